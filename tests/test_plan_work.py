"""Work lists of a plan, counted on the host (dxg2_plan_dry_run): no GPU."""
import ctypes
import math

import numpy as np
import pytest

from dynamix_amd import _lib
from dynamix_amd.synth import annular_qmask

GRAM_ITEMS, EVENT_ITEMS, DENSE_BYTES, EVENT_BYTES, NEEDED_BYTES = 8, 9, 12, 13, 14  # of the summary


def _desc(shape, nframes, q, dtype=_lib.DXG2_U8, flags=0):
    return _lib.PlanDesc(shape[0], shape[1], nframes, dtype, q.ctypes.data, None, 0, flags)


def _dry_run(shape, nframes, q, dtype=_lib.DXG2_U8, flags=0):
    q = np.ascontiguousarray(q, dtype=np.int32)
    d = _desc(shape, nframes, q, dtype, flags)
    s = (ctypes.c_int64 * 15)()
    _lib.check(_lib.load().dxg2_plan_dry_run(ctypes.byref(d), s, 15))
    return list(s)


@pytest.mark.parametrize("shape,nframes,bins", [((128, 128), 100000, 5), ((128, 128), 1000000, 5),
                                                ((64, 64), 2000000, 1), ((300, 300), 150000, 6),
                                                ((512, 512), 500000, 10)])
def test_event_items_of_several_lag_windows(shape, nframes, bins):
    """Every item clears and flushes all the counters of every lag window (32,704 lags), which
    costs about as much as 512 of its pixels: over the windows, the items of a small detector
    are no more than twice the 256 CUs, unless they have 1,024 pixels and more."""
    q = annular_qmask(shape, bins)
    pixels = int((q > 0).sum())
    windows = math.ceil(nframes / 32704)
    items = _dry_run(shape, nframes, q)[EVENT_ITEMS]
    assert items <= max(2 * 256 / windows, pixels / 1024) + bins
    assert items >= pixels / 8192


def _batch(jobs, dtype=_lib.DXG2_U8):
    masks = [np.ascontiguousarray(annular_qmask(s, b), dtype=np.int32) for s, _, b in jobs]
    d = (_lib.PlanDesc * len(jobs))(*[_desc(s, n, q, dtype) for (s, n, _), q in zip(jobs, masks)])
    out = (ctypes.c_int64 * 3)()
    _lib.check(_lib.load().dxg2_batch_dry_run(d, len(jobs), out, 3))
    return list(out), masks


def _whole(jobs, masks):
    """(items, k-blocks of the longest) with a bin's k-blocks in one item: a tile pair and bin each."""
    items = longest = 0
    for (_, n, _), q in zip(jobs, masks):
        nt = math.ceil(n / 256)
        kb = np.ceil(np.bincount(q.ravel())[1:] / 64)
        items += nt * (nt + 1) // 2 * int((kb > 0).sum())
        longest = max(longest, int(kb.max()))
    return items, longest


def test_grouped_items_are_cut_for_the_joined_list():
    """A small plan cuts its few tiles along k to fill the chip alone; sixteen of them in one
    launch fill it with whole items, and their order among bigger jobs does not matter."""
    small, large = ((96, 96), 500, 5), ((256, 256), 3000, 8)
    alone, masks = _batch([small])
    assert alone[0] > _whole([small], masks)[0]
    assert alone[0] == _dry_run(small[0], small[1], masks[0])[GRAM_ITEMS]
    for jobs in ([small] * 16, [large] * 4 + [small], [small] + [large] * 4):
        got, masks = _batch(jobs)
        assert (got[0], got[2]) == _whole(jobs, masks)


def test_grouped_items_of_uint16_plans_and_empty_masks():
    """HH and LL of every tile pair in the plain list, both halves of the cross product in the
    other; a plan without bins adds none."""
    small = ((96, 96), 500, 5)
    jobs = [small] * 16
    got, masks = _batch(jobs, _lib.DXG2_U16)
    assert got[0] == got[1] == 2 * _whole(jobs, masks)[0]
    q = np.zeros((8, 8), np.int32)
    d = (_lib.PlanDesc * 1)(_desc((8, 8), 10, q))
    out = (ctypes.c_int64 * 3)()
    _lib.check(_lib.load().dxg2_batch_dry_run(d, 1, out, 3))
    assert list(out) == [0, 0, 0]


@pytest.mark.parametrize("flags", [0, _lib.DXG2_FLAG_NO_QUEUE])
def test_serving_reserves_at_least_what_a_job_takes(flags):
    """GpuExecutor.footprint_bound() against what the plan it stands for cannot do without, outputs
    and input included, on both sides of the line from which a plan may have a narrow slab."""
    from dynamix_amd import serving
    specs = serving.make_jobs(14, 10.0, 17)
    specs += serving.make_jobs(20, 10.0, 18, shapes=((64, 48), (96, 96), (131, 77)),
                               nframes=(100, 3000), bins=(1, 12))
    specs += serving.make_jobs(10, 10.0, 19, shapes=((256, 256),), nframes=(2400, 3400))
    seen = set()
    for spec in specs:
        h, w = spec.shape
        n, q = spec.nframes, serving.job_qmask(spec)
        nb = int(q.max())
        s = _dry_run(spec.shape, n, q, flags=flags)
        out = nb * n * 28
        bound = serving.GpuExecutor.footprint_bound(None, spec)
        if spec.layout == "dense":
            need = s[NEEDED_BYTES] + out + n * h * w
            seen.add(s[DENSE_BYTES] >= s[NEEDED_BYTES] + s[2] // 2)   # a narrow slab beside it
            assert s[DENSE_BYTES] >= s[NEEDED_BYTES] > s[2]
            if min(spec.shape) >= 256:
                assert bound <= 1.25 * need or flags
        else:
            events = int(1.25 * serving.EVENT_MEAN * n * h * w)
            need = s[EVENT_BYTES] + out + 5 * events + 4 * (h * w + 1)
        assert need <= bound, spec
    assert seen == ({False} if flags else {True, False})
