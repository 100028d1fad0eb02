"""Work lists of a plan, counted on the host (dxg2_plan_dry_run): no GPU."""
import ctypes
import math

import numpy as np
import pytest

from dynamix_amd import _lib
from dynamix_amd.synth import annular_qmask

EVENT_ITEMS = 9      # index of the summary


def _dry_run(shape, nframes, q, dtype=_lib.DXG2_U8, flags=0):
    q = np.ascontiguousarray(q, dtype=np.int32)
    d = _lib.PlanDesc(shape[0], shape[1], nframes, dtype, q.ctypes.data, None, 0, flags)
    s = (ctypes.c_int64 * 12)()
    _lib.check(_lib.load().dxg2_plan_dry_run(ctypes.byref(d), s, 12))
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
