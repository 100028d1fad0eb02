"""The narrow slab (FP4) is an option of the dense call: where it cannot be had, or would not
be used, the call takes the i8 slab alone and gives the same integers."""
import ctypes

import numpy as np
import pytest

from oracle import g2 as og

pytestmark = pytest.mark.gpu

SHAPE, N = (40, 48), 520


class _Allocator(object):
    """Device memory from torch's allocator, but for the size `refuse`; every size asked for."""

    def __init__(self, refuse=0):
        import torch
        from dynamix_amd import _lib
        self.refuse, self.sizes, self.live = refuse, [], 0
        dev = torch.cuda.current_device()

        def alloc(nbytes, stream, ctx):
            self.sizes.append(int(nbytes))
            if nbytes == self.refuse:
                return None
            self.live += 1
            return torch.cuda.caching_allocator_alloc(int(nbytes), dev, int(stream or 0))

        def free(ptr, stream, ctx):
            self.live -= 1
            torch.cuda.caching_allocator_delete(int(ptr))

        self.lib = _lib.load()
        self._alloc, self._free = _lib.ALLOC_FN(alloc), _lib.FREE_FN(free)

    def plan(self, q, dtype):
        """A plan that keeps this allocator."""
        from dynamix_amd import _lib
        from dynamix_amd.correlator.common import Plan
        _lib.check(self.lib.dxg2_set_allocator(self._alloc, self._free, None))
        try:
            return Plan(SHAPE, N, q, dtype)
        finally:
            _lib.check(self.lib.dxg2_set_allocator(_lib.ALLOC_FN(), _lib.FREE_FN(), None))


def _inputs(dtype=np.uint8):
    rng = np.random.default_rng(5)
    q = rng.integers(0, 4, size=SHAPE).astype(np.int32)
    f = np.where(rng.random((N,) + SHAPE) < 0.1, rng.integers(1, 6, size=(N,) + SHAPE), 0)
    return q, f.astype(dtype)


def _slab4(q):
    """Bytes of the narrow slab: half a byte an entry of the lists padded to 64 pixels, 768
    rows (520 frames in steps of 256)."""
    n = np.bincount(q.ravel(), minlength=4)[1:]
    return int(((n + 63) // 64 * 64).sum()) * 768 // 2


def _outs(nb):
    import torch
    return (torch.zeros((nb, N), dtype=torch.int64, device="cuda"),
            torch.zeros((nb, N), dtype=torch.int64, device="cuda"),
            torch.zeros((nb, N), dtype=torch.float64, device="cuda"),
            torch.zeros((nb, N), dtype=torch.float32, device="cuda"))


def _call(plan, frames, outs):
    import torch
    from dynamix_amd import _lib
    st = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    _lib.check(plan.lib.dxg2_correlate_dense(plan.handle, _lib.ptr(frames),
                                             *[_lib.ptr(x) for x in outs], st))


def _check(outs, ref):
    np.testing.assert_array_equal(outs[0].cpu().numpy(), ref["num"])
    np.testing.assert_array_equal(outs[1].cpu().numpy(), ref["sums"])
    np.testing.assert_array_equal(outs[2].cpu().numpy(), np.asarray(ref["den"], np.float64))


@pytest.mark.parametrize("which", ["slab", "lists"])
def test_refused_workspace_leaves_the_i8_route(which, monkeypatch):
    """The narrow slab, or its wide pixels' list, is refused: the call succeeds on the i8 slab,
    keeps nothing of the workspace and does not ask again."""
    import torch
    print("[case] narrow workspace refused: %s" % which, flush=True)
    monkeypatch.setenv("DXG2_NARROW", "2")
    q, f = _inputs()
    slab4 = _slab4(q)
    refuse = slab4 if which == "slab" else SHAPE[0] * SHAPE[1] + 16   # the flags of the pixels
    a = _Allocator(refuse)
    plan = a.plan(q, np.uint8)
    outs, ref = _outs(3), og.dense_g2(f, q)
    d = torch.from_numpy(f).cuda()
    before = a.live
    for _ in range(2):
        _call(plan, d, outs)
        _check(outs, ref)
    assert a.sizes.count(refuse) == 1 and a.sizes.count(slab4) == 1
    assert a.live == before + 1           # the i8 slab
    plan.close()
    assert a.live == 0


def test_frames_that_cannot_use_it_do_not_make_it(monkeypatch):
    """Frames at an odd address take the general gather: no narrow slab is allocated for them."""
    import torch
    print("[case] narrow workspace, frames at an odd address", flush=True)
    monkeypatch.setenv("DXG2_NARROW", "2")
    q, f = _inputs()
    a = _Allocator()
    plan = a.plan(q, np.uint8)
    outs, ref = _outs(3), og.dense_g2(f, q)
    buf = torch.empty(f.size + 16, dtype=torch.uint8, device="cuda")
    odd = buf[1:1 + f.size].view(f.shape)
    odd.copy_(torch.from_numpy(f))
    _call(plan, odd, outs)
    _check(outs, ref)
    assert _slab4(q) not in a.sizes
    _call(plan, torch.from_numpy(f).cuda(), outs)
    _check(outs, ref)
    assert a.sizes.count(_slab4(q)) == 1
    plan.close()


def test_capture_after_another_dense_call(monkeypatch):
    """A plan that has its i8 slab (from a calc_std call) and is then captured by its user's
    graph: the plain call allocates and clears nothing under the capture.  Several replays,
    each against the oracle."""
    import torch
    from dynamix_amd import _lib
    from dynamix_amd.correlator.common import Plan
    print("[case] plain dense call first made under capture", flush=True)
    monkeypatch.setenv("DXG2_NARROW", "2")
    q, f = _inputs()
    other = (f[::-1] % 5).copy()
    refs = [og.dense_g2(f, q), og.dense_g2(other, q)]
    plan = Plan(SHAPE, N, q, np.uint8)
    outs = _outs(3)
    d = torch.from_numpy(f).cuda()
    dev = torch.zeros((3, N), dtype=torch.float32, device="cuda")
    st = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    _lib.check(plan.lib.dxg2_correlate_dense_std(plan.handle, _lib.ptr(d),
                                                 *[_lib.ptr(x) for x in outs], _lib.ptr(dev), st))
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        _call(plan, d, outs)
    for k in range(4):
        d.copy_(torch.from_numpy(other if k % 2 else f))
        for x in outs:
            x.zero_()
        g.replay()
        torch.cuda.synchronize()
        _check(outs, refs[k % 2])
        (torch.randn(1 << 16, device="cuda") * 2).sum().item()
    _call(plan, d, outs)                  # the same plan, eagerly, may take the narrow route
    _check(outs, refs[1])


def test_settings_are_read_when_the_plan_is_created(monkeypatch):
    """DXG2_NARROW is a setting of the plan: a change after its creation moves neither its
    footprint nor its route."""
    import torch
    print("[case] DXG2_NARROW changed after the plan's creation", flush=True)
    q, f = _inputs()
    ref, outs, d = og.dense_g2(f, q), _outs(3), torch.from_numpy(f).cuda()
    size = {}
    for made, later in (("2", "0"), ("0", "2")):
        monkeypatch.setenv("DXG2_NARROW", made)
        a = _Allocator()
        plan = a.plan(q, np.uint8)
        size[made] = plan.footprint(0)
        monkeypatch.setenv("DXG2_NARROW", later)
        assert plan.footprint(0) == size[made]
        _call(plan, d, outs)
        _check(outs, ref)
        assert (_slab4(q) in a.sizes) == (made == "2")
        plan.close()
    assert size["2"] > size["0"] + _slab4(q)


def test_a_plan_that_declines_the_narrow_slab(monkeypatch):
    """set_narrow(False): no narrow slab, the footprint without it, the same integers; and back."""
    import torch
    print("[case] narrow slab declined", flush=True)
    monkeypatch.setenv("DXG2_NARROW", "2")
    q, f = _inputs()
    ref, outs, d = og.dense_g2(f, q), _outs(3), torch.from_numpy(f).cuda()
    a = _Allocator()
    plan = a.plan(q, np.uint8)
    assert plan.footprint(0) >= plan.footprint(5) + _slab4(q)
    for k, on in enumerate((False, True, False)):
        plan.set_narrow(on)
        assert (plan.footprint(0) > plan.footprint(5)) == on
        _call(plan, d, outs)
        _check(outs, ref)
        assert on or plan.dense_route() == (False, 0)
        assert a.sizes.count(_slab4(q)) == (k > 0)
    plan.close()
    assert a.live == 0
