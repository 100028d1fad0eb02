"""Narrow pixels in FP4 (counts of at most 4 in magnitude): the dense call's numerators, sums
and denominators are the same integers as the oracle's whichever pixels are narrow."""
import numpy as np
import pytest

from oracle import g2 as og

pytestmark = pytest.mark.gpu


def _correlate(frames, q, calls=1):
    import torch
    from dynamix_amd.correlator.dense import MatMulCorrelator
    c = MatMulCorrelator(frames.shape[1:], frames.shape[0], q)
    d = torch.from_numpy(frames).cuda()
    for _ in range(calls):
        g2 = c.correlate(d)
    return c, g2


def _check(c, g2, ref):
    np.testing.assert_array_equal(c.last_numerators.cpu().numpy(), ref["num"])
    np.testing.assert_array_equal(c.last_sums.cpu().numpy(), ref["sums"])
    np.testing.assert_array_equal(c.last_denominators.cpu().numpy(),
                                  np.asarray(ref["den"], np.float64))
    fin = np.isfinite(ref["g2"])
    assert np.array_equal(fin, np.isfinite(g2))
    np.testing.assert_allclose(g2[fin], ref["g2"][fin], rtol=1e-6)


def _frames(n, shape, dtype, kind):
    rng = np.random.default_rng(n + len(kind))
    f = np.where(rng.random((n,) + shape) < 0.1, rng.integers(1, 5, size=(n,) + shape), 0)
    if dtype == np.int8:
        f = f * rng.choice([-1, 1], size=f.shape)
    if kind == "edges":                   # one count past the line, in the first and last frame
        f[0, 0, 0] = f[-1, 2, 3] = 5
        f[n // 2, shape[0] - 1, shape[1] - 1] = -128 if dtype == np.int8 else 255
    elif kind == "hot":                   # a share of the pixels always wide
        f[:, ::4, ::3] = rng.integers(0, 100, size=f[:, ::4, ::3].shape)
    elif kind == "all":                   # no narrow pixel worth keeping
        f = rng.integers(-128 if dtype == np.int8 else 0, 128 if dtype == np.int8 else 256,
                         size=f.shape)
    return f.astype(dtype)


@pytest.mark.parametrize("kind", ["none", "edges", "hot", "all"])
@pytest.mark.parametrize("dtype", [np.uint8, np.int8])
@pytest.mark.parametrize("n,shape", [(31, (20, 24)), (257, (33, 37)), (700, (48, 64))])
def test_narrow_against_oracle(n, shape, dtype, kind, monkeypatch):
    """Odd k-block counts, partial k-blocks and frame groups, several bins and one empty one;
    a second call on the same plan after one with other pixels wide."""
    print("[case] narrow n=%d %s %s %s" % (n, shape, np.dtype(dtype).name, kind), flush=True)
    monkeypatch.setenv("DXG2_NARROW", "2")
    q = np.random.default_rng(n).integers(0, 3, size=shape).astype(np.int32)
    q[:, : shape[1] // 2] = 4             # bin 3 is empty
    f = _frames(n, shape, dtype, kind)
    c, g2 = _correlate(f, q)
    _check(c, g2, og.dense_g2(f, q))
    import torch
    other = _frames(n, shape, dtype, "hot" if kind != "hot" else "edges")
    g2 = c.correlate(torch.from_numpy(other).cuda())
    _check(c, g2, og.dense_g2(other, q))


@pytest.mark.parametrize("mean", [0.02, 0.12, 0.4])
@pytest.mark.parametrize("n,shape", [(3000, (260, 300)), (4500, (192, 256))])
def test_narrow_by_work_equals_i8(n, shape, mean, monkeypatch):
    """At sizes that take the narrow route by themselves (short and long finish): equal to
    the i8 path, for few, some and mostly wide pixels."""
    from dynamix_amd import synth
    from dynamix_amd.correlator.dense import MatMulCorrelator
    print("[case] narrow by work n=%d %s mean=%g" % (n, shape, mean), flush=True)
    f = synth.speckle_frames_device(shape, n, mean, 50.0, 3, np.dtype(np.uint8))
    q = synth.annular_qmask(shape, 4)
    out = []
    for opt in ("1", "0"):
        monkeypatch.setenv("DXG2_NARROW", opt)
        c = MatMulCorrelator(shape, n, q, extra_options={"return_device": True})
        g2 = c.correlate(f)
        out.append([x.cpu().numpy() for x in (g2, c.last_numerators, c.last_sums,
                                              c.last_denominators)])
    for a, b in zip(*out):
        np.testing.assert_array_equal(a, b)


def _route(c):
    return next(iter(c._plans.values())).dense_route()


@pytest.mark.parametrize("dtype", [np.uint8, np.int8])
@pytest.mark.parametrize("kind,fp4", [("none", True), ("edges", True), ("all", False)])
def test_narrow_route_taken(kind, fp4, dtype, monkeypatch):
    """The integers are those of either route: which one ran, and with which wide pixels, is
    what the plan says.  Then a call of another kind, a plan without the option, and a replay."""
    import torch
    from dynamix_amd.correlator.dense import MatMulCorrelator
    print("[case] narrow route %s %s" % (kind, np.dtype(dtype).name), flush=True)
    monkeypatch.setenv("DXG2_NARROW", "2")
    n, shape = 257, (33, 37)
    q = np.ones(shape, np.int32)
    q[2, 3] = 0                               # one of the three wide pixels of "edges" is masked
    f = _frames(n, shape, dtype, kind)
    wide = int(((np.abs(f.astype(np.int32)) > 4).any(0) & (q > 0)).sum())
    c, g2 = _correlate(f, q)
    _check(c, g2, og.dense_g2(f, q))
    assert _route(c) == (fp4, wide if fp4 else 0)
    c.correlate(torch.from_numpy(f).cuda(), calc_std=True)
    assert _route(c) == (False, 0)
    graph = MatMulCorrelator(shape, n, q, extra_options={"graph": True})
    d = torch.from_numpy(f).cuda()
    for _ in range(3):
        _check(graph, graph.correlate(d), og.dense_g2(f, q))
    assert _route(graph) == (fp4, wide if fp4 else 0)
    monkeypatch.setenv("DXG2_NARROW", "0")
    c, g2 = _correlate(f, q)
    assert _route(c) == (False, 0)
