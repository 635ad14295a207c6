"""The matrix products and convolutions compute fp32 products from three bfloat16 terms per operand: rounding against float64 at the
edges of the tiles, and what the three terms cannot hold (infinities, NaN, values that round up to infinity, values near the
smallest normal one), which the kernels compute again with fp32 instructions."""
import functools

import numpy as np
import pytest
import torch

from lantern_amd import Tensor, TensorR, _lib, gradR_loss
from tests.util import Dev

pytestmark = pytest.mark.gpu


def _sgemm(be, ta, tb, A, B):
    m, k = A.shape
    n = B.shape[1]
    a, b = be.fromHost(np.ascontiguousarray(A.T if ta else A)), be.fromHost(np.ascontiguousarray(B.T if tb else B))
    c = be.fromHost(np.zeros((m, n), np.float32))
    be.lib.lh_sgemm(ta, tb, m, n, k, 1.0, a.ptr, m if ta else k, b.ptr, k if tb else n, 0.0, c.ptr, n)
    _lib.check()
    return be.toHost(c, m * n).reshape(m, n)


# Root mean square of the error over sum |a b|.  Normal operands: rounding of a running sum of j terms is at most 2^-24 of its
# size, sqrt(j); eight roundings per 16 k (the fp32 instructions) make 2^-24 / sqrt(3) * k / 2 over 2 / pi * k = 2.7e-8 at any
# length, six (the three terms) 2.3e-8.  A row's figure, from 160 or 192 elements, stays within twice that.
ROUNDING = 2.0 * 2.7e-8


def _rounding(got, A, B, axis=None):
    A64, B64 = A.astype(np.float64), B.astype(np.float64)
    return np.sqrt((((got.astype(np.float64) - A64 @ B64) / (np.abs(A64) @ np.abs(B64))) ** 2).mean(axis))


@pytest.mark.parametrize("tt", [(0, 0), (0, 1), (1, 0), (1, 1)])
@pytest.mark.parametrize("dims", [(16, 64, 512), (64, 129, 257), (129, 128, 100), (333, 257, 31), (512, 640, 2048), (200, 136, 5000)])
@pytest.mark.parametrize("spread", [0.0, 4.0])
def test_products_against_float64(on_hip, tt, dims, spread):
    """Per element: the six products of a group of 16 k are six roundings of the running sum (at most one unit, 2^-23, of its
    size, which no partial sum's exceeds sum |a b|), a slice of a cut reduction (256 k and more) at most one more group and its
    own addition, and the three products left out are below 3 * 2^-25 of |a b|.  Root mean square: no more than the fp32
    instructions (2.7e-8 at any length for normal operands; of wide spread, 4.6e-7 measured at 8192 and less below), where any
    one product more left out would be 5.4e-8 and more at these sizes (1.5e-6 and more for wide spread)."""
    m, n, k = dims
    rng = np.random.RandomState(7)
    draw = lambda *s: (rng.standard_normal(s) * np.exp(spread * rng.standard_normal(s))).astype(np.float32)      # noqa: E731
    A, B = draw(m, k), draw(k, n)
    got = _sgemm(on_hip, tt[0], tt[1], A, B).astype(np.float64)
    A64, B64 = A.astype(np.float64), B.astype(np.float64)
    bound = (6 * -(-k // 16) + k // 32 + 2) * 2.0 ** -23 * (np.abs(A64) @ np.abs(B64))
    assert (np.abs(got - A64 @ B64) <= bound).all()
    assert _rounding(got, A, B) <= (2.8e-8 if spread == 0.0 else 4.6e-7)


@pytest.mark.parametrize("scale", [1e-25, 1e-33, 1e-36])
def test_products_of_tiny_values(on_hip, scale):
    rng = np.random.RandomState(8)
    A, B = (scale * rng.standard_normal((192, 192))).astype(np.float32), rng.standard_normal((192, 160)).astype(np.float32)
    A64, B64 = A.astype(np.float64), B.astype(np.float64)
    got = _sgemm(on_hip, 0, 0, A, B).astype(np.float64)
    assert (np.abs(got - A64 @ B64) <= 192 * 2.0 ** -23 * (np.abs(A64) @ np.abs(B64))).all()


@pytest.mark.parametrize("tt", [(0, 0), (0, 1), (1, 0), (1, 1)])
@pytest.mark.parametrize("k", [1, 2, 3, 4, 5, 8])
@pytest.mark.parametrize("spread", [0.0, 2.0])
def test_short_sums_are_no_further_off_than_fused_multiply_adds(on_hip, tt, k, spread):
    """One product is the rounded product itself; over a few the error is at most that of a chain of fused multiply-adds (here: of
    float64 sums rounded after every term; 2 % for the sampling over half a million sums)."""
    rng = np.random.RandomState(14)
    draw = lambda *s: (rng.standard_normal(s) * np.exp(spread * rng.standard_normal(s))).astype(np.float32)      # noqa: E731
    A, B = draw(512, k), draw(k, 1024)
    got = _sgemm(on_hip, tt[0], tt[1], A, B)
    chain = np.zeros((512, 1024), np.float32)
    for i in range(k):
        chain = (chain + A[:, i:i + 1].astype(np.float64) * B[i:i + 1].astype(np.float64)).astype(np.float32)
    if k == 1:
        np.testing.assert_array_equal(got, chain)
    assert _rounding(got, A, B) <= 1.02 * _rounding(chain, A, B)


@pytest.mark.parametrize("k", [100, 192, 4096])
@pytest.mark.parametrize("sa,sb", [(1e-35, 1e20), (1e-37, 1e30), (1e-38, 1e30), (1e-40, 1e36), (1e-41, 1e37), (1e30, 1e-38), (1e36, 1e-40)])
def test_operands_below_the_range_of_three_terms(on_hip, sa, sb, k):
    """Small operands against large ones: the sums are of ordinary size, the third term of the small operand is not."""
    rng = np.random.RandomState(11)
    A, B = (sa * rng.standard_normal((192, k))).astype(np.float32), (sb * rng.standard_normal((k, 160))).astype(np.float32)
    assert (_rounding(_sgemm(on_hip, 0, 0, A, B), A, B, 1) <= ROUNDING).all()


@pytest.mark.parametrize("k", [100, 192, 4096])
@pytest.mark.parametrize("scale", [1e-34, 1e-36, 1e-38, 1e-40, 1e-42])
def test_small_rows_and_columns_beside_ordinary_ones(on_hip, scale, k):
    rng = np.random.RandomState(12)
    A, B = rng.standard_normal((192, k)), 1e10 * rng.standard_normal((k, 160))
    A[5] *= scale
    A[70] *= scale
    A, B = A.astype(np.float32), B.astype(np.float32)
    assert (_rounding(_sgemm(on_hip, 0, 0, A, B), A, B, 1) <= ROUNDING).all()
    assert (_rounding(_sgemm(on_hip, 0, 1, A, B), A, B, 1) <= ROUNDING).all()
    At, Bt = np.ascontiguousarray(B.T), np.ascontiguousarray(A.T)
    assert (_rounding(_sgemm(on_hip, 1, 0, At, Bt), At, Bt, 0) <= ROUNDING).all()


@pytest.mark.parametrize("k", [64, 250, 4096])
def test_products_with_infinities_and_nan_are_those_of_fp32(on_hip, k):
    rng = np.random.RandomState(9)
    A, B = rng.standard_normal((200, k)).astype(np.float32), (0.1 * rng.standard_normal((k, 150))).astype(np.float32)
    A[3, 5], A[7, 9], A[150, 1], A[100, k - 1] = np.inf, np.nan, -np.inf, 3.4e38
    A[20, 3], A[20, 4] = np.inf, -np.inf
    B[5, 2] = 0.0
    B[k - 1] = np.clip(B[k - 1], -0.9, 0.9)
    got = _sgemm(on_hip, 0, 0, A, B)
    with np.errstate(all="ignore"):
        want = A.astype(np.float64) @ B.astype(np.float64)
    np.testing.assert_array_equal(np.isnan(got), np.isnan(want))
    inf = np.isinf(want)
    np.testing.assert_array_equal(np.isinf(got), inf)
    np.testing.assert_array_equal(got[inf], want[inf])
    ok = np.isfinite(want)
    mag = np.abs(np.where(np.isfinite(A), A, 0)).astype(np.float64) @ np.abs(B).astype(np.float64)
    assert (np.abs(got - want)[ok] <= k * 2.0 ** -23 * mag[ok]).all()


@pytest.mark.parametrize("geom", [(2, 3, 17, 20, 7, 2, 3), (2, 32, 14, 64, 3, 1, 1), (3, 64, 7, 160, 1, 1, 0), (2, 16, 20, 24, 5, 1, 0)])
def test_convolutions_with_infinities(on_hip, geom):
    """An infinity and a NaN in the input reach the outputs and filter gradients whose window holds them, and only those."""
    N, C, H, K, R, s, p = geom
    rng = np.random.RandomState(10)
    x, w = rng.standard_normal((N, C, H, H)).astype(np.float32), (0.2 * rng.standard_normal((K, C, R, R))).astype(np.float32)
    x[0, 1, 2, 3], x[1, 2, H - 1, 0] = np.inf, np.nan
    xt, wt = torch.from_numpy(x).double(), torch.from_numpy(w).double().requires_grad_()
    yt = torch.nn.functional.conv2d(xt, wt, stride=s, padding=p)
    yt.sum().backward()
    xin, kern = TensorR(Tensor.fromNumpy(x), isInput=True), TensorR(Tensor.fromNumpy(w))
    ys = []

    def objective(dummy):
        y = xin.convBBP(kern, None, (s, s), (p, p))
        ys.append(y.x.toCPU().reshape(yt.shape))
        return y.sum()
    gradR_loss(objective)(Tensor.zeros(1))
    for got, want, terms in ((ys[0], yt.detach().numpy(), C * R * R), (kern.d.toCPU().reshape(w.shape), wt.grad.numpy(), N * H * H)):
        np.testing.assert_array_equal(np.isnan(got), np.isnan(want))
        np.testing.assert_array_equal(np.isinf(got), np.isinf(want))
        ok = np.isfinite(want)
        # sums of `terms` products of size about one: that many roundings of a unit of a running sum below 8 sqrt(terms)
        assert (np.abs(got - want)[ok] <= terms * 2.0 ** -23 * 8 * np.sqrt(terms)).all()


@pytest.mark.parametrize("dims", [(8, 64, 28, 28, 128, 3, 3, 1, 1, 1, 1), (4, 256, 14, 14, 256, 1, 1, 1, 1, 0, 0), (6, 96, 15, 15, 160, 3, 3, 1, 1, 1, 1),
                                  (16, 32, 28, 28, 32, 3, 3, 1, 1, 1, 1), (8, 128, 28, 28, 256, 1, 1, 2, 2, 0, 0)], ids=lambda d: "x".join(map(str, d)))
@pytest.mark.parametrize("plant", ["infinity", "small"])
def test_plain_tile_plans_give_the_same_bits_around_what_the_terms_cannot_hold(on_hip, dims, plant, monkeypatch):
    """Deterministic mode leaves the choice among the plans with whole tiles to a timing, so an infinity or a value below the range
    of the three terms may change the arithmetic of the 32x32 blocks it is in only, which all tile shapes share."""
    dev = Dev(on_hip)
    lib = on_hip.lib
    N, Cc, H, W, K, R, S, sH, sW, pH, pW = dims
    P, Q = (H + 2 * pH - R) // sH + 1, (W + 2 * pW - S) // sW + 1
    rng = np.random.RandomState(13)
    x, w, dy = rng.randn(N, Cc, H, W).astype(np.float32), (rng.randn(K, Cc, R, S) / np.sqrt(Cc * R * S)).astype(np.float32), rng.randn(N, K, P, Q).astype(np.float32)
    value = np.float32(np.inf) if plant == "infinity" else np.float32(1.2345678e-38)
    x[1, 3, 4, 6] = dy[1, 3, 4, 5] = dy[N - 1, K - 1, P - 1, 0] = x[N - 1, 2, H - 4, 0] = value       # (even rows and columns: under a stride of two too)
    if plant == "small":
        w[7, 1, 0, 0] = w[K - 1, Cc - 1, R - 1, S - 1] = value
    xd, wd, dyd = dev.up(x), dev.up(w), dev.up(dy)
    ny, nx = N * K * P * Q, N * Cc * H * W
    lib.lh_set_deterministic(1)
    try:
        outs = {}
        for plan in (3, 2, 1, 10):
            monkeypatch.setenv("LH_FORCE_PLAN", str(plan))
            y = dev.up(np.full(ny, 7.0, np.float32)); lib.lh_conv2d_fwd(xd.ptr, wd.ptr, 0, y.ptr, *dims)
            dx = dev.up(np.full(nx, 7.0, np.float32)); lib.lh_conv2d_bwd_data(dyd.ptr, wd.ptr, dx.ptr, 0.0, *dims)
            dev.check()
            outs[plan] = (dev.down(y, (ny,)).copy(), dev.down(dx, (nx,)).copy())
        for plan in (2, 1, 10):
            np.testing.assert_array_equal(outs[plan][0], outs[3][0], err_msg="forward, plan %d against plan 3" % plan)
            np.testing.assert_array_equal(outs[plan][1], outs[3][1], err_msg="input gradient, plan %d against plan 3" % plan)
        assert plant == "small" or (np.isinf(outs[3][0]).any() and np.isinf(outs[3][1]).any())
    finally:
        monkeypatch.delenv("LH_FORCE_PLAN", raising=False)
        lib.lh_set_deterministic(0)


REDO_SHAPES = [(4, 256, 14, 14, 256, 1, 1, 1, 1, 0, 0), (16, 128, 7, 7, 128, 3, 3, 1, 1, 1, 1), (8, 128, 28, 28, 96, 3, 3, 2, 2, 1, 1), (4, 24, 30, 26, 32, 5, 3, 2, 1, 0, 1)]


@functools.lru_cache(maxsize=1)
def _odd_convolution(dims):
    """Inputs with an infinity, a NaN and a value below the range of the three terms in every 997th place; results and summed
    magnitudes in float64 (forward, input gradient, filter gradient)."""
    N, Cc, H, W, K, R, S, sH, sW, pH, pW = dims
    P, Q = (H + 2 * pH - R) // sH + 1, (W + 2 * pW - S) // sW + 1
    rng = np.random.RandomState(15)
    x, w, dy = rng.randn(N, Cc, H, W).astype(np.float32), rng.randn(K, Cc, R, S).astype(np.float32), rng.randn(N, K, P, Q).astype(np.float32)
    x.reshape(-1)[::997] = dy.reshape(-1)[::997] = w.reshape(-1)[::997] = 1.2345678e-39
    x[1, 3, 4, 6] = dy[1, 3, 4, 5] = np.inf
    x[N - 1, 2, H - 4, 0] = dy[N - 1, K - 1, P - 1, 0] = np.nan
    conv = lambda a, b: torch.nn.functional.conv2d(a, b, stride=(sH, sW), padding=(pH, pW))      # noqa: E731

    def all_three(x, w, dy):
        xt, wt = (torch.from_numpy(a).double().requires_grad_() for a in (x, w))
        y = conv(xt, wt)
        return [y.detach().numpy()] + [g.numpy() for g in torch.autograd.grad(y, (xt, wt), torch.from_numpy(dy).double())]
    clean = [np.abs(np.where(np.isfinite(a), a, 0)).astype(np.float32) for a in (x, w, dy)]
    return x, w, dy, all_three(x, w, dy), all_three(*clean)


def _check_odd(got, want, mag, what):
    np.testing.assert_array_equal(np.isnan(got), np.isnan(want), err_msg=what)
    np.testing.assert_array_equal(np.isinf(got), np.isinf(want), err_msg=what)
    inf, ok = np.isinf(want), np.isfinite(want) & (mag > 0)
    np.testing.assert_array_equal(got[inf], want[inf], err_msg=what)
    err = np.abs(got[ok].astype(np.float64) - want[ok]) / mag[ok]
    assert np.sqrt((err ** 2).mean()) <= ROUNDING, what
    assert (got[np.isfinite(want) & (mag == 0)] == 0).all(), what


@pytest.mark.parametrize("dims", REDO_SHAPES, ids=lambda d: "x".join(map(str, d)))
@pytest.mark.parametrize("plan", [-1, 1, 2, 3, 4, 5, 6, 7, 8, 9, 11, 12, 13, 14, 15, "m32"])
def test_what_the_terms_cannot_hold_under_every_launch_plan(on_hip, dims, plan, monkeypatch):
    """Whole tiles, stream-K segments, sliced last tiles, the 32-row tile, the grouped launch of a strided input gradient, the filter
    gradient's slices (added atomically and in order): infinities and NaN where float64 has them, the rest to rounding."""
    x, w, dy, want, mag = _odd_convolution(dims)
    dev, lib = Dev(on_hip), on_hip.lib
    xd, wd, dyd = dev.up(x), dev.up(w), dev.up(dy)
    if plan == "m32":
        monkeypatch.setenv("LH_FORCE_M32", "1")
    elif plan >= 0:
        monkeypatch.setenv("LH_FORCE_PLAN", str(plan))
    y, dx = dev.up(np.full(want[0].size, 7.0, np.float32)), dev.up(np.full(want[1].size, 7.0, np.float32))
    lib.lh_conv2d_fwd(xd.ptr, wd.ptr, 0, y.ptr, *dims)
    lib.lh_conv2d_bwd_data(dyd.ptr, wd.ptr, dx.ptr, 0.0, *dims)
    dev.check()
    _check_odd(dev.down(y, want[0].shape), want[0], mag[0], "forward")
    _check_odd(dev.down(dx, want[1].shape), want[1], mag[1], "input gradient")
    if plan in (-1, "m32"):
        for deterministic in (0, 1):
            lib.lh_set_deterministic(deterministic)
            try:
                dw = dev.up(np.full(want[2].size, 7.0, np.float32))
                lib.lh_conv2d_bwd_filter(xd.ptr, dyd.ptr, dw.ptr, 0, 0.0, *dims)
                dev.check()
                _check_odd(dev.down(dw, want[2].shape), want[2], mag[2], "filter gradient, deterministic %d" % deterministic)
            finally:
                lib.lh_set_deterministic(0)


@pytest.mark.parametrize("tile", [1, 2, 3, 5, 6, 7])
def test_small_filter_rows_with_the_statistics_of_their_outputs(on_hip, tile, monkeypatch):
    """The forward launch that leaves batch-norm statistics: filter rows below the range of the three terms against large inputs."""
    dims = (6, 96, 15, 15, 160, 3, 3, 1, 1, 1, 1)
    N, Cc, H, W, K = dims[:5]
    rng = np.random.RandomState(16)
    x, w = (1e10 * rng.randn(N, Cc, H, W)).astype(np.float32), 1e-10 * rng.randn(K, Cc, 3, 3)
    w[5], w[70], w[159] = 1e-28 * w[5], 1e-30 * w[70], 1e-32 * w[159]
    w = w.astype(np.float32)
    want, mag = (torch.nn.functional.conv2d(*(torch.from_numpy(f(a).astype(np.float64)) for a in (x, w)), padding=1).numpy() for f in (np.array, np.abs))
    dev, lib = Dev(on_hip), on_hip.lib
    monkeypatch.setenv("LH_FORCE_STATS_TILE", str(tile))
    xd, wd = dev.up(x), dev.up(w)
    y, sm, si, rm, rv = dev.zeros(want.size), dev.zeros(K), dev.zeros(K), dev.zeros(K), dev.zeros(K)
    lib.lh_conv2d_fwd_bnstats(xd.ptr, wd.ptr, 0, y.ptr, *dims, sm.ptr, si.ptr, rm.ptr, rv.ptr, 1e-5, 0.1)
    dev.check()
    err = (dev.down(y, want.shape).astype(np.float64) - want) / mag
    assert (np.sqrt((err ** 2).mean((0, 2, 3))) <= ROUNDING).all()
    # a channel's mean: 1350 sums, each off by at most a few units of its magnitudes
    assert (np.abs(dev.down(sm, (K,)) - want.mean((0, 2, 3))) <= 1e-6 * mag.mean((0, 2, 3))).all()
    assert (np.abs(dev.down(si, (K,)) * np.sqrt(want.var((0, 2, 3)) + 1e-5) - 1) <= 1e-5).all()
