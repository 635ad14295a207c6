"""Softmax over rows held in registers, a bias added to rows, and column sums (a bias gradient), at the edges of their forms: row
lengths around a wavefront, a block and the longest row in registers, few and many rows, odd lengths and unaligned rows; infinities,
the lowest float and NaN; in place; gradients into fresh and into used memory."""
import numpy as np
import pytest

from lantern_amd import _lib
from lantern_amd import backend as B
from tests.util import Dev

pytestmark = pytest.mark.gpu
LENGTHS = [1, 2, 63, 64, 65, 255, 256, 257, 1000, 1024, 1025, 4095, 4096, 4097]


@pytest.mark.parametrize("c", LENGTHS)
@pytest.mark.parametrize("rows", [1, 5, 2051])
def test_softmax_rows_and_gradient(on_hip, rows, c):
    """Against 64 bits: the exponent of a value is off by its own rounding (2^-24 of values up to about 20), a sum of c positive terms
    and the functions by a few roundings more: 1e-5 relative, the gradients the same of their terms' magnitudes."""
    if rows * c > 4 << 20:
        rows = (4 << 20) // c
    d = Dev(on_hip)
    be, mark = d.be, on_hip.getMallocAddr()
    rng = np.random.RandomState(c)
    x, g, base = (rng.standard_normal((rows, c)).astype(np.float32) * s for s in (4, 1, 1))
    x64 = x.astype(np.float64)
    e = np.exp(x64 - x64.max(1, keepdims=True))
    prob = e / e.sum(1, keepdims=True)
    for log in (True, False):
        want = np.log(prob) if log else prob
        X = d.up(x)
        y = be.softmax(log, X, rows, c, 1)
        got = d.down(y, (rows, c))
        assert (np.abs(got - want) <= 1e-5 * (np.abs(want) + (np.abs(x64).max() if log else 0)) + 1e-37).all()
        be.lib.lh_softmax(int(log), X.ptr, X.ptr, rows, c, 1); _lib.check()                # in place
        np.testing.assert_array_equal(d.down(X, (rows, c)), got)
        g64, y64 = g.astype(np.float64), got.astype(np.float64)
        grad = g64 - np.exp(y64) * g64.sum(1, keepdims=True) if log else y64 * (g64 - (g64 * y64).sum(1, keepdims=True))
        mag = np.abs(g64) + (np.exp(y64) if log else np.abs(y64)) * (np.abs(g64).sum(1, keepdims=True) if log else (np.abs(g64) + (np.abs(g64) * np.abs(y64)).sum(1, keepdims=True)))
        G = d.up(g)
        fresh, used = d.zeros(rows * c), d.up(base)
        be.lib.lh_softmax_grad(int(log), y.ptr, G.ptr, fresh.ptr, rows, c, 1)
        be.lib.lh_softmax_grad(int(log), y.ptr, G.ptr, used.ptr, rows, c, 1); _lib.check()
        assert (np.abs(d.down(fresh, (rows, c)) - grad) <= 1e-6 * mag + 1e-37).all()
        assert (np.abs(d.down(used, (rows, c)) - (grad + base)) <= 1e-6 * (mag + np.abs(base)) + 1e-37).all()
        be.resetMallocAddr(mark)


def test_softmax_of_rows_without_a_finite_maximum(on_hip):
    d, low = Dev(on_hip), np.float32(-3.402823466e38)
    mark = on_hip.getMallocAddr()
    for c in (5, 300, 2000):
        x = np.zeros((4, c), np.float32)
        x[0], x[1, :] = low, -np.inf
        x[2, 1], x[3, 0] = np.nan, -np.inf
        y = d.down(on_hip.softmax(True, d.up(x), 4, c, 1), (4, c))
        np.testing.assert_allclose(d.down(on_hip.softmax(False, d.up(x[:1]), 1, c, 1), (c,)), 1 / c, rtol=1e-6)       # (log: the maximum swallows the sum's logarithm)
        assert np.isnan(y[2]).all() and y[3, 0] == -np.inf and np.allclose(y[3, 1:], -np.log(c - 1), rtol=1e-6)
        assert not np.isfinite(y[1]).any()
    on_hip.resetMallocAddr(mark)


SHAPES = [((7, 5), (5,)), ((1000, 3), (3,)), ((64, 1000), (1000,)), ((2, 4096), (4096,)), ((8192, 66), (66,)), ((3, 5, 4, 8), (4, 8)), ((3, 5, 4, 8), (5, 4, 8)),
          ((6, 5, 4, 4), (5, 1, 1)), ((2, 1, 9), (9,)), ((70000, 4), (4,)), ((33, 257), (257,)),
          # rows side by side in a block: up to 128 threads a row (of one element or of four), remainders of rows and of threads
          ((1031, 2), (2,)), ((600001, 3), (3,)), ((2051, 127), (127,)), ((2051, 128), (128,)), ((2051, 129), (129,)), ((517, 508), (508,)), ((517, 512), (512,)), ((517, 516), (516,)), ((3, 6), (6,))]


@pytest.mark.parametrize("full,small", SHAPES)
@pytest.mark.parametrize("op", [B.ADD, B.SUB, B.MUL, B.DIV])
def test_broadcast_over_rows(on_hip, full, small, op):
    """One operation an element: numpy's bits.  Column sums (+= and -=, and the gradients of + and -): within sqrt(rows) + 8 roundings
    of the terms' root sum of squares, and the same bits twice."""
    d = Dev(on_hip)
    mark = on_hip.getMallocAddr()
    rng = np.random.RandomState(7)
    a, b = rng.standard_normal(full).astype(np.float32), (rng.standard_normal(small) + 3).astype(np.float32)
    fn = [np.add, np.subtract, np.multiply, np.divide][op]
    r = len(full)
    sd = (1,) * (r - len(small)) + small
    A, Bb = d.up(a), d.up(b)
    out = d.zeros(a.size)
    on_hip.lib.lh_bcast_op(op, A.ptr, B._ints(full), Bb.ptr, B._ints(sd), out.ptr, B._ints(full), r); _lib.check()
    np.testing.assert_array_equal(d.down(out, full), fn(a, b))
    on_hip.lib.lh_bcast_update(op, A.ptr, B._ints(full), Bb.ptr, B._ints(sd), r); _lib.check()
    np.testing.assert_array_equal(d.down(A, full), fn(a, b))
    if op in (B.ADD, B.SUB):
        axes = tuple(i for i in range(r) if sd[i] == 1 and full[i] != 1)
        s64, mag = a.astype(np.float64).sum(axes, keepdims=True).reshape(small), np.sqrt((a.astype(np.float64) ** 2).sum(axes, keepdims=True)).reshape(small)
        rows = a.size // b.size
        tol = (np.sqrt(rows) + 8) * 2.0 ** -24 * (mag + np.abs(b))
        A = d.up(a)
        got = []
        for _ in range(2):
            t = d.up(b)
            on_hip.lib.lh_bcast_update(op, t.ptr, B._ints(sd), A.ptr, B._ints(full), r); _lib.check()
            got.append(d.down(t, small))
        np.testing.assert_array_equal(got[0], got[1])
        assert (np.abs(got[0] - (b + s64 if op == B.ADD else b - s64)) <= tol).all()
        gb = d.up(b)
        ga = d.zeros(a.size)
        on_hip.lib.lh_bcast_op_grad(op, A.ptr, ga.ptr, B._ints(full), 0, Bb.ptr, gb.ptr, B._ints(sd), 0, A.ptr, B._ints(full), r); _lib.check()
        assert (np.abs(d.down(gb, small) - (b + s64 if op == B.ADD else b - s64)) <= tol).all()
        np.testing.assert_array_equal(d.down(ga, full), a)
    on_hip.resetMallocAddr(mark)


@pytest.mark.parametrize("rows,cols", [(64, 1000), (65, 300), (129, 77), (256, 1000), (2048, 512), (2049, 64), (4096, 4096), (5000, 800), (1024, 65536)])
def test_column_sums_round_no_more_than_a_wavefront_per_column(on_hip, rows, cols):
    """The order of the sum this one replaced: 64 lanes that add up every 64th row, then halves of the lanes onto each other.  The rms of
    the error against 64 bits over the columns (a statistic of `cols` samples: 4 / sqrt(cols) wide) is not above that order's."""
    d = Dev(on_hip)
    mark = on_hip.getMallocAddr()
    a = np.random.RandomState(rows).standard_normal((rows, cols)).astype(np.float32)
    exact = np.sum(a, 0, dtype=np.float64)
    t, A = d.zeros(cols), d.up(a)
    on_hip.lib.lh_bcast_update(B.ADD, t.ptr, B._ints((1, cols)), A.ptr, B._ints((rows, cols)), 2); _lib.check()
    got = d.down(t, (cols,))
    lanes = np.zeros((64, cols), np.float32)
    for r in range(0, rows, 64):
        part = a[r:r + 64]
        lanes[:len(part)] += part
    while len(lanes) > 1:
        lanes = lanes[:len(lanes) // 2] + lanes[len(lanes) // 2:]
    rms = lambda e: float(np.sqrt(np.mean(np.square(e))))      # noqa: E731
    assert rms(got - exact) <= rms(lanes[0] - exact) * (1 + 4 / np.sqrt(cols)), (rms(got - exact), rms(lanes[0] - exact))
    on_hip.resetMallocAddr(mark)


def test_recorded_column_sums_leave_memory_handed_out_later_alone(on_hip):
    """A graph's replay runs what was recorded at the addresses it was recorded with: partial sums kept above the arena's top would land
    in what the program has allocated there since."""
    d, rows, cols = Dev(on_hip), 4096, 96
    mark = on_hip.getMallocAddr()
    a = np.random.RandomState(3).standard_normal((rows, cols)).astype(np.float32)
    A, t = d.up(a), d.zeros(cols)
    on_hip.toHost(t, cols)
    on_hip.captureBegin()
    on_hip.lib.lh_bcast_update(B.ADD, t.ptr, B._ints((1, cols)), A.ptr, B._ints((rows, cols)), 2); _lib.check()
    graph = on_hip.captureEnd()
    later = np.arange(1 << 16, dtype=np.float32)
    held = d.up(later)
    for r in range(1, 4):
        on_hip.graphLaunch(graph)
        tol = r * (np.sqrt(rows) + 8) * 2.0 ** -24 * np.sqrt(rows * 16.0)
        assert (np.abs(d.down(t, (cols,)) - r * a.astype(np.float64).sum(0)) <= tol).all()
        np.testing.assert_array_equal(d.down(held, (1 << 16,)), later)
    on_hip.graphDestroy(graph)
    on_hip.resetMallocAddr(mark)


@pytest.mark.parametrize("N,K,P,Q", [(100, 10, 24, 24), (1, 3, 64, 64), (7, 5, 24, 25), (33, 16, 8, 16), (64, 700, 2, 2), (300, 1, 31, 33), (4097, 2, 1, 1)])
@pytest.mark.parametrize("masked", [False, True])
def test_bias_gradient(on_hip, N, K, P, Q, masked):
    """Slices of the batch around 16 KiB, masked by a relu on the way or not: sums of N P Q terms, each rounding at most 2^-24 of a partial
    sum (below four times the terms' root sum of squares), the roundings like their square root, 8 for the rest."""
    d = Dev(on_hip)
    mark = on_hip.getMallocAddr()
    rng = np.random.RandomState(N)
    y, dy = rng.standard_normal((N, K, P, Q)).astype(np.float32), rng.standard_normal((N, K, P, Q)).astype(np.float32)
    base = rng.standard_normal(K).astype(np.float32)
    X, Y, G, db, dw = d.up(rng.standard_normal((N, 1, P, Q)).astype(np.float32)), d.up(y), d.up(dy), d.up(base), d.zeros(K)
    if masked:
        on_hip.lib.lh_unary_grad(B.RELU, Y.ptr, Y.ptr, G.ptr, G.ptr, y.size, 1, 0.0, 0.0)
    on_hip.lib.lh_conv2d_bwd_filter(X.ptr, G.ptr, dw.ptr, db.ptr, 1.0, N, 1, P, Q, K, 1, 1, 1, 1, 0, 0); _lib.check()
    g = np.where(y > 0, dy, 0).astype(np.float64) if masked else dy.astype(np.float64)
    bound = (4 * np.sqrt(N * P * Q) + 8) * 2.0 ** -24 * (np.sqrt((g ** 2).sum((0, 2, 3))) + np.abs(base))
    assert (np.abs(d.down(db, (K,)) - (base + g.sum((0, 2, 3)))) <= bound).all()
    np.testing.assert_array_equal(d.down(G, y.shape), g.astype(np.float32))
    on_hip.resetMallocAddr(mark)


@pytest.mark.parametrize("outer,dim,inner", [(1, 1, 5), (3, 7, 70), (1, 8, 257), (2, 9, 64), (5, 17, 3), (1, 384, 800), (1, 511, 1600), (300, 700, 64)])
def test_sums_over_the_middle_add_in_row_order(on_hip, outer, dim, inner):
    """One thread an output, rows in their order: numpy's bits for the same order."""
    d = Dev(on_hip)
    mark = on_hip.getMallocAddr()
    x = np.random.RandomState(dim).standard_normal((outer, dim, inner)).astype(np.float32)
    X, y = d.up(x), d.zeros(outer * inner)
    on_hip.lib.lh_sum_dim(X.ptr, y.ptr, outer, dim, inner); _lib.check()
    want = np.zeros((outer, inner), np.float32)
    for r in range(dim):
        want += x[:, r]
    np.testing.assert_array_equal(d.down(y, want.shape), want)
    on_hip.resetMallocAddr(mark)
