"""The recurrence as one launch (lh_rnn_seq.hip) against the same layer with one launch per time step (LH_RNN_SEQ=0), which
test_parity_ops.py holds to the oracle: at the edges of its tiles (16 units, 16 batch rows, groups of 16 k dealt to 4 wavefronts),
of its register forms and of its launch plans; replayed from a graph; and when a block gives up waiting."""
import ctypes

import numpy as np
import pytest

from lantern_amd._lib import LanternHipError
from tests.util import Dev

pytestmark = pytest.mark.gpu
GATES = {0: 1, 1: 1, 2: 4, 3: 3}          # relu, tanh, LSTM, GRU


def _one_launch_passes(be):
    stats = (ctypes.c_int64 * 9)()
    be.lib.lh_fusion_stats(stats, 9)
    return stats[8]


def _waited(be):
    """An event the host has waited for, without the error check of lh_sync."""
    e = be.lib.lh_event_create()
    be.lib.lh_event_record(e)
    assert be.lib.lh_event_elapsed_ms(e, e) == 0
    return e


def _layer(d, mode, T, B, I, H, bidir, init, seed=5):
    """Forward and backward of one layer; everything it returns or leaves behind."""
    be, rng, D, G = d.be, np.random.RandomState(seed), 2 if bidir else 1, GATES[mode] * H
    f = lambda *s: rng.standard_normal(s).astype(np.float32)      # noqa: E731
    x, w, dy = f(T, B, I), f(D * (G * I + G * H + 2 * G)) * np.float32(0.7 / np.sqrt(H)), f(T, B, D * H)
    hx, cx = (d.up(f(D, B, H)) if init else None), (d.up(f(D, B, H)) if init and mode == 2 else None)
    X, W, DY, dx, dw = d.up(x), d.up(w), d.up(dy), d.zeros(x.size), d.zeros(w.size)
    if mode < 2:
        y = be.rnn_forward(mode, X, W, T, B, I, H, bidir, hx=hx)
        be.rnn_backward(mode, X, y, DY, W, dx, dw, T, B, I, H, bidir, 1.0, hx=hx)
    else:
        y, reserve = be.rnn_gated_forward(mode, X, W, T, B, I, H, bidir, hx=hx, cx=cx)
        be.rnn_gated_backward(mode, X, y, DY, W, reserve, dx, dw, T, B, I, H, bidir, 1.0, hx=hx, cx=cx)
    return [d.down(y, dy.shape), d.down(dx, x.shape), d.down(dw, w.shape)]


CASES = [  # mode, T, B, I, H, both directions, initial state
    (1, 12, 1, 5, 1, False, False), (1, 12, 16, 7, 15, True, True), (0, 13, 17, 9, 16, False, True), (1, 14, 33, 8, 17, True, False),
    (1, 12, 3, 12, 255, False, False), (1, 13, 2, 12, 257, True, False), (0, 12, 5, 20, 1023, False, False), (1, 12, 2, 20, 1025, False, True),
    (1, 12, 1, 20, 2048, False, False),
    (2, 4, 1, 5, 1, True, True), (2, 7, 16, 6, 63, False, True), (2, 5, 17, 6, 64, True, False), (2, 5, 31, 6, 66, False, True),
    (2, 6, 2, 16, 129, True, True), (2, 4, 48, 16, 320, True, False), (2, 4, 64, 16, 800, True, True), (2, 4, 1, 16, 800, False, False),
    (2, 9, 16, 6, 257, True, False),
    (3, 4, 2, 5, 3, False, True), (3, 8, 16, 6, 48, True, False), (3, 5, 17, 6, 65, False, True), (3, 6, 40, 16, 257, True, True),
    (3, 4, 64, 16, 512, True, False), (3, 4, 33, 16, 800, False, True),
]


@pytest.mark.parametrize("case", CASES, ids=lambda c: "-".join(map(str, c)))
def test_one_launch_against_one_per_step(hip_backend, monkeypatch, case):
    """Both sum fp32 products of the same operands in fp32, in another order (backward: through bfloat16 terms that hold the
    operands exactly).  A sum of K <= 4 H products differs by about sqrt(K) * 2^-24 of its rms term, a step hands its difference to
    the next with a factor around one (weights of norm about 0.7), and T <= 14 of them add up: below 1e-5 of the result's rms, four
    times which is allowed."""
    d = Dev(hip_backend)
    mark, before = d.be.getMallocAddr(), _one_launch_passes(d.be)
    got = _layer(d, *case)
    d.be.resetMallocAddr(mark)
    assert _one_launch_passes(d.be) == before + 2, "forward and backward are one launch each"
    monkeypatch.setenv("LH_RNN_SEQ", "0")
    want = _layer(d, *case)
    d.be.resetMallocAddr(mark)
    assert _one_launch_passes(d.be) == before + 2
    for name, a, b in zip(("y", "dx", "dw"), got, want):
        rms = float(np.sqrt(np.mean(np.square(b, dtype=np.float64))))
        assert np.isfinite(a).all() and np.abs(a - b).max() <= 4e-5 * (np.abs(b).max() + rms), name


@pytest.mark.parametrize("T,B,H,forward,backward", [(47, 512, 128, 0, 1), (48, 512, 128, 1, 1), (12, 256, 129, 1, 1), (12, 256, 128, 1, 1), (11, 2, 16, 0, 0)])
def test_which_layers_are_one_launch(hip_backend, T, B, H, forward, backward):
    """Both directions of a tanh layer: below 12 steps, and forward below 48 where the directions follow each other and have 128 units
    at most, one launch per step is faster."""
    d = Dev(hip_backend)
    be = d.be
    mark = be.getMallocAddr()
    X, W = d.zeros(T * B * 4), d.zeros(2 * (H * 4 + H * H + 2 * H))
    before = _one_launch_passes(be)
    y = be.rnn_forward(1, X, W, T, B, 4, H, True)
    assert _one_launch_passes(be) == before + forward
    be.rnn_backward(1, X, y, d.zeros(T * B * 2 * H), W, d.zeros(X.n), d.zeros(W.n), T, B, 4, H, True)
    assert _one_launch_passes(be) == before + forward + backward
    be.sync()
    be.resetMallocAddr(mark)


@pytest.mark.parametrize("mode", [1, 2, 3])
def test_not_a_number_stays_in_its_batch_row(hip_backend, mode):
    """One NaN in the input of a sample (with the bits the ring uses for an empty word): that sample's later states are NaN, no
    other sample's are, and nobody waits for it."""
    d, T, B, I, H = Dev(hip_backend), 12, 18, 8, 40
    be, rng = d.be, np.random.RandomState(2)
    mark = be.getMallocAddr()
    x = rng.standard_normal((T, B, I)).astype(np.float32)
    x[2, 4, 1] = np.array([0xffffffff], np.uint32).view(np.float32)[0]
    G = GATES[mode] * H
    W = d.up((rng.standard_normal(G * I + G * H + 2 * G) * 0.1).astype(np.float32))
    X = d.up(x)
    y = be.rnn_forward(mode, X, W, T, B, I, H, False) if mode < 2 else be.rnn_gated_forward(mode, X, W, T, B, I, H, False)[0]
    y = d.down(y, (T, B, H))
    assert np.isnan(y[2:, 4]).all() and np.isfinite(y[:2]).all() and np.isfinite(np.delete(y, 4, axis=1)).all()
    be.resetMallocAddr(mark)


def test_replayed_from_a_graph(hip_backend):
    d, T, B, I, H, G = Dev(hip_backend), 12, 20, 24, 96, 4 * 96
    be, rng = d.be, np.random.RandomState(3)
    mark = be.getMallocAddr()
    x = rng.standard_normal((T, B, I)).astype(np.float32)
    W = d.up((rng.standard_normal(G * I + G * H + 2 * G) * 0.1).astype(np.float32))
    X = d.up(x)
    want = d.down(be.rnn_gated_forward(2, X, W, T, B, I, H, False)[0], (T, B, H))
    be.sync()
    be.lib.lh_capture_begin()
    y, _ = be.rnn_gated_forward(2, X, W, T, B, I, H, False)
    graph = be.lib.lh_capture_end(); d.check()
    for _ in range(4):
        be.fillInPlace(y, y.n, 7.0)
        be.lib.lh_graph_launch(graph); d.check()
        np.testing.assert_array_equal(d.down(y, (T, B, H)), want)
        np.testing.assert_array_equal(d.down(be.rnn_gated_forward(2, X, W, T, B, I, H, False)[0], (T, B, H)), want)     # eager work in between
    be.lib.lh_graph_destroy(graph)
    be.resetMallocAddr(mark)


@pytest.mark.parametrize("mode", [1, 2, 3])
def test_a_recording_leaves_memory_handed_out_later_alone(hip_backend, mode):
    """The ring is not arena memory: what a program allocates behind a recording, where the arena's top was, stays as it is in every
    replay; replayed from the side stream the recurrence still runs by itself (the ring has one user at a time)."""
    d, T, B, I, H, D = Dev(hip_backend), 13, 33, 8, 72, 2
    be, lib, rng, G = d.be, d.be.lib, np.random.RandomState(6), GATES[mode] * 72
    mark = be.getMallocAddr()
    x = rng.standard_normal((T, B, I)).astype(np.float32)
    X, W = d.up(x), d.up((rng.standard_normal(D * (G * I + G * H + 2 * G)) * 0.1).astype(np.float32))
    Y, Y2, R = d.zeros(T * B * D * H), d.zeros(T * B * D * H), d.zeros(be.lib.lh_rnn_gated_reserve_floats(mode, T, B, H, 1)) if mode > 1 else None

    def forward(y):
        if mode < 2:
            lib.lh_rnn_fwd(mode, X.ptr, W.ptr, y.ptr, T, B, I, H, 1)
        else:
            lib.lh_rnn_gated_fwd(mode, X.ptr, W.ptr, y.ptr, R.ptr, T, B, I, H, 1)
        d.check()
    forward(Y)
    want = d.down(Y, (T, B, D * H))
    be.captureBegin()
    forward(Y)
    graph = be.captureEnd()
    later = np.arange(2 << 20, dtype=np.float32)
    held = d.up(later)
    for side in (False, True, False, True):
        be.fillInPlace(Y, Y.n, 7.0)
        be.fillInPlace(Y2, Y2.n, 7.0)
        if side:
            lib.lh_side_begin()
        be.graphLaunch(graph)
        if side:
            lib.lh_side_end()
            if mode < 2:                    # (the gated modes' reserve has one user at a time)
                forward(Y2)
                np.testing.assert_array_equal(d.down(Y2, want.shape), want)
        np.testing.assert_array_equal(d.down(Y, want.shape), want)
        np.testing.assert_array_equal(d.down(held, later.shape), later)
    be.graphDestroy(graph)
    be.resetMallocAddr(mark)


def test_a_wait_that_runs_out_is_reported_once(hip_backend, monkeypatch):
    d = Dev(hip_backend)
    be, rng = d.be, np.random.RandomState(4)
    mark = be.getMallocAddr()
    X, W = d.up(rng.standard_normal((40, 33, 8)).astype(np.float32)), d.up((rng.standard_normal(64 * 8 + 64 * 64 + 128) * 0.1).astype(np.float32))
    monkeypatch.setenv("LH_RNN_SEQ_SPINS", "0")            # every block goes on at once where its words are not there
    be.rnn_forward(1, X, W, 40, 33, 8, 64, False)
    with pytest.raises(LanternHipError, match="waited too long"):
        be.sync()
    monkeypatch.delenv("LH_RNN_SEQ_SPINS")
    be.sync()
    before = _one_launch_passes(be)
    y = be.rnn_forward(1, X, W, 40, 33, 8, 64, False)           # one launch per time step from here on
    assert np.isfinite(d.down(y, (40, 33, 64))).all() and _one_launch_passes(be) == before
    monkeypatch.setenv("LH_RNN_SEQ", "1")
    be.rnn_forward(1, X, W, 40, 33, 8, 64, False)
    monkeypatch.delenv("LH_RNN_SEQ")
    again = be.rnn_forward(1, X, W, 40, 33, 8, 64, False)
    assert _one_launch_passes(be) == before + 2
    np.testing.assert_allclose(d.down(again, (40, 33, 64)), d.down(y, (40, 33, 64)), atol=1e-5)
    monkeypatch.setenv("LH_RNN_SEQ_SPINS", "0")            # given up by a call that no wait has reported yet: the next one knows
    be.rnn_forward(1, X, W, 40, 33, 8, 64, False)
    monkeypatch.delenv("LH_RNN_SEQ_SPINS")
    be.lib.lh_event_destroy(_waited(be))
    be.rnn_forward(1, X, W, 40, 33, 8, 64, False)
    assert _one_launch_passes(be) == before + 3
    with pytest.raises(LanternHipError, match="waited too long"):
        be.sync()
    monkeypatch.setenv("LH_RNN_SEQ", "1")
    be.rnn_forward(1, X, W, 40, 33, 8, 64, False)
    assert _one_launch_passes(be) == before + 4
    be.sync()
    be.resetMallocAddr(mark)


def test_the_bound_is_a_waits_own(hip_backend, monkeypatch):
    """60000 steps, many of them with a poll or more that finds words missing, pass under a bound that every single wait stays far below."""
    d, T, B, I, H = Dev(hip_backend), 60000, 1, 4, 256
    be, rng = d.be, np.random.RandomState(7)
    mark = be.getMallocAddr()
    X, W = d.up(rng.standard_normal((T, B, I)).astype(np.float32)), d.up((rng.standard_normal(H * I + H * H + 2 * H) * 0.1).astype(np.float32))
    dy, dx, dw = d.up(rng.standard_normal((T, B, H)).astype(np.float32)), d.zeros(T * B * I), d.zeros(W.n)
    monkeypatch.setenv("LH_RNN_SEQ_SPINS", "1000")
    y = be.rnn_forward(1, X, W, T, B, I, H, False)
    be.sync()
    be.rnn_backward(1, X, y, dy, W, dx, dw, T, B, I, H, False)
    be.sync()
    be.resetMallocAddr(mark)
