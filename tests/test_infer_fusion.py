"""conv2D_batch -> batchNormInference [-> + shortcut] [-> relu in place] in one launch (lh_conv_infer.hip, lh_defer.hip) against the same
calls run as issued: the bookkeeping on the host over random programs, the launch on the device at the edges of its tiles."""
import os
import shutil
import subprocess

import numpy as np
import pytest

from lantern_amd import _lib
from lantern_amd import backend as B

HERE = os.path.join(os.path.dirname(os.path.abspath(__file__)), "host_cpp")


def _build_host_check(tmp_path, name):
    if shutil.which("g++") is None:
        pytest.skip("no host C++ compiler")
    exe = str(tmp_path / name)
    r = subprocess.run(["g++", "-std=c++17", "-O1", "-g", "-fsanitize=address,undefined", "-fno-sanitize-recover=all", "-x", "c++", "-I", os.path.join(HERE, "fake_hip"),
                        "-o", exe, os.path.join(HERE, name + ".cpp")], capture_output=True, text=True)
    if r.returncode != 0 and "cannot find" in r.stderr:
        pytest.skip("the sanitizer runtimes are not installed: " + r.stderr[-300:])
    assert r.returncode == 0, r.stderr[-3000:]
    env = dict(os.environ)
    env.pop("LD_PRELOAD", None)
    return exe, env


@pytest.mark.parametrize("seed", [1, 2])
def test_chains_give_what_the_calls_as_issued_give(tmp_path, seed):
    exe, env = _build_host_check(tmp_path, "defer_infer_check")
    r = subprocess.run([exe, "2000", str(seed)], capture_output=True, text=True, timeout=600, env=env)
    assert r.returncode == 0 and "identical" in r.stdout and " 0 chains" not in r.stdout, (r.stdout + r.stderr)[-3000:]


def test_chains_cost_no_more_launches_than_the_calls_as_issued(tmp_path):
    exe, env = _build_host_check(tmp_path, "defer_infer_launches")
    r = subprocess.run([exe], capture_output=True, text=True, timeout=600, env=env)
    assert r.returncode == 0 and "defer_infer_launches: ok" in r.stdout, (r.stdout + r.stderr)[-3000:]


# N, C, H, W, K, filter, stride, padding, bias, join, relu, launch form (LH_FORCE_PLAN; None: the measured one)
CASES = [
    (2, 16, 9, 11, 64, 1, 1, 0, False, False, True, 3), (2, 16, 9, 11, 65, 3, 1, 1, True, True, True, 3), (1, 32, 7, 7, 40, 3, 2, 1, False, True, False, 2),
    (3, 64, 14, 14, 128, 3, 1, 1, False, True, True, 1), (3, 64, 14, 14, 130, 1, 1, 0, True, False, False, 1), (2, 128, 14, 14, 96, 1, 2, 0, False, True, True, 2),
    (2, 256, 7, 7, 512, 1, 1, 0, False, True, True, 13), (1, 256, 14, 14, 64, 3, 1, 1, False, False, True, 14), (2, 128, 20, 20, 136, 3, 1, 1, True, True, True, 15),
    (1, 64, 56, 56, 64, 1, 1, 0, False, False, True, 16), (1, 16, 9, 11, 70, 3, 1, 1, True, True, True, 16), (1, 512, 7, 7, 512, 3, 1, 1, False, True, True, 17),
    (1, 144, 14, 14, 230, 1, 1, 0, True, True, True, 18), (2, 48, 15, 13, 66, 3, 2, 1, False, False, False, 18), (1, 512, 7, 7, 512, 3, 1, 1, False, True, True, 19),
    (1, 1008, 7, 7, 70, 1, 1, 0, False, False, True, 19),
    (1, 512, 7, 7, 512, 3, 1, 1, False, True, True, 4), (1, 512, 7, 7, 100, 1, 1, 0, False, False, False, 4),
    (2, 3, 33, 31, 64, 7, 2, 3, False, False, True, None), (2, 5, 8, 8, 7, 3, 1, 1, True, True, True, None), (8, 64, 28, 28, 256, 1, 1, 0, False, True, True, None),
    (1, 16, 1, 1, 32, 1, 1, 0, False, True, True, None),
    (2, 20, 12, 12, 50, 5, 1, 0, True, False, True, 2), (2, 20, 12, 12, 65, 5, 1, 0, False, True, True, 3), (2, 20, 12, 12, 50, 5, 1, 0, False, True, False, 4),
    (3, 9, 13, 11, 130, 3, 2, 1, False, True, True, 2), (3, 9, 13, 11, 64, 3, 1, 1, True, True, True, 3), (3, 9, 13, 11, 33, 3, 1, 1, True, False, True, 4),
    (2, 100, 7, 7, 100, 3, 1, 1, False, True, True, None), (4, 200, 7, 7, 30, 3, 1, 1, False, False, True, None), (1, 512, 14, 14, 96, 3, 1, 1, False, True, True, 4),
]


def _chain(be, lib, ops, case, seed=3):
    N, C, H, W, K, R, s, p, with_bias, join, relu, _ = case
    P, Q = (H + 2 * p - R) // s + 1, (W + 2 * p - R) // s + 1
    n = N * K * P * Q
    rng = np.random.RandomState(seed)
    f = lambda *d: be.fromHost(np.ascontiguousarray(rng.standard_normal(d).astype(np.float32)))      # noqa: E731
    x, w, bias, gamma, beta, mean = f(N, C, H, W), f(K, C, R, R), f(K), f(K), f(K), f(K)
    var, sc = be.fromHost(rng.uniform(0.3, 2.0, K).astype(np.float32)), f(n)
    y, t, out = be.mallocArray(n), be.mallocArray(n), be.mallocArray(n)
    lib.lh_conv2d_fwd(x.ptr, w.ptr, bias.ptr if with_bias else 0, y.ptr, N, C, H, W, K, R, R, s, s, p, p)
    lib.lh_bn_infer(y.ptr, gamma.ptr, beta.ptr, mean.ptr, var.ptr, t.ptr, N, K, P * Q, 1e-5)
    res = t
    if join:
        dims = B._ints((n,))
        lib.lh_bcast_op(B.ADD, t.ptr, dims, sc.ptr, dims, out.ptr, dims, 1)
        res = out
    if relu:
        lib.lh_unary(B.RELU, res.ptr, res.ptr, n, 0.0, 0.0)
    _lib.check()
    got = [be.toHost(res, n)]
    for late in (t, y):                                # what the launch left out is there when it is read
        got.append(be.toHost(late, n) if (late is not res) else got[0])
    return got, (be.toHost(x, N * C * H * W).reshape(N, C, H, W), be.toHost(w, K * C * R * R).reshape(K, C, R, R), be.toHost(bias, K) if with_bias else None,
                 [be.toHost(v, K) for v in (gamma, beta, mean, var)], be.toHost(sc, n) if join else None)


@pytest.mark.gpu
@pytest.mark.parametrize("case", CASES, ids=lambda c: "-".join(map(str, c)))
def test_chain_against_its_parts(on_hip, monkeypatch, case):
    """Deterministic mode (whole tiles only): the parts' bits.  With the launch form of the case, against 64 bits: a sum of n = C R S
    products is rounded six times per 16 of them, each time by at most 2^-24 of a partial sum; partial sums stay below four times the
    terms' root sum of squares m (4 sigma), and the roundings add up like their square root: 4 sqrt(6 n / 16) 2^-24 m, with 8 2^-24
    for the product's own rounding and the operations behind the sum, scaled as the batch norm scales them."""
    import torch
    be, lib = on_hip, on_hip.lib
    mark = be.getMallocAddr()
    N, C, H, W, K, R, s, p, with_bias, join, relu, form = case
    try:
        be.setDeterministic(True)
        det, _ = _chain(be, lib, B, case)
        lib.lh_set_fusion(0)
        parts, ops = _chain(be, lib, B, case)
        lib.lh_set_fusion(1)
        for a, b in zip(det, parts):
            np.testing.assert_array_equal(a, b)
        be.setDeterministic(False)
        if form is not None:
            monkeypatch.setenv("LH_FORCE_PLAN", str(form))
        import ctypes
        stats = (ctypes.c_int64 * 8)()
        lib.lh_fusion_stats(stats, 8); before = stats[0]
        got, _ = _chain(be, lib, B, case)
        lib.lh_fusion_stats(stats, 8)
        assert stats[0] == before + 1, "the chain did not run as one launch"
    finally:
        lib.lh_set_fusion(1)
        be.setDeterministic(False)
        be.resetMallocAddr(mark)
    x, w, bias, (gamma, beta, mean, var), sc = ops
    d = lambda a: torch.from_numpy(np.asarray(a)).double()      # noqa: E731
    y = torch.nn.functional.conv2d(d(x), d(w), d(bias) if with_bias else None, s, p)
    mag = torch.nn.functional.conv2d(d(x) ** 2, d(w) ** 2, None, s, p).sqrt()
    ch = lambda a: d(a).reshape(1, -1, 1, 1)      # noqa: E731
    scale = ch(gamma) / (ch(var) + 1e-5).sqrt()
    t = (y - ch(mean)) * scale + ch(beta)
    r = t + d(sc).reshape(t.shape) if join else t
    mag = mag * max(1.0, (4 * np.sqrt(6 * C * R * R / 16) + 8) / 8)
    tol = 8 * 2.0 ** -24 * (mag * scale.abs() + (y - ch(mean)).abs() * scale.abs() + ch(beta).abs() + r.abs() + 1)
    want = [r.clamp(min=0) if relu else r, t if join else (t.clamp(min=0) if relu else t), y]
    for g, v, name in zip(got, want, ("result", "batch norm", "convolution")):
        err = (torch.from_numpy(g).double().reshape(v.shape) - v).abs()
        bound = 8 * 2.0 ** -24 * (mag + y.abs() + 1) if name == "convolution" else tol
        assert bool((err <= bound).all()), (name, float((err / bound).max()))


@pytest.mark.gpu
@pytest.mark.parametrize("case", [(3, 20, 30, 30, 51, 5, 1, 0), (5, 9, 31, 29, 30, 3, 1, 1)], ids=lambda c: "-".join(map(str, c)))
def test_the_form_is_measured_for_any_channel_count(on_hip, case):
    """Channel counts that are no multiple of the slab's depth: among the forms is the convolution by itself with its own choice of
    plans, which a whole tile under a long reduction is far behind (100 -> 100 channels over 7x7: 81 against 31 us)."""
    import ctypes
    be, lib = on_hip, on_hip.lib
    measured, remembered = ctypes.c_int64(), ctypes.c_int64()
    seen = []
    mark = be.getMallocAddr()
    for _ in range(2):
        _chain(be, lib, B, case + (False, False, True, None))
        be.resetMallocAddr(mark)
        lib.lh_tune_counters(ctypes.byref(measured), ctypes.byref(remembered))
        seen.append((measured.value, remembered.value))
    lib.lh_set_fusion(0)
    _chain(be, lib, B, case + (False, False, True, None))          # the convolution's own plan
    lib.lh_set_fusion(1)
    be.resetMallocAddr(mark)
    lib.lh_tune_counters(ctypes.byref(measured), ctypes.byref(remembered))
    assert measured.value == seen[1][0] == seen[0][0], "the first chain measured its form and, for one of the forms, the convolution's plan"
    assert seen[1][1] > seen[0][1]


@pytest.mark.gpu
def test_outputs_outside_the_arena_outlast_a_rewind(on_hip):
    """A rewind releases arena memory: outputs of a chain in memory of the caller's own are there behind it, stored or not."""
    import ctypes
    be, lib = on_hip, on_hip.lib
    rng = np.random.RandomState(4)
    N, C, H, K = 2, 16, 8, 32
    n = N * K * H * H
    up = lambda a: be.fromHost(np.ascontiguousarray(a.astype(np.float32)))      # noqa: E731
    x, w = up(rng.standard_normal((N, C, H, H))), up(rng.standard_normal((K, C, 3, 3)))
    g, b, m, v, sc = up(rng.standard_normal(K)), up(rng.standard_normal(K)), up(rng.standard_normal(K)), up(rng.uniform(0.5, 1, K)), up(rng.standard_normal(n))
    dims = B._ints((n,))
    own = [ctypes.c_void_p() for _ in range(3)]
    for a in own:
        assert lib["hipMalloc"](ctypes.byref(a), ctypes.c_size_t(4 * n)) == 0          # (of the runtime the library is linked with)
    results = []
    try:
        be.setDeterministic(True)
        for fusion in (0, 1):
            lib.lh_set_fusion(fusion)
            y, t, o = (B.Buf(own[i].value, n) for i in range(3))
            for a in (y, t, o):
                be.fillInPlace(a, n, 7.0)
            mark = be.getMallocAddr()
            be.mallocArray(1 << 20)
            lib.lh_conv2d_fwd(x.ptr, w.ptr, 0, y.ptr, N, C, H, H, K, 3, 3, 1, 1, 1, 1)
            lib.lh_bn_infer(y.ptr, g.ptr, b.ptr, m.ptr, v.ptr, t.ptr, N, K, H * H, 1e-5)
            lib.lh_bcast_op(B.ADD, t.ptr, dims, sc.ptr, dims, o.ptr, dims, 1)
            lib.lh_unary(B.RELU, o.ptr, o.ptr, n, 0.0, 0.0)
            _lib.check()
            be.resetMallocAddr(mark)
            results.append([be.toHost(a, n) for a in (y, t, o)])
    finally:
        lib.lh_set_fusion(1)
        be.setDeterministic(False)
        be.sync()
        for a in own:
            lib["hipFree"](a)
    for a, c in zip(*results):
        np.testing.assert_array_equal(a, c)


@pytest.mark.gpu
def test_infinities_and_nan_pass_as_through_the_parts(on_hip):
    be, lib = on_hip, on_hip.lib
    mark = be.getMallocAddr()
    case = (1, 16, 6, 6, 70, 1, 1, 0, False, True, True, None)
    n = 70 * 36
    x = np.random.RandomState(1).standard_normal((1, 16, 6, 6)).astype(np.float32)
    x[0, 2, 1, 1], x[0, 3, 4, 4], x[0, 5, 0, 5] = np.inf, -np.inf, np.nan
    outs = []
    try:
        be.setDeterministic(True)
        for fusion in (1, 0):
            lib.lh_set_fusion(fusion)
            rng = np.random.RandomState(2)
            up = lambda a: be.fromHost(np.ascontiguousarray(a.astype(np.float32)))      # noqa: E731
            X, w, g, b, m, v = up(x), up(rng.standard_normal((70, 16))), up(rng.standard_normal(70)), up(rng.standard_normal(70)), up(rng.standard_normal(70)), up(rng.uniform(0.5, 1, 70))
            y, t = be.mallocArray(n), be.mallocArray(n)
            lib.lh_conv2d_fwd(X.ptr, w.ptr, 0, y.ptr, 1, 16, 6, 6, 70, 1, 1, 1, 1, 0, 0)
            lib.lh_bn_infer(y.ptr, g.ptr, b.ptr, m.ptr, v.ptr, t.ptr, 1, 70, 36, 1e-5)
            lib.lh_unary(B.RELU, t.ptr, t.ptr, n, 0.0, 0.0)
            outs.append(be.toHost(t, n))
    finally:
        lib.lh_set_fusion(1)
        be.setDeterministic(False)
        be.resetMallocAddr(mark)
    np.testing.assert_array_equal(outs[0], outs[1])
    assert np.isnan(outs[0]).any()
