"""Op::RmsNorm (rlx-cpu/src/thunk.rs:8839-8869) fused into the decode GEMV's activation staging, alone and in front of
the SwiGLU and LM-head epilogues."""
import ctypes as C

import numpy as np
import pytest

import oracle
import rlx_amd
from rlx_amd import QuantScheme, ops
from helpers import Q4K, Q4_0, Q6K, Q8_0, make_weights, random_blocks, rel_err


# ---- oracle pins ------------------------------------------------------------------------------------------------

def test_rms_norm_closed_forms():
    h = 64
    gamma = np.linspace(0.5, 2.0, h).astype(np.float32)
    beta = np.linspace(-1.0, 1.0, h).astype(np.float32)
    x = np.full((1, h), -3.0, np.float32)  # constant row: x / rms = -1 up to eps
    assert np.allclose(oracle.rms_norm(x, gamma, beta, 0.0), -gamma + beta, rtol=0, atol=1e-6)
    assert np.array_equal(oracle.rms_norm(np.zeros((1, h), np.float32), gamma, beta, 1e-5), beta.reshape(1, h))  # 0 * finite
    r = np.random.default_rng(0).standard_normal((3, h)).astype(np.float32)
    a, b = oracle.rms_norm(r, gamma, None, 0.0), oracle.rms_norm(4.0 * r, gamma, None, 0.0)  # scale invariant (4 is exact)
    assert np.allclose(a, b, rtol=2e-7, atol=0)


def test_rms_norm_matches_numpy_f64():
    rng = np.random.default_rng(1)
    x = rng.standard_normal((5, 4096)).astype(np.float32) * 3
    gamma, beta = rng.standard_normal(4096).astype(np.float32), rng.standard_normal(4096).astype(np.float32)
    x64 = x.astype(np.float64)
    want = x64 / np.sqrt((x64 ** 2).mean(axis=1, keepdims=True) + 1e-5) * gamma + beta
    got = oracle.rms_norm(x, gamma, beta, 1e-5)
    assert np.max(np.abs(got - want) / np.maximum(np.abs(want), 1.0)) < 5e-6  # 4096 sequential f32 additions


# ---- GPU ---------------------------------------------------------------------------------------------------------

def weights(scheme, n, k, seed):
    if scheme == Q6K:
        return random_blocks(scheme, n, k, seed=seed, d_std=5e-6)
    return make_weights(scheme, n, k, seed=seed)[0]


@pytest.mark.gpu
@pytest.mark.parametrize("scheme,m,k,ns,with_beta", [(Q4_0, 1, 4096, (4096, 1024, 1024), True), (Q4K, 3, 2048, (300, 77), False),
                                                      (Q8_0, 8, 512, (130,), True), (Q6K, 2, 768, (96, 48), True),
                                                      (Q4_0, 1, 28672, (64,), False)])
def test_rmsnorm_prologue_matches_norm_then_matmul(scheme, m, k, ns, with_beta):
    rng = np.random.default_rng(2)
    x = (rng.standard_normal((m, k)) * 2.5).astype(np.float32)
    gamma = (1.0 + 0.1 * rng.standard_normal(k)).astype(np.float32)
    beta = (0.05 * rng.standard_normal(k)).astype(np.float32) if with_beta else None
    packed = [weights(scheme, n, k, 10 + i) for i, n in enumerate(ns)]
    ws = [ops.QWeight(QuantScheme(scheme), p, n, k) for p, n in zip(packed, ns)]
    got = ops.rmsnorm_gguf_matmul_bt_batch(x, gamma, beta, 1e-5, ws, m)
    xn = oracle.rms_norm(x, gamma, beta, 1e-5)  # the reference's two ops: RmsNorm, then DequantMatMul
    for g, p, n, w in zip(got, packed, ns, ws):
        assert rel_err(g, oracle.gguf_matmul_f64(xn, p, m, k, n, scheme)) <= 2e-3
        sep = ops.gguf_matmul_bt(xn, w, m)  # the unfused device path on the oracle's normalized vector
        assert np.max(np.abs(g - sep) / np.maximum(np.abs(sep), 1.0)) <= 2e-5
        w.free()


@pytest.mark.gpu
@pytest.mark.parametrize("scheme,m,k,n", [(Q4_0, 1, 128, 33), (Q8_0, 5, 2080, 48), (Q4K, 7, 1024, 272), (Q4_0, 3, 4096, 4112), (Q8_0, 8, 14336, 16)])
@pytest.mark.parametrize("size", [1e-6, 1.0, 1e6, 1e21])
def test_rmsnorm_scale_is_applied_to_the_sums(scheme, m, k, n, size):
    """x gamma times a power of two is staged and the sums are scaled; squares that overflow (the last size) make a factor of 0, as in
    the reference's own f32 arithmetic."""
    rng = np.random.default_rng(5)
    x = (rng.standard_normal((m, k)) * size).astype(np.float32)
    gamma = (1.0 + 0.1 * rng.standard_normal(k)).astype(np.float32)
    p = weights(scheme, n, k, 20)
    w = ops.QWeight(QuantScheme(scheme), p, n, k)
    got = ops.rmsnorm_gguf_matmul_bt_batch(x, gamma, None, 1e-12, [w], m)[0]
    if size > 1e20:
        assert not oracle.rms_norm(x, gamma, None, 1e-12).any() and not got.any()
    else:
        x64 = x.astype(np.float64)
        xn = x64 / np.sqrt((x64 ** 2).mean(axis=1, keepdims=True) + 1e-12) * gamma
        ref = xn @ oracle.dequant(scheme, p, n * k).reshape(n, k).astype(np.float64).T
        # at most 448 f32 additions of block sums, a random walk of half an ulp of the row's largest values: 2^-24 sqrt(448)
        assert np.max(np.abs(got - ref)) <= 1.3e-6 * np.max(np.abs(ref))
    w.free()


@pytest.mark.gpu
@pytest.mark.parametrize("scheme,m,k,n", [(Q4_0, 1, 128, 33), (Q4_0, 1, 4096, 64), (Q8_0, 8, 14336, 16), (Q4K, 6, 2048, 272)])
def test_rmsnorm_launch_takes_rows_of_any_size(scheme, m, k, n):
    """Without eps the outputs of x and of x 2^p have the same bits as long as both go the same way: every factor on it is a power of two.
    (The slow pass stages normalized values, whose roundings differ.)"""
    rng = np.random.default_rng(6)
    x = rng.standard_normal((m, k)).astype(np.float32)
    gamma = (1.0 + 0.1 * rng.standard_normal(k)).astype(np.float32)
    w = ops.QWeight(QuantScheme(scheme), weights(scheme, n, k, 21), n, k)
    first = ops.rmsnorm_gguf_matmul_bt_batch(x, gamma, None, 0.0, [w], m)[0]
    for p in (-40, -13, -9, 12, 14, 30):
        assert np.array_equal(ops.rmsnorm_gguf_matmul_bt_batch(x * np.float32(2.0 ** p), gamma, None, 0.0, [w], m)[0], first), p
    w.free()


@pytest.mark.gpu
@pytest.mark.parametrize("scheme,m,k,n", [(Q4_0, 1, 512, 33), (Q8_0, 3, 2080, 48), (Q4K, 8, 14336, 16)])
@pytest.mark.parametrize("first,largest", [(0.0, 2.0 ** p) for p in (-13, -10, -9, -8, -7, 0, 14, 15, 17)] +
                         [(1.0, 2.0 ** p) for p in (13, 14, 15, 16, 20)] + [(2.0 ** -20, 1.0), (2.0 ** 40, 2.0 ** 41)])
@pytest.mark.parametrize("gamma_size,with_beta", [(1.0, False), (1.0, True), (2.0 ** 16, True)])
def test_rmsnorm_range_around_the_limits(scheme, m, k, n, first, largest, gamma_size, with_beta):
    """Rows whose first columns (`first`) say little about the largest value: zeros, or smaller by as much as the range of binary16. With
    a beta, or a large gamma, normalized values are staged."""
    rng = np.random.default_rng(7)
    x = np.clip(rng.standard_normal((m, k)) / 4, -1, 1) * largest
    x[:, 300] = largest
    x[:, :256] = np.clip(rng.standard_normal((m, 256)) / 2, -1, 1) * first
    x = x.astype(np.float32)
    gamma = (gamma_size * (1.0 + 0.1 * rng.standard_normal(k))).astype(np.float32)
    beta = (0.05 * rng.standard_normal(k)).astype(np.float32) if with_beta else None
    p = weights(scheme, n, k, 22)
    w = ops.QWeight(QuantScheme(scheme), p, n, k)
    got = ops.rmsnorm_gguf_matmul_bt_batch(x, gamma, beta, 1e-12, [w], m)[0]
    w.free()
    x64 = x.astype(np.float64)
    xn = x64 / np.sqrt((x64 ** 2).mean(axis=1, keepdims=True) + 1e-12) * gamma + (0 if beta is None else beta)
    ref = xn @ oracle.dequant(scheme, p, n * k).reshape(n, k).astype(np.float64).T
    # at most 448 f32 additions of block sums, a random walk of half an ulp of the row's largest values: 2^-24 sqrt(448)
    assert np.max(np.abs(got - ref)) <= 1.3e-6 * np.max(np.abs(ref))


@pytest.mark.gpu
def test_rmsnorm_swiglu_and_argmax():
    rng = np.random.default_rng(3)
    m, k, n = 1, 2048, 700
    x = (rng.standard_normal((m, k)) * 1.5).astype(np.float32)
    gamma = (1.0 + 0.1 * rng.standard_normal(k)).astype(np.float32)
    up_b, gate_b = weights(Q4_0, n, k, 1), weights(Q4_0, n, k, 2)
    w_up, w_gate = ops.QWeight(QuantScheme.GgufQ4_0, up_b, n, k), ops.QWeight(QuantScheme.GgufQ4_0, gate_b, n, k)
    xn = oracle.rms_norm(x, gamma, None, 1e-6)
    got = ops.rmsnorm_gguf_matmul_swiglu(x, gamma, None, 1e-6, w_up, w_gate, m)
    u64, g64 = (oracle.gguf_matmul_f64(xn, b, m, k, n, Q4_0) for b in (up_b, gate_b))
    assert rel_err(got, u64 * g64 / (1 + np.exp(-g64))) <= 2e-3
    assert np.max(np.abs(got - ops.gguf_matmul_swiglu(xn, w_up, w_gate, m))) <= 2e-5
    idx, val = ops.rmsnorm_gguf_tied_lm_argmax(x[0], gamma, None, 1e-6, w_up)
    logits = ops.gguf_matmul_bt(xn, w_up, 1)[0]
    assert idx == int(np.argmax(logits)) and abs(val - logits[idx]) <= 2e-5 * max(abs(logits[idx]), 1.0)
    # top-k behind the same fused norm: its first entry is the argmax, its values are the (normalised) logits, in order
    tidx, tval = ops.rmsnorm_gguf_tied_lm_topk(x[0], gamma, None, 1e-6, w_up, 12)
    assert (int(tidx[0]), float(tval[0])) == (idx, val) and np.all(np.diff(tval) <= 0) and len(set(tidx.tolist())) == 12
    assert np.all(np.abs(tval - logits[tidx]) <= 2e-5 * np.maximum(np.abs(logits[tidx]), 1.0))
    assert tval[-1] >= np.sort(logits)[-12] - 2e-5
    w_up.free()
    w_gate.free()


@pytest.mark.gpu
@pytest.mark.parametrize("scheme,m", [(Q4_0, 1), (Q4K, 6)])
def test_rmsnorm_swiglu_and_argmax_take_rows_of_any_size(scheme, m):
    """As test_rmsnorm_launch_takes_rows_of_any_size, through the other two epilogues."""
    rng = np.random.default_rng(8)
    k, n = 2048, 700
    x = rng.standard_normal((m, k)).astype(np.float32)
    gamma = (1.0 + 0.1 * rng.standard_normal(k)).astype(np.float32)
    up, gate = (ops.QWeight(QuantScheme(scheme), weights(scheme, n, k, 23 + i), n, k) for i in range(2))
    first = ops.rmsnorm_gguf_matmul_swiglu(x, gamma, None, 0.0, up, gate, m)
    best = ops.rmsnorm_gguf_tied_lm_argmax(x[0], gamma, None, 0.0, up)
    for p in (-40, -12, 15, 30):
        scaled = x * np.float32(2.0 ** p)
        assert np.array_equal(ops.rmsnorm_gguf_matmul_swiglu(scaled, gamma, None, 0.0, up, gate, m), first), p
        assert ops.rmsnorm_gguf_tied_lm_argmax(scaled[0], gamma, None, 0.0, up) == best, p
    up.free()
    gate.free()


@pytest.mark.gpu
@pytest.mark.parametrize("m,k", [(1, 4096), (6, 2048)])
def test_rmsnorm_follows_what_the_launch_before_wrote(m, k):
    """The row's power of two is read through the scalar cache. Launches stand one behind the other on one buffer that
    a copy on the stream rewrites in between with rows of very different sizes, and nothing is waited for."""
    rng = np.random.default_rng(9)
    n = 512
    gamma = (1.0 + 0.1 * rng.standard_normal(k)).astype(np.float32)
    w = ops.QWeight(QuantScheme.GgufQ4_0, weights(Q4_0, n, k, 25), n, k)
    rows = [rng.standard_normal((m, k)).astype(np.float32) for _ in range(3)]
    want = [ops.rmsnorm_gguf_matmul_bt_batch(x, gamma, None, 0.0, [w], m)[0] for x in rows]
    L, check = rlx_amd._lib.lib(), rlx_amd._lib.check
    stream = C.c_void_p()
    check(L.rlx_mi355x_stream_create(C.byref(stream)))
    sizes = (0, -30, 25, -12, 40, 14)
    inputs = {(i, p): ops.DeviceBuffer.from_numpy(x * np.float32(2.0 ** p)) for i, x in enumerate(rows) for p in sizes}
    slot, gd = ops.DeviceBuffer(m * k * 4), ops.DeviceBuffer.from_numpy(gamma)
    order = [(int(rng.integers(3)), sizes[int(rng.integers(len(sizes)))]) for _ in range(150)]
    outs = [ops.DeviceBuffer(m * n * 4) for _ in order]
    wp = (C.c_void_p * 1)(w.ptr)
    ops.sync()
    for key, out in zip(order, outs):
        check(L.rlx_mi355x_memcpy_d2d(slot.ptr, inputs[key].ptr, m * k * 4, stream))
        check(L.rlx_mi355x_rmsnorm_gguf_matmul_bt_batch(slot.ptr, gd.ptr, None, 0.0, wp, (C.c_void_p * 1)(out.ptr), 1, m,
                                                        stream))
    check(L.rlx_mi355x_stream_sync(stream))
    for key, out in zip(order, outs):
        assert np.array_equal(out.to_numpy(np.float32).reshape(m, n), want[key[0]]), key
    check(L.rlx_mi355x_stream_destroy(stream))
    w.free()


@pytest.mark.gpu
def test_rmsnorm_argument_errors():
    w = ops.QWeight(QuantScheme.GgufQ4_0, weights(Q4_0, 32, 256, 1), 32, 256)
    with pytest.raises(rlx_amd.RlxError, match="decode path"):
        ops.rmsnorm_gguf_matmul_bt_batch(np.zeros((9, 256), np.float32), np.ones(256, np.float32), None, 1e-5, [w], 9)
    w.free()


@pytest.mark.gpu
@pytest.mark.parametrize("h", [2048, 2052, 2056, 4096, 4100, 8192, 8196, 14336, 16384, 16388, 4097])
@pytest.mark.parametrize("rows,with_beta", [(1, True), (700, False)])
def test_rms_norm_rows_kept_in_registers(h, rows, with_beta):
    """Both sides of every row length at which rlx_rmsnorm_rows_keep changes its workgroup or hands over to the kernel that reads a row twice."""
    rng = np.random.default_rng(h + rows)
    x = (rng.standard_normal((rows, h)) * 3).astype(np.float32)
    gamma = rng.standard_normal(h).astype(np.float32)
    beta = rng.standard_normal(h).astype(np.float32) if with_beta else None
    got = ops.rms_norm(x, gamma, beta, 1e-5)
    x64 = x.astype(np.float64)
    want = x64 / np.sqrt((x64 ** 2).mean(axis=1, keepdims=True) + 1e-5) * gamma + (0 if beta is None else beta)
    # per thread at most 64 additions of squares, then a tree: the factor is good to 32 ulp, the element itself adds four roundings
    assert np.max(np.abs(got - want) / np.maximum(np.abs(want), 1.0)) <= 36 * 2.0 ** -24


@pytest.mark.gpu
@pytest.mark.parametrize("rows,h", [(300, 3072), (300, 3076), (256, 10240), (257, 10240), (1400, 11996), (1399, 12000), (1400, 12000), (900, 14996), (899, 15000), (900, 15000), (257, 15996), (257, 16000)])
def test_rms_norm_rows_around_the_dispatch(rows, h):
    """Both sides of the lines between rows kept in registers, on three sizes of workgroup, and rows read twice."""
    rng = np.random.default_rng(h + rows)
    x = (rng.standard_normal((rows, h), dtype=np.float32) * 3)
    gamma = rng.standard_normal(h).astype(np.float32)
    got = ops.rms_norm(x, gamma, None, 1e-5)
    want = x / np.sqrt((x.astype(np.float64) ** 2).mean(axis=1, keepdims=True) + 1e-5) * gamma
    assert np.max(np.abs(got - want) / np.maximum(np.abs(want), 1.0)) <= 36 * 2.0 ** -24  # as above
