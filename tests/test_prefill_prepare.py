"""Activation preparation of the prefill path (rlx_xrowscale, rlx_xprep): a workspace that holds NaN everywhere, so that an image row read
without having been written shows, around the 64-row passes of small batches; both ways of scanning the rows; and an image made once for
matmuls of two schemes."""
import ctypes as C

import numpy as np
import pytest

import rlx_amd
from helpers import Q2K, Q4_0, Q4K, Q5K, Q6K, Q8_0, f32_to_bf16_bits, make_weights, random_blocks, rel_err
from rlx_amd import DType, QuantScheme, ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("scheme", [Q4_0, Q4K, Q2K])
@pytest.mark.parametrize("m,x_dtype", [(17, DType.F32), (33, DType.F32), (64, DType.F32), (65, DType.F32), (33, DType.BF16), (64, DType.BF16),
                                       (65, DType.BF16), (128, DType.BF16), (129, DType.BF16), (100, DType.F16)])
def test_no_image_row_is_read_that_was_not_written(oracle, scheme, m, x_dtype):
    n, k = 208, 1280
    check(oracle, scheme, n, k, m, x_dtype)


# a workgroup per row below 2048 rows of 16384 bytes or more, else a wave per row: both sides of both lines
@pytest.mark.parametrize("m,k,x_dtype", [(2047, 64, DType.F32), (2049, 32, DType.F32), (70, 4064, DType.F32), (70, 4096, DType.F32), (70, 16416, DType.F32),
                                         (2047, 4096, DType.F32), (2048, 4096, DType.F32), (70, 8160, DType.BF16), (70, 8192, DType.BF16)])
def test_row_scan_by_waves_and_by_workgroups(oracle, m, k, x_dtype):
    check(oracle, Q4_0, 48, k, m, x_dtype, rows=[0, 3, 5, m // 2, m - 1])


@pytest.mark.parametrize("first,second,m,n,k,x_dtype,leaves", [
    (Q4K, Q4_0, 1111, 4100, 4608, DType.F32, "rlx_gemm_big_q4_0: 1 matrix, shared tiles"),  # pieces of tiles
    (Q4K, Q8_0, 40, 1100, 4096, DType.F32, "rlx_gemvw_q8_0: 1 matrix, split K"),            # 64 rows a pass
    (Q2K, Q6K, 40, 200, 2048, DType.BF16, "rlx_gemm64_q6_k: 1 matrix, split K"),            # 64-row tiles
    (Q5K, Q6K, 300, 200, 2048, DType.F32, "rlx_gemm_q6_k: 1 matrix, split K"),              # 256-row tiles
])
def test_an_image_stays_whole_through_matmuls_of_other_schemes(first, second, m, n, k, x_dtype, leaves):
    # prepared once for a scheme with block sums; between two matmuls of that scheme another scheme's partial results go into the
    # same workspace, which holds what either scheme asks for
    rng = np.random.default_rng(m + n)
    x = rng.standard_normal((m, k)).astype(np.float32)
    xd = ops.DeviceBuffer.from_numpy(f32_to_bf16_bits(x) if x_dtype == DType.BF16 else x)
    L = rlx_amd._lib.lib()
    ws = [ops.QWeight(QuantScheme(s), random_blocks(s, n, k, seed=i, d_std=2e-3, dmin_std=2e-3) if s in (Q2K, Q5K, Q6K) else make_weights(s, n, k, seed=i)[0], n, k)
          for i, s in enumerate((first, second))]
    need = max(L.rlx_mi355x_gguf_matmul_workspace(s, int(x_dtype), m, k, n) for s in (first, second))
    assert leaves in ops.matmul_plan(second, x_dtype, m, k, [n], need)[1][0]
    wsb, od = ops.DeviceBuffer(need), ops.DeviceBuffer(m * n * 4)
    rlx_amd._lib.check(L.rlx_mi355x_gguf_matmul_prepare(xd.ptr, int(x_dtype), first, m, k, wsb.ptr, need, None))

    def product(w):
        rlx_amd._lib.check(L.rlx_mi355x_gguf_matmul_bt_prepared(wsb.ptr, need, int(x_dtype), (C.c_void_p * 1)(w.ptr), (C.c_void_p * 1)(od.ptr), 1, m, None))
        ops.sync()
        return od.to_numpy(np.uint32)

    before = product(ws[0])
    product(ws[1])
    assert np.array_equal(product(ws[0]), before)
    for w in ws:
        w.free()


def check(oracle, scheme, n, k, m, x_dtype, rows=None):
    rng = np.random.default_rng(m + k)
    x = rng.standard_normal((m, k)).astype(np.float32)
    x[5, -1] = 0 if x_dtype == DType.F16 else 30000.0  # the largest value of its row stands last: found by the last thread of the scan
    xin = x
    if x_dtype == DType.BF16:
        xin = f32_to_bf16_bits(x)
        x = (xin.astype(np.uint32) << 16).view(np.float32)
    elif x_dtype == DType.F16:
        xin = x.astype(np.float16)
        x = xin.astype(np.float32)
    packed = random_blocks(scheme, n, k, seed=k, d_std=2e-3, dmin_std=2e-3) if scheme == Q2K else make_weights(scheme, n, k, seed=k)[0]
    w = ops.QWeight(QuantScheme(scheme), packed, n, k)
    L = rlx_amd._lib.lib()
    need = L.rlx_mi355x_gguf_matmul_workspace(scheme, int(x_dtype), m, k, n)
    ws = ops.DeviceBuffer.from_numpy(np.full(need, 0xFF, np.uint8))
    xd, od = ops.DeviceBuffer.from_numpy(xin), ops.DeviceBuffer(m * n * 4)
    rlx_amd._lib.check(L.rlx_mi355x_gguf_matmul_bt(xd.ptr, int(x_dtype), w.ptr, od.ptr, m, ws.ptr, need, None))
    ops.sync()
    got = od.to_numpy(np.float32).reshape(m, n)
    assert np.isfinite(got).all()
    rows = np.arange(m) if rows is None else np.array(rows)
    rest = rows[rows != 5]
    assert rel_err(got[rest], oracle.gguf_matmul_f64(x[rest], packed, len(rest), k, n, scheme)) <= 2e-3
    want = oracle.gguf_matmul_f64(x[5:6], packed, 1, k, n, scheme)[0]  # the row with the large value: a weight's rounding is 2^-12 of it at most
    assert np.linalg.norm(got[5] - want) <= 2.0 ** -11 * np.linalg.norm(want)
    w.free()
