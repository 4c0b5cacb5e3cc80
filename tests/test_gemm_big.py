"""The 256 x 256 tile prefill kernel (csrc/kernels/gemm_big.hip): tiles handed out whole and shared between workgroups, ragged rows, columns
and K, f32 and 16-bit activations, code images, several matrices in one launch. Which of these a size is comes from an estimate of
times, so every case asks the plan of its launch first: a changed estimate fails here instead of testing another kernel."""
import ctypes as C

import numpy as np
import pytest

import rlx_amd
from helpers import Q4_0, Q8_0, f32_to_bf16_bits, rel_err
from rlx_amd import DType, QuantScheme, ops
from test_bench_launches import tiled_packed

pytestmark = pytest.mark.gpu
TOL = 2e-3  # the matmul's bound: one rounding of d * code to binary16 per weight


def planned(scheme, m, ns, k, x_dtype, room=None):
    launches = ops.matmul_plan(scheme, x_dtype, m, k, ns, room)[1]
    assert len(launches) == 1
    kernel, rest = launches[0].split(": ")
    return kernel, rest.split(", ")[1]


def run(scheme, m, ns, k, x_dtype, seed, plan, lean=False, offset=0):
    rng = np.random.default_rng(seed)
    x = rng.standard_normal((m, k)).astype(np.float32)
    x[3] *= 3e4  # a row whose values are carried with a power of two
    bits = f32_to_bf16_bits(x)
    if x_dtype == DType.BF16:
        x = (bits.astype(np.uint32) << 16).view(np.float32)
    packs = [tiled_packed(scheme, n, k, seed + i, 0.02).reshape(-1) for i, n in enumerate(ns)]
    ws = [ops.QWeight(QuantScheme(scheme), p, n, k) for p, n in zip(packs, ns)]
    L = rlx_amd._lib.lib()
    need = L.rlx_mi355x_gguf_matmul_workspace(scheme, int(x_dtype), m, k, 0) if lean else ops.matmul_plan(scheme, x_dtype, m, k, ns)[0]
    assert planned(scheme, m, ns, k, x_dtype, need) == plan
    wsb, xd = ops.DeviceBuffer(need), ops.DeviceBuffer.from_numpy(bits if x_dtype == DType.BF16 else x)
    outs = [ops.DeviceBuffer(m * n * 4 + 16) for n in ns]
    xp = (C.c_void_p * len(ns))(*[xd.ptr] * len(ns))
    wp = (C.c_void_p * len(ns))(*[w.ptr for w in ws])
    op = (C.c_void_p * len(ns))(*[o.ptr + offset for o in outs])
    got = []
    for _ in range(2):
        rlx_amd._lib.check(L.rlx_mi355x_gguf_matmul_bt_batch(xp, int(x_dtype), wp, op, len(ns), m, wsb.ptr, need, None))
        ops.sync()
        got.append([o.to_numpy(np.float32)[offset // 4:offset // 4 + m * n].reshape(m, n) for o, n in zip(outs, ns)])
    for a, b in zip(*got):
        assert np.array_equal(a.view(np.uint32), b.view(np.uint32))
    for w in ws:
        w.free()
    return x, packs, got[0]


@pytest.mark.parametrize("scheme,m,ns,k,x_dtype,offset,tiles", [
    (Q4_0, 1111, [4100], 4608, DType.F32, 0, "shared tiles"),          # ragged rows and columns
    (Q8_0, 1100, [4093], 4128, DType.F32, 0, "shared tiles"),          # odd columns: no 16-byte stores; K ends inside a 128-column unit of the image
    (Q4_0, 1111, [4096], 4096, DType.F32, 4, "shared tiles"),          # an output that is only 4-byte aligned
    (Q8_0, 2050, [6143], 8992, DType.BF16, 0, "whole"),                # a tile per workgroup, 16-bit rows
    (Q4_0, 1090, [4096, 1030, 1024], 8992, DType.F32, 0, "whole"),     # three matrices side by side
    (Q4_0, 700, [4096, 1030, 1024], 8192, DType.F32, 0, "shared tiles"),  # the same with pieces of the second and third
    (Q8_0, 2050, [3900], 8192, DType.BF16, 0, "shared tiles"),         # 16-bit rows
])
def test_large_tiles_match_the_oracle(oracle, scheme, m, ns, k, x_dtype, offset, tiles):
    x, packs, got = run(scheme, m, ns, k, x_dtype, m + k, ("rlx_gemm_big_q4_0" if scheme == Q4_0 else "rlx_gemm_big_q8_0", tiles), offset=offset)
    rows = [0, 1, 2, 127, 128, 255, 256, m // 2, m - 2, m - 1]
    for p, n, y in zip(packs, ns, got):
        assert rel_err(y[rows], oracle.gguf_matmul_f64(x[rows], p, len(rows), k, n, scheme)) <= TOL
        # the scaled row, and every other row through the sum of them all: a weight's rounding is 2^-12 of it at most
        rest = np.delete(x.astype(np.float64), 3, 0).sum(0, keepdims=True)
        for part, mine in ((x[3:4], y[3].astype(np.float64)), (rest.astype(np.float32), np.delete(y.astype(np.float64), 3, 0).sum(0))):
            want = oracle.gguf_matmul_f64(part, p, 1, k, n, scheme)[0]
            assert np.linalg.norm(mine - want) <= 2.0 ** -11 * np.linalg.norm(want)


def test_shared_tiles_need_room_for_their_pieces(oracle):
    # without room for partial results the tiles are not shared: the same numbers up to the order of the sums
    m, n, k = 1111, 4100, 4608
    _, _, full = run(Q4_0, m, [n], k, DType.F32, 5, ("rlx_gemm_big_q4_0", "shared tiles"))
    plan = planned(Q4_0, m, [n], k, DType.F32, 0)
    assert plan[1] == "whole"
    _, _, lean = run(Q4_0, m, [n], k, DType.F32, 5, plan, lean=True)
    keep = np.arange(m) != 3
    assert rel_err(lean[0][keep], full[0][keep].astype(np.float64)) <= 1e-5


@pytest.mark.parametrize("n,offset", [(6141, 0), (6142, 4), (6143, 8), (6144, 12)])
def test_rows_of_any_length_and_alignment(oracle, n, offset):
    """Whole tiles that end one, two and three columns past a store of four, and outputs that start at any word."""
    m, k = 700, 2048
    x, packs, (y,) = run(Q4_0, m, [n], k, DType.F32, n, ("rlx_gemm_big_q4_0", "whole"), offset=offset)
    rows = [0, 1, 127, 128, 255, 256, m - 1]
    assert rel_err(y[rows], oracle.gguf_matmul_f64(x[rows], packs[0], len(rows), k, n, Q4_0)) <= TOL
    assert np.all(np.isfinite(y))


@pytest.mark.parametrize("m,k,n,plan", [
    (8192, 512, 3900, ("rlx_gemm_img_f16w", "whole")),         # short K
    (8000, 2304, 4001, ("rlx_gemm_img_f16w", "whole")),        # the last K of the eight-wave kernel
    (8000, 2336, 4001, ("rlx_gemm_big_f16w", "whole")),        # the first K of the four-wave kernel, ragged
    (4000, 4096, 2500, ("rlx_gemm_big_f16w", "whole")),        # a single round of whole tiles
    (2050, 6016, 7500, ("rlx_gemm_big_f16w", "shared tiles")),  # pieces of tiles, a K offset into the ready images
])
def test_code_images_of_many_rows(oracle, m, k, n, plan):
    from rlx_amd import Graph, Op, Session, Shape
    assert planned(Q8_0, m, [n], k, DType.I8) == plan
    rng = np.random.default_rng(k)
    x = rng.standard_normal((m, k)).astype(np.float32)
    packed = tiled_packed(Q8_0, n, k, 7, 0.02).reshape(-1)
    g = Graph.new("chain")
    w = g.param("w", Shape.new([len(packed)], DType.U8))
    q = g.fake_quantize(g.input("x", Shape.new([m, k], DType.F32)), 8, 1)
    g.set_outputs([g.add_node(Op.DequantMatMul(QuantScheme.GgufQ8_0), [q, w], Shape.new([m, n], DType.F32))])
    c = Session.new().compile(g)
    c.set_param_typed("w", packed, DType.U8)
    got = np.asarray(c.run([("x", x)])[0]).reshape(m, n)
    s = np.maximum(np.abs(x).max(0) / np.float32(127), np.float32(1e-12)).astype(np.float32)
    xq = np.clip(np.round(x / s), -127, 127).astype(np.float32) * s
    rows = [0, 1, 255, 256, m // 2, m - 1]
    assert rel_err(got[rows], oracle.gguf_matmul_f64(xq[rows], packed, len(rows), k, n, Q8_0)) <= TOL
