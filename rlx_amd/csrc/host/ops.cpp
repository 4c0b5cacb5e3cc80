// Operator-level entry points: packed weights in HBM, dequant, matmul dispatch, FakeQuantize.
#include <algorithm>
#include <cstdlib>
#include <cstring>
#include <vector>

#include "common.hpp"

#include <new>

namespace rlx {
int repack_host(int scheme, uint32_t flags, const uint8_t *src, size_t nbytes, int64_t n, int64_t k, uint8_t *out);
}

struct rlx_qweight {
    int scheme;
    rlx::Layout layout;    // device layout it was repacked into
    rlx::WeightDims dims;  // of one [n, k] matrix
    uint8_t *dev;
    bool owns;
    int experts;           // matrices stacked dims.bytes apart (1 for a plain weight)
    uint32_t flags;        // rlx_qweight_flags it was created with
    int sc_off() const { return (flags & RLX_QW_Q6K_SIGNED_SCALES) ? 128 : 0; }
};

namespace rlx {

// Kernel argument blocks: must match the structs in kernels/*.hip field for field.
struct DequantArgs {
    const uint8_t *w;
    float *out;
    long long n, k, units;
    int sc_off;
};
constexpr int GEMV_MAX_SEG = 8;
struct GemvSeg {
    const uint8_t *w;
    const void *x;
    float *out;
    int n, k, row_tiles, units, wg_begin, tiles_per_wg, tile_stride;
    const uint8_t *w_pair;
};
struct GemvArgs {
    GemvSeg seg[GEMV_MAX_SEG];
    int nseg, m, kc_units, x_dtype, max_tiles_per_wg;
    const float *expert_idx;
    long long slab_bytes;
    int num_experts;
    unsigned long long *argmax_key;
    const float *gamma;
    const float *beta;
    float eps;
    int lds_bytes;
    int kw;
    int sc_off;
    int tw, slices;
    uint32_t kw_div, tw_div, slices_div, m_div;
};
struct RmsNorm {  // RMSNorm prologue of a decode launch (f32 activations only)
    const float *gamma, *beta;
    float eps;
};
struct FqArgs {
    const float *x;
    float *out;
    int8_t *codes;
    uint32_t *max_bits;
    float *scale;
    float *state;
    long long len, chan_dim, inner;
    float q_max, decay;
    int scale_mode, round_mode, rows_per_block;
    float *partial;
    int parts;
    void *img;
    float *rowfac;
    int k_pad, m_rows, write_out;
    float *colscale;
    uint32_t *smax_bits;
};
struct WScaleArgs {  // mirrors kernels/dequant.hip
    const uint8_t *w;
    void *wimg;
    const float *cs;
    const float *rowfac;
    long long row_tiles, units;
    int k_pad, sc_off;
};

constexpr int GEMM_MAX_SEG = 4;
struct GemmSeg {
    const uint8_t *w;
    float *out;
    int n, row_tiles, tile_begin;
};
struct GemmArgs {
    GemmSeg seg[GEMM_MAX_SEG];
    int nseg;
    const void *xh;
    const void *sxh;
    int m_rows, m_out, k_pad, units, pair_rows, steps_per_split, split_out, sc_off;
    const float *rowfac;
    const int *tile_expert;
    const int *perm;
    long long slab_bytes;
};
struct GemmBigSeg {  // mirrors kernels/gemm_big.hip
    const void *w;
    float *out;
    int n, row_tiles, tile_begin;
};
struct GemmBigArgs {
    GemmBigSeg seg[GEMM_MAX_SEG];
    int nseg;
    const void *a_img;
    const float *rowfac;
    float *part;
    int m_out, tiles_m, tiles_n, a_steps, quads, pair_rows;
};
struct GemmImgArgs {  // mirrors kernels/gemm.hip
    const void *a_img;
    const void *b_img;
    float *out;
    const float *rowfac;
    int m_out, n, steps;
};
constexpr int GEMVW_MAX_SEG = 8;
struct GemvWSeg {  // mirrors kernels/gemv_wide.hip
    const void *w;
    float *out;
    int n, row_tiles, wg_begin, k_slices, slice_units;
};
struct GemvWArgs {
    GemvWSeg seg[GEMVW_MAX_SEG];
    int nseg, m, pair_rows, units, k_steps;
    const void *xh;
    const float *rowfac;
    const int *tile_expert;
    const int *perm;
    long long slab_bytes;
};
struct SplitReduceArgs {  // mirrors kernels/gemm.hip
    const float *part[8];
    float *out[8];
    long long elems[8];
    int split[8];
};
// One launch adds the K slices of up to eight matrices (ascending K, fixed order) into their outputs.
static int launch_split_reduce(const SplitReduceArgs &ra, int nseg, hipStream_t stream) {
    if (nseg == 0) return RLX_OK;
    long long most = 0;
    for (int i = 0; i < nseg; i++) most = std::max(most, (ra.elems[i] + 3) / 4);
    SplitReduceArgs a = ra;
    void *rparams[] = {&a};
    return launch3(K_SPLITK_REDUCE, (unsigned)std::min<long long>((most + 255) / 256, 2048), (unsigned)nseg, 1, 256, 0, stream, rparams);
}
struct XPrepArgs {
    const void *x;
    void *xh;
    void *sxh;
    int m, k, k_pad, m_rows, x_dtype;
    float *rowfac;
    const int *perm;
    int perm_len;
    int row_group, subs_log2;
    int sums16;
};
constexpr int MOE_MAX_EXPERTS = 256;
struct MoeSortArgs {  // mirrors kernels/moe.hip
    const float *expert_idx;
    int m, num_experts, group_rows, perm_len;
    int *perm;
    int *tile_expert;
};

// Kinds of activation operand: 0 f32, 1 bf16, 2 f16 tensors; XK_CODES: the workspace image a FakeQuantize left
// (rlx_mi355x_fake_quantize_image: integer codes as binary16 plus the column scales), named RLX_I8 at the boundary.
constexpr int XK_CODES = 3;
static bool code_image_scheme(int scheme) { return scheme == SCHEME_Q4_0 || scheme == SCHEME_Q8_0; }
static int x_kind(int x_dtype) {
    switch (x_dtype) {
    case RLX_F32: return 0;
    case RLX_BF16: return 1;
    case RLX_F16: return 2;
    default: return -1;
    }
}

// One decode launch over `count` (<= GEMV_MAX_SEG) matmuls of one scheme, batch and activation dtype; each has
// its own activations, K and N.
// Rows one launch of the decode kernels takes: two groups of 16 MFMA rows, an f32 row being a hi and a lo row. Above
// that the prefill GEMM runs (measured on a 70B layer at 32 bf16 rows: 205 us against 317).
static int64_t decode_rows(int xk) { return xk == 0 ? 16 : 32; }

constexpr int ARGMAX_MAX_WGS = 4096;  // keys in the tied-LM-head scratch: one per workgroup of the decode launch

// div_by() of kernels/gemv.hip
static uint32_t div_magic(uint32_t d) { return d <= 1 ? 0u : (uint32_t)(((1ull << 32) + d - 1) / d); }

struct GemvLaunch {
    KernelId kernel;
    GemvArgs a;
    int wgs, waves;
    size_t lds;
};
static int plan_gemv(const void *const *xs, int xk, const rlx_qweight *const *ws, float *const *outs, int count, int m, const float *expert_idx,
                     unsigned long long *argmax_key, const rlx_qweight *const *pairs, const RmsNorm *norm, GemvLaunch &out) {
    const int scheme = ws[0]->scheme;
    const Layout L = ws[0]->layout;
    for (int i = 0; i < count; i++) {
        if ((uintptr_t)xs[i] % 16 != 0) {
            set_error("gguf_matmul_bt: activations must be 16-byte aligned");
            return RLX_ERR_INVALID;
        }
        if (ws[i]->sc_off() != ws[0]->sc_off() || (pairs && pairs[i]->sc_off() != ws[0]->sc_off())) {
            set_error("gguf_matmul_bt: the Q6_K weights of one launch must share one reading of their scale bytes");
            return RLX_ERR_INVALID;
        }
    }
    const int rv = xk == 0 ? 2 * m : m;
    const int ng = (rv + 3) / 4;
    const bool r2 = rv <= 2;
    // groups of 16 activation rows per weight fragment: 1 (the decode kernels) or 2 (plain epilogue only)
    const int rg = rv <= 16 ? 1 : 2;
    if (rv > 32 || (rg > 1 && (argmax_key || pairs || norm || expert_idx))) {
        set_error("gemv: %d activation rows are beyond this kernel", rv);
        return RLX_ERR_UNSUPPORTED;
    }
    // kernel = scheme family x {r2, r4, r2_argmax, r2_paired, r4_paired}
    const int family = scheme == SCHEME_Q4_0 ? K_GEMV_Q4_0_R2 : scheme == SCHEME_Q8_0 ? K_GEMV_Q8_0_R2
                       : scheme == SCHEME_Q6K ? K_GEMV_Q6_K_R2 : scheme == SCHEME_Q5K ? K_GEMV_Q5_K_R2
                       : scheme == SCHEME_Q8K ? K_GEMV_Q8_K_R2 : scheme == SCHEME_Q2K ? K_GEMV_Q2_K_R2 : K_GEMV_Q4_K_R2;
    if (argmax_key && !r2) {
        set_error("gemv: the argmax epilogue takes one activation row");
        return RLX_ERR_INVALID;
    }
    if (norm && xk != 0) {
        set_error("gemv: the RMSNorm prologue takes f32 activations");
        return RLX_ERR_UNSUPPORTED;
    }
    const int variant = argmax_key ? (norm ? 9 : 2) : pairs ? (norm ? (r2 ? 7 : 8) : (r2 ? 3 : 4)) : (norm ? (r2 ? 5 : 6) : (r2 ? 0 : 1));
    KernelId id = (KernelId)(family + variant);
    if (rg > 1) id = (KernelId)(K_GEMV_Q4_0_G2 + (family - K_GEMV_Q4_0_R2) / 10);
    static const int env_waves = getenv("RLX_GEMV_WAVES") ? atoi(getenv("RLX_GEMV_WAVES")) : 8;
    static const int env_wgs_per_cu = getenv("RLX_GEMV_WGS_PER_CU") ? atoi(getenv("RLX_GEMV_WGS_PER_CU")) : 2;
    int max_units = 0;
    long long work = 0;  // (tile, unit) items in the launch
    for (int i = 0; i < count; i++) {
        max_units = std::max(max_units, (int)ws[i]->dims.units);
        work += ws[i]->dims.row_tiles * ws[i]->dims.units * (pairs ? 2 : 1);
    }
    // Segments with the longest K last (equal K keeps the caller's order, which the expert routing relies on: segment s
    // is token s). Measured on the seven projections of a layer: 5185 GB/s with the 14336-wide down projection at the
    // end of the workgroup order, 5050 with it at the front, whatever the order of the others.
    int order[GEMV_MAX_SEG];
    for (int i = 0; i < count; i++) order[i] = i;
    std::stable_sort(order, order + count, [&](int a, int b) { return ws[a]->dims.units < ws[b]->dims.units; });
    const int cus = device_props().cu_count > 0 ? device_props().cu_count : 256;  // (none opened: a plan query)
    const size_t slot_bytes = (size_t)ng * 256;
    auto stage_bytes = [&](int kcu) {
        size_t b = ((size_t)rv * ((size_t)kcu * L.unit_k + 8) * 2 + 15) & ~(size_t)15;
        if (r2 && (scheme == SCHEME_Q4K || scheme == SCHEME_Q5K)) b += (size_t)kcu * (L.unit_k / 32) * 16 * 4;  // block sums
        return b;
    };
    // Two K units per loop item halve the per-item bookkeeping; every chunk of every segment must then hold an even number of units, and
    // every wave still needs an item.
    static const bool env_u1 = getenv("RLX_GEMV_UPI") && atoi(getenv("RLX_GEMV_UPI")) == 1;
    auto two_units = [&](int nwaves) {
        bool ok = family == K_GEMV_Q4_0_R2 && rg == 1 && !env_u1 && nwaves * 2 <= max_units;
        for (int i = 0; i < count; i++) ok = ok && ws[i]->dims.units % 2 == 0;
        return ok;
    };
    // A launch shape: `wgs_per_cu` workgroups of `waves` waves per CU, every one resident at once, each with the same
    // number of (tile, unit) items (a segment with a longer K gets fewer row tiles per workgroup), LDS split between
    // the per-(tile, wave) partial sums and the staged activation chunk (rv rows of halfs, 16 B row padding, with one
    // row plus the Q4_K / Q5_K block sums).
    struct Shape {
        GemvArgs a;
        int nwaves, wg, kcu;
        size_t lds;
        bool fits;
    };
    auto shape = [&](int waves, int wgs_per_cu, size_t budget, int kw_req) {
        Shape sh{};
        sh.nwaves = std::max(1, std::min(std::min(16, std::max(1, waves)), max_units));
        // kw waves share a tile (its K units alternate between them), nwaves / kw tiles run side by side
        const int kw = (kw_req > 0 && kw_req < sh.nwaves && sh.nwaves % kw_req == 0) ? kw_req : sh.nwaves;
        const int tw = sh.nwaves / kw;
        const long long slots = (long long)std::max(1, wgs_per_cu) * cus;
        // share of the LDS for the partial sums; the rest stages activations
        const size_t part_budget = tw > 1 ? budget / 2 : budget * 2 / 5;
        const int tpw_cap = (int)std::max<size_t>(1, part_budget / (kw * slot_bytes));
        int max_tpw = 1;
        // With tw > 1 a workgroup's tile count is rounded up to whole rounds of tw tiles; the per-workgroup target then
        // grows until one round of workgroups covers the launch (a few stragglers in a second round would double it).
        for (double grow = 1.0;; grow += 0.04) {
            const long long target_items = std::max<long long>(1, (long long)((double)((work + slots - 1) / slots) * grow));
            sh.wg = 0;
            max_tpw = 1;
            for (int oi = 0; oi < count; oi++) {
                const int i = order[oi];
                const WeightDims &D = ws[i]->dims;
                const int per_tile = pairs ? 2 : 1;  // partial-sum slots and K runs per row tile
                int tpw = (int)std::max<long long>(1, (target_items + D.units * per_tile / 2) / (D.units * per_tile));
                tpw = std::min((tpw + tw - 1) / tw * tw, std::max(1, tpw_cap / per_tile / tw * tw));
                tpw = std::max(tpw, 1);
                max_tpw = std::max(max_tpw, tpw * per_tile);
                const int seg_wgs = (int)((D.row_tiles + tpw - 1) / tpw);
                static const bool contiguous = getenv("RLX_GEMV_CONTIGUOUS") != nullptr;
                sh.a.seg[oi] = GemvSeg{ws[i]->dev, xs[i], outs[i], (int)D.n, (int)D.k, (int)D.row_tiles, (int)D.units, sh.wg, tpw,
                                      contiguous ? 1 : seg_wgs, pairs ? pairs[i]->dev : nullptr};
                sh.wg += seg_wgs;
            }
            if (tw == 1 || sh.wg <= slots || grow > 2.0) break;
        }
        const size_t part_bytes = (size_t)max_tpw * kw * slot_bytes;
        sh.kcu = max_units;
        // the last LDS_TAIL bytes: the per-row factors of the binary16 range prescale and its bookkeeping, the sums of squares of
        // the RMSNorm prologue (GEMV_LDS_TAIL in kernels/gemv.hip)
        constexpr size_t LDS_TAIL = 384;
        while (sh.kcu > 1 && part_bytes + stage_bytes(sh.kcu) + LDS_TAIL > budget) sh.kcu--;
        // A chunk of 17 units leaves fifteen of sixteen waves waiting for one, chunk after chunk: it is cut to whole rounds of a tile's waves
        // (of their two-unit items, or at least of units) where that takes at most a fifth of it and no chunk more, or a sixteenth and
        // at most a quarter more chunks. 2650 launches of more than one chunk (six schemes, twenty matrices of 7168 - 28672 columns,
        // 1 - 16 f32 and 1 - 32 bf16 rows): 1150 change, 1.04 times as fast on average, 0.967 at worst, 1.25 at best; cut wherever that
        // takes more chunks, 0.96 on average and 0.74 at worst. us, as many as fit / cut: [4096, 14336] Q4_0, 8 f32 rows, 34 -> 32
        // units 22.2 / 20.3; 5 rows, 57 -> 48, a third chunk, 15.0 / 16.2; [8192, 28672] Q4_0, 16 rows, 17 -> 16 91 / 79.
        if (sh.kcu < max_units) {
            auto chunks = [&](int kcu) {
                int c = 0;
                for (int i = 0; i < count; i++) c += ((int)ws[i]->dims.units + kcu - 1) / kcu;
                return c;
            };
            for (int step : {two_units(sh.nwaves) ? 2 * kw : kw, kw}) {
                const int cut = sh.kcu % step;
                if (cut == sh.kcu) continue;
                const int now = chunks(sh.kcu), more = chunks(sh.kcu - cut) - now;
                if (cut * (more > 0 ? 16 : 5) > sh.kcu || more * 4 > now) continue;
                sh.kcu -= cut;
                break;
            }
        }
        sh.fits = part_bytes + stage_bytes(sh.kcu) + LDS_TAIL <= budget;
        sh.lds = part_bytes + stage_bytes(sh.kcu) + LDS_TAIL;
        sh.a.nseg = count;
        sh.a.m = m;
        sh.a.kc_units = sh.kcu;
        sh.a.x_dtype = xk;
        sh.a.max_tiles_per_wg = max_tpw;
        sh.a.expert_idx = expert_idx;
        sh.a.argmax_key = argmax_key;
        sh.a.gamma = norm ? norm->gamma : nullptr;
        sh.a.beta = norm ? norm->beta : nullptr;
        sh.a.eps = norm ? norm->eps : 0.f;
        sh.a.lds_bytes = (int)sh.lds;
        sh.a.kw = kw;
        sh.a.tw = tw;
        sh.a.slices = m >= sh.nwaves ? 1 : (sh.nwaves + m - 1) / m;
        sh.a.kw_div = div_magic((uint32_t)kw);
        sh.a.tw_div = div_magic((uint32_t)tw);
        sh.a.slices_div = div_magic((uint32_t)sh.a.slices);
        sh.a.m_div = div_magic((uint32_t)m);
        sh.a.slab_bytes = ws[0]->dims.bytes;
        sh.a.num_experts = ws[0]->experts;
        sh.a.sc_off = ws[0]->sc_off();
        return sh;
    };
    // Two workgroups of 8 waves per CU with 80 KB each: holds a 14336-wide f32 vector (hi + lo rows) in one chunk.
    Shape sh = shape(env_waves, env_wgs_per_cu, (size_t)(env_wgs_per_cu <= 1 ? 156 : 80) * 1024, 0);
    // With four or more activation rows every workgroup restages all of x, and that traffic (workgroups x rows x K)
    // rivals the weights: one workgroup of 16 waves per CU with the whole LDS halves it, provided a single round of
    // workgroups still covers the matrix.
    if (rv >= 4 && !getenv("RLX_GEMV_WGS_PER_CU")) {
        // From five rows on, the per-(tile, wave) partial-sum slots (256 B per four rows) are what limits the tiles of
        // a workgroup: two waves per tile instead of sixteen, eight tiles side by side, keeps the slot area small
        // enough that one workgroup per CU covers the launch and the activations are staged once per CU. The kernels
        // for more than 16 rows run eight waves per workgroup (their register budget), one wave per tile when the
        // launch has the tiles for it.
        static const int env_kw = getenv("RLX_GEMV_KW") ? atoi(getenv("RLX_GEMV_KW")) : -1;
        const int fat_waves = rg > 1 ? 8 : 16;
        int kw = 0;
        if (rv >= 5) {  // as many tiles side by side (at most eight) as the segment with the fewest tiles per workgroup has
            double min_tpw = 1e30;
            for (int i = 0; i < count; i++)
                min_tpw = std::min(min_tpw, (double)work / cus / (double)(ws[i]->dims.units * (pairs ? 2 : 1)));
            int tw = 8;
            while (tw > 1 && tw > min_tpw * 1.2) tw /= 2;
            kw = tw > 1 ? fat_waves / tw : 0;
        }
        if (env_kw >= 0) kw = env_kw;
        Shape fat = shape(fat_waves, 1, (size_t)156 * 1024, kw);
        if (kw && !(fat.fits && fat.wg <= cus) && rg == 1) fat = shape(fat_waves, 1, (size_t)156 * 1024, 0);
        if (fat.fits && (fat.wg <= cus || rg > 1)) sh = fat;
        else if (rg > 1) sh = shape(fat_waves, 1, (size_t)156 * 1024, 0);
    }
    if (!sh.fits) {
        set_error("gemv: one K unit of %d activation rows does not fit LDS", rv);
        return RLX_ERR_INVALID;
    }
    if (two_units(sh.nwaves) && sh.kcu % 2 == 0) id = (KernelId)(K_GEMV_Q4_0_U2_R2 + variant);
    if (argmax_key && sh.wg > ARGMAX_MAX_WGS) {
        set_error("gemv: %d workgroups are more than the argmax key scratch holds (%d)", sh.wg, ARGMAX_MAX_WGS);
        return RLX_ERR_UNSUPPORTED;
    }
    out = GemvLaunch{id, sh.a, sh.wg, sh.nwaves, sh.lds};
    return RLX_OK;
}
static int launch_gemv(const void *const *xs, int xk, const rlx_qweight *const *ws, float *const *outs, int count, int m,
                       hipStream_t stream, const float *expert_idx = nullptr, unsigned long long *argmax_key = nullptr,
                       const rlx_qweight *const *pairs = nullptr, const RmsNorm *norm = nullptr, int *wgs_out = nullptr) {
    GemvLaunch g;
    RLX_TRY(plan_gemv(xs, xk, ws, outs, count, m, expert_idx, argmax_key, pairs, norm, g));
    if (wgs_out) *wgs_out = g.wgs;
    void *params[] = {&g.a};
    return launch(g.kernel, (unsigned)g.wgs, 1, (unsigned)g.waves * 64, (unsigned)g.lds, stream, params);
}

// How K is cut across workgroups when the output tiles alone would leave most of the chip idle: `split` slices of
// `units_per_split` K units (whole groups of four 64-column steps). Each slice writes its partial result and
// rlx_splitk_reduce adds the slices in ascending K.
struct GemmSplit {
    int split, units_per_split;
};
static GemmSplit gemm_split(long long tiles_x, long long tiles_y, int64_t k_units, int steps_per_unit, bool skinny, int max_split = 1 << 30) {
    // workgroup slots to fill: one per CU for the 256-row tile (144 KB of LDS), two for the 64-row tile; sized for the
    // 256 CUs of the part when no device has been opened (planning a graph needs none)
    const int cus = device_props().cu_count > 0 ? device_props().cu_count : 256;
    const long long slots = (long long)cus * (skinny ? 2 : 1);
    int split = 1;
    if (tiles_x * tiles_y * 5 < slots * 4) split = (int)std::min<long long>(k_units, slots / (tiles_x * tiles_y));
    split = std::max(1, std::min(split, max_split));
    int units_per_split = (int)((k_units + split - 1) / split);
    const int upq = std::max(1, 4 / steps_per_unit);  // units in four steps: every slice is a multiple of that
    units_per_split = (units_per_split + upq - 1) / upq * upq;
    split = (int)((k_units + units_per_split - 1) / units_per_split);
    return GemmSplit{split, units_per_split};
}

// Workspace of a prefill matmul: [per-row factors][column scales][image of x][block sums][image of the scaled weights]
// [partial results of a split K]. The second and the fifth exist only for a FakeQuantize code image (XK_CODES), whose
// matmul runs on ready binary16 weights W * diag(s) (n is the widest matrix multiplied from the image, one at a time).
// The image may have been made for another scheme than the one that multiplies it (rlx_mi355x_gguf_matmul_prepare), and that
// scheme's matmul may follow: partial results begin past the widest block sums any scheme's image has, whatever the scheme.
struct GemmPlan {
    int64_t m_rows, k_pad;
    size_t xh_bytes, sxh_bytes, fac_bytes;  // the image, the block sums (Q4_K / Q5_K per 32 columns, Q2_K per 16), the per-row prescale factors
    size_t cs_bytes, wimg_bytes;
    size_t part_off;                        // where partial results begin
    size_t part_bytes;                      // the partial results of one launch with room for all it wants (0: it leaves none)
    int sums_kind;                          // act_sums_kind of the scheme the plan was made for
    size_t image_end() const { return fac_bytes + cs_bytes + xh_bytes + sxh_bytes; }
    size_t total() const { return part_bytes ? part_off + part_bytes : image_end() + wimg_bytes; }
};
static bool gemm_skinny(int xk, int64_t m) { return (xk == 0 ? 2 * m : m) <= 128; }
// Up to 192 image rows of Q4_0 / Q8_0 run rlx_gemvw_* (kernels/gemv_wide.hip): weights decoded in registers by the wave
// that multiplies them, 256-row blocks of W per workgroup, one pass over the weights per 64 image rows (grid.y). One 70B
// layer, us, against the 64-row / 256-row prefill tiles: 96 rows 333 against 476, 128 rows 348 against 491, 160 rows 474
// against 514, 192 rows 486 against 527; at 256 rows (four passes) 575 against 552, so the 256-row tile takes over there.
static bool gemm_wide(int scheme, int xk, int64_t m) {
    return (scheme == SCHEME_Q4_0 || scheme == SCHEME_Q8_0) && xk != XK_CODES && (xk == 0 ? 2 * m : m) <= 192;
}
// K slices of one matrix in a launch of `launch_bytes` packed bytes in all: a workgroup should get about one CU's share
// of the launch, at least 512 KB (one 70B layer at 64 rows, us: 218 with half a CU's share and 256 KB, 203 with this, 230
// with at least 1 MB); the slices' partial results (written and read once: 8 m n bytes per slice) may cost up to half
// the matrix's own bytes. Slices are whole 256-column chunks of at least four units.
static GemmSplit wide_split(const Layout &L, const WeightDims &D, int64_t m, size_t launch_bytes) {
    const int cus = device_props().cu_count > 0 ? device_props().cu_count : 256;
    const size_t target = std::max<size_t>(launch_bytes / (size_t)cus, 512u << 10);
    const size_t block_bytes = (size_t)16 * (size_t)D.units * (size_t)L.unit_bytes;
    int64_t split = (int64_t)((block_bytes + target / 2) / target);
    split = std::min<int64_t>(split, (int64_t)((size_t)D.bytes / 2 / ((size_t)8 * (size_t)m * (size_t)D.n)));
    split = std::max<int64_t>(1, std::min<int64_t>(split, D.units / 4));
    int units_per_split = (int)((D.units + split - 1) / split);
    units_per_split = (units_per_split + 1) / 2 * 2;
    return GemmSplit{(int)((D.units + units_per_split - 1) / units_per_split), units_per_split};
}
// The 256 x 256 tiles of kernels/gemm_big.hip (Q4_0, Q8_0, code images) against the 256 x 128 tiles of kernels/gemm.hip, and how the
// former are handed out: a tile per workgroup, or the whole line of (tile, 128 columns of K) items in equal runs, one per CU, with
// the pieces of shared tiles added by a launch of their own. `groups` = 0: the 256 x 128 tiles. Estimated times decide. Their constants,
// in us, are free parameters of a fit: what they are named after is what they stand for, not what it measures alone. Fitted to 1180, 1140
// and 1080 random launches of f32 rows, 16-bit rows and code images whose rows are whole groups of four columns and half as many of
// other lengths (97 - 8192 rows, K 256 - 28672, one to four matrices), each timed all three ways. On 330, 320 and 345 others of the
// former kind, which the fit has not seen, the whole call takes 1.001, 1.003 and 1.003 times the fastest of the three ways on
// average (1.05, 1.11 and 1.11 at worst) and is 1.02, 1.01 and 1.04 times as fast as with the smaller tiles alone; on 167, 162 and 136 of
// the latter 1.002, 1.001 and 1.009 (1.06, 1.08, 1.38) and 1.02, 1.08, 1.08. Some, smaller / whole / shared: f32 [528, 6944] x 3426
// 107 / 188 / 101, [1111, 4096] x 28672 551 / 519 / 529, [417, 256] x 288 14.6 / 23.4 / -; bf16 [1424, 8416] x 2794 129 / 224 / 121; codes
// [3763, 6432] x 2598 212 / 163 / 219, [3138, 6720] x 5014 323 / 301 / 246.
// Shared tiles of one row of A are at the same K at the same time, and read A together, where their workgroups, 256 / tiles_n apart, are
// a whole number apart: gcd(tiles_n, 256) at a time. Alone, each reads A by itself: the kernel on code images of 22 x 12 tiles of 6912
// columns 212 us, of 24 x 11 tiles 305. Packed weights, whose bytes are a quarter or half, feel it less.
struct BigPlan {
    int groups;
    size_t part_bytes;
};
struct BigCosts {
    double half_start, half_quad;      // a round of 256 x 128 tiles: start, every 128 columns
    double half_idle;                  // share of it that a last round takes however few its tiles are
    double split_start, split_byte;    // a split of K on top: its reduce launch, its partial results per byte
    double whole_start, whole_quad;    // a round of whole 256 x 256 tiles
    double shared_start, shared_quad;  // shared tiles: the pieces, written and added by the reduce launch; every 128 columns of a run
                                       // (whose tiles each take whole_start, too)
    double alone, pairs;               // added share of the latter where A is read by one workgroup or two at a time
    double sparse_margin;              // shared tiles against a grid that is not full: the estimate's error there
    double half_word;                  // a result that the 256 x 128 tiles store as a single word (rows that are no multiple of four long)
};
constexpr BigCosts BIG_COSTS_F32{0, 1.64, 0.96, 4.91, 0, 4.09, 2.929, 28.2, 2.838, 0.024, 0.016, 0.917, 8.7e-7};
constexpr BigCosts BIG_COSTS_16{0.8, 1.83, 0.85, 4.17, 3e-7, 6.17, 3.143, 53, 3.022, 0.073, 0.042, 0.99, 1.35e-6};
constexpr BigCosts BIG_COSTS_CODES{3.8, 1.485, 0.737, 5.13, 1.7e-7, 9.54, 1.815, 36.6, 2.056, 0.8, 0.21, 0.943, 1.25e-6};
constexpr double IMG_START = 4.31, IMG_QUAD = 2.49;  // a round of rlx_gemm_img_f16w, every 128 columns of it
// up to here rlx_gemm_img_f16w instead of rlx_gemm_big_f16w: its way in and out of a tile is shorter (kernels/gemm.hip)
constexpr int64_t IMG_MAX_K = 2304;
static BigPlan big_plan(int scheme, int xk, int64_t m, int64_t m_rows, int64_t tiles_n, int64_t half_tiles_n, int64_t n_sum, int64_t n_words, int64_t quads,
                        const GemmSplit &sp, int64_t slice_quads, size_t part_room) {
    BigPlan none{0, 0};
    if (scheme != SCHEME_Q4_0 && scheme != SCHEME_Q8_0) return none;
    const bool codes = xk == XK_CODES;
    const BigCosts &c = codes ? BIG_COSTS_CODES : xk == 0 ? BIG_COSTS_F32 : BIG_COSTS_16;
    const long long cus = device_props().cu_count > 0 ? device_props().cu_count : 256;
    const long long tiles_m = m_rows / 256, tiles = tiles_m * tiles_n, half = tiles_m * half_tiles_n;
    auto rounds = [&](long long t) { return (t + cus - 1) / cus; };
    // code images run whole tiles from two rounds on in any case ([8192, 4096] x [4096, 4096] 310 -> 282 us; half tiles 14 % slower at K = 1024)
    if (codes && tiles >= 2 * cus) return BigPlan{(int)tiles, 0};
    const bool sparse = half * 5 < cus * 4;  // where gemm_split cuts K if two slices or more find a CU each
    double t_half;
    if (sp.split > 1) {
        t_half = c.half_start + (double)slice_quads * c.half_quad + c.split_start + c.split_byte * 4.0 * (double)sp.split * (double)m * (double)n_sum;
    } else {
        const double last = (double)(half - cus * (rounds(half) - 1)) / (double)cus;
        t_half = ((double)(rounds(half) - 1) + c.half_idle + (1 - c.half_idle) * last) * (c.half_start + (double)quads * c.half_quad) +
                 c.half_word * (double)m * (double)n_words;
    }
    const double t_whole = (double)rounds(tiles) * (codes && quads * 128 <= IMG_MAX_K ? IMG_START + (double)quads * IMG_QUAD : c.whole_start + (double)quads * c.whole_quad);
    const bool whole = t_whole < t_half;
    const size_t part = (size_t)cus * 2 * (size_t)(xk == 0 ? 128 : 256) * 1024;  // a workgroup leaves at most two pieces
    if (part <= part_room && tiles * quads >= cus) {
        const double quad = c.shared_quad * (1 + (tiles_n % 2 ? c.alone : tiles_n % 4 ? c.pairs : 0));
        const double margin = sparse ? c.sparse_margin : 1;
        const double t_shared = c.shared_start + (double)tiles / (double)cus * c.whole_start + (double)rounds(tiles * quads) * quad;
        if (t_shared < margin * (whole ? t_whole : t_half)) return BigPlan{(int)cus, part};
    }
    return whole ? BigPlan{(int)tiles, 0} : none;
}

// How the launch over `count` matrices [ns[i], k] of one scheme that multiply the same x is carried out, decided here for the launch
// itself, the workspace queries, the graph planner and the plan query. `part_room`: bytes there are for partial results.
struct GemmLaunch {
    KernelId kernel;
    int groups;                      // rlx_gemm_big_* / rlx_gemm_img_*: workgroups
    bool shared;                     // rlx_gemm_big_*: tiles shared between workgroups, pieces added by rlx_gemm_big_reduce
    GemmSplit split[GEMVW_MAX_SEG];  // the other kernels: K slices, of every matrix (rlx_gemvw_*) or, in [0], of all of them
    size_t part_bytes;               // partial results it leaves
};
static GemmLaunch launch_plan(int scheme, int xk, int64_t m, int64_t k, const int64_t *ns, int count, size_t part_room) {
    scheme = kernel_scheme(scheme);
    const bool codes = xk == XK_CODES, skinny = gemm_skinny(xk, m);
    const Layout L = codes ? Layout{64, 0, 0, 0, 0} : layout_of(scheme);
    const int64_t rv = xk == 0 ? 2 * m : m, m_rows = (rv + 255) / 256 * 256, k_pad = (k + 255) / 256 * 256;
    int64_t n_sum = 0, n_words = 0, tiles_n = 0, half_tiles_n = 0;
    for (int i = 0; i < count; i++) {
        n_sum += ns[i];
        n_words += ns[i] % 4 ? ns[i] : 0;
        tiles_n += (ns[i] + 255) / 256;
        half_tiles_n += (ns[i] + 127) / 128;
    }
    GemmLaunch g{};
    if (gemm_wide(scheme, xk, m)) {
        g.kernel = scheme == SCHEME_Q4_0 ? K_GEMVW_Q4_0 : K_GEMVW_Q8_0;
        // every 64 image rows are a pass of their own over the weights (a second one finds part of them in L2)
        size_t launch_bytes = 0;
        for (int i = 0; i < count; i++) launch_bytes += (size_t)weight_dims(L, ns[i], k).bytes * (size_t)((rv + 63) / 64);
        for (int i = 0; i < count; i++) {
            g.split[i] = wide_split(L, weight_dims(L, ns[i], k), m, launch_bytes);
            if (g.split[i].split > 1) g.part_bytes += (size_t)g.split[i].split * (size_t)m * (size_t)ns[i] * 4;
        }
        if (g.part_bytes > part_room) {  // a workspace without room for the slices: every matrix in one piece
            for (int i = 0; i < count; i++) g.split[i] = GemmSplit{1, (int)((weight_dims(L, ns[i], k).units + 1) / 2 * 2)};
            g.part_bytes = 0;
        }
        return g;
    }
    if (!skinny) {
        const int64_t quads = codes ? k_pad / 128 : (k + L.unit_k - 1) / L.unit_k;
        // the 256 x 128 tiles' slices of K, were there room for all of them
        const GemmSplit sp = gemm_split(half_tiles_n, m_rows / 256, codes ? k_pad / 64 : quads, L.unit_k / 64, false);
        const int64_t slice_quads = std::min<int64_t>(quads, (int64_t)sp.units_per_split * L.unit_k / 128);
        const BigPlan bp = big_plan(scheme, xk, m, m_rows, tiles_n, half_tiles_n, n_sum, n_words, quads, sp, slice_quads, part_room);
        if (bp.groups) {
            g.shared = bp.part_bytes > 0;
            g.groups = bp.groups;
            g.part_bytes = bp.part_bytes;
            g.kernel = !codes                            ? (scheme == SCHEME_Q4_0 ? K_GEMM_BIG_Q4_0 : K_GEMM_BIG_Q8_0)
                       : !g.shared && k_pad <= IMG_MAX_K ? K_GEMM_IMG_F16W
                                                         : K_GEMM_BIG_F16W;
            return g;
        }
    }
    // Up to 128 image rows run the 64-row tile (the weights are decoded once per 64 rows, but nothing is spent on padding rows); beyond
    // that the 256-row tile.
    g.kernel = codes                     ? (skinny ? K_GEMM64_F16W : K_GEMM_F16W)
               : scheme == SCHEME_Q4K    ? (skinny ? K_GEMM64_Q4_K : K_GEMM_Q4_K)
               : scheme == SCHEME_Q4_0   ? (skinny ? K_GEMM64_Q4_0 : K_GEMM_Q4_0)
               : scheme == SCHEME_Q6K    ? (skinny ? K_GEMM64_Q6_K : K_GEMM_Q6_K)
               : scheme == SCHEME_Q5K    ? (skinny ? K_GEMM64_Q5_K : K_GEMM_Q5_K)
               : scheme == SCHEME_Q8K    ? (skinny ? K_GEMM64_Q8_K : K_GEMM_Q8_K)
               : scheme == SCHEME_Q2K    ? (skinny ? K_GEMM64_Q2_K : K_GEMM_Q2_K)
                                         : (skinny ? K_GEMM64_Q8_0 : K_GEMM_Q8_0);
    // A workspace sized for fewer slices gets fewer.
    const int64_t k_units = codes ? k_pad / 64 : (k + L.unit_k - 1) / L.unit_k;  // K units of the operand the kernel reads
    const int steps_per_unit = L.unit_k / 64;
    const int64_t gy = skinny ? (rv + 63) / 64 : m_rows / 256;
    const size_t slice_bytes = (size_t)m * (size_t)n_sum * 4;
    GemmSplit sp = gemm_split(half_tiles_n, gy, k_units, steps_per_unit, skinny);
    if (sp.split > 1 && (size_t)sp.split * slice_bytes > part_room)
        sp = gemm_split(half_tiles_n, gy, k_units, steps_per_unit, skinny, (int)std::max<size_t>(1, part_room / slice_bytes));
    if (sp.split > 1 && (size_t)sp.split * slice_bytes > part_room) sp = gemm_split(half_tiles_n, gy, k_units, steps_per_unit, skinny, 1);
    g.split[0] = sp;
    if (sp.split > 1) g.part_bytes = (size_t)sp.split * slice_bytes;
    return g;
}
// Operands of a prefill matmul and, with `count` matrices in one launch, its partial results.
static GemmPlan gemm_plan(int scheme, int xk, int64_t m, int64_t k, const int64_t *ns = nullptr, int count = 0) {
    GemmPlan p;
    const int64_t rv = xk == 0 ? 2 * m : m;
    p.m_rows = (rv + 255) / 256 * 256;
    p.k_pad = (k + 255) / 256 * 256;
    p.xh_bytes = ((size_t)p.m_rows * p.k_pad * 2 + 255) & ~(size_t)255;
    p.sums_kind = xk == XK_CODES ? 0 : act_sums_kind(scheme);
    p.sxh_bytes = (size_t)p.m_rows * (p.k_pad / 256) * 32 * p.sums_kind;  // 16 or 32 halfs per row and super-block
    p.fac_bytes = ((size_t)m * 8 + 255) & ~(size_t)255;
    p.cs_bytes = xk == XK_CODES ? (size_t)p.k_pad * 4 : 0;
    int64_t widest = 0;
    for (int i = 0; i < count; i++) widest = std::max(widest, ns[i]);
    p.wimg_bytes = xk == XK_CODES ? (size_t)((widest + 255) / 256 * 256) * p.k_pad * 2 : 0;  // whole 256-row tiles of the large-m kernels
    p.part_off = xk == XK_CODES ? p.image_end() + p.wimg_bytes
                                : p.fac_bytes + p.xh_bytes + (size_t)p.m_rows * (p.k_pad / 256) * 32 * ACT_SUMS_KIND_MAX;
    p.part_bytes = count > 0 ? launch_plan(scheme, xk, m, k, ns, count, SIZE_MAX).part_bytes : 0;
    return p;
}
// Matrices on one x that one prefill launch takes
static int prefill_launch_max(int scheme, int xk, int64_t m) {
    return xk == XK_CODES ? 1 : gemm_wide(kernel_scheme(scheme), xk, m) ? GEMVW_MAX_SEG : GEMM_MAX_SEG;
}

// The conversion of x [m, k] into the workspace: one look at every row for its prescale factor (none for binary16: a launch of
// 5 us less), then the image.
// With `perm` the image's row i is row perm[i] of x (tokens sorted by expert, padding rows -1), m still counting the rows of x.
static int launch_xprep(const void *x, int xk, int64_t m, int64_t k, const GemmPlan &p, void *workspace, hipStream_t stream,
                        const int *perm = nullptr, int perm_len = 0) {
    float *fac = (float *)workspace;
    void *xh = (uint8_t *)workspace + p.fac_bytes;
    void *sxh = p.sxh_bytes ? (uint8_t *)workspace + p.fac_bytes + p.cs_bytes + p.xh_bytes : nullptr;
    // Up to 128 image rows every kernel that reads the image does so 64 rows at a pass (rlx_gemvw_*, rlx_gemm64_*): the rest of the
    // 256-row tile is not written. 64 bf16 rows of 28672: 7.1 -> 5.0 us.
    const int64_t rv = xk == 0 ? 2 * m : m;
    const int subs_log2 = perm || rv > 128 ? 3 : rv > 64 ? 2 : 1;
    // A workgroup per row of the scan where a row is two or more memory latencies long for a wave (8 KB each) and one wave per row would
    // leave CUs short of waves: 1111 f32 rows of 14336 15.5 -> 13.1 us; on 1500 bf16 rows of 2048 it would lose 1 us.
    const int row_group = m < 2048 && k * (xk == 0 ? 4 : 2) >= 16384;
    XPrepArgs xa{x, xh, sxh, (int)m, (int)k, (int)p.k_pad, (int)p.m_rows, xk, fac, perm, perm_len, row_group, subs_log2, p.sums_kind == 2};
    void *xparams[] = {&xa};
    if (xk != 2) RLX_TRY(launch(K_XROWSCALE, (unsigned)(row_group ? m : (m + 3) / 4), 1, 256, 0, stream, xparams));
    const long long xblocks = (p.m_rows / 256) * (p.k_pad / 64) << subs_log2;  // (tile, step, 32-row sub-tile)
    return launch(K_XPREP, (unsigned)xblocks, 1, 256, 0, stream, xparams);
}

// Prefill path: convert the activations once (xprep), then the MFMA GEMM over `count` (<= GEMM_MAX_SEG) matrices of one
// scheme and K that multiply the same x (q, k, v or gate, up of a layer): one launch, their tiles side by side, so
// a small matrix fills the chip together with its neighbours instead of being cut into slivers of K on its own.
// K is split across workgroups (slices written to the workspace, added in ascending K by one reduce launch) only when
// the tile grid alone would leave most CUs idle. Q4_0 / Q8_0 up to 192 image rows go to the register-decode kernel instead.
// `prepared`: the workspace already holds this x (same pointer, k, m, dtype, and the block sums if this scheme needs
// them) from the previous launch of a batch on the same stream, so the conversion pass is skipped.
static int launch_gemm(const void *x, int xk, const rlx_qweight *const *ws, float *const *outs, int count, int64_t m,
                       void *workspace, size_t workspace_bytes, hipStream_t stream, bool prepared = false) {
    if (count < 1 || count > prefill_launch_max(ws[0]->scheme, xk, m)) {
        set_error("gguf_matmul_bt: %d matrices in one prefill launch", count);
        return RLX_ERR_INVALID;
    }
    const rlx_qweight *w = ws[0];
    const bool codes = xk == XK_CODES;  // the workspace holds a FakeQuantize code image; the weights are scaled into it first
    const Layout L = codes ? Layout{64, 0, 0, 0, 0} : w->layout;
    int64_t ns[GEMVW_MAX_SEG];
    for (int i = 0; i < count; i++) ns[i] = ws[i]->dims.n;
    const GemmPlan p = gemm_plan(w->scheme, xk, m, w->dims.k, ns, codes ? 1 : 0);  // the operands; partial results are fitted below
    for (int i = 1; i < count; i++)
        if (ws[i]->scheme != w->scheme || ws[i]->dims.k != w->dims.k || ws[i]->dims.units != w->dims.units ||
            ws[i]->layout.unit_bytes != L.unit_bytes || ws[i]->sc_off() != w->sc_off()) {
            set_error("gguf_matmul_bt: matrices of one prefill launch differ in scheme or K");
            return RLX_ERR_INVALID;
        }
    const size_t ops_end = p.image_end() + p.wimg_bytes;  // the operands
    if (!workspace || workspace_bytes < ops_end) {
        set_error("gguf_matmul_bt: m=%lld needs a %zu-byte workspace, got %zu", (long long)m, ops_end, workspace_bytes);
        return RLX_ERR_INVALID;
    }
    if ((uintptr_t)workspace % 16 != 0 || (uintptr_t)x % 16 != 0) {
        set_error("gguf_matmul_bt: activations and workspace must be 16-byte aligned");
        return RLX_ERR_INVALID;
    }
    // workspace: [per-row prescale factors][binary16 image of x][block sums] ..., so that an image made for a scheme
    // with block sums is found at the same place by a scheme without
    float *fac = (float *)workspace;
    void *xh = (uint8_t *)workspace + p.fac_bytes + p.cs_bytes;
    void *sxh = p.sxh_bytes ? (uint8_t *)workspace + p.fac_bytes + p.cs_bytes + p.xh_bytes : nullptr;
    uint8_t *wimg = (uint8_t *)workspace + p.image_end();
    uint8_t *part_base = (uint8_t *)workspace + p.part_off;  // partial results; every part of the workspace is a multiple of 256 bytes
    RLX_TRY(runtime_init());  // the plan counts the device's CUs
    const GemmLaunch g = launch_plan(w->scheme, xk, m, w->dims.k, ns, count, workspace_bytes > p.part_off ? workspace_bytes - p.part_off : 0);
    if (codes) {  // B = fl16(W * diag(s) / S) as stage images; fac holds (1 / S, S) for every row
        WScaleArgs wa{w->dev, wimg, (const float *)((uint8_t *)workspace + p.fac_bytes), fac, w->dims.row_tiles, w->dims.units, (int)p.k_pad, w->sc_off()};
        void *wparams[] = {&wa};
        const KernelId wid = w->scheme == SCHEME_Q4_0 ? K_WSCALE_Q4_0 : K_WSCALE_Q8_0;
        RLX_TRY(launch(wid, (unsigned)(p.k_pad / w->layout.unit_k), (unsigned)((w->dims.n + 255) / 256 * 16), 64, 0, stream, wparams));
    } else if (!prepared) {
        RLX_TRY(launch_xprep(x, xk, m, w->dims.k, p, workspace, stream));
    }
    if (g.kernel == K_GEMVW_Q4_0 || g.kernel == K_GEMVW_Q8_0) {
        GemvWArgs wa{};
        long long wgs = 0;
        size_t off = 0;
        for (int i = 0; i < count; i++) {
            float *dst = outs[i];
            if (g.split[i].split > 1) {
                dst = (float *)(part_base + off);
                off += (size_t)g.split[i].split * (size_t)m * (size_t)ws[i]->dims.n * 4;
            }
            wa.seg[i] = GemvWSeg{ws[i]->dev, dst, (int)ws[i]->dims.n, (int)ws[i]->dims.row_tiles, (int)wgs, g.split[i].split, g.split[i].units_per_split};
            wgs += (ws[i]->dims.row_tiles + 15) / 16 * g.split[i].split;
        }
        wa.nseg = count;
        wa.m = (int)m;
        wa.pair_rows = xk == 0 ? 1 : 0;
        wa.units = (int)w->dims.units;
        wa.k_steps = (int)(p.k_pad / 64);
        wa.xh = xh;
        wa.rowfac = fac;
        void *wparams[] = {&wa};
        RLX_TRY(launch3(g.kernel, (unsigned)wgs, (unsigned)(((xk == 0 ? 2 * m : m) + 63) / 64), 1, 512, 2 * 32768, stream, wparams));
        SplitReduceArgs ra{};
        int nred = 0;
        for (int i = 0; i < count; i++)
            if (g.split[i].split > 1) {
                ra.part[nred] = wa.seg[i].out;
                ra.out[nred] = outs[i];
                ra.elems[nred] = (long long)m * ws[i]->dims.n;
                ra.split[nred++] = g.split[i].split;
            }
        return launch_split_reduce(ra, nred, stream);
    }

    if (g.kernel == K_GEMM_IMG_F16W) {
        GemmImgArgs ia{xh, wimg, outs[0], fac, (int)m, (int)w->dims.n, (int)(p.k_pad / 64)};
        void *iparams[] = {&ia};
        return launch3(g.kernel, (unsigned)((w->dims.n + 255) / 256), (unsigned)(p.m_rows / 256), 1, 512, 2 * 65536, stream, iparams);
    }
    if (g.groups) {
        GemmBigArgs ba{};
        for (int i = 0; i < count; i++) {
            ba.seg[i] = GemmBigSeg{codes ? (const void *)wimg : ws[i]->dev, outs[i], (int)ws[i]->dims.n, (int)ws[i]->dims.row_tiles, ba.tiles_n};
            ba.tiles_n += (int)((ws[i]->dims.n + 255) / 256);
        }
        ba.nseg = count;
        ba.a_img = xh;
        ba.rowfac = fac;
        ba.part = (float *)part_base;
        ba.m_out = (int)m;
        ba.tiles_m = (int)(p.m_rows / 256);
        ba.a_steps = (int)(p.k_pad / 64);
        ba.quads = codes ? (int)(p.k_pad / 128) : (int)w->dims.units;
        ba.pair_rows = xk == 0 ? 1 : 0;
        int groups = g.groups;
        void *bparams[] = {&ba, &groups};
        RLX_TRY(launch(g.kernel, (unsigned)groups, 1, 256, 5 * 32768, stream, bparams));
        if (!g.shared) return RLX_OK;
        return launch(K_GEMM_BIG_REDUCE, (unsigned)(ba.tiles_m * ba.tiles_n), ba.pair_rows ? 8 : 16, 256, 0, stream, bparams);
    }

    const int steps_per_unit = L.unit_k / 64;
    const int64_t rv = xk == 0 ? 2 * m : m;
    const bool skinny = gemm_skinny(xk, m);
    GemmArgs a{};
    long long gx = 0;
    for (int i = 0; i < count; i++) {
        a.seg[i] = GemmSeg{codes ? wimg : ws[i]->dev, outs[i], (int)ws[i]->dims.n, (int)ws[i]->dims.row_tiles, (int)gx};
        gx += (ws[i]->dims.row_tiles * 16 + 127) / 128;
    }
    a.nseg = count;
    const int gy = skinny ? (int)((rv + 63) / 64) : (int)(p.m_rows / 256);
    // Split K: every slice writes its partial result behind the images in the workspace, then one reduce launch adds the slices in
    // ascending K into the outputs.
    const int split = g.split[0].split, units_per_split = g.split[0].units_per_split;
    if (split > 1) {
        size_t off = 0;
        for (int i = 0; i < count; i++) {
            a.seg[i].out = (float *)(part_base + off);
            off += (size_t)split * (size_t)m * (size_t)ws[i]->dims.n * 4;
        }
    }
    a.xh = xh;
    a.sxh = sxh;
    a.m_rows = (int)p.m_rows;
    a.m_out = (int)m;
    a.k_pad = (int)p.k_pad;
    a.units = codes ? (int)(p.k_pad / 64) : (int)w->dims.units;
    a.pair_rows = xk == 0 ? 1 : 0;
    a.steps_per_split = units_per_split * steps_per_unit;
    a.split_out = split > 1 ? 1 : 0;
    a.sc_off = w->sc_off();
    a.rowfac = fac;
    void *params[] = {&a};
    RLX_TRY(launch3(g.kernel, (unsigned)gx, (unsigned)gy, (unsigned)split, 512, skinny ? 3 * 24 * 1024 : 3 * 48 * 1024, stream, params));
    SplitReduceArgs ra{};
    if (split > 1)
        for (int i = 0; i < count; i++) {
            ra.part[i] = a.seg[i].out;
            ra.out[i] = outs[i];
            ra.elems[i] = (long long)m * ws[i]->dims.n;
            ra.split[i] = split;
        }
    return launch_split_reduce(ra, split > 1 ? count : 0, stream);
}

}  // namespace rlx

extern "C" {

// One or `num_experts` [n, k] matrices: validate, repack on the host, upload into `device_mem` (or fresh memory).
int rlx_mi355x_qweight_create_ex(int scheme, uint32_t flags, const void *gguf_bytes, size_t nbytes, int64_t n, int64_t k,
                                 int64_t num_experts, void *device_mem, size_t device_capacity, rlx_qweight **out) {
    using namespace rlx;
    if (!gguf_bytes || !out) {
        set_error("qweight: null argument");
        return RLX_ERR_INVALID;
    }
    *out = nullptr;
    const Layout HL = layout_of(scheme);
    if (HL.unit_k == 0 || HL.block_elems == 0) {
        set_error("qweight: scheme %d is not a claimed GGUF scheme", scheme);
        return RLX_ERR_UNSUPPORTED;
    }
    if (flags & ~(uint32_t)RLX_QW_Q6K_SIGNED_SCALES) {
        set_error("qweight: unknown flags 0x%x", flags);
        return RLX_ERR_INVALID;
    }
    if (n <= 0 || k <= 0 || k % HL.block_elems != 0 || num_experts < 1 || num_experts > 0x7FFFFFFF) {
        set_error("qweight: need n > 0, k a positive multiple of %d and 1 <= experts; got n=%lld k=%lld experts=%lld", HL.block_elems,
                  (long long)n, (long long)k, (long long)num_experts);
        return RLX_ERR_INVALID;
    }
    const int64_t slab = rlx_mi355x_bytes_for(scheme, n * k);
    if (slab < 0 || nbytes != (size_t)slab * (size_t)num_experts) {
        set_error("qweight: got %zu bytes, %lld x [%lld x %lld] needs %lld", nbytes, (long long)num_experts, (long long)n, (long long)k,
                  (long long)(slab < 0 ? -1 : slab * num_experts));
        return RLX_ERR_INVALID;
    }
    const WeightDims D = weight_dims(HL, n, k);
    const size_t total = (size_t)D.bytes * (size_t)num_experts;
    if (device_mem && device_capacity < total) {
        set_error("qweight: the device layout takes %zu bytes, the slot holds %zu", total, device_capacity);
        return RLX_ERR_INVALID;
    }
    RLX_TRY(runtime_init());
    bool owns = false;
    rlx_qweight *qw = nullptr;
    try {
        std::vector<uint8_t> staging(total);
        for (int64_t e = 0; e < num_experts; e++)
            RLX_TRY(repack_host(scheme, flags, (const uint8_t *)gguf_bytes + e * slab, (size_t)slab, n, k, staging.data() + e * D.bytes));
        // `scheme` of a weight names the kernels that read it: Q3_K units are Q6_K units with signed scale bytes
        const uint32_t kflags = scheme == SCHEME_Q3K ? (uint32_t)RLX_QW_Q6K_SIGNED_SCALES : flags;
        qw = new rlx_qweight{kernel_scheme(scheme), HL, D, nullptr, false, (int)num_experts, kflags};
        if (!device_mem) {
            hipError_t me = hipMalloc(&device_mem, total);
            if (me != hipSuccess) {
                delete qw;
                set_error("qweight: hipMalloc(%zu) failed: %s", total, hipGetErrorString(me));
                return me == hipErrorOutOfMemory ? RLX_ERR_NO_MEMORY : RLX_ERR_HIP;
            }
            owns = true;
        }
        hipError_t e = hipMemcpy(device_mem, staging.data(), total, hipMemcpyHostToDevice);
        if (e != hipSuccess) {
            if (owns) (void)hipFree(device_mem);
            delete qw;
            set_error("qweight upload: %s", hipGetErrorString(e));
            return RLX_ERR_HIP;
        }
    } catch (const std::bad_alloc &) {
        delete qw;
        set_error("qweight: out of host memory staging %zu bytes", total);
        return RLX_ERR_NO_MEMORY;
    }
    qw->dev = (uint8_t *)device_mem;
    qw->owns = owns;
    *out = qw;
    return RLX_OK;
}

int rlx_mi355x_qweight_create_at(int scheme, const void *gguf_bytes, size_t nbytes, int64_t n, int64_t k,
                                 void *device_mem, rlx_qweight **out) {
    return rlx_mi355x_qweight_create_ex(scheme, 0, gguf_bytes, nbytes, n, k, 1, device_mem, device_mem ? (size_t)-1 : 0, out);
}

int rlx_mi355x_qweight_create(int scheme, const void *gguf_bytes, size_t nbytes, int64_t n, int64_t k,
                              rlx_qweight **out) {
    return rlx_mi355x_qweight_create_ex(scheme, 0, gguf_bytes, nbytes, n, k, 1, nullptr, 0, out);
}

int rlx_mi355x_qweight_create_experts_at(int scheme, const void *gguf_bytes, size_t nbytes, int64_t n, int64_t k,
                                         int64_t num_experts, void *device_mem, rlx_qweight **out) {
    return rlx_mi355x_qweight_create_ex(scheme, 0, gguf_bytes, nbytes, n, k, num_experts, device_mem, device_mem ? (size_t)-1 : 0, out);
}

int rlx_mi355x_qweight_create_experts(int scheme, const void *gguf_bytes, size_t nbytes, int64_t n, int64_t k,
                                      int64_t num_experts, rlx_qweight **out) {
    return rlx_mi355x_qweight_create_ex(scheme, 0, gguf_bytes, nbytes, n, k, num_experts, nullptr, 0, out);
}

void rlx_mi355x_qweight_destroy(rlx_qweight *w) {
    if (!w) return;
    if (w->owns) (void)hipFree(w->dev);
    delete w;
}

size_t rlx_mi355x_qweight_device_bytes(const rlx_qweight *w) { return w ? (size_t)w->dims.bytes * (size_t)w->experts : 0; }

int rlx_mi355x_dequant(const rlx_qweight *w, float *out_dev, void *stream) {
    using namespace rlx;
    if (!w || !out_dev) {
        set_error("dequant: null argument");
        return RLX_ERR_INVALID;
    }
    DequantArgs a{w->dev, out_dev, w->dims.n, w->dims.k, w->dims.units, w->sc_off()};
    void *params[] = {&a};
    KernelId id = w->scheme == SCHEME_Q4_0 ? K_DEQUANT_Q4_0 : w->scheme == SCHEME_Q8_0 ? K_DEQUANT_Q8_0
                  : w->scheme == SCHEME_Q6K ? K_DEQUANT_Q6_K : w->scheme == SCHEME_Q5K ? K_DEQUANT_Q5_K
                  : w->scheme == SCHEME_Q8K ? K_DEQUANT_Q8_K : w->scheme == SCHEME_Q2K ? K_DEQUANT_Q2_K : K_DEQUANT_Q4_K;
    return launch(id, (unsigned)w->dims.units, (unsigned)w->dims.row_tiles, 64, 0, (hipStream_t)stream, params);
}

size_t rlx_mi355x_gguf_matmul_workspace(int scheme, int x_dtype, int64_t m, int64_t k, int64_t n) {
    using namespace rlx;
    if (x_dtype == RLX_I8)  // a FakeQuantize code image and the scaled weights of the widest matrix it is multiplied by
        return !code_image_scheme(scheme) || m <= 0 || k <= 0 || n < 0 ? 0 : gemm_plan(scheme, XK_CODES, m, k, &n, n > 0).total();
    int xk = x_kind(x_dtype);
    if (xk < 0 || layout_of(scheme).unit_k == 0 || m <= decode_rows(xk)) return 0;  // decode path: no workspace
    return gemm_plan(scheme, xk, m, k, &n, n > 0).total();  // n = 0: the operand image alone (what ..._prepare writes)
}

int rlx_mi355x_gguf_matmul_plan(int scheme, int x_dtype, int64_t m, int64_t k, const int64_t *ns, int count, size_t workspace_bytes,
                                size_t *want_bytes, char *buf, size_t cap) {
    using namespace rlx;
    const int xk = x_dtype == RLX_I8 ? XK_CODES : x_kind(x_dtype);
    bool ok = ns && count > 0 && xk >= 0 && m > 0 && k > 0 && layout_of(scheme).unit_k != 0 && (xk != XK_CODES || code_image_scheme(scheme));
    for (int i = 0; ok && i < count; i++) ok = ns[i] > 0;
    if (!ok) {
        set_error("gguf_matmul_plan: needs a claimed scheme (Q4_0 / Q8_0 on a code image), F32 / BF16 / F16 / I8 activations and sizes above zero");
        return RLX_ERR_INVALID;
    }
    if (want_bytes) *want_bytes = 0;
    if (buf && cap) buf[0] = 0;
    if (xk != XK_CODES && m <= decode_rows(xk)) return 0;
    size_t pos = 0;
    int launches = 0;
    for (int i = 0; i < count; launches++) {
        const int c = std::min(count - i, prefill_launch_max(scheme, xk, m));
        const GemmPlan p = gemm_plan(scheme, xk, m, k, ns + i, c);
        if (want_bytes) *want_bytes = std::max(*want_bytes, p.total());
        const GemmLaunch g = launch_plan(scheme, xk, m, k, ns + i, c, workspace_bytes > p.part_off ? workspace_bytes - p.part_off : 0);
        if (buf && pos < cap) {
            pos += (size_t)snprintf(buf + pos, cap - pos, "%s: %d %s, %s, %zu bytes of partial results\n", kernel_name(g.kernel), c,
                                    c == 1 ? "matrix" : "matrices", g.shared ? "shared tiles" : g.part_bytes ? "split K" : "whole", g.part_bytes);
        }
        i += c;
    }
    return launches;
}

int rlx_mi355x_gguf_decode_plan(int scheme, int x_dtype, int64_t m, int64_t k, const int64_t *ns, int count, char *buf, size_t cap) {
    using namespace rlx;
    const int xk = x_kind(x_dtype);
    bool ok = ns && count > 0 && count <= GEMV_MAX_SEG && xk >= 0 && m > 0 && k > 0 && layout_of(scheme).unit_k != 0 && m <= decode_rows(xk);
    for (int i = 0; ok && i < count; i++) ok = ns[i] > 0;
    if (!ok) {
        set_error("gguf_decode_plan: needs a claimed scheme, F32 / BF16 / F16 activations, sizes above zero, up to %d matrices and a decode batch", GEMV_MAX_SEG);
        return RLX_ERR_INVALID;
    }
    rlx_qweight w[GEMV_MAX_SEG];
    const rlx_qweight *ws[GEMV_MAX_SEG];
    const void *xs[GEMV_MAX_SEG] = {};
    float *outs[GEMV_MAX_SEG] = {};
    const int kernels = kernel_scheme(scheme);  // as a weight of this scheme is kept
    for (int i = 0; i < count; i++) {
        w[i] = rlx_qweight{kernels, layout_of(scheme), weight_dims(scheme, ns[i], k), nullptr, false, 1, 0};
        ws[i] = &w[i];
    }
    GemvLaunch g;
    RLX_TRY(plan_gemv(xs, xk, ws, outs, count, (int)m, nullptr, nullptr, nullptr, nullptr, g));
    if (buf && cap) {
        snprintf(buf, cap, "%s: %d workgroups, %d waves, %d on a tile, up to %d tiles, chunks of %d units", kernel_name(g.kernel), g.wgs, g.waves, g.a.kw,
                 g.a.max_tiles_per_wg, g.a.kc_units);
    }
    return RLX_OK;
}

int rlx_mi355x_gguf_matmul_bt_batch(const void *const *xs_dev, int x_dtype, const rlx_qweight *const *ws,
                                    float *const *outs_dev, int count, int64_t m, void *workspace, size_t workspace_bytes,
                                    void *stream) {
    using namespace rlx;
    if (!xs_dev || !ws || !outs_dev || count <= 0 || m <= 0) {
        set_error("gguf_matmul_bt: null argument, count=%d or m=%lld", count, (long long)m);
        return RLX_ERR_INVALID;
    }
    for (int i = 0; i < count; i++) {
        if (!ws[i] || !outs_dev[i] || !xs_dev[i]) {
            set_error("gguf_matmul_bt: null activations / weight / output %d", i);
            return RLX_ERR_INVALID;
        }
        if (ws[i]->scheme != ws[0]->scheme) {
            set_error("gguf_matmul_bt_batch: weight %d differs in scheme from weight 0", i);
            return RLX_ERR_INVALID;
        }
    }
    int xk = x_kind(x_dtype);
    if (xk < 0) {
        set_error("gguf_matmul_bt: activation dtype %d unsupported (F32, BF16, F16 only)", x_dtype);
        return RLX_ERR_UNSUPPORTED;
    }
    const int64_t cap = decode_rows(xk);  // activation rows one pass of the decode kernels holds
    const size_t esz = xk == 0 ? 4 : 2;
    if (m > cap) {  // prefill: one GEMM per weight, sharing the workspace (same stream, so launches are ordered)
        // q, k, v (and gate, up) of a layer share their input: its f16 image in the workspace is made once. An image
        // with block sums (Q4_K / Q5_K: per 32 columns; Q2_K: per 16) also serves a scheme that reads none, not the
        // other way round, and not a scheme that reads the other kind.
        // Consecutive matrices with the same input and K go into one launch, up to GEMM_MAX_SEG at a time (GEMVW_MAX_SEG for the 64-rows-a-pass kernel).
        const void *have_x = nullptr;
        int64_t have_k = -1;
        int have_sums = 0;
        for (int i = 0; i < count;) {
            int c = 1;
            const int most = prefill_launch_max(ws[i]->scheme, xk, m);
            while (i + c < count && c < most && xs_dev[i + c] == xs_dev[i] && ws[i + c]->dims.k == ws[i]->dims.k &&
                   ws[i + c]->layout.unit_bytes == ws[i]->layout.unit_bytes && ws[i + c]->sc_off() == ws[i]->sc_off())
                c++;
            const int sums = act_sums_kind(ws[i]->scheme);
            const bool prepared = xs_dev[i] == have_x && ws[i]->dims.k == have_k && (sums == 0 || sums == have_sums);
            RLX_TRY(launch_gemm(xs_dev[i], xk, ws + i, outs_dev + i, c, m, workspace, workspace_bytes, (hipStream_t)stream, prepared));
            if (!prepared) {
                have_x = xs_dev[i];
                have_k = ws[i]->dims.k;
                have_sums = sums;
            }
            i += c;
        }
        return RLX_OK;
    }
    for (int64_t r0 = 0; r0 < m; r0 += cap) {
        int rows = (int)std::min<int64_t>(cap, m - r0);
        for (int c0 = 0; c0 < count; c0 += GEMV_MAX_SEG) {
            int c = std::min(GEMV_MAX_SEG, count - c0);
            float *outs[GEMV_MAX_SEG];
            const void *xs[GEMV_MAX_SEG];
            for (int i = 0; i < c; i++) {
                outs[i] = outs_dev[c0 + i] + r0 * ws[c0 + i]->dims.n;
                xs[i] = (const uint8_t *)xs_dev[c0 + i] + (size_t)r0 * ws[c0 + i]->dims.k * esz;
            }
            RLX_TRY(launch_gemv(xs, xk, ws + c0, outs, c, rows, (hipStream_t)stream));
        }
    }
    return RLX_OK;
}

// The two halves of the prefill path as calls of their own, for a caller that multiplies one activation tensor by several
// weights at different points of its schedule (or wants the conversion outside a timed region): prepare converts x into
// the workspace image once, prepared multiplies that image by up to four matrices of one scheme and K per launch.
int rlx_mi355x_gguf_matmul_prepare(const void *x_dev, int x_dtype, int scheme, int64_t m, int64_t k, void *workspace,
                                   size_t workspace_bytes, void *stream) {
    using namespace rlx;
    const int xk = x_kind(x_dtype);
    const Layout L = layout_of(scheme);
    if (!x_dev || xk < 0 || L.unit_k == 0 || m <= decode_rows(xk) || k <= 0 || k % 32 != 0) {
        set_error("gguf_matmul_prepare: needs F32 / BF16 / F16 activations, a claimed scheme, k a multiple of 32 and m above the decode limit (%lld)",
                  (long long)decode_rows(xk < 0 ? 0 : xk));
        return RLX_ERR_INVALID;
    }
    const GemmPlan p = gemm_plan(scheme, xk, m, k);
    if (!workspace || workspace_bytes < p.total() || (uintptr_t)workspace % 16 != 0 || (uintptr_t)x_dev % 16 != 0) {
        set_error("gguf_matmul_prepare: a 16-byte aligned workspace of %zu bytes is needed, got %zu", p.total(), workspace_bytes);
        return RLX_ERR_INVALID;
    }
    return launch_xprep(x_dev, xk, m, k, p, workspace, (hipStream_t)stream);
}

int rlx_mi355x_gguf_matmul_bt_prepared(const void *workspace, size_t workspace_bytes, int x_dtype, const rlx_qweight *const *ws,
                                       float *const *outs_dev, int count, int64_t m, void *stream) {
    using namespace rlx;
    const int xk = x_dtype == RLX_I8 ? XK_CODES : x_kind(x_dtype);
    if (!workspace || !ws || !outs_dev || count <= 0 || xk < 0 || m <= (xk == XK_CODES ? 0 : decode_rows(xk))) {
        set_error("gguf_matmul_bt_prepared: null argument, count=%d, or m=%lld within the decode limit", count, (long long)m);
        return RLX_ERR_INVALID;
    }
    for (int i = 0; i < count; i++)
        if (!ws[i] || !outs_dev[i]) {
            set_error("gguf_matmul_bt_prepared: null weight / output %d", i);
            return RLX_ERR_INVALID;
        }
    if (xk == XK_CODES) {  // one matrix at a time: each is scaled into the workspace's weight image first
        for (int i = 0; i < count; i++)
            if (!code_image_scheme(ws[i]->scheme)) {
                // the other schemes' prefill operands are exact integers; a weight rounded to binary16 would cost them accuracy
                set_error("gguf_matmul_bt_prepared: a FakeQuantize code image multiplies Q4_0 / Q8_0 weights only (weight %d is scheme %d)", i, ws[i]->scheme);
                return RLX_ERR_UNSUPPORTED;
            }
        for (int i = 0; i < count; i++)
            RLX_TRY(launch_gemm(workspace, xk, ws + i, outs_dev + i, 1, m, const_cast<void *>(workspace), workspace_bytes, (hipStream_t)stream, true));
        return RLX_OK;
    }
    for (int i = 0; i < count;) {
        int c = 1;
        while (i + c < count && c < GEMM_MAX_SEG && ws[i + c]->scheme == ws[i]->scheme && ws[i + c]->dims.k == ws[i]->dims.k &&
               ws[i + c]->sc_off() == ws[i]->sc_off())
            c++;
        // of `workspace` only what lies past every scheme's image is written; the x pointer is not looked at when the image is already there
        RLX_TRY(launch_gemm(workspace, xk, ws + i, outs_dev + i, c, m, const_cast<void *>(workspace), workspace_bytes, (hipStream_t)stream, true));
        i += c;
    }
    return RLX_OK;
}

int rlx_mi355x_gguf_matmul_bt(const void *x_dev, int x_dtype, const rlx_qweight *w, float *out_dev, int64_t m,
                              void *workspace, size_t workspace_bytes, void *stream) {
    return rlx_mi355x_gguf_matmul_bt_batch(&x_dev, x_dtype, &w, &out_dev, 1, m, workspace, workspace_bytes, stream);
}

// Shared checks of the RMSNorm-prologue entry points: f32 activations, decode sizes, 16-byte aligned gamma / beta.
static int check_norm(const char *who, const void *x_dev, const float *gamma_dev, const float *beta_dev, int64_t m) {
    if (!x_dev || !gamma_dev || m <= 0) {
        rlx::set_error("%s: null argument or m <= 0", who);
        return RLX_ERR_INVALID;
    }
    if (m > 8) {
        rlx::set_error("%s: the fused RMSNorm covers the decode path (m <= 8 f32 rows)", who);
        return RLX_ERR_UNSUPPORTED;
    }
    if ((uintptr_t)gamma_dev % 16 != 0 || (uintptr_t)beta_dev % 16 != 0) {
        rlx::set_error("%s: gamma and beta must be 16-byte aligned", who);
        return RLX_ERR_INVALID;
    }
    return RLX_OK;
}

int rlx_mi355x_rmsnorm_gguf_matmul_bt_batch(const float *x_dev, const float *gamma_dev, const float *beta_dev, float eps,
                                            const rlx_qweight *const *ws, float *const *outs_dev, int count, int64_t m,
                                            void *stream) {
    using namespace rlx;
    RLX_TRY(check_norm("rmsnorm_gguf_matmul_bt_batch", x_dev, gamma_dev, beta_dev, m));
    if (!ws || !outs_dev || count <= 0) {
        set_error("rmsnorm_gguf_matmul_bt_batch: null argument or count <= 0");
        return RLX_ERR_INVALID;
    }
    const RmsNorm norm{gamma_dev, beta_dev, eps};
    for (int i0 = 0; i0 < count; i0 += GEMV_MAX_SEG) {
        const int c = std::min(GEMV_MAX_SEG, count - i0);
        const void *xs[GEMV_MAX_SEG];
        for (int i = 0; i < c; i++) {
            if (!ws[i0 + i] || !outs_dev[i0 + i] || ws[i0 + i]->experts != 1) {
                set_error("rmsnorm_gguf_matmul_bt_batch: null weight / output or an expert stack at %d", i0 + i);
                return RLX_ERR_INVALID;
            }
            const bool same = ws[i0 + i]->scheme == ws[i0]->scheme;
            if (!same || ws[i0 + i]->dims.k != ws[0]->dims.k) {
                set_error("rmsnorm_gguf_matmul_bt_batch: the matrices share one normalized input, so one scheme and one k");
                return RLX_ERR_INVALID;
            }
            xs[i] = x_dev;
        }
        RLX_TRY(launch_gemv(xs, 0, ws + i0, outs_dev + i0, c, (int)m, (hipStream_t)stream, nullptr, nullptr, nullptr, &norm));
    }
    return RLX_OK;
}

int rlx_mi355x_rmsnorm_gguf_matmul_swiglu(const float *x_dev, const float *gamma_dev, const float *beta_dev, float eps,
                                          const rlx_qweight *w_up, const rlx_qweight *w_gate, float *out_dev, int64_t m,
                                          void *stream) {
    using namespace rlx;
    RLX_TRY(check_norm("rmsnorm_gguf_matmul_swiglu", x_dev, gamma_dev, beta_dev, m));
    if (!w_up || !w_gate || !out_dev) {
        set_error("rmsnorm_gguf_matmul_swiglu: null argument");
        return RLX_ERR_INVALID;
    }
    const bool same_layout = w_up->scheme == w_gate->scheme;
    if (!same_layout || w_up->dims.n != w_gate->dims.n || w_up->dims.k != w_gate->dims.k || w_up->experts != 1 ||
        w_gate->experts != 1) {
        set_error("rmsnorm_gguf_matmul_swiglu: the up and gate projections must share scheme, n and k");
        return RLX_ERR_INVALID;
    }
    const RmsNorm norm{gamma_dev, beta_dev, eps};
    const void *xs[1] = {x_dev};
    const rlx_qweight *ws[1] = {w_up};
    const rlx_qweight *ps[1] = {w_gate};
    float *outs[1] = {out_dev};
    return launch_gemv(xs, 0, ws, outs, 1, (int)m, (hipStream_t)stream, nullptr, nullptr, ps, &norm);
}

int rlx_mi355x_rmsnorm_gguf_tied_lm_argmax(const float *hidden_dev, const float *gamma_dev, const float *beta_dev, float eps,
                                           const rlx_qweight *embed, uint32_t *out_idx_dev, float *out_val_dev,
                                           void *key_scratch_dev, void *stream) {
    using namespace rlx;
    RLX_TRY(check_norm("rmsnorm_gguf_tied_lm_argmax", hidden_dev, gamma_dev, beta_dev, 1));
    if (!embed || !out_idx_dev || !out_val_dev || !key_scratch_dev || (uintptr_t)key_scratch_dev % 8 != 0) {
        set_error("rmsnorm_gguf_tied_lm_argmax: null argument or misaligned key scratch");
        return RLX_ERR_INVALID;
    }
    const RmsNorm norm{gamma_dev, beta_dev, eps};
    const void *xs[1] = {hidden_dev};
    const rlx_qweight *ws[1] = {embed};
    float *outs[1] = {nullptr};
    int wgs = 0;
    RLX_TRY(launch_gemv(xs, 0, ws, outs, 1, 1, (hipStream_t)stream, nullptr, (unsigned long long *)key_scratch_dev, nullptr, &norm, &wgs));
    void *params[] = {&key_scratch_dev, &wgs, &out_idx_dev, &out_val_dev};
    return launch(K_ARGMAX_FINISH, 1, 1, 256, 0, (hipStream_t)stream, params);
}

int rlx_mi355x_gguf_matmul_swiglu(const void *x_dev, int x_dtype, const rlx_qweight *w_up, const rlx_qweight *w_gate,
                                  float *out_dev, int64_t m, void *stream) {
    using namespace rlx;
    if (!x_dev || !w_up || !w_gate || !out_dev || m <= 0) {
        set_error("gguf_matmul_swiglu: null argument or m <= 0");
        return RLX_ERR_INVALID;
    }
    int xk = x_kind(x_dtype);
    if (xk < 0) {
        set_error("gguf_matmul_swiglu: activation dtype %d is not F32 / BF16 / F16", x_dtype);
        return RLX_ERR_UNSUPPORTED;
    }
    const bool same_layout = w_up->scheme == w_gate->scheme;
    if (!same_layout || w_up->dims.n != w_gate->dims.n || w_up->dims.k != w_gate->dims.k || w_up->experts != 1 ||
        w_gate->experts != 1) {
        set_error("gguf_matmul_swiglu: the up and gate projections must share scheme, n and k");
        return RLX_ERR_INVALID;
    }
    if (m > (xk == 0 ? 8 : 16)) {
        set_error("gguf_matmul_swiglu: the fused form covers the decode path (m <= %d for this dtype); run two matmuls above it",
                  xk == 0 ? 8 : 16);
        return RLX_ERR_UNSUPPORTED;
    }
    const void *xs[1] = {x_dev};
    const rlx_qweight *ws[1] = {w_up};
    const rlx_qweight *ps[1] = {w_gate};
    float *outs[1] = {out_dev};
    return launch_gemv(xs, xk, ws, outs, 1, (int)m, (hipStream_t)stream, nullptr, nullptr, ps);
}

namespace rlx {
struct RowOpArgs {  // mirrors kernels/rowops.hip
    const float *x;
    const float *gamma;
    const float *beta;
    float *out;
    long long rows, h;
    float eps;
    int gate_first;
    int vec4;
};
}  // namespace rlx

int rlx_mi355x_rms_norm(const float *x_dev, const float *gamma_dev, const float *beta_dev, float eps, float *out_dev, int64_t rows,
                        int64_t h, void *stream) {
    using namespace rlx;
    if (!x_dev || !gamma_dev || !out_dev || rows <= 0 || h <= 0) {
        set_error("rms_norm: null argument, rows=%lld or h=%lld", (long long)rows, (long long)h);
        return RLX_ERR_INVALID;
    }
    RowOpArgs a{x_dev, gamma_dev, beta_dev, out_dev, rows, h, eps, 0, 0};
    a.vec4 = h % 4 == 0 && ((uintptr_t)x_dev | (uintptr_t)gamma_dev | (uintptr_t)beta_dev | (uintptr_t)out_dev) % 16 == 0;
    void *params[] = {&a};
    // Rows that up to 1024 threads can hold, four 16-byte groups each (ROW_KEEP in kernels/rowops.hip), on as few threads as do, so that
    // the rows of a prompt are on the chip at once. us, read twice / kept, three buffers in turn: 1111 rows of 4096 10.5 / 8.4, 4096 rows
    // of 4096 33.8 / 27.3, 1500 of 2052 7.5 / 7.0 (on 256 threads 7.9), 2000 of 16384 63.7 / 58.8; rows of 2048 and less are no faster
    // kept. Between 8192 and 16384 columns 1024 threads hold more than there is, and with 85 registers a CU has room for one such
    // workgroup: kept pays where a row has a CU to itself (64 rows of 10240 4.6 / 4.3; 300 rows 8.1 / 9.4) and, the fuller the
    // threads, the earlier again where there are many rows (12288: 1111 rows 27.0 / 28.2, 1500 34.8 / 32.6; 15360: 700 rows 20.2 / 20.4, 1024 32.4 / 30.3).
    const int64_t kept_from = h <= 8192 || h >= 16000 ? 0 : h >= 15000 ? 900 : h >= 12000 ? 1400 : INT64_MAX;
    const bool keep = a.vec4 && h > 2048 && h <= 16384 && (rows <= 256 || rows >= kept_from);
    const unsigned bx = keep ? (h <= 3072 ? 192 : h <= 4096 ? 256 : h <= 8192 ? 512 : 1024) : h >= 4096 ? 1024 : 256;
    return launch(keep ? K_RMSNORM_ROWS_KEEP : K_RMSNORM_ROWS, (unsigned)std::min<int64_t>(rows, 1 << 20), 1, bx, 0, (hipStream_t)stream, params);
}

int rlx_mi355x_fused_swiglu(const float *in_dev, float *out_dev, int64_t rows, int64_t n_half, int gate_first, void *stream) {
    using namespace rlx;
    if (!in_dev || !out_dev || rows <= 0 || n_half <= 0) {
        set_error("fused_swiglu: null argument, rows=%lld or n_half=%lld", (long long)rows, (long long)n_half);
        return RLX_ERR_INVALID;
    }
    RowOpArgs a{in_dev, nullptr, nullptr, out_dev, rows, n_half, 0.f, gate_first ? 1 : 0, 0};
    a.vec4 = n_half % 4 == 0 && ((uintptr_t)in_dev | (uintptr_t)out_dev) % 16 == 0;
    void *params[] = {&a};
    const int64_t items = a.vec4 ? rows * n_half / 4 : rows * n_half;
    const unsigned gx = (unsigned)std::min<int64_t>((items + 255) / 256, 16 * (int64_t)device_props().cu_count);
    return launch(K_SWIGLU_ROWS, gx, 1, 256, 0, (hipStream_t)stream, params);
}

int rlx_mi355x_qweight_rows(const rlx_qweight *w, int64_t row0, int64_t rows, rlx_qweight **out) {
    using namespace rlx;
    if (out) *out = nullptr;
    if (!w || !out || w->experts != 1 || row0 < 0 || rows <= 0 || row0 + rows > w->dims.n || row0 % TILE_ROWS != 0 ||
        (rows % TILE_ROWS != 0 && row0 + rows != w->dims.n)) {
        set_error("qweight_rows: rows [%lld, %lld) of a plain %lld-row weight must begin and end on a multiple of %d", (long long)row0,
                  (long long)(row0 + rows), w ? (long long)w->dims.n : 0LL, TILE_ROWS);
        return RLX_ERR_INVALID;
    }
    rlx_qweight *v = new (std::nothrow) rlx_qweight(*w);
    if (!v) {
        set_error("qweight_rows: out of host memory");
        return RLX_ERR_NO_MEMORY;
    }
    v->dims = weight_dims(w->layout, rows, w->dims.k);
    v->dev = w->dev + (row0 / TILE_ROWS) * w->dims.units * (int64_t)w->layout.unit_bytes;
    v->owns = false;
    *out = v;
    return RLX_OK;
}

int rlx_mi355x_gguf_tied_lm_argmax(const void *hidden_dev, int x_dtype, const rlx_qweight *embed, uint32_t *out_idx_dev,
                                   float *out_val_dev, void *key_scratch_dev, void *stream) {
    using namespace rlx;
    if (!hidden_dev || !embed || !out_idx_dev || !out_val_dev || !key_scratch_dev) {
        set_error("gguf_tied_lm_argmax: null argument");
        return RLX_ERR_INVALID;
    }
    int xk = x_kind(x_dtype);
    if (xk < 0) {
        set_error("gguf_tied_lm_argmax: hidden dtype %d is not F32 / BF16 / F16", x_dtype);
        return RLX_ERR_UNSUPPORTED;
    }
    if ((uintptr_t)key_scratch_dev % 8 != 0) {
        set_error("gguf_tied_lm_argmax: the key scratch must be 8-byte aligned");
        return RLX_ERR_INVALID;
    }
    const void *xs[1] = {hidden_dev};
    const rlx_qweight *ws[1] = {embed};
    float *outs[1] = {nullptr};
    int wgs = 0;
    RLX_TRY(launch_gemv(xs, xk, ws, outs, 1, 1, (hipStream_t)stream, nullptr, (unsigned long long *)key_scratch_dev, nullptr, nullptr, &wgs));
    void *params[] = {&key_scratch_dev, &wgs, &out_idx_dev, &out_val_dev};
    return launch(K_ARGMAX_FINISH, 1, 1, 256, 0, (hipStream_t)stream, params);
}

namespace rlx {
struct TopkArgs {  // mirrors kernels/topk.hip
    const float *vals;
    const unsigned long long *keys_in;
    int n, cap;
    unsigned long long *keys_out;
    uint32_t *out_idx;
    float *out_val;
};
constexpr int64_t TOPK_GROUP = 1024;   // candidates one wave of rlx_topk_serial / rlx_topk_select reduces to `cap`
constexpr int64_t TOPK_FINISH = 8192;  // candidates rlx_topk_finish takes
// Winners one by one or by threshold, in us of the whole call on Q8_0 rows of 1024 columns. Reducing 1024s: 128256 rows at cap 1 29.7
// one by one, 30.0 by threshold; 9000 rows at cap 8 18.3 either way, at cap 11 19.0 against 18.7.
constexpr int TOPK_SERIAL_CAP = 8;
// The end, one by one in a single wave or by threshold in a workgroup of sixteen, which up to 128 candidates has nothing to cut: 128 rows
// at cap 1 7.9 against 9.7, at cap 8 9.7 either way; 300 rows at cap 1 7.9 against 9.7, at cap 20 12.8 against 13.1, at cap 24 14.0
// against 13.1; 1000 rows at cap 1 8.0 against 9.9, at cap 4 8.8 against 14.3, at cap 24 14.1 against 14.4.
static bool topk_serial_end(int64_t count, int cap) { return cap <= (count <= 128 ? 8 : count <= 512 ? 20 : count <= TOPK_GROUP ? 24 : 0); }
constexpr int TOPK_MAX_CAP = 64;
static int64_t topk_groups(int64_t n) { return (n + TOPK_GROUP - 1) / TOPK_GROUP; }
}  // namespace rlx

size_t rlx_mi355x_tied_lm_argmax_scratch_bytes(void) { return (size_t)rlx::ARGMAX_MAX_WGS * 8; }

size_t rlx_mi355x_tied_lm_topk_scratch_bytes(int64_t n_vocab, int cap) {
    using namespace rlx;
    if (n_vocab <= 0 || cap <= 0) return 0;
    const int64_t c = std::min<int64_t>(std::min<int64_t>(cap, TOPK_MAX_CAP), n_vocab);
    // the logits, then two key areas the passes alternate between (the first pass writes the largest)
    const int64_t keys = topk_groups(n_vocab) * c;
    return (size_t)((n_vocab * 4 + 7) / 8 * 8 + 2 * keys * 8);
}

static int tied_lm_topk(const char *who, const void *hidden_dev, int xk, const rlx::RmsNorm *norm, const rlx_qweight *embed, int cap,
                        uint32_t *out_idx_dev, float *out_val_dev, void *scratch_dev, size_t scratch_bytes, void *stream) {
    using namespace rlx;
    const int64_t n = embed->dims.n;
    if (cap < 1) cap = 1;  // the reference's cap.min(n_vocab).max(1)
    if (cap > n) cap = (int)n;
    if (cap > TOPK_MAX_CAP) {
        set_error("%s: cap %d is beyond the selection kernel (cap <= %d)", who, cap, TOPK_MAX_CAP);
        return RLX_ERR_UNSUPPORTED;
    }
    if ((uintptr_t)scratch_dev % 8 != 0 || scratch_bytes < rlx_mi355x_tied_lm_topk_scratch_bytes(n, cap)) {
        set_error("%s: scratch of %zu bytes (8-byte aligned) needed, got %zu", who, rlx_mi355x_tied_lm_topk_scratch_bytes(n, cap),
                  scratch_bytes);
        return RLX_ERR_INVALID;
    }
    float *logits = (float *)scratch_dev;
    unsigned long long *keys[2];
    keys[0] = (unsigned long long *)((uint8_t *)scratch_dev + (n * 4 + 7) / 8 * 8);
    keys[1] = keys[0] + topk_groups(n) * cap;
    const void *xs[1] = {hidden_dev};
    const rlx_qweight *ws[1] = {embed};
    float *outs[1] = {logits};
    RLX_TRY(launch_gemv(xs, xk, ws, outs, 1, 1, (hipStream_t)stream, nullptr, nullptr, nullptr, norm));
    // One launch orders up to TOPK_FINISH candidates; more than that first lose all but the cap best of every 1024.
    int64_t count = n;
    int side = 0;
    bool first = true;
    for (; count > TOPK_FINISH; first = false, side ^= 1) {
        const int64_t groups = topk_groups(count);
        TopkArgs p{first ? logits : nullptr, first ? nullptr : keys[side ^ 1], (int)count, cap, keys[side], nullptr, nullptr};
        void *params[] = {&p};
        RLX_TRY(launch(cap <= TOPK_SERIAL_CAP ? K_TOPK_SERIAL : K_TOPK_SELECT, (unsigned)groups, 1, 64, 0, (hipStream_t)stream, params));
        count = groups * cap;
    }
    TopkArgs p{first ? logits : nullptr, first ? nullptr : keys[side ^ 1], (int)count, cap, nullptr, out_idx_dev, out_val_dev};
    void *params[] = {&p};
    const bool serial = topk_serial_end(count, cap);
    return launch(serial ? K_TOPK_SERIAL : K_TOPK_FINISH, 1, 1, serial ? 64 : 1024, 0, (hipStream_t)stream, params);
}

int rlx_mi355x_gguf_tied_lm_topk(const void *hidden_dev, int x_dtype, const rlx_qweight *embed, int cap, uint32_t *out_idx_dev,
                                 float *out_val_dev, void *scratch_dev, size_t scratch_bytes, void *stream) {
    using namespace rlx;
    if (!hidden_dev || !embed || !out_idx_dev || !out_val_dev || !scratch_dev) {
        set_error("gguf_tied_lm_topk: null argument");
        return RLX_ERR_INVALID;
    }
    const int xk = x_kind(x_dtype);
    if (xk < 0) {
        set_error("gguf_tied_lm_topk: hidden dtype %d is not F32 / BF16 / F16", x_dtype);
        return RLX_ERR_UNSUPPORTED;
    }
    return tied_lm_topk("gguf_tied_lm_topk", hidden_dev, xk, nullptr, embed, cap, out_idx_dev, out_val_dev, scratch_dev, scratch_bytes, stream);
}

int rlx_mi355x_rmsnorm_gguf_tied_lm_topk(const float *hidden_dev, const float *gamma_dev, const float *beta_dev, float eps,
                                         const rlx_qweight *embed, int cap, uint32_t *out_idx_dev, float *out_val_dev,
                                         void *scratch_dev, size_t scratch_bytes, void *stream) {
    using namespace rlx;
    RLX_TRY(check_norm("rmsnorm_gguf_tied_lm_topk", hidden_dev, gamma_dev, beta_dev, 1));
    if (!embed || !out_idx_dev || !out_val_dev || !scratch_dev) {
        set_error("rmsnorm_gguf_tied_lm_topk: null argument");
        return RLX_ERR_INVALID;
    }
    const RmsNorm norm{gamma_dev, beta_dev, eps};
    return tied_lm_topk("rmsnorm_gguf_tied_lm_topk", hidden_dev, 0, &norm, embed, cap, out_idx_dev, out_val_dev, scratch_dev, scratch_bytes,
                        stream);
}

namespace rlx {
// Sizes of the expert-sorted path: an expert's run of tokens is padded to one 64-row tile of the prefill image (64 tokens,
// or 32 where an f32 token takes two image rows), so the sorted order holds at most m + experts * (group - 1) rows.
struct MoePlan {
    int group;        // tokens per tile
    int64_t perm_len; // rows of the sorted, padded order
    size_t head;      // bytes of perm + tile_expert in front of the GEMM workspace
    GemmPlan gemm;
    size_t total() const { return head + gemm.total(); }
};
static MoePlan moe_plan(int scheme, int xk, int64_t m, int64_t k, int64_t experts) {
    MoePlan p;
    p.group = xk == 0 ? 32 : 64;
    p.perm_len = (m + experts * (p.group - 1) + p.group - 1) / p.group * p.group;
    p.head = ((size_t)(p.perm_len + p.perm_len / p.group) * 4 + 255) & ~(size_t)255;
    p.gemm = gemm_plan(scheme, xk, p.perm_len, k);
    return p;
}
static bool moe_sorted_applies(int xk, int64_t m, int64_t experts) { return m > decode_rows(xk) && experts <= MOE_MAX_EXPERTS; }
}  // namespace rlx

size_t rlx_mi355x_gguf_grouped_matmul_workspace(int scheme, int x_dtype, int64_t m, int64_t k, int64_t num_experts) {
    using namespace rlx;
    const int xk = x_kind(x_dtype);
    if (xk < 0 || layout_of(scheme).unit_k == 0 || m <= 0 || k <= 0 || num_experts < 1 || !moe_sorted_applies(xk, m, num_experts)) return 0;
    return moe_plan(scheme, xk, m, k, num_experts).total();
}

int rlx_mi355x_gguf_grouped_matmul_bt_ws(const void *x_dev, int x_dtype, const rlx_qweight *w, const float *expert_idx_dev,
                                         float *out_dev, int64_t m, void *workspace, size_t workspace_bytes, void *stream) {
    using namespace rlx;
    if (!x_dev || !w || !expert_idx_dev || !out_dev || m <= 0) {
        set_error("gguf_grouped_matmul_bt: null argument or m=%lld", (long long)m);
        return RLX_ERR_INVALID;
    }
    const int xk = x_kind(x_dtype);
    if (xk < 0) {
        set_error("gguf_grouped_matmul_bt: activation dtype %d is not F32 / BF16 / F16", x_dtype);
        return RLX_ERR_UNSUPPORTED;
    }
    if (!moe_sorted_applies(xk, m, w->experts))  // decode sizes (or more experts than the sort kernel counts): a launch per eight tokens
        return rlx_mi355x_gguf_grouped_matmul_bt(x_dev, x_dtype, w, expert_idx_dev, out_dev, m, stream);
    const MoePlan p = moe_plan(w->scheme, xk, m, w->dims.k, w->experts);
    if (!workspace || workspace_bytes < p.total() || (uintptr_t)workspace % 16 != 0 || (uintptr_t)x_dev % 16 != 0) {
        set_error("gguf_grouped_matmul_bt: m=%lld over %d experts needs a 16-byte aligned workspace of %zu bytes, got %zu", (long long)m,
                  w->experts, p.total(), workspace_bytes);
        return RLX_ERR_INVALID;
    }
    if (p.gemm.m_rows > 0x7FFFFFFF || m > 0x7FFFFFFF / 2) {
        set_error("gguf_grouped_matmul_bt: m=%lld is beyond the 32-bit row indices of the sorted path", (long long)m);
        return RLX_ERR_UNSUPPORTED;
    }
    RLX_TRY(runtime_init());
    hipStream_t s = (hipStream_t)stream;
    int *perm = (int *)workspace, *tile_expert = perm + p.perm_len;
    void *gws = (uint8_t *)workspace + p.head;
    MoeSortArgs sa{expert_idx_dev, (int)m, w->experts, p.group, (int)p.perm_len, perm, tile_expert};
    void *sparams[] = {&sa};
    RLX_TRY(launch(K_MOE_SORT, 1, 1, 1024, 0, s, sparams));
    RLX_TRY(launch_xprep(x_dev, xk, m, w->dims.k, p.gemm, gws, s, perm, (int)p.perm_len));
    if (w->scheme == SCHEME_Q4_0 || w->scheme == SCHEME_Q8_0) {  // a tile is 64 image rows: the 64-rows-a-pass kernel, one expert slab per tile
        GemvWArgs wa{};
        wa.seg[0] = GemvWSeg{w->dev, out_dev, (int)w->dims.n, (int)w->dims.row_tiles, 0, 1, (int)((w->dims.units + 1) / 2 * 2)};
        wa.nseg = 1;
        wa.m = (int)p.perm_len;  // bound of the sorted rows; every perm entry is a token below m <= perm_len
        wa.pair_rows = xk == 0 ? 1 : 0;
        wa.units = (int)w->dims.units;
        wa.k_steps = (int)(p.gemm.k_pad / 64);
        wa.xh = (uint8_t *)gws + p.gemm.fac_bytes;
        wa.rowfac = (const float *)gws;
        wa.tile_expert = tile_expert;
        wa.perm = perm;
        wa.slab_bytes = w->dims.bytes;
        void *wparams[] = {&wa};
        return launch3(w->scheme == SCHEME_Q4_0 ? K_GEMVWG_Q4_0 : K_GEMVWG_Q8_0, (unsigned)((w->dims.row_tiles + 15) / 16),
                       (unsigned)(p.perm_len / p.group), 1, 512, 2 * 32768, s, wparams);
    }
    const Layout L = w->layout;
    GemmArgs a{};
    a.seg[0] = GemmSeg{w->dev, out_dev, (int)w->dims.n, (int)w->dims.row_tiles, 0};
    a.nseg = 1;
    a.xh = (uint8_t *)gws + p.gemm.fac_bytes;
    a.sxh = p.gemm.sxh_bytes ? (uint8_t *)gws + p.gemm.fac_bytes + p.gemm.xh_bytes : nullptr;
    a.m_rows = (int)p.gemm.m_rows;
    a.m_out = (int)p.perm_len;  // bound of the sorted rows; every perm entry is a token below m <= perm_len
    a.k_pad = (int)p.gemm.k_pad;
    a.units = (int)w->dims.units;
    a.pair_rows = xk == 0 ? 1 : 0;
    a.steps_per_split = (int)w->dims.units * (L.unit_k / 64);
    a.split_out = 0;
    a.sc_off = w->sc_off();
    a.rowfac = (const float *)gws;
    a.tile_expert = tile_expert;
    a.perm = perm;
    a.slab_bytes = w->dims.bytes;
    void *params[] = {&a};
    const KernelId id = w->scheme == SCHEME_Q4K    ? K_GEMM64G_Q4_K
                        : w->scheme == SCHEME_Q4_0 ? K_GEMM64G_Q4_0
                        : w->scheme == SCHEME_Q6K  ? K_GEMM64G_Q6_K
                        : w->scheme == SCHEME_Q5K  ? K_GEMM64G_Q5_K
                        : w->scheme == SCHEME_Q8K  ? K_GEMM64G_Q8_K
                        : w->scheme == SCHEME_Q2K  ? K_GEMM64G_Q2_K
                                                   : K_GEMM64G_Q8_0;
    const unsigned gx = (unsigned)((w->dims.row_tiles * 16 + 127) / 128), gy = (unsigned)(p.perm_len / p.group);
    return launch3(id, gx, gy, 1, 512, 3 * 24 * 1024, s, params);
}

int rlx_mi355x_gguf_grouped_matmul_bt(const void *x_dev, int x_dtype, const rlx_qweight *w, const float *expert_idx_dev,
                                      float *out_dev, int64_t m, void *stream) {
    using namespace rlx;
    if (!x_dev || !w || !expert_idx_dev || !out_dev || m <= 0) {
        set_error("gguf_grouped_matmul_bt: null argument or m=%lld", (long long)m);
        return RLX_ERR_INVALID;
    }
    const int xk = x_kind(x_dtype);
    if (xk < 0) {
        set_error("gguf_grouped_matmul_bt: activation dtype %d is not F32 / BF16 / F16", x_dtype);
        return RLX_ERR_UNSUPPORTED;
    }
    RLX_TRY(runtime_init());
    // Every token is its own one-row matmul against the slab its index names: up to eight tokens per launch, each
    // a segment of the decode kernel. Tokens that share an expert stream its slab again (once from HBM, then from L2).
    const size_t esz = xk == 0 ? 4 : 2;
    for (int64_t t0 = 0; t0 < m; t0 += GEMV_MAX_SEG) {
        const int c = (int)std::min<int64_t>(GEMV_MAX_SEG, m - t0);
        const void *xs[GEMV_MAX_SEG];
        const rlx_qweight *ws[GEMV_MAX_SEG];
        float *outs[GEMV_MAX_SEG];
        for (int i = 0; i < c; i++) {
            xs[i] = (const uint8_t *)x_dev + (size_t)(t0 + i) * w->dims.k * esz;
            ws[i] = w;
            outs[i] = out_dev + (size_t)(t0 + i) * w->dims.n;
        }
        RLX_TRY(launch_gemv(xs, xk, ws, outs, c, 1, (hipStream_t)stream, expert_idx_dev + t0));
    }
    return RLX_OK;
}

// Column layout (channels along the last axis, 16-byte aligned rows): pass A and pass B use their own row blocking.
struct FqColPlan {
    bool col;
    unsigned gx, gy_absmax, gy_apply;
    int rpb_absmax, rpb_apply;
};
static FqColPlan fq_col_plan(int64_t len, int64_t chan_dim, int64_t inner) {
    FqColPlan p{};
    p.col = inner == 1 && chan_dim >= 4 && chan_dim % 4 == 0 && len % chan_dim == 0 && len > 0;
    if (!p.col) return p;
    p.gx = (unsigned)((chan_dim / 4 + 255) / 256);
    const int64_t rows = len / chan_dim;
    auto block = [&](int64_t groups, int64_t min_rows, unsigned *gy, int *rpb) {
        int64_t want = std::max<int64_t>(1, groups / p.gx);
        int64_t r = std::max<int64_t>(min_rows, (rows + want - 1) / want);
        *rpb = (int)r;
        *gy = (unsigned)((rows + r - 1) / r);
    };
    block(1024, 16, &p.gy_absmax, &p.rpb_absmax);  // read only: a thousand workgroups keep enough loads in flight
    block(2048, 16, &p.gy_apply, &p.rpb_apply);
    return p;
}

size_t rlx_mi355x_fake_quantize_scratch_bytes(int64_t len, int64_t chan_dim, int64_t inner) {
    if (chan_dim < 1) chan_dim = 1;
    if (inner < 1) inner = 1;
    const FqColPlan p = fq_col_plan(len, chan_dim, inner);
    return (size_t)chan_dim * 8 + (p.col ? (size_t)p.gy_absmax * chan_dim * 4 + 256 : 0);  // maxima, scales; column layout: partial maxima, the largest scale
}

// img_ws != nullptr: column layout only; the apply pass also writes the prefill image of the result (and its per-row
// factors) into img_ws, and skips the f32 tensor when out_dev is null.
static int fake_quantize_impl(const float *x_dev, float *out_dev, int8_t *codes_dev, int64_t len, int64_t chan_dim,
                              int64_t inner, int bits, int scale_mode, float ema_decay, float *state_dev,
                              int round_mode, void *scratch_dev, void *stream, void *img_ws, size_t img_ws_bytes) {
    using namespace rlx;
    float q_max;
    switch (bits) {
    case 8: q_max = 127.0f; break;
    case 4: q_max = 7.0f; break;
    case 2: q_max = 1.0f; break;
    default:
        set_error("FakeQuantize: unsupported bits %d", bits);  // the reference panics with this text (thunk.rs:11179)
        return RLX_ERR_UNSUPPORTED;
    }
    if (chan_dim < 1) chan_dim = 1;
    if (inner < 1) inner = 1;
    if (!x_dev || (!out_dev && !img_ws) || !scratch_dev || len < 0 || scale_mode < 0 || scale_mode > 2) {
        set_error("FakeQuantize: null buffer, negative length or bad scale mode %d", scale_mode);
        return RLX_ERR_INVALID;
    }
    if (scale_mode != RLX_SCALE_PER_BATCH && !state_dev) {
        set_error("FakeQuantize: EMA / Fixed scale modes need the state tensor");  // "EMA needs state_off"
        return RLX_ERR_INVALID;
    }
    if (len == 0) return RLX_OK;
    hipStream_t s = (hipStream_t)stream;
    uint32_t *max_bits = (uint32_t *)scratch_dev;
    float *scale = (float *)scratch_dev + chan_dim;
    const FqColPlan plan = fq_col_plan(len, chan_dim, inner);
    // the scratch is sized for the column plan whether or not the pointers allow it, so alignment only picks kernels
    const bool col = plan.col && ((uintptr_t)x_dev % 16 == 0) && ((uintptr_t)out_dev % 16 == 0) &&
                     ((uintptr_t)scratch_dev % 16 == 0) && (!codes_dev || (uintptr_t)codes_dev % 8 == 0 || (!img_ws && (uintptr_t)codes_dev % 4 == 0));
    FqArgs a{x_dev, out_dev, codes_dev, max_bits, scale, state_dev, len, chan_dim, inner, q_max, ema_decay,
             scale_mode, round_mode, 0, nullptr, 0, nullptr, nullptr, 0, 0, 1, nullptr, nullptr};
    GemmPlan ip{};
    if (img_ws) {
        const int64_t m = chan_dim > 0 ? len / chan_dim : 0;
        ip = gemm_plan(SCHEME_Q8_0, XK_CODES, m, chan_dim);  // one image row of integer codes per row, plus the column scales
        if (!col || chan_dim % 8 != 0 || (uintptr_t)img_ws % 16 != 0 || img_ws_bytes < ip.image_end()) {
            set_error("FakeQuantize: the prefill image needs column channels in multiples of 8, 16-byte aligned buffers and %zu bytes of workspace",
                      ip.image_end());
            return RLX_ERR_INVALID;
        }
    }
    void *params[] = {&a};
    if (scale_mode != RLX_SCALE_FIXED) {
        if (col) {
            a.partial = (float *)scratch_dev + 2 * chan_dim;
            a.parts = (int)plan.gy_absmax;
            a.smax_bits = (uint32_t *)(a.partial + (size_t)plan.gy_absmax * chan_dim);
            a.rows_per_block = plan.rpb_absmax;
            RLX_TRY(launch(K_FQ_COL_ABSMAX, plan.gx, plan.gy_absmax, 256, 0, s, params));
        } else {
            RLX_TRY(rlx_mi355x_memset_u32(max_bits, 0, (size_t)chan_dim, stream));
            if (inner >= 256 && len % inner == 0 && len / inner <= 0x7FFFFFFF) {
                // one workgroup per contiguous run of `inner` elements, long runs split into parts of >= 16K elements
                unsigned bx = inner >= 4096 ? 1024 : 256;
                unsigned parts = (unsigned)std::min<int64_t>(1024, std::max<int64_t>(1, inner / 16384));
                a.rows_per_block = (int)((inner + parts - 1) / parts);
                RLX_TRY(launch(K_FQ_SEG_ABSMAX, (unsigned)(len / inner), parts, bx, 0, s, params));
            } else {
                int64_t threads = (len + 31) / 32;
                RLX_TRY(launch(K_FQ_FLAT_ABSMAX, (unsigned)((threads + 255) / 256), 1, 256, 0, s, params));
            }
        }
    }
    if (a.partial) RLX_TRY(launch(K_FQ_SCALE_PARTS, (unsigned)((chan_dim + 63) / 64), 1, 1024, 0, s, params));
    else RLX_TRY(launch(K_FQ_SCALE, (unsigned)((chan_dim + 255) / 256), 1, 256, 0, s, params));
    if (img_ws) {
        a.img = (uint8_t *)img_ws + ip.fac_bytes + ip.cs_bytes;
        a.rowfac = (float *)img_ws;
        a.colscale = (float *)((uint8_t *)img_ws + ip.fac_bytes);
        a.k_pad = (int)ip.k_pad;
        a.m_rows = (int)ip.m_rows;
        a.write_out = out_dev ? 1 : 0;
        const unsigned gx = (unsigned)((ip.k_pad + 255) / 256);
        // about 4096 workgroups (2048: 2 us slower, 1024: 7 us slower on [8192, 4096])
        const int64_t want = std::max<int64_t>(1, 4096 / gx), lrows = ip.m_rows;  // image rows, padding included (a multiple of 256)
        a.rows_per_block = (int)std::max<int64_t>(32, ((lrows + want - 1) / want + 31) / 32 * 32);
        RLX_TRY(launch(K_FQ_COL_APPLY_IMG, gx, (unsigned)((lrows + a.rows_per_block - 1) / a.rows_per_block), 256, 0, s, params));
    } else if (col) {
        a.rows_per_block = plan.rpb_apply;
        RLX_TRY(launch(K_FQ_COL_APPLY, plan.gx, plan.gy_apply, 256, 0, s, params));
    } else {
        bool v4 = inner % 4 == 0 && len % 4 == 0 && ((uintptr_t)x_dev % 16 == 0) && ((uintptr_t)out_dev % 16 == 0) &&
                  (!codes_dev || (uintptr_t)codes_dev % 4 == 0);
        int64_t work = v4 ? len / 4 : len;
        unsigned blocks = (unsigned)std::min<int64_t>((work + 255) / 256, 256 * 16);
        RLX_TRY(launch(v4 ? K_FQ_FLAT4_APPLY : K_FQ_FLAT_APPLY, blocks, 1, 256, 0, s, params));
    }
    return RLX_OK;
}

int rlx_mi355x_fake_quantize(const float *x_dev, float *out_dev, int8_t *codes_dev, int64_t len, int64_t chan_dim,
                             int64_t inner, int bits, int scale_mode, float ema_decay, float *state_dev,
                             int round_mode, void *scratch_dev, void *stream) {
    return fake_quantize_impl(x_dev, out_dev, codes_dev, len, chan_dim, inner, bits, scale_mode, ema_decay, state_dev, round_mode,
                              scratch_dev, stream, nullptr, 0);
}

int rlx_mi355x_fake_quantize_image(const float *x_dev, float *out_dev, int8_t *codes_dev, int64_t m, int64_t k, int bits,
                                   int scale_mode, float ema_decay, float *state_dev, int round_mode, void *scratch_dev,
                                   void *workspace, size_t workspace_bytes, void *stream) {
    if (!workspace || m <= 0 || k <= 0) {
        rlx::set_error("fake_quantize_image: null workspace or empty tensor");
        return RLX_ERR_INVALID;
    }
    return fake_quantize_impl(x_dev, out_dev, codes_dev, m * k, k, 1, bits, scale_mode, ema_decay, state_dev, round_mode, scratch_dev,
                              stream, workspace, workspace_bytes);
}

}  // extern "C"
