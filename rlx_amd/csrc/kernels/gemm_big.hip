// Prefill matmul for many rows: out[m, n] = x[m, k] . W[n, k]^T, replacing rlx_cpu::gguf_matmul::gguf_matmul_bt
// (rlx-cpu/src/gguf_matmul.rs:40-95) where the 256 x 256 tiles of the result fill the chip. A is the operand image of the
// prefill path (rlx_xprep, or the code image a FakeQuantize writes; 32 KB per 256 rows x 64 columns). W is read in one of
// two forms: packed Q4_0 / Q8_0 units, decoded to fl16(d * code) in registers and written to LDS by the workgroup that
// multiplies them (rlx_gemm_big_{q4_0,q8_0}), or ready binary16 images (rlx_gemm_big_f16w: rlx_wscale_*'s, 16 KB per 128
// rows x 64 columns, the second half of the reference's FakeQuantize -> DequantMatMul chain,
// rlx-cpu/src/thunk.rs:11242-11251 then rlx-cpu/src/gguf_matmul.rs:81-94).
//
// Four waves, one per SIMD, own 128 x 128 of the 256 x 256 tile each (256 accumulator registers): sixteen fragment reads feed 64
// matrix instructions. K advances in 32-column quanta through a ring of LDS slots that buffer loads fill directly; one barrier per
// quantum. What bounds it: on [8192, 4096] x [4096, 4096] ready images the loop takes 160 K clocks a tile, 19.5 per matrix instruction (16
// and a bubble of 2 at best), and the way in and out 20 K: 159 us at the 2.3 GHz it runs at on zeros, 1.73 PFLOP/s. On drawn data the
// chip draws more and clocks lower: 206 us for one launch after a pause (1.33 PFLOP/s), 199 in a row of a thousand (1.38), 205 - 270
// for those of a row of sixteen or sixty-four, while the clock settles. With packed weights decoded in it the loop issues for 26.6
// clocks per matrix instruction, which is what bounds it then. 16 x 16 x 32 instructions read and write half the accumulator bits per
// product of 32 x 32 x 16 ones: 210 us against 229 (and 232 for eight waves of 128 x 64 on 32 x 32 x 16, the kernel before).
// An XCD-wise tile order and a ring without address arithmetic (four slots, depth two) measured the same or 2 % slower.
//
// Decoding packed weights here costs what writing them out as images first would (about 10 % of the kernel), without 2 bytes per weight
// of workspace. A wave issues its own vector instructions under its matrix instructions: 16 x 16 x 32 alone takes 18.1 clocks, with one
// vector instruction behind each 20.1, two 20.6, three 25.1, four 29.1. Layer of 1111 f32 tokens (Llama-3-8B, Q4_0): 1280 -> 1074 - 1118 us
// with an epilogue through LDS, 6 % less without.
#include "common.h"

namespace rlx {

constexpr int BIG_STAGE_A = 32768;         // operand image of A: 256 rows x 64 columns
constexpr int BIG_SLOT = 32768;            // ring slot: a 32-column quantum, 16 KB of A then 16 KB of B
constexpr int BIG_SLOTS = 5;               // all of the CU's 160 KB
constexpr int BIG_MAX_SEG = 4;
constexpr float BIG_LO_SCALE = 2048.0f;

struct GemmBigSeg {
    const uint8_t *w;  // packed units, or images [256-row tile][2][steps][16 KB]
    float *out;        // [m_out][n]
    int n, row_tiles;  // logical columns of the result; 16-row tiles of the device layout
    int tile_begin;    // first 256-column tile of this matrix
};
struct GemmBigArgs {
    GemmBigSeg seg[BIG_MAX_SEG];
    int nseg;
    const uint8_t *a_img;  // [tiles_m][a_steps][32 KB]
    const float *rowfac;   // [m_out][2]: row i of the result is multiplied by rowfac[2 i + 1]
    float *part;           // [workgroup][2][rows of a tile][256]: pieces of tiles that are shared between workgroups
    int m_out, tiles_m, tiles_n, a_steps;
    int quads;             // K in 128-column units
    int pair_rows;         // 1: image rows 2i, 2i+1 are hi / lo*2048 of logical row i (f32 activations)
};

// Work is a line of tiles_m * tiles_n * quads items (a tile's K items next to each other, the M tiles of a column of tiles
// next); workgroup g of G takes items [g T / G, (g + 1) T / G). With G = the number of tiles that is a tile each.
__device__ __forceinline__ long long big_begin(long long total, int groups, int g) { return total * g / groups; }

template <int SCHEME>
__device__ __forceinline__ void gemm_big_body(const GemmBigArgs &a) {
    constexpr bool IMG = SCHEME == SCHEME_F16W;
    constexpr Layout L = IMG ? Layout{64, 0, 0, 0, 0} : layout_of(SCHEME);
    constexpr bool Q8 = SCHEME == SCHEME_Q8_0;
    extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave >> 1, wn = wave & 1;
    const int lr = lane & 15, lg = lane >> 4;
    typedef __attribute__((address_space(3))) void *lds_ptr;

    // Fragment addresses: register tile t of 16 rows, 8-column chunk c = 4 * (quantum & 1) + lg of the 64-column image.
    int a_rd[2][2], b_rd[2][2], b_wr[2];  // [quantum parity][tile parity]
#pragma unroll
    for (int p = 0; p < 2; p++) {
        const int c = 4 * p + lg, at = (lg & 1) * 512;
#pragma unroll
        for (int t = 0; t < 2; t++) {
            const int slot = (((16 * t + lr) ^ c) & 31) * 16 + at;
            a_rd[p][t] = ((lg >> 1) * 8 + 4 * wm) * 1024 + slot;
            b_rd[p][t] = 16384 + wn * 8192 + (lg >> 1) * 4096 + slot;
        }
        // this wave decodes rows 64 wave .. + 63 of the tile: 16-row tile i goes to sub-tile (2 wave + i / 2) & 3 of half wave / 2
        b_wr[p] = 16384 + (wave >> 1) * 8192 + ((lg >> 1) * 4 + (wave & 1) * 2) * 1024 + ((lr ^ c) & 15) * 16 + at;
    }

    const long long total = (long long)a.tiles_m * a.tiles_n * a.quads;
    long long item = big_begin(total, gridDim.x, blockIdx.x);
    const long long item_end = big_begin(total, gridDim.x, blockIdx.x + 1);
    while (item < item_end) {
        const int tile = (int)(item / a.quads), k0 = (int)(item - (long long)tile * a.quads);
        const int k1 = (int)min((long long)a.quads, k0 + (item_end - item));
        item += k1 - k0;
        const int by = tile % a.tiles_m, nt = tile / a.tiles_m;
        int si = 0;
#pragma unroll
        for (int i = 1; i < BIG_MAX_SEG; i++)
            if (i < a.nseg && nt >= a.seg[i].tile_begin) si = i;
        const GemmBigSeg sg = a.seg[si];
        const int bx = nt - sg.tile_begin;
        const int nq = 4 * (k1 - k0), q0 = 4 * k0, last = 4 * k1 - 1;

        const uint8_t *a_base = a.a_img + (long long)by * a.a_steps * BIG_STAGE_A;
        const __amdgpu_buffer_rsrc_t a_rsrc = __builtin_amdgcn_make_buffer_rsrc((void *)a_base, 0, 0x7FFFFFFF, 0x00020000);
        const uint8_t *b_base = IMG ? sg.w + (long long)(2 * bx) * a.a_steps * 16384 : sg.w + (long long)bx * 16 * a.quads * L.unit_bytes;
        const __amdgpu_buffer_rsrc_t b_rsrc = __builtin_amdgcn_make_buffer_rsrc((void *)b_base, 0, 0x7FFFFFFF, 0x00020000);
        // quantum i of this piece into its ring slot; past the end the last one again (never read), so that the number of
        // loads in flight is the same in every iteration
        auto fill_one = [&](int i, int slot, int j) {  // the j-th of this wave's 1 KB chunks: four of A, then (images) four of B
            const int q = min(q0 + i, last), chunk = wave + 4 * (j < 4 ? j : j & 1), h = (j >> 1) & 1;
            uint8_t *d = smem + slot + chunk * 1024;
            if (j < 4) __builtin_amdgcn_raw_ptr_buffer_load_lds(a_rsrc, (lds_ptr)d, 16, lane * 16, q * 16384 + chunk * 1024, 0, 0);
            else __builtin_amdgcn_raw_ptr_buffer_load_lds(b_rsrc, (lds_ptr)(d + 16384 + h * 8192), 16, lane * 16, h * a.a_steps * 16384 + q * 8192 + chunk * 1024, 0, 0);
        };
        // Packed W: the wave's four 16-row tiles, one lane slot each. A set holds half a unit, i.e. two quanta (two words of a Q4_0
        // slot, four of a Q8_0 slot); wd[0] / wd[1] the scales of the unit being decoded / of the next one.
        uint32_t wq[2][4][Q8 ? 4 : 2];
        uint2_t wd[2][4];
        int w_off[4];
        uint32_t w_keep[4];
        if constexpr (!IMG) {
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const int t16 = bx * 16 + wave * 4 + i;
                w_keep[i] = t16 < sg.row_tiles ? 0xFFFFFFFFu : 0u;  // a tile past the matrix reads the last one and decodes to zeros
                w_off[i] = (min(t16, sg.row_tiles - 1) - bx * 16) * a.quads * L.unit_bytes;
            }
        }
        auto fetch_w = [&](int unit, int h, int dset = 1) {  // half h of a unit of this piece into set h, with half 0 the unit's scales
            const int u = min(k0 + unit, k1 - 1) * L.unit_bytes;
#pragma unroll
            for (int i = 0; i < 4; i++) {
                if constexpr (Q8) {
                    const uint4_t v = __builtin_amdgcn_raw_buffer_load_b128(b_rsrc, lane * 16, w_off[i] + u + h * 1024, 0);
#pragma unroll
                    for (int e = 0; e < 4; e++) wq[h][i][e] = v[e];
                } else {
                    const uint2_t v = __builtin_amdgcn_raw_buffer_load_b64(b_rsrc, lane * 16 + h * 8, w_off[i] + u, 0);
                    wq[h][i][0] = v[0];
                    wq[h][i][1] = v[1];
                }
                if (h == 0) wd[dset][i] = __builtin_amdgcn_raw_buffer_load_b64(b_rsrc, lr * 8, w_off[i] + u + L.quant_bytes, 0);
            }
        };
        // One of 28 parts of decoding quantum t of a unit into the ring slot: for each of the four 16-row tiles the scale and six parts of
        // two to four vector instructions (columns 0 - 3, then 4 - 7 of every eight: the codes, the offset, the product), then the store.
        Frag f;
        half2_t d2;
        auto decode = [&](int t, int part, int slot) {
            const int i = part / 7, s = part % 7;
            if (s == 6) {  // row tile i: sub-tile i / 2, slot rows 16 (i & 1) .. + 15
                *(uint4_t *)(smem + slot + b_wr[t & 1] + (i >> 1) * 1024 + (i & 1) * 256) = f.u4;
                return;
            }
            const int h = s / 3;
            half2_t *v = f.h2 + 2 * h;
            if (s == 0) {
                const uint32_t dw = wd[0][i][t >> 1] & w_keep[i];
                d2 = as_half2(__builtin_amdgcn_perm(dw, dw, (t & 1) ? 0x07060706u : 0x05040504u));
            }
            if (s % 3 == 0) {
                if constexpr (Q8) q8_magic(wq[t >> 1][i][2 * (t & 1) + h], v);
                else q4_magic(h ? wq[t >> 1][i][t & 1] >> 8 : wq[t >> 1][i][t & 1], v);
            } else if (s % 3 == 1) {
                if constexpr (Q8) q8_signed(v);
                else q4_signed<8>(v);
            } else {
                v[0] = v[0] * d2;
                v[1] = v[1] * d2;
            }
        };

        float4_t acc[8][8];
#pragma unroll
        for (int i = 0; i < 8; i++)
#pragma unroll
            for (int j = 0; j < 8; j++) acc[i][j] = float4_t{0.f, 0.f, 0.f, 0.f};
        Frag fa[8], fb[2][8];  // A: one set, see below; B: [quantum parity]
        auto load_a = [&](int slot, int p, int i) { fa[i].u4 = *(const uint4_t *)(smem + slot + a_rd[p][i & 1] + (i >> 1) * 1024); };
        auto load_b = [&](int slot, int p, int i) { fb[p][i].u4 = *(const uint4_t *)(smem + slot + b_rd[p][i & 1] + (i >> 1) * 1024); };

        int s0 = 0, s1 = BIG_SLOT, s2 = 2 * BIG_SLOT, s4 = 4 * BIG_SLOT;  // ring slots of quanta q, q + 1, q + 2, q + 4
        auto turn = [&]() {
            s4 = s0;
            s0 = s1;
            s1 = s2;
            s2 = s2 == (BIG_SLOTS - 1) * BIG_SLOT ? 0 : s2 + BIG_SLOT;
        };
        if constexpr (!IMG) {
            fetch_w(0, 0, 0);
            fetch_w(0, 1);
        }
#pragma unroll
        for (int i = 0; i < BIG_SLOTS - 1; i++)
#pragma unroll
            for (int j = 0; j < (IMG ? 8 : 4); j++) fill_one(i, i * BIG_SLOT, j);
        if constexpr (!IMG) {
#pragma unroll
            for (int x = 0; x < 56; x++) decode(x / 28, x % 28, x / 28 * BIG_SLOT);
            fetch_w(1, 0);
        }
        __builtin_amdgcn_sched_barrier(0);
        __builtin_amdgcn_s_waitcnt(IMG ? 0x4078 : 0x007C);  // quantum 0 has landed, three more are on their way: vmcnt(24) / vmcnt(12), lgkmcnt(0)
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int x = 0; x < 8; x++) load_b(0, 0, x);
#pragma unroll
        for (int x = 0; x < 4; x++) load_a(0, 0, x);

        // One quantum: 64 matrix instructions, row r of register tiles at a time. On entry its B fragments and rows 0 - 3 of A are in
        // registers (or on their way). The barrier says that quantum i + 1 is complete in LDS and that every wave is done with
        // quantum i - 1, whose slot takes i + 4. Rows 4 - 7 of A are read while rows 0 - 3 are multiplied and the next quantum's
        // rows 0 - 3 after that, so one set of registers serves both; only B has two.
        auto quantum = [&](int i, int ph) {  // i = quantum of the piece, ph = i & 3, compile-time
            __builtin_amdgcn_sched_barrier(0);
            asm volatile("" ::: "memory");
            // vmcnt: quanta i + 2 and i + 3 may still be on their way (packed W loads between them only make the wait longer);
            // lgkmcnt: everything up to the two fragment reads issued last, the stores of decoded W among it
            __builtin_amdgcn_s_waitcnt(IMG ? 0x4270 : 0x0278);  // vmcnt(16) / vmcnt(8), lgkmcnt(2)
            __builtin_amdgcn_s_barrier();
            asm volatile("" ::: "memory");
            __builtin_amdgcn_sched_barrier(0);
            // 32 steps of two matrix instructions, the rest of the work spread under them: the vector instructions of this wave
            // issue while its matrix instructions run (two per 16 x 16 x 32 one cost 2.5 clocks on top of its 18, every further one 4 - 5), but
            // only if they stand between them. The fences keep the compiler from gathering them in front.
#pragma unroll
            for (int st = 0; st < 32; st++) {
                const int e = st >> 1;
                if (!(st & 1)) {
                    if (e < 4) load_a(s0, ph & 1, 4 + e);
                    else if (e < 12) load_b(s1, (ph + 1) & 1, e - 4);
                    else load_a(s1, (ph + 1) & 1, e - 12);
                    if (IMG) {
                        if (e < 8) fill_one(i + 4, s4, e);
                    }
                } else if (!IMG && e < 4) {
                    fill_one(i + 4, s4, e);
                }
                if constexpr (!IMG)
                    if (st < 28) decode((ph + 2) & 3, st, s2);  // quantum i + 2
                const int r = st >> 2;
#pragma unroll
                for (int jj = 0; jj < 2; jj++) {
                    const int x = (st & 3) * 2 + jj, j = (r & 1) ? 7 - x : x;
                    acc[r][j] = mfma16(fb[ph & 1][j], fa[r], acc[r][j]);  // rows of the product: columns of the result
                }
                __builtin_amdgcn_sched_barrier(0);
            }
            if constexpr (!IMG) {
                if (ph == 1) {  // a unit's second half has just been decoded
#pragma unroll
                    for (int j = 0; j < 4; j++) wd[0][j] = wd[1][j];
                    fetch_w((i >> 2) + 1, 1);
                }
                if (ph == 3) fetch_w((i >> 2) + 2, 0);
            }
            turn();
        };
        for (int i = 0; i < nq; i += 4) {
            quantum(i, 0);
            quantum(i + 1, 1);
            quantum(i + 2, 2);
            quantum(i + 3, 3);
        }
        // The sums stay in accumulation registers until their row is stored (here and below): left to itself the allocator moves them
        // between the register files inside the loop, some four hundred moves a quad, and spills around the epilogue.
#pragma unroll
        for (int i = 0; i < 8; i++)
#pragma unroll
            for (int j = 0; j < 8; j++) asm volatile("" : "+a"(acc[i][j]));
        __builtin_amdgcn_s_waitcnt(0);
        __syncthreads();  // nothing is on its way into LDS any more

        // Epilogue. W is the first operand of the products, so register r of tile (i, j) is row 16 i + lr, column 16 j + 4 lg + r of the
        // wave's quarter: a lane holds four neighbouring columns and stores them as they are, four lanes 64 bytes of a row. With
        // the rows in the registers the wave had to turn its quarter around in LDS first: 41 K clocks of the 205 K of a tile of
        // [8192, 4096] x [4096, 4096], 17 K now; f32 rows 30 K and 12.5 K (no stores at all: 4 K). A lower clock takes some of it back:
        // 277 -> 262 us in a row of a few dozen launches, 519 -> 506 on [2222 image rows, 4096] x [28672, 4096]. The rows' factors come through LDS.
        const int rows = a.pair_rows ? 128 : 256;
        float *fac_s = (float *)smem;
        if (tid < rows) {
            const int row = by * rows + tid;
            fac_s[tid] = row < a.m_out ? a.rowfac[2 * row + 1] : 0.f;
        }
        __syncthreads();
        const bool piece = k0 > 0 || k1 < a.quads;
        float *dst = piece ? a.part + ((long long)blockIdx.x * 2 + (k0 > 0 ? 0 : 1)) * rows * 256 : sg.out + ((long long)by * rows * sg.n + bx * 256);
        const int ld = piece ? 256 : sg.n;
        const int row_lim = piece ? rows : min(rows, a.m_out - by * rows), col_lim = piece ? 256 : min(256, sg.n - bx * 256);
        // One store whatever the row's alignment (a 16-byte store needs no more than that of its words). In four, rows of odd length took
        // 277 us instead of 236 ([2048, 4096] bf16 x 14335 columns; 490 and 430 for 8192 code rows x 8191).
        typedef float4_t __attribute__((aligned(4))) float4_words_t;
        auto store4 = [&](float *o, int col, float4_t v) {
            if (col + 4 <= col_lim) {
                *(float4_words_t *)(o + col) = v;
            } else {
#pragma unroll
                for (int e = 0; e < 3; e++)
                    if (col + e < col_lim) o[col + e] = v[e];
            }
        };
        const bool odd = lr & 1;
#pragma unroll
        for (int i = 0; i < 8; i++) {
            __builtin_amdgcn_sched_barrier(0);
            const int t0 = wm * 128 + i * 16 + lr, row = a.pair_rows ? t0 >> 1 : t0;  // image row, output row
            const float fac = fac_s[row];
            float *o = dst + (long long)row * ld;
#pragma unroll
            for (int j = 0; j < 8; j++) asm volatile("" : "+a"(acc[i][j]));
            if (a.pair_rows) {
                // neighbouring lanes hold the leading and the residual sums of one row: the even lane finishes tile j, the odd one j + 1
#pragma unroll
                for (int j = 0; j < 8; j += 2) {
                    float4_t v;
#pragma unroll
                    for (int r = 0; r < 4; r++) {
                        const float keep = odd ? acc[i][j + 1][r] : acc[i][j][r], give = odd ? acc[i][j][r] : acc[i][j + 1][r];
                        const float got = __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, give), 0xB1, 0xF, 0xF, true));
                        v[r] = ((odd ? got : keep) + (odd ? keep : got) * (1.0f / BIG_LO_SCALE)) * fac;
                    }
                    if (row < row_lim) store4(o, wn * 128 + (j + (odd ? 1 : 0)) * 16 + lg * 4, v);
                }
            } else if (row < row_lim) {
#pragma unroll
                for (int j = 0; j < 8; j++) {
                    float4_t v;
#pragma unroll
                    for (int r = 0; r < 4; r++) v[r] = acc[i][j][r] * fac;
                    store4(o, wn * 128 + j * 16 + lg * 4, v);
                }
            }
        }
        __syncthreads();  // the factors are read before the next piece overwrites them
    }
}

// A tile that several workgroups share: its pieces, in ascending K, added into the output. Grid: x = tile, y = rows / 16.
__device__ __forceinline__ void big_reduce_body(const GemmBigArgs &a, int groups) {
    const long long total = (long long)a.tiles_m * a.tiles_n * a.quads;
    const int tile = blockIdx.x;
    const long long u0 = (long long)tile * a.quads;
    const int g0 = (int)(((u0 + 1) * groups - 1) / total), g1 = (int)(((u0 + a.quads) * groups - 1) / total);  // owners of the first and last item
    if (g0 == g1) return;  // written whole
    const int rows = a.pair_rows ? 128 : 256;
    const int by = tile % a.tiles_m, nt = tile / a.tiles_m;
    int si = 0;
#pragma unroll
    for (int i = 1; i < BIG_MAX_SEG; i++)
        if (i < a.nseg && nt >= a.seg[i].tile_begin) si = i;
    const GemmBigSeg sg = a.seg[si];
    const int bx = nt - sg.tile_begin;
    const int col = bx * 256 + (threadIdx.x & 63) * 4;
    const bool wide = (sg.n & 3) == 0 && ((uintptr_t)sg.out & 15) == 0;
#pragma unroll
    for (int rr = 0; rr < 4; rr++) {
        const int trow = blockIdx.y * 16 + (threadIdx.x >> 6) * 4 + rr, row = by * rows + trow;
        if (row >= a.m_out || col >= sg.n) continue;
        float4_t v = {0.f, 0.f, 0.f, 0.f};
        for (int g = g0; g <= g1; g++) {
            // only the owner of the first item has the head of the tile (slot 1), the others begin inside it (slot 0)
            const float *p = a.part + ((long long)g * 2 + (g == g0 ? 1 : 0)) * rows * 256 + trow * 256 + (threadIdx.x & 63) * 4;
            const float4_t x = __builtin_nontemporal_load((const float4_t *)p);
            v = g == g0 ? x : v + x;
        }
        float *o = sg.out + (long long)row * sg.n + col;
        if (wide) __builtin_nontemporal_store(v, (float4_t *)o);
        else
#pragma unroll
            for (int e = 0; e < 4; e++)
                if (col + e < sg.n) o[e] = v[e];
    }
}

}  // namespace rlx

extern "C" __global__ __launch_bounds__(256, 1) void rlx_gemm_big_f16w(rlx::GemmBigArgs a) { rlx::gemm_big_body<rlx::SCHEME_F16W>(a); }
extern "C" __global__ __launch_bounds__(256, 1) void rlx_gemm_big_q4_0(rlx::GemmBigArgs a) { rlx::gemm_big_body<rlx::SCHEME_Q4_0>(a); }
extern "C" __global__ __launch_bounds__(256, 1) void rlx_gemm_big_q8_0(rlx::GemmBigArgs a) { rlx::gemm_big_body<rlx::SCHEME_Q8_0>(a); }
extern "C" __global__ __launch_bounds__(256) void rlx_gemm_big_reduce(rlx::GemmBigArgs a, int groups) { rlx::big_reduce_body(a, groups); }
