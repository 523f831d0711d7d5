// mmq_q80.hip — batched mat-mul (2 columns and up) for Q8_0 weights on the gfx950 INTEGER matrix cores.
//
// ggml-cpu's ggml_vec_dot_q8_0_q8_0 quantises the activations to Q8_0 as well and sums,
// per 32-value block, sumi * (d_w * d_x) in f32.  A block is exactly the K extent of v_mfma_i32_32x32x32_i8, so one MFMA
// with a zero accumulator yields the 32x32 integer block sums, and the f32 scale-accumulate follows at once — there is no
// super-block to amortise it over, which makes these kernels VALU-bound: 3 VALU per output and block up to 32 columns (convert, d_w * d_x,
// fused multiply-add), 2 in the column kernel above that (the factors come from the matrix core), 4 with the 128 x 128 tiles.
//
// The first two take their operands straight from global memory into the MFMA's registers: the weights from their panel copy
// (repack.hip: k_repack_q80_panels; or, without one, from the 2-byte-aligned blocks), the activations in panel order
// (quantize.hip) — a wave-instruction reads 1 KB of consecutive bytes either way, no LDS tile and no barrier per K step.
// An output is a few partial sums, added in order, over interleaved chunks of four blocks: eight (chunk c to sum c mod 8) up to 32 columns, four (c mod 4) above.  Its bits depend on
// which side of that line the batch is, not on the number of columns otherwise, the kernel, the wave or the matrices that share the launch.
#include <algorithm>
#include <cstdlib>
#include <type_traits>

#include "dev_util.h"
#include "kernels.h"

namespace mi355x {

typedef float float16q __attribute__((ext_vector_type(16)));
typedef int int4q __attribute__((ext_vector_type(4)));
typedef int int16q __attribute__((ext_vector_type(16)));
typedef float float32q __attribute__((ext_vector_type(32)));

// ------------------------------------------------------------------------------------------------ 2 .. 32 columns
// (Two to eight took 2-, 4- and 8-column mat-vec passes, with launches of their own for norm, quantiser, SwiGLU, rotation and stores.  A step of TinyLlama, 2 / 4 / 8 sequences of 200 tokens:
// 1706 / 2265 / 2832 us; on this kernel, fused as the wider batches are, 1251 / 1253 / 1303; with 16 rows a workgroup where that is faster, below, 1117 / 1114 / 1158.)
// A -np decode step of a Q8_0 model (as 8-column mat-vec passes the weights streamed once per pass: 61 us per matrix of Llama-3-8B Q8_0 at 32 columns, a 16 ms
// step).  Here the WEIGHTS stream once: a workgroup owns 32 weight rows, its eight waves take the K range in interleaved chunks of four blocks (128 values:
// one cache line of every row), one v_mfma_i32_32x32x32_i8 per block gives the 32 x 32 integer block sums, and the f32 scale-accumulate follows
// (sumf += sumi * (d_w * d_x), ggml_vec_dot_q8_0_q8_0's expression, with the fused multiply-add its SIMD builds use).  Weight bytes go from global memory straight
// into the MFMA operand registers (a lane = a row and a 16-value half of the block); the activations' blocks (32 columns x K / 32 x 36 B: L2-resident) likewise; the
// 32 row scales of a block reach the 16 accumulator rows of a lane through a wave-private LDS line.  The eight partial tiles meet in LDS and are added in wave order.
struct mmq80s_mat {
    const uint8_t * W;   // the tensor (block layout), or its panel copy (repack.hip: k_repack_q80_panels) — template WP
    int64_t w_nb1;
    int N;
    int panel_end;       // workgroups [previous matrix's panel_end, panel_end) are this matrix's 32-row panels
    float * dst;
    int64_t dst_stride;
    const float * add;
    int64_t add_stride;
};
struct mmq80s_args {    // up to three matrices over the same activations in one launch (wq / wk / wv, gate / up: graph.cpp try_merge_q80_skinny)
    mmq80s_mat m[3];
    int K, M;
    const char * act;    // the activations in panel order (quantize.hip: k_quantize_q8_0<true>): 1152 B per block
};
typedef uint32_t __attribute__((ext_vector_type(4), aligned(2))) q80s_u32x4_a2;
typedef uint32_t __attribute__((ext_vector_type(4), aligned(4))) q80s_u32x4_a4;

// the sum v of column m and row n (of matrix mi), a row a lane: into the result, or (EPI) through the rotation into where its kind goes.  Every lane of a wave comes here.
// Q8: kinds 5 and 6 are among them; 32 lanes hold the rows of a block
template <bool EPI, bool Q8> __device__ __forceinline__ void q80s_result(const mmq80s_args & a, const mmq80s_mat & mt, const mmq_epi & epi, const int mi, const int m, const int n, float v) {
    if (!EPI && (m >= a.M || n >= mt.N)) return;
    const int tk = min(m, a.M - 1);
    if (mt.add) v += mt.add[(size_t) tk * mt.add_stride + n];
    if constexpr (!EPI) mt.dst[(size_t) m * mt.dst_stride + n] = v;
    else {
        const float partner = __shfl_xor(v, 1);  // the other element of the rotation pair
        const int kind = epi.kind[mi], head = n / epi.head_dim, dd = n - head * epi.head_dim;
        char * const out = epi.out[mi];
        float x = v;
        if ((kind < 3 || kind == 5) && dd < epi.n_dims) {
            const float2 t = *(const float2 *) (epi.tab + ((size_t) tk * (epi.n_dims >> 1) + (dd >> 1)) * 2);
            const float x0 = (dd & 1) ? partner : v, x1 = (dd & 1) ? v : partner;
            x = (dd & 1) ? x0 * t.y + x1 * t.x : x0 * t.x - x1 * t.y;
        }
        float amax = fabsf(x);
        if (Q8 && kind >= 5) {  // (uniform) the 32 rows are one Q8_0 block of the cache row
#pragma unroll
            for (int o = 1; o < 32; o <<= 1) amax = fmaxf(amax, __shfl_xor(amax, o));
        }
        if (m >= a.M) return;
        if (kind == 1) *(float *) (out + (int64_t) head * epi.nb1[mi] + (int64_t) m * epi.nb2[mi] + (int64_t) dd * 4) = x;
        else if (kind == 4) ((uint16_t *) out)[epi.v_idx[(int64_t) m * mt.N + n]] = f2h(x);
        else if (Q8 && kind >= 5) {
            const float d8 = amax / 127.0f, id8 = d8 != 0.0f ? 1.0f / d8 : 0.0f;
            char * const blk = out + epi.idx[m] * epi.nb1[mi] + (n >> 5) * 34;
            blk[2 + (n & 31)] = (char) (int) roundf(x * id8);
            if ((n & 31) == 0) *(uint16_t *) blk = f2h(d8);
        } else ((uint16_t *) (out + epi.idx[m] * epi.nb1[mi]))[n] = f2h(x);
    }
}

constexpr int Q80S_WV = 8;
// EPI: wq / wk / wv of a batch whose rotation and cache stores follow — done here, as in the K-quants' epilogue (mmq_skinny.hip; the arithmetic of k_rope_qk_store).  16 tokens of TinyLlama: the
// launch of its own cost 5.8 us a layer; this one takes 7.1 us (6.7 without the epilogue; 7.8 with a branch around the next chunk's loads, behind which each product waited for what had just been requested).
template <bool WP, bool EPI> __global__ void __launch_bounds__(Q80S_WV * 64, 2) k_mmq_q80_skinny(const mmq80s_args a, const mmq_epi epi) {
    __shared__ float dwl[Q80S_WV][4][32];       // a chunk's row scales, per wave
    __shared__ float red[Q80S_WV][16][65];      // the waves' partial tiles
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int fr = lane & 31, kg = lane >> 5;
    const int mi = (int) blockIdx.x < a.m[0].panel_end ? 0 : ((int) blockIdx.x < a.m[1].panel_end ? 1 : 2);  // (uniform)
    const mmq80s_mat & mt = a.m[mi];
    const int panel = (int) blockIdx.x - (mi ? a.m[mi - 1].panel_end : 0);
    const int n0 = panel * 32;
    const int nblk = a.K / 32, nchunk = nblk / 4;
    const uint8_t * wrow = WP ? mt.W + (size_t) panel * nchunk * 4352 : mt.W + (size_t) min(n0 + fr, mt.N - 1) * mt.w_nb1;
    const int colc = min(fr, a.M - 1);
    float C[16];
#pragma unroll
    for (int r = 0; r < 16; ++r) C[r] = 0.0f;
    int16q zi;
#pragma unroll
    for (int r = 0; r < 16; ++r) zi[r] = 0;

    int4q fa[4], fb[4], nfa[4], nfb[4];
    uint16_t dw[4], ndw[4];
    float dy[4], ndy[4];
    auto load_chunk = [&](const int c, int4q * A, int4q * B, uint16_t * dW, float * dY) {
#pragma unroll
        for (int b = 0; b < 4; ++b) {
            if constexpr (WP) {  // the chunk's tile of the panel copy: a wave-instruction reads 1 KB of consecutive bytes
                const uint8_t * tile = wrow + (size_t) c * 4352;
                A[b] = *(const int4q *) (tile + b * 1024 + kg * 512 + fr * 16);
                dW[b] = *(const uint16_t *) (tile + 4096 + b * 64 + fr * 2);
            } else {
                const uint8_t * blk = wrow + (size_t) (c * 4 + b) * 34;
                dW[b] = ld16(blk);
                A[b] = __builtin_bit_cast(int4q, *(const q80s_u32x4_a2 *) (blk + 2 + 16 * kg));
            }
            const char * yt = a.act + (size_t) (c * 4 + b) * 1152;
            B[b] = *(const int4q *) (yt + kg * 512 + colc * 16);
            dY[b] = *(const float *) (yt + 1024 + colc * 4);
        }
    };
    auto multiply = [&]() __attribute__((always_inline)) {
        // the block scales of the 32 rows: written by the row's first lane, read back as the 16 rows of this lane's accumulator registers
        if (kg == 0) {
#pragma unroll
            for (int b = 0; b < 4; ++b) dwl[wave][b][fr] = h2f(dw[b]);
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
        for (int b = 0; b < 4; ++b) {
            float x[16];
#pragma unroll
            for (int g4 = 0; g4 < 4; ++g4) {
                const float4 v = *(const float4 *) &dwl[wave][b][8 * g4 + 4 * kg];
                x[4 * g4] = v.x; x[4 * g4 + 1] = v.y; x[4 * g4 + 2] = v.z; x[4 * g4 + 3] = v.w;
            }
            const int16q s = __builtin_amdgcn_mfma_i32_32x32x32_i8(fa[b], fb[b], zi, 0, 0, 0);
#pragma unroll
            for (int r = 0; r < 16; ++r) C[r] = __builtin_fmaf((float) s[r], x[r] * dy[b], C[r]);
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();  // (the next chunk's scales overwrite the line)
    };
    int c = wave;
    if (c < nchunk) {
        load_chunk(c, fa, fb, dw, dy);
        for (; c + Q80S_WV < nchunk; c += Q80S_WV) {  // (no branch around the next chunk's loads: behind a join the products would wait for them)
            load_chunk(c + Q80S_WV, nfa, nfb, ndw, ndy);
            multiply();
            __builtin_amdgcn_sched_barrier(0);  // (... as they would behind copies that move up between them)
#pragma unroll
            for (int b = 0; b < 4; ++b) { fa[b] = nfa[b]; fb[b] = nfb[b]; dw[b] = ndw[b]; dy[b] = ndy[b]; }
        }
        multiply();
    }
#pragma unroll
    for (int r = 0; r < 16; ++r) red[wave][r][lane] = C[r];
    __syncthreads();
    for (int e = tid; e < 16 * 64; e += Q80S_WV * 64) {
        const int m = e >> 5, i = e & 31, r = (i >> 3) * 4 + (i & 3), l = m + 32 * ((i >> 2) & 1), n = n0 + i;  // (32 lanes: the 32 rows of one column)
        float v = red[0][r][l];
#pragma unroll
        for (int w = 1; w < Q80S_WV; ++w) v += red[w][r][l];
        q80s_result<EPI, true>(a, mt, epi, mi, m, n, v);
    }
}

// ------------------------------------------------------------------------------------------------ 2 .. 32 columns, few rows
// The same product where 32 rows a workgroup leave CUs idle or each wave a chain of dependent round trips: 16 rows and 16 columns (CT: times two) a workgroup on v_mfma_i32_16x16x32_i8, four
// chunks of a wave in flight at once (18 registers each: 32-row tiles hold one ahead).  A lane fetches 16 bytes of one half of a block for two blocks at a time, 256 consecutive bytes per 16
// lanes, and v_permlane32_swap turns them into the operands of the two blocks (the K order inside a block is the same on both sides, so the integer sums are).  One v_mfma_f32_16x16x1 (four outer
// products) gives d_w * d_x of a chunk's four blocks.  The chunks go to the eight sums, and these are added, as above: the same bits.
template <int CT, bool EPI> __global__ void __launch_bounds__(Q80S_WV * 64, 2) k_mmq_q80_rows16(const mmq80s_args a, const mmq_epi epi) {
    args_ahead<sizeof(mmq80s_args)>();
    constexpr int DEPTH = 4;
    __shared__ float red[Q80S_WV][4 * CT][64];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int fr = lane & 15, q = lane >> 4;
    const int gp = (int) blockIdx.x >> 1;
    const int mi = gp < a.m[0].panel_end ? 0 : (gp < a.m[1].panel_end ? 1 : 2);  // (uniform)
    const mmq80s_mat & mt = a.m[mi];
    const int panel = gp - (mi ? a.m[mi - 1].panel_end : 0), r0 = 16 * ((int) blockIdx.x & 1);
    const int nchunk = a.K / 128;
    const uint8_t * const wp = mt.W + (size_t) panel * nchunk * 4352;
    const int w_off = (q >> 1) * 1024 + (q & 1) * 512 + (r0 + fr) * 16, dw_off = 4096 + q * 64 + (r0 + fr) * 2;
    int y_off[CT], dy_off[CT];
#pragma unroll
    for (int t = 0; t < CT; ++t) {
        const int col = min(16 * t + fr, a.M - 1);
        y_off[t] = (q >> 1) * 1152 + (q & 1) * 512 + col * 16;
        dy_off[t] = q * 1152 + 1024 + col * 4;
    }
    struct chunk { int4q w[2], y[CT][2]; uint32_t dw; float dy[CT]; };
    auto fetch = [&](const int c, chunk & o) __attribute__((always_inline)) {
        const uint8_t * const t = wp + (size_t) c * 4352;
        const char * const yt = a.act + (size_t) c * 4608;
#pragma unroll
        for (int u = 0; u < 2; ++u) o.w[u] = *(const int4q *) (t + w_off + u * 2048);
        o.dw = *(const uint16_t *) (t + dw_off);
#pragma unroll
        for (int k = 0; k < CT; ++k) {
#pragma unroll
            for (int u = 0; u < 2; ++u) o.y[k][u] = *(const int4q *) (yt + y_off[k] + u * 2304);
            o.dy[k] = *(const float *) (yt + dy_off[k]);
        }
    };
    float C[CT][4];
#pragma unroll
    for (int k = 0; k < CT; ++k)
#pragma unroll
        for (int r = 0; r < 4; ++r) C[k][r] = 0.0f;
    const int4q zi = {0, 0, 0, 0};
    float16q zf;
#pragma unroll
    for (int r = 0; r < 16; ++r) zf[r] = 0.0f;
    auto blocks = [](const int4q v, long & b0, long & b1) __attribute__((always_inline)) {  // lanes 0 .. 31 hold the first block's halves, lanes 32 .. 63 the second's -> 8 bytes of each for every lane
        const auto x = __builtin_amdgcn_permlane32_swap((unsigned) v[0], (unsigned) v[2], false, false);
        const auto y = __builtin_amdgcn_permlane32_swap((unsigned) v[1], (unsigned) v[3], false, false);
        b0 = (long) (((unsigned long) y[0] << 32) | x[0]);
        b1 = (long) (((unsigned long) y[1] << 32) | x[1]);
    };
    auto multiply = [&](const chunk & o) __attribute__((always_inline)) {
        long w[4];
        blocks(o.w[0], w[0], w[1]);
        blocks(o.w[1], w[2], w[3]);
        const float dw = h2f((uint16_t) o.dw);
#pragma unroll
        for (int k = 0; k < CT; ++k) {
            long y[4];
            blocks(o.y[k][0], y[0], y[1]);
            blocks(o.y[k][1], y[2], y[3]);
            const float16q p = __builtin_amdgcn_mfma_f32_16x16x1f32(o.dy[k], dw, zf, 0, 0, 0);
#pragma unroll
            for (int b = 0; b < 4; ++b) {
                const int4q s = __builtin_amdgcn_mfma_i32_16x16x32_i8(y[b], w[b], zi, 0, 0, 0);
#pragma unroll
                for (int r = 0; r < 4; ++r) C[k][r] = __builtin_fmaf((float) s[r], p[4 * b + r], C[k][r]);
            }
        }
    };
    const int mine = wave < nchunk ? (nchunk - wave + Q80S_WV - 1) / Q80S_WV : 0;  // chunks wave, wave + 8, ..
    if (mine) {
        auto at = [&](const int i) { return wave + Q80S_WV * min(i, mine - 1); };  // (past the last: that one again, read and not used)
        chunk o[DEPTH];
#pragma unroll
        for (int d = 0; d < DEPTH; ++d) fetch(at(d), o[d]);
        __builtin_amdgcn_sched_barrier(0);
        int i = 0;
        for (; i + DEPTH < mine; i += DEPTH) {
#pragma unroll
            for (int d = 0; d < DEPTH; ++d) {
                multiply(o[d]);
                __builtin_amdgcn_sched_barrier(0);  // (the next loads into these registers, and not further down)
                fetch(at(i + DEPTH + d), o[d]);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
#pragma unroll
        for (int d = 0; d < DEPTH; ++d)
            if (i + d < mine) multiply(o[d]);
    }
#pragma unroll
    for (int k = 0; k < CT; ++k)
#pragma unroll
        for (int r = 0; r < 4; ++r) red[wave][4 * k + r][lane] = C[k][r];
    __syncthreads();
    for (int e = tid; e < 256 * CT; e += Q80S_WV * 64) {  // (16 lanes: the 16 rows of one column)
        const int m = e >> 4, i = e & 15, r = (m >> 4) * 4 + (m & 3), l = ((m >> 2) & 3) * 16 + i;
        float v = red[0][r][l];
#pragma unroll
        for (int w = 1; w < Q80S_WV; ++w) v += red[w][r][l];
        q80s_result<EPI, false>(a, mt, epi, mi, m, panel * 32 + r0 + i, v);
    }
}

// ------------------------------------------------------------------------------------------------ 33 columns and up
// A prompt's micro-batch, drafts of several sequences.  A workgroup owns 32 weight rows x 64 columns, its four waves take the K range in interleaved chunks of four
// blocks and make one partial sum each, added in wave order: an output has the same bits whatever matrices and columns share the launch.  Per two blocks and 32
// columns: two v_mfma_i32_32x32x32_i8 for the integer block sums, and ONE v_mfma_f32_32x32x1 (two outer products) for the factors d_w * d_x of all 2 x 1024 outputs —
// the multiplication that would be a third VALU instruction per output and block, and the row scales need no way through LDS to the accumulator's rows.  Two VALU
// are left (convert, fused multiply-add): 128 issue cycles per block beside the matrix core's 64, which would be 1.26 POP/s for the chip.  The tighter bound is the operands' way: a wave fetches 3 KB
// for the 2048 outputs of a block, four SIMDs 96 bytes a clock where a CU's L1 gives 64, 0.84 POP/s.  The next step of two blocks is in flight
// while one is multiplied, three waves per SIMD (160 registers; three steps in flight at two waves per SIMD: 55 us below).  Workgroups that read the same weights
// (the column tiles of a panel) follow one another on one XCD, so the weights cross HBM once per 1024 columns: an XCD runs about 96 workgroups at once, and 6 panels x 16 tiles draw
// fewer different operands than 3 x 32 (2048 columns in two groups / in one, 128 x 128 tiles: 14336 x 4096 385 / 571 / 473 us, 4096 x 4096 124 / 175 / 149).
// TinyLlama, 512 columns: wq + wk + wv / gate + up / a whole 700-token prompt.  128 x 128 LDS tiles, one launch per matrix: 3 x 45 us / 2 x 45 us / 17.2 ms; this kernel
// with the factors on the VALU: 40 / 66 us / 9.1 ms; as it is: 15 / 44 us / 5.9 ms (23.6 GFLOP in 44 us: 0.53 POP/s).
constexpr int Q80C_WV = 4;
template <bool WP> __global__ void __launch_bounds__(Q80C_WV * 64, 3) k_mmq_q80_cols(const mmq80s_args a, const int n_panels, const int m_tiles) {
    args_ahead<sizeof(mmq80s_args) + 8>();
    __shared__ float red[Q80C_WV][16][65];                         // the waves' partial tiles, one 32-column half at a time
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int fr = lane & 31, kg = lane >> 5;
    const int xcd = blockIdx.x & 7, qb = blockIdx.x >> 3;
    // m_tiles: the column tiles of one group of them (blockIdx.y)
    const int gp = (qb / m_tiles) * 8 + xcd, m0 = ((int) blockIdx.y * m_tiles + qb % m_tiles) * 64;  // the panel, counted over all matrices
    if (gp >= n_panels || m0 >= a.M) return;
    const int mi = gp < a.m[0].panel_end ? 0 : (gp < a.m[1].panel_end ? 1 : 2);
    const mmq80s_mat & mt = a.m[mi];
    const int panel = gp - (mi ? a.m[mi - 1].panel_end : 0);
    const int n0 = panel * 32;
    const int nchunk = a.K / 128;
    const bool two = m0 + 32 < a.M;                                // (uniform) the second half of the tile has columns
    // uniform bases + a lane's offset (columns are clamped inside the tile's own groups of 32: group m0 / 32, and the next one when it has columns)
    const uint8_t * wbase = WP ? mt.W + (size_t) panel * nchunk * 4352 : mt.W;
    const size_t wlane = WP ? 0 : (size_t) min(n0 + fr, mt.N - 1) * mt.w_nb1;
    const size_t ygroup = (size_t) (a.K / 32) * 1152;
    const char * y0 = a.act + (size_t) (m0 >> 5) * ygroup, * y1 = two ? y0 + ygroup : y0;
    const int f0 = min(fr, a.M - 1 - m0), f1 = two ? min(fr, a.M - 1 - m0 - 32) : f0;

    int16q zi;
#pragma unroll
    for (int r = 0; r < 16; ++r) zi[r] = 0;
    float32q zp;
#pragma unroll
    for (int r = 0; r < 32; ++r) zp[r] = 0.0f;
    // the operands of two blocks (scales: lanes 0 .. 31 the first block's, lanes 32 .. 63 the second's); two sets: one multiplied, one in flight
    struct opset { int4q A[2], B0[2], B1[2]; uint32_t dW; float dY0, dY1; };
    auto load2 = [&](const int c, const int half, opset & o) {
        const size_t yo = (size_t) (c * 4 + 2 * half) * 1152;
        if constexpr (WP) o.dW = *(const uint16_t *) (wbase + (size_t) c * 4352 + 4096 + half * 128 + lane * 2);
        else o.dW = ld16(wbase + wlane + (size_t) (c * 4 + 2 * half + kg) * 34);
        o.dY0 = *(const float *) (y0 + yo + (kg * 1152 + 1024 + f0 * 4));
        o.dY1 = *(const float *) (y1 + yo + (kg * 1152 + 1024 + f1 * 4));
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            const int b = 2 * half + u;
            if constexpr (WP) o.A[u] = *(const int4q *) (wbase + (size_t) c * 4352 + b * 1024 + lane * 16);  // [K half][row][16]
            else o.A[u] = __builtin_bit_cast(int4q, *(const q80s_u32x4_a2 *) (wbase + wlane + (size_t) (c * 4 + b) * 34 + 2 + 16 * kg));
            o.B0[u] = *(const int4q *) (y0 + yo + u * 1152 + (kg * 512 + f0 * 16));
            o.B1[u] = *(const int4q *) (y1 + yo + u * 1152 + (kg * 512 + f1 * 16));
        }
    };
    float C0[16], C1[16];
    auto mul2 = [&](const opset & o, const auto both) {
        const float dw = h2f((uint16_t) o.dW);
        auto tile = [&](const int4q * B, const float dy, float (&C)[16]) {
            // d_w * d_x of two blocks' 32 x 32 outputs in one matrix instruction (two outer products; a product of two 11-bit significands is exact)
            const float32q p = __builtin_amdgcn_mfma_f32_32x32x1f32(dw, dy, zp, 0, 0, 0);
            const int16q s0 = __builtin_amdgcn_mfma_i32_32x32x32_i8(o.A[0], B[0], zi, 0, 0, 0);
            const int16q s1 = __builtin_amdgcn_mfma_i32_32x32x32_i8(o.A[1], B[1], zi, 0, 0, 0);
#pragma unroll
            for (int r = 0; r < 16; ++r) C[r] = __builtin_fmaf((float) s0[r], p[r], C[r]);
#pragma unroll
            for (int r = 0; r < 16; ++r) C[r] = __builtin_fmaf((float) s1[r], p[16 + r], C[r]);
        };
        tile(o.B0, o.dY0, C0);
        if constexpr (decltype(both)::value) tile(o.B1, o.dY1, C1);
    };
    auto sums = [&](const auto both) {
        if (wave >= nchunk) return;
        const int steps = 2 * ((nchunk - wave + 3) / 4);           // step h: half h & 1 of chunk wave + 4 (h >> 1)
        auto fetch = [&](const int h, opset & o) {                 // (past the last step: the last one's again, read and not used)
            const int hc = min(h, steps - 1);
            load2(wave + 4 * (hc >> 1), hc & 1, o);
            __builtin_amdgcn_sched_barrier(0);                     // (the scheduler would move the loads down to their uses)
        };
        opset o0, o1;
        fetch(0, o0);
        for (int h = 0; h < steps; h += 2) {                       // (an even number of steps)
            fetch(h + 1, o1);
            mul2(o0, both);
            fetch(h + 2, o0);
            mul2(o1, both);
        }
    };
#pragma unroll
    for (int r = 0; r < 16; ++r) { C0[r] = 0.0f; C1[r] = 0.0f; }
    if (two) sums(std::true_type{});
    else sums(std::false_type{});
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        if (h == 1 && !two) break;
        if (h == 1) __syncthreads();
#pragma unroll
        for (int r = 0; r < 16; ++r) red[wave][r][lane] = h ? C1[r] : C0[r];
        __syncthreads();
        // the sums of a column's 32 rows go to consecutive threads: whole 128-byte lines
        for (int e = tid; e < 32 * 32; e += Q80C_WV * 64) {
            const int row = e & 31, col = e >> 5;
            const int r = (row & 3) + 4 * (row >> 3), l = col + 32 * ((row >> 2) & 1);
            float v = red[0][r][l];
#pragma unroll
            for (int w = 1; w < Q80C_WV; ++w) v += red[w][r][l];
            const int m = m0 + 32 * h + col, n = n0 + row;
            if (m < a.M && n < mt.N) {
                if (mt.add) v += mt.add[(size_t) m * mt.add_stride + n];
                mt.dst[(size_t) m * mt.dst_stride + n] = v;
            }
        }
    }
}

// ------------------------------------------------------------------------------------------------ 33 columns and up: 128 x 128 tiles
// Tile 128 weight rows x 128 columns x 128 K (4 blocks) per trip, 8 waves (32 x 64 each), double-buffered LDS: raw int8 of both operands in the XOR-swizzled [row][128 B] image of
// mmq_i8.hip plus the 4 block scales of every row / column.  Four VALU per output and block, one workgroup a CU — but an operand is fetched once for 128 outputs, where the kernel
// above fetches it for 32 or 64: for rows without a panel copy, whose 34-byte blocks come in pieces, and for K of one or two chunks, where that kernel has work for one or
// two of its four waves.  The chunks are taken in its order (sum c mod 4, sums added in order): the same bits.
constexpr int Q80_T = 128 * 128;                // bytes of one operand tile
constexpr int Q80_STAGE = 2 * Q80_T + 2 * 128 * 16;  // A | B | dw[4][128] | da[4][128]
__device__ __forceinline__ int sw_offq(const int row, const int chunk) { return row * 128 + ((chunk ^ ((row >> 1) & 7)) << 4); }

template <bool WP> __global__ void __launch_bounds__(512, 1) k_mmq_q80_tile(const mmq80s_args a, const int n_panels, const int m_tiles) {
    extern __shared__ __attribute__((aligned(16))) char smem[];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int xcd = blockIdx.x & 7, qb = blockIdx.x >> 3;
    const int panel = (qb / m_tiles) * 8 + xcd, mt = qb % m_tiles;
    if (panel >= n_panels) return;
    const mmq80s_mat & w = a.m[0];
    const int n0 = panel * 128, m0 = mt * 128;
    const int nb32 = a.K / 32, trips = a.K / 128;
    const int nslab = wave & 3, mhalf = wave >> 2;

    // staging roles: thread -> (row | column, block of the trip)
    const int srow = tid >> 2, sq = tid & 3;
    const int wrow_c = min(n0 + srow, w.N - 1), ycol_c = min(m0 + srow, a.M - 1);
    const uint8_t * const wblk = WP ? w.W + (size_t) (wrow_c >> 5) * (size_t) trips * 4352 + (size_t) sq * 1024 + (size_t) (wrow_c & 31) * 16 : w.W + (size_t) wrow_c * w.w_nb1 + (size_t) sq * 34;
    const uint8_t * const wscale = WP ? w.W + (size_t) (wrow_c >> 5) * (size_t) trips * 4352 + 4096 + (size_t) sq * 64 + (size_t) (wrow_c & 31) * 2 : wblk;
    const char * const ytile = a.act + ((size_t) (ycol_c >> 5) * (size_t) nb32 + (size_t) sq) * 1152;
    const int off0 = sw_offq(srow, 2 * sq), off1 = sw_offq(srow, 2 * sq + 1);

    uint4 ga0, ga1, gb0, gb1;
    uint16_t gad = 0;
    float gbd = 0.0f;
    auto issue_loads = [&](const int c) {
        if constexpr (WP) {
            ga0 = *(const uint4 *) (wblk + (size_t) c * 4352);
            ga1 = *(const uint4 *) (wblk + (size_t) c * 4352 + 512);
            gad = *(const uint16_t *) (wscale + (size_t) c * 4352);
        } else {
            const uint8_t * p = wblk + (size_t) c * 4 * 34;  // (blocks are 2-byte aligned)
            gad = ld16(p);
            ga0 = make_uint4(ld32_a2(p + 2), ld32_a2(p + 6), ld32_a2(p + 10), ld32_a2(p + 14));
            ga1 = make_uint4(ld32_a2(p + 18), ld32_a2(p + 22), ld32_a2(p + 26), ld32_a2(p + 30));
        }
        const char * yt = ytile + (size_t) c * 4 * 1152;
        gb0 = *(const uint4 *) (yt + (ycol_c & 31) * 16);
        gb1 = *(const uint4 *) (yt + 512 + (ycol_c & 31) * 16);
        gbd = *(const float *) (yt + 1024 + (ycol_c & 31) * 4);
    };
    auto stage = [&](const int t) {
        char * buf = smem + (t & 1) * Q80_STAGE;
        *(uint4 *) (buf + off0) = ga0;
        *(uint4 *) (buf + off1) = ga1;
        *(uint4 *) (buf + Q80_T + off0) = gb0;
        *(uint4 *) (buf + Q80_T + off1) = gb1;
        ((float *) (buf + 2 * Q80_T))[sq * 128 + srow] = h2f(gad);              // scales are stored [block][row] so that the four
        ((float *) (buf + 2 * Q80_T + 128 * 16))[sq * 128 + srow] = gbd;        // consecutive rows of an accumulator quad are one 16-byte read
    };
    auto next = [&](const int c) { return c + 4 < trips ? c + 4 : (c & 3) + 1; };  // the chunk behind chunk c: 0, 4, 8, .., 1, 5, ..

    const int fr = lane & 31, kg = lane >> 5;
    const int swz = (fr >> 1) & 7;
    const int arow_off = (nslab * 32 + fr) * 128;
    const int brow_off0 = (mhalf * 64 + fr) * 128, brow_off1 = (mhalf * 64 + 32 + fr) * 128;
    float C0[16], C1[16], S0[16], S1[16];
    int16q zi;
#pragma unroll
    for (int r = 0; r < 16; ++r) { C0[r] = 0.0f; C1[r] = 0.0f; zi[r] = 0; }

    int c = 0, cl = 0;  // the chunk multiplied, the chunk loaded last
    issue_loads(0);
    stage(0);
    if (trips > 1) { cl = next(0); issue_loads(cl); }
    __syncthreads();
    for (int t = 0; t < trips; ++t) {
        if (t + 1 < trips) {
            stage(t + 1);
            if (t + 2 < trips) { cl = next(cl); issue_loads(cl); }
        }
        const char * buf = smem + (t & 1) * Q80_STAGE;
        const float * dwt = (const float *) (buf + 2 * Q80_T);
        const float * dat = (const float *) (buf + 2 * Q80_T + 128 * 16);
#pragma unroll
        for (int blk = 0; blk < 4; ++blk) {
            const int co = ((2 * blk + kg) ^ swz) << 4;
            const int4q fa = *(const int4q *) (buf + arow_off + co);
            const int4q fb0 = *(const int4q *) (buf + Q80_T + brow_off0 + co), fb1 = *(const int4q *) (buf + Q80_T + brow_off1 + co);
            const float y0 = dat[blk * 128 + mhalf * 64 + fr], y1 = dat[blk * 128 + mhalf * 64 + 32 + fr];
            float x[16];  // block scale of the 16 rows this lane's accumulator registers belong to
#pragma unroll
            for (int g4 = 0; g4 < 4; ++g4) {
                const float4 v = *(const float4 *) (dwt + blk * 128 + nslab * 32 + 8 * g4 + 4 * kg);
                x[4 * g4] = v.x; x[4 * g4 + 1] = v.y; x[4 * g4 + 2] = v.z; x[4 * g4 + 3] = v.w;
            }
            const int16q s0 = __builtin_amdgcn_mfma_i32_32x32x32_i8(fa, fb0, zi, 0, 0, 0);
            const int16q s1 = __builtin_amdgcn_mfma_i32_32x32x32_i8(fa, fb1, zi, 0, 0, 0);
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                C0[r] = __builtin_fmaf((float) s0[r], x[r] * y0, C0[r]);
                C1[r] = __builtin_fmaf((float) s1[r], x[r] * y1, C1[r]);
            }
        }
        const int cn = next(c);
        if ((cn & 3) != (c & 3)) {  // (the last chunk of a sum; past the last sum nothing reads C)
            const bool first = (c & 3) == 0;
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                S0[r] = first ? C0[r] : S0[r] + C0[r];
                S1[r] = first ? C1[r] : S1[r] + C1[r];
                C0[r] = 0.0f;
                C1[r] = 0.0f;
            }
        }
        c = cn;
        __syncthreads();
    }
#pragma unroll
    for (int tt = 0; tt < 2; ++tt) {
        const int m = m0 + mhalf * 64 + tt * 32 + fr;
        if (m >= a.M) continue;
        float * out = w.dst + (size_t) m * w.dst_stride;
        const float * ad = w.add ? w.add + (size_t) m * w.add_stride : nullptr;
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            const int n = n0 + nslab * 32 + 8 * g + 4 * kg;
            float c4[4];
#pragma unroll
            for (int r = 0; r < 4; ++r) c4[r] = tt ? S1[4 * g + r] : S0[4 * g + r];
            if (ad) {
#pragma unroll
                for (int r = 0; r < 4; ++r) if (n + r < w.N) c4[r] += ad[n + r];
            }
            if (n + 3 < w.N && ((((uintptr_t) (out + n)) & 15) == 0)) {
                *(float4 *) (out + n) = make_float4(c4[0], c4[1], c4[2], c4[3]);
            } else {
#pragma unroll
                for (int r = 0; r < 4; ++r) if (n + r < w.N) out[n + r] = c4[r];
            }
        }
    }
}

bool mmq_q80_batch_supported(int type, int64_t K, int64_t N, int64_t M) {
    static const bool on = !getenv("GGML_MI355X_Q80_SKINNY") || atoi(getenv("GGML_MI355X_Q80_SKINNY")) != 0;
    return (on || M > 32) && type == GGML_TYPE_Q8_0 && (K % 128) == 0 && N >= 1 && M >= 2;  // (off: the mat-vec passes up to 32 columns)
}
// Tiles of 128 x 128 instead of the column kernel (N: rows of all matrices of the launch)?  Measured (us, one product with its quantiser, tiles / columns):
// - K of one or two chunks: from about two million outputs on.  K 128, 5632 x 256 10.8 / 9.2, 4096 x 512 10.6 / 12.5, 14336 x 512 19.9 / 27.4; K 256, 4096 x 384 12.9 / 10.5,
//   4096 x 512 13.4 / 13.5, 14336 x 512 24.4 / 29.5.  K 512, up to 512 columns: 14336 x 384 31.2 / 27.5, 14336 x 512 31.9 / 33.3, 32000 x 256 32.4 / 36.2.
// - without a panel copy, any K: K 2048, 4000 x 512 47.8 / 41.6, 5600 x 512 45.8 / 56.4, 14000 x 256 45.2 / 65.8; K 5632, 5600 x 512 104.8 / 110.8, 14000 x 512 197 / 244.
// With a panel copy and longer rows the column kernel wins everywhere: K 2048, 14336 x 512 77.4 / 61.1, 32000 x 2048 570 / 438.
static bool q80_tile_pays(int64_t K, int64_t N, int64_t M, bool panels) {
    if (K <= 256) return N * M >= ((int64_t) 15 << 17);
    if (!panels) return N * M >= ((int64_t) 5 << 19);
    return K <= 512 && M <= 512 && N * M >= ((int64_t) 7 << 20);
}
// 16 rows a workgroup instead of 32 (panels: groups of 32 rows of all matrices of the launch; over panel copies)?  Measured at 16 .. 1000 panels, K 1024 .. 14336, one product with its quantiser
// (us, 32 rows / 16 rows):
// - up to 128 panels the 32-row tiles leave half of the CUs idle.  16 columns: K 2048, 64 panels 8.4 / 7.4, K 5632 12.8 / 10.6, K 14336, 128 panels 27.5 / 21.3; K 1024 6.5 / 6.2; 32 columns: K 2048,
//   64 panels 9.1 / 8.7, K 14336, 128 panels 29.5 / 26.2, but K 1024 6.7 / 7.1.
// - 129 to 256: one 32-row workgroup a CU against two that share it: K 1024, 160 panels 7.4 / 8.5, K 14336 28.8 / 30.8 (K 4096 13.1 / 12.3).
// - beyond, up to 16 columns, four chunks in flight a wave against one: K 2048, 352 panels 13.8 / 12.6, K 4096, 448 22.0 / 20.6, 1000 42.4 / 36.5, K 14336, 300 46.5 / 45.0; K 1024, 700 14.1 / 15.3; and at
//   449 to 512, where the 32-row tiles fill the chip twice, only up to 8 columns: K 8192, 512 panels x 4 36.3 / 34.2, x 16 37.3 / 38.5.  32 columns the other way: K 4096, 352 21.9 / 23.8.
static bool q80_rows16_pays(int64_t K, int panels, int64_t M) {
    if (panels <= 128) return M <= 16 || K >= 2048;
    return panels > 256 && K >= 2048 && M <= (panels > 448 && panels <= 512 ? 8 : 16);
}
// n matrices (1 .. 3) over the same activations; returns the launches; panels[q] != nullptr for ALL of them or for none (the template form is per launch)
int launch_mmq_q80_multi(hipStream_t s, int n, const mmq80s_desc * mats, int K, int M, const void * act_q80, const mmq_epi * epi) {
    mmq80s_args a;
    int pe = 0;
    const bool wp = mats[0].W_panels != nullptr;
    for (int q = 0; q < 3; ++q) {
        const mmq80s_desc & d = mats[q < n ? q : n - 1];
        if (q < n) pe += (d.N + 31) / 32;
        a.m[q] = {wp ? d.W_panels : d.W, d.w_nb1, d.N, pe, d.dst, d.dst_stride, d.add, d.add_stride};
    }
    a.K = K;
    a.M = M;
    a.act = (const char *) act_q80;
    if (M <= 32) {
        const mmq_epi none{};
        const dim3 grid((unsigned) pe), block(Q80S_WV * 64);
        if (wp && q80_rows16_pays(K, pe, M) && !(epi && (epi->kind[0] >= 5 || epi->kind[1] >= 5 || epi->kind[2] >= 5))) {
            const dim3 grid16(2 * (unsigned) pe);
            if (M <= 16) { if (epi) hipLaunchKernelGGL((k_mmq_q80_rows16<1, true>), grid16, block, 0, s, a, *epi); else hipLaunchKernelGGL((k_mmq_q80_rows16<1, false>), grid16, block, 0, s, a, none); }
            else { if (epi) hipLaunchKernelGGL((k_mmq_q80_rows16<2, true>), grid16, block, 0, s, a, *epi); else hipLaunchKernelGGL((k_mmq_q80_rows16<2, false>), grid16, block, 0, s, a, none); }
            return 1;
        }
        if (epi) { if (wp) hipLaunchKernelGGL((k_mmq_q80_skinny<true, true>), grid, block, 0, s, a, *epi); else hipLaunchKernelGGL((k_mmq_q80_skinny<false, true>), grid, block, 0, s, a, *epi); }
        else { if (wp) hipLaunchKernelGGL((k_mmq_q80_skinny<true, false>), grid, block, 0, s, a, none); else hipLaunchKernelGGL((k_mmq_q80_skinny<false, false>), grid, block, 0, s, a, none); }
        return 1;
    }
    int64_t n_total = 0;
    for (int q = 0; q < n; ++q) n_total += mats[q].N;
    if (q80_tile_pays(K, n_total, M, wp)) {
        for (int q = 0; q < n; ++q) {
            mmq80s_args one = a;
            one.m[0] = a.m[q];
            const int np = (mats[q].N + 127) / 128, mt = (M + 127) / 128;
            static std::atomic<uint32_t> raised{0}, raised_p{0};  // one bit per device (common.h: ensure_dyn_lds)
            (void) ensure_dyn_lds(wp ? (const void *) k_mmq_q80_tile<true> : (const void *) k_mmq_q80_tile<false>, 2 * (size_t) Q80_STAGE, wp ? raised_p : raised);  // on failure the launch below fails and graph_compute reports it
            const dim3 grid((unsigned) ((np + 7) / 8 * 8 * mt));
            if (wp) hipLaunchKernelGGL(k_mmq_q80_tile<true>, grid, dim3(512), 2 * Q80_STAGE, s, one, np, mt);
            else hipLaunchKernelGGL(k_mmq_q80_tile<false>, grid, dim3(512), 2 * Q80_STAGE, s, one, np, mt);
        }
        return n;
    }
    const int tiles = (M + 63) / 64, groups = (tiles + 15) / 16, m_tiles = (tiles + groups - 1) / groups;
    const dim3 grid((unsigned) ((pe + 7) / 8 * 8 * m_tiles), (unsigned) groups), block(Q80C_WV * 64);
    if (wp) hipLaunchKernelGGL(k_mmq_q80_cols<true>, grid, block, 0, s, a, pe, m_tiles);
    else hipLaunchKernelGGL(k_mmq_q80_cols<false>, grid, block, 0, s, a, pe, m_tiles);
    return 1;
}
void launch_mmq_q80(hipStream_t s, const uint8_t * W, const uint8_t * W_panels, int64_t w_nb1, int K, int N, int M, const void * act_q80, float * dst, int64_t dst_stride, const float * add,
                           int64_t add_stride) {
    const mmq80s_desc d{W, W_panels, w_nb1, N, dst, dst_stride, add, add_stride};
    launch_mmq_q80_multi(s, 1, &d, K, M, act_q80);
}

MI_TU_TOUCH(mmq_q80)

}  // namespace mi355x
