// mmq_panel.hip — K-quant weights x 2 .. 32 activation columns on the integer matrix cores, over PANEL COPIES of the matrices (repack.hip: k_repack_k_panels).
//
// The launch is a weight stream, in mmq_skinny.hip's arithmetic: int8 products of plain codes, each sub-block's sum folded with its scale in integers, mins (Q6_K: the codes' offset) by one f16 MFMA
// on the blocks' 16-value sums.  What is different is the way of the operands, and that no tile size divides the work:
//   * a unit is 16 rows x one super-block, 2 to 3 KB that lie together in the panel copy: a wave reads whole lines, non-temporally, straight into the registers that the MFMAs (16 x 16 x 32) take —
//     no staging through LDS, no barrier in the loop, four units of a wave in flight;
//   * the activations are put into LDS once per workgroup, in operand order, and asked for ahead of the weights (behind those they would come with them);
//   * sixteen (Q6_K: eight) waves of one workgroup a CU walk tiles; 1 to 16 of them share one, whichever leaves the fewest units in a row (mp_launch).  The 128-row groups of the skinny kernel's
//     tile-parallel form take two rounds as soon as there are more groups than CUs.
// With the products left out a launch takes 1.3 us less (gate/up of Llama-3-8B, 66 MB): it is 4.5 us + bytes / 5.5 TB/s + the 1.2 us by which a second wave of units a SIMD does not hide its first.
// Us a launch with its quantiser, 2 / 9 / 16 columns, mmq_skinny.hip -> here: 28672 x 4096 Q4_K 25.1 / 27.5 / 28.6 -> 23.6 / 23.9 / 24.6; 37888 x 3584 Q5_K 60.6 / 61.2 / 61.4 -> 34.1 / 36.0 / 35.7;
// 128256 x 4096 Q6_K 127.7 / 145.6 / 143.9 -> 98.2 / 97.5 / 106.9.  Steps: Qwen2-7B Q5_K_M, 4 / 16 / 32 sequences 3575 / 3919 / 4331 -> 2766 / 3117 / 3769; Llama-3-8B Q4_K_M 4 / 16 2511 / 2883 ->
// 2488 / 2829.
#include <algorithm>

#include "dev_util.h"
#include "kernels.h"
#include "mmvq_types.h"

namespace mi355x {

typedef _Float16 mp_half2 __attribute__((ext_vector_type(2)));
typedef _Float16 mp_half4 __attribute__((ext_vector_type(4)));
typedef float mp_float4 __attribute__((ext_vector_type(4)));
typedef int mp_int4 __attribute__((ext_vector_type(4)));

constexpr int MP_RS = 80;  // floats between the registers of a partial tile in LDS (64 lanes + 16: a wave that sums four registers' rows reads 64 banks)

__device__ __forceinline__ long mp_long(const uint32_t lo, const uint32_t hi) { return (long) (((unsigned long) hi << 32) | lo); }
// byte K of w replicated into both 16-bit lanes: 0x00bb00bb
template <int K> __device__ __forceinline__ uint32_t mp_rep_byte(const uint32_t w) { return __builtin_amdgcn_perm(0u, w, 0x0c000c00u | (uint32_t) K | ((uint32_t) K << 16)); }
__device__ __forceinline__ uint32_t mp_h2(const float a, const float b) {
    const mp_half2 h = {(_Float16) a, (_Float16) b};
    return __builtin_bit_cast(uint32_t, h);
}

// one unit of weights as a lane holds it: row lane % 16, the eight quants of every 32 that belong to lane group q = lane / 16
template <int QT> struct mp_unit;
template <> struct mp_unit<4> { static constexpr int BYTES = 144; uint4 w[2], hdr; };
template <> struct mp_unit<5> { static constexpr int BYTES = 176; uint4 w[2], hdr; uint2 h; };
template <> struct mp_unit<6> { static constexpr int BYTES = 210; uint4 w[3], sc; uint32_t scq; uint16_t d; };

// the activations of one super-block for 16 columns: column lane % 16
struct mp_act { uint4 y[4]; mp_half4 bs; };
template <int CT> constexpr int mp_sb_bytes() { return CT * (4096 + 512 + 64); }  // LDS of a super-block's activations: [16 columns][4][lane][16] quants, [lane][8] 16-value sums, [column] scales

template <int QT, int CT, int NW>
__global__ void __launch_bounds__(NW * 64) k_mmq_panel(const mmqp_args a) {
    args_ahead<sizeof(mmqp_args)>();
    constexpr int DEPTH = CT == 2 && NW == 16 ? 2 : 4, NT = NW * 64, NP = CT == 1 ? 5 : 9;
    extern __shared__ __attribute__((aligned(16))) char smem[];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int fr = lane & 15, q = lane >> 4;
    const int nblk = a.K / 256;
    const int S = a.split, P = NW / S;                                     // waves that share a tile's super-blocks; tiles at once
    const int sub = wave / S, w0 = wave - sub * S;
    char * const ysm = smem, * const bsm = smem + nblk * CT * 4096;
    float * const dyl = (float *) (bsm + nblk * CT * 512);
    float * const red = (float *) (smem + a.red_off);                      // [2][NW][4 CT][MP_RS], S > 1 only
    const int stride = (int) gridDim.x * P, t0 = (int) blockIdx.x * P;
    const int n_it = (a.n_tiles - t0 + stride - 1) / stride;
    const int cnt = w0 < nblk ? (nblk - w0 + S - 1) / S : 0;               // super-blocks w0, w0 + S, ..
    const int total = n_it * cnt;

    // ---- the activations into LDS in operand order.  First of all requests: behind the weights' they would come with those.  Columns beyond M are not filled, nor their results stored
    const char * const act = (const char *) a.act;
    const int tok = nblk * (int) sizeof(q8k_dev), n_pc = nblk * a.M * 18;   // 16-byte pieces: 16 of quants and two of sums a block
    uint4 pc[NP];
    auto piece_load = [&](const int i) {
        const int blk = i / 18, c = i - blk * 18, col = blk / nblk, sb = blk - col * nblk;
        return *(const uint4 *) (act + (size_t) col * tok + (size_t) sb * sizeof(q8k_dev) + 16 * c);
    };
    auto piece_store = [&](const int i, const uint4 v) {
        const int blk = i / 18, c = i - blk * 18, col = blk / nblk, sb = blk - col * nblk, k = col >> 4, l = col & 15;
        if (c < 16) {  // values 16 c .. + 7 and + 8 .. + 15: lane groups c & 1 and 2 + (c & 1) of sub-block c / 2
            char * const o = ysm + (((size_t) (sb * CT + k) * 4 + (c >> 2)) * 64 + 16 * (c & 1) + l) * 16 + 8 * ((c >> 1) & 1);
            *(uint2 *) o = make_uint2(v.x, v.y);
            *(uint2 *) (o + 512) = make_uint2(v.z, v.w);
        } else {       // sums 8 (c - 16) .. + 7: lane groups 2 (c - 16) and the next
            char * const o = bsm + ((size_t) (sb * CT + k) * 64 + 32 * (c - 16) + l) * 8;
            *(uint2 *) o = make_uint2(v.x, v.y);
            *(uint2 *) (o + 128) = make_uint2(v.z, v.w);
        }
    };
#pragma unroll
    for (int j = 0; j < NP; ++j) pc[j] = piece_load(min(tid + j * NT, n_pc - 1));
    const int n_dy = nblk * a.M;
    auto dy_load = [&](const int i) { const int col = i / nblk, sb = i - col * nblk; return *(const float *) (act + (size_t) col * tok + (size_t) sb * sizeof(q8k_dev) + 304); };
    auto dy_store = [&](const int i, const float v) { const int col = i / nblk, sb = i - col * nblk; dyl[sb * 16 * CT + col] = v; };
    const float dy0 = dy_load(min(tid, n_dy - 1));
    __builtin_amdgcn_sched_barrier(0);

    auto tile_of = [&](const int it) { return min(t0 + sub + it * stride, a.n_tiles - 1); };  // (past the last: that one again, not stored)
    auto tile_base = [&](const int tile) -> const uint8_t * {
        const int mi = tile < a.m[0].tile_end ? 0 : (tile < a.m[1].tile_end ? 1 : 2);
        const int first = mi == 0 ? 0 : (mi == 1 ? a.m[0].tile_end : a.m[1].tile_end);
        const uint8_t * W = mi == 0 ? a.m[0].W : (mi == 1 ? a.m[1].W : a.m[2].W);
        return W + (size_t) (tile - first) * (size_t) (nblk * 16 * mp_unit<QT>::BYTES);
    };
    auto fetch = [&](const int it, const int sb, mp_unit<QT> & u) __attribute__((always_inline)) {
        const uint8_t * tb = tile_base(tile_of(it));
        if constexpr (QT == 4) {
            const uint8_t * p = tb + (size_t) sb * 2304;
            u.hdr = ld_nt(p + 16 * fr);
            u.w[0] = ld_nt(p + 256 + 16 * lane);
            u.w[1] = ld_nt(p + 1280 + 16 * lane);
        } else if constexpr (QT == 5) {
            const uint8_t * p = tb + (size_t) sb * 2816;
            u.hdr = ld_nt(p + 16 * fr);
            u.h = ld_nt8(p + 256 + 8 * lane);
            u.w[0] = ld_nt(p + 768 + 16 * lane);
            u.w[1] = ld_nt(p + 1792 + 16 * lane);
        } else {
            const uint8_t * p = tb + (size_t) sb * 3328;
#pragma unroll
            for (int i = 0; i < 3; ++i) u.w[i] = ld_nt(p + 1024 * i + 16 * lane);
            u.sc = ld_nt(p + 3072 + 16 * fr);
            u.scq = *(const uint32_t *) (p + 3072 + 16 * fr + 4 * q);
            u.d = *(const uint16_t *) (tb + (size_t) nblk * 3328 + (size_t) sb * 32 + 2 * fr);
        }
    };

    float acc[CT][4];
#pragma unroll
    for (int k = 0; k < CT; ++k)
#pragma unroll
        for (int r = 0; r < 4; ++r) acc[k][r] = 0.0f;
    const mp_int4 zi = {0, 0, 0, 0};
    const mp_float4 zf = {0, 0, 0, 0};
    const uint32_t mask0 = (q & 1) ? 0u : ~0u;  // (Q6_K: lane groups of the first / second 16 values of 32)

    // the unit's contribution: D of the MFMAs is column 4 q + r of the weight row fr
    auto multiply = [&](const mp_unit<QT> & u, const int sb) __attribute__((always_inline)) {
        mp_act y[CT];
#pragma unroll
        for (int k = 0; k < CT; ++k) {
#pragma unroll
            for (int i = 0; i < 4; ++i) y[k].y[i] = *(const uint4 *) (ysm + ((size_t) (sb * CT + k) * 4 + i) * 1024 + lane * 16);
            y[k].bs = *(const mp_half4 *) (bsm + (size_t) (sb * CT + k) * 512 + lane * 8);
        }
        int isum[CT][4];
        mp_float4 ms[CT];
        float d, dmin = 0.0f;
#pragma unroll
        for (int k = 0; k < CT; ++k)
#pragma unroll
            for (int r = 0; r < 4; ++r) isum[k][r] = 0;
        if constexpr (QT == 4 || QT == 5) {
            d = h2f((uint16_t) (u.hdr.x & 0xFFFF));
            dmin = h2f((uint16_t) (u.hdr.x >> 16));
            const uint32_t slo = u.hdr.y & 0x3F3F3F3Fu, shi = (u.hdr.w & 0x0F0F0F0Fu) | ((u.hdr.y >> 2) & 0x30303030u);
            const uint32_t mlo = u.hdr.z & 0x3F3F3F3Fu, mhi = ((u.hdr.w >> 4) & 0x0F0F0F0Fu) | ((u.hdr.z >> 2) & 0x30303030u);
            {   // the mins: bsums 4 q .. 4 q + 3 against min 2 q twice and min 2 q + 1 twice (0x6400 | n is 1024 + n in f16)
                const uint32_t msrc = ((lane & 32) ? mhi : mlo) >> (lane & 16);
                const mp_half2 k1024 = {(_Float16) 1024.0f, (_Float16) 1024.0f};
                uint2 mf;
                mf.x = __builtin_bit_cast(uint32_t, __builtin_bit_cast(mp_half2, mp_rep_byte<0>(msrc) | 0x64006400u) - k1024);
                mf.y = __builtin_bit_cast(uint32_t, __builtin_bit_cast(mp_half2, mp_rep_byte<1>(msrc) | 0x64006400u) - k1024);
#pragma unroll
                for (int k = 0; k < CT; ++k) ms[k] = __builtin_amdgcn_mfma_f32_16x16x16f16(y[k].bs, __builtin_bit_cast(mp_half4, mf), zf, 0, 0, 0);
            }
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const uint4 v = u.w[j >> 1];
                const uint32_t x = (j & 1) ? v.z : v.x, z = (j & 1) ? v.w : v.y;
                uint32_t l0 = x & 0x0F0F0F0Fu, l1 = z & 0x0F0F0F0Fu, h0 = (x >> 4) & 0x0F0F0F0Fu, h1 = (z >> 4) & 0x0F0F0F0Fu;
                if constexpr (QT == 5) {
                    l0 |= ((u.h.x >> (2 * j)) & 0x01010101u) << 4;
                    l1 |= ((u.h.y >> (2 * j)) & 0x01010101u) << 4;
                    h0 |= ((u.h.x >> (2 * j + 1)) & 0x01010101u) << 4;
                    h1 |= ((u.h.y >> (2 * j + 1)) & 0x01010101u) << 4;
                }
                const long wl = mp_long(l0, l1), wh = mp_long(h0, h1);
                const uint32_t src = j < 2 ? slo : shi;
                const int s0 = (int) ((src >> (16 * (j & 1))) & 0xFF), s1 = (int) ((src >> (16 * (j & 1) + 8)) & 0xFF);
#pragma unroll
                for (int k = 0; k < CT; ++k) {
                    const mp_int4 ta = __builtin_amdgcn_mfma_i32_16x16x32_i8(mp_long(y[k].y[j].x, y[k].y[j].y), wl, zi, 0, 0, 0);
                    const mp_int4 tb = __builtin_amdgcn_mfma_i32_16x16x32_i8(mp_long(y[k].y[j].z, y[k].y[j].w), wh, zi, 0, 0, 0);
#pragma unroll
                    for (int r = 0; r < 4; ++r) isum[k][r] += __mul24(ta[r], s0) + __mul24(tb[r], s1);
                }
            }
        } else {
            d = h2f(u.d);
            {   // the codes are q + 32: 32 sum_s sc_s bsum_s comes off
                uint2 sf;
                sf.x = mp_h2((float) (int8_t) u.scq, (float) (int8_t) (u.scq >> 8));
                sf.y = mp_h2((float) (int8_t) (u.scq >> 16), (float) (int8_t) (u.scq >> 24));
#pragma unroll
                for (int k = 0; k < CT; ++k) ms[k] = __builtin_amdgcn_mfma_f32_16x16x16f16(y[k].bs, __builtin_bit_cast(mp_half4, sf), zf, 0, 0, 0);
            }
            const uint32_t scw[4] = {u.sc.x, u.sc.y, u.sc.z, u.sc.w};
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const uint32_t a0 = u.w[h].x, a1 = u.w[h].y, b0 = u.w[h].z, b1 = u.w[h].w, c0 = h ? u.w[2].z : u.w[2].x, c1 = h ? u.w[2].w : u.w[2].y;
#pragma unroll
                for (int g = 0; g < 4; ++g) {  // values 128 h + 32 g ..: sub-blocks 8 h + 2 g and 8 h + 2 g + 1, 16 values each
                    const uint32_t x0 = (g & 1) ? b0 : a0, x1 = (g & 1) ? b1 : a1;
                    const uint32_t n0 = g < 2 ? x0 & 0x0F0F0F0Fu : (x0 >> 4) & 0x0F0F0F0Fu, n1 = g < 2 ? x1 & 0x0F0F0F0Fu : (x1 >> 4) & 0x0F0F0F0Fu;
                    const uint32_t u0 = g == 0 ? c0 << 4 : g == 1 ? c0 << 2 : g == 2 ? c0 : c0 >> 2, u1 = g == 0 ? c1 << 4 : g == 1 ? c1 << 2 : g == 2 ? c1 : c1 >> 2;
                    const uint32_t v0 = n0 | (u0 & 0x30303030u), v1 = n1 | (u1 & 0x30303030u);
                    const long wa = mp_long(v0 & mask0, v1 & mask0), wb = mp_long(v0 & ~mask0, v1 & ~mask0);
                    const int s = 8 * h + 2 * g;
                    const int sa = (int) (int8_t) (scw[s >> 2] >> (8 * (s & 3))), sb1 = (int) (int8_t) (scw[s >> 2] >> (8 * (s & 3) + 8));
#pragma unroll
                    for (int k = 0; k < CT; ++k) {
                        const uint4 yv = y[k].y[2 * h + (g >> 1)];
                        const long yg = (g & 1) ? mp_long(yv.z, yv.w) : mp_long(yv.x, yv.y);
                        const mp_int4 ta = __builtin_amdgcn_mfma_i32_16x16x32_i8(yg, wa, zi, 0, 0, 0);
                        const mp_int4 tb = __builtin_amdgcn_mfma_i32_16x16x32_i8(yg, wb, zi, 0, 0, 0);
#pragma unroll
                        for (int r = 0; r < 4; ++r) isum[k][r] += __mul24(ta[r], sa) + __mul24(tb[r], sb1);
                    }
                }
            }
        }
#pragma unroll
        for (int k = 0; k < CT; ++k) {
            const float4 dy = *(const float4 *) (dyl + sb * 16 * CT + 16 * k + 4 * q);
            const float dyv[4] = {dy.x, dy.y, dy.z, dy.w};
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                float v;
                if constexpr (QT == 6) v = d * (float) (isum[k][r] - 32 * (int) ms[k][r]);
                else v = __builtin_fmaf(-dmin, ms[k][r], d * (float) isum[k][r]);
                acc[k][r] = __builtin_fmaf(dyv[r], v, acc[k][r]);
            }
        }
    };

    mp_unit<QT> o[DEPTH];
    int f_it = 0, f_sb = w0;                                               // the next item to request
    auto request = [&](mp_unit<QT> & u) __attribute__((always_inline)) {
        fetch(f_it, f_sb, u);
        f_sb += S;
        if (f_sb >= nblk) { f_sb = w0; f_it = min(f_it + 1, n_it - 1); }    // (past the last item: the last tile again, read and not used)
    };
    if (cnt) {
#pragma unroll
        for (int i = 0; i < DEPTH; ++i) request(o[i]);
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int j = 0; j < NP; ++j)
        if (tid + j * NT < n_pc) piece_store(tid + j * NT, pc[j]);
    for (int i = tid + NP * NT; i < n_pc; i += NT) piece_store(i, piece_load(i));
    if (tid < n_dy) dy_store(tid, dy0);
    for (int i = tid + NT; i < n_dy; i += NT) dy_store(i, dy_load(i));
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");

    auto store = [&](const int tile, const int m, const int i, float v) __attribute__((always_inline)) {
        if (tile >= a.n_tiles || m >= a.M) return;
        const int mi = tile < a.m[0].tile_end ? 0 : (tile < a.m[1].tile_end ? 1 : 2);
        const int first = mi == 0 ? 0 : (mi == 1 ? a.m[0].tile_end : a.m[1].tile_end);
        const mmqp_mat & mt = a.m[mi];
        const int n = (tile - first) * 16 + i;
        if (mt.add) v += mt.add[(size_t) m * mt.add_stride + n];
        mt.dst[(size_t) m * mt.dst_stride + n] = v;
    };
    int it = 0, left = cnt;
    auto tile_end = [&]() __attribute__((always_inline)) {
        if (S == 1) {  // the wave has the whole of K: lane = weight row, register r = column 4 q + r
#pragma unroll
            for (int k = 0; k < CT; ++k)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    store(t0 + sub + it * stride, 16 * k + 4 * q + r, fr, acc[k][r]);
                    acc[k][r] = 0.0f;
                }
            ++it;
            return;
        }
        if (a.red_off == 0) asm volatile("s_barrier" ::: "memory");        // (one round: the sums take the place of the activations)
        float * const buf = red + (it & 1) * NW * 4 * CT * MP_RS;
        float * const own = buf + wave * 4 * CT * MP_RS;
#pragma unroll
        for (int k = 0; k < CT; ++k)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                own[(4 * k + r) * MP_RS + lane] = acc[k][r];
                acc[k][r] = 0.0f;
            }
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");  // (the other buffer's readers have passed it when it is written next)
        const int waves = 4 * CT * P;                                      // 256 CT results a tile, P tiles; the waves that add them take turns
        for (int rw = (wave + NW - (it * waves) % NW) % NW; rw < waves; rw += NW) {
            const int e = rw * 64 + lane, ps = e / (256 * CT), x = e - ps * 256 * CT, m = x >> 4, i = x & 15;
            const float * src = buf + ps * S * 4 * CT * MP_RS + (4 * (m >> 4) + (m & 3)) * MP_RS + ((m >> 2) & 3) * 16 + i;
            float v = src[0];
            for (int s = 1; s < S; ++s) v += src[s * 4 * CT * MP_RS];
            store(t0 + ps + it * stride, m, i, v);
        }
        ++it;
    };
    if (!cnt) {
        if (S > 1)
            for (int t = 0; t < n_it; ++t) tile_end();
        return;
    }
    int sb = w0;
    for (int i = 0; i < total; i += DEPTH) {
#pragma unroll
        for (int j = 0; j < DEPTH; ++j) {
            if (i + j >= total) break;
            multiply(o[j], sb);
            __builtin_amdgcn_sched_barrier(0);
            request(o[j]);
            __builtin_amdgcn_sched_barrier(0);
            sb += S;
            if (--left == 0) {
                tile_end();
                left = cnt;
                sb = w0;
            }
        }
    }
}

template <int QT, int CT, int NW> static void mp_launch(hipStream_t s, mmqp_args & a) {
    const int nblk = a.K / 256, acts = mp_sb_bytes<CT>() * nblk, sums = NW * 4 * CT * MP_RS * 4;
    // waves a tile: the fewest units in a row for a wave, the sum of a round's partial tiles counted as one
    const int T = (a.n_tiles + 255) / 256;
    int best = 1 << 30;
    for (int S = NW; S >= 1; S /= 2) {
        const int P = NW / S, rounds = (T + P - 1) / P, cost = rounds * ((nblk + S - 1) / S + (S > 1));
        if (S > 1 && rounds > 1 && acts + 2 * sums > 160 * 1024) continue;
        if (cost < best) {
            best = cost;
            a.split = S;
            a.red_off = rounds > 1 ? acts : 0;
        }
    }
    const int P = NW / a.split;
    const size_t lds = (size_t) (a.split == 1 ? acts : a.red_off ? acts + 2 * sums : std::max(acts, sums));
    static std::atomic<uint32_t> raised{0};  // one bit per device (common.h: ensure_dyn_lds)
    (void) ensure_dyn_lds((const void *) k_mmq_panel<QT, CT, NW>, 160 * 1024, raised);  // on failure the launch below fails and graph_compute reports it
    hipLaunchKernelGGL((k_mmq_panel<QT, CT, NW>), dim3((unsigned) std::min(256, (a.n_tiles + P - 1) / P)), dim3(NW * 64), lds, s, a);
}
template <int QT> static void mp_launch_q(hipStream_t s, mmqp_args & a) {
    if (a.M <= 16) mp_launch<QT, 1, QT == 6 ? 8 : 16>(s, a);
    else if constexpr (QT != 4) mp_launch<QT, 2, QT == 6 ? 8 : 16>(s, a);
}
bool mmq_panel_applies(int type, int64_t K, int64_t n_total, int64_t M) {
    if (!(type == GGML_TYPE_Q4_K || type == GGML_TYPE_Q5_K || type == GGML_TYPE_Q6_K) || K < 256 || (K % 256) != 0 || M < 2 || M > 32) return false;
    if (K / 256 * (M <= 16 ? mp_sb_bytes<1>() : mp_sb_bytes<2>()) > 160 * 1024) return false;  // (the activations stay in LDS)
    // Measured against mmq_skinny.hip (mmq_i8.hip for long Q6_K matrices) at 400 .. 6000 tiles, K 1024 .. 8192, two matrices a launch, 2 .. 32 columns (us there / here):
    // - below 576 tiles that kernel splits K, and its partial sums are added by the next kernel: 400 tiles, K 2048 9.5 / 9.4, K 8192 x 16 19.6 / 20.6;
    // - Q5_K and Q6_K up to 16 columns: 0.49 .. 0.96 of the time (K 1024: 0.72 .. 0.96).  Q4_K, whose eight-wave form suits up to 8 columns when its groups fill the chip: K 4096 0.72 .. 0.97, K 3584, 2048
    //   tiles x 2 24.0 / 24.6, K 2048 16.8 / 18.3; x 9 to 16 K 2048 0.74 .. 1.00, K 1024 13.4 / 13.7;
    // - 17 to 32 columns, twice the activations in LDS and registers: Q5_K from K 2048 0.69 .. 0.99 (K 1024, 2048 tiles 16.4 / 17.1); Q6_K, eight waves a workgroup and a tile each, where 2048 tiles a round
    //   leave few of them idle: 2048 tiles, K 4096 55.3 / 47.9, 8016 178.6 / 151.8, but 2368 68.3 / 72.7; Q4_K 1792 tiles, K 4096 30.1 / 31.5.
    const int64_t tiles = n_total / 16;
    if (tiles < 576 || K < 1024) return false;
    if (M <= 16) return type != GGML_TYPE_Q4_K || K >= (M <= 8 ? 4096 : 2048);
    if (type == GGML_TYPE_Q6_K) return 10 * tiles >= 8 * ((tiles + 2047) / 2048 * 2048);
    return type == GGML_TYPE_Q5_K && K >= 2048;
}
// n matrices (1 .. 3) of one format over the same activations
void launch_mmq_panel(hipStream_t s, int type, int n, const mmqp_mat * mats, int K, int M, const void * act_q8k) {
    mmqp_args a{};
    int t = 0;
    for (int i = 0; i < 3; ++i) {
        a.m[i] = mats[i < n ? i : n - 1];
        if (i < n) t += a.m[i].N / 16;
        a.m[i].tile_end = t;
    }
    a.n_tiles = t;
    a.K = K;
    a.M = M;
    a.act = (const q8k_dev *) act_q8k;
    if (type == GGML_TYPE_Q4_K) mp_launch_q<4>(s, a);
    else if (type == GGML_TYPE_Q5_K) mp_launch_q<5>(s, a);
    else mp_launch_q<6>(s, a);
}

MI_TU_TOUCH(mmq_panel)

}  // namespace mi355x
