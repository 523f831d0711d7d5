// mmf_tile.hip — MUL_MAT / MUL_MAT_ID of a batch of columns by f16 / bf16 matrices: LDS-tiled, on v_mfma_f32_32x32x16_{f16,bf16}.
//
// The contract is mmf.hip's (ggml_compute_forward_mul_mat): src1 is rounded to src0's 16-bit type (nearest even), products
// are exact in f32 and accumulated in f32.  One accumulator per output walks K in steps of 16, in order, whatever the tile: the result does not depend on the tile
// chosen, on the matrices that share the launch or on the other columns.
//
// A workgroup of four waves owns TM src1 columns x TN src0 rows, a quarter of them each, and advances K by 64.  Both operands arrive by LDS-DMA (global_load_lds_dwordx4, 1 KB = 8 rows of
// 128 bytes per wave-instruction) into a ring of S stages, up to S - 1 of them in flight: with one stage ahead in registers a step of 128 x 128 took 1.7 us, the latency of
// its loads, against 0.2 us of matrix work.  The operands of the next 16 values of K leave LDS under the products of these, across the steps too: a step's one barrier lies ahead of its
// last products (128 x 128, K 4096, 6144 rows, 512 columns: 43 us, 70 with the first reads of a step behind its barrier).  src1 is rounded to 16 bits once per tensor (k_to_16: the q / k / v / gate projections read the same copy), which halves
// its share of what a CU fetches.  LDS rows hold the 16-byte chunk index XORed by (row >> 1) & 7 (the lanes
// of the DMA fetch the permuted chunks): the 16 lanes a ds_read_b128 serves at once hit 16 distinct slots.  One barrier per step.  Workgroups that read the same src0
// rows follow one another on one XCD.
#include <algorithm>
#include <atomic>
#include <cstdlib>

#include "dev_util.h"
#include "kernels.h"

namespace mi355x {

typedef _Float16 mt_half8 __attribute__((ext_vector_type(8)));
typedef __bf16 mt_bf8 __attribute__((ext_vector_type(8)));
typedef float mt_float16 __attribute__((ext_vector_type(16)));

// lane i's 16 bytes at base + off land at LDS[lds + 16 i]; base and lds are wave-uniform (M0 is written in the statement that uses it).  No memory clobber: the stage
// written is one that nobody reads before the next barrier, so the compiler may move LDS reads across
__device__ __forceinline__ void mt_dma16(const char * base, const uint32_t off, const uint32_t lds) {
    uint32_t keep;
    asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %3\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2\n\ts_mov_b32 m0, %0" : "=&s"(keep) : "v"(off), "s"(base), "s"(lds));
}

// f32 rows -> dense rows of src0's 16-bit type, nearest even.  Two float4 in, one uint4 out per thread
template <bool BF> __global__ void __launch_bounds__(256) k_to_16(const char * __restrict__ x, const int64_t nb1, const int64_t K8, const int64_t total, uint4 * __restrict__ out) {
    const int64_t i = (int64_t) blockIdx.x * 256 + threadIdx.x;
    if (i >= total) return;
    const int64_t r = i / K8, c = i - r * K8;
    const float4 p = *(const float4 *) (x + r * nb1 + c * 32), q = *(const float4 *) (x + r * nb1 + c * 32 + 16);
    const float v[8] = {p.x, p.y, p.z, p.w, q.x, q.y, q.z, q.w};
    uint4 o;
    if constexpr (BF) {
        mt_bf8 h;
#pragma unroll
        for (int k = 0; k < 8; ++k) h[k] = (__bf16) v[k];
        o = __builtin_bit_cast(uint4, h);
    } else {
        mt_half8 h;
#pragma unroll
        for (int k = 0; k < 8; ++k) h[k] = (_Float16) v[k];
        o = __builtin_bit_cast(uint4, h);
    }
    out[i] = o;
}

struct mt_mat {
    const char * W;
    int64_t nb1;
    int64_t N;
    int tile_end;  // row tiles [previous matrix's tile_end, tile_end) are this matrix's
    char * dst;
    int64_t dst_nb1;
};
struct mt_args {
    mt_mat m[4];    // up to four matrices over the same columns
    int64_t K, M;
    const char * x;  // src1 in 16 bits, dense rows
    int n_tiles, m_tiles;
    // ID: the columns of expert blockIdx.z are list[off[e] .. off[e] + cnt[e]), entry u + n_used t: src1 row (u % ne11) + ne11 t, result row (u, t)
    const int32_t * cnt, * off, * list;
    int64_t n_used, ne11, w_nb2, d_nb2;
};

template <bool BF, int TM, int TN, int S, bool ID> __global__ void __launch_bounds__(256, 1) k_mul_mat_tile(const mt_args a) {
    args_ahead<sizeof(mt_args)>();
    constexpr int MT = TM / 64, NT = TN / 64;
    constexpr int STAGE = (TM + TN) * 128, L = (TM + TN) / 32, Q = L / 4;  // bytes of a stage, DMA instructions per wave and stage, of which the first quarter
    static_assert(S >= 2 && S <= 5 && (S - 1) * L <= 63, "ring");
    extern __shared__ __attribute__((aligned(16))) char smem[];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int fr = lane & 31, g = lane >> 5;
    int tile, mt0, e = 0;
    int64_t M = a.M;
    if constexpr (ID) {
        tile = blockIdx.x;
        mt0 = blockIdx.y;
        e = blockIdx.z;
        M = a.cnt[e];
    } else {
        const int xcd = blockIdx.x & 7, q = blockIdx.x >> 3;
        tile = (q / a.m_tiles) * 8 + xcd;
        mt0 = q % a.m_tiles;
        if (tile >= a.n_tiles) return;
    }
    int mi = 0;
    if constexpr (!ID) mi = tile < a.m[0].tile_end ? 0 : (tile < a.m[1].tile_end ? 1 : (tile < a.m[2].tile_end ? 2 : 3));
    const mt_mat & mat = a.m[mi];
    const int64_t n0 = (int64_t) (tile - (mi ? a.m[mi - 1].tile_end : 0)) * TN, N = mat.N, K = a.K;
    const int32_t * cols = ID ? a.list + a.off[e] : nullptr;
    const char * const wbase = mat.W + n0 * mat.nb1 + (ID ? e * a.w_nb2 : 0);
    const int steps = (int) (K / 64);
    const int swz = (fr >> 1) & 7, wm = wave & 1, wn = wave >> 1;
    const char * const fx = smem + (wm * (TM / 2) + fr) * 128, * const fw = smem + (TM + wn * (TN / 2) + fr) * 128;
    const uint32_t lds0 = (uint32_t) (uintptr_t) smem;

    // (a workgroup of an expert walks the expert's column tiles, the grid's second dimension strides them)
    for (int mt = mt0; ; mt += ID ? (int) gridDim.y : 0) {
        const int64_t m0 = (int64_t) mt * TM;
        if (ID && m0 >= M) return;
        auto uniform = [](const char * q) {  // (wave-uniform by construction; into scalar registers)
            const uint64_t v = (uint64_t) (uintptr_t) q;
            return (const char *) (uintptr_t) (((uint64_t) (uint32_t) __builtin_amdgcn_readfirstlane((int) (v >> 32)) << 32) | (uint32_t) __builtin_amdgcn_readfirstlane((int) v));
        };
        // this wave's DMA instructions: 8 rows each, of src1 below TM and of src0 from there; lane -> row lane / 8, the permuted chunk of slot lane % 8
        const char * base[L];
        uint32_t off[L];
#pragma unroll
        for (int j = 0; j < L; ++j) {
            const int r0 = (wave * L + j) * 8, row = r0 + (lane >> 3), chunk = (lane & 7) ^ ((row >> 1) & 7);
            if (r0 < TM) {
                int64_t m = std::min<int64_t>(m0 + row, M - 1);
                if constexpr (ID) {
                    const int32_t ci = cols[m];
                    m = (ci % a.n_used) % a.ne11 + (ci / a.n_used) * a.ne11;
                    base[j] = uniform(a.x);
                    off[j] = (uint32_t) (m * K * 2 + chunk * 16);
                } else {
                    base[j] = uniform(a.x + m0 * K * 2);
                    off[j] = (uint32_t) ((m - m0) * K * 2 + chunk * 16);
                }
            } else {
                base[j] = uniform(wbase);
                off[j] = (uint32_t) (std::min<int64_t>(row - TM, N - 1 - n0) * mat.nb1 + chunk * 16);
            }
        }
        auto issue = [&](const int s, const int j) __attribute__((always_inline)) {
            mt_dma16(base[j] + (int64_t) s * 128, off[j], lds0 + (uint32_t) (s % S) * STAGE + (uint32_t) (wave * L + j) * 1024);
        };
        mt_float16 acc[MT][NT];
#pragma unroll
        for (int t = 0; t < MT; ++t)
#pragma unroll
            for (int u = 0; u < NT; ++u) acc[t][u] = (mt_float16){0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
        if (ID && mt != mt0) asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");  // (the ring is free, no store is counted in vmcnt)
#pragma unroll
        for (int s = 0; s < S; ++s)
            if (s < steps)
#pragma unroll
                for (int j = 0; j < (s < S - 1 ? L : Q); ++j) issue(s, j);
        auto landed = [&](const int later) __attribute__((always_inline)) {  // a step's pieces are there once no more than those of the `later` steps behind it may fly (0 .. S - 2 of them)
            if (later == 0) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            else if (later == 1) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(L) : "memory");
            else if (later == 2) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 * L) : "memory");
            else asm volatile("s_waitcnt vmcnt(%0)" ::"n"(3 * L) : "memory");
        };
        if (steps >= S) asm volatile("s_waitcnt vmcnt(%0)" ::"n"((S - 2) * L + Q) : "memory");
        else landed(steps - 1);
        asm volatile("s_barrier" ::: "memory");
        uint4 xa[2][MT], wb[2][NT];
        auto frags = [&](const int s, const int ks, const int set) __attribute__((always_inline)) {
            const int bo = (s % S) * STAGE + (((2 * ks + g) ^ swz) << 4);
#pragma unroll
            for (int t = 0; t < MT; ++t) xa[set][t] = *(const uint4 *) (fx + bo + t * 4096);
#pragma unroll
            for (int u = 0; u < NT; ++u) wb[set][u] = *(const uint4 *) (fw + bo + u * 4096);
        };
        frags(0, 0, 0);
        auto products = [&](const int set, const int req, const int j0, const int j1) __attribute__((always_inline)) {  // ... and the requests j0 .. j1 - 1 of step req on the way
#pragma unroll
            for (int t = 0; t < MT; ++t)
#pragma unroll
                for (int u = 0; u < NT; ++u) {
                    if constexpr (BF) acc[t][u] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(mt_bf8, xa[set][t]), __builtin_bit_cast(mt_bf8, wb[set][u]), acc[t][u], 0, 0, 0);
                    else acc[t][u] = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(mt_half8, xa[set][t]), __builtin_bit_cast(mt_half8, wb[set][u]), acc[t][u], 0, 0, 0);
                    const int i = t * NT + u;  // (spread over the products: the CU's one address pipeline takes 16 clocks for each)
#pragma unroll
                    for (int j = j0 + (j1 - j0) * i / (MT * NT); j < j0 + (j1 - j0) * (i + 1) / (MT * NT); ++j) {
                        issue(req, j);
                        __builtin_amdgcn_sched_barrier(0);
                    }
                }
        };
        int s = 0;
        for (; s + S < steps; ++s) {
#pragma unroll
            for (int ks = 0; ks < 4; ++ks) {
                if (ks == 3) {
                    // this wave has the rest of step s in registers and its pieces of step s + 1 have landed (in-order vmcnt: only the S - 2 steps behind it may still fly);
                    // then so has everybody: the stage of step s is the one requested next
                    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"((S - 2) * L) : "memory");
                    frags(s + 1, 0, 0);
                } else frags(s, ks + 1, (ks + 1) & 1);
                __builtin_amdgcn_sched_barrier(0);  // (the reads of the next products travel under these)
                if (ks == 3) products(1, s + S, 0, Q);
                else products(ks & 1, s + S - 1, Q + (L - Q) * ks / 3, Q + (L - Q) * (ks + 1) / 3);
            }
        }
        if (steps >= S)
#pragma unroll
            for (int j = Q; j < L; ++j) issue(steps - 1, j);
        while (true) {  // the rest has been requested
#pragma unroll
            for (int ks = 0; ks < 4; ++ks) {
                if (ks < 3) frags(s, ks + 1, (ks + 1) & 1);
                __builtin_amdgcn_sched_barrier(0);
                products(ks & 1, 0, 0, 0);
            }
            if (++s >= steps) break;
            landed(steps - 1 - s);
            asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
            frags(s, 0, 0);
        }
        // lane: src0 row; register i: src1 column (i & 3) + 8 (i >> 2) + 4 g — 32 lanes store a whole 128-byte line
#pragma unroll
        for (int u = 0; u < NT; ++u) {
            const int64_t n = n0 + wn * (TN / 2) + u * 32 + fr;
            if (n >= N) continue;
#pragma unroll
            for (int t = 0; t < MT; ++t)
#pragma unroll
                for (int i = 0; i < 16; ++i) {
                    const int64_t m = m0 + wm * (TM / 2) + t * 32 + (i & 3) + 8 * (i >> 2) + 4 * g;
                    if (m < M) {
                        char * out;
                        if constexpr (ID) {
                            const int32_t ci = cols[m];
                            out = mat.dst + (ci % a.n_used) * mat.dst_nb1 + (ci / a.n_used) * a.d_nb2;
                        } else out = mat.dst + m * mat.dst_nb1;
                        *(float *) (out + n * 4) = acc[t][u][i];
                    }
                }
        }
        if constexpr (!ID) return;
    }
}

// The tile and its ring: the form whose rounds over the 256 CUs take least.  A round of a form costs the same whatever the shape, in proportion to K (us for K = 4096, weights from
// memory): 256 x 128 in three stages 66, 128 x 128 in four 43, 128 x 64 and 64 x 128 in five 33, 64 x 64 in four 23 with one workgroup per CU and 38 with two.  Measured (us; bf16, 512 columns unless
// stated; 256 x 128 / 128 x 128 / 128 x 64 / 64 x 64; before, where a step's first operands were read behind its barrier: 128 x 128 in two stages, 64 x 128 in five or 64 x 64):
// K 4096 N 14336: 70 / 87 / 117 / 116 (84), N 28672: 139 / 173 / 208 / 227 (161), N 10240: 66 / 85 / 88 / 85 (78), N 6144: 63 / 43 / 59 / 53 (63), N 4096: 62 / 42 / 33 / 38 (34);
// K 14336 N 4096: 192 / 130 / 96 / 119 (107); K 8192 N 2048: 107 / 71 / 51 / 39 (56); K 2048 N 8192: 40 / 28 / 39 / 39 (39), N 2048: 33 / 19 / 14 / 11 (17); 256 columns, K 4096 N 14336:
// 69 / 50 / 63 / 69 (65); 128 columns, N 14336: 60 / 49 / 38 / 42 (39), N 4096: 56 / 42 / 31 / 23 (23).  What bounds a round: from memory a CU fetches at most 50 KB per us however deep
// the ring (142 from L2), so a tile's share of src0 is 0.3 us a step whatever its columns.
// Rows of fewer than 1024 values (MT_SHORT): a round is its latencies and the stores behind it, which only other workgroups of the CU hide, so more of them take turns: 64 x 64 in four stages while the CUs
// have two each, in three (three each) beyond, and 128 x 128 in two stages (two each) where its rounds, 1.9 times as long, are that much fewer.  Measured (us with the rounding; 64 x 64 in
// four / in three / 128 x 128 in two / the form the rounds above would choose): K 128, 6000 x 190 7.7 / 7.8 / 11.4 / 9.1, 12081 x 330 18.1 / 15.8 / 16.4 / 20.4, 24000 x 190 15.9 / 13.9 / 15.6 / 20.0,
// 24000 x 512 30.9 / 27.2 / 23.8 / 29.7; K 448, 2638 x 512 10.5 / 10.5 / 15.6 / 11.5, 24000 x 330 33.1 / 30.1 / 33.4 / 38.2, 24000 x 512 47.1 / 41.2 / 37.2 / 42.2; K 960, 24000 x 330 48.4 / 47.6 /
// 50.8 / 53.1, 12081 x 190 23.4 / 22.5 / 26.7 / 21.2; K 1536 the other way: 12081 x 190 30.6 / 30.4 / 35.9 / 26.8.
constexpr int64_t MT_SHORT = 1024;
struct mt_form { int tm, tn, stages; };
static mt_form mt_pick(const mul_mat_tile_desc * m, int n, int64_t K, int64_t M) {
    auto count = [&](int64_t TM, int64_t TN) {
        int64_t t = 0;
        for (int q = 0; q < n; ++q) t += (m[q].N + TN - 1) / TN;
        return t * ((M + TM - 1) / TM);
    };
    auto rounds = [](int64_t c, int64_t at_once) { return (c + at_once - 1) / at_once; };
    const int64_t small = count(64, 64);
    mt_form best = {64, 64, 4};
    if (M <= 64) return best;  // (wider tiles would be half empty)
    if (K < MT_SHORT) {
        if (small > 512) best = rounds(count(128, 128), 512) * 1460 <= small ? mt_form{128, 128, 2} : mt_form{64, 64, 3};  // (1460 = 1.9 x 768)
        return best;
    }
    int64_t least = small <= 256 ? 23 : 38 * rounds(small, 512);
    const struct { mt_form f; int cost; } forms[4] = {{{128, 64, 5}, 33}, {{128, 128, 4}, 43}, {{256, 128, 3}, 66}, {{64, 128, 5}, 33}};
    for (const auto & o : forms) {
        const int64_t cost = o.cost * rounds(count(o.f.tm, o.f.tn), 256);
        if (cost < least) { least = cost; best = o.f; }
    }
    return best;
}
template <bool BF, int TM, int TN, int S, bool ID> static void mt_launch_t(hipStream_t s, const dim3 grid, const mt_args & a) {
    const size_t lds = (size_t) S * (TM + TN) * 128;
    static std::atomic<uint32_t> raised{0};  // one bit per device (common.h: ensure_dyn_lds)
    (void) ensure_dyn_lds((const void *) k_mul_mat_tile<BF, TM, TN, S, ID>, lds, raised);  // on failure the launch below fails and graph_compute reports it
    hipLaunchKernelGGL((k_mul_mat_tile<BF, TM, TN, S, ID>), grid, dim3(256), lds, s, a);
}
bool mul_mat_tile_ok(int type, int64_t K, int64_t N, int64_t nb0, int64_t nb1, const void * W) {
    return (type == GGML_TYPE_F16 || type == GGML_TYPE_BF16) && nb0 == 2 && K >= 64 && (K % 64) == 0 && N >= 1 && (nb1 % 16) == 0 && (((uintptr_t) W) & 15) == 0 && 128 * nb1 < ((int64_t) 1 << 31);
}
// Rounding and tiles (a workgroup of 64 x 64 walks all of K) against one launch of mmf.hip's kernels.  Measured (us for one product of 17 .. 2048 columns, the rounding included; mmf.hip / tiles):
// - K >= 1024: mmf.hip gives a 16 x 16 tile to 8 waves (16 from K = 4096), which share K in trips of 1024 (2048) values.  While all tiles run at once that is the faster way: K 4096, 512 rows,
//   64 columns 14.5 / 22.0; N 2048 x 32 14.7 / 23.8; K 11008, 8 rows x 17 16 / 46.  With more it is not: N 2048 x 64 25.4 / 25.5, N 4096 x 64 45.8 / 22.6.  The line, in 16 x 16 tiles'
//   worth of outputs: 512 for K of one or two whole trips (K 2048: 448 14.3 / 15.3, 516 17.0 / 14.7), 288 where the last trip is part empty (K 1536: 272 11.7 / 12.0, 320 14.4 / 12.7),
//   304 up to K = 4096 (258 19.6 / 22.9, 384 22.5 / 21.6), 256 beyond (K 11008: 256 35.7 / 49, 272 52 / 47).
// - K below 1024: mmf.hip has one wave walk K for 32 x 32 outputs.  K 512, 128 rows x 64 14.0 / 7.7; K 256 9.0 / 6.8, but x 32 6.4 / 6.8, x 17 5.5 / 6.4; K 128, 1024 rows x 64 6.5 / 6.5, 128 rows
//   x 512 6.4 / 6.6, 11008 x 128 10.1 / 8.2; K 64, 4096 x 256 6.5 / 6.8, 11008 x 512 17.9 / 14.5; at most 32 rows leave the tiles half empty: K 256, 8 rows x 128 5.9 / 6.8, K 512 8.0 / 7.6.
bool mul_mat_tile_pays(int64_t K, int64_t N, int64_t M) {
    if (K >= 1024) return (N + 15) / 16 * M > 16 * (K <= 2048 ? (K % 1024 == 0 ? 512 : 288) : K <= 4096 ? 304 : 256);
    if (N <= 32) return K >= 512 && M <= 1024;
    if (K < 128) return N * M >= (int64_t) 3 << 20;
    if (K < 192) return N >= 256 && M > 48;
    if (K < 384) return M > 32;
    return true;
}
// ... and the experts' columns, `even` of them for each when they are spread evenly: the rounding and tiles against mmf.hip's launch of one wave per 32 x 32 outputs, which lists and tiles of
// few columns hardly fill.  The longer K, the earlier the tiles win.  Measured at 1592 shapes of 4 .. 128 experts of 32 .. 4096 rows (us, mmf.hip / tiles): K 64, 64 x 2048 x 16 columns 17.7 / 41.5
// (every workgroup of 64 x 128 waits for its first stage); K 128 within 10 % from 64 columns on, 1.1 .. 1.5 times as long below; K 192, 128 rows x 32 1.03 times, x 64 0.97; K 256, 8 x 2048 x
// 16 columns 11.8 / 12.1, x 32 17.0 / 13.5, 64 x 2048 x 2 22.3 / 33.7; K 384, 512 rows x 16 1.0 .. 1.08 times, 1408 rows 0.76 .. 0.94; K 512 at most 1.05 times, 0.4 .. 0.9 mostly; up to 32 rows, which
// leave half a tile empty, K 512 x 16 1.05 times, x 32 0.94 .. 1.02, K 768 0.95.  (Drawn with the tiles as they were before their fragments ran ahead of the products; 105 shapes since: 0.99 of that time,
// 0.91 .. 1.02.)
bool mul_mat_id_tile_pays(int64_t K, int64_t N, int64_t even) {
    if (N < 64) return K >= 768 || (K >= 512 && even >= 32);
    if (K >= 512) return true;
    if (K >= 384) return even >= 24 || N >= 1024;
    return (K >= 256 && even >= 24) || (K >= 192 && even >= 48);
}
void launch_to_16(hipStream_t s, int type, const char * x, int64_t nb1, int64_t K, int64_t rows, void * out) {
    const int64_t total = rows * (K / 8);
    const dim3 grid((unsigned) ((total + 255) / 256));
    if (type == GGML_TYPE_BF16) hipLaunchKernelGGL(k_to_16<true>, grid, dim3(256), 0, s, x, nb1, K / 8, total, (uint4 *) out);
    else hipLaunchKernelGGL(k_to_16<false>, grid, dim3(256), 0, s, x, nb1, K / 8, total, (uint4 *) out);
}
int launch_mul_mat_tile(hipStream_t s, int type, const mul_mat_tile_desc * m, int n, int64_t K, int64_t M, const void * x16) {
    mt_args a{};
    const mt_form f = mt_pick(m, n, K, M);
    const int tm = f.tm, tn = f.tn;
    int64_t t = 0;
    for (int q = 0; q < 4; ++q) {
        const mul_mat_tile_desc & d = m[q < n ? q : n - 1];
        if (q < n) t += (d.N + tn - 1) / tn;
        a.m[q] = {(const char *) d.W, d.nb1, d.N, (int) t, (char *) d.dst, d.dst_nb1};
    }
    a.K = K;
    a.M = M;
    a.x = (const char *) x16;
    a.n_tiles = (int) t;
    a.m_tiles = (int) ((M + tm - 1) / tm);
    const dim3 grid((unsigned) ((a.n_tiles + 7) / 8 * 8 * a.m_tiles));
    const bool bf = type == GGML_TYPE_BF16;
#define MT(TM_, TN_, S_) { if (bf) mt_launch_t<true, TM_, TN_, S_, false>(s, grid, a); else mt_launch_t<false, TM_, TN_, S_, false>(s, grid, a); }
    if (tm == 256) MT(256, 128, 3)
    else if (tm == 128 && tn == 128) { if (f.stages == 2) MT(128, 128, 2) else MT(128, 128, 4) }
    else if (tn == 128) MT(64, 128, 5)
    else if (tm == 128) MT(128, 64, 5)
    else if (f.stages == 3) MT(64, 64, 3)
    else MT(64, 64, 4)
#undef MT
    return f.stages * 1000000 + tm * 1000 + tn;
}

void launch_mul_mat_id_tile(hipStream_t s, const tdesc & as, int64_t n_b, int64_t n_used, int64_t T, const tdesc & d, const int32_t * cnt, const int32_t * off, const int32_t * list, const void * x16) {
    mt_args a{};
    const int64_t even = (n_used * T + as.ne[2] - 1) / as.ne[2];  // columns per expert when they are spread evenly (the loop inside covers an expert that drew more)
    for (int q = 0; q < 4; ++q) a.m[q] = {as.data, as.nb[1], as.ne[1], 0, d.data, d.nb[1]};
    a.K = as.ne[0];
    a.x = (const char *) x16;
    a.cnt = cnt; a.off = off; a.list = list;
    a.n_used = n_used; a.ne11 = n_b; a.w_nb2 = as.nb[2]; a.d_nb2 = d.nb[2];
    const int64_t slots = std::max<int64_t>(1, std::min<int64_t>(64, (even + 63) / 64 * 2));
    const int tn = (as.ne[1] + 127) / 128 * std::max<int64_t>(1, even / 64) * as.ne[2] >= 192 ? 128 : 64;
    const dim3 grid((unsigned) ((as.ne[1] + tn - 1) / tn), (unsigned) slots, (unsigned) as.ne[2]);
    const bool bf = as.type == GGML_TYPE_BF16;
    if (tn == 128) { if (bf) mt_launch_t<true, 64, 128, 3, true>(s, grid, a); else mt_launch_t<false, 64, 128, 3, true>(s, grid, a); }
    else { if (bf) mt_launch_t<true, 64, 64, 4, true>(s, grid, a); else mt_launch_t<false, 64, 64, 4, true>(s, grid, a); }
}

MI_TU_TOUCH(mmf_tile)

}  // namespace mi355x
