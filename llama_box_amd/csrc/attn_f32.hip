// attn_f32.hip — FLASH_ATTN_EXT in 32-bit arithmetic over a cache read in place (f32, bf16 or f16 rows), for ANY head sizes: the
// query/key size and the value size may differ and need not be 64 or 128.  Scores, soft-max weights and the weighted sum of V are f32
// from start to end (a cache value is widened exactly; nothing is rounded to 16 bits on the way), so an f32 cache gives true 32-bit
// attention.  Optional sinks: one extra score per head that takes part in the soft-max denominator and carries no value (src[4] of the op).
//
// Two kernels:
//   k_attn_f32_rows  — one workgroup per (query token, head), its four waves take the cache in interleaved blocks of 64 cells and merge
//                      their (max, sum, accumulator) through LDS; a block none of whose cells the mask lets through is skipped after
//                      one 128-byte mask read (attention confined to a window or a chunk touches few blocks).  Decode steps and
//                      small batches.  With few (token, head) pairs over a long cache the cells are split over several workgroups
//                      whose partial (max, sum, accumulator) records k_attn_f32_combine merges — and, where the graph gates the
//                      heads behind the attention, multiplies by the gate's sigmoid on the way out.
//   k_attn_f32_tile  — prompt batches: a workgroup owns 64 query tokens of one head; K and V blocks of 64 cells are staged through LDS as
//                      f32 once per workgroup and every wave runs 16 of the queries against them (a lane owns one cell for the scores
//                      and one or more value columns for the sum); blocks the mask hides from all 64 queries are skipped.
#include <algorithm>
#include <cstdlib>

#include "dev_util.h"
#include "kernels.h"

namespace mi355x {

template <int T> __device__ __forceinline__ float kv_ld(const char * __restrict__ row, const int i) {
    if constexpr (T == GGML_TYPE_F32) return ((const float *) row)[i];
    else if constexpr (T == GGML_TYPE_BF16) return __uint_as_float((uint32_t) ((const uint16_t *) row)[i] << 16);
    else return h2f(((const uint16_t *) row)[i]);
}

__device__ __forceinline__ float wave_max_f(float v) {
    for (int o = 32; o > 0; o >>= 1) v = fmaxf(v, __shfl_xor(v, o, 64));
    return v;
}
__device__ __forceinline__ float wave_sum_f(float v) {
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    return v;
}

constexpr int ATTN_F32_MAX_D = 640;   // largest head size (query/key or value): a latent cache row (latent + rotated part) serves as the key of every head
constexpr int ATTN_F32_MAX_SPLITS = 32;  // workgroups over the cells of one (token, head) at most
constexpr float ATTN_F32_LOW = -1e30f;  // "no score yet": finite, so that differences of maxima never give NaN

// mask element -> additive term (f16 or f32 mask rows; -inf hides the cell)
__device__ __forceinline__ float mask_ld(const char * __restrict__ mrow, const int mtype, const int64_t j) {
    return mtype == GGML_TYPE_F16 ? h2f(((const uint16_t *) mrow)[j]) : ((const float *) mrow)[j];
}

// the additive term of a visible cell: the mask's value itself, or — with a per-head distance penalty — the mask's value read as the distance between query and cell:
// -r1 ln(1 + r2 distance), or -r1 distance (kernels.h: ATTN_PEN_LOG, ATTN_PEN_LINEAR)
__device__ __forceinline__ float mask_term(const float mv, const int pen, const float r1, const float r2) {
    return pen == 0 ? mv : pen == ATTN_PEN_LINEAR ? -(r1 * mv) : -r1 * logf(1.0f + r2 * mv);
}

// the score of a visible cell before the mask's term: dot product x scale x a per-head factor, then optionally soft-capped (cap tanh(. / cap))
__device__ __forceinline__ float attn_score(const float d, const float scale, const float temp, const float cap) {
    const float sc = d * scale * temp;
    return cap > 0.0f ? cap * tanhf(sc / cap) : sc;
}
// weights that are no soft-max: sigmoid(score + bias) for every visible cell on its own, nothing normalised over the cells (`sig` = per head a factor on the score,
// then per head the bias).  The kernels keep their running maximum at 0, rescale by 1 and skip the division by the sum.
__device__ __forceinline__ float attn_sigmoid(const float z) { return 1.0f / (1.0f + expf(-z)); }

// acc[r] += sum over the block's visible cells of p[cell] * V[cell][lane + 64 r]: no branches around the loads (a lane beyond the row's end re-reads the last
// column, its sum is dropped later; hidden cells enter with weight 0)
template <int VT, int CELLS, int RR>
__device__ __forceinline__ void attn_f32_pv(const float p, const uint64_t live, const char * __restrict__ vbase, const int64_t v_nb1, const int64_t j0, const int64_t n_kv, const int DV,
                                            const int lane, float (&acc)[ATTN_F32_MAX_D / 64]) {
    const uint64_t gmask = CELLS == 64 ? ~0ull : ((1ull << CELLS) - 1ull);
    for (int jj0 = 0; jj0 < 64; jj0 += CELLS) {
        if (!((live >> jj0) & gmask)) continue;
        float vv[CELLS][RR];
#pragma unroll
        for (int u = 0; u < CELLS; ++u) {
            const int64_t cell = j0 + jj0 + u < n_kv ? j0 + jj0 + u : n_kv - 1;
            const char * vrow = vbase + cell * v_nb1;
#pragma unroll
            for (int r = 0; r < RR; ++r) {
                const int dcol = lane + 64 * r;
                vv[u][r] = kv_ld<VT>(vrow, dcol < DV ? dcol : DV - 1);
            }
        }
#pragma unroll
        for (int u = 0; u < CELLS; ++u) {
            const float pj = __shfl(p, jj0 + u, 64);
#pragma unroll
            for (int r = 0; r < RR; ++r) acc[r] = fmaf(pj, vv[u][r], acc[r]);
        }
    }
}

// the same sum for 2-byte value rows of 256 .. 512 entries with a lane owning EIGHT NEIGHBOURING columns (8 lane .. 8 lane + 7): one 16-byte load per cell and lane instead
// of eight 2-byte ones.  Cells enter every column's sum in the same order as above, so the results are the same bit for bit.
template <int VT, int CELLS>
__device__ __forceinline__ void attn_f32_pv8(const float p, const uint64_t live, const char * __restrict__ vbase, const int64_t v_nb1, const int64_t j0, const int64_t n_kv, const int DV,
                                             const int lane, float (&acc)[ATTN_F32_MAX_D / 64]) {
    const uint64_t gmask = (1ull << CELLS) - 1ull;
    const int col = 8 * lane < DV ? 8 * lane : DV - 8;  // (a lane beyond the row's end re-reads the last group; its sums are dropped later)
    for (int jj0 = 0; jj0 < 64; jj0 += CELLS) {
        if (!((live >> jj0) & gmask)) continue;
        uint4 vv[CELLS];
#pragma unroll
        for (int u = 0; u < CELLS; ++u) {
            const int64_t cell = j0 + jj0 + u < n_kv ? j0 + jj0 + u : n_kv - 1;
            vv[u] = *(const uint4 *) (vbase + cell * v_nb1 + col * 2);
        }
#pragma unroll
        for (int u = 0; u < CELLS; ++u) {
            const float pj = __shfl(p, jj0 + u, 64);
            const uint32_t w[4] = {vv[u].x, vv[u].y, vv[u].z, vv[u].w};
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                float lo, hi;
                if constexpr (VT == GGML_TYPE_BF16) { lo = __uint_as_float(w[e] << 16); hi = __uint_as_float(w[e] & 0xFFFF0000u); }
                else { lo = h2f((uint16_t) (w[e] & 0xFFFFu)); hi = h2f((uint16_t) (w[e] >> 16)); }
                acc[2 * e] = fmaf(pj, lo, acc[2 * e]);
                acc[2 * e + 1] = fmaf(pj, hi, acc[2 * e + 1]);
            }
        }
    }
}

template <int KT, int VT>
__global__ void __launch_bounds__(256) k_attn_f32_rows(const tdesc q, const tdesc k, const tdesc v, const tdesc mask, const int has_mask, const float * __restrict__ sinks,
                                                       const float * __restrict__ r12, const tdesc dst, const float scale, const float * __restrict__ sig, const float softcap, const int pen_kind,
                                                       float * __restrict__ parts) {
    __shared__ float qs[ATTN_F32_MAX_D];
    __shared__ float part_acc[4][ATTN_F32_MAX_D];
    __shared__ float part_m[4], part_l[4];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int64_t t = blockIdx.x, h = blockIdx.y;
    const int DK = (int) q.ne[0], DV = (int) v.ne[0];
    const int64_t n_kv = k.ne[1];
    const int64_t g = h / (q.ne[2] / k.ne[2]);
    const char * qrow = q.data + t * q.nb[1] + h * q.nb[2];
    for (int i = threadIdx.x; i < DK; i += 256) qs[i] = ((const float *) qrow)[i];
    __syncthreads();
    const char * mrow = has_mask ? mask.data + t * mask.nb[1] : nullptr;
    const char * kbase = k.data + g * k.nb[2];
    const char * vbase = v.data + g * v.nb[2];
    const int pen = r12 ? pen_kind : 0;
    const float r1 = pen ? r12[h] : 0.0f, r2 = pen == ATTN_PEN_LOG ? r12[q.ne[2] + h] : 0.0f;
    // (value rows of 256 .. 512 two-byte entries: a lane owns eight neighbouring columns)
    const bool v_vec8 = VT != GGML_TYPE_F32 && DV > 256 && DV <= 512 && (DV % 8) == 0 && (v.nb[1] % 16) == 0 && (v.nb[2] % 16) == 0 && (((uintptr_t) v.data) & 15) == 0;
    const bool k_vec = KT != GGML_TYPE_F32 && (DK % 8) == 0 && (k.nb[1] % 16) == 0 && (k.nb[2] % 16) == 0 && (((uintptr_t) k.data) & 15) == 0;
    const bool sgm = sig != nullptr;
    const float s_temp = sgm ? sig[h] : 1.0f, s_bias = sgm ? sig[q.ne[2] + h] : 0.0f;
    float m = sgm ? 0.0f : ATTN_F32_LOW, l = 0.0f;
    if (sinks && wave == 0 && blockIdx.z == 0 && !sgm) { m = sinks[h]; l = 1.0f; }  // the sink: exp(sink - m) = 1 in the denominator, nothing in the numerator
    float acc[ATTN_F32_MAX_D / 64];
#pragma unroll
    for (int r = 0; r < ATTN_F32_MAX_D / 64; ++r) acc[r] = 0.0f;
    for (int64_t j0 = (int64_t) (blockIdx.z * 4 + wave) * 64; j0 < n_kv; j0 += 256 * (int64_t) gridDim.z) {
        const int64_t j = j0 + lane;
        float mv = -INFINITY;
        if (j < n_kv) mv = has_mask ? mask_ld(mrow, mask.type, j) : 0.0f;
        const bool vis = mv > -INFINITY;
        const uint64_t live = __ballot(vis);
        if (!live) continue;
        float s = -INFINITY;
        if (vis) {
            const char * krow = kbase + j * k.nb[1];
            float d = 0.0f;
            if constexpr (KT != GGML_TYPE_F32) {
                if (k_vec) {  // 16-byte loads of eight 2-byte values; the sum runs over i in the same order as the scalar loop below
                    for (int i = 0; i < DK; i += 8) {
                        const uint4 w = *(const uint4 *) (krow + i * 2);
                        const uint32_t u[4] = {w.x, w.y, w.z, w.w};
#pragma unroll
                        for (int e = 0; e < 4; ++e) {
                            float lo, hi;
                            if constexpr (KT == GGML_TYPE_BF16) { lo = __uint_as_float(u[e] << 16); hi = __uint_as_float(u[e] & 0xFFFF0000u); }
                            else { lo = h2f((uint16_t) (u[e] & 0xFFFFu)); hi = h2f((uint16_t) (u[e] >> 16)); }
                            d = fmaf(qs[i + 2 * e], lo, d);
                            d = fmaf(qs[i + 2 * e + 1], hi, d);
                        }
                    }
                } else
                for (int i = 0; i < DK; ++i) d = fmaf(qs[i], kv_ld<KT>(krow, i), d);
            } else
            for (int i = 0; i < DK; ++i) d = fmaf(qs[i], kv_ld<KT>(krow, i), d);
            s = attn_score(d, scale, s_temp, softcap) + mask_term(mv, pen, r1, r2);
        }
        float p, corr;
        if (sgm) {
            p = vis ? attn_sigmoid(s + s_bias) : 0.0f;
            corr = 1.0f;
        } else {
            const float m_new = fmaxf(m, wave_max_f(s));
            p = vis ? expf(s - m_new) : 0.0f;
            corr = expf(m - m_new);
            l = l * corr + wave_sum_f(p);
            m = m_new;
        }
#pragma unroll
        for (int r = 0; r < ATTN_F32_MAX_D / 64; ++r) acc[r] *= corr;
        // the visible cells' value rows, CELLS at a time with all their loads in flight together: a wave pays one trip to memory per group (measured: 2 us
        // on an otherwise idle chip), so the groups are as large as the registers allow — 32 cells for value sizes up to 128, 16 beyond
        if constexpr (VT != GGML_TYPE_F32) {
            if (v_vec8) { attn_f32_pv8<VT, 16>(p, live, vbase, v.nb[1], j0, n_kv, DV, lane, acc); continue; }
        }
        if (DV <= 128) attn_f32_pv<VT, 32, 2>(p, live, vbase, v.nb[1], j0, n_kv, DV, lane, acc);
        else if (DV <= 256) attn_f32_pv<VT, 16, 4>(p, live, vbase, v.nb[1], j0, n_kv, DV, lane, acc);
        else attn_f32_pv<VT, 8, ATTN_F32_MAX_D / 64>(p, live, vbase, v.nb[1], j0, n_kv, DV, lane, acc);
    }
    if (lane == 0) { part_m[wave] = m; part_l[wave] = l; }
    if (v_vec8) {
#pragma unroll
        for (int e = 0; e < 8; ++e) if (8 * lane + e < DV) part_acc[wave][8 * lane + e] = acc[e];
    } else {
#pragma unroll
        for (int r = 0; r < ATTN_F32_MAX_D / 64; ++r) {
            const int dcol = lane + 64 * r;
            if (dcol < DV) part_acc[wave][dcol] = acc[r];
        }
    }
    __syncthreads();
    if (wave != 0) return;
    float M = part_m[0];
    for (int w = 1; w < 4; ++w) M = fmaxf(M, part_m[w]);
    float L = 0.0f, cw[4];
    for (int w = 0; w < 4; ++w) { cw[w] = expf(part_m[w] - M); L += part_l[w] * cw[w]; }
    if (gridDim.z > 1) {  // one of several workgroups over the cells of this (token, head): its record for the merge
        float * rec = parts + ((t * q.ne[2] + h) * gridDim.z + blockIdx.z) * (int64_t) (DV + 2);
        if (lane == 0) { rec[0] = M; rec[1] = L; }
        for (int dcol = lane; dcol < DV; dcol += 64) {
            float o = 0.0f;
            for (int w = 0; w < 4; ++w) o += part_acc[w][dcol] * cw[w];
            rec[2 + dcol] = o;
        }
        return;
    }
    const float inv = sgm ? 1.0f : (L > 0.0f ? 1.0f / L : 0.0f);
    float * out = (float *) (dst.data + h * dst.nb[1] + t * dst.nb[2]);
    for (int dcol = lane; dcol < DV; dcol += 64) {
        float o = 0.0f;
        for (int w = 0; w < 4; ++w) o += part_acc[w][dcol] * cw[w];
        out[dcol] = o * inv;
    }
}

// k_attn_f32_rows for what a decode step of most models is: 2-byte rows of up to 128 entries that vector loads reach, the soft-max alone (no distance penalty, sigmoid or cap).  What bounds such a
// launch is its chain of round trips and the instructions between them, not bytes: the general kernel fetches its arguments in five rounds round two 64-bit divisions, then the query, then the mask,
// then a K row in loads that wait for one another, then the values in two trips, out of 40 KB of code of which each launch runs a tenth.  Here the arguments are one struct with the group size in it,
// query and mask are requested together, a block's K rows (sixteen lanes a row) and its values (a lane two neighbouring columns) in one trip each; sums across lanes by DPP.
// 2 tokens x 16 heads of 128 over 1800 cells, 900 of them visible, in 8 splits: 11.2 us, 7.9 here (9.9 with a lane fetching a row); one token x 32 heads over 300 cells 11.2, 7.5.
struct attn_rows_args {
    const char * q, * k, * v, * mask;
    const float * sinks;
    char * dst;
    float * parts;
    int64_t q_nb1, q_nb2, k_nb1, k_nb2, v_nb1, v_nb2, mask_nb1, dst_nb1, dst_nb2;
    int n_kv, DK, DV, H, gq, mask_f16;
    float scale;
};
template <int T>  // K and V rows: bf16 or f16
__global__ void __launch_bounds__(256) k_attn_f32_rows128(const attn_rows_args a) {
    args_ahead<sizeof(attn_rows_args)>();
    __shared__ float part_acc[4][128], part_m[4], part_l[4];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int t = blockIdx.x, h = blockIdx.y, g = h / a.gq, DK = a.DK, DV = a.DV, n_kv = a.n_kv;
    const int c16 = lane & 15, r16 = lane >> 4;  // sixteen lanes fetch a K row, 16 bytes each; the lane's own cell of a block is 4 c16 + r16
    const char * const mrow = a.mask ? a.mask + t * a.mask_nb1 : nullptr;
    auto mask_at = [&](const int j) -> float {
        if (j >= n_kv) return -INFINITY;
        if (!mrow) return 0.0f;
        return a.mask_f16 ? h2f(((const uint16_t *) mrow)[j]) : ((const float *) mrow)[j];
    };
    auto two = [](const uint32_t w, float & lo, float & hi) {
        if constexpr (T == GGML_TYPE_BF16) { lo = __uint_as_float(w << 16); hi = __uint_as_float(w & 0xFFFF0000u); }
        else { lo = h2f((uint16_t) (w & 0xFFFFu)); hi = h2f((uint16_t) (w >> 16)); }
    };
    int j0 = ((int) blockIdx.z * 4 + wave) * 64;
    float mv_next = mask_at(j0 + 4 * c16 + r16);
    const bool has_q = 8 * c16 < DK;
    const float4 * const qrow = (const float4 *) (a.q + t * a.q_nb1 + h * a.q_nb2) + (has_q ? 2 * c16 : 0);
    const float4 qa = qrow[0], qb = qrow[1];
    const float qv[8] = {qa.x, qa.y, qa.z, qa.w, qb.x, qb.y, qb.z, qb.w};
    const char * const kbase = a.k + g * a.k_nb2 + (has_q ? 16 * c16 : 0), * const vbase = a.v + g * a.v_nb2 + 2 * min(2 * lane, DV - 2);
    float m = ATTN_F32_LOW, l = 0.0f, acc0 = 0.0f, acc1 = 0.0f;
    if (a.sinks && wave == 0 && blockIdx.z == 0) { m = a.sinks[h]; l = 1.0f; }  // the sink: exp(sink - m) = 1 in the denominator, nothing in the numerator
    for (; j0 < n_kv; j0 += 256 * (int) gridDim.z) {
        const float mv = mv_next;
        mv_next = mask_at(j0 + 256 * (int) gridDim.z + 4 * c16 + r16);
        const bool vis = mv > -INFINITY;
        const uint64_t live = __ballot(vis);
        if (!live) continue;
        uint4 w[16];
#pragma unroll
        for (int i = 0; i < 16; ++i)  // cells 4 i .. 4 i + 3
            if ((live >> i) & 0x0001000100010001ull) w[i] = *(const uint4 *) (kbase + (int64_t) min(j0 + 4 * i + r16, n_kv - 1) * a.k_nb1);
        float s = 0.0f;
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            if (((live >> i) & 0x0001000100010001ull) == 0) continue;
            const uint32_t u[4] = {w[i].x, w[i].y, w[i].z, w[i].w};
            float d = 0.0f;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                float lo, hi;
                two(u[e], lo, hi);
                d = fmaf(qv[2 * e], lo, d);
                d = fmaf(qv[2 * e + 1], hi, d);
            }
            d = row16_sum(has_q ? d : 0.0f);
            s = c16 == i ? d : s;
        }
        s = vis ? s * a.scale + mv : -INFINITY;
        const float m_new = fmaxf(m, wave_max(s));
        const float p = vis ? expf(s - m_new) : 0.0f, corr = expf(m - m_new);
        l = l * corr + wave_sum(p);
        m = m_new;
        acc0 *= corr;
        acc1 *= corr;
        uint32_t vv[4][16];
#pragma unroll
        for (int c = 0; c < 4; ++c) {  // cells 16 c .. 16 c + 15
            if (((live >> (4 * c)) & 0x000F000F000F000Full) == 0) continue;
#pragma unroll
            for (int u = 0; u < 16; ++u) vv[c][u] = *(const uint32_t *) (vbase + (int64_t) min(j0 + 16 * c + u, n_kv - 1) * a.v_nb1);
        }
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            if (((live >> (4 * c)) & 0x000F000F000F000Full) == 0) continue;
#pragma unroll
            for (int u = 0; u < 16; ++u) {
                const float pj = readlane_f32(p, 4 * c + (u >> 2) + 16 * (u & 3));
                float lo, hi;
                two(vv[c][u], lo, hi);
                acc0 = fmaf(pj, lo, acc0);
                acc1 = fmaf(pj, hi, acc1);
            }
        }
    }
    if (lane == 0) { part_m[wave] = m; part_l[wave] = l; }
    part_acc[wave][2 * lane] = acc0;
    part_acc[wave][2 * lane + 1] = acc1;
    __syncthreads();
    if (wave != 0) return;
    float M = part_m[0];
#pragma unroll
    for (int w = 1; w < 4; ++w) M = fmaxf(M, part_m[w]);
    float L = 0.0f, cw[4];
#pragma unroll
    for (int w = 0; w < 4; ++w) { cw[w] = expf(part_m[w] - M); L += part_l[w] * cw[w]; }
    float o[2] = {0.0f, 0.0f};
#pragma unroll
    for (int w = 0; w < 4; ++w) {
        o[0] += part_acc[w][lane] * cw[w];
        o[1] += part_acc[w][lane + 64] * cw[w];
    }
    float * out = (float *) (a.dst + h * a.dst_nb1 + t * a.dst_nb2);
    if (gridDim.z > 1) {  // one of several workgroups over the cells of this (token, head): its record for the merge
        out = a.parts + (((int64_t) t * a.H + h) * gridDim.z + blockIdx.z) * (DV + 2);
        if (lane == 0) { out[0] = M; out[1] = L; }
        out += 2;
    } else {
        const float inv = L > 0.0f ? 1.0f / L : 0.0f;
        o[0] *= inv;
        o[1] *= inv;
    }
    if (lane < DV) out[lane] = o[0];
    if (lane + 64 < DV) out[lane + 64] = o[1];
}
// (what the general kernel reads entry by entry stays with it)
static bool attn_f32_rows128_ok(const tdesc & q, const tdesc & k, const tdesc & v, const float * r12, const float * sig, float softcap) {
    if (k.type != v.type || (k.type != GGML_TYPE_BF16 && k.type != GGML_TYPE_F16) || r12 || sig || softcap > 0.0f) return false;
    if (q.ne[0] < 8 || q.ne[0] > 128 || (q.ne[0] % 8) || v.ne[0] < 2 || v.ne[0] > 128 || (v.ne[0] % 2) || k.ne[1] < 1 || k.ne[1] > (1 << 30)) return false;
    if ((q.nb[1] % 16) || (q.nb[2] % 16) || (((uintptr_t) q.data) & 15) || (k.nb[1] % 16) || (k.nb[2] % 16) || (((uintptr_t) k.data) & 15) || (v.nb[1] % 4) || (v.nb[2] % 4) || (((uintptr_t) v.data) & 3)) return false;
    return true;
}

// the merge of k_attn_f32_rows' partial records: one workgroup per (token, head).  gate (may be null): the output is multiplied by sigmoid(gate), one number per head or per entry
__global__ void __launch_bounds__(128) k_attn_f32_combine(const float * __restrict__ parts, const int S, const int H, const int DV, const tdesc dst, const int sgm, const float * __restrict__ gate,
                                                          const int gate_heads) {
    // Lane s of each wave holds split s's (maximum, sum); they, the values of the first eight splits and the gate are requested together.  (One after the other, a round trip a split: 2 tokens x 16 heads
    // in 8 splits 6.0 us a launch; so 4.4.)
    static_assert(ATTN_F32_MAX_SPLITS <= 64, "a lane a split");
    const int64_t t = blockIdx.x, h = blockIdx.y, DR = DV + 2;
    const int lane = threadIdx.x & 63;
    const float * rec = parts + (t * H + h) * S * DR;
    const float ms = lane < S ? rec[lane * DR] : -INFINITY, ls = lane < S ? rec[lane * DR + 1] : 0.0f;
    float v[8], gt = 0.0f;
    auto request = [&](const int d, const int s0) {
#pragma unroll
        for (int u = 0; u < 8; ++u) v[u] = rec[min(s0 + u, S - 1) * DR + 2 + d];
    };
    if ((int) threadIdx.x < DV) {
        request(threadIdx.x, 0);
        if (gate) gt = gate[gate_heads ? t * H + h : (t * H + h) * DV + threadIdx.x];
    }
    const float M = wave_max(ms), c = expf(ms - M), lc = ls * c;
    float L = 0.0f;
    for (int s = 0; s < S; ++s) L += readlane_f32(lc, s);
    const float inv = sgm ? 1.0f : (L > 0.0f ? 1.0f / L : 0.0f);
    float * out = (float *) (dst.data + h * dst.nb[1] + t * dst.nb[2]);
    for (int d0 = 0; d0 < DV; d0 += 128) {  // (whole waves stay: the coefficients come out of their lanes)
        const int d = d0 + (int) threadIdx.x, dl = min(d, DV - 1);
        float o = 0.0f;
        for (int s0 = 0; s0 < S; s0 += 8) {
            if (d0 > 0 || s0 > 0) request(dl, s0);
#pragma unroll
            for (int u = 0; u < 8; ++u)
                if (s0 + u < S) o += v[u] * readlane_f32(c, s0 + u);
        }
        o = o * inv;
        if (gate) {
            if (d0 > 0) gt = gate[gate_heads ? t * H + h : (t * H + h) * DV + dl];
            o = o * (1.f / (1.f + expf(-gt)));
        }
        if (d < DV) out[d] = o;
    }
}

// prompt batches: 64 query tokens x one head per workgroup; K / V blocks of 64 cells staged in LDS as f32
template <int KT, int VT, int DKP, int DVP>   // DKP / DVP: head sizes rounded up to a multiple of 32 / 64 (LDS row lengths)
__global__ void __launch_bounds__(256) k_attn_f32_tile(const tdesc q, const tdesc k, const tdesc v, const tdesc mask, const float * __restrict__ sinks,
                                                       const float * __restrict__ r12, const tdesc dst, const float scale, const float * __restrict__ sig, const float softcap, const int pen_kind) {
    constexpr int QT = 64, KB = 64, QW = QT / 4;  // queries per workgroup, cells per block, queries per wave
    constexpr int KS = DKP + 1;                   // K row stride in LDS (odd: lanes that read column i of 64 different rows hit 64 different banks)
    extern __shared__ float lds[];
    float * Ks = lds;                    // [KB][KS]
    float * Vs = Ks + KB * KS;           // [KB][DVP]
    float * Qs = Vs + KB * DVP;          // [QT][DKP]
    __shared__ int blk_live;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int64_t t0 = (int64_t) blockIdx.x * QT, h = blockIdx.y;
    const int DK = (int) q.ne[0], DV = (int) v.ne[0];
    const int64_t n_kv = k.ne[1], n_q = q.ne[1];
    const int64_t g = h / (q.ne[2] / k.ne[2]);
    const char * kbase = k.data + g * k.nb[2];
    const char * vbase = v.data + g * v.nb[2];
    const int pen = r12 ? pen_kind : 0;
    const float r1 = pen ? r12[h] : 0.0f, r2 = pen == ATTN_PEN_LOG ? r12[q.ne[2] + h] : 0.0f;
    for (int e = threadIdx.x; e < QT * DKP; e += 256) {
        const int qi = e / DKP, i = e % DKP;
        const int64_t t = t0 + qi;
        Qs[e] = (t < n_q && i < DK) ? ((const float *) (q.data + t * q.nb[1] + h * q.nb[2]))[i] : 0.0f;
    }
    const bool sgm = sig != nullptr;
    const float s_temp = sgm ? sig[h] : 1.0f, s_bias = sgm ? sig[q.ne[2] + h] : 0.0f;
    float m[QW], l[QW], acc[QW][DVP / 64];
#pragma unroll
    for (int qi = 0; qi < QW; ++qi) {
        m[qi] = sgm ? 0.0f : (sinks ? sinks[h] : ATTN_F32_LOW);
        l[qi] = (sinks && !sgm) ? 1.0f : 0.0f;
#pragma unroll
        for (int r = 0; r < DVP / 64; ++r) acc[qi][r] = 0.0f;
    }
    for (int64_t j0 = 0; j0 < n_kv; j0 += KB) {
        // does any of the 64 queries see any of the 64 cells?  (one mask element per thread and query row quarter)
        __syncthreads();
        if (threadIdx.x == 0) blk_live = 0;
        __syncthreads();
        {
            bool any = false;
            for (int qi = wave; qi < QT; qi += 4) {
                const int64_t t = t0 + qi, j = j0 + lane;
                if (t < n_q && j < n_kv) any = any || mask_ld(mask.data + t * mask.nb[1], mask.type, j) > -INFINITY;
            }
            if (__ballot(any) && lane == 0) blk_live = 1;
        }
        __syncthreads();
        if (!blk_live) continue;
        for (int e = threadIdx.x; e < KB * DKP; e += 256) {
            const int r = e / DKP, i = e % DKP;
            const int64_t j = j0 + r;
            Ks[r * KS + i] = (j < n_kv && i < DK) ? kv_ld<KT>(kbase + j * k.nb[1], i) : 0.0f;
        }
        for (int e = threadIdx.x; e < KB * DVP; e += 256) {
            const int r = e / DVP, i = e % DVP;
            const int64_t j = j0 + r;
            Vs[e] = (j < n_kv && i < DV) ? kv_ld<VT>(vbase + j * v.nb[1], i) : 0.0f;
        }
        __syncthreads();
#pragma unroll
        for (int qi = 0; qi < QW; ++qi) {
            const int ql = wave * QW + qi;
            const int64_t t = t0 + ql, j = j0 + lane;
            float mv = -INFINITY;
            if (t < n_q && j < n_kv) mv = mask_ld(mask.data + t * mask.nb[1], mask.type, j);
            const bool vis = mv > -INFINITY;
            const uint64_t live = __ballot(vis);
            if (!live) continue;
            float d = 0.0f;
            const float * qr = Qs + ql * DKP;
            const float * kr = Ks + lane * KS;
            for (int i = 0; i < DK; ++i) d = fmaf(qr[i], kr[i], d);
            const float s = vis ? attn_score(d, scale, s_temp, softcap) + mask_term(mv, pen, r1, r2) : -INFINITY;
            float p, corr;
            if (sgm) {
                p = vis ? attn_sigmoid(s + s_bias) : 0.0f;
                corr = 1.0f;
            } else {
                const float m_new = fmaxf(m[qi], wave_max_f(s));
                p = vis ? expf(s - m_new) : 0.0f;
                corr = expf(m[qi] - m_new);
                l[qi] = l[qi] * corr + wave_sum_f(p);
                m[qi] = m_new;
            }
#pragma unroll
            for (int r = 0; r < DVP / 64; ++r) acc[qi][r] *= corr;
            uint64_t todo = live;
            while (todo) {
                const int jj = __builtin_ctzll(todo);
                todo &= todo - 1;
                const float pj = __shfl(p, jj, 64);
#pragma unroll
                for (int r = 0; r < DVP / 64; ++r) acc[qi][r] = fmaf(pj, Vs[jj * DVP + lane + 64 * r], acc[qi][r]);
            }
        }
    }
#pragma unroll
    for (int qi = 0; qi < QW; ++qi) {
        const int64_t t = t0 + wave * QW + qi;
        if (t >= n_q) continue;
        const float inv = sgm ? 1.0f : (l[qi] > 0.0f ? 1.0f / l[qi] : 0.0f);
        float * out = (float *) (dst.data + h * dst.nb[1] + t * dst.nb[2]);
#pragma unroll
        for (int r = 0; r < DVP / 64; ++r) {
            const int dcol = lane + 64 * r;
            if (dcol < DV) out[dcol] = acc[qi][r] * inv;
        }
    }
}

// ------------------------------------------------------------------------------------------------ prompt batches over a bf16 cache: the matrix cores
// k_attn_mma_bf16: a workgroup of four waves owns 32 query tokens of one head; wave w takes every fourth block of 32 cells (w, w + 4, ..), alone, and the four meet at the end.  Per block
//   S^T = K . Q^T   on v_mfma_f32_32x32x16_bf16 (first operand: the cells' bf16 rows; second: the queries, rounded to bf16 once and kept in registers) — a lane
//                   then holds 16 scores of ITS query (its half-wave's cells), so the running maximum, the sum and the rescaling are per-lane scalars and one
//                   exchange with the other half-wave;
//   scores, maxima, exponentials and sums are f32;
//   O^T += V^T . P^T  on the same instruction, the weights P given as TWO bf16 terms (p = hi + lo, |lo| <= 2^-9 |p|): the f32 weights enter the sum to 2^-17, not rounded to 8 bits.
// The key order inside the second product is the order the first product's registers come in (both operands permuted alike).
// K and V rows reach the wave's own LDS by LDS-DMA as they lie (a lane-per-row load of K touches 32 lines an instruction), V is transposed by ds_read_b64_tr_b16 on the way out; a wave needs
// no barrier: the next block's K is requested when this one's has left LDS, its V when the second product has read this one's.  First the mask of the 32 queries is scanned, row by row, for
// the blocks that any of them sees, and for those where its terms are not all zero: only these read it again.  Head sizes: multiples of 8 up to 16 DK16 / 32 DVT.
// What bounds it: the vector ALU, about 350 instructions a block beside 24 matrix ones, with two waves a SIMD; with few cells its chain of round trips (queries and mask, rows, sums), so that each
// requests all it needs before anything waits.  512 queries x 32 heads of 128 on 8 key heads, the last of n cells (us, launches in a row; in brackets with 32 queries a wave, all cells, V^T staged
// by the workgroup): n = 512 22.3 (45.8), 1024 35.0 (80.0), 2048 58.3 (147), 8192 205 (569); 16 heads on 4, n = 2048 49.7 (147); 2048 queries x 64 heads 313 (525); 64 queries x 16 heads, n = 512
// 18.6 (44.8); a first prompt of 128 tokens, 256 cells, 12.0 (19.9), of 32, which see one block, 9.9 (10.0; 11.1 with the four waves meeting and the queries waited for piece by piece).
typedef __bf16 att_bf8 __attribute__((ext_vector_type(8)));
typedef float att_f16v __attribute__((ext_vector_type(16)));
__device__ __forceinline__ uint32_t att_bf16_bits(const float f) {
    const uint32_t u = __float_as_uint(f);
    return (u + 0x7FFFu + ((u >> 16) & 1u)) >> 16;
}
typedef __bf16 att_bf2 __attribute__((ext_vector_type(2)));
typedef float att_f2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ uint32_t att_bf16_pack(const float a, const float b) {  // two values to bf16, nearest even, in one instruction
    return __builtin_bit_cast(uint32_t, __builtin_convertvector((att_f2){a, b}, att_bf2));
}
// e^t for t <= 88: 2^(t log2 e) with the rounding error of the product put back (v_exp_f32's own last place remains, as in expf); 0 from -150 down, NaN stays NaN
__device__ __forceinline__ float att_exp(float t) {
    constexpr float L2E = 1.44269504f, L2E_LO = 1.92596299e-8f, LN2 = 0.693147181f;
    t = t < -150.0f ? -150.0f : t;
    const float a = t * L2E, p = __builtin_amdgcn_exp2f(a);
    return fmaf(p, fmaf(t, L2E_LO, fmaf(t, L2E, -a)) * LN2, p);
}
// lane i's 16 bytes at base + off land at LDS[lds + 16 i]; base and lds are wave-uniform
__device__ __forceinline__ void att_dma16(const char * base, const uint32_t off, const uint32_t lds) {
    uint32_t keep;
    asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %3\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2\n\ts_mov_b32 m0, %0" : "=&s"(keep) : "v"(off), "s"(base), "s"(lds) : "memory");
}
typedef short att_s4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ att_s4 att_read_tr(const uint16_t * at) {  // 16 lanes read 4 rows of 16 values (4 lanes a row, 4 values each), lane i of them receives column i
    return __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) att_s4 *) (__attribute__((address_space(3))) void *) at);
}
// PLAIN: scores are q.k x scale + mask (no sigmoid, cap or distance penalty), head sizes exactly 16 DK16 / 32 DVT.
constexpr int ATT_SCAN_BITS = 16384;  // blocks beyond these are taken as visible, with a bias
template <int DK16, int DVT, bool PLAIN>
__global__ void __launch_bounds__(256, 2) k_attn_mma_bf16(const tdesc q, const tdesc k, const tdesc v, const tdesc mask, const float * __restrict__ sinks, const float * __restrict__ r12, const tdesc dst,
                                                       const float scale, const float * __restrict__ sig, const float softcap, const int pen_kind) {
    args_ahead<args_bytes<tdesc, tdesc, tdesc, tdesc, const float *, const float *, tdesc, float>()>();
    constexpr int W = 4;  // waves
    // 16-byte pieces of a cell's K and V rows in LDS, a piece's index XORed by the cell's: the 16 K rows read at once, and the 4 x 64 bytes of V, hit all banks once
    constexpr int CP = DK16 <= 2 ? 4 : DK16 <= 4 ? 8 : 16, CV = DVT <= 1 ? 4 : DVT <= 2 ? 8 : 16;
    constexpr int KT = 32 * CP * 8, VB = 32 * CV * 8;  // elements of a block's K, V
    __shared__ __attribute__((aligned(16))) uint16_t pool[W * std::max(KT + VB, DVT * 32 * 64)];  // K and V of a wave, in the end its 32 x 32 DVT sums as f32
    __shared__ uint32_t bits[ATT_SCAN_BITS / 32], mixed[ATT_SCAN_BITS / 32];  // block seen by any query; by some only, or with a bias
    __shared__ float meet[W][2][32];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int) threadIdx.x >> 6);
    const int n = lane & 31, g = lane >> 5;
    int h = blockIdx.y, qt = blockIdx.x;
    if (gridDim.y % 8 == 0) {  // an XCD has neighbouring heads, so that their K and V stay in its L2; the late query tiles first, then the early ones upward: a CU's two see equally much
        const int id = blockIdx.x + gridDim.x * blockIdx.y, hx = gridDim.y / 8, t = (id >> 3) / hx, half = (gridDim.x + 1) / 2;
        h = (id & 7) * hx + (id >> 3) % hx;
        qt = t < half ? (int) gridDim.x - 1 - t : t - half;
    }
    const int64_t n_q = q.ne[1], n_kv = k.ne[1];
    const int DK = PLAIN ? 16 * DK16 : (int) q.ne[0], DV = PLAIN ? 32 * DVT : (int) v.ne[0];
    const int64_t tq = (int64_t) qt * 32 + n;  // this lane's query
    const bool q_live = tq < n_q;
    const int kvh = h / ((int) q.ne[2] / (int) k.ne[2]);
    const char * vbase = v.data + kvh * v.nb[2];
    const char * mrow = mask.data + (q_live ? tq : n_q - 1) * mask.nb[1];
    const int n_blk = (int) ((n_kv + 31) / 32), n_scan = min(n_blk, ATT_SCAN_BITS);
    // this lane's 16 mask terms of a block: cells 32 blk + 8 b + 4 g .. + 3, b = 0 .. 3 (register i = 4 b + r)
    auto load_mask = [&](const int blk, float (&mv)[16]) {
        const int64_t j0 = (int64_t) blk * 32 + 4 * g;
        if ((int64_t) blk * 32 + 32 <= n_kv) {  // (uniform)
#pragma unroll
            for (int b = 0; b < 4; ++b) {
                const float4 t = *(const float4 *) (mrow + (j0 + 8 * b) * 4);
                mv[4 * b] = t.x; mv[4 * b + 1] = t.y; mv[4 * b + 2] = t.z; mv[4 * b + 3] = t.w;
            }
        } else {
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                const int64_t j = j0 + 8 * (i >> 2) + (i & 3);
                mv[i] = j < n_kv ? ((const float *) mrow)[j] : -INFINITY;
            }
        }
    };
    for (int i = threadIdx.x; i < (n_scan + 31) / 32; i += blockDim.x) bits[i] = mixed[i] = n_blk == 1 ? 1 : 0;  // (a lone block is not looked at)
    // the queries as second operands: element group (16 s + 8 g .. + 7) of query n; all of a row requested ahead of the mask's scan, rounded behind it
    const float * const qrow = (const float *) (q.data + (q_live ? tq : 0) * q.nb[1] + h * q.nb[2]);
    float qx[PLAIN ? DK16 : 1][8];
    if constexpr (PLAIN) {
        if ((((uintptr_t) q.data | (uintptr_t) q.nb[1] | (uintptr_t) q.nb[2]) & 15) == 0) {  // (uniform)
#pragma unroll
            for (int s = 0; s < DK16; ++s) {
                const float4 x = *(const float4 *) (qrow + 16 * s + 8 * g), y = *(const float4 *) (qrow + 16 * s + 8 * g + 4);
                qx[s][0] = x.x; qx[s][1] = x.y; qx[s][2] = x.z; qx[s][3] = x.w;
                qx[s][4] = y.x; qx[s][5] = y.y; qx[s][6] = y.z; qx[s][7] = y.w;
            }
        } else {
#pragma unroll
            for (int s = 0; s < DK16; ++s)
#pragma unroll
                for (int e = 0; e < 8; ++e) qx[s][e] = qrow[16 * s + 8 * g + e];
        }
    }
    __syncthreads();  // (bits and mixed are clear)
    {  // a wave reads eight of the 32 rows, 256 cells at a time; cells behind the last whole four of a row count as seen, with a bias
        const char * const m0 = mask.data + (int64_t) qt * 32 * mask.nb[1];
        const int rows = (int) std::min<int64_t>(32, n_q - (int64_t) qt * 32) - 1;
        const int64_t n4 = n_kv & ~(int64_t) 3;
        for (int c = 0; n_blk > 1 && c < n_scan; c += 8) {
            const int64_t j = (int64_t) c * 32 + 4 * lane;
            bool any = false, odd = false;
            float4 t[8];  // (no branch between the eight loads: lanes past the end read the row's last four)
#pragma unroll
            for (int r = 0; r < 8; ++r) t[r] = *(const float4 *) (m0 + (int64_t) std::min(8 * wave + r, rows) * mask.nb[1] + std::min(j, n4 - 4) * 4);
#pragma unroll
            for (int r = 0; r < 8; ++r) {
                any |= t[r].x > -INFINITY || t[r].y > -INFINITY || t[r].z > -INFINITY || t[r].w > -INFINITY;
                odd |= t[r].x != 0.0f || t[r].y != 0.0f || t[r].z != 0.0f || t[r].w != 0.0f;
            }
            any = j < n4 ? any : j < n_kv;
            odd |= j >= n4;
            const uint64_t va = __ballot(any), vo = __ballot(odd);  // eight lanes a block
            uint32_t wa = 0, wo = 0;
#pragma unroll
            for (int b = 0; b < 8; ++b) {
                wa |= ((va >> (8 * b)) & 0xFF) ? 1u << b : 0u;
                wo |= ((vo >> (8 * b)) & 0xFF) ? 1u << b : 0u;
            }
            if (lane == 0) {
                const uint32_t in = n_scan - c >= 8 ? 0xFFu : (1u << (n_scan - c)) - 1u;
                if (wa & in) atomicOr(&bits[c >> 5], (wa & in) << (c & 31));
                if (wo & in) atomicOr(&mixed[c >> 5], (wo & in) << (c & 31));
            }
        }
    }
    uint4 qf[DK16];
    {
        const uint32_t keep = q_live ? 0xFFFFFFFFu : 0u;
#pragma unroll
        for (int s = 0; s < DK16; ++s) {
            const int i0 = 16 * s + 8 * g;
            uint32_t b[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                if constexpr (PLAIN) b[e] = att_bf16_pack(qx[s][2 * e], qx[s][2 * e + 1]) & keep;
                else {
                    const float x = (q_live && i0 + 2 * e < DK) ? qrow[i0 + 2 * e] : 0.0f, y = (q_live && i0 + 2 * e + 1 < DK) ? qrow[i0 + 2 * e + 1] : 0.0f;
                    b[e] = att_bf16_pack(x, y);
                }
            }
            qf[s] = make_uint4(b[0], b[1], b[2], b[3]);
        }
    }
    __syncthreads();
    // ONE visible block is the first wave's alone, which stores the result itself (uniform)
    const bool alone = n_blk <= 64 && __builtin_amdgcn_readfirstlane(__builtin_popcount(bits[0]) + (n_blk > 32 ? __builtin_popcount(bits[1]) : 0)) <= 1;
    if (alone && wave != 0) return;
    const uint32_t mine = alone ? 0xFFFFFFFFu : 0x11111111u << wave;
    auto next_block = [&](int blk) {  // this wave's first visible block from blk on (n_blk: none); uniform
        while (blk < n_scan) {
            const uint32_t w = (uint32_t) __builtin_amdgcn_readfirstlane((int) (bits[blk >> 5] & mine)) >> (blk & 31);
            if (w) { blk += __builtin_ctz(w); break; }
            blk = (blk | 31) + 1;
        }
        if (blk >= n_scan) blk += (wave - blk) & (W - 1);
        return min(blk, n_blk);
    };
    const int pen = PLAIN ? 0 : (r12 ? pen_kind : 0);
    const float r1 = pen ? r12[h] : 0.0f, r2 = pen == ATTN_PEN_LOG ? r12[q.ne[2] + h] : 0.0f;
    const bool sgm = PLAIN ? false : sig != nullptr;
    const float s_temp = sgm ? sig[h] : 1.0f, s_bias = sgm ? sig[q.ne[2] + h] : 0.0f;
    float m = sgm ? 0.0f : (sinks && wave == 0 ? sinks[h] : ATTN_F32_LOW), l = (sinks && wave == 0 && !sgm) ? 1.0f : 0.0f;
    att_f16v O[DVT];
#pragma unroll
    for (int dt = 0; dt < DVT; ++dt)
#pragma unroll
        for (int i = 0; i < 16; ++i) O[dt][i] = 0.0f;
    float mv[16];
    bool bias = true;  // the fetched block's mask terms are not all zero
    auto fetch_mask = [&](const int blk) {
        bias = blk >= n_scan || (__builtin_amdgcn_readfirstlane((int) mixed[blk >> 5]) >> (blk & 31) & 1) != 0;
        if (bias) load_mask(blk, mv);
    };
    // Lane and instruction -> cell 64 / C i + lane / C, the piece that slot lane % C holds (past the row's end: its first one, which nobody uses)
    uint16_t * const Kt = pool + wave * (KT + VB), * const Vl = Kt + KT;
    uint32_t koff[CP / 4], voff;  // (the XOR patterns of K repeat every 16 cells, those of V every four)
    auto kpiece = [&](const int i, const int64_t last) {
        const int c = i * (64 / CP) + lane / CP, p = (lane % CP) ^ ((c / (16 / CP)) & (CP - 1));
        return (uint32_t) std::min<int64_t>(c, last) * (uint32_t) k.nb[1] + (p < DK / 8 ? p * 16 : 0);
    };
    auto vpiece = [&](const int i, const int64_t last) {
        const int c = i * (64 / CV) + lane / CV, p = (lane % CV) ^ (4 * ((c / (16 / CV)) & (CV / 4 - 1)));
        return (uint32_t) std::min<int64_t>(c, last) * (uint32_t) v.nb[1] + (p < DV / 8 ? p * 16 : 0);
    };
#pragma unroll
    for (int i = 0; i < CP / 4; ++i) koff[i] = kpiece(i, 31);
    voff = vpiece(0, 31);
    auto dma_k = [&](const int blk) {
        const int64_t j0 = (int64_t) blk * 32;
        const char * const from = k.data + kvh * k.nb[2] + j0 * k.nb[1];
        const uint32_t to = (uint32_t) (uintptr_t) Kt;
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // (the block before has left LDS)
        if (j0 + 32 <= n_kv) {
#pragma unroll
            for (int i = 0; i < CP / 2; ++i) att_dma16(from + (i / (CP / 4)) * 16 * k.nb[1], koff[i % (CP / 4)], to + i * 1024);
        } else {
#pragma unroll
            for (int i = 0; i < CP / 2; ++i) att_dma16(from, kpiece(i, n_kv - 1 - j0), to + i * 1024);
        }
    };
    auto dma_v = [&](const int blk) {
        const int64_t j0 = (int64_t) blk * 32;
        const char * const from = vbase + j0 * v.nb[1];
        const uint32_t to = (uint32_t) (uintptr_t) Vl;
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        if (j0 + 32 <= n_kv) {
#pragma unroll
            for (int i = 0; i < CV / 2; ++i) att_dma16(from + i * (64 / CV) * v.nb[1], voff, to + i * 1024);
        } else {
#pragma unroll
            for (int i = 0; i < CV / 2; ++i) att_dma16(from, vpiece(i, n_kv - 1 - j0), to + i * 1024);
        }
    };
    int blk = next_block(wave);
    if (blk < n_blk) {
        fetch_mask(blk);
        dma_k(blk);
        dma_v(blk);
    }
    while (blk < n_blk) {
        const int64_t j0 = (int64_t) blk * 32;
        const bool tail = j0 + 32 > n_kv;  // (cells past the end: weight 0 and value 0 — a value read for them may be anything)
        if (bias)
#pragma unroll
            for (int i = 0; i < 16; ++i) mv[i] = q_live ? mv[i] : -INFINITY;
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"(CV / 2) : "memory");  // (its K has landed: only its V may still fly)
        att_f16v S;
#pragma unroll
        for (int i = 0; i < 16; ++i) S[i] = 0.0f;
#pragma unroll
        for (int s = 0; s < DK16; ++s) {
            uint4 kf = *(const uint4 *) ((const char *) Kt + (n * CP + ((2 * s + g) ^ ((n / (16 / CP)) & (CP - 1)))) * 16);
            if (!PLAIN && 16 * s + 8 * g >= DK) kf = make_uint4(0, 0, 0, 0);
            S = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(att_bf8, kf), __builtin_bit_cast(att_bf8, qf[s]), S, 0, 0, 0);
        }
        float mx = ATTN_F32_LOW;
        if (!bias) {
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                if constexpr (PLAIN) S[i] = S[i] * scale;
                else S[i] = attn_score(S[i], scale, s_temp, softcap) + mask_term(0.0f, pen, r1, r2);
                mx = fmaxf(mx, S[i]);
            }
        } else {
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                if constexpr (PLAIN) S[i] = mv[i] > -INFINITY ? S[i] * scale + mv[i] : -INFINITY;
                else S[i] = mv[i] > -INFINITY ? attn_score(S[i], scale, s_temp, softcap) + mask_term(mv[i], pen, r1, r2) : -INFINITY;
                mx = fmaxf(mx, S[i]);
            }
        }
        blk = next_block(blk + 1);
        if (blk < n_blk) {
            fetch_mask(blk);
            dma_k(blk);
        }
        __builtin_amdgcn_sched_barrier(0);
        mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
        // the reference of the exponents follows the maximum only when that is e^8 ahead: weights stay below e^8, and the sums are rescaled a few times a row instead of at almost every block
        const float m_new = sgm ? 0.0f : (mx > m + 8.0f ? mx : m);
        const float corr = sgm ? 1.0f : expf(m - m_new);
        float ps = 0.0f;
        uint32_t hi[8], lo[8];
#pragma unroll
        for (int i = 0; i < 16; i += 2) {
            float p0, p1;
            if constexpr (PLAIN) { p0 = att_exp(S[i] - m_new); p1 = att_exp(S[i + 1] - m_new); }
            else {
                p0 = sgm ? (S[i] > -INFINITY ? attn_sigmoid(S[i] + s_bias) : 0.0f) : att_exp(S[i] - m_new);
                p1 = sgm ? (S[i + 1] > -INFINITY ? attn_sigmoid(S[i + 1] + s_bias) : 0.0f) : att_exp(S[i + 1] - m_new);
            }
            ps += p0 + p1;
            const uint32_t h2 = att_bf16_pack(p0, p1);
            hi[i >> 1] = h2;
            lo[i >> 1] = att_bf16_pack(p0 - __uint_as_float(h2 << 16), p1 - __uint_as_float(h2 & 0xFFFF0000u));
        }
        ps += __shfl_xor(ps, 32, 64);
        l = l * corr + ps;
        m = m_new;
        if (__ballot(corr != 1.0f) != 0) {  // (a running maximum that stays rescales by 1)
#pragma unroll
            for (int dt = 0; dt < DVT; ++dt)
#pragma unroll
                for (int i = 0; i < 16; ++i) O[dt][i] *= corr;
        }
        if (blk < n_blk) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(CP / 2) : "memory");  // (the V of this block has landed: only the next one's K may still fly)
        else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        if (tail) {  // cells past the end: weight 0 and value 0 (a value read for them may be anything)
            for (int i = lane; i < 32 * CV; i += 64)
                if (j0 + i / CV >= n_kv) *(uint4 *) (Vl + i * 8) = make_uint4(0, 0, 0, 0);
            asm volatile("" ::: "memory");  // (a wave's LDS accesses happen in the order they are written down in)
        }
#pragma unroll
        for (int s2 = 0; s2 < 2; ++s2) {
            const uint4 ph = make_uint4(hi[4 * s2], hi[4 * s2 + 1], hi[4 * s2 + 2], hi[4 * s2 + 3]);
            const uint4 pl = make_uint4(lo[4 * s2], lo[4 * s2 + 1], lo[4 * s2 + 2], lo[4 * s2 + 3]);
            uint4 vf[DVT];
#pragma unroll
            for (int dt = 0; dt < DVT; ++dt) {
                // a lane reads entries 4 (l & 3) .. + 3 of 16 of one cell and receives one entry (its lane's, l & 15) of four cells: 4 g .. + 3 and 8 + 4 g .. + 3 of the half block
                const int l = lane & 15, c = 16 * s2 + 4 * g + (l >> 2), p = 4 * dt + 2 * ((lane >> 4) & 1) + ((l & 3) >> 1);
                const uint16_t * vr = Vl + (c * CV + (p ^ (4 * ((c / (16 / CV)) & (CV / 4 - 1))))) * 8 + 4 * (l & 1);
                const uint2 a0 = __builtin_bit_cast(uint2, att_read_tr(vr)), a1 = __builtin_bit_cast(uint2, att_read_tr(vr + 8 * CV * 8));
                vf[dt] = make_uint4(a0.x, a0.y, a1.x, a1.y);
            }
#pragma unroll
            for (int dt = 0; dt < DVT; ++dt) O[dt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(att_bf8, vf[dt]), __builtin_bit_cast(att_bf8, ph), O[dt], 0, 0, 0);
#pragma unroll
            for (int dt = 0; dt < DVT; ++dt) O[dt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(att_bf8, vf[dt]), __builtin_bit_cast(att_bf8, pl), O[dt], 0, 0, 0);
        }
        if (blk < n_blk) dma_v(blk);
    }
    float * out = (float *) (dst.data + h * dst.nb[1] + (q_live ? tq : 0) * dst.nb[2]);
    auto store = [&](const int d0, const float4 v) {
        if (PLAIN || d0 + 3 < DV) *(float4 *) (out + d0) = v;
        else {
            const float e[4] = {v.x, v.y, v.z, v.w};
            for (int r = 0; r < 4; ++r) if (d0 + r < DV) out[d0 + r] = e[r];
        }
    };
    if (alone) {
        if (!q_live) return;
        const float inv = sgm ? 1.0f : (l > 0.0f ? 1.0f / l : 0.0f);
#pragma unroll
        for (int dt = 0; dt < DVT; ++dt)
#pragma unroll
            for (int b = 0; b < 4; ++b) store(32 * dt + 8 * b + 4 * g, make_float4(O[dt][4 * b] * inv, O[dt][4 * b + 1] * inv, O[dt][4 * b + 2] * inv, O[dt][4 * b + 3] * inv));
        return;
    }
    // the waves' sums, relative to the largest of their references, added in the waves' order; a wave stores DVT of the 4 DVT groups of 8 entries
    if (g == 0) {
        meet[wave][0][n] = m;
        meet[wave][1][n] = l;
    }
    __syncthreads();  // (nobody reads K or V any more)
    float mm = meet[0][0][n];
#pragma unroll
    for (int w = 1; w < W; ++w) mm = fmaxf(mm, meet[w][0][n]);
    l = 0.0f;
#pragma unroll
    for (int w = 0; w < W; ++w) l += meet[w][1][n] * (sgm ? 1.0f : expf(meet[w][0][n] - mm));
    const float f = sgm ? 1.0f : expf(m - mm);
    float4 * const sums = (float4 *) pool;
#pragma unroll
    for (int dt = 0; dt < DVT; ++dt)
#pragma unroll
        for (int b = 0; b < 4; ++b) sums[(wave * DVT * 4 + dt * 4 + b) * 64 + lane] = make_float4(O[dt][4 * b] * f, O[dt][4 * b + 1] * f, O[dt][4 * b + 2] * f, O[dt][4 * b + 3] * f);
    __syncthreads();
    if (!q_live) return;
    const float inv = sgm ? 1.0f : (l > 0.0f ? 1.0f / l : 0.0f);
#pragma unroll
    for (int i = 0; i < DVT; ++i) {
        const int gi = wave * DVT + i, d0 = 32 * (gi >> 2) + 8 * (gi & 3) + 4 * g;
        float4 p[W];
#pragma unroll
        for (int w = 0; w < W; ++w) p[w] = sums[(w * DVT * 4 + gi) * 64 + lane];
        store(d0, make_float4(((p[0].x + p[1].x) + (p[2].x + p[3].x)) * inv, ((p[0].y + p[1].y) + (p[2].y + p[3].y)) * inv, ((p[0].z + p[1].z) + (p[2].z + p[3].z)) * inv,
                              ((p[0].w + p[1].w) + (p[2].w + p[3].w)) * inv));
    }
}

// k_attn_mma_bf16_wide: the same scheme for ONE key/value head shared by all query heads and rows wider than a wave can hold — a latent cache row [latent | rotated part] of
// several hundred values, its leading part the value.  The queries of a workgroup are 32 (token, head) pairs (head fastest); its four waves share them: wave w computes the
// partial scores over a quarter of the key entries, the partials meet in LDS (every wave adds them in the order 0 .. 3 and so holds the same scores), every wave runs the f32
// soft-max, and wave w accumulates a quarter of the value entries (O^T tiles of 32).  V^T of the block is staged once for all four.  DKQ: 16-entry key groups per wave, DVQ:
// 32-entry value tiles per wave.
template <int DKQ, int DVQ>
__global__ void __launch_bounds__(256) k_attn_mma_bf16_wide(const tdesc q, const tdesc k, const tdesc v, const tdesc mask, const float * __restrict__ sinks, const float * __restrict__ r12,
                                                            const tdesc dst, const float scale, const float * __restrict__ sig, const float softcap, const int pen_kind) {
    constexpr int VS = 36;
    constexpr int DVT = 4 * DVQ;
    __shared__ __attribute__((aligned(16))) uint16_t Vt[DVT * 32 * VS];
    __shared__ float Sp[4][16][64];
    __shared__ int flag[2];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int n = lane & 31, g = lane >> 5;
    const int64_t H = q.ne[2], n_tok = q.ne[1], n_kv = k.ne[1];
    const int DK = (int) q.ne[0], DV = (int) v.ne[0];
    const int64_t qi = (int64_t) blockIdx.x * 32 + n;  // this lane's (token, head) pair
    const bool q_live = qi < n_tok * H;
    const int64_t tq = q_live ? qi / H : 0, h = q_live ? qi % H : 0;
    const char * kbase = k.data;
    const char * vbase = v.data;
    uint4 qf[DKQ];
    {
        const float * qrow = (const float *) (q.data + tq * q.nb[1] + h * q.nb[2]);
#pragma unroll
        for (int s = 0; s < DKQ; ++s) {
            const int i0 = 16 * (wave * DKQ + s) + 8 * g;
            uint32_t b[8];
#pragma unroll
            for (int e = 0; e < 8; ++e) b[e] = (q_live && i0 + e < DK) ? att_bf16_bits(qrow[i0 + e]) : 0u;
            qf[s] = make_uint4(b[0] | (b[1] << 16), b[2] | (b[3] << 16), b[4] | (b[5] << 16), b[6] | (b[7] << 16));
        }
    }
    const int pen = r12 ? pen_kind : 0;
    const float r1 = pen ? r12[h] : 0.0f, r2 = pen == ATTN_PEN_LOG ? r12[H + h] : 0.0f;
    const bool sgm = sig != nullptr;
    const float s_temp = sgm ? sig[h] : 1.0f, s_bias = sgm ? sig[q.ne[2] + h] : 0.0f;
    float m = sgm ? 0.0f : (sinks ? sinks[h] : ATTN_F32_LOW), l = (sinks && !sgm) ? 1.0f : 0.0f;
    att_f16v O[DVQ];
#pragma unroll
    for (int dt = 0; dt < DVQ; ++dt)
#pragma unroll
        for (int i = 0; i < 16; ++i) O[dt][i] = 0.0f;
    const char * mrow = mask.data + tq * mask.nb[1];
    if (threadIdx.x < 2) flag[threadIdx.x] = 0;
    __syncthreads();
    auto load_mask = [&](const int64_t j0, float (&mv)[16]) {
#pragma unroll
        for (int b = 0; b < 4; ++b) {
            const int64_t j = j0 + 8 * b + 4 * g;
            float4 t = make_float4(-INFINITY, -INFINITY, -INFINITY, -INFINITY);
            if (q_live && j + 3 < n_kv) t = *(const float4 *) (mrow + j * 4);
            else if (q_live) {
                if (j < n_kv) t.x = ((const float *) mrow)[j];
                if (j + 1 < n_kv) t.y = ((const float *) mrow)[j + 1];
                if (j + 2 < n_kv) t.z = ((const float *) mrow)[j + 2];
            }
            mv[4 * b] = t.x; mv[4 * b + 1] = t.y; mv[4 * b + 2] = t.z; mv[4 * b + 3] = t.w;
        }
    };
    float mv_next[16];
    load_mask(0, mv_next);
    for (int64_t j0 = 0, blk = 0; j0 < n_kv; j0 += 32, ++blk) {
        float mv[16];
        bool any = false;
#pragma unroll
        for (int i = 0; i < 16; ++i) { mv[i] = mv_next[i]; any = any || mv[i] > -INFINITY; }
        if (j0 + 32 < n_kv) load_mask(j0 + 32, mv_next);
        const bool wave_any = __ballot(any) != 0;  // (the four waves hold the same queries: the same answer in each)
        if (threadIdx.x == 0) flag[(blk + 1) & 1] = 0;
        if (wave_any && lane == 0) flag[blk & 1] = 1;
        __syncthreads();
        if (!flag[blk & 1]) continue;
        // this wave's quarter of the block's key entries, straight from the cache rows
        uint4 kf[DKQ];
        {
            const int64_t cell = j0 + n < n_kv ? j0 + n : n_kv - 1;
            const char * krow = kbase + cell * k.nb[1] + g * 16;
#pragma unroll
            for (int s = 0; s < DKQ; ++s) {
                const int sg = wave * DKQ + s;
                kf[s] = make_uint4(0, 0, 0, 0);
                if (16 * sg + 8 * g < DK) kf[s] = *(const uint4 *) (krow + sg * 32);
            }
        }
        // V^T of the block (all value entries) into LDS, as in k_attn_mma_bf16
        for (int e0 = threadIdx.x; e0 < 8 * (DVT * 4); e0 += 256) {
            const int cg = e0 / (DVT * 4), c8 = e0 % (DVT * 4);
            uint32_t u[4][4];
#pragma unroll
            for (int cc = 0; cc < 4; ++cc) {
                uint4 t = make_uint4(0, 0, 0, 0);
                if (j0 + 4 * cg + cc < n_kv && 8 * c8 < DV) t = *(const uint4 *) (vbase + (j0 + 4 * cg + cc) * v.nb[1] + c8 * 16);
                u[cc][0] = t.x; u[cc][1] = t.y; u[cc][2] = t.z; u[cc][3] = t.w;
            }
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const uint2 lo2 = make_uint2((u[0][e] & 0xFFFFu) | (u[1][e] << 16), (u[2][e] & 0xFFFFu) | (u[3][e] << 16));
                const uint2 hi2 = make_uint2((u[0][e] >> 16) | (u[1][e] & 0xFFFF0000u), (u[2][e] >> 16) | (u[3][e] & 0xFFFF0000u));
                *(uint2 *) (Vt + (8 * c8 + 2 * e) * VS + 4 * cg) = lo2;
                *(uint2 *) (Vt + (8 * c8 + 2 * e + 1) * VS + 4 * cg) = hi2;
            }
        }
        // partial scores over this wave's key entries
        {
            att_f16v Sw;
#pragma unroll
            for (int i = 0; i < 16; ++i) Sw[i] = 0.0f;
#pragma unroll
            for (int s = 0; s < DKQ; ++s) Sw = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(att_bf8, kf[s]), __builtin_bit_cast(att_bf8, qf[s]), Sw, 0, 0, 0);
#pragma unroll
            for (int i = 0; i < 16; ++i) Sp[wave][i][lane] = Sw[i];
        }
        __syncthreads();
        att_f16v S;
#pragma unroll
        for (int i = 0; i < 16; ++i) S[i] = ((Sp[0][i][lane] + Sp[1][i][lane]) + Sp[2][i][lane]) + Sp[3][i][lane];
        float mx = ATTN_F32_LOW;
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            S[i] = mv[i] > -INFINITY ? attn_score(S[i], scale, s_temp, softcap) + mask_term(mv[i], pen, r1, r2) : -INFINITY;
            mx = fmaxf(mx, S[i]);
        }
        mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
        const float m_new = sgm ? 0.0f : fmaxf(m, mx);
        const float corr = sgm ? 1.0f : expf(m - m_new);
        float ps = 0.0f;
        uint32_t hi[8], lo[8];
#pragma unroll
        for (int i = 0; i < 16; i += 2) {
            const float p0 = sgm ? (S[i] > -INFINITY ? attn_sigmoid(S[i] + s_bias) : 0.0f) : expf(S[i] - m_new);
            const float p1 = sgm ? (S[i + 1] > -INFINITY ? attn_sigmoid(S[i + 1] + s_bias) : 0.0f) : expf(S[i + 1] - m_new);
            ps += p0 + p1;
            const uint32_t h0 = att_bf16_bits(p0), h1 = att_bf16_bits(p1);
            hi[i >> 1] = h0 | (h1 << 16);
            lo[i >> 1] = att_bf16_bits(p0 - __uint_as_float(h0 << 16)) | (att_bf16_bits(p1 - __uint_as_float(h1 << 16)) << 16);
        }
        ps += __shfl_xor(ps, 32, 64);
        l = l * corr + ps;
        m = m_new;
#pragma unroll
        for (int dt = 0; dt < DVQ; ++dt)
#pragma unroll
            for (int i = 0; i < 16; ++i) O[dt][i] *= corr;
#pragma unroll
        for (int s2 = 0; s2 < 2; ++s2) {
            const uint4 ph = make_uint4(hi[4 * s2], hi[4 * s2 + 1], hi[4 * s2 + 2], hi[4 * s2 + 3]);
            const uint4 pl = make_uint4(lo[4 * s2], lo[4 * s2 + 1], lo[4 * s2 + 2], lo[4 * s2 + 3]);
#pragma unroll
            for (int dt = 0; dt < DVQ; ++dt) {
                const uint16_t * vr = Vt + (32 * (wave * DVQ + dt) + n) * VS + 16 * s2 + 4 * g;
                const uint2 a0 = *(const uint2 *) vr, a1 = *(const uint2 *) (vr + 8);
                const uint4 vf = make_uint4(a0.x, a0.y, a1.x, a1.y);
                O[dt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(att_bf8, vf), __builtin_bit_cast(att_bf8, ph), O[dt], 0, 0, 0);
                O[dt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(att_bf8, vf), __builtin_bit_cast(att_bf8, pl), O[dt], 0, 0, 0);
            }
        }
    }
    if (!q_live) return;
    const float inv = sgm ? 1.0f : (l > 0.0f ? 1.0f / l : 0.0f);
    float * out = (float *) (dst.data + h * dst.nb[1] + tq * dst.nb[2]);
#pragma unroll
    for (int dt = 0; dt < DVQ; ++dt)
#pragma unroll
        for (int b = 0; b < 4; ++b) {
            const int d0 = 32 * (wave * DVQ + dt) + 8 * b + 4 * g;
            if (d0 + 3 < DV) *(float4 *) (out + d0) = make_float4(O[dt][4 * b] * inv, O[dt][4 * b + 1] * inv, O[dt][4 * b + 2] * inv, O[dt][4 * b + 3] * inv);
            else
                for (int r = 0; r < 4; ++r) if (d0 + r < DV) out[d0 + r] = O[dt][4 * b + r] * inv;
        }
}
// one key/value head, rows beyond what k_attn_mma_bf16 holds (up to 640 key and 512 value entries), at least 128 (token, head) pairs: a workgroup walks the whole cache for 32
// pairs, so a decode step's few pairs are better served by the row kernel's workgroup per pair
static bool attn_mma_bf16_wide_ok(const tdesc & q, const tdesc & k, const tdesc & v, const tdesc * mask, const tdesc & dst) {
    if (!mask || mask->type != GGML_TYPE_F32 || (mask->nb[1] % 16) != 0 || (((uintptr_t) mask->data) & 15)) return false;
    if (k.type != GGML_TYPE_BF16 || v.type != GGML_TYPE_BF16 || k.ne[2] != 1 || q.ne[1] * q.ne[2] < 128) return false;
    if ((q.ne[0] % 8) != 0 || (v.ne[0] % 8) != 0 || (q.ne[0] <= 128 && v.ne[0] <= 128) || q.ne[0] > 640 || v.ne[0] > 512) return false;
    if ((k.nb[1] % 16) || (v.nb[1] % 16) || (((uintptr_t) k.data | (uintptr_t) v.data | (uintptr_t) dst.data) & 15)) return false;
    if ((dst.nb[1] % 16) || (dst.nb[2] % 16)) return false;
    return true;
}

static bool attn_mma_bf16_ok(const tdesc & q, const tdesc & k, const tdesc & v, const tdesc * mask, const tdesc & dst) {
    if (!mask || mask->type != GGML_TYPE_F32 || (mask->nb[1] % 16) != 0 || (((uintptr_t) mask->data) & 15)) return false;
    if (k.type != GGML_TYPE_BF16 || v.type != GGML_TYPE_BF16 || q.ne[1] < 32) return false;
    if ((q.ne[0] % 8) != 0 || (v.ne[0] % 8) != 0 || q.ne[0] > 128 || v.ne[0] > 128) return false;
    if (k.nb[1] >= (1 << 26) || v.nb[1] >= (1 << 26)) return false;  // (a block's offsets in 32 bits)
    if ((k.nb[1] % 16) || (k.nb[2] % 16) || (v.nb[1] % 16) || (v.nb[2] % 16) || (((uintptr_t) k.data | (uintptr_t) v.data | (uintptr_t) dst.data) & 15)) return false;
    if ((dst.nb[1] % 16) || (dst.nb[2] % 16)) return false;
    return true;
}

// how many workgroups share the cells of one (token, head) — 1 unless the row kernel serves the op with few pairs over a cache of several blocks.  Every split walks whole groups of
// 256 cells (a block of 64 per wave)
int attn_f32_row_splits(const tdesc & q, const tdesc & k, const tdesc & v, const tdesc * mask, const tdesc & dst) {
    static const bool on = !getenv("GGML_MI355X_ATTN_SPLIT") || atoi(getenv("GGML_MI355X_ATTN_SPLIT")) != 0;
    static const bool mma_on = !getenv("GGML_MI355X_ATTN_MMA") || atoi(getenv("GGML_MI355X_ATTN_MMA")) != 0;
    const int64_t pairs = q.ne[1] * q.ne[2], groups = (k.ne[1] + 255) / 256;
    if (!on || groups < 2 || pairs >= 512) return 1;
    if (mask && q.ne[1] >= 32 && q.ne[0] <= 128 && v.ne[0] <= 128) return 1;  // (the tile or the matrix-core kernel)
    if (mma_on && (attn_mma_bf16_wide_ok(q, k, v, mask, dst) || attn_mma_bf16_ok(q, k, v, mask, dst))) return 1;
    return (int) std::max<int64_t>(1, std::min<int64_t>({groups, (int64_t) ATTN_F32_MAX_SPLITS, 1024 / std::max<int64_t>(1, pairs)}));
}
size_t attn_f32_workspace_bytes(const tdesc & q, const tdesc & k, const tdesc & v, const tdesc * mask, const tdesc & dst) {
    const int S = attn_f32_row_splits(q, k, v, mask, dst);
    return S > 1 ? (size_t) q.ne[1] * (size_t) q.ne[2] * (size_t) S * (size_t) (v.ne[0] + 2) * sizeof(float) : 0;
}

static bool attn_f32_type_ok(int t) { return t == GGML_TYPE_F32 || t == GGML_TYPE_BF16 || t == GGML_TYPE_F16; }

// may launch_attn_f32 serve this op?  q f32 [DK, n_q, H], k [DK, n_kv, G], v [DV, n_kv, G] of one type each, rows contiguous, one batch
bool attn_f32_applies(const tdesc & q, const tdesc & k, const tdesc & v, const tdesc * mask, const tdesc & dst) {
    if (q.type != GGML_TYPE_F32 || dst.type != GGML_TYPE_F32 || !attn_f32_type_ok(k.type) || !attn_f32_type_ok(v.type)) return false;
    if (q.ne[0] != k.ne[0] || k.ne[1] != v.ne[1] || k.ne[2] != v.ne[2] || k.ne[2] <= 0 || q.ne[2] % k.ne[2] != 0) return false;
    if (q.ne[0] < 1 || q.ne[0] > ATTN_F32_MAX_D || v.ne[0] < 1 || v.ne[0] > ATTN_F32_MAX_D) return false;
    if (q.ne[3] != 1 || k.ne[3] != 1 || v.ne[3] != 1) return false;
    if (q.nb[0] != 4 || dst.nb[0] != 4 || k.nb[0] != (k.type == GGML_TYPE_F32 ? 4 : 2) || v.nb[0] != (v.type == GGML_TYPE_F32 ? 4 : 2)) return false;
    if (dst.ne[0] != v.ne[0] || dst.ne[1] != q.ne[2] || dst.ne[2] != q.ne[1]) return false;
    if (mask && ((mask->type != GGML_TYPE_F16 && mask->type != GGML_TYPE_F32) || mask->ne[0] < k.ne[1] || mask->ne[1] < q.ne[1] || mask->ne[2] != 1 || mask->ne[3] != 1)) return false;
    return true;
}

template <int KT, int VT>
static void attn_f32_launch_t(hipStream_t s, const tdesc & q, const tdesc & k, const tdesc & v, const tdesc * mask, const float * sinks, const float * r12, const tdesc & dst, float scale,
                              const float * sig, float softcap, int pen_kind, const attn_f32_extra & x) {
    const int64_t n_q = q.ne[1], H = q.ne[2];
    const int DK = (int) q.ne[0], DV = (int) v.ne[0];
    if constexpr (KT == GGML_TYPE_BF16 && VT == GGML_TYPE_BF16) {
        static const bool mma_on = !getenv("GGML_MI355X_ATTN_MMA") || atoi(getenv("GGML_MI355X_ATTN_MMA")) != 0;
        if (mma_on && attn_mma_bf16_wide_ok(q, k, v, mask, dst)) {  // one shared key/value head with wide rows (latent attention): four waves per 32 (token, head) pairs
            const dim3 grid((unsigned) ((n_q * H + 31) / 32));
            const int dkq = ((DK + 15) / 16 + 3) / 4, dvq = ((DV + 31) / 32 + 3) / 4;  // per wave: 16-entry key groups (<= 10), 32-entry value tiles (<= 4)
#define MI_ATT_WIDE(A, B) hipLaunchKernelGGL((k_attn_mma_bf16_wide<A, B>), grid, dim3(256), 0, s, q, k, v, *mask, sinks, r12, dst, scale, sig, softcap, pen_kind)
            const int a = dkq <= 3 ? 3 : (dkq <= 5 ? 5 : 10), b = dvq <= 1 ? 1 : (dvq <= 2 ? 2 : 4);
            if (a == 3 && b == 1) MI_ATT_WIDE(3, 1); else if (a == 3 && b == 2) MI_ATT_WIDE(3, 2); else if (a == 3) MI_ATT_WIDE(3, 4);
            else if (a == 5 && b == 1) MI_ATT_WIDE(5, 1); else if (a == 5 && b == 2) MI_ATT_WIDE(5, 2); else if (a == 5) MI_ATT_WIDE(5, 4);
            else if (b == 1) MI_ATT_WIDE(10, 1); else if (b == 2) MI_ATT_WIDE(10, 2); else MI_ATT_WIDE(10, 4);
#undef MI_ATT_WIDE
            return;
        }
        if (mma_on && attn_mma_bf16_ok(q, k, v, mask, dst)) {  // prompt portions over a bf16 cache: the matrix cores
            const dim3 grid((unsigned) ((n_q + 31) / 32), (unsigned) H);
            const int dk16 = (DK + 15) / 16, dvt = (DV + 31) / 32;
            const bool plain = !sig && !r12 && softcap <= 0.0f && DK == 16 * dk16 && DV == 32 * dvt;
#define MI_ATT_MMA2(A, B, P) hipLaunchKernelGGL((k_attn_mma_bf16<A, B, P>), grid, dim3(256), 0, s, q, k, v, *mask, sinks, r12, dst, scale, sig, softcap, pen_kind)
#define MI_ATT_MMA(A, B) do { if (plain && dk16 == A && dvt == B) MI_ATT_MMA2(A, B, true); else MI_ATT_MMA2(A, B, false); } while (0)
            const int a = dk16 <= 2 ? 2 : (dk16 <= 4 ? 4 : (dk16 <= 6 ? 6 : 8)), b = dvt <= 1 ? 1 : (dvt <= 2 ? 2 : (dvt <= 3 ? 3 : 4));
            if (a == 2 && b == 1) MI_ATT_MMA(2, 1); else if (a == 2 && b == 2) MI_ATT_MMA(2, 2); else if (a == 2) MI_ATT_MMA(2, 4);
            else if (a == 6 && b == 3) MI_ATT_MMA(6, 3);
            else if (b == 3) MI_ATT_MMA(8, 4);  // (between the tilings: the next larger one)
            else if (a == 6 && b == 4) MI_ATT_MMA(8, 4);
            else if (a == 6 && b == 2) MI_ATT_MMA(8, 2);
            else if (a == 6) MI_ATT_MMA(8, 1);
            else if (a == 4 && b == 1) MI_ATT_MMA(4, 1); else if (a == 4 && b == 2) MI_ATT_MMA(4, 2); else if (a == 4) MI_ATT_MMA(4, 4);
            else if (b == 1) MI_ATT_MMA(8, 1); else if (b == 2) MI_ATT_MMA(8, 2); else MI_ATT_MMA(8, 4);
#undef MI_ATT_MMA
#undef MI_ATT_MMA2
            return;
        }
    }
    // the tile kernel: batches of 32 queries and more under a mask, head sizes up to 128 (its LDS: 64 cells of K and V plus 64 queries as f32)
    if (mask && n_q >= 32 && DK <= 128 && DV <= 128) {
        const dim3 grid((unsigned) ((n_q + 63) / 64), (unsigned) H);
        auto go = [&](auto kern, int dkp, int dvp) {
            const size_t lds = ((size_t) 64 * (dkp + 1) + (size_t) 64 * dvp + (size_t) 64 * dkp) * sizeof(float);
            // (more than the 64 KB a kernel gets by default: up to 97 KB of the CU's 160 KB; the attribute is per device and cheap to set again)
            if (lds > 48 * 1024) (void) hipFuncSetAttribute((const void *) kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int) lds);
            hipLaunchKernelGGL(kern, grid, dim3(256), lds, s, q, k, v, *mask, sinks, r12, dst, scale, sig, softcap, pen_kind);
        };
        const bool k64 = DK <= 64, v64 = DV <= 64;
        if (k64 && v64) go(k_attn_f32_tile<KT, VT, 64, 64>, 64, 64);
        else if (k64) go(k_attn_f32_tile<KT, VT, 64, 128>, 64, 128);
        else if (v64) go(k_attn_f32_tile<KT, VT, 128, 64>, 128, 64);
        else go(k_attn_f32_tile<KT, VT, 128, 128>, 128, 128);
        return;
    }
    const int S = attn_f32_row_splits(q, k, v, mask, dst);
    const bool split = S > 1 && x.ws && attn_f32_workspace_bytes(q, k, v, mask, dst) <= x.ws_bytes;
    const dim3 grid((unsigned) n_q, (unsigned) H, split ? (unsigned) S : 1u);
    bool served = false;
    if constexpr (KT == VT && KT != GGML_TYPE_F32) {
        if (attn_f32_rows128_ok(q, k, v, r12, sig, softcap)) {
            const attn_rows_args a{q.data, k.data, v.data, mask ? mask->data : nullptr, sinks, dst.data, (float *) x.ws, q.nb[1], q.nb[2], k.nb[1], k.nb[2], v.nb[1], v.nb[2], mask ? mask->nb[1] : 0,
                                   dst.nb[1], dst.nb[2], (int) k.ne[1], DK, DV, (int) H, (int) (H / k.ne[2]), mask && mask->type == GGML_TYPE_F16 ? 1 : 0, scale};
            hipLaunchKernelGGL(k_attn_f32_rows128<KT>, grid, dim3(256), 0, s, a);
            served = true;
        }
    }
    if (!served)
        hipLaunchKernelGGL((k_attn_f32_rows<KT, VT>), grid, dim3(256), 0, s, q, k, v, mask ? *mask : q, mask ? 1 : 0, sinks, r12, dst, scale, sig,
                       softcap, pen_kind, (float *) x.ws);
    if (!split) return;
    tdesc o = dst;
    if (x.gate) o.data = (char *) x.gated;
    hipLaunchKernelGGL(k_attn_f32_combine, dim3((unsigned) n_q, (unsigned) H), dim3(128), 0, s, (const float *) x.ws, S, (int) H, DV, o, sig ? 1 : 0, x.gate, x.gate_heads);
}

void launch_attn_f32(hipStream_t s, const tdesc & q, const tdesc & k, const tdesc & v, const tdesc * mask, const float * sinks, const float * r12, const tdesc & dst, float scale,
                     const float * sig, float softcap, int pen_kind, const attn_f32_extra & x) {
    if (q.ne[1] == 0 || q.ne[2] == 0) return;
#define MI_ATTN_F32_CASE(KT, VT) if (k.type == KT && v.type == VT) { attn_f32_launch_t<KT, VT>(s, q, k, v, mask, sinks, r12, dst, scale, sig, softcap, pen_kind, x); return; }
    MI_ATTN_F32_CASE(GGML_TYPE_F32, GGML_TYPE_F32)
    MI_ATTN_F32_CASE(GGML_TYPE_BF16, GGML_TYPE_BF16)
    MI_ATTN_F32_CASE(GGML_TYPE_F16, GGML_TYPE_F16)
    MI_ATTN_F32_CASE(GGML_TYPE_F32, GGML_TYPE_BF16)
    MI_ATTN_F32_CASE(GGML_TYPE_BF16, GGML_TYPE_F32)
    MI_ATTN_F32_CASE(GGML_TYPE_F32, GGML_TYPE_F16)
    MI_ATTN_F32_CASE(GGML_TYPE_F16, GGML_TYPE_F32)
    MI_ATTN_F32_CASE(GGML_TYPE_BF16, GGML_TYPE_F16)
    MI_ATTN_F32_CASE(GGML_TYPE_F16, GGML_TYPE_BF16)
#undef MI_ATTN_F32_CASE
}

MI_TU_TOUCH(attn_f32)

}  // namespace mi355x
