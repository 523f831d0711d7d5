// mmq_args.h — argument block shared by the integer matrix-core mat-mul kernels (mmq_i8.hip: prompt batches; mmq_skinny.hip:
// continuous-batching decode steps of <= 32 columns).
#pragma once
#include "dev_util.h"
#include "kernels.h"

namespace mi355x {

// Up to three weight matrices of one type that multiply the SAME activations (wq / wk / wv, ffn_gate / ffn_up) share a launch:
// their row panels form one list (matrix i owns panels [panel0_i, panel0_{i+1})), which fills the chip where each of them
// alone needed a K split — and a second kernel — to do so.
struct mmq8_mat {
    const uint8_t * W;
    int64_t w_nb1;
    int N, panel0;
    float * dst;
    int64_t dst_stride;
    float * part;        // ksplit > 1: partial [ksplit][M][N] results of this matrix (summed in a fixed order by k_splitk_reduce)
    const float * add;   // optional epilogue: + add[m * add_stride + n] (bias row: stride 0, residual: stride N)
    int64_t add_stride;
    int qt;              // two-format launches of the skinny kernel: 4 / 5 / 6 = how THIS matrix is stored (0 otherwise)
};
struct mmq8_args {
    mmq8_mat mat[3];
    int n_mat;
    int K, M;
    const q8k_dev * act;  // [M][K/256]
    int n_panels, m_tiles;
    int ksplit;          // > 1: blockIdx.y owns a contiguous range of super-blocks and writes its partial result
    int has_epi;         // skinny kernel: `epi` describes what happens to the results instead of the plain store
    mmq_epi epi;
};

void launch_mmq_skinny(hipStream_t s, int type, const mmq8_args & a);
// matrices of two K-quant formats in one launch (a.mat[].qt set); false: this pair of formats is not built
bool launch_mmq_skinny_mixed(hipStream_t s, const mmq8_args & a);
// prompt batches on the same unit (mmq_skinny.hip): 0 = not there, 1 = k_mmq_wide (no K split), 2 / 3 = k_mmq_wide_few with that many token tiles a workgroup
int mmq_wide_form(int type, int64_t K, const int64_t * N, int n_mat, int64_t M, int64_t w_nb1);
int mmq_wide_ksplit(int type, int64_t K, int64_t N, int64_t M);  // K slices of such a launch (0: it does not apply)
int mmq_tiled_ksplit(int64_t K, int64_t N, int64_t M);  // K slices of the tiled GEMM (mmq_i8.hip; Q6_K of more than 64 columns: mmq_q6_tile)
struct q6_tile { int bn, ks; double us; };  // its panel rows, K slices and expected time for a Q6_K product of more than 64 columns
q6_tile mmq_q6_tile(int64_t K, int64_t N, int64_t M);
double q6_slices_us(int64_t N, int64_t M, int64_t ks);  // ... the part of that time that its slices cost
void launch_mmq_wide(hipStream_t s, int type, int form, const mmq8_args & a);  // mmq_skinny.hip; a.mat[].panel0 / n_panels are set by the launcher

}  // namespace mi355x
