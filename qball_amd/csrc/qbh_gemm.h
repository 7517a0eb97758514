// Hand-written matrix-core GEMMs of the Γ projector contractions (qbh_gemm.hip).
#pragma once
#include <hip/hip_runtime.h>

namespace qbh {

// Slices the reduction of an R x C output with reduction length Q is cut into, at most 64; the
// count actually used (every slice non-empty).  want > 0: that many, each slice at least 512
// long.  Else FP32: enough for about 2048 workgroups of the 128 x 128 tile, each slice at least
// 512 long, whatever the tile; FP64: the same with that tile, and the cheapest count with a
// smaller one, slices down to 64 long (tile_cost).
int mfma_slices(bool fp32, int R, int C, long Q, int want);
// Length of each slice for `slices` slices (a multiple of the 16-element stage).
long mfma_slice_len(long Q, int slices);

// O_s[r + c ldo] = sum_{q in slice s} X[q + r ldx] Y[q + c ldy], s < slices, with
// O_s = O + s ostride (the fnl product: r = projector, c = band, q = real-view row).
// FP64 or FP32 operands and outputs.  Returns 0, or -1 for invalid sizes.
int mfma_gemm_qq(hipStream_t st, bool fp32, int R, int C, long Q, const void* X, long ldx,
                 const void* Y, long ldy, void* O, long ldo, int slices, long ostride);

// O[c + r ldo] (+)= sum_q X[q + r ldx] Y[c + q ldy] (the enl product taken transposed:
// r = band, c = real-view row, q = projector; X = F, Y = the projector table).
int mfma_gemm_qc(hipStream_t st, bool fp32, int R, int C, long Q, const void* X, long ldx,
                 const void* Y, long ldy, void* O, long ldo, bool accumulate);

// FP64, lower triangle (r >= c) of the symmetric product, whole tiles of it:
// O_s[r + c R] = sum_{q in slice s} X[q + r ldx] X[q + c ldx], s < slices (as mfma_gemm_qq; the
// count from mfma_sym_slices).
int mfma_sym_slices(int R, long Q);
int mfma_gemm_sym(hipStream_t st, int R, long Q, const double* X, long ldx, double* O, int slices,
                  long ostride);

// FP64, X lower triangular (zero above its diagonal): O[c + r ldo] = sum_{q <= r} X[q + r ldx]
// Y[c + q ldy], q < R (as mfma_gemm_qc without the zero half of the reduction; O apart from Y).
int mfma_gemm_tri(hipStream_t st, int R, int C, const double* X, long ldx, const double* Y,
                  long ldy, double* O, long ldo);

// Width of the tiles (32, 64, 128), and the slices, of a product of these sizes under the
// built-in rule, for the tests: which 0, 1: F in FP64, FP32 (mfma_gemm_qq); 2, 3: βF
// (mfma_gemm_qc; mfma_gemm_tri is as 2); 4: the symmetric product (C = R).
extern "C" int qbh_product_tile(int which, int R, int C, long Q, int* slices);

}  // namespace qbh
