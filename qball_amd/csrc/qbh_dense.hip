// Dense band-space operations in FP64 on gfx950: overlap matrix + Cholesky
// orthonormalisation (SlaterDet::gram, src/qball/SlaterDet.cc:1043-1143) and subspace
// diagonalisation (Wavefunction::diag, src/qball/Wavefunction.cc:1510-1715).
//
// The band-space products S = C^H X (nst x nst, contraction over ~1e5 plane waves) run as
// K-split strided-batched rocBLAS GEMMs whose slices are summed by one kernel that also
// applies the Γ weights (2 Re sum over the half sphere, G = 0 counted once); the subspace
// eigensolver is rocSOLVER's (syevd/heevd), as is the factorisation of complex bases (potrf,
// trsm).
//
// Γ orthonormalisation runs on this library's kernels: the lower tiles of S = 2 C^T C - c0 c0^T
// on the matrix cores (half the product), a blocked Cholesky factorisation S = L L^T and the
// inverse of L in 64 x 64 blocks, and C L^-T as one matrix-core product that skips the zero
// half of L^-1 (in place of a triangular solve).
#include <hip/hip_runtime.h>
#include <rocblas/rocblas.h>
#include <rocsolver/rocsolver.h>

#include <algorithm>
#include <string>
#include <vector>

#include "../../include/qbh.h"
#include "qbh_gemm.h"
#include "qbh_ham.h"

namespace qbh {
Basis* basis_of(qbh_basis b);
Ctx* ctx_of_basis(qbh_basis b);
}  // namespace qbh

using namespace qbh;

static int dfail(Ctx* c, int code, const std::string& msg) {
  c->last_error = msg;
  return code;
}

// S = alpha * sum_k P[k] - (real ? a0 b0^T : 0), P slices of M*N (complex: 2*M*N doubles)
__global__ void k_sum_band_splits(int M, int N, int nsplit, int cplx, const double* __restrict__ P,
                                  double alpha, const double* __restrict__ A, long lda,
                                  const double* __restrict__ B, long ldb, int real,
                                  double* __restrict__ S) {
  const long e = cplx ? 2 : 1;
  const long total = (long)M * N * e;
  const long i = blockIdx.x * 256L + threadIdx.x;
  if (i >= total) return;
  double s = P[i];
  for (int k = 1; k < nsplit; ++k) s += P[(long)k * total + i];
  s = alpha * s;
  if (real) {
    const long m = i % M, n = i / M;
    s -= A[m * lda] * B[n * ldb];  // rank-1 G = 0 correction (ger -1.0 on row 0)
  }
  S[i] = s;
}

// S (M x N, ld M) = alpha * A^T B (real view, K rows) or A^H B (complex, K rows)
int qbh::band_product(Ctx* c, void* bhv, bool real, int M, int N, long K, const double* A,
                      long lda, const double* B, long ldb, double alpha, double* S,
                      double*& scratch, size_t& scratch_bytes) {
  rocblas_handle bh = static_cast<rocblas_handle>(bhv);
  const long tiles = (long)((M + 127) / 128) * ((N + 127) / 128);
  long ns = std::min<long>((4096 + tiles - 1) / tiles, 32);
  ns = std::max<long>(1, std::min<long>(ns, K / 1024));
  const long kc = (K + ns - 1) / ns;
  const long nfull = K / kc, rem = K - nfull * kc;
  const int nparts = (int)(nfull + (rem ? 1 : 0));
  const size_t e = real ? 1 : 2;
  const size_t need = sizeof(double) * e * (size_t)M * N * nparts;
  if (scratch_bytes < need) {
    if (scratch) hipFree(scratch);
    scratch = nullptr;
    scratch_bytes = 0;
    if (hipMalloc(&scratch, need) != hipSuccess) return dfail(c, QBH_ERR_ALLOC, "band product scratch");
    scratch_bytes = need;
  }
  rocblas_status st = rocblas_status_success;
  const long pst = (long)M * N;  // partial stride in BLAS elements
  if (real) {
    const double one = 1.0, zero = 0.0;
    if (nfull > 0)
      st = rocblas_dgemm_strided_batched(bh, rocblas_operation_transpose, rocblas_operation_none, M,
                                         N, (int)kc, &one, A, lda, kc, B, ldb, kc, &zero, scratch,
                                         M, pst, (int)nfull);
    if (st == rocblas_status_success && rem)
      st = rocblas_dgemm(bh, rocblas_operation_transpose, rocblas_operation_none, M, N, (int)rem,
                         &one, A + nfull * kc, lda, B + nfull * kc, ldb, &zero,
                         scratch + nfull * pst, M);
  } else {
    const rocblas_double_complex one(1.0, 0.0), zero(0.0, 0.0);
    auto* Az = reinterpret_cast<const rocblas_double_complex*>(A);
    auto* Bz = reinterpret_cast<const rocblas_double_complex*>(B);
    auto* Pz = reinterpret_cast<rocblas_double_complex*>(scratch);
    if (nfull > 0)
      st = rocblas_zgemm_strided_batched(bh, rocblas_operation_conjugate_transpose,
                                         rocblas_operation_none, M, N, (int)kc, &one, Az, lda, kc,
                                         Bz, ldb, kc, &zero, Pz, M, pst, (int)nfull);
    if (st == rocblas_status_success && rem)
      st = rocblas_zgemm(bh, rocblas_operation_conjugate_transpose, rocblas_operation_none, M, N,
                         (int)rem, &one, Az + nfull * kc, lda, Bz + nfull * kc, ldb, &zero,
                         Pz + nfull * pst, M);
  }
  if (st != rocblas_status_success)
    return dfail(c, QBH_ERR_BLAS, std::string("band product: ") + rocblas_status_to_string(st));
  const long total = (long)M * N * e;
  k_sum_band_splits<<<(unsigned)((total + 255) / 256), 256, 0, c->stream>>>(
      M, N, nparts, real ? 0 : 1, scratch, alpha, A, lda, B, ldb, real ? 1 : 0, S);
  return 0;
}

namespace {
struct Scratch {
  double* p = nullptr;
  size_t bytes = 0;
  ~Scratch() {
    if (p) hipFree(p);
  }
};
}  // namespace

// ------------------------------------------------------------------------------------
// Blocked Cholesky factorisation and triangular inverse, FP64.  S is n x n, column-major, lower
// triangle (S[i + j n], i >= j), overwritten below its diagonal blocks by L; W receives L^-1,
// row-major (W[i n + j]), zero above the diagonal; T is scratch.  Per 64-wide block column: the
// diagonal block (one workgroup: elimination of [A | 1], one barrier a column), the panel
// L_ik = A_ik L_kk^-T, the trailing update A_ij -= L_ik L_jk^T; then the inverse by doubling,
// [A 0; B C]^-1 = [A^-1 0; -C^-1 B A^-1 C^-1].  Bound by the latency of the n sequential columns
// (about 0.6 us each) and of the launches.  Whole orthonormalisation against rocBLAS products,
// rocSOLVER potrf and rocBLAS trsm, MI355X: 16 bands of 1151 plane waves 129 -> 82 us, 64 of
// 5198 272 -> 99, 128 of 9139 525 -> 247, 512 of 37963 2.99 -> 2.01 ms, 1024 of 72919 12.7 -> 8.4
// (product 2.9, factor and inverse 1.5, rotation 3.9); errors against 64-bit references the same.
constexpr int CB = 64;       // block
constexpr int CS = CB + 1;   // LDS row

// Diagonal block: elimination of [A | 1] without pivoting, one column and one barrier a step.
// Thread (i, g) holds the elements m = g (mod 4) of row i of A (those from the current column
// group on, shifted down as the groups are done) and of X in registers; a step exchanges column
// j of A and row j of X through LDS, in the order the readers hold them.
__global__ void __launch_bounds__(256)
k_chol_diag(int n, int k0, const double* __restrict__ S, double* __restrict__ W,
            int* __restrict__ info) {
  // column j of A at [m % 4][m / 4 - j / 4], then row j of X at [m % 4][m / 4]; two buffers
  __shared__ double xch[2][2][4][16];
  __shared__ double piv[CB];
  const int nb = min(CB, n - k0);
  const int i = threadIdx.x & 63, g = threadIdx.x >> 6;
  double a[16], x[16];
#pragma unroll
  for (int u = 0; u < 16; ++u) {
    const int m = g + 4 * u;
    a[u] = i < nb && m <= i ? S[(long)(k0 + i) + (long)(k0 + m) * n] : (i == m ? 1.0 : 0.0);
    x[u] = i == m ? 1.0 : 0.0;
  }
  for (int jj = 0; jj < CB / 4; ++jj) {
#pragma unroll
    for (int gj = 0; gj < 4; ++gj) {
      const int j = 4 * jj + gj;
      double (*col)[16] = xch[gj & 1][0];
      double (*row)[16] = xch[gj & 1][1];
      if (g == gj && i >= 4 * jj) col[i & 3][(i >> 2) - jj] = a[0];
      if (i == j)
#pragma unroll
        for (int u = 0; u < 16; ++u) row[g][u] = x[u];
      __syncthreads();
      const double p = col[gj][0];
      if (threadIdx.x == 0) {
        piv[j] = p;
        if (j < nb && !(p > 0.0) && *info == 0) *info = k0 + j + 1;
      }
      if (i > j) {
        const double f = col[i & 3][(i >> 2) - jj] / p;
#pragma unroll
        for (int u = 0; u < 16; ++u)
          if (jj + u < 16) a[u] -= f * col[g][u];
#pragma unroll
        for (int u = 0; u < 16; ++u) x[u] -= f * row[g][u];
      }
    }
#pragma unroll
    for (int u = 0; u < 15; ++u) a[u] = a[u + 1];
    a[15] = 0.0;
  }
  __syncthreads();
  if (i < nb) {
    const double s = sqrt(piv[i]);
#pragma unroll
    for (int u = 0; u < 16; ++u) {
      const int m = g + 4 * u;
      if (m < nb) W[(long)(k0 + i) * n + k0 + m] = m <= i ? x[u] / s : 0.0;
    }
  }
}

// acc[a][b] += sum_m U[ty + 16 a][m] V[tx + 16 b][m] over one staged block pair
__device__ __forceinline__ void block_fma(const double* U, const double* V, int tx, int ty,
                                          double (&acc)[4][4]) {
#pragma unroll 4
  for (int m = 0; m < CB; ++m) {
    double u[4], v[4];
#pragma unroll
    for (int a = 0; a < 4; ++a) {
      u[a] = U[(ty + 16 * a) * CS + m];
      v[a] = V[(tx + 16 * a) * CS + m];
    }
#pragma unroll
    for (int a = 0; a < 4; ++a)
#pragma unroll
      for (int b = 0; b < 4; ++b) acc[a][b] += u[a] * v[b];
  }
}

// L_ik = A_ik W_kk^T (W_kk = L_kk^-1), in place; block row k + 1 + blockIdx.x
__global__ void __launch_bounds__(256)
k_chol_panel(int n, int k0, double* __restrict__ S, const double* __restrict__ W) {
  __shared__ double U[CB * CS], V[CB * CS];
  const int i0 = k0 + CB * (1 + blockIdx.x);
  for (int e = threadIdx.x; e < CB * CB; e += 256) {
    const int i = e % CB, m = e / CB;
    U[i * CS + m] = i0 + i < n ? S[(long)(i0 + i) + (long)(k0 + m) * n] : 0.0;
    V[m * CS + i] = W[(long)(k0 + m) * n + k0 + i];  // row m of W_kk, element i
  }
  __syncthreads();
  const int tx = threadIdx.x & 15, ty = threadIdx.x >> 4;
  double acc[4][4] = {};
  block_fma(U, V, ty, tx, acc);  // rows of A run along tx: consecutive lanes store consecutively
#pragma unroll
  for (int a = 0; a < 4; ++a)
#pragma unroll
    for (int b = 0; b < 4; ++b) {
      const int i = i0 + tx + 16 * a, j = k0 + ty + 16 * b;
      if (i < n) S[(long)i + (long)j * n] = acc[a][b];
    }
}

// A_ij -= L_ik L_jk^T for the block pairs i >= j > k
__global__ void __launch_bounds__(256)
k_chol_trail(int n, int k0, double* __restrict__ S) {
  __shared__ double U[CB * CS], V[CB * CS];
  int bi = (int)((sqrtf(8.0f * blockIdx.x + 1.0f) - 1.0f) * 0.5f);
  while ((bi + 1) * (bi + 2) / 2 <= (int)blockIdx.x) ++bi;
  while (bi * (bi + 1) / 2 > (int)blockIdx.x) --bi;
  const int bj = blockIdx.x - bi * (bi + 1) / 2;
  const int i0 = k0 + CB * (1 + bi), j0 = k0 + CB * (1 + bj);
  for (int e = threadIdx.x; e < CB * CB; e += 256) {
    const int i = e % CB, m = e / CB;
    U[i * CS + m] = i0 + i < n ? S[(long)(i0 + i) + (long)(k0 + m) * n] : 0.0;
    V[i * CS + m] = j0 + i < n ? S[(long)(j0 + i) + (long)(k0 + m) * n] : 0.0;
  }
  __syncthreads();
  const int tx = threadIdx.x & 15, ty = threadIdx.x >> 4;
  double acc[4][4] = {};
  block_fma(U, V, ty, tx, acc);
#pragma unroll
  for (int a = 0; a < 4; ++a)
#pragma unroll
    for (int b = 0; b < 4; ++b) {
      const int i = i0 + tx + 16 * a, j = j0 + ty + 16 * b;
      if (i < n && j <= i) S[(long)i + (long)j * n] -= acc[a][b];
    }
}

// One doubling step over pairs of h-block triangles: FIRST: T = B A^-1, else W = -C^-1 T on the
// blocks (C rows, A columns).  blockIdx: x = block column within A, y = block row within C,
// z = pair.
template <bool FIRST>
__global__ void __launch_bounds__(256)
k_tri_double(int n, int h, const double* __restrict__ S, double* __restrict__ W,
             double* __restrict__ T) {
  __shared__ double U[CB * CS], V[CB * CS];
  const int nblk = (n + CB - 1) / CB;
  const int b0 = blockIdx.z * 2 * h, bi = b0 + h + blockIdx.y, bj = b0 + blockIdx.x;
  if (bi >= nblk) return;
  const int i0 = bi * CB, j0 = bj * CB;
  const int tx = threadIdx.x & 15, ty = threadIdx.x >> 4;
  double acc[4][4] = {};
  // A^-1 (FIRST) and C^-1 are lower triangular: only blocks m >= j, m <= i
  const int m0 = FIRST ? bj : b0 + h, m1 = FIRST ? b0 + h : bi + 1;
  for (int bm = m0; bm < m1; ++bm) {
    const int k0 = bm * CB;
    __syncthreads();
    for (int e = threadIdx.x; e < CB * CB; e += 256) {
      const int x = e % CB, y = e / CB;
      // U: row i, element m; V: column j, element m
      if (FIRST) {
        U[x * CS + y] = i0 + x < n ? S[(long)(i0 + x) + (long)(k0 + y) * n] : 0.0;
        V[x * CS + y] = W[(long)(k0 + y) * n + j0 + x];
      } else {
        U[y * CS + x] = i0 + y < n && k0 + x < n ? W[(long)(i0 + y) * n + k0 + x] : 0.0;
        V[x * CS + y] = k0 + y < n ? T[(long)(k0 + y) * n + j0 + x] : 0.0;
      }
    }
    __syncthreads();
    block_fma(U, V, tx, ty, acc);
  }
#pragma unroll
  for (int a = 0; a < 4; ++a)
#pragma unroll
    for (int b = 0; b < 4; ++b) {
      const int i = i0 + ty + 16 * a, j = j0 + tx + 16 * b;
      if (i >= n) continue;
      if (FIRST)
        T[(long)i * n + j] = acc[a][b];
      else
        W[(long)i * n + j] = -acc[a][b];
    }
}

__global__ void k_dense_zero(long n, double* __restrict__ p, int* __restrict__ info) {
  const long i = blockIdx.x * 256L + threadIdx.x;
  if (i < n) p[i] = 0.0;
  if (i == 0) *info = 0;
}

// lower triangle of S = 2 sum_k P[k] - c0 c0^T (column-major slices of n x n)
__global__ void __launch_bounds__(256)
k_sum_lower(int n, int nsplit, const double* __restrict__ P, const double* __restrict__ c0, long ld,
            double* __restrict__ S) {
  const int j = blockIdx.y;
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i >= n || i < j) return;
  const long e = i + (long)j * n, st = (long)n * n;
  double s = P[e];
  int k = 1;
  for (; k + 4 <= nsplit; k += 4) {
    const double a = P[k * st + e], b = P[(k + 1) * st + e], c = P[(k + 2) * st + e],
                 d = P[(k + 3) * st + e];
    s += a;
    s += b;
    s += c;
    s += d;
  }
  for (; k < nsplit; ++k) s += P[k * st + e];
  S[e] = 2.0 * s - c0[i * ld] * c0[j * ld];
}

// psi (rows of w doubles from column q0, leading dimension ld) = src (compact), unless the
// factorisation failed; grid (ceil(w / 512), bands)
__global__ void __launch_bounds__(256)
k_store_rows(long w, const double* __restrict__ src, double* __restrict__ psi, long ld,
             const int* __restrict__ info) {
  if (*info) return;
  const long q = (blockIdx.x * 256L + threadIdx.x) * 2;
  if (q >= w) return;  // w is even
  const double* s = src + blockIdx.y * w + q;
  double* d = psi + blockIdx.y * ld + q;
  const double a = s[0], b = s[1];
  d[0] = a;
  d[1] = b;
}

// Γ orthonormalisation of n bands of K = 2 ngw reals (ld doubles apart); info (host) receives 0 or
// the order of the first non-positive pivot (psi is then left as it was)
static int gram_real(Ctx* c, int n, long K, double* psi, long ld, int* hinfo) {
  const int slices = mfma_sym_slices(n, K);
  const size_t nn = (size_t)n * n;
  // partials, S, W, T and the pivot flag
  CallBuffer buf(c, sizeof(double) * ((slices + 3) * nn + 2));
  double* P = static_cast<double*>(buf.p);
  // rotated bands, whole or a range of coefficients at a time within the workspace cap (and what
  // memory there is)
  const size_t room = std::max<size_t>(c->ws_cap / (8 * (size_t)n), 128);
  long w = (size_t)K <= room ? K : (long)(room / 128 * 128);
  double* out = static_cast<double*>(ws_get(c, sizeof(double) * w * n));
  while (!out && w > 128) {
    w = std::max(w / 256 * 128, 128L);
    out = static_cast<double*>(ws_get(c, sizeof(double) * w * n));
  }
  if (!P || !out) return dfail(c, QBH_ERR_ALLOC, "gram scratch allocation failed");
  double* S = P + slices * nn;
  double* W = S + nn;
  double* T = W + nn;
  int* info = reinterpret_cast<int*>(T + nn);
  hipStream_t st = c->stream;
  {
    TimedLaunch tl(c, "gram_product");
    if (mfma_gemm_sym(st, n, K, psi, ld, P, slices, (long)nn))
      return dfail(c, QBH_ERR_ARG, "gram: invalid sizes");
    k_sum_lower<<<dim3((n + 255) / 256, n), 256, 0, st>>>(n, slices, P, psi, ld, S);
  }
  {
    TimedLaunch tl(c, "gram_cholesky");
    k_dense_zero<<<(unsigned)((nn + 255) / 256), 256, 0, st>>>((long)nn, W, info);
    const int nblk = (n + CB - 1) / CB;
    for (int k = 0; k < nblk; ++k) {
      k_chol_diag<<<1, 256, 0, st>>>(n, k * CB, S, W, info);
      const int rest = nblk - k - 1;
      if (rest == 0) break;
      k_chol_panel<<<rest, 256, 0, st>>>(n, k * CB, S, W);
      k_chol_trail<<<rest * (rest + 1) / 2, 256, 0, st>>>(n, k * CB, S);
    }
    for (int h = 1; h < nblk; h *= 2) {
      const dim3 grid(h, h, (nblk + 2 * h - 1) / (2 * h));
      k_tri_double<true><<<grid, 256, 0, st>>>(n, h, S, W, T);
      k_tri_double<false><<<grid, 256, 0, st>>>(n, h, S, W, T);
    }
  }
  for (long q = 0; q < K; q += w) {
    const long m = std::min(w, K - q);
    TimedLaunch tl(c, "gram_rotate");
    if (mfma_gemm_tri(st, n, (int)m, W, n, psi + q, ld, out, m))
      return dfail(c, QBH_ERR_ARG, "gram: invalid sizes");
    k_store_rows<<<dim3((unsigned)((m + 511) / 512), n), 256, 0, st>>>(m, out, psi + q, ld, info);
  }
  hipMemcpyAsync(hinfo, info, sizeof(int), hipMemcpyDeviceToHost, st);
  hipStreamSynchronize(st);
  return 0;
}

extern "C" int qbh_gram(qbh_basis basis, double* psi_dev, long ld, int nst) {
  if (!basis || !psi_dev || nst <= 0) return QBH_ERR_ARG;
  Basis* b = basis_of(basis);
  Ctx* c = ctx_of_basis(basis);
  hipSetDevice(c->device);
  const int ngw = b->g.ngw;
  if (ld < ngw) return dfail(c, QBH_ERR_ARG, "ld < ngw");
  const bool real = b->g.real;
  // the matrix-core products read element pairs; up to 65535 bands (grid rows)
  if (real && (reinterpret_cast<uintptr_t>(psi_dev) & 15) == 0 && nst <= 65535) {
    int bad = 0;
    if (int r = gram_real(c, nst, 2L * ngw, psi_dev, 2 * ld, &bad)) return r;
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return dfail(c, QBH_ERR_DEVICE, hipGetErrorString(e));
    if (bad) return dfail(c, QBH_ERR_ARG, "gram: overlap matrix not positive definite");
    return QBH_OK;
  }
  void* hb;
  if (int r = blas_handle(c, &hb)) return r;
  rocblas_handle bh = static_cast<rocblas_handle>(hb);
  double* S = nullptr;
  rocblas_int* info = nullptr;
  const size_t ssz = (size_t)nst * nst * (real ? 1 : 2);
  if (hipMalloc(&S, ssz * sizeof(double)) != hipSuccess ||
      hipMalloc(&info, sizeof(rocblas_int)) != hipSuccess) {
    if (S) hipFree(S);
    return dfail(c, QBH_ERR_ALLOC, "gram scratch allocation failed");
  }
  Scratch scr;
  // S = 2 C^T C - c0 c0^T (SlaterDet.cc:1065-1066) or C^H C
  int r = band_product(c, bh, real, nst, nst, real ? 2L * ngw : (long)ngw, psi_dev,
                       real ? 2 * ld : ld, psi_dev, real ? 2 * ld : ld, real ? 2.0 : 1.0, S,
                       scr.p, scr.bytes);
  rocblas_status st = rocblas_status_success;
  if (!r) {
    if (real) {
      const double one = 1.0;
      st = rocsolver_dpotrf(bh, rocblas_fill_lower, nst, S, nst, info);
      if (st == rocblas_status_success)
        st = rocblas_dtrsm(bh, rocblas_side_right, rocblas_fill_lower, rocblas_operation_transpose,
                           rocblas_diagonal_non_unit, 2 * ngw, nst, &one, S, nst, psi_dev, 2 * ld);
    } else {
      const rocblas_double_complex zone(1.0, 0.0);
      auto* C = reinterpret_cast<rocblas_double_complex*>(psi_dev);
      auto* Sz = reinterpret_cast<rocblas_double_complex*>(S);
      st = rocsolver_zpotrf(bh, rocblas_fill_lower, nst, Sz, nst, info);
      if (st == rocblas_status_success)
        st = rocblas_ztrsm(bh, rocblas_side_right, rocblas_fill_lower,
                           rocblas_operation_conjugate_transpose, rocblas_diagonal_non_unit, ngw,
                           nst, &zone, Sz, nst, C, ld);
    }
  }
  rocblas_int hinfo = 0;
  hipMemcpyAsync(&hinfo, info, sizeof(rocblas_int), hipMemcpyDeviceToHost, c->stream);
  hipStreamSynchronize(c->stream);
  hipFree(S);
  hipFree(info);
  if (r) return r;
  if (st != rocblas_status_success)
    return dfail(c, QBH_ERR_BLAS, std::string("gram: ") + rocblas_status_to_string(st));
  if (hinfo != 0) return dfail(c, QBH_ERR_ARG, "gram: overlap matrix not positive definite");
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return dfail(c, QBH_ERR_DEVICE, hipGetErrorString(e));
  return QBH_OK;
}

extern "C" int qbh_subspace_diag(qbh_basis basis, double* psi_dev, long ld,
                                 const double* hpsi_dev, long ldh, int nst, double* eig,
                                 int eigvec) {
  if (!basis || !psi_dev || !hpsi_dev || nst <= 0 || !eig) return QBH_ERR_ARG;
  Basis* b = basis_of(basis);
  Ctx* c = ctx_of_basis(basis);
  hipSetDevice(c->device);
  const int ngw = b->g.ngw;
  if (ld < ngw || ldh < ngw) return dfail(c, QBH_ERR_ARG, "leading dimension < ngw");
  void* hb;
  if (int r = blas_handle(c, &hb)) return r;
  rocblas_handle bh = static_cast<rocblas_handle>(hb);
  const bool real = b->g.real;
  const size_t e = real ? 1 : 2;
  double *H = nullptr, *W = nullptr, *E = nullptr, *C0 = nullptr;
  rocblas_int* info = nullptr;
  const size_t csz = sizeof(double) * 2 * (size_t)ngw * nst;
  bool ok = hipMalloc(&H, sizeof(double) * e * nst * nst) == hipSuccess &&
            hipMalloc(&W, sizeof(double) * nst) == hipSuccess &&
            hipMalloc(&E, sizeof(double) * nst) == hipSuccess &&
            hipMalloc(&info, sizeof(rocblas_int)) == hipSuccess &&
            (!eigvec || hipMalloc(&C0, csz) == hipSuccess);
  auto release = [&]() {
    for (void* p : {(void*)H, (void*)W, (void*)E, (void*)C0, (void*)info})
      if (p) hipFree(p);
  };
  if (!ok) {
    release();
    return dfail(c, QBH_ERR_ALLOC, "subspace diag scratch allocation failed");
  }
  Scratch scr;
  // H = 2 C^T (HC) - c0 (hc)0^T (Wavefunction.cc:1546-1548) or C^H (HC) (:1634)
  int r = band_product(c, bh, real, nst, nst, real ? 2L * ngw : (long)ngw, psi_dev,
                       real ? 2 * ld : ld, hpsi_dev, real ? 2 * ldh : ldh, real ? 2.0 : 1.0, H,
                       scr.p, scr.bytes);
  rocblas_status st = rocblas_status_success;
  const rocblas_evect ev = eigvec ? rocblas_evect_original : rocblas_evect_none;
  if (!r) {
    if (real)
      st = rocsolver_dsyevd(bh, ev, rocblas_fill_lower, nst, H, nst, W, E, info);
    else
      st = rocsolver_zheevd(bh, ev, rocblas_fill_lower, nst,
                            reinterpret_cast<rocblas_double_complex*>(H), nst, W, E, info);
  }
  if (!r && st == rocblas_status_success && eigvec) {
    // C <- C Z (Wavefunction.cc:1605-1607)
    hipMemcpy2DAsync(C0, 2 * sizeof(double) * ngw, psi_dev, 2 * sizeof(double) * ld,
                     2 * sizeof(double) * ngw, nst, hipMemcpyDeviceToDevice, c->stream);
    if (real) {
      const double one = 1.0, zero = 0.0;
      st = rocblas_dgemm(bh, rocblas_operation_none, rocblas_operation_none, 2 * ngw, nst, nst,
                         &one, C0, 2 * ngw, H, nst, &zero, psi_dev, 2 * ld);
    } else {
      const rocblas_double_complex one(1.0, 0.0), zero(0.0, 0.0);
      st = rocblas_zgemm(bh, rocblas_operation_none, rocblas_operation_none, ngw, nst, nst, &one,
                         reinterpret_cast<rocblas_double_complex*>(C0), ngw,
                         reinterpret_cast<rocblas_double_complex*>(H), nst, &zero,
                         reinterpret_cast<rocblas_double_complex*>(psi_dev), ld);
    }
  }
  rocblas_int hinfo = 0;
  hipMemcpyAsync(&hinfo, info, sizeof(rocblas_int), hipMemcpyDeviceToHost, c->stream);
  hipMemcpyAsync(eig, W, sizeof(double) * nst, hipMemcpyDeviceToHost, c->stream);
  hipStreamSynchronize(c->stream);
  release();
  if (r) return r;
  if (st != rocblas_status_success)
    return dfail(c, QBH_ERR_BLAS, std::string("subspace diag: ") + rocblas_status_to_string(st));
  if (hinfo != 0) return dfail(c, QBH_ERR_ARG, "subspace diag: eigensolver did not converge");
  hipError_t err = hipGetLastError();
  if (err != hipSuccess) return dfail(c, QBH_ERR_DEVICE, hipGetErrorString(err));
  return QBH_OK;
}
