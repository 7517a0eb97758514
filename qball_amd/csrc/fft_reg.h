// Register-resident small DFTs (lengths 2..16) and a two-factor row transform.
//
// A row of length n = N1*N2 is transformed in two register stages with one LDS
// exchange between them (Cooley-Tukey "four-step" with the transposition folded into
// the LDS addressing):
//   stage A : for each j2 < N2, DFT_N1 over x[j2 + N2*j1], twiddle W_n^{j2*k1}
//   stage B : for each k1 < N1, DFT_N2 over the N2 contiguous values -> X[k1 + N1*k2]
// Small DFTs of composite length use the prime-factor (Good-Thomas) index maps when the
// factors are coprime (6, 10, 12, 14, 15) and Cooley-Tukey with constant twiddles
// otherwise (9 = 3*3, 16 = 4*4).
#pragma once
#include "fft_device.h"
#include "qbh_fft_edges.h"

namespace qbh {

// cos/sin(2 pi m / L) tables for the Cooley-Tukey small lengths
template <int L> struct WTab;
template <> struct WTab<9> {
  static constexpr double c[9] = {1.0, 0.766044443118978, 0.17364817766693036, -0.5,
                                  -0.9396926207859084, -0.9396926207859084, -0.5,
                                  0.17364817766693036, 0.766044443118978};
  static constexpr double s[9] = {0.0, 0.6427876096865394, 0.984807753012208,
                                  0.8660254037844386, 0.3420201433256687, -0.3420201433256687,
                                  -0.8660254037844386, -0.984807753012208, -0.6427876096865394};
};
template <> struct WTab<16> {
  static constexpr double c[16] = {1.0, 0.9238795325112867, 0.7071067811865476, 0.3826834323650898,
                                   0.0, -0.3826834323650898, -0.7071067811865476,
                                   -0.9238795325112867, -1.0, -0.9238795325112867,
                                   -0.7071067811865476, -0.3826834323650898, 0.0,
                                   0.3826834323650898, 0.7071067811865476, 0.9238795325112867};
  static constexpr double s[16] = {0.0, 0.3826834323650898, 0.7071067811865476, 0.9238795325112867,
                                   1.0, 0.9238795325112867, 0.7071067811865476, 0.3826834323650898,
                                   0.0, -0.3826834323650898, -0.7071067811865476,
                                   -0.9238795325112867, -1.0, -0.9238795325112867,
                                   -0.7071067811865476, -0.3826834323650898};
};

constexpr int inv_mod(int a, int m) {
  for (int x = 1; x < m; ++x)
    if ((a * x) % m == 1) return x;
  return 1;
}

template <int L, int DIR, typename T> __device__ __forceinline__ void sdft(cplx<T>* a);

// Good-Thomas: L = A*B, gcd(A,B) = 1.  Input n = (a*B + b*A) mod L, output
// k = (ka*B*inv(B,A) + kb*A*inv(A,B)) mod L.
template <int A, int B, int DIR, typename T>
__device__ __forceinline__ void pfa(cplx<T>* x) {
  constexpr int L = A * B;
  cplx<T> m[B][A];
#pragma unroll
  for (int b = 0; b < B; ++b) {
#pragma unroll
    for (int a = 0; a < A; ++a) m[b][a] = x[(a * B + b * A) % L];
    sdft<A, DIR>(m[b]);
  }
  constexpr int cb = B * inv_mod(B % A, A);
  constexpr int ca = A * inv_mod(A % B, B);
#pragma unroll
  for (int ka = 0; ka < A; ++ka) {
    cplx<T> col[B];
#pragma unroll
    for (int b = 0; b < B; ++b) col[b] = m[b][ka];
    sdft<B, DIR>(col);
#pragma unroll
    for (int kb = 0; kb < B; ++kb) x[(ka * cb + kb * ca) % L] = col[kb];
  }
}

// Cooley-Tukey L = A*B with constant twiddles: X[k1 + A*k2] =
//   sum_j2 W_B^{j2 k2} W_L^{j2 k1} sum_j1 x[j2 + B*j1] W_A^{j1 k1}
template <int A, int B, int DIR, typename T>
__device__ __forceinline__ void ct(cplx<T>* x) {
  constexpr int L = A * B;
  cplx<T> m[B][A];
#pragma unroll
  for (int j2 = 0; j2 < B; ++j2) {
#pragma unroll
    for (int j1 = 0; j1 < A; ++j1) m[j2][j1] = x[j2 + B * j1];
    sdft<A, DIR>(m[j2]);
#pragma unroll
    for (int k1 = 1; k1 < A; ++k1) {
      const int e = (j2 * k1) % L;
      if (e != 0) {
        const cplx<T> w = {T(WTab<L>::c[e]), T(DIR * WTab<L>::s[e])};
        m[j2][k1] = cmul(m[j2][k1], w);
      }
    }
  }
#pragma unroll
  for (int k1 = 0; k1 < A; ++k1) {
    cplx<T> col[B];
#pragma unroll
    for (int j2 = 0; j2 < B; ++j2) col[j2] = m[j2][k1];
    sdft<B, DIR>(col);
#pragma unroll
    for (int k2 = 0; k2 < B; ++k2) x[k1 + A * k2] = col[k2];
  }
}

template <int L, int DIR, typename T>
__device__ __forceinline__ void sdft(cplx<T>* a) {
  if constexpr (L == 1) {
  } else if constexpr (L == 2 || L == 3 || L == 4 || L == 5 || L == 7 || L == 8 || L == 11) {
    dft<L, DIR>(a);
  } else if constexpr (L == 6) {
    pfa<2, 3, DIR>(a);
  } else if constexpr (L == 10) {
    pfa<2, 5, DIR>(a);
  } else if constexpr (L == 12) {
    pfa<4, 3, DIR>(a);
  } else if constexpr (L == 14) {
    pfa<2, 7, DIR>(a);
  } else if constexpr (L == 15) {
    pfa<3, 5, DIR>(a);
  } else if constexpr (L == 9) {
    ct<3, 3, DIR>(a);
  } else if constexpr (L == 16) {
    ct<4, 4, DIR>(a);
  } else {
    static_assert(L == 2, "unsupported small DFT length");
  }
}

// FP32 transforms in the radix order of the Stockham passes (n = N1*N2 an F length): the first
// stage is a chain of the plan's leading radices with their twiddles W_N1^e = W_n^{e N2} read
// from the table tw of length n, the second the last radix, and each twiddle product stands
// right before the radix it feeds, as in those passes, and rounds as theirs do (cmul_fused).
template <typename T, int N1, int N2> constexpr bool stockham_order() {
  return sizeof(T) == 4 && stockham_length(N1 * N2);
}

// a * w (DIR < 0: a * conj w) with the fused operations that the compiler makes of the
// Stockham passes' cmul; left to itself it fuses some products of the unrolled chains the
// other way round.
template <int DIR>
__device__ __forceinline__ cplx<float> cmul_fused(cplx<float> a, cplx<float> w) {
  if (DIR < 0) w.y = -w.y;
  return {fmaf(a.x, w.x, -(a.y * w.y)), fmaf(a.y, w.x, a.x * w.y)};
}

// length A*B as radix A then B (Cooley-Tukey, see ct), twiddles tw[e * stride]
template <int A, int B, int DIR, typename T>
__device__ __forceinline__ void ct_tab(cplx<T>* x, const cplx<T>* tw, int stride) {
  cplx<T> m[B][A];
#pragma unroll
  for (int j2 = 0; j2 < B; ++j2) {
#pragma unroll
    for (int j1 = 0; j1 < A; ++j1) m[j2][j1] = x[j2 + B * j1];
    dft<A, DIR>(m[j2]);
  }
#pragma unroll
  for (int k1 = 0; k1 < A; ++k1) {
    cplx<T> col[B];
#pragma unroll
    for (int j2 = 0; j2 < B; ++j2) {
      col[j2] = m[j2][k1];
      if (j2 > 0) {
        col[j2] = cmul_fused<DIR>(col[j2], tw[j2 * k1 * stride]);
      }
    }
    dft<B, DIR>(col);
#pragma unroll
    for (int k2 = 0; k2 < B; ++k2) x[k1 + A * k2] = col[k2];
  }
}

// first-stage DFT of length N1 of a transform of length N1*N2 (twiddle table tw)
template <int N1, int N2, int DIR, typename T>
__device__ __forceinline__ void stage_a(cplx<T>* a, const cplx<T>* tw) {
  if constexpr (!stockham_order<T, N1, N2>()) {
    sdft<N1, DIR>(a);
  } else if constexpr (N1 == 4 || N1 == 8) {
    dft<N1, DIR>(a);
  } else if constexpr (N1 == 12 || N1 == 16) {
    ct_tab<4, N1 / 4, DIR>(a, tw, N2);
  } else {
    static_assert(N1 == 6 || N1 == 10 || N1 == 14, "no Stockham chain");
    ct_tab<2, N1 / 2, DIR>(a, tw, N2);
  }
}

// second-stage DFT of length N2 at k1 of the first stage (F forms: with the stage twiddles)
template <int N1, int N2, int DIR, typename T>
__device__ __forceinline__ void stage_b(cplx<T>* b, const cplx<T>* tw, int k1) {
  if constexpr (stockham_order<T, N1, N2>()) {
#pragma unroll
    for (int j2 = 1; j2 < N2; ++j2) b[j2] = cmul_fused<DIR>(b[j2], tw[k1 * j2]);
  }
  sdft<N2, DIR>(b);
}

// a[k] *= W_n^{DIR e k}, k < K, n the length of the table tw (e (K - 1) < n).  FP64 and TAB read
// every power from the table: local Hψ is 1.2 to 1.9 times closer to 64-bit reference transforms
// than with the repeated products of w = tw[e] that FP32 forms otherwise (140^3: 5.3e-16 against
// 8.2e-16 of the result), in the same time up to edge 180 (140^3 x pass, 300 slots, 3.75 against
// 3.73 ms); from 192 on local Hψ takes 3 to 12 % longer (256^3, 32 bands 5.24 against 4.78 ms).
template <int K, int DIR, bool TAB = false, typename T>
__device__ __forceinline__ void twiddle_row(cplx<T>* a, const cplx<T>* tw, int e) {
  if (e == 0) return;
  cplx<T> w = tw[e];
  if (DIR < 0) w.y = -w.y;
  cplx<T> p = w;
#pragma unroll
  for (int k = 1; k < K; ++k) {
    a[k] = cmul(a[k], p);
    if (k + 1 < K) {
      if constexpr (sizeof(T) == 8 || TAB) {
        p = tw[e * (k + 1)];
        if (DIR < 0) p.y = -p.y;
      } else {
        p = cmul(p, w);
      }
    }
  }
}

// Padded LDS row layout for the two-factor transform: element x of a row lives at
// x + x / N2 when N2 is even, so the stage-B lanes (stride N2 + 1 elements, odd) hit
// distinct LDS banks; the row occupies N1 * (N2 + 1) elements.  N1 = 0 (no register
// factorisation) means an unpadded row.
// Off by default (QBH_LDS_PAD=0): measured on MI355X the padded rows raise the LDS
// footprint of the y/z passes from 38 to 42 KB per workgroup (4 -> 3 workgroups per CU)
// and cost more than the 2-way stage-B conflicts they remove.
#ifndef QBH_LDS_PAD
#define QBH_LDS_PAD 0
#endif
template <int N1, int N2, int ON = QBH_LDS_PAD> struct Pad {
  static constexpr int P = (ON && N1 > 0 && N2 % 2 == 0) ? 1 : 0;
  static __host__ __device__ constexpr int idx(int x) { return P ? x + x / N2 : x; }
  static __host__ __device__ constexpr int row(int n) { return P ? n + n / N2 : n; }
};

// Wavefront-local transform of `nrows` (<= RPW) LDS rows of length n = N1*N2 at
// buf + r*ld (padded layout, Pad<N1,N2,PAD>), natural order in and out, direction DIR:
//   stage A: task (r, j2): DFT_N1 over x[j2 + N2*j1], twiddle W_n^{DIR j2 k1}, in place
//   stage B: task (r, k1): DFT_N2 over the contiguous block N2*k1 + j2 -> X[k1 + N1*k2],
//            held in registers until every lane has read its block, then stored at the
//            natural positions.
// TAB: FP32 stage twiddles from the table too (twiddle_row).
template <int N1, int N2, int RPW, int DIR, int PAD = QBH_LDS_PAD, bool TAB = false, typename T>
__device__ __forceinline__ void rows_fft(cplx<T>* buf, int nrows, int ld, const cplx<T>* tw,
                                         int lane) {
  constexpr int TA = RPW * N2, TB = RPW * N1;
  constexpr int IA = (TA + 63) / 64, IB = (TB + 63) / 64;
  constexpr int S = N2 + Pad<N1, N2, PAD>::P;  // padded stride of the N2-blocks
#pragma unroll
  for (int ia = 0; ia < IA; ++ia) {
    const int t = lane + 64 * ia;
    const int r = t / N2, j2 = t % N2;
    if (t < TA && r < nrows) {
      cplx<T>* row = buf + r * ld + j2;
      cplx<T> a[N1];
#pragma unroll
      for (int j1 = 0; j1 < N1; ++j1) a[j1] = row[S * j1];
      stage_a<N1, N2, DIR>(a, tw);
      if constexpr (!stockham_order<T, N1, N2>()) twiddle_row<N1, DIR, TAB>(a, tw, j2);
#pragma unroll
      for (int k1 = 0; k1 < N1; ++k1) row[S * k1] = a[k1];
    }
  }
  wave_sync();
  cplx<T> b[IB][N2];
#pragma unroll
  for (int ib = 0; ib < IB; ++ib) {
    const int t = lane + 64 * ib;
    const int r = t / N1, k1 = t % N1;
    if (t < TB && r < nrows) {
      const cplx<T>* blk = buf + r * ld + S * k1;
#pragma unroll
      for (int j2 = 0; j2 < N2; ++j2) b[ib][j2] = blk[j2];
      stage_b<N1, N2, DIR>(b[ib], tw, k1);
    }
  }
  wave_sync();
#pragma unroll
  for (int ib = 0; ib < IB; ++ib) {
    const int t = lane + 64 * ib;
    const int r = t / N1, k1 = t % N1;
    if (t < TB && r < nrows) {
      cplx<T>* row = buf + r * ld;
#pragma unroll
      for (int k2 = 0; k2 < N2; ++k2) row[Pad<N1, N2, PAD>::idx(k1 + N1 * k2)] = b[ib][k2];
    }
  }
  wave_sync();
}

}  // namespace qbh
