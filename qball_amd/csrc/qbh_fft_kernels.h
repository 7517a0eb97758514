// G-sphere <-> grid transform pipeline on gfx950.
//
// Behaviour follows qball's FourierTransform (src/qball/FourierTransform.cc): backward
// = unnormalised exp(+iG.r) sum of the sphere coefficients (Γ: c(G) at +G and conj(c(G))
// at -G, the -G value winning at G=0, :1624-1720); forward = exp(-iG.r)/N (:1338-1342)
// followed by the Γ pair unpacking c1 = (z+ + conj z-)/2, c2 = (z+ - conj z-)/(2i)
// (:1723-1752).  The decomposition is this library's own: a z pass over the nonzero
// columns only, a y pass over the x-lines that hold sphere points, and an x pass that
// owns whole real-space rows, so v(r)*psi(r) and |psi(r)|^2 are applied while a row is
// in LDS and the real-space grid never goes to HBM.
//
// Work split: every workgroup has 4 wavefronts; each wavefront owns LPW lines of LDS and
// transforms them on its own (fft_lines_w: no workgroup barrier inside a transform).
// Global reads and writes are arranged so that a wavefront touches contiguous segments
// of >= 64 bytes.
//
// This header holds the kernels and the launch functions of one edge length; every length
// with a two-factor register transform (QBH_EDGES) is compiled in one of the units made from
// qbh_fft_edges.hip, the Stockham forms of the other lengths in qbh_fft.hip, which also holds
// the dispatch.
#pragma once
#include <hip/hip_runtime.h>

#include <algorithm>
#include <string>

#include "fft_reg.h"
#include "qbh_internal.h"

namespace qbh {

constexpr int NTHR = 256;  // threads per workgroup, every pipeline kernel
constexpr int NWAVE = 4;
constexpr int ZLPW = 4;    // z-pass lines per wavefront (16 per group)

// per precision: lines per wavefront in the y and x passes, y-pass plane block
template <typename T> struct Cfg;
// launch tuning (compile-time knobs)
// x pass: slots whose sphere lines are loaded ahead (register buffers of GPW elements
// each).  Measured on MI355X at Si512: two slots ahead slowed the FP32 x pass from 4.26
// to 4.60 ms per Hψ at three waves per SIMD (register spills) and to 5.57 ms at two; FP64
// has no registers to spare.
#ifndef QBH_XPF64
#define QBH_XPF64 1
#endif
#ifndef QBH_XPF32
#define QBH_XPF32 1
#endif
// x pass: minimum waves per SIMD the register allocation must allow (the counts the
// kernels reach without spilling: FP32 three, FP64 two)
#ifndef QBH_XWPE64
#define QBH_XWPE64 2
#endif
#ifndef QBH_XWPE32
#define QBH_XWPE32 3
#endif
// x pass: stage-B forward twiddles held in registers across slots (1) or formed per slot
#ifndef QBH_XTWB
#define QBH_XTWB 1
#endif
// x pass: padded LDS rows (element x at x + x/N2).  The x pass holds two workgroups per CU
// (VGPR-bound), so the larger rows cost it no occupancy, unlike the y/z passes.
#ifndef QBH_XLDS_PAD
#define QBH_XLDS_PAD 1
#endif
// y pass: ZB z-planes x LB x-lines per workgroup, LPW lines per wavefront (ZB*LB = 4*LPW).
// Measured on MI355X at Si512 (140^3): 16 x 1 beats 8 x 2, 4 x 4, 32 x 1 and the 8-line
// shapes in both precisions (FP64 forward y pass 4.58 -> 4.05 ms, FP32 y passes 5.78 ->
// 3.63 ms per Hψ): one x-line per workgroup and 256-byte (FP64) column segments.
#ifndef QBH_YZB64
#define QBH_YZB64 16
#endif
#ifndef QBH_YLB64
#define QBH_YLB64 1
#endif
#ifndef QBH_YZB32
#define QBH_YZB32 16
#endif
#ifndef QBH_YLB32
#define QBH_YLB32 1
#endif
template <> struct Cfg<double> {
  static constexpr int XPF = QBH_XPF64;  // x pass: slots of sphere lines in flight
  static constexpr int XWPE = QBH_XWPE64;  // x pass: minimum waves per SIMD asked of the compiler
  static constexpr int ZB = QBH_YZB64;  // y pass: z-planes per workgroup (column segments)
  static constexpr int LB = QBH_YLB64;  // y pass: x-lines per workgroup
  static constexpr int LPW = ZB * LB / 4;
};
template <> struct Cfg<float> {
  static constexpr int XPF = QBH_XPF32;
  static constexpr int XWPE = QBH_XWPE32;
  static constexpr int ZB = QBH_YZB32;
  static constexpr int LB = QBH_YLB32;
  static constexpr int LPW = ZB * LB / 4;
};

// x pass: rows per wavefront for edge n = N1*N2.  A row gives the wavefront N2 stage-A and N1
// stage-B tasks, one per lane, so it takes as many rows as keep both within its 64 lanes, and
// of those the fewest that cover n rows with as many workgroups (whole last workgroups on
// cubic grids): 4 rows at 140 = 14*10, 5 at 120 = 12*10, 6 at 72 = 9*8, 8 at 64 = 8*8.  Where
// that saves less than an eighth of the workgroups (144 = 12*12: 8 against 9) it stays at 4,
// whose 256-byte segments suit the memory better (500 Al atoms, whole FP64 Hψ: 5 rows 1 % slower).  The
// pass is bound by vector-instruction issue, so idle lanes cost their full share.  Against 4
// rows at every edge (x pass of one local Hψ, MI355X): 64^3 128 bands 111 -> 87 us (FP32 53 ->
// 40), 72^3 128 bands 149 -> 103 (FP32 79 -> 67), 60^3 64 bands 56 -> 47, 144^3 unchanged.
constexpr int x_rows(int n1, int n2) {
  const int most = 64 / (n1 > n2 ? n1 : n2);
  const int nb = (n1 * n2 + 4 * most - 1) / (4 * most), nb4 = (n1 * n2 + 15) / 16;
  return 8 * nb > 7 * nb4 ? 4 : (n1 * n2 + 4 * nb - 1) / (4 * nb);
}

// y pass: lines (z planes) per wavefront for edge n = N1*N2.  Filling the lanes as in the x
// pass helps the short edges, whose passes are not yet bound by HBM, but only where the
// workgroups' z blocks then cover n with fewer planes past its end (FP32: not more) than
// blocks of 16, or exactly.  Backward / forward y pass of one local FP64 Hψ against 4 lines,
// MI355X: 72^3 128 bands 68 / 66 -> 59 / 56 us, 64^3 128 bands 45 / 41 -> 41 / 36, 120^3 300 bands 543 /
// 419 -> 484 / 391; without the rule 96^3 (5 lines: 100 planes) 342 -> 363 backward.
template <typename T> constexpr int y_lines(int n1, int n2) {
  const int n = n1 * n2, r = x_rows(n1, n2);
  const int p4 = (n + 15) / 16 * 16, pr = (n + 4 * r - 1) / (4 * r) * 4 * r;
  return pr < p4 || n % (4 * r) == 0 || (sizeof(T) == 4 && pr == p4) ? r : 4;
}
template <typename T, int N1, int N2> struct YCfg {
  static constexpr int LPW = N1 > 0 ? y_lines<T>(N1 > 0 ? N1 : 1, N2 > 0 ? N2 : 1) : Cfg<T>::LPW;
  static constexpr int LB = Cfg<T>::LB;
  static constexpr int ZB = NWAVE * LPW / LB;
};

// x pass: line elements per thread of the short variant, for spheres up to half the edge, and of
// the middle one, for up to eight lines more, of the potential multiply and the density
// (registers per element; with the full count, which the middle one avoids, 180^3 with 97 lines,
// 64 bands: Hψ 2.80 ms against 2.55; with the middle count in place of the short one 160^3, 79
// lines: density 0.94 against 0.88 ms)
constexpr int x_short(int n, int yb) { return (yb * (n / 2) + NTHR - 1) / NTHR; }
constexpr int x_middle(int n, int yb) { return (yb * (n / 2 + 8) + NTHR - 1) / NTHR; }

template <typename T>
__device__ __forceinline__ const cplx<T>* twtab(const GridDev& g, int axis);
template <>
__device__ __forceinline__ const cplx<double>* twtab<double>(const GridDev& g, int axis) {
  return g.tw64[axis];
}
template <>
__device__ __forceinline__ const cplx<float>* twtab<float>(const GridDev& g, int axis) {
  return g.tw32[axis];
}

__device__ __forceinline__ int wrap(int l, int n) { return l < 0 ? l + n : l; }

// elements per lane of a wavefront owning `lpw` lines of length <= NMAX
template <int LPW, int NMAX> struct Epl { static constexpr int v = (LPW * NMAX + 63) / 64; };

// Wavefront-local transform of nl lines of length ld: the two-factor register transform
// when the length has an instantiated factorisation n = N1*N2, else the LDS Stockham passes.
template <int DIR, int EPL, int N1, int N2, int RPW, typename T>
__device__ __forceinline__ void line_fft(cplx<T>* buf, int nl, int ld, const AxisPlan& ax,
                                         const cplx<T>* tw, int lane) {
  if constexpr (N1 > 0)
    rows_fft<N1, N2, RPW, DIR>(buf, nl, ld, tw, lane);
  else
    fft_lines_w<DIR, EPL>(buf, nl, ld, ax, tw, lane);
}

// ------------------------------------------------------------------------------------
// z pass, backward: gather sphere coefficients of one slot into its columns, transform
// along z (exp(+i)), store T1[slot][col][z].  Line e of a group belongs to wavefront e/4.
template <typename T, int MODE, int NMAX, int N1, int N2>
__global__ void __launch_bounds__(NTHR)
k_zpass_bwd(GridDev g, const double* __restrict__ psi, long ld, int nst, int band0,
            cplx<T>* __restrict__ t1) {
  constexpr int EPL = Epl<ZLPW, NMAX>::v;
  extern __shared__ __align__(16) unsigned char smem_raw[];
  const int np2 = g.np2;
  cplx<T>* tw = reinterpret_cast<cplx<T>*>(smem_raw);
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int grp = blockIdx.x;
  const int slot = blockIdx.y;
  // this wavefront's lines and the rod of the line its 16-lane group gathers, read before
  // the workgroup barrier so the table loads overlap the twiddle load
  const int e0 = g.grp_start[grp] + wave * ZLPW;
  const int nl = min(ZLPW, g.grp_start[grp + 1] - e0);
  const int le = lane >> 4;
  const int sub = lane & 15;
  int kind = 4, first = 0, lmin = 0, size = 0;
  if (le < nl) {
    kind = g.ent_kind[e0 + le];
    if (kind != 4) {
      const int rod = g.ent_rod[e0 + le];
      first = g.rod_first[rod];
      lmin = g.rod_lmin[rod];
      size = g.rod_size[rod];
    }
  }
  const cplx<T>* twg = twtab<T>(g, 2);
  for (int i = threadIdx.x; i < np2; i += NTHR) tw[i] = twg[i];
  __syncthreads();
  if (nl <= 0) return;
  using PD = Pad<N1, N2>;
  const int LD = PD::row(np2);
  cplx<T>* buf = tw + np2 + wave * ZLPW * LD;
  for (int i = lane; i < nl * LD; i += 64) buf[i] = {T(0), T(0)};
  wave_sync();

  int n1, n2;
  if (MODE == SLOT_PAIR) {
    n1 = band0 + 2 * slot;
    n2 = n1 + 1;
  } else {
    n1 = band0 + slot;
    n2 = nst;
  }
  const bool has2 = (MODE == SLOT_PAIR) && (n2 < nst);
  const double* p1 = psi + 2 * (long)n1 * ld;
  const double* p2 = psi + 2 * (long)(has2 ? n2 : n1) * ld;

  // 16 lanes per line; KZ coefficients per lane loaded together before they are stored
  constexpr int KZ = 4;
  if (le < nl && kind != 4) {
    cplx<T>* line = buf + le * LD;
    for (int i0 = sub; i0 < size; i0 += 16 * KZ) {
      double a[KZ], b[KZ], c[KZ], d[KZ];
      // branch-free: every lane loads an element of its rod (past the end: the last one,
      // never stored), so all KZ loads are in flight together
#pragma unroll
      for (int k = 0; k < KZ; ++k) {
        const long e = 2 * (long)(first + min(i0 + 16 * k, size - 1));
        a[k] = p1[e];
        b[k] = p1[e + 1];
        c[k] = d[k] = 0.0;
        if (MODE == SLOT_PAIR) {  // p2 is p1 for a lone last band; its values are dropped
          c[k] = p2[e];
          d[k] = p2[e + 1];
        }
      }
      if (!has2)
#pragma unroll
        for (int k = 0; k < KZ; ++k) c[k] = d[k] = 0.0;
#pragma unroll
      for (int k = 0; k < KZ; ++k) {
        const int i = i0 + 16 * k;
        if (i >= size) continue;
        const int l = lmin + i;
        double pr, pi, mr, mi;  // +G and -G values
        if (MODE == SLOT_PAIR) {
          pr = a[k] - d[k]; pi = b[k] + c[k]; mr = a[k] + d[k]; mi = c[k] - b[k];
        } else {
          pr = a[k]; pi = b[k]; mr = a[k]; mi = -b[k];
        }
        if (kind == 0) {
          if (i > 0) line[PD::idx(wrap(l, np2))] = {T(pr), T(pi)};
          line[PD::idx(wrap(-l, np2))] = {T(mr), T(mi)};
        } else if (kind == 1 || kind == 3) {
          line[PD::idx(wrap(l, np2))] = {T(pr), T(pi)};
        } else {
          line[PD::idx(wrap(-l, np2))] = {T(mr), T(mi)};
        }
      }
    }
  }
  wave_sync();
  line_fft<+1, EPL, N1, N2, ZLPW>(buf, nl, LD, g.ax[2], tw, lane);
  for (int ll = 0; ll < nl; ++ll) {
    const int col = g.ent_col[e0 + ll];
    if (col < 0) continue;
    cplx<T>* dst = t1 + ((long)slot * g.ncol + col) * np2;
    for (int z = lane; z < np2; z += 64) dst[z] = buf[ll * LD + PD::idx(z)];
  }
}

// ------------------------------------------------------------------------------------
// y pass, backward: T1 columns of ZB planes x LB x-lines -> y transform -> T2 lines.
// The workgroup gathers its columns cooperatively (ZB-element segments), then each
// wavefront transforms and stores its own LPW lines.
template <typename T, int NMAX, int N1, int N2>
__global__ void __launch_bounds__(NTHR)
k_ypass_bwd(GridDev g, const cplx<T>* __restrict__ t1, cplx<T>* __restrict__ t2) {
  constexpr int ZB = YCfg<T, N1, N2>::ZB, LB = YCfg<T, N1, N2>::LB, LPW = YCfg<T, N1, N2>::LPW;
  constexpr int EPL = Epl<LPW, NMAX>::v;
  extern __shared__ __align__(16) unsigned char smem_raw[];
  const int np1 = g.np1, np2 = g.np2, nlx = g.nlx;
  cplx<T>* tw = reinterpret_cast<cplx<T>*>(smem_raw);
  cplx<T>* buf = tw + np1;
  using PD = Pad<N1, N2>;
  const int LD = PD::row(np1);
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int nzb = (np2 + ZB - 1) / ZB;
  const int zb = blockIdx.x % nzb;
  const int lb = blockIdx.x / nzb;
  const int slot = blockIdx.y;
  const int z0 = zb * ZB, lx0 = lb * LB;
  const int lx1 = min(lx0 + LB, nlx);
  const cplx<T>* twg = twtab<T>(g, 1);
  for (int i = threadIdx.x; i < np1; i += NTHR) tw[i] = twg[i];
  for (int i = threadIdx.x; i < ZB * LB * LD; i += NTHR) buf[i] = {T(0), T(0)};
  __syncthreads();
  const int c0 = g.line_start[lx0], c1 = g.line_start[lx1];
  const int nwork = (c1 - c0) * ZB;
  if constexpr (sizeof(T) == 4) {
    // FP32: KG elements per thread and round, all loaded (with their column indices) before
    // any is stored; past the end a thread reloads the last element and stores nothing
    // (at Si512 1.64 -> 1.49 ms per Hψ; in FP64 the same form measured 3.33 -> 3.40-3.55 ms)
    constexpr int KG = 4;
    for (int f0 = threadIdx.x; f0 < nwork; f0 += NTHR * KG) {
      cplx<T> v[KG];
      int col[KG], cc[KG];
#pragma unroll
      for (int k = 0; k < KG; ++k) {
        const int f = min(f0 + k * NTHR, nwork - 1);
        const int c = c0 + f / ZB;
        const int z = min(z0 + f % ZB, np2 - 1);
        cc[k] = c;
        col[k] = g.col_y[c];
        v[k] = t1[((long)slot * g.ncol + c) * np2 + z];
      }
#pragma unroll
      for (int k = 0; k < KG; ++k) {
        const int f = f0 + k * NTHR;
        const int dz = f % ZB;
        if (f < nwork && z0 + dz < np2) {
          int dl = 0;
          while (lx0 + dl + 1 < lx1 && cc[k] >= g.line_start[lx0 + dl + 1]) ++dl;
          buf[(dz + ZB * dl) * LD + PD::idx(col[k])] = v[k];
        }
      }
    }
  } else {
    for (int f = threadIdx.x; f < nwork; f += NTHR) {
      const int dz = f % ZB;
      const int c = c0 + f / ZB;
      const int z = z0 + dz;
      if (z < np2) {
        int dl = 0;
        while (lx0 + dl + 1 < lx1 && c >= g.line_start[lx0 + dl + 1]) ++dl;
        buf[(dz + ZB * dl) * LD + PD::idx(g.col_y[c])] = t1[((long)slot * g.ncol + c) * np2 + z];
      }
    }
  }
  __syncthreads();
  // line li = dz + ZB*dl; wavefront w owns lines [w*LPW, (w+1)*LPW)
  cplx<T>* wbuf = buf + wave * LPW * LD;
  line_fft<+1, EPL, N1, N2, LPW>(wbuf, LPW, LD, g.ax[1], tw, lane);
  for (int ll = 0; ll < LPW; ++ll) {
    const int li = wave * LPW + ll;
    const int dz = li % ZB, dl = li / ZB;
    const int z = z0 + dz, lx = lx0 + dl;
    if (z >= np2 || lx >= lx1) continue;
    cplx<T>* dst = t2 + (((long)slot * np2 + z) * nlx + lx) * np1;
    for (int y = lane; y < np1; y += 64) dst[y] = wbuf[ll * LD + PD::idx(y)];
  }
}

// y pass, forward: T2 lines -> y transform (exp(-i)) -> sphere columns of T1.
template <typename T, int NMAX, int N1, int N2>
__global__ void __launch_bounds__(NTHR)
k_ypass_fwd(GridDev g, const cplx<T>* __restrict__ t2, cplx<T>* __restrict__ t1) {
  constexpr int ZB = YCfg<T, N1, N2>::ZB, LB = YCfg<T, N1, N2>::LB, LPW = YCfg<T, N1, N2>::LPW;
  constexpr int EPL = Epl<LPW, NMAX>::v;
  extern __shared__ __align__(16) unsigned char smem_raw[];
  const int np1 = g.np1, np2 = g.np2, nlx = g.nlx;
  cplx<T>* tw = reinterpret_cast<cplx<T>*>(smem_raw);
  cplx<T>* buf = tw + np1;
  using PD = Pad<N1, N2>;
  const int LD = PD::row(np1);
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int nzb = (np2 + ZB - 1) / ZB;
  const int zb = blockIdx.x % nzb;
  const int lb = blockIdx.x / nzb;
  const int slot = blockIdx.y;
  const int z0 = zb * ZB, lx0 = lb * LB;
  const int lx1 = min(lx0 + LB, nlx);
  const cplx<T>* twg = twtab<T>(g, 1);
  for (int i = threadIdx.x; i < np1; i += NTHR) tw[i] = twg[i];
  // LDS offset (without the z-plane term) of each column of this workgroup's lines, staged
  // once so the column scatter below waits on no index-table load
  int* cof = reinterpret_cast<int*>(buf + ZB * LB * LD);
  const int c0 = g.line_start[lx0], c1 = g.line_start[lx1];
  for (int i = threadIdx.x; i < c1 - c0; i += NTHR) {
    const int c = c0 + i;
    int dl = 0;
    while (lx0 + dl + 1 < lx1 && c >= g.line_start[lx0 + dl + 1]) ++dl;
    cof[i] = ZB * dl * LD + PD::idx(g.col_y[c]);
  }
  __syncthreads();
  cplx<T>* wbuf = buf + wave * LPW * LD;
  {
    // the wave's LPW lines (KY elements per lane each) are all loaded before any is stored
    // to LDS, so no load waits on the one before it (lines past the grid read a valid
    // line and store zeros)
    // elements per lane: a register transform's length is N1 N2 (which can exceed NMAX),
    // a generic one's at most NMAX
    constexpr int KY = ((N1 > 0 ? N1 * N2 : NMAX) + 63) / 64;
    cplx<T> v[LPW][KY];
    bool in[LPW][KY];
#pragma unroll
    for (int ll = 0; ll < LPW; ++ll) {
      const int li = wave * LPW + ll;
      const int dz = li % ZB, dl = li / ZB;
      const int z = z0 + dz, lx = lx0 + dl;
      const bool ok = z < np2 && lx < lx1;
      const cplx<T>* src = t2 + (((long)slot * np2 + (ok ? z : 0)) * nlx + (ok ? lx : 0)) * np1;
#pragma unroll
      for (int k = 0; k < KY; ++k) {
        const int y = lane + 64 * k;
        in[ll][k] = ok && y < np1;
        v[ll][k] = src[in[ll][k] ? y : 0];
      }
    }
#pragma unroll
    for (int ll = 0; ll < LPW; ++ll)
#pragma unroll
      for (int k = 0; k < KY; ++k) {
        const int y = lane + 64 * k;
        if (y < np1) wbuf[ll * LD + PD::idx(y)] = in[ll][k] ? v[ll][k] : cplx<T>{T(0), T(0)};
      }
  }
  wave_sync();
  line_fft<-1, EPL, N1, N2, LPW>(wbuf, LPW, LD, g.ax[1], tw, lane);
  __syncthreads();
  const int nwork = (c1 - c0) * ZB;
  for (int f = threadIdx.x; f < nwork; f += NTHR) {
    const int dz = f % ZB;
    const int c = c0 + f / ZB;
    const int z = z0 + dz;
    if (z < np2) t1[((long)slot * g.ncol + c) * np2 + z] = buf[dz * LD + cof[c - c0]];
  }
}

// ------------------------------------------------------------------------------------
// x pass.  Wavefront w of a workgroup owns LPW consecutive real-space rows (z fixed,
// y = y0 + w*LPW ...) and loops over the slots [s0, s1) with no workgroup barrier; the
// next slot's sphere lines are loaded into registers while the current slot transforms.
enum XOp { X_VMUL = 0, X_STORE = 1, X_LOAD = 2, X_LOAD_REAL = 3, X_DENSITY = 4 };

template <typename T, int OP, int NMAX>
__global__ void __launch_bounds__(NTHR)
k_xpass(GridDev g, cplx<T>* __restrict__ t2, int nslots, int slots_per_wg,
        const double* __restrict__ v,      // VMUL: potential; LOAD*: input grid
        double* __restrict__ out,          // STORE: complex grid; DENSITY: rho, or one
                                           // partial grid per slot range (gridDim.y > 1)
        const double* __restrict__ dens,   // DENSITY: per slot (fac1, fac2, beta1, beta2)
        double scale, int cplx_density) {
  constexpr int LPW = Cfg<T>::LPW;
  constexpr int YB = LPW * NWAVE;
  constexpr int EPL = Epl<LPW, NMAX>::v;          // row elements per lane
  constexpr int GPL = EPL;  // sphere-line elements per lane (nlx <= np0)
  extern __shared__ __align__(16) unsigned char smem_raw[];
  const int np0 = g.np0, np1 = g.np1, np2 = g.np2, nlx = g.nlx;
  cplx<T>* tw = reinterpret_cast<cplx<T>*>(smem_raw);
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int nyb = (np1 + YB - 1) / YB;
  const int z = blockIdx.x / nyb;
  const int y0 = (blockIdx.x % nyb) * YB + wave * LPW;  // this wavefront's first row
  const int nyl = min(LPW, np1 - y0);                   // rows of this wavefront
  const int s0 = blockIdx.y * slots_per_wg;
  const int s1 = min(nslots, s0 + slots_per_wg);
  const cplx<T>* twg = twtab<T>(g, 0);
  for (int i = threadIdx.x; i < np0; i += NTHR) tw[i] = twg[i];
  __syncthreads();
  if (nyl <= 0) return;
  cplx<T>* buf = tw + np0 + wave * LPW * np0;
  const int nel = nyl * np0;
  const long grow0 = ((long)z * np1 + y0) * np0;  // grid offset of the wavefront's first row
  const long N = (long)np0 * np1 * np2;
  const int ng = nlx * LPW;                       // sphere-line elements of the rows

  T vr[EPL];
  double acc[EPL];
  if (OP == X_VMUL) {
#pragma unroll
    for (int k = 0; k < EPL; ++k) {
      const int e = lane + k * 64;
      vr[k] = e < nel ? T(v[grow0 + e]) : T(0);
    }
  }
  if (OP == X_DENSITY) {
#pragma unroll
    for (int k = 0; k < EPL; ++k) acc[k] = 0.0;
  }

  // sphere-line element q = lane + k*64: row dy = q % LPW, line lx = q / LPW.  Its LDS
  // offset (-1 past the lines) and its T2 offset within a slot do not depend on the slot:
  // computed once, so the slot loop issues no index-table loads.
  const long sstride = (long)np2 * nlx * np1;
  int lofs[GPL], gofs[GPL];
#pragma unroll
  for (int k = 0; k < GPL; ++k) {
    const int q = lane + k * 64;
    const int dy = q % LPW, lx = q / LPW;
    lofs[k] = q < ng ? dy * np0 + g.line_x[lx] : -1;
    gofs[k] = (q < ng && dy < nyl) ? (z * nlx + lx) * np1 + y0 + dy : -1;
  }
  cplx<T> pf[GPL];
  auto prefetch = [&](int s) {
    const cplx<T>* src = t2 + s * sstride;
#pragma unroll
    for (int k = 0; k < GPL; ++k)
      pf[k] = gofs[k] >= 0 ? src[gofs[k]] : cplx<T>{T(0), T(0)};
  };
  const bool sparse_in = !(OP == X_LOAD || OP == X_LOAD_REAL);
  if (sparse_in && s0 < s1) prefetch(s0);

  for (int s = s0; s < s1; ++s) {
    if (sparse_in) {
      for (int i = lane; i < LPW * np0; i += 64) buf[i] = {T(0), T(0)};
      wave_sync();
#pragma unroll
      for (int k = 0; k < GPL; ++k)
        if (lofs[k] >= 0) buf[lofs[k]] = pf[k];
      wave_sync();
      if (s + 1 < s1) prefetch(s + 1);
      fft_lines_w<+1, EPL>(buf, LPW, np0, g.ax[0], tw, lane);
    } else {
      for (int e = lane; e < LPW * np0; e += 64) {
        cplx<T> val = {T(0), T(0)};
        if (e < nel) {
          if (OP == X_LOAD) {
            const double* fp = v + 2 * ((long)s * N + grow0 + e);
            val = {T(fp[0]), T(fp[1])};
          } else {
            val = {T(scale * v[(long)s * N + grow0 + e]), T(0)};
          }
        }
        buf[e] = val;
      }
      wave_sync();
    }

    if (OP == X_VMUL) {
#pragma unroll
      for (int k = 0; k < EPL; ++k) {
        const int e = lane + k * 64;
        if (e < nel) {
          const cplx<T> p = buf[e];
          buf[e] = {vr[k] * p.x, vr[k] * p.y};
        }
      }
      wave_sync();
    } else if (OP == X_STORE) {
      for (int e = lane; e < nel; e += 64) {
        double* fp = out + 2 * ((long)s * N + grow0 + e);
        fp[0] = double(buf[e].x);
        fp[1] = double(buf[e].y);
      }
      wave_sync();
      continue;
    } else if (OP == X_DENSITY) {
      if (cplx_density) {
        const double f = dens[s];
#pragma unroll
        for (int k = 0; k < EPL; ++k) {
          const int e = lane + k * 64;
          if (e < nel && f > 0.0) {
            const double re = double(buf[e].x), im = double(buf[e].y);
            acc[k] += f * (re * re + im * im);
          }
        }
      } else {
        const double f1 = dens[4 * s + 0], f2 = dens[4 * s + 1];
        const double b1 = dens[4 * s + 2], b2 = dens[4 * s + 3];
#pragma unroll
        for (int k = 0; k < EPL; ++k) {
          const int e = lane + k * 64;
          if (e < nel) {
            const cplx<T> p = buf[e];
            // f = psi1 + i psi2 with psi_j = X_j + conj(c_j(G=0)): Re psi1 = Re f - beta2,
            // Re psi2 = Im f + beta1, Im psi_j = -beta_j
            if (f1 > 0.0) {
              const double r1 = double(p.x) - b2;
              acc[k] += f1 * (r1 * r1 + b1 * b1);
            }
            if (f2 > 0.0) {
              const double r2 = double(p.y) + b1;
              acc[k] += f2 * (r2 * r2 + b2 * b2);
            }
          }
        }
      }
      wave_sync();
      continue;
    }

    // VMUL / LOAD*: forward x transform and store of the sphere lines
    fft_lines_w<-1, EPL>(buf, LPW, np0, g.ax[0], tw, lane);
    {
      cplx<T>* dst = t2 + s * sstride;
#pragma unroll
      for (int k = 0; k < GPL; ++k)
        if (gofs[k] >= 0) dst[gofs[k]] = buf[lofs[k]];
    }
    wave_sync();
  }
  if (OP == X_DENSITY) {
    double* o = out + blockIdx.y * N + grow0;
    const bool one = gridDim.y == 1;  // one slot range: accumulate
#pragma unroll
    for (int k = 0; k < EPL; ++k) {
      const int e = lane + k * 64;
      if (one && e < nel) acc[k] += o[e];
    }
#pragma unroll
    for (int k = 0; k < EPL; ++k) {
      const int e = lane + k * 64;
      if (e < nel) o[e] = acc[k];
    }
  }
}

// ------------------------------------------------------------------------------------
// x pass with the two-factor register transform (fft_reg.h), rows of n = N1*N2:
//   stage A  (bwd): DFT_N1 over stride-N2 elements, twiddle W_n^{j2 k1}
//   stage B  (bwd): DFT_N2 over contiguous blocks -> psi(r) at x = k1 + N1*k2, in
//                   registers; VMUL multiplies by v(r) there and runs stage B of the
//                   forward transform (DFT_N2, twiddle W_n^{-k1 m2}) without leaving
//                   registers; DENSITY accumulates |psi|^2 there; STORE puts psi(r)
//                   back into the rows in natural order and writes the rows to the grid
//   stage A' (fwd): DFT_N1 over stride-N2 elements -> natural order
// Three LDS round trips per slot instead of one per radix pass, and the x-dependent
// multiply touches each element once, in registers.
template <typename T, int OP, int N1, int N2, int GPW>
__global__ void __launch_bounds__(NTHR)
__attribute__((amdgpu_waves_per_eu(Cfg<T>::XWPE)))
k_xpass2(GridDev g, cplx<T>* __restrict__ t2, int nslots, int slots_per_wg,
         const double* __restrict__ v, double* __restrict__ out, const double* __restrict__ dens,
         int cplx_density) {
  constexpr int LPW = x_rows(N1, N2);
  constexpr int YB = LPW * NWAVE;
  constexpr int n = N1 * N2;
  constexpr int TA = LPW * N2, TB = LPW * N1;
  constexpr int IA = (TA + 63) / 64, IB = (TB + 63) / 64;
  extern __shared__ __align__(16) unsigned char smem_raw[];
  const int np1 = g.np1, np2 = g.np2, nlx = g.nlx;
  cplx<T>* tw = reinterpret_cast<cplx<T>*>(smem_raw);
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int nyb = (np1 + YB - 1) / YB;
  const int z = blockIdx.x / nyb;
  const int ywg = (blockIdx.x % nyb) * YB;  // the workgroup's first row
  const int y0 = ywg + wave * LPW;
  // rows of this wavefront; a wavefront with none still takes part in the workgroup
  // barriers below (its transforms run on zeros and every store it would make is masked)
  const int nyl = min(LPW, np1 - y0);
  const int s0 = blockIdx.y * slots_per_wg;
  const int s1 = min(nslots, s0 + slots_per_wg);
  const cplx<T>* twg = twtab<T>(g, 0);
  for (int i = threadIdx.x; i < n; i += NTHR) tw[i] = twg[i];
  __syncthreads();
  using PD = Pad<N1, N2, QBH_XLDS_PAD>;
  constexpr int LD = PD::row(n);
  constexpr int S = N2 + PD::P;
  cplx<T>* buf = tw + n + wave * LPW * LD;
  const long grow0 = ((long)z * np1 + y0) * n;

  T vr[IB][N2];
  double acc[IB][N2];
  // stage-B forward twiddles W_n^{-k1 m2}, m2 = 1..N2-1, of this lane's k1: the same
  // factors twiddle_row forms, computed once instead of per slot (measured at
  // 140 = 14*10: x pass 6.24 -> 6.01 ms per FP64 Hψ).  Not for the FP64 kernels with the
  // full line-element count, which have no registers to spare.
  constexpr int GT = LPW == 4 ? x_middle(n, YB) : x_short(n, YB);
  constexpr bool TWB = QBH_XTWB && (sizeof(T) == 4 || GPW <= GT) && !stockham_order<T, N1, N2>();
  cplx<T> twb[IB][TWB ? N2 - 1 : 1];
  if constexpr (TWB && OP == X_VMUL) {
#pragma unroll
    for (int ib = 0; ib < IB; ++ib) {
      const int k1 = (lane + 64 * ib) % N1;
      cplx<T> w = tw[k1];
      w.y = -w.y;
      cplx<T> p = w;
#pragma unroll
      for (int m = 1; m < N2; ++m) {
        if constexpr (sizeof(T) == 8) p = {tw[k1 * m].x, -tw[k1 * m].y};
        twb[ib][m - 1] = p;
        if (m + 1 < N2) p = cmul(p, w);
      }
    }
  }
#pragma unroll
  for (int ib = 0; ib < IB; ++ib) {
    const int t = lane + 64 * ib;
    const int r = t / N1, k1 = t % N1;
#pragma unroll
    for (int k2 = 0; k2 < N2; ++k2) {
      if (OP == X_VMUL) vr[ib][k2] = (t < TB && r < nyl) ? T(v[grow0 + r * n + k1 + N1 * k2]) : T(0);
      if (OP == X_DENSITY) acc[ib][k2] = 0.0;
    }
  }

  // The workgroup moves the sphere lines of its YB rows together: element q = tid + NTHR*k
  // is row dy = q % YB of line lx = q / YB, so one load instruction covers YB consecutive
  // rows of NTHR/YB lines (YB*sizeof(cplx) contiguous bytes per line) instead of each
  // wavefront's LPW rows.  GPW (a launch parameter) covers
  // nlx*YB elements.  LDS offset (relative to the first row buffer) and T2 offset within a
  // slot are computed once, and the loads and LDS stores are unconditional: an element past
  // the lines loads element 0 of the slot and stores it to this thread's dump entry after
  // the row buffers; a row past np1 loads element 0 into its own (never stored) row.
  const long sstride = (long)np2 * nlx * np1;
  const int ngw = nlx * YB;
  cplx<T>* rows = tw + n;  // row buffers of all wavefronts, row dy at dy * LD
  constexpr int DUMP = NWAVE * LPW * LD;  // + threadIdx.x: one LDS entry per thread
  int lofs[GPW], gofs[GPW];
  unsigned gok = 0;  // bit k: element k is a line entry of a row below np1
#pragma unroll
  for (int k = 0; k < GPW; ++k) {
    const int q = threadIdx.x + k * NTHR;
    const int dy = q % YB, lx = q / YB;
    const bool in = q < ngw, rowok = ywg + dy < np1;
    lofs[k] = in ? dy * LD + PD::idx(g.line_x[lx]) : DUMP + (int)threadIdx.x;
    gofs[k] = (in && rowok) ? (z * nlx + lx) * np1 + ywg + dy : 0;
    if (in && rowok) gok |= 1u << k;
  }
  // the sphere lines of the next XPF slots are in flight in registers while a slot
  // transforms (buffer p of slot s is refilled with slot s + XPF)
  constexpr int XPF = Cfg<T>::XPF;
  cplx<T> pf[XPF][GPW];
  auto prefetch = [&](int s, cplx<T>(&p)[GPW]) {
    const cplx<T>* src = t2 + s * sstride;
#pragma unroll
    for (int k = 0; k < GPW; ++k) {
      const cplx<T> e = src[gofs[k]];
      p[k].x = e.x;
      p[k].y = e.y;
    }
  };
#pragma unroll
  for (int d = 0; d < XPF; ++d)
    if (s0 + d < s1) prefetch(s0 + d, pf[d]);

  // The sphere lines occupy x in [0, xpos_max] and [xneg_min, n).  Stage A input index
  // j1 in [ja, jb] is zero for every j2 and is not read; stage A' outputs there are not
  // needed (FP32 stores them anyway; they are never read).  Only the rest of the rows
  // outside the lines has to be cleared per slot:
  // nz0 <= N2-1 positions below N2*ja and nz1 <= N2-1 below xneg_min, so LPW*(nz0+nz1)
  // < LPW*2*N2 entries, ZK per lane, offsets again computed once.
  const int ja = g.xpos_max / N2 + 1;
  const int jb = g.xneg_min / N2 - 1;
  const int z0a = g.xpos_max + 1, z0b = min(N2 * ja, g.xneg_min);
  const int z1a = max(N2 * (jb + 1), z0b), z1b = g.xneg_min;
  const int nz0 = max(0, z0b - z0a), nz1 = max(0, z1b - z1a);
  constexpr int ZK = (LPW * 2 * N2 + 63) / 64;
  int zofs[ZK];
#pragma unroll
  for (int k = 0; k < ZK; ++k) {
    const int i = lane + 64 * k;
    const int nz = nz0 + nz1;
    zofs[k] = -1;
    if (i < LPW * nz) {
      const int r = i / nz, j = i % nz;
      zofs[k] = r * LD + PD::idx(j < nz0 ? z0a + j : z1a + j - nz0);
    }
  }

  // Per slot: clear (own rows) and scatter (all rows), barrier, transforms on own rows,
  // barrier, gather (all rows), barrier.  Cleared positions are never line positions, so
  // the clear needs no barrier against the scatter or the previous gather.
  auto run_slot = [&](int s, cplx<T>(&p)[GPW]) {
#pragma unroll
    for (int k = 0; k < ZK; ++k)
      if (zofs[k] >= 0) buf[zofs[k]] = {T(0), T(0)};
#pragma unroll
    for (int k = 0; k < GPW; ++k) rows[lofs[k]] = cplx<T>{p[k].x, p[k].y};
    __syncthreads();
    if (s + XPF < s1) prefetch(s + XPF, p);

    // stage A, backward
#pragma unroll
    for (int ia = 0; ia < IA; ++ia) {
      const int t = lane + 64 * ia;
      if (t < TA) {
        const int r = t / N2, j2 = t % N2;
        cplx<T>* row = buf + r * LD + j2;
        cplx<T> a[N1];
#pragma unroll
        for (int j1 = 0; j1 < N1; ++j1)
          a[j1] = (j1 < ja || j1 > jb) ? row[S * j1] : cplx<T>{T(0), T(0)};
        stage_a<N1, N2, +1>(a, tw);
        if constexpr (!stockham_order<T, N1, N2>()) twiddle_row<N1, +1>(a, tw, j2);
#pragma unroll
        for (int k1 = 0; k1 < N1; ++k1) row[S * k1] = a[k1];
      }
    }
    wave_sync();
    if constexpr (OP == X_STORE) {
      // stage B backward for every block of the wavefront's rows first (in registers), then
      // psi(r) back into the rows in natural order and out to the slot's grid: each
      // wavefront's rows are one contiguous stretch of the grid (z fixed, y consecutive)
      cplx<T> bs[IB][N2];
#pragma unroll
      for (int ib = 0; ib < IB; ++ib) {
        const int t = lane + 64 * ib;
        if (t < TB) {
          const int r = t / N1, k1 = t % N1;
          const cplx<T>* blk = buf + r * LD + S * k1;
#pragma unroll
          for (int j2 = 0; j2 < N2; ++j2) bs[ib][j2] = blk[j2];
          stage_b<N1, N2, +1>(bs[ib], tw, k1);
        }
      }
      wave_sync();
#pragma unroll
      for (int ib = 0; ib < IB; ++ib) {
        const int t = lane + 64 * ib;
        if (t < TB) {
          const int r = t / N1, k1 = t % N1;
#pragma unroll
          for (int k2 = 0; k2 < N2; ++k2) buf[r * LD + PD::idx(k1 + N1 * k2)] = bs[ib][k2];
        }
      }
      wave_sync();
      const long ngrid = (long)n * np1 * np2;
      for (int e = lane; e < nyl * n; e += 64) {
        const int r = e / n, x = e - r * n;
        const cplx<T> q = buf[r * LD + PD::idx(x)];
        double* fp = out + 2 * ((long)s * ngrid + grow0 + e);
        fp[0] = double(q.x);
        fp[1] = double(q.y);
      }
      __syncthreads();  // the next scatter overwrites the rows read above
      return;
    }
    if constexpr (OP == X_VMUL && stockham_order<T, N1, N2>()) {
      // F forms: v psi(r) back into the rows in natural order, then the forward transform in
      // the same radix order: one LDS round trip more than the transposed form below, whose
      // reversed radix order rounds differently (110^3, 300 bands: x pass 1.66 -> 0.67 ms
      // against the Stockham passes)
      cplx<T> bs[IB][N2];
#pragma unroll
      for (int ib = 0; ib < IB; ++ib) {
        const int t = lane + 64 * ib;
        if (t < TB) {
          const cplx<T>* blk = buf + (t / N1) * LD + S * (t % N1);
#pragma unroll
          for (int j2 = 0; j2 < N2; ++j2) bs[ib][j2] = blk[j2];
          stage_b<N1, N2, +1>(bs[ib], tw, t % N1);
        }
      }
      wave_sync();
#pragma unroll
      for (int ib = 0; ib < IB; ++ib) {
        const int t = lane + 64 * ib;
        if (t < TB) {
          const int r = t / N1, k1 = t % N1;
#pragma unroll
          for (int k2 = 0; k2 < N2; ++k2)
            buf[r * LD + PD::idx(k1 + N1 * k2)] = {vr[ib][k2] * bs[ib][k2].x,
                                                   vr[ib][k2] * bs[ib][k2].y};
        }
      }
      wave_sync();
      rows_fft<N1, N2, LPW, -1, QBH_XLDS_PAD>(buf, LPW, LD, tw, lane);
      __syncthreads();
      cplx<T>* dst = t2 + s * sstride;
#pragma unroll
      for (int k = 0; k < GPW; ++k)
        if ((gok >> k) & 1u) dst[gofs[k]] = rows[lofs[k]];
      __syncthreads();
      return;
    }
    // stage B: backward DFT_N2 -> psi(r); multiply / accumulate; forward DFT_N2
    double f1 = 0, f2 = 0, b1 = 0, b2 = 0;
    if (OP == X_DENSITY) {
      if (cplx_density) {
        f1 = dens[s];
      } else {
        f1 = dens[4 * s + 0];
        f2 = dens[4 * s + 1];
        b1 = dens[4 * s + 2];
        b2 = dens[4 * s + 3];
      }
    }
#pragma unroll
    for (int ib = 0; ib < IB; ++ib) {
      const int t = lane + 64 * ib;
      if (t < TB) {
        const int r = t / N1, k1 = t % N1;
        cplx<T>* blk = buf + r * LD + S * k1;
        cplx<T> b[N2];
#pragma unroll
        for (int j2 = 0; j2 < N2; ++j2) b[j2] = blk[j2];
        stage_b<N1, N2, +1>(b, tw, k1);
        if (OP == X_VMUL) {
#pragma unroll
          for (int k2 = 0; k2 < N2; ++k2) b[k2] = {vr[ib][k2] * b[k2].x, vr[ib][k2] * b[k2].y};
          sdft<N2, -1>(b);
          if constexpr (TWB) {
            if (k1 != 0) {
#pragma unroll
              for (int m = 1; m < N2; ++m) b[m] = cmul(b[m], twb[ib][m - 1]);
            }
          } else {
            twiddle_row<N2, -1>(b, tw, k1);
          }
#pragma unroll
          for (int m2 = 0; m2 < N2; ++m2) blk[m2] = b[m2];
        } else {
#pragma unroll
          for (int k2 = 0; k2 < N2; ++k2) {
            const double re = double(b[k2].x), im = double(b[k2].y);
            if (cplx_density) {
              if (f1 > 0.0) acc[ib][k2] += f1 * (re * re + im * im);
            } else {
              // f = psi1 + i psi2, psi_j = X_j + conj(c_j(G=0)) (see k_xpass)
              if (f1 > 0.0) {
                const double r1 = re - b2;
                acc[ib][k2] += f1 * (r1 * r1 + b1 * b1);
              }
              if (f2 > 0.0) {
                const double r2 = im + b1;
                acc[ib][k2] += f2 * (r2 * r2 + b2 * b2);
              }
            }
          }
        }
      }
    }
    if (OP == X_DENSITY) {
      __syncthreads();  // the next scatter overwrites line positions read above
      return;
    }
    wave_sync();
    // stage A', forward: natural order
#pragma unroll
    for (int ia = 0; ia < IA; ++ia) {
      const int t = lane + 64 * ia;
      if (t < TA) {
        const int r = t / N2, m2 = t % N2;
        cplx<T>* row = buf + r * LD + m2;
        cplx<T> a[N1];
#pragma unroll
        for (int k1 = 0; k1 < N1; ++k1) a[k1] = row[S * k1];
        sdft<N1, -1>(a);
        // FP32: all N1 outputs, the unneeded ones in [ja, jb] too (stage A of the next slot
        // never reads them and the gather reads line positions only), with no branch per
        // store: FP32 x pass 3.62 -> 3.41 ms at Si512; FP64 3.00 -> 3.06 ms, so FP64 skips
        // them
#pragma unroll
        for (int m1 = 0; m1 < N1; ++m1)
          if (sizeof(T) == 4 || m1 < ja || m1 > jb) row[S * m1] = a[m1];
      }
    }
    __syncthreads();
    {
      cplx<T>* dst = t2 + s * sstride;
#pragma unroll
      for (int k = 0; k < GPW; ++k)
        if ((gok >> k) & 1u) dst[gofs[k]] = rows[lofs[k]];
    }
    __syncthreads();
  };
  for (int s = s0; s < s1; s += XPF) {
#pragma unroll
    for (int d = 0; d < XPF; ++d)
      if (s + d < s1) run_slot(s + d, pf[d]);
  }
  if (OP == X_DENSITY) {
    double* o = out + (long)blockIdx.y * n * np1 * np2 + grow0;
    const bool one = gridDim.y == 1;  // one slot range: accumulate
#pragma unroll
    for (int ib = 0; ib < IB; ++ib) {
      const int t = lane + 64 * ib;
      const int r = t / N1, k1 = t % N1;
      if (t < TB && r < nyl) {
        double* e = o + r * n + k1;
        if (one) {  // (a lane's loads in flight together)
#pragma unroll
          for (int k2 = 0; k2 < N2; ++k2) acc[ib][k2] += e[N1 * k2];
        }
#pragma unroll
        for (int k2 = 0; k2 < N2; ++k2) e[N1 * k2] = acc[ib][k2];
      }
    }
  }
}

// ------------------------------------------------------------------------------------
// x pass of the forward transform from a grid in memory (f complex, or REAL: scale * f + 0i):
// each wavefront reads its rows (one contiguous stretch of the grid, all of a lane's loads in
// flight together), transforms them with the two-factor register transform and the workgroup
// stores the nlx sphere lines, YB consecutive rows of a line at a time.  Bound by HBM: it
// reads the grid and writes T2.  With the LDS Stockham pass it replaces at these edges (198 us
// of it) a backward and a forward transform of 65 orbitals at 72^3 took 343 us, now 208 us.
// FP32 reads its stage twiddles from the table like the Stockham pass: with the repeated products
// of the other FP32 passes a forward transform was 5 to 24 % further from the 64-bit one at the E
// edges (64 along x: 1.54e-7 of the result; tabled 1.30e-7, Stockham 1.30e-7).
template <typename T, bool REAL, int N1, int N2, int GPW>
__global__ void __launch_bounds__(NTHR)
k_xload2(GridDev g, cplx<T>* __restrict__ t2, int nslots, int slots_per_wg,
         const double* __restrict__ f, double scale) {
  constexpr int LPW = x_rows(N1, N2), YB = LPW * NWAVE, n = N1 * N2;
  using PD = Pad<N1, N2, QBH_XLDS_PAD>;
  constexpr int LD = PD::row(n);
  constexpr int EPL = (LPW * n + 63) / 64;  // row elements per lane
  extern __shared__ __align__(16) unsigned char smem_raw[];
  const int np1 = g.np1, np2 = g.np2, nlx = g.nlx;
  cplx<T>* tw = reinterpret_cast<cplx<T>*>(smem_raw);
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int nyb = (np1 + YB - 1) / YB;
  const int z = blockIdx.x / nyb;
  const int ywg = (blockIdx.x % nyb) * YB;
  const int y0 = ywg + wave * LPW;
  const int nyl = max(0, min(LPW, np1 - y0));
  const int s0 = blockIdx.y * slots_per_wg;
  const int s1 = min(nslots, s0 + slots_per_wg);
  const cplx<T>* twg = twtab<T>(g, 0);
  for (int i = threadIdx.x; i < n; i += NTHR) tw[i] = twg[i];
  cplx<T>* rows = tw + n;
  cplx<T>* buf = rows + wave * LPW * LD;
  const long N = (long)n * np1 * np2;
  const long grow0 = ((long)z * np1 + y0) * n;
  const int nel = nyl * n;
  const long sstride = (long)np2 * nlx * np1;
  const int ngw = nlx * YB;
  int lofs[GPW], gofs[GPW];
#pragma unroll
  for (int k = 0; k < GPW; ++k) {
    const int q = threadIdx.x + k * NTHR;
    const int dy = q % YB, lx = q / YB;
    const bool ok = q < ngw && ywg + dy < np1;
    lofs[k] = ok ? dy * LD + PD::idx(g.line_x[lx]) : 0;
    gofs[k] = ok ? (z * nlx + lx) * np1 + ywg + dy : -1;
  }
  __syncthreads();
  for (int s = s0; s < s1; ++s) {
    if (nel > 0) {
      // clamped, branch-free loads: past the rows a lane rereads their last element
      cplx<T> v[EPL];
#pragma unroll
      for (int k = 0; k < EPL; ++k) {
        const long e = (long)s * N + grow0 + min(lane + 64 * k, nel - 1);
        if constexpr (REAL) {
          v[k] = {T(scale * f[e]), T(0)};
        } else {
          v[k] = {T(f[2 * e]), T(f[2 * e + 1])};
        }
      }
#pragma unroll
      for (int k = 0; k < EPL; ++k) {
        const int e = lane + 64 * k;
        if (e < nel) buf[(e / n) * LD + PD::idx(e % n)] = v[k];
      }
    }
    wave_sync();
    rows_fft<N1, N2, LPW, -1, QBH_XLDS_PAD, true>(buf, nyl, LD, tw, lane);
    __syncthreads();
    cplx<T>* dst = t2 + s * sstride;
#pragma unroll
    for (int k = 0; k < GPW; ++k)
      if (gofs[k] >= 0) dst[gofs[k]] = rows[lofs[k]];
    __syncthreads();
  }
}

// ------------------------------------------------------------------------------------
// x pass of band sums of products of transforms, without a grid per band:
//   part[range][d][r] = sum_s w_s Re (IM: Im) (conj(a_s(r)) b_{d,s}(r)),  d < NB
// over the slots with w_s > 0 of a range per blockIdx.y (w null: 1).  a and the b_d are
// y-transformed lines (T2); a workgroup takes the NB + 1 fields of a slot one after the other
// through the same row buffers, the next field's lines in flight, holds a(r) in registers and
// accumulates in FP64.  Against storing the transforms as grids and multiplying them from memory (16 bytes a
// point and band written and read, per field), MI355X: current
// density of 128 bands at 72^3 2.90 -> 1.54 ms, of 64 bands at 60^3 1.19 -> 0.55; TD gradient of
// 64 Si atoms, two steps, 103 -> 87 ms.  Bound like k_xpass2 by vector issue; at two waves per
// SIMD the longest edges with NB = 3 spill (110^3, 64 bands: 8.9 -> 3.0 ms all the same).
struct CrossFields {
  const cplx<double>* t2[4];  // a, b_0 .. b_{NB-1}
};
template <int N1, int N2, int GPW, int NB, bool IM>
__global__ void __launch_bounds__(NTHR) __attribute__((amdgpu_waves_per_eu(2)))
k_xcross2(GridDev g, CrossFields fields, int nslots, int slots_per_wg,
          const double* __restrict__ w, double* __restrict__ part) {
  using C = cplx<double>;
  constexpr int LPW = x_rows(N1, N2), YB = LPW * NWAVE, n = N1 * N2;
  constexpr int TA = LPW * N2, TB = LPW * N1;
  static_assert(TA <= 64 && TB <= 64, "one task per lane and stage");
  using PD = Pad<N1, N2, QBH_XLDS_PAD>;
  constexpr int LD = PD::row(n), S = N2 + PD::P;
  extern __shared__ __align__(16) unsigned char smem_raw[];
  const int np1 = g.np1, np2 = g.np2, nlx = g.nlx;
  C* tw = reinterpret_cast<C*>(smem_raw);
  C* rows = tw + n;
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  C* buf = rows + wave * LPW * LD;
  const int nyb = (np1 + YB - 1) / YB;
  const int z = blockIdx.x / nyb;
  const int ywg = (blockIdx.x % nyb) * YB;
  const int y0 = ywg + wave * LPW;
  const int nyl = min(LPW, np1 - y0);
  const int s0 = blockIdx.y * slots_per_wg;
  const int s1 = min(nslots, s0 + slots_per_wg);
  for (int i = threadIdx.x; i < n; i += NTHR) tw[i] = g.tw64[0][i];

  // line elements of this thread, and the row positions outside the lines that stage A reads
  // and that are cleared per field (see k_xpass2)
  const long sstride = (long)np2 * nlx * np1;
  constexpr int DUMP = YB * LD;
  int lofs[GPW], gofs[GPW];
#pragma unroll
  for (int k = 0; k < GPW; ++k) {
    const int q = threadIdx.x + k * NTHR;
    const int dy = q % YB, lx = q / YB;
    const bool in = q < nlx * YB;
    lofs[k] = in ? dy * LD + PD::idx(g.line_x[lx]) : DUMP + (int)threadIdx.x;
    gofs[k] = in && ywg + dy < np1 ? (z * nlx + lx) * np1 + ywg + dy : 0;
  }
  const int ja = g.xpos_max / N2 + 1;
  const int jb = g.xneg_min / N2 - 1;
  const int z0a = g.xpos_max + 1, z0b = min(N2 * ja, g.xneg_min);
  const int z1a = max(N2 * (jb + 1), z0b), z1b = g.xneg_min;
  const int nz0 = max(0, z0b - z0a), nz = nz0 + max(0, z1b - z1a);
  constexpr int ZK = (LPW * 2 * N2 + 63) / 64;
  int zofs[ZK];
#pragma unroll
  for (int k = 0; k < ZK; ++k) {
    const int i = lane + 64 * k;
    zofs[k] = -1;
    if (i < LPW * nz) {
      const int r = i / nz, j = i % nz;
      zofs[k] = r * LD + PD::idx(j < nz0 ? z0a + j : z1a + j - nz0);
    }
  }
  C pf[GPW];
  auto prefetch = [&](const C* t2, int s) {
    const C* src = t2 + s * sstride;
#pragma unroll
    for (int k = 0; k < GPW; ++k) {
      const C e = src[gofs[k]];
      pf[k].x = e.x;
      pf[k].y = e.y;
    }
  };
  // transforms the field in pf, prefetching the next; out: its values at x = k1 + N1 k2
  const int rb = lane / N1, k1 = lane % N1;
  auto transform = [&](const C* next, int snext, C(&out)[N2]) {
#pragma unroll
    for (int k = 0; k < ZK; ++k)
      if (zofs[k] >= 0) buf[zofs[k]] = {0.0, 0.0};
#pragma unroll
    for (int k = 0; k < GPW; ++k) rows[lofs[k]] = C{pf[k].x, pf[k].y};
    __syncthreads();
    if (next) prefetch(next, snext);
    if (lane < TA) {
      const int j2 = lane % N2;
      C* row = buf + (lane / N2) * LD + j2;
      C a[N1];
#pragma unroll
      for (int j1 = 0; j1 < N1; ++j1)
        a[j1] = (j1 < ja || j1 > jb) ? row[S * j1] : C{0.0, 0.0};
      sdft<N1, +1>(a);
      twiddle_row<N1, +1>(a, tw, j2);
#pragma unroll
      for (int j1 = 0; j1 < N1; ++j1) row[S * j1] = a[j1];
    }
    wave_sync();
    if (lane < TB) {
      const C* blk = buf + rb * LD + S * k1;
#pragma unroll
      for (int j2 = 0; j2 < N2; ++j2) out[j2] = blk[j2];
      sdft<N2, +1>(out);
    }
    __syncthreads();  // the next scatter overwrites rows read above
  };

  double acc[NB][N2];
#pragma unroll
  for (int d = 0; d < NB; ++d)
#pragma unroll
    for (int k2 = 0; k2 < N2; ++k2) acc[d][k2] = 0.0;
  // slots without a positive weight are left out, whatever their transforms hold (0 * NaN)
  auto weighted = [&](int s) {
    if (w)
      while (s < s1 && !(w[s] > 0.0)) ++s;
    return s;
  };
  int s = weighted(s0);
  if (s < s1) prefetch(fields.t2[0], s);
  __syncthreads();
  while (s < s1) {
    C a[N2], b[N2];
    transform(fields.t2[1], s, a);
    const double ws = w ? w[s] : 1.0;
    const int sn = weighted(s + 1);
#pragma unroll
    for (int d = 0; d < NB; ++d) {
      const bool last = d + 1 == NB;
      transform(last ? (sn < s1 ? fields.t2[0] : nullptr) : fields.t2[d + 2 < 4 ? d + 2 : 0],
                last ? sn : s, b);
      if (lane < TB) {
#pragma unroll
        for (int k2 = 0; k2 < N2; ++k2)
          acc[d][k2] += ws * (IM ? a[k2].x * b[k2].y - a[k2].y * b[k2].x
                                 : a[k2].x * b[k2].x + a[k2].y * b[k2].y);
      }
    }
    s = sn;
  }
  if (lane < TB && rb < nyl) {
    const long N = (long)n * np1 * np2;
    double* o = part + (long)blockIdx.y * NB * N + ((long)z * np1 + y0 + rb) * n + k1;
#pragma unroll
    for (int d = 0; d < NB; ++d)
#pragma unroll
      for (int k2 = 0; k2 < N2; ++k2) o[d * N + N1 * k2] = acc[d][k2];
  }
}

// ------------------------------------------------------------------------------------
// z pass, forward: T1 columns -> z transform (exp(-i)) -> x 1/N -> unpack -> output.
// store 0: out[n][G] = ((out + add32) + kin[G]*psi[n][G]) + value;
// store 1: out[n][G] = value;
// store 2: out[n][G] = (add32 + kin[G]*psi[n][G]) + value, out not read (a cleared output:
//          the same sums as store 0 on zeros).
template <typename T, int MODE, int NMAX, int N1, int N2>
__global__ void __launch_bounds__(NTHR)
k_zpass_fwd(GridDev g, const cplx<T>* __restrict__ t1, const double* __restrict__ psi, long ld,
            int nst, int band0, double* __restrict__ out, long ldo,
            const double* __restrict__ kin, int store, const float* __restrict__ add32) {
  constexpr int EPL = Epl<ZLPW, NMAX>::v;
  extern __shared__ __align__(16) unsigned char smem_raw[];
  const int np2 = g.np2;
  cplx<T>* tw = reinterpret_cast<cplx<T>*>(smem_raw);
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int grp = blockIdx.x;
  const int slot = blockIdx.y;
  // this wavefront's lines and the rod its 16-lane group writes out, read before the
  // workgroup barrier so the table loads overlap the twiddle load and the transform
  const int e0 = g.grp_start[grp] + wave * ZLPW;
  const int nl = min(ZLPW, g.grp_start[grp + 1] - e0);
  const int le = lane >> 4;
  const int sub = lane & 15;
  int kind = 4, first = 0, lmin = 0, size = 0;
  if (le < nl) {
    kind = g.ent_kind[e0 + le];
    if (kind != 2 && kind != 4) {
      const int rod = g.ent_rod[e0 + le];
      first = g.rod_first[rod];
      lmin = g.rod_lmin[rod];
      size = g.rod_size[rod];
    }
  }
  const cplx<T>* twg = twtab<T>(g, 2);
  for (int i = threadIdx.x; i < np2; i += NTHR) tw[i] = twg[i];
  __syncthreads();
  if (nl <= 0) return;
  using PD = Pad<N1, N2>;
  const int LD = PD::row(np2);
  cplx<T>* buf = tw + np2 + wave * ZLPW * LD;
  for (int ll = 0; ll < nl; ++ll) {
    const int col = g.ent_col[e0 + ll];
    const cplx<T>* src = t1 + ((long)slot * g.ncol + (col < 0 ? 0 : col)) * np2;
    for (int z = lane; z < np2; z += 64)
      buf[ll * LD + PD::idx(z)] = col < 0 ? cplx<T>{T(0), T(0)} : src[z];
  }
  wave_sync();
  line_fft<-1, EPL, N1, N2, ZLPW>(buf, nl, LD, g.ax[2], tw, lane);

  const double fac = 1.0 / ((double)g.np0 * (double)g.np1 * (double)g.np2);
  int n1, n2;
  if (MODE == SLOT_PAIR) {
    n1 = band0 + 2 * slot;
    n2 = n1 + 1;
  } else {
    n1 = band0 + slot;
    n2 = nst;
  }
  const bool has2 = (MODE == SLOT_PAIR) && (n2 < nst);
  if (le >= nl) return;
  if (kind == 2 || kind == 4) return;  // -G image: handled with its +G partner (next line)
  const cplx<T>* lp = buf + le * LD;
  const cplx<T>* lm = (kind == 1) ? buf + (le + 1) * LD : lp;
  double* o1 = out + 2 * (long)n1 * ldo;
  double* o2 = out + 2 * (long)(has2 ? n2 : n1) * ldo;
  const double* q1 = psi ? psi + 2 * (long)n1 * ld : nullptr;
  const double* q2 = psi ? psi + 2 * (long)(has2 ? n2 : n1) * ld : nullptr;
  // KZ coefficients per lane: the accumulate mode loads hpsi, psi, kin and the FP32 term
  // of all KZ first, then combines and stores them
  constexpr int KZ = 2;
  for (int i0 = sub; i0 < size; i0 += 16 * KZ) {
    double h[KZ][4], q[KZ][4], kk[KZ];
#pragma unroll
    for (int k = 0; k < KZ; ++k) {
      const int i = i0 + 16 * k;
      const int ig = first + i;
      kk[k] = 0.0;
#pragma unroll
      for (int j = 0; j < 4; ++j) h[k][j] = q[k][j] = 0.0;
      if (store == 1 || i >= size) continue;
      if (store == 0) {
        h[k][0] = o1[2 * ig];
        h[k][1] = o1[2 * ig + 1];
      }
      if (add32) {  // FP32 projector term, in the order of a separate add before this pass
        h[k][0] += double(add32[2 * ((long)n1 * g.ngw + ig)]);
        h[k][1] += double(add32[2 * ((long)n1 * g.ngw + ig) + 1]);
      }
      if (kin) {
        kk[k] = kin[ig];
        q[k][0] = q1[2 * ig];
        q[k][1] = q1[2 * ig + 1];
      }
      if (has2) {
        if (store == 0) {
          h[k][2] = o2[2 * ig];
          h[k][3] = o2[2 * ig + 1];
        }
        if (add32) {
          h[k][2] += double(add32[2 * ((long)n2 * g.ngw + ig)]);
          h[k][3] += double(add32[2 * ((long)n2 * g.ngw + ig) + 1]);
        }
        if (kin) {
          q[k][2] = q2[2 * ig];
          q[k][3] = q2[2 * ig + 1];
        }
      }
    }
#pragma unroll
    for (int k = 0; k < KZ; ++k) {
      const int i = i0 + 16 * k;
      if (i >= size) continue;
      const int l = lmin + i;
      const int ig = first + i;
      const cplx<T> zp = lp[PD::idx(wrap(l, np2))];
      double r1, i1, r2 = 0.0, i2 = 0.0;
      if (MODE == SLOT_PAIR) {
        const cplx<T> zm = lm[PD::idx(wrap(-l, np2))];
        const double a = double(zp.x) * fac, b = double(zp.y) * fac;
        const double c = double(zm.x) * fac, d = double(zm.y) * fac;
        r1 = 0.5 * (a + c);
        i1 = 0.5 * (b - d);
        r2 = 0.5 * (b + d);
        i2 = 0.5 * (c - a);
      } else {
        r1 = double(zp.x) * fac;
        i1 = double(zp.y) * fac;
      }
      if (store == 1) {
        o1[2 * ig] = r1;
        o1[2 * ig + 1] = i1;
        if (has2) {
          o2[2 * ig] = r2;
          o2[2 * ig + 1] = i2;
        }
      } else {
        double h0 = h[k][0], h1 = h[k][1];
        if (kin) {
          h0 += kk[k] * q[k][0];
          h1 += kk[k] * q[k][1];
        }
        o1[2 * ig] = h0 + r1;
        o1[2 * ig + 1] = h1 + i1;
        if (has2) {
          double g0 = h[k][2], g1 = h[k][3];
          if (kin) {
            g0 += kk[k] * q[k][2];
            g1 += kk[k] * q[k][3];
          }
          o2[2 * ig] = g0 + r2;
          o2[2 * ig + 1] = g1 + i2;
        }
      }
    }
  }
}

// ------------------------------------------------------------------------------------
// rho += scale * (sum of the nparts partial grids, in slot order; bound by HBM: nparts + 2
// grids)
template <int U>
__global__ void __launch_bounds__(NTHR)
k_density_sum(long N, int nparts, double scale, const double* __restrict__ part,
              double* __restrict__ rho) {
  const long i = blockIdx.x * (long)NTHR + threadIdx.x;
  if (i >= N) return;
  double r = 0.0;
  int p = 0;
  for (; p + U <= nparts; p += U) {  // U partials in flight together
    double v[U];
#pragma unroll
    for (int u = 0; u < U; ++u) v[u] = part[(p + u) * N + i];
#pragma unroll
    for (int u = 0; u < U; ++u) r += v[u];
  }
  for (; p < nparts; ++p) r += part[p * N + i];
  rho[i] += scale * r;
}

// ------------------------------------------------------------------------------------
// y and x passes in one kernel (FP64, both edges n; qbh_fft_plane.h)
struct PlaneOps {
  using Launch = void (*)(hipStream_t st, const GridDev& g, const PipelineArgs& a, int spw,
                          const double* in, double* out, const double* dens, int cplx_density,
                          double scale);
  bool (*fits)(const GridDev& g) = nullptr;
  int (*rounds)(const GridDev& g) = nullptr;  // dependent rounds of one direction (plane_rounds)
  int wgs = 0;  // workgroups per compute unit
  Launch vmul = nullptr, density = nullptr;
  Launch store = nullptr, load = nullptr, load_real = nullptr;  // null: separate passes
};

// Launches.  EdgeOps holds the launch functions of one edge length and precision: the
// z, y and x passes pick theirs by the length of their own axis.
struct EdgeOps {
  int n;  // edge length n1 * n2
  int xr;  // x pass: rows per wavefront
  void (*zbwd)(hipStream_t st, const GridDev& g, const PipelineArgs& a);
  void (*ybwd)(hipStream_t st, const GridDev& g, const PipelineArgs& a);
  void (*yfwd)(hipStream_t st, const GridDev& g, const PipelineArgs& a);
  void (*zfwd)(hipStream_t st, const GridDev& g, const PipelineArgs& a, double* out, long ldo,
               const double* kin, int store);
  // register x passes: potential multiply, store, density (null in the Stockham forms)
  void (*xvmul)(hipStream_t st, const GridDev& g, const PipelineArgs& a, int spw,
                const double* in, double* out, const double* dens, int cplx_density);
  void (*xstore)(hipStream_t st, const GridDev& g, const PipelineArgs& a, int spw,
                 const double* in, double* out, const double* dens, int cplx_density);
  void (*xdensity)(hipStream_t st, const GridDev& g, const PipelineArgs& a, int spw,
                   const double* in, double* out, const double* dens, int cplx_density);
  // register x pass of the forward transform, from a complex or (scaled) real grid
  void (*xload)(hipStream_t st, const GridDev& g, const PipelineArgs& a, int spw,
                const double* f, bool real_input, double scale);
  // band sums of products (FP64): nb fields b of 1 (real part) or 3 (imaginary part)
  void (*xcross)(hipStream_t st, const GridDev& g, const CrossFields& fields, int nslots, int spw,
                 int nb, const double* w, double* part);
  PlaneOps plane;
};

// register-transform edges compiled by unit `part` (qbh_fft_edges.hip)
struct EdgeTable {
  const EdgeOps* ops;
  int count;
};

template <typename T, int N1, int N2, int NMAX>
void launch_zbwd(hipStream_t st, const GridDev& g, const PipelineArgs& a) {
  auto* t1 = static_cast<cplx<T>*>(a.t1);
  const dim3 grid(g.ngroups, a.nslots);
  const size_t lds = sizeof(cplx<T>) *
                     ((size_t)g.np2 + (size_t)NWAVE * ZLPW * Pad<N1, N2>::row(g.np2));
  if (a.mode == SLOT_PAIR)
    k_zpass_bwd<T, SLOT_PAIR, NMAX, N1, N2><<<grid, NTHR, lds, st>>>(g, a.psi, a.ld, a.nst,
                                                                     a.band0, t1);
  else if (a.mode == SLOT_SINGLE_REAL)
    k_zpass_bwd<T, SLOT_SINGLE_REAL, NMAX, N1, N2><<<grid, NTHR, lds, st>>>(g, a.psi, a.ld, a.nst,
                                                                            a.band0, t1);
  else
    k_zpass_bwd<T, SLOT_COMPLEX, NMAX, N1, N2><<<grid, NTHR, lds, st>>>(g, a.psi, a.ld, a.nst,
                                                                        a.band0, t1);
}

template <typename T, int N1, int N2, int NMAX>
void launch_zfwd(hipStream_t st, const GridDev& g, const PipelineArgs& a, double* out, long ldo,
                 const double* kin, int store) {
  auto* t1 = static_cast<cplx<T>*>(a.t1);
  const dim3 grid(g.ngroups, a.nslots);
  const size_t lds = sizeof(cplx<T>) *
                     ((size_t)g.np2 + (size_t)NWAVE * ZLPW * Pad<N1, N2>::row(g.np2));
  if (a.mode == SLOT_PAIR)
    k_zpass_fwd<T, SLOT_PAIR, NMAX, N1, N2><<<grid, NTHR, lds, st>>>(
        g, t1, a.psi, a.ld, a.nst, a.band0, out, ldo, kin, store, a.add32);
  else if (a.mode == SLOT_SINGLE_REAL)
    k_zpass_fwd<T, SLOT_SINGLE_REAL, NMAX, N1, N2><<<grid, NTHR, lds, st>>>(
        g, t1, a.psi, a.ld, a.nst, a.band0, out, ldo, kin, store, a.add32);
  else
    k_zpass_fwd<T, SLOT_COMPLEX, NMAX, N1, N2><<<grid, NTHR, lds, st>>>(
        g, t1, a.psi, a.ld, a.nst, a.band0, out, ldo, kin, store, a.add32);
}

// twiddles, ZB*LB lines, and (forward pass) one int per column of LB lines
template <typename T, int N1, int N2>
size_t lds_y(const GridDev& g) {
  return sizeof(cplx<T>) *
             ((size_t)g.np1 + (size_t)NWAVE * YCfg<T, N1, N2>::LPW * Pad<N1, N2>::row(g.np1)) +
         sizeof(int) * (size_t)YCfg<T, N1, N2>::LB * g.np1;
}

template <typename T, int N1, int N2, int NMAX>
void launch_ybwd(hipStream_t st, const GridDev& g, const PipelineArgs& a) {
  constexpr int ZB = YCfg<T, N1, N2>::ZB, LB = YCfg<T, N1, N2>::LB;
  const dim3 grid(((g.np2 + ZB - 1) / ZB) * ((g.nlx + LB - 1) / LB), a.nslots);
  k_ypass_bwd<T, NMAX, N1, N2><<<grid, NTHR, lds_y<T, N1, N2>(g), st>>>(
      g, static_cast<const cplx<T>*>(a.t1), static_cast<cplx<T>*>(a.t2));
}

template <typename T, int N1, int N2, int NMAX>
void launch_yfwd(hipStream_t st, const GridDev& g, const PipelineArgs& a) {
  constexpr int ZB = YCfg<T, N1, N2>::ZB, LB = YCfg<T, N1, N2>::LB;
  const dim3 grid(((g.np2 + ZB - 1) / ZB) * ((g.nlx + LB - 1) / LB), a.nslots);
  k_ypass_fwd<T, NMAX, N1, N2><<<grid, NTHR, lds_y<T, N1, N2>(g), st>>>(
      g, static_cast<const cplx<T>*>(a.t2), static_cast<cplx<T>*>(a.t1));
}

// register x pass; line elements per thread: a short count for spheres up to half the edge (the
// usual Hψ grid), a middle one for a few lines more, the full edge otherwise
template <typename T, int OP, int N1, int N2>
void launch_x2(hipStream_t st, const GridDev& g, const PipelineArgs& a, int spw, const double* in,
               double* out, const double* dens, int cplx_density) {
  constexpr int n = N1 * N2, YB = x_rows(N1, N2) * NWAVE;
  constexpr int GS = x_short(n, YB), GF = (YB * n + NTHR - 1) / NTHR;
  const dim3 grid(g.np2 * ((g.np1 + YB - 1) / YB), (a.nslots + spw - 1) / spw);
  // twiddles, row buffers and one dump entry per thread
  const size_t lds =
      sizeof(cplx<T>) * ((size_t)n + (size_t)YB * Pad<N1, N2, QBH_XLDS_PAD>::row(n) + NTHR);
  auto* t2 = static_cast<cplx<T>*>(a.t2);
  constexpr int GM = OP == X_VMUL || OP == X_DENSITY ? x_middle(n, YB) : GS;
  const int need = (g.nlx * YB + NTHR - 1) / NTHR;
  if (need <= GS)
    k_xpass2<T, OP, N1, N2, GS><<<grid, NTHR, lds, st>>>(g, t2, a.nslots, spw, in, out, dens,
                                                         cplx_density);
  else if (GM < GF && need <= GM)
    k_xpass2<T, OP, N1, N2, GM><<<grid, NTHR, lds, st>>>(g, t2, a.nslots, spw, in, out, dens,
                                                         cplx_density);
  else
    k_xpass2<T, OP, N1, N2, GF><<<grid, NTHR, lds, st>>>(g, t2, a.nslots, spw, in, out, dens,
                                                         cplx_density);
}

// factors of n = n1 * n2 in the order of k_xload2: FP32 takes the one with more powers of two
// first, like the Stockham plans, which lead with them (error of an FP32 forward transform, 72 along
// x: 1.29e-7 of the result as 8 * 9, 1.36e-7 as 9 * 8, 1.32e-7 with the Stockham x pass)
constexpr int twos(int n) { return n % 2 ? 0 : 1 + twos(n / 2); }
template <typename T, int N1, int N2> struct LoadFactors {
  static constexpr bool swap = sizeof(T) == 4 && !stockham_order<T, N1, N2>() && twos(N2) > twos(N1);
  static constexpr int A = swap ? N2 : N1, B = swap ? N1 : N2;
};

template <typename T, int N1, int N2>
void launch_xload2(hipStream_t st, const GridDev& g, const PipelineArgs& a, int spw,
                   const double* f, bool real_input, double scale) {
  constexpr int n = N1 * N2, YB = x_rows(N1, N2) * NWAVE;
  constexpr int A = LoadFactors<T, N1, N2>::A, B = LoadFactors<T, N1, N2>::B;
  constexpr int GF = (YB * n + NTHR - 1) / NTHR;
  const dim3 grid(g.np2 * ((g.np1 + YB - 1) / YB), (a.nslots + spw - 1) / spw);
  const size_t lds = sizeof(cplx<T>) * ((size_t)n + (size_t)YB * Pad<A, B, QBH_XLDS_PAD>::row(n));
  auto* t2 = static_cast<cplx<T>*>(a.t2);
  if (real_input)
    k_xload2<T, true, A, B, GF><<<grid, NTHR, lds, st>>>(g, t2, a.nslots, spw, f, scale);
  else
    k_xload2<T, false, A, B, GF><<<grid, NTHR, lds, st>>>(g, t2, a.nslots, spw, f, scale);
}

template <int N1, int N2>
void launch_xcross2(hipStream_t st, const GridDev& g, const CrossFields& fields, int nslots,
                    int spw, int nb, const double* w, double* part) {
  constexpr int n = N1 * N2, YB = x_rows(N1, N2) * NWAVE;
  constexpr int GS = x_short(n, YB), GF = (YB * n + NTHR - 1) / NTHR;
  const dim3 grid(g.np2 * ((g.np1 + YB - 1) / YB), (nslots + spw - 1) / spw);
  const size_t lds =
      sizeof(cplx<double>) * ((size_t)n + (size_t)YB * Pad<N1, N2, QBH_XLDS_PAD>::row(n) + NTHR);
  const bool small = (g.nlx * YB + NTHR - 1) / NTHR <= GS;
  if (nb == 1 && small)
    k_xcross2<N1, N2, GS, 1, false><<<grid, NTHR, lds, st>>>(g, fields, nslots, spw, w, part);
  else if (nb == 1)
    k_xcross2<N1, N2, GF, 1, false><<<grid, NTHR, lds, st>>>(g, fields, nslots, spw, w, part);
  else if (small)
    k_xcross2<N1, N2, GS, 3, true><<<grid, NTHR, lds, st>>>(g, fields, nslots, spw, w, part);
  else
    k_xcross2<N1, N2, GF, 3, true><<<grid, NTHR, lds, st>>>(g, fields, nslots, spw, w, part);
}

}  // namespace qbh
#include "qbh_fft_plane.h"
namespace qbh {

template <typename T, int N1, int N2>
constexpr EdgeOps make_edge() {
  return EdgeOps{N1 * N2,
                 x_rows(N1, N2),
                 launch_zbwd<T, N1, N2, 144>,
                 launch_ybwd<T, N1, N2, 144>,
                 launch_yfwd<T, N1, N2, 144>,
                 launch_zfwd<T, N1, N2, 144>,
                 launch_x2<T, X_VMUL, N1, N2>,
                 launch_x2<T, X_STORE, N1, N2>,
                 launch_x2<T, X_DENSITY, N1, N2>,
                 launch_xload2<T, N1, N2>,
                 sizeof(T) == 8 ? launch_xcross2<N1, N2> : nullptr,
                 plane_edge<T, N1, N2>()};
}

}  // namespace qbh
