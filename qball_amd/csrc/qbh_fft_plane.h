// y, x and y passes of one FP64 local Hψ in one kernel, for grids of np0 = np1 = n, and with the
// y and x passes alone the density and the transforms to and from grids: a workgroup
// holds the (slot, z) plane of the pruned transform in LDS (n rows of the nlx lines that hold
// sphere points), so T2 never exists and T1 is read and written once.  At 72^3 with 128 complex
// bands the three passes move 1.65 GB and this kernel 0.25 GB.
//
// Per plane: the columns are scattered into cleared rows; the y transforms run in place with
// lanes across the lines (stage A rows j2 + N2 j1 -> j2 + N2 k1, stage B N2 k1 + j2 ->
// N2 k1 + k2, which then holds y = k1 + N1 k2: the rows stay in that order and only the look-up
// of v knows it); each wavefront takes LPW rows at a time through the x transforms of k_xpass2
// in a row buffer of its own; the forward y transforms run the stages in reverse, back to
// natural order.  Absent positions of a row are read from a line that stays zero and written to
// one that is never read: with per-element branches instead, which skip the zero rows and
// positions, 72^3 took 334 us against 320.
//
// Bound by LDS and FP64 instruction issue, each busy about 40 % of the time, with too few
// wavefronts to overlap them fully: two workgroups of four wavefronts per compute unit up to
// n = 80, one of eight above.  Workgroups are placed from the same SIMD on, so 5 or 6
// wavefronts each (445, 487 us at 72^3) leave room for only one; one workgroup of 12: 422 us.
// y, x and y passes before -> here (MI355X): 72^3, 128 complex bands 446 -> 317 us, 128 real
// bands 223 -> 166; 64^3, 128 real bands 160 -> 98; 88^3, 195 real bands 759 -> 558; 40^3, 16
// real bands 27 -> 13.5; 48^3 with nlx = 35, 64 real bands 82 -> 44.
#pragma once

namespace qbh {

template <int N1, int N2> struct Plane {
  static constexpr int n = N1 * N2;
  static constexpr int NW = n <= 80 ? 4 : 8;  // wavefronts
  static constexpr int WGS = n <= 80 ? 2 : 1;  // workgroups per compute unit
  static constexpr int LPW = x_rows(N1, N2);
  static constexpr int LDX = Pad<N1, N2, 1>::row(n);
  static constexpr int KC = 4;  // columns per thread loaded ahead
  // row stride: the lines, one that stays zero and one for unwanted output
  static __host__ __device__ int ldp(int nlx) { return (nlx + 2) | 1; }
  static size_t lds(int nlx) {
    return sizeof(cplx<double>) * ((size_t)n + (size_t)n * ldp(nlx) + (size_t)NW * LPW * LDX) +
           sizeof(int) * n;
  }
};

template <int OP, int N1, int N2>
__global__ void __launch_bounds__((Plane<N1, N2>::NW * 64))
__attribute__((amdgpu_waves_per_eu(Plane<N1, N2>::n <= 60 ? 3 : 2)))
k_plane(GridDev g, cplx<double>* __restrict__ t1, int nslots, int spw, int nwork,
        const double* __restrict__ in,     // VMUL: potential; LOAD*: grid
        double* __restrict__ out,          // STORE: grid; DENSITY: as k_xpass2
        const double* __restrict__ dens, int cplx_density, double scale) {
  constexpr bool LOAD = OP == X_LOAD || OP == X_LOAD_REAL;
  constexpr bool BWD = !LOAD, FWD = LOAD || OP == X_VMUL;
  using T = double;
  using C = Plane<N1, N2>;
  constexpr int n = C::n, NW = C::NW, NT = NW * 64, LPW = C::LPW, LDX = C::LDX, KC = C::KC;
  constexpr int S = N2 + Pad<N1, N2, 1>::P;
  constexpr int TA = LPW * N2, TB = LPW * N1;
  static_assert(TA <= 64 && TB <= 64, "one task per lane");
  extern __shared__ __align__(16) unsigned char smem_raw[];
  // consecutive planes of a slot range to one XCD: 8 of them share every 128-byte line of T1
  const int chunk = (nwork + 7) / 8;
  const int work = (blockIdx.x & 7) * chunk + (blockIdx.x >> 3);
  if (work >= nwork) return;
  const int np2 = g.np2, nlx = g.nlx, ncol = g.ncol;
  const int z = work % np2;
  const int s0 = work / np2 * spw, s1 = min(nslots, s0 + spw);
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int LDP = C::ldp(nlx);
  cplx<T>* tw = reinterpret_cast<cplx<T>*>(smem_raw);
  cplx<T>* P = tw + n;
  cplx<T>* buf = P + n * LDP + wave * LPW * LDX;
  int* xl = reinterpret_cast<int*>(P + n * LDP + NW * LPW * LDX);
  const cplx<T>* twx = g.tw64[0];
  for (int i = tid; i < n; i += NT) {
    tw[i] = twx[i];
    xl[i] = nlx;
  }
  __syncthreads();
  for (int i = tid; i < nlx; i += NT) xl[g.line_x[i]] = i;
  __syncthreads();
  const int ra = lane / N2, j2a = lane % N2;
  const int rb = lane / N1, k1b = lane % N1;
  int px[N1];
#pragma unroll
  for (int j1 = 0; j1 < N1; ++j1) px[j1] = xl[j2a + N2 * j1];
  auto col_ofs = [&](int c) {
    int lo = 0, hi = nlx;  // line of column c
    while (hi - lo > 1) {
      const int m = (lo + hi) >> 1;
      if (g.line_start[m] <= c) lo = m;
      else hi = m;
    }
    return g.col_y[c] * LDP + lo;
  };
  int pofs[KC];
#pragma unroll
  for (int k = 0; k < KC; ++k) {
    const int c = tid + k * NT;
    pofs[k] = c < ncol ? col_ofs(c) : -1;
  }
  // stage twiddles of the x transforms held in registers where LDS allows two wavefronts per
  // SIMD anyway and the registers suffice (72^3, 128 real bands: 174 -> 166 us)
  constexpr bool TWR = OP == X_VMUL && n > 60 && n <= 80;
  cplx<T> twa[TWR ? N1 : 1], twb[TWR ? N2 : 1];
  if constexpr (TWR) {
#pragma unroll
    for (int k = 1; k < N1; ++k) twa[k] = tw[j2a * k];
#pragma unroll
    for (int k = 1; k < N2; ++k) twb[k] = {tw[k1b * k].x, -tw[k1b * k].y};
  }
  cplx<T> pf[KC];
  auto prefetch = [&](int s) {
    const cplx<T>* src = t1 + (long)s * ncol * np2 + z;
#pragma unroll
    for (int k = 0; k < KC; ++k) {
      const cplx<T> e = src[(long)(pofs[k] >= 0 ? tid + k * NT : 0) * np2];
      pf[k].x = e.x;
      pf[k].y = e.y;
    }
  };
  if constexpr (BWD) prefetch(s0);
  const long N = (long)n * n * np2, gz = (long)z * n * n;
  constexpr int RND = (n + NW * LPW - 1) / (NW * LPW);  // x rounds of a wavefront
  double acc[OP == X_DENSITY ? RND : 1][N2];
  if constexpr (OP == X_DENSITY)
#pragma unroll
    for (int i = 0; i < RND; ++i)
#pragma unroll
      for (int k2 = 0; k2 < N2; ++k2) acc[i][k2] = 0.0;
  for (int s = s0; s < s1; ++s) {
    cplx<T>* tp = t1 + (long)s * ncol * np2 + z;
    if constexpr (BWD) {
      for (int i = tid; i < n * LDP; i += NT) P[i] = {0.0, 0.0};
      __syncthreads();
#pragma unroll
      for (int k = 0; k < KC; ++k)
        if (pofs[k] >= 0) P[pofs[k]] = cplx<T>{pf[k].x, pf[k].y};
      for (int c = tid + KC * NT; c < ncol; c += NT) P[col_ofs(c)] = tp[(long)c * np2];
      __syncthreads();
      if (s + 1 < s1) prefetch(s + 1);
      // y backward: rows j2 + N2 j1 -> j2 + N2 k1 -> N2 k1 + k2 holds y = k1 + N1 k2
      for (int t = tid; t < nlx * N2; t += NT) {
        const int j2 = t / nlx;
        cplx<T>* p = P + j2 * LDP + (t - j2 * nlx);
        cplx<T> a[N1];
#pragma unroll
        for (int j1 = 0; j1 < N1; ++j1) a[j1] = p[N2 * j1 * LDP];
        sdft<N1, +1>(a);
        twiddle_row<N1, +1>(a, tw, j2);
#pragma unroll
        for (int k1 = 0; k1 < N1; ++k1) p[N2 * k1 * LDP] = a[k1];
      }
      __syncthreads();
      for (int t = tid; t < nlx * N1; t += NT) {
        const int k1 = t / nlx;
        cplx<T>* p = P + N2 * k1 * LDP + (t - k1 * nlx);
        cplx<T> b[N2];
#pragma unroll
        for (int j2 = 0; j2 < N2; ++j2) b[j2] = p[j2 * LDP];
        sdft<N2, +1>(b);
#pragma unroll
        for (int k2 = 0; k2 < N2; ++k2) p[k2 * LDP] = b[k2];
      }
      __syncthreads();
    }
    double f1 = 0, f2 = 0, b1 = 0, b2 = 0;
    if constexpr (OP == X_DENSITY) {
      f1 = dens[cplx_density ? s : 4 * s];
      if (!cplx_density) {
        f2 = dens[4 * s + 1];
        b1 = dens[4 * s + 2];
        b2 = dens[4 * s + 3];
      }
    }
    auto rows = [&](int p0, double* ac) {
      const int nr = min(LPW, n - p0);
      const int prow = (p0 + ra) * LDP;
      // grid offset of row r of the round
      auto grow = [&](int r) {
        const int p = p0 + r;
        return gz + (long)(p / N2 + N1 * (p % N2)) * n;
      };
      if constexpr (LOAD) {
        constexpr int EPL = (LPW * n + 63) / 64;
        const int nel = nr * n;
        cplx<T> e[EPL];
#pragma unroll
        for (int k = 0; k < EPL; ++k) {  // past the rows a lane rereads their last element
          const int i = min(lane + 64 * k, nel - 1);
          const long o = (long)s * N + grow(i / n) + i % n;
          if constexpr (OP == X_LOAD_REAL) {
            e[k] = {scale * in[o], 0.0};
          } else {
            e[k] = {in[2 * o], in[2 * o + 1]};
          }
        }
#pragma unroll
        for (int k = 0; k < EPL; ++k) {
          const int i = lane + 64 * k;
          if (i < nel) buf[(i / n) * LDX + Pad<N1, N2, 1>::idx(i % n)] = e[k];
        }
        wave_sync();
        rows_fft<N1, N2, LPW, -1, 1>(buf, nr, LDX, tw, lane);
        if (ra < nr)
#pragma unroll
          for (int j1 = 0; j1 < N1; ++j1)
            P[prow + px[j1] + (px[j1] == nlx)] = buf[ra * LDX + j2a + S * j1];
        wave_sync();
        return;
      }
      double vr[N2];
      if constexpr (OP == X_VMUL) {
        const double* vy = in + grow(min(rb, nr - 1)) + k1b;
#pragma unroll
        for (int k2 = 0; k2 < N2; ++k2) vr[k2] = vy[N1 * k2];
      }
      if (ra < nr) {
        cplx<T> a[N1];
#pragma unroll
        for (int j1 = 0; j1 < N1; ++j1) a[j1] = P[prow + px[j1]];
        sdft<N1, +1>(a);
        if constexpr (TWR) {
#pragma unroll
          for (int k1 = 1; k1 < N1; ++k1) a[k1] = cmul(a[k1], twa[k1]);
        } else {
          twiddle_row<N1, +1>(a, tw, j2a);
        }
        cplx<T>* w = buf + ra * LDX + j2a;
#pragma unroll
        for (int k1 = 0; k1 < N1; ++k1) w[S * k1] = a[k1];
      }
      wave_sync();
      cplx<T>* blk = buf + rb * LDX + S * k1b;
      cplx<T> b[N2];
      if (rb < nr) {
#pragma unroll
        for (int j2 = 0; j2 < N2; ++j2) b[j2] = blk[j2];
        sdft<N2, +1>(b);
        if constexpr (OP == X_VMUL) {
#pragma unroll
          for (int k2 = 0; k2 < N2; ++k2) b[k2] = {vr[k2] * b[k2].x, vr[k2] * b[k2].y};
          sdft<N2, -1>(b);
          if constexpr (TWR) {
#pragma unroll
            for (int m2 = 1; m2 < N2; ++m2) b[m2] = cmul(b[m2], twb[m2]);
          } else {
            twiddle_row<N2, -1>(b, tw, k1b);
          }
#pragma unroll
          for (int m2 = 0; m2 < N2; ++m2) blk[m2] = b[m2];
        }
        if constexpr (OP == X_DENSITY) {
#pragma unroll
          for (int k2 = 0; k2 < N2; ++k2) {
            if (cplx_density) {
              if (f1 > 0.0) ac[k2] += f1 * (b[k2].x * b[k2].x + b[k2].y * b[k2].y);
            } else {  // psi_j = X_j + conj(c_j(G=0)) (see k_xpass)
              const double r1 = b[k2].x - b2, r2 = b[k2].y + b1;
              if (f1 > 0.0) ac[k2] += f1 * (r1 * r1 + b1 * b1);
              if (f2 > 0.0) ac[k2] += f2 * (r2 * r2 + b2 * b2);
            }
          }
        }
      }
      wave_sync();
      if constexpr (OP == X_STORE) {
        if (rb < nr)
#pragma unroll
          for (int k2 = 0; k2 < N2; ++k2)
            buf[rb * LDX + Pad<N1, N2, 1>::idx(k1b + N1 * k2)] = b[k2];
        wave_sync();
        for (int i = lane; i < nr * n; i += 64) {
          const int r = i / n, x = i - r * n;
          const cplx<T> q = buf[r * LDX + Pad<N1, N2, 1>::idx(x)];
          double* o = out + 2 * ((long)s * N + grow(r) + x);
          o[0] = q.x;
          o[1] = q.y;
        }
        wave_sync();
      }
      if constexpr (OP == X_VMUL) {
        if (ra < nr) {
          const cplx<T>* w = buf + ra * LDX + j2a;
          cplx<T> a[N1];
#pragma unroll
          for (int k1 = 0; k1 < N1; ++k1) a[k1] = w[S * k1];
          sdft<N1, -1>(a);
#pragma unroll
          for (int m1 = 0; m1 < N1; ++m1) P[prow + px[m1] + (px[m1] == nlx)] = a[m1];
        }
        wave_sync();
      }
    };
    if constexpr (OP == X_DENSITY) {
#pragma unroll
      for (int i = 0; i < RND; ++i)
        if ((i * NW + wave) * LPW < n) rows((i * NW + wave) * LPW, acc[i]);
    } else {
      for (int p0 = wave * LPW; p0 < n; p0 += NW * LPW) rows(p0, nullptr);
    }
    __syncthreads();
    if constexpr (!FWD) continue;
    for (int t = tid; t < nlx * N1; t += NT) {
      const int k1 = t / nlx;
      cplx<T>* p = P + N2 * k1 * LDP + (t - k1 * nlx);
      cplx<T> b[N2];
#pragma unroll
      for (int k2 = 0; k2 < N2; ++k2) b[k2] = p[k2 * LDP];
      sdft<N2, -1>(b);
      twiddle_row<N2, -1>(b, tw, k1);
#pragma unroll
      for (int m2 = 0; m2 < N2; ++m2) p[m2 * LDP] = b[m2];
    }
    __syncthreads();
    for (int t = tid; t < nlx * N2; t += NT) {
      const int m2 = t / nlx;
      cplx<T>* p = P + m2 * LDP + (t - m2 * nlx);
      cplx<T> a[N1];
#pragma unroll
      for (int k1 = 0; k1 < N1; ++k1) a[k1] = p[N2 * k1 * LDP];
      sdft<N1, -1>(a);
#pragma unroll
      for (int m1 = 0; m1 < N1; ++m1) p[N2 * m1 * LDP] = a[m1];
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < KC; ++k)
      if (pofs[k] >= 0) tp[(long)(tid + k * NT) * np2] = P[pofs[k]];
    for (int c = tid + KC * NT; c < ncol; c += NT) tp[(long)c * np2] = P[col_ofs(c)];
    __syncthreads();
  }
  if constexpr (OP == X_DENSITY) {
    const bool one = nwork == np2;  // one slot range: accumulate
    double* o = out + (long)(work / np2) * N + gz;
#pragma unroll
    for (int i = 0; i < RND; ++i) {
      const int p = (i * NW + wave) * LPW + rb;
      if (rb < LPW && p < n) {
#pragma unroll
        for (int k2 = 0; k2 < N2; ++k2) {
          double* e = o + (long)(p / N2 + N1 * (p % N2)) * n + k1b + N1 * k2;
          *e = one ? *e + acc[i][k2] : acc[i][k2];
        }
      }
    }
  }
}

template <int N1, int N2>
bool plane_fits(const GridDev& g) {
  return Plane<N1, N2>::WGS * Plane<N1, N2>::lds(g.nlx) <= 163840;
}

// rounds of tasks that follow one another in the workgroup for one direction of a plane: the
// two stages of the y transforms (nlx lines) and the row groups of the x transforms
template <int N1, int N2>
int plane_rounds(const GridDev& g) {
  using C = Plane<N1, N2>;
  constexpr int NT = C::NW * 64, R = C::NW * C::LPW;
  return (g.nlx * N1 + NT - 1) / NT + (g.nlx * N2 + NT - 1) / NT + (C::n + R - 1) / R;
}

template <int OP, int N1, int N2>
void launch_plane(hipStream_t st, const GridDev& g, const PipelineArgs& a, int spw,
                  const double* in, double* out, const double* dens, int cplx_density,
                  double scale) {
  using C = Plane<N1, N2>;
  const int nwork = g.np2 * ((a.nslots + spw - 1) / spw);
  k_plane<OP, N1, N2><<<(nwork + 7) / 8 * 8, C::NW * 64, C::lds(g.nlx), st>>>(
      g, static_cast<cplx<double>*>(a.t1), a.nslots, spw, nwork, in, out, dens, cplx_density,
      scale);
}

// The plane forms of an edge, none where its plane never fits.  Transforms to and from grids in
// memory only up to edge 64: above, the plane's short runs of grid loads and stores cost what
// T2 does (y and x pass -> plane, backward / forward: 40^3, 16 real bands 17.6 -> 12.5 / 17.7 ->
// 12.4 us; 64^3, 128 real bands 123 -> 77 / 119 -> 103; 72^3, 65 real bands 91 -> 88 / 96 -> 97,
// both directions with their z passes 202 -> 212).
template <typename T, int N1, int N2>
constexpr PlaneOps plane_edge() {
  PlaneOps p;
  if constexpr (sizeof(T) == 8 && N1 * N2 <= 108) {
    p.fits = plane_fits<N1, N2>;
    p.rounds = plane_rounds<N1, N2>;
    p.wgs = Plane<N1, N2>::WGS;
    p.vmul = launch_plane<X_VMUL, N1, N2>;
    p.density = launch_plane<X_DENSITY, N1, N2>;
    if constexpr (N1 * N2 <= 64) {
      p.store = launch_plane<X_STORE, N1, N2>;
      p.load = launch_plane<X_LOAD, N1, N2>;
      p.load_real = launch_plane<X_LOAD_REAL, N1, N2>;
    }
  }
  return p;
}

}  // namespace qbh
