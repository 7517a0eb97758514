// G-sphere <-> grid transform pipeline: dispatch by edge length, and the LDS Stockham forms
// of the passes (the kernels and their design are in qbh_fft_kernels.h).
#include <cstdio>
#include <optional>

#include "qbh_fft_edges.h"
#include "qbh_fft_kernels.h"

namespace qbh {

size_t slot_bytes(const Basis* b, int prec) {
  const size_t c = prec == PREC_FP64 ? 16 : 8;
  const GridDev& g = b->g;
  return c * ((size_t)g.ncol * g.np2 + (size_t)g.np2 * g.nlx * g.np1);
}

static int check_launch(Ctx* ctx, const char* what) {
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) {
    ctx->last_error = std::string(what) + ": " + hipGetErrorString(e);
    return -3;
  }
  return 0;
}

#define QBH_DECLARE_PART(p) EdgeTable edge_table_##p(int prec);
QBH_EDGE_PARTS(QBH_DECLARE_PART)
#undef QBH_DECLARE_PART

// launch functions of the register transforms of length n, null if it has none
static const EdgeOps* register_ops(int n, int prec) {
  static const struct Tables {
    const EdgeOps* ops[2][257] = {};
    Tables() {
      for (int pr : {PREC_FP64, PREC_FP32}) {
#define QBH_ADD_PART(p)                                                       \
  {                                                                           \
    const EdgeTable t = edge_table_##p(pr);                                   \
    for (int i = 0; i < t.count; ++i) ops[pr][t.ops[i].n] = &t.ops[i];        \
  }
        QBH_EDGE_PARTS(QBH_ADD_PART)
#undef QBH_ADD_PART
      }
    }
  } tables;
  return n >= 0 && n <= 256 ? tables.ops[prec][n] : nullptr;
}

bool register_edge(int n) { return register_ops(n, PREC_FP64) != nullptr; }

// Stockham forms of the z and y passes; NMAX 144 covers every edge up to 144 (9 elements per
// lane for 4-line wavefronts), 256 the rest
template <typename T, int NMAX>
static constexpr EdgeOps stockham_edge() {
  return EdgeOps{0,
                 Cfg<T>::LPW,
                 launch_zbwd<T, 0, 0, NMAX>,
                 launch_ybwd<T, 0, 0, NMAX>,
                 launch_yfwd<T, 0, 0, NMAX>,
                 launch_zfwd<T, 0, 0, NMAX>,
                 nullptr,
                 nullptr,
                 nullptr,
                 nullptr,
                 nullptr,
                 {}};
}
static const EdgeOps kStockham[2][2] = {
    {stockham_edge<double, 144>(), stockham_edge<double, 256>()},
    {stockham_edge<float, 144>(), stockham_edge<float, 256>()}};

// z / y passes of edge length n: the register transform where there is one, unless the
// basis' tuning turns it off
static const EdgeOps& zy_ops(const Basis* b, int n, int prec) {
  const EdgeOps* r = b->tune.zy_reg ? register_ops(n, prec) : nullptr;
  return r ? *r : kStockham[prec][n <= 144 ? 0 : 1];
}

static int bwd_z(Ctx* ctx, Basis* b, const PipelineArgs& a) {
  const GridDev& g = b->g;
  {
    TimedLaunch tl(ctx, "zpass_bwd");
    zy_ops(b, g.np2, a.prec).zbwd(ctx->stream, g, a);
  }
  return check_launch(ctx, "zpass_bwd");
}

static int bwd_yz(Ctx* ctx, Basis* b, const PipelineArgs& a) {
  const GridDev& g = b->g;
  if (int r = bwd_z(ctx, b, a)) return r;
  {
    TimedLaunch tl(ctx, "ypass_bwd");
    zy_ops(b, g.np1, a.prec).ybwd(ctx->stream, g, a);
  }
  return check_launch(ctx, "ypass_bwd");
}

static int fwd_z(Ctx* ctx, Basis* b, const PipelineArgs& a, double* out, long ldo,
                 const double* kin, int store) {
  const GridDev& g = b->g;
  if (a.wait_z) hipStreamWaitEvent(ctx->stream, a.wait_z, 0);
  {
    TimedLaunch tl(ctx, "zpass_fwd");
    zy_ops(b, g.np2, a.prec).zfwd(ctx->stream, g, a, out, ldo, kin, store);
  }
  return check_launch(ctx, "zpass_fwd");
}

static int fwd_zy(Ctx* ctx, Basis* b, const PipelineArgs& a, double* out, long ldo,
                  const double* kin, int store) {
  const GridDev& g = b->g;
  {
    TimedLaunch tl(ctx, "ypass_fwd");
    zy_ops(b, g.np1, a.prec).yfwd(ctx->stream, g, a);
  }
  if (int r = check_launch(ctx, "ypass_fwd")) return r;
  return fwd_z(ctx, b, a, out, ldo, kin, store);
}

// slots per x-pass workgroup: keep >= 4096 workgroups in flight while amortising the
// potential rows and twiddles over several slots.  Measured on the Si64 complex basis (72^3,
// 128 slots): 4 slots per workgroup (11520 workgroups) 0.760/0.516 ms per FP64/FP32 Hψ, 8
// (5760) 0.747/0.495 ms, 16 (2880) 0.754/0.484 ms; Si512 and Al500 reach the cap of 16.
static int x_slots_per_wg(const GridDev& g, int nslots, int yb) {
  const long rows = (long)g.np2 * ((g.np1 + yb - 1) / yb);
  int spw = 1;
  while (spw < 16 && rows * ((nslots + 2 * spw - 1) / (2 * spw)) >= 4096) spw *= 2;
  return spw;
}

// Stockham x pass
template <typename T, int OP>
static void launch_x(hipStream_t st, const GridDev& g, const PipelineArgs& a, int spw,
                     const double* in, double* out, const double* dens, double scale,
                     int cplx_density) {
  constexpr int YB = Cfg<T>::LPW * NWAVE;
  const dim3 grid(g.np2 * ((g.np1 + YB - 1) / YB), (a.nslots + spw - 1) / spw);
  const size_t lds = sizeof(cplx<T>) * ((size_t)g.np0 + (size_t)YB * g.np0);
  auto* t2 = static_cast<cplx<T>*>(a.t2);
  if (g.np0 <= 144)
    k_xpass<T, OP, 144><<<grid, NTHR, lds, st>>>(g, t2, a.nslots, spw, in, out, dens, scale,
                                                 cplx_density);
  else
    k_xpass<T, OP, 256><<<grid, NTHR, lds, st>>>(g, t2, a.nslots, spw, in, out, dens, scale,
                                                 cplx_density);
}

template <typename T, int OP>
static int xpass_t(Ctx* ctx, Basis* b, const PipelineArgs& a, const double* in, double* out,
                   const double* dens, double scale, int cplx_density, const char* name) {
  const GridDev& g = b->g;
  const EdgeOps* r = b->tune.x_reg ? register_ops(g.np0, a.prec) : nullptr;
  auto reg = !r ? nullptr
             : OP == X_VMUL ? r->xvmul
             : OP == X_STORE ? r->xstore
             : OP == X_DENSITY ? r->xdensity
                               : nullptr;
  constexpr bool LOAD = OP == X_LOAD || OP == X_LOAD_REAL;
  // rows per workgroup
  const int yb = (reg || (LOAD && r) ? r->xr : Cfg<T>::LPW) * NWAVE;
  const int spw = OP == X_DENSITY ? (a.nslots + a.dens_parts - 1) / a.dens_parts
                  : b->tune.x_spw > 0 ? std::min(b->tune.x_spw, a.nslots)
                                      : x_slots_per_wg(g, a.nslots, yb);
  {
    TimedLaunch tl(ctx, name);
    if (reg)
      reg(ctx->stream, g, a, spw, in, out, dens, cplx_density);
    else if (LOAD && r)
      r->xload(ctx->stream, g, a, spw, in, OP == X_LOAD_REAL, scale);
    else
      launch_x<T, OP>(ctx->stream, g, a, spw, in, out, dens, scale, cplx_density);
  }
  return check_launch(ctx, name);
}

// row transforms of a plane (n rows of nlx lines) per wavefront
static long plane_work(const GridDev& g, const PlaneOps* p) {
  return (long)g.np0 * g.nlx * p->wgs / 8;
}

// plane forms of the call `use` for nslots slots of this basis and precision, or null (FP32 has
// none).
//
// A plane is one chain of dependent stages in one workgroup; the passes take three launches instead
// and spread the same work over more workgroups.  So the plane pays where its chain is short
// (transforms and density: four rounds, or 1300 row elements per SIMD; Hψ, which saves one more
// launch: 2100, or 2600 in spheres up to half the edge), or where there are enough planes for
// their work.
// Passes against plane, one slot, cubes (MI355X): Hψ 64^3 nlx 31 30 -> 25 us, 48^3 nlx 37 29 -> 29,
// 60^3 nlx 45 33 -> 38, 60^3 nlx 57 36 -> 46; backward 64^3 nlx 31 (4 rounds) 17 -> 14, 60^3 nlx 29
// (6) 15 -> 17, 48^3 nlx 45 (6) 16 -> 20; forward 54^3 nlx 27 (4) 19 -> 16, 60^3 nlx 45 (7) 20 -> 24;
// density 64^3 nlx 31 37 -> 34, 72^3 nlx 35 (7) 38 -> 40; with four slots Hψ of 60^3 nlx 45 51 -> 46.
// Stores of fat spheres on the longest edges pay at no count (60^3 nlx 57, 64 slots 232 -> 261).
enum PlaneUse { PLANE_VMUL, PLANE_STORE, PLANE_LOAD, PLANE_DENSITY };
static const PlaneOps* plane_ops(const Basis* b, int prec, int nslots, PlaneUse use) {
  const GridDev& g = b->g;
  if (prec != PREC_FP64 || g.np0 != g.np1 || !b->tune.zy_reg || !b->tune.x_reg) return nullptr;
  const EdgeOps* r = register_ops(g.np0, prec);
  if (!r || !r->plane.fits || !r->plane.fits(g)) return nullptr;
  const long work = 4 * plane_work(g, &r->plane);
  const bool alone = use == PLANE_VMUL ? work <= (g.nlx <= g.np0 / 2 + 1 ? 2600 : 2100)
                                       : work <= 1300 || r->plane.rounds(g) <= 4;
  if (!alone && work > 21L * g.np2 * nslots) return nullptr;
  if (use == PLANE_STORE && work > 2700 && 8 * g.nlx > 5 * g.np0) return nullptr;
  return &r->plane;
}

// slots per plane workgroup: as many as leave 2048 workgroups (72^3, 128 complex bands: 1, 2,
// 4, 8 slots 360, 330, 320, 346 us; 64^3, 128 real bands 108, 100, 98, 97)
static int plane_spw(const Basis* b, int nslots) {
  if (b->tune.x_spw > 0) return std::min(b->tune.x_spw, nslots);
  int spw = 1;
  while (spw < 16 && (long)b->g.np2 * ((nslots + 2 * spw - 1) / (2 * spw)) >= 2048) spw *= 2;
  return spw;
}

static int plane_pass(Ctx* ctx, Basis* b, const PipelineArgs& a, PlaneOps::Launch f, int spw,
                      const double* in, double* out, const double* dens, int cplx_density,
                      double scale, const char* name) {
  {
    TimedLaunch tl(ctx, name);
    f(ctx->stream, b->g, a, spw, in, out, dens, cplx_density, scale);
  }
  return check_launch(ctx, name);
}

int pipeline_vmul(Ctx* ctx, Basis* b, const PipelineArgs& a, const double* v, double* out,
                  long ldo, const double* kin, int store) {
  if (const PlaneOps* p = plane_ops(b, a.prec, a.nslots, PLANE_VMUL)) {
    if (int e = bwd_z(ctx, b, a)) return e;
    if (int e = plane_pass(ctx, b, a, p->vmul, plane_spw(b, a.nslots), v, nullptr, nullptr, 0, 1.0,
                           "plane_vmul"))
      return e;
    return fwd_z(ctx, b, a, out, ldo, kin, store);
  }
  if (int e = bwd_yz(ctx, b, a)) return e;
  const int e = a.prec == PREC_FP64
      ? xpass_t<double, X_VMUL>(ctx, b, a, v, nullptr, nullptr, 1.0, 0, "xpass_vmul")
      : xpass_t<float, X_VMUL>(ctx, b, a, v, nullptr, nullptr, 1.0, 0, "xpass_vmul");
  return e ? e : fwd_zy(ctx, b, a, out, ldo, kin, store);
}

int pipeline_store(Ctx* ctx, Basis* b, const PipelineArgs& a, double* f) {
  if (const PlaneOps* p = plane_ops(b, a.prec, a.nslots, PLANE_STORE); p && p->store) {
    if (int e = bwd_z(ctx, b, a)) return e;
    return plane_pass(ctx, b, a, p->store, plane_spw(b, a.nslots), nullptr, f, nullptr, 0, 1.0,
                      "plane_store");
  }
  if (int e = bwd_yz(ctx, b, a)) return e;
  return a.prec == PREC_FP64
             ? xpass_t<double, X_STORE>(ctx, b, a, nullptr, f, nullptr, 1.0, 0, "xpass_store")
             : xpass_t<float, X_STORE>(ctx, b, a, nullptr, f, nullptr, 1.0, 0, "xpass_store");
}

int pipeline_load(Ctx* ctx, Basis* b, const PipelineArgs& a, const double* f, int real_input,
                  double scale, double* out, long ldo) {
  int e;
  if (const PlaneOps* p = plane_ops(b, a.prec, a.nslots, PLANE_LOAD); p && p->load) {
    e = plane_pass(ctx, b, a, real_input ? p->load_real : p->load, plane_spw(b, a.nslots), f,
                   nullptr, nullptr, 0, scale, "plane_load");
    return e ? e : fwd_z(ctx, b, a, out, ldo, nullptr, 1);
  }
  if (a.prec == PREC_FP64)
    e = real_input ? xpass_t<double, X_LOAD_REAL>(ctx, b, a, f, nullptr, nullptr, scale, 0, "xpass_load")
                   : xpass_t<double, X_LOAD>(ctx, b, a, f, nullptr, nullptr, 1.0, 0, "xpass_load");
  else
    e = real_input ? xpass_t<float, X_LOAD_REAL>(ctx, b, a, f, nullptr, nullptr, scale, 0, "xpass_load")
                   : xpass_t<float, X_LOAD>(ctx, b, a, f, nullptr, nullptr, 1.0, 0, "xpass_load");
  return e ? e : fwd_zy(ctx, b, a, out, ldo, nullptr, 1);
}

// Slot ranges of the density x pass for chunks of nslots slots: each workgroup sums all slots
// of its rows, so the rows alone give np2 * np1 / rows-per-workgroup workgroups (216 at 72^3,
// 1260 at 140^3: 2.5 rounds of two per CU).  Ranges for about 4096 workgroups, with at most
// cap_bytes of partial grids; a range costs a partial grid written and read, so it takes at
// least 4 slots, and 16 where the rows alone fill the chip and it only evens out the last
// round.  One range against n, density with its z and y passes (MI355X, FP64 unless noted):
// 36 x 42 x 36, 32 slots 87 -> 52 us (8); 72 x 84 x 72, 128 slots 471 -> 345 (14); 108^3, 128
// slots 996 -> 930 (7); 140^3, 400 slots 6.45 -> 6.27 ms (4), 32 slots 561 -> 553 us (2; FP32 339
// -> 330), with 4 561 (339); 8 slots 167 us (FP32 112), with 2 181 (121).
static int density_parts(const Basis* b, int nslots, int prec, size_t cap_bytes) {
  const GridDev& g = b->g;
  const EdgeOps* r = b->tune.x_reg ? register_ops(g.np0, prec) : nullptr;
  const int yb = (r ? r->xr : prec == PREC_FP64 ? Cfg<double>::LPW : Cfg<float>::LPW) * NWAVE;
  const long rows = (long)g.np2 * ((g.np1 + yb - 1) / yb);
  const long N = (long)g.np0 * g.np1 * g.np2;
  long p = std::min<long>((4096 + rows - 1) / rows, 16);
  p = std::min<long>({p, nslots / (rows < 512 ? 4 : 16), (long)(cap_bytes / (8 * (size_t)N))});
  return (int)std::max<long>(p, 1);
}

// The same for the plane form, whose workgroups are few and long: of up to 16 ranges the number
// with the least time for its rounds of resident workgroups and its partial grids, the smaller
// one if equal.  A slot of a plane takes about 1.5 us and 14 ns per n * nlx / wavefronts (36^3
// 4 us, 72^3 10.5, 90^3 8, 100^3 10), a range 16 bytes a point at 4.5 TB/s, and the sum of the
// partial grids one more and a launch (4 us).  Density without z passes, passes -> plane: 24^3,
// 16 real bands 23 -> 15 us; 64^3, 128 real bands 98 -> 66; 72^3, 64 complex bands 136 -> 122;
// 88^3, 100 real bands 231 -> 196.  Against the fewest rounds alone, whole density: 100^3, 16
// slots 172 -> 133 us (2 ranges, not 16); 90^3, 8 slots 88 -> 82 (2, not 8).
static int plane_parts(const Basis* b, const PlaneOps* p, int nslots, size_t cap_bytes) {
  const GridDev& g = b->g;
  const size_t grid = 8 * (size_t)g.np0 * g.np1 * g.np2;
  const long most = std::min<long>({16, nslots, (long)(cap_bytes / grid)});
  const double slot = 1.5 + 0.014 * plane_work(g, p);
  long best = 1;
  double cost = 0.0;
  for (long k = 1; k <= most; ++k) {
    const double c = (g.np2 * k + 256L * p->wgs - 1) / (256L * p->wgs) * ((nslots + k - 1) / k) * slot +
                     (k > 1 ? 4.0 + (k + 1) * 2.0 * grid / 4.5e6 : 0.0);
    if (k == 1 || c < cost) {
      best = k;
      cost = c;
    }
  }
  return (int)best;
}

int pipeline_density_parts(const Basis* b, int nslots, int prec, size_t cap_bytes) {
  const PlaneOps* p = plane_ops(b, prec, nslots, PLANE_DENSITY);
  return p ? plane_parts(b, p, nslots, cap_bytes) : density_parts(b, nslots, prec, cap_bytes);
}

int pipeline_density(Ctx* ctx, Basis* b, const PipelineArgs& a, const double* dens, double* rho) {
  const int cd = a.mode == SLOT_COMPLEX ? 1 : 0;
  // slot ranges actually used (every one non-empty)
  const int spw = (a.nslots + a.dens_parts - 1) / a.dens_parts;
  const int parts = (a.nslots + spw - 1) / spw;
  double* out = parts > 1 ? a.dens_part : rho;
  int r;
  if (const PlaneOps* p = plane_ops(b, a.prec, a.nslots, PLANE_DENSITY)) {
    if (int e = bwd_z(ctx, b, a)) return e;
    r = plane_pass(ctx, b, a, p->density, spw, nullptr, out, dens, cd, 1.0, "plane_density");
  } else {
    if (int e = bwd_yz(ctx, b, a)) return e;
    r = a.prec == PREC_FP64
            ? xpass_t<double, X_DENSITY>(ctx, b, a, nullptr, out, dens, 1.0, cd, "xpass_density")
            : xpass_t<float, X_DENSITY>(ctx, b, a, nullptr, out, dens, 1.0, cd, "xpass_density");
  }
  if (r || parts == 1) return r;
  const long N = (long)b->g.np0 * b->g.np1 * b->g.np2;
  TimedLaunch tl(ctx, "density_sum");
  k_density_sum<4><<<(unsigned)((N + NTHR - 1) / NTHR), NTHR, 0, ctx->stream>>>(N, parts, 1.0, out,
                                                                               rho);
  return check_launch(ctx, "density_sum");
}

bool cross_edge(const Basis* b) {
  const EdgeOps* r = b->tune.x_reg ? register_ops(b->g.np0, PREC_FP64) : nullptr;
  return r && r->xcross;
}

int pipeline_cross(Ctx* ctx, Basis* b, const double* a, long lda, const double* const* bs,
                   long ldb, int nbands, int nb, const double* w, double scale, double* out) {
  const GridDev& g = b->g;
  const EdgeOps* r = register_ops(g.np0, PREC_FP64);
  const size_t c = sizeof(cplx<double>);
  const size_t t1 = c * g.ncol * g.np2, t2 = c * g.np2 * g.nlx * g.np1;
  const size_t per = t1 + (nb + 1) * t2;
  const long N = (long)g.np0 * g.np1 * g.np2;
  // slots in flight: up to 2 GiB of T1 and T2, in chunks of about equal size (the current of 128
  // bands at 72^3 in one, its gradient's 512 columns in two; with 1 GiB in unequal chunks both
  // calls took 1 % longer), and half as many as long as there is no memory for them
  const size_t room = std::min<size_t>(ctx->ws_cap, size_t(2) << 30);
  int S = (int)std::min<size_t>({std::max<size_t>(1, room / per), (size_t)nbands, 65535});
  const int chunks = (nbands + S - 1) / S;
  S = (nbands + chunks - 1) / chunks;
  char* ws = static_cast<char*>(ws_get(ctx, S * per));
  while (!ws && S > 1) ws = static_cast<char*>(ws_get(ctx, (S /= 2) * per));
  // partial grids per slot range: one range at least, more as for the density
  int parts = density_parts(b, S, PREC_FP64, kept_cap(ctx) / nb);
  std::optional<CallBuffer> buf;
  buf.emplace(ctx, sizeof(double) * parts * nb * N, &Ctx::inner);
  if (!buf->p && parts > 1) buf.emplace(ctx, sizeof(double) * (parts = 1) * nb * N, &Ctx::inner);
  double* part = static_cast<double*>(buf->p);
  if (!ws || !part) {
    ctx->last_error = "transform workspace allocation failed";
    return -2;
  }
  CrossFields f{};
  for (int d = 0; d <= nb; ++d)
    f.t2[d] = reinterpret_cast<cplx<double>*>(ws + S * (t1 + d * t2));
  for (int n0 = 0; n0 < nbands; n0 += S) {
    PipelineArgs p{};
    p.nslots = std::min(S, nbands - n0);
    p.nst = nbands;
    p.band0 = n0;
    p.mode = g.real ? SLOT_SINGLE_REAL : SLOT_COMPLEX;
    p.prec = PREC_FP64;
    p.t1 = ws;
    for (int d = 0; d <= nb; ++d) {
      p.psi = d ? bs[d - 1] : a;
      p.ld = d ? ldb : lda;
      p.t2 = const_cast<cplx<double>*>(f.t2[d]);
      if (int e = bwd_yz(ctx, b, p)) return e;
    }
    const int pn = std::min(parts, p.nslots);
    const int spw = (p.nslots + pn - 1) / pn, used = (p.nslots + spw - 1) / spw;
    {
      TimedLaunch tl(ctx, "xpass_cross");
      r->xcross(ctx->stream, g, f, p.nslots, spw, nb, w ? w + n0 : nullptr, part);
    }
    if (int e = check_launch(ctx, "xpass_cross")) return e;
    TimedLaunch tl(ctx, "density_sum");
    k_density_sum<4><<<(unsigned)((nb * N + NTHR - 1) / NTHR), NTHR, 0, ctx->stream>>>(
        nb * N, used, scale, part, out);
    if (int e = check_launch(ctx, "density_sum")) return e;
  }
  return 0;
}

}  // namespace qbh
