// phlx_diffusion.hip -- THERMAL_DIFFUSION_STS: RKL2 super-time-stepping of
// the radiative diffusion of internal energy, Strang-split around the hydro
// step (source/source.F90:6672-6688, thermal_diffusion_step :19949-20269).
//
// One diffusion step over dt/2 with s >= 3 stages (s from dt / dt_par on the
// host):
//   k_diff_stage<FIRST>          Me_0 = M(T), e_1
//   s-1 x k_diff_stage           ideal gas: T from e_jm1 on the fly, residual,
//                                RKL2 stage, and at the last one p and T
//   Helmholtz: s-1 x (k_diff_temp, k_diff_stage), then k_diff_final
// (3D: k_diff_march for k_diff_stage.)
// e_0 stays in g.eint until the last stage; e_j alternates between the two
// g.rkl buffers, over e_jm2, which only the thread of its own cell reads.
// The residual is sum_d (F(+) - F(-)) / dx_d of the face flux
// F = (4/3) a c K_int dT/dx, K = T^3 / (rho kappa), K_int the harmonic
// mean of the two cells; each face flux is recomputed by the two cells that
// share it (same operands, same bits) instead of a face array round trip.
//
// HBM bound: a middle stage of the ideal gas moves 56 bytes per cell (e_jm1, rho,
// kappa, e_jm2, e_0, Me_0 in, e_j out; the neighbours from LDS in 3D, from cache
// in 2D), where a T pass and an in-place update took 96 and two launches: a half
// step's stages at 128^3 took 50 us each, 37 in one pass, 28 marching (4.2 TB/s).
#include "phlx_internal.hpp"

namespace phlx {

constexpr double kRad = 7.565767381646406e-15;  // source/source.F90:614
constexpr double kClight = 2.99792458e10;        // source/source.F90:622

__device__ __forceinline__ long long kapix(const Grid &g, int i, int j, int k) {
  const int k0 = (g.sd == 3) ? 1 : 0;
  return ((long long)(k + k0) * (g.n2 + 2) + (j + 1)) * (g.n1 + 2) + (i + 1);
}

// Where a stage's temperatures come from: the g.tdiff array, p / (rho R / mu)
// of the hydro state (source/source.F90:13670-13674), or eint_to_temp of the
// ideal gas in closed form (:20271-20392).
enum { DT_ARRAY = 0, DT_P = 1, DT_E = 2 };
template <int TS>
__device__ __forceinline__ double diff_temp_of(const Grid &g, double v, double rho) {
  if (TS == DT_P) return Recip(rho * kRgas * g.inv_mu).div(v);
  if (TS == DT_E) return Recip(g.inv_mu * rho * kRgas).div(g.gmm1 * v);
  return v;
}
template <int SD, int TS>
__device__ __forceinline__ double diff_temp_at(const Grid &g, const double *e, long long c,
                                               double rho) {
  const double *v = TS == DT_P ? g.P + (long long)(SD + 1) * g.N : TS == DT_E ? e : g.tdiff;
  return diff_temp_of<TS>(g, v[c], rho);
}

// (T, rho) of the cell beside (i, j, k) along axis a at offset o = -1/+1;
// ghosts per bcs_thermal_diffusion (:20837-21068): periodic copies, else rho
// extrapolated linearly from the wall cells and T copied from the wall cell
// or set to 2 T_wall - T (FIX_TEMPERATURE_AT_*).
template <int SD, int TS>
__device__ __forceinline__ void diff_cell(const Grid &g, const double *e, int i, int j, int k,
                                          int a, int o, double &T, double &rho) {
  int x[3] = {i, j, k};
  const int n[3] = {g.n1, g.n2, g.n3};
  x[a] += o;
  const int side = o < 0 ? 0 : 1;
  const bool out = x[a] < 0 || x[a] >= n[a];
  const bool wall = out && g.bc[2 * a + side] != BC_PERIODIC;
  if (out) x[a] = (wall ? side : !side) ? n[a] - 1 : 0;
  const long long c = cix(g, x[0], x[1], x[2]);
  rho = g.P[c];
  T = diff_temp_at<SD, TS>(g, e, c, rho);
  if (wall) {
    x[a] = side ? n[a] - 2 : 1;
    rho = 2.0 * rho - g.P[cix(g, x[0], x[1], x[2])];
    const double tw = g.fix_t[2 * a + side];
    if (tw == tw) T = 2.0 * tw - T;
  }
}

// Radiative flux of the face between cells m and p from their T and K
// (:20488-20509).
__device__ __forceinline__ double diff_face(double tm, double km, double tp, double kp,
                                            double inv_dl) {
  const double krad = (4.0 / 3.0) * kRad * kClight;
  const double kint = Recip(km + kp).div(2.0 * (km * kp));
  const double grad = (tp - tm) * inv_dl;
  return krad * kint * grad;
}
__device__ __forceinline__ double diff_k(double T, double rho, double kappa) {
  return Recip(rho * kappa).div(T * T * T);
}

// residuals_thermal_diffusion (:20394-20835), Cartesian, x1 first: 2D (3D:
// k_diff_march's).
template <int TS>
__device__ __forceinline__ double diff_residual(const Grid &g, const double *e, int i, int j,
                                                double rc) {
  const double tc = diff_temp_at<2, TS>(g, e, cix(g, i, j, 0), rc);
  const double kc = diff_k(tc, rc, g.kappa[kapix(g, i, j, 0)]);
  double m = 0.0;
#pragma unroll
  for (int a = 0; a < 2; a++) {
    double tm, rm, tq, rq;
    diff_cell<2, TS>(g, e, i, j, 0, a, -1, tm, rm);
    diff_cell<2, TS>(g, e, i, j, 0, a, +1, tq, rq);
    const double km = diff_k(tm, rm, g.kappa[kapix(g, i - (a == 0), j - (a == 1), 0)]);
    const double kq = diff_k(tq, rq, g.kappa[kapix(g, i + (a == 0), j + (a == 1), 0)]);
    const double fm = diff_face(tm, km, tc, kc, g.inv_dx[a]);
    const double fp = diff_face(tc, kc, tq, kq, g.inv_dx[a]);
    const double d = (fp - fm) * g.inv_dx[a];
    m = (a == 0) ? d : m + d;
  }
  return m;
}

template <int SD>
__device__ __forceinline__ bool diff_coords(const Grid &g, int &i, int &j, int &k) {
  i = blockIdx.x * blockDim.x + threadIdx.x;
  j = blockIdx.y * blockDim.y + threadIdx.y;
  k = blockIdx.z;
  return i < g.n1 && j < g.n2;
}

// Stage 1 (FIRST): Me_0 = M, e_1 = e_0 + (dt/2 mu~_1) Me_0.
// Stage j: e_j = mu e_jm1 + nu e_jm2 + (1 - mu - nu) e_0 + (dt/2 mu~) M
//                + (dt/2 gamma~) Me_0 (:20129-20190).
// LAST (ideal gas): the step's end with it, eint = e_s, eint_to_temp and p.
template <int SD, bool FIRST, bool LAST>
__device__ __forceinline__ void diff_combine(const Grid &g, long long c, double rho, double m,
                                             double ejm1, const double *ejm2, double *ej, double mu,
                                             double nu, double c0, double hm, double hg) {
  if (FIRST) {
    g.me0[c] = m;
    ej[c] = ejm1 + hm * m;
  } else {
    const double e = mu * ejm1 + nu * ejm2[c] + c0 * g.eint[c] + hm * m + hg * g.me0[c];
    if (LAST) {
      const double T = diff_temp_of<DT_E>(g, e, rho);
      g.eint[c] = e;
      g.tdiff[c] = T;
      g.P[(long long)(SD + 1) * g.N + c] = kRgas * rho * T * g.inv_mu;
    } else {
      ej[c] = e;
    }
  }
}

// The 2D stage, flat.  The block order gives each XCD contiguous rows, and the
// rows beside them to its L2.
template <int TS, bool FIRST, bool LAST>
__global__ void __launch_bounds__(256)
    k_diff_stage(Grid g, unsigned nbx, const double *ejm1, const double *ejm2, double *ej,
                 double mu, double nu, double c0, double hm, double hg) {
  if (!g.sc->active) return;
  const unsigned w = xcd_contiguous(blockIdx.x, gridDim.x);
  const int i = (w % nbx) * blockDim.x + threadIdx.x;
  const int j = (w / nbx) * blockDim.y + threadIdx.y;
  if (i >= g.n1 || j >= g.n2) return;
  const long long c = cix(g, i, j, 0);
  const double rho = g.P[c];
  const double m = diff_residual<TS>(g, ejm1, i, j, rho);
  diff_combine<2, FIRST, LAST>(g, c, rho, m, ejm1[c], ejm2, ej, mu, nu, c0, hm, hg);
}

// The 3D stage, marching: a block takes kDiffX x kDiffY columns through kc
// planes.  T and K of a cell are computed once and reach the four in-plane
// neighbours through LDS and the next plane in registers, where the flat kernel
// computes them seven times per cell; the x3 flux is carried (the same operands,
// the same bits) and the next plane's loads are in flight.  About 2048 blocks of
// at most 16 planes.  All stages of a half step: 128^3 168 -> 138 us, 256^3 1507 ->
// 1138; 64 x 48 x 40, a plane per block, the same 33.
constexpr int kDiffX = 32, kDiffY = 8, kDiffW = kDiffX + 2, kDiffN = kDiffW * (kDiffY + 2);
template <int TS, bool FIRST, bool LAST>
__global__ void __launch_bounds__(256)
    k_diff_march(Grid g, unsigned nbx, unsigned nby, int kc, const double *ejm1,
                 const double *ejm2, double *ej, double mu, double nu, double c0, double hm,
                 double hg) {
  if (!g.sc->active) return;
  __shared__ double lt[2][kDiffN], lk[2][kDiffN];
  const unsigned w = xcd_contiguous(blockIdx.x, gridDim.x);
  const int i0 = (w % nbx) * kDiffX, j0 = (w / nbx % nby) * kDiffY, k0 = (w / nbx / nby) * kc;
  const int k1 = min(k0 + kc, g.n3);
  const int tid = threadIdx.x, a = tid % kDiffX, b = tid / kDiffX;
  const int i = i0 + a, j = j0 + b;
  const bool in = i < g.n1 && j < g.n2;
  // columns past the grid repeat its last one (their flux is not used)
  const int ic = min(i, g.n1 - 1), jc = min(j, g.n2 - 1);
  // halo cell of this thread: rows -1 and kDiffY, then columns -1 and kDiffX; one
  // per tile edge, where the grid has a cell or a ghost beside it
  const bool row = tid < 2 * kDiffX, halo = tid < 2 * kDiffX + 2 * kDiffY;
  const int u = tid - 2 * kDiffX;
  const int axis = row ? 1 : 0, o = (row ? tid < kDiffX : u < kDiffY) ? -1 : 1;
  const int ha = row ? a : (o < 0 ? -1 : min(kDiffX, g.n1 - i0));
  const int hb = row ? (o < 0 ? -1 : min(kDiffY, g.n2 - j0)) : u % kDiffY;
  const bool hin = halo && (row ? i0 + ha < g.n1 : j0 + hb < g.n2);
  const int hcell = (hb + 1) * kDiffW + ha + 1, mine = (b + 1) * kDiffW + a + 1;

  // what T and K of this column's cell at kk (-1 .. n3) need: the source of T,
  // rho and, beyond a wall, the second wall cell's rho
  struct Raw {
    double v, rho, rho1, kap;
  };
  auto ghost = [&](int kk) { return (kk < 0 || kk >= g.n3) && g.bc[kk < 0 ? 4 : 5] != BC_PERIODIC; };
  auto load = [&](int kk, Raw &r) {
    const bool wall = ghost(kk);
    const int kw = kk < 0 ? (wall ? 0 : g.n3 - 1) : kk >= g.n3 ? (wall ? g.n3 - 1 : 0) : kk;
    const long long c = cix(g, ic, jc, kw);
    r.rho = g.P[c];
    r.v = TS == DT_P ? g.P[4 * g.N + c] : TS == DT_E ? ejm1[c] : g.tdiff[c];
    r.kap = g.kappa[kapix(g, ic, jc, kk)];
    r.rho1 = wall ? g.P[cix(g, ic, jc, kk < 0 ? 1 : g.n3 - 2)] : 0.0;
  };
  auto value = [&](int kk, const Raw &r, double &T, double &K) {
    T = diff_temp_of<TS>(g, r.v, r.rho);
    double rho = r.rho;
    if (ghost(kk)) {
      rho = 2.0 * rho - r.rho1;
      const double tw = g.fix_t[kk < 0 ? 4 : 5];
      if (tw == tw) T = 2.0 * tw - T;
    }
    K = diff_k(T, rho, r.kap);
  };

  Raw r;
  double tm, km, tc, kcur;
  load(k0 - 1, r);
  value(k0 - 1, r, tm, km);
  load(k0, r);
  double rho = r.rho, e = r.v;  // of the current plane
  value(k0, r, tc, kcur);
  double fm3 = diff_face(tm, km, tc, kcur, g.inv_dx[2]);
  load(k0 + 1, r);
  for (int k = k0; k < k1; k++) {
    const int s = k & 1;
    if (in) {
      lt[s][mine] = tc;
      lk[s][mine] = kcur;
    }
    if (hin) {
      double T, rh;
      const int hi = i0 + ha - (axis == 0 ? o : 0), hj = j0 + hb - (axis == 1 ? o : 0);
      diff_cell<3, TS>(g, ejm1, hi, hj, k, axis, o, T, rh);
      lt[s][hcell] = T;
      lk[s][hcell] = diff_k(T, rh, g.kappa[kapix(g, i0 + ha, j0 + hb, k)]);
    }
    __syncthreads();
    const double rho_n = r.rho, e_n = r.v;
    double tn, kn;
    value(k + 1, r, tn, kn);
    if (k + 1 < k1) load(k + 2, r);
    const double fp3 = diff_face(tc, kcur, tn, kn, g.inv_dx[2]);
    if (in) {
      const double *t = lt[s] + mine, *q = lk[s] + mine;
      const double fm1 = diff_face(t[-1], q[-1], tc, kcur, g.inv_dx[0]);
      const double fp1 = diff_face(tc, kcur, t[1], q[1], g.inv_dx[0]);
      const double fm2 = diff_face(t[-kDiffW], q[-kDiffW], tc, kcur, g.inv_dx[1]);
      const double fp2 = diff_face(tc, kcur, t[kDiffW], q[kDiffW], g.inv_dx[1]);
      double m = (fp1 - fm1) * g.inv_dx[0];
      m = m + (fp2 - fm2) * g.inv_dx[1];
      m = m + (fp3 - fm3) * g.inv_dx[2];
      const long long c = cix(g, i, j, k);
      diff_combine<3, FIRST, LAST>(g, c, rho, m, TS == DT_E ? e : ejm1[c], ejm2, ej, mu, nu, c0,
                                   hm, hg);
    }
    fm3 = fp3;
    tc = tn;
    kcur = kn;
    rho = rho_n;
    e = e_n;
  }
}

// eint_to_temp (:20271-20392) with Helmholtz: helm_rhoe_given from the
// carried T.
__device__ __forceinline__ double diff_eint_to_temp(const Grid &g, long long c, double rho,
                                                    double eint, double abar, double zbar) {
  double T = g.tdiff[c], pr, sound;
  helm_rhoe_given(g.helm, rho, eint / rho, abar, zbar, T, pr, sound, false);
  return T;
}

template <int SD>
__global__ void __launch_bounds__(256) k_diff_temp(Grid g, const double *e) {
  if (!g.sc->active) return;
  int i, j, k;
  if (!diff_coords<SD>(g, i, j, k)) return;
  const long long c = cix(g, i, j, k);
  double ye, abar;
  cell_ye_abar(g, c, ye, abar);
  g.tdiff[c] = diff_eint_to_temp(g, c, g.P[c], e[c], abar, ye * abar);
}

// The step's end with Helmholtz (:20193-20267): eint_to_temp, then p and
// eint = rho e(T) from (rho, T), and the FASTEOS gammas.
template <int SD>
__global__ void __launch_bounds__(256) k_diff_final(Grid g, const double *es) {
  if (!g.sc->active) return;
  int i, j, k;
  if (!diff_coords<SD>(g, i, j, k)) return;
  constexpr int IP = SD + 1;
  const long long c = cix(g, i, j, k), N = g.N;
  const double rho = g.P[c];
  double ye, abar;
  cell_ye_abar(g, c, ye, abar);
  const double T = diff_eint_to_temp(g, c, rho, es[c], abar, ye * abar);
  g.tdiff[c] = T;
  double pr, e, sound, cv;
  helm_full(g.helm, rho, T, abar, abar * ye, pr, e, sound, cv);
  helm_pin(pr);
  helm_pin(sound);
  const double eint = rho * e;
  g.P[IP * N + c] = pr;
  g.eint[c] = eint;
  if (g.fasteos) {
    g.gam[c] = pr / eint + 1.0;
    g.gam[N + c] = sound * sound * rho / pr;
  }
}

// compute_parabolic_dt (:19804-19947) without USE_TIMMES_KAPPA: per-block
// partial maxima of 2 D sum 1/dx^2, D = c / (3 kappa rho).
template <int SD>
__global__ void __launch_bounds__(256) k_parabolic(Grid g, double inv_dl2) {
  __shared__ double red[4];
  int i, j, k;
  double v = 0.0;
  if (diff_coords<SD>(g, i, j, k)) {
    const double rho = g.P[cix(g, i, j, k)];
    const double drad = (1.0 / 3.0) * kClight / (g.kappa[kapix(g, i, j, k)] * rho);
    v = 2.0 * drad * inv_dl2;
  }
  // block maximum (max is exact, so the order does not matter)
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v = fmax(v, __shfl_xor(v, o));
  const int tid = threadIdx.y * blockDim.x + threadIdx.x;
  if ((tid & 63) == 0) red[tid >> 6] = v;
  __syncthreads();
  if (threadIdx.x == 0 && threadIdx.y == 0) {
    const double m = fmax(fmax(red[0], red[1]), fmax(red[2], red[3]));
    g.red[blockIdx.x + (long long)gridDim.x * (blockIdx.y + (long long)gridDim.y * blockIdx.z)] = m;
  }
}

static dim3 diff_grid(const Grid &g) {
  const dim3 b = cell_block(g);
  return dim3((g.n1 + b.x - 1) / b.x, (g.n2 + b.y - 1) / b.y, g.n3);
}

template <int SD, int TS, bool FIRST, bool LAST>
static void diff_stage(const Grid &g, const double *ejm1, const double *ejm2, double *ej, double mu,
                       double nu, double c0, double hm, double hg, hipStream_t st) {
  if constexpr (SD == 3) {
    const int nbx = (g.n1 + kDiffX - 1) / kDiffX, nby = (g.n2 + kDiffY - 1) / kDiffY;
    const long long planes = (long long)nbx * nby * g.n3;
    const int kc = (int)std::min(std::max(planes / 2048, 1LL), 16LL);
    const int nbz = (g.n3 + kc - 1) / kc;
    k_diff_march<TS, FIRST, LAST><<<nbx * nby * nbz, 256, 0, st>>>(g, nbx, nby, kc, ejm1, ejm2, ej,
                                                                  mu, nu, c0, hm, hg);
  } else {
    const dim3 b = cell_block(g), n = diff_grid(g);
    k_diff_stage<TS, FIRST, LAST>
        <<<n.x * n.y, b, 0, st>>>(g, n.x, ejm1, ejm2, ej, mu, nu, c0, hm, hg);
  }
}
template <int SD>
static void diff_stage(const Grid &g, int form, const double *ejm1, const double *ejm2, double *ej,
                       double mu, double nu, double c0, double hm, double hg, hipStream_t st) {
  const auto go = [&](auto f) { f(g, ejm1, ejm2, ej, mu, nu, c0, hm, hg, st); };
  switch (form) {
    case DIFF_FIRST_ARRAY: return go(diff_stage<SD, DT_ARRAY, true, false>);
    case DIFF_FIRST_P: return go(diff_stage<SD, DT_P, true, false>);
    case DIFF_ARRAY: return go(diff_stage<SD, DT_ARRAY, false, false>);
    case DIFF_E: return go(diff_stage<SD, DT_E, false, false>);
    default: return go(diff_stage<SD, DT_E, false, true>);
  }
}

void launch_diff_stage(const Grid &g, int form, const double *ejm1, const double *ejm2, double *ej,
                       double mu, double nu, double c0, double hm, double hg, hipStream_t st) {
  if (g.sd == 3) diff_stage<3>(g, form, ejm1, ejm2, ej, mu, nu, c0, hm, hg, st);
  else diff_stage<2>(g, form, ejm1, ejm2, ej, mu, nu, c0, hm, hg, st);
}

void launch_diff_temp(const Grid &g, const double *e, hipStream_t st) {
  const dim3 blk = cell_block(g);
  if (g.sd == 3) k_diff_temp<3><<<diff_grid(g), blk, 0, st>>>(g, e);
  else k_diff_temp<2><<<diff_grid(g), blk, 0, st>>>(g, e);
}

void launch_diff_final(const Grid &g, const double *es, hipStream_t st) {
  const dim3 blk = cell_block(g);
  if (g.sd == 3) k_diff_final<3><<<diff_grid(g), blk, 0, st>>>(g, es);
  else k_diff_final<2><<<diff_grid(g), blk, 0, st>>>(g, es);
}

void launch_parabolic(const Grid &g, double inv_dl2, hipStream_t st) {
  const dim3 blk = cell_block(g);
  if (g.sd == 3) k_parabolic<3><<<diff_grid(g), blk, 0, st>>>(g, inv_dl2);
  else k_parabolic<2><<<diff_grid(g), blk, 0, st>>>(g, inv_dl2);
}

}  // namespace phlx
