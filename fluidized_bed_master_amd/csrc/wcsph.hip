// Weakly compressible SPH step (SOPHIA_single, WCSPH_Calc.cuh:4-340) on
// gfx950: the stages that differ from the ISPH step.  KGC, porosity, the
// Shepard / delta-SPH prep, the wall Neumann interpolation and XSPH are the
// ISPH kernels (the WCSPH reference kernels are the same text).
// KERNEL_set_alpha (functions_ALE.cuh:2-20) makes every SPH particle
// Eulerian, so the neighbour list of step 0 stays valid.
#include "common.hpp"
#include "nbr.hpp"

namespace sophia {

namespace {

constexpr int kMoving = 9;  // MOVING (Parameters.cuh:12)

// KERNEL_clc_predictor (functions_TIME.cuh:77-292): half step of x
// (Lagrangian only), u, rho (continuity) and T with the previous step's
// ftotal, drho and dtemp; saves the start-of-step state.
template <typename R>
__global__ void k_wc_predictor(DevParams P, SphView<R> v) {
  int i = particle_index();
  if (i >= v.n) return;
  if (v.itype[i] == 3) return;
  const int t = v.ptype[i];
  const double dt = P.dt_sph;
  const double el = P.eulerian ? 0.0 : 1.0;
  const double bz = (v.btype[i] == 0);
  if (t != kMoving) {
    const double x0 = v.x[i], y0 = v.y[i], z0 = v.z[i];
    const double ux0 = (double)v.ux[i], uy0 = (double)v.uy[i], uz0 = (double)v.uz[i];
    if (t >= 0) {
      v.x[i] = x0 + ux0 * (dt * 0.5) * (t > 0) * el;
      v.y[i] = y0 + uy0 * (dt * 0.5) * (t > 0) * el;
      v.z[i] = z0 + uz0 * (dt * 0.5) * (t > 0) * el;
      v.ux[i] = (R)(ux0 + (double)v.fx[i] * bz * (dt * 0.5));
      v.uy[i] = (R)(uy0 + (double)v.fy[i] * bz * (dt * 0.5));
      v.uz[i] = (R)(uz0 + (double)v.fz[i] * bz * (dt * 0.5));
    }
    v.x0[i] = x0; v.y0[i] = y0; v.z0[i] = z0;
    v.ux0[i] = (R)ux0; v.uy0[i] = (R)uy0; v.uz0[i] = (R)uz0;
  }
  const double rho = v.rho[i];
  if (P.first_step) v.rho_ref[i] = rho;
  if (P.rho_type == 1 && t > 0) {
    if (P.first_step) v.vol0[i] = v.m[i] / rho;
    v.rho0[i] = rho;
    v.rho[i] = rho + (double)v.drho[i] * (dt * 0.5);
  } else {
    const double hv = v.h[i] / P.h_over_dx;
    if (P.first_step) v.vol0[i] = hv * hv * hv;
    v.rho0[i] = rho;
  }
  if (P.con_solve == 1) {
    v.temp0[i] = v.temp[i];
    v.temp[i] = (R)((double)v.temp[i] + (double)v.dtemp[i] * (dt * 0.5));
  }
}

// P3 reset after the predictor (WCSPH_Calc.cuh:59-60)
template <typename R>
__global__ void k_wc_reset(SphView<R> v) {
  int i = particle_index();
  if (i >= v.n) return;
  const int n = v.n;
  v.fx[i] = 0; v.fy[i] = 0; v.fz[i] = 0; v.fmag[i] = 0;
  v.fpx[i] = 0; v.fpy[i] = 0; v.fpz[i] = 0;
  v.dtemp[i] = 0; v.drho[i] = 0;
  for (int c = 0; c < 6; c++) v.cm[c * n + i] = 0;
}

// KERNEL_clc_volume_update3D (functions_MASS.cuh:148-222): Shepard-corrected
// volume over the +-3 cells (Eulerian particles at count 0 only), then
// KERNEL_clc_mass_update (functions_MASS.cuh:45-60): m = rho vol.
template <typename R>
__global__ void k_volume_update(DevParams P, SphView<R> v, CellView cv, int count) {
  int i = particle_index();
  if (i >= v.n) return;
  if (v.itype[i] > 2) return;
  if (P.eulerian && count > 0) return;
  if (v.ptype[i] >= 1000) return;
  const double h = v.h[i], A = knl_tmpA<double>(P.kernel_type, P.dim, h), Rs = P.kappa * h;
  const double xi = v.x[i], yi = v.y[i], zi = v.z[i];
  double tR = 0, filt = 0;
  for_cells_r(P, xi, yi, zi, cv, 3, [&](int j) {
    if (!(v.ptype[j] < 1000) || v.itype[j] == 4) return;
    const double r = dist_exact(xi - v.x[j], yi - v.y[j], zi - v.z[j]) + 1e-20;
    if (!(r < Rs)) return;
    const double w = knl_w<double>(P.kernel_type, A, h, r);
    tR += w;
    filt += v.m[j] / v.rho[j] / v.vol0[j] * w;
  });
  v.vol[i] = v.vol0[i] * 1.0 / tR * filt;
}

template <typename R>
__global__ void k_mass_update(DevParams P, SphView<R> v) {
  int i = particle_index();
  if (i >= v.n) return;
  if (v.ptype[i] > 1000 || v.itype[i] > 2) return;
  if (!P.eulerian) return;  // elix == eliy == 1
  v.m[i] = v.rho[i] * v.vol[i];
}

// KERNEL_clc_continuity_norm3D (functions_MASS.cuh:771-914) -> drho: the
// velocity divergence, the eps-advection term of Eulerian particles and
// the delta-SPH diffusion (Molteni, or Antuono with the density gradient).
// FP64 sums: drho integrates into rho, which the Tait EOS raises to gamma.
// Bound by its gathers and FP64 arithmetic: the mixed path reads one 64 B
// record per neighbour in place of thirteen field gathers, with V_j and the two
// ratios taken once per particle in place of seven FP64 divisions per pair.
__global__ void k_pack_cont(SphView<float> v) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= v.n) return;
  RecCont r;
  r.p = v.pos4[i];
  const double rho = v.rho[i];
  r.vol = v.m[i] / rho;
  r.rhopor = rho / v.por[i];
  r.ratio = rho / v.rho_ref[i];
  r.ux = v.ux[i]; r.uy = v.uy[i]; r.uz = v.uz[i];
  r.grx = v.grx[i]; r.gry = v.gry[i]; r.grz = v.grz[i];
  v.rc[i] = r;
}

// One neighbour of the continuity sums.
struct NbC {
  double dx, dy, dz, vol, rhopor, ratio;
  double ux, uy, uz, grx, gry, grz;
};
// f(neighbour, counted) over the list by G lanes, from the records (mixed) or
// the fields
template <int G, typename R, class F>
__device__ inline void for_nbrs_cont(const SphView<R>& v, int i, F&& f) {
  if constexpr (std::is_same<R, float>::value) {
    const int cnt = min(v.nbr_cnt[i], v.nbr_cap);
    if (cnt <= 0) return;
    const int n = v.n, last4 = (cnt - 1) & ~3, k0 = 4 * pair_sub<G>();
    const float4 pi4 = v.pos4[i];
    uint4 en4 = *(const uint4*)(v.nbr + nbr_slot(min(k0, last4), i, n));
    for (int k = k0; k < cnt; k += 4 * G) {
      const uint32_t en[4] = {en4.x, en4.y, en4.z, en4.w};
      RecCont r[4];
#pragma unroll
      for (int u = 0; u < 4; u++) r[u] = v.rc[(int)(en[u] & ~kNbrFlag)];
      en4 = *(const uint4*)(v.nbr + nbr_slot(min(k + 4 * G, last4), i, n));
#pragma unroll
      for (int u = 0; u < 4; u++) {
        const float3 d = rel_diff(pi4, r[u].p, v.pgrid, v.pmask);
        const NbC q{d.x, d.y, d.z, r[u].vol, r[u].rhopor, r[u].ratio, r[u].ux, r[u].uy, r[u].uz,
                    r[u].grx, r[u].gry, r[u].grz};
        f(q, k + u < cnt && !(en[u] & kNbrFlag));
      }
    }
  } else {
    for_nbrs4<true, G>(v, i, true, [&](const Nb<R>& q, bool on) {
      const NbC c{q.dx, q.dy, q.dz, q.m / q.rho, q.rho / q.por, q.rho / q.rref, q.ux, q.uy, q.uz, q.grx, q.gry, q.grz};
      f(c, on);
    });
  }
}

template <typename R, int G>
__global__ __launch_bounds__(kBlock) void k_continuity(DevParams P, SphView<R> v) {
  typedef double T;
  const int i = pair_particle<G>();
  if (i >= v.n) return;
  if (v.itype[i] > 2 || v.ptype[i] > 1000) return;
  if (P.open_boundary > 0 && v.btype[i] > 0) return;
  if (v.ptype[i] <= 0) return;
  const int n = v.n;
  const T h = v.h[i], ih = 1.0 / h, A = knl_tmpA<T>(P.kernel_type, P.dim, h);
  const T uxi = v.ux[i], uyi = v.uy[i], uzi = v.uz[i];
  const T rhoi = v.rho[i], pori = v.por[i];
  const T gxi = v.grx[i], gyi = v.gry[i], gzi = v.grz[i];
  const T rri = v.rho_ref[i], rpi = rhoi / pori, ratio_i = rhoi / rri;
  const T el = P.eulerian ? 0.0 : 1.0;
  const bool dsph = P.delsph > 0, anto = P.delsph == 2;
  const Kgc<T> K(P.kgc == 1, v.cm, n, i);
  T wx = uxi, wy = uyi, wz = uzi;  // u_i . (Cm g) = (Cm u_i) . g
  K.apply(wx, wy, wz);
  // sums over V_j: (u_i - u_j) . grad~W, (rho_i/eps_i - rho_j/eps_j) u_i . grad~W
  // and the delta-SPH term; the per-particle factors follow
  T td = 0, pd = 0, tR = 0;
  for_nbrs_cont<G>(v, i, [&](const NbC& q, bool use) {
    const T dx = q.dx, dy = q.dy, dz = q.dz;
    const T d2 = dx * dx + dy * dy + dz * dz, ir = pair_rinv(d2);
    const T vs = q.vol * (knl_dw_ih<T>(P.kernel_type, A, h, ih, d2 * ir) * ir);
    T cx = dx, cy = dy, cz = dz;
    K.apply(cx, cy, cz);
    td += use ? vs * ((uxi - q.ux) * cx + (uyi - q.uy) * cy + (uzi - q.uz) * cz) : 0.0;
    pd += use ? vs * (rpi - q.rhopor) * (wx * dx + wy * dy + wz * dz) : 0.0;
    if (dsph) {
      T phi = (gxi + q.grx) * -dx;
      phi += (gyi + q.gry) * -dy;
      phi += (gzi + q.grz) * -dz;
      phi = (-0.5 * phi) * (anto ? 1.0 : 0.0) + (q.ratio - ratio_i);
      tR += use ? vs * phi : 0.0;
    }
  });
  td = group_sum<G>(td);
  pd = group_sum<G>(pd);
  tR = group_sum<G>(tR);
  if (G > 1 && pair_sub<G>() != 0) return;
  const T ds = -2 * P.delta_sph * h * rri * P.soundspeed;
  v.drho[i] = (R)(rhoi * td + pori * pd * (1 - el) + (dsph ? ds * tR : 0.0));
}

// KERNEL_EOS (functions_PROP.cuh:7-28): p = B ((rho / rho_ref)^gamma - 1)
// with B = b c0^2 / gamma; the reference's b is 1.186 (an air density: it
// applies no rho0 factor), eos_b_factor sets it
template <typename R>
__global__ void k_eos(DevParams P, SphView<R> v) {
  int i = particle_index();
  if (i >= v.n) return;
  if (v.itype[i] > 2 || v.ptype[i] > 1000 || v.btype[i] != 0) return;
  const double B = P.soundspeed * P.soundspeed * (P.eos_b) / P.gamma;
  v.pres[i] = B * (pow(v.rho[i] / v.rho_ref[i], P.gamma) - 1.0);
}

// KERNEL_interaction3D (functions_INTERACTION.cuh:413-832), i_type 1:
// pressure, laminar and artificial viscosity, gravity, conduction and the
// Eulerian advection term (interface, repulsive, surface-tension,
// Boussinesq and concentration terms are off in this build).  Geometry and
// the pressure term in FP64, as in the ISPH force kernels.
// Neighbours from the packed records of the ISPH advection (NbP), with V_j in
// place of m_j and rho_j, and the KGC inverse on the sums where they are linear
// in the gradient.
template <typename R, int G>
__global__ __launch_bounds__(kBlock) void k_wc_interaction(DevParams P, SphView<R> v) {
  typedef R T;
  const int i = pair_particle<G>();
  if (i >= v.n) return;
  if (v.itype[i] != 1 || v.ptype[i] > 1000) return;
  const int pti = v.ptype[i];
  const int n = v.n;
  const double hd = v.h[i], ihd = 1.0 / hd;
  const T h = (T)hd;
  const double Ad = knl_tmpA<double>(P.kernel_type, P.dim, hd);
  const T uxi = v.ux[i], uyi = v.uy[i], uzi = v.uz[i], tempi = v.temp[i];
  const double pid = v.pres[i], rhoid = v.rho[i], porid = v.por[i];
  const T mi = (T)v.m[i], rhoi = (T)rhoid, pori = (T)porid;
  const bool tab = P.prop_table != 0;
  const T visi = tab ? v.visp[i] : (T)P.mu_fluid, visf = (T)P.mu_fluid;
  const T vis_const = (visi * visf) / (visi + visf);
  const T cv_i = 4 * pori / rhoi;
  const T eta = (T)(0.001 * hd);
  const T kci = tab ? v.condp[i] : (T)(pti > 1000 || pti < -1000 ? P.k_dem : P.k_fluid);
  const T cpi = (T)(pti > 1000 || pti < -1000 ? P.cp_dem : P.cp_fluid);
  const T el = P.eulerian ? (T)0 : (T)1;
  const bool euler = el < (T)1;
  const Kgc<double> K(P.kgc == 1, v.cm, n, i);
  double wx = (double)uxi, wy = (double)uyi, wz = (double)uzi;  // u_i . (Cm g) = (Cm u_i) . g
  K.apply(wx, wy, wz);
  T tx = 0, ty = 0, tz = 0, Rc = 0, ex = 0, ey = 0, ez = 0, et = 0;
  double px = 0, py = 0, pz = 0;  // sum_j V_j pp grad W
  for_nbrs4_pk<true, G>(v, i, true, [&](const NbP<R>& q, bool on) {
    const bool use = on && q.pt <= 1000;
    const double dxd = q.dx, dyd = q.dy, dzd = q.dz;
    const double d2 = dxd * dxd + dyd * dyd + dzd * dzd;
    const double ird = pair_rinv(d2), rd = d2 * ird;
    const double dwd = knl_dw_ih<double>(P.kernel_type, Ad, hd, ihd, rd);
    const double sd = dwd * ird;  // grad W = sd (x_i - x_j)
    if (P.fp_solve) {
      const double pp = P.pgrad_form ? q.pres - pid : pid + q.pres;
      const double c = use ? q.vol * pp * sd : 0.0;
      px += c * dxd;
      py += c * dyd;
      pz += c * dzd;
    }
    const T Vj = (T)q.vol, dw = (T)dwd;
    const T uxj = q.ux, uyj = q.uy, uzj = q.uz;
    if (P.fv_solve && pti > 0) {
      const T visj = tab ? v.visp[q.j] : visf;
      const T vm = tab ? (visi * visj) / (visi + visj) : vis_const;
      // x . (Cm grad W) / r^2
      const T Cv = (T)(sd * K.quad(dxd, dyd, dzd) * ird * ird) * (vm * cv_i * Vj);
      tx += use ? Cv * (uxi - uxj) : (T)0;
      ty += use ? Cv * (uyi - uyj) : (T)0;
      tz += use ? Cv * (uzi - uzj) : (T)0;
    }
    if (P.fva_solve) {
      const T dx = (T)dxd, dy = (T)dyd, dz = (T)dzd, r = (T)rd;
      T uij_xij = (uxi - uxj) * dx + (uyi - uyj) * dy + (uzi - uzj) * dz;
      T hij = (h + (T)q.h) * (T)0.5;
      T phi = hij * uij_xij;
      phi /= (r * r + (T)0.01 * hij * hij);
      T Pij = mi * phi * ((T)(-0.1 * P.soundspeed) + (T)0.02 * phi);
      Pij /= (rhoi + (T)v.rho[q.j]);  // not m / V: there may be no mass
      Pij *= (T)0.5;
      double gx = dxd, gy = dyd, gz = dzd;  // Cm x
      K.apply(gx, gy, gz);
      const T c = use && uij_xij < 0 ? -Pij : (T)0;
      tx += c * (T)(sd * gx);
      ty += c * (T)(sd * gy);
      tz += c * (T)(sd * gz);
    }
    if (P.con_solve) {
      const int ptj = q.pt;
      T kcj = tab ? v.condp[q.j] : (T)(ptj > 1000 || ptj < -1000 ? P.k_dem : P.k_fluid);
      T H = (T)4.0 * Vj * kcj * kci * (tempi - (T)q.temp) * dw;
      H /= cpi * ((T)rd + eta * eta) * rhoi * (kci + kcj);
      Rc += use ? H : (T)0;
    }
    if (euler) {
      const T ug = (T)(sd * (wx * dxd + wy * dyd + wz * dzd)) * Vj * (1 - el);
      ex += use ? ug * (uxj - uxi) : (T)0;
      ey += use ? ug * (uyj - uyi) : (T)0;
      ez += use ? ug * (uzj - uzi) : (T)0;
      if (P.con_solve) et += use ? ug * ((T)q.temp - tempi) : (T)0;
    }
  });
  tx = group_sum<G>(tx);
  ty = group_sum<G>(ty);
  tz = group_sum<G>(tz);
  Rc = group_sum<G>(Rc);
  ex = group_sum<G>(ex);
  ey = group_sum<G>(ey);
  ez = group_sum<G>(ez);
  et = group_sum<G>(et);
  px = group_sum<G>(px);
  py = group_sum<G>(py);
  pz = group_sum<G>(pz);
  if (G > 1 && pair_sub<G>() != 0) return;
  K.apply(px, py, pz);
  // pressure -eps_i / rho_i V_j pp, then the other terms; FP32 rounding of the
  // sum of both is below the tests' tolerance
  const double ci = -porid / rhoid;
  double fx = ci * px + (double)tx, fy = ci * py + (double)ty, fz = ci * pz + (double)tz;
  if (P.fg_solve) fz += -P.gravity;
  v.fx[i] = (R)(fx - (double)ex);
  v.fy[i] = (R)(fy - (double)ey);
  v.fz[i] = (R)(fz - (double)ez);
  v.pgx[i] = (R)-px;
  v.pgy[i] = (R)-py;
  v.pgz[i] = (R)-pz;
  v.fmag[i] = (R)sqrt(fx * fx + fy * fy + fz * fz);
  if (P.con_solve) v.dtemp[i] = Rc * (T)(pti != -3) - et;
}

// KERNEL_time_update_single (functions_TIME.cuh:676-877): full step from the
// start-of-step state with the half-step forces.  The temperature branch
// reads `k_con_solve==1 * p_type_i>0`, i.e. k_con_solve == (p_type_i > 0):
// with conduction off, walls take temp0 + dtemp dt and fluid keeps T.
template <typename R>
__global__ void k_wc_corrector(DevParams P, SphView<R> v) {
  int i = particle_index();
  if (i >= v.n) return;
  if (v.itype[i] == 3) return;
  const int t = v.ptype[i];
  const double dt = P.dt_sph;
  const double el = P.eulerian ? 0.0 : 1.0;
  const double bz = (v.btype[i] == 0);
  if (t == kMoving) {
    v.x[i] = v.x0[i] + (double)v.ux[i] * dt;
    v.y[i] = v.y0[i] + (double)v.uy[i] * dt;
    v.z[i] = v.z0[i] + (double)v.uz[i] * dt;
  } else {
    const double ux0 = (double)v.ux0[i], uy0 = (double)v.uy0[i], uz0 = (double)v.uz0[i];
    double ax = 0, ay = 0, az = 0;
    if (t > 0) {
      ax = (double)v.fx[i] * bz;
      ay = (double)v.fy[i] * bz;
      az = (double)v.fz[i] * bz;
    }
    double uxc = ux0 + ax * dt, uyc = uy0 + ay * dt, uzc = uz0 + az * dt;
    if (uxc * uxc + uyc * uyc + uzc * uzc >= P.u_limit * P.u_limit) {
      uxc = ux0;
      uyc = uy0;
      uzc = uz0;
    }
    if (!P.xsph_solve) {
      v.x[i] = v.x0[i] + uxc * dt * (t > 0) * el;
      v.y[i] = v.y0[i] + uyc * dt * (t > 0) * el;
      v.z[i] = v.z0[i] + uzc * dt * (t > 0) * el;
    }
    v.ux[i] = (R)uxc;
    v.uy[i] = (R)uyc;
    v.uz[i] = (R)uzc;
  }
  if (P.rho_type == 1 && t > 0) v.rho[i] = v.rho0[i] + (double)v.drho[i] * dt;
  if (P.con_solve == (t > 0 ? 1 : 0)) v.temp[i] = (R)((double)v.temp0[i] + (double)v.dtemp[i] * dt);
}

}  // namespace

#define WC_LAUNCH(kern, ...)                                        \
  do {                                                              \
    if (v.n > 0) {                                                  \
      kern<R><<<grid_xcd(v.n), kBlock, 0, s>>>(__VA_ARGS__);        \
      HIP_TRY(hipGetLastError());                                   \
    }                                                               \
    return 0;                                                       \
  } while (0)

template <typename R> int wc_predictor(hipStream_t s, const DevParams& P, const SphView<R>& v) { WC_LAUNCH(k_wc_predictor, P, v); }
template <typename R> int wc_reset_p3(hipStream_t s, const SphView<R>& v) { WC_LAUNCH(k_wc_reset, v); }
template <typename R>
int wc_volume_mass(hipStream_t s, const DevParams& P, const SphView<R>& v, const CellView& cv, int count) {
  if (v.n <= 0) return 0;
  k_volume_update<R><<<grid_xcd(v.n), kBlock, 0, s>>>(P, v, cv, count);
  k_mass_update<R><<<grid_xcd(v.n), kBlock, 0, s>>>(P, v);
  HIP_TRY(hipGetLastError());
  return 0;
}
template <typename R> int wc_continuity(hipStream_t s, const DevParams& P, const SphView<R>& v) {
  if (v.n <= 0) return 0;
  if constexpr (std::is_same<R, float>::value) k_pack_cont<<<grid_for(v.n), kBlock, 0, s>>>(v);
  return pair_launch(v.n, [&](auto g, int grid) { k_continuity<R, decltype(g)::value><<<grid, kBlock, 0, s>>>(P, v); });
}
template <typename R> int wc_eos(hipStream_t s, const DevParams& P, const SphView<R>& v) { WC_LAUNCH(k_eos, P, v); }
template <typename R> int wc_interaction(hipStream_t s, const DevParams& P, const SphView<R>& v) {
  TRY(sph_pack_velocity_records(s, v, false));
  return pair_launch(v.n,
                     [&](auto g, int grid) { k_wc_interaction<R, decltype(g)::value><<<grid, kBlock, 0, s>>>(P, v); });
}
template <typename R> int wc_corrector(hipStream_t s, const DevParams& P, const SphView<R>& v) { WC_LAUNCH(k_wc_corrector, P, v); }

#define WC_INST(R)                                                                                           \
  template int wc_predictor<R>(hipStream_t, const DevParams&, const SphView<R>&);                           \
  template int wc_reset_p3<R>(hipStream_t, const SphView<R>&);                                               \
  template int wc_volume_mass<R>(hipStream_t, const DevParams&, const SphView<R>&, const CellView&, int);   \
  template int wc_continuity<R>(hipStream_t, const DevParams&, const SphView<R>&);                          \
  template int wc_eos<R>(hipStream_t, const DevParams&, const SphView<R>&);                                 \
  template int wc_interaction<R>(hipStream_t, const DevParams&, const SphView<R>&);                         \
  template int wc_corrector<R>(hipStream_t, const DevParams&, const SphView<R>&);
WC_INST(float)
WC_INST(double)

}  // namespace sophia
