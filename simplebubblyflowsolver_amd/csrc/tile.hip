// k_tile: the stage kernel (march.hip) for grids too small to fill the device.
//
// The marching kernel's wavefront walks its band row by row, 10 rows at least
// for a band of 4 (6 of ring fill), and a row with interface cells is a chain of
// about 4 us (square roots, divisions, tanh and log in FP64): a floor of 40 us
// per stage however small the grid.  Here a workgroup takes a strip of kStrip
// columns and H output rows, and each of its H + 5 wavefronts one row: what the
// marching kernel keeps in register rings goes through LDS, between barriers:
//
//   row s of a wavefront            read from the rows around it
//   0  velocities of the previous stage's projection (folded variant)
//   1  corner gradients at the bottom of row s
//   2  normals, curvature, THINC and mass flux in x      gradients s+1, u s-1, s+1
//   3  THINC and mass flux through the bottom face,
//      stresses                                          normals s-1
//   4  new vof and density, momentum fluxes              face fluxes s-1, s+1, txy s+1
//   5  predicted velocity, the rows' outputs             density, curvature, tyy s-1
//   6  Poisson right-hand side                           face terms s+1
//
// Rows jb-2 .. je+3 are needed for output rows jb .. je; a wavefront ends before
// the first phase that needs nothing of its row (a barrier waits for the ones
// that remain: k_tile at 512 x 512 28.5 -> 27.6 us).  Columns, lanes, masks
// and every expression are the marching kernel's, so the fields are the same bit
// for bit.  The latency of the seven phases bounds it (121 VGPRs in FP64, 98 in
// FP32: 4 and 5 wavefronts per SIMD, but one workgroup of H = 11 fills a CU's LDS
// by half), so the marching kernel keeps the grids where the device is full.
// The three stages together, us with about 15 of the timing events:
//                      64 x 128  128 x 256  256 x 512  512 x 1024  1024 x 1024
//   FP64   march            139        131        140         173          241
//          H = 3             44         44         74         183          338
//          H = 11            71         70         63         153          260
//   mixed  march             86         86        101         128          179
//          H = 3             31         35         64         158          284
//          H = 11            40         41         45         129          218
#include "march_dev.hpp"

namespace sbfs {

// LDS rows of 64 lanes, one of each per wavefront; a slot is reused once every
// wavefront has passed the barrier after its last read
enum {
  S_GX, S_GY,          // gradients (1, read in 2)
  S_NX, S_NY, S_NZ,    // normals (2, read in 3)
  S_K, S_MFX,          // curvature, x mass flux (2, read in 5 and 4)
  S_UX, S_UY,          // corrected velocities (0, read in 2)
  S_COUNT,
  S_FY = S_GX, S_MFY = S_GY,    // y fluxes (3, read in 4)
  S_TXY = S_UX, S_CTYY = S_UY,  // stresses (3, read in 4)
  S_DN = S_NX,                  // new density (4, read in 5)
  S_CU = S_GX, S_CG = S_GY,     // face terms of the right-hand side (5, read in 6)
};

template <typename R, bool CORR, int H>
__device__ __forceinline__ void tile_body(const MarchArgs& a, int bx, int by) {
  using A = Arith<R>;
  using V3 = V3R<R>;
  constexpr int kTileRows = H, kTileWaves = H + 5;
  __shared__ double st[T_N][64];
  __shared__ double slots[S_COUNT][kTileWaves][64];
  const int lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int nx = a.nx, ny = a.ny;
  const int i0 = 1 + bx * kStrip;
  const int cl = i0 - 3;  // column held by lane 0
  const int c = cl + lane;
  const int jb = 1 + by * kTileRows;
  const int je = min(ny, jb + kTileRows - 1);
  const int s = jb - 2 + w;  // this wavefront's row
  const bool c_vof = c >= 0 && c <= nx + 1;   // cells incl. wall ghosts
  const bool c_in = c >= 1 && c <= nx;        // interior cells
  const bool c_fx = c >= 1 && c <= nx + 1;    // x faces incl. walls
  const bool c_out = c >= i0 && c < i0 + kStrip && c <= nx;
  const bool outrow = s >= jb && s <= je;
  const int ll = lane > 0 ? lane - 1 : 0, lr = lane < 63 ? lane + 1 : 63;
  auto TB = [&](int t) { return st[t][lane]; };
  auto TR = [&](int t) { return st[t][lr]; };
  auto SB = [&](int t) { return R(st[t][lane]); };
  auto SL = [&](int t) { return R(st[t][ll]); };
  auto SR = [&](int t) { return R(st[t][lr]); };
  // this row's slot, and a neighbouring row's (the outermost rows read their
  // own: what they would form from it is not used)
  const int wm = max(w - 1, 0), wp = min(w + 1, kTileWaves - 1);
  auto put_r = [&](int k, R v) { ((R*)slots[k][w])[lane] = v; };
  auto get_r = [&](int k, int row) { return ((const R*)slots[k][row])[lane]; };
  auto put_d = [&](int k, double v) { slots[k][w][lane] = v; };
  auto get_d = [&](int k, int row) { return slots[k][row][lane]; };
  constexpr bool kExactQ = std::is_same<R, double>::value;
  auto per_h = [&](double x) { return kExactQ ? x / TB(T_HXXF) : x * TB(T_RHF); };
  const double hy = a.hy, rhy = a.cf.rhy;
  auto per_hy = [&](double x) { return kExactQ ? x / hy : x * rhy; };
  const R hyr = R(hy), rhyr = R(rhy);
  auto DEN = [&](double v) { return mix_clamp(a.denr, a.dlo, a.dhi, v); };
  auto VISUX = [&](int col, R vl, R vr) {
    R v;
    if (col == 1) v = vl;
    else if (col == nx + 1) v = vr;
    else v = R(0.5) * vl + R(0.5) * vr;
    return mixr<R>(a.visr, a.vlo, a.vhi, v);
  };
  auto VISUY = [&](R vb, R vt) { return mixr<R>(a.visr, a.vlo, a.vhi, R(0.5) * vb + R(0.5) * vt); };
  auto rw = [&](auto* f, ptrdiff_t e) {
    return RowRef<std::remove_reference_t<decltype(*f)>>{f, (unsigned)(e * (ptrdiff_t)sizeof(*f))};
  };
  const ptrdiff_t wc = nx + 2, wf = nx + 1;
  auto vof_row = [&](auto* f, int j) { return rw(f, (ptrdiff_t)(j + 1) * wc + cl); };         // L::vof
  auto cc_row = [&](auto* f, int j) { return rw(f, (ptrdiff_t)j * wc + cl); };                // L::cc
  auto xf_row = [&](auto* f, int j) { return rw(f, (ptrdiff_t)j * wf + cl - 1); };            // L::xf
  auto ci_row = [&](auto* f, int j) { return rw(f, (ptrdiff_t)(j - 1) * nx + cl - 1); };      // L::ci
  auto fx_row = [&](auto* f, int j) { return rw(f, (ptrdiff_t)(j - 1) * (nx - 1) + cl - 2); };  // L::fx
  const unsigned loff = (unsigned)lane * 8u;
  auto AT = [&](auto r) -> auto& { return lane_at(r, loff); };
  auto ld_vof = [&](int jw) { return c_vof ? AT(vof_row(a.vof, jw)) : 0.; };
  auto ld_ux = [&](int jw) { return c_fx ? AT(xf_row(a.ux, jw)) : 0.; };
  auto ld_cc = [&](const double* f, int jw) { return c_vof ? AT(cc_row(f, jw)) : 0.; };
  auto msrc = [&](auto* f, auto rowf, int j) -> auto& {
    if constexpr (std::is_same<R, float>::value) {
      using F = std::conditional_t<std::is_const<std::remove_pointer_t<decltype(f)>>::value, const float, float>;
      return lane_at(rowf((F*)f, j), loff >> 1);
    } else {
      return AT(rowf(f, j));
    }
  };

  // -- every input, issued together ------------------------------------------
  const int w0 = wrap_r(s, ny), wm1 = wrap_r(s - 1, ny), wp1 = wrap_r(s + 1, ny);
  const double vm = ld_vof(wm1), v0 = ld_vof(w0), vp = ld_vof(wp1);
  double ux0 = ld_ux(w0), uy0 = ld_cc(a.uy, w0);
  double uxm = 0., uxp = 0., uym = 0., uyp = 0.;
  if (!CORR) {
    uxm = ld_ux(wm1);
    uxp = ld_ux(wp1);
    uym = ld_cc(a.uy, wm1);
    uyp = ld_cc(a.uy, wp1);
  }
  double p0 = ld_cc(a.p, w0), pm = ld_cc(a.p, wm1);
  const double ps0 = ld_cc(a.psi0, w0), psm = ld_cc(a.psi0, wm1);
  double po0 = 0., pom = 0.;
  if (CORR) {
    po0 = ld_cc(a.psi_old, w0);
    pom = ld_cc(a.psi_old, wm1);
  }
  const bool has_b = a.stage != 0;
  double sbv = 0., sby = 0., sbx = 0.;
  if (has_b && c_in) {
    sbv = AT(ci_row(a.srcb_vof, w0));
    if (s >= jb) sby = msrc(a.srcb_uy, ci_row, w0);
    if (outrow && c >= 2) sbx = msrc(a.srcb_ux, fx_row, w0);
  }
  float kl = 0.f;
  if (a.kappa && *a.kappa_n != 0u && c_in) kl = lane_at(ci_row(a.kappa, w0), loff >> 1);
  {
    const double* tabs[T_N] = {a.cf.rhf, a.cf.rhc, a.cf.rjf, a.cf.rjc, a.cf.qf, a.cf.qc, a.cf.eqf,
                               a.cf.ecy, a.cf.cyc, a.cf.cyf, a.cf.dfx, a.cf.dcx, a.hxxf1, a.hxxc1};
    const int cc = c < 0 ? 0 : (c > nx + 1 ? nx + 1 : c);
#pragma unroll
    for (int t = 0; t < T_N; t++)
      if (t % kTileWaves == w) st[t][lane] = tabs[t][cc];
  }
  const double dt = uni(*a.dt);
  const double dtca = dt * a.ca, dtcb = dt * a.cb, dtcg = dt * a.cg;
  const double dt_old = a.g_old * dt, dt_new = a.g_new * dt;
  const double c0 = 1. / a.norm / dt_new * a.refden;
  const double c1 = 1. / a.norm * -1. / dt_new * dt_old;
  const R denr1 = R(a.denr) - R(1);
  const R refdeninv = R(a.refdeninv), tension = R(a.tension), grav = R(a.grav);
  __syncthreads();

  // -- 0: the previous stage's projection (correct_velocity/ux.c, uy.c,
  // update_pressure.c), k_post's expressions
  if (CORR) {
    const double pdtn = a.pg_new * dt, pdto = a.pg_old * dt;
    const double pcoef = -1. / pdtn * pdto;
    const double pdtc = pdtn * pcoef, irefden = 1. / a.refden;
    const double pcx0 = pdtn / a.refden, pcy = pdtn / a.refden / hy;
    const double da = DEN(vm), db = DEN(v0);
    const double dbl = from_left(db);
    const double psl = from_left(ps0), pol = from_left(po0);
    {
      double u = 0.;
      if (c >= 2 && c <= nx) {
        u = ux0;
        u -= per_h(pcx0) * (-psl + ps0);
        const double d = 0.5 * dbl + 0.5 * db;
        u += per_h(pdtc * (1. / d - irefden)) * (-pol + po0);
      }
      ux0 = u;
    }
    {
      double u = 0.;
      if (c == 0) u = kUyXm;
      else if (c == nx + 1) u = kUyXp;
      else if (c_in) {
        u = uy0;
        u -= pcy * (-psm + ps0);
        const double d = 0.5 * da + 0.5 * db;
        u += per_hy(pdtc * (1. / d - irefden)) * (-pom + po0);
      }
      uy0 = u;
    }
    if (c_in) {
      p0 = (a.p_twice ? p0 + po0 : p0) + ps0;
      pm = (a.p_twice ? pm + pom : pm) + psm;
    }
    put_d(S_UX, ux0);
    put_d(S_UY, uy0);
  }
  // -- 1: corner gradients at the bottom of row s (curvature_tensor.c:16-49) ---
  R g0x = 0, g0y = 0;
  {
    const double mm = from_left(vm), pm_ = vm, mp = from_left(v0), pp = v0;
    if (c_fx && !(mm == pm_ && mm == mp && mm == pp)) {
      const R rmm = R(mm), rpm = R(pm_), rmp = R(mp), rpp = R(pp);
      g0x = SB(T_RHF) * (-rmm + rpm - rmp + rpp);
      g0y = rhyr * (-rmm - rpm + rmp + rpp);
      const R norm = A::sqr(g0x * g0x + g0y * g0y);
      const R ninv = A::div(R(1), fmax(norm, A::eps()));
      g0x = g0x * ninv;
      g0y = g0y * ninv;
    }
  }
  put_r(S_GX, g0x);
  put_r(S_GY, g0y);
  __syncthreads();
  if (s > je + 2) return;
  if (CORR) {
    uxm = get_d(S_UX, wm);
    uxp = get_d(S_UX, wp);
    uym = get_d(S_UY, wm);
    uyp = get_d(S_UY, wp);
  }
  const R rux0 = R(ux0), ruxm = R(uxm), ruxp1 = R(uxp);
  const R ruy0 = R(uy0), ruym = R(uym), ruyp1 = R(uyp);
  const R rvm1 = R(vm), rv0 = R(v0), rvp1 = R(vp);
  // -- 2: normals and curvature of row s, fluxes through its x faces ----------
  R n0x = 0, n0y = 0, n0z = 0, k0 = 0, fx0 = 0, mfx0 = 0;
  {
    const R g1x = get_r(S_GX, wp), g1y = get_r(S_GY, wp);
    const R g0xr = A::right(g0x), g0yr = A::right(g0y), g1xr = A::right(g1x), g1yr = A::right(g1y);
    if (c_in && in_band(v0)) {
      R nxv = g0x + g0xr + g1x + g1xr;
      R nyv = g0y + g0yr + g1y + g1yr;
      nxv = A::div(nxv, SB(T_HXXC));
      nyv = A::div(nyv, hyr);
      const R norm = A::sqr(nxv * nxv + nyv * nyv);
      const R ninv = A::div(R(1), fmax(norm, A::eps()));
      n0x = nxv * ninv;
      n0y = nyv * ninv;
      n0z = A::intercept(v0);
    }
    if (c_in) {
      const R nxm = R(0.5) * g0x + R(0.5) * g1x;
      const R nxp = R(0.5) * g0xr + R(0.5) * g1xr;
      const R nym = R(0.5) * g0y + R(0.5) * g0yr;
      const R nyp = R(0.5) * g1y + R(0.5) * g1yr;
      const R div = SB(T_RJC) * (-SB(T_QF) * nxm + SR(T_QF) * nxp - SB(T_CYC) * nym + SB(T_CYC) * nyp);
      k0 = R(-1) * div;
      if (kl == kl && kl != 0.f) k0 = R(kl);
    }
    const double vl = from_left(v0);
    const R nlx = A::left(n0x), nly = A::left(n0y), nlz = A::left(n0z);
    if (c_fx) {
      const R vel = rux0;
      if (c != 1 && c != nx + 1) {
        const bool up = vel < R(0);
        const double v = up ? v0 : vl;
        const V3 n = up ? V3{n0x, n0y, n0z} : V3{nlx, nly, nlz};
        fx0 = thinc_flux<R, true>(vel, v, in_band(v) ? n : V3{0, 0, 0});
      }
      mfx0 = vel + denr1 * fx0;
    }
  }
  put_r(S_NX, n0x);
  put_r(S_NY, n0y);
  put_r(S_NZ, n0z);
  put_r(S_K, k0);
  put_r(S_MFX, mfx0);
  __syncthreads();
  if (s < jb - 1) return;
  // -- 3: fluxes through the bottom face of row s, stresses -------------------
  R fy0 = 0, mfy0 = 0;
  {
    const V3 nm{get_r(S_NX, wm), get_r(S_NY, wm), get_r(S_NZ, wm)};
    if (c_vof) {
      const R vel = ruy0;
      if (c != 0 && c != nx + 1) {
        const bool up = vel < R(0);
        const double v = up ? v0 : vm;
        const V3 n = up ? V3{n0x, n0y, n0z} : nm;
        fy0 = thinc_flux<R, false>(vel, v, in_band(v) ? n : V3{0, 0, 0});
      }
      mfy0 = vel + denr1 * fy0;
    }
  }
  put_r(S_FY, fy0);
  put_r(S_MFY, mfy0);
  const R rux0r = A::right(rux0), ruy0l = A::left(ruy0);
  R txx0 = 0, txy0 = 0, tyy0 = 0;
  {
    const R visx0 = VISUX(c, A::left(rv0), rv0), visxm = VISUX(c, A::left(rvm1), rvm1);
    const R visy0 = VISUY(rvm1, rv0), visy1 = VISUY(rv0, rvp1);
    const R visx0r = A::right(visx0), visy0l = A::left(visy0);
    if (c_in) {
      const R vx = R(0.5) * visx0 + R(0.5) * visx0r;
      const R l = SB(T_RHC) * (-rux0 + rux0r);
      txx0 = vx * l + vx * l;
    }
    if (c_in) {
      const R vy = R(0.5) * visy0 + R(0.5) * visy1;
      const R l = rhyr * (-ruy0 + ruyp1);
      tyy0 = vy * l + vy * l;
    }
    if (c_fx) {
      const R vx = R(0.5) * visxm + R(0.5) * visx0;
      const R vy = R(0.5) * visy0l + R(0.5) * visy0;
      const R lxy = rhyr * (-ruxm + rux0);
      const R lyx = SB(T_RHF) * (-ruy0l + ruy0);
      txy0 = vx * lxy + vy * lyx;
    }
  }
  const R cyc_tyy0 = SB(T_CYC) * tyy0;
  put_r(S_TXY, txy0);
  put_r(S_CTYY, cyc_tyy0);
  __syncthreads();
  if (s > je + 1) return;
  // -- 4: new vof (update/main.c:54-120) and density, momentum fluxes ----------
  const R fyp1 = get_r(S_FY, wp), mfyp1 = get_r(S_MFY, wp), txy1 = get_r(S_TXY, wp);
  const R mfym1 = get_r(S_MFY, wm), mfxm1 = get_r(S_MFX, wm), cyc_tyym1 = get_r(S_CTYY, wm);
  double src = 0., vn0 = 0.;
  {
    const double fx0d = double(fx0);
    const double fx0r = A::right(fx0);
    if (c_in) {
      src = TB(T_RJC) * (+TB(T_QF) * fx0d - TR(T_QF) * fx0r + TB(T_CYC) * double(fy0) - TB(T_CYC) * double(fyp1));
      vn0 = v0;
      vn0 += dtca * src;
      if (has_b) vn0 += dtcb * sbv;
    }
  }
  const double dn0 = DEN(vn0);
  put_d(S_DN, dn0);
  const R mfx0r = A::right(mfx0), mfyp1l = A::left(mfyp1), mfy0l = A::left(mfy0);
  const R qx = (SB(T_EQF) * mfx0 + SR(T_EQF) * mfx0r) * (R(0.5) * rux0 + R(0.5) * rux0r);
  const R qm = (SB(T_EQF) * mfxm1 + SB(T_EQF) * mfx0) * (R(0.5) * ruy0l + R(0.5) * ruy0);
  const R qxl = A::left(qx), qmr = A::right(qm);
  const R qt = SB(T_QC) * txx0;
  const R qtl = A::left(qt);
  const R qf_txy0 = SB(T_QF) * txy0;
  const R qf_txy0r = A::right(qf_txy0);
  const R qy_ux = (SL(T_ECY) * mfy0l + SB(T_ECY) * mfy0) * (R(0.5) * ruxm + R(0.5) * rux0);
  const R qy_ux_new = (SL(T_ECY) * mfyp1l + SB(T_ECY) * mfyp1) * (R(0.5) * rux0 + R(0.5) * ruxp1);
  const R qy_uy = (SB(T_ECY) * mfym1 + SB(T_ECY) * mfy0) * (R(0.5) * ruym + R(0.5) * ruy0);
  const R qy_uy_new = (SB(T_ECY) * mfy0 + SB(T_ECY) * mfyp1) * (R(0.5) * ruy0 + R(0.5) * ruyp1);
  const R cyf_txy0 = SB(T_CYF) * txy0, cyf_txy1 = SB(T_CYF) * txy1;
  __syncthreads();
  if (s < jb) return;
  // -- 5: predicted velocity (predict/ux.c, uy.c, force.c), outputs ------------
  const double dnm1 = get_d(S_DN, wm);
  const R km1 = get_r(S_K, wm);
  const double d_0 = DEN(v0), d_m1 = DEN(vm);
  const double d_0l = from_left(d_0), dn0l = from_left(dn0);
  const double dfx = 0.5 * d_0l + 0.5 * d_0;    // x face c, old vof
  const double dfy = 0.5 * d_m1 + 0.5 * d_0;    // y face s, old vof
  const double d1x = 0.5 * dn0l + 0.5 * dn0;    // x face c, new vof
  const double d1y = 0.5 * dnm1 + 0.5 * dn0;    // y face s, new vof
  double uxs = 0., uys = 0.;
  {
    const double p0l = from_left(p0);
    const R k0l = A::left(k0), rv0l = A::left(rv0);
    if (c >= 2 && c <= nx) {
      R s_ = 0;
      s_ -= SB(T_RJF) * (-qxl + qx);
      s_ -= SB(T_RJF) * (-qy_ux + qy_ux_new);
      s_ += SB(T_DFX) * (-qtl + qt);
      s_ += SB(T_DFX) * (-cyf_txy0 + cyf_txy1);
      double g = 0.;
      g -= TB(T_RHF) * (-p0l + p0);
      const R rdfx = R(dfx);
      {
        const R k = R(0.5) * k0l + R(0.5) * k0;
        const R delta = SB(T_RHF) * (-rv0l + rv0);
        s_ += rdfx * refdeninv * tension * k * delta;
      }
      s_ += grav * rdfx;
      const double sd = double(s_);
      if (a.srca_ux && outrow && c_out) msrc(a.srca_ux, fx_row, s) = s_;
      uxs = dfx * ux0 + dtca * sd + dtcb * sbx + dtcg * g;
      uxs /= d1x;
    }
    if (c_in) {
      R s_ = 0;
      s_ -= SB(T_RJC) * (-qm + qmr);
      s_ -= SB(T_RJC) * (-qy_uy + qy_uy_new);
      s_ += SB(T_DCX) * (-qf_txy0 + qf_txy0r);
      s_ += SB(T_DCX) * (-cyc_tyym1 + cyc_tyy0);
      double g = 0.;
      g -= rhy * (-pm + p0);
      {
        const R k = R(0.5) * km1 + R(0.5) * k0;
        const R delta = rhyr * (-rvm1 + rv0);
        s_ += R(dfy) * refdeninv * tension * k * delta;
      }
      const double sd = double(s_);
      if (a.srca_uy && outrow && c_out) msrc(a.srca_uy, ci_row, s) = s_;
      uys = dfy * uy0 + dtca * sd + dtcb * sby + dtcg * g;
      uys /= d1y;
    }
  }
  const double txy0r = double(A::right(txy0));
  if (a.cut) {
    const uint64_t m = __ballot(outrow && c_out && vn0 >= kCutLo && vn0 <= kCutHi);
    if (outrow && lane == 0) a.cut[(size_t)(s - 1) * march_strips(nx) + bx] = m >> 3;
  }
  if (outrow && c_out) {
    auto put_at = [&](double* f, int nh, auto row, int off, double v) {
      AT(row(f, s) + off) = v;
      if (s > ny - nh) AT(row(f, s - ny) + off) = v;
      if (s <= nh) AT(row(f, s + ny) + off) = v;
    };
    auto put = [&](double* f, int nh, auto row, double v) { put_at(f, nh, row, 0, v); };
    auto rv = [&](double* f, int j) { return vof_row(f, j); };
    auto rc = [&](double* f, int j) { return cc_row(f, j); };
    auto rx = [&](double* f, int j) { return xf_row(f, j); };
    put(a.vofn, 2, rv, vn0);
    if (c == 1) put_at(a.vofn, 2, rv, -1, 0.);
    if (c == nx) put_at(a.vofn, 2, rv, 1, 0.);
    if (a.srca_vof) AT(ci_row(a.srca_vof, s)) = src;
    put(a.uxs, 1, rx, c == 1 ? 0. : uxs);
    if (c == nx) put_at(a.uxs, 1, rx, 1, 0.);
    put(a.uys, 1, rc, uys);
    if (c == 1) put_at(a.uys, 1, rc, -1, kUyXm);
    if (c == nx) put_at(a.uys, 1, rc, 1, kUyXp);
    if (a.den1) {
      const double dg = DEN(0.);
      put(a.den1, 1, rc, dn0);
      if (c == 1) put_at(a.den1, 1, rc, -1, dg);
      if (c == nx) put_at(a.den1, 1, rc, 1, dg);
    }
    if (a.txy) {
      put(a.txy, 1, rx, double(txy0));
      if (c == nx) put_at(a.txy, 1, rx, 1, txy0r);
    }
    if (CORR && a.p_out) {
      put(a.p_out, 1, rc, p0);
      if (c == 1) put_at(a.p_out, 1, rc, -1, p0);
      if (c == nx) put_at(a.p_out, 1, rc, 1, p0);
    }
  }
  // -- 6: Poisson right-hand side of row s (compute_potential.c:315-360) -------
  const double cyc_uys = TB(T_CYC) * uys;
  const double gym = per_hy((a.refden / d1y - 1.) * (-psm + ps0));
  const double cg_ym = TB(T_CYC) * gym;
  put_d(S_CU, cyc_uys);
  put_d(S_CG, cg_ym);
  const double q_uxs = TB(T_QF) * uxs;
  const double q_uxsr = from_right(q_uxs);
  const double psl = from_left(ps0);
  const double gxm = per_h((a.refden / d1x - 1.) * (-psl + ps0));
  const double qgx = TB(T_QF) * gxm;
  const double qgxr = from_right(qgx);
  __syncthreads();
  if (outrow && c_out) {
    const double cyc_uysp = get_d(S_CU, wp), cg_yp = get_d(S_CG, wp);
    const double div = TB(T_RJC) * (-q_uxs + q_uxsr - cyc_uys + cyc_uysp);
    const double add = TB(T_RJC) * (-qgx + qgxr - cg_ym + cg_yp);
    AT(ci_row(a.rhs, s)) = c0 * div + c1 * add;
  }
}

template <typename R, bool CORR, int H>
__global__ __launch_bounds__(64 * (H + 5)) void k_tile(const MarchArgs* __restrict__ args) {
  tile_body<R, CORR, H>(*args, blockIdx.x, blockIdx.y);
}

// ensembles: one map entry (case, tile of the case) per workgroup
template <typename R, bool CORR, int H>
__global__ __launch_bounds__(64 * (H + 5)) void k_tile_batch(const MarchArgs* __restrict__ tab,
                                                             const uint2* __restrict__ map) {
  const uint2 m = map[blockIdx.x];
  const MarchArgs& a = tab[m.x];
  const int strips = march_strips(a.nx);
  tile_body<R, CORR, H>(a, (int)m.y % strips, (int)m.y / strips);
}

static const char* const kNames[2][2] = {{"k_tile", "k_tile_corr"}, {"k_tile_mixed", "k_tile_mixed_corr"}};

void tile_launch(const MarchArgs* ma, int nx, int ny, int rows, bool mixed, bool corr) {
  const dim3 grid(march_strips(nx), cdiv(ny, rows)), block(64 * (rows + 5));
  auto pick = [&](auto h) {
    constexpr int H = decltype(h)::value;
    return mixed ? (corr ? k_tile<float, true, H> : k_tile<float, false, H>)
                 : (corr ? k_tile<double, true, H> : k_tile<double, false, H>);
  };
  const auto k = rows == kTileShort ? pick(std::integral_constant<int, kTileShort>())
                                    : pick(std::integral_constant<int, kTileTall>());
  SBFS_TIMED(kNames[mixed][corr], hipLaunchKernelGGL(k, grid, block, 0, stream(), ma));
}

void tile_launch_batch(const MarchArgs* tab, const uint2* map, unsigned blocks, int rows, bool mixed, bool corr) {
  const dim3 grid(blocks), block(64 * (rows + 5));
  auto pick = [&](auto h) {
    constexpr int H = decltype(h)::value;
    return mixed ? (corr ? k_tile_batch<float, true, H> : k_tile_batch<float, false, H>)
                 : (corr ? k_tile_batch<double, true, H> : k_tile_batch<double, false, H>);
  };
  const auto k = rows == kTileShort ? pick(std::integral_constant<int, kTileShort>())
                                    : pick(std::integral_constant<int, kTileTall>());
  SBFS_TIMED(kNames[mixed][corr], hipLaunchKernelGGL(k, grid, block, 0, stream(), tab, map));
}

}  // namespace sbfs
