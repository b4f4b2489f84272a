// k_march: the whole Runge-Kutta stage up to the Poisson right-hand side,
// marching down the rows.
//
// One wavefront owns a strip of kStrip output columns [i0, i0 + kStrip) and
// a band of output rows.  Lane l holds column c = i0 - 3 + l (64 lanes cover
// the strip plus 3 halo columns on each side).  The wavefront walks the band row
// by row; at step s it loads one new row of vof, u, p, psi and computes one
// new row of every intermediate of the reference's stages:
//
//   corner gradients     row s+2   (curvature_tensor.c:16-49)
//   normals + intercept  row s+1   (curvature_tensor.c:51-97, band only)
//   curvature            row s     (curvature_tensor.c:100-135)
//   THINC / mass flux x  row s     (update/fluxx.c, mass_flux.c)
//   THINC / mass flux y  face s+1  (update/fluxy.c, mass_flux.c)
//   txx row s, tyy row s, txy corner row s+1  (predict/txx.c, tyy.c, txy.c)
//   new vof              row s     (update/main.c:54-120)
//   predicted ux, uy     row s     (predict/ux.c, uy.c, force.c)
//   Poisson rhs          row s-1   (compute_potential.c:285-363)
//
// Older rows stay in register rings, x-neighbours come from DPP wavefront
// shifts, so nothing is recomputed across rows and no LDS tile or barrier is
// needed; a term shared by two neighbouring faces or rows is formed once.  Every
// value is formed with the reference's operation order (the per-column quotients
// come from the coefficient tables), which keeps the result bitwise equal to the
// staged kernels.
#include "march_dev.hpp"

#ifndef SBFS_FP64_WAVES
#define SBFS_FP64_WAVES 2
#endif
#ifndef SBFS_MIXED_WAVES
#define SBFS_MIXED_WAVES 3
#endif

namespace sbfs {

// LDS of one wavefront: the column tables, and the older rows that the folded
// FP32 body keeps there (it has no VGPRs left for them; each lane reads back
// only what it wrote, so no barrier is needed).  The FP64 body has: with them
// in LDS a step takes 1484 us instead of 1480 at 2048 x 4096 and 569 instead of
// 566 at 1024 x 2048 with diagnostics.  The streaming one, of larger grids, keeps
// them in LDS all the same: at 4096 x 8192 a step takes 5931 us (5916 to 5949)
// instead of 5957 (5923 to 5986) with the bubbles at random, 5947 instead of 5974
// on a regular pattern (eight runs each, after 60 steps).
enum { RG_QUXS, RG_CYCUYS, RG_D1X, RG_CGY, RG_PSM1, RG_PM1, RG_DNM1, RG_N };
// The FP32 body's FP64 tables are the four that its FP64 parts read (fp64_slot).
template <typename R>
constexpr int fp64_slot(int t) {
  return std::is_same<R, double>::value ? t : t == T_RHF ? 0 : t == T_RJC ? 1 : t == T_QF ? 2 : t == T_CYC ? 3 : -1;
}
template <typename R, bool LR>
struct MarchLds {
  static constexpr bool kSingle = std::is_same<R, float>::value;
  double st[kSingle ? 4 : T_N][64];
  float sf[kSingle ? T_N : 1][64];
  double rings[LR ? RG_N : 1][64];
};
template <typename R, bool CORR, bool ALT>
constexpr bool kLdsRings = CORR && (std::is_same<R, float>::value || ALT);

// R = double: the plain FP64 step.  R = float: the stencils of the
// interface (gradients, normals, curvature, THINC and mass fluxes) and of the
// momentum sources (viscosities, stresses, advection, surface tension,
// buoyancy) in FP32; the vof update, the density-weighted velocity update,
// the pressure gradient and the Poisson right-hand side stay FP64.
// (bx, by): the strip and band of this wavefront
// IN: every lane of the strip holds an interior cell that touches no wall
// (march_inner): only the interface and the strip's output columns mask lanes
// ALT: the FP64 bodies store their output rows streaming (see ST below); the
// FP32 ones address rows by 64 bits (see row below)
template <typename R, bool CORR, bool ALT, bool IN>
__device__ __forceinline__ void march_body(const MarchArgs& a, int bx, int by,
                                           MarchLds<R, kLdsRings<R, CORR, ALT>>& lds) {
  using A = Arith<R>;
  using V3 = V3R<R>;
  constexpr bool NT = ALT && std::is_same<R, double>::value, WIDE = ALT && std::is_same<R, float>::value;
  auto& st = lds.st;
  auto& rings = lds.rings;
  const int lane = threadIdx.x;
  const int nx = a.nx, ny = a.ny;
  // (the strip and rows are the same in every lane, but read from the dispatch
  // order the compiler keeps them, and all that follows from them, in vector
  // registers; said to be uniform they leave 26 of the FP64 bodies' 227 and 12
  // of the mixed bodies' 168, whose row loop then spills nothing: at
  // 2048 x 4096 mixed 215 -> 198 us, with the fold 287 -> 261 us)
  const int i0 = __builtin_amdgcn_readfirstlane(1 + bx * kStrip);
  const int cl = i0 - 3;  // column held by lane 0
  const int c = cl + lane;
  const int jb = __builtin_amdgcn_readfirstlane(1 + by * a.band);
  const int je = __builtin_amdgcn_readfirstlane(min(ny, jb + a.band - 1));
  const bool c_vof = IN || (c >= 0 && c <= nx + 1);   // cells incl. wall ghosts
  const bool c_in = IN || (c >= 1 && c <= nx);        // interior cells
  const bool c_fx = IN || (c >= 1 && c <= nx + 1);    // x faces incl. walls
  const bool c_ux = IN || (c >= 2 && c <= nx);        // x faces between interior cells
  const bool c_first = !IN && c == 1, c_last = !IN && c == nx;
  const bool c_out = c >= i0 && c < i0 + kStrip && (IN || c <= nx);
  const int cc = c < 0 ? 0 : (c > nx + 1 ? nx + 1 : c);
  // The column tables and dt are loaded first and used last before the row
  // loop, after the first rows' loads have been issued: the wavefront waits for
  // memory once, not for each in turn, which was 6 of 31 us at 512 x 1024
  // mixed (k_march at 1024 x 2048 103 -> 98 us, with the fold 127 -> 119).
  double tab[T_N];
  {
    const double* tabs[T_N] = {a.cf.rhf, a.cf.rhc, a.cf.rjf, a.cf.rjc, a.cf.qf, a.cf.qc, a.cf.eqf,
                               a.cf.ecy, a.cf.cyc, a.cf.cyf, a.cf.dfx, a.cf.dcx, a.hxxf1, a.hxxc1};
#pragma unroll
    for (int t = 0; t < T_N; t++) tab[t] = tabs[t][cc];
  }
  const double dt_in = *a.dt;
  constexpr bool LR = kLdsRings<R, CORR, ALT>;
  const int ll = lane > 0 ? lane - 1 : 0, lr = lane < 63 ? lane + 1 : 63;
  // tables in FP64 (the FP64 parts) and in the stencil type
  // (those in FP32 are rounded once here: converted at each use they cost 20
  // instructions per row step, k_march_mixed 194 -> 188 us at 2048 x 4096)
  auto TB = [&](int t) { return st[fp64_slot<R>(t)][lane]; };
  auto TR = [&](int t) { return st[fp64_slot<R>(t)][lr]; };
  auto stencil = [&](int t, int l) {
    if constexpr (std::is_same<R, float>::value) return lds.sf[t][l];
    else return st[t][l];
  };
  auto SB = [&](int t) { return stencil(t, lane); };
  auto SL = [&](int t) { return stencil(t, ll); };
  auto SR = [&](int t) { return stencil(t, lr); };
  // x / HXXF of the lane's column and x / hy: divided in the FP64 body,
  // multiplied by the stored reciprocals in the mixed one
  constexpr bool kExactQ = std::is_same<R, double>::value;
  auto per_h = [&](double x) {
    if constexpr (kExactQ) return x / TB(T_HXXF);
    else return x * TB(T_RHF);
  };
  const double hy = a.hy, rhy = a.cf.rhy;
  auto per_hy = [&](double x) { return kExactQ ? x / hy : x * rhy; };
  const R hyr = uni(R(hy)), rhyr = uni(R(rhy));
  const bool has_b = a.stage != 0;

  // Rows of each layout, shifted to lane 0's column: a (field, byte offset)
  // pair, see RowRef, or a row pointer for fields of 4 GiB or more.
  const ptrdiff_t wc = nx + 2, wf = nx + 1;
  auto row = [&](auto* f, ptrdiff_t e) {
    if constexpr (WIDE) return f + e;
    else return RowRef<std::remove_reference_t<decltype(*f)>>{f, (unsigned)(e * (ptrdiff_t)sizeof(*f))};
  };
  auto vof_row = [&](auto* f, int j) { return row(f, (ptrdiff_t)(j + 1) * wc + cl); };         // L::vof
  auto cc_row = [&](auto* f, int j) { return row(f, (ptrdiff_t)j * wc + cl); };                // L::cc
  auto xf_row = [&](auto* f, int j) { return row(f, (ptrdiff_t)j * wf + cl - 1); };            // L::xf
  auto ci_row = [&](auto* f, int j) { return row(f, (ptrdiff_t)(j - 1) * nx + cl - 1); };      // L::ci
  auto fx_row = [&](auto* f, int j) { return row(f, (ptrdiff_t)(j - 1) * (nx - 1) + cl - 2); };  // L::fx
  const unsigned loff = (unsigned)lane * 8u;
  auto AT = [&](auto r) -> auto& { return lane_at(r, loff); };
  // Output rows: with NT (fields too large for the Infinity Cache to keep,
  // stream_fields) the FP64 bodies store them streaming (non-temporal), which
  // measured k_march 1198 -> 1164 us and k_march_corr 1502 -> 1446 us at
  // 4096 x 8192; the FP32 bodies slowed by 4-5 % with it and keep ordinary
  // stores.
  auto ST = [&](auto r, double v) {
    if constexpr (NT) __builtin_nontemporal_store(v, lane_gp(r, loff));
    else AT(r) = v;
  };
  // loads of row jw, already wrapped into 1..ny
  auto ld_vof = [&](int jw) { return c_vof ? AT(vof_row(a.vof, jw)) : 0.; };
  auto ld_ux = [&](int jw) { return c_fx ? AT(xf_row(a.ux, jw)) : 0.; };
  auto ld_cc = [&](const double* f, int jw) { return c_vof ? AT(cc_row(f, jw)) : 0.; };
  auto DEN = [&](double v) { return mix_clamp(a.denr, a.dlo, a.dhi, v); };
  // viscosity at x face c from the vof on its two sides (viscosity.c:37-53)
  auto VISUX = [&](int col, R vl, R vr) {
    R v;
    if (!IN && col == 1) v = vl;
    else if (!IN && col == nx + 1) v = vr;
    else v = R(0.5) * vl + R(0.5) * vr;
    return mixr<R>(a.visr, a.vlo, a.vhi, v);
  };
  auto VISUY = [&](R vb, R vt) { return mixr<R>(a.visr, a.vlo, a.vhi, R(0.5) * vb + R(0.5) * vt); };

  // Rings (row offsets relative to the current step s).  Several terms of
  // the reference's stencils are the same expression evaluated at the next
  // column or row (the right face of cell c is the left face of cell c+1);
  // they are formed once and taken from the neighbouring lane (DPP) or from
  // the previous step, which gives the same bits.
  double v0 = 0., vp1 = 0., vp2 = 0.;                       // vof s..s+2
  R rvm1 = 0;                                               // vof s-1, stencil type
  R g0x = 0, g0y = 0, g1x = 0, g1y = 0, g2x = 0, g2y = 0;   // corners s..s+2
  R g1xr = 0, g1yr = 0;                                     // corners of c+1, row s+1
  R n0x = 0, n0y = 0, n0z = 0, n1x = 0, n1y = 0, n1z = 0;   // normals s, s+1
  R km1 = 0, k0 = 0;                                        // curvature s-1, s
  R mfxm1 = 0, mfx0 = 0;                                    // x mass fluxes s-1, s
  R fy0 = 0, fyp1 = 0, mfy0 = 0, mfyp1 = 0;                 // y faces s, s+1
  R visx0 = 0, visx1 = 0, visy0 = 0, visy1 = 0;             // viscosities rows / faces s, s+1
  R txy0 = 0, cyf_txy0 = 0, cyc_tyym1 = 0;                  // stress terms of rows s, s-1
  double d_0 = 0.;                                          // density of vof row s
  double vn0 = 0., dnm1 = 0., dn0 = 0.;                     // new vof row s, its density s-1, s
  double ux0 = 0., uxp1 = 0., uy0 = 0., uyp1 = 0.;
  double pm1 = 0., p0 = 0.;
  double psm1 = 0., ps0 = 0., psp1 = 0.;                    // psi[0] s-1..s+1 (s+1: folded projection)
  double pop1 = 0.;                                         // previous potential s+1
  R qy_ux = 0, qy_uy = 0;                                   // y momentum fluxes at face s
  double q_uxs_m1 = 0., cyc_uys_m1 = 0.;                    // rhs terms of row s-1
  double d1x_m1 = 0., d1y = 0., cg_ym = 0.;                 // rhs densities / y gradient
  const int s_first = jb - (CORR ? kWarmCorr : kWarm);
  auto ring_ld = [&](int k, double reg) { return LR ? rings[k][lane] : reg; };
  auto ring_st = [&](int k, double& reg, double v) {
    if (LR) rings[k][lane] = v;
    else reg = v;
  };
  // Every input of step s+1 is loaded during step s, unconditionally (the
  // rows wrap, so the last step's loads stay in bounds and go unused), and
  // is first read by the fence below, after the bulk of the step's
  // arithmetic and before its first store.  The vector-memory counter
  // retires loads and stores in issue order, so a wait placed after the
  // step's stores would also wait for them; at the fence only the step's
  // loads and the previous step's stores are outstanding.
  // w1..w3: rows s+1..s+3 wrapped into 1..ny, advanced with s
  int w1 = wrap_r(s_first + 1, ny), w2 = wrap_r(s_first + 2, ny), w3 = wrap_r(s_first + 3, ny);
  // prefetched inputs of the next step (the folded projection needs psi one
  // row further ahead)
  double nv = ld_vof(w2), nux = ld_ux(w1), nuy = ld_cc(a.uy, w1);
  double np = ld_cc(a.p, wrap_r(s_first, ny)), nps = ld_cc(a.psi0, CORR ? w1 : wrap_r(s_first, ny));
  double npo = CORR ? ld_cc(a.psi_old, w1) : 0.;
  // learned curvature of row s, prefetched a row ahead (0 where absent)
  // (no listed cell: every value is NaN, so none is read)
  const float* kap = (a.kappa && *a.kappa_n != 0u) ? a.kappa : nullptr;
  auto ld_kap = [&](int jw) { return (kap && c_in) ? lane_at(ci_row(kap, jw), loff >> 1) : 0.f; };
  float nkap = ld_kap(wrap_r(s_first, ny));
  // Momentum sources between stages: the FP32 bodies form them in FP32 and
  // store them so (4-byte elements in the same layout, the first half of the
  // buffer), which the next stage reads back exactly; half the bytes and the
  // same bits as an FP64 copy (measured 1287 -> 1189 us for the folded mixed
  // kernel at 4096 x 8192).  The vof source is formed in FP64 and stays so.
  auto msrc = [&](auto* f, auto rowf, int j) -> auto& {
    if constexpr (std::is_same<R, float>::value) {
      using F = std::conditional_t<std::is_const<std::remove_pointer_t<decltype(f)>>::value, const float, float>;
      return lane_at(rowf((F*)f, j), loff >> 1);
    } else {
      return AT(rowf(f, j));
    }
  };
  // beta sources of row s (stages 1, 2): the vof's for every marched row,
  // uy's from the first output row on (the predicted uy of row je+1 enters
  // the Poisson rhs of row je), ux's on output rows
  // (the FP32 stage-0 body keeps the prefetched momentum sources as float
  // until they are used, after the fence: widened at the load, each waits
  // for its load and with it for every load issued before it, which cost
  // k_march_mixed 928 against 860 us at 4096 x 8192; the folded body
  // measured faster with the early widening, 1158 against 1189-1205 us)
  using MS = std::conditional_t<std::is_same<R, float>::value && !CORR, float, double>;
  auto ld_sb = [&](int s_, int jw, double& bv, MS& by, MS& bx) {
    bv = 0.;
    by = bx = MS(0);
    if (has_b && c_in) {
      bv = AT(ci_row(a.srcb_vof, jw));
      if (s_ >= jb) by = msrc(a.srcb_uy, ci_row, jw);
      if (s_ >= jb && s_ <= je && (IN || c >= 2)) bx = msrc(a.srcb_ux, fx_row, jw);
    }
  };
  double nsbv;
  MS nsby, nsbx;
  ld_sb(s_first, wrap_r(s_first, ny), nsbv, nsby, nsbx);
  // the fence below, for the first step's inputs: without it the loop entry
  // would carry outstanding loads into every step's first reads
  auto fence = [&]() {
    asm volatile("" : "+v"(nv), "+v"(nux), "+v"(nuy), "+v"(np), "+v"(nps), "+v"(nkap), "+v"(nsbv), "+v"(nsby),
                 "+v"(nsbx));
    if constexpr (CORR) asm volatile("" : "+v"(npo));
  };
  // the vof ring holds rows s_first and s_first + 1 before the first step,
  // so the first step's corner gradients are already valid
  vp1 = ld_vof(wrap_r(s_first, ny));
  vp2 = ld_vof(w1);
#pragma unroll
  for (int t = 0; t < T_N; t++) {
    if (fp64_slot<R>(t) >= 0) st[fp64_slot<R>(t)][lane] = tab[t];
    if (lds.kSingle) lds.sf[t][lane] = float(tab[t]);
  }
  if (LR)
    for (int k = 0; k < RG_N; k++) rings[k][lane] = 0.;
  __syncthreads();
  const double dt = uni(dt_in);
  // (dt * a.ca equals a.ca * dt bit for bit)
  const double dtca = uni(dt * a.ca), dtcb = uni(dt * a.cb), dtcg = uni(dt * a.cg);
  const double dt_old = a.g_old * dt, dt_new = a.g_new * dt;
  const double c0 = uni(1. / a.norm / dt_new * a.refden);
  const double c1 = uni(1. / a.norm * -1. / dt_new * dt_old);
  const R denr1 = uni(R(a.denr) - R(1));
  // the previous stage's projection (correct_velocity/ux.c, uy.c): the same
  // expressions as k_post, with the lane's face distance in the divisions
  const double pdtn = a.pg_new * dt, pdto = a.pg_old * dt;
  const double pcoef = -1. / pdtn * pdto;
  const double pdtc = uni(pdtn * pcoef), irefden = uni(1. / a.refden);
  const R refdeninv = uni(R(a.refdeninv)), tension = uni(R(a.tension)), grav = uni(R(a.grav));
  const double pcx0 = uni(pdtn / a.refden), pcy = uni(pdtn / a.refden / hy);
  asm volatile("" : "+v"(vp1), "+v"(vp2));
  fence();
  unsigned weight = 0;  // marched rows with an interface cell
  for (int s = s_first; s <= je + 1; s++) {
    // -- new input rows -----------------------------------------------------
    rvm1 = R(v0); v0 = vp1; vp1 = vp2; vp2 = nv;
    ux0 = uxp1; uxp1 = nux;
    uy0 = uyp1; uyp1 = nuy;
    if (!LR) pm1 = p0;
    p0 = np;
    if (CORR) {
      ps0 = psp1; psp1 = nps;   // row s-1 of the potential is in LDS
      pop1 = npo;
    } else {
      psm1 = ps0; ps0 = nps;
    }
    const bool outrow = s >= jb && s <= je;
    if (a.weight) weight += __ballot(c_vof && in_band(v0)) != 0ull ? 1u : 0u;
    const float kap = nkap;
    const double sbv = nsbv;
    const MS sby = nsby, sbx = nsbx;
    // (the folded bodies load the beta sources first: the FP32 folded body
    // widens them at the load, and the wait that needs then covers them
    // alone rather than every prefetch of the step, 1158 -> 1139 us at
    // 4096 x 8192)
    if (CORR) ld_sb(s + 1, w1, nsbv, nsby, nsbx);
    nv = ld_vof(w3);
    nux = ld_ux(w2);
    nuy = ld_cc(a.uy, w2);
    np = ld_cc(a.p, w1);
    nps = ld_cc(a.psi0, CORR ? w2 : w1);
    if (CORR) npo = ld_cc(a.psi_old, w2);
    nkap = ld_kap(w1);
    if (!CORR) ld_sb(s + 1, w1, nsbv, nsby, nsbx);
    w1 = w2;
    w2 = w3;
    w3 = w3 == ny ? 1 : w3 + 1;
    const R rux0 = R(ux0), ruxp1 = R(uxp1), ruy0 = R(uy0), ruyp1 = R(uyp1);
    const R rv0 = R(v0), rvp1 = R(vp1);
    // -- corner gradients, row s+2 (curvature_tensor.c:16-49) ----------------
    g0x = g1x; g0y = g1y; g1x = g2x; g1y = g2y;
    // (corners of c+1, row s: shifted again rather than kept, one register
    // pair fewer)
    const R g0xr = A::right(g0x), g0yr = A::right(g0y);
    {
      const double mm = from_left(vp1), pm = vp1, mp = from_left(vp2), pp = vp2;
      R gx = 0, gy = 0;
      if (c_fx && !(mm == pm && mm == mp && mm == pp)) {
        const R rmm = R(mm), rpm = R(pm), rmp = R(mp), rpp = R(pp);
        gx = SB(T_RHF) * (-rmm + rpm - rmp + rpp);
        gy = rhyr * (-rmm - rpm + rmp + rpp);
        const R norm = A::sqr(gx * gx + gy * gy);
        const R ninv = A::div(R(1), fmax(norm, A::eps()));
        gx = gx * ninv;
        gy = gy * ninv;
      }
      g2x = gx;
      g2y = gy;
    }
    const R g2xr = A::right(g2x), g2yr = A::right(g2y);
    g1xr = A::right(g1x);
    g1yr = A::right(g1y);
    // -- normals, row s+1 (curvature_tensor.c:51-97) ---------------------------
    n0x = n1x; n0y = n1y; n0z = n1z;
    {
      R nxv = 0, nyv = 0, nz = 0;
      if (c_in && in_band(vp1)) {
        nxv = g1x + g1xr + g2x + g2xr;
        nyv = g1y + g1yr + g2y + g2yr;
        nxv = A::div(nxv, SB(T_HXXC));
        nyv = A::div(nyv, hyr);
        const R norm = A::sqr(nxv * nxv + nyv * nyv);
        const R ninv = A::div(R(1), fmax(norm, A::eps()));
        nxv *= ninv;
        nyv *= ninv;
        nz = A::intercept(vp1);
      }
      n1x = nxv;
      n1y = nyv;
      n1z = nz;
    }
    // -- curvature, row s (curvature_tensor.c:100-135) -------------------------
    km1 = k0;
    {
      R kk = 0;
      // the learned value of row s replaces the plain one where the network
      // gave one
      const float kl = kap;
      if (c_in) {
        const R nxm = R(0.5) * g0x + R(0.5) * g1x;
        const R nxp = R(0.5) * g0xr + R(0.5) * g1xr;
        const R nym = R(0.5) * g0y + R(0.5) * g0yr;
        const R nyp = R(0.5) * g1y + R(0.5) * g1yr;
        const R div = SB(T_RJC) * (-SB(T_QF) * nxm + SR(T_QF) * nxp - SB(T_CYC) * nym + SB(T_CYC) * nyp);
        kk = R(-1) * div;
        if (kl == kl && kl != 0.f) kk = R(kl);
      }
      k0 = kk;
    }
    // -- THINC and mass fluxes at x face c, row s (fluxx.c, mass_flux.c) -------
    mfxm1 = mfx0;
    R fx0 = 0;
    {
      const double vl = from_left(v0);
      const R nlx = A::left(n0x), nly = A::left(n0y), nlz = A::left(n0z);
      R mf = 0;
      if (c_fx) {
        const R vel = rux0;
        if (IN || (c != 1 && c != nx + 1)) {
          const bool up = vel < R(0);
          const double v = up ? v0 : vl;
          const V3 n = up ? V3{n0x, n0y, n0z} : V3{nlx, nly, nlz};
          fx0 = thinc_flux<R, true>(vel, v, in_band(v) ? n : V3{0, 0, 0});
        }
        mf = vel + denr1 * fx0;
      }
      mfx0 = mf;
    }
    // -- THINC and mass fluxes at y face s+1 (fluxy.c, mass_flux.c) ------------
    fy0 = fyp1;
    mfy0 = mfyp1;
    {
      R f = 0, mf = 0;
      if (c_vof) {
        const R vel = ruyp1;
        if (IN || (c != 0 && c != nx + 1)) {
          const bool up = vel < R(0);
          const double v = up ? vp1 : v0;
          const V3 n = up ? V3{n1x, n1y, n1z} : V3{n0x, n0y, n0z};
          f = thinc_flux<R, false>(vel, v, in_band(v) ? n : V3{0, 0, 0});
        }
        mf = vel + denr1 * f;
      }
      fyp1 = f;
      mfyp1 = mf;
    }
    // -- viscosities (viscosity.c) ------------------------------------------------
    // (every DPP shift runs in uniform control flow: an inactive source lane
    // would not deliver its value)
    const double v0l = from_left(v0);
    const R rv0l = R(v0l), rvp1l = A::left(rvp1);
    const R rux0r = A::right(rux0);
    const R ruyp1l = A::left(ruyp1);
    visx0 = visx1;
    visx1 = VISUX(c, rvp1l, rvp1);   // x face c, row s+1
    visy0 = visy1;
    visy1 = VISUY(rv0, rvp1);        // y face s+1
    // -- new vof, row s (update/main.c:54-120), FP64 ---------------------------
    double src = 0.;
    const double fx0d = double(fx0);
    const double fx0r = A::right(fx0);
    {
      double v = 0.;
      if (c_in) {
        src = TB(T_RJC) * (+TB(T_QF) * fx0d - TR(T_QF) * fx0r + TB(T_CYC) * double(fy0) - TB(T_CYC) * double(fyp1));
        v = v0;
        v += dtca * src;
        if (has_b) v += dtcb * sbv;
      }
      vn0 = v;
    }
    // -- densities (density.c) and their face averages -------------------------
    const double d_m1 = d_0;
    d_0 = DEN(v0);
    if (!LR) dnm1 = dn0;
    dn0 = DEN(vn0);
    const double d_0l = from_left(d_0), dn0l = from_left(dn0);
    const double dfx = 0.5 * d_0l + 0.5 * d_0;    // x face c, row s, old vof
    const double dfy = 0.5 * d_m1 + 0.5 * d_0;    // y face s, old vof
    const double d1x = 0.5 * dn0l + 0.5 * dn0;    // x face c, row s, new vof
    d1y = 0.5 * ring_ld(RG_DNM1, dnm1) + 0.5 * dn0;  // y face s, new vof
    // Rows before jb - 1 only fill the interface and density rings: their
    // stresses, momentum fluxes, predicted velocity and Poisson rhs reach no
    // output, since every ring that row jb's predicted velocity reads is
    // refilled by row jb - 1, and the rhs of row jb is formed at step jb + 1
    // from the rings of step jb.  So the stresses and momentum fluxes start
    // at row jb - 1, the predicted velocity and the rhs at row jb.  (The
    // flags are uniform: the DPP shifts inside stay in uniform control flow.)
    // Measured on the 2048 x 4096 swarm: the folded body gains from both
    // (k_march_corr 452 -> 414 us); the plain one gains from the later start
    // of the predicted velocity and the rhs (k_march 296 -> 288 us) but loses
    // with the stresses and fluxes skipped too (361 us, its code laid out
    // worse), so it computes those on every row.
    const bool mom = !CORR || s >= jb - 1, pred = s >= jb;
    const R txy_prev = txy0;   // corner row s
    R txx0 = 0, tyy0 = 0, txy1 = 0;
    R qx = 0, qm = 0, qxl = 0, qmr = 0, qt = 0, qtl = 0, qf_txy0 = 0, qf_txy0r = 0;
    R qy_ux_new = 0, qy_uy_new = 0, cyf_txy1 = 0, cyc_tyy0 = 0;
    if (mom) {
      // -- stress tensor (predict/txx.c, tyy.c, txy.c) --------------------------
      const R visx0r = A::right(visx0), visy1l = A::left(visy1);
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
        const R vx = R(0.5) * visx0 + R(0.5) * visx1;
        const R vy = R(0.5) * visy1l + R(0.5) * visy1;
        const R lxy = rhyr * (-rux0 + ruxp1);
        const R lyx = SB(T_RHF) * (-ruyp1l + ruyp1);
        txy1 = vx * lxy + vy * lyx;
      }
      // -- momentum fluxes shared between neighbouring faces -------------------
      const R mfx0r = A::right(mfx0), mfyp1l = A::left(mfyp1);
      const R ruy0l = A::left(ruy0);
      // ux, x direction: cell-centre flux (mp * up) of the cell right of face c
      qx = (SB(T_EQF) * mfx0 + SR(T_EQF) * mfx0r) * (R(0.5) * rux0 + R(0.5) * rux0r);
      // uy, x direction: corner flux (mm * um) at face c
      qm = (SB(T_EQF) * mfxm1 + SB(T_EQF) * mfx0) * (R(0.5) * ruy0l + R(0.5) * ruy0);
      qxl = A::left(qx);
      qmr = A::right(qm);
      qt = SB(T_QC) * txx0;
      qtl = A::left(qt);
      qf_txy0 = SB(T_QF) * txy_prev;
      qf_txy0r = A::right(qf_txy0);
      // ux, y direction: corner flux (mp * up) at face s+1
      qy_ux_new = (SL(T_ECY) * mfyp1l + SB(T_ECY) * mfyp1) * (R(0.5) * rux0 + R(0.5) * ruxp1);
      // uy, y direction: cell-centre flux (mp * up) of row s
      qy_uy_new = (SB(T_ECY) * mfy0 + SB(T_ECY) * mfyp1) * (R(0.5) * ruy0 + R(0.5) * ruyp1);
      cyf_txy1 = SB(T_CYF) * txy1;
      cyc_tyy0 = SB(T_CYC) * tyy0;
    }
    // The fence: an empty statement that reads and redefines the next step's
    // inputs, so the compiler waits for their loads here, ahead of this
    // step's first store, rather than where the loop carries them over.
    fence();
    double uxs = 0., uys = 0.;
    if (mom) {
      if (pred) {
        const double p0l = from_left(p0);
        const R k0l = A::left(k0);
        // -- predicted ux, row s (predict/ux.c, force.c) -----------------------
        if (c_ux) {
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
          uxs = dfx * ux0 + dtca * sd + dtcb * double(sbx) + dtcg * g;
          uxs /= d1x;
        }
        // -- predicted uy, row s (predict/uy.c, force.c) -----------------------
        if (c_in) {
          R s_ = 0;
          s_ -= SB(T_RJC) * (-qm + qmr);
          s_ -= SB(T_RJC) * (-qy_uy + qy_uy_new);
          s_ += SB(T_DCX) * (-qf_txy0 + qf_txy0r);
          s_ += SB(T_DCX) * (-cyc_tyym1 + cyc_tyy0);
          double g = 0.;
          g -= rhy * (-ring_ld(RG_PM1, pm1) + p0);
          {
            const R k = R(0.5) * km1 + R(0.5) * k0;
            const R delta = rhyr * (-rvm1 + rv0);
            s_ += R(dfy) * refdeninv * tension * k * delta;
          }
          const double sd = double(s_);
          if (a.srca_uy && outrow && c_out) msrc(a.srca_uy, ci_row, s) = s_;
          uys = dfy * uy0 + dtca * sd + dtcb * double(sby) + dtcg * g;
          uys /= d1y;
        }
      }
      qy_ux = qy_ux_new;
      qy_uy = qy_uy_new;
      cyf_txy0 = cyf_txy1;
      cyc_tyym1 = cyc_tyy0;
      txy0 = txy1;
      // -- outputs of row s -----------------------------------------------------
      const double txy0r = double(A::right(txy_prev));
      if (a.cut) {
        const uint64_t m = __ballot(outrow && c_out && vn0 >= kCutLo && vn0 <= kCutHi);
        if (outrow && lane == 0) a.cut[(size_t)(s - 1) * march_strips(nx) + bx] = m >> 3;
      }
      if (outrow && c_out) {
        auto put = [&](double* f, int nh, auto row, double v) {
          ST(row(f, s), v);
          if (s > ny - nh) ST(row(f, s - ny), v);
          if (s <= nh) ST(row(f, s + ny), v);
        };
        auto put_at = [&](double* f, int nh, auto row, int off, double v) {
          ST(row(f, s) + off, v);
          if (s > ny - nh) ST(row(f, s - ny) + off, v);
          if (s <= nh) ST(row(f, s + ny) + off, v);
        };
        auto rv = [&](double* f, int j) { return vof_row(f, j); };
        auto rc = [&](double* f, int j) { return cc_row(f, j); };
        auto rx = [&](double* f, int j) { return xf_row(f, j); };
        put(a.vofn, 2, rv, vn0);
        if (c_first) put_at(a.vofn, 2, rv, -1, 0.);
        if (c_last) put_at(a.vofn, 2, rv, 1, 0.);
        if (a.srca_vof) ST(ci_row(a.srca_vof, s), src);
        put(a.uxs, 1, rx, c_first ? 0. : uxs);
        if (c_last) put_at(a.uxs, 1, rx, 1, 0.);
        put(a.uys, 1, rc, uys);
        if (c_first) put_at(a.uys, 1, rc, -1, kUyXm);
        if (c_last) put_at(a.uys, 1, rc, 1, kUyXp);
        if (a.den1) {
          const double dg = DEN(0.);
          put(a.den1, 1, rc, dn0);
          if (c_first) put_at(a.den1, 1, rc, -1, dg);
          if (c_last) put_at(a.den1, 1, rc, 1, dg);
        }
        if (a.txy) {
          put(a.txy, 1, rx, double(txy_prev));
          if (c_last) put_at(a.txy, 1, rx, 1, txy0r);
        }
        if (CORR && a.p_out) {
          // the previous stage's updated pressure, with its Neumann ghosts
          put(a.p_out, 1, rc, p0);
          if (c_first) put_at(a.p_out, 1, rc, -1, p0);
          if (c_last) put_at(a.p_out, 1, rc, 1, p0);
        }
      }
    }
    // -- Poisson right-hand side of row s-1 (compute_potential.c:315-360), FP64
    if (pred) {
      // u* divergence: the x-face terms of cell c+1 come from lane c+1
      const double q_uxs = ring_ld(RG_QUXS, q_uxs_m1);     // QF * ux* at face c, row s-1
      const double q_uxsr = from_right(q_uxs);
      const double cyc_uys0 = TB(T_CYC) * uys;
      // explicit split-pressure term: the gradient at face c+1 is lane c+1's
      // gradient at its left face; the top y face of row s-1 is the bottom
      // face of row s, kept for the next step
      const double psm1v = ring_ld(RG_PSM1, psm1);
      const double psl = from_left(psm1v);
      const double dxm = ring_ld(RG_D1X, d1x_m1);
      const double gxm = per_h((a.refden / dxm - 1.) * (-psl + psm1v));
      const double qgx = TB(T_QF) * gxm;
      const double qgxr = from_right(qgx);
      const double gyp = per_hy((a.refden / d1y - 1.) * (-psm1v + ps0));
      const double cg_yp = TB(T_CYC) * gyp;
      const int r = s - 1;
      if (r >= jb && r <= je && c_out) {
        const double div = TB(T_RJC) * (-q_uxs + q_uxsr - ring_ld(RG_CYCUYS, cyc_uys_m1) + cyc_uys0);
        const double add = TB(T_RJC) * (-qgx + qgxr - ring_ld(RG_CGY, cg_ym) + cg_yp);
        ST(ci_row(a.rhs, r), c0 * div + c1 * add);
      }
      ring_st(RG_CGY, cg_ym, cg_yp);
      ring_st(RG_CYCUYS, cyc_uys_m1, cyc_uys0);
    }
    ring_st(RG_QUXS, q_uxs_m1, TB(T_QF) * uxs);
    ring_st(RG_D1X, d1x_m1, d1x);
    if (CORR) ring_st(RG_PSM1, psm1, ps0);
    if (LR) {
      rings[RG_PM1][lane] = p0;
      rings[RG_DNM1][lane] = dn0;
    }
    if (CORR) {
      // The previous stage's projection of the rows prefetched for the next
      // step (unused after the last step), formed here where the stencil's
      // temporaries are dead: ux of row
      // s+2, uy of face s+2 (correct_velocity/ux.c:26-45, uy.c:26-43) and the
      // pressure of row s+1 (update_pressure.c:13-24, written with the
      // outputs of that row), with k_post's expressions and the lane's own
      // face distance.  The vof is this stage's input, i.e. the previous
      // stage's new vof.
      const double da = DEN(vp1), db = DEN(vp2);   // rows s+1, s+2
      const double dbl = from_left(db);
      const double nps_l = from_left(nps), npo_l = from_left(npo);
      {
        double u = 0.;
        if (c_ux) {
          u = nux;
          u -= per_h(pcx0) * (-nps_l + nps);
          const double d = 0.5 * dbl + 0.5 * db;
          u += per_h(pdtc * (1. / d - irefden)) * (-npo_l + npo);
        }
        nux = u;
      }
      {
        double u = 0.;
        if (!IN && c == 0) u = kUyXm;
        else if (!IN && c == nx + 1) u = kUyXp;
        else if (c_in) {
          u = nuy;
          u -= pcy * (-psp1 + nps);
          const double d = 0.5 * da + 0.5 * db;
          u += per_hy(pdtc * (1. / d - irefden)) * (-pop1 + npo);
        }
        nuy = u;
      }
      // (stage 2 of a folded step: the input pressure plus stage 0's
      // potential, which stage 1 formed and did not store, then stage 1's)
      if (c_in) np = (a.p_twice ? np + pop1 : np) + psp1;
    }
  }
  if (a.weight && lane == 0) a.weight[by * march_strips(nx) + bx] = weight;
}

__global__ __launch_bounds__(1024) void k_march_order(const unsigned* __restrict__ weight,
                                                      unsigned* __restrict__ order, int n, int max_weight) {
  constexpr int kB = 32, kPer = 8, kT = 1024;
  __shared__ unsigned cnt[kB], next[kB];
  const int t = threadIdx.x;
  const unsigned mw = max_weight > 0 ? (unsigned)max_weight : 1u;
  // the buckets of kPer units per thread, their loads issued together
  // (kB: no unit)
  auto buckets = [&](int base, int* b) {
    unsigned w[kPer];
#pragma unroll
    for (int i = 0; i < kPer; i++) {
      const int u = base + i * kT + t;
      w[i] = u < n ? weight[u] : 0u;
    }
#pragma unroll
    for (int i = 0; i < kPer; i++) {
      const int u = base + i * kT + t;
      b[i] = u < n ? (int)((unsigned long long)min(w[i], mw) * (kB - 1) / mw) : kB;
    }
  };
  // Adds the wavefront's lanes with a unit to their buckets of h and gives
  // each such lane a distinct slot: one atomic per distinct bucket in the
  // wavefront (most units share the bucket of weight 0, and lane-by-lane
  // atomics on one LDS word serialise).  Called in uniform control flow.
  const int lane = t & 63;
  auto add = [&](unsigned* h, int b) -> unsigned {
    unsigned slot = 0;
    unsigned long long left = __ballot(b < kB);
    while (left) {
      const int lead = __ffsll((long long)left) - 1;
      const int bl = __shfl(b, lead);
      const unsigned long long m = __ballot(b == bl);
      unsigned first = 0;
      if (lane == lead) first = atomicAdd(&h[bl], (unsigned)__popcll(m));
      first = __shfl(first, lead);
      if ((m >> lane) & 1ull) slot = first + (unsigned)__popcll(m & ((1ull << lane) - 1ull));
      left &= ~m;
    }
    return slot;
  };
  if (t < kB) cnt[t] = 0;
  __syncthreads();
  for (int base = 0; base < n; base += kPer * kT) {
    int b[kPer];
    buckets(base, b);
#pragma unroll
    for (int i = 0; i < kPer; i++) add(cnt, b[i]);
  }
  __syncthreads();
  if (t == 0) {
    unsigned s = 0;
    for (int b = kB - 1; b >= 0; b--) {
      next[b] = s;
      s += cnt[b];
    }
  }
  __syncthreads();
  for (int base = 0; base < n; base += kPer * kT) {
    int b[kPer];
    buckets(base, b);
#pragma unroll
    for (int i = 0; i < kPer; i++) {
      const unsigned slot = add(next, b[i]);
      if (b[i] < kB) order[slot] = (unsigned)(base + i * kT + t);
    }
  }
}

// The FP64 bodies need 199 to 222 VGPRs, two wavefronts per SIMD (three
// would spill dozens of registers to scratch, measured 1.4x slower).  The
// FP32 bodies need 155 of 168 VGPRs, three wavefronts per SIMD, which hides more of
// their latency (the folded variant 1.35x faster than at two).
// The arguments arrive through a pointer to device memory, not by value:
// held as kernel arguments, the ~50 uniform pointers and constants of
// MarchArgs outgrow the scalar registers, and the compiler spills them into
// vector lanes (v_writelane / v_readlane in the row loop, up to 185 of them
// in the FP64 folded body); from memory it reloads them with scalar loads.

// the (strip, band) of this workgroup: from the grid, or from the dispatch
// order (false: a slot past the last unit)
// In the grid's order, XCD x (the hardware deals workgroups to the 8 XCDs in turn)
// takes the x-th eighth of the units, band by band: neighbouring strips, whose rows
// overlap by 6 columns and share their end lines, run on one XCD and read them from
// its L2.  Dealt out in turn, each XCD fetched them again: k_march_mixed 930 -> 763
// us and folded 1180 -> 948 at 4096 x 8192, 213 -> 186 and 285 -> 249 at 2048 x 4096,
// 49 -> 47 and 63 -> 60 at 1024 x 1500.  In the dispatch order, whose units of equal
// weight are mostly neighbours too, an XCD takes runs of kOrderChunk entries of each
// 8 kOrderChunk: an FP64 step 1524 -> 1488 us at 2048 x 4096 (k_march 261 -> 260 and
// folded 346 -> 333), 6006 -> 5950 at 4096 x 8192 with the bubbles on a regular
// pattern and level with them at random (5934 and 5925); k_march 99.5 -> 98 and folded
// 120.5 -> 119.4 at 1024 x 2048.  (Runs of 64 took the folded kernel from 356 to 350
// at 2048 x 4096 but from 119 to 122 at 1024 x 2048; of 128, where the heaviest no
// longer start first, to 418 and 149.  Without the order, eighths as above and three
// rounds took 4000 us instead of 3880 for a step's three at 4096 x 8192.)
__device__ __forceinline__ bool march_unit(const MarchArgs& a, int& bx, int& by) {
  bx = blockIdx.x;
  by = blockIdx.y;
  if (a.order) {
    const unsigned b = blockIdx.x, n = (unsigned)march_units(a.nx, a.ny, a.band);
    constexpr unsigned C = kOrderChunk;
    const unsigned at = b / (8 * C) * (8 * C) + b % 8 * C + b / 8 % C;
    if (at >= n) return false;
    const unsigned u = (unsigned)__builtin_amdgcn_readfirstlane((int)a.order[at]);
    if (u >= n) return false;
    const int strips = march_strips(a.nx);
    bx = (int)u % strips;
    by = (int)u / strips;
  } else {
    const int strips = (int)gridDim.x, n = strips * (int)gridDim.y, b = by * strips + bx;
    const int xcd = b & 7;
    const int u = xcd * (n >> 3) + min(xcd, n & 7) + (b >> 3);
    bx = u % strips;
    by = u / strips;
  }
  return true;
}
// Whether every lane of strip bx holds an interior cell away from the walls
// (all strips but the first and the last one or two): in FP64 those run the body
// without the walls' lane masks.  In the masked body about 170 exec-mask blocks
// with their branches interrupt a row step, which every strip paid for the few
// at the walls; without them k_march takes 264 us instead of 283 at 2048 x 4096
// and the folded kernel 333 instead of 352.  At 4096 x 8192, where the card's power
// bounds the FP64 step, the folded kernel's inner body takes the step from 6004 to
// 5950 us with the bubbles on a regular pattern and is level with them at random (5913
// and 5925).  The FP32 bodies, which wait for memory more than they compute, got
// slower (2048 x 4096: 206 us against 198, with the fold 273 against 261) and keep the
// one masked body.
__device__ __forceinline__ bool march_inner(int nx, int bx) { return bx >= 1 && 1 + bx * kStrip + 60 <= nx; }
template <typename R, bool CORR, bool ALT>
__device__ __forceinline__ void march_strip(const MarchArgs& a, int bx, int by) {
  __shared__ MarchLds<R, kLdsRings<R, CORR, ALT>> lds;
  if (std::is_same<R, double>::value && march_inner(a.nx, bx)) march_body<R, CORR, ALT, true>(a, bx, by, lds);
  else march_body<R, CORR, ALT, false>(a, bx, by, lds);
}
#define SBFS_MARCH_KERNEL(name, R, CORR, WAVES)                                            \
  __global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(WAVES))) void name( \
      const MarchArgs* __restrict__ args) {                                               \
    const MarchArgs& a = *args;                                                           \
    int bx, by;                                                                           \
    if (march_unit(a, bx, by)) march_strip<R, CORR, false>(a, bx, by);                    \
  }                                                                                       \
  __global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(WAVES))) void name##_batch( \
      const MarchArgs* __restrict__ tab, const uint2* __restrict__ map) {                \
    const uint2 m = map[blockIdx.x];                                                      \
    const MarchArgs& a = tab[m.x];                                                        \
    const int strips = (a.nx + kStrip - 1) / kStrip;                                      \
    march_strip<R, CORR, false>(a, (int)m.y % strips, (int)m.y / strips);                 \
  }
SBFS_MARCH_KERNEL(k_march, double, false, SBFS_FP64_WAVES)
SBFS_MARCH_KERNEL(k_march_corr, double, true, SBFS_FP64_WAVES)
SBFS_MARCH_KERNEL(k_march_mixed, float, false, SBFS_MIXED_WAVES)
SBFS_MARCH_KERNEL(k_march_mixed_corr, float, true, SBFS_MIXED_WAVES)
#undef SBFS_MARCH_KERNEL
// the FP64 stage kernels with streaming output stores (single cases whose
// fields the Infinity Cache cannot keep, stream_fields), and the FP32 ones for
// fields of 4 GiB or more
#define SBFS_MARCH_ALT_KERNEL(name, R, CORR, WAVES)                                       \
  __global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(WAVES))) void name( \
      const MarchArgs* __restrict__ args) {                                               \
    const MarchArgs& a = *args;                                                           \
    int bx, by;                                                                           \
    if (march_unit(a, bx, by)) march_strip<R, CORR, true>(a, bx, by);                     \
  }
SBFS_MARCH_ALT_KERNEL(k_march_nt, double, false, SBFS_FP64_WAVES)
SBFS_MARCH_ALT_KERNEL(k_march_corr_nt, double, true, SBFS_FP64_WAVES)
SBFS_MARCH_ALT_KERNEL(k_march_mixed_wide, float, false, SBFS_MIXED_WAVES)
SBFS_MARCH_ALT_KERNEL(k_march_mixed_corr_wide, float, true, SBFS_MIXED_WAVES)
#undef SBFS_MARCH_ALT_KERNEL

}  // namespace sbfs
