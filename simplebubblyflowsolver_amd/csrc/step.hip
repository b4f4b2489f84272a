// Time-step control (reference src/decide_dt.c), device diagnostics and the
// integrator (src/integrate.c).
#include <algorithm>
#include <cfloat>
#include <cmath>

#include "decide_dt.h"
#include "fluid_solver.h"
#include "integrate.h"
#include "interface_solver.h"
#include "sbfs.h"
#include "reduce.hpp"
#include "sbfs_internal.hpp"

namespace sbfs {

static const double kPiDt = 3.1415926535897932384626433832;  // decide_dt.c:16
static const double kDtMax = 1.;                              // decide_dt.c:25


// decide_dt in one launch: the advective limit, min over faces of
// h / (|u| + small) (decide_dt.c:49-64), and its combination with the other
// limits (:157-167).  A workgroup takes kRedThreads consecutive columns of `rows`
// rows, each thread one column, so the loads of a thread are independent and in
// flight together; its minimum m joins the others through an atomic, and the
// last workgroup writes dt to device memory, for the step's kernels, and to
// pinned host memory, for the caller.  (As a second launch and a copy queued after
// the step, the combination and the caller's dt cost 10 us of a 138 us step at
// 64 x 128.)  A min does not depend on the combination order.
// DtWord::key holds the largest ~bits(m): m is positive and no NaN, so its bits
// grow with it, and 0 is the identity.  A workgroup adds to the counter after
// its update of the key has returned, that is, has been performed where every XCD
// sees it, so the workgroup that counts the last sees every minimum, and returns
// both words to 0 for the next launch.  Updates of one address take about 10 ns
// each, one after another (k_dt of 2048 workgroups on one pair of words: 74 us at
// 2048 x 4096), so above kDtFlat workgroups they combine in kDtWords groups first,
// each on its own cache lines, and the last of each group in the first pair.
// (Stored partial minima with an acquire / release counter, whose cache
// write-backs and invalidations every workgroup pays, took 76 us there.)
template <int B, bool NT>
__device__ __forceinline__ double dt_column(const DtArgs& a, int i, int j0) {
  // The column's minimum of h / (|u| + small) is h over its largest
  // |u| + small, bit for bit: a correctly rounded quotient does not grow
  // with its divisor, so the largest divisor gives the smallest quotient
  // (and fmax passes over a NaN as fmin does).  One division per field
  // and thread instead of one per cell.
  const double small = 1.e-8;
  double mx = 0., my = 0.;
  // rows past ny repeat row ny (a repeated value leaves a max unchanged),
  // so the loads carry no branch and are all in flight together; with NT
  // they are streaming loads (read once; 124 -> 88 us at 4096 x 8192, see
  // stream_fields)
  auto ld = [](const double* p) {
    if constexpr (NT) return __builtin_nontemporal_load(p);
    else return *p;
  };
  for (int r0 = 0; r0 < a.rows; r0 += B) {
#pragma unroll
    for (int r = 0; r < B; r++) {
      const int j = min(j0 + r0 + r, a.ny);
      if (i >= 2) mx = fmax(mx, fabs(ld(a.ux + L::xf(i, j, a.nx))) + small);
      my = fmax(my, fabs(ld(a.uy + L::cc(i, j, a.nx))) + small);
    }
  }
  double m = kDtMax;
  if (i >= 2) m = fmin(m, a.hxxf[i - 1] / mx);
  return fmin(m, a.hy / my);
}

template <bool NT>
__device__ __forceinline__ void dt_body(const DtArgs& a, int bx, int by) {
  __shared__ double sh[kRedThreads / 64];
  double m = kDtMax;
  const int i = 1 + (int)(bx * kRedThreads + threadIdx.x);
  const int j0 = 1 + by * a.rows;
  if (i <= a.nx) m = a.rows >= 16 ? dt_column<16, NT>(a, i, j0) : dt_column<4, NT>(a, i, j0);
  m = block_reduce<0>(m, sh);
  if (threadIdx.x != 0) return;
  unsigned long long key = ~(unsigned long long)__double_as_longlong(m);
  // joins the key of `n` workgroups; true for the last, with the joined key
  auto join = [&key](DtWord* w, unsigned n) {
    unsigned long long old = __hip_atomic_fetch_max(&w->key, key, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    // (an empty statement that reads the update's return: the wait for it comes
    // here, before the counter's update, which stays behind the statement)
    asm volatile("" : "+v"(old)::"memory");
    if (__hip_atomic_fetch_add(&w->count, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) + 1u != n) return false;
    key = __hip_atomic_exchange(&w->key, 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __hip_atomic_store(&w->count, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    return true;
  };
  unsigned groups = (unsigned)a.nblk;
  if (groups > kDtFlat) {
    const unsigned g = (unsigned)(by * a.gx + bx) % kDtWords;
    if (!join(&a.slot->word[1 + g], (groups - g + kDtWords - 1) / kDtWords)) return;
    groups = kDtWords;
  }
  if (!join(&a.slot->word[0], groups)) return;
  double r = __longlong_as_double((long long)~key) * a.cadv;
  r = fmin(r, a.dif0);
  r = fmin(r, a.dif1);
  r = fmin(r, a.dint);
  a.slot->dt = r;
  __hip_atomic_store(a.host, r, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

template <bool NT>
__global__ __launch_bounds__(kRedThreads) void k_dt(DtArgs a) {
  dt_body<NT>(a, blockIdx.x, blockIdx.y);
}

// ensembles: one map entry (case, local block) per workgroup
__global__ __launch_bounds__(kRedThreads) void k_dt_batch(const DtArgs* __restrict__ tab,
                                                         const uint2* __restrict__ map) {
  const uint2 m = map[blockIdx.x];
  const DtArgs& a = tab[m.x];
  dt_body<false>(a, (int)(m.y % a.gx), (int)(m.y / a.gx));
}

// grid-only limits (decide_dt.c:79-130); host arithmetic identical to the
// reference, including pow(h, 3.) from libm
void dt_limits(const domain_t* d, const fluid_t* f, const interface_t* s, double* dif0,
               double* dif1, double* dint) {
  const Options& o = options();
  const size_t nx = d->mysizes[0];
  double gs[2] = {DBL_MAX, d->hy};
  for (size_t i = 2; i <= nx; i++) gs[0] = fmin(gs[0], d->hxxf[i - 1]);
  const double diffusivity = 1. / f->Re;
  double dif[2];
  for (int k = 0; k < 2; k++) {
    dif[k] = fmin(1., f->denr / f->visr) / diffusivity * 0.5 / 2. * (gs[k] * gs[k]);
    dif[k] *= o.cdif;
  }
  const double tension = 1. / s->We;
  double di = kDtMax;
  for (int k = 0; k < 2; k++) di = fmin(di, sqrt(1. / tension / 4. / kPiDt * pow(gs[k], 3.)));
  di *= o.cint;
  *dif0 = dif[0];
  *dif1 = dif[1];
  *dint = di;
}

// the arguments of one case's decide_dt, into `slot` and the pinned `host`.
// Rows per workgroup: 4, doubled to at most 64 while the workgroups are more than
// 2048, eight per CU (4096 x 8192: 90 us against 100 with at most 16 rows).
int dt_args(const domain_t* d, const DomainCtx* c, const fluid_t* f, const interface_t* s, DtSlot* slot, double* host,
            DtArgs* a) {
  if (load_dt_coefs()) return 1;
  dt_limits(d, f, s, &a->dif0, &a->dif1, &a->dint);
  a->ux = (const double*)f->ux.data;
  a->uy = (const double*)f->uy.data;
  a->hxxf = c->hxxf;
  a->hy = c->hy;
  a->cadv = options().cadv;
  a->slot = slot;
  a->host = host;
  a->nx = (int)c->nx;
  a->ny = (int)c->ny;
  a->gx = (int)cdiv(a->nx, kRedThreads);
  SBFS_REQUIRE(a->gx <= kDtMaxGx, "decide_dt: %d columns, more than %d", a->nx, kDtMaxGx * kRedThreads);
  a->rows = 4;
  while (a->gx * cdiv(a->ny, a->rows) > 2048 && a->rows < 64) a->rows *= 2;
  a->nblk = a->gx * (int)cdiv(a->ny, a->rows);
  return 0;
}

int dt_launch(const DtArgs& a) {
  const dim3 grd(a.gx, cdiv(a.ny, a.rows));
  SBFS_TIMED("k_dt", hipLaunchKernelGGL((stream_fields(a.nx, a.ny) ? k_dt<true> : k_dt<false>), grd, dim3(kRedThreads),
                                        0, stream(), a));
  return check_launch("decide_dt");
}

// dt into the domain's own slot, c->dt->dt, and, after the stream is
// synchronised, *dt_host(c)
int compute_dt_device(const domain_t* d, DomainCtx* c, const fluid_t* f,
                      const interface_t* s) {
  DtArgs a;
  if (dt_args(d, c, f, s, c->dt, dt_host(c), &a)) return 1;
  return dt_launch(a);
}

// ---------------------------------------------------------------------------
// diagnostics: volume, centroid, rise velocity, max |div|, vof extrema, area
// ---------------------------------------------------------------------------
// The workgroup's five sums, minimum and two maxima, in block_reduce's order, with
// the eight quantities' exchanges in flight together and one barrier.
// (valid in the first thread)
__device__ __forceinline__ void diag_reduce(double (&q)[8]) {
  __shared__ double sh[kRedThreads / 64][8];
  auto join = [](int k, double a, double b) { return k < 5 ? a + b : k == 5 ? fmin(a, b) : fmax(a, b); };
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    double x[8];
#pragma unroll
    for (int k = 0; k < 8; k++) x[k] = __shfl_xor(q[k], o, 64);
#pragma unroll
    for (int k = 0; k < 8; k++) q[k] = join(k, q[k], x[k]);
  }
  if ((threadIdx.x & 63) == 0)
#pragma unroll
    for (int k = 0; k < 8; k++) sh[threadIdx.x >> 6][k] = q[k];
  __syncthreads();
#pragma unroll
  for (int w = 1; w < kRedThreads / 64; w++)
#pragma unroll
    for (int k = 0; k < 8; k++) q[k] = join(k, q[k], sh[w][k]);
}

// A thread takes a column of `rows` rows: the column's quotients are formed once
// and the row below is kept from the step before.  With the cells dealt out in
// turn, each paid two 64-bit divisions for its indices and six FP64 ones, and the
// eight reductions ran one after another: sbfs_diagnostics 47.6 -> 30.9 us at
// 1024 x 2048, 105 -> 51 at 2048 x 4096 (their fields read once: 10 and 39 us),
// 23.4 -> 19.9 at 64 x 128, the launches, the wait and the call.  Four rows at least:
// eight took 21.0 there, sixteen 22.8.
__global__ __launch_bounds__(kRedThreads) void k_diag_partial(
    const double* __restrict__ vof, const double* __restrict__ ux, const double* __restrict__ uy,
    const double* __restrict__ xc, const double* __restrict__ hxxf, const double* __restrict__ jdxf,
    const double* __restrict__ jdxc, double hy, int nx, int ny, int rows, double* __restrict__ part) {
  double vol = 0., sds = 0., xm = 0., um = 0., area = 0.;
  double vmin = 1., vmax = 0., dmax = 0.;
  const int j0 = 1 + (int)blockIdx.y * rows, j1 = min(ny, j0 + rows - 1);
  for (int i = 1 + (int)(blockIdx.x * kRedThreads + threadIdx.x); i <= nx; i += (int)gridDim.x * kRedThreads) {
    const double ds = jdxc[i - 1], x = xc[i];
    const double fm = jdxf[i - 1] / hxxf[i - 1], fp = jdxf[i] / hxxf[i], fy = ds / hy, rj = 1. / ds;
    double vb = vof[L::vof(i, j0 - 1, nx)], uyb = uy[L::cc(i, j0, nx)];
#pragma unroll 4
    for (int j = j0; j <= j1; j++) {
      const double lv = vof[L::vof(i, j, nx)], vl = vof[L::vof(i - 1, j, nx)];
      const double uxm = ux[L::xf(i, j, nx)], uxp = ux[L::xf(i + 1, j, nx)], uyt = uy[L::cc(i, j + 1, nx)];
      vmin = fmin(vmin, lv);
      vmax = fmax(vmax, lv);
      vol += lv * ds;
      sds += ds;
      xm += lv * x * ds;
      um += lv * (0.5 * uxm + 0.5 * uxp) * ds;
      // x and y face area terms, src/logging/interface.c:121-127
      area += fabs(lv - vl) * fm;
      area += fabs(lv - vb) * fy;
      if (i == nx) area += fabs(vof[L::vof(nx + 1, j, nx)] - lv) * fp;
      // src/logging/divergence.c:44-58
      const double div = rj * (-fm * uxm + fp * uxp - fy * uyb + fy * uyt);
      dmax = fmax(dmax, fabs(div));
      vb = lv;
      uyb = uyt;
    }
  }
  double q[8] = {vol, sds, xm, um, area, vmin, vmax, dmax};
  diag_reduce(q);
  if (threadIdx.x == 0)
#pragma unroll
    for (int k = 0; k < 8; k++) part[8 * (blockIdx.y * gridDim.x + blockIdx.x) + k] = q[k];
}

__global__ __launch_bounds__(kRedThreads) void k_diag_final(const double* __restrict__ part, int n,
                                                            double* __restrict__ out) {
  double r[8] = {0., 0., 0., 0., 0., 1., 0., 0.};
#pragma unroll 4
  for (int k = threadIdx.x; k < n; k += kRedThreads) {
#pragma unroll
    for (int q = 0; q < 5; q++) r[q] += part[8 * k + q];
    r[5] = fmin(r[5], part[8 * k + 5]);
    r[6] = fmax(r[6], part[8 * k + 6]);
    r[7] = fmax(r[7], part[8 * k + 7]);
  }
  diag_reduce(r);
  if (threadIdx.x == 0) {
    const double vol = r[0];
    out[0] = vol;
    out[1] = vol != 0. ? r[2] / vol : 0.;
    out[2] = vol != 0. ? r[3] / vol : 0.;
    out[3] = r[7];
    out[4] = r[5];
    out[5] = r[6];
    out[6] = vol / r[1];
    out[7] = r[4];
  }
}

// ---------------------------------------------------------------------------
// staged integrator: the reference's composition, stage by stage
// ---------------------------------------------------------------------------
static int integrate_staged(const domain_t* domain, fluid_t* fluid, interface_t* interface,
                            double* dt) {
  if (decide_dt(domain, fluid, interface, dt)) return 1;
  for (size_t k = 0; k < 3; k++) {
    if (fluid_compute_density(domain, fluid, interface, 0)) return 1;
    if (fluid_compute_viscosity(domain, fluid, interface)) return 1;
    if (interface_compute_curvature_tensor(domain, interface)) return 1;
    if (interface_compute_force(domain, fluid, interface)) return 1;
    if (interface_update_vof(domain, k, *dt, fluid, interface)) return 1;
    if (fluid_compute_density(domain, fluid, interface, 1)) return 1;
    if (interface_compute_mass_flux(domain, fluid, interface)) return 1;
    if (fluid_predict_field(domain, k, *dt, fluid, interface)) return 1;
    const double dt_old = rk((k + 2) % 3).g * (*dt);
    const double dt_new = rk(k).g * (*dt);
    if (fluid_compute_potential(domain, dt_old, dt_new, fluid)) return 1;
    if (fluid_correct_velocity(domain, dt_old, dt_new, fluid)) return 1;
    if (fluid_update_pressure(domain, fluid)) return 1;
  }
  return 0;
}

int integrate_fused(const domain_t* domain, fluid_t* fluid, interface_t* interface, double* dt);

}  // namespace sbfs

using namespace sbfs;

extern "C" {

int decide_dt(const domain_t* domain, const fluid_t* fluid, const interface_t* interface,
              double* dt) {
  DomainCtx* c = domain_ctx(domain);
  if (!c) return 1;
  SBFS_REQUIRE(dt != nullptr, "decide_dt: null dt");
  if (check_array(domain, &fluid->ux, NA_UX, 8, "ux")) return 1;
  if (check_array(domain, &fluid->uy, NA_UY, 8, "uy")) return 1;
  if (compute_dt_device(domain, c, fluid, interface)) return 1;
  SBFS_HIP(hipStreamSynchronize(stream()));
  *dt = *dt_host(c);
  return 0;
}

int integrate(const domain_t* domain, fluid_t* fluid, interface_t* interface, double* dt) {
  if (init_runtime()) return 1;
  SBFS_REQUIRE(domain && fluid && interface && dt, "integrate: null argument");
  if (options().path == SBFS_PATH_FUSED) {
    if (options().precision == SBFS_PRECISION_MIXED ||
        fp64_march_addressable(domain->mysizes[0], domain->mysizes[1]))
      return integrate_fused(domain, fluid, interface, dt);
    // fields of 4 GiB or more: the FP64 step runs on the staged path
    SBFS_REQUIRE(options().curvature != SBFS_CURVATURE_LEARNED,
                 "integrate: the learned curvature runs on the fused path, whose FP64 step needs fields below 4 GiB "
                 "(%zu x %zu cells); use mixed precision", domain->mysizes[0], domain->mysizes[1]);
  }
  return integrate_staged(domain, fluid, interface, dt);
}

int sbfs_diagnostics(const domain_t* domain, const fluid_t* fluid, const interface_t* interface,
                     double out[SBFS_NDIAG]) {
  DomainCtx* c = domain_ctx(domain);
  if (!c) return 1;
  if (check_array(domain, &fluid->ux, NA_UX, 8, "ux")) return 1;
  if (check_array(domain, &fluid->uy, NA_UY, 8, "uy")) return 1;
  if (check_array(domain, &interface->vof, NA_VOF, 8, "vof")) return 1;
  const int nx = (int)c->nx, ny = (int)c->ny;
  const int gx = std::min<int>(kRedBlocks, cdiv(nx, kRedThreads));
  const int rows = std::max<int>(4, cdiv(ny, kRedBlocks / gx)), gy = cdiv(ny, rows), nblk = gx * gy;
  hipLaunchKernelGGL(k_diag_partial, dim3(gx, gy), dim3(kRedThreads), 0, stream(),
                     (const double*)interface->vof.data, (const double*)fluid->ux.data,
                     (const double*)fluid->uy.data, c->xc, c->hxxf, c->jdxf, c->jdxc, c->hy, nx,
                     ny, rows, c->red);
  // (into pinned host memory: no copy behind it)
  hipLaunchKernelGGL(k_diag_final, dim3(1), dim3(kRedThreads), 0, stream(), (const double*)c->red,
                     nblk, c->host_pin);
  if (check_launch("sbfs_diagnostics")) return 1;
  SBFS_HIP(hipStreamSynchronize(stream()));
  for (int k = 0; k < SBFS_NDIAG; k++) out[k] = c->host_pin[k];
  return 0;
}

}  // extern "C"
