// Fused integrator: per Runge-Kutta stage
//
//   k_march*     the marching stage kernel (march.hip): every stage of the
//                reference from fluid_compute_density to
//                fluid_predict_field and the Poisson right-hand side, one
//                wavefront per strip of columns walking a band of rows;
//                from stage 1 on it also applies the previous stage's
//                projection and pressure update (k_march*_corr)
//   k_dct2_rows  DCT-II per row of the right-hand side
//   k_part_*     partitioned tridiagonal solve (tdm_partition.hip)
//   k_dct3_psi   DCT-III per row -> psi[1]
//   k_post       projection of u and the pressure update of the last stage
//
// Every value is computed with the same device functions and operation
// order as the staged kernels (stencils.hpp), so the fused path reproduces
// the staged path bitwise.  dt stays in device memory for the whole step.
#include <cfloat>
#include <cmath>
#include <cstdint>
#include <cstdlib>
#include <cstring>
#include <vector>

#include "decide_dt.h"
#include "fluid_solver.h"
#include "integrate.h"
#include "interface_solver.h"
#include "march.hpp"
#include "poisson.hpp"
#include "sbfs.h"
#include "sbfs_internal.hpp"
#include "scratch_pool.hpp"
#include "stencils.hpp"

namespace sbfs {

// Per-column quotients of the metrics (struct Coef, march.hpp), each
// evaluated on the host with the expression (and so the rounding) the
// reference uses inside its loops:
//   rhf = 1./HXXF  rhc = 1./HXXC  rjf = 1./JDXF  rjc = 1./JDXC
//   qf  = JDXF/HXXF   qc = JDXC/HXXC   eqf = 0.5*JDXF/HXXF
//   ecy = 0.5*JDXC/hy  cyc = JDXC/hy  cyf = JDXF/hy
//   dfx = (1/Re)/JDXF  dcx = (1/Re)/JDXC
// Indexed by the 1-based column i.  Multiplying by a stored quotient gives
// the same bits as the reference's left-to-right `a / b * x`, so the fused
// kernels keep bitwise parity while only data-dependent divisions remain.

// ---------------------------------------------------------------------------
// projection + pressure (correct_velocity/ux.c, uy.c; update_pressure.c)
// ---------------------------------------------------------------------------
// Column i = 0..nx+1, rows j0 .. j0 + kPostRows - 1 (up to ny) of one
// thread: the quotients that depend on the column or on nothing are formed
// once per thread, and the potentials and the density of row j - 1 come from
// the previous row.  Every cell's expressions are those of the reference
// (left to right, the same roundings), so the rows a thread takes do not
// change a bit.  O: the type of the element offsets (32 bits while every
// field stays below 4 GiB, so the loads take a scalar base and a 32-bit
// offset).

template <typename O>
__device__ __forceinline__ double post_ld(const double* f, O e) {
  using G = __attribute__((address_space(1))) const char;
  return *(const double*)((G*)f + e * (O)sizeof(double));
}
// (with NT, streaming stores: the velocities and the pressure are read again
// only by the next step; 487 -> 463 us at 4096 x 8192, see stream_fields)
template <typename O, bool NT>
__device__ __forceinline__ void post_st(double* f, O e, double v) {
  using G = __attribute__((address_space(1))) char;
  auto* q = (__attribute__((address_space(1))) double*)((G*)f + e * (O)sizeof(double));
  if constexpr (NT) __builtin_nontemporal_store(v, q);
  else *q = v;
}

// rows j0 .. j0 + N - 1 of column i; with All every load is issued before
// the first row's arithmetic (the full tiles), otherwise row by row
template <typename O, int N, bool All, bool NT>
__device__ __forceinline__ void post_column(const PostArgs& a, int i, int j0, int nj) {
  const int nx = a.nx, ny = a.ny;
  const double dt = *a.dt;
  const double dtn = a.g_new * dt;
  const double dto = a.g_old * dt;
  const double coef = -1. / dtn * dto;
  // dtn / a.refden / h * dpsi is ((dtn / refden) / h) * dpsi, and
  // dtn * coef * (1 / d - 1 / refden) / h * dpsi is
  // (((dtn coef) (1 / d - 1 / refden)) / h) * dpsi
  const double dtr = dtn / a.refden, cdc = dtn * coef, rr = 1. / a.refden;
  const bool fx = i >= 2 && i <= nx;  // an interior x face
  const bool cin = i >= 1 && i <= nx;  // an interior cell column
  const double h = fx ? a.hxxf[i - 1] : 1.;
  const double qx = dtr / h, qy = dtr / a.hy;
  const O wc = (O)nx + 2, wf = (O)nx + 1;
  // element offsets of (i, j0 - 1): cc and xf layouts (L::cc, L::xf); the
  // vof of cell (i, j) is at its cc offset + wc (L::vof)
  const O oc0 = (O)(j0 - 1) * wc + (O)i;
  const O ox0 = (O)(j0 - 1) * wf + (O)(i - 1);
  // potentials and vof of rows j0 - 1 .. j0 + N - 1 in this column (k = row
  // - j0 + 1), and the inputs of rows j0 .. j0 + N - 1
  double p1[N + 1] = {}, p0[N + 1] = {}, vf[N + 1] = {};
  double p1l[N] = {}, p0l[N] = {}, vfl[N] = {}, us[N] = {}, vs[N] = {}, pp[N] = {};
  auto load_row = [&](int k) {
    const O oc = oc0 + (O)k * wc;
    if (cin) {
      p1[k] = post_ld(a.psi1, oc);
      p0[k] = post_ld(a.psi0, oc);
      vf[k] = post_ld(a.vofn, oc + wc);
    }
    if (k == 0) return;
    if (fx) {
      p1l[k - 1] = post_ld(a.psi1, oc - 1);
      p0l[k - 1] = post_ld(a.psi0, oc - 1);
      vfl[k - 1] = post_ld(a.vofn, oc + wc - 1);
      us[k - 1] = post_ld(a.uxs, ox0 + (O)k * wf);
    }
    if (cin) {
      vs[k - 1] = post_ld(a.uys, oc);
      pp[k - 1] = post_ld(a.p, oc);
    }
  };
  if (All) {
#pragma unroll
    for (int k = 0; k <= N; k++) load_row(k);
  } else {
    load_row(0);
  }
  double du = cin ? mix_clamp(a.denr, a.dlo, a.dhi, vf[0]) : 0.;
#pragma unroll
  for (int r = 0; r < N; r++) {
    if (!All) {
      if (r >= nj) break;
      load_row(r + 1);
    }
    const int j = j0 + r;
    const O oc = oc0 + (O)(r + 1) * wc, ox = ox0 + (O)(r + 1) * wf;
    const double d = cin ? mix_clamp(a.denr, a.dlo, a.dhi, vf[r + 1]) : 0.;
    if (i >= 1) {
      double u = 0.;
      if (fx) {
        u = us[r];
        u -= qx * (-p1l[r] + p1[r + 1]);
        const double dd = 0.5 * mix_clamp(a.denr, a.dlo, a.dhi, vfl[r]) + 0.5 * d;
        u += cdc * (1. / dd - rr) / h * (-p0l[r] + p0[r + 1]);
      }
      post_st<O, NT>(a.ux, ox, u);
      if (j > ny - 1) post_st<O, NT>(a.ux, ox - (O)ny * wf, u);
      if (j <= 1) post_st<O, NT>(a.ux, ox + (O)ny * wf, u);
    }
    {
      double u;
      if (i == 0) u = kUyXm;
      else if (i == nx + 1) u = kUyXp;
      else {
        u = vs[r];
        u -= qy * (-p1[r] + p1[r + 1]);
        const double dd = 0.5 * du + 0.5 * d;
        u += cdc * (1. / dd - rr) / a.hy * (-p0[r] + p0[r + 1]);
      }
      post_st<O, NT>(a.uy, oc, u);
      if (j > ny - 1) post_st<O, NT>(a.uy, oc - (O)ny * wc, u);
      if (j <= 1) post_st<O, NT>(a.uy, oc + (O)ny * wc, u);
    }
    if (cin) {
      const double v = pp[r] + p1[r + 1];
      auto put = [&](O o) {
        post_st<O, NT>(a.p, o, v);
        if (j > ny - 1) post_st<O, NT>(a.p, o - (O)ny * wc, v);
        if (j <= 1) post_st<O, NT>(a.p, o + (O)ny * wc, v);
      };
      put(oc);
      if (i == 1) put(oc - 1);
      if (i == nx) put(oc + 1);
    }
    du = d;
  }
}

template <typename O, bool NT>
__device__ __forceinline__ void post_rows(const PostArgs& a, int i, int j0) {
  if (i > a.nx + 1 || j0 > a.ny) return;
  const int nj = min(kPostRows, a.ny - j0 + 1);
  if (nj == kPostRows) post_column<O, kPostRows, true, NT>(a, i, j0, nj);
  else post_column<O, kPostRows, false, NT>(a, i, j0, nj);
}

// tiles of 64 columns x 4 kPostRows rows, a thread per column and kPostRows rows
template <typename O, bool NT>
__global__ __launch_bounds__(256) void k_post(PostArgs a) {
  post_rows<O, NT>(a, (int)(blockIdx.x * 64 + threadIdx.x), 1 + (int)(blockIdx.y * 4 + threadIdx.y) * kPostRows);
}

// one tile per map entry (case, local tile); ensemble fields stay below 4 GiB
__global__ __launch_bounds__(256) void k_post_batch(const PostArgs* __restrict__ tab, const uint2* __restrict__ map) {
  const uint2 m = map[blockIdx.x];
  const PostArgs& a = tab[m.x];
  const int gx = (a.nx + 2 + 63) / 64;
  post_rows<unsigned, false>(a, (int)((m.y % gx) * 64 + threadIdx.x),
                      1 + (int)((m.y / gx) * 4 + threadIdx.y) * kPostRows);
}

// ---------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------
struct CoefTables {
  double re = 0.;
  double* buf = nullptr;
  Coef cf{};
};

// A step graph's key, and the state it leaves
struct StepKey {
  std::vector<uint64_t> v;
  bool operator==(const StepKey& o) const { return v == o.v; }
};

constexpr int kStateArrays = 17;
struct StepGraph {
  StepKey key;
  hipGraphExec_t exec = nullptr;
  // state pointers after the step, then the scratch vof and pressure, which
  // a step swaps with the state's (the pressure once per step)
  void* after[kStateArrays + 2] = {};
  uint64_t last_use = 0;
};

// Everything the fused step keeps from one step of a domain to the next, owned
// by the domain's context: scratch, coefficient tables, the stage kernels'
// arguments in device memory and the captured steps.  One set per process made
// every step of a program that advances several cases in turn rebuild the
// tables (a synchronisation, a hipFree and a hipMalloc) and launch eagerly, the
// two graphs having been captured for other cases: 294 us per step for three
// 64 x 128 bubbles in turn against 233 for one, 1946 against 1544 for three
// 2048 x 4096 swarms.  A step has two pointer states, so four graphs serve
// two fluids on one domain.
struct ArgsSlot {
  MarchArgs host;
  MarchArgs* dev;
};
constexpr int kStepGraphs = 4;
constexpr size_t kMaxArgSlots = 64;
struct FusedState {
  FusedScratch scr;
  CoefTables coef;
  std::vector<ArgsSlot> args;
  MarchArgs* args_dev = nullptr;  // kMaxArgSlots
  StepGraph graph[kStepGraphs];
  StepKey seen[kStepGraphs];
  uint64_t clock = 0;
};

struct DeviceMemory {
  static int alloc(void** p, size_t bytes) {
    const hipError_t e = hipMalloc(p, bytes);
    if (e != hipSuccess) {
      *p = nullptr;
      (void)hipGetLastError();  // (a later launch check would report it)
    }
    return e;
  }
  static void free(void* p) { (void)hipFree(p); }
  static int zero(void* p, size_t bytes) { return hipMemsetAsync(p, 0, bytes, stream()); }
};
static ScratchPool<DeviceMemory> g_pool;

hipError_t device_malloc_bytes(void** p, size_t bytes) { return (hipError_t)g_pool.alloc(p, bytes); }

// (the caller has synchronised the stream)
void fused_destroy(FusedState* s) {
  if (!s) return;
  for (StepGraph& g : s->graph)
    if (g.exec) (void)hipGraphExecDestroy(g.exec);
  (void)hipFree(s->coef.buf);
  (void)hipFree(s->args_dev);
  g_pool.put(s->scr);
  delete s;
}

static int scratch(DomainCtx* c, const interface_t* s, const fluid_t* f, bool learned) {
  FusedScratch& scr = c->fused->scr;
  const size_t cells = c->nx * c->ny;
  if (!scr.vof)
    SBFS_HIP((hipError_t)g_pool.get(
        {c->nx, c->ny, f->ux.datasize, f->uy.datasize, f->p.datasize, s->vof.datasize}, learned, &scr));
  if (learned && !scr.cut) {
    // (what a failed call here allocated stays in the set)
    auto part = [&scr](auto** p, size_t bytes) -> int {
      if (*p) return 0;
      SBFS_HIP(device_malloc(p, bytes));
      scr.bytes += bytes;
      return 0;
    };
    if (part(&scr.kappa, sizeof(float) * cells)) return 1;
    for (unsigned*& l : scr.klist)
      if (part(&l, sizeof(unsigned) * (cells + 1))) return 1;
    if (curv_field_init(scr.kappa, scr.klist, 3, (long)cells, stream())) return 1;
    scr.klast = -1;
    if (part(&scr.cut, sizeof(unsigned long long) * c->ny * march_strips((int)c->nx))) return 1;
  }
  return 0;
}

// weight and order buffers for n units (zero weights at first: any order)
static int order_buffers(DomainCtx* c, int n) {
  FusedScratch& scr = c->fused->scr;
  if (scr.units >= n) return 0;
  (void)hipStreamSynchronize(stream());
  c->epoch++;
  (void)hipFree(scr.weight);
  (void)hipFree(scr.order);
  scr.weight = scr.order = nullptr;
  scr.units = 0;
  SBFS_HIP(device_malloc(&scr.weight, sizeof(unsigned) * (size_t)n));
  SBFS_HIP(device_malloc(&scr.order, sizeof(unsigned) * (size_t)n));
  SBFS_HIP(hipMemsetAsync(scr.weight, 0, sizeof(unsigned) * (size_t)n, stream()));
  scr.units = n;
  return 0;
}

// the 14 per-column quotient tables of one domain and Re in a new device
// buffer (*buf, owned by the caller)
int coef_build(const domain_t* d, double Re, double** buf, Coef* out) {
  const size_t nx = d->mysizes[0], w = nx + 2;
  std::vector<double> h(14 * w, 0.);
  double* t[14];
  for (int k = 0; k < 14; k++) t[k] = h.data() + k * w;
  const double hy = d->hy;
  const double diffusivity = 1. / Re;
  for (size_t i = 1; i <= nx + 1; i++) {
    const double hf = d->hxxf[i - 1], jf = d->jdxf[i - 1];
    t[0][i] = 1. / hf;
    t[2][i] = 1. / jf;
    t[4][i] = jf / hf;
    t[6][i] = 0.5 * jf / hf;
    t[9][i] = jf / hy;
    t[10][i] = diffusivity / jf;
    t[12][i] = hf;
  }
  for (size_t i = 1; i <= nx; i++) {
    const double hc = d->hxxc[i - 1], jc = d->jdxc[i - 1];
    t[1][i] = 1. / hc;
    t[3][i] = 1. / jc;
    t[5][i] = jc / hc;
    t[7][i] = 0.5 * jc / hy;
    t[8][i] = jc / hy;
    t[11][i] = diffusivity / jc;
    t[13][i] = hc;
  }
  SBFS_HIP(device_malloc(buf, sizeof(double) * h.size()));
  SBFS_HIP(hipMemcpy(*buf, h.data(), sizeof(double) * h.size(), hipMemcpyHostToDevice));
  const double* b = *buf;
  Coef cf;
  cf.rhf = b + 0 * w;
  cf.rhc = b + 1 * w;
  cf.rjf = b + 2 * w;
  cf.rjc = b + 3 * w;
  cf.qf = b + 4 * w;
  cf.qc = b + 5 * w;
  cf.eqf = b + 6 * w;
  cf.ecy = b + 7 * w;
  cf.cyc = b + 8 * w;
  cf.cyf = b + 9 * w;
  cf.dfx = b + 10 * w;
  cf.dcx = b + 11 * w;
  cf.hxxf1 = b + 12 * w;
  cf.hxxc1 = b + 13 * w;
  cf.rhy = 1. / hy;
  *out = cf;
  return 0;
}

static int coef_tables(const domain_t* d, DomainCtx* c, double Re, Coef* out) {
  CoefTables& t = c->fused->coef;
  if (!t.buf || t.re != Re) {
    (void)hipStreamSynchronize(stream());
    c->epoch++;
    (void)hipFree(t.buf);
    t.buf = nullptr;
    if (coef_build(d, Re, &t.buf, &t.cf)) return 1;
    t.re = Re;
  }
  *out = t.cf;
  return 0;
}

int poisson_transform_fused(const domain_t* d, DomainCtx* c, fluid_t* f, double** rhs);  // poisson.hip

 // poisson.hip

#define D(a) ((double*)(a).data)

static void swap_data(array_t& x, array_t& y) {
  void* t = x.data;
  x.data = y.data;
  y.data = t;
}

__global__ void k_march(const MarchArgs* a);             // march.hip, plain FP64
__global__ void k_march_corr(const MarchArgs* a);        // + the previous stage's projection
__global__ void k_march_nt(const MarchArgs* a);          // k_march with streaming output stores
__global__ void k_march_corr_nt(const MarchArgs* a);     // k_march_corr with streaming output stores
__global__ void k_march_mixed(const MarchArgs* a);       // FP32 stencils
__global__ void k_march_mixed_corr(const MarchArgs* a);  // FP32 stencils + projection
__global__ void k_march_mixed_wide(const MarchArgs* a);       // k_march_mixed, fields of 4 GiB or more
__global__ void k_march_mixed_corr_wide(const MarchArgs* a);  // k_march_mixed_corr, fields of 4 GiB or more

// Stages 1 and 2 fold the previous stage's projection and pressure update
// into their stage kernel (k_march_corr), which reads the predicted velocity,
// both potentials and the pressure, corrects each row as it enters its rings
// and writes the new pressure; only the last stage keeps its k_post.
// SBFS_MARCH_FOLD=0 runs k_post after every stage instead.
static bool march_fold() {
  static int on = -1;
  if (on < 0) {
    const char* e = getenv("SBFS_MARCH_FOLD");
    on = (e && e[0] == '0') ? 0 : 1;
  }
  return on == 1;
}

// Whether the stage kernels run their units heaviest first (k_march_order):
// with several rounds of bands, the FP64 default.  SBFS_MARCH_ORDER=0 keeps
// the grid's own order, =1 orders the FP32 kernels too.
static bool march_ordered(bool mixed) {
  const char* e = getenv("SBFS_MARCH_ORDER");
  if (e && e[0] == '0') return false;
  if (e && e[0] == '1') return true;
  return !mixed;
}

// The tile height of the small grids' stage kernel (tile.hip), 0 for the
// marching kernel.  The short tile while its workgroups all run at once (two per
// CU, 512: 256 x 256 has 430, 256 x 512 would take 855 and is faster with 235
// tall ones, 63 against 74 us per step).  The tall one for up to four rounds of
// one per CU in FP64 and two and a half in mixed precision, where the marching
// kernel's lower redundancy catches up (512 x 1024, 846 tall tiles: 153 against
// 173 us in FP64, 129 against 128 mixed; 1024 x 1024, 1692: 260 against 241 and
// 218 against 179).  SBFS_MARCH_TILE=0 takes the marching kernel, =3 or =11 the
// tile of that height (the results are bitwise the same).
int tile_rows(unsigned short_groups, unsigned tall_groups, bool mixed) {
  if (const char* e = getenv("SBFS_MARCH_TILE")) {
    const int h = atoi(e);
    return h == kTileShort || h == kTileTall ? h : 0;
  }
  if (short_groups <= 512) return kTileShort;
  return tall_groups <= (mixed ? 640u : 1024u) ? kTileTall : 0;
}
static int tile_rows(int nx, int ny, bool mixed) {
  if (!fp64_march_addressable(nx, ny) || (mixed && mixed_march_wide(nx, ny))) return 0;
  return tile_rows(tile_groups(nx, ny, kTileShort), tile_groups(nx, ny, kTileTall), mixed);
}

// Rows per band of k_march.  Every wavefront marches its band plus kWarm + 2
// rows of ring fill, and a wavefront lives for the whole band, so the grid
// is sized in rounds of the device: multiples of the resident wavefront
// slots per strip (occupancy x CUs), each band as short as that allows.  In
// the grid's own order a partial last round would leave most SIMDs idle
// while it runs, so the rounds are whole.
// The FP64 bodies take about twice as long over a row with interface cells
// (the THINC flux's tanh and log), so in a single round the bands a bubble
// crosses finish last, 1.5x after the mean wavefront.  Several rounds let
// the dispatcher balance them, for more ring fill: 1.75 rounds when the
// units run heaviest first (k_march_order; the partial last round holds the
// lightest units), three in the grid's own order.  Measured on the 2048 x
// 4096 swarm, k_march / k_march_corr: 397 / 522 us for one round, 363 / 510
// for three unordered, 304 / 404 for two ordered and 289 / 398 for 1.75
// ordered (band 41; 2.4 and 1.5 rounds were slower).  The FP32 bodies'
// cheaper fluxes leave less to balance: one round is fastest for them while
// its bands are short (48 rows on the 2048 x 4096 swarm), two when one round
// would give bands of 160 rows or more (4096 x 8192: 96-row bands, 6.16 ms
// per mixed step against 6.22 with 191 rows; 128 rows 6.32, ordered 6.47-7.0).
// Where a round has room for shorter bands, the ring fill costs more than the
// idle slots: 5 rows at least in mixed precision (512 x 1024, three stages: 4 rows
// 108 us, 5 rows 104, 6 rows 112).
// SBFS_MARCH_BAND overrides the choice.
static int march_band(int nx, int ny, bool mixed) {
  static long slots[2] = {0, 0};
  long& sl = slots[mixed ? 1 : 0];
  if (sl == 0) {
    int dev = 0, per_cu = 0;
    hipDeviceProp_t prop;
    SBFS_HIP(hipGetDevice(&dev));
    SBFS_HIP(hipGetDeviceProperties(&prop, dev));
    if (mixed) SBFS_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, k_march_mixed, 64, 0));
    else SBFS_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, k_march, 64, 0));
    sl = (long)(per_cu > 0 ? per_cu : 1) * prop.multiProcessorCount;
  }
  const long slots_now = sl;
  if (const char* e = getenv("SBFS_MARCH_BAND")) {
    const int b = atoi(e);
    if (b >= 1) return b < ny ? b : ny;
  }
  const long strips = (nx + kStrip - 1) / kStrip;
  // rounds of the device, in quarters
  long quarters = mixed ? 4 : (march_ordered(mixed) ? 7 : 12);
  long bands = quarters * slots_now / (4 * strips);
  if (bands < 1) bands = 1;
  if (mixed && !march_ordered(mixed) && (ny + bands - 1) / bands >= 160) {
    quarters = 8;
    bands = quarters * slots_now / (4 * strips);
  }
  long band = (ny + bands - 1) / bands;
  const long least = mixed ? 5 : 4;
  if (band < least) band = least;
  return (int)(band < ny ? band : ny);
}

// Arguments of stage k's stage kernel from the state's current pointers:
// with the fold (corr) it reads the previous stage's predicted velocity
// us/vs[k-1] and writes us/vs[k]; stage 2 writes the pressure after stage
// 1's update to p_out (stage 1 writes none, see MarchArgs::p_out).
static void fill_march(const domain_t* domain, const DomainCtx* c, const fluid_t* fluid,
                       const interface_t* interface, const Coef& cf, double* rhs, int band, int k, bool corr,
                       double* const us[3], double* const vs[3], double* vofn, double* p_out,
                       const double* dtp, MarchArgs& m) {
  const RK r = rk(k);
  m.vof = D(interface->vof);
  m.ux = corr ? us[k - 1] : D(fluid->ux);
  m.uy = corr ? vs[k - 1] : D(fluid->uy);
  m.p = D(fluid->p);
  m.psi0 = D(fluid->psi[0]);
  m.psi_old = corr ? D(fluid->psi[1]) : nullptr;
  // stage 1's updated pressure is formed again by stage 2 (p_twice), so
  // only stage 2 stores one
  m.p_out = corr && k == 2 ? p_out : nullptr;
  m.p_twice = corr && k == 2;
  m.pg_old = rk((k + 1) % 3).g;  // gammas of stage k-1's dt_old / dt_new
  m.pg_new = rk((k + 2) % 3).g;
  m.kappa = nullptr;
  m.kappa_n = nullptr;
  m.cut = nullptr;
  m.order = nullptr;
  m.weight = nullptr;
  m.srcb_vof = D(interface->src[1]);
  m.srcb_ux = D(fluid->srcux[1]);
  m.srcb_uy = D(fluid->srcuy[1]);
  m.vofn = vofn;
  m.uxs = us[k];
  m.uys = vs[k];
  m.rhs = rhs;
  // the alpha sources of the last stage are never read again (beta of
  // stage 0 is zero), so they are not written
  m.srca_vof = k < 2 ? D(interface->src[0]) : nullptr;
  m.srca_ux = k < 2 ? D(fluid->srcux[0]) : nullptr;
  m.srca_uy = k < 2 ? D(fluid->srcuy[0]) : nullptr;
  m.den1 = k == 2 ? D(fluid->den[1]) : nullptr;
  m.txy = k == 2 ? D(fluid->txy) : nullptr;
  m.hxxf1 = cf.hxxf1;
  m.hxxc1 = cf.hxxc1;
  m.cf = cf;
  m.hy = c->hy;
  m.denr = fluid->denr;
  m.dlo = fmin(1., fluid->denr);
  m.dhi = fmax(1., fluid->denr);
  m.visr = fluid->visr;
  m.vlo = fmin(1., fluid->visr);
  m.vhi = fmax(1., fluid->visr);
  m.refdeninv = 2. / (1. + fluid->denr);
  m.tension = 1. / interface->We;
  m.grav = -1. / fluid->Fr / fluid->Fr;
  m.refden = fluid->refden;
  m.norm = 2. * (double)domain->glsizes[0];
  m.dt = dtp;
  m.ca = r.a;
  m.cb = r.b;
  m.cg = r.g;
  m.g_old = rk((k + 2) % 3).g;
  m.g_new = r.g;
  m.stage = k;
  m.nx = (int)c->nx;
  m.ny = (int)c->ny;
  m.band = band;
}

// arguments of the projection after stage k (predicted velocity uxs / uys)
static void fill_post(const DomainCtx* c, const fluid_t* fluid, const interface_t* interface, double* uxs,
                      double* uys, const double* dtp, int k, PostArgs& q) {
  q.uxs = uxs;
  q.uys = uys;
  q.psi1 = D(fluid->psi[1]);
  q.psi0 = D(fluid->psi[0]);
  q.vofn = D(interface->vof);
  q.ux = D(fluid->ux);
  q.uy = D(fluid->uy);
  q.p = D(fluid->p);
  q.hxxf = c->hxxf;
  q.hy = c->hy;
  q.denr = fluid->denr;
  q.dlo = fmin(1., fluid->denr);
  q.dhi = fmax(1., fluid->denr);
  q.refden = fluid->refden;
  q.dt = dtp;
  q.g_new = rk(k).g;
  q.g_old = rk((k + 2) % 3).g;
  q.nx = (int)c->nx;
  q.ny = (int)c->ny;
}

// The stage kernels' arguments in device memory (the kernels read them
// through a pointer, march.hip).  A step configuration builds the same
// arguments at every step, so they sit in a small cache of the domain keyed by
// their bytes: the eager first pass of a configuration stores them with a
// one-workgroup kernel (no host synchronisation), and the graph captured on its
// second pass finds the same bytes and records only the pointer.
__global__ void k_store_args(MarchArgs m, MarchArgs* __restrict__ out) {
  static_assert(sizeof(MarchArgs) % 8 == 0, "copied by 8-byte words");
  const unsigned long long* s = (const unsigned long long*)&m;
  unsigned long long* d = (unsigned long long*)out;
  for (int k = threadIdx.x; k < (int)(sizeof(MarchArgs) / 8); k += blockDim.x) d[k] = s[k];
}

static int device_args(DomainCtx* c, const MarchArgs& m, const MarchArgs** out) {
  FusedState& s = *c->fused;
  for (const ArgsSlot& a : s.args)
    if (memcmp(&a.host, &m, sizeof(m)) == 0) {
      *out = a.dev;
      return 0;
    }
  hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
  SBFS_HIP(hipStreamIsCapturing(stream(), &cs));
  SBFS_REQUIRE(cs == hipStreamCaptureStatusNone,
               "integrate: stage arguments of a captured step were not prepared by its eager pass");
  if (!s.args_dev) SBFS_HIP(device_malloc(&s.args_dev, sizeof(MarchArgs) * kMaxArgSlots));
  if (s.args.size() >= kMaxArgSlots) {
    // captured graphs hold pointers to these slots: move the epoch so that
    // none of them replays (queued steps read them before the stores below)
    s.args.clear();
    c->epoch++;
  }
  MarchArgs* d = s.args_dev + s.args.size();
  hipLaunchKernelGGL(k_store_args, dim3(1), dim3(64), 0, stream(), m, d);
  if (check_launch("integrate: stage arguments")) return 1;
  s.args.push_back({m, d});
  *out = d;
  return 0;
}

// Every launch of one fused time step (decide_dt, then per Runge-Kutta stage
// the stage kernel, the Poisson solve and the projection) plus the host-side
// pointer swaps the reference performs.  No allocation and no host
// synchronisation, so the sequence can be captured into a graph.
static int fused_body(const domain_t* domain, DomainCtx* c, fluid_t* fluid, interface_t* interface,
                      const Coef& cf, double* rhs, int band, double learned_h) {
  FusedScratch& scr = c->fused->scr;
  const int nx = (int)c->nx, ny = (int)c->ny;
  // learned curvature of each stage's input vof: on the side stream, forked
  // after the kernel that wrote that vof and joined before the stage kernel
  // that reads kappa, so it overlaps the dt reduction (stage 0) or the
  // previous stage's Poisson solve; with per-launch timing it stays on the
  // library stream, right before the stage kernel
  const bool learned = learned_h > 0.;
  const bool overlap = learned && !prof_active();
  // (stages 1 and 2 list their cells from the previous stage kernel's
  // bitmask of the vof it wrote; stage 0 from the state's vof, which the
  // caller may have changed since the last step)
  auto cut_of = [&scr](int k) -> const unsigned long long* { return k > 0 ? scr.cut : nullptr; };
  // stage k lists into list k; the launch before it wrote list klast, and
  // the launch after it writes list (k + 1) % 3
  auto curv_launch = [&](int k, const double* vof, hipStream_t st) -> int {
    if (scr.klast == k) {
      // only after a step that stopped part way: start the field afresh
      if (curv_field_init(scr.kappa, scr.klist, 3, (long)nx * ny, st)) return 1;
      scr.klast = -1;
    }
    const unsigned* prev = scr.klast >= 0 ? scr.klist[scr.klast] : nullptr;
    if (curv_mlp_launch(vof, cut_of(k), scr.kappa, scr.klist[k], prev, scr.klist[(k + 1) % 3], nx, ny,
                        learned_h, st))
      return 1;
    scr.klast = k;
    return 0;
  };
  auto fork_curv = [&](int k, const double* vof) -> int {
    SBFS_HIP(hipEventRecord(fork_event(k), stream()));
    SBFS_HIP(hipStreamWaitEvent(side_stream(), fork_event(k), 0));
    if (curv_launch(k, vof, side_stream())) return 1;
    SBFS_HIP(hipEventRecord(join_event(k), side_stream()));
    return 0;
  };
  if (overlap && fork_curv(0, D(interface->vof))) return 1;
  if (compute_dt_device(domain, c, fluid, interface)) return 1;
  const double* dtp = &c->dt->dt;
  const bool fold = march_fold();
  const bool nt = stream_fields(nx, ny);  // streaming accesses of the rows touched once
  // the units in order of the interface rows the last stage kernel found in
  // them (the previous step's; the bubbles move a fraction of a cell per
  // step), for all three stages of this step
  const bool mixed = options().precision == SBFS_PRECISION_MIXED;
  const bool wide = mixed && mixed_march_wide(nx, ny);
  const int tile = tile_rows(nx, ny, mixed);
  const bool ordered = tile == 0 && march_ordered(mixed);
  const int units = march_units(nx, ny, band);
  if (ordered) {
    SBFS_REQUIRE(scr.units >= units, "integrate: no dispatch-order buffers for %d units", units);
    SBFS_TIMED("k_march_order", hipLaunchKernelGGL(k_march_order, dim3(1), dim3(1024), 0, stream(),
                                                   (const unsigned*)scr.weight, scr.order, units,
                                                   march_max_weight(band)));
    if (check_launch("integrate: k_march_order")) return 1;
  }
  // predicted velocity of each stage: with the fold, stage 1 writes the
  // second pair while it reads the first
  double* const us[3] = {scr.ux, fold ? scr.ux2 : scr.ux, scr.ux};
  double* const vs[3] = {scr.uy, fold ? scr.uy2 : scr.uy, scr.uy};
  for (int k = 0; k < 3; k++) {
    const bool corr = fold && k > 0;  // this stage applies stage k-1's projection
    if (k != 0) {
      swap_data(interface->src[0], interface->src[1]);
      swap_data(fluid->srcux[0], fluid->srcux[1]);
      swap_data(fluid->srcuy[0], fluid->srcuy[1]);
    }
    {
      MarchArgs m;
      memset(&m, 0, sizeof(m));  // padding too: the arguments are compared bytewise
      fill_march(domain, c, fluid, interface, cf, rhs, band, k, corr, us, vs, scr.vof, scr.p, dtp, m);
      if (learned) {
        if (overlap) {
          SBFS_HIP(hipStreamWaitEvent(stream(), join_event(k), 0));
        } else if (curv_launch(k, D(interface->vof), stream())) {
          return 1;
        }
        m.kappa = scr.kappa;
        m.kappa_n = scr.klist[k];
        if (k < 2) m.cut = scr.cut;
      }
      if (ordered) {
        m.order = scr.order;
        m.weight = scr.weight;
      }
      const dim3 block(64), grid = ordered ? dim3(cdiv(units, 8 * kOrderChunk) * 8 * kOrderChunk)
                                           : dim3(cdiv(nx, kStrip), cdiv(ny, band));
      const MarchArgs* ma = nullptr;
      if (device_args(c, m, &ma)) return 1;
      if (tile) {
        tile_launch(ma, nx, ny, tile, mixed, corr);
      } else if (mixed && corr)
        SBFS_TIMED("k_march_mixed_corr",
                   hipLaunchKernelGGL((wide ? k_march_mixed_corr_wide : k_march_mixed_corr), grid, block, 0, stream(),
                                      ma));
      else if (mixed)
        SBFS_TIMED("k_march_mixed",
                   hipLaunchKernelGGL((wide ? k_march_mixed_wide : k_march_mixed), grid, block, 0, stream(), ma));
      else if (corr)
        SBFS_TIMED("k_march_corr",
                   hipLaunchKernelGGL((nt ? k_march_corr_nt : k_march_corr), grid, block, 0, stream(), ma));
      else
        SBFS_TIMED("k_march", hipLaunchKernelGGL((nt ? k_march_nt : k_march), grid, block, 0, stream(), ma));
      if (check_launch("integrate: k_march")) return 1;
      if (corr && k == 2) {
        // the stage kernel wrote the pressure after stage 1's update
        double* t = (double*)fluid->p.data;
        fluid->p.data = scr.p;
        scr.p = t;
      }
    }
    {
      // the new vof becomes the state; the old one is the next scratch
      void* t = interface->vof.data;
      interface->vof.data = scr.vof;
      scr.vof = (double*)t;
    }
    // the next stage's curvature from the new vof, beside this stage's
    // Poisson solve (the stage kernel that read kappa has been launched)
    if (overlap && k < 2 && fork_curv(k + 1, D(interface->vof))) return 1;
    if (poisson_transform_fused(domain, c, fluid, nullptr)) return 1;
    if (fold && k < 2) {
      // projected by the next stage's kernel
      swap_data(fluid->psi[0], fluid->psi[1]);
      continue;
    }
    PostArgs q;
    fill_post(c, fluid, interface, us[k], vs[k], dtp, k, q);
    const dim3 pg(cdiv(nx + 2, 64), cdiv(ny, 4 * kPostRows)), pb(64, 4);
    // (fields of 4 GiB or more are always streamed)
    if (!fp64_march_addressable(nx, ny))
      SBFS_TIMED("k_post", hipLaunchKernelGGL((k_post<size_t, true>), pg, pb, 0, stream(), q));
    else if (stream_fields(nx, ny))
      SBFS_TIMED("k_post", hipLaunchKernelGGL((k_post<unsigned, true>), pg, pb, 0, stream(), q));
    else
      SBFS_TIMED("k_post", hipLaunchKernelGGL((k_post<unsigned, false>), pg, pb, 0, stream(), q));
    if (check_launch("integrate: k_post")) return 1;
    swap_data(fluid->psi[0], fluid->psi[1]);
  }
  return 0;
}

// ---------------------------------------------------------------------------
// Graph replay of the fused step.  The step's launches depend only on the
// array pointers, the case parameters and the options, and the pointers
// return to one of two states (psi and vof swap an odd number of times per
// step), so two captured graphs serve a run and a domain keeps four.  A configuration is
// captured the second time it is seen: the first, eager, pass builds every
// plan and table the step needs, so the captured sequence allocates and
// synchronises nothing.  Profiling (per-launch events) and SBFS_GRAPH=0
// keep the eager path.
// ---------------------------------------------------------------------------
static void key_add(StepKey& k, const void* p) { k.v.push_back((uint64_t)(uintptr_t)p); }
static void key_add(StepKey& k, double x) {
  uint64_t u;
  memcpy(&u, &x, sizeof(u));
  k.v.push_back(u);
}

static array_t* state_arrays(fluid_t* f, interface_t* s, int k) {
  array_t* a[] = {&f->ux, &f->uy, &f->p, &f->psi[0], &f->psi[1], &f->den[0], &f->den[1],
                  &f->txy, &f->srcux[0], &f->srcux[1], &f->srcux[2], &f->srcuy[0],
                  &f->srcuy[1], &f->srcuy[2], &s->vof, &s->src[0], &s->src[1]};
  return k < 17 ? a[k] : nullptr;
}

static StepKey step_key(const DomainCtx* c, fluid_t* f, interface_t* s, const Coef& cf, double* rhs,
                        int band) {
  const FusedScratch& scr = c->fused->scr;
  StepKey k;
  k.v.reserve(64);
  key_add(k, c);
  k.v.push_back(c->hash);
  for (int n = 0; n < kStateArrays; n++) key_add(k, state_arrays(f, s, n)->data);
  key_add(k, scr.vof);
  key_add(k, scr.ux);
  key_add(k, scr.uy);
  key_add(k, scr.ux2);
  key_add(k, scr.uy2);
  key_add(k, scr.p);
  k.v.push_back(march_fold() ? 1 : 0);
  key_add(k, cf.rhf);
  key_add(k, rhs);
  for (double x : {f->Re, f->Fr, f->denr, f->visr, f->refden, s->We, options().cadv, options().cdif,
                   options().cint})
    key_add(k, x);
  k.v.push_back((uint64_t)band);
  k.v.push_back((uint64_t)options().gauge | ((uint64_t)options().tdm << 8) |
                ((uint64_t)options().chunk << 16) | ((uint64_t)options().precision << 48) |
                ((uint64_t)options().curvature << 56));
  key_add(k, scr.kappa);
  for (const unsigned* l : scr.klist) key_add(k, l);
  k.v.push_back((uint64_t)(int64_t)scr.klast);
  key_add(k, scr.cut);
  const bool mixed = options().precision == SBFS_PRECISION_MIXED;
  k.v.push_back((march_ordered(mixed) ? 1 : 0) | ((uint64_t)tile_rows((int)c->nx, (int)c->ny, mixed) << 1));
  k.v.push_back((stream_fields(c->nx, c->ny) ? 1 : 0) | (mixed_march_wide(c->nx, c->ny) ? 2 : 0));
  key_add(k, scr.order);
  k.v.push_back(c->epoch);
  k.v.push_back(poisson_epoch(c));
  return k;
}

static bool graphs_enabled() {
  static int on = -1;
  if (on < 0) {
    const char* e = getenv("SBFS_GRAPH");
    on = (e && e[0] == '0') ? 0 : 1;
  }
  return on == 1 && !prof_active();
}

static int step_graph(const domain_t* domain, DomainCtx* c, fluid_t* fluid, interface_t* interface,
                      const Coef& cf, double* rhs, int band, double learned_h) {
  if (!graphs_enabled()) return fused_body(domain, c, fluid, interface, cf, rhs, band, learned_h);
  FusedState& fs = *c->fused;
  FusedScratch& scr = fs.scr;
  const StepKey key = step_key(c, fluid, interface, cf, rhs, band);
  fs.clock++;
  for (StepGraph& g : fs.graph) {
    if (g.exec && g.key == key) {
      SBFS_HIP(hipGraphLaunch(g.exec, stream()));
      for (int n = 0; n < kStateArrays; n++) state_arrays(fluid, interface, n)->data = g.after[n];
      scr.vof = (double*)g.after[kStateArrays];
      scr.p = (double*)g.after[kStateArrays + 1];
      g.last_use = fs.clock;
      return 0;
    }
  }
  bool seen = false;
  for (const StepKey& k : fs.seen) seen = seen || k == key;
  if (!seen) {
    // first sight of this configuration: run eagerly (builds plans / tables);
    // one that failed has not built them all, and the next one runs eagerly too
    const int rc = fused_body(domain, c, fluid, interface, cf, rhs, band, learned_h);
    if (!rc) fs.seen[fs.clock % kStepGraphs] = key;
    return rc;
  }
  StepGraph* slot = &fs.graph[0];
  for (StepGraph& g : fs.graph)
    if (g.last_use < slot->last_use) slot = &g;
  StepGraph& g = *slot;
  if (g.exec) {
    (void)hipGraphExecDestroy(g.exec);
    g.exec = nullptr;
  }
  hipGraph_t graph = nullptr;
  SBFS_HIP(hipStreamBeginCapture(stream(), hipStreamCaptureModeRelaxed));
  const int rc = fused_body(domain, c, fluid, interface, cf, rhs, band, learned_h);
  const hipError_t ce = hipStreamEndCapture(stream(), &graph);
  if (rc) {
    if (graph) (void)hipGraphDestroy(graph);
    return 1;
  }
  SBFS_HIP(ce);
  const hipError_t ie = hipGraphInstantiate(&g.exec, graph, nullptr, nullptr, 0);
  (void)hipGraphDestroy(graph);
  SBFS_HIP(ie);
  g.key = key;
  for (int n = 0; n < kStateArrays; n++) g.after[n] = state_arrays(fluid, interface, n)->data;
  g.after[kStateArrays] = scr.vof;
  g.after[kStateArrays + 1] = scr.p;
  g.last_use = fs.clock;
  SBFS_HIP(hipGraphLaunch(g.exec, stream()));
  return 0;
}

int integrate_fused(const domain_t* domain, fluid_t* fluid, interface_t* interface, double* dt) {
  DomainCtx* c = domain_ctx(domain);
  if (!c) return 1;
  const Nadds* nas[] = {&NA_UX, &NA_UY, &NA_P, &NA_P, &NA_P, &NA_DEN, &NA_DEN, &NA_TXY};
  const array_t* arrs[] = {&fluid->ux, &fluid->uy, &fluid->p, &fluid->psi[0], &fluid->psi[1],
                           &fluid->den[0], &fluid->den[1], &fluid->txy};
  for (int k = 0; k < 8; k++)
    if (check_array(domain, arrs[k], *nas[k], 8, "fluid array")) return 1;
  for (int n = 0; n < 3; n++) {
    if (check_array(domain, &fluid->srcux[n], NA_SRCUX, 8, "srcux")) return 1;
    if (check_array(domain, &fluid->srcuy[n], NA_SRCUY, 8, "srcuy")) return 1;
  }
  if (check_array(domain, &interface->vof, NA_VOF, 8, "vof")) return 1;
  for (int n = 0; n < 2; n++)
    if (check_array(domain, &interface->src[n], NA_SRC, 8, "src")) return 1;
  if (!c->fused) c->fused = new FusedState();
  if (scratch(c, interface, fluid, options().curvature == SBFS_CURVATURE_LEARNED)) return 1;
  Coef cf;
  if (coef_tables(domain, c, fluid->Re, &cf)) return 1;
  const int nx = (int)c->nx, ny = (int)c->ny;
  double* rhs = nullptr;
  if (poisson_transform_fused(domain, c, fluid, &rhs)) return 1;
  const int band = march_band(nx, ny, options().precision == SBFS_PRECISION_MIXED);
  if (band <= 0) return 1;
  const bool mixed = options().precision == SBFS_PRECISION_MIXED;
  if (march_ordered(mixed) && tile_rows(nx, ny, mixed) == 0 &&
      order_buffers(c, march_units(nx, ny, band)))
    return 1;
  if (load_dt_coefs()) return 1;
  double learned_h = 0.;
  if (options().curvature == SBFS_CURVATURE_LEARNED) {
    // the network sees 5 x 5 stencils of square cells of one size
    const double h = domain->hy;
    for (int i = 0; i < nx; i++)
      SBFS_REQUIRE(fabs(domain->hxxc[i] - h) <= 1e-12 * h,
                   "learned curvature: needs uniform square cells (HXXC(%d) = %g, hy = %g)", i + 1,
                   domain->hxxc[i], h);
    learned_h = h;
  }
  if (step_graph(domain, c, fluid, interface, cf, rhs, band, learned_h)) return 1;
  SBFS_HIP(hipStreamSynchronize(stream()));
  *dt = *dt_host(c);
  return 0;
}

// One fused step of one ensemble case, planned without launching: the
// pointer choreography of fused_body (projection folded, plain curvature,
// sequential tridiagonal solve) applied to the case's structs and scratch,
// recording the arguments of every launch.  On return the structs and
// scratch hold the pointer state after the step.
int ensemble_plan_step(const domain_t* domain, DomainCtx* c, fluid_t* fluid, interface_t* interface,
                       const Coef& cf, int band, double* host_dt, CaseScratch& scr, CaseStep& out) {
  if (dt_args(domain, c, fluid, interface, c->dt, host_dt, &out.dt)) return 1;
  const double* dtp = &c->dt->dt;
  double* rhs = nullptr;
  if (poisson_transform_fused(domain, c, fluid, &rhs)) return 1;
  double* const us[3] = {scr.ux[0], scr.ux[1], scr.ux[0]};
  double* const vs[3] = {scr.uy[0], scr.uy[1], scr.uy[0]};
  for (int k = 0; k < 3; k++) {
    const bool corr = k > 0;
    if (k != 0) {
      swap_data(interface->src[0], interface->src[1]);
      swap_data(fluid->srcux[0], fluid->srcux[1]);
      swap_data(fluid->srcuy[0], fluid->srcuy[1]);
    }
    fill_march(domain, c, fluid, interface, cf, rhs, band, k, corr, us, vs, scr.vof, scr.p, dtp, out.march[k]);
    if (corr && k == 2) {
      double* t = (double*)fluid->p.data;
      fluid->p.data = scr.p;
      scr.p = t;
    }
    {
      void* t = interface->vof.data;
      interface->vof.data = scr.vof;
      scr.vof = (double*)t;
    }
    if (poisson_row_args(domain, c, (double*)fluid->psi[1].data, &out.rows[k])) return 1;
    if (k == 2) fill_post(c, fluid, interface, us[k], vs[k], dtp, k, out.post);
    swap_data(fluid->psi[0], fluid->psi[1]);
  }
  return 0;
}

}  // namespace sbfs
