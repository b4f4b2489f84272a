// decide_dt without allocation, for callers that cannot allocate device
// memory (code under graph capture, tight serving loops, harnesses that
// forbid hipMalloc).
//
// decide_dt reduces into a slot that the library allocates with the domain's
// device context.  decide_dt_noalloc runs the same kernel on a file-scope
// device variable instead.  Each GPU holds its own copy until the process ends;
// its device address is looked up once per device (hipGetSymbolAddress, at the
// library's set-up for the current device, otherwise at the first call on
// another device) and only that address is handed to kernels.
//
// The slot needs no clearing: it starts as 0, and every launch leaves it so.
// Every call on a GPU shares that GPU's slot and the library stream, so calls
// that overlap on one GPU (from several host threads) race.
#include <cfloat>

#include "decide_dt.h"
#include "sbfs.h"
#include "sbfs_internal.hpp"

namespace sbfs {

static __device__ DtSlot slot_;

constexpr int kMaxDevices = 64;
static DtSlot* g_slot_ptr[kMaxDevices] = {};

// device address of `slot_` on the current device, looked up once per
// device
static int slot_ptr(DtSlot** out) {
  int dev = 0;
  SBFS_HIP(hipGetDevice(&dev));
  SBFS_REQUIRE(dev >= 0 && dev < kMaxDevices, "decide_dt_noalloc: device %d out of range", dev);
  if (!g_slot_ptr[dev]) {
    void* p = nullptr;
    SBFS_HIP(hipGetSymbolAddress(&p, HIP_SYMBOL(slot_)));
    SBFS_REQUIRE(p != nullptr, "decide_dt_noalloc: no device address for its slot");
    g_slot_ptr[dev] = (DtSlot*)p;
  }
  *out = g_slot_ptr[dev];
  return 0;
}

int noalloc_setup() {
  DtSlot* p = nullptr;
  return slot_ptr(&p);
}

}  // namespace sbfs

using namespace sbfs;

extern "C" {

int decide_dt_noalloc(const domain_t* domain, const fluid_t* fluid, const interface_t* interface,
                      double* dt) {
  SBFS_REQUIRE(domain && fluid && interface && dt, "decide_dt_noalloc: null argument");
  DomainCtx* c = domain_ctx_find(domain);
  SBFS_REQUIRE(c != nullptr,
               "decide_dt_noalloc: the domain has no device context (create it first with fluid_init, "
               "interface_init, sbfs_domain_create or decide_dt)");
  if (check_array(domain, &fluid->ux, NA_UX, 8, "ux")) return 1;
  if (check_array(domain, &fluid->uy, NA_UY, 8, "uy")) return 1;
  DtSlot* s = nullptr;
  if (slot_ptr(&s)) return 1;
  DtArgs a;
  if (dt_args(domain, c, fluid, interface, s, dt_host(c), &a)) return 1;
  if (dt_launch(a)) return 1;
  SBFS_HIP(hipStreamSynchronize(stream()));
  *dt = *dt_host(c);
  return 0;
}

}  // extern "C"
