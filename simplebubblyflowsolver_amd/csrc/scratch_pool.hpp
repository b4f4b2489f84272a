// The fused step's scratch of a domain, and the pool of the sets that closed
// domains gave back.
//
// Api is the memory the sets live in (fused.hip: device memory; a CPU test:
// counted blocks): int alloc(void** p, size_t bytes), 0 for success;
// void free(void* p), which takes null; int zero(void* p, size_t bytes).
#pragma once

#include <cstddef>
#include <mutex>
#include <utility>
#include <vector>

namespace sbfs {

struct FusedScratch {
  size_t nx = 0, ny = 0;
  size_t bytes = 0;  // of all that the set holds
  double* vof = nullptr;
  double* ux = nullptr;   // predicted velocity of stages 0 and 2
  double* uy = nullptr;
  double* ux2 = nullptr;  // predicted velocity of stage 1 (folded projection)
  double* uy2 = nullptr;
  double* p = nullptr;    // pressure written by a stage kernel with the folded projection
  // learned curvature only (allocated when it is first used):
  float* kappa = nullptr;  // learned curvature of a stage's input vof (interior cells)
  unsigned* klist[3] = {};  // its listed cells (count first), one list per stage
  int klast = -1;            // the list of the last launch (-1: none since the fill)
  unsigned long long* cut = nullptr;  // cut-cell bitmask of a stage kernel's new vof
  // the stage kernels' dispatch order and unit weights (march.hpp)
  unsigned* weight = nullptr;
  unsigned* order = nullptr;
  int units = 0;
};

// bytes of the fields a domain's scratch twins
struct ScratchSizes {
  size_t nx, ny, ux, uy, p, vof;
};

template <typename Api>
void scratch_free(FusedScratch& s) {
  for (double* q : {s.vof, s.ux, s.uy, s.ux2, s.uy2, s.p}) Api::free(q);
  Api::free(s.kappa);
  for (unsigned* l : s.klist) Api::free(l);
  Api::free(s.cut);
  Api::free(s.weight);
  Api::free(s.order);
  s = FusedScratch();
}

// The sets of closed domains, for the next ones of their sizes: a program that
// closes a case and opens another allocates and frees no scratch (a hipFree of
// 268 MB takes 0.24 ms, a close of a 256 x 256 learned case 13 of them).
//  * The last set given back always stays, the others while all together are
//    at most kMost (1/36 of the card, room for three 4096 x 8192 learned cases).
//  * A domain that needs a set leaves at most kIdle of other sizes in the pool.
//  * Of several the largest goes first, among equals the oldest.
//  * An allocation that fails empties the pool and is tried again.
template <typename Api>
class ScratchPool {
 public:
  static constexpr size_t kMost = 8ull << 30, kIdle = 1ull << 30;

  // A domain's scratch: a set from the pool (one with the learned curvature's
  // buffers if they are wanted, and without them if not, where there is a
  // choice), or a new one.  All of it or, with a non-zero result, nothing.
  int get(const ScratchSizes& z, bool learned, FusedScratch* out) {
    {
      std::lock_guard<std::mutex> lock(m_);
      trim(kIdle, false, [&z](const FusedScratch& s) { return s.nx != z.nx || s.ny != z.ny; });
      int at = -1;
      for (int k = (int)sets_.size() - 1; k >= 0; k--)
        if (sets_[k].nx == z.nx && sets_[k].ny == z.ny && (at < 0 || ((sets_[k].cut != nullptr) == learned &&
                                                                      (sets_[at].cut != nullptr) != learned)))
          at = k;
      if (at >= 0) {
        *out = sets_[at];
        bytes_ -= out->bytes;
        sets_.erase(sets_.begin() + at);
        return 0;
      }
    }
    FusedScratch s;
    const std::pair<double**, size_t> bufs[] = {{&s.vof, z.vof}, {&s.ux, z.ux},   {&s.uy, z.uy},
                                                {&s.ux2, z.ux},  {&s.uy2, z.uy}, {&s.p, z.p}};
    for (const auto& b : bufs) {
      int rc = alloc((void**)b.first, b.second);
      if (!rc) rc = Api::zero(*b.first, b.second);
      if (rc) {
        scratch_free<Api>(s);
        return rc;
      }
      s.bytes += b.second;
    }
    s.nx = z.nx;
    s.ny = z.ny;
    *out = s;
    return 0;
  }

  // takes a closed domain's set (nothing uses it any more)
  void put(FusedScratch& s) {
    if (!s.vof) return;
    std::lock_guard<std::mutex> lock(m_);
    sets_.push_back(s);
    bytes_ += s.bytes;
    s = FusedScratch();
    trim(kMost, true, all);
  }

  // an allocation that may take the pool's memory
  int alloc(void** p, size_t bytes) {
    const int rc = Api::alloc(p, bytes);
    if (!rc) return 0;
    {
      std::lock_guard<std::mutex> lock(m_);
      if (sets_.empty()) return rc;
      trim(0, false, all);
    }
    return Api::alloc(p, bytes);
  }

  size_t bytes() {
    std::lock_guard<std::mutex> lock(m_);
    return bytes_;
  }

 private:
  static bool all(const FusedScratch&) { return true; }

  // frees sets that `of` names, all but the last if that one stays, until they hold `most` bytes
  template <typename Of>
  void trim(size_t most, bool last_stays, Of of) {
    for (;;) {
      size_t held = 0;
      int at = -1;
      const int n = (int)sets_.size();
      for (int k = 0; k < n; k++) {
        if (!of(sets_[k])) continue;
        held += sets_[k].bytes;
        if (!(last_stays && k == n - 1) && (at < 0 || sets_[k].bytes > sets_[at].bytes)) at = k;
      }
      if (held <= most || at < 0) return;
      bytes_ -= sets_[at].bytes;
      scratch_free<Api>(sets_[at]);
      sets_.erase(sets_.begin() + at);
    }
  }

  std::mutex m_;
  std::vector<FusedScratch> sets_;
  size_t bytes_ = 0;
};

}  // namespace sbfs
