// graph_workspace.h -- a workspace that grows with what is asked of it and that
// calls under stream capture are given too.
#pragma once
#include <stddef.h>

#include <algorithm>

namespace ffmi {

// A graph holds the address that its captured calls were given for as long as it
// lives, which nobody reports here.  So a block that a captured call was given is
// never freed; the one that replaces it is at least twice as large, and all that
// are kept together stay below the current one.  Any other block is freed when
// it is replaced.  (A captured call that needs more frees nothing either: that
// takes a synchronisation, which a capture forbids.)
class GraphWorkspace {
 public:
  // A block of at least `need` bytes, nullptr if it cannot be had (the present one
  // stays, unless it was freed).  alloc(bytes) -> pointer or nullptr; release(p):
  // waits for the device and frees, false if that fails.
  template <class Alloc, class Release>
  void *get(size_t need, bool captured, Alloc alloc, Release release) {
    if (need > bytes_) {
      const bool keep = p_ && (recorded_ || captured);
      if (p_ && !keep) {
        void *old = p_;
        p_ = nullptr, bytes_ = 0;
        if (!release(old)) return nullptr;
      }
      const size_t want = keep ? std::max(need, 2 * bytes_) : need;
      void *q = alloc(want);
      if (!q) return nullptr;
      if (keep) kept_ += bytes_;
      p_ = q, bytes_ = want, recorded_ = false;
    }
    recorded_ |= captured;
    return p_;
  }
  size_t bytes() const { return bytes_; }
  size_t kept() const { return kept_; }

 private:
  void *p_ = nullptr;
  size_t bytes_ = 0, kept_ = 0;  // of the current block, of the earlier ones in graphs
  bool recorded_ = false;        // a captured call was given the current block
};

}  // namespace ffmi
