// logit_rows.h -- rows of a step's logits to the caller's host memory, as fp32.
#pragma once
#include <stdint.h>
#include <string.h>

#include <algorithm>

#include "../ffmi_internal.h"

namespace ffmi {

// A kernel converts the rows and writes them through PCIe into pinned staging,
// kRows at a time; while one half of the staging is copied to the caller, the
// next rows go into the other.  The first rows follow the step on its stream, so
// that they are there when the step is waited for.  (One blocking copy per row
// and a conversion on one core took 90 us per row of 32000 fp16 logits, a
// pageable copy of 8 fp32 rows 110 us.)  The caller's memory is mostly fresh from its
// allocator: its pages are touched while the step runs, not by the copy behind it (8 rows
// of 32000, 1 MB: the copy 160 us into fresh pages, 25 into touched ones).
class LogitRows {
 public:
  ~LogitRows() {
    for (auto e : done_)
      if (e) (void)hipEventDestroy(e);
    if (staging_) (void)hipHostFree(staging_);
  }
  // logits: [.][ld] on the device, fp16 (half) or fp32; rows[0, n): which
  // (null: 0 .. n - 1); out: [n][V] of host memory.  The first rows are put on the
  // stream, and out is made ready (its contents stay) while the stream works.
  ffmi_status begin(const void *logits, bool half, size_t ld, const int *rows, int n, int V, hipStream_t s,
                    float *out) {
    src_ = logits, half_ = half, ld_ = ld, rows_ = rows, n_ = n, V_ = V, stream_ = s;
    if (n <= 0) return FFMI_OK;
    if (staged_ < (size_t)V) {
      if (staging_) (void)hipHostFree(staging_);
      staging_ = nullptr, staged_ = 0;
      FFMI_HIP(hipHostMalloc((void **)&staging_, (size_t)2 * kRows * V * sizeof(float),
                             hipHostMallocCoherent | hipHostMallocMapped));
      staged_ = V;
    }
    for (auto &e : done_)
      if (!e) FFMI_HIP(hipEventCreateWithFlags(&e, hipEventDisableTiming));
    out_ = out;
    const ffmi_status st = put(0);
    if (st == FFMI_OK) touch(out, (size_t)n * V * sizeof(float));
    return st;
  }
  // every row to out [n][V]
  ffmi_status finish() {
    float *const out = out_;
    for (int at = 0, half = 0; at < n_; at += kRows, half ^= 1) {
      if (at + kRows < n_) {
        const ffmi_status st = put(at + kRows);
        if (st != FFMI_OK) return st;
      }
      FFMI_HIP(hipEventSynchronize(done_[half]));
      memcpy(out + (size_t)at * V_, staging_ + (size_t)half * kRows * V_,
             (size_t)std::min(kRows, n_ - at) * V_ * sizeof(float));
    }
    return FFMI_OK;
  }

 private:
  static void touch(void *p, size_t bytes) {
    constexpr size_t kPage = 4096;
    volatile char *at = (volatile char *)p, *end = at + bytes;
    for (; at < end; at = (volatile char *)(((uintptr_t)at | (kPage - 1)) + 1)) *at = *at;
  }
  static constexpr int kRows = LogitRowIds::kMax;
  ffmi_status put(int at) {
    const int half = at / kRows & 1;
    LogitRowIds ids;
    const int n = std::min(kRows, n_ - at);
    for (int i = 0; i < n; ++i) ids.row[i] = rows_ ? rows_[at + i] : at + i;
    FFMI_HIP(launch_logit_rows(src_, half_, ld_, ids, n, V_, staging_ + (size_t)half * kRows * V_, stream_));
    FFMI_HIP(hipEventRecord(done_[half], stream_));
    return FFMI_OK;
  }
  float *staging_ = nullptr, *out_ = nullptr;
  size_t staged_ = 0;  // row width that the staging holds
  hipEvent_t done_[2] = {nullptr, nullptr};
  const void *src_ = nullptr;
  const int *rows_ = nullptr;
  bool half_ = false;
  size_t ld_ = 0;
  int n_ = 0, V_ = 0;
  hipStream_t stream_ = nullptr;
};

}  // namespace ffmi
