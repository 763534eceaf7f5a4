// logit_rows.h -- rows of a step's logits to the caller's host memory, as fp32.
#pragma once
#include <stdint.h>
#include <string.h>

#include <algorithm>

#include "../ffmi_internal.h"

namespace ffmi {

// A kernel converts the rows and writes them through PCIe into pinned staging,
// kRows at a time; a row is copied to the caller as soon as it is there, while the rows
// after it arrive (and, beyond kRows, while the next rows go into the other half).  The
// first rows follow the step on its stream.  (One blocking copy per row
// and a conversion on one core took 90 us per row of 32000 fp16 logits, a
// pageable copy of 8 fp32 rows 110 us; 8 rows copied after the last of them was there
// took about 20 us a step more than this.)  The caller's memory is mostly fresh from its
// allocator: its pages are touched while the step runs, not by the copy behind it (8 rows
// of 32000, 1 MB: the copy 160 us into fresh pages, 25 into touched ones).
class LogitRows {
 public:
  ~LogitRows() {
    for (auto e : done_)
      if (e) (void)hipEventDestroy(e);
    if (step_) (void)hipEventDestroy(step_);
    if (staging_) (void)hipHostFree(staging_);
    if (there_) (void)hipHostFree(there_);
  }
  // logits: [.][ld] on the device, fp16 (half) or fp32; rows[0, n): which
  // (null: 0 .. n - 1); out: [n][V] of host memory.  The first rows are put on the
  // stream, and out is made ready (its contents stay) while the stream works.
  ffmi_status begin(const void *logits, bool half, size_t ld, const int *rows, int n, int V, hipStream_t s,
                    float *out) {
    src_ = logits, half_ = half, ld_ = ld, rows_ = rows, n_ = 0, V_ = V, stream_ = s;
    if (n <= 0) return FFMI_OK;
    if (!there_) {
      const size_t bytes = (size_t)2 * kRows * LogitRowIds::kParts * sizeof(uint32_t);
      FFMI_HIP(hipHostMalloc((void **)&there_, bytes, hipHostMallocCoherent | hipHostMallocMapped));
      memset(there_, 0, bytes);
    }
    if (staged_ < LogitRowIds::pitch(V)) {
      if (staging_) (void)hipHostFree(staging_);
      staging_ = nullptr, staged_ = 0;
      FFMI_HIP(hipHostMalloc((void **)&staging_, 2 * kRows * LogitRowIds::pitch(V) * sizeof(float),
                             hipHostMallocCoherent | hipHostMallocMapped));
      staged_ = LogitRowIds::pitch(V);
    }
    for (auto &e : done_)
      if (!e) FFMI_HIP(hipEventCreateWithFlags(&e, hipEventDisableTiming));
    // Rows are waited for by looking, the step before them as the device's flags say
    // (FFMI_SYNC): where threads yield or sleep, by an event of its own.  (HIP's default
    // keeps the core in either wait, and the event takes up to 4 us a step.)
    unsigned flags = 0;
    FFMI_HIP(hipGetDeviceFlags(&flags));
    sleeps_ = (flags & hipDeviceScheduleMask) == hipDeviceScheduleBlockingSync ||
              (flags & hipDeviceScheduleMask) == hipDeviceScheduleYield;
    if (sleeps_) {
      if (!step_) FFMI_HIP(hipEventCreateWithFlags(&step_, hipEventDisableTiming));
      FFMI_HIP(hipEventRecord(step_, s));
    }
    out_ = out, n_ = n;
    const ffmi_status st = put(0, n);
    if (st == FFMI_OK) touch(out, (size_t)n * V * sizeof(float));
    else n_ = 0;
    return st;
  }
  // every row to out [n][V] (nothing if begin failed or had none); then the stream's work
  // up to the rows is done, too
  ffmi_status finish() {
    const int n = n_;
    n_ = 0;
    if (n <= 0) return FFMI_OK;
    if (sleeps_) FFMI_HIP(hipEventSynchronize(step_));
    int half = 0;
    for (int at = 0;; at += kRows, half ^= 1) {
      const uint32_t mark = mark_;
      const int here = std::min(kRows, n - at);
      if (at + kRows < n) {
        const ffmi_status st = put(at + kRows, n);
        if (st != FFMI_OK) return st;
      }
      for (int i = 0, to; i < here; i = to) {  // (as many rows at once as are there)
        const ffmi_status st = await(half, i, mark);
        if (st != FFMI_OK) return st;
        for (to = i + 1; to < here && there(half, to, mark);) ++to;
        const size_t pitch = LogitRowIds::pitch(V_);
        const float *from = staging_ + ((size_t)half * kRows + i) * pitch;
        if (pitch == (size_t)V_) {
          memcpy(out_ + (size_t)(at + i) * V_, from, (to - i) * pitch * sizeof(float));
        } else {
          for (int k = i; k < to; ++k, from += pitch) memcpy(out_ + (size_t)(at + k) * V_, from, V_ * sizeof(float));
        }
      }
      if (at + kRows >= n) break;
    }
    FFMI_HIP(hipEventSynchronize(done_[half]));
    return FFMI_OK;
  }

 private:
  static void touch(void *p, size_t bytes) {
    constexpr size_t kPage = 4096;
    volatile char *at = (volatile char *)p, *end = at + bytes;
    for (; at < end; at = (volatile char *)(((uintptr_t)at | (kPage - 1)) + 1)) *at = *at;
  }
  static constexpr int kRows = LogitRowIds::kMax;
  // row i of a half is there: every workgroup's word says so
  bool there(int half, int i, uint32_t mark) const {
    const uint32_t *word = there_ + ((size_t)half * kRows + i) * LogitRowIds::kParts;
    for (int p = LogitRowIds::parts(V_) - 1; p >= 0; --p)
      if (__atomic_load_n(word + p, __ATOMIC_ACQUIRE) != mark) return false;
    return true;
  }
  // (the event behind the kernel is asked now and then, so that a stream in error ends the wait)
  ffmi_status await(int half, int i, uint32_t mark) {
    for (int spins = 1; !there(half, i, mark); ++spins) {
      if (spins % 8192 == 0) {
        const hipError_t e = hipEventQuery(done_[half]);
        if (e == hipSuccess) return FFMI_OK;
        if (e != hipErrorNotReady) FFMI_HIP(e);
        (void)hipGetLastError();  // (not an error that a later launch should find)
      }
      __builtin_ia32_pause();
    }
    return FFMI_OK;
  }
  ffmi_status put(int at, int all) {
    const int half = at / kRows & 1;
    LogitRowIds ids;
    const int n = std::min(kRows, all - at);
    for (int i = 0; i < n; ++i) ids.row[i] = rows_ ? rows_[at + i] : at + i;
    FFMI_HIP(launch_logit_rows(src_, half_, ld_, ids, n, V_,
                               staging_ + (size_t)half * kRows * LogitRowIds::pitch(V_),
                               there_ + (size_t)half * kRows * LogitRowIds::kParts, ++mark_, stream_));
    FFMI_HIP(hipEventRecord(done_[half], stream_));
    return FFMI_OK;
  }
  float *staging_ = nullptr, *out_ = nullptr;
  uint32_t *there_ = nullptr;  // [2][kRows][kParts]
  uint32_t mark_ = 0;          // of the latest kernel
  size_t staged_ = 0;  // row width that the staging holds
  hipEvent_t done_[2] = {nullptr, nullptr}, step_ = nullptr;
  bool sleeps_ = false;
  const void *src_ = nullptr;
  const int *rows_ = nullptr;
  bool half_ = false;
  size_t ld_ = 0;
  int n_ = 0, V_ = 0;
  hipStream_t stream_ = nullptr;
};

}  // namespace ffmi
