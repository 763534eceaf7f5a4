// memory.hip -- matrix memories, token by token (memory.h).
#include "memory_steps.h"

namespace ffmi {

namespace {

template <MemoryRule RULE, class E, int P, bool SPLIT>
__global__ __launch_bounds__(NT, SPLIT ? 4 : 2) void memory_steps_kernel(const char *__restrict__ blob, int off_spans, Memory a,
                                                          MemoryScratch w, int limit, MemoryStepsPlan plan) {
  extern __shared__ __attribute__((aligned(16))) float lds[];
  memory_steps<RULE, E, P, SPLIT>(blob, off_spans, a, w, limit, plan, blockIdx.x, blockIdx.y, blockIdx.z, lds);
}

template <MemoryRule RULE, class E>
hipError_t run_steps(const char *blob, int off_spans, int num_spans, const Memory &a, const MemoryScratch *w,
                     int limit, bool *left, hipStream_t s) {
  const MemoryStepsPlan plan = memory_steps_plan(a, num_spans, limit, w && sizeof(E) == 2);
  const int rows = plan.rows, parts = plan.parts;
  const size_t bytes = plan.bytes;
  if (bytes > 64 * 1024) return hipErrorInvalidValue;
  const MemoryScratch none;
  *left = parts > 1;
  const dim3 grid(a.H, num_spans, parts);
#define FFMI_MS(P)                                                                                                    \
  do {                                                                                                                \
    if constexpr (sizeof(E) == 2 && RULE != kMemoryDelta)                                                             \
      if (parts > 1) {                                                                                                \
        hipLaunchKernelGGL((memory_steps_kernel<RULE, E, P, true>), grid, dim3(NT), bytes, s, blob, off_spans, a, *w,  \
                           limit, plan);                                                                              \
        break;                                                                                                        \
      }                                                                                                               \
    hipLaunchKernelGGL((memory_steps_kernel<RULE, E, P, false>), grid, dim3(NT), bytes, s, blob, off_spans, a,        \
                       w ? *w : none, limit, plan);                                                                   \
  } while (0)
  if (rows <= 1) FFMI_MS(1);
  else if (rows <= 2) FFMI_MS(2);
  else if (rows <= 4) FFMI_MS(4);
  else if (rows <= 8) FFMI_MS(8);
  else return hipErrorInvalidValue;
#undef FFMI_MS
  return hipGetLastError();
}

}  // namespace

hipError_t launch_memory_steps(const char *blob, int off_spans, int num_spans, const Memory &a,
                               const MemoryScratch *w, bool f32, int limit, bool *left, hipStream_t s) {
  *left = false;
  if (num_spans <= 0) return hipSuccess;
  if (bad_steps_shape(a) || limit < 1 || (w && (!w->o || (a.rule == kMemoryNormed && !w->gates)))) return hipErrorInvalidValue;
#define FFMI_MR(RULE)                                                                              \
  return f32 ? run_steps<RULE, float>(blob, off_spans, num_spans, a, w, limit, left, s)            \
             : run_steps<RULE, uint16_t>(blob, off_spans, num_spans, a, w, limit, left, s)
  if (a.rule == kMemoryGated) FFMI_MR(kMemoryGated);
  if (a.rule == kMemoryDelta) FFMI_MR(kMemoryDelta);
  FFMI_MR(kMemoryNormed);
#undef FFMI_MR
}

}  // namespace ffmi
