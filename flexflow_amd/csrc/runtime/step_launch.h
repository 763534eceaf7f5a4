// step_launch.h -- whether a step's kernels are launched one by one or as a captured graph.
#pragma once
#include <hip/hip_runtime.h>
#include <stdlib.h>

namespace ffmi {

// A graph's launch takes the host about 10 us before the first kernel starts, and the GPU
// a few more behind the last one; a kernel's own launch takes 3-4 us, which the kernels
// ahead of it cover if they run that long.  So a step goes one by one where its launches
// read 22 MB each (4 us at 5.5 TB/s, and 3 of latency).  Replays as graphs / one by one, in us,
// with the MB of a launch.  4096 channels: Fesenex (60) 21320 / 21120, Nomutar (70) 18140 / 18020, Vapipel (26)
// 11760 / 11690, 1 request 12250 / 12150.  2048: LLaMA, 4 requests of 1500 tokens (30) 11970 / 11850, in full
// precision (29) 5920 / 5880, Pekarax, 38 tokens a step (24) 7190 / 7000; but LLaMA, 1 request (21) 6600 / 6650
// and 6610 / 6560 on another machine, Fesenex, 1 request (17) 5950 / 6050, Vapipel (7) 6260 / 6860, and of 1024
// channels (2 - 4) 4370 / 5210 and 4440 / 5580.  (On a third machine Fesenex's and Pekarax's were the same
// either way.)  Not where threads are to yield or sleep (FFMI_SYNC): a graph
// costs the host less.
// FFMI_STEP_GRAPHS: 1 always graphs, 0 never (A/B, tests; read per call)
inline bool launch_one_by_one(double bytes, int launches) {
  if (const char *e = getenv("FFMI_STEP_GRAPHS")) return !atoi(e);
  if (bytes < 22e6 * launches) return false;
  unsigned flags = 0;
  if (hipGetDeviceFlags(&flags) != hipSuccess) return false;
  flags &= hipDeviceScheduleMask;
  return flags != hipDeviceScheduleYield && flags != hipDeviceScheduleBlockingSync;
}

}  // namespace ffmi
