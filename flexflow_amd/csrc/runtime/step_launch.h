// step_launch.h -- whether a step's kernels are launched one by one or as a captured graph.
#pragma once
#include <hip/hip_runtime.h>
#include <stdlib.h>

#include <map>

#include "../ffmi_internal.h"

namespace ffmi {

// A graph's launch takes the host about 10 us before the first kernel starts, and the GPU
// a few more behind the last one; a kernel's own launch takes 3-4 us, which the kernels
// ahead of it cover if they run that long.  Replays as graphs / one by one, in us, with the
// MB that the step reads a launch, in processes of their own.  4096 channels: Fesenex (73) 21320 / 21120,
// Vapipel, 1 request (31) 12100 / 11890.  2048: LLaMA in full precision (33) 5915 / 5840, Nomutar, 8 requests (28)
// 9640 / 8835, Pekarax, 38 tokens a step (25) 7150 / 7150 and 7110 / 7000; LLaMA, 12 requests (23) 8860 / 7560, 8
// (22) 6010 / 5900, 1 (22) 6450 / 6460; Nomutar, 4 (22) 10400 / 9810; Fesenex, 8 (20) 5970 / 5810, 1 (20) 6140 / 6120;
// Pekarax, 3 (17) 6120 / 5950, LLaMA, 43 tokens a step (16) 13380 / 11780, SpecInfer (16) 5830 / 5860; Fesenex, 47
// tokens (13) 8810 / 8630, Pekarax, 1 request (11) 4860 / 4930, Vapipel, 2 (9) 6720 / 7180; of 1024
// channels (2 - 4) 4370 / 5210 and 4440 / 5580.  On other machines single requests of 20 - 22 MB were 1.7 % slower to 0.8 %
// faster one by one.  So from 14 MB on, half as much again as the clear losses read: there
// one by one is within 1 % of a graph or faster, and a new shape's first step needs no graph made
// (SpecInfer of 2048 channels, 3 tokens 3080 / 2750).  (Most of what LLaMA's 12 and 14 requests gain is
// that the caller's fresh pages for their logits cost more beside a graph: with kept ones 6650 / 6510 and
// 11510 / 11320.)
// A busy host pays for it only where it has no core left: LLaMA of 2048 channels, 1 request (22) 6421 / 6407,
// beside 8 busy threads of 16 cores 6446 / 6406, beside 15 6433 / 6546; Pekarax, 3 requests 4705 / 4584, 4759 / 4617 and
// 4946 / 4873.
// Not where threads are to yield or sleep (FFMI_SYNC): a graph costs the host less.
// FFMI_STEP_GRAPHS: 1 always graphs, 0 never (A/B, tests; read per call)
// (bytes: what the step reads, 0: a graph whatever it is; launches: its kernels)
inline bool launch_one_by_one(double bytes, int launches) {
  if (bytes <= 0) return false;
  if (const char *e = getenv("FFMI_STEP_GRAPHS")) return !atoi(e);
  if (bytes < 14e6 * launches) return false;
  unsigned flags = 0;
  if (hipGetDeviceFlags(&flags) != hipSuccess) return false;
  flags &= hipDeviceScheduleMask;
  return flags != hipDeviceScheduleYield && flags != hipDeviceScheduleBlockingSync;
}

// The graph of a step shape (none where it is launched one by one), and its kernels, which
// are counted where it is captured: their number goes with the form that the step takes.
struct StepGraph {
  hipGraphExec_t exec = nullptr;
  int launches = 0;
};
template <class Key>
void clear_step_graphs(std::map<Key, StepGraph> *graphs) {
  for (auto &kv : *graphs)
    if (kv.second.exec) (void)hipGraphExecDestroy(kv.second.exec);
  graphs->clear();
}
template <class Key>
long count_step_graphs(const std::map<Key, StepGraph> &graphs) {
  long n = 0;
  for (const auto &kv : graphs) n += kv.second.exec != nullptr;
  return n;
}
// *exec: the graph to launch for a step that reads `bytes`, of enqueue()'s work; null: enqueue
// it.  bound: launches that its form does not exceed; a step that goes one by one even with
// those is not captured.
template <class Key, class Enqueue>
ffmi_status step_graph(std::map<Key, StepGraph> *graphs, size_t most, const Key &key, double bytes, int bound,
                       hipStream_t stream, Enqueue &&enqueue, hipGraphExec_t *exec) {
  *exec = nullptr;
  if (launch_one_by_one(bytes, bound)) return FFMI_OK;
  auto it = graphs->find(key);
  if (it == graphs->end() || (!it->second.exec && !launch_one_by_one(bytes, it->second.launches))) {
    if (graphs->size() >= most) {
      FFMI_HIP(hipStreamSynchronize(stream));  // (a step ahead of this one may run from one)
      clear_step_graphs(graphs);
    }
    hipGraph_t g = nullptr;
    FFMI_HIP(hipStreamBeginCapture(stream, hipStreamCaptureModeThreadLocal));
    const ffmi_status st = enqueue();
    const hipError_t ce = hipStreamEndCapture(stream, &g);
    size_t nodes = 0;
    hipError_t e = ce;
    StepGraph made;
    if (st == FFMI_OK && e == hipSuccess) e = hipGraphGetNodes(g, nullptr, &nodes);
    made.launches = (int)nodes;
    if (st == FFMI_OK && e == hipSuccess && !launch_one_by_one(bytes, made.launches))
      e = hipGraphInstantiate(&made.exec, g, nullptr, nullptr, 0);
    if (g) (void)hipGraphDestroy(g);
    if (st != FFMI_OK) return st;
    FFMI_HIP(e);
    it = graphs->insert_or_assign(key, made).first;
  }
  if (!launch_one_by_one(bytes, it->second.launches)) *exec = it->second.exec;
  return FFMI_OK;
}

}  // namespace ffmi
