// Host-side interface between the C-ABI layer and the templated HIP kernels.
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>
#include <vector>

#include "pof_types.hpp"

namespace pof {

// hipMalloc on the current device.  Where it has no room, the workspaces that finished calls left there for the next
// (pof_linear_filtsmooth, pof_smoothing, pof_ekf; of every context of the process) are given back first.
// Every allocation of device memory goes through it.
hipError_t device_malloc(void** p, size_t bytes);

constexpr int kMaxLevels = 40;
constexpr int kChunk = 256;  // time points (threads) per block of the smoothed means and the stage-1 reduction

// Optional per-kernel timing with HIP events (instrumented runs only).
constexpr int kMaxTimed = 256;
enum KernelClass : int {
  kKFilterLeaf = 0,
  kKFilterUp,
  kKFilterDown,
  kKFilterPost,
  kKSmoothUp,
  kKSmoothDown,
  kKSmoothPost,
  kKReduce,
  kKOutput,
  kNumKernelClasses
};
struct KernelTimer {
  int n = 0;
  hipEvent_t ev[kMaxTimed + 1];
  int cls[kMaxTimed];
  long long work[kMaxTimed];  // elements processed by the launch
  bool ready = false;
};

// Scan-level widths (combines per level, summed over the batch's IVPs) from which a scan level of a
// state dimension D <= 16 is a launch of its own; narrower levels, bound by the latency of one
// combine, share launches of up to kStageLevels levels.  The default is one wavefront of four
// combines on each of the chip's 1,024 SIMDs.
struct Tuning {
  int filter_up = 4096;
  int filter_down = 4096;
  int smooth_up = 4096;
  int smooth_down = 4096;
};

// A launch of a scan with one row per lane (D <= 16): nlev consecutive levels from l0 (the one with
// the most entries), in blocks of kStageWorkers workers.  Block b of an IVP owns the combines
// [b c, (b + 1) c) of each level, c = kStageWorkers >> (level - l0): in the up-sweep their inputs, in the
// down-sweep their prefixes, are the block's own (but for one prefix, that of everything before the block).
constexpr int kStageWorkers = 16;
// Blocks of an up-sweep stage up to which two workers share a combine (k_filter_up16): one block per CU, whose eight
// wavefronts are two per SIMD.
constexpr int kTwoBlocks = 256;
constexpr int kStageLevels = 5;  // kStageWorkers >> (kStageLevels - 1) = 1
struct Stage {
  int l0 = 0, nlev = 0;
  int off = 0, blocks = 0;  // table of blocks per IVP
  long long work = 0;       // combines
};

// Launch maps of one active set of a group (host view of a device int buffer):
// the active IVPs' records, then one prefix table per launch kind and level.
struct LaunchPlan {
  const int* dev = nullptr;  // device buffer
  IvpRec first{};            // the first active IVP's record
  int m = 0;                 // active IVPs
  int fl = 0, sl = 0;        // filter / smoother levels (maximum over the active IVPs)
  int leaf_off = 0, leaf_total = 0;    // per IVP: Ns work items
  int one_off = 0, one_total = 0;      // 1 (the first element)
  int leaf1_off = 0, leaf1_total = 0;  // Ns - 1 (the other elements)
  int pts_off = 0, pts_total = 0;      // Ns + 1
  int chunk_off = 0, chunk_total = 0;  // ceil((Ns + 1) / kChunk)
  // D <= 16: the stages of the four sweeps, in launch order
  int n_fup = 0, n_fdn = 0, n_sup = 0, n_sdn = 0;
  Stage fup[kMaxLevels], fdn[kMaxLevels], sup[kMaxLevels], sdn[kMaxLevels];
  // D > 16: a table per level
  int fup_off[kMaxLevels] = {}, fup_total[kMaxLevels] = {};  // Ns >> (l + 1)
  int fdn_off[kMaxLevels] = {}, fdn_total[kMaxLevels] = {};  // ((Ns >> l) + 1) / 2
  int sup_off[kMaxLevels] = {}, sup_total[kMaxLevels] = {};  // (Ns + 1) >> (l + 1)
  int sdn_off[kMaxLevels] = {}, sdn_total[kMaxLevels] = {};  // (((Ns + 1) >> l) + 1) / 2
  int fdn_ivps[kMaxLevels] = {}, sdn_ivps[kMaxLevels] = {};  // active IVPs that have level l
  LaunchMap map(int off, int total) const {
    return LaunchMap{reinterpret_cast<const IvpRec*>(dev), dev + off, m, total, first};
  }
};

// Kernel entry points per (D, d) instantiation, all over one group's active set.
struct EngineFns {
  int D, d;
  // one IEKS iteration for every active IVP: filter scan, smoother elements and
  // S statistics, smoother scan, smoothed means, objective, convergence
  // partials, and the per-IVP reduction into scal[a * 8 + 0..4] (a = active index)
  hipError_t (*iteration)(const GroupArgs& g, const LaunchPlan& p, double* scal, hipStream_t s, KernelTimer* t);
  // smoother scan with factors over the smoother elements of the last iteration
  hipError_t (*smooth_chol)(const GroupArgs& g, const LaunchPlan& p, hipStream_t s, KernelTimer* t);
  // project smoothed states into the caller's outputs (g.out_* tables, g.out_scale)
  hipError_t (*output)(const GroupArgs& g, const LaunchPlan& p, hipStream_t s);
  // filtered states of IVP ivp[0] (x0, then the level-0 filter prefixes)
  hipError_t (*filtered)(const GroupArgs& g, const LaunchPlan& p, double* fm, double* fL, hipStream_t s);
  // sequential filter + smoother iteration (at_pred: the EKF/EKS single pass)
  hipError_t (*seq_iteration)(const GroupArgs& g, const LaunchPlan& p, double* scal, int at_pred, hipStream_t s,
                              KernelTimer* t);
  hipError_t (*seq_smooth_chol)(const GroupArgs& g, const LaunchPlan& p, hipStream_t s, KernelTimer* t);
  // the smoother alone over filtered states in the filter prefix arrays (parallel or sequential)
  hipError_t (*smooth_only)(const GroupArgs& g, const LaunchPlan& p, double* scal, int sequential, hipStream_t s,
                            KernelTimer* t);
  // EK1 linearisation at n points: H [n, d, D], c [n, d]
  hipError_t (*linearize)(const ModelArgs& a, const double* m, int n, double* H, double* c, hipStream_t s);
  // linearisation of the given LinMethod at n states (m [n, D], L [n, D, D]):
  // H [n, dO, D], c [n, dO], R [n, dO, dO]; work: n * lin_work<D, d>() doubles
  hipError_t (*linearize_alt)(const ModelArgs& a, int method, const LinParams& p, const double* m, const double* L,
                              int n, double* H, double* c, double* R, double* work, hipStream_t s);
};

const EngineFns* find_engine(int D, int d);

}  // namespace pof
