// mbir_host.h -- host-side state of the engine shared by the C-ABI (mbir_capi.cpp)
// and the request server (mbir_serve.cpp): the context, one job's device buffers
// and the sweep helpers both drive.
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <cstdio>
#include <memory>
#include <mutex>
#include <vector>

#include "../../include/mbir_tem.h"
#include "mbir_internal.h"

#define HIP_TRY(expr)                                                                    \
  do {                                                                                   \
    hipError_t _e = (expr);                                                              \
    if (_e != hipSuccess) {                                                              \
      std::fprintf(stderr, "mbir: HIP error %s at %s:%d: %s\n", hipGetErrorName(_e),    \
                   __FILE__, __LINE__, #expr);                                           \
      return MBIR_ERR_HIP;                                                               \
    }                                                                                    \
  } while (0)

// Memory that a context and its jobs share (the last of them gives it back): one block of
// device scratch, at most kScratchKeep bytes, and 16 MB of pinned staging, both made on
// first use.  One caller at a time holds either; any other falls back to an allocation of
// its own and to a plain copy.  The scratch of a larger call is freed at its end: 64 MiB hold
// the projection and the volume of 512x64x256 at 91 views, whose two allocations cost 0.8 ms
// of a 3 ms call; a larger call spends a smaller part on them.
struct mbir_pool {
  static constexpr size_t kScratchKeep = (size_t)64 << 20;
  static constexpr int kCopyThreads = 4;
  static constexpr size_t kCopyChunk = (size_t)2 << 20;
  int device = 0;
  std::mutex scratch_mu, stage_mu;
  char* scratch = nullptr;
  size_t scratch_bytes = 0;
  char* stage = nullptr;  // 2 chunks per copying thread
  hipEvent_t ev[2 * kCopyThreads] = {};
  hipError_t make_stage();  // with stage_mu held
  // hipMalloc; when the card is full, again without the scratch block
  hipError_t device_alloc(void** p, size_t bytes);
  // gives the scratch block back if it is larger than `room` and no call uses it (a call that
  // does is charged for it elsewhere, and its end is the time to ask again)
  void trim(size_t room);
  // dst = src (device) of stream s, there when it returns (dst: host memory; device memory is
  // taken too, as a plain copy does)
  hipError_t copy_out(void* dst, const void* src, size_t bytes, hipStream_t s);
  ~mbir_pool();
};

template <typename T>
struct DevBuf {
  T* p = nullptr;
  size_t n = 0;
  bool own = true;  // false: part of a DevArena
  hipError_t alloc(mbir_pool& pool, size_t count)
  {
    n = count;
    own = true;
    return pool.device_alloc((void**)&p, std::max<size_t>(count, 1) * sizeof(T));
  }
  void release()
  {
    if (p && own) (void)hipFree(p);
    p = nullptr;
  }
};

// Buffers that live and die together, laid out in one device allocation: mapping and
// unmapping one of 4 .. 200 MB costs 0.1 .. 0.25 ms each way whatever its size, and a job
// has thirty.
class DevArena {
 public:
  template <typename T>
  void add(DevBuf<T>& b, size_t count)
  {
    b.n = count;
    b.own = false;
    parts_.push_back({reinterpret_cast<void**>(&b.p), bytes_});
    bytes_ += (std::max<size_t>(count, 1) * sizeof(T) + 255) & ~(size_t)255;
  }
  hipError_t alloc(mbir_pool& pool)  // places every buffer added so far
  {
    const hipError_t e = pool.device_alloc((void**)&p_, std::max<size_t>(bytes_, 256));
    for (const Part& q : parts_) *q.p = e == hipSuccess ? p_ + q.at : nullptr;
    return e;
  }
  ~DevArena()
  {
    if (p_) (void)hipFree(p_);
  }

 private:
  struct Part {
    void** p;
    size_t at;
  };
  std::vector<Part> parts_;
  size_t bytes_ = 0;
  char* p_ = nullptr;
};

// Device scratch for the duration of one call on stream s.
class Scratch {
 public:
  Scratch(mbir_pool& p, hipStream_t s) : pool_(p), s_(s) {}
  Scratch(const Scratch&) = delete;
  hipError_t take(size_t bytes);
  char* p() const { return p_; }
  ~Scratch();

 private:
  mbir_pool& pool_;
  hipStream_t s_;
  char* p_ = nullptr;
  bool held_ = false;
};

using mbir::DevJob;
using mbir::SweepAccum;
using mbir::MixEntry;
using mbir::LineRef;

struct mbir_ctx {
  int device = 0;
  int verbose = 0;
  uint64_t budget = 0;
  std::mutex mu;
  std::shared_ptr<mbir_pool> pool = std::make_shared<mbir_pool>();
  hipStream_t stream = nullptr;  // stream of batched launches
  DevBuf<DevJob> djobs;          // job table of a batched sweep
  DevBuf<MixEntry> ents;       // entry table of a batched sweep
  mbir::LineTuning tune;         // form of the batched line kernels per shape and size
  // autotuning: when set, batched sweeps force this form (0 / 1) and time each launch
  struct Probe {
    int force = -1;
    std::vector<hipEvent_t> ev;       // two per launch
    std::vector<int> ypl, nv, nwg;    // per launch
  }* probe = nullptr;
  ~mbir_ctx()
  {
    djobs.release(); ents.release();
    if (stream) (void)hipStreamDestroy(stream);
  }
};

struct mbir_job {
  mbir_ctx* ctx = nullptr;
  std::shared_ptr<mbir_pool> pool;
  mbir_problem prob{};
  mbir_geometry g{};
  hipStream_t stream = nullptr;
  DevJob J{};
  double offsetR = 0, offsetT = 0;
  int spacing = 1;  // conflict-free x spacing of lines in one step
  int ysplit = 1;   // y-slabs of the schedule: a step updates one unit (line, slab) per
                    // line of its row class in every slab (1 = whole lines)
  int zshift = 0;   // z offset between the row classes of neighbouring slabs in a step
  size_t sched_cap() const { return (size_t)g.N_z * g.N_x * ysplit; }
  std::vector<double> angles_rad, H;
  std::vector<double> I0h, muh, alphah;
  // device buffers: all but those of the graph and the column table in `arena`, the column
  // table (its size is known later) in `columns`
  DevArena arena, columns;
  DevBuf<float> x, e, y, wview, vlr_val;
  DevBuf<mbir::VoxelProfile> prof;  // per view: corners of the voxel profile
  DevBuf<double> cosv, sinv, Hd, beam, I0, mu, alpha, I0b, mub, sums6, cost;
  DevBuf<int2> vlr_p;
  DevBuf<int> vlr_t0, vlr_n, line_nnz, col_ptr, col_row;
  DevBuf<LineRef> sched;
  DevBuf<float> col_a, col_ka, col_kw;
  DevBuf<double> line_kk;  // per line: the column factor of theta2 (plain weights)
  DevBuf<float> wfull;       // bright field: per-entry weights, sign = selector
  DevBuf<float> bfs;         // HAADF with a bright-field sinogram: per-element scale
  DevBuf<double> alpha_b;    // bright field: the next shared variance
  double bragg = 0;          // bright field: current Bragg threshold
  std::vector<int> nnz_h;  // per-line column entries (host copy)
  unsigned int bad_counts = 0;  // bright-field setup: counts that are not positive
  int64_t nnz_total = 0;
  DevBuf<uint8_t> mask;
  DevBuf<SweepAccum> acc;
  DevBuf<mbir::UnitStat> ustat;  // per schedule position: the unit's sweep statistics
  DevBuf<double> red;             // block sums of the statistics (5 kReduceBlocks)
  // the sweep's schedule: step k is row class step_class[k] (empty: listed lines, in
  // sched_h), its units [step_ptr[k], step_ptr[k + 1]); sched_h then holds the list only in a
  // graph's sweeps (fill_schedule)
  std::vector<int> step_class, step_ptr;
  std::vector<int> class_n;   // units of every row class
  std::vector<int> steps_h;   // step_class and step_ptr as uploaded to `steps`
  DevBuf<int> steps;
  std::vector<LineRef> sched_h;
  int units() const { return step_ptr.empty() ? 0 : step_ptr.back(); }
  std::vector<int> cptr_h;  // column-table offsets of all lines (host copy)
  // bright-field NHICD: per-line update magnitudes, the seeded random list of all
  // lines, and the ROI mask on the host
  DevBuf<float> magmap;
  std::vector<float> magmap_h;
  std::vector<int> nh_all;
  std::vector<uint8_t> mask_h;
  // reach[d + N_z - 1]: the least x distance at which a line d rows away never shares a
  // detector bin with this one (every view) nor is a prior neighbour; subadditive in d
  std::vector<int> nh_reach;
  // the conflict-free steps of each homogeneous part (fixed lists: packed once)
  std::vector<std::vector<std::vector<int>>> nh_parts;
  int nh_log_on = 0;                 // record the lines of every NHICD call
  std::vector<int> nh_log;           // lines of all calls of the last run
  std::vector<int64_t> nh_log_ptr;   // call c: nh_log[nh_log_ptr[c] .. nh_log_ptr[c + 1])
  // kernel_mode 3: the sweep's step launches as a HIP graph over a padded schedule
  // (step k's lines at gsched[k * graph_lines], unused entries line = -1)
  DevBuf<LineRef> gsched;
  std::vector<LineRef> gsched_h;
  hipGraph_t graph = nullptr;
  hipGraphExec_t graph_exec = nullptr;
  DevJob graph_J{};
  int graph_steps = 0, graph_lines = 0;
  std::atomic<int> cancel{0};
  int timing = 0;
  int sweep_counter = 0;
  double stop_threshold = 0;
  double sigma_x = 0;  // current prior scale (TomoInputs::SigmaX), re-estimated with estimate_prior
  int64_t bytes = 0;
  ~mbir_job()
  {
    gsched.release(); ustat.release();  // a graph's own
    if (graph_exec) (void)hipGraphExecDestroy(graph_exec);
    if (graph) (void)hipGraphDestroy(graph);
    if (stream) (void)hipStreamDestroy(stream);
  }
};

namespace mbir {

// Sweep helpers (mbir_capi.cpp).  prepare_sweep builds the seeded step schedule
// of the job's next sweep, uploads it and clears the sweep accumulators on stream s;
// sweep_status applies the stop test to the accumulators (1 continue, 0 converged)
// and counts the sweep; nuisance_update_on enqueues joint estimation, the noise
// update and the column-weight refresh on s without waiting.
void build_schedule(mbir_job* j, bool drop_empty_steps);
void fill_schedule(mbir_job* j);
const LineRef* step_refs(const mbir_job* j, int k, LineRef* buf);
int prepare_sweep_on(mbir_job* j, hipStream_t s, int* steps);
int sweep_status(mbir_job* j, const SweepAccum& a, double ms, mbir_sweep_stats* st);
int nuisance_update_on(mbir_job* j, hipStream_t s);
// Bright field: the Bragg threshold used by the next launches (DevJob fields).
void set_bragg(mbir_job* j, double T);
// QGGMRF constants of the prior scale sigma_x (DevJob fields).
void set_prior(mbir_job* j, double sigma_x);

}  // namespace mbir
