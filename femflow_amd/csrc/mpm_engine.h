// Host-side engine object behind the mpm_ctx handle of the C ABI.
#pragma once
#include <hip/hip_runtime.h>

#include <map>
#include <string>
#include <tuple>
#include <vector>

#include "mpm355.h"
#include "mpm_engine_kernels.h"

namespace mpm {

void set_error(const std::string& msg);

// A captured segment fixes the particle count (launch grids, sort sizes),
// the segment length, whether it rebins first, which state buffer is current,
// the sums destination, and whether it continues the run's previous segment
// (cont) and ends the run (fin), whether it reads uploaded records, the
// substep of the segment it starts at, and which speed counts it sends; any
// of them changing needs another graph.
struct GraphKey {
  int64_t n;
  int len, parity, bin;
  uintptr_t sums;
  int nsteps, cont, fin, records, k0, speeds;
  bool operator<(const GraphKey& o) const {
    return std::tie(n, len, parity, bin, sums, nsteps, cont, fin, records, k0, speeds) <
           std::tie(o.n, o.len, o.parity, o.bin, o.sums, o.nsteps, o.cont, o.fin, o.records, o.k0, o.speeds);
  }
};
// Captured graphs kept per context; beyond this the cache is emptied first.
constexpr size_t MAX_GRAPHS = 32;
// Shortest rebin cadence the engine takes by itself.
constexpr int MIN_CADENCE = 8;
// Substeps for which a cadence below sort_every holds without new counts.
// Bodies that slowed down since would pay for rebins that they do not need: at
// most 24 of some 75 us (a run of 1,000 substeps of a body that stops early
// would pay for 125).  Bodies that stay fast go on as with sort_every until a
// run that reads counts (after a counter was read, as Engine.run does).
constexpr int CADENCE_HOLDS = 192;

struct CorrExtract {
  uint16_t* X;      // rows x 352 BF16 features
  uint32_t* nodes;  // global node index (block * 64 + node in block)
  float* vel;       // rows x 3 updated grid velocity
  int64_t max_rows;
};

// Per-substep state output (caller order): slot k of each array receives the
// state after substep k.  grids (optional, single-scene engines): slot k of
// 7 (res+1)^3 floats receives substep k's dense grids, the P2G momentum
// ((res+1)^3 x 3), the P2G mass ((res+1)^3) and the updated velocity
// ((res+1)^3 x 3), zero at nodes no particle reached.
struct StateSink {
  float *x, *v, *F, *C, *Jp;
  float* grids;
};

struct TimedLaunch {
  int kind;  // 0 P2G, 1 G2P2G, 2 G2P, 3 grid update
  hipEvent_t e0, e1;
  int launches;  // 0: a part of the launch that follows
};

struct Engine {
  // configuration
  int device = 0, num_cus = 256;
  int64_t n_max = 0, n = 0, total_blocks = 0;
  int nmat = 1;
  int chunk = 512, sort_every = 48, grid_mult = 8;  // the measured headline optimum
  int spread = 9;  // scatter start offsets per cell (3 or 9, see transfer_kernel)
  // fused passes take chunks from per-XCD ticket queues (set for engines of
  // 8 or more scenes, whose many uneven chunks the queue balances)
  bool dyn_sched = false;
  // the chunk list in use was built without regard to rows (see FEW_ROWS in
  // mpm_sort.hip), as the corrector needs it
  bool chunks_plain = false;
  // substeps between rebins for the speeds last seen (cadence_of; 0: none
  // seen, sort_every applies, which also bounds it)
  int cadence = 0;
  int cadence_left = 0;  // substeps for which it still holds; taken back at a rebin
  // Counts for the next run that is long enough to use them: none, of the last
  // run (the host has waited for it, or it was too short to use the ones that it
  // found), of an upload
  enum { SPEEDS_NONE, SPEEDS_RUN, SPEEDS_UPLOAD } speeds_at = SPEEDS_NONE;
  const uint32_t* speeds_from = nullptr;  // see EngineArgs; set while a probing segment is enqueued
  // a run's first kernel may still send its counts to h_speeds: the host's wait
  // for them ran out.  Until they are there no other run asks for counts, so that
  // what arrives is always the asking run's own.
  bool speeds_pending = false;
  // set while a segment with per-substep state output is enqueued: the fused
  // pass then writes v and C every substep
  bool store_vc = false;
  bool use_graph = true, timing = false;
  // substeps run since the particles were last binned; -1: not binned (after
  // an upload or a rebin request), so the next segment rebins first
  int since_bin = -1;
  int last_list = 0;  // active-block list the last substep's P2G appended to
  std::vector<SceneDev> scenes_host;
  // streams and graphs
  hipStream_t user_stream = nullptr, own_stream = nullptr;
  hipEvent_t ev_in = nullptr, ev_out = nullptr;
  std::map<GraphKey, hipGraphExec_t> graphs;
  std::vector<hipEvent_t> tevents;
  size_t tnext = 0;
  std::vector<TimedLaunch> tpairs;
  // device memory
  std::vector<void*> allocs;
  EngineState st[2] = {};
  int cur = 0;
  // The uploaded particles are still records (in d_rec; st[0] has only their x and
  // attr, for the rebin's keys); the first rebin moves them into st[1].  tiled()
  // unpacks them into st[0] instead, for calls that read the state before, and
  // for callers that capture.
  bool in_records = false;
  // 128 bytes per particle, of an upload or on a large download's way out.  Memory
  // of its own: a graph of the caller's may read either state copy at any time.
  float4* d_rec = nullptr;
  // something of this engine went into a graph of the caller's.  Its replays start
  // from the state that was there, so from then on (and within the capture) uploads
  // end in st[0] as tiles, and downloads leave d_rec, which holds the last upload,
  // alone.
  bool captured = false;
  SceneDev* d_scenes = nullptr;
  MatParams* d_mats = nullptr;
  int* d_block_scene = nullptr;
  float4* d_acc = nullptr;
  float4* d_vel = nullptr;
  uint32_t *d_flags = nullptr, *d_list = nullptr, *d_bstart = nullptr, *d_bend = nullptr;
  uint32_t* d_counters = nullptr;
  unsigned long long *d_oob = nullptr, *d_fallback = nullptr;
  uint32_t* d_speeds = nullptr;
  uint32_t* h_speeds = nullptr;  // pinned: totals per class, then the sent flag
  int4* d_chunks = nullptr;
  int4* d_split = nullptr;  // engines of many scenes: see EngineArgs::split
  int64_t chunk_cap = 0;
  uint32_t *d_nchunks = nullptr, *d_keys = nullptr, *d_vals = nullptr,
           *d_bocc = nullptr, *d_part = nullptr;
  uint32_t* d_sorted_keys = nullptr;
  // sort permutation of the last rebin, consumed by the next P2G (which
  // moves the particles into binned order); null once consumed
  const uint32_t* pending_perm = nullptr;
  uint32_t* d_hard = nullptr;
  uint32_t *d_cand_list = nullptr, *d_cand_flag = nullptr;
  uint2* d_cand_src = nullptr;
  float4* d_stage = nullptr;
  // learned corrector
  bool corr_on = false;
  float corr_mref = 1.f, corr_vref = 1.f;
  float4* d_pm = nullptr;
  float4* d_cellf = nullptr;
  float* d_corr_params = nullptr;
  uint16_t* d_corr_packed = nullptr;
  uint32_t* d_corr_count = nullptr;
  // sticky half-space colliders (all scenes, at most MAX_PLANES)
  std::vector<PlaneDev> planes_host;
  PlaneDev* d_planes = nullptr;
  uint32_t stage_cap = 0;
  uint32_t *d_bfirst = nullptr, *d_bcount = nullptr;
  void* d_ws = nullptr;
  size_t ws_bytes = 0;

  ~Engine();
  void release();
  int alloc(void** p, size_t bytes);
  int init(int64_t n_max, int nscenes, const mpm_scene* sc, int nmat, const mpm_material* mats);
  // small chunks in launches of their own
  bool split_small() const { return d_split && chunk == 512 && spread == 9; }
  EngineArgs args(double* sums, int max_steps, int sel) const;
  int upload(const mpm_particles* p, const int32_t* scene_ids);
  int download(mpm_particles* p);
  void tiled();
  bool capturing();  // whether the caller's stream is (noted in `captured`)
  // rebin; also starts the segment of len substeps (counters, sums index;
  // keep_speeds: not the speed counts, for a segment that is no part of a run)
  void enqueue_bin(hipStream_t s, int len, int with_sums, bool keep_speeds = false);
  void enqueue_segment(int k0, int len, bool bin, hipStream_t s, double* sums, int max_steps, float* frames,
                       int64_t step0, const StateSink* sink, bool cont, bool fin);
  // destroy every captured graph (after anything they baked in changes)
  void drop_graphs();
  int active_blocks(int64_t* out);
  void enqueue_frame(hipStream_t s, float* frames, int64_t step);
  void enqueue_state(hipStream_t s, const StateSink* sink, int64_t step);
  int positions(float* x);
  // separate_deferred: finish the FP64-deferred particles in their own
  // launch right after the transfer (needed where something reads the
  // particles before the grid update, and after the last G2P); otherwise
  // the following launch_grid(..., deferred = 1) finishes them
  void launch_transfer(int mode, hipStream_t s, const EngineArgs& a, bool separate_deferred = true);
  void launch_grid(hipStream_t s, const EngineArgs& a, int with_sums, int len, int k, int deferred = 0);
  void fill_u32(hipStream_t s, uint32_t* p, int64_t count, uint32_t v);
  void launch_cellf(hipStream_t s, const EngineArgs& a);
  // corrector after a grid update; ex != null: write features instead (sampling)
  void launch_corrector(hipStream_t s, const EngineArgs& a, const struct CorrExtract* ex);
  int set_corrector(const float* params, float m_ref, float v_ref, int enable);
  int corrector_sample(uint16_t* X, uint32_t* nodes, float* vel, int64_t max_rows, int64_t* rows);
  int grid_velocity(const uint32_t* nodes, int64_t count, float* out);
  int set_planes(int scene, int count, const double* points, const double* normals, int quirks);
  hipEvent_t tevent();
  int cadence_of(const uint32_t* counts) const;
  int run(int nsteps, double* sums, float* frames = nullptr, const StateSink* sink = nullptr);
  int take_counter(int which, int64_t* out);
  int particle_sums(double* out);
  int kernel_times(double* ms, int64_t* counts);
};

}  // namespace mpm
