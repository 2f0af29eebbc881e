// Internal: the launch plan of one compiled kernel (xg_kernel) and the helpers
// that turn one stencil statement into launch arguments.  Shared by the
// runtime (single calls) and the batch executor (many instances per launch).
#ifndef XGRID_KERNEL_H
#define XGRID_KERNEL_H

#include <array>
#include <cstdint>
#include <string>
#include <vector>

#include "xgrid_internal.h"

namespace xgi {

constexpr int kThreads = 256;
constexpr int kGroupThreads = 1024;
constexpr int64_t kFuseMaxCells = 4096;  // default of g_dev.fuse_max_cells (XGRID_FUSE_MAX_CELLS)
// A call with fewer launches runs them directly: replaying a graph takes 21 to 33 us of host time, three
// launches 12 (45^2 to 400^2, three statements, us a call: 21 and 12).  With a blocked loop among them the
// device time hides either way, and such calls stay graphs from three launches on (9^2 to 33^2
// cavities, all of whose calls are: 60 us a call, 57.5 made directly).
constexpr int64_t kGraphMinLaunches = 4, kGraphMinLaunchesLoop = 3;
// Store grids of which two levels do not fit the 256 MB last-level cache (Infinity Cache) take
// non-temporal stores in 3-D box tiles: by the time the next update reads a cell it has left the
// cache anyway, and the write stream drains faster.  The line lies where both ways meet (heat
// update, us, plain / non-temporal): 125 MiB FP32 59 / 67, 128 MiB FP64 47 / 54, 141 MiB FP64
// 66 / 64, 141 MiB FP32 86 / 82, 178 MiB 97 / 92, 200 MB FP64 97 / 89.
constexpr size_t kStreamBytes = (size_t)128 << 20;
// Freed grid memory the device pool keeps for reuse (beyond it, memory goes back at
// the next synchronisation).
constexpr uint64_t kPoolKeepBytes = (uint64_t)16 << 30;

// kRecord: the stub's statements are recorded for a batched launch instead of run
enum CallMode { kDirect = 0, kCapture = 1, kReplay = 2, kRecord = 3 };

struct StmtPlan {
  xg_stmt_desc d;
  uint64_t haz_version = 0;
  bool haz = false;
};

struct Pending {
  int32_t sid;
  size_t off;   // offset of its params in the arena
  int64_t bytes;
};

struct GraphEntry {
  std::vector<uint8_t> key;
  uint64_t hash = 0;
  int seen = 0;
  hipGraphExec_t exec = nullptr;
  bool direct = false;          // the call launches too little for a graph to pay: run it directly
  std::vector<std::vector<void*>> post_levels;
  std::vector<void*> post_scratch;
  uint64_t last_use = 0;
};

struct EventPair {
  hipEvent_t a, b;
};

// How the launches of a blocked loop on wave tiles cut a grid: which tile, waves per
// workgroup, halo, tiles per axis, and the iterations of the longest launch.
struct WaveCut {
  int32_t tile = 0, waves = 0, halo = 0, nt0 = 1, nt1 = 1, iters = 0;
  int64_t blocks() const { return (int64_t)nt0 * nt1; }
};

// What is known about a blocked loop on one mask.  A mask's version is drawn anew each time a
// grid's mask is set or a grid is made, so it names one grid and one mask for good.
struct LoopProof {
  uint64_t mask_version = 0;
  int state = 0;                // 1 exact, 0 unknown, -1 declined
  int validated = 0;            // state 1: launches of at most this many iterations are proven exact
  uint8_t reach[XG_WAVE_MAX_ITERS] = {};   // wave tiles, state 1: the halo that 1, 2, ... iterations need
};
// A program that alternates between grids keeps the proofs of this many masks per loop (a
// check costs a launch and a synchronisation).
constexpr size_t kLoopProofs = 32;

struct LoopPlan : LoopProof {
  xg_loop_desc d;
  std::vector<LoopProof> others;   // other masks' proofs, most recent first
  WaveCut cut;                     // wave tiles: the cut of the launches being made
  bool outrun = false;             // wave tiles: the last call's iterations needed too wide a halo (wave_outrun)
  // wave tiles: the cut last chosen for one grid, and what it was chosen for (choosing takes the
  // host 13 us, as long as two launches)
  WaveCut chosen;
  int32_t chosen_n0 = 0, chosen_n1 = 0;
  int64_t chosen_trip = 0;
  uint8_t chosen_reach[XG_WAVE_MAX_ITERS] = {};
  int64_t launches = 0, iterations = 0;
  std::vector<std::vector<uint8_t>> last_params;
};

// One recorded stub event: a statement (kind 0) or a whole blockable loop (kind 1).
struct Rec {
  int32_t kind;
  int32_t id;         // statement id or loop id
  int64_t trip;       // loop iterations
  size_t off;         // parameter block(s) in the record arena, 8-byte aligned each
};

}  // namespace xgi

struct xg_kernel {
  std::vector<xgi::StmtPlan> stmts;
  std::vector<xg_group_desc> groups;
  std::vector<xg_fan_desc> fans;
  std::vector<int32_t> fan_of;      // statement -> its fan, or -1 (empty: no fans)
  int32_t ngrids = 0;
  std::vector<xg_grid*> grids;
  int status = XG_OK;
  std::string status_msg;
  int mode = xgi::kDirect;
  xgi::GraphEntry* cur = nullptr;
  std::vector<xgi::Pending> pending;
  std::vector<uint8_t> arena;
  int32_t pending_group = -1;
  std::vector<xgi::Pending> run_buf;   // flush's working list (kept for its capacity)
  bool graphs = true, fuse = true;
  bool graphs_auto_off = false;
  int64_t graph_misses = 0, graph_hits = 0;
  std::vector<xgi::GraphEntry> cache;
  uint64_t tick = 0;
  int64_t n_launch = 0, n_fused = 0, n_replay = 0, n_capture = 0;
  int64_t capture_mark = 0;         // n_launch when the current capture began
  bool capture_loop = false;        // a blocked loop is in the current capture
  std::unique_lock<std::recursive_mutex> recording;   // held (g_recording) while this kernel's call is captured
  int32_t timed_sid = -1;
  std::vector<xgi::EventPair> events;
  std::vector<xgi::LoopPlan> loops;
  bool blocked = true;
  int32_t* d_fail = nullptr;        // answer of checking launches (kCheckBytes)
  std::vector<int64_t> exec_count;  // stmt() calls per statement (all modes)
  std::vector<std::vector<uint8_t>> last_params;  // parameters of each statement's last call
  std::vector<uint8_t> key_buf;
  bool record_next = false;         // the next call through the stub is recorded (batches)
  std::vector<xgi::Rec> rec;        // recorded events of the last recorded call
  std::vector<uint8_t> rec_arena;
};

namespace xgi {

extern const xg_api g_api;   // the stub function table
uint64_t fnv1a(const uint8_t* p, size_t n);
int set_status(xg_kernel* k, int code);
int effective_mode(xg_kernel* k, StmtPlan& sp);
void fill_dom(xg_dom& dom, const ClassPlan& p, const xg_grid* G, int32_t klass);
void fill_view(xg_gview& v, const xg_grid* G, void* ptr);
bool uniform_refs(xg_kernel* k, const xg_stmt_desc& d);
int32_t stream_flag(const xg_grid* G);
int fill_refs(xg_kernel* k, const xg_stmt_desc& d, std::vector<xg_gview>& refs);
// Workgroups over the box [lo, hi) for a statement's tile; cols3 = columns of a 3-D tile.
int64_t tiles_for(int D, const int32_t* lo, const int32_t* hi, int cols3 = 64);
int64_t blocks_for_dom(int D, const xg_dom& dom, int cols3 = 64);
// The 3-D tile width of a statement's run_main kernels (fn_main, fn_main_b).
int tile3_cols(const xg_stmt_desc& d);
int ensure_scratch(xg_kernel* k);
// Can loop `lid` run blocked on the bound grids (aliasing), and is its plan for
// the grid's current mask known?  Resets the plan when the grid or mask changed.
bool loop_blockable(xg_kernel* k, LoopPlan& L);
void fill_tb_hdr(xg_kernel* k, LoopPlan& L, xg_tb_hdr& TH, int iters, int32_t* fail_flag);
// A grid to be cut into wave tiles: its shape, and the halo that 1, 2, ... iterations need.
struct WaveShape {
  int32_t n0, n1;
  const uint8_t* reach;
};
inline WaveShape wave_shape(const xg_grid* G, const LoopProof& p) { return {G->shape[0], G->shape[1], p.reach}; }
// The tile, waves and iterations with which the launches for `trip` iterations run all `shapes`
// (`batch`: as one batched launch).  waves = 0: no tile holds the loop.
WaveCut wave_choose(const xg_loop_desc& d, const std::vector<WaveShape>& shapes, int64_t trip, bool batch);
// ... with the halo and tile counts of one grid.
WaveCut wave_cut_for(const xg_loop_desc& d, WaveCut c, const WaveShape& s);
// Header of a mask's checking launch, and what its answer (XG_WAVE_MAX_ITERS numbers) says.
void fill_wave_check(xg_kernel* k, LoopPlan& L, xg_tb_hdr& TH, int32_t* answer);
void wave_answer(LoopPlan& L, const int32_t* answer);
// Is a call to be left to plain launches: a launch of its trip iterations (at most tmax) would need
// too wide a halo?  Fewer iterations may still run blocked, so the proof keeps what each count needs.
bool wave_outrun(const LoopPlan& L, int64_t trip);
constexpr size_t kCheckBytes = XG_WAVE_MAX_ITERS * sizeof(int32_t);   // answer of a checking launch
constexpr int kWaveCheckThreads = 1024;
constexpr int64_t kWaveSingleIters = 1024;   // most iterations of a launch when one tile holds a grid

}  // namespace xgi

#endif
