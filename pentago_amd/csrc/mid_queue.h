// Batched midsolve plans (host side); the kernels live in mid_queue.hip.
//
// A batch is split by size.  Small boards (at most small_spots empty cells) are solved whole
// by one workgroup each: a persistent kernel whose workgroups pop board indices from a device
// queue (one atomic counter) and sweep every tile of the board (mid_tiles.h) with workgroup
// barriers between its steps, in a workspace slot owned by the workgroup.  No workgroup ever
// waits for another.  Large boards run step by step on one or more streams of their own (wins
// tables, then one launch per step over the whole device), boards of one stream reusing that
// stream's slot in stream order.
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>
#include <vector>

#include "device.h"
#include "mid.h"

namespace pe {

// A board's descriptor: what its kernels read and write.
struct MidBoardDev {
  MidInfo I;
  uint64_t* wins;           // [mover of the root, other][mask of empty cells]: halves of parity 0, 1
  uint64_t* spill;          // tile entries that the workspace has no room for
  uint64_t* work;           // tile entries, 4 u64 each
  pe_halfsupers* results;   // 19 entries
};

struct MidConfig {
  int64_t budget;        // bytes one run may hold (tables, workspaces, descriptors)
  int32_t small_spots;   // boards with at most this many empty cells: one workgroup each
  int32_t workgroups;    // persistent workgroups of the small-board kernel (upper bound)
  int32_t threads;       // threads per small-board workgroup: 256, 512 or 1024
  bool auto_threads;     // nobody asked for 512 threads: 1024 where the largest boards are few (board_threads)
  int32_t streams;       // streams carrying large boards (0: all work on the run stream)
  bool graph;            // replay the whole launch sequence through a captured hipGraph
};

// Memory of one run, as offsets into a single device allocation.
struct MidLayout {
  std::vector<int> small, big;         // board indices (big: largest first)
  std::vector<int> big_stream;         // stream of each big board (parallel to big)
  int32_t workgroups = 0;              // small-board kernel grid, within the budget
  int32_t streams = 0;                 // large-board streams (0: the run stream)
  std::vector<size_t> table_off;       // per small board
  size_t small_work = 0, small_stride = 0;   // workspace slot of each workgroup
  size_t big_slots = 0, big_stride = 0;      // per stream: tables, then workspace
  size_t bytes = 0;                    // total
  // descriptor blob at offset 0: small boards | big boards | prep prefixes | results | head (the
  // large boards' share is part of the reported bytes only: their launches take them by value)
  size_t o_big = 0, o_prefix = 0, o_res = 0, o_head = 0, blob_bytes = 0;
};
// Returns null on success, else an error message.
const char* mid_layout(const std::vector<MidInfo>& infos, const MidConfig& cfg, MidLayout* L);

struct MidPlan {
  int device = -1;
  int nb = 0;
  int board_threads = 0;               // of a small board's workgroup (cfg.threads, or board_threads' 1024)
  MidConfig cfg{};
  MidLayout layout;
  std::vector<MidInfo> infos;
  uint8_t* mem = nullptr;              // layout.bytes
  size_t mem_cap = 0;                  // block_take's size when the plan holds such a block, else 0
  hipEvent_t done = nullptr;           // the end of the last run, for such a block
  bool captured = false;               // a run was captured: nobody knows when the memory is free
  bool owns_mem = true;                // false: caller memory, not freed by the plan
  const MidBoardDev* small_dev = nullptr;
  std::vector<MidBoardDev> big;        // large boards: launches take them by value
  const int64_t* prefix = nullptr;     // small boards' prep prefix
  pe_halfsupers* results = nullptr;    // 19 per board, in board order
  unsigned int* head = nullptr;
  int64_t small_prep_total = 0;
  DevTables tables{};
  std::vector<hipStream_t> streams;    // owned, layout.streams of them
  std::vector<hipEvent_t> events;      // fork + one join per stream
  hipGraphExec_t graph_exec = nullptr;
  int64_t launches = 0;                // kernel launches per run
};

// upload_stream null: the descriptors go up by a synchronous hipMemcpy; else on that stream.  With
// pinned host memory `upload` of at least the layout's o_res bytes (which must stay untouched
// until upload_stream has passed the plan's first run), the upload is queued without
// waiting; otherwise the call waits for the upload.
// With `memory` of at least the layout's bytes the plan lives there (nothing is allocated,
// the caller keeps the memory until the plan is destroyed and its runs have finished).
pe_status mid_plan_create(const std::vector<MidInfo>& infos, const MidConfig& cfg, MidPlan* plan,
                          hipStream_t upload_stream = nullptr, void* upload = nullptr, size_t upload_bytes = 0,
                          void* memory = nullptr, size_t memory_bytes = 0);
pe_status mid_plan_run(MidPlan& plan, hipStream_t stream);
// Queue the copy of all results to host memory on `stream`; after the stream has been
// synchronized, mid_plan_zero_tail clears the entries past each board's spots.
pe_status mid_plan_copy_results(const MidPlan& plan, pe_halfsupers (*out)[19], hipStream_t stream);
void mid_plan_zero_tail(const MidPlan& plan, pe_halfsupers (*out)[19]);
// Gives the plan's own memory back (block_give).
void mid_plan_destroy(MidPlan* plan);
int mid_board_blocks_per_cu(int threads);

// Serving loop (mid_server.cc)
struct MidServer;
pe_status mid_server_create(const pe_mid_server_config* c, MidServer** out);
pe_status mid_server_submit(MidServer* S, const pe_high_board& board, int64_t* ticket);
pe_status mid_server_poll(MidServer* S, int64_t ticket, pe_halfsupers* results, int* done, double* latency_ms);
pe_status mid_server_wait(MidServer* S, int64_t ticket, pe_halfsupers* results, double* latency_ms);
void mid_server_stats(MidServer* S, pe_mid_server_info* out);
void mid_server_destroy(MidServer* S);

// Byte sizes of one board's tables, workspace, and both plus its 19 results.
size_t mid_table_bytes(const MidInfo& I);
size_t mid_work_bytes(const MidInfo& I);
size_t mid_board_bytes(const MidInfo& I);
// Lay out one board's table area (mid_table_bytes) at `base`; or tables, workspace and results
// (mid_board_bytes) at `base`.
void mid_carve_tables(MidBoardDev* B, uint8_t* base);
void mid_carve(MidBoardDev* B, uint8_t* base);
// One launch building the tables of every board: prefix[b] = prep entries before board b.
pe_status mid_launch_prep(const MidBoardDev* boards, const int64_t* prefix, int nb, int64_t total,
                          const DevTables& T, hipStream_t stream);
// Threads of a prep launch for one board; steps of a board; tiles of one step (0 past the last).
inline int64_t mid_prep_entries(const MidInfo& I) { return int64_t(2) << I.spots; }
int mid_steps(const MidInfo& I);
int64_t mid_step_tiles(const MidInfo& I, int step);
// Every launch of one board, its descriptor passed by value.
pe_status mid_launch_board(const MidBoardDev& board, const DevTables& T, hipStream_t stream);

}  // namespace pe
