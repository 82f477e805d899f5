// Midsolve kernels for gfx950.
//
// Per board: one pass building the wins tables (pentago/mid/internal.h:122-131) and then one
// launch per step of tiles (mid_tiles.h), a workgroup per tile, carrying (win, notlose)
// together.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstddef>
#include <cstring>
#include <mutex>
#include <string>
#include <vector>

#include "mid_device.h"
#include "mid_queue.h"

namespace pe {

namespace {

__device__ __forceinline__ int find_board(const int64_t* prefix, int nb, int64_t t) {
  int lo = 0, hi = nb;
  while (hi - lo > 1) {
    const int mid = (lo + hi) >> 1;
    if (prefix[mid] <= t) lo = mid; else hi = mid;
  }
  return lo;
}

__global__ __launch_bounds__(256) void mid_prep_kernel(const MidBoardDev* __restrict__ boards,
                                                       const int64_t* __restrict__ prefix, int nb,
                                                       int64_t total, DevTables T) {
  const int64_t t = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (t >= total) return;
  // the wave's first board by one search in scalar loads; a lane is a few boards past it at most
  const int wave = __builtin_amdgcn_readfirstlane(int(threadIdx.x) & ~63);
  int b = find_board(prefix, nb, int64_t(blockIdx.x) * blockDim.x + wave);
  while (b + 1 < nb && prefix[b + 1] <= t) b++;
  mid_wins_entry(boards[b], t - prefix[b], T);
}

// One board's table, by value.
__global__ __launch_bounds__(256) void mid_prep_one_kernel(MidBoardDev B, int64_t total, DevTables T) {
  const int64_t t = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (t < total) mid_wins_entry(B, t, T);
}

// Workgroup i runs on XCD i % 8: each XCD takes runs of neighbouring tiles, which read the same
// tiles.  Runs of 1 / 4 / 16 / 64 tiles measured within 3 %, 16 the fastest; one run of an eighth
// of the launch to each XCD is 20 % slower (the groups of a step differ in tile size).
constexpr int kRun = 16;
unsigned run_grid(int64_t tiles) { return unsigned((tiles + 8 * kRun - 1) / (8 * kRun) * (8 * kRun)); }
// A step that writes more than this (24 KB a tile at most) than the L2s hold together, 32 MB, is
// stored past them: 18 empty cells 2.51 -> 2.43 ms; a small step's reader finds it in the L2.
constexpr int kStreamTiles = 2048;

// Step `step` of every board that has one: workgroup w sweeps tile w - prefix[b] of the
// step's tiles of board b.
__global__ __launch_bounds__(2 * kTileThreads, 8) void mid_step_kernel(const MidBoardDev* __restrict__ boards,
                                                                     const int64_t* __restrict__ prefix, int nb,
                                                                     int step, int ntiles, MidTabsDev M) {
  __shared__ TileLds<false> lds;
  const int x = blockIdx.x & 7, y = blockIdx.x >> 3;
  const int w = (y / kRun * 8 + x) * kRun + y % kRun;
  if (w >= ntiles) return;
  const int b = find_board(prefix, nb, w);
  const int t = w - int(prefix[b]);
  const MidBoardDev& B = boards[b];
  const MidSched& S = M.sched[B.I.spots];
  mid_tile<2>(tile_job(B, B.work, S, M, ntiles > kStreamTiles), S.first[step] + t, lds, int(threadIdx.x));
}

// A step of one board, by value: `ntiles` tiles from `first` on, a workgroup each, or with kAlone a
// workgroup for each chain of a tile.
template <bool kAlone>
__global__ __launch_bounds__((kAlone ? 1 : 2) * kTileThreads, 8) void mid_step_one_kernel(TileJob J, int first,
                                                                                        int ntiles) {
  __shared__ TileLds<kAlone> lds;
  const int x = blockIdx.x & 7, y = int(blockIdx.x >> 3) / (kAlone ? 2 : 1);
  const int w = (y / kRun * 8 + x) * kRun + y % kRun;
  if (w < ntiles) mid_tile<2, kAlone>(J, first + w, lds, int(threadIdx.x), int(blockIdx.x >> 3 & 1));
}

}  // namespace

int mid_steps(const MidInfo& I) { return mid_tabs().sched[size_t(I.spots)].steps; }
int64_t mid_step_tiles(const MidInfo& I, int step) {
  const MidSched& S = mid_tabs().sched[size_t(I.spots)];
  return step < S.steps ? S.first[step + 1] - S.first[step] : 0;
}

// Allocation of one board's device scratch inside a caller-provided arena.
static size_t align256(size_t x) { return (x + 255) & ~size_t(255); }

size_t mid_table_bytes(const MidInfo& I) { return size_t(mid_table_area_bytes(I.spots)); }
size_t mid_work_bytes(const MidInfo& I) { return align256(32 * size_t(mid_work_entries(I.spots))); }
size_t mid_board_bytes(const MidInfo& I) {
  return mid_table_bytes(I) + mid_work_bytes(I) + align256(sizeof(pe_halfsupers) * 19);
}

void mid_carve_tables(MidBoardDev* B, uint8_t* base) {
  B->wins = reinterpret_cast<uint64_t*>(base);
  B->spill = B->wins + (size_t(8) << B->I.spots);   // 2 << spots entries of 4 words
}

void mid_carve(MidBoardDev* B, uint8_t* base) {
  mid_carve_tables(B, base);
  const size_t t = mid_table_bytes(B->I);
  B->work = reinterpret_cast<uint64_t*>(base + t);
  B->results = reinterpret_cast<pe_halfsupers*>(base + t + mid_work_bytes(B->I));
}


// Up to the number of tiles whose chains the chip holds at once (8 workgroups of 20 KB LDS a compute unit),
// a step's time is a tile's latency, which is shorter with a workgroup for each chain: 26 stones 62
// -> 58 us, 22 stones 153 -> 145, 20 stones 343 -> 331.  A larger step would be no faster so, and its small
// workgroups leave no room in the LDS for other streams' (65 boards of 18-30 stones 18.1 -> 20.6 ms).
constexpr int64_t kAloneTiles = 1024;

pe_status mid_launch_board(const MidBoardDev& B, const DevTables& T, hipStream_t stream) {
  const int64_t total = mid_prep_entries(B.I);
  hipLaunchKernelGGL(mid_prep_one_kernel, dim3(unsigned((total + 255) / 256)), dim3(256), 0, stream, B, total, T);
  PE_HIP(hipGetLastError(), "mid_prep_one_kernel launch");
  const MidSched& S = mid_tabs().sched[size_t(B.I.spots)];
  for (int k = 0; k < S.steps; k++) {
    const int64_t tiles = mid_step_tiles(B.I, k);
    if (tiles <= 0) continue;
    const TileJob J = tile_job(B, B.work, S, T.mid, tiles > kStreamTiles);
    if (tiles <= kAloneTiles)
      hipLaunchKernelGGL(mid_step_one_kernel<true>, dim3(2 * run_grid(tiles)), dim3(kTileThreads), 0, stream, J, S.first[k],
                         int(tiles));
    else
      hipLaunchKernelGGL(mid_step_one_kernel<false>, dim3(run_grid(tiles)), dim3(2 * kTileThreads), 0, stream, J, S.first[k],
                         int(tiles));
    PE_HIP(hipGetLastError(), "mid_step_one_kernel launch");
  }
  return PE_OK;
}

pe_status mid_launch_prep(const MidBoardDev* boards, const int64_t* prefix, int nb, int64_t total,
                          const DevTables& T, hipStream_t stream) {
  if (total <= 0) return PE_OK;
  hipLaunchKernelGGL(mid_prep_kernel, dim3(unsigned((total + 255) / 256)), dim3(256), 0, stream, boards, prefix, nb,
                     total, T);
  PE_HIP(hipGetLastError(), "mid_prep_kernel launch");
  return PE_OK;
}

// One board in device memory of at least mid_board_bytes, its 19 results stored to `results` (device
// or mapped host memory).
pe_status mid_solve_one(const MidInfo& info, uint8_t* arena, pe_halfsupers* results, hipStream_t stream) {
  DevTables T;
  std::string err;
  if (device_tables(&T, &err) != PE_OK) { set_error(err); return PE_ERR_DEVICE; }
  MidBoardDev B{};
  B.I = info;
  mid_carve(&B, arena);
  B.results = results;
  return mid_launch_board(B, T, stream);
}

// Solve of many boards, one launch a step over all of them, whose scratch lives in `arena` (device memory of
// at least the sum of mid_board_bytes).  Results land in each board's scratch; the caller
// copies them out (offsets returned in result_offsets).
pe_status mid_solve_levels(const std::vector<MidInfo>& infos, uint8_t* arena, std::vector<size_t>* result_offsets,
                           hipStream_t stream, DeviceBuffer& desc_cache) {
  DevTables T;
  std::string err;
  if (device_tables(&T, &err) != PE_OK) { set_error(err); return PE_ERR_DEVICE; }
  const int nb = int(infos.size());
  if (!nb) return PE_OK;
  std::vector<MidBoardDev> boards(nb);
  result_offsets->resize(nb);
  size_t off = 0;
  int steps = 0;
  for (int b = 0; b < nb; b++) {
    boards[b].I = infos[b];
    mid_carve(&boards[b], arena + off);
    (*result_offsets)[b] = size_t(reinterpret_cast<uint8_t*>(boards[b].results) - arena);
    off += mid_board_bytes(infos[b]);
    steps = std::max(steps, mid_steps(infos[b]));
  }
  // prefix sums: prep entries, then tiles per step
  std::vector<int64_t> prefix(size_t(nb + 1) * (steps + 1), 0);
  for (int b = 0; b < nb; b++) prefix[b + 1] = prefix[b] + mid_prep_entries(infos[b]);
  for (int t = 0; t < steps; t++) {
    int64_t* p = prefix.data() + size_t(nb + 1) * (t + 1);
    for (int b = 0; b < nb; b++) p[b + 1] = p[b] + mid_step_tiles(infos[b], t);
  }
  const size_t desc_bytes = sizeof(MidBoardDev) * nb;
  const size_t bytes = desc_bytes + sizeof(int64_t) * prefix.size();
  std::vector<uint8_t> blob(bytes);
  std::memcpy(blob.data(), boards.data(), desc_bytes);
  std::memcpy(blob.data() + desc_bytes, prefix.data(), sizeof(int64_t) * prefix.size());
  PE_HIP(desc_cache.reserve(bytes), "hipMalloc(mid descriptors)");
  void* const d = desc_cache.ptr;
  PE_HIP(hipMemcpyAsync(d, blob.data(), bytes, hipMemcpyHostToDevice, stream), "hipMemcpyAsync(mid descriptors)");
  const auto* dboards = static_cast<const MidBoardDev*>(d);
  const auto* dprefix = reinterpret_cast<const int64_t*>(static_cast<uint8_t*>(d) + desc_bytes);
  {
    const int64_t total = prefix[nb];
    if (total > 0)
      hipLaunchKernelGGL(mid_prep_kernel, dim3(unsigned((total + 255) / 256)), dim3(256), 0, stream, dboards,
                         dprefix, nb, total, T);
    PE_HIP(hipGetLastError(), "mid_prep_kernel launch");
  }
  for (int t = 0; t < steps; t++) {
    const int64_t* p = prefix.data() + size_t(nb + 1) * (t + 1);
    const int64_t total = p[nb];
    if (total <= 0) continue;
    if (total > 0x7fff0000) { set_error("too many tiles in one midsolve launch"); return PE_ERR_CAPACITY; }
    hipLaunchKernelGGL(mid_step_kernel, dim3(run_grid(total)), dim3(2 * kTileThreads), 0, stream, dboards,
                       dprefix + size_t(nb + 1) * (t + 1), nb, t, int(total), T.mid);
    PE_HIP(hipGetLastError(), "mid_step_kernel launch");
  }
  return PE_OK;
}

// ---- allocation-free single-board solve ----
// For callers that cannot allocate device memory (code under HIP graph capture, tight
// serving loops, harnesses that forbid hipMalloc); the reference has no counterpart (its
// caller passes a workspace it owns).  The board's tables, its workspace and its results live in `scratch`, a fixed array that every device the library
// runs on holds until the process ends.  Host code never uses the array's name as an
// address: each device's address comes from hipGetSymbolAddress, once per device.
constexpr size_t kScratchBytes = size_t(64) << 20;
static __device__ __align__(256) uint8_t scratch[kScratchBytes];

namespace {

constexpr int kScratchDevices = 64;
std::mutex g_scratch_mu[kScratchDevices];      // one solve at a time per device in this process
uint8_t* g_scratch_ptr[kScratchDevices];       // device address of `scratch` on each device

}  // namespace

int64_t mid_noalloc_scratch_bytes() { return int64_t(kScratchBytes); }

pe_status mid_solve_noalloc(const pe_high_board& hb, pe_halfsupers* results, hipStream_t stream) {
  MidInfo I;
  if (!make_mid_info(hb, &I)) { set_error("not a valid board with at least 18 stones"); return PE_ERR_INVALID; }
  DevTables T;
  if (!device_tables_ready(&T)) {
    set_error("the device's tables are not uploaded: call pe_init on this device first (this entry point allocates nothing)");
    return PE_ERR_INVALID;
  }
  const size_t need = mid_board_bytes(I);
  if (need > kScratchBytes) {
    set_error("board with " + std::to_string(I.spots) + " empty cells needs " + std::to_string(need) +
              " bytes of device scratch; the allocation-free solve has " + std::to_string(kScratchBytes) +
              " (boards with at most 15 empty cells, i.e. at least 21 stones)");
    return PE_ERR_CAPACITY;
  }
  int dev = 0;
  PE_HIP(hipGetDevice(&dev), "hipGetDevice");
  if (dev < 0 || dev >= kScratchDevices) { set_error("device index out of range"); return PE_ERR_DEVICE; }
  std::lock_guard<std::mutex> lock(g_scratch_mu[dev]);
  if (!g_scratch_ptr[dev]) {
    void* p = nullptr;
    PE_HIP(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)), "hipGetSymbolAddress(scratch)");
    g_scratch_ptr[dev] = static_cast<uint8_t*>(p);
  }
  uint8_t* const base = g_scratch_ptr[dev];
  // every table, workspace and result entry the kernels read is written by them first
  // (prep, then the tile layers), so nothing in the array needs clearing between calls
  MidBoardDev B{};
  B.I = I;
  mid_carve(&B, base);
  // every way out waits for the work queued on the stream: the next call (on any stream) reuses
  // the array
  struct Drain {
    hipStream_t s;
    ~Drain() { (void)hipStreamSynchronize(s); }
  } drain{stream};
  const pe_status st = mid_launch_board(B, T, stream);
  if (st != PE_OK) return st;
  PE_HIP(hipMemcpyAsync(results, B.results, sizeof(pe_halfsupers) * 19, hipMemcpyDeviceToHost, stream),
         "hipMemcpyAsync(results)");
  PE_HIP(hipStreamSynchronize(stream), "allocation-free midsolve");
  for (int i = I.spots + 1; i < 19; i++) std::memset(&results[i], 0, sizeof(pe_halfsupers));
  return PE_OK;
}

}  // namespace pe
