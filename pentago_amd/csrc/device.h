// Device-resident lookup tables and HIP error plumbing shared by the kernels.
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>
#include <new>
#include <stdexcept>
#include <string>

#include "../../include/pentago_amd.h"
#include "mid_tiles.h"

namespace pe {

// Device copies of the lookup tables (uploaded once per device by pe_init).
struct DevTables {
  const uint64_t* superwin;     // 4*512*5 supers
  const uint16_t* rmin_flat;    // packed radix-3 rotation-minimal quadrants
  const uint32_t* rmin_sides;   // the same quadrants unpacked: side0 | side1 << 16
  const uint16_t* rmin_inverse; // 19683 entries
  const uint16_t* pack;         // 512 entries
  const uint8_t* commute;       // 8*256 entries
  const uint8_t* rmin_stab;     // per rotation-minimal quadrant: log2 of its local stabilizer size
  const uint64_t* fields;       // field pool of the fused end kernels (end.h: field_pool_off)
  MidTabsDev mid;               // tiles of the midsolve
};

// Upload the tables to the current device (idempotent per device).
pe_status device_tables(DevTables* out, std::string* err);
// The current device's tables if they are already uploaded (never allocates).
bool device_tables_ready(DevTables* out);

void set_error(const std::string& e);

// hipMalloc that gives the kept block (below) back to the device before it fails.
hipError_t device_malloc(void** p, size_t bytes);

// Memory of a finished plan, kept for the next one: at most one block a device, of at most
// kKeptBytes.  Freed VRAM is cleared before it is handed out again, which costs a process that
// makes a plan a batch about 27 ms a GB once the device has no clean memory left.
// take: a block for `bytes` (its size in *cap, at most `limit` and less than twice `bytes`), the
// kept one of the current device or a new one with an eighth to spare, beside which the kept one
// stays only if both are within `limit`.  give: back from its owner, who has waited for all work
// that uses it.  The larger block is kept (large and small batches in turn: the large ones find
// theirs, 27 ms a GB), but one that two plans in a row could not use makes room for a smaller.
// Thread-safe: a block has one owner.
constexpr size_t kKeptBytes = size_t(4) << 30;
hipError_t block_take(size_t bytes, size_t limit, void** p, size_t* cap);
void block_give(int device, void* p, size_t cap);
// Memory that device_malloc can hand out on the current device: what is free, and the kept block,
// which default budgets count as the free memory that it was before (without it each plan's budget
// would depend on the plan closed before).
hipError_t device_available(size_t* bytes);

// Grow-only device allocation reused across synchronous calls (callers serialize use and
// have no work pending on it when it grows).
struct DeviceBuffer {
  void* ptr = nullptr;
  size_t cap = 0;
  hipError_t reserve(size_t bytes) {
    if (bytes <= cap) return hipSuccess;
    if (ptr) (void)hipFree(ptr);
    ptr = nullptr;
    cap = 0;
    const hipError_t e = device_malloc(&ptr, bytes);
    if (e == hipSuccess) cap = bytes;
    return e;
  }
};
// Every C entry point's body runs inside PE_GUARD_BEGIN / PE_GUARD_END: no C++ exception
// (a failed host allocation, above all) crosses the C ABI; it becomes an error status.
#define PE_GUARD_BEGIN try {
#define PE_GUARD_END                                                                \
  }                                                                                 \
  catch (const std::bad_alloc&) {                                                   \
    ::pe::set_error("host memory exhausted");                                       \
    return PE_ERR_CAPACITY;                                                         \
  }                                                                                 \
  catch (const std::exception& e_) {                                                \
    ::pe::set_error(e_.what());                                                     \
    return PE_ERR_INVALID;                                                          \
  }
#define PE_HIP(expr, msg)                                                           \
  do {                                                                              \
    hipError_t e_ = (expr);                                                         \
    if (e_ != hipSuccess) {                                                         \
      ::pe::set_error(std::string(msg) + ": " + hipGetErrorString(e_));             \
      return PE_ERR_DEVICE;                                                         \
    }                                                                               \
  } while (0)

}  // namespace pe
