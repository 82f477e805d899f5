// Supertensor block data <-> device nodes (pentago/data/supertensor.h:1-50 file format,
// pentago/data/filter.h interleave filter, pentago/end/check.cc:149-158 orientation).
//
// A .pentago file stores per node the pair (black wins, white wins); filter 1 interleaves the
// two supers bit by bit so that in each 64-bit output word bit 2i is black's and bit 2i+1
// white's: output words 2k and 2k+1 hold the low and high halves of word k of both supers.
// Device nodes are (we-win, we-win-or-tie) for the player to move: with turn = stones & 1,
// black = turn ? ~we-win-or-tie : we-win and white = turn ? we-win : ~we-win-or-tie.
//
// 64 bytes read, 64 bytes written a node, in place allowed.  HBM-bound.  A quad of lanes takes a node:
// lane k reads file words 2k and 2k+1 (the other way round: writes them), which are word k of both supers,
// and the quad exchanges words, so that a wave's loads and stores are 1024 consecutive bytes.
// 32 M nodes, one MI355X: decode 0.84 -> 0.65, encode 0.87 -> 0.65 ms (6.2 TB/s) against a lane a
// node, whose loads and stores are 16 bytes in 64.
#include <hip/hip_runtime.h>

#include <string>

#include "device.h"

namespace pe {
namespace {

constexpr int kFormatThreads = 256;

__device__ inline uint64_t spread32(uint64_t a) {   // bit i -> bit 2i, i < 32
  a &= 0x00000000ffffffffull;
  a = (a | a << 16) & 0x0000ffff0000ffffull;
  a = (a | a << 8) & 0x00ff00ff00ff00ffull;
  a = (a | a << 4) & 0x0f0f0f0f0f0f0f0full;
  a = (a | a << 2) & 0x3333333333333333ull;
  a = (a | a << 1) & 0x5555555555555555ull;
  return a;
}

__device__ inline uint64_t gather32(uint64_t a) {   // bit 2i -> bit i
  a &= 0x5555555555555555ull;
  a = (a | a >> 1) & 0x3333333333333333ull;
  a = (a | a >> 2) & 0x0f0f0f0f0f0f0f0full;
  a = (a | a >> 4) & 0x00ff00ff00ff00ffull;
  a = (a | a >> 8) & 0x0000ffff0000ffffull;
  a = (a | a >> 16) & 0x00000000ffffffffull;
  return a;
}

// A value of another lane of the quad (quad_perm of four two-bit lane numbers).
template <int kPerm>
__device__ inline uint64_t quad64(uint64_t v) {
  const uint32_t lo = uint32_t(__builtin_amdgcn_mov_dpp(int(v), kPerm, 0xf, 0xf, true));
  const uint32_t hi = uint32_t(__builtin_amdgcn_mov_dpp(int(v >> 32), kPerm, 0xf, 0xf, true));
  return uint64_t(lo) | uint64_t(hi) << 32;
}
constexpr int kEven = 0x88, kOdd = 0xDD;         // lanes 0, 2, 0, 2 and 1, 3, 1, 3
constexpr int kFirst = 0x50, kSecond = 0xFA;     // lanes 0, 0, 1, 1 and 2, 2, 3, 3

typedef uint64_t Words __attribute__((ext_vector_type(2)));

// decode: file words (filtered (black, white)) -> (we-win, we-win-or-tie)
__device__ inline Words decode_quarter(Words w, int k, int filter, int turn) {
  if (filter != 1) return k < 2 ? w : ~w;   // loaded from the super that goes here
  const uint64_t black = gather32(w.x) | gather32(w.y) << 32;
  const uint64_t white = gather32(w.x >> 1) | gather32(w.y >> 1) << 32;
  const uint64_t win = turn ? white : black, tie = ~(turn ? black : white);   // word k of each
  const uint64_t we = quad64<kEven>(win), wo = quad64<kOdd>(win), te = quad64<kEven>(tie), to = quad64<kOdd>(tie);
  return k < 2 ? Words{we, wo} : Words{te, to};
}

// encode: (we-win, we-win-or-tie) -> file words
__device__ inline Words encode_quarter(Words w, int k, int filter, int turn) {
  if (filter != 1) return (k < 2) != (turn != 0) ? w : ~w;
  // word k of we-win is word k & 1 of lane k / 2, of we-win-or-tie of lane 2 + k / 2
  const uint64_t w0 = quad64<kFirst>(w.x), w1 = quad64<kFirst>(w.y), t0 = quad64<kSecond>(w.x), t1 = quad64<kSecond>(w.y);
  const uint64_t win = k & 1 ? w1 : w0, tie = ~(k & 1 ? t1 : t0);
  const uint64_t black = turn ? tie : win, white = turn ? win : tie;
  return Words{spread32(black) | spread32(white) << 1, spread32(black >> 32) | spread32(white >> 32) << 1};
}

// kStream: buffers that the 256 MB memory-side cache cannot hold together go past the caches: decode,
// count and encode of 32 M nodes 1.63 ms, else 1.76; of 1 M nodes (64 MB a buffer) 84 us, else 76.
constexpr int64_t kStreamNodes = int64_t(1) << 21;

// Workgroup b takes nodes 256 b to 256 b + 255, 64 at a time.  (A quad's lanes are active together;
// every load of a node is done before its first store, so in and out may be the same.)
template <bool kDecode, bool kStream>
__global__ __launch_bounds__(kFormatThreads) void format_kernel(const uint64_t* in, uint64_t* out, int64_t nodes,
                                                                int filter, int turn) {
  constexpr int kRounds = 4;
  const int k = threadIdx.x & 3;
  // without the filter the supers change places when white is to move
  const int from = filter != 1 && turn ? k ^ 2 : k;
  const int64_t first = int64_t(blockIdx.x) * kFormatThreads + (threadIdx.x >> 2);
  Words w[kRounds];
#pragma unroll
  for (int r = 0; r < kRounds; r++) {
    const int64_t i = first + r * (kFormatThreads / 4);
    const Words* p = reinterpret_cast<const Words*>(in + 8 * i) + from;
    if (i < nodes) w[r] = kStream ? __builtin_nontemporal_load(p) : *p;
  }
#pragma unroll
  for (int r = 0; r < kRounds; r++) {
    const int64_t i = first + r * (kFormatThreads / 4);
    if (i >= nodes) continue;
    const Words v = kDecode ? decode_quarter(w[r], k, filter, turn) : encode_quarter(w[r], k, filter, turn);
    Words* p = reinterpret_cast<Words*>(out + 8 * i) + k;
    if (kStream) __builtin_nontemporal_store(v, p);
    else *p = v;
  }
}

}  // namespace

pe_status launch_supertensor_format(bool decode, int filter, int turn, const void* in, int64_t nodes, void* out,
                                    hipStream_t stream, std::string* err) {
  if (filter != 0 && filter != 1) { *err = "unknown supertensor filter"; return PE_ERR_INVALID; }
  if (nodes < 0 || (nodes && (!in || !out))) { *err = "bad supertensor buffer arguments"; return PE_ERR_INVALID; }
  if (!nodes) return PE_OK;
  const int64_t blocks = (nodes + kFormatThreads - 1) / kFormatThreads;
  if (blocks > 0x7fffffff) { *err = "supertensor buffer too large"; return PE_ERR_CAPACITY; }
  const bool stream_past = nodes > kStreamNodes;
  const auto kernel = decode ? (stream_past ? format_kernel<true, true> : format_kernel<true, false>)
                             : (stream_past ? format_kernel<false, true> : format_kernel<false, false>);
  hipLaunchKernelGGL(kernel, dim3(unsigned(blocks)), dim3(kFormatThreads), 0, stream,
                     static_cast<const uint64_t*>(in), static_cast<uint64_t*>(out), nodes, filter, turn & 1);
  if (hipGetLastError() != hipSuccess) { *err = "supertensor format kernel launch failed"; return PE_ERR_DEVICE; }
  return PE_OK;
}

}  // namespace pe
