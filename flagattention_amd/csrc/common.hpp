// Shared pieces of the attention kernels: launch helper, tile movers and MFMA operand readers.
//
// Conventions used by every kernel in this directory
//   * tensors are (batch, head, token, D) views with unit stride on D; strides are in elements;
//   * a "tile" is a row-major patch of tokens x D held in LDS with a padded row stride (LD);
//   * one wavefront multiplies 32x32 blocks with mfma32 (hw.hpp); its lane l owns column l % 32 of a
//     block and the half h = l / 32 selects which rows / which 8 of the 16 contraction indices.
#pragma once
#include <atomic>
#include <initializer_list>
#include <mutex>
#include <type_traits>
#include <unordered_map>
#include <utility>

#include "hw.hpp"
#include "params.hpp"

namespace fa {

using hw::u32x4;
using hw::f32x16;
using hw::short4v;

constexpr int kThreads = 256;  // 4 wavefronts per workgroup
constexpr float kLog2e = 1.4426950408889634f;
constexpr float kLn2 = 0.6931471805599453f;

FA_DEVICE int cdiv(int a, int b) { return (a + b - 1) / b; }
FA_DEVICE int imin(int a, int b) { return a < b ? a : b; }
FA_DEVICE int imax(int a, int b) { return a > b ? a : b; }
FA_DEVICE float neg_inf() { return -__builtin_inff(); }

// ---------------------------------------------------------------------------------------------
// global -> registers -> LDS movement of a ROWS x COLS tile (16 bytes per thread per step)
// ---------------------------------------------------------------------------------------------
// Loop-invariant plan of one thread's share of a ROWS x COLS tile: byte offsets inside the global
// tile are computed once, so that a steady-state fetch is one load per chunk from a uniform tile
// base plus a 32-bit lane offset, and the LDS destination is a fixed offset from the tile start.
//
// fetch() is branch-free on purpose.  With a branch per load (or per tile kind) the compiler puts
// loads in separate basic blocks and waits for ALL outstanding loads at their boundaries -- a full
// memory latency per tile.  Rows that do not exist are therefore read from the last row that does
// (always valid memory) and replaced by zeros when the tile is committed to LDS.
template <class T, int ROWS, int COLS>
struct TileMover {
  static constexpr int CPR = COLS / 8;          // 16-byte chunks per row
  static constexpr int RPP = kThreads / CPR;    // rows covered by one pass of the workgroup
  static constexpr int PASSES = (ROWS + RPP - 1) / RPP;
  static constexpr bool kExact = (PASSES * RPP == ROWS);
  u32x4 r[PASSES];
  uint32_t goff[PASSES];
  uint32_t stride_bytes, col_bytes;
  int row0, col0;
  int valid;  // rows of the fetched tile that exist
  uint32_t last_off;

  FA_DEVICE void init(int tid, int64_t row_stride) {
    row0 = tid / CPR;
    col0 = (tid % CPR) * 8;
    stride_bytes = (uint32_t)(row_stride * (int64_t)sizeof(T));
    col_bytes = (uint32_t)(col0 * (int)sizeof(T));
    valid = ROWS;
#pragma unroll
    for (int i = 0; i < PASSES; ++i) goff[i] = (uint32_t)(row0 + i * RPP) * stride_bytes + col_bytes;
  }
  // rows_valid >= 1 rows of the tile exist; rows past them load a copy of the last one
  FA_DEVICE void fetch(const T* tile_base, int rows_valid) {
    fetch_begin(rows_valid);
#pragma unroll
    for (int i = 0; i < PASSES; ++i) fetch_pass(tile_base, i);
  }
  // the same in pieces, for callers that place the loads themselves
  FA_DEVICE void fetch_begin(int rows_valid) {
    valid = rows_valid < ROWS ? rows_valid : ROWS;
    last_off = (uint32_t)(valid - 1) * stride_bytes + col_bytes;
  }
  FA_DEVICE void fetch_pass(const T* tile_base, int i) {
    const uint32_t off = (row0 + i * RPP < valid) ? goff[i] : last_off;
    r[i] = *(const u32x4*)((const char*)tile_base + off);
  }
  // one pass of commit(), without the zeroes for rows past the end: those keep the copies of the
  // last row that fetch() loaded
  template <int LD>
  FA_DEVICE void commit_pass(T* lds_tile, int i) const {
    static_assert(kExact, "whole passes only");
    *(u32x4*)(lds_tile + (row0 + i * RPP) * LD + col0) = r[i];
  }
  template <int LD>
  FA_DEVICE void commit(T* lds_tile) {
    if (valid < ROWS) {  // tail tile only (uniform): rows past the end become zeros
      hw::keep_branch();
#pragma unroll
      for (int i = 0; i < PASSES; ++i)
        if (row0 + i * RPP >= valid) r[i] = u32x4{0u, 0u, 0u, 0u};
    }
#pragma unroll
    for (int i = 0; i < PASSES; ++i)
      if (kExact || row0 + i * RPP < ROWS) *(u32x4*)(lds_tile + (row0 + i * RPP) * LD + col0) = r[i];
  }
};

// ---------------------------------------------------------------------------------------------
// MFMA operand readers
// ---------------------------------------------------------------------------------------------
// Operand whose contraction index runs along D: element (row = row0 + l % 32, k = k0 + 8h + 0..7)
// of a row-major tile, one 16-byte LDS read.
// f(integral_constant<int, 0>) ... f(integral_constant<int, N - 1>), in order: a loop whose index is a
// constant expression inside the body
template <int... I, class F>
FA_DEVICE void static_for_each(std::integer_sequence<int, I...>, F&& f) {
  (f(std::integral_constant<int, I>{}), ...);
}
template <int N, class F>
FA_DEVICE void static_for(F&& f) {
  static_for_each(std::make_integer_sequence<int, N>{}, f);
}

template <class T, int LD>
FA_DEVICE typename hw::Elem<T>::v8 operand_rowmajor(const T* lds_tile, int row0, int k0, int lane) {
  const T* p = lds_tile + (row0 + (lane & 31)) * LD + k0 + 8 * (lane >> 5);
  return hw::as_v8<T>(*(const u32x4*)p);
}

// Operand whose contraction index runs along the tile's rows (tokens) and whose free index runs
// along D: the lane needs, for column c0 + l % 32, the 8 rows
//     t0 + 4h + {0,1,2,3}  and  t0 + 8 + 4h + {0,1,2,3}
// which is exactly the order in which an mfma32 result holds rows 0..15 of a block (registers
// 0..7) -- so a 16-row slice of a result block can be multiplied against this operand directly.
// Two transposing reads fetch them from the row-major tile.
template <class T, int LD>
FA_DEVICE typename hw::Elem<T>::v8 operand_transposed(const T* lds_tile, int t0, int c0, int lane) {
  int i = lane & 15, dhalf = (lane >> 4) & 1, h = lane >> 5;
  const T* p = lds_tile + (t0 + 4 * h + (i >> 2)) * LD + c0 + 16 * dhalf + 4 * (i & 3);
  short4v lo = hw::lds_read_tr16(p);
  short4v hi = hw::lds_read_tr16(p + 8 * LD);
  return hw::join_v8<T>(lo, hi);
}

// Work distribution of the tiled kernels: a 1-D grid of (tile rank) x (batch * head) workgroups with
// the (batch, head) index running fastest.  Workgroups are dispatched in id order, so ranking tiles
// from most to least work puts every head's longest tiles first and leaves the shortest for the
// tail (balanced finish under the causal mask); and because consecutive ids go to consecutive XCDs,
// a given (batch, head) -- whose K/V or Q/dO every one of its tiles re-reads -- stays on one XCD's
// L2 whenever batch * heads is a multiple of the XCD count.
//
// `deal`: where a compute unit holds several workgroups, the first of a launch are all resident from the start, in
// rounds of one per unit, and unit i gets workgroup i of every round.  Ranked by length throughout, the unit with the
// longest tile would also hold the longest of the second round: 32768 rows of 2 heads under the causal mask (512
// workgroups of 128 rows on 256 units) give one unit 512 + 256 steps and the last one 258 + 2.  Odd rounds therefore run
// from short to long, and where the second round is not full, the longest of the first go to units of their own.
// Workgroups move by multiples of 8, so a head keeps its XCD.  dQ from dS at that size 605 -> 551 us per launch; the
// step of B=4 H=16 T=1024 D=64 with dropout (512 workgroups per launch) 127 -> 120 us.
struct TileId { int rank, head, batch; };
FA_DEVICE int dealt(int lin, int grid, Deal deal) {
  if (deal.resident < 2 || grid <= deal.unit) return lin;
  const int unit = deal.unit, round = lin / unit;
  if (round == 0 && grid < 2 * unit) {
    const int shared = (grid - unit) & ~7;   // units with a second workgroup
    return lin < shared ? lin + unit - shared : lin - shared;
  }
  if (round >= deal.resident || !(round & 1)) return lin;
  const int begin = round * unit, end = (begin + unit < grid ? begin + unit : grid) & ~7;
  return lin < end ? begin + end - 8 - (lin & ~7) + (lin & 7) : lin;
}
FA_DEVICE TileId tile_of_workgroup(int H, int B, Deal deal = Deal{0, 0}) {
  const int lin = dealt(hw::block_x(), hw::grid_x(), deal), bh = lin % (H * B);
  TileId t;
  t.rank = lin / (H * B);
  t.head = bh % H;
  t.batch = bh / H;
  return t;
}

// Row index inside a 32-row result block of register r for the lane's half h.
FA_DEVICE int block_row(int r, int h) { return 8 * (r >> 2) + 4 * h + (r & 3); }

// Packs registers 8c..8c+7 of a result block into an operand (rounded to T).
template <class T>
FA_DEVICE typename hw::Elem<T>::v8 pack_half_block(const f32x16& s, int c) {
  typename hw::Elem<T>::v8 v;
#pragma unroll
  for (int e = 0; e < 8; ++e) v[e] = (T)s[8 * c + e];
  return v;
}

// ---------------------------------------------------------------------------------------------
// dropout mask
// ---------------------------------------------------------------------------------------------
// The reference draws one number per score element with Triton's tl.rand(seed, offs, n_rounds=6)
// (src/flag_attn/flash.py:367-371, 454-457): Philox-4x32 with counter (lo(c), hi(c), 0, 0),
// c = offset + ((b * H + h) * M + m) * N + n, key (lo(seed), hi(seed)), 6 rounds, first output word;
// the word, read as int32 with negative values folded by -x - 1, times 4.6566127342e-10 is the
// uniform number, and the probability is kept when it exceeds dropout_p.
//
// What the kernels draw with: of the four words and six rounds only what reaches the first word is formed, three-way
// exclusive ors are one instruction, and the comparison is made on the integer (dropout_threshold below).  1.06e12 ->
// 1.66e12 elements/s, 95 clocks per 64 elements, which is still two to three times what the rest of the attention
// kernels does for them -- hence the mask goes from the forward to the backward as bits (KeepMask).
constexpr uint32_t kPhiloxM0 = 0xD2511F53u, kPhiloxM1 = 0xCD9E8D57u, kPhiloxW0 = 0x9E3779B9u, kPhiloxW1 = 0xBB67AE85u;

// The part of round 1 that depends on the counter's upper word alone.
struct PhiloxUpper { uint32_t x2, x3; };
FA_DEVICE PhiloxUpper philox_upper(uint32_t hi, uint32_t k0, uint32_t k1) {
  const uint64_t p = (uint64_t)kPhiloxM0 * (hi ^ k0);
  return PhiloxUpper{(uint32_t)(p >> 32) ^ (k1 + kPhiloxW1), (uint32_t)p};
}
FA_DEVICE uint32_t philox6_first_word(uint32_t lo, PhiloxUpper up, uint32_t k0, uint32_t k1) {
  const uint64_t a0 = (uint64_t)kPhiloxM0 * lo;                               // round 0: words 2 and 3 are zero
  const uint64_t b1 = (uint64_t)kPhiloxM1 * ((uint32_t)(a0 >> 32) ^ k1);      // round 1
  uint32_t c0 = (uint32_t)(b1 >> 32) ^ (k0 + kPhiloxW0), c1 = (uint32_t)b1;
  uint32_t c2 = up.x2 ^ (uint32_t)a0, c3 = up.x3;
#pragma unroll
  for (int round = 2; round < 5; ++round) {
    const uint64_t p0 = (uint64_t)kPhiloxM0 * c0, p1 = (uint64_t)kPhiloxM1 * c2;
    c0 = hw::xor3((uint32_t)(p1 >> 32), c1, k0 + (uint32_t)round * kPhiloxW0);
    c2 = hw::xor3((uint32_t)(p0 >> 32), c3, k1 + (uint32_t)round * kPhiloxW1);
    c1 = (uint32_t)p1;
    c3 = (uint32_t)p0;
  }
  return hw::xor3((uint32_t)(((uint64_t)kPhiloxM1 * c2) >> 32), c1, k0 + 5u * kPhiloxW0);
}
// The word x is kept when v = (x as int32, negative folded by -x - 1), times 4.6566127342e-10 in fp32, exceeds
// dropout_p.  v -> (float)v * c is monotonic, so there is a smallest kept v, `threshold`; and the dropped words are
// those of [-threshold, threshold), i.e. x + threshold < 2 threshold without sign.
inline uint32_t dropout_threshold(float dropout_p) {
  uint32_t lo = 0, hi = 0x7fffffffu;   // (float)hi * c > dropout_p for every dropout_p < 1 that fp32 tells from 1
  while (lo < hi) {
    const uint32_t mid = lo + (hi - lo) / 2;
    const float u = (float)(int32_t)mid * 4.6566127342e-10f;
    if (u > dropout_p) hi = mid;
    else lo = mid + 1;
  }
  return lo;
}
FA_DEVICE bool dropout_keeps(uint64_t counter, uint64_t seed, uint32_t threshold) {
  const uint32_t k0 = (uint32_t)seed, k1 = (uint32_t)(seed >> 32);
  return philox6_first_word((uint32_t)counter, philox_upper((uint32_t)(counter >> 32), k0, k1), k0, k1) + threshold >= 2u * threshold;
}
// Bits r = 0..15: whether the element at counter + block_row(r, 0) is kept (16 elements of a result block whose rows
// run along the counter).
FA_DEVICE uint32_t dropout_draw16(uint64_t counter, uint64_t seed, uint32_t threshold) {
  const uint32_t k0 = (uint32_t)seed, k1 = (uint32_t)(seed >> 32), lo = (uint32_t)counter, hi = (uint32_t)(counter >> 32);
  uint32_t bits = 0u;
  if (hw::wave_any(lo > 0xffffffffu - 27u)) {   // the counter's upper word changes inside the block
    hw::keep_branch();
#pragma unroll 1
    for (int r = 15; r >= 0; --r)
      bits = 2u * bits + (dropout_keeps(counter + (uint64_t)(8 * (r >> 2) + (r & 3)), seed, threshold) ? 1u : 0u);
    return bits;
  }
  const PhiloxUpper up = philox_upper(hi, k0, k1);
#pragma unroll
  for (int r = 15; r >= 0; --r)
    hw::append_at_least(bits, philox6_first_word(lo + (uint32_t)(8 * (r >> 2) + (r & 3)), up, k0, k1) + threshold, 2u * threshold);
  return bits;
}

// The mask of a forward as the backward reads it: one 32-bit word per query row and block of 32 keys (bit = key inside
// the block), words of one key block contiguous along the rows.  Blocks that no row of a 32-row block sees under the
// causal mask are neither written nor read.
struct KeepMask {
  int64_t rows, blocks;   // words per key block, key blocks per (batch, head)
  FA_DEVICE KeepMask(int M, int N) : rows(32 * (int64_t)cdiv(M, 32)), blocks(2 * (int64_t)cdiv(N, 64)) {}
  FA_DEVICE int64_t head(int64_t bh) const { return bh * blocks * rows; }
  FA_DEVICE int64_t block(int kb) const { return (int64_t)(kb < blocks ? kb : blocks - 1) * rows; }
};
// The 16 bits a lane holds (keys block_row(r, half) of a block) in their places in the word.
FA_DEVICE uint32_t keep_spread(uint32_t bits16, int half) {
  uint32_t x = (bits16 | (bits16 << 8)) & 0x00ff00ffu;
  x = (x | (x << 4)) & 0x0f0f0f0fu;
  return x << (4 * half);
}

// ---------------------------------------------------------------------------------------------
// launch
// ---------------------------------------------------------------------------------------------
constexpr int kMaxDevices = 64;   // devices whose per-device facts are remembered

// A kernel that needs more than 48 KB of LDS has to be given the limit before its first launch, once per
// device (the attribute belongs to the device's copy of the function).  The runtime call costs about as
// much as a launch, so the devices on which it has been made are remembered per kernel.
template <class P>
int allow_lds(void (*kern)(P), size_t lds_bytes) {
  static std::mutex lock;
  static std::unordered_map<const void*, uint64_t> done;   // kernel -> bit per device
  int dev = -1;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0) dev = kMaxDevices;
  const uint64_t bit = dev < kMaxDevices ? (uint64_t)1 << dev : 0;
  if (bit) {
    std::lock_guard<std::mutex> g(lock);
    auto it = done.find((const void*)kern);
    if (it != done.end() && (it->second & bit)) return 0;
  }
  hipError_t e = hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds_bytes);
  if (e != hipSuccess) return (int)e;
  if (bit) {
    std::lock_guard<std::mutex> g(lock);
    done[(const void*)kern] |= bit;
  }
  return 0;
}

template <class P>
int launch(void (*kern)(P), dim3 grid, size_t lds_bytes, hipStream_t stream, const P& p) {
  if (lds_bytes > 48 * 1024) {
    const int rc = allow_lds(kern, lds_bytes);
    if (rc) return rc;
  }
  hipLaunchKernelGGL(kern, grid, dim3(kThreads), lds_bytes, stream, p);
  return (int)hipGetLastError();
}

// Workgroups of a 1-D launch (the product of the factors), 0 if there are more than a grid can hold.  Formed in 64 bits and
// compared factor by factor: a product of ints that wraps would launch part of the tiles, or none, without an error.
inline unsigned workgroups(std::initializer_list<int64_t> factors) {
  int64_t n = 1;
  for (int64_t f : factors)
    if ((n *= f) > 0x7fffffff) return 0;
  return (unsigned)n;
}

// Workgroups of a kernel that a compute unit of the current device holds; asked once per kernel and device.
template <class P>
int resident_workgroups(void (*kern)(P), size_t lds_bytes) {
  static std::mutex lock;
  static std::unordered_map<const void*, int> known[kMaxDevices];
  int dev = -1, n = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices) return 1;
  std::lock_guard<std::mutex> g(lock);
  auto it = known[dev].find((const void*)kern);
  if (it != known[dev].end()) return it->second;
  if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, (const void*)kern, kThreads, lds_bytes) != hipSuccess) return 1;
  return known[dev][(const void*)kern] = n;
}

// A launch whose tiles differ in length under the causal mask: the kernel deals them by tile_of_workgroup.
template <class P>
int launch_dealt(void (*kern)(P), dim3 grid, size_t lds_bytes, hipStream_t stream, P p) {
  const int unit = num_cus_of_current_device();
  if (p.causal && unit > 0 && unit % 8 == 0 && (int64_t)grid.x > unit) {
    if (lds_bytes > 48 * 1024) {
      const int rc = allow_lds(kern, lds_bytes);
      if (rc) return rc;
    }
    p.deal = Deal{unit, resident_workgroups(kern, lds_bytes)};
  }
  return launch(kern, grid, lds_bytes, stream, p);
}

// error codes of the C entry points (positive values are hipError_t)
constexpr int kOk = 0;
constexpr int kBadArgument = -1;
constexpr int kUnsupported = -2;

constexpr int kDtypeF16 = 0;
constexpr int kDtypeBF16 = 1;

}  // namespace fa
