// Device helpers shared by the attention kernels: operand types and LDS
// layout, buffer resources, waits, item decode, masks and the arrival count of
// split row blocks.
#ifndef TRIANGLEMIX_DEVICE_H
#define TRIANGLEMIX_DEVICE_H

#include <hip/hip_runtime.h>

#include <stdint.h>

#include "trianglemix_kernel.h"

namespace tmx {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x4_t __attribute__((ext_vector_type(4)));
typedef short i16x4_t __attribute__((ext_vector_type(4)));
typedef float f32x16_t __attribute__((ext_vector_type(16)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));
typedef unsigned u32x4_t __attribute__((ext_vector_type(4)));

// Phase clocks (diagnostic builds only, -DTRIANGLEMIX_PHASE_CLOCKS): lane 0 of
// every wave stores the 100 MHz s_memrealtime clock at the TM_PHASE(slot)
// points of the kernels, one 64-bit slot per (workgroup, wave, phase), for grids
// of up to kPhaseClockWorkgroups workgroups.  Slots, the same in both kernels:
//   0 entry, 1 page tables complete, 2 Q landed, 3 scores of the first tile done,
//   4 + i iteration i opened (i < 8), 12 loop done, 13 KV parts merged,
//   14 output stored (nothing split); of a split row block: 16 partials stored,
//   17 arrival counted, 18 first batch of pieces merged, 19 all merged, 15 output
//   stored.
// Each source file has an array of its own; a launch fills that of its kernel
// and the read-back joins them.  The product library is built without.
#ifdef TRIANGLEMIX_PHASE_CLOCKS
constexpr int kMaxWaves = 8;  // waves of the largest workgroup shape
constexpr int kPhaseClockWorkgroups = 4096;
constexpr int kPhaseClockSlots = 32;
static __device__ unsigned long long phase_clocks[kPhaseClockWorkgroups * kMaxWaves * kPhaseClockSlots];
hipError_t wide_phase_clocks(void** ptr);  // the array of trianglemix_wide.hip
#define TM_PHASE(slot)                                                                                   \
  do {                                                                                                   \
    const unsigned long long tm_clock_ = __builtin_amdgcn_s_memrealtime();                               \
    if ((threadIdx.x & 63) == 0 && blockIdx.x < kPhaseClockWorkgroups)                                   \
      phase_clocks[(blockIdx.x * kMaxWaves + (threadIdx.x >> 6)) * kPhaseClockSlots + (slot)] = tm_clock_; \
  } while (0)
#else
#define TM_PHASE(slot) \
  do {                 \
  } while (0)
#endif

#define TM_LDS(p) ((__attribute__((address_space(3))) void*)(p))

constexpr int kRowBytes = kHeadDim * 2;          // 256 B: one key row
constexpr int kTileBytes = kKvTile * kRowBytes;  // 8 KB: K or V of one tile
constexpr int kDmaPerTile = kTileBytes / 1024;   // 1 KB (4 key rows) per DMA instruction


// Buffer-resource word 3 for raw (unformatted, stride 0) dword loads on gfx9.
constexpr int kBufferFlags = 0x00020000;
// A buffer offset past every range used here: such a load returns 0.
constexpr unsigned kOutOfRange = 0x40000000u;

static_assert(kKvTile == 32 && kPageSize % kKvTile == 0, "a tile must stay inside one page");
static_assert(kRowBlock == 32, "one MFMA column per query token");
static_assert(kDmaPerTile == 8, "a tile is eight 1 KB DMA instructions, one per MFMA step at most");

// Wait until every LDS DMA (and other vector-memory load) this wave issued has
// landed: s_waitcnt vmcnt(0), expcnt / lgkmcnt unconstrained.  Each wave runs
// it before a barrier that publishes DMA'd tiles to the other waves -- the
// barrier alone does not order the DMA's LDS writes.
__device__ __forceinline__ void wait_dma() { __builtin_amdgcn_s_waitcnt(0x0F70); }
// All but the last N (< 64) vector-memory operations of this wave have landed
// (vmcnt bits 3:0 and 15:14 of the gfx9 s_waitcnt immediate).
template <int N>
__device__ __forceinline__ void wait_dma_but() {
  static_assert(N >= 0 && N < 64, "vmcnt field");
  __builtin_amdgcn_s_waitcnt(0x0F70 | (N & 15) | ((N >> 4) << 14));
}

// All but the last N (< 16) LDS reads of this wave have returned (lgkmcnt, bits
// 11:8; LDS operations of a wave return in order).
template <int N>
__device__ __forceinline__ void wait_lds_but() {
  static_assert(N >= 0 && N < 16, "lgkmcnt field");
  __builtin_amdgcn_s_waitcnt(0xC07F | (N << 8));
}

__device__ __forceinline__ int k_slot(int row, int chunk) { return chunk ^ (row & 15); }
__device__ __forceinline__ int v_slot(int row, int chunk) { return chunk ^ ((row & 3) << 2); }

// The launch fields the prologue needs before its first memory round trip.
// They are the kernel's leading scalar arguments, which the command processor
// preloads into SGPRs (the library is built with
// -amdgpu-kernarg-preload-count): the block-table loads and the Q DMA issue
// without waiting for a kernarg load first (measured 0.3-0.4 us per launch).
// KernelParams, an aggregate passed by reference and never preloaded, carries
// the rest, which is first needed after that round trip.
struct PrologueArgs {
  const int32_t* block_table;
  const __bf16* query;
  int query_start;
  int seq_len;
  int num_row_blocks;
  int sparse_begin;
  int sparse_end;
  int split_items;
  int split_row_blocks;
  int tiles_per_split;
};

// Work item -> (row-block order index, split index, split count), computed
// by every wave from the split counts of the first p.split_row_blocks row
// blocks in issue order (lane i: row block base + i), which hold items
// 0 .. p.split_items - 1.
// The exclusive prefix sum over the lanes needs no cross-lane data move: bit
// by bit, it adds 2^b times the number of lower lanes whose count has bit b
// set (v_mbcnt of a ballot).  That is a few VALU and SALU instructions per
// bit -- six bits cover 63 splits, and a non-negative int has at most 31 --
// instead of a chain of dependent ds_bpermute round trips.
__device__ __forceinline__ void decode_item(const PrologueArgs& p, int sparse_begin, int sparse_end, int item,
                                            int lane, int& order, int& split, int& nsplit) {
  int acc = 0;
  order = 0;
  split = 0;
  nsplit = 1;
  for (int base = 0; base < p.split_row_blocks; base += 64) {
    const int o = base + lane;
    const int cnt = o < p.split_row_blocks ? row_block_splits(o, p.num_row_blocks, p.query_start, p.seq_len,
                                                            sparse_begin, sparse_end, p.tiles_per_split)
                                         : 0;
    int excl = 0;   // items of the row blocks on lower lanes
    int total = 0;  // items of the 64 row blocks
    for (int b = 0; __ballot((cnt >> b) != 0) != 0; ++b) {
      const unsigned long long bit = __ballot(((cnt >> b) & 1) != 0);
      excl += (int)__builtin_amdgcn_mbcnt_hi((unsigned)(bit >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)bit, 0u)) << b;
      total += __popcll(bit) << b;
    }
    if (item < acc + total) {
      const bool mine = cnt > 0 && item >= acc + excl && item < acc + excl + cnt;
      const int src = __ffsll((unsigned long long)__ballot(mine)) - 1;
      order = base + src;
      split = item - acc - __builtin_amdgcn_readlane(excl, src);
      nsplit = __builtin_amdgcn_readlane(cnt, src);
      return;
    }
    acc += total;
  }
}

// Rescale the running O / row sum only when some row's max grew by more than
// 2^kLazyRescale (log2 units); otherwise keep the stale max as the exponent
// shift, so p <= 2^kLazyRescale -- exact in fp32 and bf16 range -- and the
// 64 multiplies of the O rescale are skipped on most tiles.
constexpr float kLazyRescale = 8.0f;

// max / sum of x over the lane pair (i, i ^ 32), in every lane: v_permlane32_swap
// hands each lane both halves, so no lane select is needed.
__device__ __forceinline__ float half_max(float x) {
  const unsigned u = __float_as_uint(x);
  const auto r = __builtin_amdgcn_permlane32_swap(u, u, false, false);
  return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
__device__ __forceinline__ float half_sum(float x) {
  const unsigned u = __float_as_uint(x);
  const auto r = __builtin_amdgcn_permlane32_swap(u, u, false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

// Key offset inside the tile of accumulator element v, for lanes of the
// first 32-lane half (the second half adds 4).
__device__ __forceinline__ constexpr int elem_key(int v) { return 8 * (v >> 2) + (v & 3); }

// MFMA step c of S^T = K Q^T (dims 16c .. 16c+15): the K operand from LDS, by
// kKOperandReads read instructions.
constexpr int kKOperandReads = 1;
__device__ __forceinline__ bf16x8_t k_operand(const char* kt, const int* k_off, int c) {
  return *reinterpret_cast<const bf16x8_t*>(kt + k_off[c]);
}

// MFMA step k of O^T += V^T P^T (k = 0..7: d-block m = k % 4, k-group j = k / 4
// of 16 keys): the V^T operand, kVOperandReads transposed reads.  k-slot e of half h in
// k-group j is key 16j + 8(e/4) + 4h + e%4 -- the keys of P's bf16 lane
// vector pb[j].
constexpr int kVOperandReads = 2;
__device__ __forceinline__ bf16x8_t v_operand(const char* vt, const int* v_off, int k) {
  const char* a0 = vt + 16 * (k >> 2) * kRowBytes + v_off[k & 3];
  const i16x4_t lo4 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) i16x4_t*)(a0));
  const i16x4_t hi4 =
      __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) i16x4_t*)(a0 + 8 * kRowBytes));
  const i16x4_t lohi[2] = {lo4, hi4};
  bf16x8_t a;
  __builtin_memcpy(&a, lohi, sizeof(a));
  return a;
}

// Causal bound: keep elements whose key offset is <= thr (per lane).
__device__ __forceinline__ void mask_causal(f32x16_t& s, int thr) {
#pragma unroll
  for (int v = 0; v < 16; ++v) s[v] = elem_key(v) <= thr ? s[v] : -INFINITY;
}

// Window bound: keep elements whose key offset is >= thr; the elements that
// can hold sink keys (v < 4 on tile 0) compare against thr_sink instead.
__device__ __forceinline__ void mask_window(f32x16_t& s, int thr, int thr_sink) {
#pragma unroll
  for (int v = 0; v < 16; ++v) s[v] = elem_key(v) >= (v < 4 ? thr_sink : thr) ? s[v] : -INFINITY;
}


// Arrival word of (KV head, row block, workgroup position): this launch's
// epoch above the count of splits arrived under it.  A word that carries
// another epoch (another workspace's launches, a fresh buffer, or whatever
// the workspace held) counts as zero.  Each arrival adds one: when the word
// already carries this launch's epoch that is its count (one round trip:
// every arrival on a word a previous launch of this workspace left clean,
// and every arrival after the first otherwise).  An arrival that finds
// another epoch has added to a void word; it then installs this launch's
// epoch with a count of one, or -- if another arrival installed it first
// -- adds itself under it, by compare-and-swap from the value last seen.
// Either way each arrival is counted exactly once under the epoch.
// Returns the number of splits arrived, this one included.
__device__ __forceinline__ unsigned long long count_arrival(unsigned long long* ctr, unsigned long long epoch) {
  const unsigned long long old = __hip_atomic_fetch_add(ctr, 1ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  unsigned long long mine = old + 1;
  if ((old >> kEpochShift) != epoch) {
    unsigned long long seen = old + 1;  // the word if nobody else changed it since
    do {
      mine = (seen >> kEpochShift) == epoch ? seen + 1 : (epoch << kEpochShift) + 1;
    } while (!__hip_atomic_compare_exchange_strong(ctr, &seen, mine, __ATOMIC_RELAXED, __ATOMIC_RELAXED,
                                                    __HIP_MEMORY_SCOPE_AGENT));
  }
  return mine & ((1ull << kEpochShift) - 1);
}

}  // namespace tmx

#endif  // TRIANGLEMIX_DEVICE_H
