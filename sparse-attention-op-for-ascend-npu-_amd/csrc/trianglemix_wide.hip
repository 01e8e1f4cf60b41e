// The attention kernel for long work items: 64 query rows per wave.
//
// Same operator, items, splits, tiles, LDS layout and numerics as
// triangle_paged_attention_kernel (trianglemix_kernel.hip), and the same masks
// in the result (a block of sparse and dense rows takes its tiles in another
// order); another shape of wave.  There a wave owns 32 rows (one query head) and two waves share a
// SIMD; here it owns 64 (a pair of heads of the GQA group over the same 32
// tokens) and has the SIMD, with up to 512 registers, to itself:
//  * P = 4: four waves, one head pair x four KV parts, 16 workgroups per item;
//  * P = 2: four waves, two head pairs x two KV parts, 8 workgroups per item;
//  * P = 1: two waves, two head pairs, 8 workgroups per item, two per CU.
//
// What bounds it, and why this shape: at full load the chip runs this loop at
// a power-limited clock (1.8-2.1 GHz of 2.4), so time follows the energy of an
// iteration.  Every K and V operand read from LDS feeds two MFMAs instead of
// one, which halves the LDS reads of the loop, and the waves need no common
// barrier per tile (P = 4: a tile belongs to one wave alone, none at all).  A
// P = 2 iteration (32 keys of both parts for four heads) takes 0.80-0.82 us at
// 2.0 GHz where the eight-wave kernel takes 0.89 us at 1.96 GHz.  Measured, us
// before -> after: dense 2048 rows at 32768 keys 956 -> 888, TriangleMix's
// last 2048 rows of 131072 308 -> 291, dense 512 rows at 4608 keys 42.4 -> 40.6
// and at 4096 39.0 -> 35.2, the 100-row rest of an 8292-token prompt 26.2 ->
// 24.5, 2048 sparse rows 24.5 -> 23.9.  With one wave per SIMD nothing
// else covers the prologue and the merge: short items run faster in the
// eight-wave kernel (512 sparse rows 9.4 us there, 9.8 here); the rule that
// chooses is in trianglemix_capi.cpp.
//
// Pipeline of a wave with heads a and b, per tile: two windows of 16 steps.
//   window 1: QK^T of b's next tile | PV of a's present tile | softmax of a's next
//   window 2: QK^T of a's tile after | PV of b's present tile | softmax of b's next
// One MFMA per step, QK^T and PV in turn, so neither chain waits for itself;
// the K operands are read once for both heads (in window 1, for window 2 and
// the next window 1), the V operands too (in window 2).  Between the MFMAs of
// one wave about four other instructions are free; the loop has eight (tile
// addresses, byte counts and mask flags come from per-lane tables by
// v_readlane, and the running max is tested by one compare and a vote).
// The program order is fixed with scheduling barriers.
//
// Memory: tiles come by LDS DMA.  P = 4: each wave loads its own tiles (16
// instructions per iteration) into two K and two V slots of its own and waits
// for them by count; the next DMA into a slot is issued once the slot's last
// LDS read has returned.  P = 2 and 1: the two waves of a part load half a tile
// each, into three slots, and one barrier per iteration publishes tiles and
// frees slots.
#include <hip/hip_runtime.h>

#include <float.h>
#include <stdint.h>

#include "trianglemix_device.h"
#include "trianglemix_kernel.h"

namespace tmx {
namespace {

// Lambdas called from a cold branch are inlined too: as calls, their captures
// would have to live in memory.
#define TM_INLINE __attribute__((always_inline))

struct Yes { static constexpr bool value = true; };
struct No { static constexpr bool value = false; };
// Workgroup: kParts KV parts x kPairs head pairs, one wave each.
template <int P>
struct Wide {
  static constexpr int kParts = P;                       // KV parts: tiles kq, kq + P, ...
  static constexpr int kPairs = P == 4 ? 1 : 2;          // head pairs (two heads, one wave each) per part
  static constexpr int kWaves = P * kPairs;              // 4, 4, 2
  static constexpr int kThreads = kWaves * 64;
  static constexpr int kHeads = 2 * kPairs;              // query heads per workgroup
  static constexpr int kWgPerKvHead = kGroup / kHeads;   // workgroups per (row block, KV head)
  static constexpr int kSlotBytes = P * kTileBytes;      // the tiles of all parts of one iteration
  static constexpr int kDma = kDmaPerTile / kPairs;      // DMA instructions per wave, tensor and iteration
  static constexpr int kOwned = (kHeadDim / 32) / P;     // 32-wide d-blocks per head a wave keeps in the merge
  static constexpr int kQBlocksPerWave = 8 * kHeads / kWaves;  // 1 KB blocks of Q each wave DMAs
  static constexpr int kStages = P == 4 ? 2 : 3;         // K and V slots
  static_assert(kDma * kPairs == kDmaPerTile && kQBlocksPerWave * kWaves == 8 * kHeads, "the waves load whole tiles and Q");
  static_assert((P == 1 ? 2 : 1) * (2 * kStages * kSlotBytes + kHeads * kRowBlock * kRowBytes) <= 160 * 1024,
                "the workgroups of a CU (P = 1: two) fit its LDS");
};

// Wave-private tiles (P = 4): the operand that a step of a window reads, or -1.
// Window 1 reads K, window 2 V; its last read falls behind the last step.
constexpr int k_operand_at(int st) { return (st & 1) != 0 ? st >> 1 : -1; }
constexpr int v_operand_at(int st) { return (st & 1) == 0 && st > 0 ? (st >> 1) - 1 : -1; }
static_assert(k_operand_at(15) == 7 && v_operand_at(16) == 7, "a window reads eight operands");
// From this step of a window on its DMA refills the slot that the window before
// read; `but` counts the LDS reads issued since the last of those.
constexpr int kRefillStep = 6;
constexpr int k_reads_but() {
  int n = 0;
  for (int st = 0; st < kRefillStep; ++st) n += k_operand_at(st) >= 0 ? kKOperandReads : 0;
  return n;
}
constexpr int v_reads_but() {
  int n = 0;
  for (int st = 0; st < kRefillStep; ++st) n += v_operand_at(st) >= 0 ? kVOperandReads : 0;
  return n;
}

// Row max (log2 units) of a row that has met no attended key: finite, so that
// exp2(-inf - max) = 0 without a test, and so low that any real max's rescale
// factor is 0.
constexpr float kNoKeys = -FLT_MAX;

template <bool kSparse, int P>
__global__ void __launch_bounds__(Wide<P>::kThreads) __attribute__((amdgpu_waves_per_eu(1, 1)))
wide_attention_kernel(const int32_t* block_table, const __bf16* query, int query_start, int seq_len,
                      int num_row_blocks, int sparse_begin_arg, int sparse_end_arg, int split_items,
                      int split_row_blocks, int tiles_per_split, KernelParams p) {
  const PrologueArgs pa{block_table,    query,          query_start, seq_len,          num_row_blocks,
                        sparse_begin_arg, sparse_end_arg, split_items, split_row_blocks, tiles_per_split};
  using S = Wide<P>;
  constexpr int H = S::kHeads;
  constexpr int kPairs = S::kPairs;
  constexpr int NS = S::kStages;
  __shared__ __attribute__((aligned(1024))) char k_lds0[S::kSlotBytes];
  __shared__ __attribute__((aligned(1024))) char k_lds1[S::kSlotBytes];
  __shared__ __attribute__((aligned(1024))) char v_lds0[S::kSlotBytes];
  __shared__ __attribute__((aligned(1024))) char v_lds1[S::kSlotBytes];
  __shared__ __attribute__((aligned(1024))) char k_lds2[NS == 3 ? S::kSlotBytes : 16];
  __shared__ __attribute__((aligned(1024))) char v_lds2[NS == 3 ? S::kSlotBytes : 16];
  __shared__ __attribute__((aligned(1024))) char q_lds[H * kRowBlock * kRowBytes];

  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int pr = wave % kPairs;  // head pair inside the workgroup
  const int kq = wave / kPairs;  // KV part
  const int lane = tid & 63;
  const int n = lane & 31;
  const int half = lane >> 5;
  TM_PHASE(0);

  const int sparse_begin = kSparse ? pa.sparse_begin : 0;
  const int sparse_end = kSparse ? pa.sparse_end : 0;

  const int kvh = blockIdx.x % kKvHeads;
  const int hp = (blockIdx.x / kKvHeads) % S::kWgPerKvHead;
  const int item = blockIdx.x / (kKvHeads * S::kWgPerKvHead);
  int order, split, nsplit;
  if (item < pa.split_items) {
    decode_item(pa, sparse_begin, sparse_end, item, lane, order, split, nsplit);
    order = __builtin_amdgcn_readfirstlane(order);
    split = __builtin_amdgcn_readfirstlane(split);
    nsplit = __builtin_amdgcn_readfirstlane(nsplit);
  } else {
    order = pa.split_row_blocks + (item - pa.split_items);
    split = 0;
    nsplit = 1;
  }
  const int rb = pa.num_row_blocks - 1 - order;
  const int tb = pa.query_start + rb * kRowBlock;
  const int te = min(tb + kRowBlock, pa.seq_len);
  const int q = tb + n;

  TileRuns runs = row_block_tiles(tb, te, sparse_begin, sparse_end);
  const int all_tiles = runs.count();
  // A block of sparse and dense-tail rows visits every tile, and its sparse rows
  // attend none of those between the sink and their windows: nearly all.  Masking
  // them (a compare and a select for each of 16 scores of two heads, with no
  // second wave on the SIMD to hide them) makes an iteration half as long again,
  // so the sink tile is visited last, those tiles first and unmasked, and the
  // sparse rows start anew behind them (below).  Measured, us, masked -> so
  // (eight-wave kernel): the last 300 rows of 10300 52.9 -> 41.0 (48.0), the last
  // 400 of 4496 28.0 -> 23.4 (26.5), a whole 33000-token prompt 567 -> 446 (473).
  int far_block = 0;  // the first far_block tiles of the block are such
  if (kSparse && __builtin_expect(tb < sparse_end && te > sparse_end, 0)) {
    far_block = max((max(tb, sparse_begin) - kLocalWindow) / kKvTile - 1, 0);
    if (far_block > 0) runs = TileRuns{1, all_tiles - 1, 0, 1};
  }
  int t_lo = 0;
  int num_tiles = all_tiles;
  if (nsplit > 1) {
    const int base = all_tiles / nsplit;
    const int rem = all_tiles - base * nsplit;
    t_lo = split * base + min(split, rem);
    num_tiles = base + (split < rem ? 1 : 0);
  }
  const int num_iters = (num_tiles + P - 1) / P;
  // This wave's tiles: iteration j is tile kq + P j of the item, j < iters.
  const int iters = (num_tiles - kq + P - 1) / P;
  // ---- page table of this wave's tiles, Q DMA ----
  // V runs kVLag tiles behind K, the masks kMaskLag: their tables are shifted
  // by that, so one lane index serves all three.
  constexpr int kVLag = kPairs == 1 ? 2 : 1;
  constexpr int kMaskLag = 3;
  const int logical_pages = (pa.seq_len + kPageSize - 1) / kPageSize;
  const __amdgpu_buffer_rsrc_t bt_rsrc = __builtin_amdgcn_make_buffer_rsrc(
      (void*)pa.block_table, (short)0, logical_pages * 4, kBufferFlags);
  auto tile_k0 = [&](int j) TM_INLINE { return runs.tile(t_lo + kq + P * j) * kKvTile; };
  auto lane_k0 = [&](int j) TM_INLINE { return j >= 0 && j < iters ? tile_k0(j) : 0; };
  auto lane_page = [&](int j) TM_INLINE {
    const unsigned off = j >= 0 && j < iters ? (unsigned)(lane_k0(j) / kPageSize) * 4u : kOutOfRange;
    return __builtin_amdgcn_raw_buffer_load_b32(bt_rsrc, off, 0, 0);
  };
  const int phys0 = lane_page(lane);
  const int vphys0 = lane_page(lane - kVLag);
  int next_phys = lane_page(kTableTiles + lane);
  int next_vphys = lane_page(kTableTiles + lane - kVLag);
  {
    const __amdgpu_buffer_rsrc_t q_rsrc = __builtin_amdgcn_make_buffer_rsrc(
        (void*)(pa.query + ((size_t)(tb - pa.query_start) * kQueryHeads + kvh * kGroup + H * hp) * kHeadDim),
        (short)0, (te - tb - 1) * kQueryHeads * kRowBytes + H * kRowBytes, kBufferFlags);
#pragma unroll
    for (int j = 0; j < S::kQBlocksPerWave; ++j) {
      const int g = S::kQBlocksPerWave * wave + j;
      const int row = 4 * (g & 7) + (lane >> 4);
      const unsigned off = (unsigned)(row * kQueryHeads * kRowBytes + (g >> 3) * kRowBytes + 16 * k_slot(row, lane & 15));
      __builtin_amdgcn_raw_ptr_buffer_load_lds(q_rsrc, TM_LDS(q_lds + g * 1024), 16, off, 0, 0, 0);
    }
  }
  __builtin_amdgcn_sched_barrier(0);

  // ---- mask geometry ----
  const bool sparse_row = kSparse && q >= sparse_begin && q < sparse_end;
  const int lo = sparse_row ? q - kLocalWindow : 0;
  int lo_max = 0;  // the largest window start of the block's sparse rows
  if (kSparse) {
    const int last_sparse = min(te, sparse_end) - 1;
    if (last_sparse >= max(tb, sparse_begin)) lo_max = last_sparse - kLocalWindow;
  }
  const int q_rel = q - 4 * half;
  const int lo_rel = lo - 4 * half;
  // This wave's tiles that no sparse row attends come first.  The sparse rows
  // start anew at the first iteration of a round of NS at which all tiles behind
  // it are such (one place in the code, at the head of the unrolled loop); the
  // far tiles after it are masked.  Without any other tile they start anew at the
  // item's end.
  int unmasked = 0, anew = -1;  // leading tiles not masked; the iteration to start anew at
  bool none_near = false;
  if (kSparse && __builtin_expect(far_block > t_lo + kq, 0)) {
    const int far_tiles = min((far_block - t_lo - kq + P - 1) / P, iters);
    none_near = far_tiles == iters;
    anew = none_near ? -1 : (far_tiles - 1) / NS * NS;
    unmasked = none_near ? iters : anew + 1;
  }

  // Buffer base (low and high word) and byte count of a tile; first key and
  // bit 0 = some (row, key) pair of the tile is masked.
  unsigned tab_k_lo, tab_k_hi, tab_v_lo, tab_v_hi;
  int tab_k_bytes, tab_v_bytes, tab_mask;
  auto lane_addr = [&](const __bf16* cache, int j, int phys, unsigned& w0, unsigned& w1) TM_INLINE {
    phys = min(max(phys, 0), p.num_pages - 1);
    const unsigned row = ((unsigned)phys * kPageSize + (unsigned)(lane_k0(j) % kPageSize)) * kKvHeads + kvh;
    const uint64_t at = (uint64_t)cache + (uint64_t)row * kRowBytes;
    w0 = (unsigned)at;
    w1 = (unsigned)(at >> 32);
  };
  auto lane_bytes = [&](int j) TM_INLINE {
    const int valid_rows = j >= 0 && j < iters ? min(kKvTile, pa.seq_len - lane_k0(j)) : 0;
    return valid_rows > 0 ? (valid_rows - 1) * kKvHeads * kRowBytes + kRowBytes : 0;
  };
  auto lane_mask = [&](int j) TM_INLINE {
    const int k0 = lane_k0(j);
    return k0 | (int)((k0 + kKvTile - 1 > tb) | (kSparse && k0 < lo_max && j >= unmasked));
  };
  auto fill_tables = [&](int j, int phys, int vphys) TM_INLINE {  // j: this lane's tile for K
    lane_addr(p.key_cache, j, phys, tab_k_lo, tab_k_hi);
    lane_addr(p.value_cache, j - kVLag, vphys, tab_v_lo, tab_v_hi);
    tab_k_bytes = lane_bytes(j);
    tab_v_bytes = lane_bytes(j - kVLag);
    tab_mask = lane_mask(j - kMaskLag);
  };
  fill_tables(lane, phys0, vphys0);
  TM_PHASE(1);
  auto read_rsrc = [&](unsigned w0, unsigned w1, int bytes, int i) TM_INLINE {
    const uint64_t at = (uint64_t)(unsigned)__builtin_amdgcn_readlane(w0, i) |
                        ((uint64_t)(unsigned)__builtin_amdgcn_readlane(w1, i) << 32);
    return __builtin_amdgcn_make_buffer_rsrc((void*)at, (short)0, __builtin_amdgcn_readlane(bytes, i), kBufferFlags);
  };
  // Tile j of block 0 of the tables.
  auto tile_rsrc = [&](int j, int t) TM_INLINE {
    return t == 0 ? read_rsrc(tab_k_lo, tab_k_hi, tab_k_bytes, j) : read_rsrc(tab_v_lo, tab_v_hi, tab_v_bytes, j + kVLag);
  };
  // DMA instruction j of a tile loads its rows 4j .. 4j + 3 (lane / 16 within);
  // the part of the offset that no lane changes goes into the scalar offset,
  // which the buffer's range check includes.
  const int dma_j0 = (kPairs == 2 ? pr : 0) * S::kDma;
  unsigned k_voff[4];  // by j % 4
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int row = 4 * j + (lane >> 4);
    k_voff[j] = (unsigned)(row * kKvHeads * kRowBytes + 16 * k_slot(row, lane & 15));
  }
  const unsigned v_voff = (unsigned)((lane >> 4) * kKvHeads * kRowBytes + 16 * v_slot(lane >> 4, lane & 15));
  const int tile_off = kq * kTileBytes;
  const int dma_base = tile_off + dma_j0 * 1024;  // this wave's share of its part's tile
  auto dma_k = [&](__amdgpu_buffer_rsrc_t rsrc, char* lds, int j, int at) TM_INLINE {
    __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, TM_LDS(lds + at + j * 1024), 16, k_voff[j & 3],
                                             ((dma_j0 + j) >> 2) * (16 * kKvHeads * kRowBytes), 0, 0);
  };
  auto dma_v = [&](__amdgpu_buffer_rsrc_t rsrc, char* lds, int j, int at) TM_INLINE {
    __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, TM_LDS(lds + at + j * 1024), 16, v_voff,
                                             (dma_j0 + j) * (4 * kKvHeads * kRowBytes), 0, 0);
  };
  auto issue_k = [&](int i, char* lds) TM_INLINE {
    const __amdgpu_buffer_rsrc_t rsrc = tile_rsrc(i, 0);
#pragma unroll
    for (int j = 0; j < S::kDma; ++j) dma_k(rsrc, lds, j, dma_base);
    __builtin_amdgcn_sched_barrier(0);
  };
  auto issue_v = [&](int i, char* lds) TM_INLINE {
    const __amdgpu_buffer_rsrc_t rsrc = tile_rsrc(i, 1);
#pragma unroll
    for (int j = 0; j < S::kDma; ++j) dma_v(rsrc, lds, j, dma_base);
    __builtin_amdgcn_sched_barrier(0);
  };
  issue_k(0, k_lds0);

  float m_a = kNoKeys, m_b = kNoKeys;
  float l_a = 0.0f, l_b = 0.0f;
  f32x16_t o_a[kHeadDim / 32], o_b[kHeadDim / 32];
#pragma unroll
  for (int m = 0; m < kHeadDim / 32; ++m) {
    o_a[m] = f32x16_t{};
    o_b[m] = f32x16_t{};
  }

  int k_off[kHeadDim / 16];
#pragma unroll
  for (int c = 0; c < kHeadDim / 16; ++c) k_off[c] = tile_off + n * kRowBytes + 16 * k_slot(n, 2 * c + half);
  const int tr_key = 4 * (lane >> 5) + ((lane & 15) >> 2);
  int v_off[kHeadDim / 32];
#pragma unroll
  for (int m = 0; m < kHeadDim / 32; ++m) {
    const int d = 32 * m + 16 * ((lane >> 4) & 1) + 4 * (lane & 3);
    v_off[m] = tile_off + tr_key * kRowBytes + 16 * v_slot(tr_key, d >> 3) + 2 * (d & 7);
  }
  const float c2 = p.scale_log2;

  auto mask_tile = [&](f32x16_t& s, int k0) TM_INLINE {
    if (k0 + kKvTile - 1 > tb) mask_causal(s, q_rel - k0);
    if (kSparse && k0 < lo_max) {
      const int thr = lo_rel - k0;
      mask_window(s, thr, (k0 == 0 && sparse_row) ? -kKvTile : thr);
    }
  };

  // Q landed; with tiles shared by two waves, K of iteration 0 too.
  if (kPairs == 1) {
    wait_dma_but<S::kDma>();
  } else {
    issue_k(1, k_lds1);
    issue_v(0, v_lds0);
    wait_dma_but<2 * S::kDma>();
  }
  __builtin_amdgcn_s_barrier();
  TM_PHASE(2);
  bf16x8_t q_a[kHeadDim / 16], q_b[kHeadDim / 16];
  auto read_q = [&](bf16x8_t* qr, int head) TM_INLINE {
    const unsigned qb = (unsigned)(size_t)TM_LDS(q_lds + head * kRowBlock * kRowBytes) - (unsigned)tile_off;
    asm volatile(
        "ds_read_b128 %0, %8\n\t"
        "ds_read_b128 %1, %9\n\t"
        "ds_read_b128 %2, %10\n\t"
        "ds_read_b128 %3, %11\n\t"
        "ds_read_b128 %4, %12\n\t"
        "ds_read_b128 %5, %13\n\t"
        "ds_read_b128 %6, %14\n\t"
        "ds_read_b128 %7, %15\n\t"
        "s_waitcnt lgkmcnt(0)"
        : "=&a"(qr[0]), "=&a"(qr[1]), "=&a"(qr[2]), "=&a"(qr[3]), "=&a"(qr[4]), "=&a"(qr[5]),
          "=&a"(qr[6]), "=&a"(qr[7])
        : "v"(qb + k_off[0]), "v"(qb + k_off[1]), "v"(qb + k_off[2]), "v"(qb + k_off[3]), "v"(qb + k_off[4]),
          "v"(qb + k_off[5]), "v"(qb + k_off[6]), "v"(qb + k_off[7])
        : "memory");
  };
  read_q(q_a, 2 * pr);
  read_q(q_b, 2 * pr + 1);

  f32x16_t s_a, s_b;
  bf16x8_t kf[kHeadDim / 16], va[8];
  u32x4_t p_a[2], p_b[2];  // bf16 probabilities, two per word
  // Lazy rescale: O and the row sum are rescaled only when some raw score of
  // the tile exceeds thr = (largest raw score of the row at the last rescale)
  // + 8 / c2, i.e. when some probability would exceed 2^8.  A row without
  // attended keys so far has thr = -inf and m = kNoKeys.  A lane compares its
  // own half of the row's keys: the vote over the wave sees both halves.
  const float lazy = fminf(kLazyRescale / c2, FLT_MAX);  // finite: -inf + lazy stays -inf
  float thr_a = -INFINITY, thr_b = -INFINITY;
  auto mfma = [](bf16x8_t a, bf16x8_t b, f32x16_t c)
                  TM_INLINE { return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0); };
  auto prob = [](const u32x4_t* pp, int j) TM_INLINE { return __builtin_bit_cast(bf16x8_t, pp[j]); };
  // exponentials of elements 2i, 2i + 1
  auto exp_pair = [&](const f32x16_t& s, int i, float shift, float* x) TM_INLINE {
    x[0] = __builtin_amdgcn_exp2f(__builtin_fmaf(s[2 * i], c2, -shift));
    x[1] = __builtin_amdgcn_exp2f(__builtin_fmaf(s[2 * i + 1], c2, -shift));
  };
  // Adds them to the tile's sum (pair 0 starts it) and rounds them to bf16.
  auto add_pair = [&](const float* x, int i, float& sum, u32x4_t* pp) TM_INLINE {
    typedef float f32x2_t __attribute__((ext_vector_type(2)));
    typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
    sum = i == 0 ? x[0] : sum + x[0];
    sum += x[1];
    unsigned w = __builtin_bit_cast(unsigned, __builtin_convertvector((f32x2_t{x[0], x[1]}), bf16x2_t));
    asm volatile("" : "+v"(sum), "+v"(w));
    pp[i >> 2][i & 3] = w;
  };
  // The sparse rows of a head start anew: by selects, as what they summed may be infinite or NaN.
  auto start_anew = [&](float& m_x, float& thr_x, float& l_x, f32x16_t* o_x, u32x4_t* p_x) TM_INLINE {
    m_x = sparse_row ? kNoKeys : m_x;
    thr_x = sparse_row ? -INFINITY : thr_x;
    l_x = sparse_row ? 0.0f : l_x;
#pragma unroll
    for (int m = 0; m < kHeadDim / 32; ++m) {
#pragma unroll
      for (int v = 0; v < 16; ++v) o_x[m][v] = sparse_row ? 0.0f : o_x[m][v];
    }
#pragma unroll
    for (int i = 0; i < 8; ++i) p_x[i >> 2][i & 3] = sparse_row ? 0u : p_x[i >> 2][i & 3];
  };
  // Half an iteration of the pipeline, 16 steps: the QK^T MFMAs of head y
  // (even steps) alternate with the PV MFMAs of head x's present tile (odd
  // steps) -- two independent chains -- while the VALU takes the row max and
  // the exponentials of head x's next tile (scores s_x; its QK^T ended the
  // window before) into p_x.  `mem` issues each step's LDS reads and DMA.  A tile's 16 probabilities per lane are summed by themselves and
  // added once to the running row sum, so that the row sum is rounded once per
  // tile against the whole sum, as in the eight-wave kernel, and not 16 times
  // (one dominant key and all others alike, 1024 tiles: the outputs were 2.8e-4
  // off in the mean, now 9.7e-6; the calls take the same time, 890 us).
  auto window = [&](auto qk, auto pv, auto first, f32x16_t& s_y, const bf16x8_t* q_y, f32x16_t& s_x, int mask_x,
                    u32x4_t* p_x, float& m_x, float& thr_x, float& l_x, f32x16_t* o_x, auto mem) TM_INLINE {
    constexpr bool kQk = decltype(qk)::value, kPv = decltype(pv)::value, kFirst = decltype(first)::value;
    u32x4_t pn[2];
    float t = 0.0f, alpha = 1.0f, tile_sum = 0.0f;
    bool grow = false;
    float x[2];
#pragma unroll
    for (int k = 0; k < 16; ++k) {
      mem(k);
      if ((k & 1) == 0) {
        if (kQk) s_y = mfma(kf[k >> 1], q_y[k >> 1], k == 0 ? f32x16_t{} : s_y);
      } else if (kPv) {
        o_x[(k >> 1) & 3] = mfma(va[k >> 1], prob(p_x, k >> 3), o_x[(k >> 1) & 3]);
      }
      if (k == 0) {
        __builtin_amdgcn_sched_barrier(0);
        if (__builtin_expect(mask_x & 1, 0)) mask_tile(s_x, mask_x & ~1);
      }
      if (k == 1) {
        t = fmaxf(s_x[0], s_x[1]);
#pragma unroll
        for (int v = 2; v < 8; ++v) t = fmaxf(t, s_x[v]);
        asm volatile("" : "+v"(t));
      }
      if (k == 2) {
#pragma unroll
        for (int v = 8; v < 16; ++v) t = fmaxf(t, s_x[v]);
        asm volatile("" : "+v"(t));
      }
      if (k == 3) {
        if (kFirst) {
          t = half_max(t);
          m_x = fmaxf(t * c2, kNoKeys);
          thr_x = t + lazy;
        } else {
          grow = __any(t > thr_x);
          if (__builtin_expect(grow, 0)) {
            t = half_max(t);
            const float m_new = fmaxf(m_x, t * c2);
            alpha = __builtin_amdgcn_exp2f(m_x - m_new);
            thr_x = fmaxf(thr_x, t + lazy);
            l_x *= alpha;
            m_x = m_new;
          }
        }
      }
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        if (k == 5 + (i * 10) / 8) add_pair(x, i, tile_sum, pn);
        if (k == 4 + (i * 10) / 8) exp_pair(s_x, i, m_x, x);
      }
      if (k == 15) l_x += tile_sum;
      __builtin_amdgcn_sched_barrier(0);
    }
    mem(16);
    if (kPv && !kFirst) {
      if (__builtin_expect(grow, 0)) {
#pragma unroll
        for (int m = 0; m < kHeadDim / 32; ++m) o_x[m] *= alpha;
      }
    }
    p_x[0] = pn[0];
    p_x[1] = pn[1];
  };
  auto read_k = [&](const char* slot, int c) TM_INLINE { kf[c] = k_operand(slot, k_off, c); };
  auto read_v = [&](const char* slot, int c) TM_INLINE { va[c] = v_operand(slot, v_off, c); };
  // vmcnt bookkeeping below: each wave's DMA is issued in the order K(0), K(1),
  // V(0), then K(2), V(1), K(3), V(2), ... (wave-private tiles) or V(1), K(2),
  // V(2), K(3), ... (shared tiles), kDma instructions each.
  constexpr int kD = S::kDma;
  if (kPairs == 1) {
    issue_k(1, k_lds1);
    wait_dma_but<kD>();  // K(0) landed
  }
  if (iters > 0) {
    const int mask0 = __builtin_amdgcn_readlane(tab_mask, kMaskLag);
    const __amdgpu_buffer_rsrc_t v0 = tile_rsrc(0, 1), v1 = tile_rsrc(1, 1), k2 = tile_rsrc(2, 0);
#pragma unroll
    for (int c = 0; c < kHeadDim / 16; ++c) read_k(k_lds0, c);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int c = 0; c < kHeadDim / 16; ++c) {
      if (kPairs == 1) dma_v(v0, v_lds0, c, dma_base);
      s_a = mfma(kf[c], q_a[c], c == 0 ? f32x16_t{} : s_a);
      __builtin_amdgcn_sched_barrier(0);
    }
    TM_PHASE(3);
    const __amdgpu_buffer_rsrc_t v2 = tile_rsrc(2, 1), k3 = tile_rsrc(3, 0);
    window(Yes{}, No{}, Yes{}, s_b, q_b, s_a, mask0, p_a, m_a, thr_a, l_a, o_a, [&](int st) TM_INLINE {
      // K(0) has been read: its last operand was waited for by the first QK^T
      if (kPairs == 1) {
        if (st < 8) dma_k(k2, k_lds0, st, dma_base);
        if (st == 8) wait_dma_but<2 * kD>();  // K(1) landed; behind it V(0), K(2)
        if (st >= 8 && st < 16) dma_v(v1, v_lds1, st - 8, dma_base);
      } else {
        if (st < 8 && (st & 1) == 0) dma_v(v1, v_lds1, st >> 1, dma_base);
        if (st < 8 && (st & 1)) dma_k(k2, k_lds2, st >> 1, dma_base);
        if (st == 8) {
          // K(1) and V(0) landed, behind them V(1), K(2); every wave has read K(0)
          wait_dma_but<2 * kD>();
          __builtin_amdgcn_s_barrier();
        }
        if (st >= 9 && (st & 1)) dma_v(v2, v_lds2, (st - 9) >> 1, dma_base);
        if (st >= 10 && (st & 1) == 0) dma_k(k3, k_lds0, (st - 10) >> 1, dma_base);
      }
      if (st >= 9) read_k(k_lds1, st - 9);
    });
    if (kPairs == 1) wait_dma_but<2 * kD>();  // V(0) landed; behind it K(2), V(1)
    if (iters > 1) {
      window(Yes{}, No{}, Yes{}, s_a, q_a, s_b, mask0, p_b, m_b, thr_b, l_b, o_b, [&](int st) TM_INLINE {
        if (kPairs == 1) {
          // K(1) has been read
          if (st == kRefillStep) wait_lds_but<v_reads_but()>();
          if (st >= kRefillStep && st < kRefillStep + 8) dma_k(k3, k_lds1, st - kRefillStep, dma_base);
        }
        if (v_operand_at(st) >= 0) read_v(v_lds0, v_operand_at(st));
      });
    } else {
      window(No{}, No{}, Yes{}, s_a, q_a, s_b, mask0, p_b, m_b, thr_b, l_b, o_b, [&](int st) TM_INLINE {
        if (st < 8) read_v(v_lds0, st);
      });
    }
  } else if (kPairs == 2) {
    __builtin_amdgcn_s_barrier();  // the other part's barrier above
  }

  // Iteration it: [QK b of it + 1, PV a of it, softmax a of it + 1], then
  // [QK a of it + 2, PV b of it, softmax b of it + 1].  kr: K slot of it + 2;
  // kw: K slot of it + 1 (shared tiles: takes K of it + 1 + NS); vw: V slot of
  // it (takes V of it + NS); vr: V slot of it + 1.
  auto iteration = [&](int it, char* kr, char* kw, char* vw, char* vr) TM_INLINE {
    if (it < 8) TM_PHASE(4 + it);
    const int kj = kPairs == 1 ? it + 2 + NS : it + 1 + NS;
    if (__builtin_expect((kj & (kTableTiles - 1)) == 0, 0)) {
      fill_tables(kj + lane, next_phys, next_vphys);
      next_phys = lane_page(kj + kTableTiles + lane);
      next_vphys = lane_page(kj + kTableTiles + lane - kVLag);
    }
    // An opaque zero per iteration keeps the 32 LDS addresses of the DMA from
    // being hoisted into as many scalar registers.
    int zero;
    asm volatile("s_mov_b32 %0, 0" : "=s"(zero));
    const int dma_at = __builtin_amdgcn_readfirstlane(dma_base + zero);
    const __amdgpu_buffer_rsrc_t v_rsrc = read_rsrc(tab_v_lo, tab_v_hi, tab_v_bytes, kj);
    const __amdgpu_buffer_rsrc_t k_rsrc = read_rsrc(tab_k_lo, tab_k_hi, tab_k_bytes, kj);
    const int mask0 = __builtin_amdgcn_readlane(tab_mask, kj);
    if (kPairs == 1) wait_dma_but<2 * kD>();  // K(it + 2) landed; behind it V(it + 1), K(it + 3)
    window(Yes{}, Yes{}, No{}, s_b, q_b, s_a, mask0, p_a, m_a, thr_a, l_a, o_a, [&](int st) {
      if (kPairs == 2) {
        if (st == 6) {
          // V(it) has been read by this wave, K(it + 2) and V(it + 1) landed;
          // behind them V(it + 2), K(it + 3)
          __builtin_amdgcn_s_waitcnt(0x0070 | (2 * kD & 15) | ((2 * kD >> 4) << 14));
          __builtin_amdgcn_s_barrier();
        }
        if (st >= 7 && st <= 13) read_k(kr, st - 7);
        if (st == 15) read_k(kr, 7);
        if (st >= 7 && st < 15) {
          if (st & 1) dma_v(v_rsrc, vw, (st - 7) >> 1, dma_at);
          else dma_k(k_rsrc, kw, (st - 8) >> 1, dma_at);
        }
      } else {
        // V(it) has been read
        if (st == kRefillStep) wait_lds_but<k_reads_but()>();
        if (k_operand_at(st) >= 0) read_k(kr, k_operand_at(st));
        if (st >= kRefillStep && st < kRefillStep + 8) dma_v(v_rsrc, vw, st - kRefillStep, dma_at);
      }
    });
    if (kPairs == 1) wait_dma_but<2 * kD>();  // V(it + 1) landed; behind it K(it + 3), V(it + 2)
    window(Yes{}, Yes{}, No{}, s_a, q_a, s_b, mask0, p_b, m_b, thr_b, l_b, o_b, [&](int st) {
      if (kPairs == 1) {
        // K(it + 2) has been read
        if (st == kRefillStep) wait_lds_but<v_reads_but()>();
        if (st >= kRefillStep && st < kRefillStep + 8) dma_k(k_rsrc, kr, st - kRefillStep, dma_at);
      }
      if (v_operand_at(st) >= 0) read_v(vr, v_operand_at(st));
    });
  };
  int it = 0;
  const int full = iters - 2;
  // At the head of an iteration both heads' probabilities of its tile are not
  // multiplied yet and the scores of head a's next tile not looked at.
  auto check_anew = [&]() TM_INLINE {
    if (kSparse && __builtin_expect(it == anew, 0)) {
      start_anew(m_a, thr_a, l_a, o_a, p_a);
      start_anew(m_b, thr_b, l_b, o_b, p_b);
    }
  };
  if constexpr (NS == 2) {
    for (; it + 1 < full; it += 2) {
      check_anew();
      iteration(it, k_lds0, k_lds1, v_lds0, v_lds1);
      iteration(it + 1, k_lds1, k_lds0, v_lds1, v_lds0);
    }
  } else {
    for (; it + 2 < full; it += 3) {
      check_anew();
      iteration(it, k_lds2, k_lds1, v_lds0, v_lds1);
      iteration(it + 1, k_lds0, k_lds2, v_lds1, v_lds2);
      iteration(it + 2, k_lds1, k_lds0, v_lds2, v_lds0);
    }
  }
  check_anew();
  if (it < full) {
    iteration(it, NS == 2 ? k_lds0 : k_lds2, k_lds1, v_lds0, v_lds1);
    ++it;
    if (NS == 3 && it < full) {
      iteration(it, k_lds0, k_lds2, v_lds1, v_lds2);
      ++it;
    }
  }
  // The last two tiles: no QK^T follows the last one's.
  wait_dma();
  if (iters > 1) {
    if (it < 8) TM_PHASE(4 + it);
    const int mask0 = __builtin_amdgcn_readfirstlane(lane_mask(iters - 1));
    window(Yes{}, Yes{}, No{}, s_b, q_b, s_a, mask0, p_a, m_a, thr_a, l_a, o_a, [&](int st) {
      if (kPairs == 2 && st == 2) __builtin_amdgcn_s_barrier();  // V of the last tile landed
    });
    const int vs = (iters - 1) % NS;
    const char* vr = vs == 0 ? v_lds0 : (vs == 1 ? v_lds1 : v_lds2);
    window(No{}, Yes{}, No{}, s_a, q_a, s_b, mask0, p_b, m_b, thr_b, l_b, o_b, [&](int st) {
      if (v_operand_at(st) >= 0) read_v(vr, v_operand_at(st));
    });
  }
  if (kPairs == 2) {
    // the parts with a tile less take the barriers of the others
    for (int b = max(iters - 1, 0); b < num_iters - 1; ++b) __builtin_amdgcn_s_barrier();
  }
  if (iters > 0) {
#pragma unroll
    for (int k = 0; k < 8; ++k) o_a[k & 3] = mfma(va[k], prob(p_a, k >> 2), o_a[k & 3]);
#pragma unroll
    for (int k = 0; k < 8; ++k) o_b[k & 3] = mfma(va[k], prob(p_b, k >> 2), o_b[k & 3]);
    if (kSparse && __builtin_expect(none_near, 0)) {
      start_anew(m_a, thr_a, l_a, o_a, p_a);
      start_anew(m_b, thr_b, l_b, o_b, p_b);
    }
  }

  TM_PHASE(12);
  // ---- merge the P KV parts through LDS ----
  // Part kq keeps d-blocks kq * O .. + O - 1 of both heads.
  constexpr int O = S::kOwned;
  f32x16_t keep_a[kHeadDim / 32], keep_b[kHeadDim / 32];
  if constexpr (P == 1) {
#pragma unroll
    for (int m = 0; m < kHeadDim / 32; ++m) {
      keep_a[m] = o_a[m];
      keep_b[m] = o_b[m];
    }
  } else {
    // Where a wave hands a d-block over: 4 KB stretches [v/4][lane][4].
    // P = 4: its own K and V slots (its DMA has landed and nobody else reads
    // them), so it writes as soon as its own last PV is done.  P = 2: the K
    // slots and q_lds, which no wave reads or loads any more once all have
    // taken the barrier of the second-to-last iteration; an item of one
    // iteration had no such barrier.
    if (kPairs == 2 && num_iters == 1) __syncthreads();
    constexpr int kStretch = 4 * 64 * 16, kStats = 4 * 64 * 4;
    static_assert(P != 4 || (S::kWaves * kTileBytes == S::kSlotBytes && 2 * kStretch <= kTileBytes &&
                             kStats <= kTileBytes && 4 - O == 3),
                  "P = 4: a given block of both heads fits the wave's tile of each of three slots, the statistics the fourth's");
    static_assert(P != 2 || (S::kWaves * kStretch <= S::kSlotBytes && S::kWaves * kStretch <= 16384 && 4 - O == 2 &&
                             16384 + S::kWaves * kStats <= H * kRowBlock * kRowBytes),
                  "P = 2: three K slots and half of q_lds hold the given blocks, the rest of q_lds the statistics");
    auto xo = [&](int g, int gi, int w) -> f32x4_t* {  // head g, gi-th given block, wave w
      if constexpr (P == 4) {
        char* base = gi == 0 ? k_lds0 : (gi == 1 ? k_lds1 : v_lds0);
        return reinterpret_cast<f32x4_t*>(base + w * kTileBytes + g * 4096);
      } else {
        char* base = gi == 0 ? (g == 0 ? k_lds0 : k_lds1) : (g == 0 ? k_lds2 : q_lds);
        return reinterpret_cast<f32x4_t*>(base + w * 4096);
      }
    };
    // [m a, l a, m b, l b][lane] of wave w
    auto xs = [&](int w) -> float* {
      return reinterpret_cast<float*>(P == 4 ? v_lds1 + w * kTileBytes : q_lds + 16384 + w * 1024);
    };
    auto given_index = [](int m, int r) { return m < r * O ? m : m - O; };
#pragma unroll
    for (int m = 0; m < kHeadDim / 32; ++m) {
      if (m / O == kq) continue;
      f32x4_t* da = xo(0, given_index(m, kq), wave) + lane;
      f32x4_t* db = xo(1, given_index(m, kq), wave) + lane;
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        da[g * 64] = f32x4_t{o_a[m][4 * g], o_a[m][4 * g + 1], o_a[m][4 * g + 2], o_a[m][4 * g + 3]};
        db[g * 64] = f32x4_t{o_b[m][4 * g], o_b[m][4 * g + 1], o_b[m][4 * g + 2], o_b[m][4 * g + 3]};
      }
    }
    float* own = xs(wave) + lane;
    own[0] = m_a;
    own[64] = l_a;
    own[128] = m_b;
    own[192] = l_b;
    __syncthreads();
    auto merge = [&](int g, const f32x16_t* o, f32x16_t* keep, float& m_run, float& l_run) {
      float mq[4], lq[4];
      float mu = kNoKeys;
#pragma unroll
      for (int r = 0; r < P; ++r) {
        const float* st = xs(r * kPairs + pr) + 128 * g + lane;
        mq[r] = st[0];
        lq[r] = st[64];
        mu = fmaxf(mu, mq[r]);
      }
      float lt = 0.0f;
#pragma unroll
      for (int r = 0; r < P; ++r) lt += lq[r] * __builtin_amdgcn_exp2f(mq[r] - mu);
      const float self_scale = __builtin_amdgcn_exp2f(m_run - mu);
#pragma unroll
      for (int m = 0; m < kHeadDim / 32; ++m) {
        if (m / O != kq) continue;
        f32x16_t acc = o[m] * self_scale;
#pragma unroll
        for (int r = 0; r < P; ++r) {
          if (r == kq) continue;
          const float a = __builtin_amdgcn_exp2f(mq[r] - mu);
          const f32x4_t* src = xo(g, given_index(m, r), r * kPairs + pr) + lane;
#pragma unroll
          for (int v = 0; v < 4; ++v) {
            const f32x4_t x = src[v * 64];
#pragma unroll
            for (int e = 0; e < 4; ++e) acc[4 * v + e] += x[e] * a;
          }
        }
        keep[m % O] = acc;
      }
      l_run = lt;
      m_run = mu;
    };
    merge(0, o_a, keep_a, m_a, l_a);
    merge(1, o_b, keep_b, m_b, l_b);
  }

  constexpr int kCpolAgent = 16;  // sc1
  constexpr int kStageRow = H * kRowBytes;
  constexpr int kChunksPerRow = kStageRow / 16;
  constexpr int kRowsPerStore = 64 / kChunksPerRow;
  constexpr int kStores = kRowBlock / (kRowsPerStore * S::kWaves);
  static_assert(kRowsPerStore * kChunksPerRow == 64 && kStores * kRowsPerStore * S::kWaves == kRowBlock,
                "the stores cover the row block");
  static_assert(kRowBlock * kStageRow <= H * kRowBlock * kRowBytes, "the stage fits q_lds");
  auto stage_block = [&](const f32x16_t& blk, float inv, int head, int m, char* stage) TM_INLINE {
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      bf16x4_t o4;
#pragma unroll
      for (int e = 0; e < 4; ++e) o4[e] = (__bf16)(blk[4 * g + e] * inv);
      const int chunk = (head * (kRowBytes / 16) + 4 * m + g) ^ (n & 15);
      *reinterpret_cast<bf16x4_t*>(stage + n * kStageRow + 16 * chunk + 8 * half) = o4;
    }
  };
  auto inverse = [&](float l_lane) TM_INLINE {
    const float l_tot = half_sum(l_lane);
    return l_tot > 0.0f ? 1.0f / l_tot : 0.0f;
  };
  auto stage_rows = [&](const f32x16_t* blocks, float l_lane, int head, char* stage) TM_INLINE {
    const float inv = inverse(l_lane);
#pragma unroll
    for (int o = 0; o < O; ++o) stage_block(blocks[o], inv, head, kq * O + o, stage);
  };
  auto store_stage = [&](const char* stage) TM_INLINE {
    __syncthreads();
    const __amdgpu_buffer_rsrc_t out_rsrc = __builtin_amdgcn_make_buffer_rsrc(
        (void*)(p.out + ((size_t)(tb - pa.query_start) * kQueryHeads + kvh * kGroup + H * hp) * kHeadDim), (short)0,
        (te - tb - 1) * kQueryHeads * kRowBytes + kStageRow, kBufferFlags);
    const int c = lane % kChunksPerRow;
#pragma unroll
    for (int j = 0; j < kStores; ++j) {
      const int r = (wave * kStores + j) * kRowsPerStore + lane / kChunksPerRow;
      const u32x4_t v = *reinterpret_cast<const u32x4_t*>(stage + r * kStageRow + 16 * (c ^ (r & 15)));
      __builtin_amdgcn_raw_buffer_store_b128(v, out_rsrc, (unsigned)(r * kQueryHeads * kRowBytes + 16 * c), 0,
                                             kCpolAgent);
    }
  };
  // Stage: q_lds, last read in the prologue (P = 2: by the merge above, which
  // must end first).
  char* const stage = q_lds;
  TM_PHASE(13);
  if (nsplit == 1) {
    if constexpr (P == 2) __syncthreads();
    stage_rows(keep_a, l_a, 2 * pr, stage);
    stage_rows(keep_b, l_b, 2 * pr + 1, stage);
    store_stage(stage);
    TM_PHASE(14);
    return;
  }

  // ---- split-KV, merged in this launch ----
  // Records, arrival words and their protocol are those of the eight-wave
  // kernel (trianglemix_kernel.hip): every split writes its partial through to
  // the level where all L2s are coherent and counts its arrival, and the
  // workgroup that counts last merges all partials in split order.
  constexpr int kStatM = kGroup * 64 * 64;
  constexpr int kStatL = kGroup * 64 * 65;
  const int first = item - split;
  const int hq = H * hp + 2 * pr;  // head a inside the GQA group; head b is hq + 1
  const __amdgpu_buffer_rsrc_t rec = __builtin_amdgcn_make_buffer_rsrc(
      (void*)(p.partials + ((size_t)kvh * pa.split_items + first) * kPartialFloats), (short)0,
      nsplit * (int)kPartialBytes, kBufferFlags);
  auto blk_off = [&](int s, int h, int o, int g) {
    return (unsigned)(s * (int)kPartialBytes + (((((hq + h) * 4 + kq * O + o) * 4 + g) * 64 + lane) * 4) * 4);
  };
#pragma unroll
  for (int o = 0; o < O; ++o) {
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const f32x4_t xa = {keep_a[o][4 * g], keep_a[o][4 * g + 1], keep_a[o][4 * g + 2], keep_a[o][4 * g + 3]};
      const f32x4_t xb = {keep_b[o][4 * g], keep_b[o][4 * g + 1], keep_b[o][4 * g + 2], keep_b[o][4 * g + 3]};
      __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4_t, xa), rec, blk_off(split, 0, o, g), 0, kCpolAgent);
      __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4_t, xb), rec, blk_off(split, 1, o, g), 0, kCpolAgent);
    }
  }
  if (kq == 0) {
    const unsigned so = (unsigned)(split * (int)kPartialBytes + (hq * 64 + lane) * 4);
    __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(m_a), rec, so + kStatM * 4, 0, kCpolAgent);
    __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(l_a), rec, so + kStatL * 4, 0, kCpolAgent);
    __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(m_b), rec, so + 256 + kStatM * 4, 0, kCpolAgent);
    __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(l_b), rec, so + 256 + kStatL * 4, 0, kCpolAgent);
  }
  wait_dma();
  TM_PHASE(16);
  __syncthreads();
  // the merge's reads of k_lds0 ended before the barrier above
  volatile int* s_last = reinterpret_cast<volatile int*>(k_lds0);
  unsigned long long* ctr = p.counters + ((size_t)kvh * pa.split_row_blocks + order) * S::kWgPerKvHead + hp;
  if (tid == 0) {
    *s_last = (int)(count_arrival(ctr, p.epoch) == (unsigned long long)nsplit);
  }
  __syncthreads();
  TM_PHASE(17);
  if (!*s_last) return;
  if (tid == 0) __hip_atomic_store(ctr, p.epoch << kEpochShift, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);

  constexpr int kMergeBatch = P == 2 ? 2 : 4;
  if constexpr (P != 1) {
    f32x16_t acc[2][kHeadDim / 32];
    float mt[2] = {kNoKeys, kNoKeys}, lt[2] = {0.0f, 0.0f};
#pragma unroll
    for (int h = 0; h < 2; ++h) {
#pragma unroll
      for (int o = 0; o < O; ++o) acc[h][o] = f32x16_t{};
    }
    for (int s0 = 0; s0 < nsplit; s0 += kMergeBatch) {
      float ms[2][4], ls[2][4];  // fixed sizes (see keep_a); the first kMergeBatch are used
      f32x4_t xs[2][4][kHeadDim / 32][4];
#pragma unroll
      for (int b = 0; b < kMergeBatch; ++b) {
        const int sb = s0 + b;
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          if (sb == split || sb >= nsplit) {
            // This workgroup's own partial: the values it stored are still in
            // registers, so it is not loaded back.
            ms[h][b] = h == 0 ? m_a : m_b;
            ls[h][b] = h == 0 ? l_a : l_b;
#pragma unroll
            for (int o = 0; o < O; ++o) {
              const f32x16_t own = h == 0 ? keep_a[o] : keep_b[o];
#pragma unroll
              for (int g = 0; g < 4; ++g) {
                xs[h][b][o][g] = f32x4_t{own[4 * g], own[4 * g + 1], own[4 * g + 2], own[4 * g + 3]};
              }
            }
            continue;
          }
          const unsigned so = (unsigned)(sb * (int)kPartialBytes + ((hq + h) * 64 + lane) * 4);
          ms[h][b] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(rec, so + kStatM * 4, 0, kCpolAgent));
          ls[h][b] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(rec, so + kStatL * 4, 0, kCpolAgent));
#pragma unroll
          for (int o = 0; o < O; ++o) {
#pragma unroll
            for (int g = 0; g < 4; ++g) {
              xs[h][b][o][g] = __builtin_bit_cast(
                  f32x4_t, __builtin_amdgcn_raw_buffer_load_b128(rec, blk_off(sb, h, o, g), 0, kCpolAgent));
            }
          }
        }
      }
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        float mu = mt[h];
#pragma unroll
        for (int b = 0; b < kMergeBatch; ++b) mu = s0 + b < nsplit ? fmaxf(mu, ms[h][b]) : mu;
        const float scale = __builtin_amdgcn_exp2f(mt[h] - mu);
        lt[h] *= scale;
#pragma unroll
        for (int o = 0; o < O; ++o) acc[h][o] *= scale;
#pragma unroll
        for (int b = 0; b < kMergeBatch; ++b) {
          const float w = s0 + b < nsplit ? __builtin_amdgcn_exp2f(ms[h][b] - mu) : 0.0f;
          lt[h] += ls[h][b] * w;
#pragma unroll
          for (int o = 0; o < O; ++o) {
#pragma unroll
            for (int g = 0; g < 4; ++g) {
#pragma unroll
              for (int e = 0; e < 4; ++e) acc[h][o][4 * g + e] += xs[h][b][o][g][e] * w;
            }
          }
        }
        mt[h] = mu;
      }
      if (s0 == 0) TM_PHASE(18);
    }
    TM_PHASE(19);
    stage_rows(acc[0], lt[0], 2 * pr, stage);
    stage_rows(acc[1], lt[1], 2 * pr + 1, stage);
  } else {
    // One head and d-block after the other, kMergeBatch splits at a time with all
    // of a batch's loads in flight: the sums of one block stay in 16 registers,
    // whatever the shape.  Slots past the last split load the last one again
    // (weight 0).
  #pragma unroll
    for (int h = 0; h < 2; ++h) {
  #pragma unroll 1
      for (int o = 0; o < O; ++o) {
        f32x16_t acc{};
        float mt = kNoKeys, lt = 0.0f;
        for (int s0 = 0; s0 < nsplit; s0 += kMergeBatch) {
          float ms[kMergeBatch], ls[kMergeBatch];
          f32x4_t xs[kMergeBatch][4];
  #pragma unroll
          for (int b = 0; b < kMergeBatch; ++b) {
            const int sb = min(s0 + b, nsplit - 1);
            const unsigned so = (unsigned)(sb * (int)kPartialBytes + ((hq + h) * 64 + lane) * 4);
            ms[b] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(rec, so + kStatM * 4, 0, kCpolAgent));
            ls[b] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(rec, so + kStatL * 4, 0, kCpolAgent));
  #pragma unroll
            for (int g = 0; g < 4; ++g) {
              xs[b][g] =
                  __builtin_bit_cast(f32x4_t, __builtin_amdgcn_raw_buffer_load_b128(rec, blk_off(sb, h, o, g), 0, kCpolAgent));
            }
          }
          float mu = mt;
  #pragma unroll
          for (int b = 0; b < kMergeBatch; ++b) mu = fmaxf(mu, ms[b]);
          const float scale = __builtin_amdgcn_exp2f(mt - mu);
          lt *= scale;
          acc *= scale;
  #pragma unroll
          for (int b = 0; b < kMergeBatch; ++b) {
            const float w = s0 + b < nsplit ? __builtin_amdgcn_exp2f(ms[b] - mu) : 0.0f;
            lt += ls[b] * w;
  #pragma unroll
            for (int g = 0; g < 4; ++g) {
  #pragma unroll
              for (int e = 0; e < 4; ++e) acc[4 * g + e] += xs[b][g][e] * w;
            }
          }
          mt = mu;
          if (h == 0 && o == 0 && s0 == 0) TM_PHASE(18);
        }
        stage_block(acc, inverse(lt), 2 * pr + h, kq * O + o, stage);
      }
    }
    TM_PHASE(19);
  }
  store_stage(stage);
  TM_PHASE(15);
}

template <bool kSparse, int P>
hipError_t launch(const KernelParams& p, hipStream_t stream) {
  hipLaunchKernelGGL((wide_attention_kernel<kSparse, P>),
                     dim3((unsigned)(p.items_per_head * Wide<P>::kWgPerKvHead * kKvHeads)),
                     dim3(Wide<P>::kThreads), 0,
                     stream, p.block_table, p.query, p.query_start, p.seq_len, p.num_row_blocks, p.sparse_begin,
                     p.sparse_end, p.split_items, p.split_row_blocks, p.tiles_per_split, p);
  return hipGetLastError();
}

}  // namespace

#ifdef TRIANGLEMIX_PHASE_CLOCKS
hipError_t wide_phase_clocks(void** ptr) { return hipGetSymbolAddress(ptr, HIP_SYMBOL(phase_clocks)); }
#endif

hipError_t launch_wide_attention(const KernelParams& p, bool sparse, int kv_parts, hipStream_t stream) {
  if (kv_parts == 1) return sparse ? launch<true, 1>(p, stream) : launch<false, 1>(p, stream);
  if (kv_parts == 2) return sparse ? launch<true, 2>(p, stream) : launch<false, 2>(p, stream);
  return sparse ? launch<true, 4>(p, stream) : launch<false, 4>(p, stream);
}

}  // namespace tmx
