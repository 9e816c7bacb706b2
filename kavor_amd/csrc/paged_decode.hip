// Paged decode attention: one query token per sequence against its paged KV cache.
//
// Restates flash_attn_with_kvcache(q.unsqueeze(1), k_cache, v_cache, cache_seqlens,
// block_table, softmax_scale, causal=True) as used at
// kavor/layers/attention/flash_attention_kvcache.py:80-83.
//
// What bounds it: HBM, since every K/V byte is read exactly once; for the smallest batches
// the chain of dependent loads and the instructions around it.
//
// Work decomposition -- stream-K
//   Work is counted in steps of 32 tokens of one sequence; the steps of all sequences are
//   laid end to end (prefix sums of ceil(ctx / 32), built in LDS by every workgroup from
//   context_lens).  The grid is the number of workgroups the GPU holds at once (one of 4
//   waves per CU; two for many sequences at G = 1, see steps_ahead), and no more than the
//   block tables can hold steps for, so a captured graph launches few empty workgroups.  A
//   workgroup's waves are 4 kv heads; ceil(Hkv / 4) workgroups walk one contiguous range of
//   steps for all kv heads (kv heads of one token row share HBM pages and are fetched
//   together).  Every range gets the same number of steps (exact balance whatever the context
//   lengths).  A wave owns all G = Hq / Hkv query heads of its kv head, so GQA costs no extra
//   KV traffic.
//
// Why the matrix cores, although the work is HBM-bound: on the vector ALUs the q.k dot
// products, their lane sums and the P V products grow with G while the K/V bytes do not.
// At G = 8 a wave needed more issue cycles for a step than HBM needs to deliver it, and the
// registers that held the K/V double buffer were short.  Here both products run as
// v_mfma_f32_16x16x32_bf16 with the G heads as columns, a fixed 16 (G <= 5) or 24 (G = 8)
// matrix instructions per step.  Measured against the vector-ALU kernel (MI355X, whole
// calls, the two in turn): 64 sequences of 1000-9000 tokens at G = 8, one-launch step:
// 382 -> 215 us (3.4 -> 6.1 TB/s); 256 sequences of 100-2048 tokens at G = 2, with the append:
// 182 -> 177 us; 8 sequences of 600-3000 tokens at G = 2: 22.8 -> 20.5 us per layer.  128
// sequences of 1024-32768 tokens at G = 4 take what a streaming read takes (1.27 ms, 7.0 TB/s)
// with either.
//
// K and V rows go from memory into the wave's own LDS tiles (32 tokens x 256 bytes, two of
// each) with direct-to-LDS buffer loads: no register holds them, no barrier is needed, and
// a tile is refilled as soon as its step has read it, two steps ahead, so 24-32 KiB per
// wave are in flight all the time.  Where sequences are short, their starts and ends take
// longer than their steps: a wave has one SIMD to itself and nothing to hide the vector work
// behind.  So a sequence's lengths, block id and slot come from lanes (SeqWindow), its q and new
// token with its first tiles, q and the new k share their norms and rotations, and the waits
// count what is in flight (see the loop): 4096 sequences of 1-60 tokens, one-launch step,
// G = 2 223 -> 152 us, G = 1 219 -> 136; 1024 of 10-100 70.7 -> 63.2 and 68.2 -> 55.9; one of
// 611 tokens, 28 layers 307 -> 288.  The rows are read with the nontemporal hint.  Those past
// the context are clamped onto its last token, so no branch guards a load; the softmax masks
// them, and their V is cleared (0 times an infinity is a NaN).
//
// Layouts (lane l: n = l % 16, q4 = l / 16).  S = K Q^T: A is the K tile (row n of 16
// tokens, dims 8 q4 + e of each 32), B is q (column n); the lane gets the scores of tokens
// 4 q4 + j, j = 0..3, of both 16-token halves for its column.  O^T += V^T P^T: A is V^T by
// the LDS transpose load, B is P straight from the score registers (the k index of
// (q4, e) is token 4 q4 + e of the first half for e < 4, of the second for e >= 4), and the
// lane gets dims 16 mt + 4 q4 + j of its column.
//
// P stays exact to fp32: the weight is split into bf16 parts p = p0 + p1 + p2 (8 bits of
// mantissa each), and the 16 columns hold the parts of the G heads side by side (column n:
// part n / G of head n % G; q is repeated, so every column forms its own part from its own
// scores).  Three parts fit for G <= 5; G = 8 holds two and adds the third with a second
// product (8 more instructions).  The parts of a head are summed in fp32 when the state is written.  Tile rows are
// swizzled by 16-byte chunks, K by row & 15 and V by 2 (row & 7), so neither the 16-byte
// reads nor the transpose reads share a bank.  Softmax: online, base 2, scale*log2(e)
// folded into the scores, one running max per column (over all row groups) and a running sum
// per column and row group.
//
// Output: where a wave's range ends or a sequence ends its state is written; a sequence
// covered by one range gives bf16 directly, otherwise each range writes (max, sum,
// unnormalised acc) in fp32 to the workspace and decode_merge_kernel combines them with the
// same online-softmax rule.  Partial traffic is about 2 states per group per sequence
// boundary: well under 1% of the KV bytes.
//
// Partial slots: the state that range r writes for sequence b goes to slot r + b.
// Sequence b's ranges are first_b .. last_b (first_b = cum_b / spr), and the next
// sequence with steps starts at a range >= last_b, so slots are unique, and one
// sequence's slots are consecutive.  A launch with R ranges over B sequences uses at
// most R + B slots of num_q_heads states each, whatever the context lengths.
#include <math.h>

#include <algorithm>
#include <atomic>
#include <type_traits>

#include "common.h"

namespace kvp {

constexpr int kDecodeHeadDim = 128;
constexpr int kDecodeWaves = 4;  // kv heads per workgroup
constexpr int kDecodeThreads = 64 * kDecodeWaves;
constexpr int kStep = 32;               // tokens per step
constexpr int kTileBytes = kStep * 256;  // one K or V tile
// The workspace formula counts the ranges a launch may have: one per 128 tokens of its block
// tables.  The kernel cuts the actual steps into that many ranges, so a table wider than its
// contexts gives shorter ones, down to one step.  A small batch wants the shortest, because
// its waves run their steps one after the other while most CUs idle: per call, one sequence
// of 611 tokens 15.0 us with 128-token ranges, 12.2 us with one-step ranges; 37 sequences of
// 17-118 tokens 20.9 and 12.5 us.  A large batch is split by the grid and sees no difference.
constexpr int kWorkspaceRangeTokens = 128;
// Sequences per launch: as many as the step prefix has LDS for beside the tiles of `ahead` steps
// and the sequences' inputs.  More run as consecutive launches.
constexpr int seqs_per_launch(int g, bool fused, int ahead) {
  if (ahead == 1) return 2048;
  return fused ? (g <= 2 ? 4096 : g <= 5 ? 2048 : 1024) : (g <= 5 ? 4096 : 2048);
}
// Steps whose tiles a wave has in flight ahead of the one it computes: two, with one workgroup on
// a CU; or one, with two workgroups, whose waves compute while the others wait, for batches of
// many short sequences at G = 1, where a sequence's start and end take longer than its steps.
// 8q/8kv, one-launch step, two steps ahead against one: 1024 sequences of 1-32 tokens 37.8 and
// 30.3 us, 1024 of 10-100 59.7 and 55.9, 512 of 100-200 64.0 and 63.1, 1024 of 200-400 214.6 and
// 215.7; 32 of 200-800 23.4 and 24.4, one of 20000 29.5 and 33.0, 128 of 1024-16384 667 and 673.
constexpr int kManySeqs = 512;
static int steps_ahead(int g, int num_seqs) { return g == 1 && num_seqs >= kManySeqs ? 1 : 2; }
constexpr int kHeaderSeqs = 4096;     // sequences the workspace formula counts at most
constexpr int64_t kMaxDmaRow = 1 << 24;  // row stride (elements) up to which 32 rows are addressed in 32 bits
constexpr int kHeaderInts = 16;          // workspace header before the prefix table
// Upper bound of the persistent grid; the cap makes the workspace bound independent of the
// device.
constexpr int kMaxDecodeGrid = 1024;

// n / d for 0 <= n < 2^31 by a multiplication (the compiler's division is some 30
// instructions, most of them executed once per launch from a cold instruction cache).
// With l = ceil(log2 d) and mul = ceil(2^(31 + l) / d), n * mul / 2^(31 + l) exceeds n / d
// by less than n / 2^(31 + l) <= 1 / d for n < 2^31, so the floor is exact.
struct Divisor {
  uint32_t mul, shift;  // shift = l - 1 beyond the high word; d = 1: mul = 0
};
static Divisor divisor(uint32_t d) {
  if (d <= 1) return Divisor{0, 0};
  uint32_t l = 0;
  while ((1ull << l) < d) ++l;
  return Divisor{static_cast<uint32_t>(((1ull << (31 + l)) + d - 1) / d), l - 1};
}
__device__ __forceinline__ int div_by(int n, const Divisor& d) {
  return d.mul ? static_cast<int>(__umulhi(static_cast<uint32_t>(n), d.mul) >> d.shift) : n;
}

struct DecodeParams {
  const uint16_t* q;
  int64_t q_seq_stride, q_head_stride;
  const uint16_t* k_cache;
  const uint16_t* v_cache;
  int64_t blk_stride, slot_stride, head_stride;
  int32_t num_cache_blocks;
  const int32_t* block_tables;
  int64_t bt_stride;
  const int32_t* context_lens;
  int32_t num_seqs;  // <= seqs_per_launch
  int32_t num_q_heads;
  int32_t num_kv_heads;
  int32_t block_size;
  int32_t max_blocks;
  float scale_log2;  // softmax_scale * log2(e)
  uint16_t* out;
  int64_t o_seq_stride, o_head_stride;
  int32_t* header;  // [0] steps per range, [kHeaderInts ..] step prefix sums (B + 1)
  float* part_o;    // [slot][num_q_heads][128], slot = range + sequence (ranges + B slots)
  float* part_ml;   // [slot][num_q_heads][2] = (max, sum)
  // Fused q/k norm + RoPE + append (FUSED kernels): row b of qkv holds the token's
  // num_q_heads q heads, then num_kv_heads k heads, then num_kv_heads v heads.
  // The token's position is context_lens[b] - 1.
  const uint16_t* qkv;
  int64_t qkv_stride;
  const float* cos_sin;  // [max_position][128] fp32: cos of the 64 frequencies, then sin
  int32_t max_position;
  const uint16_t* q_weight;
  const uint16_t* k_weight;
  float eps;
  const int32_t* slot_mapping;
  int64_t num_cache_slots;
  Divisor div_block, div_ranges;  // by block_size and by the launch's range count
  // 32 token rows / the q heads of one kv head fit 32-bit byte offsets
  bool rows_by_dma, q_by_dma;
};

__device__ __forceinline__ uint4 load16(const uint16_t* ptr) {
  return *reinterpret_cast<const uint4*>(ptr);
}

// A wave-uniform read of read-only metadata (context lengths, block tables) through the
// constant address space, so it compiles to a scalar load.  Scalar loads are counted
// apart from the vector loads of the K/V stream: waiting for a block id does not wait
// for the KV loads in flight (as a vector load's wait would, vector loads complete in
// order), and a block id loaded one block ahead is waited for only where it is used.
__device__ __forceinline__ int load_uniform(const int32_t* base, int64_t idx) {
  return ((const __attribute__((address_space(4))) int32_t*)(base))[idx];
}

// Steps of a sequence; 0 for empty or impossible contexts (written separately).
__device__ __forceinline__ int seq_steps(int ctx, const DecodeParams& p) {
  if (ctx <= 0 || ctx > p.max_blocks * p.block_size) return 0;
  return (ctx + kStep - 1) / kStep;
}

// Rows with nothing to attend (ctx 0: graph padding) read as zeros; impossible lengths read
// as NaN.  Neither has steps.
__device__ __forceinline__ void fill_row(const DecodeParams& p, int b, int ctx) {
  const u32 w = ctx <= 0 ? 0u : 0x7fc07fc0u;
#pragma unroll 1
  for (int o = 0; o < p.num_q_heads * kDecodeHeadDim; o += 8)
    *reinterpret_cast<uint4*>(p.out + b * p.o_seq_stride + (o / kDecodeHeadDim) * p.o_head_stride +
                              o % kDecodeHeadDim) = make_uint4(w, w, w, w);
}

// Keeps a load whose value is not used.
__device__ __forceinline__ void keep(int x) { asm volatile("" ::"v"(x)); }

// s_cum[b] = steps of sequences 0..b-1 (b = 0..num_seqs), built by the whole workgroup: each
// thread sums a contiguous run of sequences, then the 256 run totals are scanned with DPP
// within each wave and the 4 wave totals through LDS.
__device__ __forceinline__ void build_step_prefix(const DecodeParams& p, int* s_cum, int* s_part) {
  const int tid = threadIdx.x;
  const int B = p.num_seqs;
  const int per = (B + kDecodeThreads - 1) / kDecodeThreads;
  const int j0 = tid * per, j1 = min(j0 + per, B);
  int warm = 0;
  const int wg = blockIdx.y * gridDim.x + blockIdx.x, wgs = gridDim.x * gridDim.y;
  int local = 0;
#pragma unroll 1
  for (int b0 = j0; b0 < j1; b0 += 4) {  // four lengths in flight
    int ctx[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) ctx[i] = p.context_lens[min(b0 + i, j1 - 1)];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int b = b0 + i;
      if (b >= j1) break;
      const int steps = seq_steps(ctx[i], p);
      s_cum[b] = steps;
      local += steps;
      if (steps == 0 && b % wgs == wg) fill_row(p, b, ctx[i]);
      // the first entry of a sequence's block-table row, so that the table read behind the
      // prefix finds its line in L2; no entry is read of a row without steps
      if (steps > 0 && per == 1) warm = p.block_tables[b * p.bt_stride];
    }
  }
  const int lane = tid & 63, wave = tid >> 6;
  const int incl = wave_incl_scan(local);
  if (lane == 63) s_part[wave] = incl;
  __syncthreads();
  int before = 0;
#pragma unroll
  for (int w = 0; w < kDecodeWaves - 1; ++w)
    if (w < wave) before += s_part[w];
  int run = before + incl - local;
#pragma unroll 1
  for (int b = j0; b < j1; ++b) {
    const int steps = s_cum[b];
    s_cum[b] = run;
    run += steps;
  }
  if (tid == kDecodeThreads - 1) s_cum[B] = before + incl;
  keep(warm);
  __syncthreads();
}

// Ranges [cum_b / spr, (cum_b1 - 1) / spr] touch sequence b's steps [cum_b, cum_b1).
__device__ __forceinline__ int num_parts(int cum_b, int cum_b1, int spr) {
  return (cum_b1 - 1) / spr - cum_b / spr + 1;
}

// Per-wave cursor over the steps of one range.
struct StepCursor {
  int b;        // sequence
  int j;        // step within the sequence
  int nsteps;   // steps of sequence b
  int ctx;      // context length of sequence b
  int slot;     // FUSED: where its new token goes
  int lblk;     // logical block whose id is cached in blk (-1: none)
  int blk;      // physical block id of lblk
  int pf_blk;   // id of block lblk + 1, loaded one block ahead (-1: not loaded)
  int buf;      // which of the wave's input regions holds the sequence's q
  int bad;      // a needed block id was out of range (an int: the struct copies stay in registers)
  int mark;     // vector memory operations issued up to the step's K tile (its V tile follows)
};

// 64 consecutive sequences' metadata, one per lane, so that moving to the next sequence waits for
// no memory and no LDS: lane i holds sequence base + i.
struct SeqWindow {
  int base;
  uint64_t live;  // the lanes with steps
  int ctx, blk, slot;  // length, first block id (0 without steps), FUSED: the new token's slot
};
template <bool FUSED>
__device__ __forceinline__ void fill_window(const DecodeParams& p, const int* s_cum, int base, int lane, SeqWindow& w) {
  const int b = min(base + lane, p.num_seqs - 1);
  const bool has = base + lane < p.num_seqs && s_cum[b + 1] > s_cum[b];
  w.base = base;
  w.live = __ballot(has);
  w.ctx = p.context_lens[b];
  w.slot = FUSED ? p.slot_mapping[b] : 0;
  w.blk = 0;
  if (has) w.blk = p.block_tables[b * p.bt_stride];
  // waited for here, so that no later read waits for what has been issued since
  asm volatile("" : "+v"(w.ctx), "+v"(w.slot), "+v"(w.blk));
}

// Puts the cursor into logical block lblk, whose id is blk, and loads the next one's ahead.
__device__ __forceinline__ void cursor_enter_block(const DecodeParams& p, StepCursor& cur, int lblk, int blk) {
  const int bad = blk < 0 || blk >= p.num_cache_blocks;
  cur.bad |= bad;
  cur.blk = bad ? 0 : blk;
  cur.lblk = lblk;
  cur.pf_blk = (lblk + 1) * p.block_size < cur.ctx ? load_uniform(p.block_tables + cur.b * p.bt_stride, lblk + 1) : -1;
}

// The cursor of the first step of sequence base + i.
__device__ __forceinline__ void cursor_start_seq(const DecodeParams& p, StepCursor& cur, const SeqWindow& w, int i,
                                                 int buf) {
  cur.buf = buf;
  cur.b = w.base + i;
  cur.j = 0;
  cur.ctx = __builtin_amdgcn_readlane(w.ctx, i);
  cur.slot = __builtin_amdgcn_readlane(w.slot, i);
  cur.nsteps = (cur.ctx + kStep - 1) / kStep;
  cur.bad = 0;
  cursor_enter_block(p, cur, 0, __builtin_amdgcn_readlane(w.blk, i));
}

// Element offset of the cursor's step in the caches, and the number of valid tokens of the
// step.  On entering a block it takes the id prefetched one block earlier (or loads it) and
// prefetches the next block's id, so the scalar load is off the critical path.
__device__ __forceinline__ int64_t step_base(const DecodeParams& p, StepCursor& cur, int64_t head_off, int& nvalid) {
  const int t0 = cur.j * kStep;
  const int lblk = div_by(t0, p.div_block);
  if (lblk != cur.lblk)
    cursor_enter_block(p, cur, lblk, lblk == cur.lblk + 1 && cur.pf_blk != -1
                                         ? cur.pf_blk
                                         : load_uniform(p.block_tables + cur.b * p.bt_stride, lblk));
  nvalid = min(kStep, cur.ctx - t0);
  return static_cast<int64_t>(cur.blk) * p.blk_stride +
         static_cast<int64_t>(t0 - lblk * p.block_size) * p.slot_stride + head_off;
}

// ---- fused q/k norm + RoPE + append (FUSED kernels)
//
// The inputs of a sequence -- its cos/sin row, raw q heads, and its new token's raw k and v heads
// -- reach one of two per-wave LDS regions with direct-to-LDS buffer loads, issued with the tiles
// of the sequence's first step, two steps ahead, so the wave never waits on a dependent load
// chain at a sequence boundary and no VGPR holds them meanwhile.  The token's position is
// context_lens[b] - 1.
constexpr int kFzRow = 512;  // bytes: one cos/sin row, 128 fp32
__device__ __forceinline__ BufferRsrc cos_sin_rsrc(const DecodeParams& p) {
  return buffer_rsrc(p.cos_sin, static_cast<uint32_t>(p.max_position) * kFzRow);
}
__device__ __forceinline__ BufferRsrc qkv_rsrc(const DecodeParams& p) {
  return buffer_rsrc(p.qkv, static_cast<uint32_t>(p.num_seqs * p.qkv_stride * 2));
}
__device__ __forceinline__ int fz_row_bytes(const DecodeParams& p, int ctx) {
  const int pos = ctx - 1;
  return (pos >= 0 && pos < p.max_position ? pos : 0) * kFzRow;
}

// Weights: lanes 0-15 the q norm weight, 16-31 the k norm weight.
__device__ __forceinline__ void fz_issue_weights(const DecodeParams& p, int lane, char* region) {
  if (lane < 16) lds_dma16(buffer_rsrc(p.q_weight, 256), 16 * lane, region);
  else if (lane < 32) lds_dma16(buffer_rsrc(p.k_weight, 256), 16 * (lane - 16), region);
}

// A sequence's region: the cos/sin row (bytes 0-511), the G raw q heads of kv head kvh, the raw k
// head, the raw v head.  Instruction i of the qkv part fills bytes 1024 i .. + 1023 of the region.
template <int G>
struct FzRegion {
  static constexpr int kNew = kFzRow + 256 * G;  // where the new token's k and v start
  static constexpr int kBytes = kNew + 512;
  static constexpr int kLoads = (kBytes + 1023) / 1024;
  static constexpr int kOps = 1 + kLoads;  // vector memory operations
};
// Byte offset in a qkv row of what the lane loads in instruction i.
template <int G>
__device__ __forceinline__ int fz_row_offset(const DecodeParams& p, int kvh, int lane, int i) {
  const int at = 1024 * i + 16 * lane;
  const int head = at < FzRegion<G>::kNew         ? kvh * G + (at - kFzRow) / 256
                   : at < FzRegion<G>::kNew + 256 ? p.num_q_heads + kvh
                                                  : p.num_q_heads + p.num_kv_heads + kvh;
  return head * 256 + at % 256;
}
template <int G>
__device__ __forceinline__ void fz_issue(const DecodeParams& p, int b, int ctx, const int (&row_at)[FzRegion<G>::kLoads],
                                         int lane, char* region) {
  typedef __attribute__((address_space(3))) void* Lds;
  if (lane < kFzRow / 16) raw_buffer_load_lds(cos_sin_rsrc(p), (Lds)region, 16, 16 * lane, fz_row_bytes(p, ctx), 0, 0);
  const int row = b * static_cast<int>(p.qkv_stride) * 2;
#pragma unroll
  for (int i = 0; i < FzRegion<G>::kLoads; ++i) {
    const int at = 1024 * i + 16 * lane;
    if (at >= kFzRow && at < FzRegion<G>::kBytes)
      raw_buffer_load_lds(qkv_rsrc(p), (Lds)(region + 1024 * i), 16, row_at[i], row, 0, 0);
  }
}

typedef __bf16 mfma_bf16x8_t __attribute__((ext_vector_type(8)));
typedef float mfma_f32x4_t __attribute__((ext_vector_type(4)));

__device__ __forceinline__ mfma_f32x4_t mfma16(u32x4_t a, u32x4_t b, mfma_f32x4_t c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(mfma_bf16x8_t, a),
                                                 __builtin_bit_cast(mfma_bf16x8_t, b), c, 0, 0, 0);
}
// All LDS accesses of the wave are done: what they read may be overwritten.
__device__ __forceinline__ void wait_lds() { asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); }

// Tile accesses are written out, each block with its own wait: the compiler cannot tell a
// tile from the one being filled and would wait for every load in flight.
__device__ __forceinline__ u32 lds_addr(const void* p) {
  return static_cast<u32>(reinterpret_cast<uintptr_t>((const __attribute__((address_space(3))) void*)(p)));
}
// The 16 bytes at a[i] and at a[i] + 4096 (the tile's two 16-token halves), i = 0..3.
__device__ __forceinline__ void read_k_tile(const u32 (&a)[4], u32x4_t (&k)[8]) {
  asm volatile(
      "ds_read_b128 %0, %8\n\tds_read_b128 %1, %8 offset:4096\n\t"
      "ds_read_b128 %2, %9\n\tds_read_b128 %3, %9 offset:4096\n\t"
      "ds_read_b128 %4, %10\n\tds_read_b128 %5, %10 offset:4096\n\t"
      "ds_read_b128 %6, %11\n\tds_read_b128 %7, %11 offset:4096\n\t"
      "s_waitcnt lgkmcnt(0)"
      : "=&v"(k[0]), "=&v"(k[1]), "=&v"(k[2]), "=&v"(k[3]), "=&v"(k[4]), "=&v"(k[5]), "=&v"(k[6]), "=&v"(k[7])
      : "v"(a[0]), "v"(a[1]), "v"(a[2]), "v"(a[3])
      : "memory");
}
typedef u32 u32x2_t __attribute__((ext_vector_type(2)));
// Transposed 8-byte reads at a[i] (first half) and a[i] + 4096 (second half), i = 0..7.
__device__ __forceinline__ void read_v_tile(const u32 (&a)[8], u32x2_t (&lo)[8], u32x2_t (&hi)[8]) {
  asm volatile(
      "ds_read_b64_tr_b16 %0, %16\n\tds_read_b64_tr_b16 %8, %16 offset:4096\n\t"
      "ds_read_b64_tr_b16 %1, %17\n\tds_read_b64_tr_b16 %9, %17 offset:4096\n\t"
      "ds_read_b64_tr_b16 %2, %18\n\tds_read_b64_tr_b16 %10, %18 offset:4096\n\t"
      "ds_read_b64_tr_b16 %3, %19\n\tds_read_b64_tr_b16 %11, %19 offset:4096\n\t"
      "ds_read_b64_tr_b16 %4, %20\n\tds_read_b64_tr_b16 %12, %20 offset:4096\n\t"
      "ds_read_b64_tr_b16 %5, %21\n\tds_read_b64_tr_b16 %13, %21 offset:4096\n\t"
      "ds_read_b64_tr_b16 %6, %22\n\tds_read_b64_tr_b16 %14, %22 offset:4096\n\t"
      "ds_read_b64_tr_b16 %7, %23\n\tds_read_b64_tr_b16 %15, %23 offset:4096\n\t"
      "s_waitcnt lgkmcnt(0)"
      : "=&v"(lo[0]), "=&v"(lo[1]), "=&v"(lo[2]), "=&v"(lo[3]), "=&v"(lo[4]), "=&v"(lo[5]), "=&v"(lo[6]),
        "=&v"(lo[7]), "=&v"(hi[0]), "=&v"(hi[1]), "=&v"(hi[2]), "=&v"(hi[3]), "=&v"(hi[4]), "=&v"(hi[5]),
        "=&v"(hi[6]), "=&v"(hi[7])
      : "v"(a[0]), "v"(a[1]), "v"(a[2]), "v"(a[3]), "v"(a[4]), "v"(a[5]), "v"(a[6]), "v"(a[7])
      : "memory");
}
// N (1 or 2) heads' chunks normalised and rotated: chunk c of the head at x_at[i], by the norm
// weights at w_at[i] and the cos/sin row at table_at.
template <int N>
__device__ __forceinline__ void norm_rope_chunks(const u32 (&w_at)[N], u32 table_at, const u32 (&x_at)[N], int c,
                                                 bool pos_ok, float eps, uint4 (&out)[N]) {
  u32x4_t hw[2], hx[2], hc[2], hs[2];
  if constexpr (N == 1) {
    asm volatile(
        "ds_read_b128 %0, %6\n\tds_read_b128 %1, %8\n\tds_read_b128 %2, %7\n\tds_read_b128 %3, %7 offset:16\n\t"
        "ds_read_b128 %4, %7 offset:256\n\tds_read_b128 %5, %7 offset:272\n\ts_waitcnt lgkmcnt(0)"
        : "=&v"(hw[0]), "=&v"(hx[0]), "=&v"(hc[0]), "=&v"(hc[1]), "=&v"(hs[0]), "=&v"(hs[1])
        : "v"(w_at[0]), "v"(table_at), "v"(x_at[0])
        : "memory");
  } else {
    asm volatile(
        "ds_read_b128 %0, %8\n\tds_read_b128 %1, %9\n\tds_read_b128 %2, %11\n\tds_read_b128 %3, %12\n\t"
        "ds_read_b128 %4, %10\n\tds_read_b128 %5, %10 offset:16\n\tds_read_b128 %6, %10 offset:256\n\t"
        "ds_read_b128 %7, %10 offset:272\n\ts_waitcnt lgkmcnt(0)"
        : "=&v"(hw[0]), "=&v"(hw[1]), "=&v"(hx[0]), "=&v"(hx[1]), "=&v"(hc[0]), "=&v"(hc[1]), "=&v"(hs[0]), "=&v"(hs[1])
        : "v"(w_at[0]), "v"(w_at[1]), "v"(table_at), "v"(x_at[0]), "v"(x_at[1])
        : "memory");
  }
  float cs[8], sn[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    cs[e] = __uint_as_float(hc[e >> 2][e & 3]);
    sn[e] = __uint_as_float(hs[e >> 2][e & 3]);
  }
#pragma unroll
  for (int i = 0; i < N; ++i) {
    float w[8], x[8];
    unpack8(__builtin_bit_cast(uint4, hw[i]), w);
    unpack8(__builtin_bit_cast(uint4, hx[i]), x);
    norm_rope_head(x, w, cs, sn, c < 8, pos_ok, eps);
    out[i] = pack8(x);
  }
}
// Two 16-byte chunks.
__device__ __forceinline__ void read_pair(u32 a, u32 b, u32x4_t& x, u32x4_t& y) {
  asm volatile("ds_read_b128 %0, %2\n\tds_read_b128 %1, %3\n\ts_waitcnt lgkmcnt(0)"
               : "=&v"(x), "=&v"(y)
               : "v"(a), "v"(b)
               : "memory");
}
// q of one column in the B layout: 16 bytes at a, a + 64, a + 128, a + 192.
__device__ __forceinline__ void read_q(u32 a, u32x4_t (&q)[4]) {
  asm volatile(
      "ds_read_b128 %0, %4\n\tds_read_b128 %1, %4 offset:64\n\t"
      "ds_read_b128 %2, %4 offset:128\n\tds_read_b128 %3, %4 offset:192\n\ts_waitcnt lgkmcnt(0)"
      : "=&v"(q[0]), "=&v"(q[1]), "=&v"(q[2]), "=&v"(q[3])
      : "v"(a)
      : "memory");
}
__device__ __forceinline__ void write_tile16(u32 addr, uint4 v) {
  asm volatile("ds_write_b128 %0, %1" ::"v"(addr), "v"(__builtin_bit_cast(u32x4_t, v)) : "memory");
}

// Stores that the waits count: one instruction each.
template <int OFFSET>
__device__ __forceinline__ void store8(void* ptr, u32x2_t v) {
  asm volatile("global_store_dwordx2 %0, %1, off offset:%2" ::"v"(ptr), "v"(v), "n"(OFFSET) : "memory");
}
template <int OFFSET>
__device__ __forceinline__ void store16(void* ptr, u32x4_t v) {
  asm volatile("global_store_dwordx4 %0, %1, off offset:%2" ::"v"(ptr), "v"(v), "n"(OFFSET) : "memory");
}

// Waits until at most `most` vector memory operations of the wave are in flight (uniform; rounded
// down to a multiple of 8).
__device__ __forceinline__ void wait_upto(int most) {
  if (most >= 24) {
    if (most >= 40) wait_vmem<40>();
    else if (most >= 32) wait_vmem<32>();
    else wait_vmem<24>();
  } else if (most >= 16) {
    wait_vmem<16>();
  } else if (most >= 8) {
    wait_vmem<8>();
  } else {
    wait_vmem<0>();
  }
}

// x of the lane N places up in the 16-lane row (0 past its end).
template <int N>
__device__ __forceinline__ float row_up(float x) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), 0x100 + N, 0xf, 0xf, false));
}

// The lane's parts of the tile fills.  Instruction i fills rows 4 i .. 4 i + 3 of a tile:
// lane l writes row r = 4 i + l / 16 at physical chunk l % 16, which holds logical chunk
// (l % 16) ^ (r & 15) of K and (l % 16) ^ 2 (r & 7) of V.
struct TileLane {
  int r, c;        // l / 16, l % 16
  int row_off;     // byte offset of row r
  int k_chunk[4];  // 16 (c ^ (4 i + r)), i = 0..3
  int v_chunk[2];  // 16 (c ^ 2 ((4 i + r) & 7)), i = 0..1
};
// Rows of a tile from element `base` of the cache: row r is token r, rows past the last one
// repeat it, so every load is in bounds.  Strides whose 32 rows do not fit 32-bit byte
// offsets go through registers.
template <bool V>
__device__ __forceinline__ void issue_tile(const DecodeParams& p, const TileLane& ln, int64_t base, int rows,
                                                char* tile) {
  const uint16_t* src = (V ? p.v_cache : p.k_cache) + base;
  if (p.rows_by_dma) {  // uniform
    const int row_bytes = static_cast<int>(p.slot_stride) * 2;
    const BufferRsrc rsrc = buffer_rsrc(src, static_cast<uint32_t>((kStep - 1) * row_bytes + 256));
    const int last = (rows - 1) * row_bytes;
#pragma unroll
    for (int i = 0; i < 8; ++i)  // nontemporal: every row is read once
      raw_buffer_load_lds(rsrc, (__attribute__((address_space(3))) void*)(tile + 1024 * i), 16,
                          min(ln.row_off + 4 * i * row_bytes, last) + (V ? ln.v_chunk[i & 1] : ln.k_chunk[i & 3]), 0,
                          0, 2);
  } else {
#pragma unroll 1
    for (int row = ln.r; row < kStep; row += 4) {
      const int chunk = 16 * (ln.c ^ (V ? 2 * (row & 7) : row & 15));
      const char* at = reinterpret_cast<const char*>(src + min(row, rows - 1) * p.slot_stride) + chunk;
      write_tile16(lds_addr(tile) + 256 * row + 16 * ln.c, load16_nt(at));
    }
  }
}

// f(0) .. f(7) with constant arguments.
template <typename F>
__device__ __forceinline__ void each8(F f) {
  f(std::integral_constant<int, 0>{});
  f(std::integral_constant<int, 1>{});
  f(std::integral_constant<int, 2>{});
  f(std::integral_constant<int, 3>{});
  f(std::integral_constant<int, 4>{});
  f(std::integral_constant<int, 5>{});
  f(std::integral_constant<int, 6>{});
  f(std::integral_constant<int, 7>{});
}

template <int G>
struct State {
  float m, l;
  mfma_f32x4_t acc[8];               // column n's part; dims 16 mt + 4 q4 + j
  mfma_f32x4_t acc2[G > 5 ? 8 : 1];  // G = 8: the third part, in columns 8..15
};
template <int G>
__device__ __forceinline__ void reset_state(State<G>& st) {
  st.m = kMaxFloor;
  st.l = 0.f;
#pragma unroll
  for (int mt = 0; mt < 8; ++mt) {
    st.acc[mt] = mfma_f32x4_t{0.f, 0.f, 0.f, 0.f};
    if (G > 5) st.acc2[mt] = mfma_f32x4_t{0.f, 0.f, 0.f, 0.f};
  }
}

// The state of (b, kvh) for this range: the parts of each head summed, then the bf16
// output when one range covers the sequence, otherwise an fp32 partial.
// Returns its vector memory operations.
template <int G>
__device__ __forceinline__ int emit_state(const DecodeParams& p, int b, int kvh, int slot, bool single, bool bad,
                                          int n, int q4, const State<G>& st) {
  float l = xor32_sum(xor16_sum(st.l));
  if (bad) l = NAN;
  float o[8][4], odd = 0.f;  // odd: NaN once a value is not finite
#pragma unroll
  for (int mt = 0; mt < 8; ++mt) {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const float a = st.acc[mt][j];
      o[mt][j] = a + row_up<G>(a);
      if (G <= 5) o[mt][j] += row_up<2 * (G <= 5 ? G : 1)>(a);
      else o[mt][j] += row_up<G>(st.acc2[mt][j]);
      odd = fmaf(o[mt][j], 0.f, odd);
    }
  }
  if (__any(odd != odd)) {  // an infinite value in V: the first part has the result, the others inf - inf
#pragma unroll
    for (int mt = 0; mt < 8; ++mt)
#pragma unroll
      for (int j = 0; j < 4; ++j) o[mt][j] = __builtin_isfinite(st.acc[mt][j]) ? o[mt][j] : st.acc[mt][j];
  }
  const int h = kvh * G + n;
  if (single) {
    const float inv = 1.f / l;
    uint16_t* out = p.out + b * p.o_seq_stride + h * p.o_head_stride + 4 * q4;
    auto row = [&](auto mt_c) {
      constexpr int mt = decltype(mt_c)::value;
      store8<32 * mt>(out, u32x2_t{pack_bf16x2(o[mt][0] * inv, o[mt][1] * inv),
                                   pack_bf16x2(o[mt][2] * inv, o[mt][3] * inv)});
    };
    if (n < G) each8(row);
    return 8;
  }
  const int64_t at = static_cast<int64_t>(slot) * p.num_q_heads + h;
  float* part = p.part_o + at * kDecodeHeadDim + 4 * q4;
  auto row = [&](auto mt_c) {
    constexpr int mt = decltype(mt_c)::value;
    store16<64 * mt>(part, u32x4_t{__float_as_uint(o[mt][0]), __float_as_uint(o[mt][1]), __float_as_uint(o[mt][2]),
                                   __float_as_uint(o[mt][3])});
  };
  if (n < G) {
    each8(row);
    if (q4 == 0) store8<0>(p.part_ml + at * 2, u32x2_t{__float_as_uint(st.m), __float_as_uint(l)});
  }
  return 9;
}

template <int G, bool FUSED, int A>
__global__ __launch_bounds__(kDecodeThreads)
void paged_decode_kernel(const DecodeParams p) {
  // per wave: K and V tiles of the steps in flight, and the inputs of as many sequences (FUSED:
  // FzRegion, else the G q heads); FUSED: norm weights, which every wave loads (the same bytes)
  __shared__ __attribute__((aligned(16))) char s_tile[kDecodeWaves][A][2 * kTileBytes];
  constexpr int kQRow = FUSED ? kFzRow : 0;
  constexpr int kQBytes = FUSED ? FzRegion<G>::kBytes : 256 * G;
  __shared__ __attribute__((aligned(16))) char s_q[kDecodeWaves][A][kQBytes];
  __shared__ __attribute__((aligned(16))) char s_fw[FUSED ? 512 : 16];
  __shared__ int s_cum[seqs_per_launch(G, FUSED, A) + 1];  // steps of sequences 0 .. b - 1
  __shared__ int s_part[kDecodeWaves];

  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lane = tid & 63;
  const int n = lane & 15, q4 = lane >> 4;

  build_step_prefix(p, s_cum, s_part);
  const int B = p.num_seqs;
  const int total_steps = __builtin_amdgcn_readfirstlane(s_cum[B]);  // uniform, and a scalar
  const int spr = max(1, div_by(total_steps + static_cast<int>(gridDim.y) - 1, p.div_ranges));
  if (blockIdx.x == 0 && blockIdx.y == 0) {  // for the merge kernel
    if (tid == 0) p.header[0] = spr;
    for (int b = tid; b <= B; b += kDecodeThreads) p.header[kHeaderInts + b] = s_cum[b];
  }
  const int range = blockIdx.y;  // workgroup x of a range: kv heads 4 x .. 4 x + 3
  const int kvh = blockIdx.x * kDecodeWaves + wave;
  const int S0 = range * spr;
  const int S1 = min(total_steps, S0 + spr);
  if (kvh >= p.num_kv_heads || S0 >= S1) return;  // no barrier follows

  // Sequence holding step S0: s_cum[b] <= S0 < s_cum[b + 1].
  int lo = 0, hi = B;
  while (hi - lo > 1) {
    const int mid = (lo + hi) >> 1;
    if (s_cum[mid] <= S0) lo = mid;
    else hi = mid;
  }
  lo = __builtin_amdgcn_readfirstlane(lo);
  const int64_t head_off = static_cast<int64_t>(kvh) * p.head_stride;
  const int hg = n % G;     // this column's head and the part of P it holds
  const int part = n / G;

  TileLane ln;
  ln.r = q4;
  ln.c = n;
  ln.row_off = q4 * static_cast<int>(p.rows_by_dma ? p.slot_stride : 0) * 2;
#pragma unroll
  for (int i = 0; i < 4; ++i) ln.k_chunk[i] = 16 * (n ^ (4 * i + q4));
#pragma unroll
  for (int i = 0; i < 2; ++i) ln.v_chunk[i] = 16 * (n ^ (2 * ((4 * i + q4) & 7)));
  // LDS addresses of the lane's operands in a tile at address 0 (see the swizzles)
  u32 ka[4], va[8];
#pragma unroll
  for (int kk = 0; kk < 4; ++kk) ka[kk] = 256 * n + 16 * ((4 * kk + q4) ^ n);
  const int vrow = 4 * q4 + (n >> 2);
#pragma unroll
  for (int mt = 0; mt < 8; ++mt) va[mt] = kTileBytes + 256 * vrow + 8 * (n & 3) + 32 * (mt ^ (vrow & 7));

  // q of a sequence reaches the wave's region with the tiles of its first step, then the
  // B layout (column n is head hg, dims 32 kk + 8 q4 + e).  FUSED: the raw heads are normalised
  // and rotated in place first (row group r takes heads r, r + 4).  Returns the vector memory
  // operations that the waits may count.
  int row_at[FUSED ? FzRegion<G>::kLoads : 1] = {};
  if constexpr (FUSED) {
#pragma unroll
    for (int i = 0; i < FzRegion<G>::kLoads; ++i) row_at[i] = fz_row_offset<G>(p, kvh, lane, i);
  }
  auto issue_q = [&](const StepCursor& c) {
    char* region = s_q[wave][c.buf];
    if constexpr (FUSED) {
      fz_issue<G>(p, c.b, c.ctx, row_at, lane, region);
      return FzRegion<G>::kOps;
    } else {
      const uint16_t* src = p.q + c.b * p.q_seq_stride + static_cast<int64_t>(kvh) * G * p.q_head_stride;
#pragma unroll
      for (int u = 0; u < (G + 3) / 4; ++u) {
        const int g = q4 + 4 * u;
        if (p.q_by_dma) {  // uniform
          const int head_bytes = static_cast<int>(p.q_head_stride) * 2;
          const BufferRsrc rsrc = buffer_rsrc(src, static_cast<uint32_t>((G - 1) * head_bytes + 256));
          if (g < G) lds_dma16(rsrc, g * head_bytes + 16 * n, region + 1024 * u);
        } else if (g < G) {
          write_tile16(lds_addr(region) + 256 * g + 16 * n, load16(src + g * p.q_head_stride + 8 * n));
        }
      }
      return p.q_by_dma ? (G + 3) / 4 : 0;
    }
  };
  const u32 q_base = lds_addr(s_q[wave][0]), w_at = lds_addr(s_fw);
  // At a range's first step of a sequence.  `ends`: the sequence's last step is in the range.
  auto finish_q = [&](const StepCursor& c, bool ends, u32x4_t (&dst)[4]) {
    const u32 q_at = q_base + kQBytes * c.buf;
    if constexpr (FUSED) {  // four heads to a pass, two passes interleaved; head G is the new token's k
      const bool pos_ok = c.ctx - 1 >= 0 && c.ctx - 1 < p.max_position;
      auto passes = [&](auto n_c, int g0) {  // heads g0 + q4, and g0 + 4 + q4
        constexpr int N = decltype(n_c)::value;
        u32 x[N], w[N];
        uint4 y[N];
#pragma unroll
        for (int i = 0; i < N; ++i) {
          const int g = min(g0 + 4 * i + q4, G);
          x[i] = q_at + kQRow + 256 * g + 16 * n;
          w[i] = w_at + (g == G ? 256 : 0) + 16 * n;
        }
        norm_rope_chunks<N>(w, q_at + 32 * (n & 7), x, n, pos_ok, p.eps, y);
#pragma unroll
        for (int i = 0; i < N; ++i)
          if (g0 + 4 * i + q4 <= G) write_tile16(x[i], y[i]);
      };
      constexpr std::integral_constant<int, 1> one{};
      constexpr std::integral_constant<int, 2> two{};
      if (G < 4 || (G == 4 && !ends)) passes(one, 0);
      else passes(two, 0);
      if (G == 8 && ends) passes(one, 8);
    }
    read_q(q_at + kQRow + 256 * hg + 16 * q4, dst);
  };
  // FUSED: the new token of the sequence that ends at this step: k (normalised and rotated with
  // q) and v appended at the slot and put into the step's tiles, where the loads left them out;
  // the rows of V past it are cleared, so that no unwritten slot is multiplied (those of K give
  // scores that are masked).  Returns the vector memory operations.
  auto finish_new = [&](const StepCursor& c, int nv, u32 tile) {
    const u32 new_at = q_base + kQBytes * c.buf + kQRow + 256 * G + 16 * n;
    u32x4_t knew, vnew;
    read_pair(new_at, new_at + 256, knew, vnew);
    int ops = 0;
    if (c.slot >= 0 && c.slot < p.num_cache_slots) {  // uniform
      const int blk = div_by(c.slot, p.div_block), off = c.slot - blk * p.block_size;
      const int64_t at = static_cast<int64_t>(blk) * p.blk_stride + static_cast<int64_t>(off) * p.slot_stride +
                         head_off + 8 * n;
      if (q4 == 0) {
        store16<0>(const_cast<uint16_t*>(p.k_cache) + at, knew);
        store16<0>(const_cast<uint16_t*>(p.v_cache) + at, vnew);
      }
      ops = 2;
    }
    const int last = nv - 1;
    if (q4 == 0) write_tile16(tile + 256 * last + 16 * (n ^ (last & 15)), __builtin_bit_cast(uint4, knew));
    for (int row = (last & ~3) + q4; row < kStep; row += 4)
      if (row >= last)
        write_tile16(tile + kTileBytes + 256 * row + 16 * (n ^ (2 * (row & 7))),
                     row == last ? __builtin_bit_cast(uint4, vnew) : make_uint4(0, 0, 0, 0));
    wait_lds();
    return ops;
  };
  // The rows of V past a sequence's end repeat its last token (see issue_tile); their weights
  // are 0, but 0 times an infinity is not: they are cleared.  (finish_new clears its own.)
  auto clear_past = [&](int nv, u32 tile) {
#pragma unroll 1
    for (int row = (nv & ~3) + q4; row < kStep; row += 4)
      if (row >= nv) write_tile16(tile + kTileBytes + 256 * row + 16 * n, make_uint4(0, 0, 0, 0));
    wait_lds();
  };

  // The loop.  Iteration S computes step S and issues the tiles of step S + A, each as soon as its
  // tile has been read, with the inputs of the sequence before them if it starts one; the first A
  // iterations (S < S0) only issue.  c[i]: cursor of step S + i.  Vector memory operations
  // complete in issue order, so the waits count back from the operations issued so far to the
  // mark of what they need; an operation that is not counted only makes them stricter.
  StepCursor c[A + 1] = {};
  StepCursor &c0 = c[0], &cn = c[A];
  u32x4_t qv[4] = {};
  State<G> st;
  reset_state<G>(st);
  int issued = 0;
  const int tile_ops = p.rows_by_dma ? 8 : 0;
  if (FUSED) fz_issue_weights(p, lane, s_fw);
  // The first step, and, if the range goes on into other sequences, their window: all of it loaded
  // together.  (The first sequence from the window as well: one of 19008 tokens, a step or five to
  // a range, 25.9 -> 26.3 us per layer.)
  const int cum_lo = __builtin_amdgcn_readfirstlane(s_cum[lo]), cum_hi = __builtin_amdgcn_readfirstlane(s_cum[lo + 1]);
  cn.b = lo;
  cn.j = S0 - cum_lo;
  cn.nsteps = cum_hi - cum_lo;
  cn.ctx = load_uniform(p.context_lens, lo);
  cn.slot = FUSED ? load_uniform(p.slot_mapping, lo) : 0;
  const int lblk0 = div_by(cn.j * kStep, p.div_block);
  const int blk0 = load_uniform(p.block_tables + lo * p.bt_stride, lblk0);
  SeqWindow win{};
  if (cum_hi < S1) fill_window<FUSED>(p, s_cum, lo + 1, lane, win);
  cursor_enter_block(p, cn, lblk0, blk0);
  for (int S = S0 - A; S < S1; ++S) {
    char* const tiles = s_tile[wave][(S - S0) & (A - 1)];
    const u32 tile = lds_addr(tiles);
    const bool live = S >= S0, issue = S + A < S1;
    const bool seq_end = live && c0.j + 1 == c0.nsteps;
    const int nv0 = min(kStep, c0.ctx - c0.j * kStep);
    const bool starts = S == S0 || c0.j == 0;
    const bool early_v = seq_end && (FUSED || nv0 < kStep);  // the tile's last rows are rewritten
    if (live) {
      wait_upto(issued - c0.mark - (early_v ? tile_ops : 0));
      if (starts) finish_q(c0, c0.nsteps - c0.j <= S1 - S, qv);
      if (early_v) {
        if constexpr (FUSED) issued += finish_new(c0, nv0, tile);
        else clear_past(nv0, tile);
      }
    }

    // ---- scores
    mfma_f32x4_t s[2] = {mfma_f32x4_t{0.f, 0.f, 0.f, 0.f}, mfma_f32x4_t{0.f, 0.f, 0.f, 0.f}};
    if (live) {
      u32x4_t k[8];
      const u32 at[4] = {tile + ka[0], tile + ka[1], tile + ka[2], tile + ka[3]};
      read_k_tile(at, k);
#pragma unroll
      for (int i = 0; i < 8; ++i) s[i & 1] = mfma16(k[i], qv[i >> 1], s[i & 1]);
    }
    int64_t base = 0;
    int rows = 0;
    if (issue) {  // K has been read: its tile takes step S + A
      const StepCursor& prev = c[A - 1];
      const bool next_seq = S + A != S0 && prev.j + 1 == prev.nsteps;
      if (next_seq) {
        int at = prev.b + 1 - win.base;
        while (at >= 64 || (win.live >> at) == 0) {  // a sequence with steps follows
          fill_window<FUSED>(p, s_cum, win.base + 64, lane, win);
          at = 0;
        }
        cursor_start_seq(p, cn, win, at + __builtin_ctzll(win.live >> at), A == 2 ? prev.buf ^ 1 : 0);
      } else if (S + A != S0) {
        cn = prev;
        cn.j = prev.j + 1;
      }
      if (S + A == S0 || next_seq) issued += issue_q(cn);
      int nv;
      base = step_base(p, cn, head_off, nv);
      // FUSED: a sequence's final step holds the token this launch appends, whose slot is
      // not written yet; its row is filled by finish_new
      rows = FUSED && cn.j + 1 == cn.nsteps && nv > 1 ? nv - 1 : nv;
      issue_tile<false>(p, ln, base, rows, tiles);
      issued += tile_ops;
      cn.mark = issued;
    }
    u32 pk[4] = {}, pk2[4] = {};
    if (live) {
      // ---- online softmax of the lane's 8 tokens and, over the row groups, all 32
      float sc[8], mx = kMaxFloor;
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const float x = s[e >> 2][e & 3] * p.scale_log2;
        sc[e] = 16 * (e >> 2) + 4 * q4 + (e & 3) < nv0 ? x : -INFINITY;
        mx = fmaxf(mx, sc[e]);
      }
      mx = xor32_max(xor16_max(mx));
      const float m_new = fmaxf(st.m, mx);
      const float alpha = fast_exp2(st.m - m_new);
      st.m = m_new;
      if (!starts && __any(alpha != 1.f)) {  // a new state is zero
        st.l *= alpha;
#pragma unroll
        for (int mt = 0; mt < 8; ++mt) {
          st.acc[mt] *= alpha;
          if (G > 5) st.acc2[mt] *= alpha;
        }
      }
#pragma unroll
      for (int e = 0; e < 8; e += 2) {
        float v[2], w[2];
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          const float p0 = fast_exp2(sc[e + i] - m_new);
          st.l += p0;
          const float r1 = p0 - round_bf16(p0);
          const float r2 = r1 - round_bf16(r1);
          v[i] = part == 0 ? p0 : (part == 1 ? r1 : r2);
          w[i] = r2;
        }
        pk[e >> 1] = pack_bf16x2(v[0], v[1]);
        if (G > 5) pk2[e >> 1] = pack_bf16x2(w[0], w[1]);
      }
      // ---- O^T += V^T P^T
      if (!early_v) wait_upto(issued - c0.mark - tile_ops);
      u32x2_t vlo[8], vhi[8];
      const u32 at[8] = {tile + va[0], tile + va[1], tile + va[2], tile + va[3],
                         tile + va[4], tile + va[5], tile + va[6], tile + va[7]};
      read_v_tile(at, vlo, vhi);
      const u32x4_t pf = {pk[0], pk[1], pk[2], pk[3]}, pf2 = {pk2[0], pk2[1], pk2[2], pk2[3]};
#pragma unroll
      for (int mt = 0; mt < 8; ++mt) {
        const u32x4_t vt = {vlo[mt].x, vlo[mt].y, vhi[mt].x, vhi[mt].y};
        st.acc[mt] = mfma16(vt, pf, st.acc[mt]);
        if (G > 5) st.acc2[mt] = mfma16(vt, pf2, st.acc2[mt]);
      }
    }
    if (issue) {
      issue_tile<true>(p, ln, base, rows, tiles + kTileBytes);
      issued += tile_ops;
    }
    if (seq_end || S + 1 == S1) {
      // the whole sequence in this range: it ends here and began here
      issued += emit_state<G>(p, c0.b, kvh, range + c0.b, seq_end && S + 1 - c0.nsteps >= S0, c0.bad, n, q4, st);
      reset_state<G>(st);
    }
#pragma unroll
    for (int i = 0; i < A; ++i) c[i] = c[i + 1];
  }
}
// Combines the per-range partial states of sequences that span several ranges.
// grid = (ceil(num_q_heads / 4), num_seqs), one wave per query head: the four 16-lane rows
// take the sequence's slots (consecutive, from first_b + b) round robin, 8 dims per lane,
// and are merged across the wave at the end.
// Latency-bound: the header words (one round trip), then one slot per row (a second one,
// which ends it for up to 4 parts), then 16 slots per round trip, so that a sequence cut
// into many short ranges does not wait for its slots a few at a time.  Against 32 lanes per
// head with 4, then 8 slots per round trip (whole calls): 2 sequences of 3000-4000 tokens
// (up to 62 parts) 21.7 -> 17.4 us, 8 of 600-3000 21.9 -> 20.6 us, one of 611 12.2 -> 11.2 us.
// Rows past the part count are clamped onto the last part and ignored.
constexpr int kMergeHeads = 4;
constexpr int kMergeThreads = 64 * kMergeHeads;
__global__ __launch_bounds__(kMergeThreads) void decode_merge_kernel(const DecodeParams p) {
  constexpr int D = kDecodeHeadDim;
  const int h = blockIdx.x * kMergeHeads + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int b = blockIdx.y;
  const int r = (threadIdx.x >> 4) & 3, d = 8 * (threadIdx.x & 15);
  if (h >= p.num_q_heads) return;
  const int cb = load_uniform(p.header, kHeaderInts + b), cb1 = load_uniform(p.header, kHeaderInts + b + 1);
  const int spr = load_uniform(p.header, 0);
  if (cb1 <= cb) return;  // no steps: written by the main kernel
  const int np = num_parts(cb, cb1, spr);
  if (np <= 1) return;  // written by the main kernel
  const int64_t row0 = static_cast<int64_t>(cb / spr + b) * p.num_q_heads + h;  // first slot's row
  const int64_t hq = p.num_q_heads;  // rows between consecutive slots
  const float* ml = p.part_ml + row0 * 2;
  const float* po = p.part_o + row0 * D + d;
  float m = kMaxFloor, l = 0.f, o[8] = {};
  auto add = [&](float2 s, float4 x, float4 y) {
    const float m_new = fmaxf(m, s.x), alpha = fast_exp2(m - m_new), w = fast_exp2(s.x - m_new);
    const float v[8] = {x.x, x.y, x.z, x.w, y.x, y.y, y.z, y.w};
    m = m_new;
    l = l * alpha + w * s.y;
#pragma unroll
    for (int j = 0; j < 8; ++j) o[j] = o[j] * alpha + w * v[j];
  };
  {
    const int64_t s = min(r, np - 1) * hq;
    const float2 st = *reinterpret_cast<const float2*>(ml + 2 * s);
    const float4 x = *reinterpret_cast<const float4*>(po + s * D), y = *reinterpret_cast<const float4*>(po + s * D + 4);
    if (r < np) add(st, x, y);
  }
#pragma unroll 1
  for (int k0 = 4 + r; k0 - r < np; k0 += 16) {
    float2 st[4];
    float4 x[4], y[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int64_t s = min(k0 + 4 * u, np - 1) * hq;
      st[u] = *reinterpret_cast<const float2*>(ml + 2 * s);
      x[u] = *reinterpret_cast<const float4*>(po + s * D);
      y[u] = *reinterpret_cast<const float4*>(po + s * D + 4);
    }
#pragma unroll
    for (int u = 0; u < 4; ++u)
      if (k0 + 4 * u < np) add(st[u], x[u], y[u]);
  }
  const float mm = xor32_max(xor16_max(m));
  const float w = fast_exp2(m - mm);
  const float inv = 1.f / xor32_sum(xor16_sum(l * w));
#pragma unroll
  for (int j = 0; j < 8; ++j) o[j] = xor32_sum(xor16_sum(o[j] * w)) * inv;
  if (r == 0) *reinterpret_cast<uint4*>(p.out + b * p.o_seq_stride + h * p.o_head_stride + d) = pack8(o);
}

constexpr int64_t kHeaderBytes = ((kHeaderInts + kHeaderSeqs + 1) * 4 + 255) / 256 * 256;
constexpr int64_t kStateBytes = (kDecodeHeadDim + 2) * 4;  // one (acc[128], max, sum) state

// Ranges of one launch: the grid's groups, and no more than minimum-size ranges over the
// largest possible work (max_tokens = sequences * table width * block_size).
static int64_t range_cap(int64_t max_tokens, int64_t range_tokens) {
  return std::max<int64_t>(1, (max_tokens + range_tokens - 1) / range_tokens);
}

// Workspace bytes for a launch of `seqs` sequences over `ranges` ranges.
static int64_t decode_workspace_need(int64_t seqs, int64_t q_heads, int64_t ranges) {
  return kHeaderBytes + (ranges + seqs) * q_heads * kStateBytes;
}

// Workspace bytes that cover every launch of up to `seqs` sequences, on any device:
// a launch has at most kMaxDecodeGrid ranges.
static int64_t decode_workspace_bound(int64_t seqs, int64_t q_heads, int64_t max_blocks, int64_t block_size) {
  const int64_t ranges = std::min<int64_t>(kMaxDecodeGrid, range_cap(seqs * max_blocks * block_size, kWorkspaceRangeTokens));
  return decode_workspace_need(seqs, q_heads, ranges);
}

// f(G, A) with constants for a batch of num_seqs sequences at GQA ratio g.
template <typename F>
static auto with_variant(int g, int num_seqs, F f) {
  using std::integral_constant;
  const integral_constant<int, 2> two;
  switch (g) {
    case 1:
      if (steps_ahead(1, num_seqs) == 1) return f(integral_constant<int, 1>{}, integral_constant<int, 1>{});
      return f(integral_constant<int, 1>{}, two);
    case 2: return f(integral_constant<int, 2>{}, two);
    case 4: return f(integral_constant<int, 4>{}, two);
    case 5: return f(integral_constant<int, 5>{}, two);
    default: return f(integral_constant<int, 8>{}, two);
  }
}

// Workgroups of the kernel resident on the whole current device (cached per device once
// the queries succeed), capped at kMaxDecodeGrid.
template <int G, bool FUSED, int A>
static int resident_workgroups() {
  static std::atomic<int> cached[16];
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 16) dev = 0;
  int v = cached[dev].load(std::memory_order_relaxed);
  if (v > 0) return v;
  int cus = 0, per_cu = 0;
  bool ok = hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) == hipSuccess && cus > 0;
  if (!ok) cus = 256;
  if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, paged_decode_kernel<G, FUSED, A>, kDecodeThreads, 0) !=
          hipSuccess || per_cu <= 0) {
    per_cu = 1;
    ok = false;
  }
  v = std::min(cus * per_cu, kMaxDecodeGrid);
  if (ok) cached[dev].store(v, std::memory_order_relaxed);
  return v;
}

template <int G, bool FUSED, int A>
static void launch_decode(DecodeParams p, int64_t ranges, hipStream_t s) {
  const int64_t groups_per_range = (p.num_kv_heads + kDecodeWaves - 1) / kDecodeWaves;
  p.div_ranges = divisor(static_cast<uint32_t>(ranges));
  const dim3 grid(static_cast<unsigned>(groups_per_range), static_cast<unsigned>(ranges));
  hipLaunchKernelGGL((paged_decode_kernel<G, FUSED, A>), grid, dim3(kDecodeThreads), 0, s, p);
  hipLaunchKernelGGL(decode_merge_kernel, dim3((p.num_q_heads + kMergeHeads - 1) / kMergeHeads, p.num_seqs),
                     dim3(kMergeThreads), 0, s, p);
}

struct DecodeArgs {
  const void* q;
  int64_t q_seq_stride, q_head_stride;
  const void* k_cache;
  const void* v_cache;
  int64_t cache_block_stride, cache_slot_stride, cache_head_stride;
  int32_t num_cache_blocks;
  const int32_t* block_tables;
  int64_t block_table_stride;
  const int32_t* context_lens;
  int32_t num_seqs, num_q_heads, num_kv_heads, head_dim, block_size, max_blocks_per_seq;
  float softmax_scale;
  void* out;
  int64_t out_seq_stride, out_head_stride;
};

// Host-side argument checks shared by both decode entry points (no HIP call).
static int check_decode_args(const char* fn, const DecodeArgs& a) {
  if (a.num_seqs < 0) return fail(KVP_EINVAL, "%s: num_seqs=%d < 0", fn, a.num_seqs);
  if (a.head_dim != kDecodeHeadDim)
    return fail(KVP_EUNSUPPORTED, "%s: head_dim=%d (supported: 128)", fn, a.head_dim);
  if (a.num_kv_heads <= 0 || a.num_q_heads <= 0 || a.num_q_heads % a.num_kv_heads != 0)
    return fail(KVP_EINVAL, "%s: num_q_heads=%d not a multiple of num_kv_heads=%d", fn, a.num_q_heads,
                a.num_kv_heads);
  const int G = a.num_q_heads / a.num_kv_heads;
  if (G != 1 && G != 2 && G != 4 && G != 5 && G != 8)
    return fail(KVP_EUNSUPPORTED, "%s: GQA ratio %d (supported: 1, 2, 4, 5, 8)", fn, G);
  if (a.block_size <= 0 || a.block_size % 64 != 0)
    return fail(KVP_EINVAL, "%s: block_size=%d must be a positive multiple of 64", fn, a.block_size);
  if (a.max_blocks_per_seq <= 0 || a.num_cache_blocks <= 0)
    return fail(KVP_EINVAL, "%s: max_blocks_per_seq=%d num_cache_blocks=%d", fn, a.max_blocks_per_seq,
                a.num_cache_blocks);
  if (static_cast<int64_t>(a.max_blocks_per_seq) * a.block_size > (1ll << 30))
    return fail(KVP_EINVAL, "%s: max_blocks_per_seq*block_size too large", fn);
  if (a.block_table_stride < a.max_blocks_per_seq)
    return fail(KVP_EINVAL, "%s: block_table_stride=%lld < max_blocks_per_seq=%d", fn,
                static_cast<long long>(a.block_table_stride), a.max_blocks_per_seq);
  if (!a.q || !a.k_cache || !a.v_cache || !a.block_tables || !a.context_lens || !a.out)
    return fail(KVP_EINVAL, "%s: null pointer", fn);
  if (!aligned16(a.q) || !aligned16(a.k_cache) || !aligned16(a.v_cache))
    return fail(KVP_EINVAL, "%s: q and cache pointers must be 16-byte aligned", fn);
  if (!aligned16(a.out) || (reinterpret_cast<uintptr_t>(a.block_tables) & 3u) ||
      (reinterpret_cast<uintptr_t>(a.context_lens) & 3u))
    return fail(KVP_EINVAL, "%s: misaligned out/block_tables/context_lens", fn);
  if (!mult8(a.q_seq_stride) || !mult8(a.q_head_stride) || !mult8(a.cache_block_stride) ||
      !mult8(a.cache_slot_stride) || !mult8(a.cache_head_stride) || !mult8(a.out_seq_stride) ||
      !mult8(a.out_head_stride))
    return fail(KVP_EINVAL, "%s: q, cache and out strides must be multiples of 8 elements", fn);
  return KVP_OK;
}

// The ranges of the batch's first (largest) launch: no more than workgroups resident at once,
// nor than the workspace formula counts, so that the plain decode cuts a batch the same way,
// and gives the same bits, whatever workspace it has.  The one-launch step takes a range for
// every step of its tables where `capacity` bytes hold their states.
template <bool FUSED = false>
static int64_t batch_ranges(const DecodeArgs& a, int64_t capacity = 0) {
  const int g = a.num_q_heads / a.num_kv_heads;
  const int nb = std::min(a.num_seqs, seqs_per_launch(g, FUSED, steps_ahead(g, a.num_seqs)));
  const int64_t max_tokens = static_cast<int64_t>(nb) * a.max_blocks_per_seq * a.block_size;
  const int64_t groups = (a.num_kv_heads + kDecodeWaves - 1) / kDecodeWaves;
  const int resident = with_variant(g, a.num_seqs, [](auto G, auto A) {
    return resident_workgroups<decltype(G)::value, FUSED, decltype(A)::value>();
  });
  const int64_t most = std::max<int64_t>(1, resident / groups);
  const int64_t fine = std::min(most, range_cap(max_tokens, kStep));
  if (FUSED && decode_workspace_need(nb, a.num_q_heads, fine) <= capacity) return fine;
  return std::min(most, range_cap(max_tokens, kWorkspaceRangeTokens));
}

// Enqueues the decode of a checked batch on `s` with `ws` as workspace (ws_bytes must
// cover decode_workspace_need of every launch; checked by the callers).  Batches beyond
// the LDS prefix table run as consecutive launches of up to seqs_per_launch sequences; they
// reuse the workspace in stream order.
template <bool FUSED>
static int enqueue_decode(const char* fn, const DecodeArgs& a, int64_t ranges, char* ws, hipStream_t s,
                          const DecodeParams* fused = nullptr) {
  const int g = a.num_q_heads / a.num_kv_heads;
  const int most = seqs_per_launch(g, FUSED, steps_ahead(g, a.num_seqs));
  for (int b0 = 0; b0 < a.num_seqs; b0 += most) {
    const int nb = std::min(most, a.num_seqs - b0);
    DecodeParams p = fused ? *fused : DecodeParams{};
    if (FUSED) {  // this chunk's rows of the per-sequence inputs
      p.qkv += b0 * p.qkv_stride;
      p.slot_mapping += b0;
    }
    p.q = static_cast<const uint16_t*>(a.q) + b0 * a.q_seq_stride;
    p.q_seq_stride = a.q_seq_stride;
    p.q_head_stride = a.q_head_stride;
    p.k_cache = static_cast<const uint16_t*>(a.k_cache);
    p.v_cache = static_cast<const uint16_t*>(a.v_cache);
    p.blk_stride = a.cache_block_stride;
    p.slot_stride = a.cache_slot_stride;
    p.head_stride = a.cache_head_stride;
    p.rows_by_dma = a.cache_slot_stride >= 0 && a.cache_slot_stride <= kMaxDmaRow;
    p.q_by_dma = a.q_head_stride >= 0 && a.q_head_stride <= kMaxDmaRow;
    p.num_cache_blocks = a.num_cache_blocks;
    p.block_tables = a.block_tables + b0 * a.block_table_stride;
    p.bt_stride = a.block_table_stride;
    p.context_lens = a.context_lens + b0;
    p.num_seqs = nb;
    p.num_q_heads = a.num_q_heads;
    p.num_kv_heads = a.num_kv_heads;
    p.block_size = a.block_size;
    p.max_blocks = a.max_blocks_per_seq;
    p.div_block = divisor(static_cast<uint32_t>(a.block_size));
    p.scale_log2 = a.softmax_scale * 1.4426950408889634f;
    p.out = static_cast<uint16_t*>(a.out) + b0 * a.out_seq_stride;
    p.o_seq_stride = a.out_seq_stride;
    p.o_head_stride = a.out_head_stride;
    p.header = reinterpret_cast<int32_t*>(ws);
    p.part_o = reinterpret_cast<float*>(ws + kHeaderBytes);
    p.part_ml = p.part_o + static_cast<size_t>(ranges + nb) * a.num_q_heads * kDecodeHeadDim;
    with_variant(g, a.num_seqs, [&](auto G, auto A) {
      launch_decode<decltype(G)::value, FUSED, decltype(A)::value>(p, ranges, s);
    });
    const int rc = launch_status(fn);
    if (rc != KVP_OK) return rc;
  }
  return KVP_OK;
}

// ---------------------------------------------------------------- no-allocation variant

// Workspace of kvp_paged_decode_bf16_noalloc: one per device, held until the process ends.
constexpr size_t kScratchBytes = 34u << 20;
static __device__ __align__(256) char scratch[kScratchBytes];

// Device address of this device's `scratch`, looked up once per device with that device
// current.  The host-side symbol is not a device address and is never passed to a kernel.
// The lookup may load the library's code object (and the array) on that device, which is
// not an operation to record into a graph: a first call on a device while `stream` is
// being captured is refused, and one call outside capture (any batch) sets the device up.
static int scratch_address(const char* fn, hipStream_t stream, char** out) {
  constexpr int kMaxDevices = 64;
  static std::atomic<char*> addr[kMaxDevices];
  int dev = -1;
  hipError_t err = hipGetDevice(&dev);
  if (err != hipSuccess) return fail(static_cast<int>(err), "%s: hipGetDevice: %s", fn, hipGetErrorString(err));
  if (dev < 0 || dev >= kMaxDevices) return fail(KVP_EINVAL, "%s: device %d beyond %d", fn, dev, kMaxDevices);
  char* ptr = addr[dev].load(std::memory_order_acquire);
  if (!ptr) {
    hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
    err = hipStreamIsCapturing(stream, &cap);
    if (err != hipSuccess)
      return fail(static_cast<int>(err), "%s: hipStreamIsCapturing: %s", fn, hipGetErrorString(err));
    if (cap != hipStreamCaptureStatusNone)
      return fail(KVP_EINVAL,
                  "%s: first call on device %d is inside a graph capture; call it once outside capture "
                  "(any batch) to set up the device's static scratch, then capture",
                  fn, dev);
    void* sym = nullptr;
    err = hipGetSymbolAddress(&sym, HIP_SYMBOL(scratch));
    if (err != hipSuccess || !sym)
      return fail(err != hipSuccess ? static_cast<int>(err) : KVP_EINVAL, "%s: hipGetSymbolAddress(scratch): %s",
                  fn, hipGetErrorString(err));
    ptr = static_cast<char*>(sym);
    addr[dev].store(ptr, std::memory_order_release);
  }
  *out = ptr;
  return KVP_OK;
}

}  // namespace kvp

using namespace kvp;

extern "C" size_t kvp_decode_workspace_bytes(int32_t max_num_seqs, int32_t num_q_heads, int32_t head_dim,
                                             int32_t max_blocks_per_seq, int32_t block_size) {
  if (max_num_seqs <= 0 || num_q_heads <= 0 || head_dim != kDecodeHeadDim || max_blocks_per_seq <= 0 ||
      block_size <= 0)
    return 0;
  const int64_t seqs = std::min<int64_t>(max_num_seqs, kHeaderSeqs);
  return static_cast<size_t>(decode_workspace_bound(seqs, num_q_heads, max_blocks_per_seq, block_size));
}

extern "C" int kvp_paged_decode_bf16(const void* q, int64_t q_seq_stride, int64_t q_head_stride,
                                     const void* k_cache, const void* v_cache,
                                     int64_t cache_block_stride, int64_t cache_slot_stride,
                                     int64_t cache_head_stride, int32_t num_cache_blocks,
                                     const int32_t* block_tables, int64_t block_table_stride,
                                     const int32_t* context_lens, int32_t num_seqs,
                                     int32_t num_q_heads, int32_t num_kv_heads, int32_t head_dim,
                                     int32_t block_size, int32_t max_blocks_per_seq,
                                     float softmax_scale,
                                     void* out, int64_t out_seq_stride, int64_t out_head_stride,
                                     void* workspace, size_t workspace_bytes, void* stream) {
  static const char fn[] = "kvp_paged_decode_bf16";
  clear_error();
  const DecodeArgs a = {q, q_seq_stride, q_head_stride, k_cache, v_cache, cache_block_stride,
                        cache_slot_stride, cache_head_stride, num_cache_blocks, block_tables,
                        block_table_stride, context_lens, num_seqs, num_q_heads, num_kv_heads,
                        head_dim, block_size, max_blocks_per_seq, softmax_scale, out,
                        out_seq_stride, out_head_stride};
  int rc = check_decode_args(fn, a);
  if (rc != KVP_OK) return rc;
  if (num_seqs == 0) return KVP_OK;
  const int chunk_seqs = std::min(num_seqs, kHeaderSeqs);
  const size_t need =
      static_cast<size_t>(decode_workspace_bound(chunk_seqs, num_q_heads, max_blocks_per_seq, block_size));
  if (!workspace || workspace_bytes < need)
    return fail(KVP_EWORKSPACE, "%s: workspace of %zu bytes, %zu needed", fn, workspace_bytes, need);
  if (reinterpret_cast<uintptr_t>(workspace) & 255u)
    return fail(KVP_EINVAL, "%s: workspace must be 256-byte aligned", fn);
  return enqueue_decode<false>(fn, a, batch_ranges(a), static_cast<char*>(workspace),
                               static_cast<hipStream_t>(stream));
}

extern "C" int kvp_paged_decode_bf16_noalloc(const void* q, int64_t q_seq_stride, int64_t q_head_stride,
                                             const void* k_cache, const void* v_cache,
                                             int64_t cache_block_stride, int64_t cache_slot_stride,
                                             int64_t cache_head_stride, int32_t num_cache_blocks,
                                             const int32_t* block_tables, int64_t block_table_stride,
                                             const int32_t* context_lens, int32_t num_seqs,
                                             int32_t num_q_heads, int32_t num_kv_heads, int32_t head_dim,
                                             int32_t block_size, int32_t max_blocks_per_seq,
                                             float softmax_scale,
                                             void* out, int64_t out_seq_stride, int64_t out_head_stride,
                                             void* stream) {
  static const char fn[] = "kvp_paged_decode_bf16_noalloc";
  clear_error();
  const DecodeArgs a = {q, q_seq_stride, q_head_stride, k_cache, v_cache, cache_block_stride,
                        cache_slot_stride, cache_head_stride, num_cache_blocks, block_tables,
                        block_table_stride, context_lens, num_seqs, num_q_heads, num_kv_heads,
                        head_dim, block_size, max_blocks_per_seq, softmax_scale, out,
                        out_seq_stride, out_head_stride};
  int rc = check_decode_args(fn, a);
  if (rc != KVP_OK) return rc;
  if (num_seqs == 0) return KVP_OK;
  const int64_t ranges = batch_ranges(a);
  const int64_t need = decode_workspace_need(std::min(num_seqs, kHeaderSeqs), num_q_heads, ranges);
  if (need > static_cast<int64_t>(kScratchBytes))
    return fail(KVP_EWORKSPACE,
                "%s: %d sequences x %d query heads need %lld bytes of decode scratch; the static scratch "
                "holds %zu (use kvp_paged_decode_bf16 with a caller workspace)",
                fn, std::min(num_seqs, kHeaderSeqs), num_q_heads, static_cast<long long>(need), kScratchBytes);
  char* ws = nullptr;
  rc = scratch_address(fn, static_cast<hipStream_t>(stream), &ws);
  if (rc != KVP_OK) return rc;
  return enqueue_decode<false>(fn, a, ranges, ws, static_cast<hipStream_t>(stream));
}

extern "C" int kvp_paged_decode_fused_bf16(
    const void* qkv, int64_t qkv_tok_stride, const float* cos_sin,
    int32_t max_position, const void* q_norm_weight, const void* k_norm_weight, float eps,
    void* k_cache, void* v_cache, int64_t cache_block_stride, int64_t cache_slot_stride,
    int64_t cache_head_stride, int32_t num_cache_blocks, const int32_t* slot_mapping,
    const int32_t* block_tables, int64_t block_table_stride, const int32_t* context_lens,
    int32_t num_seqs, int32_t num_q_heads, int32_t num_kv_heads, int32_t head_dim,
    int32_t block_size, int32_t max_blocks_per_seq, float softmax_scale,
    void* out, int64_t out_seq_stride, int64_t out_head_stride,
    void* workspace, size_t workspace_bytes, void* stream) {
  static const char fn[] = "kvp_paged_decode_fused_bf16";
  clear_error();
  // q is read from the qkv rows: the q pointer and strides of the shared checks stand in
  // for them (the q heads of row b start at qkv + b * qkv_tok_stride).
  const DecodeArgs a = {qkv, qkv_tok_stride, kRopeDim, k_cache, v_cache, cache_block_stride,
                        cache_slot_stride, cache_head_stride, num_cache_blocks, block_tables,
                        block_table_stride, context_lens, num_seqs, num_q_heads, num_kv_heads,
                        head_dim, block_size, max_blocks_per_seq, softmax_scale, out,
                        out_seq_stride, out_head_stride};
  int rc = check_decode_args(fn, a);
  if (rc != KVP_OK) return rc;
  if (!cos_sin || !q_norm_weight || !k_norm_weight || !slot_mapping)
    return fail(KVP_EINVAL, "%s: null pointer", fn);
  if (max_position < 1) return fail(KVP_EINVAL, "%s: max_position=%d", fn, max_position);
  if (!aligned16(cos_sin) || !aligned16(q_norm_weight) || !aligned16(k_norm_weight) ||
      (reinterpret_cast<uintptr_t>(slot_mapping) & 3u))
    return fail(KVP_EINVAL, "%s: misaligned cos_sin / norm weights / slot_mapping", fn);
  if (qkv_tok_stride < static_cast<int64_t>(num_q_heads + 2 * num_kv_heads) * head_dim)
    return fail(KVP_EINVAL, "%s: qkv row stride %lld is shorter than (hq + 2 hkv) * head_dim", fn,
                static_cast<long long>(qkv_tok_stride));
  if (num_seqs == 0) return KVP_OK;
  const int chunk_seqs = std::min(num_seqs, kHeaderSeqs);
  // the kernel addresses the table and one launch's qkv rows with 32-bit byte offsets
  if (static_cast<int64_t>(max_position) * kRopeDim * 4 > INT32_MAX ||
      static_cast<int64_t>(chunk_seqs) * qkv_tok_stride * 2 > INT32_MAX)
    return fail(KVP_EINVAL, "%s: the cos/sin table or %d qkv rows exceed 2 GiB", fn, chunk_seqs);
  const size_t need =
      static_cast<size_t>(decode_workspace_bound(chunk_seqs, num_q_heads, max_blocks_per_seq, block_size));
  if (!workspace || workspace_bytes < need)
    return fail(KVP_EWORKSPACE, "%s: workspace of %zu bytes, %zu needed", fn, workspace_bytes, need);
  if (reinterpret_cast<uintptr_t>(workspace) & 255u)
    return fail(KVP_EINVAL, "%s: workspace must be 256-byte aligned", fn);
  DecodeParams f{};
  f.qkv = static_cast<const uint16_t*>(qkv);
  f.qkv_stride = qkv_tok_stride;
  f.cos_sin = cos_sin;
  f.max_position = max_position;
  f.q_weight = static_cast<const uint16_t*>(q_norm_weight);
  f.k_weight = static_cast<const uint16_t*>(k_norm_weight);
  f.eps = eps;
  f.slot_mapping = slot_mapping;
  f.num_cache_slots = static_cast<int64_t>(num_cache_blocks) * block_size;
  return enqueue_decode<true>(fn, a, batch_ranges<true>(a, static_cast<int64_t>(workspace_bytes)),
                              static_cast<char*>(workspace), static_cast<hipStream_t>(stream), &f);
}
