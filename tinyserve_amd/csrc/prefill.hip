// Varlen causal prefill attention over the paged KV cache, on gfx950 MFMA.
//
// Reference behaviour: src/tinyserve/triton_prefill.py:50-125 (one program per
// (sequence, query tile, kv head), keys walked in chunks from position 0 to the tile's
// last query position, online softmax, P rounded to the value dtype before P.V) and
// src/tinyserve/attention.py:62-111 for the math it must equal.
//
// Work decomposition. A workgroup of 8 wave64s owns one kv head of one sequence and
// 32 * QB consecutive queries of HG of that kv head's query heads (HG * QB = 8): wave w
// takes query head hg = w % HG and the 32 queries of block qb = w / HG. All eight waves
// share each 64-key tile of K and V.
//
// Memory pipeline. K/V tiles are gathered from the paged cache (slot = table[pos / bs]
// * bs + pos % bs) straight into LDS with gfx950's direct-to-LDS loads
// (global_load_lds_dwordx4: lane l's 16 bytes land at the instruction's LDS base +
// 16 l), through a ring of three stages: while tile t is computed, tiles t + 1 and t + 2
// are in flight. No registers stage the data and no LDS store instructions are issued.
// One load instruction covers RPI consecutive keys (4 at D=128). When a cache block holds
// at least RPI slots those keys share one block, so the block id is a scalar load of the
// table and the address a scalar base plus a per-lane row/unit offset: the gather costs
// the VALU almost nothing. Smaller blocks take per-lane ids from a window of 512 table
// entries staged in LDS (refilled when a gather passes its end). Either way the
// vector-memory counter covers exactly the ring's loads and each stage is waited for with
// an exact vmcnt.
//
// Dispatch order. Workgroup b = (tile_rev * R + r) * heads + head: every sequence's last
// query tile (the one with the most keys) is dispatched, for all kv heads, before any
// earlier tile, so the long-running workgroups start first; and since the hardware
// deals workgroups to the 8 XCDs round-robin, with 8 kv heads each head's workgroups
// share one XCD's L2, where its K/V blocks are re-read by every query tile.
//
// Few query tiles behind long cached prefixes are also cut along the keys over several
// workgroups and merged by a second kernel (the key cut, below).
//
// Three shapes: 8 waves with a 3-stage ring of 64-key tiles (one workgroup per CU, 98 KB
// of LDS, two waves per SIMD) for large launches and prefix-hit chunks; for launches of few
// query tiles and long walks (one or two prompts, chunks behind cached keys), 8 waves over the
// queries of the 4-wave shape (64 x 2 heads) with the keys split in two: waves w and
// w + 4 walk the lower and upper half of the key tiles (a 2-stage ring holding one tile
// of each half, 128 KB) and merge their softmax states through LDS at the end, which
// halves the longest workgroup's walk and puts two waves on each SIMD; and for mid-size
// launches and short prompts, 4 waves over 32-key tiles (a 2-stage ring of 34 KB, 157 VGPRs: three
// workgroups, so three waves, per SIMD), whose extra wave per SIMD and finer key tiles
// outweigh the doubled barriers there. (Block sizes under 4 slots, 8 at D=64, run 4
// waves without the split: the halves' block ids come from the scalar-id gather.)
//
// MFMA formulation (v_mfma_f32_32x32x16_{f16,bf16}). Scores are computed transposed,
// S^T[key, query] = K . Q^T, with K as the A operand (one 16-byte LDS read per lane) and
// Q^T as the B operand (held in registers for the whole kernel). In the 32x32
// accumulator layout lane l holds column l % 32 -- one query -- and rows (keys)
// 8j + 4(l / 32) + i at item 4j + i, so each lane owns 16 of its query's scores per 32
// keys: the softmax max/sum are in-lane plus one exchange between the lane halves. The
// output is accumulated transposed too, O^T[d, query] += V^T . P^T: P^T is the B operand
// straight from the score registers (lane half h supplies keys {4h..4h+3, 8+4h..8+4h+3}
// of each 16-key chunk), and V^T is the A operand, read from the row-major V tile with
// two ds_read_b64_tr_b16 per MFMA. That instruction works on groups of 16 lanes: lane j
// of a group reads 4 consecutive 16-bit values ("row j") and lane i receives element
// i % 4 of rows i / 4, 4 + i / 4, 8 + i / 4, 12 + i / 4. Pointing lane j at
// V[key0 + j / 4][d0 + 4 (j % 4)] gives lane i the values V[key0 .. key0 + 3][d0 + i]:
// four keys of one d, the transposed operand.
//
// LDS layout: K and V tiles are [64 keys][D], rows unpadded, their 16-byte units
// XOR-swizzled per row (K by row & 15, V by a 4-row pattern), which keeps the K operand
// reads and the transposing V reads free of bank conflicts.
#include <algorithm>
#include <type_traits>

#include "common.h"

namespace ts {

typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef short s16x8 __attribute__((ext_vector_type(8)));

#define TS_LDS __attribute__((address_space(3)))
#define TS_CONST __attribute__((address_space(4)))

template <typename T>
struct Mfma;
template <>
struct Mfma<f16> {
  using V8 = f16x8;
  static __device__ __forceinline__ f32x16 mma(V8 a, V8 b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
  }
};
template <>
struct Mfma<bf16> {
  using V8 = bf16x8;
  static __device__ __forceinline__ f32x16 mma(V8 a, V8 b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
  }
};

struct PrefillArgs {
  const void* q;
  const void* k;
  const void* v;
  void* out;
  const int32_t* bt;
  const int32_t* q_starts;
  const int32_t* q_lens;
  const int32_t* ctx_lens;
  int R;
  int group;
  int hchunks;  // group / HG
  int lbs;
  int n_qtiles;
  int n_kvh;
  int seq_group;  // > 0: dispatch in groups of this many sequences ranked by length
  int64_t q_st, q_sh, o_st, o_sh, k_ss, k_sh, bt_s;
  float scale_log2;
  int o_vec;  // output rows 16-byte aligned: stored as whole rows
  // Key cut (0 units: none): fp32 states of the cut items' parts, and the launch's units
  // and CUs per (kv head, head chunk).
  float* ws;
  int32_t* ws_plan;  // [64][2]: each item's parts and first unit
  int units;
  int conc;
};

constexpr int kWin = 512;   // block ids held in LDS
// Before any score: at or below every finite one, so a part of very low scores (bf16 reaches
// -1e34) still starts from its own maximum.
constexpr float kLowest = -3.402823466e38f;
constexpr int kCutKeys = 64;  // keys per tile of the cut shapes

// ---- key cut -----------------------------------------------------------------------------
// A launch with fewer query tiles than CUs and long keys (prompt chunks behind a cached
// prefix) waits for the workgroup with the longest walk while most of the chip idles. The
// cut gives each item (sequence, query tile) several workgroups ("units") over near-equal
// shares of its key tiles; cut items write fp32 softmax states (m, l, O^T) to the
// workspace and prefill_merge_kernel merges them. The host knows sizes only, so every wave
// derives the cut from the lengths itself: lane i holds item i's key tiles, lane j < 63
// prices a share of about 4 x 1.12^j tiles and lane 63 whole items (written directly), and
// the cheapest wins. In steps of one tile, on `conc` CUs: a unit costs its share plus
// kCutUnit of start, end and state traffic; cutting at all costs kCutMerge, and kCutPart
// per part of the longest item; all three are twice as many of the shorter steps of D = 64.
constexpr float kWholeUnit = 2.0f, kCutUnit = 4.0f, kCutMerge = 4.0f, kCutPart = 0.25f;

// No share of four tiles or more is cheaper than whole items of up to this many (4 + kCutUnit +
// kCutMerge against t + kWholeUnit steps, at D = 64 with the longer terms doubled). Such launches,
// short contexts under wide tables, skip the pricing: 16 x 100 fresh tokens under a table of
// 4096 13.1 -> 10.8 us (uncut 9.2), 1 x 40 9.8 -> 8.8 (6.8).
constexpr int kCutNever = 10;

struct CutItem {
  int item;   // r * n_qtiles + tile; -1: this unit has no work
  int part;   // of `parts`
  int parts;  // 1: whole
  int tiles;  // key tiles per part (the last part may hold fewer)
  int unit0;  // the item's first unit
};

// Key tiles of item i (0: no such query tile). BQ queries per tile.
__device__ __forceinline__ int cut_tiles(const PrefillArgs& a, int i, int BQ) {
  const int r = i / a.n_qtiles, tile = i - r * a.n_qtiles;
  const int q_len = a.q_lens[r];
  if (tile * BQ >= q_len) return 0;
  const int keys = a.ctx_lens[r] - q_len + min((tile + 1) * BQ, q_len);
  return (keys + kCutKeys - 1) / kCutKeys;
}

// Where every item's units lie: lane i gets item i's part count, tiles per part and first
// unit (items <= 64; all lanes of the wave call).
template <int D>
__device__ __forceinline__ CutItem cut_plan(const PrefillArgs& a, int BQ) {
  constexpr float kStep = 128.0f / D;
  const int lane = threadIdx.x & (kWave - 1);
  const int items = a.R * a.n_qtiles;
  const int t = lane < items ? cut_tiles(a, lane, BQ) : 0;
  CutItem c;
  c.item = lane;
  c.part = 0;
  const uint64_t live_items = __ballot(t > 0);
  if (__builtin_expect(__all(t <= kCutNever), 0)) {  // out of the priced plan's way: 0.3 us a launch
    c.parts = t > 0;
    c.tiles = t;
    c.unit0 = __popcll(live_items & ((uint64_t{1} << lane) - 1));
    return c;
  }
  const float share = __builtin_floorf(4.0f * fast_exp2(static_cast<float>(lane) * 0.1635f));
  const float inv = 1.0f / share;
  float n = 0.f, total = 0.f, tmax = 1.f, live = 0.f;
  for (int i = 0; i < items; ++i) {
    const float ti = static_cast<float>(__builtin_amdgcn_readlane(t, i));
    const float one = fminf(ti, 1.0f);
    total += ti;
    live += one;
    tmax = fmaxf(tmax, ti);
    n += fmaxf(__builtin_ceilf(ti * inv - 1e-3f), one);
  }
  const bool whole = lane == kWave - 1;
  if (whole) n = live;
  const float conc = static_cast<float>(a.conc);
  // One round waits for its longest unit; several are balanced by the dispatch order but
  // for about half a unit.
  const float ps = whole ? tmax : fminf(share, tmax);
  const float busy = n <= conc ? ps : fmaxf(ps, total / conc + 0.5f * ps);
  float cost = busy + kStep * __builtin_ceilf(n / conc) * (whole ? kWholeUnit : kCutUnit);
  if (!whole) cost += kStep * (kCutMerge + kCutPart * tmax * inv);
  if (n > static_cast<float>(a.units)) cost = 3.0e6f;
  // Cheapest share; ties to the larger one.
  int key = static_cast<int>(fminf(cost, 3.0e6f) * 8.0f) * kWave + (kWave - 1 - lane);
  for (int o = 1; o < kWave; o *= 2) key = min(key, __shfl_xor(key, o));
  const int win = kWave - 1 - (__builtin_amdgcn_readfirstlane(key) & (kWave - 1));
  const float win_inv = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(inv), win));
  c.parts = c.tiles = c.unit0 = 0;
  if (t > 0) {
    c.parts = win == kWave - 1 ? 1 : max(static_cast<int>(__builtin_ceilf(static_cast<float>(t) * win_inv - 1e-3f)), 1);
    c.tiles = (t + c.parts - 1) / c.parts;
    c.parts = (t + c.tiles - 1) / c.tiles;  // no empty last part
  }
  // Units in order of falling size (ties by item), so that the longest start first.
  const int size = c.tiles * kWave + (kWave - 1 - lane);
  for (int i = 0; i < items; ++i)
    c.unit0 += __builtin_amdgcn_readlane(size, i) > size ? __builtin_amdgcn_readlane(c.parts, i) : 0;
  return c;
}

// The item and part that unit u works on (item -1: none), uniform over the wave. The
// launch's first workgroup leaves every item's parts and first unit for the merge.
template <int D>
__device__ __forceinline__ CutItem cut_unit(const PrefillArgs& a, int BQ, int u) {
  const CutItem p = cut_plan<D>(a, BQ);
  if (blockIdx.x == 0 && threadIdx.x < kWave) {
    a.ws_plan[2 * threadIdx.x] = p.parts;
    a.ws_plan[2 * threadIdx.x + 1] = p.unit0;
  }
  const uint64_t hit = __ballot(p.parts > 0 && u >= p.unit0 && u < p.unit0 + p.parts);
  CutItem c;
  if (hit == 0) {
    c.item = -1;
    return c;
  }
  const int ln = __builtin_ctzll(hit);
  c.item = ln;
  c.parts = __builtin_amdgcn_readlane(p.parts, ln);
  c.tiles = __builtin_amdgcn_readlane(p.tiles, ln);
  c.unit0 = __builtin_amdgcn_readlane(p.unit0, ln);
  c.part = u - c.unit0;
  return c;
}

constexpr int kCutPlanFloats = 2 * kWave;  // the plan, at the workspace's start

// Floats of one wave's state in the workspace: O^T [D / 32][4][64 lanes][4], m, l [64].
template <int D>
__host__ __device__ constexpr int64_t cut_state_floats() {
  return static_cast<int64_t>(D / 2 + 2) * kWave;
}

template <int D, int W, int BN>
struct TileShape {
  static constexpr int kUPR = D / 8;          // 16-byte units per row
  static constexpr int kRPI = kWave / kUPR;   // rows one direct-to-LDS instruction fills
  static constexpr int kIPW = BN / kRPI / W;  // such instructions per wave per tensor
  static_assert(kIPW >= 1 && kIPW * kRPI * W == BN, "D in {64, 128}");
};

// Physical 16-byte unit of data unit u in row `row` of a tile is u ^ swz(row).
template <int D>
__device__ __forceinline__ int k_swz(int row) {
  return row & (D / 8 - 1);
}
template <int D>
__device__ __forceinline__ int v_swz(int row) {
  // 4-row patterns: {0, 6, 10, 12} for 16-unit rows, {0, 6, 4, 2} for 8-unit rows.
  constexpr uint32_t kTab = D == 128 ? 0x0C0A0600u : 0x02040600u;
  return (kTab >> ((row & 3) * 8)) & 0xFF;
}

// Instruction classes of __builtin_amdgcn_sched_group_barrier.
constexpr int kSchedMfma = 0x008;
constexpr int kSchedDsRead = 0x100;

// One direct-to-LDS load of 16 bytes per lane (global_load_lds_dwordx4; M0 holds the
// LDS base). Issued as inline asm on purpose: the compiler's wait-count pass would
// otherwise guard every later LDS read with a wait for all such loads in flight (it
// cannot tell ring stages apart), draining the ring each step. The kernel orders these
// loads itself with counted waits before every ring barrier; loads the compiler does not
// count can only make its own waits stricter. Only the device pass sees the asm.
__device__ __forceinline__ void lds_load16(const void* src, TS_LDS void* dst) {
#if defined(__HIP_DEVICE_COMPILE__)
  // M0 is reserved to the compiler: the asm saves and restores it around the load.
  const uint32_t lds = static_cast<uint32_t>(reinterpret_cast<uintptr_t>(dst));
  uint32_t saved;
  asm volatile(
      "s_mov_b32 %0, m0\n\t"
      "s_mov_b32 m0, %1\n\t"
      "global_load_lds_dwordx4 %2, off\n\t"
      "s_mov_b32 m0, %0"
      : "=&s"(saved)
      : "s"(lds), "v"(src)
      : "memory");
#endif
}

// The same load with a scalar base address and a 32-bit per-lane byte offset
// (global_load_lds_dwordx4 voffset, saddr): the address arithmetic of a gather whose
// lanes share one cache block stays on the scalar unit.
// M0 is bound through the asm operand, so the compiler sets it (one instruction) and
// knows it is taken.
__device__ __forceinline__ void lds_load16_s(const void* base, uint32_t voff, TS_LDS void* dst) {
#if defined(__HIP_DEVICE_COMPILE__)
  const uint32_t lds = static_cast<uint32_t>(reinterpret_cast<uintptr_t>(dst));
  asm volatile("global_load_lds_dwordx4 %0, %1" : : "v"(voff), "s"(base), "{m0}"(lds) : "memory");
#endif
}

// Wait until at most N of this wave's vector-memory operations are in flight and all its
// LDS operations are done, then meet the other waves at s_barrier. __syncthreads() would
// also fence workgroup memory, which waits for every load in flight (vmcnt(0)) and so
// drains the ring; the tiles' visibility needs only each wave's own counted wait. The
// signal fences (no instructions) keep the compiler from moving memory accesses across.
template <int N>
__device__ __forceinline__ void ring_barrier() {
  static_assert(N >= 0 && N < 64, "vmcnt field");
  // vmcnt N (bits 3:0 and 15:14), expcnt 7 (no wait), lgkmcnt 0
  __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | 0x0070);
  __atomic_signal_fence(__ATOMIC_SEQ_CST);
  __builtin_amdgcn_s_barrier();
  __atomic_signal_fence(__ATOMIC_SEQ_CST);
}

template <typename T, int D, int HG, int QB, int kWaves, int kStages, int kBN, int kOcc,
          bool kScalarIds, int kParts, bool kCut>
__global__ __launch_bounds__(kWaves * kWave) __attribute__((amdgpu_waves_per_eu(kOcc, kOcc))) void
prefill_mfma_kernel(const PrefillArgs a) {
  using V8 = typename Mfma<T>::V8;
  // Key split (kParts > 1): waves w, w + kGW, ... take the same queries and heads; part
  // kh walks the kh-th contiguous share of the workgroup's key tiles, and the parts'
  // softmax states are merged through LDS at the end. kGW waves share a tile.
  constexpr bool kSplitK = kParts > 1;
  constexpr int kGW = kWaves / kParts;
  static_assert(kGW * kParts == kWaves, "whole waves per key part");
  static_assert(!kSplitK || (kScalarIds && kStages == 2), "key split: scalar ids, 2 stages");
  using Sh = TileShape<D, kGW, kBN>;
  constexpr int NH = kBN / 32;  // 32-key halves of S^T (one MFMA accumulator each)
  constexpr int NC = kBN / 16;  // 16-key chunks of P^T (one PV B operand each)
  static_assert(kStages == 2 || kStages == 3, "ring of 2 or 3 stages");
  constexpr int UPR = Sh::kUPR, RPI = Sh::kRPI, IPW = Sh::kIPW;
  constexpr int BQ = 32 * QB;
  constexpr int DT = D / 32;  // 32-row output tiles
  constexpr int KC = D / 16;  // 16-wide MFMA k-chunks of the head dim
  constexpr int TILE = kBN * D;
  constexpr int DMA_PER_TILE = 2 * IPW;  // direct-to-LDS instructions per wave per tile
  constexpr float kRescale = 8.0f;
  // bf16 keeps 8 significant bits: P rounded once would move outputs by up to ~1e-2
  // against the fp32 reference, so P is carried as hi + lo bf16 parts (about 16 bits)
  // and P.V takes two MFMAs. fp16's 11 bits meet the tolerance with one.
  constexpr bool kSplitP = std::is_same_v<T, bf16>;

  constexpr int kStageStride = kParts * TILE;  // one tile per key part
  constexpr int kRing = kStages * kStageStride;
  __shared__ __attribute__((aligned(16))) T rings[2 * kRing];
  T* const k_ring = rings;
  T* const v_ring = rings + kRing;
  __shared__ int32_t ids_lds[kWin];

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int kh = kSplitK ? wave / kGW : 0;           // key part
  const int wl = kSplitK ? wave - kh * kGW : wave;  // wave within its part
  const int col = lane & 31;  // this lane's query within the wave's 32
  const int half = lane >> 5;

  const int n_hc = a.n_kvh * a.hchunks;
  const int bid = blockIdx.x;
  const int rest = bid / n_hc;
  const int hcx = bid - rest * n_hc;
  int tile_rev, r;
  CutItem cut;  // kCut: this workgroup's share of its item's key tiles
  if constexpr (kCut) {
    cut = cut_unit<D>(a, BQ, rest);
    if (cut.item < 0) return;
    r = cut.item / a.n_qtiles;
    tile_rev = 0;
  } else if (a.seq_group > 0) {
    // Groups of seq_group sequences of similar length, longest group first; within a
    // group, heaviest query tiles first. A group's K/V (one kv head per XCD) stays in
    // that XCD's L2 while its tiles run, which the plain order below loses when many
    // sequences are in flight at once. Lane b ranks sequence b by context length
    // (ties by index; R <= 64).
    const int per_group = a.n_qtiles * a.seq_group;
    const int gi = rest / per_group;
    const int rem = rest - gi * per_group;
    tile_rev = rem / a.seq_group;
    const int want = gi * a.seq_group + (rem - tile_rev * a.seq_group);
    if (want >= a.R) return;
    const int ln = threadIdx.x & (kWave - 1);
    const int mine = ln < a.R ? a.ctx_lens[ln] : -1;
    // Already in rank order (non-increasing lengths): no ranking loop.
    const int next = __shfl_down(mine, 1);
    int rank = ln;
    if (!__all(ln + 1 >= a.R || mine >= next)) {
      rank = 0;
      if (__all(mine < (1 << 25))) {
        // Unique keys (length, then lower index first): rank = keys above this one.
        const int key = ln < a.R ? mine * kWave + (kWave - 1 - ln) : -1;
        // Eight lanes at a time, their numbers immediate (lanes past R rank below all): a
        // loop of one is mostly its own counting, paid by every workgroup.
        // (us, fp16 at 16 / 8 heads: 64 prompts of U[16, 300] 35.5 -> 31.8, 32 of U[16, 2048]
        // 188 -> 185.)
#pragma unroll
        for (int j0 = 0; j0 < kWave; j0 += 8) {
          if (j0 >= a.R) break;
#pragma unroll
          for (int j = 0; j < 8; ++j) rank += __builtin_amdgcn_readlane(key, j0 + j) > key;
        }
      } else {
        for (int j = 0; j < a.R; ++j) {
          const int other = __builtin_amdgcn_readlane(mine, j);
          rank += (other > mine) | ((other == mine) & (j < ln));
        }
      }
    }
    r = __builtin_ctzll(__ballot(ln < a.R && rank == want));
  } else {
    tile_rev = rest / a.R;
    r = rest - tile_rev * a.R;
  }
  const int q_len = a.q_lens[r];
  const int tile = kCut ? cut.item - r * a.n_qtiles : (q_len + BQ - 1) / BQ - 1 - tile_rev;
  if (tile < 0) return;
  const int q0 = tile * BQ;
  const int ctx = a.ctx_lens[r];
  const int q_start = a.q_starts[r];
  const int kvh = hcx / a.hchunks;
  const int hc = hcx - kvh * a.hchunks;
  const int hg = wl % HG;
  const int qb = wl / HG;
  const int head = kvh * a.group + hc * HG + hg;
  const int past = ctx - q_len;  // position of query 0 is past + 0

  const int wq0 = q0 + qb * 32;
  const int qi = wq0 + col;
  const bool q_ok = qi < q_len;
  const int pos = past + qi;
  // Keys the workgroup needs: key_lo .. key_end - 1.
  const int key_lo = kCut ? cut.part * cut.tiles * kBN : 0;
  const int item_end = past + min(q0 + BQ, q_len);
  const int key_end = kCut ? min(item_end, key_lo + cut.tiles * kBN) : item_end;
  const int key_last = key_end - 1;
  const int wave_key_end = wq0 < q_len ? past + min(wq0 + 32, q_len) : 0;
  const int wave_pos_min = past + wq0;

  // Q^T as B operands: lane (col, half) holds d = 16 kc + 8 half .. + 7 of its query.
  V8 qreg[KC];
  {
    const T* qp = static_cast<const T*>(a.q) + static_cast<int64_t>(q_start + qi) * a.q_st +
                  static_cast<int64_t>(head) * a.q_sh + 8 * half;
#pragma unroll
    for (int kc = 0; kc < KC; ++kc) {
      Pack16<T> x;
      if (q_ok) x = load16(qp + 16 * kc);
      else x.raw = u32x4{0, 0, 0, 0};
      qreg[kc] = __builtin_bit_cast(V8, x.raw);
    }
  }

  // Q is complete before the loop: without this wait the compiler re-checks the Q loads
  // with a full vmcnt(0) at every step, which would also wait for the ring's loads.
  __builtin_amdgcn_s_waitcnt(0x0070);

  f32x16 oacc[DT];
#pragma unroll
  for (int dt = 0; dt < DT; ++dt) oacc[dt] = f32x16{};
  float m_run = kLowest;  // running max of scale*log2e*score; finite, so 2^(m_run - x) is 0
  float l_run = 0.f;       // this lane half's share of the softmax denominator

  // ---- the gather: one tile of K and V into a ring stage --------------------------------
  // Block ids of the keys [win_key0, win_key0 + kWin << lbs) sit in LDS, so a gather
  // reads its ids with LDS loads and the vector-memory counter sees only the ring's
  // loads. The window is refilled (with the ring drained) when a gather passes its end:
  // every kWin blocks, i.e. never below 8192 keys for 16-slot blocks.
  const int32_t* btrow = a.bt + static_cast<int64_t>(r) * a.bt_s;
  const int lbs = a.lbs;
  const int bs_mask = (1 << lbs) - 1;
  const int nblk = (key_end + bs_mask) >> lbs;  // blocks holding keys 0 .. key_end - 1
  int win_blk0 = 0;                              // first block id index in the window
  auto fill_window = [&](int blk0) {
    win_blk0 = blk0;
    for (int i = tid; i < kWin; i += kWaves * kWave) {
      const int j = min(blk0 + i, nblk - 1);
      ids_lds[i] = btrow[j];
    }
  };
  const T* kbase = static_cast<const T*>(a.k) + static_cast<int64_t>(kvh) * a.k_sh;
  const T* vbase = static_cast<const T*>(a.v) + static_cast<int64_t>(kvh) * a.k_sh;
  const int dma_row = lane / UPR;   // row within an instruction's RPI rows
  const int dma_unit = lane % UPR;  // physical unit this lane fills

  // Keys past key_end read key_last (finite, owned data): their scores are masked and
  // their V rows meet P = 0.
  //
  // kScalarIds (block size >= RPI): the RPI rows of one load lie in one cache block, so
  // its block id comes from a scalar load of the table (cached in the scalar cache), its
  // base address is scalar, and a lane adds only its row and 16-byte unit.
  const TS_CONST int32_t* bt_c = (const TS_CONST int32_t*)(btrow);
  const uint32_t k_ss_bytes = static_cast<uint32_t>(a.k_ss) * sizeof(T);
  const uint32_t row_bytes = static_cast<uint32_t>(dma_row) * k_ss_bytes;
  uint32_t kunit[IPW], vunit[IPW], rows_bytes[IPW];
#pragma unroll
  for (int m = 0; m < IPW; ++m) {
    const int row = (wl * IPW + m) * RPI + dma_row;
    kunit[m] = 16u * static_cast<uint32_t>(dma_unit ^ k_swz<D>(row));
    vunit[m] = 16u * static_cast<uint32_t>(dma_unit ^ v_swz<D>(row));
    rows_bytes[m] = static_cast<uint32_t>(m * RPI + dma_row) * k_ss_bytes;
  }
  // A wave's IPW * RPI rows of a tile share one block when blocks hold that many slots.
  const bool wave_block = (1 << lbs) >= IPW * RPI;
  auto gather = [&](T* k_lds, T* v_lds, int n0) {
    if constexpr (kScalarIds) {
      if (wave_block) {
        // One block id and one base for all of the wave's loads; rows past key_last
        // read key_last, which lies in the same block.
        const int kw = __builtin_amdgcn_readfirstlane(min(n0 + wl * IPW * RPI, key_last));
        const int blk = bt_c[kw >> lbs];
        const uint64_t boff = ((static_cast<uint64_t>(static_cast<uint32_t>(blk)) << lbs) +
                               static_cast<uint32_t>(kw & bs_mask)) * k_ss_bytes;
        const uint32_t lim = static_cast<uint32_t>(key_last - kw) * k_ss_bytes;
        const char* kb = reinterpret_cast<const char*>(kbase) + boff;
        const char* vb = reinterpret_cast<const char*>(vbase) + boff;
#pragma unroll
        for (int m = 0; m < IPW; ++m) {
          const int row0 = (wl * IPW + m) * RPI;
          const uint32_t voff = min(rows_bytes[m], lim);
          lds_load16_s(kb, voff + kunit[m], (TS_LDS void*)(k_lds + row0 * D));
          lds_load16_s(vb, voff + vunit[m], (TS_LDS void*)(v_lds + row0 * D));
        }
        return;
      }
      // Every id first (scalar loads issued together, one wait), then the loads.
      int key0[IPW], blk[IPW];
#pragma unroll
      for (int m = 0; m < IPW; ++m) {
        key0[m] = __builtin_amdgcn_readfirstlane(min(n0 + (wl * IPW + m) * RPI, key_last));
        blk[m] = bt_c[key0[m] >> lbs];
      }
#pragma unroll
      for (int m = 0; m < IPW; ++m) {
        const int row0 = (wl * IPW + m) * RPI;
        const uint64_t slot0 = (static_cast<uint64_t>(static_cast<uint32_t>(blk[m])) << lbs) +
                               static_cast<uint32_t>(key0[m] & bs_mask);
        const uint64_t boff = slot0 * k_ss_bytes;
        // Rows past key_last read key_last.
        const uint32_t voff = min(row_bytes, static_cast<uint32_t>(key_last - key0[m]) * k_ss_bytes);
        lds_load16_s(reinterpret_cast<const char*>(kbase) + boff, voff + kunit[m],
                     (TS_LDS void*)(k_lds + row0 * D));
        lds_load16_s(reinterpret_cast<const char*>(vbase) + boff, voff + vunit[m],
                     (TS_LDS void*)(v_lds + row0 * D));
      }
      return;
    }
#pragma unroll
    for (int m = 0; m < IPW; ++m) {
      const int row0 = (wl * IPW + m) * RPI;
      const int row = row0 + dma_row;
      const int key = min(n0 + row, key_last);
      const int blk = ids_lds[(key >> lbs) - win_blk0];
      const int64_t slot = (static_cast<int64_t>(blk) << lbs) + (key & bs_mask);
      const int64_t off = slot * a.k_ss;
      lds_load16(kbase + off + 8 * (dma_unit ^ k_swz<D>(row)), (TS_LDS void*)(k_lds + row0 * D));
      lds_load16(vbase + off + 8 * (dma_unit ^ v_swz<D>(row)), (TS_LDS void*)(v_lds + row0 * D));
    }
  };
  // Whether the ids of keys up to min(n0 + kBN, key_end) - 1 lie in the window.
  auto in_window = [&](int n0) {
    if constexpr (kScalarIds) return true;  // no window
    return ((min(n0 + kBN, key_end) - 1) >> lbs) < win_blk0 + kWin;
  };

  // ---- per-lane constants of the operand reads -------------------------------------------
  const int kphys = k_swz<D>(col);  // K rows col and col + 32 swizzle alike
  // This lane's K operand of 16-wide chunk kc: row col, 16-byte unit (2 kc + half)
  // swizzled; the whole offset is kept per chunk, so a read is one address register plus
  // an immediate (stage and 32-key part).
  int kofs[KC];
#pragma unroll
  for (int kc = 0; kc < KC; ++kc) kofs[kc] = col * D + ((2 * kc + half) ^ kphys) * 8;
  // V^T operand: lane j of its 16-lane group points at V[key0 + j / 4][d0 + 4 (j % 4)].
  const int vj = lane & 15;
  const int vdsub = (lane >> 4) & 1;
  const int vkey_lane = 4 * half + (vj >> 2);     // + 16 c0 + 8 t
  const int vd_lane = 16 * vdsub + 4 * (vj & 3);  // + 32 dt
  const int vswz = v_swz<D>(vkey_lane);           // key & 3 = vj >> 2 for every read

  int first_key = 0;  // key of this wave's first tile
  auto attend = [&](const T* k_lds, const T* v_lds, int n0) __attribute__((always_inline)) {
    // S^T = K . Q^T for the tile's 32-key parts: NH independent MFMA chains. The K
    // operands of chunk kc + 1 are read while chunk kc multiplies.
    f32x16 s[NH];
#pragma unroll
    for (int h = 0; h < NH; ++h) s[h] = f32x16{};
    {
      auto kread = [&](int kc, V8 (&x)[NH]) {
#pragma unroll
        for (int h = 0; h < NH; ++h) x[h] = *reinterpret_cast<const V8*>(k_lds + kofs[kc] + 32 * h * D);
      };
      V8 ka[2][NH];
      kread(0, ka[0]);
#pragma unroll
      for (int kc = 0; kc < KC; ++kc) {
        if (kc + 1 < KC) kread(kc + 1, ka[(kc + 1) & 1]);
#pragma unroll
        for (int h = 0; h < NH; ++h) s[h] = Mfma<T>::mma(ka[kc & 1][h], qreg[kc], s[h]);
      }
      // Keep that order through scheduling: reads of chunk kc + 1, then MFMAs of kc.
      __builtin_amdgcn_sched_group_barrier(kSchedDsRead, NH, 0);
#pragma unroll
      for (int kc = 0; kc < KC; ++kc) {
        if (kc + 1 < KC) __builtin_amdgcn_sched_group_barrier(kSchedDsRead, NH, 0);
        __builtin_amdgcn_sched_group_barrier(kSchedMfma, NH, 0);
      }
    }
    // Causal mask, only on a tile that crosses this wave's diagonal: item v of part h
    // holds key n0 + 32 h + 8 (v / 4) + 4 half + v % 4.
    if (n0 + kBN - 1 > wave_pos_min) {
      const int lim = pos - n0 - 4 * half;
#pragma unroll
      for (int h = 0; h < NH; ++h)
#pragma unroll
        for (int v = 0; v < 16; ++v)
          if (32 * h + 8 * (v >> 2) + (v & 3) > lim) s[h][v] = -INFINITY;
    }

    // Online softmax for this lane's query, in base 2 with the scale folded into one
    // FMA: p = 2^(s * c - m), c = scale * log2(e) > 0.
    const float c = a.scale_log2;
    V8 pk[NC];
    V8 pk_lo[kSplitP ? NC : 1];
    typedef float F2 __attribute__((ext_vector_type(2)));
    typedef T T2 __attribute__((ext_vector_type(2)));
    typedef T T4 __attribute__((ext_vector_type(4)));
    // P^T of the tile against the running maximum m_run; returns this lane's sum of P.
    auto make_p = [&]() -> float {
      const float neg_m = -m_run;
      float psum = 0.f;
#pragma unroll
      for (int c0 = 0; c0 < NC; ++c0) {
        const f32x16& sv = s[c0 >> 1];
        T2 h[4], lo[4];
#pragma unroll
        for (int e2 = 0; e2 < 4; ++e2) {
          const int v = 8 * (c0 & 1) + 2 * e2;
          const F2 pf = {fast_exp2(fmaf(sv[v], c, neg_m)), fast_exp2(fmaf(sv[v + 1], c, neg_m))};
          h[e2] = __builtin_convertvector(pf, T2);
          if constexpr (kSplitP) {
            psum += pf[0] + pf[1];
            lo[e2] = __builtin_convertvector(pf - __builtin_convertvector(h[e2], F2), T2);
          } else {
            // The denominator sums the rounded P that P.V uses: one v_dot2 per pair.
            psum = __builtin_amdgcn_fdot2(h[e2], T2{T(1), T(1)}, psum, false);
          }
        }
        const T4 a01 = __builtin_shufflevector(h[0], h[1], 0, 1, 2, 3);
        const T4 a23 = __builtin_shufflevector(h[2], h[3], 0, 1, 2, 3);
        pk[c0] = __builtin_shufflevector(a01, a23, 0, 1, 2, 3, 4, 5, 6, 7);
        if constexpr (kSplitP) {
          const T4 b01 = __builtin_shufflevector(lo[0], lo[1], 0, 1, 2, 3);
          const T4 b23 = __builtin_shufflevector(lo[2], lo[3], 0, 1, 2, 3);
          pk_lo[c0] = __builtin_shufflevector(b01, b23, 0, 1, 2, 3, 4, 5, 6, 7);
        }
      }
      return psum;
    };
    // Lazy rescaling without a maximum on the common path: P is first computed against
    // the old running maximum. A lane's sum bounds each of its P, so if no lane's sum
    // exceeds 2^kRescale every P is at most 2^kRescale (exact in fp32, representable in
    // fp16/bf16) and the tile is done. Otherwise (whenever the scores grew by more than
    // kRescale) the exact maximum is taken, O and l are rescaled, and P is recomputed. A
    // wave's first tile starts from the exact maximum, so it needs no second pass: at
    // n0 == 0 every row has a key (key 0), so the maximum is finite; a cut part's first
    // tile may mask a whole row, whose maximum then stays at m_run's finite start.
    auto tile_max = [&]() -> float {
      float mx = s[0][0];
#pragma unroll
      for (int h = 0; h < NH; ++h)
#pragma unroll
        for (int v = (h == 0 ? 1 : 0); v < 16; ++v) mx = fmaxf(mx, s[h][v]);
      return halves_max(mx) * c;
    };
    if constexpr (kCut) {
      if (n0 == first_key) m_run = fmaxf(m_run, tile_max());
    } else {
      if (n0 == 0) m_run = tile_max();
    }
    float psum = make_p();
    if (__any(!(psum <= exp2f(kRescale)))) {
      const float m_new = fmaxf(m_run, tile_max());
      const float alpha = fast_exp2(m_run - m_new);
      l_run *= alpha;
#pragma unroll
      for (int dt = 0; dt < DT; ++dt) oacc[dt] *= alpha;
      m_run = m_new;
      psum = make_p();
    }
    l_run += psum;

    // O^T += V^T . P^T, the V^T operand by two transposing reads per MFMA; the operand
    // of step i + 1 is read while step i multiplies (step i = (dt, c0), c0 fastest).
    auto vread = [&](int i) -> V8 {
      const int dt = i / NC, c0 = i % NC;
      const int d = dt * 32 + vd_lane;
      s16x4 part[2];
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        const int key = 16 * c0 + 8 * t + vkey_lane;
        const T* p = v_lds + key * D + (((d >> 3) ^ vswz) << 3) + (d & 7);
        part[t] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((TS_LDS s16x4*)(p));
      }
      return __builtin_bit_cast(V8, __builtin_shufflevector(part[0], part[1], 0, 1, 2, 3, 4, 5, 6, 7));
    };
    V8 va[2];
    va[0] = vread(0);
#pragma unroll
    for (int i = 0; i < NC * DT; ++i) {
      if (i + 1 < NC * DT) va[(i + 1) & 1] = vread(i + 1);
      const int dt = i / NC, c0 = i % NC;
      oacc[dt] = Mfma<T>::mma(va[i & 1], pk[c0], oacc[dt]);
      if constexpr (kSplitP) oacc[dt] = Mfma<T>::mma(va[i & 1], pk_lo[c0], oacc[dt]);
    }
    __builtin_amdgcn_sched_group_barrier(kSchedDsRead, 2, 1);
#pragma unroll
    for (int i = 0; i < NC * DT; ++i) {
      if (i + 1 < NC * DT) __builtin_amdgcn_sched_group_barrier(kSchedDsRead, 2, 1);
      __builtin_amdgcn_sched_group_barrier(kSchedMfma, kSplitP ? 2 : 1, 1);
    }
  };

  // ---- the ring: tile t lives in stage t % kStages --------------------------------------
  // Before computing tile t a wave waits for its own loads of tile t (with three stages
  // the loads of tile t + 1, if issued, may stay in flight), then the barrier makes every
  // wave's loads of tile t visible and certifies that all waves finished tile t - 1,
  // whose stage receives tile t + kStages - 1. Stage indices are compile-time constants
  // (the loop is unrolled kStages times), so every LDS address is a base plus an offset.
  auto step = [&](const T* k_cur, const T* v_cur, T* k_nx, T* v_nx, int n0) {
    if constexpr (kStages == 3) {
      if (n0 + kBN < key_end) ring_barrier<DMA_PER_TILE>();
      else ring_barrier<0>();
    } else {
      ring_barrier<0>();
    }
    const int nn = n0 + (kStages - 1) * kBN;
    if (nn < key_end) {
      if (!in_window(nn)) {  // rare: drain, move the window to the gather's first block
        __builtin_amdgcn_s_waitcnt(0x0070);
        __syncthreads();
        fill_window(nn >> lbs);
        __syncthreads();
      }
      gather(k_nx, v_nx, nn);
    }
    if (n0 < wave_key_end) attend(k_cur, v_cur, n0);
  };
  // Stage s of this wave's key part: one tile, at (s * kParts + kh) tiles.
  T* const k0 = k_ring + kh * TILE;
  T* const v0 = v_ring + kh * TILE;
  T* const k1 = k0 + kStageStride;
  T* const v1 = v0 + kStageStride;
  T* const k2 = k0 + (kStages - 1) * kStageStride;  // == k1 with two stages (never used)
  T* const v2 = v0 + (kStages - 1) * kStageStride;

  if constexpr (!kScalarIds) {
    fill_window(0);
    __syncthreads();
  }
  if constexpr (kSplitK) {
    // Part kh takes tiles kh * n_lo .. (kh + 1) * n_lo - 1 (the last part the rest); all
    // parts step n_lo times (the same barriers), later parts' last steps possibly with no
    // tile.
    const int ntiles = (key_end - key_lo + kBN - 1) / kBN;
    const int n_lo = (ntiles + kParts - 1) / kParts;
    const int base = key_lo + kh * n_lo * kBN;
    const int half_end = kh == kParts - 1 ? key_end : min(key_lo + (kh + 1) * n_lo * kBN, key_end);
    first_key = base;
    auto sstep = [&](const T* k_cur, const T* v_cur, T* k_nx, T* v_nx, int n0) {
      ring_barrier<0>();
      if (n0 + kBN < half_end) gather(k_nx, v_nx, n0 + kBN);
      if (n0 < half_end && n0 < wave_key_end) attend(k_cur, v_cur, n0);
    };
    if (base < half_end) gather(k0, v0, base);
    for (int i = 0; i < n_lo; i += 2) {
      sstep(k0, v0, k1, v1, base + i * kBN);
      if (i + 1 >= n_lo) break;
      sstep(k1, v1, k0, v0, base + (i + 1) * kBN);
    }
  } else {
    first_key = key_lo;
    gather(k0, v0, key_lo);
    if constexpr (kStages == 3) {
      if (key_lo + kBN < key_end) gather(k1, v1, key_lo + kBN);
      for (int n0 = key_lo; n0 < key_end; n0 += 3 * kBN) {
        step(k0, v0, k2, v2, n0);
        if (n0 + kBN >= key_end) break;
        step(k1, v1, k0, v0, n0 + kBN);
        if (n0 + 2 * kBN >= key_end) break;
        step(k2, v2, k1, v1, n0 + 2 * kBN);
      }
    } else {
      for (int n0 = key_lo; n0 < key_end; n0 += 2 * kBN) {
        step(k0, v0, k1, v1, n0);
        if (n0 + kBN >= key_end) break;
        step(k1, v1, k0, v0, n0 + kBN);
      }
    }
  }
  // No load may still be writing this workgroup's LDS when its waves end.
  __builtin_amdgcn_s_waitcnt(0x0070);

  if constexpr (kSplitK) {
    // Merge every later part's state into part 0's, lane by lane (the waves have the same
    // layout), one part at a time: m, l and O^T[0] through k_ring, O^T[1..] through
    // v_ring, lane-fastest so that the accesses are conflict-free. Scores are in base-2
    // units.
    static_assert(kGW * (2 + 16) * kWave * 4 <= kRing * sizeof(T), "parked m, l, O^T[0] fit");
    static_assert(kGW * (DT - 1) * 16 * kWave * 4 <= kRing * sizeof(T), "parked O^T[1..] fit");
    float* xk = reinterpret_cast<float*>(k_ring) + wl * (2 + 16) * kWave + lane;
    float* xv = reinterpret_cast<float*>(v_ring) + wl * (DT - 1) * 16 * kWave + lane;
#pragma unroll
    for (int part = kParts - 1; part >= 1; --part) {
      __syncthreads();  // every wave is done with the ring (or with the previous merge)
      if (kh == part) {
        xk[0] = m_run;
        xk[kWave] = l_run;
#pragma unroll
        for (int e = 0; e < 16; ++e) xk[(2 + e) * kWave] = oacc[0][e];
#pragma unroll
        for (int dt = 1; dt < DT; ++dt)
#pragma unroll
          for (int e = 0; e < 16; ++e) xv[((dt - 1) * 16 + e) * kWave] = oacc[dt][e];
      }
      __syncthreads();
      if (kh == 0) {
        const float m1 = xk[0];
        const float mn = fmaxf(m_run, m1);
        const float a0 = fast_exp2(m_run - mn), a1 = fast_exp2(m1 - mn);
        l_run = l_run * a0 + xk[kWave] * a1;
#pragma unroll
        for (int e = 0; e < 16; ++e) oacc[0][e] = oacc[0][e] * a0 + xk[(2 + e) * kWave] * a1;
#pragma unroll
        for (int dt = 1; dt < DT; ++dt)
#pragma unroll
          for (int e = 0; e < 16; ++e)
            oacc[dt][e] = oacc[dt][e] * a0 + xv[((dt - 1) * 16 + e) * kWave] * a1;
        m_run = mn;
      }
    }
    if (kh != 0) return;
  }

  const float l_tot = halves_sum(l_run);
  if constexpr (kCut) {
    if (cut.parts > 1) {
      if (wq0 >= q_len) return;
      float* st = a.ws + ((static_cast<int64_t>(rest) * n_hc + hcx) * kGW + wl) * cut_state_floats<D>();
#pragma unroll
      for (int dt = 0; dt < DT; ++dt)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          typedef float F4 __attribute__((ext_vector_type(4)));
          *reinterpret_cast<F4*>(st + ((dt * 4 + j) * kWave + lane) * 4) =
              F4{oacc[dt][4 * j], oacc[dt][4 * j + 1], oacc[dt][4 * j + 2], oacc[dt][4 * j + 3]};
        }
      st[D / 2 * kWave + lane] = m_run;
      st[(D / 2 + 1) * kWave + lane] = l_tot;
      return;
    }
  }
  const float inv = 1.f / l_tot;
  if (a.o_vec) {
    // Whole rows through LDS (the ring is done with): each lane holds 8 bytes of 16 pieces
    // of its row, and storing those directly gives the L2 16 bytes of each row per
    // instruction, 16 requests per 256-byte row (the launch without its key loop: 32 mixed
    // prompts 63.6 us, 47.7 this way; whole 196 -> 188, 1 x 2048 33.4 -> 32.4, six prompts of
    // 355-576 23.0 -> 20.9). Instead the wave's 32 x D tile goes to its
    // own part of the rings, 16-byte units XOR-swizzled by row, and comes back as 16 bytes
    // per lane, UPR consecutive lanes a row.
    typedef T T4 __attribute__((ext_vector_type(4)));
    static_assert(kGW * 32 * D <= 2 * kRing, "the rings hold every wave's rows");
    __syncthreads();  // every wave is done with the ring and the key halves' merge
    T* const mine = rings + wl * 32 * D;
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        T4 x;
#pragma unroll
        for (int i = 0; i < 4; ++i) x[i] = static_cast<T>(oacc[dt][4 * j + i] * inv);
        *reinterpret_cast<T4*>(mine + col * D + ((dt * 4 + j) ^ (col & (UPR - 1))) * 8 + 4 * half) = x;
      }
    // The wave's own writes, in order before its reads: no barrier.
    const int row0 = lane / UPR, unit = lane % UPR;
    T* const op = static_cast<T*>(a.out) + static_cast<int64_t>(q_start + wq0) * a.o_st +
                  static_cast<int64_t>(head) * a.o_sh + unit * 8;
#pragma unroll
    for (int i = 0; i < 32 / RPI; ++i) {
      const int row = i * RPI + row0;
      if (wq0 + row < q_len)
        store16(op + row * a.o_st, load16(mine + row * D + (unit ^ (row & (UPR - 1))) * 8));
    }
    return;
  }
  if (!q_ok) return;
  T* op = static_cast<T*>(a.out) + static_cast<int64_t>(q_start + qi) * a.o_st +
          static_cast<int64_t>(head) * a.o_sh;
#pragma unroll
  for (int dt = 0; dt < DT; ++dt)
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      typedef T T4 __attribute__((ext_vector_type(4)));
      T4 x;
#pragma unroll
      for (int i = 0; i < 4; ++i) x[i] = static_cast<T>(oacc[dt][4 * j + i] * inv);
      *reinterpret_cast<T4*>(op + dt * 32 + 8 * j + 4 * half) = x;
    }
}

// Merges the parts of the cut items. One workgroup per (item, kv head and head chunk, wave
// of 32 queries of one head); wave (pg, dt) takes 32 output dims of parts pg, pg + PG, ...:
// it reads their m, then their l and O^T weighted by 2^(m - max m), and the PG groups merge
// through LDS. Bound by the states' traffic (4 (D + 2) bytes per row and part, mostly still
// in the last-level cache) or, with few items, by the round trips of one item's parts: PG
// is 4 there. Whole items have been written by the main kernel.
template <typename T, int D, int HG, int QB, int PG>
__global__ __launch_bounds__(PG * D / 32 * kWave) void prefill_merge_kernel(const PrefillArgs a) {
  constexpr int BQ = 32 * QB, GW = HG * QB, DT = D / 32;
  typedef float F4 __attribute__((ext_vector_type(4)));
  typedef T T4 __attribute__((ext_vector_type(4)));
  __shared__ float red[PG > 1 ? (PG - 1) * DT * 18 * kWave : 1];
  const int lane = threadIdx.x & (kWave - 1);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int dt = wave % DT, pg = wave / DT;
  const int n_hc = a.n_kvh * a.hchunks;
  const int wl = blockIdx.x % GW;
  const int hcx = blockIdx.x / GW % n_hc;
  const int item = blockIdx.x / GW / n_hc;
  const int parts = a.ws_plan[2 * item];
  if (parts <= 1) return;
  const int unit0 = a.ws_plan[2 * item + 1];
  const int r = item / a.n_qtiles, tile = item - r * a.n_qtiles;
  const int wq0 = tile * BQ + wl / HG * 32;
  const int q_len = a.q_lens[r];
  if (wq0 >= q_len) return;
  const int64_t stride = static_cast<int64_t>(n_hc) * GW * cut_state_floats<D>();  // one unit
  const float* st = a.ws + unit0 * stride + (static_cast<int64_t>(hcx) * GW + wl) * cut_state_floats<D>();
  const float* ml = st + D / 2 * kWave + lane;
  float m = kLowest;
#pragma unroll 8
  for (int i = pg; i < parts; i += PG) m = fmaxf(m, ml[i * stride]);
  float l = 0.f;
  F4 acc[4] = {};
#pragma unroll 4
  for (int i = pg; i < parts; i += PG) {
    const float w = fast_exp2(ml[i * stride] - m);
    l += w * ml[i * stride + kWave];
#pragma unroll
    for (int j = 0; j < 4; ++j)
      acc[j] += w * *reinterpret_cast<const F4*>(st + i * stride + ((dt * 4 + j) * kWave + lane) * 4);
  }
  if constexpr (PG > 1) {
    auto slot = [&](int g) { return red + (g * DT + dt) * 18 * kWave + lane; };
    if (pg > 0) {
      float* x = slot(pg - 1);
      x[0] = m;
      x[kWave] = l;
#pragma unroll
      for (int e = 0; e < 16; ++e) x[(2 + e) * kWave] = acc[e / 4][e % 4];
    }
    __syncthreads();
    if (pg > 0) return;
#pragma unroll
    for (int g = 0; g < PG - 1; ++g) {
      const float* x = slot(g);
      const float mn = fmaxf(m, x[0]);
      const float a0 = fast_exp2(m - mn), a1 = fast_exp2(x[0] - mn);
      l = l * a0 + x[kWave] * a1;
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[e / 4][e % 4] = acc[e / 4][e % 4] * a0 + x[(2 + e) * kWave] * a1;
      m = mn;
    }
  }
  const int qi = wq0 + (lane & 31);
  if (qi >= q_len) return;
  const int kvh = hcx / a.hchunks;
  const int head = kvh * a.group + (hcx - kvh * a.hchunks) * HG + wl % HG;
  T* op = static_cast<T*>(a.out) + static_cast<int64_t>(a.q_starts[r] + qi) * a.o_st +
          static_cast<int64_t>(head) * a.o_sh + dt * 32 + 4 * (lane >> 5);
  const float inv = 1.f / l;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    T4 x;
#pragma unroll
    for (int i = 0; i < 4; ++i) x[i] = static_cast<T>(acc[j][i] * inv);
    *reinterpret_cast<T4*>(op + 8 * j) = x;
  }
}

// KP > 1: the key-split shape (W waves, W / KP per key part); its caller checks that the
// block size allows the scalar-id gather.
template <typename T, int D, int HG, int W, int S, int BN, int OCC, int KP = 1>
static int launch_prefill_mfma(const PrefillArgs& a, int Hkv, hipStream_t stream) {
  constexpr int QB = W / KP / HG;
  const int seqs = a.seq_group > 0 ? (a.R + a.seq_group - 1) / a.seq_group * a.seq_group : a.R;
  dim3 grid(static_cast<unsigned>(a.n_qtiles) * seqs * Hkv * a.hchunks);
  if constexpr (KP > 1) {
    hipLaunchKernelGGL((prefill_mfma_kernel<T, D, HG, QB, W, S, BN, OCC, true, KP, false>), grid,
                       dim3(W * kWave), 0, stream, a);
  } else {
    // A load's RPI rows share a cache block when blocks hold at least RPI slots.
    if ((1 << a.lbs) >= TileShape<D, W, BN>::kRPI)
      hipLaunchKernelGGL((prefill_mfma_kernel<T, D, HG, QB, W, S, BN, OCC, true, 1, false>), grid, dim3(W * kWave), 0, stream, a);
    else
      hipLaunchKernelGGL((prefill_mfma_kernel<T, D, HG, QB, W, S, BN, OCC, false, 1, false>), grid, dim3(W * kWave), 0, stream, a);
  }
  return launch_status();
}

// Query tiles of 32 * (W / KP / HG) queries (KP: key parts), and the dispatch order. Which
// shape a launch runs is prefill_shape's choice.
template <typename T, int D, int W, int S, int BN, int OCC, int KP = 1>
static int dispatch_hg_w(PrefillArgs& a, int Hkv, int max_q_len, int64_t n_rows, hipStream_t stream) {
  constexpr int WQ = W / KP;  // waves over the queries and heads
  const int hg = a.group < WQ ? a.group : WQ;
  a.hchunks = a.group / hg;
  const int bq = 32 * (WQ / hg);
  a.n_qtiles = (max_q_len + bq - 1) / bq;
  a.n_kvh = Hkv;
  // Length-ranked groups of 4096 / (mean new tokens) sequences (1 to 8, at most R: a
  // group's K/V about fits one XCD's L2), for 8-16 sequences, short prompts (mean up to
  // 512 new tokens), or 32 or more prompts of one length, up to 64 sequences; pairs for
  // 17-64 prompts of mixed lengths above that mean. Measured at Qwen3 shapes: +43% on 8
  // mixed prompts, +27% on 64 x 256, +5% on 16 x 512, +4-6% on 48-64 x 1024, +2% on
  // 32 x 2048, +5.6% on average (-0.4% to +24%) over 16 batches of 24-64 mixed prompts;
  // for a few long prompts (-2.6% at 4 x 2048; -7 to -12% for 4 equal ones) the plain
  // order is kept.
  a.seq_group = 0;
  if (a.R > 1 && a.R <= kWave && n_rows > 0) {
    const int64_t mean = (n_rows + a.R - 1) / a.R;
    const bool uniform = n_rows == static_cast<int64_t>(a.R) * max_q_len;
    if (a.R > 16 && !uniform && mean > 512) {
      a.seq_group = 2;
    } else if ((a.R >= 8 && a.R <= 16) || mean <= 512 || (uniform && a.R >= 32)) {
      const int g = static_cast<int>(std::min<int64_t>(8, std::max<int64_t>(1, 4096 / std::max<int64_t>(mean, 1))));
      a.seq_group = g < a.R ? g : a.R;
    }
  }
  switch (hg) {
    case 1: return launch_prefill_mfma<T, D, 1, W, S, BN, OCC, KP>(a, Hkv, stream);
    case 2: return launch_prefill_mfma<T, D, 2, W, S, BN, OCC, KP>(a, Hkv, stream);
    case 4:
      if constexpr (WQ >= 4) return launch_prefill_mfma<T, D, 4, W, S, BN, OCC, KP>(a, Hkv, stream);
      return TS_EUNSUPPORTED;
    case 8:
      if constexpr (WQ >= 8) return launch_prefill_mfma<T, D, 8, W, S, BN, OCC, KP>(a, Hkv, stream);
      return TS_EUNSUPPORTED;
    default: return TS_EUNSUPPORTED;
  }
}

// Which of the three workgroup shapes a launch runs (see the header comment). wg8 is the
// 8-wave grid, n4 the key-split shape's workgroups with query tiles in them (counted from
// the rows where the host knows them: a grid sized by the longest of mixed prompts is mostly
// empty), max_keys a bound on every context (0: unknown, taken for long). The key-split shape
// runs one workgroup per CU and halves the longest walk; the 4-wave, 32-key shape (three per
// CU) starts and ends sooner, and takes what is left of the small and mid-size launches. So
// the key-split one wins from a walk on (keys a query of the longest sequence sees, cached
// ones included) that grows with the rounds of n4: 250 keys times their square, and 150 at
// least. Measured, us (16 q / 8 kv heads, D = 128, fp16, key-split / 32-key / 8-wave): 1 x 512
// 12.7 / 14.2 / 16.7, 8 x 512 23.4 / 19.8 / 21.7, 16 x 200 19.0 / 14.1 / 14.0, six prompts of
// 355-576 20.3 / 18.4 / 19.4, three of up to 2294 36.2 / 49.0 / 56.7, 2 x 2048 45.8 / 51.8 /
// 55.8; behind cached keys (cached + new, bf16) 1 x (14474 + 214) 235 / 372 / 439, 5 x (629 +
// 219) 23.3 / 28.6 / 33.5, 25 x (2849 + 143) 68 / 57 / 66. Over 920 drawn batches that the line
// decides: 1.2% over the better shape of each; two lose over 5% against the key-split shape
// throughout (the most 14%). By the new tokens alone, without the cached keys, up to 58% were
// lost. Up to 128 new tokens without a long prefix (8 tiles of 32 keys): 1 x 64 7.3 / 5.7 / 5.6,
// 8 x 128 8.8 / 7.5 / 8.9, 47 x (U[123, 247] + U[1, 10]) 32-key 14.0, 8-wave 20.7. Grids of up to 8
// 8-wave workgroups per CU (3-16 prompts of 2048, 1-4 of 4096-8192: +1-10%), and of up to 16
// when the mean new tokens per sequence is at most 1280 (8-32 mixed prompts: +5-14%), the
// 32-key shape; larger grids the 8-wave one.
enum class PrefillShape { kW8, kW4, kW4Short };

static PrefillShape prefill_shape(int R, int group, int Hkv, int max_q_len, int64_t n_rows, int64_t max_keys) {
  const int hg8 = group < 8 ? group : 8;
  const int64_t wg8 = static_cast<int64_t>((max_q_len + 32 * (8 / hg8) - 1) / (32 * (8 / hg8))) *
                      R * Hkv * (group / hg8);
  const int64_t cus = compute_units();
  if (group > 4) return PrefillShape::kW8;
  // Up to 128 new tokens and no long cached prefix: a few key tiles, all start and end.
  if (max_q_len <= 128 && max_keys > 0 && max_keys <= 256) return PrefillShape::kW4Short;
  // Up to 64 new tokens per sequence in a launch of at most half an 8-wave workgroup per
  // CU: the key-split shape (its 64 queries hold each sequence, and it halves every walk
  // of the long cached prefix; +5-25% there, -4% to -11% in larger launches).
  if (max_q_len <= 64 && 2 * wg8 <= cus) return PrefillShape::kW4;
  // Up to 128 new tokens per sequence: one 8-wave query tile holds a whole sequence, so
  // its K/V (the whole cached prefix) is read once per kv head, not once per 64 queries.
  if (max_q_len <= 128) return PrefillShape::kW8;
  const int oq = 32 * (4 / group);
  const int64_t longest = static_cast<int64_t>(R) * ((max_q_len + oq - 1) / oq);
  const bool mixed = n_rows > 0 && n_rows < static_cast<int64_t>(R) * max_q_len;
  const int64_t n4 = Hkv * (mixed ? std::min(longest, n_rows / oq + (R + 1) / 2) : longest);
  const int64_t past = max_keys > 0 ? std::max<int64_t>(max_keys - max_q_len, 0) : int64_t{1} << 31;
  const int64_t walk = past + max_q_len / 2;
  if (2 * wg8 < 3 * cus && walk >= 150 && walk * cus * cus >= 250 * n4 * n4) return PrefillShape::kW4;
  const bool short_mean = n_rows > 0 && n_rows <= 1280 * static_cast<int64_t>(R);
  if (wg8 <= 8 * cus || (short_mean && wg8 <= 16 * cus)) return PrefillShape::kW4Short;
  return PrefillShape::kW8;
}

// ---- the key cut's launches --------------------------------------------------------------
// Its two shapes, both over 64-key tiles: the key-split one (64 queries x 2 heads, two key
// halves inside the workgroup) up to 64 new tokens per sequence and where the launch would
// run it uncut, so that a launch with nothing to cut (short contexts under a wide table) costs
// no more than the plan and the merge's launch (1 x 500 fresh tokens under 16384 keys: 18.8 us
// in the 8-wave shape, 14.1 in this, 13.1 uncut); else the 8-wave one.
struct CutShape {
  int hg, waves;  // heads per workgroup; waves over the queries and heads
  int n_qtiles, hchunks, units, conc;
};

// Whether a launch of these sizes may cut its keys, and how. max_keys: the block table's
// width in keys, the most any sequence can have. The line: what a cut can save must exceed
// the plan (~1 us), the merge launch (2 us empty, 9-10 us with 2-4 parts of 100 rows x 16
// sequences) and the states' traffic. Measured at 16 q / 8 kv heads, D = 128, fp16 in graph
// replay (cached + new tokens, uncut -> cut, us): 16 x (U[500, 5000] + U[20, 128]) 122 -> 78, 1 x
// (8192 + 64) 110 -> 27, 1 x (8192 + 200) 109 -> 36, 1 x (8192 + 512) 113 -> 56, 1 x (16000 + 32)
// 204 -> 30, 6 x (3000 + 128) 81 -> 43, 24 x (U[0, 6000] + U[10, 128]) 140 -> 107, 8 x (2000 + 16)
// 33 -> 27; with equal lengths on most of the chip the plan keeps items whole (24 x (4096 + 128)
// 152 -> 149-153). Below the line it lost, on other prefixes of these sizes: 4 x (1024 + 64) 21
// -> 26, 4 x (8192 + 300) 115 -> 125, 1 x (1500 + 256) 29 -> 33, 16 x (4096 + 64) 73 -> 75, 32 x
// (2048 + 128) 94 -> 99.
static bool cut_shape(int R, int group, int Hkv, int D, int lbs, int max_q_len, int64_t max_keys, CutShape* c) {
  if (max_q_len > 512 || max_keys < 1024 || max_keys < 4 * static_cast<int64_t>(max_q_len)) return false;
  if ((1 << lbs) < kWave / (D / 8)) return false;  // scalar-id gather
  const bool halves = prefill_shape(R, group, Hkv, max_q_len, 0, max_keys) == PrefillShape::kW4;
  c->waves = (halves || max_q_len <= 64) && group <= 4 ? 4 : 8;
  c->hg = group < c->waves ? group : c->waves;
  c->hchunks = group / c->hg;
  const int bq = 32 * (c->waves / c->hg);
  c->n_qtiles = (max_q_len + bq - 1) / bq;
  const int n_hc = Hkv * c->hchunks;
  const int64_t items = static_cast<int64_t>(R) * c->n_qtiles;
  const int cus = compute_units();
  if (items > kWave) return false;
  // What a cut can gain, in steps of the longest workgroup of the shape that runs
  // otherwise (`fill`: its workgroups per CU).
  if (!halves && max_q_len > 128) return false;
  const int hg = halves ? std::min(group, 4) : std::min(group, 8);
  const int oq = 32 * ((halves ? 4 : 8) / hg);
  const double fill = static_cast<double>((max_q_len + oq - 1) / oq) * R * Hkv * (group / hg) / cus;
  const double steps = static_cast<double>(max_keys) / (halves ? 2 * kCutKeys : kCutKeys);
  const double gain = steps * (1.0 - (halves ? 1.6 : 1.0) * fill);
  if (gain < (halves && (max_q_len > 128 || D == 64) ? 20.0 : 9.0 * (128 / D))) return false;
  c->conc = cus / n_hc > 1 ? cus / n_hc : 1;
  c->units = static_cast<int>(std::max<int64_t>(items, 2 * c->conc));
  return true;
}

template <typename T, int D, int HG, int W, int S, int KP>
static int launch_cut(const PrefillArgs& a, hipStream_t stream) {
  constexpr int GW = W / KP, QB = GW / HG;
  const int n_hc = a.n_kvh * a.hchunks;
  hipLaunchKernelGGL((prefill_mfma_kernel<T, D, HG, QB, W, S, kCutKeys, 2, true, KP, true>), dim3(a.units * n_hc),
                     dim3(W * kWave), 0, stream, a);
  if (const int rc = launch_status()) return rc;
  const int items = a.R * a.n_qtiles;
  if (items <= 8)
    hipLaunchKernelGGL((prefill_merge_kernel<T, D, HG, QB, 4>), dim3(items * n_hc * GW), dim3(4 * D / 32 * kWave), 0,
                       stream, a);
  else
    hipLaunchKernelGGL((prefill_merge_kernel<T, D, HG, QB, 1>), dim3(items * n_hc * GW), dim3(D / 32 * kWave), 0,
                       stream, a);
  return launch_status();
}

template <typename T, int D>
static int dispatch_cut(PrefillArgs& a, const CutShape& c, int Hkv, hipStream_t stream) {
  a.hchunks = c.hchunks;
  a.n_qtiles = c.n_qtiles;
  a.n_kvh = Hkv;
  a.seq_group = 0;
  a.units = c.units;
  a.conc = c.conc;
  a.ws += kCutPlanFloats;  // the plan comes first
  if (c.waves == 4) {
    switch (c.hg) {
      case 1: return launch_cut<T, D, 1, 8, 2, 2>(a, stream);
      case 2: return launch_cut<T, D, 2, 8, 2, 2>(a, stream);
      default: return launch_cut<T, D, 4, 8, 2, 2>(a, stream);
    }
  }
  switch (c.hg) {
    case 1: return launch_cut<T, D, 1, 8, 3, 1>(a, stream);
    case 2: return launch_cut<T, D, 2, 8, 3, 1>(a, stream);
    case 4: return launch_cut<T, D, 4, 8, 3, 1>(a, stream);
    default: return launch_cut<T, D, 8, 8, 3, 1>(a, stream);
  }
}

template <typename T, int D>
static int dispatch_hg(PrefillArgs& a, int Hkv, int max_q_len, int64_t n_rows, int64_t max_keys,
                       hipStream_t stream) {
  switch (prefill_shape(a.R, a.group, Hkv, max_q_len, n_rows, max_keys)) {
    case PrefillShape::kW4Short: return dispatch_hg_w<T, D, 4, 2, 32, 3>(a, Hkv, max_q_len, n_rows, stream);
    case PrefillShape::kW4:
      // Two key halves per workgroup (8 waves, one workgroup and two waves per SIMD per
      // CU) where the scalar-id gather applies; else the plain 4-wave shape.
      if ((1 << a.lbs) >= TileShape<D, 4, 64>::kRPI)
        return dispatch_hg_w<T, D, 8, 2, 64, 2, 2>(a, Hkv, max_q_len, n_rows, stream);
      return dispatch_hg_w<T, D, 4, 2, 64, 2>(a, Hkv, max_q_len, n_rows, stream);
    default: return dispatch_hg_w<T, D, 8, 3, 64, 2>(a, Hkv, max_q_len, n_rows, stream);
  }
}

int prefill_rows_generic(const void* q, const void* k, const void* v, void* out,
                         const int32_t* bt, const int32_t* q_starts, const int32_t* q_lens,
                         const int32_t* ctx_lens, int R, int Hq, int Hkv, int D, int lbs,
                         int max_q_len, int64_t q_st, int64_t q_sh, int64_t o_st, int64_t o_sh,
                         int64_t k_ss, int64_t k_sh, int64_t bt_s, float scale, int dtype,
                         hipStream_t stream);

}  // namespace ts

using namespace ts;

// Whether the MFMA kernels take these types and rows: their direct-to-LDS gather moves
// 16-byte units, so rows must start 16-byte aligned.
static bool mfma_rows(const void* k, const void* v, int64_t k_ss, int64_t k_sh, int D, int dtype) {
  return (dtype == TS_F16 || dtype == TS_BF16) && (D == 64 || D == 128) && k_ss % 8 == 0 && k_sh % 8 == 0 &&
         reinterpret_cast<uintptr_t>(k) % 16 == 0 && reinterpret_cast<uintptr_t>(v) % 16 == 0;
}

extern "C" int64_t ts_prefill_workspace(int R, int Hq, int Hkv, int D, int block_size, int max_q_len,
                                        int64_t max_keys, int dtype) {
  if (R <= 0 || max_q_len <= 0 || Hq <= 0 || Hkv <= 0 || Hq % Hkv || !is_pow2(Hq / Hkv) || !is_pow2(block_size))
    return 0;
  CutShape c;
  if ((dtype != TS_F16 && dtype != TS_BF16) || (D != 64 && D != 128) ||
      !cut_shape(R, Hq / Hkv, Hkv, D, ilog2(block_size), max_q_len, max_keys, &c))
    return 0;
  return kCutPlanFloats + static_cast<int64_t>(c.units) * Hkv * c.hchunks * c.waves *
         (D == 128 ? cut_state_floats<128>() : cut_state_floats<64>());
}

extern "C" int ts_prefill_plan(int R, int Hq, int Hkv, int D, int block_size, int max_q_len, int64_t n_rows,
                               int64_t max_keys, int dtype) {
  if (R <= 0 || max_q_len <= 0 || Hq <= 0 || Hkv <= 0 || Hq % Hkv || !is_pow2(Hq / Hkv) || !is_pow2(block_size))
    return TS_EINVAL;
  if ((dtype != TS_F16 && dtype != TS_BF16) || (D != 64 && D != 128)) return 0;
  CutShape c;
  if (cut_shape(R, Hq / Hkv, Hkv, D, ilog2(block_size), max_q_len, max_keys, &c)) return c.waves == 4 ? 5 : 4;
  switch (prefill_shape(R, Hq / Hkv, Hkv, max_q_len, n_rows, max_keys)) {
    case PrefillShape::kW8: return 1;
    case PrefillShape::kW4: return 2;
    default: return 3;
  }
}

extern "C" int ts_prefill_varlen(const void* q, const void* k_cache, const void* v_cache,
                                 void* out, const int32_t* block_tables,
                                 const int32_t* q_starts, const int32_t* q_lens,
                                 const int32_t* context_lens, int R, int Hq, int Hkv, int D,
                                 int block_size, int max_q_len, int64_t n_rows,
                                 int64_t q_stride_t,
                                 int64_t q_stride_h, int64_t o_stride_t, int64_t o_stride_h,
                                 int64_t k_stride_slot, int64_t k_stride_head,
                                 int64_t bt_stride, float scale, int dtype, void* stream) {
  return ts_prefill_varlen_ws(q, k_cache, v_cache, out, block_tables, q_starts, q_lens, context_lens, R, Hq, Hkv, D,
                              block_size, max_q_len, n_rows, q_stride_t, q_stride_h, o_stride_t, o_stride_h,
                              k_stride_slot, k_stride_head, bt_stride, scale, dtype, 0, nullptr, 0, stream);
}

extern "C" int ts_prefill_varlen_ws(const void* q, const void* k_cache, const void* v_cache, void* out,
                                    const int32_t* block_tables, const int32_t* q_starts, const int32_t* q_lens,
                                    const int32_t* context_lens, int R, int Hq, int Hkv, int D, int block_size,
                                    int max_q_len, int64_t n_rows, int64_t q_stride_t, int64_t q_stride_h,
                                    int64_t o_stride_t, int64_t o_stride_h, int64_t k_stride_slot,
                                    int64_t k_stride_head, int64_t bt_stride, float scale, int dtype,
                                    int64_t max_keys, float* workspace, int64_t workspace_floats, void* stream) {
  if (R < 0 || max_q_len < 0 || n_rows < 0 || Hq <= 0 || Hkv <= 0 || Hq % Hkv || !is_pow2(Hq / Hkv) ||
      !is_pow2(block_size))
    return TS_EINVAL;
  if (R == 0 || max_q_len == 0) return 0;
  hipStream_t st = static_cast<hipStream_t>(stream);
  const int lbs = ilog2(block_size);
  if (mfma_rows(k_cache, v_cache, k_stride_slot, k_stride_head, D, dtype)) {
    const int o_vec = o_stride_t % 8 == 0 && o_stride_h % 8 == 0 && reinterpret_cast<uintptr_t>(out) % 16 == 0;
    PrefillArgs a{q, k_cache, v_cache, out, block_tables, q_starts, q_lens, context_lens,
                  R, Hq / Hkv, 1, lbs, 1, Hkv, 0, q_stride_t, q_stride_h, o_stride_t, o_stride_h,
                  k_stride_slot, k_stride_head, bt_stride, scale * kLog2e, o_vec, workspace, reinterpret_cast<int32_t*>(workspace), 0, 0};
    CutShape c;
    const int64_t need = workspace ? ts_prefill_workspace(R, Hq, Hkv, D, block_size, max_q_len, max_keys, dtype) : 0;
    if (need > 0 && workspace_floats >= need && reinterpret_cast<uintptr_t>(workspace) % 16 == 0 &&
        cut_shape(R, Hq / Hkv, Hkv, D, lbs, max_q_len, max_keys, &c)) {
      if (dtype == TS_F16)
        return D == 64 ? dispatch_cut<f16, 64>(a, c, Hkv, st) : dispatch_cut<f16, 128>(a, c, Hkv, st);
      return D == 64 ? dispatch_cut<bf16, 64>(a, c, Hkv, st) : dispatch_cut<bf16, 128>(a, c, Hkv, st);
    }
    if (dtype == TS_F16) {
      return D == 64 ? dispatch_hg<f16, 64>(a, Hkv, max_q_len, n_rows, max_keys, st)
                     : dispatch_hg<f16, 128>(a, Hkv, max_q_len, n_rows, max_keys, st);
    }
    return D == 64 ? dispatch_hg<bf16, 64>(a, Hkv, max_q_len, n_rows, max_keys, st)
                   : dispatch_hg<bf16, 128>(a, Hkv, max_q_len, n_rows, max_keys, st);
  }
  return prefill_rows_generic(q, k_cache, v_cache, out, block_tables, q_starts, q_lens,
                              context_lens, R, Hq, Hkv, D, lbs, max_q_len, q_stride_t,
                              q_stride_h, o_stride_t, o_stride_h, k_stride_slot,
                              k_stride_head, bt_stride, scale, dtype, st);
}
