// Kernel 4: chunked-prefill attention on MFMA, history read straight from the paged pool.
//
// Behaviour of a chunked-prefill layer of the reference: the history gather of
// PagedKVCachePool.gather_blocks (src/mini_infra/worker/paged_kv_cache.py:54-72), the concat of
// history and chunk in Qwen3Attention.forward (src/mini_infra/model/qwen3.py:325-330), the visibility
// mask of PagedRunner.run_prefill_chunk_step (src/mini_infra/worker/paged_runner.py:83-89) with the
// causal mask of Qwen3Model._prepare_position_ids_and_allowed_mask (qwen3.py:477-484), and
// Qwen3Attention._attend (qwen3.py:219-255) -- as one flash-style kernel.
//
// Row b of the batch: chunk of padded length L whose last len_b positions are real (left
// padding), logical start start_b, history = the first nh = min(start_b, 16 * max_history_blocks)
// pool slots of its block table.  Query i (i >= L - len_b) sees every history slot k < nh and
// chunk keys j with L - len_b <= j <= i.  Rows i < L - len_b (padding) get a zero output.
//
// Tiling for gfx950 (v_mfma_f32_16x16x32_bf16, 64-lane wavefronts):
//  * workgroup = (row b, query-head pair p of KV head g, 128-query tile), 8 wavefronts (one
//    workgroup per CU at two waves per SIMD): wave w serves query head G g + 2 p + (w >> 2) of the
//    GQA group of G heads on KV head g and queries [32 (w & 3), +32) of the tile, so the two
//    heads share every K/V tile staged in LDS.  A group of G heads takes ceil(G / 2) pairs; when G
//    is odd, the second half of its last pair repeats the group's last head and writes nothing.
//  * Dispatch order: the query tiles of one (row, head pair) stay on one XCD (shared L2), and each
//    XCD's queue runs in rounds of as many whole pairs as its CUs hold, heaviest query tiles first
//    inside a round, so the causal chunk's light and heavy tiles pair up on every CU.
//  * KV tiles of 64 keys: history tiles first (pool blocks through the block table -- the
//    gather is fused, nothing is materialised), then chunk tiles up to the causal limit.
//    K and V tiles go from memory straight into double-buffered LDS (global_load_lds_dwordx4, no
//    registers on the way), row-major with 256-byte rows whose 16-byte chunks are XOR-swizzled by
//    the row; tile t + 1 is in flight while tile t is multiplied.
//  * S^T = K Q^T: A = K rows from LDS, B = Q^T from registers (loaded once), C lane layout =
//    (query = lane % 16, keys 4 (lane / 16) + i).  Each query's softmax state lives in the
//    lanes of its column; the row max needs two cross-lane steps, the row sum is deferred.
//  * O^T = V^T P^T: the probabilities of a 32-key step are already in the B-operand lanes if
//    the MFMA's k index is read as key 16 (k' / 4) + 4 (lane / 16) + k' % 4.  The A operand (V^T)
//    comes from the row-major V tile by two transposing reads (ds_read_b64_tr_b16), 4 keys each.
//  * Softmax and accumulation are fp32 with lazy rescaling of the running max as in the decode
//    kernel.  Scores keep the reference's bf16 rounding points (bf16 product, then bf16 product
//    with the scale), one packed bf16 convert per rounding: for N(0,1) inputs those roundings
//    move logits by ~1e-2, so dropping them would leave the 2e-2 parity band.
//  * The two waves of a SIMD run in step (one workgroup barrier per tile), so per tile the
//    matrix work, the score roundings, exponentials and converts, and the LDS operand latency
//    largely add up: of 655 us at 4 x 2048 queries behind 10240 tokens, a timing copy without the softmax
//    took 299, one without the products 385, one with neither (the loads alone) 216.  Orders in which one
//    wave of a SIMD multiplies while the other does its softmax were no gain (779 us with one barrier per
//    tile, 806 with one per phase): a wave alone issues a VALU instruction in about 5 cycles, two
//    together in 3.
#include <algorithm>
#include <initializer_list>

#include "decode_block.h"

namespace mi {
namespace {

constexpr int kGroup = 2;  // query heads per workgroup (a pair of one GQA group)
constexpr int kKTile = 64;                 // keys per KV tile
constexpr int kSpans = kKTile / 4;         // 1 KiB LDS spans (4 rows of 256 B) per K or V tile

// Shape of a workgroup.  kNt: 16-query MFMA column tiles per wave; kWavesPerHead: waves side by side on
// the queries of a head; kKeySplit: wave groups that take every kKeySplit-th KV tile of the same queries
// and merge their states at the end.
template <int kNtV, int kWavesPerHeadV, int kKeySplitV>
struct Shape {
  static constexpr int kNt = kNtV, kWavesPerHead = kWavesPerHeadV, kKeySplit = kKeySplitV;
  static constexpr int kQPerWave = 16 * kNt;
  static constexpr int kQTile = kQPerWave * kWavesPerHead;       // queries per head per workgroup
  static constexpr int kGroupWaves = kGroup * kWavesPerHead;     // waves that share a KV tile
  static constexpr int kThreads = 64 * kGroupWaves * kKeySplit;
  static constexpr int kTileBytes = kKTile * 256;                // one K or V tile
  static constexpr int kLdsBytes = 4 * kTileBytes * kKeySplit;   // K and V, double-buffered, per wave group
  static constexpr int kSpansPerWave = kSpans / kGroupWaves;
  static_assert(kSpans % kGroupWaves == 0, "every wave moves the same number of spans");
  static_assert(kBlockSize % (4 * kSpansPerWave) == 0, "a wave's spans of a tile must lie in one pool block");
};
using Wide = Shape<2, 4, 1>;       // 128 queries, 8 waves
using Half = Shape<2, 2, 1>;       // 64 queries, 4 waves: two workgroups a CU, not in step
using HalfSplit = Shape<2, 2, 2>;  // 64 queries, 8 waves, the keys in two halves
using Narrow = Shape<1, 2, 2>;     // 32 queries, 8 waves, the keys in two halves
constexpr int kLdsPerGroup = 160 * 1024;
constexpr int kMaxHistoryBlocks = 16384;   // history table staged in LDS: 64 KiB at most (256k tokens)

struct PrefillArgs {
  uint16_t* out;
  int64_t out_row, out_tok;                 // elements
  const uint16_t* query;
  int64_t q_row, q_head, q_tok;
  const uint16_t* key;
  int64_t k_row, k_head, k_tok;
  const uint16_t* value;
  int64_t v_row, v_head, v_tok;
  uint16_t* key_pool;
  uint16_t* value_pool;
  int64_t num_blocks;
  const int64_t* history_blocks;
  int64_t history_stride;
  int32_t max_history_blocks;
  const int64_t* start_lens;
  const int64_t* chunk_lens;
  int64_t lens_stride;
  int32_t padded_len;
  int32_t group;   // query heads per KV head (G)
  int32_t pairs;   // workgroups per KV head: ceil(G / 2)
  float scale;
  int32_t tiles;   // query tiles per row: ceil(padded_len / kQTile)
  int32_t batch;   // rows
  int32_t groups;  // workgroups of these rows: tiles x num_kv_heads x pairs x batch
  int32_t round_pairs;  // (row, head pair) units per dispatch round of one workgroup queue
  // Decode rows (a mixed step's single new tokens, padded_len 1): start_lens holds each row's
  // context length including its token, so the history is the context minus one and a row with
  // context 0 is padding; the token's K/V row is appended to pool slot slot_mapping[b] (skipped
  // when outside the pool) by the workgroup of the first head pair of each KV head.
  int32_t decode_rows;
  const int64_t* slot_mapping;
  int64_t slot_stride;
  // Decode rows only: one workgroup per (row, KV head) attends them block by block (decode_row) instead
  // of as one-query tiles.
  int32_t stripes;
  // Ragged chunk rows (a mixed step's chunks packed back to back): when set, the len_b real tokens
  // of row b are flat tokens row_first[b] .. row_first[b] + len_b - 1 of query / key / value / out
  // (the token strides apply, the row strides are unused; row_first[b] is clamped to
  // [0, row_tokens - len_b]), and padding positions are neither read nor written.
  const int64_t* row_first;
  int64_t row_tokens;
};

// The reference's scores: bf16(bf16(q . k) * scale) (src/mini_infra/model/qwen3.py:243), in place.
__device__ __forceinline__ void reference_scores(f32x4& v, float scale) {
#pragma unroll
  for (int i = 0; i < 4; ++i) v[i] = round_bf16(round_bf16(v[i]) * scale);
}

// One 16-byte-per-lane load straight into LDS, from a uniform base and a byte offset per lane: lane i
// writes bytes [16 i, 16 i + 16) of the 1 KiB span at LDS address lds (wave-uniform, passed in M0; one wait state between the M0 write
// and the load).  Issued by inline assembly: the compiler's own form ties every later LDS read to
// the completion of all such loads (it cannot tell the two tile buffers apart), which would wait
// for tile t + 1 before reading tile t.  The compiler does not see these loads, so the kernel waits
// for them itself (vmcnt(0) before each tile barrier).  The LDS address goes in through an M0
// operand constraint, so the compiler writes M0 itself and knows its value across the asm.
__device__ __forceinline__ void dma16(const void* base, uint32_t off, uint32_t lds) {
  asm volatile("s_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(off), "s"(base), "{m0}"(lds) : "memory");
}

// A decode row of a mixed step (its single new token) by one workgroup of kStripes wavefronts per KV head,
// with the arithmetic of the decode kernels: stripe v attends blocks v, v + kStripes, ... of the history
// and the token, whose K and V rows (not yet in the pool, and appended here) are put in place of what its
// position's slot held, with zeros after them: the rest of that block was never part of the row, and an infinity or
// NaN among it would survive the product with a weight of zero.  As a one-query tile a row took 2 us per 64 keys, and the longest decode context
// was the longest chain of the launch.
constexpr int kRowDepth = 3;                             // blocks of a stripe in registers
constexpr int kRowStageElems = kBlockSize * kKStageRow;  // a wavefront's K staging; its output rows overlay it
constexpr int kRowMaxBlocks = 64 * kStripes - 1;         // a lane holds one block id; one more for the token
constexpr int kRowMaxGroup = 8;
template <int kKvHeads>
__device__ __forceinline__ void decode_row(const PrefillArgs& a, const int unit, unsigned char* smem) {
  constexpr int kRowElems = kKvHeads * kHeadDim;
  constexpr int kBlockElems = kBlockSize * kRowElems;
  static_assert(kRowMaxGroup * kHeadDim * sizeof(float) <= kRowStageElems * sizeof(uint16_t), "rows fit the staging");
  uint16_t* s_kst = reinterpret_cast<uint16_t*>(smem);                                                  // [kStripes]
  float* s_ml = reinterpret_cast<float*>(smem + kStripes * kRowStageElems * sizeof(uint16_t));          // [kStripes][8][2]
  const int b = unit / kKvHeads;
  const int g = (unit + b) % kKvHeads;  // every XCD gets every head in turn
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  const int dl = lane & 15, r = lane >> 4;
  int64_t id = a.history_blocks[b * a.history_stride + min(w + kStripes * lane, a.max_history_blocks - 1)];
  const int64_t ctx = a.start_lens[b * a.lens_stride];
  const u32x4 k_new = *reinterpret_cast<const u32x4*>(a.key + b * a.k_row + g * a.k_head + 8 * dl);
  const u32x4 v_new = *reinterpret_cast<const u32x4*>(a.value + b * a.v_row + g * a.v_head + 8 * dl);
  bf16x8 qf[4];
#pragma unroll
  for (int ks = 0; ks < 4; ++ks)
    qf[ks] = dl < a.group ? *reinterpret_cast<const bf16x8*>(a.query + b * a.q_row + (g * a.group + dl) * a.q_head +
                                                             32 * ks + 8 * r)
                          : bf16x8{};
  uint16_t* out_b = a.out + b * a.out_row + g * a.group * kHeadDim;
  if (ctx <= 0) {  // a padding row (uniform)
    if (threadIdx.x < a.group * 16) *reinterpret_cast<uint4*>(out_b + 8 * threadIdx.x) = uint4{0, 0, 0, 0};
    return;
  }
  const int nh = static_cast<int>(min(ctx - 1, static_cast<int64_t>(a.max_history_blocks) * kBlockSize));
  const int nblk = nh / kBlockSize + 1;  // the last one holds the token, at position nh
  const int cnt = nblk > w ? (nblk - 1 - w) / kStripes + 1 : 0;
  if (id < 0 || id >= a.num_blocks) id = 0;
  const uint32_t id_lo = static_cast<uint32_t>(id);  // the pool has fewer than 2^31 blocks
  if (threadIdx.x < 32) {  // append the token's K and V rows of KV head g
    const int64_t slot = a.slot_mapping[b * a.slot_stride];
    if (slot >= 0 && slot < a.num_blocks * kBlockSize) {
      uint16_t* pool = threadIdx.x < 16 ? a.key_pool : a.value_pool;
      *reinterpret_cast<u32x4*>(pool + (slot * kKvHeads + g) * kHeadDim + 8 * dl) = threadIdx.x < 16 ? k_new : v_new;
    }
  }
  const uint32_t k_off = 2u * (r * kRowElems + g * kHeadDim + 8 * dl);
  const uint32_t v_off = 2u * (4 * r * kRowElems + g * kHeadDim + 8 * dl);
  u32x4 kbuf[kRowDepth][4], vbuf[kRowDepth][4];
  auto issue = [&](int ring, int i) {
    const int64_t base = static_cast<int64_t>(__builtin_amdgcn_readlane(id_lo, i)) * kBlockElems;
    const char* kp = reinterpret_cast<const char*>(a.key_pool + base);
    const char* vp = reinterpret_cast<const char*>(a.value_pool + base);
#pragma unroll
    for (int t = 0; t < 4; ++t) kbuf[ring][t] = load_vec<true>(reinterpret_cast<const u32x4*>(kp + t * 8 * kRowElems + k_off));
#pragma unroll
    for (int t = 0; t < 4; ++t) vbuf[ring][t] = load_vec<true>(reinterpret_cast<const u32x4*>(vp + t * 2 * kRowElems + v_off));
  };
#pragma unroll
  for (int s = 0; s < kRowDepth - 1; ++s)
    if (s < cnt) issue(s, s);  // wave-uniform
  MfmaState ms;
  ms.m = -INFINITY;
  ms.l = 0.0f;
#pragma unroll
  for (int t = 0; t < 8; ++t) ms.o[t] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  for (int i0 = 0; i0 < cnt; i0 += kRowDepth) {
#pragma unroll
    for (int s = 0; s < kRowDepth; ++s) {
      const int i = i0 + s;
      if (i >= cnt) break;  // wave-uniform
      if (i + kRowDepth - 1 < cnt) issue((s + kRowDepth - 1) % kRowDepth, i + kRowDepth - 1);
      if (w + kStripes * i == nblk - 1) {
        const int t = nh % kBlockSize;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          kbuf[s][e] = 4 * e + r == t ? k_new : kbuf[s][e];
          vbuf[s][e] = 4 * r + e < t ? vbuf[s][e] : 4 * r + e == t ? v_new : u32x4{};
        }
      }
      attend_block_mfma(ms, qf, kbuf[s], vbuf[s], s_kst + w * kRowStageElems, a.scale, (w + kStripes * i) * kBlockSize,
                        nh + 1, lane);
    }
  }
  // Lane: heads 4 r + i, dims 8 dl .. +8; head j's max and sum live in lane j.
  const float lsum = xsum32_f32(xsum16_f32(ms.l));
  float* rows = reinterpret_cast<float*>(s_kst + w * kRowStageElems);  // [group][128]
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int j = 4 * r + i;
    const float Lj = __shfl(lsum, j);
    const float Mj = __shfl(ms.m, j);
    if (j >= a.group) continue;
    float4* dst = reinterpret_cast<float4*>(rows + j * kHeadDim + 8 * dl);
    dst[0] = make_float4(ms.o[0][i], ms.o[1][i], ms.o[2][i], ms.o[3][i]);
    dst[1] = make_float4(ms.o[4][i], ms.o[5][i], ms.o[6][i], ms.o[7][i]);
    if (dl == 0) *reinterpret_cast<float2*>(s_ml + (w * kRowMaxGroup + j) * 2) = make_float2(Mj, Lj);
  }
  __syncthreads();
  if (threadIdx.x < a.group * 16) {
    const int h = threadIdx.x >> 4, dm = threadIdx.x & 15;
    StripeMerge sm;
#pragma unroll
    for (int v = 0; v < kStripes; ++v) {
      const float4* src = reinterpret_cast<const float4*>(reinterpret_cast<const float*>(s_kst + v * kRowStageElems) +
                                                          h * kHeadDim + 8 * dm);
      sm.m[v] = s_ml[(v * kRowMaxGroup + h) * 2];
      sm.l[v] = s_ml[(v * kRowMaxGroup + h) * 2 + 1];
      sm.x[v] = src[0];
      sm.y[v] = src[1];
    }
    sm.store(out_b + h * kHeadDim + 8 * dm);
  }
}

// One launch serves up to two sets of rows (a mixed step's chunk rows and its decode rows): the
// first a0.groups workgroups take a0, the next a1.groups a1; the last z.groups write zero rows.
template <int kKvHeads, typename S>
__global__ __launch_bounds__(S::kThreads, 2) void chunked_prefill_kernel(const PrefillArgs a0, const PrefillArgs a1,
                                                                   const ZeroRows z) {
  constexpr int kNt = S::kNt, kQPerWave = S::kQPerWave, kQTile = S::kQTile, kThreads = S::kThreads;
  constexpr int kKeySplit = S::kKeySplit, kSpansPerWave = S::kSpansPerWave;
  constexpr uint32_t kTileBytes = S::kTileBytes;
  // Dynamic LDS.  Per wave group two K tiles, then two V tiles: row-major, 256-byte rows, 16-byte chunk
  // c of row r stored at chunk c ^ (r % 16).  Then the history block ids of this row, [ceil(nh / 16)].
  extern __shared__ __align__(1024) unsigned char s_raw[];
  int* s_hblk = reinterpret_cast<int*>(s_raw + S::kLdsBytes);

  if (static_cast<int>(blockIdx.x) >= a0.groups + a1.groups) {  // uniform
    zero_uncovered_rows(z, static_cast<int>(blockIdx.x) - a0.groups - a1.groups, kThreads);
    return;
  }
  const bool second = static_cast<int>(blockIdx.x) >= a0.groups;  // uniform
  if constexpr (kThreads == 64 * kStripes) {
    if (second && a1.stripes) {  // uniform
      decode_row<kKvHeads>(a1, static_cast<int>(blockIdx.x) - a0.groups, s_raw);
      return;
    }
  }
  const PrefillArgs a = second ? a1 : a0;

  // Workgroup -> (row b, head pair hp, query tile qt).  Consecutive workgroup ids go round-robin to
  // the kXcds XCDs, each with its own L2, and each XCD starts its ids in order on whichever CU
  // frees first.  When the pair count is a multiple of kXcds, id L runs on XCD L % kXcds and takes
  // place L / kXcds in the queue of that XCD's own pairs, so the query tiles of one (row, head
  // pair) -- which stream the same K/V tiles -- share an L2; otherwise one queue holds every pair.
  // A queue is cut into rounds of round_pairs pairs (as many as its CUs hold with all their query
  // tiles at once), and inside a round the tiles go heaviest (latest) first, pair by pair: the CUs
  // that finish a round's light tiles first take the next round's heavy ones, so every CU ends up
  // with about the same number of key tiles under the causal mask.
  int b, hp, qt;
  {
    const int tiles = a.tiles;
    const int per_row = kKvHeads * a.pairs;
    const int pairs = per_row * a.batch;
    const int lin = static_cast<int>(blockIdx.x) - (second ? a0.groups : 0);
    const bool by_xcd = pairs % kXcds == 0;
    const int units = by_xcd ? pairs / kXcds : pairs;  // pairs in this queue
    const int slot = by_xcd ? lin / kXcds : lin;       // place in this queue
    const int round_idx = slot / (a.round_pairs * tiles);
    const int within = slot - round_idx * a.round_pairs * tiles;
    const int round_size = min(a.round_pairs, units - round_idx * a.round_pairs);
    const int rank = within / round_size;
    const int unit = round_idx * a.round_pairs + (within - rank * round_size);
    const int pair = by_xcd ? unit * kXcds + lin % kXcds : unit;
    hp = pair % per_row;
    b = pair / per_row;
    qt = tiles - 1 - rank;
  }
  const int q0 = qt * kQTile;
  const int L = a.padded_len;
  int64_t len64, start64;
  if (a.decode_rows) {
    const int64_t ctx = a.start_lens[b * a.lens_stride];
    len64 = ctx > 0 ? 1 : 0;
    start64 = ctx > 0 ? ctx - 1 : 0;
  } else {
    len64 = a.chunk_lens[b * a.lens_stride];
    start64 = a.start_lens[b * a.lens_stride];
  }
  len64 = len64 < 0 ? 0 : (len64 > L ? L : len64);
  const int pad = L - static_cast<int>(len64);
  start64 = start64 < 0 ? 0 : start64;
  // Element offset of padded position rpad of row b (its first stored token): position i >= rpad
  // of a tensor with row / token strides (r, t) is at base + (i - rpad) t.
  const bool ragged = a.row_first != nullptr;  // uniform
  if (ragged && len64 == 0) return;             // an empty ragged row stores nothing
  int64_t first = 0;
  if (ragged) {
    first = a.row_first[b];
    first = first < 0 ? 0 : (first > a.row_tokens - len64 ? a.row_tokens - len64 : first);
  }
  const int rpad = ragged ? pad : 0;
  const int64_t q_base = ragged ? first * a.q_tok : b * a.q_row;
  const int64_t k_base = ragged ? first * a.k_tok : b * a.k_row;
  const int64_t v_base = ragged ? first * a.v_tok : b * a.v_row;
  const int64_t o_base = ragged ? first * a.out_tok : b * a.out_row;
  const int64_t hist_cap = static_cast<int64_t>(a.max_history_blocks) * kBlockSize;
  const int nh = static_cast<int>(start64 < hist_cap ? start64 : hist_cap);

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);  // wave index, uniform: keeps edge-tile branches real
  const int wk = w / S::kGroupWaves;      // wave group (key split)
  const int wt = w % S::kGroupWaves;      // wave of the group
  const int hh = wt / S::kWavesPerHead;
  const int qs = wt % S::kWavesPerHead;
  const int g = hp / a.pairs;                    // KV head
  const int j0 = (hp - g * a.pairs) * kGroup;    // first head of the pair within the group
  const bool head_live = j0 + hh < a.group;      // wave-uniform: false for the spare half of an odd group
  const int h = g * a.group + min(j0 + hh, a.group - 1);
  const int ql = lane & 15;
  const int gq = lane >> 4;

  if (a.decode_rows && j0 == 0 && tid < 32 && len64 > 0) {  // append the token's K and V rows of KV head g
    const int64_t slot = a.slot_mapping[b * a.slot_stride];
    if (slot >= 0 && slot < a.num_blocks * kBlockSize) {
      const int piece = (tid & 15) * 8;
      const uint16_t* src = tid < 16 ? a.key + b * a.k_row + g * a.k_head : a.value + b * a.v_row + g * a.v_head;
      uint16_t* dst = (tid < 16 ? a.key_pool : a.value_pool) + (slot * kKvHeads + g) * kHeadDim;
      *reinterpret_cast<uint4*>(dst + piece) = *reinterpret_cast<const uint4*>(src + piece);
    }
  }

  uint16_t* out_b = a.out + o_base;  // padded position rpad
  if (q0 + kQTile <= pad) {  // the whole tile is padding: zero rows (a ragged row stores none)
    if (ragged) return;
    for (int c = tid; c < kQTile * kGroup * (kHeadDim / 8); c += kThreads) {
      const int qi = q0 + c / (kGroup * (kHeadDim / 8));
      const int rem = c % (kGroup * (kHeadDim / 8));
      const int jj = j0 + rem / (kHeadDim / 8);
      const int head = g * a.group + jj;
      if (qi < L && jj < a.group)
        *reinterpret_cast<uint4*>(out_b + qi * a.out_tok + head * kHeadDim + (rem % (kHeadDim / 8)) * 8) =
            uint4{0, 0, 0, 0};
    }
    return;
  }

  // ---- Q^T fragments (B operand): query column n = ql of n-tile nt, dims 32 ks + 8 gq .. +8
  bf16x8 qf[kNt][4];
  const int qw0 = q0 + kQPerWave * qs;  // first query of this wave
#pragma unroll
  for (int nt = 0; nt < kNt; ++nt) {
    const int qi = qw0 + 16 * nt + ql;
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) {
      uint4 v = uint4{0, 0, 0, 0};
      if (qi < L && qi >= rpad)
        v = *reinterpret_cast<const uint4*>(a.query + q_base + h * a.q_head + (qi - rpad) * a.q_tok + ks * 32 + gq * 8);
      qf[nt][ks] = __builtin_bit_cast(bf16x8, v);
    }
  }

  const int n_hist_tiles = (nh + kKTile - 1) / kKTile;
  const int c_lo = pad / kKTile;
  const int last_q = min(q0 + kQTile, L) - 1;
  const int c_hi = last_q / kKTile;
  const int n_tiles = n_hist_tiles + (c_hi - c_lo + 1);

  // ---- tile loads straight into LDS (global_load_lds_dwordx4: lane i of an instruction writes
  // bytes [16 i, 16 i + 16) of a 1 KiB LDS span).  A tile is kSpans such spans of 4 rows for K and
  // as many for V; wave wt of a group moves spans [kSpansPerWave wt, kSpansPerWave (wt + 1)) of each.  Lane i of
  // span m fetches row 4 m + i / 16, global chunk (i % 16) ^ (row % 16), so that the chunk lands at
  // its swizzled place: the 16 lanes of an MFMA operand read (16 rows, one logical chunk) then hit
  // 16 different chunk positions, i.e. all banks.  In a history tile a wave's spans lie in one pool
  // block, whose id comes from the history table the workgroup staged in LDS; the id for tile t + 1
  // is read while tile t - 1 is computed, so no tile waits for that read.  Chunk rows past L - 1
  // read row L - 1, and a ragged row's padding rows its first stored row (their keys are masked).
  const int nhb = (nh + kBlockSize - 1) / kBlockSize;
  for (int i = tid; i < nhb; i += kThreads) {
    const int64_t x = a.history_blocks[b * a.history_stride + i];
    s_hblk[i] = (x < 0 || x >= a.num_blocks) ? 0 : static_cast<int>(x);
  }
  constexpr int64_t kBlkElems = static_cast<int64_t>(kBlockSize) * kKvHeads * kHeadDim;
  const int drow = lane >> 4;
  const int dchunk = lane & 15;
  const uint16_t* k_rows = a.key + k_base + g * a.k_head;  // padded position rpad
  const uint16_t* v_rows = a.value + v_base + g * a.v_head;
  const uint32_t k_tok = static_cast<uint32_t>(a.k_tok);  // < 2^24, checked by the entry point
  const uint32_t v_tok = static_cast<uint32_t>(a.v_tok);
  typedef __attribute__((address_space(3))) void* lds_ptr_t;
  const int wave_blk = 4 * kSpansPerWave * wt / kBlockSize;  // pool block of this wave's rows within a tile
  const auto hist_slot = [&](const int t) { return min(t * (kKTile / kBlockSize) + wave_blk, max(nhb - 1, 0)); };
  // LDS byte addresses of this wave's first K and V span in buffer 0 (buffer 1 follows at + kTileBytes).
  unsigned char* tiles = s_raw + wk * 4 * kTileBytes;  // this wave group's
  const uint32_t k_lds0 = static_cast<uint32_t>(reinterpret_cast<uintptr_t>((lds_ptr_t)(tiles + kSpansPerWave * wt * 1024)));
  const uint32_t v_lds0 = k_lds0 + 2 * kTileBytes;

  // Byte offsets of the lane's pieces: from the pool block in a history tile, from the tile's first row in
  // a chunk tile that lies inside the row (63 rows at most: below 2^31, token strides being below 2^24).
  uint32_t hist_off[kSpansPerWave], k_off_in[kSpansPerWave], v_off_in[kSpansPerWave];
#pragma unroll
  for (int i = 0; i < kSpansPerWave; ++i) {
    const int r = 4 * (kSpansPerWave * wt + i) + drow;
    const uint32_t c16 = static_cast<uint32_t>((dchunk ^ (r & 15)) * 16);
    hist_off[i] = static_cast<uint32_t>(((r & 15) * kKvHeads + g) * kHeadDim) * 2 + c16;
    k_off_in[i] = 2 * r * k_tok + c16;
    v_off_in[i] = 2 * r * v_tok + c16;
  }
  // hblk: this wave's history block id for tile t (unused for chunk tiles).
  auto dma_tile = [&](const int t, const int buf, const int hblk) {
    const char *kbase, *vbase;
    uint32_t ko[kSpansPerWave], vo[kSpansPerWave];
    if (t < n_hist_tiles) {
      const int64_t at = __builtin_amdgcn_readfirstlane(hblk) * kBlkElems;
      kbase = reinterpret_cast<const char*>(a.key_pool + at);
      vbase = reinterpret_cast<const char*>(a.value_pool + at);
#pragma unroll
      for (int i = 0; i < kSpansPerWave; ++i) ko[i] = vo[i] = hist_off[i];
    } else {
      const int key0 = (c_lo + t - n_hist_tiles) * kKTile;
      const int row0 = min(max(key0, rpad), L - 1);  // the clamp of the tile's first row: below every row's
      kbase = reinterpret_cast<const char*>(k_rows + static_cast<int64_t>(row0 - rpad) * k_tok);
      vbase = reinterpret_cast<const char*>(v_rows + static_cast<int64_t>(row0 - rpad) * v_tok);
      if (key0 >= rpad && key0 + kKTile <= L) {
#pragma unroll
        for (int i = 0; i < kSpansPerWave; ++i) {
          ko[i] = k_off_in[i];
          vo[i] = v_off_in[i];
        }
      } else {
#pragma unroll
        for (int i = 0; i < kSpansPerWave; ++i) {
          const int r = 4 * (kSpansPerWave * wt + i) + drow;
          const uint32_t c16 = static_cast<uint32_t>((dchunk ^ (r & 15)) * 16);
          const uint32_t kc = static_cast<uint32_t>(min(max(key0 + r, rpad), L - 1) - row0);
          ko[i] = 2 * kc * k_tok + c16;
          vo[i] = 2 * kc * v_tok + c16;
        }
      }
    }
#pragma unroll
    for (int i = 0; i < kSpansPerWave; ++i) {
      dma16(kbase, ko[i], __builtin_amdgcn_readfirstlane(k_lds0 + buf * kTileBytes + i * 1024));
      dma16(vbase, vo[i], __builtin_amdgcn_readfirstlane(v_lds0 + buf * kTileBytes + i * 1024));
    }
  };
  // Per-lane LDS byte offsets of the MFMA operands.  K (A of S^T = K Q^T): row 16 mt + ql, global
  // chunk 4 ks + gq.  V (A of O^T = V^T P^T, by transposing 8-byte reads): lane L of a 16-lane group
  // addresses row k0 + L / 4, dims 16 dt + 4 (L % 4) .. + 3, and receives dim 16 dt + L of rows
  // k0 .. k0 + 3; k0 = 32 ks2 + 4 gq, then + 16, gives the 8 keys in the MFMA's k order.
  uint32_t k_off[4];
#pragma unroll
  for (int ks = 0; ks < 4; ++ks) k_off[ks] = ql * 256 + (((4 * ks + gq) ^ ql) & 15) * 16;
  const int vr = 4 * gq + (ql >> 2);
  uint32_t v_off[8];
#pragma unroll
  for (int dt = 0; dt < 8; ++dt) v_off[dt] = vr * 256 + (((2 * dt + ((ql >> 1) & 1)) ^ vr) & 15) * 16 + (ql & 1) * 8;

  // oacc[0..7]: O^T dims 16 dt + 4 gq + i; oacc[8]: the softmax row sums.  Tile 8 multiplies P^T by
  // a constant A with ones in rows 0, 4, 8, 12: its rows 0, 4, 8, 12 -- element 0 of every lane group
  // -- accumulate sum_k bf16(p_k) on the matrix cores instead of 32 VALU adds per tile, and the
  // lazy rescale of oacc covers them.
  f32x4 oacc[9][kNt];
#pragma unroll
  for (int dt = 0; dt < 9; ++dt)
#pragma unroll
    for (int nt = 0; nt < kNt; ++nt) oacc[dt][nt] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  const __bf16 one_or_zero = (ql & 3) == 0 ? static_cast<__bf16>(1.0f) : static_cast<__bf16>(0.0f);
  const bf16x8 ones_frag = {one_or_zero, one_or_zero, one_or_zero, one_or_zero,
                            one_or_zero, one_or_zero, one_or_zero, one_or_zero};
  float m_run[kNt];
#pragma unroll
  for (int nt = 0; nt < kNt; ++nt) m_run[nt] = -INFINITY;
  const float scale = a.scale;

  // The three parts of a tile's work.  sacc: scores of 64 keys x kQPerWave queries; pf: [nt][ks2]
  // probabilities as B operands.
  f32x4 sacc[4][kNt];
  bf16x8 pf[kNt][2];
  auto tile_scores = [&](const char* sKb) {
    // ---- S^T = K Q^T for 64 keys x 32 queries
#pragma unroll
    for (int mt = 0; mt < 4; ++mt)
#pragma unroll
      for (int nt = 0; nt < kNt; ++nt) sacc[mt][nt] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) {
#pragma unroll
      for (int mt = 0; mt < 4; ++mt) {
        const bf16x8 kf = *reinterpret_cast<const bf16x8*>(sKb + mt * 4096 + k_off[ks]);
#pragma unroll
        for (int nt = 0; nt < kNt; ++nt)
          sacc[mt][nt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf, qf[nt][ks], sacc[mt][nt], 0, 0, 0);
      }
    }
  };
  auto tile_softmax = [&](const int t) {
    // ---- scores, masks (uniform branch: only edge tiles need them)
    const bool is_hist = t < n_hist_tiles;
    const int key0 = is_hist ? t * kKTile : (c_lo + t - n_hist_tiles) * kKTile;
    bool need_mask;
    if (is_hist) {
      need_mask = key0 + kKTile > nh || qw0 < pad || qw0 + kQPerWave - 1 >= L;
    } else {
      need_mask = key0 + kKTile - 1 > qw0 || key0 < pad || qw0 < pad || qw0 + kQPerWave - 1 >= L;
    }
    // Scores rounded like the reference; log2(e) is applied inside the exp2 FMA below.
#pragma unroll
    for (int mt = 0; mt < 4; ++mt)
#pragma unroll
      for (int nt = 0; nt < kNt; ++nt) reference_scores(sacc[mt][nt], scale);
    if (__builtin_expect(__builtin_amdgcn_readfirstlane(static_cast<int>(need_mask)) != 0, 0)) {
      // Bitwise (not short-circuit) conditions keep the edge-tile path free of branches.
#pragma unroll
      for (int nt = 0; nt < kNt; ++nt) {
        const int qi = qw0 + 16 * nt + ql;
        const bool row_ok = (qi >= pad) & (qi < L);
        const int lo = is_hist ? 0 : pad;        // visible key range [lo, hi] of this query
        const int hi = is_hist ? nh - 1 : qi;
#pragma unroll
        for (int mt = 0; mt < 4; ++mt)
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const int kpos = key0 + mt * 16 + 4 * gq + i;
            const bool vis = row_ok & (kpos >= lo) & (kpos <= hi);
            sacc[mt][nt][i] = vis ? sacc[mt][nt][i] : -INFINITY;
          }
      }
    }

    // ---- online softmax per query column (lanes ql, ql+16, ql+32, ql+48 hold its 64 keys)
    // Lazy rescale: m_run (shared by the four lanes of a query column) only has to bound every
    // score to within kRescaleSlack, so each lane tests its own 16 scores and the cross-lane
    // column max is taken only on the rare tiles that raise m_run.
    constexpr float to_log2 = kLog2e;
    float mx[kNt];
#pragma unroll
    for (int nt = 0; nt < kNt; ++nt) {
      float v = -INFINITY;
#pragma unroll
      for (int mt = 0; mt < 4; ++mt)
#pragma unroll
        for (int i = 0; i < 4; ++i) v = fmaxf(v, sacc[mt][nt][i]);
      mx[nt] = v * to_log2;
    }
    bool grow = false;
#pragma unroll
    for (int nt = 0; nt < kNt; ++nt) grow = grow || mx[nt] > m_run[nt] + kRescaleSlack;
    if (__builtin_amdgcn_ballot_w64(grow) != 0) {
#pragma unroll
      for (int nt = 0; nt < kNt; ++nt) {
        mx[nt] = fmaxf(mx[nt], __shfl_xor(mx[nt], 16));
        mx[nt] = fmaxf(mx[nt], __shfl_xor(mx[nt], 32));
        const float mn = fmaxf(m_run[nt], mx[nt]);
        const float alpha = mn == -INFINITY ? 1.0f : __builtin_amdgcn_exp2f(m_run[nt] - mn);
        m_run[nt] = mn;
#pragma unroll
        for (int dt = 0; dt < 9; ++dt) oacc[dt][nt] *= alpha;
      }
    }
#pragma unroll
    for (int nt = 0; nt < kNt; ++nt) {
      const float ref = m_run[nt] == -INFINITY ? 0.0f : m_run[nt];
#pragma unroll
      for (int mt = 0; mt < 4; ++mt)
#pragma unroll
        for (int i = 0; i < 4; ++i) sacc[mt][nt][i] = __builtin_amdgcn_exp2f(__builtin_fmaf(sacc[mt][nt][i], to_log2, -ref));
#pragma unroll
      for (int ks2 = 0; ks2 < 2; ++ks2) {
        const f32x8 pv = {sacc[2 * ks2][nt][0], sacc[2 * ks2][nt][1], sacc[2 * ks2][nt][2], sacc[2 * ks2][nt][3],
                          sacc[2 * ks2 + 1][nt][0], sacc[2 * ks2 + 1][nt][1], sacc[2 * ks2 + 1][nt][2],
                          sacc[2 * ks2 + 1][nt][3]};
        pf[nt][ks2] = __builtin_convertvector(pv, bf16x8);
      }
    }
  };
  auto tile_values = [&](const char* sVb) {
    // ---- O^T += V^T P^T
#pragma unroll
    for (int ks2 = 0; ks2 < 2; ++ks2) {
#pragma unroll
      for (int dt = 0; dt < 8; ++dt) {
        typedef short s16x4 __attribute__((ext_vector_type(4)));
        typedef __attribute__((address_space(3))) s16x4* lds_s16x4;
        const s16x4 v0 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4)(sVb + 32 * ks2 * 256 + v_off[dt]));
        const s16x4 v1 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4)(sVb + (32 * ks2 + 16) * 256 + v_off[dt]));
        const bf16x8 vf = __builtin_bit_cast(bf16x8, __builtin_shufflevector(v0, v1, 0, 1, 2, 3, 4, 5, 6, 7));
#pragma unroll
        for (int nt = 0; nt < kNt; ++nt)
          oacc[dt][nt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf, pf[nt][ks2], oacc[dt][nt], 0, 0, 0);
      }
#pragma unroll
      for (int nt = 0; nt < kNt; ++nt)
        oacc[8][nt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ones_frag, pf[nt][ks2], oacc[8][nt], 0, 0, 0);
    }
  };
  const char* k_tiles = reinterpret_cast<const char*>(tiles);
  const char* v_tiles = k_tiles + 2 * kTileBytes;

  __syncthreads();  // s_hblk ready
  // Tile t + 1 moves into the other buffer while tile t is computed; each wave waits for its own
  // loads before the tile barrier, after which every wave's part is in place.
  if (wk < n_tiles) dma_tile(wk, 0, s_hblk[hist_slot(wk)]);  // wave group wk takes tiles wk, wk + kKeySplit, ...
  int hblk_next = s_hblk[hist_slot(wk + kKeySplit)];
  // s_waitcnt vmcnt(0) (expcnt and lgkmcnt unconstrained) as a real instruction, so that the
  // compiler also counts the Q fragment loads as complete and waits for nothing inside the loop.
  __builtin_amdgcn_s_waitcnt(0x0F70);
  __syncthreads();
  auto tile_step = [&](const int t, const int buf) {
    if (t + kKeySplit < n_tiles) dma_tile(t + kKeySplit, buf ^ 1, hblk_next);
    hblk_next = s_hblk[hist_slot(t + 2 * kKeySplit)];
    tile_scores(k_tiles + buf * kTileBytes);
    tile_softmax(t);
    tile_values(v_tiles + buf * kTileBytes);
  };
  // Every wave of the workgroup passes every barrier: the rounds are uniform, and a wave group without
  // a tile in the last round only waits.
  auto round_end = [&] {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
  };
  for (int t0 = 0; t0 < n_tiles; t0 += 2 * kKeySplit) {
    if (kKeySplit == 1 || t0 + wk < n_tiles) tile_step(t0 + wk, 0);
    round_end();
    if (t0 + kKeySplit < n_tiles) {
      if (kKeySplit == 1 || t0 + kKeySplit + wk < n_tiles) tile_step(t0 + kKeySplit + wk, 1);
      round_end();
    }
  }
  if constexpr (kKeySplit > 1) {
    // Join the wave groups' states: group 0's waves fold in the others' (log-sum-exp), which they leave
    // in LDS over the tiles (no longer read: the last round's barrier is behind every wave).
    constexpr int kStateFloats = 33 * kNt * 64;  // per wave: 8 x 4 accumulators and the row sum per column tile
    static_assert((kKeySplit - 1) * S::kGroupWaves * (kStateFloats + 64 * kNt) * 4 <= S::kLdsBytes, "the states fit the tiles");
    float* st = reinterpret_cast<float*>(s_raw) + ((wk > 0 ? wk - 1 : 0) * S::kGroupWaves + wt) * (kStateFloats + 64 * kNt) + lane;
    if (wk > 0) {
#pragma unroll
      for (int nt = 0; nt < kNt; ++nt) {
#pragma unroll
        for (int e = 0; e < 32; ++e) st[(33 * nt + e) * 64] = oacc[e >> 2][nt][e & 3];
        st[(33 * nt + 32) * 64] = oacc[8][nt][0];
        st[(33 * kNt + nt) * 64] = m_run[nt];
      }
    }
    __syncthreads();
    if (wk > 0) return;
#pragma unroll
    for (int k = 1; k < kKeySplit; ++k) {
      const float* other = st + (k - 1) * S::kGroupWaves * (kStateFloats + 64 * kNt);
#pragma unroll
      for (int nt = 0; nt < kNt; ++nt) {
        const float mo = other[(33 * kNt + nt) * 64];
        const float mn = fmaxf(m_run[nt], mo);
        const float e0 = m_run[nt] == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(m_run[nt] - mn);
        const float e1 = mo == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(mo - mn);
        m_run[nt] = mn;
#pragma unroll
        for (int e = 0; e < 32; ++e)
          oacc[e >> 2][nt][e & 3] = e0 * oacc[e >> 2][nt][e & 3] + e1 * other[(33 * nt + e) * 64];
        oacc[8][nt][0] = e0 * oacc[8][nt][0] + e1 * other[(33 * nt + 32) * 64];
      }
    }
  }

  // ---- normalise and write: lane holds query qw0 + 16 nt + ql, dims 16 dt + 4 gq + i
#pragma unroll
  for (int nt = 0; nt < kNt; ++nt) {
    const float lt = oacc[8][nt][0];
    const float inv = lt > 0.0f ? 1.0f / lt : 0.0f;
    const int qi = qw0 + 16 * nt + ql;
    if (qi >= L || qi < rpad || !head_live) continue;
    uint16_t* orow = out_b + (qi - rpad) * a.out_tok + h * kHeadDim + 4 * gq;
#pragma unroll
    for (int dt = 0; dt < 8; ++dt) {
      uint2 v;
      v.x = pack_bf16x2(oacc[dt][nt][0] * inv, oacc[dt][nt][1] * inv);
      v.y = pack_bf16x2(oacc[dt][nt][2] * inv, oacc[dt][nt][3] * inv);
      *reinterpret_cast<uint2*>(orow + dt * 16) = v;
    }
  }
}

}  // namespace
}  // namespace mi

namespace mi {
namespace {

// Checks shared by the entry points (sizes, head shape, strides, alignment).
int32_t check_common(const char* name, int32_t num_heads, int32_t num_kv_heads, int32_t head_dim, int32_t block_size,
                     int64_t num_blocks, std::initializer_list<int64_t> strides, std::initializer_list<const void*> tensors) {
  if (head_dim != kHeadDim || block_size != kBlockSize || num_kv_heads <= 0 || num_heads <= 0 ||
      num_heads % num_kv_heads != 0)
    return fail(MI_ERR_UNSUPPORTED,
                "%s: needs head_dim %d, block_size %d, num_heads a multiple of num_kv_heads (got head_dim %d, "
                "block_size %d, heads %d/%d)",
                name, kHeadDim, kBlockSize, head_dim, block_size, num_heads, num_kv_heads);
  if (num_kv_heads != 1 && num_kv_heads != 2 && num_kv_heads != 4 && num_kv_heads != 8)
    return fail(MI_ERR_UNSUPPORTED, "%s: num_kv_heads %d not in {1,2,4,8}", name, num_kv_heads);
  for (int64_t st : strides)
    if (st % 8 != 0) return fail(MI_ERR_UNSUPPORTED, "%s: strides must be multiples of 8", name);
  for (const void* t : tensors)
    if (t && !aligned16(t)) return fail(MI_ERR_UNSUPPORTED, "%s: tensors must be 16-byte aligned", name);
  if (num_blocks > 0x7fffffff) return fail(MI_ERR_UNSUPPORTED, "%s: pool too large", name);
  return MI_OK;
}

// Fills the row-independent fields; the caller sets the pointers and strides of its rows.
PrefillArgs rows_args(int32_t batch, int32_t padded_len, int32_t num_heads, int32_t num_kv_heads, float scale,
                      int q_tile) {
  PrefillArgs a{};
  a.batch = batch;
  a.padded_len = padded_len;
  a.group = num_heads / num_kv_heads;
  a.pairs = (a.group + kGroup - 1) / kGroup;
  a.scale = scale;
  a.tiles = (padded_len + q_tile - 1) / q_tile;
  const int64_t pairs = static_cast<int64_t>(num_kv_heads) * a.pairs * batch;
  const int64_t groups = a.tiles * pairs;
  a.groups = groups > 0x3fffffff ? -1 : static_cast<int32_t>(groups);
  // Dispatch rounds: the queue of one XCD (or of the whole device when the pairs do not split
  // evenly over the XCDs) holds its CUs' worth of whole pairs per round.
  const bool by_xcd = pairs % kXcds == 0;
  const int64_t units = by_xcd ? pairs / kXcds : pairs;
  const int64_t cus = by_xcd ? device_cus() / kXcds : device_cus();
  const int64_t per_round = std::min(a.tiles > 0 ? cus / a.tiles : int64_t{1}, units);
  a.round_pairs = static_cast<int32_t>(std::max(per_round, int64_t{1}));
  return a;
}

enum class Form { kWide, kHalf, kHalfSplit, kNarrow };

// Whether a row's history table fits beside `tile_bytes` of K/V tiles in LDS.
bool table_fits(int tile_bytes, int32_t max_history_blocks) {
  return tile_bytes + static_cast<int64_t>(sizeof(int)) * max_history_blocks <= kLdsPerGroup;
}

#ifndef MI_PREFILL_FORM
#define MI_PREFILL_FORM -1
#endif
// Which workgroup shape takes a launch of `batch` chunk rows: by the workgroups it would have in the narrow and the
// wide shape, and by whether its query tiles see about as many keys each (history tables next to the
// chunk's length) or the later ones more, so that light tiles fill the last round of a finer cut.
// Measured, us, wide / half / half split / narrow (16 query, 8 KV heads; rows x queries behind tokens of
// history, and the workgroups that decide):
//   narrow: one round of its workgroups (cus; 11/8 of that without much history)
//     1 x 60 behind 4000     16 narrow       147 / 115 /  85 /  57
//     3 x 300               240               20 /  16 /  17 /  13
//     1 x 1000              256               46 /  35 /  29 /  22
//     2 x 700               352               33 /  27 /  24 /  19
//   half: short rows without history
//     15 x 128              120 wide          17 /  12 /  14 /  17
//     64 x 128              512               38 /  31 /  47 /  58
//     40 x 256              640               54 /  40 /  62 /  79
//   half split: up to half of cus wide workgroups, one round of its own
//     3 x 450                96               28 /  21 /  19 /  20
//     16 x 128 behind 1000  128               49 /  37 /  35 /  44
//     1 x 2048 behind 2000  128              127 /  94 /  83 /  86
//   up to cus: wide with history, else half split for long rows, half for shorter ones
//     20 x 128 behind 2000  160               81 /  83 /  96 /  99
//     2 x 1792 behind 4000  224              179 / 186 / 186 / 233
//     3 x 700               144               36 /  30 /  26 /  30
//     1 x 4096              256              128 / 103 /  94 / 117
//     5 x 640               200               34 /  31 /  33 /  38
//   half: a second wide round at most 9/16 full (400)
//     3 x 1408 behind 6000  264              370 / 320 / 332 / 380
//     3 x 2048              384               88 /  81 /  97 / 106
//     25 x 256 behind 2000  400              165 / 162 / 194 / 235
//   wide beyond
//     4 x 1664              416               66 /  82 /  81 / 105
//     4 x 1900 behind 1000  480              142 / 163 / 165 / 213
//     4 x 2048 behind 10240 512              729 / 750 / 801 / 1025
Form form_for(int32_t batch, int32_t padded_len, int32_t num_heads, int32_t num_kv_heads, int32_t max_history_blocks) {
  if (MI_PREFILL_FORM >= 0) return static_cast<Form>(MI_PREFILL_FORM);
  static_assert(Narrow::kLdsBytes == HalfSplit::kLdsBytes, "one limit");
  const int64_t cus = device_cus();
  const int64_t pairs = static_cast<int64_t>(num_kv_heads) * ((num_heads / num_kv_heads + kGroup - 1) / kGroup) * batch;
  const int64_t wide = pairs * ((padded_len + Wide::kQTile - 1) / Wide::kQTile);
  const int64_t narrow = pairs * ((padded_len + Narrow::kQTile - 1) / Narrow::kQTile);
  const int64_t history = static_cast<int64_t>(max_history_blocks) * kBlockSize;
  const bool split_fits = table_fits(Narrow::kLdsBytes, max_history_blocks);
  if (split_fits && 8 * narrow <= (2 * history >= padded_len ? 8 : 11) * cus) return Form::kNarrow;
  if (history == 0 && padded_len <= 256) return Form::kHalf;
  if (2 * wide <= cus) return split_fits ? Form::kHalfSplit : Form::kHalf;
  if (wide <= cus && history >= padded_len) return Form::kWide;
  if (wide <= cus) return padded_len > 640 && split_fits ? Form::kHalfSplit : Form::kHalf;
  return 16 * wide <= 25 * cus ? Form::kHalf : Form::kWide;
}

int q_tile_of(Form f) {
  return f == Form::kWide ? Wide::kQTile : f == Form::kNarrow ? Narrow::kQTile : Half::kQTile;
}

template <int kKvHeads, typename S>
int32_t launch_shape(const char* name, const PrefillArgs& a0, const PrefillArgs& a1, const ZeroRows& z, int groups,
                     int32_t max_history_blocks, hipStream_t s) {
  if (const int32_t rc = allow_lds<&chunked_prefill_kernel<kKvHeads, S>>(kLdsPerGroup, name)) return rc;
  const size_t lds = S::kLdsBytes + sizeof(int) * static_cast<size_t>(max_history_blocks > 0 ? max_history_blocks : 1);
  chunked_prefill_kernel<kKvHeads, S><<<groups, S::kThreads, lds, s>>>(a0, a1, z);
  return check_launch(name);
}

template <typename S>
int32_t launch_rows(const char* name, const PrefillArgs& a0, const PrefillArgs& a1, ZeroRows z, int32_t num_kv_heads,
                    int32_t max_history_blocks, void* stream) {
  z.groups = static_cast<int32_t>((z.tokens + S::kThreads - 1) / S::kThreads);
  if (a0.groups < 0 || a1.groups < 0 || static_cast<int64_t>(a0.groups) + a1.groups + z.groups > 0x3fffffff)
    return fail(MI_ERR_UNSUPPORTED, "%s: too many workgroups", name);
  if (max_history_blocks > kMaxHistoryBlocks)
    return fail(MI_ERR_UNSUPPORTED, "%s: history of %d blocks exceeds %d", name, max_history_blocks, kMaxHistoryBlocks);
  const int groups = a0.groups + a1.groups + z.groups;
  if (groups == 0) return ok();
  hipStream_t s = as_stream(stream);
  switch (num_kv_heads) {
    case 1: return launch_shape<1, S>(name, a0, a1, z, groups, max_history_blocks, s);
    case 2: return launch_shape<2, S>(name, a0, a1, z, groups, max_history_blocks, s);
    case 4: return launch_shape<4, S>(name, a0, a1, z, groups, max_history_blocks, s);
    default: return launch_shape<8, S>(name, a0, a1, z, groups, max_history_blocks, s);
  }
}

int32_t launch_form(Form form, const char* name, const PrefillArgs& a0, const PrefillArgs& a1, const ZeroRows& z,
                    int32_t num_kv_heads, int32_t max_history_blocks, void* stream) {
  switch (form) {
    case Form::kWide: return launch_rows<Wide>(name, a0, a1, z, num_kv_heads, max_history_blocks, stream);
    case Form::kHalf: return launch_rows<Half>(name, a0, a1, z, num_kv_heads, max_history_blocks, stream);
    case Form::kHalfSplit: return launch_rows<HalfSplit>(name, a0, a1, z, num_kv_heads, max_history_blocks, stream);
    default: return launch_rows<Narrow>(name, a0, a1, z, num_kv_heads, max_history_blocks, stream);
  }
}

}  // namespace
}  // namespace mi

extern "C" int32_t mi_chunked_prefill_attention(
    void* out, int64_t out_row_stride, int64_t out_tok_stride, const void* query, int64_t query_row_stride,
    int64_t query_head_stride, int64_t query_tok_stride, const void* key, int64_t key_row_stride,
    int64_t key_head_stride, int64_t key_tok_stride, const void* value, int64_t value_row_stride,
    int64_t value_head_stride, int64_t value_tok_stride, const void* key_pool, const void* value_pool,
    int64_t num_blocks, const int64_t* history_blocks, int64_t history_stride, int32_t max_history_blocks,
    const int64_t* start_lens, const int64_t* chunk_lens, int64_t lens_stride, int32_t batch, int32_t padded_len,
    int32_t num_heads, int32_t num_kv_heads, int32_t head_dim, int32_t block_size, float scale, void* stream) {
  using namespace mi;
  const char* name = "mi_chunked_prefill_attention";
  if (batch < 0 || padded_len < 0 || max_history_blocks < 0 || num_blocks < 0)
    return fail(MI_ERR_INVALID_ARGUMENT, "%s: negative size", name);
  if (batch == 0 || padded_len == 0) return ok();
  if (const int32_t rc = reject_empty_pool(name, num_blocks, max_history_blocks > 0)) return rc;
  if (!out || !query || !key || !value || !start_lens || !chunk_lens ||
      (max_history_blocks > 0 && (!history_blocks || !key_pool || !value_pool)))
    return fail(MI_ERR_INVALID_ARGUMENT, "%s: null pointer argument", name);
  int32_t rc = check_common(name, num_heads, num_kv_heads, head_dim, block_size, num_blocks,
                            {out_row_stride, out_tok_stride, query_row_stride, query_head_stride, query_tok_stride,
                             key_row_stride, key_head_stride, key_tok_stride, value_row_stride, value_head_stride,
                             value_tok_stride},
                            {out, query, key, value, max_history_blocks > 0 ? key_pool : nullptr,
                             max_history_blocks > 0 ? value_pool : nullptr});
  if (rc != MI_OK) return rc;
  if (max_history_blocks > 0 && history_stride < max_history_blocks)
    return fail(MI_ERR_INVALID_ARGUMENT, "%s: history_stride < max_history_blocks", name);
  if (lens_stride <= 0) return fail(MI_ERR_INVALID_ARGUMENT, "%s: lens_stride must be > 0", name);
  if (key_tok_stride < 0 || key_tok_stride >= (1 << 24) || value_tok_stride < 0 || value_tok_stride >= (1 << 24))
    return fail(MI_ERR_UNSUPPORTED, "%s: key/value token strides must be in [0, 2^24)", name);
  if (batch > 65535) return fail(MI_ERR_UNSUPPORTED, "%s: batch > 65535", name);

  const Form form = form_for(batch, padded_len, num_heads, num_kv_heads, max_history_blocks);
  PrefillArgs a = rows_args(batch, padded_len, num_heads, num_kv_heads, scale, q_tile_of(form));
  a.out = static_cast<uint16_t*>(out);
  a.out_row = out_row_stride;
  a.out_tok = out_tok_stride;
  a.query = static_cast<const uint16_t*>(query);
  a.q_row = query_row_stride;
  a.q_head = query_head_stride;
  a.q_tok = query_tok_stride;
  a.key = static_cast<const uint16_t*>(key);
  a.k_row = key_row_stride;
  a.k_head = key_head_stride;
  a.k_tok = key_tok_stride;
  a.value = static_cast<const uint16_t*>(value);
  a.v_row = value_row_stride;
  a.v_head = value_head_stride;
  a.v_tok = value_tok_stride;
  a.key_pool = static_cast<uint16_t*>(const_cast<void*>(key_pool));
  a.value_pool = static_cast<uint16_t*>(const_cast<void*>(value_pool));
  a.num_blocks = num_blocks;
  a.history_blocks = history_blocks;
  a.history_stride = history_stride;
  a.max_history_blocks = max_history_blocks;
  a.start_lens = start_lens;
  a.chunk_lens = chunk_lens;
  a.lens_stride = lens_stride;
  return launch_form(form, name, a, PrefillArgs{}, ZeroRows{}, num_kv_heads, max_history_blocks, stream);
}

extern "C" int32_t mi_mixed_paged_attention(
    void* out, int64_t out_tok_stride, const void* query, int64_t query_tok_stride, int64_t query_head_stride,
    const void* key, int64_t key_tok_stride, int64_t key_head_stride, const void* value, int64_t value_tok_stride,
    int64_t value_head_stride, void* key_pool, void* value_pool, int64_t num_blocks, int32_t prefill_rows,
    int32_t prefill_width, int64_t chunk_tokens, const int64_t* chunk_first, const int64_t* history_blocks,
    int64_t history_stride, int32_t max_history_blocks, const int64_t* start_lens, const int64_t* chunk_lens,
    int64_t lens_stride, int32_t decode_rows, const int64_t* block_tables, int64_t block_table_stride,
    int32_t max_blocks, const int64_t* context_lens, int64_t context_lens_stride, const int64_t* slot_mapping,
    int64_t slot_stride, int32_t num_heads, int32_t num_kv_heads, int32_t head_dim, int32_t block_size, float scale,
    void* stream) {
  using namespace mi;
  const char* name = "mi_mixed_paged_attention";
  if (prefill_rows < 0 || prefill_width < 0 || decode_rows < 0 || max_history_blocks < 0 || max_blocks < 0 ||
      num_blocks < 0 || (chunk_first && chunk_tokens < 0))
    return fail(MI_ERR_INVALID_ARGUMENT, "%s: negative size", name);
  const bool chunks = prefill_rows > 0 && prefill_width > 0;
  const bool ragged = chunk_first && chunk_tokens > 0;  // writes a zero row for every uncovered token
  if (!chunks && decode_rows == 0 && !ragged) return ok();
  if (const int32_t rc = reject_empty_pool(name, num_blocks, (chunks && max_history_blocks > 0) ||
                                                                 (decode_rows > 0 && max_blocks > 0)))
    return rc;
  if (!out || !query || !key || !value || (chunks && (!start_lens || !chunk_lens)) ||
      (chunks && max_history_blocks > 0 && !history_blocks) ||
      (decode_rows > 0 && (!context_lens || !slot_mapping || (max_blocks > 0 && !block_tables))) ||
      ((decode_rows > 0 || max_history_blocks > 0) && (!key_pool || !value_pool)))
    return fail(MI_ERR_INVALID_ARGUMENT, "%s: null pointer argument", name);
  const bool pools = decode_rows > 0 || max_history_blocks > 0;
  int32_t rc = check_common(name, num_heads, num_kv_heads, head_dim, block_size, num_blocks,
                            {out_tok_stride, query_tok_stride, query_head_stride, key_tok_stride, key_head_stride,
                             value_tok_stride, value_head_stride},
                            {out, query, key, value, pools ? key_pool : nullptr, pools ? value_pool : nullptr});
  if (rc != MI_OK) return rc;
  if (chunks && max_history_blocks > 0 && history_stride < max_history_blocks)
    return fail(MI_ERR_INVALID_ARGUMENT, "%s: history_stride < max_history_blocks", name);
  if (decode_rows > 0 && max_blocks > 0 && block_table_stride < max_blocks)
    return fail(MI_ERR_INVALID_ARGUMENT, "%s: block_table_stride < max_blocks", name);
  if ((chunks && lens_stride <= 0) || (decode_rows > 0 && (context_lens_stride <= 0 || slot_stride <= 0)))
    return fail(MI_ERR_INVALID_ARGUMENT, "%s: lens, context_lens and slot strides must be > 0", name);
  if (key_tok_stride < 0 || key_tok_stride >= (1 << 24) || value_tok_stride < 0 || value_tok_stride >= (1 << 24))
    return fail(MI_ERR_UNSUPPORTED, "%s: key/value token strides must be in [0, 2^24)", name);
  if (prefill_rows > 65535 || decode_rows > 65535) return fail(MI_ERR_UNSUPPORTED, "%s: more than 65535 rows", name);

  // Chunk rows: tokens [0, P L), row b at token b L, or with chunk_first the ragged rows of tokens
  // [0, chunk_tokens).  Decode rows: the D tokens after them, one each.
  const int64_t n = chunk_first ? chunk_tokens : (chunks ? static_cast<int64_t>(prefill_rows) * prefill_width : 0);
  auto fill = [&](PrefillArgs& a, int64_t tok0, int64_t rows_tokens) {
    a.out = static_cast<uint16_t*>(out) + tok0 * out_tok_stride;
    a.out_row = rows_tokens * out_tok_stride;
    a.out_tok = out_tok_stride;
    a.query = static_cast<const uint16_t*>(query) + tok0 * query_tok_stride;
    a.q_row = rows_tokens * query_tok_stride;
    a.q_head = query_head_stride;
    a.q_tok = query_tok_stride;
    a.key = static_cast<const uint16_t*>(key) + tok0 * key_tok_stride;
    a.k_row = rows_tokens * key_tok_stride;
    a.k_head = key_head_stride;
    a.k_tok = key_tok_stride;
    a.value = static_cast<const uint16_t*>(value) + tok0 * value_tok_stride;
    a.v_row = rows_tokens * value_tok_stride;
    a.v_head = value_head_stride;
    a.v_tok = value_tok_stride;
    a.key_pool = static_cast<uint16_t*>(key_pool);
    a.value_pool = static_cast<uint16_t*>(value_pool);
    a.num_blocks = num_blocks;
  };
  PrefillArgs a0{}, a1{};
  // The chunk rows' shape is the one mi_chunked_prefill_attention gives them (with the same bits: the wide shape sums
  // in the half one's order).  Decode rows alone: the wide shape, two workgroups of which share a CU.
  Form form = chunks ? form_for(prefill_rows, prefill_width, num_heads, num_kv_heads, max_history_blocks) : Form::kWide;
  if (form == Form::kHalf && decode_rows > 0) form = Form::kWide;  // decode rows take eight wavefronts
  const int q_tile = q_tile_of(form);
  if (chunks) {
    a0 = rows_args(prefill_rows, prefill_width, num_heads, num_kv_heads, scale, q_tile);
    fill(a0, 0, prefill_width);
    a0.history_blocks = history_blocks;
    a0.history_stride = history_stride;
    a0.max_history_blocks = max_history_blocks;
    a0.start_lens = start_lens;
    a0.chunk_lens = chunk_lens;
    a0.lens_stride = lens_stride;
    a0.row_first = chunk_first;
    a0.row_tokens = chunk_tokens;
  }
  if (decode_rows > 0) {
    a1 = rows_args(decode_rows, 1, num_heads, num_kv_heads, scale, q_tile);
    fill(a1, n, 1);
    a1.history_blocks = block_tables;
    a1.history_stride = block_table_stride;
    a1.max_history_blocks = max_blocks;
    a1.start_lens = context_lens;
    a1.chunk_lens = context_lens;
    a1.lens_stride = context_lens_stride;
    a1.decode_rows = 1;
    a1.slot_mapping = slot_mapping;
    a1.slot_stride = slot_stride;
    // Block by block where the table has blocks and their ids fit a wavefront's lanes; otherwise one-query tiles.
    a1.stripes = max_blocks >= 1 && max_blocks <= kRowMaxBlocks && a1.group <= kRowMaxGroup;
    if (a1.stripes) a1.groups = decode_rows * num_kv_heads;
  }
  ZeroRows z{};
  if (ragged) {
    rc = zero_rows(z, name, out, out_tok_stride, num_heads * head_dim, chunk_first, chunk_lens, lens_stride,
                   chunks ? prefill_rows : 0, prefill_width, chunk_tokens);
    if (rc != MI_OK) return rc;
  }
  const int32_t chunk_hist = chunks ? max_history_blocks : 0;
  const int32_t decode_hist = decode_rows > 0 ? max_blocks : 0;
  if (q_tile != Wide::kQTile && !table_fits(Narrow::kLdsBytes, decode_hist)) {
    // Decode tables too long for the split shapes' LDS: those rows in a launch of their own, with the wide shape.
    if (decode_hist > kMaxHistoryBlocks)
      return fail(MI_ERR_UNSUPPORTED, "%s: history of %d blocks exceeds %d", name, decode_hist, kMaxHistoryBlocks);
    rc = launch_form(form, name, a0, PrefillArgs{}, z, num_kv_heads, chunk_hist, stream);
    if (rc != MI_OK) return rc;
    return launch_form(Form::kWide, name, PrefillArgs{}, a1, ZeroRows{}, num_kv_heads, decode_hist, stream);
  }
  return launch_form(form, name, a0, a1, z, num_kv_heads, std::max(chunk_hist, decode_hist), stream);
}
