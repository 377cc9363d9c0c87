// Kernel 3: paged GQA decode attention (one query token per sequence).
//
// Behaviour of the reference's paged decode branch: the pool gather of
// Qwen3Attention._apply_paged_kv_pool (src/mini_infra/model/qwen3.py:285-292), the context-length
// bias of Qwen3Model._build_paged_inputs (:513-528) and Qwen3Attention._attend with
// _repeat_key_value (:219-255, :147-156) -- computed straight from the pool, without
// materialising the padded history or the repeated K/V.
//
// Work decomposition (MI355X: 256 CUs in 8 XCDs, 64-lane wavefronts, bandwidth-bound):
//  * The work of one launch is the list of (sequence, pool block) pairs, sequences in order,
//    N blocks in all.  It is cut into `streams` contiguous ranges of N / streams blocks (+-1),
//    and workgroup (stream s, head group hg) streams range s for the kWaves KV heads of hg.
//    Every workgroup gets the same number of blocks whatever the context lengths, and the
//    head groups of one range run side by side (adjacent workgroup ids), so the 2 KiB pool
//    rows of a block are read by concurrent workgroups.  Wavefront w of a group serves KV
//    head g and all G query heads G g .. G g + G - 1 that share it (the GQA group; 2 for
//    Qwen3-0.6B, kernels compiled for G in {1, 2, 4, 5, 8}): every K/V byte is loaded exactly
//    once.
//  * Each workgroup first turns the context lengths into a prefix sum of blocks per sequence
//    in LDS (so a block index maps to its sequence by binary search); block ids of the next
//    64 blocks of the range are fetched one per lane, a window ahead, and broadcast with
//    readlane.
//  * Inside a wavefront, lane = 16 * row + dl.  Lane dl holds dims [8 dl, 8 dl + 8) of the
//    G queries; row r owns tokens 4 i + r (i = 0..3) of every 16-token block.  One
//    16-byte load per lane per i brings four 256-byte (token, head) rows per instruction.
//  * QK^T: bf16 v_dot2 on packed pairs, then a 16-lane DPP butterfly (quad_perm, half-row
//    mirror, row mirror) leaves the full dot product in every lane of the row.
//  * Each row keeps its own online-softmax state (running max m, sum l, fp32 accumulator
//    of G heads x 8 dims), so no cross-row traffic happens inside the block loop.  The max
//    is rescaled lazily: only when a new score exceeds the running max by more than
//    kRescaleSlack (log2 units) -- exact, since l and the accumulator share the same m.
//  * PV: probabilities of token pairs are packed to bf16 and v_perm regroups V so that one
//    v_dot2 covers two tokens of one dim.
//  * K/V of the next kDepth-1 blocks are in flight in registers while the current block
//    is computed (a register ring: the VGPR file is 512 KiB per CU, LDS is 160 KiB).  The
//    ring runs straight across sequence boundaries, so the memory pipeline never drains
//    inside a range.
//  * At the end of a sequence's segment the four rows merge (log-sum-exp).  A sequence whose
//    blocks all lie in one range writes its bf16 output directly.  A sequence cut by a range
//    boundary leaves (m, l, acc) partials: a range holds at most two cut sequences (its first
//    and its last), so the caller's workspace is 2 slots per range per head, whatever the
//    batch and context lengths.  A second, small kernel merges the cut sequences and writes
//    zero rows for empty contexts.  (Merging inside the first kernel needs device-scope
//    release/acquire fences, and on this GPU each such fence writes back and invalidates a
//    whole XCD L2: far more costly than a launch.)
#include <cstdlib>
#include <cstring>
#include <mutex>

#include "decode_block.h"

namespace mi {
namespace {

#ifndef MI_DECODE_DEPTH
#define MI_DECODE_DEPTH 2
#endif
#ifndef MI_DECODE_MAX_WAVES
#define MI_DECODE_MAX_WAVES 2
#endif
#ifndef MI_DECODE_NT_LOADS
#define MI_DECODE_NT_LOADS 1
#endif
#ifndef MI_DECODE_GROUPS_PER_CU
#define MI_DECODE_GROUPS_PER_CU 4
#endif
constexpr int kDepth = MI_DECODE_DEPTH;            // register ring depth (blocks in flight incl. current)
constexpr int kMaxWaves = MI_DECODE_MAX_WAVES;     // wavefronts (KV heads) per workgroup
constexpr bool kNtLoads = MI_DECODE_NT_LOADS != 0; // K/V stream with the non-temporal hint
constexpr int kGroupsPerCu = MI_DECODE_GROUPS_PER_CU;
#ifndef MI_DECODE_XCD_RUN
#define MI_DECODE_XCD_RUN 0
#endif
// Consecutive stream-kernel workgroups per XCD run (0: launch order, which deals a range's head
// groups to different XCDs).  Unlike the scatter and the gather, decode loses with runs: at batch
// 256 (Σctx 755,887, 28 layers, three repetitions) 461-462 µs per layer without, 476.6-478.0 with
// runs of 4, 8, 16 or 32; four KV heads per workgroup (MI_DECODE_MAX_WAVES=4) 523-526 µs.
constexpr int kXcdRun = MI_DECODE_XCD_RUN;
constexpr int kMaxBatchPerLaunch = 4096;           // sequences whose prefix sum one workgroup holds in LDS
constexpr int kMinBlocksPerStream = 16;            // small launches use fewer, longer ranges
constexpr int kWindow = 64;                        // block ids fetched per window, one per lane

static_assert(kDepth >= 2 && kDepth - 1 < kWindow, "the ring looks ahead less than one id window");

#ifndef MI_DECODE_MFMA_GROUP
#define MI_DECODE_MFMA_GROUP 4
#endif
// GQA groups from this size up use the matrix-core form of the stream kernel (at most 16 heads,
// the MFMA's column count); smaller groups (Qwen3-0.6B / 1.7B's 2, multi-head 1) use the
// dot-product form, whose v_dot2 + DPP row reduction needs no zero-padded columns.  Measured at batch 256
// (8 KV heads, Σctx 755,887, attention + merge), TB/s for groups 1 / 2 / 4 / 5 / 8:
// dot-product form 6.75 / 6.67 / 6.40 / 6.27 / 4.67 (its per-token arithmetic grows with the
// group); matrix-core form 6.75 / 6.71 / 6.56 / 6.51 / 6.35.  At group 2, interleaved in one
// process (8 x 20 launches each), the matrix-core form took 461.5 µs (median) against 463.3.
constexpr int kMfmaGroup = MI_DECODE_MFMA_GROUP;
struct DecodeArgs {
  uint16_t* out;
  int64_t out_row;                 // elements
  const uint16_t* query;
  int64_t q_row, q_head;           // elements
  const uint16_t* key_pool;
  const uint16_t* value_pool;
  int64_t num_blocks;
  const int64_t* block_tables;
  int64_t bt_stride;
  const int64_t* context_lens;
  int64_t ctx_stride;
  int32_t batch;                   // sequences of this launch
  int32_t max_blocks;
  int32_t streams;                 // block ranges; grid = streams x head groups
  int32_t part_blocks;             // parts kernel: table blocks of a part; 0: the stripe kernel
  int32_t splits;                  // parts per sequence, ceil(max_blocks / part_blocks); stripe kernel:
                                   // workgroups per (sequence, KV head) (1: no partials)
  float scale;                     // softmax scale (natural units)
  // Partials, [slots, heads, 128] and [slots, heads, 2] = (m, l) in log2 units.  Stream kernel: slots
  // 2 s and 2 s + 1 are range s's first (cut) and last sequence; parts kernel: b splits + part; stripe
  // kernel: b kStripes + stripe.
  float* ws_acc;
  float* ws_ml;
  // Fused form of the per-sequence kernel: raw q / k / v projection rows of the new tokens, the
  // q/k norm weights, cos / sin rows [batch, 128] and the slots of the new K/V rows.
  const uint16_t* q_raw;
  const uint16_t* k_raw;
  const uint16_t* v_raw;
  int64_t q_raw_row, k_raw_row, v_raw_row;  // elements
  const uint16_t* q_weight;
  const uint16_t* k_weight;
  const uint16_t* cos;
  const uint16_t* sin;
  const int64_t* slot_mapping;
  int64_t slot_stride;
  int64_t num_slots;
  float eps;
};

__device__ __forceinline__ float dpp_sum16(float x) {
  // Butterfly over the 16 lanes of a DPP row: xor 1, xor 2, 8-lane mirror, 16-lane mirror.
  x += __builtin_amdgcn_update_dpp(0.0f, x, 0xB1, 0xf, 0xf, false);   // quad_perm [1,0,3,2]
  x += __builtin_amdgcn_update_dpp(0.0f, x, 0x4E, 0xf, 0xf, false);   // quad_perm [2,3,0,1]
  x += __builtin_amdgcn_update_dpp(0.0f, x, 0x141, 0xf, 0xf, false);  // row_half_mirror
  x += __builtin_amdgcn_update_dpp(0.0f, x, 0x140, 0xf, 0xf, false);  // row_mirror
  return x;
}

__device__ __forceinline__ float dot8(const uint4 q, const u32x4 k) {
  // Elements are copied to scalars before the bit casts: a bit cast of an ext-vector
  // component expression (k.y) must not be used, it can read component 0.
  const uint32_t k0 = k[0], k1 = k[1], k2 = k[2], k3 = k[3];
  float d = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2, q.x), __builtin_bit_cast(bf16x2, k0), 0.0f, false);
  d = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2, q.y), __builtin_bit_cast(bf16x2, k1), d, false);
  d = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2, q.z), __builtin_bit_cast(bf16x2, k2), d, false);
  d = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2, q.w), __builtin_bit_cast(bf16x2, k3), d, false);
  return d;
}

__device__ __forceinline__ uint32_t pack_p(float lo, float hi) {
  return __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2){lo, hi}, bf16x2));
}

__device__ __forceinline__ float fdot2(uint32_t a, uint32_t b, float c) {
  return __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2, a), __builtin_bit_cast(bf16x2, b), c, false);
}

__device__ __forceinline__ int64_t context_of(const DecodeArgs& a, int b) {
  const int64_t n = a.context_lens[b * a.ctx_stride];
  return min(n, static_cast<int64_t>(a.max_blocks) * kBlockSize);
}

// Pool blocks of a context of n tokens (0 for an empty context).
__device__ __forceinline__ int blocks_of(int64_t n) {
  return n <= 0 ? 0 : static_cast<int>((n + kBlockSize - 1) / kBlockSize);
}

// The cut of N > 0 blocks into min(streams, N) ranges, none empty: range s starts at block
// s q + min(s, rem) (the first rem ranges hold q + 1 blocks, the rest q).  32-bit arithmetic: N < 2^31,
// checked by the entry point.
struct Ranges {
  int count, q, rem;
  __device__ __forceinline__ Ranges(int total, int streams) {
    count = max(min(streams, total), 1);
    q = total / count;
    rem = total - q * count;
  }
  __device__ __forceinline__ int begin(int s) const { return s * q + min(s, rem); }
  __device__ __forceinline__ int of(int x) const {  // the range holding block x
    const int wide = rem * (q + 1);                 // blocks of the first rem ranges
    return x < wide ? x / (q + 1) : rem + (x - wide) / q;
  }
};

// Exclusive prefix sums of the blocks per sequence into s_off[0..batch]; returns the total.
template <int kThreads>
__device__ int scan_blocks(const DecodeArgs& a, int* s_off, int* s_wave) {
  constexpr int kWavesPerGroup = kThreads / 64;
  static_assert(kThreads % 64 == 0, "whole wavefronts");
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  int carry = 0;
  for (int base = 0; base < a.batch; base += kThreads) {
    const int i = base + threadIdx.x;
    int v = i < a.batch ? blocks_of(context_of(a, i)) : 0;
    for (int d = 1; d < 64; d <<= 1) {
      const int y = __shfl_up(v, d);
      if (lane >= d) v += y;
    }
    if (lane == 63) s_wave[w] = v;
    __syncthreads();
    int prefix = 0, total = 0;
#pragma unroll
    for (int k = 0; k < kWavesPerGroup; ++k) {
      const int t = s_wave[k];
      prefix += k < w ? t : 0;
      total += t;
    }
    if (i < a.batch) s_off[i + 1] = carry + prefix + v;
    carry += total;
    __syncthreads();
  }
  if (threadIdx.x == 0) s_off[0] = 0;
  __syncthreads();
  return carry;
}

// Sequence of block x (x < total): the last b with s_off[b] <= x (empty sequences are skipped).
__device__ __forceinline__ int row_of(const int* s_off, int batch, int x) {
  int lo = 0, hi = batch;  // s_off[lo] <= x < s_off[hi]
  while (hi - lo > 1) {
    const int mid = (lo + hi) >> 1;
    if (s_off[mid] <= x) lo = mid; else hi = mid;
  }
  return lo;
}

// Softmax state of one lane row (tokens 4 i + r of every block) for the kG query heads of its KV
// head: running max m (log2 units), sum l and the fp32 accumulator of the lane's 8 dims.
template <int kG>
struct RowState {
  float m[kG], l[kG], acc[kG][8];
  __device__ __forceinline__ void init() {
#pragma unroll
    for (int h = 0; h < kG; ++h) {
      m[h] = -INFINITY;
      l[h] = 0.0f;
#pragma unroll
      for (int d = 0; d < 8; ++d) acc[h][d] = 0.0f;
    }
  }
};

// One 16-token block (first token tok_base of a context of n tokens) for lane row r: scores of
// tokens 4 i + r against the kG queries, lazy rescale, then P V.  Only a sequence's last block
// can reach past its context; full blocks skip the masking (uniform branch).
template <int kG>
__device__ __forceinline__ void attend_block(RowState<kG>& st, const uint4 (&q)[kG], const u32x4 (&kb)[4],
                                             const u32x4 (&vb)[4], float scale, int tok_base, int n, int r) {
  float s[kG][4];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int h = 0; h < kG; ++h) s[h][i] = score_log2(dpp_sum16(dot8(q[h], kb[i])), scale);
  if (tok_base + kBlockSize > n) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const bool valid = tok_base + 4 * i + r < n;
#pragma unroll
      for (int h = 0; h < kG; ++h) s[h][i] = valid ? s[h][i] : -INFINITY;
    }
  }
  float mb[kG];
  bool grow = false;
#pragma unroll
  for (int h = 0; h < kG; ++h) {
    mb[h] = fmaxf(fmaxf(s[h][0], s[h][1]), fmaxf(s[h][2], s[h][3]));
    grow = grow || mb[h] > st.m[h] + kRescaleSlack;
  }
  if (__builtin_amdgcn_ballot_w64(grow) != 0) {  // lazy rescale (wave-uniform branch)
#pragma unroll
    for (int h = 0; h < kG; ++h) {
      const float nm = fmaxf(st.m[h], mb[h]);
      const float al = (nm == -INFINITY) ? 1.0f : __builtin_amdgcn_exp2f(st.m[h] - nm);
      st.m[h] = nm;
      st.l[h] *= al;
#pragma unroll
      for (int d = 0; d < 8; ++d) st.acc[h][d] *= al;
    }
  }
  // exp2(-inf) = 0 covers masked tokens; a row with no valid token yet keeps m = -inf, so the
  // reference point falls back to 0 there to avoid -inf - -inf.
  uint32_t ph[kG][2];
#pragma unroll
  for (int h = 0; h < kG; ++h) {
    const float ref = st.m[h] == -INFINITY ? 0.0f : st.m[h];
    float p[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) p[i] = __builtin_amdgcn_exp2f(s[h][i] - ref);
    st.l[h] += (p[0] + p[1]) + (p[2] + p[3]);
    ph[h][0] = pack_p(p[0], p[1]);
    ph[h][1] = pack_p(p[2], p[3]);
  }
  // P V over token pairs (0,1) and (2,3): v_perm regroups V so that one v_dot2 covers two tokens
  // of one dim; the regrouped V serves every head of the group.
#pragma unroll
  for (int pr = 0; pr < 2; ++pr) {
    const u32x4 va = vb[2 * pr];
    const u32x4 vc = vb[2 * pr + 1];
    const uint32_t aw[4] = {va[0], va[1], va[2], va[3]};
    const uint32_t cw[4] = {vc[0], vc[1], vc[2], vc[3]};
#pragma unroll
    for (int w = 0; w < 4; ++w) {
      const uint32_t plo = __builtin_amdgcn_perm(cw[w], aw[w], 0x05040100u);  // (a.lo, c.lo)
      const uint32_t phi = __builtin_amdgcn_perm(cw[w], aw[w], 0x07060302u);  // (a.hi, c.hi)
#pragma unroll
      for (int h = 0; h < kG; ++h) {
        st.acc[h][2 * w] = fdot2(ph[h][pr], plo, st.acc[h][2 * w]);
        st.acc[h][2 * w + 1] = fdot2(ph[h][pr], phi, st.acc[h][2 * w + 1]);
      }
    }
  }
}

// Merges the four lane rows of a wavefront (log-sum-exp): afterwards every row holds, per head,
// the wavefront's max M, sum l and accumulator.
template <int kG>
__device__ __forceinline__ void merge_rows(RowState<kG>& st, float (&M)[kG]) {
#pragma unroll
  for (int h = 0; h < kG; ++h) {
    float mx = fmaxf(st.m[h], __shfl_xor(st.m[h], 16));
    mx = fmaxf(mx, __shfl_xor(mx, 32));
    M[h] = mx;
    const float wt = (st.m[h] == -INFINITY) ? 0.0f : __builtin_amdgcn_exp2f(st.m[h] - mx);
    st.l[h] *= wt;
    st.l[h] += __shfl_xor(st.l[h], 16);
    st.l[h] += __shfl_xor(st.l[h], 32);
#pragma unroll
    for (int d = 0; d < 8; ++d) {
      st.acc[h][d] *= wt;
      st.acc[h][d] += __shfl_xor(st.acc[h][d], 16);
      st.acc[h][d] += __shfl_xor(st.acc[h][d], 32);
    }
  }
}

template <int kKvHeads, int kWaves, int kG>
// Second bound: minimum wavefronts per SIMD, so that kGroupsPerCu workgroups fit on a CU
// (4 SIMDs per CU) and the whole grid is resident.
__global__ __launch_bounds__(64 * kWaves, (kGroupsPerCu * kWaves + 3) / 4) void paged_decode_kernel(const DecodeArgs a) {
  constexpr int kThreads = 64 * kWaves;
  constexpr int kRowElems = kKvHeads * kHeadDim;     // elements of one pool row (token)
  constexpr int kBlockElems = kBlockSize * kRowElems;
  constexpr int kHeadGroups = kKvHeads / kWaves;
  constexpr int kHeads = kKvHeads * kG;
  constexpr bool kMfma = kG >= kMfmaGroup;
  static_assert(kG <= 16, "at most 16 query heads per KV head");

  extern __shared__ int s_off[];                     // [batch + 1] block prefix sums
  __shared__ int s_wave[kWaves];
  __shared__ __align__(16) uint16_t s_kst[kMfma ? kWaves : 1][kMfma ? kBlockSize * kKStageRow : 8];
  const int total = scan_blocks<kThreads>(a, s_off, s_wave);
  int wg = blockIdx.x;
  if (kXcdRun > 0) {
    // Workgroups go round-robin to the XCDs: within each super-run of kXcds * kXcdRun workgroups,
    // those on XCD i take [i kXcdRun, (i + 1) kXcdRun) in order, so the head groups of a range share
    // an XCD; the partial tail keeps identity.
    constexpr int kSuper = kXcds * kXcdRun;
    const int n = a.streams * kHeadGroups;
    if (wg < n / kSuper * kSuper) {
      const int base = wg / kSuper * kSuper, r = wg - base;
      wg = base + (r % kXcds) * kXcdRun + r / kXcds;
    }
  }
  const int stream = wg / kHeadGroups;
  const int hg = wg - stream * kHeadGroups;
  const Ranges rg(total, a.streams);
  if (total == 0 || stream >= rg.count) return;
  const int lo = rg.begin(stream), hi = rg.begin(stream + 1);

  const int lane = threadIdx.x & 63;
  const int dl = lane & 15;
  const int r = lane >> 4;
  const int g = hg * kWaves + (threadIdx.x >> 6);
  const float scale = a.scale;
  // Lane offsets (elements) of its first K and V pieces inside a block, and the step between its
  // four pieces.  K (both forms) and V of the dot-product form: tokens 4 i + r, dims 8 dl .. +8;
  // V of the matrix-core form: token 4 r + i, dims 8 dl .. +8.
  const int k_off = r * kRowElems + g * kHeadDim + 8 * dl;
  const int v_off = kMfma ? 4 * r * kRowElems + g * kHeadDim + 8 * dl : k_off;
  constexpr int kKStep = 4 * kRowElems;
  constexpr int kVStep = kMfma ? kRowElems : 4 * kRowElems;

  // Block ids of window [base, base + 64), one per lane (indices past the range repeat its
  // last block; ids outside the pool read block 0).
  auto fetch_ids = [&](int base, uint32_t& id_lo, uint32_t& id_hi) {
    const int x = min(base + lane, hi - 1);
    const int b = row_of(s_off, a.batch, x);
    int64_t id = a.block_tables[b * a.bt_stride + (x - s_off[b])];
    if (id < 0 || id >= a.num_blocks) id = 0;
    id_lo = static_cast<uint32_t>(id);
    id_hi = static_cast<uint32_t>(static_cast<uint64_t>(id) >> 32);
  };
  int wbase = lo;
  uint32_t cur_lo, cur_hi, nxt_lo, nxt_hi;
  fetch_ids(wbase, cur_lo, cur_hi);
  fetch_ids(wbase + kWindow, nxt_lo, nxt_hi);

  u32x4 kbuf[kDepth][4], vbuf[kDepth][4];
  // Loads block y (clamped to the range) into ring slot `slot`; y never passes the next window.
  auto issue = [&](int slot, int y) {
    y = min(y, hi - 1);
    if (y >= wbase + kWindow) {  // wave-uniform: slide the window, fetch the one after
      wbase += kWindow;
      cur_lo = nxt_lo;
      cur_hi = nxt_hi;
      fetch_ids(wbase + kWindow, nxt_lo, nxt_hi);
    }
    const int j = y - wbase;
    const uint32_t blo = __builtin_amdgcn_readlane(cur_lo, j);
    const uint32_t bhi = __builtin_amdgcn_readlane(cur_hi, j);
    const int64_t base = static_cast<int64_t>((static_cast<uint64_t>(bhi) << 32) | blo) * kBlockElems;
    const uint16_t* kp = a.key_pool + base + k_off;
    const uint16_t* vp = a.value_pool + base + v_off;
#pragma unroll
    for (int i = 0; i < 4; ++i) kbuf[slot][i] = load_vec<kNtLoads>(reinterpret_cast<const u32x4*>(kp + i * kKStep));
#pragma unroll
    for (int i = 0; i < 4; ++i) vbuf[slot][i] = load_vec<kNtLoads>(reinterpret_cast<const u32x4*>(vp + i * kVStep));
  };
#pragma unroll
  for (int s = 0; s < kDepth - 1; ++s) issue(s, lo + s);  // ring slot of block x: (x - lo) % kDepth

  int b = row_of(s_off, a.batch, lo);
  int x = lo;
  while (x < hi) {
    const int row_lo = s_off[b], row_hi = s_off[b + 1];
    const int seg_end = min(hi, row_hi);
    const int n32 = static_cast<int>(context_of(a, b));  // contexts are bounded by max_blocks * 16 < 2^31
    const uint16_t* qp = a.query + b * a.q_row + (g * kG) * a.q_head;
    uint4 q[kMfma ? 1 : kG];
    bf16x8 qf[4];
    RowState<kMfma ? 1 : kG> st;
    MfmaState ms;
    if constexpr (kMfma) {  // Q^T fragments: head dl (zero past the group), dims 32 ks + 8 r .. +8
#pragma unroll
      for (int ks = 0; ks < 4; ++ks)
        qf[ks] = dl < kG ? *reinterpret_cast<const bf16x8*>(qp + dl * a.q_head + 32 * ks + 8 * r) : bf16x8{};
      ms.m = -INFINITY;
      ms.l = 0.0f;
#pragma unroll
      for (int t = 0; t < 8; ++t) ms.o[t] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    } else {
#pragma unroll
      for (int j = 0; j < kG; ++j) q[j] = *reinterpret_cast<const uint4*>(qp + j * a.q_head + 8 * dl);
      st.init();
    }

    const int seg_begin = x;
    for (int x0 = x - (x - lo) % kDepth; x0 < seg_end; x0 += kDepth) {
#pragma unroll
      for (int s = 0; s < kDepth; ++s) {
        const int xb = x0 + s;
        if (xb < seg_begin || xb >= seg_end) continue;  // wave-uniform
        issue((s + kDepth - 1) % kDepth, xb + kDepth - 1);
        const int tok_base = (xb - row_lo) * kBlockSize;
        if constexpr (kMfma)
          attend_block_mfma(ms, qf, kbuf[s], vbuf[s], s_kst[threadIdx.x >> 6], scale, tok_base, n32, lane);
        else
          attend_block<kG>(st, q, kbuf[s], vbuf[s], scale, tok_base, n32, r);
      }
    }
    x = seg_end;
    const bool whole = row_lo >= lo && row_hi <= hi;  // the whole sequence is in this range

    if constexpr (kMfma) {
      // Column sums, then each lane's heads 4 r + i (their m and sum live in lanes 4 r + i).
      float lsum = ms.l + __shfl_xor(ms.l, 16);
      lsum += __shfl_xor(lsum, 32);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int j = 4 * r + i;
        const float Lj = __shfl(lsum, j);
        const float Mj = __shfl(ms.m, j);
        if (j >= kG) continue;
        const int h = g * kG + j;
        float o[8];
#pragma unroll
        for (int t = 0; t < 8; ++t) o[t] = ms.o[t][i];
        if (whole) {
          store_bf16x8(a.out + b * a.out_row + h * kHeadDim + 8 * dl, o, 1.0f / Lj);
        } else {  // cut sequence: slot 0 if it began before this range (its first), else 1 (its last)
          const int64_t slot = (static_cast<int64_t>(stream) * 2 + (row_lo < lo ? 0 : 1)) * kHeads + h;
          float4* dst = reinterpret_cast<float4*>(a.ws_acc + slot * kHeadDim + 8 * dl);
          dst[0] = make_float4(o[0], o[1], o[2], o[3]);
          dst[1] = make_float4(o[4], o[5], o[6], o[7]);
          if (dl == 0) {
            a.ws_ml[slot * 2 + 0] = Mj;
            a.ws_ml[slot * 2 + 1] = Lj;
          }
        }
      }
      if (x < hi) {  // next non-empty sequence (uniform)
        while (s_off[b + 1] <= x) ++b;
      }
      continue;
    }

    float M[kMfma ? 1 : kG];
    merge_rows<kMfma ? 1 : kG>(st, M);
    // Row r writes query heads g kG + j for j = r, r + 4, ... (every row has all after the merge).
#pragma unroll
    for (int j = 0; j < (kMfma ? 0 : kG); ++j) {
      if ((j & 3) != r) continue;
      const int h = g * kG + j;
      if (whole) {
        store_bf16x8(a.out + b * a.out_row + h * kHeadDim + 8 * dl, st.acc[j], 1.0f / st.l[j]);
      } else {  // cut sequence: slot 0 if it began before this range (its first), else 1 (its last)
        const int64_t slot = (static_cast<int64_t>(stream) * 2 + (row_lo < lo ? 0 : 1)) * kHeads + h;
        float4* dst = reinterpret_cast<float4*>(a.ws_acc + slot * kHeadDim + 8 * dl);
        dst[0] = make_float4(st.acc[j][0], st.acc[j][1], st.acc[j][2], st.acc[j][3]);
        dst[1] = make_float4(st.acc[j][4], st.acc[j][5], st.acc[j][6], st.acc[j][7]);
        if (dl == 0) {
          a.ws_ml[slot * 2 + 0] = M[j];
          a.ws_ml[slot * 2 + 1] = st.l[j];
        }
      }
    }
    if (x < hi) {  // next non-empty sequence (uniform)
      while (s_off[b + 1] <= x) ++b;
    }
  }
}

// ---- Small launches.  Two forms share the prologue below; both spread long tables over more CUs than
// they have (sequence, KV head) pairs, because one CU takes in no more than 47-62 bytes/ns of K/V
// whatever the loads in flight (8192 tokens on one CU per KV head: 87-92 us with rings of 2 to 4, 8 or 16
// wavefronts), and both are chains of dependent memory round trips of 1.4-2 us each, so everything
// that depends on nothing (context, block ids, the projection rows and tables of the prologue) is
// loaded together and no load is issued for a block that is not used.
//  * stripes, tables of up to kStripeMaxBlocks blocks: a sequence always falls into kStripes stripes,
//    stripe v being blocks v, v + kStripes, ..., each attended by one wavefront with the stream
//    kernel's per-block arithmetic and merged in order.  One workgroup holds all stripes (and writes
//    the rows), or kStripeWaves each hold some and the merge launch joins them: the bits are the same.
//  * parts, longer tables or more pairs: contiguous ranges of the table, two blocks a step.
// Spreading is for launches whose workspace is their own: mi_paged_decode_attention keeps small launches whole
// (one workgroup per pair), the spread entry points cut them.
// Measured against the form before (the stripes of a pair always in one workgroup, with a ring that
// re-read the last block past its end), us per layer with the prologue and the merge, passes in a graph:
// one sequence of 417 tokens 8.4 -> 6.9 (stripes in one workgroup); 8 of U[32, 1150] 18.4 -> 13.3, 24
// 21.6 -> 17.7, 12 with 4 heads per KV head 18.0 -> 14.3 (stripes spread one by one; by twos 13.5 / 18.4 /
// 14.9, by fours 15.0 / 21.2 / 15.0); 3 lognormal to 8192 89 -> 17.7, 21 with 8 heads per KV head 102 ->
// 54.7 (parts).  Rings of 2 / 3 / 4 blocks: 13.4 / 13.3 / 13.3 at 8 sequences, 14.8 / 14.3 / 15.5 at 12.
#ifndef MI_DECODE_STRIPE_WAVES
#define MI_DECODE_STRIPE_WAVES 1
#endif
#ifndef MI_DECODE_STRIPE_DEPTH
#define MI_DECODE_STRIPE_DEPTH 3
#endif
constexpr int kStripeWaves = MI_DECODE_STRIPE_WAVES;  // stripes (wavefronts) of a workgroup when they are spread
constexpr int kStripeDepth = MI_DECODE_STRIPE_DEPTH;  // blocks of a stripe in registers, the current one included
constexpr int kPartWaves = 4;
constexpr int kPartMaxBlocks = 64 * kPartWaves;  // a lane holds one block id of its wavefront
constexpr int kSeqMaxBlocks = 64 * kStripes;
constexpr int kPairTokens = 2 * kBlockSize;

// The fused form's prologue: what mi_qk_norm_rope's decode form does for KV head g of sequence b.  16
// lanes per head normalise and rotate the kG query heads and the key head into LDS; the workgroup told
// to append writes the key head with value head g into the sequence's new slot.  The wavefronts that
// attend the slot's block do not read that row back: they put the key head and the value row in place
// of what they loaded, so no load waits for the append, in this workgroup or another.
template <int kKvHeads, int kG, int kWaves>
struct Prologue {
  static constexpr int kUnits = kG + 1;  // query heads, then the new key
  static constexpr int kPasses = (kUnits + 4 * kWaves - 1) / (4 * kWaves);
  u32x4 x[kPasses], w[kPasses], c, s, v;
  int64_t slot;  // the new token's slot; -1: none

  // Unit of 16-lane row r in a pass; past the last one the key head again.
  static __device__ __forceinline__ int unit(int pass, int wave, int r) {
    return min(4 * (pass * kWaves + wave) + r, kG);
  }
  __device__ __forceinline__ void load(const DecodeArgs& a, int b, int g, int wave, int r, int dl) {
    slot = a.slot_mapping[b * a.slot_stride];
#pragma unroll
    for (int p = 0; p < kPasses; ++p) {
      const int u = unit(p, wave, r);
      x[p] = *reinterpret_cast<const u32x4*>((u < kG ? a.q_raw + b * a.q_raw_row + (g * kG + u) * kHeadDim
                                                     : a.k_raw + b * a.k_raw_row + g * kHeadDim) + 8 * dl);
      w[p] = *reinterpret_cast<const u32x4*>((u < kG ? a.q_weight : a.k_weight) + 8 * dl);
    }
    c = *reinterpret_cast<const u32x4*>(a.cos + b * kHeadDim + 8 * dl);
    s = *reinterpret_cast<const u32x4*>(a.sin + b * kHeadDim + 8 * dl);
    v = *reinterpret_cast<const u32x4*>(a.v_raw + b * a.v_raw_row + g * kHeadDim + 8 * dl);
  }
  // heads: [kUnits][128] in LDS, complete after the barrier inside.
  __device__ __forceinline__ void run(const DecodeArgs& a, int g, int wave, int r, int dl, bool append,
                                      uint16_t (*heads)[kHeadDim]) {
    if (slot >= a.num_slots || slot < 0) slot = -1;
#pragma unroll
    for (int p = 0; p < kPasses; ++p) {
      if (4 * (p * kWaves + wave) >= kUnits) break;  // wave-uniform
      const int u = unit(p, wave, r);
      const u32x4 o = norm_rope_piece(x[p], w[p], c, s, a.eps, dl);
      *reinterpret_cast<u32x4*>(&heads[u][8 * dl]) = o;
      if (append && u == kG && slot >= 0) {  // the repeated units write the same bytes
        const int64_t at = (slot * kKvHeads + g) * kHeadDim + 8 * dl;
        *reinterpret_cast<u32x4*>(const_cast<uint16_t*>(a.key_pool) + at) = o;
        *reinterpret_cast<u32x4*>(const_cast<uint16_t*>(a.value_pool) + at) = v;
      }
    }
    __syncthreads();
  }
};

// Workgroup -> (KV head, sequence, split): ids go round-robin to the XCDs; the heads of one (sequence,
// split) are neighbours, and the head an XCD gets rotates from one to the next, so every XCD gets an
// even share of each sequence and of the heads' columns of the pool rows.
struct SeqUnit {
  int g, b, split;
};
template <int kKvHeads>
__device__ __forceinline__ SeqUnit seq_unit(int batch) {
  const int u = static_cast<int>(blockIdx.x) / kKvHeads;
  const int split = u / batch;
  return {(static_cast<int>(blockIdx.x) + u) % kKvHeads, u - split * batch, split};
}

// Q^T fragments of a wavefront: head dl (zero past the group), dims 32 ks + 8 r .. +8.
template <int kG, bool kFused>
__device__ __forceinline__ void query_fragments(const DecodeArgs& a, int b, int g, int r, int dl,
                                                const uint16_t (*heads)[kHeadDim], bf16x8 (&qf)[4]) {
#pragma unroll
  for (int ks = 0; ks < 4; ++ks) {
    if constexpr (kFused)
      qf[ks] = dl < kG ? *reinterpret_cast<const bf16x8*>(&heads[dl < kG ? dl : 0][32 * ks + 8 * r]) : bf16x8{};
    else
      qf[ks] = dl < kG ? *reinterpret_cast<const bf16x8*>(a.query + b * a.q_row + (g * kG + dl) * a.q_head + 32 * ks + 8 * r)
                       : bf16x8{};
  }
}

// kWaves stripes per workgroup: kStripes (rows written here) or kStripeWaves (states to the workspace).
template <int kKvHeads, int kG, bool kFused, int kWaves>
__global__ __launch_bounds__(64 * kWaves, 2) void paged_decode_stripe_kernel(const DecodeArgs a) {
  constexpr int kRowElems = kKvHeads * kHeadDim;
  constexpr int kBlockElems = kBlockSize * kRowElems;
  static_assert(kG <= 8, "a stripe's merged rows overlay its K staging");
  // Each wavefront's K staging; its output rows overlay it after the last block.
  __shared__ __align__(16) uint16_t s_kst[kWaves][kBlockSize * kKStageRow];
  __shared__ float s_ml[kWaves][kG][2];
  __shared__ __align__(16) uint16_t s_q[kFused ? kG + 1 : 1][kHeadDim];
  const SeqUnit unit = seq_unit<kKvHeads>(a.batch);
  const int g = unit.g, b = unit.b;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  const int dl = lane & 15;
  const int r = lane >> 4;
  const int stripe = unit.split * kWaves + w;

  // Lane i holds the id of block stripe + kStripes i (ids outside the pool read block 0; entries past
  // the table repeat its last one and are not used).
  int64_t id = a.block_tables[b * a.bt_stride + min(stripe + kStripes * lane, a.max_blocks - 1)];
  const int64_t ctx = a.context_lens[b * a.ctx_stride];
  Prologue<kKvHeads, kG, kWaves> pro;
  if constexpr (kFused) pro.load(a, b, g, w, r, dl);
  const int n = static_cast<int>(min(ctx, static_cast<int64_t>(a.max_blocks) * kBlockSize));
  const int nblk = blocks_of(n);
  if (id < 0 || id >= a.num_blocks) id = 0;
  const uint32_t id_lo = static_cast<uint32_t>(id), id_hi = static_cast<uint32_t>(static_cast<uint64_t>(id) >> 32);
  const int cnt = nblk > stripe ? (nblk - 1 - stripe) / kStripes + 1 : 0;  // blocks stripe + kStripes i, i < cnt <= 64

  // Byte offsets of the lane's first pieces inside a block (the block's base address is uniform).
  const uint32_t k_off = 2u * (r * kRowElems + g * kHeadDim + 8 * dl);
  const uint32_t v_off = 2u * (4 * r * kRowElems + g * kHeadDim + 8 * dl);
  u32x4 kbuf[kStripeDepth][4], vbuf[kStripeDepth][4];
  auto issue = [&](int ring, int i) {
    const uint32_t blo = __builtin_amdgcn_readlane(id_lo, i);
    const uint32_t bhi = __builtin_amdgcn_readlane(id_hi, i);
    const int64_t base = static_cast<int64_t>((static_cast<uint64_t>(bhi) << 32) | blo) * kBlockElems;
    const char* kp = reinterpret_cast<const char*>(a.key_pool + base);
    const char* vp = reinterpret_cast<const char*>(a.value_pool + base);
#pragma unroll
    for (int t = 0; t < 4; ++t) kbuf[ring][t] = load_vec<kNtLoads>(reinterpret_cast<const u32x4*>(kp + t * 8 * kRowElems + k_off));
#pragma unroll
    for (int t = 0; t < 4; ++t) vbuf[ring][t] = load_vec<kNtLoads>(reinterpret_cast<const u32x4*>(vp + t * 2 * kRowElems + v_off));
  };
#pragma unroll
  for (int s = 0; s < kStripeDepth - 1; ++s)
    if (s < cnt) issue(s, s);  // wave-uniform; in flight during the prologue

  uint64_t slot_lanes = 0;  // lanes whose block holds the new token's slot
  if constexpr (kFused) {
    pro.run(a, g, w, r, dl, unit.split == 0, s_q);
    if (pro.slot >= 0) slot_lanes = __builtin_amdgcn_ballot_w64(id == (pro.slot >> 4));
  }
  uint16_t* out_b = a.out + b * a.out_row + (g * kG) * kHeadDim;  // query heads g kG .. g kG + kG - 1
  if (nblk == 0) {  // empty context: zero rows (uniform over the workgroup)
    if (unit.split == 0)
      for (int i = threadIdx.x; i < kG * 16; i += 64 * kWaves) *reinterpret_cast<uint4*>(out_b + 8 * i) = uint4{0, 0, 0, 0};
    return;
  }
  bf16x8 qf[4];
  query_fragments<kG, kFused>(a, b, g, r, dl, s_q, qf);
  MfmaState ms;
  ms.m = -INFINITY;
  ms.l = 0.0f;
#pragma unroll
  for (int t = 0; t < 8; ++t) ms.o[t] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  for (int i0 = 0; i0 < cnt; i0 += kStripeDepth) {
#pragma unroll
    for (int s = 0; s < kStripeDepth; ++s) {
      const int i = i0 + s;
      if (i >= cnt) break;  // wave-uniform
      if (i + kStripeDepth - 1 < cnt) issue((s + kStripeDepth - 1) % kStripeDepth, i + kStripeDepth - 1);
      if constexpr (kFused) {
        if ((slot_lanes >> i) & 1) {  // the new token's rows in place of what was loaded
          const int t = static_cast<int>(pro.slot & 15);
          const u32x4 kn = *reinterpret_cast<const u32x4*>(&s_q[kFused ? kG : 0][8 * dl]);
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            kbuf[s][e] = 4 * e + r == t ? kn : kbuf[s][e];
            vbuf[s][e] = 4 * r + e == t ? pro.v : vbuf[s][e];
          }
        }
      }
      attend_block_mfma(ms, qf, kbuf[s], vbuf[s], s_kst[w], a.scale, (stripe + kStripes * i) * kBlockSize, n, lane);
    }
  }

  // Lane: heads 4 r + i, dims 8 dl .. +8; head j's max and sum live in lane j.
  const float lsum = xsum32_f32(xsum16_f32(ms.l));
  float* s_acc = reinterpret_cast<float*>(s_kst[w]);  // [kG][128]
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int j = 4 * r + i;
    const float Lj = __shfl(lsum, j);
    const float Mj = __shfl(ms.m, j);
    if (j >= kG) continue;
    float4 lo4 = make_float4(ms.o[0][i], ms.o[1][i], ms.o[2][i], ms.o[3][i]);
    float4 hi4 = make_float4(ms.o[4][i], ms.o[5][i], ms.o[6][i], ms.o[7][i]);
    float4* dst;
    float* ml;
    if constexpr (kWaves == kStripes) {
      dst = reinterpret_cast<float4*>(s_acc + j * kHeadDim + 8 * dl);
      ml = s_ml[w][j];
    } else {
      const int64_t at = (static_cast<int64_t>(b) * kStripes + stripe) * (kKvHeads * kG) + g * kG + j;
      dst = reinterpret_cast<float4*>(a.ws_acc + at * kHeadDim + 8 * dl);
      ml = a.ws_ml + at * 2;
    }
    dst[0] = lo4;
    dst[1] = hi4;
    if (dl == 0) {
      ml[0] = Mj;
      ml[1] = Lj;
    }
  }
  if constexpr (kWaves == kStripes) {
    __syncthreads();
    if (threadIdx.x < kG * 16) {
      const int h = threadIdx.x >> 4, dm = threadIdx.x & 15;
      StripeMerge sm;
#pragma unroll
      for (int v = 0; v < kStripes; ++v) {
        const float4* src = reinterpret_cast<const float4*>(reinterpret_cast<const float*>(s_kst[v]) + h * kHeadDim + 8 * dm);
        sm.m[v] = s_ml[v][h][0];
        sm.l[v] = s_ml[v][h][1];
        sm.x[v] = src[0];
        sm.y[v] = src[1];
      }
      sm.store(out_b + h * kHeadDim + 8 * dm);
    }
  }
}

// The merge launch of spread stripes: one thread per (query head of the KV head, 8 dims), every load
// issued at once; empty contexts have been written.
template <int kKvHeads, int kG>
__global__ __launch_bounds__(kG * 16 < 64 ? 64 : kG * 16) void paged_decode_stripe_merge_kernel(const DecodeArgs a) {
  const int b = blockIdx.x, g = blockIdx.y;
  const int h = min(static_cast<int>(threadIdx.x) >> 4, kG - 1), dm = threadIdx.x & 15;
  StripeMerge sm;
  const int64_t n = context_of(a, b);
#pragma unroll
  for (int v = 0; v < kStripes; ++v) {
    const int64_t at = (static_cast<int64_t>(b) * kStripes + v) * (kKvHeads * kG) + g * kG + h;
    const float2 ml = *reinterpret_cast<const float2*>(a.ws_ml + at * 2);
    const float4* src = reinterpret_cast<const float4*>(a.ws_acc + at * kHeadDim + 8 * dm);
    sm.m[v] = ml.x;
    sm.l[v] = ml.y;
    sm.x[v] = src[0];
    sm.y[v] = src[1];
  }
  if (n <= 0 || threadIdx.x >= kG * 16) return;
  sm.store(a.out + b * a.out_row + (g * kG + h) * kHeadDim + 8 * dm);
}

// ---- Parts.  Part p is the a.part_blocks table blocks from p part_blocks on (those inside the context),
// so that its block ids do not wait for the context length.  Its kPartWaves wavefronts take pairs of
// blocks w, w + kPartWaves, ... (32 tokens a step), each pair's K registers loaded again as soon as they
// are in LDS and its V registers as soon as they are multiplied, then merge their states through LDS.
// kb / vb: the lane's K pieces (token 4 i + r of each block, dims 8 dl .. +8: whole 256-byte rows per
// instruction) and V pieces (token 4 r + i).  kst: the wavefront's 32-row K staging in LDS, through
// which K reaches the MFMA A layout.
//  * S^T = K Q^T per block as in attend_block_mfma; lane: head dl, tokens 4 r + i of both blocks.
//  * O += P V in one v_mfma_f32_16x16x32_bf16 per output tile: k index 8 r + e is token 4 r + e of the
//    first block for e < 4, token 4 r + e - 4 of the second for the rest, so P and V both stay in the
//    lanes that hold them.
__device__ __forceinline__ void stage_pair(const u32x4 (&kb)[2][4], uint16_t* kst, int lane) {
  const int dl = lane & 15, r = lane >> 4;
#pragma unroll
  for (int h = 0; h < 2; ++h)
#pragma unroll
    for (int i = 0; i < 4; ++i)
      *reinterpret_cast<u32x4*>(kst + (kBlockSize * h + 4 * i + r) * kKStageRow + 8 * dl) = kb[h][i];
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Probabilities of the staged pair (first token tok_base, tokens from n on masked) as the A operand.
__device__ __forceinline__ bf16x8 pair_probs(MfmaState& st, const bf16x8 (&qf)[4], const uint16_t* kst, float scale,
                                             int tok_base, int n, int lane) {
  const int dl = lane & 15, r = lane >> 4;
  f32x4 acc[2] = {{0.0f, 0.0f, 0.0f, 0.0f}, {0.0f, 0.0f, 0.0f, 0.0f}};
#pragma unroll
  for (int ks = 0; ks < 4; ++ks)
#pragma unroll
    for (int h = 0; h < 2; ++h)
      acc[h] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
          *reinterpret_cast<const bf16x8*>(kst + (kBlockSize * h + dl) * kKStageRow + 32 * ks + 8 * r), qf[ks], acc[h],
          0, 0, 0);
  // The next pair's staging stores follow these reads in the wavefront's LDS order.
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  float sc[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) sc[e] = score_log2(acc[e >> 2][e & 3], scale);
  if (tok_base + kPairTokens > n) {  // uniform
#pragma unroll
    for (int e = 0; e < 8; ++e) sc[e] = tok_base + kBlockSize * (e >> 2) + 4 * r + (e & 3) < n ? sc[e] : -INFINITY;
  }
  float mb = sc[0];
#pragma unroll
  for (int e = 1; e < 8; ++e) mb = fmaxf(mb, sc[e]);
  if (__builtin_amdgcn_ballot_w64(mb > st.m + kRescaleSlack) != 0) {  // lazy rescale (wave-uniform)
    const float nm = fmaxf(st.m, xmax32(xmax16(mb)));
    const float al = (nm == -INFINITY) ? 1.0f : __builtin_amdgcn_exp2f(st.m - nm);
    st.m = nm;
    st.l *= al;
#pragma unroll
    for (int i = 0; i < 4; ++i) {  // O rows are heads 4 r + i: lane h holds head h's factor
      const float ai = __shfl(al, 4 * r + i);
#pragma unroll
      for (int t = 0; t < 8; ++t) st.o[t][i] *= ai;
    }
  }
  const float ref = st.m == -INFINITY ? 0.0f : st.m;
  f32x8 p;
#pragma unroll
  for (int e = 0; e < 8; ++e) p[e] = __builtin_amdgcn_exp2f(sc[e] - ref);
  st.l += ((p[0] + p[1]) + (p[2] + p[3])) + ((p[4] + p[5]) + (p[6] + p[7]));
  return __builtin_convertvector(p, bf16x8);
}

__device__ __forceinline__ void pair_values(MfmaState& st, const bf16x8 pa, const u32x4 (&vb)[2][4]) {
#pragma unroll
  for (int t = 0; t < 8; ++t) {
    const uint32_t sel = (t & 1) ? 0x07060302u : 0x05040100u;
    u32x4 v;  // tokens 0, 1 | 2, 3 of the first block, then of the second, at dim t
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      v[2 * h] = __builtin_amdgcn_perm(vb[h][1][t >> 1], vb[h][0][t >> 1], sel);
      v[2 * h + 1] = __builtin_amdgcn_perm(vb[h][3][t >> 1], vb[h][2][t >> 1], sel);
    }
    st.o[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(pa, __builtin_bit_cast(bf16x8, v), st.o[t], 0, 0, 0);
  }
}

// Three wavefronts per SIMD (a budget of 128 registers would spill: 2-3 times slower).
template <int kKvHeads, int kG, bool kFused>
__global__ __launch_bounds__(64 * kPartWaves, 3) void paged_decode_parts_kernel(const DecodeArgs a) {
  constexpr int kRowElems = kKvHeads * kHeadDim;
  constexpr int kBlockElems = kBlockSize * kRowElems;
  static_assert(kG <= 16, "at most 16 query heads per KV head");
  // Each wavefront's K staging; its merged output rows overlay it after the last pair.
  constexpr int kStageElems = kPairTokens * kKStageRow;
  static_assert(kStageElems * sizeof(uint16_t) >= kG * kHeadDim * sizeof(float), "the output rows fit the staging");
  __shared__ __align__(16) uint16_t s_kst[kPartWaves][kStageElems];
  __shared__ float s_ml[kPartWaves][kG][2];
  __shared__ __align__(16) uint16_t s_q[kFused ? kG + 1 : 1][kHeadDim];
  const SeqUnit unit = seq_unit<kKvHeads>(a.batch);
  const int g = unit.g, b = unit.b, part = unit.split;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  const int dl = lane & 15;
  const int r = lane >> 4;
  const int lo = part * a.part_blocks;

  // Lane 2 j + h holds the id of block h of the wavefront's pair j (ids outside the pool read block 0).
  // Entries past the table repeat its last one (not used).
  const int my_blk = lo + 2 * (w + kPartWaves * (lane >> 1)) + (lane & 1);
  int64_t id = a.block_tables[b * a.bt_stride + min(my_blk, a.max_blocks - 1)];
  const int64_t ctx = a.context_lens[b * a.ctx_stride];
  Prologue<kKvHeads, kG, kPartWaves> pro;
  if constexpr (kFused) pro.load(a, b, g, w, r, dl);
  const int n = static_cast<int>(min(ctx, static_cast<int64_t>(a.max_blocks) * kBlockSize));
  const int nblk = blocks_of(n);
  if (part > 0 && lo >= nblk) return;  // uniform
  if (id < 0 || id >= a.num_blocks) id = 0;
  const uint32_t id_lo = static_cast<uint32_t>(id), id_hi = static_cast<uint32_t>(static_cast<uint64_t>(id) >> 32);
  const int hi = min(lo + a.part_blocks, nblk);
  const int tok_end = min(n, hi * kBlockSize);
  const int pairs = (hi - lo + 1) / 2;
  const int cnt = pairs > w ? (pairs - 1 - w) / kPartWaves + 1 : 0;  // pairs w + kPartWaves j, j < cnt <= 32

  // Byte offsets of the lane's first pieces inside a block (the block's base address is uniform).
  const uint32_t k_off = 2u * (r * kRowElems + g * kHeadDim + 8 * dl);
  const uint32_t v_off = 2u * (4 * r * kRowElems + g * kHeadDim + 8 * dl);
  u32x4 kb[2][4], vb[2][4];
  // The lane that holds block h of pair j; past the part's end that of the block before (masked).
  auto id_lane = [&](int j, int h) { return 2 * j + ((lo + 2 * (w + kPartWaves * j) + h < hi) ? h : 0); };
  auto block_id = [&](int j, int h) {
    const int i = id_lane(j, h);
    const uint32_t blo = __builtin_amdgcn_readlane(id_lo, i);
    const uint32_t bhi = __builtin_amdgcn_readlane(id_hi, i);
    return static_cast<int64_t>((static_cast<uint64_t>(bhi) << 32) | blo);
  };
  auto load_keys = [&](int j) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const char* kp = reinterpret_cast<const char*>(a.key_pool + block_id(j, h) * kBlockElems);
#pragma unroll
      for (int t = 0; t < 4; ++t) kb[h][t] = load_vec<kNtLoads>(reinterpret_cast<const u32x4*>(kp + t * 8 * kRowElems + k_off));
    }
  };
  auto load_values = [&](int j) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const char* vp = reinterpret_cast<const char*>(a.value_pool + block_id(j, h) * kBlockElems);
#pragma unroll
      for (int t = 0; t < 4; ++t) vb[h][t] = load_vec<kNtLoads>(reinterpret_cast<const u32x4*>(vp + t * 2 * kRowElems + v_off));
    }
  };
  if (cnt > 0) {  // wave-uniform
    load_keys(0);
    load_values(0);
  }

  uint64_t slot_lanes = 0;  // lanes whose block holds the new token's slot
  if constexpr (kFused) {
    pro.run(a, g, w, r, dl, part == 0, s_q);
    if (pro.slot >= 0) slot_lanes = __builtin_amdgcn_ballot_w64(id == (pro.slot >> 4));
  }
  uint16_t* out_b = a.out + b * a.out_row + (g * kG) * kHeadDim;  // query heads g kG .. g kG + kG - 1
  if (nblk == 0) {  // empty context: zero rows (uniform over the workgroup)
    if (threadIdx.x < kG * 16) *reinterpret_cast<uint4*>(out_b + 8 * threadIdx.x) = uint4{0, 0, 0, 0};
    return;
  }
  bf16x8 qf[4];
  query_fragments<kG, kFused>(a, b, g, r, dl, s_q, qf);
  MfmaState ms;
  ms.m = -INFINITY;
  ms.l = 0.0f;
#pragma unroll
  for (int t = 0; t < 8; ++t) ms.o[t] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};

  uint16_t* kst = s_kst[w];
  const float scale = a.scale;
  // The new token's rows in place of what was loaded from its slot (wave-uniform branch).
  auto in_slot_block = [&](int j, int h) { return (slot_lanes >> id_lane(j, h)) & 1; };
  auto patch_keys = [&](int j) {
    if constexpr (kFused) {
      const int t = static_cast<int>(pro.slot & 15);
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        if (!in_slot_block(j, h)) continue;
        const u32x4 kn = *reinterpret_cast<const u32x4*>(&s_q[kFused ? kG : 0][8 * dl]);
#pragma unroll
        for (int i = 0; i < 4; ++i) kb[h][i] = 4 * i + r == t ? kn : kb[h][i];
      }
    }
  };
  auto patch_values = [&](int j) {
    if constexpr (kFused) {
      const int t = static_cast<int>(pro.slot & 15);
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        if (!in_slot_block(j, h)) continue;
#pragma unroll
        for (int i = 0; i < 4; ++i) vb[h][i] = 4 * r + i == t ? pro.v : vb[h][i];
      }
    }
  };
  auto tok_base = [&](int j) { return (lo + 2 * (w + kPartWaves * j)) * kBlockSize; };
  for (int j = 0; j + 1 < cnt; ++j) {
    patch_keys(j);
    stage_pair(kb, kst, lane);
    load_keys(j + 1);
    const bf16x8 pa = pair_probs(ms, qf, kst, scale, tok_base(j), tok_end, lane);
    patch_values(j);
    pair_values(ms, pa, vb);
    load_values(j + 1);
  }
  if (cnt > 0) {
    patch_keys(cnt - 1);
    stage_pair(kb, kst, lane);
    const bf16x8 pa = pair_probs(ms, qf, kst, scale, tok_base(cnt - 1), tok_end, lane);
    patch_values(cnt - 1);
    if (lo + 2 * (w + kPartWaves * (cnt - 1)) + 1 >= hi) {  // wave-uniform: the second block repeats the first
#pragma unroll
      for (int i = 0; i < 4; ++i) vb[1][i] = u32x4{};       // its weights are zero, but an infinite value is not
    }
    pair_values(ms, pa, vb);
  }

  // ---- merge the wavefronts through LDS (log-sum-exp).  Lane: heads 4 r + i, dims 8 dl .. +8; head
  // j's max and sum live in lane j.
  float* s_acc = reinterpret_cast<float*>(kst);  // [kG][128]
  const float lsum = xsum32_f32(xsum16_f32(ms.l));
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int j = 4 * r + i;
    const float Lj = __shfl(lsum, j);
    const float Mj = __shfl(ms.m, j);
    if (j >= kG) continue;
#pragma unroll
    for (int t = 0; t < 8; ++t) s_acc[j * kHeadDim + 8 * dl + t] = ms.o[t][i];
    if (dl == 0) {
      s_ml[w][j][0] = Mj;
      s_ml[w][j][1] = Lj;
    }
  }
  __syncthreads();
  if (threadIdx.x < kG * 16) {
    const int h = threadIdx.x >> 4;
    const int dm = threadIdx.x & 15;
    float Mx = -INFINITY;
#pragma unroll
    for (int v = 0; v < kPartWaves; ++v) Mx = fmaxf(Mx, s_ml[v][h][0]);
    float L = 0.0f, o[8];
#pragma unroll
    for (int d = 0; d < 8; ++d) o[d] = 0.0f;
#pragma unroll
    for (int v = 0; v < kPartWaves; ++v) {
      const float mv = s_ml[v][h][0];
      const float e = mv == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(mv - Mx);
      L += e * s_ml[v][h][1];
      const float4* src = reinterpret_cast<const float4*>(reinterpret_cast<const float*>(s_kst[v]) + h * kHeadDim + 8 * dm);
      const float4 x = src[0], y = src[1];
      o[0] += e * x.x; o[1] += e * x.y; o[2] += e * x.z; o[3] += e * x.w;
      o[4] += e * y.x; o[5] += e * y.y; o[6] += e * y.z; o[7] += e * y.w;
    }
    if (nblk <= a.part_blocks) {  // in one part
      store_bf16x8(out_b + h * kHeadDim + 8 * dm, o, 1.0f / L);
    } else {
      const int64_t at = (static_cast<int64_t>(b) * a.splits + part) * (kKvHeads * kG) + g * kG + h;
      float4* dst = reinterpret_cast<float4*>(a.ws_acc + at * kHeadDim + 8 * dm);
      dst[0] = make_float4(o[0], o[1], o[2], o[3]);
      dst[1] = make_float4(o[4], o[5], o[6], o[7]);
      if (dm == 0) *reinterpret_cast<float2*>(a.ws_ml + at * 2) = make_float2(Mx, L);
    }
  }
}

// ---- The merge launch: one workgroup per (sequence, KV head) joins the partials its sequence left
// (log-sum-exp) and writes the bf16 rows; a sequence in one piece has been written already.
//  * stream kernel (kParts false): a sequence cut by range boundaries left the first range's
//    last-sequence slot, then the first-sequence slot of every later range up to the one holding its
//    last block; empty contexts get their zero rows here.
//  * parts kernel (kParts true): slot b splits + part for each part (that kernel writes the zero rows
//    itself).
// A launch of a few microseconds is a chain of latencies, so it is kept short: 16 lanes cover the
// 128 dims and 16 partials are read side by side, every head's loads before any is used, with
// one reduction over the contexts (stream form) and 32-bit range arithmetic.  Many short sequences take the
// rows form below.
constexpr int kMergeThreads = 256;
constexpr int kMergeRows = kMergeThreads / 16;  // partials read side by side

template <int kKvHeads, int kG, bool kParts>
__global__ __launch_bounds__(kMergeThreads) void paged_decode_merge_kernel(const DecodeArgs a) {
  constexpr int kHeads = kKvHeads * kG;
  constexpr int kWaves = kMergeThreads / 64;
  __shared__ float s_acc[kWaves][kG][kHeadDim];
  __shared__ float s_ml[kWaves][kG][2];
  const int b = blockIdx.x, g = blockIdx.y;
  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int dm = tid & 15, row = tid >> 4;
  uint16_t* out_b = a.out + b * a.out_row + g * kG * kHeadDim;
  // Partial p of the sequence, this lane's 8 dims of every head.
  float2 ml[kG];
  float4 x[kG], y[kG];
  auto load_partial = [&](int64_t slot) {
    const int64_t unit = slot * kHeads + g * kG;
#pragma unroll
    for (int j = 0; j < kG; ++j) {
      ml[j] = *reinterpret_cast<const float2*>(a.ws_ml + (unit + j) * 2);
      const float4* src = reinterpret_cast<const float4*>(a.ws_acc + (unit + j) * kHeadDim + 8 * dm);
      x[j] = src[0];
      y[j] = src[1];
    }
  };
  const int64_t ctx = context_of(a, b);
  int first = 0, count;  // partials [first, first + count)
  if constexpr (kParts) {
    // The first round goes out beside the context (slots no part wrote are read and not used).
    load_partial(static_cast<int64_t>(b) * a.splits + min(row, a.splits - 1));
    count = (blocks_of(ctx) + a.part_blocks - 1) / a.part_blocks;
  } else {
    __shared__ int s_sum[kWaves][2];
    const int nblk = blocks_of(ctx);
    int before = 0, total = 0;  // blocks of the sequences before b, and of all
    for (int i = tid; i < a.batch; i += kMergeThreads) {
      const int v = blocks_of(context_of(a, i));
      total += v;
      before += i < b ? v : 0;
    }
    before = wave_sum_i32(before);
    total = wave_sum_i32(total);
    if (lane == 0) {
      s_sum[w][0] = before;
      s_sum[w][1] = total;
    }
    __syncthreads();
    before = total = 0;
#pragma unroll
    for (int v = 0; v < kWaves; ++v) {
      before += s_sum[v][0];
      total += s_sum[v][1];
    }
    if (nblk == 0) {  // uniform
      if (tid < kG * 16) *reinterpret_cast<uint4*>(out_b + 8 * tid) = uint4{0, 0, 0, 0};
      return;
    }
    const Ranges rg(total, a.streams);
    first = rg.of(before);
    count = rg.of(before + nblk - 1) - first + 1;
  }
  if (count <= 1) return;  // uniform: written by the attention kernel

  float m[kG], l[kG], acc[kG][8];
#pragma unroll
  for (int j = 0; j < kG; ++j) {
    m[j] = -INFINITY;
    l[j] = 0.0f;
#pragma unroll
    for (int d = 0; d < 8; ++d) acc[j][d] = 0.0f;
  }
  for (int p = row; p < count; p += kMergeRows) {
    if (!kParts)
      load_partial(static_cast<int64_t>(first + p) * 2 + (p == 0 ? 1 : 0));
    else if (p >= kMergeRows)
      load_partial(static_cast<int64_t>(b) * a.splits + p);
#pragma unroll
    for (int j = 0; j < kG; ++j) {
      const float nm = fmaxf(m[j], ml[j].x);
      const float e0 = m[j] == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(m[j] - nm);
      const float e1 = ml[j].x == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(ml[j].x - nm);
      m[j] = nm;
      l[j] = e0 * l[j] + e1 * ml[j].y;
      const float v[8] = {x[j].x, x[j].y, x[j].z, x[j].w, y[j].x, y[j].y, y[j].z, y[j].w};
#pragma unroll
      for (int d = 0; d < 8; ++d) acc[j][d] = e0 * acc[j][d] + e1 * v[d];
    }
  }
  // The wavefront's four rows, then the wavefronts through LDS.
#pragma unroll
  for (int j = 0; j < kG; ++j) {
    const float mx = xmax32(xmax16(m[j]));
    const float e = m[j] == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(m[j] - mx);
    const float ls = xsum32_f32(xsum16_f32(l[j] * e));
#pragma unroll
    for (int d = 0; d < 8; ++d) acc[j][d] = xsum32_f32(xsum16_f32(acc[j][d] * e));
    if (lane < 16) {
#pragma unroll
      for (int d = 0; d < 8; ++d) s_acc[w][j][8 * dm + d] = acc[j][d];
      if (dm == 0) {
        s_ml[w][j][0] = mx;
        s_ml[w][j][1] = ls;
      }
    }
  }
  __syncthreads();
  if (tid < kG * 16) {
    const int h = row;
    float Mx = -INFINITY;
#pragma unroll
    for (int v = 0; v < kWaves; ++v) Mx = fmaxf(Mx, s_ml[v][h][0]);
    float L = 0.0f, o[8];
#pragma unroll
    for (int d = 0; d < 8; ++d) o[d] = 0.0f;
#pragma unroll
    for (int v = 0; v < kWaves; ++v) {
      const float mv = s_ml[v][h][0];
      const float e = mv == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(mv - Mx);
      L += e * s_ml[v][h][1];
#pragma unroll
      for (int d = 0; d < 8; ++d) o[d] += e * s_acc[v][h][8 * dm + d];
    }
    store_bf16x8(out_b + h * kHeadDim + 8 * dm, o, 1.0f / L);
  }
}

// The stream form's merge where a sequence spans under two ranges on average: one workgroup per sequence, a thread
// per (query head, 8 dims) of all heads, kMergeUnroll partials a step.  A sequence is cut into two or three
// then, or not at all, and the launch is its pass over the contexts, which the form above makes once per
// KV head beside reads for 16 partials: 512 sequences with 16 heads 5-6 us where that form takes 12, with 64
// heads 9 / 37, 2048 with 16 heads 14 / 32 (200 of U[32, 300], attention and merge, 33.7 / 36.4).
template <int kHeads>
constexpr int merge_rows_threads() {
  return kHeads * 16 < 256 ? 256 : kHeads * 16;
}
template <int kHeads>
__global__ __launch_bounds__(merge_rows_threads<kHeads>()) void paged_decode_merge_rows_kernel(const DecodeArgs a) {
  constexpr int kThreads = merge_rows_threads<kHeads>();
  constexpr int kWaves = kThreads / 64;
  constexpr int kMergeUnroll = 4;
  __shared__ int s_sum[kWaves][2];
  const int b = blockIdx.x, tid = threadIdx.x;
  const int nblk = blocks_of(context_of(a, b));
  int before = 0, total = 0;  // blocks of the sequences before b, and of all
  for (int i = tid; i < a.batch; i += kThreads) {
    const int v = blocks_of(context_of(a, i));
    total += v;
    before += i < b ? v : 0;
  }
  before = wave_sum_i32(before);
  total = wave_sum_i32(total);
  if ((tid & 63) == 0) {
    s_sum[tid >> 6][0] = before;
    s_sum[tid >> 6][1] = total;
  }
  __syncthreads();
  if (tid >= kHeads * 16) return;
  before = total = 0;
#pragma unroll
  for (int v = 0; v < kWaves; ++v) {
    before += s_sum[v][0];
    total += s_sum[v][1];
  }
  const int h = tid >> 4, dm = tid & 15;
  uint16_t* dst = a.out + b * a.out_row + h * kHeadDim + 8 * dm;
  if (nblk == 0) {
    *reinterpret_cast<uint4*>(dst) = uint4{0, 0, 0, 0};
    return;
  }
  const Ranges rg(total, a.streams);
  const int first = rg.of(before), last = rg.of(before + nblk - 1);
  if (first == last) return;  // written by the stream kernel
  auto slot_of = [&](int k) -> int64_t { return (static_cast<int64_t>(k) * 2 + (k == first ? 1 : 0)) * kHeads + h; };
  float M = -INFINITY;
  for (int k0 = first; k0 <= last; k0 += kMergeUnroll) {
    float m[kMergeUnroll];
#pragma unroll
    for (int u = 0; u < kMergeUnroll; ++u) m[u] = a.ws_ml[slot_of(min(k0 + u, last)) * 2];
#pragma unroll
    for (int u = 0; u < kMergeUnroll; ++u) M = fmaxf(M, m[u]);
  }
  float L = 0.0f, acc[8];
#pragma unroll
  for (int d = 0; d < 8; ++d) acc[d] = 0.0f;
  for (int k0 = first; k0 <= last; k0 += kMergeUnroll) {
    float2 ml[kMergeUnroll];
    float4 x[kMergeUnroll], y[kMergeUnroll];
#pragma unroll
    for (int u = 0; u < kMergeUnroll; ++u) {  // past the last one: that one again, with no weight
      const int64_t slot = slot_of(min(k0 + u, last));
      ml[u] = *reinterpret_cast<const float2*>(a.ws_ml + slot * 2);
      const float4* src = reinterpret_cast<const float4*>(a.ws_acc + slot * kHeadDim + 8 * dm);
      x[u] = src[0];
      y[u] = src[1];
    }
#pragma unroll
    for (int u = 0; u < kMergeUnroll; ++u) {
      if (k0 + u > last) break;
      const float w = ml[u].x == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(ml[u].x - M);
      L += w * ml[u].y;
      const float v[8] = {x[u].x, x[u].y, x[u].z, x[u].w, y[u].x, y[u].y, y[u].z, y[u].w};
#pragma unroll
      for (int d = 0; d < 8; ++d) acc[d] += w * v[d];
    }
  }
  store_bf16x8(dst, acc, 1.0f / L);
}

int head_groups_for(int32_t num_kv_heads) {
  const int waves = num_kv_heads < kMaxWaves ? num_kv_heads : kMaxWaves;
  return num_kv_heads / waves;
}

// Ranges of one launch of `batch` sequences: enough to fill the device (kGroupsPerCu resident
// workgroups per CU), fewer when the launch cannot hold kMinBlocksPerStream blocks per range.
int streams_for(int32_t batch, int32_t max_blocks, int32_t num_kv_heads) {
  const int64_t groups = head_groups_for(num_kv_heads);
  const int64_t resident = static_cast<int64_t>(device_cus()) * kGroupsPerCu / groups;
  const int64_t rows = batch < kMaxBatchPerLaunch ? batch : kMaxBatchPerLaunch;
  const int64_t by_work = (rows * max_blocks + kMinBlocksPerStream - 1) / kMinBlocksPerStream;
  const int64_t s = by_work < resident ? by_work : resident;
  return static_cast<int>(s < 1 ? 1 : s);
}

#ifndef MI_DECODE_PART_GROUPS
#define MI_DECODE_PART_GROUPS 6
#endif
#ifndef MI_DECODE_STRIPE_BLOCKS
#define MI_DECODE_STRIPE_BLOCKS 128
#endif
#ifndef MI_DECODE_STRIPE_PAIRS
#define MI_DECODE_STRIPE_PAIRS 256
#endif
// Workgroups per CU that the parts of a launch aim at, by the table's length (contexts fill part of it):
// 21 sequences lognormal to 8192 took 65 / 62 / 56 / 56 us with 2 / 3 / 6 / 10.
constexpr int kPartGroupsPerCu = MI_DECODE_PART_GROUPS;
// Stripes up to this table length and number of (sequence, KV head) pairs: beyond 128 blocks a stripe
// is a serial chain of more than 16 of them; beyond 256 pairs, parts won (64 sequences of U[32, 1150]
// 39.5 against 41.7 us, 40 of them 26.0 against 27.1, with the prologue in the launch, as it was then).
constexpr int kStripeMaxBlocks = MI_DECODE_STRIPE_BLOCKS;
constexpr int kStripeMaxPairs = MI_DECODE_STRIPE_PAIRS;

// Which small-launch form takes a launch, from its table length and the partials the workspace (sized by
// streams_for, two slots per range; has_workspace false: none) holds.
void cut_sequences(DecodeArgs& a, int32_t num_kv_heads, bool has_workspace) {
  const int64_t pairs = static_cast<int64_t>(a.batch) * num_kv_heads;
  const int64_t slots = has_workspace ? 2ll * streams_for(a.batch, a.max_blocks, num_kv_heads) / a.batch : 0;
  a.part_blocks = 0;
  a.splits = 1;
  if (a.max_blocks <= kStripeMaxBlocks && pairs <= kStripeMaxPairs) {
    // Spread where the workspace holds a partial per stripe (tables from 64 blocks on).
    if (slots >= kStripes) a.splits = kStripes / kStripeWaves;
    return;
  }
  int64_t parts = (static_cast<int64_t>(device_cus()) * kPartGroupsPerCu + pairs - 1) / pairs;
  parts = parts < slots ? parts : slots;
  if (parts < 2) return;
  const int64_t step = 2 * kPartWaves;
  int64_t blocks = ((a.max_blocks + parts - 1) / parts + step - 1) / step * step;
  blocks = blocks < kPartMaxBlocks ? blocks : kPartMaxBlocks;
  a.part_blocks = static_cast<int32_t>(blocks < a.max_blocks ? blocks : a.max_blocks);
  a.splits = (a.max_blocks + a.part_blocks - 1) / a.part_blocks;
}

// The per-sequence kernels serve launches of at most one (sequence, KV head) pair per CU, and larger ones while
// each sequence can be cut in two (fewer than kPartGroupsPerCu pairs per CU) and their tables hold no more
// than kSeqWork (block, KV head) pairs; beyond that the stream kernel's equal ranges win.  Measured, us per
// layer without the prologue, per-sequence / stream: 64 sequences of U[1, 64] 7.4 / 21.7, of U[1, 700] 25.5 / 26.2,
// 128 of U[1, 300] 22.4 / 25.1, 190 of U[1, 700] 58 / 62; uncut, with eight stripes in a workgroup: 256 of U[1, 420]
// 53 / 50.5, 512 of U[32, 300] 86 / 74, 1024 of U[32, 190] 131 / 103, 4096 of U[1, 48] 342 / 163; 40 lognormal to 8192
// with 5 heads per KV head (163,840 pairs) 112 / 94, 100 of them with 2 264 / 216.  MI_DECODE_PATH=stream or
// =seq (environment) forces one form where both apply.
constexpr int64_t kSeqWork = 98304;
bool use_seq_path(int32_t batch, int32_t max_blocks, int32_t num_kv_heads) {
  if (max_blocks <= 0 || max_blocks > kSeqMaxBlocks) return false;
  const char* forced = getenv("MI_DECODE_PATH");
  if (forced && strcmp(forced, "stream") == 0) return false;
  if (forced && strcmp(forced, "seq") == 0) return true;
  const int64_t pairs = static_cast<int64_t>(batch) * num_kv_heads;
  const int64_t cus = device_cus();
  return pairs <= cus || (pairs < cus * kPartGroupsPerCu && pairs * max_blocks <= kSeqWork);
}

template <int kKvHeads, int kG, bool kFused>
int32_t launch_decode(const DecodeArgs& a, bool seq_path, hipStream_t s) {
  constexpr int kWaves = kKvHeads < kMaxWaves ? kKvHeads : kMaxWaves;
  constexpr int kHeadGroups = kKvHeads / kWaves;
  const size_t lds = sizeof(int) * (static_cast<size_t>(a.batch) + 1);
  const dim3 pairs(a.batch, kKvHeads);
  if (seq_path) {
    if (a.max_blocks > kSeqMaxBlocks) return fail(MI_ERR_UNSUPPORTED, "mi_paged_decode_attention: table too long");
    const uint32_t groups = static_cast<uint32_t>(a.batch) * a.splits * kKvHeads;
    if (a.part_blocks > 0) {
      paged_decode_parts_kernel<kKvHeads, kG, kFused><<<groups, 64 * kPartWaves, 0, s>>>(a);
      const int32_t rc = check_launch("mi_paged_decode_attention(parts)");
      if (rc != MI_OK || a.splits == 1) return rc;
      paged_decode_merge_kernel<kKvHeads, kG, true><<<pairs, kMergeThreads, 0, s>>>(a);
      return check_launch("mi_paged_decode_attention(merge)");
    }
    if (a.splits == 1) {
      paged_decode_stripe_kernel<kKvHeads, kG, kFused, kStripes><<<groups, 64 * kStripes, 0, s>>>(a);
      return check_launch("mi_paged_decode_attention(stripes)");
    }
    paged_decode_stripe_kernel<kKvHeads, kG, kFused, kStripeWaves><<<groups, 64 * kStripeWaves, 0, s>>>(a);
    const int32_t rc = check_launch("mi_paged_decode_attention(stripes)");
    if (rc != MI_OK) return rc;
    paged_decode_stripe_merge_kernel<kKvHeads, kG><<<pairs, kG * 16 < 64 ? 64 : kG * 16, 0, s>>>(a);
    return check_launch("mi_paged_decode_attention(merge)");
  }
  if constexpr (kFused) return fail(MI_ERR_UNSUPPORTED, "mi_paged_decode_attention: fused form needs the per-sequence kernel");
  if (a.max_blocks > 0) {
    paged_decode_kernel<kKvHeads, kWaves, kG><<<static_cast<uint32_t>(a.streams) * kHeadGroups, 64 * kWaves, lds, s>>>(a);
    int32_t rc = check_launch("mi_paged_decode_attention");
    if (rc != MI_OK) return rc;
  }
  // A sequence spans under two ranges on average: 192 sequences to 8192 tokens 343 / 345 us with the rows form /
  // the other, 128 of them 236 / 229, 16 of 5000-20000 144 / 137, one of 30000 72 / 30.
  if (a.streams < 2 * a.batch)
    paged_decode_merge_rows_kernel<kKvHeads * kG><<<a.batch, merge_rows_threads<kKvHeads * kG>(), 0, s>>>(a);
  else
    paged_decode_merge_kernel<kKvHeads, kG, false><<<pairs, kMergeThreads, 0, s>>>(a);
  return check_launch("mi_paged_decode_attention(merge)");
}

// GQA groups (query heads per KV head) with compiled kernels: Qwen3 dense models use 2 (0.6B,
// 1.7B), 4 (4B, 8B), 5 (14B) and 8 (32B); 1 is multi-head attention.
bool group_supported(int group) { return group == 1 || group == 2 || group == 4 || group == 5 || group == 8; }

template <int kG, bool kFused>
int32_t launch_for_kv_heads(const DecodeArgs& a, int32_t num_kv_heads, bool seq_path, hipStream_t s) {
  switch (num_kv_heads) {
    case 1: return launch_decode<1, kG, kFused>(a, seq_path, s);
    case 2: return launch_decode<2, kG, kFused>(a, seq_path, s);
    case 4: return launch_decode<4, kG, kFused>(a, seq_path, s);
    default: return launch_decode<8, kG, kFused>(a, seq_path, s);
  }
}

template <bool kFused>
int32_t launch_for_heads(const DecodeArgs& a, int32_t num_heads, int32_t num_kv_heads, bool seq_path, hipStream_t s) {
  switch (num_heads / num_kv_heads) {
    case 1: return launch_for_kv_heads<1, kFused>(a, num_kv_heads, seq_path, s);
    case 2: return launch_for_kv_heads<2, kFused>(a, num_kv_heads, seq_path, s);
    case 4: return launch_for_kv_heads<4, kFused>(a, num_kv_heads, seq_path, s);
    case 5: return launch_for_kv_heads<5, kFused>(a, num_kv_heads, seq_path, s);
    default: return launch_for_kv_heads<8, kFused>(a, num_kv_heads, seq_path, s);
  }
}

// Shape checks shared by the entry points; returns MI_OK or the error it recorded.
int32_t check_heads(const char* what, int32_t num_heads, int32_t num_kv_heads, int32_t head_dim, int32_t block_size) {
  if (head_dim != kHeadDim || block_size != kBlockSize || num_kv_heads <= 0 || num_heads <= 0 ||
      num_heads % num_kv_heads != 0)
    return fail(MI_ERR_UNSUPPORTED,
                "%s: needs head_dim %d, block_size %d, num_heads a multiple of num_kv_heads "
                "(got head_dim %d, block_size %d, heads %d/%d)",
                what, kHeadDim, kBlockSize, head_dim, block_size, num_heads, num_kv_heads);
  if (num_kv_heads != 1 && num_kv_heads != 2 && num_kv_heads != 4 && num_kv_heads != 8)
    return fail(MI_ERR_UNSUPPORTED, "%s: num_kv_heads %d not in {1,2,4,8}", what, num_kv_heads);
  if (!group_supported(num_heads / num_kv_heads))
    return fail(MI_ERR_UNSUPPORTED, "%s: %d query heads per KV head not in {1,2,4,5,8}", what,
                num_heads / num_kv_heads);
  return MI_OK;
}

}  // namespace
}  // namespace mi

extern "C" int64_t mi_paged_decode_workspace_bytes(int32_t batch, int32_t max_blocks, int32_t num_heads,
                                                   int32_t num_kv_heads, int32_t head_dim, int32_t block_size) {
  using namespace mi;
  if (batch <= 0 || max_blocks <= 0 || num_heads <= 0 || num_kv_heads <= 0 || head_dim <= 0 ||
      block_size != kBlockSize || num_heads % num_kv_heads != 0)
    return 0;
  const int64_t streams = streams_for(batch, max_blocks, num_kv_heads);
  return streams * 2 * num_heads * (head_dim + 2) * static_cast<int64_t>(sizeof(float));
}

namespace mi {
namespace {

// Whose workspace a launch has.  kShared: the caller's, which other calls may use at the same time while all of
// them are small (at most one (sequence, KV head) pair per CU), so small launches leave it untouched.
// kOwn: this call's alone, so small launches may spread their sequences through it.  kNone: the launch is
// small, needs none and takes none.
enum class Workspace { kShared, kOwn, kNone };

// Small launches, to which the promise of an untouched workspace applies.
bool is_small(int32_t batch, int32_t num_kv_heads) {
  return static_cast<int64_t>(batch) * num_kv_heads <= device_cus();
}

// The checks of mi_paged_decode_attention (batch > 0), which launch nothing.
int32_t check_attention(const void* out, int64_t out_row_stride, const void* query, int64_t query_row_stride,
                        int64_t query_head_stride, const void* key_pool, const void* value_pool, int64_t num_blocks,
                        const int64_t* block_tables, int64_t block_table_stride, int32_t max_blocks,
                        const int64_t* context_lens, int64_t context_lens_stride, int32_t batch, int32_t num_heads,
                        int32_t num_kv_heads, int32_t head_dim, int32_t block_size, const void* workspace,
                        int64_t workspace_bytes, Workspace use) {
  if (const int32_t rc = reject_empty_pool("mi_paged_decode_attention", num_blocks, max_blocks > 0)) return rc;
  if (!out || !query || !key_pool || !value_pool || !context_lens || (max_blocks > 0 && !block_tables))
    return fail(MI_ERR_INVALID_ARGUMENT, "mi_paged_decode_attention: null pointer argument");
  if (const int32_t rc = check_heads("mi_paged_decode_attention", num_heads, num_kv_heads, head_dim, block_size))
    return rc;
  if (!aligned16(out) || !aligned16(query) || !aligned16(key_pool) || !aligned16(value_pool) ||
      out_row_stride % 8 != 0 || query_row_stride % 8 != 0 || query_head_stride % 8 != 0)
    return fail(MI_ERR_UNSUPPORTED, "mi_paged_decode_attention: query/out/pools must be 16-byte aligned");
  if (max_blocks > 0 && block_table_stride < max_blocks)
    return fail(MI_ERR_INVALID_ARGUMENT, "mi_paged_decode_attention: block_table_stride < max_blocks");
  if (context_lens_stride <= 0)
    return fail(MI_ERR_INVALID_ARGUMENT, "mi_paged_decode_attention: context_lens_stride must be > 0");
  if (static_cast<int64_t>(kMaxBatchPerLaunch) * max_blocks >= (1ll << 31))
    return fail(MI_ERR_UNSUPPORTED, "mi_paged_decode_attention: max_blocks %d too large", max_blocks);

  const int64_t need = mi_paged_decode_workspace_bytes(batch, max_blocks, num_heads, num_kv_heads, head_dim, block_size);
  if (use != Workspace::kNone && max_blocks > 0 && (!workspace || workspace_bytes < need))
    return fail(MI_ERR_WORKSPACE, "mi_paged_decode_attention: workspace of %lld bytes needed, got %lld",
                static_cast<long long>(need), static_cast<long long>(workspace_bytes));
  if (use != Workspace::kNone && max_blocks > 0 && !aligned16(workspace))
    return fail(MI_ERR_UNSUPPORTED, "mi_paged_decode_attention: workspace must be 16-byte aligned");
  return MI_OK;
}

// mi_paged_decode_attention.
int32_t decode_attention(void* out, int64_t out_row_stride, const void* query, int64_t query_row_stride,
                         int64_t query_head_stride, const void* key_pool, const void* value_pool, int64_t num_blocks,
                         const int64_t* block_tables, int64_t block_table_stride, int32_t max_blocks,
                         const int64_t* context_lens, int64_t context_lens_stride, int32_t batch, int32_t num_heads,
                         int32_t num_kv_heads, int32_t head_dim, int32_t block_size, float scale, void* workspace,
                         int64_t workspace_bytes, Workspace use, void* stream) {
  if (batch < 0 || max_blocks < 0 || num_blocks < 0)
    return fail(MI_ERR_INVALID_ARGUMENT, "mi_paged_decode_attention: negative size");
  if (batch == 0) return ok();
  if (const int32_t rc = check_attention(out, out_row_stride, query, query_row_stride, query_head_stride, key_pool, value_pool,
                                         num_blocks, block_tables, block_table_stride, max_blocks, context_lens,
                                         context_lens_stride, batch, num_heads, num_kv_heads, head_dim, block_size,
                                         workspace, workspace_bytes, use))
    return rc;
  const int32_t streams = streams_for(batch, max_blocks, num_kv_heads);
  float* ws_acc = static_cast<float*>(workspace);
  float* ws_ml = ws_acc ? ws_acc + static_cast<int64_t>(streams) * 2 * num_heads * kHeadDim : nullptr;

  hipStream_t s = as_stream(stream);
  const bool seq_path = use_seq_path(batch, max_blocks, num_kv_heads);
  const bool cut = use == Workspace::kOwn || !is_small(batch, num_kv_heads);
  // Sequences go in slices of at most kMaxBatchPerLaunch (the per-workgroup prefix sum lives in
  // LDS); the slices reuse the workspace one after the other on the stream.
  for (int32_t b0 = 0; b0 < batch; b0 += kMaxBatchPerLaunch) {
    const int32_t nb = batch - b0 < kMaxBatchPerLaunch ? batch - b0 : kMaxBatchPerLaunch;
    DecodeArgs a{};
    a.out = static_cast<uint16_t*>(out) + b0 * out_row_stride;
    a.out_row = out_row_stride;
    a.query = static_cast<const uint16_t*>(query) + b0 * query_row_stride;
    a.q_row = query_row_stride;
    a.q_head = query_head_stride;
    a.key_pool = static_cast<const uint16_t*>(key_pool);
    a.value_pool = static_cast<const uint16_t*>(value_pool);
    a.num_blocks = num_blocks;
    a.block_tables = block_tables ? block_tables + b0 * block_table_stride : nullptr;
    a.bt_stride = block_table_stride;
    a.context_lens = context_lens + b0 * context_lens_stride;
    a.ctx_stride = context_lens_stride;
    a.batch = nb;
    a.max_blocks = max_blocks;
    a.streams = streams;
    if (seq_path) cut_sequences(a, num_kv_heads, cut);
    a.scale = scale;
    a.ws_acc = ws_acc;
    a.ws_ml = ws_ml;
    const int32_t rc = launch_for_heads<false>(a, num_heads, num_kv_heads, seq_path, s);
    if (rc != MI_OK) return rc;
  }
  return ok();
}

}  // namespace
}  // namespace mi

extern "C" int32_t mi_paged_decode_attention(void* out, int64_t out_row_stride, const void* query,
                                             int64_t query_row_stride, int64_t query_head_stride,
                                             const void* key_pool, const void* value_pool, int64_t num_blocks,
                                             const int64_t* block_tables, int64_t block_table_stride,
                                             int32_t max_blocks, const int64_t* context_lens,
                                             int64_t context_lens_stride, int32_t batch, int32_t num_heads,
                                             int32_t num_kv_heads, int32_t head_dim, int32_t block_size, float scale,
                                             void* workspace, int64_t workspace_bytes, void* stream) {
  return mi::decode_attention(out, out_row_stride, query, query_row_stride, query_head_stride, key_pool, value_pool,
                              num_blocks, block_tables, block_table_stride, max_blocks, context_lens,
                              context_lens_stride, batch, num_heads, num_kv_heads, head_dim, block_size, scale,
                              workspace, workspace_bytes, mi::Workspace::kShared, stream);
}

extern "C" int32_t mi_paged_decode_attention_spread(void* out, int64_t out_row_stride, const void* query,
                                                    int64_t query_row_stride, int64_t query_head_stride,
                                                    const void* key_pool, const void* value_pool, int64_t num_blocks,
                                                    const int64_t* block_tables, int64_t block_table_stride,
                                                    int32_t max_blocks, const int64_t* context_lens,
                                                    int64_t context_lens_stride, int32_t batch, int32_t num_heads,
                                                    int32_t num_kv_heads, int32_t head_dim, int32_t block_size, float scale,
                                                    void* workspace, int64_t workspace_bytes, void* stream) {
  return mi::decode_attention(out, out_row_stride, query, query_row_stride, query_head_stride, key_pool, value_pool,
                              num_blocks, block_tables, block_table_stride, max_blocks, context_lens,
                              context_lens_stride, batch, num_heads, num_kv_heads, head_dim, block_size, scale,
                              workspace, workspace_bytes, mi::Workspace::kOwn, stream);
}

extern "C" int64_t mi_paged_decode_spread_bytes(int32_t batch, int32_t max_blocks, int32_t num_heads,
                                                int32_t num_kv_heads, int32_t head_dim, int32_t block_size) {
  using namespace mi;
  const int64_t need = mi_paged_decode_workspace_bytes(batch, max_blocks, num_heads, num_kv_heads, head_dim, block_size);
  if (need == 0 || !is_small(batch, num_kv_heads) || !use_seq_path(batch, max_blocks, num_kv_heads)) return 0;
  DecodeArgs a{};
  a.batch = batch;
  a.max_blocks = max_blocks;
  cut_sequences(a, num_kv_heads, true);
  return a.splits > 1 ? need : 0;
}

namespace mi {
namespace {

// mi_paged_decode_attention_fused.
int32_t decode_attention_fused(
    void* out, int64_t out_row_stride, const void* q, int64_t q_row_stride, const void* k, int64_t k_row_stride,
    const void* v, int64_t v_row_stride, const void* q_weight, const void* k_weight, const void* cos, const void* sin,
    float eps, const int64_t* slot_mapping, int64_t slot_stride, void* key_pool, void* value_pool, int64_t num_blocks,
    const int64_t* block_tables, int64_t block_table_stride, int32_t max_blocks, const int64_t* context_lens,
    int64_t context_lens_stride, int32_t batch, int32_t num_heads, int32_t num_kv_heads, int32_t head_dim,
    int32_t block_size, float scale, void* q_scratch, void* workspace, int64_t workspace_bytes, Workspace use,
    void* stream) {
  if (batch < 0 || max_blocks < 0 || num_blocks < 0)
    return fail(MI_ERR_INVALID_ARGUMENT, "mi_paged_decode_attention_fused: negative size");
  if (batch == 0) return ok();
  if (const int32_t rc = reject_empty_pool("mi_paged_decode_attention_fused", num_blocks, max_blocks > 0)) return rc;
  if (!q || !k || !v || !q_weight || !k_weight || !cos || !sin || !slot_mapping || !q_scratch)
    return fail(MI_ERR_INVALID_ARGUMENT, "mi_paged_decode_attention_fused: null pointer argument");
  if (num_blocks > INT64_MAX / kBlockSize)
    return fail(MI_ERR_INVALID_ARGUMENT, "mi_paged_decode_attention_fused: pool too large");
  if (const int32_t rc = check_heads("mi_paged_decode_attention_fused", num_heads, num_kv_heads, head_dim, block_size))
    return rc;
  // Rows may share blocks (two tokens of one sequence as two rows, one token apart): a launch of more pairs
  // than CUs appends in a launch of its own, before any row reads.  Up to one pair per CU each row's slot has
  // to be its own (the entry point's contract), and only its own workgroups put its rows in place.
  const bool small = is_small(batch, num_kv_heads);
  // The prologue of the per-sequence kernel moves 16-byte pieces of the projection rows and tables.
  const bool pieces = aligned16(q) && aligned16(k) && aligned16(v) && aligned16(q_weight) && aligned16(k_weight) &&
                      aligned16(cos) && aligned16(sin) && q_row_stride % 8 == 0 && k_row_stride % 8 == 0 &&
                      v_row_stride % 8 == 0;
  const int64_t need = mi_paged_decode_workspace_bytes(batch, max_blocks, num_heads, num_kv_heads, head_dim, block_size);
  // Where a small launch may cut its sequences; without that they stay whole.
  const bool room = use == Workspace::kOwn && workspace && workspace_bytes >= need && aligned16(workspace);
  const bool sequences = small && use_seq_path(batch, max_blocks, num_kv_heads);  // the per-sequence kernels serve it
  if (!sequences || !pieces) {
    // The append and q rotation in a launch of their own (large launches; rows of other alignments), once
    // nothing can refuse the attention after it.
    const Workspace given = sequences && !room ? Workspace::kNone : use;
    const int64_t q_head = head_dim, q_row = num_heads * q_head;
    int32_t rc = check_attention(out, out_row_stride, q_scratch, q_row, q_head, key_pool, value_pool, num_blocks,
                                 block_tables, block_table_stride, max_blocks, context_lens, context_lens_stride, batch,
                                 num_heads, num_kv_heads, head_dim, block_size, workspace, workspace_bytes, given);
    if (rc != MI_OK) return rc;
    rc = mi_qk_norm_rope(q_scratch, nullptr, nullptr, q, q_row_stride, k, k_row_stride, v, v_row_stride,
                                 q_weight, k_weight, cos, sin, batch, num_heads, num_kv_heads, head_dim, eps,
                                 slot_mapping, slot_stride, key_pool, value_pool, num_blocks * block_size, stream);
    if (rc != MI_OK) return rc;
    return decode_attention(out, out_row_stride, q_scratch, q_row, q_head, key_pool, value_pool, num_blocks, block_tables,
                            block_table_stride, max_blocks, context_lens, context_lens_stride, batch, num_heads,
                            num_kv_heads, head_dim, block_size, scale, workspace, workspace_bytes, given, stream);
  }
  // The per-sequence kernel with the prologue.  Shape checks as in the two entry points.
  if (!out || !key_pool || !value_pool || !context_lens || !block_tables)
    return fail(MI_ERR_INVALID_ARGUMENT, "mi_paged_decode_attention_fused: null pointer argument");
  if (!aligned16(out) || !aligned16(key_pool) || !aligned16(value_pool) || out_row_stride % 8 != 0)
    return fail(MI_ERR_UNSUPPORTED, "mi_paged_decode_attention_fused: out/pools must be 16-byte aligned");
  if (block_table_stride < max_blocks || context_lens_stride <= 0 || q_row_stride < num_heads * head_dim ||
      k_row_stride < num_kv_heads * head_dim || v_row_stride < num_kv_heads * head_dim)
    return fail(MI_ERR_INVALID_ARGUMENT, "mi_paged_decode_attention_fused: bad stride");
  DecodeArgs a{};
  a.out = static_cast<uint16_t*>(out);
  a.out_row = out_row_stride;
  a.key_pool = static_cast<const uint16_t*>(key_pool);
  a.value_pool = static_cast<const uint16_t*>(value_pool);
  a.num_blocks = num_blocks;
  a.block_tables = block_tables;
  a.bt_stride = block_table_stride;
  a.context_lens = context_lens;
  a.ctx_stride = context_lens_stride;
  a.batch = batch;
  a.max_blocks = max_blocks;
  a.streams = 1;
  cut_sequences(a, num_kv_heads, room);
  if (room) {
    a.ws_acc = static_cast<float*>(workspace);
    a.ws_ml = a.ws_acc + static_cast<int64_t>(streams_for(batch, max_blocks, num_kv_heads)) * 2 * num_heads * kHeadDim;
  }
  a.scale = scale;
  a.q_raw = static_cast<const uint16_t*>(q);
  a.k_raw = static_cast<const uint16_t*>(k);
  a.v_raw = static_cast<const uint16_t*>(v);
  a.q_raw_row = q_row_stride;
  a.k_raw_row = k_row_stride;
  a.v_raw_row = v_row_stride;
  a.q_weight = static_cast<const uint16_t*>(q_weight);
  a.k_weight = static_cast<const uint16_t*>(k_weight);
  a.cos = static_cast<const uint16_t*>(cos);
  a.sin = static_cast<const uint16_t*>(sin);
  a.slot_mapping = slot_mapping;
  a.slot_stride = slot_stride;
  a.num_slots = num_blocks * kBlockSize;
  a.eps = eps;
  return launch_for_heads<true>(a, num_heads, num_kv_heads, true, as_stream(stream));
}

}  // namespace
}  // namespace mi

extern "C" int32_t mi_paged_decode_attention_fused(
    void* out, int64_t out_row_stride, const void* q, int64_t q_row_stride, const void* k, int64_t k_row_stride,
    const void* v, int64_t v_row_stride, const void* q_weight, const void* k_weight, const void* cos, const void* sin,
    float eps, const int64_t* slot_mapping, int64_t slot_stride, void* key_pool, void* value_pool, int64_t num_blocks,
    const int64_t* block_tables, int64_t block_table_stride, int32_t max_blocks, const int64_t* context_lens,
    int64_t context_lens_stride, int32_t batch, int32_t num_heads, int32_t num_kv_heads, int32_t head_dim,
    int32_t block_size, float scale, void* q_scratch, void* workspace, int64_t workspace_bytes, void* stream) {
  return mi::decode_attention_fused(
      out, out_row_stride, q, q_row_stride, k, k_row_stride, v, v_row_stride, q_weight, k_weight, cos, sin, eps,
      slot_mapping, slot_stride, key_pool, value_pool, num_blocks, block_tables, block_table_stride, max_blocks,
      context_lens, context_lens_stride, batch, num_heads, num_kv_heads, head_dim, block_size, scale, q_scratch,
      workspace, workspace_bytes, mi::Workspace::kShared, stream);
}

extern "C" int32_t mi_paged_decode_attention_fused_spread(
    void* out, int64_t out_row_stride, const void* q, int64_t q_row_stride, const void* k, int64_t k_row_stride,
    const void* v, int64_t v_row_stride, const void* q_weight, const void* k_weight, const void* cos, const void* sin,
    float eps, const int64_t* slot_mapping, int64_t slot_stride, void* key_pool, void* value_pool, int64_t num_blocks,
    const int64_t* block_tables, int64_t block_table_stride, int32_t max_blocks, const int64_t* context_lens,
    int64_t context_lens_stride, int32_t batch, int32_t num_heads, int32_t num_kv_heads, int32_t head_dim,
    int32_t block_size, float scale, void* q_scratch, void* workspace, int64_t workspace_bytes, void* stream) {
  return mi::decode_attention_fused(
      out, out_row_stride, q, q_row_stride, k, k_row_stride, v, v_row_stride, q_weight, k_weight, cos, sin, eps,
      slot_mapping, slot_stride, key_pool, value_pool, num_blocks, block_tables, block_table_stride, max_blocks,
      context_lens, context_lens_stride, batch, num_heads, num_kv_heads, head_dim, block_size, scale, q_scratch,
      workspace, workspace_bytes, mi::Workspace::kOwn, stream);
}

// ---- The no-allocation variant.  The partials of sequences that the stream or the parts kernel cuts go to
// `scratch`, a fixed device array of this library (each GPU holds its own copy for the life of the
// process), instead of a caller workspace.  No part of it needs clearing: a partial slot is written
// before the merge launch uses it.  Every call on one GPU shares the array, so calls that overlap on
// one GPU (different streams, or threads) race on it.
namespace mi {
namespace {
constexpr int64_t kScratchBytes = MI_PAGED_NOALLOC_SCRATCH_BYTES;  // 4.3 MB used at 16 / 8 heads on 256 CUs
constexpr int kMaxScratchDevices = 64;
}  // namespace
}  // namespace mi

static __device__ __align__(256) unsigned char scratch[mi::kScratchBytes];

namespace mi {
namespace {

// Device address of `scratch` on the current device, looked up once per device with that device
// current (the array's name is only a host-side stand-in for it).
int32_t scratch_on_current_device(void** out) {
  static std::mutex mu;
  static void* ptrs[kMaxScratchDevices] = {nullptr};
  int dev = 0;
  const hipError_t derr = hipGetDevice(&dev);
  if (derr != hipSuccess)
    return fail(MI_ERR_DEVICE, "mi_paged_decode_attention_noalloc: hipGetDevice: %s", hipGetErrorString(derr));
  if (dev < 0 || dev >= kMaxScratchDevices)
    return fail(MI_ERR_UNSUPPORTED, "mi_paged_decode_attention_noalloc: device %d beyond %d", dev, kMaxScratchDevices);
  std::lock_guard<std::mutex> lock(mu);
  if (ptrs[dev] == nullptr) {
    void* p = nullptr;
    const hipError_t err = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (err != hipSuccess || p == nullptr)
      return fail(MI_ERR_DEVICE, "mi_paged_decode_attention_noalloc: hipGetSymbolAddress(scratch): %s",
                  hipGetErrorString(err));
    ptrs[dev] = p;
  }
  *out = ptrs[dev];
  return MI_OK;
}

}  // namespace
}  // namespace mi

extern "C" int32_t mi_paged_decode_attention_noalloc(void* out, int64_t out_row_stride, const void* query,
                                                     int64_t query_row_stride, int64_t query_head_stride,
                                                     const void* key_pool, const void* value_pool, int64_t num_blocks,
                                                     const int64_t* block_tables, int64_t block_table_stride,
                                                     int32_t max_blocks, const int64_t* context_lens,
                                                     int64_t context_lens_stride, int32_t batch, int32_t num_heads,
                                                     int32_t num_kv_heads, int32_t head_dim, int32_t block_size,
                                                     float scale, void* stream) {
  using namespace mi;
  if (batch < 0 || max_blocks < 0 || num_blocks < 0)
    return fail(MI_ERR_INVALID_ARGUMENT, "mi_paged_decode_attention_noalloc: negative size");
  if (batch == 0) return ok();
  if (const int32_t rc = reject_empty_pool("mi_paged_decode_attention_noalloc", num_blocks, max_blocks > 0))
    return rc;
  if (const int32_t rc = check_heads("mi_paged_decode_attention_noalloc", num_heads, num_kv_heads, head_dim,
                                     block_size))
    return rc;
  // The size check comes before any launch, copy or scratch lookup (it only queries the current
  // device and its CU count): a launch that needs more than the fixed array is rejected before
  // any work reaches the GPU.
  const int64_t need =
      mi_paged_decode_workspace_bytes(batch, max_blocks, num_heads, num_kv_heads, head_dim, block_size);
  if (need > kScratchBytes)
    return fail(MI_ERR_WORKSPACE,
                "mi_paged_decode_attention_noalloc: this launch needs %lld bytes of scratch, the fixed array "
                "holds %lld (use mi_paged_decode_attention with a workspace)",
                static_cast<long long>(need), static_cast<long long>(kScratchBytes));
  void* ws = nullptr;
  if (need > 0) {
    if (const int32_t rc = scratch_on_current_device(&ws)) return rc;
  }
  return mi_paged_decode_attention(out, out_row_stride, query, query_row_stride, query_head_stride, key_pool,
                                   value_pool, num_blocks, block_tables, block_table_stride, max_blocks, context_lens,
                                   context_lens_stride, batch, num_heads, num_kv_heads, head_dim, block_size, scale,
                                   ws, need > 0 ? kScratchBytes : 0, stream);
}
