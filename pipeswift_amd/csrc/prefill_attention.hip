// Prefill attention over the FP8 E4M3FN KV cache for MI355X (gfx950): the same
// attention as the decode reader of paged_attention.hip, for steps with many
// query tokens per sequence.  The kernel here gives every query block a
// workgroup of its own; prefill_runs.hip holds the one that cuts the step into
// equal runs; prefers_runs() says which is faster, here where the bounds on the
// lengths settle it and on the device where they do not.
//
// C ABI: include/pipeswift_kv.h.  Nothing here allocates or synchronizes.

#include <algorithm>
#include <cmath>
#include <type_traits>

#include "prefill_runs.h"

using namespace psk_detail;

namespace {

// psk_paged_prefill_attention computes what the decode reader computes, for
// sequences with more query rows per kv head than one 16-row MFMA tile holds
// (prefill, chunked prefill, long speculative drafts, groups of more than 16
// query heads).  One workgroup per (query block, kv head): kPfWaves waves of
// kPfSets sets of 16 MFMA rows, kPfRows rows in all; row r is query token
// i0 + r / G, query head g = r % G of the block's tq = kPfRows / G tokens, so
// every K/V row of the block's keys is read from the cache once per tq query
// tokens.  The keys stream through two LDS stages of kPfKeys keys, filled by
// the first wave of each SIMD (two 16-byte chunks of K and two of V per
// thread, converted once, exactly, K to bf16 and V to fp16) and consumed by
// every wave, as 256-byte rows:
//   * K: 16-byte chunk c of key t at chunk c ^ (t & 15), so the lanes of one
//     ds_read_b128 phase (consecutive keys, one chunk) hit distinct banks;
//   * V: chunk c of key t at c ^ (2 (t & 7)), read transposed by
//     ds_read_b64_tr_b16 (four keys of one column per lane and read).
// Per 32 keys and 16 rows: S^T = K Q^T on v_mfma_f32_16x16x32_bf16 (two
// 16-key tiles, four MFMAs each, exactly converted FP8 operands as in the
// decode reader), the softmax in the exp2 domain, then O^T = V^T P^T on
// v_mfma_f32_16x16x32_f16 with P rounded to fp16 once (11 significant bits,
// where the decode reader keeps ~16 in a bf16 hi + lo pair and runs P V
// twice; FA3's FP8 path keeps 4).  Transposed products leave each
// lane one query row (lane % 16): its scores, maximum and sum, and output
// columns 16 b + 4 (lane / 16) + r.  The 32-key MFMA step takes as its
// k = 8 s + j (s = lane / 16) key 4 s + j of the first 16-key tile for j < 4
// and key 4 s + j - 4 of the second for j >= 4: the lane's S^T results of the
// two tiles are then its P^T operand as they stand, and one transposed V read
// per tile gives the matching V^T operand.  A row's maximum is fixed by its
// first 32 keys (see the kernel), so the loop has no rescale.
constexpr int kPfWaves = 8;
constexpr int kPfSets = 2;
constexpr int kPfRows = kPfWaves * kPfSets * 16;
constexpr int kPfKeys = 64;  // keys per LDS stage
constexpr int kPfThreads = kPfWaves * 64;
// The first wave of each SIMD loads, converts and stores the stages.  Waves
// w and w + kPfWaves / 2 share a SIMD; the older one issues first and ends
// its blocks of a stage about a quarter of a stage early, so giving it all
// the staging work evens the two out at the barrier.
constexpr int kPfLoaders = kPfThreads / 2;
constexpr int kPfLoads = kPfKeys * 8 / kPfLoaders;  // 16-byte chunks of K (and of V) per loader per stage
static_assert(kPfKeys % 32 == 0 && kPfLoads >= 1 && kPfLoads * kPfLoaders == kPfKeys * 8,
              "a stage is whole 32-key blocks, its chunks spread evenly over the loaders");

static_assert(kPfRows == kBlockRows && kPfThreads == kRunThreads, "the blocks of both prefill kernels are the same");

struct PrefillArgs {
  DecodeArgs a;
  const int32_t* blocks;  // [num_seqs + 1]: query blocks before launch position k; the total last
  const int32_t* order;   // [num_seqs]: the sequence at launch position k
  int32_t num_seqs;
  int32_t tq;             // query tokens per block
  int32_t narrow;         // K/V page and row strides below 2^32: offsets from 32 x 32-bit products
};

__global__ void __launch_bounds__(1024) prefill_blocks_kernel(DecodeArgs a, int num_seqs, int tq, int32_t* blocks,
                                                              int32_t* order) {
  __shared__ OrderLds lds;
  if (num_seqs <= kOrderMax) {
    const int b = int(threadIdx.x);
    if (b < num_seqs) put_sequence(lds, b, q_count(a, b), max(a.seq_lens[b], 0));
    __syncthreads();
  }
  order_blocks<1024>(a, num_seqs, tq, blocks, order, lds);
}

// The launch position of query block u (blocks[0] = 0 <= u < blocks[num_seqs]):
// the last k with blocks[k] <= u, by a 64-way search of the wave (one round up
// to 64 sequences, two up to 4096).
__device__ __forceinline__ int block_sequence(const int32_t* blocks, int num_seqs, int u, int lane) {
  int lo = 0, n = num_seqs;  // the answer lies in [lo, lo + n) and blocks[lo] <= u
  while (n > 1) {
    const int step = (n + 63) / 64;
    const bool le = lane * step < n && blocks[lo + lane * step] <= u;  // true on a prefix of the lanes
    const uint64_t m = __ballot(le);
    const int last = 63 - __builtin_clzll(m);
    lo += last * step;
    n = min(step, n - last * step);
  }
  return lo;
}

template <int OUT_DT>
__device__ __forceinline__ void store_row4(char* dst, f32x4 v);
template <>
__device__ __forceinline__ void store_row4<PSK_DTYPE_F32>(char* dst, f32x4 v) {
  *reinterpret_cast<f32x4*>(dst) = v;
}
template <>
__device__ __forceinline__ void store_row4<PSK_DTYPE_BF16>(char* dst, f32x4 v) {
  using E = Elt<PSK_DTYPE_BF16>;
  const uint32_t lo = uint32_t(E::from_f32(v[0])) | (uint32_t(E::from_f32(v[1])) << 16);
  const uint32_t hi = uint32_t(E::from_f32(v[2])) | (uint32_t(E::from_f32(v[3])) << 16);
  typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
  *reinterpret_cast<u32x2*>(dst) = u32x2{lo, hi};
}

struct StageLds {
  u32x4 k[2][kPfKeys * 16];  // bf16 K rows, chunk c of key t at c ^ (t & 15)
  u32x4 v[2][kPfKeys * 16];  // fp16 V rows, chunk c of key t at c ^ (2 (t & 7))
};

// One workgroup's query block, of `total`.
template <int Q_DT, int OUT_DT>
__device__ __forceinline__ void attend_block(const PrefillArgs& p, int total, StageLds& lds) {
  const DecodeArgs& a = p.a;
  auto& s_k = lds.k;
  auto& s_v = lds.v;
  const int lane = int(threadIdx.x) & 63;
  const int wave = __builtin_amdgcn_readfirstlane(int(threadIdx.x) >> 6);
  const int Hkv = a.num_kv_heads;
  const int idx = int(blockIdx.x) / Hkv, h = int(blockIdx.x) - idx * Hkv;
  if (idx >= total) return;
  const int k = __builtin_amdgcn_readfirstlane(block_sequence(p.blocks, p.num_seqs, idx, lane));
  const int b = p.order[k];
  // a sequence's blocks from its last (the most keys, when causal) to its first
  const int i0 = (p.blocks[k + 1] - 1 - idx) * p.tq;
  const int n = q_count(a, b);
  const int ni = min(p.tq, n - i0);
  const int64_t qf = q_first(a, b);
  const int L = max(a.seq_lens[b], 0);
  const int G = a.heads;
  // causal: query token i sees keys below base + i (FA's bottom-right alignment)
  const int base = a.causal ? L - n + 1 : L;
  const int key_end = a.causal ? min(max(base + i0 + ni - 1, 0), L) : L;  // keys any row of the block sees
  const int mask_from = a.causal ? min(max(base + i0, 0), L) : L;         // keys every row sees
  const float qd = descale(a.qd, a.qd_b, a.qd_h, b, h);
  const float kd = descale(a.kd, a.kd_b, a.kd_h, b, h);
  const float vd = descale(a.vd, a.vd_b, a.vd_h, b, h);
  // exp2-domain score scale; a negative one is applied as -q~ (exact) times |sl|
  const float sl_signed = a.scale_log2 * qd * kd;
  const float sl = __builtin_fabsf(sl_signed);

  int row_lim[kPfSets];
  bf16x8 qop[kPfSets][4];
#pragma unroll
  for (int s = 0; s < kPfSets; ++s) {
    const int r = (wave * kPfSets + s) * 16 + (lane & 15);
    const int ti = r / G, g = r - ti * G;
    const bool live = ti < ni;
    row_lim[s] = live ? (a.causal ? min(max(base + i0 + ti, 0), L) : L) : 0;
    uint32_t qw[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) qw[i] = 0;
    if (live)
      load_query_as<Q_DT>(a.q + (qf + i0 + ti) * a.q_tok_stride + int64_t(h * G + g) * a.q_head_stride, qd,
                          32 * (lane >> 4), qw);
    if (sl_signed < 0.0f) {
#pragma unroll
      for (int i = 0; i < 8; ++i) qw[i] ^= 0x80808080u;  // -q~: E4M3 sign bits
    }
#pragma unroll
    for (int c = 0; c < 4; ++c) qop[s][c] = e4m3x8_to_bf16(qw[2 * c], qw[2 * c + 1]);
  }
  // Softmax state per row set.  m is fixed by the row's first 32 keys and
  // never raised, so the hot loop has no rescale and checks nothing: while
  // every lane's share of a row's sum stays below 2^kPfHeadroom, every p
  // (each below that too) is a finite fp16 value (at most 65504) and every
  // sum and accumulator is finite.  A score
  // far above the first keys' maximum makes a share reach it (or overflow),
  // and the workgroup then redoes the row with exact maxima: a pass for the
  // maxima, then the accumulation again.  Rows without a query token keep
  // m = +kBig (every p is 0).
  constexpr float kPfHeadroom = 15.0f;
  constexpr float kBig = 1.0e30f;
  float m[kPfSets], l[kPfSets];
  f32x4 o[kPfSets][8];
  bool live_row[kPfSets];
#pragma unroll
  for (int s = 0; s < kPfSets; ++s) live_row[s] = ((wave * kPfSets + s) * 16 + (lane & 15)) / G < ni;
  auto reset = [&](float m0) {
#pragma unroll
    for (int s = 0; s < kPfSets; ++s) {
      m[s] = live_row[s] ? m0 : kBig;
      l[s] = 0.0f;
#pragma unroll
      for (int c = 0; c < 8; ++c) o[s][c] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    }
  };

  // loads, by the loader waves (threads below kPfLoaders): chunk i =
  // threadIdx.x + u * kPfLoaders of a stage (u < kPfLoads) is 16-byte chunk
  // i & 7 of key i >> 3, of K and of V; keys past key_end and rows on
  // missing pages load as zeros
  const int lc = int(threadIdx.x) & 7;
  auto lkey = [&](int u) { return (int(threadIdx.x) + u * kPfLoaders) >> 3; };
  const bool loader = wave < kPfLoaders / 64;
  const int32_t* bt_row = a.block_table + int64_t(b) * a.bt_stride;
  // the table entry as stored (range-checked where it is used, a stage
  // later: a check here would wait for the load, and with it for the K/V
  // loads issued before it)
  auto page_id = [&](int t, int u) -> int32_t {
    const int key = t * kPfKeys + lkey(u);
    if (key >= key_end) return -1;
    const int pi = page_index(a, key);
    return pi < a.bt_width ? bt_row[pi] : -1;
  };
  const uint8_t* kbase = a.k + int64_t(h) * a.k_head + 16 * lc;
  const uint8_t* vbase = a.v + int64_t(h) * a.v_head + 16 * lc;
  auto fetch = [&](int t, int u, int32_t pid, u32x4& kr, u32x4& vr) {
    kr = u32x4(0);
    vr = u32x4(0);
    if (pid >= 0 && pid < a.num_blocks) {
      const int key = t * kPfKeys + lkey(u);
      const int row = a.bs_shift >= 0 ? key & (a.block_size - 1) : key - page_index(a, key) * a.block_size;
      uint64_t ko, vo;
      if (p.narrow) {  // two v_mad_u64_u32 each
        ko = uint64_t(uint32_t(pid)) * uint32_t(a.k_blk) + uint64_t(uint32_t(row)) * uint32_t(a.k_row);
        vo = uint64_t(uint32_t(pid)) * uint32_t(a.v_blk) + uint64_t(uint32_t(row)) * uint32_t(a.v_row);
      } else {
        ko = uint64_t(int64_t(pid) * a.k_blk + int64_t(row) * a.k_row);
        vo = uint64_t(int64_t(pid) * a.v_blk + int64_t(row) * a.v_row);
      }
      kr = *reinterpret_cast<const u32x4*>(kbase + ko);
      vr = *reinterpret_cast<const u32x4*>(vbase + vo);
    }
  };
  // K as bf16 and V as fp16 (both exact), converted once here for every wave
  auto stage_store = [&](int st, int u, const u32x4& kr, const u32x4& vr) {
    const int lk = lkey(u);
    const int ks = lk & 15, vs = 2 * (lk & 7);
    s_k[st][lk * 16 + ((2 * lc) ^ ks)] = __builtin_bit_cast(u32x4, e4m3x8_to_bf16(kr[0], kr[1]));
    s_k[st][lk * 16 + ((2 * lc + 1) ^ ks)] = __builtin_bit_cast(u32x4, e4m3x8_to_bf16(kr[2], kr[3]));
    s_v[st][lk * 16 + ((2 * lc) ^ vs)] = __builtin_bit_cast(u32x4, e4m3x8_to_f16(vr[0], vr[1]));
    s_v[st][lk * 16 + ((2 * lc + 1) ^ vs)] = __builtin_bit_cast(u32x4, e4m3x8_to_f16(vr[2], vr[3]));
  };

  // read side.  K (the A operand of S^T): key kx = lane % 16 of a 16-key
  // tile, chunk 4 (lane / 16) + c for MFMA c.  V^T (the A operand of O^T):
  // ds_read_b64_tr_b16 gives lane i of a 16-lane group element j of the row
  // that lane 4 j + i / 4 of the group addressed, at its element i % 4; lane
  // r of group s addresses key 4 s + r / 4 of the tile, columns 16 c + 4 (r %
  // 4) .. + 3 (chunk 2 c + (r % 4) / 2, half r % 2), so lane i receives column
  // 16 c + i of keys 4 s .. 4 s + 3.
  const int kx = lane & 15, kc0 = 4 * (lane >> 4);
  const int vkey = 4 * (lane >> 4) + (kx >> 2);  // this lane's V row in a 16-key tile
  const uint32_t vrow = uint32_t(256 * vkey + 8 * (kx & 1));
  const int vq = (kx & 3) >> 1, vsw = 2 * (vkey & 7);  // keys 16 j + vkey: (vkey & 7) is the tile-free swizzle

  // raw scores y = q~ . K of the 32 keys from key0 (-inf where masked), the
  // lane's 8 of each row set
  auto scores = [&](auto masked_tag, int st, int key0, int kb, float (&y)[kPfSets][8]) {
    constexpr bool MASKED = decltype(masked_tag)::value;
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int kk = 32 * kb + 16 * j + kx;
      bf16x8 kop[4];
#pragma unroll
      for (int c = 0; c < 4; ++c) kop[c] = __builtin_bit_cast(bf16x8, s_k[st][kk * 16 + ((kc0 + c) ^ kx)]);
#pragma unroll
      for (int s = 0; s < kPfSets; ++s) {
        f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int c = 0; c < 4; ++c) acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kop[c], qop[s][c], acc, 0, 0, 0);
#pragma unroll
        for (int r = 0; r < 4; ++r)
          y[s][4 * j + r] = !MASKED || key0 + 16 * j + kc0 + r < row_lim[s] ? acc[r] : -__builtin_inff();
      }
    }
  };
  // a lane's largest scaled score of a set (sl >= 0: max(y) * sl); IEEE
  // maximum, so no canonicalizing moves, and a NaN score propagates
  auto lane_max = [&](const float (&y)[8]) {
    return __builtin_elementwise_maximum(
               __builtin_elementwise_maximum(__builtin_elementwise_maximum(y[0], y[1]),
                                             __builtin_elementwise_maximum(y[2], y[3])),
               __builtin_elementwise_maximum(__builtin_elementwise_maximum(y[4], y[5]),
                                             __builtin_elementwise_maximum(y[6], y[7]))) * sl;
  };
  auto row_max = [&](float v) {
    v = __builtin_fmaxf(v, __shfl_xor(v, 16));
    return __builtin_fmaxf(v, __shfl_xor(v, 32));
  };
  // FIRST: the block fixes m (the row's maximum of these keys)
  auto block = [&](auto masked_tag, auto first_tag, int st, int key0, int kb) {
    constexpr bool MASKED = decltype(masked_tag)::value;
    constexpr bool FIRST = decltype(first_tag)::value;
    float y[kPfSets][8];
    scores(masked_tag, st, key0, kb, y);
    const char* vb = reinterpret_cast<const char*>(&s_v[st][0]) + 256 * 32 * kb;
    // set by set: set s + 1's softmax (VALU) is independent of set s's P V
    // (MFMA), so the two overlap; V^T is read again for each set rather than
    // held in registers
#pragma unroll
    for (int s = 0; s < kPfSets; ++s) {
      if constexpr (FIRST) m[s] = live_row[s] ? __builtin_fmaxf(row_max(lane_max(y[s])), kNegBig) : kBig;
      // P rounded to fp16 (RNE, relative error <= 2^-11 from 2^-14 up; every
      // p is below 2^15 in the pass that is kept, see the headroom)
      float pv[8], ps = 0.0f;
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const float e = __builtin_fmaf(y[s][i], sl, -m[s]);
        pv[i] = __builtin_amdgcn_exp2f(MASKED && y[s][i] == -__builtin_inff() ? -__builtin_inff() : e);
        ps += pv[i];
      }
      l[s] += ps;
      uint32_t pw[4];
#pragma unroll
      for (int i = 0; i < 4; ++i)
        pw[i] = __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2{pv[2 * i], pv[2 * i + 1]}), f16x2));
      const f16x8 pop = __builtin_bit_cast(f16x8, u32x4{pw[0], pw[1], pw[2], pw[3]});
#pragma unroll
      for (int c = 0; c < 8; ++c) {
        const uint32_t off = vrow + uint32_t(16 * ((2 * c + vq) ^ vsw));
        const s16x4 t0 =
            __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4*)(vb + off));
        const s16x4 t1 =
            __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4*)(vb + 256 * 16 + off));
        const f16x8 vop = __builtin_bit_cast(f16x8, __builtin_shufflevector(t0, t1, 0, 1, 2, 3, 4, 5, 6, 7));
        o[s][c] = __builtin_amdgcn_mfma_f32_16x16x32_f16(vop, pop, o[s][c], 0, 0, 0);
      }
    }
    // Ask the scheduler to alternate one MFMA with up to four VALU
    // instructions over the block's 32 MFMAs, so that each wave's softmax
    // issues under its own matrix work as well as under the other wave's.
    // With P V run twice (P as bf16 hi + lo) this was 2-3 % faster on three
    // boxes; with P in fp16, one MFMA to 2, 3 or 4 VALU and no hint measure
    // within 1.5 % of each other and six VALU 2 % slower.
    constexpr int kBlockMfmas = kPfSets * (8 + 8);  // per set: S^T 2 x 4, then P V 8
#pragma unroll
    for (int i = 0; i < kBlockMfmas; ++i) {
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);  // one MFMA
      __builtin_amdgcn_sched_group_barrier(0x002, 4, 0);  // up to four VALU
    }
  };
  // the maxima pass of a redo: the lane's largest scaled score per set into m
  auto block_max = [&](auto masked_tag, int st, int key0, int kb) {
    float y[kPfSets][8];
    scores(masked_tag, st, key0, kb, y);
#pragma unroll
    for (int s = 0; s < kPfSets; ++s) m[s] = __builtin_fmaxf(m[s], lane_max(y[s]));
  };

  // The keys of the block stream through two LDS stages: the loads of stage
  // t + 1 fly while stage t is consumed, and the page id of stage t + 2 while
  // those land.  Stage 0, the stages every row sees whole and the rest (the
  // causal band and the end of the keys) each run as straight-line code over
  // their 32-key blocks; every wave takes the same (uniform) path, so the
  // barriers match.
  const int n_tiles = (key_end + kPfKeys - 1) / kPfKeys;
  const int t_open = min(n_tiles, mask_from / kPfKeys);  // stages [0, t_open) need no mask
  using T = std::true_type;
  using F = std::false_type;
  // one stage's 32-key blocks.  MODE 0: the pass with m fixed by the first
  // block (FIRST); 1: the maxima of a redo; 2: the accumulation of a redo (m
  // exact)
  auto run_stage = [&](auto mode, auto masked_tag, auto first_tag, int st, int t) {
    constexpr int MODE = decltype(mode)::value;
#pragma unroll
    for (int kb = 0; kb < kPfKeys / 32; ++kb) {
      const int key0 = t * kPfKeys + 32 * kb;
      if (decltype(masked_tag)::value && key0 >= key_end) break;
      if constexpr (MODE == 1) {
        block_max(masked_tag, st, key0, kb);
      } else if (kb == 0) {
        block(masked_tag, first_tag, st, key0, kb);
      } else {
        block(masked_tag, F{}, st, key0, kb);
      }
    }
  };
  auto stream = [&](auto mode) {
    u32x4 kr[kPfLoads], vr[kPfLoads];
    int32_t pid_next[kPfLoads];
#pragma unroll
    for (int u = 0; u < kPfLoads; ++u) pid_next[u] = -1;
    if (n_tiles > 0 && loader) {
      int32_t pid0[kPfLoads];
#pragma unroll
      for (int u = 0; u < kPfLoads; ++u) {
        pid0[u] = page_id(0, u);
        pid_next[u] = n_tiles > 1 ? page_id(1, u) : -1;
      }
#pragma unroll
      for (int u = 0; u < kPfLoads; ++u) fetch(0, u, pid0[u], kr[u], vr[u]);
#pragma unroll
      for (int u = 0; u < kPfLoads; ++u) stage_store(0, u, kr[u], vr[u]);
    }
    __syncthreads();
    auto stage = [&](int t, auto masked_tag, auto first_tag) {
      const bool more = t + 1 < n_tiles && loader;
      if (more) {
#pragma unroll
        for (int u = 0; u < kPfLoads; ++u) fetch(t + 1, u, pid_next[u], kr[u], vr[u]);
#pragma unroll
        for (int u = 0; u < kPfLoads; ++u) pid_next[u] = t + 2 < n_tiles ? page_id(t + 2, u) : -1;
      }
      run_stage(mode, masked_tag, first_tag, t & 1, t);
      if (more) {
#pragma unroll
        for (int u = 0; u < kPfLoads; ++u) stage_store((t + 1) & 1, u, kr[u], vr[u]);
      }
      __syncthreads();
    };
    constexpr bool kFirst = decltype(mode)::value == 0;
    if (n_tiles > 0) {
      if (t_open > 0) stage(0, F{}, std::integral_constant<bool, kFirst>{});
      else stage(0, T{}, std::integral_constant<bool, kFirst>{});
    }
    int t = 1;
    for (; t < t_open; ++t) stage(t, F{}, F{});
    for (; t < n_tiles; ++t) stage(t, T{}, F{});
  };
  reset(kNegBig);
  stream(std::integral_constant<int, 0>{});
  bool ex = false;  // NaN shares also fail the test
#pragma unroll
  for (int s = 0; s < kPfSets; ++s) ex |= !(l[s] < __builtin_ldexpf(1.0f, int(kPfHeadroom)));
  if (__syncthreads_or(ex ? 1 : 0)) {
    // a score past the headroom: exact maxima, then the accumulation again
    reset(kNegBig);
    stream(std::integral_constant<int, 1>{});
    float mx[kPfSets];
#pragma unroll
    for (int s = 0; s < kPfSets; ++s) mx[s] = live_row[s] ? __builtin_fmaxf(row_max(m[s]), kNegBig) : kBig;
    reset(kNegBig);
#pragma unroll
    for (int s = 0; s < kPfSets; ++s) m[s] = mx[s];
    stream(std::integral_constant<int, 2>{});
  }

#pragma unroll
  for (int s = 0; s < kPfSets; ++s) {
    float lt = l[s];
    lt += __shfl_xor(lt, 16);
    lt += __shfl_xor(lt, 32);
    const int r = (wave * kPfSets + s) * 16 + (lane & 15);
    const int ti = r / G, g = r - ti * G;
    if (ti < ni) {
      const int64_t tok = qf + i0 + ti;
      const float inv = lt > 0.0f ? vd / lt : 0.0f;  // a row that sees no key: zeros and lse = -inf
      char* dst = a.out + tok * a.out_tok_stride + int64_t(h * G + g) * a.out_head_stride;
      constexpr int kEsz = Elt<OUT_DT>::kSize;
#pragma unroll
      for (int c = 0; c < 8; ++c) store_row4<OUT_DT>(dst + (16 * c + kc0) * kEsz, o[s][c] * inv);
      if (lane < 16 && a.lse)
        a.lse[int64_t(h * G + g) * a.lse_head_stride + tok] =
            lt > 0.0f ? (m[s] + __builtin_log2f(lt)) * 0.6931471805599453f : -__builtin_inff();
    }
  }
}

template <int Q_DT, int OUT_DT>
__global__ void __launch_bounds__(kPfThreads) __attribute__((amdgpu_waves_per_eu(2)))
prefill_attention_kernel(PrefillArgs p) {
  __shared__ StageLds lds;
  attend_block<Q_DT, OUT_DT>(p, p.blocks[p.num_seqs], lds);
}

// After prefill_runs_kernel: the merge of its records where it took the step,
// a workgroup per query block where it left it.
template <int Q_DT, int OUT_DT>
__global__ void __launch_bounds__(kPfThreads) __attribute__((amdgpu_waves_per_eu(2)))
prefill_either_kernel(PrefillArgs p, RunSpace s) {
  __shared__ StageLds lds;
  static_assert(sizeof(MergeLds) <= sizeof(StageLds), "the stages hold the merge's scratch");
  const int total = uniform(p.blocks[p.num_seqs]);
  if (total < 0)
    merge_records<OUT_DT, 8>(p.a, p.tq, s, reinterpret_cast<MergeLds&>(lds));
  else
    attend_block<Q_DT, OUT_DT>(p, total, lds);
}

template <int Q_DT, int OUT_DT>
void launch_prefill_out(const PrefillArgs& p, const RunSpace* s, dim3 grid, hipStream_t st) {
  if (s)
    hipLaunchKernelGGL((prefill_either_kernel<Q_DT, OUT_DT>), grid, dim3(kPfThreads), 0, st, p, *s);
  else
    hipLaunchKernelGGL((prefill_attention_kernel<Q_DT, OUT_DT>), grid, dim3(kPfThreads), 0, st, p);
}

template <int Q_DT>
void launch_prefill_q(const PrefillArgs& p, const RunSpace* s, int out_dtype, dim3 grid, hipStream_t st) {
  if (out_dtype == PSK_DTYPE_BF16) launch_prefill_out<Q_DT, PSK_DTYPE_BF16>(p, s, grid, st);
  else launch_prefill_out<Q_DT, PSK_DTYPE_F32>(p, s, grid, st);
}

// What the host can tell of a step whose sequences have at most `keys` keys,
// and its query tokens at least: kBlocks where no such lengths prefer the equal
// runs, kRuns where all do, else kEither.
enum Route { kBlocks, kRuns, kEither };
Route route(int64_t total_q, int64_t max_q, int64_t num_seqs, int64_t num_kv_heads, int64_t tq, bool causal,
            int64_t keys, int64_t cus) {
  const int64_t nb = ceil_div(total_q, tq), wgs = nb * num_kv_heads;
  if (num_seqs > kOrderMax || 2 * num_kv_heads > cus || wgs > 4 * cus) return kBlocks;
  keys = std::min<int64_t>(keys, INT32_MAX);
  // a CU's share of the costs: at least with the query tokens as the only keys
  // (the longest sequence's blocks, and one tq each for the others) ...
  const int64_t m = std::min(ceil_div(max_q, tq), nb);
  const int64_t least = (nb * kBlockCost + tq * (m * (m + 1) / 2 + nb - m)) * num_kv_heads / cus;
  if (!prefers_runs(keys, least, max_q, wgs, cus)) return kBlocks;
  // ... at most with all the keys there can be, for one causal sequence from
  // block to block, else in every block
  const int64_t most = (num_seqs == 1 && causal
                            ? nb * (kBlockCost + std::max<int64_t>(keys - total_q, 0) + tq) + tq * (nb * (nb - 1) / 2)
                            : (nb + num_seqs) * (kBlockCost + keys)) * num_kv_heads / cus;
  return prefers_runs(std::min(keys, max_q), most, max_q, wgs, cus) ? kRuns : kEither;
}

// Words of workspace: the launch order, and the runs' part.
int64_t order_words(int64_t num_seqs) { return 2 * num_seqs + 1; }

}  // namespace

extern "C" {

int64_t psk_paged_prefill_workspace_len(int64_t num_seqs) {
  if (num_seqs < 0) return PSK_E_ARG;
  return order_words(num_seqs) + (num_seqs <= kOrderMax ? prefill_runs_words() : 0);
}

int64_t psk_paged_prefill_step_workspace_len(int64_t num_seqs, int64_t total_q, int64_t max_seqlen_q,
                                             int64_t num_q_heads, int64_t num_kv_heads, int64_t max_seqlen_k) {
  if (num_seqs < 0 || total_q < 0 || total_q > INT32_MAX || max_seqlen_q <= 0 || num_kv_heads <= 0 || num_q_heads <= 0 ||
      num_q_heads % num_kv_heads || num_q_heads / num_kv_heads > kPfRows)
    return PSK_E_ARG;
  // (kRunMaxWgs: a device with fewer CUs takes the runs for no step that one with more does not)
  const bool blocks = route(total_q, max_seqlen_q, num_seqs, num_kv_heads, kPfRows / (num_q_heads / num_kv_heads), true,
                            max_seqlen_k, kRunMaxWgs) == kBlocks;
  return order_words(num_seqs) + (blocks ? 0 : prefill_runs_words());
}

int psk_paged_prefill_attention(const void* q, int64_t q_tok_stride, int64_t q_head_stride, int q_dtype,
                                const void* k_cache, const void* v_cache, const int64_t* k_strides,
                                const int64_t* v_strides, const int32_t* block_table, int64_t block_table_stride,
                                int64_t block_table_width, const int32_t* seq_lens, int64_t num_seqs,
                                int64_t num_q_heads, int64_t num_kv_heads, int64_t head_size, int64_t block_size,
                                int64_t num_blocks, int64_t total_q, int64_t max_seqlen_q,
                                const int32_t* cu_seqlens_q, int causal, float softmax_scale, const float* q_descale,
                                const float* k_descale, const float* v_descale, const int64_t* descale_strides,
                                void* out, int64_t out_tok_stride, int64_t out_head_stride, int out_dtype, float* lse,
                                int64_t lse_head_stride, int32_t* workspace, int64_t workspace_len, void* stream) {
  begin_device_call();
  if (num_seqs < 0 || num_kv_heads <= 0 || num_q_heads <= 0 || num_q_heads % num_kv_heads)
    return fail(PSK_E_ARG, "bad head counts (q %lld, kv %lld)", (long long)num_q_heads, (long long)num_kv_heads);
  const int64_t group = num_q_heads / num_kv_heads;
  if (group > kPfRows)
    return fail(PSK_E_ARG, "at most %d query heads per kv head (got %lld)", kPfRows, (long long)group);
  if (max_seqlen_q <= 0 || max_seqlen_q > INT32_MAX) return fail(PSK_E_ARG, "max_seqlen_q %lld", (long long)max_seqlen_q);
  if (total_q < 0 || total_q > INT32_MAX) return fail(PSK_E_ARG, "total_q %lld", (long long)total_q);
  if (!cu_seqlens_q && total_q != num_seqs * max_seqlen_q)
    return fail(PSK_E_ARG, "without cu_seqlens_q every sequence has max_seqlen_q rows (%lld != %lld x %lld)",
                (long long)total_q, (long long)num_seqs, (long long)max_seqlen_q);
  if (head_size != kHead) return fail(PSK_E_ARG, "head_size must be %d (got %lld)", kHead, (long long)head_size);
  if (block_size <= 0 || block_size > INT32_MAX || num_blocks <= 0 || num_blocks > INT32_MAX ||
      block_table_width <= 0)
    return fail(PSK_E_ARG, "bad cache geometry");
  if (q_dtype != PSK_DTYPE_FP8_E4M3FN && q_dtype != PSK_DTYPE_BF16 && q_dtype != PSK_DTYPE_F16 &&
      q_dtype != PSK_DTYPE_F32)
    return fail(PSK_E_DTYPE, "query dtype %d", q_dtype);
  if (out_dtype != PSK_DTYPE_BF16 && out_dtype != PSK_DTYPE_F32)
    return fail(PSK_E_DTYPE, "output dtype %d (bf16 or f32)", out_dtype);
  if (num_seqs == 0 || total_q == 0) return PSK_OK;
  if (!q || !k_cache || !v_cache || !k_strides || !v_strides || !block_table || !seq_lens || !out || !workspace)
    return fail(PSK_E_ARG, "NULL pointer");
  if (!std::isfinite(softmax_scale)) return fail(PSK_E_ARG, "softmax_scale is not finite");
  if (workspace_len < order_words(num_seqs))
    return fail(PSK_E_WORKSPACE, "workspace of %lld words, need %lld", (long long)workspace_len,
                (long long)order_words(num_seqs));
  const int qsz = dtype_size(q_dtype), osz = dtype_size(out_dtype);
  const uint64_t kv_align[8] = {uint64_t(uintptr_t(k_cache)), uint64_t(uintptr_t(v_cache)), uint64_t(k_strides[0]),
                                uint64_t(k_strides[1]),       uint64_t(k_strides[2]),       uint64_t(v_strides[0]),
                                uint64_t(v_strides[1]),       uint64_t(v_strides[2])};
  if (common_align(kv_align, 8, 16) < 16) return fail(PSK_E_ARG, "K/V caches need 16-byte aligned bases and strides");
  const uint64_t q_align[3] = {uint64_t(uintptr_t(q)), uint64_t(q_tok_stride * qsz), uint64_t(q_head_stride * qsz)};
  if (common_align(q_align, 3, 16) < 16) return fail(PSK_E_ARG, "query rows need 16-byte alignment");
  const uint64_t o_align[3] = {uint64_t(uintptr_t(out)), uint64_t(out_tok_stride * osz),
                               uint64_t(out_head_stride * osz)};
  if (common_align(o_align, 3, 4 * osz) < 4 * osz)
    return fail(PSK_E_ARG, "output rows need %d-byte alignment", 4 * osz);

  PrefillArgs p{};
  DecodeArgs& a = p.a;
  a.q = static_cast<const char*>(q);
  a.q_tok_stride = q_tok_stride * qsz;
  a.q_head_stride = q_head_stride * qsz;
  a.k = static_cast<const uint8_t*>(k_cache);
  a.v = static_cast<const uint8_t*>(v_cache);
  a.k_blk = k_strides[0];
  a.k_row = k_strides[1];
  a.k_head = k_strides[2];
  a.v_blk = v_strides[0];
  a.v_row = v_strides[1];
  a.v_head = v_strides[2];
  a.block_table = block_table;
  a.bt_stride = block_table_stride;
  a.bt_width = block_table_width;
  a.seq_lens = seq_lens;
  a.num_blocks = int32_t(num_blocks);
  a.block_size = int32_t(block_size);
  a.bs_shift = log2_exact(block_size);
  a.num_kv_heads = int32_t(num_kv_heads);
  a.group = int32_t(group);
  a.heads = int32_t(group);
  a.q_len = int32_t(max_seqlen_q);
  a.cu_q = cu_seqlens_q;
  a.causal = causal ? 1 : 0;
  a.scale_log2 = softmax_scale * 1.4426950408889634f;
  const int64_t zero[6] = {0, 0, 0, 0, 0, 0};
  const int64_t* ds = descale_strides ? descale_strides : zero;
  a.qd = q_descale;
  a.qd_b = ds[0];
  a.qd_h = ds[1];
  a.kd = k_descale;
  a.kd_b = ds[2];
  a.kd_h = ds[3];
  a.vd = v_descale;
  a.vd_b = ds[4];
  a.vd_h = ds[5];
  a.out = static_cast<char*>(out);
  a.out_tok_stride = out_tok_stride * osz;
  a.out_head_stride = out_head_stride * osz;
  a.lse = lse;
  a.lse_head_stride = lse_head_stride;
  p.blocks = workspace;
  p.order = workspace + num_seqs + 1;
  p.num_seqs = int32_t(num_seqs);
  p.tq = int32_t(kPfRows / group);
  constexpr int64_t k32 = int64_t(1) << 32;
  p.narrow = k_strides[0] >= 0 && k_strides[0] < k32 && k_strides[1] >= 0 && k_strides[1] < k32 &&
             v_strides[0] >= 0 && v_strides[0] < k32 && v_strides[1] >= 0 && v_strides[1] < k32;
  // query blocks: at most ceil(total_q / tq) whole ones plus one partial per sequence
  const int64_t max_blocks = ceil_div(total_q, p.tq) + num_seqs;
  if (num_seqs > (INT32_MAX - 1) / 2 || max_blocks * num_kv_heads > INT32_MAX)
    return fail(PSK_E_ARG, "too many query blocks (%lld x %lld kv heads)", (long long)max_blocks,
                (long long)num_kv_heads);

  hipStream_t st = static_cast<hipStream_t>(stream);
  const int64_t cus = prefill_cus();
  const Route r = workspace_len < order_words(num_seqs) + prefill_runs_words()
                      ? kBlocks
                      : route(total_q, max_seqlen_q, num_seqs, num_kv_heads, p.tq, a.causal != 0,
                              block_table_width * block_size, cus);
  RunSpace space;
  int st1;
  if (r != kBlocks) {
    st1 = launch_prefill_runs(a, num_seqs, ceil_div(total_q, p.tq) * num_kv_heads, r == kRuns, q_dtype, out_dtype,
                              workspace + order_words(num_seqs), workspace, workspace + num_seqs + 1, &space, st);
  } else {
    hipLaunchKernelGGL(prefill_blocks_kernel, dim3(1), dim3(1024), 0, st, a, int(num_seqs), int(p.tq), workspace,
                       workspace + num_seqs + 1);
    st1 = check_launch("prefill_blocks_kernel launch");
  }
  if (r == kRuns || st1 != PSK_OK) return st1;
  // (kEither: a workgroup per CU for the merge, where the blocks are fewer)
  const dim3 grid{unsigned(std::max(max_blocks * num_kv_heads, r == kEither ? cus : 1)), 1u, 1u};
  const RunSpace* s = r == kEither ? &space : nullptr;
  switch (q_dtype) {
    case PSK_DTYPE_FP8_E4M3FN: launch_prefill_q<PSK_DTYPE_FP8_E4M3FN>(p, s, out_dtype, grid, st); break;
    case PSK_DTYPE_BF16: launch_prefill_q<PSK_DTYPE_BF16>(p, s, out_dtype, grid, st); break;
    case PSK_DTYPE_F16: launch_prefill_q<PSK_DTYPE_F16>(p, s, out_dtype, grid, st); break;
    default: launch_prefill_q<PSK_DTYPE_F32>(p, s, out_dtype, grid, st); break;
  }
  return check_launch("prefill_attention_kernel launch");
}

}  // extern "C"
