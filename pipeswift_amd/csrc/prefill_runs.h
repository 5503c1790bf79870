// What the two prefill kernels share (prefill_attention.hip: a workgroup per
// query block; prefill_runs.hip: the step cut into equal runs): which of them a
// step takes, the launch order of the query blocks, and the merge of the
// partial records that runs leave of the blocks they share.
//
// The host knows only how long a sequence can be (the block table's width) and
// that each has its query tokens at least.  Where that does not
// settle the choice it is the device's, in two launches: prefill_runs_kernel
// reads the lengths and either runs the step or leaves the blocks' launch
// order, and prefill_either_kernel then merges the records or runs the blocks.

#ifndef PSK_PREFILL_RUNS_H
#define PSK_PREFILL_RUNS_H

#include <type_traits>

#include "paged_attention.h"

namespace psk_detail {

constexpr int kBlockRows = 256;        // rows of a query block: kBlockRows / heads query tokens of one kv head
constexpr int kRunWaves = 8;           // waves of a workgroup, in both kernels
constexpr int kRunThreads = kRunWaves * 64;
constexpr int kOrderMax = 1024;        // sequences that are ordered by length (more: batch order)
constexpr int kRunMaxWgs = 256;        // workgroups that share a step cut into runs, at most

// A query block costs kBlockCost (its queries, its first loads, its result)
// plus the keys it reads.
constexpr int64_t kBlockCost = 384;

// Whether a step runs faster cut into equal runs than with a workgroup per
// query block, from the longest sequence that has query tokens (`keys`), a
// CU's share of the blocks' costs, the most query tokens of a sequence, the
// workgroups that its blocks are (ceil(total_q / tq) per kv head) and the
// device's CUs.  A workgroup per block takes about as long as its longest
// block, runs as long as the share; their records, merge and second start of a
// block cost another 10-25 us, more where more blocks are shared.  So runs win
// where the longest block stands out: any long prefix, and fresh prompts that
// leave the chip idle.  Where the blocks fill the chip several times over, or
// get shorter from a fresh prompt's last block to its first and so fill each
// other's gaps, a workgroup per block is the faster.  Of 807 measured steps (1
// to 30 sequences, 48 to 8192 new tokens over up to 45000 cached, 1 to 8 kv
// heads) the choice takes 1.3 % more time than always taking the faster side
// (workgroups per block alone 32 %, runs alone 11 %), and for none over 1 % more
// than a workgroup per block.  Some of them, us, runs / workgroup per block,
// fresh prompts by query heads / kv heads:
//   tokens    500        1000       1400       2000       3000        4000        8000
//   32 / 8  29.2/25.0  40.1/38.4  47.1/49.9  66.7/66.2  101.7/94.5  153/137    487/479
//   32 / 4  28.8/25.1  38.1/39.2  48.0/50.3  69.8/66.8  102.9/93.7  155/135    493/479
//   16 / 2  28.3/24.9  34.6/38.7  40.2/48.7  49.0/65.6   64.7/92.1  95.4/119   262/246
//   8 / 2   28.4/24.4  31.3/37.5  33.5/48.5  38.9/65.0   47.3/90.8  60.1/117   145/226
//   8 / 1   28.3/24.5  33.4/38.1  37.1/48.2  40.0/64.5   48.0/90.4  59.0/118   147/225
// over a prefix (32 / 8): 64 tokens over 1000 32/42, 128 over 4096 41/126, 256
// over 1000 35/47, 512 over 32768 260/920; six prompts of 500 beside a decode
// of 20000 64/554; 32 / 4: seven of 600 over 20000 each 1190/2030.
constexpr int64_t kRunsLeast = 980;  // no step of shorter sequences does
__host__ __device__ inline bool prefers_runs(int64_t keys, int64_t share, int64_t max_q, int64_t wgs, int64_t cus) {
  const bool prefix = keys >= 4 * max_q;  // blocks of about one length
  if (wgs > cus) return prefix && keys >= 1024 && wgs <= 4 * cus;
  if (keys < 1536) return keys >= kRunsLeast && share <= (keys < 1280 ? 450 : 800);
  return prefix || keys >= 4096 || 4 * keys >= 5 * share + 1100;
}

// A value that is the same in every lane, in scalar registers.
__device__ __forceinline__ int uniform(int v) { return __builtin_amdgcn_readfirstlane(v); }
__device__ __forceinline__ int64_t uniform(int64_t v) {
  const uint64_t lo = uint32_t(uniform(int(v))), hi = uint32_t(uniform(int(v >> 32)));
  return int64_t(hi << 32 | lo);
}

// LDS of order_blocks: each sequence's query tokens and its length, -1 if it
// has none of them (put_sequence, for at most kOrderMax sequences), and scratch.
struct OrderLds {
  int32_t n[kOrderMax], key[kOrderMax], order[kOrderMax], wave[16];
};
__device__ __forceinline__ void put_sequence(OrderLds& lds, int b, int n, int len) {
  lds.n[b] = n;
  lds.key[b] = n > 0 ? len : -1;
}

// The launch order of the query blocks, by one workgroup of NT threads:
// sequences by decreasing length (the keys their last block reads; without
// query tokens last), ties in batch order, then each sequence's blocks from
// its last (the most keys, when causal) to its first.  Writes order[k] and
// the exclusive prefix blocks[k] of ceil(n_b / tq) over launch positions,
// blocks[num_seqs] = the total.  Past kOrderMax sequences the batch order is
// kept (and lds.n and lds.key not read).
template <int NT>
__device__ __forceinline__ void order_blocks(const DecodeArgs& a, int num_seqs, int tq, int32_t* blocks, int32_t* order,
                                             OrderLds& lds) {
  const int tid = int(threadIdx.x), lane = tid & 63, wave = tid >> 6;
  const bool sorted = num_seqs <= kOrderMax;
  if (sorted) {
    for (int b = tid; b < num_seqs; b += NT) {
      const int key = lds.key[b];
      int rank = 0;
      for (int j = 0; j < num_seqs; ++j) {
        const int kj = lds.key[j];
        rank += (kj > key || (kj == key && j < b)) ? 1 : 0;
      }
      lds.order[rank] = b;
    }
    __syncthreads();
  }
  int carry = 0;
  for (int c0 = 0; c0 < num_seqs; c0 += NT) {
    const int k = c0 + tid;
    const int b = k < num_seqs ? (sorted ? lds.order[k] : k) : 0;
    const int nb = k < num_seqs ? ((sorted ? lds.n[b] : q_count(a, b)) + tq - 1) / tq : 0;
    int x = nb;  // inclusive prefix over the wave
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const int y = __shfl_up(x, o);
      if (lane >= o) x += y;
    }
    if (lane == 63) lds.wave[wave] = x;
    __syncthreads();
    int before = 0, total = 0;
    for (int w = 0; w < NT / 64; ++w) {
      const int t = lds.wave[w];
      before += w < wave ? t : 0;
      total += t;
    }
    if (k < num_seqs) {
      blocks[k] = carry + before + x - nb;
      order[k] = b;
    }
    carry += total;
    __syncthreads();
  }
  if (tid == 0) blocks[num_seqs] = carry;
}

// A partial record: per wave 16 x 64 lanes x 4 floats of O^T as the lanes hold
// it, then 32 maxima and 32 sums.
constexpr int64_t kRunSlab = 16 * 64 * 4 + 64;
constexpr int64_t kRunRecord = kRunSlab * kRunWaves;

// What run j left as a partial record in its slot: its block (b, i), if any,
// and the sequence's query tokens.
struct RunDesc {
  int32_t valid, b, i, n;
};

// The runs' part of the workspace.
struct RunSpace {
  RunDesc* desc;     // of each run: [0] its first piece, [1] its last
  float* records;    // 2 per run and kv head
  int32_t max_runs;  // runs per kv head at most
};

template <int OUT_DT>
__device__ __forceinline__ void store_cols4(char* dst, f32x4 v);
template <>
__device__ __forceinline__ void store_cols4<PSK_DTYPE_F32>(char* dst, f32x4 v) {
  *reinterpret_cast<f32x4*>(dst) = v;
}
template <>
__device__ __forceinline__ void store_cols4<PSK_DTYPE_BF16>(char* dst, f32x4 v) {
  *reinterpret_cast<bf16x4*>(dst) = __builtin_convertvector(v, bf16x4);  // RNE
}

// Row lane % 32 of a wave's 32 of a block of ni query tokens from row `first`
// of q: columns 32 d + 8 q + 4 (lane / 32) .. + 3 of O^T in o[4 (d - d0) + q]
// for d0 <= d < d0 + ND, the sum lt and the maximum m, times vd to the output
// and (with d0 = 0) to the lse.
template <int OUT_DT, int ND>
__device__ __forceinline__ void write_row(const DecodeArgs& a, int64_t first, int ni, int h, float vd, int wave, int lane,
                                          int d0, const f32x4 (&o)[4 * ND], float m, float lt) {
  const int G = a.heads;
  const int r = wave * 32 + (lane & 31);
  const int ti = r / G, g = r - ti * G;
  if (ti >= ni) return;
  const int64_t tok = first + ti;
  const float inv = lt > 0.0f ? vd / lt : 0.0f;  // no key seen: zeros, lse = -inf
  char* dst = a.out + tok * a.out_tok_stride + int64_t(h * G + g) * a.out_head_stride;
  constexpr int kEsz = Elt<OUT_DT>::kSize;
#pragma unroll
  for (int c = 0; c < 4 * ND; ++c)
    store_cols4<OUT_DT>(dst + (32 * (d0 + (c >> 2)) + 8 * (c & 3) + 4 * (lane >> 5)) * kEsz, o[c] * inv);
  if (lane < 32 && d0 == 0 && a.lse)
    a.lse[int64_t(h * G + g) * a.lse_head_stride + tok] =
        lt > 0.0f ? (m + __builtin_log2f(lt)) * 0.6931471805599453f : -__builtin_inff();
}

// LDS of merge_records.
struct MergeLds {
  RunDesc first[kRunMaxWgs], last[kRunMaxWgs];
  int32_t begin[kRunMaxWgs];  // the runs that begin a block they do not end
  int32_t wave[kRunWaves];
};

// Merges the partial records of the blocks that several runs share, by all
// workgroups of the launch (kRunThreads threads).  Run j's record in slot 1 is
// the first of such a block, whose others are the first pieces of the runs that
// follow.  A task is one wave's: 32 columns of the 32 rows of a wave of one
// block and kv head, so that the wave's 4 KiB of a record are in flight at
// once; the tasks of the blocks there are go round the launch's workgroups,
// then their waves, so that a few use every CU's share of the bandwidth.
// R records' columns are in flight at a time.  Bound by the latency of the loads, so the
// rounds of them count: 7 appends of 11-65 tokens over 4-11k cached, 8 query heads on
// 2 kv heads, the whole call with this merge in the launch the device chooses for:
// 54.7 us with the tasks on the first workgroups, 50.6-52.2 spread over all of them
// (R = 4 and 8), 42.1 (R = 4) and 39.3 (R = 8) with the maxima 16 a round as well.
template <int OUT_DT, int R>
__device__ __forceinline__ void merge_records(const DecodeArgs& a, int tq, const RunSpace& s, MergeLds& lds) {
  const int tid = int(threadIdx.x), lane = tid & 63, wave = uniform(tid >> 6);
  const int Hkv = a.num_kv_heads;
  static_assert(kRunMaxWgs <= kRunThreads, "a run per thread");
  const bool own = tid < s.max_runs;
  RunDesc last{0, 0, 0, 0};
  if (own) {
    lds.first[tid] = s.desc[2 * tid];
    last = s.desc[2 * tid + 1];
    lds.last[tid] = last;
  }
  const uint64_t begins = __ballot(own && last.valid);
  if (lane == 0) lds.wave[wave] = __popcll(begins);
  __syncthreads();
  int before = 0, total = 0;
#pragma unroll
  for (int w = 0; w < kRunWaves; ++w) {
    const int t = lds.wave[w];
    before += w < wave ? t : 0;
    total += t;
  }
  if (own && last.valid) lds.begin[before + __popcll(begins & ((uint64_t(1) << lane) - 1))] = tid;
  __syncthreads();
  total = uniform(total);
  const int tasks = total * Hkv * kRunWaves * 4;
  for (int t = wave * int(gridDim.x) + int(blockIdx.x); t < tasks; t += int(gridDim.x) * kRunWaves) {
    const int d0 = t & 3, row_wave = (t >> 2) & (kRunWaves - 1);
    const int rest = t / (4 * kRunWaves);
    const int at = rest / Hkv, h = rest - at * Hkv;
    const int j = uniform(lds.begin[at]);
    const int b = uniform(lds.last[j].b), i = uniform(lds.last[j].i);
    const int ni = min(tq, uniform(lds.last[j].n) - i * tq);
    if (row_wave * 32 >= ni * a.heads) continue;  // no query rows
    const int64_t first = q_first(a, b) + i * tq;
    const float vd = descale(a.vd, a.vd_b, a.vd_h, b, h);
    // how many of the following runs' first pieces are of the same block
    int n = 0;
    for (int k = j + 1;; k += 64) {
      const int jl = min(k + lane, s.max_runs - 1);
      const RunDesc other = lds.first[jl];
      const uint64_t same = __ballot(k + lane < s.max_runs && other.valid && other.b == b && other.i == i);
      n += same == ~0ull ? 64 : __builtin_ctzll(~same);
      if (same != ~0ull) break;
    }
    // record r of the block: run j's slot 1, then slot 0 of run j + r
    auto record = [&](int r) {
      return s.records + ((int64_t(j + r) * Hkv + h) * 2 + (r == 0 ? 1 : 0)) * kRunRecord + row_wave * kRunSlab;
    };
    // a batch of records at a time, their maxima, sums and columns in flight
    // together (past the last a record is read again and not used): two where
    // two runs share the block, else R
    auto max_of = [&](int r) { return record(r)[4096 + (lane & 31)]; };
    float m = max_of(0), l = 0.0f;
    f32x4 o[4];
#pragma unroll
    for (int c = 0; c < 4; ++c) o[c] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    auto add = [&](auto batch_tag, int r0) {
      constexpr int N = decltype(batch_tag)::value;
      float rm[N], rl[N];
      f32x4 x[N][4];
#pragma unroll
      for (int k = 0; k < N; ++k) {
        const float* rec = record(min(r0 + k, n));
        rm[k] = rec[4096 + (lane & 31)];
        rl[k] = rec[4096 + 32 + (lane & 31)];
#pragma unroll
        for (int c = 0; c < 4; ++c) x[k][c] = *reinterpret_cast<const f32x4*>(rec + ((4 * d0 + c) * 64 + lane) * 4);
      }
      if (r0 == 0) {
#pragma unroll
        for (int k = 1; k < N; ++k) m = __builtin_fmaxf(m, rm[k]);
      }
#pragma unroll
      for (int k = 0; k < N; ++k) {
        if (r0 + k > n) break;
        const float w = __builtin_amdgcn_exp2f(rm[k] - m);
        l += rl[k] * w;
#pragma unroll
        for (int c = 0; c < 4; ++c) o[c] += x[k][c] * w;
      }
    };
    if (n == 1) {
      add(std::integral_constant<int, 2>{}, 0);
    } else {
#pragma unroll 16
      for (int r = R; r <= n; ++r) m = __builtin_fmaxf(m, max_of(r));
      for (int r0 = 0; r0 <= n; r0 += R) add(std::integral_constant<int, R>{}, r0);
    }
    write_row<OUT_DT, 1>(a, first, ni, h, vd, row_wave, lane, d0, o, m, l);
  }
}

// prefill_runs.hip.  `a` as the decode reader's, with a.q_len the most query
// tokens of a sequence, a.heads at most kBlockRows; for at most kOrderMax
// sequences and prefill_cus() / 2 kv heads.
int64_t prefill_cus();         // CUs of the device, at most kRunMaxWgs (0 if unknown)
int64_t prefill_runs_words();  // int32 words of a RunSpace, no initial contents needed
// A step cut into equal runs, with its merge: `sure`.  Else the first launch of
// a step that may take either kernel (`wgs`: its blocks' workgroups, for
// prefers_runs): where it does not run the step itself `blocks` and `order`
// receive the launch order, else blocks[num_seqs] = -1.  Fills `space` from
// `workspace`.
int launch_prefill_runs(const DecodeArgs& a, int64_t num_seqs, int64_t wgs, bool sure, int q_dtype, int out_dtype,
                        int32_t* workspace, int32_t* blocks, int32_t* order, RunSpace* space, hipStream_t st);

}  // namespace psk_detail

#endif  // PSK_PREFILL_RUNS_H
