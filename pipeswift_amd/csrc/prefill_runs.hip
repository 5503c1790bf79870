// Prefill attention over the FP8 E4M3FN KV cache for MI355X (gfx950), the work
// of a step cut into equal runs: for steps with few query blocks, or with long
// cached prefixes, where a workgroup per block (prefill_attention.hip) leaves
// CUs idle.
//
// Nothing here allocates or synchronizes.

#include <algorithm>
#include <map>
#include <mutex>
#include <type_traits>

#include "prefill_runs.h"

using namespace psk_detail;

namespace {

// A query block is kPfRows = 256 rows of one kv head, 32 per wave; row r is
// query token i0 + r / G, query head g = r % G of the block's tq = kPfRows / G
// tokens, so every K/V row of the block's keys is read from the cache once per
// tq query tokens.  The keys stream through three LDS
// stages of kPfKeys keys (converted once, exactly, K to bf16 and V to fp16,
// as 256-byte rows):
//   * K: 16-byte chunk c of key t at chunk c ^ (t & 15), so the lanes of one
//     ds_read_b128 phase (consecutive keys, one chunk) hit distinct banks;
//   * V: chunk c of key t at c ^ (4 (t & 3) | (t & 1)), read transposed by
//     ds_read_b64_tr_b16 (four keys of one column per lane and read): the four
//     64-byte pieces a half wave reads cover all banks once, and the staging
//     stores of neighbouring keys fall in different banks.
// Per 32 keys and 32 rows: S^T = K Q^T is eight v_mfma_f32_32x32x16_bf16
// (exactly converted FP8 operands as in the decode reader), the softmax runs
// in the exp2 domain, then O^T = V^T P^T is eight v_mfma_f32_32x32x16_f16 with
// P rounded to fp16 once (11 significant bits, where the decode reader keeps
// ~16 in a bf16 hi + lo pair and runs P V twice; FA3's FP8 path keeps 4).
// Transposed products leave each lane one query row (lane % 32): its scores of
// keys 8 (i / 4) + 4 (lane / 32) + i % 4, its maximum and sum.  MFMA step u of
// P V takes as its k = 8 s + j (s = lane / 32) key 16 u + 8 (j / 4) + 4 s +
// j % 4, so the lane's scores are its P^T operand as they stand, and two
// transposed V reads give the matching V^T operand.
// The 32x32 shape: one MFMA holds the matrix pipe for 32 cycles, twice as long
// as the 16x16 one for the same operand issue, and the softmax's VALU
// instructions go out under it.  A probe of two waves per SIMD, each running
// MFMAs with 4 FMA and 2 exp2 per 32 matrix cycles, took 346 cycles per 256
// matrix cycles with it against 420 with 16x16.  The wave's own stream is
// pipelined by two tiles: while the softmax of a tile runs, the scores of the
// next one and P V of the one before are on the matrix cores (tile_step).
// What bounds it: power.  On a quarter of the chip a stage takes 1.5 us (start
// to end, 8 waves; 1.7 us for the 16x16 kernel of prefill_attention.hip), on the
// whole chip 1.9-2.0, where the clock falls to 1.8 GHz with the matrix cores 56 %
// busy (2.2 GHz and 43 % there).  4096 new tokens over six prefixes of 14k-45k, 32
// query heads over 4 kv heads, on five boxes: 1380-1465 us (1150-1080 TFLOP/s),
// against 1740-1880 with a workgroup per block; 512 new tokens over 32768, 8 kv
// heads: 257-272 against 890-924.
constexpr int kPfWaves = kRunWaves;
constexpr int kPfRows = kPfWaves * 32;
static_assert(kPfRows == kBlockRows, "the blocks of both prefill kernels are the same");
constexpr int kPfKeys = 64;  // keys per LDS stage
constexpr int kPfThreads = kPfWaves * 64;
constexpr int kPfBufs = 3;                            // converted stages in LDS
constexpr int kPfRaws = 3;                            // FP8 stages in LDS, before their conversion
constexpr uint32_t kPfRaw = 2 * kPfKeys * 128;        // bytes of one: K rows, then V rows
constexpr uint32_t kPfHalf = kPfKeys * 256;           // bytes of a stage's K (its V follows)
constexpr uint32_t kPfStage = 2 * kPfHalf;
static_assert(kPfKeys * 8 == kPfThreads, "every thread stages one 16-byte chunk of K and of V");

// The work of a step is cut into equal runs: every query block costs kPfCost
// (its queries, its first loads, its result) plus its keys, per kv head
// the blocks of all sequences follow each other, and run j of M takes cost
// [T j / M, T (j + 1) / M), whatever blocks it belongs to.  M x kv heads
// workgroups, one per CU, so the chip is full and ends together however few
// blocks a step has; a block shared by several runs leaves one partial record
// per run (fp32 sums), for merge_records.  The cost and the
// least run as measured: 128, 256, 384 and 512 keys a block gave 182, 166, 161
// and 161 us on a fresh prompt of 4000 tokens, and runs of at least 1024 or
// 2048 took 52 and 75 us where 512 take 44 (128 tokens over 4096 keys).
constexpr int64_t kPfCost = kBlockCost;
constexpr int kPfSnap = 3;          // a run boundary this close (in stages) to a block's end moves there
constexpr int64_t kPfMinRun = 512;  // least cost of a run
struct RunArgs {
  DecodeArgs a;
  RunSpace s;
  int32_t num_seqs;
  int32_t tq;        // query tokens per block
  int32_t wgs, cus;  // for prefers_runs
  int32_t sure;      // the step is cut into runs whatever its lengths
  int32_t* blocks;   // the launch order of the blocks, where they are not run here
  int32_t* order;
};

// A sequence's blocks: nb of them, block i costs base + i * step.
struct PfSeq {
  int n, len, nb;
  int64_t base, step;
  // cost of the first i blocks
  __device__ __forceinline__ int64_t upto(int64_t i) const { return i * base + step * (i * (i - 1) / 2); }
};

__device__ __forceinline__ PfSeq pf_seq(const DecodeArgs& a, int tq, int n, int len) {
  PfSeq s;
  s.n = n;
  s.len = len;
  s.nb = (s.n + tq - 1) / tq;
  // causal: block i reads about len - n + (i + 1) tq keys; else all of them
  s.base = kPfCost + (a.causal ? int64_t(max(s.len - s.n, 0)) + tq : int64_t(s.len));
  s.step = a.causal ? tq : 0;
  return s;
}

// One query block of a step and the cost range it covers.
struct PfBlock {
  int b, i, n, len, nb;
  int64_t at, cost, step;
  // keys any row of the block sees
  __device__ __forceinline__ int key_end(const DecodeArgs& a, int tq) const {
    if (!a.causal) return len;
    return min(max(len - n + min((i + 1) * tq, n), 0), len);
  }
  __device__ __forceinline__ int stages(const DecodeArgs& a, int tq) const {
    return (key_end(a, tq) + kPfKeys - 1) / kPfKeys;
  }
  // first stage at or past cost x of the step; a boundary next to the block's start or end moves there
  __device__ __forceinline__ int stage_at(int64_t x, int ns) const {
    if (x <= at) return 0;
    if (x >= at + cost) return ns;
    const int64_t s = (x - at - kPfCost) / kPfKeys;
    return s < kPfSnap ? 0 : s > ns - kPfSnap ? ns : int(s);
  }
};

// The block that cost x (0 <= x < prefix[num_seqs]) falls in.
__device__ __forceinline__ PfBlock pf_block(const RunArgs& p, const int64_t* prefix, int64_t x) {
  int lo = 0, hi = p.num_seqs - 1;  // the last sequence with prefix <= x (those without blocks share the next one's)
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (prefix[mid] <= x) lo = mid; else hi = mid - 1;
  }
  lo = uniform(lo);
  const PfSeq s = pf_seq(p.a, p.tq, q_count(p.a, lo), max(p.a.seq_lens[lo], 0));
  const int64_t before = lo > 0 ? int64_t(prefix[lo]) : 0;  // prefix[0] is not stored
  const int64_t y = x - before;
  int i = 0, last = s.nb - 1;  // the last block with upto(i) <= y
  while (i < last) {
    const int mid = (i + last + 1) >> 1;
    if (s.upto(mid) <= y) i = mid; else last = mid - 1;
  }
  i = uniform(i);
  return PfBlock{lo, i, uniform(s.n), uniform(s.len), uniform(s.nb), uniform(before + s.upto(i)),
                 uniform(s.base + i * s.step), uniform(s.step)};
}

// Runs per kv head for total cost T.
__device__ __forceinline__ int pf_runs(const RunArgs& p, int64_t T) {
  return int(max(int64_t(1), min(int64_t(p.s.max_runs), T / kPfMinRun)));
}

// First cost of run j of M for total cost T: 0 for j = 0, T for j = M, and
// monotone between, from a 32-bit division (M < 2^15, T < 2^47).
__device__ __forceinline__ int64_t pf_run_start(int64_t T, int j, int M) {
  return (T * int64_t((uint32_t(j) << 16) / uint32_t(M))) >> 16;
}

// What every workgroup finds out about the step's sequences first.
struct PfStep {
  bool take;  // the step is cut into runs
  int64_t T;  // its cost
};

// Inclusive prefix and maximum over the wave's first `lanes` lanes (the maximum
// in every lane): as many steps as they need.
__device__ __forceinline__ int64_t wave_prefix(int64_t x, int lane, int lanes) {
  for (int o = 1; o < lanes; o <<= 1) {
    const int64_t y = __shfl_up(x, o);
    if (lane >= o) x += y;
  }
  return x;
}
__device__ __forceinline__ int wave_longest(int keys, int lanes) {
  for (int o = 1; o < lanes; o <<= 1) keys = max(keys, __shfl_xor(keys, o));
  return uniform(keys);
}

__device__ __forceinline__ bool pf_take(const RunArgs& p, int keys, int64_t T) {
  return p.sure || prefers_runs(keys, T * p.a.num_kv_heads / p.cus, p.a.q_len, p.wgs, p.cus);
}

// Whether the step is cut into runs, by the threads of a workgroup (the same
// answer in every one; the launch that follows reads it): if so the cost prefix
// of the sequences (prefix[b + 1]: up to b), else their query tokens and
// lengths in `seqs`.  Up to 64 sequences every wave does it for itself, a
// sequence a lane, without a barrier.
template <int NT>
__device__ __forceinline__ PfStep pf_step(const RunArgs& p, int64_t* prefix, int64_t* s_wave, OrderLds& seqs) {
  const int tid = int(threadIdx.x), lane = tid & 63, wave = tid >> 6;
  const DecodeArgs& a = p.a;
  if (p.num_seqs <= 64) {
    const bool in = lane < p.num_seqs;
    const int n = in ? q_count(a, lane) : 0, len = in ? max(a.seq_lens[lane], 0) : 0;
    const int keys = wave_longest(n > 0 ? len : 0, p.num_seqs);
    PfStep found{false, 0};
    if (p.sure || keys >= kRunsLeast) {  // else the costs do not matter
      const PfSeq s = pf_seq(a, p.tq, n, len);
      const int64_t x = wave_prefix(in ? s.upto(s.nb) : 0, lane, p.num_seqs);
      if (in) prefix[lane + 1] = x;  // the same from every wave
      const int last = p.num_seqs - 1;
      found.T = int64_t(uint64_t(uint32_t(__builtin_amdgcn_readlane(int(x >> 32), last))) << 32 |
                        uint32_t(__builtin_amdgcn_readlane(int(x), last)));
      found.take = pf_take(p, keys, found.T);
    }
    if (!found.take && in) put_sequence(seqs, lane, n, len);
    return found;
  }
  int keys = 0;
  int64_t carry = 0;
  for (int c0 = 0; c0 < p.num_seqs; c0 += NT) {
    const int b = c0 + tid;
    int64_t own = 0;
    if (b < p.num_seqs) {
      const int n = q_count(a, b), len = max(a.seq_lens[b], 0);
      put_sequence(seqs, b, n, len);
      const PfSeq s = pf_seq(a, p.tq, n, len);
      own = s.upto(s.nb);
      if (n > 0) keys = max(keys, len);
    }
    const int64_t x = wave_prefix(own, lane, 64);
    if (lane == 63) s_wave[wave] = x;
    __syncthreads();
    int64_t before = 0, total = 0;
    for (int w = 0; w < NT / 64; ++w) {
      const int64_t t = s_wave[w];
      before += w < wave ? t : 0;
      total += t;
    }
    if (b < p.num_seqs) prefix[b + 1] = carry + before + x;
    carry += total;
    __syncthreads();
  }
  keys = wave_longest(keys, 64);
  if (lane == 0) s_wave[wave] = keys;
  __syncthreads();
#pragma unroll
  for (int w = 0; w < NT / 64; ++w) keys = max(keys, int(s_wave[w]));
  return PfStep{pf_take(p, uniform(keys), uniform(carry)), uniform(carry)};
}

// LDS at a byte address
template <class T>
__device__ __forceinline__ __attribute__((address_space(3))) T* lds_at(uint32_t at) {
  return (__attribute__((address_space(3))) T*)size_t(at);
}

// Workgroup barrier that orders LDS only: the global loads of a coming stage
// stay in flight across it.
__device__ __forceinline__ void lds_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// 16 bytes per lane from global memory straight to LDS: lane i's to at + 16 i.
// In asm because the compiler, unable to tell which LDS bytes such a load
// writes, would wait for all of them before every LDS read.  It writes no
// register and leaves m0 as it was; wait_loads() orders the reads of the bytes.
__device__ __forceinline__ void load_lds(uint32_t at, const uint8_t* base, uint32_t offset) {
  uint32_t m0;
  asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %2, %3\n\ts_mov_b32 m0, %0"
               : "=&s"(m0) : "s"(at), "v"(offset), "s"(base) : "memory");
}
__device__ __forceinline__ void load_lds(uint32_t at, const uint8_t* p) {
  uint32_t m0;
  asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %2, off\n\ts_mov_b32 m0, %0"
               : "=&s"(m0) : "s"(at), "v"(p) : "memory");
}
// Until at most N of this wave's loads are in flight.
template <int N>
__device__ __forceinline__ void wait_loads() {
  asm volatile("s_waitcnt vmcnt(%0)" :: "n"(N) : "memory");
}

template <int Q_DT, int OUT_DT, bool GEN>
__global__ void __launch_bounds__(kPfThreads) __attribute__((amdgpu_waves_per_eu(2)))
prefill_runs_kernel(RunArgs p) {
  const DecodeArgs& a = p.a;
  __shared__ __attribute__((aligned(1024))) char s_lds[kPfRaws * kPfRaw + kPfBufs * kPfStage];
  __shared__ int64_t s_prefix[kOrderMax + 1];  // every workgroup scans the sequences' costs
  __shared__ int64_t s_wave[kPfWaves];
  const int tid = int(threadIdx.x);
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int Hkv = a.num_kv_heads;
  OrderLds& seqs = *reinterpret_cast<OrderLds*>(s_lds);
  static_assert(sizeof(OrderLds) <= sizeof(s_lds), "the stages hold it until the first one");
  const PfStep found = pf_step<kPfThreads>(p, s_prefix, s_wave, seqs);
  if (!found.take) {
    __syncthreads();
    if (blockIdx.x == 0) order_blocks<kPfThreads>(a, p.num_seqs, p.tq, p.blocks, p.order, seqs);
    return;
  }
  if (blockIdx.x == 0 && tid == 0) p.blocks[p.num_seqs] = -1;
  const int64_t T = found.T;
  const int M = uniform(pf_runs(p, T));
  // Workgroup w runs on XCD w % 8: a kv head's runs, in order, on as few XCDs
  // as there are for it, since neighbouring runs read the same keys.
  const int w = int(blockIdx.x);
  int j = w / Hkv, h = w - j * Hkv;
  if (Hkv < 8 && 8 % Hkv == 0 && gridDim.x % 8 == 0) {
    const int per = 8 / Hkv, xcd = w & 7;
    const int share = (M + per - 1) / per;
    h = xcd % Hkv;
    j = (w >> 3) < share ? (xcd / Hkv) * share + (w >> 3) : p.s.max_runs;
  }
  // run j's partial records: slot 0 the one of its first block, unless it
  // begins that block; slot 1 of a block it begins and does not end (its last)
  if (w == 0)
    for (int i = tid; i < 2 * (p.s.max_runs - M); i += kPfThreads) p.s.desc[2 * M + i].valid = 0;
  if (j >= M) return;
  if (h == 0 && tid < 2) p.s.desc[2 * j + tid].valid = 0;
  if (T == 0) return;
  const int64_t x_begin = uniform(pf_run_start(T, j, M));
  const int64_t x_end = uniform(pf_run_start(T, j + 1, M));
  const PfBlock k_first = pf_block(p, s_prefix, x_begin);
  __syncthreads();  // the descriptors' initial stores come before run j's own

  // staging: thread t moves 16-byte chunk t & 7 of key t >> 3 of a stage, of K and of V
  const int lk = tid >> 3, lc = tid & 7;
  const uint32_t raw0 = (uint32_t)(size_t)(lvoid*)s_lds;
  const uint32_t stage0 = raw0 + kPfRaws * kPfRaw;
  const uint32_t st_k = stage0 + uint32_t(lk * 256 + (((2 * lc) ^ (lk & 15)) << 4));
  const uint32_t st_v = stage0 + kPfHalf + uint32_t(lk * 256 + (((2 * lc) ^ (4 * (lk & 3) | (lk & 1))) << 4));
  // read side (see the comment above): K key lane % 32, chunk 8 (lane / 32) + t
  // for MFMA t; V key 4 (lane / 32) + (lane % 16) / 4 of each 8, columns 32 d +
  // 16 ((lane / 16) % 2) + 4 (lane % 4) .. + 3
  const int kk = lane & 31, half = lane >> 5;
  const uint32_t rd_k0 = stage0 + uint32_t(kk * 256 + (((8 * half) ^ (kk & 15)) << 4));
  const int vk = (lane & 15) >> 2;
  const uint32_t rd_v0 = stage0 + kPfHalf +
                         uint32_t((4 * half + vk) * 256 +
                                  (((2 * ((lane >> 4) & 1) + ((lane & 3) >> 1)) ^ (4 * vk | (vk & 1))) << 4) +
                                  8 * (lane & 1));

  // The pieces of the run: its blocks after its first, in order, then its part
  // of the first.  For blocks of about one length the runs of a sequence then
  // read the same keys at the same time (whole blocks and heads of blocks from
  // the start of the keys; the tails, which begin as far into the keys as the
  // heads before them ended, a fixed distance behind), out of one XCD's L2.
  struct Piece {
    PfBlock k;
    int sa, sb, ns, key_end;  // stages [sa, sb) of the block's ns
  };
  const int64_t x_first = min(x_end, k_first.at + k_first.cost);
  int64_t x = x_first;
  PfBlock k_last = k_first;
  bool first_left = true;
  auto next_piece = [&](Piece& c) {  // uniform over the workgroup
    for (;;) {
      int64_t lo, hi;
      if (x < x_end) {
        if (k_last.i + 1 < k_last.nb) {
          ++k_last.i;
          k_last.at += k_last.cost;
          k_last.cost += k_last.step;
        } else {
          k_last = pf_block(p, s_prefix, x);
        }
        c.k = k_last;
        lo = x;
        hi = min(x_end, c.k.at + c.k.cost);
        x = hi;
      } else if (first_left) {
        first_left = false;
        c.k = k_first;
        lo = x_begin;
        hi = x_first;
      } else {
        return false;
      }
      c.ns = uniform(c.k.stages(a, p.tq));
      c.key_end = uniform(c.k.key_end(a, p.tq));
      const bool begins = lo == c.k.at;
      c.sa = uniform(c.k.stage_at(lo, c.ns));
      c.sb = uniform(c.k.stage_at(hi, c.ns));
      if (c.sa < c.sb || (begins && c.ns == 0)) return true;
    }
  };

  const uint8_t* kbase = a.k + int64_t(h) * a.k_head;
  const uint8_t* vbase = a.v + int64_t(h) * a.v_head;
  const uint32_t off_k = uint32_t((lane >> 3) * a.k_row + 16 * lc);
  const uint32_t off_v = uint32_t((lane >> 3) * a.v_row + 16 * lc);
  // The pages of a piece's stages.  Without GEN the block size is a multiple
  // of 8, so the 8 keys a wave stages lie in one page: its id and row are
  // wave-uniform (lane i holds those of stage win + i), the row addresses
  // scalar and each lane's offset fixed.  With GEN every thread looks up its
  // own key's page, a stage ahead.  Missing pages are -1.
  struct Pages {
    int32_t id, row;
  };
  auto look_up = [&](const Piece& c, int t0) {
    const int key = (t0 + (GEN ? 0 : lane)) * kPfKeys + (GEN ? lk : 8 * wave);
    Pages g{-1, 0};
    if (key < c.key_end && t0 < c.sb) {
      const int pi = page_index(a, key);
      g.row = key - pi * a.block_size;
      if (pi < a.bt_width) g.id = a.block_table[int64_t(c.k.b) * a.bt_stride + pi];
      if (g.id >= a.num_blocks) g.id = -1;
    }
    return g;
  };
  int win = 0;
  Pages pages{-1, 0};
  bool holes = false;  // some stage of the piece started fewer loads than two
  // starts the loads of stage t into raw buffer `slot`, straight to LDS (each
  // wave's 1 KiB of K and of V, a lane's 16 bytes at 16 * tid); keys past
  // key_end and rows on missing pages are zeroed instead
  auto issue = [&](const Piece& c, int t, uint32_t slot) {
    if (t >= c.sb) return;
    const uint32_t lds_k = raw0 + slot + uint32_t(1024 * wave), lds_v = lds_k + kPfRaw / 2;
    bool in = t * kPfKeys + lk < c.key_end;
    if constexpr (GEN) {
      in = in && pages.id >= 0;
      const bool full = __all(in);
      if (in) {
        load_lds(lds_k, kbase + int64_t(pages.id) * a.k_blk + int64_t(pages.row) * a.k_row + 16 * lc);
        load_lds(lds_v, vbase + int64_t(pages.id) * a.v_blk + int64_t(pages.row) * a.v_row + 16 * lc);
      }
      pages = look_up(c, t + 1);
      if (full) return;
    } else {
      if (t - win >= 64) {
        win = t;
        pages = look_up(c, t);
      }
      const int64_t id = __builtin_amdgcn_readlane(pages.id, t - win);
      const int64_t row = __builtin_amdgcn_readlane(pages.row, t - win);
      const uint8_t* kp = kbase + (id * a.k_blk + row * a.k_row);
      const uint8_t* vp = vbase + (id * a.v_blk + row * a.v_row);
      if (id >= 0 && (t + 1) * kPfKeys <= c.key_end) {
        load_lds(lds_k, kp, off_k);
        load_lds(lds_v, vp, off_v);
        return;
      }
      in = in && id >= 0;
      if (in) {
        load_lds(lds_k, kp, off_k);
        load_lds(lds_v, vp, off_v);
      }
    }
    holes = true;
    if (!in) {
      *lds_at<u32x4>(raw0 + slot + uint32_t(16 * tid)) = u32x4(0);
      *lds_at<u32x4>(raw0 + slot + kPfRaw / 2 + uint32_t(16 * tid)) = u32x4(0);
    }
  };
  // a piece's first three stages, given the pages of its first
  auto open = [&](const Piece& c, const Pages& g) {
    win = c.sa;
    pages = g;
    holes = false;
    issue(c, c.sa, 0);
    issue(c, c.sa + 1, kPfRaw);
    issue(c, c.sa + 2, 2 * kPfRaw);
  };

  Piece c;
  if (!next_piece(c)) return;
  open(c, look_up(c, c.sa));
  for (;;) {  // over the pieces
    const PfBlock& k = c.k;
    const int sa = c.sa, sb = c.sb, ns = c.ns, key_end = c.key_end;
    const int b = k.b, i0 = k.i * p.tq;
    const int n = k.n, L = k.len;
    const int ni = min(p.tq, n - i0);
    const int64_t qf = q_first(a, b);
    const int G = a.heads;
    // causal: query token i sees keys below base + i (FA's bottom-right alignment)
    const int base = a.causal ? L - n + 1 : L;
    const int mask_from = a.causal ? min(max(base + i0, 0), L) : L;  // keys every row sees
    const float qd = descale(a.qd, a.qd_b, a.qd_h, b, h);
    const float kd = descale(a.kd, a.kd_b, a.kd_h, b, h);
    // exp2-domain score scale; a negative one is applied as -q~ (exact) times |sl|
    const float sl_signed = a.scale_log2 * qd * kd;
    const float sl = __int_as_float(uniform(__float_as_int(__builtin_fabsf(sl_signed))));

    const int r = wave * 32 + kk;
    const int ti = r / G, g = r - ti * G;
    const bool live = ti < ni;
    // this lane's scores are of keys 4 half + const: the row's limit less that
    const int row_lim = (live ? (a.causal ? min(max(base + i0 + ti, 0), L) : L) : 0) - 4 * half;

    bf16x8 qop[8];
    {
      uint32_t qw[16];
      // (rows without a query token read the block's first, and zero it)
      {
        const char* src = a.q + (qf + i0 + (live ? ti : 0)) * a.q_tok_stride + int64_t(h * G + g) * a.q_head_stride;
        uint32_t q0[8], q1[8];
        load_query_as<Q_DT>(src, qd, 64 * half, q0);
        load_query_as<Q_DT>(src, qd, 64 * half + 32, q1);
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          qw[i] = live ? q0[i] : 0u;
          qw[8 + i] = live ? q1[i] : 0u;
        }
      }
      if (sl_signed < 0.0f) {
#pragma unroll
        for (int i = 0; i < 16; ++i) qw[i] ^= 0x80808080u;  // -q~: E4M3 sign bits
      }
#pragma unroll
      for (int c = 0; c < 8; ++c) qop[c] = e4m3x8_to_bf16(qw[2 * c], qw[2 * c + 1]);
    }
    // Softmax state: m, the row's maximum of the first 32 keys of the run, is
    // raised only when a lane's 16 weights of a tile pass 2^15 in sum (until
    // then each is a finite fp16 value), so the common path has one compare
    // and branch per tile and no rescale.  Rows without a query token keep m =
    // +kBig (every p is 0).
    constexpr float kBig = 1.0e30f;
    constexpr float kMaxTileSum = 32768.0f;
    float m = kBig, l = 0.0f;
    f32x16 o[4];
#pragma unroll
    for (int d = 0; d < 4; ++d) o[d] = f32x16{};
    const bool busy = wave * 32 < ni * G;  // waves without a query row only stage

    // K as bf16 and V as fp16 (both exact), converted once here for every
    // wave, from the raw bytes this thread loaded
    auto stage_read = [&](uint32_t slot, u32x4& kr, u32x4& vr) {
      kr = *lds_at<u32x4>(raw0 + slot + uint32_t(16 * tid));
      vr = *lds_at<u32x4>(raw0 + slot + kPfRaw / 2 + uint32_t(16 * tid));
    };
    auto stage_store = [&](uint32_t buf, const u32x4& kr, const u32x4& vr, int quarter) {
      switch (quarter) {
        case 0: *lds_at<u32x4>(st_k + buf) = __builtin_bit_cast(u32x4, e4m3x8_to_bf16(kr[0], kr[1])); break;
        case 1: *lds_at<u32x4>((st_k ^ 16u) + buf) = __builtin_bit_cast(u32x4, e4m3x8_to_bf16(kr[2], kr[3])); break;
        case 2: *lds_at<u32x4>(st_v + buf) = __builtin_bit_cast(u32x4, e4m3x8_to_f16(vr[0], vr[1])); break;
        default: *lds_at<u32x4>((st_v ^ 16u) + buf) = __builtin_bit_cast(u32x4, e4m3x8_to_f16(vr[2], vr[3])); break;
      }
    };
    // LDS addresses of this lane's K and V reads in the stage being read, moved
    // from buffer to buffer (the empty asm keeps them in registers: left
    // alone, the compiler forms every address anew at its read)
    uint32_t rd_k[8], rd_v[4];
#pragma unroll
    for (int c = 0; c < 8; ++c) rd_k[c] = rd_k0 ^ uint32_t(16 * c);
#pragma unroll
    for (int d = 0; d < 4; ++d) rd_v[d] = rd_v0 ^ uint32_t(64 * d);
    auto move_k = [&](uint32_t by) {
#pragma unroll
      for (int c = 0; c < 8; ++c) {
        rd_k[c] += by;
        asm volatile("" : "+v"(rd_k[c]));
      }
    };
    auto move_v = [&](uint32_t by) {
#pragma unroll
      for (int d = 0; d < 4; ++d) {
        rd_v[d] += by;
        asm volatile("" : "+v"(rd_v[d]));
      }
    };
    // the V^T operand of step u of a tile, columns 32 d .. + 31
    auto load_v = [&](int tile, int u, int d) {
      const uint32_t at = rd_v[d] + uint32_t(8192 * tile + 4096 * u);
      const s16x4 t0 = __builtin_amdgcn_ds_read_tr16_b64_v4i16(lds_at<s16x4>(at));
      const s16x4 t1 = __builtin_amdgcn_ds_read_tr16_b64_v4i16(lds_at<s16x4>(at + 2048));
      return __builtin_bit_cast(f16x8, __builtin_shufflevector(t0, t1, 0, 1, 2, 3, 4, 5, 6, 7));
    };
    // the lane's key i of a tile, before its 4 half
    auto key_of = [](int i) { return 8 * (i >> 2) + (i & 3); };
    // the row's largest scaled score of a tile (sl >= 0: max(y) * sl)
    auto tile_max = [&](const f32x16& y, int key0) {
      float v = -__builtin_inff();
#pragma unroll
      for (int i = 0; i < 16; ++i) v = __builtin_fmaxf(v, key0 + key_of(i) < row_lim ? y[i] : -__builtin_inff());
      v *= sl;
      v = __builtin_fmaxf(v, __shfl_xor(v, 32));
      return live ? __builtin_fmaxf(v, kNegBig) : kBig;
    };
    // P of two keys (elements i, i + 1) of a tile in fp16 (RNE, relative error
    // <= 2^-11 from 2^-14 up), and their sums
    auto weigh = [&](auto masked_tag, const f32x16& y, int key0, int i, float& s0, float& s1, uint32_t (&pw)[8]) {
      constexpr bool MASKED = decltype(masked_tag)::value;
      float e0 = __builtin_fmaf(y[i], sl, -m), e1 = __builtin_fmaf(y[i + 1], sl, -m);
      if (MASKED && key0 + key_of(i) >= row_lim) e0 = -__builtin_inff();
      if (MASKED && key0 + key_of(i + 1) >= row_lim) e1 = -__builtin_inff();
      const float p0 = __builtin_amdgcn_exp2f(e0), p1 = __builtin_amdgcn_exp2f(e1);
      s0 += p0;
      s1 += p1;
      pw[i / 2] = __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2{p0, p1}), f16x2));
    };
    // One tile's step of the wave's pipeline, three independent strands that
    // fill the matrix and vector units together: the softmax of a tile (scores
    // y, its weights to pw), the scores of the tile after it (returned; K tile
    // k_tile) and P V of the tile before it (weights pv, V tile v_tile), in
    // eight groups of one MFMA of each product, two keys' softmax and the LDS
    // reads of two groups on.  The order is fixed (sched_barrier): left alone,
    // the compiler reads each operand right before its MFMA and waits for it.
    // extra(c): more work for group c.
    auto tile_step = [&](auto masked_tag, const f32x16& y, int key0, int k_tile, int v_tile, const uint32_t (&pv)[8],
                         uint32_t (&pw)[8], const auto& extra) {
      u32x4 kw[8];
      f16x8 vw[8];
      auto read = [&](int c) {
        kw[c] = *lds_at<u32x4>(rd_k[c] + uint32_t(8192 * k_tile));
        vw[c] = load_v(v_tile, c >> 2, c & 3);
      };
      float s0 = 0.0f, s1 = 0.0f;
      f32x16 yn = {};
      read(0);
      read(1);
      __builtin_amdgcn_sched_barrier(0);
      weigh(masked_tag, y, key0, 0, s0, s1, pw);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int c = 0; c < 8; ++c) {
        const int u = c >> 2, d = c & 3;
        if (c + 2 < 8) read(c + 2);
        yn = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, kw[c]), qop[c], yn, 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
        if (c < 7) weigh(masked_tag, y, key0, 2 * c + 2, s0, s1, pw);
        const f16x8 pop = __builtin_bit_cast(f16x8, u32x4{pv[4 * u], pv[4 * u + 1], pv[4 * u + 2], pv[4 * u + 3]});
        o[d] = __builtin_amdgcn_mfma_f32_32x32x16_f16(vw[c], pop, o[d], 0, 0, 0);
        extra(c);
        __builtin_amdgcn_sched_barrier(0);
      }
      float sum = s0 + s1;
      if (__builtin_expect(__any(!(sum <= kMaxTileSum)), 0)) {  // (NaN scores come here too)
        const float mn = __builtin_fmaxf(m, tile_max(y, key0));
        const float f = __builtin_amdgcn_exp2f(m - mn);
        m = mn;
        l *= f;
#pragma unroll
        for (int d = 0; d < 4; ++d) o[d] *= f;
        s0 = s1 = 0.0f;
#pragma unroll
        for (int i = 0; i < 16; i += 2) weigh(std::true_type{}, y, key0, i, s0, s1, pw);
        sum = s0 + s1;
      }
      l += sum;
      return yn;
    };

    // The run's stages.  Stage t + 1 is complete in its buffer from the barrier
    // of step t on.  Step t starts the loads of stage t + 4 and converts stage
    // t + 2 into the third buffer at its end (every wave left that one before
    // the step's barrier); a wave converts what it loaded itself, so its own
    // load counter is all it waits for: two loads each of the two later
    // stages may be in flight.  Past the run's last stage stale bytes are
    // converted, and the scores of stale bytes taken, and neither is used.
    const int t_open = min(sb, mask_from / kPfKeys);  // stages below need no mask
    // the next piece and its first pages, while this one's first loads fly
    Piece c_next;
    const bool more = next_piece(c_next);
    Pages pages_next{-1, 0};
    if (more) pages_next = look_up(c_next, c_next.sa);
    {
      u32x4 kr, vr;
      wait_loads<0>();
      lds_barrier();  // the buffers' previous readers are done
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        stage_read(i * kPfRaw, kr, vr);
#pragma unroll
        for (int q = 0; q < 4; ++q) stage_store(i * kPfStage, kr, vr, q);
      }
      issue(c, sa + 3, 0);
      lds_barrier();
    }
    uint32_t raw = kPfRaw;        // the raw buffer of stage t + 1, then of t + 4
    uint32_t to = 2 * kPfStage;   // the buffer that stage t + 2 goes to
    uint32_t to_next = kPfStage;  // from the buffer of stage t to that of stage t + 1
    f32x16 y0 = {};
    uint32_t p0[8], p1[8];  // weights of the stage's two tiles
#pragma unroll
    for (int i = 0; i < 8; ++i) p1[i] = 0u;  // before the first tile: zero weights (on that stage's own V)
    if (busy) {
#pragma unroll
      for (int c = 0; c < 8; ++c)
        y0 = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, *lds_at<u32x4>(rd_k[c])), qop[c], y0, 0,
                                                     0, 0);
      m = tile_max(y0, sa * kPfKeys);
    }
    uint32_t from_last = 0;  // from the buffer of stage t - 1 to that of stage t
    auto step = [&](int t, auto masked_tag) {
      issue(c, t + 4, raw);
      raw = raw == 2 * kPfRaw ? 0 : raw + kPfRaw;
      f32x16 y1;
      if (busy) {
        y1 = tile_step(masked_tag, y0, t * kPfKeys, 1, 1, p1, p0, [&](int c) {
          if (c == 6) move_k(to_next);
          if (c == 7) move_v(from_last);
        });
      }
      lds_barrier();
      u32x4 kr, vr;
      if (t + 4 < sb && !holes) wait_loads<4>(); else wait_loads<0>();
      stage_read(raw, kr, vr);
      if (busy) {
        y0 = tile_step(masked_tag, y1, t * kPfKeys + 32, 0, 0, p0, p1, [&](int c) {
          if (c >= 4) stage_store(to, kr, vr, c - 4);
        });
      } else {
#pragma unroll
        for (int q = 0; q < 4; ++q) stage_store(to, kr, vr, q);
      }
      from_last = to_next;
      to = to == 2 * kPfStage ? 0 : to + kPfStage;
      to_next = to == 2 * kPfStage ? kPfStage : to == 0 ? kPfStage : 0u - 2 * kPfStage;
    };
    // nothing is left in flight into registers the loop reads: the compiler
    // would wait for it, and with it for the coming stages' loads, in every step
    __builtin_amdgcn_s_waitcnt(0xF70);  // vmcnt(0)
    int t = sa;
    for (; t < t_open; ++t) step(t, std::false_type{});
    for (; t < sb; ++t) step(t, std::true_type{});
    if (busy && sa < sb) {  // the last tile's P V
#pragma unroll
      for (int c = 0; c < 8; ++c) {
        const int u = c >> 2, d = c & 3;
        const f16x8 pop = __builtin_bit_cast(f16x8, u32x4{p1[4 * u], p1[4 * u + 1], p1[4 * u + 2], p1[4 * u + 3]});
        o[d] = __builtin_amdgcn_mfma_f32_32x32x16_f16(load_v(1, u, d), pop, o[d], 0, 0, 0);
      }
    }

    // the next piece's first loads fly while this one's result is written
    if (more) open(c_next, pages_next);
    const float lt = l + __shfl_xor(l, 32);
    f32x4 frag[16];
#pragma unroll
    for (int c = 0; c < 16; ++c)
      frag[c] = f32x4{o[c >> 2][4 * (c & 3)], o[c >> 2][4 * (c & 3) + 1], o[c >> 2][4 * (c & 3) + 2],
                      o[c >> 2][4 * (c & 3) + 3]};
    if (sa == 0 && sb == ns) {
      write_row<OUT_DT, 4>(a, q_first(a, b) + i0, ni, h, descale(a.vd, a.vd_b, a.vd_h, b, h), wave, lane, 0, frag, m, lt);
    } else {
      const int slot = sa == 0 ? 1 : 0;
      if (h == 0 && tid == 0) p.s.desc[2 * j + slot] = RunDesc{1, b, k.i, q_count(a, b)};
      if (busy) {
        float* rec = p.s.records + ((int64_t(j) * Hkv + h) * 2 + slot) * kRunRecord + wave * kRunSlab;
#pragma unroll
        for (int c = 0; c < 16; ++c) *reinterpret_cast<f32x4*>(rec + (c * 64 + lane) * 4) = frag[c];
        if (lane < 32) {
          rec[4096 + lane] = m;
          rec[4096 + 32 + lane] = lt;
        }
      }
    }
    if (!more) return;
    c = c_next;
  }
}

// The merge of a step that is cut into runs whatever its lengths.
template <int OUT_DT>
__global__ void __launch_bounds__(kRunThreads) prefill_merge_kernel(DecodeArgs a, int tq, RunSpace s) {
  __shared__ MergeLds lds;
  merge_records<OUT_DT, 4>(a, tq, s, lds);
}

template <int Q_DT, bool GEN>
void launch_prefill_q(const RunArgs& p, int out_dtype, dim3 grid, hipStream_t st) {
  if (out_dtype == PSK_DTYPE_BF16)
    hipLaunchKernelGGL((prefill_runs_kernel<Q_DT, PSK_DTYPE_BF16, GEN>), grid, dim3(kPfThreads), 0, st, p);
  else
    hipLaunchKernelGGL((prefill_runs_kernel<Q_DT, PSK_DTYPE_F32, GEN>), grid, dim3(kPfThreads), 0, st, p);
}

template <bool GEN>
void launch_prefill(const RunArgs& p, int q_dtype, int out_dtype, dim3 grid, hipStream_t st) {
  switch (q_dtype) {
    case PSK_DTYPE_FP8_E4M3FN: launch_prefill_q<PSK_DTYPE_FP8_E4M3FN, GEN>(p, out_dtype, grid, st); break;
    case PSK_DTYPE_BF16: launch_prefill_q<PSK_DTYPE_BF16, GEN>(p, out_dtype, grid, st); break;
    case PSK_DTYPE_F16: launch_prefill_q<PSK_DTYPE_F16, GEN>(p, out_dtype, grid, st); break;
    default: launch_prefill_q<PSK_DTYPE_F32, GEN>(p, out_dtype, grid, st); break;
  }
}

}  // namespace

namespace psk_detail {

// One workgroup per CU (its LDS stages and 256 registers a wave leave no room
// for a second).
int64_t prefill_cus() {
  static std::mutex mu;
  static std::map<int, int64_t> cache;
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess) return 0;
  std::lock_guard<std::mutex> lock(mu);
  auto it = cache.find(dev);
  if (it != cache.end()) return it->second;
  int cus = 0;
  if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess) return 0;
  cache[dev] = std::min(cus, kRunMaxWgs);
  return cache[dev];
}

// Alignment to 16 bytes, the descriptors and the records.
int64_t prefill_runs_words() { return 4 + 2 * kRunMaxWgs * (kRunRecord + int64_t(sizeof(RunDesc) / 4)); }

int launch_prefill_runs(const DecodeArgs& a, int64_t num_seqs, int64_t wgs, bool sure, int q_dtype, int out_dtype,
                        int32_t* workspace, int32_t* blocks, int32_t* order, RunSpace* space, hipStream_t st) {
  RunArgs p{};
  p.a = a;
  p.num_seqs = int32_t(num_seqs);
  p.tq = kPfRows / a.heads;
  p.wgs = int32_t(std::min<int64_t>(wgs, INT32_MAX));
  p.cus = int32_t(prefill_cus());
  p.sure = sure ? 1 : 0;
  p.blocks = blocks;
  p.order = order;
  p.s.max_runs = p.cus / a.num_kv_heads;
  p.s.desc = reinterpret_cast<RunDesc*>((reinterpret_cast<uintptr_t>(workspace) + 15) & ~uintptr_t(15));
  p.s.records = reinterpret_cast<float*>(p.s.desc + 2 * p.s.max_runs);
  *space = p.s;
  const dim3 grid{unsigned(p.s.max_runs * a.num_kv_heads), 1u, 1u};
  // pages of a multiple of 8 keys whose rows lie within 32-bit offsets: a
  // wave's staged keys share a page
  const bool uniform_pages = a.block_size % 8 == 0 && a.k_row >= 0 && a.v_row >= 0 &&
                             8 * std::max(a.k_row, a.v_row) < (int64_t(1) << 31);
  if (uniform_pages) launch_prefill<false>(p, q_dtype, out_dtype, grid, st);
  else launch_prefill<true>(p, q_dtype, out_dtype, grid, st);
  const int st1 = check_launch("prefill_runs_kernel launch");
  if (!sure || st1 != PSK_OK) return st1;
  const dim3 grid2{unsigned(4 * p.s.max_runs * a.num_kv_heads), 1u, 1u};  // a task a wave where every run shares a block
  if (out_dtype == PSK_DTYPE_BF16)
    hipLaunchKernelGGL((prefill_merge_kernel<PSK_DTYPE_BF16>), grid2, dim3(kRunThreads), 0, st, a, p.tq, p.s);
  else
    hipLaunchKernelGGL((prefill_merge_kernel<PSK_DTYPE_F32>), grid2, dim3(kRunThreads), 0, st, a, p.tq, p.s);
  return check_launch("prefill_merge_kernel launch");
}

}  // namespace psk_detail
