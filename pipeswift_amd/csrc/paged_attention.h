// What the FP8 paged attention kernels share (the decode reader of
// paged_attention.hip and the prefill kernel of prefill_attention.hip): their
// arguments, the exact FP8 conversions and the query load.

#ifndef PSK_PAGED_ATTENTION_H
#define PSK_PAGED_ATTENTION_H

#include <hip/hip_runtime.h>

#include <stdint.h>

#include "pipeswift_kv.h"
#include "psk_common.h"

namespace psk_detail {

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef int i32x2 __attribute__((ext_vector_type(2)));
typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));

constexpr int kHead = 128;  // head_dim of the MFMA tiling
constexpr float kNegBig = -1.0e30f;  // finite "no token yet" maximum

typedef __attribute__((address_space(1))) void gvoid;
typedef __attribute__((address_space(3))) void lvoid;

// Runs of the decode reader's balanced schedule that hold a sequence's first and last tile.
struct RunSpan {
  uint16_t first, last;
};

struct DecodeArgs {
  const char* q;
  int64_t q_tok_stride;   // bytes
  int64_t q_head_stride;  // bytes
  const uint8_t* k;
  const uint8_t* v;
  int64_t k_blk, k_row, k_head;  // bytes
  int64_t v_blk, v_row, v_head;
  const int32_t* block_table;
  int64_t bt_stride;
  int64_t bt_width;
  const int32_t* seq_lens;
  int32_t num_blocks;
  int32_t block_size;
  int32_t bs_shift;  // log2(block_size) or -1
  int32_t num_kv_heads;
  int32_t group;     // MFMA rows per (sequence, kv head): q_len query tokens x heads
  int32_t heads;     // query heads per kv head
  int32_t q_len;     // query token slots per sequence (the most query tokens any sequence has)
  const int32_t* cu_q;  // query tokens of sequence b: [cu_q[b], cu_q[b+1]); NULL: [b q_len, (b+1) q_len)
  int32_t causal;    // query token i of n of a sequence of length L sees keys [0, L - n + 1 + i)
  int32_t split;     // tokens per workgroup
  int32_t max_splits;
  float scale_log2;  // softmax_scale * log2(e)
  const float* qd;
  int64_t qd_b, qd_h;
  const float* kd;
  int64_t kd_b, kd_h;
  const float* vd;
  int64_t vd_b, vd_h;
  float* part;       // partial records of G * (kHead + 2) floats: [B][Hkv][max_splits] (splits) or
                     // [(B + stream_wgs) * Hkv] (balanced schedule)
  RunSpan* spans;    // balanced schedule: of each sequence with tokens, [B]
  int32_t stream_wgs;  // balanced schedule: runs per kv head; 0 with splits
  int32_t seq_units;   // balanced schedule: units that stand for the start of a sequence
  char* out;
  int64_t out_tok_stride;   // bytes
  int64_t out_head_stride;  // bytes
  float* lse;               // [Hq][lse_head_stride] (entry [hq][b]) or nullptr
  int64_t lse_head_stride;
};

// First query token of sequence b and how many it has (at most q_len).
__device__ __forceinline__ int64_t q_first(const DecodeArgs& a, int b) {
  return a.cu_q ? int64_t(a.cu_q[b]) : int64_t(b) * a.q_len;
}
__device__ __forceinline__ int q_count(const DecodeArgs& a, int b) {
  return a.cu_q ? max(0, min(a.q_len, a.cu_q[b + 1] - a.cu_q[b])) : a.q_len;
}

__device__ __forceinline__ float descale(const float* p, int64_t sb, int64_t sh, int b, int h) {
  return p ? p[b * sb + h * sh] : 1.0f;
}

// Eight E4M3FN bytes (w0 then w1, in byte order) -> eight bf16, exactly: every
// E4M3FN value is a bf16 value.
__device__ __forceinline__ bf16x8 e4m3x8_to_bf16(uint32_t w0, uint32_t w1) {
  const bf16x2 a = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(w0, 1.0f, false);
  const bf16x2 b = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(w0, 1.0f, true);
  const bf16x2 c = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(w1, 1.0f, false);
  const bf16x2 d = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(w1, 1.0f, true);
  return bf16x8{a[0], a[1], b[0], b[1], c[0], c[1], d[0], d[1]};
}

// The same to fp16, exactly: E4M3FN's 3-bit mantissas and exponents 2^-9 ..
// 2^8 (448 at most) all lie in fp16's range and precision.
__device__ __forceinline__ f16x8 e4m3x8_to_f16(uint32_t w0, uint32_t w1) {
  const f16x2 a = __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(w0, 1.0f, false);
  const f16x2 b = __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(w0, 1.0f, true);
  const f16x2 c = __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(w1, 1.0f, false);
  const f16x2 d = __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(w1, 1.0f, true);
  return f16x8{a[0], a[1], b[0], b[1], c[0], c[1], d[0], d[1]};
}

__device__ __forceinline__ int page_index(const DecodeArgs& a, int t) {
  return a.bs_shift >= 0 ? (t >> a.bs_shift) : (t / a.block_size);
}

// 32 FP8 query bytes of this lane's MFMA row (query head h*G + lane%16, d from
// 32 * (lane / 16)); zero rows beyond the group.
template <int Q_DT>
__device__ __forceinline__ void load_query_as(const char* src, float qd, int d0, uint32_t qw[8]) {
  if constexpr (Q_DT == PSK_DTYPE_FP8_E4M3FN) {
    const u32x4 lo = *reinterpret_cast<const u32x4*>(src + d0);
    const u32x4 hi = *reinterpret_cast<const u32x4*>(src + d0 + 16);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      qw[i] = lo[i];
      qw[4 + i] = hi[i];
    }
  } else {
    constexpr int kEsz = Elt<Q_DT>::kSize;
    constexpr int E = 16 / kEsz;  // elements per 16-byte load
    using QC = QuantConv<Q_DT, E, kNanTorch>;  // the query is quantized as fp8_kv.quantize does
    const QScale qs = make_qscale(qd);
    uint8_t bytes[32];
#pragma unroll
    for (int i = 0; i < 32 / E; ++i) {
      const typename QC::In x = *reinterpret_cast<const typename QC::In*>(src + (d0 + E * i) * kEsz);
      const typename QC::Out y = QC::apply(x, qs);
      __builtin_memcpy(bytes + E * i, &y, E);
    }
    __builtin_memcpy(qw, bytes, 32);
  }
}

}  // namespace psk_detail

#endif  // PSK_PAGED_ATTENTION_H
