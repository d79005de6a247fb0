// Per-head q/k RMSNorm + RoPE + KV store of one token, shared by the fused
// call-site kernels (csrc/fused.hip) and the QKV projection's epilogue
// (csrc/gemm.hip): the arithmetic of model/model.py:47-52 and :86-99 with
// the reference's rounding points, and the K/V destination row of the
// llm.py:171-174 store or the model/model.py:233-240 decode append.
#pragma once

#include "aac_common.h"

namespace aac {

constexpr int kHeadDimFused = 128;

namespace fz {

template <Dt DT> struct Cvt;
template <> struct Cvt<Dt::BF16> {
  __device__ static inline float lo(u32 w) { return bf16lo(w); }
  __device__ static inline float hi(u32 w) { return bf16hi(w); }
  // v_cvt_pk_bf16_f32 (round to nearest even): the same bits as
  // f32_to_bf16_bits for every number, a fifth of its instructions
  __device__ static inline u32 pack(float a, float b) { return Elem<Dt::BF16>::pack2_hw(a, b); }
  __device__ static inline float round(float x) { return bf16lo(pack(x, x)); }
};
template <> struct Cvt<Dt::FP16> {
  __device__ static inline float lo(u32 w) { return f16lo(w); }
  __device__ static inline float hi(u32 w) { return f16hi(w); }
  __device__ static inline u32 pack(float a, float b) { return pack_f16x2(a, b); }
  __device__ static inline float round(float x) { return (float)(_Float16)x; }
};

template <Dt DT>
__device__ __forceinline__ void unpack8(const u32x4& w, float* f) {
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    f[2 * i] = Cvt<DT>::lo(w[i]);
    f[2 * i + 1] = Cvt<DT>::hi(w[i]);
  }
}
template <Dt DT>
__device__ __forceinline__ u32x4 pack8(const float* f) {
  u32x4 w;
#pragma unroll
  for (int i = 0; i < 4; ++i) w[i] = Cvt<DT>::pack(f[2 * i], f[2 * i + 1]);
  return w;
}

// Both values rounded to the activation type: bf16 has a convert of pairs (and
// two unpacks), fp16 converts one by one.
template <Dt DT>
__device__ __forceinline__ void round2(float& a, float& b) {
  if constexpr (DT == Dt::BF16) {
    const u32 w = Cvt<DT>::pack(a, b);
    a = Cvt<DT>::lo(w);
    b = Cvt<DT>::hi(w);
  } else {
    a = Cvt<DT>::round(a);
    b = Cvt<DT>::round(b);
  }
}

// 16 bytes to memory; NT: non-temporal, past the caches.
template <bool NT> __device__ __forceinline__ void put16(u16* p, const u32x4& w) {
  if constexpr (NT) __builtin_nontemporal_store(w, reinterpret_cast<u32x4*>(p));
  else *reinterpret_cast<u32x4*>(p) = w;
}

// 16 bytes read once; NT: non-temporal.
template <bool NT> __device__ __forceinline__ u32x4 get16(const u16* p) {
  if constexpr (NT) return __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(p));
  else return *reinterpret_cast<const u32x4*>(p);
}

__device__ __forceinline__ float wave_sum(float x) {
  x = row16_sum(x);
  x += __shfl_xor(x, 16);
  x += __shfl_xor(x, 32);
  return x;
}

// ------------------------------------------------- q/k RMSNorm + RoPE + store
struct QkArgs {
  const u16* qkv;
  int64_t qkv_stride;  // elements between tokens
  int64_t n_tokens;
  int32_t hq, hkv;
  const u16* qw;  // q_norm weight [128]
  const u16* kw;  // k_norm weight [128]
  float eps;
  const u16* cos;  // [max_pos, 128]
  const u16* sin;
  const int32_t* positions;  // [T]
  int32_t max_pos;
  u16* q_out;  // [T, hq, 128]
  u16* k_out;  // [T, hkv, 128] or null
  u16* k_cache;
  u16* v_cache;  // rows [*, hkv, 128]; null: no store
  const int64_t* slot_mapping;  // explicit rows, or null: paged append
  int64_t num_rows;
  const int32_t* block_tables;
  int32_t max_blocks;
  const int32_t* cache_seqlens;  // append position of token t (= sequence t)
  int32_t block_size;
  int64_t num_blocks;
};

// Destination cache row of token t for the K/V store, or -1 (none or out of range).
__device__ __forceinline__ int64_t cache_row(const QkArgs& a, int64_t t) {
  int64_t crow = -1;
  if (a.v_cache == nullptr) return crow;
  if (a.slot_mapping != nullptr) {
    crow = a.slot_mapping[t];
    if (crow >= a.num_rows) crow = -1;
  } else {
    const int p = a.cache_seqlens[t];
    if (p >= 0 && (int64_t)p < (int64_t)a.max_blocks * a.block_size) {
      const int blk = a.block_tables[t * a.max_blocks + p / a.block_size];
      if (blk >= 0 && blk < a.num_blocks) crow = (int64_t)blk * a.block_size + p % a.block_size;
    }
  }
  return crow;
}

// One query or key head row, held by the 16 lanes of a DPP row (lane li owns
// dims [8li, 8li+8)): RMSNorm over the head (model/model.py:47-52) and RoPE, out =
// x*cos + rotate_half(x)*sin with each product and the sum rounded
// (model/model.py:90-99); rotate_half pairs dim d with d +- 64, i.e. lane li
// with lane li ^ 8 (DPP row_ror:8).  The caller keeps the row's 16 lanes
// together on every branch.  sf holds sin with the sign of rotate_half folded
// in: negative in the lanes of the first half (li < 8), see signed_sin.
template <Dt DT>
__device__ __forceinline__ u32x4 norm_rope_row(const u32x4& xr, float eps, const float* wf, const float* cf,
                                               const float* sf) {
  // Each product and the sum are rounded separately; for fp16 those rounds
  // become half-precision operations, which contraction would merge into one
  // fused multiply-add (a single rounding, unlike the torch expression).
#pragma clang fp contract(off)
  float x[8];
  unpack8<DT>(xr, x);
  float ss = 0.f;
#pragma unroll
  for (int i = 0; i < 8; ++i) ss = fmaf(x[i], x[i], ss);
  ss = row16_sum(ss);
  const float rs = __frsqrt_rn(ss / (float)kHeadDimFused + eps);
#pragma unroll
  for (int i = 0; i < 8; ++i) x[i] *= rs;
#pragma unroll
  for (int i = 0; i < 8; i += 2) round2<DT>(x[i], x[i + 1]);
#pragma unroll
  for (int i = 0; i < 8; ++i) x[i] *= wf[i];
#pragma unroll
  for (int i = 0; i < 8; i += 2) round2<DT>(x[i], x[i + 1]);
  u32x4 packed;
#pragma unroll
  for (int i = 0; i < 8; i += 2) {
    float c[2], r[2];
#pragma unroll
    for (int e = 0; e < 2; ++e) {
      const float partner = __int_as_float(
          __builtin_amdgcn_update_dpp(0, __float_as_int(x[i + e]), 0x128, 0xF, 0xF, false));
      c[e] = x[i + e] * cf[i + e];
      r[e] = partner * sf[i + e];
    }
    round2<DT>(c[0], c[1]);
    round2<DT>(r[0], r[1]);
    packed[i / 2] = Cvt<DT>::pack(c[0] + r[0], c[1] + r[1]);
  }
  return packed;
}

// One head row of token t: a value head is copied into the cache, a query or
// key head goes through norm_rope_row.
template <Dt DT, bool NT = false>
__device__ __forceinline__ void norm_rope_head(const QkArgs& a, int64_t t, int hh, int li,
                                               const u32x4& xr, int64_t crow, const float* wf,
                                               const float* cf, const float* sf) {
  if (hh >= a.hq + a.hkv) {  // value head
    if (crow >= 0)
      put16<NT>(a.v_cache + (crow * a.hkv + (hh - a.hq - a.hkv)) * kHeadDimFused + li * 8, xr);
    return;
  }
  const u32x4 packed = norm_rope_row<DT>(xr, a.eps, wf, cf, sf);
  if (hh < a.hq) {
    put16<NT>(a.q_out + (t * a.hq + hh) * kHeadDimFused + li * 8, packed);
  } else {
    const int kh = hh - a.hq;
    if (a.k_out != nullptr) put16<NT>(a.k_out + (t * a.hkv + kh) * kHeadDimFused + li * 8, packed);
    if (crow >= 0) put16<NT>(a.k_cache + (crow * a.hkv + kh) * kHeadDimFused + li * 8, packed);
  }
}

// sin of the lane's dims, negated in the first half (a sign bit per packed value:
// as fp16 the products then still fold into half-precision operations): rounding
// is symmetric, so (-partner) * sin and partner * (-sin) are the same bits.
template <Dt DT>
__device__ __forceinline__ void signed_sin(const u32x4& sin8, int li, float* sf) {
  const u32 sign = li < 8 ? 0x80008000u : 0u;
  unpack8<DT>(u32x4{sin8[0] ^ sign, sin8[1] ^ sign, sin8[2] ^ sign, sin8[3] ^ sign}, sf);
}
template <Dt DT>
__device__ __forceinline__ void signed_sin(const u16* sin8, int li, float* sf) {
  signed_sin<DT>(*reinterpret_cast<const u32x4*>(sin8), li, sf);
}

__device__ __forceinline__ int clamp_pos(const QkArgs& a, int p) {
  return p < 0 ? 0 : (p >= a.max_pos ? a.max_pos - 1 : p);
}

}  // namespace fz
}  // namespace aac
