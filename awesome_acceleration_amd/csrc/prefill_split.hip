// Varlen causal GQA prefill of few queries (gfx950, bf16/fp16 MFMA): the call
// of prefill_wide.hip (flash_attn_varlen_func, llm.py:178-184; with the store
// llm.py:171-184) where its work items leave CUs idle.
//
// What bounds it: one request of a few hundred tokens is 1-10 us of matrix work
// for the chip, and the time is the chain of the longest item: start, first
// tiles, one key tile after the other, epilogue.  The wide kernel's item (128
// queries at G = 2, every key of its KV head in turn) makes 56 items of up to
// 13 tiles from 777 tokens at 16/8 heads, on 256 CUs.  Here an item is 32
// queries of two query heads of a KV head, and the keys are split over the
// workgroup's waves: wave (c, s) takes head c and the 32-key sub-tiles s, s + 4,
// s + 8, ..., so the chain is a sixteenth of the context's sub-tiles per
// 128 keys.  Two waves per SIMD run the two heads of a slice, one's softmax
// beside the other's MFMAs.  The four partial results of a head (reference
// max, row sum, O) are merged through LDS at the end.
//
// Tiles: per iteration the workgroup stages 128 keys of K and V (64 KiB)
// straight from global memory into one of two LDS stages; wave (0, s) brings
// slice s's K rows, wave (1, s) its V rows.  One barrier per iteration: past it
// every wave's tile has landed and the other stage is free for the next loads.
// Row layouts, fragments, masks, lazy rescaling and the probability rounding
// are those of prefill_wide.hip.

#include <algorithm>

#include "prefill_common.h"
#include "prefill_split.h"

namespace aac {
namespace ps {

using pf::Args;
using pf::D;
using pf::kRescale;

constexpr int kWaves = 8, kThreads = 64 * kWaves;
constexpr int kSlices = 4;                  // key slices (32 keys each per iteration)
constexpr int kSubBytes = 32 * D * 2;       // 8 KiB: a sub-tile of K or V
constexpr int kStageBytes = kSlices * 2 * kSubBytes;
constexpr int kOutPitch = D * 2 + 16;       // bytes of an output staging row
constexpr int kOutOff = 2 * kStageBytes;    // [2 heads][32 queries]
constexpr int kMlOff = kOutOff + 2 * 32 * kOutPitch;
constexpr int kLdsBytes = kMlOff + kWaves * 32 * 8;

typedef __attribute__((address_space(3))) unsigned char lds_u8;
typedef short v4s __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) v4s lds_v4s;

// 1 KiB from a buffer resource straight into LDS (dst + 16 lane); inline
// assembly, so that the compiler neither counts it nor guards LDS reads with
// waits for it: the waits are explicit.  M0 is used by nothing else here.
__device__ __forceinline__ void load_lds16(__amdgpu_buffer_rsrc_t r, int voff, int soff, u32 dst) {
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
  asm volatile("s_mov_b32 m0, %3\n\ts_nop 0\n\tbuffer_load_dwordx4 %0, %1, %2 offen lds"
               :
               : "v"(voff), "s"(r), "s"(soff), "s"(dst)
               : "memory", "m0");
#pragma clang diagnostic pop
}

// this wave's loads into LDS and LDS reads are done, then the workgroup's
__device__ __forceinline__ void landed_barrier() {
  asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

template <bool CAUSAL, bool STORE, bool F16>
__global__ __launch_bounds__(kThreads, 1) void prefill_split_kernel(Args a) {
  static_assert(CAUSAL || !STORE, "the store variant is causal self-attention");
  typedef pf::Mfma<F16> M;
  __shared__ __attribute__((aligned(1024))) unsigned char lds[kLdsBytes];
  const u32 lds0 = (u32)(uintptr_t)(lds_u8*)lds;

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int c = wave & 1, sl = wave >> 1;  // query head of the pair, key slice
  const int hl = lane >> 5, col = lane & 31;

  if (STORE && blockIdx.x == 0) {  // tokens outside [cu[0], cu[n])
    pf::store_kv_span<kThreads>(a, tid, 0, a.cu_q[0], 0, a.hkv);
    pf::store_kv_span<kThreads>(a, tid, a.cu_q[a.n_seqs], a.n_tok, 0, a.hkv);
  }

  // items: KV head fastest (one XCD per head when there are eight), heaviest
  // causal q-blocks first
  const int G = a.hq / a.hkv, pairs = G >> 1;
  int it = blockIdx.x;
  const int h = it % a.hkv;
  it /= a.hkv;
  const int pr = it % pairs;
  it /= pairs;
  const int sg = it % a.n_seqs, z = it / a.n_seqs;
  typedef const int32_t __attribute__((address_space(4))) cint;  // scalar loads
  const cint* cuq = (const cint*)(uintptr_t)a.cu_q;
  const cint* cuk = (const cint*)(uintptr_t)a.cu_k;
  const int q_beg = cuq[sg], Lq = cuq[sg + 1] - q_beg;
  const int k_beg = cuk[sg], Lk = min(cuk[sg + 1] - k_beg, a.max_k);
  const int nqb = (Lq + 31) / 32;
  if (z >= nqb) return;  // workgroup-uniform
  const int qb = CAUSAL ? nqb - 1 - z : z;
  const int q0 = qb * 32, qmax = min(q0 + 31, Lq - 1), shift = Lk - Lq;
  const int kv_end = CAUSAL ? max(0, min(Lk, qmax + 1 + shift)) : max(0, Lk);
  const int full = CAUSAL ? max(0, min(Lk, q0 + 1 + shift)) : Lk;  // keys below need no mask
  const int my_lim = CAUSAL ? min(Lk, q0 + col + 1 + shift) : Lk;
  const int nsub = (kv_end + 31) / 32, n_it = (nsub + kSlices - 1) / kSlices;
  const int head = h * G + 2 * pr;  // first query head of the pair

  // staging: instruction i brings rows 4 i + lane / 16 of this wave's sub-tile;
  // 16-byte chunk ch of row r sits at ch ^ (r & 15) (K) or ch ^ 4 (r & 3) (V)
  const int row_bytes = (int)((c == 0 ? a.k_stride : a.v_stride) * 2);
  const u16* base = (c == 0 ? a.k + (int64_t)k_beg * a.k_stride : a.v + (int64_t)k_beg * a.v_stride) + h * D;
  const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<u16*>(base), 0, kv_end > 0 ? (kv_end - 1) * row_bytes + D * 2 : 0, 0x00020000);
  const int r4 = lane >> 4;
  int voff[4];
#pragma unroll
  for (int i = 0; i < 4; ++i)
    voff[i] = r4 * row_bytes + 16 * ((lane & 15) ^ (c == 0 ? 4 * i + r4 : 4 * r4));
  const u32 dst0 = lds0 + (u32)(sl * 2 * kSubBytes + c * kSubBytes);
  auto issue = [&](int n) {
    const int key0 = 32 * (n * kSlices + sl);
#pragma unroll
    for (int i = 0; i < 8; ++i)
      load_lds16(rs, voff[i & 3], (key0 + 4 * i) * row_bytes, dst0 + (u32)((n & 1) * kStageBytes + i * 1024));
  };
  if (n_it > 0) issue(0);

  // Q fragments (B operand of S^T = K Q^T: lane = query)
  u32x4 qf[8];
  {
    const u16* qp = a.q + (int64_t)(q_beg + min(q0 + col, Lq - 1)) * a.q_stride + (head + c) * D + hl * 8;
#pragma unroll
    for (int t = 0; t < 8; ++t) qf[t] = *reinterpret_cast<const u32x4*>(qp + 16 * t);
  }
  // fragment addresses within a sub-tile (see prefill_wide.hip)
  int koff[8], vo[4];
#pragma unroll
  for (int t = 0; t < 8; ++t) koff[t] = col * 256 + 16 * ((2 * t + hl) ^ (col & 15));
  {
    const int g = lane >> 4, i = lane & 15;
    const int l0 = (4 * (g >> 1) + (i >> 2)) * 256 + 32 * (g & 1) + 8 * (i & 3);
#pragma unroll
    for (int db = 0; db < 4; ++db) vo[db] = l0 + 64 * (db ^ (i >> 2));
  }

  const float cs = a.scale_log2, kthr = kRescale / cs;
  f32x16 o[4];
#pragma unroll
  for (int db = 0; db < 4; ++db)
#pragma unroll
    for (int i = 0; i < 16; ++i) o[db][i] = 0.f;
  float m = -1e30f, l = 0.f;  // reference max (raw scores), lane-partial row sum

  for (int n = 0; n < n_it; ++n) {
    landed_barrier();
    if (n + 1 < n_it) issue(n + 1);
    const int j = n * kSlices + sl;
    if (j >= nsub) continue;  // the last iteration's slices past the end
    const lds_u8* kb = (const lds_u8*)lds + (n & 1) * kStageBytes + sl * 2 * kSubBytes;
    const lds_u8* vb = kb + kSubBytes;
    f32x16 s;
#pragma unroll
    for (int i = 0; i < 16; ++i) s[i] = 0.f;
#pragma unroll
    for (int t = 0; t < 8; ++t) {
      const u32x4 kf = *reinterpret_cast<const __attribute__((address_space(3))) u32x4*>(kb + koff[t]);
      s = M::run(kf, qf[t], s);
    }
    if (32 * j + 32 > full) {
      const int lim = my_lim - 32 * j - 4 * hl;
#pragma unroll
      for (int i = 0; i < 16; ++i) s[i] = 8 * (i >> 2) + (i & 3) < lim ? s[i] : -INFINITY;
    }
    float mx = vmax3(s[0], s[1], s[2]);
#pragma unroll
    for (int i = 3; i < 15; i += 2) mx = vmax3(mx, s[i], s[i + 1]);
    mx = vmax(mx, s[15]);
    if (__ballot(mx > m + kthr)) {  // any lane: rescale (rare after the first sub-tile)
      const auto sw = __builtin_amdgcn_permlane32_swap(__float_as_uint(mx), __float_as_uint(mx), false, false);
      mx = vmax(__uint_as_float(sw[0]), __uint_as_float(sw[1]));
      const float mn = vmax(m, mx), alpha = fast_exp2((m - mn) * cs);
      m = mn;
      l *= alpha;
#pragma unroll
      for (int db = 0; db < 4; ++db)
#pragma unroll
        for (int i = 0; i < 16; ++i) o[db][i] *= alpha;
    }
    const float nb = -m * cs;
    u32 pw[8];
#pragma unroll
    for (int w = 0; w < 8; ++w) {
      pw[w] = M::pack(fast_exp2(fmaf(s[2 * w], cs, nb)), fast_exp2(fmaf(s[2 * w + 1], cs, nb)));
      l = M::dot2_ones(pw[w], l);
    }
#pragma unroll
    for (int tt = 0; tt < 2; ++tt) {
      const u32x4 p = {pw[4 * tt], pw[4 * tt + 1], pw[4 * tt + 2], pw[4 * tt + 3]};
#pragma unroll
      for (int db = 0; db < 4; ++db) {
        const v4s lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4s*)(vb + vo[db] + 4096 * tt));
        const v4s hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4s*)(vb + vo[db] + 4096 * tt + 2048));
        const u32x2 a0 = __builtin_bit_cast(u32x2, lo), a1 = __builtin_bit_cast(u32x2, hi);
        o[db] = M::run(u32x4{a0[0], a0[1], a1[0], a1[1]}, p, o[db]);
      }
    }
  }

  // KV-cache store: the item's own 32 rows taken as keys (one pair per KV
  // head), loaded here and written after the output
  u32x4 ok[2];
  int64_t oslot = -1;
  const int orow = tid >> 4, och = (tid & 15) * 8;  // 32 rows x 16 chunks
  if constexpr (STORE) {
    const int64_t tok = (int64_t)k_beg + q0 + orow;
    if (pr == 0 && q0 + orow < Lq && tok < a.n_tok) {
      oslot = a.slots[tok];
      ok[0] = *reinterpret_cast<const u32x4*>(a.k + tok * a.k_stride + h * D + och);
      ok[1] = *reinterpret_cast<const u32x4*>(a.v + tok * a.v_stride + h * D + och);
    }
  }

  // merge the four slices of each head: partial O over the (dead) stages,
  // [wave][16 float4][64 lanes]; then wave (c, s) sums dims 32 s .. + 31
  {
    const auto sw = __builtin_amdgcn_permlane32_swap(__float_as_uint(l), __float_as_uint(l), false, false);
    l = __uint_as_float(sw[0]) + __uint_as_float(sw[1]);
  }
  __syncthreads();
  float2* ml = reinterpret_cast<float2*>(lds + kMlOff);
  if (lane < 32) ml[wave * 32 + col] = make_float2(m, l);
  f32x4* part = reinterpret_cast<f32x4*>(lds + wave * 16384);
#pragma unroll
  for (int db = 0; db < 4; ++db)
#pragma unroll
    for (int r = 0; r < 4; ++r)
      part[(4 * db + r) * 64 + lane] = f32x4{o[db][4 * r], o[db][4 * r + 1], o[db][4 * r + 2], o[db][4 * r + 3]};
  __syncthreads();
  float2 mls[kSlices];
  float mx = -1e30f;
#pragma unroll
  for (int k = 0; k < kSlices; ++k) {
    mls[k] = ml[(2 * k + c) * 32 + col];
    mx = vmax(mx, mls[k].x);
  }
  float wt[kSlices], lt = 0.f;
#pragma unroll
  for (int k = 0; k < kSlices; ++k) {
    wt[k] = fast_exp2((mls[k].x - mx) * cs);
    lt = fmaf(mls[k].y, wt[k], lt);
  }
  const float inv = lt > 0.f ? __builtin_amdgcn_rcpf(lt) : 0.f;
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    f32x4 v = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int k = 0; k < kSlices; ++k) {
      const f32x4 x = *reinterpret_cast<const f32x4*>(lds + (2 * k + c) * 16384 + ((4 * sl + r) * 64 + lane) * 16);
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = fmaf(x[e], wt[k], v[e]);
    }
    u32x2 w;
    w[0] = M::pack(v[0] * inv, v[1] * inv);
    w[1] = M::pack(v[2] * inv, v[3] * inv);
    *reinterpret_cast<u32x2*>(lds + kOutOff + (c * 32 + col) * kOutPitch + (32 * sl + 8 * r + 4 * hl) * 2) = w;
  }
  __syncthreads();
  if (q0 + orow < Lq) {
#pragma unroll
    for (int k = 0; k < 2; ++k)
      *reinterpret_cast<u32x4*>(a.out + (int64_t)(q_beg + q0 + orow) * a.o_stride + (head + k) * D + och) =
          *reinterpret_cast<const u32x4*>(lds + kOutOff + (k * 32 + orow) * kOutPitch + och * 2);
  }
  if constexpr (STORE) {
    if (oslot >= 0 && oslot < a.num_rows) {
      const int64_t dst = (oslot * a.hkv + h) * D + och;
      *reinterpret_cast<u32x4*>(a.kc + dst) = ok[0];
      *reinterpret_cast<u32x4*>(a.vc + dst) = ok[1];
    }
    // q-blocks of the segment that no item owns (max_seqlen below its length)
    if (z == 0 && pr == 0 && nqb > a.n_qblocks)
      pf::store_kv_span<kThreads>(a, tid, k_beg, k_beg + (int64_t)(nqb - a.n_qblocks) * 32, h, h + 1);
  }
}

template <bool CAUSAL, bool STORE, bool F16>
static void launch_t(const Args& a, unsigned grid, hipStream_t st) {
  hipLaunchKernelGGL((prefill_split_kernel<CAUSAL, STORE, F16>), dim3(grid), dim3(kThreads), 0, st, a);
}

}  // namespace ps

// Up to one item per CU the call runs here; up to two per CU from 512 keys on.
// Measured (us, the other kernel -> this one; causal, graph replay): 16/8 heads,
// one request of 128 tokens 11.5 -> 6.8, 777 23.3 -> 12.3 (with the store 24.8 ->
// 13.3), 1024 28.6 -> 15.0, 2048 (512 items) 48.9 -> 31.3; 8 x 128 (256 items)
// 12.0 -> 7.4; two items per CU: 4 x 512 18.8 -> 17.0 but 8 x 256 13.6 -> 14.7 and
// 32 x 64 10.1 -> 13.1; four per CU: 1 x 4096 93 -> 97, 2 x 2048 54 -> 61, 8 x 512
// 20 -> 33 (the wide kernel's tiles serve four times the queries).  32/8 and 8/4
// heads lie alike at equal item counts.
bool prefill_split_takes(int g, float scale, int n_seqs, int hkv, int max_q, int max_k, int n_cu) {
  if ((g != 2 && g != 4 && g != 8) || !(scale > 0.f)) return false;
  const int64_t items = (int64_t)n_seqs * hkv * (g / 2) * cdiv(max_q, 32);
  return items <= n_cu || (items <= 2 * (int64_t)n_cu && max_k >= 512);
}

int prefill_split_launch(const pf::Args& a0, int g, bool causal, bool store, bool f16, int max_q, hipStream_t st) {
  if (store && !causal) return AAC_ERR_UNSUPPORTED;
  pf::Args a = a0;
  a.n_qblocks = (int)cdiv(max_q, 32);
  const unsigned grid = (unsigned)((int64_t)a.n_seqs * a.hkv * (g / 2) * a.n_qblocks);
  if (store) {
    if (f16) ps::launch_t<true, true, true>(a, grid, st); else ps::launch_t<true, true, false>(a, grid, st);
  } else if (causal) {
    if (f16) ps::launch_t<true, false, true>(a, grid, st); else ps::launch_t<true, false, false>(a, grid, st);
  } else {
    if (f16) ps::launch_t<false, false, true>(a, grid, st); else ps::launch_t<false, false, false>(a, grid, st);
  }
  return AAC_OK;
}

}  // namespace aac
