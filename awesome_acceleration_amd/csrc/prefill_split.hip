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
// workgroup's waves: with SL slices, wave (c, s) takes head c and the 32-key
// sub-tiles s, s + SL, s + 2 SL, ...  The partial results of a head (reference
// max, row sum, O) are merged through LDS at the end.  Two forms:
//   SL = 4: eight waves, two LDS stages of 128 keys, one workgroup per CU: the
//     shortest chain, for fewer items than CUs.  Two waves per SIMD run the two
//     heads of a slice, one's softmax beside the other's MFMAs.
//   SL = 2: four waves, one stage of 64 keys, three workgroups per CU: one's
//     loads, merge and stores run beside the others' products.  For short
//     segments and a few items per CU.
//
// Tiles go straight from global memory into LDS; wave (0, s) brings slice s's
// K rows, wave (1, s) its V rows.  With two stages there is one barrier per
// iteration: past it every wave's tile has landed and the other stage is free
// for the next loads.  Row layouts, fragments, masks, lazy rescaling and the
// probability rounding are those of prefill_wide.hip.

#include <algorithm>

#include "prefill_common.h"
#include "prefill_split.h"

namespace aac {
namespace ps {

using pf::Args;
using pf::D;
using pf::kRescale;

constexpr int kSubBytes = 32 * D * 2;   // 8 KiB: a sub-tile of K or V
constexpr int kOutPitch = D * 2 + 16;   // bytes of an output staging row

// SL key slices (32 keys each per iteration) on 2 SL waves, STAGES LDS stages.
template <int SL, int STAGES> struct Shape {
  static constexpr int kWaves = 2 * SL, kThreads = 64 * kWaves;
  static constexpr int kStageBytes = SL * 2 * kSubBytes;
  // partial O of the merge, over the dead stages: 4 KiB per 32 dims that a wave
  // hands to another slice's
  static constexpr int kPartBytes = kWaves * (SL == 4 ? 4 : 2) * 4096;
  static constexpr int kTiles = STAGES * kStageBytes > kPartBytes ? STAGES * kStageBytes : kPartBytes;
  static constexpr int kOutOff = kTiles;  // [2 heads][32 queries]
  static constexpr int kMlOff = kOutOff + 2 * 32 * kOutPitch;
  static constexpr int kLdsBytes = kMlOff + kWaves * 32 * 8;
};

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

template <int SL, int STAGES, bool CAUSAL, bool STORE, bool F16>
__global__ __launch_bounds__(128 * SL, SL == 4 ? 2 : 3) void prefill_split_kernel(Args a) {
  static_assert(CAUSAL || !STORE, "the store variant is causal self-attention");
  static_assert((SL == 4 && STAGES == 2) || (SL == 2 && STAGES == 1), "the two forms");
  typedef pf::Mfma<F16> M;
  typedef Shape<SL, STAGES> S;
  constexpr int kThreads = S::kThreads, kSlices = SL, kStageBytes = S::kStageBytes;
  constexpr int kOutOff = S::kOutOff, kMlOff = S::kMlOff;
  __shared__ __attribute__((aligned(1024))) unsigned char lds[S::kLdsBytes];
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
      load_lds16(rs, voff[i & 3], (key0 + 4 * i) * row_bytes, dst0 + (u32)(n % STAGES * kStageBytes + i * 1024));
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
    if constexpr (STAGES == 1) {
      if (n > 0) {
        __syncthreads();  // every wave is done with the tile before
        issue(n);
      }
      landed_barrier();
    } else {
      landed_barrier();
      if (n + 1 < n_it) issue(n + 1);
    }
    const int j = n * kSlices + sl;
    if (j >= nsub) continue;  // the last iteration's slices past the end
    const lds_u8* kb = (const lds_u8*)lds + n % STAGES * kStageBytes + sl * 2 * kSubBytes;
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
  // head), loaded here and written after the output: 16 threads a row
  constexpr int kRows = kThreads / 16, kPass = 32 / kRows;
  u32x4 ok[kPass], ov[kPass];
  int64_t oslot[kPass];
  const int orow = tid >> 4, och = (tid & 15) * 8;
  if constexpr (STORE) {
#pragma unroll
    for (int i = 0; i < kPass; ++i) {
      const int row = q0 + orow + i * kRows;
      const int64_t tok = (int64_t)k_beg + row;
      oslot[i] = -1;
      if (pr == 0 && row < Lq && tok < a.n_tok) {
        oslot[i] = a.slots[tok];
        ok[i] = *reinterpret_cast<const u32x4*>(a.k + tok * a.k_stride + h * D + och);
        ov[i] = *reinterpret_cast<const u32x4*>(a.v + tok * a.v_stride + h * D + och);
      }
    }
  }

  // Merge the slices of each head: slice s takes dims 128 s / SL and up, its own
  // part from registers, the others' through LDS (over the dead stages).
  {
    const auto sw = __builtin_amdgcn_permlane32_swap(__float_as_uint(l), __float_as_uint(l), false, false);
    l = __uint_as_float(sw[0]) + __uint_as_float(sw[1]);
  }
  auto part = [&](int w, int db) {  // 4 KiB of wave w's dims 32 db .. + 31: [4][64 lanes]
    return reinterpret_cast<f32x4*>(lds + (SL == 4 ? 4 * w + db : 2 * w + (db & 1)) * 4096);
  };
  __syncthreads();
  float2* ml = reinterpret_cast<float2*>(lds + kMlOff);
  if (lane < 32) ml[wave * 32 + col] = make_float2(m, l);
#pragma unroll
  for (int db = 0; db < 4; ++db)
    if (db * SL / 4 != sl) {
#pragma unroll
      for (int r = 0; r < 4; ++r)
        part(wave, db)[r * 64 + lane] = f32x4{o[db][4 * r], o[db][4 * r + 1], o[db][4 * r + 2], o[db][4 * r + 3]};
    }
  __syncthreads();
  float2 mls[SL];
  float mx = -1e30f;
#pragma unroll
  for (int k = 0; k < SL; ++k) {
    mls[k] = ml[(2 * k + c) * 32 + col];
    mx = vmax(mx, mls[k].x);
  }
  float wt[SL], lt = 0.f;
#pragma unroll
  for (int k = 0; k < SL; ++k) {
    wt[k] = fast_exp2((mls[k].x - mx) * cs);
    lt = fmaf(mls[k].y, wt[k], lt);
  }
  const float inv = lt > 0.f ? __builtin_amdgcn_rcpf(lt) : 0.f;
#pragma unroll
  for (int db = 0; db < 4; ++db)
    if (db * SL / 4 == sl) {
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        float v[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int k = 0; k < SL; ++k) {  // in slice order
          if (k == db * SL / 4) {
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] = fmaf(o[db][4 * r + e], wt[k], v[e]);
          } else {
            const f32x4 x = part(2 * k + c, db)[r * 64 + lane];
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] = fmaf(x[e], wt[k], v[e]);
          }
        }
        u32x2 w;
        w[0] = M::pack(v[0] * inv, v[1] * inv);
        w[1] = M::pack(v[2] * inv, v[3] * inv);
        *reinterpret_cast<u32x2*>(lds + kOutOff + (c * 32 + col) * kOutPitch + (32 * db + 8 * r + 4 * hl) * 2) = w;
      }
    }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < kPass; ++i) {
    const int row = orow + i * kRows;
    if (q0 + row < Lq) {
#pragma unroll
      for (int k = 0; k < 2; ++k)
        *reinterpret_cast<u32x4*>(a.out + (int64_t)(q_beg + q0 + row) * a.o_stride + (head + k) * D + och) =
            *reinterpret_cast<const u32x4*>(lds + kOutOff + (k * 32 + row) * kOutPitch + och * 2);
    }
  }
  if constexpr (STORE) {
#pragma unroll
    for (int i = 0; i < kPass; ++i)
      if (oslot[i] >= 0 && oslot[i] < a.num_rows) {
        const int64_t dst = (oslot[i] * a.hkv + h) * D + och;
        *reinterpret_cast<u32x4*>(a.kc + dst) = ok[i];
        *reinterpret_cast<u32x4*>(a.vc + dst) = ov[i];
      }
    // q-blocks of the segment that no item owns (max_seqlen below its length)
    if (z == 0 && pr == 0 && nqb > a.n_qblocks)
      pf::store_kv_span<kThreads>(a, tid, k_beg, k_beg + (int64_t)(nqb - a.n_qblocks) * 32, h, h + 1);
  }
}

template <bool CAUSAL, bool STORE, bool F16>
static void launch_t(const Args& a, bool four, unsigned grid, hipStream_t st) {
  if (four)
    hipLaunchKernelGGL((prefill_split_kernel<4, 2, CAUSAL, STORE, F16>), dim3(grid), dim3(Shape<4, 2>::kThreads), 0, st, a);
  else
    hipLaunchKernelGGL((prefill_split_kernel<2, 1, CAUSAL, STORE, F16>), dim3(grid), dim3(Shape<2, 1>::kThreads), 0, st, a);
}

}  // namespace ps

// Where the lines lie, by items (32 queries of two heads) per CU.  Measured on
// MI355X (graph replay, us): W the wide kernel, P the eight-wave kernel's two pieces
// per item, 4 and 2 the slices here; over 1,794 shapes of 16-2048 queries, up to
// 32,768 keys and groups 2, 4 and 8 the choice is at most 5% behind W or P.
//
// Causal, with keys for the queries alone or half as many more:
//   up to one item: 16/8 heads, 1 x 128 W 11.5, 4 6.4, 2 5.7; 1 x 256 12.9, 7.5,
//     7.5; 1 x 777 23.3, 12.1, 15.1 (with the store 24.8, 12.9); 1 x 1024 28.6,
//     14.5, 18.9: four slices for more than 256 keys
//   up to two: 4 x 512 W 18.9, 4 16.6, 2 13.1; 1 x 2048 48.7, 29.2, 33.6; 8/4 heads
//     3 x 1024 28.4, 17.9, 19.3: four from 640 keys on
//   up to three: 6 x 512 W 19.0, 2 15.9; 1 x 3072 69.1, 57.0; 12 x 250 13.1, 11.8
//   up to four: 1 x 4096 W 93.1, 2 84.7; 2 x 2048 50.7, 47.8, but 16 x 256 15.2,
//     18.0: from 1024 keys on; where there are more keys than queries from 3072 on
//     (4 x 1024 queries, 1536 keys W 44.3, 2 50.5).  Beyond, the wide kernel, whose
//     tiles serve four times the queries (8 x 1024 46.4, 55.9)
//   segments of one block of 32 queries keep one of its four waves busy: 256 x 32
//     at 16/8 heads W 50.3, 2 21.6, at 32/8 55.5, 33.4; of two blocks 57.0, 40.8,
//     but at 32/8 67.7, 82.0
//
// Every item sees all or most of its keys (not causal, or many more keys than
// queries).  Each item here reads them for itself, where W reads them once for 128
// queries, and the longer they are the more of the time that is:
//   up to one item: 16/8 heads, 8 x 128 queries, 2048 keys P 47.2, 4 30.8, 2 44.7;
//     1 x 512, 8192 keys 133.8, 89.6, 145.6.  But when the keys and values pass
//     the 256 MiB last-level cache the call is bound by drawing them, and P draws
//     with twice the CUs where it finds them idle: 16 x 32, 8192 keys P 127, 4 164;
//     8 x 64, 16,384 keys 200, 273
//   up to two: 16 x 128, 512 keys W 21.8, 2 18.6; 64 x 32, 512 keys 34.9, 26.8; 16 x
//     128, 2048 keys P 57.6, 2 50.7, but 32/8 32 x 32, 2048 keys W 55.7, 2 63.8
//   up to three: 24 x 128, 160 keys W 13.8, 2 13.4; 24 x 64, 1024 keys 39, 42.  From
//     3072 keys on P has more pieces than CUs: 12 x 256, 4096 keys P 160, 2 119
//   beyond: 64 x 64, 4096 keys W 234, 2 409; 32 x 128, 2048 keys 72, 159; one block of
//     queries, 256 x 32, 512 keys 134, 125, at 32/8 144, 156; 64 x 16, 256 keys at
//     32/8 26.5, 21.6
static int pick_slices(int g, int n_seqs, int hkv, int max_q, int max_k, bool causal, int n_cu, bool idle_pieces) {
  const int64_t cu = n_cu, items = (int64_t)n_seqs * hkv * (g / 2) * cdiv(max_q, 32);
  if (causal && 2 * (int64_t)max_k <= 3 * (int64_t)max_q) {
    if ((items <= cu && max_k > 256) || (items <= 2 * cu && max_k >= 640)) return 4;
    if (items <= 3 * cu || (items <= 4 * cu && max_k >= (max_k <= max_q ? 1024 : 3072))) return 2;
    if (max_k <= max_q) return max_q <= 32 || (max_q <= 64 && g == 2) ? 2 : 0;
  } else if (items <= cu) {
    if (max_k <= 256) return 2;
    return idle_pieces && (int64_t)n_seqs * hkv * max_k * (2 * pf::D * 2) > (int64_t(256) << 20) ? 0 : 4;
  } else if (items <= 2 * cu) {
    return max_k <= 1024 || (max_k <= 2048 && max_q > 32) ? 2 : 0;
  } else if (items <= 3 * cu) {
    return max_k <= 512 || max_k >= 3072 ? 2 : 0;
  }
  if (max_q <= 32) return max_k <= (g == 2 ? 512 : g == 4 ? 256 : max_q <= 16 || items <= 8 * cu ? 64 : 0) ? 2 : 0;
  return g == 2 && max_q <= 64 && max_k <= 128 ? 2 : 0;
}

int prefill_split_slices(int g, float scale, bool f16, int n_seqs, int hkv, int max_q, int max_k, bool causal,
                         int n_cu, bool idle_pieces) {
  if ((g != 2 && g != 4 && g != 8) || !(scale > 0.f)) return 0;
  const int slices = pick_slices(g, n_seqs, hkv, max_q, max_k, causal, n_cu, idle_pieces);
  // fp16 calls of more items would run on the eight-wave kernel (see
  // prefill_wide_takes), which loses less on short items than the wide one: two
  // slices only where they beat it as well (eight-wave / two: 64 x 64 queries at 16/8
  // heads 12.9 / 16.4, 24 x 128, not causal 11.7 / 13.0, 64 x 32, 40 keys at 32/8 12.9
  // / 16.9; 256 x 32 at 16/8 32 / 21, 6 x 512 21.5 / 21.4, 3 x 1129 36 / 27)
  const int64_t cu = n_cu, items = (int64_t)n_seqs * hkv * (g / 2) * cdiv(max_q, 32);
  if (!f16 || slices != 2 || 2 * items <= 3 * cu) return slices;
  const bool keep = g == 2 && max_q <= 32 ? true
                    : items <= 2 * cu     ? max_q > 64
                    : items <= 3 * cu     ? max_k > 256
                                          : items <= 4 * cu && max_k >= 1024;
  return keep ? 2 : 0;
}

int prefill_split_launch(const pf::Args& a0, int slices, int g, bool causal, bool store, bool f16, int max_q,
                         hipStream_t st) {
  if (store && !causal) return AAC_ERR_UNSUPPORTED;
  pf::Args a = a0;
  a.n_qblocks = (int)cdiv(max_q, 32);
  const unsigned grid = (unsigned)((int64_t)a.n_seqs * a.hkv * (g / 2) * a.n_qblocks);
  const bool four = slices == 4;
  if (store) {
    if (f16) ps::launch_t<true, true, true>(a, four, grid, st); else ps::launch_t<true, true, false>(a, four, grid, st);
  } else if (causal) {
    if (f16) ps::launch_t<true, false, true>(a, four, grid, st); else ps::launch_t<true, false, false>(a, four, grid, st);
  } else {
    if (f16) ps::launch_t<false, false, true>(a, four, grid, st); else ps::launch_t<false, false, false>(a, four, grid, st);
  }
  return AAC_OK;
}

}  // namespace aac
