// Projections of a decode step of few sequences (gfx950, bf16/fp16 MFMA):
// Y = X W^T for X [m, k], m <= 32, and a torch Linear weight W [n, k]
// (model/model.py:132-154, :178-188, :258), optionally with the residual add
// and RMSNorm before it (model/model.py:47-52, :259, :265) in the prologue and
// SiLU * up (model/model.py:188) in the epilogue.
//
// What bounds it: with a few rows the product is the time to stream W once,
// 1-2 us at the HBM rate, and a launch costs more than that, so the number of
// CUs that pull on W and the chain of latencies inside a launch are what
// counts.  The tiles of gemm.hip leave a 1024-column projection on 16-32 of
// 256 CUs.  Here a workgroup owns 8 or 16 output columns and all of K; its
// eight waves split K.
//
// Each wave stages exactly the W (and X) columns that it multiplies, in units
// of 64 columns, straight into its own part of LDS (global_load_lds_dwordx4:
// one instruction fills 8 rows x 128 bytes, whole cache lines; loaded into
// the MFMA register layout instead, an instruction touches 16 rows x 64 bytes
// and a CU drew W at about half the rate).  Nothing is shared between waves,
// so there is no barrier before the end: as many units as fit LDS are in
// flight from the start and a wave waits only for its own.  A unit's rows are
// stored with their 16-byte chunks XOR-swizzled by the row (chunk c of row r
// at c ^ ((r >> 1) & 7)), so that 16 rows' fragment reads cover all banks.
//
// v_mfma_f32_16x16x32: A = 16 W rows x 32 k (lane l: row l % 16, k 8 (l / 16)
// .. + 7), B = 32 k x 16 X rows (the same layout); a lane ends with one token
// (l % 16) and four consecutive output columns 4 (l / 16) .. + 3.  With 8
// columns or 8 tokens the upper half of the operand repeats the lower.  The
// eight partial tiles are summed through LDS in wave order.
//
// The norm: the rows of X are normalised by one wave each, in the order of
// the RMSNorm kernel of fused.hip (so the result is the same bit for bit),
// while the W loads are in flight, and shared through LDS.  Every workgroup
// normalises all rows again (m x 2 KB from L2 at hidden 1024), which costs
// less than the launch it saves as long as a wave has a few rows at most.  The
// workgroup of column tile 0 writes the new residual.  Loads return in order, so
// with at most one row per wave (m <= 8) the row, its residual and the norm weight
// are staged through LDS before W and normalised while W is on its way: loaded
// into registers after W they were waited for together with all of it.  QKV 4.7
// -> 3.9 us and gate/up 6.3 -> 5.3 at 4 rows (trace), a 28-layer step 870 -> 826.

#include "gemm_small.h"
#include "qk_head.h"

namespace aac {
namespace gs {

template <bool F16> struct Mma;
template <> struct Mma<false> {
  static constexpr Dt DT = Dt::BF16;
  __device__ static inline f32x4 run(const u32x4& a, const u32x4& b, const f32x4& c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a),
                                                    __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
  }
};
template <> struct Mma<true> {
  static constexpr Dt DT = Dt::FP16;
  __device__ static inline f32x4 run(const u32x4& a, const u32x4& b, const f32x4& c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a),
                                                   __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
  }
};

constexpr int KS = 8;                  // waves; each owns k / 8 columns of K
constexpr int kUnitK = 64;             // columns of K per unit
constexpr int kBlock = 1024;           // bytes of one staged block: 8 rows x 128
constexpr int kLdsMax = 160 * 1024;

// 8 rows x 128 bytes from global memory straight into LDS at dst + 16 lane.
// Inline assembly: the compiler neither counts the load nor guards LDS reads
// with waits for it; the waits are explicit.  The LDS reads that may still be
// on their way from the same place are waited for first.  M0 is used by
// nothing else here.
typedef __attribute__((address_space(3))) unsigned char lds_u8;
__device__ __forceinline__ void stage8(const u16* src, u32 dst) {
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off"
               :
               : "v"(src), "s"(dst)
               : "memory", "m0");
#pragma clang diagnostic pop
}

template <int N> __device__ __forceinline__ void wait_vm() {
  static_assert(N < 64, "vmcnt is six bits");
  asm volatile("s_waitcnt vmcnt(%0)" : : "n"(N) : "memory");
}

// LDS exchange between waves; loads from global memory stay in flight.
__device__ __forceinline__ void lds_barrier() {
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

// WR: W rows (output columns) per workgroup, 8 or 16 (twice that with SILU).
// XR: X rows per workgroup, 8, 16 or 32.  NORMK: 0, or the depth k of a call
// with the norm.
// Units in flight per wave at most: MAXU.
template <int WR, int XR, bool SILU, bool F16, int NORMK, bool RESID, int MAXU>
__global__ __launch_bounds__(64 * KS) void small_kernel(Args a) {
  typedef Mma<F16> M;
  constexpr Dt DT = M::DT;
  typedef fz::Cvt<DT> C;
  constexpr bool NORM = NORMK > 0;
  constexpr int NB = SILU ? 2 : 1;                 // W row groups (gate, up)
  constexpr int MT = XR > 16 ? XR / 16 : 1;        // 16-token MFMA tiles
  constexpr int WBLK = WR / 8 * NB, XBLK = NORM ? 0 : XR / 8;
  constexpr int IPU = WBLK + XBLK;                 // staged blocks (loads) per unit
  constexpr int XPITCH = NORMK * 2 + 16;           // bytes of a normalised row
  // with at most one row to normalise per wave its x, residual and norm weight
  // are staged too, before W
  constexpr int NC = NORMK / 512;
  constexpr bool STAGED = NORM && XR == KS;
  constexpr int kIn = STAGED ? NC * (RESID ? 3 : 2) * kBlock : 0;
  constexpr int kXn = (NORM ? XR * XPITCH : 0) + KS * kIn;
  constexpr int kFit = (kLdsMax - kXn) / (KS * IPU * kBlock);
  constexpr int kWant = NORM ? NORMK / (KS * kUnitK) : MAXU;
  constexpr int NBUF = kFit < kWant ? kFit : kWant;  // units in flight per wave
  constexpr int kStage = NBUF * IPU * kBlock, kPart = NB * MT * 1024;
  constexpr int kWave = kStage > kPart ? kStage : kPart;  // a wave's own LDS
  static_assert(NBUF >= 2 || (NORM && NBUF == kWant), "two units, or all of them, in flight");
  static_assert(!STAGED || NBUF == kWant, "all of W in flight behind the staged row");
  __shared__ __attribute__((aligned(1024))) unsigned char lds[KS * kWave + kXn];

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int col = lane & 15, kg = lane >> 4;

  const int n_mt = (a.m + XR - 1) / XR;
  // the row tiles of one column tile on one XCD, as in gemm.hip: W comes from
  // HBM once
  const int T = n_mt * a.n_tiles;
  int t = blockIdx.x;
  if ((T & 7) == 0) t = (t & 7) * (T >> 3) + (t >> 3);
  const int m0 = (t % n_mt) * XR, nt = t / n_mt, n0 = nt * WR;

  const int units = a.k / (KS * kUnitK);
  const int kbeg = wave * units * kUnitK;
  // staging: block j holds rows 8 j + lane / 8, this lane's chunk swizzled
  const int r8 = lane >> 3;
  const u16* src[IPU];
#pragma unroll
  for (int j = 0; j < IPU; ++j) {
    if (j < WBLK) {
      const int nb = j / (WR / 8), row = 8 * (j % (WR / 8)) + r8;
      src[j] = a.w + (int64_t)(nb * a.silu_off + n0 + row) * a.w_stride + kbeg + 8 * ((lane & 7) ^ ((row >> 1) & 7));
    } else {
      const int row = 8 * (j - WBLK) + r8;
      src[j] = a.x + (int64_t)min(m0 + row, a.m - 1) * a.x_stride + kbeg + 8 * ((lane & 7) ^ ((row >> 1) & 7));
    }
  }
  const u32 lds0 = (u32)(uintptr_t)(lds_u8*)lds + (u32)(wave * kWave);
  auto issue = [&](int u, int buf) {
#pragma unroll
    for (int j = 0; j < IPU; ++j) stage8(src[j] + u * kUnitK, lds0 + (u32)((buf * IPU + j) * kBlock));
  };
  const int first = units < NBUF ? units : NBUF;
  constexpr int kInOff = KS * kWave + (NORM ? XR * XPITCH + 15 : 0) / 16 * 16;
  if constexpr (STAGED) {
    const int row = m0 + wave;
    if (row < a.m) {  // wave-uniform
      const u32 in = (u32)(uintptr_t)(lds_u8*)lds + (u32)(kInOff + wave * kIn);
#pragma unroll
      for (int c = 0; c < NC; ++c) {
        stage8(a.x + (int64_t)row * a.x_stride + c * 512 + lane * 8, in + (u32)(c * kBlock));
        stage8(a.norm_w + c * 512 + lane * 8, in + (u32)((NC + c) * kBlock));
        if constexpr (RESID)
          stage8(a.res + (int64_t)row * NORMK + c * 512 + lane * 8, in + (u32)((2 * NC + c) * kBlock));
      }
    }
  }
  for (int u = 0; u < first; ++u) issue(u, u);

  if constexpr (NORM) {
    // row `wave`, `wave` + 8, ...: one wavefront per row, 8 consecutive
    // elements per lane and 512-element chunk
    constexpr int RW = XR / KS;
    u32x4 xr[RW][NC], rr[RESID ? RW : 1][NC], nw[NC];
    if constexpr (STAGED) {
      // the depth is NORMK, so W's loads behind these are known
      wait_vm<kWant * IPU>();
      const unsigned char* in = lds + kInOff + wave * kIn + lane * 16;
#pragma unroll
      for (int c = 0; c < NC; ++c) {
        xr[0][c] = *reinterpret_cast<const u32x4*>(in + c * kBlock);
        nw[c] = *reinterpret_cast<const u32x4*>(in + (NC + c) * kBlock);
        if constexpr (RESID) rr[0][c] = *reinterpret_cast<const u32x4*>(in + (2 * NC + c) * kBlock);
      }
    } else {
#pragma unroll
      for (int i = 0; i < RW; ++i) {
        const int row = m0 + wave + KS * i;
        if (row < a.m) {  // wave-uniform
#pragma unroll
          for (int c = 0; c < NC; ++c) {
            xr[i][c] = *reinterpret_cast<const u32x4*>(a.x + (int64_t)row * a.x_stride + c * 512 + lane * 8);
            if constexpr (RESID)
              rr[i][c] = *reinterpret_cast<const u32x4*>(a.res + (int64_t)row * NORMK + c * 512 + lane * 8);
          }
        }
      }
#pragma unroll
      for (int c = 0; c < NC; ++c) nw[c] = *reinterpret_cast<const u32x4*>(a.norm_w + c * 512 + lane * 8);
    }
#pragma unroll
    for (int i = 0; i < RW; ++i) {
      const int row = m0 + wave + KS * i;
      if (row < a.m) {
        float v[NC][8], ss = 0.f;
#pragma unroll
        for (int c = 0; c < NC; ++c) {
          fz::unpack8<DT>(xr[i][c], v[c]);
          if constexpr (RESID) {
            float r[8];
            fz::unpack8<DT>(rr[i][c], r);
#pragma unroll
            for (int e = 0; e < 8; ++e) v[c][e] = C::round(v[c][e] + r[e]);
            if (nt == 0)
              *reinterpret_cast<u32x4*>(a.res_out + (int64_t)row * NORMK + c * 512 + lane * 8) =
                  fz::pack8<DT>(v[c]);
          }
#pragma unroll
          for (int e = 0; e < 8; ++e) ss = fmaf(v[c][e], v[c][e], ss);
        }
        ss = fz::wave_sum(ss);
        const float rs = __frsqrt_rn(ss / (float)NORMK + a.eps);
#pragma unroll
        for (int c = 0; c < NC; ++c) {
          float w[8], o[8];
          fz::unpack8<DT>(nw[c], w);
#pragma unroll
          for (int e = 0; e < 8; ++e) o[e] = w[e] * C::round(v[c][e] * rs);
          *reinterpret_cast<u32x4*>(lds + KS * kWave + (wave + KS * i) * XPITCH + c * 1024 + lane * 16) =
              fz::pack8<DT>(o);
        }
      }
    }
    lds_barrier();
  }

  f32x4 acc[NB][MT];
#pragma unroll
  for (int nb = 0; nb < NB; ++nb)
#pragma unroll
    for (int i = 0; i < MT; ++i) acc[nb][i] = f32x4{0.f, 0.f, 0.f, 0.f};

  const unsigned char* mine = lds + wave * kWave;
  const int wrow = col & (WR - 1), xrow = XR < 16 ? col & (XR - 1) : col;
  auto multiply = [&](int u, int buf) {
    const unsigned char* b = mine + buf * (IPU * kBlock);
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      const int c = 4 * s + kg;  // 16-byte chunk of the unit
      u32x4 w[NB], x[MT];
#pragma unroll
      for (int nb = 0; nb < NB; ++nb)
        w[nb] = *reinterpret_cast<const u32x4*>(b + nb * (WR / 8) * kBlock + wrow * 128 + 16 * (c ^ ((wrow >> 1) & 7)));
#pragma unroll
      for (int i = 0; i < MT; ++i) {
        if constexpr (NORM)
          x[i] = *reinterpret_cast<const u32x4*>(lds + KS * kWave + (16 * i + xrow) * XPITCH +
                                                  (kbeg + u * kUnitK) * 2 + 16 * c);
        else
          x[i] = *reinterpret_cast<const u32x4*>(b + WBLK * kBlock + (16 * i + xrow) * 128 +
                                                  16 * (c ^ ((xrow >> 1) & 7)));
      }
#pragma unroll
      for (int nb = 0; nb < NB; ++nb)
#pragma unroll
        for (int i = 0; i < MT; ++i) acc[nb][i] = M::run(w[nb], x[i], acc[nb][i]);
    }
  };
  int u = 0, buf = 0;
  for (; u + NBUF < units; ++u) {  // refill the buffer just read
    wait_vm<(NBUF - 1) * IPU>();
    multiply(u, buf);
    issue(u + NBUF, buf);
    buf = buf + 1 == NBUF ? 0 : buf + 1;
  }
  for (; u < units; ++u) {  // the last units: fewer loads behind each
    switch (units - 1 - u) {
      case 0: wait_vm<0>(); break;
      case 1: wait_vm<1 * IPU>(); break;
      case 2: wait_vm<(NBUF > 2 ? 2 : 1) * IPU>(); break;
      case 3: wait_vm<(NBUF > 3 ? 3 : 1) * IPU>(); break;
      case 4: wait_vm<(NBUF > 4 ? 4 : 1) * IPU>(); break;
      default: wait_vm<(NBUF - 1) * IPU>(); break;
    }
    multiply(u, buf);
    buf = buf + 1 == NBUF ? 0 : buf + 1;
  }

  // this wave's partial tiles into its own LDS (its staged data is dead)
  f32x4* part = reinterpret_cast<f32x4*>(lds + wave * kWave);
#pragma unroll
  for (int nb = 0; nb < NB; ++nb)
#pragma unroll
    for (int i = 0; i < MT; ++i) part[(nb * MT + i) * 64 + lane] = acc[nb][i];
  lds_barrier();
  if (tid >= MT * 64) return;
  const int i = tid >> 6;
  auto total = [&](int tile) {
    f32x4 v = *reinterpret_cast<const f32x4*>(lds + (tile * 64 + lane) * 16);
#pragma unroll
    for (int j = 1; j < KS; ++j)
      v += *reinterpret_cast<const f32x4*>(lds + j * kWave + (tile * 64 + lane) * 16);
    return v;
  };
  f32x4 v = total(i);
  if constexpr (SILU) {
    const f32x4 up = total(MT + i);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      // torch rounds the gate_up product, then F.silu, then the product
      const float g = C::round(v[e]);
      v[e] = C::round(g / (1.f + __expf(-g))) * C::round(up[e]);
    }
  }
  const int row = m0 + 16 * i + col;
  if (row < a.m && (XR >= 16 || col < XR) && 4 * kg < WR) {
    u32x2 o;
    o[0] = C::pack(v[0], v[1]);
    o[1] = C::pack(v[2], v[3]);
    *reinterpret_cast<u32x2*>(a.y + (int64_t)row * a.y_stride + n0 + 4 * kg) = o;
  }
}

template <int WR, int XR, bool SILU, bool F16, int NORMK, bool RESID>
static void launch_t(Args a, int n_out, hipStream_t st) {
  a.n_tiles = n_out / WR;
  const dim3 grid((unsigned)(cdiv(a.m, XR) * a.n_tiles)), block(64 * KS);
  // k up to 1024 has two units per wave: less LDS, more workgroups per CU
  if constexpr (NORMK == 0) {
    if (a.k > 2 * KS * kUnitK) {
      hipLaunchKernelGGL((small_kernel<WR, XR, SILU, F16, NORMK, RESID, 6>), grid, block, 0, st, a);
      return;
    }
  }
  hipLaunchKernelGGL((small_kernel<WR, XR, SILU, F16, NORMK, RESID, 2>), grid, block, 0, st, a);
}

template <int WR, bool SILU, bool F16, int NORMK, bool RESID>
static void launch_x(const Args& a, int n_out, hipStream_t st) {
  if (a.m <= 8) launch_t<WR, 8, SILU, F16, NORMK, RESID>(a, n_out, st);
  else if (a.m <= 16) launch_t<WR, 16, SILU, F16, NORMK, RESID>(a, n_out, st);
  else launch_t<WR, 32, SILU, F16, NORMK, RESID>(a, n_out, st);
}

// 16 columns per workgroup when that gives at least 128 workgroups, else 8.
template <bool SILU, bool F16, int NORMK, bool RESID>
static void launch_w(const Args& a, int n_out, hipStream_t st) {
  if (n_out >= 2048) launch_x<16, SILU, F16, NORMK, RESID>(a, n_out, st);
  else launch_x<8, SILU, F16, NORMK, RESID>(a, n_out, st);
}

template <bool SILU, bool F16>
static int launch_f(const Args& a, int n_out, hipStream_t st) {
  if (a.norm_w == nullptr) {
    launch_w<SILU, F16, 0, false>(a, n_out, st);
  } else if (a.k == 512) {
    if (a.res) launch_w<SILU, F16, 512, true>(a, n_out, st);
    else launch_w<SILU, F16, 512, false>(a, n_out, st);
  } else if (a.k == 1024) {
    if (a.res) launch_w<SILU, F16, 1024, true>(a, n_out, st);
    else launch_w<SILU, F16, 1024, false>(a, n_out, st);
  } else {
    return AAC_ERR_UNSUPPORTED;
  }
  return AAC_OK;
}

// Measured in HIP-graph replay with cold weights (28 sets), us per launch
// against the best tiling of gemm.hip: m = 4: o_proj (1024 x 2048) 3.3 against
// 5.7, down (1024 x 3072) 3.8 against 6.9, gate/up + SiLU (3072 x 1024) 4.9
// against 9.5, QKV (4096 x 1024) 3.6 against 4.9; m = 32: 4.5, 5.4, 5.6 and 3.9
// against 6.0, 7.3, 9.4 and 4.9; m = 64 (two row tiles, W drawn twice): 4.7, 5.6,
// 8.9 and 6.0 against 5.9, 7.2, 9.4 and 4.9, the last with 512 workgroups; m = 96:
// 7.5, 9.2 and 12.0 against 5.9, 7.1 and 9.6.
bool small_takes(int m, int n, int k) {
  if (k % (KS * kUnitK) || n % 32) return false;
  if (m <= 32) return true;
  return m <= 64 && 2 * (n / (n >= 2048 ? 16 : 8)) <= 384;
}

int launch_small(const Args& a, int n_out, bool silu, bool f16, hipStream_t st) {
  if (silu) return f16 ? launch_f<true, true>(a, n_out, st) : launch_f<true, false>(a, n_out, st);
  return f16 ? launch_f<false, true>(a, n_out, st) : launch_f<false, false>(a, n_out, st);
}

}  // namespace gs
}  // namespace aac

using namespace aac;

// Whether [a, a + na) and [b, b + nb) share a byte (null: nothing).
static bool overlap(const void* a, size_t na, const void* b, size_t nb) {
  return a && b && (uintptr_t)a < (uintptr_t)b + nb && (uintptr_t)b < (uintptr_t)a + na;
}

extern "C" int aac_rmsnorm_gemm_nt(const void* x, int64_t x_row_stride, const void* residual,
                                   void* residual_out, const void* norm_weight, float eps,
                                   const void* w, int64_t w_row_stride, void* y, int64_t y_row_stride,
                                   int32_t m, int32_t n, int32_t k, int32_t silu_intermediate,
                                   int32_t dtype, void* stream) {
  if (dtype != AAC_DTYPE_BF16 && dtype != AAC_DTYPE_FP16) return AAC_ERR_UNSUPPORTED;
  if (m < 0 || n <= 0 || k <= 0 || silu_intermediate < 0) return AAC_ERR_INVALID_ARGUMENT;
  if (silu_intermediate > 0 && silu_intermediate != n) return AAC_ERR_SHAPE;
  if (x_row_stride < k || w_row_stride < k || y_row_stride < n) return AAC_ERR_SHAPE;
  if (n % 32 || (k != 512 && k != 1024)) return AAC_ERR_UNSUPPORTED;
  if (m == 0) return AAC_OK;
  if (!x || !norm_weight || !w || !y || ((residual == nullptr) != (residual_out == nullptr)))
    return AAC_ERR_INVALID_ARGUMENT;
  if (((uintptr_t)x | (uintptr_t)w | (uintptr_t)norm_weight | (uintptr_t)residual |
       (uintptr_t)residual_out) % 16 || (uintptr_t)y % 8 || x_row_stride % 8 || w_row_stride % 8 ||
      y_row_stride % 4)
    return AAC_ERR_MISALIGNED;
  if (cdiv(m, 8) * (n / 8) >= (int64_t(1) << 31)) return AAC_ERR_UNSUPPORTED;
  // every workgroup reads all rows of x and residual, with no order between them
  const size_t rows = (size_t)m * k * 2, xb = ((size_t)(m - 1) * x_row_stride + k) * 2;
  const size_t yb = ((size_t)(m - 1) * y_row_stride + n) * 2;
  if (overlap(residual_out, rows, x, xb) || overlap(residual_out, rows, residual, rows) ||
      overlap(y, yb, x, xb) || overlap(y, yb, residual, rows) || overlap(y, yb, residual_out, rows))
    return AAC_ERR_INVALID_ARGUMENT;
  gs::Args a{};
  a.x = (const u16*)x;
  a.x_stride = x_row_stride;
  a.res = (const u16*)residual;
  a.res_out = (u16*)residual_out;
  a.norm_w = (const u16*)norm_weight;
  a.eps = eps;
  a.w = (const u16*)w;
  a.w_stride = w_row_stride;
  a.y = (u16*)y;
  a.y_stride = y_row_stride;
  a.m = m;
  a.k = k;
  a.silu_off = silu_intermediate;
  const int rc = gs::launch_small(a, n, silu_intermediate > 0, dtype == AAC_DTYPE_FP16, (hipStream_t)stream);
  if (rc != AAC_OK) return rc;
  hipError_t e = hipGetLastError();
  return e == hipSuccess ? AAC_OK : (int)e;
}
