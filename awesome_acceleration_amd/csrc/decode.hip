// Paged decode attention (gfx950): one query token per sequence against a
// paged KV cache -- the attend half of the reference's
// flash_attn_with_kvcache call (model/model.py:233-240).
//
// Work decomposition
//   grid = (kv_head, partition, sequence), 256 threads (4 wavefronts); the KV
//   heads of one token range are adjacent in dispatch order, so the 256-byte
//   head slices of each 2 KiB cache row are fetched at about the same time.
//   A workgroup owns one KV head of one sequence over a partition of
//   `part_tokens` consecutive context tokens and serves all G = Hq/Hkv query
//   heads that share that KV head, so each K/V byte is read from HBM once.
//   Without a split (up to 1024 sequences), blockIdx.z is a rank in
//   descending context-length order, which every workgroup maps to its
//   sequence: the dispatcher, which hands out workgroups in index order as
//   slots free up, then starts long sequences first and fills the end of the
//   launch with short ones instead of leaving a few long ones running alone
//   (256 sequences of 1024..2047 tokens: 264 -> 254 us).
//   Inside the workgroup every 16-lane DPP row owns one token row at a time:
//   lane li holds head dims [8*li, 8*li+8) and loads them with one 16-byte
//   global load (two for fp32), so a wavefront reads 4 token rows (4 x 256 B
//   in bf16) per load instruction and U=8 rows per DPP row (4 for G=8) are in
//   flight before the first use: the block-table entries of an iteration are
//   loaded one iteration ahead and all K/V loads are issued before any math
//   (with in-order load counters, a block-table load waited for in between
//   would also wait for every earlier K/V load).  The 16 rows of a workgroup
//   walk the partition in lock step (row slot r takes tokens t0 + r,
//   t0 + r + 16, ...); slots past the partition end re-read token t0's row
//   (finite, probability 0) so the loads never branch.  K/V are read with
//   non-temporal loads: each byte is used once per step, so it should not
//   displace anything from L2/MALL (measured +10% bandwidth).  Power-of-two
//   block sizes use shift/mask for the block-table lookup.
//
// Softmax
//   Each DPP row keeps its own online-softmax state (running max m, running
//   sum l, fp32 accumulator for its 8 dims x G heads; Milakov & Gimelshein
//   2018), in the log2 domain (exponentiated with v_exp_f32).  bf16/fp16: q.k
//   is v_dot2 on the packed rows, the probabilities are rounded to the input
//   type and P.V is v_dot2 over V words paired across two tokens (v_perm);
//   fp32: unpacked fp32 FMAs with q pre-scaled.  The 16 row states of a workgroup are
//   merged at the end (cross-row shuffles inside a wave, LDS across waves).
//   A sequence whose context spans one partition writes the final output
//   directly; longer contexts write a normalised partial output and its
//   log-sum-exp to the workspace, and a second kernel combines the
//   partitions (the FlashDecoding split-K method).
//
// The new token (aac_decode_append_paged, aac_decode_qkv_paged): appended by
// the attention launch itself, see NEW at the kernel.  Against a store launch
// before it: 24 slot-layout sequences of 100-2063 tokens 27.1 -> 25.6 us (graph
// replay), a 28-layer step of 4 sequences some 40 us less with the q/k norm + RoPE
// folded in too.  The search for rows that share blocks is 0.3-1.2 us of that a
// launch (without it 24.4; the step 824 against 838).
//
// Bytes per launch (the HBM roofline): every context token's K and V row of
// each KV head is read exactly once, 2 * Hkv * D * elem_bytes per token, plus
// q and out; the reduction adds 2 * B * Hq * P * (D + 1) * 4 bytes when split.

#include <algorithm>
#include <climits>
#include <mutex>

#include "qk_head.h"


namespace aac {

constexpr int kHeadDim = 128;
constexpr int kRowLanes = 16;  // lanes per token row: 128 dims / 8 per lane

struct DecodeArgs {
  const void* q;
  int64_t q_seq_stride;  // elements
  const void* k_cache;
  const void* v_cache;
  int64_t num_blocks;
  int32_t block_size;
  const int32_t* block_tables;
  int32_t max_blocks;
  const int32_t* lens;  // context length of sequence b = lens[b] + lens_add
  int32_t lens_add;
  int32_t n_seqs;
  int32_t hq;
  int32_t hkv;
  float scale_log2;  // softmax scale * log2(e)
  void* out;
  int64_t out_seq_stride;  // elements
  float* ws_o;             // [B][Hq][P][D] normalised partial outputs
  float* ws_lse;           // [B][Hq][P]    log2-sum-exp of each partition
  // [B][Hkv] finished partitions, or null: a second launch combines them
  unsigned long long* ws_cnt;
  int32_t n_parts;
  int32_t part_tokens;
  int32_t bs_shift;  // log2(block_size) when it is a power of two
  // otherwise t / block_size = (t * bs_magic) >> bs_mshift for 0 <= t < 2^31
  // (Granlund & Montgomery 1994, Thm 4.2: bs_magic = floor(2^(31+l) / d) + 1
  // with l = ceil(log2 d), bs_mshift = 31 + l)
  uint64_t bs_magic;
  int32_t bs_mshift;
  int32_t lpt;       // 1: blockIdx.z is a rank in descending context order
  int32_t lpt_max;   // context bound the length classes are scaled to
  // The new token's rows of sequence b (NEW): [n_seqs, hkv, 128] with these
  // sequence strides (elements); lens[b] is its position.  The caches are
  // written here.
  const void* k_new;
  const void* v_new;
  int64_t k_new_stride, v_new_stride;
  // NEW == kQkv: q and k_new are the projection's raw rows; norm weights, RoPE
  // tables [max_pos, 128] and positions as in qk_head.h
  const u16 *qw, *kw, *cos, *sin;
  const int32_t* positions;
  int32_t max_pos;
  float eps;
};

// What the launch does with the step's new token: nothing (its rows are in the
// caches already), append its K/V rows, or also make q and k from the QKV
// projection's rows (q/k RMSNorm + RoPE).
// kAppendMerge: kAppend, and the partition that finishes last combines them all
// (a form of its own, as its code costs the others 0.85 us a launch: a 28-layer
// step of 4 sequences 872 -> 896 us).
enum { kNone = 0, kAppend = 1, kQkv = 2, kAppendMerge = 3 };

// Raw storage for the 8 elements one lane owns in one token row.
template <Dt DT> struct Raw8 {
  static constexpr int kWords = Elem<DT>::kBytes * 8 / 16;  // u32x4 words
  u32x4 w[kWords];
  __device__ inline void load(const char* p) {
#pragma unroll
    for (int i = 0; i < kWords; ++i)
      w[i] = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(p + 16 * i));
  }
  __device__ inline void zero() {
#pragma unroll
    for (int i = 0; i < kWords; ++i) w[i] = u32x4{0, 0, 0, 0};
  }
  __device__ inline void store(char* p) const {
#pragma unroll
    for (int i = 0; i < kWords; ++i) *reinterpret_cast<u32x4*>(p + 16 * i) = w[i];
  }
  __device__ inline void unpack(float* f) const {
    if constexpr (DT == Dt::FP32) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        f[i] = __uint_as_float(w[0][i]);
        f[4 + i] = __uint_as_float(w[1][i]);
      }
    } else {
      Elem<DT>::unpack8(w[0], f);
    }
  }
};

__device__ __forceinline__ int clip_len(const DecodeArgs& a, int len) {
  int ctx = len + a.lens_add;
  const int64_t cap = (int64_t)a.max_blocks * a.block_size;  // may lie past 2^31
  ctx = ctx < 0 ? 0 : ctx;
  return ctx > cap ? (int)cap : ctx;
}
__device__ __forceinline__ int context_len(const DecodeArgs& a, int b) { return clip_len(a, a.lens[b]); }

__device__ __forceinline__ int parts_of(const DecodeArgs& a, int ctx) {
  const int n = (int)(((uint32_t)ctx + (uint32_t)a.part_tokens - 1) / (uint32_t)a.part_tokens);
  return n > a.n_parts ? a.n_parts : n;
}

// Sequence of rank `rank` in descending context-length order, by length
// class: class c = ctx * 64 / (lpt_max + 1) (64 classes, longest first),
// index order inside a class.  Counts, prefix sums and ballots do not depend
// on timing, so every workgroup derives the same bijection rank -> sequence:
//   1. histogram of the classes (LDS atomics; the counts are exact),
//   2. one wavefront scans the 64 counts and finds the class and position of
//      `rank`,
//   3. per 64-sequence chunk a ballot of "in that class" and its popcounts
//      give each sequence its position inside the class.
constexpr int kLptMaxSeqs = 1024;
constexpr int kLptClasses = 64;
__device__ __forceinline__ int seq_of_rank(const DecodeArgs& a, int rank, int tid) {
  __shared__ int s_cnt[kLptClasses];
  __shared__ int s_wcnt[kLptMaxSeqs / 64];
  __shared__ int s_sel[2];
  __shared__ int s_pick;
  const int n = a.n_seqs, lane = tid & 63, wave = tid >> 6;
  if (tid < kLptClasses) s_cnt[tid] = 0;
  __syncthreads();
  int cls[kLptMaxSeqs / 256];  // descending class index of sequences tid + 256k (-1: none)
#pragma unroll
  for (int k = 0; k < kLptMaxSeqs / 256; ++k) {
    const int i = tid + 256 * k;
    cls[k] = -1;
    if (i < n) {
      const int64_t c = (int64_t)context_len(a, i) * kLptClasses / ((int64_t)a.lpt_max + 1);
      cls[k] = kLptClasses - 1 - (int)(c < kLptClasses - 1 ? c : kLptClasses - 1);
      atomicAdd(&s_cnt[cls[k]], 1);
    }
  }
  __syncthreads();
  if (wave == 0) {
    const int v = s_cnt[lane];
    int incl = v;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
      const int t = __shfl_up(incl, off);
      if (lane >= off) incl += t;
    }
    if (rank >= incl - v && rank < incl) {
      s_sel[0] = lane;
      s_sel[1] = rank - (incl - v);
    }
  }
  __syncthreads();
  const int csel = s_sel[0], psel = s_sel[1];
  unsigned long long bal[kLptMaxSeqs / 256];
#pragma unroll
  for (int k = 0; k < kLptMaxSeqs / 256; ++k) {
    bal[k] = __ballot(cls[k] == csel);
    if (lane == 0) s_wcnt[4 * k + wave] = __popcll(bal[k]);
  }
  __syncthreads();
  int base = 0;
#pragma unroll
  for (int k = 0; k < kLptMaxSeqs / 256; ++k) {
    const int chunk = 4 * k + wave;  // 64-sequence chunks in index order
    int before = base;
    for (int m = 4 * k; m < chunk; ++m) before += s_wcnt[m];
    const int pos = before + (int)__builtin_amdgcn_mbcnt_hi((unsigned)(bal[k] >> 32),
                                                          __builtin_amdgcn_mbcnt_lo((unsigned)bal[k], 0u));
    if (cls[k] == csel && pos == psel) s_pick = tid + 256 * k;
    for (int m = 4 * k; m < 4 * k + 4; ++m) base += s_wcnt[m];
  }
  __syncthreads();
  return s_pick;
}

template <Dt DT>
__device__ __forceinline__ void store_out2(void* out, int64_t idx, float x0, float x1) {
  if constexpr (DT == Dt::FP32) {
    *reinterpret_cast<float2*>(reinterpret_cast<float*>(out) + idx) = make_float2(x0, x1);
  } else {
    *reinterpret_cast<u32*>(reinterpret_cast<u16*>(out) + idx) = Elem<DT>::pack2(x0, x1);
  }
}

// A (sequence, KV head)'s partial rows and log-sum-exps in the workspace
constexpr int kSc1 = 16;  // cache policy: coherent across XCDs
constexpr unsigned long long kCntTag = 0xa3c59e176b2dull << 16;
template <int G> __device__ __forceinline__ __amdgpu_buffer_rsrc_t ws_rows(const DecodeArgs& a, int b, int h) {
  return __builtin_amdgcn_make_buffer_rsrc(a.ws_o + ((int64_t)b * a.hq + h * G) * a.n_parts * kHeadDim, 0,
                                           G * a.n_parts * kHeadDim * 4, 0x00020000);
}
template <int G> __device__ __forceinline__ __amdgpu_buffer_rsrc_t ws_lses(const DecodeArgs& a, int b, int h) {
  return __builtin_amdgcn_make_buffer_rsrc(a.ws_lse + ((int64_t)b * a.hq + h * G) * a.n_parts, 0,
                                           G * a.n_parts * 4, 0x00020000);
}

// One dword per lane from global memory straight into LDS at p + lane.  Inline
// assembly: the compiler neither moves the load (it sinks ordinary ones to their
// first use, behind the wait for the context length) nor waits for it; read p
// behind landed().
__device__ __forceinline__ void to_lds4(const int32_t* src, int* p) {
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
  asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dword %0, off"
               :
               : "v"(src), "s"((u32)(uintptr_t)(__attribute__((address_space(3))) int*)p)
               : "memory", "m0");
#pragma clang diagnostic pop
}
__device__ __forceinline__ void landed() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }

// NEW: the workgroup that holds the new token (the last one of the context)
// starts its online softmax from it, straight from the given rows, and writes
// them to the caches: the loop is that of kNone, and there is no launch before
// this one.  The result is that of a store launch before the attention also
// where rows of the call share blocks (one sequence given as several rows, at
// positions n, n + 1, ...): in a workgroup whose tokens include another row's new
// one, each wave first writes that row to the cache too, the same bytes as its
// owner, and reads what it wrote.  Looked for before the loop: beside its first
// loads, or behind it with a second pass, the search's registers spilled or its
// code cost more than the latency (step of 4 sequences 857 us, and 833-850 with the
// tables scanned entry by entry, whose cost grows with them: 64 x 10-500 21 us).
template <Dt DT, int G, int U, bool POW2, int NEW>
// Occupancy: with G <= 2 the kernel fits 128 VGPRs, i.e. four workgroups per
// CU (16 wavefronts); larger groups hold more accumulators.
__global__ __launch_bounds__(256, G <= 2 ? 4 : 2) void decode_paged_kernel(DecodeArgs a) {
  constexpr int ES = Elem<DT>::kBytes;
  // The KV heads of one token range are dispatched together.  Workgroups go
  // to the 8 XCDs round-robin, so with an even head count workgroup x runs
  // on an XCD of x's parity; it attends head x ^ 1, on the XCD of the other
  // parity: measured on MI355X over all eight rotations of heads to XCDs,
  // the odd ones (256 seqs x 1-2k, 16/8 heads: 246.4-247.0 us) beat the even
  // ones (253.2-253.3 us), and likewise at 8/4 heads (129.4-129.7 against
  // 132.8-133.0 us).
  const int h = (a.hkv & 1) ? (int)blockIdx.x : (int)(blockIdx.x ^ 1u);
  const int part = blockIdx.y;
  const int tid = threadIdx.x;
  // Longest contexts first: the dispatcher hands out workgroups in index
  // order as slots free up, so the short sequences fill the tail instead of
  // a few long ones running alone at the end.
  const int b = a.lpt ? __builtin_amdgcn_readfirstlane(seq_of_rank(a, blockIdx.z, tid))
                     : (int)blockIdx.z;  // wave-uniform (SGPR) either way
  constexpr int R = 16;  // token rows of the workgroup (one per DPP row)
  const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int li = lane & 15, grp = lane >> 4;
  const int rslot = wave * 4 + grp;  // 0 .. R - 1
  const int t0 = (int)((uint32_t)part * (uint32_t)a.part_tokens);  // past 2^31: no such partition
  const int32_t* bt = a.block_tables + (int64_t)b * a.max_blocks;
  const uint32_t nb32 = a.num_blocks < 0x7fffffff ? (uint32_t)a.num_blocks : 0x7fffffffu;
  auto block_index = [&](int t) {
    return POW2 ? t >> a.bs_shift : (int)(((uint64_t)(uint32_t)t * a.bs_magic) >> a.bs_mshift);
  };
  // an entry of the row's table for any t, before it is known to be a token
  auto entry = [&](int i) { return bt + min((uint32_t)i, (uint32_t)a.max_blocks - 1u); };

  // A call of few sequences is a chain of latencies, so everything that does not
  // depend on the context length is loaded beside it: the block numbers of the
  // first iteration (clamped to the table; past the context replaced below)
  // and the query rows.  The first K/V loads then wait for one load, not four,
  // and the query's preparation runs while they are in flight (28-layer step of
  // 4 sequences 879 -> 870 us; 256 x 1-2k 241.2 -> 240.2, 64 x 16k-32k 989.5 -> 984.5).
  const int len = a.lens[b];
  int blk[U];
#pragma unroll
  for (int u = 0; u < U; ++u) blk[u] = *entry(block_index((int)((uint32_t)t0 + rslot + R * u)));
  const int blk0 = *entry(block_index(t0));
  Raw8<DT> qr[G];
  {
    const char* qb = reinterpret_cast<const char*>(a.q) +
                     ((int64_t)b * a.q_seq_stride + (int64_t)h * G * kHeadDim + li * 8) * ES;
#pragma unroll
    for (int g = 0; g < G; ++g) qr[g].load(qb + (int64_t)g * kHeadDim * ES);
  }
  // NEW == kQkv: the norm weight and RoPE rows of the query heads
  struct Rope {
    u32x4 c, s;
  };
  auto rope_of = [&](int row) {
    Rope r = {};
    if constexpr (NEW == kQkv) {
      const int64_t at = (int64_t)min(max(a.positions[row], 0), a.max_pos - 1) * kHeadDim + li * 8;
      r.c = *reinterpret_cast<const u32x4*>(a.cos + at);
      r.s = *reinterpret_cast<const u32x4*>(a.sin + at);
    }
    return r;
  };
  const Rope rope = rope_of(b);
  u32x4 wraw;
  if constexpr (NEW == kQkv) wraw = *reinterpret_cast<const u32x4*>(a.qw + li * 8);
  // NEW: wave 3 looks for rows that share blocks (below), from the positions of the
  // call's first 64 rows and the first 64 blocks of this partition.  One wave, as at
  // the start all waves of a CU compete for issue.
  __shared__ int s_new[NEW == kNone ? 1 : 2][64];
  __shared__ int s_share;
  if (NEW != kNone && wave == 3) {
    to_lds4(a.lens + min(lane, a.n_seqs - 1), s_new[0]);
    to_lds4(entry((int)((uint32_t)block_index(t0) + lane)), s_new[1]);
  }
  // RMSNorm + RoPE of one head row
  auto new_head = [&](const u32x4& raw, const u32x4& w, const Rope& r) {
    u32x4 o = raw;
    if constexpr (NEW == kQkv) {
      float wf[8], cf[8], sf[8];
      fz::unpack8<DT>(w, wf);
      fz::unpack8<DT>(r.c, cf);
      fz::signed_sin<DT>(r.s, li, sf);
      o = fz::norm_rope_row<DT>(raw, a.eps, wf, cf, sf);
    }
    return o;
  };

  const int ctx = clip_len(a, len);
  const int np = parts_of(a, ctx);
  if (part >= np) {
    if (part == 0) {  // empty context: zeros (FA2 convention)
      for (int i = tid; i < G * (kHeadDim / 2); i += 256) {
        const int g = i / (kHeadDim / 2), d2 = (i % (kHeadDim / 2)) * 2;
        store_out2<DT>(a.out, (int64_t)b * a.out_seq_stride + (int64_t)(h * G + g) * kHeadDim + d2,
                       0.f, 0.f);
      }
    }
    if constexpr (NEW != kNone) landed();
    return;
  }
  // NEW: the last partition takes the new token (position lens[b], unless that
  // lies outside the table) apart from the loop, which ends before it.
  const bool has_new = NEW != kNone && part == np - 1 && len == ctx - 1;
  const int t1 = (part == np - 1) ? ctx - (has_new ? 1 : 0) : t0 + a.part_tokens;

  const int64_t tok_bytes = (int64_t)a.hkv * kHeadDim * ES;  // cache row stride
  const char* kbase = reinterpret_cast<const char*>(a.k_cache) + ((int64_t)h * kHeadDim + li * 8) * ES;
  const char* vbase = reinterpret_cast<const char*>(a.v_cache) + ((int64_t)h * kHeadDim + li * 8) * ES;

  // Token t of this partition, or t0 (a valid token whose row is finite and
  // whose probability is set to 0) past its end, so loads never branch.
  auto token = [&](int t) { return t < t1 ? t : t0; };
  // byte offset of token t's cache row in block `b` (bad entries read block 0)
  auto row_off = [&](int t, int b) {
    const int off = POW2 ? t & (a.block_size - 1) : t - block_index(t) * a.block_size;
    return ((int64_t)((uint32_t)b < nb32 ? (uint32_t)b : 0u) * a.block_size + off) * tok_bytes;
  };
  // The block numbers of an iteration's U tokens are loaded one iteration
  // ahead: a block-table load waited for right before the K/V loads would,
  // with in-order load counters, also wait for every K/V load issued before
  // it and leave one token per wave in flight.
#pragma unroll
  for (int u = 0; u < U; ++u) blk[u] = t0 + rslot + R * u < t1 ? blk[u] : blk0;

  // q for the G heads of this KV head.  fp32: unpacked and pre-scaled into
  // the log2 domain.  bf16/fp16 (PK): kept packed and exact for v_dot2; the
  // scale is applied to the scores instead.
  constexpr bool PK = DT != Dt::FP32;
  float qf[PK ? 1 : G][8];
  u32 qp[PK ? G : 1][4];
  float m[G], l[G], acc[G][8];
  // the query: once a row's first K/V loads are on their way, or before them
  // where its registers beside theirs would spill
  constexpr bool kQueryFirst = NEW == kQkv || G == 8 || DT == Dt::FP32;
  auto prepare = [&]() {
#pragma unroll
    for (int g = 0; g < G; ++g) {
      if constexpr (NEW == kQkv) qr[g].w[0] = new_head(qr[g].w[0], wraw, rope);
      if constexpr (PK) {
#pragma unroll
        for (int w = 0; w < 4; ++w) qp[g][w] = qr[g].w[0][w];
      } else {
        qr[g].unpack(qf[g]);
#pragma unroll
        for (int i = 0; i < 8; ++i) qf[g][i] *= a.scale_log2;
      }
    }

#pragma unroll
    for (int g = 0; g < G; ++g) {
      m[g] = -1e30f;
      l[g] = 0.f;
#pragma unroll
      for (int i = 0; i < 8; ++i) acc[g][i] = 0.f;
    }
  };

  bool ready = kQueryFirst;
  if constexpr (kQueryFirst) prepare();

  // The rows r0 .. r0 + 63 whose new token is one of [t0, t1), as a lane mask, with
  // their positions and blocks: rows in lanes, the partition's blocks one by one.
  // From memory, or the first ones from LDS.
  struct New {
    int pos, blk;
  };
  auto shared_rows = [&](int r0, bool lds, New& e) {
    const int row = min(r0 + lane, a.n_seqs - 1);
    e.pos = lds ? s_new[0][lane] : a.lens[row];
    const int bi = block_index(max(e.pos, 0)), off = e.pos - bi * a.block_size;
    e.blk = a.block_tables[(int64_t)row * a.max_blocks + min(bi, a.max_blocks - 1)];
    bool hit = false;
    if (t1 > t0) {
      const int first = block_index(t0), last = block_index(t1 - 1);
      for (int i0 = first; i0 <= last; i0 += 64) {
        const int own = lds && i0 == first ? s_new[1][lane] : *entry(i0 + lane);
        const int n = min(64, last + 1 - i0);
        for (int j = 0; j < n; ++j) {
          const int t = (i0 + j) * a.block_size + off;
          hit |= __builtin_amdgcn_readlane(own, j) == e.blk && t >= t0 && t < t1;
        }
      }
    }
    // the row's new token is inside the table, its block inside the cache
    return __ballot(hit && r0 + lane < a.n_seqs && e.pos >= 0 && bi < a.max_blocks && (uint32_t)e.blk < nb32);
  };
  // Write those rows to the caches (every wave for itself).
  auto settle = [&]() {
    for (int r0 = 0; r0 < a.n_seqs; r0 += 64) {
      New e;
      for (unsigned long long rows = shared_rows(r0, false, e); rows; rows &= rows - 1) {
        const int i = __ffsll(rows) - 1, row = r0 + i;
        const int64_t to = row_off(__builtin_amdgcn_readlane(e.pos, i), __builtin_amdgcn_readlane(e.blk, i));
        const int64_t hd = (int64_t)h * kHeadDim + li * 8;
        Raw8<DT> kx, vx;
        kx.load(reinterpret_cast<const char*>(a.k_new) + (row * a.k_new_stride + hd) * ES);
        vx.load(reinterpret_cast<const char*>(a.v_new) + (row * a.v_new_stride + hd) * ES);
        if constexpr (NEW == kQkv)
          kx.w[0] = new_head(kx.w[0], *reinterpret_cast<const u32x4*>(a.kw + li * 8), rope_of(row));
        if (lane < kRowLanes) {
          kx.store(const_cast<char*>(kbase) + to);
          vx.store(const_cast<char*>(vbase) + to);
        }
      }
    }
    landed();
  };
  if constexpr (NEW != kNone) {
    if (wave == 3) {
      landed();
      unsigned long long rows = 0;
      New e;
      for (int r0 = 0; r0 < a.n_seqs; r0 += 64) rows |= shared_rows(r0, r0 == 0, e);
      if (lane == 0) s_share = rows != 0;
    }
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    if (s_share) settle();
  }

  // The new token: row 0 of the workgroup starts its online softmax from the
  // given rows and writes them to the caches (not to a block outside the
  // cache: then the row that a bad entry reads takes their place).
  if (NEW != kNone && has_new && wave == 0) {
    if constexpr (!kQueryFirst) {
      prepare();
      ready = true;
    }
    const int pos = ctx - 1, bk = bt[block_index(pos)];
    const bool store = (uint32_t)bk < nb32;  // wave-uniform
    const int64_t off = row_off(pos, bk);
    const int64_t hd = (int64_t)h * kHeadDim + li * 8;
    Raw8<DT> kx, vx;
    kx.load(store ? reinterpret_cast<const char*>(a.k_new) + (b * a.k_new_stride + hd) * ES : kbase + off);
    vx.load(store ? reinterpret_cast<const char*>(a.v_new) + (b * a.v_new_stride + hd) * ES : vbase + off);
    if constexpr (NEW == kQkv) {
      if (store) kx.w[0] = new_head(kx.w[0], *reinterpret_cast<const u32x4*>(a.kw + li * 8), rope);
    }
    float vf[8], kf[PK ? 1 : 8];
    vx.unpack(vf);
    if constexpr (!PK) kx.unpack(kf);
    const bool first = lane < kRowLanes;
#pragma unroll
    for (int g = 0; g < G; ++g) {
      float d = 0.f;
      if constexpr (PK) {
#pragma unroll
        for (int w = 0; w < 4; ++w) d = Elem<DT>::dot2(kx.w[0][w], qp[g][w], d);
      } else {
#pragma unroll
        for (int i = 0; i < 8; ++i) d = fmaf(qf[g][i], kf[i], d);
      }
      d = row16_sum(d);
      m[g] = first ? (PK ? d * a.scale_log2 : d) : m[g];
      l[g] = first ? 1.f : 0.f;
#pragma unroll
      for (int i = 0; i < 8; ++i) acc[g][i] = first ? vf[i] : 0.f;
    }
    if (first && store) {
      kx.store(const_cast<char*>(kbase) + off);
      vx.store(const_cast<char*>(vbase) + off);
    }
  }

  for (int tb = t0 + rslot; tb < t1; tb += R * U) {
    Raw8<DT> kr[U], vr[U];
    bool valid[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      valid[u] = tb + R * u < t1;
      const int64_t off = row_off(token(tb + R * u), blk[u]);
      kr[u].load(kbase + off);
      vr[u].load(vbase + off);
    }
#pragma unroll
    for (int u = 0; u < U; ++u) blk[u] = bt[block_index(token(tb + R * U + R * u))];
    // Every load above is issued before any arithmetic below (the scheduler
    // would otherwise pull each token's math up behind its load and wait).
    __builtin_amdgcn_sched_barrier(0);
    if (!kQueryFirst && !ready) {
      prepare();
      ready = true;
    }
    float s[U][G];
    if constexpr (PK) {
      // Packed bf16/fp16: q.k with v_dot2 on the packed rows (no unpacking),
      // raw scores; the probabilities are rounded to the input type (as the
      // MFMA prefill and FA2 do for the PV product) and packed per token pair,
      // so that P V is v_dot2 too, over V words paired across two tokens by
      // v_perm.  The row sum l adds the same rounded probabilities.
      typedef Elem<DT> E;
#pragma unroll
      for (int u = 0; u < U; ++u)
#pragma unroll
        for (int g = 0; g < G; ++g) {
          float d = 0.f;
#pragma unroll
          for (int w = 0; w < 4; ++w) d = E::dot2(kr[u].w[0][w], qp[g][w], d);
          d = row16_sum(d);
          s[u][g] = valid[u] ? d : -INFINITY;
        }
      u32 pp[U / 2][G];
#pragma unroll
      for (int g = 0; g < G; ++g) {
        float mr = s[0][g];
#pragma unroll
        for (int u = 1; u + 1 < U; u += 2) mr = vmax3(mr, s[u][g], s[u + 1][g]);
        mr = vmax(mr, s[U - 1][g]);
        const float mx = vmax(m[g], mr * a.scale_log2);
        const float alpha = fast_exp2(m[g] - mx);
        m[g] = mx;
        l[g] *= alpha;
#pragma unroll
        for (int i = 0; i < 8; ++i) acc[g][i] *= alpha;
#pragma unroll
        for (int v = 0; v < U / 2; ++v) {
          const float p0 = fast_exp2(fmaf(s[2 * v][g], a.scale_log2, -mx));
          const float p1 = fast_exp2(fmaf(s[2 * v + 1][g], a.scale_log2, -mx));
          pp[v][g] = E::pack2_hw(p0, p1);
          l[g] = E::dot2(pp[v][g], E::kOnes, l[g]);
        }
      }
#pragma unroll
      for (int v = 0; v < U / 2; ++v)
#pragma unroll
        for (int w = 0; w < 4; ++w) {
          // (token 2v, token 2v+1) of dims 2w and 2w+1
          const u32 lo = __builtin_amdgcn_perm(vr[2 * v + 1].w[0][w], vr[2 * v].w[0][w], kSelLo);
          const u32 hi = __builtin_amdgcn_perm(vr[2 * v + 1].w[0][w], vr[2 * v].w[0][w], kSelHi);
#pragma unroll
          for (int g = 0; g < G; ++g) {
            acc[g][2 * w] = E::dot2(lo, pp[v][g], acc[g][2 * w]);
            acc[g][2 * w + 1] = E::dot2(hi, pp[v][g], acc[g][2 * w + 1]);
          }
        }
    } else {
#pragma unroll
      for (int u = 0; u < U; ++u) {
        float kf[8];
        kr[u].unpack(kf);
#pragma unroll
        for (int g = 0; g < G; ++g) {
          float d = 0.f;
#pragma unroll
          for (int i = 0; i < 8; ++i) d = fmaf(qf[g][i], kf[i], d);
          d = row16_sum(d);
          s[u][g] = valid[u] ? d : -INFINITY;
        }
      }
#pragma unroll
      for (int g = 0; g < G; ++g) {
        float mx = m[g];
#pragma unroll
        for (int u = 0; u < U; ++u) mx = fmaxf(mx, s[u][g]);
        const float alpha = fast_exp2(m[g] - mx);
        m[g] = mx;
        l[g] *= alpha;
#pragma unroll
        for (int i = 0; i < 8; ++i) acc[g][i] *= alpha;
#pragma unroll
        for (int u = 0; u < U; ++u) s[u][g] = fast_exp2(s[u][g] - mx);
      }
#pragma unroll
      for (int u = 0; u < U; ++u) {
        float vf[8];
        vr[u].unpack(vf);
#pragma unroll
        for (int g = 0; g < G; ++g) {
          l[g] += s[u][g];
#pragma unroll
          for (int i = 0; i < 8; ++i) acc[g][i] = fmaf(s[u][g], vf[i], acc[g][i]);
        }
      }
    }
  }
  if (!kQueryFirst && !ready) prepare();

  // Merge the 4 DPP rows of this wave (lanes li, li+16, li+32, li+48 hold the
  // same dims).
#pragma unroll
  for (int g = 0; g < G; ++g) {
    float mx = fmaxf(m[g], __shfl_xor(m[g], 16));
    mx = fmaxf(mx, __shfl_xor(mx, 32));
    const float f = fast_exp2(m[g] - mx);
    m[g] = mx;
    l[g] *= f;
    l[g] += __shfl_xor(l[g], 16);
    l[g] += __shfl_xor(l[g], 32);
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      float x = acc[g][i] * f;
      x += __shfl_xor(x, 16);
      x += __shfl_xor(x, 32);
      acc[g][i] = x;
    }
  }

  __shared__ float sm_m[4][G], sm_l[4][G];
  __shared__ float sm_acc[4][G][kHeadDim];
  if (grp == 0) {
#pragma unroll
    for (int g = 0; g < G; ++g) {
#pragma unroll
      for (int i = 0; i < 8; ++i) sm_acc[wave][g][li * 8 + i] = acc[g][i];
      if (li == 0) {
        sm_m[wave][g] = m[g];
        sm_l[wave][g] = l[g];
      }
    }
  }
  __syncthreads();

  for (int i = tid; i < G * (kHeadDim / 2); i += 256) {
    const int g = i / (kHeadDim / 2), d2 = (i % (kHeadDim / 2)) * 2;
    float mx = sm_m[0][g];
#pragma unroll
    for (int w = 1; w < 4; ++w) mx = fmaxf(mx, sm_m[w][g]);
    float L = 0.f, o0 = 0.f, o1 = 0.f;
#pragma unroll
    for (int w = 0; w < 4; ++w) {
      const float f = fast_exp2(sm_m[w][g] - mx);
      L += sm_l[w][g] * f;
      o0 += sm_acc[w][g][d2] * f;
      o1 += sm_acc[w][g][d2 + 1] * f;
    }
    const float inv = 1.f / L;
    const int hq = h * G + g;
    if (np == 1) {
      store_out2<DT>(a.out, (int64_t)b * a.out_seq_stride + (int64_t)hq * kHeadDim + d2, o0 * inv,
                     o1 * inv);
    } else if constexpr (NEW != kAppendMerge) {
      const int64_t slot = ((int64_t)b * a.hq + hq) * a.n_parts + part;
      *reinterpret_cast<float2*>(a.ws_o + slot * kHeadDim + d2) = make_float2(o0 * inv, o1 * inv);
      if (d2 == 0) a.ws_lse[slot] = mx + __log2f(L);
    } else {
      const u32x2 v = {__float_as_uint(o0 * inv), __float_as_uint(o1 * inv)};
      __builtin_amdgcn_raw_buffer_store_b64(v, ws_rows<G>(a, b, h), ((g * a.n_parts + part) * kHeadDim + d2) * 4, 0, kSc1);
      if (d2 == 0)
        __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(mx + __log2f(L)), ws_lses<G>(a, b, h),
                                              (g * a.n_parts + part) * 4, 0, kSc1);
    }
  }
  if constexpr (NEW != kAppendMerge) return;
  if (np == 1) return;

  // The partition that finishes last combines them all, in partition order
  // whichever it is.  Partial results are written and read past the XCDs' L2s
  // (sc1, as the compiler's agent-scope atomics are), every lane waits for its
  // own before the workgroup counts itself, and nothing waits for another
  // workgroup.  A counter holds kCntTag in its upper 48 bits from its first
  // use on (a workspace comes as it is) and goes back to zero finished.
  __shared__ int s_last;
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  if (tid == 0) {
    unsigned long long* cnt = a.ws_cnt + (int64_t)b * a.hkv + h;
    unsigned long long v = __hip_atomic_load(cnt, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if ((v & ~0xffffull) != kCntTag)
      __hip_atomic_compare_exchange_strong(cnt, &v, kCntTag, __ATOMIC_RELAXED, __ATOMIC_RELAXED,
                                           __HIP_MEMORY_SCOPE_AGENT);
    v = __hip_atomic_fetch_add(cnt, 1ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    s_last = (int)(v & 0xffff) == np - 1;
    if (s_last) __hip_atomic_store(cnt, kCntTag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  __syncthreads();
  if (!s_last) return;
  const __amdgpu_buffer_rsrc_t rows = ws_rows<G>(a, b, h), lses = ws_lses<G>(a, b, h);
  // wave w: head g, partitions c, c + C, ...; lane: two dims
  constexpr int C = G >= 4 ? 1 : 4 / G;
  __shared__ float sm_w[C][G];
  __shared__ float2 sm_o[C][G][64];
#pragma unroll
  for (int k = 0; k < (G > 4 ? G / 4 : 1); ++k) {
    const int g = G >= 4 ? wave + 4 * k : wave % G, c = G >= 4 ? 0 : wave / G;
    float mx = -INFINITY;
    for (int p = lane; p < np; p += 64)
      mx = fmaxf(mx, __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(lses, (g * a.n_parts + p) * 4, 0, kSc1)));
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) mx = fmaxf(mx, __shfl_xor(mx, o));
    constexpr int V = 8;  // partitions in flight
    float W = 0.f, o0 = 0.f, o1 = 0.f;
    for (int p0 = c; p0 < np; p0 += V * C) {
      u32 ls[V];
      u32x2 ov[V];
#pragma unroll
      for (int u = 0; u < V; ++u) {
        const int i = g * a.n_parts + min(p0 + u * C, np - 1);
        ls[u] = __builtin_amdgcn_raw_buffer_load_b32(lses, i * 4, 0, kSc1);
        ov[u] = __builtin_amdgcn_raw_buffer_load_b64(rows, (i * kHeadDim + 2 * lane) * 4, 0, kSc1);
      }
#pragma unroll
      for (int u = 0; u < V; ++u) {
        // past the end: nothing, not 0 x the last partition's (infinite?) result
        const bool in = p0 + u * C < np;
        const float w = fast_exp2(__uint_as_float(ls[u]) - mx);
        W += in ? w : 0.f;
        o0 = in ? fmaf(w, __uint_as_float(ov[u][0]), o0) : o0;
        o1 = in ? fmaf(w, __uint_as_float(ov[u][1]), o1) : o1;
      }
    }
    if constexpr (C > 1) {
      if (lane == 0) sm_w[c][g] = W;
      sm_o[c][g][lane] = make_float2(o0, o1);
      __syncthreads();
      if (c) return;
#pragma unroll
      for (int j = 1; j < C; ++j) {
        W += sm_w[j][g];
        o0 += sm_o[j][g][lane].x;
        o1 += sm_o[j][g][lane].y;
      }
    }
    const float inv = 1.f / W;
    store_out2<DT>(a.out, (int64_t)b * a.out_seq_stride + (int64_t)(h * G + g) * kHeadDim + 2 * lane,
                   o0 * inv, o1 * inv);
  }
}

// Combine the partitions of every (sequence, query head) whose context was
// split: out = sum_p 2^(lse_p - LSE) o_p with LSE = log2 sum_p 2^lse_p.
// Four wavefronts per (sequence, query head): each finds the largest lse (one
// load per 64 partitions), then wave w sums partitions w, w + 4, ... with four
// in flight, and the four sums meet in LDS.  The chain of loads is what it
// costs: one wave walking the partitions one by one took 5.2 us at 11 partitions
// of 24 sequences.
template <Dt DT>
__global__ __launch_bounds__(256) void decode_reduce_kernel(DecodeArgs a) {
  const int hq = blockIdx.x, b = blockIdx.y;
  const int np = parts_of(a, context_len(a, b));
  if (np <= 1) return;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int64_t slot0 = ((int64_t)b * a.hq + hq) * a.n_parts;
  float mx = -INFINITY;
  for (int p = lane; p < np; p += 64) mx = fmaxf(mx, a.ws_lse[slot0 + p]);
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) mx = fmaxf(mx, __shfl_xor(mx, o));
  float W = 0.f, o0 = 0.f, o1 = 0.f;
  for (int p = wave; p < np; p += 16) {
    float lse[4];
    float2 o[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int64_t slot = slot0 + min(p + 4 * u, np - 1);
      lse[u] = a.ws_lse[slot];
      o[u] = *reinterpret_cast<const float2*>(a.ws_o + slot * kHeadDim + 2 * lane);
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      // past the end: nothing, not 0 x the last partition's (infinite?) result
      const bool in = p + 4 * u < np;
      const float w = fast_exp2(lse[u] - mx);
      W += in ? w : 0.f;
      o0 = in ? fmaf(w, o[u].x, o0) : o0;
      o1 = in ? fmaf(w, o[u].y, o1) : o1;
    }
  }
  __shared__ float sw[4];
  __shared__ float2 so[4][64];
  so[wave][lane] = make_float2(o0, o1);
  if (lane == 0) sw[wave] = W;
  __syncthreads();
  if (wave) return;
#pragma unroll
  for (int w = 1; w < 4; ++w) {
    W += sw[w];
    o0 += so[w][lane].x;
    o1 += so[w][lane].y;
  }
  const float inv = 1.f / W;
  store_out2<DT>(a.out, (int64_t)b * a.out_seq_stride + (int64_t)hq * kHeadDim + 2 * lane, o0 * inv,
                 o1 * inv);
}

// ------------------------------------------------------------------ planning
struct DecodePlan {
  int32_t part_tokens;
  int32_t n_parts;
  size_t ws_bytes;
};

static DecodePlan plan_decode(int32_t n_seqs, int32_t hq, int32_t hkv, int32_t block_size,
                              int32_t max_blocks, int32_t max_context_len, int32_t part_tokens,
                              int32_t elem_bytes) {
  // tokens of one iteration of a workgroup: 16 rows x 8 in flight (fp32: 4)
  const int iter_tokens = elem_bytes == 4 ? 64 : 128;
  DecodePlan p;
  int64_t cap = (int64_t)max_blocks * block_size;
  if (max_context_len > 0 && max_context_len < cap) cap = max_context_len;
  if (cap < 1) cap = 1;
  int64_t part = part_tokens;
  if (part <= 0) {
    // Measured on MI355X (block 256, graph replay, us).  From 512 (sequence, KV
    // head) items and contexts up to 4096 tokens one workgroup per item needs no
    // reduction and is the fastest (64 x 1-2k at 8 KV heads 66.7 against 68.3-73
    // in partitions of 128-1024; 64 x 10-200 10.8 against 13.9-16.3), and up to
    // two iterations of tokens for any number (1 x 93: 4.9 against 6.2).  Else the
    // smallest partition, from one iteration up in whole iterations (parts of one
    // cost a whole one: 24 x 100-2063 in 128 24.6, 192 26.8, 256 24.1), that keeps
    // the tables' capacity within twelve workgroups per CU, sixteen in fp32 (about half
    // of them have tokens: 46 x 49-4548 GQA-4 in 384 92, 768 93, 2048 107; 93 x 77-2504
    // at 4 KV heads in 384 47.7, 1024 54.9; fp32, 40 x 577-1837 in 192 84, 512 105)
    // and the reduction at some 50 partitions (one of 30,000: 1024 25.1, 512 26.7,
    // 128 32.9; one of 25,000 at 4 KV heads: 512 17.5, 1024 23.6; 2 x 6-7k GQA-4: 256
    // 18.4, 128 20.2), twice that in fp32, whose rows are twice as long (one of
    // 20,000: 128 39.4, 256 40.7, 512 47.2).  At most 3072 (64 x 16k-32k GQA-4 over
    // four context draws: 75.4% of HBM peak against 73.8% for 2048, 75.1% for 2560,
    // 74.3% for 3584 and 72.5% for 4096).
    const int64_t items = (int64_t)n_seqs * hkv;
    const int64_t most_parts = elem_bytes == 4 ? 96 : 52, most_groups = elem_bytes == 4 ? 4096 : 3072;
    if ((items >= 512 && cap <= 4096) || cap <= 2 * iter_tokens) {
      part = cap;
    } else {
      for (int k : {1, 2, 3, 4, 6, 8, 12, 16, 24, 32, 48}) {
        part = std::min(k * iter_tokens, 3072);
        if (items * cdiv(cap, part) <= most_groups && cdiv(cap, part) <= most_parts) break;
      }
    }
  }
  if (part > cap) part = cap;
  p.part_tokens = (int32_t)part;
  p.n_parts = (int32_t)cdiv(cap, part);
  p.ws_bytes = p.n_parts > 1 ? (size_t)n_seqs * hq * p.n_parts * (kHeadDim + 1) * sizeof(float) : 0;
  return p;
}

template <Dt DT, int G, int U, int NEW>
static void launch_decode_p(const DecodeArgs& a, hipStream_t s) {
  const dim3 grid(a.hkv, a.n_parts, a.n_seqs);
  if (a.bs_shift >= 0)
    hipLaunchKernelGGL((decode_paged_kernel<DT, G, U, true, NEW>), grid, dim3(256), 0, s, a);
  else
    hipLaunchKernelGGL((decode_paged_kernel<DT, G, U, false, NEW>), grid, dim3(256), 0, s, a);
}

template <Dt DT, int G>
static void launch_decode_t(const DecodeArgs& a, hipStream_t s) {
  // Token rows in flight per DPP row: eight for bf16/fp16, four for fp32,
  // whose rows take twice the registers (at eight, the fp32 instances of
  // groups 1 and 2 spill under the 128-VGPR bound of four workgroups per
  // CU).  At bf16 group 8, eight rows (233 VGPRs, 2 workgroups per CU) beat
  // four (181) by 3% on 256 seqs x 1-2k at 64/8 heads (318.0 against
  // 328.2 us).
  constexpr int U = DT == Dt::FP32 ? 4 : 8;
  if (a.qw) {
    if constexpr (DT != Dt::FP32) launch_decode_p<DT, G, U, kQkv>(a, s);
  } else if (a.ws_cnt) {
    launch_decode_p<DT, G, U, kAppendMerge>(a, s);
  } else if (a.k_new) {
    launch_decode_p<DT, G, U, kAppend>(a, s);
  } else {
    launch_decode_p<DT, G, U, kNone>(a, s);
  }
  if (a.n_parts > 1 && a.ws_cnt == nullptr)
    hipLaunchKernelGGL((decode_reduce_kernel<DT>), dim3(a.hq, a.n_seqs), dim3(256), 0, s, a);
}

template <Dt DT>
static int launch_decode_g(const DecodeArgs& a, int g, hipStream_t s) {
  switch (g) {
    case 1: launch_decode_t<DT, 1>(a, s); break;
    case 2: launch_decode_t<DT, 2>(a, s); break;
    case 4: launch_decode_t<DT, 4>(a, s); break;
    case 8: launch_decode_t<DT, 8>(a, s); break;
    default: return AAC_ERR_UNSUPPORTED;
  }
  return AAC_OK;
}

}  // namespace aac

using namespace aac;

extern "C" size_t aac_decode_workspace_bytes(int32_t n_seqs, int32_t n_q_heads, int32_t n_kv_heads,
                                             int32_t head_dim, int32_t block_size,
                                             int32_t max_blocks_per_seq, int32_t max_context_len,
                                             int32_t partition_tokens) {
  (void)head_dim;
  if (n_seqs <= 0 || n_q_heads <= 0 || n_kv_heads <= 0 || block_size <= 0 || max_blocks_per_seq <= 0)
    return 0;
  // the element type is not known here: the larger of the two plans
  size_t most = 0;
  for (int es : {2, 4})
    most = std::max(most, plan_decode(n_seqs, n_q_heads, n_kv_heads, block_size, max_blocks_per_seq,
                                      max_context_len, partition_tokens, es).ws_bytes);
  return most;
}

// The new token of a step, when the launch appends it (DecodeArgs)
struct NewToken {
  const void *k = nullptr, *v = nullptr;
  int64_t k_stride = 0, v_stride = 0;
  void* counters = nullptr;  // [n_seqs, n_kv_heads] x 8 bytes, or null
  const void *qw = nullptr, *kw = nullptr, *cos = nullptr, *sin = nullptr;
  const int32_t* positions = nullptr;
  int32_t max_pos = 0;
  float eps = 0.f;
};

static int decode_common(const void* q, int64_t q_seq_stride, const void* k_cache,
                         const void* v_cache, int64_t num_blocks, int32_t block_size,
                         const int32_t* block_tables, int32_t max_blocks_per_seq,
                         const int32_t* lens, int32_t lens_add, int32_t n_seqs,
                         int32_t max_context_len, int32_t n_q_heads, int32_t n_kv_heads,
                         int32_t head_dim, float scale, void* out, int64_t out_seq_stride,
                         void* workspace, size_t workspace_bytes, int32_t partition_tokens,
                         int32_t dtype, hipStream_t stream, const NewToken& nt = {}) {
  if (n_seqs < 0 || n_q_heads <= 0 || n_kv_heads <= 0 || num_blocks <= 0 || block_size <= 0 ||
      max_blocks_per_seq <= 0 || q_seq_stride < 0 || out_seq_stride < 0)
    return AAC_ERR_INVALID_ARGUMENT;
  if (head_dim != kHeadDim) return AAC_ERR_UNSUPPORTED;
  if (n_q_heads % n_kv_heads) return AAC_ERR_SHAPE;
  if (n_seqs == 0) return AAC_OK;
  if (!q || !k_cache || !v_cache || !block_tables || !lens || !out) return AAC_ERR_INVALID_ARGUMENT;
  if (q_seq_stride < (int64_t)n_q_heads * head_dim || out_seq_stride < (int64_t)n_q_heads * head_dim)
    return AAC_ERR_SHAPE;
  int es;
  Dt dt;
  switch (dtype) {
    case AAC_DTYPE_BF16: es = 2; dt = Dt::BF16; break;
    case AAC_DTYPE_FP16: es = 2; dt = Dt::FP16; break;
    case AAC_DTYPE_FP32: es = 4; dt = Dt::FP32; break;
    default: return AAC_ERR_UNSUPPORTED;
  }
  if (((uintptr_t)q | (uintptr_t)k_cache | (uintptr_t)v_cache) % 16 ||
      (q_seq_stride * es) % 16 || (uintptr_t)out % 8 || (out_seq_stride * es) % 8)
    return AAC_ERR_MISALIGNED;
  const DecodePlan plan = plan_decode(n_seqs, n_q_heads, n_kv_heads, block_size,
                                      max_blocks_per_seq, max_context_len, partition_tokens, es);
  if (plan.ws_bytes) {
    if (!workspace || workspace_bytes < plan.ws_bytes) return AAC_ERR_WORKSPACE;
    if ((uintptr_t)workspace % 16) return AAC_ERR_MISALIGNED;
  }
  DecodeArgs a = {};
  a.q = q;
  a.q_seq_stride = q_seq_stride;
  a.k_cache = k_cache;
  a.v_cache = v_cache;
  a.num_blocks = num_blocks;
  a.block_size = block_size;
  a.block_tables = block_tables;
  a.max_blocks = max_blocks_per_seq;
  a.lens = lens;
  a.lens_add = lens_add;
  a.n_seqs = n_seqs;
  a.hq = n_q_heads;
  a.hkv = n_kv_heads;
  a.scale_log2 = scale * kLog2e;
  a.out = out;
  a.out_seq_stride = out_seq_stride;
  a.n_parts = plan.n_parts;
  a.part_tokens = plan.part_tokens;
  a.bs_shift = (block_size & (block_size - 1)) == 0 ? __builtin_ctz((unsigned)block_size) : -1;
  if (a.bs_shift < 0) {  // block_size >= 3 here
    const int l = 32 - __builtin_clz((unsigned)(block_size - 1));
    a.bs_magic = (uint64_t(1) << (31 + l)) / (uint64_t)block_size + 1;
    a.bs_mshift = 31 + l;
  } else {
    a.bs_magic = 0;
    a.bs_mshift = 0;
  }
  // Length order only without a split (split partitions are already uniform
  // work units), and not for contexts of a few iterations that are all resident
  // at once: finding the order costs every workgroup some 1.7 us (8 sequences of
  // 69-250 tokens 8.6 us with it, 6.9 without; 64 of 10-500 17.1 and 17.6, 100 of
  // 100-2000 82.5 and 100.1).
  a.lpt = plan.n_parts == 1 && n_seqs >= 2 && n_seqs <= kLptMaxSeqs &&
          (plan.part_tokens > 256 || (int64_t)n_seqs * n_kv_heads > 1024);
  a.lpt_max = max_context_len > 0
                  ? max_context_len
                  : (int32_t)std::min<int64_t>((int64_t)max_blocks_per_seq * block_size, INT32_MAX);
  if (plan.ws_bytes) {
    a.ws_o = reinterpret_cast<float*>(workspace);
    a.ws_lse = a.ws_o + (size_t)n_seqs * n_q_heads * plan.n_parts * kHeadDim;
    // With counters a small append call combines its partitions in its launch.
    // Writes past the L2s, the counting and the second read take the GPU longer than
    // a second launch from some 4 partitions on (24 sequences in 9 partitions 29.9 us
    // against 25.7), but a caller that launches each call itself is bound by its
    // launches (fp32, 4 sequences in 8 partitions: 15.3 us a call with the second
    // launch, 13.5 without).
    if (nt.counters && plan.n_parts <= 8 && (int64_t)n_seqs * n_kv_heads * plan.n_parts <= 512)
      a.ws_cnt = reinterpret_cast<unsigned long long*>(nt.counters);
  }
  a.k_new = nt.k;
  a.v_new = nt.v;
  a.k_new_stride = nt.k_stride;
  a.v_new_stride = nt.v_stride;
  a.qw = (const u16*)nt.qw;
  a.kw = (const u16*)nt.kw;
  a.cos = (const u16*)nt.cos;
  a.sin = (const u16*)nt.sin;
  a.positions = nt.positions;
  a.max_pos = nt.max_pos;
  a.eps = nt.eps;
  const int g = n_q_heads / n_kv_heads;
  int rc;
  switch (dt) {
    case Dt::BF16: rc = launch_decode_g<Dt::BF16>(a, g, stream); break;
    case Dt::FP16: rc = launch_decode_g<Dt::FP16>(a, g, stream); break;
    default: rc = launch_decode_g<Dt::FP32>(a, g, stream); break;
  }
  if (rc != AAC_OK) return rc;
  hipError_t e = hipGetLastError();
  return e == hipSuccess ? AAC_OK : (int)e;
}

extern "C" int aac_decode_paged(const void* q, int64_t q_seq_stride, const void* k_cache,
                                const void* v_cache, int64_t num_blocks, int32_t block_size,
                                const int32_t* block_tables, int32_t max_blocks_per_seq,
                                const int32_t* context_lens, int32_t n_seqs,
                                int32_t max_context_len, int32_t n_q_heads, int32_t n_kv_heads,
                                int32_t head_dim, float scale, void* out, int64_t out_seq_stride,
                                void* workspace, size_t workspace_bytes, int32_t partition_tokens,
                                int32_t dtype, void* stream) {
  return decode_common(q, q_seq_stride, k_cache, v_cache, num_blocks, block_size, block_tables,
                       max_blocks_per_seq, context_lens, 0, n_seqs, max_context_len, n_q_heads,
                       n_kv_heads, head_dim, scale, out, out_seq_stride, workspace,
                       workspace_bytes, partition_tokens, dtype, (hipStream_t)stream);
}

// ------------------------------------------------------------------ static scratch
// Split-K scratch of aac_decode_paged_noalloc: one array per GPU, held until
// the process ends.  In host code `scratch` names a host-side stand-in, not
// device memory; the array's device address on each GPU comes from
// hipGetSymbolAddress (looked up once per device, with that device current)
// and only that address is handed to the kernels.
static __device__ __align__(256) unsigned char scratch[AAC_DECODE_SCRATCH_BYTES];

static int scratch_address(void** out) {
  constexpr int kMaxDevices = 64;
  static std::mutex mu;
  static void* addr[kMaxDevices] = {};
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return (int)e;
  if (dev < 0 || dev >= kMaxDevices) return AAC_ERR_UNSUPPORTED;
  std::lock_guard<std::mutex> lock(mu);
  if (!addr[dev]) {
    void* p = nullptr;
    e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess) return (int)e;
    if (!p) return AAC_ERR_SCRATCH;
    addr[dev] = p;
  }
  *out = addr[dev];
  return AAC_OK;
}

extern "C" int aac_decode_paged_noalloc(const void* q, int64_t q_seq_stride, const void* k_cache,
                                        const void* v_cache, int64_t num_blocks, int32_t block_size,
                                        const int32_t* block_tables, int32_t max_blocks_per_seq,
                                        const int32_t* context_lens, int32_t n_seqs,
                                        int32_t max_context_len, int32_t n_q_heads,
                                        int32_t n_kv_heads, int32_t head_dim, float scale,
                                        void* out, int64_t out_seq_stride,
                                        int32_t partition_tokens, int32_t dtype, void* stream) {
  // the plan is host arithmetic: a call it does not fit is rejected before
  // the device is touched
  const size_t need = aac_decode_workspace_bytes(n_seqs, n_q_heads, n_kv_heads, head_dim,
                                                 block_size, max_blocks_per_seq, max_context_len,
                                                 partition_tokens);
  if (need > AAC_DECODE_SCRATCH_BYTES) return AAC_ERR_SCRATCH;
  void* ws = nullptr;
  if (need) {
    const int rc = scratch_address(&ws);
    if (rc != AAC_OK) return rc;
  }
  return decode_common(q, q_seq_stride, k_cache, v_cache, num_blocks, block_size, block_tables,
                       max_blocks_per_seq, context_lens, 0, n_seqs, max_context_len, n_q_heads,
                       n_kv_heads, head_dim, scale, out, out_seq_stride, ws,
                       need ? (size_t)AAC_DECODE_SCRATCH_BYTES : 0, partition_tokens, dtype,
                       (hipStream_t)stream);
}

extern "C" int aac_decode_append_merge_paged(
    const void* q, int64_t q_seq_stride, const void* k, const void* v, int64_t k_tok_stride,
    int64_t v_tok_stride, void* k_cache, void* v_cache, int64_t num_blocks, int32_t block_size,
    const int32_t* block_tables, int32_t max_blocks_per_seq, const int32_t* cache_seqlens,
    int32_t n_seqs, int32_t max_context_len, int32_t n_q_heads, int32_t n_kv_heads,
    int32_t head_dim, float scale, void* out, int64_t out_seq_stride, void* workspace,
    size_t workspace_bytes, void* counters, int32_t partition_tokens, int32_t dtype, void* stream) {
  if (head_dim != kHeadDim) return AAC_ERR_UNSUPPORTED;
  if ((uintptr_t)counters % 8) return AAC_ERR_MISALIGNED;
  // The append runs inside the attention launch when its rows suit the 16-byte
  // loads there, there are at most 64 of them, a lane each in the search for shared
  // blocks, and a partition has at most 64 blocks to search; anything else takes the
  // general append first (graph replay, one launch against two, us: 24 x 100-2063
  // 25.6 and 27.1, 64 x 10-500 16.0 and 17.4, 1 x 20,000 at 32/8 heads 24.7 and 25.9;
  // 256 x 1-2k 249.5 and 245.3; partitions of 192 blocks of 16, 37 x 15k 390 and 383).
  const int es = dtype == AAC_DTYPE_FP32 ? 4 : 2;
  const int g = n_kv_heads > 0 && n_q_heads > 0 && n_q_heads % n_kv_heads == 0 ? n_q_heads / n_kv_heads : 0;
  if (n_seqs > 0 && n_seqs <= 64 && (g == 1 || g == 2 || g == 4 || g == 8) && k && v && k_cache && v_cache &&
      block_tables && cache_seqlens && num_blocks > 0 && k_tok_stride >= (int64_t)n_kv_heads * head_dim &&
      v_tok_stride >= (int64_t)n_kv_heads * head_dim && ((uintptr_t)k | (uintptr_t)v) % 16 == 0 &&
      (k_tok_stride * es) % 16 == 0 && (v_tok_stride * es) % 16 == 0 && block_size > 0 &&
      max_blocks_per_seq > 0 &&
      plan_decode(n_seqs, n_q_heads, n_kv_heads, block_size, max_blocks_per_seq, max_context_len,
                  partition_tokens, es).part_tokens <= 64 * (int64_t)block_size) {
    NewToken nt;
    nt.k = k;
    nt.v = v;
    nt.k_stride = k_tok_stride;
    nt.v_stride = v_tok_stride;
    nt.counters = counters;
    return decode_common(q, q_seq_stride, k_cache, v_cache, num_blocks, block_size, block_tables,
                         max_blocks_per_seq, cache_seqlens, 1, n_seqs, max_context_len, n_q_heads,
                         n_kv_heads, head_dim, scale, out, out_seq_stride, workspace,
                         workspace_bytes, partition_tokens, dtype, (hipStream_t)stream, nt);
  }
  const int rc = aac_kv_append_paged(k, v, k_tok_stride, v_tok_stride, k_cache, v_cache, num_blocks,
                                     block_size, block_tables, max_blocks_per_seq, cache_seqlens,
                                     n_seqs, n_kv_heads, head_dim, dtype, stream);
  if (rc != AAC_OK) return rc;
  return decode_common(q, q_seq_stride, k_cache, v_cache, num_blocks, block_size, block_tables,
                       max_blocks_per_seq, cache_seqlens, 1, n_seqs, max_context_len, n_q_heads,
                       n_kv_heads, head_dim, scale, out, out_seq_stride, workspace,
                       workspace_bytes, partition_tokens, dtype, (hipStream_t)stream);
}

extern "C" int aac_decode_append_paged(const void* q, int64_t q_seq_stride, const void* k,
                                       const void* v, int64_t k_tok_stride, int64_t v_tok_stride,
                                       void* k_cache, void* v_cache, int64_t num_blocks,
                                       int32_t block_size, const int32_t* block_tables,
                                       int32_t max_blocks_per_seq, const int32_t* cache_seqlens,
                                       int32_t n_seqs, int32_t max_context_len, int32_t n_q_heads,
                                       int32_t n_kv_heads, int32_t head_dim, float scale, void* out,
                                       int64_t out_seq_stride, void* workspace,
                                       size_t workspace_bytes, int32_t partition_tokens,
                                       int32_t dtype, void* stream) {
  return aac_decode_append_merge_paged(q, q_seq_stride, k, v, k_tok_stride, v_tok_stride, k_cache,
                                       v_cache, num_blocks, block_size, block_tables,
                                       max_blocks_per_seq, cache_seqlens, n_seqs, max_context_len,
                                       n_q_heads, n_kv_heads, head_dim, scale, out, out_seq_stride,
                                       workspace, workspace_bytes, nullptr, partition_tokens, dtype,
                                       stream);
}

extern "C" int aac_decode_qkv_paged(
    const void* qkv, int64_t qkv_row_stride, const void* q_norm_weight, const void* k_norm_weight,
    float eps, const void* cos_table, const void* sin_table, int32_t max_position,
    const int32_t* positions, void* k_cache, void* v_cache, int64_t num_blocks, int32_t block_size,
    const int32_t* block_tables, int32_t max_blocks_per_seq, const int32_t* cache_seqlens,
    int32_t n_seqs, int32_t max_context_len, int32_t n_q_heads, int32_t n_kv_heads,
    int32_t head_dim, float scale, void* out, int64_t out_seq_stride, void* workspace,
    size_t workspace_bytes, int32_t partition_tokens, int32_t dtype, void* stream) {
  if (dtype != AAC_DTYPE_BF16 && dtype != AAC_DTYPE_FP16) return AAC_ERR_UNSUPPORTED;
  if (head_dim != kHeadDim) return AAC_ERR_UNSUPPORTED;
  if (n_seqs < 0 || n_q_heads <= 0 || n_kv_heads <= 0 || max_position <= 0) return AAC_ERR_INVALID_ARGUMENT;
  if (qkv_row_stride < (int64_t)(n_q_heads + 2 * n_kv_heads) * head_dim) return AAC_ERR_SHAPE;
  if (n_seqs == 0) return AAC_OK;
  if (!qkv || !q_norm_weight || !k_norm_weight || !cos_table || !sin_table || !positions)
    return AAC_ERR_INVALID_ARGUMENT;
  if (((uintptr_t)qkv | (uintptr_t)q_norm_weight | (uintptr_t)k_norm_weight | (uintptr_t)cos_table |
       (uintptr_t)sin_table) % 16 || qkv_row_stride % 8)
    return AAC_ERR_MISALIGNED;
  NewToken nt;
  nt.k = (const u16*)qkv + (int64_t)n_q_heads * kHeadDim;
  nt.v = (const u16*)qkv + (int64_t)(n_q_heads + n_kv_heads) * kHeadDim;
  nt.k_stride = nt.v_stride = qkv_row_stride;
  nt.qw = q_norm_weight;
  nt.kw = k_norm_weight;
  nt.cos = cos_table;
  nt.sin = sin_table;
  nt.positions = positions;
  nt.max_pos = max_position;
  nt.eps = eps;
  return decode_common(qkv, qkv_row_stride, k_cache, v_cache, num_blocks, block_size, block_tables,
                       max_blocks_per_seq, cache_seqlens, 1, n_seqs, max_context_len, n_q_heads,
                       n_kv_heads, head_dim, scale, out, out_seq_stride, workspace,
                       workspace_bytes, partition_tokens, dtype, (hipStream_t)stream, nt);
}
