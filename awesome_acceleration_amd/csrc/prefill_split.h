// The prefill kernel for calls of few or short segments (prefill_split.hip),
// launched by the varlen prefill entry points in prefill.hip.
#pragma once

#include "prefill_common.h"

namespace aac {

// The key slices the call runs with in this kernel, or 0 where another kernel
// is the faster one (see prefill_split.hip for where the lines lie).  idle_pieces:
// the other one is the eight-wave kernel with two pieces per item, all on CUs of
// their own.
int prefill_split_slices(int g, float scale, bool f16, int n_seqs, int hkv, int max_q, int max_k, bool causal,
                         int n_cu, bool idle_pieces);

// a.n_qblocks is set by the launcher.  store: also write the K/V rows to the
// KV cache through a.slots (causal self-attention only).
int prefill_split_launch(const pf::Args& a, int slices, int g, bool causal, bool store, bool f16, int max_q,
                         hipStream_t st);

}  // namespace aac
