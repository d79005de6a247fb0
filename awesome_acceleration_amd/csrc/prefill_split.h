// The prefill kernel for calls of few queries (prefill_split.hip), launched by
// the varlen prefill entry points in prefill.hip.
#pragma once

#include "prefill_common.h"

namespace aac {

// Whether the call goes to this kernel (see prefill_split.hip for where the
// line lies).
bool prefill_split_takes(int g, float scale, int n_seqs, int hkv, int max_q, int max_k, int n_cu);

// a.n_qblocks is set by the launcher.  store: also write the K/V rows to the
// KV cache through a.slots (causal self-attention only).
int prefill_split_launch(const pf::Args& a, int g, bool causal, bool store, bool f16, int max_q, hipStream_t st);

}  // namespace aac
