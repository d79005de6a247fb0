// The four-wave, two-columns-per-wave prefill kernel (prefill_wide.hip),
// launched by the varlen prefill entry points in prefill.hip.
#pragma once

#include "prefill_common.h"

namespace aac {

// Whether the wide kernel takes a call: GQA groups 2, 4, 8 and a positive scale, in
// fp16 only where it is the faster one.
bool prefill_wide_takes(int g, float scale, bool f16, bool store, int n_seqs, int hkv, int max_q, int n_cu);

// Launch on the persistent grid (min(items, n_cu) workgroups).  a.n_qblocks
// is set by the launcher.  store: also write the K/V rows to the KV cache
// through a.slots (causal self-attention only).
int prefill_wide_launch(const pf::Args& a, int g, bool causal, bool store, bool f16, int max_q,
                        int n_cu, hipStream_t st);

}  // namespace aac
