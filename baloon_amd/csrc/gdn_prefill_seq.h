// gdn_prefill_seq.h -- the one-workgroup-per-(sequence, v head) prefill (gdn_prefill_seq.hip).
#pragma once
#include "gdn_chunk.h"

namespace ixg {

constexpr int kSeqThreads = 512;

// Workgroups (of kSeqThreads) per sequence.
long long seq_workgroups(const Layer& L);

// Prefill of every sequence of the batch that has no chunk in the plan's chunk table: states, outputs
// (p.o, p.o_bf16 from the batch's first token on; the gated norm's when gate is given) and conv
// histories. Two launches on s; p.ws.order lists the sequences.
void launch_prefill_seq(const PrefillParams& p, const OutGate* gate, bool silu, hipStream_t s);

}  // namespace ixg
