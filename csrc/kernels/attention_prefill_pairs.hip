// Prefill attention of 64 rows a wave (attention_prefill_long.h), in pairs of half blocks; attention_prefill.hip chooses.
#include "attention_prefill_long.h"

int launch_prefill_pairs(DLI_LONG_ARGS) {
  return launch_rows<true>(out, out_stride, qkv, row_stride, cu_seqlens, num_seqs, max_seqlen, hq, hkv, scale_log2, ctx_lens, k_cache, v_cache,
                           block_tables, bt_stride, block_size, st);
}
