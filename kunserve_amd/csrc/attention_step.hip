// The attention stage of one layer of a step (LlamaOp.pforward,
// kunserve/worker.py:298-312) as one host call: the prologue (rotary
// embedding and append, or append alone), then the decode rows, then the
// prefill rows, all enqueued on the caller's stream. The step's arrays and
// plans are described once (kunserve_step) and shared by its layers; a layer
// passes only its tensors. Small decode steps are bound by the host's work
// between launches: through three separate calls from Python a layer of one
// row took 23 us of host time, its kernels 16.
#include "common.hpp"

using namespace kunserve;

extern "C" int kunserve_attention_step(const kunserve_step* step, int32_t layer,
                                       const kunserve_step_io* io, kunserve_stream_t stream) {
  clear_error();
  KSV_CHECK_ARG(step && io, "null step or tensors");
  kunserve_tensor3 q = io->q, out = io->out;
  DecodeFusion fusion;
  fusion.counters = step->counters_dev;
  fusion.num_counters = step->num_counters;
  int rc = KUNSERVE_OK;
  if (io->inv_freq_dev) {
    rc = kunserve_rope_append_kv(&step->pool, layer, &step->table, step->q_indptr_dev,
                                 step->num_tokens, &q, step->num_qo_heads, &io->k, &io->v,
                                 io->inv_freq_dev, io->interleave, stream);
  } else if (step->decode_appends && step->prefill_table.num_seqs == 0) {
    fusion.k_new = &io->k;
    fusion.v_new = &io->v;
  } else {
    rc = kunserve_append_kv(&step->pool, layer, &step->table, step->q_indptr_dev,
                            step->num_tokens, &io->k, &io->v, stream);
  }
  if (rc) return rc;
  if (step->decode_table.num_seqs > 0) {
    rc = paged_decode(&step->pool, layer, &step->decode_table, step->decode_q_token_dev, &q, &out,
                      step->num_qo_heads, step->sm_scale, step->decode_plan_dev,
                      &step->decode_info, step->workspace_dev, step->workspace_bytes, fusion,
                      stream);
    if (rc) return rc;
  }
  if (step->prefill_table.num_seqs > 0) {
    rc = paged_prefill(&step->pool, layer, &step->prefill_table, step->prefill_q_indptr_dev,
                       step->prefill_q_start_dev, &q, &out, step->num_qo_heads, step->sm_scale,
                       step->prefill_plan_dev, &step->prefill_info, step->workspace_dev,
                       step->workspace_bytes, step->prefill_counters_dev,
                       step->num_prefill_counters, stream);
    if (rc) return rc;
  }
  return KUNSERVE_OK;
}
