// The attention stage of one layer of a step (LlamaOp.pforward,
// kunserve/worker.py:298-312) as one host call: the prologue (rotary
// embedding and append, or append alone, which the attention launches take
// on where they can), then the decode rows, then the prefill rows, all
// enqueued on the caller's stream. The step's arrays and
// plans are described once (kunserve_step) and shared by its layers; a layer
// passes only its tensors. Small decode steps are bound by the host's work
// between launches: through three separate calls from Python a layer of one
// row took 23 us of host time, its kernels 16.
#include <algorithm>
#include <new>
#include <vector>

#include "common.hpp"

using namespace kunserve;

extern "C" int kunserve_tensors_overlap(const kunserve_tensor3* a, int32_t heads_a,
                                        const kunserve_tensor3* b, int32_t heads_b,
                                        int32_t num_tokens, int32_t head_dim) {
  clear_error();
  KSV_CHECK_ARG(a && b && heads_a >= 0 && heads_b >= 0 && num_tokens >= 0 && head_dim >= 0,
                "null tensor or negative size");
  if (heads_a == 0 || heads_b == 0 || num_tokens == 0 || head_dim == 0) return 0;
  // Bytes from `data` to the first element and past the last, strides of
  // either sign.
  struct Range { int64_t lo, hi; };
  auto range = [&](const kunserve_tensor3& t, int32_t heads) {
    const int64_t tok = int64_t(num_tokens - 1) * t.token_stride;
    const int64_t head = int64_t(heads - 1) * t.head_stride;
    const int64_t base = int64_t(reinterpret_cast<intptr_t>(t.data));
    return Range{base + 2 * (std::min<int64_t>(tok, 0) + std::min<int64_t>(head, 0)),
                 base + 2 * (std::max<int64_t>(tok, 0) + std::max<int64_t>(head, 0) + head_dim)};
  };
  const Range ra = range(*a, heads_a), rb = range(*b, heads_b);
  if (ra.hi <= rb.lo || rb.hi <= ra.lo) return 0;
  // Slices of the rows of one buffer (a QKV projection's): disjoint where they
  // are in one row.
  const int64_t row = 2 * a->token_stride;
  if (row <= 0 || a->token_stride != b->token_stride || a->head_stride < 0 || b->head_stride < 0)
    return 1;
  const int64_t wa = 2 * (int64_t(heads_a - 1) * a->head_stride + head_dim);
  const int64_t wb = 2 * (int64_t(heads_b - 1) * b->head_stride + head_dim);
  if (wa > row || wb > row) return 1;
  const int64_t at = ((ra.lo - rb.lo) % row + row) % row;   // a's start in b's row
  return at < wb || at + wa > row;
}

extern "C" int kunserve_attention_step(const kunserve_step* step, int32_t layer,
                                       const kunserve_step_io* io, kunserve_stream_t stream) {
  clear_error();
  KSV_CHECK_ARG(step && io, "null step or tensors");
  kunserve_tensor3 q = io->q, out = io->out;
  StepFusion decode, prefill;
  decode.counters = step->counters_dev;
  decode.num_counters = step->num_counters;
  prefill.counters = step->prefill_counters_dev;
  prefill.num_counters = step->num_prefill_counters;
  // Launches that append read k and v while other workgroups of theirs, or the
  // launch before them, write out: where out is in k's or v's memory, both are
  // first copied into their pages.
  auto out_overlaps_new = [&] {
    for (const kunserve_tensor3* t : {&io->k, &io->v})
      if (kunserve_tensors_overlap(&out, step->num_qo_heads, t, step->pool.num_kv_heads,
                                   step->num_tokens, step->pool.head_dim))
        return true;
    return false;
  };
  int rc = KUNSERVE_OK;
  if (io->inv_freq_dev) {
    rc = kunserve_rope_append_kv(&step->pool, layer, &step->table, step->q_indptr_dev,
                                 step->num_tokens, &q, step->num_qo_heads, &io->k, &io->v,
                                 io->inv_freq_dev, io->interleave, stream);
  } else if (step->appends && !out_overlaps_new()) {
    decode.k_new = prefill.k_new = &io->k;
    decode.v_new = prefill.v_new = &io->v;
  } else {
    rc = kunserve_append_kv(&step->pool, layer, &step->table, step->q_indptr_dev,
                            step->num_tokens, &io->k, &io->v, stream);
  }
  if (rc) return rc;
  if (step->decode_table.num_seqs > 0) {
    rc = paged_decode(&step->pool, layer, &step->decode_table, step->decode_q_token_dev, &q, &out,
                      step->num_qo_heads, step->sm_scale, step->decode_plan_dev,
                      &step->decode_info, step->workspace_dev, step->workspace_bytes, decode,
                      stream);
    if (rc) return rc;
  }
  if (step->prefill_table.num_seqs > 0) {
    rc = paged_prefill(&step->pool, layer, &step->prefill_table, step->prefill_q_indptr_dev,
                       step->prefill_q_start_dev, &q, &out, step->num_qo_heads, step->sm_scale,
                       step->prefill_plan_dev, &step->prefill_info, step->workspace_dev,
                       step->workspace_bytes, prefill, stream);
    if (rc) return rc;
  }
  return KUNSERVE_OK;
}

// A launch that appends its own rows must not write what another of its
// workgroups reads: the pages of a row's new tokens are in no other place of
// the table.
extern "C" int kunserve_new_pages_private(const int32_t* indptr_host, const int32_t* indices_host,
                                          const int32_t* q_indptr_host,
                                          const int32_t* kv_len_host, int32_t num_seqs,
                                          int32_t page_size, int64_t num_pages) {
  clear_error();
  KSV_CHECK_ARG(num_seqs >= 0 && page_size > 0 && num_pages > 0 && num_pages < (int64_t(1) << 31),
                "bad num_seqs, page_size or num_pages");
  KSV_CHECK_ARG(num_seqs == 0 || (indptr_host && indices_host && q_indptr_host && kv_len_host),
                "null table");
  try {
    // The pages of new tokens in a hash table, so that the cost is the step's and
    // not the pool's: linear probing, at most half full.
    int64_t count = 0;
    for (int32_t b = 0; b < num_seqs; ++b) {
      const int32_t n = q_indptr_host[b + 1] - q_indptr_host[b], kv = kv_len_host[b];
      if (n <= 0) continue;
      if (kv < n || (kv - 1) / page_size >= indptr_host[b + 1] - indptr_host[b]) return 0;
      count += (kv - 1) / page_size - (kv - n) / page_size + 1;
    }
    int bits = 4;
    while ((int64_t(1) << bits) < 2 * count) ++bits;
    struct Slot {
      int32_t page = -1;
      bool met = false;   // in the table
    };
    std::vector<Slot> slots(size_t(1) << bits);
    auto find = [&](int32_t p) -> Slot& {   // p's slot, or the free one it would take
      size_t i = (uint32_t(p) * 2654435769u) >> (32 - bits);
      while (slots[i].page >= 0 && slots[i].page != p) i = (i + 1) & (slots.size() - 1);
      return slots[i];
    };
    for (int32_t b = 0; b < num_seqs; ++b) {
      const int32_t n = q_indptr_host[b + 1] - q_indptr_host[b], kv = kv_len_host[b];
      if (n <= 0) continue;
      for (int32_t i = (kv - n) / page_size; i <= (kv - 1) / page_size; ++i) {
        const int32_t p = indices_host[indptr_host[b] + i];
        if (p < 0 || p >= num_pages) return 0;
        Slot& slot = find(p);
        if (slot.page == p) return 0;
        slot.page = p;
      }
    }
    for (int32_t i = num_seqs ? indptr_host[0] : 0, e = num_seqs ? indptr_host[num_seqs] : 0; i < e; ++i) {
      const int32_t p = indices_host[i];
      if (p < 0 || p >= num_pages) continue;
      Slot& slot = find(p);
      if (slot.page < 0) continue;
      if (slot.met) return 0;
      slot.met = true;
    }
  } catch (const std::bad_alloc&) {
    set_error("out of host memory");
    return KUNSERVE_ENOSPC;
  }
  return 1;
}
