// Paged decode attention (q_len == 1 rows of LlamaOp.pforward,
// kunserve/worker.py:298-312; head counts kunserve/models.py:55-56, page
// size kunserve/models.py:57).
//
// HBM-bound: every K/V byte of a sequence is read exactly once per layer.
// Design for gfx950 (wave64, 256 CUs):
//  * The host plan cuts every sequence into partitions of part_tokens and
//    deals them, longest first, to 8 XCD lanes by estimated finish time;
//    the grid is lane entries x head groups, each XCD running all head
//    groups of one item at a time, so mixed context lengths still give an
//    even, device-filling grid that is dispatched longest item first on
//    every XCD.
//  * A workgroup (4 waves) owns one partition of one KV head and all
//    `G` query heads that share it (GQA: one KV read serves G heads).
//  * The partition's slice of the page table is staged in LDS once; after
//    that each K/V access is one 16-byte load per lane. A wave reads 1 KiB
//    of K and 1 KiB of V per load instruction (4 tokens x 256 B for
//    head_dim 128), four of each in flight per 16-token chunk.
//  * fp16 and bf16 pools (kernels are templates over the element type).
//  * Q.K uses v_dot2_f32_f16 / _bf16 and a DPP butterfly inside each 16-lane row;
//    the softmax is an online (running max) softmax in fp32 kept per row,
//    merged across rows with shuffles and across waves through LDS.
//  * Sequences longer than one partition write fp32 partial results with
//    their log-sum-exp (base 2). The last workgroup of a row to finish combines
//    them where the caller gives counters (decode_finish), else a small merge
//    kernel does.
//  * With the step's new k and v the launch appends them (append_row).
#include <algorithm>
#include <cmath>
#include <mutex>
#include <vector>

#include "common.hpp"

namespace kunserve {
namespace {

constexpr int kThreads = 256;
constexpr int kWaves = kThreads / kWave;
constexpr int kLoadsPerChunk = 4;        // 16-byte loads per lane per chunk (K and V each)
constexpr int kMaxPartTokens = 4096;
constexpr int kMinPageSize = 4;
constexpr int kMaxPartPages = kMaxPartTokens / kMinPageSize + 2;
constexpr int kMinPartTokens = 256;
constexpr int kMinAutoPartTokens = 128;  // shortest the grouped plan chooses by itself: a step of every wave
constexpr int kMaxCountedParts = 8;      // partitions a counting workgroup combines (one batch)
constexpr int kMaxGroup = 16;            // query heads of one workgroup (MFMA columns)
constexpr int kXcds = 8;                 // MI355X: workgroup b runs on XCD b % 8
constexpr float kNegBig = -1.0e30f;      // finite "minus infinity" for running maxima

// Source of the loads of lanes past a partition's end and of bad page ids:
// one zero K/V row (head_dim <= 256), so loaded data is never masked.
__device__ __attribute__((aligned(16))) f16 g_zero_row[256];

struct DecodeArgs {
  const int32_t* q_token;   // null, or [num_seqs]: token of q and out of each sequence
  const f16* q;
  int64_t q_tok, q_head;
  f16* out;
  int64_t o_tok, o_head;
  const f16* k;             // pool K at the layer
  const f16* v;
  int64_t page_stride, head_stride, token_stride;
  int32_t num_pages;
  int32_t page_shift;
  const int32_t* indptr;
  const int32_t* indices;
  const int32_t* kv_len;    // for k_new and counters (null without them)
  // The step's new K/V rows of the same tokens as q, or null: they are then
  // in the pages already. With them the launch appends as well: the new
  // token's row (position kv_len - 1) is read from here instead of from its
  // page, and the workgroup that reads it writes it there. No other row's
  // table holds that page (the caller checks), so no other workgroup
  // reads what this launch writes.
  const f16* k_new;
  const f16* v_new;
  int64_t kn_tok, kn_head, vn_tok, vn_head;
  // null, or one zeroed counter per (first slot of a split row, head group):
  // the last of the row's workgroups to finish combines the partials.
  int32_t* counters;
  int32_t part_tokens;
  const int32_t* work;      // [num_work][4]: seq (-1: padding), tok_begin, tok_end, slot (-1: direct)
  float* part_o;            // [slots][num_qo_heads][D]
  float* part_lse;          // [slots][num_qo_heads]
  int32_t num_qo_heads;
  int32_t group;            // G: query heads of a workgroup
  int32_t head_groups;      // num_qo_heads / G
  int32_t num_work;         // work items of the plan
  int32_t ratio;            // num_qo_heads / num_kv_heads
  float scale_log2;         // sm_scale * log2(e)
};

// Work record and head group of workgroup b. The hardware hands workgroup
// b to XCD b % 8. The plan's records are 8 lanes interleaved (record
// 8 r + x is entry r of XCD x's lane), and XCD x runs every head group of
// its lane's entries in order, an entry's head groups back to back, so the
// pages an XCD reads at a time are those of its own few items (measured
// 1-2% faster than spreading each item's head groups over all XCDs). A
// lane's padding records (seq -1) end the workgroup at once.
__device__ __forceinline__ bool decode_work(const DecodeArgs& a, int& item, int& hg) {
  const int b = int(blockIdx.x);
  const int j = b >> 3;
  const int local = j / a.head_groups;
  hg = j - local * a.head_groups;
  item = 8 * local + (b & 7);
  return item < a.num_work;
}

// Where an item's new K/V row is: its position (-1: not in this launch's
// care) and its distance in elements from the KV head's base in the pool, so
// that a lane's load address takes one select of two offsets.
struct NewRow {
  int pos;
  int64_t k, v;
};
__device__ __forceinline__ NewRow new_row(const DecodeArgs& a, int seq, int tok, int hkv) {
  if (!a.k_new) return {-1, 0, 0};
  auto distance = [&](const f16* row, const f16* pool) {   // both 16-byte aligned
    return (reinterpret_cast<intptr_t>(row) - reinterpret_cast<intptr_t>(pool + int64_t(hkv) * a.head_stride)) / 2;
  };
  return {a.kv_len[seq] - 1,
          distance(a.k_new + int64_t(tok) * a.kn_tok + int64_t(hkv) * a.kn_head, a.k),
          distance(a.v_new + int64_t(tok) * a.vn_tok + int64_t(hkv) * a.vn_head, a.v)};
}
// Writes the new row into its page (`page`, -1: outside the pool), by the
// workgroup of the KV head's first query heads whose partition holds it.
template <int D>
__device__ __forceinline__ void append_row(const DecodeArgs& a, const NewRow& nr, int page,
                                           int hkv) {
  constexpr int CH = D / 8;
  const int tid = threadIdx.x;
  if (page < 0 || tid >= 2 * CH) return;
  const int c = tid % CH;
  const int64_t off = int64_t(page) * a.page_stride +
                      int64_t(nr.pos & ((1 << a.page_shift) - 1)) * a.token_stride;
  const bool v = tid >= CH;
  f16* base = const_cast<f16*>(v ? a.v : a.k) + int64_t(hkv) * a.head_stride + 8 * c;
  store_f16x8(base + off, load_f16x8(base + (v ? nr.v : nr.k)));
}

__device__ __forceinline__ void store_agent(float* p, float x, float y) {
  const uint64_t w = uint64_t(uint32_t(f32_to_bits(x))) | uint64_t(uint32_t(f32_to_bits(y))) << 32;
  __hip_atomic_store(reinterpret_cast<uint64_t*>(p), w, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Writes a workgroup's result, `result(g, d, x, y, lse)` giving head g's dims
// d, d + 1 and log-sum-exp (base 2): to out (slot -1), or as the partial of
// `slot`. With counters, the last workgroup of the row and head group to
// finish then combines the row's partials, in partition order, and no merge
// launch follows (about 3 us and the gap before it). A release/acquire pair
// at agent scope would write back and invalidate the XCD's whole L2 once per
// workgroup (10 times the launch's time). Instead the partials themselves are
// agent-scope atomic stores and loads, which do not stay in an L2: every
// wave waits for its stores (vmcnt counts stores on this part), the
// workgroup meets at a barrier, and only then is it counted.
template <typename T, int D, int THREADS, typename F>
__device__ __forceinline__ void decode_finish(const DecodeArgs& a, int seq, int tok, int tb,
                                              int slot, int hq0, int hg, int G, F result) {
  __shared__ int s_last;
  const int tid = threadIdx.x;
  const int pairs = G * (D / 2);
  auto write_out = [&](int g, int d, float x, float y) {
    T* op = reinterpret_cast<T*>(a.out) + int64_t(tok) * a.o_tok + int64_t(hq0 + g) * a.o_head + d;
    op[0] = T(x);
    op[1] = T(y);
  };
  for (int idx = tid; idx < pairs; idx += THREADS) {
    const int g = idx / (D / 2), d = 2 * (idx % (D / 2));
    float x, y, lse;
    result(g, d, x, y, lse);
    if (slot < 0) {
      write_out(g, d, x, y);
      continue;
    }
    const int64_t row = int64_t(slot) * a.num_qo_heads + hq0 + g;
    float* po = a.part_o + row * D + d;
    if (a.counters) {
      store_agent(po, x, y);
      if (d == 0)
        __hip_atomic_store(a.part_lse + row, lse, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    } else {
      po[0] = x;
      po[1] = y;
      if (d == 0) a.part_lse[row] = lse;
    }
  }
  if (slot < 0 || !a.counters) return;
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  const int s0 = slot - tb / a.part_tokens;   // the row's first slot
  const int n = (a.kv_len[seq] + a.part_tokens - 1) / a.part_tokens;
  if (tid == 0) {
    int32_t* counter = a.counters + int64_t(s0) * a.head_groups + hg;
    const int before = __hip_atomic_fetch_add(counter, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    s_last = before == n - 1;
    if (before == n - 1)   // zero again for the next layer
      __hip_atomic_store(counter, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  __syncthreads();   // also keeps the compiler from moving the loads below before the count
  if (!s_last) return;
  for (int idx = tid; idx < pairs; idx += THREADS) {
    const int g = idx / (D / 2), d = 2 * (idx % (D / 2));
    const int64_t row0 = int64_t(s0) * a.num_qo_heads + hq0 + g;
    constexpr int kBatch = 8;   // partials read together, so their latencies overlap
    float mx = -INFINITY, wsum = 0.f, x = 0.f, y = 0.f;
    for (int j = 0; j < n; j += kBatch) {
      float lse[kBatch];
      uint64_t po[kBatch];
#pragma unroll
      for (int u = 0; u < kBatch; ++u) {
        const int64_t row = row0 + int64_t(min(j + u, n - 1)) * a.num_qo_heads;
        lse[u] = __hip_atomic_load(a.part_lse + row, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        po[u] = __hip_atomic_load(reinterpret_cast<const uint64_t*>(a.part_o + row * D + d),
                                  __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
      float m2 = mx;
#pragma unroll
      for (int u = 0; u < kBatch; ++u) m2 = j + u < n ? fmaxf(m2, lse[u]) : m2;
      if (m2 == -INFINITY) continue;
      const float keep = fast_exp2(mx - m2);
      mx = m2;
      wsum *= keep;
      x *= keep;
      y *= keep;
#pragma unroll
      for (int u = 0; u < kBatch; ++u) {
        if (j + u >= n) break;   // uniform: the last partial again, of no weight (0 x inf)
        const float w = fast_exp2(lse[u] - m2);
        wsum += w;
        x = fmaf(w, bits_to_f32(int(uint32_t(po[u]))), x);
        y = fmaf(w, bits_to_f32(int(uint32_t(po[u] >> 32))), y);
      }
    }
    const float inv = wsum > 0.f ? 1.f / wsum : 0.f;
    write_out(g, d, x * inv, y * inv);
  }
}

// Waves per SIMD the VALU kernel's registers are held to (each 4 waves a CU
// fewer costs bandwidth).
template <typename T, int G>
constexpr int valu_waves() { return G == 1 ? (__is_same(T, f16) ? 5 : 4) : G == 2 ? 4 : 3; }

template <typename T, int D, int G>
__global__ __launch_bounds__(kThreads, (valu_waves<T, G>())) void paged_decode_kernel(DecodeArgs a) {
  typedef typename Vec<T>::v8 V8;
  constexpr int LPT = D / 8;            // lanes per token row (16 for D = 128)
  constexpr int TPL = kWave / LPT;      // tokens per load instruction (4)
  constexpr int CHUNK = TPL * kLoadsPerChunk;  // tokens per wave iteration (16)

  __shared__ int s_pages[kMaxPartPages];
  __shared__ float s_m[kWaves][G];
  __shared__ float s_l[kWaves][G];
  __shared__ float s_acc[kWaves][G][D];

  const int tid = threadIdx.x;
  const int lane = tid & (kWave - 1);
  const int wave = tid >> 6;
  const int row = lane / LPT;
  const int col = lane % LPT;

  int item, hg;
  if (!decode_work(a, item, hg)) return;   // padding workgroup (uniform: no barrier reached)
  const int32_t* w = a.work + 4 * item;
  const int seq = w[0], tb = w[1], te = w[2], slot = w[3];
  if (seq < 0) return;   // a lane's padding record (uniform: no barrier reached)
  const int tok = a.q_token ? a.q_token[seq] : seq;   // q / out token of the sequence
  const int hq0 = hg * G;
  const int hkv = hq0 / a.ratio;
  const int page_mask = (1 << a.page_shift) - 1;

  // Stage this partition's page ids; invalid ids become -1 (masked).
  const int pb = tb >> a.page_shift;
  const int np = te > tb ? ((te - 1) >> a.page_shift) + 1 - pb : 0;
  const int32_t* seq_pages = a.indices + a.indptr[seq];
  for (int i = tid; i < np; i += kThreads) {
    const int p = seq_pages[pb + i];
    s_pages[i] = (p >= 0 && p < a.num_pages) ? p : -1;
  }

  V8 qv[G];
#pragma unroll
  for (int g = 0; g < G; ++g)
    qv[g] = load_v8<T>(a.q + int64_t(tok) * a.q_tok + int64_t(hq0 + g) * a.q_head + col * 8);

  float m[G], l[G], acc[G][8];
#pragma unroll
  for (int g = 0; g < G; ++g) {
    m[g] = kNegBig;
    l[g] = 0.f;
#pragma unroll
    for (int j = 0; j < 8; ++j) acc[g][j] = 0.f;
  }
  __syncthreads();

  const NewRow nr = new_row(a, seq, tok, hkv);
  if (nr.pos >= tb && nr.pos < te && hq0 % a.ratio == 0)
    append_row<D>(a, nr, s_pages[(nr.pos >> a.page_shift) - pb], hkv);
  const f16* kb = a.k + int64_t(hkv) * a.head_stride + col * 8;
  const f16* vb = a.v + int64_t(hkv) * a.head_stride + col * 8;
  const int nchunks = (te - tb + CHUNK - 1) / CHUNK;

  // One chunk = kLoadsPerChunk token rows per lane, K and V. Loads are
  // non-temporal: every K/V byte is read once, so it should not displace
  // the page table and q in the caches.
  struct Chunk {
    V8 k[kLoadsPerChunk], v[kLoadsPerChunk];
    bool ok[kLoadsPerChunk];
  };
  // Loads are issued unconditionally (lanes past the partition read the
  // cache-resident zero row): with no branch around them and no use of the
  // data until it is consumed, the compiler waits for the current chunk
  // while the next chunk's loads stay in flight.
  auto load_chunk = [&](int c, Chunk& ch) {
    const int t0 = tb + c * CHUNK;
#pragma unroll
    for (int i = 0; i < kLoadsPerChunk; ++i) {
      const int t = t0 + i * TPL + row;
      const int pi = min((t >> a.page_shift) - pb, kMaxPartPages - 1);
      const int p = (c < nchunks && t < te) ? s_pages[pi] : -1;
      ch.ok[i] = p >= 0;
      const int64_t off = int64_t(max(p, 0)) * a.page_stride + int64_t(t & page_mask) * a.token_stride;
      ch.k[i] = load_v8_nt<T>(ch.ok[i] ? kb + (t == nr.pos ? nr.k : off) : g_zero_row + col * 8);
      ch.v[i] = load_v8_nt<T>(ch.ok[i] ? vb + (t == nr.pos ? nr.v : off) : g_zero_row + col * 8);
    }
  };
  auto consume = [&](const Chunk& ch) {
    float vf[kLoadsPerChunk][8];
#pragma unroll
    for (int i = 0; i < kLoadsPerChunk; ++i)
#pragma unroll
      for (int j = 0; j < 8; ++j) vf[i][j] = float(ch.v[i][j]);
#pragma unroll
    for (int g = 0; g < G; ++g) {
      float s[kLoadsPerChunk];
      float mx = m[g];
#pragma unroll
      for (int i = 0; i < kLoadsPerChunk; ++i) {
        s[i] = group_sum<LPT>(dot8(qv[g], ch.k[i], 0.f)) * a.scale_log2;
        s[i] = ch.ok[i] ? s[i] : -INFINITY;
        mx = fmaxf(mx, s[i]);
      }
      const float alpha = fast_exp2(m[g] - mx);
      m[g] = mx;
      float p[kLoadsPerChunk];
      float ps = 0.f;
#pragma unroll
      for (int i = 0; i < kLoadsPerChunk; ++i) {
        p[i] = fast_exp2(s[i] - mx);
        ps += p[i];
      }
      l[g] = l[g] * alpha + ps;
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        float x = acc[g][j] * alpha;
#pragma unroll
        for (int i = 0; i < kLoadsPerChunk; ++i) x = fmaf(p[i], vf[i][j], x);
        acc[g][j] = x;
      }
    }
  };

  // Software pipeline over this wave's chunks (wave, wave + 4, ...): the
  // loads of the next chunk are in flight while the current one is reduced.
  if (wave < nchunks) {
    Chunk c0, c1;
    int c = wave;
    load_chunk(c, c0);
    while (true) {
      load_chunk(c + kWaves, c1);
      consume(c0);
      c += kWaves;
      if (c >= nchunks) break;
      load_chunk(c + kWaves, c0);
      consume(c1);
      c += kWaves;
      if (c >= nchunks) break;
    }
  }

  // Merge the TPL rows of each wave (lanes col, col+LPT, ...).
#pragma unroll
  for (int off = LPT; off < kWave; off <<= 1) {
#pragma unroll
    for (int g = 0; g < G; ++g) {
      const float m2 = __shfl_xor(m[g], off);
      const float l2 = __shfl_xor(l[g], off);
      const float mx = fmaxf(m[g], m2);
      const float f1 = fast_exp2(m[g] - mx), f2 = fast_exp2(m2 - mx);
      m[g] = mx;
      l[g] = l[g] * f1 + l2 * f2;
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const float a2 = __shfl_xor(acc[g][j], off);
        acc[g][j] = acc[g][j] * f1 + a2 * f2;
      }
    }
  }
  if (row == 0) {
#pragma unroll
    for (int g = 0; g < G; ++g) {
      if (col == 0) {
        s_m[wave][g] = m[g];
        s_l[wave][g] = l[g];
      }
#pragma unroll
      for (int j = 0; j < 8; ++j) s_acc[wave][g][col * 8 + j] = acc[g][j];
    }
  }
  __syncthreads();

  // Merge the waves and write the output (direct) or a partial (split).
  decode_finish<T, D, kThreads>(a, seq, tok, tb, slot, hq0, hg, G,
                                [&](int g, int d, float& x, float& y, float& lse) {
    float mx = kNegBig;
#pragma unroll
    for (int wv = 0; wv < kWaves; ++wv) mx = fmaxf(mx, s_m[wv][g]);
    float lsum = 0.f;
    x = y = 0.f;
#pragma unroll
    for (int wv = 0; wv < kWaves; ++wv) {
      const float f = fast_exp2(s_m[wv][g] - mx);
      lsum += s_l[wv][g] * f;
      x += s_acc[wv][g][d] * f;
      y += s_acc[wv][g][d + 1] * f;
    }
    x = lsum > 0.f ? x / lsum : 0.f;
    y = lsum > 0.f ? y / lsum : 0.f;
    lse = lsum > 0.f ? mx + __log2f(lsum) : -INFINITY;
  });
}

// GQA decode on MFMA: every group of 2 to 16 query heads that share a KV head
// (at head_dim 64, 128 and 256).
// With G query heads sharing each K/V byte the VALU form above needs ~G
// dot products and G x 8 FMAs per token row and lane, which caps it below
// the HBM rate from G = 3 on, and it has only groups that are powers of two:
// at a ratio of 3 or 5 it would read K and V once per query head. Here both
// contractions run on 16x16x32 MFMAs with the heads as the 16 columns, so
// one workgroup serves any group and K/V is read once.
//  * K and V are read exactly as in the VALU kernel (each load instruction
//    covers whole token rows, 1 KiB contiguous per wave: measured ~15%
//    more bandwidth than reading MFMA operands straight from memory). A step
//    is 8 loads of K and of V per lane: 8 tokens x one 16-byte chunk.
//  * S^T[16 tokens x 16 heads] = K . Q^T: K goes through a per-wave LDS
//    block, row-major with the 16-byte chunk index XORed with token bits
//    (DecodeTile::swz), and comes back as the A operand (ds_read_b128); B
//    operand = Q^T (head lane%16, zero for lanes >= G). Which token is which
//    tile row is free, and chosen so that lane group tg of the result holds
//    the 8 tokens whose V rows lane group tg loaded.
//  * O^T[dims x 16 heads] += V^T . P^T without LDS: a lane's 8 tokens x 8
//    dims are transposed in registers (one v_perm per result dword), and
//    MFMA e takes dim 8 c + e of chunk c as its row. P^T is the S^T
//    accumulator itself in 16 bits. (Through LDS with 16-bit reads, 64 per
//    step, one 777-token row by one workgroup took 22.7 us; 15.9 so.)
//  * At head_dim 64 lanes j and j + 8 hold the same chunk of even and odd
//    tokens, so two MFMAs, each with its tokens' P, fill two accumulators of
//    which a lane group uses one; at 256 lane groups 2 g and 2 g + 1 hold
//    the two halves of the row of the same tokens, so two MFMAs take P
//    with the other half's groups zeroed, and every score is formed twice.
//    Twice the MFMAs of head_dim 128 per byte, still hidden by the loads.
//  * The probabilities go in as two 16-bit terms, the rounded value and the
//    rounded remainder: 22 significant bits in fp16 and 16 in bf16 where the
//    VALU kernel has 24, which the sums see (2^-17 of a term in bf16) and the
//    rounded output does not: over 108 combinations of dtype, head_dim, 1 to 16
//    heads per KV head and flat to peaked rows its error against 64 bits is at
//    most 0.01% above that of the kernels that served the groups before
//    (2.1e-4 in fp16, 1.65e-3 in bf16; one bf16 term had 2.15e-3).
//  * Infinite and NaN values in V do not survive the two terms; a wave that
//    meets one does its tokens again (wave_rows).
//  * Online softmax per head column in fp32 with a lazy running max, merged
//    across waves through LDS; partial results as in the VALU kernel.
template <int D>
struct DecodeTile {
  static constexpr int CH = D / 8;            // 16-byte chunks per token row
  static constexpr int TPL = kWave / CH;      // token rows per load instruction
  static constexpr int LOADS = 8;             // loads per lane per step (K and V each)
  static constexpr int STEP = TPL * LOADS;    // tokens per wave iteration
  static constexpr int PAIRS = D == 64 ? 2 : 1;   // pairs of 16-token score tiles per step
  static constexpr int ACCS = D == 128 ? 1 : 2;   // accumulator sets of 8
  // Step token of element i (0..7) of lane group g, score pair p.
  static __device__ __forceinline__ int token(int i, int g, int p) {
    return D == 64 ? 8 * i + 2 * g + p : D == 128 ? 4 * i + g : 2 * i + (g >> 1);
  }
  // XOR of token t's chunk index in the LDS block: the 8 rows that 8
  // consecutive lanes read differ in it.
  static __device__ __forceinline__ int swz(int t) {
    return D == 64 ? ((t >> 3) & 3) | ((t & 2) << 1) : D == 128 ? t & 15 : t & 7;
  }
};

// Maximum and sum over the four 16-lane groups.
__device__ __forceinline__ float groups_max(float x) {
  const auto a = __builtin_amdgcn_permlane16_swap(f32_to_bits(x), f32_to_bits(x), false, false);
  x = fmaxf(bits_to_f32(a[0]), bits_to_f32(a[1]));
  const auto b = __builtin_amdgcn_permlane32_swap(f32_to_bits(x), f32_to_bits(x), false, false);
  return fmaxf(bits_to_f32(b[0]), bits_to_f32(b[1]));
}

// One head's attention over the tokens of a wave's steps, in fp32 on the vector
// units and a load at a time: what the MFMA kernel falls back to for values
// that its products do not carry. Lane (row lane / CH, chunk lane % CH) holds
// dims 8 chunk .. + 7 in acc, the same in every row after the merge; kb and vb
// point at the lane's chunk.
template <typename T, int D, int W>
__device__ __forceinline__ void wave_rows(const DecodeArgs& a, typename Vec<T>::v8 q, const f16* kb,
                                          const f16* vb, int tb, int te, const int* s_pages,
                                          const NewRow& nr, float& m, float& l, float (&acc)[8]) {
  typedef DecodeTile<D> L;
  const int lane = threadIdx.x & (kWave - 1);
  const int wave = threadIdx.x >> 6;
  m = kNegBig;
  l = 0.f;
#pragma unroll
  for (int e = 0; e < 8; ++e) acc[e] = 0.f;
  for (int t0 = tb + wave * L::STEP; t0 < te; t0 += W * L::STEP)
#pragma unroll 1
    for (int i = 0; i < L::LOADS; ++i) {
      const int t = t0 + L::TPL * i + lane / L::CH;
      const int p = t < te ? s_pages[(t >> a.page_shift) - (tb >> a.page_shift)] : -1;
      const int64_t off = int64_t(max(p, 0)) * a.page_stride +
                          int64_t(t & ((1 << a.page_shift) - 1)) * a.token_stride;
      const f16* zero = g_zero_row + 8 * (lane % L::CH);
      const auto k = load_v8<T>(p >= 0 ? kb + (t == nr.pos ? nr.k : off) : zero);
      const auto v = load_v8<T>(p >= 0 ? vb + (t == nr.pos ? nr.v : off) : zero);
      float s = group_sum<L::CH>(dot8(q, k, 0.f)) * a.scale_log2;
      s = p >= 0 ? s : -INFINITY;
      const float mx = fmaxf(m, s);
      const float alpha = fast_exp2(m - mx), pr = fast_exp2(s - mx);
      m = mx;
      l = fmaf(l, alpha, pr);
#pragma unroll
      for (int e = 0; e < 8; ++e) acc[e] = fmaf(pr, float(v[e]), acc[e] * alpha);
    }
#pragma unroll
  for (int off = L::CH; off < kWave; off <<= 1) {
    const float m2 = __shfl_xor(m, off), l2 = __shfl_xor(l, off);
    const float mx = fmaxf(m, m2);
    const float f1 = fast_exp2(m - mx), f2 = fast_exp2(m2 - mx);
    m = mx;
    l = l * f1 + l2 * f2;
#pragma unroll
    for (int e = 0; e < 8; ++e) acc[e] = acc[e] * f1 + __shfl_xor(acc[e], off) * f2;
  }
}

template <typename T, int D, int W>
__global__ __launch_bounds__(W * kWave) __attribute__((amdgpu_waves_per_eu(2)))
void paged_decode_mfma_kernel(DecodeArgs a) {
  typedef typename Vec<T>::v8 V8;
  typedef DecodeTile<D> L;
  constexpr int STEP = L::STEP, TPL = L::TPL, LOADS = L::LOADS, PAIRS = L::PAIRS;
  constexpr int BLK = STEP * D;             // halves of a wave's K block
  constexpr int KS = D / 32;                // 32-dim k-steps of a score tile

  __shared__ int s_pages[kMaxPartPages];
  __shared__ int s_bad[W];
  // The waves' K blocks; after the loop, their O (fp32, G x D each).
  constexpr int kKBytes = W * BLK * int(sizeof(T)), kOBytes = W * kMaxGroup * D * int(sizeof(float));
  __shared__ __attribute__((aligned(16))) char s_raw[kKBytes > kOBytes ? kKBytes : kOBytes];
  __shared__ float s_m[W][kMaxGroup];
  __shared__ float s_l[W][kMaxGroup];
  // Q at head_dim 256 (head g's chunk c at c ^ (g & 7)): in registers it
  // would push the step's buffers out.
  constexpr bool kQInLds = D == 256;
  __shared__ __attribute__((aligned(16))) T s_q[kQInLds ? kMaxGroup * D : 8];

  const int tid = threadIdx.x;
  const int lane = tid & (kWave - 1);
  const int wave = tid >> 6;
  const int j = lane & 15;          // MFMA row / column index of this lane
  const int tg = lane >> 4;         // MFMA k group / C row group
  const int lrow = lane / L::CH;    // load layout: token row within a load
  const int lcol = lane % L::CH;    // load layout: 16-byte chunk of the row
  const int G = a.group;

  int item, hg;
  if (!decode_work(a, item, hg)) return;   // padding workgroup (uniform: no barrier reached)
  const int32_t* w = a.work + 4 * item;
  const int seq = w[0], tb = w[1], te = w[2], slot = w[3];
  if (seq < 0) return;   // a lane's padding record (uniform: no barrier reached)
  const int tok = a.q_token ? a.q_token[seq] : seq;   // q / out token of the sequence
  const int hq0 = hg * G;
  const int hkv = hq0 / a.ratio;
  const int page_mask = (1 << a.page_shift) - 1;

  const int pb = tb >> a.page_shift;
  const int np = te > tb ? ((te - 1) >> a.page_shift) + 1 - pb : 0;
  const int32_t* seq_pages = a.indices + a.indptr[seq];
  bool bad_id = false;
  for (int i = tid; i < np; i += W * kWave) {
    const int p = seq_pages[pb + i];
    const bool ok = p >= 0 && p < a.num_pages;
    s_pages[i] = ok ? p : -1;
    bad_id |= !ok;
  }
  // Whether any staged id is outside the pool (one vote per wave, read after
  // the barrier below): only then do the scores need a per-page mask.
  const bool wave_bad = __any(bad_id);
  if (lane == 0) s_bad[wave] = wave_bad;

  // Q^T as the B operand: dim step s covers dims 32s + 8tg .. +8 of head j.
  V8 qb[kQInLds ? 1 : KS];
  const f16* qp = a.q + int64_t(tok) * a.q_tok + int64_t(hq0) * a.q_head;
  if constexpr (kQInLds) {
    for (int i = tid; i < kMaxGroup * L::CH; i += W * kWave) {
      const int g = i / L::CH, c = i % L::CH;
      *reinterpret_cast<V8*>(&s_q[g * D + 8 * (c ^ (g & 7))]) =
          g < G ? load_v8<T>(qp + int64_t(g) * a.q_head + 8 * c) : V8{};
    }
  } else {
#pragma unroll
    for (int s = 0; s < KS; ++s)
      qb[s] = j < G ? load_v8<T>(qp + int64_t(j) * a.q_head + 32 * s + 8 * tg) : V8{};
  }
  f32x4 o[L::ACCS][8];
#pragma unroll
  for (int x = 0; x < L::ACCS; ++x)
#pragma unroll
    for (int e = 0; e < 8; ++e) o[x][e] = f32x4{};
  float m = kNegBig;   // running max of head j, scaled log2 units (same in all tg)
  float lsum = 0.f;    // this lane's share of head j's sum
  __syncthreads();
  int bad_votes = 0;
#pragma unroll
  for (int wv = 0; wv < W; ++wv) bad_votes |= s_bad[wv];
  const bool any_bad = __builtin_amdgcn_readfirstlane(bad_votes) != 0;   // the same in every lane

  const NewRow nr = new_row(a, seq, tok, hkv);
  if (nr.pos >= tb && nr.pos < te && hq0 % a.ratio == 0)
    append_row<D>(a, nr, s_pages[(nr.pos >> a.page_shift) - pb], hkv);
  const f16* kb = a.k + int64_t(hkv) * a.head_stride + lcol * 8;
  const f16* vb = a.v + int64_t(hkv) * a.head_stride + lcol * 8;
  const int nsteps = (te - tb + STEP - 1) / STEP;
  T* sk = reinterpret_cast<T*>(s_raw) + wave * BLK;

  // Unconditional loads (see the VALU kernel): past-the-end lanes and bad
  // page ids read the zero row.
  V8 k[LOADS], v[LOADS];
  auto load = [&](int c) {
#pragma unroll
    for (int i = 0; i < LOADS; ++i) {
      const int t = tb + c * STEP + TPL * i + lrow;
      const int pi = min((t >> a.page_shift) - pb, kMaxPartPages - 1);
      const int p = (c < nsteps && t < te) ? s_pages[pi] : -1;
      const int64_t off = int64_t(max(p, 0)) * a.page_stride + int64_t(t & page_mask) * a.token_stride;
      k[i] = load_v8_nt<T>(p >= 0 ? kb + (t == nr.pos ? nr.k : off) : g_zero_row + lcol * 8);
      v[i] = load_v8_nt<T>(p >= 0 ? vb + (t == nr.pos ? nr.v : off) : g_zero_row + lcol * 8);
    }
  };
  // vt[e]: dim 8 lcol + e of the lane's 8 tokens.
  auto transpose = [&](V8 (&vt)[8]) {
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      u32x4 d;
#pragma unroll
      for (int x = 0; x < 4; ++x)
        d[x] = __builtin_amdgcn_perm(__builtin_bit_cast(u32x4, v[2 * x + 1])[e >> 1],
                                     __builtin_bit_cast(u32x4, v[2 * x])[e >> 1],
                                     (e & 1) ? 0x07060302u : 0x05040100u);
      vt[e] = __builtin_bit_cast(V8, d);
    }
  };

  if (wave < nsteps) load(wave);
  for (int c = wave; c < nsteps; c += W) {
    // Park K in LDS and transpose V in registers, which frees both for the
    // next step's loads: they land during this step's math.
#pragma unroll
    for (int i = 0; i < LOADS; ++i) {
      const int t = TPL * i + lrow;
      *reinterpret_cast<V8*>(&sk[t * D + ((lcol ^ L::swz(t)) << 3)]) = k[i];
    }
    V8 vt[8];
    transpose(vt);
    load(c + W);

    // Scores. LDS runs a wave's accesses in order; keep the compiler from
    // moving them.
    f32x4 sc[PAIRS][2];
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int p = 0; p < PAIRS; ++p)
#pragma unroll
      for (int sub = 0; sub < 2; ++sub) {
        const int t = L::token(4 * sub + (j & 3), j >> 2, p);   // tile row j
        sc[p][sub] = f32x4{};
#pragma unroll
        for (int s = 0; s < KS; ++s) {
          const V8 ka = *reinterpret_cast<const V8*>(&sk[t * D + (((4 * s + tg) ^ L::swz(t)) << 3)]);
          V8 qs;
          if constexpr (kQInLds)
            qs = *reinterpret_cast<const V8*>(&s_q[j * D + 8 * ((4 * s + tg) ^ (j & 7))]);
          else
            qs = qb[s];
          sc[p][sub] = mfma16(ka, qs, sc[p][sub]);
        }
      }
    __builtin_amdgcn_wave_barrier();

    // Softmax. Tokens past the partition are masked, and those of an
    // out-of-range page id (their K/V rows read as zeros), so that they drop
    // out as in the VALU kernel.
    const int t0 = tb + c * STEP;
    float mx = -INFINITY;
#pragma unroll
    for (int p = 0; p < PAIRS; ++p)
#pragma unroll
      for (int sub = 0; sub < 2; ++sub)
#pragma unroll
        for (int x = 0; x < 4; ++x) {
          const int t = t0 + L::token(4 * sub + x, tg, p);
          bool drop = t >= te;
          if (any_bad) drop |= s_pages[min((min(t, te - 1) >> a.page_shift) - pb, kMaxPartPages - 1)] < 0;
          if (drop) sc[p][sub][x] = -INFINITY;
          mx = fmaxf(mx, sc[p][sub][x]);
        }
    mx = groups_max(mx) * a.scale_log2;
    if (__any(mx > m + 8.f)) {
      const float m_new = mx > m + 8.f ? mx : m;
      const float alpha = fast_exp2(m - m_new);
      m = m_new;
      lsum *= alpha;
#pragma unroll
      for (int x = 0; x < L::ACCS; ++x)
#pragma unroll
        for (int e = 0; e < 8; ++e) o[x][e] *= alpha;
    }
    V8 ph[L::ACCS], pl[L::ACCS];   // probabilities: rounded, and what rounding left
#pragma unroll
    for (int p = 0; p < PAIRS; ++p)
#pragma unroll
      for (int sub = 0; sub < 2; ++sub)
#pragma unroll
        for (int x = 0; x < 4; ++x) {
          const float pr = fast_exp2(fmaf(sc[p][sub][x], a.scale_log2, -m));
          lsum += pr;
          const T hi = T(pr);
          ph[p][4 * sub + x] = hi;
          pl[p][4 * sub + x] = T(pr - float(hi));
        }
    if constexpr (D == 256) {   // set x takes the lane groups of its half of the row
      const V8 zero = {};
      ph[1] = (tg & 1) ? ph[0] : zero;
      pl[1] = (tg & 1) ? pl[0] : zero;
      ph[0] = (tg & 1) ? zero : ph[0];
      pl[0] = (tg & 1) ? zero : pl[0];
    }
#pragma unroll
    for (int e = 0; e < 8; ++e)
#pragma unroll
      for (int x = 0; x < L::ACCS; ++x) o[x][e] = mfma16(vt[e], ph[x], o[x][e]);
#pragma unroll
    for (int e = 0; e < 8; ++e)
#pragma unroll
      for (int x = 0; x < L::ACCS; ++x) o[x][e] = mfma16(vt[e], pl[x], o[x][e]);
  }

  // Head j's sum over the 4 row groups of this wave (at 256 every token is
  // in two of them).
  lsum += __shfl_xor(lsum, 16);
  lsum += __shfl_xor(lsum, 32);
  if constexpr (D == 256) lsum *= 0.5f;
  // At 64 a group's rows are chunks 4 (tg % 2) + row of set tg / 2's tokens:
  // add the other set's, held by group tg ^ 2.
  if constexpr (D == 64) {
#pragma unroll
    for (int e = 0; e < 8; ++e)
#pragma unroll
      for (int x = 0; x < 4; ++x) {
        const float own = tg >> 1 ? o[1][e][x] : o[0][e][x];
        o[0][e][x] = own + __shfl_xor(own, 32);
      }
  }
  // An infinite or NaN value in V must not leave its dim, and an infinite one
  // must stay infinite: the two terms of P turn it into NaN (0 x inf, inf - inf),
  // at 256 in both halves of the row. Such a value shows in the sums; the wave
  // then does its tokens again, head by head in fp32 on the vector units.
  float z[4] = {};   // 0 x every sum: NaN where one is not finite
#pragma unroll
  for (int x = 0; x < (D == 256 ? 2 : 1); ++x)
#pragma unroll
    for (int e = 0; e < 8; ++e)
#pragma unroll
      for (int i = 0; i < 4; ++i) z[i] = fmaf(o[x][e][i], 0.f, z[i]);
  const bool again = __any(!(z[0] + z[1] + z[2] + z[3] == 0.f));
  __syncthreads();   // every wave is done with its K block: reuse them for the merge
  // O as [W][G][D]; 4-float unit u of head g's row is stored at u ^ (g & 7).
  float* s_o = reinterpret_cast<float*>(s_raw);
  auto unit_at = [&](int g, int unit) { return &s_o[(wave * G + g) * D + 4 * (unit ^ (g & 7))]; };
  if (again) {
#pragma unroll 1
    for (int g = 0; g < G; ++g) {
      float m1, l1, acc[8];
      wave_rows<T, D, W>(a, load_v8<T>(qp + int64_t(g) * a.q_head + 8 * lcol), kb, vb, tb, te,
                         s_pages, nr, m1, l1, acc);
      if (lrow == 0) {
        if (lcol == 0) {
          s_m[wave][g] = m1;
          s_l[wave][g] = l1;
        }
#pragma unroll
        for (int half = 0; half < 2; ++half)
          *reinterpret_cast<f32x4*>(unit_at(g, 2 * lcol + half)) =
              f32x4{acc[4 * half], acc[4 * half + 1], acc[4 * half + 2], acc[4 * half + 3]};
      }
    }
  } else if (j < G) {
    if (tg == 0) {
      s_m[wave][j] = m;
      s_l[wave][j] = lsum;
    }
    if (D != 64 || tg < 2) {
#pragma unroll
      for (int x = 0; x < (D == 256 ? 2 : 1); ++x)
#pragma unroll
        for (int row = 0; row < 4; ++row)
#pragma unroll
          for (int half = 0; half < 2; ++half) {
            // dims 8 (4 tg + row + 16 x) + 4 half ..
            const int unit = 2 * (4 * tg + row + 16 * x) + half;
            *reinterpret_cast<f32x4*>(unit_at(j, unit)) =
                f32x4{o[x][4 * half][row], o[x][4 * half + 1][row], o[x][4 * half + 2][row],
                      o[x][4 * half + 3][row]};
          }
    }
  }
  __syncthreads();
  decode_finish<T, D, W * kWave>(a, seq, tok, tb, slot, hq0, hg, G,
                                 [&](int g, int d, float& x, float& y, float& lse) {
    float mxw = kNegBig;
#pragma unroll
    for (int wv = 0; wv < W; ++wv) mxw = fmaxf(mxw, s_m[wv][g]);
    float ls = 0.f;
    x = y = 0.f;
#pragma unroll
    for (int wv = 0; wv < W; ++wv) {
      const float f = fast_exp2(s_m[wv][g] - mxw);
      const float* oc = &s_o[(wv * G + g) * D + 4 * ((d >> 2) ^ (g & 7)) + (d & 3)];
      ls += s_l[wv][g] * f;
      x += oc[0] * f;
      y += oc[1] * f;
    }
    x = ls > 0.f ? x / ls : 0.f;
    y = ls > 0.f ? y / ls : 0.f;
    lse = ls > 0.f ? mxw + __log2f(ls) : -INFINITY;
  });
}

// Combines the partitions of split sequences: one wave per (sequence,
// q head). Lane j first reads the log-sum-exp of partition j, so the
// weights come from one round of loads; each lane then accumulates D/64
// dimensions over the partitions.
template <typename T, int D>
__global__ __launch_bounds__(kWave) void decode_merge_kernel(const int32_t* merges,
                                                             const int32_t* q_token,
                                                             const float* part_o,
                                                             const float* part_lse, T* out,
                                                             int64_t o_tok, int64_t o_head,
                                                             int32_t num_qo_heads) {
  constexpr int DPL = D / kWave;
  typedef float PartVec __attribute__((ext_vector_type(DPL)));
  const int32_t* mg = merges + 4 * blockIdx.x;
  const int seq = mg[0], s0 = mg[1], n = mg[2];
  const int hq = blockIdx.y;
  const int lane = threadIdx.x;

  // Partials are read kBatch at a time, each batch's loads issued together
  // (one partial at a time waits a memory round trip per partial), and
  // summed in partition order, so the result does not depend on timing.
  // The first batch goes out with the first 64 log-sum-exps, before the
  // maximum they are weighted by is known.
  constexpr int kBatch = 8;
  PartVec x[kBatch];
  auto load_batch = [&](int first, int cnt) {   // partials first .. first + min(cnt, kBatch)
#pragma unroll
    for (int u = 0; u < kBatch; ++u) {
      const float* src = part_o + (int64_t(s0 + first + u) * num_qo_heads + hq) * D + lane * DPL;
      x[u] = u < cnt ? *reinterpret_cast<const PartVec*>(src) : PartVec{};
    }
  };
  float lse = lane < n ? part_lse[int64_t(s0 + lane) * num_qo_heads + hq] : -INFINITY;
  load_batch(0, n);
  float mx = lse;
  for (int j = lane + kWave; j < n; j += kWave)
    mx = fmaxf(mx, part_lse[int64_t(s0 + j) * num_qo_heads + hq]);
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) mx = fmaxf(mx, __shfl_xor(mx, off));

  float o[DPL] = {};
  float wsum = 0.f;
  if (mx > -INFINITY) {
    for (int base = 0; base < n; base += kWave) {
      const int j = base + lane;
      if (base > 0) lse = j < n ? part_lse[int64_t(s0 + j) * num_qo_heads + hq] : -INFINITY;
      const float w = j < n ? fast_exp2(lse - mx) : 0.f;
      wsum += w;
      const int cnt = min(kWave, n - base);   // uniform
      for (int t0 = 0; t0 < cnt; t0 += kBatch) {
        if (base + t0 > 0) load_batch(base + t0, cnt - t0);
#pragma unroll
        for (int u = 0; u < kBatch; ++u) {
          const float wt = __shfl(w, t0 + u);   // every lane: t0 + u < kWave
          if (t0 + u < cnt) {
#pragma unroll
            for (int e = 0; e < DPL; ++e) o[e] = fmaf(wt, x[u][e], o[e]);
          }
        }
      }
    }
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) wsum += __shfl_xor(wsum, off);
  const float inv = wsum > 0.f ? 1.f / wsum : 0.f;
  const int tok = q_token ? q_token[seq] : seq;
  T* dst = out + int64_t(tok) * o_tok + int64_t(hq) * o_head + lane * DPL;
#pragma unroll
  for (int e = 0; e < DPL; ++e) dst[e] = T(o[e] * inv);
}

// Query heads a workgroup serves, `ratio` of them sharing a KV head:
// powers of two (kunserve_decode_plan), or the largest divisor up to the
// MFMA's 16 columns (kunserve_decode_plan_grouped).
int pick_group(int ratio, bool any_divisor) {
  if (any_divisor) {
    for (int g = std::min(ratio, kMaxGroup); g > 1; --g)
      if (ratio % g == 0) return g;
    return 1;
  }
  for (int g : {8, 4, 2}) {
    if (ratio % g == 0) return g;
  }
  return 1;
}

// From 3 query heads per KV head on, MFMA; for 1 and 2 the VALU kernel is
// as fast or faster. Per launch, MFMA against VALU: 8 heads per KV head 117
// against 169 us (head_dim 256, 589 MB) and 52 against 74 us (64, 213 MB);
// 4 heads 109.5 against 111.8 us (256), but 54.5 against 53.2 us (64, where
// the MFMA kernel works on half-empty tiles: VALU there); 2 heads
// 95.6 against 94.7 us (128), 108 against 104 us (256), 58.9 against 54.6 us
// (64). At 128, 3 heads (106 MB) take 26-31 us against 35 us with K and V
// read three times, 7 heads (64 MB) 20-24 against 39-42 us.
constexpr bool uses_mfma(int group, int head_dim) {
  return group > 2 && !(head_dim == 64 && group == 4);
}
// Workgroups of the launch that a CU holds: what the MFMA kernel's registers
// allow, or the launch bounds of the VALU kernel's fewest waves (fp16 with one
// query head holds 5).
int resident_workgroups(int group, int head_dim) {
  return uses_mfma(group, head_dim) ? 2 : group == 4 ? 3 : 4;
}

// Most workgroups of a launch that combines its split rows itself: one round,
// at most 3 to a CU and at head_dim 256 one. A workgroup that counts waits for its
// stores and an atomic's round trip before its CU takes the next one, and the
// combining one reads the partials alone. Launch and merge launch against the
// launch alone, 80 drawn steps: up to these numbers 0.2-1.3 us more (one row of 1850
// tokens, 3 heads on 8, in 48 workgroups 10.9 against 10.1), beyond them less (16 rows
// of 7202, head_dim 256, in 512: 155.3 against 158.1; 93 of 553-4426 in 1008: 139.1
// against 141.2; 48 rows in 1072 at head_dim 128: 49.5 against 50.7).
int64_t max_counted_workgroups(int group, int head_dim, int64_t cus) {
  return cus * (head_dim == 256 ? 1 : std::min(3, resident_workgroups(group, head_dim)));
}

template <typename T, int D>
int launch_decode(const DecodeArgs& a, dim3 grid, hipStream_t s) {
  if (uses_mfma(a.group, D))
    paged_decode_mfma_kernel<T, D, 4><<<grid, kThreads, 0, s>>>(a);
  else if (a.group == 2)
    paged_decode_kernel<T, D, 2><<<grid, kThreads, 0, s>>>(a);
  else if (D == 64 && a.group == 4)
    paged_decode_kernel<T, D == 64 ? D : 64, 4><<<grid, kThreads, 0, s>>>(a);
  else
    paged_decode_kernel<T, D, 1><<<grid, kThreads, 0, s>>>(a);
  KSV_CHECK_LAUNCH();
  return KUNSERVE_OK;
}

template <typename T, int D>
int launch_merge(const int32_t* merges, int num_merge, const int32_t* q_token, const float* po,
                 const float* pl, f16* out, int64_t o_tok, int64_t o_head, int hq, hipStream_t s) {
  dim3 grid(num_merge, hq);
  decode_merge_kernel<T, D><<<grid, kWave, 0, s>>>(merges, q_token, po, pl,
                                                   reinterpret_cast<T*>(out),
                                                   o_tok, o_head, hq);
  KSV_CHECK_LAUNCH();
  return KUNSERVE_OK;
}

// Partition kernel, then (for split rows) the merge, for element type T.
template <typename T>
int run_decode(const DecodeArgs& a, const kunserve_decode_plan_info& info, const int32_t* plan_dev,
               int head_dim, int num_qo_heads, dim3 grid, hipStream_t s) {
  int rc;
  switch (head_dim) {
    case 64: rc = launch_decode<T, 64>(a, grid, s); break;
    case 128: rc = launch_decode<T, 128>(a, grid, s); break;
    case 256: rc = launch_decode<T, 256>(a, grid, s); break;
    default: set_error("head_dim %d not compiled", head_dim); return KUNSERVE_EUNSUPPORTED;
  }
  if (rc || info.num_merge == 0 || a.counters) return rc;
  const int32_t* merges = plan_dev + 4 * int64_t(info.num_work);
  switch (head_dim) {
    case 64:
      return launch_merge<T, 64>(merges, info.num_merge, a.q_token, a.part_o, a.part_lse, a.out, a.o_tok,
                                 a.o_head, num_qo_heads, s);
    case 128:
      return launch_merge<T, 128>(merges, info.num_merge, a.q_token, a.part_o, a.part_lse, a.out, a.o_tok,
                                  a.o_head, num_qo_heads, s);
    default:
      return launch_merge<T, 256>(merges, info.num_merge, a.q_token, a.part_o, a.part_lse, a.out, a.o_tok,
                                  a.o_head, num_qo_heads, s);
  }
}

int64_t ceil_div(int64_t a, int64_t b) { return (a + b - 1) / b; }

}  // namespace
}  // namespace kunserve

using namespace kunserve;

extern "C" int64_t kunserve_decode_plan_bound(const int32_t* kv_len_host, int32_t num_seqs) {
  if (num_seqs < 0 || (num_seqs > 0 && !kv_len_host)) return -1;
  int64_t parts = 0;
  for (int32_t b = 0; b < num_seqs; ++b)
    parts += std::max<int64_t>(1, ceil_div(std::max(kv_len_host[b], 0), kMinAutoPartTokens));
  // work records (8 lanes, each at most every item) and merge records
  return 4 * (8 * parts + num_seqs);
}

// Partition length of a grouped plan: the power of two with the least
// estimated time, in us:
//   max(bytes / bandwidth, longest item alone) + a quarter of the longest item
//   over (1 + rounds) + rounds x the start of a round + combining.
// A lone workgroup takes 11.5 ns per token at head_dim 128 (777 tokens whole
// 16.2 us, in 512s 13.3, in 256s 10.3) and 30 at 256; the launch streams
// 6.6 TB/s; workgroups of the MFMA kernel cost 2.5 and of the VALU kernel 1.6
// us per round of the device (resident_workgroups to a CU) that later items do
// not hide; rows of up to 8 partitions are combined by the launch itself (2 us;
// kunserve_paged_decode, which has no counters, merges in a second launch: the
// same plans measured within 0.6 us of the step's there), others by a second one.
// Measured against the rule of kunserve_decode_plan (per layer): 28 rows of
// 241-7578 tokens on 4 KV heads 62.7 -> 48.7 us, 96 rows of 272-2110 with 8
// heads per KV head 87.7 -> 75.3, 28 rows of 1584 at head_dim 256 78.2 -> 64.5,
// 20 rows of 102-2998 with 3 heads per KV head 31.1 -> 26.0, 48 rows of 256-4096
// at head_dim 64 with 4 heads per KV head on 4 KV heads 36.9 -> 28.2 (44.4 with
// the MFMA kernel's costs, which keep whole rows), one row of 777
// 10.4 -> 8.9; 64 rows without GQA and 128 rows of 1034-8002 keep 4096.
static int32_t grouped_part_tokens(const int32_t* kv_len, int32_t n, int64_t head_groups,
                                   int group, int head_dim, int64_t cus) {
  int64_t total = 0;
  int32_t max_len = 0;
  for (int32_t b = 0; b < n; ++b) {
    total += kv_len[b];
    max_len = std::max(max_len, kv_len[b]);
  }
  const double dim = head_dim / 128.0;
  const double stream = double(total) * double(head_groups) * 4.0 * head_dim / (6.6e6 * cus / 256.0);
  const double slots = double(cus) * resident_workgroups(group, head_dim);
  const double round_start = uses_mfma(group, head_dim) ? 2.5 * std::max(1.0, dim) : 1.6;
  const int64_t counted = max_counted_workgroups(group, head_dim, cus);
  int32_t best = kMaxPartTokens;
  double best_us = 0.0;
  for (int32_t part = kMaxPartTokens; part >= kMinAutoPartTokens; part /= 2) {
    if (part / 2 >= max_len && part > kMinAutoPartTokens) continue;   // whole rows with a shorter one
    int64_t items = 0;
    for (int32_t b = 0; b < n; ++b) items += std::max<int64_t>(1, ceil_div(kv_len[b], part));
    const double rounds = double(items) * double(head_groups) / slots;
    const double longest = 0.0115 * std::pow(dim, 1.4) *
                           std::max(kMinAutoPartTokens, std::min(part, max_len));
    const int64_t parts = ceil_div(max_len, part);
    const double us = std::max(stream, longest) + 0.25 * longest / (1.0 + rounds) +
                      rounds * round_start +
                      (parts <= 1 ? 0.0
                       : parts <= kMaxCountedParts && items * head_groups <= counted
                           ? 2.0
                           : 3.5 + 0.03 * double(parts));
    if (best_us == 0.0 || us < 0.99 * best_us) {
      best_us = us;
      best = part;
    }
  }
  return best;
}

static int decode_plan(const int32_t* kv_len_host, int32_t num_seqs, int32_t num_qo_heads,
                       int32_t num_kv_heads, int32_t head_dim, int32_t num_cus,
                       int32_t part_tokens, bool grouped, int32_t* plan_host,
                       int64_t plan_capacity, kunserve_decode_plan_info* info) {
  clear_error();
  KSV_CHECK_ARG(info && plan_host, "null plan buffer or info");
  KSV_CHECK_ARG(num_seqs >= 0 && (num_seqs == 0 || kv_len_host), "bad kv_len / num_seqs");
  KSV_CHECK_ARG(num_qo_heads > 0 && num_kv_heads > 0 && num_qo_heads % num_kv_heads == 0,
                "num_qo_heads %d not a multiple of num_kv_heads %d", num_qo_heads, num_kv_heads);
  for (int32_t b = 0; b < num_seqs; ++b)
    KSV_CHECK_ARG(kv_len_host[b] >= 0, "kv_len[%d] = %d < 0", b, kv_len_host[b]);
  const int group = pick_group(num_qo_heads / num_kv_heads, grouped);
  const int64_t head_groups = num_qo_heads / group;

  const int32_t min_part = grouped && part_tokens == 0 ? kMinAutoPartTokens : kMinPartTokens;
  if (part_tokens == 0 && grouped) {
    part_tokens = grouped_part_tokens(kv_len_host, num_seqs, head_groups, group, head_dim,
                                      std::max(num_cus, 1));
  } else if (part_tokens == 0) {
    // The longest power-of-two partition whose longest work item is at most
    // 3/4 of one CU's share of the launch (a workgroup streams nearly as
    // fast alone as a CU's share of the device, so an item that long still
    // ends with the others when it starts first) and that gives every CU
    // at least 4 workgroups. Longer partitions mean fewer splits, fewer
    // partials and, once no row is split, no merge launch: the Llama-2-7B
    // decode (64 rows of lognormal(700) tokens, 32 heads) takes 136.0 us
    // per layer at 4096 (whole rows) against 138.7 at 2048, 139.0 at 1024
    // and 140.3 at 512, and the Llama-3-8B GQA and Llama-2-70B layers run
    // 1.4% and 2.4% faster at 4096 than at 2048.
    int64_t total = 0;
    int32_t max_len = 0;
    for (int32_t b = 0; b < num_seqs; ++b) {
      total += kv_len_host[b];
      max_len = std::max(max_len, kv_len_host[b]);
    }
    const int64_t cus = std::max(num_cus, 1);
    const double share = double(total) * double(head_groups) / double(cus);
    auto workgroups = [&](int64_t part) {
      int64_t n = 0;
      for (int32_t b = 0; b < num_seqs; ++b)
        n += std::max<int64_t>(1, ceil_div(kv_len_host[b], part));
      return n * head_groups;
    };
    part_tokens = kMinPartTokens;
    for (int64_t part = kMaxPartTokens; part > kMinPartTokens; part /= 2) {
      if (double(std::min<int64_t>(part, max_len)) <= 0.75 * share &&
          workgroups(part) >= 4 * cus) {
        part_tokens = int32_t(part);
        break;
      }
    }
    // A short launch (under 8 minimum partitions per CU) whose whole rows
    // already give every CU a work item, none longer than two partitions:
    // splitting would at most halve the longest item and add the merge
    // launch, which costs more than that here (single-layer batch of 8
    // rows of U[128, 512] tokens: 10.2 us unsplit against 12.2-13.2 us
    // split at 256). Keep whole rows then.
    const int64_t per = total * head_groups / (cus * 8);
    if (part_tokens == kMinPartTokens && per < kMinPartTokens &&
        int64_t(num_seqs) * head_groups >= cus && max_len <= 2 * part_tokens) {
      while (part_tokens < max_len && part_tokens < kMaxPartTokens) part_tokens *= 2;
    }
  }
  KSV_CHECK_ARG(part_tokens >= min_part && part_tokens <= kMaxPartTokens &&
                    part_tokens % 64 == 0,
                "part_tokens %d must be a multiple of 64 in [%d, %d]", part_tokens,
                kMinPartTokens, kMaxPartTokens);

  // Work items: (seq, begin, end, slot). Full partitions first, then tails
  // by decreasing length, so the longest items start first.
  struct Item { int32_t seq, b, e, slot; };
  std::vector<Item> items;
  std::vector<int32_t> merges;
  int32_t slots = 0;
  for (int32_t b = 0; b < num_seqs; ++b) {
    const int32_t len = kv_len_host[b];
    const int32_t n = std::max<int32_t>(1, int32_t(ceil_div(len, part_tokens)));
    if (n == 1) {
      items.push_back({b, 0, len, -1});
    } else {
      merges.insert(merges.end(), {b, slots, n, 0});
      for (int32_t j = 0; j < n; ++j)
        items.push_back({b, j * part_tokens, std::min(len, (j + 1) * part_tokens), slots + j});
      slots += n;
    }
  }
  std::stable_sort(items.begin(), items.end(),
                   [](const Item& x, const Item& y) { return (x.e - x.b) > (y.e - y.b); });
  // One lane per XCD, dealt longest first to the lane that would finish it
  // first at that XCD's streaming rate. On MI355X the odd XCDs stream decode
  // about 7% slower than the even ones (10.8 against 11.6 tokens per us per
  // workgroup at the Llama-2-7B shape, the same on every layer and with the
  // items rotated across XCDs: a property of the XCD, not of the data), so
  // an even share left them finishing 5-7 us after the even XCDs. A
  // workgroup's start costs about 32 tokens of streaming.
  constexpr double kXcdRate[kXcds] = {1.0, 0.93, 1.0, 0.93, 1.0, 0.93, 1.0, 0.93};
  constexpr double kItemStartTokens = 32.0;
  std::vector<Item> lanes[kXcds];
  double load[kXcds] = {};
  for (const Item& it : items) {
    const double cost = double(it.e - it.b) + kItemStartTokens;
    int best = 0;
    for (int x = 1; x < kXcds; ++x)
      if ((load[x] + cost) / kXcdRate[x] < (load[best] + cost) / kXcdRate[best]) best = x;
    lanes[best].push_back(it);
    load[best] += cost;
  }
  size_t depth = 0;
  for (const auto& l : lanes) depth = std::max(depth, l.size());
  const int64_t need = 4 * int64_t(kXcds) * int64_t(depth) + int64_t(merges.size());
  if (need > plan_capacity) {
    set_error("plan needs %lld ints, capacity %lld", (long long)need, (long long)plan_capacity);
    return KUNSERVE_ENOSPC;
  }
  int32_t* p = plan_host;
  for (size_t r = 0; r < depth; ++r)
    for (int x = 0; x < kXcds; ++x) {
      const Item it = r < lanes[x].size() ? lanes[x][r] : Item{-1, 0, 0, -1};
      *p++ = it.seq;
      *p++ = it.b;
      *p++ = it.e;
      *p++ = it.slot;
    }
  std::copy(merges.begin(), merges.end(), p);
  info->num_work = int32_t(kXcds * depth);
  info->num_merge = int32_t(merges.size() / 4);
  info->num_slots = slots;
  info->part_tokens = part_tokens;
  info->group_size = group;
  info->plan_ints = int32_t(need);
  return KUNSERVE_OK;
}

extern "C" int kunserve_decode_plan(const int32_t* kv_len_host, int32_t num_seqs,
                                    int32_t num_qo_heads, int32_t num_kv_heads, int32_t num_cus,
                                    int32_t part_tokens, int32_t* plan_host,
                                    int64_t plan_capacity, kunserve_decode_plan_info* info) {
  return no_throw([&] {
    return decode_plan(kv_len_host, num_seqs, num_qo_heads, num_kv_heads, 128, num_cus, part_tokens,
                       false, plan_host, plan_capacity, info);
  });
}

extern "C" int kunserve_decode_plan_grouped(const int32_t* kv_len_host, int32_t num_seqs,
                                            int32_t num_qo_heads, int32_t num_kv_heads,
                                            int32_t head_dim, int32_t num_cus,
                                            int32_t part_tokens, int32_t* plan_host,
                                            int64_t plan_capacity,
                                            kunserve_decode_plan_info* info) {
  clear_error();
  KSV_CHECK_ARG(head_dim > 0 && head_dim <= 1024, "bad head_dim %d", head_dim);
  return no_throw([&] {
    return decode_plan(kv_len_host, num_seqs, num_qo_heads, num_kv_heads, head_dim, num_cus,
                       part_tokens, true, plan_host, plan_capacity, info);
  });
}

// Up to one batch of partials a row (24 partitions: 14.9 us against 13.4 with a
// second launch) and max_counted_workgroups.
extern "C" int64_t kunserve_decode_counters(const int32_t* kv_len_host, int32_t num_seqs,
                                            int32_t num_qo_heads, int32_t head_dim, int32_t num_cus,
                                            const kunserve_decode_plan_info* info) {
  clear_error();
  KSV_CHECK_ARG(info && num_seqs >= 0 && (num_seqs == 0 || kv_len_host), "null argument");
  KSV_CHECK_ARG(info->part_tokens > 0 && info->group_size > 0 && num_qo_heads > 0, "bad plan");
  if (info->num_merge == 0) return 0;
  const int64_t head_groups = num_qo_heads / info->group_size;
  int64_t items = 0;
  for (int32_t b = 0; b < num_seqs; ++b) {
    const int64_t parts = ceil_div(std::max(kv_len_host[b], 0), info->part_tokens);
    if (parts > kMaxCountedParts) return 0;
    items += std::max<int64_t>(1, parts);
  }
  return items * head_groups <= max_counted_workgroups(
                                     info->group_size, head_dim, std::max(num_cus, 1)) ? int64_t(info->num_slots) * head_groups : 0;
}

extern "C" int64_t kunserve_decode_workspace_bytes(const kunserve_decode_plan_info* info,
                                                   int32_t num_qo_heads, int32_t head_dim) {
  if (!info || num_qo_heads <= 0 || head_dim <= 0) return -1;
  const int64_t slots = info->num_slots;
  return slots * num_qo_heads * (int64_t(head_dim) + 1) * int64_t(sizeof(float));
}

int kunserve::paged_decode(const kunserve_kv_pool* pool, int32_t layer,
                           const kunserve_page_table* table, const int32_t* q_token_dev,
                           const kunserve_tensor3* q, kunserve_tensor3* out, int32_t num_qo_heads,
                           float sm_scale, const int32_t* plan_dev,
                           const kunserve_decode_plan_info* info, void* workspace_dev,
                           int64_t workspace_bytes, const StepFusion& fusion,
                           kunserve_stream_t stream) {
  clear_error();
  int rc = check_pool(pool, true);
  if (rc) return rc;
  KSV_CHECK_ARG(table && q && out && info, "null argument");
  KSV_CHECK_ARG(layer >= 0 && layer < pool->num_layers, "layer %d outside [0, %d)", layer,
                pool->num_layers);
  KSV_CHECK_ARG(std::isfinite(sm_scale) && sm_scale > 0.f,
                "sm_scale %g must be finite and positive", double(sm_scale));
  KSV_CHECK_ARG(num_qo_heads > 0 && num_qo_heads % pool->num_kv_heads == 0,
                "num_qo_heads %d not a multiple of num_kv_heads %d", num_qo_heads,
                pool->num_kv_heads);
  const int ratio = num_qo_heads / pool->num_kv_heads;
  KSV_CHECK_ARG(info->group_size >= 1 && ratio % info->group_size == 0,
                "plan group size %d does not divide the GQA ratio %d", info->group_size, ratio);
  if (info->group_size > kMaxGroup) {
    set_error("unsupported group size %d", info->group_size);
    return KUNSERVE_EUNSUPPORTED;
  }
  if (info->num_work == 0) return KUNSERVE_OK;
  KSV_CHECK_ARG(plan_dev && table->indptr_dev && table->indices_dev, "null plan or table");
  KSV_CHECK_ARG(q->data && out->data && aligned16(q->data) &&
                    (q->token_stride % 8) == 0 && (q->head_stride % 8) == 0,
                "q must be 16-byte aligned with strides that are multiples of 8");
  const int64_t ws_need = kunserve_decode_workspace_bytes(info, num_qo_heads, pool->head_dim);
  if (info->num_slots > 0 && (workspace_bytes < ws_need || !workspace_dev)) {
    set_error("decode workspace holds %lld bytes, %lld needed", (long long)workspace_bytes,
              (long long)ws_need);
    return KUNSERVE_ENOSPC;
  }
  DecodeArgs a{};
  a.q_token = q_token_dev;
  a.q = static_cast<const f16*>(q->data);
  a.q_tok = q->token_stride;
  a.q_head = q->head_stride;
  a.out = static_cast<f16*>(out->data);
  a.o_tok = out->token_stride;
  a.o_head = out->head_stride;
  a.k = static_cast<const f16*>(pool->k) + int64_t(layer) * pool->layer_stride;
  a.v = static_cast<const f16*>(pool->v) + int64_t(layer) * pool->layer_stride;
  a.page_stride = pool->page_stride;
  a.head_stride = pool->head_stride;
  a.token_stride = pool->token_stride;
  a.num_pages = int32_t(pool->num_pages);
  a.page_shift = __builtin_ctz(pool->page_size);
  a.indptr = table->indptr_dev;
  a.indices = table->indices_dev;
  a.work = plan_dev;
  float* ws = static_cast<float*>(workspace_dev);
  a.part_o = ws;
  a.part_lse = ws ? ws + int64_t(info->num_slots) * num_qo_heads * pool->head_dim : nullptr;
  if (fusion.k_new) {
    KSV_CHECK_ARG(fusion.v_new && table->kv_len_dev, "null v_new or kv_len");
    for (const kunserve_tensor3* t : {fusion.k_new, fusion.v_new})
      KSV_CHECK_ARG(t->data && aligned16(t->data) && t->token_stride % 8 == 0 &&
                        t->head_stride % 8 == 0,
                    "k_new / v_new must be 16-byte aligned with strides that are multiples of 8");
    a.k_new = static_cast<const f16*>(fusion.k_new->data);
    a.v_new = static_cast<const f16*>(fusion.v_new->data);
    a.kn_tok = fusion.k_new->token_stride;
    a.kn_head = fusion.k_new->head_stride;
    a.vn_tok = fusion.v_new->token_stride;
    a.vn_head = fusion.v_new->head_stride;
  }
  // The counting workgroups store partials 8 bytes at a time.
  if (info->num_merge > 0 && table->kv_len_dev && fusion.counters &&
      fusion.num_counters >= int64_t(info->num_slots) * (num_qo_heads / info->group_size) &&
      (reinterpret_cast<uintptr_t>(ws) & 7) == 0)
    a.counters = fusion.counters;
  a.kv_len = a.k_new || a.counters ? table->kv_len_dev : nullptr;
  a.part_tokens = info->part_tokens;
  a.num_qo_heads = num_qo_heads;
  a.ratio = ratio;
  a.scale_log2 = sm_scale * 1.4426950408889634f;

  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  // One dimension, mapped to (record, head group) by decode_work: on every
  // XCD the dispatch order is its lane's longest-first order (a launch ends
  // on short items), with an item's head groups, which read the same pages,
  // back to back.
  a.group = info->group_size;
  a.head_groups = num_qo_heads / info->group_size;
  a.num_work = info->num_work;
  const int64_t nblocks = 8 * ceil_div(info->num_work, 8) * a.head_groups;
  KSV_CHECK_ARG(nblocks < (int64_t(1) << 31), "decode grid of %lld workgroups is too large",
                (long long)nblocks);
  const dim3 grid(static_cast<unsigned>(nblocks));
  if (pool->dtype == KUNSERVE_DTYPE_BF16)
    return run_decode<bf16>(a, *info, plan_dev, pool->head_dim, num_qo_heads, grid, s);
  return run_decode<f16>(a, *info, plan_dev, pool->head_dim, num_qo_heads, grid, s);
}

extern "C" int kunserve_paged_decode(const kunserve_kv_pool* pool, int32_t layer,
                                     const kunserve_page_table* table,
                                     const int32_t* q_token_dev,
                                     const kunserve_tensor3* q, kunserve_tensor3* out,
                                     int32_t num_qo_heads, float sm_scale,
                                     const int32_t* plan_dev,
                                     const kunserve_decode_plan_info* info, void* workspace_dev,
                                     int64_t workspace_bytes, kunserve_stream_t stream) {
  return kunserve::paged_decode(pool, layer, table, q_token_dev, q, out, num_qo_heads, sm_scale,
                                plan_dev, info, workspace_dev, workspace_bytes,
                                StepFusion{}, stream);
}

// ------------------------------------------------ access-pattern calibration
// kunserve_decode_slab_probe reads a decode launch's K/V slabs (one page's
// tokens of one head: page_size x head_dim elements, contiguous) in the
// partition kernel's shape, with the slab offsets precomputed and no
// arithmetic on the data: workgroup i x heads + h reads item i's slabs of
// head h, its 4 waves striding them, two slabs in flight per wave, 1 KiB per
// load instruction, non-temporal. Each workgroup XORs what it read into
// sink[workgroup], so a test can check the bytes.
namespace kunserve {
namespace {

constexpr int kMaxSlabLoads = 16;   // 1 KiB loads per slab and tensor (slabs up to 16 KiB)

template <int NL>
__device__ __forceinline__ void probe_slab(const char* k, const char* v, int64_t off, int lane,
                                           u32x4 (&x)[2 * NL]) {
#pragma unroll
  for (int i = 0; i < NL; ++i) {
    x[i] = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(k + off + i * 1024 + lane * 16));
    x[NL + i] = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(v + off + i * 1024 + lane * 16));
  }
}

template <int NL>
__global__ __launch_bounds__(kThreads) void decode_slab_probe_kernel(
    const char* k, const char* v, const int64_t* offs, const int32_t* counts, int max_slabs,
    int64_t head_bytes, int heads, uint32_t* sink) {
  __shared__ int64_t s_off[kMaxPartPages];
  __shared__ uint32_t s_x[kWaves];
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  // The decode's dispatch order: an item's heads on one XCD, items of the
  // 8 XCD lanes interleaved.
  const int j = int(blockIdx.x) >> 3;
  const int local = j / heads;
  const int head = j - local * heads;
  const int item = 8 * local + (int(blockIdx.x) & 7);
  const int n = min(counts[item], max_slabs);
  // The item's offsets are staged in LDS, as the decode stages its page ids.
  const int64_t* o = offs + int64_t(item) * max_slabs;
  for (int i = threadIdx.x; i < n; i += kThreads) s_off[i] = o[i];
  __syncthreads();
  const int64_t hoff = int64_t(head) * head_bytes;
  u32x4 acc = {0u, 0u, 0u, 0u};
  u32x4 a[2 * NL], b[2 * NL];
  int s = wave;
  if (s < n) probe_slab<NL>(k, v, s_off[s] + hoff, lane, a);
  while (s < n) {
    const int s2 = s + kWaves;
    if (s2 < n) probe_slab<NL>(k, v, s_off[s2] + hoff, lane, b);
#pragma unroll
    for (int i = 0; i < 2 * NL; ++i) acc ^= a[i];
    s = s2;
    if (s >= n) break;
    const int s3 = s + kWaves;
    if (s3 < n) probe_slab<NL>(k, v, s_off[s3] + hoff, lane, a);
#pragma unroll
    for (int i = 0; i < 2 * NL; ++i) acc ^= b[i];
    s = s3;
  }
  uint32_t x = acc[0] ^ acc[1] ^ acc[2] ^ acc[3];
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) x ^= uint32_t(__shfl_xor(int(x), off));
  if (lane == 0) s_x[wave] = x;
  __syncthreads();
  if (threadIdx.x == 0) {
    uint32_t r = 0;
#pragma unroll
    for (int w = 0; w < kWaves; ++w) r ^= s_x[w];
    sink[item * heads + head] = r;
  }
}

}  // namespace
}  // namespace kunserve

extern "C" int kunserve_decode_slab_probe(const void* k_dev, const void* v_dev,
                                          const int64_t* slab_offsets_dev,
                                          const int32_t* counts_dev, int32_t num_items,
                                          int32_t max_slabs, int64_t head_stride_bytes,
                                          int32_t num_heads, int32_t slab_bytes,
                                          uint32_t* sink_dev, kunserve_stream_t stream) {
  using namespace kunserve;
  clear_error();
  KSV_CHECK_ARG(k_dev && v_dev && slab_offsets_dev && counts_dev && sink_dev, "null argument");
  KSV_CHECK_ARG(aligned16(k_dev) && aligned16(v_dev), "pools must be 16-byte aligned");
  KSV_CHECK_ARG(num_items >= 0 && num_items % 8 == 0 && max_slabs > 0 &&
                    max_slabs <= kMaxPartPages && num_heads > 0 && head_stride_bytes >= 0,
                "bad item (a multiple of 8), slab (at most %d) or head count", kMaxPartPages);
  KSV_CHECK_ARG(slab_bytes > 0 && slab_bytes % 1024 == 0 && slab_bytes / 1024 <= kMaxSlabLoads,
                "slab_bytes %d must be a multiple of 1024 up to %d", slab_bytes,
                kMaxSlabLoads * 1024);
  KSV_CHECK_ARG(int64_t(num_items) * num_heads < (int64_t(1) << 31), "too many workgroups");
  if (num_items == 0) return KUNSERVE_OK;
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  const char* k = static_cast<const char*>(k_dev);
  const char* v = static_cast<const char*>(v_dev);
  const dim3 grid(static_cast<unsigned>(int64_t(num_items) * num_heads));
  switch (slab_bytes / 1024) {
    case 1: decode_slab_probe_kernel<1><<<grid, kThreads, 0, s>>>(k, v, slab_offsets_dev, counts_dev, max_slabs, head_stride_bytes, num_heads, sink_dev); break;
    case 2: decode_slab_probe_kernel<2><<<grid, kThreads, 0, s>>>(k, v, slab_offsets_dev, counts_dev, max_slabs, head_stride_bytes, num_heads, sink_dev); break;
    case 4: decode_slab_probe_kernel<4><<<grid, kThreads, 0, s>>>(k, v, slab_offsets_dev, counts_dev, max_slabs, head_stride_bytes, num_heads, sink_dev); break;
    case 8: decode_slab_probe_kernel<8><<<grid, kThreads, 0, s>>>(k, v, slab_offsets_dev, counts_dev, max_slabs, head_stride_bytes, num_heads, sink_dev); break;
    case 16: decode_slab_probe_kernel<16><<<grid, kThreads, 0, s>>>(k, v, slab_offsets_dev, counts_dev, max_slabs, head_stride_bytes, num_heads, sink_dev); break;
    default: set_error("slab_bytes %d: 1, 2, 4, 8 or 16 KiB", slab_bytes); return KUNSERVE_EINVAL;
  }
  KSV_CHECK_LAUNCH();
  return KUNSERVE_OK;
}

// ------------------------------------------------ decode without allocation
// kunserve_paged_decode_noalloc keeps the split partials in `scratch`, a
// file-scope device array of kNoAllocScratchBytes that every device the
// library runs on holds until the process ends. In host code `scratch` is
// only a stand-in for the symbol: its device address, one per device, comes
// from hipGetSymbolAddress with that device current, and only that address
// is ever handed to a kernel.
namespace kunserve {
namespace {

constexpr int64_t kNoAllocScratchBytes = int64_t(32) << 20;
static __device__ __align__(256) unsigned char scratch[kNoAllocScratchBytes];

std::mutex g_scratch_mutex;
std::vector<void*> g_scratch_ptr;   // by device ordinal

// Device address of `scratch` on `device`, looked up once per device.
int scratch_address(int device, void** out) {
  std::lock_guard<std::mutex> lock(g_scratch_mutex);
  if (device >= int(g_scratch_ptr.size())) g_scratch_ptr.resize(device + 1, nullptr);
  if (!g_scratch_ptr[device]) {
    int current = 0;
    KSV_CHECK_HIP(hipGetDevice(&current));
    if (current != device) KSV_CHECK_HIP(hipSetDevice(device));
    void* ptr = nullptr;
    const hipError_t e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
    if (current != device) KSV_CHECK_HIP(hipSetDevice(current));
    if (e != hipSuccess || !ptr) {
      set_error("hipGetSymbolAddress(scratch) on device %d failed: %s", device,
                hipGetErrorString(e));
      return KUNSERVE_EHIP;
    }
    g_scratch_ptr[device] = ptr;
  }
  *out = g_scratch_ptr[device];
  return KUNSERVE_OK;
}

}  // namespace
}  // namespace kunserve

extern "C" int64_t kunserve_paged_decode_noalloc_max_bytes(void) {
  return kunserve::kNoAllocScratchBytes;
}

extern "C" int kunserve_paged_decode_noalloc(const kunserve_kv_pool* pool, int32_t layer,
                                             const kunserve_page_table* table,
                                             const int32_t* q_token_dev,
                                             const kunserve_tensor3* q, kunserve_tensor3* out,
                                             int32_t num_qo_heads, float sm_scale,
                                             const int32_t* plan_dev,
                                             const kunserve_decode_plan_info* info,
                                             kunserve_stream_t stream) {
  using namespace kunserve;
  clear_error();
  int rc = check_pool(pool, true);
  if (rc) return rc;
  KSV_CHECK_ARG(info != nullptr, "null plan info");
  const int64_t need = kunserve_decode_workspace_bytes(info, num_qo_heads, pool->head_dim);
  KSV_CHECK_ARG(need >= 0, "bad plan or head counts");
  if (need > kNoAllocScratchBytes) {
    set_error("decode partials need %lld bytes, more than the %lld bytes of the static "
              "scratch of kunserve_paged_decode_noalloc; use kunserve_paged_decode with a "
              "workspace", (long long)need, (long long)kNoAllocScratchBytes);
    return KUNSERVE_ENOSPC;
  }
  void* ws = nullptr;
  if (need > 0) {
    int device = 0;
    if (stream) {
      KSV_CHECK_HIP(hipStreamGetDevice(reinterpret_cast<hipStream_t>(stream), &device));
    } else {
      KSV_CHECK_HIP(hipGetDevice(&device));
    }
    rc = scratch_address(device, &ws);
    if (rc) return rc;
  }
  return kunserve_paged_decode(pool, layer, table, q_token_dev, q, out, num_qo_heads, sm_scale,
                               plan_dev, info, ws, need > 0 ? kNoAllocScratchBytes : 0, stream);
}
