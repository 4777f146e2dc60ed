// Paged KV append, paged decode attention and causal paged (prefill)
// attention for gfx950 (CDNA4, wave64).
//
// Slab layout (reference src/paged_attention_kernel.cu:2,18-19 and
// minitorch/paged_kv_cache.py:30): every slab is
//   [layers][2 (K,V)][pages_per_slab][heads][page_size][head_dim]
// and physical page p lives in slab p / pages_per_slab at slot
// p % pages_per_slab; slab base addresses come from a uint64 device table.
//
// Decode attention is a GEMV over paged K/V (about one flop per byte), so it
// is bound by HBM bandwidth and uses no MFMA. The design:
//   * one workgroup (4 or 8 waves) owns one (request, head, context split);
//   * a wave covers 8 tokens per step: eight lanes per token, each lane owning
//     head_dim/8 contiguous dims, so for fp16/bf16 at D = 64 every 16-byte-per-
//     lane load instruction reads 1 KiB of one page-head block contiguously
//     (8 whole token rows), non-temporally: each K/V byte is read once;
//   * every 8-lane token group keeps its own online-softmax state (running max,
//     denominator, fp32 accumulator), so the stream needs no cross-lane
//     reduction except the 8-lane dot-product sum; groups, waves and splits are
//     merged once at the end with the log-sum-exp rule;
//   * the slab table of a small pool is staged in LDS and each lane resolves
//     the page of one of its wave's row-blocks before streaming (broadcast with
//     readlane), so the dependent table -> slab -> K/V chain is paid once;
//   * the KV append of the new token is fused: the workgroup that owns the
//     last split scores the new token from the K/V inputs and writes it into
//     its page, so append + attention is a single launch;
//   * a row longer than one split writes (max, denominator, accumulator)
//     partials to a workspace and a small reduction kernel merges them. (A
//     last-arriving-workgroup merge inside the decode kernel needs device-scope
//     release/acquire fences, which write back and invalidate the XCD's L2 per
//     workgroup; measured on MI355X that made the decode 10x slower than a
//     separate launch.)
//
// Causal attention of several queries per request (a prefill) runs on the
// matrix cores for every type and head dims of whole 16-byte chunks
// (causal_kernel: 32 queries a wave, S^T = K Q^T and O^T += V^T P^T), a single
// query on the decode kernel; other rows, and few queries where that is faster,
// use the per-query query_kernel.
#include "mt_device.h"
#include "../../include/mt_paged.h"
#include <algorithm>
#include <atomic>
#include <climits>

// The decode kernel streams every K/V byte of a launch exactly once, so its
// loads are non-temporal (streamed past the caches). Measured on MI355X
// (config 2, cold pools): 24.5 -> 21.2 us together with 8 lanes per token.
#ifndef MT_DECODE_NT_LOADS
#define MT_DECODE_NT_LOADS 1
#endif
#include <cmath>
#include <mutex>
#include <type_traits>
#include <vector>

using namespace mt;

namespace {

constexpr int kWave = 64;
constexpr int kWaves = 4;
constexpr int kThreads = kWave * kWaves;
constexpr int kGroup = 4;                    // lanes per token
constexpr int kRowBlock = kWave / kGroup;    // tokens per wave step
constexpr int kMaxSplitTokens = 2048;
constexpr int kMaxSplitPages = kMaxSplitTokens / 8;
constexpr int kDefaultSplitTokens = 1024;
constexpr int kMaxSplitsPerRow = 8;
constexpr float kLog2e = 1.4426950408889634f;
#ifndef MT_STAGES
#define MT_STAGES 1
#endif
constexpr int kStages = MT_STAGES;  // register stages of the K/V stream
// Lanes per token in the decode kernel: 8 lanes of 8 dims (fp16/bf16, D 64)
// make each 16-byte-per-lane load instruction one contiguous 1 KiB of a page
// (8 whole token rows); with 4 lanes of 16 dims an instruction touches every
// row of the 2 KiB page-row block half each.
#ifndef MT_DECODE_GROUP
#define MT_DECODE_GROUP 8
#endif
constexpr int kDecodeGroup = MT_DECODE_GROUP;
constexpr bool kDecodeNT = MT_DECODE_NT_LOADS != 0;
// Pools of at most this many slabs have their slab table staged in LDS by the
// decode kernel, so that page resolution after the block-table read is an LDS
// read instead of a second dependent global load.
constexpr int kLdsSlabs = 512;

#ifdef MT_DECODE_TIMELINE
// Measurement builds only (bench.py --timeline): wall-clock stamps of each
// decode workgroup's first item, taken by thread 0 at 100 MHz
// (s_memrealtime), workgroups below kTimelineMax. Record: [start, work entry
// returned, table/query/offset returned, past the staging barrier, K/V
// stream start, end, HW_ID register, XCC_ID register]. A stamp that follows
// a load takes that load's value as an operand, so it waits for the data.
// The product build has none of this.
constexpr int kTimelineMax = 8192;
constexpr int kTimelineFields = 8;
__device__ uint64_t g_decode_timeline[kTimelineMax * kTimelineFields];
template <class T>
__device__ __forceinline__ uint64_t stamp_after(T dep) {
  uint64_t t;
  asm volatile("s_memrealtime %0\n\ts_waitcnt lgkmcnt(0)" : "=s"(t) : "v"(dep) : "memory");
  return t;
}
#endif

struct Geometry {
  int heads, dim, page_size, log2_page, pps, num_slabs, columns, layer;
  int64_t kind_stride;  // elements between the K and V planes of one layer
  // p / pps for 0 <= p < 2^31 as (p * pps_magic) >> pps_shift, so that page
  // resolution needs no division: pps_magic = ceil(2^(31+s) / pps) with
  // s = ceil(log2 pps), pps_shift = 31 + s (the error n * e / 2^(31+s),
  // e < 1, stays below 1 / pps for n < 2^31 since pps <= 2^s).
  uint64_t pps_magic;
  int pps_shift;
};

__device__ __forceinline__ int slab_index(int physical, const Geometry& g) {
  return int((uint64_t(uint32_t(physical)) * g.pps_magic) >> g.pps_shift);
}

__device__ __forceinline__ float fast_exp2(float x) { return __builtin_amdgcn_exp2f(x); }

// Address of (slot, head, row 0, col 0) in the K plane of `layer`, or nullptr
// for the cases the reference treats as a missing page
// (src/paged_attention_kernel.cu:11-16): logical column out of range, negative
// or out-of-pool physical page, or a null slab.
template <class T>
__device__ __forceinline__ const T* page_base(const uint64_t* slabs, const int* table_row,
                                              int64_t logical, const Geometry& g, int head) {
  if (logical < 0 || logical >= g.columns) return nullptr;
  const int physical = table_row[logical];
  if (physical < 0 || int64_t(physical) >= int64_t(g.num_slabs) * g.pps) return nullptr;
  const int slab = slab_index(physical, g);
  const uint64_t address = slabs[slab];
  if (!address) return nullptr;
  const int slot = physical - slab * g.pps;
  const int64_t i = ((int64_t(g.layer) * 2 * g.pps + slot) * g.heads + head) *
                    int64_t(g.page_size) * g.dim;
  return reinterpret_cast<const T*>(address) + i;
}

// Page base from an already loaded physical page ID (the table read is
// issued separately so that it overlaps other loads).
template <class T>
__device__ __forceinline__ const T* resolve_page(const uint64_t* slabs, int physical,
                                                 const Geometry& g, int head) {
  if (physical < 0 || int64_t(physical) >= int64_t(g.num_slabs) * g.pps) return nullptr;
  const int slab = slab_index(physical, g);
  const uint64_t address = slabs[slab];
  if (!address) return nullptr;
  const int slot = physical - slab * g.pps;
  const int64_t i = ((int64_t(g.layer) * 2 * g.pps + slot) * g.heads + head) *
                    int64_t(g.page_size) * g.dim;
  return reinterpret_cast<const T*>(address) + i;
}

// Page base from a physical page ID and its slab's base address (already
// looked up); nullptr for a null slab.
template <class T>
__device__ __forceinline__ const T* page_in_slab(uint64_t address, int physical, const Geometry& g,
                                                 int head) {
  if (!address) return nullptr;
  const int slot = physical - slab_index(physical, g) * g.pps;
  const int64_t i = ((int64_t(g.layer) * 2 * g.pps + slot) * g.heads + head) *
                    int64_t(g.page_size) * g.dim;
  return reinterpret_cast<const T*>(address) + i;
}

__device__ __forceinline__ bool physical_in_pool(int physical, const Geometry& g) {
  return physical >= 0 && int64_t(physical) < int64_t(g.num_slabs) * g.pps;
}

// Online-softmax state of one token group, in base-2 units (scores are
// pre-multiplied by log2(e)). A missing page contributes a NaN score, which
// fmaxf drops from the running max and which then poisons the denominator,
// matching the reference's NaN propagation (src/paged_attention_kernel.cu:53,66-69,84).
template <int N, int G = kGroup>
struct Softmax {
  float m, l, acc[N];
  __device__ __forceinline__ void init() {
    m = -INFINITY; l = 0.f;
#pragma unroll
    for (int i = 0; i < N; ++i) acc[i] = 0.f;
  }
  __device__ __forceinline__ void add(float s, const float* v) {
    const float mn = fmaxf(m, s);
    const float alpha = (m == -INFINITY) ? 0.f : fast_exp2(m - mn);
    const float p = fast_exp2(s - mn);
    l = fmaf(l, alpha, p);
#pragma unroll
    for (int i = 0; i < N; ++i) acc[i] = fmaf(p, v[i], acc[i] * alpha);
    m = mn;
  }
  // Add U tokens with one rescale: the running max moves once per call.
  template <int U, class VF>
  __device__ __forceinline__ void add_many(const float* s, const bool* valid, VF&& v_of) {
    float mx = m;
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (valid[u]) mx = fmaxf(mx, s[u]);
    const float alpha = (m == -INFINITY) ? 0.f : fast_exp2(m - mx);
    l *= alpha;
#pragma unroll
    for (int i = 0; i < N; ++i) acc[i] *= alpha;
#pragma unroll
    for (int u = 0; u < U; ++u) {
      if (valid[u]) {
        const float p = fast_exp2(s[u] - mx);
        l += p;
        float v[N];
        v_of(u, v);
#pragma unroll
        for (int i = 0; i < N; ++i) acc[i] = fmaf(p, v[i], acc[i]);
      }
    }
    m = mx;
  }
  __device__ __forceinline__ void merge(float mo, float lo, const float* ao) {
    const float mn = fmaxf(m, mo);
    const float sa = (m == -INFINITY) ? 0.f : fast_exp2(m - mn);
    const float sb = (mo == -INFINITY) ? 0.f : fast_exp2(mo - mn);
    l = l * sa + lo * sb;
#pragma unroll
    for (int i = 0; i < N; ++i) acc[i] = acc[i] * sa + ao[i] * sb;
    m = mn;
  }
  // Merge with the state held `rot` lanes further along the same 16-lane row
  // (DPP row rotate; no LDS traffic).
  template <int CTRL>
  __device__ __forceinline__ void merge_dpp() {
    float ao[N];
    const float mo = __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(m), CTRL, 0xF, 0xF, false));
    const float lo = __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(l), CTRL, 0xF, 0xF, false));
#pragma unroll
    for (int i = 0; i < N; ++i)
      ao[i] = __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(acc[i]), CTRL, 0xF, 0xF, false));
    merge(mo, lo, ao);
  }
  // Merge the token groups of each 16-lane row: afterwards lanes with
  // lane % 16 < G hold their row's state for chunk lane % G.
  __device__ __forceinline__ void row_merge() {
    static_assert(G == 4 || G == 8, "row_merge expects 4 or 8 lanes per token");
    if constexpr (G == 4) merge_dpp<0x124>();  // row_ror:4
    merge_dpp<0x128>();                        // row_ror:8
  }
  // Merge the states of the token groups of a wave (lanes with equal
  // lane % G): afterwards lanes 0..G-1 hold the wave's state for their chunk.
  __device__ __forceinline__ void wave_merge() {
#pragma unroll
    for (int off = G; off < kWave; off <<= 1) {
      float ao[N];
      const float mo = __shfl_xor(m, off);
      const float lo = __shfl_xor(l, off);
#pragma unroll
      for (int i = 0; i < N; ++i) ao[i] = __shfl_xor(acc[i], off);
      merge(mo, lo, ao);
    }
  }
};

__device__ __forceinline__ float finalize(float acc, float l) {
  return l > 0.f ? acc / l : (isnan(l) ? NAN : 0.f);
}

// Sum of a value over the G lanes of a token group with DPP: quad permutes
// for 4 lanes, then the half-row mirror (lane i <-> 7 - i) for 8 lanes.
template <int G = kGroup>
__device__ __forceinline__ float group_sum(float x) {
  x += __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(x), 0xB1, 0xF, 0xF, true));
  x += __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(x), 0x4E, 0xF, 0xF, true));
  if constexpr (G == 8)
    x += __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(x), 0x141, 0xF, 0xF, true));
  return x;
}

// How a decode reads rows: element by element, masked to the head dim; in
// 16-byte loads when the head dim is the kernel's (64 or 128); in 16-byte
// loads masked to a smaller head dim of whole 16-byte chunks (80 of 128, 32 of
// 64), whose other lanes hold zeros.
enum Rows : int { kRowsElements = 0, kRowsFull = 1, kRowsPadded = 2 };

// Per-lane chunk of one token row: DL values at `p` (K or V plane), converted
// to fp32. VEC (Rows) uses 16-byte loads; otherwise element loads masked to `dim`.
// The G lanes of a row take its 16-byte chunks in turn (lane g chunks g, g + G,
// ..), so that each load instruction covers consecutive bytes also where a lane
// owns several chunks; with a lane's chunks next to each other fp32 and head
// dim 128 streamed at 2.1-2.8 TB/s, fp32's 8 x 900 tokens x 25 heads of 128 in
// 64 us. col_of(i): the column of a lane's value i less its first.
template <int DT, int DL, int VEC, int G>
struct Chunk {
  static __device__ __forceinline__ constexpr int col_of(int i) {
    return VEC ? i / per16<DT>() * (G * per16<DT>()) + i % per16<DT>() : i;
  }
  static __device__ __forceinline__ int first_col(int g) { return VEC ? g * per16<DT>() : g * DL; }
  using T = typename Elem<DT>::T;
  static constexpr int NV = VEC ? DL * elem_bytes<DT>() / 16 : 1;
  u32x4 raw[VEC ? NV : 1];
  float val[VEC ? 1 : DL];
  // NTL: non-temporal loads (data read once, not kept in the caches).
  template <bool NTL = false>
  __device__ __forceinline__ void load(const T* p, int col0, int dim) {
    if constexpr (VEC) {
      const auto* v = global_view(reinterpret_cast<const u32x4*>(p));
#pragma unroll
      for (int i = 0; i < NV; ++i) {
        if (VEC == kRowsPadded && col0 + i * G * per16<DT>() >= dim) raw[i] = u32x4{0u, 0u, 0u, 0u};
        else if constexpr (NTL) raw[i] = __builtin_nontemporal_load(v + i * G);
        else raw[i] = v[i * G];
      }
    } else {
      const auto* g = global_view(p);
#pragma unroll
      for (int i = 0; i < DL; ++i) val[i] = (col0 + i < dim) ? to_f32<DT>(g[i]) : 0.f;
    }
  }
  // Same chunk from an LDS copy of the row (p points at column col0).
  __device__ __forceinline__ void load_lds(const T* p, int col0, int dim) {
    if constexpr (VEC) {
#pragma unroll
      for (int i = 0; i < NV; ++i) raw[i] = reinterpret_cast<const u32x4*>(p)[i * G];
    } else {
#pragma unroll
      for (int i = 0; i < DL; ++i) val[i] = (col0 + i < dim) ? to_f32<DT>(p[i]) : 0.f;
    }
  }
  __device__ __forceinline__ void nan_fill() {
    if constexpr (VEC) {
#pragma unroll
      for (int i = 0; i < NV; ++i) raw[i] = u32x4{~0u, ~0u, ~0u, ~0u};
    } else {
#pragma unroll
      for (int i = 0; i < DL; ++i) val[i] = NAN;
    }
  }
  __device__ __forceinline__ void to_float(float* o) const {
    if constexpr (VEC) {
      constexpr int E = per16<DT>();
#pragma unroll
      for (int i = 0; i < NV; ++i) unpack16<DT>(raw[i], o + i * E);
    } else {
#pragma unroll
      for (int i = 0; i < DL; ++i) o[i] = val[i];
    }
  }
};

// One query vector split over the 4 lanes of a token group. For fp16/bf16
// with 16-byte access the query stays packed in its input type and q.k uses
// the fp32-accumulating dot2 instructions (v_dot2c_f32_f16 / _bf16), so no
// K conversion is needed and the query takes DL/2 registers; the 1/sqrt(D)
// and log2(e) factors are applied to the summed score. fp32 and the masked
// path keep a pre-scaled fp32 query.
template <int DT, int D, int VEC, int G = kGroup>
struct Query {
  using T = typename Elem<DT>::T;
  static constexpr int DL = D / G;
  static constexpr bool PACKED = VEC && DT != kF32;
  uint32_t qp[PACKED ? DL / 2 : 1];
  float qf[PACKED ? 1 : DL];
  float post_scale;
  __device__ __forceinline__ void load(const T* q, int col0, int dim, float scale) {
    Chunk<DT, DL, VEC, G> c;
    c.load(q + col0, col0, dim);
    if constexpr (PACKED) {
#pragma unroll
      for (int w = 0; w < DL / 2; ++w) qp[w] = c.raw[w / 4][w % 4];
      post_scale = scale;
    } else {
      c.to_float(qf);
#pragma unroll
      for (int i = 0; i < DL; ++i) qf[i] *= scale;
      post_scale = 1.f;
    }
  }
  // This lane's part of q.k (before the group sum and post_scale).
  __device__ __forceinline__ float partial(const Chunk<DT, DL, VEC, G>& k) const {
    float s = 0.f;
    if constexpr (PACKED) {
      typedef _Float16 h2 __attribute__((ext_vector_type(2)));
      typedef __bf16 b2 __attribute__((ext_vector_type(2)));
#pragma unroll
      for (int w = 0; w < DL / 2; ++w) {
        const uint32_t kw = k.raw[w / 4][w % 4];
        if constexpr (DT == kF16)
          s = __builtin_amdgcn_fdot2(__builtin_bit_cast(h2, qp[w]), __builtin_bit_cast(h2, kw), s, false);
        else
          s = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(b2, qp[w]), __builtin_bit_cast(b2, kw), s, false);
      }
    } else {
      float kf[DL];
      k.to_float(kf);
#pragma unroll
      for (int i = 0; i < DL; ++i) s = fmaf(qf[i], kf[i], s);
    }
    return s;
  }
  __device__ __forceinline__ float score(const Chunk<DT, DL, VEC, G>& k) const {
    return group_sum<G>(partial(k)) * post_scale;
  }
};

// Stream the tokens [t0, t0 + ntok) of one (request, head) whose page bases
// (K plane) are in s_page (entry j covers tokens t0 + j*P ...). Row-blocks
// rb = rb_first, rb_first + rb_step, ... are processed U at a time; with
// STAGES = 2 the loads of the next U row-blocks are in flight while the
// current ones are scored and accumulated.
template <int DT, int D, int VEC, int U, int STAGES>
__device__ __forceinline__ void stream_rows(Softmax<D / kGroup>& st, const Query<DT, D, VEC>& q,
                                            typename Elem<DT>::T const* const* s_page,
                                            int ntok, int rb_first, int rb_step,
                                            const Geometry& g, int dim) {
  using T = typename Elem<DT>::T;
  constexpr int DL = D / kGroup;
  const int lane = threadIdx.x & (kWave - 1);
  const int tok = lane >> 2;
  const int col0 = Chunk<DT, DL, VEC, kGroup>::first_col(lane & 3);
  const int nrb = (ntok + kRowBlock - 1) / kRowBlock;
  const int pmask = g.page_size - 1;
  using C = Chunk<DT, DL, VEC, kGroup>;
  auto issue = [&](int rb0, C* kc, C* vc, bool* valid) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int rel = (rb0 + u * rb_step) * kRowBlock + tok;
      valid[u] = rel < ntok;
      const T* base = valid[u] ? s_page[rel >> g.log2_page] : nullptr;
      if (base) {
        const T* kp = base + (rel & pmask) * dim + col0;
        kc[u].load(kp, col0, dim);
        vc[u].load(kp + g.kind_stride, col0, dim);
      } else {
        kc[u].nan_fill();
        vc[u].nan_fill();
      }
    }
  };
  auto consume = [&](const C* kc, const C* vc, const bool* valid) {
    float s[U];
#pragma unroll
    for (int u = 0; u < U; ++u) s[u] = q.score(kc[u]);
    st.template add_many<U>(s, valid, [&](int u, float* vf) { vc[u].to_float(vf); });
  };
  if constexpr (STAGES == 1) {
    for (int rb0 = rb_first; rb0 < nrb; rb0 += rb_step * U) {
      C kc[U], vc[U];
      bool valid[U];
      issue(rb0, kc, vc, valid);
      consume(kc, vc, valid);
    }
  } else {
    C kc[U], vc[U];
    bool valid[U];
    int rb0 = rb_first;
    if (rb0 < nrb) issue(rb0, kc, vc, valid);
    while (rb0 < nrb) {
      const int nxt = rb0 + rb_step * U;
      C nk[U], nv[U];
      bool nvalid[U];
      if (nxt < nrb) issue(nxt, nk, nv, nvalid);
      consume(kc, vc, valid);
#pragma unroll
      for (int u = 0; u < U; ++u) { kc[u] = nk[u]; vc[u] = nv[u]; valid[u] = nvalid[u]; }
      rb0 = nxt;
    }
  }
}

struct DecodeArgs {
  void* out;
  const void* q;
  const void* k;
  const void* v;
  const uint64_t* slabs;
  const int* table;
  const int* offsets;
  int batch;
  int split_tokens;
  int nsplit_max;
  float qscale;
  int64_t items;
  Geometry g;
  float* partials;
  // Optional work list: work_items (row, split) pairs in visiting order,
  // then merge_rows row indices whose splits need the reduction. Without it
  // every (split, row, head) is an item and every row is a merge candidate.
  const int* work;
  int work_items;
  int merge_rows;
  int64_t qkv_stride;  // elements between the rows of q, k and v (h * d when contiguous)
  // Without a work list and with one split per row: when rank_rows is set,
  // every workgroup ranks the batch's rows by context length from `offsets`
  // (longest first, ties by row) into dynamic LDS and visits them in the
  // order a host work list would give -- passes of rank_per rows, every
  // other pass reversed. Needs 2 * (batch rounded up to 4) ints of dynamic LDS.
  int rank_rows;
  int rank_per;
  // > 0: every row attends this many keys (kVisitUniform; offsets is null).
  // With k null they all lie in the pages, else the last is the new token.
  int uniform_len;
  // Work list built on the device (order_kernel) for a batch whose rows may
  // split: work_count[0] (row, split) pairs at `work`, then work_count[1]
  // merge rows. `items` is then only the capacity (batch * nsplit_max *
  // heads) and the grid one residency round that strides over the list.
  const int* work_count;
};

// How decode_kernel finds its items, a template parameter so that each
// instantiation carries only its own prologue (the kernel's start is
// latency-bound, and measured slower when unused prologue code grew):
// from a work list (host- or device-built), by ranking the rows in every
// workgroup, or as the plain (split, row, head) grid, of rows of their own
// lengths or of one length known to the host.
constexpr int kVisitList = 0, kVisitRank = 1, kVisitGrid = 2, kVisitUniform = 3;

// Rows a decode workgroup ranks on its own (the ranking costs each thread
// batch / threads * batch LDS reads).
constexpr int kRankRows = 256;
// Rows order_kernel orders in its one workgroup; larger batches are visited
// in batch order.
constexpr int kOrderRows = 2048;
constexpr int kOrderThreads = 1024;

// Stream one wave's share of a split: row-blocks j = wave + waves * i
// (16 tokens each) of tokens [t0, t0 + ntok). Lane s of the wave holds in
// `base` the page base (K plane) of page slot s, resolved in the prologue:
// slot i for page sizes >= 16 (one page per row-block), slots 2i and 2i + 1
// for page size 8. Page bases are broadcast with readlane (scalar registers)
// or, for page size 8, a lane shuffle; no LDS and no barrier are involved.
template <int DT, int D, int VEC, int U, int STAGES, int G>
__device__ __forceinline__ void stream_wave(Softmax<D / G, G>& st, const Query<DT, D, VEC, G>& q,
                                            uint64_t base, int ntok, int wave, int waves,
                                            const Geometry& g, int dim) {
  using T = typename Elem<DT>::T;
  constexpr int DL = D / G;
  constexpr int RB = kWave / G;  // tokens per wave step
  using C = Chunk<DT, DL, VEC, G>;
  const int lane = threadIdx.x & (kWave - 1);
  const int tok = lane / G;
  const int col0 = Chunk<DT, DL, VEC, G>::first_col(lane % G);
  const int pmask = g.page_size - 1;
  const bool two_pages = g.page_size < RB;
  const int nrb = (ntok + RB - 1) / RB;
  const int mine = nrb > wave ? (nrb - wave + waves - 1) / waves : 0;
  const uint32_t base_lo = uint32_t(base), base_hi = uint32_t(base >> 32);
  auto issue = [&](int i0, C* kc, C* vc, bool* valid) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int i = i0 + u;
      const int rel = (wave + waves * i) * RB + tok;
      valid[u] = i < mine && rel < ntok;
      uint64_t pb;
      if (two_pages) {
        const int slot = 2 * i + (tok >> 3);
        pb = (uint64_t(uint32_t(__shfl(int(base_hi), slot))) << 32) | uint32_t(__shfl(int(base_lo), slot));
      } else {
        const int slot = i < kWave ? i : kWave - 1;
        pb = (uint64_t(uint32_t(__builtin_amdgcn_readlane(int(base_hi), slot))) << 32) |
             uint32_t(__builtin_amdgcn_readlane(int(base_lo), slot));
      }
      const T* page = reinterpret_cast<const T*>(pb);
      if (valid[u] && page) {
        const T* kp = page + (rel & pmask) * dim + col0;
        kc[u].template load<kDecodeNT>(kp, col0, dim);
        vc[u].template load<kDecodeNT>(kp + g.kind_stride, col0, dim);
      } else {
        kc[u].nan_fill();
        vc[u].nan_fill();
      }
    }
  };
  auto consume = [&](const C* kc, const C* vc, const bool* valid) {
    float s[U];
#pragma unroll
    for (int u = 0; u < U; ++u) s[u] = q.score(kc[u]);
    st.template add_many<U>(s, valid, [&](int u, float* vf) { vc[u].to_float(vf); });
  };
  if constexpr (STAGES == 1) {
    for (int i0 = 0; i0 < mine; i0 += U) {
      C kc[U], vc[U];
      bool valid[U];
      issue(i0, kc, vc, valid);
      consume(kc, vc, valid);
    }
  } else {
    C kc[U], vc[U];
    bool valid[U];
    if (mine > 0) issue(0, kc, vc, valid);
    for (int i0 = 0; i0 < mine; i0 += U) {
      C nk[U], nv[U];
      bool nvalid[U];
      if (i0 + U < mine) issue(i0 + U, nk, nv, nvalid);
      consume(kc, vc, valid);
#pragma unroll
      for (int u = 0; u < U; ++u) { kc[u] = nk[u]; vc[u] = nv[u]; valid[u] = nvalid[u]; }
    }
  }
}

// Fused KV append + decode attention over (request, head, split) items.
// Items come from the work list when one is given (visiting order chosen by
// the caller, e.g. longest first), else from the full (split, row, head) grid.
// 8-wave fp16/bf16 workgroups at D = 64 (config 2's shape) are meant to be
// resident three per compute unit, i.e. six waves per SIMD and at most 80
// VGPRs: one VGPR more drops a whole workgroup per compute unit (and the
// launcher then picks 4-wave workgroups), so the bound is stated. Other
// shapes need more registers and keep the compiler's choice.
template <int DT, int D, int VEC, int U, int STAGES, int WAVES, int G, int MODE>
__global__ __launch_bounds__(WAVES * kWave)
__attribute__((amdgpu_waves_per_eu(WAVES == 8 && D == 64 && VEC == kRowsFull && DT != kF32 && U <= 2 ? 6 : 1)))
void decode_kernel(DecodeArgs a) {
  using T = typename Elem<DT>::T;
  constexpr int DL = D / G;
  constexpr int RB = kWave / G;
  constexpr int PSTRIDE = D + 2;
  constexpr int NT = WAVES * kWave;
  constexpr int NS = WAVES * 4;  // partial states per item: one per 16-lane row
  constexpr int SLABS_PER_THREAD = (kLdsSlabs + NT - 1) / NT;
  constexpr int GROUPS = NT / D;    // thread groups of the first merge level
  constexpr int PER = NS / GROUPS;  // row states each group merges
  static_assert(NT % D == 0 && NS % GROUPS == 0, "merge partition");
  __shared__ float s_m[NS], s_l[NS];
  __shared__ float s_acc[NS][D];
  __shared__ float s2_m[GROUPS], s2_l[GROUPS];
  __shared__ float s2_acc[GROUPS][D];
  __shared__ uint64_t s_slabs[kLdsSlabs];
  __shared__ __align__(16) T s_new[2][D];  // the new token's K and V rows

#ifdef MT_DECODE_TIMELINE
  const uint64_t tl_start = wall_clock64();
  uint64_t tl_entry = 0, tl_loads = 0, tl_barrier = 0, tl_stream = 0;
#endif
  const Geometry& g = a.g;
  const int dim = VEC == kRowsFull ? D : g.dim;
  const int tid = threadIdx.x;
  const int64_t bh_count = int64_t(a.batch) * g.heads;
  // The slab table of a small pool is staged in LDS. A workgroup whose first
  // item is certain to have work (every work-list item; split 0 of the full
  // grid) reads it before anything else, so that it arrives while the
  // item's own loads are in flight; others read it once an item has work.
  const bool lds_slabs = g.num_slabs <= kLdsSlabs;
  bool slabs_staged = !lds_slabs;
  bool slabs_loaded = false;
  uint64_t slab_reg[SLABS_PER_THREAD];
  auto load_slabs = [&]() {
#pragma unroll
    for (int j = 0; j < SLABS_PER_THREAD; ++j) {
      const int i = tid + j * NT;
      slab_reg[j] = i < g.num_slabs ? a.slabs[i] : 0;
    }
    slabs_loaded = true;
  };
  if (lds_slabs && (MODE != kVisitGrid || blockIdx.x < bh_count)) load_slabs();
  // In-kernel longest-first order (see DecodeArgs::rank_rows): s_len holds
  // the offsets, s_order[k] the row of rank k; (length desc, row asc) is a
  // strict order, so the ranks are a permutation whatever the offsets hold.
  // s_len is padded to a multiple of 4 rows with INT_MIN, which no row
  // ranks behind, and read 4 rows per LDS load. Each row's rank is counted
  // by tpr consecutive lanes (the largest power of two up to 64 with
  // tpr * batch <= threads), each over its own slice of the candidates, and
  // summed with lane shuffles: the count runs on every wave, not one.
  extern __shared__ __align__(16) int s_rank[];
  const int len4 = (a.batch + 3) & ~3;
  int* const s_len = s_rank;
  int* const s_order = s_rank + len4;
  if constexpr (MODE == kVisitRank) {
    for (int r = tid; r < len4; r += NT) s_len[r] = r < a.batch ? a.offsets[r] : INT_MIN;
    __syncthreads();
    const int4* len_v = reinterpret_cast<const int4*>(s_len);
    int tpr = 1;
    while (tpr < kWave && 2 * tpr * a.batch <= NT) tpr *= 2;
    const int n4 = len4 / 4;
    const int per_part = (n4 + tpr - 1) / tpr;  // int4 candidates per lane
    for (int t0 = 0; t0 < a.batch * tpr; t0 += NT) {
      const int t = t0 + tid;
      const int r = t / tpr, part = t - r * tpr;
      int rank = 0;
      if (r < a.batch) {
        const int lr = s_len[r];
        const int c1 = min(n4, (part + 1) * per_part);
        for (int q4 = part * per_part; q4 < c1; ++q4) {
          const int4 l = len_v[q4];
          const int q = 4 * q4;
          rank += (l.x > lr) | ((l.x == lr) & (q < r));
          rank += (l.y > lr) | ((l.y == lr) & (q + 1 < r));
          rank += (l.z > lr) | ((l.z == lr) & (q + 2 < r));
          rank += (l.w > lr) | ((l.w == lr) & (q + 3 < r));
        }
      }
      for (int o = 1; o < tpr; o <<= 1) rank += __shfl_xor(rank, o);
      if (r < a.batch && part == 0) s_order[rank] = r;
    }
    __syncthreads();
  }
  const int wave = tid >> 6;
  const int lane = tid & (kWave - 1);
  const int col0 = Chunk<DT, DL, VEC, G>::first_col(lane % G);
  const int64_t cap = int64_t(g.columns) * g.page_size;
  const int sub_shift = g.page_size < RB ? 1 : 0;
  const int rb_per_wave = a.split_tokens / RB / WAVES;
  const T* qp = static_cast<const T*>(a.q);
  const T* kin = static_cast<const T*>(a.k);
  const T* vin = static_cast<const T*>(a.v);
  T* out = static_cast<T*>(a.out);
  const uint64_t* work64 = reinterpret_cast<const uint64_t*>(a.work);

  // A device-built list's length is read together with the workgroup's first
  // entry (within the list's capacity, which bounds the grid), so the count
  // adds no round trip before the first item.
  int64_t items = a.items;
  uint64_t first_entry = 0;
  if (MODE == kVisitList && a.work_count) {
    first_entry = work64[blockIdx.x / unsigned(g.heads)];
    items = std::min(int64_t(a.work_count[0]) * g.heads, a.items);  // never past the list
  }

  for (int64_t item = blockIdx.x; item < items; item += gridDim.x) {
    int split, b, head;
    if constexpr (MODE == kVisitList) {
      // (row, split) read as one 8-byte load: the workgroup's first dependent
      // round trip.
      const int w = int(unsigned(item) / unsigned(g.heads));
      head = int(item) - w * g.heads;
      const uint64_t e = (a.work_count && item == blockIdx.x) ? first_entry : work64[w];
      b = int(uint32_t(e));
      split = int(uint32_t(e >> 32));
#ifdef MT_DECODE_TIMELINE
      if (item == blockIdx.x) tl_entry = stamp_after(b);
#endif
      if (!((unsigned(b) < unsigned(a.batch)) & (unsigned(split) < unsigned(a.nsplit_max)))) continue;
    } else if constexpr (MODE == kVisitRank) {
      // item = (visiting position, head); one split per row
      const int pos = int(unsigned(item) / unsigned(g.heads));
      head = int(item) - pos * g.heads;
      const int pass = pos / a.rank_per, within = pos - pass * a.rank_per;
      const int width = min(a.rank_per, a.batch - pass * a.rank_per);
      b = s_order[pass * a.rank_per + ((pass & 1) ? width - 1 - within : within)];
      split = 0;
    } else {
      split = int(unsigned(item) / unsigned(bh_count));
      const int bhi = int(item) - split * int(bh_count);
      b = int(unsigned(bhi) / unsigned(g.heads));
      head = bhi - b * g.heads;
    }
    const int64_t bh = int64_t(b) * g.heads + head;

    // Loads that do not depend on the context length are issued first, all
    // in one round trip: the table entry of each of this wave's page slots
    // (the next link of the chain to the K/V loads), the query, the new
    // token's K/V (wave 0) and the offset.
    const int* table_row = a.table + int64_t(b) * g.columns;
    const int t0i = split * a.split_tokens;
    const int slot_i = lane >> sub_shift;
    const int slot_tok = (wave + WAVES * slot_i) * RB + ((lane & sub_shift) << 3);
    const int64_t slot_logical = (int64_t(t0i) + slot_tok) >> g.log2_page;
    int physical = -1;
    if (slot_i < rb_per_wave && slot_logical < g.columns) physical = table_row[slot_logical];
    Query<DT, D, VEC, G> qv;
    const int64_t qrow = int64_t(b) * a.qkv_stride + int64_t(head) * dim;  // q, k, v row
    qv.load(qp + qrow, col0, dim, a.qscale);
    T new_k{}, new_v{};
    const bool has_new = MODE != kVisitUniform || a.k;
    if (has_new && tid < dim) { new_k = kin[qrow + tid]; new_v = vin[qrow + tid]; }
    const int offset = MODE == kVisitRank ? s_len[b] : MODE == kVisitUniform ? a.uniform_len - 1 : a.offsets[b];
#ifdef MT_DECODE_TIMELINE
    if (item == blockIdx.x) tl_loads = stamp_after(offset + physical);
#endif

    const int64_t L = offset < 0 ? 0 : int64_t(offset) + 1;
    T* orow = out + bh * dim;
    if (L > cap) {
      // A token beyond the table's columns reads as a missing page: NaN row.
      if (split == 0)
        for (int t = tid; t < dim; t += NT) orow[t] = from_f32<DT>(NAN);
      continue;
    }
    const int nsplit = L == 0 ? 1 : int((uint32_t(L) + uint32_t(a.split_tokens) - 1) / uint32_t(a.split_tokens));
    if (split >= nsplit) continue;
    const int64_t t0 = t0i;
    const int64_t t1 = L < t0 + a.split_tokens ? L : t0 + a.split_tokens;
    const bool owns_new = has_new && L > 0 && split == nsplit - 1;
    const int ntok_paged = int((owns_new ? t1 - 1 : t1) - t0);  // tokens read from pages
    // Staged in LDS once the loads above are in flight: the slab table (first
    // item only) and the new token's K/V row, which is needed only after the
    // stream and so holds no registers during it.
    if (!slabs_staged) {
      if (!slabs_loaded) load_slabs();
#pragma unroll
      for (int j = 0; j < SLABS_PER_THREAD; ++j)
        if (tid + j * NT < kLdsSlabs) s_slabs[tid + j * NT] = slab_reg[j];
    }
    if (tid < (VEC == kRowsPadded ? D : dim)) { s_new[0][tid] = new_k; s_new[1][tid] = new_v; }
    __syncthreads();
    slabs_staged = true;
#ifdef MT_DECODE_TIMELINE
    if (item == blockIdx.x) tl_barrier = wall_clock64();
#endif
    auto slab_of = [&](int physical) -> uint64_t {
      return lds_slabs ? s_slabs[slab_index(physical, g)] : a.slabs[slab_index(physical, g)];
    };
    auto resolve = [&](int physical) -> const T* {
      return physical_in_pool(physical, g) ? page_in_slab<T>(slab_of(physical), physical, g, head)
                                           : nullptr;
    };

    const T* my_page = (slot_i < rb_per_wave && t0 + slot_tok < t1) ? resolve(physical) : nullptr;
    // The new token's page (wave 0, scalar loads; needed only after the stream).
    const T* new_page = nullptr;
    if (owns_new && wave == 0) {
      const int64_t logical = (L - 1) >> g.log2_page;
      new_page = logical < g.columns ? resolve(table_row[logical]) : nullptr;
    }

    Softmax<DL, G> st;
    st.init();
#ifdef MT_DECODE_TIMELINE
    if (item == blockIdx.x) tl_stream = wall_clock64();
#endif
    stream_wave<DT, D, VEC, U, STAGES, G>(st, qv, reinterpret_cast<uint64_t>(my_page), ntok_paged,
                                           wave, WAVES, g, dim);

    if (owns_new && wave == 0) {
      // The new token: read from the K/V inputs, scored by group 0 of wave 0,
      // and written into its page when the page exists (reference append,
      // src/paged_attention_kernel.cu:23-33). A missing page reads as NaN.
      const int64_t pos = L - 1;
      Chunk<DT, DL, VEC, G> kn, vn;
      kn.load_lds(&s_new[0][col0], col0, dim);
      vn.load_lds(&s_new[1][col0], col0, dim);
      if (lane < G && new_page) {
        T* kp = const_cast<T*>(new_page) + (pos & (g.page_size - 1)) * dim + col0;
        T* vp = kp + g.kind_stride;
        if constexpr (VEC) {
#pragma unroll
          for (int i = 0; i < Chunk<DT, DL, VEC, G>::NV; ++i) {
            if (VEC == kRowsPadded && col0 + i * G * per16<DT>() >= dim) break;
            global_view(reinterpret_cast<u32x4*>(kp))[i * G] = kn.raw[i];
            global_view(reinterpret_cast<u32x4*>(vp))[i * G] = vn.raw[i];
          }
        } else {
          for (int i = 0; i < DL && col0 + i < dim; ++i) {
            kp[i] = kin[qrow + col0 + i];
            vp[i] = vin[qrow + col0 + i];
          }
        }
      }
      if (!new_page) { kn.nan_fill(); vn.nan_fill(); }
      const float sc = qv.score(kn);
      if (lane < G) {
        float vf[DL];
        vn.to_float(vf);
        st.add(sc, vf);
      }
    }

    // Row merges by DPP, then the WAVES * 4 row states meet in LDS.
    st.row_merge();
    const int row = lane >> 4;
    if ((lane & 15) < G) {
      const int si = wave * 4 + row;
#pragma unroll
      for (int i = 0; i < DL; ++i) s_acc[si][col0 + Chunk<DT, DL, VEC, G>::col_of(i)] = st.acc[i];
      if ((lane & 15) == 0) { s_m[si] = st.m; s_l[si] = st.l; }
    }
    __syncthreads();

    // Two-level merge with every thread busy: group q of D threads merges
    // row states [q*PER, (q+1)*PER) per dim, then D threads merge the groups.
    {
      const int d = tid % D, q = tid / D;
      float M = -INFINITY;
#pragma unroll
      for (int j = 0; j < PER; ++j) M = fmaxf(M, s_m[q * PER + j]);
      float lq = 0.f, aq = 0.f;
#pragma unroll
      for (int j = 0; j < PER; ++j) {
        const int w = q * PER + j;
        const float mw = s_m[w];
        const float sc = (mw == -INFINITY) ? 0.f : fast_exp2(mw - M);
        lq = fmaf(s_l[w], sc, lq);
        aq = fmaf(s_acc[w][d], sc, aq);
      }
      s2_acc[q][d] = aq;
      if (d == 0) { s2_m[q] = M; s2_l[q] = lq; }
    }
    __syncthreads();

    const int t = tid;
    if (t < dim) {
      float M = -INFINITY;
#pragma unroll
      for (int q = 0; q < GROUPS; ++q) M = fmaxf(M, s2_m[q]);
      float lsum = 0.f, asum = 0.f;
#pragma unroll
      for (int q = 0; q < GROUPS; ++q) {
        const float mq = s2_m[q];
        const float sc = (mq == -INFINITY) ? 0.f : fast_exp2(mq - M);
        lsum = fmaf(s2_l[q], sc, lsum);
        asum = fmaf(s2_acc[q][t], sc, asum);
      }
      if (nsplit == 1) {
        orow[t] = from_f32<DT>(finalize(asum, lsum));
      } else {
        float* part = a.partials + (bh * a.nsplit_max + split) * PSTRIDE;
        part[2 + t] = asum;
        if (t == 0) { part[0] = M; part[1] = lsum; }
      }
    }
    __syncthreads();  // LDS is reused by the next item
  }
#ifdef MT_DECODE_TIMELINE
  if (tid == 0 && blockIdx.x < unsigned(kTimelineMax)) {
    uint64_t* rec = g_decode_timeline + kTimelineFields * blockIdx.x;
    rec[0] = tl_start;
    rec[1] = tl_entry;
    rec[2] = tl_loads;
    rec[3] = tl_barrier;
    rec[4] = tl_stream;
    rec[5] = wall_clock64();
    rec[6] = __builtin_amdgcn_s_getreg(4 | (31 << 11));   // HW_ID: wave, SIMD, CU, SH, SE
    rec[7] = __builtin_amdgcn_s_getreg(20 | (15 << 11));  // XCC_ID
  }
#endif
}

// Split-context reduction: for every (request, head) whose context spans more
// than one split, merge the per-split (max, denominator, accumulator) partials
// with the log-sum-exp rule and write the output row. Rows with a single split
// were written by decode_kernel. The kernel boundary orders it after the
// partial writes, so no device-scope fences are needed.
template <int DT, int D>
__global__ __launch_bounds__(128) void merge_kernel(DecodeArgs a) {
  using T = typename Elem<DT>::T;
  constexpr int PSTRIDE = D + 2;
  const Geometry& g = a.g;
  const int dim = g.dim;
  // a device-built list's counts, bounded by its capacity
  const int64_t work_items = a.work_count ? std::min(int64_t(a.work_count[0]), a.items / g.heads) : a.work_items;
  const int64_t rows = a.work_count ? std::min(a.work_count[1], a.batch) : a.work ? a.merge_rows : a.batch;
  const int64_t count = rows * g.heads;
  const int64_t cap = int64_t(g.columns) * g.page_size;
  T* out = static_cast<T*>(a.out);
  for (int64_t i = blockIdx.x; i < count; i += gridDim.x) {
    const int64_t m = i / g.heads;
    const int head = int(i - m * g.heads);
    const int b = a.work ? a.work[2 * work_items + m] : int(m);
    if (b < 0 || b >= a.batch) continue;
    const int64_t bh = int64_t(b) * g.heads + head;
    const float* base = a.partials + bh * a.nsplit_max * PSTRIDE;
    const int t = threadIdx.x;
    // Partials of up to kChunk splits are loaded per pass; the first pass is
    // issued together with the context-length read that says how many exist.
    constexpr int kChunk = 8;
    float pm[kChunk], pl[kChunk], pa[kChunk];
    auto load_chunk = [&](int s0) {
#pragma unroll
      for (int j = 0; j < kChunk; ++j) {
        const int sj = s0 + j < a.nsplit_max ? s0 + j : a.nsplit_max - 1;
        pm[j] = base[sj * PSTRIDE];
        pl[j] = base[sj * PSTRIDE + 1];
        pa[j] = t < dim ? base[sj * PSTRIDE + 2 + t] : 0.f;
      }
    };
    load_chunk(0);
    const int offset = a.offsets ? a.offsets[b] : a.uniform_len - 1;
    const int64_t L = offset < 0 ? 0 : int64_t(offset) + 1;
    if (L > cap) continue;
    const int nsplit = L == 0 ? 1 : int((L + a.split_tokens - 1) / a.split_tokens);
    if (nsplit == 1) continue;
    // Online log-sum-exp merge over the chunks, a chunk's terms added in pairs:
    // one chain over a row's splits rounds at each of them, and a row of many
    // splits then ends further from 64 bits than one of few (fp32, one row of
    // 8000 tokens x 12 heads: 2.17e-7 in 63 splits, 1.96e-7 in 8; in pairs
    // 1.87e-7 in 63, in the same 16.3 us).
    float M = -INFINITY, lsum = 0.f, asum = 0.f;
    for (int s0 = 0; s0 < nsplit; s0 += kChunk) {
      if (s0 > 0) load_chunk(s0);
      float cm = M;
#pragma unroll
      for (int j = 0; j < kChunk; ++j)
        if (s0 + j < nsplit) cm = fmaxf(cm, pm[j]);
      const float rescale = (M == -INFINITY) ? 0.f : fast_exp2(M - cm);
      float tl[kChunk], ta[kChunk];
#pragma unroll
      for (int j = 0; j < kChunk; ++j) {
        const float sc = s0 + j < nsplit && pm[j] != -INFINITY ? fast_exp2(pm[j] - cm) : 0.f;
        tl[j] = s0 + j < nsplit ? pl[j] * sc : 0.f;
        ta[j] = s0 + j < nsplit ? pa[j] * sc : 0.f;
      }
#pragma unroll
      for (int w = kChunk / 2; w > 0; w /= 2)
#pragma unroll
        for (int j = 0; j < w; ++j) { tl[j] += tl[j + w]; ta[j] += ta[j + w]; }
      lsum = fmaf(lsum, rescale, tl[0]);
      asum = fmaf(asum, rescale, ta[0]);
      M = cm;
    }
    if (t < dim) out[bh * dim + t] = from_f32<DT>(finalize(asum, lsum));
  }
}

// Work list of a decode launch built on the device from offsets[], for the
// reference entry, which has no work-list argument: the list a host caller
// builds from the lengths it knows (paged_ops.decode_work_list), bit for bit.
// Row r attends L = offsets[r] + 1 keys (0 for a negative offset) in
// n = max(1, ceil(L / S)) splits: splits 0 .. n-2 of S tokens and a last one
// of t = L - (n-1) S (a row past its table: one entry, t = 0, which the
// decode turns into a NaN row). Entries are ordered by tokens descending,
// then row, then split; position p of that order goes to slot f(p) of
// passes of `per` entries with every other pass reversed. The S-token
// entries form the first run, in (row, split) order, so entry (r, s) of it
// sits at the count of S-token entries of rows before r, plus s (a prefix
// sum). The last splits of fewer than S tokens follow, sorted by (tokens
// descending, row): a stable LDS radix sort of the rows on S - 1 - t, rows
// whose last split is full keyed past every other. The rows with more than
// one split follow the list, ascending: list[2W + m]. count = (W, M).
struct OrderArgs {
  const int* offsets;
  int* list;   // 2 * capacity + batch ints
  int* count;  // [2]
  int batch, split_tokens, per;
  int capacity;  // (row, split) pairs the list holds: batch * nsplit_max
  int64_t cap;   // tokens a table holds
};

constexpr int kOrderWaves = kOrderThreads / 64;
constexpr int kRadixBits = 6;
constexpr int kRadixDigits = 1 << kRadixBits;  // one digit per lane
constexpr int kOrderBlocks = kOrderRows / kOrderThreads;  // rows per thread (striped)
constexpr int kRadixCounts = kRadixDigits * kOrderBlocks * kOrderWaves;
static_assert(kRadixDigits == 64 && kRadixCounts % kOrderThreads == 0, "order_kernel layout");

// Exclusive prefix sums of V per-thread values over a workgroup of
// kOrderThreads, in thread order; totals in tot[].
template <int V>
__device__ __forceinline__ void order_scan(int (&v)[V], int (&tot)[V], int (*s_wave)[kOrderWaves]) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  int inc[V];
#pragma unroll
  for (int j = 0; j < V; ++j) inc[j] = wave_inclusive_add(v[j]);
  if (lane == 63) {
#pragma unroll
    for (int j = 0; j < V; ++j) s_wave[j][wave] = inc[j];
  }
  __syncthreads();
#pragma unroll
  for (int j = 0; j < V; ++j) {
    int before = 0, all = 0;
#pragma unroll
    for (int w = 0; w < kOrderWaves; ++w) {
      const int x = s_wave[j][w];
      before += w < wave ? x : 0;
      all += x;
    }
    v[j] = before + inc[j] - v[j];
    tot[j] = all;
  }
  __syncthreads();
}

__global__ __launch_bounds__(kOrderThreads) void order_kernel(OrderArgs o) {
  __shared__ int s_full[kOrderRows];   // S-token entries of the rows before
  __shared__ int s_merge[kOrderRows];  // merge rows before
  __shared__ int s_key[2][kOrderRows];  // radix sort: keys, ping-pong
  __shared__ short s_row[2][kOrderRows];
  // per (digit, block, wave) counts of one radix pass, scanned in that order
  __shared__ int s_cnt[kRadixCounts];
  __shared__ int s_wave[2 * kOrderBlocks + kOrderBlocks][kOrderWaves];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int b = o.batch;
  const uint32_t S = uint32_t(o.split_tokens);
  const int blocks = (b + kOrderThreads - 1) / kOrderThreads;
  // Striped rows: thread tid holds rows tid + j * kOrderThreads.
  int n[kOrderBlocks], t[kOrderBlocks];
#pragma unroll
  for (int j = 0; j < kOrderBlocks; ++j) {
    const int r = tid + j * kOrderThreads;
    n[j] = 0; t[j] = 0;
    if (r < b) {
      const int off = o.offsets[r];
      const uint32_t L = off < 0 ? 0u : uint32_t(off) + 1u;
      if (int64_t(L) > o.cap) {
        n[j] = 1;
      } else {
        const uint32_t nn = L == 0 ? 1u : (L + S - 1) / S;
        n[j] = int(nn);
        t[j] = int(L - (nn - 1) * S);
      }
    }
    // sort key: S - 1 - t ascending is tokens descending; a full last split
    // (not sorted here) and padding rows go behind every other
    s_key[0][r] = (r < b && t[j] < int(S)) ? int(S) - 1 - t[j] : 4095;
    s_row[0][r] = short(r);
  }
  // Prefix sums in row order of the S-token entries, the last splits below
  // S and the merge rows: block j's sums follow block j - 1's.
  int v[3 * kOrderBlocks], tot[3 * kOrderBlocks];
#pragma unroll
  for (int j = 0; j < kOrderBlocks; ++j) {
    const bool in = tid + j * kOrderThreads < b;
    v[3 * j] = in ? n[j] - 1 + (t[j] == int(S)) : 0;
    v[3 * j + 1] = in ? int(t[j] < int(S)) : 0;
    v[3 * j + 2] = in ? int(n[j] > 1) : 0;
  }
  order_scan<3 * kOrderBlocks>(v, tot, s_wave);
  int full_total = 0, last_count = 0, M = 0;
#pragma unroll
  for (int j = 0; j < kOrderBlocks; ++j) {
    const int r = tid + j * kOrderThreads;
    if (r < b) { s_full[r] = full_total + v[3 * j]; s_merge[r] = M + v[3 * j + 2]; }
    full_total += tot[3 * j];
    last_count += tot[3 * j + 1];
    M += tot[3 * j + 2];
  }
  const int W = full_total + last_count;
  // Stable LSD radix sort of (key, row) over 12 bits, 6 per pass. Six
  // ballots give every lane the lanes of its wave with the same digit, and
  // lane d the count of digit d in its wave; a position is the scanned count
  // of (digit, block, wave) plus the same-digit lanes below it.
  const uint64_t lt = (uint64_t(1) << lane) - 1;
  int src = 0;
  for (int shift = 0; shift < 12; shift += kRadixBits, src ^= 1) {
    int digit[kOrderBlocks], within[kOrderBlocks];
#pragma unroll
    for (int j = 0; j < kOrderBlocks; ++j) {
      digit[j] = 0; within[j] = 0;
      int count = 0;
      if (j < blocks) {
        const int d = (s_key[src][tid + j * kOrderThreads] >> shift) & (kRadixDigits - 1);
        uint64_t peers = ~uint64_t(0), mine = ~uint64_t(0);
#pragma unroll
        for (int bit = 0; bit < kRadixBits; ++bit) {
          const uint64_t m = __ballot((d >> bit) & 1);
          peers &= ((d >> bit) & 1) ? m : ~m;
          mine &= ((lane >> bit) & 1) ? m : ~m;
        }
        digit[j] = d;
        within[j] = __popcll(peers & lt);
        count = __popcll(mine);
      }
      s_cnt[(lane * kOrderBlocks + j) * kOrderWaves + wave] = count;
    }
    __syncthreads();
    {
      constexpr int PER = kRadixCounts / kOrderThreads;
      int c[PER], sv[1] = {0}, st[1];
#pragma unroll
      for (int i = 0; i < PER; ++i) { c[i] = s_cnt[tid * PER + i]; sv[0] += c[i]; }
      order_scan<1>(sv, st, s_wave);
      int run = sv[0];
#pragma unroll
      for (int i = 0; i < PER; ++i) { s_cnt[tid * PER + i] = run; run += c[i]; }
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < kOrderBlocks; ++j) {
      if (j < blocks) {
        const int i = tid + j * kOrderThreads;
        const int pos = s_cnt[(digit[j] * kOrderBlocks + j) * kOrderWaves + wave] + within[j];
        if (unsigned(pos) < unsigned(kOrderRows)) {
          s_key[src ^ 1][pos] = s_key[src][i];
          s_row[src ^ 1][pos] = s_row[src][i];
        }
      }
    }
    __syncthreads();
  }
  const int per = o.per;
  auto place = [&](int p, int r, int s) {
    const int pass = p / per, within = p - pass * per;
    const int width = min(per, W - pass * per);
    const int f = pass * per + ((pass & 1) ? width - 1 - within : within);
    if (unsigned(f) < unsigned(min(W, o.capacity))) {
      o.list[2 * f] = r;
      o.list[2 * f + 1] = s;
    }
  };
  // The sorted last splits below S.
  for (int p = tid; p < last_count; p += kOrderThreads) {
    const int r = s_row[src][p];
    if (unsigned(r) >= unsigned(b)) continue;
    const int full = (r + 1 < b ? s_full[r + 1] : full_total) - s_full[r];
    place(full_total + p, r, full);
  }
  // Each row's S-token splits and its merge entry.
#pragma unroll
  for (int j = 0; j < kOrderBlocks; ++j) {
    const int r = tid + j * kOrderThreads;
    if (r < b) {
      const int full = n[j] - 1 + (t[j] == int(S));
      for (int s = 0; s < full; ++s) place(s_full[r] + s, r, s);
      const int m = s_merge[r];
      if (n[j] > 1 && W <= o.capacity && unsigned(m) < unsigned(b)) o.list[2 * W + m] = r;
    }
  }
  if (tid == 0) { o.count[0] = W; o.count[1] = M; }
}

struct QueryArgs {
  void* out;
  const void* q;
  const uint64_t* slabs;
  const int* table;
  int batch, nq, nk, offset;
  float qscale;
  int64_t items;
  Geometry g;
  // Element strides of q and out per request, head and query: [b, h, nq, d]
  // by default, [b, nq, row] for head-interleaved token rows.
  int64_t q_b, q_h, q_r, o_b, o_h, o_r;
  // The prompt's own K/V rows (strides of q), or null. When set (causal
  // kernel only), keys at or past the offset are read from these rows and the
  // workgroup of each query tile writes its tokens' K/V to their pages, which
  // replaces a separate append.
  const void* k;
  const void* v;
  // Key-split prefill: per (slot, head, query of the tile) D accumulators,
  // max and denominator of one piece's keys, merged by uniform_merge_kernel or
  // ragged_merge_kernel.
  float* partials;
};

// Floats per query in the key-split partials: D accumulators, then max and
// denominator, padded so every row starts 16-byte aligned.
template <int D>
constexpr int pf_part_row() { return D + 4; }

// Causal paged attention for nq >= 1 queries per (request, head)
// (reference paged_forward with offsets == nullptr, src/paged_attention_kernel.cu:35-85):
// query qi attends keys kj < nk with kj <= offset + qi. One wave per query,
// four queries per workgroup; page bases are resolved per 2048-token chunk.
template <int DT, int D, int VEC, int U>
__global__ __launch_bounds__(kThreads) void query_kernel(QueryArgs a) {
  using T = typename Elem<DT>::T;
  constexpr int DL = D / kGroup;
  __shared__ const T* s_page[kMaxSplitPages];
  const Geometry& g = a.g;
  const int dim = VEC == kRowsFull ? D : g.dim;
  const int tid = threadIdx.x;
  const int wave = tid >> 6;
  const int lane = tid & (kWave - 1);
  const int col0 = Chunk<DT, DL, VEC, kGroup>::first_col(lane & 3);
  const int qblocks = (a.nq + kWaves - 1) / kWaves;
  const T* qp = static_cast<const T*>(a.q);
  T* out = static_cast<T*>(a.out);
  for (int64_t item = blockIdx.x; item < a.items; item += gridDim.x) {
    const int64_t bh = item / qblocks;
    const int qb = int(item - bh * qblocks);
    const int b = int(bh / g.heads), head = int(bh - int64_t(b) * g.heads);
    const int qi = qb * kWaves + wave;
    const bool has_q = qi < a.nq;
    const int64_t klen = has_q ? (int64_t(a.offset) + qi + 1 < a.nk ? int64_t(a.offset) + qi + 1 : a.nk) : 0;
    const int qlast = (qb * kWaves + kWaves - 1 < a.nq ? qb * kWaves + kWaves - 1 : a.nq - 1);
    const int64_t kmax = int64_t(a.offset) + qlast + 1 < a.nk ? int64_t(a.offset) + qlast + 1 : a.nk;
    const int* table_row = a.table + int64_t(b) * g.columns;
    Query<DT, D, VEC> qv;
    qv.load(qp + b * a.q_b + head * a.q_h + (has_q ? qi : 0) * a.q_r, col0, dim, a.qscale);
    Softmax<DL> st;
    st.init();
    for (int64_t c0 = 0; c0 < kmax; c0 += kMaxSplitTokens) {
      const int64_t c1 = c0 + kMaxSplitTokens < kmax ? c0 + kMaxSplitTokens : kmax;
      const int npg = int((c1 - c0 + g.page_size - 1) >> g.log2_page);
      __syncthreads();
      for (int j = tid; j < npg; j += kThreads)
        s_page[j] = page_base<T>(a.slabs, table_row, (c0 >> g.log2_page) + j, g, head);
      __syncthreads();
      const int64_t mine = klen - c0 < c1 - c0 ? klen - c0 : c1 - c0;
      if (mine > 0) stream_rows<DT, D, VEC, U, 2>(st, qv, s_page, int(mine), 0, 1, g, dim);
    }
    st.wave_merge();
    if (has_q && lane < kGroup) {
      T* orow = out + b * a.o_b + head * a.o_h + qi * a.o_r;
      for (int i = 0; i < DL; ++i) {
        const int c = col0 + Chunk<DT, DL, VEC, kGroup>::col_of(i);
        if (c < dim) orow[c] = from_f32<DT>(finalize(st.acc[i], st.l));
      }
    }
    __syncthreads();
  }
}

struct AppendArgs {
  const void* k;
  const void* v;
  const uint64_t* slabs;
  const int* table;
  int batch, n, offset;
  int64_t vectors;  // number of per-thread units
  Geometry g;
  int64_t src_b, src_h, src_r;  // element strides of k/v per request, head and token
};


// ---------------------------------------------------------------------------
// Causal paged attention of several queries per request on the matrix cores,
// same semantics as query_kernel: query qi attends keys kj < nk with
// kj <= offset + qi, and a query whose keys touch a missing page reads NaN.
//
// A workgroup owns a tile of 32 QT queries of one (request, head). It has
// QT x KG waves: wave (qt, kg) holds 32 of the tile's queries and takes every
// KG-th block of KB keys; the KG groups' softmax states meet in LDS at the
// end. A staged round is KG blocks, copied from the pages (or from the
// prompt's own K/V rows) to LDS by all waves while the round before it is
// computed.
//
// Per block a wave computes S^T = K Q^T with 32x32 MFMAs (keys x queries, so
// two lanes share a query and each holds half of the block's scores of it),
// updates that query's online softmax in registers and accumulates
// O^T += V^T P^T, feeding the scores' own register layout as the B operand
// (the MFMA sums over its k index in any order, so A's key order is chosen to
// match). K and V both lie row-major in LDS; for 16-bit types V's operand is
// read transposed by ds_read_b64_tr_b16, for fp32 a lane reads single
// elements. Rows are swizzled in 16-byte chunks so that these reads are free
// of bank conflicts. Rounds go from memory to LDS without passing through
// registers, so that a wave's registers hold its queries, scores and output:
// two to four waves per SIMD, which is what the kernel lives on. Its bound is
// the issue of a block's ~170 VALU instructions (exponentials, the split of
// P) between 12 MFMAs; rounds deeper in flight, and all loads through
// registers, measured the same or slower. Against the 16-query waves with V
// transposed by 2-byte LDS stores that it replaces (us per call, bf16): 2048
// tokens at offset 2048 x 16 heads 59-65 by box against 134 (400-435 against 192
// TFLOP/s), 1000 tokens x 16 heads 15.0 against 22.7, 16 prompts of 32-512 tokens
// x 12 heads fp16 19.0-19.8 against 26.3; fp32, which query_kernel read K/V for
// once per query: 4 x 333 tokens x 12 heads 22 against 106.
//
// For fp16/bf16 the MFMA takes P in the input type, so P is split into a high
// and a low part of that type (two MFMAs): the weights keep about 16 (bf16)
// or 22 (fp16) significant bits instead of 8 or 11, which holds the output to
// the fp32 path's accuracy when |V| is large. fp32 runs on the fp32 MFMA
// (v_mfma_f32_32x32x2_f32), nothing is rounded below fp32.
//
// The running reference of the exponentials moves only when a score exceeds
// it by kRescale (base 2), so most blocks skip the rescaling of O: weights
// are then at most 2^kRescale, which neither fp32 nor the hi/lo split minds.
// fp16 has nothing below 2^-24, so its weights are taken 2^kHalfShift larger,
// denominator and all: the split then keeps a weight's 22 bits down to 2^-11 of
// the largest and ends at 2^-33 of it. Ending at 2^-24, weights of 2.9e-6 beside
// one of 1 in every block lost 1 % of their sum.
constexpr int kPfWindowPages = 512;  // page bases resolved into LDS at a time
constexpr int kPfBlock = 64;         // keys per unit of a split over workgroups
constexpr float kRescale = 6.f;
constexpr float kHalfShift = 9.f;  // 2^(kRescale + kHalfShift) is below fp16's largest
constexpr int kPfMinQueries = 2;     // a single query runs the decode kernel or query_kernel

// x of lanes l and l ^ 32 (in either order): the permlane swap of two copies
// of x leaves x[l % 32] in one and x[l % 32 + 32] in the other.
__device__ __forceinline__ float max_halves(float x) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
__device__ __forceinline__ float add_halves(float x) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

// Two probabilities as the high and low packed MFMA operands: hi = p rounded
// to the input type (fp16 toward zero, one packed conversion; bf16 to nearest
// even), lo = the remainder, rounded the same way.
template <int DT>
struct SplitP;
template <>
struct SplitP<kF16> {
  static __device__ __forceinline__ void split(float p0, float p1, uint32_t& hi, uint32_t& lo) {
    const auto h = __builtin_amdgcn_cvt_pkrtz(p0, p1);
    hi = __builtin_bit_cast(uint32_t, h);
    lo = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_pkrtz(p0 - float(h[0]), p1 - float(h[1])));
  }
};
template <>
struct SplitP<kBF16> {
  typedef __bf16 bf2 __attribute__((ext_vector_type(2)));
  static __device__ __forceinline__ void split(float p0, float p1, uint32_t& hi, uint32_t& lo) {
    const bf2 h = {static_cast<__bf16>(p0), static_cast<__bf16>(p1)};
    hi = __builtin_bit_cast(uint32_t, h);
    asm("" : "+v"(hi));  // keeps the halves' unpacking from becoming two more conversions
    const float r0 = p0 - __uint_as_float(hi << 16), r1 = p1 - __uint_as_float(hi & 0xffff0000u);
    const bf2 r = {static_cast<__bf16>(r0), static_cast<__bf16>(r1)};
    lo = __builtin_bit_cast(uint32_t, r);
  }
};

// What one workgroup works on: query tile `tile` of `head` of a request whose
// queries start at element q0 of q (o0 of out), nq queries at key offset
// `offset` over the pages of table_row.
struct PfItem {
  int tile, head, nq, offset;
  int64_t q0, o0;
  const int* table_row;
  int kb0, kb1;  // kPfBlock-key blocks [kb0, kb1) of the tile's keys that this item attends
  int slot;      // partials slot of a split tile, -1: the item writes the output rows
};

constexpr int kAllKeyBlocks = 1 << 24;

// Blocks of kPfBlock keys that query tile `tile` (tq queries a tile) attends.
__host__ __device__ __forceinline__ int key_blocks(int tile, int tq, int nq, int offset) {
  const int64_t end = int64_t(tile + 1) * tq < nq ? int64_t(tile + 1) * tq : nq;
  return int((offset + end + kPfBlock - 1) / kPfBlock);
}

// The uniform batch of QueryArgs (b requests of nq queries at one offset):
// items ordered by tile, last (longest) tiles first. With `share` > 0 each
// tile's keys are cut into pieces of at most `share` blocks, at most `pieces`
// per tile (a tile with one piece writes its output rows).
struct UniformItems {
  int tiles, pieces, share;
  __device__ __forceinline__ int64_t count(const QueryArgs& a) const { return a.items; }
  __device__ __forceinline__ bool get(int64_t item, const QueryArgs& a, int tq, PfItem& it) const {
    const unsigned bh_count = unsigned(a.batch) * unsigned(a.g.heads);
    const unsigned tp = unsigned(item) / bh_count;  // (tile, piece), from the last tile down
    const unsigned bh = unsigned(item) - tp * bh_count;
    const unsigned t = tp / unsigned(pieces);
    const int piece = int(tp - t * unsigned(pieces));
    const int b = int(bh / unsigned(a.g.heads));
    it.tile = tiles - 1 - int(t);
    it.head = int(bh) - b * a.g.heads;
    it.nq = a.nq;
    it.offset = a.offset;
    it.q0 = b * a.q_b + it.head * a.q_h;
    it.o0 = b * a.o_b + it.head * a.o_h;
    it.table_row = a.table + int64_t(b) * a.g.columns;
    it.kb0 = 0; it.kb1 = kAllKeyBlocks; it.slot = -1;
    if (pieces > 1) {
      const int nb = key_blocks(it.tile, tq, it.nq, it.offset);
      it.kb0 = piece * share;
      it.kb1 = it.kb0 + share < nb ? it.kb0 + share : nb;
      if (nb > share) it.slot = (b * tiles + it.tile) * pieces + piece;
      return it.kb0 < nb;
    }
    return true;
  }
};

// Prompts of different lengths in one launch (token-major rows, prompt r at
// rows [first_row[r], first_row[r] + n[r]) of q/k/v/out, with its own table
// row and key offset), passed by value: every (prompt, tile) pair in the
// order of pair_prompt / pair_tile (heaviest first), times the heads.
constexpr int kRaggedPrompts = 16;
constexpr int kRaggedTiles = 256;
struct RaggedItems {
  int prompts, pairs;
  int first_row[kRaggedPrompts], n[kRaggedPrompts], offset[kRaggedPrompts];
  const int* table[kRaggedPrompts];
  unsigned char pair_prompt[kRaggedTiles];
  unsigned short pair_tile[kRaggedTiles];
  // Key blocks [kb0, kb1) of the pair's tile and its partials slot (-1: the
  // pair covers all of the tile's keys and writes the output rows).
  unsigned short pair_kb0[kRaggedTiles], pair_kb1[kRaggedTiles];
  short pair_slot[kRaggedTiles];
  __device__ __forceinline__ int64_t count(const QueryArgs& a) const { return int64_t(pairs) * a.g.heads; }
  __device__ __forceinline__ bool get(int64_t item, const QueryArgs& a, int, PfItem& it) const {
    const int p = int(unsigned(item) / unsigned(a.g.heads));
    const int r = pair_prompt[p];
    it.tile = pair_tile[p];
    it.head = int(item) - p * a.g.heads;
    it.nq = n[r];
    it.offset = offset[r];
    it.q0 = int64_t(first_row[r]) * a.q_r + it.head * a.q_h;
    it.o0 = int64_t(first_row[r]) * a.o_r + it.head * a.o_h;
    it.table_row = table[r];
    it.slot = pair_slot[p];
    it.kb0 = it.slot >= 0 ? pair_kb0[p] : 0;
    it.kb1 = it.slot >= 0 ? pair_kb1[p] : kAllKeyBlocks;
    return true;
  }
};

// Shape of a workgroup's staged round, per element type, padded head dim DP
// (64 or 128), QT x KG waves and SW, the waves per SIMD its registers are held
// to (512 registers a lane over the waves of a SIMD). With SW 4 two 8-wave
// workgroups share a compute unit and hide each other's waits; with fewer the
// operands of a block are all read before its first MFMA.
template <int DT, int DP, int QT, int KG, int SW>
struct CausalShape {
  static constexpr int ES = elem_bytes<DT>();
  static constexpr int EC = 16 / ES;     // elements per 16-byte chunk
  static constexpr int CPR = DP / EC;    // chunks per LDS row
  static constexpr int KB = 32;          // keys per group and round
  static constexpr int KI = KG * KB;     // keys per round, a multiple of every page size
  static constexpr int W = QT * KG;      // waves
  static constexpr int NT = W * kWave;
  static constexpr int NC = KI * CPR / NT;     // 16-byte chunks per lane, K and V each
  static constexpr int RW = kWave / CPR;       // rows one load instruction of a wave fills
  static constexpr int DT32 = DP / 32;
  static constexpr int OS = DP + 4;      // row stride of the groups' accumulators in LDS
  // Parts of a block's keys that an fp32 output sums on its own, four chains
  // each. Two in the shape for one key block, whose output is one chain's
  // (60 tokens, head dim 64: 1.040e-7 with one, 1.035e-7 with two, 1.031e-7 in
  // query_kernel).
  static constexpr int kSums = DP == 64 && KG == 1 ? 2 : 1;
  static constexpr int kPlane = KI * DP * ES;  // bytes of a round's K (and V)
  // Rounds of LDS: one computed, the others in flight.
  static constexpr int kRing = SW == 4 || KG <= 2 ? 2 : 131072 / (2 * kPlane) < 4 ? 131072 / (2 * kPlane) : 4;
  static constexpr size_t kStage = size_t(2 * kRing) * kPlane;
  static constexpr size_t kMerge = KG > 1 ? size_t(KG) * 32 * QT * (OS + 2) * sizeof(float) : 0;
  static constexpr size_t kLds = kStage > kMerge ? kStage : kMerge;
  static_assert(NC * NT == KI * CPR && NC >= 1 && kWave % CPR == 0, "a round divides over the workgroup");
  // Chunk p of key row r lies at chunk kpos / vpos of the row (both their own
  // inverse). K is read as 16-byte chunks of 32 consecutive rows, V as 4 rows
  // x 64 bytes (16-bit) or as two rows 4 apart x 128 bytes (fp32).
  static __device__ __forceinline__ int kpos(int r, int p) { return CPR == 8 ? p ^ ((r >> 1) & 7) : p ^ (r & 15); }
  static __device__ __forceinline__ int vpos(int r, int p) {
    if constexpr (DT == kF32) return p ^ (((r >> 2) & 1) << 3);
    else return CPR == 8 ? p ^ (((r >> 1) & 1) << 2) : p ^ ((r & 3) << 2);
  }
};

typedef float floatx16 __attribute__((ext_vector_type(16)));

template <int DT>
__device__ __forceinline__ floatx16 mfma32(const u32x4& x, const u32x4& y, const floatx16& c) {
  if constexpr (DT == kF16)
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(Mfma<kF16>::v8, x),
                                                  __builtin_bit_cast(Mfma<kF16>::v8, y), c, 0, 0, 0);
  else
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(Mfma<kBF16>::v8, x),
                                                   __builtin_bit_cast(Mfma<kBF16>::v8, y), c, 0, 0, 0);
}

// Four keys of one dim: lane t of each 16 lanes passes row t / 4, columns
// 4 (t % 4) .. + 3 of a 4 x 16 block of 16-bit elements and receives column t.
__device__ __forceinline__ uint2 read_transposed(const void* p) {
  typedef short s4 __attribute__((ext_vector_type(4)));
  const s4 r = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s4*)(p));
  return __builtin_bit_cast(uint2, r);
}

// acc / l by the output rule (0 for l = 0, NaN for a NaN l) with inv =
// inverse(l): one multiplication for 16-bit results, corrected to fp32's
// rounding for fp32 ones.
__device__ __forceinline__ float inverse(float l) { return l > 0.f ? 1.f / l : (isnan(l) ? NAN : 0.f); }
template <int DT>
__device__ __forceinline__ float divided(float acc, float l, float inv) {
  const float x = acc * inv;
  if constexpr (DT == kF32) return fabsf(x) < INFINITY ? fmaf(fmaf(-x, l, acc), inv, x) : x;
  else return x;
}

// What a staged row reads where there is nothing to read: NaN keys (a missing
// page: its scores are NaN) and zeros, each a 16-byte load.
__device__ __align__(16) const uint32_t g_fill[8] = {~0u, ~0u, ~0u, ~0u, 0u, 0u, 0u, 0u};

// Copies 16 bytes per lane from global memory to LDS without passing through
// registers: lane l's bytes land at lds + 16 l. The compiler does not see the
// write, nor count it in its own waits: wait_staged() before the barrier that
// publishes a round.
__device__ __forceinline__ void stage16(const void* src, uint32_t lds) {
  asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off" ::"v"(src), "s"(lds) : "m0", "memory");
}
__device__ __forceinline__ void stage16(const void* base, uint32_t offset, uint32_t lds) {
  asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %0" ::"s"(base), "v"(offset), "s"(lds)
               : "m0", "memory");
}
__device__ __forceinline__ const char* uniform(const char* p) {
  const uint64_t x = reinterpret_cast<uintptr_t>(p);
  const uint32_t lo = __builtin_amdgcn_readfirstlane(uint32_t(x)), hi = __builtin_amdgcn_readfirstlane(uint32_t(x >> 32));
  return reinterpret_cast<const char*>(uint64_t(hi) << 32 | lo);
}
// Waits until at most N of this wave's memory operations are outstanding.
template <int N>
__device__ __forceinline__ void wait_staged() { asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory"); }

// Queries of item `item` (tiles of TQ) that the matrix cores left non-finite,
// a bit each of 32-query group t in `left`: every WAVES-th of them from the
// `wave`-th on is attended once more, by one wave on the VALU, over the keys it
// attends and no others. On the matrix cores a key that a query does not attend
// has weight 0, and 0 * Inf or 0 * NaN of its V is NaN; so is the 0 * Inf of a
// weight's low part. For kernels whose arguments are (QueryArgs, Items): they
// are read anew, and the walk is kept small (a lane scores a key, then holds one
// or two columns of the output), so that this rare path costs the kernel's own
// no registers. Finite calls, us without and with the check: 16 prompts of
// 32-512 tokens fp16 19.6 and 19.6, 4 x 333 tokens fp32 25.6 and 26.1.
template <int DT, int DP, int TQ, int WAVES, class Items, bool FUSED>
__device__ __forceinline__ void attend_again(int64_t item, int t, int wave, uint32_t left) {
  using T = typename Elem<DT>::T;
  constexpr int E = per16<DT>(), COLS = DP / kWave;
  struct Args { QueryArgs a; Items items; };
  uint64_t at = reinterpret_cast<uintptr_t>(__builtin_amdgcn_kernarg_segment_ptr());
  asm volatile("" : "+s"(at));
  const QueryArgs& a = reinterpret_cast<const Args*>(at)->a;
  const Geometry& g = a.g;
  PfItem it;
  reinterpret_cast<const Args*>(at)->items.get(item, a, TQ, it);
  int lane = threadIdx.x & (kWave - 1);
  asm volatile("" : "+v"(lane));
  const int kend = it.offset + ((it.tile + 1) * TQ < it.nq ? (it.tile + 1) * TQ : it.nq);
  const int kstop = int64_t(it.kb1) * kPfBlock < kend ? it.kb1 * kPfBlock : kend;
#pragma unroll 1
  for (int turn = 0; left; left &= left - 1, ++turn) {
    if (turn % WAVES != wave) continue;
    const int q = 32 * t + __builtin_ctz(left);
    const int row = it.tile * TQ + q;
    const int k1 = min(kstop, it.offset + row + 1);
    const T* qrow = static_cast<const T*>(a.q) + it.q0 + row * a.q_r;
    float m = -INFINITY, l = 0.f, acc[COLS];
#pragma unroll
    for (int e = 0; e < COLS; ++e) acc[e] = 0.f;
#pragma unroll 1
    for (int k0 = it.kb0 * kPfBlock; k0 < k1; k0 += kWave) {
      const int key = k0 + lane;
      const T* page = key < k1 ? page_base<T>(a.slabs, it.table_row, key >> g.log2_page, g, it.head) : nullptr;
      const T *kp = nullptr, *vp = nullptr;
      float s = key < k1 ? NAN : -INFINITY;  // a missing page's score is NaN
      if (page) {
        const bool fresh = FUSED && key >= it.offset;
        const int64_t row_at = fresh ? it.q0 + int64_t(key - it.offset) * a.q_r : (key & (g.page_size - 1)) * g.dim;
        kp = (fresh ? static_cast<const T*>(a.k) : page) + row_at;
        vp = (fresh ? static_cast<const T*>(a.v) : page + g.kind_stride) + row_at;
        float sum[E];
#pragma unroll
        for (int i = 0; i < E; ++i) sum[i] = 0.f;
#pragma unroll 1
        for (int c = 0; c < g.dim; c += E) {
          float x[E], y[E];
          const u32x4 qx = *global_view(reinterpret_cast<const u32x4*>(qrow + c));
          const u32x4 kx = *global_view(reinterpret_cast<const u32x4*>(kp + c));
          unpack16<DT>(qx, x);
          unpack16<DT>(kx, y);
#pragma unroll
          for (int i = 0; i < E; ++i) sum[i] = fmaf(x[i], y[i], sum[i]);
        }
#pragma unroll
        for (int w = E / 2; w > 0; w /= 2)
#pragma unroll
          for (int i = 0; i < w; ++i) sum[i] += sum[i + w];
        s = sum[0] * a.qscale;
      }
      float top = s;
#pragma unroll
      for (int w = kWave / 2; w > 0; w /= 2) top = fmaxf(top, __shfl_xor(top, w));
      top = fmaxf(m, top);
      const float alpha = m == -INFINITY ? 0.f : fast_exp2(m - top);
      const float p = fast_exp2(s - (top == -INFINITY ? 0.f : top));
      m = top;
      l = fmaf(l, alpha, p);  // this lane's keys
#pragma unroll
      for (int e = 0; e < COLS; ++e) acc[e] *= alpha;
      const uint64_t v_at = reinterpret_cast<uintptr_t>(vp);
#pragma unroll 4
      for (int j = 0; j < min(kWave, k1 - k0); ++j) {
        const float pj = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(p), j));
        const T* vj = reinterpret_cast<const T*>(
            uint64_t(uint32_t(__builtin_amdgcn_readlane(int(v_at >> 32), j))) << 32 |
            uint32_t(__builtin_amdgcn_readlane(int(v_at), j)));
#pragma unroll
        for (int e = 0; e < COLS; ++e)
          if (vj && lane + kWave * e < g.dim)
            acc[e] = fmaf(pj, to_f32<DT>(global_view(vj)[lane + kWave * e]), acc[e]);
      }
    }
#pragma unroll
    for (int w = kWave / 2; w > 0; w /= 2) l += __shfl_xor(l, w);
    float* const part =
        it.slot >= 0 ? a.partials + ((int64_t(it.slot) * g.heads + it.head) * TQ + q) * pf_part_row<DP>() : nullptr;
#pragma unroll
    for (int e = 0; e < COLS; ++e) {
      const int c = lane + kWave * e;
      if (part) part[c] = acc[e];
      else if (c < g.dim) static_cast<T*>(a.out)[it.o0 + row * a.o_r + c] = from_f32<DT>(finalize(acc[e], l));
    }
    if (part && lane == 0) *reinterpret_cast<float2*>(part + DP) = float2{m, l};
  }
}

template <int DT, int DP, int QT, int KG, int SW, class Items, bool FUSED>
__global__ __launch_bounds__(QT * KG * kWave) __attribute__((amdgpu_waves_per_eu(SW)))
void causal_kernel(QueryArgs a, Items items) {
  using T = typename Elem<DT>::T;
  using S = CausalShape<DT, DP, QT, KG, SW>;
  constexpr int EC = S::EC, CPR = S::CPR, KB = S::KB, KI = S::KI, NT = S::NT, NC = S::NC, DT32 = S::DT32;
  constexpr int TQ = 32 * QT;
  constexpr int QW = DT == kF32 ? DP / 8 : DP / 16;  // 16-byte query registers
  constexpr float kShift = DT == kF16 ? kHalfShift : 0.f;
  __shared__ const T* s_page[kPfWindowPages];
  __shared__ int s_missing;  // whether a page of a window was missing
  __shared__ uint32_t s_redo[QT];  // queries of the tile to attend alone, a bit each
  __shared__ __align__(16) char s_raw[S::kLds];
  const uint32_t lds0 = uint32_t(reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) char*)s_raw));

  const Geometry& g = a.g;
  const int dim = g.dim;
  const int chunks = dim / EC;  // 16-byte chunks per row; the rest of DP is zero
  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lane = tid & (kWave - 1);
  const int kg = wave / QT, qt = wave - kg * QT;
  const int grp = lane >> 5;  // 0..1: which half of a block's keys this lane scores
  const int col = lane & 31;  // this lane's query within its wave's 32
  const T* qp = static_cast<const T*>(a.q);
  T* out = static_cast<T*>(a.out);
  const int win_keys = kPfWindowPages << g.log2_page;
  // Load n of a wave fills rows row0 + n W RW .. of a round; this lane its row
  // `sr` further, chunk position `spos`. Pages are at most 32 keys and rounds
  // start at multiples of 32, so a row's place in its page is fixed.
  const int sr = wave * S::RW + lane / CPR, spos = lane % CPR;
  if (tid == 0) s_missing = 0;

  const int64_t n_items = items.count(a);
  for (int64_t item = blockIdx.x; item < n_items; item += gridDim.x) {
    PfItem it;
    if (!items.get(item, a, TQ, it)) continue;
    const int head = it.head;
    const int nq = it.nq, offset = it.offset;

    // B operand of S^T = K Q^T: 16-bit types dims [16 s + 8 grp, + 8) of the
    // lane's query, fp32 dims [DP / 2 * grp, + DP / 2).
    const int q0 = it.tile * TQ + qt * 32;
    const int qi = q0 + col;
    const bool q_ok = qi < nq;
    const T* qrow = qp + it.q0 + (q_ok ? qi : 0) * a.q_r;
    u32x4 qv[QW];
#pragma unroll
    for (int s = 0; s < QW; ++s) {
      const int p = DT == kF32 ? CPR / 2 * grp + s : 2 * s + grp;
      qv[s] = *global_view(reinterpret_cast<const u32x4*>(p < chunks ? qrow + p * EC : reinterpret_cast<const T*>(g_fill + 4)));
    }
    const int qpos = offset + qi;
    const bool wave_live = q0 < nq;
    const int wave_last = offset + (q0 + 31 < nq ? q0 + 31 : nq - 1);
    const int kend = offset + ((it.tile + 1) * TQ < nq ? (it.tile + 1) * TQ : nq);

    float m = -INFINITY, l = 0.f;
    floatx16 o[DT32];
#pragma unroll
    for (int d = 0; d < DT32; ++d)
#pragma unroll
      for (int i = 0; i < 16; ++i) o[d][i] = 0.f;

    // Staging of a round into LDS half `buf`. Keys past the item's range are
    // zero; a missing page is NaN in K (so its score is NaN) and zero in V (so
    // a query that does not attend it is unaffected). FUSED: keys from the
    // offset on come from the prompt's own K/V rows, and this workgroup writes
    // the keys of its own queries, [own0, kend), to the pages.
    const T* krows = FUSED ? static_cast<const T*>(a.k) + it.q0 : nullptr;
    const T* vrows = FUSED ? static_cast<const T*>(a.v) + it.q0 : nullptr;
    const int own0 = offset + it.tile * TQ;
    const uint64_t row_bytes = uint64_t(a.q_r) * S::ES;
    const bool short_rows = row_bytes * KI < (uint64_t(1) << 31);
    auto stage = [&](int k0, int w0, int w1, int buf, bool known, bool plain) {
      const uint32_t lk = lds0 + buf * 2 * S::kPlane + wave * 1024, lv = lk + S::kPlane;
      const bool whole = chunks == CPR && plain && k0 + KI <= w1;
      if (FUSED && whole && k0 >= offset && short_rows) {
        // a round of the prompt's own rows: one base
        int row = sr;
        asm volatile("" : "+v"(row));
        const char* kb = uniform(reinterpret_cast<const char*>(krows) + uint64_t(uint32_t(k0 - offset)) * row_bytes);
        const char* vb = uniform(reinterpret_cast<const char*>(vrows) + uint64_t(uint32_t(k0 - offset)) * row_bytes);
#pragma unroll
        for (int n = 0; n < NC; ++n) {
          const int r = row + n * S::W * S::RW;
          const uint32_t at = uint32_t(r) * uint32_t(row_bytes);
          stage16(kb, at + S::kpos(r, spos) * 16, lk + n * S::W * 1024);
          stage16(vb, at + S::vpos(r, spos) * 16, lv + n * S::W * 1024);
        }
      } else if (whole && (!FUSED || k0 + KI <= offset)) {
        // a round of present pages
#pragma unroll
        for (int n = 0; n < NC; ++n) {
          const int r = sr + n * S::W * S::RW;
          const T* page = s_page[(k0 + r - w0) >> g.log2_page] + (r & (g.page_size - 1)) * dim;
          stage16(page + S::kpos(r, spos) * EC, lk + n * S::W * 1024);
          stage16(page + g.kind_stride + S::vpos(r, spos) * EC, lv + n * S::W * 1024);
        }
      } else {
        int row = sr;
        asm volatile("" : "+v"(row));  // keeps this rare path's terms out of the registers of the loop
#pragma unroll
        for (int n = 0; n < NC; ++n) {
          // a block wholly past the keys is never read
          if (k0 + ((wave * S::RW + n * S::W * S::RW) & ~(KB - 1)) >= w1) continue;
          const int r = row + n * S::W * S::RW;
          const int key = k0 + r;
          const int pk = S::kpos(r, spos), pv = S::vpos(r, spos);
          const T* kp = reinterpret_cast<const T*>(g_fill + 4);
          const T* vp = kp;
          if (key < w1) {
            const T* page = known ? s_page[(key - w0) >> g.log2_page] : qp;  // qp: any page, taken as present
            if (page) {
              const bool fresh = FUSED && key >= offset;
              const int64_t at = fresh ? int64_t(uint32_t(key - offset)) * a.q_r : (r & (g.page_size - 1)) * dim;
              if (pk < chunks) kp = (fresh ? krows : page) + at + pk * EC;
              if (pv < chunks) vp = (fresh ? vrows : page + g.kind_stride) + at + pv * EC;
            } else {
              kp = reinterpret_cast<const T*>(g_fill);
            }
          }
          stage16(kp, lk + n * S::W * 1024);
          stage16(vp, lv + n * S::W * 1024);
        }
      }
    };
    // This item's keys: blocks [kb0, kb1) of [0, kend).
    const int kstart = it.kb0 * kPfBlock;
    const int kstop = int64_t(it.kb1) * kPfBlock < kend ? it.kb1 * kPfBlock : kend;
    for (int w0 = kstart; w0 < kstop; w0 += win_keys) {
      const int w1 = w0 + win_keys < kstop ? w0 + win_keys : kstop;
      const int npg = (w1 - w0 + g.page_size - 1) >> g.log2_page;
      __syncthreads();  // every wave is done with the LDS of the window before
      if (KG > 1 && tid < QT) s_redo[tid] = 0;
      // The first round is staged before the window's pages are known when it
      // holds only the prompt's own rows, and again if one turns out missing.
      const bool early = FUSED && w0 >= offset;
      bool plain = true;
#pragma unroll 1
      for (int pass = early ? 0 : 1; pass < 2; ++pass) {
        if (pass == 1) {
          bool hole = false;
          for (int j = tid; j < npg; j += NT) {
            const T* page = page_base<T>(a.slabs, it.table_row, (w0 >> g.log2_page) + j, g, head);
            s_page[j] = page;
            hole |= !page;
          }
          if (hole) s_missing = 1;  // stays set: the careful staging is right for any window
          __syncthreads();
          plain = !s_missing;
          if (!plain) wait_staged<0>();
        }
        if (pass == 0 || !early || !plain)
#pragma unroll 1
          for (int i = 0; i < S::kRing - 1 && w0 + i * KI < w1; ++i)
            stage(w0 + i * KI, w0, w1, i, pass == 1, plain);
      }
#pragma unroll
      for (int s = 0; s < QW; ++s) asm volatile("" : "+v"(qv[s]));  // the query has arrived before the loop
      int buf = 0, ahead = S::kRing - 1;  // the round's LDS, and that of the round staged next
      for (int k0 = w0; k0 < w1; k0 += KI) {
        // this wave's part of the round (a round cut short has fewer loads to count)
        if (k0 + (S::kRing - 1) * KI <= w1) wait_staged<(S::kRing - 2) * 2 * NC>();
        else wait_staged<0>();
        __syncthreads();  // everybody's, and the round before is done with
        if (k0 + (S::kRing - 1) * KI < w1) stage(k0 + (S::kRing - 1) * KI, w0, w1, ahead, true, plain);
        const T* const s_k = reinterpret_cast<const T*>(s_raw + buf * 2 * S::kPlane);
        const T* const s_v = reinterpret_cast<const T*>(s_raw + buf * 2 * S::kPlane + S::kPlane);
        ahead = buf;
        buf = buf + 1 < S::kRing ? buf + 1 : 0;
        if (FUSED && k0 + KI > own0) {
          // keys of this tile's own tokens: their page copies
          int row = sr;
          asm volatile("" : "+v"(row));
#pragma unroll
          for (int n = 0; n < NC; ++n) {
            const int r = row + n * S::W * S::RW;
            const int key = k0 + r;
            if (key < own0 || key >= w1) continue;
            T* page = const_cast<T*>(s_page[(key - w0) >> g.log2_page]);
            if (!page) continue;
            page += (r & (g.page_size - 1)) * dim;
            const int pk = S::kpos(r, spos), pv = S::vpos(r, spos);
            const u32x4 kk = *reinterpret_cast<const u32x4*>(s_k + r * DP + spos * EC);
            const u32x4 vv = *reinterpret_cast<const u32x4*>(s_v + r * DP + spos * EC);
            if (pk < chunks) *global_view(reinterpret_cast<u32x4*>(page + pk * EC)) = kk;
            if (pv < chunks) *global_view(reinterpret_cast<u32x4*>(page + g.kind_stride + pv * EC)) = vv;
          }
        }
        const int base = k0 + kg * KB;  // this wave's block
        if (!wave_live || base > wave_last || base >= w1) continue;

        // Scores: lane holds keys base + 8 (i / 4) + 4 grp + i % 4 of query qi.
        floatx16 sc;
#pragma unroll
        for (int i = 0; i < 16; ++i) sc[i] = 0.f;
        auto read_k = [&](int s) {
          const int p = DT == kF32 ? CPR / 2 * grp + s : 2 * s + grp;
          return *reinterpret_cast<const u32x4*>(s_k + (kg * KB + col) * DP + S::kpos(col, p) * EC);
        };
        u32x4 kf[SW < 4 ? QW : 1];
        if constexpr (SW < 4) {
#pragma unroll
          for (int s = 0; s < QW; ++s) kf[s] = read_k(s);
        }
        // With registers to spare V's operands are read before the scores are worked on.
        const int t16 = lane & 15;
        auto read_v = [&](int s, int d) {
          const int rr = 4 * grp + (t16 >> 2);
          const int p = 4 * d + ((lane >> 4) & 1) * 2 + ((t16 & 3) >> 1);
          const T* at = s_v + (kg * KB + 16 * s + rr) * DP + S::vpos(rr, p) * 8 + (t16 & 1) * 4;
          const uint2 x = read_transposed(at);
          const uint2 y = read_transposed(at + 8 * DP);
          return u32x4{x.x, x.y, y.x, y.y};
        };
        u32x4 vf[KB / 16][DT32];
        if constexpr (DT != kF32 && SW < 4) {
#pragma unroll
          for (int s = 0; s < KB / 16; ++s)
#pragma unroll
            for (int d = 0; d < DT32; ++d) vf[s][d] = read_v(s, d);
          __builtin_amdgcn_sched_barrier(0);
        }
        if constexpr (DT == kF32) {
          // four short chains of sums instead of one of DP / 2
          floatx16 part[3];
#pragma unroll
          for (int j = 0; j < 3; ++j)
#pragma unroll
            for (int i = 0; i < 16; ++i) part[j][i] = 0.f;
#pragma unroll
          for (int s = 0; s < QW; ++s)
#pragma unroll
            for (int j = 0; j < 4; ++j) {
              floatx16& c = j == 0 ? sc : part[j - 1];
              c = __builtin_amdgcn_mfma_f32_32x32x2f32(__uint_as_float(kf[s][j]), __uint_as_float(qv[s][j]), c, 0, 0, 0);
            }
#pragma unroll
          for (int i = 0; i < 16; ++i) sc[i] = (sc[i] + part[0][i]) + (part[1][i] + part[2][i]);
        } else {
#pragma unroll
          for (int s = 0; s < QW; ++s) sc = mfma32<DT>(SW < 4 ? kf[s] : read_k(s), qv[s], sc);
        }
        // Causal / length mask, only for blocks that reach past the wave's
        // first query or past the item's keys (a wave-uniform test).
        if (base + KB - 1 > offset + q0 || base + KB > w1) {
          const int last = min(qpos, w1 - 1) - base - 4 * grp;
#pragma unroll
          for (int i = 0; i < 16; ++i)
            if (8 * (i >> 2) + (i & 3) > last) sc[i] = -INFINITY;
        }
        // Block max of the raw scores (qscale > 0 commutes with the max; NaN
        // scores are dropped by fmaxf), shared by the two lanes of a query.
        float bmax = sc[0];
#pragma unroll
        for (int i = 1; i < 16; ++i) bmax = fmaxf(bmax, sc[i]);
        bmax = max_halves(bmax) * a.qscale;
        if (__any(bmax > m + kRescale)) {  // also a query's first keys, m = -inf
          const float mn = fmaxf(m, bmax);
          const float alpha = (m == -INFINITY) ? 0.f : fast_exp2(m - mn);
          l *= alpha;
#pragma unroll
          for (int d = 0; d < DT32; ++d)
#pragma unroll
            for (int i = 0; i < 16; ++i) o[d][i] *= alpha;
          m = mn;
        }
        const float mref = (m == -INFINITY) ? 0.f : m - kShift;  // masked scores give exp2(-inf) = 0
#pragma unroll
        for (int i = 0; i < 16; ++i) sc[i] = fast_exp2(fmaf(sc[i], a.qscale, -mref));
        float psum[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) psum[i] = sc[i] + sc[i + 8];
#pragma unroll
        for (int w = 4; w > 0; w /= 2)
#pragma unroll
          for (int i = 0; i < w; ++i) psum[i] += psum[i + w];
        l += psum[0];  // this lane's keys; the lanes of a query are added at the end

        if constexpr (DT == kF32) {
          // The block's sums start at zero, in short chains that are added in
          // pairs and then to the running ones: a chain rounds at every key.
          // All 32 keys in one chain, 4 x 333 tokens of head dim 64 end 1.38e-7
          // from 64 bits (2-norm, relative), where query_kernel's short chains
          // end 1.25e-7; four chains end 1.25e-7 as well, for 2 % of the time
          // (13 % at head dim 128, one wave per SIMD).
          constexpr int STEP = 16 / S::kSums;
#pragma unroll
          for (int d = 0; d < DT32; ++d) {
            floatx16 sum;
#pragma unroll
            for (int h = 0; h < 16; h += STEP) {
              floatx16 ob[4];
#pragma unroll
              for (int j = 0; j < 4; ++j)
#pragma unroll
                for (int i = 0; i < 16; ++i) ob[j][i] = 0.f;
#pragma unroll
              for (int i = h; i < h + STEP; ++i) {
                const int rr = 8 * (i >> 2) + 4 * grp + (i & 3), dd = 32 * d + col;
                const float vv = s_v[(kg * KB + rr) * DP + S::vpos(rr, dd >> 2) * 4 + (dd & 3)];
                ob[i & 3] = __builtin_amdgcn_mfma_f32_32x32x2f32(vv, sc[i], ob[i & 3], 0, 0, 0);
              }
#pragma unroll
              for (int i = 0; i < 16; ++i) {
                const float x = (ob[0][i] + ob[1][i]) + (ob[2][i] + ob[3][i]);
                sum[i] = h ? sum[i] + x : x;
              }
            }
#pragma unroll
            for (int i = 0; i < 16; ++i) o[d][i] += sum[i];
          }
        } else {
          // 16 keys a step: slot j < 4 of a lane holds key 16 s + 4 grp + j,
          // slot j >= 4 key 16 s + 8 + 4 grp + j - 4, in P as in V^T.
#pragma unroll
          for (int s = 0; s < KB / 16; ++s) {
            u32x4 hi, lo;
#pragma unroll
            for (int w = 0; w < 4; ++w) {
              uint32_t h2, l2;
              SplitP<DT>::split(sc[8 * s + 2 * w], sc[8 * s + 2 * w + 1], h2, l2);
              hi[w] = h2;
              lo[w] = l2;
            }
#pragma unroll
            for (int d = 0; d < DT32; ++d) {
              const u32x4 vv = SW < 4 ? vf[s][d] : read_v(s, d);
              o[d] = mfma32<DT>(vv, hi, o[d]);
              o[d] = mfma32<DT>(vv, lo, o[d]);
            }
          }
        }
      }
    }

    // O^T lane layout: dims 32 d + 8 (i / 4) + 4 grp + i % 4 of query qi. A
    // piece of the tile's keys leaves (accumulators, max, denominator) in
    // base-2 units for the merge kernels, a whole tile the output rows.
    l = add_halves(l);
    m -= kShift;  // what the sums are relative to
    float* const part = it.slot >= 0 ? a.partials + (int64_t(it.slot) * g.heads + head) * TQ * pf_part_row<DP>() : nullptr;
    if constexpr (KG == 1) {
      // Queries left non-finite (and not by a missing page, whose NaN is the
      // denominator's too) are attended once more, alone.
      float zero[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int d = 0; d < DT32; ++d)
#pragma unroll
        for (int i = 0; i < 16; ++i) zero[i & 3] = fmaf(o[d][i], 0.f, zero[i & 3]);
      const uint64_t lanes = __ballot(q_ok && isnan((zero[0] + zero[1]) + (zero[2] + zero[3])) && !isnan(l));
      const uint32_t redo = uint32_t(lanes) | uint32_t(lanes >> 32);
      const float inv = inverse(l);
#pragma unroll
      for (int d = 0; d < DT32; ++d)
#pragma unroll
        for (int i = 0; i < 16; i += 4) {
          const int dd = 32 * d + 2 * i + 4 * grp;
          if (!q_ok) continue;
          if (part)
            *reinterpret_cast<float4*>(part + (qt * 32 + col) * pf_part_row<DP>() + dd) =
                float4{o[d][i], o[d][i + 1], o[d][i + 2], o[d][i + 3]};
          else if (dd < dim)
            store4<DT>(out + it.o0 + qi * a.o_r + dd, divided<DT>(o[d][i], l, inv), divided<DT>(o[d][i + 1], l, inv),
                       divided<DT>(o[d][i + 2], l, inv), divided<DT>(o[d][i + 3], l, inv));
        }
      if (part && q_ok && grp == 0)
        *reinterpret_cast<float2*>(part + (qt * 32 + col) * pf_part_row<DP>() + DP) = float2{m, l};
      if (__builtin_expect(redo != 0, 0)) {
        __threadfence_block();  // after the stores above, which it repeats
        attend_again<DT, DP, TQ, 1, Items, FUSED>(item, qt, 0, redo);
      }
    } else {
      // The groups' states meet in LDS, then every thread merges four dims of
      // a query over the groups. A group none of whose keys a query attends
      // holds l = 0; a NaN denominator (missing page) poisons the sum.
      float* const s_o = reinterpret_cast<float*>(s_raw);
      float2* const s_ml = reinterpret_cast<float2*>(s_o + KG * TQ * S::OS);
      __syncthreads();
      {
        float* row = s_o + ((kg * TQ) + qt * 32 + col) * S::OS + 4 * grp;
#pragma unroll
        for (int d = 0; d < DT32; ++d)
#pragma unroll
          for (int i = 0; i < 16; i += 4)
            *reinterpret_cast<float4*>(row + 32 * d + 2 * i) = float4{o[d][i], o[d][i + 1], o[d][i + 2], o[d][i + 3]};
        if (grp == 0) s_ml[kg * TQ + qt * 32 + col] = float2{m, l};
      }
      __syncthreads();
      int first = tid;
      asm volatile("" : "+v"(first));  // keeps the addresses below out of the registers of the loop
      for (int u = first; u < TQ * DP / 4; u += NT) {
        const int q = u / (DP / 4), dd = 4 * (u - q * (DP / 4));
        const int row = it.tile * TQ + q;
        if (row >= nq) break;
        float2 ml[KG];
        float M = -INFINITY, L = 0.f;
#pragma unroll
        for (int k = 0; k < KG; ++k) { ml[k] = s_ml[k * TQ + q]; M = fmaxf(M, ml[k].x); }
        float4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int k = 0; k < KG; ++k) {
          const float w = ml[k].x == -INFINITY ? 0.f : fast_exp2(ml[k].x - M);
          const float4 x = *reinterpret_cast<const float4*>(s_o + (k * TQ + q) * S::OS + dd);
          L = fmaf(ml[k].y, w, L);
          acc.x = fmaf(x.x, w, acc.x); acc.y = fmaf(x.y, w, acc.y);
          acc.z = fmaf(x.z, w, acc.z); acc.w = fmaf(x.w, w, acc.w);
        }
        // left non-finite, and not by a missing page: attended once more, alone
        if (__builtin_expect(isnan(0.f * acc.x + 0.f * acc.y + 0.f * acc.z + 0.f * acc.w) && !isnan(L), 0))
          atomicOr(&s_redo[q >> 5], 1u << (q & 31));
        if (part) {
          float* dst = part + q * pf_part_row<DP>();
          *reinterpret_cast<float4*>(dst + dd) = acc;
          if (dd == 0) *reinterpret_cast<float2*>(dst + DP) = float2{M, L};
        } else if (dd < dim) {
          const float inv = inverse(L);
          store4<DT>(out + it.o0 + row * a.o_r + dd, divided<DT>(acc.x, L, inv), divided<DT>(acc.y, L, inv),
                     divided<DT>(acc.z, L, inv), divided<DT>(acc.w, L, inv));
        }
      }
      // (a workgroup's stores to a row are in the order of its barriers)
      __syncthreads();
      uint32_t any = 0;
#pragma unroll
      for (int t = 0; t < QT; ++t) any |= s_redo[t];
      if (__builtin_expect(__builtin_amdgcn_readfirstlane(any) != 0, 0))
#pragma unroll 1
        for (int t = 0; t < QT; ++t)
          attend_again<DT, DP, TQ, S::W, Items, FUSED>(item, t, wave, __builtin_amdgcn_readfirstlane(s_redo[t]));
    }
  }
}

// Merge of tiles whose keys were split over workgroups: every query's output
// from its pieces' (accumulators, max, denominator) by the log-sum-exp rule,
// with the finalize rule of the unsplit kernel (a NaN denominator stays NaN, a
// zero one gives 0). One workgroup per (tile, head), four threads per query,
// each taking every fourth 16-byte chunk of the row; one online pass over the
// pieces, unrolled so that several pieces' loads are in flight.
template <int DT, int D>
__device__ __forceinline__ void merge_query(const QueryArgs& a, int head, int q, int sub, int tq, int first_slot,
                                            int n, typename Elem<DT>::T* orow) {
  constexpr int R = pf_part_row<D>(), C = D / 16;
  const float* base = a.partials + ((int64_t(first_slot) * a.g.heads + head) * tq + q) * R;
  const int64_t step = int64_t(a.g.heads) * tq * R;
  float M = -INFINITY, L = 0.f;
  float4 acc[C];
#pragma unroll
  for (int c = 0; c < C; ++c) acc[c] = float4{0.f, 0.f, 0.f, 0.f};
#pragma unroll 4
  for (int s = 0; s < n; ++s) {
    const float* p = base + s * step;
    const float2 ml = *reinterpret_cast<const float2*>(p + D);
    float4 x[C];
#pragma unroll
    for (int c = 0; c < C; ++c) x[c] = *reinterpret_cast<const float4*>(p + 4 * (sub + 4 * c));
    const float Mn = fmaxf(M, ml.x);
    const float wo = M == -INFINITY ? 0.f : fast_exp2(M - Mn);
    const float wn = ml.x == -INFINITY ? 0.f : fast_exp2(ml.x - Mn);
    L = fmaf(L, wo, ml.y * wn);  // a NaN denominator (missing page) poisons the sum
#pragma unroll
    for (int c = 0; c < C; ++c) {
      acc[c].x = fmaf(acc[c].x, wo, x[c].x * wn);
      acc[c].y = fmaf(acc[c].y, wo, x[c].y * wn);
      acc[c].z = fmaf(acc[c].z, wo, x[c].z * wn);
      acc[c].w = fmaf(acc[c].w, wo, x[c].w * wn);
    }
    M = Mn;
  }
#pragma unroll
  for (int c = 0; c < C; ++c) {
    const int dd = 4 * (sub + 4 * c);
    if (dd < a.g.dim)
      store4<DT>(orow + dd, finalize(acc[c].x, L), finalize(acc[c].y, L), finalize(acc[c].z, L),
                 finalize(acc[c].w, L));
  }
}

// Tiles of a uniform batch: one workgroup per (tile, request, head).
template <int DT, int D>
__global__ __launch_bounds__(256) void uniform_merge_kernel(QueryArgs a, UniformItems u, int tq) {
  using T = typename Elem<DT>::T;
  const unsigned bh_count = unsigned(a.batch) * unsigned(a.g.heads);
  const int tile = int(blockIdx.x / bh_count);
  const int bh = int(blockIdx.x - unsigned(tile) * bh_count);
  const int b = bh / a.g.heads, head = bh - b * a.g.heads;
  const int nb = key_blocks(tile, tq, a.nq, a.offset);
  if (nb <= u.share) return;  // one piece: its workgroup wrote the output
  for (int q = threadIdx.x >> 2; q < tq; q += 64) {
    const int qi = tile * tq + q;
    if (qi >= a.nq) return;
    T* orow = static_cast<T*>(a.out) + b * a.o_b + head * a.o_h + int64_t(qi) * a.o_r;
    merge_query<DT, D>(a, head, q, threadIdx.x & 3, tq, (b * u.tiles + tile) * u.pieces, (nb + u.share - 1) / u.share,
                       orow);
  }
}

// Key splits of ragged prompts: per split tile, its first output row (in the
// launch's rows), its valid queries, first partials slot and piece count.
struct RaggedMerge {
  int tiles;
  int row0[kRaggedTiles];
  unsigned short nq[kRaggedTiles], first_slot[kRaggedTiles];
  unsigned char splits[kRaggedTiles];
};

// Kernel arguments stay within the 4 KiB kernarg limit.
static_assert(sizeof(QueryArgs) + sizeof(RaggedItems) <= 4096, "ragged prefill arguments");
static_assert(sizeof(QueryArgs) + sizeof(RaggedMerge) <= 4096, "ragged merge arguments");

template <int DT, int D>
__global__ __launch_bounds__(256) void ragged_merge_kernel(QueryArgs a, RaggedMerge mg, int tq) {
  using T = typename Elem<DT>::T;
  const int t = int(blockIdx.x / unsigned(a.g.heads));
  const int head = int(blockIdx.x - unsigned(t) * a.g.heads);
  if (t >= mg.tiles) return;
  for (int q = threadIdx.x >> 2; q < mg.nq[t]; q += 64) {
    T* orow = static_cast<T*>(a.out) + head * a.o_h + (int64_t(mg.row0[t]) + q) * a.o_r;
    merge_query<DT, D>(a, head, q, threadIdx.x & 3, tq, mg.first_slot[t], mg.splits[t], orow);
  }
}

// Multi-token append at a common offset (reference paged_append with
// offsets == nullptr, src/paged_attention_kernel.cu:23-33): K/V[b,h,pos,:]
// goes to token offset + pos of request b; rows whose page is missing are
// skipped. VEC moves 16 bytes per thread.
template <int DT, bool VEC>
__global__ __launch_bounds__(256) void append_kernel(AppendArgs a) {
  using T = typename Elem<DT>::T;
  constexpr int E = VEC ? per16<DT>() : 1;
  const Geometry& g = a.g;
  const int dim = g.dim;
  const int per_row = dim / E;
  for (int64_t i = blockIdx.x * int64_t(blockDim.x) + threadIdx.x; i < a.vectors;
       i += int64_t(gridDim.x) * blockDim.x) {
    const int64_t row = i / per_row;  // (b*h + head)*n + pos
    const int col = int(i - row * per_row) * E;
    const int64_t bhh = row / a.n;
    const int pos_in = int(row - bhh * a.n);
    const int b = int(bhh / g.heads), head = int(bhh - int64_t(b) * g.heads);
    const int64_t pos = int64_t(a.offset) + pos_in;
    const T* base = page_base<T>(a.slabs, a.table + int64_t(b) * g.columns, pos >> g.log2_page, g, head);
    if (!base) continue;
    T* kp = const_cast<T*>(base) + (pos & (g.page_size - 1)) * dim + col;
    T* vp = kp + g.kind_stride;
    const int64_t src = b * a.src_b + head * a.src_h + pos_in * a.src_r + col;
    if constexpr (VEC) {
      *global_view(reinterpret_cast<u32x4*>(kp)) = *global_view(reinterpret_cast<const u32x4*>(static_cast<const T*>(a.k) + src));
      *global_view(reinterpret_cast<u32x4*>(vp)) = *global_view(reinterpret_cast<const u32x4*>(static_cast<const T*>(a.v) + src));
    } else {
      *kp = static_cast<const T*>(a.k)[src];
      *vp = static_cast<const T*>(a.v)[src];
    }
  }
}

// Shape guard of the reference (src/paged_attention_kernel.cu:87-94 and
// src/includes/flash_common.cuh:17-20): the same inputs are rejected.
bool paged_shape(int b, int h, int nq, int nk, int d, int page_size, int pps, int num_slabs,
                 int columns, int layer, int layers, int offset) {
  return b > 0 && h > 0 && nq > 0 && nk > 0 && d > 0 && d <= 128 &&
         int64_t(b) * h * nq * d <= INT32_MAX && int64_t(b) * h * nk * d <= INT32_MAX &&
         int64_t(b) * h <= 65535 && (page_size == 8 || page_size == 16 || page_size == 32) &&
         pps > 0 && num_slabs > 0 && int64_t(pps) * num_slabs <= INT32_MAX && columns > 0 &&
         int64_t(b) * columns <= INT32_MAX && nk <= int64_t(columns) * page_size && layers > 0 &&
         layer >= 0 && layer < layers && offset >= 0 && int64_t(offset) + nq == nk;
}

Geometry make_geometry(int h, int d, int page_size, int pps, int num_slabs, int columns, int layer) {
  Geometry g{};
  g.heads = h; g.dim = d; g.page_size = page_size;
  g.log2_page = page_size == 8 ? 3 : page_size == 16 ? 4 : 5;
  g.pps = pps; g.num_slabs = num_slabs; g.columns = columns; g.layer = layer;
  int sh = 0;
  while ((int64_t(1) << sh) < pps) ++sh;
  g.pps_shift = 31 + sh;
  g.pps_magic = ((uint64_t(1) << (31 + sh)) + uint64_t(pps) - 1) / uint64_t(pps);
  g.kind_stride = int64_t(pps) * h * page_size * d;
  return g;
}

bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

constexpr int64_t kMaxGrid = int64_t(1) << 30;

int grid_for(int64_t items) { return int(items < kMaxGrid ? items : kMaxGrid); }

// Split length for a decode launch: kDefaultSplitTokens unless the longest
// possible context (columns * page_size) would need more than
// kMaxSplitsPerRow splits, then longer splits (multiple of 64, at most 2048).
int choose_split(int64_t cap, int requested) {
  if (requested > 0) return requested;
  int64_t s = kDefaultSplitTokens;
  if ((cap + s - 1) / s > kMaxSplitsPerRow) {
    s = (cap + kMaxSplitsPerRow - 1) / kMaxSplitsPerRow;
    s = (s + 63) / 64 * 64;
    if (s > kMaxSplitTokens) s = kMaxSplitTokens;
  }
  return int(s);
}

size_t workspace_bytes_for(int64_t bh, int nsplit_max) {
  // (max, denominator, accumulator[128]) per (row, head, split)
  return size_t(bh) * nsplit_max * (128 + 2) * sizeof(float);
}

// How the decode reads the rows of these operands.
Rows decode_rows(int d, int dtype, const void* out, const void* q, const void* k, const void* v,
                 int64_t qkv_stride) {
  const int esize = dtype == kF32 ? 4 : 2;
  if ((d * esize) % 16 || !aligned16(out) || !aligned16(q) || !aligned16(k) || !aligned16(v) ||
      (qkv_stride * esize) % 16)
    return kRowsElements;
  return d == 64 || d == 128 ? kRowsFull : kRowsPadded;
}

// Bytes of split partials a decode launch writes: (max, denominator,
// accumulator[D]) per (row, head, split), D being the kernel's head-dim
// template (64 for the 16-byte kernel at d = 64, else 128).
size_t partial_bytes(int64_t bh, int64_t nsplit_max, bool vec, int d) {
  const int dt = (vec && d == 64) ? 64 : 128;
  return size_t(bh) * size_t(nsplit_max) * size_t(dt + 2) * sizeof(float);
}

// Compute units of the current device (cached per device).
int device_compute_units() {
  static int cached[64] = {};
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 0;
  if (!cached[dev]) {
    int n = 0;
    if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess) return 0;
    cached[dev] = n;
  }
  return cached[dev];
}

// A wave resolves the page of each of its steps into one lane, so a split
// may give a wave at most 64 steps (32 when a step spans two pages): 2-wave
// workgroups take splits of at most 1024 tokens (512 for pages below 8).
bool two_wave_split_ok(const DecodeArgs& a) {
  constexpr int RB = kWave / kDecodeGroup;  // tokens per wave step
  const int steps = a.split_tokens / RB / 2;
  return a.split_tokens % (2 * RB) == 0 && steps * (a.g.page_size < RB ? 2 : 1) <= kWave;
}

// Workgroups of decode_kernel<DT, D, VEC, U, kStages, WAVES, G> resident per
// compute unit (0 if the query fails), looked up once per instantiation.
template <int DT, int D, int VEC, int U, int WAVES, int G>
int decode_occupancy() {
  static const int per_cu = [] {
    int n = 0;
    return hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, decode_kernel<DT, D, VEC, U, kStages, WAVES, G, kVisitList>,
                                                        WAVES * kWave, 0) == hipSuccess ? n : 0;
  }();
  return per_cu;
}

// The instantiation of the launch's visiting mode.
template <int DT, int D, int VEC, int U, int WAVES, int G>
void launch_decode_mode(const DecodeArgs& a, int64_t blocks, size_t lds) {
  constexpr int NT = WAVES * kWave;
  if (a.work) decode_kernel<DT, D, VEC, U, kStages, WAVES, G, kVisitList><<<grid_for(blocks), NT, lds>>>(a);
  else if (a.uniform_len) decode_kernel<DT, D, VEC, U, kStages, WAVES, G, kVisitUniform><<<grid_for(blocks), NT, lds>>>(a);
  else if (a.rank_rows) decode_kernel<DT, D, VEC, U, kStages, WAVES, G, kVisitRank><<<grid_for(blocks), NT, lds>>>(a);
  else decode_kernel<DT, D, VEC, U, kStages, WAVES, G, kVisitGrid><<<grid_for(blocks), NT, lds>>>(a);
}

template <int DT, int D, int VEC, int WAVES, int G>
hipError_t launch_decode_w(const DecodeArgs& a, int64_t blocks, int unroll) {
  // Row bytes per lane bound the useful unroll: register stages beyond it spill.
  constexpr int kMaxUnroll = !VEC ? 1 : (VEC == kRowsPadded || D * elem_bytes<DT>() >= 256 ? 2 : 4);
  constexpr int NT = WAVES * kWave;
  if (unroll == 0) {
    if constexpr (G == 8) {
      // Two row-blocks per register stage: measured best or within 1 % of
      // the best at every decode shape of configs 2, 4 and 5. A grid of at
      // most one 8-wave workgroup per compute unit has registers for four,
      // which keep twice the bytes in flight: one row of 1000 tokens x 16
      // heads bf16 8.8 against 9.5 us, 4 rows to 500 x 25 heads 7.5 against 8.0.
      unroll = WAVES == 8 && kMaxUnroll >= 4 && blocks <= device_compute_units() ? 4 : 2;
    } else if constexpr (kMaxUnroll >= 4) {
      // The deepest unroll when the whole grid is resident at its
      // occupancy (more loads in flight per wave), else unroll 1, whose
      // lower register count keeps the most workgroups per compute unit.
      unroll = blocks <= int64_t(decode_occupancy<DT, D, VEC, 4, WAVES, G>()) * device_compute_units() ? 4 : 1;
    } else {
      unroll = 1;
    }
  }
  // Requests between the supported values round down (3 -> 2, 5+ -> 4).
  unroll = unroll >= 4 ? 4 : unroll >= 2 ? 2 : 1;
  const size_t rank_lds = a.rank_rows ? size_t(2) * ((a.batch + 3) & ~3) * sizeof(int) : 0;
  if (unroll > kMaxUnroll) unroll = kMaxUnroll;
  if (a.work_count) {
    // A device-built list of unknown length: one residency round of
    // workgroups strides over it.
    int occ = 0;
    if (unroll == 4) occ = decode_occupancy<DT, D, VEC, (kMaxUnroll >= 4 ? 4 : 1), WAVES, G>();
    else if (unroll == 2) occ = decode_occupancy<DT, D, VEC, (kMaxUnroll >= 2 ? 2 : 1), WAVES, G>();
    else occ = decode_occupancy<DT, D, VEC, 1, WAVES, G>();
    const int64_t resident = int64_t(occ > 0 ? occ : 1) * std::max(1, device_compute_units());
    blocks = std::min(blocks, resident);
  }
  if constexpr (kMaxUnroll >= 4) {
    if (unroll == 4) launch_decode_mode<DT, D, VEC, 4, WAVES, G>(a, blocks, rank_lds);
  }
  if constexpr (kMaxUnroll >= 2) {
    if (unroll == 2) launch_decode_mode<DT, D, VEC, 2, WAVES, G>(a, blocks, rank_lds);
  }
  if (unroll == 1) launch_decode_mode<DT, D, VEC, 1, WAVES, G>(a, blocks, rank_lds);
  hipError_t e = hipGetLastError();
  const int64_t merge_rows = a.work && !a.work_count ? a.merge_rows : a.batch;
  if (e != hipSuccess || a.nsplit_max == 1 || merge_rows == 0) return e;
  int64_t merge_blocks = merge_rows * a.g.heads;
  // Device-built list: the merge rows' count is on the device; a grid of
  // four workgroups per compute unit strides over them.
  if (a.work_count) merge_blocks = std::min(merge_blocks, 4 * int64_t(std::max(1, device_compute_units())));
  merge_kernel<DT, (D > 64 ? 128 : 64)><<<grid_for(merge_blocks), 128>>>(a);
  return hipGetLastError();
}

// waves 0 = automatic: 8-wave workgroups when the whole grid is resident at
// their occupancy (a (row, head) streamed by 8 waves finishes its longest
// rows sooner; config 2: 21.0 us vs 21.9 us with 4), else 4 (more
// workgroups per compute unit for grids of several residency rounds;
// config 5: 256 us vs 267 us with 8), and 2 when even 2-wave workgroups take
// more than two residency rounds (finer-grained hand-out of the tail; config
// 5: 261-263 us vs 267 us with 4; config 4's layer, 2048 workgroups that 2
// waves would make resident at once, took 9 % longer per step with 2).
template <int DT, int D, int VEC>
hipError_t launch_decode_t(const DecodeArgs& a, int64_t blocks, int unroll, int waves) {
  constexpr int G = kDecodeGroup;
  constexpr int U8 = VEC && G == 8 ? 2 : 1;
  if (waves == 0) {
    const int64_t cus = device_compute_units();
    waves = blocks <= int64_t(decode_occupancy<DT, D, VEC, U8, 8, G>()) * cus ? 8 : 4;
    if (waves == 4 && two_wave_split_ok(a) && blocks > 2 * int64_t(decode_occupancy<DT, D, VEC, U8, 2, G>()) * cus)
      waves = 2;
  }
  if (a.split_tokens % ((kWave / G) * waves) != 0 || (waves == 2 && !two_wave_split_ok(a))) waves = 4;
  if (waves == 8) return launch_decode_w<DT, D, VEC, 8, G>(a, blocks, unroll);
  if (waves == 2) return launch_decode_w<DT, D, VEC, 2, G>(a, blocks, unroll);
  return launch_decode_w<DT, D, VEC, 4, G>(a, blocks, unroll);
}

template <int DT>
hipError_t launch_decode_dt(const DecodeArgs& a, int64_t blocks, Rows rows, int d, int unroll, int waves) {
  if (rows == kRowsFull && d == 64) return launch_decode_t<DT, 64, kRowsFull>(a, blocks, unroll, waves);
  if (rows == kRowsFull) return launch_decode_t<DT, 128, kRowsFull>(a, blocks, unroll, waves);
  if (rows == kRowsPadded && d < 64) return launch_decode_t<DT, 64, kRowsPadded>(a, blocks, unroll, waves);
  if (rows == kRowsPadded) return launch_decode_t<DT, 128, kRowsPadded>(a, blocks, unroll, waves);
  return launch_decode_t<DT, 128, kRowsElements>(a, blocks, 1, waves);
}

// Split length of a decode of bh (row, head) pairs whose longest context is
// `longest` tokens, where the library chooses: choose_split's, unless that
// leaves compute units idle. Then enough splits for two workgroups per
// compute unit, but no split below kSplitBytes of K and V (a split's own
// prologue and its share of the merge take about 5 us, in which a workgroup
// streams that much). One row of 8000 tokens x 12 heads fp16: 12.0 us at 512
// tokens a split, 13.4 at 1024, 15.2 at 128; 8 rows to 1500: 12.6 against 13.4.
constexpr int64_t kSplitBytes = 128 * 1024;
int idle_split(int64_t bh, int64_t longest, int d, int dtype) {
  const int S = choose_split(longest, 0);
  const int64_t row_bytes = int64_t(2) * d * (dtype == kF32 ? 4 : 2);
  const int64_t least = (kSplitBytes / row_bytes + 63) / 64 * 64;
  const int64_t want = (longest * bh / (2 * std::max(1, device_compute_units())) + 63) / 64 * 64;
  return int(std::min<int64_t>(S, std::max(least, want)));
}

int decode_common(void* out, const void* q, const void* k, const void* v, const uint64_t* slabs,
                  const int* table, const int* offsets, int b, int h, int d, int page_size,
                  int pps, int num_slabs, int columns, int layer, int layers, int dtype,
                  int split_tokens, int unroll, int waves, int qkv_stride, const int* work,
                  int work_items, int merge_rows, void* workspace, size_t workspace_bytes,
                  bool rank_order = false, int* order = nullptr) {
  const int64_t cap = int64_t(columns) * page_size;
  // A work list is built for one split length, so it must be given.
  if (work && split_tokens <= 0) return hipErrorInvalidValue;
  const int S = choose_split(cap, split_tokens);
  if (S < 64 || S % 64 != 0 || S > kMaxSplitTokens) return hipErrorInvalidValue;
  if (waves != 0 && waves != 2 && waves != 4 && waves != 8) return hipErrorInvalidValue;
  const int64_t nsplit_max = (cap + S - 1) / S;
  const int64_t bh = int64_t(b) * h;
  if (nsplit_max > INT_MAX) return hipErrorInvalidValue;
  if (work && (work_items < 0 || merge_rows < 0 || merge_rows > b ||
               work_items > int64_t(b) * nsplit_max || (reinterpret_cast<uintptr_t>(work) & 7u)))
    return hipErrorInvalidValue;
  if (work && work_items == 0) return hipSuccess;
  const int64_t stride = qkv_stride ? qkv_stride : int64_t(h) * d;
  const Rows rows = decode_rows(d, dtype, out, q, k, v, stride);
  if (nsplit_max > 1 && (!workspace || workspace_bytes < partial_bytes(bh, nsplit_max, rows == kRowsFull, d)))
    return hipErrorInvalidValue;
  DecodeArgs a{};
  a.out = out; a.q = q; a.k = k; a.v = v; a.slabs = slabs; a.table = table; a.offsets = offsets;
  a.batch = b; a.split_tokens = S; a.nsplit_max = int(nsplit_max);
  a.qscale = (1.0f / std::sqrt(float(d))) * kLog2e;
  a.items = work ? int64_t(work_items) * h : bh * nsplit_max;
  // The kernels index items with 32-bit arithmetic.
  if (a.items > INT32_MAX) return hipErrorInvalidValue;
  a.g = make_geometry(h, d, page_size, pps, num_slabs, columns, layer);
  a.partials = static_cast<float*>(workspace);
  a.qkv_stride = stride;
  a.work = work;
  a.work_items = work ? work_items : 0;
  a.merge_rows = work ? merge_rows : 0;
  // Entries without a work list visit rows longest first when every row has
  // one split and the batch is small enough to rank in each workgroup.
  // Where every workgroup has a compute unit to itself the order does not
  // matter, and the ranking only lengthens the prologue.
  if (rank_order && !work && nsplit_max == 1 && b <= kRankRows && bh > device_compute_units()) {
    a.rank_rows = 1;
    a.rank_per = std::max(1, device_compute_units() / h);
  } else if (rank_order && !work && order) {
    // Larger batches, and rows that may split: order_kernel writes the work
    // list a host caller would build (count, then the list) into `order`.
    OrderArgs oa{};
    oa.offsets = offsets; oa.count = order; oa.list = order + 2;
    oa.batch = b; oa.split_tokens = S; oa.cap = cap; oa.capacity = int(int64_t(b) * nsplit_max);
    oa.per = std::max(1, device_compute_units() / h);
    order_kernel<<<1, kOrderThreads>>>(oa);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    a.work = order + 2;
    if (nsplit_max > 1) {
      a.work_count = order;  // a.items stays the capacity, bh * nsplit_max
    } else {
      a.work_items = b;      // one entry per row
      a.items = bh;
    }
  }
  if (dtype == kF32) return launch_decode_dt<kF32>(a, a.items, rows, d, unroll, waves);
  if (dtype == kF16) return launch_decode_dt<kF16>(a, a.items, rows, d, unroll, waves);
  if (dtype == kBF16) return launch_decode_dt<kBF16>(a, a.items, rows, d, unroll, waves);
  return hipErrorInvalidValue;
}

// Whether the reference entries have order_kernel build their visiting
// order (batches past the in-workgroup ranking, or rows that may split, up to
// kOrderRows rows), and the bytes it writes: the count pair, the (row, split)
// list and the merge rows.
// Not for grids of few rounds of the compute units: the launch (8 us) costs
// more than the order saves (40 rows to 3000 tokens x 25 heads fp16, 3000
// workgroups: 71.4 us in batch order, 77.2 with it; 512 rows to 8192 x 25
// heads, 102,400: 334 against 270).
constexpr int kOrderBlocksPerUnit = 16;
bool device_order(int b, int h, int64_t nsplit_max) {
  return b <= kOrderRows && (nsplit_max > 1 || b > kRankRows) && int64_t(b) * nsplit_max <= INT32_MAX / 2 &&
         int64_t(b) * h * nsplit_max > int64_t(kOrderBlocksPerUnit) * device_compute_units();
}
size_t order_bytes(int b, int64_t nsplit_max) {
  return size_t(2 + 2 * int64_t(b) * nsplit_max + b) * sizeof(int);
}
size_t align256(size_t n) { return (n + 255) & ~size_t(255); }

// Library-owned split workspace of the reference entry points, which have no
// workspace argument (mt_paged_decode_batch for tables longer than one split,
// the key-split prefill of mt_paged_attention / mt_paged_prefill). One buffer
// per (host thread, device): every launch of these libraries goes to the
// calling thread's default stream (they are built with per-thread default
// streams), so a buffer private to the thread is private to the stream its
// kernels run on, and calls from several host threads never share one. It
// grows stream-ordered on that stream: hipMallocAsync for the larger buffer
// and hipFreeAsync for the old one, which is released only after the work
// queued before it, so growing neither synchronizes the device nor blocks the
// host. A buffer whose address a captured graph holds is not released while
// its thread lives, nor is one that a capture outgrows, where a release would be
// a node of the graph; the buffer that takes its place is at least twice as
// large, so that those kept add up to less than the current one. Under capture
// the larger buffer is a plain allocation: a stream-ordered one would be a node
// too, there only while the graph runs. A thread's buffers are released when it
// exits.
// Callers that cannot allocate use mt_paged_decode_split with their own
// workspace, or mt_paged_decode_batch_noalloc.
struct Workspace {
  void* ptr = nullptr;
  size_t bytes = 0;
  bool pooled = false;    // from hipMallocAsync
  bool captured = false;  // a graph holds its address
};

struct ThreadWorkspaces {
  struct PerDevice {
    Workspace current;
    std::vector<Workspace> kept;
  };
  std::vector<PerDevice> per_device;
  static void release(const Workspace& w) {
    if (w.ptr) (void)(w.pooled ? hipFreeAsync(w.ptr, hipStreamPerThread) : hipFree(w.ptr));
  }
  ~ThreadWorkspaces() {
    int current = 0;
    if (hipGetDevice(&current) != hipSuccess) return;
    for (size_t dev = 0; dev < per_device.size(); ++dev) {
      if (!per_device[dev].current.ptr || hipSetDevice(int(dev)) != hipSuccess) continue;
      release(per_device[dev].current);
      for (const Workspace& w : per_device[dev].kept) release(w);
    }
    (void)hipSetDevice(current);
  }
};
thread_local ThreadWorkspaces t_workspaces;

int library_workspace(size_t bytes, void** out) {
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return e;
  hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
  e = hipStreamIsCapturing(hipStreamPerThread, &status);
  if (e != hipSuccess) return e;
  const bool capturing = status != hipStreamCaptureStatusNone;
  auto& per_device = t_workspaces.per_device;
  if (per_device.size() <= size_t(dev)) per_device.resize(dev + 1);
  auto& ws = per_device[dev];
  if (ws.current.bytes < bytes) {
    Workspace w;
    const bool keep = ws.current.ptr && (capturing || ws.current.captured);
    w.bytes = keep ? std::max(bytes, 2 * ws.current.bytes) : bytes;
    w.pooled = !capturing;
    if (capturing) {
      hipStreamCaptureMode mode = hipStreamCaptureModeRelaxed;
      e = hipThreadExchangeStreamCaptureMode(&mode);
      if (e != hipSuccess) return e;
      e = hipMalloc(&w.ptr, w.bytes);
      (void)hipThreadExchangeStreamCaptureMode(&mode);
    } else {
      e = hipMallocAsync(&w.ptr, w.bytes, hipStreamPerThread);
    }
    if (e != hipSuccess) {
      (void)hipGetLastError();  // the caller reports the status; keep it off the next launch
      return e;
    }
    if (keep) ws.kept.push_back(ws.current);
    else if (ws.current.ptr) (void)hipFreeAsync(ws.current.ptr, hipStreamPerThread);
    ws.current = w;
  }
  ws.current.captured |= capturing;
  *out = ws.current.ptr;
  return hipSuccess;
}

// Split partials of mt_paged_decode_batch_noalloc: a fixed device array, so
// that entry point allocates nothing. Every call on a device shares that
// device's copy. The decode writes every partial of a split row before the
// merge reads it, so nothing carries over between calls and nothing needs
// clearing; calls that overlap on one device (other streams) would race.
}  // namespace

static __device__ __align__(256) float scratch[MT_PAGED_NOALLOC_SCRATCH_BYTES / sizeof(float)];

namespace {

constexpr size_t kNoAllocScratchBytes = MT_PAGED_NOALLOC_SCRATCH_BYTES;

// Device address of `scratch` on the current device, looked up once per
// device (the host-side name of the array is not a device address).
int scratch_address(void** out) {
  static std::mutex mutex;
  static std::vector<void*> addresses;
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return e;
  std::lock_guard<std::mutex> lock(mutex);
  if (addresses.size() <= size_t(dev)) addresses.resize(dev + 1, nullptr);
  if (!addresses[dev]) {
    void* p = nullptr;
    e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess) return e;
    if (!p) return hipErrorInvalidSymbol;
    addresses[dev] = p;
  }
  *out = addresses[dev];
  return hipSuccess;
}

// One query per request over `len` keys, on the decode kernel: every key from
// the pages (k null), or the last one appended from the k/v rows. out is [b,
// h * d]. hipErrorNotSupported where the rows need element loads or there is
// no room for the partials.
hipError_t decode_uniform(void* out, const void* q, const void* k, const void* v, const uint64_t* slabs,
                          const int* table, int b, int len, int64_t qkv_stride, int dtype, const Geometry& g) {
  const Rows rows = decode_rows(g.dim, dtype, out, q, k, v, qkv_stride);
  if (rows == kRowsElements) return hipErrorNotSupported;
  const int64_t bh = int64_t(b) * g.heads;
  const int row_bytes = 2 * g.dim * (dtype == kF32 ? 4 : 2);
  // Unsplit while a row is short or the rows fill the compute units: the
  // merge is a launch of its own (1000 tokens x 16 heads bf16, 256 KB a row:
  // 8.8 us unsplit, 10.1 split; 700 x 12 fp32, 358 KB: 14.7 against 10.4).
  const bool whole = len <= kMaxSplitTokens &&
                     (int64_t(len) * row_bytes <= 300 * 1024 || bh >= device_compute_units());
  DecodeArgs a{};
  const int most = whole ? len : idle_split(bh, len, g.dim, dtype);
  const int pieces = (len + most - 1) / most;  // of even length
  a.split_tokens = ((len + pieces - 1) / pieces + 63) / 64 * 64;
  a.nsplit_max = (len + a.split_tokens - 1) / a.split_tokens;
  if (a.nsplit_max > 1) {
    void* ws = nullptr;
    if (library_workspace(workspace_bytes_for(bh, a.nsplit_max), &ws) != hipSuccess) return hipErrorNotSupported;
    a.partials = static_cast<float*>(ws);
  }
  a.out = out; a.q = q; a.k = k; a.v = v; a.slabs = slabs; a.table = table;
  a.batch = b; a.uniform_len = len;
  a.qscale = (1.0f / std::sqrt(float(g.dim))) * kLog2e;
  a.items = bh * a.nsplit_max;
  if (a.items > INT32_MAX) return hipErrorNotSupported;
  a.g = g;
  a.qkv_stride = qkv_stride;
  if (dtype == kF32) return launch_decode_dt<kF32>(a, a.items, rows, g.dim, 0, 0);
  if (dtype == kF16) return launch_decode_dt<kF16>(a, a.items, rows, g.dim, 0, 0);
  return launch_decode_dt<kBF16>(a, a.items, rows, g.dim, 0, 0);
}

// Launch of the append kernel for any source strides; the 16-byte path needs
// 16-byte aligned rows.
hipError_t launch_append(AppendArgs& a, int dtype) {
  const int d = a.g.dim;
  const int esize = dtype == kF32 ? 4 : 2;
  const int E = 16 / esize;
  const bool vec = d % E == 0 && aligned16(a.k) && aligned16(a.v) &&
                   (a.src_b * esize) % 16 == 0 && (a.src_h * esize) % 16 == 0 &&
                   (a.src_r * esize) % 16 == 0;
  a.vectors = int64_t(a.batch) * a.g.heads * a.n * (vec ? d / E : d);
  const int blocks = int((a.vectors + 255) / 256 < 65536 * 16 ? (a.vectors + 255) / 256 : 65536 * 16);
#define MT_APPEND(DT)                                                        \
  if (vec) append_kernel<DT, true><<<blocks, 256>>>(a);                      \
  else append_kernel<DT, false><<<blocks, 256>>>(a);
  if (dtype == kF32) { MT_APPEND(kF32) }
  else if (dtype == kF16) { MT_APPEND(kF16) }
  else { MT_APPEND(kBF16) }
#undef MT_APPEND
  return hipGetLastError();
}

// Whether query_kernel is the faster one for rows that both take (head dims 64
// and 128, where it reads rows in full 16-byte loads). It walks the keys once
// per query, four queries of a head side by side; the causal kernel computes
// tiles of 32 queries however few there are, and fp32 products at a sixteenth
// of the 16-bit rate. us per call of attention, causal kernel and query_kernel,
// 12 heads:
// * fp32, up to four queries: one walk serves them all. 2 queries of 64 requests
//   at 500 keys 122 and 50, of one request at 60 keys 10.2 and 6.3. Past 512
//   keys only where the requests fill the compute units (head dim 128: half of
//   them, its tiles split their keys two ways only): 24 requests at 800 keys 52
//   and 30, but 16 at 1500 47 and 56; past 1024 for three (64 requests at 1500
//   keys: 147 in narrow tiles, 139 and 162 for three and four).
// * fp32, head dim 128, up to eight where the tiles come to between one and two
//   rounds of the compute units: 32 requests at 500 keys 98 and 91.
// * fp32, any number of queries while their walks take one round of the compute
//   units and are short: 64 tokens 9.9 and 6.5, 20 at 120 keys 11.4 and 9.4 (head
//   dim 128: 23 and 14; 8 at 500 keys 33 and 26). A walk of 16 keys a step ends
//   later from 256 keys on (384 at head dim 128, 512 for twelve queries).
// * fp16 and bf16, head dim 64, up to three queries (four to 512 keys) of
//   requests for more than two rounds: 2 of 64 requests at 500 keys 26 and 20,
//   of 32 requests 14 and 18. Head dim 128: between one and two rounds to 320
//   keys, 2 of 32 requests at 200 keys 20 and 15.
bool query_kernel_faster(const QueryArgs& a, int dtype) {
  const int d = a.g.dim;
  if (d != 64 && d != 128) return false;
  const bool wide = d == 128;
  const int64_t cus = std::max(1, device_compute_units());
  const int64_t bh = int64_t(a.batch) * a.g.heads;
  const int64_t tiles = bh * ((a.nq + 31) / 32), groups = bh * ((a.nq + kWaves - 1) / kWaves);
  const int keys = a.nk;
  const bool second_round = tiles > cus && tiles <= 2 * cus;
  if (dtype != kF32) {
    if (wide) return a.nq <= 3 && second_round && keys > 128 && keys <= 320;
    return (a.nq <= 3 || (a.nq == 4 && keys <= 512)) && tiles > 2 * cus && keys > 128;
  }
  if (a.nq <= 4 && keys > 32) {
    if (keys <= 512) return true;
    if (wide ? 2 * tiles > cus : tiles > cus && (a.nq <= 3 || keys <= 1024)) return true;
  }
  if (wide && a.nq <= 8 && second_round && keys > 64) return true;
  if (keys <= 64) return groups <= (wide ? cus : 2 * cus);
  return groups <= cus && keys <= (wide ? (a.nq <= 12 ? 512 : 384) : 256);
}

// Whether launch_query runs the matrix-core causal kernel: rows of whole
// 16-byte chunks (head dims 8, 16, .. 128 in fp16/bf16, 4, 8, .. in fp32) at
// 16-byte aligned addresses and at least kPfMinQueries queries, where
// query_kernel is not the faster one.
bool causal_kernel_takes(const QueryArgs& a, int dtype) {
  const int d = a.g.dim;
  const int esize = dtype == kF32 ? 4 : 2;
  auto rows16 = [&](int64_t x) { return (x * esize) % 16 == 0; };
  return rows16(d) && a.nq >= kPfMinQueries && aligned16(a.out) && aligned16(a.q) && rows16(a.q_b) &&
         rows16(a.q_h) && rows16(a.q_r) && rows16(a.o_b) && rows16(a.o_h) && rows16(a.o_r) &&
         !query_kernel_faster(a, dtype);
}

// Launches that split prompts' keys over workgroups (a diagnostic for tests).
std::atomic<long long> g_key_split_launches{0};

// Workgroup shapes of a causal launch (QT x KG waves, SW): queries per tile
// and how many ways the tile's keys are split inside the workgroup.
enum CausalConfig : int {
  kTiny,    // 64 queries, unsplit: two waves and rounds of 32 keys, for prompts of one key block
  kShort,   // 64 queries, 2 ways: four waves and rounds of 64 keys, for two key blocks
  kNarrow,  // 32 queries, up to 8 ways
  kDeep,    // 64 queries, 4 ways
  kDense,   // 64 queries, 4 ways, two workgroups per compute unit (16-bit types, head dims to 64)
  kWide     // 128 queries, 2 ways, two workgroups per compute unit likewise
};
int config_queries(int config) { return config == kNarrow ? 32 : config == kWide ? 128 : 64; }

// How a causal launch runs: its shape, and with share > 0 the blocks of
// kPfBlock keys after which a tile's keys go to another workgroup.
struct CausalPlan {
  int config, share;
};

// tiles32/64/128: workgroups (tiles x heads, over all prompts) for tiles of
// that many queries; blocks: key blocks of the longest tile; row_bytes: a K
// row in LDS; queries: of the longest prompt; fp32: the type. Where the lines lie (MI355X, 256 compute units, us per call):
// * kTiny and kShort for prompts of one and two key blocks, which end before
//   wider workgroups have met: 8 x 100 tokens x 25 heads fp16 9.3 kShort
//   against 11.5 kDense. Two blocks of a 16-bit type run kDeep while 64-query
//   tiles take one round, whose eight waves stage and compute them at once: 16
//   prompts of 20-60 tokens at offset 60 x 12 heads bf16 9.6 kShort and 8.7, 27
//   of 31-62 at 29 18.7 and 16.6 (17.6 on the kernel before); in fp32 the two
//   are within 3 % of each other either way.
// * kNarrow while its workgroups take one round of the compute units (an
//   eighth more still end with the long tiles): 300 tokens x 12 heads bf16 8.0
//   against 8.8 kDeep, 700 x 12 fp32 (264 workgroups) 25.8 against 33.1; but
//   1000 x 16 bf16 (512) 17.5 against 15.2 kDeep.
//   Also for every launch of prompts of at most 32 queries in rows of more than
//   128 bytes: half the waves of a wider tile would have none (fp32, 8 queries
//   of 64 requests at 500 keys x 12 heads 62 against 120 kDeep, head dim 128 177
//   against 247). Shorter rows keep kDense, whose second workgroup per compute
//   unit makes up for it (fp16: 26 against 28).
// * kDeep while 64-query tiles take one round; then kDense, whose second
//   workgroup per compute unit covers for the first: 1000 x 25 bf16 18.9
//   against 21.5 kDeep and 24.8 kWide.
// * kWide from one and a half rounds of 128-query tiles on, when what a tile
//   spends outside its key loop counts: 8 x 512 tokens x 25 heads 33.1
//   against 42.9 kDense; below it kDense (2048 at offset 2048 x 16: 60 against 76).
// * Splitting over workgroups costs a merge launch (about 5 us): only when
//   narrow tiles leave half the compute units idle and the longest walks at
//   least 8 rounds, in pieces of at least 3 (40 tokens at offset 4000 x 12
//   heads bf16: 15.5 against 26.9).
CausalPlan causal_plan(int64_t tiles32, int64_t tiles64, int64_t tiles128, int blocks, int row_bytes, int queries, bool fp32) {
  const int64_t cus = std::max(1, device_compute_units());
  CausalPlan plan{};
  const bool narrow = 8 * tiles32 <= 9 * cus || (queries <= 32 && row_bytes > 128);
  plan.config = blocks == 1             ? kTiny
                : blocks == 2           ? (tiles64 <= cus && !fp32 ? kDeep : kShort)
                : narrow                ? kNarrow
                : tiles64 <= cus        ? kDeep
                : 2 * tiles128 < 3 * cus ? kDense
                                        : kWide;
  const int round = std::max(1, 4 * 128 / row_bytes);  // blocks a narrow workgroup takes per round
  if (plan.config == kNarrow && 2 * tiles32 <= cus && blocks >= 8 * round) {
    const int64_t pieces = std::min<int64_t>(std::min<int64_t>(cus / tiles32, 64), blocks / (3 * round));
    plan.share = int((blocks + pieces - 1) / pieces);
  }
  return plan;
}

template <int DT, int DP, class Items, bool FUSED>
void launch_causal_t(int config, int blocks, const QueryArgs& a, const Items& items) {
  constexpr int CPR = DP * elem_bytes<DT>() / 16;
  constexpr int SW = CPR == 32 ? 1 : 2;              // waves per SIMD the operands leave room for
  constexpr int NK = CPR == 8 ? 8 : CPR == 16 ? 4 : 2;  // ways a narrow tile's keys are split
  constexpr int DK = CPR == 32 ? 2 : 4;
  if (config == kTiny) {
    causal_kernel<DT, DP, 2, 1, SW, Items, FUSED><<<blocks, 2 * kWave>>>(a, items);
  } else if (config == kShort) {
    causal_kernel<DT, DP, 2, 2, CPR == 8 ? 3 : SW, Items, FUSED><<<blocks, 4 * kWave>>>(a, items);
  } else if (config == kNarrow) {
    causal_kernel<DT, DP, 1, NK, CPR == 8 ? 2 : 1, Items, FUSED><<<blocks, NK * kWave>>>(a, items);
  } else if constexpr (CPR == 8) {
    if (config == kDeep) causal_kernel<DT, DP, 2, 4, 2, Items, FUSED><<<blocks, 8 * kWave>>>(a, items);
    else if (config == kDense) causal_kernel<DT, DP, 2, 4, 4, Items, FUSED><<<blocks, 8 * kWave>>>(a, items);
    else causal_kernel<DT, DP, 4, 2, 4, Items, FUSED><<<blocks, 8 * kWave>>>(a, items);
  } else if (config == kWide) {
    causal_kernel<DT, DP, 4, DK / 2, SW, Items, FUSED><<<blocks, 2 * DK * kWave>>>(a, items);
  } else {
    causal_kernel<DT, DP, 2, DK, SW, Items, FUSED><<<blocks, 2 * DK * kWave>>>(a, items);
  }
}
template <int DT, class Items>
void launch_causal_dt(int config, int blocks, const QueryArgs& a, const Items& items) {
  const bool small = a.g.dim <= 64;
  if constexpr (std::is_same<Items, RaggedItems>::value) {
    if (small) launch_causal_t<DT, 64, Items, true>(config, blocks, a, items);
    else launch_causal_t<DT, 128, Items, true>(config, blocks, a, items);
  } else if (a.k) {
    if (small) launch_causal_t<DT, 64, Items, true>(config, blocks, a, items);
    else launch_causal_t<DT, 128, Items, true>(config, blocks, a, items);
  } else {
    if (small) launch_causal_t<DT, 64, Items, false>(config, blocks, a, items);
    else launch_causal_t<DT, 128, Items, false>(config, blocks, a, items);
  }
}
template <class Items>
void launch_causal(int config, int dtype, int64_t items_count, const QueryArgs& a, const Items& items) {
  const int blocks = grid_for(items_count);
  if (dtype == kF32) launch_causal_dt<kF32>(config, blocks, a, items);
  else if (dtype == kF16) launch_causal_dt<kF16>(config, blocks, a, items);
  else launch_causal_dt<kBF16>(config, blocks, a, items);
}

// Causal attention launch for any q/out strides: the matrix-core causal
// kernel where causal_kernel_takes, the per-query kernel otherwise (which
// reads every key from the pages: a.k must then be null).
hipError_t launch_query(QueryArgs& a, int dtype) {
  const int d = a.g.dim;
  const int esize = dtype == kF32 ? 4 : 2;
  auto rows16 = [&](int64_t x) { return (x * esize) % 16 == 0; };
  const bool vec = (d == 64 || d == 128) && aligned16(a.out) && aligned16(a.q) && rows16(a.q_b) &&
                   rows16(a.q_h) && rows16(a.q_r) && rows16(a.o_b) && rows16(a.o_h) && rows16(a.o_r);
  a.qscale = (1.0f / std::sqrt(float(d))) * kLog2e;
  const int h = a.g.heads;
  if (causal_kernel_takes(a, dtype)) {
    const int64_t bh = int64_t(a.batch) * h;
    auto tiles = [&](int tq) { return (a.nq + tq - 1) / tq; };
    const int most = key_blocks(tiles(64) - 1, 64, a.nq, a.offset);
    const CausalPlan plan = causal_plan(bh * tiles(32), bh * tiles(64), bh * tiles(128), most,
                                         (d <= 64 ? 64 : 128) * esize, a.nq, dtype == kF32);
    const int tq = config_queries(plan.config);
    UniformItems items{tiles(tq), 1, 0};
    if (plan.share > 0) {
      const int pieces = (most + plan.share - 1) / plan.share;
      void* ws = nullptr;
      // Without room for the partials the launch runs unsplit.
      if (pieces > 1 && library_workspace(size_t(bh) * items.tiles * pieces * tq * (d <= 64 ? 68 : 132) * sizeof(float),
                                          &ws) == hipSuccess) {
        items.pieces = pieces;
        items.share = plan.share;
        a.partials = static_cast<float*>(ws);
      }
    }
    a.items = bh * items.tiles * items.pieces;
    launch_causal(plan.config, dtype, a.items, a, items);
    if (items.pieces > 1) {
      const int blocks = grid_for(bh * items.tiles);
#define MT_MERGE(DT)                                                              \
  if (d <= 64) uniform_merge_kernel<DT, 64><<<blocks, 256>>>(a, items, tq);       \
  else uniform_merge_kernel<DT, 128><<<blocks, 256>>>(a, items, tq);
      if (dtype == kF32) { MT_MERGE(kF32) }
      else if (dtype == kF16) { MT_MERGE(kF16) }
      else { MT_MERGE(kBF16) }
#undef MT_MERGE
      g_key_split_launches.fetch_add(1, std::memory_order_relaxed);
    }
    return hipGetLastError();
  }
  if (a.k) return hipErrorInvalidValue;
  a.items = int64_t(a.batch) * h * ((a.nq + kWaves - 1) / kWaves);
  const int blocks = grid_for(a.items);
#define MT_QUERY(DT)                                                                   \
  if (vec && d == 64) query_kernel<DT, 64, true, 2><<<blocks, kThreads>>>(a);          \
  else if (vec && d == 128) query_kernel<DT, 128, true, 2><<<blocks, kThreads>>>(a);   \
  else query_kernel<DT, 128, false, 1><<<blocks, kThreads>>>(a);
  if (dtype == kF32) { MT_QUERY(kF32) }
  else if (dtype == kF16) { MT_QUERY(kF16) }
  else { MT_QUERY(kBF16) }
#undef MT_QUERY
  return hipGetLastError();
}

}  // namespace

extern "C" {

int mt_paged_append(const void* k, const void* v, const uint64_t* slabs, const int* table, int b,
                    int h, int n, int d, int page_size, int pages_per_slab, int num_slabs,
                    int columns, int layer, int layers, int offset, int dtype) {
  if (!k || !v || !slabs || !table) return hipErrorInvalidValue;
  if (int64_t(offset) + n > INT32_MAX ||
      !paged_shape(b, h, n, offset + n, d, page_size, pages_per_slab, num_slabs, columns, layer,
                   layers, offset))
    return hipErrorInvalidValue;
  if (dtype < 0 || dtype > 2) return hipErrorInvalidValue;
  AppendArgs a{};
  a.k = k; a.v = v; a.slabs = slabs; a.table = table; a.batch = b; a.n = n; a.offset = offset;
  a.g = make_geometry(h, d, page_size, pages_per_slab, num_slabs, columns, layer);
  a.src_b = int64_t(h) * n * d; a.src_h = int64_t(n) * d; a.src_r = d;
  return launch_append(a, dtype);
}

int mt_paged_attention(void* out, const void* q, const uint64_t* slabs, const int* table, int b,
                       int h, int nq, int nk, int d, int page_size, int pages_per_slab,
                       int num_slabs, int columns, int layer, int layers, int offset, int dtype) {
  if (!out || !q || !slabs || !table) return hipErrorInvalidValue;
  if (!paged_shape(b, h, nq, nk, d, page_size, pages_per_slab, num_slabs, columns, layer, layers,
                   offset))
    return hipErrorInvalidValue;
  if (dtype < 0 || dtype > 2) return hipErrorInvalidValue;
  QueryArgs a{};
  a.out = out; a.q = q; a.slabs = slabs; a.table = table;
  a.batch = b; a.nq = nq; a.nk = nk; a.offset = offset;
  a.g = make_geometry(h, d, page_size, pages_per_slab, num_slabs, columns, layer);
  a.q_b = a.o_b = int64_t(h) * nq * d;
  a.q_h = a.o_h = int64_t(nq) * d;
  a.q_r = a.o_r = d;
  if (nq == 1) {
    const hipError_t e = decode_uniform(out, q, nullptr, nullptr, slabs, table, b, nk, int64_t(h) * d, dtype, a.g);
    if (e != hipErrorNotSupported) return e;
  }
  return launch_query(a, dtype);
}

int mt_paged_prefill(void* out, const void* q, const void* k, const void* v, const uint64_t* slabs,
                     const int* table, int b, int h, int n, int d, int page_size,
                     int pages_per_slab, int num_slabs, int columns, int layer, int layers,
                     int offset, int dtype, int qkv_stride, int out_stride) {
  if (!out || !q || !k || !v || !slabs || !table) return hipErrorInvalidValue;
  const int64_t hd = int64_t(h) * d;
  if (qkv_stride == 0) qkv_stride = int(hd);
  if (out_stride == 0) out_stride = int(hd);
  if (int64_t(offset) + n > INT32_MAX || qkv_stride < hd || out_stride < hd ||
      int64_t(b) * n * qkv_stride > INT32_MAX || int64_t(b) * n * out_stride > INT32_MAX ||
      !paged_shape(b, h, n, offset + n, d, page_size, pages_per_slab, num_slabs, columns, layer,
                   layers, offset))
    return hipErrorInvalidValue;
  if (dtype < 0 || dtype > 2) return hipErrorInvalidValue;
  QueryArgs a{};
  a.out = out; a.q = q; a.slabs = slabs; a.table = table;
  a.batch = b; a.nq = n; a.nk = offset + n; a.offset = offset;
  a.g = make_geometry(h, d, page_size, pages_per_slab, num_slabs, columns, layer);
  a.q_b = int64_t(n) * qkv_stride; a.q_h = d; a.q_r = qkv_stride;
  a.o_b = int64_t(n) * out_stride; a.o_h = d; a.o_r = out_stride;
  if (n == 1 && out_stride == hd) {
    // one token: append and attention in the decode's one launch
    const hipError_t e = decode_uniform(out, q, k, v, slabs, table, b, offset + 1, qkv_stride, dtype, a.g);
    if (e != hipErrorNotSupported) return e;
  }
  if (causal_kernel_takes(a, dtype) && aligned16(k) && aligned16(v)) {
    // The causal kernel reads the new keys from k/v and writes them to
    // their pages itself: no separate append.
    a.k = k; a.v = v;
    return launch_query(a, dtype);
  }
  AppendArgs ap{};
  ap.k = k; ap.v = v; ap.slabs = slabs; ap.table = table; ap.batch = b; ap.n = n; ap.offset = offset;
  ap.g = a.g;
  ap.src_b = int64_t(n) * qkv_stride; ap.src_h = d; ap.src_r = qkv_stride;
  hipError_t e = launch_append(ap, dtype);
  if (e != hipSuccess) return e;
  return launch_query(a, dtype);
}

int mt_paged_prefill_ragged(void* out, const void* q, const void* k, const void* v,
                            const uint64_t* slabs, const int* const* tables, const int* tokens,
                            const int* offsets, int requests, int h, int d, int page_size,
                            int pages_per_slab, int num_slabs, int columns, int layer, int layers,
                            int dtype, int qkv_stride, int out_stride) {
  if (!out || !q || !k || !v || !slabs || !tables || !tokens || !offsets || requests < 1 || h < 1 ||
      d < 1 || dtype < 0 || dtype > 2)
    return hipErrorInvalidValue;
  const int64_t hd = int64_t(h) * d;
  if (qkv_stride == 0) qkv_stride = int(hd);
  if (out_stride == 0) out_stride = int(hd);
  if (qkv_stride < hd || out_stride < hd) return hipErrorInvalidValue;
  int64_t total = 0;
  for (int r = 0; r < requests; ++r) {
    if (!tables[r] || tokens[r] < 1 || offsets[r] < 0 || int64_t(offsets[r]) + tokens[r] > INT32_MAX ||
        !paged_shape(1, h, tokens[r], offsets[r] + tokens[r], d, page_size, pages_per_slab, num_slabs,
                     columns, layer, layers, offsets[r]))
      return hipErrorInvalidValue;
    total += tokens[r];
  }
  if (total * qkv_stride > INT32_MAX || total * out_stride > INT32_MAX) return hipErrorInvalidValue;
  const size_t e = dtype == kF32 ? 4 : 2;
  auto rows16 = [&](int64_t x) { return (x * int64_t(e)) % 16 == 0; };
  const bool mfma = aligned16(out) && aligned16(q) && aligned16(k) && aligned16(v) && rows16(qkv_stride) &&
                    rows16(out_stride) && rows16(d);
  if (!mfma) {
    // Shapes the matrix-core kernel does not take: one call per prompt.
    int64_t first = 0;
    for (int r = 0; r < requests; ++r) {
      const int st = mt_paged_prefill(static_cast<char*>(out) + size_t(first) * out_stride * e,
                                      static_cast<const char*>(q) + size_t(first) * qkv_stride * e,
                                      static_cast<const char*>(k) + size_t(first) * qkv_stride * e,
                                      static_cast<const char*>(v) + size_t(first) * qkv_stride * e, slabs,
                                      tables[r], 1, h, tokens[r], d, page_size, pages_per_slab, num_slabs,
                                      columns, layer, layers, offsets[r], dtype, qkv_stride, out_stride);
      if (st) return st;
      first += tokens[r];
    }
    return hipSuccess;
  }
  const Geometry g = make_geometry(h, d, page_size, pages_per_slab, num_slabs, columns, layer);
  // Chunks of at most kRaggedPrompts prompts and kRaggedTiles query tiles.
  int r0 = 0;
  int64_t row0 = 0;
  while (r0 < requests) {
    RaggedItems it{};
    int r1 = r0;
    int64_t rows = 0;
    int most = 0;  // key blocks of the longest tile
    int queries = 0;  // tokens of the longest prompt
    int64_t tiles32 = 0, tiles64 = 0, tiles128 = 0;
    while (r1 < requests && r1 - r0 < kRaggedPrompts && tiles64 + (tokens[r1] + 63) / 64 <= kRaggedTiles) {
      const int p = r1 - r0;
      it.first_row[p] = int(rows);
      it.n[p] = tokens[r1];
      it.offset[p] = offsets[r1];
      it.table[p] = tables[r1];
      queries = std::max(queries, tokens[r1]);
      most = std::max(most, key_blocks((tokens[r1] - 1) / 64, 64, tokens[r1], offsets[r1]));
      tiles32 += (tokens[r1] + 31) / 32;
      tiles64 += (tokens[r1] + 63) / 64;
      tiles128 += (tokens[r1] + 127) / 128;
      rows += tokens[r1];
      ++r1;
    }
    if (r1 == r0) {
      // One prompt with more query tiles than a launch describes: on its own.
      const size_t qo = size_t(row0) * qkv_stride * e;
      const int st = mt_paged_prefill(static_cast<char*>(out) + size_t(row0) * out_stride * e,
                                      static_cast<const char*>(q) + qo, static_cast<const char*>(k) + qo,
                                      static_cast<const char*>(v) + qo, slabs, tables[r0], 1, h, tokens[r0], d,
                                      page_size, pages_per_slab, num_slabs, columns, layer, layers,
                                      offsets[r0], dtype, qkv_stride, out_stride);
      if (st) return st;
      row0 += tokens[r0];
      ++r0;
      continue;
    }
    it.prompts = r1 - r0;
    // (narrow tiles only where the launch can list them)
    const CausalPlan plan = causal_plan(tiles32 <= kRaggedTiles ? tiles32 * h : INT64_MAX / 16, tiles64 * h,
                                        tiles128 * h, most, (d <= 64 ? 64 : 128) * int(e),
                                        tiles32 <= kRaggedTiles ? queries : INT_MAX, dtype == kF32);
    const int tq = config_queries(plan.config);
    // (prompt, tile) pairs and their key blocks, the longest first; with a
    // share, cut into pieces of at most that many blocks as far as the
    // launch describes them.
    struct Piece { int p, t, kb0, kb1, slot, at; };
    Piece list[kRaggedTiles];
    RaggedMerge mg{};
    int share = plan.share, pairs = 0, slots = 0;
    auto cut = [&](bool write) {
      int count = 0;
      for (int p = 0; p < it.prompts; ++p)
        for (int t = 0; t * tq < it.n[p]; ++t) {
          const int nb = key_blocks(t, tq, it.n[p], it.offset[p]);
          const int n = share > 0 ? (nb + share - 1) / share : 1;
          if (write) {
            if (n > 1) {
              mg.row0[mg.tiles] = it.first_row[p] + t * tq;
              mg.nq[mg.tiles] = static_cast<unsigned short>(std::min(tq, it.n[p] - t * tq));
              mg.first_slot[mg.tiles] = static_cast<unsigned short>(slots);
              mg.splits[mg.tiles] = static_cast<unsigned char>(n);
              ++mg.tiles;
            }
            for (int j = 0; j < n; ++j)
              list[count + j] = {p, t, j * share, n > 1 ? std::min(nb, (j + 1) * share) : nb, n > 1 ? slots++ : -1, count + j};
          }
          count += n;
        }
      return count;
    };
    while (share > 0 && cut(false) > kRaggedTiles) ++share;
    void* ws = nullptr;
    if (share > 0) {
      // Without room for the partials the launch runs unsplit.
      pairs = cut(true);
      if (most > 65535 ||
          (slots && library_workspace(size_t(slots) * h * tq * (d <= 64 ? 68 : 132) * sizeof(float), &ws) != hipSuccess)) {
        share = slots = 0;
        mg = RaggedMerge{};
      }
    }
    if (share == 0) pairs = cut(true);
    std::sort(list, list + pairs, [](const Piece& x, const Piece& y) {
      const int nx = x.kb1 - x.kb0, ny = y.kb1 - y.kb0;
      return nx != ny ? nx > ny : x.at < y.at;
    });
    const bool split = slots > 0;
    it.pairs = pairs;
    for (int i = 0; i < pairs; ++i) {
      it.pair_prompt[i] = static_cast<unsigned char>(list[i].p);
      it.pair_tile[i] = static_cast<unsigned short>(list[i].t);
      it.pair_kb0[i] = static_cast<unsigned short>(list[i].kb0);
      it.pair_kb1[i] = static_cast<unsigned short>(list[i].kb1);
      it.pair_slot[i] = static_cast<short>(list[i].slot);
    }
    const size_t qoff = size_t(row0) * qkv_stride * e, ooff = size_t(row0) * out_stride * e;
    QueryArgs a{};
    a.out = static_cast<char*>(out) + ooff;
    a.q = static_cast<const char*>(q) + qoff;
    a.k = static_cast<const char*>(k) + qoff;  // the kernel appends the prompts' K/V itself
    a.v = static_cast<const char*>(v) + qoff;
    a.slabs = slabs;
    a.g = g;
    a.qscale = (1.0f / std::sqrt(float(d))) * kLog2e;
    a.q_h = d; a.q_r = qkv_stride;
    a.o_h = d; a.o_r = out_stride;
    a.partials = static_cast<float*>(ws);
    launch_causal(plan.config, dtype, int64_t(pairs) * h, a, it);
    if (split) {
      const unsigned mblocks = unsigned(mg.tiles * h);
#define MT_MERGE(DT)                                                            \
  if (d <= 64) ragged_merge_kernel<DT, 64><<<mblocks, 256>>>(a, mg, tq);        \
  else ragged_merge_kernel<DT, 128><<<mblocks, 256>>>(a, mg, tq);
      if (dtype == kF32) { MT_MERGE(kF32) }
      else if (dtype == kF16) { MT_MERGE(kF16) }
      else { MT_MERGE(kBF16) }
#undef MT_MERGE
      g_key_split_launches.fetch_add(1, std::memory_order_relaxed);
    }
    const hipError_t err = hipGetLastError();
    if (err != hipSuccess) return err;
    r0 = r1;
    row0 += rows;
  }
  return hipSuccess;
}

int mt_paged_decode_batch(void* out, const void* q, const void* k, const void* v,
                          const uint64_t* slabs, const int* table, const int* offsets, int b,
                          int h, int d, int page_size, int pages_per_slab, int num_slabs,
                          int columns, int layer, int layers, int dtype) {
  if (!out || !q || !k || !v || !slabs || !table || !offsets ||
      !paged_shape(b, h, 1, 1, d, page_size, pages_per_slab, num_slabs, columns, layer, layers, 0) ||
      int64_t(columns) * page_size > INT32_MAX)
    return hipErrorInvalidValue;
  if (dtype < 0 || dtype > 2) return hipErrorInvalidValue;
  const int64_t cap = int64_t(columns) * page_size;
  const int S = cap > kDefaultSplitTokens ? idle_split(int64_t(b) * h, cap, d, dtype) : choose_split(cap, 0);
  const int64_t nsplit_max = (cap + S - 1) / S;
  const bool ordered = device_order(b, h, nsplit_max);
  // Workspace: split partials, then the device-built visiting order.
  const size_t part = nsplit_max > 1 ? align256(workspace_bytes_for(int64_t(b) * h, int(nsplit_max))) : 0;
  const size_t ws_bytes = part + (ordered ? order_bytes(b, nsplit_max) : 0);
  void* ws = nullptr;
  if (ws_bytes) {
    const int e = library_workspace(ws_bytes, &ws);
    if (e != hipSuccess) return e;
  }
  int* order = ordered ? reinterpret_cast<int*>(static_cast<char*>(ws) + part) : nullptr;
  return decode_common(out, q, k, v, slabs, table, offsets, b, h, d, page_size, pages_per_slab,
                       num_slabs, columns, layer, layers, dtype, S, 0, 0, 0,
                       nullptr, 0, 0, part ? ws : nullptr, part, true, order);
}

int mt_paged_decode_batch_noalloc(void* out, const void* q, const void* k, const void* v,
                                  const uint64_t* slabs, const int* table, const int* offsets,
                                  int b, int h, int d, int page_size, int pages_per_slab,
                                  int num_slabs, int columns, int layer, int layers, int dtype) {
  if (!out || !q || !k || !v || !slabs || !table || !offsets ||
      !paged_shape(b, h, 1, 1, d, page_size, pages_per_slab, num_slabs, columns, layer, layers, 0) ||
      int64_t(columns) * page_size > INT32_MAX)
    return hipErrorInvalidValue;
  if (dtype < 0 || dtype > 2) return hipErrorInvalidValue;
  const int64_t cap = int64_t(columns) * page_size;
  const int S = cap > kDefaultSplitTokens ? idle_split(int64_t(b) * h, cap, d, dtype) : choose_split(cap, 0);
  const int64_t nsplit_max = (cap + S - 1) / S;
  const bool ordered = device_order(b, h, nsplit_max);
  // The fixed array holds the split partials, then the device-built visiting
  // order; a shape that needs more is refused before any launch.
  const bool vec = decode_rows(d, dtype, out, q, k, v, int64_t(h) * d) == kRowsFull;
  const size_t part = nsplit_max > 1 ? align256(partial_bytes(int64_t(b) * h, nsplit_max, vec, d)) : 0;
  const size_t need = part + (ordered ? order_bytes(b, nsplit_max) : 0);
  if (need > kNoAllocScratchBytes) return hipErrorInvalidValue;
  void* ws = nullptr;
  if (need) {
    const int e = scratch_address(&ws);
    if (e != hipSuccess) return e;
  }
  int* order = ordered ? reinterpret_cast<int*>(static_cast<char*>(ws) + part) : nullptr;
  return decode_common(out, q, k, v, slabs, table, offsets, b, h, d, page_size, pages_per_slab,
                       num_slabs, columns, layer, layers, dtype, S, 0, 0, 0,
                       nullptr, 0, 0, part ? ws : nullptr, part, true, order);
}

int mt_paged_prefill_key_splits(long long* launches) {
  if (!launches) return hipErrorInvalidValue;
  *launches = g_key_split_launches.load(std::memory_order_relaxed);
  return hipSuccess;
}

int mt_paged_decode_workspace_bytes(int b, int h, int page_size, int columns, int split_tokens,
                                    size_t* bytes) {
  if (!bytes || b < 1 || h < 1 || columns < 1 ||
      !(page_size == 8 || page_size == 16 || page_size == 32))
    return hipErrorInvalidValue;
  const int64_t cap = int64_t(columns) * page_size;
  const int S = choose_split(cap, split_tokens);
  if (S < 64 || S % 64 != 0 || S > kMaxSplitTokens) return hipErrorInvalidValue;
  const int64_t nsplit_max = (cap + S - 1) / S;
  *bytes = nsplit_max > 1 ? workspace_bytes_for(int64_t(b) * h, int(nsplit_max)) : 0;
  return hipSuccess;
}

#ifdef MT_DECODE_TIMELINE
// Measurement builds only: copies the first `count` workgroups' records
// (kTimelineFields x uint64 each, see g_decode_timeline) of the last decode
// launch to host memory `dst`, after the calling thread's stream has drained.
int mt_decode_timeline(unsigned long long* dst, int count) {
  if (!dst || count < 1 || count > kTimelineMax) return hipErrorInvalidValue;
  hipError_t e = hipStreamSynchronize(hipStreamPerThread);
  if (e == hipSuccess)
    e = hipMemcpyFromSymbol(dst, HIP_SYMBOL(g_decode_timeline), size_t(count) * kTimelineFields * 8);
  return e;
}
#endif

int mt_paged_decode_split_tokens(int page_size, int columns, int requested, int* split_tokens) {
  if (!split_tokens || columns < 1 || requested < 0 ||
      !(page_size == 8 || page_size == 16 || page_size == 32))
    return hipErrorInvalidValue;
  const int S = choose_split(int64_t(columns) * page_size, requested);
  if (S < 64 || S % 64 != 0 || S > kMaxSplitTokens) return hipErrorInvalidValue;
  *split_tokens = S;
  return hipSuccess;
}

int mt_paged_decode_order(const int* offsets, int b, int h, int page_size, int columns,
                          int split_tokens, int compute_units, int* list, int* count) {
  if (!offsets || !list || !count || b < 1 || b > kOrderRows || h < 1 || columns < 1 ||
      split_tokens < 0 || compute_units < 0 || !(page_size == 8 || page_size == 16 || page_size == 32) ||
      int64_t(columns) * page_size > INT32_MAX)
    return hipErrorInvalidValue;
  const int64_t cap = int64_t(columns) * page_size;
  const int S = choose_split(cap, split_tokens);
  if (S < 64 || S % 64 != 0 || S > kMaxSplitTokens) return hipErrorInvalidValue;
  OrderArgs oa{};
  oa.offsets = offsets; oa.count = count; oa.list = list;
  oa.batch = b; oa.split_tokens = S; oa.cap = cap;
  const int64_t nsplit_max = (cap + S - 1) / S;
  if (int64_t(b) * nsplit_max > INT32_MAX / 2) return hipErrorInvalidValue;
  oa.capacity = int(int64_t(b) * nsplit_max);
  oa.per = std::max(1, (compute_units ? compute_units : device_compute_units()) / h);
  order_kernel<<<1, kOrderThreads>>>(oa);
  return hipGetLastError();
}

int mt_paged_decode_split(void* out, const void* q, const void* k, const void* v,
                          const uint64_t* slabs, const int* table, const int* offsets, int b,
                          int h, int d, int page_size, int pages_per_slab, int num_slabs,
                          int columns, int layer, int layers, int dtype, int split_tokens,
                          int unroll, int waves, int qkv_stride, const int* work,
                          int work_items, int merge_rows, void* workspace,
                          size_t workspace_bytes) {
  if (!out || !q || !k || !v || !slabs || !table || !offsets ||
      !paged_shape(b, h, 1, 1, d, page_size, pages_per_slab, num_slabs, columns, layer, layers, 0) ||
      int64_t(columns) * page_size > INT32_MAX || split_tokens < 0 || unroll < 0 ||
      (waves != 0 && waves != 2 && waves != 4 && waves != 8) ||
      (qkv_stride != 0 && int64_t(qkv_stride) < int64_t(h) * d) || qkv_stride < 0)
    return hipErrorInvalidValue;
  if (dtype < 0 || dtype > 2) return hipErrorInvalidValue;
  return decode_common(out, q, k, v, slabs, table, offsets, b, h, d, page_size, pages_per_slab,
                       num_slabs, columns, layer, layers, dtype, split_tokens,
                       unroll, waves, qkv_stride,
                       work, work_items, merge_rows, workspace, workspace_bytes);
}

}  // extern "C"
