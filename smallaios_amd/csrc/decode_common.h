// Device helpers shared by the int8 and int4 decode kernels: lane-group
// reductions, the hi/lo pair swap, vector loads of a Q chunk, RoPE of one
// element, and the (sequence, split) mapping of a decode workgroup.
//
// Wave layout used by both kernels: lane = r + 16 g (r = lane & 15 is the
// MFMA row/column index, g = lane >> 4 the lane group, i.e. the page of the
// current 64-token tile).
#pragma once

#include "sai_internal.h"

namespace sai {

typedef int v4i __attribute__((ext_vector_type(4)));

constexpr int kMaxSplitPages = 1024;  // split_tokens <= 16384 (page ids staged in LDS)

// RoPE of one element; `first` = this element is x0 of its pair. Both
// products are rounded on their own and the select picks the sign of the
// second, so x0: c*x0 - s*x1 and x1: s*x0 + c*x1 (== c*x1 + s*x0) without a
// branch per lane.
__device__ __forceinline__ float rope_elem(float c, float s, float own, float partner,
                                           bool first) {
#pragma clang fp contract(off)
  const float a = c * own;
  const float b = s * partner;
  return a + (first ? -b : b);
}

__device__ __forceinline__ int pack4(int a, int b, int c, int d) {
  return (a & 0xFF) | ((b & 0xFF) << 8) | ((c & 0xFF) << 16) | ((int)((unsigned)d << 24));
}

// exchange with the neighbouring lane: quad_perm(1,0,3,2)
__device__ __forceinline__ int swap_pair(int v) {
  return __builtin_amdgcn_mov_dpp(v, 0xB1, 0xF, 0xF, false);
}

// max / sum over the four lane groups (lanes r, r+16, r+32, r+48)
__device__ __forceinline__ float xgroup_max(float v) {
  auto a = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  v = fmaxf(__uint_as_float(a[0]), __uint_as_float(a[1]));
  auto b = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return fmaxf(__uint_as_float(b[0]), __uint_as_float(b[1]));
}
__device__ __forceinline__ float xgroup_sum(float v) {
  auto a = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  v = __uint_as_float(a[0]) + __uint_as_float(a[1]);
  auto b = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return __uint_as_float(b[0]) + __uint_as_float(b[1]);
}

__device__ __forceinline__ float fast_exp2(float x) { return __builtin_amdgcn_exp2f(x); }

template <int K>
__device__ __forceinline__ float comp4(const float4& v) {
  if constexpr (K == 0) return v.x;
  else if constexpr (K == 1) return v.y;
  else if constexpr (K == 2) return v.z;
  else return v.w;
}

// Element I of 16 table entries loaded as four float4 q[0..3] from the run's
// start: split-half pairs take entry I, interleaved pairs entry I / 2. Both
// candidates are constant components of SSA values, so the select stays a
// v_cndmask (a select between two elements of one local array is turned into
// dynamic register indexing, which waits for the loads at once).
template <int I>
__device__ __forceinline__ float rope_pick(const float4 (&q)[4], bool interleaved) {
  const float split_half = comp4<I & 3>(q[I >> 2]);
  const float inter = comp4<(I >> 1) & 3>(q[I >> 3]);
  return interleaved ? inter : split_half;
}

template <int I>
__device__ __forceinline__ void rope_pick_all(const float4 (&qc)[4], const float4 (&qs)[4],
                                              bool interleaved, float (&c)[16], float (&s)[16]) {
  c[I] = rope_pick<I>(qc, interleaved);
  s[I] = rope_pick<I>(qs, interleaved);
  if constexpr (I + 1 < 16) rope_pick_all<I + 1>(qc, qs, interleaved, c, s);
}

// The cos / sin table entries of the 16 dims [c0, c0 + 16) of a query row at
// one position (cr, sr: that position's table rows of head_dim / 2 entries,
// 16-byte aligned): split-half pairs use entries c0 mod (D/2) + i,
// interleaved pairs entry (c0 + i) / 2. rope_load16 issues four 16-byte loads
// per table whatever the pairing (interleaved needs the first two; the other
// two repeat them, since base + 16 may pass the row end), 8 loads instead of
// 32; rope_pick_all turns them into per-dim values where they are used, so
// that nothing waits for the loads before then.
template <int D>
__device__ __forceinline__ void rope_load16(const float* cr, const float* sr, int c0,
                                            int interleaved, float4 (&qc)[4], float4 (&qs)[4]) {
  constexpr int HALF = D / 2;
  const bool il = interleaved != 0;
  const int base = il ? (c0 >> 1) : (c0 < HALF ? c0 : c0 - HALF);
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int off = base + 4 * (il ? (j & 1) : j);
    qc[j] = *(const float4*)(cr + off);
    qs[j] = *(const float4*)(sr + off);
  }
}

// Split partials handed between workgroups of one launch. The workgroups of
// a (sequence, kv head) run on different XCDs, whose L2 caches are not kept
// coherent with each other for ordinary stores. An agent-scope atomic store or
// load is coherent across them by itself (gfx950 emits global_store /
// global_load with sc1), so the handoff needs no L2 writeback or invalidate:
// the writer stores its partial this way, waits for the stores to complete
// (partials_complete), and only then takes a ticket from the counter; the
// workgroup with the last ticket loads the other partials this way.
__device__ __forceinline__ void store_partial(float* a, float v) {
  __hip_atomic_store(a, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ float load_partial(const float* a) {
  return __hip_atomic_load(a, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// Two neighbouring floats at once (8-byte aligned: a partial's rows hold an
// even number of floats).
__device__ __forceinline__ void store_partial2(float* a, float v0, float v1) {
  __hip_atomic_store((unsigned long long*)a,
                     (unsigned long long)__float_as_uint(v0) |
                         ((unsigned long long)__float_as_uint(v1) << 32),
                     __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ float2 load_partial2(const float* a) {
  const unsigned long long w = __hip_atomic_load((const unsigned long long*)a, __ATOMIC_RELAXED,
                                                 __HIP_MEMORY_SCOPE_AGENT);
  return float2{__uint_as_float((uint32_t)w), __uint_as_float((uint32_t)(w >> 32))};
}
// Every vector memory access of this wave issued so far has completed (on
// gfx9 vmcnt counts stores until they are acknowledged); also a compiler
// barrier, so no store is moved past it.
__device__ __forceinline__ void partials_complete() {
  __asm__ volatile("s_waitcnt vmcnt(0)" ::: "memory");
}
// One ticket of the split counter of a (sequence, kv head); true for the
// workgroup that takes the last one, which then resets the counter for the
// next launch. Call after partials_complete() and a workgroup barrier.
__device__ __forceinline__ bool last_ticket(int* counter, int nsplit) {
  return __hip_atomic_fetch_add(counter, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) ==
         nsplit - 1;
}
__device__ __forceinline__ void reset_ticket(int* counter) {
  __hip_atomic_store(counter, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Online merge of the splits' (m, l, o) entries for one (head, dim) into
// (M, Ls, O), C splits per round trip, in split order, skipping splits with no
// visible key; `ph` points at split 0's (m, l, o[...]) block of this head,
// `stride` floats apart per split, `d` the dim.
template <int C>
__device__ __forceinline__ void merge_partials(const float* ph, size_t stride, int d, int nsplit,
                                               float& M, float& Ls, float& O) {
  for (int s0 = 0; s0 < nsplit; s0 += C) {
    float m[C], l[C], o[C];
#pragma unroll
    for (int i = 0; i < C; ++i) {
      const int s = min(s0 + i, nsplit - 1);
      const float* ps = ph + (size_t)s * stride;
      m[i] = load_partial(ps);
      l[i] = load_partial(ps + 1);
      o[i] = load_partial(ps + 2 + d);
    }
#pragma unroll
    for (int i = 0; i < C; ++i) {
      const int s = s0 + i;
      if (s >= nsplit || m[i] == -INFINITY) continue;
      const float mn = fmaxf(M, m[i]);
      const float fa = M == -INFINITY ? 0.0f : fast_exp2(M - mn);
      const float fb = fast_exp2(m[i] - mn);
      Ls = Ls * fa + l[i] * fb;
      O = O * fa + o[i] * fb;
      M = mn;
    }
  }
}

// The merge of a (sequence, kv head)'s nsplit partials by one workgroup of NT
// threads: p0 points at split 0's block [G][m, l, o[D]], `stride` floats to
// the next split's. A thread takes pairs of neighbouring dims; the loads of C
// splits for all its pairs go out together with the (m, l) of those splits,
// which reach the other threads through LDS (sm: C * G float2). Every load of
// partials written on other XCDs is a full memory latency, so what counts is
// the number of dependent rounds: one per C splits, whatever the entries per
// thread. (One entry after the other, each loading its own m and l, took a
// round per entry: 1 x 16384 in 32 splits, 8Q/1KV, D = 128, 30.1 us per step,
// in one round per 16 splits 22.6; 1 x 8192 in 16, 32Q/8KV, 15.8 -> 13.9; the
// Gemma 3 4B window layer in 5, 16.9 -> 16.0.) The result does not depend on
// which workgroup merges.
// store(head, dim, v0, v1) takes dims dim, dim + 1.
template <int D, int G, int NT, int C, class F>
__device__ __forceinline__ void merge_splits_by(const float* p0, size_t stride, int nsplit,
                                                float2* sm, F&& store) {
  constexpr int E = G * D / 2;  // pairs
  constexpr int PER = (E + NT - 1) / NT;
  const int tid = threadIdx.x;
  float M[PER], L[PER], O0[PER], O1[PER];
#pragma unroll
  for (int k = 0; k < PER; ++k) {
    M[k] = -INFINITY;
    L[k] = O0[k] = O1[k] = 0.0f;
  }
  for (int s0 = 0; s0 < nsplit; s0 += C) {
    const int n = min(C, nsplit - s0);
    const float* ps = p0 + (size_t)s0 * stride;
    float2 o[PER][C];
#pragma unroll
    for (int k = 0; k < PER; ++k) {
      const int e = min(tid + k * NT, E - 1), hd = e / (D / 2), d = 2 * (e % (D / 2));
#pragma unroll
      for (int i = 0; i < C; ++i)
        o[k][i] = load_partial2(ps + (size_t)min(i, n - 1) * stride + hd * (D + 2) + 2 + d);
    }
    for (int t = tid; t < C * G; t += NT) {
      const int i = t / G;
      const float2 ml = load_partial2(ps + (size_t)min(i, n - 1) * stride + (t % G) * (D + 2));
      sm[t] = i < n ? ml : float2{-INFINITY, 0.0f};
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < PER; ++k) {
      const int hd = min(tid + k * NT, E - 1) / (D / 2);
      float2 ml[C];  // read together: no branch between the LDS reads
#pragma unroll
      for (int i = 0; i < C; ++i) ml[i] = sm[i * G + hd];
      float mb = M[k];
#pragma unroll
      for (int i = 0; i < C; ++i) mb = fmaxf(mb, ml[i].x);
      // splits without a visible key (m = -inf, l = o = 0) weigh 2^-inf = 0
      const float ref = mb == -INFINITY ? 0.0f : mb;
      const float f0 = fast_exp2(M[k] - ref);
      L[k] *= f0;
      O0[k] *= f0;
      O1[k] *= f0;
#pragma unroll
      for (int i = 0; i < C; ++i) {
        const float f = fast_exp2(ml[i].x - ref);
        L[k] += ml[i].y * f;
        O0[k] += o[k][i].x * f;
        O1[k] += o[k][i].y * f;
      }
      M[k] = mb;
    }
    if (s0 + C < nsplit) __syncthreads();  // sm is written again
  }
#pragma unroll
  for (int k = 0; k < PER; ++k) {
    const int e = tid + k * NT;
    if (E % NT != 0 && e >= E) break;
    store(e / (D / 2), 2 * (e % (D / 2)), L[k] > 0.0f ? O0[k] / L[k] : 0.0f,
          L[k] > 0.0f ? O1[k] / L[k] : 0.0f);
  }
}

// Rounds of 4, 8 or 16 splits by the split count (uniform).
template <int D, int G, int NT, class F>
__device__ __forceinline__ void merge_splits(const float* p0, size_t stride, int nsplit,
                                             float2* sm, F&& store) {
  if constexpr (G * D <= NT) {
    // An entry per thread, each reading its own (m, l), has no barrier in the
    // way. One wave (G * D <= 64) always takes it (int4, 1 x 4585, 8Q/8KV, D =
    // 64, 9 splits: 11.96 against 12.60 us per step), more waves up to 4 splits
    // (2: int4 2 x 409, 8Q/2KV, 128, 10.7 against 11.05 us, int8 16 x 516, 10.8
    // against 11.05; 3: int4 3 x 590 11.2 against 11.25; 5: int4 6 x 1200 12.35
    // against 12.25).
    if (G * D <= 64 || nsplit <= 4) {
      const int t = threadIdx.x;
      if (t < G * D) {
        const int hd = t / D, d = t % D;
        const float* ph = p0 + hd * (D + 2);
        float M = -INFINITY, L = 0.0f, O = 0.0f;
        if (nsplit <= 2)
          merge_partials<2>(ph, stride, d, nsplit, M, L, O);
        else if (nsplit <= 4)
          merge_partials<4>(ph, stride, d, nsplit, M, L, O);
        else if (nsplit <= 8)
          merge_partials<8>(ph, stride, d, nsplit, M, L, O);
        else
          merge_partials<16>(ph, stride, d, nsplit, M, L, O);
        const float v = L > 0.0f ? O / L : 0.0f;
        const float next = __int_as_float(swap_pair(__float_as_int(v)));
        if ((d & 1) == 0) store(hd, d, v, next);
      }
      return;
    }
  }
  if (nsplit <= 4)
    merge_splits_by<D, G, NT, 4>(p0, stride, nsplit, sm, store);
  else if (nsplit <= 8)
    merge_splits_by<D, G, NT, 8>(p0, stride, nsplit, sm, store);
  else
    merge_splits_by<D, G, NT, 16>(p0, stride, nsplit, sm, store);
}

// 16 consecutive elements (f32 or bf16) starting at element `off`; the
// offset is a multiple of 16 and the row 32-byte aligned.
__device__ __forceinline__ void load16(const void* base, size_t off, int dtype, float (&x)[16]) {
  if (dtype == kDtypeBf16) {
    const uint4* p = (const uint4*)((const uint16_t*)base + off);
    const uint4 a = p[0], b = p[1];
    const uint32_t w[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      x[2 * i] = __uint_as_float(w[i] << 16);
      x[2 * i + 1] = __uint_as_float(w[i] & 0xFFFF0000u);
    }
  } else {
    const float4* p = (const float4*)((const float*)base + off);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float4 v = p[i];
      x[4 * i] = v.x, x[4 * i + 1] = v.y, x[4 * i + 2] = v.z, x[4 * i + 3] = v.w;
    }
  }
}

// The parameters lie in three 64-byte lines of the kernel-argument memory.
// Loaded where each is used, those behind the branches of decode_work_item
// were a memory round trip of their own: 0.1 to 0.2 us of a call. So one of
// each line, and those that the first loads need, are asked for together at
// the start (int8, us per call: 1 x 512, 8Q/2KV, 64, 7.66 -> 7.52; 7 x 200..1900,
// 32Q/8KV, 128, 12.06 -> 11.83; the Gemma 3 4B window layer 14.33 -> 14.12; 16 x
// 8192 the same). The int4 kernel does without: its short calls gain as much
// (14 x 72 9.53 -> 9.33), but its long ones lose 1 % at lengths of 2^14 and 2^15
// (4 x 32768 34.2 -> 34.5).
__device__ __forceinline__ void load_params(const DecodeParams& p) {
  __asm__ volatile("" ::"s"(p.kv_heads), "s"(p.uniform_nsplit), "s"(p.window), "s"(p.page_table),
                   "s"(p.seq_lens), "s"(p.max_pages), "s"(p.pending), "s"(p.split_tokens),
                   "s"(p.k_new), "s"(p.q), "s"(p.q_dtype), "s"(p.pool));
}

// (sequence, split) of a decode workgroup and its split's length in 64-token
// tiles. Uniform split count: direct mapping, splits of split_tokens.
// Ragged: the host's table of work items (p.ordered), or for larger batches a
// prefix scan over the per-sequence split counts of seq_lens[b] + pending
// tokens; a sequence's streamed tiles are dealt evenly to its splits
// (ceil(T / nsplit) each, the last split taking the rest, never none), so no
// split is a short remainder. Returns b = -1 past the last work item.
// (The scan waits for the lengths and then for six lane shuffles: 1.6 us of
// every workgroup at 7 ragged sequences, whose step went from 18.8 to 16.7 us
// with the table and the merge in the kernel.)
__device__ __forceinline__ void decode_work_item(const DecodeParams& p, int work, int lane, int& b,
                                                 int& split, int& nsplit, int& split_base,
                                                 int& tps) {
  b = -1;
  split = nsplit = split_base = 0;
  tps = p.split_tokens / 64;
  if (p.uniform_nsplit > 0) {
    nsplit = p.uniform_nsplit;
    b = work / nsplit;
    split = work - b * nsplit;
    split_base = b * nsplit;
    return;
  }
  if (p.ordered) {
    // the host's table: no lengths, no scan, one round trip
    for (int c0 = 0; c0 < p.batch; c0 += 64) {
      const int i = min(c0 + lane, p.batch - 1);
      const int end = p.item_end[i];
      const int begin = i > 0 ? p.item_end[i - 1] : 0;
      const int sb = p.order[i], tp = p.item_tps[i];
      const unsigned long long m = __ballot(end > work);
      if (m == 0) continue;
      const int first = __ffsll((long long)m) - 1;
      b = __builtin_amdgcn_readlane(sb, first);
      split_base = __builtin_amdgcn_readlane(begin, first);
      nsplit = __builtin_amdgcn_readlane(end, first) - split_base;
      tps = __builtin_amdgcn_readlane(tp, first);
      split = work - split_base;
      return;
    }
    return;
  }
  int base = 0;
  for (int c0 = 0; c0 < p.batch; c0 += 64) {
    const int bi = c0 + lane;
    const int sb = bi < p.batch ? bi : 0;
    const int Lb = bi < p.batch ? p.seq_lens[sb] + p.pending : 0;
    const int span = Lb - window_origin(Lb, p.window);
    const int n = (span + p.split_tokens - 1) / p.split_tokens;
    int incl = n;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
      const int t = __shfl_up(incl, off, 64);
      if (lane >= off) incl += t;
    }
    const int total = __shfl(incl, 63, 64);
    if (work < base + total) {
      const unsigned long long m = __ballot(base + incl > work);
      const int first = __ffsll((long long)m) - 1;
      b = __shfl(sb, first, 64);
      split_base = base + __shfl(incl - n, first, 64);
      nsplit = __shfl(n, first, 64);
      const int tiles = (__shfl(span, first, 64) + 63) / 64;
      tps = (tiles + nsplit - 1) / nsplit;
      split = work - split_base;
      return;
    }
    base += total;
  }
}

// The length of sequence b (seq_lens[b] + pending) and the split's page ids,
// staged into sm_pg (page slot i of the split = sm_pg[i]). The length is a
// scalar load (b is uniform), so it waits on its own counter; without a
// window the split's first page does not depend on it, and the page-id loads
// go out beside it instead of after it: one memory round trip less before the
// first tile. With a window the split starts at the tile holding the first
// visible key, which needs the length first. NT = threads of the workgroup.
template <int NT>
__device__ __forceinline__ void stage_split_pages(const DecodeParams& p, int b, int split, int tps,
                                                  int* sm_pg, int& L, int& k_lo,
                                                  int& first_page) {
  b = __builtin_amdgcn_readfirstlane(b);
  const int32_t* pt = p.page_table + (size_t)b * p.max_pages;
  const int split_pages = tps * (64 / kPageTokens);
  const int len = p.seq_lens[b];
  if (p.window <= 0) {
    first_page = split * split_pages;
    for (int i = threadIdx.x; i < split_pages; i += NT)
      sm_pg[i] = pt[min(first_page + i, p.max_pages - 1)];
    L = len + p.pending;
    k_lo = 0;
  } else {
    L = len + p.pending;
    k_lo = window_first_key(L, p.window);
    first_page = (k_lo / 64) * 64 / kPageTokens + split * split_pages;
    for (int i = threadIdx.x; i < split_pages; i += NT)
      sm_pg[i] = pt[min(first_page + i, p.max_pages - 1)];
  }
}

}  // namespace sai
