// Shared by the kernels that stream a row's keys in splits (paged_attention.hip, few_query.hip): the decode work
// list, and the merge of a split row inside the launch that attends it.
#pragma once

#include "attn_common.h"

namespace lv {

constexpr int kWaves = 4;  // waves per workgroup

// Steps of few queries per row (few_query.hip): at most kFewMaxQueries queries a row, and kFewMaxRows (position, head)
// query rows per kv head -- what one item's accumulators hold at two workgroups per CU.
constexpr int kFewMaxQueries = 16;
constexpr int kFewMaxRows = 64;
// Launches the decode list (at most `items` items of hp kv heads each), rows of at most query_rows (position, head)
// query rows per kv head in one pass over their keys (rows of more take several).
void launch_few_query(const AttnParams& p, int d, int query_rows, int hp, int dtype, int items, hipStream_t stream);

// Decode item i (below the launch's bound, so inside the list's memory), the number of decode items and the keys per
// split, in one round trip: a decode workgroup's start is a chain of dependent loads (item, then lengths and page,
// then keys), and a step of a few short rows is little more than that chain.
struct DecodeWork {
  int row, split, count, per;
};
__device__ __forceinline__ DecodeWork decode_work(const AttnParams& p, int i) {
  DecodeWork w;
  int64_t item;
  asm volatile("s_load_dwordx2 %0, %3, 0x0\n\ts_load_dword %1, %4, %5\n\ts_load_dword %2, %4, %6\n\t"
               "s_waitcnt lgkmcnt(0)"
               : "=&s"(item), "=&s"(w.count), "=&s"(w.per)
               : "s"(p.items + i), "s"(p.n_items), "n"(4 * kPlanDecodes), "n"(4 * kPlanSplit));
  w.row = (int)(uint32_t)item;
  w.split = (int)(item >> 32);
  return w;
}

// A split row's partials pass between workgroups that may run on different XCDs, whose L2 caches are not coherent
// with each other. They are stored and loaded as device-scope relaxed atomics (global_store / global_load with sc1:
// written through to memory, read past the L2), so neither side needs a whole-L2 writeback or invalidate.
__device__ __forceinline__ void coherent_store(float* ptr, float v) {
  __hip_atomic_store(ptr, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ float coherent_load(const float* ptr) {
  return __hip_atomic_load(ptr, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// Two adjacent floats (8-byte aligned) in one access.
__device__ __forceinline__ void coherent_store2(float* ptr, float a, float b) {
  const uint64_t v = (uint64_t)__float_as_uint(a) | (uint64_t)__float_as_uint(b) << 32;
  __hip_atomic_store(reinterpret_cast<uint64_t*>(ptr), v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void coherent_load2(const float* ptr, float& a, float& b) {
  const uint64_t v =
      __hip_atomic_load(reinterpret_cast<const uint64_t*>(ptr), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  a = __uint_as_float((uint32_t)v);
  b = __uint_as_float((uint32_t)(v >> 32));
}

// Merge of a split row's partial outputs: o = sum_s 2^(lse_s - M) o_s / sum_s 2^(lse_s - M). A piece is two adjacent
// dims of one query head's output (its partials in slots slot, slot + stride, ...); a thread merges NP pieces at
// once, reading kMergeLoads / NP splits of each at a time, every load issued before the first is used, with the max
// and the sums carried from batch to batch. The merge is the serial end of a row's step: one round trip past the L2
// per batch, and one set of them per kMergeLoads loads a thread has to make. Each output element's arithmetic depends
// only on its own head, dim and NP, so any spread of the pieces over threads gives the same bits.
constexpr int kMergeLoads = 32;
struct MergePiece {
  int slot, tok, head, d0;  // slot < 0: no piece
};
template <typename T, int D, int NP>
__device__ __forceinline__ void merge_split_partials(const AttnParams& p, const MergePiece (&pc)[NP], int stride,
                                                     int nsplit) {
  using E = Elem<T>;
  constexpr int B = kMergeLoads / NP;
  float m[NP], den[NP], o0[NP], o1[NP];
#pragma unroll
  for (int q = 0; q < NP; ++q) {
    m[q] = -INFINITY;
    den[q] = o0[q] = o1[q] = 0.f;
  }
  for (int s0 = 0; s0 < nsplit; s0 += B) {
    float ls[NP][B], x[NP][B][2];
#pragma unroll
    for (int q = 0; q < NP; ++q)
#pragma unroll
      for (int i = 0; i < B; ++i) {
        ls[q][i] = -INFINITY;
        x[q][i][0] = x[q][i][1] = 0.f;
        if (s0 + i < nsplit && pc[q].slot >= 0) {  // s0 + i < nsplit: uniform over the threads of a row
          const int64_t at = (int64_t)(pc[q].slot + (s0 + i) * stride) * p.hq + pc[q].head;
          ls[q][i] = coherent_load(p.part_lse + at);
          coherent_load2(p.part_o + at * D + pc[q].d0, x[q][i][0], x[q][i][1]);
        }
      }
#pragma unroll
    for (int q = 0; q < NP; ++q) {
      float bm = m[q];
#pragma unroll
      for (int i = 0; i < B; ++i) bm = fmaxf(bm, ls[q][i]);
      const float base = merge_base(bm);
      const float alpha = fast_exp2(m[q] - base);  // 0 while m is -inf
      den[q] *= alpha;
      o0[q] *= alpha;
      o1[q] *= alpha;
#pragma unroll
      for (int i = 0; i < B; ++i) {
        const float w = fast_exp2(ls[q][i] - base);  // 0 past the last split
        den[q] += w;
        o0[q] = fmaf(w, x[q][i][0], o0[q]);
        o1[q] = fmaf(w, x[q][i][1], o1[q]);
      }
      m[q] = bm;
    }
  }
#pragma unroll
  for (int q = 0; q < NP; ++q) {
    if (pc[q].slot < 0) continue;
    const float inv = inv_sum(den[q]);
    *reinterpret_cast<uint32_t*>(p.out + pc[q].tok * p.o_st + pc[q].head * p.o_sh + (int64_t)pc[q].d0 * 2) =
        E::pack(o0[q] * inv, o1[q] * inv);
  }
}

// All pieces of an item, `pieces` of them (piece_of(i): piece i), by its workgroup of 64 kWaves threads; up to four
// at a time per thread where there are that many.
template <typename T, int D, int NP, typename F>
__device__ __forceinline__ void merge_pieces(const AttnParams& p, int pieces, int stride, int nsplit, F&& piece_of) {
  constexpr int NT = 64 * kWaves;
  for (int at = 0; at < pieces; at += NP * NT) {
    MergePiece pc[NP];
#pragma unroll
    for (int q = 0; q < NP; ++q) {
      const int i = at + q * NT + (int)threadIdx.x;
      pc[q] = i < pieces ? piece_of(i) : MergePiece{-1, 0, 0, 0};
    }
    merge_split_partials<T, D, NP>(p, pc, stride, nsplit);
  }
}
template <typename T, int D, typename F>
__device__ __forceinline__ void merge_item(const AttnParams& p, int pieces, int stride, int nsplit, F&& piece_of) {
  constexpr int NT = 64 * kWaves;
  if (pieces > 2 * NT) merge_pieces<T, D, 4>(p, pieces, stride, nsplit, piece_of);
  else if (pieces > NT) merge_pieces<T, D, 2>(p, pieces, stride, nsplit, piece_of);
  else merge_pieces<T, D, 1>(p, pieces, stride, nsplit, piece_of);
}

}  // namespace lv
