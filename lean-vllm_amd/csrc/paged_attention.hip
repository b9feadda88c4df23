// Paged attention for a continuous-batching step on gfx950: pure decode, chunked prefill, or both in one launch.
//
// Work items (one workgroup of 4 waves each):
//   decode item  = (row, split, kv head or pair of kv heads, query-head group): a row with one query, keys
//                  [split*S, (split+1)*S). Streaming, bandwidth-bound: each wave takes every 4th tile of the
//                  range; a token's head row (D elements) is spread over 16 lanes as 16-byte loads (the two head
//                  rows of a pair, adjacent in the cache, over 32); q.k by v_dot2 with a DPP butterfly inside the
//                  16-lane row; online softmax per tile; p.v on the VALU in fp32. The four waves and, for long
//                  rows, the splits are merged by log-sum-exp (a row's splits by whichever finishes last).
//   prompt item  = (row, q tile, kv head): a row with several queries; the MFMA tile of attn_common.h.
// A step whose rows all have few queries (drafted tokens, or decode of GQA groups other than 1, 2 and 4) runs on the
// items of few_query.hip instead, listed as decode items.
// Launches read a work list built on the device by plan_kernel from the key lengths (and cu_seqlens_q), longest
// work first; its workspace also holds the split rows' partials and their merge counters.
//
// Math: TorchAttention.decode / prefill (lean_vllm/attention/torch_backend.py:62-103,159-181): query head h reads
// key head h / (Hq/Hkv); query j of a row with lq queries and lk keys sees keys 0..lk-lq+j.
#include <algorithm>
#include <mutex>

#include "split_rows.h"

namespace lv {

constexpr int kTile = 16;           // decode tokens per tile; block sizes are multiples of it: a tile is in one block
constexpr int kPlanMaxRows = 4096;  // rows of a step with prompts (the work-list scan lives in LDS)

constexpr int kPromptRing = 2;        // LDS stages of the prompt tiles' ring
constexpr int kOverlapCusPct = 44;    // percent of the CUs that hold a prompt workgroup in a mixed step by default
constexpr int kOverlapCusMaxPct = 75;  // at most this percent when the caller sizes the prompt share
constexpr int kDecodeWgs = 2;         // persistent decode workgroups per CU outside the overlap
constexpr int kOverlapDecodeWgs = 3;  // persistent decode workgroups per CU beside a mixed step's prompt workgroups
                                      // (at most: pair items at D = 128 fit two)
constexpr int kMaxPromptPieces = 8;   // workgroups a prompt item is split into at most
constexpr int kPieceKeys = 1024;      // and keys per piece at least, of the longest row
constexpr int kSplitTarget = 4096;    // decode items (x kv heads x query-head groups) a step with split rows aims for
constexpr int kMaxRowSplits = 128;    // and splits per row on average at most
constexpr int kMinSplit = 256;        // keys per decode item at least
constexpr int kSplitStep = 64;        // and a multiple of this: one tile of every wave
constexpr int kFewRound = 512;        // workgroups that an MI355X holds at once, two per CU (kMaxPieces is its bound)
// Pieces of a step's split prompt items at most: n items are cut into (kFewRound + n / 2) / n >= 2 pieces each, so n
// is at most 2/3 kFewRound, and n pieces of each come to at most kFewRound + n / 2.
constexpr int kMaxPieces = kFewRound * 4 / 3;
// Partials of a step of few queries per row at most (within the static workspace).
constexpr int64_t kFewPartBytes = 14 << 20;
constexpr int kSmallStepRounds = 8;   // a mixed step of at most this many GPU-fulls of workgroups is one launch

// ---------------------------------------------------------------------------------------------------------
// Decode item.
//
// Lane layout (D = 128): 16 lanes hold one token's head row, 16 bytes (8 dims) each. With one kv head per item
// (HP = 1) the wave's 4 lane groups take 4 tokens at a time, 4 times per 16-token tile; with a pair (HP = 2) lanes
// 0-31 take one token's two head rows (512 contiguous bytes of an NHD token row) and lanes 32-63 the next token's.
// Scores stay in raw q.k units; the softmax scale (positive) and log2(e) are folded into the exp2 argument. The
// running max is uniform over the lanes of a head, so rescaling the accumulators is a branch taken only when a
// tile raises some head's max. p.v runs as 2-term dot products over token pairs with p in
// the 16-bit format of the cache (fp32 accumulation), as the MFMA path does with its probability tiles.

// Reduce over the lane groups of a wave that hold different tokens of one head (lanes i, i + LPH, i + 2 LPH, ...;
// LPH lanes hold a token's piece of the item's head rows).
template <int LPH>
__device__ inline float groups_max(float x) {
  static_assert(LPH == 8 || LPH == 16 || LPH == 32, "8, 16 or 32 lanes per token piece");
  if constexpr (LPH == 8) x = vmax(x, dpp_ror8(x));  // lanes i and i ^ 8 of each 16-lane row
  if constexpr (LPH <= 16) x = xor16_max(x);
  return xor32_max(x);
}
template <int LPH>
__device__ inline float groups_sum(float x) {
  static_assert(LPH == 8 || LPH == 16 || LPH == 32, "8, 16 or 32 lanes per token piece");
  if constexpr (LPH == 8) x += dpp_ror8(x);
  if constexpr (LPH <= 16) x = xor16_sum(x);
  return xor32_sum(x);
}

// publish (persistent launches): thread 0 stores publish_value there before the item's merge barrier, and the
// barrier is met even by an item with nothing to do, so the whole workgroup reads the value after the call.
template <typename T, int D, int GS, int HP, int US = 0>
__device__ void decode_item(const AttnParams& p, int row, int split, int per, int kvh, int qg, char* smem,
                            int* publish = nullptr, int publish_value = 0) {
  using E = Elem<T>;
  static_assert(D == 64 || D == 128, "head_dim 64 or 128");
  static_assert(HP == 1 || HP == 2, "one or two kv heads per item");
  constexpr int LPT = D / 8;      // lanes per token head row, 16 bytes each
  constexpr int LPH = LPT * HP;   // lanes per token piece: the item's HP head rows, adjacent in a token's NHD row
  constexpr int TPI = 64 / LPH;   // tokens per wave step
  constexpr int KT = US > 0 ? TPI * US : kTile / HP;  // tokens per wave tile
  constexpr int U = KT / TPI;     // load steps per wave tile
  static_assert(U % 2 == 0, "token pairs");
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int grp = lane / LPH, hs = (lane / LPT) % HP, part = lane % LPT;

  // The row's key length, its first query and the page of the item's first key, in one round trip (the page exists: the
  // plan lists splits that hold keys, and a row of none has a table all the same).
  const int kbeg = split * per;  // per: keys per split
  const int32_t* table = p.tables + (int64_t)row * p.t_stride;
  const int pg0 = (int)p.bs.div(kbeg);
  const int32_t* len = p.lens_k ? p.lens_k + row : p.cu_k + row;
  const int32_t* const where[4] = {len, p.lens_k ? len : len + 1, p.cu_q ? p.cu_q + row : len, table + pg0};
  int got[4];
  sload_n<4>(where, got);
  const int lk = p.lens_k ? got[0] : got[1] - got[0];
  const int tok = p.cu_q ? got[2] : row;
  const bool valid = split == 0 || kbeg < lk;  // else past the row's end: the row has shrunk since the plan
  if (!valid && !publish) return;
  const int kend = valid ? min(lk, kbeg + per) : kbeg;
  const int nsplit = lk > per ? (lk + per - 1) / per : 1;
  const int head0 = (kvh + hs) * p.group + qg * GS;  // this lane's query heads (kvh: the item's first kv head)
  const float c = p.scale_log2;

  u32x4 qv[GS];
#pragma unroll
  for (int g = 0; g < GS; ++g) qv[g] = ld16(p.q + tok * p.q_st + (head0 + g) * p.q_sh + part * 16);

  float m[GS], l[GS], acc[GS][8];
#pragma unroll
  for (int g = 0; g < GS; ++g) {
    m[g] = -INFINITY;
    l[g] = 0.f;
#pragma unroll
    for (int e = 0; e < 8; ++e) acc[g][e] = 0.f;
  }

  // Byte offset of this lane's 16 bytes of step u inside a tile (tile rows are p.c_st apart; fits 32 bits).
  uint32_t loff[U];
#pragma unroll
  for (int u = 0; u < U; ++u) loff[u] = (uint32_t)((u * TPI + grp) * p.c_st + hs * p.c_sh + part * 16);

  // Page numbers come through the scalar cache, once per page this wave enters: a vector load of the table would
  // be waited for in order with the K/V loads already in flight.
  int cached_pg = pg0;
  int64_t cached_base = (int64_t)got[3] * p.c_sb + (int64_t)kvh * p.c_sh;
  auto tile_base = [&](int t0) {
    const int pg = (int)p.bs.div(t0);
    if (pg != cached_pg) {
      cached_pg = pg;
      cached_base = (int64_t)sload(table + pg) * p.c_sb + (int64_t)kvh * p.c_sh;
    }
    return cached_base + (int64_t)(t0 - pg * (int)p.bs.d) * p.c_st;
  };
  auto load_rows = [&](const char* cache, int64_t base, u32x4 (&x)[U]) {
    const char* b = cache + base;
#pragma unroll
    for (int u = 0; u < U; ++u) x[u] = ld16_stream(b + loff[u]);
  };
  // Scores of a tile -> online-softmax update -> probabilities packed in token pairs, per query head.
  auto qk = [&](int t0, const u32x4 (&kv)[U], uint32_t (&pp)[GS][U / 2]) {
    float s[U][GS];
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int g = 0; g < GS; ++g) {
        float d = E::dot2(qv[g][0], kv[u][0], 0.f);
#pragma unroll
        for (int w = 1; w < 4; ++w) d = E::dot2(qv[g][w], kv[u][w], d);
        s[u][g] = group_sum<LPT>(d);
      }
    if (t0 + KT > kend) {  // wave-uniform: the row's last tile; tokens past it get no weight
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const bool in = t0 + u * TPI + grp < kend;
#pragma unroll
        for (int g = 0; g < GS; ++g) s[u][g] = in ? s[u][g] : -INFINITY;
      }
    }
    float mt[GS];
    int grow = 0;
#pragma unroll
    for (int g = 0; g < GS; ++g) {
      float x = s[0][g];
#pragma unroll
      for (int u = 1; u < U; ++u) x = vmax(x, s[u][g]);
      mt[g] = groups_max<LPH>(x);  // finite: every tile holds a token in range
      grow |= mt[g] > m[g];
    }
    // One kv head per item: the max is wave-uniform. Two: each head's lanes hold their own, and a lane whose max did
    // not grow rescales by 1.
    if (HP == 1 ? __builtin_amdgcn_readfirstlane(grow) != 0 : __builtin_amdgcn_ballot_w64(grow) != 0) {
#pragma unroll
      for (int g = 0; g < GS; ++g) {
        const float mn = vmax(m[g], mt[g]);
        const float alpha = fast_exp2((m[g] - mn) * c);
        m[g] = mn;
        l[g] *= alpha;
#pragma unroll
        for (int e = 0; e < 8; ++e) acc[g][e] *= alpha;
      }
    }
#pragma unroll
    for (int g = 0; g < GS; ++g) {
      const float mc = m[g] * c;
#pragma unroll
      for (int u = 0; u < U; u += 2) {
        const float p0 = fast_exp2(fmaf(s[u][g], c, -mc));
        const float p1 = fast_exp2(fmaf(s[u + 1][g], c, -mc));
        l[g] += p0 + p1;
        pp[g][u / 2] = E::pack(p0, p1);
      }
    }
  };
  // acc += p . V over the tile: value rows of token pairs interleaved per dim, 2-term dot products.
  auto pv = [&](int t0, u32x4 (&vv)[U], const uint32_t (&pp)[GS][U / 2]) {
    if (t0 + KT > kend) {  // values past the range may be NaN: zero them (their p is 0)
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const bool in = t0 + u * TPI + grp < kend;
#pragma unroll
        for (int w = 0; w < 4; ++w) vv[u][w] = in ? vv[u][w] : 0u;
      }
    }
#pragma unroll
    for (int u = 0; u < U; u += 2)
#pragma unroll
      for (int w = 0; w < 4; ++w) {
        const uint32_t lo = __builtin_amdgcn_perm(vv[u + 1][w], vv[u][w], 0x05040100u);
        const uint32_t hi = __builtin_amdgcn_perm(vv[u + 1][w], vv[u][w], 0x07060302u);
#pragma unroll
        for (int g = 0; g < GS; ++g) {
          acc[g][2 * w] = E::dot2(pp[g][u / 2], lo, acc[g][2 * w]);
          acc[g][2 * w + 1] = E::dot2(pp[g][u / 2], hi, acc[g][2 * w + 1]);
        }
      }
  };

  constexpr int kStride = KT * kWaves;
  int t0 = kbeg + KT * wave;
  if (t0 < kend) {
    // Staggered: the next tile's keys load during this tile's p.v, its values during its own q.k.
    u32x4 kv[U], vv[U];
    uint32_t pp[GS][U / 2];
    int64_t base = tile_base(t0);
    load_rows(p.k_cache, base, kv);
    load_rows(p.v_cache, base, vv);
    while (true) {
      qk(t0, kv, pp);
      const int t1 = t0 + kStride;
      int64_t next = 0;
      if (t1 < kend) {
        next = tile_base(t1);
        load_rows(p.k_cache, next, kv);
      }
      pv(t0, vv, pp);
      if (t1 >= kend) break;
      load_rows(p.v_cache, next, vv);
      t0 = t1;
    }
  }

  // Sum the token groups of the wave (they share m); m moves to the log2 domain of the merges.
#pragma unroll
  for (int g = 0; g < GS; ++g) {
    l[g] = groups_sum<LPH>(l[g]);
#pragma unroll
    for (int e = 0; e < 8; ++e) acc[g][e] = groups_sum<LPH>(acc[g][e]);
    m[g] *= c;
  }
  // Merge the waves through LDS: wm/wl [kWaves][HG], wacc [kWaves][HG][D] for the item's HG = HP GS query heads
  // (lanes of token group 0 hold their head's sums).
  constexpr int HG = HP * GS;
  float* wm = reinterpret_cast<float*>(smem);
  float* wl = wm + kWaves * HG;
  float* wacc = wl + kWaves * HG;
  if (lane < LPH) {
#pragma unroll
    for (int g = 0; g < GS; ++g) {
      const int hg = wave * HG + hs * GS + g;
#pragma unroll
      for (int e = 0; e < 8; ++e) wacc[hg * D + part * 8 + e] = acc[g][e];
      if (part == 0) {
        wm[hg] = m[g];
        wl[hg] = l[g];
      }
    }
  }
  if (publish && threadIdx.x == 0) *publish = publish_value;
  __syncthreads();
  if (!valid) return;
  // The waves' sums of the item's query head g, dims d0 .. d0 + N - 1, merged; returns the log2-sum-exp2.
  auto merge_waves = [&](int g, int d0, auto& o) {
    constexpr int N = sizeof(o) / sizeof(o[0]);
    float mmax = -INFINITY, den = 0.f;
#pragma unroll
    for (int w = 0; w < kWaves; ++w) mmax = fmaxf(mmax, wm[w * HG + g]);
#pragma unroll
    for (int e = 0; e < N; ++e) o[e] = 0.f;
    mmax = merge_base(mmax);
#pragma unroll
    for (int w = 0; w < kWaves; ++w) {
      const float wt = fast_exp2(wm[w * HG + g] - mmax);
      den += wt * wl[w * HG + g];
#pragma unroll
      for (int e = 0; e < N; ++e) o[e] += wt * wacc[(w * HG + g) * D + d0 + e];
    }
    const float inv = inv_sum(den);
#pragma unroll
    for (int e = 0; e < N; ++e) o[e] *= inv;
    return mmax + fast_log2(den);  // no key seen: -inf
  };
  auto head_of = [&](int g) { return (kvh + g / GS) * p.group + qg * GS + g % GS; };  // g: hs-major
  if (nsplit <= 1) {
    // One thread per 8 output elements.
    for (int c = threadIdx.x; c < HG * D / 8; c += blockDim.x) {
      const int g = c / (D / 8), d0 = (c % (D / 8)) * 8;
      float o[8];
      merge_waves(g, d0, o);
      u32x4 packed;
#pragma unroll
      for (int w = 0; w < 4; ++w) packed[w] = E::pack(o[2 * w], o[2 * w + 1]);
      st16(p.out + tok * p.o_st + head_of(g) * p.o_sh + (int64_t)d0 * 2, packed);
    }
    return;
  }
  // One thread per two elements of the partial: a wave writes 512 consecutive bytes.
  const int slot0 = p.part_base[row];  // the row's partial slots
  for (int c = threadIdx.x; c < HG * D / 2; c += blockDim.x) {
    const int g = c / (D / 2), d0 = (c % (D / 2)) * 2;
    float o[2];
    const float lse = merge_waves(g, d0, o);
    const int64_t slot = (int64_t)(slot0 + split) * p.hq + head_of(g);
    coherent_store2(p.part_o + slot * D + d0, o[0], o[1]);
    if (d0 == 0) coherent_store(p.part_lse + slot, lse);
  }
  // The split that counts in last merges the item's heads. Each wave waits until its partial stores are complete
  // (written through to memory) before the barrier that precedes the count, so every split's partials are in memory
  // before its count; the merger reads them past its L2 after its own count has returned.
  __shared__ int s_last;
  __builtin_amdgcn_s_waitcnt(0);
  __syncthreads();
  int32_t* count = p.merge_count + (row * (p.hkv / HP) + kvh / HP) * p.qgroups + qg;
  if (threadIdx.x == 0)
    s_last = __hip_atomic_fetch_add(count, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == nsplit - 1;
  __syncthreads();
  if (s_last) {
    merge_item<T, D>(p, HG * D / 2, 1, nsplit, [&](int c) {
      return MergePiece{slot0, tok, head_of(c / (D / 2)), (c % (D / 2)) * 2};
    });
    // Back to zero for the next layer on this plan.
    if (threadIdx.x == 0) __hip_atomic_store(count, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
}

// ---------------------------------------------------------------------------------------------------------
// Kernels.

template <int D, int GS, int HP>
struct SmemBytes {
  static constexpr int kDecode = kWaves * HP * GS * (D + 2) * 4;
};

// Work-list kernels. blockIdx.x walks the device work list with the query-head groups innermost, so workgroups
// are dispatched in list order (longest first). The step's prompt items and its decode items are two lists. Decode
// items run in decode_list_kernel at the decode item's register budget; prompt items in prompt_list_kernel, whose MFMA
// tile needs more registers and LDS.

template <typename T, int D, int GS, int HP, int US = 0>
__global__ __launch_bounds__(256) void decode_list_kernel(AttnParams p) {
  __shared__ __attribute__((aligned(16))) char smem[SmemBytes<D, GS, HP>::kDecode];
  const int ny = p.hkv / HP * p.qgroups;
  const int bx = blockIdx.x / ny, by = blockIdx.x - bx * ny;
  const int kh = by / p.qgroups, qg = by - kh * p.qgroups;
  const DecodeWork w = decode_work(p, bx);
  if (bx >= w.count) return;
  decode_item<T, D, GS, HP, US>(p, w.row, w.split, w.per, kh * HP, qg, smem);
}

// Decode items of the work list on a persistent grid beside a mixed step's prompt workgroups: each workgroup takes
// items by ticket (an atomic counter the plan kernel zeroes), in list order, so the longest still go first. A
// fixed number of workgroups per CU lets the prompt workgroups stay resident beside them (outside the overlap,
// one workgroup per item measured as fast or faster). The next ticket is drawn at the start of an item and
// published at its merge barrier; the merge alternates between two LDS buffers, so one barrier per item suffices.
// The last workgroup to finish puts the ticket and the exit count back to zero, so the next layer of the step can
// run on the same plan without a plan launch: every workgroup's ticket draws have returned (their values were
// read) before it counts itself out, so no draw can follow the reset.
template <typename T, int D, int GS, int HP, int US = 0>
__device__ __forceinline__ void decode_persistent(const AttnParams& p) {
  __shared__ __attribute__((aligned(16))) char smem[2][SmemBytes<D, GS, HP>::kDecode];
  __shared__ int s_ticket[2];
  const int ny = p.hkv / HP * p.qgroups;
  const int total = p.n_items[kPlanDecodes] * ny;
  if (threadIdx.x == 0) s_ticket[0] = atomicAdd(p.ticket, 1);
  __syncthreads();
  int f = __builtin_amdgcn_readfirstlane(s_ticket[0]);
  for (int k = 0; f < total; ++k) {
    int next = 0;
    if (threadIdx.x == 0) next = atomicAdd(p.ticket, 1);
    const int bx = f / ny, by = f - bx * ny;
    const int kh = by / p.qgroups, qg = by - kh * p.qgroups;
    const DecodeWork w = decode_work(p, bx);
    decode_item<T, D, GS, HP, US>(p, w.row, w.split, w.per, kh * HP, qg, smem[k & 1], &s_ticket[(k + 1) & 1], next);
    f = __builtin_amdgcn_readfirstlane(s_ticket[(k + 1) & 1]);
  }
  if (threadIdx.x == 0 && atomicAdd(p.ticket + 1, 1) == (int)gridDim.x - 1) {
    atomicExch(p.ticket, 0);
    atomicExch(p.ticket + 1, 0);
  }
}

// Load steps of a wave tile: pair items at D = 128 hold 16-token wave tiles (8 load steps, twice the bytes in
// flight per wave of the 8-token tile, about 210 registers); other shapes keep the kTile / HP default.
template <int D, int HP>
constexpr int kWideSteps = HP == 2 && D == 128 ? 8 : 0;

// Beside a mixed step's prompt workgroups (one per CU; a prompt wave takes 193 registers, allocated as 200) the
// decode workgroups share each SIMD's 512 registers per lane: one pair-item workgroup at D = 128 (210) beside a
// prompt wave and two on the other CUs; the smaller items of other shapes (131 or fewer) two beside a prompt wave
// and three on the others. The grid asks for up to three per CU, as many as fit alone.
template <typename T, int D, int GS, int HP>
__global__ __launch_bounds__(256, 2) void decode_beside_kernel(AttnParams p) {
  decode_persistent<T, D, GS, HP, kWideSteps<D, HP>>(p);
}

// TP: pages per 64-key prompt tile. TP > 0 (pages of a multiple of 64 keys, or of 32 or 16): the tiles stream
// through an LDS ring of kPromptRing stages; TP = 0 (other page sizes): through registers.
template <int TP>
constexpr int kRingOf = TP > 0 ? kPromptRing : 0;

template <typename T, int D, int TP>
__global__ __launch_bounds__(256, 2) void prompt_list_kernel(AttnParams p) {
  constexpr int RING = kRingOf<TP>;
  __shared__ __attribute__((aligned(16))) char smem[(RING > 0 ? RING : 1) * PromptSmem<D, D, (TP > 1)>::kBytes];
  const int bx = blockIdx.x / p.hkv, kvh = blockIdx.x - bx * p.hkv;
  if (bx >= p.n_items[kPlanPrompts]) return;
  const int2 it = p.prompts[bx];
  prefill_item<T, D, D, true, false, RING, 4, false, (TP > 0 ? TP : 1)>(p, it.x, -1 - it.y, kvh, smem);
}

// A few prompt items with long key ranges (a chunk late in a long prompt), each split over its keys into p.pieces
// workgroups, and the merge of their partials: one thread per four dims of a query row. MFMA-bound, as the unsplit
// items, but 128 of those leave half the CUs without one and every SIMD of the others with one wave. 32/8 heads,
// d128, a chunk on a 24,576-token prefix: 512 tokens 505 -> 222 us (412 -> 940 TFLOP/s), 32 tokens 494 -> 84, 1024
// tokens 517 -> 417; on 16-token pages 618 -> 235; 256 tokens on 4096 97 -> 47. (Pieces of at least kPieceKeys keys:
// 512 tokens on 2048 62 -> 53.) The number of pieces is the step's, by its longest row; a piece is that part of its
// own item's tiles, so a short row's or an early tile's pieces are shorter, or empty.
template <typename T, int D, int TP>
__global__ __launch_bounds__(256, 2) void prompt_split_kernel(AttnParams p) {
  constexpr int RING = kRingOf<TP>;
  __shared__ __attribute__((aligned(16))) char smem[RING * PromptSmem<D, D, (TP > 1)>::kBytes];
  const int f = blockIdx.x / p.hkv, kvh = blockIdx.x - f * p.hkv;
  const int bx = f / p.pieces, piece = f - bx * p.pieces;
  if (bx >= p.n_items[kPlanPrompts]) return;
  const int2 it = p.prompts[bx];
  prefill_item<T, D, D, true, false, RING, 4, false, TP, true>(p, it.x, -1 - it.y, kvh, smem, piece,
                                                               (bx * p.hkv + kvh) * p.pieces + piece);
}

template <typename T, int D>
__global__ __launch_bounds__(256) void prompt_merge_kernel(AttnParams p) {
  using E = Elem<T>;
  constexpr int LPR = D / 4, RPB = 256 / LPR;  // threads per row, rows per workgroup
  const int item = blockIdx.x / (kPrefillRows / RPB);
  const int r = (blockIdx.x - item * (kPrefillRows / RPB)) * RPB + threadIdx.x / LPR, d0 = threadIdx.x % LPR * 4;
  const int bx = item / p.hkv, kvh = item - bx * p.hkv;
  if (bx >= p.n_items[kPlanPrompts]) return;
  const int2 it = p.prompts[bx];
  const int qp = kPrefillRows / p.group;
  const int q0 = p.cu_q[it.x], lq = p.cu_q[it.x + 1] - q0;
  const int pos = (-1 - it.y) * qp + r / p.group, head = kvh * p.group + r % p.group;
  if (r >= qp * p.group || pos >= lq) return;
  float ls[kMaxPromptPieces];
  f32x4 x[kMaxPromptPieces];
  float m = -INFINITY;
#pragma unroll
  for (int i = 0; i < kMaxPromptPieces; ++i) {
    ls[i] = -INFINITY;
    x[i] = f32x4{0, 0, 0, 0};
    if (i < p.pieces) {
      const int64_t at = ((int64_t)item * p.pieces + i) * kPrefillRows + r;
      ls[i] = p.piece_lse[at];
      x[i] = *reinterpret_cast<const f32x4*>(p.piece_o + at * D + d0);
    }
  }
#pragma unroll
  for (int i = 0; i < kMaxPromptPieces; ++i) m = fmaxf(m, ls[i]);
  m = merge_base(m);
  float den = 0.f;
  f32x4 o = {0, 0, 0, 0};
#pragma unroll
  for (int i = 0; i < kMaxPromptPieces; ++i) {
    const float w = fast_exp2(ls[i] - m);
    den += w;
    o += w * x[i];
  }
  o *= inv_sum(den);
  *reinterpret_cast<u32x2*>(p.out + (int64_t)(q0 + pos) * p.o_st + (int64_t)head * p.o_sh + d0 * 2) =
      u32x2{E::pack(o[0], o[1]), E::pack(o[2], o[3])};
}

// Prompt items of a mixed step, run at the same time as its decode items: one workgroup per CU, each walking the
// prompt items blockIdx.x, + gridDim.x, ... in list order. Its LDS request (padded at launch, so the compiler still
// budgets registers for 2 waves per SIMD) leaves room for no second one, and the decode workgroups take the CU's
// remaining registers: the MFMA work of the prompt tiles hides under the decode rows' memory streaming.
constexpr int kOverlapLds = 84 * 1024;
template <typename T, int D, int TP>
__global__ __launch_bounds__(256, 2) void prompt_overlap_kernel(AttnParams p) {
  constexpr int RING = kRingOf<TP>;
  __shared__ __attribute__((aligned(16))) char smem[(RING > 0 ? RING : 1) * PromptSmem<D, D, (TP > 1)>::kBytes];
  // The prompt tiles are the step's critical path beside the decode waves, which need few issue slots: the prompt
  // waves win the SIMD's issue arbitration (1% on the Qwen3-8B mixed step; favouring the decode waves costs 15%).
  __builtin_amdgcn_s_setprio(1);
  const int n = p.n_items[kPlanPrompts] * p.hkv;
  for (int f = blockIdx.x; f < n; f += gridDim.x) {
    const int bx = f / p.hkv, kvh = f - bx * p.hkv;
    const int2 it = p.prompts[bx];
    prefill_item<T, D, D, true, true, RING, 4, false, (TP > 0 ? TP : 1)>(p, it.x, -1 - it.y, kvh, smem);
    __syncthreads();  // the next item restages the LDS tiles
  }
}

// A small mixed step in one launch: workgroups [0, prompt_wgs) take the prompt items (one per item and kv head, the
// longest first), the rest the decode items in list order. Dispatched in that order, the prompt workgroups start
// first and the decode workgroups stream through the slots they leave, as in the overlapped schedule but without a
// second stream, its events and one launch: for steps of a few hundred rows, whose launch sequence is a large share
// of their time.
template <typename T, int D, int GS, int TP, int HP>
__global__ __launch_bounds__(256, 2) void mixed_small_kernel(AttnParams p, int32_t prompt_wgs) {
  constexpr int RING = kRingOf<TP>;
  static_assert(SmemBytes<D, GS, HP>::kDecode <= (RING > 0 ? RING : 1) * PromptSmem<D, D, (TP > 1)>::kBytes,
                "LDS for both");
  __shared__ __attribute__((aligned(16))) char smem[(RING > 0 ? RING : 1) * PromptSmem<D, D, (TP > 1)>::kBytes];
  const int b = blockIdx.x;
  if (b < prompt_wgs) {
    const int bx = b / p.hkv, kvh = b - bx * p.hkv;
    if (bx >= p.n_items[kPlanPrompts]) return;
    const int2 it = p.prompts[bx];
    prefill_item<T, D, D, true, false, RING, 4, false, (TP > 0 ? TP : 1)>(p, it.x, -1 - it.y, kvh, smem);
  } else {
    const int ny = p.hkv / HP * p.qgroups;
    const int f = b - prompt_wgs, bx = f / ny, by = f - bx * ny;
    const int kh = by / p.qgroups, qg = by - kh * p.qgroups;
    const DecodeWork w = decode_work(p, bx);
    if (bx >= w.count) return;
    decode_item<T, D, GS, HP>(p, w.row, w.split, w.per, kh * HP, qg, smem);
  }
}

// Decode of more rows than the planner holds: blockIdx.x is the row, blockIdx.y the kv head (or pair) and query-head
// group. Such a step's rows are not split: a split row's partials need the slots and merge counters of a work list.
template <typename T, int D, int GS, int HP>
__global__ __launch_bounds__(256) void decode_grid_kernel(AttnParams p) {
  __shared__ __attribute__((aligned(16))) char smem[SmemBytes<D, GS, HP>::kDecode];
  const int kh = blockIdx.y / p.qgroups, qg = blockIdx.y % p.qgroups;
  decode_item<T, D, GS, HP>(p, blockIdx.x, 0, INT32_MAX, kh * HP, qg, smem);
}

constexpr int kLenBuckets = 64;
// Bucket of a split that is `short_of` keys short of a whole one: longer splits get smaller buckets (dispatched first).
__device__ inline int len_bucket(int short_of, float per_key) {
  return min(max((int)((float)short_of * per_key), 0), kLenBuckets - 1);
}

// Work lists of a step, longest work first: the prompt items (row, -1 - tile); and the decode items, every full split
// (row, s), then each row's last split (row, n - 1) by decreasing key count (counting sort over length buckets).
// In-order dispatch of that list approximates longest-processing-time scheduling, so the launch ends with short
// items instead of a tail of full ones. A prompt row's tiles go last tile first (most keys) when the prompt items
// have the GPU to themselves (last_first: a step of prompts, or the serial schedule): the Qwen3-8B chunks 5-6%
// faster than first tile first. Beside the decode rows (the overlapped schedule) the order made no measurable
// difference, and the first tile goes first there as before. The split rows' merge counters start at zero.
//
// Keys per decode split: the decode rows' own keys over `pieces`, at least kMinSplit (or two) and a multiple of
// kSplitStep, so that a step is cut into about the same number of items whatever its lengths (at most pieces + rows).
// The caller's bound on key lengths only sizes the buffers: a captured graph's bound is the longest context it may
// ever serve, and a batch of a few rows far apart in length has most of its keys in one of them. pieces 0: rows are
// not split, and one split holds the longest row. The partials of split rows lie in consecutive slots from
// part_base[row]. few: rows of several queries are streamed as decode items too, one slot per query and split.
//
// few: a row's merge is one workgroup's work, and takes as long as its splits where they hold `least` keys: n splits
// of lk keys take lk / n keys' stream (12 KB a microsecond) and lq G D n / 512 loads a thread (19 a microsecond),
// equal at lk / n = sqrt(0.3 lk lq G). One row of 64,000 keys, 128 splits and with this bound: 8/2 heads, d128, 16
// queries 160 -> 114 us (56 splits); 16/1 heads, 4 queries, two rows 157 -> 113; 40/1 heads, one query 114 -> 91. It
// is below kMinSplit, and changes nothing, while lk lq G < 218,000 (4 queries of group 4 on 13,000 keys).
//
// A split that needs more slots than there are grows until they fit: a long row of more queries than the others (to
// fewer_pieces first), more queries or lengths than the caller said (by the slots' ratio, a sixteenth at least).
__host__ __device__ inline int least_split(int lk, int query_rows) {
  return (int)sqrtf(0.3f * (float)(lk > 0 ? lk : 0) * (float)query_rows);
}
// VALU items (few: kv_heads 0): two kMinSplit where that still gives every CU an item of its own kv head. Over 80
// decode steps of random shapes 3% faster than kMinSplit everywhere (one to nine long rows of one or two kv heads
// 15-35%), over 120 mixed steps 1%; one row of 8K keys of 8 kv heads, below the line, 34.6 us against 40.1 with it.
__host__ __device__ inline int split_keys(float keys, int longest, int least, int pieces, int kv_heads) {
  if (keys * (float)kv_heads >= 2.f * kMinSplit * (kFewRound / 2) && least < 2 * kMinSplit) least = 2 * kMinSplit;
  int64_t want = longest;
  if (pieces > 0) {
    int64_t share = (int64_t)(keys * 1.00001f / (float)pieces) + 1;
    share = share > least ? share : least;
    want = want < share ? want : share;
  }
  want = (want + kSplitStep - 1) / kSplitStep * kSplitStep;
  return want < INT32_MAX ? (int)want : INT32_MAX;
}

struct PlanOut {
  int2* prompts;    // the prompt items
  int2* items;      // the decode items
  int32_t* counts;  // kPlan* entries
  int32_t* part_base;
  int32_t* merge_count;
};

// ROWS: rows a thread at most. The kernel is its barriers, its round trips to memory and its code, which a step's one
// plan meets cold: the rows' loads are issued together, once, and all that is known of a row stays in registers. 3 /
// 256 / 1024 / 4096 rows of a decode step 6.0 / 6.4 / 7.4 / 12.8 us with later rows loaded again in each pass and
// 64-bit bucket divisions, 5.4 / 5.9 / 6.6 / 10.4 so (with splits of a size fixed on the host 5.6 / 4.5 / 5.0 / 8.9).
// PROMPTS: the caller says that no row is a decode row (LV_ATTN_PROMPTS_ONLY), so no split is sized and no decode item
// listed: a step of one or two short prompts, whose layers take 9 us each, 2.5 us instead of 4.9 (1100
// rows 4.4 instead of 7.8).
template <int ROWS, bool PROMPTS>
__global__ __launch_bounds__(kScanThreads) void plan_kernel(const int32_t* __restrict__ cu_q,
                                                            const int32_t* __restrict__ lens_k,
                                                            const int32_t* __restrict__ cu_k, int32_t rows,
                                                            int32_t pieces, int32_t max_slots, int32_t qp,
                                                            int32_t max_prompts, int32_t max_items,
                                                            int32_t last_first, int32_t few, int32_t fewer_pieces,
                                                            int32_t group, int32_t kv_heads, int32_t n_merge,
                                                            PlanOut out) {
  __shared__ int pre[ROWS * kScanThreads + 1];
  __shared__ int full[ROWS * kScanThreads + 1];
  __shared__ int slots[ROWS * kScanThreads + 1];
  __shared__ int bucket[kLenBuckets + 1];
  __shared__ int wave_tot[3][kScanThreads / 64];
  __shared__ float wave_keys[kScanThreads / 64];
  __shared__ int wave_max_of[kScanThreads / 64];
  __shared__ int wave_least[kScanThreads / 64];
  const int tid = threadIdx.x;
  int lq[ROWS], lk[ROWS], n[ROWS];  // of rows tid, tid + kScanThreads, ...: queries, keys, decode items
#pragma unroll
  for (int i = 0; i < ROWS; ++i) {
    const int r = tid + i * kScanThreads;
    lq[i] = lk[i] = n[i] = 0;
    if (r < rows) {
      lq[i] = cu_q ? cu_q[r + 1] - cu_q[r] : 1;
      lk[i] = lens_k ? lens_k[r] : cu_k[r + 1] - cu_k[r];
    }
  }
  // Prompt items and full splits, one thread each (a few long rows hold hundreds: a thread per row would write them
  // one by one, 9 us for seven prompts' 260 items, 5 so).
  auto row_of = [&](const int* before, int i) {  // the last row with at most i items before its own
    int lo = 0, hi = rows - 1;
    while (lo < hi) {
      const int mid = (lo + hi + 1) >> 1;
      if (before[mid] <= i) lo = mid; else hi = mid - 1;
    }
    return lo;
  };
  auto list_prompts = [&] {
    for (int i = tid; i < min(pre[rows], max_prompts); i += kScanThreads) {
      const int r = row_of(pre, i);
      out.prompts[i] = make_int2(r, -1 - (last_first ? pre[r + 1] - 1 - i : i - pre[r]));
    }
  };
  if constexpr (PROMPTS) {
    __shared__ int prompt_tot[1][kScanThreads / 64];
    for (int i = tid; i < n_merge; i += kScanThreads) out.merge_count[i] = 0;
#pragma unroll
    for (int i = 0; i < ROWS; ++i)
      if (tid + i * kScanThreads < rows) pre[tid + i * kScanThreads] = lq[i] > 1 ? (lq[i] + qp - 1) / qp : 0;
    __syncthreads();
    block_scan(pre, rows, prompt_tot);
    list_prompts();
    if (tid == 0) {
      out.counts[kPlanDecodes] = 0;
      out.counts[kPlanPrompts] = min(pre[rows], max_prompts);
      out.counts[kPlanTicket] = 0;
      out.counts[kPlanDone] = 0;
      out.counts[kPlanSplit] = kSplitStep;
    }
    return;
  }
  auto streamed = [&](int i) { return few ? lq[i] > 0 : lq[i] == 1; };  // a row of decode items
  for (int b = tid; b <= kLenBuckets; b += kScanThreads) bucket[b] = 0;
  for (int i = tid; i < n_merge; i += kScanThreads) out.merge_count[i] = 0;
  // The decode rows' keys in all (fp32 is enough: the count is rounded up past its error) and at most.
  float keys = 0.f;
  int longest = 1, least = kMinSplit;  // least: keys per split at least
#pragma unroll
  for (int i = 0; i < ROWS; ++i)
    if (streamed(i)) {
      keys += (float)max(lk[i], 0);
      longest = max(longest, lk[i]);
      if (few) least = max(least, least_split(lk[i], lq[i] * group));
    }
  keys = wave_sum(keys);
  longest = wave_max(longest);
  if (few) least = wave_max(least);
  if ((tid & 63) == 0) {
    wave_keys[tid >> 6] = keys;
    wave_max_of[tid >> 6] = longest;
    wave_least[tid >> 6] = least;
  }
  __syncthreads();
  keys = 0.f;
#pragma unroll
  for (int w = 0; w < kScanThreads / 64; ++w) {
    keys += wave_keys[w];
    longest = max(longest, wave_max_of[w]);
    least = max(least, wave_least[w]);
  }
  int split = split_keys(keys, longest, least, pieces, few ? 0 : kv_heads);
  for (;;) {  // every thread leaves together: slots[rows] is the same for all, and split reaches the longest row
#pragma unroll
    for (int i = 0; i < ROWS; ++i) {
      const int r = tid + i * kScanThreads;
      if (r >= rows) break;
      n[i] = streamed(i) ? (lk[i] > split ? (lk[i] + split - 1) / split : 1) : 0;
      pre[r] = lq[i] > 1 && !few ? (lq[i] + qp - 1) / qp : 0;
      full[r] = max(n[i] - 1, 0);
      slots[r] = n[i] > 1 ? n[i] * lq[i] : 0;
    }
    __syncthreads();
    int* const sums[3] = {pre, full, slots};  // one pass over all
    block_scan<3>(sums, rows, wave_tot);
    if (slots[rows] <= max_slots || split >= longest) break;
    int64_t grown = max((int64_t)split * slots[rows] / max(max_slots, 1), (int64_t)split + split / 16);
    if (fewer_pieces > 0) {
      grown = max((int64_t)split, (int64_t)(keys / (float)fewer_pieces));
      fewer_pieces = 0;  // the next time by the slots' ratio
    }
    grown = (grown + kSplitStep) / kSplitStep * kSplitStep;
    split = grown <= (1 << 30) ? (int)grown : INT32_MAX;
    __syncthreads();  // every thread has read slots[rows]
  }
  const float per_key = (float)kLenBuckets / (float)split;
  int at[ROWS];  // the bucket of a row's last split
#pragma unroll
  for (int i = 0; i < ROWS; ++i)
    if (n[i] > 0) {
      const int r = tid + i * kScanThreads;
      at[i] = len_bucket(split - (lk[i] - (n[i] - 1) * split), per_key);
      atomicAdd(&bucket[at[i]], 1);
      if (n[i] > 1) out.part_base[r] = slots[r];
    }
  __syncthreads();
  if (tid < kLenBuckets) {  // wave 0: the bucket counts to offsets (one bucket per lane)
    static_assert(kLenBuckets == 64, "one wave scans the buckets");
    const int v = bucket[tid];
    const int x = wave_incl_scan(v);
    bucket[tid] = x - v;
    if (tid == kLenBuckets - 1) bucket[kLenBuckets] = x;
  }
  __syncthreads();
  const int npre = pre[rows], nfull = full[rows], npart = bucket[kLenBuckets];
  list_prompts();
  for (int i = tid; i < min(nfull, max_items); i += kScanThreads) {
    const int r = row_of(full, i);
    out.items[i] = make_int2(r, i - full[r]);
  }
#pragma unroll
  for (int i = 0; i < ROWS; ++i)
    if (n[i] > 0) {
      const int pos = nfull + atomicAdd(&bucket[at[i]], 1);
      if (pos < max_items) out.items[pos] = make_int2(tid + i * kScanThreads, n[i] - 1);
    }
  if (tid == 0) {
    out.counts[kPlanDecodes] = min(nfull + npart, max_items);
    out.counts[kPlanPrompts] = min(npre, max_prompts);
    out.counts[kPlanTicket] = 0;
    out.counts[kPlanDone] = 0;
    out.counts[kPlanSplit] = split;
  }
}

// ---------------------------------------------------------------------------------------------------------
// Host side.

struct Shape {
  int32_t max_items, max_prompt_items, max_decode_items, gs;
  int32_t pieces;      // the plan cuts the decode rows' keys into this many (0: rows are not split)
  int32_t fewer_pieces;  // few queries: and into this many where the partials of those do not fit
  int32_t route_items; // decode items by which a mixed step's route is chosen
  int32_t max_splits;  // the most items one row may be split into
  int32_t slots;       // split rows' partial slots
  int32_t prompt_pieces;  // workgroups per prompt item outside the overlap
  int64_t merges;      // split rows' merge counters (rows x kv heads x query-head groups)
  size_t items_off, count_off, base_off, lse_off, o_off, merge_off, bytes;
  size_t piece_bytes;  // beside them, split prompt items' partials: outputs, then log-sum-exps
};

static int pick_gs(int group) {
  if (group % 4 == 0) return 4;
  if (group % 2 == 0) return 2;
  return 1;
}

// Queries per row that a step of few queries may have (0: the GQA group is too wide). Past 32 query rows per kv head
// an item at D = 128 streams its keys into LDS twice; its steps are few-query steps while rows x kv heads are at most
// a quarter of the GPU's workgroups. At D = 64 it stays with one copy: two layers, 16 queries a row of 32/8 heads, 48
// rows 231 against 308 us on the prompt items, 8 rows 83 against 256 (unsplit).
//
// What the line weighs, D = 128, 16 queries a row of 32/8 heads, us a layer, few-query items / split prompt items,
// contexts of 2K, 8K, 32K: 1 row 29 / 55, 53 / 42, 94 / 114; 4 rows 33 / 55, 71 / 45, 223 / 122; 8 rows 46 / 56, 121
// / 76, 423 / 243; 16 rows 70 / 57, 221 / 123, 830 / 426. One row of 64,000 keys among short ones (8/2 heads): 114 /
// 212. Few-query items win on short contexts and where the long rows are one or two; a step of equal rows past 4K
// would be faster on the prompt items, but the host knows the bound on the contexts, not the contexts.
//
// (A decode row of a group that wide is a few-query row all the same: the VALU items would read its keys once per
// four heads.)
static int few_queries(int64_t rows, int32_t hkv, int32_t d, int group) {
  const int most = d == 64 || group > 32 || rows * hkv <= kFewRound / 4 ? kFewMaxRows : kFewMaxRows / 2;
  return std::min(kFewMaxQueries, most / group);
}

// max_q: queries per row at most, of a step of few queries.
static Shape plan_shape(int32_t rows, int32_t tokens, int32_t hq, int32_t hkv, int32_t d, int32_t max_k,
                        bool listed, bool few, int32_t max_q, bool split_prompts) {
  Shape s{};
  const int group = hq / hkv;
  s.gs = pick_gs(group);
  const int64_t per_split = few ? hkv : (int64_t)hkv * (group / s.gs);  // decode items per row and split
  const int64_t keys = max_k > 0 ? max_k : 1;
  // Rows split only in a listed step (whose workspace holds the partial slots and merge counters). The number of pieces
  // weighs the list's balance against the merge of a row, its round trips past the L2 after its last split.
  //
  // Where unsplit items fill the GPU (VALU: more than half the items aimed for; few queries: more than one round),
  // the longest-first list balances them as they are, and only a row of more than two workgroups' share of all keys
  // is split.
  //
  // VALU decode items: 4096 one-head items for many rows, fewer for a few long ones. 32/8 heads, d128, contexts
  // U[32K, 128K], 1024 / 2048 / 3072 / 4096 items (before, 4096 of sizes set by the longest row): 1 row 93 / 113 /
  // 125 / 132 us (166), 2 rows 174 / 181 / 192 / 190 (219), 3 rows 252 / 250 / 256 / 261 (272), 8 rows 594 / 557 /
  // 567 / 569 (585), 24 rows 1494 / 1399 / 1372 / 1384 (1452); 48 rows U[4K, 64K] 1431 / 1283 / 1237 / 1241 (1309):
  // the lines at 2 and 16 rows lie between measured counts, and 3072 items for more rows would be within 1%.
  //
  // Steps of few queries (few_query.hip, two workgroups per CU whatever the group): a full piece is one workgroup's
  // share of all keys, so the full pieces run in one round and the rows' remainders pack beside them; up to kFewRound
  // / 8 rows' remainders are counted in, so that all run at once. More pieces cost more than they balance, their
  // partials being several query rows each. 32/8 heads, d128, 4 queries a row, contexts U[512, 8192], two layers,
  // pieces of half a share / two thirds / one: 12 rows 121 / 117 / 110 us, 24 rows 193 / 192 / 182, 48 rows 346 / 353
  // / 336; 4 rows with their remainders beside the round 66.7, in it 57.9; 100 rows split by shares 631, unsplit 624.
  const int64_t units = rows * per_split;
  const int64_t row_queries = few ? ((int64_t)tokens + rows - 1) / rows : 1;  // a row's on average
  const int64_t slot_bytes = (int64_t)hq * (d + 1) * (int64_t)sizeof(float);
  const int64_t share = std::max<int64_t>(1, kFewRound / per_split);  // splits of one round of workgroups
  int64_t pieces = std::max<int64_t>(1, share / 2);
  const int64_t remainders = 8 * rows <= share ? rows : 0;
  const bool light = few && row_queries * group <= 4;
  if (few && !light) {
    if (units <= kFewRound) pieces = std::min(share - remainders, (int64_t)kMaxRowSplits * rows);
    const int64_t max_slots = kFewPartBytes / slot_bytes;
    if ((pieces + std::min<int64_t>(rows, pieces)) * row_queries > max_slots) pieces = max_slots / row_queries / 2;
  } else {  // up to four query rows an item weighs no more than a VALU item and splits as one
    const int64_t items = rows <= 2 ? kSplitTarget / 4 : rows <= 16 ? kSplitTarget / 2 : kSplitTarget;
    const int64_t splits = std::min<int64_t>((items + per_split - 1) / per_split, (int64_t)kMaxRowSplits * rows);
    if (2 * (int64_t)rows <= splits) pieces = splits - rows;
  }
  int64_t route_split = kMinSplit;
  while (route_split < keys && units * ((keys + route_split - 1) / route_split) > kSplitTarget) route_split *= 2;
  if (!listed || keys <= kMinSplit) pieces = 0;
  s.pieces = (int32_t)pieces;
  const int64_t most = pieces > 0 ? (keys + kMinSplit - 1) / kMinSplit : 1;  // splits of one row
  const int64_t splits = std::min(rows * most, pieces + rows);  // of all rows
  s.max_splits = (int32_t)std::min(most, splits);
  const int qp = kPrefillRows / (group > 0 ? group : 1);
  // In 64 bits, saturated: a count past INT32_MAX is far past what one launch holds (check_grids refuses it).
  auto sat = [](int64_t x) { return (int32_t)std::min<int64_t>(x, INT32_MAX); };
  s.max_prompt_items = listed && !few ? sat(((int64_t)tokens + qp - 1) / qp + rows) : 0;
  s.max_decode_items = listed ? sat(splits) : 0;
  s.max_items = sat((int64_t)s.max_prompt_items + s.max_decode_items);
  s.route_items = sat(rows * ((keys + route_split - 1) / route_split));
  // Rows of more than one split hold more keys than a split, so there are at most `pieces` of them, and their splits
  // have slots for row_queries each. In a step of few queries most keys may be in a row of more than that: slots for
  // max_q each, where they fit in kFewPartBytes with the counters, at half the pieces (one workgroup per CU streams
  // about as fast and leaves half the partials to merge), or one round of the light ones. One long row among short
  // ones, us, with the split doubled until slots for the average row held it (before), and so: 32/8 heads, d128, 8
  // queries on 64,000 keys among 15 of one on 300 108.9 -> 74.8; 16 on 60,000 beside 9 on 5000 and two short 214 ->
  // 136.5; 4 on 64,000 beside 7 of one on 1000 59.9 -> 60.6; 8/8 heads, 8 queries on 64,000 beside 3 of one on 4000
  // 66.2 -> 65.8.
  const int64_t merges = s.max_splits > 1 ? (int64_t)rows * per_split : 0;
  if (s.max_splits > 1) {
    const int64_t split_rows = std::min<int64_t>(rows, pieces);
    int64_t slots = std::min(splits, pieces + split_rows) * row_queries;
    if (few) {
      s.fewer_pieces = (int32_t)std::max<int64_t>(1, light ? share - remainders : pieces / 2);
      slots = std::max(slots, std::min(std::min(splits, s.fewer_pieces + split_rows) * std::min(max_q, tokens),
                                       (kFewPartBytes - merges * (int64_t)sizeof(int32_t)) / slot_bytes));
    }
    s.slots = sat(slots);
  }
  size_t off = 0;
  s.items_off = off;
  off += (size_t)s.max_items * sizeof(int2);
  off = (off + 255) / 256 * 256;
  s.count_off = off;
  off += 256;
  s.base_off = off;
  off += s.slots > 0 ? (size_t)rows * sizeof(int32_t) : 0;
  off = (off + 255) / 256 * 256;
  const size_t parts = (size_t)s.slots * hq;
  s.lse_off = off;
  off += parts * sizeof(float);
  off = (off + 255) / 256 * 256;
  s.o_off = off;
  off += parts * d * sizeof(float);
  off = (off + 255) / 256 * 256;
  s.merges = merges;
  s.merge_off = off;
  off += (size_t)s.merges * sizeof(int32_t);
  // Prompt items that fill at most two thirds of the GPU's workgroups are split over their keys, into as many pieces
  // as come nearest to one round. Their bound counts a tile per decode row too, so a serial step's chunk beside many
  // decode rows stays whole (512 tokens beside 32 rows of 32/8 heads: 128 items, 400 counted).
  const int64_t prompts = (int64_t)s.max_prompt_items * hkv;
  s.prompt_pieces = 1;
  if (split_prompts && prompts > 0)
    s.prompt_pieces = (int32_t)std::max<int64_t>(
        1, std::min<int64_t>({kMaxPromptPieces, (kFewRound + prompts / 2) / prompts, keys / kPieceKeys}));
  s.bytes = off;
  if (s.prompt_pieces > 1) s.piece_bytes = (size_t)prompts * s.prompt_pieces * kPrefillRows * (d + 1) * sizeof(float);
  return s;
}

// A caller's workspace: the lists and the rows' partials, then the pieces'.
static size_t piece_off(const Shape& s) { return (s.bytes + 255) / 256 * 256; }
static size_t workspace_bytes_of(const Shape& s) { return s.piece_bytes > 0 ? piece_off(s) + s.piece_bytes : s.bytes; }

// A second stream per device and the fork/join events that tie it to the caller's stream, created on first use.
// The mutex makes each call's record / wait / launch sequence atomic against calls from other host threads that
// share the device's second stream.
struct SideStream {
  hipStream_t stream = nullptr;
  hipEvent_t fork = nullptr, join = nullptr;
  std::mutex lock;
};
static SideStream* side_stream() {
  static SideStream side[64];
  static std::mutex create;
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return nullptr;
  SideStream& s = side[dev];
  std::lock_guard<std::mutex> g(create);
  if (!s.stream) {  // default priority, non-blocking with respect to the legacy stream
    hipStream_t st = nullptr;
    hipEvent_t f = nullptr, j = nullptr;
    if (hipStreamCreateWithFlags(&st, hipStreamNonBlocking) != hipSuccess) return nullptr;
    if (hipEventCreateWithFlags(&f, hipEventDisableTiming) != hipSuccess) {
      (void)hipStreamDestroy(st);
      return nullptr;
    }
    if (hipEventCreateWithFlags(&j, hipEventDisableTiming) != hipSuccess) {
      (void)hipEventDestroy(f);
      (void)hipStreamDestroy(st);
      return nullptr;
    }
    s.fork = f;
    s.join = j;
    s.stream = st;
  }
  return &s;
}

// Workgroups of kernel K (256 threads) that one CU holds at once, from its register and LDS needs (cached per
// kernel and device).
template <auto K>
static int resident_per_cu() {
  static int cached[64];
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) dev = 0;
  if (cached[dev] > 0) return cached[dev];
  int n = 0;
  if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, K, 256, 0) != hipSuccess || n <= 0) n = 1;
  cached[dev] = n;
  return n;
}

// The kernels of one call, decided on the host from the step's shape (the same decision for a launch and for
// lv_paged_attention_launch_info).
struct StepKind {
  bool listed;        // the step's items come from a device work list (at most kPlanMaxRows rows)
  bool mixed;         // some row has more than one query
  bool overlap;       // the caller's schedule lets prompt tiles run beside the decode items
  bool prompts_only;  // the caller says every row has more than one query
  bool few;           // every row's query heads fit one MFMA item per kv head (few_query.hip)
  int max_q;          // queries per row at most
  int tokens;
  int prompt_wgs;     // the caller's prompt share of the CUs in an overlap (0: the default)
};
struct Route {
  int hp = 1;                                    // kv heads per decode item
  int decode = LV_KERNEL_NONE, decode_grid = 0;  // the launch running the decode items, its workgroups
  int prompt = LV_KERNEL_NONE, prompt_grid = 0;  // the launch running the prompt items (MIXED_SMALL: the same one)
  bool two_streams = false;                      // decode items on the second stream beside prompt_overlap_kernel
  bool merge = false;                            // rows split over items, merged by their last split
};

// CUs that hold a prompt workgroup in an overlapped step: the caller's count clamped to [default, max] and
// rounded down to a multiple of 8, or the default share for 0; never more than there are prompt items.
static int prompt_grid(const Shape& s, const AttnParams& p, int requested) {
  const int cus = device_cus();
  const int lo = std::max(8, cus * kOverlapCusPct / 100 / 8 * 8), hi = std::max(lo, cus * kOverlapCusMaxPct / 100);
  const int n = requested > 0 ? std::min(hi, std::max(lo, requested / 8 * 8)) : lo;
  return std::min(s.max_prompt_items * p.hkv, n);
}

// The route of a step:
// - a step of prompts: its prompt items one workgroup each on the whole GPU;
// - more rows than the work list holds (decode only): one workgroup per (row, split, item head group), no list;
// - a mixed step under the overlapped schedule whose workgroups (bounds: prompt bounds past a row's queries exit at
//   once; decode items at a power of two of keys, the largest number up to kSplitTarget: by the finer splits that the
//   plan may make, a step of few rows with long contexts would be a large one, 235 rows of 16/8 heads beside a
//   1154-token chunk 151 us a layer here and 206 there, 23 rows of 12/1 heads 61 and 80) fill the GPU at most
//   kSmallStepRounds times: prompt and decode items in one launch (mixed_small_kernel);
// - a larger one: prompt items on a persistent share of the CUs, decode items beside them on a second stream, on the
//   persistent ticket grid where the item bound gives each of its workgroups at least eight items (else one
//   workgroup per item: few short items finish sooner all at once than in rounds);
// - otherwise (the serial schedule, or decode only): the prompt items on the whole GPU if any, then the decode items
//   one workgroup each. Outside the overlap one workgroup per item measured as fast as the persistent grid or faster
//   (Qwen3-8B batch-256 decode of kv-head pairs 0.727 against 0.771 ms, same box, medians of 3).
template <typename T, int D, int GS, int TP, int HP>
static Route route_of(const AttnParams& p, const Shape& s, const StepKind& k) {
  Route r;
  r.hp = HP;
  const int ny = p.hkv / HP * p.qgroups;
  const int cus = device_cus();
  const int64_t pw = k.listed && k.mixed ? (int64_t)s.max_prompt_items * p.hkv : 0;
  const int64_t rw = (int64_t)s.route_items * ny;
  const int64_t dw = k.listed ? (int64_t)s.max_decode_items * ny : (int64_t)p.rows * ny;
  r.merge = s.max_splits > 1 && !k.prompts_only;
  if (k.prompts_only) {
    r.prompt = LV_KERNEL_PROMPT_LIST;
    r.prompt_grid = (int)pw * (TP > 0 ? s.prompt_pieces : 1);
  } else if (!k.listed) {
    r.decode = LV_KERNEL_DECODE_GRID;
    r.decode_grid = (int)dw;
  } else if (k.mixed && k.overlap &&
             pw + rw <= (int64_t)kSmallStepRounds * resident_per_cu<mixed_small_kernel<T, D, GS, TP, HP>>() * cus) {
    r.prompt = r.decode = LV_KERNEL_MIXED_SMALL;
    r.prompt_grid = (int)pw;
    r.decode_grid = (int)dw;
  } else if (k.mixed && k.overlap) {
    r.two_streams = true;
    r.prompt = LV_KERNEL_PROMPT_OVERLAP;
    r.prompt_grid = prompt_grid(s, p, k.prompt_wgs);
    const int grid = std::min(kOverlapDecodeWgs, resident_per_cu<decode_beside_kernel<T, D, GS, HP>>()) * cus;
    r.decode = rw >= 8 * (int64_t)grid ? LV_KERNEL_DECODE_BESIDE : LV_KERNEL_DECODE_LIST;
    r.decode_grid = r.decode == LV_KERNEL_DECODE_BESIDE ? grid : (int)dw;
  } else {
    if (k.mixed) {
      r.prompt = LV_KERNEL_PROMPT_LIST;
      r.prompt_grid = (int)pw * (TP > 0 ? s.prompt_pieces : 1);
    }
    r.decode = LV_KERNEL_DECODE_LIST;
    r.decode_grid = (int)dw;
  }
  return r;
}

// The decode launch of a route on `stream`.
template <typename T, int D, int GS, int HP>
static void launch_decode(const AttnParams& p, const Route& r, hipStream_t stream) {
  if (r.decode == LV_KERNEL_DECODE_BESIDE)
    hipLaunchKernelGGL((decode_beside_kernel<T, D, GS, HP>), dim3(r.decode_grid), dim3(256), 0, stream, p);
  else if (r.decode == LV_KERNEL_DECODE_GRID)
    hipLaunchKernelGGL((decode_grid_kernel<T, D, GS, HP>), dim3(p.rows, p.hkv / HP * p.qgroups),
                       dim3(256), 0, stream, p);
  else if (r.decode == LV_KERNEL_DECODE_LIST)
    hipLaunchKernelGGL((decode_list_kernel<T, D, GS, HP, kWideSteps<D, HP>>), dim3(r.decode_grid), dim3(256), 0,
                       stream, p);
}

// A step's kernels after the plan. An overlapped mixed step forks the decode items onto the device's second stream
// and joins it back into `stream` with events; if the second stream cannot be set up, or the fork's record or wait
// fails before anything is launched, the step runs serially instead (the same results, but for the rounding where
// the serial schedule splits few prompt items). A failure after the prompt
// launch leaves the two streams unordered and is returned as LV_EHIP. With `info` set nothing is launched: the
// route is reported instead.
template <typename T, int D, int GS, int TP, int HP>
static int launch(const AttnParams& p, const Shape& s, const StepKind& k, hipStream_t stream, Route* info) {
  const Route r = route_of<T, D, GS, TP, HP>(p, s, k);
  if (info) {
    *info = r;
    return LV_OK;
  }
  if (r.prompt == LV_KERNEL_MIXED_SMALL) {
    hipLaunchKernelGGL((mixed_small_kernel<T, D, GS, TP, HP>), dim3(r.prompt_grid + r.decode_grid), dim3(256), 0,
                       stream, p, (int32_t)r.prompt_grid);
    LV_LAUNCH_CHECK("mixed_small_kernel");
  } else {
    SideStream* side = r.two_streams ? side_stream() : nullptr;
    bool forked = false;
    if (side) {
      // The prompt items go first, to the caller's stream, then the decode items to the second one: the prompt
      // workgroups (one per CU) are dispatched as soon as the plan ends, the decode workgroups fill the rest. On an
      // idle GPU decode workgroups launched first fill every CU, and the prompt items start when they end: the
      // Qwen3-8B mixed step alone 4.62 ms, so 2.95; among others 2.97 and 2.93.
      std::lock_guard<std::mutex> g(side->lock);
      if (hipEventRecord(side->fork, stream) == hipSuccess &&
          hipStreamWaitEvent(side->stream, side->fork, 0) == hipSuccess) {
        forked = true;
        constexpr int pad = std::max(0, kOverlapLds - std::max(1, kRingOf<TP>) * PromptSmem<D, D, (TP > 1)>::kBytes);
        hipLaunchKernelGGL((prompt_overlap_kernel<T, D, TP>), dim3(r.prompt_grid), dim3(256), pad, stream, p);
        LV_LAUNCH_CHECK("prompt_overlap_kernel");
        launch_decode<T, D, GS, HP>(p, r, side->stream);
        LV_LAUNCH_CHECK("decode kernel beside the prompt tiles");
        LV_HIP_CHECK(hipEventRecord(side->join, side->stream));
        LV_HIP_CHECK(hipStreamWaitEvent(stream, side->join, 0));
      } else {
        (void)hipGetLastError();  // the failed record or wait: fall back to the serial schedule
      }
    }
    if (!forked) {
      if (r.prompt != LV_KERNEL_NONE) {  // the serial schedule (or its fallback): prompt items on the whole GPU
        const int items = s.max_prompt_items * p.hkv;
        if constexpr (TP > 0) {
          if (s.prompt_pieces > 1) {
            hipLaunchKernelGGL((prompt_split_kernel<T, D, TP>), dim3(items * s.prompt_pieces), dim3(256), 0, stream, p);
            hipLaunchKernelGGL((prompt_merge_kernel<T, D>), dim3(items * (kPrefillRows * D / 4 / 256)), dim3(256), 0,
                               stream, p);
          }
        }
        if (TP == 0 || s.prompt_pieces == 1)
          hipLaunchKernelGGL((prompt_list_kernel<T, D, TP>), dim3(items), dim3(256), 0, stream, p);
      }
      if (r.decode != LV_KERNEL_NONE) {
        Route serial = r;
        if (serial.decode == LV_KERNEL_DECODE_BESIDE) {  // the fallback: one workgroup per item
          serial.decode = LV_KERNEL_DECODE_LIST;
          serial.decode_grid = s.max_decode_items * (p.hkv / HP) * p.qgroups;
        }
        launch_decode<T, D, GS, HP>(p, serial, stream);
      }
      LV_LAUNCH_CHECK("paged attention kernels");
    }
  }
  return LV_OK;
}

// Pages per 64-key prompt tile for the LDS ring: 1 for pages of a multiple of 64 keys, 2 or 4 for pages of 32 or
// 16; 0 (register staging) for any other size.
static int tile_pages(int block_size) {
  if (block_size % kPrefillKeys == 0) return 1;
  if (block_size == 32) return 2;
  if (block_size == 16) return 4;
  return 0;
}

template <typename T, int D, int GS, int HP>
static int launch_tp(const AttnParams& p, const Shape& s, const StepKind& k, hipStream_t stream, Route* info) {
  switch (tile_pages((int)p.bs.d)) {
    case 1: return launch<T, D, GS, 1, HP>(p, s, k, stream, info);
    case 2: return launch<T, D, GS, 2, HP>(p, s, k, stream, info);
    case 4: return launch<T, D, GS, 4, HP>(p, s, k, stream, info);
    default: return launch<T, D, GS, 0, HP>(p, s, k, stream, info);
  }
}

// Decode items of a streaming step take two kv heads where the step has an even number: a token's two head rows are
// adjacent in the NHD cache, so each 64-lane load covers 512-byte pieces of token rows instead of 256-byte ones (a
// math-free stream of 512-byte pieces at a 2 KB stride reads 7.15 TB/s on an MI355X, of 256-byte pieces
// 6.5-6.7 TB/s). The split of a row's keys stays as planned, so such items are half as many and twice as long;
// steps of fewer than kPairItems one-head items per CU (a few short rows, latency-bound) keep one head per item.
// A lane addresses the second head's row with a 32-bit offset (the head stride) inside its tile, so pairs also need
// a head stride under 2^30 bytes.
constexpr int kPairItems = 8;
template <typename T, int D, int GS>
static int launch_hp(const AttnParams& p, const Shape& s, const StepKind& k, hipStream_t stream, Route* info) {
  const int64_t items = (int64_t)(k.listed ? s.max_decode_items : p.rows) * p.hkv * p.qgroups;
  if (p.hkv % 2 == 0 && p.c_sh >= 0 && p.c_sh < ((int64_t)1 << 30) && items >= (int64_t)kPairItems * device_cus())
    return launch_tp<T, D, GS, 2>(p, s, k, stream, info);
  return launch_tp<T, D, GS, 1>(p, s, k, stream, info);
}

template <typename T, int D>
static int launch_gs(const AttnParams& p, int gs, const Shape& s, const StepKind& k, hipStream_t stream,
                     Route* info) {
  if (gs == 4) return launch_hp<T, D, 4>(p, s, k, stream, info);
  if (gs == 2) return launch_hp<T, D, 2>(p, s, k, stream, info);
  return launch_hp<T, D, 1>(p, s, k, stream, info);
}

template <typename T>
static int launch_d(const AttnParams& p, int d, int gs, const Shape& s, const StepKind& k, hipStream_t stream,
                    Route* info) {
  switch (d) {
    case 64: return launch_gs<T, 64>(p, gs, s, k, stream, info);
    case 128: return launch_gs<T, 128>(p, gs, s, k, stream, info);
    default: set_error("paged_attention: head_dim %d is not 64 or 128", d); return LV_EINVAL;
  }
}

// A step's kernels after the plan, by its kind: rows of few queries on few_query.hip's items, else by dtype, head dim,
// lane group, kv heads per item and pages.
static int launch_step(const AttnParams& p, int d, const Shape& s, const StepKind& k, int dtype, hipStream_t stream,
                       Route* info) {
  if (k.few) {
    Route r;
    r.decode = LV_KERNEL_DECODE_LIST;
    // Pairs of kv heads (512-byte pieces of a token's row): where two rounds of workgroups remain without splits (200
    // rows of 4 queries 1178 -> 1114 us, two layers; 100 rows 631 -> 737), or items are light and fill the CUs.
    const int64_t items = (int64_t)s.max_decode_items * p.hkv;
    const bool light = ((int64_t)k.tokens + p.rows - 1) / p.rows * p.group <= 4;  // as plan_shape has it
    const bool pairs = light ? items >= kFewRound : (int64_t)p.rows * p.hkv >= 2 * kFewRound;
    r.hp = p.hkv % 2 == 0 && k.max_q * p.group <= 32 && pairs ? 2 : 1;
    r.decode_grid = s.max_decode_items * (p.hkv / r.hp);
    r.merge = s.max_splits > 1;
    if (info) {
      *info = r;
      return LV_OK;
    }
    launch_few_query(p, d, k.max_q * p.group, r.hp, dtype, s.max_decode_items, stream);
    LV_LAUNCH_CHECK("few_list_kernel");
    return LV_OK;
  }
  return dtype == LV_DTYPE_BF16 ? launch_d<BF16>(p, d, s.gs, s, k, stream, info)
                                : launch_d<F16>(p, d, s.gs, s, k, stream, info);
}

// --------------------------------------------------------------------------------------------------------- The
// workspace of lv_paged_attention_static: file-scope device arrays (each GPU that loads the library holds its own
// copies until the process ends), one for the lists and the rows' partials, one for the pieces of split prompt items
// (its size covers every step that splits them). Host code must not pass an array's name to a kernel -- in host code
// it is a stand-in, not a device address; its address on the current device comes from hipGetSymbolAddress, resolved
// once per device and kept. The same set-up creates the device's second stream and its fork/join events, so that no
// later call creates anything.
constexpr size_t kStaticPieceBytes = (size_t)kMaxPieces * kPrefillRows * (128 + 1) * sizeof(float);
static __device__ __align__(256) char scratch[LV_STATIC_WORKSPACE_BYTES];
static __device__ __align__(256) char piece_scratch[kStaticPieceBytes];

struct Scratch {
  void *ws, *pieces;
};
static Scratch scratch_on_current_device() {
  static Scratch addr[64];
  static std::mutex lock;
  int dev = 0;
  const hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) {
    set_error("paged_attention_static: hipGetDevice failed: %s", hipGetErrorString(e));
    return Scratch{};
  }
  if (dev < 0 || dev >= 64) {
    set_error("paged_attention_static: device %d is past the 64 devices served", dev);
    return Scratch{};
  }
  std::lock_guard<std::mutex> g(lock);
  if (!addr[dev].ws) {
    Scratch s{};
    hipError_t r = hipGetSymbolAddress(&s.ws, HIP_SYMBOL(scratch));
    if (r == hipSuccess) r = hipGetSymbolAddress(&s.pieces, HIP_SYMBOL(piece_scratch));
    if (r != hipSuccess || !s.ws || !s.pieces) {
      set_error("paged_attention_static: hipGetSymbolAddress of the static workspace failed on device %d: %s", dev,
                hipGetErrorString(r));
      return Scratch{};
    }
    if (!side_stream()) {
      set_error("paged_attention_static: the second stream of device %d could not be created", dev);
      return Scratch{};
    }
    addr[dev] = s;
  }
  return addr[dev];
}

// What a work list was planned for, per workspace: a caller's request to reuse the plan already in a workspace
// (LV_ATTN_REUSE_PLAN, for the later layers of a step) is honoured only if the workspace's last plan was made for the
// same rows, shape and row-length arrays; otherwise the call plans again.
struct PlanSig {
  const void* ws = nullptr;
  const int32_t *cu_q = nullptr, *lens = nullptr, *cu_k = nullptr;
  int64_t rows = 0, tokens = 0, max_k = 0, pieces = 0, slots = 0, qp = 0, max_items = 0, merge_off = 0, bytes = 0;
  bool mixed = false, last_first = false, few = false, prompts = false;
  bool operator==(const PlanSig& o) const {
    return ws == o.ws && cu_q == o.cu_q && lens == o.lens && cu_k == o.cu_k && rows == o.rows &&
           tokens == o.tokens && max_k == o.max_k && pieces == o.pieces && slots == o.slots && qp == o.qp &&
           max_items == o.max_items && merge_off == o.merge_off && bytes == o.bytes && mixed == o.mixed &&
           last_first == o.last_first && few == o.few && prompts == o.prompts;
  }
};
constexpr int kPlanRecords = 32;
static std::mutex g_plan_lock;
static PlanSig g_plans[kPlanRecords];

// True if a caller asks to reuse the plan in `sig`'s workspace and that workspace's last plan is the one `sig`
// describes.
static bool plan_is_current(const PlanSig& sig, bool reuse) {
  if (!reuse) return false;
  std::lock_guard<std::mutex> g(g_plan_lock);
  for (int i = 0; i < kPlanRecords; ++i)
    if (g_plans[i].ws == sig.ws) return g_plans[i] == sig;
  return false;
}

// Records what workspace `ws` now holds: the plan `sig` (after its launch was accepted), or nothing (sig null: a
// call that failed after choosing to plan, whose list may never be written).
static void record_plan(const void* ws, const PlanSig* sig) {
  std::lock_guard<std::mutex> g(g_plan_lock);
  int slot = -1;
  for (int i = 0; i < kPlanRecords; ++i)
    if (g_plans[i].ws == ws) slot = i;
  if (!sig) {
    if (slot >= 0) g_plans[slot] = PlanSig{};
    return;
  }
  if (slot < 0) {  // a new workspace: take a free record, else the first
    slot = 0;
    for (int i = 0; i < kPlanRecords; ++i)
      if (!g_plans[i].ws) {
        slot = i;
        break;
      }
  }
  g_plans[slot] = *sig;
}

// The checks on a step's shape and options, shared by the call and the launch-info query.
static int check_shape(int32_t num_rows, int32_t num_tokens, int32_t num_heads, int32_t num_kv_heads,
                       int32_t head_dim, int32_t block_size, bool has_cu_q, int32_t max_seqlen_q,
                       int32_t max_seqlen_k, int32_t schedule, int32_t prompt_workgroups, int32_t flags,
                       int32_t dtype) {
  LV_REQUIRE(dtype == LV_DTYPE_BF16 || dtype == LV_DTYPE_F16, "paged_attention: dtype %d is not bf16 or fp16",
             dtype);
  LV_REQUIRE(num_rows >= 0 && num_tokens >= 0, "paged_attention: negative row or token count");
  LV_REQUIRE(schedule == LV_SCHEDULE_AUTO || schedule == LV_SCHEDULE_SERIAL || schedule == LV_SCHEDULE_OVERLAP,
             "paged_attention: unknown schedule %d", schedule);
  LV_REQUIRE(prompt_workgroups >= 0, "paged_attention: negative prompt_workgroups %d", prompt_workgroups);
  LV_REQUIRE((flags & ~(LV_ATTN_REUSE_PLAN | LV_ATTN_PROMPTS_ONLY)) == 0, "paged_attention: unknown flags 0x%x",
             flags);
  LV_REQUIRE(!(flags & LV_ATTN_PROMPTS_ONLY) || (has_cu_q && max_seqlen_q > 1),
             "paged_attention: LV_ATTN_PROMPTS_ONLY needs cu_seqlens_q and max_seqlen_q > 1");
  if (num_rows == 0 || num_tokens == 0) return LV_OK;
  LV_REQUIRE(num_heads > 0 && num_kv_heads > 0 && num_heads % num_kv_heads == 0,
             "paged_attention: %d query heads do not group over %d key heads", num_heads, num_kv_heads);
  LV_REQUIRE(num_heads / num_kv_heads <= kPrefillRows, "paged_attention: query group %d exceeds %d",
             num_heads / num_kv_heads, kPrefillRows);
  LV_REQUIRE(head_dim == 64 || head_dim == 128, "paged_attention: head_dim %d is not 64 or 128", head_dim);
  LV_REQUIRE(block_size > 0 && block_size % kTile == 0, "paged_attention: block_size %d is not a multiple of %d",
             block_size, kTile);
  LV_REQUIRE(has_cu_q || num_tokens == num_rows, "paged_attention: without cu_seqlens_q, T (%d) must equal B (%d)",
             num_tokens, num_rows);
  LV_REQUIRE(max_seqlen_k >= 0 && max_seqlen_k <= (1 << 30), "paged_attention: max_seqlen_k %d is negative or above "
             "2^30 keys", max_seqlen_k);
  LV_REQUIRE(!(has_cu_q && max_seqlen_q > 1) || num_rows <= kPlanMaxRows,
             "paged_attention: a step with prompts holds at most %d rows, got %d", kPlanMaxRows, num_rows);
  return LV_OK;
}

static StepKind step_kind(int32_t num_rows, int32_t num_tokens, int32_t num_heads, int32_t num_kv_heads,
                          int32_t head_dim, bool has_cu_q, int32_t max_seqlen_q, int32_t schedule,
                          int32_t prompt_workgroups, int32_t flags) {
  const int group = num_heads / num_kv_heads;
  const int few = few_queries(num_rows, num_kv_heads, head_dim, group);
  StepKind k;
  k.mixed = has_cu_q && max_seqlen_q > 1;
  k.listed = num_rows <= kPlanMaxRows;
  k.overlap = schedule != LV_SCHEDULE_SERIAL;
  k.prompts_only = (flags & LV_ATTN_PROMPTS_ONLY) != 0;
  k.prompt_wgs = prompt_workgroups;
  k.max_q = k.mixed ? max_seqlen_q : 1;
  k.tokens = num_tokens;
  k.few = k.listed && k.max_q <= few && num_tokens <= (int64_t)num_rows * few &&
          (k.mixed || pick_gs(group) != group);
  return k;
}

// A launch counts its work-items (workgroups x 256) in 32 bits: the step's largest grid must stay below that.
static int check_grids(const Shape& s, int32_t num_rows, int32_t num_heads, int32_t num_kv_heads) {
  const int64_t prompt = (int64_t)s.max_prompt_items * num_kv_heads;
  const int64_t decode = std::max<int64_t>(s.max_decode_items, num_rows) * num_heads;
  LV_REQUIRE(fits_one_launch(prompt + decode, 256),
             "paged_attention: the step needs %lld + %lld workgroups, more than one launch holds", (long long)prompt,
             (long long)decode);
  return LV_OK;
}

// The shape part of a step's parameters (what the route depends on).
static void shape_params(AttnParams& p, const Shape& s, int32_t num_rows, int32_t num_heads, int32_t num_kv_heads,
                         int32_t block_size, int64_t cache_stride_head) {
  p.bs = FastDiv::make((uint32_t)block_size);
  p.c_sh = cache_stride_head * 2;
  p.rows = num_rows;
  p.hq = num_heads;
  p.hkv = num_kv_heads;
  p.group = num_heads / num_kv_heads;
  p.qgroups = p.group / s.gs;
}

// One step, with the workspace given (workspace != nullptr or an empty shape) or, for static_ws, the device's
// static workspace.
static int paged_attention(const void* q, int64_t q_stride_t, int64_t q_stride_h, const void* k_cache,
                           const void* v_cache, int64_t cache_stride_block, int64_t cache_stride_token,
                           int64_t cache_stride_head, int32_t block_size, const int32_t* block_tables,
                           int64_t table_stride, const int32_t* cu_seqlens_q, const int32_t* seqlens_k,
                           const int32_t* cu_seqlens_k, int32_t num_rows, int32_t num_tokens, int32_t num_heads,
                           int32_t num_kv_heads, int32_t head_dim, float scale, int32_t max_seqlen_q,
                           int32_t max_seqlen_k, void* out, int64_t out_stride_t, int64_t out_stride_h,
                           void* workspace, size_t workspace_bytes, bool static_ws, int32_t schedule,
                           int32_t prompt_workgroups, int32_t flags, int32_t dtype, void* stream) {
  const int rc0 = check_shape(num_rows, num_tokens, num_heads, num_kv_heads, head_dim, block_size,
                              cu_seqlens_q != nullptr, max_seqlen_q, max_seqlen_k, schedule, prompt_workgroups,
                              flags, dtype);
  if (rc0 != LV_OK || num_rows == 0 || num_tokens == 0) return rc0;
  LV_REQUIRE(q && k_cache && v_cache && out && block_tables, "paged_attention: null tensor pointer");
  LV_REQUIRE(seqlens_k || cu_seqlens_k, "paged_attention: neither key lengths nor cu_seqlens_k given");
  // 16-byte rows: q, out and cache head rows are read and written as 16-byte vectors.
  LV_REQUIRE(aligned(q, 16) && aligned(out, 16) && aligned(k_cache, 16) && aligned(v_cache, 16) &&
                 (q_stride_t * 2) % 16 == 0 && (q_stride_h * 2) % 16 == 0 && (out_stride_t * 2) % 16 == 0 &&
                 (out_stride_h * 2) % 16 == 0 && (cache_stride_block * 2) % 16 == 0 &&
                 (cache_stride_token * 2) % 16 == 0 && (cache_stride_head * 2) % 16 == 0,
             "paged_attention: tensors and their strides must be 16-byte aligned");
  // Lanes address their rows inside a 16-token decode tile or a 64-key prompt tile with 32-bit byte offsets, the
  // prompt tile's as 24-bit products (key row times token stride).
  LV_REQUIRE(cache_stride_token >= 0 && (int64_t)kPrefillKeys * cache_stride_token * 2 < (int64_t)1 << 30,
             "paged_attention: cache token stride %lld is negative or too large", (long long)cache_stride_token);
  LV_REQUIRE(scale > 0.f, "paged_attention: the softmax scale must be positive, got %g", (double)scale);
  const StepKind kind = step_kind(num_rows, num_tokens, num_heads, num_kv_heads, head_dim, cu_seqlens_q != nullptr,
                                  max_seqlen_q, schedule, prompt_workgroups, flags);
  const Shape s = plan_shape(num_rows, num_tokens, num_heads, num_kv_heads, head_dim, max_seqlen_k, kind.listed,
                             kind.few, kind.max_q, kind.mixed);
  const int rg = check_grids(s, num_rows, num_heads, num_kv_heads);
  if (rg != LV_OK) return rg;
  char* pieces = nullptr;
  if (static_ws) {
    LV_REQUIRE(s.bytes <= (size_t)LV_STATIC_WORKSPACE_BYTES,
               "paged_attention_static: this step needs %zu bytes of workspace; the static workspace holds %zu "
               "(LV_STATIC_WORKSPACE_BYTES): call lv_paged_attention with a workspace instead",
               s.bytes, (size_t)LV_STATIC_WORKSPACE_BYTES);
    LV_REQUIRE(s.piece_bytes <= kStaticPieceBytes, "paged_attention_static: %zu bytes of prompt pieces, more than %zu",
               s.piece_bytes, kStaticPieceBytes);
    const Scratch scratch = scratch_on_current_device();
    if (!scratch.ws) return LV_EHIP;
    workspace = scratch.ws;
    pieces = (char*)scratch.pieces;
  } else {
    const size_t need = workspace_bytes_of(s);
    LV_REQUIRE(workspace_bytes >= need && (need == 0 || workspace),
               "paged_attention: workspace of %zu bytes given, %zu needed", workspace_bytes, need);
    LV_REQUIRE(aligned(workspace, 256), "paged_attention: workspace must be 256-byte aligned");
    if (s.piece_bytes > 0) pieces = (char*)workspace + piece_off(s);
  }

  AttnParams p{};
  shape_params(p, s, num_rows, num_heads, num_kv_heads, block_size, cache_stride_head);
  p.q = (const char*)q;
  p.q_st = q_stride_t * 2;
  p.q_sh = q_stride_h * 2;
  p.k_cache = (const char*)k_cache;
  p.v_cache = (const char*)v_cache;
  p.c_sb = cache_stride_block * 2;
  p.c_st = cache_stride_token * 2;
  p.v_st = p.c_st;
  p.v_sh = p.c_sh;
  p.paged = true;
  p.causal = 1;
  // Decode items read their row's first page before its length; with no keys at all a table may hold no entry, so the
  // lengths (any readable ints) stand in for it.
  p.tables = max_seqlen_k > 0 ? block_tables : seqlens_k ? seqlens_k : cu_seqlens_k;
  p.t_stride = max_seqlen_k > 0 ? table_stride : 0;
  p.cu_q = cu_seqlens_q;
  p.lens_k = seqlens_k;
  p.cu_k = cu_seqlens_k;
  p.scale_log2 = scale * kLog2e;
  p.out = (char*)out;
  p.o_st = out_stride_t * 2;
  p.o_sh = out_stride_h * 2;
  char* ws = (char*)workspace;
  p.part_base = s.slots > 0 ? reinterpret_cast<const int32_t*>(ws + s.base_off) : nullptr;
  p.part_lse = s.slots > 0 ? reinterpret_cast<float*>(ws + s.lse_off) : nullptr;
  p.part_o = s.slots > 0 ? reinterpret_cast<float*>(ws + s.o_off) : nullptr;
  p.prompts = kind.listed ? reinterpret_cast<const int2*>(ws + s.items_off) : nullptr;
  p.items = kind.listed ? p.prompts + s.max_prompt_items : nullptr;
  p.pieces = s.prompt_pieces;
  if (s.piece_bytes > 0) {
    p.piece_o = reinterpret_cast<float*>(pieces);
    p.piece_lse = p.piece_o + (s.piece_bytes / sizeof(float)) / (head_dim + 1) * head_dim;
  }
  p.n_items = kind.listed ? reinterpret_cast<const int32_t*>(ws + s.count_off) : nullptr;
  p.ticket = kind.listed ? reinterpret_cast<int32_t*>(ws + s.count_off) + kPlanTicket : nullptr;
  p.merge_count = s.merges > 0 ? reinterpret_cast<int32_t*>(ws + s.merge_off) : nullptr;

  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  const int qp = kPrefillRows / p.group;
  PlanSig sig;
  sig.ws = workspace;
  sig.cu_q = kind.mixed ? cu_seqlens_q : nullptr;
  sig.lens = seqlens_k;
  sig.cu_k = cu_seqlens_k;
  sig.rows = num_rows;
  sig.tokens = num_tokens;
  sig.max_k = max_seqlen_k;
  sig.pieces = s.pieces;
  sig.slots = s.slots;
  sig.qp = qp;
  sig.max_items = s.max_items;
  sig.merge_off = (int64_t)s.merge_off;
  sig.bytes = (int64_t)s.bytes;
  sig.mixed = kind.mixed;
  sig.few = kind.few;
  sig.prompts = kind.prompts_only && !kind.few;
  sig.last_first = kind.prompts_only || !kind.overlap;  // prompt items with the GPU to themselves: last tile first
  bool planned = false;
  if (kind.listed && !plan_is_current(sig, (flags & LV_ATTN_REUSE_PLAN) != 0)) {
    record_plan(workspace, nullptr);  // until this plan's launch is accepted, the workspace holds no plan
    int2* lists = reinterpret_cast<int2*>(ws + s.items_off);
    const PlanOut out{lists, lists + s.max_prompt_items, reinterpret_cast<int32_t*>(ws + s.count_off),
                      reinterpret_cast<int32_t*>(ws + s.base_off), p.merge_count};
    // Few-query items take a row's queries from cu_seqlens_q, so its partial slots are counted from there too, also
    // in a step that was said to have one query a row.
    constexpr int kMany = kPlanMaxRows / kScanThreads;
    const bool many = num_rows > kScanThreads;
    auto* const plan = sig.prompts ? (many ? &plan_kernel<kMany, true> : &plan_kernel<1, true>)
                                   : (many ? &plan_kernel<kMany, false> : &plan_kernel<1, false>);
    hipLaunchKernelGGL(plan, dim3(1), dim3(kScanThreads), 0, st,
                       kind.mixed || kind.few ? cu_seqlens_q : nullptr, seqlens_k, cu_seqlens_k, num_rows, s.pieces,
                       s.slots, qp, s.max_prompt_items, s.max_decode_items, (int32_t)sig.last_first, (int32_t)kind.few,
                       s.fewer_pieces, p.group, p.hkv, (int32_t)s.merges, out);
    LV_LAUNCH_CHECK("plan_kernel");
    planned = true;
  }
  const int rc = launch_step(p, head_dim, s, kind, dtype, st, nullptr);
  if (rc != LV_OK) {
    // A failed launch may leave the persistent grid's ticket unreset: the next call on this workspace plans again.
    record_plan(workspace, nullptr);
    return rc;
  }
  if (planned) record_plan(workspace, &sig);
  return LV_OK;
}

}  // namespace lv

using namespace lv;

extern "C" size_t lv_paged_attention_workspace_bytes(int32_t num_rows, int32_t num_tokens, int32_t num_heads,
                                                     int32_t num_kv_heads, int32_t head_dim, int32_t max_seqlen_k,
                                                     int32_t decode_only) {
  if (num_rows <= 0 || num_heads <= 0 || num_kv_heads <= 0 || num_heads % num_kv_heads || max_seqlen_k < 0 ||
      max_seqlen_k > (1 << 30))
    return 0;
  const bool mixed = decode_only == 0;
  const bool listed = mixed || num_rows <= kPlanMaxRows;
  const int group = num_heads / num_kv_heads;
  const int few_q = few_queries(num_rows, num_kv_heads, head_dim, group);
  const bool may_be_few =
      listed && num_tokens <= (int64_t)num_rows * few_q && (mixed || pick_gs(group) != group);
  auto bytes = [&](bool few) {
    return workspace_bytes_of(plan_shape(num_rows, num_tokens, num_heads, num_kv_heads, head_dim, max_seqlen_k,
                                         listed, few, mixed ? few_q : 1, mixed));
  };
  // The longest row's queries are not known here: a step whose rows may all have few takes the larger of the two.
  return may_be_few ? std::max(bytes(false), bytes(true)) : bytes(false);
}

extern "C" int lv_paged_attention_launch_info(int32_t num_rows, int32_t num_tokens, int32_t num_heads,
                                              int32_t num_kv_heads, int32_t head_dim, int32_t block_size,
                                              int64_t cache_stride_head, int32_t has_cu_seqlens_q,
                                              int32_t max_seqlen_q, int32_t max_seqlen_k, int32_t schedule,
                                              int32_t prompt_workgroups, int32_t flags, int32_t dtype,
                                              lv_launch_info* info) {
  LV_REQUIRE(info, "paged_attention_launch_info: info is null");
  *info = lv_launch_info{};
  const int rc0 = check_shape(num_rows, num_tokens, num_heads, num_kv_heads, head_dim, block_size,
                              has_cu_seqlens_q != 0, max_seqlen_q, max_seqlen_k, schedule, prompt_workgroups, flags,
                              dtype);
  if (rc0 != LV_OK || num_rows == 0 || num_tokens == 0) return rc0;
  const StepKind kind = step_kind(num_rows, num_tokens, num_heads, num_kv_heads, head_dim, has_cu_seqlens_q != 0,
                                  max_seqlen_q, schedule, prompt_workgroups, flags);
  const Shape s = plan_shape(num_rows, num_tokens, num_heads, num_kv_heads, head_dim, max_seqlen_k, kind.listed,
                             kind.few, kind.max_q, kind.mixed);
  const int rg = check_grids(s, num_rows, num_heads, num_kv_heads);
  if (rg != LV_OK) return rg;
  AttnParams p{};
  shape_params(p, s, num_rows, num_heads, num_kv_heads, block_size, cache_stride_head);
  Route r;
  const int rc = launch_step(p, head_dim, s, kind, dtype, nullptr, &r);
  if (rc != LV_OK) return rc;
  info->decode_kernel = r.decode;
  info->decode_workgroups = r.decode_grid;
  info->prompt_kernel = r.prompt;
  info->prompt_workgroups = r.prompt_grid;
  info->kv_heads_per_item = r.hp;
  info->two_streams = r.two_streams;
  const int least = kind.few ? least_split(max_seqlen_k, std::min(kind.max_q, num_tokens) * p.group) : 0;
  info->keys_per_split = split_keys((float)num_rows * (float)max_seqlen_k, std::max(max_seqlen_k, 1),
                                    std::max(kMinSplit, least), s.pieces, kind.few ? 0 : num_kv_heads);
  info->max_splits = s.max_splits;
  info->splitk_merge = r.merge;
  return LV_OK;
}

extern "C" int lv_paged_attention(const void* q, int64_t q_stride_t, int64_t q_stride_h, const void* k_cache,
                                  const void* v_cache, int64_t cache_stride_block, int64_t cache_stride_token,
                                  int64_t cache_stride_head, int32_t block_size, const int32_t* block_tables,
                                  int64_t table_stride, const int32_t* cu_seqlens_q, const int32_t* seqlens_k,
                                  const int32_t* cu_seqlens_k, int32_t num_rows, int32_t num_tokens,
                                  int32_t num_heads, int32_t num_kv_heads, int32_t head_dim, float scale,
                                  int32_t max_seqlen_q, int32_t max_seqlen_k, void* out, int64_t out_stride_t,
                                  int64_t out_stride_h, void* workspace, size_t workspace_bytes, int32_t schedule,
                                  int32_t prompt_workgroups, int32_t flags, int32_t dtype, void* stream) {
  return paged_attention(q, q_stride_t, q_stride_h, k_cache, v_cache, cache_stride_block, cache_stride_token,
                         cache_stride_head, block_size, block_tables, table_stride, cu_seqlens_q, seqlens_k,
                         cu_seqlens_k, num_rows, num_tokens, num_heads, num_kv_heads, head_dim, scale, max_seqlen_q,
                         max_seqlen_k, out, out_stride_t, out_stride_h, workspace, workspace_bytes, false, schedule,
                         prompt_workgroups, flags, dtype, stream);
}

extern "C" int lv_paged_attention_static(const void* q, int64_t q_stride_t, int64_t q_stride_h, const void* k_cache,
                                         const void* v_cache, int64_t cache_stride_block, int64_t cache_stride_token,
                                         int64_t cache_stride_head, int32_t block_size, const int32_t* block_tables,
                                         int64_t table_stride, const int32_t* cu_seqlens_q, const int32_t* seqlens_k,
                                         const int32_t* cu_seqlens_k, int32_t num_rows, int32_t num_tokens,
                                         int32_t num_heads, int32_t num_kv_heads, int32_t head_dim, float scale,
                                         int32_t max_seqlen_q, int32_t max_seqlen_k, void* out, int64_t out_stride_t,
                                         int64_t out_stride_h, int32_t schedule, int32_t prompt_workgroups,
                                         int32_t flags, int32_t dtype, void* stream) {
  return paged_attention(q, q_stride_t, q_stride_h, k_cache, v_cache, cache_stride_block, cache_stride_token,
                         cache_stride_head, block_size, block_tables, table_stride, cu_seqlens_q, seqlens_k,
                         cu_seqlens_k, num_rows, num_tokens, num_heads, num_kv_heads, head_dim, scale, max_seqlen_q,
                         max_seqlen_k, out, out_stride_t, out_stride_h, nullptr, 0, true, schedule, prompt_workgroups,
                         flags, dtype, stream);
}
