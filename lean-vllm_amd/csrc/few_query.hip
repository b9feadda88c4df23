// Paged attention of rows with few queries on MFMA: drafted tokens (2 to 16 queries a row), and decode rows whose GQA
// group is not 1, 2 or 4 query heads.
//
// An item is (row, split, kv head): all of the row's (position, head) query rows of one GQA group, up to 64, against
// the keys [split * S, (split + 1) * S) of the row, so the keys and values are read from memory once. Bound by HBM:
// 16 to 64 query rows do 16 to 64 flops a byte. The VALU decode item takes one query and 1, 2 or 4 heads of a group,
// and would read the keys once for each such share; the MFMA prompt item holds 128 query rows and walks the row's
// keys in one workgroup, which leaves most of the chip idle on a few long rows.
//
// Each of a workgroup's four waves takes every 4th tile of the item's keys through a private two-stage LDS ring, filled
// straight from memory; no barrier until the waves merge. A tile's keys are refilled as soon as their scores are in
// registers and its values as soon as P.V has read them, so a wave keeps 12 KB to 16 KB in flight. S^T = K Q^T on MFMA
// 16x16x32, O^T += V^T P^T with V^T operands from the transposing LDS read, the softmax per query row in between.
// Math: TorchAttention.decode / prefill (lean_vllm/attention/torch_backend.py:62-103), as paged_attention.hip.
#include "split_rows.h"

namespace lv {

// Keys per wave tile: 4 KB of keys and 4 KB of values.
template <int D>
constexpr int kFewTile = 2048 / D;
constexpr int kFewHalf = 4096;           // bytes of a tile's keys or values
constexpr int kFewStage = 2 * kFewHalf;  // a stage: keys, then values
constexpr int kFewStages = 2;
constexpr int kFewLoads = kFewHalf / 1024;  // 64-lane 16-byte loads of a tile's keys or values

template <int N>
__device__ __forceinline__ void few_wait() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

// NB: 16-row blocks of (position, head) query rows that a wave holds. How the waves share an item:
// - kOneSet: each takes every 4th tile;
// - kTwoHeads: the item is a pair of kv heads (kvh: the first); waves 0 and 2 take its first, 1 and 3 its second, each
//   every 2nd tile;
// - kTwoBlocks: waves 0 and 2 hold the first 16 NB query rows, 1 and 3 the next, each every 2nd tile, which two waves
//   then load. For 33 to 64 query rows at D = 128, where a wave of four 16-row blocks spills: three times the time.
enum FewSets { kOneSet, kTwoHeads, kTwoBlocks };
template <typename T, int D, int NB, FewSets SETS>
__device__ __forceinline__ void few_item(const AttnParams& p, int row, int split, int per, int kvh, char* smem) {
  using E = Elem<T>;
  constexpr int KT = kFewTile<D>, KB = KT / 16;  // keys per tile, 16-key blocks
  constexpr int KS = D / 32, DB = D / 16, CH = D / 8;
  constexpr int KPL = 64 / CH;  // keys per load
  constexpr int NS = SETS == kOneSet ? 1 : 2;  // sets of waves
  constexpr int HP = SETS == kTwoHeads ? 2 : 1;  // kv heads
  constexpr int WT = kWaves / NS;                // waves that share the tiles
  constexpr int SET_ROWS = SETS == kTwoBlocks ? 16 * NB : 0;  // query rows between the sets
  static_assert(KB == 1 || KB == 2, "16 or 32 keys per tile");
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int n = lane & 15, j4 = lane >> 4;
  const int G = p.group, set = wave % NS, wh = kvh + (HP > 1 ? set : 0);  // this wave's kv head
  const float c = p.scale_log2;

  const int32_t* len = p.lens_k ? p.lens_k + row : p.cu_k + row;
  const int32_t* first = p.cu_q ? p.cu_q + row : len;
  const int32_t* const where[4] = {len, p.lens_k ? len : len + 1, first, p.cu_q ? first + 1 : first};
  int got[4];
  sload_n<4>(where, got);
  const int lk = p.lens_k ? got[0] : got[1] - got[0];
  const int tok = p.cu_q ? got[2] : row, lq = p.cu_q ? got[3] - got[2] : 1;
  const int kbeg = split * per;
  if (split > 0 && kbeg >= lk) return;  // past the row's end: the row has shrunk since the plan
  const int kend = min(lk, kbeg + per);
  const int nsplit = lk > per ? (lk + per - 1) / per : 1;
  const int qrows = lq * G;
  const int slot0 = nsplit > 1 ? p.part_base[row] : 0;  // the row's partial slots, lq per split
  const int32_t* table = p.tables + (int64_t)row * p.t_stride;
  // This wave's tiles t = 0 .. nt - 1 start at key k0 + KT WT t.
  const int k0 = kbeg + KT * (wave / NS);
  const int nt = kend > k0 ? (kend - k0 + KT * WT - 1) / (KT * WT) : 0;

  // Loads of a tile: load j holds keys KPL j .. + KPL - 1, lane l the 16-byte chunk that belongs at position l of their
  // swizzled rows.
  const int st = (int)p.c_st;
  int chunk[kFewLoads], key[kFewLoads];
  uint32_t voff[kFewLoads];  // byte offset inside the 16-key block
#pragma unroll
  for (int j = 0; j < kFewLoads; ++j) {
    key[j] = KPL * j + lane / CH;
    chunk[j] = 16 * swz<CH, true>(key[j], lane % CH);
    voff[j] = __umul24(key[j] & 15, st) + chunk[j];
  }
  int kpos[KS], vpos[DB];
#pragma unroll
  for (int k = 0; k < KS; ++k) kpos[k] = 8 * swz<CH, true>(n, 4 * k + j4);
#pragma unroll
  for (int b = 0; b < DB; ++b) vpos[b] = 8 * swz<CH, true>(4 * j4 + (n >> 2), 2 * b + ((n & 3) >> 1)) + 4 * (n & 1);

  // Pages of the wave's next 64 tiles, one tile per lane (a 16-key block lies in one page).
  int pages[KB];
  // A block past the end: block 0.
  auto block_start = [&](int t0, int b) { return t0 + 16 * b < kend ? t0 + 16 * b : t0; };
  auto load_pages = [&](int t) {
    const int t0 = min(k0 + KT * WT * (t + lane), kend - 1);
#pragma unroll
    for (int b = 0; b < KB; ++b) pages[b] = table[p.bs.div(block_start(t0, b))];
  };

  char* ring = smem + wave * kFewStages * kFewStage;
  int64_t off[KB];  // byte offsets of the tile being filled, in either cache
  auto locate = [&](int t) {
    if ((t & 63) == 0) load_pages(t);
    const int t0 = k0 + KT * WT * t;
#pragma unroll
    for (int b = 0; b < KB; ++b) {
      const int s = block_start(t0, b);
      const int pg = (int)p.bs.div(s);
      off[b] = (int64_t)__builtin_amdgcn_readlane(pages[b], t & 63) * p.c_sb +
               (int64_t)(s - pg * (int)p.bs.d) * p.c_st + (int64_t)wh * p.c_sh;
    }
  };
  // The keys or the values of tile t, located before. Keys past the item's end load its last key (finite; weight 0).
  auto fill = [&](int t, const char* cache, char* dst) {
    const int t0 = k0 + KT * WT * t, last = kend - 1 - t0;
    const uint32_t at = lds_addr(dst);
    if (last >= KT - 1) {
#pragma unroll
      for (int j = 0; j < kFewLoads; ++j) lds_dma16(cache + off[KPL * j / 16], voff[j], at + 1024 * j);
    } else {
#pragma unroll
      for (int j = 0; j < kFewLoads; ++j) {
        const int b = KPL * j / 16;
        const int r = min(key[j], last) - (block_start(t0, b) - t0);
        lds_dma16(cache + off[b], __umul24(r, st) + chunk[j], at + 1024 * j);
      }
    }
  };

  // One pass, unless the row has more query rows than the launch expects.
  for (int q0 = 0; q0 < qrows; q0 += 16 * NB + SET_ROWS) {
    // Query rows q0 + SET_ROWS set + 16 nb + n: Q^T operands (dims 32 k + 8 j4 .. + 7) and the keys each sees.
    int lim[NB];
    u32x4 qb[NB][KS];
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) {
      const int r = q0 + SET_ROWS * set + 16 * nb + n, pos = r / G;
      const bool in = r < qrows;
      lim[nb] = in ? lk - lq + pos + 1 : lk;
      const char* src = p.q + (int64_t)(tok + pos) * p.q_st + (int64_t)(wh * G + r - pos * G) * p.q_sh + 16 * j4;
#pragma unroll
      for (int k = 0; k < KS; ++k) qb[nb][k] = in ? ld16(src + 64 * k) : u32x4{0, 0, 0, 0};
    }
    const int all = lk - lq + q0 / G + 1;  // keys below it are seen by every query row of the pass
    float m[NB], l[NB];
    f32x4 o[NB][DB];
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) {
      m[nb] = -INFINITY;
      l[nb] = 0.f;
#pragma unroll
      for (int b = 0; b < DB; ++b) o[nb][b] = f32x4{0, 0, 0, 0};
    }
    // q in registers before the tile loads are counted.
#pragma unroll
    for (int nb = 0; nb < NB; ++nb)
#pragma unroll
      for (int k = 0; k < KS; ++k) asm volatile("" ::"v"(qb[nb][k]));
#pragma unroll
    for (int t = 0; t < kFewStages; ++t)
      if (t < nt) {
        locate(t);
        fill(t, p.k_cache, ring + t * kFewStage);
        fill(t, p.v_cache, ring + t * kFewStage + kFewHalf);
      }
    for (int t = 0; t < nt; ++t) {
      char* stage = ring + (t & 1) * kFewStage;
      const uint16_t* ks = reinterpret_cast<const uint16_t*>(stage);
      const uint16_t* vs = reinterpret_cast<const uint16_t*>(stage + kFewHalf);
      const bool next = t + 1 < nt, refill = t + 2 < nt;
      // In order of issue: keys t, values t, keys t + 1, values t + 1.
      if (next) few_wait<3 * kFewLoads>(); else few_wait<kFewLoads>();
      // S^T: s[kb][nb] lane holds keys t0 + 16 kb + 4 j4 + r of query row (nb, n).
      f32x4 s[KB][NB];
#pragma unroll
      for (int kb = 0; kb < KB; ++kb)
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) s[kb][nb] = f32x4{0, 0, 0, 0};
#pragma unroll
      for (int k = 0; k < KS; ++k)
#pragma unroll
        for (int kb = 0; kb < KB; ++kb) {
          const u32x4 a = *reinterpret_cast<const u32x4*>(ks + (16 * kb + n) * D + kpos[k]);
#pragma unroll
          for (int nb = 0; nb < NB; ++nb) s[kb][nb] = E::mfma16x16x32(a, qb[nb][k], s[kb][nb]);
        }
      if (refill) {
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // the keys are in registers
        locate(t + 2);
        fill(t + 2, p.k_cache, stage);
      }
      const int t0 = k0 + KT * WT * t;
      if (t0 + KT > all) {
#pragma unroll
        for (int kb = 0; kb < KB; ++kb)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const int k = t0 + 16 * kb + 4 * j4 + r;
#pragma unroll
            for (int nb = 0; nb < NB; ++nb) s[kb][nb][r] = k < lim[nb] ? s[kb][nb][r] : -INFINITY;
          }
      }
      float mx[NB];
      bool grow = false;
#pragma unroll
      for (int nb = 0; nb < NB; ++nb) {
        float x = vmax(vmax(s[0][nb][0], s[0][nb][1]), vmax(s[0][nb][2], s[0][nb][3]));
        if constexpr (KB == 2) x = vmax(x, vmax(vmax(s[1][nb][0], s[1][nb][1]), vmax(s[1][nb][2], s[1][nb][3])));
        mx[nb] = xor32_max(xor16_max(x));
        grow |= mx[nb] > m[nb] && (m[nb] == -INFINITY || (mx[nb] - m[nb]) * c > kRescaleSlack);
      }
      if (__any(grow)) {
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) {
          const float mn = vmax(m[nb], mx[nb]);
          const float alpha = m[nb] == -INFINITY ? 0.f : fast_exp2((m[nb] - mn) * c);
          m[nb] = mn;
          l[nb] *= alpha;
#pragma unroll
          for (int b = 0; b < DB; ++b) o[nb][b] *= alpha;
        }
      }
      // P^T operands: k slots 4 j4 .. + 3 (and, of 32 keys, 16 + 4 j4 .. + 3). Probabilities as a sum of two 16-bit
      // numbers, the second MFMA being free beside the stream: one alone would leave a rounding as large as the
      // output's (against 64 bits 2.3e-3 in bf16, where the VALU item, whose maxima are exactly 1, has 2.1e-3; so
      // 1.7e-3).
      uint32_t pb[NB][2 * KB], pl[NB][2 * KB];
#pragma unroll
      for (int nb = 0; nb < NB; ++nb) {
        const float mc = m[nb] == -INFINITY ? 0.f : m[nb] * c;  // no key seen yet: every score is -inf
#pragma unroll
        for (int kb = 0; kb < KB; ++kb) {
          float pr[4];
#pragma unroll
          for (int r = 0; r < 4; ++r) pr[r] = fast_exp2(fmaf(s[kb][nb][r], c, -mc));
          l[nb] += (pr[0] + pr[1]) + (pr[2] + pr[3]);
#pragma unroll
          for (int w = 0; w < 2; ++w) {
            const uint32_t hi = E::pack(pr[2 * w], pr[2 * w + 1]);
            pb[nb][2 * kb + w] = hi;
            pl[nb][2 * kb + w] = E::pack(pr[2 * w] - E::lo(hi), pr[2 * w + 1] - E::hi(hi));
          }
        }
      }
      if (refill) few_wait<3 * kFewLoads>(); else if (next) few_wait<2 * kFewLoads>(); else few_wait<0>();
      const uint16_t* vrow = vs + (4 * j4 + (n >> 2)) * D;
#pragma unroll
      for (int b = 0; b < DB; ++b) {
        const u32x2 lo = lds_read_tr16(vrow + vpos[b]);
        if constexpr (KB == 1) {
#pragma unroll
          for (int nb = 0; nb < NB; ++nb) {
            o[nb][b] = E::mfma16x16x16(lo, u32x2{pb[nb][0], pb[nb][1]}, o[nb][b]);
            o[nb][b] = E::mfma16x16x16(lo, u32x2{pl[nb][0], pl[nb][1]}, o[nb][b]);
          }
        } else {
          const u32x2 hi = lds_read_tr16(vrow + 16 * D + vpos[b]);
          const u32x4 a = {lo[0], lo[1], hi[0], hi[1]};
#pragma unroll
          for (int nb = 0; nb < NB; ++nb) {
            const u32x4 ph = {pb[nb][0], pb[nb][1], pb[nb][2 * KB - 2], pb[nb][2 * KB - 1]};
            const u32x4 pr = {pl[nb][0], pl[nb][1], pl[nb][2 * KB - 2], pl[nb][2 * KB - 1]};
            o[nb][b] = E::mfma16x16x32(a, ph, o[nb][b]);
            o[nb][b] = E::mfma16x16x32(a, pr, o[nb][b]);
          }
        }
      }
      if (refill) {
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // the values are in registers
        fill(t + 2, p.v_cache, stage + kFewHalf);
      }
    }

    // Merge the waves, 16 query rows at a time, through the rings' memory: wacc [wave][16][PITCH], wm / wl [wave][16].
    constexpr int PITCH = D + 4;
    float* wacc = reinterpret_cast<float*>(smem);
    float* wm = wacc + kWaves * 16 * PITCH;
    float* wl = wm + kWaves * 16;
    static_assert((kWaves * 16 * (PITCH + 2)) * 4 <= kWaves * kFewStages * kFewStage, "the merge fits the rings");
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) {
      if (q0 + 16 * nb >= qrows) break;
      __syncthreads();  // the rings (or the block before) are read
      const float ls = xor32_sum(xor16_sum(l[nb]));
#pragma unroll
      for (int b = 0; b < DB; ++b)
        *reinterpret_cast<f32x4*>(wacc + (wave * 16 + n) * PITCH + 16 * b + 4 * j4) = o[nb][b];
      if (j4 == 0) {
        wm[wave * 16 + n] = m[nb] * c;
        wl[wave * 16 + n] = ls;
      }
      __syncthreads();
      // Row i of this block of set w0, dims d0 .. d0 + N - 1 over its waves; returns the log2-sum-exp2.
      auto merge_waves = [&](int w0, int i, int d0, auto& x) {
        constexpr int N = sizeof(x) / sizeof(x[0]);
        float mmax = -INFINITY, den = 0.f;
#pragma unroll
        for (int w = w0; w < kWaves; w += NS) mmax = fmaxf(mmax, wm[w * 16 + i]);
#pragma unroll
        for (int e = 0; e < N; ++e) x[e] = 0.f;
        mmax = merge_base(mmax);
#pragma unroll
        for (int w = w0; w < kWaves; w += NS) {
          const float wt = fast_exp2(wm[w * 16 + i] - mmax);
          den += wt * wl[w * 16 + i];
#pragma unroll
          for (int e = 0; e < N; ++e) x[e] += wt * wacc[(w * 16 + i) * PITCH + d0 + e];
        }
        const float inv = inv_sum(den);
#pragma unroll
        for (int e = 0; e < N; ++e) x[e] *= inv;
        return mmax + fast_log2(den);  // no key seen: -inf
      };
      for (int i = threadIdx.x; i < NS * 16 * (D / 4); i += 64 * kWaves) {
        const int row16 = i / (D / 4), d0 = (i % (D / 4)) * 4, w0 = row16 / 16, ri = row16 % 16;
        const int r = q0 + SET_ROWS * w0 + 16 * nb + ri, pos = r / G;
        const int head = (kvh + (HP > 1 ? w0 : 0)) * G + r - pos * G;
        if (r >= qrows) continue;
        float x[4];
        const float lse = merge_waves(w0, ri, d0, x);
        if (nsplit <= 1) {
          *reinterpret_cast<u32x2*>(p.out + (int64_t)(tok + pos) * p.o_st + (int64_t)head * p.o_sh + d0 * 2) =
              u32x2{E::pack(x[0], x[1]), E::pack(x[2], x[3])};
        } else {
          const int64_t slot = (int64_t)(slot0 + split * lq + pos) * p.hq + head;
          coherent_store2(p.part_o + slot * D + d0, x[0], x[1]);
          coherent_store2(p.part_o + slot * D + d0 + 2, x[2], x[3]);
          if (d0 == 0) coherent_store(p.part_lse + slot, lse);
        }
      }
    }
    __syncthreads();  // before another pass refills the rings
  }
  if (nsplit <= 1) return;
  // The split that counts in last merges the row (as decode_item in paged_attention.hip).
  __shared__ int s_last;
  __builtin_amdgcn_s_waitcnt(0);
  __syncthreads();
  int32_t* count = p.merge_count + (row * p.hkv + kvh) / HP;
  if (threadIdx.x == 0)
    s_last = __hip_atomic_fetch_add(count, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == nsplit - 1;
  __syncthreads();
  if (!s_last) return;
  merge_item<T, D>(p, HP * qrows * (D / 2), lq, nsplit, [&](int i) {
    const int hr = i / (D / 2), h = hr / qrows, r = hr - h * qrows, pos = r / G;
    return MergePiece{slot0 + pos, tok + pos, (kvh + h) * G + r - pos * G, (i % (D / 2)) * 2};
  });
  if (threadIdx.x == 0) __hip_atomic_store(count, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

template <typename T, int D, int NB, FewSets SETS>
__global__ __launch_bounds__(64 * kWaves, 2) void few_list_kernel(AttnParams p) {
  __shared__ __attribute__((aligned(16))) char smem[kWaves * kFewStages * kFewStage];
  constexpr int HP = SETS == kTwoHeads ? 2 : 1;
  const int ny = p.hkv / HP, bx = blockIdx.x / ny, kh = blockIdx.x - bx * ny;
  const DecodeWork w = decode_work(p, bx);
  if (bx >= w.count) return;
  few_item<T, D, NB, SETS>(p, w.row, w.split, w.per, kh * HP, smem);
}

template <typename T, int D>
static void launch_rows(const AttnParams& p, int query_rows, int hp, int items, hipStream_t stream) {
  const dim3 grid(items * (p.hkv / hp)), block(64 * kWaves);
  if (query_rows > 32)
    hipLaunchKernelGGL((few_list_kernel<T, D, (D == 64 ? 4 : 2), (D == 64 ? kOneSet : kTwoBlocks)>), grid, block, 0,
                       stream, p);
  else if (query_rows > 16 && hp == 2)
    hipLaunchKernelGGL((few_list_kernel<T, D, 2, kTwoHeads>), grid, block, 0, stream, p);
  else if (query_rows > 16)
    hipLaunchKernelGGL((few_list_kernel<T, D, 2, kOneSet>), grid, block, 0, stream, p);
  else if (hp == 2)
    hipLaunchKernelGGL((few_list_kernel<T, D, 1, kTwoHeads>), grid, block, 0, stream, p);
  else
    hipLaunchKernelGGL((few_list_kernel<T, D, 1, kOneSet>), grid, block, 0, stream, p);
}

void launch_few_query(const AttnParams& p, int d, int query_rows, int hp, int dtype, int items, hipStream_t stream) {
  if (dtype == LV_DTYPE_BF16) {
    if (d == 64) launch_rows<BF16, 64>(p, query_rows, hp, items, stream);
    else launch_rows<BF16, 128>(p, query_rows, hp, items, stream);
  } else {
    if (d == 64) launch_rows<F16, 64>(p, query_rows, hp, items, stream);
    else launch_rows<F16, 128>(p, query_rows, hp, items, stream);
  }
}

}  // namespace lv
