// MLA absorbed decode on gfx950: each row's last queries attend its paged latents as one key head shared by all
// query heads; values are the latents' leading v_dim entries.
//
// Math of TorchAttention.mla_decode (lean_vllm/attention/torch_backend.py:105-119), called by
// MLAAttention._decode_latents (lean_vllm/layers/attention.py:319-335) with q = [q_nope W_UK_T | q_pe] of width
// 576 (kv_lora_rank 512 + rope 64) and v_dim 512: query j of a row with lq queries and L cached latents sees
// latents 0 .. L - lq + j.
//
// Two schedules, both streaming latents from HBM straight into an LDS ring (global_load_lds_dwordx4):
//   balanced runs (mla_run_kernel)  pages a multiple of 16 latents: the units' 32-latent stages, end to end, are cut
//                                   into equal runs, one per workgroup; units cut by run boundaries are merged by
//                                   log-sum-exp in mla_run_merge_kernel.
//   split schedule (mla_decode_dma_kernel)  other page sizes, or more units than the runs' in-kernel scan holds:
//                                   one workgroup per (row, split of <= 4096 latents, query, 16-head tile); split
//                                   rows are merged by log-sum-exp in mla_merge_kernel.
// Per 16 latents: S^T = Lat Q^T (16 latents x 16 columns, K = 576) on MFMA 16x16x32, the online softmax per
// column, and O^T += V^T P^T (512 dims) on MFMA 16x16x32 or 16x16x16 with V^T operands from gfx950's transposing LDS
// read (ds_read_b64_tr_b16).
#include <algorithm>

#include "lv_common.h"

namespace lv {

constexpr int kLatent = 576;              // latent width served: kv_lora_rank 512 + rope 64
constexpr int kVDim = 512;                // value width: the latents' leading entries
constexpr int kMlaPitch = kLatent + 16;   // LDS row pitch in elements (1184 bytes): conflict-free operand reads and
                                          // transposing reads (a 1168-byte pitch halves the latter's rate)
constexpr int kLatChunks = kLatent / 8;   // 16-byte chunks per latent row

constexpr int kMlaMaxSplit = 4096;        // latents per work item at most
constexpr int kMlaMaxBlocks = kMlaMaxSplit / 16 + 2;  // pages one work item touches at most (pages >= 16 latents)

constexpr int kMlaSplitStages = 4;    // ring depth of the split schedule
constexpr int kMlaSplitTarget = 4096;  // split-schedule items (x queries x head tiles) a grid aims for

struct MlaParams {
  const char* q;
  int64_t q_st, q_sh;  // bytes
  const char* cache;
  int64_t c_sb, c_st;  // bytes
  FastDiv bs;  // latents per page
  const int32_t* tables;
  int64_t t_stride;  // elements
  const int32_t* lens;
  int32_t rows, lq, heads, htiles;
  float scale_log2;
  char* out;
  int64_t o_st, o_sh;  // bytes
  int32_t split, max_splits;
  float* part_o;    // split schedule: [rows * lq][heads][max_splits][kVDim]; runs: [runs][2][16 NB][kVDim]
  float* part_lse;  // split schedule: [rows * lq][heads][max_splits]; runs: [runs][2][16 NB]; log2 domain
  int32_t units;    // runs: (row, tile of 16 NB (query, head) columns) units
  int32_t tiles;    // runs: units per row
  int32_t* prefix;  // runs: [units + 2] prefix of places over units, then their total and the run length
};

// ---------------------------------------------------------------------------------------------------------
// Split schedule: latents move from HBM straight into LDS (global_load_lds_dwordx4), a ring of kMlaSplitStages
// 16-latent stages with all but one in flight while one is consumed; no registers stage data. Each wave computes
// the stage's whole S^T (16 latents x 16 heads, K = 576) from LDS, then O^T for its 128 output dims with MFMA
// 16x16x16 whose V^T operands come from one transposing LDS read each. One unfenced barrier per stage; every wait
// on the stage loads is an explicit vmcnt.

constexpr int kDmaTile = 16;                            // latents per stage
constexpr int kDmaRowSlots = kLatChunks + 2;            // 16-byte slots per LDS row (two pad slots: pitch 1184 B)
constexpr int kDmaStageSlots = kDmaTile * kDmaRowSlots;  // 1184
constexpr int kDmaInstr = (kDmaStageSlots + 63) / 64;   // 64-lane loads per stage: 19, 5 per wave (4 for wave 3)
constexpr int kDmaStageElems = kDmaStageSlots * 8;
static_assert(kDmaRowSlots * 8 == kMlaPitch, "the slots make up the LDS row pitch");
static_assert(kDmaInstr == 19, "the stage waits count 5 loads for waves 0-2 and 4 for wave 3");

// Wait until at most `ahead` (<= 2) stages of this wave's loads (5 per stage, 4 for wave 3) are outstanding, then meet
// the other waves. No fence: the stage's LDS writes are exactly the loads waited for, and a fence would wait for
// the stages still in flight as well.
#define LV_WAIT_BARRIER(N) asm volatile("s_waitcnt vmcnt(" #N ")\n\ts_barrier" ::: "memory")
__device__ __forceinline__ void dma_stage_barrier(int ahead, int wave) {
  if (wave < 3) {
    switch (ahead) {
      case 0: LV_WAIT_BARRIER(0); break;
      case 1: LV_WAIT_BARRIER(5); break;
      default: LV_WAIT_BARRIER(10); break;
    }
  } else {
    switch (ahead) {
      case 0: LV_WAIT_BARRIER(0); break;
      case 1: LV_WAIT_BARRIER(4); break;
      default: LV_WAIT_BARRIER(8); break;
    }
  }
}
#undef LV_WAIT_BARRIER

// STAGES: ring depth (STAGES - 1 stages in flight while one is consumed; at most 4). ONE_PAGE: block_size is a
// multiple of 16, so a stage (16 latents starting at a multiple of 16) lies in one page: one page lookup per
// stage, every lane's load a fixed offset from it.
template <typename T, int STAGES, bool ONE_PAGE>
__global__ __launch_bounds__(256) void mla_decode_dma_kernel(MlaParams p) {
  static_assert(STAGES >= 2 && STAGES <= 4, "the stage waits cover up to three stages in flight");
  using E = Elem<T>;
  __shared__ __attribute__((aligned(16))) uint16_t ring[STAGES * kDmaStageElems];
  __shared__ int64_t page_off[kMlaMaxBlocks];
  const int row = blockIdx.x / p.max_splits, split = blockIdx.x % p.max_splits;
  const int qj = blockIdx.y / p.htiles, ht = blockIdx.y % p.htiles;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n = lane & 15, g = lane >> 4;

  const int lk = p.lens[row] - p.lq + qj + 1;  // latents this query sees
  const int kbeg = split * p.split;
  if ((split > 0 && kbeg >= lk) || split >= p.max_splits) return;
  const int kend = min(lk, kbeg + p.split);
  const int nsplit = lk > 0 ? min((lk + p.split - 1) / p.split, p.max_splits) : 0;
  const int tokq = row * p.lq + qj;
  const int head = ht * 16 + n;
  const bool hvalid = head < p.heads;
  const float c = p.scale_log2;

  // Q^T operand over the whole latent: lane holds dims 32 s + 8 g .. + 7 of head n.
  u32x4 qb[18];
  {
    const char* qrow = p.q + tokq * p.q_st + (int64_t)head * p.q_sh;
#pragma unroll
    for (int s = 0; s < 18; ++s) qb[s] = hvalid ? ld16(qrow + (int64_t)(32 * s + 8 * g) * 2) : u32x4{0, 0, 0, 0};
  }
  const int page0 = kend > kbeg ? (int)p.bs.div(kbeg) : 0;
  const int npages = kend > kbeg ? (int)p.bs.div(kend - 1) - page0 + 1 : 0;
  {
    const int32_t* table = p.tables + (int64_t)row * p.t_stride + page0;
    for (int i = tid; i < npages; i += 256) page_off[i] = (int64_t)table[i] * p.c_sb;
  }
  // This wave's loads j = wave + 4 i (i < 5) of a stage's 19: slot 64 j + lane is 16-byte chunk `part` of latent
  // row r of the stage. Slots 74 r + 72 and 74 r + 73 of row r are LDS padding, filled with copies of chunk 71.
  int lrow[5], lpart[5];
#pragma unroll
  for (int i = 0; i < 5; ++i) {
    const int slot = min(64 * (wave + 4 * i) + lane, kDmaStageSlots - 1);
    lrow[i] = slot / kDmaRowSlots;
    lpart[i] = min(slot - lrow[i] * kDmaRowSlots, kLatChunks - 1) * 16;
  }
  __builtin_amdgcn_s_waitcnt(0xF70);  // vmcnt(0): q is in registers before the stage loads are counted
  __syncthreads();

  // Stage load of latents t0 .. t0 + 15; latents at or past kend load a latent of the range instead (finite
  // values; their weight is 0).
  auto fill = [&](int t0, uint16_t* stage) {
    const int last = kend - 1 - t0;  // rows past it are clamped
    int64_t base = 0;
    if (ONE_PAGE) {
      const int pg = (int)p.bs.div(t0);
      const int64_t po = page_off[pg - page0];
      // Uniform: move it to scalar registers. The low half is widened unsigned (offsets reach past 2 GiB).
      base = (int64_t)((uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)po) |
                       ((uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(po >> 32)) << 32));
      base += (int64_t)(t0 - pg * (int)p.bs.d) * p.c_st;
    }
#pragma unroll
    for (int i = 0; i < 5; ++i) {
      const int j = wave + 4 * i;
      if (j < kDmaInstr && 64 * j + lane < kDmaStageSlots) {
        const int r = min(lrow[i], last);
        if (ONE_PAGE) {
          lds_dma16(p.cache + base, (uint32_t)(r * (int)p.c_st + lpart[i]), lds_addr(stage + 64 * 8 * j));
        } else {
          const int tok = t0 + r;
          const int pg = (int)p.bs.div(tok);
          lds_dma16(p.cache + page_off[pg - page0] + (int64_t)(tok - pg * (int)p.bs.d) * p.c_st + lpart[i],
                    lds_addr(stage + 64 * 8 * j));
        }
      }
    }
  };

  float m = -INFINITY, lsum = 0.f;
  f32x4 o[8];
#pragma unroll
  for (int j = 0; j < 8; ++j) o[j] = f32x4{0, 0, 0, 0};

  const int ntiles = kend > kbeg ? (kend - kbeg + kDmaTile - 1) / kDmaTile : 0;
  for (int t = 0; t < STAGES - 1 && t < ntiles; ++t) fill(kbeg + t * kDmaTile, ring + t * kDmaStageElems);
  for (int it = 0; it < ntiles; ++it) {
    const int t0 = kbeg + it * kDmaTile;
    dma_stage_barrier(min(STAGES - 2, ntiles - 1 - it), wave);  // stage `it` has landed for every wave
    const bool refill = it + STAGES - 1 < ntiles;
    // Refill the stage read last iteration (every wave has passed the barrier, so its reads are done), then
    // consume this one.
    auto step = [&](uint16_t* next, const uint16_t* stage) {
      if (refill) fill(t0 + (STAGES - 1) * kDmaTile, next);
      f32x4 sc = {0, 0, 0, 0};  // latents t0 + 4 g + r of head n
      const uint16_t* arow = stage + n * kMlaPitch + 8 * g;
#pragma unroll
      for (int s = 0; s < 18; ++s) sc = E::mfma16x16x32(*reinterpret_cast<const u32x4*>(arow + 32 * s), qb[s], sc);
      if (t0 + kDmaTile > kend) {
#pragma unroll
        for (int r = 0; r < 4; ++r) sc[r] = t0 + 4 * g + r < kend ? sc[r] : -INFINITY;
      }
      float mx = vmax(vmax(sc[0], sc[1]), vmax(sc[2], sc[3]));
      mx = xor32_max(xor16_max(mx));
      if (__any(mx > m && (m == -INFINITY || (mx - m) * c > kRescaleSlack))) {
        const float mn = vmax(m, mx);
        const float alpha = m == -INFINITY ? 0.f : fast_exp2((m - mn) * c);
        m = mn;
        lsum *= alpha;
#pragma unroll
        for (int j = 0; j < 8; ++j) o[j] *= alpha;
      }
      const float mc = m * c;
      float pr[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) pr[r] = fast_exp2(fmaf(sc[r], c, -mc));
      lsum += (pr[0] + pr[1]) + (pr[2] + pr[3]);
      const u32x2 pb = {E::pack(pr[0], pr[1]), E::pack(pr[2], pr[3])};
      const uint16_t* v = stage + (4 * g + (n >> 2)) * kMlaPitch + 128 * wave + 4 * (n & 3);
#pragma unroll
      for (int j = 0; j < 8; ++j) o[j] = E::mfma16x16x16(lds_read_tr16(v + 16 * j), pb, o[j]);
    };
    step(ring + ((it + STAGES - 1) % STAGES) * kDmaStageElems, ring + (it % STAGES) * kDmaStageElems);
  }

  lsum = xor32_sum(xor16_sum(lsum));
  if (!hvalid) return;
  const float inv = lsum > 0.f ? 1.f / lsum : 0.f;
  if (nsplit <= 1) {
    char* dst = p.out + tokq * p.o_st + (int64_t)head * p.o_sh;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const int d = 128 * wave + 16 * j + 4 * g;
      const u32x2 v = {E::pack(o[j][0] * inv, o[j][1] * inv), E::pack(o[j][2] * inv, o[j][3] * inv)};
      *reinterpret_cast<u32x2*>(dst + d * 2) = v;
    }
  } else {
    const int64_t slot = ((int64_t)tokq * p.heads + head) * p.max_splits + split;
    float* dst = p.part_o + slot * kVDim;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const int d = 128 * wave + 16 * j + 4 * g;
      *reinterpret_cast<f32x4*>(dst + d) = o[j] * inv;
    }
    if (wave == 0 && g == 0) p.part_lse[slot] = lsum > 0.f || lsum != lsum ? m * c + fast_log2(lsum) : -INFINITY;
  }
}

// ---------------------------------------------------------------------------------------------------------
// Balanced schedule over equal runs of stages, for pages whose size is a multiple of 16 latents.
//
// A row's columns are its (query j, head) pairs, c = j * heads + head. Unit u = (row, tile of 16 NB columns), u = row
// * tiles + tile, needs T_u = ceil(L_u / 32) stages of 32 latents (L_u: the latents its last query sees; a column of
// an earlier query masks its last ones), and kRunEnter more places ahead of them for its queries and its output,
// which cost a run about as much. Laid end to end (prefix P_u) the units' stages are cut into equal runs, one per
// workgroup of a grid that fills the GPU once; every workgroup streams its run through an LDS ring, each unit it
// enters preceded by a stage holding that unit's query rows. A unit that lies wholly inside one run is finished in
// place. A unit cut by run boundaries leaves (o / l, log2 l + m) per column in slot 0 (the run's first unit) or slot
// 1 (its last unit) of every run it touches, and mla_run_merge_kernel combines them; that kernel also writes the zero
// output of columns that see no latents. Every run does equal work, whatever the spread of row lengths, and partials
// are written only where a row crosses a run boundary.
//
// NB is 1 for rows of up to 16 columns, else 2: drafts and heads past 16 share the latents that a workgroup has in LDS
// instead of streaming them again. (Four blocks spill: 64 heads 1047 us against 458.)
//
// One workgroup of 8 waves per CU, a ring of three 36 KB stages, two in flight. Wave (lb, cb) of the first 2 NB
// computes the scores of 16 latents for 16 columns over the whole K = 576 (its Q^T in registers) and leaves their
// probabilities in LDS as the P^T operand; the other waves meanwhile issue the stage loads; after a barrier every
// wave adds P.V for 64 of the 512 output dims and all columns, V^T from the transposing read. Two barriers per 32
// latents. The max of a column is shared: a score past it by more than kRescaleSlack makes the workgroup take the
// stage's maxima from LDS, rescale and write the probabilities again (rare: the first stage of a unit, seldom
// another).
//
// Bound by HBM up to 32 columns (a build without the scores and P.V streams 128 rows of 1024-16384 latents in 201 us,
// 6.55 TB/s; the scores' serial chain through LDS and the two barriers are what is left). Against the schedule
// before, two workgroups of 4 waves per CU with a 16-latent stage each, every query and every 16 heads a unit of
// their own: 128 rows, 16 heads 216 us (215.4), 32 heads 229 (426), 64 heads 454 (850), 128 heads 890 (1670); two
// layers of 20 rows, 1024-8192 latents, 16 heads, 2 queries 73 us (108), 3 queries 104 (138), 128 heads 171 (298); 4
// rows 57 (70).

constexpr int kRunTile = 32;         // latents per stage
constexpr int kRunEnter = 3;         // places of a unit's start (0 / 1 / 2 / 3: 60 rows 136.6 / 135.1 / 134.4 / 133.2
                                     // us, 128 rows 217.5 / 216.4 / 216.9 / 216.0, within the spread of runs)
constexpr int kRunMin = 4;           // places per run at least (past a unit's start)
constexpr int kRunStages = 3;        // ring depth (four stream no faster)
constexpr int kRunWaves = 8;
constexpr int kRunsPerCU = 1;        // run workgroups per CU
enum : int { kGrow = 1, kUnseen = 2 };
constexpr int kRunMaxUnits = 8192;   // units the in-kernel scan serves
constexpr int kRunRow = kLatent;     // LDS row pitch in elements: no padding, 16-byte chunk c of row r at c ^ (r & 6),
                                     // so that operand and transposing reads meet no bank conflicts
constexpr int kRunElems = kRunTile * kRunRow;
constexpr int kRunLoads = kRunTile * kLatChunks / 64;  // 64-lane loads per stage, 18 per 16 rows

// At most N of this wave's loads outstanding and its LDS reads of the stage before done; then the other waves' are.
template <int N>
__device__ __forceinline__ void run_wait() {
  asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(N) : "memory");
}

// Latents that the last query of unit u = (row, tile) sees, from the row's cached latents.
template <int NB>
__device__ __forceinline__ int unit_latents(const MlaParams& p, int tile, int len) {
  const int last = min((tile + 1) * 16 * NB, p.lq * p.heads) - 1;  // the unit's last column
  return len - p.lq + last / p.heads + 1;
}

// Places of a unit of lk latents in the runs; none without latents.
__device__ __forceinline__ int stage_places(int lk) {
  return lk > 0 ? (lk + kRunTile - 1) / kRunTile + kRunEnter : 0;
}
template <int NB>
__device__ __forceinline__ int unit_places(const MlaParams& p, int u) {
  const int row = u / p.tiles;
  return stage_places(unit_latents<NB>(p, u - row * p.tiles, p.lens[row]));
}

// Position in a run's stage sequence: unit u (first stage at place pu, tu stages, lk latents), next tile t (-1: its
// queries). The unit's row and column tile and its block-table row are kept here, so a stage's loads need no division.
struct RunCursor {
  int u, pu, tu, lk, t;
  int row, len, tile, pg[2];
  const int32_t* table;
  const char* page[2];  // cache pages pg[] of the last stage's two blocks
  bool done;
};

template <typename T, int NB>
__global__ __launch_bounds__(64 * kRunWaves, 2) void mla_run_kernel(MlaParams p) {
  using E = Elem<T>;
  constexpr int W = kRunWaves, LB = kRunTile / 16;  // 16-latent blocks of a stage
  constexpr int DB = kVDim / 16 / W;                // 16-dim output blocks per wave
  constexpr int SW = LB * NB;                       // waves that compute scores
  // The other waves load the stages: their cursor and address work runs beside the scores.
  constexpr int LW = W - SW;
  constexpr int kPer = kRunLoads / LW;              // loads per stage
  static_assert(kPer * LW == kRunLoads && kRunStages == 3, "as many for each; one stage ahead of the awaited one");
  static_assert(SW < W && LB == 2 && NB <= LB, "waves for scores and loads; a stage holds a unit's query rows");
  __shared__ __attribute__((aligned(16))) uint16_t ring[kRunStages * kRunElems];
  __shared__ u32x2 s_p[NB][LB][64];      // P^T operands of the stage
  __shared__ float s_max[NB][LB][16];    // its maxima
  __shared__ float s_sum[NB][LB][16];    // row sums at a unit's end
  __shared__ int s_state[8];             // what its score waves found: kGrow, kUnseen
  __shared__ int wave_tot[W];
  __shared__ int first[3];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n = lane & 15, g = lane >> 4;
  const float c = p.scale_log2;
  const int lb = wave % LB, cb = wave / LB;  // the scores this wave computes (wave < SW)
  const int columns = p.lq * p.heads;

  // Places over units; thread tid sums units [ulo, uhi). Exclusive scan of those sums across the block.
  const int per_thread = (p.units + 64 * W - 1) / (64 * W);
  const int ulo = min(tid * per_thread, p.units), uhi = min(ulo + per_thread, p.units);
  int local = 0, len0 = 0;  // len0: latents of unit ulo's row
  for (int u = ulo; u < uhi; ++u) {
    const int row = u / p.tiles, len = p.lens[row];
    const int lk = unit_latents<NB>(p, u - row * p.tiles, len);
    local += stage_places(lk);
    len0 = u == ulo ? len : len0;
  }
  const int x = wave_incl_scan(local);
  if (lane == 63) wave_tot[wave] = x;
  if (tid < 8) s_state[tid] = 0;
  __syncthreads();
  int excl = x - local, total = 0;
#pragma unroll
  for (int w = 0; w < W; ++w) {
    excl += w < wave ? wave_tot[w] : 0;
    total += wave_tot[w];
  }
  total = __builtin_amdgcn_readfirstlane(total);
  const int per = max((total + (int)gridDim.x - 1) / (int)gridDim.x, kRunMin);
  if (blockIdx.x == 0) {  // the prefix, for the merge
    int run = excl;
    for (int u = ulo; u < uhi; ++u) {
      p.prefix[u] = run;
      run += unit_places<NB>(p, u);
    }
    if (tid == 0) {
      p.prefix[p.units] = total;
      p.prefix[p.units + 1] = per;
    }
  }
  const int start = blockIdx.x * per;
  if (start >= total) return;
  const int end = min(start + per, total);
  if (local > 0 && excl <= start && start < excl + local) {
    int u = ulo, acc = excl;
    if (per_thread > 1)
      for (int tu = unit_places<NB>(p, u); acc + tu <= start; tu = unit_places<NB>(p, u)) {
        acc += tu;
        ++u;
      }
    first[0] = u;
    first[1] = acc;
    first[2] = u == ulo ? len0 : p.lens[u / p.tiles];
  }
  __syncthreads();

  // Both cursors walk the same sequence: for each unit, its query stage, then its tiles inside [start, end).
  auto enter = [&](RunCursor& r, int u, int pu, int len = -1) {
    for (;; ++u) {  // units without latents hold no stages
      r.row = u / p.tiles;
      r.tile = u - r.row * p.tiles;
      r.len = len >= 0 ? len : sload(p.lens + r.row);
      r.lk = unit_latents<NB>(p, r.tile, r.len);
      if (r.lk > 0) break;
    }
    r.u = u;
    r.pu = pu + kRunEnter;
    r.tu = (r.lk + kRunTile - 1) / kRunTile;
    r.t = -1;
    r.table = p.tables + (int64_t)r.row * p.t_stride;
    r.pg[0] = r.pg[1] = -1;
    r.done = false;
  };
  auto advance = [&](RunCursor& r) {
    if (r.t < 0) {
      r.t = max(start, r.pu) - r.pu;
    } else if (r.pu + r.t + 1 == end) {
      r.done = true;
    } else if (r.t + 1 == r.tu) {
      if (r.pu + r.tu + kRunEnter >= end) r.done = true;  // the next unit's stages lie past the run
      else enter(r, r.u + 1, r.pu + r.tu);
    } else {
      ++r.t;
    }
  };
  RunCursor prod, cons;
  enter(prod, __builtin_amdgcn_readfirstlane(first[0]), __builtin_amdgcn_readfirstlane(first[1]),
        __builtin_amdgcn_readfirstlane(first[2]));
  cons = prod;

  // Loader wave lw's loads j = lw + LW i of a stage's 36: each lies in 16-row block j / 18, slot 64 (j % 18) + lane
  // of it holding position slot % 72 of its row slot / 72, so the chunk that belongs there.
  const bool loader = wave >= SW;
  const int lw = loader ? wave - SW : 0;
  // Whether load i of this wave lies in the second block: known for most i, whatever the wave.
  auto second = [&](int i) {
    return LW * i >= kRunLoads / LB || (LW * i + LW > kRunLoads / LB && lw >= kRunLoads / LB - LW * i);
  };
  int lrow[kPer], lchunk[kPer];
#pragma unroll
  for (int i = 0; i < kPer; ++i) {
    const int slot = 64 * ((lw + LW * i) % (kRunLoads / LB)) + lane;
    lrow[i] = slot / kLatChunks;
    lchunk[i] = ((slot - lrow[i] * kLatChunks) ^ (lrow[i] & 6)) * 16;
  }
  // Query stage: the 32 columns from the unit's first (columns past the row's last load the last; unused).
  // Latent stage: latents t0 .. t0 + 31 of the row, each 16 in one page (the page size is a multiple of 16); latents at
  // or past lk load latent lk - 1 instead (finite values; their weight is 0).
  auto fill = [&](RunCursor& r, uint16_t* stage) {
    if (r.t < 0) {
      const int c0 = r.tile * NB * 16;
#pragma unroll
      for (int i = 0; i < kPer; ++i) {
        const int j = lw + LW * i;
        const int col = min(c0 + (second(i) ? 16 : 0) + lrow[i], columns - 1), qj = col / p.heads;
        lds_dma16(p.q + (int64_t)(r.row * p.lq + qj) * p.q_st + (int64_t)(col - qj * p.heads) * p.q_sh + lchunk[i],
                  lds_addr(stage + 64 * 8 * j));
      }
    } else {
      const int t0 = r.t * kRunTile;
      const int s0 = t0, s1 = min(t0 + 16, r.lk - 1);  // first latent of either block
      const int g0 = (int)p.bs.div(s0), g1 = (int)p.bs.div(s1);
      if (g0 != r.pg[0] || g1 != r.pg[1]) {
        const int32_t* const where[2] = {r.table + g0, r.table + g1};
        int page[2];
        sload_n<2>(where, page);
        r.pg[0] = g0;
        r.pg[1] = g1;
        r.page[0] = p.cache + (int64_t)page[0] * p.c_sb;
        r.page[1] = p.cache + (int64_t)page[1] * p.c_sb;
      }
      const char* b0 = r.page[0] + (int64_t)(s0 - g0 * (int)p.bs.d) * p.c_st;
      const char* b1 = r.page[1] + (int64_t)(s1 - g1 * (int)p.bs.d) * p.c_st;
      const int last0 = r.lk - 1 - s0, last1 = r.lk - 1 - s1;
#pragma unroll
      for (int i = 0; i < kPer; ++i) {
        const int j = lw + LW * i;
        lds_dma16(second(i) ? b1 : b0, (uint32_t)(min(lrow[i], second(i) ? last1 : last0) * (int)p.c_st + lchunk[i]),
                  lds_addr(stage + 64 * 8 * j));
      }
    }
  };

  // Element offsets of this lane's operand reads: scores, k-steps of even and odd index (latent row n, chunk 4 k + g);
  // values, output block j (latent rows 4 g + n / 4 (+ 16), dims 64 wave + 16 j + 4 (n % 4)).
  const int kpos[2] = {n * kRunRow + 8 * (g ^ (n & 6)), n * kRunRow + 8 * ((4 + g) ^ (n & 6))};
  int vpos[DB];
#pragma unroll
  for (int j = 0; j < DB; ++j) {
    const int r = 4 * g + (n >> 2), chunk = 2 * DB * wave + 2 * j + ((n & 3) >> 1);
    vpos[j] = r * kRunRow + 8 * (chunk ^ (r & 6)) + 4 * (n & 1);
  }

  u32x4 qb[18];  // Q^T operand: lane holds dims 32 k + 8 g .. + 7 of column n of block cb
  int sees = 0;  // latents that column sees
  int later = 0;  // latents that the unit's first query does not see and its last does
  float m[NB], lsum = 0.f;
  f32x4 o[NB][DB];
  int issued = 0;
  for (; loader && issued < kRunStages - 1 && !prod.done; ++issued) {
    fill(prod, ring + issued * kRunElems);
    advance(prod);
  }
  for (int k = 0; !cons.done; ++k) {
    // Stage k has landed for every wave (one that loads nothing meets the barrier).
    const int ahead = issued - k - 1;
    if (!loader) run_wait<63>();
    else if (ahead <= 0) run_wait<0>();
    else run_wait<kPer>();
    // Refill the slot read last iteration (every wave has passed the barrier, so its reads are done).
    auto refill = [&] {
      if (!loader || prod.done) return;
      fill(prod, ring + (issued % kRunStages) * kRunElems);
      advance(prod);
      ++issued;
    };
    // With the value reads below before it, one column block: 128 rows of 16 heads 207.7 -> 205.0 us, 60 rows 98.2 ->
    // 97.1, 256 shorter rows 121.8 -> 120.9, 20 rows 30.2 -> 30.4; after it, two column blocks: 77.8 -> 74.8.
    constexpr bool kValuesFirst = NB == 1;
    if (cons.t < 0 || !kValuesFirst) refill();
    const uint16_t* stage = ring + (k % kRunStages) * kRunElems;
    if (cons.t < 0) {
      later = cons.lk - cons.len + p.lq - 1 - (cons.tile > 0 ? cons.tile * NB * 16 / p.heads : 0);
      if (wave < SW) {
        const uint16_t* qs = stage + cb * 16 * kRunRow;
#pragma unroll
        for (int s = 0; s < 18; ++s) qb[s] = *reinterpret_cast<const u32x4*>(qs + kpos[s & 1] + 64 * (s >> 1));
        const int col = min((cons.tile * NB + cb) * 16 + n, columns - 1);
        sees = cons.len - p.lq + col / p.heads + 1;
        lsum = 0.f;
      }
#pragma unroll
      for (int nb = 0; nb < NB; ++nb) {
        m[nb] = -INFINITY;
#pragma unroll
        for (int j = 0; j < DB; ++j) o[nb][j] = f32x4{0, 0, 0, 0};
      }
      advance(cons);
      continue;
    }
    f32x4 sc = {0, 0, 0, 0};  // latents t0 + 16 lb + 4 g + r of column n
    float mc = 0.f, psum = 0.f;
    const int t0 = cons.t * kRunTile;
    // Probabilities of the wave's scores under the column's max, to LDS.
    auto put_probabilities = [&] {
      float pr[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) pr[r] = fast_exp2(fmaf(sc[r], c, -mc));
      psum = (pr[0] + pr[1]) + (pr[2] + pr[3]);
      s_p[cb][lb][lane] = u32x2{E::pack(pr[0], pr[1]), E::pack(pr[2], pr[3])};
    };
    auto own_max = [&] {
      float x = m[0];
#pragma unroll
      for (int nb = 1; nb < NB; ++nb) x = cb == nb ? m[nb] : x;
      return x;
    };
    // The stage's V^T operands wait for nobody; a wave with scores reads them after those.
    u32x4 va[DB];
    auto read_values = [&] {
#pragma unroll
      for (int j = 0; j < DB; ++j) {
        const u32x2 lo = lds_read_tr16(stage + vpos[j]), hi = lds_read_tr16(stage + 16 * kRunRow + vpos[j]);
        va[j] = u32x4{lo[0], lo[1], hi[0], hi[1]};
      }
    };
    if (wave >= SW) {
      read_values();
      if (kValuesFirst) refill();
    }
    if (wave < SW) {
      const uint16_t* rows = stage + lb * 16 * kRunRow;
      f32x4 sd = {0, 0, 0, 0};  // two chains
#pragma unroll
      for (int s = 0; s < 18; s += 2) {
        sc = E::mfma16x16x32(*reinterpret_cast<const u32x4*>(rows + kpos[0] + 32 * s), qb[s], sc);
        sd = E::mfma16x16x32(*reinterpret_cast<const u32x4*>(rows + kpos[1] + 32 * s), qb[s + 1], sd);
      }
      // Six operands read ahead of the MFMAs (left alone, the compiler waits for each read in turn).
      __builtin_amdgcn_sched_group_barrier(0x100, 6, 0);
#pragma unroll
      for (int s = 0; s < 6; ++s) {
        __builtin_amdgcn_sched_group_barrier(0x008, 2, 0);
        __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
      }
      __builtin_amdgcn_sched_group_barrier(0x008, 6, 0);
      sc += sd;
      bool unseen = false;  // a latent that the column does not see is no number (then its score is none)
      if (t0 + kRunTile > cons.lk - (p.lq - 1)) {  // else every column sees the stage
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const bool in = t0 + 16 * lb + 4 * g + r < sees;
          unseen |= !in && !__builtin_isfinite(sc[r]);
          sc[r] = in ? sc[r] : -INFINITY;
        }
      }
      float mx = vmax(vmax(sc[0], sc[1]), vmax(sc[2], sc[3]));
      mx = xor32_max(xor16_max(mx));
      const float mo = own_max();
      const bool grow = mx > mo && (mo == -INFINITY || (mx - mo) * c > kRescaleSlack);
      mc = mo == -INFINITY ? 0.f : mo * c;
      if (g == 0) s_max[cb][lb][n] = mx;
      const bool grows = __any(grow), drafts = __any(unseen);
      if (lane == 0) s_state[wave] = (grows ? kGrow : 0) | (drafts ? kUnseen : 0);
      if (!grows) put_probabilities();
      read_values();
    }
    // LDS only: the stage loads in flight are not waited for.
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    int state = 0;
#pragma unroll
    for (int w = 0; w < SW; ++w) state |= s_state[w];
    state = __builtin_amdgcn_readfirstlane(state);  // the same in every wave
    u32x4 pb[NB];
    auto get_probabilities = [&] {
#pragma unroll
      for (int nb = 0; nb < NB; ++nb) {
        const u32x2 lo = s_p[nb][0][lane], hi = s_p[nb][1][lane];
        pb[nb] = u32x4{lo[0], lo[1], hi[0], hi[1]};
      }
    };
    get_probabilities();
    if (state & kGrow) {
#pragma unroll
      for (int nb = 0; nb < NB; ++nb) {
        const float mn = vmax(m[nb], vmax(s_max[nb][0][n], s_max[nb][1][n]));
        const float alpha = m[nb] == -INFINITY ? 0.f : fast_exp2((m[nb] - mn) * c);
        m[nb] = mn;
        if (cb == nb) lsum *= alpha;
#pragma unroll
        for (int j = 0; j < DB; ++j) o[nb][j] *= alpha;
      }
      if (wave < SW) {
        const float mo = own_max();
        mc = mo == -INFINITY ? 0.f : mo * c;  // a column that has seen no latent
        put_probabilities();
      }
      asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
      get_probabilities();
    }
    lsum += psum;
    // Latents from `common` on are drafts that the unit's first query does not see. Its weights there are 0, but a
    // value that is no number would reach its sums all the same: where a stage has one, such latents are left out of
    // the product and added to the columns that see them one by one.
    const int common = cons.lk - later;
    if (state & kUnseen) {
#pragma unroll
      for (int w = 0; w < 4; ++w) {  // word w of an operand: latents t0 + 16 (w / 2) + 4 g + 2 (w % 2) and the next
        const int t = t0 + 16 * (w >> 1) + 4 * g + 2 * (w & 1);
        const uint32_t keep = t + 1 < common ? 0xffffffffu : t < common ? 0xffffu : 0u;
#pragma unroll
        for (int j = 0; j < DB; ++j) va[j][w] &= keep;
      }
    }
#pragma unroll
    for (int j = 0; j < DB; ++j)
#pragma unroll
      for (int nb = 0; nb < NB; ++nb) o[nb][j] = E::mfma16x16x32(va[j], pb[nb], o[nb][j]);
    if (state & kUnseen) {
      for (int t = max(t0, common); t < min(t0 + kRunTile, cons.lk); ++t) {
        const int r = t - t0;
        // Its first column in the tile: query t - (len - lq) is the first to see it.
        const int c0 = (t - cons.len + p.lq) * p.heads - cons.tile * NB * 16;
#pragma unroll
        for (int j = 0; j < DB; ++j) {
          const int chunk = 2 * DB * wave + 2 * j + (g >> 1);  // dims 16 DB wave + 16 j + 4 g .. + 3
          const u32x2 v = *reinterpret_cast<const u32x2*>(stage + r * kRunRow + 8 * (chunk ^ (r & 6)) + 4 * (g & 1));
#pragma unroll
          for (int nb = 0; nb < NB; ++nb) {
            const uint32_t pair = s_p[nb][r >> 4][n + 4 * (r & 12)][(r >> 1) & 1];
            const float pr = r & 1 ? E::hi(pair) : E::lo(pair);
            if (16 * nb + n >= c0)
              o[nb][j] += f32x4{pr * E::lo(v[0]), pr * E::hi(v[0]), pr * E::lo(v[1]), pr * E::hi(v[1])};
          }
        }
      }
    }

    if (cons.t + 1 == cons.tu || cons.pu + cons.t + 1 == end) {  // the unit's last stage in this run
      const bool whole = cons.pu >= start && cons.pu + cons.tu <= end;
      if (wave < SW) {
        const float l = xor32_sum(xor16_sum(lsum));
        if (g == 0) s_sum[cb][lb][n] = l;
      }
      asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
#pragma unroll
      for (int nb = 0; nb < NB; ++nb) {
        const int col = (cons.tile * NB + nb) * 16 + n;
        if (col >= columns) continue;
        const float l = s_sum[nb][0][n] + s_sum[nb][1][n];
        const float inv = inv_sum(l);  // 0: an earlier query sees none of the run's latents
        if (whole) {
          const int qj = col / p.heads;
          char* dst = p.out + (int64_t)(cons.row * p.lq + qj) * p.o_st + (int64_t)(col - qj * p.heads) * p.o_sh;
#pragma unroll
          for (int j = 0; j < DB; ++j) {
            const int d = 16 * DB * wave + 16 * j + 4 * g;
            const u32x2 val = {E::pack(o[nb][j][0] * inv, o[nb][j][1] * inv),
                               E::pack(o[nb][j][2] * inv, o[nb][j][3] * inv)};
            *reinterpret_cast<u32x2*>(dst + d * 2) = val;
          }
        } else {
          const int slot = (blockIdx.x * 2 + (cons.pu - kRunEnter <= start ? 0 : 1)) * 16 * NB + 16 * nb + n;
          float* dst = p.part_o + (int64_t)slot * kVDim;
#pragma unroll
          for (int j = 0; j < DB; ++j) {
            const int d = 16 * DB * wave + 16 * j + 4 * g;
            *reinterpret_cast<f32x4*>(dst + d) = o[nb][j] * inv;
          }
          if (wave == 0 && g == 0) p.part_lse[slot] = l > 0.f || l != l ? m[nb] * c + fast_log2(l) : -INFINITY;
        }
      }
    }
    advance(cons);
  }
}

// Finish units cut by run boundaries (log-sum-exp over the runs that touched them) and zero the output of units
// that see no latents; units finished in place are left alone. Block (unit, four columns of its tile), one wave each.
template <typename T, int NB>
__global__ __launch_bounds__(256) void mla_run_merge_kernel(MlaParams p) {
  using E = Elem<T>;
  const int u = blockIdx.x, lane = threadIdx.x & 63;
  const int h = blockIdx.y * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int row = u / p.tiles, col = (u - row * p.tiles) * 16 * NB + h;
  if (col >= p.lq * p.heads) return;
  const int qj = col / p.heads, tq = row * p.lq + qj, head = col - qj * p.heads;
  const int at = p.prefix[u], pu = at + kRunEnter, tu = p.prefix[u + 1] - pu, per = p.prefix[p.units + 1];
  constexpr int PER = kVDim / 64;
  float o[PER];
#pragma unroll
  for (int e = 0; e < PER; ++e) o[e] = 0.f;
  if (tu > 0) {
    const int b0 = pu / per, b1 = (pu + tu - 1) / per;
    if (b0 == b1) return;
    // The runs' partials, kRunMergeBatch at a time with every load of a batch issued before the first is used;
    // the max and the sums carry from batch to batch.
    constexpr int kRunMergeBatch = 8;
    float m = -INFINITY, den = 0.f;
    for (int c0 = b0; c0 <= b1; c0 += kRunMergeBatch) {
      float ls[kRunMergeBatch];
      f32x4 x[kRunMergeBatch][PER / 4];
#pragma unroll
      for (int i = 0; i < kRunMergeBatch; ++i) {
        const int b = c0 + i;
        ls[i] = -INFINITY;
#pragma unroll
        for (int e = 0; e < PER / 4; ++e) x[i][e] = f32x4{0, 0, 0, 0};
        if (b <= b1) {  // wave-uniform
          const int slot = (b * 2 + (b == b0 && at > b0 * per ? 1 : 0)) * 16 * NB + h;
          ls[i] = p.part_lse[slot];
          const f32x4* src = reinterpret_cast<const f32x4*>(p.part_o + (int64_t)slot * kVDim + lane * PER);
#pragma unroll
          for (int e = 0; e < PER / 4; ++e) x[i][e] = src[e];
        }
      }
      float bm = m;
#pragma unroll
      for (int i = 0; i < kRunMergeBatch; ++i) bm = fmaxf(bm, ls[i]);
      const float base = merge_base(bm);
      const float alpha = fast_exp2(m - base);  // 0 while m is -inf
      den *= alpha;
#pragma unroll
      for (int e = 0; e < PER; ++e) o[e] *= alpha;
#pragma unroll
      for (int i = 0; i < kRunMergeBatch; ++i) {
        const float w = fast_exp2(ls[i] - base);  // 0 past the last run
        den += w;
#pragma unroll
        for (int e = 0; e < PER / 4; ++e)
#pragma unroll
          for (int r = 0; r < 4; ++r) o[4 * e + r] = fmaf(w, x[i][e][r], o[4 * e + r]);
      }
      m = bm;
    }
    const float inv = inv_sum(den);
#pragma unroll
    for (int e = 0; e < PER; ++e) o[e] *= inv;
  }
  u32x4 packed;
#pragma unroll
  for (int w = 0; w < 4; ++w) packed[w] = E::pack(o[2 * w], o[2 * w + 1]);
  *reinterpret_cast<u32x4*>(p.out + tq * p.o_st + (int64_t)head * p.o_sh + lane * PER * 2) = packed;
}

// Combine a split query's partials: o = sum_s 2^(lse_s - M) o_s / sum_s 2^(lse_s - M).
template <typename T>
__global__ __launch_bounds__(64) void mla_merge_kernel(MlaParams p) {
  using E = Elem<T>;
  const int tokq = blockIdx.x, head = blockIdx.y, lane = threadIdx.x;
  const int row = tokq / p.lq, qj = tokq - row * p.lq;
  const int lk = p.lens[row] - p.lq + qj + 1;
  const int nsplit = lk > 0 ? min((lk + p.split - 1) / p.split, p.max_splits) : 0;
  if (nsplit <= 1) return;
  const int64_t slot0 = ((int64_t)tokq * p.heads + head) * p.max_splits;
  float mmax = -INFINITY;
  for (int s = 0; s < nsplit; ++s) mmax = fmaxf(mmax, p.part_lse[slot0 + s]);
  constexpr int PER = kVDim / 64;
  float o[PER];
#pragma unroll
  for (int e = 0; e < PER; ++e) o[e] = 0.f;
  float den = 0.f;
  mmax = merge_base(mmax);
  for (int s = 0; s < nsplit; ++s) {
    const float w = fast_exp2(p.part_lse[slot0 + s] - mmax);
    den += w;
    const f32x4* src = reinterpret_cast<const f32x4*>(p.part_o + (slot0 + s) * kVDim + lane * PER);
#pragma unroll
    for (int e = 0; e < PER / 4; ++e) {
      const f32x4 x = src[e];
#pragma unroll
      for (int r = 0; r < 4; ++r) o[4 * e + r] = fmaf(w, x[r], o[4 * e + r]);
    }
  }
  const float inv = inv_sum(den);
  u32x4 packed;
#pragma unroll
  for (int w = 0; w < 4; ++w) packed[w] = E::pack(o[2 * w] * inv, o[2 * w + 1] * inv);
  *reinterpret_cast<u32x4*>(p.out + tokq * p.o_st + (int64_t)head * p.o_sh + lane * PER * 2) = packed;
}

struct MlaShape {
  int32_t split, max_splits;  // split schedule
  int32_t runs, units;        // run schedule: workgroups, units
  int32_t nb, tiles;          // and 16-column blocks per unit, units per row
  size_t lse_off, o_off, prefix_off, bytes;
};


template <typename T>
static void launch_dma(const MlaParams& p, bool one_page, dim3 grid, hipStream_t st) {
  if (one_page)
    hipLaunchKernelGGL((mla_decode_dma_kernel<T, kMlaSplitStages, true>), grid, dim3(256), 0, st, p);
  else
    hipLaunchKernelGGL((mla_decode_dma_kernel<T, kMlaSplitStages, false>), grid, dim3(256), 0, st, p);
}

static MlaShape mla_shape(int32_t rows, int32_t lq, int32_t heads, int32_t max_k) {
  MlaShape s{};
  const int64_t units = (int64_t)rows * lq * ((heads + 15) / 16);
  const int64_t keys = max_k > 0 ? max_k : 1;
  // Split schedule (pages not a multiple of 16 latents, or too many units for the in-kernel scan).
  int64_t split = 256;
  while (split < kMlaMaxSplit && split < keys && units * ((keys + split - 1) / split) > kMlaSplitTarget)
    split *= 2;
  s.split = (int32_t)split;
  s.max_splits = (int32_t)((keys + split - 1) / split);
  const size_t parts = s.max_splits > 1 ? (size_t)rows * lq * heads * s.max_splits : 0;
  // Run schedule: one workgroup per CU, fewer when the stages cannot fill runs of kRunMin.
  const int64_t columns = (int64_t)lq * heads;
  s.nb = columns <= 16 ? 1 : 2;
  const int64_t tiles = (columns + 16 * s.nb - 1) / (16 * s.nb);
  const int64_t run_units = rows * tiles;
  const int64_t stages = run_units * ((keys + kRunTile - 1) / kRunTile + kRunEnter);
  s.tiles = (int32_t)std::min<int64_t>(tiles, INT32_MAX);
  s.units = (int32_t)std::min<int64_t>(run_units, INT32_MAX);
  s.runs = (int32_t)std::max<int64_t>(
      1, std::min<int64_t>(kRunsPerCU * device_cus(), (stages + kRunMin - 1) / kRunMin));
  const size_t run_parts = (size_t)s.runs * 2 * 16 * s.nb;
  const size_t nparts = std::max(parts, run_parts);
  s.lse_off = 0;
  s.o_off = (nparts * sizeof(float) + 255) / 256 * 256;
  s.prefix_off = s.o_off + nparts * kVDim * sizeof(float);
  s.bytes = s.prefix_off + (size_t)(run_units + 2) * sizeof(int32_t);
  return s;
}

template <typename T, int NB>
static void launch_runs(const MlaParams& p, int runs, hipStream_t st) {
  hipLaunchKernelGGL((mla_run_kernel<T, NB>), dim3(runs), dim3(64 * kRunWaves), 0, st, p);
  hipLaunchKernelGGL((mla_run_merge_kernel<T, NB>), dim3(p.units, 4 * NB), dim3(256), 0, st, p);
}

template <typename T>
static void launch_runs(const MlaParams& p, const MlaShape& s, hipStream_t st) {
  if (s.nb == 1) launch_runs<T, 1>(p, s.runs, st);
  else launch_runs<T, 2>(p, s.runs, st);
}

}  // namespace lv

using namespace lv;

extern "C" size_t lv_mla_decode_workspace_bytes(int32_t num_rows, int32_t queries_per_row, int32_t num_heads,
                                                int32_t max_seqlen_k) {
  if (num_rows <= 0 || queries_per_row <= 0 || num_heads <= 0) return 0;
  return mla_shape(num_rows, queries_per_row, num_heads, max_seqlen_k).bytes;
}

extern "C" int lv_mla_decode(const void* q, int64_t q_stride_t, int64_t q_stride_h, const void* latent_cache,
                             int64_t cache_stride_block, int64_t cache_stride_token, int32_t block_size,
                             const int32_t* block_tables, int64_t table_stride, const int32_t* context_lens,
                             int32_t num_rows, int32_t queries_per_row, int32_t num_heads, int32_t latent_dim,
                             int32_t v_dim, float scale, int32_t max_seqlen_k, void* out, int64_t out_stride_t,
                             int64_t out_stride_h, void* workspace, size_t workspace_bytes, int32_t dtype,
                             void* stream) {
  LV_REQUIRE(dtype == LV_DTYPE_BF16 || dtype == LV_DTYPE_F16, "mla_decode: dtype %d is not bf16 or fp16", dtype);
  LV_REQUIRE(num_rows >= 0 && queries_per_row > 0 && num_heads > 0, "mla_decode: bad sizes B=%d Lq=%d H=%d",
             num_rows, queries_per_row, num_heads);
  LV_REQUIRE(latent_dim == kLatent && v_dim == kVDim, "mla_decode: latent %d / values %d; %d / %d are served",
             latent_dim, v_dim, kLatent, kVDim);
  if (num_rows == 0) return LV_OK;
  LV_REQUIRE(block_size >= 16, "mla_decode: block_size must be at least 16, got %d", block_size);
  LV_REQUIRE(q && latent_cache && block_tables && context_lens && out, "mla_decode: null tensor pointer");
  LV_REQUIRE(max_seqlen_k >= 0, "mla_decode: negative max_seqlen_k");
  LV_REQUIRE(scale > 0.f, "mla_decode: the softmax scale must be positive, got %g", (double)scale);
  LV_REQUIRE(aligned(q, 16) && aligned(out, 16) && aligned(latent_cache, 16) && (q_stride_t * 2) % 16 == 0 &&
                 (q_stride_h * 2) % 16 == 0 && (out_stride_t * 2) % 16 == 0 && (out_stride_h * 2) % 16 == 0 &&
                 (cache_stride_block * 2) % 16 == 0 && (cache_stride_token * 2) % 16 == 0,
             "mla_decode: tensors and their strides must be 16-byte aligned");
  const MlaShape s = mla_shape(num_rows, queries_per_row, num_heads, max_seqlen_k);
  LV_REQUIRE(workspace_bytes >= s.bytes && (s.bytes == 0 || workspace),
             "mla_decode: workspace of %zu bytes given, %zu needed", workspace_bytes, s.bytes);
  LV_REQUIRE(aligned(workspace, 256), "mla_decode: workspace must be 256-byte aligned");
  LV_REQUIRE(fits_one_launch((int64_t)num_rows * s.max_splits, 256) &&
                 fits_one_launch((int64_t)num_rows * queries_per_row, 64) &&
                 (int64_t)queries_per_row * ((num_heads + 15) / 16) < 65536,
             "mla_decode: %d rows x %d queries x %d splits need a grid larger than one launch holds", num_rows,
             queries_per_row, s.max_splits);

  MlaParams p{};
  p.q = (const char*)q;
  p.q_st = q_stride_t * 2;
  p.q_sh = q_stride_h * 2;
  p.cache = (const char*)latent_cache;
  p.c_sb = cache_stride_block * 2;
  p.c_st = cache_stride_token * 2;
  p.bs = FastDiv::make((uint32_t)block_size);
  p.tables = block_tables;
  p.t_stride = table_stride;
  p.lens = context_lens;
  p.rows = num_rows;
  p.lq = queries_per_row;
  p.heads = num_heads;
  p.htiles = (num_heads + 15) / 16;
  p.scale_log2 = scale * kLog2e;
  p.out = (char*)out;
  p.o_st = out_stride_t * 2;
  p.o_sh = out_stride_h * 2;
  p.split = s.split;
  p.max_splits = s.max_splits;
  char* ws = (char*)workspace;
  p.part_lse = s.max_splits > 1 ? reinterpret_cast<float*>(ws + s.lse_off) : nullptr;
  p.part_o = s.max_splits > 1 ? reinterpret_cast<float*>(ws + s.o_off) : nullptr;

  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  const bool one_page = block_size % kDmaTile == 0 && p.c_st * kDmaTile < ((int64_t)1 << 31);
  // The run schedule counts places in 32 bits on the device.
  const int64_t keys = std::max(max_seqlen_k, 1);
  const int64_t places = (int64_t)s.units * ((keys + kRunTile - 1) / kRunTile + kRunEnter);
  if (one_page && s.units <= kRunMaxUnits && places < ((int64_t)1 << 30)) {
    p.units = s.units;
    p.tiles = s.tiles;
    p.part_lse = reinterpret_cast<float*>(ws + s.lse_off);
    p.part_o = reinterpret_cast<float*>(ws + s.o_off);
    p.prefix = reinterpret_cast<int32_t*>(ws + s.prefix_off);
    if (dtype == LV_DTYPE_BF16)
      launch_runs<BF16>(p, s, st);
    else
      launch_runs<F16>(p, s, st);
    LV_LAUNCH_CHECK("mla_run_kernel");
    return LV_OK;
  }
  const dim3 grid(num_rows * s.max_splits, queries_per_row * p.htiles);
  if (dtype == LV_DTYPE_BF16)
    launch_dma<BF16>(p, one_page, grid, st);
  else
    launch_dma<F16>(p, one_page, grid, st);
  LV_LAUNCH_CHECK("mla_decode_dma_kernel");
  if (s.max_splits > 1) {
    const dim3 mgrid(num_rows * queries_per_row, num_heads);
    if (dtype == LV_DTYPE_BF16)
      hipLaunchKernelGGL(mla_merge_kernel<BF16>, mgrid, dim3(64), 0, st, p);
    else
      hipLaunchKernelGGL(mla_merge_kernel<F16>, mgrid, dim3(64), 0, st, p);
    LV_LAUNCH_CHECK("mla_merge_kernel");
  }
  return LV_OK;
}
