// Whole vector searches in few launches: query preparation, list probing and planning (IVF), one scan of the
// vectors with the top-k folded in, and the merge that already gives external ids.
//
// The work of a scan is one sequence of 128-row tiles over all (list, query group) items, cut into equal runs, one
// run per workgroup. A run that crosses from one item into the next ends its top-k there and starts again, so lists
// of any sizes load the chip evenly: with a fixed count of workgroups per list the longest list decided (1M x 1024
// in 64 lists of unequal size, 16 probed, one query: scan 143 us, so 102; the whole search 189 us, so 113; in one launch with its
// probing, further below, 103).
#include <algorithm>
#include "common.h"
#include "kernels.h"

namespace nga {

namespace {
constexpr int SS_W = 4;               // waves of a scan workgroup
constexpr int SS_ROWS = 32 * SS_W;    // rows of a tile
constexpr int SS_LDS = 160 * 1024;
constexpr int SEL_CAP = 1024;         // candidates that the selection sorts in LDS

__device__ __forceinline__ uint32_t ss_key(float f) {
  const uint32_t u = __float_as_uint(f);
  return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}
constexpr uint32_t KEY_NEG_INF = 0x007fffffu;

// Scores that are no numbers as the selection leaves them out; no register list takes them in. As keys those without a sign would come first
// (the matrix unit's have one, a bias may have none)
__device__ __forceinline__ f32x4 ss_drop_nan(f32x4 v) {
#pragma unroll
  for (int i = 0; i < 4; ++i) v[i] = v[i] == v[i] ? v[i] : -INFINITY;
  return v;
}

// order of results: the higher value, of equal ones the lower row
__device__ __forceinline__ bool ss_first(float av, int ar, float bv, int br) { return (av > bv) | ((av == bv) & (ar < br)); }

// a lane sees its rows in ascending order: one of equal value goes behind, and what it pushes down keeps its order
template <int K>
__device__ __forceinline__ void ss_insert(float (&v)[K], int (&r)[K], float x, int row) {
  float cv = x;
  int cr = row;
#pragma unroll
  for (int j = 0; j < K; ++j) {
    const bool sw = x > v[j];   // from the place of x on
    const float tv = v[j];
    const int tr = r[j];
    v[j] = sw ? cv : tv;
    r[j] = sw ? cr : tr;
    cv = sw ? tv : cv;
    cr = sw ? tr : cr;
  }
}

// (v, r) := top K of itself and of the list held by lane ^ mask (both sorted, descending)
template <int K>
__device__ __forceinline__ void ss_merge_xor(float (&v)[K], int (&r)[K], int mask) {
  float ov[K];
  int orr[K];
#pragma unroll
  for (int j = 0; j < K; ++j) {
    ov[j] = __shfl_xor(v[j], mask, 64);
    orr[j] = __shfl_xor(r[j], mask, 64);
  }
#pragma unroll
  for (int j = 0; j < K; ++j) {
    const bool tb = ss_first(ov[K - 1 - j], orr[K - 1 - j], v[j], r[j]);
    v[j] = tb ? ov[K - 1 - j] : v[j];
    r[j] = tb ? orr[K - 1 - j] : r[j];
  }
#pragma unroll
  for (int st = K / 2; st > 0; st >>= 1) {
#pragma unroll
    for (int j = 0; j < K; ++j) {
      if ((j & st) == 0) {
        const bool sw = ss_first(v[j + st], r[j + st], v[j], r[j]);
        const float a = v[j], b = v[j + st];
        const int ra = r[j], rb = r[j + st];
        v[j] = sw ? b : a;
        v[j + st] = sw ? a : b;
        r[j] = sw ? rb : ra;
        r[j + st] = sw ? ra : rb;
      }
    }
  }
}
}  // namespace

// ---------------------------------------------------------------- queries
// The bf16 form of one query as the stored vectors have it, divided by its norm for cosine; by one wave. Lane l holds
// elements 4 l + 256 j (D a multiple of 128 up to 1,024).
namespace {
struct WaveQuery {
  f32x4 v[4];
  __device__ __forceinline__ void load(const float* __restrict__ x, int D, int metric, int lane) {
    float ss = 0.f;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int i = 4 * lane + 256 * j;
      v[j] = (f32x4)(0.f);
      if (i < D) {
#pragma unroll
        for (int e = 0; e < 4; ++e) v[j][e] = x[i + e];
      }
#pragma unroll
      for (int e = 0; e < 4; ++e) ss += v[j][e] * v[j][e];
    }
    if (metric == SEARCH_COSINE) {
      const float nrm = fmaxf(sqrtf(wave_sum(ss)), 1e-12f);
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int e = 0; e < 4; ++e) v[j][e] /= nrm;
    }
  }
  __device__ __forceinline__ u16x4 bf(int j) const {
    return (u16x4){f2bf(v[j][0]), f2bf(v[j][1]), f2bf(v[j][2]), f2bf(v[j][3])};
  }
};
}  // namespace

// One wave per query: its bf16 form. Replaces four elementwise and reduction launches of 4 to 5 us each.
__global__ void __launch_bounds__(256) search_prep_kernel(const float* __restrict__ q, int64_t q_stride, int nq, int D, int metric,
                                                          uint16_t* __restrict__ qb, int packed) {
  const int64_t row = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  if (row >= nq) return;
  WaveQuery wq;
  wq.load(q + row * q_stride, D, metric, lane);
#pragma unroll
  for (int j = 0; j < 4; ++j)
    if (4 * lane + 256 * j < D) *reinterpret_cast<u16x4*>(qb + (packed ? packed_at((int)row, 4 * lane + 256 * j, D) : row * D + 4 * lane + 256 * j)) = wq.bf(j);
}

// Plans of the scan by one workgroup of 1,024 threads, thread t for list t with `mine` probing queries: items of sl query slots
// in list order, and run_item[b], the item with which workgroup b of the scan begins, so that a scan workgroup is two dependent loads
// away from its first vectors. Returns the first item of the thread's list.
namespace {
struct PlanShared {
  int items[1024], tiles[1024], len[1024];   // of a list: its first item, its tiles and those before it, tiles of an item
  int wave[2][16];
};

__device__ __forceinline__ int ivf_plan(PlanShared& s, int mine, int nlist, int sl, int blocks, const int64_t* __restrict__ lbeg,
                                        const int64_t* __restrict__ lend, ScanItem* __restrict__ items, int32_t* __restrict__ run_item) {
  const int t = threadIdx.x, lane = t & 63, w = t >> 6;
  int m = 0, tl = 0;
  int64_t lb = 0, le = 0;
  if (t < nlist) {
    m = (mine + sl - 1) / sl;
    lb = lbeg[t];
    le = lend[t];
    tl = le > lb ? (int)((le - lb + SS_ROWS - 1) / SS_ROWS) : 0;
  }
  int si = m, st = m * tl;   // sums up to this list
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const int a = __shfl_up(si, o, 64), b = __shfl_up(st, o, 64);
    si += lane >= o ? a : 0;
    st += lane >= o ? b : 0;
  }
  if (lane == 63) {
    s.wave[0][w] = si;
    s.wave[1][w] = st;
  }
  __syncthreads();
  int total = 0;
#pragma unroll
  for (int o = 0; o < 16; ++o) {
    si += o < w ? s.wave[0][o] : 0;
    st += o < w ? s.wave[1][o] : 0;
    total += s.wave[1][o];
  }
  const int ib = si - m, tb = st - m * tl;
  s.items[t] = ib;
  s.tiles[t] = st;
  s.len[t] = tl;
  for (int j = 0; j < m; ++j) {
    ScanItem it;
    it.tile0 = tb + j * tl;
    it.tile1 = it.tile0 + tl;
    it.nq = mine - j * sl < sl ? mine - j * sl : sl;
    it.unused = 0;
    it.beg = lb;
    it.end = le;
    items[ib + j] = it;
  }
  __syncthreads();
  for (int b = t; b < blocks; b += 1024) {
    const int g = (int)((int64_t)total * b / blocks);
    if (total == 0) break;
    int l = 0;   // the first list whose tiles end behind g
#pragma unroll
    for (int o = 512; o > 0; o >>= 1) l += s.tiles[l + o - 1] <= g ? o : 0;
    run_item[b] = s.items[l] + (g - (l ? s.tiles[l - 1] : 0)) / s.len[l];
  }
  if (t == 0) run_item[blocks] = total;
  return ib;
}
}  // namespace

// One workgroup per query: its bf16 form, its products with every centroid (rounded to bf16 as the stored vectors are,
// sums in fp32; a wave takes four centroids at once, all their loads in flight), each centroid's rank by counting, the
// nprobe first ones. Takes the place of the preparation, a cast, a score launch over one row tile (11 us) and a radix
// selection (9 us).
__global__ void __launch_bounds__(1024) ivf_probe_kernel(const float* __restrict__ q, int64_t q_stride, int D, int metric,
                                                         const float* __restrict__ cent, int nlist, int nprobe,
                                                         uint16_t* __restrict__ qb, int32_t* __restrict__ cnt,
                                                         int32_t* __restrict__ probes, IvfOne one) {
  __shared__ uint32_t sk[IVF_SCAN_MAX_LISTS];
  __shared__ PlanShared ps;
  const int64_t row = blockIdx.x;
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  WaveQuery wq;
  wq.load(q + row * q_stride, D, metric, lane);
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const u16x4 b = wq.bf(j);
    if (w == 0 && 4 * lane + 256 * j < D) *reinterpret_cast<u16x4*>(qb + row * D + 4 * lane + 256 * j) = b;
#pragma unroll
    for (int e = 0; e < 4; ++e) wq.v[j][e] = bf2f(b[e]);
  }
  if (threadIdx.x == 0) cnt[row] = 0;
  for (int c0 = 4 * w; c0 < nlist; c0 += 64) {
    f32x4 v[4][4];
#pragma unroll
    for (int u = 0; u < 4; ++u)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int i = 4 * lane + 256 * j;
        v[u][j] = (f32x4)(0.f);
        if (i < D && c0 + u < nlist) v[u][j] = *reinterpret_cast<const f32x4*>(cent + (int64_t)(c0 + u) * D + i);
      }
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      float s = 0.f;
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int e = 0; e < 4; ++e) s += wq.v[j][e] * bf2f(f2bf(v[u][j][e]));
      s = wave_sum(s);
      if (lane == 0 && c0 + u < nlist) sk[c0 + u] = ss_key(s);
    }
  }
  __syncthreads();
  const int c = threadIdx.x;
  bool first = false;
  if (c < nlist) {
    const uint32_t mine = sk[c];
    int rank = 0;
#pragma unroll 16
    for (int o = 0; o < nlist; ++o) {
      const uint32_t x = sk[o];
      rank += x > mine || (x == mine && o < c);
    }
    first = rank < nprobe;
    if (first) probes[row * nprobe + rank] = c;
  }
  if (one.items == nullptr) return;
  // the only query: its items, one a list, here, instead of in a launch of 8 us
  const int item = ivf_plan(ps, first, nlist, one.sl, one.blocks, one.lbeg, one.lend, one.items, one.run_item);
  if (first)
    for (int o = 0; o < one.sl; ++o) one.qtab[item * one.sl + o] = o ? -1 : 0;
}

// One workgroup groups the (query, probe) pairs by list: list l with n probing queries becomes ceil(n / sl) items of sl
// query slots (-1: empty).
__global__ void __launch_bounds__(1024) ivf_items_kernel(const int32_t* __restrict__ probes, int npairs, int nprobe, int nlist,
                                                         int sl, int max_items, int blocks, const int64_t* __restrict__ lbeg,
                                                         const int64_t* __restrict__ lend, ScanItem* __restrict__ items,
                                                         int32_t* __restrict__ run_item, int32_t* __restrict__ qtab) {
  __shared__ int cnt[IVF_SCAN_MAX_LISTS], base[IVF_SCAN_MAX_LISTS];
  __shared__ PlanShared ps;
  const int t = threadIdx.x;
  cnt[t] = 0;
  for (int i = t; i < max_items * sl; i += 1024) qtab[i] = -1;
  __syncthreads();
  for (int i = t; i < npairs; i += 1024) atomicAdd(&cnt[probes[i]], 1);
  __syncthreads();
  base[t] = ivf_plan(ps, cnt[t], nlist, sl, blocks, lbeg, lend, items, run_item);
  cnt[t] = 0;   // its own, read above
  __syncthreads();
  for (int i = t; i < npairs; i += 1024) {
    const int p = probes[i], rank = atomicAdd(&cnt[p], 1);
    qtab[(base[p] + rank / sl) * sl + rank % sl] = i / nprobe;
  }
}

// ---------------------------------------------------------------- scan
// Per wave a 32-row x CH-dim LDS slot, filled by lane-linear LDS-DMA (1 KiB per instruction, non-temporal) and read
// into registers as MFMA fragments; the next unit's DMA goes out before the MFMAs of this one. NG groups of 16 queries
// lie in LDS beside the slots: one workgroup fills a CU at D 1,024. Bound by the stream of vectors: 6.6 TB/s at one
// query (1M x 1024; whole search 312 us, 340 with the launches around it that are now in it). More queries of lists, or of
// vectors that scan_wide_kernel below does not take, halve what is left of LDS for the stream (33 of them, 250k x 1,024: 4.5 TB/s);
// reading MFMA fragments from HBM directly, 16 rows x 64 B an instruction, took 187 us.
// K > 0: a register list of K per lane and group, merged over lanes and waves at the end of a run, and appended to the
// query's candidates. K = 0 (more results than the lists hold, or where scan_scores_flat or scan_scores_lists finds it faster): scores
// to S, of lists too, at their rows' places.
template <int NG, int K, int CH>
__global__ void __launch_bounds__(256, 1) scan_kernel(ScanArgs p) {
  constexpr int SL = 16 * NG;
  constexpr int SLOT = 32 * CH;     // elements of a wave's slot
  constexpr int NC = CH / 8;        // 16-B positions of a row chunk
  constexpr int NI = NC / 2;        // DMA instructions of a unit: 32 rows x NC positions / 64 lanes
  constexpr int NS = CH / 32;       // MFMA k-steps of a unit
  constexpr int KR = K > 0 ? K : 1;
  extern __shared__ __attribute__((aligned(16))) uint16_t smem[];
  uint16_t* const q_s = smem + SS_W * SLOT;
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const int col = lane & 15, h = lane >> 4;
  const int D = p.D, nch = D / 8, nchx = D / CH;
  const bool flat = p.items == nullptr;
  uint16_t* const slot = smem + w * SLOT;
  // flat: workgroup b takes tiles part, part + parts, ... of query group `item` (neighbouring workgroups read
  // neighbouring tiles: 309 us for 1M x 1024 with the preparation of the query, 311 with one stretch of rows each and
  // without it). p.fine: its wave w takes the 32-row tiles w parts + part, so many times 4 parts behind it, since with up to two tiles a
  // CU whole ones leave CUs idle (us, whole / 32 rows: 13k x 1,024, 2 queries, 22.2 19.8; 40k 35.0 32.9; 20k, one query, 22.8 22.3; 40k x 384
  // 35.8 27.5 with scores; but 250k x 1,024 95.1 96.3). Lists: tiles [g0, g1) of the sequence of all items' tiles
  int item = 0, part = 0;
  int64_t g0 = 0, g1 = 1, stride = 1;
  if (flat) {
    item = blockIdx.x / p.parts;
    part = blockIdx.x % p.parts;
    stride = p.fine ? SS_W * p.parts : p.parts;
  } else {
    const int64_t total = p.run_item[gridDim.x];
    g0 = total * blockIdx.x / gridDim.x;
    g1 = total * (blockIdx.x + 1) / gridDim.x;
    if (g0 >= g1) return;
    item = p.run_item[blockIdx.x];
  }
  for (; g0 < g1; ++item) {
    int64_t beg = 0, end = p.N, t0 = p.fine ? w * p.parts + part : part, t1 = p.fine ? (p.N + 31) / 32 : (p.N + SS_ROWS - 1) / SS_ROWS;
    int nql;
    if (flat) {
      nql = p.nq - item * SL < SL ? p.nq - item * SL : SL;
      g0 = g1;
    } else {
      const ScanItem it = p.items[item];
      if (it.tile1 <= g0) continue;   // an empty list
      beg = it.beg;
      end = it.end;
      nql = it.nq;
      t0 = g0 - it.tile0;
      t1 = (g1 < it.tile1 ? g1 : it.tile1) - it.tile0;
      g0 = it.tile0 + t1;
    }
    auto row_of = [&](int64_t tile) -> int64_t { return p.fine ? tile * 32 : beg + tile * SS_ROWS + w * 32; };
    auto slot_q = [&](int s) -> int { return flat ? item * SL + s : p.qtab[(int64_t)item * SL + s]; };
    const int ngrp = (nql + 15) / 16;

    float bnext[2][4], bcur[2][4];
    auto issue = [&](int64_t tile, int c) {
      const int64_t rbase = row_of(tile);
#pragma unroll
      for (int i = 0; i < NI; ++i) {
        const unsigned li = i * 64 + lane, row = li / NC, pos = li % NC;
        int64_t gr = rbase + row;
        if (gr >= end) gr = end - 1;
        const uint16_t* src = p.X + gr * D + c * CH + ((pos ^ (row & 15)) << 3);
        __builtin_amdgcn_global_load_lds((gptr_t)src, (lptr_t)(slot + i * 512), 16, 0, 2);
      }
      if (c == 0) {   // the tile's biases arrive with its first unit
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
          for (int rr = 0; rr < 4; ++rr) {
            const int64_t r = rbase + 16 * i + 4 * h + rr;
            bnext[i][rr] = (p.bias && r < end) ? p.bias[r] : 0.f;
          }
      }
    };
    if (t0 < t1) issue(t0, 0);
    int64_t qs[K > 0 ? 1 : NG];   // the queries whose scores this lane has
    if constexpr (K == 0) {
#pragma unroll
      for (int g = 0; g < NG; ++g) qs[g] = 16 * g + col < nql ? slot_q(16 * g + col) : -1;
    }
    if (NG == 1 && p.qf) {   // unprepared queries: a wave makes the bf16 form of four of them
      for (int r = w; r < SL; r += SS_W) {
        WaveQuery wq;
#pragma unroll
        for (int j = 0; j < 4; ++j) wq.v[j] = (f32x4)(0.f);
        if (r < nql) wq.load(p.qf + (int64_t)slot_q(r) * p.q_stride, D, p.metric, lane);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const int i = 4 * lane + 256 * j;
          if (i < D) *reinterpret_cast<u16x4*>(&q_s[r * D + (((i >> 3) ^ (r & 15)) << 3) + (i & 7)]) = wq.bf(j);
        }
      }
    } else {
      for (int i = tid; i < SL * nch; i += 256) {
        const int r = i / nch, ch = i % nch;
        u16x8 v = (u16x8)(0);
        if (r < nql) v = load8(p.Q + (int64_t)slot_q(r) * D + ch * 8);
        *reinterpret_cast<u16x8*>(&q_s[r * D + ((ch ^ (r & 15)) * 8)]) = v;
      }
    }
    __syncthreads();

    float tv[NG][KR];
    int tr[NG][KR];
#pragma unroll
    for (int g = 0; g < NG; ++g)
#pragma unroll
      for (int j = 0; j < KR; ++j) {
        tv[g][j] = -INFINITY;
        tr[g][j] = -1;
      }
    f32x4 acc[2][NG];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int g = 0; g < NG; ++g) acc[i][g] = (f32x4)(0.f);
    int64_t t = t0;
    int c = 0;
    while (t < t1) {
      int c2 = c + 1;
      int64_t t2 = t;
      if (c2 == nchx) {
        c2 = 0;
        t2 = t + stride;
      }
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      if (c == 0) {
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
          for (int rr = 0; rr < 4; ++rr) bcur[i][rr] = bnext[i][rr];
      }
      u16x8 a[2][NS];
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int s = 0; s < NS; ++s)
          a[i][s] = *reinterpret_cast<const u16x8*>(slot + (16 * i + col) * CH + (((4 * s + h) ^ col) << 3));
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");   // the slot is free
      if (t2 < t1) issue(t2, c2);
#pragma unroll
      for (int s = 0; s < NS; ++s) {
        const int ch = c * NC + 4 * s + h;
#pragma unroll
        for (int g = 0; g < NG; ++g) {
          if (g < ngrp) {
            const bf16x8 bq = as_bf16x8(*reinterpret_cast<const u16x8*>(&q_s[(16 * g + col) * D + ((ch ^ col) << 3)]));
            acc[0][g] = mfma16(as_bf16x8(a[0][s]), bq, acc[0][g]);
            acc[1][g] = mfma16(as_bf16x8(a[1][s]), bq, acc[1][g]);
          }
        }
      }
      if (c == nchx - 1) {
        // acc[i][g][rr]: row tile + 16 i + 4 h + rr, query slot 16 g + col
        const int64_t rbase = row_of(t);
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          const int64_t rb = rbase + 16 * i + 4 * h;
#pragma unroll
          for (int g = 0; g < NG; ++g) {
            if constexpr (K > 0) {
              if (g < ngrp) {
#pragma unroll
                for (int rr = 0; rr < 4; ++rr) {
                  const float sc = acc[i][g][rr] * p.dot_scale + bcur[i][rr];
                  if (rb + rr < end && sc > tv[g][K - 1]) ss_insert<KR>(tv[g], tr[g], sc, (int)(rb + rr));
                }
              }
            } else {
              if (qs[g] >= 0) {
                float* dst = p.S + qs[g] * p.s_stride + rb;
                f32x4 v;
#pragma unroll
                for (int rr = 0; rr < 4; ++rr) v[rr] = acc[i][g][rr] * p.dot_scale + bcur[i][rr];
                v = ss_drop_nan(v);
                if (rb + 3 < end) {
                  __builtin_memcpy(dst, &v, 16);   // lists begin at any row
                } else {
#pragma unroll
                  for (int rr = 0; rr < 4; ++rr)
                    if (rb + rr < end) dst[rr] = v[rr];
                }
              }
            }
            acc[i][g] = (f32x4)(0.f);
          }
        }
      }
      t = t2;
      c = c2;
    }
    if constexpr (K > 0) {
#pragma unroll
      for (int g = 0; g < NG; ++g) {
        if (g < ngrp) {
          ss_merge_xor<KR>(tv[g], tr[g], 16);
          ss_merge_xor<KR>(tv[g], tr[g], 32);
        }
      }
      __syncthreads();   // every wave is past its last DMA wait and done with the query tile
      float* mv = reinterpret_cast<float*>(smem);   // [SL][4][K]
      int* mr = reinterpret_cast<int*>(mv + SL * SS_W * K);
      if (h == 0) {
#pragma unroll
        for (int g = 0; g < NG; ++g) {
#pragma unroll
          for (int j = 0; j < K; ++j) {
            mv[((16 * g + col) * SS_W + w) * K + j] = tv[g][j];
            mr[((16 * g + col) * SS_W + w) * K + j] = tr[g][j];
          }
        }
      }
      __syncthreads();
      if (tid < nql) {
        const int q = slot_q(tid);
        const float* lv = mv + tid * SS_W * K;
        const int* lr = mr + tid * SS_W * K;
        int n = 0;
        for (int j = 0; j < SS_W * K; ++j) n += lr[j] >= 0;
        n = n < p.k ? n : p.k;
        // flat: the workgroup's own k places; lists: behind what other runs have appended
        const int pos = flat ? part * p.k : atomicAdd(&p.cnt[q], n);
        if (flat)
          for (int j = n; j < p.k; ++j) {
            p.cand_v[(int64_t)q * p.cap + pos + j] = -INFINITY;
            p.cand_r[(int64_t)q * p.cap + pos + j] = -1;
          }
        int head[SS_W] = {0, 0, 0, 0};
        for (int j = 0; j < n && pos + j < p.cap; ++j) {
          float x[SS_W], best = -INFINITY;
          int xr[SS_W], bu = 0, row = -1;
#pragma unroll
          for (int u = 0; u < SS_W; ++u) {
            const int at = u * K + (head[u] < K ? head[u] : K - 1);
            x[u] = head[u] < K ? lv[at] : -INFINITY;
            xr[u] = lr[at];
          }
#pragma unroll
          for (int u = 0; u < SS_W; ++u) {
            const bool first = ss_first(x[u], xr[u], best, row);
            best = first ? x[u] : best;
            bu = first ? u : bu;
            row = first ? xr[u] : row;
          }
#pragma unroll
          for (int u = 0; u < SS_W; ++u)
            if (u == bu) ++head[u];
          p.cand_v[(int64_t)q * p.cap + pos + j] = best;
          p.cand_r[(int64_t)q * p.cap + pos + j] = row;
        }
      }
    }
    __syncthreads();   // the slots and the query tile are free for the next item
  }
}

// Flat scan for 17 to 64 queries. Held in LDS they leave a wave half of it to stream through; here a wave holds a quarter of every
// query in registers (NG x KS fragments), reads that quarter of every row, and the four waves add up in LDS, 32 rows at a time.
// LDS is then a ring of NSL units (16 rows) a wave, which all stay under way. The sums are handed over in the accumulators'
// layout, so that a lane ends with four rows of one query as in the other kernel; wave w takes rows 16 (w & 1) .. and every
// second group of queries. Bound by the stream: 1M x 1,024, k 4, whole search, before and here, 17 / 33 / 64 queries: 322 372
// 493 us, 307 299 336; k 25 (scores) 434 473 568, 412 445 504; 250k x 768, k 4: 88 100 126, 69 81 96; 10k x 384: 20 23 27, 17 19 20; 1M x 512,
// k 4: 200 240 315, 183 218 272; x 640, 33 / 64: 287 371, 232 285; x 896, 17 / 33 / 64: 316 358 451, 267 283 343; x 256, 17 / 64: 153 245, 140 228.
// Of 128 dimensions two barriers for 8 KB cost more than the smaller queries in LDS (1M, 17 / 33 / 64: 77 111 103, here 126 175 215); left there
// too are 33 to 48 queries of 256 (1M 178, 189; 100k 41, 36) and 17 to 32 of 640 (1M 207, 214; 100k 39, 36). Each dimension takes its own registers.
// Where results are kept in lists, four more waves (wide_apart) take the sums in: inserting, some 10 operations a place of the list whenever one of
// 64 lanes takes a value in, then no longer holds up the DMA and the products of the next tile. Us, whole search, in the stream's waves / apart:
// k 4, 64 queries: 1M x 1,024 341 318, 600k x 896 224 174, 900k x 512 246 180, 130k x 384 52 45, 10k x 768 22.9 22.4; 33 queries: 900k x 512
// 197 156; 20 queries: 130k x 384 36.6 33.2; k 8: 250k x 1,024, 64 queries, 146 105, 600k x 896, 40 queries, 235 187, 900k x 512, 20 queries, 195 160;
// k 12, 20 queries: 600k x 768 226 162, 60k x 1,024 47 44. Writing scores so gains nothing (33 x 250k x 1,024 124 126, 64 x 1M 479
// 502; their 33 MB cost some 18 us there, where a copy writes as much in 7); lists of 32, or of 16 for more than 32 queries, remain slower than scores (33 x 900k x 512, k 12, 223 372).
namespace {
constexpr int WIDE_BIAS = 8;   // where the stream's waves take the sums in: tiles whose biases have a place, more than are under way
// which numbers of groups (NG) it takes of 128 KS dimensions
constexpr bool wide_takes(int KS, int NG) { return NG >= 2 && NG <= 4 && KS >= 2 && KS <= 8 && !(KS == 2 && NG == 3) && !(KS == 5 && NG == 2); }
// units of 4 KS KiB for all waves that fill the LDS beside the sums and the biases, ten at most (384 dimensions, 33 queries: 205 us with ten and
// 213 with eleven)
constexpr int wide_slots(int KS, int NG, bool apart) {
  const int n = (160 - 8 * NG - (apart ? 0 : WIDE_BIAS / 4)) / (4 * KS);
  return n < 10 ? n : 10;
}
// whether waves of their own take the sums in: lists do not hold up the stream then. Not where it is what bounds: 1M x 1,024, k 4, 20 / 33 queries, in
// the stream's waves / apart, 315 311 / 323 323; 64 queries 345 / 318, k 8, 20 queries 250k 97 / 98
constexpr bool wide_apart(int NG, int K, int KS) { return K > 0 && !(KS == 8 && K == 4 && NG < 4); }
constexpr int wide_swizzle(int KS) { return KS % 4 == 0 ? 15 : KS % 2 == 0 ? 7 : 3; }
template <int N>
__device__ __forceinline__ void wide_wait() {
  static_assert(N >= 0 && N < 64, "vmcnt is 6 bits");
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}
// an accumulator to LDS while DMAs are under way (an ordinary store would wait for them); the compiler does not see that the
// instruction reads an MFMA's result, which is there after 19 cycles
__device__ __forceinline__ void wide_store(float* p, f32x4 v) {
  asm volatile("s_nop 15\n\ts_nop 7\n\tds_write_b128 %0, %1" ::"v"((uint32_t)(uintptr_t)(__attribute__((address_space(3))) void*)p), "v"(v)
               : "memory");
}
__device__ __forceinline__ void wide_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }
}  // namespace

static size_t wide_lds(int NG, int KS, bool apart) {
  return (size_t)SS_W * wide_slots(KS, NG, apart) * KS * 1024 + 8192 * NG + (apart ? 0 : WIDE_BIAS * SS_W * 64);
}

template <int NG, int K, int KS>
__global__ void __launch_bounds__(wide_apart(NG, K, KS) ? 512 : 256, 1) scan_wide_kernel(ScanArgs p) {
  constexpr bool APART = wide_apart(NG, K, KS);
  constexpr int SL = 16 * NG, NSL = wide_slots(KS, NG, APART), UNIT = 512 * KS, NC = 4 * KS, SW = wide_swizzle(KS), GW = (NG + 1) / 2;
  constexpr int KR = K > 0 ? K : 1;
  extern __shared__ __attribute__((aligned(16))) uint16_t smem[];
  float* const xch = reinterpret_cast<float*>(smem + SS_W * NSL * UNIT);
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), w = wave % SS_W;
  const int col = lane & 15, h = lane >> 4;
  const int D = 128 * KS;
  const int item = blockIdx.x / p.parts, part = blockIdx.x % p.parts;
  const int nql = p.nq - item * SL < SL ? p.nq - item * SL : SL, ngrp = (nql + 15) / 16;
  const int tiles = (int)((p.N + 31) / 32), nt = part < tiles ? (tiles - 1 - part) / p.parts + 1 : 0, units = 2 * nt;

  float tv[GW][KR];
  int tr[GW][KR];
#pragma unroll
  for (int g = 0; g < GW; ++g)
#pragma unroll
    for (int j = 0; j < KR; ++j) {
      tv[g][j] = -INFINITY;
      tr[g][j] = -1;
    }
  // the sums of tile n: rows 16 (w & 1) .. of it and every second group, with the biases b of this lane's four rows
  auto take = [&](int n, const f32x4 b) {
    const int64_t rb = (part + (int64_t)n * p.parts) * 32 + 16 * (w & 1) + 4 * h;
#pragma unroll
    for (int gg = 0; gg < GW; ++gg) {
      const int g = 2 * gg + (w >> 1);
      if (g >= ngrp) continue;
      f32x4 v = (f32x4)(0.f);
#pragma unroll
      for (int o = 0; o < SS_W; ++o) v += *reinterpret_cast<const f32x4*>(xch + (((o * 2 + (w & 1)) * NG + g) * 64 + lane) * 4);
#pragma unroll
      for (int rr = 0; rr < 4; ++rr) v[rr] = v[rr] * p.dot_scale + b[rr];
      if constexpr (K > 0) {
#pragma unroll
        for (int rr = 0; rr < 4; ++rr)
          if (rb + rr < p.N && v[rr] > tv[gg][K - 1]) ss_insert<KR>(tv[gg], tr[gg], v[rr], (int)(rb + rr));
      } else if (16 * g + col < nql) {
        v = ss_drop_nan(v);
        float* dst = p.S + (int64_t)(item * SL + 16 * g + col) * p.s_stride + rb;   // s_stride % 4 == 0
        if (rb + 3 < p.N) {
          *reinterpret_cast<f32x4*>(dst) = v;
        } else {
#pragma unroll
          for (int rr = 0; rr < 4; ++rr)
            if (rb + rr < p.N) dst[rr] = v[rr];
        }
      }
    }
  };
  if (!APART || wave < SS_W) {
    float* const bias_s = xch + 2048 * NG + w * 16;   // unless APART: [WIDE_BIAS][SS_W][16]
    uint16_t* const ring = smem + w * NSL * UNIT;
    bf16x8 bq[NG][KS];
#pragma unroll
    for (int g = 0; g < NG; ++g)
#pragma unroll
      for (int s = 0; s < KS; ++s) {
        u16x8 v = load8(p.Q + packed_at(item * SL + 16 * g + col, w * (D / 4) + 32 * s + 8 * h, D));
        bq[g][s] = as_bf16x8(16 * g + col < nql ? v : (u16x8)(0));
      }
    int off[KS], row[KS];   // of this lane's 16 bytes of instruction i: chunk c of row r lies at c ^ (r & SW)
#pragma unroll
    for (int i = 0; i < KS; ++i) {
      const int li = 64 * i + lane;
      row[i] = li / NC;
      off[i] = w * (D / 4) + (((li % NC) ^ (row[i] & SW)) << 3);
    }
    auto issue = [&](int u, bool first) {   // first: of a tile, whose biases come before it
      const int64_t rbase = (part + (int64_t)(u >> 1) * p.parts) * 32 + (u & 1) * 16;
      if (!APART && first && lane < 16) {
        const int64_t r = rbase + 16 * (w & 1) + lane;
        __builtin_amdgcn_global_load_lds((gptr_t)(p.bias + (r < p.N ? r : p.N - 1)), (lptr_t)(bias_s + ((u >> 1) % WIDE_BIAS) * (SS_W * 16)), 4, 0, 0);
      }
      uint16_t* to = ring + (u % NSL) * UNIT;
#pragma unroll
      for (int i = 0; i < KS; ++i) {
        const int64_t r = rbase + row[i];
        __builtin_amdgcn_global_load_lds((gptr_t)(p.X + (r < p.N ? r : p.N - 1) * D + off[i]), (lptr_t)(to + i * 512), 16, 0, 2);
      }
    };
#pragma unroll
    for (int u = 0; u < NSL; ++u) issue(u, u % 2 == 0);
    // the queries are used here, so that the compiler's wait for them lies before the loop
#pragma unroll
    for (int g = 0; g < NG; ++g)
#pragma unroll
      for (int s = 0; s < KS; ++s) asm volatile("" : "+v"(bq[g][s]));

    f32x4 acc[2][NG];
    auto multiply = [&](int u, int i) {
      const uint16_t* from = ring + (u % NSL) * UNIT + col * (NC * 8);
      u16x8 a[KS];
#pragma unroll
      for (int s = 0; s < KS; ++s) a[s] = *reinterpret_cast<const u16x8*>(from + (((4 * s + h) ^ (col & SW)) << 3));
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");   // the unit's place is free
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int g = 0; g < NG; ++g) acc[i][g] = (f32x4)(0.f);
#pragma unroll
      for (int s = 0; s < KS; ++s)
#pragma unroll
        for (int g = 0; g < NG; ++g) acc[i][g] = mfma16(as_bf16x8(a[s]), bq[g][s], acc[i][g]);
    };
    auto finish = [&](int n) {   // tile n of this workgroup
      wide_barrier();   // the sums of the tile before have been read
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int g = 0; g < NG; ++g) wide_store(xch + (((w * 2 + i) * NG + g) * 64 + lane) * 4, acc[i][g]);
      wide_barrier();
      if constexpr (!APART) take(n, *reinterpret_cast<const f32x4*>(bias_s + (n % WIDE_BIAS) * (SS_W * 16) + 4 * h));
    };
    // younger than unit u when its turn comes: the NSL - 1 units behind it, a bias before each even one. Stores of scores are not
    // counted: they may be done before older loads
    static_assert(APART || NSL / 2 + 2 <= WIDE_BIAS, "biases under way and of the tile in hand lie apart");
    constexpr int Y0 = (NSL - 1) * KS + (APART ? 0 : (NSL - 1) / 2), Y1 = (NSL - 1) * KS + (APART ? 0 : NSL / 2);
    int n = 0;
    for (; 2 * n + 1 + NSL < units; ++n) {
      wide_wait<Y0>();
      multiply(2 * n, 0);
      issue(2 * n + NSL, NSL % 2 == 0);
      wide_wait<Y1>();
      multiply(2 * n + 1, 1);
      issue(2 * n + 1 + NSL, NSL % 2 == 1);
      finish(n);
    }
    for (; n < nt; ++n) {   // the last units: nothing more to ask for, but one unit if it is the ring's first place that is missing
      wide_wait<0>();
      multiply(2 * n, 0);
      if (2 * n + NSL < units) issue(2 * n + NSL, NSL % 2 == 0);
      multiply(2 * n + 1, 1);
      finish(n);
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // the ring is free
  } else {
    for (int n = 0; n < nt; ++n) {   // as many barriers as the other waves pass
      f32x4 b;
#pragma unroll
      for (int rr = 0; rr < 4; ++rr) {
        const int64_t r = (part + (int64_t)n * p.parts) * 32 + 16 * (w & 1) + 4 * h + rr;
        b[rr] = p.bias[r < p.N ? r : p.N - 1];
      }
      wide_barrier();
      wide_barrier();
      take(n, b);
    }
  }

  if constexpr (K > 0) {
#pragma unroll
    for (int g = 0; g < GW; ++g) {
      ss_merge_xor<KR>(tv[g], tr[g], 16);
      ss_merge_xor<KR>(tv[g], tr[g], 32);
    }
    __syncthreads();
    float* mv = reinterpret_cast<float*>(smem);   // [SL][2][K]
    int* mr = reinterpret_cast<int*>(mv + SL * 2 * K);
    if ((!APART || wave >= SS_W) && h == 0) {
#pragma unroll
      for (int gg = 0; gg < GW; ++gg) {
        const int g = 2 * gg + (w >> 1);
        if (g < NG) {
#pragma unroll
          for (int j = 0; j < K; ++j) {
            mv[((16 * g + col) * 2 + (w & 1)) * K + j] = tv[gg][j];
            mr[((16 * g + col) * 2 + (w & 1)) * K + j] = tr[gg][j];
          }
        }
      }
    }
    __syncthreads();
    if (tid < nql) {
      const float* lv = mv + tid * 2 * K;
      const int* lr = mr + tid * 2 * K;
      int a = 0, b = 0;
      const int64_t at = (int64_t)(item * SL + tid) * p.cap + part * p.k;
      for (int j = 0; j < p.k; ++j) {   // k <= K; empty places are -inf, row -1
        const float av = a < K ? lv[a] : -INFINITY, bv = b < K ? lv[K + b] : -INFINITY;
        const int ar = a < K ? lr[a] : -1, br = b < K ? lr[K + b] : -1;
        const bool first = br < 0 || (ar >= 0 && ss_first(av, ar, bv, br));
        p.cand_v[at + j] = first ? av : bv;
        p.cand_r[at + j] = first ? ar : br;
        a += first;
        b += !first;
      }
    }
  }
}

// ---------------------------------------------------------------- lists, one query
// Probing, plan and scan of a single query in one launch. Every workgroup does the probing itself: of few centroids that is shorter (some 4 us
// for 64) than a launch of one workgroup, the way from it to the next one and that one's tables (13). And one query's lists need no
// restarts: the rows of all probed lists are one sequence of 32-row tiles, cut into equal runs, one a wave, which keeps its register list
// and its DMA under way from one list to the next. Bound by the stream of vectors. Whole search, us, before (probing with the plan in a launch
// of its own, runs that end with their list) and here: 1M x 1,024, 16 of 64 lists 88 75, 4 of 64 32.8 27.0; 500k x 768, 8 of 64 58 48; 200k x
// 768, 8 of 64, k 10 39.7 33.1; 1M x 384, 16 of 64, k 25 122 108; 100k x 384, 8 of 16 32 25.
template <int K, int CH>
__global__ void __launch_bounds__(256, 1) ivf_one_kernel(ScanArgs p, IvfLists l) {
  constexpr int SLOT = 32 * CH, NC = CH / 8, NI = NC / 2, NS = CH / 32, NB = 4;
  extern __shared__ __attribute__((aligned(16))) uint16_t smem[];
  uint16_t* const q_s = smem + SS_W * SLOT;                       // the query, and a row of zeros
  int64_t* const beg_s = reinterpret_cast<int64_t*>(q_s + 2 * p.D);         // of the probed lists
  int64_t* const end_s = beg_s + IVF_ONE_MAX_LISTS;
  int* const start_s = reinterpret_cast<int*>(end_s + IVF_ONE_MAX_LISTS);   // the first tile of each, and the count of tiles
  uint32_t* const sk = reinterpret_cast<uint32_t*>(start_s + IVF_ONE_MAX_LISTS + 1);
  int* const sum_s = reinterpret_cast<int*>(sk + IVF_ONE_MAX_LISTS);        // [2][SS_W]
  const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int col = lane & 15, h = lane >> 4;
  const int D = p.D, nchx = D / CH;
  uint16_t* const slot = smem + w * SLOT;

  // probing, as in ivf_probe_kernel
  int64_t lb = 0, le = 0;
  if (tid < l.nlist) {
    lb = l.beg[tid];
    le = l.end[tid];
  }
  WaveQuery wq;
  f32x4 va[NB][4], vb[NB][4];
  auto ask = [&](f32x4 (&v)[NB][4], int c0) {   // a centroid beyond the last: the last one's again, not used
#pragma unroll
    for (int j = 0; j < 4; ++j)
      if (256 * j < D) {
        const int i = 4 * lane + 256 * j;
#pragma unroll
        for (int u = 0; u < NB; ++u) v[u][j] = *reinterpret_cast<const f32x4*>(l.cent + (uint32_t)(min(c0 + u, l.nlist - 1) * D) + (uint32_t)(i < D ? i : 0));
      }
  };
  auto products = [&](f32x4 (&v)[NB][4], int c0) {
    float s[NB];
#pragma unroll
    for (int u = 0; u < NB; ++u) s[u] = 0.f;
#pragma unroll
    for (int j = 0; j < 4; ++j)
      if (256 * j < D) {
        const bool in = 4 * lane + 256 * j < D;
#pragma unroll
        for (int u = 0; u < NB; ++u)
#pragma unroll
          for (int e = 0; e < 4; ++e) s[u] += wq.v[j][e] * bf2f(f2bf(in ? v[u][j][e] : 0.f));
      }
    // wave_sum of all at once: one after another they would take 5 us
#pragma unroll
    for (int o = 32; o > 0; o >>= 1)
#pragma unroll
      for (int u = 0; u < NB; ++u) s[u] += __shfl_xor(s[u], o, 64);
    float own = s[0];
#pragma unroll
    for (int u = 1; u < NB; ++u) own = lane == u ? s[u] : own;
    if (lane < NB && c0 + lane < l.nlist) sk[c0 + lane] = ss_key(own);
  };
  constexpr int RB = NB * SS_W;   // centroids of a round
  ask(va, NB * w);
  ask(vb, NB * w + RB);
  wq.load(p.qf, D, p.metric, lane);
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const u16x4 b = wq.bf(j);
    const int i = 4 * lane + 256 * j;
    if (w == 0 && i < D) {
      *reinterpret_cast<u16x4*>(&q_s[i]) = b;
      *reinterpret_cast<u16x4*>(&q_s[D + i]) = (u16x4)(0);
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) wq.v[j][e] = bf2f(b[e]);
  }
  for (int c0 = NB * w; c0 - NB * w < l.nlist; c0 += 2 * RB) {
    products(va, c0);
    if (c0 + 2 * RB < l.nlist) ask(va, c0 + 2 * RB);
    products(vb, c0 + RB);
    if (c0 + 3 * RB < l.nlist) ask(vb, c0 + 3 * RB);
  }
  __syncthreads();
  bool first = false;
  if (tid < l.nlist) {
    const uint32_t mine = sk[tid];
    int rank = 0;
#pragma unroll 16
    for (int o = 0; o < l.nlist; ++o) {
      const uint32_t x = sk[o];
      rank += x > mine || (x == mine && o < tid);
    }
    first = rank < l.nprobe && le > lb;
  }
  // the probed lists that hold rows, in the order of their rows: that of the lists, or else found by counting
  const int mine = first ? (int)((le - lb + 31) / 32) : 0;
  const uint64_t who = __ballot(first);
  int tiles = mine;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const int a = __shfl_up(tiles, o, 64);
    tiles += lane >= o ? a : 0;
  }
  if (lane == 63) {
    sum_s[w] = tiles;
    sum_s[SS_W + w] = __popcll(who);
  }
  __syncthreads();
  int before = 0, place = __popcll(who & ((uint64_t(1) << lane) - 1)), total = 0, lists = 0;
#pragma unroll
  for (int u = 0; u < SS_W; ++u) {
    before += u < w ? sum_s[u] : 0;
    place += u < w ? sum_s[SS_W + u] : 0;
    total += sum_s[u];
    lists += sum_s[SS_W + u];
  }
  if (__syncthreads_or(tid + 1 < l.nlist && lb > l.beg[tid + 1])) {
    if (tid < l.nlist) {
      beg_s[tid] = lb;
      start_s[tid] = mine;
    }
    __syncthreads();
    place = before = 0;
    for (int o = 0; o < l.nlist; ++o) {
      const int to = start_s[o];   // 0: not of them
      const int64_t bo = beg_s[o];
      if (to > 0 && (bo < lb || (bo == lb && o < tid))) {
        ++place;
        before += to;
      }
    }
    tiles = mine;
    __syncthreads();
  }
  if (first) {
    beg_s[place] = lb;
    end_s[place] = le;
    start_s[place] = before + tiles - mine;
  }
  if (tid == 0) start_s[lists] = total;
  __syncthreads();

  const int64_t runs = (int64_t)gridDim.x * SS_W, run = (int64_t)blockIdx.x * SS_W + w;
  int t = __builtin_amdgcn_readfirstlane((int)(total * run / runs));
  const int t1 = __builtin_amdgcn_readfirstlane((int)(total * (run + 1) / runs));
  float tv[K];
  int tr[K];
#pragma unroll
  for (int j = 0; j < K; ++j) {
    tv[j] = -INFINITY;
    tr[j] = -1;
  }
  if (t < t1) {
    // the list of the tile that is asked for, and that tile's rows
    int at = 0, next = 0;
    int64_t nrow = 0, nend = 0, row = 0, end = 0;
    for (int o = 0; o < lists; o += 64) at += __popcll(__ballot(o + lane < lists && start_s[o + lane] <= t));
    at -= 1;
    auto open = [&](int tile) {
      while (tile >= start_s[at + 1]) ++at;   // start_s[lists] = total lies behind every tile
      at = __builtin_amdgcn_readfirstlane(at);
      next = tile;
      nrow = beg_s[at] + (int64_t)(tile - start_s[at]) * 32;
      nend = end_s[at];
    };
    float bnext[2][4], bcur[2][4];
    auto issue = [&](int c) {
#pragma unroll
      for (int i = 0; i < NI; ++i) {
        const unsigned li = i * 64 + lane, r = li / NC, pos = li % NC;
        int64_t gr = nrow + r;
        if (gr >= nend) gr = nend - 1;
        __builtin_amdgcn_global_load_lds((gptr_t)(p.X + gr * D + c * CH + ((pos ^ (r & 15)) << 3)), (lptr_t)(slot + i * 512), 16, 0, 2);
      }
      if (c == 0) {   // the tile's biases arrive with its first unit
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
          for (int rr = 0; rr < 4; ++rr) {
            const int64_t r = nrow + 16 * i + 4 * h + rr;
            bnext[i][rr] = r < nend ? p.bias[r] : 0.f;
          }
      }
    };
    f32x4 acc[2] = {(f32x4)(0.f), (f32x4)(0.f)};   // column 0 is the query's
    open(t);
    issue(0);
    int c = 0;
    while (t < t1) {
      const int c2 = c + 1 == nchx ? 0 : c + 1, t2 = c2 == 0 ? t + 1 : t;
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      if (c == 0) {
        row = nrow;
        end = nend;
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
          for (int rr = 0; rr < 4; ++rr) bcur[i][rr] = bnext[i][rr];
      }
      u16x8 a[2][NS];
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int s = 0; s < NS; ++s)
          a[i][s] = *reinterpret_cast<const u16x8*>(slot + (16 * i + col) * CH + (((4 * s + h) ^ col) << 3));
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");   // the slot is free
      if (t2 < t1) {
        if (t2 != next) open(t2);
        issue(c2);
      }
#pragma unroll
      for (int s = 0; s < NS; ++s) {
        const bf16x8 bq = as_bf16x8(*reinterpret_cast<const u16x8*>(&q_s[(col ? D : 0) + (c * NC + 4 * s + h) * 8]));
        acc[0] = mfma16(as_bf16x8(a[0][s]), bq, acc[0]);
        acc[1] = mfma16(as_bf16x8(a[1][s]), bq, acc[1]);
      }
      if (c == nchx - 1) {
#pragma unroll
        for (int i = 0; i < 2; ++i) {
#pragma unroll
          for (int rr = 0; rr < 4; ++rr) {
            const int64_t r = row + 16 * i + 4 * h + rr;
            const float sc = acc[i][rr] * p.dot_scale + bcur[i][rr];
            if (r < end && sc > tv[K - 1]) ss_insert<K>(tv, tr, sc, (int)r);
          }
          acc[i] = (f32x4)(0.f);
        }
      }
      t = t2;
      c = c2;
    }
  }
  ss_merge_xor<K>(tv, tr, 16);
  ss_merge_xor<K>(tv, tr, 32);
  __syncthreads();   // every wave is past its last DMA wait
  float* const mv = reinterpret_cast<float*>(smem);   // [SS_W][K]
  int* const mr = reinterpret_cast<int*>(mv + SS_W * K);
  if (lane == 0) {   // the query's column
#pragma unroll
    for (int j = 0; j < K; ++j) {
      mv[w * K + j] = tv[j];
      mr[w * K + j] = tr[j];
    }
  }
  __syncthreads();
  // each of the 4 K finds its place among all
  if (tid < SS_W * K) {
    const float x = mv[tid];
    const int r = mr[tid];
    int rank = 0;
    for (int o = 0; o < SS_W * K; ++o) {
      const int orow = mr[o];
      rank += orow >= 0 ? (r < 0 || ss_first(mv[o], orow, x, r)) : (r < 0 && o < tid);
    }
    if (rank < p.k) {
      p.cand_v[(int64_t)blockIdx.x * p.k + rank] = r >= 0 ? x : -INFINITY;
      p.cand_r[(int64_t)blockIdx.x * p.k + rank] = r;
    }
  }
}

// ---------------------------------------------------------------- selection
// The k <= 256 largest of n values, sorted, by one workgroup. The k-th largest of the 256 threads' maxima (of 64 groups'
// maxima where k is at most 32) is a lower bound of the k-th largest value, so a first pass takes maxima, their ranks (by
// counting) give the bound, and a second pass collects what reaches it: a few more than k values, which are ranked by
// counting again, as keys of 64 bits, sixteen comparisons' reads in flight. Up to 256 RV values stay in registers between the
// passes. Values of -inf (removed rows) are left out. Should more than
// 1,024 values reach the bound (equal scores), the k-th key is found bit by bit, and the last row that is taken of those with
// that key in the same way. Three passes over 2,048 LDS counters,
// most of them on the same few exponents, took 82 us for both levels of 33 x 250k scores, k 25; two reads of the scores, and ranks
// from one LDS read after another, 30; these took 23, and 21 with loads of 16 bytes, one operation a value and pass, and 64 registers (of 64 x 1M
// scores the whole search 476, 465; with 115 registers 480).
// Order: value, then row (the lower first).
namespace {
struct SelShared {
  uint64_t kr[SEL_CAP];   // key, then the row's complement: their order is that of results
  uint32_t tmax[256];
  uint32_t bound, n_got;
  int red[4];
};

__device__ __forceinline__ int sel_block_count(int c, int* red) {
  for (int o = 32; o > 0; o >>= 1) c += __shfl_xor(c, o, 64);
  __syncthreads();
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = c;
  __syncthreads();
  return red[0] + red[1] + red[2] + red[3];
}

// returns how many of the first k places are filled; emit(place, value, row, fetch(row)) is called for each of them, where fetch comes before
// the places are counted. mid() is called once while the first values are on their way. More than 256 RV values are read twice.
template <int RV, typename Mid, typename Fetch, typename Emit>
__device__ __forceinline__ int sel_topk(const float* __restrict__ v, const int32_t* __restrict__ r, int64_t row0, int64_t n, int k,
                                        SelShared& s, Mid mid, Fetch fetch, Emit emit) {
  const int t = threadIdx.x;
  const bool kept = n <= 256 * RV;
  float mxf = -INFINITY;
  float x[RV];
  int32_t xr[RV];
  // values c0 .. of a turn: a thread's are 256 apart, or where all are there four in a row, in loads of 16 bytes
  auto whole = [&](int64_t c0) -> bool { return !r && n - c0 >= 256 * RV; };
  auto load = [&](int64_t c0) {
    if (whole(c0)) {
#pragma unroll
      for (int u = 0; u < RV; u += 4) __builtin_memcpy(&x[u], v + c0 + 4 * t + 256 * u, 16);   // lists begin at any row
      return;
    }
    const int left = (int)(n - c0 < 256 * RV ? n - c0 : 256 * RV) - t;
#pragma unroll
    for (int u = 0; u < RV; ++u) x[u] = 256 * u < left ? v[c0 + t + 256 * u] : -INFINITY;
    if (r && kept)
#pragma unroll
      for (int u = 0; u < RV; ++u) xr[u] = 256 * u < left ? r[c0 + t + 256 * u] : -1;
  };
  for (int64_t c0 = 0; c0 < (kept ? 1 : n); c0 += RV * 256) {
    load(c0);
    if (kept) mid();
#pragma unroll
    for (int u = 0; u < RV; ++u) mxf = fmaxf(mxf, x[u]);
  }
  if (!kept) mid();
  uint32_t mx = ss_key(mxf);
  const int ngr = k <= 32 ? 64 : 256;   // groups of four threads, or threads
  if (ngr == 64) {
    uint32_t o = __shfl_xor(mx, 1, 64);
    mx = o > mx ? o : mx;
    o = __shfl_xor(mx, 2, 64);
    mx = o > mx ? o : mx;
    if ((t & 3) == 0) s.tmax[t >> 2] = mx;
  } else {
    s.tmax[t] = mx;
  }
  if (t == 0) s.n_got = 0;
  __syncthreads();
  if (t < ngr) {
    const uint32_t own = s.tmax[t];
    int rank = 0;
#pragma unroll 16
    for (int o = 0; o < ngr; ++o) {
      const uint32_t m = s.tmax[o];
      rank += m > own || (m == own && o < t);
    }
    if (rank == k - 1) s.bound = own > KEY_NEG_INF ? own : KEY_NEG_INF + 1;
  }
  __syncthreads();
  const uint32_t bound = s.bound;
  const float least = __uint_as_float((bound & 0x80000000u) ? (bound & 0x7fffffffu) : ~bound);
  for (int64_t c0 = 0; c0 < (kept ? 1 : n); c0 += RV * 256) {
    if (!kept) load(c0);
    const bool four = whole(c0);
#pragma unroll
    for (int u = 0; u < RV; ++u) {
      if (!(x[u] < least)) {   // one operation a value; the key orders what is left
        const uint32_t key = ss_key(x[u]);
        if (key < bound) continue;
        const uint32_t pos = atomicAdd(&s.n_got, 1u);
        if (pos < SEL_CAP) {
          const int64_t i = c0 + (four ? 4 * t + 256 * (u & ~3) + (u & 3) : t + 256 * u);
          const int32_t row = r ? (kept ? xr[u] : r[i]) : (int32_t)(row0 + i);
          s.kr[pos] = (uint64_t)key << 32 | (uint32_t)~row;
        }
      }
    }
  }
  __syncthreads();
  int got = (int)s.n_got;
  if (got > SEL_CAP) {   // the k-th largest key, its bits from the highest down
    uint32_t kth = 0;
    for (int b = 31; b >= 0; --b) {
      const uint32_t cand = kth | (1u << b);
      int c = 0;
      for (int64_t i = t; i < n; i += 256) c += ss_key(v[i]) >= cand;
      if (sel_block_count(c, s.red) >= k) kth = cand;
    }
    int above = 0;
    for (int64_t i = t; i < n; i += 256) above += ss_key(v[i]) > kth;
    const int left = k - sel_block_count(above, s.red);   // at least one of those that are equal
    uint32_t last = 0;   // the largest row such that fewer than `left` of them lie below it; rows are not negative
    for (int b = 30; b >= 0; --b) {
      const uint32_t cand = last | (1u << b);
      int c = 0;
      for (int64_t i = t; i < n; i += 256) c += ss_key(v[i]) == kth && (uint32_t)(r ? r[i] : (int32_t)(row0 + i)) < cand;
      if (sel_block_count(c, s.red) < left) last = cand;
    }
    __syncthreads();
    if (t == 0) s.n_got = 0;
    __syncthreads();
    for (int64_t i = t; i < n; i += 256) {
      const uint32_t key = ss_key(v[i]);
      const int32_t row = r ? r[i] : (int32_t)(row0 + i);
      if (key > kth || (key == kth && (uint32_t)row <= last)) {
        const uint32_t pos = atomicAdd(&s.n_got, 1u);
        if (pos < (uint32_t)k) s.kr[pos] = (uint64_t)key << 32 | (uint32_t)~row;
      }
    }
    __syncthreads();
    got = (int)s.n_got < k ? (int)s.n_got : k;
  }
  for (int i = t; i < got; i += 256) {
    const uint64_t own = s.kr[i];
    const int32_t row = (int32_t)~(uint32_t)own;
    const auto with = fetch(row);
    int place = 0;
#pragma unroll 16
    for (int o = 0; o < got; ++o) {
      const uint64_t x = s.kr[o];
      place += x > own || (x == own && o < i);
    }
    const uint32_t key = (uint32_t)(own >> 32);
    if (place < k) emit(place, __uint_as_float((key & 0x80000000u) ? (key & 0x7fffffffu) : ~key), row, with);
  }
  return got < k ? got : k;
}
}  // namespace

// the k best of each segment of a row of scores, as candidates
__global__ void __launch_bounds__(256, 8) select_segments_kernel(const float* __restrict__ S, int64_t s_stride, int64_t N,
                                                              int64_t seg, int k, int32_t cap, float* __restrict__ cand_v,
                                                              int32_t* __restrict__ cand_r) {
  __shared__ SelShared s;
  const int64_t q = blockIdx.y, beg = blockIdx.x * seg;
  const int64_t n = N - beg < seg ? N - beg : seg;
  float* ov = cand_v + q * cap + (int64_t)blockIdx.x * k;
  int32_t* orow = cand_r + q * cap + (int64_t)blockIdx.x * k;
  const int got = sel_topk<32>(S + q * s_stride + beg, (const int32_t*)nullptr, beg, n, k, s, [] {}, [](int32_t) { return 0; }, [&](int place, float v, int32_t r, int) {
    ov[place] = v;
    orow[place] = r;
  });
  for (int i = got + threadIdx.x; i < k; i += 256) {
    ov[i] = -INFINITY;
    orow[i] = -1;
  }
}

// the same of each list that a query probes
__global__ void __launch_bounds__(256, 8) select_lists_kernel(const float* __restrict__ S, int64_t s_stride, const int32_t* __restrict__ probes,
                                                           const int64_t* __restrict__ lbeg, const int64_t* __restrict__ lend, int k,
                                                           float* __restrict__ cand_v, int32_t* __restrict__ cand_r) {
  __shared__ SelShared s;
  const int64_t q = blockIdx.y, nprobe = gridDim.x, at = (q * nprobe + blockIdx.x) * k;
  const int list = probes[q * nprobe + blockIdx.x];
  const int64_t beg = lbeg[list], n = lend[list] > beg ? lend[list] - beg : 0;
  const int got = sel_topk<32>(S + q * s_stride + beg, (const int32_t*)nullptr, beg, n, k, s, [] {}, [](int32_t) { return 0; }, [&](int place, float v, int32_t r, int) {
    cand_v[at + place] = v;
    cand_r[at + place] = r;
  });
  for (int i = got + threadIdx.x; i < k; i += 256) {
    cand_v[at + i] = -INFINITY;
    cand_r[at + i] = -1;
  }
}

// a query's result from its candidates: the k best, less |q|^2 (l2), with the external ids of finite scores. A chain of latencies: the
// query's squares are added up while the candidates are on their way, the ids come while the places are counted
__global__ void __launch_bounds__(256) search_finish_kernel(const float* __restrict__ cand_v, const int32_t* __restrict__ cand_r,
                                                            const int32_t* __restrict__ cnt, int32_t n_fixed, int32_t cap,
                                                            int k, const float* __restrict__ qf, int64_t q_stride, int D,
                                                            const int64_t* __restrict__ ids, float* __restrict__ out_v,
                                                            int64_t* __restrict__ out_id) {
  __shared__ SelShared s;
  __shared__ float red[4];
  const int64_t q = blockIdx.x;
  int n = n_fixed >= 0 ? n_fixed : cnt[q];
  n = n < cap ? n : cap;
  const int t = threadIdx.x;
  float qv[4] = {0.f, 0.f, 0.f, 0.f};
  if (qf)   // l2; D <= 1,024
#pragma unroll
    for (int j = 0; j < 4; ++j)
      if (t + 256 * j < D) qv[j] = qf[q * q_stride + t + 256 * j];
  auto squares = [&]() {
    if (!qf) return;
    float less = 0.f;
#pragma unroll
    for (int j = 0; j < 4; ++j) less = __builtin_fmaf(qv[j], qv[j], less);
    less = wave_sum(less);
    if ((t & 63) == 0) red[t >> 6] = less;   // read behind the selection's barriers
  };
  const int got = sel_topk<16>(cand_v + q * cap, cand_r + q * cap, 0, n, k, s, squares, [&](int32_t r) { return r >= 0 ? ids[r] : (int64_t)-1; },
                               [&](int place, float v, int32_t, int64_t id) {
    const float x = qf ? v - (((red[0] + red[1]) + red[2]) + red[3]) : v;
    out_v[q * k + place] = x;
    out_id[q * k + place] = isfinite(x) ? id : -1;
  });
  for (int i = got + threadIdx.x; i < k; i += 256) {
    out_v[q * k + i] = -INFINITY;
    out_id[q * k + i] = -1;
  }
}

// ---------------------------------------------------------------- launches
// dims of a unit: the largest of 512, 384, 256, 128 that divides D and fits beside the queries (more bytes in flight)
int scan_chunk(int D, int ng) {
  if (D % 128 != 0 || D < 128 || D > 1024 || ng < 1 || ng > 4) return 0;
  for (int ch : {512, 384, 256, 128})
    if (D % ch == 0 && (ng == 1 || ch < 512) && SS_W * 32 * ch * 2 + 16 * ng * D * 2 <= SS_LDS) return ch;
  return 0;
}

static size_t scan_lds(int D, int ng, int ch, int K) {
  const size_t tiles = (size_t)(SS_W * 32 * ch + 16 * ng * D) * 2, merge = (size_t)16 * ng * SS_W * K * 8;
  return tiles > merge ? tiles : merge;
}

int scan_blocks(int D, int ng, int cus) {
  const int ch = scan_chunk(D, ng);
  const int per_cu = (int)(SS_LDS / scan_lds(D, ng, ch, 32));
  return cus * (per_cu < 1 ? 1 : per_cu > 4 ? 4 : per_cu);
}

template <int NG, int K, int CH>
static void scan_go(const ScanArgs& a, int blocks, hipStream_t stream) {
  static const bool attr = [] {
    (void)hipFuncSetAttribute((const void*)scan_kernel<NG, K, CH>, hipFuncAttributeMaxDynamicSharedMemorySize, SS_LDS);
    (void)hipGetLastError();
    return true;
  }();
  (void)attr;
  scan_kernel<NG, K, CH><<<blocks, 256, scan_lds(a.D, NG, CH, K), stream>>>(a);
}

template <int NG, int K>
static void scan_ch(const ScanArgs& a, int blocks, hipStream_t stream) {
  switch (scan_chunk(a.D, NG)) {
    case 512: if constexpr (NG == 1) scan_go<NG, K, 512>(a, blocks, stream); break;
    case 384: scan_go<NG, K, 384>(a, blocks, stream); break;
    case 256: scan_go<NG, K, 256>(a, blocks, stream); break;
    case 128: scan_go<NG, K, 128>(a, blocks, stream); break;
    default: break;
  }
}

// lists: 4, 8, 16, 32 results with up to 32 queries of an item, 4, 8 with up to 64; K = 0: scores
int scan_list(int k, int ng, bool ivf) {
  const int most = ng <= 2 ? (ivf ? 32 : 16) : 8;
  return k > most ? 0 : k <= 4 ? 4 : k <= 8 ? 8 : k <= 16 ? 16 : 32;
}

bool scan_wide_covers(int D, int ng) { return D % 128 == 0 && wide_takes(D / 128, ng); }   // flat scans of 17 to 64 queries, prepared

// Whether scores go to memory and are selected from there where register lists could hold the results: a list of 16 or 32 costs every
// lane some 100 or 200 operations whenever one of a wave's takes a value in, and on merging, whatever the rows' length: some 5 to 20 us, more
// with fewer dimensions. A score costs 4 bytes twice, and the writes hold up the stream the more, the more of its time is the vectors' own:
// the line is one of rows x (queries + 2). Up to 128 MiB of scores. Whole searches, us, lists / scores, on either side of the lines:
// 512 dimensions, k 9, at 1 / 16 queries: 60k 37 39, 29 33; 2M 350 452, 325 424 (fewer gain more: 128, 2M 168 204, 111 154).
// 640, k 9, at 1 / 8 / 16: 250k 85 89 91, 67 77 86; 1M 244 254 257, 221 268 286; 2M 441 463 468, 432 518 551; at 17 / 32: 250k 88 90, 80 86; 700k 187 194,
// 191 208. 768, at 1 / 8 / 16: 250k 96 100 100, 79 88 97; 1M 257 287 290, 249 302 324; one of 2M 470, 480. 896: 250k 88 90 92, 81 91 100; 1M 276 282 285, 283
// 329 350. 1,024: 250k 110 113 114, 96 106 116; 1M 321 335 338, 324 378 402. k 16 moves the lines out a little: 896, 8 of 250k 102 / 93.
// 17 to 64 queries of the dimensions of scan_wide_kernel stay in its lists, which waves of their own keep: 600k x 768, 20 queries, k 12, 161 208, 33, k
// 8, 161 230; 900k x 512, 33, k 8, 222 247; closest 130k x 384, 20, k 12, 51 48. 33 to 48 of 256 dimensions, k 5 / 8, at 34 / 48: 12k 27 27, 23 24; 100k 52 51,
// 42 45; 600k 178 193, 122 127
bool scan_scores_flat(int64_t nq, int64_t N, int D, int k) {
  if (nq > 64 || nq * N > (int64_t(1) << 25)) return false;
  if (nq > 16 && scan_wide_covers(D, nq <= 32 ? 2 : nq <= 48 ? 3 : 4)) return false;
  if (nq > 32) return D == 256 && k > 4 && k <= 8;   // what is left of 128 dimensions keeps its lists
  if (k <= 8 || k > 16) return false;
  const int64_t cost = N * (nq + 2);
  return D <= 512 || cost <= (nq > 16 ? 12000000 : D <= 768 ? 5000000 : D == 896 ? 2000000 : 2500000);   // above 16 queries: 640 dimensions
}
// The same of lists. What register lists cost here is a merge for every run of a query's rows; what scores cost, beside the writes, is a selection by one
// workgroup a query and list (which reads more than 8,192 scores twice): a few long lists leave the chip waiting for it, and of many short ones, or few rows
// in all, it is a launch too much. Measured on 4,000 searches of any sizes; us, register lists / scores:
// k 25, 16 of 64 lists, at 1 / 5 / 12 / 32 queries: 1M x 1,024 165 386 470 453, 133 299 376 418; 200k x 768 69 130 137 144, 47 80 88 94; 60k x 384 49 75 76 79, 35 41
// 42 45. No search of 17 to 32 results was faster in lists.
// k 9 to 16: 8 of 64, k 14, 2 / 5 / 12 / 20 / 32 queries: 1M x 1,024 135 210 299 357 376, 123 196 297 361 392; 200k x 768 60 80 93 102 111, 47 63 73 81 89. On either side of the
// lists' length, 6 x 1.3M x 128, 8 of 8, 163 138, 3 x 885k x 384, 2 of 2, 196 232; 6 x 317k x 768, 8 of 8, 139 131, 3 x 1.1M x 768, 1 of 16, 154 191; of the scores
// (and the rows read), 8 x 1.5M x 768, 8 of 64, 307 284, 8 x 1.5M x 640, 32 of 32, 365 417, 8 x 1.3M x 1,024, 16 of 64, 444 452; more than 16 queries write whole lines: 32 x 490k x 768, 64 of 64, 235 212.
// k 5 to 8: 20 x 109k x 256, 16 of 64, 26 % less, 12 x 93k x 128 15, 4 x 95k x 384 10, 6 x 220k x 640 9; beyond the lines 6 x 416k x 512, 8 of 8, 112 141; 12 x 817k x 640, 4 of
// 16, 203 242; 64 x 16k x 128, 64 of 256, 50 58; 8 x 15k x 256, 4 of 4, 28 31; 12 x 927k x 768, 16 of 64, 260 277. Of the 290 of 1,500 that these lines take 16 are slower, by
// 1.5 to 5 %. One query of k 12 is the one launch's, where that takes it (1M x 1,024 128 / 131).
bool scan_scores_lists(int64_t nq, int64_t N, int D, int k, int64_t nlist, int64_t nprobe) {
  if (k <= 4 || nq * N > (int64_t(1) << 25)) return false;
  const int64_t rows = N / nlist, pairs = nq * nprobe, n = pairs * rows;   // a list's rows and all scores, with lists of one length
  if (k > 16) return true;
  if (k > 8) {
    if (D <= 512) return rows <= 262144;
    return rows <= (D <= 768 ? 49152 : 32768) && (nq > 16 || n + 2 * std::min(pairs, nlist) * rows <= (D <= 768 ? 6000000 : 3000000));
  }
  return rows <= (D <= 256 ? 24576 : 8192) && pairs >= 32 && pairs <= 2048 && N >= 30000 && n >= 30000 && n <= 3000000 &&
         (D <= 512 || (D <= 768 && nq <= 16));
}

void launch_scan(const ScanArgs& a, int ng, int K, int blocks, hipStream_t stream) {
#define NGA_SCAN(NG_, K_) if (ng == NG_ && K == K_) return scan_ch<NG_, K_>(a, blocks, stream)
  NGA_SCAN(1, 0); NGA_SCAN(1, 4); NGA_SCAN(1, 8); NGA_SCAN(1, 16); NGA_SCAN(1, 32);
  NGA_SCAN(2, 0); NGA_SCAN(2, 4); NGA_SCAN(2, 8); NGA_SCAN(2, 16); NGA_SCAN(2, 32);
  NGA_SCAN(3, 0); NGA_SCAN(3, 4); NGA_SCAN(3, 8);
  NGA_SCAN(4, 0); NGA_SCAN(4, 4); NGA_SCAN(4, 8);
#undef NGA_SCAN
}

// The dimensions whose slots fill a CU with one workgroup; with several (128, 256, 640, 896) all of them would probe: 100k x 640, 64 lists 30
// us, here 54. And as many centroids as take no longer here than in a launch of their own; both, us, at 128 and 160 lists: 500k x 1,024
// 50.4 43.9, 41.3 42.7; 100k x 1,024 35.6 32.9, 37.3 38.0; 100k x 768 33.9 29.2, 35.3 33.0; 100k x 384 30.9 25.1, 32.2 28.2 (256 lists, 200k:
// 39.0 35.9; x 1,024 44.2 46.4).
bool ivf_one_covers(int64_t nq, int64_t nlist, int D, int k) {
  return nq == 1 && nlist <= IVF_ONE_MAX_LISTS && nlist * D <= 128 * 1024 && k >= 1 && k <= 32 && scan_chunk(D, 1) >= 384;
}

template <int K, int CH>
static void one_go(const ScanArgs& a, const IvfLists& l, int blocks, hipStream_t stream) {
  constexpr size_t lds = (size_t)SS_W * 32 * CH * 2 + 2 * 1024 * 2 + IVF_ONE_MAX_LISTS * 24 + 4 + 2 * SS_W * 4;
  static_assert(lds <= SS_LDS, "LDS");
  static const bool attr = [] {
    (void)hipFuncSetAttribute((const void*)ivf_one_kernel<K, CH>, hipFuncAttributeMaxDynamicSharedMemorySize, SS_LDS);
    (void)hipGetLastError();
    return true;
  }();
  (void)attr;
  ivf_one_kernel<K, CH><<<blocks, 256, lds, stream>>>(a, l);
}

template <int K>
static void one_ch(const ScanArgs& a, const IvfLists& l, int blocks, hipStream_t stream) {
  if (scan_chunk(a.D, 1) == 512) one_go<K, 512>(a, l, blocks, stream);
  else one_go<K, 384>(a, l, blocks, stream);
}

void launch_ivf_one(const ScanArgs& a, const IvfLists& l, int blocks, hipStream_t stream) {
  switch (scan_list(a.k, 1, true)) {
    case 4: return one_ch<4>(a, l, blocks, stream);
    case 8: return one_ch<8>(a, l, blocks, stream);
    case 16: return one_ch<16>(a, l, blocks, stream);
    case 32: return one_ch<32>(a, l, blocks, stream);
    default: return;
  }
}

template <int NG, int K, int KS>
static void wide_go(const ScanArgs& a, int blocks, hipStream_t stream) {
  if constexpr (wide_takes(KS, NG)) {
    static const bool attr = [] {
      (void)hipFuncSetAttribute((const void*)scan_wide_kernel<NG, K, KS>, hipFuncAttributeMaxDynamicSharedMemorySize, SS_LDS);
      (void)hipGetLastError();
      return true;
    }();
    (void)attr;
    scan_wide_kernel<NG, K, KS><<<blocks, wide_apart(NG, K, KS) ? 512 : 256, wide_lds(NG, KS, wide_apart(NG, K, KS)), stream>>>(a);
  }
}

void launch_scan_wide(const ScanArgs& a, int ng, int K, int blocks, hipStream_t stream) {
#define NGA_WIDE(NG_, K_)                                              \
  if (ng == NG_ && K == K_) {                                          \
    switch (a.D / 128) {                                               \
      case 2: return wide_go<NG_, K_, 2>(a, blocks, stream);           \
      case 3: return wide_go<NG_, K_, 3>(a, blocks, stream);           \
      case 4: return wide_go<NG_, K_, 4>(a, blocks, stream);           \
      case 5: return wide_go<NG_, K_, 5>(a, blocks, stream);           \
      case 6: return wide_go<NG_, K_, 6>(a, blocks, stream);           \
      case 7: return wide_go<NG_, K_, 7>(a, blocks, stream);           \
      case 8: return wide_go<NG_, K_, 8>(a, blocks, stream);           \
    }                                                                  \
  }
  NGA_WIDE(2, 0); NGA_WIDE(2, 4); NGA_WIDE(2, 8); NGA_WIDE(2, 16);
  NGA_WIDE(3, 0); NGA_WIDE(3, 4); NGA_WIDE(3, 8);
  NGA_WIDE(4, 0); NGA_WIDE(4, 4); NGA_WIDE(4, 8);
#undef NGA_WIDE
}

void launch_search_prep(const float* q, int64_t q_stride, int nq, int D, int metric, uint16_t* qb, bool packed,
                        hipStream_t stream) {
  search_prep_kernel<<<(nq + 3) / 4, 256, 0, stream>>>(q, q_stride, nq, D, metric, qb, packed);
}

void launch_ivf_probe(const float* q, int64_t q_stride, int nq, int D, int metric, const float* cent, int nlist, int nprobe,
                      uint16_t* qb, int32_t* cnt, int32_t* probes, const IvfOne& one, hipStream_t stream) {
  ivf_probe_kernel<<<nq, 1024, 0, stream>>>(q, q_stride, D, metric, cent, nlist, nprobe, qb, cnt, probes, one);
}

void launch_ivf_items(const int32_t* probes, int npairs, int nprobe, int nlist, int sl, int max_items, int blocks,
                      const int64_t* lbeg, const int64_t* lend, ScanItem* items, int32_t* run_item, int32_t* qtab,
                      hipStream_t stream) {
  ivf_items_kernel<<<1, 1024, 0, stream>>>(probes, npairs, nprobe, nlist, sl, max_items, blocks, lbeg, lend, items, run_item,
                                           qtab);
}

void launch_select_segments(const float* S, int64_t s_stride, int nq, int64_t N, int64_t seg, int k, int32_t cap, float* cand_v,
                            int32_t* cand_r, hipStream_t stream) {
  dim3 grid((unsigned)((N + seg - 1) / seg), (unsigned)nq);
  select_segments_kernel<<<grid, 256, 0, stream>>>(S, s_stride, N, seg, k, cap, cand_v, cand_r);
}

void launch_select_lists(const float* S, int64_t s_stride, int nq, const int32_t* probes, int nprobe, const int64_t* lbeg, const int64_t* lend,
                         int k, float* cand_v, int32_t* cand_r, hipStream_t stream) {
  select_lists_kernel<<<dim3(nprobe, nq), 256, 0, stream>>>(S, s_stride, probes, lbeg, lend, k, cand_v, cand_r);
}

void launch_search_finish(const float* cand_v, const int32_t* cand_r, const int32_t* cnt, int32_t n_fixed, int32_t cap, int nq,
                          int k, const float* qf, int64_t q_stride, int D, const int64_t* ids, float* out_v, int64_t* out_id,
                          hipStream_t stream) {
  search_finish_kernel<<<nq, 256, 0, stream>>>(cand_v, cand_r, cnt, n_fixed, cap, k, qf, q_stride, D, ids, out_v, out_id);
}

}  // namespace nga
