// Token sampling over a full vocabulary row (up to 256K: Gemma) (K7 in SURVEY.md §2.C), one 1024-thread
// workgroup per sequence, no full sort:
//   * repetition penalty (TRT-LLM semantics: divide positive / multiply negative logits of
//     every token seen in prompt+output) through an LDS bitmap of the row's history;
//   * temperature; greedy when temperature <= 0 or top_k == 1;
//   * top-k / top-p thresholds, fast path: one pass bins every token with v > M - 16 by its
//     distance to the row max (2048 linear bins, so the LDS atomics spread out instead of piling
//     onto a few exponent bins; the far tail takes no atomic), a scan finds the bin where the
//     running count / probability mass reaches the target, a second pass gathers that bin's keys
//     (at most 2048) into LDS, and a bitonic sort + scan there gives the exact threshold;
//   * exact fallback when the crossing lies in the far tail or its bin is too full (flat rows,
//     p close to 1): 3-level (11/11/10-bit) radix descent on order-preserving float keys;
//   * the draw itself is Gumbel-max over the kept tokens with a counter-based RNG keyed on
//     (seed, step, token): deterministic for a given seed, no global RNG state.
// Every pass over the row keeps eight 16-byte loads in flight per thread. Histogram weights are
// 64-bit fixed point (2^-40 units of exp(v - M)) so the LDS atomics are ds_add_u64: LDS
// ds_add_f32 measured ~8x slower on gfx950 (scripts/dev/lds_atomic_bench.hip).
//   * rows of 30,000 values and more, up to some dozens of them, first go through sample_slices_kernel, some 2,000 values a workgroup,
//     which finds the largest value and the partition function's part of each slice and lists its values close to that maximum. One
//     workgroup a row is bound by its own arithmetic: a pass over 128,256 values takes it 14 to 20 us. Where the lists reach far enough below the row's maximum (at the
//     temperature of 0.2 that the servers use by default they do, with some 20 of 2,000 values) all passes of the fast path go over
//     them, in registers, instead of the row. More in sample_slices.
// Also returns the chosen token's log-probability under the temperature-scaled distribution.
#include "common.h"
#include "kernels.h"

namespace nga {

namespace {
constexpr int NT = 1024;
constexpr int NBINS = 2048;
constexpr int CAP = 2048;        // keys the fast path sorts in LDS
constexpr float DRANGE = 16.f;   // fast-path bins cover v in (M - DRANGE, M]
constexpr float DSCALE = NBINS / DRANGE;
constexpr int UNROLL = 8;

__device__ __forceinline__ uint32_t fkey(float f) {
  const uint32_t u = __float_as_uint(f);
  return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}

__device__ __forceinline__ float fval(uint32_t k) {
  return __uint_as_float((k & 0x80000000u) ? (k & 0x7fffffffu) : ~k);
}

struct ArgMax {
  float v;
  int i;
};
struct SampleEntry {   // a value that a slice lists, before the temperature
  float v;
  int i;
};
struct SampleSlice {
  float m, z;   // the largest value, and the sum of exp(v - m)
  int i, n;     // where it is; how many are listed
  float range;  // those less than this below m
};

constexpr int SLICE = 2048;        // values of a slice: 8 a thread
constexpr int MAX_SLICES = 128;    // of a row (262,144 values)
constexpr int LISTED = 64;         // values that a slice can list

constexpr double FIX = 1099511627776.0;  // 2^40: fixed-point unit of the mass histograms

struct Smem {
  union {
    uint32_t bitmap[8192];  // history bitmap (repetition penalty only), V <= 262144 (Gemma: 256000)
    struct {
      union {
        uint64_t q[NBINS];  // bin weights: counts or fixed-point mass
        float w[NBINS];     // candidate weights (fast path, after the bin scan)
      } h;
      uint32_t cand[CAP];
      union {
        uint64_t q[NT];
        float f[NT];
      } scan;
    } s;
  } u;
  float red[NT / 64];
  ArgMax ared[NT / 64];
  int ncand;
  int sel;
  float sel_above_f;
  uint64_t sel_above_q;
};

// Top-down crossing over nb <= 2*NT values (bins[nb-1] is the top): inclusive suffix scan,
// returns the bin where the running total first reaches `target` and the total strictly above
// it, or -1 (with the grand total in *above_out) when the total stays below target.
template <typename T>
__device__ __forceinline__ int find_crossing(const T* bins, int nb, T target, T* above_out, T* scan, Smem& sm) {
  const int t = threadIdx.x;
  // thread t owns bins (nb-1-2t) and (nb-2-2t): descending order
  const int b0 = nb - 1 - 2 * t, b1 = b0 - 1;
  const T v0 = b0 >= 0 ? bins[b0] : (T)0, v1 = b1 >= 0 ? bins[b1] : (T)0;
  const T mine = v0 + v1;
  scan[t] = mine;
  __syncthreads();
  for (int off = 1; off < NT; off <<= 1) {
    T add = t >= off ? scan[t - off] : (T)0;
    __syncthreads();
    scan[t] += add;
    __syncthreads();
  }
  const T incl = scan[t];
  const T excl = incl - mine;
  if (t == 0) sm.sel = -1;
  __syncthreads();
  if (excl < target && incl >= target) {
    const bool first = excl + v0 >= target;
    sm.sel = first ? b0 : b1;
    const T a = first ? excl : excl + v0;
    if constexpr (sizeof(T) == 8)
      sm.sel_above_q = a;
    else
      sm.sel_above_f = a;
  }
  __syncthreads();
  const int s = sm.sel;
  T a;
  if constexpr (sizeof(T) == 8)
    a = sm.sel_above_q;
  else
    a = sm.sel_above_f;
  *above_out = s >= 0 ? a : scan[NT - 1];
  __syncthreads();
  return s;
}

// Visit every element of a row: UNROLL float4 loads in flight per thread for the body (rows
// of the [B, V] fp32 logits are 16-B aligned when V % 4 == 0), scalar loads for any tail.
// f(index, value) is called by every lane of the workgroup in step for the unrolled body.
template <typename F>
__device__ __forceinline__ void for_row(const float* __restrict__ x, int V, F f) {
  const int t = threadIdx.x;
  if ((V & 3) == 0) {
    const float4* x4 = reinterpret_cast<const float4*>(x);
    const int n4 = V >> 2;
    int j = t;
    for (; j + (UNROLL - 1) * NT < n4; j += UNROLL * NT) {
      float4 v[UNROLL];
#pragma unroll
      for (int u = 0; u < UNROLL; ++u) v[u] = x4[j + u * NT];
#pragma unroll
      for (int u = 0; u < UNROLL; ++u) {
        const int i = 4 * (j + u * NT);
        f(i, v[u].x);
        f(i + 1, v[u].y);
        f(i + 2, v[u].z);
        f(i + 3, v[u].w);
      }
    }
    for (; j < n4; j += NT) {
      const float4 v = x4[j];
      f(4 * j, v.x);
      f(4 * j + 1, v.y);
      f(4 * j + 2, v.z);
      f(4 * j + 3, v.w);
    }
  } else {
    for (int i = t; i < V; i += NT) f(i, x[i]);
  }
}

// A row as the fast path sees it: all its values, or those that the slices list, a thread's share of them in its registers
constexpr int OWN = MAX_SLICES * LISTED / NT;
struct Row {
  const float* x;
  int V;
  bool listed;
  SampleEntry own[OWN];   // i < 0: none
};

template <typename F>
__device__ __forceinline__ void for_near(const Row& r, F f) {
  if (!r.listed) {
    for_row(r.x, r.V, f);
    return;
  }
#pragma unroll
  for (int j = 0; j < OWN; ++j)
    if (r.own[j].i >= 0) f(r.own[j].i, r.own[j].v);
}

__device__ __forceinline__ ArgMax am_max(ArgMax a, ArgMax b) {
  return (b.v > a.v || (b.v == a.v && b.i < a.i)) ? b : a;
}

__device__ __forceinline__ ArgMax wave_argmax(ArgMax a) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    ArgMax b;
    b.v = __shfl_xor(a.v, o, 64);
    b.i = __shfl_xor(a.i, o, 64);
    a = am_max(a, b);
  }
  return a;
}

__device__ ArgMax block_argmax(ArgMax a, ArgMax* red) {
  a = wave_argmax(a);
  __syncthreads();
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = a;
  __syncthreads();
  ArgMax r = red[0];
  for (int k = 1; k < NT / 64; ++k) r = am_max(r, red[k]);
  return r;
}

__device__ __forceinline__ int dist_bin(float d) { return min((int)(d * DSCALE), NBINS - 1); }

// exp(v - M) <= 1 in units of 2^-40; a row's total stays below 2^58
__device__ __forceinline__ uint64_t fixed_mass(float dv) {
  return (uint64_t)(__expf(dv) * (float)FIX);
}
template <bool MASS>
__device__ __forceinline__ uint64_t to_fixed(float w) {
  return MASS ? (uint64_t)((double)w * FIX) : (uint64_t)w;
}
template <bool MASS>
__device__ __forceinline__ float from_fixed(uint64_t q) {
  return MASS ? (float)((double)q * (1.0 / FIX)) : (float)q;
}

// Fast threshold: the largest key thr >= floor_key whose weight {key >= thr} reaches target,
// weight = 1 per token (MASS = false: top-k) or exp(v - M) (MASS = true: top-p). Also returns
// the probability mass (relative to exp(M)) kept by that threshold. Returns false, uniformly
// over the workgroup, when the caller must take the radix descent instead.
template <bool MASS>
__device__ __forceinline__ bool fast_select(const Row& row, float inv_t, float M,
                            uint32_t floor_key, float target, Smem& sm, uint32_t* thr_out,
                            float* kept_out) {
  const int t = threadIdx.x, lane = t & 63;
  for (int i = t; i < NBINS; i += NT) sm.u.s.h.q[i] = 0ull;
  if (t == 0) sm.ncand = 0;
  __syncthreads();
  for_near(row, [&](int, float raw) {
    const float v = raw * inv_t;
    const float d = M - v;
    if (d < DRANGE && fkey(v) >= floor_key)
      atomicAdd(&sm.u.s.h.q[NBINS - 1 - dist_bin(d)], MASS ? fixed_mass(v - M) : 1ull);
  });
  __syncthreads();
  uint64_t above_q;
  const int bin = find_crossing<uint64_t>(sm.u.s.h.q, NBINS, to_fixed<MASS>(target), &above_q,
                                          sm.u.s.scan.q, sm);
  if (bin < 0) return false;
  const float above = from_fixed<MASS>(above_q);
  const int cbin = NBINS - 1 - bin;  // crossing bin in distance order

  // gather the crossing bin's keys (wave-aggregated slots), and the mass of the bins above it
  float m_above = 0.f;
  for_near(row, [&](int, float raw) {
    const float v = raw * inv_t;
    const float d = M - v;
    const uint32_t key = fkey(v);
    bool want = false;
    if (d < DRANGE && key >= floor_key) {
      const int db = dist_bin(d);
      if (db < cbin) m_above += __expf(v - M);
      want = db == cbin;
    }
    const uint64_t m = __ballot(want);
    if (m != 0) {
      const int leader = __ffsll((unsigned long long)m) - 1;
      int base = 0;
      if (lane == leader) base = atomicAdd(&sm.ncand, __popcll(m));
      base = __shfl(base, leader, 64);
      if (want) {
        const int pos = base + __popcll(m & ((1ull << lane) - 1ull));
        if (pos < CAP) sm.u.s.cand[pos] = key;
      }
    }
  });
  m_above = block_sum(m_above, sm.red);  // starts and ends with a barrier
  const int n = sm.ncand;
  if (n > CAP || n == 0) return false;
  int sn = 2;
  while (sn < n) sn <<= 1;
  for (int i = n + t; i < sn; i += NT) sm.u.s.cand[i] = 0u;  // pads sort below every real key
  // bitonic sort, ascending
  for (int size = 2; size <= sn; size <<= 1)
    for (int stride = size >> 1; stride > 0; stride >>= 1) {
      __syncthreads();
      if (t < (sn >> 1)) {
        const int i = 2 * t - (t & (stride - 1));
        const int j = i + stride;
        const uint32_t a = sm.u.s.cand[i], b = sm.u.s.cand[j];
        if ((a > b) == ((i & size) == 0)) {
          sm.u.s.cand[i] = b;
          sm.u.s.cand[j] = a;
        }
      }
    }
  __syncthreads();
  const int lo = sn - n;  // first real key
  for (int i = t; i < sn; i += NT)
    sm.u.s.h.w[i] = i < lo ? 0.f : (MASS ? __expf(fval(sm.u.s.cand[i]) - M) : 1.f);
  __syncthreads();
  float above2;
  int c = find_crossing<float>(sm.u.s.h.w, sn, target - above, &above2, sm.u.s.scan.f, sm);
  if (c < lo) c = lo;  // rounding: keep the whole bin
  const uint32_t thr = sm.u.s.cand[c];
  float km = 0.f;
  for (int i = lo + t; i < sn; i += NT)
    if (sm.u.s.cand[i] >= thr) km += __expf(fval(sm.u.s.cand[i]) - M);
  km = block_sum(km, sm.red);
  *thr_out = thr;
  *kept_out = m_above + km;
  return true;
}

// Exact radix descent (11/11/10 bits of the key) on counts (top-k) or fixed-point mass (top-p,
// restricted to key >= floor_key). Used when the fast path declines.
template <bool MASS>
__device__ __forceinline__ uint32_t radix_select(const float* __restrict__ x, int V, float inv_t,
                                                 float M, uint32_t floor_key, float target, Smem& sm) {
  const int t = threadIdx.x;
  uint32_t prefix = 0, mask = 0;
  uint64_t remaining = to_fixed<MASS>(target);
  for (int lvl = 0; lvl < 3; ++lvl) {
    for (int i = t; i < NBINS; i += NT) sm.u.s.h.q[i] = 0ull;
    __syncthreads();
    const int sh = lvl == 0 ? 21 : lvl == 1 ? 10 : 0;
    const uint32_t bm = lvl == 2 ? 0x3ffu : 0x7ffu;
    for_row(x, V, [&](int, float raw) {
      const float v = raw * inv_t;
      const uint32_t key = fkey(v);
      if ((key & mask) == prefix && key >= floor_key)
        atomicAdd(&sm.u.s.h.q[(key >> sh) & bm], MASS ? fixed_mass(v - M) : 1ull);
    });
    __syncthreads();
    uint64_t above;
    int bin = find_crossing<uint64_t>(sm.u.s.h.q, NBINS, remaining, &above, sm.u.s.scan.q, sm);
    if (bin < 0) {  // target beyond total (rounding): take the lowest populated bin
      bin = 0;
      above -= sm.u.s.h.q[0];
    }
    remaining -= above;
    prefix |= ((uint32_t)bin) << sh;
    mask |= bm << sh;
    __syncthreads();
  }
  return prefix;
}
}  // namespace

// One slice of a row: its largest value and where, the sum of exp(v - it) over the slice, and unless the row is greedy its values near
// the largest one: less than DRANGE below it, or a half, a quarter, an eighth of that if they are too many. (What counts is DRANGE below the
// row's largest value; a slice of a smaller one need not reach as far.)
__global__ void __launch_bounds__(256) sample_slices_kernel(const float* __restrict__ logits, int V, const float* __restrict__ temperature,
                                                            const int32_t* __restrict__ top_k, const float* __restrict__ penalty,
                                                            SampleSlice* __restrict__ slices, SampleEntry* __restrict__ list) {
  __shared__ ArgMax ared[4];
  __shared__ float red[4];
  __shared__ int counts[4][4];
  const int row = blockIdx.y, t = threadIdx.x;
  if (penalty && penalty[row] != 1.f) return;   // sample_kernel changes the row first
  const float* x = logits + (int64_t)row * V;
  const float temp = temperature[row];
  const bool greedy = !(temp > 0.f) || (top_k && top_k[row] == 1);
  const float inv_t = greedy ? 1.f : 1.f / temp;
  const int b = blockIdx.x * SLICE;
  float raw[8];
  const bool vec = (V & 3) == 0;   // rows at 16-byte addresses
  auto at = [&](int j) { return vec ? b + 1024 * (j >> 2) + 4 * t + (j & 3) : b + 256 * j + t; };
  if (vec) {
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const float4 v = at(4 * u) < V ? *reinterpret_cast<const float4*>(x + at(4 * u)) : make_float4(-INFINITY, -INFINITY, -INFINITY, -INFINITY);
      raw[4 * u] = v.x;
      raw[4 * u + 1] = v.y;
      raw[4 * u + 2] = v.z;
      raw[4 * u + 3] = v.w;
    }
  } else {
#pragma unroll
    for (int j = 0; j < 8; ++j) raw[j] = at(j) < V ? x[at(j)] : -INFINITY;
  }
  ArgMax am{-INFINITY, 0x7fffffff};
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    const float v = raw[j] * inv_t;
    if (v > am.v) am = ArgMax{v, at(j)};   // a thread's values in ascending order
  }
  am = wave_argmax(am);
  if ((t & 63) == 0) ared[t >> 6] = am;
  __syncthreads();
  am = am_max(am_max(ared[0], ared[1]), am_max(ared[2], ared[3]));
  SampleEntry* const own = list + ((int64_t)row * gridDim.x + blockIdx.x) * LISTED;
  float z = 0.f, range = 0.f;
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    const float v = raw[j] * inv_t;
    if (v > -INFINITY) z += v == am.v ? 1.f : __expf(v - am.v);
  }
  int count = 0;
  if (!greedy) {
    const int w = t >> 6, lane = t & 63;
    int n[4] = {0, 0, 0, 0};
#pragma unroll
    for (int j = 0; j < 8; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) n[r] += __popcll(__ballot(am.v - raw[j] * inv_t < DRANGE / (1 << r)));
    if (lane < 4) counts[w][lane] = lane == 0 ? n[0] : lane == 1 ? n[1] : lane == 2 ? n[2] : n[3];
    __syncthreads();
    // places by wave, then j, then lane: the passes over the lists add up in their order, so it is the same at every call
    int place = 0;
#pragma unroll
    for (int r = 3; r >= 0; --r) {
      const int all = counts[0][r] + counts[1][r] + counts[2][r] + counts[3][r];
      if (all > LISTED) continue;
      range = DRANGE / (1 << r);
      count = all;
      place = (w > 0 ? counts[0][r] : 0) + (w > 1 ? counts[1][r] : 0) + (w > 2 ? counts[2][r] : 0);
    }
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const bool in = am.v - raw[j] * inv_t < range;
      const uint64_t m = __ballot(in);
      if (in) own[place + __popcll(m & ((1ull << lane) - 1ull))] = SampleEntry{raw[j], at(j)};
      place += __popcll(m);
    }
  }
  z = block_sum(z, red);
  if (t == 0) slices[(int64_t)row * gridDim.x + blockIdx.x] = SampleSlice{am.v, z, am.i, count, range};
}

__global__ void __launch_bounds__(NT) sample_kernel(
    float* __restrict__ logits, int V, const float* __restrict__ temperature,
    const int32_t* __restrict__ top_k, const float* __restrict__ top_p,
    const float* __restrict__ rep_penalty, const int32_t* __restrict__ history, int hist_len,
    const int64_t* __restrict__ seeds, const int64_t* __restrict__ steps,
    const SampleSlice* __restrict__ slices, const SampleEntry* __restrict__ list, int nslices,
    int32_t* __restrict__ out_tok, float* __restrict__ out_logprob) {
  __shared__ Smem sm;

  const int row = blockIdx.x, t = threadIdx.x;
  float* x = logits + (int64_t)row * V;
  const float pen = rep_penalty ? rep_penalty[row] : 1.f;

  const bool changed = pen != 1.f && history != nullptr;
  if (changed) {
    for (int i = t; i < 8192; i += NT) sm.u.bitmap[i] = 0;
    __syncthreads();
    const int32_t* hs = history + (int64_t)row * hist_len;
    for (int i = t; i < hist_len; i += NT) {
      const int tok = hs[i];
      if (tok >= 0 && tok < V) atomicOr(&sm.u.bitmap[tok >> 5], 1u << (tok & 31));
    }
    __syncthreads();
    for (int i = t; i < V; i += NT)
      if (sm.u.bitmap[i >> 5] & (1u << (i & 31))) {
        const float v = x[i];
        x[i] = v > 0.f ? v / pen : v * pen;
      }
    __syncthreads();
  }

  const float temp = temperature[row];
  const int k = top_k ? top_k[row] : 0;
  const float p = top_p ? top_p[row] : 1.f;
  const bool greedy = !(temp > 0.f) || k == 1;
  const float inv_t = greedy ? 1.f : 1.f / temp;

  // argmax and the partition function: the slices', or in one pass (online: per-thread running max + rescaled sum)
  ArgMax am{-INFINITY, 0x7fffffff};
  float z = 0.f;
  Row near;
  near.x = x;
  near.V = V;
  near.listed = false;
  float range = DRANGE;   // of this thread's slice values less than this below its largest one are listed
  if (nslices > 0 && !changed) {
    const SampleSlice* const own = slices + (int64_t)row * nslices;
#pragma unroll
    for (int j = 0; j < OWN; ++j) {
      const int e = t + j * NT;
      near.own[j].i = -1;
      if (e < nslices * LISTED && !greedy) {
        const SampleEntry v = list[(int64_t)row * nslices * LISTED + e];
        near.own[j] = SampleEntry{v.v, e % LISTED < own[e / LISTED].n ? v.i : -1};
      }
    }
    if (t < nslices) {
      am = ArgMax{own[t].m, own[t].i};
      z = own[t].z;
      range = own[t].range;
    }
  } else {
    for_row(x, V, [&](int i, float raw) {
      const float v = raw * inv_t;
      if (v > am.v) {
        z = z * __expf(am.v - v) + 1.f;
        am = ArgMax{v, i};
      } else if (v > -INFINITY) {
        z += __expf(v - am.v);
        if (v == am.v && i < am.i) am.i = i;
      }
    });
  }
  const float m_thr = am.v;
  am = block_argmax(am, sm.ared);
  if (am.i == 0x7fffffff) am.i = 0;   // a row of NaN or -inf alone
  const float M = am.v;
  // Every value less than DRANGE below M is listed, as the passes work that distance out: a slice's own list that goes so far does (no value
  // is nearer to M than to the slice's largest), a shorter one by a margin for the roundings. (M - DRANGE is M itself from 2^28 up.)
  near.listed = __syncthreads_and(nslices > 0 && !changed && (range == DRANGE || M - m_thr + range >= DRANGE * 1.00001f));
  const float Z = block_sum(m_thr == -INFINITY ? 0.f : m_thr == M ? z : z * __expf(m_thr - M), sm.red);
  const float logZ = __logf(Z);

  if (greedy) {
    if (t == 0) {
      out_tok[row] = am.i;
      out_logprob[row] = 0.f - logZ;  // x[am] * inv_t - M == 0
    }
    return;
  }

  uint32_t thr = 0u;  // keep tokens with fkey(x * inv_t) >= thr
  float kept_mass = Z;
  if (k > 0 && k < V) {
    if (!fast_select<false>(near, inv_t, M, 0u, (float)k, sm, &thr, &kept_mass)) {
      thr = radix_select<false>(x, V, inv_t, M, 0u, (float)k, sm);
      float km = 0.f;
      for_row(x, V, [&](int, float raw) {
        const float v = raw * inv_t;
        if (fkey(v) >= thr) km += __expf(v - M);
      });
      kept_mass = block_sum(km, sm.red);
    }
  }
  if (p < 1.f) {
    uint32_t tp;
    float unused;
    if (!fast_select<true>(near, inv_t, M, thr, p * kept_mass, sm, &tp, &unused))
      tp = radix_select<true>(x, V, inv_t, M, thr, p * kept_mass, sm);
    thr = tp > thr ? tp : thr;
  }

  // Gumbel-max draw over kept tokens
  const uint64_t seed = (uint64_t)seeds[row];
  const uint64_t base = (uint64_t)steps[row] * (uint64_t)V;
  ArgMax best{-INFINITY, 0x7fffffff};
  if (!(M - fval(thr) < DRANGE)) near.listed = false;   // keeps values that the lists leave out (thr 0 is NaN's key: all)
  for_near(near, [&](int i, float raw) {
    const float v = raw * inv_t;
    if (fkey(v) >= thr) {
      const float u = hash_uniform(seed, base + i);
      const float g = -__logf(-__logf(u));
      best = am_max(best, ArgMax{v + g, i});
    }
  });
  best = block_argmax(best, sm.ared);
  if (t == 0) {
    const int tok = best.i == 0x7fffffff ? am.i : best.i;
    out_tok[row] = tok;
    out_logprob[row] = x[tok] * inv_t - M - logZ;
  }
}

// Slices of a row, 0: none. Their launch costs 3 us and up, and where the lists are of no use or too short the passes over the row come
// besides: short rows are through as soon, and many rows fill the chip by themselves. The line is where that worst case costs nothing, but
// for up to 4 rows of 16 to 23 slices, where it costs 1 to 4 % and the others gain 40. Both, us, without / with: (a) at temperature 0.2 and
// top-p 0.7, the servers' defaults, (b) greedy, (c) normal logits of deviation 3 at temperature 1, top-p 0.9, where lists are of no use:
//   rows x values    (a)          (b)          (c)             rows x values    (a)          (b)          (c)
//    1 x  24,576  20.5  16.9    7.0   7.9   31.5  34.0          1 x 128,256  53.0  19.0   19.5   7.9    113   104
//    1 x  32,000  24.1  17.2    8.0   7.9   37.9  39.4         16 x 128,256  54.0  20.4   20.1   9.0    114   107
//   16 x  32,000  25.2  26.8    8.4   8.4   39.2  40.8         64 x 128,256  60.3  29.0   21.4  14.1    119   119
//    8 x  49,152  30.3  17.7   10.5   8.4   52.7  52.3        128 x 128,256  66.9  39.0   22.7  21.0    123   131
//   48 x  49,152  31.8  33.0   10.6   9.3   53.6  54.9         32 x 256,000  92.0  31.2   35.2  13.9    213   200
//   32 x  65,536  34.6  19.3   12.2   8.9   64.3  63.5        128 x 256,000   107  59.8   37.6  32.3    219   232
//   48 x 100,352  45.6  45.0   16.4  11.3   90.5  90.8
// The partition function adds up in another order with slices than without: a row's log-probability, and with it the target of its top-p, can
// differ in the last bit between a batch that is sliced and one that is not.
int sample_slices(int B, int V) {
  const int n = (V + SLICE - 1) / SLICE;
  const int most = n < 16 || n > MAX_SLICES ? 0 : n < 24 ? 4 : n < 60 ? n : 4096 / n;   // rows
  return B <= most ? n : 0;
}
int64_t sample_scratch(int B, int V) { return (int64_t)B * sample_slices(B, V) * (sizeof(SampleSlice) + LISTED * sizeof(SampleEntry)); }

void launch_sample(float* logits, int B, int V, const float* temperature, const int32_t* top_k,
                   const float* top_p, const float* rep_penalty, const int32_t* history,
                   int hist_len, const int64_t* seeds, const int64_t* steps, void* scratch, int32_t* out_tok,
                   float* out_logprob, hipStream_t stream) {
  if (B == 0) return;
  const int n = scratch ? sample_slices(B, V) : 0;
  SampleEntry* const list = static_cast<SampleEntry*>(scratch);
  SampleSlice* const slices = reinterpret_cast<SampleSlice*>(list + (int64_t)B * n * LISTED);
  if (n > 0)
    sample_slices_kernel<<<dim3(n, B), 256, 0, stream>>>(logits, V, temperature, top_k, history ? rep_penalty : nullptr, slices, list);
  sample_kernel<<<B, NT, 0, stream>>>(logits, V, temperature, top_k, top_p, rep_penalty, history,
                                      hist_len, seeds, steps, slices, list, n, out_tok, out_logprob);
}

}  // namespace nga
