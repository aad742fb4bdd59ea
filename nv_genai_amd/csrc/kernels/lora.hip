// Gradients of a low-rank adapter, y = x w^T + scale h b^T with h = x a^T (x [T, K], a [r, K], b [N, r], r <= 64), beside w's:
//   dh = scale dy b,  db = scale dy^T h,  da = dh^T x,  dx += dh a
// Each of the four products has one side of r: it reads dy, x or dx once and computes next to nothing, so it is bound by memory
// and, at a few thousand rows, by launches and by how many CUs it occupies. At T 1,024, K 4,096, N 6,144, r 32 library products
// (64 to 96 workgroups each, with their scaling, casts and a copy of dx around them, ten launches) took 74 us; these three launches
// take 21, of which the bytes are 8. At 16,384 rows 195 for 308. All sizes measured are faster: T 1 to 16,384, K 768 to 14,336, N 2,304
// to 28,672, r 8 to 64; the least, T 16,384 and N 28,672, 522 for 534.
//   1. dh in parts of N's columns, beside db;  2. the parts' sum, as bf16;  3. dx, beside da
// A sum over rows has a workgroup for 64 columns; where these are few and the rows many they are sliced, and the slices added up in
// launch 2 (db) or in a fourth (da): K 768, N 2,304, T 16,384 179 us without, 60 with slices of 1,024 rows or more; slices of 512
// lose at 1,024 rows (24 for 21) what they gain nowhere.
// The operands that a product over rows needs transposed (dy and h for db, x and dh for da, b for dh, a for dx) are read as they
// lie, 8 rows of E neighbouring columns a lane, and transposed in registers: fragment e then holds columns e, E + e, 2 E + e, ...
// in the place of 16 neighbours, and a lane's results are neighbours again. No LDS but for the sum over a workgroup's waves.
#include "common.h"
#include "kernels.h"

#include <algorithm>

namespace nga {

namespace {

constexpr int WAVES = 8;
constexpr int COLS = 64;     // of a workgroup that sums over rows
constexpr int SLICE = 1024;  // rows of one that sums over rows, at least
constexpr int ROWS = 64;     // of one that sums over columns, and of one of dx

// f[e]: rows r0 + 8 (lane / 16) + 0 .. 7 of column c0 + E (lane % 16) + e; zero outside [R, C], where C % E == 0
template <int E>
__device__ __forceinline__ void load_t(const uint16_t* p, int64_t ld, int64_t r0, int64_t R, int64_t c0, int64_t C, int lane,
                                       bf16x8 (&f)[E]) {
  const int64_t c = c0 + E * (lane & 15), r = r0 + 8 * (lane >> 4);
  typedef uint16_t vec __attribute__((ext_vector_type(E == 1 ? 2 : E)));   // one value alone is in no vector
  const uint16_t* at = p + (c < C ? c : 0);
  u16x8 t[E];
  uint16_t v[8][E];
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const uint16_t* row = at + (r + i < R ? r + i : R - 1) * ld;
    if constexpr (E == 1) {
      v[i][0] = *row;
    } else {
      const vec x = *reinterpret_cast<const vec*>(row);
#pragma unroll
      for (int e = 0; e < E; ++e) v[i][e] = x[e];
    }
  }
#pragma unroll
  for (int e = 0; e < E; ++e)
#pragma unroll
    for (int i = 0; i < 8; ++i) t[e][i] = c < C && r + i < R ? v[i][e] : (uint16_t)0;
#pragma unroll
  for (int e = 0; e < E; ++e) f[e] = __builtin_bit_cast(bf16x8, t[e]);
}

// acc of all waves, summed in wave 0 in a fixed order
template <int E>
__device__ __forceinline__ void sum_waves(f32x4 (&acc)[4][E], float* red, int w, int lane) {
#pragma unroll
  for (int s = WAVES / 2; s; s >>= 1) {
    f32x4* own = reinterpret_cast<f32x4*>(red) + (w % s) * 4 * E * 64 + lane;
    if (w >= s && w < 2 * s)
#pragma unroll
      for (int i = 0; i < 4 * E; ++i) own[i * 64] = acc[i / E][i % E];
    __syncthreads();
    if (w < s)
#pragma unroll
      for (int i = 0; i < 4 * E; ++i) acc[i / E][i % E] += own[i * 64];
    __syncthreads();
  }
}

// out = scale m^T s over rows first .. T for COLS columns of m [., C], s [., r]: [C, r], or turned [r, C]
template <int E, bool TURNED>
__device__ void over_rows(const uint16_t* m, const uint16_t* s, int64_t lds, int64_t first, int64_t T, int64_t C, int r, float scale,
                          float* out, int64_t c0, float* red) {
  const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
  f32x4 acc[4][E] = {};
#pragma unroll 2
  for (int64_t t0 = first + 32 * w; t0 < T; t0 += 32 * WAVES) {
    bf16x8 fm[4], fs[E];
    load_t<4>(m, C, t0, T, c0, C, lane, fm);
    load_t<E>(s, lds, t0, T, 0, r, lane, fs);
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int e = 0; e < E; ++e) acc[i][e] = mfma16(fm[i], fs[e], acc[i][e]);
  }
  sum_waves<E>(acc, red, w, lane);
  const int j0 = E * (lane & 15);
  if (w || j0 >= r) return;
#pragma unroll
  for (int v = 0; v < 4; ++v) {
    const int64_t c = c0 + 16 * (lane >> 4) + 4 * v;   // C % 4 == 0
    if (c >= C) continue;
    if constexpr (TURNED) {
#pragma unroll
      for (int e = 0; e < E; ++e)
        *reinterpret_cast<f32x4*>(out + (j0 + e) * C + c) =
            (f32x4){scale * acc[0][e][v], scale * acc[1][e][v], scale * acc[2][e][v], scale * acc[3][e][v]};
    } else {
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int e = 0; e < E; ++e) out[(c + i) * r + j0 + e] = scale * acc[i][e][v];
    }
  }
}

// part [T, 16 E] = m b for ROWS rows of m [T, N] and its columns n0 .. n1, b [N, r]
template <int E>
__device__ void over_cols(const uint16_t* m, const uint16_t* b, int64_t T, int64_t N, int r, int64_t t0, int64_t n0, int64_t n1,
                          float* part, float* red) {
  const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
  f32x4 acc[4][E] = {};
#pragma unroll 2
  for (int64_t n = n0 + 32 * w; n < n1; n += 32 * WAVES) {
    bf16x8 fm[4], fb[E];
    const int64_t k = n + 8 * (lane >> 4);   // N % 8 == 0
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int64_t t = t0 + 16 * i + (lane & 15);
      const u16x8 v = load8(m + (t < T ? t : T - 1) * N + (k < N ? k : 0));
      fm[i] = __builtin_bit_cast(bf16x8, t < T && k < N ? v : (u16x8)(0));
    }
    load_t<E>(b, r, n, N, 0, r, lane, fb);
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int e = 0; e < E; ++e) acc[i][e] = mfma16(fm[i], fb[e], acc[i][e]);
  }
  sum_waves<E>(acc, red, w, lane);
  if (w) return;
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int64_t t = t0 + 16 * i + 4 * (lane >> 4) + v;
#pragma unroll
      for (int e = 0; e < E; ++e)
        if (t < T) part[t * 16 * E + E * (lane & 15) + e] = acc[i][e][v];
    }
}

template <int E>
__global__ __launch_bounds__(64 * WAVES) void lora_dy_kernel(LoraGrads p) {
  __shared__ __align__(16) float red[WAVES / 2 * 4 * E * 64 * 4];
  const int64_t g = blockIdx.x, nd = p.part ? (p.T + ROWS - 1) / ROWS * p.parts : 0;
  if (g < nd) {   // the row workgroups first: they read more
    const int64_t q = g % p.parts, n0 = q * p.chunk;
    over_cols<E>(p.dy, p.b, p.T, p.N, p.r, g / p.parts * ROWS, n0, n0 + p.chunk < p.N ? n0 + p.chunk : p.N,
                 p.part + q * p.T * 16 * E, red);
  } else {
    const int64_t q = (g - nd) % p.slices_n, t0 = q * p.slice_n;
    over_rows<E, false>(p.dy, p.h, p.r, t0, min(t0 + p.slice_n, p.T), p.N, p.r, p.scale,
                        p.slices_n > 1 ? p.sums + q * p.N * p.r : p.db, (g - nd) / p.slices_n * COLS, red);
  }
}

// dh [T, 32 or 64], zero from column 16 E on; behind them out [n4 float4] as the sum of its slices
template <int E>
__global__ __launch_bounds__(256) void lora_sum_kernel(LoraGrads p, int64_t rows, float* out, int64_t n4, int slices) {
  constexpr int W = E == 4 ? 64 : 32;
  int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  f32x4 s = {};
  if (i < rows * (W / 4)) {
    const int64_t t = i / (W / 4);
    const int j = i % (W / 4) * 4;
    if (j < 16 * E) {
      const float* at = p.part + t * 16 * E + j;
#pragma unroll 4
      for (int q = 0; q < p.parts; ++q) s += *reinterpret_cast<const f32x4*>(at + q * p.T * 16 * E);
    }
    u16x4 o;
#pragma unroll
    for (int k = 0; k < 4; ++k) o[k] = f2bf(p.scale * s[k]);
    *reinterpret_cast<u16x4*>(p.dh + t * W + j) = o;
  } else if ((i -= rows * (W / 4)) < n4) {
    for (int q = 0; q < slices; ++q) s += reinterpret_cast<const f32x4*>(p.sums)[q * n4 + i];
    reinterpret_cast<f32x4*>(out)[i] = s;
  }
}

// dx += dh a for ROWS rows and 64 columns a wave
template <int E>
__device__ void add_dx(const LoraGrads& p, int64_t t0, int64_t c0) {
  constexpr int W = E == 4 ? 64 : 32;
  const int lane = threadIdx.x & 63;
  if (c0 >= p.K) return;
  const int64_t c = c0 + 16 * (lane >> 4);
  bf16x8 fa[W / 32][4];
#pragma unroll
  for (int k = 0; k < W / 32; ++k) load_t<4>(p.a, p.K, 32 * k, p.r, c0, p.K, lane, fa[k]);
#pragma unroll
  for (int i = 0; i < ROWS / 16; ++i) {
    const int64_t t = t0 + 16 * i + (lane & 15), tc = t < p.T ? t : p.T - 1;
    uint16_t* at = p.dx + tc * p.K;
    u16x8 x[2];
#pragma unroll
    for (int k = 0; k < 2; ++k) x[k] = load8(at + (c + 8 * k < p.K ? c + 8 * k : 0));
    f32x4 acc[4] = {};
#pragma unroll
    for (int k = 0; k < W / 32; ++k) {
      const bf16x8 fd = __builtin_bit_cast(bf16x8, load8(p.dh + tc * W + 32 * k + 8 * (lane >> 4)));
#pragma unroll
      for (int j = 0; j < 4; ++j) acc[j] = mfma16(fa[k][j], fd, acc[j]);
    }
#pragma unroll
    for (int k = 0; k < 2; ++k) {
#pragma unroll
      for (int j = 0; j < 8; ++j) x[k][j] = f2bf(bf2f(x[k][j]) + acc[j % 4][2 * k + j / 4]);
      if (t < p.T && c + 8 * k < p.K) *reinterpret_cast<u16x8*>(at + c + 8 * k) = x[k];
    }
  }
}

template <int E>
__global__ __launch_bounds__(64 * WAVES) void lora_x_kernel(LoraGrads p) {
  __shared__ __align__(16) float red[WAVES / 2 * 4 * E * 64 * 4];
  const int64_t g = blockIdx.x, nc = p.da ? (p.K + COLS - 1) / COLS * p.slices_k : 0;
  if (g < nc) {   // the longer ones first
    const int64_t q = g % p.slices_k, t0 = q * p.slice_k;
    over_rows<E, true>(p.x, p.dh, E == 4 ? 64 : 32, t0, min(t0 + p.slice_k, p.T), p.K, p.r, 1.f,
                       p.slices_k > 1 ? p.sums + q * p.K * p.r : p.da, g / p.slices_k * COLS, red);
  } else {
    const int64_t across = (p.K + 64 * WAVES - 1) / (64 * WAVES), q = g - nc;
    add_dx<E>(p, q / across * ROWS, (q % across) * 64 * WAVES + (threadIdx.x >> 6) * 64);
  }
}

template <int E>
void launch(const LoraGrads& p, hipStream_t st) {
  const int64_t tiles = (p.T + ROWS - 1) / ROWS;
  const auto sum = [&](int64_t rows, float* out, int64_t n4, int slices) {
    const int64_t n = rows * (E == 4 ? 16 : 8) + n4;
    if (n) lora_sum_kernel<E><<<dim3((unsigned)((n + 255) / 256)), 256, 0, st>>>(p, rows, out, n4, slices);
  };
  const int64_t one = (p.part ? tiles * p.parts : 0) + (p.db ? (p.N + COLS - 1) / COLS * p.slices_n : 0);
  if (one) lora_dy_kernel<E><<<dim3((unsigned)one), 64 * WAVES, 0, st>>>(p);
  sum(p.part ? p.T : 0, p.db, p.db && p.slices_n > 1 ? p.N * p.r / 4 : 0, p.slices_n);
  const int64_t two = p.part ? (p.da ? (p.K + COLS - 1) / COLS * p.slices_k : 0) +
                                   (p.dx ? tiles * ((p.K + 64 * WAVES - 1) / (64 * WAVES)) : 0) : 0;
  if (two) lora_x_kernel<E><<<dim3((unsigned)two), 64 * WAVES, 0, st>>>(p);
  sum(0, p.da, p.da && p.slices_k > 1 ? p.K * p.r / 4 : 0, p.slices_k);
}

// rows of a slice of a sum over T rows for C columns
int64_t slice(int64_t T, int64_t C) {
  const int64_t groups = (C + COLS - 1) / COLS, n = std::max<int64_t>(1, std::min((256 + groups - 1) / groups, T / SLICE));
  return (T + n * 32 * WAVES - 1) / (n * 32 * WAVES) * 32 * WAVES;
}

}  // namespace

void lora_plan(LoraGrads& p) {
  // columns of dy to a workgroup of dh: some 128 workgroups, beside those of db, of at least one step a wave
  const int64_t tiles = (p.T + ROWS - 1) / ROWS, want = (128 + tiles - 1) / tiles, least = 32 * WAVES;
  p.chunk = (p.N + want * least - 1) / (want * least) * least;
  p.parts = (int)((p.N + p.chunk - 1) / p.chunk);
  p.slice_n = slice(p.T, p.N);
  p.slice_k = slice(p.T, p.K);
  p.slices_n = (int)((p.T + p.slice_n - 1) / p.slice_n);
  p.slices_k = (int)((p.T + p.slice_k - 1) / p.slice_k);
}

void launch_lora_grads(const LoraGrads& p, hipStream_t st) {
  if (p.r <= 16) launch<1>(p, st);
  else if (p.r <= 32) launch<2>(p, st);
  else launch<4>(p, st);
}

}  // namespace nga
