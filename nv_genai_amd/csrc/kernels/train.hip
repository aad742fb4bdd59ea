// Training steps around the matrix products: norms with their residual, activations, rotation, cross entropy and column
// sums. Activations bf16, statistics, sums and weights' gradients fp32. Each takes the place of a chain of single
// torch operations (a norm and its residual: 10 launches forward, 14 backward; a rotation: 14 each way).
//
// Steps marked "as written" round where that chain rounds, in its order, without contraction: their results are its bits (one
// other bit in an activation is an independent rounding error of the whole gradient a few layers later). The means and sums
// over a row that such a step needs are left to torch, whose order of summation is its own. Column sums, the gradients of
// norms' weights and biases, are in this file's order, and so within fp32 rounding of torch's.
#include "common.h"
#include "kernels.h"

namespace nga {

namespace {
// single roundings: nothing is contracted to an fma
__device__ __forceinline__ float mul(float a, float b) {
#pragma clang fp contract(off)
  return a * b;
}
__device__ __forceinline__ float add(float a, float b) {
#pragma clang fp contract(off)
  return a + b;
}

// weights and biases are fp32 masters or bf16
__device__ __forceinline__ void ldw8(const void* p, bool f32, int64_t i, float (&v)[8]) {
  if (f32) {
    const f32x4 a = *reinterpret_cast<const f32x4*>(static_cast<const float*>(p) + i);
    const f32x4 b = *reinterpret_cast<const f32x4*>(static_cast<const float*>(p) + i + 4);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      v[j] = a[j];
      v[4 + j] = b[j];
    }
  } else {
    const u16x8 a = load8(static_cast<const uint16_t*>(p) + i);
#pragma unroll
    for (int j = 0; j < 8; ++j) v[j] = bf2f(a[j]);
  }
}

__device__ __forceinline__ void unpack8(u16x8 a, float (&v)[8]) {
#pragma unroll
  for (int j = 0; j < 8; ++j) v[j] = bf2f(a[j]);
}

__device__ __forceinline__ u16x8 pack8(const float (&v)[8]) {
  u16x8 o;
#pragma unroll
  for (int j = 0; j < 8; ++j) o[j] = f2bf(v[j]);
  return o;
}

__device__ __forceinline__ void store8f(float* p, const float (&v)[8]) {
  *reinterpret_cast<f32x4*>(p) = (f32x4){v[0], v[1], v[2], v[3]};
  *reinterpret_cast<f32x4*>(p + 4) = (f32x4){v[4], v[5], v[6], v[7]};
}

}  // namespace

// ---------------------------------------------------------------- RMS norm
// as written: xn = x + o (o null: x itself, not written), sq = xn^2 in fp32
__global__ void __launch_bounds__(256) rms_sq_kernel(const uint16_t* __restrict__ x, const uint16_t* __restrict__ o, int64_t n8,
                                                     uint16_t* __restrict__ xn, float* __restrict__ sq) {
  for (int64_t i = blockIdx.x * 256ll + threadIdx.x; i < n8; i += gridDim.x * 256ll) {
    float v[8];
    unpack8(load8(x + 8 * i), v);
    if (o) {
      float d[8];
      unpack8(load8(o + 8 * i), d);
#pragma unroll
      for (int j = 0; j < 8; ++j) v[j] += d[j];
      const u16x8 s = pack8(v);
      store8(xn + 8 * i, s);
      unpack8(s, v);
    }
#pragma unroll
    for (int j = 0; j < 8; ++j) v[j] = mul(v[j], v[j]);
    store8f(sq + 8 * i, v);
  }
}

// as written: y = (xn * r) * w, r = rsqrt(ms + eps), ms [R] the means of sq
__global__ void __launch_bounds__(1024) rms_apply_kernel(const uint16_t* __restrict__ xn, const float* __restrict__ ms,
                                                         const void* __restrict__ w, int w32, float eps, int H,
                                                         uint16_t* __restrict__ y, float* __restrict__ rstd) {
  const int64_t row = blockIdx.x;
  const int c = threadIdx.x * 8;
  const float r = (float)(1. / sqrt((double)add(ms[row], eps)));   // torch's is rounded correctly, the instruction is not
  if (threadIdx.x == 0) rstd[row] = r;
  if (c >= H) return;
  float v[8], wv[8];
  unpack8(load8(xn + row * H + c), v);
  ldw8(w, w32, c, wv);
#pragma unroll
  for (int j = 0; j < 8; ++j) v[j] = mul(mul(v[j], r), wv[j]);
  store8(y + row * H + c, pack8(v));
}

// as written: prod = (dy * w) * xn, whose row sums are the gradient of r; part[blk][H]: column sums of dy (xn r) (null: none)
__global__ void __launch_bounds__(1024) rms_prod_kernel(const uint16_t* __restrict__ dy, const uint16_t* __restrict__ xn,
                                                        const void* __restrict__ w, int w32, const float* __restrict__ rstd,
                                                        int64_t R, int H, float* __restrict__ prod, float* __restrict__ part) {
  const int c = threadIdx.x * 8;
  if (c >= H) return;
  float wv[8], dw[8] = {0, 0, 0, 0, 0, 0, 0, 0};
  ldw8(w, w32, c, wv);
  for (int64_t row = blockIdx.x; row < R; row += gridDim.x) {
    const float r = rstd[row];
    float g[8], v[8];
    unpack8(load8(dy + row * H + c), g);
    unpack8(load8(xn + row * H + c), v);
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      dw[j] += g[j] * (v[j] * r);
      v[j] = mul(mul(g[j], wv[j]), v[j]);
    }
    store8f(prod + row * H + c, v);
  }
  if (part) store8f(part + (int64_t)blockIdx.x * H + c, dw);
}

// as written: dx = bf16((dy w) r + (dms * inv_h) (2 xn)) [+ dxn], dms = (-0.5 dr) r^3
__global__ void __launch_bounds__(1024) rms_dx_kernel(const uint16_t* __restrict__ dy, const uint16_t* __restrict__ xn,
                                                      const void* __restrict__ w, int w32, const float* __restrict__ rstd,
                                                      const float* __restrict__ dr, const uint16_t* __restrict__ dxn, int H,
                                                      float inv_h, uint16_t* __restrict__ dx) {
  const int64_t row = blockIdx.x;
  const int c = threadIdx.x * 8;
  if (c >= H) return;
  const float r = rstd[row];
  const float dms = mul(mul(mul(-0.5f, dr[row]), mul(mul(r, r), r)), inv_h);
  float g[8], v[8], wv[8];
  unpack8(load8(dy + row * H + c), g);
  unpack8(load8(xn + row * H + c), v);
  ldw8(w, w32, c, wv);
#pragma unroll
  for (int j = 0; j < 8; ++j)
    v[j] = add(mul(mul(g[j], wv[j]), r), mul(dms, mul(2.f, v[j])));
  u16x8 o = pack8(v);
  if (dxn) {
    unpack8(o, v);
    unpack8(load8(dxn + row * H + c), g);
#pragma unroll
    for (int j = 0; j < 8; ++j) v[j] += g[j];
    o = pack8(v);
  }
  store8(dx + row * H + c, o);
}

// the same gradient in one pass, its sums in this kernel's order (adapters, whose base has no gradient):
// dx = dxn + rstd (dy w - n mean(dy w n)), n = xn rstd; part[blk][H]: column sums of dy n (null: no gradient of w)
__global__ void __launch_bounds__(1024) rms_bwd_kernel(const uint16_t* __restrict__ xn, const float* __restrict__ rstd,
                                                       const void* __restrict__ w, int w32, const uint16_t* __restrict__ dy,
                                                       const uint16_t* __restrict__ dxn, int64_t R, int H,
                                                       uint16_t* __restrict__ dx, float* __restrict__ part) {
  __shared__ float red[16];
  const int c = threadIdx.x * 8;
  const bool active = c < H;
  float wv[8] = {0, 0, 0, 0, 0, 0, 0, 0}, dw[8] = {0, 0, 0, 0, 0, 0, 0, 0};
  if (active) ldw8(w, w32, c, wv);
  for (int64_t row = blockIdx.x; row < R; row += gridDim.x) {
    const float r = rstd[row];
    float n[8], g[8], s = 0.f;
    if (active) {
      unpack8(load8(xn + row * H + c), n);
      unpack8(load8(dy + row * H + c), g);
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        n[j] *= r;
        dw[j] += g[j] * n[j];
        g[j] *= wv[j];
        s += g[j] * n[j];
      }
    }
    s = block_sum(s, red) / (float)H;
    if (active) {
      float a[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) a[j] = r * (g[j] - n[j] * s);
      if (dxn) {
        float d[8];
        unpack8(load8(dxn + row * H + c), d);
#pragma unroll
        for (int j = 0; j < 8; ++j) a[j] += d[j];
      }
      store8(dx + row * H + c, pack8(a));
    }
  }
  if (part && active) store8f(part + (int64_t)blockIdx.x * H + c, dw);
}

// ---------------------------------------------------------------- layer norm behind a residual
// as written: s = x + o in fp32
__global__ void __launch_bounds__(256) add_f32_kernel(const uint16_t* __restrict__ x, const uint16_t* __restrict__ o, int64_t n8,
                                                      float* __restrict__ s) {
  for (int64_t i = blockIdx.x * 256ll + threadIdx.x; i < n8; i += gridDim.x * 256ll) {
    float a[8], b[8];
    unpack8(load8(x + 8 * i), a);
    unpack8(load8(o + 8 * i), b);
#pragma unroll
    for (int j = 0; j < 8; ++j) a[j] += b[j];
    store8f(s + 8 * i, a);
  }
}

// part[blk][2][H]: column sums of dy n and dy, n = (s - mean) rstd
__global__ void __launch_bounds__(1024) ln_sums_kernel(const float* __restrict__ s, const float* __restrict__ mean,
                                                       const float* __restrict__ rstd, const uint16_t* __restrict__ dy, int64_t R,
                                                       int H, float* __restrict__ part) {
  const int c = threadIdx.x * 8;
  if (c >= H) return;
  float sg[8] = {0, 0, 0, 0, 0, 0, 0, 0}, sb[8] = {0, 0, 0, 0, 0, 0, 0, 0};
  for (int64_t row = blockIdx.x; row < R; row += gridDim.x) {
    const float m = mean[row], r = rstd[row];
    float d[8], v[8];
    unpack8(load8(dy + row * H + c), d);
    ldw8(s, true, row * H + c, v);
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      sg[j] += d[j] * ((v[j] - m) * r);
      sb[j] += d[j];
    }
  }
  float* p = part + (int64_t)blockIdx.x * 2 * H + c;
  store8f(p, sg);
  store8f(p + H, sb);
}

// out[n] = sum over P rows of part [P, n]. The chain of loads bounds it: 64 columns a workgroup, 16 rows at a time and four of
// those in flight (512 x 4,096: four rows at a time, one in flight, 39 us, now 6)
template <typename OUT>
__global__ void __launch_bounds__(1024) sum_parts_kernel(const float* __restrict__ part, int P, int64_t n, OUT* __restrict__ out) {
  __shared__ float red[1024];
  const int64_t c = (int64_t)blockIdx.x * 64 + (threadIdx.x & 63);
  float s = 0.f;
  if (c < n) {
    int r = threadIdx.x >> 6;
    for (; r + 48 < P; r += 64) {
      const float a = part[r * n + c], b = part[(r + 16) * n + c], d = part[(r + 32) * n + c], e = part[(r + 48) * n + c];
      s += (a + b) + (d + e);
    }
    for (; r < P; r += 16) s += part[r * n + c];
  }
  red[threadIdx.x] = s;
  __syncthreads();
  for (int o = 512; o >= 64; o >>= 1) {
    if (threadIdx.x < o) red[threadIdx.x] += red[threadIdx.x + o];
    __syncthreads();
  }
  if (threadIdx.x < 64 && c < n) {
    if constexpr (sizeof(OUT) == 2) out[c] = f2bf(red[threadIdx.x]);
    else out[c] = red[threadIdx.x];
  }
}

// ---------------------------------------------------------------- activations
// as written: GELU (erf form) of bf16 values in fp32; dh: its gradient
__global__ void __launch_bounds__(256) gelu_kernel(const uint16_t* __restrict__ z, const uint16_t* __restrict__ dh, int64_t n8,
                                                   uint16_t* __restrict__ out) {
  for (int64_t i = blockIdx.x * 256ll + threadIdx.x; i < n8; i += gridDim.x * 256ll) {
    float v[8];
    unpack8(load8(z + 8 * i), v);
    if (dh) {
      float d[8];
      unpack8(load8(dh + 8 * i), d);
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const float cdf = 0.5f * (1.f + erff(v[j] * 0.70710678118654752440f));
        const float pdf = expf(-0.5f * v[j] * v[j]) * 0.39894228040143267794f;
        v[j] = d[j] * (cdf + v[j] * pdf);
      }
    } else {
#pragma unroll
      for (int j = 0; j < 8; ++j) v[j] = v[j] * 0.5f * (1.f + erff(v[j] * 0.70710678118654752440f));
    }
    store8(out + 8 * i, pack8(v));
  }
}

// part[blk][F]: column sums of bf16 rows
__global__ void __launch_bounds__(256) col_sums_kernel(const uint16_t* __restrict__ x, int64_t ld, int64_t R, int F,
                                                       float* __restrict__ part) {
  const int c = (blockIdx.x * 256 + threadIdx.x) * 8;
  if (c >= F) return;
  float s[8] = {0, 0, 0, 0, 0, 0, 0, 0};
  for (int64_t row = blockIdx.y; row < R; row += gridDim.y) {
    float d[8];
    unpack8(load8(x + row * ld + c), d);
#pragma unroll
    for (int j = 0; j < 8; ++j) s[j] += d[j];
  }
  store8f(part + (int64_t)blockIdx.y * F + c, s);
}

namespace {
__device__ __forceinline__ int cast_tensor(const CastTable& t, int& chunk) {
  int i = 0;
  while (i + 1 < t.n && chunk >= t.first[i + 1]) ++i;
  chunk -= t.first[i];
  return i;
}
}  // namespace

// Matrices and biases of a layer to bf16, and their gradients back, of two uses added: one launch for the dozens of tensors whose
// casts, casts back and additions took a launch each, 4.5 us for a bias of 2 to 8 KB. Memory bounds it
// (a layer of 12.6M weights: 75 MB in 17.8 us, back 100 MB in 25.8; BERT-large, both passes: 62.0 -> 59.4 ms of kernels a step).
__global__ void __launch_bounds__(256) half_copies_kernel(CastTable t) {
  int chunk = blockIdx.x;
  const int i = cast_tensor(t, chunk);
  const int64_t beg = (int64_t)chunk * CAST_CHUNK, end = min(t.len[i], beg + CAST_CHUNK);
  const float* f = t.f[i];
  uint16_t* a = t.a[i];
#pragma unroll 4
  for (int64_t c = beg + 8 * threadIdx.x; c < end; c += 2048) {
    if (c + 7 < end) {
      const f32x4 u = *reinterpret_cast<const f32x4*>(f + c), v = *reinterpret_cast<const f32x4*>(f + c + 4);
      u16x8 o;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        o[j] = f2bf(u[j]);
        o[4 + j] = f2bf(v[j]);
      }
      store8(a + c, o);
    } else {
      for (int64_t k = c; k < end; ++k) a[k] = f2bf(f[k]);
    }
  }
}

__global__ void __launch_bounds__(256) half_grads_kernel(CastTable t) {
  int chunk = blockIdx.x;
  const int i = cast_tensor(t, chunk);
  const int64_t beg = (int64_t)chunk * CAST_CHUNK, end = min(t.len[i], beg + CAST_CHUNK);
  float* f = t.f[i];
  const uint16_t *a = t.a[i], *b = t.b[i];
#pragma unroll 4
  for (int64_t c = beg + 8 * threadIdx.x; c < end; c += 2048) {
    if (c + 7 < end) {
      float u[8];
      unpack8(load8(a + c), u);
      if (b) {
        float v[8];
        unpack8(load8(b + c), v);
#pragma unroll
        for (int j = 0; j < 8; ++j) u[j] += v[j];
      }
      store8f(f + c, u);
    } else {
      for (int64_t k = c; k < end; ++k) f[k] = b ? bf2f(a[k]) + bf2f(b[k]) : bf2f(a[k]);
    }
  }
}

// as written: h = bf16(silu(gate)) up of gu [R, 2F] = [gate | up]; BWD: dgu from dh
template <bool BWD>
__global__ void __launch_bounds__(256) swiglu_kernel(const uint16_t* __restrict__ gu, const uint16_t* __restrict__ dh, int64_t R, int F,
                                                     uint16_t* __restrict__ out) {
  const int64_t nv = F / 8, total = R * nv;
  for (int64_t i = blockIdx.x * 256ll + threadIdx.x; i < total; i += gridDim.x * 256ll) {
    const int64_t row = i / nv, c = (i - row * nv) * 8;
    float g[8], u[8];
    unpack8(load8(gu + row * 2 * F + c), g);
    unpack8(load8(gu + row * 2 * F + F + c), u);
    if constexpr (!BWD) {
#pragma unroll
      for (int j = 0; j < 8; ++j) g[j] = bf2f(f2bf(g[j] / (1.f + expf(-g[j])))) * u[j];
      store8(out + row * F + c, pack8(g));
    } else {
      float t[8];
      unpack8(load8(dh + row * F + c), t);
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const float x = g[j], a = bf2f(f2bf(x / (1.f + expf(-x))));
        const float s = 1.f / (1.f + expf(-x)), da = bf2f(f2bf(t[j] * u[j]));
        g[j] = da * s * (1.f + x * (1.f - s));
        u[j] = t[j] * a;
      }
      store8(out + row * 2 * F + c, pack8(g));
      store8(out + row * 2 * F + F + c, pack8(u));
    }
  }
}

// as written: y = bf16(y + bf16(scale d))
__global__ void __launch_bounds__(256) add_scaled_kernel(const uint16_t* __restrict__ d, float scale, int64_t n8, uint16_t* __restrict__ y) {
  for (int64_t i = blockIdx.x * 256ll + threadIdx.x; i < n8; i += gridDim.x * 256ll) {
    float a[8], b[8];
    unpack8(load8(y + 8 * i), a);
    unpack8(load8(d + 8 * i), b);
#pragma unroll
    for (int j = 0; j < 8; ++j) a[j] += bf2f(f2bf(b[j] * scale));
    store8(y + 8 * i, pack8(a));
  }
}

// ---------------------------------------------------------------- rotation
// out = rows [q heads | k heads | v heads] with the first nr = Hq + Hkv heads rotated (halves) by cs [P, D] = [cos | sin] of
// row t % P (sign -1: back), the others copied; as written: products, then their sum. 8 pairs a thread
__global__ void __launch_bounds__(256) rope_rows_kernel(const uint16_t* __restrict__ in, const float* __restrict__ cs, int64_t T,
                                                        int64_t P, int nr, int nh, int D, float sign, uint16_t* __restrict__ out) {
  const int per = D / 16;
  const int64_t total = T * nh * per;
  for (int64_t i = blockIdx.x * 256ll + threadIdx.x; i < total; i += gridDim.x * 256ll) {
    const int64_t t = i / (nh * per);
    const int r = (int)(i - t * nh * per), hd = r / per, c = (r % per) * 8;
    const int64_t at = (t * nh + hd) * D + c;
    const u16x8 a = load8(in + at), b = load8(in + at + D / 2);
    if (hd >= nr) {
      if (in != out) {
        store8(out + at, a);
        store8(out + at + D / 2, b);
      }
      continue;
    }
    const float* p = cs + (t % P) * D + c;
    float x[8], y[8], co[8], si[8];
    unpack8(a, x);
    unpack8(b, y);
    ldw8(p, true, 0, co);
    ldw8(p, true, D / 2, si);
    float u[8], v[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const float s = sign * si[j];
      u[j] = add(mul(x[j], co[j]), -mul(y[j], s));
      v[j] = add(mul(y[j], co[j]), mul(x[j], s));
    }
    store8(out + at, pack8(u));
    store8(out + at + D / 2, pack8(v));
  }
}

// ---------------------------------------------------------------- cross entropy
// lse[r] = log sum exp of a row of bf16 logits, loss[r] = lse - logit[y] (a label outside the row: NaN). One workgroup a row,
// one pass: running maximum and sum per thread
__global__ void __launch_bounds__(512) ce_fwd_kernel(const uint16_t* __restrict__ lg, const int64_t* __restrict__ y, int64_t V,
                                                     float* __restrict__ lse, float* __restrict__ loss) {
  __shared__ float red[32];
  const int64_t row = blockIdx.x;
  const uint16_t* p = lg + row * V;
  float m = -INFINITY, s = 0.f;
  for (int64_t c = threadIdx.x * 8ll; c < V; c += 512 * 8) {
    float v[8], mx;
    unpack8(load8(p + c), v);
    mx = v[0];
#pragma unroll
    for (int j = 1; j < 8; ++j) mx = fmaxf(mx, v[j]);
    if (mx > m) {
      s *= __expf(m - mx);
      m = mx;
    }
    if (m > -INFINITY) {
#pragma unroll
      for (int j = 0; j < 8; ++j) s += __expf(v[j] - m);
    } else {   // -inf throughout, or NaN, which the maximum leaves out
#pragma unroll
      for (int j = 0; j < 8; ++j) s += v[j] == v[j] ? 0.f : v[j];
    }
  }
  const float M = block_max(m, red);
  if (m > -INFINITY) s *= __expf(m - M);
  s = block_sum(s, red);
  if (threadIdx.x == 0) {
    const float l = M + logf(s);
    const int64_t t = y[row];
    lse[row] = l;
    loss[row] = t >= 0 && t < V ? l - bf2f(p[t]) : NAN;
  }
}

// d = (softmax - one-hot) * scale[0]; LP: as written, from fp32 log softmax rows x (lse null). 2,048 x 50,304 logits, both
// directions: 120 us, with the log softmax 490, from torch's operations 874
template <bool LP>
__global__ void __launch_bounds__(512) ce_bwd_kernel(const void* __restrict__ x, const int64_t* __restrict__ y,
                                                     const float* __restrict__ lse, const float* __restrict__ scale, int64_t V,
                                                     uint16_t* __restrict__ d) {
  const int64_t row = blockIdx.x, t = y[row];
  const float l = LP ? 0.f : lse[row], sc = scale[0];
  for (int64_t c = threadIdx.x * 8ll; c < V; c += 512 * 8) {
    float v[8];
    ldw8(x, LP, row * V + c, v);
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      if (LP) v[j] = expf(v[j]) * sc + (c + j == t ? -sc : 0.f);
      else v[j] = (__expf(v[j] - l) - (c + j == t ? 1.f : 0.f)) * sc;
    }
    store8(d + row * V + c, pack8(v));
  }
}

// ---------------------------------------------------------------- launches
static int tr_threads(int H) { return (H / 8 + 63) / 64 * 64; }

// workgroups of the kernels that leave column sums: enough to fill the chip, few enough that the sums stay small
int train_parts(int64_t R) { return (int)(R < 512 ? R : 512); }
int train_col_parts(int64_t R, int F) {
  const int64_t gx = (F + 2047) / 2048, want = 512 / gx;
  return (int)(R < want ? R : want);
}

static unsigned tr_grid(int64_t n) {
  const int64_t g = (n + 255) / 256;
  return (unsigned)(g < 8192 ? g : 8192);
}

void launch_rms_sq(const uint16_t* x, const uint16_t* o, int64_t n, uint16_t* xn, float* sq, hipStream_t st) {
  if (n) rms_sq_kernel<<<tr_grid(n / 8), 256, 0, st>>>(x, o, n / 8, xn, sq);
}

void launch_rms_apply(const uint16_t* xn, const float* ms, const void* w, bool w32, float eps, int64_t R, int H, uint16_t* y,
                      float* rstd, hipStream_t st) {
  if (R) rms_apply_kernel<<<(unsigned)R, tr_threads(H), 0, st>>>(xn, ms, w, w32, eps, H, y, rstd);
}

void launch_rms_prod(const uint16_t* dy, const uint16_t* xn, const void* w, bool w32, const float* rstd, int64_t R, int H,
                     float* prod, float* part, float* dw, hipStream_t st) {
  if (!R) return;
  const int P = train_parts(R);
  rms_prod_kernel<<<part ? P : (unsigned)(R < 65536 ? R : 65536), tr_threads(H), 0, st>>>(dy, xn, w, w32, rstd, R, H, prod, part);
  if (part) sum_parts_kernel<<<(H + 63) / 64, 1024, 0, st>>>(part, P, H, dw);
}

void launch_rms_dx(const uint16_t* dy, const uint16_t* xn, const void* w, bool w32, const float* rstd, const float* dr,
                   const uint16_t* dxn, int64_t R, int H, uint16_t* dx, hipStream_t st) {
  if (R) rms_dx_kernel<<<(unsigned)R, tr_threads(H), 0, st>>>(dy, xn, w, w32, rstd, dr, dxn, H, 1.f / (float)H, dx);
}

void launch_rms_bwd(const uint16_t* xn, const float* rstd, const void* w, bool w32, const uint16_t* dy, const uint16_t* dxn,
                    int64_t R, int H, uint16_t* dx, float* part, float* dw, hipStream_t st) {
  if (!R) return;
  const int P = train_parts(R);
  const unsigned grid = part ? P : (unsigned)(R < 65536 ? R : 65536);
  rms_bwd_kernel<<<grid, tr_threads(H), 0, st>>>(xn, rstd, w, w32, dy, dxn, R, H, dx, part);
  if (part) sum_parts_kernel<<<(H + 63) / 64, 1024, 0, st>>>(part, P, H, dw);
}

void launch_add_f32(const uint16_t* x, const uint16_t* o, int64_t n, float* s, hipStream_t st) {
  if (n) add_f32_kernel<<<tr_grid(n / 8), 256, 0, st>>>(x, o, n / 8, s);
}

void launch_ln_sums(const float* s, const float* mean, const float* rstd, const uint16_t* dy, int64_t R, int H, float* part,
                    float* sums, hipStream_t st) {
  if (!R) return;
  const int P = train_parts(R);
  ln_sums_kernel<<<P, tr_threads(H), 0, st>>>(s, mean, rstd, dy, R, H, part);
  sum_parts_kernel<<<(2 * H + 63) / 64, 1024, 0, st>>>(part, P, 2 * (int64_t)H, sums);
}

void launch_gelu(const uint16_t* z, const uint16_t* dh, int64_t n, uint16_t* out, hipStream_t st) {
  if (n) gelu_kernel<<<tr_grid(n / 8), 256, 0, st>>>(z, dh, n / 8, out);
}

void launch_col_sums(const uint16_t* x, int64_t ld, int64_t R, int F, float* part, uint16_t* out, hipStream_t st) {
  if (!R) return;
  const int P = train_col_parts(R, F);
  col_sums_kernel<<<dim3((F + 2047) / 2048, P), 256, 0, st>>>(x, ld, R, F, part);
  sum_parts_kernel<<<(F + 63) / 64, 1024, 0, st>>>(part, P, F, out);
}

void launch_half_copies(const CastTable& t, hipStream_t st) { half_copies_kernel<<<t.first[t.n], 256, 0, st>>>(t); }
void launch_half_grads(const CastTable& t, hipStream_t st) { half_grads_kernel<<<t.first[t.n], 256, 0, st>>>(t); }

void launch_swiglu(const uint16_t* gu, const uint16_t* dh, int64_t R, int F, uint16_t* out, hipStream_t st) {
  if (R * F == 0) return;
  if (dh) swiglu_kernel<true><<<tr_grid(R * (F / 8)), 256, 0, st>>>(gu, dh, R, F, out);
  else swiglu_kernel<false><<<tr_grid(R * (F / 8)), 256, 0, st>>>(gu, nullptr, R, F, out);
}

void launch_add_scaled(const uint16_t* d, float scale, int64_t n, uint16_t* y, hipStream_t st) {
  if (n) add_scaled_kernel<<<tr_grid(n / 8), 256, 0, st>>>(d, scale, n / 8, y);
}

void launch_rope_rows(const uint16_t* in, const float* cs, int64_t T, int64_t P, int nr, int nh, int D, float sign, uint16_t* out,
                      hipStream_t st) {
  const int64_t n = (T * nh * (D / 16) + 255) / 256;
  if (!n) return;
  rope_rows_kernel<<<(unsigned)(n < 16384 ? n : 16384), 256, 0, st>>>(in, cs, T, P, nr, nh, D, sign, out);
}

void launch_ce_fwd(const uint16_t* lg, const int64_t* y, int64_t R, int64_t V, float* lse, float* loss, hipStream_t st) {
  if (R) ce_fwd_kernel<<<(unsigned)R, 512, 0, st>>>(lg, y, V, lse, loss);
}

void launch_ce_bwd(const void* x, const int64_t* y, const float* lse, const float* scale, int64_t R, int64_t V, uint16_t* d,
                   hipStream_t st) {
  if (!R) return;
  if (lse) ce_bwd_kernel<false><<<(unsigned)R, 512, 0, st>>>(x, y, lse, scale, V, d);
  else ce_bwd_kernel<true><<<(unsigned)R, 512, 0, st>>>(x, y, lse, scale, V, d);
}

}  // namespace nga
