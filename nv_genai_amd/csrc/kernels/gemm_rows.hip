// Projections of few rows (an encoder on one query): out[M, N] = x[M, K] . W[N, K]^T + bias for up to 32 rows, with the
// bias, GELU or a K split for the norm that follows; that norm; and the embedding sum with its norm.
//
// With tens of rows a projection is its weight stream, 2 to 8 MB of a BERT-large layer: about a microsecond of HBM time,
// so latency decides. Every wave loads the MFMA fragments of its whole share of K straight into registers, all in flight
// at once (W rows are the A operand, token rows the B operand, 16 bytes a lane each), multiplies, and the eight waves of a
// workgroup, which share 16 features and split K, meet once in LDS. No staging, no loop of barriers. BERT-large at 19
// rows, weights from HBM (us, library / here): q/k/v 11.1 / 5.1, output 5.8 / 3.0, up 11.3 / 5.4 and its GELU launch
// saved, down 14.1 / 4.9. Token rows come from L2 again for each workgroup: from 33 rows on the LDS tiles of
// gemm_skinny.hip are faster (64 rows: q/k/v 8.2 here, 7.6 there).
#include "common.h"
#include "kernels.h"

namespace nga {

namespace {
// 0.5 x (1 + erf(x / sqrt 2))
__device__ __forceinline__ float gr_gelu(float x) { return 0.5f * x * (1.f + erff(x * 0.70710678118654752f)); }
}  // namespace

// MT x 16 token rows and 16 features per workgroup; PD k-steps of 32 in flight per wave, twice.
// EPI 0: bf16 out, + bias; 1: fp32 slab [split, M, N]; 2: bf16 out, GELU(. + bias)
template <int MT, int EPI>
__global__ void __launch_bounds__(512) row_gemm_kernel(RowGemmParams P) {
  constexpr int PD = 4, NW = 8;
  __shared__ __attribute__((aligned(16))) float part[NW * MT * 256];
  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int col = lane & 15, h = lane >> 4;
  const int f0 = blockIdx.x * 16, t0 = blockIdx.y * 16 * MT, ks = blockIdx.z;
  const int steps = P.K / 32, slices = NW * P.split, sl = ks * NW + w;
  const int s0 = steps * sl / slices, s1 = steps * (sl + 1) / slices;
  const uint16_t *wp = P.w + (int64_t)(f0 + col) * P.K + 8 * h, *xp[MT];
#pragma unroll
  for (int i = 0; i < MT; ++i) xp[i] = P.x + (int64_t)min(t0 + 16 * i + col, P.M - 1) * P.ldx + 8 * h;
  f32x4 acc[MT];
#pragma unroll
  for (int j = 0; j < MT; ++j) acc[j] = (f32x4)(0.f);
  u16x8 a[PD], b[PD][MT], an[PD], bn[PD][MT];
  auto load = [&](int s, u16x8 (&av)[PD], u16x8 (&bv)[PD][MT]) {
#pragma unroll
    for (int d = 0; d < PD; ++d)
      if (s + d < s1) {
        av[d] = load8(wp + 32 * (s + d));
#pragma unroll
        for (int i = 0; i < MT; ++i) bv[d][i] = load8(xp[i] + 32 * (s + d));
      }
  };
  load(s0, a, b);
  for (int s = s0; s < s1; s += PD) {
    if (s + PD < s1) load(s + PD, an, bn);
#pragma unroll
    for (int d = 0; d < PD; ++d)
      if (s + d < s1) {
#pragma unroll
        for (int j = 0; j < MT; ++j) acc[j] = mfma16(as_bf16x8(a[d]), as_bf16x8(b[d][j]), acc[j]);
      }
    if (s + PD < s1) {
#pragma unroll
      for (int d = 0; d < PD; ++d) {
        a[d] = an[d];
#pragma unroll
        for (int i = 0; i < MT; ++i) b[d][i] = bn[d][i];
      }
    }
  }
#pragma unroll
  for (int j = 0; j < MT; ++j) *reinterpret_cast<f32x4*>(&part[((w * MT + j) * 64 + lane) * 4]) = acc[j];
  __syncthreads();
  // tile j: features f0 + 4 h + 0..3 of token t0 + 16 j + col; one wave each
#pragma unroll
  for (int j = 0; j < MT; ++j) {
    if (j != w) continue;
    f32x4 v = (f32x4)(0.f);
#pragma unroll
    for (int u = 0; u < NW; ++u) v += *reinterpret_cast<const f32x4*>(&part[((u * MT + j) * 64 + lane) * 4]);
    const int t = t0 + 16 * j + col, n = f0 + 4 * h;
    if (t >= P.M) continue;
    if constexpr (EPI == 1) {
      *reinterpret_cast<f32x4*>(reinterpret_cast<float*>(P.out) + ((int64_t)ks * P.M + t) * P.N + n) = v;
    } else {
      u16x4 o;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const float y = v[r] + bf2f(P.bias[n + r]);
        o[r] = f2bf(EPI == 2 ? gr_gelu(y) : y);
      }
      *reinterpret_cast<u16x4*>(reinterpret_cast<uint16_t*>(P.out) + (int64_t)t * P.ldo + n) = o;
    }
  }
}

// out = LN(sum_s P[s] + bias + resid): the norm behind a K-split projection (P [S, M, H] fp32)
__global__ void __launch_bounds__(1024) splitk_layernorm_kernel(const float* __restrict__ P, int S, int M,
                                                                const uint16_t* __restrict__ bias,
                                                                const uint16_t* __restrict__ resid,
                                                                const uint16_t* __restrict__ g, const uint16_t* __restrict__ b,
                                                                float eps, int H, uint16_t* __restrict__ out) {
  __shared__ float red[16];
  const int64_t row = blockIdx.x;
  const int c = threadIdx.x * 8;
  const bool active = c < H;
  const int64_t slab = (int64_t)M * H;
  float x[8], s = 0.f;
  u16x8 gv, bv;
  if (active) {
    const float* p = P + row * H + c;
    f32x4 a0 = *reinterpret_cast<const f32x4*>(p), a1 = *reinterpret_cast<const f32x4*>(p + 4);
    for (int k = 1; k < S; ++k) {
      a0 += *reinterpret_cast<const f32x4*>(p + k * slab);
      a1 += *reinterpret_cast<const f32x4*>(p + k * slab + 4);
    }
    const u16x8 r = load8(resid + row * H + c), bi = load8(bias + c);
    gv = load8(g + c);
    bv = load8(b + c);
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      x[i] = (i < 4 ? a0[i] : a1[i - 4]) + bf2f(bi[i]) + bf2f(r[i]);
      s += x[i];
    }
  }
  const float mean = block_sum(s, red) / (float)H;
  float vs = 0.f;
  if (active) {
#pragma unroll
    for (int i = 0; i < 8; ++i) vs += (x[i] - mean) * (x[i] - mean);
  }
  const float rstd = rsqrtf(block_sum(vs, red) / (float)H + eps);
  if (active) {
    u16x8 o;
#pragma unroll
    for (int i = 0; i < 8; ++i) o[i] = f2bf((x[i] - mean) * rstd * bf2f(gv[i]) + bf2f(bv[i]));
    store8(out + row * H + c, o);
  }
}

// x[t] = LN(word[ids[t]] + pos_table[pos[t]] + type[types[t]]), the sum in fp32 (types null: row 0). An index outside its
// table gives a row of NaN. Six gather, addition and norm launches before.
__global__ void __launch_bounds__(1024) embed_layernorm_kernel(const int32_t* __restrict__ ids, const int32_t* __restrict__ pos,
                                                               const int32_t* __restrict__ types,
                                                               const uint16_t* __restrict__ word, int n_word,
                                                               const uint16_t* __restrict__ ptab, int n_pos,
                                                               const uint16_t* __restrict__ ttab, int n_type,
                                                               const uint16_t* __restrict__ g, const uint16_t* __restrict__ b,
                                                               float eps, int H, uint16_t* __restrict__ out) {
  __shared__ float red[16];
  const int64_t row = blockIdx.x;
  const int c = threadIdx.x * 8;
  const bool active = c < H;
  float x[8], s = 0.f;
  if (active) {
    const int a0 = ids[row], a1 = pos[row], a2 = types ? types[row] : 0;
    const bool ok = a0 >= 0 && a0 < n_word && a1 >= 0 && a1 < n_pos && a2 >= 0 && a2 < n_type;
    const int64_t i0 = ok ? a0 : 0, i1 = ok ? a1 : 0, i2 = ok ? a2 : 0;
    const u16x8 v0 = load8(word + i0 * H + c), v1 = load8(ptab + i1 * H + c), v2 = load8(ttab + i2 * H + c);
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      x[i] = ok ? bf2f(v0[i]) + bf2f(v1[i]) + bf2f(v2[i]) : NAN;
      s += x[i];
    }
  }
  const float mean = block_sum(s, red) / (float)H;
  float vs = 0.f;
  if (active) {
#pragma unroll
    for (int i = 0; i < 8; ++i) vs += (x[i] - mean) * (x[i] - mean);
  }
  const float rstd = rsqrtf(block_sum(vs, red) / (float)H + eps);
  if (active) {
    const u16x8 gv = load8(g + c), bv = load8(b + c);
    u16x8 o;
#pragma unroll
    for (int i = 0; i < 8; ++i) o[i] = f2bf((x[i] - mean) * rstd * bf2f(gv[i]) + bf2f(bv[i]));
    store8(out + row * H + c, o);
  }
}

void launch_row_gemm(const RowGemmParams& p, int epi, hipStream_t stream) {
  if (p.M == 0 || p.N == 0) return;
  const int mt = p.M <= 16 ? 1 : 2;
  const dim3 grid(p.N / 16, (p.M + 16 * mt - 1) / (16 * mt), p.split);
#define NGA_RG(MT_)                                                               \
  if (mt == MT_) {                                                                \
    if (epi == 0) row_gemm_kernel<MT_, 0><<<grid, 512, 0, stream>>>(p);           \
    else if (epi == 1) row_gemm_kernel<MT_, 1><<<grid, 512, 0, stream>>>(p);      \
    else row_gemm_kernel<MT_, 2><<<grid, 512, 0, stream>>>(p);                    \
    return;                                                                       \
  }
  NGA_RG(1) NGA_RG(2)
#undef NGA_RG
}

static int rows_threads(int H) { return (H / 8 + 63) / 64 * 64; }

void launch_splitk_layernorm(const float* P, int S, int M, const uint16_t* bias, const uint16_t* resid, const uint16_t* g,
                             const uint16_t* b, float eps, int H, uint16_t* out, hipStream_t stream) {
  if (M == 0) return;
  splitk_layernorm_kernel<<<M, rows_threads(H), 0, stream>>>(P, S, M, bias, resid, g, b, eps, H, out);
}

void launch_embed_layernorm(const int32_t* ids, const int32_t* pos, const int32_t* types, const uint16_t* word, int n_word,
                            const uint16_t* ptab, int n_pos, const uint16_t* ttab, int n_type, const uint16_t* g,
                            const uint16_t* b, float eps, int64_t rows, int H, uint16_t* out, hipStream_t stream) {
  if (rows == 0) return;
  embed_layernorm_kernel<<<(unsigned)rows, rows_threads(H), 0, stream>>>(ids, pos, types, word, n_word, ptab, n_pos, ttab, n_type,
                                                                         g, b, eps, H, out);
}

}  // namespace nga
