// Projections of few rows (an encoder on one query): out[M, N] = x[M, K] . W[N, K]^T + bias for up to 32 rows, with the
// bias, GELU or a K split for the norm that follows; that norm; and the embedding sum with its norm.
//
// With tens of rows a projection is its weight stream, 2 to 8 MB of a BERT-large layer: about a microsecond of HBM time,
// so latency decides, and the cycles of a CU's load path: every workgroup reads all token rows beside its 16 rows of weights. Every wave
// loads its whole share of K straight into registers, all in flight at once, multiplies (W rows are the A operand, token rows the B
// operand), and the eight waves of a workgroup, which share 16 features and split K, meet once in LDS. No staging, no loop of barriers.
// What bounds it is how the lanes of a load lie: as an MFMA operand wants them, 16 rows to neighbouring lanes, a load takes a cycle a
// lane (37 bytes a nanosecond and CU from L2); with four lanes to 64 bytes of a row 107. So weights come in that order and change
// lanes (gr_fragment), and token rows lie packed, a step of 16 rows in one piece, written so by what makes them. BERT-large at 19 rows,
// weights from HBM, us, library / as fragments / so: q/k/v 11.1 / 5.1 / 3.7, output behind its attention - / 5.3 / 4.5, up 11.3 / 5.9 /
// 3.9 and its GELU launch saved, down 14.1 / 5.3 / 3.9. Token rows come from L2 again for each workgroup, up
// to two tiles of 16. A layer of an encoder at 16 / 20 / 32 rows, us, here / in the LDS tiles of gemm_skinny.hip: hidden size 384 22.1 23.2 23.7 / 26.7 27.3
// 27.4, 768 23.5 24.9 25.2 / 29.6 30.1 30.4, 1,024 26.9 28.2 28.7 / 34.6 34.8 35.4 (at 36 rows 25.5, 31.0, 36.8 there). Three tiles and more were slower than LDS
// tiles while every load came as fragments (64 rows: q/k/v 8.2, 7.6 there), and have not been tried with these loads.
#include "common.h"
#include "gelu.h"
#include "kernels.h"

namespace nga {

namespace {
typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) s16x4* ltr_t;

// 16 rows x 32 values as an instruction brings them fastest, four lanes for 64 bytes of a row (lane 4 r + c: row r, values 8 c ..),
// as the MFMA operand: lane r + 16 c
__device__ __forceinline__ bf16x8 gr_fragment(u16x8 v, int lane) {
  typedef int i32x4 __attribute__((ext_vector_type(4)));
  const int from = ((lane & 15) * 4 + (lane >> 4)) * 4;
  i32x4 a = __builtin_bit_cast(i32x4, v);
#pragma unroll
  for (int i = 0; i < 4; ++i) a[i] = __builtin_amdgcn_ds_bpermute(from, a[i]);
  return __builtin_bit_cast(bf16x8, a);
}

}  // namespace

// MT x 16 token rows and 16 features per workgroup; PD k-steps of 32 in flight per wave, twice.
// EPI 0: bf16 out, + bias; 1: fp32 slab [split, M, N]; 2: bf16 out, GELU(. + bias)
template <int MT, int EPI, bool XP>
__global__ void __launch_bounds__(512) row_gemm_kernel(RowGemmParams P) {
  constexpr int PD = 4, NW = 8;
  __shared__ __attribute__((aligned(16))) float part[NW * MT * 256];
  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int col = lane & 15, h = lane >> 4;
  const int f0 = blockIdx.x * 16, ks = blockIdx.y;
  const int steps = P.K / 32, slices = NW * P.split, sl = ks * NW + w;
  const int s0 = steps * sl / slices, s1 = steps * (sl + 1) / slices;
  const int lr = lane >> 2, lc = 8 * (lane & 3);   // a lane's row and values of the loads
  const uint16_t* wp = P.w + (int64_t)(f0 + lr) * P.K + lc;
  const uint16_t* xp[MT];
#pragma unroll
  for (int i = 0; i < MT; ++i) xp[i] = XP ? P.x + ((int64_t)i * steps * 64 + lane) * 8 : P.x + (int64_t)min(16 * i + lr, P.M - 1) * P.ldx + lc;
  u16x4 bias = (u16x4)(0);   // asked for with the rest: at the end it would be a latency of its own
  if (EPI == 2) bias[0] = P.bias[f0 + ((tid >> 7) & 1) * 8 + (tid & 7)];
  if (EPI == 0 && w < MT) bias = *reinterpret_cast<const u16x4*>(P.bias + f0 + 4 * h);
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
        for (int i = 0; i < MT - 1; ++i) bv[d][i] = load8(xp[i] + (XP ? 512 : 32) * (s + d));
      }
#pragma unroll
    for (int d = 0; d < PD; ++d) bv[d][MT - 1] = (u16x8)(0);
    if ((XP ? col : lr) < P.M - 16 * (MT - 1)) {   // lanes of rows that are not there bring nothing
#pragma unroll
      for (int d = 0; d < PD; ++d)
        if (s + d < s1) bv[d][MT - 1] = load8(xp[MT - 1] + (XP ? 512 : 32) * (s + d));
    }
  };
  load(s0, a, b);
  for (int s = s0; s < s1; s += PD) {
    if (s + PD < s1) load(s + PD, an, bn);
#pragma unroll
    for (int d = 0; d < PD; ++d)
      if (s + d < s1) {
        const bf16x8 af = gr_fragment(a[d], lane);
#pragma unroll
        for (int j = 0; j < MT; ++j) acc[j] = mfma16(af, XP ? as_bf16x8(b[d][j]) : gr_fragment(b[d][j], lane), acc[j]);
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
  if constexpr (EPI == 2) {
    // a value each thread, eight of a row side by side: with four to a lane of MT waves the four GELUs were half a microsecond
    if (tid >= MT * 256) return;
    const int t = (tid >> 8) * 16 + ((tid >> 3) & 15), f = ((tid >> 7) & 1) * 8 + (tid & 7);
    if (t >= P.M) return;
    const float* const at = part + ((t >> 4) * 64 + (f >> 2) * 16 + (t & 15)) * 4 + (f & 3);
    float v = at[0];
#pragma unroll
    for (int u = 1; u < NW; ++u) v += at[u * MT * 256];
    reinterpret_cast<uint16_t*>(P.out)[packed_at(t, f0 + f, P.N)] = f2bf(gelu_f(v + bf2f(bias[0])));
  } else {
    // tile w: features f0 + 4 h + 0..3 of token 16 w + col
    const int t = 16 * w + col, n = f0 + 4 * h;
    if (w >= MT || t >= P.M) return;
    f32x4 v = (f32x4)(0.f);
#pragma unroll
    for (int u = 0; u < NW; ++u) v += *reinterpret_cast<const f32x4*>(&part[((u * MT + w) * 64 + lane) * 4]);
    if constexpr (EPI == 1) {
      *reinterpret_cast<f32x4*>(reinterpret_cast<float*>(P.out) + ((int64_t)ks * P.M + t) * P.N + n) = v;
    } else {
      u16x4 o;
#pragma unroll
      for (int r = 0; r < 4; ++r) o[r] = f2bf(v[r] + bf2f(bias[r]));
      *reinterpret_cast<u16x4*>(reinterpret_cast<uint16_t*>(P.out) + (P.packed ? packed_at(t, n, P.N) : t * P.ldo + n)) = o;
    }
  }
}

// The attention of one sequence of up to 32 rows and the output projection behind it, as slabs [split, M, N]: x = q | k | v, a
// K slice is a few heads, and each of its N / 16 workgroups computes those heads by itself, a head's 16 queries a wave. As in
// attention_decode.hip the key order of S^T makes P^T the next operand; V comes transposed from LDS (ds_read_b64_tr_b16).
// (BERT-large, 19 rows: attention 4.5 and output 3.6 us in two launches, 5.4 in one.)
template <int MT, int D>
__global__ void __launch_bounds__(512) row_attn_gemm_kernel(RowGemmParams P) {
  constexpr int NW = 8, PD = 4, VL = D + 8, DS = D / 32, DT = D / 16;
  extern __shared__ __attribute__((aligned(16))) uint16_t sm[];   // [16 MT][columns + 8] rows, then V of each wave; partial sums
  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int col = lane & 15, h = lane >> 4;
  const int f0 = blockIdx.x * 16, ks = blockIdx.y, heads = P.K / D;
  const int h0 = heads * ks / P.split, h1 = heads * (ks + 1) / P.split, cols = (h1 - h0) * D, ld = cols + 8;
  const int steps = cols / 32, s0 = steps * w / NW, s1 = steps * (w + 1) / NW;
  const uint16_t* wp = P.w + (int64_t)(f0 + (lane >> 2)) * P.K + h0 * D + 8 * (lane & 3);
  u16x8 a[PD];
#pragma unroll
  for (int d = 0; d < PD; ++d) a[d] = s0 + d < s1 ? load8(wp + 32 * (s0 + d)) : (u16x8)(0);
  // rows beside the sequence are clamped into it: whatever those hold, it would be multiplied by 0
  const int lo = max(0, P.cu[0]), hi = min(P.M, P.cu[1]);
  auto row = [&](int r) { return min(max(lo, min(r, hi - 1)), P.M - 1); };
  uint16_t* const vh = sm + 16 * MT * ld + w * (16 * MT * VL);
  for (int u = w; u < (h1 - h0) * MT; u += NW) {
    const int hd = u / MT, i = u % MT;   // queries 16 i .. of head h0 + hd
    bf16x8 kf[MT][DS], qf[DS];
    u16x8 vr[MT * D / 32];
    const int at = (h0 + hd) * D;
#pragma unroll
    for (int s = 0; s < DS; ++s) {
      qf[s] = as_bf16x8(load8(P.x + packed_at(row(16 * i + col), at + 32 * s + 8 * h, 3 * P.K)));
#pragma unroll
      for (int t = 0; t < MT; ++t)   // row `col` of key tile t: key 8 (col / 4) + 4 t + col % 4 (of 16 keys: their order)
        kf[t][s] = as_bf16x8(load8(P.x + packed_at(row(MT == 2 ? 8 * (col >> 2) + 4 * t + (col & 3) : col), P.K + at + 32 * s + 8 * h, 3 * P.K)));
    }
    auto vrow = [&](int j) { return (64 * j + lane) % (16 * MT); };
    auto vcol = [&](int j) { return (64 * j + lane) / (16 * MT) * 8; };
#pragma unroll
    for (int j = 0; j < MT * D / 32; ++j) vr[j] = load8(P.x + packed_at(row(vrow(j)), 2 * P.K + at + vcol(j), 3 * P.K));
#pragma unroll
    for (int j = 0; j < MT * D / 32; ++j) store8(vh + vrow(j) * VL + vcol(j), vr[j]);
    f32x4 S[MT];
    float mx = -INFINITY;
#pragma unroll
    for (int t = 0; t < MT; ++t) {
      S[t] = (f32x4)(0.f);
#pragma unroll
      for (int s = 0; s < DS; ++s) S[t] = mfma16(kf[t][s], qf[s], S[t]);
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int key = MT == 2 ? 8 * h + 4 * t + r : 4 * h + r;
        S[t][r] = key >= lo && key < hi ? S[t][r] * (P.scale * 1.4426950408889634f) : -INFINITY;
        mx = fmaxf(mx, S[t][r]);
      }
    }
    mx = fmaxf(mx, __shfl_xor(mx, 16, 64));
    mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
    float l = 0.f;
    u16x8 pf = (u16x8)(0);
#pragma unroll
    for (int t = 0; t < MT; ++t)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const float e = __builtin_amdgcn_exp2f(S[t][r] - mx);
        l += e;
        pf[4 * t + r] = f2bf(e);
      }
    l += __shfl_xor(l, 16, 64);
    l += __shfl_xor(l, 32, 64);
    const float inv = l > 0.f ? 1.f / l : 0.f;
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) {
      // lane: dim 16 dt + col; keys 8 h .. 8 h + 7, of 16 keys 4 h .. 4 h + 3 and zeros
      uint16_t* const at = vh + ((MT == 2 ? 8 : 4) * h + (col >> 2)) * VL + 16 * dt + 4 * (col & 3);
      const s16x4 va = __builtin_amdgcn_ds_read_tr16_b64_v4i16((ltr_t)at);
      const s16x4 vb = MT == 2 ? __builtin_amdgcn_ds_read_tr16_b64_v4i16((ltr_t)(at + 4 * VL)) : (s16x4)(0);
      const auto v8 = __builtin_shufflevector(va, vb, 0, 1, 2, 3, 4, 5, 6, 7);
      const f32x4 o = mfma16(__builtin_bit_cast(bf16x8, v8), as_bf16x8(pf), (f32x4)(0.f));
      u16x4 ob;
#pragma unroll
      for (int r = 0; r < 4; ++r) ob[r] = f2bf(o[r] * inv);
      *reinterpret_cast<u16x4*>(sm + (16 * i + col) * ld + hd * D + 16 * dt + 4 * h) = ob;
    }
  }
  f32x4 acc[MT];
#pragma unroll
  for (int j = 0; j < MT; ++j) acc[j] = (f32x4)(0.f);
  __syncthreads();
  for (int s = s0; s < s1; s += PD) {
    if (s > s0)
#pragma unroll
      for (int d = 0; d < PD; ++d)
        if (s + d < s1) a[d] = load8(wp + 32 * (s + d));
#pragma unroll
    for (int d = 0; d < PD; ++d) {
      if (s + d >= s1) continue;
      const bf16x8 af = gr_fragment(a[d], lane);
#pragma unroll
      for (int j = 0; j < MT; ++j) acc[j] = mfma16(af, as_bf16x8(load8(sm + (16 * j + col) * ld + 32 * (s + d) + 8 * h)), acc[j]);
    }
  }
  float* const part = reinterpret_cast<float*>(sm + 16 * MT * ld);   // V is read
#pragma unroll
  for (int j = 0; j < MT; ++j) *reinterpret_cast<f32x4*>(&part[((w * MT + j) * 64 + lane) * 4]) = acc[j];
  __syncthreads();
#pragma unroll
  for (int j = 0; j < MT; ++j) {
    const int t = 16 * j + col;
    if (j != w || t >= P.M) continue;
    f32x4 v = (f32x4)(0.f);
#pragma unroll
    for (int u = 0; u < NW; ++u) v += *reinterpret_cast<const f32x4*>(&part[((u * MT + j) * 64 + lane) * 4]);
    *reinterpret_cast<f32x4*>(reinterpret_cast<float*>(P.out) + ((int64_t)ks * P.M + t) * P.N + f0 + 4 * h) = v;
  }
}

// A norm has a workgroup a row and waits for memory, and HBM lies idle: workgroups beside its own read the weights that the next
// launch streams, a word of each 64 bytes, so that they lie in the L2 that will ask for them. Workgroup `wg` of the `n` of a die. The
// norm takes 0.5 us longer for 8 MB, the product behind it up to 1.5 less: one query of 19 tokens of BERT-large 696 -> 655 us, eight
// queries 1,061 -> 1,040. From workgroups beside a product's own, whose end waits for HBM then, or with two products' weights: slower.
__device__ void read_ahead(const ReadAhead& R, int die, int wg, int n) {
  const int waves = blockDim.x >> 6, lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane(wg * waves + (threadIdx.x >> 6));
  constexpr int CH = 64 * 32, U = 8;   // values that a load of a wave touches; loads under way
  const int64_t piece = R.tiled ? (int64_t)(R.N / 8) * R.K : (int64_t)16 * R.K;
  const int per = (int)(piece / CH), total = R.tiled ? per : R.N / 128 * per;
  for (int k = w; k < total; k += U * n * waves) {
    uint32_t v[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int c = min(k + u * n * waves, total - 1);
      const int64_t at = R.tiled ? die * piece + (int64_t)c * CH : (die + 8 * (int64_t)(c / per)) * piece + (int64_t)(c % per) * CH;
      v[u] = *reinterpret_cast<const uint32_t*>(R.w + at + lane * 32);
    }
#pragma unroll
    for (int u = 0; u < U; ++u) asm volatile("" ::"v"(v[u]));
  }
}

// out = LN(sum_s P[s] + bias + resid): the norm behind a K-split projection (P [S, M, H] fp32). NS: S, with all slabs' loads
// in flight at once, or 0 (a loop waits for
// each: 19 rows of 8 slabs 4.6 us, here 3.7)
template <int NS>
__global__ void __launch_bounds__(1024) splitk_layernorm_kernel(const float* __restrict__ P, int S, int M,
                                                                const uint16_t* __restrict__ bias,
                                                                const uint16_t* __restrict__ resid,
                                                                const uint16_t* __restrict__ g, const uint16_t* __restrict__ b,
                                                                float eps, int H, uint16_t* __restrict__ out, uint16_t* __restrict__ packed,
                                                                ReadAhead next) {
  __shared__ float red[16];
  if ((int)blockIdx.x >= M) {
    read_ahead(next, blockIdx.x & 7, (blockIdx.x - M) >> 3, (gridDim.x - M) >> 3);
    return;
  }
  const int64_t row = blockIdx.x;
  const int c = threadIdx.x * 8;
  const bool active = c < H;
  const int64_t slab = (int64_t)M * H;
  float x[8], s = 0.f;
  u16x8 gv, bv;
  if (active) {
    const float* p = P + row * H + c;
    f32x4 a0, a1;
    const u16x8 r = load8(resid + row * H + c), bi = load8(bias + c);
    gv = load8(g + c);
    bv = load8(b + c);
    if constexpr (NS > 0) {
      f32x4 v[NS][2];
#pragma unroll
      for (int k = 0; k < NS; ++k) {
        v[k][0] = *reinterpret_cast<const f32x4*>(p + k * slab);
        v[k][1] = *reinterpret_cast<const f32x4*>(p + k * slab + 4);
      }
      a0 = v[0][0];
      a1 = v[0][1];
#pragma unroll
      for (int k = 1; k < NS; ++k) {
        a0 += v[k][0];
        a1 += v[k][1];
      }
    } else {
      a0 = *reinterpret_cast<const f32x4*>(p);
      a1 = *reinterpret_cast<const f32x4*>(p + 4);
      for (int k = 1; k < S; ++k) {
        a0 += *reinterpret_cast<const f32x4*>(p + k * slab);
        a1 += *reinterpret_cast<const f32x4*>(p + k * slab + 4);
      }
    }
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
    if (packed != nullptr) store8(packed + packed_at((int)row, c, H), o);
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
                                                               float eps, int H, uint16_t* __restrict__ out, uint16_t* __restrict__ packed) {
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
    if (packed != nullptr) store8(packed + packed_at((int)row, c, H), o);
  }
}

void launch_row_gemm(const RowGemmParams& p, int epi, hipStream_t stream) {
  if (p.M == 0 || p.N == 0) return;
  const int mt = p.M <= 16 ? 1 : 2;
  const dim3 grid(p.N / 16, p.split);
#define NGA_RG(MT_)                                                                                \
  if (mt == MT_) {                                                                                 \
    if (epi == 0) row_gemm_kernel<MT_, 0, true><<<grid, 512, 0, stream>>>(p);                      \
    else if (epi == 2) row_gemm_kernel<MT_, 2, true><<<grid, 512, 0, stream>>>(p);                 \
    else if (p.ldx == 0) row_gemm_kernel<MT_, 1, true><<<grid, 512, 0, stream>>>(p);               \
    else row_gemm_kernel<MT_, 1, false><<<grid, 512, 0, stream>>>(p);                              \
    return;                                                                                        \
  }
  NGA_RG(1) NGA_RG(2)
#undef NGA_RG
}

// K slices of it: four heads each, eight at most
int row_attn_split(int heads) { return heads <= 4 ? 1 : heads <= 32 ? (heads + 3) / 4 : 8; }

void launch_row_attn_gemm(const RowGemmParams& p, int D, hipStream_t stream) {
  if (p.M == 0 || p.N == 0) return;
  const int mt = p.M <= 16 ? 1 : 2, heads = p.K / D;
  const size_t cols = (size_t)((heads + p.split - 1) / p.split) * D, sums = (size_t)8 * mt * 1024, v = (size_t)8 * 16 * mt * (D + 8) * 2;
  const size_t lds = 16 * mt * (cols + 8) * 2 + (v > sums ? v : sums);
#define NGA_RA(MT_, DD)                                                                                    \
  {                                                                                                        \
    static const hipError_t attr = hipFuncSetAttribute((const void*)row_attn_gemm_kernel<MT_, DD>,         \
                                                       hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024); \
    (void)attr;                                                                                            \
    row_attn_gemm_kernel<MT_, DD><<<dim3(p.N / 16, p.split), 512, lds, stream>>>(p);                    \
  }
#define NGA_RD(MT_) if (D == 32) NGA_RA(MT_, 32) else if (D == 64) NGA_RA(MT_, 64) else NGA_RA(MT_, 128)
  if (mt == 1) { NGA_RD(1) } else { NGA_RD(2) }
#undef NGA_RD
#undef NGA_RA
}

static int rows_threads(int H) { return (H / 8 + 63) / 64 * 64; }

// Up to how many weights reading ahead gains: what a die's 4 MB of L2 do not hold until the product comes is read twice, and the norm takes as long as
// the whole stream. A layer, us, without / q/k/v's / up's too, at 19 rows: hidden 1,024 27.6 26.5 25.8, 1,536 44.2 42.1 41.4, 2,048 51.9 51.1 50.7,
// 2,304 66.2 66.2 66.3, 2,560 74.2 74.1 76.0, 4,096 137 143 153. Tiles come with token rows beside their weights, so their line lies lower, and lower
// still with many: at 64 / 208 / 512 / 768 rows 1,024 38.2 43.4 56.6 69.2, 37.9 42.7 55.9 69.2, 37.6 42.5 54.7 68.4; 1,280 43.4 56.8 74.6 81.9, 42.8 56.6
// 73.1 82.2, 42.4 54.9 72.8 83.2; 1,536 46.1 64.2 85.5 126, 45.8 63.6 85.7 127, 46.3 63.4 86.2 129; 2,048 54.7 74.5 107 181, 55.7 76.7 109 184, 57.2 78.5
// 112 186. Other numbers of weights than multiples of 128 are not dealt out
bool norm_reads_ahead(int64_t M, int64_t N, int64_t K, bool tiled) {
  return N % 128 == 0 && K % 128 == 0 && N * K <= (!tiled ? 1 << 24 : M <= 512 ? 6600000 : 1 << 22);
}

void launch_splitk_layernorm(const float* P, int S, int M, const uint16_t* bias, const uint16_t* resid, const uint16_t* g,
                             const uint16_t* b, float eps, int H, uint16_t* out, uint16_t* packed, const ReadAhead& next, hipStream_t stream) {
  if (M == 0) return;
  // 32 workgroups a die have 8 MB under way at once; 16 and 64 a die were 1 % slower
  const int beside = next.w != nullptr && norm_reads_ahead(M, next.N, next.K, next.tiled) ? 256 : 0;
#define NGA_SL(NS) splitk_layernorm_kernel<NS><<<M + beside, rows_threads(H), 0, stream>>>(P, S, M, bias, resid, g, b, eps, H, out, packed, next)
  if (S == 1) NGA_SL(1);
  else if (S == 2) NGA_SL(2);
  else if (S == 3) NGA_SL(3);
  else if (S == 4) NGA_SL(4);
  else if (S == 8) NGA_SL(8);
  else NGA_SL(0);
#undef NGA_SL
}

void launch_embed_layernorm(const int32_t* ids, const int32_t* pos, const int32_t* types, const uint16_t* word, int n_word,
                            const uint16_t* ptab, int n_pos, const uint16_t* ttab, int n_type, const uint16_t* g,
                            const uint16_t* b, float eps, int64_t rows, int H, uint16_t* out, uint16_t* packed, hipStream_t stream) {
  if (rows == 0) return;
  embed_layernorm_kernel<<<(unsigned)rows, rows_threads(H), 0, stream>>>(ids, pos, types, word, n_word, ptab, n_pos, ttab, n_type,
                                                                         g, b, eps, H, out, packed);
}

}  // namespace nga
