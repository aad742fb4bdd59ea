// Gradients of causal attention over packed variable-length sequences, head_dim 32, 64 or 128, 32x32x16 MFMA. Probabilities are
// formed again from the scores and the row's log-sum:
//   P = 2^(s - lse),  dV = P^T dO,  dP = dO V^T,  dS = P (dP - delta),  dQ = scale dS K,  dK = scale dS^T Q,
// delta = rowsum(dO O). Two kernels, so that nothing is added up through memory and the result does not depend on order:
//   dk/dv  a wave owns 32 keys. S[q][key] = Q K^T with the Q rows of an LDS tile as A operand and the keys in registers as
//          B; a lane then holds one key and 8 consecutive queries per register half, which is the B operand of
//          dV^T[d][key] = dO^T[d][q] P[q][key] and of dK^T = Q^T dS. dO^T and Q^T come from the row-major LDS tiles by the
//          transpose read. The query heads of a KV head follow one another.
//   dq     a wave owns 32 queries: the forward's loop over key tiles with dP^T = V dO^T beside S^T, and
//          dQ^T[d][q] = K^T[d][key] dS^T[key][q], K^T by the transpose read.
// A wave alone on its SIMD waits for its own products, exponentials and LDS reads in turn (heads of 128, whose sums and operands
// fill 440 registers), so there two waves share each 32 keys or queries and take the halves of every tile (HW 2): their sums meet
// in LDS at the end, and V (dk/dv) stays in LDS. Three buffers instead of two were 8 to 16 % slower: it is not the tiles' latency.
// 8 x 2,048 tokens, 32 / 8 heads of 128: 1.20 ms (574 TFLOP/s; one wave 1.80; torch's flash attention 4.00), 2 x 512 54 us (74),
// 32 x 16 30 (32); 4 x 1,024, 12 heads of 64: 71 us (84). Of these, rows brought in and out in whole pieces through LDS gave 8 % and 5 %,
// masks in a branch and tile addresses from a scalar 7 % (12 % with heads of 64), delta from the dq kernel's rows instead of a launch 4 %.
// Tiles by LDS-DMA as they lie in memory, two buffers, as in the forward. Chunk swizzle: 16 rows of one chunk and 64 bytes of
// 4 consecutive rows both fall into distinct banks.
#include "common.h"
#include "kernels.h"

namespace nga {

namespace {
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) s16x4* ltr_t;

constexpr float AB_LOG2E = 1.4426950408889634f;

template <int D>
__device__ __forceinline__ int ab_swz(int row) {
  if constexpr (D == 128) return ((row & 3) << 2) | ((row >> 2) & 3);
  if constexpr (D == 64) return (((row >> 1) & 1) << 2) | ((row >> 2) & 3);
  return (row >> 2) & 3;
}

__device__ __forceinline__ f32x16 ab_mfma(bf16x8 a, bf16x8 b, f32x16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
}

// 32 dims (rows of the MFMA) x 8 tile rows of a row-major LDS tile; four rows on, the swizzle's lowest bit (the eighth
// element) is the other one
template <int D>
__device__ __forceinline__ bf16x8 ab_tr(const uint16_t* tile, int off) {
  uint16_t* p = const_cast<uint16_t*>(tile);
  const s16x4 a = __builtin_amdgcn_ds_read_tr16_b64_v4i16((ltr_t)(p + off));
  const s16x4 b = __builtin_amdgcn_ds_read_tr16_b64_v4i16((ltr_t)(p + (off ^ 8) + 4 * D));
  return __builtin_bit_cast(bf16x8, __builtin_shufflevector(a, b, 0, 1, 2, 3, 4, 5, 6, 7));
}

// a lane's part of transposed fragments: 32-dim tile dt, tile rows 16 s + 8 h + 0..7 at base + off[dt] + 16 s D
template <int D>
__device__ __forceinline__ void ab_tr_offsets(int lane, int (&off)[D / 32]) {
  const int h = lane >> 5, row = 8 * h + ((lane & 15) >> 2), dim = 16 * ((lane >> 4) & 1) + 4 * (lane & 3);
#pragma unroll
  for (int dt = 0; dt < D / 32; ++dt) {
    const int d = 32 * dt + dim;
    off[dt] = row * D + (((d >> 3) ^ ab_swz<D>(row)) << 3) + (d & 7);
  }
}

// 128 rows acc[dt][j] (dim 32 dt + (j & 3) + 8 (j >> 2) + 4 h, one row a lane, 32 a wave with `mine`) times f, through LDS to the
// first `rows` rows of out: a lane's own pieces are 8 or 16 bytes at the rows' stride
template <int D, typename T>
__device__ __forceinline__ void ab_store(T* out, int64_t stride, int rows, const f32x16 (&acc)[D / 32], float f, bool mine, int group,
                                         int lane, void* lds) {
  constexpr int E = 16 / sizeof(T), C = D / E;   // values of a 16-byte chunk, chunks of a row: chunk c of row r lies at c ^ r (mod C)
  T* const tile = static_cast<T*>(lds);
  const int h = lane >> 5, row = 32 * group + (lane & 31);
  __syncthreads();
  if (mine)
#pragma unroll
    for (int dt = 0; dt < D / 32; ++dt)
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const int d = 32 * dt + 8 * g + 4 * h;
        T* to = tile + row * D + (((d / E) ^ (row % C)) * E) + d % E;
        f32x4 v;
#pragma unroll
        for (int j = 0; j < 4; ++j) v[j] = acc[dt][4 * g + j] * f;
        if constexpr (E == 4) *reinterpret_cast<f32x4*>(to) = v;
        else *reinterpret_cast<u16x4*>(to) = (u16x4){f2bf(v[0]), f2bf(v[1]), f2bf(v[2]), f2bf(v[3])};
      }
  __syncthreads();
  for (int i = threadIdx.x; i < min(rows, 128) * C; i += blockDim.x) {
    const int r = i / C, c = i % C;
    *reinterpret_cast<f32x4*>(out + r * stride + c * E) = *reinterpret_cast<const f32x4*>(tile + r * D + ((c ^ (r % C)) * E));
  }
}

// Up to 128 rows to LDS as they lie, chunks swizzled, by 8 waves; and a wave's fragments of 32 of them. Of rows past the last
// nothing is asked, and what their lanes compute from the LDS as it was stays in those lanes and is not stored.
template <int D>
__device__ __forceinline__ void ab_rows_in(const uint16_t* src, int64_t stride, int rows, uint16_t* lds, int w, int lane) {
  constexpr int N = 128 * (D / 8) / 512;
#pragma unroll
  for (int i = 0; i < N; ++i) {
    const int p = (N * w + i) * 64 + lane, row = p / (D / 8);
    if ((N * w + i) * 512 / D < rows) glds16(src + min(row, rows - 1) * stride + ((p % (D / 8)) ^ ab_swz<D>(row)) * 8, lds + (N * w + i) * 512);
  }
}
template <int D>
__device__ __forceinline__ bf16x8 ab_frag(const uint16_t* lds, int row, int chunk) {
  return as_bf16x8(*reinterpret_cast<const u16x8*>(lds + row * D + ((chunk ^ ab_swz<D>(row)) << 3)));
}

// acc of the wave that took the first halves += that of the one that took the second
template <int DT>
__device__ __forceinline__ void ab_add_halves(f32x16 (&acc)[DT], float* red, int group, int half, int lane) {
  f32x4* at = reinterpret_cast<f32x4*>(red) + group * DT * 4 * 64 + lane;
  __syncthreads();
#pragma unroll
  for (int i = 0; i < DT * 4; ++i)
    if (half) at[64 * i] = (f32x4){acc[i / 4][4 * (i % 4)], acc[i / 4][4 * (i % 4) + 1], acc[i / 4][4 * (i % 4) + 2], acc[i / 4][4 * (i % 4) + 3]};
  __syncthreads();
  if (half) return;
#pragma unroll
  for (int i = 0; i < DT * 4; ++i) {
    const f32x4 v = at[64 * i];
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i / 4][4 * (i % 4) + j] += v[j];
  }
}
}  // namespace

// a row's log-sum from lse_in
__device__ __forceinline__ float ab_lse(const AttnBwdParams& P, uint32_t t, int hq) {
  const uint32_t S = (uint32_t)P.S;
  return P.lse_in[((int64_t)(t / S) * P.Hq + hq) * S + t % S] * AB_LOG2E;
}

// delta[hq][t] = sum_d dO O; 8 dims a lane. Where two waves share 32 rows the dq kernel works it out instead. Log-sums as torch's attention
// leaves them, natural and by sequence, become lse beside it (single operations: 9.6 us a call at 2 x 512 tokens, 32 heads).
template <int D>
__global__ void __launch_bounds__(256) attn_delta_kernel(AttnBwdParams P) {
  constexpr int LPR = D / 8;
  const int64_t i = ((int64_t)blockIdx.x * 256 + threadIdx.x) / LPR;
  const int c = (threadIdx.x % LPR) * 8;
  if (i >= P.T * P.Hq) return;
  const int64_t t = i / P.Hq;
  const int hq = (int)(i % P.Hq);
  const u16x8 a = load8(P.out + t * P.out_stride + (int64_t)hq * D + c), b = load8(P.dout + t * P.dout_stride + (int64_t)hq * D + c);
  float s = 0.f;
#pragma unroll
  for (int j = 0; j < 8; ++j) s += bf2f(a[j]) * bf2f(b[j]);
#pragma unroll
  for (int o = LPR / 2; o > 0; o >>= 1) s += __shfl_xor(s, o, 64);
  if (c == 0) {
    P.delta[(int64_t)hq * P.T + t] = s;
    if (P.lse_in) P.lse[(int64_t)hq * P.T + t] = ab_lse(P, (uint32_t)t, hq);
  }
}

// dk, dv [T, Hkv D] = the sums over the head parts of part [parts, 2, T, Hkv D]
__global__ void __launch_bounds__(256) attn_sum_parts_kernel(AttnBwdParams P, int width) {
  const int64_t n = P.T * width, i = (blockIdx.x * 256ll + threadIdx.x) * 4;
  if (i >= n) return;
  f32x4 a = (f32x4)(0.f), b = (f32x4)(0.f);
  for (int u = 0; u < P.parts; ++u) {
    a += *reinterpret_cast<const f32x4*>(P.part + 2 * u * n + i);
    b += *reinterpret_cast<const f32x4*>(P.part + (2 * u + 1) * n + i);
  }
  const int64_t at = i / width * P.dkv_stride + i % width;
  *reinterpret_cast<u16x4*>(P.dk + at) = (u16x4){f2bf(a[0]), f2bf(a[1]), f2bf(a[2]), f2bf(a[3])};
  *reinterpret_cast<u16x4*>(P.dv + at) = (u16x4){f2bf(b[0]), f2bf(b[1]), f2bf(b[2]), f2bf(b[3])};
}

template <int D, int HW>
__global__ void __launch_bounds__(256 * HW, D == 128 ? HW : 2) attn_bwd_dkdv_kernel(AttnBwdParams P) {
  constexpr int QT = 64, NC = D / 8, TILE = QT * D, NI = D / 32 / HW, DS = D / 16, DT = D / 32, KW = 128;
  // one LDS object: [Q 0 | Q 1 | dO 0 | dO 1 | lse 0 | lse 1 | delta 0 | delta 1], then V, which the registers of two waves a SIMD do
  // not hold, and K on its way into them
  constexpr int VS = 4 * TILE + 4 * 2 * QT;
  __shared__ __attribute__((aligned(16))) uint16_t smem[VS + (HW == 2 ? 2 * KW * D : 0)];
  uint16_t *const qbuf = smem, *const obuf = smem + 2 * TILE;
  float* const lbuf = reinterpret_cast<float*>(smem + 4 * TILE);
  const int pblk = blockIdx.x, Lb = (pblk & 7) * P.per_xcd + (pblk >> 3);
  if (Lb >= P.total) return;
  // a part takes some of the query heads of its KV head
  const int kb = Lb % P.ntiles, pu = (Lb / P.ntiles) % P.parts, kvh = (Lb / (P.ntiles * P.parts)) % P.Hkv;
  const int b = Lb / (P.ntiles * P.parts * P.Hkv);
  const int q0 = P.cu[b], len = P.cu[b + 1] - q0;
  if (kb * KW >= len) return;
  const int G = P.Hq / P.Hkv / P.parts, hq0 = (kvh * P.parts + pu) * G;
  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6), kg = w % 4;
  const int r32 = lane & 31, h = lane >> 5;
  const int k0 = kb * KW + 32 * kg;           // the wave's first key
  const bool active = k0 < len;
  const int key = k0 + r32, kr = min(key, len - 1);

  bf16x8 kf[DS], vf[HW == 2 ? 1 : DS];
  uint16_t *const vt = smem + VS, *const kt = vt + KW * D;
  {
    const int64_t at = (int64_t)(q0 + kb * KW) * P.kv_stride + (int64_t)kvh * D;
    if constexpr (HW == 2) {
      ab_rows_in<D>(P.k + at, P.kv_stride, len - kb * KW, kt, w, lane);
      ab_rows_in<D>(P.v + at, P.kv_stride, len - kb * KW, vt, w, lane);
    } else if (active) {
#pragma unroll
      for (int s = 0; s < DS; ++s) {
        kf[s] = as_bf16x8(load8(P.k + at + (kr - kb * KW) * P.kv_stride + 8 * h + 16 * s));
        vf[s] = as_bf16x8(load8(P.v + at + (kr - kb * KW) * P.kv_stride + 8 * h + 16 * s));
      }
    }
  }
  // query tiles that see any key of the workgroup, for each head of the group in turn
  const int n_tiles = (len - 1) / QT + 1;
  const int t_first = kb * KW / QT;
  const int per_head = n_tiles - t_first, total = per_head * G;

  // a lane's place in a tile, to be added to the tile's address (scalar); a last tile that is not full repeats its last row, and
  // what comes of the repeated ones is masked
  const uint32_t qstep = (uint32_t)P.q_stride, ostep = (uint32_t)P.dout_stride;
  uint32_t prow_[NI], pcol[NI], qoff[NI], ooff[NI];
#pragma unroll
  for (int i = 0; i < NI; ++i) {
    const int p = (NI * w + i) * 64 + lane;
    prow_[i] = p / NC;
    pcol[i] = ((p % NC) ^ ab_swz<D>(prow_[i])) * 8;
    qoff[i] = prow_[i] * qstep + pcol[i];
    ooff[i] = prow_[i] * ostep + pcol[i];
  }
  auto issue = [&](int it, int buf) {
    const int hq = hq0 + it / per_head, t = t_first + it % per_head;
    const uint32_t left = len - 1 - t * QT;
    const uint16_t* const qt = P.q + (int64_t)(q0 + t * QT) * P.q_stride + (int64_t)hq * D;
    const uint16_t* const ot = P.dout + (int64_t)(q0 + t * QT) * P.dout_stride + (int64_t)hq * D;
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      uint32_t a = qoff[i], c = ooff[i];
      if (left < QT - 1) {
        a = min(prow_[i], left) * qstep + pcol[i];
        c = min(prow_[i], left) * ostep + pcol[i];
      }
      glds16(qt + a, qbuf + buf * TILE + (NI * w + i) * 512);
      glds16(ot + c, obuf + buf * TILE + (NI * w + i) * 512);
    }
    if (w < 2) {
      const float* src = (w == 0 ? P.lse : P.delta) + (int64_t)hq * P.T + q0 + min(t * QT + lane, len - 1);
      __builtin_amdgcn_global_load_lds((gptr_t)src, (lptr_t)(lbuf + (2 * w + buf) * QT), 4, 0, 0);
    }
  };
  const int prow = (r32 & ~12) | ((r32 & 4) << 1) | ((r32 & 8) >> 1);
  const int psw = ab_swz<D>(prow);   // of prow + 32 too
  int troff[DT];
  ab_tr_offsets<D>(lane, troff);
  const float sl2 = P.scale * AB_LOG2E;
  f32x16 dk[DT], dv[DT];
#pragma unroll
  for (int dt = 0; dt < DT; ++dt) dk[dt] = dv[dt] = (f32x16)(0.f);

  if (total > 0) issue(0, 0);
  if constexpr (HW == 2) {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
#pragma unroll
    for (int s = 0; s < DS; ++s) kf[s] = ab_frag<D>(kt, 32 * kg + r32, 2 * s + h);
  }
  for (int it = 0; it < total; ++it) {
    const int buf = it & 1, t = t_first + it % per_head;
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    if (it + 1 < total) issue(it + 1, buf ^ 1);
    if (!active || t * QT + QT - 1 < k0) continue;
    const uint16_t *qs = qbuf + buf * TILE, *os = obuf + buf * TILE;
    const float *ls = lbuf + buf * QT, *ds = lbuf + (2 + buf) * QT;
#pragma unroll
    for (int u = 0; u < 2 / HW; ++u) {
      const int h2 = HW == 2 ? w / 4 : u;
      f32x16 S = (f32x16)(0.f), dP = (f32x16)(0.f);
#pragma unroll
      for (int s = 0; s < DS; ++s) {
        const int at = (32 * h2 + prow) * D + (((2 * s + h) ^ psw) << 3);
        S = ab_mfma(as_bf16x8(*reinterpret_cast<const u16x8*>(qs + at)), kf[s], S);
        const bf16x8 v = HW == 2 ? ab_frag<D>(vt, 32 * kg + r32, 2 * s + h) : vf[HW == 2 ? 0 : s];
        dP = ab_mfma(as_bf16x8(*reinterpret_cast<const u16x8*>(os + at)), v, dP);
      }
      const int qbase = t * QT + 32 * h2;
      const bool need = qbase + 32 > len || qbase < k0 + 31;
      bf16x8 pf[2], df[2];
      const int ql = 32 * h2 + 8 * h;
#pragma unroll
      for (int j = 0; j < 16; ++j) S[j] = __builtin_amdgcn_exp2f(__builtin_fmaf(S[j], sl2, -ls[ql + 16 * (j >> 3) + (j & 7)]));
      if (need) {   // the diagonal and the end, a branch of the whole wave: its 64 instructions are a third of the others
        asm volatile("");
#pragma unroll
        for (int j = 0; j < 16; ++j) {
          const int q = t * QT + ql + 16 * (j >> 3) + (j & 7);
          S[j] = q < len && key <= q ? S[j] : 0.f;
        }
      }
#pragma unroll
      for (int j = 0; j < 16; ++j) {
        pf[j >> 3][j & 7] = (__bf16)S[j];
        df[j >> 3][j & 7] = (__bf16)(S[j] * (dP[j] - ds[ql + 16 * (j >> 3) + (j & 7)]));
      }
#pragma unroll
      for (int dt = 0; dt < DT; ++dt)
#pragma unroll
        for (int s = 0; s < 2; ++s) {
          const int at = troff[dt] + (32 * h2 + 16 * s) * D;
          dv[dt] = ab_mfma(ab_tr<D>(os, at), pf[s], dv[dt]);
          dk[dt] = ab_mfma(ab_tr<D>(qs, at), df[s], dk[dt]);
        }
    }
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // no DMA may outlive the workgroup
  if constexpr (HW == 2) {
    ab_add_halves<DT>(dk, reinterpret_cast<float*>(smem), kg, w / 4, lane);
    ab_add_halves<DT>(dv, reinterpret_cast<float*>(smem), kg, w / 4, lane);
  }
  const int rows = len - kb * KW;
  if (P.parts > 1) {
    const int64_t n = P.T * P.Hkv * D, width = (int64_t)P.Hkv * D;
    float* pk = P.part + 2 * pu * n + (int64_t)(q0 + kb * KW) * width + (int64_t)kvh * D;
    ab_store<D>(pk, width, rows, dk, P.scale, w < 4, kg, lane, smem);
    ab_store<D>(pk + n, width, rows, dv, 1.f, w < 4, kg, lane, smem);
  } else {
    const int64_t at = (int64_t)(q0 + kb * KW) * P.dkv_stride + (int64_t)kvh * D;
    ab_store<D>(P.dk + at, P.dkv_stride, rows, dk, P.scale, w < 4, kg, lane, smem);
    ab_store<D>(P.dv + at, P.dkv_stride, rows, dv, 1.f, w < 4, kg, lane, smem);
  }
}

template <int D, int HW>
__global__ void __launch_bounds__(256 * HW, D == 128 ? HW : 2) attn_bwd_dq_kernel(AttnBwdParams P) {
  constexpr int KT = 64, NC = D / 8, TILE = KT * D, NI = D / 32 / HW, DS = D / 16, DT = D / 32, RW = 128;
  // [K 0 | K 1 | V 0 | V 1], then Q and dO on their way into registers
  __shared__ __attribute__((aligned(16))) uint16_t smem[4 * TILE + (HW == 2 ? 2 * RW * D : 0)];
  uint16_t *const kbuf = smem, *const vbuf = smem + 2 * TILE;
  const int pblk = blockIdx.x, Lb = (pblk & 7) * P.per_xcd + (pblk >> 3);
  if (Lb >= P.total) return;
  const int qb = P.ntiles - 1 - Lb % P.ntiles, hq = (Lb / P.ntiles) % P.Hq, b = Lb / (P.ntiles * P.Hq);
  const int q0 = P.cu[b], len = P.cu[b + 1] - q0;
  if (qb * RW >= len) return;
  const int kvh = hq / (P.Hq / P.Hkv);
  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r32 = lane & 31, h = lane >> 5;
  const int row0 = qb * RW + 32 * (w % 4);
  const bool active = row0 < len;
  const int qr = min(row0 + r32, len - 1);
  bf16x8 qf[DS], of[DS];
  uint16_t *const qt = smem + 4 * TILE, *const ot = qt + RW * D;
  {
    const uint16_t* qp = P.q + (int64_t)(q0 + qb * RW) * P.q_stride + (int64_t)hq * D;
    const uint16_t* op = P.dout + (int64_t)(q0 + qb * RW) * P.dout_stride + (int64_t)hq * D;
    if constexpr (HW == 2) {
      ab_rows_in<D>(qp, P.q_stride, len - qb * RW, qt, w, lane);
      ab_rows_in<D>(op, P.dout_stride, len - qb * RW, ot, w, lane);
      // O, for delta, in the second tile's buffers, which lie a tile apart
      ab_rows_in<D>(P.out + (int64_t)(q0 + qb * RW) * P.out_stride + (int64_t)hq * D, P.out_stride, len - qb * RW,
                    smem + (w < 4 ? 1 : 2) * TILE, w, lane);
    } else if (active) {
#pragma unroll
      for (int s = 0; s < DS; ++s) {
        qf[s] = as_bf16x8(load8(qp + (qr - qb * RW) * P.q_stride + 8 * h + 16 * s));
        of[s] = as_bf16x8(load8(op + (qr - qb * RW) * P.dout_stride + 8 * h + 16 * s));
      }
    }
  }
  const int64_t stat = (int64_t)hq * P.T + q0 + qr;
  float lse = P.lse_in ? ab_lse(P, q0 + qr, hq) : P.lse[stat], delta = HW == 2 ? 0.f : P.delta[stat];
  const int hi_w = min(len - 1, row0 + 31);
  const int n_tiles = min(len - 1, qb * RW + RW - 1) / KT + 1;
  const int w_last = hi_w / KT;
  const uint32_t step = (uint32_t)P.kv_stride;   // as in dk/dv
  uint32_t prow_[NI], pcol[NI], off[NI];
#pragma unroll
  for (int i = 0; i < NI; ++i) {
    const int p = (NI * w + i) * 64 + lane;
    prow_[i] = p / NC;
    pcol[i] = ((p % NC) ^ ab_swz<D>(prow_[i])) * 8;
    off[i] = prow_[i] * step + pcol[i];
  }
  const uint16_t* const kp = P.k + (int64_t)q0 * P.kv_stride + (int64_t)kvh * D;
  const uint16_t* const vp = P.v + (int64_t)q0 * P.kv_stride + (int64_t)kvh * D;
  auto issue = [&](int t, int buf) {
    const uint32_t left = len - 1 - t * KT;
    const uint16_t *const kt = kp + (int64_t)t * KT * P.kv_stride, *const vt = vp + (int64_t)t * KT * P.kv_stride;
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      uint32_t a = off[i];
      if (left < KT - 1) a = min(prow_[i], left) * step + pcol[i];
      glds16(kt + a, kbuf + buf * TILE + (NI * w + i) * 512);
      glds16(vt + a, vbuf + buf * TILE + (NI * w + i) * 512);
    }
  };
  const int prow = (r32 & ~12) | ((r32 & 4) << 1) | ((r32 & 8) >> 1);
  const int psw = ab_swz<D>(prow);
  int troff[DT];
  ab_tr_offsets<D>(lane, troff);
  const float sl2 = P.scale * AB_LOG2E;
  f32x16 dq[DT];
#pragma unroll
  for (int dt = 0; dt < DT; ++dt) dq[dt] = (f32x16)(0.f);

  issue(0, 0);
  if constexpr (HW == 2) {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
#pragma unroll
    for (int s = 0; s < DS; ++s) {
      qf[s] = ab_frag<D>(qt, 32 * (w % 4) + r32, 2 * s + h);
      of[s] = ab_frag<D>(ot, 32 * (w % 4) + r32, 2 * s + h);
      const bf16x8 o = ab_frag<D>(smem + (w % 4 < 2 ? 1 : 2) * TILE, 32 * (w % 4) + r32, 2 * s + h);
#pragma unroll
      for (int j = 0; j < 8; ++j) delta = __builtin_fmaf((float)of[s][j], (float)o[j], delta);
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");   // the second tile comes behind the next barrier
    delta += __shfl_xor(delta, 32, 64);
    if (w < 4 && h == 0 && row0 + r32 < len) {
      P.delta[stat] = delta;
      if (P.lse_in) P.lse[stat] = lse;
    }
  }
  for (int t = 0; t < n_tiles; ++t) {
    const int buf = t & 1;
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    if (t + 1 < n_tiles) issue(t + 1, buf ^ 1);
    if (!active || t > w_last) continue;
    const uint16_t *ks = kbuf + buf * TILE, *vs = vbuf + buf * TILE;
#pragma unroll
    for (int u = 0; u < 2 / HW; ++u) {
      const int h2 = HW == 2 ? w / 4 : u;
      f32x16 S = (f32x16)(0.f), dP = (f32x16)(0.f);
#pragma unroll
      for (int s = 0; s < DS; ++s) {
        const int at = (32 * h2 + prow) * D + (((2 * s + h) ^ psw) << 3);
        S = ab_mfma(as_bf16x8(*reinterpret_cast<const u16x8*>(ks + at)), qf[s], S);
        dP = ab_mfma(as_bf16x8(*reinterpret_cast<const u16x8*>(vs + at)), of[s], dP);
      }
      const int kbase = t * KT + 32 * h2;
      const bool need = kbase + 32 > len || kbase + 31 > row0;
      bf16x8 df[2];
#pragma unroll
      for (int j = 0; j < 16; ++j) S[j] = __builtin_amdgcn_exp2f(__builtin_fmaf(S[j], sl2, -lse));
      if (need) {
        asm volatile("");
#pragma unroll
        for (int j = 0; j < 16; ++j) S[j] = kbase + 8 * h + 16 * (j >> 3) + (j & 7) <= qr ? S[j] : 0.f;
      }
#pragma unroll
      for (int j = 0; j < 16; ++j) df[j >> 3][j & 7] = (__bf16)(S[j] * (dP[j] - delta));
#pragma unroll
      for (int dt = 0; dt < DT; ++dt)
#pragma unroll
        for (int s = 0; s < 2; ++s) dq[dt] = ab_mfma(ab_tr<D>(ks, troff[dt] + (32 * h2 + 16 * s) * D), df[s], dq[dt]);
    }
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  if constexpr (HW == 2) ab_add_halves<DT>(dq, reinterpret_cast<float*>(smem), w % 4, w / 4, lane);
  ab_store<D>(P.dq + (int64_t)(q0 + qb * RW) * P.dq_stride + (int64_t)hq * D, P.dq_stride, len - qb * RW, dq, P.scale, w < 4, w % 4, lane,
              smem);
}

template <int D, int HW>
static void attn_bwd(AttnBwdParams p, int num_seqs, int max_len, hipStream_t stream) {
  p.ntiles = (max_len + 127) / 128;
  const auto dq = [&](AttnBwdParams p) {
    p.total = p.ntiles * p.Hq * num_seqs;
    p.per_xcd = (p.total + 7) / 8;
    attn_bwd_dq_kernel<D, HW><<<8 * p.per_xcd, 256 * HW, 0, stream>>>(p);
  };
  if (HW == 1) {
    const int64_t dl = p.T * p.Hq * (D / 8);
    attn_delta_kernel<D><<<(unsigned)((dl + 255) / 256), 256, 0, stream>>>(p);
  } else {
    dq(p);
  }
  p.total = p.ntiles * p.parts * p.Hkv * num_seqs;
  p.per_xcd = (p.total + 7) / 8;
  attn_bwd_dkdv_kernel<D, HW><<<8 * p.per_xcd, 256 * HW, 0, stream>>>(p);
  if (p.parts > 1) attn_sum_parts_kernel<<<(unsigned)((p.T * p.Hkv * D / 4 + 255) / 256), 256, 0, stream>>>(p, p.Hkv * D);
  if (HW == 1) dq(p);
}

// The query heads of a KV head one workgroup each, their sums added up after, while key tiles alone leave most CUs idle
// (2 x 512 tokens, 32 / 8 heads of 128: 64 workgroups in one part, 256 in four; backward 153 -> 78 us; torch's
// flash attention 155).
int attn_bwd_parts(int num_seqs, int max_len, int Hq, int Hkv) {
  return (int64_t)((max_len + 127) / 128) * Hkv * num_seqs < 256 ? Hq / Hkv : 1;
}

// Two waves for 32 rows where a sequence is longer than one tile of 64, us against one wave: 32 x 64 tokens 50 47, 8 x 64 31 30, 2 x 96 28
// 30, 32 x 128 81 85, 16 x 32 42 34; 32 / 8 heads
void launch_varlen_attention_backward(const AttnBwdParams& p, int num_seqs, int max_len, int D, hipStream_t stream) {
  if (num_seqs == 0 || max_len == 0 || p.T == 0) return;
  if (D == 128 && max_len > 64) attn_bwd<128, 2>(p, num_seqs, max_len, stream);
  else if (D == 128) attn_bwd<128, 1>(p, num_seqs, max_len, stream);
  else if (D == 64) attn_bwd<64, 1>(p, num_seqs, max_len, stream);
  else if (D == 32) attn_bwd<32, 1>(p, num_seqs, max_len, stream);
}

}  // namespace nga
