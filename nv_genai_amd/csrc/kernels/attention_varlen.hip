// Attention over packed variable-length sequences without a cache (K10: encoders, rerankers, vision towers, reward
// models), bidirectional or causal, head_dim 32, 64 or 128, 32x32x16 MFMA.
//
// Workgroup = 4 waves, each with 32 query rows: four row blocks of one head, or (HPW 4, a multiple of four query heads
// per KV head) the same 32 rows of four heads, so that short sequences waste fewer rows. Per 64-key tile:
//   S^T = K . Q^T     A = K rows from LDS (row order perm: bits 2 and 3 swapped), B = Q^T in registers; register j of a
//                     lane then holds key (j & 7) + 8 h + 16 (j >> 3) of a 32-key half: the order that P^T needs below.
//   softmax           per query column in the exp2 domain; the running maximum moves only when a row grows by 2^8.
//   O^T += V^T . P^T  A = V^T, read from the row-major V tile by the LDS transpose read (ds_read_b64_tr_b16: a group of
//                     16 lanes reads 4 keys x 16 dims and each lane receives 4 keys of one dim).
// K and V tiles come by LDS-DMA as the rows lie in memory, 16-byte chunks swizzled through the source address, two
// buffers; the DMA of tile t + 1 goes out behind the barrier that opens tile t.
//
// Bound by the softmax: 32 exponentials and about 100 other vector operations per lane and tile against 16 MFMAs of 32
// cycles at head_dim 64, and by rounding up short sequences: 670 to 770 TFLOP/s at 512 and 2,048 tokens, 390 for 90 to 512
// tokens. The 16x16 form before it wrote V transposed into LDS two bytes at a time. Layers as measured: 64 sequences of 90
// to 512 tokens, 16 heads of 64: 170 -> 96 us, with deal_xcds 71; 20 sequences, 32 / 8 heads of 128: 298 -> 81 us. With queries and
// results in whole rows through LDS, where a lane's own pieces of 16 and 8 bytes lie a row's stride apart, and tile addresses from a
// scalar and a lane's fixed offset: 67 and 74 us (64 of 512 tokens, 32 / 8 heads: 382 -> 359). (The transpose read as an asm block that
// waits for its own reads alone, where the compiler waits for the next tile's DMA too: equal; the maximum over both halves by
// permlane32_swap: 1 % either way.)
#include "common.h"
#include "kernels.h"

namespace nga {

namespace {
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) s16x4* ltr_t;

constexpr float VL_LOG2E = 1.4426950408889634f;
constexpr float VL_RESCALE_LOG2 = 8.f;

// 16-byte chunk swizzles: K, distinct banks for the same chunk of 16 rows; V, for 64 bytes of 4 consecutive rows
template <int D>
__device__ __forceinline__ int vl_kswz(int row) {
  return D == 128 ? row & 15 : D == 64 ? (row >> 1) & 7 : (row >> 2) & 3;
}
template <int D>
__device__ __forceinline__ int vl_vswz(int row) {
  return D == 128 ? (row & 3) << 2 : D == 64 ? ((row >> 1) & 1) << 2 : 0;
}
}  // namespace

template <int D, bool CAUSAL, int HPW>
__global__ void __launch_bounds__(256, D == 128 ? 2 : 3) varlen_attn_kernel(PrefillParams P) {
  constexpr int KT = 64, NC = D / 8, TILE = KT * D;
  constexpr int NI = D / 32;            // DMA instructions of a wave per tile and operand
  constexpr int DS = D / 16, DT = D / 32;
  constexpr int RB = 4 / HPW, RW = 32 * RB;
  // one LDS object: [K 0 | K 1 | V 0 | V 1]
  __shared__ __attribute__((aligned(16))) uint16_t smem[4 * TILE];
  uint16_t* const kbuf = smem;
  uint16_t* const vbuf = smem + 2 * TILE;

  const int L = xcd_item(P);
  if (L >= P.total) return;
  const int G = P.Hq / P.Hkv, ngrp = P.Hq / HPW;
  const int qb = P.ntiles - 1 - L % P.ntiles;
  const int hg = (L / P.ntiles) % ngrp;
  const int b = L / (P.ntiles * ngrp);
  const int q0 = P.cu_q[b], qlen = P.cu_q[b + 1] - q0;
  if (qb * RW >= qlen) return;

  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int hq = hg * HPW + w % HPW, kvh = hq / G, rb = w / HPW;
  const int r32 = lane & 31, h = lane >> 5;
  const int row0 = qb * RW + rb * 32;                 // the wave's first query row
  const bool active = row0 < qlen;                    // wave-uniform; idle waves still fill the tiles
  const int qr = min(row0 + r32, qlen - 1);
  const int W = CAUSAL ? P.window : 0;

  // tiles of the workgroup; a wave computes those that its own rows see
  const int hi_wg = min(qlen - 1, qb * RW + RW - 1), hi_w = min(qlen - 1, row0 + 31);
  const int n_tiles = (CAUSAL ? hi_wg : qlen - 1) / KT + 1;
  const int t_first = W > 0 ? max(0, qb * RW - W + 1) / KT : 0;
  const int w_last = CAUSAL ? hi_w / KT : n_tiles - 1;

  // DMA: wave instruction i fills chunk positions [64 (NI w + i), +64) of a tile, position p holding chunk
  // (p % NC) ^ swizzle of row p / NC
  const uint32_t step = (uint32_t)P.kv_stride;
  uint32_t krow[NI], kcol[NI], vcol[NI], koff[NI], vplace[NI];   // a lane's place, to be added to the tile's address (scalar)
#pragma unroll
  for (int i = 0; i < NI; ++i) {
    const int p = (NI * w + i) * 64 + lane;
    krow[i] = p / NC;
    kcol[i] = ((p % NC) ^ vl_kswz<D>(krow[i])) * 8;
    vcol[i] = ((p % NC) ^ vl_vswz<D>(krow[i])) * 8;
    koff[i] = krow[i] * step + kcol[i];
    vplace[i] = krow[i] * step + vcol[i];
  }
  const uint16_t* const kp = P.k + (int64_t)q0 * P.kv_stride + (int64_t)kvh * D;
  const uint16_t* const vp = P.v + (int64_t)q0 * P.kv_stride + (int64_t)kvh * D;
  auto issue = [&](int t, int buf) {
    const uint32_t left = qlen - 1 - t * KT;
    const uint16_t *const kt = kp + (int64_t)t * KT * P.kv_stride, *const vt = vp + (int64_t)t * KT * P.kv_stride;
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      uint32_t a = koff[i], c = vplace[i];
      if (left < KT - 1) {   // keys past the end are masked
        a = min(krow[i], left) * step + kcol[i];
        c = min(krow[i], left) * step + vcol[i];
      }
      glds16(kt + a, kbuf + buf * TILE + (NI * w + i) * 512);
      glds16(vt + c, vbuf + buf * TILE + (NI * w + i) * 512);
    }
  };
  // A wave's 32 rows pass through its quarter of a tile buffer, that of K or V, in whole pieces: the queries through the second
  // one before its first tile comes, the results through the one whose tile everyone has read. Chunk c of row r lies at c ^ r (mod NC).
  auto rows_at = [&](int buf) { return smem + ((w >> 1) * 2 + buf) * TILE + (w & 1) * (TILE / 2); };
  constexpr int NR = D / 16;   // instructions for 32 rows
  bf16x8 qf[DS];
  {
    const uint16_t* qp = P.q + (int64_t)(q0 + row0) * P.q_stride + (int64_t)hq * D;
    if (active)
#pragma unroll
      for (int i = 0; i < NR; ++i) {
        const int p = i * 64 + lane, r = p / NC;
        glds16(qp + min(r, qlen - 1 - row0) * P.q_stride + ((p % NC) ^ (r % NC)) * 8, rows_at(1) + i * 512);
      }
  }

  const int prow = (r32 & ~12) | ((r32 & 4) << 1) | ((r32 & 8) >> 1);   // perm(r32)
  const int ksw = vl_kswz<D>(prow);                                     // of prow + 32 too
  // transpose read: lane i of a 16-lane group names key i / 4 and dims 4 (i % 4) .. of the group's 4 x 16 block
  const int tkey = 8 * h + ((lane & 15) >> 2), tdim = 16 * ((lane >> 4) & 1) + 4 * (lane & 3);
  int voff[DT];   // the swizzle of a key is that of key + 4 and key + 16
#pragma unroll
  for (int dt = 0; dt < DT; ++dt) {
    const int d = 32 * dt + tdim;
    voff[dt] = tkey * D + (((d >> 3) ^ vl_vswz<D>(tkey)) << 3) + (d & 7);
  }

  const float sl2 = P.scale * VL_LOG2E;
  float m = -INFINITY, l = 0.f;
  f32x16 o[DT];
#pragma unroll
  for (int dt = 0; dt < DT; ++dt) o[dt] = (f32x16)(0.f);

  issue(t_first, 0);
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 * NI) : "memory");
#pragma unroll
  for (int s = 0; s < DS; ++s) qf[s] = as_bf16x8(*reinterpret_cast<const u16x8*>(rows_at(1) + r32 * D + (((2 * s + h) ^ (r32 % NC)) << 3)));
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);
  for (int t = t_first; t < n_tiles; ++t) {
    const int buf = (t - t_first) & 1;
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // this wave's part of tile t is there
    __builtin_amdgcn_s_barrier();                      // everyone's is, and tile t - 1 is read
    if (t + 1 < n_tiles) issue(t + 1, buf ^ 1);
    if (!active || t > w_last) continue;
    const uint16_t* ks = kbuf + buf * TILE;
    f32x16 S[2];
#pragma unroll
    for (int h2 = 0; h2 < 2; ++h2) {
      S[h2] = (f32x16)(0.f);
#pragma unroll
      for (int s = 0; s < DS; ++s) {
        const bf16x8 a = as_bf16x8(*reinterpret_cast<const u16x8*>(ks + (32 * h2 + prow) * D + (((2 * s + h) ^ ksw) << 3)));
        S[h2] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, qf[s], S[h2], 0, 0, 0);
      }
    }
    const int kbase = t * KT;
    const bool need = CAUSAL ? (kbase + KT - 1 > row0 || (W > 0 && kbase <= hi_w - W)) : kbase + KT > qlen;
    if (need) {
      const int lo = W > 0 ? qr - W : -1, hi = CAUSAL ? qr : qlen - 1;
#pragma unroll
      for (int h2 = 0; h2 < 2; ++h2)
#pragma unroll
        for (int j = 0; j < 16; ++j) {
          const int key = kbase + 32 * h2 + 8 * h + 16 * (j >> 3) + (j & 7);
          S[h2][j] = key <= hi && key > lo ? S[h2][j] : -INFINITY;
        }
    }
    float mx = S[0][0];
#pragma unroll
    for (int j = 1; j < 32; ++j) mx = fmaxf(mx, S[j >> 4][j & 15]);
    mx = fmaxf(mx, __shfl_xor(mx, 32, 64)) * sl2;   // scale > 0
    const bool grow = mx > m + VL_RESCALE_LOG2;
    if (__ballot(grow)) {
      const float m_new = grow ? mx : m;
      const float alpha = grow ? __builtin_amdgcn_exp2f(m - m_new) : 1.f;
      m = m_new;
      l *= alpha;
#pragma unroll
      for (int dt = 0; dt < DT; ++dt) o[dt] *= alpha;
    }
    const float mo = m == -INFINITY ? 0.f : -m;   // a row may see nothing of a tile (window)
    bf16x8 pf[4];
    float ls0 = 0.f, ls1 = 0.f;
#pragma unroll
    for (int j = 0; j < 32; j += 2) {
      const float e0 = __builtin_amdgcn_exp2f(__builtin_fmaf(S[j >> 4][j & 15], sl2, mo));
      const float e1 = __builtin_amdgcn_exp2f(__builtin_fmaf(S[j >> 4][(j & 15) + 1], sl2, mo));
      ls0 += e0;
      ls1 += e1;
      pf[j >> 3][j & 7] = (__bf16)e0;
      pf[j >> 3][(j & 7) + 1] = (__bf16)e1;
    }
    l += ls0 + ls1;
    // pf[s]: keys 16 s + 8 h + 0..7 of the tile
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) {
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        uint16_t* const at = vbuf + buf * TILE + voff[dt] + 16 * s * D;
        const s16x4 va = __builtin_amdgcn_ds_read_tr16_b64_v4i16((ltr_t)at);
        const s16x4 vb = __builtin_amdgcn_ds_read_tr16_b64_v4i16((ltr_t)(at + 4 * D));
        const auto v8 = __builtin_shufflevector(va, vb, 0, 1, 2, 3, 4, 5, 6, 7);
        o[dt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, v8), pf[s], o[dt], 0, 0, 0);
      }
    }
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // no DMA may outlive the workgroup
  l += __shfl_xor(l, 32, 64);
  if (!active) return;
  const float inv = l > 0.f ? 1.f / l : 0.f;
  uint16_t* const rows = rows_at((n_tiles - t_first) & 1);
  // o[dt][j]: dim 32 dt + (j & 3) + 8 (j >> 2) + 4 h
#pragma unroll
  for (int dt = 0; dt < DT; ++dt)
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      u16x4 v;
#pragma unroll
      for (int j = 0; j < 4; ++j) v[j] = f2bf(o[dt][4 * g + j] * inv);
      *reinterpret_cast<u16x4*>(rows + r32 * D + (((4 * dt + g) ^ (r32 % NC)) << 3) + 4 * h) = v;
    }
  uint16_t* const op = P.out + (int64_t)(q0 + row0) * P.out_stride + (int64_t)hq * D;
#pragma unroll
  for (int i = 0; i < NR; ++i) {
    const int p = i * 64 + lane, r = p / NC;
    const u16x8 v = *reinterpret_cast<const u16x8*>(rows + r * D + (((p % NC) ^ (r % NC)) << 3));
    if (row0 + r < qlen) store8_any(op + r * P.out_stride + (p % NC) * 8, v);
  }
}

void launch_varlen_attention(const PrefillParams& p, int num_seqs, int max_q_len, int D, bool causal, hipStream_t stream) {
  const int hpw = (p.Hq / p.Hkv) % 4 == 0 ? 4 : 1;
  const int rw = 128 / hpw;
  PrefillParams pp = p;
  pp.ntiles = (max_q_len + rw - 1) / rw;
  const dim3 grid(deal_xcds(pp, num_seqs, pp.ntiles * (p.Hq / hpw / p.Hkv)));
#define NGA_VL(DD)                                                                                         \
  do {                                                                                                     \
    if (hpw == 4) {                                                                                        \
      if (causal) varlen_attn_kernel<DD, true, 4><<<grid, 256, 0, stream>>>(pp);                           \
      else varlen_attn_kernel<DD, false, 4><<<grid, 256, 0, stream>>>(pp);                                 \
    } else {                                                                                               \
      if (causal) varlen_attn_kernel<DD, true, 1><<<grid, 256, 0, stream>>>(pp);                           \
      else varlen_attn_kernel<DD, false, 1><<<grid, 256, 0, stream>>>(pp);                                 \
    }                                                                                                      \
  } while (0)
  if (D == 128) NGA_VL(128);
  else if (D == 64) NGA_VL(64);
  else if (D == 32) NGA_VL(32);
#undef NGA_VL
}

}  // namespace nga
