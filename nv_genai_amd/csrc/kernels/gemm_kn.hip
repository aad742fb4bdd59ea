// out[M, N] = x[M, K] . w[K, N] in bf16 with fp32 sums: the gradient of a frozen projection's inputs, dy . W with W as it lies.
//
// A decoder's rows of one micro-batch give few output tiles (1,024 x 4,096: 64 of 256 x 256) and a long K (28,672 behind gate and
// up), so K is split over the chip, the slices' fp32 sums are added up by splitk_reduce_kernel, and the workgroups of a die share
// one slice's rows of W. The matrix cores bound it: a workgroup of four waves, 128 x 128 of the tile each (the least LDS traffic a
// product: 64 KiB read for 32 KiB brought in), a ring of four 32-deep stages of x and w filled by LDS-DMA, one barrier a stage; the
// fragments of the next stage are read between this stage's products, so these wait for nothing. w is transposed by the LDS
// transpose read (a group of 16 lanes reads 4 k x 16 n and each lane receives 4 k of one n); it is the A operand, so that a lane
// ends with four neighbouring columns of one row. M 1,024, N 4,096, K 28,672: 192 us, 1,250 TFLOP/s with the sum of the slabs (library
// 348); K 128,256: 785 us, 1,370 (1,442). More in ops.gemm_kn_covers.
//
// XT: x lies as [K, M], for the gradient of a weight, dy^T . x: rows of the micro-batch are the long K then, both operands are read
// transposed. K of any size from 256 on: the last stage is the last 32 rows, of which the ones that were there before count as zero. 10,240 rows:
// 4,096 x 1,024 84 us (library 105), 1,024 x 1,024 39 (66). More in ops.weight_grad_covers.
#include <algorithm>

#include "gemm_tile.h"
#include "kernels.h"

namespace nga {

namespace {
typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) s16x4* ltr_t;
constexpr int KN_T = 256, KN_K = 32, KN_STAGE = 2 * KN_T * KN_K, KN_NST = 4;   // tile, depth, elements and count of stages

// w's stage: 16-column unit u of row k lies at u ^ kn_swz(k): the eight rows that are read together lie in different banks
__device__ __forceinline__ int kn_swz(int k) { return (k & 3) | (((k >> 3) & 1) << 2); }
}  // namespace

template <bool SLABS, bool XT>
__global__ void __launch_bounds__(256, 1) gemm_kn_kernel(GemmKnParams p) {
  __shared__ __attribute__((aligned(16))) uint16_t smem[KN_NST * KN_STAGE];
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int col = lane & 15, h = lane >> 4, wm = w >> 1, wn = w & 1;
  // workgroups of one die (every eighth) take neighbouring tiles of one slice
  const int nb = gridDim.x, id = nb % 8 == 0 ? (blockIdx.x & 7) * (nb >> 3) + (blockIdx.x >> 3) : blockIdx.x;
  const int tm = (p.M + KN_T - 1) / KN_T, per = tm * (p.N / KN_T), sl = id / per, r = id - sl * per;
  const int m0 = (r % tm) * KN_T, n0 = (r / tm) * KN_T;
  const int all = (p.K + KN_K - 1) / KN_K, i0 = (int)((int64_t)all * sl / p.split), steps = (int)((int64_t)all * (sl + 1) / p.split) - i0;   // >= 8

  // this wave's part of a stage: 64 rows of x, 4 chunks of 8 each (chunk c of row r at c ^ (r >> 2 & 3)); 8 rows of w
  uint32_t xo[4], wo[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int row = w * 64 + 16 * i + (lane >> 2), c = (lane & 3) ^ ((row >> 2) & 3);
    const int k = w * 8 + 2 * i + (lane >> 5), pos = lane & 31, at = (((pos >> 1) ^ kn_swz(k)) << 4) + ((pos & 1) << 3);
    xo[i] = 2 * (uint32_t)(XT ? k * (int)p.ldx + at : min(row, p.M - 1 - m0) * (int)p.ldx + 8 * c);
    wo[i] = 2 * (uint32_t)(k * p.N + at);
  }
  const uint16_t* const xb = p.x + (XT ? m0 : (int64_t)m0 * p.ldx);
  const uint16_t* const wb = p.w + n0;
  auto issue_one = [&](int i, int j) {   // j-th of eight
    uint16_t* const s = smem + (i % KN_NST) * KN_STAGE;
    const int k = min((i0 + i) * KN_K, p.K - KN_K);
    if (j < 4) tile_dma(xb + (XT ? k * p.ldx : k), xo[j & 3], s + (XT ? (w * 8 + 2 * j) * KN_T : (w * 64 + 16 * j) * KN_K));
    else tile_dma(wb + (int64_t)k * p.N, wo[j & 3], s + KN_T * KN_K + (w * 8 + 2 * (j - 4)) * KN_T);
  };
  auto issue = [&](int i) {
#pragma unroll
    for (int j = 0; j < 8; ++j) issue_one(i, j);
  };
  // a lane's fragments in a stage: 8 k of a row of x (16 j rows on for the j-th), of a column of w
  const int fx0 = (wm * 128 + col) * KN_K + ((h ^ ((col >> 2) & 3)) << 3);
  const int kr = 8 * h + (col >> 2);
  int fw0[8], fxt[8];
#pragma unroll
  for (int t = 0; t < 8; ++t) {
    fw0[t] = KN_T * KN_K + kr * KN_T + (((wn * 8 + t) ^ kn_swz(kr)) << 4) + 4 * (col & 3);
    fxt[t] = kr * KN_T + (((wm * 8 + t) ^ kn_swz(kr)) << 4) + 4 * (col & 3);
  }
  auto transposed = [&](uint16_t* s) {   // four rows on the swizzle is the same
    const s16x4 a = __builtin_amdgcn_ds_read_tr16_b64_v4i16((ltr_t)s);
    const s16x4 b = __builtin_amdgcn_ds_read_tr16_b64_v4i16((ltr_t)(s + 4 * KN_T));
    return __builtin_bit_cast(bf16x8, __builtin_shufflevector(a, b, 0, 1, 2, 3, 4, 5, 6, 7));
  };
  auto read_one = [&](int i, int t, bf16x8& x, bf16x8& y) {   // t-th of eight of each
    uint16_t* const s = smem + (i % KN_NST) * KN_STAGE;
    if constexpr (XT) x = transposed(s + fxt[t]);
    else x = as_bf16x8(*reinterpret_cast<const u16x8*>(s + fx0 + 16 * KN_K * t));
    y = transposed(s + fw0[t]);
  };
  auto read = [&](int i, bf16x8 (&x)[8], bf16x8 (&y)[8]) {
#pragma unroll
    for (int t = 0; t < 8; ++t) read_one(i, t, x[t], y[t]);
  };
  const int again = all * KN_K - p.K;   // rows of the last stage that the one before it has
  f32x4 acc[8][8];   // [columns][rows]
#pragma unroll
  for (int t = 0; t < 8; ++t)
#pragma unroll
    for (int j = 0; j < 8; ++j) acc[t][j] = (f32x4)(0.f);
  auto multiply = [&](bf16x8 (&x)[8], bf16x8 (&y)[8]) {
#pragma unroll
    for (int t = 0; t < 8; ++t)
#pragma unroll
      for (int j = 0; j < 8; ++j) tile_mfma(acc[t][j], y[t], x[j]);
  };

  bf16x8 xa[8], ya[8], xc[8], yc[8];
  issue(0);
  issue(1);
  issue(2);
  issue(3);
  asm volatile("s_waitcnt vmcnt(24)\n\ts_barrier" ::: "memory");
  read(0, xa, ya);
  // stage i, whose fragments x, y are in registers: stage i + 1 has landed (two younger ones of 8 DMAs may be under way), every
  // wave has read stage i, whose place stage i + 4 takes
  auto step = [&](int i, bf16x8 (&x)[8], bf16x8 (&y)[8], bf16x8 (&nx)[8], bf16x8 (&ny)[8]) {
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("s_waitcnt vmcnt(16) lgkmcnt(0)\n\ts_barrier" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int t = 0; t < 8; ++t) {   // between two products there is time for another instruction
#pragma unroll
      for (int j = 0; j < 4; ++j) tile_mfma(acc[t][j], y[t], x[j]);
      __builtin_amdgcn_sched_barrier(0);
      issue_one(i + 4, t);
      read_one(i + 1, t, nx[t], ny[t]);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int j = 4; j < 8; ++j) tile_mfma(acc[t][j], y[t], x[j]);
      __builtin_amdgcn_sched_barrier(0);
    }
    __builtin_amdgcn_sched_barrier(0);
  };
  auto last = [&](int i, bf16x8 (&x)[8], bf16x8 (&y)[8], bf16x8 (&nx)[8], bf16x8 (&ny)[8]) {
    if (i >= steps) return;
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
    if (i + 4 < steps) issue(i + 4);
    if (i + 1 < steps) {
      read(i + 1, nx, ny);
      if (XT && again > 0 && i0 + i + 1 == all - 1) {
#pragma unroll
        for (int t = 0; t < 8; ++t)
#pragma unroll
          for (int e = 0; e < 8; ++e) {
            nx[t][e] = 8 * h + e >= again ? nx[t][e] : (__bf16)0.f;
            ny[t][e] = 8 * h + e >= again ? ny[t][e] : (__bf16)0.f;
          }
      }
    }
    multiply(x, y);
  };
  int i = 0;
  for (; i + 8 <= steps; i += 4) {   // i is a multiple of 4: the stages' places are constants
    step(0 + i, xa, ya, xc, yc);
    step(1 + i, xc, yc, xa, ya);
    step(2 + i, xa, ya, xc, yc);
    step(3 + i, xc, yc, xa, ya);
  }
#pragma unroll
  for (int j = 0; j < 4; ++j) {   // 4 to 7 stages
    last(i + 2 * j, xa, ya, xc, yc);
    last(i + 2 * j + 1, xc, yc, xa, ya);
  }

  tile_settle(acc);
  const int64_t at = (int64_t)sl * p.M * p.N + n0 + wn * 128 + 4 * h;
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    const int m = m0 + wm * 128 + 16 * j + col;
    if (m >= p.M) continue;
#pragma unroll
    for (int t = 0; t < 8; ++t) {
      const int64_t o = at + (int64_t)m * p.N + 16 * t;
      if constexpr (SLABS) {
        *reinterpret_cast<f32x4*>(static_cast<float*>(p.out) + o) = acc[t][j];
      } else {
        u16x4 v;
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = f2bf(acc[t][j][e]);
        *reinterpret_cast<u16x4*>(static_cast<uint16_t*>(p.out) + o) = v;
      }
    }
  }
}

// slices of K: as many as the tiles leave CUs for, of eight stages at least, at most 16
int gemm_kn_split(int64_t M, int64_t N, int64_t K) {
  const int64_t tiles = (M + KN_T - 1) / KN_T * (N / KN_T);
  if (tiles < 1) return 1;
  const int64_t s = 256 / tiles, most = (K + KN_K - 1) / KN_K / 8;
  return (int)std::max<int64_t>(1, std::min<int64_t>(std::min<int64_t>(s, 16), most));
}

void launch_gemm_kn(const GemmKnParams& p, bool xt, hipStream_t stream) {
  const int blocks = (p.M + KN_T - 1) / KN_T * (p.N / KN_T) * p.split;
  if (blocks == 0) return;
  if (xt) {
    if (p.split > 1) gemm_kn_kernel<true, true><<<blocks, 256, 0, stream>>>(p);
    else gemm_kn_kernel<false, true><<<blocks, 256, 0, stream>>>(p);
  } else {
    if (p.split > 1) gemm_kn_kernel<true, false><<<blocks, 256, 0, stream>>>(p);
    else gemm_kn_kernel<false, false><<<blocks, 256, 0, stream>>>(p);
  }
}

}  // namespace nga
