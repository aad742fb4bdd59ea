// out[M, N] = GELU(x[M, K] . w[N, K]^T + bias) in bf16 with fp32 sums and one rounding, for many rows: an encoder's up projection.
//
// The matrix cores bound it, as gemm_kn.hip: 256 x 256 tiles, four waves of 128 x 128, a ring of four 32-deep stages of x and w filled
// by LDS-DMA, one barrier a stage, the next stage's fragments read between this one's products. A K of 1,024 is 32 stages, so what
// lies before and behind them counts: workgroups stay for all their tiles, one a CU, and ask for the next tile's stages before they
// write the sums of the last; the sums start as the bias. w is the A operand: a lane ends with four neighbouring features of a row.
// Those of one die walk blocks of eight tiles of rows by four of features, so that its L2 serves both.
//
// The product alone is no faster than the library's (K 1,024, 4,096 features: 4,096 rows 36.5 us, library 29.1; 19,264 rows 160, 155; nor
// with other features or K); the launch of bias and GELU that it saves is what it gains. Both, us, library / here, at 2,048 / 3,072 /
// 4,096 / 8,192 / 19,264 rows: K 1,024, 4,096 features 34.6 45.0 50.0 94.0 238, 37.9 40.0 43.5 80.0 190; K 768, 3,072 features 27.8 39.6
// 40.1 74.7 145, 30.7 31.5 33.6 63.0 125.
#include "gelu.h"
#include "gemm_tile.h"
#include "kernels.h"

namespace nga {

namespace {
constexpr int NT_T = 256, NT_K = 32, NT_STAGE = 2 * NT_T * NT_K, NT_NST = 4, NT_GM = 8;
}  // namespace

__global__ void __launch_bounds__(256, 1) gemm_nt_gelu_kernel(GemmNtParams p) {
  __shared__ __attribute__((aligned(16))) uint16_t smem[NT_NST * NT_STAGE];
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int col = lane & 15, h = lane >> 4, wm = w >> 1, wn = w & 1;
  const int tm = (p.M + NT_T - 1) / NT_T, tn = p.N / NT_T, tiles = tm * tn, steps = p.K / NT_K;   // >= 8
  // die c has tiles [c0, c1), its workgroups every so-manyeth of them
  const int die = blockIdx.x & 7, q8 = tiles >> 3, r8 = tiles & 7;
  const int c0 = die * q8 + min(die, r8), c1 = c0 + q8 + (die < r8 ? 1 : 0), stride = (gridDim.x - die + 7) >> 3;

  int m0, n0;
  uint32_t xo[4], wo[4];   // of this lane's 16 bytes of a stage: 64 rows a wave, chunk c of row r at c ^ (r >> 2 & 3)
  const uint16_t *xb, *wb;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int row = w * 64 + 16 * i + (lane >> 2), c = (lane & 3) ^ ((row >> 2) & 3);
    wo[i] = 2 * (uint32_t)(row * p.K + 8 * c);
  }
  u16x4 bias[8];
  auto open = [&](int tile) {   // its place, its biases, its first four stages
    const int g = tile / (NT_GM * tn), fm = g * NT_GM, gm = min(tm - fm, NT_GM), r = tile - g * NT_GM * tn;
    m0 = (fm + r % gm) * NT_T;
    n0 = r / gm * NT_T;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int row = w * 64 + 16 * i + (lane >> 2), c = (lane & 3) ^ ((row >> 2) & 3);
      xo[i] = 2 * (uint32_t)(min(row, p.M - 1 - m0) * (int)p.ldx + 8 * c);
    }
    xb = p.x + (int64_t)m0 * p.ldx;
    wb = p.w + (int64_t)n0 * p.K;
#pragma unroll
    for (int t = 0; t < 8; ++t) bias[t] = *reinterpret_cast<const u16x4*>(p.bias + n0 + wn * 128 + 16 * t + 4 * h);
  };
  auto issue_one = [&](int i, int j) {   // j-th of eight
    uint16_t* const s = smem + (i % NT_NST) * NT_STAGE + (j >> 2) * (NT_T * NT_K) + (w * 64 + 16 * (j & 3)) * NT_K;
    if (j < 4) tile_dma(xb + (int64_t)i * NT_K, xo[j & 3], s);
    else tile_dma(wb + (int64_t)i * NT_K, wo[j & 3], s);
  };
  auto issue = [&](int i) {
#pragma unroll
    for (int j = 0; j < 8; ++j) issue_one(i, j);
  };
  const int fx0 = (wm * 128 + col) * NT_K + ((h ^ ((col >> 2) & 3)) << 3);
  const int fw0 = NT_T * NT_K + (wn * 128 + col) * NT_K + ((h ^ ((col >> 2) & 3)) << 3);
  auto read_one = [&](int i, int t, bf16x8& x, bf16x8& y) {
    const uint16_t* const s = smem + (i % NT_NST) * NT_STAGE + 16 * NT_K * t;
    x = as_bf16x8(*reinterpret_cast<const u16x8*>(s + fx0));
    y = as_bf16x8(*reinterpret_cast<const u16x8*>(s + fw0));
  };
  f32x4 acc[8][8];   // [features][rows]
  bf16x8 xa[8], ya[8], xc[8], yc[8];
  // as in gemm_kn.hip: stage i + 1 has landed, every wave has read stage i, whose place stage i + 4 takes
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
  };
  auto last = [&](int i, bf16x8 (&x)[8], bf16x8 (&y)[8], bf16x8 (&nx)[8], bf16x8 (&ny)[8]) {
    if (i >= steps) return;
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
    if (i + 4 < steps) issue(i + 4);
    if (i + 1 < steps)
#pragma unroll
      for (int t = 0; t < 8; ++t) read_one(i + 1, t, nx[t], ny[t]);
#pragma unroll
    for (int t = 0; t < 8; ++t)
#pragma unroll
      for (int j = 0; j < 8; ++j) tile_mfma(acc[t][j], y[t], x[j]);
  };

  int tile = c0 + (blockIdx.x >> 3);
  if (tile >= c1) return;
  open(tile);
  issue(0);
  issue(1);
  issue(2);
  issue(3);
  while (true) {
#pragma unroll
    for (int t = 0; t < 8; ++t)
#pragma unroll
      for (int j = 0; j < 8; ++j)
#pragma unroll
        for (int e = 0; e < 4; ++e) acc[t][j][e] = bf2f(bias[t][e]);
    // 32 DMAs, and behind them the stores of the tile before: at most 24 operations left, so the first stage is there
    asm volatile("s_waitcnt vmcnt(24)\n\ts_barrier" ::: "memory");
#pragma unroll
    for (int t = 0; t < 8; ++t) read_one(0, t, xa[t], ya[t]);
    int i = 0;
    for (; i + 8 <= steps; i += 4) {
      step(i, xa, ya, xc, yc);
      step(i + 1, xc, yc, xa, ya);
      step(i + 2, xa, ya, xc, yc);
      step(i + 3, xc, yc, xa, ya);
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) {   // 4 to 7 stages
      last(i + 2 * j, xa, ya, xc, yc);
      last(i + 2 * j + 1, xc, yc, xa, ya);
    }
    // behind the last barrier no wave reads the ring any more
    const int at = n0 + wn * 128 + 4 * h;
    const int row0 = m0 + wm * 128 + col;
    tile += stride;
    const bool more = tile < c1;
    if (more) {
      open(tile);
      issue(0);
      issue(1);
      issue(2);
      issue(3);
    }
    tile_settle(acc);
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const int m = row0 + 16 * j;
      if (m >= p.M) continue;
#pragma unroll
      for (int t = 0; t < 8; ++t) {
        u16x4 v;
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = f2bf(gelu_f(acc[t][j][e]));
        *reinterpret_cast<u16x4*>(p.out + (int64_t)m * p.N + at + 16 * t) = v;
      }
    }
    if (!more) return;
  }
}

bool gemm_nt_gelu_covers(int64_t M, int64_t N, int64_t K) {
  return M >= 3072 && M < (1 << 24) && N >= 256 && N % NT_T == 0 && N < (1 << 20) && K >= 256 && K % NT_K == 0 && K < (1 << 20);
}

void launch_gemm_nt_gelu(const GemmNtParams& p, hipStream_t stream) {
  const int64_t tiles = (int64_t)((p.M + NT_T - 1) / NT_T) * (p.N / NT_T);
  if (tiles == 0) return;
  gemm_nt_gelu_kernel<<<(unsigned)(tiles < 256 ? tiles : 256), 256, 0, stream>>>(p);
}

}  // namespace nga
