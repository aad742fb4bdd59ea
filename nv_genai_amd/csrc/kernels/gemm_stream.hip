// Decode projections of up to 16 rows: out[M, N] = x[M, K] . W[N, K]^T as one stream of the weights.
//
// Nothing but the weights' bytes counts here, and HBM gives them at full rate only in long pieces with much in flight. A wave
// therefore has a stream of its own: 16 or 32 weight rows (NT), 512 or 256 bytes of each at a time, by LDS-DMA into two private
// 8-KiB buffers, eight waves a CU, and no barrier before the end. The weight rows are the A operand of 16x16x32 MFMA, the token
// rows the B operand, from L2 straight into registers one stage ahead. The four waves of a workgroup share the rows and split K;
// they meet once in LDS, so no partial sums go through memory.
//
// Weights from HBM, us at 1 / 4 / 8 / 16 rows, the kernel that did it before and here (before: gemv.hip, then gemm_skinny.hip's
// table, the K split's sums not counted; its 128 weight rows come in pieces of 128 bytes):
//   4,096 x 4,096    9.1  8.8  9.2  9.6    7.8  7.9  8.2  9.5
//   6,144 x 4,096   10.9 11.1 11.5 12.1   10.4 10.6 10.9 12.1
//   4,096 x 14,336  25.3 22.3 22.7 23.6   21.3 21.5 22.4 26.6
//   SwiGLU 2 x 14,336 x 4,096   39.4 45.3 48.8 49.1   39.5 39.7 40.6 44.7   (235 MB: 5.3 to 5.9 TB/s)
// One wave a tile and eight waves were slower everywhere (28,672 rows: 44.8 and 44.4 us for 38.7), and so are 17 to 32 rows,
// whose tokens cost as much L2 traffic as the weights (SwiGLU above at 32 rows: 55.6, table 49.6).
#include "common.h"
#include "kernels.h"

namespace nga {

namespace {
template <int N>
__device__ __forceinline__ void st_wait_vm() {
  static_assert(N >= 0 && N < 64, "vmcnt is 6 bits");
  __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | (7 << 4) | (15 << 8));
}

__device__ __forceinline__ float st_silu(float x) { return x / (1.f + __expf(-x)); }
}  // namespace

// EPI 0: bf16 out; 1: fp32 out; 2: bf16 silu(gate) up of W = [gate | up] rows, N = F (8 NT features a tile); 3: bf16 out += product
// XP: a layer of 2 to 16 rows without launches for its norms. What adds to the residual (epi 3) leaves the rows times the next norm's
// weights, packed as the next projection's operand wants them, and the squares' sum of each row over its features; that projection's sums
// are multiplied by the rows' 1 / rms at the end. A bf16 rounding of x w for one of x w / rms, the squares in fp32 as before. 8B, us at 2 /
// 8 / 16 rows, with rows as they lie and without norms / so: q/k/v 10.5 10.9 11.8 / 11.3 11.3 11.8, output 7.0 7.2 8.1 / 7.5 7.6 8.8, SwiGLU
// 38.5 39.7 44.3 / 38.5 38.6 41.9, down 21.3 22.5 26.7 (and 22.4 in slabs) / 21.8 21.8 23.5; each of the two norms was a launch of 4.6 to 4.8.
// NJ > 0: the one row is normed first (RMSNorm, K <= 512 NJ), while the first two stages are under way. Each wave sums the row's
// squares by itself and lays the K range that it multiplies in its own part of LDS, so that none waits for another. It takes the
// place of a launch of 4.6 us (6,144 x 4,096: 10.0 us, with the norm 12.1); for two rows it costs what it saves (SwiGLU 2 x 14,336 x
// 4,096: 38.3, with the norm 43.0), since every workgroup reads them whole.
template <int NT, int EPI, int NJ, bool XP>
__global__ void __launch_bounds__(256) stream_gemm_kernel(StreamGemmParams P) {
  constexpr int NW = 4;
  constexpr int KS = 256 / NT, CPR = KS / 8, KSTEPS = KS / 32;   // k of a stage, its 16-byte chunks a row, its MFMA steps
  constexpr int XS = NW * 2 * 4096;                              // the normed row
  __shared__ __attribute__((aligned(16))) uint16_t ring[XS + 512 * NJ];
  const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int col = lane & 15, h = lane >> 4;
  const int tile = blockIdx.x;
  const int stages = P.K / KS;
  const int s0 = stages * wv / NW, s1 = stages * (wv + 1) / NW;

  // chunk c of row r lies at c ^ r (mod 16); with SwiGLU the second half of the rows are up's
  const uint16_t* wsrc[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const int r = 2 * NT * i + lane / CPR, hr = 8 * NT;
    const int64_t row = EPI == 2 ? (r < hr ? (int64_t)tile * hr + r : (int64_t)P.N + tile * hr + r - hr) : (int64_t)tile * 16 * NT + r;
    wsrc[i] = P.w + row * P.K + ((lane % CPR ^ (r & 15)) << 3);
  }
  const uint16_t* xp = XP ? P.x + (16 * h + min(col, P.M - 1)) * 8 : P.x + (int64_t)min(col, P.M - 1) * P.ldx + 8 * h;
  uint16_t* buf = ring + wv * (2 * 4096);

  auto issue = [&](int s) {
    uint16_t* b = buf + (s & 1) * 4096;
#pragma unroll
    for (int i = 0; i < 8; ++i) glds16(wsrc[i] + (int64_t)s * KS, b + i * 512);
  };
  const uint16_t* xl = ring + XS + 8 * h;
  auto load_x = [&](int s, u16x8 (&x)[KSTEPS]) {
#pragma unroll
    for (int k = 0; k < KSTEPS; ++k) x[k] = NJ ? *reinterpret_cast<const u16x8*>(xl + s * KS + 32 * k) : load8(xp + (XP ? (s * KSTEPS + k) * 512 : s * KS + 32 * k));
  };
  constexpr int XV = NJ ? 0 : KSTEPS;   // loads of token rows in flight
  f32x4 acc[NT];
#pragma unroll
  for (int i = 0; i < NT; ++i) acc[i] = (f32x4)(0.f);
  auto multiply = [&](int s, u16x8 (&x)[KSTEPS]) {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
    const uint16_t* b = buf + (s & 1) * 4096 + col * KS;
    u16x8 a[NT][KSTEPS];
#pragma unroll
    for (int k = 0; k < KSTEPS; ++k)
#pragma unroll
      for (int i = 0; i < NT; ++i) a[i][k] = *reinterpret_cast<const u16x8*>(b + i * 16 * KS + (((4 * k + h) ^ col) << 3));
#pragma unroll
    for (int k = 0; k < KSTEPS; ++k)
#pragma unroll
      for (int i = 0; i < NT; ++i) acc[i] = mfma16(as_bf16x8(a[i][k]), as_bf16x8(x[k]), acc[i]);
    __builtin_amdgcn_sched_barrier(0);   // the buffer is read before it is filled again
    asm volatile("" ::: "memory");
  };
  // ask for stage s + 1 and its rows y, wait for what was asked for before them, multiply stage s
  auto step = [&](int s, u16x8 (&x)[KSTEPS], u16x8 (&y)[KSTEPS]) {
    load_x(s + 1, y);
    __builtin_amdgcn_sched_barrier(0);
    issue(s + 1);
    __builtin_amdgcn_sched_barrier(0);
    st_wait_vm<8 + XV>();
    multiply(s, x);
  };
  // what the end needs, asked for first by the wave that adds up: the rows' squares (shared out over the waves the launch was 0.4 us
  // longer), the residual that the product is added to, the next norm's weights
  constexpr int SQ = 16;
  f32x4 sv[SQ];
  u16x4 res[NT], nw_next[NT];
  const int groups = XP ? P.n_sq >> 2 : 0;
  if (wv == 0) {
    if constexpr (XP) {
      if (P.sq != nullptr)
#pragma unroll
        for (int i = 0; i < SQ; ++i) {
          const int g = h + 4 * i;
          sv[i] = g < groups ? *reinterpret_cast<const f32x4*>(P.sq + (g * 16 + col) * 4) : (f32x4)(0.f);
        }
    }
    if constexpr (EPI == 3) {
#pragma unroll
      for (int i = 0; i < NT; ++i) {
        const int n = 16 * (NT * tile + i) + 4 * h;
        res[i] = *reinterpret_cast<const u16x4*>(reinterpret_cast<const uint16_t*>(P.out) + (int64_t)min(col, P.M - 1) * P.ldo + n);
        nw_next[i] = P.xw != nullptr ? *reinterpret_cast<const u16x4*>(P.next_w + n) : (u16x4)(0);
      }
    }
  }
  auto squares = [&]() {   // 1 / rms of row `col`
    float ss = 0.f;
#pragma unroll
    for (int i = 0; i < SQ; ++i) ss += (sv[i][0] + sv[i][1]) + (sv[i][2] + sv[i][3]);
    for (int g = h + 4 * SQ; g < groups; g += 4) {
      const f32x4 v = *reinterpret_cast<const f32x4*>(P.sq + (g * 16 + col) * 4);
      ss += (v[0] + v[1]) + (v[2] + v[3]);
    }
    ss += __shfl_xor(ss, 16, 64);
    ss += __shfl_xor(ss, 32, 64);
    return rsqrtf(ss / (float)P.K + P.eps);
  };
  float scale = 1.f;
  if (XP && s0 >= s1 && wv == 0 && P.sq != nullptr) scale = squares();   // a K of fewer stages than waves
  u16x8 xa[KSTEPS], xb[KSTEPS];
  if (s0 < s1) {
    int s = s0;
    if constexpr (NJ > 0) {
      constexpr int SJ = NJ / NW + 1;   // 512-value pieces of a wave's K range, at most
      const int k0 = s0 * KS, k1 = s1 * KS;
      u16x8 nw[SJ], xr[SJ], v[NJ];
      wave_row_load(v, P.x, P.K, lane);
#pragma unroll
      for (int j = 0; j < SJ; ++j) {
        const int k = min(k0 + 512 * j + 8 * lane, k1 - 8);
        nw[j] = load8(P.norm_w + k);
        xr[j] = load8(P.x + k);
      }
      __builtin_amdgcn_sched_barrier(0);
      issue(s0);
      if (s0 + 1 < s1) issue(s0 + 1);
      __builtin_amdgcn_sched_barrier(0);
      const float r = wave_row_rstd(v, P.K, P.eps);
#pragma unroll
      for (int j = 0; j < SJ; ++j) {
        const int k = k0 + 512 * j + 8 * lane;
        if (k < k1) lds_store8(ring + XS + k, rms_apply8(xr[j], r, nw[j]));
      }
      lds_stored();
      if (s0 + 1 < s1) {
        load_x(s0, xb);
        st_wait_vm<8>();
        multiply(s0, xb);
        s = s0 + 1;
      }
      load_x(s, xa);
    } else {
      load_x(s0, xa);
      __builtin_amdgcn_sched_barrier(0);
      issue(s0);
      __builtin_amdgcn_sched_barrier(0);
      if (XP && wv == 0 && P.sq != nullptr) scale = squares();
    }
    // the last steps apart: a branch around the loads would make the compiler wait for all of them
    for (; s + 2 < s1; s += 2) {
      step(s, xa, xb);
      step(s + 1, xb, xa);
    }
    if (s + 1 < s1) {
      step(s, xa, xb);
      st_wait_vm<0>();
      multiply(s + 1, xb);
    } else {
      st_wait_vm<0>();
      multiply(s, xa);
    }
  }

  // lane: features 4 h .. 4 h + 3 of each 16, token col; the first wave adds the four up
  float* part = reinterpret_cast<float*>(ring);
  __syncthreads();
#pragma unroll
  for (int i = 0; i < NT; ++i) *reinterpret_cast<f32x4*>(part + ((wv * NT + i) * 64 + lane) * 4) = acc[i];
  __syncthreads();
  if (wv) return;
#pragma unroll
  for (int i = 0; i < NT; ++i) {
    f32x4 v = (f32x4)(0.f);
#pragma unroll
    for (int u = 0; u < NW; ++u) v += *reinterpret_cast<const f32x4*>(part + ((u * NT + i) * 64 + lane) * 4);
    acc[i] = XP ? v * scale : v;
  }
  if constexpr (EPI == 2) {
    float up[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) up[r] = NT == 2 ? acc[NT - 1][r] : __shfl_xor(acc[0][r], 32, 64);
    if (col >= P.M || (NT == 1 && h >= 2)) return;
    u16x4 o;
#pragma unroll
    for (int r = 0; r < 4; ++r) o[r] = f2bf(st_silu(acc[0][r]) * up[r]);
    const int n = 8 * NT * tile + 4 * h;
    *reinterpret_cast<u16x4*>(reinterpret_cast<uint16_t*>(P.out) + (XP ? packed_at(col, n, P.N) : (int64_t)col * P.ldo + n)) = o;
  } else if constexpr (EPI == 3) {
#pragma unroll
    for (int i = 0; i < NT; ++i) {
      const int t = NT * tile + i, n = 16 * t + 4 * h;
      u16x4 o, y;
      float ss = 0.f;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        o[r] = f2bf(bf2f(res[i][r]) + acc[i][r]);
        const float x = bf2f(o[r]);
        y[r] = f2bf(x * bf2f(nw_next[i][r]));
        ss = __builtin_fmaf(x, x, ss);
      }
      if (col < P.M) *reinterpret_cast<u16x4*>(reinterpret_cast<uint16_t*>(P.out) + (int64_t)col * P.ldo + n) = o;
      if (P.xw == nullptr) continue;
      ss += __shfl_xor(ss, 16, 64);
      ss += __shfl_xor(ss, 32, 64);
      if (col < P.M) *reinterpret_cast<u16x4*>(P.xw + packed_at(col, n, P.N)) = y;
      if (h == 0) P.sq_out[((t >> 2) * 16 + col) * 4 + (t & 3)] = ss;
    }
  } else {
    if (col >= P.M) return;
#pragma unroll
    for (int i = 0; i < NT; ++i) {
      const int64_t at = (int64_t)col * P.ldo + 16 * (NT * tile + i) + 4 * h;
      if constexpr (EPI == 1) {
        *reinterpret_cast<f32x4*>(reinterpret_cast<float*>(P.out) + at) = acc[i];
      } else {
        u16x4 o;
#pragma unroll
        for (int r = 0; r < 4; ++r) o[r] = f2bf(acc[i][r]);
        *reinterpret_cast<u16x4*>(reinterpret_cast<uint16_t*>(P.out) + at) = o;
      }
    }
  }
}

// tiles of 16 weight rows
static int64_t st_tiles(int64_t N, bool swiglu) { return swiglu ? N / 8 : N / 16; }

// Whether this kernel is the fastest of those here for a projection (N = F with SwiGLU). Up to K = 4,096 it is for 2 to 16 rows,
// measured against what took them before over all projections of the presets with 1 to 8 ranks. gemv.hip, which splits rows of
// any count evenly over the CUs, is faster where the tiles do not come out even: for one row between 256 and 512 tiles and above
// (6,144 rows of 1,536 / 3,072: 5.5 / 8.8 us, here 5.8 / 9.5; at 256 and 512 tiles this one: 4,096 x 4,096 9.3 and 7.9, 8,192 x
// 4,096 14.0 and 13.3; up to 448 tiles of 4,096 values too: 6,144 x 4,096 10.8 and 10.7, in a decode step 10.8 and 9.9; 7,680 12.8
// and 13.2), and for two rows of SwiGLU between 512 and 768
// tiles of long rows (2 x 4,608 x 4,096: 16.9, here 18.5; of 2,048: 10.8, 10.9; 2 x 6,656 x 4,096: 22.9, 20.5). Longer rows of 16
// tokens at once keep the L2 busier than HBM: up to 256 tiles 8 rows still gain (above, and 1,280 x 8,192 at 1 / 4 / 8 rows with
// the rotation 14.8 17.9 18.1 from the table's slabs, here 13.1 14.2 15.8), beyond the others are level (8,192 x 8,192 at 4 rows:
// table 25.6, here 27.8; 10,240 x 8,192: library 35.5, here 36.7). Of the heads only 256,000 x 3,072 at 14 to 16 rows is slower
// than the library's product (278 us, here 292); 256,000 x 2,048 takes it 229, here 195.
bool stream_gemm_covers(int64_t M, int64_t N, int64_t K, bool swiglu) {
  if (M < 1 || M > 16 || K < 256 || K % 256 || N < 16 || N % 16 || N >= (int64_t(1) << 30)) return false;
  const int64_t t = st_tiles(N, swiglu);
  if (K > 4096) return t <= 256 && M <= 8;
  if (swiglu && M == 2 && K > 2048 && t > 512 && t < 768) return false;
  return M > 1 || t <= 256 || t == 512 || (!swiglu && K > 3072 && t <= 448);
}

// 32 rows a workgroup (half the token traffic) where 16 would give some CUs two workgroups and others one, or from 9 tokens on.
// 4,096 x 4,096 at 8 rows: 16 rows 8.2 us, 32 rows 9.5; 6,144 x 4,096: 12.5, 10.9; SwiGLU 14,336 x 4,096: 40.6, 42.3, at 16
// rows 49.6, 44.7
static bool st_two(int64_t M, int64_t N, int64_t t) { return t > 256 && (t < 1024 || M > 8) && N % 32 == 0; }

// The read-ahead warms the L2 of the die that runs a 16-row workgroup of this kernel; weights that others take, or that are cut into
// other pieces, would come to the wrong dies, and what is read must be there before the slowest attention workgroup ends. One row of a
// short context, a layer with / without, us: 4,096 x 4,096 (33.5 MB) 88.8 90.8, 3,072 x 3,072 55.2 56.1, 2,048 x 2,048 44.8 45.4; read ahead
// all the same, 5,120 x 5,120 111.5 107.9, 6,144 x 6,144 161.9 155.5, 8,192 x 8,192 310.5 299.5. 2 to 16 rows of 4,096: 0.3 to 0.9 less.
bool stream_gemm_reads_ahead(int64_t M, int64_t N, int64_t K) {
  return stream_gemm_covers(M, N, K, false) && !st_two(M, N, st_tiles(N, false)) && N * K <= (int64_t(1) << 24);
}

void launch_stream_gemm(const StreamGemmParams& p, int epi, hipStream_t stream) {
  const int t = (int)st_tiles(p.N, epi == 2);
  if (p.M == 0 || t == 0) return;
  const bool two = st_two(p.packed ? 1 : p.M, p.N, t);   // packed rows cost no more at 16 than at 8
#define NGA_ST(EPI, NJ)                                                                  \
  if (two) stream_gemm_kernel<2, EPI, NJ, false><<<t / 2, 256, 0, stream>>>(p);          \
  else stream_gemm_kernel<1, EPI, NJ, false><<<t, 256, 0, stream>>>(p)
#define NGA_SP(EPI)                                                                      \
  if (two) stream_gemm_kernel<2, EPI, 0, true><<<t / 2, 256, 0, stream>>>(p);            \
  else stream_gemm_kernel<1, EPI, 0, true><<<t, 256, 0, stream>>>(p)
  if (p.packed) {
    if (epi == 1) { NGA_SP(1); }
    else if (epi == 2) { NGA_SP(2); }
    else { NGA_SP(3); }
    return;
  }
  if (p.norm_w != nullptr && p.K <= 4096) {
    if (epi == 1) { NGA_ST(1, 8); }
    else { NGA_ST(2, 8); }
  } else if (p.norm_w != nullptr) {
    if (epi == 1) { NGA_ST(1, 16); }
    else { NGA_ST(2, 16); }
  } else if (epi == 0) { NGA_ST(0, 0); }
  else if (epi == 1) { NGA_ST(1, 0); }
  else if (epi == 2) { NGA_ST(2, 0); }
  else { NGA_ST(3, 0); }
#undef NGA_SP
#undef NGA_ST
}

// xw = x norm_w in bf16, packed, and the squares' sum of each row, as the epilogue above leaves them, in one group of four
__global__ void __launch_bounds__(1024) stream_open_kernel(const uint16_t* __restrict__ x, int64_t ldx, const uint16_t* __restrict__ norm_w, int H,
                                                           uint16_t* __restrict__ xw, float* __restrict__ sq) {
  __shared__ float red[16];
  const int row = blockIdx.x, c = threadIdx.x * 8;
  float ss = 0.f;
  if (c < H) {
    const u16x8 v = load8(x + row * ldx + c), w = load8(norm_w + c);
    u16x8 o;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const float a = bf2f(v[i]);
      o[i] = f2bf(a * bf2f(w[i]));
      ss = __builtin_fmaf(a, a, ss);
    }
    store8(xw + packed_at(row, c, H), o);
  }
  ss = block_sum(ss, red);
  if (threadIdx.x < 4) sq[row * 4 + threadIdx.x] = threadIdx.x ? 0.f : ss;
}

void launch_stream_open(const uint16_t* x, int64_t ldx, const uint16_t* norm_w, int M, int H, uint16_t* xw, float* sq, hipStream_t stream) {
  if (M == 0) return;
  stream_open_kernel<<<M, (H / 8 + 63) / 64 * 64, 0, stream>>>(x, ldx, norm_w, H, xw, sq);
}

}  // namespace nga
