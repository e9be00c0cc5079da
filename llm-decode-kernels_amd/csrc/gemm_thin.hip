// W4A16 GEMM of a few tokens (M <= 32) on gfx950: Y[M, N] = X[M, K] . dequant(W)[N, K]^T, formats, rounding and epilogues
// as gemm_w4a16.hip (each weight fp16((q - zero) * scale), exact products, fp32 sums).
//
// A short prompt reads every weight once for little arithmetic, so what counts is the bytes each CU pulls in: its share
// of the weights and the X it needs beside them. A CU sustains about 20-25 bytes per ns here however many loads are in
// flight (2, 3 or 4 chunks ahead measure the same), so the kernel spreads the weight rows over all CUs first and shares
// each staged X among as many rows as that leaves (thin_rows).
//   * A wave owns TI tiles of 16 weight rows and all tokens (MT tiles of 16) on v_mfma_f32_16x16x32_f16: weights are
//     operand A, straight from memory into the MFMA layout and dequantized in registers (lane 16 g + c holds words of
//     row c: WPL = CK / 32 consecutive words per chunk of CK k), tokens operand B, from LDS. k order: in step s lane g
//     takes word WPL g + s of the chunk, for both operands alike.
//   * RWV waves beside each other (rows) make a K group; the KG groups of a workgroup (and the workgroups of a split)
//     take consecutive runs of chunks, so that the two halves of a 128-byte line of weights are read by one wave; runs
//     differ by at most one chunk, and a shorter one ends on a chunk of zero X and zero scales (a branch around the
//     step would make the compiler drain every load in flight at the join).
//   * The group stages its X chunk in LDS (16-byte chunk q of token t at q ^ (t & 15): the 16 tokens of an operand read
//     fall in distinct banks), double-buffered, one barrier per chunk; the next chunk's loads are in flight.
//   * The groups' accumulators meet in LDS at the end and group 0 adds them in group order, so the result depends on
//     (N, K) and the token class (M <= 16, <= 32) only.
// With a workspace, rows of K >= 8192 that make few tiles split K over workgroups of 128 rows (X is then read by a
// quarter to an eighth of the chip per k range) and leave fp32 partials.
//
// us per launch at G 128, M 2 / 16 / 32, this kernel and the wide one (64 x 64 tiles, four K groups) it replaced there:
//   28672 x 4096 (SwiGLU)  22.5 24.0 27.6  before 39.4 43.6 44.3     11264 x 2048 (SwiGLU)  9.0 8.9 10.1  before 11.5 11.9 12.9
//   6144 x 4096             9.4 10.0 12.2  before 17.6 18.7 19.8     2560 x 2048             5.4 5.5  7.6  before 10.6 10.8 11.3
//   4096 x 4096             7.3  7.8 10.9  before 17.2 18.0 19.1     2048 x 5632             8.5 9.6 14.0  before 22.2 23.6 24.6
//   4096 x 14336           18.9 20.1 23.2  before 52.0 55.9 59.8     (split 8 ways, with its reduce launch)
// 33 tokens and more are left to the register-stationary kernel, which has four row tiles per staged X: with MT = 4 this
// one takes 42 us at 28672 x 4096 and M 64 against 29.
#include "common.hpp"
#include "launch.hpp"
#include "w4_common.hpp"

namespace dk {
namespace {

constexpr int kThinMaxM = 32;

typedef _Float16 h8 __attribute__((ext_vector_type(8)));
typedef float f4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

__device__ __forceinline__ f4 mfma32(h8 a, h8 b, f4 c) { return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0); }
__device__ __forceinline__ void phase_fence() { asm volatile("" ::: "memory"); }

// PD: chunks of loads in flight (register slots)
template <int TI, int MT, int RWV, int KG, int CK, int PD, int EPI>
__global__ void __launch_bounds__(kWave * RWV * KG)
gemm_w4a16_thin(const uint32_t* W, const uint32_t* SZ, const f16* X, f16* Y, int M, int N, int K, int gsh, int tiles,
                int per, int rem) {
  constexpr int GT = kWave * RWV;            // threads of a K group
  constexpr int WPL = CK / 32;               // packed words per lane and row tile per chunk
  constexpr int CH = CK / 8;                 // 16-byte chunks of a token row per chunk
  constexpr int XL = 16 * MT * CH / GT;      // 16-byte X loads per thread per chunk
  constexpr int XR = GT / CH;                // token rows per load index
  static_assert(XL >= 1 && XL * XR == 16 * MT, "X staging covers a chunk");
  __shared__ u32x4 Xs[KG][2][16 * MT][CH];
  const int t = (int)blockIdx.x % tiles, split = (int)blockIdx.x / tiles;
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int kg = wave / RWV, rw = wave % RWV;
  const int tid = (int)threadIdx.x % GT;
  const int c = lane & 15, g = lane >> 4;
  const int n0 = (t * RWV + rw) * 16 * TI;
  const int KW = K >> 3, NG = K >> gsh;
  // this part's chunks: the first `rem` of the KG x splits parts have per + 1, the others per
  const int part = split * KG + kg;
  const int lo = part * per + min(part, rem), cnt = per + (part < rem ? 1 : 0);
  const int steps = per + (rem > 0 ? 1 : 0);  // a part with fewer chunks ends on a chunk of zeros

  const uint32_t* wrow[TI];
  const uint32_t* srow[TI];
#pragma unroll
  for (int i = 0; i < TI; ++i) {
    const size_t row = (size_t)min(n0 + 16 * i + c, N - 1);
    wrow[i] = W + row * KW + lo * (CK / 8) + WPL * g;
    srow[i] = SZ + row * NG;
  }
  const int xq = tid % CH, xr = tid / CH;
  const f16* xrow[XL];
#pragma unroll
  for (int i = 0; i < XL; ++i) xrow[i] = X + (size_t)min(xr + XR * i, M - 1) * K + lo * CK + 8 * xq;

  u32x4 xv[PD][XL], wv[PD][TI][WPL / 4];
  uint32_t sv[PD][TI];
  auto fetch = [&](int j, int slot) {
    const int k = min(j, cnt - 1);
#pragma unroll
    for (int i = 0; i < XL; ++i) xv[slot][i] = *reinterpret_cast<const u32x4*>(xrow[i] + k * CK);
#pragma unroll
    for (int i = 0; i < TI; ++i) {
#pragma unroll
      for (int u = 0; u < WPL / 4; ++u)
        wv[slot][i][u] = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(wrow[i] + k * (CK / 8) + 4 * u));
      sv[slot][i] = srow[i][((lo + k) * CK + 8 * WPL * g) >> gsh];
    }
  };
  auto stage = [&](int j, int slot) {
    const u32x4 z = {0u, 0u, 0u, 0u};
#pragma unroll
    for (int i = 0; i < XL; ++i) Xs[kg][j & 1][xr + XR * i][xq ^ ((xr + XR * i) & 15)] = j < cnt ? xv[slot][i] : z;
  };
  f4 acc[TI][MT];
#pragma unroll
  for (int i = 0; i < TI; ++i) {
#pragma unroll
    for (int j = 0; j < MT; ++j) acc[i][j] = f4{0.f, 0.f, 0.f, 0.f};
  }
  const uint32_t mlo = vgpr_const(0x000F000Fu), mhi = vgpr_const(0x00F000F0u);
  auto compute = [&](int j, int slot) {
    const int buf = j & 1;
    f16x2 s2[TI], zk[TI], zs[TI];
#pragma unroll
    for (int i = 0; i < TI; ++i) {
      const f16x2 sz = as_f16x2(j < cnt ? sv[slot][i] : 0u);
      const f16 a = (f16)1024.0f + sz.y, b = (f16)64.0f + sz.y;
      s2[i] = f16x2{sz.x, sz.x};
      zk[i] = f16x2{a, a};
      zs[i] = f16x2{b, b};
    }
#pragma unroll
    for (int s = 0; s < WPL; ++s) {
      h8 b[MT];
#pragma unroll
      for (int jj = 0; jj < MT; ++jj) b[jj] = __builtin_bit_cast(h8, Xs[kg][buf][16 * jj + c][(WPL * g + s) ^ c]);
#pragma unroll
      for (int i = 0; i < TI; ++i) {
        const h8 a = __builtin_bit_cast(h8, dequant8_sz(wv[slot][i][s >> 2][s & 3], s2[i], zk[i], zs[i], mlo, mhi));
#pragma unroll
        for (int jj = 0; jj < MT; ++jj) acc[i][jj] = mfma32(a, b[jj], acc[i][jj]);
      }
    }
  };
#pragma unroll
  for (int u = 0; u < PD; ++u) {
    fetch(u, u);
    phase_fence();
  }
  stage(0, 0);
  __syncthreads();
  auto step = [&](int j, int u) {
    compute(j, u);
    phase_fence();
    stage(j + 1, (u + 1) % PD);
    phase_fence();
    fetch(j + PD, u);
    phase_fence();
    __syncthreads();
  };
  int j0 = 0;
  for (; j0 + PD <= steps; j0 += PD) {
#pragma unroll
    for (int u = 0; u < PD; ++u) step(j0 + u, u);
  }
#pragma unroll
  for (int u = 0; u + 1 < PD; ++u)
    if (j0 + u < steps) step(j0 + u, u);

  if constexpr (KG > 1) {
    static_assert((KG - 1) * RWV * TI * MT * kWave * 16 <= (int)sizeof(Xs), "reduction space");
    f4* red = reinterpret_cast<f4*>(&Xs[0][0][0][0]);
    if (kg > 0) {
#pragma unroll
      for (int i = 0; i < TI; ++i) {
#pragma unroll
        for (int j = 0; j < MT; ++j) red[((((kg - 1) * RWV + rw) * TI + i) * MT + j) * kWave + lane] = acc[i][j];
      }
    }
    __syncthreads();
    if (kg > 0) return;
#pragma unroll
    for (int q = 1; q < KG; ++q) {
#pragma unroll
      for (int i = 0; i < TI; ++i) {
#pragma unroll
        for (int j = 0; j < MT; ++j) acc[i][j] += red[((((q - 1) * RWV + rw) * TI + i) * MT + j) * kWave + lane];
      }
    }
  }
  const bool vec = (N & 3) == 0 && (reinterpret_cast<uintptr_t>(Y) & 7) == 0;
#pragma unroll
  for (int j = 0; j < MT; ++j) {
    const int m = 16 * j + c;
    if (m >= M) continue;
#pragma unroll
    for (int i = 0; i < TI; ++i) {
      const int n = n0 + 16 * i + 4 * g;
      if (n >= N) continue;
      if constexpr (EPI == 2) {
        *reinterpret_cast<f4*>(reinterpret_cast<float*>(Y) + ((size_t)split * M + m) * N + n) = acc[i][j];
        continue;
      }
      const f16 y0 = (f16)acc[i][j][0], y1 = (f16)acc[i][j][1], y2 = (f16)acc[i][j][2], y3 = (f16)acc[i][j][3];
      if constexpr (EPI == 0) {
        f16* dst = Y + (size_t)m * N + n;
        if (vec) {
          *reinterpret_cast<u32x2*>(dst) = u32x2{as_u32(f16x2{y0, y1}), as_u32(f16x2{y2, y3})};
        } else {
          const f16 yy[4] = {y0, y1, y2, y3};
#pragma unroll
          for (int v = 0; v < 4; ++v)
            if (n + v < N) dst[v] = yy[v];
        }
      } else {
        f16* dst = Y + (size_t)m * (N >> 1) + (n >> 1);
        const f16 a0 = silu_mul(y0, y1), a1 = silu_mul(y2, y3);
        if (vec) {
          *reinterpret_cast<uint32_t*>(dst) = as_u32(f16x2{a0, a1});
        } else {
          if (n + 1 < N) dst[0] = a0;
          if (n + 3 < N) dst[1] = a1;
        }
      }
    }
  }
}

// Weight rows per workgroup of the unsplit kernel: the most that still give 160 workgroups, since every workgroup reads
// all of X through its CU and the weights want every CU. us at M 16 with 128 / 64 / 32 / 16 rows: 28672 x 4096
// 23.4 28.3 33.3 43.2; 11264 x 2048 13.5 9.0 10.3 13.4; 6144 x 4096 21.5 13.8 9.9 13.0; 4096 x 4096 20.9 13.6 9.6 7.9.
// 16 rows up to one round of the CUs only: from 17 tokens on a workgroup's LDS fills a CU, and a few workgroups over 256
// take a second round (N 4992, K 1280, M 18: 12.3 us with 16 rows, 6.7 with 32; at 16 tokens and less 4 to 20% less too).
int thin_rows(int N) {
  for (int rows = 128; rows > 16; rows /= 2)
    if (N / rows >= 160) return rows;
  return N > 16 * 256 ? 32 : 16;
}

template <int TI, int MT, int RWV, int KG, int CK, int EPI>
void go(const void* packed, const void* sz, const void* x, void* y, int M, int N, int K, int log2G, int splits,
        hipStream_t st) {
  constexpr int rows = 16 * TI * RWV;
  const int tiles = (N + rows - 1) / rows, parts = KG * splits;
  hipLaunchKernelGGL((gemm_w4a16_thin<TI, MT, RWV, KG, CK, 2, EPI>), dim3(tiles * splits), dim3(kWave * RWV * KG), 0,
                     st, (const uint32_t*)packed, (const uint32_t*)sz, (const f16*)x, (f16*)y, M, N, K, log2G, tiles,
                     K / CK / parts, K / CK % parts);
}

template <int MT, int EPI>
void launch_rows(const void* packed, const void* sz, const void* x, void* y, int M, int N, int K, int log2G,
                 hipStream_t st) {
  switch (thin_rows(N)) {
    case 128:
      if (K % 256 == 0)
        go<2, MT, 4, 2, 256, EPI>(packed, sz, x, y, M, N, K, log2G, 1, st);
      else
        go<2, MT, 4, 2, 128, EPI>(packed, sz, x, y, M, N, K, log2G, 1, st);
      return;
    case 64: go<1, MT, 4, 2, 128, EPI>(packed, sz, x, y, M, N, K, log2G, 1, st); return;
    case 32: go<1, MT, 2, 4, 128, EPI>(packed, sz, x, y, M, N, K, log2G, 1, st); return;
    default: go<1, MT, 1, 8, 128, EPI>(packed, sz, x, y, M, N, K, log2G, 1, st); return;
  }
}

}  // namespace

// N K below 2^21: a tile or two per CU whatever the kernel; launch-bound on the wide kernel too, whose sums do not
// depend on the number of tokens there.
bool gemm_thin_fits(int M, int N, int K, int log2G) {
  return M <= kThinMaxM && K % 128 == 0 && K >= 1024 && log2G >= 6 && (long long)N * K >= 1 << 21;
}

// k ranges over 128-row tiles when a workspace is given: long rows (K >= 8192) of few tiles, the fewest that make 192
// workgroups while every K group keeps 3 chunks (4096 x 14336 at M 32, S 8: 23.2 us with the reduce launch against
// 28.4 unsplit; 20.1 against 19.7 at M 16, where the reader that sums the partials itself saves the launch). From 160
// workgroups of 64 rows on the unsplit kernel has its CUs (12000 x 8192 at M 32: 30.0 us, split 4 ways 36.6).
int gemm_thin_splits(int M, int N, int K, int log2G) {
  if (!gemm_thin_fits(M, N, K, log2G) || K % 256 != 0 || N % 4 != 0) return 1;
  if (K < 8192 || N / 64 >= 160) return 1;
  const int tiles = (N + 127) / 128, nk = K / 512;  // chunks per group of an unsplit workgroup
  int s = 1;
  while (s < 16 && tiles * s < 192 && nk / (2 * s) >= 3) s *= 2;
  return tiles * s >= 128 && s > 1 ? s : 1;
}

const char* gemm_thin_name(int N, int splits) {
  switch (splits > 1 ? 128 : thin_rows(N)) {
    case 128: return "thin 128";
    case 64: return "thin 64";
    case 32: return "thin 32";
    default: return "thin 16";
  }
}

void launch_gemm_thin(const void* packed, const void* sz, const void* x, void* y, int M, int N, int K, int log2G,
                      int epilogue, int splits, hipStream_t st) {
  if (splits > 1) {  // y = the partials
    if (M <= 16) return go<2, 1, 4, 2, 256, 2>(packed, sz, x, y, M, N, K, log2G, splits, st);
    return go<2, 2, 4, 2, 256, 2>(packed, sz, x, y, M, N, K, log2G, splits, st);
  }
  if (M <= 16) {
    if (epilogue == 1) return launch_rows<1, 1>(packed, sz, x, y, M, N, K, log2G, st);
    return launch_rows<1, 0>(packed, sz, x, y, M, N, K, log2G, st);
  }
  if (epilogue == 1) return launch_rows<2, 1>(packed, sz, x, y, M, N, K, log2G, st);
  launch_rows<2, 0>(packed, sz, x, y, M, N, K, log2G, st);
}

}  // namespace dk
