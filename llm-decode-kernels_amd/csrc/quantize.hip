// INT4 format producer on gfx950: round-to-nearest asymmetric group quantization + nibble packing, bit-identical to
// the reference's runtime/quant.py (group_params RTN branch :20-28, quantize :42-48, pack :100-109,
// pack_scale_zero :122-124):
//     scale = fp16(max((max - min) / 15, 1e-6))        (fp32 arithmetic, read back as fp32)
//     zero  = clamp(rint(-min / scale), 0, 15)
//     q     = clamp(rint(w / scale) + zero, 0, 15)
// rint is round-half-to-even and the divisions are IEEE-correctly rounded, matching torch's fp32 ops.
//
// With clip (group_params clip=True, runtime/quant.py:17-38) the range [min, max] is first shrunk by the factor of
// CLIP_GRID = (1.0, 0.95, ..., 0.7) whose (scale, zero) give the smallest squared rounding error of the group: for each
// factor a (fp32, as torch multiplies an fp32 tensor by a Python float) mn = min * a, mx = max * a, the scale and zero
// above, and err = sum((clamp(rint(w / scale) + zero, 0, 15) - zero) * scale - w)^2 over the group, each term in fp32
// exactly as the reference computes it. The terms are summed in fp64, so the choice (the first factor with the
// smallest error, the reference's strict `err < best`) is the argmin of the reference's fp32 terms up to fp64 rounding: the
// eight terms of a word in order, then the words of the group pairwise, the farthest lanes first. The reference sums them
// in fp32, so the two can pick different factors only where two errors agree to fp32 summation noise.
//
// One lane per packed word (8 weights, one 16-byte load), 1 or 4 words per thread (kManyWords); the G/8 lanes of a group are
// consecutive in one wave (G <= 512) and reduce min / max (and the clip errors) by DPP within 16 lanes, by shuffles
// beyond. Rows are whole groups, so words and groups are numbered through the matrix and no row is ever computed.
// Bound: the 2.5 bytes per weight. Before, the row's 64-bit division, ten IEEE divisions per word and eight LDS
// shuffles kept the vector ALUs busy for longer than that: 4096 x 14336 G 128 45.8 us (3.2 TB/s) against 33.3 now (4.5),
// with clip 280 against 167 (seven times the rounding per weight: vector ALUs).
#include "common.hpp"
#include "launch.hpp"

namespace dk {
namespace {

// torch.clamp semantics: a value equal to a bound (in particular -0.0 against a bound of +0.0) and NaN pass through
// unchanged. fminf / fmaxf would return +0.0 for (-0.0, +0.0) and drop NaN.
__device__ __forceinline__ float clamp_keep_sign(float v, float lo, float hi) {
  return v < lo ? lo : (v > hi ? hi : v);
}

constexpr float kClipGrid[7] = {1.0f, 0.95f, 0.9f, 0.85f, 0.8f, 0.75f, 0.7f};

// (scale, zero) of a [lo, hi] range: scale = fp16(max((hi - lo) / 15, 1e-6)) read back as fp32, zero =
// clamp(rint(-lo / scale), 0, 15) (a group whose minimum is 0 or a tiny positive value gives -0.0, which the
// reference's clamp keeps).
__device__ __forceinline__ void range_params(float lo, float hi, f16& scale16, float& scale, float& zero) {
  const float step = clamp_keep_sign((hi - lo) / 15.0f, 1e-6f, INFINITY);
  scale16 = (f16)step;
  scale = (float)scale16;
  zero = clamp_keep_sign(rintf(-lo / scale), 0.0f, 15.0f);
}

// v / s for the rounding rint(v / s), v and s fp16 values in fp32, s > 0 finite: the quotient's reciprocal estimate
// with one residual step. A quotient near a tie k + 1/2 (k < 32) is either the tie itself, which the residual step
// returns exactly (the residual v - q s is exact and its correction rounds to the representable quotient), or at least
// 2^-12 away from it (2 v - (2 k + 1) s is a whole number of units of the two 11-bit significands), while the estimate is
// within 2^-17: rint gives what it gives for the correctly rounded division.
__device__ __forceinline__ float quot(float v, float s, float rs) {
  const float q = v * rs;
  return fmaf(fmaf(-q, s, v), rs, q);
}

// clamp(rint(quotient) + zero, 0, 15) as a finite whole number (0 for NaN, as the integer conversion gives)
__device__ __forceinline__ float code(float quotient, float zero) {
  return __builtin_amdgcn_fmed3f(rintf(quotient) + zero, 0.0f, 15.0f);
}

// the value of lane ^ O (O a power of two): DPP within 16 lanes, a shuffle beyond. Lane ^ 4 is lane ^ 7 (row_half_mirror)
// of lane ^ 3 (quad_perm).
template <int O>
__device__ __forceinline__ float partner(float v) {
  if constexpr (O == 1) {
    return DK_DPP_F32(v, 0xB1, 0xF);   // quad_perm [1,0,3,2]
  } else if constexpr (O == 2) {
    return DK_DPP_F32(v, 0x4E, 0xF);   // quad_perm [2,3,0,1]
  } else if constexpr (O == 4) {
    const float t = DK_DPP_F32(v, 0x1B, 0xF);  // quad_perm [3,2,1,0]
    return DK_DPP_F32(t, 0x141, 0xF);
  } else if constexpr (O == 8) {
    return DK_DPP_F32(v, 0x128, 0xF);  // row_ror:8
  } else {
    return __shfl_xor(v, O, kWave);
  }
}
template <int O>
__device__ __forceinline__ double partner(double v) {
  const uint64_t b = __builtin_bit_cast(uint64_t, v);
  const float lo = partner<O>(__builtin_bit_cast(float, (uint32_t)b));
  const float hi = partner<O>(__builtin_bit_cast(float, (uint32_t)(b >> 32)));
  return __builtin_bit_cast(double, (uint64_t)__builtin_bit_cast(uint32_t, hi) << 32 | __builtin_bit_cast(uint32_t, lo));
}
// over the WPG lanes of a group, from the nearest partner to the farthest: when lane ^ 4 is due the lanes of a quad hold the
// same values, so lane ^ 7 serves (one instruction less: 1% of 4096 x 14336 without clip)
template <int WPG, int O = 1>
__device__ __forceinline__ void group_range(float& lo, float& hi) {
  if constexpr (O < WPG) {
    lo = fminf(lo, O == 4 ? DK_DPP_F32(lo, 0x141, 0xF) : partner<O>(lo));
    hi = fmaxf(hi, O == 4 ? DK_DPP_F32(hi, 0x141, 0xF) : partner<O>(hi));
    group_range<WPG, 2 * O>(lo, hi);
  }
}
// the same over sums, whose rounding depends on the order: from the farthest partner to the nearest
template <int WPG>
__device__ __forceinline__ void group_total(double& e) {
  if constexpr (WPG > 1) {
    e += partner<WPG / 2>(e);
    group_total<WPG / 2>(e);
  }
}

constexpr int kQuantThreads = 256;

template <int WPG, bool CLIP, int WPT>  // words (lanes) per group; range clipping; words per thread
__global__ void __launch_bounds__(kQuantThreads)
quantize_w4_kernel(const f16* __restrict__ w, uint32_t* __restrict__ packed, uint32_t* __restrict__ sz, long long words) {
  const long long base = (long long)blockIdx.x * (kQuantThreads * WPT) + threadIdx.x;
  u32x4 raw[WPT];
#pragma unroll
  for (int i = 0; i < WPT; ++i)  // dead tail lanes (whole dead groups: words % WPG == 0) re-read the last word
    raw[i] = load_stream(reinterpret_cast<const u32x4*>(w) + min(base + i * kQuantThreads, words - 1));
#pragma unroll
  for (int i = 0; i < WPT; ++i) {
    const long long gid = base + i * kQuantThreads;
    float v[8];
    unpack8(raw[i], v);
    f16x2 lo2 = as_f16x2(raw[i][0]), hi2 = lo2;
#pragma unroll
    for (int e = 1; e < 4; ++e) {
      lo2 = __builtin_elementwise_min(lo2, as_f16x2(raw[i][e]));
      hi2 = __builtin_elementwise_max(hi2, as_f16x2(raw[i][e]));
    }
    float lo = fminf((float)lo2.x, (float)lo2.y), hi = fmaxf((float)hi2.x, (float)hi2.y);
    group_range<WPG>(lo, hi);
    f16 scale16;
    float scale, zero;
    range_params(lo, hi, scale16, scale, zero);
    const bool fin = scale < INFINITY;  // an infinite weight in the group: plain divisions
    if constexpr (CLIP) {
      double best = 0.0;
#pragma unroll 1
      for (int c = 0; c < 7; ++c) {
        f16 s16;
        float sc, ze;
        range_params(lo * kClipGrid[c], hi * kClipGrid[c], s16, sc, ze);
        const float rs = __builtin_amdgcn_rcpf(sc);
        double err = 0.0;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const float c15 = fin ? code(quot(v[e], sc, rs), ze) : clamp_keep_sign(rintf(v[e] / sc) + ze, 0.0f, 15.0f);
          const float d = (c15 - ze) * sc - v[e];
          err += (double)(d * d);
        }
        group_total<WPG>(err);
        if (c == 0 || err < best) {
          best = err;
          scale16 = s16;
          scale = sc;
          zero = ze;
        }
      }
    }
    const float rs = __builtin_amdgcn_rcpf(scale);
    // the word's halves as exact fp32 sums of their four nibbles (elements 0, 2, 4, 6 and 1, 3, 5, 7)
    float half[2];
#pragma unroll
    for (int o = 0; o < 2; ++o) {
      half[o] = code(quot(v[6 + o], scale, rs), zero);
#pragma unroll
      for (int e = 4; e >= 0; e -= 2) half[o] = fmaf(half[o], 16.0f, code(quot(v[e + o], scale, rs), zero));
    }
    uint32_t word = (uint32_t)half[0] | (uint32_t)half[1] << 16;
    if (!fin) {
      asm volatile("");  // stays a branch
      word = 0;
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const float qf = clamp_keep_sign(rintf(v[e] / scale) + zero, 0.0f, 15.0f);
        word |= (uint32_t)qf << (4 * (e >> 1) + 16 * (e & 1));
      }
    }
    if (gid < words) {
      packed[gid] = word;
      if ((threadIdx.x & (WPG - 1)) == 0) sz[gid / WPG] = as_u32(f16x2{scale16, (f16)zero});
    }
  }
}

// Words per thread: a thread works through its words one after the other, so where the waves are few the chain of four is
// the kernel's time; over many rounds of waves four loads in flight per thread are a little better. us at G 128 with 1 / 4
// words (clip: 1 / 4): 256 x 1024 2.8 / 3.6 (6.0 / 18.2), 1024 x 4096 4.5 / 4.8 (15.7 / 21.5), 4096 x 4096 11.9 / 11.9 (51.5 /
// 54.7), 4096 x 14336 33.5 / 33.7 (167 / 166), 16384 x 14336 125 / 119 (648 / 628).
constexpr long long kManyWords = 1 << 22;

template <bool CLIP, int WPT>
void launch_quantize(const void* w, void* packed, void* sz, int N, int K, int log2G, hipStream_t st) {
  const long long words = (long long)N * (K >> 3);
  const int per = kQuantThreads * WPT;
  const dim3 grid((unsigned)((words + per - 1) / per)), block(kQuantThreads);
  const f16* wp = (const f16*)w;
  uint32_t* pp = (uint32_t*)packed;
  uint32_t* sp = (uint32_t*)sz;
  switch (log2G) {
    case 5: hipLaunchKernelGGL((quantize_w4_kernel<4, CLIP, WPT>), grid, block, 0, st, wp, pp, sp, words); break;
    case 6: hipLaunchKernelGGL((quantize_w4_kernel<8, CLIP, WPT>), grid, block, 0, st, wp, pp, sp, words); break;
    case 7: hipLaunchKernelGGL((quantize_w4_kernel<16, CLIP, WPT>), grid, block, 0, st, wp, pp, sp, words); break;
    case 8: hipLaunchKernelGGL((quantize_w4_kernel<32, CLIP, WPT>), grid, block, 0, st, wp, pp, sp, words); break;
    default: hipLaunchKernelGGL((quantize_w4_kernel<64, CLIP, WPT>), grid, block, 0, st, wp, pp, sp, words); break;
  }
}

}  // namespace

void launch_quantize_w4(const void* w, void* packed, void* sz, int N, int K, int log2G, int clip, hipStream_t st) {
  if ((long long)N * (K >> 3) > kManyWords) {
    if (clip) return launch_quantize<true, 4>(w, packed, sz, N, K, log2G, st);
    return launch_quantize<false, 4>(w, packed, sz, N, K, log2G, st);
  }
  if (clip) return launch_quantize<true, 1>(w, packed, sz, N, K, log2G, st);
  launch_quantize<false, 1>(w, packed, sz, N, K, log2G, st);
}

}  // namespace dk
