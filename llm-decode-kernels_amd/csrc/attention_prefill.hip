// Prefill attention on gfx950: causal attention of M prompt rows (row m at position pos + m) over the paged cache,
// which already holds their K / V.
//
// A workgroup owns one kv head and CW waves' worth of columns: a column is a (row, query head) pair, a wave has the 32
// columns of its 32 / HPG rows x HPG heads, so every column does work at any GQA ratio. KVS groups of CW waves share
// the columns and split the tokens: group h takes the blocks of BT tokens b with b % KVS == h. K / V stream through LDS
// in rounds of KVS blocks (double-buffered; the next round's loads are in flight in registers during the current
// round's MFMAs), one block per group, read there by the group's waves.
//
// Per block, on v_mfma_f32_32x32x16_f16 (32 columns per wave: half the LDS bytes per MFMA of the 16 x 16 form, at that
// form's full rate):
//   * S^T = K . Q^T: A = 32 token rows of K from LDS, B = the wave's Q columns (registers). The accumulator leaves lane
//     (h, r) with column r, tokens 8 q + 4 h + v of the 32: a column's scores, its running maximum, its sum and its
//     output all live in the lane pair (r, r + 32), so the softmax needs one exchange per block and the output's
//     rescale factor is the lane's own.
//   * online softmax in the log2 domain (the scale and log2 e in one multiplier). The reference maximum of a column
//     moves only when a block's maximum passes it by more than kLazy (2^8); until then neither the accumulators nor the
//     sum need rescaling. p = 2^(s - ref + kLift), at most 2^15: fp16 holds it, and what its two fp16 parts round away
//     (2^-25 at most, below 2^-14 a fixed amount) is 2^-32 or less of the largest weight. Each column decides
//     for itself (the wave only skips the code when none of its columns moves), so a row's result does not depend on
//     the rows it shares a wave with. Blocks wholly visible to the wave skip the causal mask.
//   * O^T += V^T . P^T with p as fp16 hi + lo parts, both rounded to nearest (22 bits, no bias: the sum of the weights
//     is taken from the unsplit p, so a truncated p lowers every output): the score accumulator is the B operand as it is
//     (k slot e of half h in step s is token 16 s + 8 (e / 4) + 4 h + e % 4, for both operands), and the V^T operand
//     comes out of the row-major V tile through the transposing LDS read (ds_read_b64_tr_b16: 4 tokens x 16 dims per 16
//     lanes, lane i receiving dim i).
//
// LDS: rows of 2 D bytes without padding. K chunk q (16 bytes) of row t at q ^ (t & 15) (D 128) or q ^ ((t >> 1) & 7)
// (D 64), so that 8 consecutive rows' reads of one chunk fall in distinct banks; V in 64-byte units, unit u of row t at
// u ^ (t & 3) (D 128) or u ^ ((t >> 1) & 1) (D 64), so that the 4 rows x 64 bytes of a transposing read do.
//
// The groups' states (reference maximum, sum, accumulator per column) meet in LDS at the end and group 0 merges them in
// group order. Every column's tokens go to the same group in the same order whatever workgroup or batch its row is in,
// and a block wholly past a column's bound changes nothing for it, so a row's result does not depend on how the prompt
// is batched for a given (KVS, BT); the launch's choice depends on the grid (launch_prefill).
#include <type_traits>

#include "common.hpp"
#include "launch.hpp"
#include "attn_common.hpp"

namespace dk {
namespace {

// Reference maximum of a column that has seen no token yet: a finite stand-in for -infinity, so that 2^(old - new) and
// 2^(score - ref) never meet -inf - (-inf).
constexpr float kPfNoMax = -1e30f;
constexpr float kLazy = 8.0f;  // log2 units
constexpr float kLift = 7.0f;  // p's exponent at the reference maximum
static_assert(kLazy + kLift <= 15.0f, "p fits fp16");

typedef _Float16 h8 __attribute__((ext_vector_type(8)));
typedef _Float16 h2 __attribute__((ext_vector_type(2)));
typedef float f2 __attribute__((ext_vector_type(2)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef short s16x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ f32x16 mfma32x32(h8 a, h8 b, f32x16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
}

// Keeps loads where they are written (no sinking to their first use).
__device__ __forceinline__ void pf_fence() { asm volatile("" ::: "memory"); }

// Transposing LDS read of 4 x 16-bit per lane.
__device__ __forceinline__ u32x2 read_tr(const uint8_t* p) {
  typedef __attribute__((address_space(3))) s16x4* lds_s16x4;
  return __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4)(p)));
}

// p - (float)(low / high half of an fp16 pair), one instruction each (the compiler converts and subtracts)
__device__ __forceinline__ float minus_lo(float p, uint32_t pair) {
  float r;
  asm("v_fma_mix_f32 %0, %1, -1.0, %2 op_sel_hi:[1,0,0]" : "=v"(r) : "v"(pair), "v"(p));
  return r;
}
__device__ __forceinline__ float minus_hi(float p, uint32_t pair) {
  float r;
  asm("v_fma_mix_f32 %0, %1, -1.0, %2 op_sel:[1,0,0] op_sel_hi:[1,0,0]" : "=v"(r) : "v"(pair), "v"(p));
  return r;
}

template <int D, int CW, int KVS, int BT, bool UP>
__global__ void __launch_bounds__(CW * KVS * kWave, 2)
attn_prefill_kernel(const f16* __restrict__ qkv, const int32_t* __restrict__ pos_ptr, const int32_t* __restrict__ bt,
                    int n_bt, const f16* kc, const f16* vc, int n_pages, int log2P, int n_q, int n_kv, int lhpg, int M,
                    int ctx_cap, int fold, float c2, f16* __restrict__ out) {
  // (kc, vc without __restrict__: the fences must order their loads)
  constexpr int NTH = CW * KVS * kWave;      // threads
  constexpr int CH = D / 8;                  // 16-byte chunks per K / V row
  constexpr int RB = 2 * D;                  // bytes per row
  constexpr int SB = BT * KVS;               // tokens per round (one block per group)
  constexpr int LPT = SB * CH / NTH;         // 16-byte K (and V) loads per thread per round
  constexpr int RPI = NTH / CH;              // token rows covered per load index
  constexpr int NT = BT / 32, DT = D / 32;   // 32-token score tiles per block, 32-dim output tiles
  constexpr int KS = D / 16;                 // k steps of the scores
  static_assert(LPT * RPI == SB && RPI % 16 == 0, "staging covers a round");
  constexpr int kTile = SB * RB;             // bytes of one K (or V) buffer
  __shared__ __align__(16) uint8_t lds[4 * kTile];  // K buffers 0, 1, then V buffers 0, 1

  const int kvh = blockIdx.x;
  // the rows with the longest contexts first; a grid that is resident at once (fold) pairs them with the shortest
  const int rb = (int)gridDim.y, y = (int)blockIdx.y;
  const int qb = fold && 2 * y >= rb ? y - (rb + 1) / 2 : rb - 1 - y;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int grp = wave / CW, gw = wave % CW;  // group, and the wave's columns within it
  const int r = lane & 31, h = lane >> 5;
  const int P = 1 << log2P;
  const int pos0 = *pos_ptr;
  // this lane's query column: prompt row m, head hd; tokens t <= lim are attended. Columns past the last row repeat it.
  const int rpw = 32 >> lhpg;                            // rows per wave
  const int mw = (qb * CW + gw) * rpw;                   // the wave's first row
  const int mcol = mw + (r >> lhpg);
  const int m = min(mcol, M - 1);
  const int hd = (kvh << lhpg) + (r & ((1 << lhpg) - 1));
  const int lim = (int)max(-1LL, min((long long)pos0 + m, (long long)ctx_cap - 1));  // the cap bounds mask and loads
  // every column of the wave sees tokens [0, lim_w] (its first row's bound)
  const int lim_w = (int)max(-1LL, min((long long)pos0 + min(mw, M - 1), (long long)ctx_cap - 1));
  const int mlast = min((qb + 1) * CW * rpw, M) - 1;
  const int ctx = (int)max(0LL, min((long long)pos0 + mlast + 1, (long long)ctx_cap));  // tokens [0, ctx) are read
  h8 q[KS];
  {
    const f16* qh = qkv + (size_t)m * (n_q + 2 * n_kv) * D + (size_t)hd * D + 8 * h;
#pragma unroll
    for (int s = 0; s < KS; ++s) q[s] = __builtin_bit_cast(h8, *reinterpret_cast<const u32x4*>(qh + 16 * s));
  }

  // Thread's share of a round: chunk tid % CH of token rows tid / CH + RPI i. The rows' pages are looked up a round
  // ahead of their K / V loads (branch-free: a lookup behind a branch waits for every load in flight). Tokens without a
  // page read page 0's row (every cache has one), those past ctx a row of the last page (UP) or of page 0; both are zeroed
  // on the way to LDS.
  // UP (pages of at least the 64 / CH rows that one load instruction of a wave covers): the instruction's rows lie in
  // one page, so lane i looks up the page of load i, and the load's base is computed on the scalar unit; with a page
  // per lane the address arithmetic alone took a tenth of the kernel's time.
  const int nrnd = (ctx + SB - 1) / SB;
  const int sch = tid % CH, sr = tid / CH;
  constexpr int RPW = kWave / CH;            // rows per load instruction of a wave
  // RPI is a multiple of 16, so the swizzles of row sr + RPI i are those of row sr
  const int kof = sr * RB + ((D == 128 ? sch ^ (sr & 15) : sch ^ ((sr >> 1) & 7)) << 4);
  const int vof = sr * RB + (((sch >> 2) ^ (D == 128 ? sr & 3 : (sr >> 1) & 1)) << 6) + ((sch & 3) << 4);
  const uint32_t lof = (uint32_t)((lane / CH) * RB + 16 * sch);  // the lane's byte within a load's rows
  u32x4 kk[LPT], vv[LPT];
  int pg[UP ? 1 : LPT];
  bool ok[LPT];
  auto lookup = [&](int rnd) {
    if constexpr (UP) {
      pg[0] = bt[min(rnd * SB + RPW * wave + RPI * (lane % LPT), ctx - 1) >> log2P];
    } else {
#pragma unroll
      for (int i = 0; i < LPT; ++i) pg[i] = bt[min(rnd * SB + sr + RPI * i, ctx - 1) >> log2P];
    }
  };
  auto fetch = [&](int rnd) {
#pragma unroll
    for (int i = 0; i < LPT; ++i) {
      const int t = rnd * SB + sr + RPI * i;
      if constexpr (UP) {
        const int t0 = rnd * SB + RPW * wave + RPI * i, p = __builtin_amdgcn_readlane(pg[0], i);
        const bool mapped = (unsigned)p < (unsigned)n_pages;
        ok[i] = t < ctx && mapped;
        const size_t off = ((((size_t)(mapped ? p : 0) * n_kv + kvh) << log2P) + (t0 & (P - 1))) * RB;
        kk[i] = *reinterpret_cast<const u32x4*>(reinterpret_cast<const uint8_t*>(kc) + off + lof);
        vv[i] = *reinterpret_cast<const u32x4*>(reinterpret_cast<const uint8_t*>(vc) + off + lof);
      } else {
        ok[i] = t < ctx && (unsigned)pg[i] < (unsigned)n_pages;
        const size_t off = ((((size_t)(ok[i] ? pg[i] : 0) * n_kv + kvh) << log2P) + (t & (P - 1))) * D + 8 * sch;
        kk[i] = *reinterpret_cast<const u32x4*>(kc + off);
        vv[i] = *reinterpret_cast<const u32x4*>(vc + off);
      }
    }
  };
  auto stage = [&](int buf) {
    uint8_t* kb = lds + buf * kTile + kof;
    uint8_t* vb = lds + (2 + buf) * kTile + vof;
    bool all = true;
#pragma unroll
    for (int i = 0; i < LPT; ++i) all = all && ok[i];
    if (!__all(all)) {  // the last round, or an unmapped page
      asm volatile("");  // stays a branch
      const u32x4 z = {0u, 0u, 0u, 0u};
#pragma unroll
      for (int i = 0; i < LPT; ++i) {
        kk[i] = ok[i] ? kk[i] : z;
        vv[i] = ok[i] ? vv[i] : z;
      }
    }
#pragma unroll
    for (int i = 0; i < LPT; ++i) {
      *reinterpret_cast<u32x4*>(kb + i * RPI * RB) = kk[i];
      *reinterpret_cast<u32x4*>(vb + i * RPI * RB) = vv[i];
    }
  };

  float mref = kPfNoMax, l = 0.f;  // the column's reference maximum (log2 units); this lane's half of its sum
  f32x16 acc[DT];
#pragma unroll
  for (int t = 0; t < DT; ++t) acc[t] = f32x16{};

  // LDS addresses: K row r of the group's block (chunk bits apart), and the lane's row of a transposing V read
  const int krow = (grp * BT + r) * RB, ksw = D == 128 ? r & 15 : (r >> 1) & 7;
  const int vt = 4 * h + ((lane & 15) >> 2);           // token (of 8) that the lane addresses
  const int vd = 32 * ((lane >> 4) & 1) + 8 * (lane & 3);  // byte of its 4 dims within the 64-byte unit
  const int vrow = (grp * BT + vt) * RB + vd, vsw = D == 128 ? vt & 3 : (vt >> 1) & 1;  // + 8 rows: the same swizzle

  auto compute = [&](int t0, int buf, bool mask) {
    const uint8_t* Kb = lds + buf * kTile + krow;
    const uint8_t* Vb = lds + (2 + buf) * kTile + vrow;
    f32x16 sc[NT];
#pragma unroll
    for (int tt = 0; tt < NT; ++tt) sc[tt] = f32x16{};
    // K fragments (k step f / NT, token tile f % NT), each read from LDS RA fragments ahead of its MFMA
    constexpr int NF = KS * NT, RA = 4;
    u32x4 ka[RA + 1];
    auto read_k = [&](int f) {
      return *reinterpret_cast<const u32x4*>(Kb + (f % NT) * 32 * RB + (((2 * (f / NT) + h) ^ ksw) << 4));
    };
#pragma unroll
    for (int f = 0; f < RA; ++f) ka[f] = read_k(f);
#pragma unroll
    for (int f = 0; f < NF; ++f) {
      if (f + RA < NF) ka[(f + RA) % (RA + 1)] = read_k(f + RA);
      sc[f % NT] = mfma32x32(__builtin_bit_cast(h8, ka[f % (RA + 1)]), q[f / NT], sc[f % NT]);
      __builtin_amdgcn_sched_barrier(0x7);
    }
    if (mask) {  // uniform per wave
      asm volatile("");  // stays a branch
#pragma unroll
      for (int tt = 0; tt < NT; ++tt) {
#pragma unroll
        for (int i = 0; i < 16; ++i)
          if (t0 + 32 * tt + 8 * (i >> 2) + 4 * h + (i & 3) > lim) sc[tt][i] = -INFINITY;
      }
    }
    float mx = sc[0][0];
#pragma unroll
    for (int tt = 0; tt < NT; ++tt) {
#pragma unroll
      for (int i = 0; i < 16; ++i) mx = fmaxf(mx, sc[tt][i]);
    }
    mx = fmaxf(mx, __shfl_xor(mx, 32, kWave)) * c2;
    const bool move = mx > mref + kLazy;
    if (__any(move)) {
      const float mn = move ? mx : mref;
      const float alpha = __builtin_amdgcn_exp2f(mref - mn);  // 1 for a column that stays
      mref = mn;
      l *= alpha;
#pragma unroll
      for (int t = 0; t < DT; ++t) {
#pragma unroll
        for (int i = 0; i < 16; ++i) acc[t][i] *= alpha;
      }
    }
    const float lift = kLift - mref;
    float ps[2] = {0.f, 0.f};
#pragma unroll
    for (int tt = 0; tt < NT; ++tt) {
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const float p = __builtin_amdgcn_exp2f(fmaf(sc[tt][i], c2, lift));
        sc[tt][i] = p;
        ps[i & 1] += p;
      }
    }
    l += ps[0] + ps[1];
#pragma unroll
    for (int ks = 0; ks < 2 * NT; ++ks) {
      h8 phi, plo;
#pragma unroll
      for (int e = 0; e < 8; e += 2) {
        const float p0 = sc[ks >> 1][8 * (ks & 1) + e], p1 = sc[ks >> 1][8 * (ks & 1) + e + 1];
        const h2 hi = __builtin_convertvector(f2{p0, p1}, h2);
        const uint32_t hw = __builtin_bit_cast(uint32_t, hi);
        const h2 lo = __builtin_convertvector(f2{minus_lo(p0, hw), minus_hi(p1, hw)}, h2);
        phi[e] = hi[0];
        phi[e + 1] = hi[1];
        plo[e] = lo[0];
        plo[e + 1] = lo[1];
      }
      h8 v[DT];
#pragma unroll
      for (int t = 0; t < DT; ++t) {
        const uint8_t* src = Vb + ks * 16 * RB + ((t ^ vsw) << 6);
        const u32x2 a = read_tr(src), b = read_tr(src + 8 * RB);
        v[t] = __builtin_bit_cast(h8, u32x4{a[0], a[1], b[0], b[1]});
      }
#pragma unroll
      for (int t = 0; t < DT; ++t) acc[t] = mfma32x32(v[t], phi, acc[t]);
#pragma unroll
      for (int t = 0; t < DT; ++t) acc[t] = mfma32x32(v[t], plo, acc[t]);
    }
  };
  // round rnd: loads of round rnd + 1 go out, the group's block is computed from LDS buffer rnd & 1, the loads land in
  // the other buffer (every wave finished reading it before the last barrier)
  if (nrnd > 0) {  // uniform
    lookup(0);
    fetch(0);
    pf_fence();
    lookup(1);
    pf_fence();
    stage(0);
    __syncthreads();
    for (int rnd = 0; rnd < nrnd; ++rnd) {
      fetch(rnd + 1);  // past the end: nothing is in the context, the rows read are never computed on
      pf_fence();
      lookup(rnd + 2);
      pf_fence();
      const int t0 = (rnd * KVS + grp) * BT;
      compute(t0, rnd & 1, t0 + BT - 1 > lim_w);
      pf_fence();
      stage((rnd + 1) & 1);
      __syncthreads();
    }
  }
  l += __shfl_xor(l, 32, kWave);
  // ---- merge: groups 1 .. KVS - 1 leave maximum and sum per column and the accumulator per lane in LDS (over the K / V
  // buffers, which every wave has finished reading at the last barrier); group 0 merges them in group order
  static_assert(KVS == 1 || (2 * KVS * CW * 32 + (KVS - 1) * CW * kWave * DT * 16) * 4 <= (int)sizeof(lds),
                "merge scratch fits the buffers");
  if constexpr (KVS > 1) {
    float* s_m = reinterpret_cast<float*>(lds);                         // [KVS][CW][32]
    float* s_l = s_m + KVS * CW * 32;                                   // [KVS][CW][32]
    float4* s_acc = reinterpret_cast<float4*>(s_l + KVS * CW * 32);     // [KVS - 1][CW][DT * 4][64]
    if (h == 0) {
      s_m[(grp * CW + gw) * 32 + r] = mref;
      s_l[(grp * CW + gw) * 32 + r] = l;
    }
    if (grp > 0) {
      float4* dst = s_acc + ((grp - 1) * CW + gw) * (DT * 4 * kWave) + lane;
#pragma unroll
      for (int t = 0; t < DT; ++t) {
#pragma unroll
        for (int i = 0; i < 4; ++i)
          dst[(4 * t + i) * kWave] = float4{acc[t][4 * i], acc[t][4 * i + 1], acc[t][4 * i + 2], acc[t][4 * i + 3]};
      }
    }
    __syncthreads();
    if (grp > 0) return;  // uniform per wave; no barrier follows
    float mx = mref;
#pragma unroll
    for (int k = 1; k < KVS; ++k) mx = fmaxf(mx, s_m[(k * CW + gw) * 32 + r]);
    const float w0 = __builtin_amdgcn_exp2f(mref - mx);  // a group that saw no token weighs 0 beside one that did
    l *= w0;
#pragma unroll
    for (int t = 0; t < DT; ++t) {
#pragma unroll
      for (int i = 0; i < 16; ++i) acc[t][i] *= w0;
    }
#pragma unroll
    for (int k = 1; k < KVS; ++k) {
      const float wk = __builtin_amdgcn_exp2f(s_m[(k * CW + gw) * 32 + r] - mx);
      l = fmaf(wk, s_l[(k * CW + gw) * 32 + r], l);
      const float4* src = s_acc + ((k - 1) * CW + gw) * (DT * 4 * kWave) + lane;
#pragma unroll
      for (int t = 0; t < DT; ++t) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const float4 o = src[(4 * t + i) * kWave];
          acc[t][4 * i] = fmaf(wk, o.x, acc[t][4 * i]);
          acc[t][4 * i + 1] = fmaf(wk, o.y, acc[t][4 * i + 1]);
          acc[t][4 * i + 2] = fmaf(wk, o.z, acc[t][4 * i + 2]);
          acc[t][4 * i + 3] = fmaf(wk, o.w, acc[t][4 * i + 3]);
        }
      }
    }
  }
  // ---- output: acc[t][4 q + v] = O[column r][dim 32 t + 8 q + 4 h + v]
  if (mcol < M) {
    const float inv = l > 0.f ? 1.0f / l : 0.f;
    f16* dst = out + (size_t)m * n_q * D + (size_t)hd * D + 4 * h;
    const bool vec = (reinterpret_cast<uintptr_t>(out) & 7) == 0;  // uniform
#pragma unroll
    for (int t = 0; t < DT; ++t) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const f16 o0 = (f16)(acc[t][4 * i] * inv), o1 = (f16)(acc[t][4 * i + 1] * inv);
        const f16 o2 = (f16)(acc[t][4 * i + 2] * inv), o3 = (f16)(acc[t][4 * i + 3] * inv);
        f16* d = dst + 32 * t + 8 * i;
        if (vec) {
          *reinterpret_cast<u32x2*>(d) = u32x2{as_u32(f16x2{o0, o1}), as_u32(f16x2{o2, o3})};
        } else {
          d[0] = o0;
          d[1] = o1;
          d[2] = o2;
          d[3] = o3;
        }
      }
    }
  }
}

// Waves of 32 columns (n_kv * M * HPG / 32) decide the workgroup shape, (CW, KVS, BT) below: few waves are spread over
// the SIMDs by giving the token blocks to more groups, many share each staged block among more columns. Measured in us
// per launch at M tokens from position 0 (TinyLlama heads 4 x 8 x 64, where waves = M; Llama-3-8B heads 8 x 4 x 128,
// likewise), the choice against its neighbours:
//   D  64:   512 tokens  (1,4,32)  8.7  (2,2,64)  9.3   |  1024 (2,2,64) 16.4  (4,1,64) 22.0  (1,4,32) 21.0
//           2048         (4,1,64) 41.2  (2,2,64) 43.1   |  4096 (4,1,64) 123   (2,2,64) 143
//   D 128:   256         (1,4,32)  9.7  (2,4,32) 10.9   |   512 (2,4,32) 15.0  (1,4,32) 21.1  (4,2,64) 17.7
//           1024         (4,2,64) 29.4  (2,4,32) 36.2   |  2048 (4,1,64) 67.4  (4,2,64) 65-75
//           3000         (4,1,64) 120   (8,1,64) 134    |  4096 (8,1,64) 205   (4,1,64) 219
// (The 16 x 16 kernel this replaced: 12.7, 32.0, 81-88, 262 and 13.3, 19.4, 48.5, 163, 320, 560.) What bounds the
// largest shapes is power: the MFMAs alone (with p as hi + lo, 1.5 times the products) take 128 us at Llama-3-8B 4096
// whether or not anything is read from LDS, 1.63 PFLOP/s at the clock that they hold; the softmax adds 40, the staging
// of K / V 57 at four waves per workgroup and 30 at eight. Interleaving one tile's softmax with the next one's scores
// in a wave (255 us) and two wave groups taking turns on the matrix cores behind barriers (217-225) were no faster.
// Pages too small for one base per load instruction (UP) take the general lookup in two of the shapes. At D 128 the
// (2,4,32) shape holds 256 VGPRs and spills 8, with and without UP.
template <int D>
void launch_prefill(const void* qkv, const int32_t* pos, const int32_t* bt, int n_bt, const void* kc, const void* vc,
                    int n_pages, int log2P, int n_q, int n_kv, int M, int max_ctx, void* out, hipStream_t st) {
  const float c2 = (float)(1.4426950408889634 / sqrt((double)D));
  const int cap = (int)min((long long)max_ctx, (long long)n_bt << log2P);
  int lhpg = 0;
  while ((n_kv << lhpg) < n_q) ++lhpg;
  auto go = [&](auto kernel, int cw, int threads) {
    const int rows = cw * (32 >> lhpg);
    const int rb = (M + rows - 1) / rows;
    const int fold = threads == 256 && (long long)n_kv * rb <= 512;  // two workgroups per CU
    hipLaunchKernelGGL(kernel, dim3(n_kv, rb), dim3(threads), 0, st, (const f16*)qkv, pos, bt, n_bt,
                       (const f16*)kc, (const f16*)vc, n_pages, log2P, n_q, n_kv, lhpg, M, cap, fold, c2, (f16*)out);
  };
  const long long waves = (long long)n_kv * ((((long long)M << lhpg) + 31) / 32);
  if ((1 << log2P) < 512 / D) {
    if (waves > 1536)
      go(attn_prefill_kernel<D, 4, 1, 64, false>, 4, 256);
    else
      go(attn_prefill_kernel<D, 2, 4, 32, false>, 2, 512);
    return;
  }
  if constexpr (D == 64) {
    if (waves <= 512)
      go(attn_prefill_kernel<64, 1, 4, 32, true>, 1, 256);
    else if (waves <= 1536)
      go(attn_prefill_kernel<64, 2, 2, 64, true>, 2, 256);
    else
      go(attn_prefill_kernel<64, 4, 1, 64, true>, 4, 256);
  } else {
    if (waves <= 256)
      go(attn_prefill_kernel<128, 1, 4, 32, true>, 1, 256);
    else if (waves <= 640)
      go(attn_prefill_kernel<128, 2, 4, 32, true>, 2, 512);
    else if (waves <= 1536)
      go(attn_prefill_kernel<128, 4, 2, 64, true>, 4, 512);
    else if (waves < 4096)
      go(attn_prefill_kernel<128, 4, 1, 64, true>, 4, 256);
    else
      go(attn_prefill_kernel<128, 8, 1, 64, true>, 8, 512);
  }
}

}  // namespace

void launch_attention_prefill(const void* qkv, const int32_t* pos, const int32_t* bt, int n_bt, const void* kc,
                              const void* vc, int n_pages, int log2P, int n_q, int n_kv, int head_dim, int M,
                              int max_ctx, void* out, hipStream_t st) {
  if (head_dim == 64)
    launch_prefill<64>(qkv, pos, bt, n_bt, kc, vc, n_pages, log2P, n_q, n_kv, M, max_ctx, out, st);
  else
    launch_prefill<128>(qkv, pos, bt, n_bt, kc, vc, n_pages, log2P, n_q, n_kv, M, max_ctx, out, st);
}

}  // namespace dk
