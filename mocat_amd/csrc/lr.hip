// Bayesian logistic regression on the GPU: fused potential + hand-written adjoint, and the fused
// HMC / MALA / underdamped-Langevin iteration built on it.
//
// Model (a user Scenario in the reference's README pattern, README.md:35-49):
//   prior_potential(theta)      = 0.5 * prec * |theta|^2 + 0.5 * d * (log 2pi - log prec)
//   likelihood_potential(theta) = sum_i softplus(x_i . theta) - y_i * (x_i . theta)
//   grad_likelihood             = X^T (sigmoid(X theta) - y)
// Chains/particles are processed in tiles of 32: the contraction over the data rows is the hot loop.
//
// Three engines evaluate (U, grad U) for a tile:
//   Fp32Engine - data rows staged through LDS in chunks, FP32 FMAs on the vector ALU.
//   Fp64Engine - the same in FP64 (the reference for the error of the other two).
//   Bf16Engine - MFMA v_mfma_f32_32x32x16_bf16 with split precision: every operand is
//                hi + lo bf16 and each product is hi*hi + hi*lo + lo*hi in FP32 accumulation.
//                Z = X Theta^T is accumulated with rows of X on the M side and the 32 chains on
//                N, so each lane's accumulator column is one chain. sigmoid(Z) - y is formed in
//                registers and reused directly as the A operand (chains x rows) of
//                G = R X: the K slots of that operand are the rows the lane already holds, and
//                X's second packed layout lists its rows in the same order.
//
// The iteration kernel follows mocat's Underdamped + Metropolis/RMMetropolis update
// (mocat/src/mcmc/standard_mcmc.py:107-153, mocat/src/utils.py:108-146,
//  mocat/src/mcmc/metropolis.py:48-161), one chain per (tile, slot), key tree per chain as mocat's
// single-chain run (mocat/src/mcmc/sampler.py:92-111).
#include <type_traits>

#include "common.hpp"

using namespace mocat;

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float floatx16 __attribute__((ext_vector_type(16)));
typedef float floatx4 __attribute__((ext_vector_type(4)));

namespace {

constexpr int CT = 32;  // chains per tile
constexpr float kLog2Pi = 1.83787706640934548356f;

MOCAT_DEV int acc_row(int r, int lane) { return 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3); }

// --- per-row likelihood pieces -------------------------------------------------------------
// r = sigmoid(z) - y ; c = softplus(z) - y z. Rows with y < 0 are padding: r = c = 0.
// Hardware exp2/log2/rcp (v_exp_f32, v_log_f32, v_rcp_f32): |error| of c per row <= ~1e-7 absolute.
MOCAT_DEV void lr_row(float z, float y, float& r, float& c) {
  const float e = __expf(-fabsf(z));
  const float ope = 1.f + e;
  const float inv = __builtin_amdgcn_rcpf(ope);
  const float sig = z >= 0.f ? inv : e * inv;
  const bool valid = y >= 0.f;
  r = valid ? sig - y : 0.f;
  c = valid ? fmaxf(z, 0.f) + __logf(ope) - y * z : 0.f;
}

// MFMA-engine rows on the hardware transcendentals only (v_exp_f32 = 2^x, v_log_f32 = log2,
// v_rcp_f32): t = 2^(-z log2 e) = exp(-z), r = 1 / (1 + t) - y; softplus(z) = max(z + ln2 log2(1 + t), 0)
// with the exponent clamped below overflow (1 + t >= 1, so no denormal inputs reach v_log_f32).
// Padding rows hold x = 0 and y = 0.5, so r = 0 there.
constexpr float kLog2E = 1.44269504088896340736f;
constexpr float kLn2 = 0.69314718055994530942f;
// Both take zs = -z log2(e), the engine's accumulator (X is packed premultiplied by -log2(e)).
MOCAT_DEV float lr_row_grad_hw(float zs, float y) {
  const float t = __builtin_amdgcn_exp2f(zs);
  return __builtin_amdgcn_rcpf(1.f + t) - y;
}
MOCAT_DEV float lr_row_full_hw(float zs, float y, float& c) {
  const float t = __builtin_amdgcn_exp2f(fminf(zs, 126.f));
  const float ope = 1.f + t;
  const float z = zs * -kLn2;
  c = fmaxf(z + kLn2 * __builtin_amdgcn_logf(ope), 0.f) - y * z;
  return __builtin_amdgcn_rcpf(ope) - y;
}

// Split two floats into packed bf16 pairs, v = hi + lo: hi keeps the upper 16 bits of v (truncation,
// one v_perm_b32 packs both), lo = v - hi exactly in FP32, rounded to bf16 by v_cvt_pk_bf16_f32.
// |v - hi - lo| <= 2^-16 |v|, the same order as a rounded split.
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float floatx2 __attribute__((ext_vector_type(2)));
MOCAT_DEV void split_pair(float v0, float v1, uint32_t& hi, uint32_t& lo) {
  const uint32_t u0 = __float_as_uint(v0) & 0xffff0000u, u1 = __float_as_uint(v1) & 0xffff0000u;
  hi = __builtin_amdgcn_perm(u1, u0, 0x07060302u);
  const floatx2 l = {v0 - __uint_as_float(u0), v1 - __uint_as_float(u1)};
  const bf16x2 lb = __builtin_convertvector(l, bf16x2);
  lo = __builtin_bit_cast(uint32_t, lb);
}

// ------------------------------------------------------------------------------------------
// FP32 engine.  LDS: X chunk [RC][DP+4], R chunk [CT][RC+4].
template <int DP, int NT>
struct Fp32Engine {
  static constexpr int RC = 64;
  static constexpr int XS = DP + 4;
  static constexpr int RS = RC + 4;
  struct alignas(16) Smem {
    alignas(16) float x[RC * XS];
    alignas(16) float r[CT * RS];
    float y[RC];
    float red[NT / kWave][CT];
  };

  // theta: LDS [CT][DP] (zero beyond d). Outputs: lik[CT], glik[CT][DP] in LDS.
  static MOCAT_DEV void eval(Smem& s, const float* __restrict__ X, const float* __restrict__ y, const void*,
                             int n, int d, const float* theta, float* lik, float* glik, bool /*want_pot*/) {
    const int t = threadIdx.x;
    const int lane = t & (kWave - 1), w = t / kWave;
    constexpr int NW = NT / kWave;
    constexpr int P1 = CT / NW;         // chains per thread in phase 1 (row = lane)
    constexpr int KPT = DP / kWave;     // k columns per thread in phase 2 (1 or 2)
    float gacc[P1][KPT];
    float cacc[P1];
#pragma unroll
    for (int m = 0; m < P1; ++m) {
      cacc[m] = 0.f;
#pragma unroll
      for (int q = 0; q < KPT; ++q) gacc[m][q] = 0.f;
    }
    for (int i0 = 0; i0 < n; i0 += RC) {
      __syncthreads();
      // stage X rows [i0, i0+RC) and y
      for (int e = t; e < RC * DP; e += NT) {
        const int i = e / DP, k = e - i * DP;
        const int gi = i0 + i;
        s.x[i * XS + k] = (gi < n && k < d) ? X[(int64_t)gi * d + k] : 0.f;
      }
      for (int i = t; i < RC; i += NT) s.y[i] = (i0 + i < n) ? y[i0 + i] : -1.f;
      __syncthreads();
      // phase 1: z[c][i] for row i = lane, chains c = w + NW*m
      {
        float z[P1];
#pragma unroll
        for (int m = 0; m < P1; ++m) z[m] = 0.f;
        const float* xr = &s.x[lane * XS];
#pragma unroll 4
        for (int k = 0; k < DP; k += 4) {
          const floatx4 xv = *reinterpret_cast<const floatx4*>(xr + k);
#pragma unroll
          for (int m = 0; m < P1; ++m) {
            const floatx4 tv = *reinterpret_cast<const floatx4*>(theta + (w + NW * m) * DP + k);
            z[m] += xv.x * tv.x + xv.y * tv.y + xv.z * tv.z + xv.w * tv.w;
          }
        }
        const float yv = s.y[lane];
#pragma unroll
        for (int m = 0; m < P1; ++m) {
          float r, c;
          lr_row(z[m], yv, r, c);
          cacc[m] += c;
          s.r[(w + NW * m) * RS + lane] = r;
        }
      }
      __syncthreads();
      // phase 2: g[c][k] += sum_i r[c][i] x[i][k], k = lane (+64), chains c = w + NW*m
#pragma unroll 2
      for (int i = 0; i < RC; i += 4) {
        float xv[4][KPT];
#pragma unroll
        for (int ii = 0; ii < 4; ++ii)
#pragma unroll
          for (int q = 0; q < KPT; ++q) xv[ii][q] = s.x[(i + ii) * XS + lane + kWave * q];
#pragma unroll
        for (int m = 0; m < P1; ++m) {
          const floatx4 rv = *reinterpret_cast<const floatx4*>(&s.r[(w + NW * m) * RS + i]);
#pragma unroll
          for (int q = 0; q < KPT; ++q)
            gacc[m][q] += rv.x * xv[0][q] + rv.y * xv[1][q] + rv.z * xv[2][q] + rv.w * xv[3][q];
        }
      }
    }
    // outputs: each (chain, k) owned by exactly one thread; potentials reduced over lanes
#pragma unroll
    for (int m = 0; m < P1; ++m) {
      const int c = w + NW * m;
#pragma unroll
      for (int q = 0; q < KPT; ++q) glik[c * DP + lane + kWave * q] = gacc[m][q];
      const float cs = wave_sum(cacc[m]);
      if (lane == 0) lik[c] = cs;
    }
    __syncthreads();
  }
};

// ------------------------------------------------------------------------------------------
// FP64 engine: the same contraction with every product, sum and row function in double (the
// reference run that error statements of the split-precision engine are made against). The tile
// state stays f32: theta is widened exactly, the outputs are rounded once. LDS: X chunk
// [RC][DP+1] and R chunk [CT][RC+1] in double.
template <int DP, int NT>
struct Fp64Engine {
  static constexpr int RC = 32;
  static constexpr int XS = DP + 1;
  static constexpr int RS = RC + 1;
  struct alignas(16) Smem {
    double x[RC * XS];
    double r[CT * RS];
    double y[RC];
  };

  static MOCAT_DEV void eval(Smem& s, const float* __restrict__ X, const float* __restrict__ y, const void*,
                             int n, int d, const float* theta, float* lik, float* glik, bool /*want_pot*/) {
    const int t = threadIdx.x;
    const int lane = t & (kWave - 1), w = t / kWave;
    constexpr int NW = NT / kWave;
    constexpr int G1 = NW * 2;          // phase 1: chain groups (row = lane % 32)
    constexpr int P1 = CT / G1;         // chains per thread in phase 1
    constexpr int P2 = CT / NW;         // chains per thread in phase 2 (column = lane (+64))
    constexpr int KPT = DP / kWave;
    static_assert(CT % G1 == 0 && CT % NW == 0, "tile shape");
    const int row = lane & 31, grp = w * 2 + (lane >> 5);
    double gacc[P2][KPT];
    double cacc[P1];
#pragma unroll
    for (int m = 0; m < P1; ++m) cacc[m] = 0.0;
#pragma unroll
    for (int m = 0; m < P2; ++m)
#pragma unroll
      for (int q = 0; q < KPT; ++q) gacc[m][q] = 0.0;
    for (int i0 = 0; i0 < n; i0 += RC) {
      __syncthreads();
      for (int e = t; e < RC * DP; e += NT) {
        const int i = e / DP, k = e - i * DP;
        const int gi = i0 + i;
        s.x[i * XS + k] = (gi < n && k < d) ? (double)X[(int64_t)gi * d + k] : 0.0;
      }
      for (int i = t; i < RC; i += NT) s.y[i] = (i0 + i < n) ? (double)y[i0 + i] : -1.0;
      __syncthreads();
      {
        double z[P1];
#pragma unroll
        for (int m = 0; m < P1; ++m) z[m] = 0.0;
        const double* xr = &s.x[row * XS];
        for (int k = 0; k < d; ++k) {
          const double xv = xr[k];
#pragma unroll
          for (int m = 0; m < P1; ++m) z[m] = fma(xv, (double)theta[(grp + G1 * m) * DP + k], z[m]);
        }
        const double yv = s.y[row];
#pragma unroll
        for (int m = 0; m < P1; ++m) {
          double r = 0.0, c = 0.0;
          if (yv >= 0.0) {
            const double e = exp(-fabs(z[m]));
            const double sig = z[m] >= 0.0 ? 1.0 / (1.0 + e) : e / (1.0 + e);
            r = sig - yv;
            c = fmax(z[m], 0.0) + log1p(e) - yv * z[m];
          }
          cacc[m] += c;
          s.r[(grp + G1 * m) * RS + row] = r;
        }
      }
      __syncthreads();
      for (int i = 0; i < RC; ++i) {
        double xv[KPT];
#pragma unroll
        for (int q = 0; q < KPT; ++q) xv[q] = s.x[i * XS + lane + kWave * q];
#pragma unroll
        for (int m = 0; m < P2; ++m) {
          const double rv = s.r[(w + NW * m) * RS + i];
#pragma unroll
          for (int q = 0; q < KPT; ++q) gacc[m][q] = fma(rv, xv[q], gacc[m][q]);
        }
      }
    }
    __syncthreads();
    // potentials: the two half-waves hold different chains; sum each chain's rows over its 32 lanes
#pragma unroll
    for (int m = 0; m < P1; ++m) {
      double v = cacc[m];
#pragma unroll
      for (int off = 16; off > 0; off >>= 1) v += __shfl_xor(v, off, 32);
      if (row == 0) lik[grp + G1 * m] = (float)v;
    }
#pragma unroll
    for (int m = 0; m < P2; ++m)
#pragma unroll
      for (int q = 0; q < KPT; ++q) glik[(w + NW * m) * DP + lane + kWave * q] = (float)gacc[m][q];
    __syncthreads();
  }
};

// ------------------------------------------------------------------------------------------
// BF16 split-precision MFMA engine.
// Packed data per block of 32 rows (rb):
//   A layout [2 parts][KB][64 lanes][8]   lane l: row l%32, columns kb*16 + (l/32)*8 + s
//   B layout [2 parts][2][NB][64][8]      lane l: column nb*32 + l%32, rows acc_row(kb2*8+s, l)
//   y layout [2][16] f32                  g = l/32: y[acc_row(r, l)], 0.5 on padding rows (x = 0 there)
template <int DP>
struct PackLayout {
  // The engine reads X premultiplied by -log2(e) in the GEMM-1 (A) layout, so that its accumulators
  // hold z' = -z log2(e) and exp(-z) = 2^z' needs no multiply; the B layout is plain X.
  static constexpr float kAScale = -kLog2E;
  static constexpr int KB = DP / 16;
  static constexpr int NB = DP / 32;
  static constexpr int A_ELEMS = 2 * KB * 512;
  static constexpr int B_ELEMS = 2 * 2 * NB * 512;
  static constexpr int BLOCK_BF16 = A_ELEMS + B_ELEMS;
  static constexpr int BLOCK_BYTES = BLOCK_BF16 * 2 + 32 * 4;
};

MOCAT_DEV void split_bf16(float v, __bf16& hi, __bf16& lo) {
  hi = (__bf16)v;
  lo = (__bf16)(v - (float)hi);
}

// ------------------------------------------------------------------------------------------
// BF16 split-precision MFMA engine (every product hi*hi + hi*lo + lo*hi, FP32 accumulation).
// Z = X Theta^T is accumulated with rows of X on the M side and 32 chains on N, so each lane's
// accumulator column is one chain; R = sigmoid(Z) - y is formed in registers and reused directly as
// the A operand (chains x rows) of G = R X: the K slots of that operand are the rows the lane already
// holds, and X's second packed layout lists its rows in the same order. With NW waves, wave w takes
// the 32-row blocks rb = w + NW j; two waves per SIMD (NW = 8) let one wave's row functions on the
// vector ALU overlap the other's MFMAs.
//
// A workgroup takes NCT tiles of 32 chains. What bounds one tile most is the first-level cache: every wave streams its
// blocks' operands through it at 64 B per clock, 32 KB per 32 rows at d > 64 (2050 clocks for four waves, their
// MFMAs 1540) and 16 KB at d <= 64 (2050 clocks for eight waves, the MFMAs 1540), and each block's labels another quarter
// of that at d <= 64 (16 bytes a lane, four times). Counters of the moves at d = 50: 0.8 accesses of 64 B a clock in
// the block loop, the return path busy 83% of all clocks, vector ALU 50%, matrix pipe 43%. Leaving out the
// transcendentals or taking the operands from a hot line changes little there, and neither do two blocks at once per wave
// (slower) or waves out of phase. Two tiles use each operand twice (0.39 accesses a clock); then the one wave per SIMD takes
// turns between the vector ALU (52% of the clocks) and the matrix pipe (50%), one of them busy in 83%: 288-309 TFLOP/s
// algorithmic at d = 100, 1105-1190 issued, where a large bf16 product reaches 1320-1344. (One MFMA for the last columns' three
// products, at d = 50 and 100 10 instead of 12 and 19 instead of 24 per block, would give another 6%, but sums them in
// another order: chains of 200 leapfrog steps then end up to 3e-5 from where they ended before.)
template <int DP, int NT, int NCT>
struct Bf16Engine {
  using L = PackLayout<DP>;
  static constexpr int KB = L::KB, NB = L::NB, NW = NT / kWave;
  static_assert(NW % 4 == 0, "whole SIMDs");
  static_assert(L::kAScale == -kLog2E, "the rows expect the scaled A layout");
  static constexpr bool kThetaRegs = DP <= 64 && NCT == 1;
  static constexpr int GS = DP + 4;  // row stride of the partial gradients (spreads LDS banks)
  struct alignas(16) Smem {
    alignas(16) float gred[NW][CT * GS];
    alignas(16) bf16x8 thl[NCT][2][KB][64];  // theta^T operands, hi and lo parts, per lane
    float ured[NW][2][NCT * CT];
  };
  struct Acc {
    floatx16 g[NCT][NB];  // the wave's partial gradients
    float u[NCT];         // and potential terms
  };
  struct ABuf {
    bf16x8 h[KB], l[KB];
  };
  struct BBuf {
    floatx4 y[4];
    bf16x8 h[2][NB], l[2][NB];
  };

  // Writes columns k .. k + 3 (k a multiple of 4) of chain c of tile ct into theta's operands.
  static MOCAT_DEV void put_theta(Smem& s, int ct, int c, int k, const float* v) {
    typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
    bf16x4 h4, l4;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      __bf16 h, l;
      split_bf16(v[q], h, l);
      h4[q] = h;
      l4[q] = l;
    }
    const int ln = c + 32 * ((k / 8) & 1);  // operand (k / 16, lane ln), elements k % 8 ..
    reinterpret_cast<bf16x4*>(&s.thl[ct][0][k / 16][ln])[(k / 4) & 1] = h4;
    reinterpret_cast<bf16x4*>(&s.thl[ct][1][k / 16][ln])[(k / 4) & 1] = l4;
  }

  // The block loop of one gradient evaluation. Theta's operands are read from s.thl (written by the
  // caller before a barrier); each wave returns its partial gradients and leaves its potential partials in
  // s.ured[w]. Two compiled passes (the potential terms are needed after the last leapfrog step only), so that
  // each block's row functions and MFMAs form one straight-line region the scheduler can interleave.
  // SPLIT: the workgroup is number `part` of `parts` that share the blocks, wave w takes rb = part NW + w + parts NW j.
  template <bool WANT_POT, bool SPLIT = false>
  static MOCAT_DEV void partials(Smem& s, const void* packed, int n, Acc& acc, int part = 0, int parts = 1) {
    const int t = threadIdx.x;
    const int lane = t & (kWave - 1), w = t / kWave, g = lane >> 5, col = lane & 31;
    const int nrb = (n + 31) / 32;
    const int rb0 = SPLIT ? part * NW + w : w, stride = SPLIT ? parts * NW : NW;
    const int nmine = nrb > rb0 ? (nrb - rb0 + stride - 1) / stride : 0;  // blocks rb = rb0 + j * stride, j < nmine
    const char* base = reinterpret_cast<const char*>(packed);
    bf16x8 th[kThetaRegs ? KB : 1], tl[kThetaRegs ? KB : 1];
    if constexpr (kThetaRegs) {
#pragma unroll
      for (int kb = 0; kb < KB; ++kb) {
        th[kb] = s.thl[0][0][kb][lane];
        tl[kb] = s.thl[0][1][kb][lane];
      }
    }
#pragma unroll
    for (int ct = 0; ct < NCT; ++ct) {
      acc.u[ct] = 0.f;
#pragma unroll
      for (int nb = 0; nb < NB; ++nb)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc.g[ct][nb][r] = 0.f;
    }

    auto blk = [&](int j) { return base + (int64_t)(rb0 + j * stride) * L::BLOCK_BYTES; };
    auto load_a = [&](ABuf& a, int j) {
      const bf16x8* A = reinterpret_cast<const bf16x8*>(blk(j));
#pragma unroll
      for (int kb = 0; kb < KB; ++kb) {
        a.h[kb] = A[(0 * KB + kb) * 64 + lane];
        a.l[kb] = A[(1 * KB + kb) * 64 + lane];
      }
    };
    auto load_b = [&](BBuf& b, int j) {
      const char* bp = blk(j);
      const floatx4* yv4 = reinterpret_cast<const floatx4*>(bp + L::BLOCK_BF16 * 2 + g * 64);
#pragma unroll
      for (int q = 0; q < 4; ++q) b.y[q] = yv4[q];
      const bf16x8* B = reinterpret_cast<const bf16x8*>(bp) + L::A_ELEMS / 8;
#pragma unroll
      for (int kb2 = 0; kb2 < 2; ++kb2)
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) {
          b.h[kb2][nb] = B[((0 * 2 + kb2) * NB + nb) * 64 + lane];
          b.l[kb2][nb] = B[((1 * 2 + kb2) * NB + nb) * 64 + lane];
        }
    };
    auto gemm1 = [&](const ABuf& a, floatx16 (&z)[NCT]) {
#pragma unroll
      for (int ct = 0; ct < NCT; ++ct)
#pragma unroll
        for (int r = 0; r < 16; ++r) z[ct][r] = 0.f;
#pragma unroll
      for (int kb = 0; kb < KB; ++kb) {
        bf16x8 h8[NCT], l8[NCT];
#pragma unroll
        for (int ct = 0; ct < NCT; ++ct) {
          h8[ct] = kThetaRegs ? th[kThetaRegs ? kb : 0] : s.thl[ct][0][kb][lane];
          l8[ct] = kThetaRegs ? tl[kThetaRegs ? kb : 0] : s.thl[ct][1][kb][lane];
        }
#pragma unroll
        for (int ct = 0; ct < NCT; ++ct) z[ct] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a.h[kb], h8[ct], z[ct], 0, 0, 0);
#pragma unroll
        for (int ct = 0; ct < NCT; ++ct) z[ct] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a.h[kb], l8[ct], z[ct], 0, 0, 0);
#pragma unroll
        for (int ct = 0; ct < NCT; ++ct) z[ct] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a.l[kb], h8[ct], z[ct], 0, 0, 0);
      }
    };
    // one block: rows of Z_j with labels and B operands bc, then G += R_j X_j
    auto step = [&](const floatx16 (&z)[NCT], const BBuf& bc) {
      float yv[16];
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        yv[4 * q] = bc.y[q].x;
        yv[4 * q + 1] = bc.y[q].y;
        yv[4 * q + 2] = bc.y[q].z;
        yv[4 * q + 3] = bc.y[q].w;
      }
#pragma unroll
      for (int ct = 0; ct < NCT; ++ct) {
        float rv[16];
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          if constexpr (WANT_POT) {
            float cc;
            rv[r] = lr_row_full_hw(z[ct][r], yv[r], cc);
            acc.u[ct] += cc;  // padding rows are taken out after the loop
          } else {
            rv[r] = lr_row_grad_hw(z[ct][r], yv[r]);
          }
        }
        typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
        u32x4 ph[2], pl[2];
#pragma unroll
        for (int q = 0; q < 8; ++q) {
          uint32_t hw, lw;
          split_pair(rv[2 * q], rv[2 * q + 1], hw, lw);
          ph[q >> 2][q & 3] = hw;
          pl[q >> 2][q & 3] = lw;
        }
#pragma unroll
        for (int kb2 = 0; kb2 < 2; ++kb2) {
          const bf16x8 rh = __builtin_bit_cast(bf16x8, ph[kb2]), rl = __builtin_bit_cast(bf16x8, pl[kb2]);
#pragma unroll
          for (int nb = 0; nb < NB; ++nb) {
            floatx16& ga = acc.g[ct][nb];
            ga = __builtin_amdgcn_mfma_f32_32x32x16_bf16(rh, bc.h[kb2][nb], ga, 0, 0, 0);
            ga = __builtin_amdgcn_mfma_f32_32x32x16_bf16(rh, bc.l[kb2][nb], ga, 0, 0, 0);
            ga = __builtin_amdgcn_mfma_f32_32x32x16_bf16(rl, bc.h[kb2][nb], ga, 0, 0, 0);
          }
        }
      }
    };
    for (int j = 0; j < nmine; ++j) {
      ABuf a;
      BBuf b;
      floatx16 z[NCT];
      load_a(a, j);
      // At two waves per SIMD a wave issuing its first GEMM and the next loads runs at raised priority, so that
      // the other wave's row functions fill the vector ALU meanwhile (measured 3% faster per HMC iteration at
      // the bench shape; at one wave per SIMD it does not apply)
      if constexpr (NW == 8) __builtin_amdgcn_s_setprio(1);
      gemm1(a, z);
      load_b(b, j);
      if constexpr (NW == 8) __builtin_amdgcn_s_setprio(0);
      step(z, b);
    }
    if constexpr (WANT_POT) {
      // padding rows of the last block (x = 0, y = 0.5: z = 0) each added the same term
      const int rbl = nrb - 1;
      if (rbl % stride == rb0) {
        float cpad;
        lr_row_full_hw(0.f, 0.5f, cpad);
        int npad = 0;
#pragma unroll
        for (int r = 0; r < 16; ++r) npad += (rbl * 32 + acc_row(r, lane) >= n);
#pragma unroll
        for (int ct = 0; ct < NCT; ++ct) acc.u[ct] -= (float)npad * cpad;
      }
#pragma unroll
      for (int ct = 0; ct < NCT; ++ct) s.ured[w][g][ct * CT + col] = acc.u[ct];
    }
  }

  // Leaves the wave's partial gradient of tile ct in s.gred[w] ([chain][GS]); readers (after a barrier) sum the
  // waves' in order.
  static MOCAT_DEV void put_partials(Smem& s, const Acc& acc, int ct) {
    const int lane = threadIdx.x & (kWave - 1), w = threadIdx.x / kWave, col = lane & 31;
#pragma unroll
    for (int nb = 0; nb < NB; ++nb)
#pragma unroll
      for (int r = 0; r < 16; ++r) s.gred[w][acc_row(r, lane) * GS + nb * 32 + col] = acc.g[ct][nb][r];
  }
  static MOCAT_DEV floatx4 gradient(const Smem& s, int c, int k) {
    floatx4 v = *reinterpret_cast<const floatx4*>(&s.gred[0][c * GS + k]);
#pragma unroll
    for (int w = 1; w < NW; ++w) v += *reinterpret_cast<const floatx4*>(&s.gred[w][c * GS + k]);
    return v;
  }
  static MOCAT_DEV float potential(const Smem& s, int c) {  // c: chain of the NCT tiles
    float lk = 0.f;
    for (int w = 0; w < NW; ++w) lk += s.ured[w][0][c] + s.ured[w][1][c];
    return lk;
  }
};

// Pack X (n x d, row-major f32) and y into the Bf16Engine layout, zero padded to DP columns and a
// multiple of 32 rows. One thread per packed element.
template <int DP>
__global__ void lr_pack_kernel(const float* __restrict__ X, const float* __restrict__ y, int n, int d,
                               char* __restrict__ out) {
  using L = PackLayout<DP>;
  const int nrb = (n + 31) / 32;
  const int64_t per = L::BLOCK_BF16 + 32;
  const int64_t total = (int64_t)nrb * per;
  for (int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; e < total; e += (int64_t)gridDim.x * blockDim.x) {
    const int rb = (int)(e / per);
    const int q = (int)(e - rb * per);
    char* blk = out + (int64_t)rb * L::BLOCK_BYTES;
    if (q < L::A_ELEMS) {
      const int s = q & 7, lane = (q >> 3) & 63, pk = q >> 9;  // pk = part*KB + kb
      const int part = pk / L::KB, kb = pk - part * L::KB;
      const int row = rb * 32 + (lane & 31), colm = kb * 16 + (lane >> 5) * 8 + s;
      const float v = (row < n && colm < d) ? X[(int64_t)row * d + colm] * L::kAScale : 0.f;
      __bf16 h, l;
      split_bf16(v, h, l);
      reinterpret_cast<__bf16*>(blk)[q] = part ? l : h;
    } else if (q < L::BLOCK_BF16) {
      const int qq = q - L::A_ELEMS;
      const int s = qq & 7, lane = (qq >> 3) & 63, rest = qq >> 9;  // rest = (part*2 + kb2)*NB + nb
      const int nb = rest % L::NB, pk2 = rest / L::NB, kb2 = pk2 & 1, part = pk2 >> 1;
      const int row = rb * 32 + acc_row(kb2 * 8 + s, lane), colm = nb * 32 + (lane & 31);
      const float v = (row < n && colm < d) ? X[(int64_t)row * d + colm] : 0.f;
      __bf16 h, l;
      split_bf16(v, h, l);
      reinterpret_cast<__bf16*>(blk)[q] = part ? l : h;
    } else {
      const int qq = q - L::BLOCK_BF16;  // 0..31 = g*16 + r
      const int gg = qq >> 4, r = qq & 15;
      const int row = rb * 32 + 8 * (r >> 2) + 4 * gg + (r & 3);
      reinterpret_cast<float*>(blk + L::BLOCK_BF16 * 2)[qq] = row < n ? y[row] : 0.5f;
    }
  }
}

// ------------------------------------------------------------------------------------------
// Diagonal Gaussian likelihood engine (mocat/src/scenarios/toy_examples.py:19-51 with a diagonal
// covariance): lik = 0.5 * sum_k lam_k (theta_k - mu_k)^2, grad = lam * (theta - mu).
// Data: X -> mu[d], y -> lam[d] (precisions); n unused.
template <int DP, int NT>
struct GaussEngine {
  struct alignas(16) Smem {
    float part[CT * DP];
  };
  static MOCAT_DEV void eval(Smem& s, const float* __restrict__ mu, const float* __restrict__ lam, const void*, int,
                             int d, const float* theta, float* lik, float* glik, bool /*want_pot*/) {
    const int t = threadIdx.x;
    for (int e = t; e < CT * DP; e += NT) {
      const int k = e % DP;
      float g = 0.f, c = 0.f;
      if (k < d) {
        const float df = theta[e] - mu[k];
        g = lam[k] * df;
        c = 0.5f * lam[k] * df * df;
      }
      glik[e] = g;
      s.part[e] = c;
    }
    __syncthreads();
    if (t < CT) {
      float acc = 0.f;
      for (int k = 0; k < d; ++k) acc += s.part[t * DP + k];
      lik[t] = acc;
    }
    __syncthreads();
  }
};

// ------------------------------------------------------------------------------------------
// Tile state shared by the evaluation and iteration kernels.
template <int DP>
struct alignas(16) TileState {
  alignas(16) float theta[CT * DP];
  float mom[CT * DP];
  float grad[CT * DP];  // grad of the tempered potential
  float glik[CT * DP];
  float lik[CT];
  float pot[CT];
  float prior[CT];
  float likv[CT];
  float pot0[CT];
  float prior0[CT];
  float lik0[CT];
  float step[CT];
  float alpha[CT];
  float kin0[CT];
  float sq[CT];
  uint32_t key[CT][2];
};

// out[c] = sum_k v[c][k]^2 for the CT chains of a tile (one wave per chain group), then a barrier.
template <int DP, int NT>
MOCAT_DEV void chain_sqnorm(const float* v, int d, float* out) {
  constexpr int NW = NT / kWave;
  const int t = threadIdx.x, lane = t & (kWave - 1), w = t / kWave;
  __syncthreads();
  for (int c = w; c < CT; c += NW) {
    float a = 0.f;
    for (int k = lane; k < d; k += kWave) a += v[c * DP + k] * v[c * DP + k];
    a = wave_sum(a);
    if (lane == 0) out[c] = a;
  }
  __syncthreads();
}

struct LrArgs {
  const float* X;
  const float* y;
  const void* packed;
  int n, d;
  float prior_prec, temperature;
};

// Evaluates prior/likelihood potentials and gradients of the tile's theta (in LDS).
// want_pot = false (intermediate leapfrog steps): the gradient only; the potentials are left as they were.
template <class Engine, int DP, int NT>
MOCAT_DEV void tile_eval(typename Engine::Smem& es, TileState<DP>& ts, const LrArgs& a, bool want_pot = true) {
  Engine::eval(es, a.X, a.y, a.packed, a.n, a.d, ts.theta, ts.lik, ts.glik, want_pot);
  const int t = threadIdx.x;
  for (int e = t; e < CT * DP; e += NT) ts.grad[e] = a.prior_prec * ts.theta[e] + a.temperature * ts.glik[e];
  if (want_pot) {
    chain_sqnorm<DP, NT>(ts.theta, a.d, ts.sq);
    if (t < CT) {
      // prec == 0: improper flat prior, potential 0 (mocat's default uniform prior, core.py:183-189)
      const float pr = a.prior_prec > 0.f
                           ? 0.5f * a.prior_prec * ts.sq[t] + 0.5f * (float)a.d * (kLog2Pi - logf(a.prior_prec))
                           : 0.f;
      ts.prior[t] = pr;
      ts.likv[t] = ts.lik[t];
      ts.pot[t] = pr + a.temperature * ts.lik[t];
    }
  }
  __syncthreads();
}

// SPLIT: gridDim.y workgroups share the rows of X, `rows` each, and write partial sums as lr_eval_bf16_kernel does.
template <class Engine, int DP, int NT, bool SPLIT = false>
__global__ __launch_bounds__(NT) void lr_eval_kernel(LrArgs a, const float* __restrict__ theta, int64_t C,
                                                     float* prior_pot, float* lik_pot, float* grad_prior,
                                                     float* grad_lik, int rows = 0) {
  if constexpr (SPLIT) {
    const int part = (int)blockIdx.y, r0 = part * rows;
    a.X += (int64_t)r0 * a.d;
    a.y += r0;
    a.n = a.n - r0 < rows ? a.n - r0 : rows;
    if (part != 0) prior_pot = grad_prior = nullptr;
    lik_pot += part * C;
    grad_lik += part * C * a.d;
  }
  __shared__ TileState<DP> ts;
  __shared__ typename Engine::Smem es;
  const int t = threadIdx.x;
  const int64_t c0 = (int64_t)blockIdx.x * CT;
  for (int e = t; e < CT * DP; e += NT) {
    const int c = e / DP, k = e - c * DP;
    ts.theta[e] = (c0 + c < C && k < a.d) ? theta[(c0 + c) * a.d + k] : 0.f;
  }
  __syncthreads();
  tile_eval<Engine, DP, NT>(es, ts, a);
  for (int e = t; e < CT * DP; e += NT) {
    const int c = e / DP, k = e - c * DP;
    if (c0 + c < C && k < a.d) {
      if (grad_lik) grad_lik[(c0 + c) * a.d + k] = ts.glik[e];
      if (grad_prior) grad_prior[(c0 + c) * a.d + k] = a.prior_prec * ts.theta[e];
    }
  }
  if (t < CT && c0 + t < C) {
    if (prior_pot) prior_pot[c0 + t] = ts.prior[t];
    if (lik_pot) lik_pot[c0 + t] = ts.likv[t];
  }
}

// The evaluation with the bf16x3 engine: thread t owns chain c = t % 32 of each of the NCT tiles and the columns
// k0 = EPT (t / 32) .. of it, whose values stay in registers.
// SPLIT: gridDim.y workgroups share the rows of X; lik_pot and grad_lik then hold each one's partial sums, [gridDim.y]
// times the arrays (lr_eval_sum_kernel adds them), and the first of them writes the prior's.
template <int DP, int NT, int NCT, bool SPLIT = false>
__global__ __launch_bounds__(NT) void lr_eval_bf16_kernel(LrArgs a, const float* __restrict__ theta, int64_t C,
                                                          float* prior_pot, float* lik_pot, float* grad_prior,
                                                          float* grad_lik) {
  const int part = SPLIT ? (int)blockIdx.y : 0, parts = SPLIT ? (int)gridDim.y : 1;
  if constexpr (SPLIT) {
    if (part != 0) prior_pot = grad_prior = nullptr;
    lik_pot += part * C;
    grad_lik += part * C * a.d;
  }
  using E = Bf16Engine<DP, NT, NCT>;
  constexpr int NG = NT / CT, EPT = DP / NG;
  static_assert(NG * EPT == DP && EPT % 4 == 0, "thread ownership");
  __shared__ typename E::Smem es;
  const int t = threadIdx.x, c = t % CT, kg = t / CT, k0 = kg * EPT;
  const int d = a.d;
  const int64_t c0 = (int64_t)blockIdx.x * (NCT * CT);
#pragma unroll
  for (int ct = 0; ct < NCT; ++ct) {
    const int64_t chain = c0 + ct * CT + c;
    float th[EPT];
#pragma unroll
    for (int q = 0; q < EPT; ++q) {
      th[q] = (chain < C && k0 + q < d) ? theta[chain * d + k0 + q] : 0.f;
      if (grad_prior && chain < C && k0 + q < d) grad_prior[chain * d + k0 + q] = a.prior_prec * th[q];
    }
#pragma unroll
    for (int q = 0; q < EPT; q += 4) E::put_theta(es, ct, c, k0 + q, &th[q]);
  }
  __syncthreads();
  typename E::Acc acc;
  if (SPLIT || lik_pot)
    E::template partials<true, SPLIT>(es, a.packed, a.n, acc, part, parts);
  else
    E::template partials<false>(es, a.packed, a.n, acc);
#pragma unroll
  for (int ct = 0; ct < NCT; ++ct) {
    if (ct) __syncthreads();  // the previous tile's partials have been read
    E::put_partials(es, acc, ct);
    __syncthreads();
    const int64_t chain = c0 + ct * CT + c;
#pragma unroll
    for (int q = 0; q < EPT; q += 4) {
      const floatx4 gv = E::gradient(es, c, k0 + q);
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (grad_lik && chain < C && k0 + q + e < d) grad_lik[chain * d + k0 + q + e] = gv[e];
    }
  }
  if (lik_pot && t < NCT * CT && c0 + t < C) lik_pot[c0 + t] = E::potential(es, t);
  if (prior_pot) {
    const int lane = t & (kWave - 1);
    for (int64_t chain = c0 + t / kWave; chain < C && chain < c0 + NCT * CT; chain += E::NW) {
      float s2 = 0.f;
      for (int q = lane; q < d; q += kWave) s2 += theta[chain * d + q] * theta[chain * d + q];
      s2 = wave_sum(s2);
      // prec == 0: improper flat prior, potential 0 (mocat's default uniform prior, core.py:183-189)
      if (lane == 0)
        prior_pot[chain] = a.prior_prec > 0.f
                               ? fmaf(0.5f * (float)d, kLog2Pi - logf(a.prior_prec), 0.5f * a.prior_prec * s2)
                               : 0.f;
    }
  }
}

// The sums of the row parts, in their order.
__global__ __launch_bounds__(256) void lr_eval_sum_kernel(const float* __restrict__ lik, const float* __restrict__ grad,
                                                          int parts, int64_t C, int64_t d, float* lik_pot,
                                                          float* grad_lik) {
  for (int64_t e = blockIdx.x * (int64_t)256 + threadIdx.x; e < C * d; e += (int64_t)gridDim.x * 256) {
    float g = 0.f;
#pragma unroll 8
    for (int p = 0; p < parts; ++p) g += grad[p * C * d + e];
    if (grad_lik) grad_lik[e] = g;
    if (e < C && lik_pot) {
      float l = 0.f;
#pragma unroll 8
      for (int p = 0; p < parts; ++p) l += lik[p * C + e];
      lik_pot[e] = l;
    }
  }
}

// ------------------------------------------------------------------------------------------
struct HmcArgs {
  LrArgs lr;
  int64_t C;
  float* theta;
  float* mom;
  float* grad;
  float* pot;
  float* prior;
  float* lik;
  float* step;
  float* alpha;
  uint32_t* keys;
  int64_t iter0;
  int n_iter;
  int leapfrog_steps;
  float friction;
  int correction;  // 0 none, 1 Metropolis, 2 Robbins-Monro-adapted Metropolis (log update)
  float target;
  float rm_scale, rm_neg_exponent;
  double adapt_cut_off;
  float* tr_value;
  float* tr_pot;
  float* tr_alpha;
  float* tr_step;
  float* tr_mom;
};

template <class Engine, int DP, int NT>
__global__ __launch_bounds__(NT) void hmc_lr_kernel(HmcArgs h) {
  __shared__ TileState<DP> ts;
  __shared__ typename Engine::Smem es;
  const int t = threadIdx.x;
  const int d = h.lr.d;
  const int64_t c0 = (int64_t)blockIdx.x * CT;
  const int nvalid = (int)((h.C - c0) < CT ? (h.C - c0) : CT);

  // load the tile (padding chains are zero and never written back)
  for (int e = t; e < CT * DP; e += NT) {
    const int c = e / DP, k = e - c * DP;
    const bool v = c < nvalid && k < d;
    ts.theta[e] = v ? h.theta[(c0 + c) * d + k] : 0.f;
    ts.mom[e] = v ? h.mom[(c0 + c) * d + k] : 0.f;
    ts.grad[e] = v ? h.grad[(c0 + c) * d + k] : 0.f;
  }
  if (t < CT) {
    const bool v = t < nvalid;
    ts.pot[t] = v ? h.pot[c0 + t] : 0.f;
    ts.prior[t] = v ? h.prior[c0 + t] : 0.f;
    ts.likv[t] = v ? h.lik[c0 + t] : 0.f;
    ts.step[t] = v ? h.step[c0 + t] : 1.f;  // padding chains: finite dummy stepsize
    ts.alpha[t] = v ? h.alpha[c0 + t] : 0.f;
    ts.key[t][0] = v ? h.keys[2 * (c0 + t)] : 0u;
    ts.key[t][1] = v ? h.keys[2 * (c0 + t) + 1] : 0u;
  }
  __syncthreads();

  const uint32_t hd = (uint32_t)(d + 1) >> 1;  // threefry blocks per normal(sub, (d,))
  for (int it = 0; it < h.n_iter; ++it) {
    const int64_t iter = h.iter0 + it + 1;
    // ---- always: p <- -p ; (key, sub) = split(key) ; OU refresh (standard_mcmc.py:107-123)
    __shared__ uint32_t sub[CT][2];
    if (t < CT) {
      Key k{ts.key[t][0], ts.key[t][1]};
      Key nk = split_at(k, 2, 0), sk = split_at(k, 2, 1);
      ts.key[t][0] = nk.a;
      ts.key[t][1] = nk.b;
      sub[t][0] = sk.a;
      sub[t][1] = sk.b;
      // keys = split(key, L+1); key = keys[0] (proposal, standard_mcmc.py:129-131)
      Key pk = split_at(nk, (uint32_t)h.leapfrog_steps + 1u, 0);
      ts.key[t][0] = pk.a;
      ts.key[t][1] = pk.b;
    }
    __syncthreads();
    for (int e = t; e < CT * (int)hd; e += NT) {
      const int c = e / hd;
      const uint32_t i = (uint32_t)(e - c * hd);
      uint32_t w0, w1;
      bits_pair(Key{sub[c][0], sub[c][1]}, (uint32_t)d, i, w0, w1);
      const float hstep = ts.step[c];
      const float decay = __expf(-h.friction * hstep);
      const float noise = sqrtf(1.f - __expf(-2.f * h.friction * hstep));
      float* p = &ts.mom[c * DP];
      p[i] = -p[i] * decay + noise * normal_from_bits(w0);
      if (i + hd < (uint32_t)d) p[i + hd] = -p[i + hd] * decay + noise * normal_from_bits(w1);
    }
    __syncthreads();
    // keep the refreshed momenta for rejection in the global momenta array (position and gradient of
    // the pre-proposal state stay in global memory until a proposal is accepted)
    for (int e = t; e < CT * DP; e += NT) {
      const int c = e / DP, k = e - c * DP;
      if (c < nvalid && k < d) h.mom[(c0 + c) * d + k] = ts.mom[e];
    }
    chain_sqnorm<DP, NT>(ts.mom, d, ts.sq);
    if (t < CT) {
      ts.pot0[t] = ts.pot[t];
      ts.prior0[t] = ts.prior[t];
      ts.lik0[t] = ts.likv[t];
      ts.kin0[t] = 0.5f * ts.sq[t] + 0.5f * (float)d * kLog2Pi;
    }
    // the pre-proposal position/gradient stay in global memory (unchanged until accepted)
    __syncthreads();
    // ---- leapfrog (utils.py:117-146)
    for (int s = 0; s < h.leapfrog_steps; ++s) {
      for (int e = t; e < CT * DP; e += NT) {
        const int c = e / DP;
        const float hh = ts.step[c];
        const float ph = ts.mom[e] - (hh / 2.f) * ts.grad[e];
        ts.mom[e] = ph;
        ts.theta[e] = ((e - c * DP) < d) ? ts.theta[e] + hh * ph : 0.f;
      }
      __syncthreads();
      tile_eval<Engine, DP, NT>(es, ts, h.lr, s == h.leapfrog_steps - 1);
      for (int e = t; e < CT * DP; e += NT) {
        const int c = e / DP;
        ts.mom[e] = ts.mom[e] - (ts.step[c] / 2.f) * ts.grad[e];
      }
      __syncthreads();
    }
    // ---- correction (metropolis.py:48-70, 118-161)
    __shared__ int accept[CT];
    chain_sqnorm<DP, NT>(ts.mom, d, ts.sq);
    if (t < CT) {
      const float kin1 = 0.5f * ts.sq[t] + 0.5f * (float)d * kLog2Pi;  // |-p|^2 == |p|^2
      float a = 1.f;
      int acc = 1;
      if (h.correction > 0) {
        a = fminf(1.f, __expf(-ts.pot[t] + ts.pot0[t] - kin1 + ts.kin0[t]));
        a = isnan(a) ? 0.f : a;
        Key k{ts.key[t][0], ts.key[t][1]};
        Key nk = split_at(k, 2, 0), sk = split_at(k, 2, 1);
        ts.key[t][0] = nk.a;
        ts.key[t][1] = nk.b;
        const float u = uniform_from_bits(bits_at(sk, 1, 0), 0.f, 1.f);
        acc = u < a;
      }
      accept[t] = acc;
      ts.alpha[t] = a;
      if (!acc) {
        ts.pot[t] = ts.pot0[t];
        ts.prior[t] = ts.prior0[t];
        ts.likv[t] = ts.lik0[t];
      }
      if (h.correction == 2 && (double)iter <= h.adapt_cut_off) {
        const float rm = h.rm_scale * powf((float)iter, -h.rm_neg_exponent);
        ts.step[t] = expf(logf(ts.step[t]) + rm * (a - h.target));
      }
    }
    __syncthreads();
    // accepted: momenta <- -p'; rejected: restore position/grad from global, momenta = refreshed
    for (int e = t; e < CT * DP; e += NT) {
      const int c = e / DP, k = e - c * DP;
      if (accept[c]) {
        ts.mom[e] = -ts.mom[e];
        if (c < nvalid && k < d) {
          h.theta[(c0 + c) * d + k] = ts.theta[e];
          h.grad[(c0 + c) * d + k] = ts.grad[e];
        }
      } else {
        ts.mom[e] = (c < nvalid && k < d) ? h.mom[(c0 + c) * d + k] : 0.f;
        if (c < nvalid && k < d) {
          ts.theta[e] = h.theta[(c0 + c) * d + k];
          ts.grad[e] = h.grad[(c0 + c) * d + k];
        } else {
          ts.theta[e] = 0.f;
          ts.grad[e] = 0.f;
        }
      }
      if (c < nvalid && k < d) {
        if (h.tr_value) h.tr_value[((int64_t)it * h.C + c0 + c) * d + k] = ts.theta[e];
        if (h.tr_mom) h.tr_mom[((int64_t)it * h.C + c0 + c) * d + k] = ts.mom[e];
      }
    }
    if (t < nvalid) {
      const int64_t o = (int64_t)it * h.C + c0 + t;
      if (h.tr_pot) h.tr_pot[o] = ts.pot[t];
      if (h.tr_alpha) h.tr_alpha[o] = ts.alpha[t];
      if (h.tr_step) h.tr_step[o] = ts.step[t];
    }
    __syncthreads();
  }
  // write back the final per-chain state
  for (int e = t; e < CT * DP; e += NT) {
    const int c = e / DP, k = e - c * DP;
    if (c < nvalid && k < d) h.mom[(c0 + c) * d + k] = ts.mom[e];
  }
  if (t < nvalid) {
    h.pot[c0 + t] = ts.pot[t];
    h.prior[c0 + t] = ts.prior[t];
    h.lik[c0 + t] = ts.likv[t];
    h.step[c0 + t] = ts.step[t];
    h.alpha[c0 + t] = ts.alpha[t];
    h.keys[2 * (c0 + t)] = ts.key[t][0];
    h.keys[2 * (c0 + t) + 1] = ts.key[t][1];
  }
}

// The iteration for a diagonal Gaussian: LPC lanes per chain, lane q of them with the columns GK q .. GK q + GK - 1 of
// position, momentum and gradient in registers, so that an iteration has neither LDS state nor global traffic (a tile of
// 32 chains in LDS as hmc_lr_kernel keeps took about 25 barriers per iteration: 70 us for 5 moves of 16384 chains
// at d = 20, here 30 us; 219 and 97 us at d = 100). What is left is the vector ALU: threefry and the normals, which the lanes of a chain share
// by blocks of two words and pass on through LDS. Sums over columns keep hmc_lr_kernel's order: the likelihood
// one column after the other, the squared norms by the butterfly of a wave that holds column k in lane k.
constexpr int GK = 8;

// The product alone, never contracted into the sum that takes it.
MOCAT_DEV float product(float a, float b) {
#pragma clang fp contract(off)
  return a * b;
}

template <int LPC>
MOCAT_DEV float gauss_sqnorm(const float (&v)[GK], int q) {
  float a[GK];
#pragma unroll
  for (int j = 0; j < GK; ++j) {
    if constexpr (LPC == 16) {  // columns k and k + 64 are one lane's
      const float o = __shfl_xor(v[j], 8, kWave);
      const float lo = (q & 8) ? o : v[j], hi = (q & 8) ? v[j] : o;
      a[j] = fmaf(hi, hi, product(lo, lo));
    } else {
      a[j] = product(v[j], v[j]);
    }
  }
#pragma unroll
  for (int o = (LPC == 16 ? 8 : LPC) / 2; o > 0; o >>= 1)
#pragma unroll
    for (int j = 0; j < GK; ++j) a[j] += __shfl_xor(a[j], o, kWave);
#pragma unroll
  for (int o = GK / 2; o > 0; o >>= 1)
#pragma unroll
    for (int j = 0; j < o; ++j) a[j] += a[j + o];
  return a[0];
}

// Orders a wave's own LDS writes and reads: a chain's lanes are of one wave.
MOCAT_DEV void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

// Words 0 and 1 of `S` words of key k, each lane of a pair computing one of their two threefry blocks.
template <int LPC>
MOCAT_DEV Key pair_words(Key k, uint32_t S, int q) {
  if constexpr (LPC == 1) {
    return Key{bits_at(k, S, 0), bits_at(k, S, 1)};
  } else {
    const uint32_t w = bits_at(k, S, (uint32_t)(q & 1)), o = __shfl_xor(w, 1, kWave);
    return (q & 1) ? Key{o, w} : Key{w, o};
  }
}

// split(k, 2): four words from two blocks.
template <int LPC>
MOCAT_DEV void pair_split(Key k, int q, Key& first, Key& second) {
  if constexpr (LPC == 1) {
    first = split_at(k, 2, 0);
    second = split_at(k, 2, 1);
  } else {
    uint32_t a, b;
    bits_pair(k, 4u, (uint32_t)(q & 1), a, b);
    const uint32_t oa = __shfl_xor(a, 1, kWave), ob = __shfl_xor(b, 1, kWave);
    first = (q & 1) ? Key{oa, a} : Key{a, oa};
    second = (q & 1) ? Key{ob, b} : Key{b, ob};
  }
}

template <int LPC>
__global__ __launch_bounds__(256) void hmc_gauss_kernel(HmcArgs h) {
  constexpr int NC = 256 / LPC;
  __shared__ float normals[NC][GK * LPC + 1];
  const int t = threadIdx.x, q = t % LPC, c = t / LPC, k0 = q * GK, first = (t & (kWave - 1)) - q;
  const int d = h.lr.d;
  const int64_t chain = (int64_t)blockIdx.x * NC + c;
  const bool live = chain < h.C;
  const float prec = h.lr.prior_prec, temp = h.lr.temperature;
  float th[GK], p[GK], g[GK], mu[GK], lam[GK];
#pragma unroll
  for (int j = 0; j < GK; ++j) {
    const bool v = k0 + j < d;
    mu[j] = v ? h.lr.X[k0 + j] : 0.f;
    lam[j] = v ? h.lr.y[k0 + j] : 0.f;
    th[j] = v && live ? h.theta[chain * d + k0 + j] : 0.f;
    p[j] = v && live ? h.mom[chain * d + k0 + j] : 0.f;
    g[j] = v && live ? h.grad[chain * d + k0 + j] : 0.f;
  }
  float pot = live ? h.pot[chain] : 0.f, prior = live ? h.prior[chain] : 0.f, lik = live ? h.lik[chain] : 0.f;
  float step = live ? h.step[chain] : 1.f, alpha = live ? h.alpha[chain] : 0.f;
  Key key = live ? Key{h.keys[2 * chain], h.keys[2 * chain + 1]} : Key{0u, 0u};
  const uint32_t hd = (uint32_t)(d + 1) >> 1, L1 = (uint32_t)h.leapfrog_steps + 1u;
  for (int it = 0; it < h.n_iter; ++it) {
    const int64_t iter = h.iter0 + it + 1;
    // ---- always: p <- -p ; (key, sub) = split(key) ; OU refresh (standard_mcmc.py:107-123); then the
    // proposal's keys = split(key, L+1), key = keys[0] (standard_mcmc.py:129-131)
    Key nk, sk;
    pair_split<LPC>(key, q, nk, sk);
    key = pair_words<LPC>(nk, 2u * L1, q);
    float u = 0.f;
    if (h.correction > 0) {  // the acceptance's uniform (metropolis.py:60-61)
      Key uk;
      pair_split<LPC>(key, q, nk, uk);
      key = nk;
      u = uniform_from_bits(bits_at(uk, 1, 0), 0.f, 1.f);
    }
#pragma unroll
    for (int j = 0; j < GK / 2; ++j) {
      const uint32_t i = (uint32_t)(j * LPC + q);
      if (j * LPC >= (int)hd) break;
      uint32_t w0, w1;
      bits_pair(sk, (uint32_t)d, i, w0, w1);
      const float z0 = normal_from_bits(w0), z1 = normal_from_bits(w1);
      if (i < hd) normals[c][i] = z0;
      if (i + hd < (uint32_t)d) normals[c][i + hd] = z1;
    }
    wave_sync();
    const float decay = __expf(-h.friction * step);
    const float noise = sqrtf(1.f - __expf(-2.f * h.friction * step));
    float p0[GK], th0[GK], g0[GK];  // the pre-proposal state, for a rejection
#pragma unroll
    for (int j = 0; j < GK; ++j) {
      if (k0 + j < d) p[j] = fmaf(noise, normals[c][k0 + j], -(p[j] * decay));
      p0[j] = p[j];
      th0[j] = th[j];
      g0[j] = g[j];
    }
    wave_sync();  // the normals have been read
    const float kin0 = fmaf(0.5f, gauss_sqnorm<LPC>(p, q), 0.5f * (float)d * kLog2Pi);
    // ---- leapfrog (utils.py:117-146)
    float pot1 = pot, prior1 = prior, lik1 = lik;
    for (int s = 0; s < h.leapfrog_steps; ++s) {
      float cost[GK];
#pragma unroll
      for (int j = 0; j < GK; ++j) {
        p[j] = fmaf(-(step / 2.f), g[j], p[j]);
        th[j] = k0 + j < d ? fmaf(step, p[j], th[j]) : 0.f;
        const float df = th[j] - mu[j];
        cost[j] = product(product(product(0.5f, lam[j]), df), df);
        g[j] = fmaf(prec, th[j], temp * product(lam[j], df));
        p[j] = fmaf(-(step / 2.f), g[j], p[j]);
      }
      if (s == h.leapfrog_steps - 1) {
        lik1 = 0.f;
#pragma unroll
        for (int r = 0; r < LPC; ++r) {
          float acc = lik1;
#pragma unroll
          for (int j = 0; j < GK; ++j) acc += cost[j];  // columns from d on: 0
          lik1 = LPC == 1 ? acc : __shfl(acc, first + r, kWave);
        }
        // prec == 0: improper flat prior, potential 0 (mocat's default uniform prior, core.py:183-189)
        prior1 = prec > 0.f ? fmaf(0.5f * prec, gauss_sqnorm<LPC>(th, q), 0.5f * (float)d * (kLog2Pi - logf(prec))) : 0.f;
        pot1 = fmaf(temp, lik1, prior1);
      }
    }
    // ---- correction (metropolis.py:48-70, 118-161)
    const float kin1 = fmaf(0.5f, gauss_sqnorm<LPC>(p, q), 0.5f * (float)d * kLog2Pi);  // |-p|^2 == |p|^2
    float a = 1.f;
    bool acc = true;
    if (h.correction > 0) {
      a = fminf(1.f, __expf(-pot1 + pot - kin1 + kin0));
      a = isnan(a) ? 0.f : a;
      acc = u < a;
    }
    alpha = a;
    if (acc) {
      pot = pot1;
      prior = prior1;
      lik = lik1;
    }
    if (h.correction == 2 && (double)iter <= h.adapt_cut_off) {
      const float rm = h.rm_scale * powf((float)iter, -h.rm_neg_exponent);
      step = expf(logf(step) + rm * (a - h.target));
    }
    // accepted: momenta <- -p'; rejected: the pre-proposal state
#pragma unroll
    for (int j = 0; j < GK; ++j) {
      p[j] = acc ? -p[j] : p0[j];
      th[j] = acc ? th[j] : th0[j];
      g[j] = acc ? g[j] : g0[j];
    }
    if (live) {
      const int64_t o = (int64_t)it * h.C + chain;
      if (h.tr_value || h.tr_mom)
#pragma unroll
        for (int j = 0; j < GK; ++j)
          if (k0 + j < d) {
            if (h.tr_value) h.tr_value[o * d + k0 + j] = th[j];
            if (h.tr_mom) h.tr_mom[o * d + k0 + j] = p[j];
          }
      if (q == 0) {
        if (h.tr_pot) h.tr_pot[o] = pot;
        if (h.tr_alpha) h.tr_alpha[o] = alpha;
        if (h.tr_step) h.tr_step[o] = step;
      }
    }
  }
  if (!live) return;
#pragma unroll
  for (int j = 0; j < GK; ++j)
    if (k0 + j < d) {
      h.theta[chain * d + k0 + j] = th[j];
      h.mom[chain * d + k0 + j] = p[j];
      h.grad[chain * d + k0 + j] = g[j];
    }
  if (q == 0) {
    h.pot[chain] = pot;
    h.prior[chain] = prior;
    h.lik[chain] = lik;
    h.step[chain] = step;
    h.alpha[chain] = alpha;
    h.keys[2 * chain] = key.a;
    h.keys[2 * chain + 1] = key.b;
  }
}

constexpr int kThreads = 512;

// The same iteration as hmc_lr_kernel for the bf16x3 engine, with the tile state in
// registers: thread t owns, in each of the NCT tiles, chain c = t % 32 and the EPT = DP / (NT / 32) columns
// k0 = EPT * (t / 32) .. of position, momentum and gradient. A leapfrog step is then: update the owned elements
// and write their bf16 hi/lo split into the engine's theta operand (barrier), the engine's block loop (barrier),
// and the owned gradient elements summed from every wave's partials. The refreshed momenta, position
// and gradient of the pre-proposal state stay in global memory until a proposal is accepted (as in
// hmc_lr_kernel); per-chain scalars and keys live in LDS and in the first NCT * 32 threads.
template <int DP, int NT, int NCT>
__global__ __launch_bounds__(NT) void hmc_lr_bf16_kernel(HmcArgs h) {
  using E = Bf16Engine<DP, NT, NCT>;
  constexpr int NG = NT / CT;  // column groups
  constexpr int EPT = DP / NG;
  constexpr int NC = NCT * CT;  // chains of the workgroup
  static_assert(NG * EPT == DP && EPT % 4 == 0 && NC <= NT, "thread ownership");
  __shared__ typename E::Smem es;
  __shared__ float sq0[NG][NC], sq1[NG][NC], sqt[NG][NC];
  __shared__ float step[NC], pot[NC], prior[NC], likv[NC], alpha[NC];
  __shared__ uint32_t sub[NC][2];
  __shared__ int accept[NC];
  const int t = threadIdx.x, c = t % CT, kg = t / CT, k0 = kg * EPT;
  const int d = h.lr.d;
  const int64_t c0 = (int64_t)blockIdx.x * NC;
  const int nvalid = (int)((h.C - c0) < NC ? (h.C - c0) : NC);
  const float prec = h.lr.prior_prec, temp = h.lr.temperature;
  auto valid = [&](int ct) { return ct * CT + c < nvalid; };
  auto row = [&](int ct) { return (c0 + ct * CT + c) * (int64_t)d; };

  float th[NCT][EPT], p[NCT][EPT], g[NCT][EPT];
#pragma unroll
  for (int ct = 0; ct < NCT; ++ct)
#pragma unroll
    for (int q = 0; q < EPT; ++q) {
      const int k = k0 + q;
      const bool v = valid(ct) && k < d;
      th[ct][q] = v ? h.theta[row(ct) + k] : 0.f;
      p[ct][q] = v ? h.mom[row(ct) + k] : 0.f;
      g[ct][q] = v ? h.grad[row(ct) + k] : 0.f;
    }
  Key key{0u, 0u};
  if (t < NC) {
    const bool v = t < nvalid;
    pot[t] = v ? h.pot[c0 + t] : 0.f;
    prior[t] = v ? h.prior[c0 + t] : 0.f;
    likv[t] = v ? h.lik[c0 + t] : 0.f;
    step[t] = v ? h.step[c0 + t] : 1.f;  // padding chains: finite dummy stepsize
    alpha[t] = v ? h.alpha[c0 + t] : 0.f;
    key = v ? Key{h.keys[2 * (c0 + t)], h.keys[2 * (c0 + t) + 1]} : Key{0u, 0u};
  }
  const uint32_t L1 = (uint32_t)h.leapfrog_steps + 1u;
  for (int it = 0; it < h.n_iter; ++it) {
    const int64_t iter = h.iter0 + it + 1;
    // ---- always: p <- -p ; (key, sub) = split(key) ; OU refresh (standard_mcmc.py:107-123); then the
    // proposal's keys = split(key, L+1), key = keys[0] (standard_mcmc.py:129-131)
    float pot0 = 0.f, prior0 = 0.f, lik0 = 0.f;
    if (t < NC) {
      const Key nk = split_at(key, 2, 0), sk = split_at(key, 2, 1);
      sub[t][0] = sk.a;
      sub[t][1] = sk.b;
      key = split_at(nk, L1, 0);
      pot0 = pot[t];
      prior0 = prior[t];
      lik0 = likv[t];
    }
    __syncthreads();
    float hh[NCT];
#pragma unroll
    for (int ct = 0; ct < NCT; ++ct) {
      hh[ct] = step[ct * CT + c];
      const float decay = __expf(-h.friction * hh[ct]);
      const float noise = sqrtf(1.f - __expf(-2.f * h.friction * hh[ct]));
      const Key sk{sub[ct * CT + c][0], sub[ct * CT + c][1]};
      float s2 = 0.f;
#pragma unroll
      for (int q = 0; q < EPT; ++q) {
        const int k = k0 + q;
        if (k < d) {
          p[ct][q] = -p[ct][q] * decay + noise * normal_from_bits(bits_at(sk, (uint32_t)d, (uint32_t)k));
          if (valid(ct)) h.mom[row(ct) + k] = p[ct][q];  // the refreshed momenta, kept for a rejection
        }
        s2 += p[ct][q] * p[ct][q];
      }
      sq0[kg][ct * CT + c] = s2;
    }
    // ---- leapfrog (utils.py:117-146)
    for (int s = 0; s < h.leapfrog_steps; ++s) {
      const bool last = s == h.leapfrog_steps - 1;
#pragma unroll
      for (int ct = 0; ct < NCT; ++ct) {
        float s2 = 0.f;
#pragma unroll
        for (int q = 0; q < EPT; ++q) {
          const float ph = p[ct][q] - (hh[ct] / 2.f) * g[ct][q];
          p[ct][q] = ph;
          th[ct][q] = (k0 + q < d) ? th[ct][q] + hh[ct] * ph : 0.f;
          s2 += th[ct][q] * th[ct][q];
        }
        if (last) sqt[kg][ct * CT + c] = s2;
#pragma unroll
        for (int q = 0; q < EPT; q += 4) E::put_theta(es, ct, c, k0 + q, &th[ct][q]);
      }
      __syncthreads();
      typename E::Acc acc;
      if (last)
        E::template partials<true>(es, h.lr.packed, h.lr.n, acc);
      else
        E::template partials<false>(es, h.lr.packed, h.lr.n, acc);
#pragma unroll
      for (int ct = 0; ct < NCT; ++ct) {
        if (ct) __syncthreads();  // the previous tile's partials have been read
        E::put_partials(es, acc, ct);
        __syncthreads();
#pragma unroll
        for (int q = 0; q < EPT; q += 4) {
          const floatx4 gv = E::gradient(es, c, k0 + q);
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            // explicit, so that every tile count contracts it alike
            g[ct][q + e] = fmaf(temp, gv[e], prec * th[ct][q + e]);
            p[ct][q + e] = p[ct][q + e] - (hh[ct] / 2.f) * g[ct][q + e];
          }
        }
      }
      if (last && t < NC) {
        const float lk = E::potential(es, t);
        float st = 0.f;
        for (int q = 0; q < NG; ++q) st += sqt[q][t];
        // prec == 0: improper flat prior, potential 0 (mocat's default uniform prior, core.py:183-189)
        const float pr = prec > 0.f ? 0.5f * prec * st + 0.5f * (float)d * (kLog2Pi - logf(prec)) : 0.f;
        prior[t] = pr;
        likv[t] = lk;
        pot[t] = pr + temp * lk;
      }
      if (NCT > 1 && !last) __syncthreads();  // the last tile's partials have been read before the next step's
    }
#pragma unroll
    for (int ct = 0; ct < NCT; ++ct) {
      float s2 = 0.f;
#pragma unroll
      for (int q = 0; q < EPT; ++q) s2 += p[ct][q] * p[ct][q];
      sq1[kg][ct * CT + c] = s2;
    }
    __syncthreads();
    // ---- correction (metropolis.py:48-70, 118-161)
    if (t < NC) {
      float k0s = 0.f, k1s = 0.f;
      for (int q = 0; q < NG; ++q) {
        k0s += sq0[q][t];
        k1s += sq1[q][t];
      }
      const float kin0 = 0.5f * k0s + 0.5f * (float)d * kLog2Pi;
      const float kin1 = 0.5f * k1s + 0.5f * (float)d * kLog2Pi;  // |-p|^2 == |p|^2
      float a = 1.f;
      int acc = 1;
      if (h.correction > 0) {
        a = fminf(1.f, __expf(-pot[t] + pot0 - kin1 + kin0));
        a = isnan(a) ? 0.f : a;
        const Key nk = split_at(key, 2, 0), sk = split_at(key, 2, 1);
        key = nk;
        const float u = uniform_from_bits(bits_at(sk, 1, 0), 0.f, 1.f);
        acc = u < a;
      }
      accept[t] = acc;
      alpha[t] = a;
      if (!acc) {
        pot[t] = pot0;
        prior[t] = prior0;
        likv[t] = lik0;
      }
      if (h.correction == 2 && (double)iter <= h.adapt_cut_off) {
        const float rm = h.rm_scale * powf((float)iter, -h.rm_neg_exponent);
        step[t] = expf(logf(step[t]) + rm * (a - h.target));
      }
    }
    __syncthreads();
    // accepted: momenta <- -p' and the proposal is stored; rejected: the pre-proposal state is read back
#pragma unroll
    for (int ct = 0; ct < NCT; ++ct) {
      const bool acc = accept[ct * CT + c] != 0;
#pragma unroll
      for (int q = 0; q < EPT; ++q) {
        const int k = k0 + q;
        const bool v = valid(ct) && k < d;
        if (acc) {
          p[ct][q] = -p[ct][q];
          if (v) {
            h.theta[row(ct) + k] = th[ct][q];
            h.grad[row(ct) + k] = g[ct][q];
          }
        } else {
          p[ct][q] = v ? h.mom[row(ct) + k] : 0.f;
          th[ct][q] = v ? h.theta[row(ct) + k] : 0.f;
          g[ct][q] = v ? h.grad[row(ct) + k] : 0.f;
        }
        if (v) {
          const int64_t o = ((int64_t)it * h.C + c0 + ct * CT + c) * d + k;
          if (h.tr_value) h.tr_value[o] = th[ct][q];
          if (h.tr_mom) h.tr_mom[o] = p[ct][q];
        }
      }
    }
    if (t < nvalid) {
      const int64_t o = (int64_t)it * h.C + c0 + t;
      if (h.tr_pot) h.tr_pot[o] = pot[t];
      if (h.tr_alpha) h.tr_alpha[o] = alpha[t];
      if (h.tr_step) h.tr_step[o] = step[t];
    }
  }
  // write back the final per-chain state (position and gradient are already in place)
#pragma unroll
  for (int ct = 0; ct < NCT; ++ct)
#pragma unroll
    for (int q = 0; q < EPT; ++q)
      if (valid(ct) && k0 + q < d) h.mom[row(ct) + k0 + q] = p[ct][q];
  if (t < nvalid) {
    h.pot[c0 + t] = pot[t];
    h.prior[c0 + t] = prior[t];
    h.lik[c0 + t] = likv[t];
    h.step[c0 + t] = step[t];
    h.alpha[c0 + t] = alpha[t];
    h.keys[2 * (c0 + t)] = key.a;
    h.keys[2 * (c0 + t) + 1] = key.b;
  }
}

template <template <int, int> class E>
int dispatch_eval(const LrArgs& a, const float* theta, int64_t C, float* pp, float* lp, float* gp, float* gl,
                  hipStream_t st) {
  const unsigned blocks = (unsigned)((C + CT - 1) / CT);
  if (a.d <= 64)
    hipLaunchKernelGGL((lr_eval_kernel<E<64, kThreads>, 64, kThreads>), dim3(blocks), dim3(kThreads), 0, st, a,
                       theta, C, pp, lp, gp, gl, 0);
  else
    hipLaunchKernelGGL((lr_eval_kernel<E<128, kThreads>, 128, kThreads>), dim3(blocks), dim3(kThreads), 0, st, a,
                       theta, C, pp, lp, gp, gl, 0);
  MOCAT_LAUNCH_CHECK();
  return MOCAT_OK;
}

template <template <int, int> class E>
int dispatch_hmc(const HmcArgs& h, hipStream_t st) {
  const unsigned blocks = (unsigned)((h.C + CT - 1) / CT);
  if (h.lr.d <= 64)
    hipLaunchKernelGGL((hmc_lr_kernel<E<64, kThreads>, 64, kThreads>), dim3(blocks), dim3(kThreads), 0, st, h);
  else
    hipLaunchKernelGGL((hmc_lr_kernel<E<128, kThreads>, 128, kThreads>), dim3(blocks), dim3(kThreads), 0, st, h);
  MOCAT_LAUNCH_CHECK();
  return MOCAT_OK;
}

template <int LPC>
void launch_gauss(const HmcArgs& h, hipStream_t st) {
  const int64_t per = 256 / LPC;
  hipLaunchKernelGGL((hmc_gauss_kernel<LPC>), dim3((unsigned)((h.C + per - 1) / per)), dim3(256), 0, st, h);
}

int dispatch_hmc_gauss(const HmcArgs& h, hipStream_t st) {
  if (h.lr.d <= GK)
    launch_gauss<1>(h, st);
  else if (h.lr.d <= 2 * GK)
    launch_gauss<2>(h, st);
  else if (h.lr.d <= 4 * GK)
    launch_gauss<4>(h, st);
  else if (h.lr.d <= 8 * GK)
    launch_gauss<8>(h, st);
  else
    launch_gauss<16>(h, st);
  MOCAT_LAUNCH_CHECK();
  return MOCAT_OK;
}

// bf16x3: two waves per SIMD at d <= 64; at d <= 128 one wave per SIMD (the operand registers of a
// 128-column block, and the LDS of eight waves' partial gradients, do not fit two waves). Two tiles of
// chains per workgroup from kTwoTiles chains (a workgroup for each of 256 CUs): X 20000 x 100, 65536 positions,
// potential and gradient 2107 -> 1697 us, one MALA move 2141 -> 1860; X 2000 x 50, 32768 positions 89 -> 70.
constexpr int kBf16Threads64 = 512, kBf16Threads128 = 256;
constexpr int64_t kTwoTiles = 256 * 2 * CT;

unsigned tiles(int64_t C, int nct) { return (unsigned)((C + nct * CT - 1) / (nct * CT)); }

template <int DP>
int launch_eval_bf16(const LrArgs& a, const float* theta, int64_t C, float* pp, float* lp, float* gp, float* gl,
                     hipStream_t st) {
  constexpr int NT = DP == 64 ? kBf16Threads64 : kBf16Threads128;
  if (C < kTwoTiles)
    hipLaunchKernelGGL((lr_eval_bf16_kernel<DP, NT, 1>), dim3(tiles(C, 1)), dim3(NT), 0, st, a, theta, C, pp, lp, gp, gl);
  else
    hipLaunchKernelGGL((lr_eval_bf16_kernel<DP, NT, 2>), dim3(tiles(C, 2)), dim3(NT), 0, st, a, theta, C, pp, lp, gp, gl);
  MOCAT_LAUNCH_CHECK();
  return MOCAT_OK;
}

// Parts the rows of X are split into for C points: few points (one workgroup per 32 of them) leave the other CUs idle. At
// least four 32-row blocks per wave are left, and nothing is split below twelve, where the second launch costs
// more than it saves. A call unsplit / split, us: X 1505x100, 40 points 26.5 / 20.2, 4096 points 29.5 / 27.0; X 3100x64, 40
// points 26.9 / 18.6; X 20000x100, 1 point 254 / 19, 1024 259 / 56, 4096 263 / 159 (about 15 us of each is the host's).
// FP32: blocks of 64 rows, from four on: X 193x64, 1 point 21.1 / 19.9, 285x100 41 / 20, 1390x100 166 / 20, 20000x100 3060 / 85; 4096
// points 37 / 28 (193x100), 172 / 98 (1390x100), 3008 / 1520 (20000x100).
constexpr int kMaxParts = 32, kFp32Rows = 64;
int eval_parts(int precision, int64_t n, int64_t d, int64_t C) {
  const int64_t tile = (C + CT - 1) / CT;
  if (tile < 1 || tile > 128) return 1;
  const int64_t most = std::min<int64_t>(kMaxParts, 256 / tile);
  if (precision == 0) {
    const int64_t blocks = (n + kFp32Rows - 1) / kFp32Rows;
    if (blocks < 4) return 1;
    const int64_t per = (blocks + most - 1) / most;
    return (int)((blocks + per - 1) / per);
  }
  if (precision != 1) return 1;
  const int64_t nw = (d <= 64 ? kBf16Threads64 : kBf16Threads128) / kWave, nrb = (n + 31) / 32;
  return nrb < 12 * nw ? 1 : (int)std::min<int64_t>(most, nrb / (4 * nw));
}

template <int DP>
int launch_eval_split(const LrArgs& a, int precision, const float* theta, int64_t C, int parts, float* ws, float* pp,
                      float* lp, float* gp, float* gl, hipStream_t st) {
  constexpr int NT = DP == 64 ? kBf16Threads64 : kBf16Threads128;
  float *lik = ws, *grad = ws + parts * C;
  if (precision == 0) {
    const int blocks = (a.n + kFp32Rows - 1) / kFp32Rows, rows = (blocks + parts - 1) / parts * kFp32Rows;
    hipLaunchKernelGGL((lr_eval_kernel<Fp32Engine<DP, kThreads>, DP, kThreads, true>), dim3(tiles(C, 1), parts),
                       dim3(kThreads), 0, st, a, theta, C, pp, lik, gp, grad, rows);
  } else {
    hipLaunchKernelGGL((lr_eval_bf16_kernel<DP, NT, 1, true>), dim3(tiles(C, 1), parts), dim3(NT), 0, st, a, theta, C, pp,
                       lik, gp, grad);
  }
  const int64_t blocks = (C * a.d + 255) / 256;
  hipLaunchKernelGGL(lr_eval_sum_kernel, dim3((unsigned)std::min<int64_t>(blocks, 65535)), dim3(256), 0, st, (const float*)lik,
                     (const float*)grad, parts, C, (int64_t)a.d, lp, gl);
  MOCAT_LAUNCH_CHECK();
  return MOCAT_OK;
}

int dispatch_eval_bf16(const LrArgs& a, const float* theta, int64_t C, float* pp, float* lp, float* gp, float* gl,
                       hipStream_t st) {
  return a.d <= 64 ? launch_eval_bf16<64>(a, theta, C, pp, lp, gp, gl, st)
                   : launch_eval_bf16<128>(a, theta, C, pp, lp, gp, gl, st);
}

int dispatch_hmc_bf16(const HmcArgs& h, hipStream_t st) {
  if (h.lr.d <= 64)  // two tiles' chain state does not fit two waves per SIMD (spilled: 576 against 518 us)
    hipLaunchKernelGGL((hmc_lr_bf16_kernel<64, kBf16Threads64, 1>), dim3(tiles(h.C, 1)), dim3(kBf16Threads64), 0, st, h);
  else if (h.C < kTwoTiles)
    hipLaunchKernelGGL((hmc_lr_bf16_kernel<128, kBf16Threads128, 1>), dim3(tiles(h.C, 1)), dim3(kBf16Threads128), 0, st,
                       h);
  else
    hipLaunchKernelGGL((hmc_lr_bf16_kernel<128, kBf16Threads128, 2>), dim3(tiles(h.C, 2)), dim3(kBf16Threads128), 0, st,
                       h);
  MOCAT_LAUNCH_CHECK();
  return MOCAT_OK;
}

int check_lr(const float* X, const float* y, const void* packed, int64_t n, int64_t d, int precision) {
  if (n <= 0 || d <= 0 || d > 128 || n > (1ll << 30)) return MOCAT_ERR_ARG;
  if (precision == 0 || precision == 2 || precision == 3) return (X && y) ? MOCAT_OK : MOCAT_ERR_ARG;
  if (precision == 1) return packed ? MOCAT_OK : MOCAT_ERR_ARG;
  return MOCAT_ERR_ARG;
}

}  // namespace

extern "C" {

int mocat_lr_packed_bytes(int64_t n, int64_t d, int64_t* bytes) {
  if (n <= 0 || d <= 0 || d > 128 || !bytes) return MOCAT_ERR_ARG;
  const int64_t nrb = (n + 31) / 32;
  *bytes = nrb * (d <= 64 ? PackLayout<64>::BLOCK_BYTES : PackLayout<128>::BLOCK_BYTES);
  return MOCAT_OK;
}

int mocat_lr_pack(const float* X, const float* y, int64_t n, int64_t d, void* packed, hipStream_t stream) {
  if (!X || !y || !packed || n <= 0 || d <= 0 || d > 128 || n > (1ll << 30)) return MOCAT_ERR_ARG;
  const int64_t nrb = (n + 31) / 32;
  const int threads = 256;
  if (d <= 64) {
    const int64_t total = nrb * (PackLayout<64>::BLOCK_BF16 + 32);
    const unsigned blocks = (unsigned)std::min<int64_t>((total + threads - 1) / threads, 65535);
    hipLaunchKernelGGL(lr_pack_kernel<64>, dim3(blocks), dim3(threads), 0, stream, X, y, (int)n, (int)d,
                       (char*)packed);
  } else {
    const int64_t total = nrb * (PackLayout<128>::BLOCK_BF16 + 32);
    const unsigned blocks = (unsigned)std::min<int64_t>((total + threads - 1) / threads, 65535);
    hipLaunchKernelGGL(lr_pack_kernel<128>, dim3(blocks), dim3(threads), 0, stream, X, y, (int)n, (int)d,
                       (char*)packed);
  }
  MOCAT_LAUNCH_CHECK();
  return MOCAT_OK;
}

int mocat_lr_potential_grad(const float* X, const float* y, const void* packed, int64_t n, int64_t d, int precision,
                            float prior_prec, float temperature, const float* theta, int64_t C, float* prior_pot,
                            float* lik_pot, float* grad_prior, float* grad_lik, hipStream_t stream) {
  int rc = check_lr(X, y, packed, n, d, precision);
  if (rc) return rc;
  if (C < 0 || (C > 0 && !theta)) return MOCAT_ERR_ARG;
  if (C == 0) return MOCAT_OK;
  LrArgs a{X, y, packed, (int)n, (int)d, prior_prec, temperature};
  if (precision == 2)
    return dispatch_eval<GaussEngine>(a, theta, C, prior_pot, lik_pot, grad_prior, grad_lik, stream);
  if (precision == 3)
    return dispatch_eval<Fp64Engine>(a, theta, C, prior_pot, lik_pot, grad_prior, grad_lik, stream);
  return precision == 0 ? dispatch_eval<Fp32Engine>(a, theta, C, prior_pot, lik_pot, grad_prior, grad_lik, stream)
                        : dispatch_eval_bf16(a, theta, C, prior_pot, lik_pot, grad_prior, grad_lik, stream);
}

int mocat_lr_eval_workspace_bytes(int64_t n, int64_t d, int precision, int64_t C, int64_t* bytes) {
  if (!bytes || n <= 0 || d <= 0 || d > 128 || C < 0) return MOCAT_ERR_ARG;
  const int parts = eval_parts(precision, n, d, C);
  *bytes = parts > 1 ? parts * C * (d + 1) * (int64_t)sizeof(float) : 0;
  return MOCAT_OK;
}

int mocat_lr_potential_grad_split(const float* X, const float* y, const void* packed, int64_t n, int64_t d, int precision,
                                  float prior_prec, float temperature, const float* theta, int64_t C, float* prior_pot,
                                  float* lik_pot, float* grad_prior, float* grad_lik, void* workspace,
                                  int64_t workspace_bytes, hipStream_t stream) {
  int rc = check_lr(X, y, packed, n, d, precision);
  if (rc) return rc;
  if (C < 0 || (C > 0 && !theta)) return MOCAT_ERR_ARG;
  int64_t need = 0;
  rc = mocat_lr_eval_workspace_bytes(n, d, precision, C, &need);
  if (rc) return rc;
  if (need == 0)
    return mocat_lr_potential_grad(X, y, packed, n, d, precision, prior_prec, temperature, theta, C, prior_pot, lik_pot,
                                   grad_prior, grad_lik, stream);
  if (!workspace || workspace_bytes < need) return MOCAT_ERR_SIZE;
  LrArgs a{X, y, packed, (int)n, (int)d, prior_prec, temperature};
  const int parts = eval_parts(precision, n, d, C);
  float* ws = static_cast<float*>(workspace);
  return d <= 64 ? launch_eval_split<64>(a, precision, theta, C, parts, ws, prior_pot, lik_pot, grad_prior, grad_lik, stream)
                 : launch_eval_split<128>(a, precision, theta, C, parts, ws, prior_pot, lik_pot, grad_prior, grad_lik, stream);
}

int mocat_hmc_lr_iterate(const float* X, const float* y, const void* packed, int64_t n, int64_t d, int precision,
                         float prior_prec, float temperature, int64_t C, float* theta, float* momenta, float* grad,
                         float* potential, float* prior_pot, float* lik_pot, float* stepsize, float* alpha,
                         uint32_t* keys, int64_t iter0, int n_iter, int leapfrog_steps, float friction,
                         int correction, float target, float rm_scale, float rm_neg_exponent, double adapt_cut_off,
                         float* trace_value, float* trace_potential, float* trace_alpha, float* trace_stepsize,
                         float* trace_momenta, hipStream_t stream) {
  int rc = check_lr(X, y, packed, n, d, precision);
  if (rc) return rc;
  if (C < 0 || n_iter < 0 || leapfrog_steps < 1 || correction < 0 || correction > 2) return MOCAT_ERR_ARG;
  if (C == 0 || n_iter == 0) return MOCAT_OK;
  if (!theta || !momenta || !grad || !potential || !prior_pot || !lik_pot || !stepsize || !alpha || !keys)
    return MOCAT_ERR_ARG;
  HmcArgs h{{X, y, packed, (int)n, (int)d, prior_prec, temperature},
            C, theta, momenta, grad, potential, prior_pot, lik_pot, stepsize, alpha, keys, iter0, n_iter,
            leapfrog_steps, friction, correction, target, rm_scale, rm_neg_exponent, adapt_cut_off,
            trace_value, trace_potential, trace_alpha, trace_stepsize, trace_momenta};
  if (precision == 2) return dispatch_hmc_gauss(h, stream);
  if (precision == 3) return dispatch_hmc<Fp64Engine>(h, stream);
  return precision == 0 ? dispatch_hmc<Fp32Engine>(h, stream) : dispatch_hmc_bf16(h, stream);
}

}  // extern "C"
