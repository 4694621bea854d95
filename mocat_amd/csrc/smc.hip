// Tempered SMC sampler pieces (mocat/src/transport/smc.py):
//   gather_rows   resampled_ensemble_state = ensemble_state[resampled_indices] (smc.py:61-71)
//   smc_temper    FP64, one workgroup or several:
//     next temperature by mocat's regula falsi ("bisect", mocat/src/utils.py:205-237) on
//       f(b) = log_ess(lw - (b - b_t) lik) - log(ess_t * retain)   (smc.py:303-326)
//     or a fixed next temperature (temperature_schedule);
//     reweight lw_new = lw - (b' - b_t) lik (MetropolisedSMCSampler.log_weight, smc.py:367-373),
//     ESS and the log-normaliser increment lse(lw_new) - lse(lw) (TemperedSMCSampler.adapt,
//     smc.py:193-217), and the Robbins-Monro stepsize step with the weighted mean acceptance
//     (RMMetropolisedSMCSampler.adapt, smc.py:406-421).
//   smc_resample, smc_move   the launches of one temperature before and after the evaluation at the
//     resampled particles (smc.py:73-99), a call each: with a call per kernel and elementwise step the host's
//     work and the elementwise launches were 2.4 of 5.8 ms (16384 particles, 20 dimensions, 13 temperatures).
#include "common.hpp"
#include "../../include/mocat_amd.h"

using namespace mocat;

namespace {

__global__ __launch_bounds__(256) void gather_kernel(const uint32_t* __restrict__ src, const int32_t* __restrict__ idx,
                                                     int64_t n_out, int64_t width, uint32_t* __restrict__ dst) {
  const int64_t total = n_out * width;
  for (int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; e < total; e += (int64_t)gridDim.x * blockDim.x) {
    const int64_t j = e / width, k = e - j * width;
    dst[e] = src[(int64_t)idx[j] * width + k];
  }
}

struct TemperArgs {
  const float* lw;        // [n] current (resampled) log weights
  const float* lik;       // [n] likelihood potentials of the moved particles
  int64_t n;
  double beta;            // current temperature b_t
  double ess;             // ESS of lw (n after a resample)
  double retain;          // ess_threshold_retain
  double max_temperature;
  double tol;
  int max_iter;
  int adaptive;           // 1: regula falsi, 0: fixed next temperature `next_beta`
  double next_beta;
  const float* alpha;     // [k_alpha][n] acceptance probabilities of the moves, or NULL
  int k_alpha;
  double log_stepsize;    // current log stepsize
  double rm_stepsize;     // 0: no RM update
  double target;
  float* lw_out;          // [n]
  double* out;            // [8]: beta_new, ess_new, lse_new, lse_prev, log_stepsize_new, alpha_mean, iters, f_min
};

// The particles of one workgroup: i = (k * G + g) * NT + t for workgroup g of G. The first kRegs per
// thread are read once and kept in registers over all evaluations, any others are read again each time.
constexpr int kRegs = 4;
template <int NT, bool ALPHA>
struct Share {
  int64_t n, stride, first;  // stride = G * NT
  const float *lw, *lik, *alpha;
  int k_alpha;
  float rl[kRegs], rk[kRegs];
  double ra[ALPHA ? kRegs : 1];  // mean acceptance probability of the moves
  MOCAT_DEV Share(const TemperArgs& a)
      : n(a.n), stride((int64_t)gridDim.x * NT), first((int64_t)blockIdx.x * NT + threadIdx.x), lw(a.lw), lik(a.lik),
        alpha(a.alpha), k_alpha(a.alpha ? a.k_alpha : 0) {
#pragma unroll
    for (int k = 0; k < kRegs; ++k) {
      const int64_t i = first + k * stride;
      rl[k] = i < n ? lw[i] : 0.f;
      rk[k] = i < n ? lik[i] : 0.f;
      if constexpr (ALPHA) ra[k] = i < n ? mean_alpha(i) : 0.0;
    }
  }
  MOCAT_DEV double mean_alpha(int64_t i) const {
    double am = 0.0;
    for (int j = 0; j < k_alpha; ++j) am += (double)alpha[(int64_t)j * n + i];
    return k_alpha > 0 ? am / (double)k_alpha : 0.0;
  }
  template <class F>
  MOCAT_DEV void each(F f) const {  // f(i, log weight, likelihood potential)
#pragma unroll
    for (int k = 0; k < kRegs; ++k) {
      const int64_t i = first + k * stride;
      if (i < n) f(i, rl[k], rk[k]);
    }
#pragma unroll 4
    for (int64_t i = first + kRegs * stride; i < n; i += stride) f(i, lw[i], lik[i]);
  }
  // s += (e, e^2, with ALPHA e * mean acceptance), e = exp(lw - db * lik - ref)
  MOCAT_DEV void sums(double db, double ref, double s[3]) const {
    auto add = [&](float l, float k, double am) {
      const double e = exp((double)l - db * (double)k - ref);
      s[0] += e;
      s[1] += e * e;
      if constexpr (ALPHA) s[2] += e * am;
    };
#pragma unroll
    for (int k = 0; k < kRegs; ++k)
      if (first + k * stride < n) add(rl[k], rk[k], ALPHA ? ra[k] : 0.0);
#pragma unroll 4
    for (int64_t i = first + kRegs * stride; i < n; i += stride) add(lw[i], lik[i], ALPHA ? mean_alpha(i) : 0.0);
  }
};

// Workgroups of a split evaluation, and what they exchange: two sets of slots used in turn, so that a
// workgroup that is one exchange ahead never overwrites what another still reads, and the barrier's
// arrival count and abort flag. A workgroup that polls max_polls times without seeing every arrival sets
// the flag and leaves, as does every workgroup that sees it; temper_kernel<false> then does the work.
// Slots are written and read by agent-scope atomics, which pass the caches: no cache is written back or
// dropped for them.
constexpr int kSlots = 10;
constexpr int kMaxSplit = 128;
struct TemperWs {
  double slot[2][kMaxSplit][kSlots];
  uint32_t bar[2];
};
struct Exchange {
  TemperWs* ws;
  uint32_t max_polls, count;

  // Wave 0: publishes this workgroup's values (the same in every lane), waits for all of them.
  template <int NV>
  MOCAT_DEV bool run(const double (&v)[NV]) {
    static_assert(NV <= kSlots, "a slot holds the values");
    const int par = count & 1;
    ++count;
    int ok = 1;
    if (threadIdx.x == 0) {
#pragma unroll
      for (int k = 0; k < NV; ++k)
        __hip_atomic_store(&ws->slot[par][blockIdx.x][k], v[k], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the values have arrived before the count does
      __hip_atomic_fetch_add(&ws->bar[0], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      const uint32_t target = count * gridDim.x;
      for (uint32_t polls = 0;; ++polls) {
        if (polls >= max_polls) {
          __hip_atomic_store(&ws->bar[1], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
          ok = 0;
          break;
        }
        if (__hip_atomic_load(&ws->bar[0], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) >= target) break;
        if ((polls & 63u) == 63u && __hip_atomic_load(&ws->bar[1], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0u) {
          ok = 0;
          break;
        }
      }
      asm volatile("" ::: "memory");
    }
    return __shfl(ok, 0, kWave) != 0;
  }
  MOCAT_DEV double get(int g, int k) const {
    return __hip_atomic_load(&ws->slot[(count - 1) & 1][g][k], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
};

struct Eval {
  double lse, lse2, am;  // lse(w), lse(2w), weighted mean acceptance
};

template <bool SPLIT>
struct Temper {
  static constexpr int NT = SPLIT ? 256 : 512, NW = NT / kWave;
  using Particles = Share<NT, SPLIT>;
  struct Smem {
    double red[6][NW];
    double mx[2][NW];
    double bc[8];
    int nan[2][NW];
    int ok;
  };

  // w_i = lw_i - db * lik_i at db = 0 and db = db1 together, FP64: the maxima, then sums of exp(w_i - max).
  // Partial sums are combined in a fixed order (lanes by butterfly, waves in index order, workgroups by lane and
  // butterfly after scaling to the common maximum), so that every workgroup finds the same values and takes the
  // same decisions. false: the exchange was given up.
  static MOCAT_DEV bool ends(const Particles& sh, double db1, Exchange& ex, Smem& s, Eval& e0, Eval& e1) {
    const int t = threadIdx.x, lane = t & (kWave - 1), w = t / kWave;
    const double db[2] = {0.0, db1};
    double mx[2] = {-INFINITY, -INFINITY};
    int bad[2] = {0, 0};
    sh.each([&](int64_t, float l, float k) {
#pragma unroll
      for (int q = 0; q < 2; ++q) {
        const double v = (double)l - db[q] * (double)k;
        if (isnan(v)) bad[q] = 1;
        else mx[q] = fmax(mx[q], v);
      }
    });
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      mx[q] = wave_max(mx[q]);
      const int any = __any(bad[q]);
      if (lane == 0) {
        s.mx[q][w] = mx[q];
        s.nan[q][w] = any;
      }
    }
    __syncthreads();
    double p[6] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      mx[q] = s.mx[q][0];
      bad[q] = s.nan[q][0];
      for (int i = 1; i < NW; ++i) {
        mx[q] = fmax(mx[q], s.mx[q][i]);
        bad[q] |= s.nan[q][i];
      }
      if (!bad[q] && mx[q] != -INFINITY) sh.sums(db[q], mx[q], p + 3 * q);
    }
#pragma unroll
    for (int k = 0; k < 6; ++k) {
      p[k] = wave_sum(p[k]);
      if (lane == 0) s.red[k][w] = p[k];
    }
    __syncthreads();
    if (w == 0) {
#pragma unroll
      for (int k = 0; k < 6; ++k) {
        p[k] = s.red[k][0];
        for (int i = 1; i < NW; ++i) p[k] += s.red[k][i];
      }
      bool ok = true;
      if constexpr (SPLIT) {
        const double v[kSlots] = {mx[0], mx[1], bad[0] ? 1.0 : 0.0, bad[1] ? 1.0 : 0.0, p[0], p[1], p[2], p[3], p[4], p[5]};
        ok = ex.run(v);
        if (ok) {
          const int G = (int)gridDim.x;
#pragma unroll
          for (int q = 0; q < 2; ++q) {
            double m = -INFINITY, nn = 0.0;
            for (int g = lane; g < G; g += kWave) {
              m = fmax(m, ex.get(g, q));
              nn = fmax(nn, ex.get(g, 2 + q));
            }
            mx[q] = wave_max(m);
            bad[q] = wave_max(nn) != 0.0;
            double a[3] = {0.0, 0.0, 0.0};
            if (mx[q] != -INFINITY)
              for (int g = lane; g < G; g += kWave) {
                const double sc = exp(ex.get(g, q) - mx[q]);
                a[0] += ex.get(g, 4 + 3 * q) * sc;
                a[1] += ex.get(g, 5 + 3 * q) * (sc * sc);
                a[2] += ex.get(g, 6 + 3 * q) * sc;
              }
#pragma unroll
            for (int k = 0; k < 3; ++k) p[3 * q + k] = wave_sum(a[k]);
          }
        }
      }
      if (lane == 0) {
        s.ok = ok;
#pragma unroll
        for (int q = 0; q < 2; ++q) {
          const double out = bad[q] ? NAN : -INFINITY;
          const bool none = bad[q] || mx[q] == -INFINITY;
          s.bc[3 * q] = none ? out : mx[q] + log(p[3 * q]);
          s.bc[3 * q + 1] = none ? out : 2.0 * mx[q] + log(p[3 * q + 1]);
          s.bc[3 * q + 2] = none ? NAN : p[3 * q + 2] / p[3 * q];
        }
      }
    }
    __syncthreads();
    e0 = {s.bc[0], s.bc[1], s.bc[2]};
    e1 = {s.bc[3], s.bc[4], s.bc[5]};
    return s.ok != 0;
  }

  // The same at one db, with the sums relative to `ref` in place of the maximum; bc: the three sums.
  static MOCAT_DEV bool inner(const Particles& sh, double db, double ref, Exchange& ex, Smem& s, Eval& e) {
    const int t = threadIdx.x, lane = t & (kWave - 1), w = t / kWave;
    double p[3] = {0.0, 0.0, 0.0};
    sh.sums(db, ref, p);
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      p[k] = wave_sum(p[k]);
      if (lane == 0) s.red[k][w] = p[k];
    }
    __syncthreads();
    if (w == 0) {
#pragma unroll
      for (int k = 0; k < 3; ++k) {
        p[k] = s.red[k][0];
        for (int i = 1; i < NW; ++i) p[k] += s.red[k][i];
      }
      bool ok = true;
      if constexpr (SPLIT) {
        ok = ex.run(p);
        if (ok) {
          double a[3] = {0.0, 0.0, 0.0};
          for (int g = lane; g < (int)gridDim.x; g += kWave)
#pragma unroll
            for (int k = 0; k < 3; ++k) a[k] += ex.get(g, k);
#pragma unroll
          for (int k = 0; k < 3; ++k) p[k] = wave_sum(a[k]);
        }
      }
      if (lane == 0) {
        s.ok = ok;
#pragma unroll
        for (int k = 0; k < 3; ++k) s.bc[k] = p[k];
      }
    }
    __syncthreads();
    const double s1 = s.bc[0], s2 = s.bc[1];
    e.lse = ref + log(s1);
    e.lse2 = 2.0 * ref + log(s2);
    e.am = s.bc[2] / s1;
    return s.ok != 0;
  }
};

// Sums below this may have lost terms to underflow: the evaluation is repeated relative to the maximum.
constexpr double kTiny = -640.0;  // log; the smallest normal number is exp(-708)

// One evaluation is an FP64 exponential per particle, and what surrounds it is latency: reductions, two barriers,
// the exchange. So the bracket's ends are evaluated together; inside the bracket the sums are taken
// relative to the chord through the ends' log-sum-exps (log-sum-exp is convex in the temperature, so no exponential
// exceeds 1) instead of to a maximum found first; and the result's values are those of the evaluation that was
// chosen.
// SPLIT: a workgroup of 256 per 256 particles (at most kMaxSplit), one exchange per evaluation, which carries the
// weighted acceptance along. Without SPLIT one workgroup of 512, which sums the acceptance at the end; with
// a workspace only if the split search gave up.
template <bool SPLIT>
__global__ __launch_bounds__(Temper<SPLIT>::NT) void temper_kernel(TemperArgs a, TemperWs* ws, uint32_t max_polls) {
  using T = Temper<SPLIT>;
  __shared__ typename T::Smem s;
  if constexpr (!SPLIT)
    if (ws && ws->bar[1] == 0u) return;
  const typename T::Particles sh(a);
  Exchange ex{ws, max_polls, 0u};
  const double logthr = log(a.ess * a.retain);
  auto f = [&](const Eval& e) { return (2.0 * e.lse - e.lse2) - logthr; };
  double bnew = a.next_beta, fmin_abs = 0.0;
  int iters = 0;
  Eval lo, hi;
  if (!T::ends(sh, (a.adaptive ? a.max_temperature : a.next_beta) - a.beta, ex, s, lo, hi)) return;
  const double lse_prev = lo.lse;
  Eval at = hi;
  if (a.adaptive) {
    double b0 = a.beta, b1 = a.max_temperature;
    double f0 = f(lo), f1 = f(hi);
    const bool increasing = f1 > f0;
    while (true) {
      const bool done = fmin(fabs(f0), fabs(f1)) < a.tol || iters >= a.max_iter || (f0 < 0 && f1 < 0) ||
                        (f0 > 0 && f1 > 0) || isnan(f0) || isnan(f1);
      if (done) break;
      const double np = b0 - f0 * (b1 - b0) / (f1 - f0);
      const double ref = lo.lse + (hi.lse - lo.lse) * ((np - b0) / (b1 - b0));
      Eval e;
      if (!T::inner(sh, np - a.beta, ref, ex, s, e)) return;
      if (!(e.lse2 - 2.0 * ref > kTiny)) {
        Eval unused;
        if (!T::ends(sh, np - a.beta, ex, s, unused, e)) return;
      }
      const double ne = f(e);
      const bool replace_upper = increasing ? ne > 0 : ne < 0;
      if (replace_upper) {
        b1 = np;
        f1 = ne;
        hi = e;
      } else {
        b0 = np;
        f0 = ne;
        lo = e;
      }
      ++iters;
    }
    // bounds[argmin |evals|] (first on ties)
    const bool upper = fabs(f1) < fabs(f0);
    bnew = upper ? b1 : b0;
    at = upper ? hi : lo;
    fmin_abs = fmin(fabs(f0), fabs(f1));
  }
  const double db = bnew - a.beta;
  // weighted mean acceptance with weights exp(lw_new - max) (normalised)
  double amean = 0.0;
  if (a.alpha && a.k_alpha > 0) {
    amean = at.am;
    if constexpr (!SPLIT) {
      double num = 0.0, den = 0.0;
      sh.each([&](int64_t i, float l, float k) {
        const double wi = exp((double)l - db * (double)k - at.lse);
        num += wi * sh.mean_alpha(i);
        den += wi;
      });
      num = block_sum(num, s.red[0]);
      den = block_sum(den, s.red[1]);
      amean = num / den;
    }
  }
  // written last so that lw_out may alias lw: each thread its own particles
  sh.each([&](int64_t i, float l, float k) { a.lw_out[i] = (float)((double)l - db * (double)k); });
  if (threadIdx.x == 0 && blockIdx.x == 0) {
    a.out[0] = bnew;
    a.out[1] = exp(2.0 * at.lse - at.lse2);
    a.out[2] = at.lse;
    a.out[3] = lse_prev;
    a.out[4] = a.rm_stepsize != 0.0 ? a.log_stepsize + a.rm_stepsize * (amean - a.target) : a.log_stepsize;
    a.out[5] = amean;
    a.out[6] = (double)iters;
    a.out[7] = fmin_abs;
  }
}

__global__ void temper_clear_kernel(TemperWs* ws) { ws->bar[threadIdx.x] = 0u; }

// One workgroup / split, the whole step with 4 search iterations: 25 / 29 us at 2048 particles, 33 / 31 at 4096, 47 / 33 at
// 8192, 74 / 34 at 16384, 233 / 44 at 65536. One workgroup of 1024 spilled registers and took 51 us at 4096.
constexpr int64_t kSplitMin = 4096;

// cleared: an earlier kernel on the stream has set ws->bar to zero.
void launch_temper(const TemperArgs& a, TemperWs* ws, uint32_t max_polls, bool cleared, hipStream_t stream) {
  if (a.n < kSplitMin) {
    hipLaunchKernelGGL((temper_kernel<false>), dim3(1), dim3(Temper<false>::NT), 0, stream, a, (TemperWs*)nullptr, 0u);
    return;
  }
  const int64_t want = (a.n + Temper<true>::NT - 1) / Temper<true>::NT;
  const dim3 grid((unsigned)(want < kMaxSplit ? want : kMaxSplit));
  if (!cleared) hipLaunchKernelGGL(temper_clear_kernel, dim3(1), dim3(2), 0, stream, ws);
  hipLaunchKernelGGL((temper_kernel<true>), grid, dim3(Temper<true>::NT), 0, stream, a, ws, max_polls);
  hipLaunchKernelGGL((temper_kernel<false>), dim3(1), dim3(Temper<false>::NT), 0, stream, a, ws, 0u);
}

unsigned blocks_for(int64_t total) {
  const int64_t b = (total + 255) / 256;
  return (unsigned)(b < 65535 ? b : 65535);
}

// keys = split(key, n + 2): particle i moves with split(keys[i], 3)[0], keys[n] resamples, keys[n + 1] is
// the next temperature's. After a resample the log weights are zero.
__global__ __launch_bounds__(256) void pass_keys_kernel(const uint32_t* __restrict__ key, int64_t n,
                                                        uint32_t* __restrict__ move_keys, uint32_t* resample_key,
                                                        uint32_t* next_key, float* lw_zero) {
  const Key k{key[0], key[1]};
  const uint32_t num = (uint32_t)n + 2u;
  for (int64_t i = blockIdx.x * (int64_t)256 + threadIdx.x; i < n + 2; i += (int64_t)gridDim.x * 256) {
    Key c = split_at(k, num, (uint32_t)i);
    uint32_t* dst = i == n ? resample_key : next_key;
    if (i < n) {
      c = split_at(c, 3u, 0u);
      dst = move_keys + 2 * i;
      if (lw_zero) lw_zero[i] = 0.f;
    }
    dst[0] = c.a;
    dst[1] = c.b;
  }
}

__global__ __launch_bounds__(256) void gather_pair_kernel(const float* __restrict__ a, const float* __restrict__ b,
                                                          const int32_t* __restrict__ idx, int64_t n, int64_t d,
                                                          float* __restrict__ a_out, float* __restrict__ b_out) {
  const float* src = blockIdx.y ? b : a;
  float* dst = blockIdx.y ? b_out : a_out;
  for (int64_t e = blockIdx.x * (int64_t)256 + threadIdx.x; e < n * d; e += (int64_t)gridDim.x * 256) {
    const int64_t j = e / d;
    dst[e] = src[(int64_t)idx[j] * d + (e - j * d)];
  }
}

// a + b * c with the product rounded (HIP contracts by default), as elementwise tensor steps give it.
MOCAT_DEV float tempered(float a, float b, float c) {
#pragma clang fp contract(off)
  const float p = b * c;
  return a + p;
}

// Potential and gradient at temperature beta; the moves' stepsizes; the counters of this call.
__global__ __launch_bounds__(256) void pass_begin_kernel(int64_t n, int64_t d, float beta, float h,
                                                         const float* __restrict__ prior, const float* __restrict__ lik,
                                                         const float* __restrict__ gp, const float* __restrict__ gl,
                                                         float* __restrict__ pot, float* __restrict__ grad,
                                                         float* __restrict__ stepsize, TemperWs* ws,
                                                         unsigned long long* nans) {
  for (int64_t e = blockIdx.x * (int64_t)256 + threadIdx.x; e < n * d; e += (int64_t)gridDim.x * 256) {
    if (e == 0) {
      ws->bar[0] = ws->bar[1] = 0u;
      *nans = 0ull;
    }
    grad[e] = tempered(gp[e], beta, gl[e]);
    if (e < n) {
      pot[e] = tempered(prior[e], beta, lik[e]);
      stepsize[e] = h;
    }
  }
}

// The potential at the temperature that was found, and how many of the values are NaN.
__global__ __launch_bounds__(256) void pass_end_kernel(int64_t n, int64_t d, const double* __restrict__ out,
                                                       const float* __restrict__ prior, const float* __restrict__ lik,
                                                       const float* __restrict__ value, float* __restrict__ pot,
                                                       unsigned long long* nans) {
  const float beta = (float)out[0];
  unsigned long long c = 0ull;
  for (int64_t e = blockIdx.x * (int64_t)256 + threadIdx.x; e < n * d; e += (int64_t)gridDim.x * 256) {
    c += isnan(value[e]) ? 1ull : 0ull;
    if (e < n) pot[e] = tempered(prior[e], beta, lik[e]);
  }
  if (c) atomicAdd(nans, c);
}

}  // namespace

extern "C" {

int mocat_gather_rows(const void* src, const int32_t* idx, int64_t n_out, int64_t width, void* dst,
                      hipStream_t stream) {
  if (!src || !idx || !dst || n_out < 0 || width <= 0) return MOCAT_ERR_ARG;
  if (n_out == 0) return MOCAT_OK;
  const int64_t total = n_out * width;
  const int64_t blocks = (total + 255) / 256;
  hipLaunchKernelGGL(gather_kernel, dim3((unsigned)(blocks < 65535 ? blocks : 65535)), dim3(256), 0, stream,
                     (const uint32_t*)src, idx, n_out, width, (uint32_t*)dst);
  MOCAT_LAUNCH_CHECK();
  return MOCAT_OK;
}

int mocat_smc_temper(const float* log_weight, const float* lik, int64_t n, double beta, double ess, double retain,
                     double max_temperature, double tol, int max_iter, int adaptive, double next_beta,
                     const float* alpha, int k_alpha, double log_stepsize, double rm_stepsize, double target,
                     float* log_weight_out, double* out, hipStream_t stream) {
  if (!log_weight || !lik || !log_weight_out || !out || n <= 0 || max_iter < 0 || k_alpha < 0) return MOCAT_ERR_ARG;
  TemperArgs a{log_weight, lik, n, beta, ess, retain, max_temperature, tol, max_iter, adaptive, next_beta,
               alpha, k_alpha, log_stepsize, rm_stepsize, target, log_weight_out, out};
  hipLaunchKernelGGL((temper_kernel<false>), dim3(1), dim3(Temper<false>::NT), 0, stream, a, (TemperWs*)nullptr, 0u);
  MOCAT_LAUNCH_CHECK();
  return MOCAT_OK;
}

int mocat_smc_temper_workspace_bytes(int64_t* bytes) {
  if (!bytes) return MOCAT_ERR_ARG;
  *bytes = (int64_t)sizeof(TemperWs);
  return MOCAT_OK;
}

int mocat_smc_temper_split(const float* log_weight, const float* lik, int64_t n, double beta, double ess, double retain,
                           double max_temperature, double tol, int max_iter, int adaptive, double next_beta,
                           const float* alpha, int k_alpha, double log_stepsize, double rm_stepsize, double target,
                           float* log_weight_out, double* out, void* workspace, int64_t workspace_bytes, int max_polls,
                           hipStream_t stream) {
  if (!log_weight || !lik || !log_weight_out || !out || n <= 0 || max_iter < 0 || k_alpha < 0 || max_polls < 0 ||
      log_weight == log_weight_out || (uintptr_t)workspace % 8)
    return MOCAT_ERR_ARG;
  if (!workspace || workspace_bytes < (int64_t)sizeof(TemperWs)) return MOCAT_ERR_SIZE;
  TemperArgs a{log_weight, lik, n, beta, ess, retain, max_temperature, tol, max_iter, adaptive, next_beta,
               alpha, k_alpha, log_stepsize, rm_stepsize, target, log_weight_out, out};
  launch_temper(a, (TemperWs*)workspace, (uint32_t)max_polls, false, stream);
  MOCAT_LAUNCH_CHECK();
  return MOCAT_OK;
}

int mocat_smc_resample_workspace_bytes(int64_t n, int64_t* bytes) {
  if (!bytes || n <= 0) return MOCAT_ERR_ARG;
  *bytes = n * (int64_t)(sizeof(uint64_t) + sizeof(int32_t)) + 2 * (int64_t)sizeof(uint32_t);
  return MOCAT_OK;
}

int mocat_smc_resample(const uint32_t* key, int64_t n, int64_t d, int method, const float* log_weight,
                       const float* value, const float* momenta, float* value_out, float* momenta_out,
                       float* log_weight_out, uint32_t* move_keys, uint32_t* next_key, void* workspace,
                       int64_t workspace_bytes, hipStream_t stream) {
  if (!key || !move_keys || !next_key || key == next_key || n <= 0 || n > 0x7FFFFFFD || d <= 0 || method < -1 || method > 2 ||
      (uintptr_t)workspace % 8)
    return MOCAT_ERR_ARG;
  if (method >= 0 && (!log_weight || !value || !momenta || !value_out || !momenta_out || !log_weight_out ||
                      value == value_out || momenta == momenta_out || log_weight == log_weight_out))
    return MOCAT_ERR_ARG;
  int64_t need = 0;
  mocat_smc_resample_workspace_bytes(n, &need);
  if (!workspace || workspace_bytes < need) return MOCAT_ERR_SIZE;
  uint64_t* csum = (uint64_t*)workspace;
  int32_t* idx = (int32_t*)(csum + n);
  uint32_t* rkey = (uint32_t*)(idx + n);
  hipLaunchKernelGGL(pass_keys_kernel, dim3(blocks_for(n + 2)), dim3(256), 0, stream, key, n, move_keys, rkey, next_key,
                     method >= 0 ? log_weight_out : (float*)nullptr);
  MOCAT_LAUNCH_CHECK();
  if (method < 0) return MOCAT_OK;
  const int rc = method == 2 ? mocat_resample_categorical(log_weight, n, n, rkey, idx, stream)
                             : mocat_resample(log_weight, n, method, 1, rkey, csum, idx, stream);
  if (rc != MOCAT_OK) return rc;
  hipLaunchKernelGGL(gather_pair_kernel, dim3(blocks_for(n * d), 2), dim3(256), 0, stream, value, momenta, (const int32_t*)idx, n,
                     d, value_out, momenta_out);
  MOCAT_LAUNCH_CHECK();
  return MOCAT_OK;
}

int mocat_smc_move(const float* X, const float* y, const void* packed, int64_t rows, int64_t d, int precision,
                   float prior_prec, int64_t n, const float* grad_prior, const float* grad_lik, float* value,
                   float* momenta, float* grad, float* potential, float* prior_pot, float* lik_pot, float* stepsizes,
                   float* alpha, uint32_t* keys, int steps, int leapfrog_steps, float friction, float* alpha_trace,
                   const float* log_weight, double beta, double stepsize, double log_stepsize, double ess,
                   double retain, double max_temperature, double tol, int max_iter, int adaptive, double next_beta,
                   double rm_stepsize, double target, float* log_weight_out, double* out, void* workspace,
                   int64_t workspace_bytes, int max_polls, hipStream_t stream) {
  if (n <= 0 || d <= 0 || !grad_prior || !grad_lik || !value || !grad || !potential || !prior_pot || !lik_pot ||
      !stepsizes || !log_weight || !log_weight_out || !out || log_weight == log_weight_out || max_iter < 0 ||
      steps < 0 || max_polls < 0 || (uintptr_t)workspace % 8)
    return MOCAT_ERR_ARG;
  if (!workspace || workspace_bytes < (int64_t)sizeof(TemperWs)) return MOCAT_ERR_SIZE;
  TemperWs* ws = (TemperWs*)workspace;
  unsigned long long* nans = (unsigned long long*)(out + 8);
  hipLaunchKernelGGL(pass_begin_kernel, dim3(blocks_for(n * d)), dim3(256), 0, stream, n, d, (float)beta, (float)stepsize,
                     (const float*)prior_pot, (const float*)lik_pot, grad_prior, grad_lik, potential, grad, stepsizes, ws,
                     nans);
  MOCAT_LAUNCH_CHECK();
  const int rc = mocat_hmc_lr_iterate(X, y, packed, rows, d, precision, prior_prec, (float)beta, n, value, momenta, grad,
                                      potential, prior_pot, lik_pot, stepsizes, alpha, keys, 0, steps, leapfrog_steps,
                                      friction, 1, 0.f, 1.f, 2.f / 3.f, INFINITY, nullptr, nullptr, alpha_trace, nullptr,
                                      nullptr, stream);
  if (rc != MOCAT_OK) return rc;
  TemperArgs a{log_weight, lik_pot, n, beta, ess, retain, max_temperature, tol, max_iter, adaptive, next_beta,
               alpha_trace, steps, log_stepsize, rm_stepsize, target, log_weight_out, out};
  launch_temper(a, ws, (uint32_t)max_polls, true, stream);
  hipLaunchKernelGGL(pass_end_kernel, dim3(blocks_for(n * d)), dim3(256), 0, stream, n, d, (const double*)out,
                     (const float*)prior_pot, (const float*)lik_pot, (const float*)value, potential, nans);
  MOCAT_LAUNCH_CHECK();
  return MOCAT_OK;
}

}  // extern "C"
