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

constexpr int NT = 1024;
constexpr int NW = NT / kWave;

__global__ __launch_bounds__(256) void gather_kernel(const uint32_t* __restrict__ src, const int32_t* __restrict__ idx,
                                                     int64_t n_out, int64_t width, uint32_t* __restrict__ dst) {
  const int64_t total = n_out * width;
  for (int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; e < total; e += (int64_t)gridDim.x * blockDim.x) {
    const int64_t j = e / width, k = e - j * width;
    dst[e] = src[(int64_t)idx[j] * width + k];
  }
}

struct Smem {
  double m[NW], s1[NW], s2[NW];
  double bc[2];
  int pass;
};

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
struct Share {
  int64_t n, stride, first;  // stride = G * NT
  const float *lw, *lik;
  float rl[kRegs], rk[kRegs];
  template <class F>
  MOCAT_DEV void each(F f) const {
#pragma unroll
    for (int k = 0; k < kRegs; ++k) {
      const int64_t i = first + k * stride;
      if (i < n) f(i, rl[k], rk[k]);
    }
    for (int64_t i = first + kRegs * stride; i < n; i += stride) f(i, lw[i], lik[i]);
  }
};
MOCAT_DEV Share share_of(const float* lw, const float* lik, int64_t n) {
  Share s;
  s.n = n;
  s.stride = (int64_t)gridDim.x * NT;
  s.first = (int64_t)blockIdx.x * NT + threadIdx.x;
  s.lw = lw;
  s.lik = lik;
#pragma unroll
  for (int k = 0; k < kRegs; ++k) {
    const int64_t i = s.first + k * s.stride;
    s.rl[k] = i < n ? lw[i] : 0.f;
    s.rk[k] = i < n ? lik[i] : 0.f;
  }
  return s;
}

// Workgroups of a split evaluation, and what they exchange: two sets of slots used in turn, so that a
// workgroup that is one exchange ahead never overwrites what another still reads, and the barrier's
// arrival count and abort flag. A workgroup that polls max_polls times without seeing every arrival sets
// the flag and leaves, as does every workgroup that sees it; temper_kernel<false> then does the work.
constexpr int kMaxSplit = 32;
static_assert(kMaxSplit <= kWave, "one wave combines the workgroups' slots");
struct TemperWs {
  double slot[2][kMaxSplit][4];
  uint32_t bar[2];
};
struct Exchange {
  TemperWs* ws;
  uint32_t max_polls, count;

  // Publishes this workgroup's values (thread 0's), waits for all: true when every workgroup arrived.
  MOCAT_DEV bool run(const double* v, int nv, bool wait, Smem& s) {
    const int par = count & 1;
    ++count;
    if (threadIdx.x == 0) {
      for (int k = 0; k < nv; ++k) ws->slot[par][blockIdx.x][k] = v[k];
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
      __hip_atomic_fetch_add(&ws->bar[0], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      int ok = 1;
      const uint32_t target = count * gridDim.x;
      for (uint32_t polls = 0; wait; ++polls) {
        if (__hip_atomic_load(&ws->bar[1], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0u) {
          ok = 0;
          break;
        }
        if (polls >= max_polls) {
          __hip_atomic_store(&ws->bar[1], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
          ok = 0;
          break;
        }
        if (__hip_atomic_load(&ws->bar[0], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) >= target) break;
        __builtin_amdgcn_s_sleep(1);
      }
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
      s.pass = ok;
    }
    __syncthreads();
    const bool ok = s.pass != 0;
    __syncthreads();
    return ok;
  }
  MOCAT_DEV const double* slots(int g) const { return ws->slot[(count - 1) & 1][g]; }
};

// (lse(w), lse(2w)) of w_i = lw_i - db * lik_i, FP64: the workgroup's maximum m and the sums of
// exp(w_i - m) and its square (one exponential per element), partial sums combined in a fixed order (lanes by
// butterfly, waves in index order, workgroups by butterfly after scaling to the common maximum), so that every
// workgroup finds the same values and takes the same decisions. false: the exchange was given up.
template <bool SPLIT>
MOCAT_DEV bool lse_pair(const Share& sh, double db, Exchange& ex, Smem& s, double& lse, double& lse2) {
  const int t = threadIdx.x, lane = t & (kWave - 1), w = t / kWave;
  double mx = -INFINITY;
  int has_nan = 0;
  sh.each([&](int64_t, float l, float k) {
    const double v = (double)l - db * (double)k;
    if (isnan(v)) has_nan = 1;
    else mx = fmax(mx, v);
  });
  const bool nan_seen = __syncthreads_or(has_nan) != 0;
  mx = wave_max(mx);
  if (lane == 0) s.m[w] = mx;
  __syncthreads();
  double m = s.m[0];
  for (int i = 1; i < NW; ++i) m = fmax(m, s.m[i]);
  double s1 = 0.0, s2 = 0.0;
  if (!nan_seen && m != -INFINITY)
    sh.each([&](int64_t, float l, float k) {
      const double e = exp((double)l - db * (double)k - m);
      s1 += e;
      s2 += e * e;
    });
  s1 = wave_sum(s1);
  s2 = wave_sum(s2);
  if (lane == 0) {
    s.s1[w] = s1;
    s.s2[w] = s2;
  }
  __syncthreads();
  double a1 = 0.0, a2 = 0.0;
  for (int i = 0; i < NW; ++i) {
    a1 += s.s1[i];
    a2 += s.s2[i];
  }
  __syncthreads();  // every thread has read the partials before a later call rewrites them
  bool bad = nan_seen;
  if constexpr (SPLIT) {
    const double v[4] = {m, a1, a2, nan_seen ? 1.0 : 0.0};
    if (!ex.run(v, 4, true, s)) return false;
    if (w == 0) {
      const bool in = lane < (int)gridDim.x;
      const double* o = ex.slots(in ? lane : 0);
      const double mg = in ? o[0] : -INFINITY, ng = in ? o[3] : 0.0;
      const double mm = wave_max(mg);
      const double sc = in && mm != -INFINITY ? exp(mg - mm) : 0.0;
      const double t1 = wave_sum(in ? o[1] * sc : 0.0), t2 = wave_sum(in ? o[2] * (sc * sc) : 0.0);
      const double nn = wave_max(ng);
      if (lane == 0) {
        s.m[0] = mm;
        s.s1[0] = t1;
        s.s2[0] = t2;
        s.bc[0] = nn;
      }
    }
    __syncthreads();
    m = s.m[0];
    a1 = s.s1[0];
    a2 = s.s2[0];
    bad = s.bc[0] != 0.0;
    __syncthreads();
  }
  if (bad || m == -INFINITY) {
    lse = lse2 = bad ? NAN : -INFINITY;
  } else {
    lse = m + log(a1);
    lse2 = 2.0 * m + log(a2);
  }
  return true;
}

// One evaluation is an FP64 exponential per particle and takes 10 us in one workgroup at 16384 particles, 132 us for
// the whole search. SPLIT: a workgroup per 1024 particles (at most kMaxSplit), one exchange per evaluation;
// the evaluations at b_t and at the chosen bound are those of the search.
// Without SPLIT one workgroup; with a workspace only if the split search gave up.
template <bool SPLIT>
__global__ __launch_bounds__(NT) void temper_kernel(TemperArgs a, TemperWs* ws, uint32_t max_polls) {
  __shared__ Smem s;
  if constexpr (!SPLIT)
    if (ws && ws->bar[1] == 0u) return;
  const int t = threadIdx.x;
  const Share sh = share_of(a.lw, a.lik, a.n);
  Exchange ex{ws, max_polls, 0u};
  const double logthr = log(a.ess * a.retain);
  double bnew, fmin_abs = 0.0, lse_prev, lse_new, lse2_new;
  int iters = 0;
  if (a.adaptive) {
    double b0 = a.beta, b1 = a.max_temperature, l0, m0, l1, m1;
    if (!lse_pair<SPLIT>(sh, 0.0, ex, s, l0, m0)) return;
    if (!lse_pair<SPLIT>(sh, b1 - a.beta, ex, s, l1, m1)) return;
    double e0 = (2.0 * l0 - m0) - logthr, e1 = (2.0 * l1 - m1) - logthr;
    lse_prev = l0;
    const bool increasing = e1 > e0;
    while (true) {
      const bool done = fmin(fabs(e0), fabs(e1)) < a.tol || iters >= a.max_iter || (e0 < 0 && e1 < 0) ||
                        (e0 > 0 && e1 > 0) || isnan(e0) || isnan(e1);
      if (done) break;
      const double np = b0 - e0 * (b1 - b0) / (e1 - e0);
      double l, m;
      if (!lse_pair<SPLIT>(sh, np - a.beta, ex, s, l, m)) return;
      const double ne = (2.0 * l - m) - logthr;
      const bool replace_upper = increasing ? ne > 0 : ne < 0;
      if (replace_upper) {
        b1 = np;
        e1 = ne;
        l1 = l;
        m1 = m;
      } else {
        b0 = np;
        e0 = ne;
        l0 = l;
        m0 = m;
      }
      ++iters;
    }
    // bounds[argmin |evals|] (first on ties)
    const bool upper = fabs(e1) < fabs(e0);
    bnew = upper ? b1 : b0;
    lse_new = upper ? l1 : l0;
    lse2_new = upper ? m1 : m0;
    fmin_abs = fmin(fabs(e0), fabs(e1));
  } else {
    bnew = a.next_beta;
    double lse_prev2;
    if (!lse_pair<SPLIT>(sh, 0.0, ex, s, lse_prev, lse_prev2)) return;
    if (!lse_pair<SPLIT>(sh, bnew - a.beta, ex, s, lse_new, lse2_new)) return;
  }
  const double db = bnew - a.beta;
  // weighted mean acceptance with weights exp(lw_new - max) (normalised)
  double amean = 0.0;
  if (a.alpha && a.k_alpha > 0) {
    double num = 0.0, den = 0.0;
    sh.each([&](int64_t i, float l, float k) {
      const double wi = exp((double)l - db * (double)k - lse_new);
      double am = 0.0;
      for (int j = 0; j < a.k_alpha; ++j) am += (double)a.alpha[(int64_t)j * a.n + i];
      am /= (double)a.k_alpha;
      num += wi * am;
      den += wi;
    });
    num = wave_sum(num);
    den = wave_sum(den);
    if ((t & (kWave - 1)) == 0) {
      s.s1[t / kWave] = num;
      s.s2[t / kWave] = den;
    }
    __syncthreads();
    double N = 0.0, D = 0.0;
    for (int i = 0; i < NW; ++i) {
      N += s.s1[i];
      D += s.s2[i];
    }
    __syncthreads();
    if constexpr (SPLIT) {
      const double v[2] = {N, D};
      if (!ex.run(v, 2, blockIdx.x == 0, s)) return;
      if (blockIdx.x == 0) {
        N = D = 0.0;
        for (int g = 0; g < (int)gridDim.x; ++g) {
          N += ex.slots(g)[0];
          D += ex.slots(g)[1];
        }
      }
    }
    amean = N / D;
  }
  // written last so that lw_out may alias lw: each thread its own particles
  sh.each([&](int64_t i, float l, float k) { a.lw_out[i] = (float)((double)l - db * (double)k); });
  if (t == 0 && blockIdx.x == 0) {
    a.out[0] = bnew;
    a.out[1] = exp(2.0 * lse_new - lse2_new);
    a.out[2] = lse_new;
    a.out[3] = lse_prev;
    a.out[4] = a.rm_stepsize != 0.0 ? a.log_stepsize + a.rm_stepsize * (amean - a.target) : a.log_stepsize;
    a.out[5] = amean;
    a.out[6] = (double)iters;
    a.out[7] = fmin_abs;
  }
}

__global__ void temper_clear_kernel(TemperWs* ws) { ws->bar[threadIdx.x] = 0u; }

// One workgroup / split, the whole step with 4 search iterations: 42 / 61 us at 4096 particles, 60 / 62 at 8192, 92 / 65 at
// 16384, 274 / 76 at 65536, 6690 / 199 at 2^20 (an exchange costs about as much as 8 particles per thread).
constexpr int64_t kSplitMin = 12288;

// cleared: an earlier kernel on the stream has set ws->bar to zero.
void launch_temper(const TemperArgs& a, TemperWs* ws, uint32_t max_polls, bool cleared, hipStream_t stream) {
  if (a.n < kSplitMin) {
    hipLaunchKernelGGL((temper_kernel<false>), dim3(1), dim3(NT), 0, stream, a, (TemperWs*)nullptr, 0u);
    return;
  }
  const int64_t want = (a.n + NT - 1) / NT;
  const dim3 grid((unsigned)(want < kMaxSplit ? want : kMaxSplit));
  if (!cleared) hipLaunchKernelGGL(temper_clear_kernel, dim3(1), dim3(2), 0, stream, ws);
  hipLaunchKernelGGL((temper_kernel<true>), grid, dim3(NT), 0, stream, a, ws, max_polls);
  hipLaunchKernelGGL((temper_kernel<false>), dim3(1), dim3(NT), 0, stream, a, ws, 0u);
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
  hipLaunchKernelGGL((temper_kernel<false>), dim3(1), dim3(NT), 0, stream, a, (TemperWs*)nullptr, 0u);
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
