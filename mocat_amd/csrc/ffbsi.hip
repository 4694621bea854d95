// Forward-filtering backward-simulation, full resampling (mocat/src/ssm/backward.py:20-39, 210-243).
//
// One backward step, for every trajectory m of M: key_m = split(key_t, M)[m] and
//   x_t[m] = particles_t[argmax_j(gumbel(key_m, (N,))[j] + log_weight_t[j] - U(particles_t[j] -> x_{t+1}[m]))]
// (random.categorical: the first maximum wins), U the model's transition potential as mocat's
// gaussian_potential evaluates it (utils.py:49-105): 0.5 |(x' - A x) @ S|^2 + nlz, S the transition
// precision square root. One wave per trajectory (or a workgroup, when there are few): the lanes take
// pairs (j, j + N/2), whose Gumbel bits come out of one threefry block (the halves layout), and keep a
// running maximum; a butterfly with the lower index winning ties combines them. Work per step: N x M / 2
// threefry blocks, N x M bounds of the scores, and the potentials and accurate logarithms of the draws that
// the bounds do not drop (gumbel.hpp; a few per trajectory). Kernel time of a step of 4096 x 4096 without and
// with the bounds: d = 1 45 and 35 us, d = 4 59 and 39, d = 8 150 and 57 (threefry and bound, about 50
// operations a pair, are then what is left); 4096 x 1024, d = 4: 28 and, four waves a trajectory, 17.5.
#include <cmath>

#include "common.hpp"
#include "gumbel.hpp"

using namespace mocat;

namespace {

// linear Gaussian: params A[D*D], S[D*D] (transition precision square root), nlz
template <int D>
struct LgTrans {
  float A[D * D], S[D * D], nlz;
  MOCAT_DEV void load(const float* p, int /*d: D*/) {
#pragma unroll
    for (int i = 0; i < D * D; ++i) A[i] = p[i];
#pragma unroll
    for (int i = 0; i < D * D; ++i) S[i] = p[D * D + i];
    nlz = p[2 * D * D];
  }
  MOCAT_DEV float pot(const float* xp, const float* xn) const {
    float diff[D];
#pragma unroll
    for (int i = 0; i < D; ++i) {
      float a = 0.f;
#pragma unroll
      for (int k = 0; k < D; ++k) a += A[i * D + k] * xp[k];
      diff[i] = xn[i] - a;
    }
    float s = 0.f;
#pragma unroll
    for (int k = 0; k < D; ++k) {
      float v = 0.f;
#pragma unroll
      for (int i = 0; i < D; ++i) v += diff[i] * S[i * D + k];
      s += v * v;
    }
    return 0.5f * s + nlz;
  }
  // u = x @ S and a = max_k sum_i |x_i S_ik|
  MOCAT_DEV void project(const float* x, float* u, float& a) const {
    a = 0.f;
#pragma unroll
    for (int k = 0; k < D; ++k) {
      float v = 0.f, b = 0.f;
#pragma unroll
      for (int i = 0; i < D; ++i) {
        v += x[i] * S[i * D + k];
        b += fabsf(x[i] * S[i * D + k]);
      }
      u[k] = v;
      a = b > a || isnan(b) ? b : a;
    }
  }
  MOCAT_DEV void project_mean(const float* xp, float* u, float& a) const {
    float ax[D];
#pragma unroll
    for (int i = 0; i < D; ++i) {
      float m = 0.f;
#pragma unroll
      for (int k = 0; k < D; ++k) m += A[i * D + k] * xp[k];
      ax[i] = m;
    }
    project(ax, u, a);
  }
};

// stochastic volatility, unit steps (stochastic_volatility.py:78-84): params phi, 1/sigma, nlz
struct SvTrans {
  float phi, isig, nlz;
  MOCAT_DEV void load(const float* p, int /*d: 1*/) {
    phi = p[0];
    isig = p[1];
    nlz = p[2];
  }
  MOCAT_DEV float pot(const float* xp, const float* xn) const {
    const float diff = xn[0] - xp[0] * phi;
    return 0.5f * (diff * diff) * (isig * isig) + nlz;
  }
  MOCAT_DEV void project(const float* x, float* u, float& a) const {
    u[0] = x[0] * isig;
    a = fabsf(u[0]);
  }
  MOCAT_DEV void project_mean(const float* xp, float* u, float& a) const {
    const float m = phi * xp[0];
    project(&m, u, a);
  }
};

// linear Gaussian at a runtime d <= kRtMaxDim (the kernels' template D = 0): A and S read from params,
// the difference vector in the calling lane's LDS row, the products in LgTrans's order
constexpr int kRtMaxDim = 16;

struct LgTransRt {
  const float *A, *S;
  float nlz;
  int d;
  MOCAT_DEV void load(const float* p, int dd) {
    d = dd;
    A = p;
    S = p + dd * dd;
    nlz = p[2 * dd * dd];
  }
  MOCAT_DEV float pot(const float* xp, const float* xn) const {
    __shared__ float DF[kRtMaxDim][256];
    const int t = threadIdx.x;
    for (int i = 0; i < d; ++i) {
      float a = 0.f;
      for (int k = 0; k < d; ++k) a += A[i * d + k] * xp[k];
      DF[i][t] = xn[i] - a;
    }
    float s = 0.f;
    for (int k = 0; k < d; ++k) {
      float v = 0.f;
      for (int i = 0; i < d; ++i) v += DF[i][t] * S[i * d + k];
      s += v * v;
    }
    return 0.5f * s + nlz;
  }
};

// Bounds of the logits lw_j - U(x_j -> x'), prepared once per filter particle: U = 0.5 |v|^2 + nlz with
// v = (x' - A x) @ S = x' @ S - p, p = (A x) @ S, so a pair's bound takes D subtractions and D FMAs from p and
// x' @ S, and no product with A or S. Rounding: a component of that difference is within
// delta = kRoundings * 2^-24 (a_j + a_m) of the v that pot() forms, a = max_k sum_i |(A x)_i S_ik| (a_m the same
// of x'), and (v - delta)^2 >= (1 - kEta) v^2 - delta^2 / kEta, with kEta also above the relative error of the
// squared norm. The sums' own rounding is below 1e-6 (|lw| + |nlz|). Filter particle j carries its share of these
// slacks in `lim`; a non-finite state leaves NaN or infinity there, which drops nothing.
constexpr float kEta = 1e-3f, kRoundings = 64.f;
MOCAT_DEV float rounding_slack(float a) {
  const float e = kRoundings * 5.9604645e-8f * a;  // (a_j + a_m)^2 <= 2 (a_j^2 + a_m^2)
  return e * e / kEta;
}

// One thread per particle of a block of time points: pre[k] = {p[D], lim}.
template <class Tr, int D>
__global__ __launch_bounds__(256) void ffbsi_prep_kernel(const float* __restrict__ params, const float* __restrict__ xs,
                                                         const float* __restrict__ lw, int64_t count,
                                                         float* __restrict__ p, float* __restrict__ lim) {
  Tr tr;
  tr.load(params, D);
  for (int64_t k = blockIdx.x * (int64_t)256 + threadIdx.x; k < count; k += (int64_t)gridDim.x * 256) {
    float pj[D], a;
    tr.project_mean(xs + k * D, pj, a);
#pragma unroll
    for (int q = 0; q < D; ++q) p[k * D + q] = pj[q];
    const float l = lw[k];
    lim[k] = l == -INFINITY ? l : l - tr.nlz + 1e-6f * (fabsf(l) + fabsf(tr.nlz)) + (float)D * rounding_slack(a);
  }
}

// W waves per trajectory: 1, or all four of a workgroup. p, lim: the prepared bounds of these particles, or
// null (then lw - nlz bounds a logit).
template <class Tr, int D, int W>
__global__ __launch_bounds__(256) void ffbsi_step_kernel(const float* __restrict__ params,
                                                         const float* __restrict__ xs, const float* __restrict__ lw,
                                                         const float* __restrict__ p, const float* __restrict__ lim,
                                                         int64_t n, const float* __restrict__ xnext, int64_t m_count,
                                                         const uint32_t* __restrict__ key, int32_t* __restrict__ idx,
                                                         float* __restrict__ xout) {
  constexpr int kWaves = 256 / kWave;
  static_assert(W == 1 || W == kWaves, "one wave or the whole workgroup per trajectory");
  __shared__ float wbest[kWaves];
  __shared__ uint32_t wi[kWaves];
  const int lane = threadIdx.x & (kWave - 1), w = threadIdx.x / kWave;
  const int64_t m = W == 1 ? (int64_t)blockIdx.x * kWaves + w : (int64_t)blockIdx.x;
  if (m >= m_count) return;
  Tr tr;
  tr.load(params, D);
  const Key km = split_at(Key{key[0], key[1]}, (uint32_t)m_count, (uint32_t)m);
  float xn[D];
#pragma unroll
  for (int q = 0; q < D; ++q) xn[q] = xnext[m * D + q];
  const uint32_t part = W == 1 ? 0u : (uint32_t)w;
  auto logit = [&](uint32_t j) { return lw[j] - tr.pot(xs + (int64_t)j * D, xn); };
  float best;
  uint32_t bi;
  if (p) {
    float u[D], a;
    tr.project(xn, u, a);
    const float slack = (float)D * rounding_slack(a);
    auto bound = [&](uint32_t j) {
      float s = 0.f;
#pragma unroll
      for (int q = 0; q < D; ++q) {
        const float v = u[q] - p[(int64_t)j * D + q];
        s = fmaf(v, v, s);
      }
      return fmaf(-0.5f * (1.f - kEta), s, lim[j] + slack);
    };
    bi = gumbel_argmax(km, (uint32_t)n, lane, part, W, bound, logit, &best);
  } else {
    bi = gumbel_argmax(km, (uint32_t)n, lane, part, W, [&](uint32_t j) { return lw[j] - tr.nlz; }, logit, &best);
  }
  if constexpr (W > 1) {
    if (lane == 0) {
      wbest[w] = best;
      wi[w] = bi;
    }
    __syncthreads();
    GumbelRow all;
    for (int k = 0; k < W; ++k) all.take(wbest[k], wi[k]);
    bi = all.bi;
    if (w != 0) return;
  }
  if (lane == 0 && idx) idx[m] = (int32_t)bi;
  if (lane < D) xout[m * D + lane] = xs[(int64_t)bi * D + lane];
}

template <class Tr, int D>
int launch_ffbsi(const float* params, const float* xs, const float* lw, const float* p, const float* lim, int64_t n,
                 const float* xnext, int64_t m, const uint32_t* key, int32_t* idx, float* xout, hipStream_t stream) {
  // with at most two waves per SIMD a wave's chain of threefry blocks is the bound: four share it
  const bool split = m <= 2048 && n >= 512;
  if (split)
    hipLaunchKernelGGL((ffbsi_step_kernel<Tr, D, 4>), dim3((unsigned)m), dim3(256), 0, stream, params, xs, lw, p, lim, n,
                       xnext, m, key, idx, xout);
  else
    hipLaunchKernelGGL((ffbsi_step_kernel<Tr, D, 1>), dim3((unsigned)((m + 3) / 4)), dim3(256), 0, stream, params, xs,
                       lw, p, lim, n, xnext, m, key, idx, xout);
  MOCAT_LAUNCH_CHECK();
  return MOCAT_OK;
}

// The full backward step for the linear-Gaussian model at a d without a compiled kernel (d <= kRtMaxDim):
// the same draw and potential (0.5 |(x' - A x) @ S|^2 + nlz, the products in LgTrans's order) with A and
// S in LDS, each wave's x_{t+1} in LDS, and each lane's particle state and difference vector in its own
// LDS rows (indexed at run time).

__global__ __launch_bounds__(256) void ffbsi_step_rt_kernel(int d, const float* __restrict__ params,
                                                            const float* __restrict__ xs,
                                                            const float* __restrict__ lw, int64_t n,
                                                            const float* __restrict__ xnext, int64_t m_count,
                                                            const uint32_t* __restrict__ key,
                                                            int32_t* __restrict__ idx, float* __restrict__ xout) {
  __shared__ float A[kRtMaxDim * kRtMaxDim], S[kRtMaxDim * kRtMaxDim];
  __shared__ float XN[256 / kWave][kRtMaxDim];
  __shared__ float XP[kRtMaxDim][256], DF[kRtMaxDim][256];
  const int t = threadIdx.x, lane = t & (kWave - 1), w = t / kWave;
  for (int k = t; k < d * d; k += 256) {
    A[k] = params[k];
    S[k] = params[d * d + k];
  }
  const float nlz = params[2 * d * d];
  const int64_t m = (int64_t)blockIdx.x * (256 / kWave) + w;
  if (lane < d && m < m_count) XN[w][lane] = xnext[m * d + lane];
  __syncthreads();
  if (m >= m_count) return;
  const Key km = split_at(Key{key[0], key[1]}, (uint32_t)m_count, (uint32_t)m);
  auto pot = [&](int64_t j) {
    for (int k = 0; k < d; ++k) XP[k][t] = xs[j * d + k];
    for (int i = 0; i < d; ++i) {
      float a = 0.f;
      for (int k = 0; k < d; ++k) a += A[i * d + k] * XP[k][t];
      DF[i][t] = XN[w][i] - a;
    }
    float s = 0.f;
    for (int k = 0; k < d; ++k) {
      float v = 0.f;
      for (int i = 0; i < d; ++i) v += DF[i][t] * S[i * d + k];
      s += v * v;
    }
    return 0.5f * s + nlz;
  };
  const int64_t bi = gumbel_argmax(km, (uint32_t)n, lane, 0u, 1u, [&](int64_t j) { return lw[j] - nlz; },
                                   [&](int64_t j) { return lw[j] - pot(j); });
  if (lane == 0 && idx) idx[m] = (int32_t)bi;
  if (lane < d) xout[m * d + lane] = xs[bi * d + lane];
}

// ---------------------------------------------------------------- rejection backward simulation
// mocat/src/ssm/backward.py:42-194 for one backward step (rejection_resampling): initial proposals
// x0[m] = categorical(k0, lw, shape=(M,))[m] with (k0, k1, k2) = split(key_t, 3), densities
// p[m] = exp(-U(x0[m] -> x1[m])), bound = max p * inflation if max p > the initial bound parameter
// (else that parameter), not_yet[m] = uniform(k1, (M,))[m] > p[m] / bound, keys[m] = split(k2, M)[m];
// then rounds while some trajectory waits and fewer than maximum_rejections rounds ran: a waiting
// trajectory splits its key into (key, choice, uniform), proposes categorical(choice, lw), and stays
// waiting iff uniform(uniform) > p / bound; a round whose largest density exceeds the bound raises it
// to that density times the inflation and sends every trajectory back to waiting. Trajectories still
// waiting at the end are drawn by full resampling with their keys. Each round is one launch over the
// trajectories (one wave each) and one single-workgroup launch for the shared bound and counts.
struct RejState {
  float bound;
  int reset;                 // the last round raised the bound: every trajectory proposes again
  int any;                   // some trajectory waits for an acceptance
  int pad;
  unsigned long long evals;  // transition-density evaluations of this step
};

struct RejBuffers {
  uint32_t* keys;   // [M][2]
  int32_t* wait;    // [M] not yet accepted
  int32_t* entered; // [M] proposed in the current round
  float* dens;      // [M] density of the current round's proposal (0 when none)
  RejState* st;
};

// D = 0: the runtime dimension rt_d (LgTransRt); otherwise rt_d is unused
template <class Tr, int D>
__global__ __launch_bounds__(256) void rej_init_kernel(const float* __restrict__ params, const float* __restrict__ xs,
                                                       const float* __restrict__ lw, int64_t n,
                                                       const float* __restrict__ xnext, int64_t M,
                                                       const uint32_t* __restrict__ key, int32_t* __restrict__ idx,
                                                       RejBuffers b, int rt_d) {
  const int64_t DD = D > 0 ? D : rt_d;
  const int lane = threadIdx.x & (kWave - 1);
  const int64_t m = (int64_t)blockIdx.x * (blockDim.x / kWave) + threadIdx.x / kWave;
  if (m >= M) return;
  Tr tr;
  tr.load(params, (int)DD);
  const Key kt{key[0], key[1]};
  const int64_t bi = gumbel_row(split_at(kt, 3, 0), (uint32_t)(M * n), (uint32_t)(m * n), (uint32_t)n, lane,
                                [&](int64_t j) { return lw[j]; });
  if (lane == 0) {
    idx[m] = (int32_t)bi;
    b.dens[m] = expf(-tr.pot(xs + bi * DD, xnext + m * DD));
  }
}

// mode 0: the initial bound from the initial densities, the step's evaluation count set to M;
// mode 1: end of a round (raise the bound if exceeded, count the round's proposals);
// mode 2: end of the step: add n per trajectory resampled in full and write the count out.
__global__ __launch_bounds__(1024) void rej_reduce_kernel(int mode, int64_t M, int64_t n, float init_bound,
                                                          float inflation, RejBuffers b, long long* evals_out) {
  __shared__ float smax[16];
  __shared__ long long scnt[2][16];
  RejState& st = *b.st;
  if (mode == 1 && !st.any) return;
  float mx = 0.f;
  long long c0 = 0, c1 = 0;
  for (int64_t m = threadIdx.x; m < M; m += blockDim.x) {
    mx = fmaxf(mx, b.dens[m]);
    c0 += b.entered[m];
    c1 += b.wait[m];
  }
  mx = wave_max(mx);
  c0 = wave_sum(c0);
  c1 = wave_sum(c1);
  const int w = threadIdx.x / kWave, nw = blockDim.x / kWave;
  if ((threadIdx.x & (kWave - 1)) == 0) {
    smax[w] = mx;
    scnt[0][w] = c0;
    scnt[1][w] = c1;
  }
  __syncthreads();
  if (threadIdx.x != 0) return;
  mx = smax[0];
  c0 = scnt[0][0];
  c1 = scnt[1][0];
  for (int q = 1; q < nw; ++q) {
    mx = fmaxf(mx, smax[q]);
    c0 += scnt[0][q];
    c1 += scnt[1][q];
  }
  if (mode == 0) {
    st.bound = mx > init_bound ? mx * inflation : init_bound;
    st.evals = (unsigned long long)M;
    st.reset = 0;
    st.any = 1;  // decided after the acceptance flags (rej_flags_kernel)
  } else if (mode == 1) {
    const bool reset = mx > st.bound;
    if (reset) st.bound = mx * inflation;
    st.evals += (unsigned long long)c0;
    st.reset = reset ? 1 : 0;
    st.any = (reset || c1 > 0) ? 1 : 0;
  } else {
    st.evals += (unsigned long long)n * (unsigned long long)c0;
    *evals_out = (long long)st.evals;
  }
}

// acceptance flags of the initial proposals and the trajectories' keys; the waiting count in entered
__global__ __launch_bounds__(256) void rej_flags_kernel(int64_t M, const uint32_t* __restrict__ key, RejBuffers b) {
  const int64_t m = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (m >= M) return;
  const Key kt{key[0], key[1]};
  const float u = uniform_from_bits(bits_at(split_at(kt, 3, 1), (uint32_t)M, (uint32_t)m), 0.f, 1.f);
  const int wait = u > b.dens[m] / b.st->bound ? 1 : 0;
  b.wait[m] = wait;
  b.entered[m] = wait;
  const Key km = split_at(split_at(kt, 3, 2), (uint32_t)M, (uint32_t)m);
  b.keys[2 * m] = km.a;
  b.keys[2 * m + 1] = km.b;
  b.dens[m] = 0.f;
}

// whether any trajectory waits after the initial flags (the first round's condition)
__global__ __launch_bounds__(1024) void rej_any_kernel(int64_t M, RejBuffers b) {
  __shared__ int sany;
  if (threadIdx.x == 0) sany = 0;
  __syncthreads();
  int a = 0;
  for (int64_t m = threadIdx.x; m < M; m += blockDim.x) a |= b.wait[m];
  if (a) sany = 1;
  __syncthreads();
  if (threadIdx.x == 0) b.st->any = sany;
}

template <class Tr, int D>
__global__ __launch_bounds__(256) void rej_round_kernel(const float* __restrict__ params, const float* __restrict__ xs,
                                                        const float* __restrict__ lw, int64_t n,
                                                        const float* __restrict__ xnext, int64_t M,
                                                        int32_t* __restrict__ idx, RejBuffers b, int rt_d) {
  const int64_t DD = D > 0 ? D : rt_d;
  const int lane = threadIdx.x & (kWave - 1);
  const int64_t m = (int64_t)blockIdx.x * (blockDim.x / kWave) + threadIdx.x / kWave;
  if (m >= M || !b.st->any) return;
  const bool wait = b.st->reset || b.wait[m];
  if (!wait) {
    if (lane == 0) {
      b.entered[m] = 0;
      b.dens[m] = 0.f;
    }
    return;
  }
  Tr tr;
  tr.load(params, (int)DD);
  const Key k{b.keys[2 * m], b.keys[2 * m + 1]};
  const Key kr = split_at(k, 3, 0), kc = split_at(k, 3, 1), ku = split_at(k, 3, 2);
  const int64_t bi = gumbel_argmax(kc, (uint32_t)n, lane, 0u, 1u, [&](int64_t j) { return lw[j]; },
                                   [&](int64_t j) { return lw[j]; });
  if (lane == 0) {
    const float dd = expf(-tr.pot(xs + bi * DD, xnext + m * DD));
    const float u = uniform_from_bits(bits_at(ku, 1, 0), 0.f, 1.f);
    idx[m] = (int32_t)bi;
    b.dens[m] = dd;
    b.wait[m] = u > dd / b.st->bound ? 1 : 0;
    b.entered[m] = 1;
    b.keys[2 * m] = kr.a;
    b.keys[2 * m + 1] = kr.b;
  }
}

// trajectories still waiting: full resampling with their own keys; then the rows of the step
template <class Tr, int D>
__global__ __launch_bounds__(256) void rej_final_kernel(const float* __restrict__ params, const float* __restrict__ xs,
                                                        const float* __restrict__ lw, int64_t n,
                                                        const float* __restrict__ xnext, int64_t M,
                                                        int32_t* __restrict__ idx, float* __restrict__ xout,
                                                        RejBuffers b, int rt_d) {
  const int64_t DD = D > 0 ? D : rt_d;
  const int lane = threadIdx.x & (kWave - 1);
  const int64_t m = (int64_t)blockIdx.x * (blockDim.x / kWave) + threadIdx.x / kWave;
  if (m >= M) return;
  const bool wait = b.st->any && (b.st->reset || b.wait[m]);
  int64_t bi;
  if (wait) {
    Tr tr;
    tr.load(params, (int)DD);
    const Key k{b.keys[2 * m], b.keys[2 * m + 1]};
    if constexpr (D > 0) {
      float xn[D];
#pragma unroll
      for (int q = 0; q < D; ++q) xn[q] = xnext[m * D + q];
      bi = gumbel_argmax(k, (uint32_t)n, lane, 0u, 1u, [&](int64_t j) { return lw[j] - tr.nlz; },
                         [&](int64_t j) { return lw[j] - tr.pot(xs + j * D, xn); });
    } else {
      const float* xn = xnext + m * DD;
      bi = gumbel_argmax(k, (uint32_t)n, lane, 0u, 1u, [&](int64_t j) { return lw[j] - tr.nlz; },
                         [&](int64_t j) { return lw[j] - tr.pot(xs + j * DD, xn); });
    }
    if (lane == 0) idx[m] = (int32_t)bi;
  } else {
    bi = idx[m];
  }
  if (lane == 0) b.entered[m] = wait ? 1 : 0;
  for (int64_t q = lane; q < DD; q += kWave) xout[m * DD + q] = xs[bi * DD + q];
}

template <class Tr, int D>
int launch_rejection(const float* params, const float* xs, const float* lw, int64_t n, const float* xnext, int64_t M,
                     const uint32_t* key, int max_rejections, float init_bound, float inflation, RejBuffers b,
                     int32_t* idx, float* xout, long long* evals_out, hipStream_t st, int rt_d = D) {
  const int per = 256 / kWave;
  const dim3 waves((unsigned)((M + per - 1) / per)), thr((unsigned)((M + 255) / 256));
  hipLaunchKernelGGL((rej_init_kernel<Tr, D>), waves, dim3(256), 0, st, params, xs, lw, n, xnext, M, key, idx, b,
                     rt_d);
  hipLaunchKernelGGL(rej_reduce_kernel, dim3(1), dim3(1024), 0, st, 0, M, n, init_bound, inflation, b, evals_out);
  hipLaunchKernelGGL(rej_flags_kernel, thr, dim3(256), 0, st, M, key, b);
  hipLaunchKernelGGL(rej_any_kernel, dim3(1), dim3(1024), 0, st, M, b);
  for (int r = 1; r < max_rejections; ++r) {
    hipLaunchKernelGGL((rej_round_kernel<Tr, D>), waves, dim3(256), 0, st, params, xs, lw, n, xnext, M, idx, b, rt_d);
    hipLaunchKernelGGL(rej_reduce_kernel, dim3(1), dim3(1024), 0, st, 1, M, n, init_bound, inflation, b, evals_out);
  }
  hipLaunchKernelGGL((rej_final_kernel<Tr, D>), waves, dim3(256), 0, st, params, xs, lw, n, xnext, M, idx, xout, b,
                     rt_d);
  hipLaunchKernelGGL(rej_reduce_kernel, dim3(1), dim3(1024), 0, st, 2, M, n, init_bound, inflation, b, evals_out);
  MOCAT_LAUNCH_CHECK();
  return MOCAT_OK;
}

int64_t rej_layout(int64_t M, RejBuffers* b, char* base) {
  int64_t o = 0;
  auto take = [&](int64_t bytes) {
    const int64_t at = o;
    o = (o + bytes + 255) / 256 * 256;
    return base ? base + at : nullptr;
  };
  char* keys = take(M * 8);
  char* wait = take(M * 4);
  char* entered = take(M * 4);
  char* dens = take(M * 4);
  char* st = take(sizeof(RejState));
  if (b) *b = RejBuffers{reinterpret_cast<uint32_t*>(keys), reinterpret_cast<int32_t*>(wait),
                         reinterpret_cast<int32_t*>(entered), reinterpret_cast<float*>(dens),
                         reinterpret_cast<RejState*>(st)};
  return o;
}

// (model, d) of the compiled transitions; the linear-Gaussian model runs at any d <= kRtMaxDim without bounds
#define MOCAT_FFBSI_SHAPES(CASE)                                             \
  if (model == 1 && d == 1) CASE(SvTrans, 1);                                \
  if (model == 0 && d == 1) CASE(LgTrans<1>, 1);                             \
  if (model == 0 && d == 2) CASE(LgTrans<2>, 2);                             \
  if (model == 0 && d == 3) CASE(LgTrans<3>, 3);                             \
  if (model == 0 && d == 4) CASE(LgTrans<4>, 4);                             \
  if (model == 0 && d == 5) CASE(LgTrans<5>, 5);                             \
  if (model == 0 && d == 8) CASE(LgTrans<8>, 8);

int ffbsi_step_dispatch(int model, int d, const float* params, const float* particles, const float* log_weight,
                        const float* p, const float* lim, int64_t n, const float* x_next, int64_t m,
                        const uint32_t* key, int32_t* idx, float* x_out, hipStream_t stream) {
#define MOCAT_FFBSI_CASE(TR, DD) \
  return launch_ffbsi<TR, DD>(params, particles, log_weight, p, lim, n, x_next, m, key, idx, x_out, stream)
  MOCAT_FFBSI_SHAPES(MOCAT_FFBSI_CASE)
#undef MOCAT_FFBSI_CASE
  if (model != 0 || d < 1 || d > kRtMaxDim) return MOCAT_ERR_ARG;
  const int per = 256 / kWave;
  hipLaunchKernelGGL(ffbsi_step_rt_kernel, dim3((unsigned)((m + per - 1) / per)), dim3(256), 0, stream, d, params,
                     particles, log_weight, n, x_next, m, key, idx, x_out);
  MOCAT_LAUNCH_CHECK();
  return MOCAT_OK;
}

template <class Tr, int D>
int launch_ffbsi_prep(const float* params, const float* xs, const float* lw, int64_t count, float* p, float* lim,
                      hipStream_t stream) {
  const int64_t blocks = (count + 255) / 256;
  hipLaunchKernelGGL((ffbsi_prep_kernel<Tr, D>), dim3((unsigned)(blocks < 4096 ? blocks : 4096)), dim3(256), 0, stream,
                     params, xs, lw, count, p, lim);
  MOCAT_LAUNCH_CHECK();
  return MOCAT_OK;
}

int ffbsi_prep_dispatch(int model, int d, const float* params, const float* xs, const float* lw, int64_t count,
                        float* p, float* lim, hipStream_t stream) {
#define MOCAT_FFBSI_CASE(TR, DD) return launch_ffbsi_prep<TR, DD>(params, xs, lw, count, p, lim, stream)
  MOCAT_FFBSI_SHAPES(MOCAT_FFBSI_CASE)
#undef MOCAT_FFBSI_CASE
  return MOCAT_ERR_ARG;
}

// Time points whose bounds are prepared together (up to 64 MB of workspace); 0: no bounds, for a dimension
// without a compiled transition and for so few trajectories that preparing costs what it saves.
int64_t ffbsi_step_bytes(int d, int64_t n) { return n * (d + 1) * (int64_t)sizeof(float); }
int64_t ffbsi_block(int model, int d, int64_t T, int64_t n, int64_t m) {
  const bool compiled = model == 1 ? d == 1 : (d >= 1 && d <= 5) || d == 8;
  if (!compiled || m < 16 || T < 2) return 0;
  const int64_t fit = (64ll << 20) / ffbsi_step_bytes(d, n);
  return fit < 1 ? 1 : fit < T - 1 ? fit : T - 1;
}

}  // namespace

extern "C" {

int mocat_ffbsi_rejection_workspace_bytes(int64_t m, int64_t* bytes) {
  if (m <= 0 || !bytes) return MOCAT_ERR_ARG;
  *bytes = rej_layout(m, nullptr, nullptr);
  return MOCAT_OK;
}

int mocat_ffbsi_rejection_step(int model, int d, const float* params, const float* particles, const float* log_weight,
                               int64_t n, const float* x_next, int64_t m, const uint32_t* key, int max_rejections,
                               float init_bound, float bound_inflation, void* workspace, int64_t workspace_bytes,
                               int32_t* idx, float* x_out, long long* evals, hipStream_t stream) {
  if (!params || !particles || !log_weight || !x_next || !key || !workspace || !idx || !x_out || !evals || n <= 0 ||
      m <= 0 || n * m >= 0xFFFFFFFFll || max_rejections < 1)
    return MOCAT_ERR_ARG;
  if (workspace_bytes < rej_layout(m, nullptr, nullptr)) return MOCAT_ERR_SIZE;
  RejBuffers b;
  rej_layout(m, &b, static_cast<char*>(workspace));
#define MOCAT_REJ(TR, DD)                                                                                          \
  return launch_rejection<TR, DD>(params, particles, log_weight, n, x_next, m, key, max_rejections, init_bound,    \
                                  bound_inflation, b, idx, x_out, evals, stream)
  if (model == 1) {
    if (d != 1) return MOCAT_ERR_ARG;
    MOCAT_REJ(SvTrans, 1);
  }
  if (model != 0) return MOCAT_ERR_ARG;
  switch (d) {
    case 1: MOCAT_REJ(LgTrans<1>, 1);
    case 2: MOCAT_REJ(LgTrans<2>, 2);
    case 3: MOCAT_REJ(LgTrans<3>, 3);
    case 4: MOCAT_REJ(LgTrans<4>, 4);
    case 5: MOCAT_REJ(LgTrans<5>, 5);
    case 8: MOCAT_REJ(LgTrans<8>, 8);
    default:
      if (d < 1 || d > kRtMaxDim) return MOCAT_ERR_ARG;
      return launch_rejection<LgTransRt, 0>(params, particles, log_weight, n, x_next, m, key, max_rejections,
                                            init_bound, bound_inflation, b, idx, x_out, evals, stream, d);
  }
#undef MOCAT_REJ
}


int mocat_ffbsi_step(int model, int d, const float* params, const float* particles, const float* log_weight,
                     int64_t n, const float* x_next, int64_t m, const uint32_t* key, int32_t* idx, float* x_out,
                     hipStream_t stream) {
  if (!params || !particles || !log_weight || !x_next || !key || !x_out || n <= 0 || n >= 0xFFFFFFFFll || m <= 0 ||
      m >= 0xFFFFFFFFll)
    return MOCAT_ERR_ARG;
  return ffbsi_step_dispatch(model, d, params, particles, log_weight, nullptr, nullptr, n, x_next, m, key, idx, x_out,
                             stream);
}

int mocat_ffbsi_workspace_bytes(int model, int d, int64_t T, int64_t n, int64_t m, int64_t* bytes) {
  if (d < 1 || T < 1 || n <= 0 || m <= 0 || !bytes) return MOCAT_ERR_ARG;
  *bytes = ffbsi_block(model, d, T, n, m) * ffbsi_step_bytes(d, n);
  return MOCAT_OK;
}

int mocat_ffbsi_run(int model, int d, const float* params, const float* particles, const float* log_weight, int64_t T,
                    int64_t n, int64_t m, const uint32_t* keys, void* workspace, int64_t workspace_bytes, int32_t* idx,
                    float* x_out, hipStream_t stream) {
  if (!params || !particles || !log_weight || !keys || !idx || !x_out || T < 1 || n <= 0 || n >= 0xFFFFFFFFll || m <= 0 ||
      m >= 0xFFFFFFFFll || d < 1)
    return MOCAT_ERR_ARG;
  const int64_t B = ffbsi_block(model, d, T, n, m);
  if (B > 0 && (!workspace || workspace_bytes < B * ffbsi_step_bytes(d, n))) return MOCAT_ERR_SIZE;
  float* p = static_cast<float*>(workspace);
  float* lim = p + B * n * d;
  int64_t lo = T - 1;  // the prepared block starts here
  for (int64_t t = T - 2; t >= 0; --t) {
    if (B > 0 && t < lo) {
      lo = t - B + 1 > 0 ? t - B + 1 : 0;
      const int rc = ffbsi_prep_dispatch(model, d, params, particles + lo * n * d, log_weight + lo * n,
                                         (t - lo + 1) * n, p, lim, stream);
      if (rc != MOCAT_OK) return rc;
    }
    const int rc = ffbsi_step_dispatch(model, d, params, particles + t * n * d, log_weight + t * n,
                                       B > 0 ? p + (t - lo) * n * d : nullptr, B > 0 ? lim + (t - lo) * n : nullptr, n,
                                       x_out + (t + 1) * m * d, m, keys + 2 * t, idx + t * m, x_out + t * m * d, stream);
    if (rc != MOCAT_OK) return rc;
  }
  return MOCAT_OK;
}

}  // extern "C"
