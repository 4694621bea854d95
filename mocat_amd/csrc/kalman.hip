// Kalman filter and Rauch-Tung-Striebel smoother of a linear-Gaussian model in FP64
// (mocat/src/ssm/linear_gaussian/kalman.py:16-98), state and observation dimensions up to 8.
//
// The recursions are serial in time and tiny (4 x 4 matrices for the usual models), so latency is all there
// is: as separate matrix operations a filter step was about 45 launches (53 ms for filter and smoother over
// 100 steps). Here one wave runs the whole filter: matrices in LDS, one element per lane, the
// Cholesky factor in every lane's registers, each lane solving for one column of the gain. The smoother's
// gains and predictions do not depend on each other and take a wave per time point; what is left to the serial
// wave is m = f + J (m' - A f) and P = F + J (P' - pred) J^T.
//
// Both dimensions are padded to M = max(d, dy) (compiled for 1 to 8): padding states have A = 0, Q = 1 and no
// observation, padding observations y = 0, H = 0 and R = 1, which leaves the others' values as they are.
#include "common.hpp"

using namespace mocat;

namespace {

struct KfModel {  // device pointers, row-major, padded to M
  const double *A, *Q, *H, *R, *m0, *P0, *y;
};

// f(row, column, element) for the M x M elements, one per lane
template <int M, class F>
MOCAT_DEV void each(F f) {
#pragma unroll
  for (int e0 = 0; e0 < M * M; e0 += kWave) {
    const int e = e0 + (int)threadIdx.x;
    if (e < M * M) f(e / M, e % M, e);
  }
}

// Whether each lane's elements of a covariance (LDS) equal their mirror images but for rounding.
template <int M>
MOCAT_DEV bool symmetric(const double* s) {
  bool ok = true;
  each<M>([&](int i, int j, int e) {
    ok = ok && !(fabs(s[e] - s[j * M + i]) > 1e-9 * (fabs(s[i * M + i]) + fabs(s[j * M + j])));
  });
  return ok;
}

// Lower Cholesky factor of the symmetric matrix s (LDS, lower triangle read) in registers, diagonal as
// its reciprocal too; false if it is not positive definite (or not a number).
template <int M>
MOCAT_DEV bool cholesky(const double* s, double (&L)[M][M], double (&inv)[M]) {
  bool ok = true;
#pragma unroll
  for (int j = 0; j < M; ++j) {
    double v = s[j * M + j];
#pragma unroll
    for (int k = 0; k < j; ++k) v -= L[j][k] * L[j][k];
    ok = ok && v > 0.0;
    const double r = sqrt(v);
    L[j][j] = r;
    inv[j] = 1.0 / r;
#pragma unroll
    for (int i = j + 1; i < M; ++i) {
      double u = s[i * M + j];
#pragma unroll
      for (int k = 0; k < j; ++k) u -= L[i][k] * L[j][k];
      L[i][j] = u * inv[j];
    }
  }
  return ok;
}

// x <- (L L^T)^-1 x
template <int M>
MOCAT_DEV void solve(const double (&L)[M][M], const double (&inv)[M], double (&x)[M]) {
#pragma unroll
  for (int i = 0; i < M; ++i) {
#pragma unroll
    for (int k = 0; k < i; ++k) x[i] -= L[i][k] * x[k];
    x[i] *= inv[i];
  }
#pragma unroll
  for (int i = M - 1; i >= 0; --i) {
#pragma unroll
    for (int k = i + 1; k < M; ++k) x[i] -= L[k][i] * x[k];
    x[i] *= inv[i];
  }
}

// stats: [T][M + 1] scratch (the factors' diagonals and the innovations' quadratic forms, whose logarithms are
// summed at the end, off the serial path); info: set to 1 when an innovation covariance has no Cholesky factor, and when
// P0 or Q, whose symmetry the gain uses, is not symmetric.
template <int M>
__global__ __launch_bounds__(kWave) void kalman_filter_kernel(KfModel g, int64_t T, int d, int dy, double* means,
                                                              double* covs, double* loglik, double* stats, int* info) {
  __shared__ double A[M * M], Q[M * M], H[M * M], R[M * M], P[M * M], W[M * M], B[M * M], S[M * M], K[M * M];
  __shared__ double m[M], mp[M], r[M];
  const int lane = threadIdx.x;
  each<M>([&](int, int, int e) {
    A[e] = g.A[e];
    Q[e] = g.Q[e];
    H[e] = g.H[e];
    R[e] = g.R[e];
    P[e] = g.P0[e];
  });
  if (lane < M) m[lane] = g.m0[lane];
  __syncthreads();
  bool ok = symmetric<M>(P) && symmetric<M>(Q);
  double yt = lane < M ? g.y[lane] : 0.0;
  for (int64_t t = 0; t < T; ++t) {
    const double ynext = (lane < M && t + 1 < T) ? g.y[(t + 1) * M + lane] : 0.0;
    __syncthreads();
    if (t > 0) {  // predict: m = A m, P = A P A^T + Q
      each<M>([&](int i, int j, int e) {
        double v = 0.0;
#pragma unroll
        for (int k = 0; k < M; ++k) v += A[i * M + k] * P[k * M + j];
        W[e] = v;
      });
      if (lane < M) {
        double v = 0.0;
#pragma unroll
        for (int k = 0; k < M; ++k) v += A[lane * M + k] * m[k];
        mp[lane] = v;
      }
      __syncthreads();
      each<M>([&](int i, int j, int e) {
        double v = 0.0;
#pragma unroll
        for (int k = 0; k < M; ++k) v += W[i * M + k] * A[j * M + k];
        P[e] = v + Q[e];
      });
    } else if (lane < M) {
      mp[lane] = m[lane];
    }
    __syncthreads();
    // B = H P, r = y - H m
    each<M>([&](int i, int j, int e) {
      double v = 0.0;
#pragma unroll
      for (int k = 0; k < M; ++k) v += H[i * M + k] * P[k * M + j];
      B[e] = v;
    });
    if (lane < M) {
      double v = 0.0;
#pragma unroll
      for (int k = 0; k < M; ++k) v += H[lane * M + k] * mp[k];
      r[lane] = yt - v;
    }
    __syncthreads();
    each<M>([&](int i, int j, int e) {
      double v = 0.0;
#pragma unroll
      for (int k = 0; k < M; ++k) v += B[i * M + k] * H[j * M + k];
      S[e] = v + R[e];
    });
    __syncthreads();
    double L[M][M], inv[M], x[M];
    ok = cholesky<M>(S, L, inv) && ok;
    // lane i < M: column i of S^-1 B, i.e. row i of the gain; lane M: S^-1 r
#pragma unroll
    for (int k = 0; k < M; ++k) x[k] = lane < M ? B[k * M + lane] : r[k];
    solve<M>(L, inv, x);
    if (lane < M) {
      double v = mp[lane];
#pragma unroll
      for (int k = 0; k < M; ++k) {
        K[lane * M + k] = x[k];
        v += x[k] * r[k];
      }
      m[lane] = v;
      if (lane < d) means[t * d + lane] = v;
    } else if (lane == M) {
      double q = 0.0;
#pragma unroll
      for (int k = 0; k < M; ++k) {
        q += r[k] * x[k];
        stats[t * (M + 1) + k] = L[k][k];
      }
      stats[t * (M + 1) + M] = q;
    }
    __syncthreads();
    each<M>([&](int i, int j, int e) {
      double v = 0.0;
#pragma unroll
      for (int k = 0; k < M; ++k) v += K[i * M + k] * B[k * M + j];
      v = P[e] - v;
      W[e] = v;
      if (i < d && j < d) covs[(t * d + i) * d + j] = v;
    });
    __syncthreads();
    each<M>([&](int, int, int e) { P[e] = W[e]; });
    yt = ynext;
  }
  __threadfence();
  __syncthreads();
  double ll = 0.0;
  for (int64_t t = lane; t < T; t += kWave) {
    double q = stats[t * (M + 1) + M] + dy * 1.83787706640934548356;
    for (int k = 0; k < M; ++k) q += 2.0 * log(stats[t * (M + 1) + k]);
    ll -= 0.5 * q;
  }
  ll = wave_sum(ll);
  ok = __all(ok);
  if (lane == 0) {
    *loglik = ll;
    *info = ok ? 0 : 1;
  }
}

// One wave per time point t < T - 1: pred = A F_t A^T + Q and the gain J = F_t A^T pred^-1, to [T - 1][M][M] each.
// J uses F_t = F_t^T and pred = pred^T, and the filter covariances are the caller's: info is also set where F_t or Q is
// not symmetric.
template <int M>
__global__ __launch_bounds__(kWave) void kalman_gain_kernel(KfModel g, int d, const double* f_covs, double* gains,
                                                            double* preds, int* info) {
  __shared__ double A[M * M], Q[M * M], F[M * M], B[M * M], S[M * M];
  const int lane = threadIdx.x;
  const int64_t t = blockIdx.x;
  each<M>([&](int i, int j, int e) {
    A[e] = g.A[e];
    Q[e] = g.Q[e];
    F[e] = (i < d && j < d) ? f_covs[(t * d + i) * d + j] : 0.0;
  });
  __syncthreads();
  each<M>([&](int i, int j, int e) {
    double v = 0.0;
#pragma unroll
    for (int k = 0; k < M; ++k) v += A[i * M + k] * F[k * M + j];
    B[e] = v;
  });
  __syncthreads();
  each<M>([&](int i, int j, int e) {
    double v = 0.0;
#pragma unroll
    for (int k = 0; k < M; ++k) v += B[i * M + k] * A[j * M + k];
    v += Q[e];
    S[e] = v;
    preds[t * M * M + e] = v;
  });
  __syncthreads();
  double L[M][M], inv[M], x[M];
  const bool ok = cholesky<M>(S, L, inv);
  if (!ok || !symmetric<M>(F) || !symmetric<M>(Q)) *info = 1;
  if (lane < M) {
#pragma unroll
    for (int k = 0; k < M; ++k) x[k] = B[k * M + lane];
    solve<M>(L, inv, x);
#pragma unroll
    for (int k = 0; k < M; ++k) gains[(t * M + lane) * M + k] = x[k];
  }
}

// The backward recursion by one wave; the next time point's gain, prediction and filter moments are read one
// step ahead.
template <int M>
__global__ __launch_bounds__(kWave) void kalman_smooth_kernel(KfModel g, int64_t T, int d, const double* f_means,
                                                              const double* f_covs, const double* gains,
                                                              const double* preds, double* means, double* covs) {
  constexpr int E = (M * M + kWave - 1) / kWave;
  __shared__ double A[M * M], J[M * M], D[M * M], W[M * M], fm[M], m[M], dm[M];
  const int lane = threadIdx.x;
  each<M>([&](int, int, int e) { A[e] = g.A[e]; });
  double cov[E], nj[E], np[E], nf[E], nm = 0.0;
  auto fetch = [&](int64_t t) {
#pragma unroll
    for (int q = 0; q < E; ++q) {
      const int e = q * kWave + lane, i = e / M, j = e % M;
      const bool in = e < M * M && t >= 0;
      nj[q] = in ? gains[t * M * M + e] : 0.0;
      np[q] = in ? preds[t * M * M + e] : 0.0;
      nf[q] = in && i < d && j < d ? f_covs[(t * d + i) * d + j] : 0.0;
    }
    nm = lane < d && t >= 0 ? f_means[t * d + lane] : 0.0;
  };
#pragma unroll
  for (int q = 0; q < E; ++q) {
    const int e = q * kWave + lane, i = e / M, j = e % M;
    cov[q] = e < M * M && i < d && j < d ? f_covs[((T - 1) * d + i) * d + j] : 0.0;
    if (e < M * M && i < d && j < d) covs[((T - 1) * d + i) * d + j] = cov[q];
  }
  if (lane < M) {
    m[lane] = lane < d ? f_means[(T - 1) * d + lane] : 0.0;
    if (lane < d) means[(T - 1) * d + lane] = m[lane];
  }
  fetch(T - 2);
  for (int64_t t = T - 2; t >= 0; --t) {
    double cf[E];
#pragma unroll
    for (int q = 0; q < E; ++q) {
      const int e = q * kWave + lane;
      cf[q] = nf[q];
      if (e < M * M) {
        J[e] = nj[q];
        D[e] = cov[q] - np[q];
      }
    }
    if (lane < M) fm[lane] = nm;
    fetch(t - 1);
    __syncthreads();
    each<M>([&](int i, int j, int e) {
      double v = 0.0;
#pragma unroll
      for (int k = 0; k < M; ++k) v += J[i * M + k] * D[k * M + j];
      W[e] = v;
    });
    if (lane < M) {
      double v = 0.0;
#pragma unroll
      for (int k = 0; k < M; ++k) v += A[lane * M + k] * fm[k];
      dm[lane] = m[lane] - v;
    }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < E; ++q) {
      const int e = q * kWave + lane, i = e / M, j = e % M;
      if (e >= M * M) continue;
      double v = 0.0;
#pragma unroll
      for (int k = 0; k < M; ++k) v += W[i * M + k] * J[j * M + k];
      cov[q] = cf[q] + v;
      if (i < d && j < d) covs[(t * d + i) * d + j] = cov[q];
    }
    if (lane < M) {
      double v = fm[lane];
#pragma unroll
      for (int k = 0; k < M; ++k) v += J[lane * M + k] * dm[k];
      m[lane] = v;
      if (lane < d) means[t * d + lane] = v;
    }
    __syncthreads();
  }
}

// mocat's lag-one term (kalman.py:79-80), one wave per t: f_t . m_t+1 + J_t (P_t+1 + (m_t+1 - f_t+1) . m_t+1)
template <int M>
__global__ __launch_bounds__(kWave) void kalman_lag_kernel(int d, const double* f_means, const double* gains,
                                                           const double* means, const double* covs, double* lags) {
  const int64_t t = blockIdx.x;
  const double *f0 = f_means + t * d, *f1 = f0 + d, *m1 = means + (t + 1) * d, *P1 = covs + (t + 1) * d * d;
  double s1 = 0.0, s2 = 0.0;
  for (int k = 0; k < d; ++k) {
    s1 += f0[k] * m1[k];
    s2 += (m1[k] - f1[k]) * m1[k];
  }
  for (int e = threadIdx.x; e < d * d; e += kWave) {
    const int i = e / d, j = e % d;
    double v = 0.0;
    for (int k = 0; k < d; ++k) v += gains[(t * M + i) * M + k] * (P1[k * d + j] + s2);
    lags[t * d * d + e] = s1 + v;
  }
}

// The packed model: A, Q, H, R, P0 (M x M each), m0 (M), then y (T x M); the smoother reads A and Q only.
KfModel unpack(const double* model, int M) {
  const int64_t q = (int64_t)M * M;
  return KfModel{model, model + q, model + 2 * q, model + 3 * q, model + 5 * q, model + 4 * q, model + 5 * q + M};
}

template <int M>
int launch_filter(const double* model, int64_t T, int d, int dy, double* means, double* covs, double* loglik,
                  double* stats, int* info, hipStream_t st) {
  hipLaunchKernelGGL((kalman_filter_kernel<M>), dim3(1), dim3(kWave), 0, st, unpack(model, M), T, d, dy, means, covs,
                     loglik, stats, info);
  MOCAT_LAUNCH_CHECK();
  return MOCAT_OK;
}

template <int M>
int launch_smoother(const double* model, int64_t T, int d, const double* f_means, const double* f_covs, double* means,
                    double* covs, double* lags, double* ws, int* info, hipStream_t st) {
  const KfModel g = unpack(model, M);
  double *gains = ws, *preds = ws + (T - 1) * M * M;
  if (T > 1)
    hipLaunchKernelGGL((kalman_gain_kernel<M>), dim3((unsigned)(T - 1)), dim3(kWave), 0, st, g, d, f_covs, gains, preds,
                       info);
  hipLaunchKernelGGL((kalman_smooth_kernel<M>), dim3(1), dim3(kWave), 0, st, g, T, d, f_means, f_covs, gains, preds,
                     means, covs);
  if (T > 1)
    hipLaunchKernelGGL((kalman_lag_kernel<M>), dim3((unsigned)(T - 1)), dim3(kWave), 0, st, d, f_means, gains, means,
                       covs, lags);
  MOCAT_LAUNCH_CHECK();
  return MOCAT_OK;
}

}  // namespace

extern "C" {

int mocat_kalman_filter(const double* model, int m_pad, int64_t T, int d, int dy, double* means, double* covs,
                        double* loglik, double* scratch, int* info, hipStream_t stream) {
  if (!model || !means || !covs || !loglik || !scratch || !info || T < 1 || d < 1 || dy < 1 || d > m_pad ||
      dy > m_pad)
    return MOCAT_ERR_ARG;
#define MOCAT_KF(MM) \
  case MM: return launch_filter<MM>(model, T, d, dy, means, covs, loglik, scratch, info, stream)
  switch (m_pad) {
    MOCAT_KF(1);
    MOCAT_KF(2);
    MOCAT_KF(3);
    MOCAT_KF(4);
    MOCAT_KF(5);
    MOCAT_KF(6);
    MOCAT_KF(7);
    MOCAT_KF(8);
    default: return MOCAT_ERR_ARG;
  }
#undef MOCAT_KF
}

int mocat_kalman_smoother(const double* model, int m_pad, int64_t T, int d, const double* filter_means,
                          const double* filter_covs, double* means, double* covs, double* lag_ones, double* scratch,
                          int* info, hipStream_t stream) {
  if (!model || !filter_means || !filter_covs || !means || !covs || !info || T < 1 || T > 0x7FFFFFFFll || d < 1 ||
      d > m_pad || (T > 1 && (!lag_ones || !scratch)))
    return MOCAT_ERR_ARG;
#define MOCAT_KS(MM)                                                                                              \
  case MM: return launch_smoother<MM>(model, T, d, filter_means, filter_covs, means, covs, lag_ones, scratch, info, \
                                      stream)
  switch (m_pad) {
    MOCAT_KS(1);
    MOCAT_KS(2);
    MOCAT_KS(3);
    MOCAT_KS(4);
    MOCAT_KS(5);
    MOCAT_KS(6);
    MOCAT_KS(7);
    MOCAT_KS(8);
    default: return MOCAT_ERR_ARG;
  }
#undef MOCAT_KS
}

}  // extern "C"
