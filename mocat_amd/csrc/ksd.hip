// Kernel Stein discrepancy (mocat/src/metrics.py:88-130) for mocat's Gaussian and IMQ kernels
// (mocat/src/kernels.py:83-111, 164-215), over the full ensemble or over random minibatches.
//
// k_0(x_i, x_j) depends on the pair only through four sums over the coordinates,
//   r2 = |x_i - x_j|^2, a = (x_i - x_j).g_j, b = (x_i - x_j).g_i, c = g_i.g_j,
// so a workgroup takes a 64 x 64 tile of pairs, stages 32-coordinate chunks of both sides in LDS and
// gives each thread a 4 x 4 block of pairs (FP32 sums over the coordinates; the weighted k_0 row
// sums in FP64). Row partial sums over each workgroup's j range go to part[js][i]; the host adds
// them, weights by w_i and divides by (sum w)^2.
//
// The discrepancy itself needs only the sum over all pairs, and k_0(i, j) + k_0(j, i) depends on the pair through
// r2, c and a - b = -(x_i - x_j).(g_i - g_j), so ksd_total_kernel takes the pairs i <= j alone: half the tiles, five
// vector operations per pair and coordinate, which bound it. At n = 4096, d = 100 the row kernel takes 502 us, a
// third of it in the FP64 power of the IMQ kernel (its usual exponent -1/2 is now a reciprocal square root); the
// sum over half the tiles 213 us.
#include "common.hpp"

using namespace mocat;

namespace {

constexpr int kTile = 64, kChunk = 32, kStride = kTile + 4, kKsdThreads = 256;

struct KsdParams {
  int kernel;  // 0 Gaussian, 1 IMQ
  float h, c, beta;
  int d;
};

// base^beta, base^(beta - 1), base^(beta - 2)
MOCAT_DEV void imq_powers(const KsdParams& p, double base, double& kb, double& kb1, double& kb2) {
  if (p.beta == -0.5f) {
    kb = rsqrt(base);
    const double inv = kb * kb;
    kb1 = kb * inv;
    kb2 = kb1 * inv;
    return;
  }
  kb = pow(base, (double)p.beta);
  kb1 = kb / base;
  kb2 = kb1 / base;
}

// mocat's k_0 (metrics.py:116-124) in terms of (r2, a, b, c)
MOCAT_DEV double k0_pair(const KsdParams& p, float r2, float a, float b, float c) {
  const float h2 = p.h * p.h;
  if (p.kernel == 0) {
    // Gaussian: diag_grad_xy summed = (d h^2 - r2) k / h^4, grad_x k = (y - x) k / h^2, grad_y k = (x - y) k / h^2
    const float k = __expf(-0.5f * r2 / h2);
    return (double)k * ((double)((float)p.d * h2 - r2) / ((double)h2 * h2) + (double)(b - a) / h2 + (double)c);
  }
  // IMQ as mocat writes it: base = c + |x - y|^2 / (2 h^2); k = base^beta;
  // grad_x = diff beta base^(beta-1); grad_y = -diff / h beta base^(beta-1);
  // diag_grad_xy = (-beta base^(beta-1) + beta (beta-1) diff^2 base^(beta-2)) / h^2, diff = (x - y) / h
  const double dd = (double)r2 / h2;
  double kb, kb1, kb2;
  imq_powers(p, (double)p.c + 0.5 * dd, kb, kb1, kb2);
  const double beta = p.beta;
  return (-(double)p.d * beta * kb1 + beta * (beta - 1.0) * dd * kb2) / h2 + beta * kb1 * a / p.h -
         beta * kb1 * b / h2 + kb * c;
}

// k_0(x_i, x_j) + k_0(x_j, x_i) in terms of r2, ab = a - b and c (swapping the pair turns (a, b) into (-b, -a)).
MOCAT_DEV double k0_both(const KsdParams& p, float r2, float ab, float c) {
  const double h2 = (double)p.h * p.h;
  if (p.kernel == 0) {
    const float k = __expf(-0.5f * r2 / (float)h2);
    return 2.0 * (double)k * (((double)p.d * h2 - (double)r2) / (h2 * h2) - (double)ab / h2 + (double)c);
  }
  const double dd = (double)r2 / h2, beta = p.beta;
  double kb, kb1, kb2;
  imq_powers(p, (double)p.c + 0.5 * dd, kb, kb1, kb2);
  return 2.0 * (beta * (beta - 1.0) * dd * kb2 - (double)p.d * beta * kb1) / h2 +
         beta * kb1 * (double)ab * (1.0 / p.h + 1.0 / h2) + 2.0 * kb * c;
}

__global__ __launch_bounds__(kKsdThreads) void ksd_rows_kernel(const float* __restrict__ x,
                                                               const float* __restrict__ g,
                                                               const float* __restrict__ w, int n, KsdParams p,
                                                               int js_count, double* __restrict__ part) {
  __shared__ alignas(16) float xi[kChunk][kStride], gi[kChunk][kStride], xj[kChunk][kStride], gj[kChunk][kStride];
  __shared__ double red[kKsdThreads / 16][kTile];
  const int t = threadIdx.x, ti = t & 15, tj = t >> 4;
  const int i0 = blockIdx.x * kTile, js = blockIdx.y;
  const int d = p.d;
  const int ntiles = (n + kTile - 1) / kTile;
  double rows[4] = {0.0, 0.0, 0.0, 0.0};
  for (int jt = js; jt < ntiles; jt += js_count) {
    const int j0 = jt * kTile;
    float r2[4][4], sa[4][4], sb[4][4], sc[4][4];
#pragma unroll
    for (int u = 0; u < 4; ++u)
#pragma unroll
      for (int v = 0; v < 4; ++v) r2[u][v] = sa[u][v] = sb[u][v] = sc[u][v] = 0.f;
    for (int k0 = 0; k0 < d; k0 += kChunk) {
      __syncthreads();
      for (int e = t; e < kTile * kChunk; e += kKsdThreads) {
        const int row = e / kChunk, k = e - row * kChunk;
        const bool kin = k0 + k < d;
        const int ii = i0 + row, jj = j0 + row;
        xi[k][row] = (kin && ii < n) ? x[(int64_t)ii * d + k0 + k] : 0.f;
        gi[k][row] = (kin && ii < n) ? g[(int64_t)ii * d + k0 + k] : 0.f;
        xj[k][row] = (kin && jj < n) ? x[(int64_t)jj * d + k0 + k] : 0.f;
        gj[k][row] = (kin && jj < n) ? g[(int64_t)jj * d + k0 + k] : 0.f;
      }
      __syncthreads();
      const int kn = min(kChunk, d - k0);
      for (int k = 0; k < kn; ++k) {
        const float4 xa = *reinterpret_cast<const float4*>(&xi[k][ti * 4]);
        const float4 ga = *reinterpret_cast<const float4*>(&gi[k][ti * 4]);
        const float4 xb = *reinterpret_cast<const float4*>(&xj[k][tj * 4]);
        const float4 gb = *reinterpret_cast<const float4*>(&gj[k][tj * 4]);
        const float xv[4] = {xa.x, xa.y, xa.z, xa.w}, gv[4] = {ga.x, ga.y, ga.z, ga.w};
        const float yv[4] = {xb.x, xb.y, xb.z, xb.w}, hv[4] = {gb.x, gb.y, gb.z, gb.w};
#pragma unroll
        for (int u = 0; u < 4; ++u)
#pragma unroll
          for (int v = 0; v < 4; ++v) {
            const float df = xv[u] - yv[v];
            r2[u][v] = fmaf(df, df, r2[u][v]);
            sa[u][v] = fmaf(df, hv[v], sa[u][v]);
            sb[u][v] = fmaf(df, gv[u], sb[u][v]);
            sc[u][v] = fmaf(gv[u], hv[v], sc[u][v]);
          }
      }
    }
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int j = j0 + tj * 4 + v;
      if (j >= n) continue;
      const double wj = w ? (double)w[j] : 1.0;
#pragma unroll
      for (int u = 0; u < 4; ++u) rows[u] += wj * k0_pair(p, r2[u][v], sa[u][v], sb[u][v], sc[u][v]);
    }
  }
  // fixed-order sum over the 16 thread columns of each row
#pragma unroll
  for (int u = 0; u < 4; ++u) red[tj][ti * 4 + u] = rows[u];
  __syncthreads();
  if (t < kTile && i0 + t < n) {
    double s = 0.0;
    for (int q = 0; q < kKsdThreads / 16; ++q) s += red[q][t];
    part[(int64_t)js * n + i0 + t] = s;
  }
}

// Tile pair k of the upper triangle (row tile <= column tile), rows in order: column tile J holds the pairs
// J (J + 1) / 2 .. J (J + 1) / 2 + J.
MOCAT_DEV void upper_pair(int64_t k, int& I, int& J) {
  int64_t j = (int64_t)((sqrt(8.0 * (double)k + 1.0) - 1.0) * 0.5);
  while (j * (j + 1) / 2 > k) --j;
  while ((j + 1) * (j + 2) / 2 <= k) ++j;
  J = (int)j;
  I = (int)(k - j * (j + 1) / 2);
}

// part[workgroup] = sum over the workgroup's pairs i <= j of w_i w_j (k_0(i, j) + k_0(j, i)), the diagonal once.
__global__ __launch_bounds__(kKsdThreads) void ksd_total_kernel(const float* __restrict__ x,
                                                                const float* __restrict__ g,
                                                                const double* __restrict__ w, int n, KsdParams p,
                                                                int64_t pairs, double* __restrict__ part) {
  __shared__ alignas(16) float xi[kChunk][kStride], gi[kChunk][kStride], xj[kChunk][kStride], gj[kChunk][kStride];
  __shared__ double red[kKsdThreads / kWave];
  const int t = threadIdx.x, ti = t & 15, tj = t >> 4;
  const int d = p.d;
  double sum = 0.0;
  for (int64_t k = blockIdx.x; k < pairs; k += gridDim.x) {
    int I, J;
    upper_pair(k, I, J);
    const int i0 = I * kTile, j0 = J * kTile;
    float r2[4][4], se[4][4], sc[4][4];
#pragma unroll
    for (int u = 0; u < 4; ++u)
#pragma unroll
      for (int v = 0; v < 4; ++v) r2[u][v] = se[u][v] = sc[u][v] = 0.f;
    for (int k0 = 0; k0 < d; k0 += kChunk) {
      __syncthreads();
      for (int e = t; e < kTile * kChunk; e += kKsdThreads) {
        const int row = e / kChunk, kk = e - row * kChunk;
        const bool kin = k0 + kk < d;
        const int ii = i0 + row, jj = j0 + row;
        xi[kk][row] = (kin && ii < n) ? x[(int64_t)ii * d + k0 + kk] : 0.f;
        gi[kk][row] = (kin && ii < n) ? g[(int64_t)ii * d + k0 + kk] : 0.f;
        xj[kk][row] = (kin && jj < n) ? x[(int64_t)jj * d + k0 + kk] : 0.f;
        gj[kk][row] = (kin && jj < n) ? g[(int64_t)jj * d + k0 + kk] : 0.f;
      }
      __syncthreads();
      const int kn = min(kChunk, d - k0);
#pragma unroll 2
      for (int kk = 0; kk < kn; ++kk) {
        const float4 xa = *reinterpret_cast<const float4*>(&xi[kk][ti * 4]);
        const float4 ga = *reinterpret_cast<const float4*>(&gi[kk][ti * 4]);
        const float4 xb = *reinterpret_cast<const float4*>(&xj[kk][tj * 4]);
        const float4 gb = *reinterpret_cast<const float4*>(&gj[kk][tj * 4]);
        const float xv[4] = {xa.x, xa.y, xa.z, xa.w}, gv[4] = {ga.x, ga.y, ga.z, ga.w};
        const float yv[4] = {xb.x, xb.y, xb.z, xb.w}, hv[4] = {gb.x, gb.y, gb.z, gb.w};
#pragma unroll
        for (int u = 0; u < 4; ++u)
#pragma unroll
          for (int v = 0; v < 4; ++v) {
            const float df = xv[u] - yv[v], dg = hv[v] - gv[u];
            r2[u][v] = fmaf(df, df, r2[u][v]);
            se[u][v] = fmaf(df, dg, se[u][v]);  // a - b
            sc[u][v] = fmaf(gv[u], hv[v], sc[u][v]);
          }
      }
    }
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int j = j0 + tj * 4 + v;
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int i = i0 + ti * 4 + u;
        if (j >= n || i > j) continue;  // i <= j < n
        const double ww = w ? w[i] * w[j] : 1.0;
        sum += (i == j ? 0.5 : 1.0) * ww * k0_both(p, r2[u][v], se[u][v], sc[u][v]);
      }
    }
  }
  sum = wave_sum(sum);
  if ((t & (kWave - 1)) == 0) red[t / kWave] = sum;
  __syncthreads();
  if (t == 0) {
    for (int q = 1; q < kKsdThreads / kWave; ++q) sum += red[q];
    part[blockIdx.x] = sum;
  }
}

// out = sqrt(sum of the parts) / sum of the weights (n without weights)
__global__ __launch_bounds__(kKsdThreads) void ksd_finish_kernel(const double* __restrict__ part, int64_t parts,
                                                                 const double* __restrict__ w, int64_t n,
                                                                 double* out) {
  __shared__ double red[2][kKsdThreads / kWave];
  const int t = threadIdx.x;
  double a = 0.0, b = 0.0;
  for (int64_t k = t; k < parts; k += kKsdThreads) a += part[k];
  if (w)
    for (int64_t k = t; k < n; k += kKsdThreads) b += w[k];
  a = wave_sum(a);
  b = wave_sum(b);
  if ((t & (kWave - 1)) == 0) {
    red[0][t / kWave] = a;
    red[1][t / kWave] = b;
  }
  __syncthreads();
  if (t == 0) {
    for (int q = 1; q < kKsdThreads / kWave; ++q) {
      a += red[0][q];
      b += red[1][q];
    }
    const double s = w ? b : (double)n;
    *out = sqrt(a / (s * s));
  }
}

// Minibatch rows: one wave per particle i; lane b takes batch entries b, b + 64, ... and sums the
// four coordinate sums of its pair in coordinate order (FP32, as the tile kernel), then k_0 in FP64;
// the lanes' FP64 partial sums are combined by a fixed butterfly.
__global__ __launch_bounds__(256) void ksd_batch_kernel(const float* __restrict__ x, const float* __restrict__ g,
                                                        const float* __restrict__ w, int n, int64_t batch,
                                                        const int32_t* __restrict__ inds, KsdParams p,
                                                        double* __restrict__ row_k, double* __restrict__ row_w) {
  const int lane = threadIdx.x & (kWave - 1);
  const int64_t i = (int64_t)blockIdx.x * (blockDim.x / kWave) + threadIdx.x / kWave;
  if (i >= n) return;
  const int d = p.d;
  const float* xi = x + i * d;
  const float* gi = g + i * d;
  double sk = 0.0, sw = 0.0;
  for (int64_t b = lane; b < batch; b += kWave) {
    const int64_t j = inds[i * batch + b];
    const float* xj = x + j * d;
    const float* gj = g + j * d;
    float r2 = 0.f, a = 0.f, bb = 0.f, c = 0.f;
    for (int k = 0; k < d; ++k) {
      const float df = xi[k] - xj[k];
      r2 = fmaf(df, df, r2);
      a = fmaf(df, gj[k], a);
      bb = fmaf(df, gi[k], bb);
      c = fmaf(gi[k], gj[k], c);
    }
    const double wj = w ? (double)w[j] : 1.0;
    sk += wj * k0_pair(p, r2, a, bb, c);
    sw += wj;
  }
  sk = wave_sum(sk);
  sw = wave_sum(sw);
  if (lane == 0) {
    row_k[i] = sk;
    row_w[i] = sw;
  }
}

// workgroups of the total: one per tile pair, up to eight waves per SIMD on 256 CUs
constexpr int64_t kKsdMaxParts = 8192;

int64_t ksd_parts(int64_t n) {
  const int64_t tiles = (n + kTile - 1) / kTile, pairs = tiles * (tiles + 1) / 2;
  return pairs < kKsdMaxParts ? pairs : kKsdMaxParts;
}

}  // namespace

extern "C" {

int mocat_ksd_rows(const float* x, const float* grad_potential, const float* weights, int64_t n, int64_t d,
                   int kernel, float bandwidth, float c, float beta, int js_count, double* part,
                   hipStream_t stream) {
  if (!x || !grad_potential || !part || n <= 0 || n > (1 << 24) || d <= 0 || d > (1 << 16) || js_count <= 0 ||
      js_count > 65535 || (kernel != 0 && kernel != 1) || !(bandwidth > 0.f) || (kernel == 1 && !(c > 0.f)))
    return MOCAT_ERR_ARG;
  const KsdParams p{kernel, bandwidth, c, beta, (int)d};
  hipLaunchKernelGGL(ksd_rows_kernel, dim3((unsigned)((n + kTile - 1) / kTile), (unsigned)js_count),
                     dim3(kKsdThreads), 0, stream, x, grad_potential, weights, (int)n, p, js_count, part);
  MOCAT_LAUNCH_CHECK();
  return MOCAT_OK;
}

int mocat_ksd_workspace_bytes(int64_t n, int64_t* bytes) {
  if (n <= 0 || n > (1 << 24) || !bytes) return MOCAT_ERR_ARG;
  *bytes = ksd_parts(n) * (int64_t)sizeof(double);
  return MOCAT_OK;
}

int mocat_ksd(const float* x, const float* grad_potential, const double* weights, int64_t n, int64_t d, int kernel,
              float bandwidth, float c, float beta, void* workspace, int64_t workspace_bytes, double* out,
              hipStream_t stream) {
  if (!x || !grad_potential || !workspace || !out || n <= 0 || n > (1 << 24) || d <= 0 || d > (1 << 16) ||
      (kernel != 0 && kernel != 1) || !(bandwidth > 0.f) || (kernel == 1 && !(c > 0.f)))
    return MOCAT_ERR_ARG;
  const int64_t parts = ksd_parts(n), tiles = (n + kTile - 1) / kTile;
  if (workspace_bytes < parts * (int64_t)sizeof(double)) return MOCAT_ERR_SIZE;
  const KsdParams p{kernel, bandwidth, c, beta, (int)d};
  double* part = static_cast<double*>(workspace);
  hipLaunchKernelGGL(ksd_total_kernel, dim3((unsigned)parts), dim3(kKsdThreads), 0, stream, x, grad_potential, weights,
                     (int)n, p, tiles * (tiles + 1) / 2, part);
  hipLaunchKernelGGL(ksd_finish_kernel, dim3(1), dim3(kKsdThreads), 0, stream, (const double*)part, parts, weights, n,
                     out);
  MOCAT_LAUNCH_CHECK();
  return MOCAT_OK;
}

int mocat_ksd_batch_rows(const float* x, const float* grad_potential, const float* weights, int64_t n, int64_t d,
                         int64_t batch, const int32_t* inds, int kernel, float bandwidth, float c, float beta,
                         double* row_k, double* row_w, hipStream_t stream) {
  if (!x || !grad_potential || !inds || !row_k || !row_w || n <= 0 || n > (1 << 24) || d <= 0 || d > (1 << 16) ||
      batch <= 0 || batch > (1ll << 31) / n || (kernel != 0 && kernel != 1) || !(bandwidth > 0.f) ||
      (kernel == 1 && !(c > 0.f)))
    return MOCAT_ERR_ARG;
  const KsdParams p{kernel, bandwidth, c, beta, (int)d};
  const int per = 256 / kWave;
  hipLaunchKernelGGL(ksd_batch_kernel, dim3((unsigned)((n + per - 1) / per)), dim3(256), 0, stream, x, grad_potential,
                     weights, (int)n, batch, inds, p, row_k, row_w);
  MOCAT_LAUNCH_CHECK();
  return MOCAT_OK;
}

}  // extern "C"
