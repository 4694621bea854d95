// Gumbel-max draws by whole wavefronts: argmax_j gumbel_j + logit_j, the first maximum, as
// random.categorical (mocat/src/ssm/filtering.py:196-199, mocat/src/ssm/backward.py:20-39). The draws are
// elements of a jax.random bits array (halves layout), gumbel = -log(-log(uniform(tiny, 1))).
//
// What bounds it: one threefry block per one or two draws (about 70 integer operations a block), then the
// two accurate logarithms of each draw. Most draws cannot win, and a bound shows it without the logarithms:
// with f the draw's uniform, -log(f) >= 1 - f, so gumbel <= -log(1 - f), and 1 - f is exact in FP32. The
// bound takes one v_log_f32 and a margin (1e-4, above the error of v_log_f32 and of both logf's: a draw's
// Gumbel is at most 16); adding the logit rounds monotonically, so a candidate whose bound is below the
// best value seen by the wave is below it too, and is dropped without changing the result. A candidate that
// is not dropped, a few per row (the chance of a new best falls as one over the draws seen), takes the exact
// value.
//
// A NaN score is never better than a number: its particle is drawn as if its log-weight were -inf, whichever lanes and
// waves share the row and whether or not the bound drops it. Only a row whose first score is NaN takes index 0.
#pragma once
#include "common.hpp"

namespace mocat {

constexpr float kGumbelTiny = 1.17549435e-38f;  // float32 tiny: the lower end of jax's gumbel uniforms
constexpr uint32_t kNoIndex = 0xffffffffu;

MOCAT_DEV float gumbel_exact(uint32_t bits) { return -logf(-logf(uniform_from_bits(bits, kGumbelTiny, 1.f))); }

MOCAT_DEV float gumbel_upper(uint32_t bits) {
  const float om = 2.0f - __uint_as_float((bits >> 9) | 0x3F800000u);  // 1 - f, in [2^-23, 1]
  return fmaf(-0.69314718f, __builtin_amdgcn_logf(om), 1e-4f);
}

// One row's running maximum: each lane keeps the best candidate it evaluated, `top` is the wave's.
// offer() is called by the whole wave (act: the lane holds a candidate). The first 64 candidates are never dropped.
struct GumbelRow {
  float best = -INFINITY, top = -INFINITY;
  uint32_t bi = kNoIndex;  // the largest index: any score, -inf too, wins against no candidate

  // bound: at least logit(j).
  template <class Logit>
  MOCAT_DEV void offer(bool act, uint32_t j, uint32_t bits, float bound, Logit logit) {
    const bool c = act && !(gumbel_upper(bits) + bound < top);
    if (__ballot(c) == 0ull) return;
    if (c) {
      float v = gumbel_exact(bits) + logit(j);
      if (j == 0u && isnan(v)) v = INFINITY;
      take(v, j);
    }
    top = wave_max(best);
  }

  // the larger score, the lower index on ties; false for a NaN
  MOCAT_DEV void take(float v, uint32_t j) {
    if (v > best || (v == best && j < bi)) {
      best = v;
      bi = j;
    }
  }

  // the maximum over the wave (first maximum); kNoIndex without candidates
  MOCAT_DEV uint32_t first_max() {
#pragma unroll
    for (int o = kWave / 2; o > 0; o >>= 1) {
      const float ob = __shfl_xor(best, o, kWave);
      take(ob, (uint32_t)__shfl_xor((int)bi, o, kWave));
    }
    return bi;
  }
};

// Row m of gumbel(k, (rows, n)) (elements m n + j of S = rows n), any S.
template <class Logit>
MOCAT_DEV uint32_t gumbel_row(Key k, uint32_t S, uint32_t off, uint32_t n, int lane, Logit logit) {
  GumbelRow row;
  for (uint64_t j0 = 0; j0 < n; j0 += kWave) {
    const bool act = j0 + (uint64_t)lane < n;
    const uint32_t j = (uint32_t)j0 + (uint32_t)lane, jc = act ? j : n - 1u;
    row.offer(act, j, bits_at(k, S, off + jc), logit(jc), logit);
  }
  return row.first_max();
}

// argmax_j gumbel(k, (n,))_j + logit(j) with logit(j) <= bound(j): elements j and j + ceil(n / 2) are the two
// words of a threefry block. Wave `part` of `parts` takes every parts-th 64 blocks; `best` and the index
// returned are its own part's.
template <class Bound, class Logit>
MOCAT_DEV uint32_t gumbel_argmax(Key k, uint32_t n, int lane, uint32_t part, uint32_t parts, Bound bound, Logit logit,
                                 float* best = nullptr) {
  const uint32_t h = (n + 1u) >> 1;
  GumbelRow row;
  for (uint64_t j0 = (uint64_t)part * kWave; j0 < h; j0 += (uint64_t)parts * kWave) {
    const bool act = j0 + (uint64_t)lane < h;
    const uint32_t j = act ? (uint32_t)j0 + (uint32_t)lane : 0u;
    const bool act1 = act && j + h < n;
    const uint32_t j1 = act1 ? j + h : 0u;
    const float b0 = bound(j), b1 = bound(j1);
    uint32_t w0, w1;
    bits_pair(k, n, j, w0, w1);
    // the bounds' loads, then most of the block's 75 vector operations before the first use of what they bring (left to
    // itself the scheduler may wait for a load first: backward simulation of 4096 x 4096, d = 4, 99 steps 5.42 ms, so 5.18)
    __builtin_amdgcn_sched_group_barrier(0x020, 16, 0);
    __builtin_amdgcn_sched_group_barrier(0x002, 60, 0);
    row.offer(act, j, w0, b0, logit);
    row.offer(act1, j1, w1, b1, logit);
  }
  row.first_max();
  if (best) *best = row.best;
  return row.bi;
}

// Rows m and m + rows / 2 of gumbel(k, (rows, n)) for an even number of rows: element m n + j and the same
// element of the other row are the two words of one threefry block. Wave `part` of `parts` takes every
// parts-th 64 columns.
template <class Logit>
MOCAT_DEV void gumbel_row_pair(Key k, uint32_t S, uint32_t off, uint32_t n, int lane, uint32_t part, uint32_t parts,
                               Logit logit, GumbelRow& a, GumbelRow& b) {
  const uint32_t h = S >> 1;
  for (uint64_t j0 = (uint64_t)part * kWave; j0 < n; j0 += (uint64_t)parts * kWave) {
    const bool act = j0 + (uint64_t)lane < n;
    const uint32_t j = (uint32_t)j0 + (uint32_t)lane, jc = act ? j : n - 1u;
    uint32_t w0 = off + jc, w1 = off + jc + h;
    threefry2x32(k.a, k.b, w0, w1);
    const float l = logit(jc);
    a.offer(act, j, w0, l, logit);
    b.offer(act, j, w1, l, logit);
  }
  a.first_max();
  b.first_max();
}

// Rows of random.categorical(key, lw, (rows,)) by one wave: unit u of the ceil(rows / 2) that cover them
// is the rows u and u + rows / 2 when rows is even (they share their threefry blocks), else 2u and 2u + 1.
MOCAT_DEV void categorical_unit(const float* __restrict__ lw, uint32_t n, uint32_t rows, Key key, uint32_t u, int lane,
                                int32_t* __restrict__ idx) {
  const uint32_t S = n * rows;
  auto logit = [&](uint32_t j) { return lw[j]; };
  if ((rows & 1u) == 0u) {
    GumbelRow a, b;
    gumbel_row_pair(key, S, u * n, n, lane, 0u, 1u, logit, a, b);
    if (lane == 0) {
      idx[u] = (int32_t)a.bi;
      idx[u + rows / 2] = (int32_t)b.bi;
    }
    return;
  }
  for (uint32_t r = 2u * u; r < 2u * u + 2u && r < rows; ++r) {
    const uint32_t a = gumbel_row(key, S, r * n, n, lane, logit);
    if (lane == 0) idx[r] = (int32_t)a;
  }
}

// The same unit by the P waves of a workgroup of P waves: each takes every P-th 64 columns of both rows, and the parts'
// first maxima are compared. Every thread of the workgroup calls it. For calls with too few rows for a wave each
// (launch_small_cat).
template <int P>
struct CategoricalParts {
  float best[2][P];
  uint32_t bi[2][P];
};
template <int P>
MOCAT_DEV void categorical_unit_parts(const float* __restrict__ lw, uint32_t n, uint32_t rows, Key key, uint32_t u,
                                      CategoricalParts<P>& s, int32_t* __restrict__ idx) {
  const uint32_t S = n * rows, lane = threadIdx.x & (kWave - 1), part = threadIdx.x / kWave;
  auto logit = [&](uint32_t j) { return lw[j]; };
  const bool pair = (rows & 1u) == 0u;
  GumbelRow a, b;
  if (pair) {
    gumbel_row_pair(key, S, u * n, n, (int)lane, part, P, logit, a, b);
  } else {
    auto draw = [&](GumbelRow& row, uint32_t off) {
      for (uint64_t j0 = (uint64_t)part * kWave; j0 < n; j0 += (uint64_t)P * kWave) {
        const bool act = j0 + (uint64_t)lane < n;
        const uint32_t j = (uint32_t)j0 + lane, jc = act ? j : n - 1u;
        row.offer(act, j, bits_at(key, S, off + jc), logit(jc), logit);
      }
      row.first_max();
    };
    draw(a, 2u * u * n);
    if (2u * u + 1u < rows) draw(b, (2u * u + 1u) * n);
  }
  if (lane == 0) {
    s.best[0][part] = a.best;
    s.bi[0][part] = a.bi;
    s.best[1][part] = b.best;
    s.bi[1][part] = b.bi;
  }
  __syncthreads();
  if (part != 0) return;
  if (lane < 2) {
    const uint32_t row = pair ? u + lane * (rows / 2) : 2u * u + lane;
    GumbelRow all;
    for (int q = 0; q < P; ++q) all.take(s.best[lane][q], s.bi[lane][q]);
    if (row < rows) idx[row] = (int32_t)all.bi;
  }
}

}  // namespace mocat
