// Global-L2 gradient clip coefficient on the device (gfx950).
//
// Restates the clip of _prepare_grads (apexw/optimizer.py:242-256) without the
// host synchronisation: per-tensor norms (torch._foreach_norm rounds each norm
// to the grad dtype), the L2 norm of those norms, and
// coef = min(clip / (total + 1e-6), 1).  The step kernels read the coefficient
// from device memory and scale the grads in registers.
//
// Three short launches, deterministic (no atomics):
//   1. one wavefront per work unit of the chunk table -> sum of squares
//   2. one wavefront per tensor (a workgroup for a tensor of many units) sums its
//      (contiguous) units -> rounded norm
//   3. one workgroup combines the tensor norms -> coefficient
// With grad centralization the pass that forms the row means also forms each row's
// sum of squares about its mean (apexw_grad_row_stats; rows of up to APEXW_ROW_SUMSQ_MAX
// elements), and 1 skips those tensors.
#include <mutex>
#include <type_traits>

#include "common.h"

namespace {

// squares of sanitize(g) (when san), unscaled in the grad dtype when unscale
// (AMP grads are unscaled before the clip, apexw/optimizer.py:227-237).
// Sanitizing changes only NaN / +-Inf grads, and one of those makes the lane's sum
// non-finite: the sum is formed without it, and a lane whose sum is not finite
// (rare) forms it again with it.
template <int GD, int N>
APEXW_DEV float sumsq_vals(const float (&g)[N], bool san, bool unscale, float inv, float acc, bool gc,
                           const float (&mean)[N]) {
#pragma unroll
  for (int j = 0; j < N; ++j) {
    float x = san ? sanitize<GD>(g[j]) : g[j];
    if (unscale) x = rnd<GD>(x * inv);
    if (gc) x = rnd<GD>(x - mean[j]);
    acc = fmaf(x, x, acc);
  }
  return acc;
}

// Row means (APEXW_FLAG_GC: `means` holds one per row of rl elements) of the 8
// elements from e0; zeros for a tensor that is not centralized (means == nullptr).
APEXW_DEV void clip_means8(const apexw_tensor& t, const float* means, int64_t rl, int64_t e0, float (&mean)[8]) {
  if (!means) {
#pragma unroll
    for (int j = 0; j < 8; ++j) mean[j] = 0.0f;
    return;
  }
  const int64_t rows = t.n / rl;
  if (rl >= 8) {
    // at most one row boundary inside the 8 elements
    const int64_t row = e0 / rl, col = e0 - row * rl;
    const float m0 = means[row < rows ? row : rows - 1];
    const float m1 = (col + 8 > rl && row + 1 < rows) ? means[row + 1] : m0;
#pragma unroll
    for (int j = 0; j < 8; ++j) mean[j] = col + j < rl ? m0 : m1;
    return;
  }
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    const int64_t r = (e0 + j) / rl;
    mean[j] = means[r < rows ? r : rows - 1];
  }
}

// means / rl: the tensor's row means and row length when it is centralized, else
// nullptr / 0
template <int GD>
APEXW_DEV float unit_sumsq(const apexw_tensor& t, int64_t start, int64_t cnt, bool san, bool unscale, float inv,
                           const float* means, int64_t rl) {
  const int lane = lane_id();
  const bool vec = !(t.flags & APEXW_FLAG_SCALAR) && (start % 8) == 0;
  float acc = 0.0f;
  const bool gc = means != nullptr;
  if (vec && cnt == 2048 && !gc) {
    // a whole 2048-element unit: the wave's four 8-element loads per lane are issued
    // together (centralized tensors take the loop below, in the same summation order,
    // so that their row means do not hold registers here)
    float g[4][8];
    const float none[8] = {0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int k = 0; k < 4; ++k) load8<GD>(t.g, start + k * 512 + lane * 8, g[k]);
#pragma unroll
    for (int k = 0; k < 4; ++k) acc = sumsq_vals<GD, 8>(g[k], false, unscale, inv, acc, false, none);
    if (san && !(acc - acc == 0.0f)) {
      // rare: a NaN / Inf grad in this lane's elements; read them again (the values need
      // not stay in registers past the first pass) and form the sum with them sanitized
      acc = 0.0f;
      for (int k = 0; k < 4; ++k) {
        float h[8];
        load8<GD>(t.g, start + k * 512 + lane * 8, h);
        acc = sumsq_vals<GD, 8>(h, true, unscale, inv, acc, false, none);
      }
    }
    return wave_sum(acc);
  }
  for (int pass = 0; pass < 2; ++pass) {
    const bool s = pass == 1;
    acc = 0.0f;
    for (int64_t rel = (int64_t)lane * 8; rel < cnt; rel += 64 * 8) {
      const int64_t e0 = start + rel;
      const int c = (cnt - rel) < 8 ? (int)(cnt - rel) : 8;
      float g[8];
      if (vec && c == 8) {
        load8<GD>(t.g, e0, g);
      } else {
#pragma unroll
        for (int j = 0; j < 8; ++j) g[j] = j < c ? load1<GD>(t.g, e0 + j) : 0.0f;
      }
      float mean[8];
      clip_means8(t, means, rl, e0, mean);
      acc = sumsq_vals<GD, 8>(g, s, unscale, inv, acc, gc, mean);
    }
    if (!san || acc - acc == 0.0f) break;
  }
  return wave_sum(acc);
}

// Whether tensor t's squares are its rows', written after its row means by
// row_means_kernel<true> (under APEXW_HP_ROW_SUMSQ, rows of up to APEXW_ROW_SUMSQ_MAX).
APEXW_DEV bool norm_by_rows(const apexw_tensor& d, int64_t t, uint32_t flags, const apexw_row_means* rows) {
  if (!(flags & APEXW_HP_ROW_SUMSQ) || !(d.flags & APEXW_FLAG_GC)) return false;
  return (rows ? rows[t].row_len : (int64_t)d.block) <= APEXW_ROW_SUMSQ_MAX;
}

// (six waves per SIMD: 80 registers)
__global__ __launch_bounds__(256, 6) void sumsq_kernel(const apexw_tensor* __restrict__ tensors,
                                                    const apexw_unit* __restrict__ units, int64_t n_units,
                                                    int64_t unit_size, float* __restrict__ partial, uint32_t flags,
                                                    float inv, const apexw_amp_dyn* __restrict__ amp,
                                                    const apexw_row_means* __restrict__ rows) {
  if (amp) inv = amp->grad_inv_scale;
  const uint32_t wave = uniform(threadIdx.x >> 6);
  const bool san = flags & APEXW_HP_SANITIZE, unscale = flags & APEXW_HP_UNSCALE;
  const bool row_sums = flags & APEXW_HP_ROW_SUMSQ;
  // a workgroup walks a contiguous chunk of 64 units, its waves interleaved, one
  // workgroup per chunk (the dispatcher balances the tail): at C4 (2.08 B grads)
  // 0.631 ms against 0.679 ms for a resident grid striding by 4 units
  for (int64_t base = (int64_t)blockIdx.x * 64; base < n_units; base += (int64_t)gridDim.x * 64) {
  const int64_t u_end = base + 64 < n_units ? base + 64 : n_units;
  // a chunk inside one tensor whose row sums the row pass has formed: nothing to do
  // (a tensor's units are contiguous)
  const uint32_t t0 = units[base].tensor;
  if (row_sums && units[u_end - 1].tensor == t0 && norm_by_rows(tensors[t0], t0, flags, rows)) continue;
  for (int64_t u = base + wave; u < u_end; u += 4) {
    const apexw_unit un = units[u];
    const apexw_tensor& t = tensors[un.tensor];
    if (row_sums && norm_by_rows(t, un.tensor, flags, rows)) continue;
    const int64_t us = unit_size > 0 ? unit_size : (t.block > 0 ? (int64_t)t.block : 64);
    const int64_t start = (int64_t)un.unit * us;
    const int64_t cnt = (t.n - start) < us ? (t.n - start) : us;
    const uint32_t gd = (t.flags >> APEXW_FLAG_GDT_SHIFT) & 3u;
    // a centralized tensor's row means: its descriptor's own fields (compact tables) or
    // its entry of the side table (8-bit / ultra tables)
    const float* means = nullptr;
    int64_t rl = 0;
    if (t.flags & APEXW_FLAG_GC) {
      means = rows ? rows[un.tensor].means : t.m_scale;
      rl = rows ? rows[un.tensor].row_len : (int64_t)t.block;
    }
    float s;
    if (gd == APEXW_F32) s = unit_sumsq<APEXW_F32>(t, start, cnt, san, unscale, inv, means, rl);
    else if (gd == APEXW_BF16) s = unit_sumsq<APEXW_BF16>(t, start, cnt, san, unscale, inv, means, rl);
    else s = unit_sumsq<APEXW_F16>(t, start, cnt, san, unscale, inv, means, rl);
    if (lane_id() == 0) partial[u] = s;
  }
  }
}

// The partial sums of one tensor: its units' (from sumsq_kernel) or its rows' (norm_by_rows).
struct NormSpan {
  const float* p;
  int64_t n;
};
APEXW_DEV NormSpan norm_span(const apexw_tensor* tensors, int64_t t, const int64_t* unit_begin, const float* partial,
                             uint32_t flags, const apexw_row_means* rows) {
  const apexw_tensor& d = tensors[t];
  if (norm_by_rows(d, t, flags, rows)) {
    const float* means = rows ? rows[t].means : d.m_scale;
    const int64_t n_rows = d.n / (rows ? rows[t].row_len : (int64_t)d.block);
    return {means + n_rows, n_rows};
  }
  return {partial + unit_begin[t], unit_begin[t + 1] - unit_begin[t]};
}

// The sum of `s` by `step` lanes, this one the `first`, in float64: eight loads in
// flight and eight running sums (a plain loop waits for memory at each addition).
APEXW_DEV double span_sum(const NormSpan& s, int64_t first, int64_t step) {
  double a[8] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
  int64_t i = first;
  for (; i + 7 * step < s.n; i += 8 * step) {
#pragma unroll
    for (int j = 0; j < 8; ++j) a[j] += (double)s.p[i + j * step];
  }
  for (; i < s.n; i += step) a[0] += (double)s.p[i];
  return ((a[0] + a[1]) + (a[2] + a[3])) + ((a[4] + a[5]) + (a[6] + a[7]));
}

APEXW_DEV double wave_sum64(double x) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) x += __shfl_xor(x, off, 64);
  return x;
}

// Each tensor's norm, rounded to its grad dtype, as torch._foreach_norm does.  A
// workgroup of 16 waves takes `per` tensors (16, or 1 when there are few), a wave
// each; a tensor of more than kNormWave partials is summed by the whole workgroup:
// one wave alone walks the 28,672 units of a 14336 x 4096 matrix serially (123 us for
// the 36 tensors of four Llama layers, 6 us so; 68 -> 5 us for GPT-2-small).
constexpr int kNormWaves = 16;
constexpr int64_t kNormWave = 1024;
__global__ __launch_bounds__(kNormWaves * 64) void tensor_norm_kernel(
    const apexw_tensor* __restrict__ tensors, int32_t n_tensors, const int64_t* __restrict__ unit_begin,
    const float* __restrict__ partial, float* __restrict__ norm, int32_t per, uint32_t flags,
    const apexw_row_means* __restrict__ rows) {
  __shared__ double s_part[kNormWaves];
  const int wave = (int)uniform(threadIdx.x >> 6);
  auto store = [&](int64_t t, double acc) {
    const uint32_t gd = (tensors[t].flags >> APEXW_FLAG_GDT_SHIFT) & 3u;
    float nrm = sqrtf((float)acc);
    nrm = gd == APEXW_BF16 ? rnd<APEXW_BF16>(nrm) : (gd == APEXW_F16 ? rnd<APEXW_F16>(nrm) : nrm);
    norm[t] = nrm;
  };
  for (int64_t t0 = (int64_t)blockIdx.x * per; t0 < n_tensors; t0 += (int64_t)gridDim.x * per) {
    const int64_t t_end = t0 + per < n_tensors ? t0 + per : n_tensors;
    bool large = false;
    if (t0 + wave < t_end) {
      const NormSpan s = norm_span(tensors, t0 + wave, unit_begin, partial, flags, rows);
      large = s.n > kNormWave;
      if (!large) {
        const double acc = wave_sum64(span_sum(s, lane_id(), 64));
        if (lane_id() == 0) store(t0 + wave, acc);
      }
    }
    if (!__syncthreads_or(large)) continue;   // (the same for every wave)
    for (int64_t t = t0; t < t_end; ++t) {
      const NormSpan s = norm_span(tensors, t, unit_begin, partial, flags, rows);
      if (s.n <= kNormWave) continue;
      const double acc = wave_sum64(span_sum(s, threadIdx.x, kNormWaves * 64));
      if (lane_id() == 0) s_part[wave] = acc;
      __syncthreads();
      if (threadIdx.x == 0) {
        double tot = 0.0;
        for (int w = 0; w < kNormWaves; ++w) tot += s_part[w];
        store(t, tot);
      }
      __syncthreads();   // s_part is the next large tensor's
    }
  }
}

__global__ __launch_bounds__(1024) void clip_coef_kernel(const float* __restrict__ norm, int32_t n_tensors, float clip,
                                                         float* __restrict__ coef) {
  __shared__ double s_part[16];
  double acc = 0.0;
  for (int32_t t = threadIdx.x; t < n_tensors; t += blockDim.x) acc += (double)norm[t] * (double)norm[t];
  acc = wave_sum64(acc);
  if (lane_id() == 0) s_part[threadIdx.x >> 6] = acc;
  __syncthreads();
  if (threadIdx.x == 0) {
    double tot = 0.0;
    for (int w = 0; w < (int)(blockDim.x >> 6); ++w) tot += s_part[w];
    const float total = sqrtf((float)tot);
    float c = clip / (total + 1e-6f);
    // torch.clamp(c, max=1) then "multiply only if c < 1": NaN / >= 1 leave grads unscaled
    coef[0] = (c < 1.0f) ? c : 1.0f;
  }
}

// ---------------------------------------------------------------------------
// Gradient preparation (sanitize, AMP unscale, centralization), one 256-thread
// workgroup per unit: a row of a centralized grad (sum pass, then subtract and
// store; the row is re-read from L2) or a 2048-element chunk of any other grad.
// ---------------------------------------------------------------------------
template <int GD> APEXW_DEV float prep_value(const void* g, int64_t i, bool san, bool unscale, float inv) {
  float x = load1<GD>(g, i);
  if (san) x = sanitize<GD>(x);
  if (unscale) x = rnd<GD>(x * inv);
  return x;
}

template <int GD> APEXW_DEV void prep_vec8(const void* g, int64_t i, bool san, bool unscale, float inv,
                                           float (&x)[8]) {
  load8<GD>(g, i, x);
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    if (san) x[j] = sanitize<GD>(x[j]);
    if (unscale) x[j] = rnd<GD>(x[j] * inv);
  }
}

// Elements [lo, hi) of a grad: the 8-aligned middle [a, b) in 8-element vectors
// (16-byte bf16 / 32-byte fp32 accesses) when both buffers are aligned for
// them, the ragged ends element by element.
struct PrepSpan {
  int64_t a, b;
};
template <int GD> APEXW_DEV PrepSpan prep_span(const apexw_grad_prep& d, int64_t lo, int64_t hi) {
  constexpr uintptr_t align = GD == APEXW_F32 ? 31 : 15;
  if ((((uintptr_t)d.g | (uintptr_t)d.out) & align) != 0) return {hi, hi};
  const int64_t a = (lo + 7) & ~(int64_t)7, b = hi & ~(int64_t)7;
  return a < b ? PrepSpan{a, b} : PrepSpan{hi, hi};
}

template <int GD>
APEXW_DEV void prep_unit(const apexw_grad_prep& d, int64_t unit, bool san, bool unscale, float inv, float* red) {
  const int tid = threadIdx.x;
  const bool row = d.row_len > 0;
  const int64_t lo = row ? unit * d.row_len : unit * APEXW_GRAD_PREP_CHUNK;
  const int64_t hi = row ? lo + d.row_len : (lo + APEXW_GRAD_PREP_CHUNK < d.n ? lo + APEXW_GRAD_PREP_CHUNK : d.n);
  const PrepSpan sp = prep_span<GD>(d, lo, hi);
  // ragged ends: [lo, a) and [b, hi) (the whole range when not vectorized)
  const int64_t head = sp.a - lo, n_end = head + (hi - sp.b);
  float mean = 0.0f;
  if (row) {
    float s = 0.0f;
    for (int64_t i = sp.a + (int64_t)tid * 8; i < sp.b; i += 2048) {
      float x[8];
      prep_vec8<GD>(d.g, i, san, unscale, inv, x);
#pragma unroll
      for (int j = 0; j < 8; ++j) s += x[j];
    }
    for (int64_t k = tid; k < n_end; k += 256) {
      const int64_t i = k < head ? lo + k : sp.b + (k - head);
      s += prep_value<GD>(d.g, i, san, unscale, inv);
    }
    s = wave_sum(s);
    if ((tid & 63) == 0) red[tid >> 6] = s;
    __syncthreads();
    // torch's mean: sum in fp32, divided by the count, result in the grad dtype
    mean = rnd<GD>(((red[0] + red[1]) + (red[2] + red[3])) / (float)d.row_len);
  }
  // second pass (the row is re-read from L2): subtract the mean and store
  for (int64_t i = sp.a + (int64_t)tid * 8; i < sp.b; i += 2048) {
    float x[8];
    prep_vec8<GD>(d.g, i, san, unscale, inv, x);
    if (row) {
#pragma unroll
      for (int j = 0; j < 8; ++j) x[j] = rnd<GD>(x[j] - mean);
    }
    store8<GD>(d.out, i, x);
  }
  for (int64_t k = tid; k < n_end; k += 256) {
    const int64_t i = k < head ? lo + k : sp.b + (k - head);
    const float x = prep_value<GD>(d.g, i, san, unscale, inv);
    store1<GD>(d.out, i, row ? rnd<GD>(x - mean) : x);
  }
}

// Row means only (the fold of centralization into the step kernels): one wave per
// row of a descriptor with row_len > 0; d.out is a float array of one mean per
// row, each the grad dtype's rounding of the fp32 row sum over row_len of the
// sanitized, unscaled grads.  SUMSQ (a clip follows): the row's sum of squares about
// that mean, each difference rounded to the grad dtype, goes to d.out[rows + row] for
// rows of up to APEXW_ROW_SUMSQ_MAX elements.
//
// Bound by the read of the grads.  A lane holds its first kRowVecs 8-element vectors
// (rows of up to 4096 16-bit elements whole), loaded before they are added, so the
// second sum reads nothing again; a longer row's rest is read in batches of four and,
// for the second sum, again.  Sanitizing changes only NaN / +-Inf grads, and one of
// those makes the row's sum non-finite: the sums are formed without it, and a row
// whose sum is not finite (rare) forms them again with it.
// Four Llama layers (0.87 B bf16 grads, 1.75 GB, all centralized), 8-bit step with clip: 3098 us
// with the means' and the clip's passes apart, 1840 us with both here and the unscale flag
// tested per element, 1751 us with each preparation (plain, unscaled, sanitized) its own loop.
//
// One wave walks a row twice in series where the clip's unit pass would spread its second
// read over the chip.  Means, clip and norms of one bf16 tensor by the unit pass / here, us:
// 64 x 4096: 94 / 20, 64 x 16384: 110 / 44, 64 x 32768: 128 / 75; without a limit
// 64 x 65536: 190 / 228, 8 x 262144: 284 / 452, 8 x 1048576: 869 / 1789; fp32 alike.  So rows
// beyond APEXW_ROW_SUMSQ_MAX leave their squares to the unit pass.
// Sixteen rows to a workgroup: enough workgroups for small models, whose rows are few.
constexpr int64_t kRowChunk = 16;
template <int GD> constexpr int kRowVecs = GD == APEXW_F32 ? 4 : 8;

// A grad as it enters the row's sums: as given, unscaled, or sanitized (and unscaled by a
// run-time flag: rows of non-finite grads are rare).
constexpr int kPlain = 0, kUnscale = 1, kSanitize = 2;
template <int GD, int PREP>
APEXW_DEV float row_value(float x, bool unscale, float inv) {
  if constexpr (PREP == kPlain) return x;
  if constexpr (PREP == kSanitize) {
    x = sanitize<GD>(x);
    if (!unscale) return x;
  }
  return rnd<GD>(x * inv);
}

// The row's sum (MEAN false) or its sum of squares about mean (MEAN true) over a lane's
// share: the held vectors r, the rest of [a, b) and the ragged ends.  Squares go to eight
// running sums, folded after each batch of at most kRowVecs additions, so that no chain of
// additions is longer than in the unit pass (32 terms) up to APEXW_ROW_SUMSQ_MAX elements.
template <int GD, int PREP, bool MEAN>
APEXW_DEV float row_sum(const apexw_grad_prep& d, const Raw8<GD> (&r)[kRowVecs<GD>], const PrepSpan& sp, int64_t lo,
                        int64_t hi, bool unscale, float inv, float mean) {
  constexpr int NV = kRowVecs<GD>;
  const int lane = lane_id();
  float s = 0.0f, q[8] = {0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
  auto add = [&](int j, float x) {
    x = row_value<GD, PREP>(x, unscale, inv);
    if constexpr (MEAN) {
      x = rnd<GD>(x - mean);
      q[j] = fmaf(x, x, q[j]);
    } else {
      s += x;
    }
  };
  auto fold = [&]() {
    if constexpr (MEAN) {
      s += ((q[0] + q[1]) + (q[2] + q[3])) + ((q[4] + q[5]) + (q[6] + q[7]));
#pragma unroll
      for (int j = 0; j < 8; ++j) q[j] = 0.0f;
    }
  };
  int64_t i = sp.a + (int64_t)lane * 8;
#pragma unroll
  for (int v = 0; v < NV; ++v, i += 512) {
    if (i < sp.b) {
      float x[8];
      unpack8<GD>(r[v], x);
#pragma unroll
      for (int j = 0; j < 8; ++j) add(j, x[j]);
    }
  }
  fold();
  for (; i + 3 * 512 < sp.b; i += 4 * 512) {
    Raw8<GD> w[4];
#pragma unroll
    for (int v = 0; v < 4; ++v) raw_load8<GD>(d.g, i + v * 512, w[v]);
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      float x[8];
      unpack8<GD>(w[v], x);
#pragma unroll
      for (int j = 0; j < 8; ++j) add(j, x[j]);
    }
    fold();
  }
  for (; i < sp.b; i += 512) {
    float x[8];
    load8<GD>(d.g, i, x);
#pragma unroll
    for (int j = 0; j < 8; ++j) add(j, x[j]);
  }
  // ragged ends: [lo, a) and [b, hi) (the whole row when not vectorized)
  const int64_t head = sp.a - lo, n_end = head + (hi - sp.b);
  for (int64_t k0 = lane; k0 < n_end; k0 += 8 * 64) {
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const int64_t k = k0 + j * 64;
      if (k < n_end) add(j, load1<GD>(d.g, k < head ? lo + k : sp.b + (k - head)));
    }
    fold();
  }
  fold();
  return wave_sum(s);
}

template <int GD, bool SUMSQ>
APEXW_DEV void mean_row(const apexw_grad_prep& d, int64_t row, bool san, bool unscale, float inv) {
  constexpr int NV = kRowVecs<GD>;
  const int lane = lane_id();
  const int64_t lo = row * d.row_len, hi = lo + d.row_len;
  const PrepSpan sp = prep_span<GD>(d, lo, hi);
  Raw8<GD> r[NV];
#pragma unroll
  for (int q = 0; q < NV; ++q) {
    const int64_t i = sp.a + (int64_t)lane * 8 + q * 512;
    if (i < sp.b) raw_load8<GD>(d.g, i, r[q]);
  }
  // both sums under one preparation of the grads
  auto sums = [&](auto prep_c, float& mean, float& s, float& q) {
    constexpr int PREP = decltype(prep_c)::value;
    s = row_sum<GD, PREP, false>(d, r, sp, lo, hi, unscale, inv, 0.0f);
    mean = rnd<GD>(s / (float)d.row_len);
    q = 0.0f;
    if (PREP != kSanitize && san && !(s - s == 0.0f)) return;   // formed again, sanitized
    if (SUMSQ && d.row_len <= APEXW_ROW_SUMSQ_MAX)
      q = row_sum<GD, PREP, true>(d, r, sp, lo, hi, unscale, inv, mean);
  };
  float mean, s, q;
  if (unscale) sums(std::integral_constant<int, kUnscale>(), mean, s, q);
  else sums(std::integral_constant<int, kPlain>(), mean, s, q);
  // wave-uniform: every lane holds the sum
  if (san && !(s - s == 0.0f)) sums(std::integral_constant<int, kSanitize>(), mean, s, q);
  if (lane == 0) {
    ((float*)d.out)[row] = mean;
    if (SUMSQ && d.row_len <= APEXW_ROW_SUMSQ_MAX) ((float*)d.out)[d.n / d.row_len + row] = q;
  }
}

template <bool SUMSQ>
__global__ __launch_bounds__(256) void row_means_kernel(const apexw_grad_prep* __restrict__ preps,
                                                        const apexw_unit* __restrict__ units, int64_t n_units,
                                                        float inv, uint32_t flags,
                                                        const apexw_amp_dyn* __restrict__ amp) {
  if (amp) inv = amp->grad_inv_scale;
  const bool san = flags & APEXW_HP_SANITIZE, unscale = flags & APEXW_HP_UNSCALE;
  const uint32_t wave = uniform(threadIdx.x >> 6);
  // workgroup b takes a contiguous chunk of kRowChunk rows, its waves interleaved
  for (int64_t base = (int64_t)blockIdx.x * kRowChunk; base < n_units; base += (int64_t)gridDim.x * kRowChunk)
  for (int64_t u = base + wave, u_end = base + kRowChunk < n_units ? base + kRowChunk : n_units; u < u_end; u += 4) {
    const apexw_unit un = units[u];
    const apexw_grad_prep& d = preps[un.tensor];
    if (d.dtype == APEXW_F32) mean_row<APEXW_F32, SUMSQ>(d, un.unit, san, unscale, inv);
    else if (d.dtype == APEXW_BF16) mean_row<APEXW_BF16, SUMSQ>(d, un.unit, san, unscale, inv);
    else mean_row<APEXW_F16, SUMSQ>(d, un.unit, san, unscale, inv);
  }
}

__global__ __launch_bounds__(256) void grad_prep_kernel(const apexw_grad_prep* __restrict__ preps,
                                                        const apexw_unit* __restrict__ units, int64_t n_units,
                                                        float inv, uint32_t flags,
                                                        const apexw_amp_dyn* __restrict__ amp) {
  __shared__ float red[4];
  if (amp) inv = amp->grad_inv_scale;
  const bool san = flags & APEXW_HP_SANITIZE, unscale = flags & APEXW_HP_UNSCALE;
  for (int64_t u = blockIdx.x; u < n_units; u += gridDim.x) {
    const apexw_unit un = units[u];
    const apexw_grad_prep& d = preps[un.tensor];
    if (d.dtype == APEXW_F32) prep_unit<APEXW_F32>(d, un.unit, san, unscale, inv, red);
    else if (d.dtype == APEXW_BF16) prep_unit<APEXW_BF16>(d, un.unit, san, unscale, inv, red);
    else prep_unit<APEXW_F16>(d, un.unit, san, unscale, inv, red);
    __syncthreads();   // red is reused by the next unit
  }
}

}  // namespace

int apexw_launch_grad_prep(const apexw_grad_prep* preps, const apexw_unit* units, int64_t n_units, float inv,
                           uint32_t flags, const apexw_amp_dyn* amp, hipStream_t stream) {
  if (n_units <= 0) return APEXW_OK;
  const int64_t want = n_units < 65536 ? n_units : 65536;
  hipLaunchKernelGGL(grad_prep_kernel, dim3((unsigned)want), dim3(256), 0, stream, preps, units, n_units, inv, flags,
                     amp);
  return hipGetLastError() == hipSuccess ? APEXW_OK : APEXW_ERR_LAUNCH;
}

int apexw_launch_clip(const apexw_tensor* tensors, int32_t n_tensors, const apexw_unit* units, int64_t n_units,
                      int64_t unit_size, const int64_t* unit_begin, float* unit_partial, float* tensor_norm,
                      float clip, float inv, uint32_t flags, float* coef, const apexw_amp_dyn* amp,
                      const apexw_row_means* rows, hipStream_t stream);

int apexw_launch_row_means(const apexw_grad_prep* preps, const apexw_unit* units, int64_t n_units, float inv,
                           uint32_t flags, const apexw_amp_dyn* amp, bool sumsq, hipStream_t stream) {
  if (n_units <= 0) return APEXW_OK;
  const int64_t chunks = (n_units + kRowChunk - 1) / kRowChunk;
  const unsigned grid = (unsigned)(chunks < INT32_MAX ? chunks : INT32_MAX);
  if (sumsq)
    hipLaunchKernelGGL(row_means_kernel<true>, dim3(grid), dim3(256), 0, stream, preps, units, n_units, inv, flags,
                       amp);
  else
    hipLaunchKernelGGL(row_means_kernel<false>, dim3(grid), dim3(256), 0, stream, preps, units, n_units, inv, flags,
                       amp);
  return hipGetLastError() == hipSuccess ? APEXW_OK : APEXW_ERR_LAUNCH;
}

// ---------------------------------------------------------------------------
// Allocation-free clip coefficient: the per-unit partials and per-tensor norms
// live in this file-scope device array instead of caller workspace.  Each GPU
// holds its own copy; its device address is looked up once per device with
// hipGetSymbolAddress (the array's name is only a host-side stand-in).
// ---------------------------------------------------------------------------
static __device__ __align__(256) float scratch[APEXW_NOALLOC_CLIP_MAX_UNITS + APEXW_NOALLOC_CLIP_MAX_TENSORS];

namespace {

constexpr int kScratchDevices = 64;
std::mutex g_scratch_mu;
float* g_scratch_ptr[kScratchDevices];

// Device address of `scratch` on device dev, or nullptr if it cannot be had.  A
// lookup that fails is not cached: the next call tries again.
float* scratch_on_device(int dev) {
  if (dev < 0 || dev >= kScratchDevices) return nullptr;
  std::lock_guard<std::mutex> lk(g_scratch_mu);
  if (g_scratch_ptr[dev]) return g_scratch_ptr[dev];
  int cur = -1;
  if (hipGetDevice(&cur) != hipSuccess) return nullptr;
  // hipGetSymbolAddress answers for the calling thread's current device
  if (cur != dev && hipSetDevice(dev) != hipSuccess) return nullptr;
  void* ptr = nullptr;
  const bool ok = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch)) == hipSuccess && ptr;
  if (cur != dev) (void)hipSetDevice(cur);
  if (ok) g_scratch_ptr[dev] = (float*)ptr;
  return ok ? (float*)ptr : nullptr;
}

}  // namespace

extern "C" int apexw_grad_clip_coef_noalloc(const apexw_tensor* tensors, int32_t n_tensors, const apexw_unit* units,
                                            int64_t n_units, int64_t unit_size, const int64_t* unit_begin,
                                            float clip, float grad_inv_scale, uint32_t flags, float* coef,
                                            const apexw_amp_dyn* amp, void* stream) {
  if (!tensors || !units || !unit_begin || !coef) return APEXW_ERR_ARG;
  if (n_tensors <= 0 || n_units < 0 || unit_size < 0 || !(clip > 0.0f)) return APEXW_ERR_ARG;
  if ((flags & APEXW_HP_UNSCALE) && !amp && !apexw_inv_scale_ok(grad_inv_scale)) return APEXW_ERR_ARG;
  if (n_units > APEXW_NOALLOC_CLIP_MAX_UNITS || n_tensors > APEXW_NOALLOC_CLIP_MAX_TENSORS) return APEXW_ERR_SIZE;
  // the array of the GPU the kernels run on: the stream's device (the null stream is
  // the current device's)
  int dev = -1;
  if (stream) {
    if (hipStreamGetDevice((hipStream_t)stream, &dev) != hipSuccess) return APEXW_ERR_ARG;
  } else if (hipGetDevice(&dev) != hipSuccess) {
    return APEXW_ERR_LAUNCH;
  }
  float* ptr = scratch_on_device(dev);
  if (!ptr) return APEXW_ERR_LAUNCH;
  return apexw_launch_clip(tensors, n_tensors, units, n_units, unit_size, unit_begin, ptr,
                           ptr + APEXW_NOALLOC_CLIP_MAX_UNITS, clip, grad_inv_scale, flags, coef, amp, nullptr,
                           (hipStream_t)stream);
}

int apexw_launch_clip(const apexw_tensor* tensors, int32_t n_tensors, const apexw_unit* units, int64_t n_units,
                      int64_t unit_size, const int64_t* unit_begin, float* unit_partial, float* tensor_norm,
                      float clip, float inv, uint32_t flags, float* coef, const apexw_amp_dyn* amp,
                      const apexw_row_means* rows, hipStream_t stream) {
  if (n_units > 0) {
    const int64_t chunks = (n_units + 63) / 64;
    const int grid_units = (int)(chunks < INT32_MAX ? chunks : INT32_MAX);
    hipLaunchKernelGGL(sumsq_kernel, dim3(grid_units), dim3(256), 0, stream, tensors, units, n_units, unit_size,
                       unit_partial, flags, inv, amp, rows);
  }
  if (n_tensors > 0) {
    // a workgroup per tensor while that fills the chip at most a few times over, 16
    // tensors to a workgroup beyond (small tensors then dominate the count)
    const int32_t per = n_tensors <= 2048 ? 1 : kNormWaves;
    const int32_t grid_tensors = (n_tensors + per - 1) / per;
    hipLaunchKernelGGL(tensor_norm_kernel, dim3(grid_tensors), dim3(kNormWaves * 64), 0, stream, tensors, n_tensors,
                       unit_begin, unit_partial, tensor_norm, per, flags, rows);
  }
  hipLaunchKernelGGL(clip_coef_kernel, dim3(1), dim3(1024), 0, stream, tensor_norm, n_tensors, clip, coef);
  return hipGetLastError() == hipSuccess ? APEXW_OK : APEXW_ERR_LAUNCH;
}

// ---------------------------------------------------------------------------
// GradScaler's scale and found_inf read on the device (apexw_amp_prepare): one
// thread turns them and the host's step counts into each launch's scalars.
// ---------------------------------------------------------------------------
namespace {

struct AmpLaunches {
  apexw_amp_launch l[APEXW_AMP_MAX_LAUNCHES];
};

__global__ __launch_bounds__(64) void amp_prepare_kernel(const float* __restrict__ found_inf,
                                                         const float* __restrict__ grad_scale,
                                                         int32_t* __restrict__ skips, int32_t folded, AmpLaunches ls,
                                                         int32_t n, apexw_amp_dyn* __restrict__ dyn) {
  if (threadIdx.x != 0) return;
  const uint32_t skip = *found_inf != 0.0f ? 1u : 0u;
  const int32_t s = *skips;
  if (skip) *skips = s + 1;
  const float inv = 1.0f / *grad_scale;
  for (int i = 0; i < n; ++i) {
    const apexw_amp_launch& L = ls.l[i];
    const double t = L.step - (double)(s - folded);
    const double bc1 = 1.0 - pow(L.beta1, t), bc2 = 1.0 - pow(L.beta2, t);
    const double bc2s = sqrt(bc2);
    apexw_amp_dyn d;
    if (L.kind == 1) {
      d.step_size = (float)(L.lr / bc1);
      d.eps_scaled = (float)L.eps;
      d.bc2_sqrt = (float)bc2s;
    } else {
      d.step_size = (float)(L.lr * bc2s / bc1);
      d.eps_scaled = (float)(L.eps * bc2s);
      d.bc2_sqrt = (float)bc2s;
    }
    d.grad_inv_scale = inv;
    d.skip = skip;
    d.reserved[0] = d.reserved[1] = d.reserved[2] = 0u;
    dyn[i] = d;
  }
}

}  // namespace

int apexw_launch_amp_prepare(const float* found_inf, const float* grad_scale, int32_t* skips, int32_t folded,
                             const apexw_amp_launch* launches, int32_t n, apexw_amp_dyn* dyn, hipStream_t stream) {
  AmpLaunches ls;
  for (int i = 0; i < n; ++i) ls.l[i] = launches[i];
  hipLaunchKernelGGL(amp_prepare_kernel, dim3(1), dim3(64), 0, stream, found_inf, grad_scale, skips, folded, ls, n,
                     dyn);
  return hipGetLastError() == hipSuccess ? APEXW_OK : APEXW_ERR_LAUNCH;
}
