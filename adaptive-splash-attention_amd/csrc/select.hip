// Key-block position bounds, tau from the sorted top-k values, and the
// dispatch of the score pass (select_kernel.hpp) by storage type.
#include <climits>
#include <type_traits>

#include "asa_compact.hpp"
#include "asa_device.hpp"
#include "asa_launch.hpp"
#include "asa_tiles.hpp"

namespace asa {
namespace {

constexpr int kThreads = 256;

__device__ __forceinline__ int wave_min(int v) { return wave_reduce_minmax<false>(v); }
__device__ __forceinline__ int wave_max(int v) { return wave_reduce_minmax<true>(v); }

// tau from the sorted top-k values of one row (best first), s(j) for
// j < k, following the reference recurrence step by step
// (adasplashattention.cu:51-125): bracket from the extreme kept values,
// midpoint start, up to five rounds of {f, f', f'' over the leading positive
// terms; exit when |f| < 1e-4; Halley step with the reference's f''
// coefficient a(a + 1 - alpha); bracket midpoint when the step leaves the
// bracket; bracket update from f at the new point; clamp}.  No contraction,
// powers in the exponent classes of alpha (pow_exact_c): bit-identical to
// the CPU oracle on equal inputs.  KMAX > 0: the caller guarantees k <= KMAX
// and s(j) is a compile-time-indexed register, so the loops are unrolled.
template <int AC, int KMAX, typename S>
__device__ float entmax_tau(S s, int k, float alpha_in) {
#pragma clang fp contract(off)
  constexpr int PA = AlphaPow<AC>::P, P1 = AlphaPow<AC>::W, P2 = AlphaPow<AC>::V;
  // register-resident values and closed-form powers: evaluate every slot
  constexpr bool kFlat = KMAX > 0 && AC != kAGen;
  const float alpha = fmaxf(1.05f, fminf(alpha_in, 3.0f));
  const float am1 = alpha - 1.0f;
  const float a = 1.0f / am1;
  const float e1 = (2.0f - alpha) * a;
  const float e2 = (3.0f - 2.0f * alpha) * a;
  const float c2 = a * ((a + 1.0f) - alpha);
  const float top = s(0);
  const float bottom = s(k - 1);
  float lo = am1 * bottom - 2.0f;
  float hi = am1 * top + 2.0f;
  float tau = 0.5f * (lo + hi);
  for (int it = 0; it < 5; ++it) {
    float f = -1.0f, df = 0.0f, d2f = 0.0f;
    // one term of f, f', f''; false once the terms end
    auto term = [&](int j) {
      if (j >= k) return false;
      const float u = am1 * s(j) - tau;
      if (u <= 0.0f) return false;
      const float ue = fmaxf(u, kEps);
      float t = pow_exact_c<PA>(ue, a);
      if (!finite(t)) t = 0.0f;
      f = f + t;
      const float t1 = -a * pow_exact_c<P1>(ue, e1);
      if (finite(t1)) df = df + t1;
      const float t2 = c2 * pow_exact_c<P2>(ue, e2);
      if (finite(t2)) d2f = d2f + t2;
      return true;
    };
    if constexpr (kFlat) {
      // Branch-free over all KMAX slots: the values are sorted, so u is
      // non-increasing in j and the terms the recurrence stops before are
      // exactly the ones with u <= 0 (or j >= k).  Those add +0.0f, which
      // leaves every sum unchanged (none of them can be -0.0f), so the
      // result is bit-identical to the early-exit loop.  The closed-form
      // powers cannot overflow here (u <= (alpha-1)(10 + 1e6) + 10 with
      // u^e, e in {-1, 0, ..., 4}, and u >= EPS), so the finiteness tests
      // of the general loop always pass and are left out.
#pragma unroll
      for (int j = 0; j < KMAX; ++j) {
        const float u = am1 * s(j) - tau;
        const bool on = j < k && !(u <= 0.0f);
        const float ue = fmaxf(u, kEps);
        f = f + (on ? pow_exact_c<PA>(ue, a) : 0.0f);
        df = df + (on ? -a * pow_exact_c<P1>(ue, e1) : 0.0f);
        d2f = d2f + (on ? c2 * pow_exact_c<P2>(ue, e2) : 0.0f);
      }
    } else if constexpr (KMAX > 0) {
#pragma unroll
      for (int j = 0; j < KMAX; ++j)
        if (!term(j)) break;
    } else {
      for (int j = 0; term(j); ++j) {
      }
    }
    if (fabsf(f) < 1e-4f) break;
    float next = tau;
    if (fabsf(df) > kEps) {
      const float den = 2.0f * df * df - f * d2f;
      if (fabsf(den) > kEps) next = tau - 2.0f * f * df / den;
    }
    if (!(next >= lo && next <= hi)) next = 0.5f * (lo + hi);
    float gsum = -1.0f;
    auto gterm = [&](int j) {
      if (j >= k) return false;
      const float u = am1 * s(j) - next;
      if (u <= 0.0f) return false;
      const float t = pow_exact_c<PA>(fmaxf(u, kEps), a);
      if (finite(t)) gsum = gsum + t;
      return true;
    };
    if constexpr (kFlat) {
#pragma unroll
      for (int j = 0; j < KMAX; ++j) {
        const float u = am1 * s(j) - next;
        gsum = gsum + (j < k && !(u <= 0.0f) ? pow_exact_c<PA>(fmaxf(u, kEps), a) : 0.0f);
      }
    } else if constexpr (KMAX > 0) {
#pragma unroll
      for (int j = 0; j < KMAX; ++j)
        if (!gterm(j)) break;
    } else {
      for (int j = 0; gterm(j); ++j) {
      }
    }
    if (gsum > 0.0f) lo = next;
    else hi = next;
    tau = next;
    tau = fmaxf(tau, bottom * am1 - 10.0f);
    tau = fminf(tau, top * am1 + 10.0f);
  }
  return tau;
}

// Smallest and largest position of every 64-key block of every (batch,
// head): kbounds[bh * nKB + kb] = (min, max) over the block's keys < NK.
// One wave per key block.  Also clears the per-call status word: this is the
// first kernel of a forward on the stream.
__global__ __launch_bounds__(kThreads) void bounds_kernel(SelectParams p) {
  const int nKB = p.d.nKB, NK = p.d.NK;
  if (blockIdx.x == 0 && threadIdx.x == 0 && p.status) *p.status = 0u;
  const int blk = blockIdx.x * (kThreads / kWave) + (threadIdx.x >> 6);
  if (blk >= p.d.BH * nKB) return;  // wave-uniform
  const int bh = blk / nKB, kb = blk % nKB, L = threadIdx.x & 63;
  const int key = kb * kBlock + L;
  const int pos = key < NK ? p.k_idx[size_t(bh) * NK + key] : 0;
  const int mn = wave_min(key < NK ? pos : INT_MAX);
  const int mx = wave_max(key < NK ? pos : INT_MIN);
  if (L == 0) p.kbounds[blk] = int2{mn, mx};
}

// tau of every row from its sorted top-k values (one thread per row):
// tkv[e * rows + row], e < k.
template <int AC, int KMAX>
__device__ __forceinline__ void tau_row(const SelectParams& p, int blk) {
  const size_t rows = size_t(p.d.BH) * p.d.NQ;
  const size_t r = size_t(blk) * kThreads + threadIdx.x;
  if (r >= rows) return;
  const int k = p.d.k;
  const float* v = p.tkv + r;
  if constexpr (KMAX > 0) {
    float reg[KMAX];
#pragma unroll
    for (int j = 0; j < KMAX; ++j) reg[j] = v[size_t(min(j, k - 1)) * rows];  // k >= 1
    p.taus[r] = entmax_tau<AC, KMAX>([&](int j) { return reg[j]; }, k, p.d.alpha);
  } else {
    p.taus[r] = entmax_tau<AC, 0>([&](int j) { return v[size_t(j) * rows]; }, k, p.d.alpha);
  }
}


template <int AC, int KMAX>
__global__ __launch_bounds__(kThreads) void tau_kernel(SelectParams p) {
  tau_row<AC, KMAX>(p, blockIdx.x);
}

// compact_kernel's blocks, then tau_kernel's (both read only what the
// score pass wrote): one launch, the compaction running beside the tau
// rows instead of after them.  The compaction's blocks come first: each
// runs longer than a block of tau rows, and on large masks they are many
// (compact_grid).
template <int AC, int KMAX>
__global__ __launch_bounds__(kThreads) void tau_compact_kernel(SelectParams p, CompactParams cp, int ncomp) {
  if (int(blockIdx.x) < ncomp) {  // block-uniform
    extern __shared__ int sm[];
    compact_detail::compact_block(cp, sm, blockIdx.x);
  } else {
    tau_row<AC, KMAX>(p, int(blockIdx.x) - ncomp);
  }
}

}  // namespace

hipError_t launch_bounds(const SelectParams& p, hipStream_t s) {
  const int blocks = p.d.BH * p.d.nKB;
  const int per = kThreads / kWave;
  hipLaunchKernelGGL(bounds_kernel, dim3(unsigned((blocks + per - 1) / per)), dim3(kThreads), 0, s, p);
  return hipGetLastError();
}

// f(AC, KMAX) for the problem's exponent class and the fewest register slots
// that hold a row's k values (0: read from memory).  The sums run over every
// slot, so their number sets a launch's time where it has few rows: at
// k = 8, 8 slots against 32 took the tau and compaction launch from 14.0 to
// 7.0 us at 2x8x1024 rows (k = 16, 3x5x1537: 14.4 -> 9.4 us).
template <typename F>
void with_tau_variant(const Dims& d, F&& f) {
  auto slots = [&](auto ac) {
    if (d.k <= 8) f(ac, std::integral_constant<int, 8>{});
    else if (d.k <= 16) f(ac, std::integral_constant<int, 16>{});
    else if (d.k <= 32) f(ac, std::integral_constant<int, 32>{});
    else f(ac, std::integral_constant<int, 0>{});
  };
  switch (alpha_class_of(d.alpha)) {
    case kA15: slots(std::integral_constant<int, kA15>{}); break;
    case kA20: slots(std::integral_constant<int, kA20>{}); break;
    case kA125: slots(std::integral_constant<int, kA125>{}); break;
    default: slots(std::integral_constant<int, kAGen>{}); break;
  }
}

hipError_t launch_tau(const SelectParams& p, hipStream_t s) {
  const size_t rows = size_t(p.d.BH) * p.d.NQ;
  const dim3 grid(unsigned((rows + kThreads - 1) / kThreads));
  with_tau_variant(p.d, [&](auto ac, auto kmax) {
    hipLaunchKernelGGL((tau_kernel<decltype(ac)::value, decltype(kmax)::value>), grid, dim3(kThreads), 0, s, p);
  });
  return hipGetLastError();
}

hipError_t launch_tau_compact(const SelectParams& p, const CompactParams& cp, hipStream_t s) {
  const size_t rows = size_t(p.d.BH) * p.d.NQ;
  const int ntau = int((rows + kThreads - 1) / kThreads);
  const int ncomp = compact_detail::compact_grid(cp);
  const dim3 grid(unsigned(ntau + ncomp));
  const size_t lds = compact_detail::compact_lds_bytes(cp);
  with_tau_variant(p.d, [&](auto ac, auto kmax) {
    hipLaunchKernelGGL((tau_compact_kernel<decltype(ac)::value, decltype(kmax)::value>), grid, dim3(kThreads),
                       lds, s, p, cp, ncomp);
  });
  return hipGetLastError();
}

hipError_t launch_select(const SelectParams& p, int dtype, bool from_scores, hipStream_t s) {
  if (from_scores) return launch_select_scores(p, s);
  if (dtype == kElemBF16) return launch_select_bf16(p, s);
  if (dtype == kElemF16) return launch_select_f16(p, s);
  return launch_select_f32(p, s);
}

}  // namespace asa
