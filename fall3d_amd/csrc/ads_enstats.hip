// ads_enstats.hip -- ensemble statistics over member fields on gfx950
// (the statistics of Sources/task_PosEns.F90:319-441, computed per grid
// point over the members of an ensemble).
//
// Input: nmem member fields of npoints values each, member-major on the
// device (x[m * npoints + p], FP64). Outputs per point, each optional:
//   mean      sum_m x_m / nmem                       (task_PosEns.F90:321-329)
//   logmean   10^(sum_m log10 x_m / nmem)            (:334-343)
//   stddev    sqrt(sum_m (x_m - mean)^2 / (nmem-1))  (:348-365, see below)
//   median    r(int(nmem/2)), r the values in ascending order, 1-based
//                                                    (:369-383; postp_rank_vector
//                                                     sorts ascending, mod_Postp.F90:181)
//   per[i]    r(min(max(int(p_i/100 nmem), 1), nmem)) (:415-437)
//   prob[i]   100 #{m : x_m >= th_i} / nmem          (:388-410)
// The reference's standard-deviation loop assigns instead of accumulating
// (:356-360), so it would keep only the last member's squared deviation;
// this computes the sum its division by nens-1 is written for.
//
// The member fields are read once. Up to 64 members a thread owns a point and
// keeps its values in registers (loads coalesced across the points): sums in
// member order, then an odd-even merge network for the ranks. Up to 1024
// members a workgroup moves the values of a few neighbouring points into LDS
// and each of its waves sorts one point at a time there.
//
// The sum of logarithms is the logarithm of the product: mantissas multiply,
// exponents add, and one log10 per point closes it (closer to the sum than
// adding rounded logarithms, and 48 log10 fewer at 48 members).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <utility>

#include "../../include/fall3d_ads.h"

namespace f3d {
namespace {

struct StatsArgs {
  const double *x;
  long npoints;
  int nmem;
  int nper, nth;
  const double *per_val;  // percentiles in percent (device)
  const double *th_val;   // thresholds (device)
  double *mean, *logmean, *stddev, *median, *per, *prob;
};

// 1-based rank of percentile p (task_PosEns.F90:429-431)
__device__ __forceinline__ int per_rank(double p, int nmem) {
  int n = (int)(p / 100.0 * nmem);
  n = n < 1 ? 1 : n;
  return n > nmem ? nmem : n;
}

// product of positive values as mantissa and exponent
struct Product {
  double mant = 1.0;
  int ex = 0;
  __device__ __forceinline__ void times(double v) {
    mant = mant * __builtin_amdgcn_frexp_mant(v);
    ex += __builtin_amdgcn_frexp_exp(v);
  }
  __device__ __forceinline__ void normalise() {  // before 1000 mantissas of at least 1/2 can underflow
    ex += __builtin_amdgcn_frexp_exp(mant);
    mant = __builtin_amdgcn_frexp_mant(mant);
  }
  // sum of the log10 of the values; neg: one of them was below zero
  __device__ __forceinline__ double log10sum(bool neg) const {
    constexpr double hi = 0x1.34413509f79ffp-2, lo = -0x1.9dc1da994fd21p-59;  // log10(2)
    const double l = fma((double)ex, hi, fma((double)ex, lo, log10(mant)));
    return neg ? NAN : l;
  }
};

// v[r] of a register array, r the same in every lane: a tree of uniform branches
template <int LO, int HI, int P>
__device__ __forceinline__ double pick(const double (&v)[P], int r) {
  if constexpr (HI - LO == 1) {
    double out = v[LO];
    __asm__ volatile("" : "+v"(out));  // a value, not one of several addresses (the array would leave the registers)
    return out;
  } else {
    constexpr int MID = (LO + HI) / 2;
    double out;
    if (r < MID)
      out = pick<LO, MID, P>(v, r);
    else
      out = pick<MID, HI, P>(v, r);
    return out;
  }
}

// Batcher's odd-even merge sort, ascending; comparators that reach past P
// fall away (the missing values count as +infinity, which never moves down).
// The network is a compile-time list, so that the values stay in registers.
template <int P>
struct Network {
  int n = 0;
  unsigned char lo[544] = {}, hi[544] = {};  // 543 comparators at 64 values
  constexpr Network() {
    for (int p = 1; p < P; p <<= 1)
      for (int k = p; k >= 1; k >>= 1)
        for (int j = k % p; j + k < 64; j += 2 * k)
          for (int i = 0; i < k; ++i) {
            const int l = i + j, h = i + j + k;
            if (h < P && l / (2 * p) == h / (2 * p)) {
              lo[n] = (unsigned char)l;
              hi[n] = (unsigned char)h;
              ++n;
            }
          }
  }
};
template <int P>
constexpr Network<P> kNetwork{};

__device__ __forceinline__ void exchange(double &a, double &b) {
  const double lo = fmin(a, b), hi = fmax(a, b);
  a = lo;
  b = hi;
}
template <int P, size_t... I>
__device__ __forceinline__ void merge_sort(double (&v)[P], std::index_sequence<I...>) {
  (exchange(v[kNetwork<P>.lo[I]], v[kNetwork<P>.hi[I]]), ...);
}

// nmem in P-7 .. P. Bound by memory (8 nmem bytes per point) and the exchanges
// of the network: 48 members of 480 000 points with 4 percentiles and 4
// thresholds take 64 us (3.6 TB/s of reads and writes); 506 us when moments,
// thresholds and ranks each read the fields again and every member took a
// log10.
template <int P>
__global__ void __launch_bounds__(256, P <= 24 ? 4 : (P <= 48 ? 3 : 2)) k_stats_reg(StatsArgs a, long first) {
  // (no loop over points: one would keep the polynomials' coefficients in
  // registers from one to the next)
  const int M = a.nmem;
  const long p0 = first + (long)blockIdx.x * 256, p = p0 + threadIdx.x;
  if (p >= a.npoints) return;
  double v[P];
  const double *row = a.x + p0;  // uniform: member m's values of this workgroup
#pragma unroll
  for (int m = 0; m < P; ++m) {
    v[m] = (m < P - 7 || m < M) ? row[threadIdx.x] : INFINITY;
    row += a.npoints;
  }
  // f(value) for the members in order (the last ones' presence is uniform)
  auto members = [&](auto &&f) {
#pragma unroll
    for (int m = 0; m < P; ++m)
      if (m < P - 7 || m < M) f(v[m]);
  };
  double s = 0.0;
  members([&](double x) { s = s + x; });
  const double mu = s / M;
  if (a.mean) a.mean[p] = mu;
  if (a.logmean) {
    Product pr;
    double least = INFINITY;
    members([&](double x) {
      pr.times(x);
      least = fmin(least, x);
    });
    a.logmean[p] = pow(10.0, pr.log10sum(least < 0.0) / M);
  }
  if (a.stddev) {
    double q = 0.0;
    members([&](double x) {
      const double d = x - mu;
      q = q + d * d;
    });
    a.stddev[p] = M > 1 ? sqrt(q / (M - 1)) : 0.0;
  }
  for (int t = 0; t < a.nth; ++t) {
    const double th = a.th_val[t];
    int n = 0;
    members([&](double x) { n += (x >= th) ? 1 : 0; });
    a.prob[(size_t)t * a.npoints + p] = 100.0 * n / M;
  }
  if (!a.median && !a.per) return;
  merge_sort<P>(v, std::make_index_sequence<kNetwork<P>.n>());
  if (a.median) a.median[p] = pick<0, P, P>(v, (M / 2 > 0 ? M / 2 : 1) - 1);
  for (int i = 0; i < a.nper; ++i) {
    const int r = __builtin_amdgcn_readfirstlane(per_rank(a.per_val[i], M) - 1);
    a.per[(size_t)i * a.npoints + p] = pick<0, P, P>(v, r);
  }
}

__device__ __forceinline__ double wave_sum(double v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  return v;
}

// T neighbouring points per workgroup of four waves, their values in LDS rows
// of P + 1 doubles (padded with +infinity); a wave takes a point at a time.
// (A wave per point that reads its values by itself touches a line of memory
// per value: 100 members of 120 000 points 4.5 ms that way, 0.33 ms in tiles.)
template <int P, int T>
__global__ void __launch_bounds__(256) k_stats_lds(StatsArgs a) {
  extern __shared__ double slds[];
  constexpr int J = P / 64;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, M = a.nmem;
  for (long p0 = (long)blockIdx.x * T; p0 < a.npoints; p0 += (long)gridDim.x * T) {
    __syncthreads();  // the previous points' rows are free
    for (int e = threadIdx.x; e < P * T; e += 256) {
      const int m = e / T, q = e % T;
      slds[q * (P + 1) + m] = (m < M && p0 + q < a.npoints) ? a.x[(size_t)m * a.npoints + p0 + q] : INFINITY;
    }
    __syncthreads();
    for (int q = wave; q < T && p0 + q < a.npoints; q += 4) {
      const long p = p0 + q;
      double *v = slds + q * (P + 1);
      double r[J];
#pragma unroll
      for (int j = 0; j < J; ++j) r[j] = v[lane + 64 * j];
      auto members = [&](auto &&f) {
#pragma unroll
        for (int j = 0; j < J; ++j)
          if (lane + 64 * j < M) f(r[j]);
      };
      double s = 0.0;
      members([&](double x) { s = s + x; });
      const double mu = wave_sum(s) / M;
      if (a.mean && lane == 0) a.mean[p] = mu;
      if (a.logmean) {
        Product pr;
        bool neg = false;
        members([&](double x) {
          pr.times(x);
          neg |= x < 0.0;
        });
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) {
          pr.mant = pr.mant * __shfl_xor(pr.mant, o, 64);
          pr.ex += __shfl_xor(pr.ex, o, 64);
          pr.normalise();
        }
        const bool any = __any(neg);
        if (lane == 0) a.logmean[p] = pow(10.0, pr.log10sum(any) / M);
      }
      if (a.stddev) {
        double d2 = 0.0;
        members([&](double x) {
          const double d = x - mu;
          d2 = d2 + d * d;
        });
        d2 = wave_sum(d2);
        if (lane == 0) a.stddev[p] = sqrt(d2 / (M - 1));
      }
      for (int t = 0; t < a.nth; ++t) {
        const double th = a.th_val[t];
        int n = 0;
#pragma unroll
        for (int j = 0; j < J; ++j) n += __popcll(__ballot(lane + 64 * j < M && r[j] >= th));
        if (lane == 0) a.prob[(size_t)t * a.npoints + p] = 100.0 * n / M;
      }
      if (!a.median && !a.per) continue;
      // bitonic sort in the wave's row: pair e of a step compares i and i + j
      auto order = [] {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
      };
      for (int k = 2; k <= P; k <<= 1)
        for (int j = k >> 1; j > 0; j >>= 1) {
#pragma unroll
          for (int e = lane; e < P / 2; e += 64) {
            const int i = ((e & ~(j - 1)) << 1) | (e & (j - 1)), l = i + j;
            const bool up = (i & k) == 0;
            const double x0 = v[i], x1 = v[l];
            const double lo = fmin(x0, x1), hi = fmax(x0, x1);
            v[i] = up ? lo : hi;
            v[l] = up ? hi : lo;
          }
          order();
        }
      if (lane == 0) {
        if (a.median) a.median[p] = v[M / 2 - 1];
        for (int i = 0; i < a.nper; ++i) a.per[(size_t)i * a.npoints + p] = v[per_rank(a.per_val[i], M) - 1];
      }
      order();
    }
  }
}

// points per workgroup of k_stats_lds: 128-byte pieces of the member rows
// while the rows of 16 points leave a CU three workgroups, fewer beyond
template <int P>
hipError_t launch_lds(const StatsArgs &a, hipStream_t st) {
  constexpr int T = P <= 256 ? 16 : (P <= 512 ? 8 : 4);
  const long blocks = std::min<long>((a.npoints + T - 1) / T, 65536);
  hipLaunchKernelGGL((k_stats_lds<P, T>), dim3((unsigned)blocks), dim3(256), (size_t)T * (P + 1) * sizeof(double), st, a);
  return hipGetLastError();
}

template <int P>
hipError_t launch_reg(const StatsArgs &a, hipStream_t st) {
  constexpr long kBlocks = 1l << 23;  // a grid axis holds fewer than 2^32 threads
  for (long first = 0; first < a.npoints; first += 256 * kBlocks) {
    const long blocks = std::min<long>((a.npoints - first + 255) / 256, kBlocks);
    hipLaunchKernelGGL(k_stats_reg<P>, dim3((unsigned)blocks), dim3(256), 0, st, a, first);
  }
  return hipGetLastError();
}

hipError_t launch_stats(const StatsArgs &a, hipStream_t st) {
  switch ((a.nmem + 7) / 8) {
    case 1: return launch_reg<8>(a, st);
    case 2: return launch_reg<16>(a, st);
    case 3: return launch_reg<24>(a, st);
    case 4: return launch_reg<32>(a, st);
    case 5: return launch_reg<40>(a, st);
    case 6: return launch_reg<48>(a, st);
    case 7: return launch_reg<56>(a, st);
    case 8: return launch_reg<64>(a, st);
  }
  if (a.nmem <= 128) return launch_lds<128>(a, st);
  if (a.nmem <= 256) return launch_lds<256>(a, st);
  if (a.nmem <= 512) return launch_lds<512>(a, st);
  return launch_lds<1024>(a, st);
}

}  // namespace
}  // namespace f3d

using namespace f3d;

extern "C" int fall3d_ens_statistics(const double *x, int nmem, long npoints, const double *percentiles, int nper,
                                     const double *thresholds, int nth, double *mean, double *logmean,
                                     double *stddev, double *median, double *per, double *prob, void *stream) {
  if (!x || nmem < 1 || nmem > 1024 || npoints < 0 || nper < 0 || nth < 0) return FALL3D_ADS_EINVAL;
  if ((nper > 0 && (!percentiles || !per)) || (nth > 0 && (!thresholds || !prob))) return FALL3D_ADS_EINVAL;
  if (npoints == 0) return FALL3D_ADS_OK;
  hipStream_t st = (hipStream_t)stream;
  StatsArgs a;
  a.x = x;
  a.npoints = npoints;
  a.nmem = nmem;
  a.nper = nper;
  a.nth = nth;
  a.per_val = percentiles;
  a.th_val = thresholds;
  a.mean = mean;
  a.logmean = logmean;
  a.stddev = stddev;
  a.median = median;
  a.per = nper > 0 ? per : nullptr;
  a.prob = nth > 0 ? prob : nullptr;
  (void)hipGetLastError();
  if (launch_stats(a, st) != hipSuccess) return FALL3D_ADS_EHIP;
  return hipStreamSynchronize(st) == hipSuccess ? FALL3D_ADS_OK : FALL3D_ADS_EHIP;
}
