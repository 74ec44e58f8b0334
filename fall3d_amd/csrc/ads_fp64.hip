// ads_fp64.hip -- the FP64 state (FALL3D_ADS_STATE_FP64): the KT sweeps of
// Sources/mod_ADS.F90 (ADS_solve_along_x/y/z :233-815, kt_rhs :1057-1120,
// flux limiters :1124-1223, free-flow ghosts :1239-1324) and the source term
// (Sources/mod_F3D.F90:1456-1473) in double precision, every statement
// rounded as the reference writes it (the library is built without
// floating-point contraction), so that the state follows an FP64 CPU
// statement of the reference bit for bit.
//
// A thread integrates one line of one bin in one pass over its cells. The
// RK4 stages run as a pipeline along the line: at step t stage 1 forms the
// flux of face t, stage s that of face t - 2(s-1). Face f of stage s needs
// stage s's input at cells f-2 .. f+1, and stage s-1 finished cell f+1 at
// its face f+2, in the same step: each value of the line is read once and
// written once, and the stage inputs and the RK4 accumulator live in
// registers (rings of 8 entries).
#include <cmath>
#include <type_traits>

#include "ads_fp64.h"
#include "ads_quotient.h"

namespace f3d {
namespace {

constexpr double kEpsilon = 1e-12;  // EPSILON, Sources/mod_KindType.F90:42

// flux-limiter ratio r of cell i from dm = c(i) - c(i-1) and dp = c(i+1) - c(i)
// (minmod 1, superbee 2, ospre 3; Sources/mod_ADS.F90:1124-1223)
template <int LIM>
__device__ __forceinline__ double limiter64(double dm, double dp) {
  if (fabs(dp) < kEpsilon) {
    if constexpr (LIM == 1) {
      return 1.0;
    } else {
      if (fabs(dm) < kEpsilon) return 0.0;
      return LIM == 2 ? 2.0 : 1.5;
    }
  }
  const double rr = dm / dp;
  if constexpr (LIM == 1) {
    const double t = fmin(1.0, rr);
    return fmax(0.0, t);
  } else if constexpr (LIM == 2) {
    const double x = fmin(2.0 * rr, 1.0);
    const double y = fmin(rr, 2.0);
    const double m = fmax(0.0, x);
    return fmax(m, y);
  } else {
    return 1.5 * (rr * rr + rr) / (rr * rr + rr + 1.0);
  }
}

// some lane of the wave has a numerator that quot() does not take (dr is the
// last of the face: a non-finite value of any of them reaches it)
__device__ __forceinline__ bool quot_fails(double kd, double dF, double dP, double dr) {
  const double low = fmin(fmin(fabs(kd), fabs(dF)), fmin(fabs(dP), fabs(dr)));
  if (!__any(low < kQuotLow || !(fabs(dr) < kQuotHigh))) return false;
  auto tiny = [](double x) { return x != 0.0 && fabs(x) < kQuotLow; };  // zeros are fine
  return __any(tiny(kd) || tiny(dF) || tiny(dP) || tiny(dr) || !(fabs(dr) < kQuotHigh));
}
constexpr Divisor kThree = {3.0, 0x1.5555555555555p-2, 0x1.5555555555555p-56};
constexpr Divisor kSix = {6.0, 0x1.5555555555555p-3, 0x1.5555555555555p-57};

// One stage's window on its line before face f: X(f-1), X(f), their
// difference, half the limiter ratio of cell f-1, and the advective and
// diffusive fluxes of face f-1.
struct Win {
  double xm, x0, dm, hr, F, P;
};

__device__ __forceinline__ double wsum64(double v) {
  for (int o = 32; o > 0; o >>= 1) v += __shfl_down(v, o, 64);
  return v;
}

// partials[blockIdx.x*4 + s] = workgroup sum of v[s] (fixed order)
__device__ __forceinline__ void block_store4(const double (&v)[4], double *partials) {
  __shared__ double red[4][4];
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
#pragma unroll
  for (int s = 0; s < 4; ++s) {
    const double r = wsum64(v[s]);
    if (lane == 0) red[s][wid] = r;
  }
  __syncthreads();
  if (threadIdx.x < 4) {
    double sum = 0.0;
    for (int w = 0; w < (int)(blockDim.x >> 6); ++w) sum += red[threadIdx.x][w];
    partials[(size_t)blockIdx.x * 4 + threadIdx.x] = sum;
  }
}

// uniform base address + this lane's byte offset (one bin of any array here
// is below 4 GiB)
__device__ __forceinline__ double ld(const char *base, uint32_t off) { return *(const double *)(base + off); }
__device__ __forceinline__ void st(char *base, uint32_t off, double v) { *(double *)(base + off) = v; }
typedef __attribute__((address_space(4))) const Quot64 cquot;  // scalar-loaded tables

// Calls f(integral_constant<int, U>) for U = U0 .. U1-1 (compile-time unrolled).
template <int U0, int U1, class F>
__device__ __forceinline__ void unroll_range(F &&f) {
  if constexpr (U0 < U1) {
    f(std::integral_constant<int, U0>{});
    unroll_range<U0 + 1, U1>(f);
  }
}

// One thread per line and bin. Bound by FP64 VALU issue: per face and stage
// one general division (the limiter ratio), four quotients by known divisors
// (dX_p, dX_b, 6 or 3) and about 25 further operations. The loop runs in
// blocks of kRing steps, so that the values in flight sit in rings with fixed
// slots instead of being shifted every step: the line's last cells and the
// RK4 sums in registers, winds and diffusion of the last faces in LDS, which
// leaves room for three waves per SIMD (two in the x sweep, whose row pieces
// in flight take 40 registers more; three with spills is 3% slower). The next
// step's fields are loaded one step ahead. On 384 x 288 x 80 cells, 12 bins,
// minmod, RK4: y 2.49 -> 1.21 ms, z 2.51 -> 1.27 ms, x 3.77 -> 1.78 ms with the
// transposes it needs (of the state and its fields; of the fields only).
constexpr int kRing = 8;
constexpr int kTileRow = 9;  // doubles per line of an LDS tile: 8 cells and a pad (the lanes' rows on different banks)
typedef double d2a __attribute__((ext_vector_type(2), aligned(8)));

// orders a wave's LDS accesses (its lanes exchange data through its own tiles)
__device__ __forceinline__ void lds_order() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// SHORT: a stage is left out at the steps outside its faces, which are most of
// a short line's (4 cells take 16 steps of 4 stages for 24 faces); the branches
// cost a long line 4 to 6%. z of 66 x 44 x 4 x 4: 29.1 -> 19.7 us, of 323 x 24 x
// 65 x 12: 140 -> 127, of 384 x 288 x 80 x 12: 1.28 -> 1.26 ms; but y of 39 x 169 x
// 33 x 2: 258 -> 278, of 13 x 116 x 30 x 2: 204 -> 207: lines of up to kShort cells.
constexpr int kShort = 80;
template <int DIR, int LIM, int NST, bool SHORT>
__global__ void __launch_bounds__(256, DIR == 0 ? 2 : 3) k_sweep64(Sweep64Args a) {
  constexpr int LAG = 2 * (NST - 1);  // faces between stage 1 and the last stage
  const int n = a.n, nx = a.nx, ny = a.ny, nz = a.nz, nb = a.nb;
  // Thread order: 64 consecutive lines of one bin per wave, the waves after
  // it the same lines for the other bins, and the blocks renumbered so that
  // consecutive ones share an XCD: every bin of a line reads the line's winds
  // and diffusion close together in time, through one L2.
  __shared__ double tile[DIR == 0 ? 4 : 1][DIR == 0 ? 64 * kTileRow : 1];  // x sweep: a block's cells in, then out
  const int wv = threadIdx.x >> 6;
  __shared__ double led[2][256];  // per thread: the running RK-weighted F - P of either end face (a line of up to 6
                                  // cells has both in the pipeline at once)
  __shared__ double fuk[2][kRing][256];  // per thread: wind and 0.5 (K(f) + K(f-1)) of the last faces f, slot f mod kRing
  const int lane = threadIdx.x & 63;
  const long nwave = (a.nlines + 63) / 64 * nb;
  const long w0 = __builtin_amdgcn_readfirstlane(xcd_block(blockIdx.x, gridDim.x) * 4 + (int)(threadIdx.x >> 6));
  const double s = a.stime, s1 = 1.0 - a.stime, dt = a.dt, hdt = 0.5 * a.dt;
  const bool lerp = DIR == 2 || s != 0.0;  // x/y winds at stime 0 are vel1 as given
  cquot *qt = (cquot *)a.quot + kQuotLead;  // qt[p]: dX_p(p) and dX_b(p)
  double acc[4] = {0.0, 0.0, 0.0, 0.0};     // reference flux beg/end, ledger beg/end
  for (long wq = w0; wq < nwave; wq += (long)gridDim.x * 4) {
    const long chunk = wq / nb;
    const int b = (int)(wq - chunk * nb);
    const long L0 = chunk * 64 + lane;
    const bool ok = L0 < a.nlines;  // the last chunk's idle lanes
    if (DIR != 0 && !ok) continue;
    // (x sweep: the wave moves its rows together; its idle lanes repeat the last line and store nothing)
    const long L = ok ? L0 : a.nlines - 1;
    int t1, t2;  // transverse indices (x: j, k; y: i, k; z: i, j)
    uint32_t vc, vv, vk;  // lane byte offsets of position 0 of c, face 0 of the winds, position -1 of K in their bin
    size_t cst, vst;      // bytes from one position to the next
    const size_t cells = (size_t)(nx + 4) * (ny + 4) * (nz + 4);
    if constexpr (DIR == 0) {
      // fields in (x, y)-transposed layouts: wind(j, f, k), kd(j, p, k)
      t1 = (int)(L % ny) + 1;
      t2 = (int)(L / ny) + 1;
      vc = (uint32_t)(8 * (1 + (size_t)(nx + 4) * ((size_t)(t1 + 1) + (size_t)(ny + 4) * (t2 + 1))));
      cst = 8;
      vv = (uint32_t)(8 * ((size_t)(t1 - 1) + (size_t)ny * (nx + 3) * (t2 - 1)));
      vk = (uint32_t)(8 * ((size_t)(t1 - 1) + (size_t)ny * (nx + 4) * (t2 - 1)));
      vst = 8 * (size_t)ny;
    } else if constexpr (DIR == 1) {
      t1 = (int)(L % nx) + 1;
      t2 = (int)(L / nx) + 1;
      vc = (uint32_t)(8 * ((size_t)(t1 + 1) + (size_t)(nx + 4) * (1 + (size_t)(ny + 4) * (size_t)(t2 + 1))));
      cst = 8 * (size_t)(nx + 4);
      vv = (uint32_t)(8 * ((size_t)(t1 - 1) + (size_t)nx * (ny + 3) * (t2 - 1)));
      vk = (uint32_t)(8 * ((size_t)(t1 - 1) + (size_t)nx * (ny + 4) * (t2 - 1)));
      vst = 8 * (size_t)nx;
    } else {
      t1 = (int)(L % nx) + 1;
      t2 = (int)(L / nx) + 1;
      vc = (uint32_t)(8 * ((size_t)(t1 + 1) + (size_t)(nx + 4) * ((size_t)(t2 + 1) + (size_t)(ny + 4))));
      cst = 8 * (size_t)(nx + 4) * (ny + 4);
      vv = vk = (uint32_t)(8 * L);
      vst = 8 * (size_t)nx * ny;
    }
    char *cb = (char *)(a.c + cells * b);
    const char *v1b = (const char *)a.vel1, *v2b = (const char *)a.vel2, *kb = (const char *)a.kd;
    const char *sb = DIR == 2 ? (const char *)(a.vs + (size_t)nx * ny * (nz + 3) * b) : nullptr;
    auto wind = [&](double w1, double w2, double vs) -> double {
      if (!lerp) return w1;
      const double v = s1 * w1 + s * w2;
      return DIR == 2 ? v - vs : v;
    };
    auto wind_at = [&](int f) -> double {
      const size_t o = (size_t)f * vst;
      return wind(ld(v1b + o, vv), lerp ? ld(v2b + o, vv) : 0.0, DIR == 2 ? ld(sb + o, vv) : 0.0);
    };

    // boundary ghosts: with free flow, inflow at a side (u(1) > 0,
    // u(n+1) < 0) gives 2 bvalue - c with bvalue = 0 and outflow a
    // zero-gradient copy; Dirichlet always gives the former, the
    // zero-gradient rule always the latter; the outer ghost copies the inner
    const double c1 = ld(cb + cst, vc);
    const bool inw = a.bc == 0 ? (wind_at(1) > 0.0) : (a.bc == 1);
    const bool ine = a.bc == 0 ? (wind_at(n + 1) < 0.0) : (a.bc == 1);
    const double gw = inw ? 2.0 * 0.0 - c1 : c1;
    if (ok) {
      st(cb, vc, gw);
      st(cb - cst, vc, gw);
    }

    const double area = a.areaB[t2] * a.areaA[t1];
    // every stage starts as if it had run over an unbounded row of west
    // ghosts (value gw, zero differences); faces below 1 have zero fluxes
    Win w[NST];
#pragma unroll
    for (int q = 0; q < NST; ++q) w[q] = Win{gw, gw, 0.0, 0.0, 0.0, 0.0};
    // rings, slot = position (face) mod kRing: the line L(p), the RK4 sum
    // nc(i), wind and 0.5 (K(f) + K(f-1)) of the faces
    double lr[kRing], nc[kRing];
#pragma unroll
    for (int j = 0; j < kRing; ++j) {
      lr[j] = gw;
      nc[j] = 0.0;
      fuk[0][j][threadIdx.x] = fuk[1][j][threadIdx.x] = 0.0;
    }
    // x sweep: a line's cells are adjacent in memory and the lanes' lines are
    // not, so each block's 8 cells per line move through an LDS tile: 4 lanes
    // read (write) the 64 bytes of a line in 16-byte pieces, 16 lines per
    // instruction, one block ahead (behind). A finished cell takes the slot
    // of the lead value that its step has consumed.
    const int prow = lane >> 2, pcol = 2 * (lane & 3);  // line and first cell of this lane's pieces
    uint32_t vrow[4];                                   // byte offsets of position 0 of lines prow + 16 m
    bool rok[4];
    d2a ahead[4];
    auto fetch = [&](int p0) {  // positions p0 .. p0+7 of every line (past n: replaced by the ghosts)
#pragma unroll
      for (int m = 0; m < 4; ++m) ahead[m] = *(const d2a *)(cb + (size_t)(p0 + pcol) * 8 + vrow[m]);
    };
    if constexpr (DIR == 0) {
#pragma unroll
      for (int m = 0; m < 4; ++m) {
        const long Lr0 = chunk * 64 + prow + 16 * m;
        rok[m] = Lr0 < a.nlines;
        const long Lr = rok[m] ? Lr0 : a.nlines - 1;
        vrow[m] = (uint32_t)(8 * (1 + (size_t)(nx + 4) * ((size_t)(Lr % ny + 2) + (size_t)(ny + 4) * (size_t)(Lr / ny + 2))));
      }
      fetch(1);
    }
    // loaded for the next step: L(t+1), and wind and K of face / position t
    double nl = c1, n1 = ld(v1b, vv), n2 = lerp ? ld(v2b, vv) : 0.0, ns = DIR == 2 ? ld(sb, vv) : 0.0;
    double nk = ld(kb + vst, vk), kprev = 0.0;

    auto step = [&](const int t0, auto U) {
      constexpr int u = decltype(U)::value;  // t mod kRing
      int t = t0;
      __asm__ volatile("" : "+s"(t));  // its comparisons are formed here, not kept for all steps of a block
      // lead value L(t+1) (east ghosts formed from L(n) and stored)
      if constexpr (DIR == 0 && u == 0) {
        lds_order();
#pragma unroll
        for (int m = 0; m < 4; ++m) {
          tile[wv][(prow + 16 * m) * kTileRow + pcol] = ahead[m].x;
          tile[wv][(prow + 16 * m) * kTileRow + pcol + 1] = ahead[m].y;
        }
        lds_order();
        fetch(t + 1 + kRing);
      }
      double v = DIR == 0 ? tile[wv][lane * kTileRow + u] : nl;
      if (t >= n) {
        const int p = t + 1;
        v = (p == n + 1 && ine) ? 2.0 * 0.0 - lr[u] : lr[u];
        if (p <= n + 2 && ok) st(cb + (size_t)p * cst, vc, v);
      }
      lr[(u + 1) % kRing] = v;
      fuk[0][u][threadIdx.x] = wind(n1, n2, ns);
      fuk[1][u][threadIdx.x] = 0.5 * (nk + kprev);
      kprev = nk;
      {  // positions past the line's end re-read its last one; nothing uses them
        const size_t oc = (size_t)min(t + 2, n + 2) * cst, ov = (size_t)min(t + 1, n + 1) * vst;
        if constexpr (DIR != 0) nl = ld(cb + oc, vc);
        n1 = ld(v1b + ov, vv);
        if (lerp) n2 = ld(v2b + ov, vv);
        if constexpr (DIR == 2) ns = ld(sb + ov, vv);
        nk = ld(kb + ov + vst, vk);
      }
      // stages; pv carries stage q's finished cell to stage q+1 (same step)
      double pv = v;
#pragma unroll
      for (int q = 0; q < NST; ++q) {
        const int f = t - 2 * q;  // face of this stage
        const int i = f - 1;      // cell completed at this face
        constexpr int R = kRing;
        const int sf = (u - 2 * q + 2 * R) % R, sl = (u - 2 * q - 1 + 2 * R) % R;  // ring slots of face f and cell i
        if constexpr (SHORT) {  // beyond its faces 0..n+1 a stage only hands its input's ghosts on
          if (f < 0 || f > n + 1) {
            pv = lr[sl];
            continue;
          }
        }
        const double dp = pv - w[q].x0;
        const double r = limiter64<LIM>(w[q].dm, dp);
        const double hr = 0.5 * r;
        const double cl = w[q].xm + w[q].hr * w[q].dm;  // left state at face f
        const double cr = w[q].x0 - hr * dp;            // right state at face f
        const double ff = fuk[0][sf][threadIdx.x];
        const double Fl = cl * ff, Fr = cr * ff;
        const double F = 0.5 * (Fl + Fr) - 0.5 * fabs(ff) * (cr - cl);
        const double kd = fuk[1][sf][threadIdx.x] * w[q].dm;
        const bool cell = f >= 2 && f <= n + 1;  // uniform: a cell 1..n is completed
        const Divisor dp_ = {qt[i].p, qt[i].ph, qt[i].pl}, db_ = {qt[i].b, qt[i].bh, qt[i].bl};
        const double Li = lr[sl];
        double P = quot(kd, dp_);
        const double dF = F - w[q].F;
        double dP = P - w[q].P;
        double rhs = -quot(dF, db_) + quot(dP, db_);
        double dr = dt * rhs;
        const bool third = q == 1 || q == 2;
        double part = NST == 1 ? dr : quot(dr, third ? kThree : kSix);
        if (quot_fails(kd, dF, dP, dr)) {
          P = kd / dp_.d;
          dP = P - w[q].P;
          rhs = -1.0 * dF / db_.d + dP / db_.d;
          dr = dt * rhs;
          part = NST == 1 ? dr : dr / (third ? 3.0 : 6.0);
        }
        double out = Li;  // stage input of cell i for the next stage (ghosts keep L)
        if (cell) {
          if (q < NST - 1) {
            out = Li + (q < 2 ? hdt * rhs : dr);
            nc[sl] = (q == 0 ? Li : nc[sl]) + part;
          } else {
            const double done = (NST == 1 ? Li : nc[sl]) + part;
            if constexpr (DIR == 0)
              tile[wv][lane * kTileRow + u] = done;
            else
              st(cb + (size_t)i * cst, vc, done);
          }
        }
        // end faces: the RK-weighted F - P for the ledger (its sum kept in
        // LDS: it is touched a few times per line) and the last stage's F + P
        const int end = f == 1 ? 0 : (f == n + 1 ? 1 : -1);
        if (end >= 0 && ok) {
          const double d = NST == 1 ? F - P : (F - P) / (third ? 3.0 : 6.0);
          const double sum = (q == 0) ? d : led[end][threadIdx.x] + d;
          if (q < NST - 1) {
            led[end][threadIdx.x] = sum;
          } else if (end == 0) {
            acc[0] = acc[0] + (F + P) * area * dt;
            acc[2] = acc[2] - sum * area * dt;  // mass leaving through the first face
            if constexpr (DIR == 2) {
              double *ap = a.acum + (size_t)(t1 + 1) + (size_t)(nx + 4) * ((size_t)(t2 + 1) + (size_t)(ny + 4) * b);
              *ap = *ap + fabs(F + P) * dt;
            }
          } else {
            acc[1] = acc[1] + (F + P) * area * dt;
            acc[3] = acc[3] + sum * area * dt;  // mass leaving through the last face
          }
        }
        w[q].xm = w[q].x0;
        w[q].x0 = pv;
        w[q].dm = dp;
        w[q].hr = hr;
        w[q].F = F;
        w[q].P = P;
        pv = out;
        // keep the scheduler from hoisting the scalar loads and offsets of
        // the whole unrolled block to its top (SGPR spills)
        __builtin_amdgcn_sched_barrier(0);
      }
      if constexpr (DIR == 0 && u == kRing - 1) {
        // cells t-LAG-8 .. t-LAG-1 of every line: whole pieces inside 1..n, single cells at the line's ends
        lds_order();
        const int i0 = t - LAG - kRing + pcol;
#pragma unroll
        for (int m = 0; m < 4; ++m) {
          const double *row = &tile[wv][(prow + 16 * m) * kTileRow + pcol];
          char *to = cb + (ptrdiff_t)i0 * 8 + (ptrdiff_t)vrow[m];
          if (i0 >= 1 && i0 + 1 <= n) {
            if (rok[m]) *(d2a *)to = d2a{row[0], row[1]};
          } else if (rok[m]) {
            if (i0 >= 1 && i0 <= n) *(double *)to = row[0];
            if (i0 + 1 >= 1 && i0 + 1 <= n) *(double *)(to + 8) = row[1];
          }
        }
        lds_order();
      }
    };
    for (int t = 0; t <= n + 1 + LAG; t += kRing)
      unroll_range<0, kRing>([&](auto U) { step(t + decltype(U)::value, U); });
  }
  block_store4(acc, a.partials);
}

template <int DIR, int LIM, int NST>
hipError_t launch_nst(const Sweep64Args &a, int nblocks, hipStream_t st) {
  if (a.n <= kShort)
    hipLaunchKernelGGL((k_sweep64<DIR, LIM, NST, true>), dim3(nblocks), dim3(256), 0, st, a);
  else
    hipLaunchKernelGGL((k_sweep64<DIR, LIM, NST, false>), dim3(nblocks), dim3(256), 0, st, a);
  return hipGetLastError();
}

template <int DIR, int LIM>
hipError_t launch_lim(int tm, const Sweep64Args &a, int nblocks, hipStream_t st) {
  return tm == 1 ? launch_nst<DIR, LIM, 1>(a, nblocks, st) : launch_nst<DIR, LIM, 4>(a, nblocks, st);
}

template <int DIR>
hipError_t launch_dir(int limiter, const Sweep64Args &a, int nblocks, hipStream_t st) {
  if (limiter == 1) return launch_lim<DIR, 1>(a.tm, a, nblocks, st);
  if (limiter == 2) return launch_lim<DIR, 2>(a.tm, a, nblocks, st);
  return launch_lim<DIR, 3>(a.tm, a, nblocks, st);
}

__global__ void k_source64(double *__restrict__ c, const size_t *__restrict__ idx, const double *__restrict__ s,
                           const double *__restrict__ vol, const double *__restrict__ meas, int nent, double dt,
                           double *__restrict__ partials) {
  const int e = blockIdx.x * blockDim.x + threadIdx.x;
  double v[4] = {0.0, 0.0, 0.0, 0.0};
  if (e < nent) {
    const size_t i = idx[e];
    const double inc = dt * s[e] / vol[e];
    c[i] = c[i] + inc;
    v[0] = inc * meas[e];
  }
  block_store4(v, partials);
}

}  // namespace

int sweep64_blocks(long nlines, int nb) {
  const long g = ((nlines + 63) / 64 * 64 * (long)nb + 255) / 256;
  return (int)(g < 1 ? 1 : (g > kSweep64MaxBlocks ? kSweep64MaxBlocks : g));
}

hipError_t launch_sweep64(int dir, int limiter, const Sweep64Args &a, int nblocks, hipStream_t st) {
  (void)hipGetLastError();  // drop errors of earlier, unrelated calls
  if (dir == 0) return launch_dir<0>(limiter, a, nblocks, st);
  if (dir == 1) return launch_dir<1>(limiter, a, nblocks, st);
  return launch_dir<2>(limiter, a, nblocks, st);
}

hipError_t source_inject64(double *c, const size_t *idx, const double *s, const double *vol, const double *meas,
                           int nent, double dt, double *partials, int *nblocks, hipStream_t st) {
  (void)hipGetLastError();
  const int nb = (nent + 255) / 256;
  *nblocks = nb;
  if (nb == 0) return hipSuccess;
  hipLaunchKernelGGL(k_source64, dim3(nb), dim3(256), 0, st, c, idx, s, vol, meas, nent, dt, partials);
  return hipGetLastError();
}

}  // namespace f3d
