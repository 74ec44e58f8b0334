// ads_output.hip -- the output post-processing of nc_IO_out_res
// (Sources/mod_nc_IO.F90:3206-4335) on the device, for the context's state:
//
//   c scaled back by the map factors, converted to g/m3 and clipped at 0 on
//   the mass points with their 2 ghosts (map factors at the clamped index)
//                                                        mod_nc_IO.F90:3397-3416
//   mass points -> cell corners, 8-point average          mod_Grid.F90:1150-1181
//   ground accumulation -> corners, 4-point average of the clamped field
//                                                        mod_Grid.F90:1190-1220
//   per species: 3-D concentration (CON), surface concentration (CON_SUR),
//   column load by the trapezoid rule over the corner heights (COL_MASS,
//   optionally in Dobson units), PM column loads (COL_MASS_PM), cloud-top
//   height at 50 ug/m3 (CLOUD_TOP), ground load total and per bin (GRN_LOAD,
//   GRN_LOAD_BIN)                                        mod_nc_IO.F90:3506-4020
//
// Corner concentrations are formed with one thread per corner (bins in order),
// then one thread per corner column walks up its levels for the integrals, so
// every sum runs in the reference's order; neighbouring threads own
// neighbouring corners (coalesced along x).
#include <algorithm>
#include <cmath>
#include <cstring>
#include <vector>

#include "ads_aux.h"
#include "ads_context.h"
#include "ads_quotient.h"

namespace f3d {
namespace {

struct OutArgs {
  const float *chi, *clo;  // FP32 state (lo: compensated) or
  const double *c64;       // FP64 state
  const double *acum;      // acum(-1:nx+2,-1:ny+2,nb)
  int nx, ny, nz, nb;
  const double *hm1, *hm2, *hm3;  // Hm1_p(1:ny), Hm2_p(-1:ny+2), Hm3_p(1:nx,1:ny)
  const double *zc;               // corner heights (nx+1)(ny+1)(nz+1)
  const int *spe;                 // per bin species code
  const int *pm_bin;              // per bin: bit p set when the bin counts for PM threshold p
  int species, so2_du, npm, pm_ok;
  // outputs (corner layouts, FP64; any may be nullptr)
  double *con_bins;     // (nx+1)(ny+1)(nz+1) nb
  double *con;          // (nx+1)(ny+1)(nz+1)
  double *con_sur;      // (nx+1)(ny+1)
  double *col_mass;     // (nx+1)(ny+1)
  double *col_mass_pm;  // (nx+1)(ny+1) npm
  double *cloud_top;    // (nx+1)(ny+1)
  double *grn_load;     // (nx+1)(ny+1)
  double *grn_load_bin; // (nx+1)(ny+1) nb
  double *wpm;          // scratch, (nx+1)(ny+1)(nz+1) npm: the PM classes' concentrations
};

constexpr int kMaxPm = 8;

__device__ __forceinline__ int clampi(int v, int lo, int hi) { return v < lo ? lo : (v > hi ? hi : v); }

// Map factor product of a column (clamped indices) as a divisor, and whether
// it is of ordinary size.
struct Scale {
  Divisor v;
  bool plain;
};
__device__ __forceinline__ Scale column_scale(const OutArgs &a, int i, int j) {
  const int jj = clampi(j, 1, a.ny), ii = clampi(i, 1, a.nx);
  const double hm1 = a.hm1[jj - 1], hm2 = a.hm2[jj + 1], hm3 = a.hm3[(size_t)(ii - 1) + (size_t)a.nx * (jj - 1)];
  const double d = hm1 * hm2 * hm3;
  return {divisor(d), fabs(d) > 0x1p-100 && fabs(d) < 0x1p100};
}
// scaled-back, clipped concentration in g/m3
__device__ __forceinline__ double unscaled(double c, const Scale &s) {
  const double x = 1e3 * c, t = fabs(x);
  const double v = (s.plain && !(t < kQuotLow && t != 0.0) && !(t >= kQuotHigh)) ? quot(x, s.v) : x / s.v.d;
  return fmax(0.0, v);
}

// Corner concentrations: 8-point averages per bin, their sum over the species'
// bins and over each PM class. A wave takes 63 corners of a row: lane l holds
// the mass points at i = first + l - 1 of the rows j and j - 1 and the levels k
// and k - 1, and hands them to the next lane, whose corner they adjoin on the
// west side. Bound by the loads of the state (each value read by two rows and
// two levels, mostly from the L2): 360 x 240 x 60 x 10 1.85 ms with one thread
// per corner column walking up and eight general divisions per corner, 0.35 ms now.
constexpr int kCornersPerWave = 63;
template <typename T, bool LOW>
__global__ void __launch_bounds__(256) k_corners(OutArgs a) {
  const T *__restrict__ c = LOW || sizeof(T) == 4 ? (const T *)a.chi : (const T *)a.c64;
  const int nx = a.nx, ny = a.ny, nz = a.nz;
  const int px = sizeof(T) == 8 ? nx + 4 : state_pitch(nx);  // x pitch of c64 / chi
  const int pieces = (nx + 1 + kCornersPerWave - 1) / kCornersPerWave;
  const size_t rows = (size_t)(ny + 1) * (nz + 1), ncol = (size_t)(nx + 1) * (ny + 1), n3 = ncol * (nz + 1);
  const int lane = threadIdx.x & 63;
  const size_t bin = (size_t)px * (ny + 4) * (nz + 4);
  for (size_t w = (size_t)blockIdx.x * 4 + (threadIdx.x >> 6); w < rows * pieces; w += (size_t)gridDim.x * 4) {
    const size_t row = w / pieces;
    const int piece = (int)(w - row * pieces);
    const int k = (int)(row / (ny + 1)) + 1, j = (int)(row % (ny + 1)) + 1;
    const int i = piece * kCornersPerWave + lane;  // mass point; corner i (lane 0's belongs to the piece before)
    const int im = i <= nx + 1 ? i : nx + 1;
    const bool out = lane > 0 && i <= nx + 1;
    const Scale s1 = column_scale(a, im, j), s0 = column_scale(a, im, j - 1);
    // mass points (im, j), (im, j-1) at levels k and k-1
    const size_t m11 = (size_t)(im + 1) + (size_t)px * ((size_t)(j + 1) + (size_t)(ny + 4) * (k + 1));
    const size_t m10 = m11 - (size_t)px * (ny + 4), o = (size_t)(i - 1) + (size_t)(nx + 1) * (j - 1) + ncol * (size_t)(k - 1);
    auto at = [&](size_t m, size_t b) -> double {
      double v = (double)c[m + bin * b];
      if constexpr (LOW) v += (double)a.clo[m + bin * b];
      return v;
    };
    double sum = 0.0, wp[kMaxPm];
    for (int p = 0; p < kMaxPm; ++p) wp[p] = 0.0;
    for (int b = 0; b < a.nb; ++b) {
      const double e11 = unscaled(at(m11, b), s1), e01 = unscaled(at(m11 - px, b), s0);
      const double e10 = unscaled(at(m10, b), s1), e00 = unscaled(at(m10 - px, b), s0);
      const double w11 = __shfl_up(e11, 1, 64), w01 = __shfl_up(e01, 1, 64);
      const double w10 = __shfl_up(e10, 1, 64), w00 = __shfl_up(e00, 1, 64);
      const double v = (e11 + w11 + e01 + w01 + e10 + w10 + e00 + w00) / 8.0;
      if (a.con_bins && out) a.con_bins[o + n3 * (size_t)b] = v;
      if (a.spe[b] != a.species) continue;
      sum = sum + v;
      if (a.pm_ok)
        for (int p = 0; p < a.npm; ++p)
          if ((a.pm_bin[b] >> p) & 1) wp[p] = wp[p] + v;
    }
    if (!out) continue;
    if (a.con) a.con[o] = sum;
    if (k == 1 && a.con_sur) a.con_sur[o] = sum;
    if (a.pm_ok)
      for (int p = 0; p < a.npm; ++p) a.wpm[o + n3 * (size_t)p] = wp[p];
  }
}

// column products and ground loads, one thread per corner column
__global__ void __launch_bounds__(256) k_columns(OutArgs a) {
  const int nx = a.nx, ny = a.ny, nz = a.nz;
  const size_t ncol = (size_t)(nx + 1) * (ny + 1);
  const size_t n3 = ncol * (nz + 1);
  for (size_t col = blockIdx.x * (size_t)blockDim.x + threadIdx.x; col < ncol; col += (size_t)gridDim.x * blockDim.x) {
    const int i = (int)(col % (nx + 1)) + 1;
    const int j = (int)(col / (nx + 1)) + 1;
    if (a.col_mass || a.cloud_top || a.pm_ok) {
      double load = 0.0, top = 0.0, wprev = 0.0, zprev = 0.0;
#pragma unroll 8
      for (int k = 1; k <= nz + 1; ++k) {
        const size_t o = col + ncol * (size_t)(k - 1);
        const double w = a.con[o], z = a.zc[o];
        if (k > 1) load = load + 0.5 * (wprev + w) * (z - zprev);
        if (w > 50e-6) top = z;  // the highest level above the threshold wins
        wprev = w;
        zprev = z;
      }
      if (a.so2_du) load = load / 64.0 * 2.238e3;
      if (a.col_mass) a.col_mass[col] = load;
      if (a.cloud_top) a.cloud_top[col] = top;
      if (a.col_mass_pm && a.pm_ok)
        for (int p = 0; p < a.npm; ++p) {
          double pm = 0.0;
          wprev = zprev = 0.0;
#pragma unroll 8
          for (int k = 1; k <= nz + 1; ++k) {
            const size_t o = col + ncol * (size_t)(k - 1);
            const double w = a.wpm[o + n3 * (size_t)p], z = a.zc[o];
            if (k > 1) pm = pm + 0.5 * (wprev + w) * (z - zprev);
            wprev = w;
            zprev = z;
          }
          a.col_mass_pm[col + ncol * (size_t)p] = pm;
        }
    }
    // ground accumulation at the corner (clamped mass points), kg/m2
    if (!a.grn_load && !a.grn_load_bin) continue;
    double g = 0.0;
    const int i0 = clampi(i - 1, 1, nx), i1 = clampi(i, 1, nx), j0 = clampi(j - 1, 1, ny), j1 = clampi(j, 1, ny);
#pragma unroll 2
    for (int b = 0; b < a.nb; ++b) {
      auto A = [&](int ii, int jj) {
        return a.acum[(size_t)(ii + 1) + (size_t)(nx + 4) * ((size_t)(jj + 1) + (size_t)(ny + 4) * b)];
      };
      const double ac = (A(i1, j1) + A(i0, j1) + A(i1, j0) + A(i0, j0)) / 4.0;
      if (a.grn_load_bin) a.grn_load_bin[col + ncol * (size_t)b] = ac;
      if (a.spe[b] == a.species) g = g + ac;
    }
    if (a.grn_load) a.grn_load[col] = g;
  }
}

hipError_t launch_output(const OutArgs &a, hipStream_t st) {
  (void)hipGetLastError();
  const size_t ncol = (size_t)(a.nx + 1) * (a.ny + 1);
  const size_t pieces = (size_t)((a.nx + kCornersPerWave) / kCornersPerWave);
  const size_t waves = pieces * (a.ny + 1) * (a.nz + 1);
  const dim3 grid((unsigned)std::min<size_t>((waves + 3) / 4, 1u << 22));
  if (a.con_bins || a.con) {
    if (a.c64)
      hipLaunchKernelGGL((k_corners<double, false>), grid, dim3(256), 0, st, a);
    else if (a.clo)
      hipLaunchKernelGGL((k_corners<float, true>), grid, dim3(256), 0, st, a);
    else
      hipLaunchKernelGGL((k_corners<float, false>), grid, dim3(256), 0, st, a);
  }
  if (a.col_mass || a.cloud_top || a.pm_ok || a.grn_load || a.grn_load_bin)
    hipLaunchKernelGGL(k_columns, dim3((unsigned)std::min<size_t>((ncol + 255) / 256, 65536)), dim3(256), 0, st, a);
  return hipGetLastError();
}

// grid_get_shapez (Sources/mod_Grid.F90:1287-1329) over v(1..n) (element
// q at v[(q-1) * stride]): the interval [v(k), v(k+1)] holding z, searched
// from the bottom, and the linear weight of v(k+1); below v(1) it gives
// (1, 0), above v(n) (n-1, 1).
__host__ __device__ inline void shapez(const double *v, size_t stride, int n, double z, int &ik, double &s) {
  if (z < v[0]) {
    ik = 1;
    s = 0.0;
    return;
  }
  if (z > v[(size_t)(n - 1) * stride]) {
    ik = n - 1;
    s = 1.0;
    return;
  }
  for (int k = 1; k < n; ++k) {
    const double lo = v[(size_t)(k - 1) * stride], hi = v[(size_t)k * stride];
    if (z >= lo && z <= hi) {
      ik = k;
      s = (z - lo) / (hi - lo);
      return;
    }
  }
  ik = 1;  // only for a column that is not ordered upward (the reference never ends its search then)
  s = 0.0;
}

// the species' corner concentration on the z levels zl(1..nz+1) above sea
// level: per corner column, interpolated over the column's own corner
// heights (mod_nc_IO.F90:3302-3313 and 4102-4117); one thread per column and
// level (360 x 240 x 60: 617 us with a thread walking all levels, 209 now)
__global__ void __launch_bounds__(256) k_zlevels(const double *__restrict__ con, const double *__restrict__ zc,
                                                 const double *__restrict__ zl, int nx, int ny, int nz,
                                                 double *__restrict__ cz) {
  const size_t ncol = (size_t)(nx + 1) * (ny + 1);
  for (size_t col = blockIdx.x * (size_t)blockDim.x + threadIdx.x; col < ncol; col += (size_t)gridDim.x * blockDim.x) {
    for (int k = blockIdx.y + 1; k <= nz + 1; k += gridDim.y) {
      int kk;
      double sh;
      shapez(zc + col, ncol, nz + 1, zl[k - 1], kk, sh);
      cz[col + ncol * (size_t)(k - 1)] =
          kk > 0 ? (1.0 - sh) * con[col + ncol * (size_t)(kk - 1)] + sh * con[col + ncol * (size_t)kk] : 0.0;
    }
  }
}

// Cuts of cz (mod_nc_IO.F90:4126-4332): mode 0 x cuts (ny+1, nz+1, ncut),
// 1 y cuts (nx+1, nz+1, ncut), 2 z or flight-level cuts (nx+1, ny+1, ncut);
// cut q interpolates between positions idx[q] and idx[q]+1 with weight sh[q].
__global__ void __launch_bounds__(256) k_cuts(const double *__restrict__ cz, int nx, int ny, int nz, int mode,
                                              int ncut, const int *__restrict__ idx, const double *__restrict__ sh,
                                              double *__restrict__ out) {
  const size_t n1 = (size_t)(mode == 0 ? ny + 1 : nx + 1), n2 = (size_t)(mode == 2 ? ny + 1 : nz + 1);
  const size_t total = n1 * n2 * (size_t)ncut;
  const size_t sx = 1, sy = (size_t)(nx + 1), sz = (size_t)(nx + 1) * (ny + 1);
  for (size_t e = blockIdx.x * (size_t)blockDim.x + threadIdx.x; e < total; e += (size_t)gridDim.x * blockDim.x) {
    const size_t a = e % n1, r = e / n1, b = r % n2;
    const int q = (int)(r / n2);
    const size_t m = (size_t)(idx[q] - 1);
    size_t lo, step;
    if (mode == 0) {  // (j, k) at x position m
      lo = m * sx + a * sy + b * sz;
      step = sx;
    } else if (mode == 1) {  // (i, k) at y position m
      lo = a * sx + m * sy + b * sz;
      step = sy;
    } else {  // (i, j) at level m
      lo = a * sx + b * sy + m * sz;
      step = sz;
    }
    out[e] = (1.0 - sh[q]) * cz[lo] + sh[q] * cz[lo + step];
  }
}

}  // namespace
}  // namespace f3d

using namespace f3d;
using namespace f3d::host;

namespace {

// cut request of fall3d_ads_postprocess_cuts: host outputs x, y, z, FL
struct CutReq {
  const fall3d_cut_args *args;
  double *out[4];
};

int postprocess_impl(fall3d_ads_ctx *c, const fall3d_output_args *o, double *con_bins, double *con, double *con_sur,
                     double *col_mass, double *col_mass_pm, double *cloud_top, double *grn_load,
                     double *grn_load_bin, const CutReq *cut) {
  if (!c) return FALL3D_ADS_EINVAL;
  if (!o) return fail(c, FALL3D_ADS_EINVAL, "null argument");
  if (cut) {
    const fall3d_cut_args *ca = cut->args;
    if (!ca) return fail(c, FALL3D_ADS_EINVAL, "null cut arguments");
    if (!o->z_c || !ca->sigma) return fail(c, FALL3D_ADS_EINVAL, "cuts need the corner heights z_c and sigma levels");
    const int ncut[4] = {ca->ncutx, ca->ncuty, ca->ncutz, ca->nfl};
    const double *pos[4] = {ca->x_cut, ca->y_cut, ca->z_cut, ca->fl_cut};
    for (int q = 0; q < 4; ++q)
      if (ncut[q] < 0 || (ncut[q] > 0 && (!pos[q] || !cut->out[q])))
        return fail(c, FALL3D_ADS_EINVAL, "cut kind %d: positive count needs positions and an output", q);
  }
  if (!c->grid_ok) return fail(c, FALL3D_ADS_ESTATE, "fall3d_ads_set_grid has not been called");
  if (o->npm < 0 || o->npm > kMaxPm) return fail(c, FALL3D_ADS_EINVAL, "at most %d PM thresholds", kMaxPm);
  if ((col_mass || col_mass_pm || cloud_top) && !o->z_c)
    return fail(c, FALL3D_ADS_EINVAL, "column loads and cloud top need the corner heights z_c");
  if (col_mass_pm && o->npm > 0 && (!o->pm_um || !o->bin_diam))
    return fail(c, FALL3D_ADS_EINVAL, "PM loads need the thresholds and the bin diameters");
  const int nx = c->nx, ny = c->ny, nz = c->nz, nb = c->nb;
  const size_t ncol = (size_t)(nx + 1) * (ny + 1), n3 = ncol * (nz + 1);
  // host-side tables: vertical and horizontal map factors (1 when not given),
  // species, PM membership
  std::vector<double> hm1(ny, 1.0), hm2(ny + 4, 1.0), hm3;
  auto hv = [&](const void *p, size_t q) {
    return c->kind == 8 ? ((const double *)p)[q] : (double)((const float *)p)[q];
  };
  if (o->Hm1_p) for (int q = 0; q < ny; ++q) hm1[q] = hv(o->Hm1_p, q);
  if (o->Hm2_p) for (int q = 0; q < ny + 4; ++q) hm2[q] = hv(o->Hm2_p, q);
  const size_t nhm3 = (size_t)nx * ny;
  if (!o->Hm3_p) hm3.assign(nhm3, 1.0);
  std::vector<int> spe(nb, 0), pmb(nb, 0);
  for (int b = 0; b < nb; ++b) spe[b] = o->bin_species ? o->bin_species[b] : 0;
  const int species = o->bin_species ? o->species : 0;
  // PM loads skip aerosol species (mod_nc_IO.F90:3750); a bin counts for
  // threshold p when its diameter is at most pm_um[p] micrometres
  const bool pm_ok = col_mass_pm && o->npm > 0 && o->species_category != 2;
  if (pm_ok)
    for (int b = 0; b < nb; ++b)
      for (int p = 0; p < o->npm; ++p)
        if (o->bin_diam[b] <= o->pm_um[p] * 1e-6) pmb[b] |= 1 << p;

  // device buffers: tables and outputs
  struct Out {
    double *host;
    size_t n;
    double *dev;
  } outs[8] = {{con_bins, n3 * nb, nullptr}, {con, n3, nullptr},           {con_sur, ncol, nullptr},
               {col_mass, ncol, nullptr},    {col_mass_pm, ncol * (size_t)std::max(o->npm, 1), nullptr},
               {cloud_top, ncol, nullptr},   {grn_load, ncol, nullptr},     {grn_load_bin, ncol * nb, nullptr}};
  // the column products and the cuts are formed from the corner concentration
  const bool need_con = cut || con_sur || col_mass || cloud_top || pm_ok;
  size_t bytes = 2 * DevArena::room<double>(n3) + 8 * DevArena::room<double>((size_t)nx + ny + nz + nb + 8) +
                 2 * DevArena::room<double>(nhm3) + (pm_ok ? DevArena::room<double>(n3 * (size_t)o->npm) : 0) +
                 (cut ? DevArena::room<double>(n3) : 0);
  for (auto &x : outs)
    if (x.host || (need_con && &x == &outs[1])) bytes += DevArena::room<double>(x.n);
  DevArena arena(bytes);
  auto dev = [&](size_t n) -> void * {
    char *p = nullptr;
    return arena.take(&p, n) == hipSuccess ? p : nullptr;
  };
  OutArgs a;
  memset(&a, 0, sizeof(a));
  a.chi = c->chi;
  a.clo = c->comp == FALL3D_ADS_STATE_FP32X2 ? c->clo : nullptr;
  a.c64 = c->c64;
  a.acum = c->acum;
  a.nx = nx;
  a.ny = ny;
  a.nz = nz;
  a.nb = nb;
  a.species = species;
  a.so2_du = o->so2_du;
  a.npm = o->npm;
  a.pm_ok = pm_ok ? 1 : 0;
  double *d_hm1 = (double *)dev(8 * hm1.size()), *d_hm2 = (double *)dev(8 * hm2.size());
  double *d_hm3 = (double *)dev(8 * nhm3);
  int *d_spe = (int *)dev(4 * (size_t)nb), *d_pmb = (int *)dev(4 * (size_t)nb);
  double *d_zc = o->z_c ? (double *)dev(8 * n3) : nullptr;
  // host arrays of the context kind go through raw into FP64
  char *raw = (o->z_c || o->Hm3_p) ? (char *)dev((size_t)c->kind * (o->z_c ? n3 : nhm3)) : nullptr;
  bool ok = d_hm1 && d_hm2 && d_hm3 && d_spe && d_pmb && (!o->z_c || d_zc) && (raw || (!o->z_c && !o->Hm3_p));
  for (auto &x : outs)
    if ((x.host || (need_con && &x == &outs[1])) && ok) ok = (x.dev = (double *)dev(8 * x.n)) != nullptr;
  double *d_wpm = nullptr;
  if (pm_ok && ok) ok = (d_wpm = (double *)dev(8 * n3 * (size_t)o->npm)) != nullptr;
  a.wpm = d_wpm;
  double *d_cz = nullptr, *d_zl = nullptr;
  if (cut && ok) ok = (d_cz = (double *)dev(8 * n3)) != nullptr && (d_zl = (double *)dev(8 * (size_t)(nz + 1))) != nullptr;
  if (!ok) return fail(c, FALL3D_ADS_EHIP, "postprocess: device allocation failed");
  hipError_t e = hipSuccess;
  auto up = [&](void *d, const void *h, size_t bytes) {
    if (e == hipSuccess) e = hipMemcpyAsync(d, h, bytes, hipMemcpyHostToDevice, c->stream);
  };
  up(d_hm1, hm1.data(), 8 * hm1.size());
  up(d_hm2, hm2.data(), 8 * hm2.size());
  auto up64 = [&](double *d, const void *h, size_t n) {
    if (e == hipSuccess) e = c->staging.in(raw, h, n * (size_t)c->kind, c->stream);
    if (e == hipSuccess) e = to_f64(raw, c->kind, d, n, c->stream);
  };
  if (o->Hm3_p)
    up64(d_hm3, o->Hm3_p, nhm3);
  else
    up(d_hm3, hm3.data(), 8 * nhm3);
  up(d_spe, spe.data(), 4 * (size_t)nb);
  up(d_pmb, pmb.data(), 4 * (size_t)nb);
  if (d_zc) up64(d_zc, o->z_c, n3);
  a.hm1 = d_hm1;
  a.hm2 = d_hm2;
  a.hm3 = d_hm3;
  a.spe = d_spe;
  a.pm_bin = d_pmb;
  a.zc = d_zc;
  a.con_bins = outs[0].dev;
  a.con = outs[1].dev;
  a.con_sur = outs[2].dev;
  a.col_mass = outs[3].dev;
  a.col_mass_pm = pm_ok ? outs[4].dev : nullptr;
  a.cloud_top = outs[5].dev;
  a.grn_load = outs[6].dev;
  a.grn_load_bin = outs[7].dev;
  if (e == hipSuccess) e = launch_output(a, c->stream);
  // cuts: the species' concentration on the z levels sigma X3max, then
  // linear interpolation to the cut positions (index and weight of each cut
  // from grid_get_shapez over the corner coordinates, on the host)
  std::vector<int> cidx[4];
  std::vector<double> csh[4], zl;
  if (cut && e == hipSuccess) {
    const fall3d_cut_args *ca = cut->args;
    zl.resize(nz + 1);
    for (int k = 0; k <= nz; ++k) zl[k] = ca->sigma[k] * ca->X3max;
    up(d_zl, zl.data(), 8 * zl.size());
    if (e == hipSuccess) {
      const size_t g = std::min<size_t>((ncol + 255) / 256, 65536);
      hipLaunchKernelGGL(k_zlevels, dim3((unsigned)std::max<size_t>(g, 1), (unsigned)std::min(nz + 1, 65535)), dim3(256), 0, c->stream, a.con, d_zc, d_zl,
                         nx, ny, nz, d_cz);
      e = hipGetLastError();
    }
    std::vector<double> xc(nx + 1), yc(ny + 1);
    for (int i = 0; i <= nx; ++i) xc[i] = ca->lonmin + (double)i * ca->dlon;
    for (int j = 0; j <= ny; ++j) yc[j] = ca->latmin + (double)j * ca->dlat;
    const int ncut[4] = {ca->ncutx, ca->ncuty, ca->ncutz, ca->nfl};
    const double *pos[4] = {ca->x_cut, ca->y_cut, ca->z_cut, ca->fl_cut};
    const std::vector<double> *coord[4] = {&xc, &yc, &zl, &zl};
    for (int q = 0; q < 4 && e == hipSuccess; ++q) {
      if (ncut[q] == 0) continue;
      cidx[q].resize(ncut[q]);
      csh[q].resize(ncut[q]);
      for (int m = 0; m < ncut[q]; ++m) {
        const double z = q == 3 ? pos[q][m] * 30.48 : pos[q][m];  // flight level (100 ft) -> m
        shapez(coord[q]->data(), 1, (int)coord[q]->size(), z, cidx[q][m], csh[q][m]);
      }
      const int mode = q < 2 ? q : 2;
      const size_t nout = (size_t)(mode == 0 ? ny + 1 : nx + 1) * (mode == 2 ? ny + 1 : nz + 1) * ncut[q];
      int *d_idx = (int *)dev(4 * (size_t)ncut[q]);
      double *d_sh = (double *)dev(8 * (size_t)ncut[q]), *d_out = (double *)dev(8 * nout);
      if (!d_idx || !d_sh || !d_out) {
        e = hipErrorOutOfMemory;
        break;
      }
      up(d_idx, cidx[q].data(), 4 * (size_t)ncut[q]);
      up(d_sh, csh[q].data(), 8 * (size_t)ncut[q]);
      if (e != hipSuccess) break;
      const size_t g = std::min<size_t>((nout + 255) / 256, 65536);
      hipLaunchKernelGGL(k_cuts, dim3((unsigned)std::max<size_t>(g, 1)), dim3(256), 0, c->stream, d_cz, nx, ny, nz,
                         mode, ncut[q], d_idx, d_sh, d_out);
      e = hipGetLastError();
      if (e == hipSuccess) e = c->staging.out(cut->out[q], d_out, 8 * nout, c->stream);
    }
  }
  for (auto &x : outs)
    if (x.host && e == hipSuccess) e = c->staging.out(x.host, x.dev, 8 * x.n, c->stream);
  if (e == hipSuccess) e = hipStreamSynchronize(c->stream);
  if (col_mass_pm && !pm_ok && e == hipSuccess)
    for (size_t q = 0; q < outs[4].n; ++q) col_mass_pm[q] = 0.0;
  if (e != hipSuccess) return fail(c, FALL3D_ADS_EHIP, "postprocess: %s", hipGetErrorString(e));
  return FALL3D_ADS_OK;
}

}  // namespace

extern "C" int fall3d_ads_postprocess(fall3d_ads_ctx *c, const fall3d_output_args *o, double *con_bins, double *con,
                                      double *con_sur, double *col_mass, double *col_mass_pm, double *cloud_top,
                                      double *grn_load, double *grn_load_bin) {
  return postprocess_impl(c, o, con_bins, con, con_sur, col_mass, col_mass_pm, cloud_top, grn_load, grn_load_bin,
                          nullptr);
}

extern "C" int fall3d_ads_postprocess_cuts(fall3d_ads_ctx *c, const fall3d_output_args *o,
                                           const fall3d_cut_args *cuts, double *cut_x, double *cut_y, double *cut_z,
                                           double *cut_fl) {
  const CutReq r = {cuts, {cut_x, cut_y, cut_z, cut_fl}};
  return postprocess_impl(c, o, nullptr, nullptr, nullptr, nullptr, nullptr, nullptr, nullptr, nullptr, &r);
}
