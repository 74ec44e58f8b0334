// ads_sweep_seg.hip -- y and z sweeps of small grids (Sources/mod_ADS.F90
// ADS_solve_along_y/z): lines cut into segments that run side by side.
//
// The streaming sweep gives a line to one thread, so its time is the length
// of a line however few lines there are: 64 x 64 x 32 cells of one bin are 32
// waves on 1024 SIMDs, and the y sweep takes 22 us for 0.5 MB. Here a workgroup
// owns X neighbouring columns of one transverse line, and X consecutive
// threads one segment of C cells of each column; the segments trade their
// edge cells and fluxes through LDS, two barriers per RK stage, and the bins
// of the group follow one another with the next bin's cells already loaded.
// Winds, diffusion and factors are read once for all bins (the settling
// velocity per bin). Stage values and fluxes are formed by the statements of
// the other sweeps (see ads_sweep_impl.h), so the fields are equal bit for bit.
#include "ads_sweep_impl.h"

namespace f3d {
namespace {

template <int DIR, int C, int LIM, bool COMP, int NST>
__global__ void __launch_bounds__(512) k_seg(SweepArgs a) {
  // per thread: last two and first cell of the segment, first face's flux and
  // its RK4 sum
  __shared__ float edge[5][512];
  const int X = a.TX, S = a.S, n = a.n, nx = a.nx, ny = a.ny, nz = a.nz;
  const int tid = threadIdx.x, seg = tid / X, col = tid - seg * X;
  const int tile = blockIdx.x % a.ntrans, t2 = blockIdx.x / a.ntrans + 1;  // x tile; k (y sweep) or j (z sweep)
  const int i = tile * X + col + 1;
  const bool act = seg < S && i <= nx;
  const int ia = i <= nx ? i : nx;
  const bool first = seg == 0, last = seg >= S - 1;
  const int s0 = (seg < S ? seg : 0) * C + 1;  // first cell; idle threads read the first segment's
  const int qn = n - s0;                       // local index of cell n in the last segment (-1: in the one before)
  const int lt = first ? tid : tid - X, rt = last ? tid : tid + X;

  // element offsets: position -1 of c, face 0 of the winds, position -1 of K; strides
  const size_t cbin = (size_t)state_pitch(nx) * (ny + 4) * (nz + 4);
  size_t c0, v0, k0, cs, vs;
  if constexpr (DIR == 1) {
    c0 = (size_t)(ia + 1) + (size_t)state_pitch(nx) * ((size_t)(ny + 4) * (t2 + 1));
    cs = (size_t)state_pitch(nx);
    v0 = (size_t)(ia - 1) + (size_t)nx * (ny + 3) * (t2 - 1);
    k0 = (size_t)(ia - 1) + (size_t)nx * (ny + 4) * (t2 - 1);
    vs = (size_t)nx;
  } else {
    c0 = (size_t)(ia + 1) + (size_t)state_pitch(nx) * (t2 + 1);
    cs = (size_t)state_pitch(nx) * (ny + 4);
    v0 = k0 = (size_t)(ia - 1) + (size_t)nx * (t2 - 1);
    vs = (size_t)nx * ny;
  }
  const size_t nvs = (size_t)nx * ny * (nz + 3);
  auto at = [n](int p) { return p < n + 2 ? p : n + 2; };  // cells and faces past the arrays' last feed nothing

  const float s = a.stime, s1 = 1.0f - a.stime;
  float wv[C], kf[C], hb[C], db[C], fb[C], wq[C];
  double f64[C];
  {
    float kk = a.kd[k0 + vs * (size_t)s0];  // cell s0-1
#pragma unroll
    for (int q = 0; q < C; ++q) {
      const int p = at(s0 + q);
      wv[q] = s1 * a.vel1[v0 + vs * (size_t)p] + s * a.vel2[v0 + vs * (size_t)p];
      const float kq = a.kd[k0 + vs * (size_t)(p + 1)];
      kf[q] = (kk + kq) * a.hdxp[p];
      kk = kq;
      const bool in = act && s0 + q <= n;
      db[q] = in ? a.dtib[p] : 0.0f;
      hb[q] = in ? a.hdtib[p] : 0.0f;
      fb[q] = in ? a.ftib[p] : 0.0f;
      f64[q] = (!COMP && in) ? a.ftib64[p] : 0.0;
      wq[q] = (float)a.dxb64[p];
    }
  }
  const float wbeg = s1 * a.vel1[v0 + vs] + s * a.vel2[v0 + vs];
  const float wend = s1 * a.vel1[v0 + vs * (size_t)(n + 1)] + s * a.vel2[v0 + vs * (size_t)(n + 1)];
  const double area = act ? a.areaB[t2] * a.areaA[ia] : 0.0, dt = (double)a.dt;

  double rb = 0.0, re = 0.0, lb = 0.0, le = 0.0, rr = 0.0;
  const int bfirst = blockIdx.y * a.nbin, blast = min(bfirst + a.nbin, a.nbins);
  float nxt[C], nlo[C], nvv[C], nvb = 0.0f, nve = 0.0f;  // the next bin's cells and settling velocities
  auto fetch = [&](int b) {
#pragma unroll
    for (int q = 0; q < C; ++q) {
      const int p = at(s0 + q);
      nxt[q] = a.chi[c0 + cbin * (size_t)b + cs * (size_t)(p + 1)];
      if constexpr (COMP) nlo[q] = a.clo[c0 + cbin * (size_t)b + cs * (size_t)(p + 1)];
      if constexpr (DIR == 2) nvv[q] = a.vs[v0 + nvs * (size_t)b + vs * (size_t)p];
    }
    if constexpr (DIR == 2) {
      nvb = a.vs[v0 + nvs * (size_t)b + vs];
      nve = a.vs[v0 + nvs * (size_t)b + vs * (size_t)(n + 1)];
    }
  };
  fetch(bfirst);
  for (int b = bfirst; b < blast; ++b) {
    float *hi = a.chi + c0 + cbin * (size_t)b + cs;  // hi[cs * p]: cell p
    float *low = COMP ? a.clo + c0 + cbin * (size_t)b + cs : nullptr;
    float cn[C], lo[C], up[C], um[C];
    float vbeg = wbeg, vend = wend;
#pragma unroll
    for (int q = 0; q < C; ++q) {
      cn[q] = nxt[q];
      lo[q] = COMP ? nlo[q] : 0.0f;
      float v = wv[q];
      if constexpr (DIR == 2) v -= nvv[q];
      up[q] = fmaxf(v, 0.0f);
      um[q] = fminf(v, 0.0f);
    }
    if constexpr (DIR == 2) {
      vbeg -= nvb;
      vend -= nve;
    }
    if (b + 1 < blast) fetch(b + 1);
    // free-flow ghosts (Sources/mod_ADS.F90:1239-1324), frozen for the sweep;
    // cell n is in the last segment, or the last cell of the one before
    edge[1][tid] = cn[C - 1];
    __syncthreads();
    const float cleft = edge[1][lt];
    float gL = 0.0f, gR = 0.0f;
    if (first) gL = (a.bc == 0 ? (vbeg > 0.0f) : (a.bc == 1)) ? (2.0f * 0.0f - cn[0]) : cn[0];
    if (last) {
      float cl = (qn < 0) ? cleft : cn[0];
#pragma unroll
      for (int q = 1; q < C; ++q) cl = (q == qn) ? cn[q] : cl;
      gR = (a.bc == 0 ? (vend < 0.0f) : (a.bc == 1)) ? (2.0f * 0.0f - cl) : cl;
#pragma unroll
      for (int q = 0; q < C; ++q) {
        cn[q] = (q > qn) ? gR : cn[q];
        lo[q] = (q > qn) ? 0.0f : lo[q];  // ghost low words are 0
      }
    }
    if (act && first) {
      hi[0] = gL;
      *(hi - cs) = gL;
      if constexpr (COMP) low[0] = *(low - cs) = 0.0f;
    }
    if (act && last) {
      hi[cs * (size_t)(n + 1)] = gR;
      hi[cs * (size_t)(n + 2)] = gR;
      if constexpr (COMP) low[cs * (size_t)(n + 1)] = low[cs * (size_t)(n + 2)] = 0.0f;
    }

    float y[C], gh[C + 1];
#pragma unroll
    for (int q = 0; q < C; ++q) y[q] = cn[q];
#pragma unroll
    for (int q = 0; q <= C; ++q) gh[q] = 0.0f;
    float RFb = 0.0f, RFe = 0.0f;
    __syncthreads();  // the last cells above have been read
#pragma unroll
    for (int st = 0; st < NST; ++st) {
      const bool last_stage = (st == NST - 1);
      edge[0][tid] = y[C - 2];
      edge[1][tid] = y[C - 1];
      edge[2][tid] = y[0];
      __syncthreads();
      float w[C + 3];
      w[0] = first ? gL : edge[0][lt];
      w[1] = first ? gL : edge[1][lt];
#pragma unroll
      for (int q = 0; q < C; ++q) w[q + 2] = y[q];
      w[C + 2] = last ? gR : edge[2][rt];
      float d_cur = w[2] - w[1];
      float m_prev = limiter_slope<LIM>(w[1] - w[0], d_cur);
      float G_prev = 0.0f;
#pragma unroll
      for (int q = 0; q < C; ++q) {
        const float d_next = w[q + 3] - w[q + 2];
        const float m_cur = limiter_slope<LIM>(d_cur, d_next);
        const float cL = fmaf(0.5f, m_prev, w[q + 1]);
        const float cR = fmaf(-0.5f, m_cur, w[q + 2]);
        // G = F - P with F = max(u,0) cL + min(u,0) cR
        const float P = kf[q] * d_cur;
        const float G = fmaf(up[q], cL, fmaf(um[q], cR, -P));
        if (last_stage) {  // reference boundary fluxes F + P
          if (q == 0) RFb = fmaf(2.0f, P, G);
          if (q == qn + 1) RFe = fmaf(2.0f, P, G);
        }
        // RK4 weights 1 2 2 1 (the 1/6 is in the final factor)
        if (st == 0)
          gh[q] = G;
        else if (last_stage)
          gh[q] = gh[q] + G;
        else
          gh[q] = fmaf(2.0f, G, gh[q]);
        if (q == 0) {
          edge[3][tid] = G;
          if (last_stage) edge[4][tid] = gh[0];
        } else if (!last_stage) {
          y[q - 1] = fmaf((st == 2) ? db[q - 1] : hb[q - 1], G_prev - G, cn[q - 1]);
        }
        G_prev = G;
        d_cur = d_next;
        m_prev = m_cur;
      }
      // Face C is the right neighbour's face 0; past the last segment it only
      // feeds frozen ghost positions (zero factors)
      __syncthreads();
      if (!last_stage) y[C - 1] = fmaf((st == 2) ? db[C - 1] : hb[C - 1], G_prev - edge[3][rt], cn[C - 1]);
    }
    gh[C] = edge[4][rt];

    // final update of cells up to n
    float tl0 = 0.0f, trn = 0.0f, res = 0.0f;
    double fl0 = 1.0, fln = 1.0;
#pragma unroll
    for (int q = 0; q < C; ++q) {
      float hv, lv = 0.0f;
      if constexpr (COMP) {
        const float tl = fb[q] * gh[q], tr = fb[q] * gh[q + 1];
        if (q == 0) tl0 = tl;
        if (q == qn) trn = tr;
        hv = cn[q];
        lv = lo[q];
        comp_add(hv, lv, tl);
        comp_add(hv, lv, -tr);
      } else {
        if (q == 0) {
          tl0 = gh[0];
          fl0 = f64[0];
        }
        if (q == qn) {
          trn = gh[q + 1];
          fln = f64[q];
        }
        hv = final_update_fp64(cn[q], gh[q], gh[q + 1], f64[q], wq[q], res);
      }
      if (act && q <= qn) {
        hi[cs * (size_t)(s0 + q)] = hv;
        if constexpr (COMP) low[cs * (size_t)(s0 + q)] = lv;
      }
    }
    if (act) {
      if (first) {
        rb += (double)RFb * area * dt;
        lb -= (double)tl0 * fl0 * a.dxb64[1] * area;
        if constexpr (DIR == 2) {
          const size_t ai = (size_t)(i + 1) + (size_t)(nx + 4) * ((size_t)(t2 + 1) + (size_t)(ny + 4) * b);
          a.acum[ai] = a.acum[ai] + fabs((double)RFb) * dt;
        }
      }
      if (qn >= -1 && qn <= C - 2) re += (double)RFe * area * dt;      // holds face n+1
      if (qn >= 0 && qn <= C - 1) le += (double)trn * fln * a.dxb64[n] * area;  // holds cell n
      rr += (double)res * area;
    }
  }
  block_partials5(rb, re, lb, le, rr, a.partials, a.rpartials, (size_t)blockIdx.y * gridDim.x + blockIdx.x);
}

template <int DIR, int C>
hipError_t launch(int limiter, bool comp, int nst, const SweepArgs &a, dim3 grid, dim3 block, hipStream_t st) {
#define F3D_SEG(L, CP, N)                                                            \
  if (limiter == L && comp == CP && nst == N) {                                      \
    hipLaunchKernelGGL((k_seg<DIR, C, L, CP, N>), grid, block, 0, st, a);            \
    return hipGetLastError();                                                        \
  }
  F3D_SEG(1, false, 4) F3D_SEG(2, false, 4) F3D_SEG(3, false, 4) F3D_SEG(1, true, 4) F3D_SEG(2, true, 4)
  F3D_SEG(3, true, 4) F3D_SEG(1, false, 1) F3D_SEG(2, false, 1) F3D_SEG(3, false, 1) F3D_SEG(1, true, 1)
  F3D_SEG(2, true, 1) F3D_SEG(3, true, 1)
#undef F3D_SEG
  return hipErrorInvalidValue;
}

}  // namespace

hipError_t launch_sweep_seg(int dir, int cells, int limiter, bool comp, int nst, const SweepArgs &a, dim3 grid, dim3 block,
                            hipStream_t st) {
  (void)hipGetLastError();
  if (block.x > 512 || a.S * a.TX > (int)block.x) return hipErrorInvalidValue;
  if (cells == 4) return dir == 1 ? launch<1, 4>(limiter, comp, nst, a, grid, block, st) : launch<2, 4>(limiter, comp, nst, a, grid, block, st);
  if (cells == 8) return dir == 1 ? launch<1, 8>(limiter, comp, nst, a, grid, block, st) : launch<2, 8>(limiter, comp, nst, a, grid, block, st);
  return hipErrorInvalidValue;
}

}  // namespace f3d
