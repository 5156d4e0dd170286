// pb_sph.hip -- SPH Navier-Stokes path of cudaParticleSPH_NS on MI355X.
//
// Reference path (cudaParticleSPH_NS.cu:71-207, kerneltemplate.hh:636-709,
// kernelinline.hh:173-215): per step a cell sort, a (cell x 27) density
// kernel writing 81 partials per particle, a 27-way reduction and two
// element-wise passes (1/rho, mu), then the same for the acceleration.
//
// Here: after pb_bin (the counting sort of the reference cell grid) the
// particles are gathered into cell order once per call (positions with the
// mass in w, velocities, per-particle material terms); one kernel computes
// the number density, rho, 1/rho and the field mu in a single pass over
// the 27 cells, and one kernel computes the acceleration.  Both test FP32
// views of the candidates, staged in LDS column by column (neighbour cells of a
// column are one contiguous range), evaluate what passes in FP64 and write
// straight to the particle's storage slot: no partial buffers, no reductions.
// Distances are non-periodic (distance2, kernelinline.hh:19-29); the density sum includes the particle itself, the
// acceleration sum excludes it; rho0 = 1 (cudaParticleSPH_NS.cu:91).
//
// The same calls also run the dam-break workload's config physics, which the
// reference's kernels do not hold (weakly compressible SPH): the M4 cubic
// spline of support 2h, summation density, the Tait equation of state
// clamped at pmin, and Monaghan's artificial viscosity; selected by
// pb_sph_set_wcsph, with the same gathered views, cell grid and launches.
#include "pb_internal.h"
#include <cmath>

struct SphGrid {
  uint32_t nb[3];
  float len[3], lo[3];
};

struct SphArgs {
  const uint32_t *perm;      // sorted slot -> storage slot
  const uint32_t *bid;       // sorted slot -> cell
  const uint32_t *cstart;    // cell -> first sorted slot (cstart[c+1] ends it)
  const float4 *fq;          // sorted filter view (sph_view)
  const double4 *rs;         // sorted (x, y, z, m)
  const double4 *vs;         // acceleration: sorted (vx, vy, vz, 1/rho; rho under the config physics)
  const double2 *ds;         // acceleration: sorted (P, mu); (p/rho^2, 0) under the config physics
  const double *mus;         // density: sorted mu0
  SphGrid g;
  uint32_t n;
  double h, w0, w1, rho0;
  // config physics: support^2, 1/h, 1/(pi h^3), 1/(pi h^5), Tait B, 1/rho0,
  // gamma, pmin, alpha c0 h, 0.01 h^2
  double sup2, hinv, ws, wf, B, rho0inv, gamma, pmin, avh, eh2;
};

// FP32 filter: the bound on |r_ij|^2 with the rounding margin, and the ranges of
// the coordinates that the margin covers
struct SphFilter {
  float r2, l2, zmax;
};

// Filter view of a particle of cell c: x and y from the middle of its cell
// column, z from the grid's edge, and x^2 + y^2; a particle beyond the margin's
// ranges (outside the grid, binned into its edge cells; NaN) passes every test.
__device__ __forceinline__ float4 sph_view(const SphGrid &g, const SphFilter &FB, uint32_t c,
                                           const double4 &p) {
  const uint32_t col = c / g.nb[2], i = col / g.nb[1], j = col % g.nb[1];
  const float x = (float)(p.x - ((double)g.lo[0] + ((double)i + 0.5) * (double)g.len[0]));
  const float y = (float)(p.y - ((double)g.lo[1] + ((double)j + 0.5) * (double)g.len[1]));
  const float z = (float)(p.z - (double)g.lo[2]);
  const float w = x * x + y * y;
  return w <= FB.l2 && fabsf(z) <= FB.zmax ? make_float4(x, y, z, w)
                                           : make_float4(0.f, 0.f, 0.f, -INFINITY);
}

// positions (mass in w), the filter view and mu0 in cell order (density call)
__global__ void k_sph_gather(const uint32_t *perm, const uint32_t *bid, const double4 *r,
                             const double4 *v, const double *mu0, SphGrid g, SphFilter FB,
                             uint32_t n, double4 *rs, float4 *fq, double *mus) {
  const uint32_t k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= n) return;
  const uint32_t s = perm[k];
  const double4 p = r[s];
  rs[k] = make_double4(p.x, p.y, p.z, 1.0 / v[s].w);
  fq[k] = sph_view(g, FB, bid[k], p);
  if (mu0) mus[k] = mu0[s];
}

// Acceleration call: positions, velocities and the per-particle terms of the
// last density call, read from the storage-order outputs, so a pb_bin
// between the two calls is harmless.  Reference physics: 1/rho, and ds =
// (c2/rho (1 - rho0/rho), mu); config physics: rho, and ds = (p/rho^2, -).
__global__ void k_sph_gather_acc(const uint32_t *perm, const uint32_t *bid, const double4 *r,
                                 const double4 *v, const double4 *num, const double *rhoinv,
                                 const double *c2, double rho0, int wc, SphGrid g, SphFilter FB,
                                 uint32_t n, double4 *rs, float4 *fq, double4 *vs, double2 *ds) {
  const uint32_t k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= n) return;
  const uint32_t s = perm[k];
  const double4 p = r[s], u = v[s], d = num[s];
  const double ri = rhoinv[s];
  rs[k] = make_double4(p.x, p.y, p.z, 1.0 / u.w);
  fq[k] = sph_view(g, FB, bid[k], p);
  vs[k] = make_double4(u.x, u.y, u.z, wc ? d.y : ri);
  ds[k] = wc ? make_double2(d.z * ri * ri, 0.0)
             : make_double2(c2[s] * ri * (1.0 - rho0 * ri), d.z);
}

// ---------------------------------------------------------------------------
// Pair kernels.  LN lanes per sorted slot, 64 / LN consecutive slots a wavefront.
// In each of the 9 neighbour columns the cells z-1 .. z+1 of a slot are one
// contiguous sorted range (its window), and the windows of a wavefront's slots
// overlap: their union is staged into LDS, SC_CAP filter views at a time (loaded
// while the column before is tested), and each lane scans its share of its own
// window, every LN-th candidate:
//   * a conservative FP32 filter, up to 32 candidates into a bit mask:
//     |ri - rj|^2 < r2max plus a margin that covers the FP32 rounding, from
//     coordinates relative to the candidates' column (6 instructions a test);
//   * the hits are appended to the lane's list in LDS, and the lists are worked
//     off together when one of them is full and at the end, so that lanes wait
//     for the largest number of hits of all columns instead of the largest of
//     each (Lucy, h = 1.7 dx: 21 in place of 36 a wavefront for 20 a particle);
//   * the FP64 pair body on the cell-order views, which applies the exact
//     support test itself (so the margin changes nothing).
// A wavefront whose slots lie thinly (a floor, a splash) can span many dense
// neighbour columns of which it needs little: past SC_DIRECT candidates the lanes
// read their windows from memory.  Such wavefronts, one in a hundred, took up
// to eight times the others' time and were the kernel's end (796,176 particles:
// 97 us with this, 114 without).
// Bound by vector instructions (about 60 % of the time) and by the latency of
// the loads between them.  Density and acceleration of 796,176 particles, Lucy,
// 20 pairs each: 202 and 270 us with a workgroup a column segment (wavefronts
// two thirds full, two barriers a column), now 95 and 134 us; 133,904 of the
// config physics, 66 pairs: 99 and 174, now 56 and 78 us.
// A slot's pairs are visited in the order of a 27-cell loop (neighbour columns in
// (a, b) order, slots ascending), each lane its share of them; the lanes' sums
// are added in a fixed order.
constexpr uint32_t SC_T = 64;       // a wavefront is a workgroup: none waits for another's end
constexpr uint32_t SC_CAP = 128;    // candidates staged at a time
constexpr uint32_t SC_DIRECT = 256; // longer unions are read directly
constexpr uint32_t SC_HITS = 20;    // hits a lane keeps
constexpr uint32_t SC_W = 2;        // hits worked off at a time
constexpr uint32_t SC_G = 8;        // tests at a time

enum { SPH_LUCY_DENS = 0, SPH_LUCY_ACC = 1, SPH_WC_DENS = 2, SPH_WC_ACC = 3 };

// 1/sqrt(x), x > 0: the hardware estimate and two Newton steps (about one
// ulp); and 1/x the same way
__device__ __forceinline__ double sph_rsqrt(double x) {
  double y = __builtin_amdgcn_rsq(x);
  const double hx = 0.5 * x;
  y = y * fma(-hx * y, y, 1.5);
  y = y * fma(-hx * y, y, 1.5);
  return y;
}
__device__ __forceinline__ double sph_rcp(double x) {
  double y = __builtin_amdgcn_rcp(x);
  y = fma(y, fma(-x, y, 1.0), y);
  y = fma(y, fma(-x, y, 1.0), y);
  return y;
}
// Tait pressure max(B ((rho/rho0)^gamma - 1), pmin); out of line, once per
// particle, so pow's registers do not weigh on the pair loop
__device__ __attribute__((noinline)) double sph_tait(double rho, double rho0inv, double gamma,
                                                     double B, double pmin) {
  return fmax(B * (pow(rho * rho0inv, gamma) - 1.0), pmin);
}

// |r| from r^2 (0 at 0)
__device__ __forceinline__ double sph_norm(double r2, double *rinv) {
  const double y = r2 > 0.0 ? sph_rsqrt(r2) : 0.0;
  *rinv = y;
  return r2 * y;
}

// the fields of a particle that pass M reads
struct SphBody {
  double4 p, v;
  double2 d;
  double mu;
};
template <int M>
__device__ __forceinline__ SphBody sph_load(const SphArgs &A, uint32_t q) {
  SphBody B;
  B.p = A.rs[q];
  if constexpr (M == SPH_LUCY_DENS) B.mu = A.mus[q];
  if constexpr (M == SPH_LUCY_ACC || M == SPH_WC_ACC) {
    B.v = A.vs[q];
    B.d = A.ds[q];
  }
  return B;
}

// one pair; self: the particle with itself
template <int M>
__device__ __forceinline__ void sph_pair(const SphArgs &A, const SphBody &I, const SphBody &J,
                                         bool self, double &acc0, double &acc1, double &acc2) {
  const double4 &pi = I.p, &vi = I.v, &pj = J.p, &vj = J.v;
  if constexpr (M == SPH_LUCY_DENS) {
    // SPHcalcDensity<SPHKernelLucy> (kerneltemplate.hh:636-656):
    // W = w0 (h + 3R)(h - R)^3, 0 beyond h (kernelinline.hh:182-188)
    const double dx = pi.x - pj.x, dy = pi.y - pj.y, dz = pi.z - pj.z;
    double ri;
    const double R = sph_norm(dx * dx + dy * dy + dz * dz, &ri);
    const double tt = fmax(A.h - R, 0.0);
    const double W = A.w0 * (A.h + 3.0 * R) * (tt * tt * tt);
    const double mW = pj.w * W;
    acc0 += W;
    acc1 += mW;
    acc2 = fma(J.mu, mW, acc2);
  } else if constexpr (M == SPH_LUCY_ACC) {
    // SPHNavierStokes<SPHKernelLucyDW> (kerneltemplate.hh:666-709)
    const double dx = pj.x - pi.x, dy = pj.y - pi.y, dz = pj.z - pi.z;
    double ri;
    const double R = sph_norm(dx * dx + dy * dy + dz * dz, &ri);
    const double tt = A.h - R;
    if (tt > 0.0 && !self) {                    // no self term, 0 beyond h
      const double mw = pj.w * (A.w1 * tt * tt);  // m_j (dW/dr)/r, kernelinline.hh:209-214
      const double p1 = I.d.x + J.d.x;
      const double v1 = (I.d.y + J.d.y) * vi.w * vj.w;
      acc0 += mw * (dx * p1 - (vj.x - vi.x) * v1);
      acc1 += mw * (dy * p1 - (vj.y - vi.y) * v1);
      acc2 += mw * (dz * p1 - (vj.z - vi.z) * v1);
    }
  } else if constexpr (M == SPH_WC_DENS) {
    // M4 spline inside the support: W = ws (t2^3/4 - t1^3),
    // t1 = max(1 - q, 0), t2 = 2 - q, q = r/h
    const double dx = pi.x - pj.x, dy = pi.y - pj.y, dz = pi.z - pj.z;
    const double R2 = dx * dx + dy * dy + dz * dz;
    if (R2 < A.sup2) {
      double ri;
      const double qq = sph_norm(R2, &ri) * A.hinv;
      const double t1 = fmax(1.0 - qq, 0.0), t2 = 2.0 - qq;
      const double W = 0.25 * (t2 * t2 * t2) - t1 * t1 * t1;
      acc0 += W;
      acc1 = fma(pj.w, W, acc1);
    }
  } else {
    // a_i = -sum m_j (P_i + P_j + Pi_ij) F(r) r_ij, F = (dW/dr)/r
    // = wf (-3 + 9/4 q) for q < 1, wf (-3/4 (2 - q)^2 / q) below 2;
    // Pi_ij = -alpha c0 h (v_ij . r_ij) / ((r^2 + 0.01 h^2) rho_bar)
    // for approaching pairs
    const double dx = pi.x - pj.x, dy = pi.y - pj.y, dz = pi.z - pj.z;
    const double R2 = dx * dx + dy * dy + dz * dz;
    if (R2 < A.sup2 && !self) {
      double ri;
      const double qq = sph_norm(R2, &ri) * A.hinv, t2 = 2.0 - qq;
      const double g = qq < 1.0 ? fma(2.25, qq, -3.0) : -0.75 * t2 * t2 * (A.h * ri);
      const double vr = (vi.x - vj.x) * dx + (vi.y - vj.y) * dy + (vi.z - vj.z) * dz;
      const double visc =
          vr < 0.0 ? -A.avh * vr * sph_rcp((R2 + A.eh2) * (0.5 * (vi.w + vj.w))) : 0.0;
      const double f = -pj.w * (I.d.x + J.d.x + visc) * g;
      acc0 = fma(f, dx, acc0);
      acc1 = fma(f, dy, acc1);
      acc2 = fma(f, dz, acc2);
    }
  }
}

template <int M, uint32_t LN>
__device__ __forceinline__ void sph_pairs(const SphArgs &A, SphFilter FB, double4 *out4,
                                          double *out1) {
  static_assert(SC_T == PB_WAVE, "the lists and the stage are a wavefront's own");
  __shared__ float4 F[SC_CAP + SC_G * LN];       // spare for a window's last tests
  __shared__ uint32_t Hs[SC_HITS][SC_T];
  const uint32_t lane = threadIdx.x;
  // consecutive workgroups share neighbour columns in an XCD's L2
  const uint32_t blk = pb_xcd_chunk<64>();
  const uint32_t k = blk * (SC_T / LN) + lane / LN, sl = lane % LN;
  const bool act = k < A.n;
  const uint32_t kk = act ? k : A.n - 1u;
  const uint32_t nz = A.g.nb[2], ny = A.g.nb[1], nx = A.g.nb[0];
  const uint32_t c = A.bid[kk], col = c / nz, z = c % nz, ci = col / ny, cj = col % ny;
  const uint32_t klo = z > 0 ? z - 1 : 0, khi = z + 1 < nz ? z + 1 : z;
  const SphBody I = sph_load<M>(A, kk);
  const float4 fi = A.fq[kk];
  double acc0 = 0.0, acc1 = 0.0, acc2 = 0.0;
  uint32_t cnt = 0;
  auto work_off = [&]() {
    for (uint32_t e = 0; e < cnt; e += SC_W) {
      SphBody J[SC_W];
      uint32_t q[SC_W];
#pragma unroll
      for (uint32_t u = 0; u < SC_W; ++u) q[u] = Hs[e + u < cnt ? e + u : e][lane];
#pragma unroll
      for (uint32_t u = 0; u < SC_W; ++u) J[u] = sph_load<M>(A, q[u]);
#pragma unroll
      for (uint32_t u = 0; u < SC_W; ++u)
        if (e + u < cnt) sph_pair<M>(A, I, J[u], q[u] == k, acc0, acc1, acc2);
    }
    cnt = 0;
    // no load of a skipped pair stays open: its registers would hold up every
    // later use of them behind the prefetches (vmcnt(0))
    __builtin_amdgcn_s_waitcnt(0x0f70);
  };
  // the lane's window in column t (false: none)
  auto window = [&](int t, uint32_t &w0, uint32_t &w1) {
    const int a = t / 3 - 1, b = t % 3 - 1;
    const bool in = act && t < 9 && (a >= 0 || ci > 0) && (a <= 0 || ci + 1 < nx) &&
                    (b >= 0 || cj > 0) && (b <= 0 || cj + 1 < ny);
    w0 = w1 = 0;
    if (in) {
      const uint32_t cb = (col + (uint32_t)(a * (int)ny + b)) * nz;
      w0 = A.cstart[cb + klo];
      w1 = A.cstart[cb + khi + 1];
    }
    return in;
  };
  // the union of the windows, which ascend with the slots
  auto span = [&](bool in, uint32_t w0, uint32_t w1, uint32_t &r0, uint32_t &r1) {
    const uint64_t any = __ballot(in);
    r0 = r1 = 0;
    if (any) {
      r0 = (uint32_t)__builtin_amdgcn_readlane((int)w0, __builtin_ctzll(any));
      r1 = (uint32_t)__builtin_amdgcn_readlane((int)w1, 63 - __builtin_clzll(any));
    }
  };
  static_assert(SC_CAP == 2 * PB_WAVE, "a batch is two views a lane");
  float4 stage0, stage1;                         // a batch on its way to LDS
  auto fetch = [&](uint32_t b0) {
    stage0 = A.fq[min(b0 + lane, A.n - 1u)];
    stage1 = A.fq[min(b0 + PB_WAVE + lane, A.n - 1u)];
  };
  uint32_t w0, w1, r0, r1, nw0, nw1;
  span(window(0, w0, w1), w0, w1, r0, r1);
  fetch(r0);
  bool nin = window(1, nw0, nw1);
#pragma unroll 1
  for (int t = 0; t < 9; ++t) {
    // the lane against this column: -2 ri and the bound less |ri|^2
    const int a = t / 3 - 1, b = t % 3 - 1;
    const float x = fi.x - (float)a * A.g.len[0], y = fi.y - (float)b * A.g.len[1];
    const bool far = fi.w < 0.f;
    const float fx = far ? 0.f : -2.0f * x, fy = far ? 0.f : -2.0f * y, fz = fi.z;
    const float lim = far ? INFINITY : FB.r2 - (x * x + y * y);
    uint32_t nr0 = 0, nr1 = 0;
    const bool direct = r1 - r0 > SC_DIRECT;
#pragma unroll 1
    for (uint32_t b0 = r0;;) {
      const uint32_t b1 = b0 + SC_CAP < r1 && !direct ? b0 + SC_CAP : r1;
      pb_wave_lds_sync();                        // the previous batch is consumed
      F[lane] = stage0;
      F[PB_WAVE + lane] = stage1;
      pb_wave_lds_sync();
      const bool last = b1 >= r1;
      if (last) span(nin, nw0, nw1, nr0, nr1);
      fetch(last ? nr0 : b1);
      // the lane's candidates: every LN-th of the window
      uint32_t q0 = w0 + sl;
      if (q0 < b0) q0 += (b0 - q0 + LN - 1u) / LN * LN;
      const uint32_t q1 = w1 < b1 ? w1 : b1;
#pragma unroll 1
      while (__any(q0 < q1)) {
        const uint32_t len = q0 < q1 ? min((q1 - q0 + LN - 1u) / LN, 32u) : 0u;
        // first test in the highest bit; tests past the window are cut off
        uint32_t mask = 0, done = 0;
        auto tests = [&](const float4 (&f)[SC_G]) {
#pragma unroll
          for (uint32_t u = 0; u < SC_G; ++u) {
            const float dz = f[u].z - fz;
            const float d = fmaf(dz, dz, fmaf(fx, f[u].x, fmaf(fy, f[u].y, f[u].w - lim)));
            mask = __builtin_amdgcn_alignbit(mask, __float_as_uint(d), 31);
          }
        };
        if (!direct) {
          const float4 *f0 = F + (q0 < q1 ? q0 - b0 : 0u);
#pragma unroll 1
          for (; done < len; done += SC_G) {
            float4 f[SC_G];
#pragma unroll
            for (uint32_t u = 0; u < SC_G; ++u) f[u] = f0[(done + u) * LN];
            tests(f);
          }
        } else {
#pragma unroll 1
          for (; done < len; done += SC_G) {
            float4 f[SC_G];
#pragma unroll
            for (uint32_t u = 0; u < SC_G; ++u) f[u] = A.fq[min(q0 + (done + u) * LN, A.n - 1u)];
            tests(f);
          }
        }
        mask = len ? (mask << (32u - done)) & (~0u << (32u - len)) : 0u;
        for (;;) {
          while (mask && cnt < SC_HITS) {
            const uint32_t u = (uint32_t)__builtin_clz(mask);
            mask &= ~(0x80000000u >> u);
            Hs[cnt++][lane] = q0 + u * LN;
          }
          if (!__any(mask)) break;
          work_off();
        }
        q0 += 32u * LN;
      }
      if (last) break;
      b0 = b1;
    }
    w0 = nw0;
    w1 = nw1;
    r0 = nr0;
    r1 = nr1;
    nin = window(t + 2, nw0, nw1);
  }
  work_off();
#pragma unroll
  for (uint32_t o = 1; o < LN; o <<= 1) {
    acc0 += __shfl_xor(acc0, (int)o, 64);
    acc1 += __shfl_xor(acc1, (int)o, 64);
    acc2 += __shfl_xor(acc2, (int)o, 64);
  }
  if (act && sl == 0) {
    const uint32_t s = A.perm[k];
    if constexpr (M == SPH_LUCY_DENS) {
      // calcDensityPost (cudaParticleSPH_NS.cu:184-207)
      const double ri = 1.0 / acc1;
      out4[s] = make_double4(acc0, acc1, acc2 * ri, 0.0);
      out1[s] = ri;
    } else if constexpr (M == SPH_WC_DENS) {
      // Tait: p = max(B ((rho/rho0)^gamma - 1), pmin)
      const double n0 = acc0 * A.ws, rho = acc1 * A.ws;
      const double p = sph_tait(rho, A.rho0inv, A.gamma, A.B, A.pmin);
      out4[s] = make_double4(n0, rho, p, 0.0);
      out1[s] = 1.0 / rho;
    } else if constexpr (M == SPH_LUCY_ACC) {
      out4[s] = make_double4(acc0, acc1, acc2, 0.0);
    } else {
      out4[s] = make_double4(acc0 * A.wf, acc1 * A.wf, acc2 * A.wf, 0.0);
    }
  }
}

template <int M, uint32_t LN>
__global__ void __launch_bounds__(SC_T) k_sph_pairs(SphArgs A, SphFilter FB, double4 *out4,
                                                    double *out1) {
  sph_pairs<M, LN>(A, FB, out4, out1);
}

// inspectDense_x (kernelfuncs.cu:772-801): per-wave partial sums of the
// number density and the count of movable particles
__global__ void k_sph_inspect(const double4 *num, const uint8_t *move, const uint32_t *orig,
                              uint32_t n, double *partials) {
  const uint32_t s = blockIdx.x * blockDim.x + threadIdx.x;
  double x = 0.0, c = 0.0;
  if (s < n && orig[s] != PB_NONE && move[s] > 0) {
    x = num[s].x;
    c = 1.0;
  }
  x = pb_wave_sum(x);
  c = pb_wave_sum(c);
  if (pb_lane() == 0 && s < n) {
    partials[4 * (s / PB_WAVE)] = x;
    partials[4 * (s / PB_WAVE) + 1] = c;
  }
}

// ------------------------------------------------------------------ host
static int sph_ready(pb_sys *s) {
  if (!s->sph_set) return pb_fail(s->ctx, PB_ERR_STATE, "SPH properties not set");
  if (!s->ref_binned) return pb_fail(s->ctx, PB_ERR_STATE, "SPH: pb_bin (calcBlockID) first");
  if (s->ref_periodic) return pb_fail(s->ctx, PB_ERR_CELLS, "SPH: cells must be non-periodic");
  const float hf = (float)(s->sph_kind == 1 ? 2.0 * s->sph_h : s->sph_h);
  if (s->blocklen[0] < hf || s->blocklen[1] < hf || s->blocklen[2] < hf)
    return pb_fail(s->ctx, PB_ERR_CELLS, "SPH: cell length below the kernel support");
  return PB_OK;
}

static SphArgs sph_args(pb_sys *s) {
  SphArgs A;
  A.perm = s->perm;
  A.bid = s->ref_bid;
  A.cstart = s->cstart;
  A.fq = s->sph_fq;
  A.rs = s->sph_rs;
  A.vs = s->sph_vs;
  A.ds = s->sph_ds;
  A.mus = s->sph_mus;
  for (int a = 0; a < 3; ++a) {
    A.g.nb[a] = s->blocknum[a];
    A.g.len[a] = s->blocklen[a];
    A.g.lo[a] = s->blocklen[a + 3];
  }
  A.n = s->n;
  A.h = s->sph_h;
  A.w0 = 105.0 / (16.0 * M_PI * std::pow(s->sph_h, 7));   // cudaParticleSPHBase.cu:121
  A.w1 = -12.0 * A.w0;
  A.rho0 = s->sph_rho0;
  const double h = s->sph_h;
  A.sup2 = 4.0 * h * h;
  A.hinv = 1.0 / h;
  A.ws = 1.0 / (M_PI * h * h * h);
  A.wf = A.ws / (h * h);
  A.B = s->sph_rho0 * s->sph_c0 * s->sph_c0 / s->sph_gamma;
  A.rho0inv = 1.0 / s->sph_rho0;
  A.gamma = s->sph_gamma;
  A.pmin = s->sph_pmin;
  A.avh = s->sph_alpha * s->sph_c0 * h;
  A.eh2 = 0.01 * h * h;
  return A;
}

// FP32 filter bound: r2max and what rounding can add.  With (cx, cy) the cell
// lengths, x^2 + y^2 of a candidate from its column's middle is at most cx^2 +
// cy^2 = L2/4 (l2) and that of a lane, up to a column away, at most L2; the
// expanded form then errs by at most ten units of 2^-24 L2 and its inputs'
// rounding by as much again.  z within [-cz, zmax] is rounded twice and
// subtracted: e = 3 units of 2^-24 zmax on |dz| <= sqrt(r2max).  Where the squares
// leave the FP32 range every pair is left to the exact test.
static SphFilter sph_filter(pb_sys *s, double r2max) {
  const double cx = s->blocklen[0], cy = s->blocklen[1], cz = s->blocklen[2];
  const double L2 = 4.0 * (cx * cx + cy * cy), zmax = (s->blocknum[2] + 1.0) * cz;
  const double e = 3.0 * 6e-8 * zmax;
  SphFilter F;
  F.r2 = (float)(r2max * (1.0 + 1e-6) + 4e-6 * L2 + 2.0 * std::sqrt(r2max) * e + e * e);
  F.l2 = L2 + zmax * zmax < 1e30 && r2max > 1e-30 ? (float)(0.25 * L2) : -1.f;
  F.zmax = (float)zmax;
  return F;
}

// Lanes a slot: as many as fill the chip's 1024 SIMDs several times over; more only
// repeat the staging.  Density + acceleration, gathers included, us with 1, 2, 4
// and 8 lanes:
//   Lucy (14 candidates a window):  15,876: 55, 41, 33, 33;  48,148: 61, 47, 46, 65;
//     133,904: 82, 83, 95, 135;  796,176: 279, 301, 402, 664
//   config (34 a window, support 2h):  7,036: 162, 79, 50, 38;  48,148: 184, 97, 70, 84;
//     133,904: 214, 147, 153, 183;  796,176: 700, 630, 705, 920
static uint32_t sph_lanes(const pb_sys *s) {
  const bool wc = s->sph_kind == 1;
  if (s->n <= 24576u) return 8u;
  if (s->n <= (wc ? 98304u : 49152u)) return 4u;
  return wc || s->n <= 131072u ? 2u : 1u;
}

template <int M>
static void sph_launch_pairs(pb_sys *s, const SphArgs &A, const SphFilter &FB, double4 *out4,
                             double *out1) {
  const uint32_t ln = sph_lanes(s);
  auto kernel = ln == 8   ? k_sph_pairs<M, 8>
                : ln == 4 ? k_sph_pairs<M, 4>
                : ln == 2 ? k_sph_pairs<M, 2>
                          : k_sph_pairs<M, 1>;
  hipLaunchKernelGGL(kernel, dim3(pb_blocks(A.n, SC_T / ln)), dim3(SC_T), 0, s->ctx->stream, A, FB,
                     out4, out1);
}

// density, 1/rho and the cell-order views, shared by both physics
static int sph_alloc_views(pb_sys *s) {
  const size_t np = s->npad;
  int rc = PB_OK;
  if (!s->sph_rs) {
    // sph_rs last: the others exist where it does
    if ((rc = pb_alloc(s->ctx, &s->sph_rhoinv, np)) || (rc = pb_alloc(s->ctx, &s->sph_num, np)) ||
        (rc = pb_alloc(s->ctx, &s->sph_vs, np)) || (rc = pb_alloc(s->ctx, &s->sph_ds, np)) ||
        (rc = pb_alloc(s->ctx, &s->sph_mus, np)) || (rc = pb_alloc(s->ctx, &s->sph_fq, np)) ||
        (rc = pb_alloc(s->ctx, &s->sph_rs, np)))
      return rc;
  }
  hipStream_t st = s->ctx->stream;
  PB_HIP(s->ctx, hipMemsetAsync(s->sph_num, 0, sizeof(double4) * np, st));
  PB_HIP(s->ctx, hipMemsetAsync(s->sph_rhoinv, 0, 8 * np, st));
  return PB_OK;
}

extern "C" int pb_sph_set_properties(pb_sys *s, const double *mu0, const double *c, double h) {
  if (!s || !mu0 || !c || !(h > 0)) return PB_ERR_ARG;
  if (s->nrep != 1) return pb_fail(s->ctx, PB_ERR_ARG, "SPH: single replica only");
  PB_HIP(s->ctx, hipSetDevice(s->ctx->device));
  int rc = PB_OK;
  const size_t np = s->npad;
  if (!s->sph_mu0) {                       // the last of them
    if ((rc = pb_alloc(s->ctx, &s->sph_c2, np)) || (rc = pb_alloc(s->ctx, &s->sph_mu0, np)))
      return rc;
  }
  if ((rc = sph_alloc_views(s))) return rc;
  if ((rc = pb_io_scatter(s, mu0, s->sph_mu0, false)) ||
      (rc = pb_io_scatter(s, c, s->sph_c2, true)))              // c^2, cudaParticleSPH_NS.cu:63-64
    return rc;
  PB_HIP(s->ctx, hipStreamSynchronize(s->ctx->stream));
  s->sph_h = h;
  s->sph_rho0 = 1.0;
  s->sph_kind = 0;
  s->sph_set = true;
  s->sph_dens = false;
  return PB_OK;
}

extern "C" int pb_sph_set_wcsph(pb_sys *s, double h, double rho0, double c0, double gamma,
                                double alpha, double pmin) {
  if (!s || !(h > 0) || !(rho0 > 0) || !(c0 > 0) || !(gamma > 0) || !(alpha >= 0) ||
      std::isnan(pmin) || !std::isfinite(h * rho0 * c0 * gamma * alpha))
    return PB_ERR_ARG;
  if (s->nrep != 1) return pb_fail(s->ctx, PB_ERR_ARG, "SPH: single replica only");
  PB_HIP(s->ctx, hipSetDevice(s->ctx->device));
  if (int rc = sph_alloc_views(s)) return rc;
  PB_HIP(s->ctx, hipStreamSynchronize(s->ctx->stream));
  s->sph_h = h;
  s->sph_rho0 = rho0;
  s->sph_c0 = c0;
  s->sph_gamma = gamma;
  s->sph_alpha = alpha;
  s->sph_pmin = pmin;
  s->sph_kind = 1;
  s->sph_set = true;
  s->sph_dens = false;
  return PB_OK;
}

extern "C" int pb_sph_density(pb_sys *s) {
  if (!s) return PB_ERR_ARG;
  if (int rc = sph_ready(s)) return rc;
  PB_HIP(s->ctx, hipSetDevice(s->ctx->device));
  hipStream_t st = s->ctx->stream;
  const uint32_t n = s->n;
  if (n == 0) return PB_OK;
  SphArgs A = sph_args(s);
  const bool wc = s->sph_kind == 1;
  const SphFilter FB = sph_filter(s, wc ? A.sup2 : A.h * A.h);
  hipLaunchKernelGGL(k_sph_gather, dim3(pb_blocks(n, 256)), dim3(256), 0, st, s->perm, s->ref_bid,
                     s->r, s->v, wc ? (const double *)nullptr : s->sph_mu0, A.g, FB, n, s->sph_rs,
                     s->sph_fq, s->sph_mus);
  if (wc) sph_launch_pairs<SPH_WC_DENS>(s, A, FB, s->sph_num, s->sph_rhoinv);
  else sph_launch_pairs<SPH_LUCY_DENS>(s, A, FB, s->sph_num, s->sph_rhoinv);
  PB_LAUNCH_CHECK(s->ctx, "k_sph_pairs (density)");
  s->sph_dens = true;
  return PB_OK;
}

extern "C" int pb_sph_acceleration(pb_sys *s) {
  if (!s) return PB_ERR_ARG;
  if (int rc = sph_ready(s)) return rc;
  if (!s->sph_dens) return pb_fail(s->ctx, PB_ERR_STATE, "SPH: pb_sph_density first");
  PB_HIP(s->ctx, hipSetDevice(s->ctx->device));
  hipStream_t st = s->ctx->stream;
  const uint32_t n = s->n;
  if (n == 0) return PB_OK;
  SphArgs A = sph_args(s);
  const bool wc = s->sph_kind == 1;
  const SphFilter FB = sph_filter(s, wc ? A.sup2 : A.h * A.h);
  // current positions and velocities, and the density call's rho, 1/rho,
  // mu or p, in the current cell order
  hipLaunchKernelGGL(k_sph_gather_acc, dim3(pb_blocks(n, 256)), dim3(256), 0, st, s->perm,
                     s->ref_bid, s->r, s->v, s->sph_num, s->sph_rhoinv,
                     s->sph_c2 ? s->sph_c2 : s->sph_rhoinv,   // not read under the config physics
                     s->sph_rho0, wc ? 1 : 0, A.g, FB, n, s->sph_rs, s->sph_fq, s->sph_vs,
                     s->sph_ds);
  if (wc) sph_launch_pairs<SPH_WC_ACC>(s, A, FB, s->a, nullptr);
  else sph_launch_pairs<SPH_LUCY_ACC>(s, A, FB, s->a, nullptr);
  PB_LAUNCH_CHECK(s->ctx, "k_sph_pairs (acceleration)");
  return PB_OK;
}

extern "C" int pb_sph_inspect_density(pb_sys *s, double *mean_num) {
  if (!s || !mean_num) return PB_ERR_ARG;
  if (!s->sph_num) return pb_fail(s->ctx, PB_ERR_STATE, "SPH: no density yet");
  hipLaunchKernelGGL(k_sph_inspect, dim3(pb_blocks(s->npad, 256)), dim3(256), 0, s->ctx->stream,
                     s->sph_num, s->move, s->orig, s->npad, s->partials);
  PB_LAUNCH_CHECK(s->ctx, "k_sph_inspect");
  const double *h = nullptr;
  if (int rc = pb_reduce_to_host(s, 2, &h)) return rc;
  *mean_num = h[0] / h[1];     // 0/0 (no movable particle) is NaN, as the reference divides
  return PB_OK;
}
