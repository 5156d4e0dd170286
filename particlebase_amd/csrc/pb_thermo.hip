// pb_thermo.hip -- MD thermostat helpers on the storage layout:
//   * Gaussian isokinetic velocity Verlet (GaussianThermo::TimeEvolution,
//     GaussianThermo.cu:29-83),
//   * adjustVelocities (cudaParticleMD.cu:177-198, GaussianThermo.cu:98-119),
//   * constTemp (cudaParticleMD.cu:140-155).
//
// Gaussian step.  The reference solves the implicit velocity half of
//   v(t) = v(t-dt) + dt/2m (F(t) + F(t-dt)) - dt/2 (v(t-dt) xi(t-dt) + v(t) xi(t)),
//   xi(t) = sum F(t).v(t) / sum m v(t)^2
// by a Newton-Raphson loop with three host round trips per pass, stopping
// when the rms update of a pass is <= tol.  Writing
// A = v(t-dt) + dt/2m (F + Fold) - dt/2 v(t-dt) xi(t-dt), the system reads
// v = A / (1 + dt/2 xi(v)); every solution is v = A / c with one scalar c,
// and xi(A/c) = c (F.A)/(m A.A) gives c = 1 / (1 - dt/2 g), g = F.A / m A.A.
// So v(t) = A (1 - dt/2 g) and xi(t) = g / (1 - dt/2 g) is the fixed point
// the loop converges to.  The loop's first pass uses the previous step's
// xi; when that pass already moves v by no more than tol (always so when
// xi(t-dt) = 0, as on the first step) the reference stops there with the
// one-pass velocity and xi of it, so that pass is evaluated too and decides
// the branch exactly as the loop's test does.  Three to five launches, no host
// synchronisation (the solves are part of the kernels after them for small
// replicas):
//   k_gt_a       A into v, v' = v + dt/2m (F + Fold) into a; partials
//                F.A, m A.A, m v'.v'
//   k_gt_solve1  per replica (fixed order): 1/c, xi of the fixed point,
//                1 / sum m v'.v'
//   k_gt_pass1   the loop's first Newton pass from v' with the previous xi:
//                v1 = v' - f/f' into a; partials (f/f')^2, F.v1, m v1.v1
//   k_gt_solve2  rms of the pass vs tol: one-pass result or fixed point
//   k_gt_drift   v = v1 or A/c ; r += v (dt - xi dt^2/2) + F dt^2/2m ;
//                Fold = F
// Per-replica xi persists on the device between steps (GaussianThermo::xi).
#include "pb_internal.h"
#include <algorithm>

#define GT_BLOCK 256
#define GT_SOLVE_WAVES 512u   // largest replica solved without launches of its own

namespace {

// gt holds 4 doubles per replica: [0] xi (persistent), [1] 1/c of the
// fixed point or -1 when the one-pass result is taken, [2] 1 / sum m v'.v',
// [3] xi of the fixed point.

__global__ void __launch_bounds__(GT_BLOCK)
    k_gt_a(double4 *v, const double4 *F, double4 *Fold, const uint32_t *orig,
           const uint32_t *waveRep, const double *gt, uint32_t n, double dt, double *partials) {
  const uint32_t s = blockIdx.x * blockDim.x + threadIdx.x;
  double fa = 0.0, ma2 = 0.0, mv2 = 0.0;
  if (s < n && orig[s] != PB_NONE) {
    const double xi = gt[4 * waveRep[s / PB_WAVE]];
    const double dt2 = 0.5 * dt;
    double4 V = v[s];
    const double4 f = F[s], fo = Fold[s];
    const double dtm2 = dt2 * V.w, xd = xi * dt2;
    const double px = V.x + (f.x + fo.x) * dtm2;     // v'
    const double py = V.y + (f.y + fo.y) * dtm2;
    const double pz = V.z + (f.z + fo.z) * dtm2;
    const double ax = px - V.x * xd, ay = py - V.y * xd, az = pz - V.z * xd;   // A
    fa = f.x * ax + f.y * ay + f.z * az;
    ma2 = (ax * ax + ay * ay + az * az) / V.w;
    mv2 = (px * px + py * py + pz * pz) / V.w;
    V.x = ax;
    V.y = ay;
    V.z = az;
    v[s] = V;
    Fold[s] = make_double4(px, py, pz, 0.0);
  }
  fa = pb_wave_sum(fa);
  ma2 = pb_wave_sum(ma2);
  mv2 = pb_wave_sum(mv2);
  if (pb_lane() == 0 && s < n) {
    double *P = partials + 4 * (s / PB_WAVE);
    P[0] = fa;
    P[1] = ma2;
    P[2] = mv2;
  }
}

// Sums of a replica's partials in every lane of a wavefront
struct GtSums {
  double x[3];
  __device__ __forceinline__ GtSums(const double *partials, const RepInfo &R) {
    const uint32_t w0[1] = {R.wave0}, nw[1] = {R.nwave};
    double y[1][3];
    pb_wave_reduce<3>(partials, w0, nw, y);
#pragma unroll
    for (int c = 0; c < 3; ++c) x[c] = y[0][c];
  }
};

// 1/c, xi of the fixed point and 1 / sum m v'^2 from the sums of k_gt_a.  A
// replica whose A vanishes (all particles at rest, no force) has no defined
// xi: g = 0.
struct GtSolve1 {
  double cinv, mv2inv, xi;
  __device__ __forceinline__ GtSolve1(double fa, double ma2, double mv2, double dt) {
    const double g = ma2 > 0.0 ? fa / ma2 : 0.0;
    cinv = 1.0 - 0.5 * dt * g;
    mv2inv = mv2 > 0.0 ? 1.0 / mv2 : 0.0;
    xi = g / cinv;
  }
};

// The loop's test after its first pass, v0 = sqrt(sum q^2 / 3N) <= tol, picks
// the one-pass result (1/c = -1); otherwise the fixed point, which has no
// solution when 1/c <= 0 (dt too large for the forces; the reference's loop does
// not converge there): bad, and taken as xi = 0, v = A.
struct GtSolve2 {
  double xi, cinv;
  bool bad;
  __device__ __forceinline__ GtSolve2(const double (&x)[3], double natoms, double tol, double cinv1,
                                      double xi1) {
    const double v0 = sqrt(x[0] / (3.0 * natoms));
    bad = false;
    xi = xi1;
    cinv = cinv1;
    if (!(v0 > tol)) {
      xi = x[2] > 0.0 ? x[1] / x[2] : 0.0;
      cinv = -1.0;
    } else if (!(cinv1 > 0.0 && isfinite(xi1))) {
      bad = true;
      xi = 0.0;
      cinv = 1.0;
    }
  }
};

// One workgroup.
__global__ void __launch_bounds__(256)
    k_gt_solve1(const double *partials, const RepInfo *reps, uint32_t nrep, double dt,
                double *out, double *gt) {
  __shared__ double sm[4 * 256];
  pb_block_reduce_reps<3>(partials, reps, nrep, out, false, sm);
  __syncthreads();
  for (uint32_t q = threadIdx.x; q < nrep; q += blockDim.x) {
    const GtSolve1 S(out[8 * q], out[8 * q + 1], out[8 * q + 2], dt);
    gt[4 * q + 1] = S.cinv;
    gt[4 * q + 2] = S.mv2inv;
    gt[4 * q + 3] = S.xi;
  }
}

// The first pass of calcGaussianThermoFoverF_F4 (kernelfuncs.cu:407-454):
// f = A - (dt/2 xi + 1) v', f' = -dt/2 (xi + (F - 2 xi m v') v' / sum m v'^2) - 1.
// SOLVE: every wavefront sums its replica's partials `in` and solves for itself,
// the first one stores the result (k_gt_solve1's).
template <bool SOLVE>
__global__ void __launch_bounds__(GT_BLOCK)
    k_gt_pass1(const double4 *v, const double4 *F, double4 *Fold, const uint32_t *orig,
               const uint32_t *waveRep, const RepInfo *reps, const double *in, double *gt,
               uint32_t n, double dt, double *partials) {
  const uint32_t s = blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= n) return;                            // whole wavefronts
  double qq = 0.0, fv = 0.0, mv2 = 0.0;
  double *G = gt + 4 * waveRep[s / PB_WAVE];
  double mv2inv;
  if constexpr (SOLVE) {
    const RepInfo &R = reps[waveRep[s / PB_WAVE]];
    const GtSums T(in, R);
    const GtSolve1 S(T.x[0], T.x[1], T.x[2], dt);
    mv2inv = S.mv2inv;
    if (pb_lane() == 0 && s / PB_WAVE == R.wave0) {
      G[1] = S.cinv;
      G[2] = S.mv2inv;
      G[3] = S.xi;
    }
  } else {
    mv2inv = G[2];
  }
  if (orig[s] != PB_NONE) {
    const double xi = G[0], dt2 = 0.5 * dt;
    const double4 A = v[s], f = F[s], p = Fold[s];
    const double m = 1.0 / A.w, k1 = dt2 * xi + 1.0, k2 = 2.0 * xi * m;
    const double qx = (A.x - k1 * p.x) / (-dt2 * (xi + (f.x - k2 * p.x) * p.x * mv2inv) - 1.0);
    const double qy = (A.y - k1 * p.y) / (-dt2 * (xi + (f.y - k2 * p.y) * p.y * mv2inv) - 1.0);
    const double qz = (A.z - k1 * p.z) / (-dt2 * (xi + (f.z - k2 * p.z) * p.z * mv2inv) - 1.0);
    const double x = p.x - qx, y = p.y - qy, z = p.z - qz;
    qq = qx * qx + qy * qy + qz * qz;
    fv = f.x * x + f.y * y + f.z * z;
    mv2 = (x * x + y * y + z * z) * m;
    Fold[s] = make_double4(x, y, z, 0.0);
  }
  qq = pb_wave_sum(qq);
  fv = pb_wave_sum(fv);
  mv2 = pb_wave_sum(mv2);
  if (pb_lane() == 0) {
    double *P = partials + 4 * (s / PB_WAVE);
    P[0] = qq;
    P[1] = fv;
    P[2] = mv2;
  }
}

// One workgroup; steps without a solution are counted in bad[0].
__global__ void __launch_bounds__(256)
    k_gt_solve2(const double *partials, const RepInfo *reps, uint32_t nrep, double tol,
                double *out, double *gt, uint32_t *bad) {
  __shared__ double sm[4 * 256];
  pb_block_reduce_reps<3>(partials, reps, nrep, out, false, sm);
  __syncthreads();
  for (uint32_t q = threadIdx.x; q < nrep; q += blockDim.x) {
    double *G = gt + 4 * q;
    const double x[3] = {out[8 * q], out[8 * q + 1], out[8 * q + 2]};
    const GtSolve2 S(x, reps[q].natoms, tol, G[1], G[3]);
    G[0] = S.xi;
    G[1] = S.cinv;
    if (S.bad) atomicAdd(bad, 1u);
  }
}

// SOLVE: as in k_gt_pass1, for k_gt_solve2; the first wavefront stores xi (the
// others may still read the fixed point's terms, which stay).
template <bool SOLVE>
__global__ void __launch_bounds__(GT_BLOCK)
    k_gt_drift(double4 *r, double4 *v, const double4 *F, double4 *Fold, const uint32_t *orig,
               const uint32_t *waveRep, const RepInfo *reps, const double *in, double *gt,
               uint32_t n, double dt, double tol, uint32_t *bad) {
  const uint32_t s = blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= n) return;
  double *G = gt + 4 * waveRep[s / PB_WAVE];
  double xi, cinv;
  if constexpr (SOLVE) {
    const RepInfo &R = reps[waveRep[s / PB_WAVE]];
    const GtSums T(in, R);
    const GtSolve2 S(T.x, R.natoms, tol, G[1], G[3]);
    xi = S.xi;
    cinv = S.cinv;
    if (pb_lane() == 0 && s / PB_WAVE == R.wave0) {
      G[0] = xi;
      if (S.bad) atomicAdd(bad, 1u);
    }
  } else {
    xi = G[0];
    cinv = G[1];
  }
  if (orig[s] == PB_NONE) return;
  double4 V = v[s];
  const double4 f = F[s];
  if (cinv < 0.0) {
    const double4 p = Fold[s];
    V.x = p.x;
    V.y = p.y;
    V.z = p.z;
  } else {
    V.x *= cinv;
    V.y *= cinv;
    V.z *= cinv;
  }
  const double dt22 = 0.5 * dt * dt;
  const double cv = dt - xi * dt22, cf = dt22 * V.w;
  double4 R = r[s];
  R.x += V.x * cv + f.x * cf;
  R.y += V.y * cv + f.y * cf;
  R.z += V.z * cv + f.z * cf;
  r[s] = R;
  v[s] = V;
  Fold[s] = make_double4(f.x, f.y, f.z, 0.0);
}

// per-wave partials of sum v (K = 3 components) for the velocity adjustment
__global__ void __launch_bounds__(GT_BLOCK)
    k_vsum_partial(const double4 *v, const uint32_t *orig, uint32_t n, double *partials) {
  const uint32_t s = blockIdx.x * blockDim.x + threadIdx.x;
  double x = 0.0, y = 0.0, z = 0.0;
  if (s < n && orig[s] != PB_NONE) {
    const double4 V = v[s];
    x = V.x;
    y = V.y;
    z = V.z;
  }
  x = pb_wave_sum(x);
  y = pb_wave_sum(y);
  z = pb_wave_sum(z);
  if (pb_lane() == 0 && s < n) {
    double *P = partials + 4 * (s / PB_WAVE);
    P[0] = x;
    P[1] = y;
    P[2] = z;
  }
}

// per-wave partials of sum (v - mean)^2 per axis; means at stats[6q + 0..2]
__global__ void __launch_bounds__(GT_BLOCK)
    k_vvar_partial(const double4 *v, const uint32_t *orig, const uint32_t *waveRep,
                   const double *stats, uint32_t n, double *partials) {
  const uint32_t s = blockIdx.x * blockDim.x + threadIdx.x;
  double x = 0.0, y = 0.0, z = 0.0;
  if (s < n && orig[s] != PB_NONE) {
    const double *S = stats + 6 * waveRep[s / PB_WAVE];
    const double4 V = v[s];
    x = V.x - S[0];
    y = V.y - S[1];
    z = V.z - S[2];
    x *= x;
    y *= y;
    z *= z;
  }
  x = pb_wave_sum(x);
  y = pb_wave_sum(y);
  z = pb_wave_sum(z);
  if (pb_lane() == 0 && s < n) {
    double *P = partials + 4 * (s / PB_WAVE);
    P[0] = x;
    P[1] = y;
    P[2] = z;
  }
}

// v = (v - mean) * v1 / sqrt(var); mean and variance per replica in
// stats[6q + 0..5] (means, then variances).
__global__ void __launch_bounds__(GT_BLOCK)
    k_vadjust(double4 *v, const uint32_t *orig, const uint32_t *waveRep, const double *stats,
              uint32_t n, double v1) {
  const uint32_t s = blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= n || orig[s] == PB_NONE) return;
  const double *S = stats + 6 * waveRep[s / PB_WAVE];
  double4 V = v[s];
  V.x = (V.x - S[0]) * (v1 / sqrt(S[3]));
  V.y = (V.y - S[1]) * (v1 / sqrt(S[4]));
  V.z = (V.z - S[2]) * (v1 / sqrt(S[5]));
  v[s] = V;
}

// means / variances from the two passes of sums; one workgroup
__global__ void __launch_bounds__(256)
    k_vstats(const double *partials, const RepInfo *reps, uint32_t nrep, double *out,
             double *stats, int pass) {
  __shared__ double sm[4 * 256];
  pb_block_reduce_reps<3>(partials, reps, nrep, out, false, sm);
  __syncthreads();
  for (uint32_t q = threadIdx.x; q < nrep; q += blockDim.x) {
    const double inv = 1.0 / (double)reps[q].natoms;
    for (int c = 0; c < 3; ++c) stats[6 * q + 3 * pass + c] = out[8 * q + c] * inv;
  }
}

// per-wave partials of sum F.v and sum m v^2 (constTemp)
__global__ void __launch_bounds__(GT_BLOCK)
    k_fv_partial(const double4 *v, const double4 *F, const uint32_t *orig, uint32_t n,
                 double *partials) {
  const uint32_t s = blockIdx.x * blockDim.x + threadIdx.x;
  double fv = 0.0, mv2 = 0.0;
  if (s < n && orig[s] != PB_NONE) {
    const double4 V = v[s], f = F[s];
    fv = f.x * V.x + f.y * V.y + f.z * V.z;
    mv2 = (V.x * V.x + V.y * V.y + V.z * V.z) / V.w;
  }
  fv = pb_wave_sum(fv);
  mv2 = pb_wave_sum(mv2);
  if (pb_lane() == 0 && s < n) {
    partials[4 * (s / PB_WAVE) + 0] = fv;
    partials[4 * (s / PB_WAVE) + 1] = mv2;
  }
}

// lambda per replica into out[8q + 4] (0 when sum m v^2 vanishes)
__global__ void __launch_bounds__(256)
    k_ct_solve(const double *partials, const RepInfo *reps, uint32_t nrep, double *out) {
  __shared__ double sm[4 * 256];
  pb_block_reduce_reps<2>(partials, reps, nrep, out, false, sm);
  __syncthreads();
  for (uint32_t q = threadIdx.x; q < nrep; q += blockDim.x) {
    const double fv = out[8 * q], mv2 = out[8 * q + 1];
    out[8 * q + 4] = mv2 > 0.0 ? fv / mv2 : 0.0;
  }
}

// F -= lambda m v (correctConstTemp_F4, kernelfuncs.cu:533-544)
__global__ void __launch_bounds__(GT_BLOCK)
    k_ct_apply(const double4 *v, double4 *F, const uint32_t *orig, const uint32_t *waveRep,
               const double *out, uint32_t n) {
  const uint32_t s = blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= n || orig[s] == PB_NONE) return;
  const double lam = out[8 * waveRep[s / PB_WAVE] + 4];
  if (lam == 0.0) return;
  const double4 V = v[s];
  double4 f = F[s];
  const double lm = lam / V.w;
  f.x -= lm * V.x;
  f.y -= lm * V.y;
  f.z -= lm * V.z;
  F[s] = f;
}

int ensure_gt(pb_sys *s) {
  if (s->gt) return PB_OK;
  if (int rc = pb_alloc(s->ctx, &s->gt_bad, 1)) return rc;
  if (int rc = pb_alloc(s->ctx, &s->gt_part, 4 * (size_t)s->nwave)) return rc;
  if (int rc = pb_alloc(s->ctx, &s->gt, 4 * (size_t)s->nrep)) return rc;
  const uint32_t zero = 0;
  PB_HIP(s->ctx, hipMemcpyAsync(s->gt_bad, &zero, sizeof(uint32_t), hipMemcpyHostToDevice,
                                s->ctx->stream));
  std::vector<double> h(4 * (size_t)s->nrep, 0.0);   // xi(0) = 0 (GaussianThermo() : xi(0))
  PB_HIP(s->ctx, hipMemcpyAsync(s->gt, h.data(), sizeof(double) * h.size(),
                                hipMemcpyHostToDevice, s->ctx->stream));
  PB_HIP(s->ctx, hipStreamSynchronize(s->ctx->stream));
  return PB_OK;
}

}  // namespace

#define GT_GRID(n) dim3(pb_blocks((n), GT_BLOCK)), dim3(GT_BLOCK), 0, s->ctx->stream

extern "C" int pb_gt_step(pb_sys *s, double dt, double tol) {
  if (!s) return PB_ERR_ARG;
  if (!(dt > 0.0)) return pb_fail(s->ctx, PB_ERR_ARG, "pb_gt_step: dt must be positive");
  if (!(tol >= 0.0)) return pb_fail(s->ctx, PB_ERR_ARG, "pb_gt_step: tol must be >= 0");
  if (int rc = ensure_gt(s)) return rc;
  hipStream_t st = s->ctx->stream;
  hipLaunchKernelGGL(k_gt_a, GT_GRID(s->npad), s->v, s->F, s->a, s->orig, s->waveRep, s->gt,
                     s->npad, dt, s->partials);
  // Replicas of few wavefronts are solved by every wavefront of the kernels that
  // need the result, two launches of one workgroup fewer; each reads all of its
  // replica's partials, so larger ones keep the launches (us a step with 3 and
  // with 5 launches: 500 particles 12.5, 20; 4924 11.4, 15.1; 16,000 12.8, 16.3;
  // 32,000 15.4, 16.5; 64,000 20.9, 18.9).
  uint32_t most = 0;
  for (const RepInfo &R : s->reps) most = std::max(most, R.nwave);
  if (most <= GT_SOLVE_WAVES) {
    hipLaunchKernelGGL(k_gt_pass1<true>, GT_GRID(s->npad), s->v, s->F, s->a, s->orig, s->waveRep,
                       s->d_reps, s->partials, s->gt, s->npad, dt, s->gt_part);
    hipLaunchKernelGGL(k_gt_drift<true>, GT_GRID(s->npad), s->r, s->v, s->F, s->a, s->orig, s->waveRep,
                       s->d_reps, s->gt_part, s->gt, s->npad, dt, tol, s->gt_bad);
  } else {
    hipLaunchKernelGGL(k_gt_solve1, dim3(1), dim3(256), 0, st, s->partials, s->d_reps, s->nrep, dt,
                       s->d_out, s->gt);
    hipLaunchKernelGGL(k_gt_pass1<false>, GT_GRID(s->npad), s->v, s->F, s->a, s->orig, s->waveRep,
                       s->d_reps, (const double *)nullptr, s->gt, s->npad, dt, s->partials);
    hipLaunchKernelGGL(k_gt_solve2, dim3(1), dim3(256), 0, st, s->partials, s->d_reps, s->nrep, tol,
                       s->d_out, s->gt, s->gt_bad);
    hipLaunchKernelGGL(k_gt_drift<false>, GT_GRID(s->npad), s->r, s->v, s->F, s->a, s->orig, s->waveRep,
                       s->d_reps, (const double *)nullptr, s->gt, s->npad, dt, tol, s->gt_bad);
  }
  PB_LAUNCH_CHECK(s->ctx, "pb_gt_step");
  return PB_OK;
}

extern "C" int pb_gt_xi(pb_sys *s, const double *set_xi, double *get_xi, uint32_t *bad_steps) {
  if (!s) return PB_ERR_ARG;
  if (int rc = ensure_gt(s)) return rc;
  std::vector<double> h(4 * (size_t)s->nrep);
  PB_HIP(s->ctx, hipMemcpyAsync(h.data(), s->gt, sizeof(double) * h.size(),
                                hipMemcpyDeviceToHost, s->ctx->stream));
  uint32_t nb = 0;
  PB_HIP(s->ctx, hipMemcpyAsync(&nb, s->gt_bad, sizeof(uint32_t), hipMemcpyDeviceToHost,
                                s->ctx->stream));
  PB_HIP(s->ctx, hipStreamSynchronize(s->ctx->stream));
  if (get_xi)
    for (uint32_t q = 0; q < s->nrep; ++q) get_xi[q] = h[4 * q];
  if (bad_steps) *bad_steps = nb;
  if (set_xi) {
    for (uint32_t q = 0; q < s->nrep; ++q) h[4 * q] = set_xi[q];
    PB_HIP(s->ctx, hipMemcpyAsync(s->gt, h.data(), sizeof(double) * h.size(),
                                  hipMemcpyHostToDevice, s->ctx->stream));
    nb = 0;
    PB_HIP(s->ctx, hipMemcpyAsync(s->gt_bad, &nb, sizeof(uint32_t), hipMemcpyHostToDevice,
                                  s->ctx->stream));
    PB_HIP(s->ctx, hipStreamSynchronize(s->ctx->stream));
  }
  return PB_OK;
}

extern "C" int pb_adjust_velocities(pb_sys *s, double v1, double *stats) {
  if (!s) return PB_ERR_ARG;
  if (!(v1 >= 0.0)) return pb_fail(s->ctx, PB_ERR_ARG, "pb_adjust_velocities: v1 < 0");
  double *dstats = s->d_out + 8 * (size_t)s->nrep;   // 6 per replica after the 8-word records
  // pass 0: sums -> means; pass 1: centred squares -> variances (two-pass)
  hipLaunchKernelGGL(k_vsum_partial, GT_GRID(s->npad), s->v, s->orig, s->npad, s->partials);
  hipLaunchKernelGGL(k_vstats, dim3(1), dim3(256), 0, s->ctx->stream, s->partials, s->d_reps,
                     s->nrep, s->d_out, dstats, 0);
  hipLaunchKernelGGL(k_vvar_partial, GT_GRID(s->npad), s->v, s->orig, s->waveRep, dstats,
                     s->npad, s->partials);
  hipLaunchKernelGGL(k_vstats, dim3(1), dim3(256), 0, s->ctx->stream, s->partials, s->d_reps,
                     s->nrep, s->d_out, dstats, 1);
  PB_LAUNCH_CHECK(s->ctx, "pb_adjust_velocities (statistics)");
  std::vector<double> h(6 * (size_t)s->nrep);
  PB_HIP(s->ctx, hipMemcpyAsync(h.data(), dstats, sizeof(double) * h.size(),
                                hipMemcpyDeviceToHost, s->ctx->stream));
  PB_HIP(s->ctx, hipStreamSynchronize(s->ctx->stream));
  for (uint32_t q = 0; q < s->nrep; ++q)
    for (int c = 0; c < 3; ++c)
      if (!(h[6 * q + 3 + c] > 0.0))
        return pb_fail(s->ctx, PB_ERR_ARG,
                       "pb_adjust_velocities: a velocity component has zero variance");
  if (stats) std::copy(h.begin(), h.end(), stats);
  hipLaunchKernelGGL(k_vadjust, GT_GRID(s->npad), s->v, s->orig, s->waveRep, dstats, s->npad, v1);
  PB_LAUNCH_CHECK(s->ctx, "pb_adjust_velocities");
  return PB_OK;
}

extern "C" int pb_const_temp(pb_sys *s, double *mv2, double *lambda) {
  if (!s) return PB_ERR_ARG;
  hipLaunchKernelGGL(k_fv_partial, GT_GRID(s->npad), s->v, s->F, s->orig, s->npad, s->partials);
  hipLaunchKernelGGL(k_ct_solve, dim3(1), dim3(256), 0, s->ctx->stream, s->partials, s->d_reps,
                     s->nrep, s->d_out);
  hipLaunchKernelGGL(k_ct_apply, GT_GRID(s->npad), s->v, s->F, s->orig, s->waveRep, s->d_out,
                     s->npad);
  PB_LAUNCH_CHECK(s->ctx, "pb_const_temp");
  if (mv2 || lambda) {
    std::vector<double> h(8 * (size_t)s->nrep);
    PB_HIP(s->ctx, hipMemcpyAsync(h.data(), s->d_out, sizeof(double) * h.size(),
                                  hipMemcpyDeviceToHost, s->ctx->stream));
    PB_HIP(s->ctx, hipStreamSynchronize(s->ctx->stream));
    for (uint32_t q = 0; q < s->nrep; ++q) {
      if (mv2) mv2[q] = h[8 * q + 1];
      if (lambda) lambda[q] = h[8 * q + 4];
    }
  }
  return PB_OK;
}
