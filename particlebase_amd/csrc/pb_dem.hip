// pb_dem.hip -- DEM contact path of cudaParticleDEM (+ cudaParticleRotation)
// on MI355X.  Compiled without FP contraction: the contact decisions
// (|r_ij|^2 < (r_i + r_j)^2 in FP64) are the same IEEE operations as the
// FP64 oracle's, so the contact CSR is reproducible bit for bit.
//
// Reference path (cudaParticleDEM.cu:29-213, kernelfuncs.cu:1088-1309,
// kerneltemplate.hh:135-168, 311-418, kernelinline.hh:235-382): a
// coordination-number pass, a single-block partial sum for the row
// pointers, a host read of nnz, a column-index pass, a per-row sort, the
// history carry-over from the previous matrix and the contact-force pass.
//
// Here the same stages run as: a gather of (x, y, z, radius) into cell order
// and an FP32 view of it -> count (one thread per particle in cell order, 27 or
// 125 neighbour cells as contiguous ranges) -> exclusive scan -> one kernel that sorts
// each row, takes the tangential history over from the previous matrix (both
// rows sorted) and computes contact force and torque.  The column arrays are
// sized from the previous step's count; that kernel stops at the capacity and
// the host reads nnz and the time-step check together at the end, repeating it
// with larger arrays in the rare step where nnz outgrew them (one host
// synchronisation per call).  Rows are indexed by the original particle index
// and hold original indices in ascending order.  Contacts use the strict
// |r_ij| < r_i + r_j for both the count and the list (the reference lists
// with <=, which overruns a row on an exact touch, kernelfuncs.cu:1158).
#include "pb_internal.h"
#include <algorithm>
#include <cmath>
#include <vector>

__global__ void k_fill_u32(uint32_t *x, uint32_t n, uint32_t val);

struct DemGrid {
  const uint32_t *perm, *bid, *cstart;
  const double4 *rs;        // cell order: (x, y, z, radius)
  const float4 *fq;         // cell order: the same for the FP32 filter (dem_view)
  const uint32_t *so;       // cell order: original index
  const uint8_t *move;
  uint32_t nb[3];
  uint32_t n;
  uint32_t cap;     // capacity of the column arrays
  uint32_t *rowbuf; // DEM_ROWBUF contacts per particle, by original index
};

// contacts a particle's row keeps from the counting scan; longer rows (more
// touching neighbours than any sphere packing gives) are scanned again
#define DEM_ROWBUF 16u

// FP32 view for a first test that passes every pair in contact: positions from
// the grid's corner, up to `span` from it, and the radius with half the margin
// that covers their rounding: 2^-24 span a coordinate and particle, so less than
// 4e-7 span a distance, and a few units of relative rounding.  A particle beyond
// the span (outside the grid, binned into its edge cells; NaN) gets an infinite
// radius.
struct DemView {
  double lo[3];
  float span;
};
__device__ __forceinline__ float4 dem_view(const DemView &V, const double4 &p) {
  const float x = (float)(p.x - V.lo[0]), y = (float)(p.y - V.lo[1]), z = (float)(p.z - V.lo[2]);
  if (!(fabsf(x) <= V.span && fabsf(y) <= V.span && fabsf(z) <= V.span))
    return make_float4(0.f, 0.f, 0.f, INFINITY);
  // at least 1e-18, so that the squares stay normal
  return make_float4(x, y, z, fmaxf(fabsf((float)p.w) * 1.000001f + 2e-7f * V.span, 1e-18f));
}

// positions with the radius in w and their view, in cell order
__global__ void k_dem_gather(const uint32_t *perm, const double4 *r, const double *rad, uint32_t n,
                             DemView V, double4 *rs, float4 *fq) {
  const uint32_t k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= n) return;
  const uint32_t s = perm[k];
  const double4 p = r[s];
  const double4 o = make_double4(p.x, p.y, p.z, rad[s]);
  rs[k] = o;
  fq[k] = dem_view(V, o);
}

// (x, y, z, radius) of both particles
__device__ __forceinline__ bool in_contact(const double4 &pi, const double4 &pj) {
  const double dx = pi.x - pj.x, dy = pi.y - pj.y, dz = pi.z - pj.z;
  const double R2 = dx * dx + dy * dy + dz * dz;
  const double rc = pi.w + pj.w;
  return R2 < rc * rc;
}

// f(original index) for every particle in contact with particle k, over the
// (2W + 1)^3 cells around its own (non-periodic: DEM distances never use an image,
// kernelinline.hh:248), in no particular order.  The scan is a chain of dependent
// reads (cell starts, candidates) at few wavefronts a SIMD, so the starts of a
// row of columns are read together, and the first candidates of several columns
// (a column holds one to three) in one go, as FP32 views; what passes is listed
// in the thread's LDS and tested exactly four at a time.
template <int W, typename F, size_t T>
__device__ __forceinline__ void dem_contacts(const DemGrid &G, uint32_t k,
                                             uint32_t (&list)[DEM_ROWBUF][T], F &&f) {
  const uint32_t tid = threadIdx.x;
  const uint32_t c = G.bid[k], nz = G.nb[2], nyz = G.nb[1] * nz;
  const int i0 = (int)(c / nyz), j0 = (int)((c / nz) % G.nb[1]), k0 = (int)(c % nz);
  const uint32_t kl = (uint32_t)max(k0 - W, 0), kh = (uint32_t)min(k0 + W, (int)nz - 1) + 1u;
  const double4 pi = G.rs[k];
  const float4 fi = G.fq[k];
  uint32_t cnt = 0;
  auto work_off = [&]() {
    for (uint32_t e = 0; e < cnt; e += 4) {
      uint32_t q[4], o[4];
      double4 pj[4];
#pragma unroll
      for (uint32_t u = 0; u < 4; ++u) q[u] = list[min(e + u, cnt - 1u)][tid];
#pragma unroll
      for (uint32_t u = 0; u < 4; ++u) {
        pj[u] = G.rs[q[u]];
        o[u] = G.so[q[u]];
      }
#pragma unroll
      for (uint32_t u = 0; u < 4; ++u)
        if (e + u < cnt && in_contact(pi, pj[u])) f(o[u]);
    }
    cnt = 0;
  };
  constexpr int NG = 2 * W + 1;                       // columns of a row, tested together,
  constexpr uint32_t U = W == 1 ? 4u : 2u;            // that many candidates each
  static_assert(NG * U <= DEM_ROWBUF, "a round's candidates fit the list");
  auto starts = [&](int a, uint32_t (&q0)[NG], uint32_t (&q1)[NG]) {
    const int i2 = i0 + a;
#pragma unroll
    for (int t = 0; t < NG; ++t) {
      const int j2 = j0 + t - W;
      const bool ok = a <= W && i2 >= 0 && i2 < (int)G.nb[0] && j2 >= 0 && j2 < (int)G.nb[1];
      const uint32_t cb = ok ? (uint32_t)i2 * nyz + (uint32_t)j2 * nz : 0u;
      q0[t] = G.cstart[cb + kl];
      q1[t] = ok ? G.cstart[cb + kh] : q0[t];
    }
  };
  uint32_t q0[NG], q1[NG], n0[NG], n1[NG];
  starts(-W, q0, q1);
#pragma unroll 1
  for (int a = -W; a <= W; ++a) {
    starts(a + 1, n0, n1);                            // the next row on its way
    bool more;
    uint32_t o = 0;
#pragma unroll 1
    do {
      float4 fj[NG][U];
#pragma unroll
      for (int t = 0; t < NG; ++t)
#pragma unroll
        for (uint32_t u = 0; u < U; ++u) {
          const uint32_t q = q0[t] + o + u;
          fj[t][u] = G.fq[q < q1[t] ? q : k];         // past the end: the particle itself
        }
      more = false;
#pragma unroll
      for (int t = 0; t < NG; ++t) {
#pragma unroll
        for (uint32_t u = 0; u < U; ++u) {
          const uint32_t q = q0[t] + o + u;
          const float dx = fi.x - fj[t][u].x, dy = fi.y - fj[t][u].y, dz = fi.z - fj[t][u].z;
          const float rr = fi.w + fj[t][u].w;
          if (q < q1[t] && q != k && dx * dx + dy * dy + dz * dz < rr * rr) list[cnt++][tid] = q;
        }
        more |= q0[t] + o + U < q1[t];
      }
      o += U;
      // room for the next round; the last row's rounds end here too
      if (cnt > DEM_ROWBUF - NG * U || (a == W && !more)) work_off();
    } while (more);
#pragma unroll
    for (int t = 0; t < NG; ++t) {
      q0[t] = n0[t];
      q1[t] = n1[t];
    }
  }
}

// calcCoord_F4 (kernelinline.hh:371-382): contacts of movable particles
// The same scan keeps the first DEM_ROWBUF contacts (original indices, in no
// particular order) in the row buffer for the rows.
// 200,000 dispersed spheres 14 us stored in lattice order and 16 in random order, a
// bed of 60,000 14 us (FP64 candidates column by column: 18 for the first, 15 for
// the bed); at most 128 registers, so that four wavefronts fit a SIMD.
template <int W>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(4)))
k_dem_count(DemGrid G, uint32_t *cnt, uint32_t *bad) {
  __shared__ uint32_t list[DEM_ROWBUF][256];
  const uint32_t k = pb_xcd_chunk8() * 256u + threadIdx.x;
  if (k == 0) *bad = 0;                               // Cundall-Strack violations of this call
  if (k >= G.n) return;
  const uint32_t i = G.so[k];
  uint32_t c = 0;
  if (G.move[G.perm[k]]) {
    uint32_t *buf = G.rowbuf + (size_t)i * DEM_ROWBUF;
    dem_contacts<W>(G, k, list, [&](uint32_t o) {
      if (c < DEM_ROWBUF) buf[c] = o;
      ++c;
    });
  }
  cnt[i] = c;
}

struct DemForceArgs {
  const uint32_t *inv;                 // original -> storage
  const uint32_t *prow, *pcol;         // previous matrix (null: none)
  const double *pval;
  const uint32_t *row;
  uint32_t *col;
  double *val;
  const double4 *r, *v, *w;
  const double *rad;
  const uint8_t *move;
  double4 *F, *T;
  uint32_t *bad;                         // Cundall-Strack violations
  uint32_t *res;                         // pinned: nnz, and 1 if there are any violations
  double E, mu, s2, gamma2, mu_r, dt;
  double kn, zeta, kt;                   // linear law
};

// a particle's state and sums
struct DemBody {
  double4 p, v, w;
  double rad;
  double f[3] = {0, 0, 0}, t[3] = {0, 0, 0};
  uint32_t bad = 0;
};

// the other particle of a contact
struct DemOther {
  double4 p, v, w;
  double rad;
  uint32_t move;
};
__device__ __forceinline__ DemOther dem_other(const DemForceArgs &A, uint32_t sj) {
  return DemOther{A.r[sj], A.v[sj], A.w[sj], A.rad[sj], A.move[sj]};
}

// DEMContact_F4 (kernelinline.hh:235-363), FP64.  h: the contact's history (1
// double: the slip length), updated in place.
__device__ __forceinline__ void contact_hertz(const DemForceArgs &A, DemBody &B, const DemOther &J, double *h) {
  const double4 &pi = B.p, &vi = B.v, &wi = B.w;
  const double ri = B.rad;
  const bool wnz = wi.x != 0 && wi.y != 0 && wi.z != 0;
  const double4 &pj = J.p, &vj = J.v, &wj = J.w;
  const double rj = J.rad;
  const double d[3] = {pi.x - pj.x, pi.y - pj.y, pi.z - pj.z};
  const double R2 = d[0] * d[0] + d[1] * d[1] + d[2] * d[2];
  const double rs = ri + rj;
  if (!(R2 < rs * rs)) return;
  const double R = sqrt(R2);
  const double nv[3] = {d[0] / R, d[1] / R, d[2] / R};
  const double c = -ri / rs;
  const double Rij[3] = {c * d[0], c * d[1], c * d[2]};
  const double vij[3] = {vi.x - vj.x, vi.y - vj.y, vi.z - vj.z};
  const double xi = rs - R;
  const double C3 = vij[0] * nv[0] + vij[1] * nv[1] + vij[2] * nv[2];
  const double Rbar = ri * rj / rs;
  const double mbar = 1.0 / (vi.w + vj.w);
  const double Kn = 2.0 / 3.0 * A.E * sqrt(Rbar * xi);
  const double C4 = Kn * xi - A.gamma2 * sqrt(mbar * Kn) * C3;
  const double Fn[3] = {nv[0] * C4, nv[1] * C4, nv[2] * C4};
  if (!(A.dt < 2.0 * sqrt(mbar / Kn))) ++B.bad;    // Cundall-Strack, kernelinline.hh:285-286
  const double F0 = sqrt(Fn[0] * Fn[0] + Fn[1] * Fn[1] + Fn[2] * Fn[2]);
  const double ws[3] = {wi.x + wj.x, wi.y + wj.y, wi.z + wj.z};
  double vt[3] = {vij[0] - C3 * nv[0], vij[1] - C3 * nv[1], vij[2] - C3 * nv[2]};
  vt[0] += ws[1] * Rij[2] - ws[2] * Rij[1];
  vt[1] += ws[2] * Rij[0] - ws[0] * Rij[2];
  vt[2] += ws[0] * Rij[1] - ws[1] * Rij[0];
  double Fs[3] = {0, 0, 0};
  if (vt[0] != 0 && vt[1] != 0 && vt[2] != 0) {   // as the reference, kernelinline.hh:296
    const double xsm = A.mu * A.s2 * xi;
    const double vn = sqrt(vt[0] * vt[0] + vt[1] * vt[1] + vt[2] * vt[2]);
    const double xs = h[0];
    const double v1 = -A.mu * F0 * ((xs < xsm) ? (xs / xsm) : 1.0) / vn;
    Fs[0] = v1 * vt[0];
    Fs[1] = v1 * vt[1];
    Fs[2] = v1 * vt[2];
    h[0] = xs + vn * A.dt;                        // history, owned by this row
  }
  const double Ts[3] = {Rij[1] * Fs[2] - Rij[2] * Fs[1], Rij[2] * Fs[0] - Rij[0] * Fs[2],
                        Rij[0] * Fs[1] - Rij[1] * Fs[0]};
  double Tr[3] = {0, 0, 0};
  if (wnz) {
    const double wn = sqrt(wi.x * wi.x + wi.y * wi.y + wi.z * wi.z);
    const double cr = -A.mu_r * ri * F0 / wn;
    Tr[0] = cr * wi.x;
    Tr[1] = cr * wi.y;
    Tr[2] = cr * wi.z;
  }
  const double Q = 2.0 - (double)J.move;
#pragma unroll
  for (int x = 0; x < 3; ++x) {
    B.f[x] += (Fn[x] + Fs[x]) * Q;
    B.t[x] += (Ts[x] + Tr[x]) * Q;
  }
}

// Linear spring-dashpot normal force with a tangential spring and a Coulomb
// cap (Cundall & Strack, Geotechnique 29 (1979) 47-65; no reference
// counterpart: the granular settle workload's law, behind the same calls as
// the Hertz law above).  Per contact, n = (r_i - r_j)/|r_ij|,
// delta = rad_i + rad_j - |r_ij|, 1/meff = minv_i + minv_j (0 for a fixed j):
//   Fn = (kn delta - 2 zeta sqrt(meff kn) v_ij.n) n
//   vt = tangential part of v_ij - (rad_i w_i + rad_j w_j) x n
//   s  = history projected on the tangent plane + vt dt, Ft = -kt s,
//        capped at mu |Fn| (the spring then follows the cap, s = -Ft/kt)
//   F_i += Fn + Ft, T_i += (-rad_i n) x Ft
// The history (3 doubles per contact) belongs to row i and is updated in
// place.
__device__ __forceinline__ void contact_linear(const DemForceArgs &A, DemBody &B, const DemOther &J, double *h) {
  const double4 &pi = B.p, &vi = B.v, &wi = B.w;
  const double ri = B.rad;
  const double4 &pj = J.p, &vj = J.v, &wj = J.w;
  const double rj = J.rad;
  const double d[3] = {pi.x - pj.x, pi.y - pj.y, pi.z - pj.z};
  const double R2 = d[0] * d[0] + d[1] * d[1] + d[2] * d[2];
  const double rs = ri + rj;
  if (!(R2 < rs * rs)) return;
  const double R = sqrt(R2);
  const double nv[3] = {d[0] / R, d[1] / R, d[2] / R};
  const double delta = rs - R;
  const double meff = 1.0 / (vi.w + (J.move ? vj.w : 0.0));
  const double gn = 2.0 * A.zeta * sqrt(meff * A.kn);
  if (!(A.dt < 2.0 * sqrt(meff / A.kn))) ++B.bad;
  const double vij[3] = {vi.x - vj.x, vi.y - vj.y, vi.z - vj.z};
  const double vn = vij[0] * nv[0] + vij[1] * nv[1] + vij[2] * nv[2];
  const double fn = A.kn * delta - gn * vn;
  const double W[3] = {ri * wi.x + rj * wj.x, ri * wi.y + rj * wj.y, ri * wi.z + rj * wj.z};
  const double Wxn[3] = {W[1] * nv[2] - W[2] * nv[1], W[2] * nv[0] - W[0] * nv[2],
                         W[0] * nv[1] - W[1] * nv[0]};
  const double h0 = h[0], h1 = h[1], h2 = h[2];
  const double hn = h0 * nv[0] + h1 * nv[1] + h2 * nv[2];
  double sp[3], ft[3];
  sp[0] = h0 - hn * nv[0] + (vij[0] - Wxn[0] - vn * nv[0]) * A.dt;
  sp[1] = h1 - hn * nv[1] + (vij[1] - Wxn[1] - vn * nv[1]) * A.dt;
  sp[2] = h2 - hn * nv[2] + (vij[2] - Wxn[2] - vn * nv[2]) * A.dt;
#pragma unroll
  for (int k = 0; k < 3; ++k) ft[k] = -A.kt * sp[k];
  const double ftm = sqrt(ft[0] * ft[0] + ft[1] * ft[1] + ft[2] * ft[2]);
  const double cap = A.mu * fabs(fn);
  if (ftm > cap) {
    const double c = cap / ftm;
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      ft[k] *= c;
      sp[k] = -ft[k] / A.kt;
    }
  }
  h[0] = sp[0];
  h[1] = sp[1];
  h[2] = sp[2];
  const double nxf[3] = {nv[1] * ft[2] - nv[2] * ft[1], nv[2] * ft[0] - nv[0] * ft[2],
                         nv[0] * ft[1] - nv[1] * ft[0]};
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    B.f[k] += fn * nv[k] + ft[k];
    B.t[k] += -ri * nxf[k];
  }
}

// ascending order of N registers (Batcher's odd-even merge sort)
template <int N>
__device__ __forceinline__ void sort_registers(uint32_t (&a)[DEM_ROWBUF]) {
#pragma unroll
  for (int p = 1; p < N; p *= 2)
#pragma unroll
    for (int k = p; k >= 1; k /= 2)
#pragma unroll
      for (int j = k % p; j <= N - 1 - k; j += 2 * k)
#pragma unroll
        for (int i = 0; i < k; ++i)
          if (i + j + k < N && (i + j) / (2 * p) == (i + j + k) / (2 * p)) {
            const uint32_t x = min(a[i + j], a[i + j + k]), y = max(a[i + j], a[i + j + k]);
            a[i + j] = x;
            a[i + j + k] = y;
          }
}

// The rows of the contact matrix, their history and the forces, one thread per
// particle in cell order: makeJlist_WithBlock2/4_F4 (kernelfuncs.cu:1120-1216),
// sortColIdx (:1262-1290), succeedPrevState (:1292-1309) and
// calcF_IJpairWithList_F4 (kerneltemplate.hh:135-168) in one pass.  F and T are
// overwritten (the reference clears both first, cudaParticleDEM.cu:168-169);
// padding slots are not visited (they stay zero).
// Bound by latency and uncoalesced reads (a particle has none to a dozen
// contacts).  A row that the counting scan kept whole is sorted in registers;
// longer rows (more touching neighbours than any sphere packing gives) are
// scanned again and sorted in memory.  A contact present in both matrices keeps
// its history (both rows are sorted); new ones start at 0.  LN lanes take every
// LN-th contact of a row (each walks the previous row by itself), and the sums
// are added in a fixed order.  Code is kept short (rolled loops): a wavefront
// passes most of it once, so its fetch counts.  Neighbouring workgroups share an
// XCD's L2.  A bed of 60,000 spheres of 6 contacts: 19 us with two lanes, 21 with
// one, 27 with four; 200,000 dispersed ones with almost none: 8.0 with two, 7.5 with
// one (9.3 stored in random order); fill, carry and force as kernels of their own
// took 31 and 16 us.
#define DEM_ROWS_BS 128
template <int LAW, int W, uint32_t LN>
__global__ void __launch_bounds__(DEM_ROWS_BS) k_dem_rows(DemGrid G, DemForceArgs A) {
  __shared__ uint32_t scol[DEM_ROWBUF][DEM_ROWS_BS];    // a row
  constexpr uint32_t HW = LAW == 1 ? 3u : 1u;
  const uint32_t tid = threadIdx.x, k = (pb_xcd_chunk<16>() * DEM_ROWS_BS + tid) / LN, sl = tid % LN;
  if (k >= G.n) return;                               // a particle's lanes leave together
  if (k == 0 && sl == 0) A.res[0] = A.row[G.n];
  const uint32_t s = G.perm[k], i = G.so[k];
  const uint32_t b = A.row[i], full = A.row[i + 1] - b;
  // rows past the capacity: redone
  const uint32_t e = min(b + full, G.cap), len = e > b ? e - b : 0u;
  DemBody B;
  if (len) {
    B.p = A.r[s];
    B.v = A.v[s];
    B.w = A.w[s];
    B.rad = A.rad[s];
    uint32_t p = 0, pe = 0;
    if (A.prow) {
      p = A.prow[i];
      pe = A.prow[i + 1];
    }
    const bool kept = full <= DEM_ROWBUF;   // the counting scan kept the whole row
    if (kept) {
      uint32_t a[DEM_ROWBUF];
      const uint4 *buf = reinterpret_cast<const uint4 *>(G.rowbuf + (size_t)i * DEM_ROWBUF);
#pragma unroll
      for (uint32_t x = 0; x < DEM_ROWBUF; x += 4) {
        const uint4 y = buf[x / 4];
        a[x] = x < full ? y.x : PB_NONE;
        a[x + 1] = x + 1 < full ? y.y : PB_NONE;
        a[x + 2] = x + 2 < full ? y.z : PB_NONE;
        a[x + 3] = x + 3 < full ? y.w : PB_NONE;
      }
      if (__ballot(full > 8) == 0ull) sort_registers<8>(a);
      else sort_registers<(int)DEM_ROWBUF>(a);
#pragma unroll
      for (uint32_t x = 0; x < DEM_ROWBUF; ++x) scol[x][tid] = a[x];
    } else if (sl == 0) {
      uint32_t m = b;
      dem_contacts<W>(G, k, scol, [&](uint32_t o) {
        if (m < e) A.col[m++] = o;
      });
      for (uint32_t x = b + 1; x < e; ++x) {
        const uint32_t v = A.col[x];
        uint32_t y = x;
        while (y > b && A.col[y - 1] > v) {
          A.col[y] = A.col[y - 1];
          --y;
        }
        A.col[y] = v;
      }
    }
    uint32_t pj = p < pe ? A.pcol[p] : PB_NONE;       // both rows ascend
    const uint32_t step = kept ? LN : 1u, first = kept || sl == 0 ? sl : len;
#pragma unroll 1
    for (uint32_t x = first; x < len; x += step) {
      const uint32_t j = kept ? scol[x][tid] : A.col[b + x];
      if (kept) A.col[b + x] = j;
      const DemOther J = dem_other(A, A.inv[j]);
      while (pj < j) {
        ++p;
        pj = p < pe ? A.pcol[p] : PB_NONE;
      }
      double h[HW];
#pragma unroll
      for (uint32_t y = 0; y < HW; ++y) h[y] = pj == j ? A.pval[(size_t)p * HW + y] : 0.0;
      if (LAW == 1) contact_linear(A, B, J, h);
      else contact_hertz(A, B, J, h);
#pragma unroll
      for (uint32_t y = 0; y < HW; ++y) A.val[(size_t)(b + x) * HW + y] = h[y];
    }
  }
#pragma unroll
  for (uint32_t o = 1; o < LN; o <<= 1) {
#pragma unroll
    for (int x = 0; x < 3; ++x) {
      B.f[x] += __shfl_xor(B.f[x], (int)o, PB_WAVE);
      B.t[x] += __shfl_xor(B.t[x], (int)o, PB_WAVE);
    }
  }
  if (sl == 0) {
    A.F[s] = make_double4(B.f[0], B.f[1], B.f[2], 0.0);
    A.T[s] = make_double4(B.t[0], B.t[1], B.t[2], 0.0);
  }
  if (B.bad) {
    atomicAdd(A.bad, B.bad);
    A.res[1] = 1u;
  }
}

__global__ void k_dem_inv(const uint32_t *orig, uint32_t n, uint32_t *inv) {
  const uint32_t s = blockIdx.x * blockDim.x + threadIdx.x;
  if (s < n && orig[s] != PB_NONE) inv[orig[s]] = s;
}

// propagateEulerianRotation_F4, kernelfuncs.cu:966-986
__global__ void k_rot_step(double4 *w, double4 *L, const double4 *T, const double *m0inv,
                           const uint8_t *move, uint32_t n, double dt) {
  const uint32_t s = blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= n) return;
  const double mv = (double)move[s];
  const double d = dt * mv, m0 = m0inv[s] * mv;
  double4 l = L[s];
  const double4 t = T[s];
  l.x += t.x * d;
  l.y += t.y * d;
  l.z += t.z * d;
  L[s] = l;
  w[s] = make_double4(l.x * m0, l.y * m0, l.z * m0, 0.0);
}

// m0inv = minv / (0.4 r0^2), cudaParticleRotation::setInertia (.cu:35-61)
__global__ void k_set_inertia(const double4 *v, const double *r0, uint32_t n, double *m0inv) {
  const uint32_t s = blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= n) return;
  const double r = r0[s];
  m0inv[s] = r > 0 ? v[s].w * (1.0 / (0.4 * r * r)) : 0.0;
}

// ------------------------------------------------------------------ host
// a radius per particle (r0, or r0_all for every one) in storage order
static int scatter_radius(pb_sys *s, const double *r0, double r0_all, double *dst,
                          const char *msg) {
  std::vector<double> all;
  if (!r0) {
    all.assign(s->n, r0_all);
    r0 = all.data();
  }
  for (size_t g = 0; g < s->n; ++g)
    if (!(r0[g] > 0)) return pb_fail(s->ctx, PB_ERR_ARG, msg);
  return pb_io_scatter(s, r0, dst, false);
}

static int upload_radius(pb_sys *s, const double *r0, double r0_all) {
  int rc = pb_ensure_radius(s);
  if (rc) return rc;
  if ((rc = scatter_radius(s, r0, r0_all, s->radius, "DEM: radius must be > 0"))) return rc;
  PB_HIP(s->ctx, hipStreamSynchronize(s->ctx->stream));
  return PB_OK;
}

// a change of contact law changes the history width: the contact matrices
// start again (as after the first set-up)
static void set_law(pb_sys *s, int law, uint32_t hw) {
  if (s->dem_hw != hw) {
    for (int b = 0; b < 2; ++b) {
      pb_free(s->cm_val[b]);
      s->cm_val[b] = nullptr;
      s->cm_cap[b] = 0;
      s->cm_nnz[b] = 0;
    }
    s->cm_cur = -1;
    s->cm_prev = false;
    s->cm_rewound = false;
  }
  s->dem_law = law;
  s->dem_hw = hw;
}

extern "C" int pb_dem_set_properties(pb_sys *s, double E, double mu, double sigma, double gamma,
                                     double mu_r, const double *r0, double r0_all) {
  if (!s) return PB_ERR_ARG;
  if (s->nrep != 1) return pb_fail(s->ctx, PB_ERR_ARG, "DEM: single replica only");
  if (!(sigma < 0.5)) return pb_fail(s->ctx, PB_ERR_ARG, "DEM: Poisson ratio must be < 0.5");
  PB_HIP(s->ctx, hipSetDevice(s->ctx->device));
  // cudaParticleDEM::setDEMProperties, cudaParticleDEM.cu:221-252
  s->dem_E = E * (1.0 - sigma * sigma);
  s->dem_mu = mu;
  s->dem_s2 = (2.0 - sigma) / 2.0 / (1.0 - sigma);
  s->dem_gamma2 = gamma;
  s->dem_mu_r = mu_r;
  if (int rc = upload_radius(s, r0, r0_all)) return rc;
  if (int rc = pb_ensure_rotation(s)) return rc;
  set_law(s, 0, 1);
  s->dem_set = true;
  return PB_OK;
}

extern "C" int pb_dem_set_linear(pb_sys *s, double kn, double e, double kt, double mu,
                                 const double *r0, double r0_all) {
  if (!s) return PB_ERR_ARG;
  if (s->nrep != 1) return pb_fail(s->ctx, PB_ERR_ARG, "DEM: single replica only");
  if (!(kn > 0) || !(kt > 0) || !(mu >= 0))
    return pb_fail(s->ctx, PB_ERR_ARG, "pb_dem_set_linear: need kn > 0, kt > 0, mu >= 0");
  if (!(e > 0 && e <= 1))
    return pb_fail(s->ctx, PB_ERR_ARG, "pb_dem_set_linear: restitution must be in (0, 1]");
  PB_HIP(s->ctx, hipSetDevice(s->ctx->device));
  const double le = std::log(e);
  s->dem_kn = kn;
  s->dem_kt = kt;
  s->dem_zeta = -le / std::sqrt(M_PI * M_PI + le * le);   // damping ratio of restitution e
  s->dem_mu = mu;
  if (int rc = upload_radius(s, r0, r0_all)) return rc;
  if (int rc = pb_ensure_rotation(s)) return rc;
  set_law(s, 1, 3);
  s->dem_set = true;
  return PB_OK;
}

extern "C" int pb_rot_set_inertia(pb_sys *s, const double *r0, double r0_all) {
  if (!s) return PB_ERR_ARG;
  PB_HIP(s->ctx, hipSetDevice(s->ctx->device));
  int rc = pb_ensure_rotation(s);
  if (rc) return rc;
  // the inertia radius may differ from the contact radius: it is staged in a
  // temporary device array in storage order
  double *d = nullptr;
  if ((rc = pb_alloc(s->ctx, &d, s->npad))) return rc;
  hipStream_t st = s->ctx->stream;
  rc = scatter_radius(s, r0, r0_all, d, "setInertia: radius must be > 0");
  if (!rc && !s->m0inv) rc = pb_alloc(s->ctx, &s->m0inv, s->npad);
  if (rc) {
    (void)hipStreamSynchronize(st);
    pb_free(d);
    return rc;
  }
  hipLaunchKernelGGL(k_set_inertia, dim3(pb_blocks(s->npad, 256)), dim3(256), 0, st, s->v, d,
                     s->npad, s->m0inv);
  hipError_t e = hipGetLastError();
  if (e == hipSuccess) e = hipMemsetAsync(s->w, 0, sizeof(double4) * s->npad, st);
  if (e == hipSuccess) e = hipMemsetAsync(s->Lm, 0, sizeof(double4) * s->npad, st);
  if (e == hipSuccess) e = hipStreamSynchronize(st);
  pb_free(d);
  if (e != hipSuccess) return pb_hip_check(s->ctx, e, "pb_rot_set_inertia");
  return PB_OK;
}

extern "C" int pb_rot_step(pb_sys *s, double dt) {
  if (!s) return PB_ERR_ARG;
  if (!s->m0inv) return pb_fail(s->ctx, PB_ERR_STATE, "rotation: pb_rot_set_inertia first");
  hipLaunchKernelGGL(k_rot_step, dim3(pb_blocks(s->npad, 256)), dim3(256), 0, s->ctx->stream,
                     s->w, s->Lm, s->T, s->m0inv, s->move, s->npad, dt);
  PB_LAUNCH_CHECK(s->ctx, "k_rot_step");
  return PB_OK;
}

static int ensure_csr(pb_sys *s, int b, uint32_t nnz) {
  int rc;
  if (!s->cm_row[b] && (rc = pb_alloc(s->ctx, &s->cm_row[b], (size_t)s->n + 1))) return rc;
  if (s->cm_cap[b] < nnz || !s->cm_cap[b]) {
    const uint32_t cap = (uint32_t)std::min<uint64_t>(((uint64_t)nnz * 5 / 4 + 512), 0xFFFFFFFFull);
    // the matrix that the arrays held is gone, also if the new ones can't be had
    s->cm_cap[b] = 0;
    if (s->cm_cur == b) s->cm_cur = -1;
    s->cm_prev = false;
    if ((rc = pb_alloc(s->ctx, &s->cm_col[b], cap)) ||
        (rc = pb_alloc(s->ctx, &s->cm_val[b], (size_t)cap * s->dem_hw)))
      return rc;
    s->cm_cap[b] = cap;
  }
  return PB_OK;
}

// lanes a particle in k_dem_rows: two while one leaves SIMDs without a wavefront
static uint32_t dem_lanes(uint32_t n) {
  return n <= 98304u ? 2u : 1u;
}

template <int LAW>
static void (*dem_rows_kernel(bool single, uint32_t ln))(DemGrid, DemForceArgs) {
  if (ln == 2) return single ? k_dem_rows<LAW, 2, 2> : k_dem_rows<LAW, 1, 2>;
  return single ? k_dem_rows<LAW, 2, 1> : k_dem_rows<LAW, 1, 1>;
}

extern "C" int pb_dem_calc_force(pb_sys *s, double dt, int autotune, uint32_t *nnz_out) {
  if (!s) return PB_ERR_ARG;
  if (!s->dem_set) return pb_fail(s->ctx, PB_ERR_STATE, "DEM properties not set");
  if (!s->ref_binned) return pb_fail(s->ctx, PB_ERR_STATE, "DEM: pb_bin (calcBlockID) first");
  PB_HIP(s->ctx, hipSetDevice(s->ctx->device));
  hipStream_t st = s->ctx->stream;
  const uint32_t n = s->n;
  int rc;
  if (!s->dem_rs) {
    if ((rc = pb_alloc(s->ctx, &s->dem_inv, (size_t)n + 1)) ||
        (rc = pb_alloc(s->ctx, &s->dem_rowbuf, (size_t)s->npad * DEM_ROWBUF)) ||
        (rc = pb_alloc(s->ctx, &s->dem_fq, s->npad)) || (rc = pb_alloc(s->ctx, &s->dem_rs, s->npad)))
      return rc;
  }
  if (s->dem_inv_order != s->order_gen) {
    hipLaunchKernelGGL(k_dem_inv, dim3(pb_blocks(s->npad, 256)), dim3(256), 0, st, s->orig, s->npad,
                       s->dem_inv);
    PB_LAUNCH_CHECK(s->ctx, "k_dem_inv");
    s->dem_inv_order = s->order_gen;
  }
  DemView V;
  double span = 0.0;
  for (int a = 0; a < 3; ++a) {
    V.lo[a] = s->blocklen[3 + a];
    span = std::max(span, (s->blocknum[a] + 1.0) * s->blocklen[a]);
  }
  V.span = span < 1e18 ? (float)span : -1.f;  // squares outside FP32: every pair exactly
  hipLaunchKernelGGL(k_dem_gather, dim3(pb_blocks(n, 256)), dim3(256), 0, st, s->perm, s->r,
                     s->radius, n, V, s->dem_rs, s->dem_fq);
  DemGrid G;
  G.perm = s->perm;
  G.bid = s->ref_bid;
  G.cstart = s->cstart;
  G.rs = s->dem_rs;
  G.fq = s->dem_fq;
  G.so = s->ref_pid;
  G.rowbuf = s->dem_rowbuf;
  G.move = s->move;
  for (int a = 0; a < 3; ++a) G.nb[a] = s->blocknum[a];
  G.n = n;
  const int b = (s->cm_cur + 1) & 1;         // the other buffer keeps the previous matrix
  // capacity from the previous matrix (ensure_csr adds a quarter)
  if ((rc = ensure_csr(s, b, s->cm_cur >= 0 ? s->cm_nnz[s->cm_cur] : 0))) return rc;
  G.cap = s->cm_cap[b];
  s->cm_prev = false;                        // the other buffer is overwritten from here on
  // per-row counts go to the sort workspace's rank array (free once pb_bin
  // has produced perm / cstart), their exclusive scan to the new row array
  uint32_t *cnt = s->rank, *bad = s->d_counter + 8;
  const bool single = s->ref_single != 0;    // 125 cells of one particle, else 27
  hipLaunchKernelGGL(single ? k_dem_count<2> : k_dem_count<1>, dim3(pb_blocks(n, 256)), dim3(256), 0,
                     st, G, cnt, bad);
  PB_LAUNCH_CHECK(s->ctx, "k_dem_count");
  if ((rc = pb_exclusive_scan(s, cnt, s->cm_row[b], n))) return rc;
  const int p = s->cm_cur;
  DemForceArgs A;
  A.inv = s->dem_inv;
  A.prow = p >= 0 ? s->cm_row[p] : nullptr;
  A.pcol = p >= 0 ? s->cm_col[p] : nullptr;
  A.pval = p >= 0 ? s->cm_val[p] : nullptr;
  A.r = s->r;
  A.v = s->v;
  A.w = s->w;
  A.rad = s->radius;
  A.move = s->move;
  A.F = s->F;
  A.T = s->T;
  A.bad = bad;
  A.E = s->dem_E;
  A.mu = s->dem_mu;
  A.s2 = s->dem_s2;
  A.gamma2 = s->dem_gamma2;
  A.mu_r = s->dem_mu_r;
  A.dt = dt;
  A.kn = s->dem_kn;
  A.zeta = s->dem_zeta;
  A.kt = s->dem_kt;
  A.res = (uint32_t *)s->ctx->res_dev;
  const uint32_t ln = dem_lanes(n);
  auto rows = s->dem_law == 1 ? dem_rows_kernel<1>(single, ln) : dem_rows_kernel<0>(single, ln);
  // rows, history and forces up to the capacity; that kernel reports nnz and
  // whether the time-step check failed (its count is fetched only then)
  uint32_t nnz = 0, nbad = 0;
  auto contacts_and_force = [&]() -> int {
    G.cap = s->cm_cap[b];
    A.row = s->cm_row[b];
    A.col = s->cm_col[b];
    A.val = s->cm_val[b];
    volatile uint32_t *res = (volatile uint32_t *)s->ctx->res;
    res[1] = 0;
    hipLaunchKernelGGL(rows, dim3(pb_blocks(n, DEM_ROWS_BS / ln)), dim3(DEM_ROWS_BS), 0, st, G, A);
    PB_LAUNCH_CHECK(s->ctx, "k_dem_rows");
    PB_HIP(s->ctx, hipStreamSynchronize(st));
    nnz = res[0];
    nbad = 0;
    return res[1] ? pb_io_download(s->ctx, &nbad, bad, sizeof(nbad)) : PB_OK;
  };
  if ((rc = contacts_and_force())) return rc;
  if (nnz > s->cm_cap[b]) {                  // the matrix outgrew the arrays: again, larger
    hipLaunchKernelGGL(k_fill_u32, dim3(1), dim3(64), 0, st, bad, 1u, 0u);
    if ((rc = ensure_csr(s, b, nnz)) || (rc = contacts_and_force())) return rc;
  }
  s->cm_nnz[b] = nnz;
  s->cm_prev = p >= 0;
  s->cm_rewound = false;
  s->cm_cur = b;
  s->dem_bad = nbad;
  if (nnz_out) *nnz_out = nnz;
  if (nbad && !autotune)
    return pb_fail(s->ctx, PB_ERR_DT, "DEM: time step above the Cundall-Strack bound 2 sqrt(m/Kn)");
  return PB_OK;
}

extern "C" int pb_dem_get_contacts(pb_sys *s, uint32_t *rowptr, uint32_t *colidx, double *val,
                                   uint32_t cap, uint32_t *nnz) {
  if (!s) return PB_ERR_ARG;
  if (s->cm_cur < 0) return pb_fail(s->ctx, PB_ERR_STATE, "DEM: no contact matrix yet");
  const int b = s->cm_cur;
  const uint32_t z = s->cm_nnz[b];
  if (nnz) *nnz = z;
  hipStream_t st = s->ctx->stream;
  if (rowptr)
    PB_HIP(s->ctx, hipMemcpyAsync(rowptr, s->cm_row[b], 4 * ((size_t)s->n + 1),
                                  hipMemcpyDeviceToHost, st));
  if ((colidx || val) && z > cap)
    return pb_fail(s->ctx, PB_ERR_ARG, "pb_dem_get_contacts: capacity below nnz");
  if (colidx && z)
    PB_HIP(s->ctx, hipMemcpyAsync(colidx, s->cm_col[b], 4 * (size_t)z, hipMemcpyDeviceToHost, st));
  if (val && z)
    PB_HIP(s->ctx, hipMemcpyAsync(val, s->cm_val[b], 8 * (size_t)z * s->dem_hw,
                                  hipMemcpyDeviceToHost, st));
  PB_HIP(s->ctx, hipStreamSynchronize(st));
  return PB_OK;
}

extern "C" int pb_dem_set_contacts(pb_sys *s, const uint32_t *rowptr, const uint32_t *colidx,
                                   const double *val, uint32_t nnz) {
  if (!s || !rowptr || (nnz && (!colidx || !val))) return PB_ERR_ARG;
  const uint32_t n = s->n;
  // a CSR the history merge can read: rows of original indices, columns
  // ascending and in range
  if (rowptr[0] != 0 || rowptr[n] != nnz)
    return pb_fail(s->ctx, PB_ERR_ARG, "pb_dem_set_contacts: rowptr does not span nnz");
  for (uint32_t i = 0; i < n; ++i) {
    if (rowptr[i + 1] < rowptr[i])
      return pb_fail(s->ctx, PB_ERR_ARG, "pb_dem_set_contacts: rowptr decreases");
    for (uint32_t k = rowptr[i]; k < rowptr[i + 1]; ++k)
      if (colidx[k] >= n || (k > rowptr[i] && colidx[k] <= colidx[k - 1]))
        return pb_fail(s->ctx, PB_ERR_ARG, "pb_dem_set_contacts: columns out of range or unsorted");
  }
  const int b = s->cm_cur < 0 ? 0 : s->cm_cur;
  if (int rc = ensure_csr(s, b, nnz)) return rc;
  hipStream_t st = s->ctx->stream;
  PB_HIP(s->ctx, hipMemcpyAsync(s->cm_row[b], rowptr, 4 * ((size_t)n + 1), hipMemcpyHostToDevice, st));
  if (nnz) {
    PB_HIP(s->ctx, hipMemcpyAsync(s->cm_col[b], colidx, 4 * (size_t)nnz, hipMemcpyHostToDevice, st));
    PB_HIP(s->ctx, hipMemcpyAsync(s->cm_val[b], val, 8 * (size_t)nnz * s->dem_hw,
                                  hipMemcpyHostToDevice, st));
  }
  PB_HIP(s->ctx, hipStreamSynchronize(st));
  s->cm_nnz[b] = nnz;
  s->cm_cur = b;
  s->cm_prev = false;                        // the other buffer is not its predecessor
  s->cm_rewound = false;
  return PB_OK;
}

// cudaParticleDEM::rollback's `_N -= 1` (cudaParticleDEM.cu:302-306): the
// matrix before the latest becomes the latest again, so the next
// pb_dem_calc_force overwrites the discarded one and carries the history
// of the step before it.  When the latest matrix has no predecessor (the
// first call, or a matrix restored by pb_dem_set_contacts) the next call
// starts every contact at zero history, as the reference's cleared second
// matrix gives.  Only one earlier step is kept, so a second rewind without a
// pb_dem_calc_force in between is refused.
extern "C" int pb_dem_rewind(pb_sys *s) {
  if (!s) return PB_ERR_ARG;
  if (s->cm_rewound)
    return pb_fail(s->ctx, PB_ERR_STATE, "pb_dem_rewind: already rewound (one step is kept)");
  if (s->cm_cur < 0)
    return pb_fail(s->ctx, PB_ERR_STATE, "pb_dem_rewind: no contact matrix to rewind");
  s->cm_cur = s->cm_prev ? (s->cm_cur ^ 1) : -1;
  s->cm_prev = false;
  s->cm_rewound = true;
  return PB_OK;
}

extern "C" int pb_dem_history_width(pb_sys *s, uint32_t *hw) {
  if (!s || !hw) return PB_ERR_ARG;
  *hw = s->dem_hw;
  return PB_OK;
}

extern "C" int pb_dem_last_violations(pb_sys *s, uint32_t *count) {
  if (!s || !count) return PB_ERR_ARG;
  *count = s->dem_bad;
  return PB_OK;
}
