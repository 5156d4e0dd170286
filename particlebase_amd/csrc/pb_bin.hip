// pb_bin.hip -- the integer-output paths that must match the reference bit
// for bit: cell ids (calcBID_F4), the cell sort (calcBlockID), neighbour
// counts (calcCoordMD_F4) and g(r) histograms (calcGR_F4).  This file is
// compiled with -ffp-contract=off: every FP32 operation is rounded exactly as
// the reference's source orders it (division and sqrt correctly rounded).
#include "pb_internal.h"
#include <cmath>
#include <cstring>
#include <type_traits>

// CUDA's float->uint conversion saturates; calcBID_F4 relies on it.
__device__ __host__ __forceinline__ uint32_t f2u_sat(float q) {
  if (!(q > 0.0f)) return 0u;
  if (q >= 4294967296.0f) return 0xFFFFFFFFu;
  return (uint32_t)q;
}
__device__ __forceinline__ uint32_t clamp_axis(uint32_t d, uint32_t c) {
  // kernelfuncs.cu:821-835
  return (d == c) ? c - 1 : ((d > c) ? 0u : d);
}

// distance2p, kernelinline.hh:47-62
__device__ __forceinline__ float distance2p(float r1x, float r1y, float r1z, float r2x,
                                            float r2y, float r2z, float cx, float cy, float cz) {
  r1x -= r2x;
  r1y -= r2y;
  r1z -= r2z;
  r1x *= r1x;
  r1y *= r1y;
  r1z *= r1z;
  if (r1x > cx) r1x += 4.0f * (cx - sqrtf(cx * r1x));
  if (r1y > cy) r1y += 4.0f * (cy - sqrtf(cy * r1y));
  if (r1z > cz) r1z += 4.0f * (cz - sqrtf(cz * r1z));
  return r1x + r1y + r1z;
}

struct RefGrid {
  float len[3], lo[3];
  uint32_t nb[3];
};

// calcBID_F4, kernelfuncs.cu:807-841; padding slots go to the extra cell
// ncell so they sort after every real particle.  The cell's particles are
// counted in the same pass.
__global__ void k_ref_bid(const double4 *r, const uint32_t *orig, uint32_t n, RefGrid g,
                          uint32_t ncell, uint32_t *cellid, uint32_t *counts, uint32_t *rank) {
  const uint32_t s = blockIdx.x * blockDim.x + threadIdx.x;
  const bool valid = s < n;
  uint32_t c = PB_NONE;
  if (valid) {
    c = ncell;
    if (orig[s] != PB_NONE) {
      const double4 p = r[s];
      const float x = (float)p.x, y = (float)p.y, z = (float)p.z;
      const uint32_t d0 = clamp_axis(f2u_sat((x - g.lo[0]) / g.len[0]), g.nb[0]);
      const uint32_t d1 = clamp_axis(f2u_sat((y - g.lo[1]) / g.len[1]), g.nb[1]);
      const uint32_t d2 = clamp_axis(f2u_sat((z - g.lo[2]) / g.len[2]), g.nb[2]);
      c = d2 + d1 * g.nb[2] + d0 * g.nb[1] * g.nb[2];
    }
    cellid[s] = c;
  }
  const uint32_t k = pb_count_rank(c, valid, counts);
  if (valid) rank[s] = k;
}

static void host_neighbor_table(const uint32_t bn[3], int w, int periodic, uint32_t *table) {
  // calc_BlockNeighbor, cudaCutoffBlock.cu:17-65
  const long bx = bn[0], by = bn[1], bz = bn[2];
  const int J = (2 * w + 1) * (2 * w + 1) * (2 * w + 1);
  for (long i = 0; i < bx; ++i)
    for (long j = 0; j < by; ++j)
      for (long k = 0; k < bz; ++k) {
        const long I = k + j * bz + i * bz * by;
        int L = 0;
        for (int i1 = -w; i1 < w + 1; ++i1)
          for (int j1 = -w; j1 < w + 1; ++j1)
            for (int k1 = -w; k1 < w + 1; ++k1) {
              long i2 = i + i1, j2 = j + j1, k2 = k + k1;
              if (i2 == bx) i2 = 0;
              if (j2 == by) j2 = 0;
              if (k2 == bz) k2 = 0;
              if (i2 == -1) i2 = bx - 1;
              if (j2 == -1) j2 = by - 1;
              if (k2 == -1) k2 = bz - 1;
              if (i2 == bx + 1) i2 = 1;
              if (j2 == by + 1) j2 = 1;
              if (k2 == bz + 1) k2 = 1;
              if (i2 == -2) i2 = bx - 2;
              if (j2 == -2) j2 = by - 2;
              if (k2 == -2) k2 = bz - 2;
              uint32_t v = PB_NONE;
              if (periodic || ((i + i1) >= 0 && (i + i1) < bx && (j + j1) >= 0 && (j + j1) < by &&
                               (k + k1) >= 0 && (k + k1) < bz))
                v = (uint32_t)(k2 + j2 * bz + i2 * bz * by);
              table[I * J + L++] = v;
            }
      }
}

extern "C" int pb_setup_cells(pb_sys *s, float rmax, int periodic, int single_particle) {
  if (!s) return PB_ERR_ARG;
  if (s->nrep != 1) return pb_fail(s->ctx, PB_ERR_ARG, "pb_setup_cells: single replica only");
  if (!s->cell_set) return pb_fail(s->ctx, PB_ERR_STATE, "pb_setup_cells: cell not set");
  if (!(rmax > 0)) return pb_fail(s->ctx, PB_ERR_ARG, "pb_setup_cells: rmax <= 0");
  // cudaCutoffBlock::setupCutoffBlock, cudaCutoffBlock.cu:97-141 (FP32)
  float cell[6];
  for (int i = 0; i < 6; ++i) cell[i] = (float)s->cells[i];
  float c[3];
  uint32_t num[3];               // the system's grid only when all is known to be good
  float len[6];
  for (int i = 0; i < 3; ++i) {
    c[i] = cell[i * 2 + 1] - cell[i * 2];
    if (periodic) {
      num[i] = f2u_sat(c[i] / rmax);
      if (num[i] == 0) return pb_fail(s->ctx, PB_ERR_CELLS, "pb_setup_cells: box smaller than rmax");
      len[i] = c[i] / (float)num[i];
    } else {
      len[i] = rmax;
      num[i] = f2u_sat(c[i] / rmax) + 1u;
    }
    if (num[i] <= 2)
      return pb_fail(s->ctx, PB_ERR_CELLS, "pb_setup_cells: fewer than 3 cells along an axis");
    len[i + 3] = cell[i * 2];
  }
  if (single_particle) {
    // cudaCutoffBlock.cu:115-138: shrink cells until the cell diagonal is
    // below the particle diameter (r0 = rmax*sqrt(3)/2)
    const double r0 = rmax * sqrt(3.0) / 2.0;
    const double R02 = (r0 * 2.0) * (r0 * 2.0);
    while ((double)(len[0] * len[0] + len[1] * len[1] + len[2] * len[2]) > R02) {
      if ((len[0] > len[1]) && (len[0] > len[2])) {
        ++num[0];
        len[0] = c[0] / num[0];
      } else if (len[1] > len[2]) {
        ++num[1];
        len[1] = c[1] / num[1];
      } else {
        ++num[2];
        len[2] = c[2] / num[2];
      }
    }
  }
  const uint64_t nc = (uint64_t)num[0] * num[1] * num[2];
  if (nc >= 0x7FFFFFFFull) return pb_fail(s->ctx, PB_ERR_CELLS, "pb_setup_cells: too many cells");
  s->ref_cells = s->ref_binned = false;
  std::memcpy(s->blocknum, num, sizeof(num));
  std::memcpy(s->blocklen, len, sizeof(len));
  s->ref_ncell = (uint32_t)nc;
  s->ref_periodic = periodic ? 1 : 0;
  s->ref_single = single_particle ? 1 : 0;
  int rc;
  if ((rc = pb_alloc(s->ctx, &s->ref_bid, s->npad)) || (rc = pb_alloc(s->ctx, &s->ref_pid, s->npad)) ||
      (rc = pb_alloc(s->ctx, &s->ref_bindex, (size_t)s->ref_ncell + 1)))
    return rc;
  if ((rc = pb_ensure_sort_ws(s, s->ref_ncell + 1))) return rc;
  s->ref_cells = true;
  return PB_OK;
}

extern "C" int pb_get_cell_info(pb_sys *s, uint32_t blocknum[3], float blocklen[6]) {
  if (!s || !s->ref_cells) return pb_fail(s ? s->ctx : nullptr, PB_ERR_STATE, "no cells");
  if (blocknum) std::memcpy(blocknum, s->blocknum, sizeof(s->blocknum));
  if (blocklen) std::memcpy(blocklen, s->blocklen, sizeof(s->blocklen));
  return PB_OK;
}

extern "C" int pb_get_neighbor_table(pb_sys *s, uint32_t *table) {
  if (!s || !table) return PB_ERR_ARG;
  if (!s->ref_cells) return pb_fail(s->ctx, PB_ERR_STATE, "no cells");
  host_neighbor_table(s->blocknum, s->ref_single ? 2 : 1, s->ref_periodic, table);
  return PB_OK;
}

static RefGrid ref_grid(const pb_sys *s) {
  RefGrid g;
  for (int a = 0; a < 3; ++a) {
    g.len[a] = s->blocklen[a];
    g.lo[a] = s->blocklen[3 + a];
    g.nb[a] = s->blocknum[a];
  }
  return g;
}

extern "C" int pb_bin(pb_sys *s) {
  if (!s) return PB_ERR_ARG;
  if (!s->ref_cells) return pb_fail(s->ctx, PB_ERR_STATE, "pb_bin: pb_setup_cells first");
  hipStream_t st = s->ctx->stream;
  const uint32_t nc = s->ref_ncell;
  int rc;
  if ((rc = pb_ensure_sort_ws(s, nc + 1)) || (rc = pb_counts_begin(s))) return rc;
  hipLaunchKernelGGL(k_ref_bid, dim3(pb_blocks(s->npad, 256)), dim3(256), 0, st, s->r, s->orig,
                     s->npad, ref_grid(s), nc, s->cellid, s->ccount, s->rank);
  PB_LAUNCH_CHECK(s->ctx, "k_ref_bid");
  PbCellOrder O;
  if ((rc = pb_counting_sort(s, nc + 1, s->orig, &O)) || (rc = pb_cell_order(s, O, nc))) return rc;
  s->ref_binned = true;
  return PB_OK;
}

extern "C" int pb_get_bins(pb_sys *s, uint32_t *pid, uint32_t *bid_sorted, uint32_t *bindex) {
  if (!s) return PB_ERR_ARG;
  if (!s->ref_binned) return pb_fail(s->ctx, PB_ERR_STATE, "pb_get_bins: pb_bin first");
  hipStream_t st = s->ctx->stream;
  if (pid) PB_HIP(s->ctx, hipMemcpyAsync(pid, s->ref_pid, 4 * (size_t)s->n, hipMemcpyDeviceToHost, st));
  if (bid_sorted)
    PB_HIP(s->ctx, hipMemcpyAsync(bid_sorted, s->ref_bid, 4 * (size_t)s->n, hipMemcpyDeviceToHost, st));
  if (bindex)
    PB_HIP(s->ctx, hipMemcpyAsync(bindex, s->ref_bindex, 4 * ((size_t)s->ref_ncell + 1),
                                  hipMemcpyDeviceToHost, st));
  PB_HIP(s->ctx, hipStreamSynchronize(st));
  return PB_OK;
}

static void half_cell2(const pb_sys *s, uint32_t q, float c[3]) {
  // cudaFrame::setCell, cudaFrame.cu:85-91, on the FP32 cell values
  for (int a = 0; a < 3; ++a) {
    const float lo = (float)s->cells[6 * q + 2 * a], hi = (float)s->cells[6 * q + 2 * a + 1];
    c[a] = (hi - lo) / 2;
    c[a] *= c[a];
  }
}

// ------------------------------------------------------------------ g(r)
// All unordered pairs of every replica (the pair set of
// calcF_IJpairWithBlock5_F4 over makePairInfo's tiles, kerneltemplate.hh:
// 423-512, cudaCalcGR.cu:30-84), binned by calcGR_F4 (kernelinline.hh:
// 440-448).  A work item is a slice (1/1 to 1/8) of the j particles of one of
// the triangular pairs of 256-particle tiles; a workgroup takes consecutive
// items, so it stays with a replica and flushes its LDS histogram seldom.
// Integer sums: the result is independent of the order.
//
// Bound by VALU issue.  The reference's rounding (per axis
// d2 + 4 (c - sqrt(c d2)) with correctly rounded roots, then sqrt and a
// double-precision bin) takes 102 instructions a pair; but the bin is decided
// by far less unless the distance lies next to a bin boundary.  So a lane
// computes r from the folded axes min(|d|, ||d| - L|) and the hardware rsqrt
// (26 instructions), with a bound on how far its bin coordinate t can be from
// the reference's, and counts the pair when no boundary (an integer t) lies
// within the bound.  The others -- about 1 % at 200 bins -- go to a queue in
// LDS that the wavefront works off 64 at a time with the reference's exact
// arithmetic.  The bound, with u = 2^-24 and c the squared half edges:
//   the reference's sum is within (34 + 5) u (cx + cy + cz) of the exact fold
//   of the same d (the root's 20 u c, c - root, d2 and sum roundings, for
//   |d| <= 1.25 L), this one within (8 + 8 + 3) u (cx + cy + cz) (the rounding
//   of L and |d| - L, the other side of the fold test, the sum), together
//   below E = 64 u (cx + cy + cz) (largest difference seen in 6e7 random
//   pairs: 0.23 E).  So t differs by at most K / (t - 0.5), K = rstepinv^2 E,
//   plus k0 = 2^-20 (rnum + 2) for the relative errors of rsqrt and products.
// Particles further than L / 8 outside the box (or not finite) and bins finer
// than the bound void it: those tile pairs take the exact arithmetic.
// 256 replicas, 7.17e9 pairs, 200 bins: 13.4 ms before, 4.1 ms now.  (The
// fold by 32-bit box fractions, one subtraction and one conversion an axis,
// took 5.5 ms: conversions issue slowly.  Copies of the histogram against
// atomics on one LDS address changed nothing.)
#define GR_T 256
#define GR_MAX_SLICES 8u
// A tile pair adds at most GR_T * GR_T = 2^16 pairs to one bin of the
// workgroup's uint32 LDS histogram; flushing at least every 2^14 work items
// keeps every bin and the pair count below 2^31, whatever the replica's size.
#define GR_FLUSH_TILES 16384u
struct GrRep {
  uint32_t atom0, natoms, ntile;
  uint64_t pair0;      // first tile-pair index of this replica
  float cx, cy, cz, rstepinv;
  float lo[3], hi[3];  // FP32 box
};

// the reference's bin of a pair (0: dropped), calcGR_F4
__device__ __forceinline__ uint32_t gr_bin(const float4 &pi, const float4 &pj, const GrRep &R,
                                           uint32_t rnum) {
  const float R2 = distance2p(pi.x, pi.y, pi.z, pj.x, pj.y, pj.z, R.cx, R.cy, R.cz);
  const float r0 = sqrtf(R2) * R.rstepinv;
  const double tt = (double)r0 + 0.5;
  return (tt < (double)rnum) ? (uint32_t)tt : 0u;
}

// Bin 0 (the pairs the reference drops: r < dr/2 and r beyond the last bin,
// about half of all pairs in a periodic box) is what is left of the items'
// pairs when a histogram is flushed.
__global__ void __launch_bounds__(GR_T) k_gr(const double4 *r, const GrRep *reps, uint32_t nrep,
                                             uint64_t nitem, uint32_t slices, uint32_t rnum,
                                             uint64_t *hist) {
  extern __shared__ uint32_t h[];
  __shared__ float4 ti[GR_T], tj[GR_T + 4];   // 4: read, not used, by the last group of j
  __shared__ uint32_t queue[GR_T / 64][5 * 64];   // fewer than 64, and a group's 4 x 64
  __shared__ uint32_t binned;
  const uint32_t tid = threadIdx.x, lane = pb_lane(), wave = tid / 64;
  for (uint32_t b = tid; b < rnum; b += GR_T) h[b] = 0;
  if (tid == 0) binned = 0;
  const uint64_t per = (nitem + gridDim.x - 1) / gridDim.x;
  const uint64_t w0 = (uint64_t)blockIdx.x * per, w1 = min(w0 + per, nitem);
  uint32_t pairs = 0, since = 0;           // of the items in the LDS histogram
  uint32_t rep = 0;
  for (uint64_t w = w0; w < w1; ++w) {     // block-uniform
    const uint64_t p = w / slices;
    const uint32_t slice = (uint32_t)(w % slices);
    if (w == w0 || (rep + 1 < nrep && p >= reps[rep + 1].pair0)) {
      uint32_t lo = rep, hi = nrep;
      while (hi - lo > 1) {
        const uint32_t mid = (lo + hi) / 2;
        if (reps[mid].pair0 <= p) lo = mid;
        else hi = mid;
      }
      rep = lo;
    }
    const GrRep R = reps[rep];
    // triangular index t -> (it <= jt): row it starts at it ntile - it (it - 1) / 2
    const uint64_t t = p - R.pair0;
    const double b2 = 2.0 * R.ntile + 1.0;
    uint32_t it = (uint32_t)(0.5 * (b2 - sqrt(fmax(b2 * b2 - 8.0 * (double)t, 0.0))));
    auto row0 = [&](uint32_t k) { return (uint64_t)k * R.ntile - (uint64_t)k * (k - 1) / 2; };
    it = min(it, R.ntile - 1u);
    while (it > 0 && row0(it) > t) --it;
    while (it + 1 < R.ntile && row0(it + 1) <= t) ++it;
    const uint32_t jt = it + (uint32_t)(t - row0(it));
    const uint32_t ni = min(GR_T, R.natoms - it * GR_T), nj = min(GR_T, R.natoms - jt * GR_T);
    const uint32_t j0 = min(nj, slice * (GR_T / slices)), j1 = min(nj, j0 + GR_T / slices);
    const bool diag = it == jt;
    pairs += diag ? (j1 * j1 - j1 - (j0 * j0 - j0)) / 2u : ni * (j1 - j0);
    const float L[3] = {R.hi[0] - R.lo[0], R.hi[1] - R.lo[1], R.hi[2] - R.lo[2]};
    __syncthreads();                       // the tiles of the item before are consumed
    // FP32 position of a particle; whether the bound holds for it
    auto load = [&](uint32_t k, float4 &q) {
      const double4 x = r[R.atom0 + k];
      q = make_float4((float)x.x, (float)x.y, (float)x.z, 0.f);
      const float c[3] = {q.x, q.y, q.z};
      bool in = true;
#pragma unroll
      for (int a = 0; a < 3; ++a) {
        const float s = 0.125f * L[a];
        in = in && c[a] >= R.lo[a] - s && c[a] <= R.hi[a] + s;
      }
      return in;
    };
    float4 pi = make_float4(0.f, 0.f, 0.f, 0.f);
    const float K = R.rstepinv * R.rstepinv * (64.0f * 5.9604645e-8f * 1.0001f) * (R.cx + R.cy + R.cz);
    bool ok = K < 0.25f * (float)rnum;
    if (tid < ni) {
      ok = load(it * GR_T + tid, pi) && ok;
      ti[tid] = pi;
    }
    if (tid >= j0 && tid < j1) ok = load(jt * GR_T + tid, tj[tid]) && ok;
    if (!__syncthreads_and(ok)) {
      if (tid < ni)
        for (uint32_t jj = diag ? max(j0, tid + 1) : j0; jj < j1; ++jj) {
          const uint32_t bin = gr_bin(pi, tj[jj], R, rnum);
          if (bin) atomicAdd(&h[bin], 1u);
        }
    } else {
      const float sc = R.rstepinv, ke = -K / sc;
      const float k0 = 0.5f - 9.5367432e-7f * (float)(rnum + 2u);
      const float tin = (float)rnum, tout = (float)(rnum + 1u);
      const uint32_t first = tid >= ni ? GR_T : (diag ? tid + 1u : 0u);
      uint32_t qn = 0;                     // queued pairs (wave-uniform)
      auto work_off = [&](uint32_t n) {    // the last n <= 64 queued pairs, exactly
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
        if (lane < n) {
          const uint32_t e = queue[wave][qn - n + lane];
          const uint32_t bin = gr_bin(ti[e >> 16], tj[e & 0xFFFFu], R, rnum);
          if (bin) atomicAdd(&h[bin], 1u);
        }
        qn -= n;
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
      };
      // four consecutive j: their loads and arithmetic interleave, and one
      // branch asks whether any lane has a pair for the queue
      auto four = [&](uint32_t jj, auto masked) {
        constexpr uint32_t U = 4;
        bool slow[U], any = false;
#pragma unroll
        for (uint32_t u = 0; u < U; ++u) {
          const float4 pj = tj[jj + u];
          const float dx = fabsf(pi.x - pj.x), dy = fabsf(pi.y - pj.y), dz = fabsf(pi.z - pj.z);
          const float ax = fminf(dx, fabsf(dx - L[0])), ay = fminf(dy, fabsf(dy - L[1])),
                      az = fminf(dz, fabsf(dz - L[2]));
          const float R2 = fmaf(az, az, fmaf(ay, ay, ax * ax));
          const float y = __builtin_amdgcn_rsqf(R2);
          const float tc = fmaf(R2 * sc, y, 0.5f);    // NaN at R2 = 0: exact arithmetic
          // half a bin less the bound; beyond rnum the bound is below 1
          const float room = fmaf(ke, y, k0);
          const bool valid = !decltype(masked)::value || (jj + u >= first && jj + u < j1);
          const bool safe = fabsf(__builtin_amdgcn_fractf(tc) - 0.5f) < room;
          if (valid && safe && tc < tin) atomicAdd(&h[(uint32_t)tc], 1u);
          slow[u] = valid && !safe && !(tc >= tout);
          any |= slow[u];
        }
        if (__ballot(any) == 0ull) return;
#pragma unroll
        for (uint32_t u = 0; u < U; ++u) {
          const uint64_t m = __ballot(slow[u]);
          if (slow[u])
            queue[wave][qn + __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32),
                                                       __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u))] =
                (tid << 16) + jj + u;
          qn += (uint32_t)__popcll(m);
        }
        while (qn >= 64u) work_off(64u);
      };
      uint32_t jj = j0;
      if (!diag && ni == GR_T)
        for (; jj + 4 <= j1; jj += 4) four(jj, std::false_type{});
      for (; jj < j1; jj += 4) four(jj, std::true_type{});
      if (qn) work_off(qn);                // fewer than 64
    }
    // flush when the replica changes, at the end (histograms are per
    // replica) and every GR_FLUSH_TILES work items (no uint32 count can wrap)
    const bool flush = w + 1 >= w1 || ++since >= GR_FLUSH_TILES ||
                       (rep + 1 < nrep && (w + 1) / slices >= reps[rep + 1].pair0);
    if (flush) {
      __syncthreads();
      uint32_t mine = 0;
      for (uint32_t b = tid; b < rnum; b += GR_T) {
        const uint32_t v = h[b];
        h[b] = 0;
        if (b && v) {
          mine += v;
          atomicAdd((unsigned long long *)&hist[(uint64_t)rep * rnum + b], (unsigned long long)v);
        }
      }
      mine = pb_wave_sum_u32(mine);
      if (lane == 0 && mine) atomicAdd(&binned, mine);
      __syncthreads();
      if (tid == 0) {
        if (pairs != binned)
          atomicAdd((unsigned long long *)&hist[(uint64_t)rep * rnum], (unsigned long long)(pairs - binned));
        binned = 0;
      }
      pairs = 0;
      since = 0;
    }
  }
}

// replica table of the g(r) kernel from the device replica records: one
// workgroup; per-replica tile-pair counts scanned in order (uint64)
__global__ void __launch_bounds__(256) k_gr_prep(const RepInfo *reps, const float *rstep,
                                                 uint32_t nrep, GrRep *out) {
  __shared__ unsigned long long part[256];
  const uint32_t per = (nrep + 255u) / 256u;
  const uint32_t q0 = threadIdx.x * per, q1 = min(nrep, q0 + per);
  unsigned long long mine = 0;
  for (uint32_t q = q0; q < q1; ++q) {
    const unsigned long long nt = (reps[q].natoms + GR_T - 1) / GR_T;
    mine += nt * (nt + 1) / 2;
  }
  part[threadIdx.x] = mine;
  __syncthreads();
  unsigned long long base = 0;
  for (uint32_t k = 0; k < threadIdx.x; ++k) base += part[k];
  for (uint32_t q = q0; q < q1; ++q) {
    const RepInfo &R = reps[q];
    GrRep g;
    g.atom0 = R.atom0;
    g.natoms = R.natoms;
    g.ntile = (R.natoms + GR_T - 1) / GR_T;
    g.pair0 = base;
    base += (unsigned long long)g.ntile * (g.ntile + 1) / 2;
    // cudaFrame::setCell (cudaFrame.cu:85-91) on the FP32 cell values
    float c[3];
    for (int a = 0; a < 3; ++a) {
      const float lo = (float)R.lo[a], hi = (float)R.hi[a];
      c[a] = (hi - lo) * 0.5f;            // = (hi - lo) / 2 exactly
      c[a] *= c[a];
    }
    g.cx = c[0];
    g.cy = c[1];
    g.cz = c[2];
    // cudaCalcGR::setup: rstepinv = 1.0 / rstep (double) stored as real
    g.rstepinv = (float)(1.0 / (double)rstep[q]);
    for (int a = 0; a < 3; ++a) {
      g.lo[a] = (float)R.lo[a];
      g.hi[a] = (float)R.hi[a];
    }
    out[q] = g;
  }
}

__global__ void k_zero_u64(uint64_t *x, size_t n) {
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) x[i] = 0;
}

// Table, cleared histograms, pairs and the histograms back to the host, on
// given device memory (rstep first written by an upload).  Storage order
// holds each replica's real particles at [atom0, atom0 + natoms) at all times
// (padding sorts after the real particles of its replica).
static int gr_run(pb_sys *s, const float *rstep, uint32_t rnum, uint64_t *hist, GrRep *dreps,
                  float *drstep, uint64_t *dhist) {
  uint64_t tot = 0;
  for (uint32_t q = 0; q < s->nrep; ++q) {
    const uint64_t nt = (s->reps[q].natoms + GR_T - 1) / GR_T;
    tot += nt * (nt + 1) / 2;
  }
  // few tile pairs: their j particles split so that 4096 workgroups (16 a
  // compute unit) have work
  uint32_t slices = 1;
  while (slices < GR_MAX_SLICES && tot * slices < 4096) slices *= 2;
  const size_t hn = (size_t)s->nrep * rnum;
  hipStream_t st = s->ctx->stream;
  if (int rc = pb_io_upload(s->ctx, drstep, rstep, sizeof(float) * s->nrep)) return rc;
  hipLaunchKernelGGL(k_gr_prep, dim3(1), dim3(256), 0, st, s->d_reps, drstep, s->nrep, dreps);
  hipLaunchKernelGGL(k_zero_u64, dim3(pb_blocks(hn, 256)), dim3(256), 0, st, dhist, hn);
  if (tot) {
    // a few items a workgroup: their number varies by the diagonal and the
    // ragged tiles (16384 workgroups at most: 6 % slower on the 256 replicas)
    const uint32_t grid = (uint32_t)std::min<uint64_t>(tot * slices, 65536);
    hipLaunchKernelGGL(k_gr, dim3(grid), dim3(GR_T), sizeof(uint32_t) * rnum, st,
                       s->r, dreps, s->nrep, tot * slices, slices, rnum, dhist);
  }
  PB_LAUNCH_CHECK(s->ctx, "k_gr");
  return pb_io_download(s->ctx, hist, dhist, sizeof(uint64_t) * hn);
}

extern "C" int pb_gr_hist(pb_sys *s, const float *rstep, uint32_t rnum, uint64_t *hist) {
  if (!s || !rstep || !hist || rnum == 0) return PB_ERR_ARG;
  if (rnum > 16384) return pb_fail(s->ctx, PB_ERR_ARG, "pb_gr_hist: rnum > 16384");
  if (!s->cell_set) return pb_fail(s->ctx, PB_ERR_STATE, "pb_gr_hist: cell not set");
  // one workspace, kept: histograms, replica table, steps
  const size_t hb = sizeof(uint64_t) * (size_t)s->nrep * rnum, rb = sizeof(GrRep) * (size_t)s->nrep;
  const size_t need = hb + rb + sizeof(float) * (size_t)s->nrep;
  if (s->gr_cap < need) {
    s->gr_cap = 0;
    if (int rc = pb_alloc(s->ctx, (uint8_t **)&s->gr_hist, need)) return rc;
    s->gr_cap = need;
  }
  uint8_t *base = (uint8_t *)s->gr_hist;
  return gr_run(s, rstep, rnum, hist, (GrRep *)(base + hb), (float *)(base + hb + rb), s->gr_hist);
}

// ---------------------------------------- g(r) without allocations
// pb_gr_hist_noalloc keeps its replica table and histograms in this
// file-scope device array instead of library-allocated memory: each device
// holds its own copy for the life of the process.  Host code never passes
// the array's name to a kernel (on the host it is only a stand-in symbol);
// it uses the device address that pb_gr_scratch_init stores in the context.
#define GR_NA_MAX_REPS 4096u                          // replicas per call
#define GR_NA_MAX_SLOTS 131072u                       // nrep * rnum histogram slots
#define GR_NA_REP_BYTES ((size_t)GR_NA_MAX_REPS * sizeof(GrRep))
#define GR_NA_RSTEP_BYTES ((size_t)GR_NA_MAX_REPS * sizeof(float))
#define GR_NA_BYTES (GR_NA_REP_BYTES + GR_NA_RSTEP_BYTES + (size_t)GR_NA_MAX_SLOTS * 8)
static __device__ __align__(256) unsigned char scratch[GR_NA_BYTES];

// the device address of `scratch` on the context's (current) device
int pb_gr_scratch_init(pb_ctx *c) {
  void *ptr = nullptr;
  const hipError_t e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
  if (e != hipSuccess || !ptr) return pb_hip_check(c, e != hipSuccess ? e : hipErrorUnknown,
                                                   "hipGetSymbolAddress(g(r) scratch)");
  c->gr_scratch = ptr;
  return PB_OK;
}

extern "C" int pb_gr_hist_noalloc(pb_sys *s, const float *rstep, uint32_t rnum, uint64_t *hist) {
  if (!s || !rstep || !hist || rnum == 0) return PB_ERR_ARG;
  if (rnum > 16384) return pb_fail(s->ctx, PB_ERR_ARG, "pb_gr_hist_noalloc: rnum > 16384");
  if (!s->cell_set) return pb_fail(s->ctx, PB_ERR_STATE, "pb_gr_hist_noalloc: cell not set");
  if (s->nrep > GR_NA_MAX_REPS)
    return pb_fail(s->ctx, PB_ERR_ARG, "pb_gr_hist_noalloc: more than 4096 replicas");
  if ((uint64_t)s->nrep * rnum > GR_NA_MAX_SLOTS)
    return pb_fail(s->ctx, PB_ERR_ARG,
                   "pb_gr_hist_noalloc: replicas x bins above the scratch limit of 131072");
  if (!s->ctx->gr_scratch)
    return pb_fail(s->ctx, PB_ERR_STATE, "pb_gr_hist_noalloc: no scratch address");
  for (uint32_t q = 0; q < s->nrep; ++q)
    if (!(rstep[q] > 0.0f)) return pb_fail(s->ctx, PB_ERR_ARG, "pb_gr_hist_noalloc: rstep <= 0");
  unsigned char *base = static_cast<unsigned char *>(s->ctx->gr_scratch);
  return gr_run(s, rstep, rnum, hist, reinterpret_cast<GrRep *>(base),
                reinterpret_cast<float *>(base + GR_NA_REP_BYTES),
                reinterpret_cast<uint64_t *>(base + GR_NA_REP_BYTES + GR_NA_RSTEP_BYTES));
}

__global__ void k_clear4_bin(double4 *x, uint32_t n) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) x[i] = make_double4(0.0, 0.0, 0.0, 0.0);
}

// ------------------------------------------- MD neighbour list (CSR) path
// cudaParticleMD::useNList / makeNList (cudaParticleMD.cu:338-394;
// calcCoordMD_F4 counts, makeJlist_WithBlock_F4 kerneltemplate.hh:725-775,
// MDNeighborRegister kernelinline.hh:404-412) and the forces of
// calcF_IJpairWithList_F4 (kerneltemplate.hh:136-168).  Rows and columns are
// original particle indices; a row holds every j != i of the 27 cells with
// FP32 distance2p < rmax2t, in ascending order (the reference leaves them
// in traversal order).

// visit the storage slots sj of the 27 cells around cell c (periodic wrap
// as calc_BlockNeighbor; non-periodic cells outside the box are skipped)
template <typename Fn>
__device__ __forceinline__ void for_27_cells(const RefGrid &g, uint32_t c, int periodic,
                                             const uint32_t *start, const uint32_t *perm, Fn &&fn) {
  const uint32_t nyz = g.nb[1] * g.nb[2];
  const int i0 = (int)(c / nyz), j0 = (int)((c / g.nb[2]) % g.nb[1]), k0 = (int)(c % g.nb[2]);
  for (int a = -1; a <= 1; ++a) {
    int i2 = i0 + a;
    if (i2 < 0 || i2 >= (int)g.nb[0]) {
      if (!periodic) continue;
      i2 = (i2 + (int)g.nb[0]) % (int)g.nb[0];
    }
    for (int b = -1; b <= 1; ++b) {
      int j2 = j0 + b;
      if (j2 < 0 || j2 >= (int)g.nb[1]) {
        if (!periodic) continue;
        j2 = (j2 + (int)g.nb[1]) % (int)g.nb[1];
      }
      for (int d = -1; d <= 1; ++d) {
        int k2 = k0 + d;
        if (k2 < 0 || k2 >= (int)g.nb[2]) {
          if (!periodic) continue;
          k2 = (k2 + (int)g.nb[2]) % (int)g.nb[2];
        }
        const uint32_t J = (uint32_t)k2 + (uint32_t)j2 * g.nb[2] + (uint32_t)i2 * nyz;
        for (uint32_t jj = start[J]; jj < start[J + 1]; ++jj) fn(perm[jj]);
      }
    }
  }
}

struct NlistArgs {
  const float4 *pos;           // cell order: FP32 position, original index
  const uint32_t *bid, *start; // cell of a sorted position, first position of a cell
  uint32_t nreal;
  RefGrid g;
  float L[3];                  // FP32 box edges
  float cx, cy, cz, rmax2t;
  int periodic;
  uint32_t cap;                // capacity of the column array
  uint32_t k0;                 // first sorted position of the launch
};

__global__ void k_md_gather(const double4 *r, const uint32_t *perm, const uint32_t *pid,
                            uint32_t n, float4 *pos) {
  const uint32_t k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= n) return;
  const double4 p = r[perm[k]];
  pos[k] = make_float4((float)p.x, (float)p.y, (float)p.z, __uint_as_float(pid[k]));
}

// Rows of the list: one wavefront a particle, 64 candidates of the 27 cells
// at a time (a column of three cells is one contiguous run of the cell order,
// two where it wraps in z), so a row's candidates are coalesced reads and
// 32,000 particles are 32,000 wavefronts.  The reference's FP32 distance2p
// decides; it is evaluated only where the distance from folded axes lies
// within the rounding bound of rmax2t (the bound of k_gr: 64 u (cx + cy + cz)
// for |d| <= 1.25 L), a few lanes in a hundred thousand.
//   FILL = false: the row's length.
//   FILL = true: the row's original indices, ascending: the hits are compacted
// into LDS and every hit counts the smaller ones.  Rows longer than the LDS
// row are written as found and sorted in place by one lane.
// 32,000 particles of a liquid (about 80 a row): 316 + 1079 us a build with a
// thread a row and an insertion sort in global memory, 48 + 69 us now.
// A launch takes NL_LAUNCH rows: its work items must fit in 32 bits, and a million
// wavefronts leave no tail worth a longer launch.
#define NL_CAP 512u
#define NL_LAUNCH (1u << 20)
template <bool FILL>
__global__ void __launch_bounds__(256) k_nlist(NlistArgs A, uint32_t *rowcnt, const uint32_t *rowptr,
                                               uint32_t *col) {
  __shared__ __align__(16) uint32_t rows[FILL ? 4 : 1][FILL ? NL_CAP : 1];
  const uint32_t lane = pb_lane(), wave = threadIdx.x / 64;
  const uint32_t k = A.k0 + __builtin_amdgcn_readfirstlane(blockIdx.x * 4u + wave);
  if (k >= A.nreal) return;
  const float4 pi = A.pos[k];
  const uint32_t oi = __float_as_uint(pi.w), c = A.bid[k];
  uint32_t b = 0, len = 0;
  if (FILL) {
    b = rowptr[oi];
    len = rowptr[oi + 1] - b;
    if (b + len > A.cap || len == 0) return;          // outgrown: filled again, larger
  }
  const float E = 64.0f * 5.9604645e-8f * 1.0001f * (A.cx + A.cy + A.cz);
  const float lim = A.rmax2t + E, sure = A.rmax2t - E;
  const float fx = 1.25f * A.L[0], fy = 1.25f * A.L[1], fz = 1.25f * A.L[2];
  const int nb0 = (int)A.g.nb[0], nb1 = (int)A.g.nb[1], nb2 = (int)A.g.nb[2];
  const int i0 = (int)(c / (A.g.nb[1] * A.g.nb[2])), j0 = (int)((c / A.g.nb[2]) % A.g.nb[1]),
            k0 = (int)(c % A.g.nb[2]);
  uint32_t cnt = 0;
  auto run = [&](uint32_t q0, uint32_t q1) {          // wave-uniform
    for (uint32_t q = q0; q < q1; q += 64u) {
      const uint32_t j = q + lane;
      bool hit = false;
      uint32_t oj = 0;
      if (j < q1 && j != k) {
        const float4 pj = A.pos[j];
        oj = __float_as_uint(pj.w);
        const float dx = fabsf(pi.x - pj.x), dy = fabsf(pi.y - pj.y), dz = fabsf(pi.z - pj.z);
        const float ax = fminf(dx, fabsf(dx - A.L[0])), ay = fminf(dy, fabsf(dy - A.L[1])),
                    az = fminf(dz, fabsf(dz - A.L[2]));
        const float R2 = fmaf(az, az, fmaf(ay, ay, ax * ax));
        const bool bound = dx <= fx && dy <= fy && dz <= fz;
        hit = R2 < sure;
        if (!bound || !(hit || R2 >= lim))
          hit = distance2p(pi.x, pi.y, pi.z, pj.x, pj.y, pj.z, A.cx, A.cy, A.cz) < A.rmax2t;
      }
      const uint64_t m = __ballot(hit);
      if (FILL && hit) {
        const uint32_t p = cnt + __builtin_amdgcn_mbcnt_hi(
                                     (uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
        if (len > NL_CAP) col[b + p] = oj;
        else rows[wave][p] = oj;
      }
      cnt += (uint32_t)__popcll(m);
    }
  };
  for (int a = -1; a <= 1; ++a) {
    int i2 = i0 + a;
    if (i2 < 0 || i2 >= nb0) {
      if (!A.periodic) continue;
      i2 = i2 < 0 ? nb0 - 1 : 0;
    }
    for (int d = -1; d <= 1; ++d) {
      int j2 = j0 + d;
      if (j2 < 0 || j2 >= nb1) {
        if (!A.periodic) continue;
        j2 = j2 < 0 ? nb1 - 1 : 0;
      }
      const uint32_t cb = ((uint32_t)i2 * A.g.nb[1] + (uint32_t)j2) * A.g.nb[2];
      const int lo = k0 > 0 ? k0 - 1 : 0, hi = k0 + 1 < nb2 ? k0 + 1 : nb2 - 1;
      run(A.start[cb + (uint32_t)lo], A.start[cb + (uint32_t)hi + 1u]);
      if (A.periodic && k0 == 0) run(A.start[cb + (uint32_t)nb2 - 1u], A.start[cb + (uint32_t)nb2]);
      if (A.periodic && k0 == nb2 - 1) run(A.start[cb], A.start[cb + 1u]);
    }
  }
  if (!FILL) {
    if (lane == 0) rowcnt[oi] = cnt;
    return;
  }
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup");
  __builtin_amdgcn_wave_barrier();
  if (len <= NL_CAP) {
    const uint32_t *row = rows[wave];
    for (uint32_t base = 0; base < len; base += 64u) {
      const uint32_t i = base + lane;
      const uint32_t x = i < len ? row[i] : 0u;
      uint32_t rank = 0, j = 0;
      for (; j + 4 <= len; j += 4) {
        const uint4 y = *reinterpret_cast<const uint4 *>(row + j);
        rank += (y.x < x ? 1u : 0u) + (y.y < x ? 1u : 0u) + (y.z < x ? 1u : 0u) + (y.w < x ? 1u : 0u);
      }
      for (; j < len; ++j) rank += row[j] < x ? 1u : 0u;
      if (i < len) col[b + rank] = x;
    }
  } else if (lane == 0) {
    for (uint32_t i = b + 1; i < b + len; ++i) {
      const uint32_t x = col[i];
      uint32_t j = i;
      while (j > b && col[j - 1] > x) {
        col[j] = col[j - 1];
        --j;
      }
      col[j] = x;
    }
  }
}

__global__ void k_inverse_perm(const uint32_t *orig, uint32_t n, uint32_t *inv) {
  const uint32_t s = blockIdx.x * blockDim.x + threadIdx.x;
  if (s < n && orig[s] != PB_NONE) inv[orig[s]] = s;
}

// FP64 minimum-image displacement (the distance2p fold of MDpairForce,
// kerneltemplate.hh:538-543, without its FP32 rounding)
__device__ __forceinline__ double min_image(double d, double L, int periodic) {
  if (periodic && d * d > 0.25 * L * L) d += d < 0 ? L : -L;
  return d;
}

struct PairArgs {
  const double4 *r;
  const uint32_t *orig, *inv;
  const uint32_t *rowptr, *col;     // list path
  const uint32_t *perm, *cellid, *start;   // cell path
  uint32_t npad;
  uint32_t block0;                  // list path: first 64 slots of the launch
  RefGrid g;
  double L[3];
  int periodic;
  const LJTable *lj;
  double rc2;
  double sc_rc, sc_f0;              // soft core
  double4 *F;
  double *partials;
};

// LJ forces, PE and virial from the CSR list (pairs with r^2 < rc2): eight
// lanes a row, each taking every eighth column, so a row's columns are read
// together and a lane waits for ten dependent gathers (column, slot, position)
// instead of eighty.  Bound by that latency: 32,000 rows of about 80 are 4000
// wavefronts; a thread a row (500 wavefronts) took 79 us, this 20 us.
// Partials per 64 slots, added in a fixed order.
#define NF_LANES 8u
__global__ void __launch_bounds__(64 * NF_LANES) k_lj_force_nlist(PairArgs A) {
  __shared__ double tab[4][PB_MAXT * PB_MAXT];
  __shared__ double sums[2][NF_LANES];
  for (uint32_t t = threadIdx.x; t < PB_MAXT * PB_MAXT; t += blockDim.x) {
    tab[0][t] = A.lj->s2[t];
    tab[1][t] = A.lj->e24[t];
    tab[2][t] = A.lj->e4[t];
    tab[3][t] = A.lj->shift[t];
  }
  __syncthreads();
  const uint32_t block = A.block0 + blockIdx.x;
  const uint32_t si = block * 64u + threadIdx.x / NF_LANES, sub = threadIdx.x % NF_LANES;
  double pe = 0.0, vir = 0.0;
  const uint32_t row = si < A.npad ? A.orig[si] : PB_NONE;
  if (row != PB_NONE) {
    const double4 pi = A.r[si];
    const uint32_t ti = (uint32_t)pi.w;
    double fx = 0.0, fy = 0.0, fz = 0.0;
    const uint32_t e = A.rowptr[row + 1];
#pragma unroll 2
    for (uint32_t k = A.rowptr[row] + sub; k < e; k += NF_LANES) {
      const double4 pj = A.r[A.inv[A.col[k]]];
      const double dx = min_image(pi.x - pj.x, A.L[0], A.periodic);
      const double dy = min_image(pi.y - pj.y, A.L[1], A.periodic);
      const double dz = min_image(pi.z - pj.z, A.L[2], A.periodic);
      const double r2 = dx * dx + dy * dy + dz * dz;
      if (!(r2 < A.rc2)) continue;
      const uint32_t t = ti * PB_MAXT + (uint32_t)pj.w;
      double s6 = tab[0][t] / r2;
      s6 = s6 * s6 * s6;
      const double fr = tab[1][t] * s6 * (2.0 * s6 - 1.0) / r2;
      fx += fr * dx;
      fy += fr * dy;
      fz += fr * dz;
      pe += 0.5 * (tab[2][t] * s6 * (s6 - 1.0) - tab[3][t]);
      vir += 0.5 * fr * r2;
    }
#pragma unroll
    for (uint32_t o = 1; o < NF_LANES; o <<= 1) {      // a row's lanes take this branch together
      fx += __shfl_xor(fx, (int)o, 64);
      fy += __shfl_xor(fy, (int)o, 64);
      fz += __shfl_xor(fz, (int)o, 64);
    }
    if (sub == 0) A.F[si] = make_double4(fx, fy, fz, 0.0);
  }
  pe = pb_wave_sum(pe);
  vir = pb_wave_sum(vir);
  if (pb_lane() == 0) {
    sums[0][threadIdx.x / 64] = pe;
    sums[1][threadIdx.x / 64] = vir;
  }
  __syncthreads();
  if (threadIdx.x < 2) {
    double t = 0.0;
    for (uint32_t w = 0; w < NF_LANES; ++w) t += sums[threadIdx.x][w];
    A.partials[4 * (size_t)block + threadIdx.x] = t;
  }
}

// Soft-core forces of initialAnnealing (potentialSC, kernelinline.hh:140-158,
// through MDpairForce, kerneltemplate.hh:524-565) over the 27 cells:
// F_i = sum_j f0 cos(r/rc pi/2) (r_i - r_j)/r for r <= rc and r^2 < rmax2.
__global__ void k_softcore_force(PairArgs A, uint32_t nreal) {
  const uint32_t k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= nreal) return;
  const uint32_t si = A.perm[k];
  const double4 pi = A.r[si];
  double fx = 0.0, fy = 0.0, fz = 0.0;
  const double hpi = 0.5 * M_PI / A.sc_rc;
  for_27_cells(A.g, A.cellid[si], A.periodic, A.start, A.perm, [&](uint32_t sj) {
    if (sj == si) return;
    const double4 pj = A.r[sj];
    const double dx = min_image(pi.x - pj.x, A.L[0], A.periodic);
    const double dy = min_image(pi.y - pj.y, A.L[1], A.periodic);
    const double dz = min_image(pi.z - pj.z, A.L[2], A.periodic);
    const double r2 = dx * dx + dy * dy + dz * dz;
    if (!(r2 < A.rc2)) return;
    const double r = sqrt(r2);
    if (r > A.sc_rc) return;
    const double f = A.sc_f0 * cos(r * hpi) / r;
    fx += f * dx;
    fy += f * dy;
    fz += f * dz;
  });
  A.F[si] = make_double4(fx, fy, fz, 0.0);
}

static int need_binned_grid(pb_sys *s, const char *who) {
  if (!s->ref_cells || s->ref_single)
    return pb_fail(s->ctx, PB_ERR_STATE, std::string(who) + ": needs a 27-neighbour cell grid");
  if (!s->ref_binned) return pb_fail(s->ctx, PB_ERR_STATE, std::string(who) + ": pb_bin first");
  return PB_OK;
}

// the 27-cell search's arguments, on the positions gathered into cell order
static int nlist_args(pb_sys *s, float rmax2t, NlistArgs *out) {
  int rc;
  if (!s->md_cnt &&                          // the last of them
      ((rc = pb_alloc(s->ctx, &s->md_pos, s->npad)) || (rc = pb_alloc(s->ctx, &s->md_cnt, (size_t)s->n + 1))))
    return rc;
  hipLaunchKernelGGL(k_md_gather, dim3(pb_blocks(s->n, 256)), dim3(256), 0, s->ctx->stream, s->r,
                     s->perm, s->ref_pid, s->n, s->md_pos);
  PB_LAUNCH_CHECK(s->ctx, "k_md_gather");
  NlistArgs &A = *out;
  A.pos = s->md_pos;
  A.bid = s->ref_bid;
  A.start = s->cstart;
  A.nreal = s->n;
  A.g = ref_grid(s);
  float c[3];
  half_cell2(s, 0, c);
  A.cx = c[0];
  A.cy = c[1];
  A.cz = c[2];
  for (int a = 0; a < 3; ++a) A.L[a] = (float)s->cells[2 * a + 1] - (float)s->cells[2 * a];
  A.rmax2t = rmax2t;
  A.periodic = s->ref_periodic;
  A.cap = 0;
  return PB_OK;
}

// all rows: their lengths to md_cnt (FILL = false), or their columns to md_col
template <bool FILL>
static int nlist_rows(pb_sys *s, NlistArgs A) {
  for (A.k0 = 0; A.k0 < A.nreal; A.k0 += NL_LAUNCH)
    hipLaunchKernelGGL(k_nlist<FILL>, dim3(pb_blocks(std::min(A.nreal - A.k0, NL_LAUNCH), 4)), dim3(256),
                       0, s->ctx->stream, A, s->md_cnt, s->md_row, s->md_col);
  PB_LAUNCH_CHECK(s->ctx, FILL ? "k_nlist (rows)" : "k_nlist (counts)");
  return PB_OK;
}

// calcCoordMD_F4 counts (kernelinline.hh:387-399) over the 27 cells of
// calcF_IJpairWithBlock_F4 (kerneltemplate.hh:244-293): the rows' lengths
extern "C" int pb_coord_counts(pb_sys *s, float rmax2t, uint32_t *counts) {
  if (!s || !counts) return PB_ERR_ARG;
  if (!s->ref_cells || s->ref_single)
    return pb_fail(s->ctx, PB_ERR_STATE, "pb_coord_counts: needs a 27-neighbour cell grid");
  const float rc = sqrtf(rmax2t);
  for (int a = 0; a < 3; ++a)
    if (s->blocklen[a] < rc)
      return pb_fail(s->ctx, PB_ERR_CELLS, "pb_coord_counts: cell length below the count radius");
  if (int e = pb_bin(s)) return e;
  NlistArgs A;
  if (int e = nlist_args(s, rmax2t, &A)) return e;
  if (int e = nlist_rows<false>(s, A)) return e;
  return pb_io_download(s->ctx, counts, s->md_cnt, 4 * (size_t)s->n);
}

extern "C" int pb_nlist_build(pb_sys *s, float rmax2t, uint32_t *nnz_out) {
  if (!s || !(rmax2t > 0.0f)) return PB_ERR_ARG;
  if (int rc = need_binned_grid(s, "pb_nlist_build")) return rc;
  const float rc = sqrtf(rmax2t);
  for (int a = 0; a < 3; ++a)
    if (s->blocklen[a] < rc)
      return pb_fail(s->ctx, PB_ERR_CELLS, "pb_nlist_build: cell length below the list radius");
  hipStream_t st = s->ctx->stream;
  const uint32_t n = s->n;
  int rc2;
  if (!s->md_row && (rc2 = pb_alloc(s->ctx, &s->md_row, (size_t)n + 1))) return rc2;
  NlistArgs A;
  if ((rc2 = nlist_args(s, rmax2t, &A))) return rc2;
  s->md_valid = false;                        // until the rows are whole
  if ((rc2 = nlist_rows<false>(s, A))) return rc2;
  if ((rc2 = pb_exclusive_scan(s, s->md_cnt, s->md_row, n))) return rc2;
  // the rows are filled before the host knows their sum, up to the capacity
  // of the last list; a list that outgrew it is filled again
  auto fill = [&]() -> int {
    A.cap = s->md_cap;
    return A.cap ? nlist_rows<true>(s, A) : PB_OK;
  };
  if ((rc2 = fill())) return rc2;
  PB_HIP(s->ctx, hipMemcpyAsync(s->ctx->res, s->md_row + n, 4, hipMemcpyDeviceToHost, st));
  PB_HIP(s->ctx, hipStreamSynchronize(st));
  uint32_t nnz;
  std::memcpy(&nnz, s->ctx->res, 4);
  if (s->md_cap < nnz || !s->md_col) {
    const uint32_t cap = (uint32_t)std::min<uint64_t>((uint64_t)nnz + nnz / 16 + 64, 0xFFFFFFF0ull);
    s->md_cap = 0;
    if ((rc2 = pb_alloc(s->ctx, &s->md_col, cap))) return rc2;
    s->md_cap = cap;
    if ((rc2 = fill())) return rc2;
  }
  s->md_nnz = nnz;
  s->md_valid = true;
  if (nnz_out) *nnz_out = nnz;
  return PB_OK;
}

extern "C" int pb_nlist_get(pb_sys *s, uint32_t *rowptr, uint32_t *colidx, uint32_t cap,
                            uint32_t *nnz) {
  if (!s) return PB_ERR_ARG;
  if (!s->md_valid) return pb_fail(s->ctx, PB_ERR_STATE, "pb_nlist_get: pb_nlist_build first");
  hipStream_t st = s->ctx->stream;
  if (nnz) *nnz = s->md_nnz;
  if (rowptr)
    PB_HIP(s->ctx, hipMemcpyAsync(rowptr, s->md_row, 4 * ((size_t)s->n + 1), hipMemcpyDeviceToHost, st));
  if (colidx) {
    if (cap < s->md_nnz) return pb_fail(s->ctx, PB_ERR_ARG, "pb_nlist_get: colidx too small");
    PB_HIP(s->ctx, hipMemcpyAsync(colidx, s->md_col, 4 * (size_t)s->md_nnz, hipMemcpyDeviceToHost, st));
  }
  PB_HIP(s->ctx, hipStreamSynchronize(st));
  return PB_OK;
}

static PairArgs pair_args(pb_sys *s) {
  PairArgs A;
  std::memset(&A, 0, sizeof(A));
  A.r = s->r;
  A.orig = s->orig;
  A.npad = s->npad;
  A.g = ref_grid(s);
  for (int a = 0; a < 3; ++a) A.L[a] = s->cells[2 * a + 1] - s->cells[2 * a];
  A.periodic = s->ref_periodic;
  A.lj = s->d_lj;
  A.rc2 = s->rc2;
  A.F = s->F;
  A.partials = s->partials;
  A.perm = s->perm;
  A.cellid = s->cellid;
  A.start = s->cstart;
  return A;
}

extern "C" int pb_lj_force_nlist(pb_sys *s, double *pe, double *virial) {
  if (!s) return PB_ERR_ARG;
  if (!s->md_valid) return pb_fail(s->ctx, PB_ERR_STATE, "pb_lj_force_nlist: pb_nlist_build first");
  if (!s->lj_set || !(s->rc2 > 0)) return pb_fail(s->ctx, PB_ERR_STATE, "LJ parameters or cutoff not set");
  if (s->nrep != 1) return pb_fail(s->ctx, PB_ERR_STATE, "pb_lj_force_nlist: single replica only");
  hipStream_t st = s->ctx->stream;
  int rc;
  if (!s->md_inv && (rc = pb_alloc(s->ctx, &s->md_inv, (size_t)s->n))) return rc;
  if (s->md_inv_order != s->order_gen) {
    hipLaunchKernelGGL(k_inverse_perm, dim3(pb_blocks(s->npad, 256)), dim3(256), 0, st, s->orig,
                       s->npad, s->md_inv);
    PB_LAUNCH_CHECK(s->ctx, "k_inverse_perm");
    s->md_inv_order = s->order_gen;
  }
  PairArgs A = pair_args(s);
  A.inv = s->md_inv;
  A.rowptr = s->md_row;
  A.col = s->md_col;
  A.periodic = 1;       // MD boxes are periodic (MDpairForce folds every pair)
  for (A.block0 = 0; A.block0 < s->nwave; A.block0 += NL_LAUNCH / 64u)
    hipLaunchKernelGGL(k_lj_force_nlist, dim3(std::min(s->nwave - A.block0, NL_LAUNCH / 64u)),
                       dim3(64 * NF_LANES), 0, st, A);
  PB_LAUNCH_CHECK(s->ctx, "k_lj_force_nlist");
  if (pe || virial) {
    const double *h = nullptr;
    if ((rc = pb_reduce_to_host(s, 2, &h))) return rc;
    if (pe) *pe = h[0];
    if (virial) *virial = h[1];
  }
  return PB_OK;
}

extern "C" int pb_softcore_force(pb_sys *s, double rc, double f0, double rmax2) {
  if (!s || !(rc > 0) || !(rmax2 > 0)) return PB_ERR_ARG;
  if (int e = need_binned_grid(s, "pb_softcore_force")) return e;
  for (int a = 0; a < 3; ++a)
    if ((double)s->blocklen[a] < std::min(rc, std::sqrt(rmax2)))
      return pb_fail(s->ctx, PB_ERR_CELLS, "pb_softcore_force: cell length below the soft-core radius");
  PairArgs A = pair_args(s);
  A.rc2 = rmax2;
  A.sc_rc = rc;
  A.sc_f0 = f0;
  hipLaunchKernelGGL(k_clear4_bin, dim3(pb_blocks(s->npad, 256)), dim3(256), 0, s->ctx->stream,
                     s->F, s->npad);
  hipLaunchKernelGGL(k_softcore_force, dim3(pb_blocks(s->n, 256)), dim3(256), 0, s->ctx->stream, A,
                     s->n);
  PB_LAUNCH_CHECK(s->ctx, "pb_softcore_force");
  return PB_OK;
}
