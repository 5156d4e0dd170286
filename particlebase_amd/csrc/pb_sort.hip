// pb_sort.hip -- deterministic counting sort of storage slots by cell.
//
// Replaces the reference's calcBlockID sort chain (sortByBID_M1 insertion
// pre-sort, single-block odd-even sortByBID and makeBindex,
// kernelfuncs.cu:844-932, cudaCutoffBlock.cu:241-256), whose in-cell order is
// unstable and timing dependent.  Here:
//   1. counting  : wave64 atomics on per-cell counters by the caller's cell-id
//                  kernel (pb_count_rank); equal cells in neighbouring lanes
//                  are aggregated into one atomic.
//   2. scan      : exclusive prefix sum, LDS-tiled (each block adds the sums,
//                  or the elements, before it), any length.
//   3. k_scatter : (key, slot, cell) to start[cell] + rank; clears the counters for
//                  the next sort.
//   4. ordering  : inside every cell, by a key (the original particle index):
//                  one thread an element counts the smaller keys of its cell
//                  (pb_cell_position) -- the order produced by the atomics is
//                  discarded, so the permutation is the canonical stable one.
//                  Done by the kernel that uses the order (k_cell_order here,
//                  k_reorder of the LJ path), not by a pass of its own.
#include "pb_internal.h"

#define SCAN_BS 256
#define SCAN_PER 8
#define SCAN_CH (SCAN_BS * SCAN_PER)

__global__ void k_fill_u32(uint32_t *x, uint32_t n, uint32_t val) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) x[i] = val;
}

// inclusive wave scan (64 lanes)
__device__ __forceinline__ uint32_t wave_incl_scan(uint32_t x) {
  const uint32_t lane = pb_lane();
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const uint32_t y = __shfl_up(x, o, 64);
    if (lane >= (uint32_t)o) x += y;
  }
  return x;
}

// exclusive block scan of one value per thread; returns the exclusive prefix
// and the block total.
__device__ __forceinline__ uint32_t block_excl_scan(uint32_t x, uint32_t *total) {
  __shared__ uint32_t wsum[SCAN_BS / 64];
  const uint32_t lane = pb_lane(), w = threadIdx.x / 64;
  const uint32_t inc = wave_incl_scan(x);
  if (lane == 63) wsum[w] = inc;
  __syncthreads();
  uint32_t off = 0, tot = 0;
  for (uint32_t k = 0; k < blockDim.x / 64; ++k) {
    if (k < w) off += wsum[k];
    tot += wsum[k];
  }
  __syncthreads();
  *total = tot;
  return off + inc - x;
}

// a thread's SCAN_PER consecutive elements (0 past the end), 16 bytes a load
__device__ __forceinline__ void scan_load(const uint32_t *in, uint32_t n, uint32_t base,
                                          uint32_t (&v)[SCAN_PER]) {
  if (base + SCAN_PER <= n) {
#pragma unroll
    for (int k = 0; k < SCAN_PER; k += 4) {
      const uint4 y = *reinterpret_cast<const uint4 *>(in + base + k);
      v[k] = y.x;
      v[k + 1] = y.y;
      v[k + 2] = y.z;
      v[k + 3] = y.w;
    }
  } else {
#pragma unroll
    for (int k = 0; k < SCAN_PER; ++k) v[k] = base + k < n ? in[base + k] : 0u;
  }
}

__global__ void __launch_bounds__(SCAN_BS) k_scan_reduce(const uint32_t *in, uint32_t n,
                                                         uint32_t *bsum) {
  const uint32_t base = blockIdx.x * SCAN_CH + threadIdx.x * SCAN_PER;
  uint32_t v[SCAN_PER], x = 0;
  scan_load(in, n, base, v);
#pragma unroll
  for (int k = 0; k < SCAN_PER; ++k) x += v[k];
  uint32_t tot;
  (void)block_excl_scan(x, &tot);
  if (threadIdx.x == 0) bsum[blockIdx.x] = tot;
}

// scan-and-add: each block adds the sums of the blocks before it (summed by
// the block itself, so no separate pass scans the block sums); the last
// block writes the total to out[n]
__global__ void __launch_bounds__(SCAN_BS) k_scan_final(const uint32_t *in, uint32_t n,
                                                        const uint32_t *bsum, uint32_t *out) {
  uint32_t pre = 0;
  for (uint32_t k = threadIdx.x; k < blockIdx.x; k += blockDim.x) pre += bsum[k];
  uint32_t before;
  (void)block_excl_scan(pre, &before);
  const uint32_t base = blockIdx.x * SCAN_CH + threadIdx.x * SCAN_PER;
  uint32_t v[SCAN_PER], x = 0;
  scan_load(in, n, base, v);
#pragma unroll
  for (int k = 0; k < SCAN_PER; ++k) x += v[k];
  uint32_t tot;
  uint32_t run = block_excl_scan(x, &tot) + before;
#pragma unroll
  for (int k = 0; k < SCAN_PER; ++k) {
    const uint32_t y = v[k];
    v[k] = run;
    run += y;
  }
  if (base + SCAN_PER <= n) {
#pragma unroll
    for (int k = 0; k < SCAN_PER; k += 4)
      *reinterpret_cast<uint4 *>(out + base + k) = make_uint4(v[k], v[k + 1], v[k + 2], v[k + 3]);
  } else {
#pragma unroll
    for (int k = 0; k < SCAN_PER; ++k)
      if (base + k < n) out[base + k] = v[k];
  }
  if (blockIdx.x == gridDim.x - 1 && threadIdx.x == 0) out[n] = before + tot;
}

// Short arrays in one launch: every block sums all elements before its own
// (at most SCAN_ONE_MAX reads a block, coalesced).  The rebuild of a small
// system is a chain of launches of about 2 us each, so one fewer is worth
// more than the extra reads; the line lies where they reach a launch's time.
#define SCAN_ONE_BS 1024
#define SCAN_ONE_CH 4096
#define SCAN_ONE_MAX 16384u
__global__ void __launch_bounds__(SCAN_ONE_BS) k_scan_one(const uint32_t *in, uint32_t n,
                                                          uint32_t *out) {
  __shared__ uint32_t wsum[SCAN_ONE_BS / 64], wpre[SCAN_ONE_BS / 64];
  const uint32_t b0 = blockIdx.x * SCAN_ONE_CH, lane = pb_lane(), w = threadIdx.x / 64;
  uint32_t pre = 0;
  for (uint32_t k = threadIdx.x; k < b0; k += SCAN_ONE_BS) pre += in[k];
  const uint32_t base = b0 + threadIdx.x * 4u;
  uint32_t v[4], x = 0;
#pragma unroll
  for (uint32_t k = 0; k < 4; ++k) {
    v[k] = base + k < n ? in[base + k] : 0u;
    x += v[k];
  }
  const uint32_t inc = wave_incl_scan(x);
  pre = pb_wave_sum_u32(pre);
  if (lane == 63) wsum[w] = inc;
  if (lane == 0) wpre[w] = pre;
  __syncthreads();
  uint32_t run = inc - x, before = 0, tot = 0;
  for (uint32_t k = 0; k < SCAN_ONE_BS / 64; ++k) {
    if (k < w) run += wsum[k];
    tot += wsum[k];
    before += wpre[k];
  }
  run += before;
#pragma unroll
  for (uint32_t k = 0; k < 4; ++k)
    if (base + k < n) {
      out[base + k] = run;
      run += v[k];
    }
  if (blockIdx.x == gridDim.x - 1 && threadIdx.x == 0) out[n] = before + tot;
}

int pb_exclusive_scan(pb_sys *s, const uint32_t *in, uint32_t *out, uint32_t n) {
  hipStream_t st = s->ctx->stream;
  if (n == 0) {
    hipLaunchKernelGGL(k_fill_u32, dim3(1), dim3(64), 0, st, out, 1u, 0u);
    PB_LAUNCH_CHECK(s->ctx, "scan(empty)");
    return PB_OK;
  }
  if (n <= SCAN_ONE_MAX) {
    hipLaunchKernelGGL(k_scan_one, dim3(pb_blocks(n, SCAN_ONE_CH)), dim3(SCAN_ONE_BS), 0, st, in, n,
                       out);
    PB_LAUNCH_CHECK(s->ctx, "pb_exclusive_scan");
    return PB_OK;
  }
  const uint32_t nb = (n + SCAN_CH - 1) / SCAN_CH;
  const size_t need = (size_t)nb + 1;
  if (s->scan_tmp_n < need) {
    s->scan_tmp_n = 0;
    if (int rc = pb_alloc(s->ctx, &s->scan_tmp, need)) return rc;
    s->scan_tmp_n = need;
  }
  hipLaunchKernelGGL(k_scan_reduce, dim3(nb), dim3(SCAN_BS), 0, st, in, n, s->scan_tmp);
  hipLaunchKernelGGL(k_scan_final, dim3(nb), dim3(SCAN_BS), 0, st, in, n, s->scan_tmp, out);
  PB_LAUNCH_CHECK(s->ctx, "pb_exclusive_scan");
  return PB_OK;
}

__global__ void k_scatter(const uint32_t *cellid, const uint32_t *rank, const uint32_t *start,
                          const uint32_t *key, uint32_t n, uint32_t *skey, uint32_t *sslot,
                          uint32_t *scell, uint32_t *counts, uint32_t ncell) {
  const uint32_t s = blockIdx.x * blockDim.x + threadIdx.x;
  if (s < ncell) counts[s] = 0;
  if (s < n) {
    const uint32_t c = cellid[s], pos = start[c] + rank[s];
    skey[pos] = key[s];
    sslot[pos] = s;
    scell[pos] = c;
  }
}

// The sorted order as arrays: perm, and for the nreal particles pid / bid, and
// bindex (calcBlockID's outputs, cudaCutoffBlock.cu:233-258).  Bound by its
// chain of dependent L2 reads (pair, cell start, keys of the cell) and 20 bytes
// of traffic a particle: 16 us at 796,176 particles in 470,000 cells, where
// ordering runs of 64 cells in LDS and a pass for the outputs took 19 + 6 us;
// 4000 particles in 125 cells 11 us (with the rows, in k_reorder) against
// 29 + 5, since two workgroups had all the cells.
__global__ void k_cell_order(PbCellOrder O, uint32_t n, uint32_t *perm, uint32_t nreal,
                             uint32_t ncell, uint32_t *pid, uint32_t *bid, uint32_t *bindex) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < ncell) {
    const uint32_t b = O.start[i];
    bindex[i] = O.start[i + 1] > b ? b : PB_NONE;
  }
  if (i == 0) bindex[ncell] = nreal;
  if (i >= n) return;
  uint32_t slot, cell;
  const uint32_t k = pb_cell_position(O, i, &slot, &cell);
  perm[k] = slot;
  if (k < nreal) {
    pid[k] = O.skey[i];
    bid[k] = cell;
  }
}

int pb_ensure_sort_ws(pb_sys *s, uint32_t ncell) {
  int rc;
  if (!s->cellid) {                        // the last of them
    if ((rc = pb_alloc(s->ctx, &s->rank, s->npad)) || (rc = pb_alloc(s->ctx, &s->perm, s->npad)) ||
        (rc = pb_alloc(s->ctx, &s->skey, s->npad)) || (rc = pb_alloc(s->ctx, &s->sslot, s->npad)) ||
        (rc = pb_alloc(s->ctx, &s->scell, s->npad)) || (rc = pb_alloc(s->ctx, &s->cellid, s->npad)))
      return rc;
  }
  if (s->ncell_cap < ncell) {
    s->ncell_cap = 0;
    s->ref_binned = false;                   // the order's cell starts go
    if ((rc = pb_alloc(s->ctx, &s->ccount, (size_t)ncell + 1)) ||
        (rc = pb_alloc(s->ctx, &s->cstart, (size_t)ncell + 1)))
      return rc;
    // the counters are zero between sorts (k_scatter clears them)
    hipLaunchKernelGGL(k_fill_u32, dim3(pb_blocks((size_t)ncell + 1, 256)), dim3(256), 0,
                       s->ctx->stream, s->ccount, ncell + 1, 0u);
    PB_LAUNCH_CHECK(s->ctx, "sort workspace");
    s->ncell_cap = ncell;
    s->counts_used = false;
  }
  return PB_OK;
}

int pb_counts_begin(pb_sys *s) {
  s->ref_binned = false;                     // the arrays of the order before are written from here on
  if (s->counts_used) {
    hipLaunchKernelGGL(k_fill_u32, dim3(pb_blocks((size_t)s->ncell_cap + 1, 256)), dim3(256), 0,
                       s->ctx->stream, s->ccount, s->ncell_cap + 1, 0u);
    PB_LAUNCH_CHECK(s->ctx, "pb_counts_begin");
  }
  s->counts_used = true;
  return PB_OK;
}

// the sort after the counting (s->ccount and s->rank filled by the caller's
// cell-id kernel) up to the scattered (key, slot, cell)
int pb_counting_sort(pb_sys *s, uint32_t ncell, const uint32_t *key, PbCellOrder *O) {
  s->lj_cont = false;             // the fused LJ run's cell order is gone
  const uint32_t n = s->npad;
  if (int rc = pb_exclusive_scan(s, s->ccount, s->cstart, ncell)) return rc;
  hipLaunchKernelGGL(k_scatter, dim3(pb_blocks(n > ncell ? n : ncell, 256)), dim3(256), 0,
                     s->ctx->stream, s->cellid, s->rank, s->cstart, key, n, s->skey, s->sslot,
                     s->scell, s->ccount, ncell);
  PB_LAUNCH_CHECK(s->ctx, "pb_counting_sort");
  s->counts_used = false;
  O->start = s->cstart;
  O->skey = s->skey;
  O->sslot = s->sslot;
  O->scell = s->scell;
  return PB_OK;
}

int pb_cell_order(pb_sys *s, const PbCellOrder &O, uint32_t ncell) {
  const uint32_t n = s->npad, m = n > ncell + 1 ? n : ncell + 1;
  hipLaunchKernelGGL(k_cell_order, dim3(pb_blocks(m, 256)), dim3(256), 0, s->ctx->stream, O, n,
                     s->perm, s->n, ncell, s->ref_pid, s->ref_bid, s->ref_bindex);
  PB_LAUNCH_CHECK(s->ctx, "k_cell_order");
  return PB_OK;
}
