// pb_internal.h -- shared types of the MI355X particle engine (host + device).
//
// Storage layout (HBM): every per-particle array is indexed by a storage
// slot s in [0, npad).  Each replica owns a 64-aligned slot range
// [atom0, atom0 + npad_r) holding its natoms real particles followed by
// padding slots, so every wavefront belongs to exactly one replica and all
// per-replica reductions are per-wave partials summed in a fixed order.
// Positions are double4 (x, y, z, w = type id), velocities double4
// (x, y, z, w = 1/mass): one 32-byte load brings everything the pair and
// integration kernels need about a particle.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>
#include <string>
#include <vector>
#include "../../include/pbamd.h"

#define PB_WAVE 64
#define PB_PAD_TYPE 0xFFFFu
#define PB_NONE 0xFFFFFFFFu
#define PB_MAXT 5

struct RepInfo {
  double lo[3], hi[3], L[3], Linv[3];
  uint32_t nb[3];      // list-cell grid of this replica (fused path)
  uint32_t cell0;      // first global list cell; the replica's pad cell is cell0 + nb0*nb1*nb2
  uint32_t atom0;      // first storage slot (multiple of 64)
  uint32_t natoms;     // real particles
  uint32_t npad;       // slots (multiple of 64)
  uint32_t wave0, nwave;
  uint32_t seg0, nseg;   // pair-kernel work units (segments) of this replica
  double rlist;          // Verlet list radius of this replica (rc + its skin)
  double half_skin2;     // (skin / 2)^2: a particle beyond it invalidates the list
  float rb2;             // FP32 list-build radius^2 (rlist + rounding margin)^2
  float inv_hs2;         // 1 / (skin / 2)^2 (0 without a skin): displacement scale
};

struct LJTable {
  int ntypes;
  double s2[PB_MAXT * PB_MAXT], e24[PB_MAXT * PB_MAXT], e4[PB_MAXT * PB_MAXT],
      shift[PB_MAXT * PB_MAXT];
  float s2f[PB_MAXT * PB_MAXT], e24f[PB_MAXT * PB_MAXT], e4f[PB_MAXT * PB_MAXT],
      shiftf[PB_MAXT * PB_MAXT];
};

#define PB_RES_DOUBLES 16384u

struct pb_ctx {
  int device = 0;
  hipStream_t stream = nullptr;
  // pinned staging ring of the host boundary (pb_io.hip; 2 MiB, made and
  // released with the context, so that no later call allocates it), its device
  // address and an event per slot
  uint8_t *io_stage = nullptr, *io_dev = nullptr;
  hipEvent_t io_ev[2] = {};
  // small results that kernels write to the host themselves: PB_RES_DOUBLES
  // doubles of pinned memory and their device address; read
  // after the stream's synchronisation that every such call ends with
  double *res = nullptr, *res_dev = nullptr;
  // device address of pb_bin.hip's static g(r) scratch array on this
  // context's device (pb_gr_hist_noalloc); set when the context is created
  void *gr_scratch = nullptr;
  std::string err;
  int cu_count = 0;
  std::string name;
  uint64_t global_mem = 0;
  uint32_t max_threads = 0, max_grid = 0, lds_per_block = 0;
  uint32_t nsys = 0;   // live systems created on this context (destroy refuses while > 0)
};

// device buffer helper
template <typename T>
struct DBuf {
  T *p = nullptr;
  size_t n = 0;
};

struct pb_sys {
  pb_ctx *ctx = nullptr;
  uint32_t nrep = 0, n = 0, npad = 0, nwave = 0;
  std::vector<uint32_t> counts, offsets;   // per replica (original order)
  std::vector<RepInfo> reps;               // host copy
  std::vector<double> cells;               // 6 per replica
  bool cell_set = false;

  // device state (storage order)
  double4 *r = nullptr, *v = nullptr, *a = nullptr, *F = nullptr;
  double4 *w = nullptr, *Lm = nullptr, *T = nullptr;   // rotation (lazy)
  double *radius = nullptr;                            // DEM (lazy)
  uint8_t *move = nullptr;
  uint16_t *type = nullptr;
  uint32_t *orig = nullptr;       // storage slot -> original index (PB_NONE: pad)
  uint32_t order_gen = 1;         // advanced whenever orig is permuted
  uint32_t *waveRep = nullptr;    // wave -> replica
  RepInfo *d_reps = nullptr;
  double *partials = nullptr;     // per-wave partial sums, 4 per wave
  uint32_t *d_counter = nullptr;  // last-block counters / flags (16 words)
  double *d_out = nullptr;        // small reduction outputs (16 per replica)
  std::vector<double> h_out;      // host copy of them where they exceed the context's results
  uint8_t *io = nullptr;          // a packed field in the caller's order (24 B a particle, lazy)

  // reference cell grid (pb_setup_cells), single replica
  bool ref_cells = false;
  int ref_periodic = 1, ref_single = 0;
  uint32_t blocknum[3] = {0, 0, 0};
  float blocklen[6] = {0, 0, 0, 0, 0, 0};
  uint32_t ref_ncell = 0;
  uint32_t *ref_table = nullptr;  // ncell * 27 (or 125)
  uint32_t *ref_bid = nullptr, *ref_pid = nullptr, *ref_bindex = nullptr;
  bool ref_binned = false;

  // counting-sort workspace (shared by pb_bin and the list rebuild)
  uint32_t *cellid = nullptr, *rank = nullptr, *perm = nullptr;
  uint32_t *skey = nullptr, *sslot = nullptr, *scell = nullptr;   // grouped by cell
  uint32_t *ccount = nullptr, *cstart = nullptr;  // ncell_cap + 1
  uint32_t ncell_cap = 0;
  bool counts_used = false;       // a sort began and its scatter, which clears ccount, was not launched
  uint32_t *scan_tmp = nullptr;
  size_t scan_tmp_n = 0;

  // LJ
  LJTable lj{};
  bool lj_set = false;
  double rc2 = 0.0;
  int shifted = 0;
  LJTable *d_lj = nullptr;

  // fused path: Verlet list
  uint16_t *nl = nullptr;          // window-local indices, entry k of slot s at nl[k * npad + s]
  uint32_t *nn = nullptr;          // list length per slot
  uint32_t maxnb = 0;              // list capacity
  float4 *rbuild = nullptr;
  double4 *r2buf = nullptr, *v2buf = nullptr;   // ping-pong partners
  uint32_t *orig2 = nullptr;
  uint16_t *type2 = nullptr;
  uint8_t *move2 = nullptr;
  double4 *a2buf = nullptr;
  uint32_t list_ncell = 0;
  double list_rlist = 0.0;         // largest list radius over the replicas
  uint32_t *list_segs = nullptr;   // list-build work units (8 words each)
  bool list_thin = false;         // some replica is one whole segment
  uint32_t list_nsegs = 0;
  uint4 *list_wtab = nullptr;      // per-segment window tables (cell order of the last sort)
  uint32_t list_wtab_cap = 0;      // segments list_wtab holds
  uint32_t list_segs_cap = 0;      // segments list_segs holds
  uint32_t partials_cap = 0;       // records `partials` holds
  // what the list cells and segments were laid out for (plan_lanes 0: none)
  uint32_t plan_lanes = 0, plan_tile_w = 0;
  double plan_rc = 0, plan_fill = 0;
  std::vector<double> plan_skins;
  double *lj_ebuf = nullptr;       // energy records
  size_t lj_ebuf_cap = 0;
  uint32_t tile_w = 2;             // list-cell columns per tile side (1 or 2)
  double tile_fill = 0.72;         // target fill of the LDS window stage
  // Continuation of the fused LJ run: the cell order, Verlet list and list
  // cells left by the last pb_lj_run stay valid for the next one when the
  // positions and the storage order are exactly those that run left (a
  // fingerprint of r and orig) and the list parameters are unchanged.  Any
  // sort (pb_counting_sort) clears lj_cont.
  bool lj_cont = false;
  uint64_t lj_cont_hash = 0;       // fingerprint of r, orig at the end of the run
  double lj_cont_rc2 = 0, lj_cont_fill = 0;
  uint32_t lj_cont_tile_w = 0, lj_cont_lanes = 0;
  std::vector<double> lj_cont_skins;
  uint32_t lj_cont_since = 0;      // steps since the list was built
  uint32_t lj_cont_d2 = 0, lj_cont_v2 = 0;   // displacement / speed maxima (float bits)
  unsigned long long *d_hash = nullptr;
  uint32_t *lj_queue = nullptr;    // persistent step kernel: 8 work queues + exit counter
  uint32_t last_rebuilds = 0, last_maxnn = 0;
  int last_skin_violation = 0;
  double last_step_ms = 0.0, last_rebuild_ms = 0.0;
  uint32_t last_nstep_timed = 0, last_nrebuild_timed = 0;
  // host-mapped ring through which step kernels publish the previous step's
  // max displacement / speed (drives the rebuild schedule without a sync)
  uint32_t *hmon = nullptr, *dmon = nullptr;

  // Gaussian thermostat: per replica {xi, 1/c} of the last step, and the
  // count of steps whose implicit velocity equation had no solution
  double *gt = nullptr;
  double *gt_part = nullptr;       // partials of its second pass, one set a wavefront
  uint32_t *gt_bad = nullptr;

  // MD neighbour list (cudaParticleMD::makeNList): CSR by original index
  uint32_t *md_row = nullptr, *md_col = nullptr, *md_inv = nullptr;
  uint32_t *md_cnt = nullptr;      // row lengths
  float4 *md_pos = nullptr;        // cell order: FP32 position, original index
  uint32_t md_cap = 0, md_nnz = 0;
  uint32_t md_inv_order = 0;       // order_gen md_inv was made for (0: none)
  bool md_valid = false;

  // g(r)
  uint64_t *gr_hist = nullptr;     // histograms, replica table, rstep
  size_t gr_cap = 0;               // bytes

  // SPH (cudaParticleSPH_NS), storage order unless noted
  double *sph_mu0 = nullptr, *sph_c2 = nullptr, *sph_rhoinv = nullptr;
  double4 *sph_num = nullptr;                  // (number density, rho, mu or p, 0)
  double4 *sph_rs = nullptr, *sph_vs = nullptr;   // cell-sorted views
  double2 *sph_ds = nullptr;
  double *sph_mus = nullptr;
  float4 *sph_fq = nullptr;
  double sph_h = 0.0, sph_rho0 = 1.0;
  bool sph_set = false, sph_dens = false;
  // 0: reference physics (Lucy, linear EOS, mu); 1: weakly compressible
  // config physics (cubic spline, Tait, artificial viscosity)
  int sph_kind = 0;
  double sph_c0 = 0.0, sph_gamma = 7.0, sph_alpha = 0.0, sph_pmin = 0.0;

  // DEM (cudaParticleDEM, cudaParticleRotation)
  double *m0inv = nullptr;                     // minv / (0.4 r0^2), storage order
  double dem_E = 0, dem_mu = 0, dem_s2 = 0, dem_gamma2 = 0, dem_mu_r = 0;
  bool dem_set = false;
  // contact law: 0 = the reference's Hertz law (scalar history per contact),
  // 1 = linear spring-dashpot + tangential spring (3 doubles per contact)
  int dem_law = 0;
  uint32_t dem_hw = 1;                         // history doubles per contact
  double dem_kn = 0, dem_zeta = 0, dem_kt = 0;
  // contact CSR by original index, double-buffered for the tangential history
  uint32_t *cm_row[2] = {nullptr, nullptr}, *cm_col[2] = {nullptr, nullptr};
  double *cm_val[2] = {nullptr, nullptr};
  uint32_t cm_cap[2] = {0, 0}, cm_nnz[2] = {0, 0};
  int cm_cur = -1;                             // buffer of the latest CSR, -1 before any
  bool cm_prev = false;                        // the other buffer holds the matrix before it
  bool cm_rewound = false;                     // the last matrix operation was pb_dem_rewind
  uint32_t *dem_inv = nullptr;                 // original index -> storage slot
  uint32_t dem_inv_order = 0;                  // order_gen dem_inv was made for (0: none)
  double4 *dem_rs = nullptr;                   // cell order: (x, y, z, radius)
  float4 *dem_fq = nullptr;                    // the same in FP32
  uint32_t *dem_rowbuf = nullptr;              // contacts kept by the counting scan
  uint32_t dem_bad = 0;                        // Cundall-Strack violations of the last call
};

// --------------------------------------------------------------- host util
int pb_fail(pb_ctx *ctx, int code, const std::string &msg);
int pb_hip_check(pb_ctx *ctx, hipError_t e, const char *what);
#define PB_HIP(ctx, call)                                              \
  do {                                                                 \
    hipError_t _e = (call);                                            \
    if (_e != hipSuccess) return pb_hip_check((ctx), _e, #call);       \
  } while (0)
#define PB_LAUNCH_CHECK(ctx, what)                                     \
  do {                                                                 \
    hipError_t _e = hipGetLastError();                                 \
    if (_e != hipSuccess) return pb_hip_check((ctx), _e, what);        \
  } while (0)

template <typename T>
int pb_alloc(pb_ctx *ctx, T **p, size_t n) {
  if (*p) {
    (void)hipFree(*p);
    *p = nullptr;
  }
  if (n == 0) n = 1;
  hipError_t e = hipMalloc((void **)p, sizeof(T) * n);
  if (e != hipSuccess) return pb_hip_check(ctx, e, "hipMalloc");
  return PB_OK;
}
template <typename T>
void pb_free(T *&p) {
  if (p) (void)hipFree(p);
  p = nullptr;
}

static inline uint32_t pb_blocks(size_t n, uint32_t bs) {
  return (uint32_t)((n + bs - 1) / bs);
}

// counting sort helpers (pb_sort.hip)
int pb_ensure_sort_ws(pb_sys *sys, uint32_t ncell);
// exclusive scan of in[0..n) into out[0..n], out[n] = total
int pb_exclusive_scan(pb_sys *sys, const uint32_t *in, uint32_t *out, uint32_t n);
// (key, slot, cell) grouped by cell, in no particular order inside a cell
struct PbCellOrder {
  const uint32_t *start;       // cell -> first position (start[c + 1] ends it)
  const uint32_t *skey, *sslot, *scell;
};
// before a counting kernel: ccount is zero (a sort given up in between leaves
// counts, and ranks on top of them lie past the arrays), and the order of the
// reference cell grid no longer holds
int pb_counts_begin(pb_sys *sys);
// cellid[s] (PB_NONE never), the counts of every cell and the rank of s among
// them given; cells start in sys->cstart
int pb_counting_sort(pb_sys *sys, uint32_t ncell, const uint32_t *key, PbCellOrder *O);
// sys->perm (sorted position -> storage slot, by cell and key) and
// calcBlockID's outputs of the reference cell grid
int pb_cell_order(pb_sys *sys, const PbCellOrder &O, uint32_t ncell);
// per-replica reduction of K = 1 or 2 per-wave partial components into out[rep*8+c]
// (device memory, or the context's small results)
int pb_reduce_waves(pb_sys *sys, int K, double *out);
// the same, waited for, into host[rep*8+c]
int pb_reduce_to_host(pb_sys *sys, int K, const double **host);
// host boundary (pb_io.hip): copies through the context's pinned ring (an
// upload is stream ordered, a download waits); the packed-field device
// buffer; a scalar per particle from the caller's order into storage order
// (squared if asked; padding 0)
int pb_io_upload(pb_ctx *ctx, void *dev, const void *host, size_t bytes);
int pb_io_download(pb_ctx *ctx, void *host, const void *dev, size_t bytes);
int pb_io_buffer(pb_sys *sys);
int pb_io_scatter(pb_sys *sys, const double *host, double *dst, bool square);
// the context's ring, its events and the small-result memory
int pb_io_create(pb_ctx *ctx);
void pb_io_release(pb_ctx *ctx);
// rotation / radius state, allocated on first use
int pb_ensure_rotation(pb_sys *sys);
int pb_gr_scratch_init(pb_ctx *ctx);          // pb_bin.hip: device address of the g(r) scratch
int pb_ensure_radius(pb_sys *sys);

// ------------------------------------------------------------ device util
__device__ __forceinline__ uint32_t pb_lane() { return __lane_id(); }

// Rank of a slot among the slots of cell c counted so far: lanes holding the
// same cell as their left neighbour form a run, whose head does one
// atomicAdd on counts[c] for the whole run and broadcasts the base (one
// atomic per run when the input is nearly cell-ordered).  All lanes of the
// wavefront call it; invalid lanes pass valid = false.
__device__ __forceinline__ uint32_t pb_count_rank(uint32_t c, bool valid, uint32_t *counts) {
  const uint32_t lane = pb_lane();
  const uint32_t left = __shfl_up(c, 1, 64);
  const bool head = valid && (lane == 0 || left != c);
  const uint64_t heads = __ballot(head);
  const uint64_t validm = __ballot(valid);
  // my run head: highest head lane <= lane
  const uint64_t le = heads & ((lane == 63) ? ~0ull : ((2ull << lane) - 1ull));
  const uint32_t hl = le ? (63u - (uint32_t)__clzll((long long)le)) : 0u;
  // run length (for heads): distance to the next head or the end of valid lanes
  uint32_t base = 0;
  if (head) {
    const uint64_t gt = heads & ~((lane == 63) ? ~0ull : ((2ull << lane) - 1ull));
    const uint32_t nextl = gt ? (uint32_t)__ffsll((long long)gt) - 1u : (uint32_t)__popcll(validm);
    base = atomicAdd(&counts[c], nextl - lane);
  }
  base = __shfl(base, (int)hl, 64);
  return base + (lane - hl);
}

// Sorted position of the pair at i: its cell's start plus the number of
// smaller keys in the cell.  Equal keys, which only the padding slots of a
// replica have, keep the order they stand in: their rows are all alike.
// Lanes of a wavefront share cells, so the reads are mostly broadcast L1 hits;
// eight are in flight at a time.
__device__ __forceinline__ uint32_t pb_cell_position(const PbCellOrder &O, uint32_t i,
                                                     uint32_t *slot, uint32_t *cell) {
  const uint32_t k = O.skey[i], c = O.scell[i];
  const uint32_t b = O.start[c], e = O.start[c + 1];
  uint32_t rank = 0;
  for (uint32_t j = b; j < e; j += 8) {
    uint32_t q[8];
#pragma unroll
    for (uint32_t u = 0; u < 8; ++u) q[u] = O.skey[min(j + u, e - 1u)];
#pragma unroll
    for (uint32_t u = 0; u < 8; ++u)
      rank += (j + u < e && (q[u] < k || (q[u] == k && j + u < i))) ? 1u : 0u;
  }
  *slot = O.sslot[i];
  *cell = c;
  return b + rank;
}

__device__ __forceinline__ double pb_wave_sum(double x) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) x += __shfl_xor(x, o, 64);
  return x;
}
__device__ __forceinline__ uint32_t pb_wave_sum_u32(uint32_t x) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) x += (uint32_t)__shfl_xor((int)x, o, 64);
  return x;
}
// LDS written by some lanes of a wavefront and read by others of it: LDS
// operations of one wavefront complete in order, so only the compiler is held
__device__ __forceinline__ void pb_wave_lds_sync() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

// XCD-aware logical block of a 1-D grid (MI355X dispatches workgroups
// round-robin over its 8 XCDs, each with its own L2): within every 64
// workgroups, XCD x takes 8 consecutive logical blocks (the tail past the
// last whole 64 keeps its order).  Neighbouring blocks share an XCD's L2 in eights while
// dense and sparse regions stay spread over all XCDs.  Bijective.
__device__ __forceinline__ uint32_t pb_xcd_chunk8() {
  const uint32_t b = blockIdx.x, full = gridDim.x & ~63u;
  return b < full ? (b & ~63u) + (b & 7u) * 8u + ((b >> 3) & 7u) : b;
}

// the same with C consecutive logical blocks a XCD within every 8 C
template <uint32_t C>
__device__ __forceinline__ uint32_t pb_xcd_chunk() {
  const uint32_t b = blockIdx.x, full = gridDim.x / (8u * C) * (8u * C);
  return b < full ? b / (8u * C) * (8u * C) + (b & 7u) * C + (b >> 3) % C : b;
}

__device__ __forceinline__ double pb_load_relaxed(const double *p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// replicas from which a reduction takes a wavefront for each (and callers a
// workgroup of 1024)
constexpr uint32_t PB_REDUCE_WAVES = 4;
// The order of a replica's sum is the same in every form that takes it, so its
// bits don't depend on the other replicas: partial w goes to running sum w mod
// 256, sums l, l + 64, l + 128 and l + 192 are added in pairs to lane l's, and the
// lanes' by pb_wave_sum.
constexpr uint32_t PB_REDUCE_SUMS = 256;

// a wavefront's part of it: Q replicas (first partial w0, number nw) at once, the
// sums of their K components in every lane
template <int K, uint32_t Q>
__device__ __forceinline__ void pb_wave_reduce(const double *partials, const uint32_t (&w0)[Q],
                                               const uint32_t (&nw)[Q], double (&out)[Q][K]) {
  constexpr uint32_t J = PB_REDUCE_SUMS / PB_WAVE;
  uint32_t most = 0;
#pragma unroll
  for (uint32_t k = 0; k < Q; ++k) most = max(most, nw[k]);
  double acc[J][Q][K] = {};
  for (uint32_t w = pb_lane(); w < most; w += PB_REDUCE_SUMS)
#pragma unroll
    for (uint32_t j = 0; j < J; ++j)
#pragma unroll
      for (uint32_t k = 0; k < Q; ++k)
        if (w + j * PB_WAVE < nw[k])
#pragma unroll
          for (int c = 0; c < K; ++c)
            acc[j][k][c] += partials[4 * (size_t)(w0[k] + w + j * PB_WAVE) + c];
#pragma unroll
  for (uint32_t k = 0; k < Q; ++k)
#pragma unroll
    for (int c = 0; c < K; ++c)
      out[k][c] = pb_wave_sum((acc[0][k][c] + acc[1][k][c]) + (acc[2][k][c] + acc[3][k][c]));
}

// sum of K per-wave partial components for every replica, executed by one
// block (used by the last-block reductions and by k_reduce_waves).
template <int K>
__device__ __forceinline__ void pb_block_reduce_reps(const double *partials, const RepInfo *reps,
                                     uint32_t nrep, double *out, bool by_segment,
                                     double *scratch) {
  // Every replica's partials: one per wave, or one per pair-kernel segment when
  // by_segment.  Callers that read partials written by other workgroups issue a
  // device-scope fence first (it invalidates this CU's vector L1), so plain loads
  // are coherent.  scratch: 4 x 256 doubles of the caller's LDS
  double (*sm)[256] = reinterpret_cast<double (*)[256]>(scratch);
  const uint32_t t = threadIdx.x, bs = blockDim.x, lane = pb_lane();
  const RepInfo &last = reps[nrep - 1u];
  const uint32_t parts = by_segment ? last.seg0 + last.nseg : last.wave0 + last.nwave;
  if (nrep >= PB_REDUCE_WAVES && parts / 2048u < nrep) {   // a product would wrap from 2^21 replicas
    // a wavefront a replica, two of them and eight partials a lane in flight (mv2
    // of 256 replicas of 8000 particles: a thread a replica, a chain of its
    // partials, 125 us a call, this 45; 15 of 500 to 4000: one after the other by
    // the whole workgroup 37.5, this 18.4).  Few replicas of very many partials
    // keep the whole workgroup on each (4 of 400,000 particles: 55 us a call
    // against 56).
    constexpr uint32_t Q = 2;
    const uint32_t nwv = bs / PB_WAVE;
    for (uint32_t q0 = t / PB_WAVE; q0 < nrep; q0 += nwv * Q) {
      uint32_t w0[Q], nw[Q];
#pragma unroll
      for (uint32_t k = 0; k < Q; ++k) {
        const RepInfo &R = reps[min(q0 + k * nwv, nrep - 1u)];
        w0[k] = by_segment ? R.seg0 : R.wave0;
        nw[k] = q0 + k * nwv < nrep ? (by_segment ? R.nseg : R.nwave) : 0u;
      }
      double x[Q][K];
      pb_wave_reduce<K>(partials, w0, nw, x);
#pragma unroll
      for (uint32_t k = 0; k < Q; ++k)
#pragma unroll
        for (int c = 0; c < K; ++c)
          if (lane == 0 && q0 + k * nwv < nrep) out[8 * (q0 + k * nwv) + c] = x[k][c];
    }
    return;
  }
  // the first 256 threads hold the running sums (any block size >= 256 may call
  // this), a wavefront a component adds them
  const uint32_t T = PB_REDUCE_SUMS;
  for (uint32_t q = 0; q < nrep; ++q) {
    const uint32_t w0 = by_segment ? reps[q].seg0 : reps[q].wave0;
    const uint32_t nw = by_segment ? reps[q].nseg : reps[q].nwave;
    double acc[K] = {};
    if (t < T) {
      for (uint32_t w = t; w < nw; w += T)
#pragma unroll
        for (int c = 0; c < K; ++c) acc[c] += partials[4 * (size_t)(w0 + w) + c];
#pragma unroll
      for (int c = 0; c < K; ++c) sm[c][t] = acc[c];
    }
    __syncthreads();
    const uint32_t c = t / PB_WAVE;
    if (c < (uint32_t)K) {
      const double x = pb_wave_sum((sm[c][lane] + sm[c][lane + 64]) + (sm[c][lane + 128] + sm[c][lane + 192]));
      if (lane == 0) out[8 * q + c] = x;
    }
    __syncthreads();
  }
}

// applyPeriodicCondition_F4 (kernelfuncs.cu:95-129) in FP64; a value that
// rounds onto the upper face is put on the lower one.
__device__ __forceinline__ double wrap1(double x, double c0, double c1) {
  const double L = c1 - c0;
  const double d0 = c0 - x;
  if (d0 > 0) x += (double)((int)(d0 / L) + 1) * L;
  const double d1 = x - c1;
  if (d1 >= 0) x -= (double)((int)(d1 / L) + 1) * L;
  if (x >= c1) x = c0;
  return x;
}
