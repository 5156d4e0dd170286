// pb_core.hip -- context, particle storage, integrators,
// boundaries and FP64 reductions of the MI355X particle engine.
//
// Reference counterparts: cudaFrame (cudaFrame.cu), cudaParticleBase
// (cudaParticleBase.cu), cudaParticleVV (cudaParticleVV.cu), cudaParticleLF
// (cudaParticleLF.cu) and the element-wise kernels of kernelfuncs.cu.
#include "pb_internal.h"
#include <algorithm>
#include <cmath>
#include <cstring>

int pb_fail(pb_ctx *ctx, int code, const std::string &msg) {
  if (ctx) ctx->err = msg;
  return code;
}
int pb_hip_check(pb_ctx *ctx, hipError_t e, const char *what) {
  std::string m = std::string(what) + ": " + hipGetErrorString(e);
  return pb_fail(ctx, PB_ERR_HIP, m);
}

// ================================================================= context
extern "C" int pb_ctx_create(int device, pb_ctx **out) {
  if (!out) return PB_ERR_ARG;
  *out = nullptr;
  int ndev = 0;
  if (hipGetDeviceCount(&ndev) != hipSuccess || ndev <= 0) return PB_ERR_HIP;
  if (device < 0 || device >= ndev) return PB_ERR_ARG;
  pb_ctx *c = new pb_ctx();
  c->device = device;
  if (hipSetDevice(device) != hipSuccess) {
    delete c;
    return PB_ERR_HIP;
  }
  hipDeviceProp_t prop;
  if (hipGetDeviceProperties(&prop, device) == hipSuccess) {
    c->cu_count = prop.multiProcessorCount;
    c->name = prop.gcnArchName;
    c->global_mem = (uint64_t)prop.totalGlobalMem;
    c->max_threads = (uint32_t)prop.maxThreadsPerBlock;
    c->max_grid = (uint32_t)prop.maxGridSize[0];
    c->lds_per_block = (uint32_t)prop.sharedMemPerBlock;
  }
  // default-priority stream (never a different priority)
  if (hipStreamCreateWithFlags(&c->stream, hipStreamNonBlocking) != hipSuccess) {
    delete c;
    return PB_ERR_HIP;
  }
  if (pb_gr_scratch_init(c) != PB_OK || pb_io_create(c) != PB_OK) {
    pb_io_release(c);
    (void)hipStreamDestroy(c->stream);
    delete c;
    return PB_ERR_HIP;
  }
  *out = c;
  return PB_OK;
}

extern "C" int pb_ctx_destroy(pb_ctx *ctx) {
  if (!ctx) return PB_ERR_ARG;
  // a system keeps its context's device and stream: destroying the context
  // first would leave every later call on the system (its destroy included)
  // with a freed context
  if (ctx->nsys)
    return pb_fail(ctx, PB_ERR_STATE,
                   "pb_ctx_destroy: " + std::to_string(ctx->nsys) +
                       " system(s) still alive on this context; pb_sys_destroy them first");
  (void)hipSetDevice(ctx->device);
  if (ctx->stream) {
    (void)hipStreamSynchronize(ctx->stream);
    pb_io_release(ctx);
    (void)hipStreamDestroy(ctx->stream);
  }
  delete ctx;
  return PB_OK;
}

extern "C" const char *pb_ctx_last_error(const pb_ctx *ctx) {
  return ctx ? ctx->err.c_str() : "null context";
}

extern "C" int pb_ctx_sync(pb_ctx *ctx) {
  if (!ctx) return PB_ERR_ARG;
  PB_HIP(ctx, hipStreamSynchronize(ctx->stream));
  return PB_OK;
}

extern "C" int pb_ctx_info(pb_ctx *ctx, char *name, size_t name_len, int *cu_count) {
  if (!ctx) return PB_ERR_ARG;
  if (name && name_len) {
    std::strncpy(name, ctx->name.c_str(), name_len - 1);
    name[name_len - 1] = 0;
  }
  if (cu_count) *cu_count = ctx->cu_count;
  return PB_OK;
}

extern "C" int pb_ctx_limits(pb_ctx *ctx, uint64_t *global_mem, uint32_t *max_threads,
                             uint32_t *max_grid, uint32_t *lds_per_block,
                             uint32_t *lanes_per_cu) {
  if (!ctx) return PB_ERR_ARG;
  if (global_mem) *global_mem = ctx->global_mem;
  if (max_threads) *max_threads = ctx->max_threads;
  if (max_grid) *max_grid = ctx->max_grid;
  if (lds_per_block) *lds_per_block = ctx->lds_per_block;
  // a CDNA compute unit issues to 4 SIMDs of 16 lanes each
  if (lanes_per_cu) *lanes_per_cu = 64;
  return PB_OK;
}

// ================================================================== system
extern "C" int pb_sys_create(pb_ctx *ctx, uint32_t nrep, const uint32_t *counts,
                             pb_sys **out) {
  if (!ctx || !out || nrep == 0 || !counts) return pb_fail(ctx, PB_ERR_ARG, "pb_sys_create: bad args");
  *out = nullptr;
  uint64_t total = 0, totpad = 0;
  for (uint32_t q = 0; q < nrep; ++q) {
    if (counts[q] == 0) return pb_fail(ctx, PB_ERR_ARG, "pb_sys_create: empty replica");
    total += counts[q];
    totpad += (counts[q] + PB_WAVE - 1) / PB_WAVE * PB_WAVE;
  }
  if (totpad >= (1ull << 31)) return pb_fail(ctx, PB_ERR_ARG, "pb_sys_create: too many particles");
  PB_HIP(ctx, hipSetDevice(ctx->device));
  pb_sys *s = new pb_sys();
  s->ctx = ctx;
  ++ctx->nsys;
  s->nrep = nrep;
  s->n = (uint32_t)total;
  s->npad = (uint32_t)totpad;
  s->nwave = s->npad / PB_WAVE;
  s->counts.assign(counts, counts + nrep);
  s->offsets.resize(nrep);
  s->reps.resize(nrep);
  s->cells.assign(6 * (size_t)nrep, 0.0);
  uint32_t off = 0, slot = 0;
  for (uint32_t q = 0; q < nrep; ++q) {
    RepInfo &R = s->reps[q];
    std::memset(&R, 0, sizeof(R));
    s->offsets[q] = off;
    R.atom0 = slot;
    R.natoms = counts[q];
    R.npad = (counts[q] + PB_WAVE - 1) / PB_WAVE * PB_WAVE;
    R.wave0 = slot / PB_WAVE;
    R.nwave = R.npad / PB_WAVE;
    off += counts[q];
    slot += R.npad;
  }
  int rc = PB_OK;
  const size_t np = s->npad;
  if ((rc = pb_alloc(ctx, &s->r, np)) || (rc = pb_alloc(ctx, &s->v, np)) ||
      (rc = pb_alloc(ctx, &s->a, np)) || (rc = pb_alloc(ctx, &s->F, np)) ||
      (rc = pb_alloc(ctx, &s->move, np)) || (rc = pb_alloc(ctx, &s->type, np)) ||
      (rc = pb_alloc(ctx, &s->orig, np)) || (rc = pb_alloc(ctx, &s->waveRep, s->nwave)) ||
      (rc = pb_alloc(ctx, &s->d_reps, nrep)) ||
      (rc = pb_alloc(ctx, &s->partials, 4 * (size_t)s->nwave)) ||
      (rc = pb_alloc(ctx, &s->d_counter, 16)) || (rc = pb_alloc(ctx, &s->d_out, 16 * (size_t)nrep)) ||
      (rc = pb_alloc(ctx, &s->d_lj, 1))) {
    pb_sys_destroy(s);
    return rc;
  }
  s->partials_cap = s->nwave;
  std::vector<uint32_t> wr(s->nwave);
  for (uint32_t q = 0; q < nrep; ++q)
    for (uint32_t k = 0; k < s->reps[q].nwave; ++k) wr[s->reps[q].wave0 + k] = q;
  std::vector<uint32_t> orig(np, PB_NONE);
  for (uint32_t q = 0; q < nrep; ++q)
    for (uint32_t i = 0; i < counts[q]; ++i) orig[s->reps[q].atom0 + i] = s->offsets[q] + i;
  std::vector<uint16_t> ty(np, (uint16_t)PB_PAD_TYPE);
  for (uint32_t q = 0; q < nrep; ++q)
    for (uint32_t i = 0; i < counts[q]; ++i) ty[s->reps[q].atom0 + i] = 0;
  hipStream_t st = ctx->stream;
  if (hipMemcpyAsync(s->waveRep, wr.data(), 4 * wr.size(), hipMemcpyHostToDevice, st) ||
      hipMemcpyAsync(s->orig, orig.data(), 4 * np, hipMemcpyHostToDevice, st) ||
      hipMemcpyAsync(s->type, ty.data(), 2 * np, hipMemcpyHostToDevice, st) ||
      hipMemsetAsync(s->r, 0, sizeof(double4) * np, st) ||
      hipMemsetAsync(s->v, 0, sizeof(double4) * np, st) ||
      hipMemsetAsync(s->a, 0, sizeof(double4) * np, st) ||
      hipMemsetAsync(s->F, 0, sizeof(double4) * np, st) ||
      hipMemsetAsync(s->move, 0, np, st) ||
      hipMemsetAsync(s->d_counter, 0, 16 * 4, st) ||
      hipStreamSynchronize(st)) {
    pb_sys_destroy(s);
    return pb_fail(ctx, PB_ERR_HIP, "pb_sys_create: upload failed");
  }
  *out = s;
  return PB_OK;
}

extern "C" void pb_sys_destroy(pb_sys *s) {
  if (!s) return;
  if (s->ctx) {
    (void)hipSetDevice(s->ctx->device);
    (void)hipStreamSynchronize(s->ctx->stream);
  }
  pb_free(s->r); pb_free(s->v); pb_free(s->a); pb_free(s->F);
  pb_free(s->w); pb_free(s->Lm); pb_free(s->T); pb_free(s->radius);
  pb_free(s->move); pb_free(s->type); pb_free(s->orig); pb_free(s->waveRep);
  pb_free(s->d_reps); pb_free(s->partials); pb_free(s->d_counter); pb_free(s->d_out);
  pb_free(s->d_hash); pb_free(s->lj_queue); pb_free(s->io);
  pb_free(s->gt); pb_free(s->gt_bad); pb_free(s->gt_part);
  pb_free(s->md_row); pb_free(s->md_col); pb_free(s->md_inv);
  pb_free(s->md_cnt); pb_free(s->md_pos);
  pb_free(s->ref_table); pb_free(s->ref_bid); pb_free(s->ref_pid); pb_free(s->ref_bindex);
  pb_free(s->cellid); pb_free(s->rank); pb_free(s->perm); pb_free(s->ccount);
  pb_free(s->skey); pb_free(s->sslot); pb_free(s->scell);
  pb_free(s->cstart); pb_free(s->scan_tmp); pb_free(s->d_lj);
  pb_free(s->nl); pb_free(s->nn); pb_free(s->rbuild); pb_free(s->r2buf); pb_free(s->v2buf);
  pb_free(s->orig2); pb_free(s->type2); pb_free(s->move2); pb_free(s->a2buf);
  pb_free(s->sph_mu0); pb_free(s->sph_c2); pb_free(s->sph_rhoinv); pb_free(s->sph_num);
  pb_free(s->sph_rs); pb_free(s->sph_vs); pb_free(s->sph_ds); pb_free(s->sph_mus); pb_free(s->sph_fq); pb_free(s->m0inv);
  pb_free(s->dem_inv); pb_free(s->dem_rs); pb_free(s->dem_fq); pb_free(s->dem_rowbuf);
  for (int b = 0; b < 2; ++b) {
    pb_free(s->cm_row[b]); pb_free(s->cm_col[b]); pb_free(s->cm_val[b]);
  }
  pb_free(s->gr_hist);
  pb_free(s->list_segs); pb_free(s->list_wtab); pb_free(s->lj_ebuf);
  if (s->hmon) (void)hipHostFree(s->hmon);
  if (s->ctx) --s->ctx->nsys;
  delete s;
}

extern "C" uint32_t pb_sys_count(const pb_sys *s) { return s ? s->n : 0; }
extern "C" uint32_t pb_sys_replicas(const pb_sys *s) { return s ? s->nrep : 0; }

static int upload_reps(pb_sys *s) {
  PB_HIP(s->ctx, hipMemcpyAsync(s->d_reps, s->reps.data(), sizeof(RepInfo) * s->nrep,
                                hipMemcpyHostToDevice, s->ctx->stream));
  return PB_OK;
}

extern "C" int pb_sys_set_cell(pb_sys *s, const double *cells) {
  if (!s || !cells) return PB_ERR_ARG;
  // nothing is written before all boxes are known to be good
  for (size_t k = 0; k < 3 * (size_t)s->nrep; ++k)
    if (!(cells[2 * k + 1] > cells[2 * k])) return pb_fail(s->ctx, PB_ERR_ARG, "pb_sys_set_cell: empty box");
  for (uint32_t q = 0; q < s->nrep; ++q) {
    RepInfo &R = s->reps[q];
    for (int a = 0; a < 3; ++a) {
      const double lo = cells[6 * q + 2 * a], hi = cells[6 * q + 2 * a + 1];
      R.lo[a] = lo;
      R.hi[a] = hi;
      R.L[a] = hi - lo;
      R.Linv[a] = 1.0 / (hi - lo);
    }
  }
  std::memcpy(s->cells.data(), cells, sizeof(double) * 6 * s->nrep);
  s->cell_set = true;
  s->lj_cont = false;             // the fused LJ run's list cells follow the box
  s->plan_lanes = 0;
  return upload_reps(s);
}

int pb_ensure_rotation(pb_sys *s) {
  if (s->w) return PB_OK;
  int rc;                                  // w last: the others exist where it does
  if ((rc = pb_alloc(s->ctx, &s->Lm, s->npad)) || (rc = pb_alloc(s->ctx, &s->T, s->npad)) ||
      (rc = pb_alloc(s->ctx, &s->w, s->npad)))
    return rc;
  hipStream_t st = s->ctx->stream;
  PB_HIP(s->ctx, hipMemsetAsync(s->w, 0, sizeof(double4) * s->npad, st));
  PB_HIP(s->ctx, hipMemsetAsync(s->Lm, 0, sizeof(double4) * s->npad, st));
  PB_HIP(s->ctx, hipMemsetAsync(s->T, 0, sizeof(double4) * s->npad, st));
  return PB_OK;
}
int pb_ensure_radius(pb_sys *s) {
  if (s->radius) return PB_OK;
  int rc = pb_alloc(s->ctx, &s->radius, s->npad);
  if (rc) return rc;
  PB_HIP(s->ctx, hipMemsetAsync(s->radius, 0, sizeof(double) * s->npad, s->ctx->stream));
  return PB_OK;
}

// ======================================================= element-wise kernels
// All take the storage slot range [0, npad) and skip padding slots via
// orig[s] == PB_NONE.

__global__ void k_clear4(double4 *x, uint32_t n) {
  const uint32_t s = blockIdx.x * blockDim.x + threadIdx.x;
  if (s < n) x[s] = make_double4(0, 0, 0, 0);
}

// x y z of *p where any bit of them changed: the passes below leave most
// particles as they are (walls, or nothing beyond the boundary), and a wavefront
// that stores nothing costs no write traffic (bound by memory; 796,176 particles,
// 37 % fixed: leap-frog 22.6 -> 17.4 us, absolute boundary 12.8 -> 6.2)
__device__ __forceinline__ void store_changed(double4 *p, const double4 &was, const double4 &is) {
  if (__double_as_longlong(was.x) != __double_as_longlong(is.x) ||
      __double_as_longlong(was.y) != __double_as_longlong(is.y) ||
      __double_as_longlong(was.z) != __double_as_longlong(is.z))
    *p = is;
}

__global__ void k_add_axis(double4 *x, const uint32_t *orig, uint32_t n, int axis, double val) {
  // addArray_F4 (value), kernelfuncs.cu:27-38
  const uint32_t s = blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= n || orig[s] == PB_NONE) return;
  reinterpret_cast<double *>(x + s)[axis] += val;
}

__global__ void k_calc_acc(double4 *a, const double4 *F, const double4 *v,
                           const uint32_t *orig, uint32_t n) {
  // calcA_F4, kernelfuncs.cu:70-82
  const uint32_t s = blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= n || orig[s] == PB_NONE) return;
  const double mi = v[s].w;
  const double4 f = F[s];
  *reinterpret_cast<double2 *>(&a[s].x) = make_double2(f.x * mi, f.y * mi);   // w stays, unread
  a[s].z = f.z * mi;
}

__global__ void k_vv_step(double4 *r, double4 *v, const double4 *F, double4 *Fold,
                          const uint32_t *orig, uint32_t n, double dt) {
  // propagateVelocityVerlet_F4, kernelfuncs.cu:333-367 (FP64)
  const uint32_t s = blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= n || orig[s] == PB_NONE) return;
  const double dt2 = dt * 0.5;
  double4 V = v[s];
  const double dtm2 = dt2 * V.w;
  const double4 f = F[s];
  const double4 fo = Fold[s];
  V.x += (f.x + fo.x) * dtm2;
  V.y += (f.y + fo.y) * dtm2;
  V.z += (f.z + fo.z) * dtm2;
  const double dt22 = dtm2 * dt;
  double4 R = r[s];
  R.x += V.x * dt + f.x * dt22;
  R.y += V.y * dt + f.y * dt22;
  R.z += V.z * dt + f.z * dt22;
  Fold[s] = make_double4(f.x, f.y, f.z, 0.0);
  v[s] = V;
  r[s] = R;
}

__global__ void k_euler_step(double4 *r, double4 *v, const double4 *a, const uint8_t *move,
                             const uint32_t *orig, uint32_t n, double dt) {
  // propagateEuler_F4, kernelfuncs.cu:174-192 (FP64): r += v dt, v += a dt
  // for movable particles
  const uint32_t s = blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= n || orig[s] == PB_NONE) return;
  const double d = move[s] ? dt : 0.0;
  double4 R = r[s], V = v[s];
  const double4 A = a[s];
  R.x += V.x * d;
  R.y += V.y * d;
  R.z += V.z * d;
  V.x += A.x * d;
  V.y += A.y * d;
  V.z += A.z * d;
  r[s] = R;
  v[s] = V;
}

__global__ void k_wrap(double4 *r, const uint32_t *orig, const uint32_t *waveRep,
                       const RepInfo *reps, uint32_t n) {
  const uint32_t s = blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= n || orig[s] == PB_NONE) return;
  const RepInfo &R = reps[waveRep[s / PB_WAVE]];
  double4 p = r[s];
  p.x = wrap1(p.x, R.lo[0], R.hi[0]);
  p.y = wrap1(p.y, R.lo[1], R.hi[1]);
  p.z = wrap1(p.z, R.lo[2], R.hi[2]);
  r[s] = p;
}

__global__ void k_absolute(double4 *r, const uint32_t *orig, const uint32_t *waveRep,
                           const RepInfo *reps, uint32_t n) {
  // treatAbsoluteBoundary_F4, kernelfuncs.cu:141-155
  const uint32_t s = blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= n || orig[s] == PB_NONE) return;
  const RepInfo &R = reps[waveRep[s / PB_WAVE]];
  const double4 was = r[s];
  double4 p = was;
  p.x = fmin(fmax(p.x, R.lo[0]), R.hi[0]);
  p.y = fmin(fmax(p.y, R.lo[1]), R.hi[1]);
  p.z = fmin(fmax(p.z, R.lo[2]), R.hi[2]);
  store_changed(r + s, was, p);
}

__global__ void k_reflect(const double4 *r, double4 *v, const uint32_t *orig,
                          const uint32_t *waveRep, const RepInfo *reps, uint32_t n) {
  // treatRefrectBoundary_F4, kernelfuncs.cu:157-172
  const uint32_t s = blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= n || orig[s] == PB_NONE) return;
  const RepInfo &R = reps[waveRep[s / PB_WAVE]];
  const double4 p = r[s];
  if (!(p.x < R.lo[0] || p.x > R.hi[0] || p.y < R.lo[1] || p.y > R.hi[1] || p.z < R.lo[2] ||
        p.z > R.hi[2]))
    return;                                     // v unread
  double4 V = v[s];
  if (p.x < R.lo[0]) V.x = fabs(V.x);
  if (p.x > R.hi[0]) V.x = -fabs(V.x);
  if (p.y < R.lo[1]) V.y = fabs(V.y);
  if (p.y > R.hi[1]) V.y = -fabs(V.y);
  if (p.z < R.lo[2]) V.z = fabs(V.z);
  if (p.z > R.hi[2]) V.z = -fabs(V.z);
  v[s] = V;
}

__global__ void k_lf_vinit(double4 *v, const double4 *F, const uint32_t *orig, uint32_t n,
                           double dt_2) {
  // calcLFVinit_F4, kernelfuncs.cu:246-258
  const uint32_t s = blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= n || orig[s] == PB_NONE) return;
  double4 V = v[s];
  const double mi = V.w * dt_2;
  const double4 f = F[s];
  V.x -= f.x * mi;
  V.y -= f.y * mi;
  V.z -= f.z * mi;
  v[s] = V;
}

__global__ void k_lf_step(double4 *r, double4 *v, const double4 *a, const uint8_t *move,
                          const uint32_t *orig, uint32_t n, double dt) {
  // propagateLeapFrog_F4, kernelfuncs.cu:260-284
  const uint32_t s = blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= n || orig[s] == PB_NONE) return;
  const double dt2 = dt * (double)move[s];
  const double4 V0 = v[s], R0 = r[s], A = a[s];
  double4 V = V0, R = R0;
  V.x += A.x * dt2;
  V.y += A.y * dt2;
  V.z += A.z * dt2;
  store_changed(v + s, V0, V);
  R.x += V.x * dt2;
  R.y += V.y * dt2;
  R.z += V.z * dt2;
  store_changed(r + s, R0, R);
}

__global__ void k_lf_rollback(double4 *r, double4 *v, const double4 *a, const uint8_t *move,
                              const uint32_t *orig, uint32_t n, double dt) {
  // rollbackLeapFrog_F4, kernelfuncs.cu:286-327
  const uint32_t s = blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= n || orig[s] == PB_NONE) return;
  const double dt2 = dt * (double)move[s];
  double4 V = v[s];
  double4 R = r[s];
  const double4 A = a[s];
  const double rx = R.x - V.x * dt2, ry = R.y - V.y * dt2, rz = R.z - V.z * dt2;
  V.x -= A.x * dt2;
  V.y -= A.y * dt2;
  V.z -= A.z * dt2;
  v[s] = V;
  R.x = rx - V.x * dt2;
  R.y = ry - V.y * dt2;
  R.z = rz - V.z * dt2;
  r[s] = R;
}

__global__ void k_scale_v(double4 *v, const uint32_t *orig, uint32_t n, double sc) {
  // mulArray on v, kerneltemplate.hh:29-35
  const uint32_t s = blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= n || orig[s] == PB_NONE) return;
  double4 V = v[s];
  V.x *= sc;
  V.y *= sc;
  V.z *= sc;
  v[s] = V;
}

// per-wave partial of m v^2 (calcV2_F4 + DOT, kernelfuncs.cu:520-530,
// cudaParticleMD.cu:124-133)
__global__ void k_mv2_partial(const double4 *v, const uint32_t *orig, uint32_t n,
                              double *partials) {
  const uint32_t s = blockIdx.x * blockDim.x + threadIdx.x;
  double x = 0.0;
  if (s < n && orig[s] != PB_NONE) {
    const double4 V = v[s];
    x = (V.x * V.x + V.y * V.y + V.z * V.z) / V.w;
  }
  x = pb_wave_sum(x);
  if (pb_lane() == 0 && s < n) partials[4 * (s / PB_WAVE)] = x;
}

// inspectV_F4 (kernelfuncs.cu:194-240): max of |v|/vlim with its original index,
// vlim already truncated to an integer; ties go to the lowest index (a total
// order, so the result does not depend on the visiting order).  Workgroups take
// several rounds of v, so that few maxima are left for the second launch; letting
// the workgroup that ends last reduce them took 16 us in all (its release and
// acquire), the two launches 7.4 + 4.3 us at 796,176 particles and 5.1 + 2.6 at
// 200,000 (7.4 + 6.5 and 4.0 + 4.4 with a maximum a wavefront).
constexpr uint32_t INSPECT_BLOCKS = 512;
struct SpeedMax {
  double m = -1.0, id = 1e300;
  __device__ __forceinline__ void take(double x, double i) {
    if (x > m || (x == m && i < id)) {
      m = x;
      id = i;
    }
  }
  __device__ __forceinline__ void block(double (*lds)[2]) {    // the block's, in thread 0
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
      const double x = __shfl_xor(m, o, PB_WAVE), i = __shfl_xor(id, o, PB_WAVE);
      take(x, i);
    }
    if (pb_lane() == 0) {
      lds[threadIdx.x / PB_WAVE][0] = m;
      lds[threadIdx.x / PB_WAVE][1] = id;
    }
    __syncthreads();
    if (threadIdx.x == 0)
      for (uint32_t w = 1; w < blockDim.x / PB_WAVE; ++w) take(lds[w][0], lds[w][1]);
  }
};
__global__ void __launch_bounds__(256) k_inspect(const double4 *v, const uint32_t *orig, uint32_t n,
                                                 double vlim, double *partials) {
  __shared__ double lds[4][2];
  const uint32_t T = gridDim.x * 256u;
  SpeedMax M;
  for (uint32_t s = blockIdx.x * 256u + threadIdx.x; s < n; s += 4u * T) {
    double4 V[4];
    uint32_t o[4];
#pragma unroll
    for (uint32_t u = 0; u < 4; ++u) {
      const uint32_t q = s + u * T < n ? s + u * T : s;
      V[u] = v[q];
      o[u] = orig[q];
    }
#pragma unroll
    for (uint32_t u = 0; u < 4; ++u)
      if (o[u] != PB_NONE)
        M.take(sqrt(V[u].x * V[u].x + V[u].y * V[u].y + V[u].z * V[u].z) / vlim, (double)o[u]);
  }
  M.block(lds);
  if (threadIdx.x == 0) {
    partials[2 * blockIdx.x] = M.m;
    partials[2 * blockIdx.x + 1] = M.id;
  }
}
__global__ void __launch_bounds__(256) k_inspect_final(const double *partials, uint32_t n,
                                                       double *out) {
  __shared__ double lds[4][2];
  SpeedMax M;
#pragma unroll
  for (uint32_t b = threadIdx.x; b < INSPECT_BLOCKS; b += 256u)
    if (b < n) M.take(partials[2 * b], partials[2 * b + 1]);
  M.block(lds);
  if (threadIdx.x == 0) {
    out[0] = M.m;
    out[1] = M.id;
  }
}

// ============================================================ reductions
template <int K>
__global__ void __launch_bounds__(1024) k_reduce_waves(const double *partials, const RepInfo *reps,
                                                      uint32_t nrep, double *out) {
  __shared__ double sm[4 * 256];
  pb_block_reduce_reps<K>(partials, reps, nrep, out, false, sm);
}

int pb_reduce_waves(pb_sys *s, int K, double *out) {
  hipLaunchKernelGGL(K == 1 ? k_reduce_waves<1> : k_reduce_waves<2>, dim3(1),
                     dim3(s->nrep >= PB_REDUCE_WAVES ? 1024 : 256), 0, s->ctx->stream, s->partials,
                     s->d_reps, s->nrep, out);
  PB_LAUNCH_CHECK(s->ctx, "k_reduce_waves");
  return PB_OK;
}

// The reduction kernel writes the sums to pinned memory itself: no copy is
// queued behind it (a copy of a few doubles into pageable memory costs about
// 10 us of host time and a 3 us kernel).
int pb_reduce_to_host(pb_sys *s, int K, const double **host) {
  if (8 * (size_t)s->nrep <= PB_RES_DOUBLES) {
    if (int rc = pb_reduce_waves(s, K, s->ctx->res_dev)) return rc;
    PB_HIP(s->ctx, hipStreamSynchronize(s->ctx->stream));
    *host = s->ctx->res;
    return PB_OK;
  }
  if (int rc = pb_reduce_waves(s, K, s->d_out)) return rc;
  s->h_out.resize(8 * (size_t)s->nrep);
  *host = s->h_out.data();
  return pb_io_download(s->ctx, s->h_out.data(), s->d_out, 8 * sizeof(double) * s->nrep);
}

// ================================================================ wrappers
#define PB_GRID(n) dim3(pb_blocks((n), 256)), dim3(256), 0, s->ctx->stream

extern "C" int pb_clear_force(pb_sys *s, int with_fold) {
  if (!s) return PB_ERR_ARG;
  hipLaunchKernelGGL(k_clear4, PB_GRID(s->npad), s->F, s->npad);
  if (with_fold) hipLaunchKernelGGL(k_clear4, PB_GRID(s->npad), s->a, s->npad);
  PB_LAUNCH_CHECK(s->ctx, "pb_clear_force");
  return PB_OK;
}

extern "C" int pb_calc_acceleration(pb_sys *s) {
  if (!s) return PB_ERR_ARG;
  hipLaunchKernelGGL(k_calc_acc, PB_GRID(s->npad), s->a, s->F, s->v, s->orig, s->npad);
  PB_LAUNCH_CHECK(s->ctx, "pb_calc_acceleration");
  return PB_OK;
}

extern "C" int pb_add_force(pb_sys *s, int axis, double value) {
  if (!s || axis < 0 || axis > 2) return PB_ERR_ARG;
  hipLaunchKernelGGL(k_add_axis, PB_GRID(s->npad), s->F, s->orig, s->npad, axis, value);
  PB_LAUNCH_CHECK(s->ctx, "pb_add_force");
  return PB_OK;
}

extern "C" int pb_add_acceleration(pb_sys *s, int axis, double value) {
  if (!s || axis < 0 || axis > 2) return PB_ERR_ARG;
  hipLaunchKernelGGL(k_add_axis, PB_GRID(s->npad), s->a, s->orig, s->npad, axis, value);
  PB_LAUNCH_CHECK(s->ctx, "pb_add_acceleration");
  return PB_OK;
}

static int need_cell(pb_sys *s) {
  return s->cell_set ? PB_OK : pb_fail(s->ctx, PB_ERR_STATE, "cell not set (pb_sys_set_cell)");
}

extern "C" int pb_treat_periodic(pb_sys *s) {
  if (!s) return PB_ERR_ARG;
  if (int rc = need_cell(s)) return rc;
  hipLaunchKernelGGL(k_wrap, PB_GRID(s->npad), s->r, s->orig, s->waveRep, s->d_reps, s->npad);
  PB_LAUNCH_CHECK(s->ctx, "pb_treat_periodic");
  return PB_OK;
}

extern "C" int pb_treat_absolute(pb_sys *s) {
  if (!s) return PB_ERR_ARG;
  if (int rc = need_cell(s)) return rc;
  hipLaunchKernelGGL(k_absolute, PB_GRID(s->npad), s->r, s->orig, s->waveRep, s->d_reps, s->npad);
  PB_LAUNCH_CHECK(s->ctx, "pb_treat_absolute");
  return PB_OK;
}

extern "C" int pb_treat_reflect(pb_sys *s) {
  if (!s) return PB_ERR_ARG;
  if (int rc = need_cell(s)) return rc;
  hipLaunchKernelGGL(k_reflect, PB_GRID(s->npad), s->r, s->v, s->orig, s->waveRep, s->d_reps,
                     s->npad);
  PB_LAUNCH_CHECK(s->ctx, "pb_treat_reflect");
  return PB_OK;
}

extern "C" int pb_vv_step(pb_sys *s, double dt) {
  if (!s) return PB_ERR_ARG;
  hipLaunchKernelGGL(k_vv_step, PB_GRID(s->npad), s->r, s->v, s->F, s->a, s->orig, s->npad, dt);
  PB_LAUNCH_CHECK(s->ctx, "pb_vv_step");
  return PB_OK;
}

extern "C" int pb_euler_step(pb_sys *s, double dt) {
  if (!s) return PB_ERR_ARG;
  hipLaunchKernelGGL(k_euler_step, PB_GRID(s->npad), s->r, s->v, s->a, s->move, s->orig, s->npad, dt);
  PB_LAUNCH_CHECK(s->ctx, "pb_euler_step");
  return PB_OK;
}

extern "C" int pb_lf_vinit(pb_sys *s, double dt) {
  if (!s) return PB_ERR_ARG;
  // cudaParticleLF::calcVinit passes dt/2 (cudaParticleLF.cu:4-7)
  hipLaunchKernelGGL(k_lf_vinit, PB_GRID(s->npad), s->v, s->F, s->orig, s->npad, dt * 0.5);
  PB_LAUNCH_CHECK(s->ctx, "pb_lf_vinit");
  return PB_OK;
}

extern "C" int pb_lf_step(pb_sys *s, double dt) {
  if (!s) return PB_ERR_ARG;
  hipLaunchKernelGGL(k_lf_step, PB_GRID(s->npad), s->r, s->v, s->a, s->move, s->orig, s->npad, dt);
  PB_LAUNCH_CHECK(s->ctx, "pb_lf_step");
  return PB_OK;
}

extern "C" int pb_lf_rollback(pb_sys *s, double dt) {
  if (!s) return PB_ERR_ARG;
  hipLaunchKernelGGL(k_lf_rollback, PB_GRID(s->npad), s->r, s->v, s->a, s->move, s->orig,
                     s->npad, dt);
  PB_LAUNCH_CHECK(s->ctx, "pb_lf_rollback");
  return PB_OK;
}

extern "C" int pb_scale_velocities(pb_sys *s, double sc) {
  if (!s) return PB_ERR_ARG;
  hipLaunchKernelGGL(k_scale_v, PB_GRID(s->npad), s->v, s->orig, s->npad, sc);
  PB_LAUNCH_CHECK(s->ctx, "pb_scale_velocities");
  return PB_OK;
}

extern "C" int pb_mv2(pb_sys *s, double *out) {
  if (!s || !out) return PB_ERR_ARG;
  hipLaunchKernelGGL(k_mv2_partial, PB_GRID(s->npad), s->v, s->orig, s->npad, s->partials);
  PB_LAUNCH_CHECK(s->ctx, "k_mv2_partial");
  const double *h = nullptr;
  if (int rc = pb_reduce_to_host(s, 1, &h)) return rc;
  for (uint32_t q = 0; q < s->nrep; ++q) out[q] = h[8 * q];
  return PB_OK;
}

extern "C" int pb_inspect_velocity(pb_sys *s, double vlim, double lim_u, double lim_l,
                                   int *result, double *vratio_max, uint32_t *imax) {
  if (!s || !result) return PB_ERR_ARG;
  // inspectV_F4 takes uint32_t vlim (kernelfuncs.h:116): the float limit is
  // truncated before the division.
  const double vl = (double)(uint32_t)(vlim > 0 ? vlim : 0);
  if (vl <= 0) return pb_fail(s->ctx, PB_ERR_ARG, "pb_inspect_velocity: vlim truncates to 0");
  const uint32_t blocks = std::min(pb_blocks(s->npad, 256), INSPECT_BLOCKS);
  hipLaunchKernelGGL(k_inspect, dim3(blocks), dim3(256), 0, s->ctx->stream, s->v, s->orig, s->npad, vl,
                     s->partials);
  hipLaunchKernelGGL(k_inspect_final, dim3(1), dim3(256), 0, s->ctx->stream, s->partials, blocks,
                     s->ctx->res_dev);
  PB_LAUNCH_CHECK(s->ctx, "pb_inspect_velocity");
  PB_HIP(s->ctx, hipStreamSynchronize(s->ctx->stream));
  const double *h = s->ctx->res;
  // float thresholds as the reference's float2 thresh (cudaParticleBase.cu:248-250)
  const double mx = h[0];
  if (mx >= (double)(float)lim_u) *result = 1;
  else if (mx >= (double)(float)lim_l) *result = 0;
  else *result = -1;
  if (vratio_max) *vratio_max = mx;
  if (imax) *imax = (uint32_t)h[1];
  return PB_OK;
}
