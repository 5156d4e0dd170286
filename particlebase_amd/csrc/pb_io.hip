// pb_io.hip -- the host boundary of a particle system: import, get and set
// (cudaParticleBase::import, getPosition & co., cudaParticleBase.cu:68-149).
//
// Host arrays are in the caller's particle order and tightly packed; the
// device keeps storage order and double4 rows.  The reordering and the
// conversion run on the GPU: a field is packed by k_unpack* into a contiguous
// device buffer in the caller's order (or scattered from one by k_pack*), and
// only the caller's bytes cross the bus, through a pinned staging ring of the
// context.  Doing it on the host (download of orig and of the double4 rows
// into fresh pageable vectors, a scalar scatter loop) cost 10.4 ms a field at
// 1,048,576 particles, almost all of it page faults and cache misses of that
// loop; here it takes 0.97 ms, and an
// import of r, v, mass and type 2.7 ms instead of 31.8.
//
// The ring has two slots: the DMA of one chunk runs while the other is copied
// between the slot and the caller's pageable memory, which is what bounds a
// large transfer (25 MB at about 30 GB/s; six threads sharing the chunks
// brought 0.97 ms to 0.87 ms and are not worth their start).  Up to IO_DIRECT
// bytes the kernel writes the pinned memory itself: no DMA, one launch and
// one wait (864 particles: 14 us a field against 30 us through a DMA; equal
// at 32,000).
#include "pb_internal.h"
#include <algorithm>
#include <cstring>

#define IO_CHUNK ((size_t)1 << 20)
#define IO_DIRECT ((size_t)256 << 10)

// ------------------------------------------------------------ staging ring
int pb_io_create(pb_ctx *ctx) {
  auto pinned = [&](void **host, void **dev, size_t bytes) -> int {
    PB_HIP(ctx, hipHostMalloc(host, bytes, hipHostMallocMapped));
    PB_HIP(ctx, hipHostGetDevicePointer(dev, *host, 0));
    return PB_OK;
  };
  int rc;
  if ((rc = pinned((void **)&ctx->io_stage, (void **)&ctx->io_dev, 2 * IO_CHUNK)) ||
      (rc = pinned((void **)&ctx->res, (void **)&ctx->res_dev, sizeof(double) * PB_RES_DOUBLES)))
    return rc;
  for (hipEvent_t &e : ctx->io_ev) PB_HIP(ctx, hipEventCreateWithFlags(&e, hipEventDisableTiming));
  return PB_OK;
}

void pb_io_release(pb_ctx *ctx) {
  if (ctx->res) (void)hipHostFree(ctx->res);
  ctx->res = ctx->res_dev = nullptr;
  if (ctx->io_stage) (void)hipHostFree(ctx->io_stage);
  ctx->io_stage = ctx->io_dev = nullptr;
  for (hipEvent_t &e : ctx->io_ev) {
    if (e) (void)hipEventDestroy(e);
    e = nullptr;
  }
}

// Device to host.  Every DMA that wrote the ring has completed on return.
int pb_io_download(pb_ctx *ctx, void *host, const void *dev, size_t bytes) {
  hipStream_t st = ctx->stream;
  const size_t nchunk = (bytes + IO_CHUNK - 1) / IO_CHUNK;
  for (size_t c = 0; c <= nchunk; ++c) {
    if (c < nchunk) {
      const size_t len = std::min(IO_CHUNK, bytes - c * IO_CHUNK);
      PB_HIP(ctx, hipMemcpyAsync(ctx->io_stage + (c & 1u) * IO_CHUNK,
                                 (const uint8_t *)dev + c * IO_CHUNK, len, hipMemcpyDeviceToHost, st));
      PB_HIP(ctx, hipEventRecord(ctx->io_ev[c & 1u], st));
    }
    if (c > 0) {
      const size_t p = c - 1, len = std::min(IO_CHUNK, bytes - p * IO_CHUNK);
      PB_HIP(ctx, hipEventSynchronize(ctx->io_ev[p & 1u]));
      std::memcpy((uint8_t *)host + p * IO_CHUNK, ctx->io_stage + (p & 1u) * IO_CHUNK, len);
    }
  }
  return PB_OK;
}

// Host to device, stream ordered; the caller's buffer is free on return.  A
// slot's last event tells when the host may write it again (an event that was
// never recorded, or one of a finished download, does not wait).
int pb_io_upload(pb_ctx *ctx, void *dev, const void *host, size_t bytes) {
  hipStream_t st = ctx->stream;
  const size_t nchunk = (bytes + IO_CHUNK - 1) / IO_CHUNK;
  for (size_t c = 0; c < nchunk; ++c) {
    const size_t len = std::min(IO_CHUNK, bytes - c * IO_CHUNK);
    uint8_t *slot = ctx->io_stage + (c & 1u) * IO_CHUNK;
    PB_HIP(ctx, hipEventSynchronize(ctx->io_ev[c & 1u]));
    std::memcpy(slot, (const uint8_t *)host + c * IO_CHUNK, len);
    PB_HIP(ctx, hipMemcpyAsync((uint8_t *)dev + c * IO_CHUNK, slot, len, hipMemcpyHostToDevice, st));
    PB_HIP(ctx, hipEventRecord(ctx->io_ev[c & 1u], st));
  }
  return PB_OK;
}

// device buffer of the packed fields: 24 bytes a particle
int pb_io_buffer(pb_sys *s) {
  if (s->io) return PB_OK;
  return pb_alloc(s->ctx, &s->io, 24 * (size_t)s->n);
}

// ----------------------------------------------------------------- kernels
// One thread a storage slot: the row is read coalesced, the caller's element
// written where orig says (coalesced while storage order is the caller's,
// 24-byte writes after a re-sort); bound by those scattered writes.
__global__ void k_unpack3(const double4 *src, const uint32_t *orig, uint32_t n, double *out) {
  const uint32_t s = blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= n) return;
  const uint32_t o = orig[s];
  if (o == PB_NONE) return;
  const double4 p = src[s];
  double *q = out + 3 * (size_t)o;
  q[0] = p.x;
  q[1] = p.y;
  q[2] = p.z;
}
__global__ void k_unpack_w(const double4 *src, const uint32_t *orig, uint32_t n, double *out) {
  const uint32_t s = blockIdx.x * blockDim.x + threadIdx.x;
  if (s < n && orig[s] != PB_NONE) out[orig[s]] = src[s].w;
}
template <typename T>
__global__ void k_unpack1(const T *src, const uint32_t *orig, uint32_t n, T *out) {
  const uint32_t s = blockIdx.x * blockDim.x + threadIdx.x;
  if (s < n && orig[s] != PB_NONE) out[orig[s]] = src[s];
}
__global__ void k_pack3(const double *in, const uint32_t *orig, uint32_t n, double4 *dst) {
  const uint32_t s = blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= n) return;
  const uint32_t o = orig[s];
  if (o == PB_NONE) return;
  const double *q = in + 3 * (size_t)o;
  dst[s] = make_double4(q[0], q[1], q[2], dst[s].w);
}
__global__ void k_pack_w(const double *in, const uint32_t *orig, uint32_t n, double4 *dst) {
  const uint32_t s = blockIdx.x * blockDim.x + threadIdx.x;
  if (s < n && orig[s] != PB_NONE) dst[s].w = in[orig[s]];
}
// padding slots get 0
template <typename T>
__global__ void k_pack1(const T *in, const uint32_t *orig, uint32_t n, T *dst) {
  const uint32_t s = blockIdx.x * blockDim.x + threadIdx.x;
  if (s < n) dst[s] = orig[s] == PB_NONE ? (T)0 : in[orig[s]];
}
// dst = in^2 (c -> c^2, cudaParticleSPH_NS.cu:63-64); padding slots get 0
__global__ void k_pack_square(const double *in, const uint32_t *orig, uint32_t n, double *dst) {
  const uint32_t s = blockIdx.x * blockDim.x + threadIdx.x;
  if (s < n) dst[s] = orig[s] == PB_NONE ? 0.0 : in[orig[s]] * in[orig[s]];
}
// 1/rho of imported densities (calcDensityPost's reciprocal,
// cudaParticleSPH_NS.cu:190-195), so that an acceleration after a density
// import uses the imported densities throughout
__global__ void k_pack_rhoinv(const double *in, const uint32_t *orig, uint32_t n, double *rhoinv) {
  const uint32_t s = blockIdx.x * blockDim.x + threadIdx.x;
  if (s < n) rhoinv[s] = orig[s] == PB_NONE ? 0.0 : 1.0 / in[3 * (size_t)orig[s] + 1];
}
__global__ void k_pack_type(const uint16_t *in, const uint32_t *orig, uint32_t n, uint16_t *type,
                            double4 *r) {
  const uint32_t s = blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= n || orig[s] == PB_NONE) return;
  const uint16_t t = in[orig[s]];
  type[s] = t;
  r[s].w = (double)t;
}

struct ImportArgs {
  const uint32_t *orig;
  const double *m;
  const uint32_t *ty;          // null: type 0
  const uint8_t *fixed;        // null: all movable
  uint32_t n;
  double4 *r, *v, *a, *F;
  uint16_t *type;
  uint8_t *move;
};
// type, mass, movable flag; padding rows and F cleared
__global__ void k_import_scalars(ImportArgs A) {
  const uint32_t s = blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= A.n) return;
  const uint32_t o = A.orig[s];
  const bool pad = o == PB_NONE;
  const uint32_t t = pad ? PB_PAD_TYPE : (A.ty ? A.ty[o] : 0u);
  A.r[s] = make_double4(0, 0, 0, (double)t);
  A.v[s] = make_double4(0, 0, 0, pad ? 0.0 : 1.0 / A.m[o]);
  A.a[s] = make_double4(0, 0, 0, 0);
  A.F[s] = make_double4(0, 0, 0, 0);
  A.type[s] = (uint16_t)t;
  A.move[s] = pad ? 0 : (A.fixed ? (A.fixed[o] ? 0 : 1) : 1);
}

// -------------------------------------------------------------------- host
#define IO_GRID(s) dim3(pb_blocks((s)->npad, 256)), dim3(256), 0, (s)->ctx->stream

// run `pack(dst)` -- a kernel launch that writes the caller's `bytes` to a
// device-visible buffer -- and bring them to `host`
template <typename F>
static int download_packed(pb_sys *s, void *host, size_t bytes, F &&pack) {
  pb_ctx *ctx = s->ctx;
  if (bytes <= IO_DIRECT) {
    pack((void *)ctx->io_dev);
    PB_LAUNCH_CHECK(ctx, "pb_sys_get");
    PB_HIP(ctx, hipStreamSynchronize(ctx->stream));
    std::memcpy(host, ctx->io_stage, bytes);
    return PB_OK;
  }
  if (int rc = pb_io_buffer(s)) return rc;
  pack((void *)s->io);
  PB_LAUNCH_CHECK(ctx, "pb_sys_get");
  return pb_io_download(ctx, host, s->io, bytes);
}

int pb_io_scatter(pb_sys *s, const double *host, double *dst, bool square) {
  if (int rc = pb_io_buffer(s)) return rc;
  if (int rc = pb_io_upload(s->ctx, s->io, host, 8 * (size_t)s->n)) return rc;
  const double *in = (const double *)s->io;
  if (square) hipLaunchKernelGGL(k_pack_square, IO_GRID(s), in, s->orig, s->npad, dst);
  else hipLaunchKernelGGL(k_pack1<double>, IO_GRID(s), in, s->orig, s->npad, dst);
  PB_LAUNCH_CHECK(s->ctx, "pb_io_scatter");
  return PB_OK;
}

extern "C" int pb_sys_import(pb_sys *s, const double *r, const double *v, const double *a,
                             const double *m, const uint32_t *type, const uint8_t *is_fixed) {
  if (!s || !r || !m) return pb_fail(s ? s->ctx : nullptr, PB_ERR_ARG, "pb_sys_import: r and m required");
  PB_HIP(s->ctx, hipSetDevice(s->ctx->device));
  const size_t n = s->n;
  // nothing is written before all values are known to be good
  for (size_t g = 0; g < n; ++g) {
    if (type && type[g] >= PB_MAXT) return pb_fail(s->ctx, PB_ERR_ARG, "pb_sys_import: type >= 5");
    if (!(m[g] > 0)) return pb_fail(s->ctx, PB_ERR_ARG, "pb_sys_import: mass must be > 0");
  }
  int rc;
  if ((rc = pb_io_buffer(s))) return rc;
  ImportArgs A;
  A.orig = s->orig;
  A.m = (const double *)s->io;
  A.ty = type ? (const uint32_t *)(s->io + 8 * n) : nullptr;
  A.fixed = is_fixed ? s->io + 12 * n : nullptr;
  A.n = s->npad;
  A.r = s->r; A.v = s->v; A.a = s->a; A.F = s->F;
  A.type = s->type; A.move = s->move;
  if ((rc = pb_io_upload(s->ctx, s->io, m, 8 * n)) ||
      (type && (rc = pb_io_upload(s->ctx, s->io + 8 * n, type, 4 * n))) ||
      (is_fixed && (rc = pb_io_upload(s->ctx, s->io + 12 * n, is_fixed, n))))
    return rc;
  hipLaunchKernelGGL(k_import_scalars, IO_GRID(s), A);
  PB_LAUNCH_CHECK(s->ctx, "k_import_scalars");
  const double *src[3] = {r, v, a};
  double4 *dst[3] = {s->r, s->v, s->a};
  for (int k = 0; k < 3; ++k) {
    if (!src[k]) continue;
    // the stream orders the upload behind the kernels that read the buffer
    if ((rc = pb_io_upload(s->ctx, s->io, src[k], 24 * n))) return rc;
    hipLaunchKernelGGL(k_pack3, IO_GRID(s), (const double *)s->io, s->orig, s->npad, dst[k]);
    PB_LAUNCH_CHECK(s->ctx, "k_pack3");
  }
  PB_HIP(s->ctx, hipStreamSynchronize(s->ctx->stream));
  s->ref_binned = false;
  return PB_OK;
}

static double4 *vec_field(pb_sys *s, int field) {
  switch (field) {
    case PB_FIELD_R: return s->r;
    case PB_FIELD_V: return s->v;
    case PB_FIELD_A: return s->a;
    case PB_FIELD_F: return s->F;
    case PB_FIELD_W: return s->w;
    case PB_FIELD_L: return s->w ? s->Lm : nullptr;
    case PB_FIELD_T: return s->w ? s->T : nullptr;
    case PB_FIELD_SPH_NUM: return s->sph_num;
    default: return nullptr;
  }
}

extern "C" int pb_sys_get(pb_sys *s, int field, void *host) {
  if (!s || !host) return PB_ERR_ARG;
  PB_HIP(s->ctx, hipSetDevice(s->ctx->device));
  const size_t n = s->n;
  if (const double4 *src = vec_field(s, field))
    return download_packed(s, host, 24 * n, [&](void *d) {
      hipLaunchKernelGGL(k_unpack3, IO_GRID(s), src, s->orig, s->npad, (double *)d);
    });
  auto scalar = [&](auto *src) {
    using T = std::remove_const_t<std::remove_pointer_t<decltype(src)>>;
    return download_packed(s, host, sizeof(T) * n, [&](void *d) {
      hipLaunchKernelGGL(k_unpack1<T>, IO_GRID(s), src, s->orig, s->npad, (T *)d);
    });
  };
  switch (field) {
    case PB_FIELD_W:
    case PB_FIELD_L:
    case PB_FIELD_T:
      return pb_fail(s->ctx, PB_ERR_STATE, "pb_sys_get: rotation state not allocated");
    case PB_FIELD_SPH_NUM:
      return pb_fail(s->ctx, PB_ERR_STATE, "pb_sys_get: no SPH density yet");
    case PB_FIELD_SPH_RHOINV:
      if (!s->sph_num) return pb_fail(s->ctx, PB_ERR_STATE, "pb_sys_get: no SPH density yet");
      return scalar(s->sph_rhoinv);
    case PB_FIELD_MINV:
      return download_packed(s, host, 8 * n, [&](void *d) {
        hipLaunchKernelGGL(k_unpack_w, IO_GRID(s), s->v, s->orig, s->npad, (double *)d);
      });
    case PB_FIELD_TYPE: return scalar(s->type);
    case PB_FIELD_MOVE: return scalar(s->move);
    case PB_FIELD_RADIUS:
      if (!s->radius) return pb_fail(s->ctx, PB_ERR_STATE, "pb_sys_get: radius not set");
      return scalar(s->radius);
    default: return pb_fail(s->ctx, PB_ERR_ARG, "pb_sys_get: unknown field");
  }
}

extern "C" int pb_sys_set(pb_sys *s, int field, const void *host) {
  if (!s || !host) return PB_ERR_ARG;
  PB_HIP(s->ctx, hipSetDevice(s->ctx->device));
  int rc = PB_OK;
  if ((field == PB_FIELD_W || field == PB_FIELD_L || field == PB_FIELD_T) && (rc = pb_ensure_rotation(s)))
    return rc;
  if (field == PB_FIELD_RADIUS && (rc = pb_ensure_radius(s))) return rc;
  if (field == PB_FIELD_SPH_NUM && !s->sph_num)
    return pb_fail(s->ctx, PB_ERR_STATE, "pb_sys_set: no SPH density yet");
  double4 *vec = vec_field(s, field);
  const size_t n = s->n;
  size_t bytes = 24 * n;
  if (!vec) {
    switch (field) {
      case PB_FIELD_MINV:
      case PB_FIELD_RADIUS: bytes = 8 * n; break;
      case PB_FIELD_TYPE:
        bytes = 2 * n;
        for (size_t g = 0; g < n; ++g)
          if (((const uint16_t *)host)[g] >= PB_MAXT)
            return pb_fail(s->ctx, PB_ERR_ARG, "pb_sys_set: type >= 5");
        break;
      case PB_FIELD_MOVE: bytes = n; break;
      default: return pb_fail(s->ctx, PB_ERR_ARG, "pb_sys_set: unknown field");
    }
  }
  if ((rc = pb_io_buffer(s)) || (rc = pb_io_upload(s->ctx, s->io, host, bytes))) return rc;
  if (vec) {
    hipLaunchKernelGGL(k_pack3, IO_GRID(s), (const double *)s->io, s->orig, s->npad, vec);
    if (field == PB_FIELD_SPH_NUM && s->sph_rhoinv)
      hipLaunchKernelGGL(k_pack_rhoinv, IO_GRID(s), (const double *)s->io, s->orig, s->npad,
                         s->sph_rhoinv);
  } else if (field == PB_FIELD_MINV) {
    hipLaunchKernelGGL(k_pack_w, IO_GRID(s), (const double *)s->io, s->orig, s->npad, s->v);
  } else if (field == PB_FIELD_TYPE) {
    hipLaunchKernelGGL(k_pack_type, IO_GRID(s), (const uint16_t *)s->io, s->orig, s->npad, s->type,
                       s->r);
  } else if (field == PB_FIELD_MOVE) {
    hipLaunchKernelGGL(k_pack1<uint8_t>, IO_GRID(s), s->io, s->orig, s->npad, s->move);
  } else {
    hipLaunchKernelGGL(k_pack1<double>, IO_GRID(s), (const double *)s->io, s->orig, s->npad,
                       s->radius);
  }
  PB_LAUNCH_CHECK(s->ctx, "pb_sys_set");
  PB_HIP(s->ctx, hipStreamSynchronize(s->ctx->stream));
  return PB_OK;
}
