// ljg_transfer.hip -- particle arrays between the caller's memory and the device, through one pinned staging
// buffer per context (at most kRingBytes).
//
// The copies of pageable memory that the runtime makes cost 10-40 us each whatever their size, and a download was
// one long copy followed by one long memcpy of the same bytes.  Here small uploads are copied into the staging
// buffer, which the kernels read directly, and downloads run as a ring of chunks: the device writes a chunk
// into the buffer while the host copies earlier ones out, from a few threads when there is much to copy.
#include <algorithm>
#include <chrono>
#include <cstring>

#include "ljg_internal.h"
#include "ljg_stage.h"

namespace ljg {

constexpr int kMoveThreads = 256;

// Pinned memory is read and written at system scope: kernels that follow each other in a stream meet at the
// scope of the device, so a plain load may find a line that an L2 kept from an earlier upload, and a plain store
// may stay there.
template <bool HOST, class T>
__device__ inline T load_from(const T *p) {
  if constexpr (HOST) return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
  else return *p;
}

// n 8-byte words from device to pinned memory (OUT) or back.  With progress given, `value` goes there first: the
// kernels queued before this one have finished.
template <bool OUT>
__global__ __launch_bounds__(kMoveThreads) void k_move(int64_t n, const unsigned long long *__restrict__ src,
                                                       unsigned long long *__restrict__ dst,
                                                       unsigned long long *progress, unsigned long long value) {
  if (progress && blockIdx.x == 0 && threadIdx.x == 0) {
    __threadfence_system();
    __hip_atomic_store(progress, value, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
  }
  const int64_t step = (int64_t)gridDim.x * kMoveThreads;
#pragma unroll 4
  for (int64_t i = (int64_t)blockIdx.x * kMoveThreads + threadIdx.x; i < n; i += step) {
    const unsigned long long v = load_from<!OUT>(src + i);
    if constexpr (OUT) __hip_atomic_store(dst + i, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    else dst[i] = v;
  }
}

template <bool OUT>
static void move_launch(Ctx &c, const double *src, double *dst, size_t n, unsigned long long *progress,
                        unsigned long long value) {
  const int nb = n > 0 ? blocks_for((int64_t)n, kMoveThreads * 4) : 1;
  hipLaunchKernelGGL(k_move<OUT>, dim3(nb < 512 ? nb : 512), dim3(kMoveThreads), 0, c.stream, (int64_t)n,
                     reinterpret_cast<const unsigned long long *>(src), reinterpret_cast<unsigned long long *>(dst),
                     progress, value);
  LJG_HIP(hipGetLastError());
}

// The staging buffer of at least `bytes` (up to kRingBytes), free of earlier uploads that kernels may still read.
static double *stage_buffer(Ctx &c, size_t bytes) {
  if (c.stage_mark > c.mark_seen) {
    stream_wait(c);  // (a marker seen after the upload was queued also shows that it was read)
  }
  c.stage_mark = 0;
  if (c.pin_stage_cap < bytes) {
    const size_t cap = stage_capacity(bytes, c.pin_stage_cap);
    if (c.pin_stage) LJG_HIP(hipHostFree(c.pin_stage));
    c.pin_stage = nullptr;
    c.pin_stage_cap = 0;
    LJG_HIP(hipHostMalloc((void **)&c.pin_stage, cap, hipHostMallocMapped | hipHostMallocCoherent));
    c.pin_stage_cap = cap;
    LJG_HIP(hipHostGetDevicePointer((void **)&c.pin_stage_dev, c.pin_stage, 0));
  }
  return c.pin_stage;
}

void release_stage(Ctx &c) {
  c.helpers.join();
  if (c.pin_stage) (void)hipHostFree(c.pin_stage);
  c.pin_stage = nullptr;
}

// dst (may be null) = src; whether every value lies in [lo, hi] (NaN does not).  Without an early exit, so that the
// loop is vectorised: the check took 0.7 ns per value on its own.
static bool copy_checked(double *__restrict__ dst, const double *__restrict__ src, size_t n, double lo, double hi) {
  bool ok = true;
  constexpr size_t kBlock = 1024;
  for (size_t b = 0; b < n; b += kBlock) {
    const size_t e = b + kBlock < n ? b + kBlock : n;
    if (dst) std::memcpy(dst + b, src + b, (e - b) * sizeof(double));
    int64_t inside = 0;
    for (size_t i = b; i < e; ++i) inside += (int64_t)((src[i] >= lo) & (src[i] <= hi));
    ok = ok && inside == (int64_t)(e - b);
  }
  return ok;
}

bool region_check(const Ctx &c, int64_t n, const double *const src[3], double *const dst[3]) {
  const double ilen = c.prm.cutoff + c.prm.skin;
  for (int d = 0; d < 3; ++d) {
    if (!c.open) {
      if (dst[d]) std::memcpy(dst[d], src[d], (size_t)n * sizeof(double));
    } else if (!copy_checked(dst[d], src[d], (size_t)n, c.open_min[d] - ilen, c.open_max[d] + ilen)) {
      return false;
    }
  }
  return true;
}

// An upload in storage order: x, y, z, velocities, types and ids (vx, type, id null: zero, zero, the index) from the
// arrays given, which may be pinned memory or the state's own; forces zero, reference positions as given, positions wrapped into
// the box (not those of an ensemble, whose boxes wrap them).
template <bool HOST>
__global__ __launch_bounds__(256) void k_init_upload(int64_t n, StateView s, const double *x,
                                                     const double *y, const double *z,
                                                     const double *vx, const double *vy,
                                                     const double *vz, const int32_t *type,
                                                     const int64_t *id, int32_t wrap, WrapArgs w) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const double px = load_from<HOST>(x + i), py = load_from<HOST>(y + i), pz = load_from<HOST>(z + i);
  const double ux = vx ? load_from<HOST>(vx + i) : 0., uy = vx ? load_from<HOST>(vy + i) : 0.;
  const double uz = vx ? load_from<HOST>(vz + i) : 0.;
  const int32_t t = type ? load_from<HOST>(type + i) : 0;
  const int64_t k = id ? load_from<HOST>(id + i) : i;
  s.rx[i] = px; s.ry[i] = py; s.rz[i] = pz;
  s.x[i] = wrap ? wrap_coord(px, 0, w) : px;
  s.y[i] = wrap ? wrap_coord(py, 1, w) : py;
  s.z[i] = wrap ? wrap_coord(pz, 2, w) : pz;
  s.vx[i] = ux; s.vy[i] = uy; s.vz[i] = uz;
  s.fx[i] = 0.; s.fy[i] = 0.; s.fz[i] = 0.;
  s.ofx[i] = 0.; s.ofy[i] = 0.; s.ofz[i] = 0.;
  s.type[i] = t;
  s.orig[i] = (int32_t)i;
  s.id[i] = k;
}

// Uploads of up to kStageUpload go through the staging buffer, where it is large enough already (a download
// makes it as large as it needs) or no more than kStageNew would be pinned: pinning takes ~0.4 ms per MiB, more
// than one upload gains.  Larger ones are copied by the runtime, whose cost per call no longer counts.
constexpr size_t kStageUpload = 4u << 20, kStageNew = 256u << 10;
static bool use_stage(const Ctx &c, size_t bytes) {
  return bytes <= kStageUpload && (bytes <= c.pin_stage_cap || bytes <= kStageNew);
}

bool upload_state(Ctx &c, int64_t n, const double *const pos[3], const double *const vel[3], const int32_t *type,
                  const int64_t *id) {
  const bool hv = vel[0] && vel[1] && vel[2];
  const size_t un = (size_t)n, stride = un + (un & 1);
  const size_t words = (hv ? 6 : 3) * stride + (id ? stride : 0) + (type ? (stride + 1) / 2 : 0);
  State &s = c.st[0];
  const WrapArgs w = wrap_args(c.prm);
  const int32_t wrap = c.nboxes == 0;
  const double *p[3] = {s.x.p, s.y.p, s.z.p}, *v[3] = {nullptr, nullptr, nullptr};
  const int32_t *dt = nullptr;
  const int64_t *di = nullptr;
  const bool staged = use_stage(c, words * sizeof(double));
  if (staged) {
    double *h = stage_buffer(c, words * sizeof(double));
    const double *dev = c.pin_stage_dev;
    size_t off = 0;
    double *const dst[3] = {h, h + stride, h + 2 * stride};
    if (!region_check(c, n, pos, dst)) return false;
    for (int d = 0; d < 3; ++d, off += stride) p[d] = dev + off;
    if (hv)
      for (int d = 0; d < 3; ++d, off += stride) {
        std::memcpy(h + off, vel[d], un * sizeof(double));
        v[d] = dev + off;
      }
    if (id) {
      std::memcpy(h + off, id, un * sizeof(int64_t));
      di = reinterpret_cast<const int64_t *>(dev + off);
      off += stride;
    }
    if (type) {
      std::memcpy(h + off, type, un * sizeof(int32_t));
      dt = reinterpret_cast<const int32_t *>(dev + off);
    }
  } else {
    double *const none[3] = {nullptr, nullptr, nullptr};
    if (c.open && !region_check(c, n, pos, none)) return false;
  }
  c.cur = 0;
  s.ensure(un);
  if (!staged) {
    double *const px[3] = {s.x.p, s.y.p, s.z.p}, *const pv[3] = {s.vx.p, s.vy.p, s.vz.p};
    for (int d = 0; d < 3; ++d) {
      LJG_HIP(hipMemcpyAsync(px[d], pos[d], un * sizeof(double), hipMemcpyHostToDevice, c.stream));
      p[d] = px[d];
    }
    if (hv)
      for (int d = 0; d < 3; ++d) {
        LJG_HIP(hipMemcpyAsync(pv[d], vel[d], un * sizeof(double), hipMemcpyHostToDevice, c.stream));
        v[d] = pv[d];
      }
    if (type) {
      LJG_HIP(hipMemcpyAsync(s.type.p, type, un * sizeof(int32_t), hipMemcpyHostToDevice, c.stream));
      dt = s.type.p;
    }
    if (id) {
      LJG_HIP(hipMemcpyAsync(s.id.p, id, un * sizeof(int64_t), hipMemcpyHostToDevice, c.stream));
      di = s.id.p;
    }
  }
  hipLaunchKernelGGL(staged ? k_init_upload<true> : k_init_upload<false>, dim3(blocks_for(n, 256)), dim3(256), 0,
                     c.stream, n, view(s), p[0], p[1], p[2], v[0], v[1], v[2], dt, di, wrap, w);
  LJG_HIP(hipGetLastError());
  // The caller's arrays are free to change once this returns.  The staging buffer is used again only after a
  // marker queued behind this launch was seen.
  if (staged) c.stage_mark = c.mark_seq + 1;
  else stream_wait(c);
  return true;
}

const double *stage_positions(Ctx &c, const double *const pos[3], const double *const vel[3], double *dev) {
  const size_t n = (size_t)c.n;
  const bool hv = vel[0] && vel[1] && vel[2];
  const size_t words = (hv ? 6 : 3) * n;
  if (!use_stage(c, words * sizeof(double))) {
    double *const none[3] = {nullptr, nullptr, nullptr};
    if (c.open && !region_check(c, c.n, pos, none)) return nullptr;
    for (int k = 0; k < (hv ? 6 : 3); ++k)
      LJG_HIP(hipMemcpyAsync(dev + k * n, k < 3 ? pos[k] : vel[k - 3], n * sizeof(double), hipMemcpyHostToDevice,
                             c.stream));
    return dev;
  }
  double *h = stage_buffer(c, words * sizeof(double));
  double *const dst[3] = {h, h + n, h + 2 * n};
  if (!region_check(c, c.n, pos, dst)) return nullptr;
  if (hv)
    for (int d = 0; d < 3; ++d) std::memcpy(h + (3 + d) * n, vel[d], n * sizeof(double));
  move_launch<false>(c, c.pin_stage_dev, dev, words, nullptr, 0);
  c.stage_mark = c.mark_seq + 1;
  return dev;
}

// From 24 MiB on with three helpers: one thread copies about 30 GB/s, the link carries 55.  Downloads of 63, 72 and
// 144 MB: 3.50, 3.74 and 7.36 -> 1.42, 1.55 and 2.95 ms.
constexpr size_t kHelpedBytes = 24u << 20;
constexpr int kHelpers = 3;

void download_arrays(Ctx &c, const double *dev, size_t count, double *const outs[9]) {
  const std::shared_ptr<Download> shared = std::make_shared<Download>();
  Download &d = *shared;
  d.count = count;
  d.total = 9 * count;
  d.chunk = download_chunk(d.total);
  d.nchunks = (int)((d.total + d.chunk - 1) / d.chunk);
  const size_t bytes = (d.nchunks > 1 ? (size_t)d.nchunks * d.chunk : d.total) * sizeof(double);
  d.ring = stage_buffer(c, bytes < kRingBytes ? bytes : kRingBytes);
  d.slots = (int)(c.pin_stage_cap / (d.chunk * sizeof(double)));
  d.slots = d.slots < 1 ? 1 : d.slots;  // (a single chunk shorter than kMinChunk)
  std::copy(outs, outs + 9, d.outs);
  d.progress = c.pin_mark + kMarkProgress;
  d.base = c.progress_seq;
  c.progress_seq += (unsigned long long)d.nchunks + 1;
  d.done.reset(new std::atomic<char>[(size_t)d.nchunks]);
  for (int k = 0; k < d.nchunks; ++k) d.done[k].store(0, std::memory_order_relaxed);
  int queued = 0;  // chunks queued, nchunks + 1 once the last progress write is
  int mine = -1;   // the chunk this thread has taken last
  auto pump = [&]() {
    while (queued <= d.nchunks &&
           (queued == d.nchunks || queued < d.slots || d.done[queued - d.slots].load(std::memory_order_acquire))) {
      const size_t b = (size_t)queued * d.chunk, n = queued == d.nchunks ? 0 : std::min(d.chunk, d.total - b);
      move_launch<true>(c, dev + (n ? b : 0), c.pin_stage_dev + (n ? (size_t)(queued % d.slots) * d.chunk : 0), n,
                  queued > 0 ? c.pin_mark_dev + kMarkProgress : nullptr, d.base + (unsigned long long)queued);
      ++queued;
    }
  };
  try {
    pump();
    if (d.total * sizeof(double) >= kHelpedBytes) {
      for (int k = 0; k < kHelpers; ++k) {
        try {
          c.helpers.start([shared]() { shared->help(); });
        } catch (const std::exception &) {
          break;  // no more threads to be had: this one copies the rest
        }
      }
    }
    auto t0 = std::chrono::steady_clock::now();
    // (device: only the device is waited for, which a synchronisation of the stream completes)
    auto wait_for = [&](bool device, auto &&met) {
      for (uint64_t spins = 0; !met(); ++spins) {
        pump();
        if ((spins & 1023) == 1023 && std::chrono::steady_clock::now() - t0 > std::chrono::seconds(2)) {
          LJG_HIP(hipStreamSynchronize(c.stream));  // reports any error
          if (device && queued > d.nchunks && !met()) throw HipError{hipErrorUnknown, "download not completed", __LINE__};
          t0 = std::chrono::steady_clock::now();
        }
      }
    };
    for (;;) {
      const int k = d.next.fetch_add(1);
      if (k >= d.nchunks) break;
      mine = k;
      wait_for(true, [&]() { return d.ready(k); });
      d.copy_out(k);
    }
    // every chunk is taken: the helpers finish theirs (which may wait for some that are not queued yet)
    for (int k = 0; k < d.nchunks; ++k)
      wait_for(false, [&]() { return d.done[k].load(std::memory_order_acquire) != 0; });
    wait_for(false, [&]() { return queued > d.nchunks; });
  } catch (...) {
    // no chunk is taken from here on; those taken end with the abort or with their copy
    const int taken = std::min(d.next.exchange(d.nchunks), d.nchunks);
    d.abort.store(true);
    for (int k = 0; k < taken; ++k)
      while (d.done[k].load(std::memory_order_acquire) == 0 && k != mine) std::this_thread::yield();
    throw;
  }
}

}  // namespace ljg
