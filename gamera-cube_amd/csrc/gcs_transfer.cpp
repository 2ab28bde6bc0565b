// Copies between device planes and the reference's array-of-structs host
// arrays (gamera_no_grid / gamera_no_storage / gamera_no_background_field,
// nonorthogonal_grid.h:12-30, nonorthogonal_storage.h:12-47): element e of an
// array with extent ext is at host[e * stride], k fastest
// (nonorthogonal_grid.c:7-10), and maps to plane position (i * SJ + j) * SK + k
// of its cube face.
//
// The planes of one array cross PCIe together through a pinned staging
// buffer (one strided copy for all its components), and the conversion to
// or from the interleaved host layout runs on a pool of host threads, each
// taking whole radial planes, so that every host element's components are
// written together.
#include <hip/hip_runtime.h>
#include <sys/mman.h>

#include <algorithm>
#include <cstdlib>
#include <cstring>
#include <vector>

#include "gcs_device.hpp"
#include "gcs_host_pool.hpp"
#include "gcs_transfer.hpp"

namespace gcs {

namespace {

// The problem's pinned staging buffer, at least `count` doubles.
double *pinned(Problem &P, size_t count) {
  if (P.pinned_count < count) {
    if (P.pinned != nullptr) (void)hipHostFree(P.pinned);
    P.pinned = nullptr;
    P.pinned_count = 0;
    if (hipHostMalloc((void **)&P.pinned, count * sizeof(double)) != hipSuccess) {
      P.pinned = nullptr;
      set_error("pinned host allocation failed");
      return nullptr;
    }
    P.pinned_count = count;
  }
  return P.pinned;
}

// ncomp consecutive planes of one cube face <-> the pinned buffer
// [ncomp][face_stride].
int planes_down(Problem &P, int first, int ncomp, int face, double *buf) {
  const Layout &L = P.L;
  GCS_HIP(hipMemcpy2D(buf, L.face_stride * sizeof(double),
                      P.plane(first) + face * L.face_stride, L.total * sizeof(double),
                      L.face_stride * sizeof(double), ncomp, hipMemcpyDeviceToHost));
  return 0;
}

int planes_up(Problem &P, int first, int ncomp, int face, const double *buf) {
  const Layout &L = P.L;
  GCS_HIP(hipMemcpy2D(P.plane(first) + face * L.face_stride, L.total * sizeof(double), buf,
                      L.face_stride * sizeof(double), L.face_stride * sizeof(double), ncomp,
                      hipMemcpyHostToDevice));
  return 0;
}

// Component c of element e at host[e * stride + c].
int to_host(Problem &P, int first, int ncomp, int face, const size_t ext[3], double *host,
            size_t stride) {
  const Layout &L = P.L;
  double *buf = pinned(P, (size_t)ncomp * L.face_stride);
  if (buf == nullptr || planes_down(P, first, ncomp, face, buf) != 0) return -1;
  HostPool::get().run((long)ext[0], [&](long i0, long i1) {
    for (size_t i = (size_t)i0; i < (size_t)i1; ++i)
      for (size_t j = 0; j < ext[1]; ++j) {
        const size_t at = (i * L.SJ + j) * L.SK;
        double *h = host + ((i * ext[1] + j) * ext[2]) * stride;
        for (size_t k = 0; k < ext[2]; ++k, h += stride)
          for (int c = 0; c < ncomp; ++c) h[c] = buf[c * L.face_stride + at + k];
      }
  });
  return 0;
}

int from_host(Problem &P, int first, int ncomp, int face, const size_t ext[3],
              const double *host, size_t stride) {
  const Layout &L = P.L;
  double *buf = pinned(P, (size_t)ncomp * L.face_stride);
  if (buf == nullptr) return -1;
  // Positions outside the array's extent are zero, as after allocation.
  HostPool::get().run((long)(L.NI + 1), [&](long i0, long i1) {
    for (int c = 0; c < ncomp; ++c)
      std::memset(buf + c * L.face_stride + (size_t)i0 * L.SJ * L.SK, 0,
                  (size_t)(i1 - i0) * L.SJ * L.SK * sizeof(double));
    for (size_t i = (size_t)i0; i < std::min((size_t)i1, ext[0]); ++i)
      for (size_t j = 0; j < ext[1]; ++j) {
        const size_t at = (i * L.SJ + j) * L.SK;
        const double *h = host + ((i * ext[1] + j) * ext[2]) * stride;
        for (size_t k = 0; k < ext[2]; ++k, h += stride)
          for (int c = 0; c < ncomp; ++c) buf[c * L.face_stride + at + k] = h[c];
      }
  });
  return planes_up(P, first, ncomp, face, buf);
}

}  // namespace

int plane_to_host(Problem &P, int plane, int face, const size_t ext[3],
                  double *host, size_t stride) {
  return to_host(P, plane, 1, face, ext, host, stride);
}

int box_planes_to_host(Problem &P, int first, int ncomp, int face, const size_t ext[3],
                       const size_t lo[3], const size_t hi[3], double *host) {
  const Layout &L = P.L;
  double *buf = pinned(P, (size_t)ncomp * L.face_stride);
  if (buf == nullptr || planes_down(P, first, ncomp, face, buf) != 0) return -1;
  HostPool::get().run((long)(hi[0] - lo[0]), [&](long i0, long i1) {
    for (size_t i = lo[0] + (size_t)i0; i < lo[0] + (size_t)i1; ++i)
      for (size_t j = lo[1]; j < hi[1]; ++j) {
        const size_t at = (i * L.SJ + j) * L.SK;
        for (size_t k = lo[2]; k < hi[2]; ++k)
          for (int c = 0; c < ncomp; ++c)
            host[((i * ext[1] + j) * ext[2] + k) * ncomp + c] = buf[c * L.face_stride + at + k];
      }
  });
  return 0;
}

void free_array(HostArray &a) {
  std::free(a.data);
  a = HostArray();
}

namespace {

// Memory for `count` doubles; large arrays on huge pages where the system
// has them (a 4 KiB page fault each costs more than the copy into it).
int size_array(HostArray &a, size_t count) {
  a.count = count;
  if (a.capacity >= count) return 0;
  std::free(a.data);
  a.capacity = 0;
  constexpr size_t huge = 2UL << 20;
  size_t bytes = std::max<size_t>(count, 1) * sizeof(double);
  if (bytes >= 2 * huge) {
    bytes = (bytes + huge - 1) / huge * huge;
    a.data = (double *)std::aligned_alloc(huge, bytes);
    if (a.data != nullptr) (void)madvise(a.data, bytes, MADV_HUGEPAGE);
  } else {
    a.data = (double *)std::malloc(bytes);
  }
  if (a.data == nullptr) {
    a = HostArray();
    set_error("host allocation failed");
    return -1;
  }
  a.capacity = count;
  return 0;
}

// memcpy on the host threads; small copies on the calling one.
void parallel_copy(void *dst, const void *src, size_t bytes, size_t block = 1UL << 18) {
  if (bytes <= 4 * block) {
    std::memcpy(dst, src, bytes);
    return;
  }
  HostPool::get().run((long)((bytes + block - 1) / block), [&](long b0, long b1) {
    const size_t from = (size_t)b0 * block, to = std::min(bytes, (size_t)b1 * block);
    std::memcpy((char *)dst + from, (const char *)src + from, to - from);
  });
}

}  // namespace

namespace {

// One plane at a time through a pageable copy: slow, and needs no device or
// pinned memory.
int planes_to_arrays_direct(Problem &P, int first, int ncomp, int face, int faces,
                            const size_t ext[3], HostArray *const out[]) {
  const Layout &L = P.L;
  std::vector<double> buf(L.face_stride);
  for (int f = 0; f < faces; ++f) {
    for (int c = 0; c < ncomp; ++c) {
      GCS_HIP(hipMemcpy(buf.data(), P.plane(first + c) + (face + f) * L.face_stride,
                        L.face_stride * sizeof(double), hipMemcpyDeviceToHost));
      double *to = out[f]->data + c;
      for (size_t i = 0; i < ext[0]; ++i)
        for (size_t j = 0; j < ext[1]; ++j)
          for (size_t k = 0; k < ext[2]; ++k, to += ncomp) *to = buf[(i * L.SJ + j) * L.SK + k];
    }
    out[f]->valid = true;
  }
  return 0;
}

}  // namespace

// The planes are interleaved on the device and cross PCIe in two alternating
// pinned chunks, each copied out by the host threads while the next one
// arrives. What bounds it is PCIe and the host's memory (6 x 96^2 x 192, U, B
// and face flux, 1.25 GB: 30 ms, 42 GB/s; a pageable copy per plane and one
// host thread that scattered it took 228 ms). A device with no room for the
// interleaved array, or a host without pinned memory, takes the direct way.
int planes_to_arrays(Problem &P, int first, int ncomp, int face, int faces,
                     const size_t ext[3], HostArray *const out[]) {
  const size_t per = ext[0] * ext[1] * ext[2] * (size_t)ncomp, total = per * faces;
  for (int f = 0; f < faces; ++f)
    if (size_array(*out[f], per) != 0) return -1;
  const size_t chunk = std::min<size_t>(total, 1UL << 20);  // doubles
  double *buf = pinned(P, 2 * chunk);
  bool staged = buf != nullptr;
  for (hipEvent_t &e : P.copied)
    if (staged && e == nullptr)
      staged = hipEventCreateWithFlags(&e, hipEventDisableTiming) == hipSuccess;
  if (!staged || pack_planes(P, first, ncomp, face, faces, ext) != 0) {
    (void)hipGetLastError();
    return planes_to_arrays_direct(P, first, ncomp, face, faces, ext, out);
  }
  const size_t chunks = (total + chunk - 1) / chunk;
  auto request = [&](size_t q) -> int {
    const size_t at = q * chunk, n = std::min(chunk, total - at);
    GCS_HIP(hipMemcpyAsync(buf + (q & 1) * chunk, P.packed + at, n * sizeof(double),
                           hipMemcpyDeviceToHost, P.stream));
    GCS_HIP(hipEventRecord(P.copied[q & 1], P.stream));
    return 0;
  };
  for (size_t q = 0; q < std::min<size_t>(chunks, 2); ++q)
    if (request(q) != 0) return -1;
  for (size_t q = 0; q < chunks; ++q) {
    GCS_HIP(hipEventSynchronize(P.copied[q & 1]));
    const size_t end = std::min(total, (q + 1) * chunk);
    for (size_t at = q * chunk; at < end;) {  // a chunk may end one face and begin another
      const size_t f = at / per, in = at - f * per, n = std::min(per - in, end - at);
      parallel_copy(out[f]->data + in, buf + (q & 1) * chunk + (at - q * chunk),
                    n * sizeof(double));
      at += n;
    }
    if (q + 2 < chunks && request(q + 2) != 0) return -1;
  }
  for (int f = 0; f < faces; ++f) out[f]->valid = true;
  return 0;
}

// Flat arrays cross in two pinned chunks of 4 MB, filled or emptied by the host
// threads (blocks of 256 KB) while the other one is on the bus; a fresh numpy
// array is then also paged in by all of them. Down from 1 MB on (the network's
// 7.8 MB of gradients: loss and gradients of 8 x 32 x 64, 1.10 -> 0.90 ms); up
// only from 16 MB on (33.5 MB of features, 8 x 128 x 256: 3.43 -> 2.92 ms with
// both), where it gains: 8.4 MB took 0.30 ms either way.
namespace {
constexpr size_t kStageChunk = 4UL << 20, kStageBlock = 1UL << 18;
constexpr size_t kStageDownFrom = 1UL << 20, kStageUpFrom = 16UL << 20;
}

void Staging::make() {
  for (int b = 0; b < 2; ++b)
    if (hipHostMalloc((void **)&buf[b], kStageChunk) != hipSuccess)
      buf[b] = nullptr;
    else
      std::memset(buf[b], 0, kStageChunk);  // paged in here, not by the first copy
  for (int b = 0; b < 2; ++b)
    if (hipEventCreateWithFlags(&done[b], hipEventDisableTiming) != hipSuccess) done[b] = nullptr;
  (void)hipGetLastError();
}

Staging::~Staging() {
  for (int b = 0; b < 2; ++b) {
    if (done[b] != nullptr) (void)hipEventDestroy(done[b]);
    if (buf[b] != nullptr) (void)hipHostFree(buf[b]);
  }
}

static bool goes_staged(const Staging &g, size_t bytes, size_t from) {
  return bytes >= from && g.buf[0] != nullptr && g.buf[1] != nullptr &&
         g.done[0] != nullptr && g.done[1] != nullptr;
}

int stage_up(Staging &g, hipStream_t stream, const void *host, void *dev, size_t bytes) {
  if (!goes_staged(g, bytes, kStageUpFrom)) {
    GCS_HIP(hipMemcpyAsync(dev, host, bytes, hipMemcpyHostToDevice, stream));
    return 0;
  }
  for (size_t at = 0, q = 0; at < bytes; at += kStageChunk, ++q) {
    const size_t n = std::min(kStageChunk, bytes - at);
    GCS_HIP(hipEventSynchronize(g.done[q & 1]));  // the chunk's last copy, here or before
    parallel_copy(g.buf[q & 1], (const char *)host + at, n, kStageBlock);
    GCS_HIP(hipMemcpyAsync((char *)dev + at, g.buf[q & 1], n, hipMemcpyHostToDevice, stream));
    GCS_HIP(hipEventRecord(g.done[q & 1], stream));
  }
  return 0;
}

int stage_down(Staging &g, hipStream_t stream, const void *dev, void *host, size_t bytes) {
  if (!goes_staged(g, bytes, kStageDownFrom)) {
    GCS_HIP(hipMemcpyAsync(host, dev, bytes, hipMemcpyDeviceToHost, stream));
    GCS_HIP(hipStreamSynchronize(stream));
    return 0;
  }
  const size_t chunks = (bytes + kStageChunk - 1) / kStageChunk;
  auto request = [&](size_t q) -> int {
    const size_t at = q * kStageChunk, n = std::min(kStageChunk, bytes - at);
    GCS_HIP(hipMemcpyAsync(g.buf[q & 1], (const char *)dev + at, n, hipMemcpyDeviceToHost,
                           stream));
    GCS_HIP(hipEventRecord(g.done[q & 1], stream));
    return 0;
  };
  for (size_t q = 0; q < std::min<size_t>(chunks, 2); ++q)
    if (request(q) != 0) return -1;
  for (size_t q = 0; q < chunks; ++q) {
    const size_t at = q * kStageChunk;
    GCS_HIP(hipEventSynchronize(g.done[q & 1]));
    parallel_copy((char *)host + at, g.buf[q & 1], std::min(kStageChunk, bytes - at), kStageBlock);
    if (q + 2 < chunks && request(q + 2) != 0) return -1;
  }
  return 0;
}

int host_to_plane(Problem &P, int plane, int face, const size_t ext[3],
                  const double *host, size_t stride) {
  return from_host(P, plane, 1, face, ext, host, stride);
}

int host_to_byte_plane(Problem &P, int plane, int face, const size_t ext[3],
                       const unsigned char *host) {
  const Layout &L = P.L;
  std::vector<uint8_t> buf(L.face_stride, 0);
  size_t e = 0;
  for (size_t i = 0; i < ext[0]; ++i)
    for (size_t j = 0; j < ext[1]; ++j)
      for (size_t k = 0; k < ext[2]; ++k, ++e)
        buf[(i * L.SJ + j) * L.SK + k] = host[e] ? 1 : 0;
  GCS_HIP(hipMemcpy(P.byte_plane(plane) + face * L.face_stride, buf.data(),
                    L.face_stride, hipMemcpyHostToDevice));
  return 0;
}

int planes_to_host(Problem &P, int first, int ncomp, int face,
                   const size_t ext[3], double *host) {
  return to_host(P, first, ncomp, face, ext, host, (size_t)ncomp);
}

int host_to_planes(Problem &P, int first, int ncomp, int face,
                   const size_t ext[3], const double *host) {
  return from_host(P, first, ncomp, face, ext, host, (size_t)ncomp);
}

}  // namespace gcs
