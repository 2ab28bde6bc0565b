// Copies between device planes and reference-layout host arrays.
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>

namespace gcs {

struct Problem;

// One plane of one cube face <-> a strided host array of extent ext
// (element e at host[e * stride]).
int plane_to_host(Problem &P, int plane, int face, const size_t ext[3],
                  double *host, size_t stride);
int host_to_plane(Problem &P, int plane, int face, const size_t ext[3],
                  const double *host, size_t stride);
int host_to_byte_plane(Problem &P, int plane, int face, const size_t ext[3],
                       const unsigned char *host);
// ncomp consecutive planes <-> an interleaved host array [element][ncomp].
int planes_to_host(Problem &P, int first, int ncomp, int face,
                   const size_t ext[3], double *host);
int host_to_planes(Problem &P, int first, int ncomp, int face,
                   const size_t ext[3], const double *host);
// planes_to_host for the elements of the box lo <= (i, j, k) < hi only; the
// host array's other elements are left as they are.
int box_planes_to_host(Problem &P, int first, int ncomp, int face, const size_t ext[3],
                       const size_t lo[3], const size_t hi[3], double *host);

// Host arrays of `faces` cube faces from `face` on, interleaved [element]
// [ncomp] with extent ext, from ncomp consecutive planes; allocates them.
struct HostArray;
int planes_to_arrays(Problem &P, int first, int ncomp, int face, int faces,
                     const size_t ext[3], HostArray *const out[]);
void free_array(HostArray &a);

// Two pinned chunks that flat arrays cross PCIe in, owned by one caller (its
// calls are in order on one stream). Without buffers (never made, or no pinned
// memory) and for short arrays the copies are direct.
struct Staging {
  char *buf[2] = {};
  hipEvent_t done[2] = {};
  Staging() = default;
  Staging(const Staging &) = delete;
  Staging &operator=(const Staging &) = delete;
  ~Staging();
  void make();
};
// The host array has been read when stage_up returns, and been written when
// stage_down does (which also waits for the stream's earlier work).
int stage_up(Staging &g, hipStream_t stream, const void *host, void *dev, size_t bytes);
int stage_down(Staging &g, hipStream_t stream, const void *dev, void *host, size_t bytes);

}  // namespace gcs
