// stage.hip -- what the caller hands in and takes out (positions, velocities,
// forces, potentials, energies, error flags), through a pinned host buffer of
// the engine that small kernels read and write directly over the host link.
//
// Per-site vectors live on the device as three planes (all x, all y, all z)
// and at the caller's as xyz triples; the kernels turn one into the other on
// the way.  Copying to pageable memory and reordering on the host cost two
// fresh buffers' page faults, a strided pass over both and the runtime's own
// staging: at 98304 sites 235 us for each of r, v and f taken out and 157 us
// for positions handed in; a flag word took 20 us.
// The link carries 55 GB/s (43 us for 98304 sites); the rest is the one
// memcpy to or from the caller's memory.
#include <sys/mman.h>

#include <cerrno>
#include <cstring>

#include "engine.hpp"

namespace mmamd {

constexpr int STAGE_TB = 256;
constexpr int STAGE_MAX_SITES = 1 << 18;   // 6 MiB of pinned memory at most
constexpr int STAGE_PUT_SITES = 1 << 14;   // handed in by parts: copied while the last part is read

__global__ void k_stage_sites(const double *__restrict__ soa, int N, int i0, int n,
                              double *__restrict__ aos) {
  const int k = blockIdx.x * STAGE_TB + threadIdx.x;
  if (k >= 3 * n) return;
  const int i = k / 3, c = k - 3 * i;
  aos[k] = soa[(long)c * N + i0 + i];
}

__global__ void k_unstage_sites(const double *__restrict__ aos, int N, int i0, int n,
                                double *__restrict__ soa) {
  const int k = blockIdx.x * STAGE_TB + threadIdx.x;
  if (k >= 3 * n) return;
  const int i = k / 3, c = k - 3 * i;
  soa[(long)c * N + i0 + i] = aos[k];
}

__global__ void k_stage_words(const int *__restrict__ d, int n, int *__restrict__ h) {
  const int k = blockIdx.x * STAGE_TB + threadIdx.x;
  if (k < n) h[k] = d[k];
}

static dim3 stage_grid(int n) { return dim3((n + STAGE_TB - 1) / STAGE_TB); }

// Maps the whole pages of [p, p + bytes), which the caller is about to fill, in
// one call: 0.4 us a page instead of 0.85 for a fault each (2.3 MB of fresh
// pages: 280 and 530 us), 12 us where they are mapped already, and the device
// fills the buffer meanwhile.  Where the system has no such advice the faults
// come as they did.
static void map_pages(void *p, size_t bytes) {
#ifdef MADV_POPULATE_WRITE
  const size_t page = 4096, lo = ((size_t)p + page - 1) & ~(page - 1), hi = ((size_t)p + bytes) & ~(page - 1);
  if (hi > lo && hi - lo >= 16 * page) {
    const int err = errno;
    madvise((void *)lo, hi - lo, MADV_POPULATE_WRITE);
    errno = err;
  }
#endif
}

// The buffer: room for every site up to the bound.  Made with the engine (90 us
// and 0.07 us a KB) and written once here, which gives it its pages: left to
// the first positions handed in, that made them take 950 us for 98304 sites
// (160 for 12288) instead of 120 (50).  Engines inside a reference-style call
// never need one.
int stage_create(Engine &e) {
  Stage &b = *e.stage;
  b.sites = std::min(std::max(e.nsite, 512), STAGE_MAX_SITES);
  MM_HIP(hipHostMalloc((void **)&b.h, 3 * sizeof(double) * b.sites));
  memset(b.h, 0, 3 * sizeof(double) * b.sites);
  return 0;
}

int stage_get_sites(Engine &e, const double *soa, double *aos) {
  std::lock_guard<std::mutex> lock(e.stage->lock);
  const Stage &b = *e.stage;
  for (int i0 = 0; i0 < e.nsite; i0 += b.sites) {
    const int n = std::min(b.sites, e.nsite - i0);
    hipLaunchKernelGGL(k_stage_sites, stage_grid(3 * n), dim3(STAGE_TB), 0, e.stream, soa, e.nsite,
                       i0, n, b.h);
    MM_HIP(hipGetLastError());
    map_pages(aos + 3 * (size_t)i0, 3 * sizeof(double) * n);
    MM_HIP(hipStreamSynchronize(e.stream));
    memcpy(aos + 3 * (size_t)i0, b.h, 3 * sizeof(double) * n);
  }
  return 0;
}

int stage_put_sites(Engine &e, double *soa, const double *aos) {
  std::lock_guard<std::mutex> lock(e.stage->lock);
  const Stage &b = *e.stage;
  for (int p0 = 0; p0 < e.nsite; p0 += b.sites) {
    const int pn = std::min(b.sites, e.nsite - p0);
    for (int j = 0; j < pn; j += STAGE_PUT_SITES) {
      const int n = std::min(STAGE_PUT_SITES, pn - j), i0 = p0 + j;
      memcpy(b.h + 3 * (size_t)j, aos + 3 * (size_t)i0, 3 * sizeof(double) * n);
      hipLaunchKernelGGL(k_unstage_sites, stage_grid(3 * n), dim3(STAGE_TB), 0, e.stream,
                         b.h + 3 * (size_t)j, e.nsite, i0, n, soa);
      MM_HIP(hipGetLastError());
    }
    MM_HIP(hipStreamSynchronize(e.stream));
  }
  return 0;
}

int stage_get(Engine &e, const void *d, void *h, size_t bytes) {
  if (!h) { set_last_error("null output"); return -1; }
  std::lock_guard<std::mutex> lock(e.stage->lock);
  const Stage &b = *e.stage;
  const size_t cap = 3 * sizeof(double) * b.sites;
  for (size_t o = 0; o < bytes; o += cap) {
    const size_t n = std::min(cap, bytes - o);
    hipLaunchKernelGGL(k_stage_words, stage_grid((int)(n / 4)), dim3(STAGE_TB), 0, e.stream,
                       (const int *)((const char *)d + o), (int)(n / 4), (int *)b.h);
    MM_HIP(hipGetLastError());
    MM_HIP(hipStreamSynchronize(e.stream));
    memcpy((char *)h + o, b.h, n);
  }
  return 0;
}

}  // namespace mmamd
