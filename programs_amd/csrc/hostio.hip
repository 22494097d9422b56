// Host transfers through a pinned buffer (hostio.h).
#include "hostio.h"

#include <algorithm>
#include <cstring>

#include "ctx.h"
#include "threads.h"

namespace fvk {

// one half of the pinned buffer: large enough that the wait for a half is
// rare, small enough to stay in the host's cache between copy and kernel
constexpr size_t kHalf = (size_t)4 << 20;

struct IoMap {
  int comp[9];
};

// Consecutive threads take consecutive host elements: the pinned buffer is
// read and written over PCIe, where only whole lines are fast.
template <bool PUT>
__global__ __launch_bounds__(BS) void k_io(double *__restrict__ pin, unsigned first, unsigned cnt, unsigned ncomp,
                                           unsigned count, int layout, const int *__restrict__ where, double *__restrict__ d,
                                           size_t ldd, IoMap map) {
  for (unsigned i = blockIdx.x * BS + threadIdx.x; i < cnt; i += gridDim.x * BS) {
    const unsigned e = first + i;
    const unsigned o = layout == IO_ENTITY ? e / ncomp : e % count, q = layout == IO_ENTITY ? e % ncomp : e / count;
    const size_t z = (size_t)map.comp[q] * ldd + (where ? (unsigned)where[o] : o);
    if (PUT) d[z] = pin[i];
    else pin[i] = d[z];
  }
}

__global__ __launch_bounds__(BS) void k_io_raw(unsigned *__restrict__ pin, const unsigned *__restrict__ d, size_t cnt) {
  for (size_t i = blockIdx.x * (size_t)BS + threadIdx.x; i < cnt; i += (size_t)gridDim.x * BS) pin[i] = d[i];
}

static int io_grid(size_t cnt) { return (int)std::max<size_t>(1, std::min<size_t>((cnt + BS - 1) / BS, 2048)); }

// Four threads from 1 MiB on: one fills a caller's fresh pages at about a
// quarter of the PCIe rate.
static void copy_bytes(void *dst, const void *src, size_t n) {
  constexpr size_t kPar = (size_t)1 << 20;
  if (n < kPar) {
    std::memcpy(dst, src, n);
    return;
  }
  constexpr int T = 4;
  on_threads(T, [=](int t) {
    const size_t a = n / T * t, b = t == T - 1 ? n : n / T * (t + 1);
    std::memcpy((char *)dst + a, (const char *)src + a, b - a);
  });
}

void HostIo::drain(int b) {
  for (const Seg &s : seg[b]) copy_bytes(s.h, s.p, s.bytes);
  seg[b].clear();
  busy[b] = false;
}

int HostIo::rotate() {
  FVK_HIP(hipEventRecord(ev[cur], stream));
  busy[cur] = true;
  cur ^= 1;
  used = 0;
  if (busy[cur]) {
    FVK_HIP(hipEventSynchronize(ev[cur]));
    drain(cur);
  }
  return 0;
}

int HostIo::room(size_t unit, size_t want, char *&p, size_t &got) {
  if (!pin) {
    FVK_HIP(hipHostMalloc((void **)&pin, 2 * kHalf, hipHostMallocDefault));
    for (auto &e : ev) FVK_HIP(hipEventCreateWithFlags(&e, hipEventDisableTiming));
  }
  used = (used + 63) / 64 * 64;
  if (used + std::min(unit * want, (size_t)65536) > kHalf) {
    const int rc = rotate();
    if (rc) return rc;
  }
  got = std::min(want, (kHalf - used) / unit);
  p = pin + (size_t)cur * kHalf + used;
  used += got * unit;
  return 0;
}

int HostIo::put(const double *h, int ncomp, int count, const int *where, double *d, size_t ldd, int layout) {
  const size_t total = (size_t)ncomp * count;
  IoMap map;
  for (int q = 0; q < 9; ++q) map.comp[q] = q;
  for (size_t e = 0; e < total;) {
    char *p;
    size_t got;
    const int rc = room(sizeof(double), total - e, p, got);
    if (rc) return rc;
    copy_bytes(p, h + e, got * sizeof(double));
    k_io<true><<<io_grid(got), BS, 0, stream>>>((double *)p, (unsigned)e, (unsigned)got, ncomp, count, layout, where, d, ldd, map);
    e += got;
  }
  FVK_HIP(hipGetLastError());
  return 0;
}

int HostIo::get(const double *d, size_t ldd, int ncomp, int count, const int *where, double *h, int layout,
                const int *comp) {
  const size_t total = (size_t)ncomp * count;
  IoMap map;
  for (int q = 0; q < 9; ++q) map.comp[q] = comp && q < ncomp ? comp[q] : q;
  for (size_t e = 0; e < total;) {
    char *p;
    size_t got;
    const int rc = room(sizeof(double), total - e, p, got);
    if (rc) return rc;
    k_io<false><<<io_grid(got), BS, 0, stream>>>((double *)p, (unsigned)e, (unsigned)got, ncomp, count, layout, where,
                                                 const_cast<double *>(d), ldd, map);
    seg[cur].push_back(Seg{h + e, p, got * sizeof(double)});
    e += got;
  }
  FVK_HIP(hipGetLastError());
  return 0;
}

int HostIo::get_raw(const void *d, size_t bytes, void *h) {
  for (size_t e = 0, total = bytes / 4; e < total;) {
    char *p;
    size_t got;
    const int rc = room(4, total - e, p, got);
    if (rc) return rc;
    k_io_raw<<<io_grid(got), BS, 0, stream>>>((unsigned *)p, (const unsigned *)d + e, got);
    seg[cur].push_back(Seg{(char *)h + 4 * e, p, got * 4});
    e += got;
  }
  FVK_HIP(hipGetLastError());
  return 0;
}

int HostIo::finish() {
  FVK_HIP(hipStreamSynchronize(stream));
  drain(cur ^ 1);
  drain(cur);
  used = 0;
  return 0;
}

void HostIo::free() {
  for (auto &e : ev)
    if (e) hipEventDestroy(e);
  if (pin) hipHostFree(pin);
  *this = HostIo();
}

}  // namespace fvk
