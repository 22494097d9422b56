// Transfers between a caller's host arrays and device arrays through a
// small pinned buffer of the context, kept as long as it lives.  A kernel
// reorders on the way (the reference's cell order and entity-major or
// column-major layout on the host, component-major rows on the device), so
// the host only copies bytes, and calls on a stream are queued in order: no
// transfer waits for another but for room in the buffer (two halves; the
// copy out of one overlaps the kernels that fill the other).
#pragma once
#include <hip/hip_runtime.h>

#include <vector>

namespace fvk {

enum { IO_ENTITY = 0, IO_COLUMN = 1 };  // host element (o, q) at o ncomp + q, or at q count + o

struct HostIo {
  hipStream_t stream = nullptr;
  // d[q ldd + (where ? where[o] : o)] = h(o, q) for o < count, q < ncomp;
  // h has been read when this returns
  int put(const double *h, int ncomp, int count, const int *where, double *d, size_t ldd, int layout = IO_ENTITY);
  // the reverse, h(o, q) from component comp[q] (null: q); h is written by
  // the time finish() returns
  int get(const double *d, size_t ldd, int ncomp, int count, const int *where, double *h, int layout = IO_ENTITY,
          const int *comp = nullptr);
  // bytes (a multiple of 4) as they are
  int get_raw(const void *d, size_t bytes, void *h);
  int finish();
  // forgets what get() has not delivered (a call that failed half way)
  void drop() {
    seg[0].clear();
    seg[1].clear();
  }
  void free();

 private:
  struct Seg {
    void *h;
    const char *p;
    size_t bytes;
  };
  char *pin = nullptr;
  hipEvent_t ev[2] = {nullptr, nullptr};
  std::vector<Seg> seg[2];
  bool busy[2] = {false, false};
  int cur = 0;
  size_t used = 0;
  int rotate();
  // room for at least one unit and at most want units, in the current half
  int room(size_t unit, size_t want, char *&p, size_t &got);
  void drain(int b);
};

// for the length of a call: nothing is delivered after it
struct IoCall {
  HostIo &io;
  explicit IoCall(HostIo &i) : io(i) {}
  ~IoCall() { io.drop(); }
};

}  // namespace fvk
