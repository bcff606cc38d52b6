// transfer.hpp -- host Fortran arrays <-> padded device boxes.
//
// A transfer is a list of fields, seen as one run of elements: the host
// arrays end to end, in the caller's layout (x fastest, their own bounds).
// It is cut into chunks.  One launch of k_xfer moves a chunk between a pinned
// host buffer and the device boxes, converting between FP64 and the storage
// type on the way, so nothing is repacked on the host and no packed copy is
// held on the device; the host only copies between the pinned buffer and the
// caller's (pageable) array.  That copy takes about 10 GB/s per thread, and
// it is the first to touch the pages of a fresh dump, so several threads
// take the chunks in turn, each with its own stream and two buffers: one is
// copied while the device works on the other.
//
// Bound by the host link: the 1.55 GB of a 256^3 state go up in 28 ms and
// down in 31 ms (55 and 50 GB/s; one thread: 43 and 116 ms).  The repacking
// through a host copy of each padded box that this replaced took 217 and
// 211 ms; at 16^3 0.08 and 0.09 ms against 0.37 and 0.23 ms.

struct XferField {
  void *dev;
  double *host;
  int wide;             // 1: FP64 box, 0: FP32 box
  int lo[3];            // lower Fortran bound of the host array per axis
  unsigned long first;  // its first element in the run
};
#define XFER_MAXF 12
struct XferSet {
  XferField f[XFER_MAXF];
  int nf;
  unsigned long total;
};

// Pinned memory costs about 0.2 ms per MiB to allocate and a thread about
// 20 us to start, so a small transfer takes small chunks and few threads: a
// 32nd of the run within XFER_CHUNK_MIN..MAX elements (1/2 and 4 MiB; the
// whole run in one launch up to 1 MiB), and a thread for each
// XFER_PER_THREAD elements.  Eight threads reach the link's
// rate; 12 or 16, or chunks of 1 or 2 MiB, made no difference at 256^3.
#define XFER_CHUNK_MIN (64ul * 1024)
#define XFER_CHUNK_MAX (512ul * 1024)
#define XFER_PER_THREAD (512ul * 1024)
#define XFER_THREADS 8

// Elements first .. first+count-1 of the run; buf holds them in order.
template <bool TO_DEV>
__global__ __launch_bounds__(256) void k_xfer(Geo g, XferSet s, unsigned long first, unsigned count,
                                              double *__restrict__ buf) {
  const unsigned t = blockIdx.x * 256u + threadIdx.x;
  if (t >= count) return;
  const unsigned long e = first + t;
  int q = 0;
  while (q + 1 < s.nf && e >= s.f[q + 1].first) ++q;
  const XferField &f = s.f[q];
  const unsigned ex = (unsigned)(g.nx + 3 - f.lo[0]), ey = (unsigned)(g.ny + 3 - f.lo[1]);
  const unsigned l = (unsigned)(e - f.first), r = l / ex, k = r / ey;
  const int c = g.idx((int)(l - r * ex) + f.lo[0], (int)(r - k * ey) + f.lo[1], (int)k + f.lo[2]);
  if (TO_DEV) {
    if (f.wide) ((double *)f.dev)[c] = buf[t];
    else ((float *)f.dev)[c] = (float)buf[t];
  } else {
    buf[t] = f.wide ? ((const double *)f.dev)[c] : (double)((const float *)f.dev)[c];
  }
}

// Pinned buffers, streams and events of the transfers, made as they are
// needed and kept until the device state is freed.
struct XferLane {
  hipStream_t stream = nullptr;  // lane 0, the calling thread's, uses the library stream
  double *buf[2] = {nullptr, nullptr};
  hipEvent_t done[2] = {nullptr, nullptr};
  unsigned long cap = 0;  // elements of each buffer
};
XferLane XL[XFER_THREADS];

void xfer_free_lane(XferLane &l) {
  for (int q = 0; q < 2; ++q) {
    if (l.buf[q]) (void)hipHostFree(l.buf[q]);
    if (l.done[q]) (void)hipEventDestroy(l.done[q]);
  }
  if (l.stream && l.stream != S.stream) (void)hipStreamDestroy(l.stream);
  l = XferLane();
}
void xfer_free() {
  for (XferLane &l : XL) xfer_free_lane(l);
}
hipError_t xfer_lane(XferLane &l, unsigned long elems, int bufs) {
  if (l.cap >= elems && l.buf[bufs - 1]) return hipSuccess;
  xfer_free_lane(l);
  hipError_t e = hipSuccess;
  if (&l == &XL[0]) l.stream = S.stream;
  else e = hipStreamCreateWithFlags(&l.stream, hipStreamNonBlocking);
  for (int q = 0; q < bufs && e == hipSuccess; ++q) {
    e = hipHostMalloc((void **)&l.buf[q], sizeof(double) * elems, hipHostMallocDefault);
    if (e == hipSuccess) e = hipEventCreateWithFlags(&l.done[q], hipEventDisableTiming);
  }
  if (e != hipSuccess) xfer_free_lane(l);
  else l.cap = elems;
  return e;
}

// the host copy of elements first .. first+count-1
void xfer_host(const XferSet &s, unsigned long first, unsigned long count, double *buf, bool to_dev) {
  for (int q = 0; q < s.nf; ++q) {
    const unsigned long f0 = s.f[q].first, f1 = q + 1 < s.nf ? s.f[q + 1].first : s.total;
    const unsigned long a = first > f0 ? first : f0, b = first + count < f1 ? first + count : f1;
    if (a >= b) continue;
    double *h = s.f[q].host + (a - f0), *p = buf + (a - first);
    if (to_dev) memcpy(p, h, sizeof(double) * (b - a));
    else memcpy(h, p, sizeof(double) * (b - a));
  }
}

// chunks `lane`, lane + lanes, ... of the run
hipError_t xfer_run(const XferSet &s, int lane, int lanes, unsigned long chunk, bool to_dev) {
  XferLane &l = XL[lane];
  const unsigned long chunks = (s.total + chunk - 1) / chunk;
  auto size = [&](unsigned long c) { return c + 1 < chunks ? chunk : s.total - c * chunk; };
  unsigned long prev = chunks;  // the chunk whose host copy is still due
  int n = 0;
  for (unsigned long c = (unsigned long)lane; c < chunks; c += (unsigned long)lanes, ++n) {
    const int q = n & 1;
    const unsigned long first = c * chunk, count = size(c);
    hipError_t e = hipSuccess;
    if (to_dev) {
      if (n >= 2) e = hipEventSynchronize(l.done[q]);
      if (e != hipSuccess) return e;
      xfer_host(s, first, count, l.buf[q], true);
    }
    const dim3 gr((unsigned)((count + 255) / 256));
    if (to_dev) hipLaunchKernelGGL(k_xfer<true>, gr, dim3(256), 0, l.stream, S.g, s, first, (unsigned)count, l.buf[q]);
    else hipLaunchKernelGGL(k_xfer<false>, gr, dim3(256), 0, l.stream, S.g, s, first, (unsigned)count, l.buf[q]);
    e = hipGetLastError();
    if (e == hipSuccess) e = hipEventRecord(l.done[q], l.stream);
    if (e != hipSuccess) return e;
    if (!to_dev) {
      if (prev < chunks) {
        e = hipEventSynchronize(l.done[q ^ 1]);
        if (e != hipSuccess) return e;
        xfer_host(s, prev * chunk, size(prev), l.buf[q ^ 1], false);
      }
      prev = c;
    }
  }
  if (!to_dev && prev < chunks) {
    const int q = (n - 1) & 1;
    const hipError_t e = hipEventSynchronize(l.done[q]);
    if (e != hipSuccess) return e;
    xfer_host(s, prev * chunk, size(prev), l.buf[q], false);
  }
  return hipStreamSynchronize(l.stream);
}

// The transfer of s; the library stream must be idle.
int transfer(const XferSet &s, bool to_dev) {
  if (s.nf == 0) return 0;
  unsigned long chunk = s.total / 32;
  if (chunk < XFER_CHUNK_MIN) chunk = XFER_CHUNK_MIN;
  if (chunk > XFER_CHUNK_MAX) chunk = XFER_CHUNK_MAX;
  if (s.total <= 2 * XFER_CHUNK_MIN) chunk = s.total;
  const unsigned long chunks = (s.total + chunk - 1) / chunk;
  int lanes = (int)(s.total / XFER_PER_THREAD < XFER_THREADS ? s.total / XFER_PER_THREAD : XFER_THREADS);
  if (lanes < 1) lanes = 1;
  int dev = 0;
  HIPCHK(hipGetDevice(&dev));
  const int bufs = chunks > 1 ? 2 : 1;
  HIPCHK(xfer_lane(XL[0], chunk, bufs));
  for (int t = 1; t < lanes; ++t)
    if (xfer_lane(XL[t], chunk, bufs) != hipSuccess) {
      (void)hipGetLastError();
      lanes = t;  // fewer pinned buffers to be had: fewer threads
    }
  hipError_t err[XFER_THREADS] = {};
  std::thread th[XFER_THREADS];
  int started = 1;
  try {
    for (; started < lanes; ++started) {
      const int t = started;
      th[t] = std::thread([&s, &err, t, lanes, chunk, to_dev, dev] {
        err[t] = hipSetDevice(dev);
        if (err[t] == hipSuccess) err[t] = xfer_run(s, t, lanes, chunk, to_dev);
      });
    }
  } catch (...) {
    // no more threads to be had: the caller takes the lanes that have none
  }
  err[0] = xfer_run(s, 0, lanes, chunk, to_dev);
  for (int t = started; t < lanes; ++t) err[t] = xfer_run(s, t, lanes, chunk, to_dev);
  for (int t = 1; t < started; ++t) th[t].join();
  for (int t = 0; t < lanes; ++t) HIPCHK(err[t]);
  return 0;
}
