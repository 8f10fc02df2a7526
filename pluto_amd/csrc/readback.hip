// Read-back of state arrays into the caller's (pageable) memory.
//
// A kernel gathers the wanted cells of all arrays straight into pinned host
// buffers over the link, a ring of four buffers ahead of the host threads
// that copy them out.  hipMemcpy to pageable memory moved 16 GB/s, one copy
// and one wait per array, and a ghosted box's arrays came whole and were cut
// on the host by one thread: 128^3 read back from a periodic box 10.4 -> 3.7
// ms (50 GB/s; the link 57), from a bounded one 20.0 -> 3.7 ms, 32^3 0.24 ->
// 0.13 and 0.31 -> 0.13 ms, 96 patches of edges 16 to 64 one by one 47 -> 26.
// A box's first read also pins its buffers: 128^3 10.5 -> 4.1 ms, 32^3 0.26 ->
// 0.19 (a process's very first ones, on new host memory, about 1 ms more).

#include "readback.hpp"

#include <algorithm>
#include <atomic>
#include <condition_variable>
#include <cstring>
#include <mutex>
#include <thread>
#include <vector>

namespace pgpu {

namespace {

// elements e0 .. e0 + n - 1 of the arrays one after another
__global__ void __launch_bounds__(256) k_gather_cells(ReadSrc s, long e0, long n, double* out)
{
  const long ni = (long)s.n[0] * s.n[1] * s.n[2];
  for (long t = (long)blockIdx.x * 256 + threadIdx.x; t < n; t += (long)gridDim.x * 256) {
    const long e = e0 + t, q = e / ni;
    const unsigned c = (unsigned)(e - q * ni);   // (a domain's arrays are under 2^32 cells)
    const unsigned r = c / (unsigned)s.n[0], i = c - r * (unsigned)s.n[0];
    const unsigned k = r / (unsigned)s.n[1], j = r - k * (unsigned)s.n[1];
    out[t] = s.a[q][s.first + (long)k * s.plane + (long)j * s.row + i];
  }
}

void drop_buffers(Readback& rb)
{
  for (auto& h : rb.h) {
    if (h) (void)hipHostFree(h);
    h = nullptr;
  }
  rb.elems = 0;
}

// Buffers for a read of `total` doubles: as large as the read, 32 KiB to 4
// MiB (a power of two), and only as many as it fills; a larger read replaces
// them.  (Four of 4 MiB whatever was read pinned 16 MiB an object, and a box's
// first read took longer: 8^3 0.09 ms, now 0.044, 32^3 0.22, now 0.19.)
int make_ring(Readback& rb, long total)
{
  long el = 1l << 12;
  while (el < 1l << 19 && el < total) el *= 2;
  if (rb.elems > el) el = rb.elems;
  for (; el >= 1l << 12; el >>= 2) {   // (less where that is refused)
    if (rb.elems != el) drop_buffers(rb);
    const int need = (int)std::min((long)Readback::NB, (total + el - 1) / el);
    hipError_t e = hipSuccess;
    for (int q = 0; q < need && e == hipSuccess; q++) {
      if (!rb.ev[q]) e = hipEventCreateWithFlags(&rb.ev[q], hipEventDisableTiming);
      if (e == hipSuccess && !rb.h[q])
        e = hipHostMalloc((void**)&rb.h[q], (size_t)el * sizeof(double), hipHostMallocDefault);
    }
    if (e == hipSuccess) {
      rb.elems = el;
      return 0;
    }
    drop_buffers(rb);
    (void)hipGetLastError();
  }
  return (int)hipErrorOutOfMemory;
}

}  // namespace

Readback::~Readback()
{
  drop_buffers(*this);
  for (auto& e : ev)
    if (e) (void)hipEventDestroy(e);
}

int readback(Readback& rb, const ReadSrc& src, double* const* dst, hipStream_t s)
{
  constexpr int NB = Readback::NB;
  const long ni = (long)src.n[0] * src.n[1] * src.n[2], total = ni * src.na;
  if (total <= 0) return (int)hipStreamSynchronize(s);   // (no array asked for: a wait)
  // (the caller's current device may be another)
  struct OnDevice {
    int was = -1;
    explicit OnDevice(hipStream_t s)
    {
      int cur = 0, own = 0;
      if (hipGetDevice(&cur) == hipSuccess && hipStreamGetDevice(s, &own) == hipSuccess && own != cur &&
          hipSetDevice(own) == hipSuccess)
        was = cur;
    }
    ~OnDevice()
    {
      if (was >= 0) (void)hipSetDevice(was);
    }
  } on(s);
  if (const int rc = make_ring(rb, total)) return rc;
  const long ch = rb.elems, nch = (total + ch - 1) / ch;

  // elements [e0, e1) of the concatenation, held from h on, to their arrays
  auto copy_out = [&](const double* h, long e0, long e1) {
    for (long e = e0; e < e1;) {
      const long q = e / ni, c = e - q * ni, m = std::min(e1 - e, ni - c);
      memcpy(dst[q] + c, h + (e - e0), (size_t)m * sizeof(double));
      e += m;
    }
  };

  // chunk c is in its buffer when ready > c; left: threads still copying it
  std::mutex m;
  std::condition_variable more;
  long ready = 0;
  bool stop = false;
  int nw = 0;
  std::atomic<int> left[NB];
  for (auto& l : left) l.store(0);
  auto work = [&](int w) {
    for (long c = 0; c < nch; c++) {
      {
        std::unique_lock<std::mutex> lk(m);
        more.wait(lk, [&] { return ready > c || stop; });
        if (ready <= c) return;
      }
      const long e0 = c * ch, len = std::min(ch, total - e0);
      const long b = len * w / nw, e = len * (w + 1) / nw;
      copy_out(rb.h[c % NB] + b, e0 + b, e0 + e);
      left[c % NB].fetch_sub(1, std::memory_order_release);
    }
  };
  std::vector<std::thread> th;

  hipError_t err = hipSuccess;
  long issued = 0, got = 0;
  while (got < nch && err == hipSuccess) {
    while (issued < nch && issued - got < NB && left[issued % NB].load(std::memory_order_acquire) == 0) {
      const long e0 = issued * ch, len = std::min(ch, total - e0);
      const long nwg = (len + 1023) / 1024;
      hipLaunchKernelGGL(k_gather_cells, dim3((unsigned)nwg), dim3(256), 0, s, src, e0, len, rb.h[issued % NB]);
      err = hipGetLastError();
      if (err == hipSuccess) err = hipEventRecord(rb.ev[issued % NB], s);
      if (err != hipSuccess) break;
      issued++;
    }
    if (err != hipSuccess) break;
    if (issued == got) {   // every buffer is still being copied out
      std::this_thread::yield();
      continue;
    }
    err = hipEventSynchronize(rb.ev[got % NB]);
    if (err != hipSuccess) break;
    if (got == 0 && nch > 1) {
      // a thread copies about 10 GB/s and starts in about 20 us: from two chunks
      // on, up to eight, started only now that there is something to copy (the
      // stream may hold a whole run of steps before the first chunk)
      const int want = (int)std::min(8u, std::max(1u, std::thread::hardware_concurrency() / 2));
      try {
        th.reserve(want);
        for (int w = 0; w < want; w++) th.emplace_back(work, w);
      } catch (...) {   // fewer threads, or none: this one copies
      }
      nw = (int)th.size();   // (read after the first chunk is published)
    }
    if (nw == 0) {
      const long e0 = got * ch;
      copy_out(rb.h[got % NB], e0, std::min(e0 + ch, total));
    }
    left[got % NB].store(nw);
    {
      std::lock_guard<std::mutex> lk(m);
      ready = ++got;
    }
    more.notify_all();
  }
  // (only a failure stops the threads: after the last chunk they still copy)
  if (err != hipSuccess) {
    {
      std::lock_guard<std::mutex> lk(m);
      stop = true;
    }
    more.notify_all();
    (void)hipStreamSynchronize(s);   // nothing writes the buffers any more
  }
  for (auto& x : th) x.join();
  return (int)err;
}

}  // namespace pgpu
