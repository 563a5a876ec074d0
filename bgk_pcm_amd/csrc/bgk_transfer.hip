// bgk_transfer.hip -- results on their way to the host.
//
// A field leaves the device through pinned staging buffers: a kernel packs rows
// (pitch and pair stride taken out) straight into mapped host memory, and the
// host copies them into the caller's array, chunk by chunk, several chunks in
// flight and each copied by a thread of its own.  hipMemcpy2DAsync into pageable
// memory moved 0.6 GB/s of a 512^2 field and 2.7 GB/s of a 4096^2 one.  Small
// results (gathers, reductions) are written by their kernel into such a buffer:
// one launch and one wait instead of copies each way.
//
// The buffers belong to the process: at most kMaxBuffers of kChunk bytes kept
// for the next use, freed with the last handle.
#include <algorithm>
#include <cstring>
#include <future>
#include <mutex>

#include "bgk_internal.h"

namespace bgk {
namespace {

constexpr size_t kChunk = (size_t)4 << 20;
constexpr int kMaxBuffers = 8;

std::mutex g_mu;
void* g_idle[kMaxBuffers];  // buffers of kChunk bytes (no container: nothing here throws)
int g_nidle = 0;
int g_users = 0;            // handles alive

// rows r0 .. r0 + gridDim.y - 1 of a plane, nx + 2 values each
__global__ void k_pack(const double* __restrict__ src, int stride, int64_t pitch, int r0, int n,
                       double* __restrict__ out) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const int r = blockIdx.y;
  out[(int64_t)r * n + i] = src[((int64_t)(r0 + r) * pitch + i) * stride];
}

void* take() {
  {
    std::lock_guard<std::mutex> lock(g_mu);
    if (g_nidle > 0) return g_idle[--g_nidle];
  }
  void* p = nullptr;
  if (hipHostMalloc(&p, kChunk, hipHostMallocPortable | hipHostMallocMapped) != hipSuccess) {
    (void)hipGetLastError();
    return nullptr;
  }
  return p;
}

void give(void* p) {
  if (!p) return;
  {
    std::lock_guard<std::mutex> lock(g_mu);
    if (g_users > 0 && g_nidle < kMaxBuffers) {
      g_idle[g_nidle++] = p;
      return;
    }
  }
  (void)hipHostFree(p);
}

void copy_rows(double* dst, int64_t ld, const double* src, int n, int rows) {
  if (ld == n) {
    std::memcpy(dst, src, (size_t)rows * n * sizeof(double));
    return;
  }
  for (int r = 0; r < rows; ++r)
    std::memcpy(dst + (int64_t)r * ld, src + (int64_t)r * n, (size_t)n * sizeof(double));
}

// A chunk in flight: its buffer, the event behind its kernel, and the thread
// that waits for it and copies it out.
struct Slot {
  void* buf = nullptr;
  hipEvent_t ev = nullptr;
  std::future<hipError_t> done;
  hipError_t wait() { return done.valid() ? done.get() : hipSuccess; }
};

}  // namespace

void staging_open() {
  std::lock_guard<std::mutex> lock(g_mu);
  ++g_users;
}

void staging_close() {
  void* idle[kMaxBuffers];
  int n = 0;
  {
    std::lock_guard<std::mutex> lock(g_mu);
    if (--g_users == 0)
      while (g_nidle > 0) idle[n++] = g_idle[--g_nidle];
  }
  while (n > 0) (void)hipHostFree(idle[--n]);
}

Staging::Staging() : p_(take()) {}
Staging::~Staging() { give(p_); }
size_t Staging::bytes() { return kChunk; }

bool download_staged(bgk_handle* h, const double* src, int stride, double* dst, int64_t ld,
                     hipError_t* err) {
  const int n = h->nx + 2, rows = h->ny + 2;
  const int per = (int)std::min<int64_t>(rows, (int64_t)(kChunk / sizeof(double)) / n);
  if (per < 1) return false;  // (a row of more than half a million nodes)
  const int chunks = (rows + per - 1) / per;
  *err = hipSuccess;
  auto pack = [&](int c, double* buf) {
    const int r0 = c * per, m = std::min(per, rows - r0);
    // at most 65535 rows per launch
    for (int r = 0; r < m; r += 65535)
      hipLaunchKernelGGL(k_pack, dim3((unsigned)((n + 255) / 256), (unsigned)std::min(m - r, 65535)),
                         dim3(256), 0, h->stream, src, stride, h->pitch, r0 + r, n,
                         buf + (int64_t)r * n);
    return hipGetLastError();
  };
  if (chunks == 1) {
    Staging s;
    if (!s.ptr()) return false;
    double* const buf = static_cast<double*>(s.ptr());
    if ((*err = pack(0, buf)) == hipSuccess) *err = hipStreamSynchronize(h->stream);
    if (*err == hipSuccess) copy_rows(dst, ld, buf, n, rows);
    return true;
  }
  Slot slot[kMaxBuffers];
  int nslot = 0;
  for (int k = 0; k < std::min(kMaxBuffers, chunks); ++k, ++nslot) {
    slot[k].buf = take();
    if (!slot[k].buf) break;
    if (hipEventCreateWithFlags(&slot[k].ev, hipEventDisableTiming) != hipSuccess) {
      (void)hipGetLastError();
      give(slot[k].buf);
      slot[k].buf = nullptr;
      break;
    }
  }
  for (int c = 0; c < chunks && nslot > 0 && *err == hipSuccess; ++c) {
    Slot& s = slot[c % nslot];
    if ((*err = s.wait()) != hipSuccess) break;
    double* const buf = static_cast<double*>(s.buf);
    if ((*err = pack(c, buf)) != hipSuccess) break;
    if ((*err = hipEventRecord(s.ev, h->stream)) != hipSuccess) break;
    const int r0 = c * per, m = std::min(per, rows - r0), device = h->device;
    const hipEvent_t ev = s.ev;
    auto out = [=]() {
      hipError_t e = hipSetDevice(device);
      if (e == hipSuccess) e = hipEventSynchronize(ev);
      if (e == hipSuccess) copy_rows(dst + (int64_t)r0 * ld, ld, buf, n, m);
      return e;
    };
    try {
      s.done = std::async(std::launch::async, out);
    } catch (...) {  // no thread to be had: copy here
      *err = out();
    }
  }
  for (int k = 0; k < nslot; ++k) {
    const hipError_t e = slot[k].wait();
    if (*err == hipSuccess) *err = e;
  }
  // (after an error a kernel may still be writing into a buffer)
  if (*err != hipSuccess) (void)hipStreamSynchronize(h->stream);
  for (int k = 0; k < nslot; ++k) {
    (void)hipEventDestroy(slot[k].ev);
    give(slot[k].buf);
  }
  return nslot > 0;
}

}  // namespace bgk
