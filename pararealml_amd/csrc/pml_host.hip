// Results on their way to the host: the channel-last copy of field-major
// states and the download into ordinary (pageable) memory.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstring>
#include <exception>
#include <mutex>
#include <thread>
#include <vector>

#include "pml_common.h"

namespace pml {

// Field-major states (n states of F planes) -> channel-last, FP64.  Bound by
// HBM (one read, one write); a thread writes the F values of one vertex, so
// the reads of a wavefront are F contiguous runs and its writes one.
template <int F>
__global__ void __launch_bounds__(256) k_channel_last(const double *__restrict__ s,
                                                      double *__restrict__ d, int64_t plane,
                                                      int64_t vertices) {
  for (int64_t v = blockIdx.x * int64_t{256} + threadIdx.x; v < vertices;
       v += int64_t{256} * gridDim.x) {
    const int64_t state = v / plane, p = v - state * plane;
    const double *from = s + state * F * plane + p;
    double x[F];
#pragma unroll
    for (int f = 0; f < F; ++f) x[f] = from[f * plane];
#pragma unroll
    for (int f = 0; f < F; ++f) d[v * F + f] = x[f];
  }
}

// Pinned staging of one download: every worker owns two slots.  At most
// kKept sets outlive their call (kKept x 16 MiB); they are given back by
// pml_graph_cache_clear().
constexpr int kWorkers = 8;
constexpr size_t kSlotBytes = size_t{1} << 20;
constexpr size_t kKept = 2;
static std::mutex g_staging_mu;
static std::vector<char *> g_staging;

static char *take_staging() {
  {
    std::lock_guard<std::mutex> lock(g_staging_mu);
    if (!g_staging.empty()) {
      char *p = g_staging.back();
      g_staging.pop_back();
      return p;
    }
  }
  void *p = nullptr;
  if (hipHostMalloc(&p, 2 * kWorkers * kSlotBytes, hipHostMallocPortable) != hipSuccess) {
    (void)hipGetLastError();
    return nullptr;
  }
  return static_cast<char *>(p);
}

static void give_staging(char *p) {
  {
    std::lock_guard<std::mutex> lock(g_staging_mu);
    if (g_staging.size() < kKept) {
      g_staging.push_back(p);
      return;
    }
  }
  (void)hipHostFree(p);
}

void release_staging() {
  std::lock_guard<std::mutex> lock(g_staging_mu);
  for (char *p : g_staging) (void)hipHostFree(p);
  g_staging.clear();
}

static int worker_count(size_t pieces) {
  const size_t cores = std::max(1u, std::thread::hardware_concurrency());
  return static_cast<int>(std::min({pieces, static_cast<size_t>(kWorkers), cores}));
}

// work(0 .. workers - 1), on as many threads as can be started (this one
// among them; it also does the work of those that could not).
template <class Work>
static void share_out(int workers, Work work) {
  std::thread threads[kWorkers];
  int started = 1;
  try {
    for (; started < workers; ++started) threads[started] = std::thread(work, started);
  } catch (const std::exception &) {
  }
  work(0);
  for (int w = started; w < workers; ++w) work(w);
  for (std::thread &t : threads)
    if (t.joinable()) t.join();
}

// Worker w copies pieces w, w + workers, ... : the next piece is on its way
// into one slot while the last one leaves the other for `dst`.
static hipError_t download_pieces(int device, char *dst, const char *src, size_t bytes, char *slots,
                                  int w, int workers, hipStream_t st) {
  hipError_t e = hipSetDevice(device);
  if (e != hipSuccess) return e;
  hipEvent_t ev[2] = {};
  for (int k = 0; k < 2 && e == hipSuccess; ++k)
    e = hipEventCreateWithFlags(&ev[k], hipEventDisableTiming);
  const size_t pieces = (bytes + kSlotBytes - 1) / kSlotBytes;
  auto size_of = [&](size_t p) { return std::min(kSlotBytes, bytes - p * kSlotBytes); };
  int slot = 0;
  auto fetch = [&](size_t p, int s) {
    if (e == hipSuccess)
      e = hipMemcpyAsync(slots + (2 * w + s) * kSlotBytes, src + p * kSlotBytes, size_of(p),
                         hipMemcpyDeviceToHost, st);
    if (e == hipSuccess) e = hipEventRecord(ev[s], st);
  };
  size_t p = static_cast<size_t>(w);
  if (p < pieces) fetch(p, slot);
  for (; p < pieces && e == hipSuccess; p += workers, slot ^= 1) {
    if (p + workers < pieces) fetch(p + workers, slot ^ 1);
    if (e == hipSuccess) e = hipEventSynchronize(ev[slot]);
    if (e == hipSuccess)
      std::memcpy(dst + p * kSlotBytes, slots + (2 * w + slot) * kSlotBytes, size_of(p));
  }
  // nothing of this worker's may still be in flight when the slots go back
  if (e != hipSuccess) (void)hipStreamSynchronize(st);
  for (int k = 0; k < 2; ++k)
    if (ev[k]) (void)hipEventDestroy(ev[k]);
  return e;
}

}  // namespace pml

using namespace pml;

extern "C" int pml_channel_last(const double *field_major, double *channel_last, int n_fields,
                                int64_t plane, int64_t n_states, void *stream) {
  if (!field_major || !channel_last || plane <= 0 || n_states < 0 || n_fields < 1 || n_fields > 4)
    return fail(PML_E_INVALID, "bad channel-last arguments");
  const int64_t vertices = plane * n_states;
  if (!vertices) return PML_OK;
  const dim3 grid(static_cast<unsigned>(std::min<int64_t>((vertices + 255) / 256, 1 << 16)));
  hipStream_t st = as_stream(stream);
  auto launch = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, grid, dim3(256), 0, st, field_major, channel_last, plane, vertices);
  };
  switch (n_fields) {
    case 1: launch(k_channel_last<1>); break;
    case 2: launch(k_channel_last<2>); break;
    case 3: launch(k_channel_last<3>); break;
    default: launch(k_channel_last<4>); break;
  }
  PML_LAUNCH_CHECK();
  return PML_OK;
}

extern "C" int pml_host_copy(void *dst, const void *src, int64_t bytes) {
  if (bytes < 0 || (bytes && (!dst || !src))) return fail(PML_E_INVALID, "bad host copy arguments");
  const size_t n = static_cast<size_t>(bytes);
  const size_t pieces = (n + kSlotBytes - 1) / kSlotBytes;
  if (!pieces) return PML_OK;
  const int workers = worker_count(pieces);
  share_out(workers, [&](int w) {
    for (size_t p = w; p < pieces; p += workers)
      std::memcpy(static_cast<char *>(dst) + p * kSlotBytes,
                  static_cast<const char *>(src) + p * kSlotBytes,
                  std::min(kSlotBytes, n - p * kSlotBytes));
  });
  return PML_OK;
}

extern "C" int pml_download(void *dst, const void *src, int64_t bytes, void *stream) {
  if (bytes < 0 || (bytes && (!dst || !src))) return fail(PML_E_INVALID, "bad download arguments");
  if (!bytes) return PML_OK;
  hipStream_t st = as_stream(stream);
  int device = 0;
  PML_HIP_CHECK(hipGetDevice(&device));
  // to the copying threads this name is another stream
  if (st == hipStreamPerThread) PML_HIP_CHECK(hipStreamSynchronize(st));
  char *slots = take_staging();
  if (!slots) {  // no pinned memory to be had: the runtime's own copy
    PML_HIP_CHECK(hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, st));
    PML_HIP_CHECK(hipStreamSynchronize(st));
    return PML_OK;
  }
  const size_t n = static_cast<size_t>(bytes);
  const size_t pieces = (n + kSlotBytes - 1) / kSlotBytes;
  const int workers = worker_count(pieces);
  hipError_t err[kWorkers] = {};
  share_out(workers, [&](int w) {
    err[w] = download_pieces(device, static_cast<char *>(dst), static_cast<const char *>(src), n,
                             slots, w, workers, st);
  });
  give_staging(slots);
  for (int w = 0; w < workers; ++w)
    if (err[w] != hipSuccess)
      return fail(PML_E_HIP, std::string("download: ") + hipGetErrorString(err[w]));
  return PML_OK;
}
