// Copies between pageable host arrays and device memory through a ring of
// pinned buffers.
//
// The runtime's own copy of a pageable array stages it with one thread, about
// 23 GB/s on a host whose bus takes 50.  Here all threads copy a piece into
// (out of) a pinned buffer while the copy engine moves the pieces before it.
// Drop-in call at 16^4 x Ls8 FP64, Nsimd 4, 10 applications (276 MB of
// arrays): 13.3 -> 7.5 ms; 24^4 x Ls16, 20 applications: 125 -> 71 ms.  Arrays
// under 1 MiB stay with the runtime (a 4^4 call: 150 us, 166 us through here).
#include <cstring>

#include "gbx_internal.h"

namespace {

// memcpy by all threads.
void copy_parallel(char *dst, const char *src, size_t n)
{
  constexpr size_t kPiece = 128 << 10;
  const int64_t pieces = (int64_t)((n + kPiece - 1) / kPiece);
#pragma omp parallel for schedule(static) if (pieces > 4)
  for (int64_t i = 0; i < pieces; i++) {
    const size_t o = (size_t)i * kPiece;
    memcpy(dst + o, src + o, o + kPiece <= n ? kPiece : n - o);
  }
}

}  // namespace

int HostRing::prepare()
{
  for (int i = 0; i < kSlots; i++) {
    if (!buf[i]) GBX_HIP(hipHostMalloc(&buf[i], kBytes, hipHostMallocDefault));
    if (!ev[i]) GBX_HIP(hipEventCreateWithFlags(&ev[i], hipEventDisableTiming));
  }
  return GBX_OK;
}

void HostRing::release()
{
  for (int i = 0; i < kSlots; i++) {
    if (ev[i]) {
      (void)hipEventSynchronize(ev[i]);
      (void)hipEventDestroy(ev[i]);
    }
    (void)hipHostFree(buf[i]);
    ev[i] = nullptr;
    buf[i] = nullptr;
    used[i] = false;
  }
}

// Enqueues host -> device on st; src has been read when it returns.
int HostRing::upload(void *dst, const void *src, size_t n, hipStream_t st)
{
  if (n < kSmall) {
    GBX_HIP(hipMemcpyAsync(dst, src, n, hipMemcpyHostToDevice, st));
    return GBX_OK;
  }
  GBX_TRY(prepare());
  for (size_t o = 0; o < n; o += kBytes) {
    const size_t len = o + kBytes <= n ? kBytes : n - o;
    const int i = next;
    next = (next + 1) % kSlots;
    if (used[i]) GBX_HIP(hipEventSynchronize(ev[i]));  // its last piece has left the buffer
    copy_parallel((char *)buf[i], (const char *)src + o, len);
    GBX_HIP(hipMemcpyAsync((char *)dst + o, buf[i], len, hipMemcpyHostToDevice, st));
    GBX_HIP(hipEventRecord(ev[i], st));
    used[i] = true;
  }
  return GBX_OK;
}

// Device -> host behind the work on st; dst is complete when it returns.
int HostRing::download(void *dst, const void *src, size_t n, hipStream_t st)
{
  if (n < kSmall) {
    GBX_HIP(hipMemcpyAsync(dst, src, n, hipMemcpyDeviceToHost, st));
    GBX_HIP(hipStreamSynchronize(st));
    return GBX_OK;
  }
  GBX_TRY(prepare());
  const size_t pieces = (n + kBytes - 1) / kBytes;
  auto len = [&](size_t p) { return (p + 1) * kBytes <= n ? kBytes : n - p * kBytes; };
  auto start = [&](size_t p) -> int {
    const int i = (int)(p % kSlots);  // stream order keeps an earlier upload's use of the buffer ahead
    GBX_HIP(hipMemcpyAsync(buf[i], (const char *)src + p * kBytes, len(p), hipMemcpyDeviceToHost, st));
    GBX_HIP(hipEventRecord(ev[i], st));
    used[i] = true;
    return GBX_OK;
  };
  for (size_t p = 0; p < pieces && p < (size_t)kSlots; p++) {
    if (used[p]) GBX_HIP(hipEventSynchronize(ev[p]));
    GBX_TRY(start(p));
  }
  for (size_t p = 0; p < pieces; p++) {
    const int i = (int)(p % kSlots);
    GBX_HIP(hipEventSynchronize(ev[i]));
    copy_parallel((char *)dst + p * kBytes, (const char *)buf[i], len(p));
    if (p + kSlots < pieces) GBX_TRY(start(p + kSlots));
  }
  GBX_HIP(hipStreamSynchronize(st));
  return GBX_OK;
}
