// HIP calls of a device with fake::room bytes left, defined in the test program
// so that the library's host code runs without a GPU: addresses are numbers,
// nothing is read or written there.
#pragma once
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <map>

inline double cospi(double x) { return std::cos(M_PI * x); }  // a device function to g++

#include "ctx.h"

namespace fake {
int64_t room = 0;
size_t refuse = 0;  // a request of this size fails
std::map<void *, int64_t> live;
char *next = (char *)((uintptr_t)1 << 44);
inline int64_t held() {
  int64_t n = 0;
  for (auto &b : live) n += b.second;
  return n;
}
}  // namespace fake

#define CHECK(x)                                                     \
  do {                                                               \
    if (!(x)) {                                                      \
      std::printf("line %d: %s is false\n", __LINE__, #x);           \
      std::exit(1);                                                  \
    }                                                                \
  } while (0)

extern "C" {
hipError_t hipMalloc(void **p, size_t n) {
  if ((int64_t)n > fake::room || n == fake::refuse) return hipErrorOutOfMemory;
  fake::room -= (int64_t)n;
  *p = fake::next;
  fake::live[*p] = (int64_t)n;
  fake::next += (n + 4095) / 4096 * 4096 + 4096;
  return hipSuccess;
}
hipError_t hipFree(void *p) {
  auto b = fake::live.find(p);
  if (b == fake::live.end()) {
    std::printf("release of an address that is not an allocation\n");
    std::exit(1);
  }
  fake::room += b->second;
  fake::live.erase(b);
  return hipSuccess;
}
hipError_t hipMemcpy(void *, const void *, size_t, hipMemcpyKind) { return hipSuccess; }
hipError_t hipMemcpyAsync(void *, const void *, size_t, hipMemcpyKind, hipStream_t) { return hipSuccess; }
hipError_t hipMemsetAsync(void *, int, size_t, hipStream_t) { return hipSuccess; }
hipError_t hipLaunchKernel(const void *, dim3, dim3, void **, size_t, hipStream_t) { return hipSuccess; }
hipError_t hipHostMalloc(void **p, size_t n, unsigned) {
  *p = std::calloc(n, 1);
  return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipGetLastError(void) { return hipSuccess; }
hipError_t hipMemGetInfo(size_t *f, size_t *t) {
  *f = (size_t)fake::room;
  *t = (size_t)(fake::room + fake::held());
  return hipSuccess;
}
const char *hipGetErrorString(hipError_t) { return "fake"; }
}
