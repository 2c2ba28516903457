// A stand-in for the HIP runtime, defined in the test program: the dynamic
// linker binds libpainty_hip.so's calls to the program's symbols first, so
// the library's host code runs where there is no device.  Memory is host
// memory, copies happen at once, and kernels are recorded instead of run.
//
// It can fail the n-th device allocation from now (fail_in), keeps the order
// of launches (launches), and notices a copy that overwrites or reads what an
// operation still queued on another stream reads or writes (hazards).
#pragma once

#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <string>
#include <vector>

struct dim3 {
  uint32_t x, y, z;
};

namespace host_hip {


struct Op {  // a queued copy
  void* stream;
  const char *src, *dst;
  size_t bytes;
};

struct State {
  std::map<const void*, std::string> kernels;
  std::map<char*, size_t> dev, pinned;  // live allocations
  size_t dev_bytes = 0, pinned_bytes = 0, pinned_most = 0;
  int fail_in = 0;  // 1: the next hipMalloc fails; 0: none
  int last_error = 0;
  std::vector<Op> queued;
  std::vector<std::string> hazards;
  void (*on_launch)(const std::string& name, void** args) = nullptr;
  struct {
    dim3 grid, block;
    size_t lds;
    void* stream;
  } call{};
};
inline State& state() {
  static State s;
  return s;
}

inline bool live(const void* p) {
  for (const auto& a : state().dev)
    if ((const char*)p >= a.first && (const char*)p < a.first + a.second) return true;
  return false;
}
// Does the 8-byte value v stand at an 8-byte boundary of [p, p + bytes)?
template <class T>
bool holds(const void* p, size_t bytes, T v) {
  static_assert(sizeof(T) == 8, "8-byte values");
  for (size_t i = 0; i + 8 <= bytes; i += 8)
    if (!std::memcmp((const char*)p + i, &v, 8)) return true;
  return false;
}
// Does the address of a live device allocation of `size` bytes?
inline bool holds_alloc(const void* p, size_t bytes, size_t size) {
  for (const auto& a : state().dev)
    if (a.second == size && holds(p, bytes, a.first)) return true;
  return false;
}
inline void drain(void* stream) {
  std::vector<Op> rest;
  for (const Op& o : state().queued)
    if (o.stream != stream) rest.push_back(o);
  state().queued.swap(rest);
}
inline int error(int e) { return e ? state().last_error = e : 0; }

}  // namespace host_hip

#define HOST_HIP extern "C" __attribute__((visibility("default"), used))

HOST_HIP int hipGetDeviceCount(int* n) { return *n = 1, 0; }
HOST_HIP int hipSetDevice(int) { return 0; }
HOST_HIP int hipGetDevice(int* d) { return *d = 0, 0; }
HOST_HIP int hipDeviceGetAttribute(int* v, int, int) { return *v = 256, 0; }
HOST_HIP int hipOccupancyMaxActiveBlocksPerMultiprocessor(int* v, const void*, int, size_t) {
  return *v = 1, 0;
}
HOST_HIP int hipGetSymbolAddress(void** p, const void* s) { return *p = (void*)s, 0; }
HOST_HIP int hipGetLastError() {
  const int e = host_hip::state().last_error;
  host_hip::state().last_error = 0;
  return e;
}
HOST_HIP const char* hipGetErrorString(int e) { return e == 2 ? "out of memory" : "error"; }
HOST_HIP int hipMemGetInfo(size_t* f, size_t* t) { return *f = *t = (size_t)64 << 30, 0; }

HOST_HIP int hipStreamCreateWithFlags(void** s, unsigned) { return *s = std::malloc(1), 0; }
HOST_HIP int hipExtStreamCreateWithCUMask(void** s, uint32_t, const uint32_t*) {
  return *s = std::malloc(1), 0;
}
HOST_HIP int hipStreamSynchronize(void* s) { return host_hip::drain(s), 0; }
HOST_HIP int hipStreamDestroy(void* s) { return host_hip::drain(s), std::free(s), 0; }
struct HostEvent {
  void* stream;
};
HOST_HIP int hipEventCreateWithFlags(void** e, unsigned) { return *e = new HostEvent{}, 0; }
HOST_HIP int hipEventCreate(void** e) { return *e = new HostEvent{}, 0; }
HOST_HIP int hipEventDestroy(void* e) { return delete (HostEvent*)e, 0; }
HOST_HIP int hipEventRecord(void* e, void* s) { return ((HostEvent*)e)->stream = s, 0; }
HOST_HIP int hipEventQuery(void*) { return 0; }
HOST_HIP int hipEventSynchronize(void* e) { return host_hip::drain(((HostEvent*)e)->stream), 0; }
HOST_HIP int hipStreamWaitEvent(void*, void* e, unsigned) { return hipEventSynchronize(e); }
HOST_HIP int hipEventElapsedTime(float* ms, void*, void*) { return *ms = 0.0f, 0; }

HOST_HIP int hipMalloc(void** p, size_t n) {
  auto& S = host_hip::state();
  if (S.fail_in > 0 && --S.fail_in == 0) return *p = nullptr, host_hip::error(2);
  char* q = (char*)std::aligned_alloc(256, (n + 511) / 256 * 256);
  std::memset(q, 0, n);
  S.dev[q] = n;
  S.dev_bytes += n;
  return *p = q, 0;
}
HOST_HIP int hipFree(void* p) {
  auto& S = host_hip::state();
  if (!p) return 0;
  S.queued.clear();  // hipFree waits for the device
  const auto it = S.dev.find((char*)p);
  if (it == S.dev.end()) return host_hip::error(1);
  S.dev_bytes -= it->second;
  S.dev.erase(it);
  std::free(p);
  return 0;
}
HOST_HIP int hipHostMalloc(void** p, size_t n, unsigned) {
  auto& S = host_hip::state();
  char* q = (char*)std::calloc(1, n ? n : 1);
  S.pinned[q] = n;
  S.pinned_bytes += n;
  if (S.pinned_bytes > S.pinned_most) S.pinned_most = S.pinned_bytes;
  return *p = q, 0;
}
HOST_HIP int hipHostFree(void* p) {
  auto& S = host_hip::state();
  const auto it = S.pinned.find((char*)p);
  if (it == S.pinned.end()) return host_hip::error(1);
  S.pinned_bytes -= it->second;
  S.pinned.erase(it);
  std::free(p);
  return 0;
}
HOST_HIP int hipHostGetDevicePointer(void** d, void* h, unsigned) { return *d = h, 0; }

HOST_HIP int hipMemcpyAsync(void* dst, const void* src, size_t n, int kind, void* s) {
  auto& S = host_hip::state();
  const char *d = (const char*)dst, *q = (const char*)src;
  const bool to_dev = kind == 1 || kind == 3, from_dev = kind == 2 || kind == 3;
  if (n && ((to_dev && !host_hip::live(dst)) || (from_dev && !host_hip::live(src))))
    S.hazards.push_back("copy to or from memory that is not allocated");
  const auto meet = [](const char* a, size_t an, const char* b, size_t bn) {
    return a < b + bn && b < a + an;
  };
  for (const auto& o : S.queued)
    if (o.stream != s && (meet(d, n, o.src, o.bytes) || meet(d, n, o.dst, o.bytes) ||
                          meet(q, n, o.dst, o.bytes)))
      S.hazards.push_back("copy overtakes one queued on another stream");
  S.queued.push_back(host_hip::Op{s, q, d, n});
  std::memcpy(dst, src, n);
  return 0;
}

HOST_HIP void** __hipRegisterFatBinary(const void* data) { return (void**)data; }
HOST_HIP void __hipUnregisterFatBinary(void**) {}
HOST_HIP void __hipRegisterFunction(void**, const void* host, char*, const char* name, unsigned,
                                    void*, void*, void*, void*, int*) {
  host_hip::state().kernels[host] = name;
}
HOST_HIP void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
HOST_HIP int __hipPushCallConfiguration(dim3 g, dim3 b, size_t lds, void* s) {
  host_hip::state().call = {g, b, lds, s};
  return 0;
}
HOST_HIP int __hipPopCallConfiguration(dim3* g, dim3* b, size_t* lds, void** s) {
  const auto& c = host_hip::state().call;
  return *g = c.grid, *b = c.block, *lds = c.lds, *s = c.stream, 0;
}
HOST_HIP int hipLaunchKernel(const void* f, dim3, dim3, void** args, size_t, void*) {
  auto& S = host_hip::state();
  if (S.on_launch) S.on_launch(S.kernels[f], args);
  return 0;
}
HOST_HIP int hipLaunchCooperativeKernel(const void* f, dim3 g, dim3 b, void** args, unsigned,
                                        void* s) {
  return hipLaunchKernel(f, g, b, args, 0, s);
}
