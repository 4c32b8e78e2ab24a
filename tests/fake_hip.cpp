// fake_hip.cpp -- a HIP runtime without a GPU, for tests of the library's host
// path: two devices, memory that counts, streams that run what they hold only
// when something waits for them (the latest that a real one may), and the few
// kernels whose results steer the host.  Loaded in front of libamdhip64
// (fake_hip.py); every other kernel does nothing.
#include <hip/hip_runtime_api.h>
#include <sys/mman.h>

#include <cmath>
#include <cstdint>
#include <cstring>
#include <functional>
#include <map>
#include <string>
#include <utility>
#include <vector>

namespace {

struct Block {
  size_t bytes;
  int device;
};
struct Stream {
  int device;
  std::vector<std::function<void()>> work;
};

int device_now = 0;
std::map<void*, Block> blocks;        // device memory
std::map<void*, size_t> host_blocks;  // pinned host memory
std::map<const void*, std::string> kernels;
std::vector<Stream*> streams;
std::vector<std::string> launched;
size_t used[2] = {0, 0}, peak[2] = {0, 0}, capacity = (size_t)288 << 30;
long n_malloc = 0, n_free = 0, n_wait = 0, n_foreign = 0;
double fail_rho = -1.0;       // a P build at this tree scale fails
int fail_launch = 0;          // countdown: the n-th launch of `fail_kernel` fails
std::string fail_kernel;
hipError_t last_error = hipSuccess;
struct Config {
  dim3 grid, block;
  size_t lds;
  hipStream_t s;
} config;

void drain(Stream* s) {
  std::vector<std::function<void()>> work;
  work.swap(s->work);
  for (auto& f : work) f();
}
void drain_all() {
  for (Stream* s : streams) drain(s);
}
Stream* of(hipStream_t s) { return reinterpret_cast<Stream*>(s); }

template <typename T>
T arg(void** a, int k) {
  return *static_cast<T*>(a[k]);
}

// the tree scales of the last P build: lpr of set k is -(ln rho_k - 0.3)^2
const double* rho_now = nullptr;
int sets_now = 0;
double lpr_of(int r, int q, int nm) {
  const double x = std::log(rho_now[sets_now == nm ? q : r * nm + q]) - 0.3 - 0.01 * q;
  return -100.0 * x * x;
}

std::function<void()> emulate(const std::string& name, dim3 grid, void** a) {
  auto is = [&](const char* n) { return name.find(n) != std::string::npos; };
  if (is("pbuild_kernel")) {
    auto rho = arg<const double*>(a, 4);
    auto active = arg<const uint8_t*>(a, 5);
    auto nbr = arg<int>(a, 7);
    auto perr = arg<unsigned long long*>(a, 15);
    const int n = (int)grid.y;
    return [=] {
      rho_now = rho;
      sets_now = n;
      for (int k = 0; k < n; ++k)
        if (active[k] && rho[k] == fail_rho)  // (set k, branch 0, row 1, column 2), check 1
          *perr = std::min(*perr, ((((unsigned long long)k * nbr) * 64 + 1) * 65 + 2) << 2 | 1);
    };
  }
  if (is("transpose_codes_kernel")) {
    auto src = arg<const uint8_t*>(a, 0);
    auto ncols = arg<int64_t>(a, 1);
    auto nl = arg<int>(a, 2);
    auto dst = arg<uint8_t*>(a, 3);
    auto ld = arg<int64_t>(a, 4);
    return [=] {
      for (int64_t c = 0; c < ncols; ++c)
        for (int l = 0; l < nl; ++l) dst[(size_t)l * ld + c] = src[(size_t)c * nl + l];
    };
  }
  if (is("region_reduce_aligned_kernel")) {
    auto active = arg<const uint8_t*>(a, 4);
    auto r0 = arg<int>(a, 5), nm = arg<int>(a, 6);
    auto l = arg<double*>(a, 8), e = arg<double*>(a, 9), sq = arg<double*>(a, 10);
    auto perr = arg<const unsigned long long*>(a, 11);
    auto head = arg<double*>(a, 12);
    const int nr = (int)grid.x;
    return [=] {
      std::memcpy(head, perr, 8);
      if (*perr != ~0ull) return;
      for (int r = 0; r < nr; ++r)
        for (int q = 0; q < nm; ++q) {
          if (active && !active[r * nm + q]) continue;
          l[(size_t)(r0 + r) * nm + q] = lpr_of(r, q, nm);
          e[(size_t)(r0 + r) * nm + q] = sq ? 0.0 : 0.5;
          if (sq) sq[(size_t)(r0 + r) * nm + q] = 1.0;
        }
    };
  }
  if (is("region_reduce_kernel")) {
    auto nm = arg<int>(a, 3);
    auto l = arg<double*>(a, 5), e = arg<double*>(a, 6);
    auto perr = arg<const unsigned long long*>(a, 7);
    auto head = arg<double*>(a, 8);
    const int nr = (int)grid.x;
    return [=] {
      if (head) std::memcpy(head, perr, 8);
      if (head && *perr != ~0ull) return;
      for (int r = 0; r < nr; ++r)
        for (int q = 0; q < nm; ++q) {
          l[(size_t)r * nm + q] = lpr_of(r, q, nm);
          e[(size_t)r * nm + q] = 0.5;
        }
    };
  }
  if (is("lik_small_kernel")) {
    auto n = arg<int>(a, 1);
    auto leaves = arg<const int32_t*>(a, 6);
    auto dist = arg<const double*>(a, 7);
    auto ncols = arg<int64_t>(a, 8);
    auto z = arg<double*>(a, 10);
    auto bad = arg<int*>(a, 13);
    return [=] {
      for (int64_t k = 0; k < ncols * ((n + 1) / 2); ++k)
        if (leaves[k] < -1 && !(dist && leaves[k] == -2)) *bad = 1;
      for (int64_t k = 0; k < ncols; ++k) z[k] = 1.0;
    };
  }
  return nullptr;
}

}  // namespace

extern "C" {

// ---- what the tests ask and set ---------------------------------------------
void fake_reset() {
  launched.clear();
  n_malloc = n_free = n_wait = n_foreign = 0;
  peak[0] = used[0], peak[1] = used[1];
  fail_rho = -1.0;
  fail_launch = 0;
}
void fake_capacity(size_t bytes) { capacity = bytes; }
void fake_fail_rho(double r) { fail_rho = r; }
void fake_fail_launch(const char* name, int nth) { fail_kernel = name, fail_launch = nth; }
size_t fake_used(int d) { return used[d]; }
size_t fake_peak(int d) { return peak[d]; }
long fake_count(int what) { return what == 0 ? n_malloc : what == 1 ? n_free : what == 2 ? n_wait : n_foreign; }
long fake_launches(const char* name) {
  long n = 0;
  for (auto& s : launched) n += s.find(name) != std::string::npos;
  return n;
}

// ---- the runtime ------------------------------------------------------------
hipError_t hipGetDeviceCount(int* n) { return *n = 2, hipSuccess; }
hipError_t hipSetDevice(int d) { return device_now = d, hipSuccess; }
hipError_t hipGetDevice(int* d) { return *d = device_now, hipSuccess; }
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600* p, int) {
  std::memset(p, 0, sizeof *p);
  p->multiProcessorCount = 256;
  return hipSuccess;
}
hipError_t hipGetLastError() { return std::exchange(last_error, hipSuccess); }
const char* hipGetErrorString(hipError_t e) { return e == hipErrorOutOfMemory ? "out of memory" : "error"; }

hipError_t hipMalloc(void** p, size_t bytes) {
  ++n_malloc;
  *p = nullptr;
  if (used[device_now] + bytes > capacity) return hipErrorOutOfMemory;
  *p = mmap(nullptr, bytes, PROT_READ | PROT_WRITE, MAP_PRIVATE | MAP_ANONYMOUS | MAP_NORESERVE, -1, 0);
  blocks[*p] = {bytes, device_now};
  used[device_now] += bytes;
  peak[device_now] = std::max(peak[device_now], used[device_now]);
  return hipSuccess;
}
hipError_t hipFree(void* p) {  // waits for the device
  ++n_free;
  drain_all();
  auto b = blocks.find(p);
  if (b == blocks.end()) return hipErrorInvalidValue;
  used[b->second.device] -= b->second.bytes;
  munmap(p, b->second.bytes);
  blocks.erase(b);
  return hipSuccess;
}
hipError_t hipHostMalloc(void** p, size_t bytes, unsigned) {
  *p = ::operator new(bytes);
  return hipSuccess;
}
hipError_t hipHostFree(void* p) { return ::operator delete(p), hipSuccess; }

hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) {
  auto* x = new Stream{device_now, {}};
  streams.push_back(x);
  return *s = reinterpret_cast<hipStream_t>(x), hipSuccess;
}
hipError_t hipStreamCreate(hipStream_t* s) { return hipStreamCreateWithFlags(s, 0); }
hipError_t hipStreamSynchronize(hipStream_t s) { return ++n_wait, drain(of(s)), hipSuccess; }
hipError_t hipDeviceSynchronize() { return ++n_wait, drain_all(), hipSuccess; }
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned) { return drain_all(), hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t s) { return drain(of(s)), hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) {
  return *e = reinterpret_cast<hipEvent_t>(&config), hipSuccess;
}
hipError_t hipEventCreate(hipEvent_t* e) { return hipEventCreateWithFlags(e, 0); }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return drain_all(), hipSuccess; }
hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t) { return *ms = 1.0f, hipSuccess; }

hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t q) {
  for (const void* p : {(const void*)d, s}) {  // memory of another device than the stream's
    auto b = blocks.upper_bound(const_cast<void*>(p));
    if (b != blocks.begin() && (--b, (const char*)p < (const char*)b->first + b->second.bytes) &&
        b->second.device != of(q)->device)
      ++n_foreign;
  }
  of(q)->work.push_back([=] { std::memcpy(d, s, n); });
  return hipSuccess;
}
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind) {
  return drain_all(), std::memcpy(d, s, n), hipSuccess;
}
hipError_t hipMemset(void* d, int v, size_t n) { return drain_all(), std::memset(d, v, n), hipSuccess; }
hipError_t hipMemsetAsync(void* d, int v, size_t n, hipStream_t q) {
  of(q)->work.push_back([=] { std::memset(d, v, n); });
  return hipSuccess;
}

hipError_t hipFuncSetAttribute(const void*, hipFuncAttribute, int) { return hipSuccess; }
hipError_t hipOccupancyMaxActiveBlocksPerMultiprocessor(int* n, const void*, int, size_t) {
  return *n = 2, hipSuccess;
}
hipError_t hipGetSymbolAddress(void** p, const void*) {
  static void* scratch = ::operator new(64u << 20);
  return *p = scratch, hipSuccess;
}
void** __hipRegisterFatBinary(const void*) { return nullptr; }
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void* host, char*, const char* name, unsigned, void*, void*, void*,
                           void*, int*) {
  kernels[host] = name;
}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t lds, hipStream_t s) {
  return config = {g, b, lds, s}, hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3* g, dim3* b, size_t* lds, hipStream_t* s) {
  return *g = config.grid, *b = config.block, *lds = config.lds, *s = config.s, hipSuccess;
}
hipError_t hipLaunchKernel(const void* f, dim3 grid, dim3, void** args, size_t, hipStream_t s) {
  const std::string& name = kernels[f];
  if (fail_launch > 0 && name.find(fail_kernel) != std::string::npos && --fail_launch == 0)
    return last_error = hipErrorLaunchFailure;
  launched.push_back(name);
  if (of(s)->device != device_now) ++n_foreign;
  if (auto run = emulate(name, grid, args)) of(s)->work.push_back(run);
  return hipSuccess;
}

}  // extern "C"
