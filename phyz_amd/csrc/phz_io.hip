// phz_io.hip — state layout kernels (ahead-of-time compiled for gfx950).
//
// The C ABI hands over world-major f64 rows (the reference wire layout,
// crates/phyz-gpu/src/layout.rs:327-373); the step kernel keeps state as
// structure-of-arrays [j][stride] in the sim's precision so that lane-per-world
// loads and stores coalesce. These kernels move rows between the two layouts.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <mutex>

constexpr int kPhzRowParts = 3;
struct PhzRowParts {  // must match phz_host.cpp
  void* soa[kPhzRowParts];
  void* rows[kPhzRowParts];
  int width[kPhzRowParts];
  int parts, first, count, stride;
};

namespace {

// World-major rows against structure-of-arrays columns, a tile of 64 worlds x
// 64 columns per workgroup through LDS so that both sides are read and written
// in whole lines; one grid row per part, so q, v and ctrl are one launch, one
// grid layer per column tile: a slot of wide rows holds few worlds (two tiles
// of 64 at 1056 values), and their columns in one workgroup's turn left PCIe
// idle. The rows are pinned host memory (move_rows in phz_host.cpp), which the
// kernels access over PCIe themselves: no device staging, no copy command,
// half the bytes where the sim is f32. Bound by PCIe in large launches and by
// the launch itself in small ones. The lane-per-world form read and wrote rows
// 8 bytes a lane, a row's pitch apart, in f64; calls before and after are with
// move_rows.
constexpr int kTile = 64;

// rows[w][c] = (R) soa[c][first + w]
template <class T, class R> __global__ void __launch_bounds__(256) rows_out(PhzRowParts p) {
  __shared__ T tile[kTile][kTile + 1];
  const int width = p.width[blockIdx.y], w0 = blockIdx.x * kTile, nw = min(kTile, p.count - w0);
  const int c0 = blockIdx.z * kTile, nc = min(kTile, width - c0);
  if (nc <= 0) return;  // a narrower part
  const T* soa = (const T*)p.soa[blockIdx.y] + p.first + w0;
  R* rows = (R*)p.rows[blockIdx.y] + (size_t)w0 * width;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  if (lane < nw)
    for (int c = wave; c < nc; c += 4) tile[lane][c] = soa[(size_t)(c0 + c) * p.stride + lane];
  __syncthreads();
  for (int k = threadIdx.x; k < nw * nc; k += 256) {
    const int w = k / nc, c = k - w * nc;
    rows[(size_t)w * width + c0 + c] = (R)tile[w][c];
  }
}

// soa[c][first + w] = rows[w][c]
template <class T> __global__ void __launch_bounds__(256) rows_in(PhzRowParts p) {
  __shared__ T tile[kTile][kTile + 1];
  const int width = p.width[blockIdx.y], w0 = blockIdx.x * kTile, nw = min(kTile, p.count - w0);
  const int c0 = blockIdx.z * kTile, nc = min(kTile, width - c0);
  if (nc <= 0) return;
  T* soa = (T*)p.soa[blockIdx.y] + p.first + w0;
  const T* rows = (const T*)p.rows[blockIdx.y] + (size_t)w0 * width;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll 4
  for (int k = threadIdx.x; k < nw * nc; k += 256) {
    const int w = k / nc, c = k - w * nc;
    tile[w][c] = rows[(size_t)w * width + c0 + c];
  }
  __syncthreads();
  if (lane < nw)
    for (int c = wave; c < nc; c += 4) soa[(size_t)(c0 + c) * p.stride + lane] = tile[lane][c];
}

// One workgroup per tile of worlds, part and tile of columns.
dim3 rows_grid(const PhzRowParts* p) {
  int width = 1;
  for (int k = 0; k < p->parts; k++) width = width > p->width[k] ? width : p->width[k];
  return dim3((p->count + kTile - 1) / kTile, p->parts, (width + kTile - 1) / kTile);
}

template <class T> __global__ void fill_zero(T* __restrict__ dst, size_t n) {
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) dst[i] = T(0);
}

// SplitMix64 world seeds (crates/phyz-gpu/src/policy_pipeline.rs:417-424).
__global__ void seed_worlds(uint64_t* __restrict__ rng, uint64_t seed, int nworld) {
  const int w = blockIdx.x * blockDim.x + threadIdx.x;
  if (w >= nworld) return;
  uint64_t z = seed + 0x9E3779B97F4A7C15ull * (uint64_t)(w + 1);
  z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
  z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
  z = z ^ (z >> 31);
  rng[w] = z ? z : 1;
}

// dst[i] = src[i], 4-byte words (state snapshots; a kernel rather than a
// memcpy node so that a captured rollout holds only kernel nodes).
__global__ void copy_words(uint32_t* __restrict__ dst, const uint32_t* __restrict__ src, size_t n) {
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) dst[i] = src[i];
}

constexpr int kBlock = 256;
inline int blocks(size_t n) { return (int)((n + kBlock - 1) / kBlock); }

constexpr size_t kScratchBytes = size_t(32) << 20;
constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
void* g_scratch_ptr[kMaxDevices] = {};
std::mutex g_scratch_use[kMaxDevices];

}  // namespace

// Held by a caller across its whole use of device `dev`'s scratch array
// (stage, copy out, synchronize), so calls from several threads or sims on
// one GPU take turns instead of overwriting each other's rows.
std::mutex& phz_io_scratch_mutex(int dev) { return g_scratch_use[dev]; }

// Staging rows for callers that cannot allocate device memory
// (phz_readback_states_noalloc): 32 MiB per GPU, held until the process ends.
// Every call on a GPU shares that GPU's copy; callers serialize their use of
// it with phz_io_scratch_mutex. In host code `scratch` names a host-side stand-in, never the device
// memory: use the address phz_io_scratch returns.
static __device__ __align__(256) double scratch[kScratchBytes / sizeof(double)];

extern "C" {

// soa_f64, rows_f64: the element types; rows of a f32 array may be f64.
hipError_t phz_io_rows_out(const PhzRowParts* p, int soa_f64, int rows_f64, hipStream_t s) {
  if (p->count <= 0 || p->parts <= 0) return hipSuccess;
  const dim3 grid = rows_grid(p), block(256);
  if (soa_f64 && rows_f64) hipLaunchKernelGGL(HIP_KERNEL_NAME(rows_out<double, double>), grid, block, 0, s, *p);
  else if (soa_f64) return hipErrorInvalidValue;
  else if (rows_f64) hipLaunchKernelGGL(HIP_KERNEL_NAME(rows_out<float, double>), grid, block, 0, s, *p);
  else hipLaunchKernelGGL(HIP_KERNEL_NAME(rows_out<float, float>), grid, block, 0, s, *p);
  return hipGetLastError();
}

hipError_t phz_io_rows_in(const PhzRowParts* p, int f64, hipStream_t s) {
  if (p->count <= 0 || p->parts <= 0) return hipSuccess;
  const dim3 grid = rows_grid(p), block(256);
  if (f64) hipLaunchKernelGGL(rows_in<double>, grid, block, 0, s, *p);
  else hipLaunchKernelGGL(rows_in<float>, grid, block, 0, s, *p);
  return hipGetLastError();
}

// Zero-fill with a kernel (no hipMemsetAsync, so a captured graph stays valid).
hipError_t phz_io_zero(void* dst, size_t bytes, hipStream_t s) {
  if (bytes == 0) return hipSuccess;
  const size_t n = bytes / 4;
  hipLaunchKernelGGL(fill_zero<uint32_t>, dim3(blocks(n)), dim3(kBlock), 0, s, (uint32_t*)dst, n);
  return hipGetLastError();
}

hipError_t phz_io_copy(void* dst, const void* src, size_t bytes, hipStream_t s) {
  if (bytes == 0) return hipSuccess;
  const size_t n = bytes / 4;
  hipLaunchKernelGGL(copy_words, dim3(blocks(n)), dim3(kBlock), 0, s, (uint32_t*)dst, (const uint32_t*)src, n);
  return hipGetLastError();
}

// The device address of the current device's scratch array, its size and the
// device's ordinal, looked up once per device (with that device current) and
// kept.
hipError_t phz_io_scratch(void** ptr, size_t* bytes, int* device) {
  int dev = -1;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return e;
  if (dev < 0 || dev >= kMaxDevices) return hipErrorInvalidDevice;
  std::lock_guard<std::mutex> lk(g_scratch_mu);
  if (!g_scratch_ptr[dev]) {
    void* p = nullptr;
    e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess) return e;
    if (!p) return hipErrorInvalidSymbol;
    g_scratch_ptr[dev] = p;
  }
  *ptr = g_scratch_ptr[dev];
  *bytes = kScratchBytes;
  *device = dev;
  return hipSuccess;
}

hipError_t phz_io_seed(uint64_t* rng, uint64_t seed, int nworld, hipStream_t s) {
  if (nworld <= 0) return hipSuccess;
  hipLaunchKernelGGL(seed_worlds, dim3(blocks(nworld)), dim3(kBlock), 0, s, rng, seed, nworld);
  return hipGetLastError();
}

}  // extern "C"
