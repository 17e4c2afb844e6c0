// Traversal order of a large ray array, for the persistent batched variants and
// for callers that ask svo_cast for it (set_cast_order_threshold); by default
// svo_cast streams such arrays, which needs no sort. Rays whose origins lie
// close together and whose directions share an octant walk the same nodes
// and bricks, so they are traversed side by side: each ray gets the key
// (Morton code of its origin on a 64^3 grid over the tree) * 8 + (direction
// octant), a stable radix sort of the keys gives the order, and the cast
// kernel's lane i traverses ray order[i] and writes that ray's own outputs.
// (A 64^3 grid orders as well as finer ones and keeps the key to 21 bits:
// three radix passes.)
// Every ray's result is computed alone, so the order changes no result; it
// changes the cache reuse and the spread of trip counts within a wave
// (incoherent rays into 512^3 and 2048^3 trees: 1.43-1.50x faster, sort
// excluded). The scratch arrays come from the stream-ordered allocator and
// go back to it on the same stream.
#include <hip/hip_runtime.h>

#include <hipcub/hipcub.hpp>

#include <algorithm>
#include <mutex>
#include <string>
#include <vector>

#include "device.hpp"
#include "launch.hpp"

namespace svo {

namespace {

constexpr uint32_t kGrid = 64;      // cells per axis
constexpr int kKeyBits = 18 + 3;    // 3 x 6 Morton bits + 3 octant bits

// Spreads the low 6 bits of v to every third bit (bit b to bit 3b).
__device__ inline uint32_t spread3(uint32_t v) {
  v &= 0x3Fu;
  v = (v | (v << 8)) & 0x0000F00Fu;
  v = (v | (v << 4)) & 0x000C30C3u;
  v = (v | (v << 2)) & 0x00249249u;
  return v;
}

// Grid cell (0..kGrid-1) of coordinate c, with cells_per_unit = kGrid / tree
// size; NaN and values outside the tree clamp to the edge cells.
__device__ inline uint32_t grid_cell(float c, float cells_per_unit) {
  const float g = c * cells_per_unit;
  return g >= static_cast<float>(kGrid - 1) ? kGrid - 1 : (g > 0.0f ? static_cast<uint32_t>(g) : 0u);
}

__global__ __launch_bounds__(256) void ray_keys_kernel(const float* __restrict__ rays, uint32_t n,
                                                       float cells_per_unit,
                                                       uint32_t* __restrict__ keys,
                                                       uint32_t* __restrict__ index) {
  const uint32_t i = blockIdx.x * 256u + threadIdx.x;
  if (i >= n) return;
  const float* r = rays + 6ull * i;
  const uint32_t m = spread3(grid_cell(r[0], cells_per_unit)) |
                     (spread3(grid_cell(r[1], cells_per_unit)) << 1) |
                     (spread3(grid_cell(r[2], cells_per_unit)) << 2);
  const uint32_t oct = static_cast<uint32_t>(__builtin_signbit(r[3]) != 0) |
                       (static_cast<uint32_t>(__builtin_signbit(r[4]) != 0) << 1) |
                       (static_cast<uint32_t>(__builtin_signbit(r[5]) != 0) << 2);
  keys[i] = (m << 3) | oct;
  index[i] = i;
}

int hip_fail(hipError_t e, const char* what, std::string* err) {
  *err = std::string(what) + ": " + hipGetErrorString(e);
  return e == hipErrorOutOfMemory ? SVO_OUT_OF_DEVICE_MEMORY : SVO_HIP_ERROR;
}

}  // namespace

int order_rays(const float* rays, uint32_t n, float tree_size, uint32_t** order, void* stream,
               std::string* err) {
  *order = nullptr;
  if (n > 0x7FFFFFFFu) return SVO_OK;  // the sort counts items in an int: left unordered
  hipStream_t s = static_cast<hipStream_t>(stream);
  {
    // the device's default pool keeps what the sort frees (by default it
    // returns it to the system at each synchronization, and every call would
    // allocate anew)
    static std::mutex mu;
    static std::vector<int> tuned;
    int dev = 0;
    if (hipGetDevice(&dev) == hipSuccess) {
      std::lock_guard<std::mutex> g(mu);
      if (std::find(tuned.begin(), tuned.end(), dev) == tuned.end()) {
        hipMemPool_t pool = nullptr;
        if (hipDeviceGetDefaultMemPool(&pool, dev) == hipSuccess) {
          uint64_t keep = UINT64_MAX;
          (void)hipMemPoolSetAttribute(pool, hipMemPoolAttrReleaseThreshold, &keep);
        }
        tuned.push_back(dev);
      }
    }
  }
  const size_t bytes = static_cast<size_t>(n) * sizeof(uint32_t);
  void* buf[4] = {nullptr, nullptr, nullptr, nullptr};  // keys in/out, index in/out
  hipError_t e = hipSuccess;
  for (int i = 0; i < 4 && e == hipSuccess; ++i) e = hipMallocAsync(&buf[i], bytes, s);
  size_t temp_bytes = 0;
  void* temp = nullptr;
  if (e == hipSuccess)
    e = hipcub::DeviceRadixSort::SortPairs(
        nullptr, temp_bytes, static_cast<const uint32_t*>(buf[0]), static_cast<uint32_t*>(buf[1]),
        static_cast<const uint32_t*>(buf[2]), static_cast<uint32_t*>(buf[3]), n, 0, kKeyBits, s);
  if (e == hipSuccess) e = hipMallocAsync(&temp, temp_bytes ? temp_bytes : 1, s);
  if (e == hipSuccess) {
    const uint32_t grid = static_cast<uint32_t>((static_cast<uint64_t>(n) + 255u) / 256u);
    e = launch(ray_keys_kernel, dim3(grid), dim3(256), s, rays, n,
               static_cast<float>(kGrid) / tree_size, static_cast<uint32_t*>(buf[0]),
               static_cast<uint32_t*>(buf[2]));
  }
  if (e == hipSuccess)
    e = hipcub::DeviceRadixSort::SortPairs(
        temp, temp_bytes, static_cast<const uint32_t*>(buf[0]), static_cast<uint32_t*>(buf[1]),
        static_cast<const uint32_t*>(buf[2]), static_cast<uint32_t*>(buf[3]), n, 0, kKeyBits, s);
  // everything but the order goes back to the pool once the stream has run
  // the sort
  for (int i = 0; i < 3; ++i)
    if (buf[i]) (void)hipFreeAsync(buf[i], s);
  if (temp) (void)hipFreeAsync(temp, s);
  if (e != hipSuccess) {
    if (buf[3]) (void)hipFreeAsync(buf[3], s);
    // (without memory the caller goes on unordered: not an error of the thread's)
    if (e == hipErrorOutOfMemory) (void)hipGetLastError();
    return hip_fail(e, "ray ordering", err);
  }
  *order = static_cast<uint32_t*>(buf[3]);
  return SVO_OK;
}

}  // namespace svo
