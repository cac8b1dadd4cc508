// Truncated distance field of an occupancy grid: for every voxel of a
// dx x dy x dz grid (x fastest: index x + y*dx + z*dx*dy) the squared
// Euclidean distance, in voxel units, to the nearest occupied voxel, capped
// at trunc2.  The reference computes the same quantity by brute force over
// every occupied voxel (kernel.cu:9-31: a 30^3 grid, cap 900, called from
// key_point.h:287-308 on a key point's occupied octree voxels and read at
// matching.h:169-188).  Here the squared distance transform is separable:
// three 1-D passes, each d'(a) = min_t (a - t)^2 + d(t) along one axis.  Every
// value below 2^24 is an integer held exactly in FP32 (larger ones only lose
// low bits and can never undercut a smaller exact value), so capped results
// equal the brute force bit for bit.  Grid dimensions are arbitrary; occupied
// coordinates outside the grid are ignored.  The points variant maps a point
// to floor((p - origin) * (1 / resolution)) in FP32.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstring>
#include <mutex>
#include <vector>

#include "../../include/rtr.h"
#include "engine.hpp"

namespace rtr {

constexpr float kTdfInf = 1.0e30f;  // far above any squared grid distance

__global__ void k_tdf_fill(float* g, size_t n) {
  for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x)
    g[i] = kTdfInf;
}

__global__ void k_tdf_mark(const int32_t* occ, size_t n_occ, int dx, int dy, int dz, float* g) {
  for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n_occ; i += (size_t)gridDim.x * blockDim.x) {
    const int x = occ[3 * i], y = occ[3 * i + 1], z = occ[3 * i + 2];
    if (x < 0 || y < 0 || z < 0 || x >= dx || y >= dy || z >= dz) continue;
    g[x + (size_t)dx * ((size_t)y + (size_t)dy * z)] = 0.f;
  }
}

// Points -> occupied voxels: floor((p - origin) / res) inside the grid.
__global__ void k_tdf_mark_points(const float* xyz, size_t n, float ox, float oy, float oz, float inv_res, int dx,
                                  int dy, int dz, float* g) {
  for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x) {
    const float fx = (xyz[3 * i] - ox) * inv_res, fy = (xyz[3 * i + 1] - oy) * inv_res,
                fz = (xyz[3 * i + 2] - oz) * inv_res;
    if (!(fx >= 0.f && fy >= 0.f && fz >= 0.f && fx < (float)dx && fy < (float)dy && fz < (float)dz)) continue;
    const int x = min((int)fx, dx - 1), y = min((int)fy, dy - 1), z = min((int)fz, dz - 1);
    g[x + (size_t)dx * ((size_t)y + (size_t)dy * z)] = 0.f;
  }
}

// One pass along axis A (0 = x, 1 = y, 2 = z): out(a) = min(cap, min_t
// (a - t)^2 + in(t)) over the line through the voxel.  The offsets go outward
// and stop at the first r with r^2 >= the best so far: no farther term can be
// smaller (its rounded sum is at least r^2), so the result is that of the whole
// line, bit for bit.  Capping every pass, not the last alone, changes nothing
// either (a term with in >= cap is >= cap) and bounds the offsets by sqrt(cap)
// where a line holds nothing.
//
// A lane takes R neighbouring voxels of its line, so that a value read serves
// them all, with U offsets to each side in flight.  Lanes run along x in the y
// and z passes, and every load is then one contiguous segment per wave.
//
// Large fields (R = 4, U = 4) are bound by their loads and addresses, most of
// all where nothing stops the offsets (a large cap, few occupied voxels): with
// one voxel a lane such passes took longer than all terms of the line from LDS
// had.  250 x 250 x 125, the three passes: one occupied voxel and cap 10^9, from
// LDS 1057 us, one voxel a lane 1641, now 851; cap 900, 1058, 369, 176; 300k
// occupied, cap 900, 1058, 155, 93.  Small fields leave the chip idle and are a
// chain of load latencies: R = 1 for more lanes, and more offsets at once.
// 30^3, five launches: from LDS 15.0-17.1 us, U = 4 17.3-20.3, U = 16 15.0-16.9;
// 50^3 27, 24 (U = 4), 23 (U = 8), 29 (R = 4); 64^3, cap 10^9: 37, 33, 35 (U = 8),
// 32 (R = 4).
template <int A, int R, int U>
__global__ __launch_bounds__(256) void k_tdf_pass(const float* in, float* out, uint32_t n_runs, int dx, int dy, int dz,
                                                  float cap) {
  const int len = A == 0 ? dx : (A == 1 ? dy : dz);
  const ptrdiff_t stride = A == 0 ? 1 : (A == 1 ? dx : (ptrdiff_t)dx * dy);
  const uint32_t per_line = (uint32_t)(len + R - 1) / R;
  for (uint32_t i = blockIdx.x * 256u + threadIdx.x; i < n_runs; i += gridDim.x * 256u) {
    // the run's first voxel: runs along x, y or z in place of voxels
    int pos;
    size_t at;
    if (A == 0) {
      const uint32_t line = i / per_line;
      pos = R * (int)(i - line * per_line);
      at = (size_t)line * dx + pos;
    } else {
      const uint32_t q = i / (uint32_t)dx, x = i - q * (uint32_t)dx;
      if (A == 1) {
        const uint32_t z = q / per_line;
        pos = R * (int)(q - z * per_line);
        at = x + (size_t)dx * ((size_t)z * dy + pos);
      } else {
        const uint32_t g = q / (uint32_t)dy;
        pos = R * (int)g;
        at = x + (size_t)dx * ((q - g * (uint32_t)dy) + (size_t)pos * dy);
      }
    }
    const int m = min(R, len - pos);  // voxels of the run: fewer at the line's end
    const float* const p = in + at;
    const float* const e = p + (m - 1) * stride;
    float v[R], best[R];
#pragma unroll
    for (int k = 0; k < R; ++k) v[k] = p[min(k, m - 1) * stride];
#pragma unroll
    for (int k = 0; k < R; ++k) {
      best[k] = fminf(v[k], cap);
#pragma unroll
      for (int j = 0; j < R; ++j)
        if (j != k) best[k] = fminf(best[k], (float)((k - j) * (k - j)) + v[j]);
    }
    // (an offset past the line's end, here and below, repeats the end voxel's
    // value at a distance no shorter than its own: never below the term it
    // stands for)
    const int lo = pos, hi = len - pos - m, both = min(lo, hi), far = max(lo, hi);
    const float *l = p - stride, *h = e + stride;
    auto largest = [&] {
      float x = best[0];
#pragma unroll
      for (int k = 1; k < R; ++k) x = fmaxf(x, best[k]);
      return x;
    };
    float lim = largest();
    for (int r = 1; r <= far && (float)r * (float)r < lim; r += U, l -= U * stride, h += U * stride) {
      float a[U], b[U];
      if (r + U - 1 <= both) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
          a[u] = l[-u * stride];
          b[u] = h[u * stride];
        }
      } else {
#pragma unroll
        for (int u = 0; u < U; ++u) {
          a[u] = p[-min(r + u, lo) * stride];
          b[u] = e[min(r + u, hi) * stride];
        }
      }
      float d[U + R - 1];
#pragma unroll
      for (int j = 0; j < U + R - 1; ++j) d[j] = (float)(r + j) * (float)(r + j);
#pragma unroll
      for (int u = 0; u < U; ++u)
#pragma unroll
        for (int k = 0; k < R; ++k) best[k] = fminf(best[k], fminf(d[u + k] + a[u], d[u + R - 1 - k] + b[u]));
      lim = largest();
    }
#pragma unroll
    for (int k = 0; k < R; ++k)
      if (k < m) out[at + k * stride] = best[k];
  }
}

// The three passes over n = dx dy dz <= 2^31 voxels, from a through b back to
// a, and into out.
template <int R, int U>
static void tdf_passes_of(float* a, float* b, float* out, const int dims[3], float cap, hipStream_t s) {
  const dim3 t(256);
  auto runs = [&](int axis) {
    return (uint32_t)((size_t)dims[0] * dims[1] * dims[2] / dims[axis] * ((dims[axis] + R - 1) / R));
  };
  auto grid = [](uint32_t n) { return dim3(std::min((n + 255u) / 256u, 1u << 20)); };
  hipLaunchKernelGGL((k_tdf_pass<0, R, U>), grid(runs(0)), t, 0, s, a, b, runs(0), dims[0], dims[1], dims[2], cap);
  hipLaunchKernelGGL((k_tdf_pass<1, R, U>), grid(runs(1)), t, 0, s, b, a, runs(1), dims[0], dims[1], dims[2], cap);
  hipLaunchKernelGGL((k_tdf_pass<2, R, U>), grid(runs(2)), t, 0, s, a, out, runs(2), dims[0], dims[1], dims[2], cap);
}

static void tdf_passes(float* a, float* b, float* out, const int dims[3], float cap, hipStream_t s) {
  const size_t n = (size_t)dims[0] * dims[1] * dims[2];
  if (n <= (size_t)1 << 16)
    tdf_passes_of<1, 16>(a, b, out, dims, cap, s);
  else if (n <= (size_t)1 << 17)
    tdf_passes_of<1, 8>(a, b, out, dims, cap, s);
  else
    tdf_passes_of<4, 4>(a, b, out, dims, cap, s);
}

// Fills, marks, transforms and reads back; mem holds two fields and the input.
static int tdf_enqueue(float* mem, const int dims[3], float trunc2, float* out, const int32_t* occ, size_t n_occ,
                       const float* xyz, size_t n_pts, size_t stride, const float origin[3], float res) {
  const int dx = dims[0], dy = dims[1], dz = dims[2];
  const size_t n = (size_t)dx * dy * dz;
  float* const a = mem;
  float* const b = mem + n;
  float* const src = mem + 2 * n;
  hipStream_t s = nullptr;
  hipLaunchKernelGGL(k_tdf_fill, dim3((unsigned)std::min<size_t>(1024, (n + 255) / 256)), dim3(256), 0, s, a, n);
  if (occ && n_occ) {
    RTR_HIP(hipMemcpy(src, occ, n_occ * 12, hipMemcpyHostToDevice));
    hipLaunchKernelGGL(k_tdf_mark, dim3(256), dim3(256), 0, s, reinterpret_cast<int32_t*>(src), n_occ, dx, dy, dz, a);
  } else if (xyz && n_pts) {
    std::vector<float> packed;
    const float* from = xyz;
    if (stride != 12) {
      packed.resize(3 * n_pts);
      const char* base = reinterpret_cast<const char*>(xyz);
      for (size_t i = 0; i < n_pts; ++i) memcpy(&packed[3 * i], base + i * stride, 12);
      from = packed.data();
    }
    RTR_HIP(hipMemcpy(src, from, n_pts * 12, hipMemcpyHostToDevice));
    hipLaunchKernelGGL(k_tdf_mark_points, dim3(256), dim3(256), 0, s, src, n_pts, origin[0], origin[1], origin[2],
                       1.0f / res, dx, dy, dz, a);
  }
  tdf_passes(a, b, b, dims, trunc2, s);
  RTR_HIP(hipGetLastError());
  RTR_HIP(hipMemcpy(out, b, n * 4, hipMemcpyDeviceToHost));
  return RTR_OK;
}

static int tdf_run(int device, const int dims[3], float trunc2, float* out, const int32_t* occ, size_t n_occ,
                   const float* xyz, size_t n_pts, size_t stride, const float origin[3], float res) {
  RTR_HIP(hipSetDevice(device));
  const size_t n = (size_t)dims[0] * dims[1] * dims[2];
  // one allocation: the two fields, then the input
  const size_t src_bytes = occ ? n_occ * 12 : n_pts * 12;
  DevBuf mem;
  RTR_TRY(mem.ensure(2 * n * 4 + src_bytes));
  const int rc = tdf_enqueue(mem.as<float>(), dims, trunc2, out, occ, n_occ, xyz, n_pts, stride, origin, res);
  mem.release();
  return rc;
}

// ---------------------------------------------------------------------------
// Allocation-free variant (rtr_tdf_noalloc): the caller's device buffers hold
// the occupied voxels and the field; the intermediate grid of the separable
// passes is this file-scope device array, one per GPU, held until the process
// ends.  Host code never passes `scratch` itself to a kernel: its device
// address, per device, comes from hipGetSymbolAddress on the first call on
// that device.
// ---------------------------------------------------------------------------
constexpr size_t kTdfScratchMax = (size_t)1 << 21;  // floats: 8 MiB, grids of up to 2^21 voxels (128^3)
__device__ __align__(256) float scratch[kTdfScratchMax];

constexpr int kMaxDevices = 64;
static float* g_scratch_dev[kMaxDevices] = {nullptr};
static std::mutex g_scratch_mu;

static int scratch_of(int device, float** out) {
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (!g_scratch_dev[device]) {
    void* p = nullptr;
    RTR_HIP(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
    if (!p) {
      set_error("hipGetSymbolAddress returned no address for the TDF scratch array");
      return RTR_ERR_DEVICE;
    }
    g_scratch_dev[device] = static_cast<float*>(p);
  }
  *out = g_scratch_dev[device];
  return RTR_OK;
}

static bool tdf_dims_ok(const int dims[3]) {
  if (!dims) return false;
  size_t n = 1;
  for (int k = 0; k < 3; ++k) {
    if (dims[k] < 1 || dims[k] > 4096) return false;
    n *= (size_t)dims[k];
  }
  return n <= ((size_t)1 << 31);
}

}  // namespace rtr

extern "C" {

int rtr_tdf(int device, const int32_t* occ, size_t n_occ, const int dims[3], float trunc2, float* out) {
  using namespace rtr;
  if (!out || (n_occ && !occ) || !tdf_dims_ok(dims) || !(trunc2 > 0.f)) {
    set_error("rtr_tdf: invalid arguments");
    return RTR_ERR_INVALID_ARG;
  }
  try {
    return tdf_run(device, dims, trunc2, out, occ, n_occ, nullptr, 0, 12, nullptr, 1.f);
  } catch (...) {
    set_error("host allocation failed");
    return RTR_ERR_CAPACITY;
  }
}

int rtr_tdf_noalloc(int device, const int32_t* occ_dev, size_t n_occ, const int dims[3], float trunc2, float* out_dev,
                    void* stream) {
  using namespace rtr;
  if (!out_dev || (n_occ && !occ_dev) || !tdf_dims_ok(dims) || !(trunc2 > 0.f)) {
    set_error("rtr_tdf_noalloc: invalid arguments");
    return RTR_ERR_INVALID_ARG;
  }
  const size_t n = (size_t)dims[0] * dims[1] * dims[2];
  if (n > kTdfScratchMax) {
    set_error("rtr_tdf_noalloc: a %d x %d x %d grid has %zu voxels, above the allocation-free limit of %zu",
              dims[0], dims[1], dims[2], n, kTdfScratchMax);
    return RTR_ERR_CAPACITY;
  }
  int n_dev = 0;
  RTR_HIP(hipGetDeviceCount(&n_dev));
  if (device < 0 || device >= n_dev || device >= kMaxDevices) {
    set_error("rtr_tdf_noalloc: device %d not available", device);
    return RTR_ERR_DEVICE;
  }
  RTR_HIP(hipSetDevice(device));
  float* g = nullptr;
  RTR_TRY(scratch_of(device, &g));
  hipStream_t s = static_cast<hipStream_t>(stream);
  const int dx = dims[0], dy = dims[1], dz = dims[2];
  // every scratch voxel is written by the fill before it is read: nothing
  // left by an earlier call on this device is used
  // (the passes go from the caller's field to the scratch and back, so that
  // the last one reads the scratch and writes the caller's)
  hipLaunchKernelGGL(k_tdf_fill, dim3(1024), dim3(256), 0, s, g, n);
  if (n_occ) hipLaunchKernelGGL(k_tdf_mark, dim3(256), dim3(256), 0, s, occ_dev, n_occ, dx, dy, dz, g);
  tdf_passes(g, out_dev, out_dev, dims, trunc2, s);
  RTR_HIP(hipGetLastError());
  return RTR_OK;
}

int rtr_tdf_points(int device, const float* xyz, size_t n, size_t stride_bytes, const float origin[3],
                   float resolution, const int dims[3], float trunc2, float* out) {
  using namespace rtr;
  if (!out || (n && !xyz) || !origin || !(resolution > 0.f) || !tdf_dims_ok(dims) || !(trunc2 > 0.f)) {
    set_error("rtr_tdf_points: invalid arguments");
    return RTR_ERR_INVALID_ARG;
  }
  if (stride_bytes == 0) stride_bytes = 12;
  if (stride_bytes < 12) {
    set_error("rtr_tdf_points: stride below 12 bytes");
    return RTR_ERR_INVALID_ARG;
  }
  try {
    return tdf_run(device, dims, trunc2, out, nullptr, 0, xyz, n, stride_bytes, origin, resolution);
  } catch (...) {
    set_error("host allocation failed");
    return RTR_ERR_CAPACITY;
  }
}

}  // extern "C"
