// Voxel-hash map: merges transformed clouds into a scene map.
//
// The reference "merges" by transforming a cloud, saving it as a PCD and
// overlaying files in a viewer (RealTimeRobot.cpp:104-114).  Here every
// point is transformed on the device (PCL transformPointCloud order), keyed
// by floor(p * inv_voxel) per axis (the truncation convention of
// key_point.h:143-160 / matching.h:181-184, floored for negative
// coordinates), and accumulated into an open-addressing hash table in HBM:
// per voxel a 64-bit key, the FP32 sum of (p - voxel corner) and a count.
// Offsets from the corner keep the FP32 sums small, so the centroid keeps
// full float precision however many frames land in the voxel.
//
// Integration kernel: each workgroup takes a contiguous run of tiles of 512
// consecutive points (a few image rows of a depth frame), stages each tile
// in LDS with coalesced loads, and merges the points voxel by voxel in an LDS
// hash table that lives across the run's tiles (neighbouring pixels, and
// neighbouring rows, share voxels); the table is flushed into the global one
// when it holds more than a quarter of its slots ahead of the next tile (so
// LDS probes stay short), and at the end of the run.  The global table then
// sees one insert and one set of atomics per distinct voxel of each flush,
// not per point.  Global probes are bounded (the table holds at most half its
// slots).  Many frames (each with its own transform) integrate in one
// launch.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cfloat>
#include <cmath>
#include <cstring>
#include <vector>

#include "../../include/rtr.h"
#include "engine.hpp"
#include "geom.hpp"
#include "wave.hpp"

namespace rtr {

constexpr uint64_t kEmpty = ~0ull;
constexpr int kBias = 1 << 20;

struct MapDev {
  unsigned long long* keys;  // capacity slots, kEmpty when free
  float4* acc;               // (sum dx, sum dy, sum dz, count bits)
  uint32_t* list;            // the occupied slots, in the order they were taken
  uint32_t* counters;        // [0] occupied slots, [1] dropped points, [2] overflow, [4..9] key box (lo, hi per axis)
  uint64_t mask;             // capacity - 1 (power of two)
  uint32_t max_voxels;
  float h, inv_h;
};

__device__ __forceinline__ uint64_t mix64(uint64_t k) {
  // SplitMix64 finaliser (Steele, Lea, Flood 2014)
  k ^= k >> 30;
  k *= 0xbf58476d1ce4e5b9ull;
  k ^= k >> 27;
  k *= 0x94d049bb133111ebull;
  k ^= k >> 31;
  return k;
}

RTR_HD bool voxel_key(float x, float y, float z, float inv_h, uint64_t* key, int* k3) {
  const float v[3] = {x * inv_h, y * inv_h, z * inv_h};
  uint64_t kk = 0;
  for (int a = 0; a < 3; ++a) {
    if (!(v[a] - v[a] == 0.f)) return false;  // inf or NaN
    const float f = floorf(v[a]);
    if (f < -(float)kBias || f >= (float)kBias) return false;
    const int k = (int)f;
    k3[a] = k;
    kk |= (uint64_t)(uint32_t)(k + kBias) << (21 * a);
  }
  *key = kk;
  return true;
}

constexpr int kMapBlock = 256;
constexpr int kMapTile = 512;    // points per workgroup tile
constexpr int kMapSlots = 2048;  // the run's LDS hash table
constexpr int kMapFlushAt = kMapSlots / 2 - kMapTile;  // flush before a tile when more keys are held
constexpr int kMapMinRun = 4;    // tiles per workgroup at least (the merging spans the run)
constexpr int kMaxProbe = 128;   // global probe bound (the table is at most half full)
static_assert(kMapFlushAt + kMapTile < kMapSlots, "every tile key must find a free LDS slot");

// One frame of an integration launch: packed xyz on the device, its point
// count, its first tile in the launch and the float rows of its transform.
struct MapFrame {
  const float* xyz;
  uint32_t n;
  uint32_t tile0;
  float m[12];
  int has_T;
  int pad_;
};

// One merged voxel of a tile into the global table: (sum of corner offsets,
// count).  False when the probe bound is reached (table too full).
__device__ __forceinline__ bool global_add(const MapDev& m, uint64_t key, float sx, float sy, float sz, uint32_t cnt) {
  uint64_t slot = mix64(key) & m.mask;
  for (int probe = 0; probe < kMaxProbe; ++probe) {
    // a stale empty read only costs a CAS; a key once written never changes
    unsigned long long cur = m.keys[slot];
    if (cur == kEmpty) {
      cur = atomicCAS(&m.keys[slot], (unsigned long long)kEmpty, (unsigned long long)key);
      if (cur == kEmpty) {
        const uint32_t occ = atomicAdd(&m.counters[0], 1u);
        m.list[occ] = (uint32_t)slot;  // occ counts slots taken: it stays below their number
        if (occ >= m.max_voxels) atomicOr(&m.counters[2], 1u);
        cur = key;
      }
    }
    if (cur == key) {
      float* a = reinterpret_cast<float*>(&m.acc[slot]);
      atomicAdd(a + 0, sx);
      atomicAdd(a + 1, sy);
      atomicAdd(a + 2, sz);
      atomicAdd(reinterpret_cast<uint32_t*>(a + 3), cnt);
      return true;
    }
    slot = (slot + 1) & m.mask;
  }
  return false;
}

// The run's merged voxels into the global table; the LDS table is left
// empty.  Every thread of the workgroup calls it.
__device__ __forceinline__ void map_flush(const MapDev& m, unsigned long long* s_key, float4* s_acc,
                                          uint32_t& dropped, uint32_t& overflow) {
  for (int i = threadIdx.x; i < kMapSlots; i += kMapBlock) {
    const unsigned long long k = s_key[i];
    if (k == kEmpty) continue;
    const float4 a = s_acc[i];
    const uint32_t c = __float_as_uint(a.w);
    if (!global_add(m, k, a.x, a.y, a.z, c)) {
      dropped += c;
      overflow = 1;
    }
    s_key[i] = kEmpty;
    s_acc[i] = make_float4(0.f, 0.f, 0.f, 0.f);
  }
}

__global__ __launch_bounds__(kMapBlock) void k_map_integrate(MapDev m, const MapFrame* frames, int n_frames,
                                                             uint32_t n_tiles, uint32_t run) {
  __shared__ float s_xyz[3 * kMapTile];
  __shared__ unsigned long long s_key[kMapSlots];
  __shared__ float4 s_acc[kMapSlots];
  __shared__ int s_frame;
  __shared__ uint32_t s_used;
  const int tid = threadIdx.x;
  uint32_t dropped = 0, overflow = 0;
  for (int i = tid; i < kMapSlots; i += kMapBlock) {
    s_key[i] = kEmpty;
    s_acc[i] = make_float4(0.f, 0.f, 0.f, 0.f);
  }
  if (tid == 0) s_used = 0u;
  const uint32_t t0 = blockIdx.x * run;
  const uint32_t t1 = min(t0 + run, n_tiles);
  for (uint32_t tile = t0; tile < t1; ++tile) {
    __syncthreads();  // the previous tile's inserts (and s_used) are complete
    if (s_used > (uint32_t)kMapFlushAt) {
      map_flush(m, s_key, s_acc, dropped, overflow);
      __syncthreads();
      if (tid == 0) s_used = 0u;
    }
    if (tid == 0) {
      // the frame of this tile: the last one whose first tile is <= tile
      int lo = 0, hi = n_frames - 1;
      while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (frames[mid].tile0 <= tile)
          lo = mid;
        else
          hi = mid - 1;
      }
      s_frame = lo;
    }
    __syncthreads();
    const MapFrame* f = frames + s_frame;
    const uint32_t base = (tile - f->tile0) * (uint32_t)kMapTile;
    const uint32_t cnt = min((uint32_t)kMapTile, f->n - base);
    // coalesced staging: consecutive lanes load consecutive floats
    const float* src = f->xyz + 3 * (size_t)base;
    for (uint32_t j = tid; j < 3 * cnt; j += kMapBlock) s_xyz[j] = src[j];
    const int has_T = f->has_T;
    float mt[12];
#pragma unroll
    for (int k = 0; k < 12; ++k) mt[k] = f->m[k];
    __syncthreads();
    for (uint32_t p = tid; p < cnt; p += kMapBlock) {
      float px = s_xyz[3 * p], py = s_xyz[3 * p + 1], pz = s_xyz[3 * p + 2];
      if (has_T) apply_f32(mt, px, py, pz, px, py, pz);
      uint64_t key;
      int k3[3];
      if (!voxel_key(px, py, pz, m.inv_h, &key, k3)) {
        ++dropped;
        continue;
      }
      const float dx = px - (float)k3[0] * m.h;
      const float dy = py - (float)k3[1] * m.h;
      const float dz = pz - (float)k3[2] * m.h;
      // the table holds at most kMapFlushAt + kMapTile < kMapSlots keys: a
      // free or matching slot always exists within kMapSlots probes
      uint32_t sl = (uint32_t)(mix64(key) & (uint64_t)(kMapSlots - 1));
      for (int probe = 0; probe < kMapSlots; ++probe) {
        unsigned long long cur = s_key[sl];
        if (cur == kEmpty) {
          cur = atomicCAS(&s_key[sl], (unsigned long long)kEmpty, (unsigned long long)key);
          if (cur == kEmpty) {
            atomicAdd(&s_used, 1u);
            cur = key;
          }
        }
        if (cur == key) {
          atomicAdd(&s_acc[sl].x, dx);
          atomicAdd(&s_acc[sl].y, dy);
          atomicAdd(&s_acc[sl].z, dz);
          atomicAdd(reinterpret_cast<uint32_t*>(&s_acc[sl].w), 1u);
          break;
        }
        sl = (sl + 1) & (uint32_t)(kMapSlots - 1);
      }
    }
  }
  __syncthreads();
  map_flush(m, s_key, s_acc, dropped, overflow);
  if (dropped) atomicAdd(&m.counters[1], dropped);
  if (overflow) atomicOr(&m.counters[2], 1u);
}

// ---------------------------------------------------------------------------
// Reading the map out, in key order
//
// The list of occupied slots, filled as voxels are inserted, spares the scan of
// the whole table (134 MB for a capacity of 8M voxels) and its one counter that
// every occupied slot incremented.  Keys are unique, so a voxel's place in key
// order is the number of occupied voxels before it: one bit per cell of the
// keys' bounding box, the bits counted by an exclusive scan of their words,
// and a voxel's rank is its word's count plus the bits below its own.  Eight
// small kernels, about 35 us together for 40k-100k voxels of a room: the
// table's scan alone took 606 us (167 us for a frame's downsample), and the
// sort on the host that followed it 1-6 ms.  A fused and read map of 8 frames
// 4.43 -> 1.67 ms, a downsampled 640 x 480 frame 1.99 -> 0.63 ms; what is left
// is the upload (0.6 and 0.1 ms), the integration's device-scope atomics (0.2
// and 0.09 ms) and copying the results out.
// ---------------------------------------------------------------------------
__device__ __forceinline__ uint32_t key_axis(uint64_t k, int a) { return (uint32_t)(k >> (21 * a)) & 0x1fffffu; }

constexpr int kBoxThreads = 1024;  // few workgroups: each ends with six atomics on the same words

__global__ __launch_bounds__(kBoxThreads) void k_map_box(MapDev m) {
  __shared__ int part[6][kBoxThreads / 64];
  const uint32_t n = m.counters[0];
  int lo[3] = {0x7fffffff, 0x7fffffff, 0x7fffffff}, hi[3] = {-1, -1, -1};
  for (uint32_t i = blockIdx.x * kBoxThreads + threadIdx.x; i < n; i += gridDim.x * kBoxThreads) {
    const uint64_t k = m.keys[m.list[i]];
    for (int a = 0; a < 3; ++a) {
      lo[a] = min(lo[a], (int)key_axis(k, a));
      hi[a] = max(hi[a], (int)key_axis(k, a));
    }
  }
  for (int a = 0; a < 3; ++a) {
    const int l = wave_min_i32(lo[a]), h = wave_max_i32(hi[a]);
    if ((threadIdx.x & 63) == 0) {
      part[a][threadIdx.x >> 6] = l;
      part[3 + a][threadIdx.x >> 6] = h;
    }
  }
  __syncthreads();
  if (threadIdx.x < 6) {
    const int a = threadIdx.x;
    int v = part[a][0];
    for (int w = 1; w < kBoxThreads / 64; ++w) v = a < 3 ? min(v, part[a][w]) : max(v, part[a][w]);
    if (a < 3 && v != 0x7fffffff) atomicMin(&m.counters[4 + a], (uint32_t)v);
    if (a >= 3 && v >= 0) atomicMax(&m.counters[4 + a], (uint32_t)v);
  }
}

__global__ void k_map_box_init(MapDev m) {
  if (threadIdx.x < 6) m.counters[4 + threadIdx.x] = threadIdx.x < 3 ? 0xffffffffu : 0u;
}

// The key box of a read-out: cells (x fastest) of [lo, lo + dim).
struct KeyBox {
  uint32_t lo[3], dim[3];
};

__device__ __forceinline__ uint32_t cell_of_key(const KeyBox& b, uint64_t k) {
  return (key_axis(k, 0) - b.lo[0]) + b.dim[0] * ((key_axis(k, 1) - b.lo[1]) + b.dim[1] * (key_axis(k, 2) - b.lo[2]));
}

__global__ __launch_bounds__(256) void k_map_bits(MapDev m, uint32_t n, KeyBox box, uint32_t* bits) {
  for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
    const uint32_t c = cell_of_key(box, m.keys[m.list[i]]);
    atomicOr(&bits[c >> 5], 1u << (c & 31u));
  }
}

__global__ __launch_bounds__(256) void k_map_popc(const uint32_t* bits, uint32_t words, uint32_t* cnt) {
  for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < words; i += gridDim.x * blockDim.x)
    cnt[i] = (uint32_t)__popc(bits[i]);
}

// A voxel's outputs: its key, its count and its sum of points, or centroid.
// The sums are kept as offsets from the voxel corner; the corner's share is
// added in FP64.
struct MapOut {
  int64_t* keys;      // (each nullable)
  float* xyz;
  uint32_t* counts;
  int as_centroids;
};

__host__ __device__ __forceinline__ void voxel_out(uint64_t k, float sx, float sy, float sz, uint32_t c, float h,
                                                   const MapOut& o, size_t at) {
  if (o.keys) o.keys[at] = (int64_t)k;
  if (o.counts) o.counts[at] = c;
  if (!o.xyz) return;
  const float s[3] = {sx, sy, sz};
  for (int a = 0; a < 3; ++a) {
    const int kk = (int)((k >> (21 * a)) & 0x1fffffull) - kBias;
    const float corner = (float)kk * h;
    const double v = (double)corner * c + (double)s[a];
    o.xyz[3 * at + a] = o.as_centroids ? (float)(v / (double)c) : (float)v;
  }
}

__global__ __launch_bounds__(256) void k_map_emit(MapDev m, uint32_t n, KeyBox box, const uint32_t* bits,
                                                  const uint32_t* first, MapOut out) {
  for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
    const uint32_t slot = m.list[i];
    const uint64_t k = m.keys[slot];
    const float4 a = m.acc[slot];
    const uint32_t c = cell_of_key(box, k), below = bits[c >> 5] & ((1u << (c & 31u)) - 1u);
    voxel_out(k, a.x, a.y, a.z, __float_as_uint(a.w), m.h, out, first[c >> 5] + (uint32_t)__popc(below));
  }
}

// The occupied voxels in the list's order (for the boxes too sparse for a bit
// per cell, which the host sorts)
__global__ __launch_bounds__(256) void k_map_gather(MapDev m, uint32_t n, unsigned long long* okeys, float4* oacc) {
  for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
    const uint32_t slot = m.list[i];
    okeys[i] = m.keys[slot];
    oacc[i] = m.acc[slot];
  }
}

// Empties the table: the n slots on the list, or every slot, and zeroes the
// counters (which no thread reads here).
__global__ __launch_bounds__(256) void k_map_clear(MapDev m, uint32_t n, int all) {
  const uint64_t stride = (uint64_t)gridDim.x * blockDim.x, i0 = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i0 < 4) m.counters[i0] = 0u;
  if (!all) {
    for (uint64_t i = i0; i < n; i += stride) {
      const uint32_t s = m.list[i];
      m.keys[s] = kEmpty;
      m.acc[s] = make_float4(0.f, 0.f, 0.f, 0.f);
    }
    return;
  }
  for (uint64_t s = i0; s <= m.mask; s += stride) {
    m.keys[s] = kEmpty;
    m.acc[s] = make_float4(0.f, 0.f, 0.f, 0.f);
  }
}

// Up to this many voxels are read in the list's order and sorted on the host: one
// launch in place of eight (100 voxels of a 0.5 m box 141 -> 59 us, 2000 139 ->
// 69; 4000 take 187 us this way and 141 by the bit map).
constexpr uint32_t kFewVoxels = 2048;

// Cells of the key box: at most this many per voxel, or in all, for the bit
// map.  64 per voxel is 2 words of bits and 2 of counts to pass over per voxel,
// far below a comparison sort's work; 2^24 cells (2 MB of bits, about 10 us)
// always pay; 2^28 bounds the workspace to 64 MB.
constexpr uint64_t kBoxCellsPerVoxel = 64, kBoxCellsFew = 1ull << 24, kBoxCellsMost = 1ull << 28;

struct VoxelMap {
  int device;
  hipStream_t stream = nullptr;
  hipEvent_t ev[2] = {nullptr, nullptr};
  bool profiling = false;
  float last_ms = 0.f;
  int cu_count = 0;
  DevBuf table, in, T;            // table: acc, keys, list, counters
  DevBuf bits, first, scan, out;  // read-out
  MapDev dev;
  size_t capacity = 0;
  static constexpr uint32_t kUnknown = 0xffffffffu;
  uint32_t used = kUnknown;       // occupied slots, as the last call left them
  uint64_t dropped_total = 0;

  int init(int dev_id, float voxel, size_t cap) {
    device = dev_id;
    int n = 0;
    RTR_HIP(hipGetDeviceCount(&n));
    if (dev_id < 0 || dev_id >= n) {
      set_error("device %d not available", dev_id);
      return RTR_ERR_DEVICE;
    }
    RTR_HIP(hipSetDevice(device));
    RTR_HIP(hipStreamCreateWithFlags(&stream, hipStreamNonBlocking));
    RTR_HIP(hipEventCreate(&ev[0]));
    RTR_HIP(hipEventCreate(&ev[1]));
    RTR_HIP(hipDeviceGetAttribute(&cu_count, hipDeviceAttributeMultiprocessorCount, device));
    uint64_t slots = 1024;
    while (slots < 2 * (uint64_t)cap) slots <<= 1;
    capacity = cap;
    // one allocation: each costs its own call and, on release, its own wait
    RTR_TRY(table.ensure(slots * (16 + 8 + 4) + 64));
    dev.acc = table.as<float4>();
    dev.keys = reinterpret_cast<unsigned long long*>(dev.acc + slots);
    dev.list = reinterpret_cast<uint32_t*>(dev.keys + slots);
    dev.counters = dev.list + slots;
    dev.mask = slots - 1;
    dev.max_voxels = (uint32_t)cap;
    dev.h = voxel;
    dev.inv_h = (float)(1.0 / (double)voxel);
    return clear();
  }
  // By the list when it is short against the table (two lines at random places
  // for each entry, against 24 bytes a slot in order: 16M slots 66 us, 40k listed
  // voxels 13 us).
  int clear() {
    RTR_HIP(hipSetDevice(device));
    const bool all = used == kUnknown || (uint64_t)used * 8 > dev.mask;
    const unsigned blocks = all ? 1024u : std::max(1u, std::min(1024u, (used + 255u) / 256u));
    hipLaunchKernelGGL(k_map_clear, dim3(blocks), dim3(256), 0, stream, dev, all ? 0u : used, all ? 1 : 0);
    used = kUnknown;
    RTR_HIP(hipGetLastError());
    RTR_HIP(hipStreamSynchronize(stream));
    used = 0;
    dropped_total = 0;
    return RTR_OK;
  }
  ~VoxelMap() {
    (void)hipSetDevice(device);
    if (stream) (void)hipStreamSynchronize(stream);
    DevBuf* b[] = {&table, &in, &T, &bits, &first, &scan, &out};
    for (DevBuf* x : b) x->release();
    for (hipEvent_t e : ev)
      if (e) (void)hipEventDestroy(e);
    if (stream) (void)hipStreamDestroy(stream);
  }
  int read_counters(uint32_t c[4]) {
    RTR_HIP(hipMemcpyAsync(c, dev.counters, 16, hipMemcpyDeviceToHost, stream));
    RTR_HIP(hipStreamSynchronize(stream));
    return RTR_OK;
  }
  // nf frames in one launch: frame f's points (packed, or with a byte
  // stride) moved by T[16 f ..] (column-major; T or its entries nullable
  // means identity)
  int integrate_frames(int nf, const float* const* xyz, const size_t* n, size_t stride, const double* Tcm) {
    RTR_HIP(hipSetDevice(device));
    if (stride == 0) stride = 12;
    size_t total = 0, tiles = 0;
    for (int f = 0; f < nf; ++f) {
      total += n[f];
      tiles += (n[f] + kMapTile - 1) / kMapTile;
    }
    if (total == 0) return RTR_OK;
    if (total >= (1ull << 32) || tiles >= (1ull << 32)) {
      set_error("too many points in one call");
      return RTR_ERR_CAPACITY;
    }
    RTR_TRY(in.ensure(total * 12));
    RTR_TRY(T.ensure(sizeof(MapFrame) * (size_t)nf));
    std::vector<MapFrame> fr(nf);
    std::vector<float> packed;
    size_t off = 0;
    uint32_t tile0 = 0;
    for (int f = 0; f < nf; ++f) {
      MapFrame& d = fr[f];
      memset(&d, 0, sizeof(d));
      d.xyz = in.as<float>() + 3 * off;
      d.n = (uint32_t)n[f];
      d.tile0 = tile0;
      d.has_T = Tcm ? 1 : 0;
      if (Tcm) tf_rows_f32(Tcm + 16 * (size_t)f, d.m);
      if (n[f]) {
        const float* src = xyz[f];
        if (stride != 12) {
          packed.resize(n[f] * 3);
          const char* b = reinterpret_cast<const char*>(xyz[f]);
          for (size_t i = 0; i < n[f]; ++i) memcpy(packed.data() + 3 * i, b + i * stride, 12);
          src = packed.data();
        }
        // synchronous for pageable memory: the staging buffer is reused
        RTR_HIP(hipMemcpyAsync(in.as<float>() + 3 * off, src, n[f] * 12, hipMemcpyHostToDevice, stream));
        if (stride != 12) RTR_HIP(hipStreamSynchronize(stream));
      }
      off += n[f];
      tile0 += (uint32_t)((n[f] + kMapTile - 1) / kMapTile);
    }
    RTR_HIP(hipMemcpyAsync(T.p, fr.data(), sizeof(MapFrame) * (size_t)nf, hipMemcpyHostToDevice, stream));
    // contiguous runs of at least kMapMinRun tiles, at most 8 workgroups per CU
    size_t blocks = std::min<size_t>((tiles + kMapMinRun - 1) / kMapMinRun, (size_t)std::max(cu_count, 1) * 8);
    const uint32_t run = (uint32_t)((tiles + blocks - 1) / blocks);
    blocks = (tiles + run - 1) / run;
    if (profiling) RTR_HIP(hipEventRecord(ev[0], stream));
    used = kUnknown;
    hipLaunchKernelGGL(k_map_integrate, dim3((unsigned)blocks), dim3(kMapBlock), 0, stream, dev, T.as<MapFrame>(), nf,
                       (uint32_t)tiles, run);
    RTR_HIP(hipGetLastError());
    if (profiling) RTR_HIP(hipEventRecord(ev[1], stream));
    uint32_t after[4];
    RTR_TRY(read_counters(after));
    used = after[0];
    if (profiling) RTR_HIP(hipEventElapsedTime(&last_ms, ev[0], ev[1]));
    dropped_total = after[1];
    if (after[2]) {
      set_error("voxel map capacity exceeded (%zu voxels)", capacity);
      return RTR_ERR_CAPACITY;
    }
    return RTR_OK;
  }
  int integrate(const float* xyz, size_t n, size_t stride, const double* Tcm) {
    return integrate_frames(1, &xyz, &n, stride, Tcm);
  }
  int size(size_t* n) {
    uint32_t c[4];
    int rc = read_counters(c);
    if (rc) return rc;
    *n = c[0];
    return RTR_OK;
  }
  // Occupied voxels in key order (z, then y, then x) into host arrays of cap
  // entries (each nullable); *n_out their number, also when it exceeds cap.
  int extract(const MapOut& host, size_t cap, size_t* n_out, const char* what) {
    RTR_HIP(hipSetDevice(device));
    uint32_t c[10];
    if (used == kUnknown) {
      RTR_TRY(read_counters(c));
      used = c[0];
    }
    const uint32_t nv = used;
    *n_out = nv;
    if (nv > cap) {
      set_error("%s capacity %zu < %u voxels", what, cap, nv);
      return RTR_ERR_CAPACITY;
    }
    if (nv == 0) return RTR_OK;
    const unsigned blocks = (unsigned)std::min<size_t>(2048, ((size_t)nv + 255) / 256);
    if (nv <= kFewVoxels) return extract_sorted_on_host(host, nv, blocks);
    hipLaunchKernelGGL(k_map_box_init, dim3(1), dim3(64), 0, stream, dev);
    hipLaunchKernelGGL(k_map_box, dim3(32), dim3(kBoxThreads), 0, stream, dev);
    RTR_HIP(hipGetLastError());
    RTR_HIP(hipMemcpyAsync(c, dev.counters, sizeof(c), hipMemcpyDeviceToHost, stream));
    RTR_HIP(hipStreamSynchronize(stream));
    KeyBox box;
    uint64_t cells = 1;
    for (int a = 0; a < 3; ++a) {
      box.lo[a] = c[4 + a];
      box.dim[a] = c[7 + a] - c[4 + a] + 1;
      cells *= box.dim[a];  // at most 2^63
    }
    if (cells > kBoxCellsMost || (cells > kBoxCellsFew && cells / kBoxCellsPerVoxel > nv))
      return extract_sorted_on_host(host, nv, blocks);
    const uint32_t words = (uint32_t)((cells + 31) / 32);
    RTR_TRY(bits.ensure((size_t)words * 4));
    RTR_TRY(first.ensure((size_t)words * 4));
    RTR_TRY(scan.ensure(scan_tmp_words(words) * 4));
    RTR_TRY(out.ensure((size_t)nv * 24));
    launch_fill_u32(bits.as<uint32_t>(), 0u, words, stream);
    hipLaunchKernelGGL(k_map_bits, dim3(blocks), dim3(256), 0, stream, dev, nv, box, bits.as<uint32_t>());
    hipLaunchKernelGGL(k_map_popc, dim3(std::min(2048u, (words + 255) / 256)), dim3(256), 0, stream,
                       bits.as<uint32_t>(), words, first.as<uint32_t>());
    launch_exclusive_scan(first.as<uint32_t>(), first.as<uint32_t>(), words, scan.as<uint32_t>(), stream);
    MapOut o = host;
    o.keys = host.keys ? out.as<int64_t>() : nullptr;
    o.xyz = host.xyz ? reinterpret_cast<float*>(out.as<int64_t>() + nv) : nullptr;
    o.counts = host.counts ? reinterpret_cast<uint32_t*>(out.as<int64_t>() + nv) + 3 * (size_t)nv : nullptr;
    hipLaunchKernelGGL(k_map_emit, dim3(blocks), dim3(256), 0, stream, dev, nv, box, bits.as<uint32_t>(),
                       first.as<uint32_t>(), o);
    RTR_HIP(hipGetLastError());
    if (host.keys) RTR_HIP(hipMemcpyAsync(host.keys, o.keys, (size_t)nv * 8, hipMemcpyDeviceToHost, stream));
    if (host.xyz) RTR_HIP(hipMemcpyAsync(host.xyz, o.xyz, (size_t)nv * 12, hipMemcpyDeviceToHost, stream));
    if (host.counts) RTR_HIP(hipMemcpyAsync(host.counts, o.counts, (size_t)nv * 4, hipMemcpyDeviceToHost, stream));
    RTR_HIP(hipStreamSynchronize(stream));
    return RTR_OK;
  }

  // The same where a bit per cell of the key box would be too many: the voxels
  // in any order, sorted on the host.
  int extract_sorted_on_host(const MapOut& host, uint32_t nv, unsigned blocks) {
    RTR_TRY(out.ensure((size_t)nv * 24));
    float4* dacc = out.as<float4>();
    unsigned long long* dkeys = reinterpret_cast<unsigned long long*>(dacc + nv);
    hipLaunchKernelGGL(k_map_gather, dim3(blocks), dim3(256), 0, stream, dev, nv, dkeys, dacc);
    RTR_HIP(hipGetLastError());
    std::vector<uint64_t> hk(nv);
    std::vector<float4> ha(nv);
    RTR_HIP(hipMemcpyAsync(hk.data(), dkeys, (size_t)nv * 8, hipMemcpyDeviceToHost, stream));
    RTR_HIP(hipMemcpyAsync(ha.data(), dacc, (size_t)nv * 16, hipMemcpyDeviceToHost, stream));
    RTR_HIP(hipStreamSynchronize(stream));
    std::vector<uint32_t> order(nv);
    for (uint32_t i = 0; i < nv; ++i) order[i] = i;
    std::sort(order.begin(), order.end(), [&](uint32_t a, uint32_t b) { return hk[a] < hk[b]; });
    for (uint32_t i = 0; i < nv; ++i) {
      const float4& a = ha[order[i]];
      uint32_t c;
      memcpy(&c, &a.w, 4);
      voxel_out(hk[order[i]], a.x, a.y, a.z, c, dev.h, host, i);
    }
    return RTR_OK;
  }
};

}  // namespace rtr

using rtr::set_error;
using rtr::VoxelMap;

struct rtr_map {
  VoxelMap m;
};

extern "C" {

int rtr_map_create(rtr_map** out, int device, float voxel_size, size_t capacity) {
  try {
    if (!out || !(voxel_size > 0) || capacity == 0 || capacity > (1ull << 31)) {
      set_error("invalid voxel map arguments (voxel %g, capacity %zu)", voxel_size, capacity);
      return RTR_ERR_INVALID_ARG;
    }
    *out = nullptr;
    rtr_map* m = new rtr_map();
    int rc = m->m.init(device, voxel_size, capacity);
    if (rc) {
      delete m;
      return rc;
    }
    *out = m;
    return RTR_OK;
  } catch (...) {
    set_error("host allocation failed");
    return RTR_ERR_CAPACITY;
  }
}

int rtr_map_destroy(rtr_map* m) {
  delete m;
  return RTR_OK;
}

int rtr_map_clear(rtr_map* m) {
  if (!m) return RTR_ERR_INVALID_ARG;
  return m->m.clear();
}

int rtr_map_integrate(rtr_map* m, const float* xyz, size_t n, size_t stride, const double T[16]) {
  if (!m || (n && !xyz) || (stride != 0 && stride < 12)) return RTR_ERR_INVALID_ARG;
  try {
    return m->m.integrate(xyz, n, stride, T);
  } catch (...) {
    set_error("host allocation failed");
    return RTR_ERR_CAPACITY;
  }
}

int rtr_map_integrate_frames(rtr_map* m, int n_frames, const float* const* xyz, const size_t* n, size_t stride,
                             const double* T) {
  if (!m || n_frames < 1 || !xyz || !n || (stride != 0 && stride < 12)) return RTR_ERR_INVALID_ARG;
  for (int f = 0; f < n_frames; ++f)
    if (n[f] && !xyz[f]) return RTR_ERR_INVALID_ARG;
  try {
    return m->m.integrate_frames(n_frames, xyz, n, stride, T);
  } catch (...) {
    set_error("host allocation failed");
    return RTR_ERR_CAPACITY;
  }
}

int rtr_map_set_profiling(rtr_map* m, int on) {
  if (!m) return RTR_ERR_INVALID_ARG;
  m->m.profiling = on != 0;
  return RTR_OK;
}

int rtr_map_last_ms(rtr_map* m, float* ms) {
  if (!m || !ms) return RTR_ERR_INVALID_ARG;
  *ms = m->m.last_ms;
  return RTR_OK;
}

int rtr_map_size(rtr_map* m, size_t* n) {
  if (!m || !n) return RTR_ERR_INVALID_ARG;
  return m->m.size(n);
}

int rtr_map_dropped(rtr_map* m, uint64_t* n) {
  if (!m || !n) return RTR_ERR_INVALID_ARG;
  *n = m->m.dropped_total;
  return RTR_OK;
}

int rtr_map_extract(rtr_map* m, int64_t* keys, float* xyz, uint32_t* counts, size_t cap,
                    size_t* n_out, int as_centroids) {
  if (!m || !n_out) return RTR_ERR_INVALID_ARG;
  try {
    const rtr::MapOut o{keys, xyz, counts, as_centroids};
    return m->m.extract(o, cap, n_out, "extract");
  } catch (...) {
    set_error("host allocation failed");
    return RTR_ERR_CAPACITY;
  }
}

int rtr_voxel_downsample(int device, const float* xyz, size_t n, size_t stride, float leaf,
                         float* out, size_t cap, size_t* n_out) {
  if ((n && !xyz) || !(leaf > 0) || !n_out) return RTR_ERR_INVALID_ARG;
  try {
    VoxelMap vm;
    int rc = vm.init(device, leaf, n > 0 ? n : 1);
    if (rc) return rc;
    rc = vm.integrate(xyz, n, stride, nullptr);
    if (rc) return rc;
    // PCL VoxelGrid order (linear index over the ijk bounding box, x fastest)
    // is key order
    return vm.extract(rtr::MapOut{nullptr, out, nullptr, 1}, cap, n_out, "downsample");
  } catch (...) {
    set_error("host allocation failed");
    return RTR_ERR_CAPACITY;
  }
}

}  // extern "C"
