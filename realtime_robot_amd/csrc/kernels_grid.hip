// Grid construction on the device: per-target uniform grids (cell-sorted
// float4 points + cell start offsets) and per-source spatial (Morton) sort,
// batched over all clouds of an engine.  Counting sort: count -> flat
// exclusive scan over every cloud's cell range -> scatter.
#include <hip/hip_runtime.h>

#include "engine_dev.hpp"
#include "geom.hpp"
#include "wave.hpp"

namespace rtr {

// ---------------------------------------------------------------------------
// fill and scan
// ---------------------------------------------------------------------------

__global__ void k_fill_u32(uint32_t* p, uint32_t v, size_t n) {
  size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  size_t stride = (size_t)gridDim.x * blockDim.x;
  for (; i < n; i += stride) p[i] = v;
}

void launch_fill_u32(uint32_t* p, uint32_t v, size_t n, hipStream_t s) {
  if (n == 0) return;
  size_t blocks = (n + kBlock - 1) / kBlock;
  if (blocks > 8192) blocks = 8192;
  hipLaunchKernelGGL(k_fill_u32, dim3((unsigned)blocks), dim3(kBlock), 0, s, p, v, n);
}

constexpr int kScanPer = 8;                    // elements per thread
constexpr int kScanTile = kBlock * kScanPer;   // 2048 per block

size_t scan_tmp_words(uint32_t n) { return (n + kScanTile - 1) / kScanTile + 1; }

__device__ __forceinline__ uint32_t wave_incl_scan(uint32_t v) {
  const int lane = threadIdx.x & 63;
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    uint32_t t = __shfl_up(v, off, 64);
    if (lane >= off) v += t;
  }
  return v;
}

// exclusive block scan of one value per thread; returns prefix, total in *tot
__device__ __forceinline__ uint32_t block_excl_scan(uint32_t v, uint32_t* tot) {
  __shared__ uint32_t wsum[kWaves];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  uint32_t inc = wave_incl_scan(v);
  if (lane == 63) wsum[w] = inc;
  __syncthreads();
  uint32_t base = 0, all = 0;
  for (int i = 0; i < kWaves; ++i) {
    if (i < w) base += wsum[i];
    all += wsum[i];
  }
  __syncthreads();
  *tot = all;
  return base + inc - v;
}

__global__ void k_scan_reduce(const uint32_t* in, uint32_t n, uint32_t* tile_sums) {
  const uint32_t base = blockIdx.x * kScanTile + threadIdx.x * kScanPer;
  uint32_t s = 0;
#pragma unroll
  for (int k = 0; k < kScanPer; ++k)
    if (base + k < n) s += in[base + k];
  uint32_t tot;
  block_excl_scan(s, &tot);
  if (threadIdx.x == 0) tile_sums[blockIdx.x] = tot;
}

__global__ void k_scan_tiles(uint32_t* tile_sums, uint32_t ntiles) {
  uint32_t carry = 0;
  for (uint32_t b = 0; b < ntiles; b += kBlock) {
    uint32_t i = b + threadIdx.x;
    uint32_t v = i < ntiles ? tile_sums[i] : 0;
    uint32_t tot;
    uint32_t ex = block_excl_scan(v, &tot);
    if (i < ntiles) tile_sums[i] = carry + ex;
    carry += tot;
  }
  if (threadIdx.x == 0) tile_sums[ntiles] = carry;
}

__global__ void k_scan_apply(const uint32_t* in, uint32_t* out, uint32_t n,
                             const uint32_t* tile_sums) {
  const uint32_t base = blockIdx.x * kScanTile + threadIdx.x * kScanPer;
  uint32_t v[kScanPer];
  uint32_t s = 0;
#pragma unroll
  for (int k = 0; k < kScanPer; ++k) {
    v[k] = (base + k < n) ? in[base + k] : 0;
    s += v[k];
  }
  uint32_t tot;
  uint32_t ex = block_excl_scan(s, &tot) + tile_sums[blockIdx.x];
#pragma unroll
  for (int k = 0; k < kScanPer; ++k) {
    if (base + k < n) out[base + k] = ex;
    ex += v[k];
  }
}

void launch_exclusive_scan(const uint32_t* in, uint32_t* out, uint32_t n, uint32_t* tmp,
                           hipStream_t s) {
  if (n == 0) return;
  uint32_t ntiles = (n + kScanTile - 1) / kScanTile;
  hipLaunchKernelGGL(k_scan_reduce, dim3(ntiles), dim3(kBlock), 0, s, in, n, tmp);
  hipLaunchKernelGGL(k_scan_tiles, dim3(1), dim3(kBlock), 0, s, tmp, ntiles);
  hipLaunchKernelGGL(k_scan_apply, dim3(ntiles), dim3(kBlock), 0, s, in, out, n, tmp);
}

// ---------------------------------------------------------------------------
// block reductions
// ---------------------------------------------------------------------------

// (wave reductions: DPP row operations, wave.hpp)


// Bounding boxes of many clouds at once: each cloud is split over many
// workgroups, whose wave minima / maxima (as order-preserving integer keys)
// and finite-point counts meet in 8 words per cloud through atomics.  Min and
// max do not depend on the order they are taken in, so the box is the same
// as a serial pass.
__device__ __forceinline__ uint32_t ord_key(float f) {
  const uint32_t u = __float_as_uint(f);
  return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}
__device__ __forceinline__ float ord_val(uint32_t k) {
  return __uint_as_float((k & 0x80000000u) ? (k & 0x7fffffffu) : ~k);
}

// words per cloud: lo key x3, hi key x3, finite count, unused
__global__ void k_bbox_init(uint32_t* bb, uint32_t n_words) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n_words) bb[i] = (i & 7u) < 3u ? 0xffffffffu : 0u;
}

template <bool TGT>
__global__ void k_cloud_bbox(DevEngine e) {
  const uint32_t c = blockIdx.y;
  const float* xyz = TGT ? e.tgt_raw + 3 * (size_t)e.tgts[c].raw_off : e.src_raw + 3 * (size_t)e.srcs[c].off;
  const uint32_t n = TGT ? e.tgts[c].n : e.srcs[c].n;
  uint32_t* bb = e.bbox_tmp + 8 * (size_t)(TGT ? c : e.n_tgt + c);
  float l[3] = {3.0e38f, 3.0e38f, 3.0e38f}, h[3] = {-3.0e38f, -3.0e38f, -3.0e38f};
  uint32_t cnt = 0;
  for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
    const float x = xyz[3 * (size_t)i], y = xyz[3 * (size_t)i + 1], z = xyz[3 * (size_t)i + 2];
    if (!(isfinite(x) && isfinite(y) && isfinite(z))) continue;
    l[0] = fminf(l[0], x);
    l[1] = fminf(l[1], y);
    l[2] = fminf(l[2], z);
    h[0] = fmaxf(h[0], x);
    h[1] = fmaxf(h[1], y);
    h[2] = fmaxf(h[2], z);
    ++cnt;
  }
  for (int a = 0; a < 3; ++a) {
    l[a] = wave_min_f32(l[a]);
    h[a] = wave_max_f32(h[a]);
  }
  cnt = wave_sum_u32(cnt);
  // the workgroup's waves combine in LDS first: one set of atomics per
  // workgroup instead of per wave (every workgroup of a cloud updates the
  // same seven words, so these atomics serialise)
  __shared__ float s_l[kBlock / 64][3], s_h[kBlock / 64][3];
  __shared__ uint32_t s_c[kBlock / 64];
  const int w = threadIdx.x >> 6;
  if ((threadIdx.x & 63) == 0) {
    for (int a = 0; a < 3; ++a) {
      s_l[w][a] = l[a];
      s_h[w][a] = h[a];
    }
    s_c[w] = cnt;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int v = 1; v < kBlock / 64; ++v) {
      for (int a = 0; a < 3; ++a) {
        l[a] = fminf(l[a], s_l[v][a]);
        h[a] = fmaxf(h[a], s_h[v][a]);
      }
      cnt += s_c[v];
    }
    if (cnt) {
      for (int a = 0; a < 3; ++a) {
        atomicMin(&bb[a], ord_key(l[a]));
        atomicMax(&bb[3 + a], ord_key(h[a]));
      }
      atomicAdd(&bb[6], cnt);
    }
  }
}

__device__ __forceinline__ void bbox_of(const uint32_t* bb, float* lo, float* hi, uint32_t* cnt) {
  *cnt = bb[6];
  for (int a = 0; a < 3; ++a) {
    lo[a] = *cnt ? ord_val(bb[a]) : 3.0e38f;
    hi[a] = *cnt ? ord_val(bb[3 + a]) : -3.0e38f;
  }
}

// ---------------------------------------------------------------------------
// target grids
// ---------------------------------------------------------------------------

// Choose the cell edge: the smallest h >= h_req (growing by 5%) whose grid
// over the bbox fits the cell budget.  dims use the same float expression as
// the cell assignment, so every point lands inside the grid.
__device__ void choose_grid(TargetDesc& t, const float* lo, const float* hi, uint32_t cnt) {
  t.n_valid = cnt;
  if (cnt == 0) {
    t.dx = t.dy = t.dz = 1;
    t.ox = t.oy = t.oz = 0.f;
    t.h = t.h_req > 0.f ? t.h_req : 1.f;
    t.inv_h = 1.0f / t.h;
    t.margin = 1e-3f * t.h;
    t.anchor[0] = t.anchor[1] = t.anchor[2] = 0.f;
    return;
  }
  const float ex = hi[0] - lo[0], ey = hi[1] - lo[1], ez = hi[2] - lo[2];
  float h = t.h_req > 0.f ? t.h_req : 1e-3f;
  const double vol = (double)ex * ey * ez;
  const double hb = cbrt(vol / (double)t.cell_budget);
  if ((float)hb > h) h = (float)hb;
  int dx = 1, dy = 1, dz = 1;
  float inv = 1.0f / h;
  bool fits = false;
  if (isfinite(ex) && isfinite(ey) && isfinite(ez)) {
    for (int it = 0; it < 400; ++it) {
      inv = 1.0f / h;
      const float fx = floorf((hi[0] - lo[0]) * inv), fy = floorf((hi[1] - lo[1]) * inv),
                  fz = floorf((hi[2] - lo[2]) * inv);
      if (fx < 1.0e7f && fy < 1.0e7f && fz < 1.0e7f) {
        dx = (int)fx + 1;
        dy = (int)fy + 1;
        dz = (int)fz + 1;
        if ((long long)dx * dy * dz <= (long long)t.cell_budget) {
          fits = true;
          break;
        }
      }
      h *= 1.05f;
    }
  }
  if (!fits) {
    // a single cell holds everything (cell_of clamps every index to 0): slow, exact
    dx = dy = dz = 1;
    h = fmaxf(fmaxf(ex, ey), ez);
    if (!(h > 0.f) || !isfinite(h)) h = 1.0f;
    inv = 1.0f / h;
  }
  t.dx = dx;
  t.dy = dy;
  t.dz = dz;
  t.ox = lo[0];
  t.oy = lo[1];
  t.oz = lo[2];
  t.h = h;
  t.inv_h = inv;
  float mag = fmaxf(fmaxf(fabsf(lo[0]), fabsf(hi[0])), fmaxf(fmaxf(fabsf(lo[1]), fabsf(hi[1])),
                                                             fmaxf(fabsf(lo[2]), fabsf(hi[2]))));
  t.margin = 1e-3f * h + 4e-6f * (mag + fmaxf(ex, fmaxf(ey, ez)));
  t.anchor[0] = lo[0] + 0.5f * ex;
  t.anchor[1] = lo[1] + 0.5f * ey;
  t.anchor[2] = lo[2] + 0.5f * ez;
}

// Distance-field parameters: a query whose cell is at Chebyshev distance >= R
// from every occupied cell is at least (R - 1) * h - margin from every target
// point; skip_ring is the smallest R for which that exceeds r_max.
__device__ void choose_dist_cap(TargetDesc& t, float r_max) {
  dist_caps(r_max, t.h, t.margin, &t.skip_ring, &t.dt_cap);
}

// one thread per target, after k_cloud_bbox<true>
__global__ void k_tgt_choose(DevEngine e) {
  const int j = blockIdx.x * blockDim.x + threadIdx.x;
  if (j >= e.n_tgt) return;
  TargetDesc& t = e.tgts[j];
  float lo[3], hi[3];
  uint32_t cnt;
  bbox_of(e.bbox_tmp + 8 * (size_t)j, lo, hi, &cnt);
  choose_grid(t, lo, hi, cnt);
  choose_dist_cap(t, e.r_max);
}

__device__ __forceinline__ bool cell_of(const TargetDesc& t, float x, float y, float z,
                                        uint32_t* c) {
  if (!(isfinite(x) && isfinite(y) && isfinite(z))) return false;
  int ix = clampi((int)floorf((x - t.ox) * t.inv_h), 0, t.dx - 1);
  int iy = clampi((int)floorf((y - t.oy) * t.inv_h), 0, t.dy - 1);
  int iz = clampi((int)floorf((z - t.oz) * t.inv_h), 0, t.dz - 1);
  *c = ((uint32_t)iz * t.dy + iy) * t.dx + ix;
  return true;
}

__global__ void k_tgt_count(DevEngine e) {
  const TargetDesc& t = e.tgts[blockIdx.y];
  const float* xyz = e.tgt_raw + 3 * (size_t)t.raw_off;
  for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < t.n; i += gridDim.x * blockDim.x) {
    uint32_t c;
    if (cell_of(t, xyz[3 * (size_t)i], xyz[3 * (size_t)i + 1], xyz[3 * (size_t)i + 2], &c)) {
      e.cell_id[t.raw_off + i] = c;
      e.cell_rank[t.raw_off + i] = atomicAdd(&e.cell_count[t.cell_off + c], 1u);
    } else {
      e.cell_id[t.raw_off + i] = 0xffffffffu;
    }
  }
}

__global__ void k_tgt_scatter(DevEngine e) {
  const TargetDesc& t = e.tgts[blockIdx.y];
  const float* xyz = e.tgt_raw + 3 * (size_t)t.raw_off;
  for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < t.n; i += gridDim.x * blockDim.x) {
    const uint32_t c = e.cell_id[t.raw_off + i];
    if (c == 0xffffffffu) continue;
    const uint32_t slot = t.cell_off + c;
    // the count pass handed every point its slot within the cell
    const uint32_t pos = e.cell_start[slot] + e.cell_rank[t.raw_off + i];
    union {
      int32_t i;
      float f;
    } w;
    w.i = (int32_t)i;
    e.tgt_sorted[pos] =
        make_float4(xyz[3 * (size_t)i], xyz[3 * (size_t)i + 1], xyz[3 * (size_t)i + 2], w.f);
    if (e.tgt_nrm_raw && e.tgt_nrm_sorted) {
      const float* nr = e.tgt_nrm_raw + 3 * ((size_t)t.raw_off + i);
      e.tgt_nrm_sorted[pos] = make_float4(nr[0], nr[1], nr[2], 0.f);
    }
  }
}

// Separable Chebyshev distance transform over each target's cells, capped at
// dt_cap + 1: pass x from the occupancy (cell_start differences), then y, then
// z, each a min over |d| <= cap of max(|d|, previous pass at offset d).  The
// offsets go outward by |d| and stop once |d| reaches the best value so far:
// no farther offset can give less than its |d|.
template <int AXIS>
__global__ void k_tgt_dist(DevEngine e, const uint8_t* src, uint8_t* dst) {
  const TargetDesc& t = e.tgts[blockIdx.y];
  const uint32_t ncell = (uint32_t)t.dx * t.dy * t.dz;
  const int K = t.dt_cap;
  const int len = AXIS == 0 ? t.dx : (AXIS == 1 ? t.dy : t.dz);
  const int stride = AXIS == 0 ? 1 : (AXIS == 1 ? t.dx : t.dx * t.dy);
  const uint32_t* cs = e.cell_start + t.cell_off;
  auto val = [&](uint32_t cc) -> int {
    if (AXIS == 0) return cs[cc + 1] > cs[cc] ? 0 : K + 1;
    return src[t.cell_off + cc];
  };
  for (uint32_t c = blockIdx.x * blockDim.x + threadIdx.x; c < ncell; c += gridDim.x * blockDim.x) {
    const int pos = AXIS == 0 ? (int)(c % t.dx) : (AXIS == 1 ? (int)((c / t.dx) % t.dy) : (int)(c / ((uint32_t)t.dx * t.dy)));
    int best = val(c);
    const int lo = min(K, pos), hi = min(K, len - 1 - pos);
    for (int a = 1; a < best && (a <= lo || a <= hi); ++a) {
      int v = K + 1;
      if (a <= lo) v = val(c - (uint32_t)(a * stride));
      if (a <= hi) {
        const int w = val(c + (uint32_t)(a * stride));
        v = w < v ? w : v;
      }
      v = v > a ? v : a;
      best = v < best ? v : best;
    }
    dst[t.cell_off + c] = (uint8_t)best;
  }
}

// workgroups per cloud of a bounding-box pass: about 16 points per thread
static unsigned bbox_blocks_for(int max_pts) {
  unsigned b = (unsigned)((max_pts + 16 * kBlock - 1) / (16 * kBlock));
  return b < 1 ? 1 : (b > 128 ? 128 : b);
}

static unsigned blocks_for(int max_pts) {
  unsigned b = (unsigned)((max_pts + kBlock - 1) / kBlock);
  if (b < 1) b = 1;
  if (b > 256) b = 256;
  return b;
}

void launch_target_grid(const DevEngine& e, int max_tgt_pts, int max_cells, hipStream_t s) {
  if (e.n_tgt == 0) return;
  launch_fill_u32(e.cell_count, 0u, e.n_cells_total, s);
  const uint32_t bw = 8u * (uint32_t)e.n_tgt;
  hipLaunchKernelGGL(k_bbox_init, dim3((bw + kBlock - 1) / kBlock), dim3(kBlock), 0, s, e.bbox_tmp, bw);
  dim3 g(blocks_for(max_tgt_pts), e.n_tgt);
  hipLaunchKernelGGL(k_cloud_bbox<true>, dim3(bbox_blocks_for(max_tgt_pts), e.n_tgt), dim3(kBlock), 0, s, e);
  hipLaunchKernelGGL(k_tgt_choose, dim3((e.n_tgt + 63) / 64), dim3(64), 0, s, e);
  hipLaunchKernelGGL(k_tgt_count, g, dim3(kBlock), 0, s, e);
  launch_exclusive_scan(e.cell_count, e.cell_start, e.n_cells_total, e.scan_tmp, s);
  hipLaunchKernelGGL(k_tgt_scatter, g, dim3(kBlock), 0, s, e);
  if (e.cell_dist) {
    dim3 gd(blocks_for(max_cells), e.n_tgt);
    hipLaunchKernelGGL(k_tgt_dist<0>, gd, dim3(kBlock), 0, s, e, (const uint8_t*)nullptr, e.cell_dist);
    hipLaunchKernelGGL(k_tgt_dist<1>, gd, dim3(kBlock), 0, s, e, (const uint8_t*)e.cell_dist, e.cell_dist_tmp);
    hipLaunchKernelGGL(k_tgt_dist<2>, gd, dim3(kBlock), 0, s, e, (const uint8_t*)e.cell_dist_tmp, e.cell_dist);
  }
}

// ---------------------------------------------------------------------------
// source spatial sort (Morton order of a coarse grid in the source frame)
// ---------------------------------------------------------------------------

__device__ __forceinline__ uint32_t spread3(uint32_t v) {
  // 5-bit value -> bits at positions 0, 3, 6, 9, 12
  uint32_t r = 0;
#pragma unroll
  for (int b = 0; b < 5; ++b) r |= ((v >> b) & 1u) << (3 * b);
  return r;
}

// one thread per source, after k_cloud_bbox<false>
__global__ void k_src_choose(DevEngine e) {
  const int j = blockIdx.x * blockDim.x + threadIdx.x;
  if (j >= e.n_src) return;
  SourceDesc& s = e.srcs[j];
  float lo[3], hi[3];
  uint32_t cnt;
  bbox_of(e.bbox_tmp + 8 * (size_t)(e.n_tgt + j), lo, hi, &cnt);
  {
    // bin_budget = P^3 with P a power of two <= 32 (chosen by the host)
    int P = 1;
    while (P * P * P < (int)s.bin_budget) P <<= 1;
    s.dx = s.dy = s.dz = P;
    float ext = cnt ? fmaxf(hi[0] - lo[0], fmaxf(hi[1] - lo[1], hi[2] - lo[2])) : 0.f;
    s.ox = cnt ? lo[0] : 0.f;
    s.oy = cnt ? lo[1] : 0.f;
    s.oz = cnt ? lo[2] : 0.f;
    s.inv_h = ext > 0.f ? (float)P / ext : 0.f;
  }
}

__device__ __forceinline__ uint32_t bin_of(const SourceDesc& s, float x, float y, float z) {
  const uint32_t last = s.bin_budget - 1;
  if (!(isfinite(x) && isfinite(y) && isfinite(z))) return last;
  const int P = s.dx;
  int ix = clampi((int)floorf((x - s.ox) * s.inv_h), 0, P - 1);
  int iy = clampi((int)floorf((y - s.oy) * s.inv_h), 0, P - 1);
  int iz = clampi((int)floorf((z - s.oz) * s.inv_h), 0, P - 1);
  uint32_t m = spread3(ix) | (spread3(iy) << 1) | (spread3(iz) << 2);
  return m > last ? last : m;
}

__global__ void k_src_count(DevEngine e) {
  const SourceDesc& s = e.srcs[blockIdx.y];
  const float* xyz = e.src_raw + 3 * (size_t)s.off;
  for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < s.n; i += gridDim.x * blockDim.x) {
    uint32_t b = bin_of(s, xyz[3 * (size_t)i], xyz[3 * (size_t)i + 1], xyz[3 * (size_t)i + 2]);
    e.bin_id[s.off + i] = b;
    e.bin_rank[s.off + i] = atomicAdd(&e.bin_count[s.bin_off + b], 1u);
  }
}

__device__ __forceinline__ uint32_t spread3_4(uint32_t v) {
  uint32_t r = 0;
#pragma unroll
  for (int b = 0; b < 4; ++b) r |= ((v >> b) & 1u) << (3 * b);
  return r;
}

// (Morton code of the point inside its bin at 16 sub-cells per axis, original
// index): ordered by it, the layout, and with it the summation order of the
// moments, is identical from run to run, and consecutive points stay compact
// below the bin size.
__device__ __forceinline__ uint64_t fine_key(const SourceDesc& sd, float x, float y, float z, uint32_t id) {
  uint32_t fine = 0xfffu;
  if (isfinite(x) && isfinite(y) && isfinite(z)) {
    const int P = sd.dx;
    const float f[3] = {(x - sd.ox) * sd.inv_h, (y - sd.oy) * sd.inv_h, (z - sd.oz) * sd.inv_h};
    uint32_t sub[3];
    for (int a = 0; a < 3; ++a) {
      const int c = clampi((int)floorf(f[a]), 0, P - 1);
      sub[a] = (uint32_t)clampi((int)floorf((f[a] - (float)c) * 16.0f), 0, 15);
    }
    fine = spread3_4(sub[0]) | (spread3_4(sub[1]) << 1) | (spread3_4(sub[2]) << 2);
  }
  return ((uint64_t)fine << 32) | id;
}

// The keys go to their bins in atomic order: the point's bin (at most 32^3, 15
// bits) above its key, so that the next pass finds the bin with it.
__global__ void k_src_scatter(DevEngine e) {
  const SourceDesc& s = e.srcs[blockIdx.y];
  const float* xyz = e.src_raw + 3 * (size_t)s.off;
  for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < s.n; i += gridDim.x * blockDim.x) {
    const uint32_t b = e.bin_id[s.off + i];
    // bin_start is global over all sources; every source point is placed, so
    // source s occupies exactly [s.off, s.off + s.n) of the sorted arrays
    const uint32_t pos = e.bin_start[s.bin_off + b] + e.bin_rank[s.off + i];
    e.src_key[pos] = ((uint64_t)b << 44) | fine_key(s, xyz[3 * (size_t)i], xyz[3 * (size_t)i + 1], xyz[3 * (size_t)i + 2], i);
  }
}

// Each point's rank in its bin, by counting the bin's smaller keys: bins hold
// tens of points whose keys lie together, so a point's loop runs in the L1 with
// several loads in flight, and every point of every cloud is a lane.  (One wave
// ordering 64 bins through LDS after the other ran at the latency of its
// loads, most of a small cloud in a few waves: 79 -> 8 us for 2k points, 455 ->
// 85 us for 256 sources of 3k to 8k.)  A bin of more than kBinCap points is ordered
// by the original index alone.
constexpr uint32_t kBinCap = 1024;

__global__ __launch_bounds__(kBlock) void k_src_order(DevEngine e) {
  const SourceDesc& s = e.srcs[blockIdx.y];
  const float* xyz = e.src_raw + 3 * (size_t)s.off;
  for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < s.n; i += gridDim.x * blockDim.x) {
    uint64_t key = e.src_key[s.off + i];
    const uint32_t slot = s.bin_off + (uint32_t)(key >> 44);
    const uint32_t lo = e.bin_start[slot], n = e.bin_count[slot];
    const uint32_t id = (uint32_t)key;
    const uint64_t mask = n > kBinCap ? 0xffffffffull : ~0ull;
    key &= mask;
    const uint64_t* k = e.src_key + lo;
    uint32_t r = 0, j = 0;
    for (; j + 8 <= n; j += 8) {
      uint64_t o[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) o[u] = k[j + u];
#pragma unroll
      for (int u = 0; u < 8; ++u) r += (o[u] & mask) < key ? 1u : 0u;
    }
    for (; j < n; ++j) r += (k[j] & mask) < key ? 1u : 0u;
    const uint32_t pos = lo + r;
    e.sx[pos] = xyz[3 * (size_t)id];
    e.sy[pos] = xyz[3 * (size_t)id + 1];
    e.sz[pos] = xyz[3 * (size_t)id + 2];
    e.perm[pos] = id;
  }
}

void launch_source_sort(const DevEngine& e, int max_src_pts, hipStream_t s) {
  if (e.n_src == 0) return;
  launch_fill_u32(e.bin_count, 0u, e.n_bins_total, s);
  const uint32_t bw = 8u * (uint32_t)e.n_src;
  hipLaunchKernelGGL(k_bbox_init, dim3((bw + kBlock - 1) / kBlock), dim3(kBlock), 0, s, e.bbox_tmp + 8 * (size_t)e.n_tgt,
                     bw);
  hipLaunchKernelGGL(k_cloud_bbox<false>, dim3(bbox_blocks_for(max_src_pts), e.n_src), dim3(kBlock), 0, s, e);
  hipLaunchKernelGGL(k_src_choose, dim3((e.n_src + 63) / 64), dim3(64), 0, s, e);
  dim3 g(blocks_for(max_src_pts), e.n_src);
  hipLaunchKernelGGL(k_src_count, g, dim3(kBlock), 0, s, e);
  launch_exclusive_scan(e.bin_count, e.bin_start, e.n_bins_total, e.scan_tmp, s);
  hipLaunchKernelGGL(k_src_scatter, g, dim3(kBlock), 0, s, e);
  hipLaunchKernelGGL(k_src_order, g, dim3(kBlock), 0, s, e);
}

}  // namespace rtr
