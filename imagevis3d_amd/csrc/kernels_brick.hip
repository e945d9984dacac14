// kernels_brick.hip -- HBM-streaming kernels of the UVF bricking / LOD path
// (RasterDataBlock::FlatDataToBrickedLOD + CombineAverage + SimpleMaxMin,
// UVFReader/DataSource.h:550-570; Histogram1D/2DDataBlock::Compute,
// UVFReader/DataSource.h:595-636).  Integer in, integer out: every result
// is bit-exact with the CPU twins in oracle/oracle.c.
//
// All of these are byte/integer streaming work bounded by HBM bandwidth:
// threads walk rows of x so each wavefront reads and writes contiguous
// runs, and reductions go through wave shuffles before one atomic per
// workgroup.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "kernels.hpp"

namespace tvk {
namespace {

constexpr int kThreads = 256;

// 2x2x2 reduction of the existing children of each parent voxel: integer
// mean floor(sum / count) (RasterDataBlock's CombineAverage rule), or with
// MEDIAN the lower median -- element (count-1)/2 of the sorted children
// (the UseMedian option of the TOC builder).
template <typename T, bool MEDIAN>
__global__ __launch_bounds__(kThreads) void downsample_kernel(const T* __restrict__ src, int64_t nx,
                                                              int64_t ny, int64_t nz,
                                                              T* __restrict__ dst, int64_t mx,
                                                              int64_t my, int64_t mz) {
  const int64_t x = (int64_t)blockIdx.x * kThreads + threadIdx.x;
  if (x >= mx) return;
  // rows of a level stay below 2^31 for every supported volume, so the
  // per-row index split uses 32-bit division.
  const uint32_t rows = (uint32_t)(my * mz), umy = (uint32_t)my;
  const int64_t x0 = 2 * x, x1 = 2 * x + 1 < nx ? 2 * x + 1 : -1;
  for (uint32_t row = blockIdx.y; row < rows; row += gridDim.y) {
    const int64_t y = row % umy, z = row / umy;
    const int64_t ys[2] = {2 * y, 2 * y + 1 < ny ? 2 * y + 1 : -1};
    const int64_t zs[2] = {2 * z, 2 * z + 1 < nz ? 2 * z + 1 : -1};
    uint32_t sum = 0, cnt = 0;
    uint32_t v[8];
#pragma unroll
    for (int dz = 0; dz < 2; ++dz) {
      if (zs[dz] < 0) continue;
#pragma unroll
      for (int dy = 0; dy < 2; ++dy) {
        if (ys[dy] < 0) continue;
        const T* r = src + (zs[dz] * ny + ys[dy]) * nx;
        if (MEDIAN) {
          v[cnt++] = r[x0];
          if (x1 >= 0) v[cnt++] = r[x1];
        } else {
          sum += r[x0];
          ++cnt;
          if (x1 >= 0) {
            sum += r[x1];
            ++cnt;
          }
        }
      }
    }
    uint32_t out;
    if (MEDIAN) {
      // insertion sort of the (at most 8) children
      for (uint32_t i = 1; i < cnt; ++i) {
        const uint32_t key = v[i];
        uint32_t j = i;
        while (j > 0 && v[j - 1] > key) {
          v[j] = v[j - 1];
          --j;
        }
        v[j] = key;
      }
      out = v[(cnt - 1) / 2];
    } else {
      out = sum / cnt;
    }
    dst[(z * my + y) * mx + x] = (T)out;
  }
}

// N consecutive voxels with one load; a volume row starts at any multiple of
// the voxel size, and unaligned global loads are legal on gfx950.
template <typename T, int N>
struct VoxelRun {
  typedef T vec __attribute__((ext_vector_type(N), aligned(sizeof(T))));
};
template <typename T, int N>
__device__ inline void load_run(const T* p, uint32_t (&out)[N]) {
  const auto v = *(const __attribute__((address_space(1))) typename VoxelRun<T, N>::vec*)p;
#pragma unroll
  for (int j = 0; j < N; ++j) out[j] = v[j];
}

__device__ inline uint32_t wave_min(uint32_t v) {
  for (int o = 32; o > 0; o >>= 1) v = min(v, (uint32_t)__shfl_xor((int)v, o, 64));
  return v;
}
__device__ inline uint32_t wave_max(uint32_t v) {
  for (int o = 32; o > 0; o >>= 1) v = max(v, (uint32_t)__shfl_xor((int)v, o, 64));
  return v;
}
__device__ inline unsigned long long wave_max64(unsigned long long v) {
  for (int o = 32; o > 0; o >>= 1) {
    unsigned long long w = __shfl_xor(v, o, 64);
    v = w > v ? w : v;
  }
  return v;
}

__device__ inline int64_t clamp64(int64_t v, int64_t lo, int64_t hi) {
  return v < lo ? lo : (v > hi ? hi : v);
}

// One row of a slot's blocks (all bx at by, bz) in the blocked slot layout:
// the 16 rows of x its blocks hold come in as contiguous runs, wait in LDS
// and leave in element order -- the row's blocks are contiguous in the slot
// -- 16 bytes a thread and step.  The slot's voxel (x, y, z) is src at (ox +
// x, oy + y, oz + z) clamped to the nx x ny x nz volume; blocks past the
// slot's edge repeat its last voxel along that axis.  lds: 16 rows of 4 (n +
// 1) voxels.  Folds the voxels' range into lo and hi.
template <typename T>
__device__ inline void slot_block_row(const T* __restrict__ src, int64_t nx, int64_t ny, int64_t nz, int64_t ox,
                                      int64_t oy, int64_t oz, int S, int by, int bz, T* __restrict__ slot, T* lds,
                                      uint32_t& lo, uint32_t& hi) {
  const int n = slot_blocks(S), segs = n + 1, stride = 4 * segs;
  const int row = (int)threadIdx.x >> 4;  // 16 rows, 16 threads each
  const int64_t y = clamp64(oy + min(by * 4 + (row & 3), S - 1), 0, ny - 1);
  const int64_t z = clamp64(oz + min(bz * 4 + (row >> 2), S - 1), 0, nz - 1);
  const T* __restrict__ line = src + (z * ny + y) * nx;
  typedef T vec4 __attribute__((ext_vector_type(4)));
  for (int seg = (int)threadIdx.x & 15; seg < segs; seg += 16) {
    const int x = 4 * seg;
    const int64_t gx = ox + x;
    uint32_t v[4];
    if (x + 3 < S && gx >= 0 && gx + 3 < nx) {
      load_run<T, 4>(line + gx, v);
    } else {
#pragma unroll
      for (int j = 0; j < 4; ++j) v[j] = line[clamp64(ox + min(x + j, S - 1), 0, nx - 1)];
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      lo = min(lo, v[j]);
      hi = max(hi, v[j]);
    }
    *(vec4*)(lds + row * stride + x) = vec4{(T)v[0], (T)v[1], (T)v[2], (T)v[3]};
  }
  __syncthreads();
  constexpr int N = 16 / (int)sizeof(T);  // a block's 80 voxels are a multiple of it
  T* __restrict__ out = slot + (int64_t)(bz * n + by) * n * kSlotBlockElems;
  for (int g = (int)threadIdx.x; g < n * (kSlotBlockElems / N); g += kThreads) {
    const uint32_t i = (uint32_t)g * N, bx = i / kSlotBlockElems, r = i % kSlotBlockElems;
    const T* q = lds + (r / 5) * stride + bx * 4;
    int e = (int)(r % 5);
    T v[N];
#pragma unroll
    for (int j = 0; j < N; ++j) {
      v[j] = q[e];
      if (++e == 5) {
        e = 0;
        q += stride;
      }
    }
    uint4 w;
    __builtin_memcpy(&w, v, sizeof w);
    *(uint4*)(out + i) = w;
  }
}

// Bricks of a flat level into pool slots.  grid.y: brick job; work-group p of
// grid.x takes the slot's block rows [p per, (p + 1) per) (row by + bz n) and
// leaves their range in part[2 (job gridDim.x + p)].  HBM stream: the level
// once (aprons from the caches), the slots once.  An element per thread and
// step (five divisions, a 2-byte load and store) and two atomics a wave on
// its brick's range took 1.17 ms for the 64 bricks of 128^3 of a 512^3 u16
// level and 3.9 ms for the 512 of 1024^3 u8; 0.18 and 1.2 now.
template <typename T>
__global__ __launch_bounds__(kThreads) void extract_bricks_kernel(
    const T* __restrict__ level, int64_t nx, int64_t ny, int64_t nz,
    const BrickJob* __restrict__ jobs, T* __restrict__ pool, int64_t slot_stride,
    int B, int apron, int per, uint32_t* __restrict__ part) {
  extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
  __shared__ uint32_t s_lo[kThreads / 64], s_hi[kThreads / 64];
  const BrickJob job = jobs[blockIdx.y];
  const int S = B + 2 * apron, n = slot_blocks(S);
  uint32_t lo = 0xffffffffu, hi = 0;
  const int r0 = (int)blockIdx.x * per, r1 = min(r0 + per, n * n);
  for (int r = r0; r < r1; ++r) {
    if (r > r0) __syncthreads();  // the last row's voxels have been written out
    slot_block_row<T>(level, nx, ny, nz, (int64_t)job.bx * B - apron, (int64_t)job.by * B - apron,
                      (int64_t)job.bz * B - apron, S, r % n, r / n, pool + job.slot * slot_stride, (T*)lds, lo, hi);
  }
  lo = wave_min(lo);
  hi = wave_max(hi);
  const int wave = (int)(threadIdx.x >> 6);
  if ((threadIdx.x & 63) == 0) {
    s_lo[wave] = lo;
    s_hi[wave] = hi;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int k = 1; k < kThreads / 64; ++k) {
      lo = min(lo, s_lo[k]);
      hi = max(hi, s_hi[k]);
    }
    const int64_t q = (int64_t)blockIdx.y * gridDim.x + blockIdx.x;
    part[2 * q] = lo;
    part[2 * q + 1] = hi;
  }
}

// The bricks' ranges from their parts' (a work-group of one wave per brick).
__global__ __launch_bounds__(64) void brick_range_kernel(const uint32_t* __restrict__ part, int parts,
                                                         const BrickJob* __restrict__ jobs,
                                                         float* __restrict__ brick_range) {
  const int64_t i = blockIdx.x;
  uint32_t lo = 0xffffffffu, hi = 0;
  for (int k = (int)threadIdx.x; k < parts; k += 64) {
    lo = min(lo, part[2 * (i * parts + k)]);
    hi = max(hi, part[2 * (i * parts + k) + 1]);
  }
  lo = wave_min(lo);
  hi = wave_max(hi);
  if (threadIdx.x == 0) {
    brick_range[2 * jobs[i].brick_id] = (float)lo;
    brick_range[2 * jobs[i].brick_id + 1] = (float)hi;
  }
}

// Overlap-inclusive bricks of a flat level, x fastest (the TOC builder's
// stored bricks): job j's brick covers level voxels [b*P - o, b*P - o + S)
// per axis (S = P + 2o); voxels outside the level repeat the nearest edge
// voxel (clamp) or are 0.  Brick j goes to out + j * S^3 (j = the job's
// slot field); its (min, max) over the stored voxels to minmax[2j], [2j+1].
// grid.x: chunks of one brick, grid.y: job.
template <typename T>
__global__ __launch_bounds__(kThreads) void extract_linear_bricks_kernel(
    const T* __restrict__ level, int64_t nx, int64_t ny, int64_t nz,
    const BrickJob* __restrict__ jobs, T* __restrict__ out, int P, int o, int clamp,
    uint32_t* __restrict__ minmax) {
  const BrickJob job = jobs[blockIdx.y];
  const int64_t S = P + 2 * o;
  const int64_t n = S * S * S;
  const int64_t ox = (int64_t)job.bx * P - o, oy = (int64_t)job.by * P - o, oz = (int64_t)job.bz * P - o;
  T* __restrict__ dst = out + job.slot * n;
  const int64_t chunk = (n + gridDim.x - 1) / gridDim.x;
  const int64_t beg = chunk * blockIdx.x;
  const int64_t end = beg + chunk < n ? beg + chunk : n;
  uint32_t lo = 0xffffffffu, hi = 0;
  for (int64_t i = beg + threadIdx.x; i < end; i += kThreads) {
    const int64_t gx = ox + i % S, gy = oy + (i / S) % S, gz = oz + i / (S * S);
    T v;
    if (gx >= 0 && gx < nx && gy >= 0 && gy < ny && gz >= 0 && gz < nz)
      v = level[(gz * ny + gy) * nx + gx];
    else if (clamp)
      v = level[(clamp64(gz, 0, nz - 1) * ny + clamp64(gy, 0, ny - 1)) * nx + clamp64(gx, 0, nx - 1)];
    else
      v = (T)0;
    dst[i] = v;
    lo = min(lo, (uint32_t)v);
    hi = max(hi, (uint32_t)v);
  }
  lo = wave_min(lo);
  hi = wave_max(hi);
  if ((threadIdx.x & 63) == 0) {
    atomicMin(&minmax[2 * job.slot], lo);
    atomicMax(&minmax[2 * job.slot + 1], hi);
  }
}

// An x-fastest S^3 brick into the blocked slot layout (grid.x: block rows),
// and back.
template <typename T>
__global__ __launch_bounds__(kThreads) void linear_to_slot_kernel(const T* __restrict__ src,
                                                                  T* __restrict__ slot, int S) {
  extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
  const int n = slot_blocks(S);
  uint32_t lo = 0xffffffffu, hi = 0;
  slot_block_row<T>(src, S, S, S, 0, 0, 0, S, (int)blockIdx.x % n, (int)blockIdx.x / n, slot, (T*)lds, lo, hi);
}

template <typename T>
__global__ __launch_bounds__(kThreads) void slot_to_linear_kernel(const T* __restrict__ slot,
                                                                  T* __restrict__ dst, int S,
                                                                  int64_t n) {
  const int64_t i = (int64_t)blockIdx.x * kThreads + threadIdx.x;
  if (i >= n) return;
  const int x = (int)(i % S), y = (int)((i / S) % S), z = (int)(i / ((int64_t)S * S));
  dst[i] = slot[slot_offset(slot_geo(S), x, y, z)];
}

// Small empty-space cells (4 <= C <= 32, the default 16 among them): a
// work-group owns the kx = 64 / C cells of a run along x, 64 voxels or a
// cache line of u16, a lane a row of one of them -- neighbouring lanes the
// neighbouring cells of a row -- and writes their packed ranges itself: no
// clearing, global atomics or packing pass.  The voxels [c*C - 1, (c+1)*C]
// (clamped) of a row come as runs of 4.  HBM stream of the level, read about
// twice from the caches (18^3 voxels for 16^3 cells).  512^3 u16 in 16^3
// cells: 0.43 ms a wave per rows of one cell, folded by atomics, 0.17 now.
template <typename T>
__global__ __launch_bounds__(kThreads) void cell_range_small_kernel(const T* __restrict__ level, int64_t nx,
                                                                    int64_t ny, int64_t nz, int C, int ncx,
                                                                    int ncy, int64_t n_groups, int gx,
                                                                    uint32_t* __restrict__ out) {
  __shared__ uint32_t s_lo[16], s_hi[16];  // kx <= 16
  const int kx = 64 / C;
  const int k = (int)threadIdx.x % kx, lrow = (int)threadIdx.x / kx, rstep = kThreads / kx;
  // the loop bound depends on blockIdx only: every thread reaches the barriers
  for (int64_t g = blockIdx.x; g < n_groups; g += gridDim.x) {
    if (threadIdx.x < 16) {
      s_lo[threadIdx.x] = 0xffffffffu;
      s_hi[threadIdx.x] = 0u;
    }
    __syncthreads();
    const int cx = (int)(g % gx) * kx + k, cy = (int)(g / gx % ncy), cz = (int)(g / ((int64_t)gx * ncy));
    const int64_t x0 = max((int64_t)cx * C - 1, (int64_t)0), x1 = min((int64_t)(cx + 1) * C, nx - 1);
    const int64_t y0 = max((int64_t)cy * C - 1, (int64_t)0), y1 = min((int64_t)(cy + 1) * C, ny - 1);
    const int64_t z0 = max((int64_t)cz * C - 1, (int64_t)0), z1 = min((int64_t)(cz + 1) * C, nz - 1);
    const int h = (int)(y1 - y0 + 1), rows = h * (int)(z1 - z0 + 1), w = (int)(x1 - x0 + 1);
    uint32_t lo = 0xffffffffu, hi = 0;
    if (cx < ncx && lrow < rstep) {
      for (int r = lrow; r < rows; r += rstep) {
        const T* row = level + ((z0 + r / h) * ny + (y0 + r % h)) * nx + x0;
        int x = 0;
        for (; x + 4 <= w; x += 4) {
          uint32_t v[4];
          load_run<T, 4>(row + x, v);
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            lo = min(lo, v[j]);
            hi = max(hi, v[j]);
          }
        }
        for (; x < w; ++x) {
          lo = min(lo, (uint32_t)row[x]);
          hi = max(hi, (uint32_t)row[x]);
        }
      }
    }
    if (hi >= lo) {
      atomicMin(&s_lo[k], lo);
      atomicMax(&s_hi[k], hi);
    }
    __syncthreads();
    if (threadIdx.x < (unsigned)kx && cx < ncx)  // thread k of the first kx is cell k's
      out[((int64_t)cz * ncy + cy) * ncx + cx] = s_lo[k] | s_hi[k] << 16;
    __syncthreads();  // s_lo / s_hi are the next group's
  }
}

// Many waves per empty-space cell: the cell's neighbourhood [c*C - 1,
// (c+1)*C] (clamped) is cut into rows of x; a wave takes max(1, 64 / w)
// rows at a time with its lanes over x, the work-groups along grid.y split
// the rows among them, and each work-group folds its minimum and maximum
// into the cell with one atomic each (lo starts at ~0, hi at 0).  The work
// per launch does not depend on the cell size.  Work-groups along grid.x
// take cells blockIdx.x, blockIdx.x + gridDim.x, ... (a 4096^3 level has
// 16.7 M cells of 16^3, more work-groups than one launch may have).
template <typename T>
__global__ __launch_bounds__(kThreads) void cell_range_rows_kernel(const T* __restrict__ level,
                                                                   int64_t nx, int64_t ny, int64_t nz,
                                                                   int C, int ncx, int ncy, int64_t n_cells,
                                                                   uint32_t* __restrict__ lo_out,
                                                                   uint32_t* __restrict__ hi_out) {
  __shared__ uint32_t s_lo[kThreads / 64], s_hi[kThreads / 64];
  const int wave = (int)(threadIdx.x >> 6), lane = (int)(threadIdx.x & 63);
  const int waves = (int)gridDim.y * (kThreads / 64);
  const int wg = (int)blockIdx.y * (kThreads / 64) + wave;
  // the loop bound depends on blockIdx only: every thread of the group runs
  // the same iterations, so the barriers below are reached by all of them
  for (int64_t cell = blockIdx.x; cell < n_cells; cell += gridDim.x) {
    const int64_t cx = cell % ncx, cy = (cell / ncx) % ncy, cz = cell / ((int64_t)ncx * ncy);
    const int64_t x0 = clamp64(cx * C - 1, 0, nx - 1), x1 = clamp64((cx + 1) * C, 0, nx - 1);
    const int64_t y0 = clamp64(cy * C - 1, 0, ny - 1), y1 = clamp64((cy + 1) * C, 0, ny - 1);
    const int64_t z0 = clamp64(cz * C - 1, 0, nz - 1), z1 = clamp64((cz + 1) * C, 0, nz - 1);
    const int w = (int)(x1 - x0 + 1), h = (int)(y1 - y0 + 1), dz = (int)(z1 - z0 + 1);
    const int rows = h * dz;
    const int rpw = w < 64 ? 64 / w : 1;            // rows per wave step
    const int lrow = w < 64 ? lane / w : 0;          // this lane's row in the step
    const int lx = w < 64 ? lane % w : lane;         // and its first x
    const int xstep = w < 64 ? w : 64;
    uint32_t lo = 0xffffffffu, hi = 0;
    if (lrow < rpw) {
      for (int r = wg * rpw + lrow; r < rows; r += waves * rpw) {
        const int y = r % h, z = r / h;
        const T* __restrict__ row = level + ((z0 + z) * ny + (y0 + y)) * nx + x0;
        for (int x = lx; x < w; x += xstep) {
          const uint32_t v = row[x];
          lo = min(lo, v);
          hi = max(hi, v);
        }
      }
    }
    lo = wave_min(lo);
    hi = wave_max(hi);
    if (lane == 0) {
      s_lo[wave] = lo;
      s_hi[wave] = hi;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
      for (int k = 1; k < kThreads / 64; ++k) {
        lo = min(lo, s_lo[k]);
        hi = max(hi, s_hi[k]);
      }
      atomicMin(lo_out + cell, lo);
      atomicMax(hi_out + cell, hi);
    }
    __syncthreads();  // s_lo / s_hi are the next cell's
  }
}

__global__ __launch_bounds__(kThreads) void fill_u32_kernel(uint32_t* __restrict__ p, int64_t n,
                                                            uint32_t v) {
  for (int64_t i = (int64_t)blockIdx.x * kThreads + threadIdx.x; i < n; i += (int64_t)gridDim.x * kThreads)
    p[i] = v;
}

// out = lo | hi << 16 (16-bit voxel values)
__global__ __launch_bounds__(kThreads) void pack_ranges_kernel(uint32_t* __restrict__ out,
                                                               const uint32_t* __restrict__ hi, int64_t n) {
  for (int64_t i = (int64_t)blockIdx.x * kThreads + threadIdx.x; i < n; i += (int64_t)gridDim.x * kThreads)
    out[i] |= hi[i] << 16;
}

// Cell ranges of one brick from its pool slot (paged pools, after upload).
// Cell c of the brick covers level voxels [c*C - 1, (c+1)*C], clamped into
// the slot, whose clamp-to-edge apron gives the values clamping to the level
// would.  Work-group (c, g) folds every gridDim.y-th row step of cell c (a
// wave takes 64/w rows of w < 64 voxels at once, else one row) into
// lo[c] / hi[c] with atomics, so a large cell spreads over many CUs
// (one wave per 256^3 cell ran 62 ms per brick); slot_cell_pack_kernel then
// writes the packed ranges and resets lo / hi for the next brick.
template <typename T>
__global__ __launch_bounds__(kThreads) void slot_cell_range_kernel(
    const T* __restrict__ slot, int S, int apron, int B, int C, int bx, int by, int bz,
    int ncx, int ncy, int ncz, uint32_t* __restrict__ lo_out, uint32_t* __restrict__ hi_out) {
  const int per = B / C;
  const int c = (int)blockIdx.x;  // < per^3
  const int cx = bx * per + c % per, cy = by * per + (c / per) % per, cz = bz * per + c / (per * per);
  if (cx >= ncx || cy >= ncy || cz >= ncz) return;  // whole work-group
  const int x0 = max(cx * C - 1 - (bx * B - apron), 0), x1 = min((cx + 1) * C - (bx * B - apron), S - 1);
  const int y0 = max(cy * C - 1 - (by * B - apron), 0), y1 = min((cy + 1) * C - (by * B - apron), S - 1);
  const int z0 = max(cz * C - 1 - (bz * B - apron), 0), z1 = min((cz + 1) * C - (bz * B - apron), S - 1);
  const int w = x1 - x0 + 1, h = y1 - y0 + 1, dz = z1 - z0 + 1;
  const int rows = h * dz;
  const int lane = (int)(threadIdx.x & 63);
  const int wave = (int)blockIdx.y * (kThreads / 64) + (int)(threadIdx.x >> 6);
  const int waves = (int)gridDim.y * (kThreads / 64);
  const int rpw = w < 64 ? 64 / w : 1;     // rows per wave step
  const int lrow = w < 64 ? lane / w : 0;  // this lane's row in the step
  const int lx = w < 64 ? lane % w : lane;  // and its first x
  const int xstep = w < 64 ? w : 64;
  const SlotGeo G = slot_geo(S);
  uint32_t lo = 0xffffffffu, hi = 0;
  if (lrow < rpw) {
    for (int r = wave * rpw + lrow; r < rows; r += waves * rpw) {
      const int y = y0 + r % h, z = z0 + r / h;
      const int64_t yz = slot_oy(G, y) + slot_oz(G, z);
      for (int x = x0 + lx; x <= x1; x += xstep) {
        const uint32_t v = slot[yz + slot_ox(x)];
        lo = min(lo, v);
        hi = max(hi, v);
      }
    }
  }
  lo = wave_min(lo);
  hi = wave_max(hi);
  if (lane == 0 && hi >= lo) {  // a wave with no rows folds nothing
    atomicMin(lo_out + c, lo);
    atomicMax(hi_out + c, hi);
  }
}

// The brick's cells' ranges into the level's cell-range array, lo / hi
// reset for the next brick.
__global__ __launch_bounds__(kThreads) void slot_cell_pack_kernel(uint32_t* __restrict__ lo,
                                                                  uint32_t* __restrict__ hi, int per,
                                                                  int bx, int by, int bz, int ncx,
                                                                  int ncy, int ncz,
                                                                  uint32_t* __restrict__ out) {
  const int c = (int)(blockIdx.x * kThreads + threadIdx.x);
  if (c >= per * per * per) return;
  const int cx = bx * per + c % per, cy = by * per + (c / per) % per, cz = bz * per + c / (per * per);
  if (cx < ncx && cy < ncy && cz < ncz) out[((int64_t)cz * ncy + cy) * ncx + cx] = lo[c] | (hi[c] << 16);
  lo[c] = 0xffffffffu;
  hi[c] = 0u;
}

__global__ void minmax_init_kernel(uint32_t* mm, int n) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) {
    mm[2 * i] = 0xffffffffu;
    mm[2 * i + 1] = 0u;
  }
}

__global__ void fill_u64_kernel(unsigned long long* p, int64_t n, unsigned long long v) {
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x)
    p[i] = v;
}

// Histograms of few bins (u8 volumes, bricks): one counter per bin and LDS
// bank column, so that at most two of a wave's 64 increments meet on an
// address -- in scans most voxels share a bin, and 64 atomics on one word are
// served one by one (the 16-bin brick histograms of 512^3 u16: 4.34 ms with a shared
// counter per bin and one work-group per brick, below 0.1 ms now).
constexpr int kHistCols = 32;

__device__ inline void cols_count(uint32_t* cols, uint32_t bin) {
  atomicAdd(&cols[bin * kHistCols + (threadIdx.x & (kHistCols - 1))], 1u);
}
__device__ inline uint32_t cols_sum(const uint32_t* cols, int bin) {
  uint32_t s = 0;
  for (int c = 0; c < kHistCols; ++c) s += cols[bin * kHistCols + ((c + bin) & (kHistCols - 1))];
  return s;
}

// u8: 256 bins, 16 voxels per load.  A work-group counts at most 2^31
// voxels (n < 2^40, 2048 work-groups).
__global__ __launch_bounds__(kThreads) void hist1d_u8_kernel(const uint8_t* __restrict__ v,
                                                             int64_t n,
                                                             unsigned long long* hist) {
  __shared__ uint32_t cols[256 * kHistCols];
  for (int i = (int)threadIdx.x; i < 256 * kHistCols; i += kThreads) cols[i] = 0;
  __syncthreads();
  const int64_t step = (int64_t)gridDim.x * kThreads * 16;
  for (int64_t i = ((int64_t)blockIdx.x * kThreads + threadIdx.x) * 16; i < n; i += step) {
    if (i + 16 <= n) {
      uint32_t x[16];
      load_run<uint8_t, 16>(v + i, x);
#pragma unroll
      for (int j = 0; j < 16; ++j) cols_count(cols, x[j]);
    } else {
      for (int64_t k = i; k < n; ++k) cols_count(cols, v[k]);
    }
  }
  __syncthreads();
  const uint32_t c = cols_sum(cols, (int)threadIdx.x);
  if (c) atomicAdd(&hist[threadIdx.x], (unsigned long long)c);
}

// u16: 65536 bins do not fit a block's LDS; count in global memory.
__global__ __launch_bounds__(kThreads) void hist1d_u16_kernel(const uint16_t* __restrict__ v,
                                                              int64_t n,
                                                              unsigned long long* hist) {
  for (int64_t i = (int64_t)blockIdx.x * kThreads + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * kThreads)
    atomicAdd(&hist[v[i]], 1ull);
}

// Integer squared gradient in units of 1/(2*maxval): central differences
// v[c+1]-v[c-1] inside, 2*(one-sided difference) at the borders (the
// numpy.gradient definition that reproduces the 2D histogram stored in
// DemoData/c60.uvf).
template <typename T>
__device__ inline long long grad_k(const T* __restrict__ v, int64_t i, int64_t c, int64_t n,
                                   int64_t stride) {
  if (n < 2) return 0;
  if (c == 0) return 2ll * ((long long)v[i + stride] - (long long)v[i]);
  if (c == n - 1) return 2ll * ((long long)v[i] - (long long)v[i - stride]);
  return (long long)v[i + stride] - (long long)v[i - stride];
}

template <typename T>
__device__ inline unsigned long long grad_K(const T* __restrict__ v, int64_t nx, int64_t ny,
                                            int64_t nz, int64_t x, int64_t y, int64_t z) {
  const int64_t i = (z * ny + y) * nx + x;
  const long long gx = grad_k(v, i, x, nx, 1);
  const long long gy = grad_k(v, i, y, ny, nx);
  const long long gz = grad_k(v, i, z, nz, nx * ny);
  return (unsigned long long)(gx * gx + gy * gy + gz * gz);
}

// grad_K of up to kRunX consecutive voxels (x .. x + n - 1) of row (y, z),
// whose values come along in c: the five rows they read arrive in one load
// each.  u8 sums stay below 2^20 and are kept in 32 bits.
constexpr int kRunX = 8;
template <typename T>
struct GradSum {
  typedef unsigned long long type;
};
template <>
struct GradSum<uint8_t> {
  typedef uint32_t type;
};

template <typename T>
__device__ inline void grad_run(const T* __restrict__ v, int64_t nx, int64_t ny, int64_t nz, int64_t x, int64_t y,
                                int64_t z, int n, uint32_t (&c)[kRunX], typename GradSum<T>::type (&K)[kRunX]) {
  typedef typename GradSum<T>::type Sum;
  const T* row = v + (z * ny + y) * nx + x;
  // per axis: rows b and a with K += (f (b - a))^2: inside b = +1, a = -1 and
  // f = 1; at a border the one-sided difference and f = 2; f = 0 for an axis
  // of one voxel
  const T* yb = row + (y + 1 < ny ? nx : 0);
  const T* ya = row - (y > 0 ? nx : 0);
  const T* zb = row + (z + 1 < nz ? nx * ny : 0);
  const T* za = row - (z > 0 ? nx * ny : 0);
  const int fy = ny < 2 ? 0 : (y == 0 || y + 1 == ny ? 2 : 1);
  const int fz = nz < 2 ? 0 : (z == 0 || z + 1 == nz ? 2 : 1);
  uint32_t b1[kRunX], a1[kRunX], b2[kRunX], a2[kRunX];
  if (n == kRunX) {
    load_run<T, kRunX>(row, c);
    load_run<T, kRunX>(yb, b1);
    load_run<T, kRunX>(ya, a1);
    load_run<T, kRunX>(zb, b2);
    load_run<T, kRunX>(za, a2);
  } else {
#pragma unroll
    for (int j = 0; j < kRunX; ++j) {
      const int q = j < n ? j : 0;
      c[j] = row[q];
      b1[j] = yb[q];
      a1[j] = ya[q];
      b2[j] = zb[q];
      a2[j] = za[q];
    }
  }
  const uint32_t left = x > 0 ? row[-1] : c[0];
  const uint32_t right = x + n < nx ? row[n] : c[kRunX - 1];
#pragma unroll
  for (int j = 0; j < kRunX; ++j) {
    // the voxel beyond the run's end, or the last voxel itself at the border
    const uint32_t nxt = j + 1 < n ? c[j + 1 < kRunX ? j + 1 : j] : (x + n < nx ? right : c[j]);
    const uint32_t prv = j > 0 ? c[j > 0 ? j - 1 : 0] : left;
    const int fx = nx < 2 ? 0 : (x + j == 0 || x + j + 1 == nx ? 2 : 1);
    const int gx = fx * ((int)nxt - (int)prv);
    const int gy = fy * ((int)b1[j] - (int)a1[j]);
    const int gz = fz * ((int)b2[j] - (int)a2[j]);
    const uint32_t ux = (uint32_t)abs(gx), uy = (uint32_t)abs(gy), uz = (uint32_t)abs(gz);
    K[j] = (Sum)ux * ux + (Sum)uy * uy + (Sum)uz * uz;
  }
}

// How a work-group of `threads` walks a volume's rows in runs of kRunX: a
// work-group takes spw runs of a row (chunk blockIdx.x of the row) and
// threads / spw rows at a time.
struct RunWalk {
  int spw;   // runs of a row per work-group pass
  int rows;  // rows per pass
};
__host__ __device__ inline RunWalk run_walk(int64_t nx, int threads) {
  const int64_t runs = (nx + kRunX - 1) / kRunX;
  const int spw = runs < threads ? (int)runs : threads;
  return RunWalk{spw, threads / spw};
}

// The largest squared integer gradient.  HBM stream: the volume once, its
// neighbour rows from the caches.  With a 2-byte load per voxel and
// neighbour and 64-bit index arithmetic, 512^3 u16 took 3.59 ms; 0.32 now.
template <typename T>
__global__ __launch_bounds__(kThreads) void gradient_kmax_kernel(const T* __restrict__ v,
                                                                 int64_t nx, int64_t ny,
                                                                 int64_t nz,
                                                                 unsigned long long* kmax) {
  const RunWalk W = run_walk(nx, kThreads);
  typename GradSum<T>::type m = 0;
  const int64_t x = ((int64_t)blockIdx.x * W.spw + (int)threadIdx.x % W.spw) * kRunX;
  const int lrow = (int)threadIdx.x / W.spw;
  if (lrow < W.rows && x < nx) {
    const int n = nx - x < kRunX ? (int)(nx - x) : kRunX;
    // rows of a level stay below 2^32 for every supported volume
    const uint32_t rows = (uint32_t)(ny * nz), uny = (uint32_t)ny;
    for (uint64_t row = (uint64_t)blockIdx.y * W.rows + lrow; row < rows; row += (uint64_t)gridDim.y * W.rows) {
      uint32_t c[kRunX];
      typename GradSum<T>::type K[kRunX];
      grad_run(v, nx, ny, nz, x, (int64_t)((uint32_t)row % uny), (int64_t)((uint32_t)row / uny), n, c, K);
#pragma unroll
      for (int j = 0; j < kRunX; ++j)
        if (j < n) m = K[j] > m ? K[j] : m;
    }
  }
  const unsigned long long w = wave_max64((unsigned long long)m);
  if ((threadIdx.x & 63) == 0 && w) atomicMax(kmax, w);
}

// The 2D histogram bin of voxel (x, y, z): value >> shift along the value
// axis, b = max{ b : b^2 kmax <= F^2 K } along the gradient axis (F =
// n_grad - 1, K and kmax squared integer gradients), decided exactly in
// integers after a float estimate.
template <typename T>
__device__ inline int64_t hist2d_bin(const T* __restrict__ v, int64_t nx, int64_t ny, int64_t nz,
                                     int64_t x, int64_t y, int64_t z, unsigned long long kmax, int shift,
                                     int n_grad) {
  const unsigned long long F = (unsigned long long)(n_grad - 1);
  const unsigned long long K = grad_K(v, nx, ny, nz, x, y, z);
  long long b = 0;
  if (kmax > 0) {
    b = (long long)floorf((float)F * sqrtf((float)K / (float)kmax));
    if (b < 0) b = 0;
    if (b > (long long)F) b = (long long)F;
    const unsigned long long rhs = F * F * K;
    while (b < (long long)F && (unsigned long long)(b + 1) * (unsigned long long)(b + 1) * kmax <= rhs) ++b;
    while (b > 0 && (unsigned long long)b * (unsigned long long)b * kmax > rhs) --b;
  }
  const int64_t vb = (int64_t)(v[(z * ny + y) * nx + x] >> shift);
  return vb * n_grad + b;
}

template <typename T>
__global__ __launch_bounds__(kThreads) void hist2d_kernel(const T* __restrict__ v, int64_t nx,
                                                          int64_t ny, int64_t nz,
                                                          const unsigned long long* kmax_p,
                                                          int shift, int n_grad,
                                                          unsigned long long* hist) {
  const int64_t x = (int64_t)blockIdx.x * kThreads + threadIdx.x;
  if (x >= nx) return;
  const unsigned long long kmax = *kmax_p;
  const uint32_t rows = (uint32_t)(ny * nz), uny = (uint32_t)ny;
  for (uint32_t row = blockIdx.y; row < rows; row += gridDim.y) {
    const int64_t y = row % uny, z = row / uny;
    atomicAdd(&hist[hist2d_bin(v, nx, ny, nz, x, y, z, kmax, shift, n_grad)], 1ull);
  }
}

// Privatised histograms of many bins: a work-group counts in LDS, 16-bit
// counters two to a 32-bit word (up to 65536 bins = 128 KiB, so one
// work-group of 16 waves per CU), and adds its non-zero bins to the global
// u64 histogram at its end.  A counter that reaches 0x8000 hands 0x8000 on
// to the global bin after the run that took it there; a work-group meets a
// barrier after at most kHistChunk counts, so a counter never passes 0x8000 + kHistChunk before
// the hand-over that its crossing started is done.  Lanes that share the
// first lane's bin add once for all of them: in scans most of a wave's
// voxels are the same.
constexpr int kHistThreads = 1024;
constexpr int kHistChunk = 3 * kHistThreads * kRunX;
static_assert(0x8000 + kHistChunk <= 0xffff, "a 16-bit counter must hold a chunk above its hand-over mark");

// Counts the first n of a run's bins; every lane of the wave calls this.  The
// run's adds are all in flight before the first returned count is looked at.
__device__ inline void lds_count(uint32_t* words, const uint32_t (&bin)[kRunX], int n, unsigned long long* hist) {
  const int lane = (int)(threadIdx.x & 63);
  uint32_t old[kRunX], k[kRunX];
#pragma unroll
  for (int j = 0; j < kRunX; ++j) {
    old[j] = 0, k[j] = 0;
    const unsigned long long act = __ballot(j < n);
    if (act == 0) continue;
    const int first = __builtin_ctzll(act);
    const uint32_t b0 = (uint32_t)__builtin_amdgcn_readlane((int)bin[j], first);
    const unsigned long long same = __ballot(j < n && bin[j] == b0);
    if (j < n) k[j] = lane == first ? (uint32_t)__popcll(same) : bin[j] != b0 ? 1u : 0u;
    if (k[j] != 0) old[j] = atomicAdd(&words[bin[j] >> 1], k[j] << ((bin[j] & 1u) * 16u));
  }
#pragma unroll
  for (int j = 0; j < kRunX; ++j) {
    const uint32_t sh = (bin[j] & 1u) * 16u, was = (old[j] >> sh) & 0xffffu;
    if (was < 0x8000u && was + k[j] >= 0x8000u) {
      atomicSub(&words[bin[j] >> 1], 0x8000u << sh);
      atomicAdd(&hist[bin[j]], 0x8000ull);
    }
  }
}

// Neighbouring lanes add neighbouring bins, and each work-group starts at its
// own part of the bins: they all end at once, and adds to one line wait for
// each other.
__device__ inline void lds_flush(const uint32_t* words, int nbins, unsigned long long* hist) {
  const int from = (int)((int64_t)nbins * blockIdx.x / gridDim.x) & ~15;
  for (int k = (int)threadIdx.x; k < nbins; k += kHistThreads) {
    const int b = k + from < nbins ? k + from : k + from - nbins;
    const uint32_t c = words[b >> 1] >> ((b & 1) * 16) & 0xffffu;
    if (c) atomicAdd(&hist[b], (unsigned long long)c);
  }
}

// 2D histogram, all bins in LDS; up to kHistThresholds gradient bins also
// their thresholds: threshold[b] = ceil(b^2 kmax / F^2), the least K of bin
// b, so a bin is a float estimate and two comparisons (more bins compare
// b^2 kmax with F^2 K, as hist2d_bin does).  Bound by the LDS atomics and the
// gradients' arithmetic.  512^3 u16 took 2.12 ms with a 2-byte load per voxel
// and neighbour, 64-bit products per voxel and a flush of all bins per 65,535
// voxels; 0.51 now.
constexpr int kHistThresholds = 1024;
template <typename T>
__global__ __launch_bounds__(kHistThreads) void hist2d_lds_kernel(const T* __restrict__ v, int64_t nx,
                                                                  int64_t ny, int64_t nz,
                                                                  const unsigned long long* kmax_p,
                                                                  int shift, int n_grad, int nbins,
                                                                  unsigned long long* hist) {
  extern __shared__ __attribute__((aligned(8))) uint32_t words[];
  const int nwords = nbins >> 1;
  unsigned long long* thr = (unsigned long long*)(words + ((nwords + 1) & ~1));
  const unsigned long long kmax = *kmax_p;
  const unsigned long long F = (unsigned long long)(n_grad - 1);
  for (int k = (int)threadIdx.x; k < nwords; k += kHistThreads) words[k] = 0;
  const bool table = n_grad <= kHistThresholds;
  for (int b = (int)threadIdx.x; table && b < n_grad; b += kHistThreads)
    thr[b] = ((unsigned long long)b * b * kmax + F * F - 1) / (F * F);
  __syncthreads();
  const float scale = kmax > 0 ? (float)F / sqrtf((float)kmax) : 0.f;
  const RunWalk W = run_walk(nx, kHistThreads);
  const int64_t xs = (int64_t)W.spw * kRunX;  // voxels of a row per pass
  const int64_t xchunks = (nx + xs - 1) / xs;
  const int lrow = (int)threadIdx.x / W.spw;
  const int64_t lx = (int64_t)((int)threadIdx.x % W.spw) * kRunX;
  const int64_t rows = ny * nz, passes = (rows + W.rows - 1) / W.rows * xchunks;
  const uint32_t uny = (uint32_t)ny;
  int counted = 0;
  // the trip count depends on blockIdx only: every thread reaches the barriers
  for (int64_t p = blockIdx.x; p < passes; p += gridDim.x) {
    const int64_t row = p / xchunks * W.rows + lrow, x = p % xchunks * xs + lx;
    const bool on = lrow < W.rows && row < rows && x < nx;
    const int n = on ? (nx - x < kRunX ? (int)(nx - x) : kRunX) : 0;
    uint32_t c[kRunX];
    typename GradSum<T>::type K[kRunX];
    if (on) {
      grad_run(v, nx, ny, nz, x, (int64_t)((uint32_t)row % uny), (int64_t)((uint32_t)row / uny), n, c, K);
    } else {
#pragma unroll
      for (int j = 0; j < kRunX; ++j) c[j] = 0, K[j] = 0;
    }
    uint32_t bin[kRunX];
#pragma unroll
    for (int j = 0; j < kRunX; ++j) {
      bin[j] = 0;
      if (j < n) {
        int b = 0;
        if (kmax > 0) {
          b = min((int)(scale * __builtin_amdgcn_sqrtf((float)K[j])), (int)F);
          const unsigned long long k = K[j];
          auto reaches = [&](int q) {
            return table ? k >= thr[q] : (unsigned long long)q * (unsigned long long)q * kmax <= F * F * k;
          };
          while (b < (int)F && reaches(b + 1)) ++b;
          while (b > 0 && !reaches(b)) --b;
        }
        bin[j] = (c[j] >> shift) * (uint32_t)n_grad + (uint32_t)b;
      }
    }
    lds_count(words, bin, n, hist);
    if (++counted == kHistChunk / (kHistThreads * kRunX)) {
      __syncthreads();
      counted = 0;
    }
  }
  __syncthreads();
  lds_flush(words, nbins, hist);
}

// 1D histogram of u16 voxels, as above, bound by the LDS atomics: 512^3 took
// 0.78 ms without the privatised counts and 0.34 with every add waited for by
// itself and all work-groups flushing from bin 0; 0.20 now.
__global__ __launch_bounds__(kHistThreads) void hist1d_u16_lds_kernel(const uint16_t* __restrict__ v,
                                                                      int64_t n,
                                                                      unsigned long long* hist) {
  extern __shared__ uint32_t words[];
  constexpr int nwords = 65536 / 2;
  for (int k = (int)threadIdx.x; k < nwords; k += kHistThreads) words[k] = 0;
  __syncthreads();
  constexpr int64_t kPass = (int64_t)kHistThreads * kRunX;
  int counted = 0;
  for (int64_t p = blockIdx.x; p * kPass < n; p += gridDim.x) {  // trip count: blockIdx only
    const int64_t i = p * kPass + (int64_t)threadIdx.x * kRunX;
    const int m = i >= n ? 0 : (n - i < kRunX ? (int)(n - i) : kRunX);
    uint32_t x[kRunX];
    if (m == kRunX) {
      load_run<uint16_t, kRunX>(v + i, x);
    } else {
#pragma unroll
      for (int j = 0; j < kRunX; ++j) x[j] = j < m ? v[i + j] : 0;
    }
    lds_count(words, x, m, hist);
    if (++counted == kHistChunk / (kHistThreads * kRunX)) {
      __syncthreads();
      counted = 0;
    }
  }
  __syncthreads();
  lds_flush(words, 65536, hist);
}

// CUs of the current device (work-groups of a kernel that takes a CU each).
int device_cus() {
  int dev = 0, cus = 0;
  if (hipGetDevice(&dev) != hipSuccess ||
      hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cus < 1)
    return 256;
  return cus;
}

// Dynamic LDS of `bytes` for kernel `k` on the current device, if it allows it.
template <typename K>
bool lds_allowed(K k, size_t bytes) {
  int dev = 0, max_lds = 0;
  if (hipGetDevice(&dev) != hipSuccess ||
      hipDeviceGetAttribute(&max_lds, hipDeviceAttributeMaxSharedMemoryPerBlock, dev) != hipSuccess)
    return false;
  if ((size_t)max_lds < bytes) return false;
  return hipFuncSetAttribute((const void*)k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes) == hipSuccess;
}

inline dim3 row_grid(int64_t nx, int64_t rows) {
  const int64_t gy = rows < 65535 ? rows : 65535;
  return dim3((unsigned)((nx + kThreads - 1) / kThreads), (unsigned)(gy > 0 ? gy : 1), 1);
}

}  // namespace

hipError_t launch_fill_u64(unsigned long long* p, int64_t n, unsigned long long v,
                           hipStream_t stream) {
  if (n <= 0) return hipSuccess;
  int64_t blocks = (n + kThreads - 1) / kThreads;
  if (blocks > 65536) blocks = 65536;
  fill_u64_kernel<<<(unsigned)blocks, kThreads, 0, stream>>>(p, n, v);
  return hipGetLastError();
}

hipError_t launch_downsample(const void* src, int bpv, const int64_t d[3], void* dst,
                             hipStream_t stream, bool median) {
  const int64_t mx = (d[0] + 1) / 2, my = (d[1] + 1) / 2, mz = (d[2] + 1) / 2;
  const dim3 grid = row_grid(mx, my * mz);
  if (bpv == 1) {
    if (median)
      downsample_kernel<uint8_t, true><<<grid, kThreads, 0, stream>>>(
          (const uint8_t*)src, d[0], d[1], d[2], (uint8_t*)dst, mx, my, mz);
    else
      downsample_kernel<uint8_t, false><<<grid, kThreads, 0, stream>>>(
          (const uint8_t*)src, d[0], d[1], d[2], (uint8_t*)dst, mx, my, mz);
  } else {
    if (median)
      downsample_kernel<uint16_t, true><<<grid, kThreads, 0, stream>>>(
          (const uint16_t*)src, d[0], d[1], d[2], (uint16_t*)dst, mx, my, mz);
    else
      downsample_kernel<uint16_t, false><<<grid, kThreads, 0, stream>>>(
          (const uint16_t*)src, d[0], d[1], d[2], (uint16_t*)dst, mx, my, mz);
  }
  return hipGetLastError();
}

// LDS of slot_block_row: 16 rows of 4 (n + 1) voxels (33 KiB for the largest
// slots of u16).
static size_t block_row_lds(int S, int bpv) { return (size_t)16 * 4 * (slot_blocks(S) + 1) * bpv; }

// Block rows per work-group: one brick's rows spread until the launch has
// about 16 work-groups per CU.
static int extract_rows(int64_t n_jobs, int S) {
  const int64_t n = slot_blocks(S), rows = n * n;
  return (int)std::max<int64_t>(1, std::min<int64_t>(rows, rows * n_jobs / 4096));
}

int64_t extract_scratch_words(int64_t n_jobs, int S) {
  const int64_t rows = (int64_t)slot_blocks(S) * slot_blocks(S), per = extract_rows(n_jobs, S);
  return 2 * n_jobs * ((rows + per - 1) / per);
}

hipError_t launch_extract_bricks(const void* level, int bpv, const int64_t d[3],
                                 const BrickJob* jobs, int n_jobs, void* pool,
                                 int64_t slot_stride, int B, int apron, float* brick_range,
                                 uint32_t* scratch, hipStream_t stream) {
  if (n_jobs <= 0) return hipSuccess;
  const int S = B + 2 * apron, n = slot_blocks(S), per = extract_rows(n_jobs, S);
  const int parts = (n * n + per - 1) / per;
  const size_t lds = block_row_lds(S, bpv);
  for (int j0 = 0; j0 < n_jobs; j0 += 65535) {
    const int nj = n_jobs - j0 < 65535 ? n_jobs - j0 : 65535;
    const dim3 grid((unsigned)parts, (unsigned)nj, 1);
    uint32_t* part = scratch + (int64_t)2 * j0 * parts;
    if (bpv == 1)
      extract_bricks_kernel<uint8_t><<<grid, kThreads, lds, stream>>>(
          (const uint8_t*)level, d[0], d[1], d[2], jobs + j0, (uint8_t*)pool, slot_stride, B, apron, per, part);
    else
      extract_bricks_kernel<uint16_t><<<grid, kThreads, lds, stream>>>(
          (const uint16_t*)level, d[0], d[1], d[2], jobs + j0, (uint16_t*)pool, slot_stride, B, apron, per, part);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
  }
  brick_range_kernel<<<(unsigned)n_jobs, 64, 0, stream>>>(scratch, parts, jobs, brick_range);
  return hipGetLastError();
}

hipError_t launch_extract_linear_bricks(const void* level, int bpv, const int64_t d[3],
                                        const BrickJob* jobs, int n_jobs, void* out, int P, int o,
                                        bool clamp, uint32_t* minmax, hipStream_t stream) {
  if (n_jobs <= 0) return hipSuccess;
  minmax_init_kernel<<<(n_jobs + 255) / 256, 256, 0, stream>>>(minmax, n_jobs);
  const int64_t S = P + 2 * o;
  int64_t chunks = (S * S * S + 8191) / 8192;
  if (chunks > 1024) chunks = 1024;
  if (chunks < 1) chunks = 1;
  for (int j0 = 0; j0 < n_jobs; j0 += 65535) {
    const int nj = n_jobs - j0 < 65535 ? n_jobs - j0 : 65535;
    const dim3 grid((unsigned)chunks, (unsigned)nj, 1);
    if (bpv == 1)
      extract_linear_bricks_kernel<uint8_t><<<grid, kThreads, 0, stream>>>(
          (const uint8_t*)level, d[0], d[1], d[2], jobs + j0, (uint8_t*)out, P, o, clamp ? 1 : 0, minmax);
    else
      extract_linear_bricks_kernel<uint16_t><<<grid, kThreads, 0, stream>>>(
          (const uint16_t*)level, d[0], d[1], d[2], jobs + j0, (uint16_t*)out, P, o, clamp ? 1 : 0, minmax);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
  }
  return hipSuccess;
}

hipError_t launch_linear_to_slot(const void* src, void* slot, int bpv, int S, hipStream_t stream) {
  const unsigned rows = (unsigned)(slot_blocks(S) * slot_blocks(S));
  const size_t lds = block_row_lds(S, bpv);
  if (bpv == 1)
    linear_to_slot_kernel<uint8_t><<<rows, kThreads, lds, stream>>>((const uint8_t*)src, (uint8_t*)slot, S);
  else
    linear_to_slot_kernel<uint16_t><<<rows, kThreads, lds, stream>>>((const uint16_t*)src, (uint16_t*)slot, S);
  return hipGetLastError();
}

hipError_t launch_slot_to_linear(const void* slot, void* dst, int bpv, int S, hipStream_t stream) {
  const int64_t n = (int64_t)S * S * S;
  const unsigned blocks = (unsigned)((n + kThreads - 1) / kThreads);
  if (bpv == 1)
    slot_to_linear_kernel<uint8_t><<<blocks, kThreads, 0, stream>>>((const uint8_t*)slot, (uint8_t*)dst, S, n);
  else
    slot_to_linear_kernel<uint16_t><<<blocks, kThreads, 0, stream>>>((const uint16_t*)slot, (uint16_t*)dst,
                                                                      S, n);
  return hipGetLastError();
}

hipError_t launch_cell_ranges(const void* level, int bpv, const int64_t d[3], int C, uint32_t* out,
                              uint32_t* tmp_hi, hipStream_t stream) {
  const int ncx = (int)((d[0] + C - 1) / C), ncy = (int)((d[1] + C - 1) / C),
            ncz = (int)((d[2] + C - 1) / C);
  const int64_t cells = (int64_t)ncx * ncy * ncz;
  if (!cell_ranges_fold(C)) {
    const int gx = (ncx + 64 / C - 1) / (64 / C);
    const int64_t n = (int64_t)gx * ncy * ncz;
    const unsigned groups = (unsigned)std::min<int64_t>(n, (int64_t)1 << 20);
    if (bpv == 1)
      cell_range_small_kernel<uint8_t><<<groups, kThreads, 0, stream>>>((const uint8_t*)level, d[0], d[1], d[2], C,
                                                                        ncx, ncy, n, gx, out);
    else
      cell_range_small_kernel<uint16_t><<<groups, kThreads, 0, stream>>>((const uint16_t*)level, d[0], d[1], d[2], C,
                                                                         ncx, ncy, n, gx, out);
    return hipGetLastError();
  }
  const unsigned fill_blocks = (unsigned)std::min<int64_t>((cells + kThreads - 1) / kThreads, 65536);
  fill_u32_kernel<<<fill_blocks, kThreads, 0, stream>>>(out, cells, 0xffffffffu);
  fill_u32_kernel<<<fill_blocks, kThreads, 0, stream>>>(tmp_hi, cells, 0u);
  // work-groups per cell: about 8 row steps per wave over the largest cell
  const int64_t w = C + 2, rows = w * w;
  const int64_t rpw = w < 64 ? 64 / w : 1;
  const int64_t per_group = (kThreads / 64) * rpw * 8;
  const unsigned gy = (unsigned)std::min<int64_t>(std::max<int64_t>(1, (rows + per_group - 1) / per_group), 65535);
  // at most 2^20 work-groups along x (a launch counts each dimension's
  // work-items in 32 bits: one work-group per cell of a 4096^3 level would
  // be 2^32 of them); more cells loop inside the kernel
  const unsigned gx = (unsigned)std::min<int64_t>(cells, (int64_t)1 << 20);
  const dim3 grid(gx, gy, 1);
  if (bpv == 1)
    cell_range_rows_kernel<uint8_t><<<grid, kThreads, 0, stream>>>((const uint8_t*)level, d[0], d[1], d[2], C,
                                                                   ncx, ncy, cells, out, tmp_hi);
  else
    cell_range_rows_kernel<uint16_t><<<grid, kThreads, 0, stream>>>((const uint16_t*)level, d[0], d[1], d[2], C,
                                                                    ncx, ncy, cells, out, tmp_hi);
  pack_ranges_kernel<<<fill_blocks, kThreads, 0, stream>>>(out, tmp_hi, cells);
  return hipGetLastError();
}

hipError_t launch_slot_cell_ranges(const void* slot, int bpv, int S, int apron, int B, int C,
                                   const int brick[3], const int cells[3], uint32_t* out,
                                   uint32_t* tmp, hipStream_t stream) {
  const int per = B / C;
  const int n = per * per * per;
  // work-groups per cell: about 8 row steps per wave over the cell
  const int64_t w = C + 2, rows = w * w;
  const int64_t rpw = w < 64 ? 64 / w : 1;
  const int64_t per_group = (kThreads / 64) * rpw * 8;
  const unsigned gy = (unsigned)std::min<int64_t>(std::max<int64_t>(1, (rows + per_group - 1) / per_group), 65535);
  const dim3 grid((unsigned)n, gy, 1);
  uint32_t* lo = tmp;
  uint32_t* hi = tmp + n;
  if (bpv == 1)
    slot_cell_range_kernel<uint8_t><<<grid, kThreads, 0, stream>>>(
        (const uint8_t*)slot, S, apron, B, C, brick[0], brick[1], brick[2], cells[0], cells[1], cells[2], lo, hi);
  else
    slot_cell_range_kernel<uint16_t><<<grid, kThreads, 0, stream>>>(
        (const uint16_t*)slot, S, apron, B, C, brick[0], brick[1], brick[2], cells[0], cells[1], cells[2], lo,
        hi);
  slot_cell_pack_kernel<<<(unsigned)((n + kThreads - 1) / kThreads), kThreads, 0, stream>>>(
      lo, hi, per, brick[0], brick[1], brick[2], cells[0], cells[1], cells[2], out);
  return hipGetLastError();
}

hipError_t launch_slot_cell_tmp_init(uint32_t* tmp, int per, hipStream_t stream) {
  const int64_t n = (int64_t)per * per * per;
  const unsigned blocks = (unsigned)std::min<int64_t>((n + kThreads - 1) / kThreads, 65536);
  fill_u32_kernel<<<blocks, kThreads, 0, stream>>>(tmp, n, 0xffffffffu);
  fill_u32_kernel<<<blocks, kThreads, 0, stream>>>(tmp + n, n, 0u);
  return hipGetLastError();
}

// How the work-groups of a per-brick reduction walk one brick of payload B
// (clipped to the level, w x h x d voxels): runs of kBrickRun voxels along x,
// thread t at run t % segs of row t / segs, kThreads / segs rows per pass,
// the rows split over gridDim.y work-groups.
constexpr int kBrickRun = 4;

// Work-groups per brick: at least 16 passes each, more for fewer bricks
// until the launch has about 8 work-groups per CU.
static inline unsigned brick_parts(int64_t bricks, int B) {
  const int64_t segs = (B + kBrickRun - 1) / kBrickRun;
  const int64_t per_pass = kThreads / segs;  // B <= 1024: segs <= 256
  const int64_t passes = ((int64_t)B * B + per_pass - 1) / per_pass;
  const int64_t want = std::max<int64_t>(1, 8 * 256 / std::max<int64_t>(1, bricks));
  // a thread sums at most 2^16 voxels (|difference| < 2^16 fits 32 bits then)
  const int64_t least = (passes + (1 << 14) - 1) >> 14;
  return (unsigned)std::max<int64_t>(least, std::min<int64_t>(want, std::max<int64_t>(1, passes / 16)));
}

// Per-brick value histogram of a flat level: `bins` equal bins over
// [0, 2^(8 bpv)), counted in bank columns (cols_count).  out is cleared by
// the caller.
template <typename T>
__global__ __launch_bounds__(kThreads) void brick_hist_kernel(const T* __restrict__ level, int64_t nx,
                                                              int64_t ny, int64_t nz, int B, int gx,
                                                              int gy, int bins, int shift,
                                                              uint32_t* __restrict__ out) {
  __shared__ uint32_t cols[64 * kHistCols];
  for (int i = (int)threadIdx.x; i < bins * kHistCols; i += kThreads) cols[i] = 0;
  __syncthreads();
  const int b = (int)blockIdx.x;
  const int bx = b % gx, by = (b / gx) % gy, bz = b / (gx * gy);
  const int64_t x0 = (int64_t)bx * B, y0 = (int64_t)by * B, z0 = (int64_t)bz * B;
  const int w = (int)min<int64_t>(B, nx - x0), h = (int)min<int64_t>(B, ny - y0),
            d = (int)min<int64_t>(B, nz - z0);
  const int segs = (w + kBrickRun - 1) / kBrickRun, rpp = kThreads / segs;
  const int lrow = (int)threadIdx.x / segs, x = (int)threadIdx.x % segs * kBrickRun;
  if (lrow < rpp) {
    const int step = rpp * (int)gridDim.y;
    for (int r = (int)blockIdx.y * rpp + lrow; r < h * d; r += step) {
      const int y = r % h, z = r / h;
      const T* row = level + ((z0 + z) * ny + (y0 + y)) * nx + (x0 + x);
      if (x + kBrickRun <= w) {
        uint32_t v[kBrickRun];
        load_run<T, kBrickRun>(row, v);
#pragma unroll
        for (int j = 0; j < kBrickRun; ++j) cols_count(cols, v[j] >> shift);
      } else {
        for (int j = 0; x + j < w; ++j) cols_count(cols, (uint32_t)row[j] >> shift);
      }
    }
  }
  __syncthreads();
  for (int i = (int)threadIdx.x; i < bins; i += kThreads) {
    const uint32_t c = cols_sum(cols, i);
    if (c) atomicAdd(&out[(int64_t)b * bins + i], c);
  }
}

// Per LOD-0 brick region and level l >= 1: the sum of |v0(x) - v_l(x >> l)|
// over the region's voxels (each LOD-0 voxel against its level-l ancestor),
// exact in integers; sums[region * n_lod + l], cleared by the caller.  HBM
// stream of level 0, the coarser levels from the caches.  One work-group per
// region, a voxel per thread step and FP32 sums took 8.57 ms for the 64
// regions of 512^3 u16; 0.18 now.
struct DetailLevels {
  const void* level[16];
  int64_t dims[16][3];
};

template <typename T>
__global__ __launch_bounds__(kThreads) void region_detail_kernel(const DetailLevels D, int n_lod, int B,
                                                                 int gx, int gy,
                                                                 unsigned long long* __restrict__ sums) {
  __shared__ unsigned long long red[16];
  if (threadIdx.x < 16) red[threadIdx.x] = 0;
  __syncthreads();
  const int reg = (int)blockIdx.x;
  const int bx = reg % gx, by = (reg / gx) % gy, bz = reg / (gx * gy);
  const int64_t nx = D.dims[0][0], ny = D.dims[0][1], nz = D.dims[0][2];
  const int64_t x0 = (int64_t)bx * B, y0 = (int64_t)by * B, z0 = (int64_t)bz * B;
  const int w = (int)min<int64_t>(B, nx - x0), h = (int)min<int64_t>(B, ny - y0),
            d = (int)min<int64_t>(B, nz - z0);
  const int segs = (w + kBrickRun - 1) / kBrickRun, rpp = kThreads / segs;
  const int lrow = (int)threadIdx.x / segs, lx = (int)threadIdx.x % segs * kBrickRun;
  uint32_t acc[16];
#pragma unroll
  for (int l = 0; l < 16; ++l) acc[l] = 0;
  const T* v0 = (const T*)D.level[0];
  if (lrow < rpp) {
    const int step = rpp * (int)gridDim.y;
    const int n = min(kBrickRun, w - lx);
    const int64_t x = x0 + lx;
    for (int r = (int)blockIdx.y * rpp + lrow; r < h * d; r += step) {
      const int64_t y = y0 + r % h, z = z0 + r / h;
      const T* row = v0 + (z * ny + y) * nx + x;
      uint32_t a[kBrickRun];
      if (n == kBrickRun) {
        load_run<T, kBrickRun>(row, a);
      } else {
#pragma unroll
        for (int j = 0; j < kBrickRun; ++j) a[j] = j < n ? row[j] : 0;
      }
#pragma unroll
      for (int l = 1; l < 16; ++l) {
        if (l >= n_lod) break;  // uniform
        const T* vl = (const T*)D.level[l] + ((z >> l) * D.dims[l][1] + (y >> l)) * D.dims[l][0];
        uint32_t last = 0;
        int64_t at = -1;
#pragma unroll
        for (int j = 0; j < kBrickRun; ++j) {
          if (j < n) {
            const int64_t q = (x + j) >> l;
            if (q != at) {  // the run's voxels share most ancestors
              last = vl[q];
              at = q;
            }
            acc[l] += (uint32_t)abs((int)a[j] - (int)last);
          }
        }
      }
    }
  }
#pragma unroll
  for (int l = 1; l < 16; ++l) {
    if (l >= n_lod) break;
    unsigned long long s = acc[l];
    for (int off = 32; off > 0; off >>= 1) s += __shfl_xor(s, off, 64);
    if ((threadIdx.x & 63) == 0) atomicAdd(&red[l], s);
  }
  __syncthreads();
  if (threadIdx.x > 0 && threadIdx.x < (unsigned)n_lod)
    atomicAdd(&sums[(int64_t)reg * n_lod + threadIdx.x], red[threadIdx.x]);
}

// out[region * n_lod + l] = sum / voxels of the region
__global__ __launch_bounds__(kThreads) void region_detail_mean_kernel(const unsigned long long* __restrict__ sums,
                                                                      int64_t n, int n_lod, int64_t nx, int64_t ny,
                                                                      int64_t nz, int B, int gx, int gy,
                                                                      float* __restrict__ out) {
  const int64_t i = (int64_t)blockIdx.x * kThreads + threadIdx.x;
  if (i >= n) return;
  const int reg = (int)(i / n_lod);
  const int bx = reg % gx, by = (reg / gx) % gy, bz = reg / (gx * gy);
  const int64_t w = min<int64_t>(B, nx - (int64_t)bx * B), h = min<int64_t>(B, ny - (int64_t)by * B),
                d = min<int64_t>(B, nz - (int64_t)bz * B);
  out[i] = (float)((double)sums[i] / (double)max<int64_t>(w * h * d, 1));
}

hipError_t launch_region_detail(const void* const* levels, const int64_t (*dims)[3], int n_lod, int bpv,
                                int B, unsigned long long* sums, float* out, hipStream_t stream) {
  DetailLevels D{};
  for (int l = 0; l < n_lod && l < 16; ++l) {
    D.level[l] = levels[l];
    for (int i = 0; i < 3; ++i) D.dims[l][i] = dims[l][i];
  }
  const int gx = (int)((dims[0][0] + B - 1) / B), gy = (int)((dims[0][1] + B - 1) / B),
            gz = (int)((dims[0][2] + B - 1) / B);
  const int64_t regions = (int64_t)gx * gy * gz, n = regions * n_lod;
  if (hipError_t e = launch_fill_u64(sums, n, 0ull, stream)) return e;
  const dim3 grid((unsigned)regions, brick_parts(regions, B), 1);
  if (bpv == 1)
    region_detail_kernel<uint8_t><<<grid, kThreads, 0, stream>>>(D, n_lod, B, gx, gy, sums);
  else
    region_detail_kernel<uint16_t><<<grid, kThreads, 0, stream>>>(D, n_lod, B, gx, gy, sums);
  if (hipError_t e = hipGetLastError()) return e;
  region_detail_mean_kernel<<<(unsigned)((n + kThreads - 1) / kThreads), kThreads, 0, stream>>>(
      sums, n, n_lod, dims[0][0], dims[0][1], dims[0][2], B, gx, gy, out);
  return hipGetLastError();
}

hipError_t launch_brick_histograms(const void* level, int bpv, const int64_t d[3], int B, int bins,
                                   uint32_t* out, hipStream_t stream) {
  const int gx = (int)((d[0] + B - 1) / B), gy = (int)((d[1] + B - 1) / B),
            gz = (int)((d[2] + B - 1) / B);
  int shift = 0;
  while ((1 << (8 * bpv - shift)) > bins) ++shift;
  const int64_t bricks = (int64_t)gx * gy * gz, n = bricks * bins;
  fill_u32_kernel<<<(unsigned)std::min<int64_t>((n + kThreads - 1) / kThreads, 65536), kThreads, 0, stream>>>(out, n,
                                                                                                             0u);
  if (hipError_t e = hipGetLastError()) return e;
  const dim3 grid((unsigned)bricks, brick_parts(bricks, B), 1);
  if (bpv == 1)
    brick_hist_kernel<uint8_t><<<grid, kThreads, 0, stream>>>((const uint8_t*)level, d[0], d[1], d[2],
                                                               B, gx, gy, bins, shift, out);
  else
    brick_hist_kernel<uint16_t><<<grid, kThreads, 0, stream>>>((const uint16_t*)level, d[0], d[1],
                                                                d[2], B, gx, gy, bins, shift, out);
  return hipGetLastError();
}

hipError_t launch_histogram_1d(const void* vol, int bpv, int64_t n, unsigned long long* hist,
                               hipStream_t stream) {
  const int64_t nb = bpv == 1 ? 256 : 65536;
  hipError_t e = launch_fill_u64(hist, nb, 0ull, stream);
  if (e != hipSuccess) return e;
  int64_t blocks = (n + kThreads * 16 - 1) / (kThreads * 16);
  if (blocks > 8192) blocks = 8192;
  if (blocks < 1) blocks = 1;
  if (bpv == 1) {
    const int64_t groups = std::min<int64_t>((n + kThreads * 16 - 1) / (kThreads * 16), 2048);
    hist1d_u8_kernel<<<(unsigned)groups, kThreads, 0, stream>>>((const uint8_t*)vol, n, hist);
    return hipGetLastError();
  }
  const size_t lds = 65536 * 2;
  if (lds_allowed(hist1d_u16_lds_kernel, lds)) {
    // A group per pass of 8192 voxels up to a quarter of the CUs, then four
    // passes a group: a group adds each of its distinct values to the global
    // bins, as many as its voxels where they hardly repeat.  128^3 voxels of
    // noise take 113 us with a group per pass and 88 so, a smooth field 100
    // and 84, a scan 72 and 75, values that share few bins 58 and 64.
    const int64_t cus = device_cus(), passes = (n + kHistThreads * kRunX - 1) / (kHistThreads * kRunX);
    const int64_t groups = std::min(cus, std::max(std::min(passes, cus / 4), passes / 4));
    hist1d_u16_lds_kernel<<<(unsigned)groups, kHistThreads, lds, stream>>>((const uint16_t*)vol, n, hist);
    if (hipGetLastError() == hipSuccess) return hipSuccess;
  }
  hist1d_u16_kernel<<<(unsigned)blocks, kThreads, 0, stream>>>((const uint16_t*)vol, n, hist);
  return hipGetLastError();
}

hipError_t launch_gradient_kmax(const void* vol, int bpv, const int64_t d[3],
                                unsigned long long* kmax, hipStream_t stream) {
  hipError_t e = launch_fill_u64(kmax, 1, 0ull, stream);
  if (e != hipSuccess) return e;
  const RunWalk W = run_walk(d[0], kThreads);
  const int64_t runs = (d[0] + kRunX - 1) / kRunX, passes = (d[1] * d[2] + W.rows - 1) / W.rows;
  const dim3 grid((unsigned)((runs + W.spw - 1) / W.spw), (unsigned)std::min<int64_t>(passes, 8192), 1);
  if (bpv == 1)
    gradient_kmax_kernel<uint8_t><<<grid, kThreads, 0, stream>>>((const uint8_t*)vol, d[0], d[1],
                                                                 d[2], kmax);
  else
    gradient_kmax_kernel<uint16_t><<<grid, kThreads, 0, stream>>>((const uint16_t*)vol, d[0],
                                                                  d[1], d[2], kmax);
  return hipGetLastError();
}

hipError_t launch_histogram_2d(const void* vol, int bpv, const int64_t d[3],
                               const unsigned long long* kmax, int n_value, int n_grad,
                               unsigned long long* hist, hipStream_t stream) {
  hipError_t e = launch_fill_u64(hist, (int64_t)n_value * n_grad, 0ull, stream);
  if (e != hipSuccess) return e;
  int shift = 0;
  while (((int64_t)n_value << shift) < ((int64_t)1 << (8 * bpv))) ++shift;
  // privatised in LDS when the bins fit 128 KiB
  const int64_t nbins = (int64_t)n_value * n_grad;
  const size_t lds = (size_t)((nbins / 2 + 1) & ~1ll) * 4 + (n_grad <= kHistThresholds ? (size_t)n_grad * 8 : 0);
  if (nbins % 2 == 0 && nbins <= 65536) {
    const RunWalk W = run_walk(d[0], kHistThreads);
    const int64_t xs = (int64_t)W.spw * kRunX;
    const int64_t passes = (d[1] * d[2] + W.rows - 1) / W.rows * ((d[0] + xs - 1) / xs);
    const unsigned groups = (unsigned)std::min<int64_t>(device_cus(), passes);
    bool ok = false;
    if (bpv == 1 && lds_allowed(hist2d_lds_kernel<uint8_t>, lds)) {
      hist2d_lds_kernel<uint8_t><<<groups, kHistThreads, lds, stream>>>(
          (const uint8_t*)vol, d[0], d[1], d[2], kmax, shift, n_grad, (int)nbins, hist);
      ok = hipGetLastError() == hipSuccess;
    } else if (bpv == 2 && lds_allowed(hist2d_lds_kernel<uint16_t>, lds)) {
      hist2d_lds_kernel<uint16_t><<<groups, kHistThreads, lds, stream>>>(
          (const uint16_t*)vol, d[0], d[1], d[2], kmax, shift, n_grad, (int)nbins, hist);
      ok = hipGetLastError() == hipSuccess;
    }
    if (ok) return hipSuccess;
  }
  const dim3 grid = row_grid(d[0], d[1] * d[2]);
  if (bpv == 1)
    hist2d_kernel<uint8_t><<<grid, kThreads, 0, stream>>>((const uint8_t*)vol, d[0], d[1], d[2],
                                                          kmax, shift, n_grad, hist);
  else
    hist2d_kernel<uint16_t><<<grid, kThreads, 0, stream>>>((const uint16_t*)vol, d[0], d[1], d[2],
                                                           kmax, shift, n_grad, hist);
  return hipGetLastError();
}

}  // namespace tvk
