// transform_data gather: border-clamped linear / bilinear / trilinear sampling
// and its backward (cpab/pytorch/interpolation.py:3-159 plus the torch
// autograd backward of those ops).
//
// Index conventions of the reference: grid coordinate k scales by
// (data.shape[2+k] - 1) and indexes data axis 2+k; the warped grid lists points
// with coordinate 0 fastest, p = i0 + o0*(i1 + o1*i2); the output is
// [B, C, o0, o1(, o2)] with the LAST axis fastest.  So the point order and the
// output order are transposes of each other.  HBM-bound, so each workgroup
// takes a kT0 x kTL tile over (i0, i_last) at fixed i_mid, reads the grid rows
// coalesced along i0 into LDS, and computes/writes with i_last across the
// lanes (whole 128-byte output lines and, for smooth warps, near-contiguous
// data rows).
// The backward does the same transpose in the other direction for grad_grid.
// The per-sample arithmetic lives in cpab_sample.hpp.
#include <hip/hip_runtime.h>
#include <limits.h>
#include <math.h>
#include <algorithm>
#include "cpab_launch.hpp"
#include "cpab_sample.hpp"

namespace cpab {
namespace {

constexpr int kT0 = kInterpTile0;      // tile extent along i0 (grid rows are contiguous in i0)
constexpr int kTL = kInterpTileLast;   // tile extent along i_last (output rows are contiguous in i_last)
constexpr int kThreads = kInterpThreads;
constexpr int kLogT0 = 5, kLogTL = 5;
static_assert(kT0 == 1 << kLogT0 && kTL == 1 << kLogTL, "tile extents");
static_assert(kThreads % kTL == 0 && kT0 % 4 == 0 && 64 % kTL == 0 && kT0 % (kThreads / kTL) == 0,
              "tile shape");
constexpr int kRows = kThreads / kTL;   // tile rows (along i0) a workgroup covers per pass
constexpr int kPerLane = kT0 / kRows;   // outputs per lane in a whole tile
// Outputs per lane whose gathers the backward issues together (4 corner-pair
// loads in flight per lane).  Larger batches cost occupancy: with the pairs,
// batches of 4 (2D) and 2 (3D) ran the C3 backward 14% and the C4 backward 8%
// slower.
constexpr int gather_batch(int nd) { return nd == 3 ? 1 : 2; }
static_assert(kPerLane % gather_batch(2) == 0 && kPerLane % gather_batch(3) == 0, "batches");
constexpr int kXcds = 8;     // MI355X: accelerator complex dies, each with its own L2

struct Shape {
  int ndim;
  int B, C;
  int in[3];     // data spatial sizes
  int o0, omid, olast;
  int64_t nP;
  int vec4;      // grid rows are 16-byte aligned along i0 (o0 % 4 == 0)
  int tiles0, tilesm, tilesl;  // tiles along i0, i_mid and i_last
  int log0, logm, logl;        // log2 of a tile's extent along each
};

// Tiles of a launch, padded to the same number for each XCD.
__host__ __device__ inline int64_t padded_tiles(const Shape& s) {
  const int64_t total = (int64_t)s.tiles0 * s.tilesl * s.B * s.tilesm;
  return (total + kXcds - 1) / kXcds * kXcds;
}

// Tile of workgroup wg, XCD-aware.  The hardware hands consecutive
// workgroup ids to the 8 XCDs in turn, and each XCD has its own L2; the
// remap gives XCD x the x-th eighth of the tile list, so an XCD works through
// whole images (tiles ordered i0 tile, then i_last tile, then i_mid tile and b)
// and the gathers of one image share that XCD's L2.  Returns false for the
// padding workgroups past the last tile.
__device__ __forceinline__ bool tile_origin(const Shape& s, int64_t wg, int& b, int& im, int& t0,
                                            int& tl) {
  const int64_t total = (int64_t)s.tiles0 * s.tilesl * s.B * s.tilesm;
  const int64_t per = (total + kXcds - 1) / kXcds;
  const int64_t n = (wg % kXcds) * per + wg / kXcds;
  if (n >= total) return false;
  const int64_t plane = (int64_t)s.tiles0 * s.tilesl;
  const int64_t z = n / plane;
  const int r = (int)(n - z * plane);
  const int ty = r / s.tiles0;
  b = (int)(z / s.tilesm);
  im = (int)(z - (int64_t)b * s.tilesm) << s.logm;
  t0 = (r - ty * s.tiles0) << s.log0;
  tl = ty << s.logl;
  return true;
}

// Grid rows of this tile -> LDS crd[k][al][a0] (lanes along i0, float4 when aligned).
template <int ND>
__device__ __forceinline__ void load_tile(const Shape& s, const float* __restrict__ grid, int b,
                                          int im, int t0, int tl, int n0, int nl,
                                          float (*crd)[kTL][kT0 + 1], int threads = kThreads) {
  const int64_t row0 = (int64_t)s.o0 * (im + (int64_t)s.omid * tl) + t0;  // point of (t0, tl)
  const int64_t rstride = (int64_t)s.o0 * s.omid;                        // next i_last
  if (s.vec4 && n0 == kT0) {
    constexpr int Q = kT0 / 4;
    for (int e = threadIdx.x; e < Q * kTL; e += threads) {
      const int q = e % Q, al = e / Q;
      if (al < nl) {
#pragma unroll
        for (int k = 0; k < ND; ++k) {
          const float4 v = *reinterpret_cast<const float4*>(
              grid + ((int64_t)b * ND + k) * s.nP + row0 + al * rstride + 4 * q);
          crd[k][al][4 * q] = v.x;
          crd[k][al][4 * q + 1] = v.y;
          crd[k][al][4 * q + 2] = v.z;
          crd[k][al][4 * q + 3] = v.w;
        }
      }
    }
  } else {
    for (int e = threadIdx.x; e < kT0 * kTL; e += threads) {
      const int a0 = e % kT0, al = e / kT0;
      if (a0 < n0 && al < nl) {
#pragma unroll
        for (int k = 0; k < ND; ++k)
          crd[k][al][a0] = grid[((int64_t)b * ND + k) * s.nP + row0 + al * rstride + a0];
      }
    }
  }
}

// The tile in crd -> grid rows (lanes along i0, float4 when aligned).
template <int ND>
__device__ __forceinline__ void store_tile(const Shape& s, float* __restrict__ grad_grid, int b,
                                           int im, int t0, int tl, int n0, int nl,
                                           const float (*crd)[kTL][kT0 + 1],
                                           int threads = kThreads) {
  const int64_t row0 = (int64_t)s.o0 * (im + (int64_t)s.omid * tl) + t0;
  const int64_t rstride = (int64_t)s.o0 * s.omid;
  if (s.vec4 && n0 == kT0) {
    constexpr int Q = kT0 / 4;
    for (int e = threadIdx.x; e < Q * kTL; e += threads) {
      const int q = e % Q, l = e / Q;
      if (l < nl) {
#pragma unroll
        for (int k = 0; k < ND; ++k) {
          float4 v;
          v.x = crd[k][l][4 * q];
          v.y = crd[k][l][4 * q + 1];
          v.z = crd[k][l][4 * q + 2];
          v.w = crd[k][l][4 * q + 3];
          *reinterpret_cast<float4*>(grad_grid + ((int64_t)b * ND + k) * s.nP + row0 + l * rstride + 4 * q) = v;
        }
      }
    }
  } else {
    for (int e = threadIdx.x; e < kT0 * kTL; e += threads) {
      const int a0 = e % kT0, l = e / kT0;
      if (a0 < n0 && l < nl) {
#pragma unroll
        for (int k = 0; k < ND; ++k)
          grad_grid[((int64_t)b * ND + k) * s.nP + row0 + l * rstride + a0] = crd[k][l][a0];
      }
    }
  }
}

template <int ND>
__global__ __launch_bounds__(kThreads) void interp_fwd_kernel(Shape s,
                                                              const float* __restrict__ data,
                                                              const float* __restrict__ grid,
                                                              float* __restrict__ out) {
  __shared__ float crd[ND][kTL][kT0 + 1];
  int b, im, t0, tl;
  if (!tile_origin(s, blockIdx.x, b, im, t0, tl)) return;
  const int n0 = min(kT0, s.o0 - t0), nl = min(kTL, s.olast - tl);
  load_tile<ND>(s, grid, b, im, t0, tl, n0, nl, crd);
  __syncthreads();
  const int al = threadIdx.x % kTL;   // lanes along i_last
  const int w = threadIdx.x / kTL;    // kRows rows at a time
  const int64_t plane_in = (int64_t)s.in[0] * s.in[1] * (ND == 3 ? s.in[2] : 1);
  const int64_t plane_out = (int64_t)s.o0 * s.omid * s.olast;
  const int64_t ostride = (int64_t)s.omid * s.olast;   // next i0 in the output
  const bool pairs = s.in[ND - 1] >= 2;                // corners read in pairs
  if (al >= nl) return;
  if (n0 == kT0) {
    // Whole tile along i0, software-pipelined: the corner loads of a lane's
    // next output are issued before the current output is blended and stored.
    for (int ch = 0; ch < s.C; ++ch) {
      const int64_t bc = (int64_t)b * s.C + ch;
      const ChannelBuf d(data + bc * plane_in, plane_in);
      float* __restrict__ o = out + bc * plane_out + (int64_t)(t0 + w) * ostride +
                              (int64_t)im * s.olast + tl + al;
      Axis ax[2], ay[2], az[2];
      float c[2][1 << ND];
#pragma unroll
      for (int j = -1; j < kPerLane; ++j) {
        if (j + 1 < kPerLane) {
          const int n = (j + 1) & 1;
          const int a0 = w + (j + 1) * kRows;
          ax[n] = axis_of(crd[0][al][a0], s.in[0]);
          ay[n] = axis_of(crd[1][al][a0], s.in[1]);
          az[n] = ND == 3 ? axis_of(crd[ND - 1][al][a0], s.in[2]) : Axis{0, 0, 0.0f};
          if (pairs) gather_pairs<ND>(s.in, d, ax[n], ay[n], az[n], c[n]);
          else gather<ND>(s.in, d, ax[n], ay[n], az[n], c[n]);
        }
        __builtin_amdgcn_sched_barrier(0);
        if (j >= 0) {
          const int k = j & 1;
          o[j * kRows * ostride] = blend<ND>(c[k], ax[k], ay[k], az[k]);
        }
      }
    }
    return;
  }
  for (int ch = 0; ch < s.C; ++ch) {
    const int64_t bc = (int64_t)b * s.C + ch;
    const float* __restrict__ d = data + bc * plane_in;
    float* __restrict__ o = out + bc * plane_out + (int64_t)im * s.olast + tl + al;
    for (int a0 = w; a0 < n0; a0 += kRows) {
      const Axis ax = axis_of(crd[0][al][a0], s.in[0]);
      const Axis ay = axis_of(crd[1][al][a0], s.in[1]);
      const Axis az = ND == 3 ? axis_of(crd[ND - 1][al][a0], s.in[2]) : Axis{0, 0, 0.0f};
      o[(int64_t)(t0 + a0) * ostride] = sample<ND>(s.in, d, ax, ay, az);
    }
  }
}

// grad_grid (the gradient of the coordinates).
template <int ND>
__global__ __launch_bounds__(kThreads) void interp_bwd_kernel(Shape s,
                                                              const float* __restrict__ data,
                                                              const float* __restrict__ grid,
                                                              const float* __restrict__ grad_out,
                                                              float* __restrict__ grad_grid) {
  __shared__ float crd[ND][kTL][kT0 + 1];
  int b, im, t0, tl;
  if (!tile_origin(s, blockIdx.x, b, im, t0, tl)) return;
  const int n0 = min(kT0, s.o0 - t0), nl = min(kTL, s.olast - tl);
  load_tile<ND>(s, grid, b, im, t0, tl, n0, nl, crd);
  __syncthreads();
  const int al = threadIdx.x % kTL;
  const int w = threadIdx.x / kTL;
  const int64_t plane_in = (int64_t)s.in[0] * s.in[1] * (ND == 3 ? s.in[2] : 1);
  const int64_t plane_out = (int64_t)s.o0 * s.omid * s.olast;
  const bool pairs = s.in[ND - 1] >= 2;   // corners read in pairs
  if (al < nl && n0 == kT0) {
    // Whole tile along i0: the gathers of gather_batch outputs of a lane
    // overlap.
    constexpr int NB = gather_batch(ND);
#pragma unroll
    for (int j0 = 0; j0 < kPerLane; j0 += NB) {
      Axis ax[NB], ay[NB], az[NB];
      float dd[NB][3];
#pragma unroll
      for (int j = 0; j < NB; ++j) {
        const int a0 = w + (j0 + j) * kRows;
        ax[j] = axis_of(crd[0][al][a0], s.in[0]);
        ay[j] = axis_of(crd[1][al][a0], s.in[1]);
        az[j] = ND == 3 ? axis_of(crd[ND - 1][al][a0], s.in[2]) : Axis{0, 0, 0.0f};
        dd[j][0] = dd[j][1] = dd[j][2] = 0.0f;
      }
      const int64_t o = ((int64_t)(t0 + w + j0 * kRows) * s.omid + im) * s.olast + tl + al;
      for (int ch = 0; ch < s.C; ++ch) {
        const int64_t bc = (int64_t)b * s.C + ch;
        const ChannelBuf d(data + bc * plane_in, plane_in);
        const float* __restrict__ go = grad_out + bc * plane_out + o;
        float g[NB], c[NB][1 << ND];
#pragma unroll
        for (int j = 0; j < NB; ++j) {
          if (pairs) gather_pairs<ND>(s.in, d, ax[j], ay[j], az[j], c[j]);
          else gather<ND>(s.in, d, ax[j], ay[j], az[j], c[j]);
        }
#pragma unroll
        for (int j = 0; j < NB; ++j) g[j] = go[(int64_t)j * kRows * s.omid * s.olast];
        // keeps the batch's loads issued before the first use of one
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int j = 0; j < NB; ++j) blend_grad<ND>(c[j], ax[j], ay[j], az[j], g[j], dd[j]);
      }
      // (size-1) chain factor of x = g*(size-1); each thread rewrites only
      // the LDS slots it read.
#pragma unroll
      for (int j = 0; j < NB; ++j)
#pragma unroll
        for (int k = 0; k < ND; ++k)
          crd[k][al][w + (j0 + j) * kRows] = dd[j][k] * (float)(s.in[k] - 1);
    }
  } else if (al < nl) {
    for (int a0 = w; a0 < n0; a0 += kRows) {
      const Axis ax = axis_of(crd[0][al][a0], s.in[0]);
      const Axis ay = axis_of(crd[1][al][a0], s.in[1]);
      const Axis az = ND == 3 ? axis_of(crd[ND - 1][al][a0], s.in[2]) : Axis{0, 0, 0.0f};
      const int64_t o = ((int64_t)(t0 + a0) * s.omid + im) * s.olast + tl + al;
      float dd[3] = {0.0f, 0.0f, 0.0f};
      for (int ch = 0; ch < s.C; ++ch) {
        const int64_t bc = (int64_t)b * s.C + ch;
        float c[1 << ND];
        gather<ND>(s.in, ChannelPtr{data + bc * plane_in}, ax, ay, az, c);
        blend_grad<ND>(c, ax, ay, az, grad_out[bc * plane_out + o], dd);
      }
#pragma unroll
      for (int k = 0; k < ND; ++k) crd[k][al][a0] = dd[k] * (float)(s.in[k] - 1);
    }
  }
  __syncthreads();
  store_tile<ND>(s, grad_grid, b, im, t0, tl, n0, nl, crd);
}

// grad_data of 2D / 3D resampling: every output adds its gradient, times each
// corner's weight, to the data positions around its coordinate.
//
// Bound by atomics: a float add to HBM costs a request per 64-byte row it
// touches (20 G/s measured; a coalesced wave adds 320 G floats/s).  So a
// workgroup takes a tile of 1024 outputs, adds its corners in an LDS box
// over the data positions the tile reaches and adds the box to HBM row by row,
// lanes along the data's contiguous axis: one coalesced add per data position
// instead of 2^ND scattered ones per output.  The box is in double because
// ds_add_f64 takes 9 cycles for a wave of distinct addresses and ds_add_f32
// 194 (3 per active lane).  A tile whose box exceeds kBoxMax (the warp
// stretches it, or the data is much finer than the output) adds its corners to
// HBM directly.  8 x 3 x 384 x 384 outputs whose positions scatter by 4 pixels:
// 48 us here (93 with a float box of 5,120 positions), 482 with every corner
// added to HBM from the gather kernel; 8 x 3 x 225 x 227 smoothly warped
// outputs: 14 us here (41 with the float box), 48 when the image backward added
// them.
// IMG: the coordinates are in output order (last axis fastest, the fused
// transform_data's final points; image_tile's tiles), else in grid order
// (coordinate 0 fastest; kT0 x kTL tiles of a slice, as the gather kernels).
// GRID: grad_grid too, with interp_bwd_kernel's arithmetic, before the box: one
// launch and one read of coordinates and gradients where both are wanted (32 x 28
// x 28 outputs, whole backward: 15.9 us as two kernels, 13.1 so; 16 x 512 x 512
// 86.0 and 80.5; 128^3 68.8 and 67.4).  At least four waves per SIMD: with the 131
// registers that 3D takes unbounded one workgroup fits a CU (128^3: 86.8 us).
// FEW: no tile of the launch has more than kScatterFew outputs (thin or small
// images): every corner goes to HBM, coordinates and grad_grid past LDS, in
// workgroups of the tile's size (64 x 8 x 8 outputs 11.4 us with the box, 9.1 so;
// 16 x 4 x 300 x 4 116 and 41; 100 x 16 x 16 12.2 and 10.2).
constexpr int kScatterThreads = 512;
constexpr int kScatterLog = 10;                       // log2 of a tile's outputs
constexpr int kScatterPer = (1 << kScatterLog) / kScatterThreads;   // outputs per lane
static_assert(kT0 * kTL == 1 << kScatterLog, "grid-order tiles");
constexpr int kBoxMax = 10000;   // doubles: 80 KB, two workgroups per CU
constexpr int kScatterFew = 256;

struct BoxSink {
  double* box;
  __device__ __forceinline__ void add(int i, float v) const {
    __hip_atomic_fetch_add(box + i, (double)v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
  }
};

template <int ND, bool IMG, bool GRID, bool FEW>
__device__ __forceinline__ void scatter_tile(const Shape& s, int64_t wg,
                                             const float* __restrict__ data,
                                             const float* __restrict__ coords,
                                             const float* __restrict__ grad_out,
                                             float* __restrict__ grad_grid,
                                             float* __restrict__ grad_data, double* box) {
  static_assert(!(IMG && GRID), "grad_grid is in grid order");
  const int threads = FEW ? (int)blockDim.x : kScatterThreads;
  __shared__ int lo[3], hi[3];
  float(*crd)[kTL][kT0 + 1] = reinterpret_cast<float(*)[kTL][kT0 + 1]>(box);
  int b, im, t0, tl;
  if (!tile_origin(s, wg, b, im, t0, tl)) return;
  const int n0 = min(1 << s.log0, s.o0 - t0), nm = min(1 << s.logm, s.omid - im);
  const int nl = min(1 << s.logl, s.olast - tl);
  if (threadIdx.x < 3) {
    lo[threadIdx.x] = INT_MAX;
    hi[threadIdx.x] = -1;
  }
  if constexpr (!FEW) {
    if constexpr (!IMG) load_tile<ND>(s, coords, b, im, t0, tl, n0, nl, crd, kScatterThreads);
    __syncthreads();
  }
  const int64_t plane_in = (int64_t)s.in[0] * s.in[1] * (ND == 3 ? s.in[2] : 1);
  const int64_t plane_out = (int64_t)s.o0 * s.omid * s.olast;

  // This lane's outputs (consecutive lanes along i_last), and the data positions
  // they reach.
  Axis at[ND][kScatterPer];
  bool live[kScatterPer];
  int64_t o[kScatterPer];   // their indices in an output plane
  const auto grid_at = [&](int al, int a0) {   // and in grid order
    return t0 + a0 + (int64_t)s.o0 * (im + (int64_t)s.omid * (tl + al));
  };
  int mn[ND], mx[ND];
#pragma unroll
  for (int k = 0; k < ND; ++k) {
    mn[k] = INT_MAX;
    mx[k] = -1;
  }
#pragma unroll
  for (int j = 0; j < kScatterPer; ++j) {
    const int e = threadIdx.x + j * threads;
    const int al = e & ((1 << s.logl) - 1), r = e >> s.logl;
    const int am = r & ((1 << s.logm) - 1), a0 = r >> s.logm;
    live[j] = al < nl && am < nm && a0 < n0;
    o[j] = ((int64_t)(t0 + a0) * s.omid + im + am) * s.olast + tl + al;
#pragma unroll
    for (int k = 0; k < ND; ++k) {
      float x = 0.0f;
      if (live[j]) {
        if constexpr (IMG) x = coords[((int64_t)b * ND + k) * s.nP + o[j]];
        else if constexpr (FEW) x = coords[((int64_t)b * ND + k) * s.nP + grid_at(al, a0)];
        else x = crd[k][al][a0];
      }
      at[k][j] = axis_of(x, s.in[k]);
      if (live[j]) {
        mn[k] = min(mn[k], at[k][j].i0);
        mx[k] = max(mx[k], at[k][j].i1);
      }
    }
  }
  const Axis none{0, 0, 0.0f};
  if constexpr (!FEW) {
#pragma unroll
    for (int k = 0; k < ND; ++k) {
#pragma unroll
      for (int off = 32; off >= 1; off >>= 1) {
        mn[k] = min(mn[k], __shfl_xor(mn[k], off));
        mx[k] = max(mx[k], __shfl_xor(mx[k], off));
      }
      if ((threadIdx.x & 63) == 0) {
        atomicMin(&lo[k], mn[k]);
        atomicMax(&hi[k], mx[k]);
      }
    }
    __syncthreads();
  }
  if constexpr (GRID) {
    float dd[kScatterPer][3] = {};
    for (int ch = 0; ch < s.C; ++ch) {
      const int64_t bc = (int64_t)b * s.C + ch;
      const ChannelBuf d(data + bc * plane_in, plane_in);
#pragma unroll
      for (int j = 0; j < kScatterPer; ++j) {
        float c[1 << ND];
        const Axis az = ND == 3 ? at[ND - 1][j] : none;
        gather<ND>(s.in, d, at[0][j], at[1][j], az, c);
        const float g = live[j] ? grad_out[bc * plane_out + o[j]] : 0.0f;
        blend_grad<ND>(c, at[0][j], at[1][j], az, g, dd[j]);
      }
    }
    // The coordinates' slots take their gradients (each lane its own).
#pragma unroll
    for (int j = 0; j < kScatterPer; ++j) {
      if (!live[j]) continue;
      const int e = threadIdx.x + j * threads, al = e & ((1 << s.logl) - 1), a0 = e >> s.logl;
#pragma unroll
      for (int k = 0; k < ND; ++k) {
        const float v = dd[j][k] * (float)(s.in[k] - 1);
        if constexpr (FEW) grad_grid[((int64_t)b * ND + k) * s.nP + grid_at(al, a0)] = v;
        else crd[k][al][a0] = v;
      }
    }
    if constexpr (!FEW) {
      __syncthreads();
      store_tile<ND>(s, grad_grid, b, im, t0, tl, n0, nl, crd, kScatterThreads);
      __syncthreads();   // the box may take their place
    }
  }
  int org[3] = {0, 0, 0}, ext[3] = {1, 1, 1};
  int64_t area = FEW ? INT64_MAX : 1;
  if constexpr (!FEW) {
#pragma unroll
    for (int k = 0; k < ND; ++k) {
      org[k] = __builtin_amdgcn_readfirstlane(lo[k]);
      ext[k] = __builtin_amdgcn_readfirstlane(hi[k]) - org[k] + 1;
      area *= ext[k];
    }
  }
  if (area > kBoxMax) {   // uniform over the workgroup
    for (int ch = 0; ch < s.C; ++ch) {
      const int64_t bc = (int64_t)b * s.C + ch;
#pragma unroll
      for (int j = 0; j < kScatterPer; ++j) {
        if (!live[j]) continue;
        scatter_to<ND>(s.in, FloatScatter{grad_data + bc * plane_in}, at[0][j], at[1][j],
                       ND == 3 ? at[ND - 1][j] : none,
                       grad_out[bc * plane_out + o[j]]);
      }
    }
    return;
  }
#pragma unroll
  for (int k = 0; k < ND; ++k)
#pragma unroll
    for (int j = 0; j < kScatterPer; ++j) {
      at[k][j].i0 -= org[k];
      at[k][j].i1 -= org[k];
    }
  for (int i = threadIdx.x; i < (int)area; i += kScatterThreads) box[i] = 0.0;
  const int rows = (int)area / ext[ND - 1];
  const int64_t base = ND == 2 ? (int64_t)org[0] * s.in[1] + org[1]
                               : ((int64_t)org[0] * s.in[1] + org[1]) * s.in[2] + org[2];
  for (int ch = 0; ch < s.C; ++ch) {
    const int64_t bc = (int64_t)b * s.C + ch;
    float g[kScatterPer];
#pragma unroll
    for (int j = 0; j < kScatterPer; ++j)
      g[j] = live[j] ? grad_out[bc * plane_out + o[j]] : 0.0f;
    __syncthreads();   // the box is clear
#pragma unroll
    for (int j = 0; j < kScatterPer; ++j)
      if (live[j])
        scatter_to<ND>(ext, BoxSink{box}, at[0][j], at[1][j], ND == 3 ? at[ND - 1][j] : none, g[j]);
    __syncthreads();
    // Half a wave per box row; each slot is cleared for the next channel.
    float* __restrict__ gd = grad_data + bc * plane_in + base;
    for (int r = threadIdx.x / 32; r < rows; r += kScatterThreads / 32) {
      const int64_t row = ND == 2 ? (int64_t)r * s.in[1]
                                  : ((int64_t)(r / ext[1]) * s.in[1] + r % ext[1]) * s.in[2];
      for (int c = threadIdx.x % 32; c < ext[ND - 1]; c += 32) {
        const float v = (float)box[r * ext[ND - 1] + c];
        box[r * ext[ND - 1] + c] = 0.0;
        if (v != 0.0f) unsafeAtomicAdd(gd + row + c, v);
      }
    }
  }
}

// One workgroup per tile up to kScatterGrid workgroups; a launch of more tiles
// (thin volumes in a large batch) walks them in strides of the grid, which
// would otherwise pass HIP's limit of 2^32 lanes.
constexpr int64_t kScatterGrid = 1 << 22;   // a multiple of kXcds

template <int ND, bool IMG, bool GRID, bool FEW>
__global__ __launch_bounds__(kScatterThreads, 4) void scatter_kernel(
    Shape s, const float* __restrict__ data, const float* __restrict__ coords,
    const float* __restrict__ grad_out, float* __restrict__ grad_grid,
    float* __restrict__ grad_data) {
  extern __shared__ __align__(16) double box[];   // kBoxMax; first the tile's coordinates
  for (int64_t wg = blockIdx.x; wg < padded_tiles(s); wg += gridDim.x) {
    scatter_tile<ND, IMG, GRID, FEW>(s, wg, data, coords, grad_out, grad_grid, grad_data, box);
    __syncthreads();   // the next tile takes the box
  }
}

// 1D: point order equals output order, one thread per (b, point).
__global__ __launch_bounds__(kThreads) void interp1d_fwd_kernel(int B, int C, int W, int64_t nP,
                                                                const float* __restrict__ data,
                                                                const float* __restrict__ grid,
                                                                float* __restrict__ out) {
  for (int64_t e = blockIdx.x * (int64_t)kThreads + threadIdx.x; e < (int64_t)B * nP;
       e += (int64_t)gridDim.x * kThreads) {
    const int64_t b = e / nP, p = e - b * nP;
    const Axis ax = axis_of(grid[e], W);
    for (int ch = 0; ch < C; ++ch) {
      const float* d = data + (b * C + ch) * W;
      out[(b * C + ch) * nP + p] = lerp_ref(load_at(d, ax.i0), load_at(d, ax.i1), ax.t);
    }
  }
}

// grad_grid and grad_data (zero before), whichever are wanted, in one pass over
// the points: a second launch with the coordinates and gradients read again took
// 1.8 us more (16 x 10,000 points, one channel: 10.3 us in all, 12.1 with two).
template <bool GRID, bool DATA>
__global__ __launch_bounds__(kThreads) void interp1d_bwd_kernel(int B, int C, int W, int64_t nP,
                                                                const float* __restrict__ data,
                                                                const float* __restrict__ grid,
                                                                const float* __restrict__ grad_out,
                                                                float* __restrict__ grad_grid,
                                                                float* __restrict__ grad_data) {
  const Axis none{0, 0, 0.0f};
  for (int64_t e = blockIdx.x * (int64_t)kThreads + threadIdx.x; e < (int64_t)B * nP;
       e += (int64_t)gridDim.x * kThreads) {
    const int64_t b = e / nP, p = e - b * nP;
    const Axis ax = axis_of(grid[e], W);
    float gx = 0.0f;
    for (int ch = 0; ch < C; ++ch) {
      const int64_t bc = b * C + ch;
      const float g = grad_out[bc * nP + p];
      if constexpr (GRID) {
        const float* d = data + bc * W;
        gx += g * (load_at(d, ax.i1) - load_at(d, ax.i0));
      }
      if constexpr (DATA)
        scatter_to<1>(nullptr, FloatScatter{grad_data + bc * W}, ax, none, none, g);
    }
    if constexpr (GRID) grad_grid[e] = gx * (float)(W - 1);
  }
}

Shape make_shape(int ndim, int64_t B, int64_t C, const int64_t* in_size, const int64_t* out_size) {
  Shape s{};
  s.vec4 = 0;
  s.ndim = ndim;
  s.B = (int)B;
  s.C = (int)C;
  for (int k = 0; k < 3; ++k) s.in[k] = k < ndim ? (int)in_size[k] : 1;
  s.o0 = (int)out_size[0];
  s.omid = ndim == 3 ? (int)out_size[1] : 1;
  s.olast = (int)out_size[ndim - 1];
  s.nP = 1;
  for (int k = 0; k < ndim; ++k) s.nP *= out_size[k];
  s.vec4 = (s.o0 % 4) == 0;
  s.tiles0 = (s.o0 + kT0 - 1) / kT0;
  s.tilesl = (s.olast + kTL - 1) / kTL;
  s.tilesm = s.omid;
  s.log0 = kLogT0;
  s.logl = kLogTL;
  return s;
}

int aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; }

dim3 tile_grid(const Shape& s) { return dim3((unsigned)padded_tiles(s)); }

// Tile of the scatter over an image or volume in output order: 32 x 32, in a
// volume 8 x 8 x 16, whose box holds 1.8 data positions for each output where
// 32 x 32 outputs of one slice reach 3.4 (whole pass, one channel, 112^3: 376 us in
// slices, 365 so, 377 with 8 x 16 x 8; three channels 423, 400, 414), longer along
// the other axes where the output is thinner (16 volumes of 4 x 300 x 4: 117 us with
// a workgroup for each slice's 16 outputs, 78 so).
void image_tile(Shape* s) {
  const int size[3] = {s->o0, s->omid, s->olast};
  int want[3] = {5, 0, 5}, most[3];
  if (s->ndim == 3) { want[0] = 3; want[1] = 3; want[2] = 4; }
  int bits = 0;
  for (int k = 0; k < 3; ++k) {
    most[k] = 0;
    while (most[k] < kScatterLog && (1 << most[k]) < size[k]) ++most[k];
    want[k] = std::min(want[k], most[k]);
    bits += want[k];
  }
  for (int k : {2, 0, 1})
    while (bits < kScatterLog && want[k] < most[k]) { ++want[k]; ++bits; }
  s->log0 = want[0];
  s->logm = want[1];
  s->logl = want[2] + (kScatterLog - bits);   // fewer outputs than a tile's
  s->tiles0 = ((s->o0 - 1) >> s->log0) + 1;
  s->tilesm = ((s->omid - 1) >> s->logm) + 1;
  s->tilesl = ((s->olast - 1) >> s->logl) + 1;
}

template <int ND, bool IMG, bool GRID>
hipError_t launch_scatter(Shape s, const float* data, const float* coords, const float* grad_out,
                          float* grad_grid, float* grad_data, hipStream_t st) {
  if (IMG) {
    image_tile(&s);
  } else {   // lanes for the outputs there are
    while (s.log0 > 0 && (1 << s.log0) >= 2 * s.o0) --s.log0;
    while (s.logl > 0 && (1 << s.logl) >= 2 * s.olast) --s.logl;
  }
  const int most = std::min(s.o0, 1 << s.log0) * std::min(s.omid, 1 << s.logm) *
                   std::min(s.olast, 1 << s.logl);   // outputs of a tile
  const int threads = std::min(std::max(1 << (s.log0 + s.logm + s.logl), 64), kScatterThreads);
  const dim3 grid((unsigned)std::min(padded_tiles(s), kScatterGrid));
  if (most <= kScatterFew) {
    hipLaunchKernelGGL((scatter_kernel<ND, IMG, GRID, true>), grid, dim3(threads), 0, st, s, data,
                       coords, grad_out, grad_grid, grad_data);
    return hipGetLastError();
  }
  constexpr size_t lds = kBoxMax * sizeof(double);
  static LdsAllowed allowed;
  auto kernel = scatter_kernel<ND, IMG, GRID, false>;
  const hipError_t e = allow_lds(reinterpret_cast<const void*>(kernel), lds, allowed);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(kernel, grid, dim3(kScatterThreads), lds, st, s, data, coords, grad_out,
                     grad_grid, grad_data);
  return hipGetLastError();
}

}  // namespace

hipError_t launch_interp_forward(int ndim, int64_t B, int64_t C, const int64_t* in_size,
                                 const int64_t* out_size, const float* data, const float* grid,
                                 float* out, hipStream_t st) {
  Shape s = make_shape(ndim, B, C, in_size, out_size);
  s.vec4 &= aligned16(grid);
  if (s.nP <= 0 || B <= 0) return hipSuccess;
  if (ndim == 1) {
    int64_t g = (B * s.nP + kThreads - 1) / kThreads;
    if (g > 65536) g = 65536;
    hipLaunchKernelGGL(interp1d_fwd_kernel, dim3((unsigned)g), dim3(kThreads), 0, st, s.B, s.C,
                       s.in[0], s.nP, data, grid, out);
  } else {
    if (ndim == 2)
      hipLaunchKernelGGL(interp_fwd_kernel<2>, tile_grid(s), dim3(kThreads), 0, st, s, data, grid, out);
    else
      hipLaunchKernelGGL(interp_fwd_kernel<3>, tile_grid(s), dim3(kThreads), 0, st, s, data, grid, out);
  }
  return hipGetLastError();
}

hipError_t launch_interp_backward(int ndim, int64_t B, int64_t C, const int64_t* in_size,
                                  const int64_t* out_size, const float* data, const float* grid,
                                  const float* grad_out, float* grad_grid, float* grad_data,
                                  hipStream_t st) {
  Shape s = make_shape(ndim, B, C, in_size, out_size);
  s.vec4 &= aligned16(grid) & (grad_grid == nullptr || aligned16(grad_grid));
  if (grad_data) {
    int64_t n = B * C;
    for (int k = 0; k < ndim; ++k) n *= in_size[k];
    hipError_t e = launch_fill(grad_data, n, 0.0f, st);
    if (e != hipSuccess) return e;
  }
  if (s.nP <= 0 || B <= 0) return hipSuccess;
  if (ndim == 1) {
    if (!grad_grid && !grad_data) return hipSuccess;
    const int64_t g = std::min<int64_t>((B * s.nP + kThreads - 1) / kThreads, 65536);
    auto kernel = grad_grid ? (grad_data ? interp1d_bwd_kernel<true, true> : interp1d_bwd_kernel<true, false>)
                            : interp1d_bwd_kernel<false, true>;
    hipLaunchKernelGGL(kernel, dim3((unsigned)g), dim3(kThreads), 0, st, s.B, s.C, s.in[0], s.nP,
                       data, grid, grad_out, grad_grid, grad_data);
  } else if (grad_grid && grad_data) {
    return ndim == 2 ? launch_scatter<2, false, true>(s, data, grid, grad_out, grad_grid, grad_data, st)
                     : launch_scatter<3, false, true>(s, data, grid, grad_out, grad_grid, grad_data, st);
  } else if (grad_data) {
    return ndim == 2
               ? launch_scatter<2, false, false>(s, nullptr, grid, grad_out, nullptr, grad_data, st)
               : launch_scatter<3, false, false>(s, nullptr, grid, grad_out, nullptr, grad_data, st);
  } else if (grad_grid) {
    hipLaunchKernelGGL(ndim == 2 ? interp_bwd_kernel<2> : interp_bwd_kernel<3>, tile_grid(s),
                       dim3(kThreads), 0, st, s, data, grid, grad_out, grad_grid);
  }
  return hipGetLastError();
}

hipError_t launch_image_scatter(int ndim, const ImageShape& img, int64_t n_batch,
                                const float* final_points, const float* grad_out,
                                float* grad_data, hipStream_t st) {
  if (img.nP <= 0 || n_batch <= 0) return hipSuccess;
  int64_t in_size[3], out_size[3];
  for (int k = 0; k < 3; ++k) {
    in_size[k] = img.in[k];
    out_size[k] = img.o[k];
  }
  const Shape s = make_shape(ndim, n_batch, img.C, in_size, out_size);
  if (ndim == 1) {
    const int64_t g = std::min<int64_t>((n_batch * s.nP + kThreads - 1) / kThreads, 65536);
    hipLaunchKernelGGL((interp1d_bwd_kernel<false, true>), dim3((unsigned)g), dim3(kThreads), 0, st,
                       s.B, s.C, s.in[0], s.nP, nullptr, final_points, grad_out, nullptr, grad_data);
  } else {
    return ndim == 2 ? launch_scatter<2, true, false>(s, nullptr, final_points, grad_out, nullptr,
                                                      grad_data, st)
                     : launch_scatter<3, true, false>(s, nullptr, final_points, grad_out, nullptr,
                                                      grad_data, st);
  }
  return hipGetLastError();
}

}  // namespace cpab
