// ss_kernels.hip -- gfx950 kernels for the slant-stack projector pair, its exact
// transpose, the FBP row filter, the fused EM epilogues and the ellipse phantoms.
//
// Arithmetic is FP32 with FP32 accumulation.  FP64 appears only in the plan (angle
// tables, exact sample ranges), in the knife-edge predicate fallback of the
// backprojection and in the EM log-likelihood sums.
#include <hip/hip_runtime.h>

#include <type_traits>

#include <algorithm>

#include "ss_kernels.h"
#include "ss_plan_logic.h"

#define SS_INV_FIX 2.3283064365386963e-10f  // 2^-32
#define SS_FIX_ONE_I64 ((int64_t)1 << 32)    // one cell in Q32.32

// =====================================================================================
// plan: exact per-ray sample ranges
// =====================================================================================

// ray_t == nullptr: the uniform detector grid.  Otherwise ray k sits at ray_t[k] (the
// arbitrary-mesh form) and its Q32.32 trajectory offset goes to ray_alpha[j][k].
__global__ __launch_bounds__(256) void k_plan_bounds(SSGeom g, const SSAngle* __restrict__ angles,
                                                     int2* __restrict__ bounds, int* __restrict__ irregular,
                                                     int* __restrict__ nirregular, int capacity,
                                                     const double* __restrict__ ray_t, int64_t* __restrict__ ray_alpha) {
  const int k = blockIdx.x * blockDim.x + threadIdx.x;
  const int j = blockIdx.y;
  if (k >= g.nrays) return;
  const SSAngle a = angles[j];
  const SSTraj tr = ss_trajectory(g, a);
  int lo, hi, irr;
  if (ray_t) {
    const double t = ray_t[k];
    const double u0 = ss_ray_alpha(g, a, t);
    ray_alpha[(size_t)j * g.nrays + k] = __double2ll_rn(u0 * SS_FIX_ONE);
    irr = ss_ray_range_t(g, a, tr.beta, t, u0, &lo, &hi);
  } else {
    irr = ss_ray_range(g, a, tr, k, &lo, &hi);
  }
  if (irr) {
    lo = 0;
    hi = -2;  // empty for the main kernels; the fixup kernels evaluate it sample by sample
    const int slot = atomicAdd(nirregular, 1);
    if (slot < capacity) irregular[slot] = j * g.nrays + k;
  }
  bounds[(size_t)j * g.nrays + k] = make_int2(lo, hi);
}

// Per (angle, group of 64 rays): union and intersection of the non-empty ranges.
__global__ __launch_bounds__(64) void k_plan_wave_bounds(SSGeom g, const int2* __restrict__ bounds,
                                                         int4* __restrict__ wbounds) {
  const int j = blockIdx.y;
  const int grp = blockIdx.x;
  const int k = grp * SS_WAVE + threadIdx.x;
  int lo = 0x7fffffff, hi = -1, ilo = -0x7fffffff, ihi = 0x7fffffff;
  bool any = false;
  if (k < g.nrays) {
    const int2 b = bounds[(size_t)j * g.nrays + k];
    if (b.y >= b.x) {
      lo = b.x;
      hi = b.y;
      ilo = b.x;
      ihi = b.y;
      any = true;
    }
  }
  // every lane takes part in every shuffle (no short-circuit around them)
  for (int off = 32; off > 0; off >>= 1) {
    lo = min(lo, __shfl_xor(lo, off));
    hi = max(hi, __shfl_xor(hi, off));
    ilo = max(ilo, __shfl_xor(ilo, off));
    ihi = min(ihi, __shfl_xor(ihi, off));
  }
  const bool any_lane = __ballot(any ? 1 : 0) != 0ull;
  if (threadIdx.x == 0) {
    int4 r;
    if (!any_lane) {
      r = make_int4(0, -1, 0, -1);
    } else {
      r = make_int4(lo, hi, ilo, ihi);
    }
    wbounds[(size_t)j * gridDim.x + grp] = r;
  }
}

hipError_t ss_launch_plan_bounds(const SSGeom& g, const SSAngle* angles, int2* bounds, int* irregular,
                                 int* nirregular, int capacity, const double* ray_t, int64_t* ray_alpha,
                                 hipStream_t stream) {
  dim3 grid((g.nrays + 255) / 256, g.nangles);
  hipLaunchKernelGGL(k_plan_bounds, grid, dim3(256), 0, stream, g, angles, bounds, irregular, nirregular, capacity,
                     ray_t, ray_alpha);
  return hipGetLastError();
}

hipError_t ss_launch_plan_wave_bounds(const SSGeom& g, const int2* bounds, int4* wbounds, hipStream_t stream) {
  dim3 grid((g.nrays + SS_WAVE - 1) / SS_WAVE, g.nangles);
  hipLaunchKernelGGL(k_plan_wave_bounds, grid, dim3(SS_WAVE), 0, stream, g, bounds, wbounds);
  return hipGetLastError();
}

// =====================================================================================
// layouts
// =====================================================================================

// image [n][n] -> pair layouts [n][pitch] of float2, q in [0, n+1] (pitch >= n+2):
//   gatherB[r][q] = (F(r, q-1), F(r, q) - F(r, q-1))      image rows
//   gatherA[c][q] = (F(q-1, c), F(q, c) - F(q-1, c))      image columns
// with F = the image inside [0, n)^2 and 0 outside.  Element m+1 of a row holds the
// lower tap of interpolation cell m and the difference to the upper tap, so a Radon
// sample is one aligned 8-byte load and a + w*d.
//
// One tile = GT values of q in both directions (GT = 32 or 64) for a block of NW waves:
// the image square with a one-pixel halo ((GT+1)^2) goes to LDS, every halo load issued
// before the first LDS write; then the waves write rows of GT records (GT * 8
// contiguous bytes), first of layout B, then of layout A, 64 / GT rows per store.  64 x 64
// tiles with 8 waves serve launches of many tiles; 32 x 32 tiles with 4 waves serve small
// ones (one 1024^2 image), where the larger tiles leave the CUs short of waves.
template <int GT, int NW>
__device__ __forceinline__ void ss_gather_tile(const float* __restrict__ src, float2* __restrict__ dA,
                                               float2* __restrict__ dB, int n, int pitch, int bx, int by,
                                               float (*T)[GT + 1], int which = SS_GATHER_BOTH) {
  constexpr int H = GT + 1;                       // halo side
  constexpr int NT = NW * SS_WAVE;                // threads
  constexpr int LOADS = (H * H + NT - 1) / NT;    // halo values per thread
  constexpr int SUB = SS_WAVE / GT;               // rows per wave store
  float v[LOADS];
#pragma unroll
  for (int i = 0; i < LOADS; ++i) {
    const int idx = (int)threadIdx.x + NT * i;
    const int a = idx / H, b = idx - a * H;
    const int r = by - 1 + a, c = bx - 1 + b;
    const bool in = idx < H * H && r >= 0 && r < n && c >= 0 && c < n;
    v[i] = in ? src[(size_t)r * n + c] : 0.f;
  }
#pragma unroll
  for (int i = 0; i < LOADS; ++i) {
    const int idx = (int)threadIdx.x + NT * i;
    if (idx < H * H) T[idx / H][idx % H] = v[i];
  }
  __syncthreads();
  const int lane = threadIdx.x & (SS_WAVE - 1);
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x / SS_WAVE);
  const int x = lane % GT, sub = lane / GT;
  // B: record (r, q) = (F(r, q-1), F(r, q) - F(r, q-1)) = T[r - by + 1][q - bx (+1)]
  const int qb = bx + x;
  for (int i = wv * SUB + sub; (which & SS_GATHER_B) && i < GT; i += NW * SUB) {
    const int r = by + i;
    if (r < n && qb <= n + 1) {
      const float lo = T[i + 1][x];
      dB[(size_t)r * pitch + qb] = make_float2(lo, T[i + 1][x + 1] - lo);
    }
  }
  // A: record (c, q) = (F(q-1, c), F(q, c) - F(q-1, c)) = T[q - by (+1)][c - bx + 1]
  const int qa = by + x;
  for (int j = wv * SUB + sub; (which & SS_GATHER_A) && j < GT; j += NW * SUB) {
    const int cc = bx + j;
    if (cc < n && qa <= n + 1) {
      const float lo = T[x][j + 1];
      dA[(size_t)cc * pitch + qa] = make_float2(lo, T[x + 1][j + 1] - lo);
    }
  }
}

template <int GT, int NW>
__global__ __launch_bounds__(NW * SS_WAVE) void k_gather_pairs(const float* __restrict__ img, float2* __restrict__ gA,
                                                               float2* __restrict__ gB, int n, int pitch, int which) {
  __shared__ float T[GT + 1][GT + 1];  // F(by-1+a, bx-1+b)
  const size_t slice = blockIdx.z;
  ss_gather_tile<GT, NW>(img + slice * n * n, gA + slice * n * pitch, gB + slice * n * pitch, n, pitch,
                         blockIdx.x * GT, blockIdx.y * GT, T, which);
}

hipError_t ss_launch_gather_layouts(const SSDevPlan& p, const float* image, float2* gatherA, float2* gatherB,
                                    int nslices, hipStream_t stream, int which) {
  const int n = p.g.n;
  const int tiles = ss_gather_tiles(n);
  if (!(which & SS_GATHER_BOTH)) return hipSuccess;
  if (p.radon_planes) return ss_launch_gather_planes(p, image, gatherA, gatherB, nslices, stream, which);
  if ((long long)tiles * tiles * nslices >= 1024) {  // at least 4 large tiles per CU
    hipLaunchKernelGGL((k_gather_pairs<SS_GATHER_TILE, 8>), dim3(tiles, tiles, nslices), dim3(8 * SS_WAVE), 0, stream,
                       image, gatherA, gatherB, n, p.g.pitch, which);
  } else {
    const int t32 = (n + 2 + 31) / 32;
    hipLaunchKernelGGL((k_gather_pairs<32, 4>), dim3(t32, t32, nslices), dim3(4 * SS_WAVE), 0, stream, image,
                       gatherA, gatherB, n, p.g.pitch, which);
  }
  return hipGetLastError();
}

// [rows][cols] -> [cols][rows], one 32x32 tile
__device__ __forceinline__ void ss_transpose_tile(const float* __restrict__ src, float* __restrict__ dst, int rows,
                                                  int cols, int bx, int by, float (*tile)[33]) {
  const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;
  for (int yy = ty; yy < 32; yy += 8) {
    const int r = by + yy, c = bx + tx;
    if (r < rows && c < cols) tile[yy][tx] = src[(size_t)r * cols + c];
  }
  __syncthreads();
  for (int xx = ty; xx < 32; xx += 8) {
    const int c = bx + xx, r = by + tx;
    if (r < rows && c < cols) dst[(size_t)c * rows + r] = tile[tx][xx];
  }
}

// [s][rows][cols] -> [s][cols][rows]
__global__ __launch_bounds__(256) void k_transpose2d(const float* __restrict__ in, float* __restrict__ out, int rows,
                                                     int cols) {
  __shared__ float tile[32][33];
  const size_t off = (size_t)blockIdx.z * rows * cols;
  ss_transpose_tile(in + off, out + off, rows, cols, blockIdx.x * 32, blockIdx.y * 32, tile);
}

hipError_t ss_launch_sino_to_t(const float* sino, float* sinoT, int R, int A, int nslices, hipStream_t stream) {
  dim3 grid((A + 31) / 32, (R + 31) / 32, nslices);
  hipLaunchKernelGGL(k_transpose2d, grid, dim3(256), 0, stream, sino, sinoT, R, A);
  return hipGetLastError();
}

hipError_t ss_launch_t_to_sino(const float* sinoT, float* sino, int R, int A, int nslices, hipStream_t stream) {
  dim3 grid((R + 31) / 32, (A + 31) / 32, nslices);
  hipLaunchKernelGGL(k_transpose2d, grid, dim3(256), 0, stream, sinoT, sino, A, R);
  return hipGetLastError();
}

// =====================================================================================
// forward: ray-driven slant-stack Radon
//
// One wave = 64 consecutive rays of one angle.  Sample s walks
// gather rows (image rows for branch B, image columns for branch A, stored
// transposed), so at each s the 64 lanes read a contiguous stretch of one padded
// row.  Loop bounds come from the plan's exact FP64 ranges: predicated head and
// tail, unpredicated middle.
// =====================================================================================

__device__ __forceinline__ double ss_block_sum_f64(double v, double* scratch) {
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off);
  const int wv = threadIdx.x >> 6;
  if ((threadIdx.x & 63) == 0) scratch[wv] = v;
  __syncthreads();
  double r = 0.0;
  if (threadIdx.x == 0)
    for (int i = 0; i < (int)(blockDim.x >> 6); ++i) r += scratch[i];
  return r;  // valid in thread 0
}

// The plan fields the forward kernel reads (kept small: in the batched kernels they
// are loaded per item into scalar registers).
struct SSRadonView {
  const SSAngle* angles;
  const int2* bounds;
  const int4* wbounds;
  const int64_t* ray_alpha;  // per-ray trajectory offsets of a mesh plan, else nullptr
  int n, R, A, pitch, nwaves;
};

__device__ __forceinline__ SSRadonView ss_radon_view(const SSDevPlan& p) {
  return SSRadonView{p.angles, p.bounds, p.wbounds, p.ray_alpha, p.g.n, p.g.nrays, p.g.nangles, p.g.pitch, p.nwaves};
}

// out / meas point at this slice's sinogram
template <int MODE>
__device__ __forceinline__ void ss_radon_store(const SSRadonView& p, int j, int k, float val, float* out,
                                               const float* meas, double* ll) {
  const int R = p.R, A = p.A;
  if (MODE == SS_OUT_SINO) {
    out[(size_t)k * A + j] = val;
  } else if (MODE == SS_OUT_SINOT) {
    out[(size_t)j * R + k] = val;
  } else {
    const size_t idx = (size_t)j * R + k;
    const float s = meas[idx];
    float rho = 0.f;
    if (val > 0.f) {
      rho = s / val;
      *ll += (double)s * log((double)val) - (double)val;
    }
    out[idx] = rho;
  }
}

// A block is 8 waves: 8 consecutive angles over the same 64-ray group, one angle per wave.
// Launches too small to fill the chip (few angles, e.g. one OSEM subset) divide the sample
// rows into slabs taken by separate blocks instead (ss_radon_slab_plan).

typedef float ss_f32x2 __attribute__((ext_vector_type(2)));

#define SS_RSRC_DWORD3 0x00020000  // gfx9 buffer word 3: 32-bit data format, no swizzle

// Structured buffer load of one 8-byte record: address = base + soffset + vindex * stride.
// The record index comes straight from the high word of the Q32.32 trajectory, so a
// sample costs no address arithmetic.
__device__ ss_f32x2 ss_struct_load_f32x2(__amdgpu_buffer_rsrc_t rsrc, int vindex, int voffset, int soffset,
                                         int aux) __asm("llvm.amdgcn.struct.ptr.buffer.load.v2f32");

// tap pair (lower tap, difference) at record `rec` of the gather row at byte offset
// `row_off` (per-slice offsets stay below 2^32 for n <= 16384; unsigned on the hardware)
__device__ __forceinline__ ss_f32x2 ss_pair(__amdgpu_buffer_rsrc_t rs, uint32_t row_off, int rec) {
  return ss_struct_load_f32x2(rs, rec, 0, (int)row_off, 0);
}

// Radon block shapes, picked per launch by the autotuner: staged (tap, difference)
// records per block and sample rows per chunk.  Shape 0: 4096 records (32 KiB), chunks
// of up to 32 rows; shape 1: 4864 records (38 KiB; four blocks still fit a CU's
// 160 KiB), chunks of up to 40 rows.
template <int SH>
struct SSRadonShape {
  static constexpr int CAP = SH == 0 ? 4096 : 4864;
  static constexpr int CHUNK = SH == 0 ? 32 : 40;
};
template <int CAP>
struct SSRadonLds {
  double red[RADON_WAVES];
  int64_t wpar[RADON_WAVES][3];  // per wave: lowest and highest trajectory offset of its rays, slope
  int wmeta[RADON_WAVES][3];     // per wave: branch (-1: no samples), first row, last row
  int wred[2][RADON_WAVES];      // per wave: widest window of a table pass (two passes in turn)
  int2 table[RADON_TABLE];       // per chunk of the super-chunk: first staged record, records per row
  __attribute__((aligned(16))) float2 stage[CAP + 2];  // chunk window; record CAP stays (0, 0)
};

// Direct sample reader: (row s, trajectory u) -> (lower tap, difference), where u is
// the Q32.32 trajectory plus one cell, its high word the record index.
struct SSGatherReader {
  __amdgpu_buffer_rsrc_t rs;
  uint32_t row_bytes;
  __device__ __forceinline__ float2 operator()(int s, int64_t u) const {
    const ss_f32x2 t = ss_pair(rs, (uint32_t)s * row_bytes, (int)(u >> 32));
    return make_float2(t.x, t.y);
  }
};

// G consecutive samples s, s+1, ... of one lane's ray from the staged window, all G
// reads issued before the first is used.  With CHECK, a sample at or beyond `end` or
// outside the lane's own range [lo, lo + span] reads record CAP (past the window), which holds
// (0, 0), instead of branching: it adds exactly zero to both sums.  u advances G steps.
template <int G, bool CHECK, int CAP>
__device__ __forceinline__ void ss_radon_group(const float2* __restrict__ st, int s, int end, int64_t& u,
                                               int64_t step, int lo, unsigned span, float& acc_a, float& acc_d) {
  float2 t[G];
  uint32_t w[G];
  int idx[G];
#pragma unroll
  for (int g = 0; g < G; ++g) {
    idx[g] = (int)(u >> 32);
    if (CHECK) idx[g] = (s + g < end && (unsigned)(s + g - lo) <= span) ? idx[g] : CAP;
    w[g] = (uint32_t)u;
    u += step;
    __asm__ volatile("" : "+v"(u));  // one 64-bit add per sample, not offsets re-derived per sample
  }
#pragma unroll
  for (int g = 0; g < G; ++g) t[g] = st[idx[g]];
  float sa = t[0].x;
  if (G == 4) sa = (t[0].x + t[1].x) + (t[2].x + t[3].x);
  if (G == 8) sa = ((t[0].x + t[1].x) + (t[2].x + t[3].x)) + ((t[4].x + t[5].x) + (t[6].x + t[7].x));
  acc_a += sa;
#pragma unroll
  for (int g = 0; g < G; ++g) acc_d = fmaf((float)w[g], t[g].y, acc_d);
}

// Samples [sa, sb) of one lane's ray from the staged window (u carries the row offset
// in its high word): groups of 4 with the range test before zlo (outside the group's
// common range), unchecked groups of 8 in [zlo, zhi1), and the rest (the last group
// of the common range and the samples from zhi1 on) again in checked groups of 4.
template <int CAP>
__device__ __forceinline__ void ss_radon_rows_staged(const float2* __restrict__ st, int sa, int sb, int zlo,
                                                     int zhi1, int64_t u, int64_t step, int lo, unsigned span,
                                                     float& acc_a, float& acc_d) {
  int s = sa;
  const int h_end = min(sb, zlo);
  if (s < h_end) {
    const int64_t u0 = u;
    for (; s < h_end; s += 4) ss_radon_group<4, true, CAP>(st, s, h_end, u, step, lo, span, acc_a, acc_d);
    s = h_end;
    u = u0 + (int64_t)(h_end - sa) * step;
  }
  const int m_end = min(sb, zhi1);
  for (; s + 8 <= m_end; s += 8) ss_radon_group<8, false, CAP>(st, s, 0, u, step, lo, span, acc_a, acc_d);
  for (; s < sb; s += 4) ss_radon_group<4, true, CAP>(st, s, sb, u, step, lo, span, acc_a, acc_d);
}

// Samples [sa, sb) of one lane's ray: predicated before zlo and from zhi1 on (outside
// the group's common range), unpredicated in between with 4 samples in flight, each
// on its own trajectory register (one 64-bit add per sample; the empty asm keeps the
// compiler from re-deriving the four from one base, which costs extra adds).
template <class Rd>
__device__ __forceinline__ void ss_radon_rows(const Rd& rd, int sa, int sb, int zlo, int zhi1, int64_t u,
                                              int64_t beta, int lo, unsigned span, float& acc_a, float& acc_d) {
  int s = sa;
  const int h_end = min(sb, zlo);
  for (; s < h_end; ++s) {
    if ((unsigned)(s - lo) <= span) {
      const float2 t = rd(s, u);
      acc_a += t.x;
      acc_d = fmaf((float)(uint32_t)u, t.y, acc_d);
    }
    u += beta;
  }
  const int m_end = min(sb, zhi1);
  if (s + 4 <= m_end) {
    int64_t u0 = u, u1 = u + beta, u2 = u + 2 * beta, u3 = u + 3 * beta;
    const int64_t beta4 = 4 * beta;
    for (; s + 4 <= m_end; s += 4) {
      const float2 t0 = rd(s, u0), t1 = rd(s + 1, u1), t2 = rd(s + 2, u2), t3 = rd(s + 3, u3);
      acc_a += (t0.x + t1.x) + (t2.x + t3.x);
      acc_d = fmaf((float)(uint32_t)u0, t0.y, acc_d);
      acc_d = fmaf((float)(uint32_t)u1, t1.y, acc_d);
      acc_d = fmaf((float)(uint32_t)u2, t2.y, acc_d);
      acc_d = fmaf((float)(uint32_t)u3, t3.y, acc_d);
      u0 += beta4;
      u1 += beta4;
      u2 += beta4;
      u3 += beta4;
      __asm__ volatile("" : "+v"(u0), "+v"(u1), "+v"(u2), "+v"(u3));
    }
    u = u0;
  }
  for (; s < m_end; ++s) {
    const float2 t = rd(s, u);
    acc_a += t.x;
    acc_d = fmaf((float)(uint32_t)u, t.y, acc_d);
    u += beta;
  }
  for (; s < sb; ++s) {
    if ((unsigned)(s - lo) <= span) {
      const float2 t = rd(s, u);
      acc_a += t.x;
      acc_d = fmaf((float)(uint32_t)u, t.y, acc_d);
    }
    u += beta;
  }
}

// One block's work: rays [grp*64, grp*64+64) of the RADON_WAVES angles starting at
// j0 + ablk*RADON_WAVES, clipped to [j0, j1), over the sample rows
// [row_lo, row_hi).  gA/gB/out/meas point at this slice's data; in EM mode the block's
// FP64 log-likelihood partial goes to *ll_slot.  In SS_OUT_PARTIAL mode the block writes
// its partial ray sums to part_out ([j - j0][k], delta not applied) for a finishing pass.
//
// All angles of the block on one branch (the usual case): the block walks its sample
// rows in chunks of up to CHUNK rows.  For each chunk it bounds the cells every
// wave can touch (the trajectory is affine in ray and row, so the extremes are at the
// corners), copies that window of the gather rows into LDS with contiguous loads, and
// the waves interpolate from LDS.  A window too wide for LDS falls back to direct
// gathers for that chunk.  A block straddling the branch switch gathers directly from
// the layouts.
template <int MODE, int SH>
__device__ __forceinline__ void ss_radon_item(const SSRadonView& p, const float2* __restrict__ gA,
                                              const float2* __restrict__ gB, int j0, int j1, int grp, int ablk,
                                              int row_lo, int row_hi, float* __restrict__ out,
                                              const float* __restrict__ meas, double* ll_slot,
                                              float* __restrict__ part_out,
                                              SSRadonLds<SSRadonShape<SH>::CAP>& lds) {
  constexpr int CAP = SSRadonShape<SH>::CAP, CHUNK = SSRadonShape<SH>::CHUNK;
  const int lane = threadIdx.x & 63;
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int j = j0 + ablk * RADON_WAVES + wv;
  const int R = p.R, n = p.n, pitch = p.pitch;
  const int k = grp * SS_WAVE + lane;
  const bool active = j < j1;
  float acc_a = 0.f, acc_d = 0.f;
  float delta = 0.f;
  int branch = -1;
  int4 wb = make_int4(0, -1, 0, -1);
  int lo = 0, hi = -1;
  int64_t alpha = 0, gamma = 0, beta = 0;
  if (active) {
    const SSAngle& a = p.angles[j];
    delta = ss_rflf(a.delta);
    alpha = ss_rfl64(a.alpha0);
    gamma = ss_rfl64(a.gamma);
    beta = ss_rfl64(a.beta);
    const int4 w4 = p.wbounds[(size_t)j * p.nwaves + grp];
    wb = make_int4(ss_rfl(w4.x), ss_rfl(w4.y), ss_rfl(w4.z), ss_rfl(w4.w));
    if (wb.y >= wb.x) branch = ss_rfl(a.branch_a);
    if (k < R) {
      const int2 b = p.bounds[(size_t)j * R + k];
      lo = b.x;
      hi = b.y;
    }
  }
  const bool empty = hi < lo;
  const unsigned span = (unsigned)(hi - lo);
  const uint32_t row_bytes = (uint32_t)pitch * 8u;
  // this lane's trajectory offset: u = a_k + s*beta
  int64_t a_k = alpha + (int64_t)k * gamma;
  if (p.ray_alpha && active && k < R) a_k = p.ray_alpha[(size_t)j * R + k];

  bool staged = false;
  {  // staged or direct: decided per block
    // the wave's extreme trajectory offsets (over its rays on the detector)
    int64_t amin = (k < R) ? a_k : INT64_MAX, amax = (k < R) ? a_k : INT64_MIN;
    for (int off = 32; off > 0; off >>= 1) {
      amin = min(amin, (int64_t)__shfl_xor((long long)amin, off));
      amax = max(amax, (int64_t)__shfl_xor((long long)amax, off));
    }
    if (lane == 0) {
      lds.wmeta[wv][0] = branch;
      lds.wmeta[wv][1] = wb.x;
      lds.wmeta[wv][2] = wb.y;
      lds.wpar[wv][0] = amin;
      lds.wpar[wv][1] = amax;
      lds.wpar[wv][2] = beta;
    }
    if (threadIdx.x == 0) lds.stage[CAP] = make_float2(0.f, 0.f);
    __syncthreads();
    int bmin = 2, bmax = -1, s_lo = 0x7fffffff, s_hi = -1;
    for (int w = 0; w < RADON_WAVES; ++w) {
      const int b = lds.wmeta[w][0];
      if (b >= 0) {
        bmin = min(bmin, b);
        bmax = max(bmax, b);
        s_lo = min(s_lo, lds.wmeta[w][1]);
        s_hi = max(s_hi, lds.wmeta[w][2]);
      }
    }
    bmin = ss_rfl(bmin);
    bmax = ss_rfl(bmax);
    s_lo = max(ss_rfl(s_lo), row_lo);
    s_hi = min(ss_rfl(s_hi), row_hi - 1);
    staged = bmax < 0 || bmin == bmax;  // block-uniform
    if (staged && bmax >= 0) {
      const float2* lay = bmax ? gA : gB;
      const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(
          (void*)lay, (short)sizeof(float2), (int)((uint32_t)n * (uint32_t)pitch * 8u), SS_RSRC_DWORD3);
      const SSGatherReader grd{rs, row_bytes};
      // the pure trajectory of this lane's ray at the first row of the current chunk
      int64_t t0 = a_k + (int64_t)s_lo * beta;
      // rows in super-chunks of up to RADON_TABLE chunks: one pass over the table gives
      // every chunk's window and the widest; chunks of CHUNK rows unless that
      // window would not fit, then of the rows it allows (a second pass)
      for (int sc = s_lo; sc <= s_hi;) {
        int rows = CHUNK;
        int nch = min(RADON_TABLE, (s_hi - sc + rows) / rows);
        const int wmax = ss_radon_windows<true>(lds, 0, sc, rows, nch, s_hi, n);
        if (wmax * rows > CAP) {
          int r2 = CAP / wmax;
          if (r2 >= RADON_ROW_ROUND) r2 = r2 / RADON_ROW_ROUND * RADON_ROW_ROUND;
          rows = max(r2, 1);
          nch = min(RADON_TABLE, (s_hi - sc + rows) / rows);
          (void)ss_radon_windows<true>(lds, 1, sc, rows, nch, s_hi, n);
        }
        const int64_t chunk_step = (int64_t)rows * beta;
        for (int c = 0; c < nch; ++c) {
          const int s0 = sc + c * rows, s1 = min(s0 + rows, s_hi + 1);
          const int2 tw = lds.table[c];
          const int rec0 = ss_rfl(tw.x), Wc = ss_rfl(tw.y);
          const bool fits = Wc > 0 && (s1 - s0) * Wc <= CAP;  // block-uniform
          if (c > 0) __syncthreads();  // every wave is done with the previous chunk
          if (fits) {
            // direct global -> LDS copies, 16 bytes (two records) per lane: wave wv copies
            // rows wv, wv+8, ...; the last record read is rec0 + Wc - 1 <= c_hi + 2 <= n + 1
            const float2* src0 = lay + (size_t)(s0 + wv) * pitch + rec0 + 2 * lane;
            for (int seg = 0; seg < Wc; seg += 2 * SS_WAVE) {
              if (seg + 2 * lane < Wc) {
                const float2* src = src0 + seg;
                float2* dst = lds.stage + wv * Wc + seg;
                for (int r = wv; r < s1 - s0; r += RADON_WAVES) {
                  __builtin_amdgcn_global_load_lds((ss_global_cptr)src, (ss_lds_ptr)dst, 16, 0, 0);
                  src += (size_t)RADON_WAVES * pitch;
                  dst += RADON_WAVES * Wc;
                }
              }
            }
          }
          __syncthreads();  // window staged
          const int ra2 = max(s0, wb.x), rb2 = min(s1 - 1, wb.y);
          if (branch >= 0 && ra2 <= rb2 && Wc > 0) {
            const int64_t t = t0 + (int64_t)(ra2 - s0) * beta;
            if (fits) {
              // high word: staged record index (cell + 1 - rec0) + (row - s0) * Wc
              int64_t u = t + ((int64_t)(1 - rec0 + (ra2 - s0) * Wc) << 32);
              int64_t step = beta + ((int64_t)Wc << 32);
              if (empty) {
                u = (int64_t)CAP << 32;
                step = 0;
              }
              ss_radon_rows_staged<CAP>(lds.stage, ra2, rb2 + 1, wb.z, wb.w + 1, u, step, lo, span, acc_a, acc_d);
            } else {
              int64_t u = t + ((int64_t)1 << 32);
              int64_t step = beta;
              if (empty) {
                u = 0;
                step = 0;
              }
              ss_radon_rows(grd, ra2, rb2 + 1, wb.z, wb.w + 1, u, step, lo, span, acc_a, acc_d);
            }
          }
          t0 += chunk_step;
        }
        sc += nch * rows;
      }
    }
  }
  if (!staged && active && branch >= 0) {
    // the group's sample range [wb.x, wb.y] within the rows
    const int sa = max(wb.x, row_lo), sb = min(wb.y + 1, row_hi);
    // u carries the trajectory plus one cell: its high word is the record index m + 1
    // of the lower tap in the gather row, its low word the interpolation weight
    int64_t u = a_k + (int64_t)sa * beta + ((int64_t)1 << 32);
    int64_t step = beta;
    if (empty) {
      // an empty ray reads record 0 (lower tap 0) with weight 0: exactly 0 in the unpredicated loop
      u = 0;
      step = 0;
    }
    const float2* lay = branch ? gA : gB;
    const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(
        (void*)lay, (short)sizeof(float2), (int)((uint32_t)n * (uint32_t)pitch * 8u), SS_RSRC_DWORD3);
    ss_radon_rows(SSGatherReader{rs, row_bytes}, sa, sb, wb.z, wb.w + 1, u, step, lo, span, acc_a, acc_d);
  }
  double ll = 0.0;
  if (active && k < R) {
    if (MODE == SS_OUT_PARTIAL) {
      part_out[(size_t)(j - j0) * R + k] = fmaf(acc_d, SS_INV_FIX, acc_a);
    } else {
      const float val = fmaf(acc_d, SS_INV_FIX, acc_a) * delta;
      ss_radon_store<MODE>(p, j, k, val, out, meas, &ll);
    }
  }
  if (MODE == SS_OUT_EM_RATIO) {
    const double tot = ss_block_sum_f64(ll, lds.red);
    if (threadIdx.x == 0) *ll_slot = tot;
  }
}

// The slabs' partial sums of one ray, added in slab order (the per-plan and batched
// finishing passes give the same bits); unrolled so that the loads issue together.
__device__ __forceinline__ float ss_slab_sum(const float* __restrict__ src, size_t per, int nslab) {
  float sum = 0.f;
#pragma unroll 8
  for (int z = 0; z < nslab; ++z) sum += src[(size_t)z * per];
  return sum;
}

// blockIdx.z = slice * nslab + z: slab z takes sample rows [z * slab_rows, (z + 1) * slab_rows).
// In SS_OUT_PARTIAL mode the blocks write partial ray sums to part[slice][z][j - j0][k] for
// k_radon_slab_finish; in the other modes (nslab = 1) they store the output themselves.
template <int MODE, int SH>
__global__ __launch_bounds__(RADON_WAVES * SS_WAVE) void k_radon(SSDevPlan p, const float2* __restrict__ gA,
                                               const float2* __restrict__ gB, int j0, int j1, int nslab,
                                               int slab_rows, float* __restrict__ out, float* __restrict__ part,
                                               SSEmRatioArgs em) {
  __shared__ SSRadonLds<SSRadonShape<SH>::CAP> lds;
  const int z = (int)(blockIdx.z % (unsigned)nslab);
  const size_t slice = blockIdx.z / (unsigned)nslab;
  const size_t lay = slice * p.g.n * p.g.pitch;
  const size_t so = slice * p.g.nangles * p.g.nrays;
  double* slot = nullptr;
  if (MODE == SS_OUT_EM_RATIO) slot = em.ll_partials + (slice * gridDim.y + blockIdx.y) * gridDim.x + blockIdx.x;
  float* po = MODE == SS_OUT_PARTIAL ? part + (slice * nslab + z) * (size_t)(j1 - j0) * p.g.nrays : nullptr;
  ss_radon_item<MODE, SH>(ss_radon_view(p), gA + lay, gB + lay, j0, j1, blockIdx.x, blockIdx.y, z * slab_rows,
                      min(p.g.n, (z + 1) * slab_rows), out + so, MODE == SS_OUT_EM_RATIO ? em.meas + so : nullptr,
                      slot, po, lds);
}

// =====================================================================================
// Radon in planes: four rays per trajectory
//
// The one-ray kernel above is bound by its LDS reads (8-byte records gamma = 1..1.41 cells
// apart; reads alone reach 13.7 lane-reads per CU-clock at 1 cell, 9.0 at 1.05 and, with two-way
// bank conflicts, 7.9 from 1.1 on) and issues 5 VALU instructions per update, three of them for the trajectory, its weight
// and the address.  Here a lane's trajectory serves four rays whose samples lie at the same
// cell of four images, the planes:
//   SS_PLANES_QUAD    on a grid symmetric about the rotation axis, over all angles of
//                     [0, pi): the image, its half turn (ray -t), its mirror x -> -x (angle
//                     pi - theta) and the half turn of that (pi - theta, -t);
//   SS_PLANES_PAIR    two slices and their half turns (any angle range);
//   SS_PLANES_SLICES  four slices (any geometry).
// The layouts hold the planes' values of a cell together (16 bytes), so one 16-byte LDS
// read gives the lower taps and another the upper taps of all four; the lanes of a read
// pass hold 16 neighbouring rays (ss_plane_ray), which keeps its conflicts two-way.  Per
// four updates: 5 VALU for the trajectory, address and the two weights, 8 FMAs, two reads
// (such pairs of reads alone: 26 updates per CU-clock at a stride of 1, 18 at 1.05, 16 from 1.1 on;
// in the order of the lanes 10.5 at 1.41).  Sums are taken in FP32 over 8 samples, those over
// a chunk's rows and those over the ray: 1e-7 from the 64-bit sums at 2048^2 x 1500 (one
// running sum per ray: 6e-7).  2048^2 x 1500: 1.07 -> 0.80 ms, the layouts' 27 us included; the
// kernel issues VALU in 0.83 and reads LDS in 0.74 of the clocks a CU is busy, which is 0.8 of
// its time (2.9 rounds of blocks).
//
// Every plane's ray keeps its own exact sample range, delta and output; rays computed twice
// (the middle ray of an odd detector, theta = 0 and pi/2, slices past the last) are stored
// once.  Plans with irregular rays don't take this form (ss_radon_planes_kind).
// =====================================================================================

// Layout row r of B (image rows) and row c of A (image columns), cells q in [0, n + 1]:
//   LB[r][q] = (G_0, .., G_3)(r, q - 1),  LA[c][q] = (G_0, .., G_3)(q - 1, c)
// with G_z plane z's image and 0 outside.  A block moves one 32 x 32 pixel tile.
__global__ __launch_bounds__(256) void k_gather_planes(const float* __restrict__ img, ss_f32x4* __restrict__ lA,
                                                       ss_f32x4* __restrict__ lB, int n, int pitch, int nslices,
                                                       int kind, int which) {
  __shared__ float T[SS_PLANES][32][33];
  const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;
  const int bx = blockIdx.x * 32, by = blockIdx.y * 32;
  const int per = ss_planes_slices(kind);
#pragma unroll
  for (int z = 0; z < SS_PLANES; ++z) {
    const SSPlane pl = ss_plane(kind, z);
    const size_t slice = (size_t)min((int)blockIdx.z * per + pl.slice, nslices - 1);
    const float* src = img + slice * n * n;
#pragma unroll
    for (int yy = ty; yy < 32; yy += 8) {
      const int r = by + yy, c = bx + tx;
      const int sr = pl.turn ? n - 1 - r : r, sc = pl.turn != pl.mirror ? n - 1 - c : c;
      T[z][yy][tx] = r < n && c < n ? src[(size_t)sr * n + sc] : 0.f;
    }
  }
  __syncthreads();
  ss_f32x4* dA = lA + (size_t)blockIdx.z * n * pitch;
  ss_f32x4* dB = lB + (size_t)blockIdx.z * n * pitch;
  const ss_f32x4 zero = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int yy = ty; yy < 32; yy += 8) {
    if (which & SS_GATHER_B) {
      const int r = by + yy, q = bx + tx + 1;
      if (r < n && q <= n) dB[(size_t)r * pitch + q] = ss_f32x4{T[0][yy][tx], T[1][yy][tx], T[2][yy][tx], T[3][yy][tx]};
      if (r < n && q == 1) dB[(size_t)r * pitch] = zero;
      if (r < n && q == n) dB[(size_t)r * pitch + n + 1] = zero;
    }
    if (which & SS_GATHER_A) {
      const int c = bx + yy, q = by + tx + 1;
      if (c < n && q <= n) dA[(size_t)c * pitch + q] = ss_f32x4{T[0][tx][yy], T[1][tx][yy], T[2][tx][yy], T[3][tx][yy]};
      if (c < n && q == 1) dA[(size_t)c * pitch] = zero;
      if (c < n && q == n) dA[(size_t)c * pitch + n + 1] = zero;
    }
  }
}

// the sample range of a lane's ray on each plane, in the sample order of plane 0's ray
struct SSPlaneRanges {
  int lo[SS_PLANES];
  unsigned span[SS_PLANES];  // valid samples lo .. lo + span
};

// G samples s, s + 1, ... from the staged window.  CHECK: a sample at or beyond `end`, or
// outside the ray's range, reads the zero cells; with OWN each plane tests its own range
// (they differ at knife-edge samples), else the planes share plane 0's.
template <int G, bool CHECK, bool OWN>
__device__ __forceinline__ void ss_planes_group(const ss_f32x4* __restrict__ st, int s, int end, int64_t& u,
                                                int64_t step, const SSPlaneRanges& rg, float (&acc)[SS_PLANES]) {
  float part[SS_PLANES];
  const unsigned stb = ss_rfl((int)(unsigned)(size_t)(ss_lds_cell)st);
#pragma unroll
  for (int h = 0; h < G; h += 4) {  // four samples' reads in flight
    ss_f32x4 a[4], b[4];
    float w[4];
    int keep[4];
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      int idx = (int)(u >> 32);
      keep[g] = 0;
      if (CHECK) {
        const int t = s + h + g;
        if (OWN) {
#pragma unroll
          for (int z = 0; z < SS_PLANES; ++z) keep[g] |= (t < end && (unsigned)(t - rg.lo[z]) <= rg.span[z]) << z;
          idx = keep[g] ? idx : PLANES_CAP;
        } else {
          idx = t < end && (unsigned)(t - rg.lo[0]) <= rg.span[0] ? idx : PLANES_CAP;
        }
      }
      // weights in [0, 1]: left at 2^32 they would overflow sums from 8e28 on
      w[g] = (float)(uint32_t)u * SS_INV_FIX;
      u += step;
      __asm__ volatile("" : "+v"(u));  // one 64-bit add per sample
      // one byte address for both cells (the second in the read's offset field): stb + 16 idx, by
      // hand, as the compiler takes it out of u's words in three instructions
      unsigned at;
      __asm__("v_lshl_add_u32 %0, %1, 4, %2" : "=v"(at) : "v"(idx), "s"(stb));
      const ss_lds_cell c = (ss_lds_cell)(size_t)at;
      a[g] = c[0];
      b[g] = c[1];
    }
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const float w1 = 1.f - w[g];
#pragma unroll
      for (int z = 0; z < SS_PLANES; ++z) {
        float lo = a[g][z], hi = b[g][z];
        if (CHECK && OWN) {
          lo = keep[g] >> z & 1 ? lo : 0.f;
          hi = keep[g] >> z & 1 ? hi : 0.f;
        }
        part[z] = h + g == 0 ? w1 * lo : fmaf(w1, lo, part[z]);
        part[z] = fmaf(w[g], hi, part[z]);
      }
    }
  }
#pragma unroll
  for (int z = 0; z < SS_PLANES; ++z) acc[z] += part[z];
}

// samples [sa, sb): checked groups before zlo and from zhi1 on, unchecked between
template <bool OWN>
__device__ __forceinline__ void ss_planes_rows(const ss_f32x4* __restrict__ st, int sa, int sb, int zlo, int zhi1,
                                               int64_t u, int64_t step, const SSPlaneRanges& rg,
                                               float (&acc)[SS_PLANES]) {
  int s = sa;
  const int h_end = min(sb, zlo);
  if (s < h_end) {
    const int64_t u0 = u;
    for (; s < h_end; s += 4) ss_planes_group<4, true, OWN>(st, s, h_end, u, step, rg, acc);
    s = h_end;
    u = u0 + (int64_t)(h_end - sa) * step;
  }
  const int m_end = min(sb, zhi1);
  for (; s + 8 <= m_end; s += 8) ss_planes_group<8, false, OWN>(st, s, 0, u, step, rg, acc);
  for (; s < sb; s += 4) ss_planes_group<4, true, OWN>(st, s, sb, u, step, rg, acc);
}

// One block: the rays of group `grp` of the RADON_WAVES angles from j0 + ablk*RADON_WAVES
// (clipped to j1: plane 0's angles), sample rows [row_lo, row_hi).  A block whose angles lie
// on both sides of a branch switch makes a pass for each.
template <int MODE>
__device__ __forceinline__ void ss_planes_item(const SSRadonView& p, const ss_f32x4* __restrict__ lA,
                                               const ss_f32x4* __restrict__ lB, int kind, int slice0, int nslices,
                                               int j0, int j1, int jpart, int npart, int nrays, int grp, int ablk,
                                               int row_lo, int row_hi, float* __restrict__ out,
                                               const float* __restrict__ meas, double* ll_slot,
                                               float* __restrict__ part_out, size_t part_slice, SSPlanesLds& lds) {
  const int lane = threadIdx.x & 63;
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int j = j0 + ablk * RADON_WAVES + wv;
  const int R = p.R, A = p.A, n = p.n, pitch = p.pitch;
  const int k = grp * SS_WAVE + ss_plane_ray(lane);
  const bool active = j < j1, on = active && k < nrays;
  int branch = -1;
  int64_t a_k = 0, beta = 0;
  SSPlaneRanges rg;
  // the group's rows: union and common range over its rays and planes
  int ulo = 0x7fffffff, uhi = -1, clo = -0x7fffffff, chi = 0x7fffffff;
  bool any = false, own = false;
  if (active) {
    const SSAngle& a = p.angles[j];
    branch = ss_rfl(a.branch_a);
    beta = ss_rfl64(a.beta);
    a_k = ss_rfl64(a.alpha0) + (int64_t)k * ss_rfl64(a.gamma);
    if (p.ray_alpha && k < R) a_k = p.ray_alpha[(size_t)j * R + k];
  }
#pragma unroll
  for (int z = 0; z < SS_PLANES; ++z) {
    const SSPlane pl = ss_plane(kind, z);
    rg.lo[z] = 0x40000000;  // empty: no sample passes the test
    rg.span[z] = 0;
    if (on) {
      const int jz = pl.mirror ? (j > 0 ? A - j : 0) : j;
      const bool rev = pl.turn != (pl.mirror && j == 0);  // angle pi is angle 0 with the rays reversed
      int2 b = p.bounds[(size_t)jz * R + (rev ? R - 1 - k : k)];
      if (b.y >= b.x) {
        // image rows (branch B) are reversed by the half turn, columns (A) by either
        if (pl.turn != (pl.mirror && branch == 1)) b = make_int2(n - 1 - b.y, n - 1 - b.x);
        rg.lo[z] = b.x;
        rg.span[z] = (unsigned)(b.y - b.x);
        any = true;
        ulo = min(ulo, b.x);
        uhi = max(uhi, b.y);
        clo = max(clo, b.x);
        chi = min(chi, b.y);
      }
    }
    own = own || rg.lo[z] != rg.lo[0] || rg.span[z] != rg.span[0];
  }
  if (own && any) {  // no common range: every sample of the ray is tested per plane
    bool whole = true;
#pragma unroll
    for (int z = 0; z < SS_PLANES; ++z) whole = whole && rg.lo[z] != 0x40000000;
    if (!whole) clo = 0x7fffffff, chi = -1;
  }
  const bool own_wave = __ballot(own) != 0ull;
  int64_t amin = on ? a_k : INT64_MAX, amax = on ? a_k : INT64_MIN;
  for (int off = 32; off > 0; off >>= 1) {
    ulo = min(ulo, __shfl_xor(ulo, off));
    uhi = max(uhi, __shfl_xor(uhi, off));
    clo = max(clo, __shfl_xor(clo, off));
    chi = min(chi, __shfl_xor(chi, off));
    amin = min(amin, (int64_t)__shfl_xor((long long)amin, off));
    amax = max(amax, (int64_t)__shfl_xor((long long)amax, off));
  }
  ulo = ss_rfl(ulo);
  uhi = ss_rfl(uhi);
  clo = ss_rfl(clo);
  chi = ss_rfl(chi);
  if (uhi < ulo) branch = -1;
  if (lane == 0) {
    lds.wmeta[wv][0] = branch;
    lds.wmeta[wv][1] = ulo;
    lds.wmeta[wv][2] = uhi;
    lds.wpar[wv][0] = amin;
    lds.wpar[wv][1] = amax;
    lds.wpar[wv][2] = beta;
  }
  if (threadIdx.x < 2) lds.stage[PLANES_CAP + threadIdx.x] = ss_f32x4{0.f, 0.f, 0.f, 0.f};
  float tot[SS_PLANES] = {0.f, 0.f, 0.f, 0.f};
  for (int pass = 0; pass < 2; ++pass) {
    __syncthreads();
    if (lane == 0) lds.wmeta[wv][0] = branch == pass ? branch : -1;  // this pass's waves
    __syncthreads();
    int s_lo = 0x7fffffff, s_hi = -1;
    for (int w = 0; w < RADON_WAVES; ++w)
      if (lds.wmeta[w][0] >= 0) {
        s_lo = min(s_lo, lds.wmeta[w][1]);
        s_hi = max(s_hi, lds.wmeta[w][2]);
      }
    s_lo = max(ss_rfl(s_lo), row_lo);
    s_hi = min(ss_rfl(s_hi), row_hi - 1);
    const bool mine = branch == pass;
    const ss_f32x4* lay = pass ? lA : lB;
    ss_planes_chunks(lds, lay, pitch, n, s_lo, s_hi, wv, lane, [&](int s0, int s1, int rec0, int Wc, bool fits) {
      const int ra2 = max(s0, ulo), rb2 = min(s1 - 1, uhi);
      if (mine && ra2 <= rb2 && Wc > 0) {
        const int64_t t = a_k + (int64_t)ra2 * beta;
        float acc[SS_PLANES] = {0.f, 0.f, 0.f, 0.f};  // the chunk's sum
        if (fits) {
          // high word: staged cell index (cell + 1 - rec0) + (row - s0) * Wc
          int64_t u = t + ((int64_t)(1 - rec0 + (ra2 - s0) * Wc) << 32);
          int64_t step = beta + ((int64_t)Wc << 32);
          if (!any) {
            u = (int64_t)PLANES_CAP << 32;
            step = 0;
          }
          if (own_wave)
            ss_planes_rows<true>(lds.stage, ra2, rb2 + 1, clo, chi + 1, u, step, rg, acc);
          else
            ss_planes_rows<false>(lds.stage, ra2, rb2 + 1, clo, chi + 1, u, step, rg, acc);
        } else if (any) {  // the window does not fit the LDS: read the layout
          int64_t u = t + ((int64_t)1 << 32);
          for (int s = ra2; s <= rb2; ++s, u += beta) {
            int keep = 0;
#pragma unroll
            for (int z = 0; z < SS_PLANES; ++z) keep |= ((unsigned)(s - rg.lo[z]) <= rg.span[z]) << z;
            if (keep) {
              const ss_f32x4* cell = lay + (size_t)s * pitch + (int)(u >> 32);
              const ss_f32x4 a = cell[0], b = cell[1];
              const float w = (float)(uint32_t)u * SS_INV_FIX, w1 = 1.f - w;
#pragma unroll
              for (int z = 0; z < SS_PLANES; ++z) {
                const float v = fmaf(w, b[z], w1 * a[z]);
                acc[z] += keep >> z & 1 ? v : 0.f;
              }
            }
          }
        }
#pragma unroll
        for (int z = 0; z < SS_PLANES; ++z) tot[z] += acc[z];
      }
    });
  }
  double ll = 0.0;
  if (on) {
#pragma unroll
    for (int z = 0; z < SS_PLANES; ++z) {
      const SSPlane pl = ss_plane(kind, z);
      const int kz = pl.turn ? R - 1 - k : k;
      const int jz = pl.mirror ? A - j : j;
      if (slice0 + pl.slice >= nslices) continue;     // a group past the last slice
      if (pl.turn && kz == k) continue;               // the middle ray, its own half turn
      if (pl.mirror && (j == 0 || jz == j)) continue;  // angles that are their own mirror
      const float sum = tot[z];
      const size_t so = (size_t)(slice0 + pl.slice) * A * R;
      if (MODE == SS_OUT_PARTIAL) {
        part_out[(size_t)pl.slice * part_slice + (size_t)(jz - jpart) * R + kz] = sum;
      } else {
        ss_radon_store<MODE>(p, jz, kz, sum * p.angles[jz].delta, out + so,
                             MODE == SS_OUT_EM_RATIO ? meas + so : nullptr, &ll);
      }
    }
  }
  if (MODE == SS_OUT_EM_RATIO) {
    const double tot = ss_block_sum_f64(ll, lds.red);
    if (threadIdx.x == 0) *ll_slot = tot;
  }
}

// blockIdx.z = group * nslab + z.  The block's rays and angles come from `order`, over plane
// 0's angles [j0, jd1) and rays [0, nrays); partial sums are laid out over [j0, j1).
template <int MODE>
__global__ __launch_bounds__(RADON_WAVES * SS_WAVE, PLANES_BLOCKS) void k_radon_planes(
    SSDevPlan p, const ss_f32x4* __restrict__ lA, const ss_f32x4* __restrict__ lB, int kind, int nslices, int j0,
    int j1, int jd1, int nrays, SSPlanesOrder order, int nslab, int slab_rows, float* __restrict__ out,
    float* __restrict__ part, SSEmRatioArgs em) {
  __shared__ SSPlanesLds lds;
  const int z = (int)(blockIdx.z % (unsigned)nslab);
  const int group = (int)(blockIdx.z / (unsigned)nslab);
  const int2 at = ss_planes_place(order, blockIdx.x);
  const int grp = at.x, ablk = at.y;
  const size_t lay = (size_t)group * p.g.n * p.g.pitch;
  const int slice0 = group * ss_planes_slices(kind);
  const size_t per = (size_t)(j1 - j0) * p.g.nrays;
  double* slot = nullptr;
  if (MODE == SS_OUT_EM_RATIO) slot = em.ll_partials + (size_t)group * gridDim.x + blockIdx.x;
  if (ablk < 0) {  // block-uniform
    if (MODE == SS_OUT_EM_RATIO && threadIdx.x == 0) *slot = 0.0;
    return;
  }
  float* po = MODE == SS_OUT_PARTIAL ? part + ((size_t)slice0 * nslab + z) * per : nullptr;
  ss_planes_item<MODE>(ss_radon_view(p), lA + lay, lB + lay, kind, slice0, nslices, j0, jd1, j0, j1 - j0, nrays,
                       grp, ablk, z * slab_rows, min(p.g.n, (z + 1) * slab_rows), out, em.meas, slot, po,
                       (size_t)nslab * per, lds);
}

// Sums the slabs' partial sums of rays [j0, j1) x [0, R) of each slice and stores them
// as k_radon does (delta applied; in EM mode the ratio, and one FP64 log-likelihood
// partial per block at ll_partials[slice * gridDim.x + blockIdx.x]).
template <int MODE>
__global__ __launch_bounds__(256) void k_radon_slab_finish(SSDevPlan p, const float* __restrict__ part, int nslab,
                                                           int j0, int j1, float* __restrict__ out, SSEmRatioArgs em) {
  __shared__ double red[4];
  const size_t slice = blockIdx.y;
  const int R = p.g.nrays;
  const size_t per = (size_t)(j1 - j0) * R;
  const size_t idx = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  const size_t so = slice * p.g.nangles * (size_t)R;
  double ll = 0.0;
  if (idx < per) {
    const int jj = (int)(idx / (unsigned)R), k = (int)(idx - (size_t)jj * R);
    const float* src = part + slice * nslab * per + idx;
    float sum = 0.f;
    sum = ss_slab_sum(src, per, nslab);
    ss_radon_store<MODE>(ss_radon_view(p), j0 + jj, k, sum * p.angles[j0 + jj].delta, out + so,
                         MODE == SS_OUT_EM_RATIO ? em.meas + so : nullptr, &ll);
  }
  if (MODE == SS_OUT_EM_RATIO) {
    const double tot = ss_block_sum_f64(ll, red);
    if (threadIdx.x == 0) em.ll_partials[slice * gridDim.x + blockIdx.x] = tot;
  }
}

// Irregular rays (knife-edge angles): one block per ray, samples across threads,
// validity evaluated per sample with the exact FP64 predicate.  `idx` indexes the
// plan's irregular list; rays outside [j0, j1) write a zero partial only.
template <int MODE>
__device__ __forceinline__ void ss_radon_fixup_item(const SSDevPlan& p, const float2* __restrict__ gA,
                                                    const float2* __restrict__ gB, int j0, int j1, int idx,
                                                    float* __restrict__ out, const float* __restrict__ meas,
                                                    double* ll_slot, float* redf) {
  const int id = p.irregular[idx];
  const int R = p.g.nrays, n = p.g.n, pitch = p.g.pitch;
  const int j = id / R, k = id % R;
  if (j < j0 || j >= j1) {
    if (MODE == SS_OUT_EM_RATIO && threadIdx.x == 0) *ll_slot = 0.0;
    return;
  }
  const SSAngle& a = p.angles[j];
  const float2* img = (a.branch_a ? gA : gB) + 1;
  const double t = p.ray_t ? p.ray_t[k] : ss_ray_t(p.g, k);
  const int64_t a_k = p.ray_alpha ? p.ray_alpha[(size_t)j * R + k] : a.alpha0 + (int64_t)k * a.gamma;
  float acc = 0.f;
  for (int s = threadIdx.x; s < n; s += blockDim.x) {
    if (ss_radon_sample_valid_t(p.g, a, t, s)) {
      const int64_t u = a_k + (int64_t)s * a.beta;
      const int m = (int)(u >> 32);
      const float w = (float)(uint32_t)u * SS_INV_FIX;
      const float2 rec = img[(size_t)s * pitch + m];
      acc += fmaf(w, rec.y, rec.x);
    }
  }
  for (int off = 32; off > 0; off >>= 1) acc += __shfl_xor(acc, off);
  if ((threadIdx.x & 63) == 0) redf[threadIdx.x >> 6] = acc;
  __syncthreads();
  if (threadIdx.x == 0) {
    float tot = 0.f;
    for (int i = 0; i < (int)(blockDim.x >> 6); ++i) tot += redf[i];
    double ll = 0.0;
    ss_radon_store<MODE>(ss_radon_view(p), j, k, tot * a.delta, out, meas, &ll);
    if (MODE == SS_OUT_EM_RATIO) *ll_slot = ll;
  }
}

template <int MODE>
__global__ __launch_bounds__(256) void k_radon_fixup(SSDevPlan p, const float2* __restrict__ gA,
                                                     const float2* __restrict__ gB, int j0, int j1,
                                                     float* __restrict__ out, SSEmRatioArgs em, int partial_base) {
  __shared__ float redf[4];
  const size_t slice = blockIdx.y;
  const size_t lay = slice * p.g.n * p.g.pitch;
  const size_t so = slice * p.g.nangles * p.g.nrays;
  double* slot = nullptr;
  if (MODE == SS_OUT_EM_RATIO) slot = em.ll_partials + partial_base + slice * gridDim.x + blockIdx.x;
  ss_radon_fixup_item<MODE>(p, gA + lay, gB + lay, j0, j1, blockIdx.x, out + so,
                            MODE == SS_OUT_EM_RATIO ? em.meas + so : nullptr, slot, redf);
}

// A launch of few blocks (a few angles: one OSEM subset) divides the sample rows of every
// (angle block, ray group) into slabs handled by separate blocks, so that every CU gets
// blocks while each block keeps the LDS-staged path; a finishing pass then adds the
// slabs' partial sums.  Rows per slab are a multiple of RADON_SLAB_ALIGN, and the divided
// launch stays within SS_RADON_SLAB_BLOCKS blocks (4 per CU, one round: a second round
// for a few blocks would double the launch time).
int ss_radon_slab_plan(int n, long long blocks, int* rows, int target) {
  *rows = n;
  if (blocks >= target) return 1;
  const long long want = target / std::max(blocks, 1LL);
  if (want <= 1) return 1;
  int L = (int)((n + want - 1) / want);
  L = (L + RADON_SLAB_ALIGN - 1) / RADON_SLAB_ALIGN * RADON_SLAB_ALIGN;
  const int count = (n + L - 1) / L;
  if (count <= 1) return 1;
  *rows = L;
  return count;
}

int ss_radon_slabs(const SSDevPlan& p, int j0, int j1, int nslices, int* rows) {
  const int n = p.g.n;
  *rows = n;
  if (j1 <= j0) return 1;
  if (p.radon_slab_rows > 0) {
    const int L = (std::min(p.radon_slab_rows, n) + RADON_SLAB_ALIGN - 1) / RADON_SLAB_ALIGN * RADON_SLAB_ALIGN;
    const int count = (n + L - 1) / L;
    if (count <= 1) return 1;
    *rows = L;
    return count;
  }
  if (p.radon_planes)
    return ss_radon_slab_plan(n, ss_planes_blocks(p, j0, j1, nslices), rows, SS_PLANES_SLAB_BLOCKS);
  return ss_radon_slab_plan(n, ss_radon_blocks(p.nwaves, j0, j1) * nslices, rows);
}

static int ss_radon_finish_blocks(int nj, int R) { return (int)(((long long)nj * R + 255) / 256); }

size_t ss_radon_layout_bytes(const SSDevPlan& p, int nslices) {
  const size_t records = (size_t)p.g.n * p.g.pitch;
  if (!p.radon_planes) return sizeof(float2) * records * nslices;
  return sizeof(ss_f32x4) * records * ss_planes_groups(p.radon_planes, nslices);
}

// Plane 0's angles and rays of a launch over [j0, j1): a quad launch's blocks walk theta in
// [0, pi/2] and half the detector, the pair form half the detector
static int ss_planes_j1(const SSDevPlan& p, int j1) {
  return p.radon_planes == SS_PLANES_QUAD ? p.g.nangles / 2 + 1 : j1;
}
static int ss_planes_rays(const SSDevPlan& p) {
  return p.radon_planes == SS_PLANES_SLICES ? p.g.nrays : (p.g.nrays + 1) / 2;
}

hipError_t ss_launch_gather_planes(const SSDevPlan& p, const float* image, float2* lA, float2* lB, int nslices,
                                   hipStream_t stream, int which) {
  const int t = (p.g.n + 31) / 32;
  hipLaunchKernelGGL(k_gather_planes, dim3(t, t, ss_planes_groups(p.radon_planes, nslices)), dim3(256), 0, stream,
                     image, reinterpret_cast<ss_f32x4*>(lA), reinterpret_cast<ss_f32x4*>(lB), p.g.n, p.g.pitch,
                     nslices, p.radon_planes, which);
  return hipGetLastError();
}

static SSPlanesOrder ss_planes_order(const SSDevPlan& p, int j0, int j1) {
  return ss_planes_order(ss_planes_rays(p), ss_planes_j1(p, j1) - j0);
}

long long ss_planes_blocks(const SSDevPlan& p, int j0, int j1, int nslices) {
  return (long long)ss_planes_order(p, j0, j1).blocks *
         ss_planes_groups(p.radon_planes, nslices);
}

// Whether an undivided planes launch has blocks with work for the whole chip, at most one
// launched block in nine without (SSPlanesOrder) and at most one plane in 17 empty
bool ss_planes_suit(const SSDevPlan& p, int j0, int j1, int nslices) {
  const SSPlanesOrder o = ss_planes_order(p, j0, j1);
  const long long groups = ss_planes_groups(p.radon_planes, nslices), work = (long long)o.g * o.y;
  return work * groups >= SS_RADON_SLAB_BLOCKS && 8LL * o.blocks <= 9 * work &&
         16 * groups * ss_planes_slices(p.radon_planes) <= 17LL * nslices;
}

size_t ss_radon_scratch(const SSDevPlan& p, int j0, int j1, int nslices) {
  int rows;
  const int nslab = ss_radon_slabs(p, j0, j1, nslices, &rows);
  return nslab > 1 ? sizeof(float) * (size_t)nslab * nslices * (size_t)(j1 - j0) * p.g.nrays : 0;
}

int ss_radon_partials(const SSDevPlan& p, int j0, int j1, int nslices) {
  int rows;
  const int nslab = ss_radon_slabs(p, j0, j1, nslices, &rows);
  if (nslab == 1 && p.radon_planes) return (int)ss_planes_blocks(p, j0, j1, nslices);
  const int main = nslab > 1 ? ss_radon_finish_blocks(j1 - j0, p.g.nrays)
                             : p.nwaves * ((j1 - j0 + RADON_WAVES - 1) / RADON_WAVES);
  return (main + p.nirregular) * nslices;
}

hipError_t ss_launch_radon(const SSDevPlan& p, const float2* gatherA, const float2* gatherB, int j0, int j1,
                           int nslices, int mode, float* out, SSEmRatioArgs em, float* scratch, hipStream_t stream) {
  if (j1 <= j0) return hipSuccess;
  int rows;
  const int nslab = ss_radon_slabs(p, j0, j1, nslices, &rows);
  if (nslab > 1 && !scratch) return hipErrorInvalidValue;
  dim3 grid(p.nwaves, (j1 - j0 + RADON_WAVES - 1) / RADON_WAVES, nslices * nslab);
  dim3 block(RADON_WAVES * SS_WAVE);
  int partial_base;
  const int jd1 = ss_planes_j1(p, j1), half = ss_planes_rays(p);
  const SSPlanesOrder order = ss_planes_order(p, j0, j1);
  if (p.radon_planes) grid = dim3(order.blocks, 1, ss_planes_groups(p.radon_planes, nslices) * nslab);
  // the main pass in the plan's form: planes, or block shape 0 or 1
#define SS_RADON_LAUNCH(MODE, OUTP, PARTP, NSLAB, ROWS, EM)                                                        \
  do {                                                                                                            \
    if (p.radon_planes)                                                                                           \
      hipLaunchKernelGGL(k_radon_planes<MODE>, grid, block, 0, stream, p,                                         \
                         reinterpret_cast<const ss_f32x4*>(gatherA), reinterpret_cast<const ss_f32x4*>(gatherB),  \
                         p.radon_planes, nslices, j0, j1, jd1, half, order, NSLAB, ROWS, OUTP, PARTP, EM);        \
    else if (p.radon_shape == 1)                                                                                       \
      hipLaunchKernelGGL((k_radon<MODE, 1>), grid, block, 0, stream, p, gatherA, gatherB, j0, j1, NSLAB, ROWS,    \
                         OUTP, PARTP, EM);                                                                        \
    else                                                                                                          \
      hipLaunchKernelGGL((k_radon<MODE, 0>), grid, block, 0, stream, p, gatherA, gatherB, j0, j1, NSLAB, ROWS,    \
                         OUTP, PARTP, EM);                                                                        \
  } while (0)
  if (nslab > 1) {
    const SSEmRatioArgs none{nullptr, nullptr};
    SS_RADON_LAUNCH(SS_OUT_PARTIAL, nullptr, scratch, nslab, rows, none);
    const int fb = ss_radon_finish_blocks(j1 - j0, p.g.nrays);
    dim3 fin(fb, nslices);
    switch (mode) {
      case SS_OUT_SINO:
        hipLaunchKernelGGL(k_radon_slab_finish<SS_OUT_SINO>, fin, dim3(256), 0, stream, p, scratch, nslab, j0, j1, out,
                           em);
        break;
      case SS_OUT_SINOT:
        hipLaunchKernelGGL(k_radon_slab_finish<SS_OUT_SINOT>, fin, dim3(256), 0, stream, p, scratch, nslab, j0, j1,
                           out, em);
        break;
      default:
        hipLaunchKernelGGL(k_radon_slab_finish<SS_OUT_EM_RATIO>, fin, dim3(256), 0, stream, p, scratch, nslab, j0, j1,
                           out, em);
        break;
    }
    partial_base = fb * nslices;
  } else {
    switch (mode) {
      case SS_OUT_SINO:
        SS_RADON_LAUNCH(SS_OUT_SINO, out, nullptr, 1, p.g.n, em);
        break;
      case SS_OUT_SINOT:
        SS_RADON_LAUNCH(SS_OUT_SINOT, out, nullptr, 1, p.g.n, em);
        break;
      default:
        SS_RADON_LAUNCH(SS_OUT_EM_RATIO, out, nullptr, 1, p.g.n, em);
        break;
    }
#undef SS_RADON_LAUNCH
    partial_base = (int)(grid.x * grid.y) * (p.radon_planes ? (int)grid.z : nslices);
  }
  hipError_t e = hipGetLastError();
  if (e != hipSuccess || p.nirregular == 0) return e;
  dim3 fgrid(p.nirregular, nslices);
  switch (mode) {
    case SS_OUT_SINO:
      hipLaunchKernelGGL(k_radon_fixup<SS_OUT_SINO>, fgrid, dim3(256), 0, stream, p, gatherA, gatherB, j0, j1, out,
                         em, partial_base);
      break;
    case SS_OUT_SINOT:
      hipLaunchKernelGGL(k_radon_fixup<SS_OUT_SINOT>, fgrid, dim3(256), 0, stream, p, gatherA, gatherB, j0, j1, out,
                         em, partial_base);
      break;
    default:
      hipLaunchKernelGGL(k_radon_fixup<SS_OUT_EM_RATIO>, fgrid, dim3(256), 0, stream, p, gatherA, gatherB, j0, j1,
                         out, em, partial_base);
      break;
  }
  return hipGetLastError();
}

// =====================================================================================
// backprojection: pixel-driven, 32 x (8*ROWS) pixel tile per block, angle blocks
// staged in LDS
//
// For each angle of a stage the block computes (FP64) the ray coordinate U of the
// tile origin and the tile's U range, then stages the W consecutive rays
// [base, base+W) that the tile can touch.  Each thread owns ROWS pixels (one column,
// rows ty, ty+8, ...) and interpolates from LDS with FP32 offsets relative to `base`
// (|u| < ~W, so FP32 resolves ~1e-5 of a detector bin).
//
// Exactness of the 0 <= m <= R-2 predicate: a tile whose U range lies inside
// [eps, R-1-eps] needs no test; one entirely outside contributes nothing; the rest
// test each pixel, and pixels within W 2^-20 bins of an edge (ss_bp_edge) re-evaluate the
// reference's FP64 expression.
// =====================================================================================

#define BP_TILE_W 32

struct alignas(16) BPAngle {
  float f0, b, c;  // read together by one 16-byte LDS read
  int flag;        // 0 outside, 1 interior, 2 boundary
  int base;
  float lo, hi;    // u of the pixels that are on the detector for certain
  int pad;
};

__device__ __forceinline__ int ss_bp_exact_valid(const SSDevPlan& p, int j, int row, int col) {
  const SSAngle& a = p.angles[j];
  return ss_bp_sample_valid(p.g, a.cost, a.sint, row, col) ? 1 : 0;
}

// Pixels this near (in rays) to the first or last ray take the exact test: a tile's pixels have
// u < W rays from its base, and its FP32 evaluation (the rounded origin, slopes times up to 63
// pixels, two fused steps) is within W 2^-22 of the FP64 coordinate; four times that.  (At
// 1e-3 for every tile one wave in ten took the test and waited for its loads.)
__device__ __forceinline__ float ss_bp_edge(int W) { return (float)W * 9.5367431640625e-7f; }

// Angle j on the tile [c0, c0 + 32) x [r0, r0 + th): its origin's ray coordinate from the base
// ray, the slopes, and whether the tile lies on the detector
__device__ __forceinline__ BPAngle ss_bp_params(const SSDevPlan& p, int j, int c0, int r0, int th) {
  BPAngle q{0.f, 0.f, 0.f, 0, 0, 0.f, 0.f, 0};
  const int R = p.g.nrays;
  const SSAngle& a = p.angles[j];
  const double U = a.bp_a + (double)c0 * a.bp_b + (double)r0 * a.bp_c;
  const double ec = (double)(BP_TILE_W - 1) * a.bp_b, er = (double)(th - 1) * a.bp_c;
  const double umin = U + fmin(0.0, ec) + fmin(0.0, er);
  const double umax = U + fmax(0.0, ec) + fmax(0.0, er);
  const double base = floor(umin) - 1.0;
  q.f0 = (float)(U - base);
  q.b = (float)a.bp_b;
  q.c = (float)a.bp_c;
  const double eps = 1e-6;
  if (umax < -eps || umin >= (double)(R - 1) + eps)
    q.flag = 0;
  else if (umin >= eps && umax < (double)(R - 1) - eps)
    q.flag = 1;
  else
    q.flag = 2;
  q.base = (int)base;
  return q;
}

template <int STAGE>
struct SSBpLds {
  // per staged ray w the PL records (value - w * difference, difference to the next ray),
  // in pairs of planes; planes 2, 3 in the second half
  alignas(16) float2 win[STAGE];
  BPAngle par[64];
};

// raw buffer load of one float at a byte offset; an offset past the buffer (also a negative
// one, as unsigned) reads 0
__device__ float ss_raw_load_f32(__amdgpu_buffer_rsrc_t rsrc, int voffset, int soffset,
                                 int aux) __asm("llvm.amdgcn.raw.ptr.buffer.load.f32");

// the value of the next lane (lane 63: 0)
__device__ __forceinline__ float ss_next_lane(float v) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x130 /* wave_shl:1 */, 0xf, 0xf, true));
}

// The sinogram row that the mirrored planes of angle j read (PL = 4): that of the angle
// pi - theta_j, A - j on the grid [0, pi); for theta = 0 its own row reversed.
struct SSBpMirror {
  int row;
  bool flip;
};
__device__ __forceinline__ SSBpMirror ss_bp_mirror(int j, int A) { return SSBpMirror{j > 0 ? A - j : 0, j == 0}; }

#define BP_BATCH (SS_BP_STAGE_BATCH / 4)  // angle windows whose loads a wave issues together

// One stage's windows of the angles jb + wv, jb + wv + 4, ... < jb + nj: the records w in
// [0, W) of each, ray base + w of every plane (lane js + jj holds base).  The loads of BP_BATCH windows are issued
// before the first is used, so that a stage waits for memory once per BP_BATCH windows and
// not once per window; a record's second ray comes from the next lane (63 records a pass);
// rays off the detector read 0 through the buffer's range check.
template <int PL, int STAGE>
__device__ __forceinline__ void ss_bp_stage(const float* __restrict__ sl, int R, int A, int W, int jb, int nj, int wv,
                                            int lane, int base, int js, float2* __restrict__ win) {
  for (int w0 = 0; w0 < W; w0 += SS_WAVE - 1) {
    const int w = w0 + lane;
    const float fw = -(float)w;
    for (int j4 = wv; j4 < nj; j4 += 4 * BP_BATCH) {
      float v[BP_BATCH][PL];
#pragma unroll
      for (int b = 0; b < BP_BATCH; ++b) {
        const int jj = min(j4 + 4 * b, nj - 1);  // past the last: its window again, not stored
        const int ray = __builtin_amdgcn_readlane(base, js + jj) + w;
        // the whole offset in the register, so that the range check sees a ray below 0
        int fwd = 4 * ray, rev = 4 * (R - 1) - 4 * ray;
        __asm__ volatile("" : "+v"(fwd), "+v"(rev));
        const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(
            (void*)(sl + (size_t)(jb + jj) * R), (short)0, R * (int)sizeof(float), SS_RSRC_DWORD3);
        v[b][0] = ss_raw_load_f32(rs, fwd, 0, 0);
        if (PL >= 2) v[b][PL >= 2 ? 1 : 0] = ss_raw_load_f32(rs, rev, 0, 0);
        if (PL == 4) {
          const SSBpMirror m = ss_bp_mirror(jb + jj, A);
          const __amdgpu_buffer_rsrc_t rm = __builtin_amdgcn_make_buffer_rsrc(
              (void*)(sl + (size_t)m.row * R), (short)0, R * (int)sizeof(float), SS_RSRC_DWORD3);
          v[b][PL == 4 ? 2 : 0] = ss_raw_load_f32(rm, m.flip ? rev : fwd, 0, 0);
          v[b][PL == 4 ? 3 : 0] = ss_raw_load_f32(rm, m.flip ? fwd : rev, 0, 0);
        }
      }
#pragma unroll
      for (int b = 0; b < BP_BATCH; ++b) {
        const int jj = j4 + 4 * b;
        // (v0 - w d, d): the value at u in [w, w + 1) is then fma(u, d, first), so the
        // interpolation needs no fraction of u
        float f[PL], d[PL];
#pragma unroll
        for (int z = 0; z < PL; ++z) {  // every lane takes part in the lane shift
          d[z] = ss_next_lane(v[b][z]) - v[b][z];
          f[z] = fmaf(fw, d[z], v[b][z]);
        }
        if (jj < nj && lane < SS_WAVE - 1 && w < W) {
          if (PL == 1) {
            win[jj * W + w] = make_float2(f[0], d[0]);
          } else {
            // planes 2, 3 in a window array of their own: neighbouring rays 16 bytes apart
            ss_f32x4* dst = reinterpret_cast<ss_f32x4*>(win) + jj * W + w;
#pragma unroll
            for (int z = 0; z + 1 < PL; z += 2)
              dst[z / 2 * (STAGE / 4)] = ss_f32x4{f[z], d[z], f[z + 1], d[z + 1]};
          }
        }
      }
    }
  }
}

// The values of the planes at ray offset u of one window.
template <int PL, int STAGE>
__device__ __forceinline__ void ss_bp_lerp(const float2* __restrict__ wrow, float u, float (&val)[PL]) {
  if (PL == 1) {
    const float2 t = wrow[(int)u];
    val[0] = fmaf(u, t.y, t.x);
  } else {
    const ss_f32x4* t = reinterpret_cast<const ss_f32x4*>(wrow) + (int)u;
#pragma unroll
    for (int z = 0; z + 1 < PL; z += 2) {
      const ss_f32x4 q = t[z / 2 * (STAGE / 4)];
      val[z] = fmaf(u, q.y, q.x);
      val[z + 1] = fmaf(u, q.w, q.z);
    }
  }
}

// the pixel of plane z that goes with pixel (row, col) of plane 0, and whether it is stored
// (not where it coincides with another plane's pixel, on the middle row or column)
template <int PL>
__device__ __forceinline__ bool ss_bp_plane_pixel(int z, int n, int row, int col, int* zr, int* zc) {
  *zr = (z == 1 || z == 3) ? n - 1 - row : row;
  *zc = (z == 1 || z == 2) ? n - 1 - col : col;
  if (PL == 1) return row < n && col < n;
  if (PL == 2) return 2 * row + z <= n - 1 && col < n;
  const int mr = z == 1 || z == 3, mc = z == 1 || z == 2;
  return 2 * row + mr <= n - 1 && 2 * col + mc <= n - 1;
}

// One pixel tile [c0, c0+32) x [r0, r0+8*ROWS) over angles [j0, j1).  sl points at this
// slice's angle-major sinogram; out (plain) or x/weight (EM update) at its image.
//
// The planes of the tile share each pixel's ray coordinate, its conversion and its address;
// only the interpolation and the sum are their own, and a ray's records lie together, so
// that one 16-byte LDS read returns two of them:
//   PL = 1  the pixel alone.
//   PL = 2  (SSDevPlan::bp_pair) on a grid symmetric about the rotation axis, pixel
//           (n-1-r, n-1-c) has the coordinate R - 1 - u of pixel (r, c)'s u: a window
//           holds for each ray also the record of ray R - 1 - ray.  Tiles cover the rows
//           r <= n-1-r.
//   PL = 4  (SSDevPlan::bp_quad) over all angles of a symmetric grid [0, pi): at the angle
//           pi - theta, pixel (r, n-1-c) has pixel (r, c)'s coordinate, and (n-1-r, c) its
//           reverse; a window also holds the rows of that angle.  Tiles cover a quadrant.
// Each pixel's range test is its own (a mirrored pixel re-evaluates its own FP64 expression).
// The tiles that some angles end in set a short launch's time: 45 angles of a 1024^2 image 21 us
// with a branch on each angle's flag and a test per pixel, 15 in the form below, 10 where no
// angle ends in the image; 720 angles 97 / 95, 2048^2 x 1500 587 / 570.
// VALU instructions per update in the loop: 5 / 3.5 / 2.75.
template <int MODE, int ROWS, int STAGE, int PL>
__device__ __forceinline__ void ss_bp_item(const SSDevPlan& p, const float* __restrict__ sl, int j0, int j1, int c0,
                                           int r0, float* __restrict__ out, float* __restrict__ xs,
                                           const float* __restrict__ ws, SSBpLds<STAGE>& lds) {
  const int n = p.g.n, R = p.g.nrays, A = p.g.nangles;
  const int W = p.bp_window;
  const int J = PL == 4 ? p.bp_quad : (PL == 2 ? p.bp_pair : p.bp_angles);
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int tx = PL == 1 ? tid & 31 : ss_bp_column(tid), ty = tid >> 5;
  const int col = c0 + tx;
  constexpr int TH = 8 * ROWS;
  float acc[ROWS][PL];
  float fty[ROWS];
#pragma unroll
  for (int i = 0; i < ROWS; ++i) {
#pragma unroll
    for (int z = 0; z < PL; ++z) acc[i][z] = 0.f;
    fty[i] = (float)(ty + 8 * i);
  }
  const float ftx = (float)tx;
  const float edge = ss_bp_edge(W);

  // Parameters of up to 64 angles at a time: lane l of every wave holds those of angle
  // ja + l, for as many whole stages as fit (in FP64: redone per stage they were 7% of the
  // kernel's instructions).
  const int JP = SS_WAVE / J * J;
  for (int ja = j0; ja < j1; ja += JP) {
    const int np = min(JP, j1 - ja);
    BPAngle q{0.f, 0.f, 0.f, 0, 0, 0.f, 0.f, 0};
    if (lane < np) q = ss_bp_params(p, ja + lane, c0, r0, TH);
    // the angles that are interior for this tile run without predicates
    const unsigned long long interior = __ballot(lane < np && q.flag == 1);
    const unsigned long long ending = __ballot(lane < np && q.flag == 2);
    for (int js = 0; js < np; js += J) {
      const int jb = ja + js, nj = min(J, np - js);
      const bool mixed = __popcll(interior >> js & (~0ull >> (SS_WAVE - nj))) != nj;
      __syncthreads();  // the previous stage (or item) is done with win / par
      if (js == 0 && wv == 0) {  // the used fields only (whole-struct copies kept the padding in scratch)
        lds.par[lane].f0 = q.f0;
        lds.par[lane].b = q.b;
        lds.par[lane].c = q.c;
        lds.par[lane].lo = (float)(-q.base) + edge;
        lds.par[lane].hi = (float)(R - 1 - q.base) - edge;
      }
      // base is at least one ray below the tile's lowest U, so every pixel has u >= 1 and
      // (int)u < W - 1
      ss_bp_stage<PL, STAGE>(sl, R, A, W, jb, nj, wv, lane, q.base, js, lds.win);
      __syncthreads();
      // one angle's updates from its window: u >= 1, so truncation is the floor
      auto add = [&](const ss_f32x4& par, const float2* wrow) {
        const float t0 = fmaf(ftx, par.y, par.x);
#pragma unroll
        for (int i = 0; i < ROWS; ++i) {
          float val[PL];
          ss_bp_lerp<PL, STAGE>(wrow, fmaf(fty[i], par.z, t0), val);
#pragma unroll
          for (int z = 0; z < PL; ++z) acc[i][z] += val[z];
        }
      };
      constexpr int RW = PL == 1 ? 1 : 2;  // records of a ray in a window array
      if (!mixed) {
#pragma unroll 2
        for (int jj = 0; jj < nj; ++jj)
          add(*reinterpret_cast<const ss_f32x4*>(&lds.par[js + jj]), lds.win + jj * RW * W);  // f0, b, c
      } else {
        // Some angles end in this tile or miss it.  By the scalar masks (a flag read per angle put
        // two LDS latencies in a row before its updates): first the interior ones, then those that
        // end here with per-pixel 0 <= m <= R-2 tests; two angles at a time.  Pixels within `edge`
        // rays of an end are left out and take the reference's FP64 expression afterwards; most
        // stages have none.
        const unsigned long long mask = ~0ull >> (SS_WAVE - nj);
        auto two = [&](unsigned long long m, auto&& one) {
          while (m) {
            const int j1 = __builtin_ctzll(m);
            m &= m - 1;
            if (m) {
              const int j2 = __builtin_ctzll(m);
              m &= m - 1;
              one(j1);
              one(j2);
            } else {
              one(j1);
            }
          }
        };
        two(interior >> js & mask, [&](int jj) {
          add(*reinterpret_cast<const ss_f32x4*>(&lds.par[js + jj]), lds.win + jj * RW * W);
        });
        bool near = false;
        const unsigned long long ends = ending >> js & mask;
        two(ends, [&](int jj) {
          const ss_f32x4 par = *reinterpret_cast<const ss_f32x4*>(&lds.par[js + jj]);
          const float lo = lds.par[js + jj].lo, hi = lds.par[js + jj].hi;
          const float t0 = fmaf(ftx, par.y, par.x);
#pragma unroll
          for (int i = 0; i < ROWS; ++i) {
            const float u = fmaf(fty[i], par.z, t0);
            const bool in = __builtin_amdgcn_fmed3f(u, lo, hi) == u;
            near = near || (!in && __builtin_amdgcn_fmed3f(u, lo - 2.f * edge, hi + 2.f * edge) == u);
            float val[PL];
            ss_bp_lerp<PL, STAGE>(lds.win + jj * RW * W, u, val);
#pragma unroll
            for (int z = 0; z < PL; ++z) acc[i][z] += in ? val[z] : 0.f;
          }
        });
        if (__ballot(near) != 0ull) {
          for (unsigned long long m = ends; m; m &= m - 1) {
            const int jj = __builtin_ctzll(m);
            const ss_f32x4 par = *reinterpret_cast<const ss_f32x4*>(&lds.par[js + jj]);
            const float lo = lds.par[js + jj].lo, hi = lds.par[js + jj].hi;
            const float t0 = fmaf(ftx, par.y, par.x);
            const int jm = PL == 4 ? ss_bp_mirror(jb + jj, A).row : jb + jj;
#pragma unroll
            for (int i = 0; i < ROWS; ++i) {
              const float u = fmaf(fty[i], par.z, t0);
              if (__builtin_amdgcn_fmed3f(u, lo, hi) == u ||
                  __builtin_amdgcn_fmed3f(u, lo - 2.f * edge, hi + 2.f * edge) != u)
                continue;
              float val[PL];
              ss_bp_lerp<PL, STAGE>(lds.win + jj * RW * W, u, val);
#pragma unroll
              for (int z = 0; z < PL; ++z) {
                int zr, zc;
                (void)ss_bp_plane_pixel<PL>(z, n, r0 + ty + 8 * i, col, &zr, &zc);
                acc[i][z] += ss_bp_exact_valid(p, z >= 2 ? jm : jb + jj, zr, zc) ? val[z] : 0.f;
              }
            }
          }
        }
      }
    }
  }
  const float dth = (float)p.g.dth;
#pragma unroll
  for (int i = 0; i < ROWS; ++i) {
#pragma unroll
    for (int z = 0; z < PL; ++z) {
      int zr, zc;
      if (!ss_bp_plane_pixel<PL>(z, n, r0 + ty + 8 * i, col, &zr, &zc)) continue;
      const size_t idx = (size_t)zr * n + zc;
      const float bp = acc[i][z] * dth;
      if (MODE == SS_BP_PLAIN) {
        out[idx] = bp;
      } else if (MODE == SS_BP_PARTIAL) {
        out[idx] = acc[i][z];
      } else {
        const float wgt = ws[idx];
        const float x = xs[idx];
        xs[idx] = wgt > 0.f ? x * bp / wgt : x;
      }
    }
  }
}

// blockIdx.z = slice * ngroups + g.  SS_BP_PARTIAL: group g takes angles
// [j0 + g*nj/ngroups, j0 + (g+1)*nj/ngroups) and writes its unscaled sums to
// out[slice][g][n][n]; the other modes have ngroups = 1.
template <int MODE, int ROWS, int STAGE, int PL>
__global__ __launch_bounds__(256) void k_backprojection(SSDevPlan p, const float* __restrict__ sinoT, int j0, int j1,
                                                        int ngroups, float* __restrict__ out, SSEmUpdateArgs em) {
  __shared__ SSBpLds<STAGE> lds;
  const size_t slice = blockIdx.z / (unsigned)ngroups;
  const int g = (int)(blockIdx.z % (unsigned)ngroups);
  const size_t so = slice * p.g.nangles * p.g.nrays;
  const size_t per = (size_t)p.g.n * p.g.n;
  const size_t io = slice * per;
  int ja = j0, jb = j1;
  if (MODE == SS_BP_PARTIAL) {
    const long long nj = j1 - j0;
    ja = j0 + (int)(g * nj / ngroups);
    jb = j0 + (int)((g + 1) * nj / ngroups);
  }
  float* dst = MODE == SS_BP_PLAIN ? out + io : (MODE == SS_BP_PARTIAL ? out + (slice * ngroups + g) * per : nullptr);
  ss_bp_item<MODE, ROWS, STAGE, PL>(p, sinoT + so, ja, jb, blockIdx.x * BP_TILE_W, blockIdx.y * 8 * ROWS, dst,
                                MODE == SS_BP_EM_UPDATE ? em.x + io : nullptr,
                                MODE == SS_BP_EM_UPDATE ? em.weight : nullptr, lds);
}

// The OSEM weights W_b = BP_b(1) of the subsets [b A / S, (b + 1) A / S), to out[b][n][n]: between
// two rays the backprojection of ones adds 1, so a pixel's sum is the count of the subset's
// angles whose ray coordinate lies on the detector, by the test of ss_bp_item.  A block takes
// a 32 x 32 pixel tile (and subset b0 + blockIdx.z), a wave's lanes the flags of 64 angles at a
// time: angles interior to the tile add to all its pixels at once, only those that end in it are
// tested per pixel.  1024^2, 16 subsets of 45 angles: 365 us as 16 backprojections, 47 here (the
// angles' FP64 terms and one wait for their loads per block).  SPLIT: launches of few tiles walk
// their angles too long (226^2, one subset of 449, an iteration: 117 us, split 84), so a block takes
// 32 x 8 pixels and each of its SPLIT waves all of them for its part of the angles: 4, and for the
// smallest launches 16 (one subset of 457 angles, many of them ending in a tile, 170^2: 37 us with
// 4 waves, 14 with 16, 25 as a backprojection of ones; an OSEM call of 1024^2 x 457 in one subset 390
// with 4, 417 with 16).
template <int SPLIT>
__global__ __launch_bounds__(SPLIT ? SPLIT * SS_WAVE : 256) void k_bp_weights(SSDevPlan p, int S, int b0,
                                                                             float* __restrict__ out) {
  const int n = p.g.n, R = p.g.nrays, A = p.g.nangles, b = b0 + blockIdx.z;
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  constexpr int TH = SPLIT ? 8 : 32, STEP = SPLIT ? 2 : 8;  // tile rows, rows between a thread's pixels
  const int tx = threadIdx.x & 31, ty = (SPLIT ? lane : (int)threadIdx.x) >> 5;
  const int c0 = blockIdx.x * BP_TILE_W, r0 = blockIdx.y * TH;
  const int col = c0 + tx;
  int j0 = (int)((long long)b * A / S), j1 = (int)((long long)(b + 1) * A / S);
  if (SPLIT) {
    const int nj = j1 - j0;
    j1 = j0 + (int)((wv + 1LL) * nj / SPLIT);
    j0 += (int)((long long)wv * nj / SPLIT);
  }
  const float edge = ss_bp_edge(2 * p.bp_window);  // these tiles may be twice the plan's
  int all = 0, count[4] = {0, 0, 0, 0};
  for (int ja = j0; ja < j1; ja += SS_WAVE) {
    const int np = min(SS_WAVE, j1 - ja);
    const BPAngle q = lane < np ? ss_bp_params(p, ja + lane, c0, r0, TH) : BPAngle{0.f, 0.f, 0.f, 0, 0, 0.f, 0.f, 0};
    all += __popcll(__ballot(q.flag == 1));
    for (unsigned long long mixed = __ballot(q.flag == 2); mixed; mixed &= mixed - 1) {
      const int jj = __builtin_ctzll(mixed);
      const float f0 = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(q.f0), jj));
      const float pb = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(q.b), jj));
      const float pc = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(q.c), jj));
      const int base = __builtin_amdgcn_readlane(q.base, jj);
      const float t0 = fmaf((float)tx, pb, f0), lo = (float)(-base), hi = (float)(R - 1 - base);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float u = fmaf((float)(ty + STEP * i), pc, t0);
        if (u > lo + edge && u < hi - edge)
          ++count[i];
        else if (!(u < lo - edge || u > hi + edge))
          count[i] += ss_bp_exact_valid(p, ja + jj, r0 + ty + STEP * i, col);
      }
    }
  }
  const float dth = (float)p.g.dth;
  if constexpr (SPLIT) {
    __shared__ int part[SPLIT][TH * 32];
#pragma unroll
    for (int i = 0; i < 4; ++i) part[wv][(ty + STEP * i) * 32 + tx] = all + count[i];
    __syncthreads();
    const int t = threadIdx.x, row = r0 + (t >> 5);
    if (t >= TH * 32) return;
    int sum = 0;
#pragma unroll
    for (int w = 0; w < SPLIT; ++w) sum += part[w][t];
    if (row < n && col < n) out[((size_t)b * n + row) * n + col] = (float)sum * dth;
  } else {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int row = r0 + ty + STEP * i;
      if (row < n && col < n) out[((size_t)b * n + row) * n + col] = (float)(all + count[i]) * dth;
    }
  }
}

hipError_t ss_launch_bp_weights(const SSDevPlan& p, int nsubsets, float* out, hipStream_t stream) {
  const int t = (p.g.n + 31) / 32;
  const long long tiles = (long long)t * t * nsubsets;
  const bool split = tiles <= SS_BP_ROUND_BLOCKS;
  const bool wide = 2 * tiles <= SS_BP_ROUND_BLOCKS && p.g.nangles / nsubsets >= 128;  // 8 angles a wave
  for (int b0 = 0; b0 < nsubsets; b0 += 65535) {  // grid dimension limit
    const dim3 grid(t, split ? (p.g.n + 7) / 8 : t, std::min(nsubsets - b0, 65535));
    if (wide)
      hipLaunchKernelGGL(k_bp_weights<16>, grid, dim3(16 * SS_WAVE), 0, stream, p, nsubsets, b0, out);
    else if (split)
      hipLaunchKernelGGL(k_bp_weights<4>, grid, dim3(4 * SS_WAVE), 0, stream, p, nsubsets, b0, out);
    else
      hipLaunchKernelGGL(k_bp_weights<0>, grid, dim3(256), 0, stream, p, nsubsets, b0, out);
  }
  return hipGetLastError();
}

// the groups' partial sums of each pixel added in group order, times dtheta, stored
// (SS_BP_PLAIN) or applied as x <- x * bp / w (SS_BP_EM_UPDATE), as ss_bp_item stores them
template <int MODE>
__global__ __launch_bounds__(256) void k_bp_groups_finish(const float* __restrict__ part, int ngroups, int n, float dth,
                                                          float* __restrict__ out, SSEmUpdateArgs em) {
  const size_t per = (size_t)n * n;
  const size_t idx = (size_t)blockIdx.x * 256 + threadIdx.x;
  if (idx >= per) return;
  const size_t slice = blockIdx.y;
  const float* src = part + slice * ngroups * per + idx;
  float sum = 0.f;
#pragma unroll 8
  for (int g = 0; g < ngroups; ++g) sum += src[(size_t)g * per];
  const float bp = sum * dth;
  const size_t o = slice * per + idx;
  if (MODE == SS_BP_PLAIN) {
    out[o] = bp;
  } else {
    const float wgt = em.weight[idx];
    const float x = em.x[o];
    em.x[o] = wgt > 0.f ? x * bp / wgt : x;
  }
}

// Planes of a backprojection over angles [j0, j1) (see ss_bp_item)
int ss_bp_planes(const SSDevPlan& p, int j0, int j1) {
  if (p.bp_quad > 0 && j0 == 0 && j1 == p.g.nangles) return 4;
  return p.bp_pair > 0 ? 2 : 1;
}

// columns and rows that the tiles of an n x n image cover
static int ss_bp_cols(int n, int planes) { return planes == 4 ? (n + 1) / 2 : n; }
static int ss_bp_rows(int n, int planes) { return planes >= 2 ? (n + 1) / 2 : n; }
static int ss_bp_tile_cols(int n, int planes) { return (ss_bp_cols(n, planes) + BP_TILE_W - 1) / BP_TILE_W; }

int ss_bp_tiles(int n, int variant, int planes) {
  const int th = 8 * kSSBpRows[variant];
  return ss_bp_tile_cols(n, planes) * ((ss_bp_rows(n, planes) + th - 1) / th);
}

// angle groups of a launch of `tiles` blocks over nj angles (the rule at SS_BP_GROUP_SCALE)
static int ss_angle_groups(long long tiles, int nj) {
  if (tiles <= 0 || nj < 2 * SS_BP_GROUP_ANGLES) return 1;
  const double g = SS_BP_GROUP_SCALE * sqrt((double)SS_BP_ROUND_BLOCKS * nj / (double)tiles);
  if (g < 2.0) return 1;  // two groups cost more than they even out (SS_BP_GROUP_SCALE)
  return (int)std::min(floor(g + 0.5), (double)(nj / SS_BP_GROUP_ANGLES));
}

// Whether a backprojection has too few angles for its tiles to be divided (SS_BP_SHORT_*)
static bool ss_bp_short(const SSDevPlan& p, int j0, int j1, int nslices) {
  const long long tiles = (long long)ss_bp_tiles(p.g.n, 1, 2) * std::max(nslices, 1);  // 32 x 16 pixels, two planes
  return j1 - j0 < SS_BP_SHORT_ANGLES ||
         (tiles >= SS_BP_SHORT_TILES && j1 - j0 <= std::min(160LL, SS_BP_SHORT_ANGLES + tiles / 8));
}

int ss_bp_launch_planes(const SSDevPlan& p, int j0, int j1, int nslices) {
  const int planes = ss_bp_planes(p, j0, j1), ns = std::max(nslices, 1);
  if (planes > 1 && (long long)ss_bp_tiles(p.g.n, 1, 2) * ns * (j1 - j0) < SS_BP_PAIR_WORK) return 1;
  if (planes < 4 || p.bp_pair <= 0) return planes;
  const long long small = (long long)ss_bp_tiles(p.g.n, 1, 4) * ns, large = (long long)ss_bp_tiles(p.g.n, 0, 4) * ns;
  if (small * (j1 - j0) < SS_BP_QUAD_WORK) return 2;
  return ss_bp_short(p, j0, j1, nslices) && large < SS_BP_SHORT_QUAD ? 2 : 4;
}

int ss_bp_groups(const SSDevPlan& p, int j0, int j1, int nslices) {
  if (ss_bp_short(p, j0, j1, nslices)) return 1;
  const int planes = ss_bp_launch_planes(p, j0, j1, nslices);
  return ss_angle_groups((long long)ss_bp_tiles(p.g.n, p.bp_variant, planes) * std::max(nslices, 1), j1 - j0);
}

size_t ss_bp_scratch(const SSDevPlan& p, int j0, int j1, int nslices) {
  const int G = ss_bp_groups(p, j0, j1, nslices);
  return G > 1 ? sizeof(float) * (size_t)G * nslices * p.g.n * p.g.n : 0;
}

// variant id -> (ROWS, STAGE); must match kSSBpRows / kSSBpStage
#define SS_BP_FOR_VARIANTS(X) X(0, 4, 4096) X(1, 2, 2048) X(2, 8, 4096) X(3, 4, 2048) X(4, 2, 4096) X(5, 8, 2048)

hipError_t ss_launch_backprojection(const SSDevPlan& p, const float* sinoT, int j0, int j1, int nslices, int mode,
                                    float* out, SSEmUpdateArgs em, float* scratch, hipStream_t stream) {
  if (j1 <= j0 && mode == SS_BP_EM_UPDATE) return hipSuccess;
  const int n = p.g.n;
  const int th = 8 * kSSBpRows[p.bp_variant];
  const int G = scratch ? ss_bp_groups(p, j0, j1, nslices) : 1;
  const int kmode = G > 1 ? SS_BP_PARTIAL : mode;
  float* kout = G > 1 ? scratch : out;
  const int planes = ss_bp_launch_planes(p, j0, j1, nslices);
  dim3 grid(ss_bp_tile_cols(n, planes), (ss_bp_rows(n, planes) + th - 1) / th, nslices * G);
#define SS_BP_LAUNCH_PL(ROWS, STAGE, PL)                                                                          \
  do {                                                                                                            \
    if (kmode == SS_BP_PLAIN)                                                                                     \
      hipLaunchKernelGGL((k_backprojection<SS_BP_PLAIN, ROWS, STAGE, PL>), grid, dim3(256), 0, stream, p, sinoT, \
                         j0, j1, 1, kout, em);                                                                    \
    else if (kmode == SS_BP_PARTIAL)                                                                              \
      hipLaunchKernelGGL((k_backprojection<SS_BP_PARTIAL, ROWS, STAGE, PL>), grid, dim3(256), 0, stream, p,      \
                         sinoT, j0, j1, G, kout, em);                                                             \
    else                                                                                                          \
      hipLaunchKernelGGL((k_backprojection<SS_BP_EM_UPDATE, ROWS, STAGE, PL>), grid, dim3(256), 0, stream, p,    \
                         sinoT, j0, j1, 1, kout, em);                                                             \
  } while (0)
#define SS_BP_LAUNCH(V, ROWS, STAGE)     \
  case V:                                \
    if (planes == 4)                     \
      SS_BP_LAUNCH_PL(ROWS, STAGE, 4);   \
    else if (planes == 2)                \
      SS_BP_LAUNCH_PL(ROWS, STAGE, 2);   \
    else                                 \
      SS_BP_LAUNCH_PL(ROWS, STAGE, 1);   \
    break;
  switch (p.bp_variant) {
    SS_BP_FOR_VARIANTS(SS_BP_LAUNCH)
    default:
      return hipErrorInvalidValue;
  }
#undef SS_BP_LAUNCH
#undef SS_BP_LAUNCH_PL
  hipError_t e = hipGetLastError();
  if (e != hipSuccess || G == 1) return e;
  const size_t per = (size_t)n * n;
  dim3 fin((unsigned)((per + 255) / 256), nslices);
  if (mode == SS_BP_PLAIN)
    hipLaunchKernelGGL(k_bp_groups_finish<SS_BP_PLAIN>, fin, dim3(256), 0, stream, scratch, G, n, (float)p.g.dth, out,
                       em);
  else
    hipLaunchKernelGGL(k_bp_groups_finish<SS_BP_EM_UPDATE>, fin, dim3(256), 0, stream, scratch, G, n,
                       (float)p.g.dth, out, em);
  return hipGetLastError();
}

// =====================================================================================
// exact transpose of the Radon: image lines accumulated in LDS from the forward's own
// sample map
//
// The forward adds (1-w)*F[m] + w*F[m+1] for every valid sample (ray k, sample s), with
// m and w from the Q32.32 trajectory u = alpha0 + k*gamma + s*beta.  Its transpose
// gives pixel m the amount (1-w)*delta*q_k and pixel m+1 the amount w*delta*q_k.
//
// k_radon_transpose_lines: one wave owns one image line along the forward's sample
// axis -- image row s for branch-B angles, image column s for branch-A angles -- as
// an LDS row of n+2 cells (pixel c at index c+1, the two pads absorb m = -1 and
// m+1 = n).  For each angle of its branch, the lanes take the rays that can cross the
// line 64 at a time, step u by 64*gamma between passes, check the sample's validity
// and add the two contributions.  Each line belongs to one wave, so no global atomics
// or block barriers are needed; the LDS holds only the lines, so up to 16384-pixel
// lines fit and many waves share a CU.  The rays' exact ranges and sinogram values are
// read from global memory (the angle's rows are shared by every line, so they stay in
// cache).  Branch-B lines are image rows and are written to the output; branch-A lines
// are image columns and go to a transposed scratch image that k_transpose_add folds
// in.  Irregular rays are added by the fixup kernel afterwards.
// =====================================================================================

#define RT_LINES 8         // image lines (waves) per block
#define RT_PHASES_MAX 8    // dense rays: lane phases before falling back to LDS atomics

// LDS of k_radon_transpose_lines: one line of n+2 cells per wave, plus two spare cells
// that lanes without a sample update with zero
__host__ __device__ inline int ss_rt_line_stride(int n) { return n + 4; }
__host__ __device__ inline size_t ss_rt_line_lds(int n, int nl) {
  return sizeof(float) * (size_t)nl * ss_rt_line_stride(n);
}

// The angle table read through the constant address space: the plan's angles are not
// written while a kernel runs, so the reads are scalar loads into wave-uniform registers.
typedef __attribute__((address_space(4))) const SSAngle* ss_const_angles;

// next angle >= j of `branch` (or j1)
__device__ __forceinline__ int ss_rt_next(ss_const_angles angles, int j, int j1, int branch) {
  while (j < j1 && angles[j].branch_a != branch) ++j;
  return j;
}

// structured buffer loads of one ray's record (address = base + vindex * stride)
typedef int ss_i32x2 __attribute__((ext_vector_type(2)));
__device__ ss_i32x2 ss_struct_load_i32x2(__amdgpu_buffer_rsrc_t rsrc, int vindex, int voffset, int soffset,
                                         int aux) __asm("llvm.amdgcn.struct.ptr.buffer.load.v2i32");
__device__ float ss_struct_load_f32(__amdgpu_buffer_rsrc_t rsrc, int vindex, int voffset, int soffset,
                                    int aux) __asm("llvm.amdgcn.struct.ptr.buffer.load.f32");

// How the lanes of a pass add their two terms to the LDS line:
//   RT_DISTINCT  rays at least one cell apart (|gamma| >= 1): the lanes hit distinct cells,
//                so plain read-modify-writes, first cell m, then cell m+1, in program order
//                (the empty asm statements keep the compiler from moving an update across
//                the previous one); lanes without a sample add zero to the spare cells;
//   RT_PHASED    denser rays: the same, one phase of lanes `phases` apart at a time;
//   RT_ATOMIC    rays denser than 1/RT_PHASES_MAX cell: LDS atomics.
// In the first two every cell takes its terms in a fixed order (deterministic sums).
enum { RT_DISTINCT = 0, RT_PHASED = 1, RT_ATOMIC = 2 };

// A wave owns image line s of SL slices (SL = 2 shares the geometry work of a pass
// between two slices of a batch; every slice has its own LDS line and sinogram row).
#define RT_SL_MAX 4  // slices per wave, at most
struct SSRtLine {
  float* line[RT_SL_MAX];    // LDS lines: cell c + 1 holds pixel c; cells n+2, n+3 are spare
  int n, s;                  // line length, line index (the forward's sample)
  int k_lo, k_hi;            // candidate rays
  bool all_edge;             // every sample reads its ray's exact range
  int p_first, p_last;       // passes p_first .. p_last - 1 hold only valid samples
  int phases, my_phase;      // RT_PHASED
  __amdgpu_buffer_rsrc_t rb;     // the angle's range row (int2)
  __amdgpu_buffer_rsrc_t rq[RT_SL_MAX];  // the angle's sinogram row (float) of each slice
  int64_t gamma;             // trajectory step per ray
  int64_t u0, step;          // trajectory (+1 cell) of ray k_lo, and its step per pass
  float delta;
};

// RT_PHASED / RT_ATOMIC update of one pass on one line: trajectory u, term qd = q * delta
// (0 if the sample is not valid)
template <int MODE>
__device__ __forceinline__ void ss_rt_update(const SSRtLine& L, float* line, bool valid, int64_t u, float qd) {
  const int idx = (int)(u >> 32);
  const float wq = (float)(uint32_t)u * SS_INV_FIX * qd;
  if (MODE == RT_PHASED) {
    float* cell = line + idx;
    for (int ph = 0; ph < L.phases; ++ph) {
      const bool mine = valid && L.my_phase == ph;
      if (mine) cell[0] += qd - wq;
      __asm__ volatile("" ::: "memory");
      if (mine) cell[1] += wq;
      __asm__ volatile("" ::: "memory");
    }
  } else if (valid) {
    atomicAdd(line + idx, qd - wq);
    atomicAdd(line + idx + 1, wq);
  }
}

// One iteration over two passes (pass, pass + 1) of the candidate rays: lane 0's ray kb and
// trajectory ub (+1 cell), the passes' sinogram values q0[], q1[] per slice; loads the
// values of the next iteration's passes into n0[], n1[] (indices clamped to the last
// candidate: the loads past the last pass stay in bounds and go unused).
//
// Passes p_first .. p_last - 1 hold only valid samples (see the kernel); a pair of them
// takes a path without range checks.  Other samples near the line's ends (every sample
// of other angles) read the ray's exact range.
template <int MODE, int SL>
__device__ __forceinline__ void ss_rt_pair(const SSRtLine& L, int lane, int pass, int npass, int kb, int64_t ub,
                                           int64_t lane_u, const float* q0, const float* q1, float* n0, float* n1) {
  const int n = L.n, s = L.s, k_hi = L.k_hi, last = k_hi - 1;
  const int64_t ub1 = ub + L.step;
  const int64_t u = ub + lane_u, u1 = ub1 + lane_u;
  const int idx0 = (int)(u >> 32), idx1 = (int)(u1 >> 32);  // m + 1, in [0, n] if valid
  const int k = kb + lane;
  if (MODE == RT_DISTINCT && pass >= L.p_first && pass + 1 < L.p_last) {
    // every sample of both passes is valid
#pragma unroll
    for (int i = 0; i < SL; ++i) {
      n0[i] = ss_struct_load_f32(L.rq[i], min(k + 2 * SS_WAVE, last), 0, 0, 0);
      n1[i] = ss_struct_load_f32(L.rq[i], min(k + 3 * SS_WAVE, last), 0, 0, 0);
    }
    const float ds = L.delta * SS_INV_FIX;
    const float f0 = (float)(uint32_t)u, f1 = (float)(uint32_t)u1;
    float w0[SL], w1[SL], x0[SL], x1[SL];
    float *c0[SL], *c1[SL];
#pragma unroll
    for (int i = 0; i < SL; ++i) {
      w0[i] = f0 * (q0[i] * ds);
      w1[i] = f1 * (q1[i] * ds);
      c0[i] = L.line[i] + idx0;
      c1[i] = L.line[i] + idx1;
      x0[i] = c0[i][0];
      x1[i] = c1[i][0];
    }
#pragma unroll
    for (int i = 0; i < SL; ++i) {
      c0[i][0] = fmaf(q0[i], L.delta, x0[i]) - w0[i];
      c1[i][0] = fmaf(q1[i], L.delta, x1[i]) - w1[i];
    }
    __asm__ volatile("" ::: "memory");
#pragma unroll
    for (int i = 0; i < SL; ++i) {
      x0[i] = c0[i][1];
      x1[i] = c1[i][1];
    }
#pragma unroll
    for (int i = 0; i < SL; ++i) {
      c0[i][1] = x0[i] + w0[i];
      c1[i][1] = x1[i] + w1[i];
    }
    __asm__ volatile("" ::: "memory");
    return;
  }
  const bool two = pass + 1 < npass;  // a second pass this iteration (uniform)
  const bool e0 = L.all_edge || (unsigned)(idx0 - 2) > (unsigned)(n - 4);
  const bool e1 = two && (L.all_edge || (unsigned)(idx1 - 2) > (unsigned)(n - 4));
  ss_i32x2 b0 = {0, -1}, b1 = {0, -1};
  if (e0) b0 = ss_struct_load_i32x2(L.rb, min(k, last), 0, 0, 0);
  if (e1) b1 = ss_struct_load_i32x2(L.rb, min(k + SS_WAVE, last), 0, 0, 0);
  // issued after the ranges, so that waiting for the ranges does not wait for these
#pragma unroll
  for (int i = 0; i < SL; ++i) {
    n0[i] = ss_struct_load_f32(L.rq[i], min(k + 2 * SS_WAVE, last), 0, 0, 0);
    n1[i] = ss_struct_load_f32(L.rq[i], min(k + 3 * SS_WAVE, last), 0, 0, 0);
  }
  bool v0 = k < k_hi, v1 = k + SS_WAVE < k_hi;
  if (e0) v0 = v0 && s >= b0.x && s <= b0.y;
  if (e1) v1 = v1 && s >= b1.x && s <= b1.y;
  if (MODE == RT_DISTINCT) {
    // the first cells of both passes are distinct, and so are their second cells: read
    // both, then write both, one cell phase at a time; lanes without a sample add zero to
    // the spare cells
    const float f0 = (float)(uint32_t)u * SS_INV_FIX, f1 = (float)(uint32_t)u1 * SS_INV_FIX;
    const int i0 = v0 ? idx0 : n + 2, i1 = v1 ? idx1 : n + 2;
    float qd0[SL], qd1[SL], w0[SL], w1[SL], x0[SL], x1[SL];
    float *c0[SL], *c1[SL];
#pragma unroll
    for (int i = 0; i < SL; ++i) {
      qd0[i] = v0 ? q0[i] * L.delta : 0.f;
      qd1[i] = v1 ? q1[i] * L.delta : 0.f;
      w0[i] = f0 * qd0[i];
      w1[i] = f1 * qd1[i];
      c0[i] = L.line[i] + i0;
      c1[i] = L.line[i] + i1;
      x0[i] = c0[i][0];
      x1[i] = c1[i][0];
    }
#pragma unroll
    for (int i = 0; i < SL; ++i) {
      c0[i][0] = x0[i] + (qd0[i] - w0[i]);
      c1[i][0] = x1[i] + (qd1[i] - w1[i]);
    }
    __asm__ volatile("" ::: "memory");
#pragma unroll
    for (int i = 0; i < SL; ++i) {
      x0[i] = c0[i][1];
      x1[i] = c1[i][1];
    }
#pragma unroll
    for (int i = 0; i < SL; ++i) {
      c0[i][1] = x0[i] + w0[i];
      c1[i][1] = x1[i] + w1[i];
    }
    __asm__ volatile("" ::: "memory");
  } else {
#pragma unroll
    for (int i = 0; i < SL; ++i) {
      ss_rt_update<MODE>(L, L.line[i], v0, u, v0 ? q0[i] * L.delta : 0.f);
      if (two) ss_rt_update<MODE>(L, L.line[i], v1, u1, v1 ? q1[i] * L.delta : 0.f);
    }
  }
}

// the passes over the candidate rays, two per ss_rt_pair; the sinogram values alternate
// between two register sets (each half loads the other half's values)
template <int MODE, int SL>
__device__ __forceinline__ void ss_rt_passes(const SSRtLine& L, int lane) {
  const int npass = (L.k_hi - L.k_lo + SS_WAVE - 1) / SS_WAVE;
  const int last = L.k_hi - 1;
  const int64_t lane_u = (int64_t)lane * L.gamma;
  int64_t ub = L.u0;  // lane 0's trajectory (+1 cell)
  int kb = L.k_lo;    // lane 0's ray
  float qa[SL], qb[SL], qc[SL], qd[SL];
#pragma unroll
  for (int i = 0; i < SL; ++i) {
    qa[i] = ss_struct_load_f32(L.rq[i], min(kb + lane, last), 0, 0, 0);
    qb[i] = ss_struct_load_f32(L.rq[i], min(kb + SS_WAVE + lane, last), 0, 0, 0);
  }
  for (int pass = 0;;) {
    ss_rt_pair<MODE, SL>(L, lane, pass, npass, kb, ub, lane_u, qa, qb, qc, qd);
    pass += 2;
    kb += 2 * SS_WAVE;
    ub += 2 * L.step;
    if (pass >= npass) break;
    ss_rt_pair<MODE, SL>(L, lane, pass, npass, kb, ub, lane_u, qc, qd, qa, qb);
    pass += 2;
    kb += 2 * SS_WAVE;
    ub += 2 * L.step;
    if (pass >= npass) break;
  }
}

// slices slice0 + blockIdx.y * SL .. + SL - 1
template <int SL>
__global__ __launch_bounds__(RT_LINES * SS_WAVE) void k_radon_transpose_lines(SSDevPlan p, const float* __restrict__ qT,
                                                                             int j0, int j1, int slice0,
                                                                             float* __restrict__ outB,
                                                                             float* __restrict__ outA) {
  extern __shared__ float sh[];
  const int n = p.g.n, R = p.g.nrays, A = p.g.nangles;
  const int lane = threadIdx.x & 63;
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int nw = (int)(blockDim.x >> 6);
  const int groups = (n + nw - 1) / nw;
  const int branch = blockIdx.x >= (unsigned)groups ? 1 : 0;
  const int s = ((int)blockIdx.x - branch * groups) * nw + wv;  // image row (B) or column (A)
  if (s >= n) return;  // waves work independently: no block barrier follows
  const size_t slice = (size_t)slice0 + (size_t)blockIdx.y * SL;
  const size_t sino_size = (size_t)A * R;
  const float* q = qT + slice * sino_size;
  SSRtLine L;
  // LDS is addressed as sh + offset, so that every access compiles to an LDS instruction
#pragma unroll
  for (int i = 0; i < SL; ++i) {
    L.line[i] = sh + (wv * SL + i) * ss_rt_line_stride(n);
    for (int c = lane; c < ss_rt_line_stride(n); c += SS_WAVE) L.line[i][c] = 0.f;
  }
  L.n = n;
  L.s = s;
  const ss_const_angles angles = (ss_const_angles)p.angles;
  for (int j = ss_rt_next(angles, j0, j1, branch); j < j1; j = ss_rt_next(angles, j + 1, j1, branch)) {
    const __attribute__((address_space(4))) SSAngle& a = angles[j];
    const int64_t gamma = a.gamma;
    // candidate rays [k_lo, k_hi) of line s: ray k sits at cell x = (k + a0(s)) / rt_ig on it,
    // and a valid sample has x in [-1, n]; two rays of margin against rounding (every
    // candidate is still checked)
    const double a0 = a.rt_a0 + (double)s * a.rt_b;
    int k_lo = 0, k_hi = R;
    if (gamma != 0) {
      const double kd = floor(a.rt_w - a0) - 2.0;
      k_lo = ss_rfl((int)fmin(fmax(kd, 0.0), (double)R));
      k_hi = ss_rfl((int)fmax(fmin(kd + (double)(a.rt_wn + 5), (double)R), 0.0));
    }
    if (k_lo >= k_hi) continue;
    L.k_lo = k_lo;
    L.k_hi = k_hi;
    L.all_edge = !(a.regular && n >= 4);
    // On a regular angle a sample whose Q32.32 cell m lies in [1, n-3] is valid: the FP64
    // coordinate of the exact predicate is within ~(k + s) 2^-33 cells of the trajectory,
    // so its floor is in [0, n-2].  Those samples are the rays reaching cells [1, n-2]; the
    // passes whose 64 rays lie at least one ray inside that interval (and below k_hi) hold
    // only valid samples.
    L.p_first = 0;
    L.p_last = 0;
    if (!L.all_edge && gamma != 0) {
      const int kf = ss_rfl((int)fmin(fmax(floor(a.rt_i0 - a0) + 2.0, -1.0), (double)R));  // first fast ray
      const int kl = min(ss_rfl((int)fmin(fmax(ceil(a.rt_i1 - a0) - 2.0, -1.0), (double)R)), k_hi - 1);
      // pass p covers rays k_lo + 64 p .. k_lo + 64 p + 63
      const int pf = kf <= k_lo ? 0 : (kf - k_lo + SS_WAVE - 1) / SS_WAVE;
      const int span = kl - k_lo - (SS_WAVE - 1);
      if (span >= 0) {
        L.p_first = pf;
        L.p_last = span / SS_WAVE + 1;  // one past the last fast pass
      }
    }
    L.delta = a.delta;
    // record k of the angle's range row (8 bytes) and sinogram rows (4 bytes); every index
    // used is clamped to [0, R-1]
    L.rb = __builtin_amdgcn_make_buffer_rsrc((void*)(p.bounds + (size_t)j * R), (short)sizeof(int2),
                                             (int)((uint32_t)R * 8u), SS_RSRC_DWORD3);
#pragma unroll
    for (int i = 0; i < SL; ++i)
      L.rq[i] = __builtin_amdgcn_make_buffer_rsrc((void*)(q + i * sino_size + (size_t)j * R), (short)sizeof(float),
                                                  (int)((uint32_t)R * 4u), SS_RSRC_DWORD3);
    L.gamma = gamma;
    L.u0 = a.alpha0 + (int64_t)s * a.beta + (int64_t)k_lo * gamma + ((int64_t)1 << 32);
    L.step = (int64_t)SS_WAVE * gamma;
    const uint64_t ag = (uint64_t)(gamma < 0 ? -gamma : gamma);
    if (ag >= (uint64_t)SS_FIX_ONE_I64) {
      ss_rt_passes<RT_DISTINCT, SL>(L, lane);
    } else if (ag * RT_PHASES_MAX >= (uint64_t)SS_FIX_ONE_I64) {
      // lanes `phases` apart are at least one cell apart
      L.phases = ss_rfl((int)(((uint64_t)SS_FIX_ONE_I64 + ag - 1) / ag));
      L.my_phase = lane % L.phases;
      ss_rt_passes<RT_PHASED, SL>(L, lane);
    } else {
      ss_rt_passes<RT_ATOMIC, SL>(L, lane);
    }
  }
#pragma unroll
  for (int i = 0; i < SL; ++i) {
    float* dst = (branch ? outA : outB) + ((slice + i) * n + s) * n;
    for (int c = lane; c < n; c += SS_WAVE) dst[c] = L.line[i][c + 1];
  }
}

// out[s][r][c] += t[s][c][r], 32x32 tiles
__global__ __launch_bounds__(256) void k_transpose_add(const float* __restrict__ t, float* __restrict__ out, int n) {
  __shared__ float tile[32][33];
  const size_t off = (size_t)blockIdx.z * n * n;
  const int bx = blockIdx.x * 32, by = blockIdx.y * 32;
  const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;
  for (int yy = ty; yy < 32; yy += 8) {
    const int r = by + yy, c = bx + tx;  // t row r (image column), column c (image row)
    if (r < n && c < n) tile[yy][tx] = t[off + (size_t)r * n + c];
  }
  __syncthreads();
  for (int xx = ty; xx < 32; xx += 8) {
    const int r = bx + xx, c = by + tx;  // image row r, column c
    if (r < n && c < n) out[off + (size_t)r * n + c] += tile[tx][xx];
  }
}

// irregular rays: scatter their exact contributions
// (qT angle-major, or with in_cols in the (R, A) layout)
__global__ __launch_bounds__(256) void k_radon_transpose_fixup(SSDevPlan p, const float* __restrict__ qT, int in_cols,
                                                               int j0, int j1, float* __restrict__ out) {
  const int id = p.irregular[blockIdx.x];
  const int slice = blockIdx.y;
  const int n = p.g.n, R = p.g.nrays, A = p.g.nangles;
  const int j = id / R, k = id % R;
  if (j < j0 || j >= j1) return;
  const SSAngle& a = p.angles[j];
  const float v = qT[(size_t)slice * A * R + (in_cols ? (size_t)k * A + j : (size_t)j * R + k)] * a.delta;
  float* img = out + (size_t)slice * n * n;
  for (int s = threadIdx.x; s < n; s += blockDim.x) {
    if (!ss_radon_sample_valid(p.g, a, k, s)) continue;
    const int64_t u = a.alpha0 + (int64_t)k * a.gamma + (int64_t)s * a.beta;
    const int m = (int)(u >> 32);
    const float w = (float)(uint32_t)u * SS_INV_FIX;
    // pixel index along the interpolation axis m (weight 1-w) and m+1 (weight w)
    if (m >= 0 && m < n) {
      const size_t idx = a.branch_a ? (size_t)m * n + s : (size_t)s * n + m;
      atomicAdd(img + idx, (1.f - w) * v);
    }
    if (m + 1 >= 0 && m + 1 < n) {
      const size_t idx = a.branch_a ? (size_t)(m + 1) * n + s : (size_t)s * n + m + 1;
      atomicAdd(img + idx, w * v);
    }
  }
}

// =====================================================================================
// exact transpose, pixel-driven (rays at least one cell apart on every line)
//
// The forward adds (1-w) F[m] + w F[m+1] for a valid sample whose Q32.32 position on its
// line is u = m + w, so pixel p of line s receives Delta q_k max(0, 1 - |u_k(s) - p|)
// from ray k: a hat one cell wide.  On line s the rays sit at u_k = (alpha0 + k gamma +
// s beta) 2^-32, so the pixel lies at the real ray index
//   kappa = (p 2^32 - alpha0 - s beta) / gamma = p rt_ig - rt_a0 - s rt_b
// and ray k contributes Delta q_k max(0, 1 - g |k - kappa|), g = |gamma| 2^-32 the ray
// spacing in cells.  With g >= 1 only k0 = floor(kappa) and k0 + 1 can contribute:
//   w0 = clamp(1 - g f),  w1 = clamp(1 - g + g f),  f = kappa - k0.
// kappa is affine in the pixel's column and row (branch B: p = column, s = row; branch A:
// p = row, s = column), so a pixel tile evaluates it as the backprojection evaluates its
// detector coordinate: per angle of an LDS stage the tile origin's kappa in FP64 relative
// to a staged base ray, FP32 offsets per pixel, and staged (Delta q_k, Delta q_{k+1})
// pairs.  Both branches add into the same pixels in one pass.
//
// Validity.  A sample is valid when its FP64 predicate coordinate x lies in [0, n-1), and x is
// within ~(k + s) 2^-33 cells of the Q32.32 trajectory.  A candidate with weight lies within a
// cell of its pixel, so on pixels p in [1, n-2] every candidate that counts is valid (one at
// the very end of the line has weight zero there), and the tiles test nothing; the image's
// first and last rows and columns are made by blocks of their own (ss_rtp_border), with the
// tests.  Irregular rays enter as zeros and the fixup kernel adds them.  The weights are FP32
// evaluations of the forward's (~1e-5 cells).
//
// What bounds it: VALU issue (8 instructions per update with one plane, 5 with two, 3.5 with
// four), once the launch has enough blocks and none of the slow border tiles runs last.
// From the (R, A) layout, us before and after the planes, angle groups and border blocks:
// 2048^2 x 1500 2440 -> 660; 1024^2 x 720 550 -> 115; 512^2 x 720 490 -> 57, 64 of those
// 4110 -> 1590; 231^2 x 1000 (a limited arc) 920 -> 35.  Border tiles that test every pixel in
// place of the border blocks: 980 at 2048^2 x 1500 (the slow tiles end last).
// =====================================================================================

#ifndef RTP_UNROLL
#define RTP_UNROLL 2  // angles per unrolled step of the pixel-driven transpose
#endif

struct alignas(16) RTPAngle {
  float f0, b, c, g;  // read together by one 16-byte LDS read
  int flag;  // 0: no candidate ray on the detector, 1: regular angle, 2: not regular
  int base;
  int branch_a;
  float gs;  // signed ray spacing in cells (gamma 2^-32)
};

// Parameters of angle j for the tile [c0, c0 + 32) x [r0, r0 + th): the tile origin's kappa
// relative to the base ray, its slopes, the spacing
__device__ __forceinline__ RTPAngle ss_rtp_params(const SSDevPlan& p, int j, int c0, int r0, int th) {
  RTPAngle q{0.f, 0.f, 0.f, 0.f, 0, 0, 0, 0.f};
  const SSAngle& a = p.angles[j];
  const double kb = a.branch_a ? -a.rt_b : a.rt_ig;  // kappa per column
  const double kc = a.branch_a ? a.rt_ig : -a.rt_b;  // kappa per row
  const double K = -a.rt_a0 + (double)c0 * kb + (double)r0 * kc;
  const double eb = (double)(BP_TILE_W - 1) * kb, ec = (double)(th - 1) * kc;
  const double kmin = K + fmin(0.0, eb) + fmin(0.0, ec);
  const double kmax = K + fmax(0.0, eb) + fmax(0.0, ec);
  const double base = floor(kmin) - 1.0;
  q.f0 = (float)(K - base);
  q.b = (float)kb;
  q.c = (float)kc;
  q.g = (float)(fabs((double)a.gamma) * (1.0 / SS_FIX_ONE));
  q.gs = (float)((double)a.gamma * (1.0 / SS_FIX_ONE));
  q.base = (int)base;
  q.branch_a = a.branch_a;
  q.flag = kmax < -1.0 || kmin >= (double)p.g.nrays ? 0 : (a.regular ? 1 : 2);
  return q;
}

// The planes of a launch (ss_rt_kind chooses): a block's pixel tile
// and PL planes that share each pixel's geometry (kappa, floor, weights).  QUAD, PAIR and
// SLICES as for the Radon (ss_plane): the half turn of pixel (r, c) has the ray coordinate
// R - 1 - kappa, the mirror (r, n-1-c) has kappa at the angle pi - theta.  TURN: one slice and
// its half turn; TWO: two slices; ONE: the pixel alone.
__device__ __host__ __forceinline__ SSPlane ss_rt_plane(int kind, int z) {
  if (kind == SS_RT_TURN) return SSPlane{0, z != 0, false};
  return ss_plane(kind, z);  // SS_RT_TWO and SS_RT_ONE: slices
}

// win holds, per staged angle, the planes' values of rays base .. base + W (rt_window W;
// windows WS = W + 4 rays apart), copied straight from the pre-scaled copy (k_rtp_planes) into
// LDS: the PL values of a ray together.  A pixel reads its two candidates with two reads of
// 4 PL bytes.
template <int STAGE>
struct SSRtpLds {
  alignas(16) float win[2 * STAGE];  // J windows of PL x WS floats (border: partial sums)
  RTPAngle par[64];
};

#define RTP_EDGE_SLICES 4  // slices of a border block (they share the geometry)

// A border block: 32 pixels of an image's first or last row or column (`side` 0, 1: rows, 2,
// 3: columns; segment `seg`), over angles [j0, j1), for slices s0 .. s0 + RTP_EDGE_SLICES - 1
// (out: the first slice's image, or its partial image).
// Only here can a candidate's sample be off its line: on a regular angle the position on
// the line decides, u = p - f gs or p + (1 - f) gs, which FP32 gives within ~2e-5 cells (u in
// [eps, n-1-eps) is valid, u < -eps or u >= n-1+eps is not) except within eps = 1e-3 of an end
// and on other angles, which read the candidate's exact range.  Thread: pixel tid % 32,
// angles tid / 32 mod 8; the eight sums are added in order.
template <int STAGE>
__device__ __forceinline__ void ss_rtp_border(const SSDevPlan& p, const float* __restrict__ planes, int kind,
                                              int nslices, int j0, int j1, int side, int seg, int s0, int ngroups,
                                              float* __restrict__ out, SSRtpLds<STAGE>& lds) {
  const int n = p.g.n, R = p.g.nrays, A = p.g.nangles, PL = ss_rt_planes(kind);
  const int tid = threadIdx.x, lane = tid & 63, i = tid & 31, sub = tid >> 5;
  const bool is_row = side < 2;
  const int fixed = side & 1 ? n - 1 : 0;
  const int row = is_row ? fixed : seg * 32 + i, col = is_row ? seg * 32 + i : fixed;
  const int c0 = col & ~31, r0 = row & ~31;  // the pixel's 32 x 32 tile
  const bool on = row < n && col < n && (is_row || (row > 0 && row < n - 1));
  const float ftx = (float)(col - c0), fty = (float)(row - r0), top = (float)(n - 1);
  constexpr float eps = 1e-3f;
  const float* src[RTP_EDGE_SLICES];
#pragma unroll
  for (int s = 0; s < RTP_EDGE_SLICES; ++s) {
    const int slice = min(s0 + s, nslices - 1), per = ss_rt_slices(kind);
    // the slice's own plane in its group
    const int z = kind == SS_PLANES_PAIR ? 2 * (slice % 2) : slice % per;
    src[s] = planes + (size_t)(slice / per) * A * R * PL + z;
  }
  float acc[RTP_EDGE_SLICES];
#pragma unroll
  for (int s = 0; s < RTP_EDGE_SLICES; ++s) acc[s] = 0.f;
  for (int ja = j0; ja < j1; ja += SS_WAVE) {
    const int np = min(SS_WAVE, j1 - ja);
    __syncthreads();
    if (tid < np) lds.par[lane] = ss_rtp_params(p, ja + lane, is_row ? seg * 32 : c0, is_row ? r0 : seg * 32, 32);
    __syncthreads();
    if (!on) continue;
    for (int jj = sub; jj < np; jj += 8) {
      const RTPAngle q = lds.par[jj];
      if (q.flag == 0) continue;
      const float kap = fmaf(fty, q.c, fmaf(ftx, q.b, q.f0));
      const int k = q.base + (int)kap;
      const float f = __builtin_amdgcn_fractf(kap);
      float w0 = __builtin_amdgcn_fmed3f(fmaf(-q.g, f, 1.f), 0.f, 1.f);
      float w1 = __builtin_amdgcn_fmed3f(fmaf(q.g, f, 1.f - q.g), 0.f, 1.f);
      const int pix = q.branch_a ? row : col;  // the pixel's cell on its sample line
      if (q.flag == 2 || pix == 0 || pix == n - 1) {
        const float u0 = fmaf(-f, q.gs, (float)pix), u1 = u0 + q.gs;
        const int2* rng = p.bounds + (size_t)(ja + jj) * R;
        const int sline = q.branch_a ? col : row;  // the candidates' sample line
        // every other u near the line reads the range (testing |u - top| < eps instead left out
        // the float below top - eps, which rounds down at some n)
        bool in0 = q.flag == 1 && u0 >= eps && u0 < top - eps, in1 = q.flag == 1 && u1 >= eps && u1 < top - eps;
        if (!in0 && (q.flag == 2 || (u0 > -eps && u0 < top + eps)) && (unsigned)k < (unsigned)R) {
          const int2 b = rng[k];
          in0 = sline >= b.x && sline <= b.y;
        }
        if (!in1 && (q.flag == 2 || (u1 > -eps && u1 < top + eps)) && (unsigned)(k + 1) < (unsigned)R) {
          const int2 b = rng[k + 1];
          in1 = sline >= b.x && sline <= b.y;
        }
        w0 = in0 ? w0 : 0.f;
        w1 = in1 ? w1 : 0.f;
      }
      const size_t at = (size_t)(ja + jj) * R;
      const int k0 = min(max(k, 0), R - 1), k1 = min(max(k + 1, 0), R - 1);
#pragma unroll
      for (int s = 0; s < RTP_EDGE_SLICES; ++s) {
        const float v0 = src[s][(at + k0) * PL], v1 = src[s][(at + k1) * PL];
        acc[s] = fmaf(w0, k0 == k ? v0 : 0.f, acc[s]);  // 0 off the detector
        acc[s] = fmaf(w1, k1 == k + 1 ? v1 : 0.f, acc[s]);
      }
    }
  }
  __syncthreads();
#pragma unroll
  for (int s = 0; s < RTP_EDGE_SLICES; ++s) lds.win[(s * 8 + sub) * 32 + i] = acc[s];
  __syncthreads();
  // thread (pixel i, slice sub < 4)
  if (!on || sub >= RTP_EDGE_SLICES || s0 + sub >= nslices) return;
  float sum = 0.f;
#pragma unroll
  for (int t = 0; t < 8; ++t) sum += lds.win[(sub * 8 + t) * 32 + i];
  const size_t img = (size_t)n * n;
  out[(size_t)(s0 + sub) * ngroups * img + (size_t)row * n + col] = sum;
}

template <int PL>
struct SSRtVec {
  typedef float type __attribute__((ext_vector_type(PL)));
};
template <>
struct SSRtVec<1> {
  typedef float type;
};
template <int PL>
__device__ __forceinline__ float ss_rt_get(const typename SSRtVec<PL>::type& v, int z) {
  if constexpr (PL == 1)
    return v;
  else
    return v[z];
}

// sp: the group's pre-scaled planes [A][R][PL].  out + plane offset: the planes' images (or,
// PARTIAL, their partial images).
template <int ROWS, int STAGE, int PL>
__device__ __forceinline__ void ss_rtp_item(const SSDevPlan& p, const float* __restrict__ sp, int kind, int slice0,
                                            int nslices, int j0, int j1, int c0, int r0, float* __restrict__ out,
                                            size_t out_slice, SSRtpLds<STAGE>& lds) {
  typedef typename SSRtVec<PL>::type vec;
  const int n = p.g.n, R = p.g.nrays, A = p.g.nangles;
  const int W = p.rt_window;
  const int WS = W + 4;
  const int J = min(SS_WAVE, 2 * STAGE / PL / WS);
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int tx = PL == 4 ? ss_bp_column(tid) : tid & 31, ty = tid >> 5;
  const int col = c0 + tx;
  constexpr int TH = 8 * ROWS;
  float acc[ROWS][PL];
  float fty[ROWS];
#pragma unroll
  for (int i = 0; i < ROWS; ++i) {
    fty[i] = (float)(ty + 8 * i);
#pragma unroll
    for (int z = 0; z < PL; ++z) acc[i][z] = 0.f;
  }
  const float ftx = (float)tx;
  const int JP = SS_WAVE / J * J;  // parameters of whole stages, up to 64 angles at a time

  for (int ja = j0; ja < j1; ja += JP) {
    const int np = min(JP, j1 - ja);
    RTPAngle q{0.f, 0.f, 0.f, 0.f, 0, 0, 0, 0.f};
    if (lane < np) q = ss_rtp_params(p, ja + lane, c0, r0, TH);
    const unsigned long long near = __ballot(lane < np && q.flag != 0);
    for (int js = 0; js < np; js += J) {
      const int jb = ja + js, nj = min(J, np - js);
      const bool every = __popcll(near >> js & (~0ull >> (SS_WAVE - nj))) == nj;
      __syncthreads();  // the previous stage is done with win / par
      if (js == 0 && wv == 0) {
        lds.par[lane].f0 = q.f0;
        lds.par[lane].b = q.b;
        lds.par[lane].c = q.c;
        lds.par[lane].g = q.g;
        lds.par[lane].flag = q.flag;
      }
      // staging: wave wv fills the windows of angles wv, wv+4, ... with direct buffer -> LDS
      // copies: with four planes a ray per lane, else a float per lane.  Rays outside [0, R)
      // (and every ray of an angle without candidates) read 0 through the buffer's range
      // check.  kappa - base >= 1 for every pixel, so the truncated offset is the floor and
      // stays below W.
      for (int jj = wv; jj < nj; jj += 4) {
        const int fl = __builtin_amdgcn_readlane(q.flag, js + jj);
        const int bs = __builtin_amdgcn_readlane(q.base, js + jj);
        const __amdgpu_buffer_rsrc_t rs =
            __builtin_amdgcn_make_buffer_rsrc((void*)(sp + (size_t)(jb + jj) * R * PL), (short)0,
                                              R * PL * (int)sizeof(float), SS_RSRC_DWORD3);
        float* dst = lds.win + jj * PL * WS;
        constexpr int UNIT = PL == 4 ? 4 : 1;         // floats per lane
        const int units = PL * (W + 1) / UNIT;
        for (int w = 0; w < units; w += 64) {
          // the whole offset in the register (none in the instruction's offset field), so
          // the range check sees a ray below 0 as out of range
          int off = fl != 0 ? (PL * bs + UNIT * (w + lane)) * (int)sizeof(float) : 0x7ffffff0;
          __asm__ volatile("" : "+v"(off));
          if (w + lane < units) {  // active lanes write their unit: stay in this window
            if constexpr (PL == 4)
              __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (ss_lds_ptr)(dst + UNIT * w), 16, off, 0, 0, 0);
            else
              __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (ss_lds_ptr)(dst + UNIT * w), 4, off, 0, 0, 0);
          }
        }
      }
      __syncthreads();
      auto add = [&](const ss_f32x4& par, const vec* wrow) {  // par: f0, b, c, g
        const float g1 = 1.f - par.w;
        const float t0 = fmaf(ftx, par.y, par.x);
#pragma unroll
        for (int i = 0; i < ROWS; ++i) {
          const float kap = fmaf(fty[i], par.z, t0);
          const int kr = (int)kap;
          const float f = __builtin_amdgcn_fractf(kap);
          const float w0 = __builtin_amdgcn_fmed3f(fmaf(-par.w, f, 1.f), 0.f, 1.f);
          const float w1 = __builtin_amdgcn_fmed3f(fmaf(par.w, f, g1), 0.f, 1.f);
          const vec q0 = wrow[kr], q1 = wrow[kr + 1];
#pragma unroll
          for (int z = 0; z < PL; ++z)
            acc[i][z] = fmaf(w1, ss_rt_get<PL>(q1, z), fmaf(w0, ss_rt_get<PL>(q0, z), acc[i][z]));
        }
      };
      if (every) {
#pragma unroll RTP_UNROLL
        for (int jj = 0; jj < nj; ++jj)
          add(*reinterpret_cast<const ss_f32x4*>(&lds.par[js + jj]),
              reinterpret_cast<const vec*>(lds.win + jj * PL * WS));
      } else {
        for (int jj = 0; jj < nj; ++jj)
          if (__builtin_amdgcn_readfirstlane(lds.par[js + jj].flag))
            add(*reinterpret_cast<const ss_f32x4*>(&lds.par[js + jj]),
                reinterpret_cast<const vec*>(lds.win + jj * PL * WS));
      }
    }
  }
#pragma unroll
  for (int i = 0; i < ROWS; ++i) {
    const int row = r0 + ty + 8 * i;
#pragma unroll
    for (int z = 0; z < PL; ++z) {
      const SSPlane pl = ss_rt_plane(kind, z);
      // tiles cover the rows (and, with the mirror, the columns) up to the middle; a pixel
      // that is its own image is stored once
      const int mr = pl.turn ? 1 : 0, mc = pl.turn != pl.mirror ? 1 : 0;
      if (slice0 + pl.slice >= nslices || row >= n || col >= n) continue;
      if (kind == SS_PLANES_QUAD ? 2 * row + mr > n - 1 || 2 * col + mc > n - 1
                                 : (kind == SS_PLANES_PAIR || kind == SS_RT_TURN) && 2 * row + mr > n - 1)
        continue;
      const int zr = mr ? n - 1 - row : row, zc = mc ? n - 1 - col : col;
      if (zr == 0 || zr == n - 1 || zc == 0 || zc == n - 1) continue;  // ss_rtp_border's
      out[(size_t)pl.slice * out_slice + (size_t)zr * n + zc] = acc[i][z];
    }
  }
}

// Blocks per CU the compiler must fit (registers): eight 256-thread blocks (8 waves per
// SIMD, 64 VGPRs) for one-plane tiles of up to 4 rows per thread, whose register need is
// near 64; the planes need more.
#define RTP_MIN_BLOCKS(ROWS, PL) ((ROWS) <= 4 && (PL) == 1 ? 8 : ((ROWS) <= 4 ? 4 : 1))

// Blocks [0, nborder): the border segments (4 sides x ceil(n / 32)) of each RTP_EDGE_SLICES
// slices and angle group; then the tiles, tile fastest, then z = group * ngroups + g: planes
// group `group` over the g-th of ngroups equal parts of the angles [j0, j1).  With ngroups > 1
// the parts' partial images go to out[slice][g][n][n], for k_bp_groups_finish.
template <int ROWS, int STAGE, int PL>
__global__ __launch_bounds__(256, RTP_MIN_BLOCKS(ROWS, PL)) void k_radon_transpose_px(
    SSDevPlan p, const float* __restrict__ planes, int kind, int nslices, int j0, int j1, int ngroups, int nborder,
    int cols, int rows, float* __restrict__ out) {
  __shared__ SSRtpLds<STAGE> lds;
  const size_t img = (size_t)p.g.n * p.g.n;
  const long long nj = j1 - j0;
  int id = blockIdx.x;
  if (id < nborder) {
    const int segs = (p.g.n + 31) / 32, part = id / (4 * segs);
    const int g = part % ngroups;
    ss_rtp_border<STAGE>(p, planes, kind, nslices, j0 + (int)(g * nj / ngroups), j0 + (int)((g + 1) * nj / ngroups),
                         id / segs % 4, id % segs, part / ngroups * RTP_EDGE_SLICES, ngroups, out + g * img, lds);
    return;
  }
  id -= nborder;
  const int z = id / (cols * rows), tile = id - z * (cols * rows);
  const int ty = tile / cols, tx = tile - ty * cols;
  const int group = z / ngroups, g = z - group * ngroups;
  const int slice0 = group * ss_rt_slices(kind);
  const int ja = j0 + (int)(g * nj / ngroups), jb = j0 + (int)((g + 1) * nj / ngroups);
  ss_rtp_item<ROWS, STAGE, PL>(p, planes + (size_t)group * p.g.nangles * p.g.nrays * PL, kind, slice0, nslices, ja, jb,
                               tx * BP_TILE_W, ty * 8 * ROWS, out + ((size_t)slice0 * ngroups + g) * img,
                               ngroups * img, lds);
}

// The transpose's pre-scaled planes: out[group][a][r][z] = plane z's sinogram value at (a, r)
// times its angle's Delta, for the angles j0 .. j1 - 1 (z >= PL: none).  Read from the
// angle-major layout or (in_cols) from the (R, A) layout, which spares that its own
// transposition pass.  A block moves 32 angles x 32 rays.
template <int PL>
__global__ __launch_bounds__(256) void k_rtp_planes(SSDevPlan p, const float* __restrict__ in, int in_cols, int kind,
                                                    int nslices, int j0, int j1, float* __restrict__ out) {
  __shared__ float T[PL][32][33];
  typedef typename SSRtVec<PL>::type vec;
  const int R = p.g.nrays, A = p.g.nangles;
  const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;
  const int br = blockIdx.x * 32, ba = j0 + blockIdx.y * 32;
#pragma unroll
  for (int z = 0; z < PL; ++z) {
    const SSPlane pl = ss_rt_plane(kind, z);
    const size_t slice = (size_t)min((int)blockIdx.z * ss_rt_slices(kind) + pl.slice, nslices - 1);
    const float* src = in + slice * A * R;
#pragma unroll
    for (int yy = ty; yy < 32; yy += 8) {
      // tx runs along the input's contiguous direction
      const int a = ba + (in_cols ? tx : yy), r = br + (in_cols ? yy : tx);
      float v = 0.f;
      if (a < j1 && r < R) {
        const SSBpMirror m = pl.mirror ? ss_bp_mirror(a, A) : SSBpMirror{a, false};
        const int rz = pl.turn != m.flip ? R - 1 - r : r;
        v = src[in_cols ? (size_t)rz * A + m.row : (size_t)m.row * R + rz] * p.angles[m.row].delta;
        // irregular rays (k_radon_transpose_fixup adds them) have the range (0, -2)
        if (p.nirregular && p.bounds[(size_t)m.row * R + rz].y == -2) v = 0.f;
      }
      T[z][in_cols ? tx : yy][in_cols ? yy : tx] = v;  // [angle][ray]
    }
  }
  __syncthreads();
  vec* dst = reinterpret_cast<vec*>(out) + (size_t)blockIdx.z * A * R;
#pragma unroll
  for (int yy = ty; yy < 32; yy += 8) {
    const int a = ba + yy, r = br + tx;
    if (a >= j1 || r >= R) continue;
    vec v;
    if constexpr (PL == 1) {
      v = T[0][yy][tx];
    } else {
#pragma unroll
      for (int z = 0; z < PL; ++z) v[z] = T[z][yy][tx];
    }
    dst[(size_t)a * R + r] = v;
  }
}

// LDS a block may use on the current device (gfx950: 160 KiB, also assumed if the query
// fails)
static size_t ss_lds_per_block() {
  int dev = 0, v = 0;
  if (hipGetDevice(&dev) != hipSuccess ||
      hipDeviceGetAttribute(&v, hipDeviceAttributeMaxSharedMemoryPerBlock, dev) != hipSuccess || v <= 0)
    return 160 * 1024;
  return (size_t)v;
}

// lines (waves) per block for the line kernel holding `sl` slices per wave: the most whose
// lines fit one block's LDS (one line of the largest image, 16384 pixels, takes 64 KiB)
static int ss_rt_lines(int n, int sl) {
  const size_t budget = ss_lds_per_block();
  for (int nl = RT_LINES; nl >= 1; nl >>= 1)
    if (ss_rt_line_lds(n, nl * sl) <= budget) return nl;
  return 0;
}

// Planes of a pixel-driven transpose over angles [j0, j1) of nslices slices.  Every plane's
// arithmetic is the same in each of them, so up to SS_PLANES_STACK slices, which also share one
// slice's angle groups (ss_rt_groups), have the bits of a launch of their own; larger stacks
// choose their groups, and with them the order of the sums, by all their tiles.
static int ss_rt_kind(const SSDevPlan& p, int j0, int j1, int nslices) {
  if (4 * (p.rt_window + 4) > 2 * kSSBpStage[p.rt_variant]) return SS_RT_ONE;  // a window of four does not fit
  if (ss_planes_stack(nslices)) return SS_PLANES_SLICES;
  if ((p.rt_sym & 2) && j0 == 0 && j1 == p.g.nangles) return SS_PLANES_QUAD;
  if (p.rt_sym & 1) return nslices >= 2 ? SS_PLANES_PAIR : SS_RT_TURN;
  return nslices >= 3 ? SS_PLANES_SLICES : (nslices == 2 ? SS_RT_TWO : SS_RT_ONE);
}

static dim3 ss_rt_grid(const SSDevPlan& p, int kind) {
  const int n = p.g.n, th = 8 * kSSBpRows[p.rt_variant];
  const int cols = kind == SS_PLANES_QUAD ? (n + 1) / 2 : n;
  const int rows = kind == SS_PLANES_QUAD || kind == SS_PLANES_PAIR || kind == SS_RT_TURN ? (n + 1) / 2 : n;
  return dim3((cols + BP_TILE_W - 1) / BP_TILE_W, (rows + th - 1) / th);
}

// Angle groups, by the backprojection's rule.  Up to SS_PLANES_STACK slices take one
// slice's groups (of the form that launch has), so that their sums have the same order.
static int ss_rt_groups(const SSDevPlan& p, int j0, int j1, int nslices) {
  const int kind = ss_rt_kind(p, j0, j1, nslices);
  const int one = nslices <= SS_PLANES_STACK ? ss_rt_kind(p, j0, j1, 1) : kind;
  const dim3 grid = ss_rt_grid(p, one);
  const long long tiles = (long long)grid.x * grid.y *
                          (nslices <= SS_PLANES_STACK ? 1 : (nslices + ss_rt_slices(kind) - 1) / ss_rt_slices(kind));
  return ss_angle_groups(tiles, j1 - j0);
}

static size_t ss_rt_planes_floats(const SSDevPlan& p, int kind, int nslices) {
  const int per = ss_rt_slices(kind);
  return (size_t)((nslices + per - 1) / per) * p.g.nangles * p.g.nrays * ss_rt_planes(kind);
}

size_t ss_radon_transpose_scratch(const SSDevPlan& p, int j0, int j1, int nslices) {
  const size_t img = (size_t)nslices * p.g.n * p.g.n;
  if (p.rt_angles <= 0) return sizeof(float) * img;
  const int kind = ss_rt_kind(p, j0, j1, nslices), G = ss_rt_groups(p, j0, j1, nslices);
  return sizeof(float) * (((ss_rt_planes_floats(p, kind, nslices) + 3) & ~(size_t)3) + (G > 1 ? G * img : 0));
}

// blocks of the border (k_radon_transpose_px), and all of them
static long long ss_rt_border_blocks(const SSDevPlan& p, int nslices, int G) {
  return 4LL * ((p.g.n + 31) / 32) * ((nslices + RTP_EDGE_SLICES - 1) / RTP_EDGE_SLICES) * G;
}
static long long ss_rt_blocks(const SSDevPlan& p, int j0, int j1, int nslices) {
  const int kind = ss_rt_kind(p, j0, j1, nslices), G = ss_rt_groups(p, j0, j1, nslices), per = ss_rt_slices(kind);
  const dim3 tiles = ss_rt_grid(p, kind);
  return ss_rt_border_blocks(p, nslices, G) + (long long)tiles.x * tiles.y * ((nslices + per - 1) / per) * G;
}

int ss_radon_transpose_slices(const SSDevPlan& p, int j0, int j1, int nslices) {
  if (p.rt_angles <= 0) return nslices;
  int most = nslices;
  while (most > SS_PLANES_STACK && ss_rt_blocks(p, j0, j1, most) * 256 > SS_GRID_THREADS) most = (most / 2 + 3) & ~3;
  return most;
}

template <int PL>
static hipError_t ss_launch_rtp(const SSDevPlan& p, const float* in, int in_cols, int kind, int j0, int j1,
                                int nslices, float* out, float* scratch, hipStream_t stream) {
  const int G = ss_rt_groups(p, j0, j1, nslices);
  const int per = ss_rt_slices(kind), groups = (nslices + per - 1) / per;
  float* planes = scratch;
  float* part = scratch + ((ss_rt_planes_floats(p, kind, nslices) + 3) & ~(size_t)3);
  hipLaunchKernelGGL(k_rtp_planes<PL>, dim3((p.g.nrays + 31) / 32, (j1 - j0 + 31) / 32, groups), dim3(256), 0, stream,
                     p, in, in_cols, kind, nslices, j0, j1, planes);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  const dim3 tiles = ss_rt_grid(p, kind);
  const int nborder = (int)ss_rt_border_blocks(p, nslices, G);
  const dim3 grid(nborder + tiles.x * tiles.y * groups * G);
#define SS_RTP_LAUNCH(V, ROWS, STAGE)                                                                             \
  case V:                                                                                                         \
    hipLaunchKernelGGL((k_radon_transpose_px<ROWS, STAGE, PL>), grid, dim3(256), 0, stream, p, planes, kind,      \
                       nslices, j0, j1, G, nborder, (int)tiles.x, (int)tiles.y, G > 1 ? part : out);              \
    break;
  switch (p.rt_variant) {
    SS_BP_FOR_VARIANTS(SS_RTP_LAUNCH)
    default:
      return hipErrorInvalidValue;
  }
#undef SS_RTP_LAUNCH
  e = hipGetLastError();
  if (e != hipSuccess || G == 1) return e;
  const size_t img = (size_t)p.g.n * p.g.n;
  hipLaunchKernelGGL(k_bp_groups_finish<SS_BP_PLAIN>, dim3((unsigned)((img + 255) / 256), nslices), dim3(256), 0,
                     stream, part, G, p.g.n, 1.0f, out, SSEmUpdateArgs{nullptr, nullptr});
  return hipGetLastError();
}

hipError_t ss_launch_radon_transpose(const SSDevPlan& p, const float* sinoT, int in_cols, int j0, int j1, int nslices,
                                     float* out, float* scratch, hipStream_t stream) {
  const int n = p.g.n;
  if (p.rt_angles > 0) {  // the pixel-driven form (every angle's rays at least one cell apart)
    if (!scratch || j1 <= j0) return hipErrorInvalidValue;
    const int kind = ss_rt_kind(p, j0, j1, nslices);
    const int pl = ss_rt_planes(kind);
    const hipError_t e = pl == 4   ? ss_launch_rtp<4>(p, sinoT, in_cols, kind, j0, j1, nslices, out, scratch, stream)
                         : pl == 2 ? ss_launch_rtp<2>(p, sinoT, in_cols, kind, j0, j1, nslices, out, scratch, stream)
                                   : ss_launch_rtp<1>(p, sinoT, in_cols, kind, j0, j1, nslices, out, scratch, stream);
    if (e != hipSuccess || p.nirregular == 0) return e;
    hipLaunchKernelGGL(k_radon_transpose_fixup, dim3(p.nirregular, nslices), dim3(256), 0, stream, p, sinoT, in_cols,
                       j0, j1, out);
    return hipGetLastError();
  }
  if (in_cols) return hipErrorInvalidValue;  // the line form reads the angle-major layout
  // several slices per wave where the image is small enough for their lines to leave
  // room for many waves per CU: four for n <= 512, two for n <= 1024 (8 KiB per wave);
  // the remaining slices go in pairs, then alone
  const int quads = (n <= 512) ? nslices / 4 : 0;
  const int pairs = (n <= 1024) ? (nslices - 4 * quads) / 2 : 0;
  const int singles = nslices - 4 * quads - 2 * pairs;
  if (quads > 0) {
    const int nl = ss_rt_lines(n, 4);
    if (nl == 0) return hipErrorInvalidConfiguration;
    const int groups = (n + nl - 1) / nl;
    hipLaunchKernelGGL(k_radon_transpose_lines<4>, dim3(2 * groups, quads), dim3(nl * SS_WAVE),
                       ss_rt_line_lds(n, 4 * nl), stream, p, sinoT, j0, j1, 0, out, scratch);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
  }
  if (pairs > 0) {
    const int nl = ss_rt_lines(n, 2);
    if (nl == 0) return hipErrorInvalidConfiguration;
    const int groups = (n + nl - 1) / nl;
    hipLaunchKernelGGL(k_radon_transpose_lines<2>, dim3(2 * groups, pairs), dim3(nl * SS_WAVE),
                       ss_rt_line_lds(n, 2 * nl), stream, p, sinoT, j0, j1, 4 * quads, out, scratch);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
  }
  if (singles > 0) {
    const int nl = ss_rt_lines(n, 1);
    if (nl == 0) return hipErrorInvalidConfiguration;  // a line does not fit the LDS
    const int groups = (n + nl - 1) / nl;
    hipLaunchKernelGGL(k_radon_transpose_lines<1>, dim3(2 * groups, singles), dim3(nl * SS_WAVE),
                       ss_rt_line_lds(n, nl), stream, p, sinoT, j0, j1, 4 * quads + 2 * pairs, out, scratch);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
  }
  const int t = (n + 31) / 32;
  hipLaunchKernelGGL(k_transpose_add, dim3(t, t, nslices), dim3(256), 0, stream, scratch, out, n);
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess || p.nirregular == 0) return e;
  hipLaunchKernelGGL(k_radon_transpose_fixup, dim3(p.nirregular, nslices), dim3(256), 0, stream, p, sinoT, 0, j0, j1,
                     out);
  return hipGetLastError();
}

// =====================================================================================
// FBP row filter: circular convolution of each length-R row with g
// (g = Re(ifft(fftshift(h))), the real kernel equivalent to pyraft's lowpassino_fbp)
// 4 rows per block; g (duplicated, length 2R) and the rows in LDS.
// =====================================================================================

#define RF_ROWS 4
// out[row][k] = sum_m in[row][m] * taps[k - m + R].  toeplitz = 0: g holds R taps of a
// circular convolution (taps[j] = g[j mod R]); toeplitz = 1: g holds the 2R Toeplitz
// taps themselves (entry 0 unused).
__global__ __launch_bounds__(256) void k_ramp_filter(const float* __restrict__ in, float* __restrict__ out,
                                                     const float* __restrict__ g, int R, int nrows, int toeplitz) {
  extern __shared__ float lds[];
  float* g2 = lds;                          // 2R
  float* rows = lds + ((2 * R + 3) & ~3);   // R x RF_ROWS, interleaved [m][row], 16-byte aligned
  const int row0 = blockIdx.x * RF_ROWS;
  if (toeplitz) {
    for (int i = threadIdx.x; i < 2 * R; i += 256) g2[i] = g[i];
  } else {
    for (int i = threadIdx.x; i < R; i += 256) {
      const float v = g[i];
      g2[i] = v;
      g2[i + R] = v;
    }
  }
  for (int i = threadIdx.x; i < R * RF_ROWS; i += 256) {
    const int rr = i / R, m = i - rr * R;
    const int row = row0 + rr;
    rows[m * RF_ROWS + rr] = row < nrows ? in[(size_t)row * R + m] : 0.f;
  }
  __syncthreads();
  for (int k = threadIdx.x; k < R; k += 256) {
    float a0 = 0.f, a1 = 0.f, a2 = 0.f, a3 = 0.f;
    const float* gk = g2 + k + R;
    for (int m = 0; m < R; ++m) {
      const float gv = gk[-m];
      const float4 s = *reinterpret_cast<const float4*>(rows + m * RF_ROWS);
      a0 = fmaf(gv, s.x, a0);
      a1 = fmaf(gv, s.y, a1);
      a2 = fmaf(gv, s.z, a2);
      a3 = fmaf(gv, s.w, a3);
    }
    if (row0 + 0 < nrows) out[(size_t)(row0 + 0) * R + k] = a0;
    if (row0 + 1 < nrows) out[(size_t)(row0 + 1) * R + k] = a1;
    if (row0 + 2 < nrows) out[(size_t)(row0 + 2) * R + k] = a2;
    if (row0 + 3 < nrows) out[(size_t)(row0 + 3) * R + k] = a3;
  }
}

hipError_t ss_launch_ramp_filter(const float* in, float* out, const float* g, int R, int nrows, hipStream_t stream,
                                 bool toeplitz) {
  if (nrows <= 0) return hipSuccess;
  if (const size_t bytes = ss_fft_taps_bytes(R)) {
    // FFT form, its spectrum in stream-ordered scratch
    void* mem = nullptr;
    hipError_t e = hipMallocAsync(&mem, bytes, stream);
    if (e != hipSuccess) return e;
    SSFftTaps t;
    e = ss_fft_taps_build(g, R, toeplitz, mem, &t, stream);
    if (e == hipSuccess) e = ss_launch_fft_filter(in, out, t, nrows, stream);
    const hipError_t f = hipFreeAsync(mem, stream);
    return e != hipSuccess ? e : f;
  }
  const size_t lds = (size_t)(((2 * R + 3) & ~3) + RF_ROWS * R) * sizeof(float);
  if (lds > 160 * 1024) return hipErrorInvalidValue;
  hipLaunchKernelGGL(k_ramp_filter, dim3((nrows + RF_ROWS - 1) / RF_ROWS), dim3(256), lds, stream, in, out, g, R,
                     nrows, toeplitz ? 1 : 0);
  return hipGetLastError();
}

// =====================================================================================
// FFT form of the row filter.  With taps2[j] (j in [0, 2R)) the filter is
//   y[n] = sum_m x[m] taps2[n - m + R],   n, m in [0, R),
// where n - m + R stays in [1, 2R - 1].  Zero-padded to a power of two M >= 2R, the
// M-point circular convolution c = x (*) taps2 holds y[n] = c[n + R]: no term wraps.
// Two rows go into one complex sequence (row 2i real, row 2i + 1 imaginary); the taps
// are real, so the real and imaginary parts of c are the two rows' convolutions.
// A block computes c = IFFT(FFT(z) * G) in LDS with G = FFT(taps2), both transforms
// Stockham autosort passes (radix 4, one radix-2 pass first when log2 M is odd) over
// a table W[k] = exp(-2 pi i k / M).  The transforms run in FP64: FP32 rounding in the
// spectrum of a smooth row (large low-frequency bins, which the ramp suppresses) would
// reach 1e-5 of the filtered row at R = 2048.
// =====================================================================================

#define FF_THREADS 512

__device__ __forceinline__ double2 ss_zadd(double2 a, double2 b) { return make_double2(a.x + b.x, a.y + b.y); }
__device__ __forceinline__ double2 ss_zsub(double2 a, double2 b) { return make_double2(a.x - b.x, a.y - b.y); }
__device__ __forceinline__ double2 ss_zmul(double2 a, double2 b) {
  return make_double2(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x);
}

// The M-point DFT (INV: with exp(+2 pi i k / M), unnormalised) of the sequence in `a`,
// with `b` as the second buffer; returns the buffer holding the result.  Every thread
// of the block takes part (the passes end with block barriers).
template <bool INV>
__device__ double2* ss_fft_lds(double2* a, double2* b, const double2* __restrict__ W, int M, int lgM) {
  const int tid = threadIdx.x;
  int Ns = 1;
  if (lgM & 1) {
    const int h = M >> 1;
    for (int j = tid; j < h; j += FF_THREADS) {
      const double2 v0 = a[j], v1 = a[j + h];
      b[2 * j] = ss_zadd(v0, v1);
      b[2 * j + 1] = ss_zsub(v0, v1);
    }
    __syncthreads();
    double2* t = a;
    a = b;
    b = t;
    Ns = 2;
  }
  const int q = M >> 2;
  for (; Ns < M; Ns <<= 2) {
    const int ts = q / Ns;  // twiddle stride: exp(-2 pi i r k / (4 Ns)) = W[r k ts]
    for (int j = tid; j < q; j += FF_THREADS) {
      const int k = j & (Ns - 1);
      double2 w1 = W[k * ts], w2 = W[2 * k * ts], w3 = W[3 * k * ts];
      if (INV) {
        w1.y = -w1.y;
        w2.y = -w2.y;
        w3.y = -w3.y;
      }
      const double2 v0 = a[j], v1 = ss_zmul(a[j + q], w1), v2 = ss_zmul(a[j + 2 * q], w2),
                    v3 = ss_zmul(a[j + 3 * q], w3);
      const double2 a0 = ss_zadd(v0, v2), a1 = ss_zsub(v0, v2), a2 = ss_zadd(v1, v3), d = ss_zsub(v1, v3);
      const double2 a3 = INV ? make_double2(-d.y, d.x) : make_double2(d.y, -d.x);  // d * (+-i)
      const int o = (j - k) * 4 + k;
      b[o] = ss_zadd(a0, a2);
      b[o + Ns] = ss_zadd(a1, a3);
      b[o + 2 * Ns] = ss_zsub(a0, a2);
      b[o + 3 * Ns] = ss_zsub(a1, a3);
    }
    __syncthreads();
    double2* t = a;
    a = b;
    b = t;
  }
  return a;
}

__global__ __launch_bounds__(256) void k_fft_twiddles(double2* __restrict__ W, int M) {
  const int k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= M) return;
  double sv, cv;
  sincospi(-2.0 * (double)k / (double)M, &sv, &cv);
  W[k] = make_double2(cv, sv);
}

// G = FFT(taps2 zero-padded to M); taps2[j] = g[j] (toeplitz) or g[j mod R]
__global__ __launch_bounds__(FF_THREADS) void k_fft_taps(const float* __restrict__ g, int R, int toeplitz,
                                                         const double2* __restrict__ W, int M, int lgM,
                                                         double2* __restrict__ G) {
  extern __shared__ double2 zb[];
  double2* a = zb;
  for (int m = threadIdx.x; m < M; m += FF_THREADS) {
    double v = 0.0;
    if (m < 2 * R) v = toeplitz ? (m > 0 ? g[m] : 0.f) : g[m < R ? m : m - R];
    a[m] = make_double2(v, 0.0);
  }
  __syncthreads();
  const double2* f = ss_fft_lds<false>(a, zb + M, W, M, lgM);
  for (int m = threadIdx.x; m < M; m += FF_THREADS) G[m] = f[m];
}

// Row r of the filter's input / output: angle-major (cols = 0: row r at r * R, unit
// stride) or the (R, A) layout (cols = A: row r = slice * A + a at slice * R * A + a,
// stride A), which spares a small sinogram the layout copies around the filter.
__device__ __forceinline__ size_t ss_ff_row(int r, int R, int cols) {
  return cols > 0 ? (size_t)(r / cols) * R * cols + (r % cols) : (size_t)r * R;
}

__global__ __launch_bounds__(FF_THREADS) void k_fft_filter(const float* __restrict__ in, float* __restrict__ out,
                                                           const double2* __restrict__ G,
                                                           const double2* __restrict__ W, int R, int M, int lgM,
                                                           int nrows, int in_cols, int out_cols) {
  extern __shared__ double2 zb[];
  double2* a = zb;
  double2* b = zb + M;
  const int r0 = 2 * blockIdx.x;
  const bool two = r0 + 1 < nrows;
  const size_t is = in_cols > 0 ? (size_t)in_cols : 1;
  const float* x0 = in + ss_ff_row(r0, R, in_cols);
  const float* x1 = in + ss_ff_row(two ? r0 + 1 : r0, R, in_cols);
  for (int m = threadIdx.x; m < M; m += FF_THREADS) {
    double2 z = make_double2(0.0, 0.0);
    if (m < R) {
      z.x = x0[m * is];
      if (two) z.y = x1[m * is];
    }
    a[m] = z;
  }
  __syncthreads();
  double2* f = ss_fft_lds<false>(a, b, W, M, lgM);
  for (int m = threadIdx.x; m < M; m += FF_THREADS) f[m] = ss_zmul(f[m], G[m]);
  __syncthreads();
  const double2* c = ss_fft_lds<true>(f, f == a ? b : a, W, M, lgM);
  const double scale = 1.0 / (double)M;
  const size_t os = out_cols > 0 ? (size_t)out_cols : 1;
  float* y0 = out + ss_ff_row(r0, R, out_cols);
  float* y1 = out + ss_ff_row(two ? r0 + 1 : r0, R, out_cols);
  for (int n = threadIdx.x; n < R; n += FF_THREADS) {
    const double2 v = c[n + R];
    y0[n * os] = (float)(v.x * scale);
    if (two) y1[n * os] = (float)(v.y * scale);
  }
}

int ss_fft_size(int R, int* lg) {
  int M = 4, l = 2;
  while (M < 2 * R) {
    M <<= 1;
    ++l;
  }
  if (M > SS_FFT_MAX) return 0;
  if (lg) *lg = l;
  return M;
}

size_t ss_fft_taps_bytes(int R) {
  const int M = ss_fft_size(R, nullptr);
  return M ? 2 * sizeof(double2) * (size_t)M : 0;
}

hipError_t ss_fft_taps_build(const float* g, int R, bool toeplitz, void* mem, SSFftTaps* t, hipStream_t stream) {
  int lg = 0;
  const int M = ss_fft_size(R, &lg);
  if (!M) return hipErrorInvalidValue;
  double2* W = reinterpret_cast<double2*>(mem);
  double2* G = W + M;
  hipLaunchKernelGGL(k_fft_twiddles, dim3((M + 255) / 256), dim3(256), 0, stream, W, M);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(k_fft_taps, dim3(1), dim3(FF_THREADS), 2 * sizeof(double2) * (size_t)M, stream, g, R,
                     toeplitz ? 1 : 0, W, M, lg, G);
  e = hipGetLastError();
  if (e != hipSuccess) return e;
  t->W = W;
  t->G = G;
  t->R = R;
  t->M = M;
  t->lgM = lg;
  return hipSuccess;
}

hipError_t ss_launch_fft_filter(const float* in, float* out, const SSFftTaps& t, int nrows, hipStream_t stream,
                                int in_cols, int out_cols) {
  if (nrows <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_fft_filter, dim3((nrows + 1) / 2), dim3(FF_THREADS), 2 * sizeof(double2) * (size_t)t.M,
                     stream, in, out, t.G, t.W, t.R, t.M, t.lgM, nrows, in_cols, out_cols);
  return hipGetLastError();
}

// =====================================================================================
// transmission EM (raft/raft_transmission_em.cu:52-61)
// =====================================================================================

// expected counts: p <- flat * exp(-p) (raft/raft_radon_gpu_function.cu:31-39 with expo = -1,
// then the product with the flat field)
__global__ __launch_bounds__(256) void k_tr_expected(float* __restrict__ p, const float* __restrict__ flat, size_t n) {
  for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x)
    p[i] = flat[i] * expf(-p[i]);
}

// x <- (x * r) * r, r = b / w: the reference applies its multiplicative update twice;
// pixels with w = 0 keep their value (the reference divides unguarded)
__global__ __launch_bounds__(256) void k_tr_update(float* __restrict__ x, const float* __restrict__ b,
                                                   const float* __restrict__ w, size_t n) {
  for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x) {
    const float wi = w[i];
    if (wi != 0.f) {
      const float r = b[i] / wi;
      x[i] = (x[i] * r) * r;
    }
  }
}

hipError_t ss_launch_tr_expected(float* p, const float* flat, size_t n, hipStream_t stream) {
  hipLaunchKernelGGL(k_tr_expected, dim3(2048), dim3(256), 0, stream, p, flat, n);
  return hipGetLastError();
}

hipError_t ss_launch_tr_update(float* x, const float* b, const float* w, size_t n, hipStream_t stream) {
  hipLaunchKernelGGL(k_tr_update, dim3(2048), dim3(256), 0, stream, x, b, w, n);
  return hipGetLastError();
}

// =====================================================================================
// small helpers
// =====================================================================================

// dst = sum(partials[0..n)) in a fixed order (one block); a store, so the caller clears nothing
__global__ __launch_bounds__(256) void k_sum_partials(const double* __restrict__ partials, int n,
                                                      double* __restrict__ dst) {
  __shared__ double red[4];
  double v = 0.0;
  for (int i = threadIdx.x; i < n; i += 256) v += partials[i];
  const double tot = ss_block_sum_f64(v, red);
  if (threadIdx.x == 0) *dst = tot;
}

hipError_t ss_launch_sum_partials(const double* partials, int n, double* dst, hipStream_t stream) {
  hipLaunchKernelGGL(k_sum_partials, dim3(1), dim3(256), 0, stream, partials, n, dst);
  return hipGetLastError();
}

__global__ __launch_bounds__(256) void k_fill(float* __restrict__ p, float v, size_t n) {
  for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (size_t)gridDim.x * 256) p[i] = v;
}

hipError_t ss_launch_fill(float* p, float v, size_t n, hipStream_t stream) {
  size_t blocks = (n + 255) / 256;
  if (blocks > 65536) blocks = 65536;
  if (blocks == 0) return hipSuccess;
  hipLaunchKernelGGL(k_fill, dim3((unsigned)blocks), dim3(256), 0, stream, p, v, n);
  return hipGetLastError();
}

// =====================================================================================
// batched execution: persistent kernels over the work items of many slices
//
// A launch covers entries (slice, angle range) of a batch whose slices differ in
// n, R and A.  Items are numbered entry by entry; a fixed grid of resident blocks
// takes items blockIdx.x, blockIdx.x + gridDim.x, ...  The host orders entries by
// decreasing item cost, so the last items to run are the cheapest.  Each item runs
// the same device function as the per-plan kernels, on that slice's plan and
// buffers, so a slice's result does not depend on what it is batched with.
// =====================================================================================

// largest entry e with entries[e].item0 <= item (entries with no items are skipped
// because a later entry shares their item0)
__device__ __forceinline__ int ss_find_entry(const SSBatchEntry* __restrict__ e, int n, int item) {
  int lo = 0, hi = n - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (e[mid].item0 <= item)
      lo = mid;
    else
      hi = mid - 1;
  }
  return lo;
}

// A copy of *src held in scalar registers: the tables live in ordinary global memory,
// which the kernels also write, so the compiler would otherwise load them per lane.
template <class T>
__device__ __forceinline__ T ss_uniform_copy(const T* src) {
  static_assert(sizeof(T) % 4 == 0, "dword-sized type");
  int w[sizeof(T) / 4];
  const int* p = reinterpret_cast<const int*>(src);
#pragma unroll
  for (int i = 0; i < (int)(sizeof(T) / 4); ++i) w[i] = __builtin_amdgcn_readfirstlane(p[i]);
  T out;
  __builtin_memcpy(&out, w, sizeof(T));
  return out;
}

// The entry of `item` with every field wave-uniform: the compiler then keeps the
// slice's plan in scalar registers instead of per-lane copies.
__device__ __forceinline__ SSBatchEntry ss_entry_of(const SSBatchLaunch& L, int item) {
  const int idx = __builtin_amdgcn_readfirstlane(ss_find_entry(L.entries, L.nentries, item));
  SSBatchEntry e = L.entries[idx];
  e.slice = __builtin_amdgcn_readfirstlane(e.slice);
  e.j0 = __builtin_amdgcn_readfirstlane(e.j0);
  e.j1 = __builtin_amdgcn_readfirstlane(e.j1);
  e.item0 = __builtin_amdgcn_readfirstlane(e.item0);
  e.nslab = __builtin_amdgcn_readfirstlane(e.nslab);
  e.slab_rows = __builtin_amdgcn_readfirstlane(e.slab_rows);
  e.part_off = ss_rfl64(e.part_off);
  e.which = __builtin_amdgcn_readfirstlane(e.which);
  e.planes = __builtin_amdgcn_readfirstlane(e.planes);
  return e;
}

// GT x GT tiles with NW waves (ss_batch_gather_tile picks the shape per launch)
template <int GT, int NW>
__global__ __launch_bounds__(NW * SS_WAVE) void k_batch_gather(SSBatchLaunch L, const float* __restrict__ images,
                                                               float2* __restrict__ gA, float2* __restrict__ gB) {
  __shared__ float T[GT + 1][GT + 1];
  for (int item = blockIdx.x; item < L.total; item += gridDim.x) {
    const SSBatchEntry e = ss_entry_of(L, item);
    const SSBatchSlice s = ss_uniform_copy(L.slices + e.slice);
    const int n = s.p.g.n;
    const int tiles = (n + 2 + GT - 1) / GT;
    const int local = item - e.item0;
    const int ty = local / tiles, tx = local - ty * tiles;
    ss_gather_tile<GT, NW>(images + s.img_off, gA + s.lay_off, gB + s.lay_off, n, s.p.g.pitch, tx * GT, ty * GT, T,
                           e.which);
    __syncthreads();
  }
}

// to_t: [R][A] -> [A][R] per slice, else [A][R] -> [R][A]
__global__ __launch_bounds__(256) void k_batch_transpose(SSBatchLaunch L, const float* __restrict__ in,
                                                         float* __restrict__ out, int to_t) {
  __shared__ float tile[32][33];
  for (int item = blockIdx.x; item < L.total; item += gridDim.x) {
    const SSBatchEntry e = ss_entry_of(L, item);
    const SSBatchSlice s = ss_uniform_copy(L.slices + e.slice);
    const int rows = to_t ? s.p.g.nrays : s.p.g.nangles;
    const int cols = to_t ? s.p.g.nangles : s.p.g.nrays;
    const int tcols = (cols + 31) / 32;
    const int local = item - e.item0;
    const int ty = local / tcols, tx = local - ty * tcols;
    ss_transpose_tile(in + s.sino_off, out + s.sino_off, rows, cols, tx * 32, ty * 32, tile);
    __syncthreads();
  }
}

// Eight waves per SIMD (four 512-thread blocks per CU, as the per-plan k_radon gets): the
// slice's plan values held in scalar registers would otherwise push the kernel to 87
// VGPRs, two blocks per CU, and a second round of blocks for a 1024^2 OSEM subset.  The
// scalar values that do not fit go to VGPR lanes (no scratch memory).
//
// Item = (row slab, ray group, block of 8 angles) of an entry, slab fastest.  In
// SS_OUT_PARTIAL mode the items write their partial ray sums for k_batch_radon_finish;
// launches in the other modes are never divided into slabs.
template <int MODE>
__global__ __launch_bounds__(RADON_WAVES * SS_WAVE) __attribute__((amdgpu_waves_per_eu(8, 8))) void k_batch_radon(
    SSBatchLaunch L, const float2* __restrict__ gA, const float2* __restrict__ gB, float* __restrict__ part,
    float* __restrict__ out, const float* __restrict__ meas, double* __restrict__ ll) {
  __shared__ SSRadonLds<SSRadonShape<0>::CAP> lds;
  for (int item = blockIdx.x; item < L.total; item += gridDim.x) {
    const SSBatchEntry e = ss_entry_of(L, item);
    const SSBatchSlice* sp = L.slices + e.slice;
    SSRadonView v;
    v.angles = ss_uniform_copy(&sp->p.angles);
    v.bounds = ss_uniform_copy(&sp->p.bounds);
    v.wbounds = ss_uniform_copy(&sp->p.wbounds);
    v.ray_alpha = ss_uniform_copy(&sp->p.ray_alpha);
    v.n = ss_uniform_copy(&sp->p.g.n);
    v.R = ss_uniform_copy(&sp->p.g.nrays);
    v.A = ss_uniform_copy(&sp->p.g.nangles);
    v.pitch = ss_uniform_copy(&sp->p.g.pitch);
    v.nwaves = ss_uniform_copy(&sp->p.nwaves);
    const int64_t lay_off = ss_uniform_copy(&sp->lay_off), sino_off = ss_uniform_copy(&sp->sino_off);
    const int local = item - e.item0;
    constexpr bool divisible = MODE == SS_OUT_PARTIAL;
    const int ns = divisible ? max(e.nslab, 1) : 1;
    const int z = local % ns, r = local / ns;
    const int ablk = r / v.nwaves, grp = r - ablk * v.nwaves;
    const int rows = ns > 1 ? e.slab_rows : v.n;
    float* po = divisible ? part + e.part_off + (size_t)z * (e.j1 - e.j0) * v.R : nullptr;
    ss_radon_item<MODE, 0>(v, gA + lay_off, gB + lay_off, e.j0, e.j1, grp, ablk, z * rows, min(v.n, (z + 1) * rows),
                        out + sino_off, MODE == SS_OUT_EM_RATIO ? meas + sino_off : nullptr,
                        MODE == SS_OUT_EM_RATIO ? ll + item : nullptr, po, lds);
    __syncthreads();
  }
}

template <int MODE>
__global__ __launch_bounds__(256) void k_batch_radon_fixup(SSBatchLaunch L, const float2* __restrict__ gA,
                                                           const float2* __restrict__ gB, float* __restrict__ out,
                                                           const float* __restrict__ meas, double* __restrict__ ll) {
  __shared__ float redf[4];
  for (int item = blockIdx.x; item < L.total; item += gridDim.x) {
    const SSBatchEntry e = ss_entry_of(L, item);
    const SSBatchSlice s = ss_uniform_copy(L.slices + e.slice);
    ss_radon_fixup_item<MODE>(s.p, gA + s.lay_off, gB + s.lay_off, e.j0, e.j1, item - e.item0, out + s.sino_off,
                              MODE == SS_OUT_EM_RATIO ? meas + s.sino_off : nullptr,
                              MODE == SS_OUT_EM_RATIO ? ll + item : nullptr, redf);
    __syncthreads();
  }
}

// Item = 256 consecutive rays [j - j0][k] of an entry: the sum of its nslab partial sums,
// stored as k_batch_radon stores (EM mode: one FP64 log-likelihood partial per item).
template <int MODE>
__global__ __launch_bounds__(256) void k_batch_radon_finish(SSBatchLaunch L, const float* __restrict__ part,
                                                            float* __restrict__ out, const float* __restrict__ meas,
                                                            double* __restrict__ ll) {
  __shared__ double red[4];
  for (int item = blockIdx.x; item < L.total; item += gridDim.x) {
    const SSBatchEntry e = ss_entry_of(L, item);
    const SSBatchSlice* sp = L.slices + e.slice;
    SSRadonView v;
    v.angles = ss_uniform_copy(&sp->p.angles);
    v.R = ss_uniform_copy(&sp->p.g.nrays);
    v.A = ss_uniform_copy(&sp->p.g.nangles);
    const int64_t sino_off = ss_uniform_copy(&sp->sino_off);
    const size_t per = (size_t)(e.j1 - e.j0) * v.R;
    const size_t idx = (size_t)(item - e.item0) * 256 + threadIdx.x;
    double l = 0.0;
    if (idx < per) {
      const int jj = (int)(idx / (unsigned)v.R), k = (int)(idx - (size_t)jj * v.R);
      const float* src = part + e.part_off + idx;
      float sum = 0.f;
      sum = ss_slab_sum(src, per, max(e.nslab, 1));
      ss_radon_store<MODE>(v, e.j0 + jj, k, sum * v.angles[e.j0 + jj].delta, out + sino_off,
                           MODE == SS_OUT_EM_RATIO ? meas + sino_off : nullptr, &l);
    }
    if (MODE == SS_OUT_EM_RATIO) {
      const double tot = ss_block_sum_f64(l, red);
      if (threadIdx.x == 0) ll[item] = tot;
    }
    __syncthreads();
  }
}

template <int MODE, int ROWS, int STAGE>
__global__ __launch_bounds__(256) void k_batch_bp(SSBatchLaunch L, const float* __restrict__ sinoT,
                                                  float* __restrict__ out, float* __restrict__ x,
                                                  const float* __restrict__ weight) {
  __shared__ SSBpLds<STAGE> lds;
  constexpr int TH = 8 * ROWS;
  for (int item = blockIdx.x; item < L.total; item += gridDim.x) {
    const SSBatchEntry e = ss_entry_of(L, item);
    const SSBatchSlice s = ss_uniform_copy(L.slices + e.slice);
    const int planes = e.planes;  // uniform over the block; 4 only over whole ranges (SS_BP_PLAIN)
    const int tiles_x = ((planes == 4 ? (s.p.g.n + 1) / 2 : s.p.g.n) + BP_TILE_W - 1) / BP_TILE_W;
    const int local = item - e.item0;
    const int ty = local / tiles_x, tx = local - ty * tiles_x;
    float* o = MODE == SS_BP_PLAIN ? out + s.img_off : nullptr;
    float* xs = MODE == SS_BP_PLAIN ? nullptr : x + s.img_off;
    const float* ws = MODE == SS_BP_PLAIN ? nullptr : weight + s.img_off;
    if (MODE == SS_BP_PLAIN && planes == 4)
      ss_bp_item<MODE, ROWS, STAGE, MODE == SS_BP_PLAIN ? 4 : 2>(s.p, sinoT + s.sino_off, e.j0, e.j1, tx * BP_TILE_W,
                                                                 ty * TH, o, xs, ws, lds);
    else if (planes == 2)
      ss_bp_item<MODE, ROWS, STAGE, 2>(s.p, sinoT + s.sino_off, e.j0, e.j1, tx * BP_TILE_W, ty * TH, o, xs, ws, lds);
    else
      ss_bp_item<MODE, ROWS, STAGE, 1>(s.p, sinoT + s.sino_off, e.j0, e.j1, tx * BP_TILE_W, ty * TH, o, xs, ws, lds);
    __syncthreads();
  }
}

// resident blocks per CU of each batched kernel, from the runtime's occupancy query
namespace {
template <class K>
int ss_resident_blocks(K kernel, int block) {
  int per_cu = 0;
  if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kernel, block, 0) != hipSuccess || per_cu < 1) per_cu = 1;
  int dev = 0, cus = 0;
  if (hipGetDevice(&dev) != hipSuccess ||
      hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cus < 1)
    cus = 256;
  return per_cu * cus;
}
}  // namespace

// Blocks take items blockIdx.x + i*gridDim.x.  Item costs repeat with the ray-group
// or tile-column count of a slice (often a power of two), so a grid that shares a
// factor with it would hand some blocks only the long central rays; a prime grid
// larger than any such period gives every block the full mix.
static int ss_prime_at_most(int g) {
  for (; g > 2; --g) {
    bool prime = (g % 2) != 0;
    for (int d = 3; prime && d * d <= g; d += 2) prime = (g % d) != 0;
    if (prime) return g;
  }
  return g;
}

int ss_batch_grid(int kind, int variant, int mode, int total) {
  if (total <= 0) return 0;
  // the layout kernels' items are single tiles: one block per item lets the dispatcher
  // overlap their loads and stores across blocks, where a resident grid walks its items
  // one after another (4% of a batched OSEM iteration at 256 slices)
  if (kind == SS_KIND_GATHER || kind == SS_KIND_TRANSPOSE || kind == SS_KIND_RADON_FINISH) return total;
  int g = 0;
  switch (kind) {
    case SS_KIND_RADON:
      g = mode == SS_OUT_EM_RATIO  ? ss_resident_blocks(k_batch_radon<SS_OUT_EM_RATIO>, RADON_WAVES * SS_WAVE)
          : mode == SS_OUT_PARTIAL ? ss_resident_blocks(k_batch_radon<SS_OUT_PARTIAL>, RADON_WAVES * SS_WAVE)
                                   : ss_resident_blocks(k_batch_radon<SS_OUT_SINOT>, RADON_WAVES * SS_WAVE);
      break;
    case SS_KIND_FIXUP:
      g = ss_resident_blocks(k_batch_radon_fixup<SS_OUT_EM_RATIO>, 256);
      break;
    default: {
#define SS_BP_OCC(V, ROWS, STAGE)                                                               \
  case V:                                                                                       \
    g = mode == SS_BP_PLAIN ? ss_resident_blocks(k_batch_bp<SS_BP_PLAIN, ROWS, STAGE>, 256)     \
                            : ss_resident_blocks(k_batch_bp<SS_BP_EM_UPDATE, ROWS, STAGE>, 256); \
    break;
      switch (variant) {
        SS_BP_FOR_VARIANTS(SS_BP_OCC)
        default:
          g = 256;
      }
#undef SS_BP_OCC
    }
  }
  return g < total ? ss_prime_at_most(g) : total;
}

int ss_batch_gather_tile(const int* n, int count) {
  long long big = 0;
  for (int i = 0; i < count; ++i) big += (long long)ss_gather_tiles(n[i]) * ss_gather_tiles(n[i]);
  return big >= 1024 ? SS_GATHER_TILE : 32;  // the per-plan rule: at least 4 large tiles per CU
}

hipError_t ss_launch_batch_gather(const SSBatchLaunch& L, int tile, const float* images, float2* gatherA,
                                  float2* gatherB, hipStream_t stream) {
  if (L.total <= 0) return hipSuccess;
  if (tile == SS_GATHER_TILE)
    hipLaunchKernelGGL((k_batch_gather<SS_GATHER_TILE, 8>), dim3(L.grid), dim3(8 * SS_WAVE), 0, stream, L, images,
                       gatherA, gatherB);
  else
    hipLaunchKernelGGL((k_batch_gather<32, 4>), dim3(L.grid), dim3(4 * SS_WAVE), 0, stream, L, images, gatherA,
                       gatherB);
  return hipGetLastError();
}

hipError_t ss_launch_batch_transpose(const SSBatchLaunch& L, const float* in, float* out, int to_angle_major,
                                     hipStream_t stream) {
  if (L.total <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_batch_transpose, dim3(L.grid), dim3(256), 0, stream, L, in, out, to_angle_major);
  return hipGetLastError();
}

hipError_t ss_launch_batch_radon(const SSBatchLaunch& L, const float2* gatherA, const float2* gatherB, float* part,
                                 int mode, float* out, const float* meas, double* ll_partials, hipStream_t stream) {
  if (L.total <= 0) return hipSuccess;
  const dim3 grid(L.grid), block(RADON_WAVES * SS_WAVE);
  if (part) mode = SS_OUT_PARTIAL;  // the output mode is the finishing pass's
  switch (mode) {
    case SS_OUT_PARTIAL:
      hipLaunchKernelGGL(k_batch_radon<SS_OUT_PARTIAL>, grid, block, 0, stream, L, gatherA, gatherB, part, out, meas,
                         ll_partials);
      break;
    case SS_OUT_SINO:
      hipLaunchKernelGGL(k_batch_radon<SS_OUT_SINO>, grid, block, 0, stream, L, gatherA, gatherB, part, out, meas,
                         ll_partials);
      break;
    case SS_OUT_SINOT:
      hipLaunchKernelGGL(k_batch_radon<SS_OUT_SINOT>, grid, block, 0, stream, L, gatherA, gatherB, part, out, meas,
                         ll_partials);
      break;
    default:
      hipLaunchKernelGGL(k_batch_radon<SS_OUT_EM_RATIO>, grid, block, 0, stream, L, gatherA, gatherB, part, out, meas,
                         ll_partials);
  }
  return hipGetLastError();
}

hipError_t ss_launch_batch_radon_finish(const SSBatchLaunch& L, const float* part, int mode, float* out,
                                        const float* meas, double* ll_partials, hipStream_t stream) {
  if (L.total <= 0) return hipSuccess;
  const dim3 grid(L.grid), block(256);
  switch (mode) {
    case SS_OUT_SINO:
      hipLaunchKernelGGL(k_batch_radon_finish<SS_OUT_SINO>, grid, block, 0, stream, L, part, out, meas, ll_partials);
      break;
    case SS_OUT_SINOT:
      hipLaunchKernelGGL(k_batch_radon_finish<SS_OUT_SINOT>, grid, block, 0, stream, L, part, out, meas, ll_partials);
      break;
    default:
      hipLaunchKernelGGL(k_batch_radon_finish<SS_OUT_EM_RATIO>, grid, block, 0, stream, L, part, out, meas,
                         ll_partials);
  }
  return hipGetLastError();
}

hipError_t ss_launch_batch_radon_fixup(const SSBatchLaunch& L, const float2* gatherA, const float2* gatherB, int mode,
                                       float* out, const float* meas, double* ll_partials, hipStream_t stream) {
  if (L.total <= 0) return hipSuccess;
  const dim3 grid(L.grid), block(256);
  switch (mode) {
    case SS_OUT_SINO:
      hipLaunchKernelGGL(k_batch_radon_fixup<SS_OUT_SINO>, grid, block, 0, stream, L, gatherA, gatherB, out, meas,
                         ll_partials);
      break;
    case SS_OUT_SINOT:
      hipLaunchKernelGGL(k_batch_radon_fixup<SS_OUT_SINOT>, grid, block, 0, stream, L, gatherA, gatherB, out, meas,
                         ll_partials);
      break;
    default:
      hipLaunchKernelGGL(k_batch_radon_fixup<SS_OUT_EM_RATIO>, grid, block, 0, stream, L, gatherA, gatherB, out,
                         meas, ll_partials);
  }
  return hipGetLastError();
}

hipError_t ss_launch_batch_backprojection(const SSBatchLaunch& L, int variant, const float* sinoT, int mode,
                                          float* out, float* x, const float* weight, hipStream_t stream) {
  if (L.total <= 0) return hipSuccess;
  const dim3 grid(L.grid), block(256);
#define SS_BP_BATCH(V, ROWS, STAGE)                                                                            \
  case V:                                                                                                      \
    if (mode == SS_BP_PLAIN)                                                                                   \
      hipLaunchKernelGGL((k_batch_bp<SS_BP_PLAIN, ROWS, STAGE>), grid, block, 0, stream, L, sinoT, out, x,     \
                         weight);                                                                              \
    else                                                                                                       \
      hipLaunchKernelGGL((k_batch_bp<SS_BP_EM_UPDATE, ROWS, STAGE>), grid, block, 0, stream, L, sinoT, out, x, \
                         weight);                                                                              \
    break;
  switch (variant) {
    SS_BP_FOR_VARIANTS(SS_BP_BATCH)
    default:
      return hipErrorInvalidValue;
  }
#undef SS_BP_BATCH
  return hipGetLastError();
}

// one block per slice: the slice's partial ranges summed in a fixed order
__global__ __launch_bounds__(256) void k_batch_ll(const int2* __restrict__ ranges, int nranges,
                                                  const double* __restrict__ partials, double* __restrict__ ll_out) {
  __shared__ double red[4];
  const size_t slice = blockIdx.x;
  double v = 0.0;
  for (int r = 0; r < nranges; ++r) {
    const int2 rg = ranges[slice * nranges + r];
    for (int i = threadIdx.x; i < rg.y; i += 256) v += partials[(size_t)rg.x + i];
  }
  const double tot = ss_block_sum_f64(v, red);
  if (threadIdx.x == 0) ll_out[slice] = tot;
}

hipError_t ss_launch_batch_ll(const int2* ranges, int nranges, int nslices, const double* partials, double* ll_out,
                              hipStream_t stream) {
  if (nslices <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_batch_ll, dim3(nslices), dim3(256), 0, stream, ranges, nranges, partials, ll_out);
  return hipGetLastError();
}

__global__ __launch_bounds__(256) void k_fill_f64(double* __restrict__ p, double v, size_t n) {
  for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (size_t)gridDim.x * 256) p[i] = v;
}

hipError_t ss_launch_fill_f64(double* p, double v, size_t n, hipStream_t stream) {
  size_t blocks = (n + 255) / 256;
  if (blocks > 65536) blocks = 65536;
  if (blocks == 0) return hipSuccess;
  hipLaunchKernelGGL(k_fill_f64, dim3((unsigned)blocks), dim3(256), 0, stream, p, v, n);
  return hipGetLastError();
}

// =====================================================================================
// ellipse phantoms, FP64 (raft/raft_image_phantom_fromdesc.c:4-59, raft/raft_radon_fromdesc.c:4-67)
// =====================================================================================

__global__ __launch_bounds__(256) void k_phantom(const SSEllipse* __restrict__ ell, int nell, int lines, int cols,
                                                 double tl_x, double tl_y, double hs, double vs,
                                                 double* __restrict__ out64, float* __restrict__ out32) {
  SS_NOCONTRACT
  const size_t idx = (size_t)blockIdx.x * 256 + threadIdx.x;
  if (idx >= (size_t)lines * cols) return;
  const int i = (int)(idx / cols), j = (int)(idx % cols);
  double acc = out64 ? out64[idx] : 0.0;
  for (int e = 0; e < nell; ++e) {
    const SSEllipse E = ell[e];
    const double x = tl_x + j * hs - E.x0;
    const double y = tl_y + i * vs - E.y0;
    double pv = (y * E.s) + (x * E.c);
    pv /= E.a;
    pv *= pv;
    double qv = (y * E.c) - (x * E.s);
    qv /= E.b;
    qv *= qv;
    pv += qv;
    pv = sqrt(pv);
    if (pv <= 1) acc += E.val;
  }
  if (out64) out64[idx] = acc;
  if (out32) out32[idx] = (float)acc;
}

hipError_t ss_launch_phantom(const SSEllipse* ell, int nell, int lines, int cols, double tl_x, double tl_y,
                             double hs, double vs, double* out64, float* out32, hipStream_t stream) {
  const size_t total = (size_t)lines * cols;
  hipLaunchKernelGGL(k_phantom, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, stream, ell, nell, lines, cols,
                     tl_x, tl_y, hs, vs, out64, out32);
  return hipGetLastError();
}

__global__ __launch_bounds__(256) void k_radon_fromdesc(const SSEllipseView* __restrict__ views, int nell,
                                                        int lines, int cols, double* __restrict__ out64) {
  SS_NOCONTRACT
  const size_t idx = (size_t)blockIdx.x * 256 + threadIdx.x;
  if (idx >= (size_t)lines * cols) return;
  const int i = (int)(idx / cols), j = (int)(idx % cols);
  double acc = out64[idx];
  for (int e = 0; e < nell; ++e) {
    const SSEllipseView v = views[(size_t)e * cols + j];
    double tp = v.mab * i - v.delt;
    tp *= tp;
    if (tp <= 1.0) acc += v.m * sqrt(1.0 - tp);
  }
  out64[idx] = acc;
}

hipError_t ss_launch_radon_fromdesc(const SSEllipseView* views, int nell, int lines, int cols, double* out64,
                                    hipStream_t stream) {
  const size_t total = (size_t)lines * cols;
  hipLaunchKernelGGL(k_radon_fromdesc, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, stream, views, nell,
                     lines, cols, out64);
  return hipGetLastError();
}
