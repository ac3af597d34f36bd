// dda_kernels.hip -- line-traversal (Bresenham / DDA) projector pair on gfx950.
//
// One lane per ray; the 64 lanes of a wave are 64 consecutive rays of one angle, so at
// each fast move they touch one line of pixels of the (fast, slow) layout chosen for
// the angle.  The move sequence is decided in FP64 with the reference's operation
// order (raft/raft_ddaiterator.c), so every ray visits the reference's pixels; taps
// are FP32, the Radon's ray sums FP64.
//
//   k_dda_radon_planes    Radon, four rays per lane on symmetric geometries and in stacks of
//                         slices; k_dda_pad_planes its image layouts
//   k_dda_radon           Radon, one ray per lane: sino[r][a] = sum over the ray's pixels of
//                         f(pixel) * len; k_dda_pad_images its image layouts
//   k_dda_gather_planes   transpose by pixels, four pixels per lane on the same geometries
//   k_dda_gather2, k_dda_gather  transpose by pixels, one pixel per lane and line
//   k_dda_scatter         transpose of traced angles: acc(pixel) += q * len with atomics (FP32 for
//                         R^T, FP64 for the normalised backprojection and its weights R^T 1)
//   k_dda_fold            the transpose's parts added, optionally / weights
#include "dda_kernels.h"
#include "ss_kernels.h"

#include <hip/hip_runtime.h>

#include <algorithm>

#define DDA_TILE 32

__device__ __forceinline__ bool dda_inside(int f, int s, int nf, int ns) {
  return (unsigned)f < (unsigned)nf && (unsigned)s < (unsigned)ns;
}

__device__ __forceinline__ double dda_ray_t(const SSDdaGeom& g, int r) {
  DDA_NOCONTRACT
  return g.t0 + (r * g.dt);
}

// ---------------------------------------------------------------- Radon (gather)

// The wave's fast index at which its first ray enters the image (all lanes share the
// angle, so the direction dfast): lanes wait until the wave's index reaches theirs and
// then advance with it, so at every step the active lanes sit on one line of the
// layout and their 64 taps fall in a few cache lines.
__device__ __forceinline__ int dda_wave_start(bool alive, int f, int dfast) {
  int key = alive ? (dfast > 0 ? f : -f) : 0x7fffffff;
  for (int off = 32; off > 0; off >>= 1) key = min(key, __shfl_xor(key, off));
  return dfast > 0 ? key : -key;
}

#ifndef DDA_RADON_U
#define DDA_RADON_U 8
#endif
#define DDA_RSRC_DWORD3 0x00020000  // gfx9 buffer word 3: 32-bit data format, no swizzle

// Exact-geometry angles in trapezoid form (SSDdaAngle::tr_*): the ray's length in the
// pixel at fast index k, slow index j is lmax z(|sigma_k - j|), and at most two slow
// indices per k have z > 0.  Each lane carries tau = sigma - half_s + DDA_PADW + 1 in Q32
// (integer part, 32-bit fraction), stepped by tr_d per fast index with an add and a
// carry; per k it adds q0 z0 + q1 z1 of its candidates (padded slow indices floor(tau),
// floor(tau) + 1), z from the FP32 fraction.  The wave runs the union of its lanes' fast
// ranges where a candidate can be inside the image; rows are summed in FP32 per block of
// rows, the blocks in FP64.  src is the slice's padded image (dda_pad_pitch lines).
//
// Wave-staged form (tr_wstage): per chunk of DDA_WS_ROWS fast indices the wave copies,
// for each, the DDA_WS_SEG padded pixels from one chunk-wide start sb into its own LDS
// rows, two fast indices per 16-byte buffer-to-LDS load (lanes 0-31 one, 32-63 the
// next), and then reads each lane's candidates from there with LDS reads: half the
// loads of the direct form, whose one 8-byte load per ray and fast index keeps the
// texture addresser busy.  sb is the lowest ray's floor(tau) at the chunk's first index,
// less 1 and the chunk's possible fall (tr_wgap), aligned down to 4: one scalar per
// chunk, stepped in Q32 by tr_qchunk, so the copies take a fixed lane offset and a
// scalar row offset.  Every lane's candidates on the chunk's rows then lie in
// [sb, sb + spread + (DDA_WS_ROWS - 1) |tr_d| + 9), inside the segment, and the DDA_PADW
// padding keeps the segment inside its line for every fast index of the wave's range.
// Two chunk buffers per wave: the next chunk's copies are in flight while the wave sums
// the current one.  Otherwise the direct form: one 8-byte buffer load per ray and fast
// index, the index clamped to the padded line (its padding makes the clamp exact).
//
// s_waitcnt immediates (gfx9 encoding: vmcnt bits 3:0 and 15:14, expcnt 6:4, lgkmcnt
// 11:8; a counter at its maximum is not waited on)
#define DDA_WAIT_VM0 0x0F70
#define DDA_WAIT_LGKM0 0xC07F
#define DDA_WAIT_VM_CHUNK (0x0F70 | (DDA_WS_ROWS / 2))  // vmcnt(DDA_WS_ROWS / 2), below 16
typedef float dda_f2v __attribute__((ext_vector_type(2)));
typedef __attribute__((address_space(3))) void* dda_lds_ptr;
typedef __attribute__((address_space(3))) const float* dda_lds_fptr;
__device__ dda_f2v dda_raw_load_f2(__amdgpu_buffer_rsrc_t rsrc, int voffset, int soffset,
                                   int aux) __asm("llvm.amdgcn.raw.ptr.buffer.load.v2f32");

struct SSDdaTrapState {
  int hi;
  unsigned lo;
};

__device__ __forceinline__ void dda_trap_step(const SSDdaAngle& a, SSDdaTrapState& st) {
  const unsigned lo = st.lo + a.tr_dlo;
  st.hi += a.tr_dhi + (lo < st.lo ? 1 : 0);
  st.lo = lo;
}

__device__ __forceinline__ float dda_trap_term(const SSDdaAngle& a, float x0, float x1, unsigned lo, float acc) {
  const float fr = (float)lo;
  const float z0 = __builtin_amdgcn_fmed3f(fmaf(-fabsf(a.tr_c1 - fr), a.tr_kz, a.tr_pz), 0.f, 1.f);
  const float z1 = __builtin_amdgcn_fmed3f(fmaf(fr, a.tr_kz, a.tr_pz1), 0.f, 1.f);
  return fmaf(x1, z1, fmaf(x0, z0, acc));
}

__device__ __forceinline__ SSDdaTrapState dda_trap_start(const SSDdaAngle& a, double tau0, int k) {
  const double v = fmin(fmax(fma((double)k, a.tr_d, tau0), -1073741824.0), 1073741824.0);
  const double fv = floor(v);
  SSDdaTrapState st;
  st.hi = (int)fv;
  st.lo = (unsigned)((v - fv) * 4294967296.0);
  return st;
}

// the wave's fast range: indices where floor(tau) can be in [DDA_PADW - 1,
// ns + DDA_PADW - 1] (a candidate inside the image) for some lane, one index of margin
__device__ __forceinline__ int2 dda_trap_range(const SSDdaAngle& a, double tau0, bool lane_ok, int nf, int ns) {
  const double ka = (DDA_PADW - 1.0 - tau0) / a.tr_d, kb = (ns + DDA_PADW - tau0) / a.tr_d;
  const double kl = fmax(fmin(ka, kb), -1.0), kh = fmin(fmax(ka, kb), (double)nf);
  int klo = nf, khi = -1;
  if (lane_ok && kl <= kh) {  // false for NaN
    klo = (int)fmax(0.0, floor(kl) - 1.0);
    khi = (int)fmin(nf - 1.0, ceil(kh) + 1.0);
  }
  for (int off = 32; off > 0; off >>= 1) {
    klo = min(klo, __shfl_xor(klo, off));
    khi = max(khi, __shfl_xor(khi, off));
  }
  // wave-uniform: rows in scalar registers
  return make_int2(__builtin_amdgcn_readfirstlane(klo), __builtin_amdgcn_readfirstlane(khi));
}

template <int N>
__device__ __forceinline__ float dda_trap_rows(const SSDdaAngle& a, __amdgpu_buffer_rsrc_t rs, int row_bytes,
                                               int pitch_bytes, int smax, SSDdaTrapState& st) {
  float blk = 0.f;
#pragma unroll
  for (int u = 0; u < N; ++u) {
    // below 0 wraps to a large unsigned value and clamps to smax: zeros there too
    const unsigned idx = min((unsigned)st.hi, (unsigned)smax);
    const dda_f2v q = dda_raw_load_f2(rs, (int)(idx * sizeof(float)), row_bytes + u * pitch_bytes, 0);
    blk = dda_trap_term(a, q[0], q[1], st.lo, blk);
    dda_trap_step(a, st);
  }
  return blk;
}

__device__ __forceinline__ double dda_radon_trap(const SSDdaAngle& a, const float* __restrict__ src, double t,
                                                 bool lane_ok, int nf, int ns) {
  const double tau0 = fma(t, a.tr_inv, a.tr_off);
  const int2 kr = dda_trap_range(a, tau0, lane_ok, nf, ns);
  if (kr.x > kr.y) return 0.0;
  SSDdaTrapState st = dda_trap_start(a, tau0, kr.x);
  const int pitch = dda_pad_pitch(ns);
  const int pitch_bytes = pitch * (int)sizeof(float);
  const __amdgpu_buffer_rsrc_t rs =
      __builtin_amdgcn_make_buffer_rsrc((void*)src, (short)0, nf * pitch_bytes, DDA_RSRC_DWORD3);
  double tot = 0.0;
  int k = kr.x;
  for (; k + DDA_RADON_U - 1 <= kr.y; k += DDA_RADON_U)
    tot += (double)dda_trap_rows<DDA_RADON_U>(a, rs, k * pitch_bytes, pitch_bytes, pitch - 2, st);
  for (; k <= kr.y; ++k) tot += (double)dda_trap_rows<1>(a, rs, k * pitch_bytes, pitch_bytes, pitch - 2, st);
  return lane_ok ? tot * a.tr_lmax : 0.0;
}

// copies chunk rows k0 .. k0 + nrow - 1 of the segments from sb into buf (DDA_WS_ROWS
// rows of DDA_WS_SEG floats), DDA_WS_ROWS / 2 loads
__device__ __forceinline__ void dda_ws_copy(__amdgpu_buffer_rsrc_t rs, float* buf, int k0, int sb, int nrow,
                                            int pitch_bytes, int l16, int upper) {
  const int chunk_bytes = k0 * pitch_bytes + sb * (int)sizeof(float);
  if (nrow == DDA_WS_ROWS) {
    // a fixed lane offset, the row pair as a scalar offset
    const int lane_off = l16 + upper * pitch_bytes;
#pragma unroll
    for (int i = 0; i < DDA_WS_ROWS / 2; ++i) {
      int off = lane_off;
      __asm__ volatile("" : "+v"(off));
      // the scalar offset through readfirstlane: a uniform value that instruction
      // selection placed in a vector register would otherwise become a waterfall loop
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (dda_lds_ptr)(buf + 2 * i * DDA_WS_SEG), 16, off,
                                               __builtin_amdgcn_readfirstlane(chunk_bytes + 2 * i * pitch_bytes), 0,
                                               0);
    }
  } else {
#pragma unroll
    for (int i = 0; i < DDA_WS_ROWS / 2; ++i) {
      // rows past the range repeat the last one (inside the image, never read); the whole
      // offset per lane, so that no scalar offset is built from lane values
      int off = chunk_bytes + l16 + min(2 * i + upper, nrow - 1) * pitch_bytes;
      __asm__ volatile("" : "+v"(off));
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (dda_lds_ptr)(buf + 2 * i * DDA_WS_SEG), 16, off, 0, 0, 0);
    }
  }
}

// the chunk's segment start from the lowest ray's Q32 state ql at its first index
__device__ __forceinline__ int dda_ws_start(const SSDdaAngle& a, long long ql) {
  return ((int)(ql >> 32) - 1 - a.tr_wgap) & ~3;
}

// wlds: this wave's two chunk buffers in LDS, DDA_WS_ROWS x DDA_WS_SEG floats each (the
// next chunk's copies are in flight while the wave sums the current one).  Every lane,
// also one past the last ray, reads inside its buffer: the lanes' tau is linear in the
// ray index, so each lies between the lowest lane's and that plus the wave's spread.
__device__ __forceinline__ double dda_radon_trap_ws(const SSDdaAngle& a, const float* __restrict__ src, double t,
                                                    bool lane_ok, int nf, int ns, float* wlds) {
  const double tau0 = fma(t, a.tr_inv, a.tr_off);
  const int2 kr = dda_trap_range(a, tau0, lane_ok, nf, ns);
  if (kr.x > kr.y) return 0.0;
  SSDdaTrapState st = dda_trap_start(a, tau0, kr.x);
  const int lane = threadIdx.x & 63;
  const int pitch_bytes = dda_pad_pitch(ns) * (int)sizeof(float);
  const __amdgpu_buffer_rsrc_t rs =
      __builtin_amdgcn_make_buffer_rsrc((void*)src, (short)0, nf * pitch_bytes, DDA_RSRC_DWORD3);
  const int l16 = (lane & 31) * 16;  // this lane's 16 bytes of a staged segment
  const int upper = lane >> 5;       // 1: the second fast index of a load
  // the lowest ray's Q32 state (scalar) at the first index of the next chunk to copy
  long long ql = (long long)(((unsigned long long)(unsigned)__builtin_amdgcn_readlane(st.hi, a.tr_lowlane) << 32) |
                             (unsigned)__builtin_amdgcn_readlane((int)st.lo, a.tr_lowlane));
  const int nchunk = (kr.y - kr.x) / DDA_WS_ROWS + 1;
  int sb = dda_ws_start(a, ql);
  dda_ws_copy(rs, wlds, kr.x, sb, min(DDA_WS_ROWS, kr.y - kr.x + 1), pitch_bytes, l16, upper);
  double tot = 0.0;
  for (int c = 0; c < nchunk; ++c) {
    const int k0 = kr.x + c * DDA_WS_ROWS;
    const int nrow = min(DDA_WS_ROWS, kr.y - k0 + 1);
    const float* __restrict__ cur = wlds + (c & 1) * (DDA_WS_ROWS * DDA_WS_SEG);
    int sb_next = 0;
    if (c + 1 < nchunk) {
      ql += a.tr_qchunk;
      sb_next = dda_ws_start(a, ql);
      // the other buffer's LDS reads (chunk c - 1) have returned before it is overwritten
      __builtin_amdgcn_s_waitcnt(DDA_WAIT_LGKM0);
      dda_ws_copy(rs, wlds + ((c + 1) & 1) * (DDA_WS_ROWS * DDA_WS_SEG), k0 + DDA_WS_ROWS, sb_next,
                  min(DDA_WS_ROWS, kr.y - k0 - DDA_WS_ROWS + 1), pitch_bytes, l16, upper);
      // buffer-to-LDS copies count on vmcnt, in order, and no barrier orders them here:
      // this chunk's have landed once at most the next chunk's are outstanding
      __builtin_amdgcn_s_waitcnt(DDA_WAIT_VM_CHUNK);
    } else {
      __builtin_amdgcn_s_waitcnt(DDA_WAIT_VM0);
    }
    // LDS byte address of a lane's first candidate on row u: a scalar row base plus 4 hi
    const int base = __builtin_amdgcn_readfirstlane((int)(size_t)(dda_lds_fptr)cur) - 4 * sb;
    float blk = 0.f;
    if (nrow == DDA_WS_ROWS) {
      // wave-uniform: a full chunk steps its rows, issues its reads together, then sums
      unsigned lo[DDA_WS_ROWS];
      float x0[DDA_WS_ROWS], x1[DDA_WS_ROWS];
#pragma unroll
      for (int u = 0; u < DDA_WS_ROWS; ++u) {
        const dda_lds_fptr q = (dda_lds_fptr)(size_t)(unsigned)(__builtin_amdgcn_readfirstlane(base + u * DDA_WS_SEG * 4) +
                                                                 4 * st.hi);
        x0[u] = q[0];
        x1[u] = q[1];
        lo[u] = st.lo;
        dda_trap_step(a, st);
      }
#pragma unroll
      for (int u = 0; u < DDA_WS_ROWS; ++u) blk = dda_trap_term(a, x0[u], x1[u], lo[u], blk);
    } else {
      for (int u = 0; u < nrow; ++u) {
        const dda_lds_fptr q = (dda_lds_fptr)(size_t)(unsigned)(base + u * DDA_WS_SEG * 4 + 4 * st.hi);
        blk = dda_trap_term(a, q[0], q[1], st.lo, blk);
        dda_trap_step(a, st);
      }
    }
    tot += (double)blk;
    sb = sb_next;
  }
  return lane_ok ? tot * a.tr_lmax : 0.0;
}

__global__ __launch_bounds__(256) void k_dda_radon(SSDdaGeom g, const SSDdaAngle* __restrict__ angles,
                                                   const float* __restrict__ img, const float* __restrict__ imgT,
                                                   float* __restrict__ sino) {
  const int r = blockIdx.x * blockDim.x + threadIdx.x;
  const int ai = blockIdx.y;
  const size_t slice = blockIdx.z;
  const bool lane_ok = r < g.nrays;
  const SSDdaAngle a = angles[ai];
  const int nf = a.fast_i ? g.lines : g.cols;
  const int ns = a.fast_i ? g.cols : g.lines;
  // padded layouts: DDA_PADW zero columns either side of each line (dda_pad_pitch)
  const int pitch = dda_pad_pitch(ns);
  const float* __restrict__ src = (a.fast_i ? img : imgT) + slice * (size_t)nf * pitch;
  if (a.fixed && (long long)nf * pitch < (1LL << 29)) {
    __shared__ float wlds[4][2 * DDA_WS_ROWS * DDA_WS_SEG];  // two chunk buffers per wave
    // every lane's own ray (past R too): the staged form takes the wave's lowest ray from
    // its lanes
    const double t = dda_ray_t(g, r);
    const double acc = a.tr_wstage ? dda_radon_trap_ws(a, src, t, lane_ok, nf, ns, wlds[threadIdx.x >> 6])
                                   : dda_radon_trap(a, src, t, lane_ok, nf, ns);
    if (lane_ok) sino[(slice * g.nrays + r) * g.nangles + ai] = (float)acc;
    return;
  }
  SSDdaRay ray = dda_ray_start(g, a, dda_ray_t(g, lane_ok ? r : 0));
  bool alive = lane_ok && dda_inside(ray.f, ray.s, nf, ns);
  // FP64 sum: the lengths are FP64 already, so a tap costs one convert and one FMA as
  // in FP32, without FP32's N*eps growth over a ray of N equal terms
  double acc = 0.0;
  int F = dda_wave_start(alive, ray.f, a.dfast);
  // the pixel's offset in the (fast, slow) image, stepped with the ray (an image side is
  // at most 16384, so a slice's offsets fit an int); meaningful while the lane is alive
  int pix = alive ? ray.f * pitch + ray.s + DDA_PADW : 0;
  {
    const int fast_step = a.dfast * pitch;
    // lanes start at most nf moves apart and then take at most nf + 1 moves each
    for (int it = 0; it <= 2 * nf + 1; ++it) {
      if (__ballot(alive) == 0) break;
      if (alive && ray.f == F) {
        acc = fma((double)src[pix], ray.len, acc);
        if (ray.slow_next) {
          ray.s = dda_step(ray.s, a.dslow);
          pix += a.dslow;
          ray.len = a.len_full - ray.len;
          ray.slow_next = 0;
          alive = dda_inside(ray.f, ray.s, nf, ns);
          if (alive) acc = fma((double)src[pix], ray.len, acc);
        }
        if (alive) {
          dda_fast_move(a, ray);
          pix += fast_step;
          alive = dda_inside(ray.f, ray.s, nf, ns);
        }
      }
      F += a.dfast;
    }
  }
  if (lane_ok) sino[(slice * g.nrays + r) * g.nangles + ai] = (float)acc;
}

// ---------------------------------------------------------------- Radon in planes

// The trapezoid form in planes.  k_dda_radon reads one 8-byte LDS pair and issues 13 VALU
// instructions per fast index and ray.  Here a lane's tau and weights serve four rays
// (SSPlane; the image, its half turn (ray R - 1 - r), its mirror x -> -x (angle A - 1 - a) and
// the half turn of that, or slices), the layouts hold the planes' values of a pixel together
// (16 bytes), and a block's 8 waves share one staged window (ss_planes_chunks).  Layout rows:
// fast index k's pixels along the slow axis with DDA_RP_PAD zeros either side; the record of
// slow index j is j + DDA_RP_PAD, and to the window code the rows are rows of an image of
// ns + 2 DDA_RP_PAD - 2 cells.  A lane takes the fast indices where floor(tau) can be a
// candidate inside the image, with an index of margin either side: tau moves by at most 2 per
// index, so those samples lie within the padding, and their terms are zeros.  Sums are taken
// in FP32 over at most 8 fast indices and those in FP64, as in k_dda_radon.
// Per four updates: 6 VALU for tau, the address and the fraction, 5 for the weights, 8 FMAs,
// two 16-byte reads.
// 2048^2 x 1500: 2470 -> 805 us, the layouts' 34 us included; 1024^2 x 721 491 -> 160; 16 x 512^2 x 360
// 660 -> 340; 256^2 x 180 80 -> 51.

// Layouts: L[group][line][pc] and LT[group][column][pl] of img[slice][lines][cols], pc (pl) =
// cols (lines) + 2 DDA_RP_PAD.  A block moves one 32 x 32 pixel tile; the first and last tile
// of a row also write its padding.
__global__ __launch_bounds__(256) void k_dda_pad_planes(int lines, int cols, int kind, int nslices,
                                                        const float* __restrict__ img, ss_f32x4* __restrict__ L,
                                                        ss_f32x4* __restrict__ LT) {
  __shared__ float T[SS_PLANES][32][33];
  const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;
  const int i0 = blockIdx.y * 32, j0 = blockIdx.x * 32;
  const int pc = cols + 2 * DDA_RP_PAD, pl = lines + 2 * DDA_RP_PAD;
#pragma unroll
  for (int z = 0; z < SS_PLANES; ++z) {
    const SSPlane p = ss_plane(kind, z);
    const size_t slice = (size_t)min((int)blockIdx.z * ss_planes_slices(kind) + p.slice, nslices - 1);
    const float* __restrict__ src = img + slice * lines * cols;
#pragma unroll
    for (int yy = ty; yy < 32; yy += 8) {
      const int i = i0 + yy, j = j0 + tx;
      const int si = p.turn ? lines - 1 - i : i, sj = p.turn != p.mirror ? cols - 1 - j : j;
      T[z][yy][tx] = i < lines && j < cols ? src[(size_t)si * cols + sj] : 0.f;
    }
  }
  __syncthreads();
  ss_f32x4* __restrict__ o = L + (size_t)blockIdx.z * lines * pc;
  ss_f32x4* __restrict__ oT = LT + (size_t)blockIdx.z * cols * pl;
  const ss_f32x4 zero = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int yy = ty; yy < 32; yy += 8) {
    const int i = i0 + yy, j = j0 + tx;
    if (i < lines) {
      ss_f32x4* __restrict__ row = o + (size_t)i * pc;
      if (j < cols) row[j + DDA_RP_PAD] = ss_f32x4{T[0][yy][tx], T[1][yy][tx], T[2][yy][tx], T[3][yy][tx]};
      if (blockIdx.x == 0 && tx < DDA_RP_PAD) row[tx] = zero;
      if (j0 + 32 >= cols && tx < DDA_RP_PAD) row[cols + DDA_RP_PAD + tx] = zero;
    }
    const int jt = j0 + yy, it = i0 + tx;
    if (jt < cols) {
      ss_f32x4* __restrict__ row = oT + (size_t)jt * pl;
      if (it < lines) row[it + DDA_RP_PAD] = ss_f32x4{T[0][tx][yy], T[1][tx][yy], T[2][tx][yy], T[3][tx][yy]};
      if (blockIdx.y == 0 && tx < DDA_RP_PAD) row[tx] = zero;
      if (i0 + 32 >= lines && tx < DDA_RP_PAD) row[lines + DDA_RP_PAD + tx] = zero;
    }
  }
}

// trapezoid terms of a wave's angle
struct SSDdaTerms {
  float c1, kz, pz, pz1;
};

// G fast indices s, s + 1, ... from the staged window; CHECK: an index at or beyond `end` or
// outside the lane's range [lo, lo + span] reads the zero records
template <int G, bool CHECK>
__device__ __forceinline__ void dda_rp_group(const ss_f32x4* __restrict__ st, int s, int end, int64_t& u, int64_t step,
                                             int lo, unsigned span, const SSDdaTerms& w, double (&tot)[SS_PLANES]) {
  float part[SS_PLANES];
  const unsigned stb = (unsigned)(size_t)(ss_lds_cell)st;
#pragma unroll
  for (int h = 0; h < G; h += 4) {  // four indices' reads in flight
    ss_f32x4 a[4], b[4];
    float fr[4];
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      int idx = (int)(u >> 32);
      if (CHECK) idx = s + h + g < end && (unsigned)(s + h + g - lo) <= span ? idx : PLANES_CAP;
      fr[g] = (float)(uint32_t)u;
      u += step;
      __asm__ volatile("" : "+v"(u));  // one 64-bit add per index
      const ss_lds_cell c = (ss_lds_cell)(size_t)(stb + ((unsigned)idx << 4));
      a[g] = c[0];
      b[g] = c[1];
    }
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const float z0 = __builtin_amdgcn_fmed3f(fmaf(-fabsf(w.c1 - fr[g]), w.kz, w.pz), 0.f, 1.f);
      const float z1 = __builtin_amdgcn_fmed3f(fmaf(fr[g], w.kz, w.pz1), 0.f, 1.f);
#pragma unroll
      for (int z = 0; z < SS_PLANES; ++z) {
        part[z] = h + g == 0 ? z0 * a[g][z] : fmaf(z0, a[g][z], part[z]);
        part[z] = fmaf(z1, b[g][z], part[z]);
      }
    }
  }
#pragma unroll
  for (int z = 0; z < SS_PLANES; ++z) tot[z] += (double)part[z];
}

struct SSDdaRadonPlanes {
  int kind, nslices;
  int nangles, nrays;      // plane 0's angles and rays
  SSPlanesOrder order;
  int nslab, slab_rows;    // fast indices in slabs of slab_rows, each with its partial sums
  const SSDdaStraight* straight;
  int nstraight;           // straight angles: blocks of 64 rays, first in the launch
  const int* walk;
  int nwalk;               // traced angles: blocks of 512 rays, before those
};

// the layout of a slice's own plane in its group: rows of `pitch` records, a float every
// SS_PLANES
__device__ __forceinline__ const float* dda_rp_plane(const SSDdaRadonPlanes& rp, const ss_f32x4* __restrict__ lay,
                                                     int slice, int nf, int pitch) {
  const int per = ss_planes_slices(rp.kind);
  const int z = rp.kind == SS_PLANES_PAIR ? 2 * (slice % 2) : slice % per;
  return reinterpret_cast<const float*>(lay + (size_t)(slice / per) * nf * pitch) + z;
}

// a traced angle's rays, as k_dda_radon walks them, DDA_RP_MOVES moves at a time: their pixels
// and lengths first, then the loads together (a move that adds nothing reads the layout's
// first record, a zero), then the sums in order
#define DDA_RP_MOVES 8
__device__ __forceinline__ void dda_rp_walk(const SSDdaGeom& g, const SSDdaAngle* __restrict__ angles,
                                            const SSDdaRadonPlanes& rp, const ss_f32x4* __restrict__ L,
                                            const ss_f32x4* __restrict__ LT, int id, float* __restrict__ sino) {
  const int nrb = (g.nrays + RADON_WAVES * SS_WAVE - 1) / (RADON_WAVES * SS_WAVE);
  const int slice = id / (nrb * rp.nwalk);
  id -= slice * (nrb * rp.nwalk);
  const int ai = rp.walk[id / nrb], r = id % nrb * (RADON_WAVES * SS_WAVE) + threadIdx.x;
  const SSDdaAngle& a = angles[ai];
  const int nf = a.fast_i ? g.lines : g.cols, ns = a.fast_i ? g.cols : g.lines;
  const int pitch = ns + 2 * DDA_RP_PAD;
  const float* __restrict__ src = dda_rp_plane(rp, a.fast_i ? L : LT, slice, nf, pitch);
  SSDdaRay ray = dda_ray_start(g, a, dda_ray_t(g, min(r, g.nrays - 1)));
  bool alive = r < g.nrays && dda_inside(ray.f, ray.s, nf, ns);
  int F = dda_wave_start(alive, ray.f, a.dfast);
  double acc = 0.0;
  // lanes start at most nf moves apart and then take at most nf + 1 moves each
  for (int it = 0; it <= 2 * nf + 1; it += DDA_RP_MOVES) {
    if (__ballot(alive) == 0) break;
    // no lane's drift passes the pixel width in these moves (close to an axis, most): the same
    // moves without their cases
    double e = ray.e;
#pragma unroll
    for (int m = 0; m < DDA_RP_MOVES; ++m) e += a.e_step;
    const int f_end = dda_step(ray.f, DDA_RP_MOVES * a.dfast);
    const bool plain = ray.f == F && !ray.slow_next && (unsigned)f_end < (unsigned)nf && e <= a.e_cap;
    if (__ballot(alive && !plain) == 0) {
      const float* at = src + (alive ? (size_t)(ray.f * pitch + ray.s + DDA_RP_PAD) : 0) * SS_PLANES;
      const ptrdiff_t step = alive ? (ptrdiff_t)a.dfast * pitch * SS_PLANES : 0;
      float v[DDA_RP_MOVES];
#pragma unroll
      for (int m = 0; m < DDA_RP_MOVES; ++m) v[m] = at[m * step];
#pragma unroll
      for (int m = 0; m < DDA_RP_MOVES; ++m) acc = fma((double)v[m], m == 0 ? ray.len : a.len_full, acc);
      if (alive) {
        ray.f = f_end;
        ray.e = e;
        ray.len = a.len_full;
      }
      F += DDA_RP_MOVES * a.dfast;
      continue;
    }
    int pix[2 * DDA_RP_MOVES];
    double len[2 * DDA_RP_MOVES];
#pragma unroll
    for (int m = 0; m < DDA_RP_MOVES; ++m) {
      pix[2 * m] = pix[2 * m + 1] = 0;
      len[2 * m] = len[2 * m + 1] = 0.0;
      if (alive && ray.f == F) {
        pix[2 * m] = ray.f * pitch + ray.s + DDA_RP_PAD;
        len[2 * m] = ray.len;
        if (ray.slow_next) {
          ray.s = dda_step(ray.s, a.dslow);
          ray.len = a.len_full - ray.len;
          ray.slow_next = 0;
          alive = dda_inside(ray.f, ray.s, nf, ns);
          if (alive) {
            pix[2 * m + 1] = ray.f * pitch + ray.s + DDA_RP_PAD;
            len[2 * m + 1] = ray.len;
          }
        }
        if (alive) {
          dda_fast_move(a, ray);
          alive = dda_inside(ray.f, ray.s, nf, ns);
        }
      }
      F += a.dfast;
    }
    float v[2 * DDA_RP_MOVES];
#pragma unroll
    for (int m = 0; m < 2 * DDA_RP_MOVES; ++m) v[m] = src[(size_t)pix[m] * SS_PLANES];
#pragma unroll
    for (int m = 0; m < 2 * DDA_RP_MOVES; ++m) acc = fma((double)v[m], len[m], acc);
  }
  if (r < g.nrays) sino[((size_t)slice * g.nrays + r) * g.nangles + ai] = (float)acc;
}

// a straight angle's rays: the block's waves sum an eighth of the fast indices each
__device__ __forceinline__ void dda_rp_straight(const SSDdaGeom& g, const SSDdaAngle* __restrict__ angles,
                                                const SSDdaRadonPlanes& rp, const ss_f32x4* __restrict__ L,
                                                const ss_f32x4* __restrict__ LT, int id, double* red,
                                                float* __restrict__ sino) {
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int nrb = (g.nrays + 63) / 64;
  const int slice = id / (nrb * rp.nstraight);
  id -= slice * (nrb * rp.nstraight);
  const int ai = rp.straight[id / nrb].a, r = id % nrb * 64 + lane;
  const SSDdaAngle& a = angles[ai];
  const int nf = a.fast_i ? g.lines : g.cols, ns = a.fast_i ? g.cols : g.lines;
  const int pitch = ns + 2 * DDA_RP_PAD;
  const float* __restrict__ src = dda_rp_plane(rp, a.fast_i ? L : LT, slice, nf, pitch);
  const SSDdaRay ray = dda_ray_start(g, a, dda_ray_t(g, min(r, g.nrays - 1)));
  const bool in = dda_inside(ray.f, ray.s, nf, ns);
  const int s = in ? ray.s : 0;
  double sum = 0.0;
  const int f0 = (int)((long long)nf * wv / RADON_WAVES), f1 = (int)((long long)nf * (wv + 1) / RADON_WAVES);
#pragma unroll 8
  for (int f = f0; f < f1; ++f) sum += (double)src[((size_t)f * pitch + s + DDA_RP_PAD) * SS_PLANES];
  red[threadIdx.x] = sum;
  __syncthreads();
  if (wv != 0 || r >= g.nrays) return;
  for (int w = 1; w < RADON_WAVES; ++w) sum += red[w * 64 + lane];
  sino[((size_t)slice * g.nrays + r) * g.nangles + ai] = in ? (float)(sum * a.len_full) : 0.f;
}

// Blocks: the traced angles' and the straight angles' (all slices), then the planes' (order.blocks per
// slab and group of planes).  PARTIAL: the slab's FP64 sums go to part[slice][slab][a][r].
template <bool PARTIAL>
__global__ __launch_bounds__(RADON_WAVES * SS_WAVE, PLANES_BLOCKS) void k_dda_radon_planes(
    SSDdaGeom g, const SSDdaAngle* __restrict__ angles, SSDdaRadonPlanes rp, const ss_f32x4* __restrict__ L,
    const ss_f32x4* __restrict__ LT, float* __restrict__ sino, double* __restrict__ part) {
  __shared__ SSPlanesLds lds;
  int id = blockIdx.x;
  const int nwk = rp.nwalk * ((g.nrays + RADON_WAVES * SS_WAVE - 1) / (RADON_WAVES * SS_WAVE)) * rp.nslices;
  if (id < nwk) {
    dda_rp_walk(g, angles, rp, L, LT, id, sino);
    return;
  }
  id -= nwk;
  const int nst = rp.nstraight * ((g.nrays + 63) / 64) * rp.nslices;
  if (id < nst) {
    dda_rp_straight(g, angles, rp, L, LT, id, reinterpret_cast<double*>(lds.stage), sino);
    return;
  }
  id -= nst;
  const int2 at = ss_planes_place(rp.order, id % rp.order.blocks);
  id /= rp.order.blocks;
  const int slab = id % rp.nslab, group = id / rp.nslab;
  if (at.y < 0) return;  // block-uniform
  const int lane = threadIdx.x & 63;
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int j = at.y * RADON_WAVES + wv, k = at.x * SS_WAVE + ss_plane_ray(lane);
  const SSDdaAngle& a = angles[min(j, rp.nangles - 1)];
  const bool active = j < rp.nangles && a.fixed;
  const bool on = active && k < rp.nrays;
  const int nf_a = a.fast_i ? g.lines : g.cols, ns_a = a.fast_i ? g.cols : g.lines;
  const SSDdaTerms w{a.tr_c1, a.tr_kz, a.tr_pz, a.tr_pz1};
  const int64_t beta = (int64_t)a.tr_dhi * ((int64_t)1 << 32) + a.tr_dlo;
  // trajectory in Q32 records, less 1 (the window code's cells): a_k + s beta
  int64_t a_k = 0;
  int lo = 0x40000000, hi = -1;
  if (on) {
    const double x = fma(dda_ray_t(g, k), a.tr_inv, a.tr_off) - DDA_PADW;  // floor: the first candidate
    const double v = fmin(fmax(x + (DDA_RP_PAD - 1), -1073741824.0), 1073741824.0), fv = floor(v);
    a_k = (int64_t)fv * ((int64_t)1 << 32) + (int64_t)(uint32_t)((v - fv) * 4294967296.0);
    const double ka = (-1.0 - x) / a.tr_d, kb = (ns_a - x) / a.tr_d;
    const double kl = fmax(fmin(ka, kb), -1.0), kh = fmin(fmax(ka, kb), (double)nf_a);
    if (kl <= kh) {  // false for NaN
      lo = (int)fmax(0.0, floor(kl) - 1.0);
      hi = (int)fmin(nf_a - 1.0, ceil(kh) + 1.0);
    }
  }
  const bool any = lo <= hi;
  const unsigned span = any ? (unsigned)(hi - lo) : 0u;
  if (!any) lo = 0x40000000;
  int ulo = any ? lo : 0x7fffffff, uhi = any ? hi : -1, clo = any ? lo : -0x7fffffff, chi = any ? hi : 0x7fffffff;
  int64_t amin = any ? a_k : INT64_MAX, amax = any ? a_k : INT64_MIN;
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
  const int branch = uhi < ulo ? -1 : (a.fast_i ? 0 : 1);
  if (lane == 0) {
    lds.wmeta[wv][0] = branch;
    lds.wmeta[wv][1] = ulo;
    lds.wmeta[wv][2] = uhi;
    lds.wpar[wv][0] = amin;
    lds.wpar[wv][1] = amax;
    lds.wpar[wv][2] = beta;
  }
  if (threadIdx.x < 2) lds.stage[PLANES_CAP + threadIdx.x] = ss_f32x4{0.f, 0.f, 0.f, 0.f};
  double tot[SS_PLANES] = {0.0, 0.0, 0.0, 0.0};
  for (int pass = 0; pass < 2; ++pass) {  // fast axis line, then column
    __syncthreads();
    if (lane == 0) lds.wmeta[wv][0] = branch == pass ? branch : -1;  // this pass's waves
    __syncthreads();
    int s_lo = 0x7fffffff, s_hi = -1;
    for (int i = 0; i < RADON_WAVES; ++i)
      if (lds.wmeta[i][0] >= 0) {
        s_lo = min(s_lo, lds.wmeta[i][1]);
        s_hi = max(s_hi, lds.wmeta[i][2]);
      }
    s_lo = max(ss_rfl(s_lo), slab * rp.slab_rows);
    s_hi = min(ss_rfl(s_hi), (slab + 1) * rp.slab_rows - 1);
    const bool mine = branch == pass;
    const int nf = pass ? g.cols : g.lines, pitch = (pass ? g.lines : g.cols) + 2 * DDA_RP_PAD;
    const ss_f32x4* lay = (pass ? LT : L) + (size_t)group * nf * pitch;
    ss_planes_chunks(lds, lay, pitch, pitch - 2, s_lo, s_hi, wv, lane, [&](int s0, int s1, int rec0, int Wc, bool fits) {
      const int ra = max(s0, ulo), rb = min(s1 - 1, uhi);
      if (!mine || ra > rb || Wc <= 0) return;
      const int64_t t = a_k + (int64_t)ra * beta;
      if (fits) {
        // high word: staged record index (cell + 1 - rec0) + (row - s0) * Wc
        int64_t u = t + ((int64_t)(1 - rec0 + (ra - s0) * Wc) << 32);
        int64_t step = beta + ((int64_t)Wc << 32);
        if (!any) {
          u = (int64_t)PLANES_CAP << 32;
          step = 0;
        }
        int s = ra;
        const int head = min(rb + 1, clo);
        if (s < head) {
          const int64_t u0 = u;
          for (; s < head; s += 4) dda_rp_group<4, true>(lds.stage, s, head, u, step, lo, span, w, tot);
          s = head;
          u = u0 + (int64_t)(head - ra) * step;
        }
        const int mid = min(rb + 1, chi + 1);
        for (; s + 8 <= mid; s += 8) dda_rp_group<8, false>(lds.stage, s, 0, u, step, lo, span, w, tot);
        for (; s <= rb; s += 4) dda_rp_group<4, true>(lds.stage, s, rb + 1, u, step, lo, span, w, tot);
      } else if (any) {  // the window does not fit the LDS: read the layout
        int64_t u = t + ((int64_t)1 << 32);
        for (int s = ra; s <= rb; ++s, u += beta) {
          if ((unsigned)(s - lo) > span) continue;
          const ss_f32x4* cell = lay + (size_t)s * pitch + (int)(u >> 32);
          const ss_f32x4 q0 = cell[0], q1 = cell[1];
          const float fr = (float)(uint32_t)u;
          const float z0 = __builtin_amdgcn_fmed3f(fmaf(-fabsf(w.c1 - fr), w.kz, w.pz), 0.f, 1.f);
          const float z1 = __builtin_amdgcn_fmed3f(fmaf(fr, w.kz, w.pz1), 0.f, 1.f);
#pragma unroll
          for (int z = 0; z < SS_PLANES; ++z) tot[z] += (double)fmaf(z1, q1[z], z0 * q0[z]);
        }
      }
    });
  }
  if (!on) return;
  const int R = g.nrays, A = g.nangles, slice0 = group * ss_planes_slices(rp.kind);
#pragma unroll
  for (int z = 0; z < SS_PLANES; ++z) {
    const SSPlane pl = ss_plane(rp.kind, z);
    const int kz = pl.turn ? R - 1 - k : k, jz = pl.mirror ? A - 1 - j : j;
    if (slice0 + pl.slice >= rp.nslices) continue;                     // a group past the last slice
    if ((pl.turn && kz == k) || (pl.mirror && jz == j)) continue;     // its own half turn or mirror
    const size_t slice = slice0 + pl.slice;
    if (PARTIAL)
      part[((slice * rp.nslab + slab) * A + jz) * R + kz] = tot[z];
    else
      sino[(slice * R + kz) * A + jz] = (float)(tot[z] * a.tr_lmax);
  }
}

// sino[slice][r][a] = lmax times the sum, in order, of the slabs' partial sums (exact-geometry
// angles).  A block moves 32 angles x 32 rays.
__global__ __launch_bounds__(256) void k_dda_radon_finish(SSDdaGeom g, const SSDdaAngle* __restrict__ angles, int nslab,
                                                          const double* __restrict__ part, float* __restrict__ sino) {
  __shared__ float T[32][33];
  const int R = g.nrays, A = g.nangles;
  const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;
  const int r0 = blockIdx.x * 32, a0 = blockIdx.y * 32;
  const size_t slice = blockIdx.z;
  for (int yy = ty; yy < 32; yy += 8) {
    const int a = a0 + yy, r = r0 + tx;
    double sum = 0.0;
    if (a < A && r < R && angles[a].fixed) {
      const double* __restrict__ src = part + (slice * nslab * A + a) * R + r;
#pragma unroll 4
      for (int s = 0; s < nslab; ++s) sum += src[(size_t)s * A * R];
      sum *= angles[a].tr_lmax;
    }
    T[yy][tx] = (float)sum;
  }
  __syncthreads();
  for (int yy = ty; yy < 32; yy += 8) {
    const int r = r0 + yy, a = a0 + tx;
    if (a < A && r < R && angles[a].fixed) sino[(slice * R + r) * A + a] = T[tx][yy];
  }
}

// ---------------------------------------------------------------- transpose (scatter)

// acc: pixels of angles whose fast axis is the line ([lines][cols]); accT: the others
// ([cols][lines]).  ones: every ray carries 1 (the normalisation R^T 1).  T = float for
// the transpose, double for the backprojection, whose normalisation can cancel (the
// reference's non-square-pixel traversal yields negative lengths).
template <typename T>
__global__ __launch_bounds__(256) void k_dda_scatter(SSDdaGeom g, const SSDdaAngle* __restrict__ angles,
                                                     const int* __restrict__ walk, const float* __restrict__ sino,
                                                     int ones, T* __restrict__ acc, T* __restrict__ accT) {
  const int r = blockIdx.x * blockDim.x + threadIdx.x;
  const int ai = walk[blockIdx.y];
  const size_t slice = blockIdx.z;
  if (r >= g.nrays) return;
  const T q = ones ? T(1) : T(sino[(slice * g.nrays + r) * g.nangles + ai]);
  if (q == T(0)) return;  // adds nothing
  const SSDdaAngle a = angles[ai];
  const int nf = a.fast_i ? g.lines : g.cols;
  const int ns = a.fast_i ? g.cols : g.lines;
  T* dst = (a.fast_i ? acc : accT) + slice * (size_t)g.lines * g.cols;
  SSDdaRay ray = dda_ray_start(g, a, dda_ray_t(g, r));
  for (int it = 0; it <= nf; ++it) {
    if (!dda_inside(ray.f, ray.s, nf, ns)) break;
    unsafeAtomicAdd(dst + (size_t)ray.f * ns + ray.s, q * T(ray.len));
    if (ray.slow_next) {
      ray.s = dda_step(ray.s, a.dslow);
      ray.len = a.len_full - ray.len;
      ray.slow_next = 0;
      if (!dda_inside(ray.f, ray.s, nf, ns)) break;
      unsafeAtomicAdd(dst + (size_t)ray.f * ns + ray.s, q * T(ray.len));
    }
    dda_fast_move(a, ray);
  }
}

// ---------------------------------------------------------------- transpose (gather)

#define DDA_GX 64     // image columns per block (one per lane)
#define DDA_GROWS 4   // image lines per thread
#define DDA_GY (4 * DDA_GROWS)

// acc[i][j] = sum over the table's angles and the rays crossing pixel (i, j) of
// q(r, a) * L(t_r - t_c) (trapezoid lengths, FP64 geometry and sums).  Overwrites acc.
// rows: the angle-major sinogram, each row scaled by its angle's lmax and padded with
// two zeros either side (row a starts at rows + a * (R + 4) + 2), so the K = 2 path reads
// its candidates r0, r0 + 1 in [-2, R + 1] without bounds tests.  K = 0: any number of
// candidates (A.k), with bounds tests.  ones: q = 1 (the normalisation R^T 1).
template <typename T, int K>
__global__ __launch_bounds__(256) void k_dda_gather(SSDdaGeom g, const SSDdaGatherAngle* __restrict__ ga, int nga,
                                                    const float* __restrict__ rows, int ones, T* __restrict__ acc) {
  const int j = blockIdx.x * DDA_GX + (threadIdx.x & (DDA_GX - 1));
  const int i0 = blockIdx.y * DDA_GY + (threadIdx.x / DDA_GX) * DDA_GROWS;
  const size_t slice = blockIdx.z;
  if (j >= g.cols || i0 >= g.lines) return;
  const double x = g.ox + j * g.hx;
  const double y0 = g.oy + i0 * g.hy;
  const double inv_dt = 1.0 / g.dt;
  const int pitch = g.nrays + 4;
  const float* __restrict__ srows = rows + slice * (size_t)g.nangles * pitch + 2;
  double sum[DDA_GROWS];
#pragma unroll
  for (int rr = 0; rr < DDA_GROWS; ++rr) sum[rr] = 0.0;
  for (int k = 0; k < nga; ++k) {
    const SSDdaGatherAngle A = ga[k];
    const float* __restrict__ q = srows + (size_t)A.a * pitch;
    double tc = fma(x, A.c, y0 * A.s);
    const double p_inv = A.p * A.inv_pq;
#pragma unroll
    for (int rr = 0; rr < DDA_GROWS; ++rr) {
      const double rc = (tc - g.t0) * inv_dt;
      const double lo = fmin(fmax(floor(rc - A.half) + 1.0, -2.0), (double)g.nrays);
      const int r0 = (int)lo;
      if (K == 2) {
        // d = t_r - t_c for r0 and r0 + 1; z = clamp((p - |d|) / (p - q))
        const double d0 = fma(lo, g.dt, g.t0) - tc;
        const double d1 = d0 + g.dt;
        const double z0 = fmin(1.0, fmax(0.0, fma(-fabs(d0), A.inv_pq, p_inv)));
        const double z1 = fmin(1.0, fmax(0.0, fma(-fabs(d1), A.inv_pq, p_inv)));
        if (ones) {  // rays that exist only
          const double w0 = (unsigned)r0 < (unsigned)g.nrays ? z0 : 0.0;
          const double w1 = (unsigned)(r0 + 1) < (unsigned)g.nrays ? z1 : 0.0;
          sum[rr] += A.lmax * (w0 + w1);
        } else {
          sum[rr] = fma((double)q[r0], z0, sum[rr]);
          sum[rr] = fma((double)q[r0 + 1], z1, sum[rr]);
        }
      } else {
        for (int m = 0; m < A.k; ++m) {
          const int r = r0 + m;
          if ((unsigned)r < (unsigned)g.nrays) {
            const double d = fma((double)r, g.dt, g.t0) - tc;
            const double z = fmin(1.0, fmax(0.0, fma(-fabs(d), A.inv_pq, p_inv)));
            sum[rr] = fma(ones ? A.lmax : (double)q[r], z, sum[rr]);
          }
        }
      }
      tc += A.hys;
    }
  }
  T* __restrict__ out = acc + slice * (size_t)g.lines * g.cols;
#pragma unroll
  for (int rr = 0; rr < DDA_GROWS; ++rr)
    if (i0 + rr < g.lines) out[(size_t)(i0 + rr) * g.cols + j] = T(sum[rr]);
}

// The two-candidate gather of a sinogram (k <= 2 for every angle) in FP32 ray units.
// A block covers DDA_G2_COLS columns x 4 G lines of pixels and takes the
// angles in groups of DDA_G2_ANGLES: each wave stages, for a quarter of the group's
// angles, the segment of the angle's (lmax-scaled, zero-padded) row that the block's
// candidate rays span into LDS (rays rb .. rb + ws - 1 with rb = floor(min over the block
// of rc - half) - 2; the resource spans the padded row, so rays off the row read 0),
// or marks the angle as missing the block.  Then per (thread, angle) FP64 gives
// rc - half - rb at the thread's first line and splits it into an integer base and an
// FP32 fraction g0 in [0, 1); each of the thread's G lines takes
// fl = floor(g), fr = fract(g) of g = g0 + rr ky, reads q[r0], q[r0 + 1]
// (r0 = rb + base + fl + 1) from the segment with one two-word LDS read and adds
// q0 z0 + q1 z1 with the angle's hat weights.  The segment index base + fl + 1 lies in
// [1, 6 + span] for span = (cols - 1)|kx| + (lines - 1)|ky| of the block (the FP32
// fraction is within 1e-5 ray units of the FP64 value, so floor is off by at most one),
// and ws >= span + 8.  Terms are summed in FP32 over a group, those sums in FP64.
__device__ float dda_raw_load_f32(__amdgpu_buffer_rsrc_t rsrc, int voffset, int soffset,
                                  int aux) __asm("llvm.amdgcn.raw.ptr.buffer.load.f32");

__device__ __forceinline__ int dda_floor_i32(float v) {
  int r;
  __asm__("v_cvt_flr_i32_f32 %0, %1" : "=v"(r) : "v"(v));
  return r;
}

#define DDA_G2_MISS (-0x7fffffff - 1)
typedef __attribute__((address_space(3))) float dda_lds_float;
typedef __attribute__((address_space(3))) const ss_f32x4* dda_lds_cell;

template <typename T, int G>
__global__ __launch_bounds__(256) void k_dda_gather2(SSDdaGeom g, const SSDdaGatherAngle* __restrict__ ga, int nga,
                                                     const float* __restrict__ rows, int ws, T* __restrict__ acc) {
  constexpr int NA = DDA_G2_ANGLES;
  __shared__ float seg[NA * DDA_G2_WSMAX];
  __shared__ int seg_rb[NA];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int jb = blockIdx.x * DDA_G2_COLS, ib = blockIdx.y * (4 * G);
  const int j = jb + lane;
  const int i0 = ib + wave * G;
  const size_t slice = blockIdx.z;
  const double jd = j, id = i0;
  const int pitch = g.nrays + 4;
  const float* __restrict__ srows = rows + slice * (size_t)g.nangles * pitch;
  double tot[G];
#pragma unroll
  for (int rr = 0; rr < G; ++rr) tot[rr] = 0.0;
  for (int k0 = 0; k0 < nga; k0 += NA) {
    const int na = min(NA, nga - k0);
    __syncthreads();  // the previous group's segments are read
    for (int t = wave; t < na; t += 4) {
      const SSDdaGatherAngle& A = ga[k0 + t];
      const double lo = fma((double)jb, A.kx, fma((double)ib, A.ky, A.k0h)) + fmin(0.0, (DDA_G2_COLS - 1) * A.kx) +
                        fmin(0.0, (4 * G - 1) * A.ky);
      const double hi = lo + (DDA_G2_COLS - 1) * fabs(A.kx) + (4 * G - 1) * fabs(A.ky);
      // candidates floor(lo) + 1 .. floor(hi) + 2 meet the rays 0 .. R - 1
      const bool meets = hi >= -4.0 && lo <= g.nrays + 4.0;
      const int rb = meets ? (int)floor(lo) - 2 : DDA_G2_MISS;
      if (lane == 0) seg_rb[t] = rb;
      if (meets) {
        const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(
            (void*)(srows + (size_t)A.a * pitch), (short)0, pitch * (int)sizeof(float), DDA_RSRC_DWORD3);
        // byte offset of padded element rb + 2 (ray rb), opaque so that no constant part
        // moves into the load's instruction offset: the range check sees the whole
        // offset, and one below 0 reads as out of range
        int off = (rb + 2) * (int)sizeof(float);
        __asm__ volatile("" : "+v"(off));
        for (int m = lane; m < ws; m += 64)
          seg[t * DDA_G2_WSMAX + m] = dda_raw_load_f32(rs, off + m * (int)sizeof(float), 0, 0);
      }
    }
    __syncthreads();
    float sum[G];
#pragma unroll
    for (int rr = 0; rr < G; ++rr) sum[rr] = 0.f;
    for (int t = 0; t < na; ++t) {
      const int rb = __builtin_amdgcn_readfirstlane(seg_rb[t]);
      if (rb == DDA_G2_MISS) continue;
      const SSDdaGatherAngle& A = ga[k0 + t];
      const double v = fma(jd, A.kx, fma(id, A.ky, A.k0h)) - (double)rb;
      const double b = floor(v);
      const float g0 = (float)(v - b);
      // the angle's segment from the pixel's base, opaque so that each line's address is
      // one shift-add of its floor
      dda_lds_float* sg = (dda_lds_float*)(seg + t * DDA_G2_WSMAX + ((int)b + 1));
      __asm__ volatile("" : "+v"(sg));
      float fr[G];
      dda_f2v q[G];
#pragma unroll
      for (int rr = 0; rr < G; ++rr) {
        const float gr = rr == 0 ? g0 : fmaf((float)rr, A.kyf, g0);
        const int fl = dda_floor_i32(gr);
        fr[rr] = __builtin_amdgcn_fractf(gr);
        q[rr][0] = sg[fl];
        q[rr][1] = sg[fl + 1];
      }
#pragma unroll
      for (int rr = 0; rr < G; ++rr) {
        const float z0 = __builtin_amdgcn_fmed3f(fmaf(-fabsf(A.c1 - fr[rr]), A.kz, A.pz), 0.f, 1.f);
        const float z1 = __builtin_amdgcn_fmed3f(fmaf(fr[rr], A.kz, A.pz1), 0.f, 1.f);
        sum[rr] = fmaf(q[rr][0], z0, sum[rr]);
        sum[rr] = fmaf(q[rr][1], z1, sum[rr]);
      }
    }
#pragma unroll
    for (int rr = 0; rr < G; ++rr) tot[rr] += (double)sum[rr];
  }
  if (j >= g.cols) return;
  T* __restrict__ out = acc + slice * (size_t)g.lines * g.cols;
#pragma unroll
  for (int rr = 0; rr < G; ++rr)
    if (i0 + rr < g.lines) out[(size_t)(i0 + rr) * g.cols + j] = T(tot[rr]);
}

// The two-candidate gather in planes.  k_dda_gather2 is bound by its LDS reads (one two-word
// read per update) and by the floor, fraction and weights of every update, and launches of few
// tiles walk all angles serially.  Here a pixel's ray coordinate rc - half, its candidates
// and weights serve four values (SSPlane):
//   SS_PLANES_QUAD    the pixel, its half turn (ray R - 1 - r), its mirror x -> -x (angle
//                     A - 1 - a) and the half turn of that, tiles over a quarter of the image;
//   SS_PLANES_PAIR    two slices and their half turns, tiles over half the image;
//   SS_PLANES_SLICES  four slices.
// sp[a][r] holds the planes' lmax-scaled values of a ray together (k_dda_rows_planes), copied
// into LDS windows of ws rays by 16-byte buffer-to-LDS loads (rays off the detector read 0
// through the range check); a lane reads a candidate's four values with one 16-byte read
// (column order: ss_bp_column).  Geometry as in k_dda_gather2: per (thread, angle) FP64 gives
// rc - half from the window's base and splits it; the thread's DDA_GP_ROWS consecutive lines
// step from that fraction by ky in FP32.  Sums are taken in FP32 over DDA_GP_ANGLES angles,
// those in FP64; with angle groups the groups' FP64 partial images are added by k_dda_fold.
// Window: a tile's rc - half lies in [lo, hi] and its candidates in floor(lo) + 1 .. floor(hi) + 2;
// the window holds floor(lo) .. floor(lo) + ws - 1, a ray of margin either side for rounding.
//
// Work per four updates: 7 VALU for the candidates and weights, 8 FMAs, two reads.
// 1024^2 x 721, backprojection: 575 -> 141 us (this kernel 555 -> 112: VALU issue and LDS reads about
// equal); 2048^2 x 1500 1670 -> 810; 16 x 512^2 x 360 430 -> 250; 256^2 x 180 136 -> 52.
__global__ __launch_bounds__(256, 4) void k_dda_gather_planes(SSDdaGeom g, const SSDdaGatherAngle* __restrict__ ga,
                                                              int nga, const ss_f32x4* __restrict__ planes, int kind,
                                                              int nslices, int ws, int ngroups, int tcols, int trows,
                                                              double* __restrict__ part) {
  constexpr int ROWS = DDA_GP_ROWS, NA = DDA_GP_ANGLES, TH = 8 * ROWS;
  __shared__ ss_f32x4 seg[NA * DDA_GP_WSMAX];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int z0 = blockIdx.x / (tcols * trows), tile = blockIdx.x - z0 * (tcols * trows);
  const int group = z0 / ngroups, gi = z0 - group * ngroups;
  const int r0 = tile / tcols * TH, c0 = tile % tcols * 32;
  const int tx = ss_bp_column(tid), ty = (tid >> 5) * ROWS;
  const int k0 = (int)((long long)gi * nga / ngroups), k1 = (int)((long long)(gi + 1) * nga / ngroups);
  const ss_f32x4* __restrict__ sp = planes + (size_t)group * g.nangles * g.nrays;
  const double txd = tx, tyd = ty;
  double tot[ROWS][SS_PLANES];
#pragma unroll
  for (int i = 0; i < ROWS; ++i)
#pragma unroll
    for (int z = 0; z < SS_PLANES; ++z) tot[i][z] = 0.0;
  for (int ka = k0; ka < k1; ka += 64) {
    const int np = min(64, k1 - ka);
    // angle ka + lane: rc - half at the tile's origin from the window's first ray, less 1
    double o = 0.0;
    int first = 0, row = 0;
    bool meets = false;
    if (lane < np) {
      const SSDdaGatherAngle& A = ga[ka + lane];
      const double v = fma((double)c0, A.kx, fma((double)r0, A.ky, A.k0h));
      const double lo = v + fmin(0.0, 31 * A.kx) + fmin(0.0, (TH - 1) * A.ky);
      const double hi = v + fmax(0.0, 31 * A.kx) + fmax(0.0, (TH - 1) * A.ky);
      meets = hi >= -4.0 && lo <= g.nrays + 4.0;  // candidates floor(rc - half) + 1 and + 2
      first = meets ? (int)floor(lo) : 0;
      o = v - (first - 1);
      row = A.a;
    }
    const unsigned long long near = __ballot(meets);
    for (int ks = 0; ks < np; ks += NA) {
      const int na = min(NA, np - ks);
      __syncthreads();  // the previous windows are read
      for (int t = wv; t < na; t += 4) {
        if (!(near >> (ks + t) & 1)) continue;
        const int a = __builtin_amdgcn_readlane(row, ks + t), base = __builtin_amdgcn_readlane(first, ks + t);
        const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(
            (void*)(sp + (size_t)a * g.nrays), (short)0, g.nrays * (int)sizeof(ss_f32x4), DDA_RSRC_DWORD3);
        for (int m = 0; m < ws; m += 64) {
          // the whole offset in the register: the range check sees a ray below 0 as out of range
          int off = (base + m + lane) * (int)sizeof(ss_f32x4);
          __asm__ volatile("" : "+v"(off));
          if (m + lane < ws)  // active lanes write their record: stay in this window
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (dda_lds_ptr)(seg + t * DDA_GP_WSMAX + m), 16, off, 0, 0, 0);
        }
      }
      __syncthreads();
      float sum[ROWS][SS_PLANES];
#pragma unroll
      for (int i = 0; i < ROWS; ++i)
#pragma unroll
        for (int z = 0; z < SS_PLANES; ++z) sum[i][z] = 0.f;
      for (int t = 0; t < na; ++t) {
        if (!(near >> (ks + t) & 1)) continue;
        const SSDdaGatherAngle& A = ga[ka + ks + t];
        const long long ob = __builtin_bit_cast(long long, o);
        const double ot = __builtin_bit_cast(
            double, ((long long)__builtin_amdgcn_readlane((int)(ob >> 32), ks + t) << 32) |
                        (unsigned)__builtin_amdgcn_readlane((int)ob, ks + t));
        const double v = fma(txd, A.kx, fma(tyd, A.ky, ot));
        const double b = floor(v);
        const float g0 = (float)(v - b);
        // candidate floor(rc - half) + 1 is record floor(v) of the window
        const dda_lds_cell q = (dda_lds_cell)(seg + t * DDA_GP_WSMAX + (int)b);
#pragma unroll
        for (int i = 0; i < ROWS; ++i) {
          const float gr = i == 0 ? g0 : fmaf((float)i, A.kyf, g0);
          const int fl = i == 0 ? 0 : dda_floor_i32(gr);
          const float fr = i == 0 ? g0 : __builtin_amdgcn_fractf(gr);
          const ss_f32x4 q0 = q[fl], q1 = q[fl + 1];
          const float w0 = __builtin_amdgcn_fmed3f(fmaf(-fabsf(A.c1 - fr), A.kz, A.pz), 0.f, 1.f);
          const float w1 = __builtin_amdgcn_fmed3f(fmaf(fr, A.kz, A.pz1), 0.f, 1.f);
#pragma unroll
          for (int z = 0; z < SS_PLANES; ++z) sum[i][z] = fmaf(w1, q1[z], fmaf(w0, q0[z], sum[i][z]));
        }
      }
#pragma unroll
      for (int i = 0; i < ROWS; ++i)
#pragma unroll
        for (int z = 0; z < SS_PLANES; ++z) tot[i][z] += (double)sum[i][z];
    }
  }
  const size_t npix = (size_t)g.lines * g.cols;
  const int slice0 = group * ss_planes_slices(kind);
#pragma unroll
  for (int i = 0; i < ROWS; ++i) {
    const int row = r0 + ty + i, col = c0 + tx;
#pragma unroll
    for (int z = 0; z < SS_PLANES; ++z) {
      const SSPlane pl = ss_plane(kind, z);
      const int mr = pl.turn ? 1 : 0, mc = pl.turn != pl.mirror ? 1 : 0;
      if (slice0 + pl.slice >= nslices || row >= g.lines || col >= g.cols) continue;
      // tiles reach the image's middle; a pixel that is its own image is stored once
      if (kind != SS_PLANES_SLICES && 2 * row + mr > g.lines - 1) continue;
      if (kind == SS_PLANES_QUAD && 2 * col + mc > g.cols - 1) continue;
      const int zr = mr ? g.lines - 1 - row : row, zc = mc ? g.cols - 1 - col : col;
      part[((size_t)(slice0 + pl.slice) * ngroups + gi) * npix + (size_t)zr * g.cols + zc] = tot[i][z];
    }
  }
}

// rows[group][a][r] = the planes' values sino[slice][r'][a'] * scale[a'] of ray r at angle a
__global__ __launch_bounds__(256) void k_dda_rows_planes(int R, int A, int kind, int nslices,
                                                         const float* __restrict__ sino,
                                                         const float* __restrict__ scale, ss_f32x4* __restrict__ rows) {
  __shared__ float T[SS_PLANES][32][33];
  const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;
  const int br = blockIdx.x * 32, ba = blockIdx.y * 32;
#pragma unroll
  for (int z = 0; z < SS_PLANES; ++z) {
    const SSPlane pl = ss_plane(kind, z);
    const size_t slice = (size_t)min((int)blockIdx.z * ss_planes_slices(kind) + pl.slice, nslices - 1);
    const float* __restrict__ src = sino + slice * (size_t)R * A;
    const int a = ba + tx, az = pl.mirror ? A - 1 - a : a;
    const float sc = a < A ? scale[az] : 0.f;
#pragma unroll
    for (int yy = ty; yy < 32; yy += 8) {
      const int r = br + yy, rz = pl.turn ? R - 1 - r : r;
      T[z][tx][yy] = a < A && r < R ? src[(size_t)rz * A + az] * sc : 0.f;
    }
  }
  __syncthreads();
  ss_f32x4* dst = rows + (size_t)blockIdx.z * A * R;
#pragma unroll
  for (int yy = ty; yy < 32; yy += 8) {
    const int a = ba + yy, r = br + tx;
    if (a < A && r < R) dst[(size_t)a * R + r] = ss_f32x4{T[0][yy][tx], T[1][yy][tx], T[2][yy][tx], T[3][yy][tx]};
  }
}

// rows[slice][a][2 + r] = sino[slice][r][a] * scale[a], two zeros either side of each row
__global__ __launch_bounds__(256) void k_dda_sino_rows(int R, int A, const float* __restrict__ sino,
                                                       const float* __restrict__ scale, float* __restrict__ rows) {
  __shared__ float tile[DDA_TILE][DDA_TILE + 1];
  const size_t slice = blockIdx.z;
  const int r0 = blockIdx.y * DDA_TILE, a0 = blockIdx.x * DDA_TILE;
  const int pitch = R + 4;
  const float* __restrict__ s = sino + slice * (size_t)R * A;
  float* __restrict__ o = rows + slice * (size_t)A * pitch;
  for (int rr = threadIdx.y; rr < DDA_TILE; rr += blockDim.y) {
    const int r = r0 + rr, a = a0 + threadIdx.x;
    tile[rr][threadIdx.x] = (r < R && a < A) ? s[(size_t)r * A + a] : 0.f;
  }
  __syncthreads();
  for (int aa = threadIdx.y; aa < DDA_TILE; aa += blockDim.y) {
    const int a = a0 + aa, r = r0 + threadIdx.x;
    if (a < A && r < R) o[(size_t)a * pitch + 2 + r] = tile[threadIdx.x][aa] * scale[a];
    if (a < A && blockIdx.y == 0 && threadIdx.x < 4) {
      const int pad = threadIdx.x < 2 ? threadIdx.x : R + threadIdx.x;  // 0, 1, R + 2, R + 3
      o[(size_t)a * pitch + pad] = 0.f;
    }
  }
}

// ---------------------------------------------------------------- layouts

template <typename T>
__global__ __launch_bounds__(256) void k_dda_fill(T* __restrict__ p, size_t n) {
  for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x) p[i] = T(0);
}

// Straight angles: vcol[slice][j] (vline[slice][i]) = sum over the straight angles whose
// slow index is the column (line) of len * (sum of q over the rays of that index), q = 1
// for `ones`; FP64 sums.  One thread per column, then per line.
template <typename T>
__global__ __launch_bounds__(256) void k_dda_straight(SSDdaGeom g, const SSDdaStraight* __restrict__ st, int nst,
                                                      const int* __restrict__ ranges, const float* __restrict__ sino,
                                                      int ones, T* __restrict__ vcol, T* __restrict__ vline) {
  const int idx = blockIdx.x * blockDim.x + threadIdx.x;
  const size_t slice = blockIdx.y;
  if (idx >= g.cols + g.lines) return;
  const int col = idx < g.cols;
  const int s = col ? idx : idx - g.cols;
  const float* __restrict__ q = sino + slice * (size_t)g.nrays * g.nangles;
  double sum = 0.0;
  for (int k = 0; k < nst; ++k) {
    const SSDdaStraight S = st[k];
    if (S.slow_col != col) continue;
    const int lo = ranges[S.off + 2 * s], hi = ranges[S.off + 2 * s + 1];
    double qs = 0.0;
    if (ones)
      qs = hi - lo;
    else
      for (int r = lo; r < hi; ++r) qs += (double)q[(size_t)r * g.nangles + S.a];
    sum = fma(qs, S.len, sum);
  }
  if (col)
    vcol[slice * g.cols + s] = T(sum);
  else
    vline[slice * g.lines + s] = T(sum);
}

// out[lines][cols] = acc[lines][cols] + more[lines][cols] + accT[cols][lines]^T + vcol[cols] +
// vline[lines] (more, accT, vcol, vline may be null), divided by w when given.  acc: the sum, in order, of
// ngroups partial images [slice][group][lines][cols] of type P.
// Block (32, 8) handles a 32 x 32 tile; accT is read along its lines through LDS.
template <typename T, typename Out, typename P>
__global__ __launch_bounds__(256) void k_dda_fold(int lines, int cols, const P* __restrict__ acc, int ngroups,
                                                  const T* __restrict__ more,
                                                  const T* __restrict__ accT, const T* __restrict__ vcol,
                                                  const T* __restrict__ vline, const double* __restrict__ w,
                                                  Out* __restrict__ out) {
  __shared__ T tile[DDA_TILE][DDA_TILE + 1];
  const size_t slice = blockIdx.z;
  const size_t npix = (size_t)lines * cols;
  const int i0 = blockIdx.y * DDA_TILE, j0 = blockIdx.x * DDA_TILE;
  const T* aT = accT ? accT + slice * npix : nullptr;
  for (int jj = threadIdx.y; jj < DDA_TILE; jj += blockDim.y) {
    const int j = j0 + jj, i = i0 + threadIdx.x;
    tile[jj][threadIdx.x] = (accT && j < cols && i < lines) ? aT[(size_t)j * lines + i] : T(0);
  }
  __syncthreads();
  for (int ii = threadIdx.y; ii < DDA_TILE; ii += blockDim.y) {
    const int i = i0 + ii, j = j0 + threadIdx.x;
    if (i < lines && j < cols) {
      const size_t p = (size_t)i * cols + j;
      P sum = P(0);
#pragma unroll 4
      for (int k = 0; k < ngroups; ++k) sum += acc[(slice * ngroups + k) * npix + p];
      T v = T(sum) + tile[threadIdx.x][ii];
      if (more) v += more[slice * npix + p];
      if (vcol) v += vcol[slice * cols + j] + vline[slice * lines + i];
      out[slice * npix + p] = w ? Out((double)v / w[p]) : Out(v);
    }
  }
}

// The Radon's padded layouts of img[slice][lines][cols]: pad[slice][lines][pc] and
// padT[slice][cols][pl] (the transpose), pc = dda_pad_pitch(cols), pl =
// dda_pad_pitch(lines): each line DDA_PADW zeros, its pixels, then zeros to the pitch.
// Block (32, 8) copies a 32 x 32 tile, the transposed copy through LDS; the first and
// last tile of a line also write its padding.
__global__ __launch_bounds__(256) void k_dda_pad_images(int lines, int cols, const float* __restrict__ src,
                                                        float* __restrict__ pad, float* __restrict__ padT) {
  __shared__ float tile[DDA_TILE][DDA_TILE + 1];
  const size_t slice = blockIdx.z;
  const int i0 = blockIdx.y * DDA_TILE, j0 = blockIdx.x * DDA_TILE;
  const int pc = dda_pad_pitch(cols), pl = dda_pad_pitch(lines);
  const float* __restrict__ s = src + slice * (size_t)lines * cols;
  float* __restrict__ o = pad + slice * (size_t)lines * pc;
  float* __restrict__ oT = padT + slice * (size_t)cols * pl;
  const int x = threadIdx.x;
  for (int ii = threadIdx.y; ii < DDA_TILE; ii += blockDim.y) {
    const int i = i0 + ii, j = j0 + x;
    const float v = (i < lines && j < cols) ? s[(size_t)i * cols + j] : 0.f;
    tile[ii][x] = v;
    if (i < lines) {
      float* __restrict__ line = o + (size_t)i * pc;
      if (j < cols) line[j + DDA_PADW] = v;
      if (blockIdx.x == 0)
        for (int c = x; c < DDA_PADW; c += DDA_TILE) line[c] = 0.f;
      if (j0 + DDA_TILE >= cols)
        for (int c = cols + DDA_PADW + x; c < pc; c += DDA_TILE) line[c] = 0.f;
    }
  }
  __syncthreads();
  for (int jj = threadIdx.y; jj < DDA_TILE; jj += blockDim.y) {
    const int j = j0 + jj, i = i0 + x;
    if (j < cols) {
      float* __restrict__ line = oT + (size_t)j * pl;
      if (i < lines) line[i + DDA_PADW] = tile[x][jj];
      if (blockIdx.y == 0)
        for (int c = x; c < DDA_PADW; c += DDA_TILE) line[c] = 0.f;
      if (i0 + DDA_TILE >= lines)
        for (int c = lines + DDA_PADW + x; c < pl; c += DDA_TILE) line[c] = 0.f;
    }
  }
}

// ---------------------------------------------------------------- launchers

static dim3 dda_tiles(int lines, int cols, int nslices) {
  return dim3((cols + DDA_TILE - 1) / DDA_TILE, (lines + DDA_TILE - 1) / DDA_TILE, nslices);
}

// The planes a launch takes
static int dda_planes_kind(const SSDdaTransposePlan& tp, int nslices) {
  if (ss_planes_stack(nslices)) return SS_PLANES_SLICES;
  if (tp.sym & DDA_SYM_MIRROR) return SS_PLANES_QUAD;
  if ((tp.sym & DDA_SYM_TURN) && nslices >= 2) return SS_PLANES_PAIR;
  return nslices >= 3 ? SS_PLANES_SLICES : SS_PLANES_NONE;
}

static SSDdaRadonPlanes dda_radon_planes(const SSDdaGeom& g, const SSDdaTransposePlan& tp, int kind, int nslices) {
  SSDdaRadonPlanes rp;
  rp.kind = kind;
  rp.nslices = nslices;
  rp.nangles = kind == SS_PLANES_QUAD ? (g.nangles + 1) / 2 : g.nangles;
  rp.nrays = kind == SS_PLANES_SLICES ? g.nrays : (g.nrays + 1) / 2;
  rp.order = ss_planes_order(rp.nrays, rp.nangles);
  const int nf = std::max(g.lines, g.cols);
  const long long blocks = (long long)rp.order.blocks * ss_planes_groups(kind, nslices);
  rp.nslab = ss_radon_slab_plan(nf, blocks, &rp.slab_rows,
                                (int)std::min<long long>(SS_PLANES_SLAB_BLOCKS, blocks * (nf / DDA_RP_MIN_ROWS)));
  rp.straight = tp.straight;
  rp.nstraight = tp.nstraight;
  rp.walk = tp.walk;
  rp.nwalk = tp.nwalk;
  return rp;
}

static long long dda_radon_planes_blocks(const SSDdaGeom& g, const SSDdaRadonPlanes& rp) {
  const int wide = RADON_WAVES * SS_WAVE;
  return (long long)rp.order.blocks * rp.nslab * ss_planes_groups(rp.kind, rp.nslices) +
         ((long long)rp.nstraight * ((g.nrays + 63) / 64) + (long long)rp.nwalk * ((g.nrays + wide - 1) / wide)) *
             rp.nslices;
}

SSDdaRadonForm dda_radon_form(const SSDdaGeom& g, const SSDdaTransposePlan& tp, int nslices) {
  SSDdaRadonForm f{SS_PLANES_NONE, 1, 0, 0};
  f.layout = sizeof(float) * dda_radon_scratch_floats(g, nslices);
  if (tp.ngather == 0) return f;
  // a traced ray's pixel offsets are ints
  if ((long long)std::max(g.lines, g.cols) * (std::max(g.lines, g.cols) + 2 * DDA_RP_PAD) >= (1LL << 31)) return f;
  const int kind = dda_planes_kind(tp, nslices);
  if (kind == SS_PLANES_NONE) return f;
  const int groups = ss_planes_groups(kind, nslices);
  const SSDdaRadonPlanes rp = dda_radon_planes(g, tp, kind, nslices);
  if (dda_radon_planes_blocks(g, rp) * RADON_WAVES * SS_WAVE > SS_GRID_THREADS) return f;
  f.kind = kind;
  f.nslab = rp.nslab;
  f.layout = sizeof(ss_f32x4) * (size_t)groups *
             ((size_t)g.lines * (g.cols + 2 * DDA_RP_PAD) + (size_t)g.cols * (g.lines + 2 * DDA_RP_PAD));
  f.part = rp.nslab > 1 ? sizeof(double) * (size_t)nslices * rp.nslab * g.nangles * g.nrays : 0;
  return f;
}

hipError_t dda_launch_radon(const SSDdaGeom& g, const SSDdaTransposePlan& tp, const float* img, void* layout,
                            double* part, float* sino, int nslices, hipStream_t stream) {
  const SSDdaAngle* angles = tp.angles;
  const SSDdaRadonForm form = dda_radon_form(g, tp, nslices);
  if (form.kind != SS_PLANES_NONE) {
    const int groups = ss_planes_groups(form.kind, nslices);
    const SSDdaRadonPlanes rp = dda_radon_planes(g, tp, form.kind, nslices);
    ss_f32x4* L = static_cast<ss_f32x4*>(layout);
    ss_f32x4* LT = L + (size_t)groups * g.lines * (g.cols + 2 * DDA_RP_PAD);
    hipLaunchKernelGGL(k_dda_pad_planes, dda_tiles(g.lines, g.cols, groups), dim3(256), 0, stream, g.lines, g.cols,
                       form.kind, nslices, img, L, LT);
    const unsigned blocks = (unsigned)dda_radon_planes_blocks(g, rp);
    if (rp.nslab > 1) {
      hipLaunchKernelGGL(k_dda_radon_planes<true>, dim3(blocks), dim3(RADON_WAVES * SS_WAVE), 0, stream, g, angles, rp,
                         (const ss_f32x4*)L, (const ss_f32x4*)LT, sino, part);
      hipLaunchKernelGGL(k_dda_radon_finish, dim3((g.nrays + 31) / 32, (g.nangles + 31) / 32, nslices), dim3(256), 0,
                         stream, g, angles, rp.nslab, (const double*)part, sino);
    } else {
      hipLaunchKernelGGL(k_dda_radon_planes<false>, dim3(blocks), dim3(RADON_WAVES * SS_WAVE), 0, stream, g, angles, rp,
                         (const ss_f32x4*)L, (const ss_f32x4*)LT, sino, part);
    }
    return hipGetLastError();
  }
  float* img_pad = static_cast<float*>(layout);
  float* imgT_pad = img_pad + (size_t)nslices * g.lines * dda_pad_pitch(g.cols);
  hipLaunchKernelGGL(k_dda_pad_images, dda_tiles(g.lines, g.cols, nslices), dim3(DDA_TILE, 8), 0, stream, g.lines,
                     g.cols, img, img_pad, imgT_pad);
  hipLaunchKernelGGL(k_dda_radon, dim3((g.nrays + 255) / 256, g.nangles, nslices), dim3(256), 0, stream, g, angles,
                     (const float*)img_pad, (const float*)imgT_pad, sino);
  return hipGetLastError();
}

static int dda_gp_cols(const SSDdaGeom& g, int kind) {
  return ((kind == SS_PLANES_QUAD ? (g.cols + 1) / 2 : g.cols) + 31) / 32;
}
static int dda_gp_rows(const SSDdaGeom& g, int kind) {
  return ((kind == SS_PLANES_SLICES ? g.lines : (g.lines + 1) / 2) + 8 * DDA_GP_ROWS - 1) / (8 * DDA_GP_ROWS);
}

SSDdaGatherForm dda_gather_form(const SSDdaGeom& g, const SSDdaTransposePlan& tp, bool ones, int nslices) {
  SSDdaGatherForm f{SS_PLANES_NONE, 1};
  if (ones || tp.ngather == 0 || tp.planes_ws <= 0) return f;
  f.kind = dda_planes_kind(tp, nslices);
  if (f.kind == SS_PLANES_NONE) return f;
  const long long tiles = (long long)dda_gp_cols(g, f.kind) * dda_gp_rows(g, f.kind) * ss_planes_groups(f.kind, nslices);
  const long long want = std::max<long long>((DDA_GP_BLOCKS + tiles / 2) / tiles, tiles <= DDA_GP_PAIR_TILES ? 2 : 1);
  f.ngroups = (int)std::min<long long>({DDA_GP_MAXGROUPS, want, (tp.ngather + DDA_GP_ANGLES - 1) / DDA_GP_ANGLES});
  if (tiles * f.ngroups * 256 > SS_GRID_THREADS) return SSDdaGatherForm{SS_PLANES_NONE, 1};
  return f;
}

SSDdaTransposeScratch dda_transpose_scratch(const SSDdaGeom& g, const SSDdaTransposePlan& tp, bool ones, int nslices,
                                            size_t sizeof_t) {
  const size_t npix = (size_t)g.lines * g.cols, n = npix * nslices;
  const SSDdaGatherForm f = dda_gather_form(g, tp, ones, nslices);
  SSDdaTransposeScratch b;
  if (f.kind != SS_PLANES_NONE) {
    b.sino = sizeof(ss_f32x4) * (size_t)g.nrays * g.nangles * ss_planes_groups(f.kind, nslices);
    b.acc = sizeof(double) * n * f.ngroups;
    // the traced angles' two images, or the straight angles' vectors
    b.accT = tp.nwalk > 0 ? 2 * sizeof_t * n : (tp.nstraight > 0 ? sizeof_t * (size_t)nslices * (g.lines + g.cols) : 0);
  } else {
    b.sino = sizeof(float) * (size_t)(g.nrays + 4) * g.nangles * nslices;
    b.acc = b.accT = sizeof_t * n;
  }
  return b;
}

template <typename T, typename Out>
hipError_t dda_launch_transpose(const SSDdaGeom& g, const SSDdaTransposePlan& tp, const float* sino, bool ones,
                                float* sinoT, void* acc_, T* accT, const double* w, Out* out, int nslices,
                                hipStream_t stream) {
  const size_t n = (size_t)g.lines * g.cols * nslices;
  T* acc = static_cast<T*>(acc_);
  const SSDdaGatherForm form = dda_gather_form(g, tp, ones, nslices);
  if (form.kind != SS_PLANES_NONE) {
    const int groups = ss_planes_groups(form.kind, nslices);
    const int tc = dda_gp_cols(g, form.kind), tr = dda_gp_rows(g, form.kind);
    ss_f32x4* rows = reinterpret_cast<ss_f32x4*>(sinoT);
    hipLaunchKernelGGL(k_dda_rows_planes, dim3((g.nrays + 31) / 32, (g.nangles + 31) / 32, groups), dim3(256), 0,
                       stream, g.nrays, g.nangles, form.kind, nslices, sino, tp.row_scale, rows);
    hipLaunchKernelGGL(k_dda_gather_planes, dim3((unsigned)(tc * tr * groups * form.ngroups)), dim3(256), 0, stream, g,
                       tp.gather, tp.ngather, (const ss_f32x4*)rows, form.kind, nslices, tp.planes_ws, form.ngroups,
                       tc, tr, static_cast<double*>(acc_));
  } else if (tp.ngather > 0) {
    if (!ones)  // angle-major, lmax-scaled, zero-padded copy of the sinogram
      hipLaunchKernelGGL(k_dda_sino_rows, dda_tiles(g.nrays, g.nangles, nslices), dim3(DDA_TILE, 8), 0, stream,
                         g.nrays, g.nangles, sino, tp.row_scale, sinoT);
    const dim3 grid((g.cols + DDA_GX - 1) / DDA_GX, (g.lines + DDA_GY - 1) / DDA_GY, nslices);
    if (tp.kmax <= 2 && !ones && tp.gather_ws > 0) {
      // the taller tiles halve the per-angle work per pixel; they need a block per CU
      const int gx = (g.cols + DDA_G2_COLS - 1) / DDA_G2_COLS;
      const int gy = (g.lines + 4 * DDA_G2_LINES - 1) / (4 * DDA_G2_LINES);
      if ((long long)gx * gy * nslices >= 256)
        hipLaunchKernelGGL((k_dda_gather2<T, DDA_G2_LINES>), dim3(gx, gy, nslices), dim3(256), 0, stream, g,
                           tp.gather, tp.ngather, (const float*)sinoT, tp.gather_ws, acc);
      else
        hipLaunchKernelGGL((k_dda_gather2<T, DDA_G2_LINES_SMALL>), dim3(gx, (g.lines + 4 * DDA_G2_LINES_SMALL - 1) /
                                                                          (4 * DDA_G2_LINES_SMALL), nslices),
                           dim3(256), 0, stream, g, tp.gather, tp.ngather, (const float*)sinoT, tp.gather_ws, acc);
    }
    else if (tp.kmax <= 2)
      hipLaunchKernelGGL((k_dda_gather<T, 2>), grid, dim3(256), 0, stream, g, tp.gather, tp.ngather,
                         (const float*)sinoT, ones ? 1 : 0, acc);
    else
      hipLaunchKernelGGL((k_dda_gather<T, 0>), grid, dim3(256), 0, stream, g, tp.gather, tp.ngather,
                         (const float*)sinoT, ones ? 1 : 0, acc);
  } else {
    hipLaunchKernelGGL(k_dda_fill<T>, dim3(1024), dim3(256), 0, stream, acc, n);
  }
  if (tp.nwalk > 0) {
    if (form.kind != SS_PLANES_NONE) acc = accT + n;  // beside the gather's FP64 images
    hipLaunchKernelGGL(k_dda_fill<T>, dim3(1024), dim3(256), 0, stream, accT, form.kind != SS_PLANES_NONE ? 2 * n : n);
    hipLaunchKernelGGL(k_dda_scatter<T>, dim3((g.nrays + 255) / 256, tp.nwalk, nslices), dim3(256), 0, stream, g,
                       tp.angles, tp.walk, sino, ones ? 1 : 0, acc, accT);
  }
  // straight angles (present only without traced ones): column and line vectors in accT,
  // [nslices][cols] then [nslices][lines] (lines * cols >= lines + cols for sides >= 2)
  T* vcol = nullptr;
  T* vline = nullptr;
  if (tp.nstraight > 0 && tp.nwalk == 0) {
    vcol = accT;
    vline = accT + (size_t)nslices * g.cols;
    hipLaunchKernelGGL(k_dda_straight<T>, dim3((g.cols + g.lines + 255) / 256, nslices), dim3(256), 0, stream, g,
                       tp.straight, tp.nstraight, tp.ranges, sino, ones ? 1 : 0, vcol, vline);
  }
  if (form.kind != SS_PLANES_NONE)
    hipLaunchKernelGGL((k_dda_fold<T, Out, double>), dda_tiles(g.lines, g.cols, nslices), dim3(DDA_TILE, 8), 0, stream,
                       g.lines, g.cols, (const double*)acc_, form.ngroups, (const T*)(tp.nwalk > 0 ? acc : nullptr),
                       (const T*)(tp.nwalk > 0 ? accT : nullptr), (const T*)vcol, (const T*)vline, w, out);
  else
    hipLaunchKernelGGL((k_dda_fold<T, Out, T>), dda_tiles(g.lines, g.cols, nslices), dim3(DDA_TILE, 8), 0, stream,
                       g.lines, g.cols, (const T*)acc, 1, (const T*)nullptr,
                       (const T*)(tp.nwalk > 0 ? accT : nullptr), (const T*)vcol, (const T*)vline, w, out);
  return hipGetLastError();
}

__global__ __launch_bounds__(256) void k_dda_to_f32(const double* __restrict__ src, float* __restrict__ dst, size_t n) {
  for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x)
    dst[i] = (float)src[i];
}

hipError_t dda_launch_to_f32(const double* src, float* dst, size_t n, hipStream_t stream) {
  hipLaunchKernelGGL(k_dda_to_f32, dim3(1024), dim3(256), 0, stream, src, dst, n);
  return hipGetLastError();
}

template hipError_t dda_launch_transpose<float, float>(const SSDdaGeom&, const SSDdaTransposePlan&, const float*,
                                                      bool, float*, void*, float*, const double*, float*, int,
                                                      hipStream_t);
template hipError_t dda_launch_transpose<double, float>(const SSDdaGeom&, const SSDdaTransposePlan&, const float*,
                                                       bool, float*, void*, double*, const double*, float*, int,
                                                       hipStream_t);
template hipError_t dda_launch_transpose<double, double>(const SSDdaGeom&, const SSDdaTransposePlan&, const float*,
                                                        bool, float*, void*, double*, const double*, double*, int,
                                                        hipStream_t);
