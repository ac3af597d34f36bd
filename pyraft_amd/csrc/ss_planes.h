// ss_planes.h -- planes: values of up to four images or sinograms that one ray coordinate
// serves, stored together (the forms are described at their kernels).
#ifndef PYRAFT_AMD_SS_PLANES_H
#define PYRAFT_AMD_SS_PLANES_H

#include <hip/hip_runtime.h>
#include <stdint.h>

#define SS_PLANES 4
#define SS_WAVE 64

// Threads of a launch along one dimension at most; HIP cuts a longer one short without an error
#define SS_GRID_THREADS 0xffffffffLL

#ifndef RADON_WAVES
#define RADON_WAVES 8  // angles (one per wave) of a Radon block
#endif

// What the four planes of a launch are, the slices that
// a group of planes covers, and the groups of a launch
enum { SS_PLANES_NONE = 0, SS_PLANES_QUAD = 1, SS_PLANES_PAIR = 2, SS_PLANES_SLICES = 3 };
static inline __host__ __device__ int ss_planes_slices(int kind) {
  return kind == SS_PLANES_QUAD ? 1 : (kind == SS_PLANES_PAIR ? 2 : 4);
}
static inline int ss_planes_groups(int kind, int nslices) {
  return (nslices + ss_planes_slices(kind) - 1) / ss_planes_slices(kind);
}

// Whether a stack goes in groups of four slices also where a symmetry would serve: above
// SS_PLANES_STACK slices (smaller launches sum in one slice's order) if at most one plane in 17
// stays empty.  The planes are then copies of different slices, not four views of one, so the
// copies take a quarter of the memory and time (us, quad against slices: Radon 64 x 512^2 x 720
// 1790 / 1643, 54 x 671^2 x 352 1709 / 1281, 64 x 128^2 x 100 91 / 54; transpose 64 x 512^2 x 720
// 1631 / 1428; line Radon 64 x 512^2 x 720 1958 / 1727).
#define SS_PLANES_STACK 8
static inline bool ss_planes_stack(int nslices) {
  return nslices > SS_PLANES_STACK && 16 * ((nslices + 3) / 4 * 4) <= 17 * nslices;
}

// Order of a planes launch's blocks: consecutive blocks go to the 8 XCDs in turn, each with an
// L2 of its own.  A unit is a c-th of a ray group's angle blocks; the units, from the long rays
// at the detector's centre to the short ones at its edge, are dealt to the XCDs there and
// back, so that each XCD gets the same mix and walks one strip of the image with slowly
// turning angles at a time.
struct SSPlanesOrder {
  int g, y;       // ray groups, angle blocks
  int c, yc;      // units per ray group, angle blocks per unit at most
  int blocks;     // blocks launched; those past a unit's angle blocks have no work
};
static inline SSPlanesOrder ss_planes_order(int nrays, int nangles) {
  SSPlanesOrder o;
  o.g = (nrays + SS_WAVE - 1) / SS_WAVE;
  o.y = (nangles + RADON_WAVES - 1) / RADON_WAVES;
  o.c = 1;
  while (o.g * o.c % 16 && o.c < o.y) o.c *= 2;
  if (o.c > o.y) o.c = o.y;
  o.yc = (o.y + o.c - 1) / o.c;
  o.blocks = (o.g * o.c + 15) / 16 * 16 * o.yc;
  return o;
}

#if defined(__HIPCC__)
typedef float ss_f32x4 __attribute__((ext_vector_type(4)));

// plane z of a launch: its slice within the group, whether it is the half turn of its image
// and whether the mirror
struct SSPlane {
  int slice;
  bool turn, mirror;
};
__device__ __host__ __forceinline__ SSPlane ss_plane(int kind, int z) {
  if (kind == SS_PLANES_QUAD) return SSPlane{0, (z & 1) != 0, (z & 2) != 0};
  if (kind == SS_PLANES_PAIR) return SSPlane{z >> 1, (z & 1) != 0, false};
  return SSPlane{z, false, false};
}

// Column of a lane in its 32-pixel tile row.  A 16-byte LDS read serves 16 lanes of a half
// wave per pass, the lanes 0-3, 12-15, 20-27 and then the others; giving each of the two
// sets 16 neighbouring columns keeps a pass within 16 neighbouring records, so that no two
// of them share a bank (pixels are at most one ray apart).
__device__ __forceinline__ int ss_bp_column(int lane) {
  const int q = (lane >> 2) & 7;
  return ((0x73261540 >> (4 * q)) & 7) * 4 + (lane & 3);
}

// Ray of a lane within its group of 64: a 16-byte LDS read serves the lanes 0-3, 12-15,
// 20-27 of a half wave in one pass and the others in the next; each set gets 16 neighbours.
__device__ __forceinline__ int ss_plane_ray(int lane) { return (lane & 32) + ss_bp_column(lane); }

// ray group and angle block of block `id`; (0, -1): no work
__device__ __forceinline__ int2 ss_planes_place(const SSPlanesOrder& o, int id) {
  const int xcd = id % 8, turn = id / 8;
  const int deal = turn / o.yc;
  const int unit = deal * 8 + (deal & 1 ? 7 - xcd : xcd);
  const int part = unit % o.c;
  const int ablk = (int)((long long)o.y * part / o.c) + turn % o.yc;
  if (unit >= o.g * o.c || ablk >= (int)((long long)o.y * (part + 1) / o.c)) return make_int2(0, -1);
  return make_int2(o.g - 1 - unit / o.c, ablk);
}

#ifndef RADON_ROW_ROUND
#define RADON_ROW_ROUND 8  // chunk rows rounded down to a multiple of this where the window allows
#endif

#define RADON_TABLE SS_WAVE  // chunks per window table: one (chunk, wave) pair per thread

typedef __attribute__((address_space(1))) const void* ss_global_cptr;
typedef __attribute__((address_space(3))) void* ss_lds_ptr;

// wave-uniform copies (scalar registers) of values the compiler cannot prove uniform
__device__ __forceinline__ int ss_rfl(int v) { return __builtin_amdgcn_readfirstlane(v); }
__device__ __forceinline__ int64_t ss_rfl64(int64_t v) {
  const uint32_t lo = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)v);
  const uint32_t hi = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)((uint64_t)v >> 32));
  return (int64_t)(((uint64_t)hi << 32) | lo);
}
__device__ __forceinline__ float ss_rflf(float v) { return __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(v))); }
typedef __attribute__((address_space(3))) const ss_f32x4* ss_lds_cell;

// staged cells per block and sample rows per chunk at most: two 512-thread blocks per CU
#define PLANES_CAP 4864
#define PLANES_CHUNK 40
#define PLANES_BLOCKS 2

struct SSPlanesLds {
  double red[RADON_WAVES];
  int64_t wpar[RADON_WAVES][3];  // as SSRadonLds
  int wmeta[RADON_WAVES][3];
  int wred[2][RADON_WAVES];
  int2 table[RADON_TABLE];
  alignas(16) ss_f32x4 stage[PLANES_CAP + 2];  // chunk window; cells CAP, CAP + 1 stay 0
};

// Window table of `nch` chunks of `rows` sample rows from row sc (the last chunk ends
// at s_hi at the latest): for each chunk, the gather records [rec0, rec0 + Wc) of each
// row that the block's waves read in its rows (Wc = 0: none).  Each thread takes one
// (chunk, wave) pair, bounds the cells of that wave's rays over the chunk's rows at the
// corners (the trajectory is affine in ray and row; valid samples have cells in
// [-1, n-1]), and the RADON_WAVES lanes of a chunk take the union.  Returns the widest
// Wc of the table (block-uniform); `pass` selects the reduction slots, so that a second
// pass right after the first needs no barrier in between.
template <bool PAIRS, class Lds>
__device__ __forceinline__ int ss_radon_windows(Lds& lds, int pass, int sc, int rows, int nch, int s_hi, int n) {
  const int t = threadIdx.x;
  const int c = t / RADON_WAVES, w = t % RADON_WAVES;
  int cmin = 0x7fffffff, cmax = -0x7fffffff;
  if (c < nch) {
    const int s0 = sc + c * rows, s1 = min(s0 + rows, s_hi + 1);
    const int ra = max(s0, lds.wmeta[w][1]), rb = min(s1 - 1, lds.wmeta[w][2]);
    if (lds.wmeta[w][0] >= 0 && ra <= rb) {
      const int64_t beta = lds.wpar[w][2];
      const int64_t c00 = lds.wpar[w][0] + (int64_t)ra * beta;
      const int64_t c10 = lds.wpar[w][1] + (int64_t)ra * beta;
      const int64_t ds = (int64_t)(rb - ra) * beta;
      const int m0 = (int)(c00 >> 32), m1 = (int)(c10 >> 32);
      const int m2 = (int)((c00 + ds) >> 32), m3 = (int)((c10 + ds) >> 32);
      cmin = max(min(min(m0, m1), min(m2, m3)), -1);
      cmax = min(max(max(m0, m1), max(m2, m3)), n - 1);
    }
  }
  for (int off = 1; off < RADON_WAVES; off <<= 1) {
    cmin = min(cmin, __shfl_xor(cmin, off));
    cmax = max(cmax, __shfl_xor(cmax, off));
  }
  // pair records: cells c_lo..c_hi need records c_lo+1..c_hi+1; rec0 is even so that rows of
  // the window start 16-byte aligned in the layout (even pitch) and in LDS (even Wc).  Plane
  // cells (16 bytes each): c_lo+1..c_hi+2, the upper tap being the next cell
  const int rec0 = PAIRS ? (cmin + 1) & ~1 : cmin + 1;
  int wc = 0;
  if (cmax >= cmin) wc = PAIRS ? ((cmax + 2 - rec0) + 1) & ~1 : cmax + 3 - rec0;
  if (c >= nch) wc = 0;
  if (c < nch && w == 0) lds.table[c] = make_int2(rec0, wc);
  for (int off = 32; off > 0; off >>= 1) wc = max(wc, __shfl_xor(wc, off));
  if ((t & (SS_WAVE - 1)) == 0) lds.wred[pass][t / SS_WAVE] = wc;
  __syncthreads();
  int wmax = 0;
  for (int i = 0; i < RADON_WAVES; ++i) wmax = max(wmax, lds.wred[pass][i]);
  return ss_rfl(wmax);
}

// The chunks of sample rows [s_lo, s_hi] of a planes block (all its waves; a block-uniform
// call): bounds the cells that every wave can touch, copies that window of the layout into
// lds.stage and calls body(s0, s1, first cell, cells per row, whether it was staged) for rows
// [s0, s1).  Super-chunks of up to RADON_TABLE chunks share one pass over the windows.
template <typename Body>
__device__ __forceinline__ void ss_planes_chunks(SSPlanesLds& lds, const ss_f32x4* __restrict__ lay, int pitch, int n,
                                                 int s_lo, int s_hi, int wv, int lane, Body body) {
  for (int sc = s_lo; sc <= s_hi;) {  // block-uniform
    int rows = PLANES_CHUNK;
    int nch = min(RADON_TABLE, (s_hi - sc + rows) / rows);
    const int wmax = ss_radon_windows<false>(lds, 0, sc, rows, nch, s_hi, n);
    if (wmax * rows > PLANES_CAP) {
      int r2 = PLANES_CAP / wmax;
      if (r2 >= RADON_ROW_ROUND) r2 = r2 / RADON_ROW_ROUND * RADON_ROW_ROUND;
      rows = max(r2, 1);
      nch = min(RADON_TABLE, (s_hi - sc + rows) / rows);
      (void)ss_radon_windows<false>(lds, 1, sc, rows, nch, s_hi, n);
    }
    for (int c = 0; c < nch; ++c) {
      const int s0 = sc + c * rows, s1 = min(s0 + rows, s_hi + 1);
      const int2 tw = lds.table[c];
      const int rec0 = ss_rfl(tw.x), Wc = ss_rfl(tw.y);
      const bool fits = Wc > 0 && (s1 - s0) * Wc <= PLANES_CAP;  // block-uniform
      if (c > 0) __syncthreads();  // every wave is done with the previous chunk
      if (fits) {
        const ss_f32x4* src0 = lay + (size_t)(s0 + wv) * pitch + rec0 + lane;
        for (int seg = 0; seg < Wc; seg += SS_WAVE) {
          if (seg + lane < Wc) {
            const ss_f32x4* src = src0 + seg;
            ss_f32x4* dst = lds.stage + wv * Wc + seg;
            for (int r = wv; r < s1 - s0; r += RADON_WAVES) {
              __builtin_amdgcn_global_load_lds((ss_global_cptr)src, (ss_lds_ptr)dst, 16, 0, 0);
              src += (size_t)RADON_WAVES * pitch;
              dst += RADON_WAVES * Wc;
            }
          }
        }
      }
      __syncthreads();  // window staged
      body(s0, s1, rec0, Wc, fits);
    }
    sc += nch * rows;
  }
}
#endif

#endif
