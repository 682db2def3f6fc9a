// Per-thread bodies of the parallel-beam projectors, shared by the
// one-problem kernels (parallel.hip) and the batched persistent kernels
// (batched.hip).  Model: Core/src/p2D.cpp (see parallel.hip).
#pragma once

#include <hip/hip_runtime.h>

#include "common.hpp"

namespace ccpi {

// Device memory reached through a pointer typed as global: loads and stores
// compile to global (not flat) accesses.  The batched kernels read their
// problems' pointers from descriptors in device memory, which leaves them
// generic to the compiler; generic accesses wait on the scalar and vector
// memory counters both and need 64-bit addresses in vector registers.  The
// bodies below reach all their arrays through gmem.
#define CCPI_GLOBAL __attribute__((address_space(1)))
template <class T>
__device__ inline CCPI_GLOBAL T *gmem(T *p) {
  return (CCPI_GLOBAL T *)p;
}

// A plan table at a uniform address: scalar loads, whatever memory the kernel
// writes meanwhile (no kernel writes the tables it reads).
#define CCPI_CONST __attribute__((address_space(4)))
template <class T>
__device__ inline const CCPI_CONST T *cmem(const T *p) {
  return (const CCPI_CONST T *)(uintptr_t)p;
}

// 16 bytes at p (4-byte aligned) as one load.
__device__ inline float4 load_f4(const CCPI_GLOBAL float *p) {
  float4 v;
  __builtin_memcpy(&v, p, sizeof(v));
  return v;
}

// Minimum and maximum of numbers, without the canonicalisation that the
// library's take for a signalling NaN.
__device__ inline double min_f64(double a, double b) {
  double r;
  asm("v_min_f64 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
  return r;
}
__device__ inline double max_f64(double a, double b) {
  double r;
  asm("v_max_f64 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
  return r;
}

// LDS byte address of a shared-memory pointer.
__device__ inline uint32_t lds_byte(const void *p) {
  return (uint32_t)(uintptr_t)(const __attribute__((address_space(3))) void *)p;
}
// Reads of 16 / 4 bytes per lane straight into LDS: lane i's go to `lds` + 16
// i / 4 i (lds uniform).  The compiler does not know them: lds_loads_done
// waits for the wavefront's, and a barrier after it shows them to the others.
__device__ inline void lds_load16(uint32_t lds, const CCPI_GLOBAL float *p) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off"
               :: "s"(__builtin_amdgcn_readfirstlane((int)lds)), "v"(p) : "m0", "memory");
}
__device__ inline void lds_load4(uint32_t lds, const CCPI_GLOBAL float *p) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dword %1, off"
               :: "s"(__builtin_amdgcn_readfirstlane((int)lds)), "v"(p) : "m0", "memory");
}
__device__ inline void lds_loads_done() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }

// One 8-byte walk-table entry.
__device__ inline uint2 load_u2(const CCPI_GLOBAL uint2 *p) {
  uint2 v;
  __builtin_memcpy(&v, p, sizeof(v));
  return v;
}

// The detector line of ray (a, h) walked through the xy grid (p2D.cpp:
// 215-458), G cells at a time: emit(cid, l, n) receives the next n <= G
// cells (column index x * ny + y and xy length; n < G only for the last
// group) in the walk's order, so a caller can issue the group's gathers
// before it accumulates them.
template <int G, class Emit>
__device__ inline void par_walk_groups(const ParArgs &g, int a, int h, Emit &&emit) {
  const int nx = g.nx, ny = g.ny;
  const double c = gmem(g.atab)[5 * a], s = gmem(g.atab)[5 * a + 1];
  const double hp = gmem(g.h_pix)[h];
  const double p2x = c * g.D - s * hp;
  const double p2y = s * g.D + c * hp;
  int cid[G];
  float l[G];
  if (fabs(c) < kEps) {
    if (fabs(s) >= kEps) {  // line parallel to y (p2D.cpp:233-260)
      const int i = (int)floor((p2x - g.ox) / g.dx);
      if (i >= 0 && i < nx) {
        for (int j0 = 0; j0 < ny; j0 += G) {
#pragma unroll
          for (int q = 0; q < G; q++) {
            cid[q] = i * ny + (s < 0.0 ? ny - 1 - (j0 + q) : j0 + q);
            l[q] = (float)g.dy;
          }
          emit(cid, l, min(G, ny - j0));
        }
      }
    }
  } else if (fabs(s) < kEps) {  // line parallel to x (p2D.cpp:261-283)
    const int j = (int)floor((p2y - g.oy) / g.dy);
    if (j >= 0 && j < ny) {
      for (int i0 = 0; i0 < nx; i0 += G) {
#pragma unroll
        for (int q = 0; q < G; q++) {
          cid[q] = (c < 0.0 ? nx - 1 - (i0 + q) : i0 + q) * ny + j;
          l[q] = (float)g.dx;
        }
        emit(cid, l, min(G, nx - i0));
      }
    }
  } else {  // general line (p2D.cpp:284-458)
    const double ix = 1.0 / c, iy = 1.0 / s;
    const double ax0 = (g.ox - p2x) * ix, ay0 = (g.oy - p2y) * iy;
    const double axn = (g.ox + (double)nx * g.dx - p2x) * ix;
    const double ayn = (g.oy + (double)ny * g.dy - p2y) * iy;
    const double amin = fmax(fmax(fmin(ax0, axn), fmin(ay0, ayn)), -g.dconv);
    const double amax = fmin(fmin(fmax(ax0, axn), fmax(ay0, ayn)), 0.0);
    if (amin < amax - kEps) {
      const int sx = c > 0.0 ? 1 : -1, sy = s > 0.0 ? 1 : -1;
      int x, y;
      {
        const double xface = sx > 0 ? ax0 : axn, yface = sy > 0 ? ay0 : ayn;
        const int xin = sx > 0 ? 0 : nx - 1, yin = sy > 0 ? 0 : ny - 1;
        bool on_x = amin == xface, on_y = amin == yface;
        if (sx > 0 && sy < 0) {
          if (on_y) on_x = false;
        } else if (!(sx < 0 && sy < 0)) {
          if (on_x) on_y = false;
        }
        if (on_x) {
          x = xin;
          y = on_y ? yin : (int)floor((p2y + amin * s - g.oy) / g.dy);
        } else if (on_y) {
          y = yin;
          x = (int)floor((p2x + amin * c - g.ox) / g.dx);
        } else {
          x = 0;
          y = 0;
        }
        x = min(max(x, 0), nx - 1);
        y = min(max(y, 0), ny - 1);
      }
      const int bxs = sx > 0, bys = sy > 0;
      double ap = amin;
      while (x >= 0 && x < nx && y >= 0 && y < ny) {
        int n = 0;
#pragma unroll
        for (int q = 0; q < G; q++) {
          const bool in = x >= 0 && x < nx && y >= 0 && y < ny;
          cid[q] = in ? x * ny + y : 0;
          l[q] = 0.f;
          if (in) {
            const double nxa = (g.ox + (double)(x + bxs) * g.dx - p2x) * ix;
            const double nya = (g.oy + (double)(y + bys) * g.dy - p2y) * iy;
            double nap;
            if (nxa < nya - kEps) {
              nap = nxa;
              x += sx;
            } else if (nya < nxa - kEps) {
              nap = nya;
              y += sy;
            } else {
              nap = fmax(nxa, nya);
              x += sx;
              y += sy;
            }
            l[q] = (float)(nap - ap);
            ap = nap;
            n = q + 1;
          }
        }
        emit(cid, l, n);
      }
    }
  }
}

// The cells of ray r (angle a, column h), G at a time as par_walk_groups
// emits them: read from the plan's walk table when it has one (the same
// cells and lengths, written at plan time by par_walk_groups), else walked.
template <int G, class Emit>
__device__ inline void par_cells(const ParArgs &g, int r, int a, int h, Emit &&emit) {
  if (g.woff) {
    const unsigned long long e0 = gmem(g.woff)[r], e1 = gmem(g.woff)[r + 1];
    int cid[G];
    float l[G];
    for (unsigned long long e = e0; e < e1; e += G) {
      const int n = (int)min((unsigned long long)G, e1 - e);
#pragma unroll
      for (int q = 0; q < G; q++) {
        uint2 t = make_uint2(0u, 0u);
        if (q < n) t = load_u2(gmem(g.went) + e + q);
        cid[q] = (int)t.x;
        l[q] = __builtin_bit_cast(float, t.y);
      }
      emit(cid, l, n);
    }
  } else {
    par_walk_groups<G>(g, a, h, emit);
  }
}

// Cells per group of the FP: in the one-row-per-slice FP the group's column
// reads are all in flight before the accumulation.
constexpr int kParFpGroup = 8;

// x of the lane that DPP control C names, within the lane's quad or half row
// of 8 (all of them active).
template <int C>
__device__ inline float par_dpp(float x) {
  return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(x), C, 0xf, 0xf, true));
}
template <int C>
__device__ inline double par_dpp(double x) {
  const unsigned long long b = __builtin_bit_cast(unsigned long long, x);
  const unsigned lo = (unsigned)__builtin_amdgcn_mov_dpp((int)(unsigned)b, C, 0xf, 0xf, true);
  const unsigned hi =
      (unsigned)__builtin_amdgcn_mov_dpp((int)(unsigned)(b >> 32), C, 0xf, 0xf, true);
  return __builtin_bit_cast(double, (unsigned long long)hi << 32 | lo);
}
constexpr int kDppMirror8 = 0x141;                           // lane i: x of 7 - i
constexpr int kDppQuad[4] = {0x00, 0x55, 0xAA, 0xFF};        // lane i of every quad
constexpr int kDppPair[2] = {0xA0, 0xF5};                    // lane i of every pair

// acc + the products of CL adjacent lanes in lane order: x of lane 0, 1, ..
// (all CL lanes hold the same acc and get the sum; with 8, lanes 0 .. 3 do).
template <int CL, class Acc>
__device__ inline Acc par_add_lanes(Acc acc, Acc x) {
  if constexpr (CL == 1) {
    acc = acc + x;
  } else if constexpr (CL == 2) {
    acc = acc + par_dpp<kDppPair[0]>(x);
    acc = acc + par_dpp<kDppPair[1]>(x);
  } else {
    acc = acc + par_dpp<kDppQuad[0]>(x);
    acc = acc + par_dpp<kDppQuad[1]>(x);
    acc = acc + par_dpp<kDppQuad[2]>(x);
    acc = acc + par_dpp<kDppQuad[3]>(x);
    if constexpr (CL == 8) {
      const Acc y = par_dpp<kDppMirror8>(x);   // lanes 0 .. 3: x of 7 .. 4
      acc = acc + par_dpp<kDppQuad[3]>(y);
      acc = acc + par_dpp<kDppQuad[2]>(y);
      acc = acc + par_dpp<kDppQuad[1]>(y);
      acc = acc + par_dpp<kDppQuad[0]>(y);
    }
  }
  return acc;
}

// Rows v0 .. v0 + 3 of column cid, one row per slice (row v is slice v),
// nval of them inside the volume; the others read as 0.
__device__ inline float4 par_rows4(const ParArgs &g, const float *__restrict__ vol, int cid,
                                   int v0, int nval) {
  const CCPI_GLOBAL float *__restrict__ cv = gmem(vol) + (size_t)cid * g.nz + v0;
  float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
  if (nval > 3) {
    v = load_f4(cv);
  } else {
    if (nval > 0) v.x = cv[0];
    if (nval > 1) v.y = cv[1];
    if (nval > 2) v.z = cv[2];
  }
  return v;
}

// FP of detector rows v0 .. v0 + 3 of ray r from the plan's walk table (one
// row per slice).  CL lanes share the ray's cells and the four rows: lane c
// of them takes cells c, c + CL, .., 8 at a time, so 8 column reads are in
// flight per lane, and the next table entries are read while they are; the
// products are added in the walk's order (par_add_lanes), so the sums are
// those of a lane that walks alone.  The chain of table read and gather per
// 8 cells is what these small launches wait for (64 x 64 x 1, 90 angles
// 0.026 -> 0.008 ms, 128 x 128 x 7, 180 angles 0.061 -> 0.035).  Returns the sum of squares
// of the rows written (lane 0 of the CL writes).
template <int CL, class Acc>
__device__ inline double par_fp_table(const ParArgs &g, int r, int v0, int c,
                                      const float *__restrict__ vol, float *__restrict__ sino,
                                      bool acc_in) {
  static_assert(CL == 1 || CL == 2 || CL == 4 || CL == 8, "adjacent lanes of a half row");
  CCPI_GLOBAL float *__restrict__ out = gmem(sino) + (size_t)r * g.nv + v0;
  const int nrow = min(4, g.nv - v0);
  const int nval = max(0, min(nrow, g.nz - v0));
  Acc acc[4];
#pragma unroll
  for (int q = 0; q < 4; q++) acc[q] = (acc_in && q < nrow) ? (Acc)out[q] : (Acc)0;
  const unsigned long long e0 = gmem(g.woff)[r], e1 = gmem(g.woff)[r + 1];
  uint2 ent[8];
  auto fetch = [&](unsigned long long e) {
#pragma unroll
    for (int i = 0; i < 8; i++) {
      const unsigned long long q = e + i * CL + c;
      ent[i] = make_uint2(0u, 0u);
      if (q < e1) ent[i] = load_u2(gmem(g.went) + q);
    }
  };
  fetch(e0);
  for (unsigned long long e = e0; e < e1; e += 8 * CL) {
    float4 f[8];
    float l[8];
#pragma unroll
    for (int i = 0; i < 8; i++) {
      // entries past the ray's last are column 0 with length 0: their reads
      // are left out (a voxel that is not finite must not enter the sum)
      const bool in = e + i * CL + c < e1;
      l[i] = __builtin_bit_cast(float, ent[i].y);
      f[i] = par_rows4(g, vol, (int)ent[i].x, v0, in ? nval : 0);
    }
    fetch(e + 8 * CL);
#pragma unroll
    for (int i = 0; i < 8; i++) {
      acc[0] = par_add_lanes<CL, Acc>(acc[0], (Acc)(f[i].x * l[i]));
      acc[1] = par_add_lanes<CL, Acc>(acc[1], (Acc)(f[i].y * l[i]));
      acc[2] = par_add_lanes<CL, Acc>(acc[2], (Acc)(f[i].z * l[i]));
      acc[3] = par_add_lanes<CL, Acc>(acc[3], (Acc)(f[i].w * l[i]));
    }
  }
  double ss = 0.0;
  if (c == 0) {
#pragma unroll
    for (int q = 0; q < 4; q++)
      if (q < nrow) {
        const float o = (float)acc[q];
        out[q] = o;
        ss += (double)o * (double)o;
      }
  }
  return ss;
}

// FP of detector rows [v0, v0 + RC) of ray r (clipped to nv), the lane
// walking the ray itself: `acc_in` selects y += A x (reference f2D) or
// y = A x.  Returns the sum of squares of the rows written.  Acc: float row
// sums (the reference's), or double (the FP64-accumulation option; each
// float product added in double).
template <int RC, class Acc = float>
__device__ inline double par_fp_rows(const ParArgs &g, int r, int v0,
                                     const float *__restrict__ vol,
                                     float *__restrict__ sino, bool acc_in) {
  static_assert(RC % 4 == 0, "rows are read in groups of four");
  const int a = r / g.nh, h = r - a * g.nh;
  const int nz = g.nz;
  CCPI_GLOBAL float *__restrict__ out = gmem(sino) + (size_t)r * g.nv + v0;
  const int nrow = min(RC, g.nv - v0);
  Acc acc[RC];
  int kmap[RC];
#pragma unroll
  for (int q = 0; q < RC; q++) {
    acc[q] = (acc_in && q < nrow) ? (Acc)out[q] : (Acc)0;
    const int k = q < nrow ? gmem(g.map)[v0 + q] : -1;
    kmap[q] = (k >= 0 && k < nz) ? k : -1;
  }
  // one row per slice (map_type 1): the rows are the contiguous slices
  // v0 .. v0 + nval - 1 of each column, read 16 bytes at a time
  const int nval = g.map_type == 1 ? max(0, min(nrow, nz - v0)) : 0;
  if (g.map_type == 1) {
    // kParFpGroup cells at a time: all their column reads are issued before
    // the accumulation, which adds the cells in the walk's order
    constexpr int Q4 = RC / 4;
    par_walk_groups<kParFpGroup>(g, a, h, [&](const int *cid, const float *l, int n) {
      float4 f[kParFpGroup][Q4];
#pragma unroll
      for (int q = 0; q < kParFpGroup; q++)
#pragma unroll
        for (int q4 = 0; q4 < Q4; q4++)
          f[q][q4] = par_rows4(g, vol, cid[q], v0 + 4 * q4, q < n ? nval - 4 * q4 : 0);
      // cells past the group's n add 0 * l = 0
#pragma unroll
      for (int q = 0; q < kParFpGroup; q++)
#pragma unroll
        for (int q4 = 0; q4 < Q4; q4++) {
          acc[4 * q4] = acc[4 * q4] + (Acc)(f[q][q4].x * l[q]);
          acc[4 * q4 + 1] = acc[4 * q4 + 1] + (Acc)(f[q][q4].y * l[q]);
          acc[4 * q4 + 2] = acc[4 * q4 + 2] + (Acc)(f[q][q4].z * l[q]);
          acc[4 * q4 + 3] = acc[4 * q4 + 3] + (Acc)(f[q][q4].w * l[q]);
        }
    });
  } else {
    par_cells<kParFpGroup>(g, r, a, h, [&](const int *cid, const float *l, int n) {
      for (int q = 0; q < n; q++) {
        const CCPI_GLOBAL float *__restrict__ col = gmem(vol) + (size_t)cid[q] * nz;
#pragma unroll
        for (int k = 0; k < RC; k++)
          if (kmap[k] >= 0) acc[k] = acc[k] + (Acc)(col[kmap[k]] * l[q]);
      }
    });
  }
  double ss = 0.0;
#pragma unroll
  for (int q = 0; q < RC; q++)
    if (q < nrow) {
      const float o = (float)acc[q];
      out[q] = o;
      ss += (double)o * (double)o;
    }
  return ss;
}

// ---- FP, the walk shared by a wavefront --------------------------------------
//
// The rows of a ray need the same cells, so the lanes that share a ray need
// not all walk it.  A workgroup takes 64 adjacent rays of one angle: the
// lanes of its first wavefront walk a ray each, 8 cells at a time, into LDS,
// a round ahead of the others, which gather and sum the cells, lr lanes of 4
// rows per ray and NS rays per lane.  Cells are par_walk_groups' (the same
// steps and lengths), added in the walk's order.
//
// Bound: the gathers' 64 bytes per cycle and CU from L1 (512 x 512 x 32, 360
// angles: TD 84 % busy, TA 78, VALU issue up to 65 % of the cycles).  With every lane walking, 8 lanes
// repeated each ray's double arithmetic (35 instructions per cell against 10
// to gather and sum it): 512 x 512 x 32 1.51 -> 0.67 ms, 383 x 383 x 29 (180
// angles) 0.52 -> 0.23, 256 x 256 x 16 (180) 0.135 -> 0.080.  A wavefront that
// walks for itself only (16 or 32 of its lanes) took 0.77, 0.29 and 0.121.

// Walk of one ray, a step at a time (par_walk_groups' arithmetic).
struct ParWalker {
  double p2x, p2y, ix, iy, ap;
  int x, y, sx, sy;    // cell and step; an axis-parallel line steps one axis
  float l;             // its constant length, or < 0 for a general line
  bool on;

  __device__ inline void start(const ParArgs &g, int a, int h) {
    const int nx = g.nx, ny = g.ny;
    const double c = gmem(g.atab)[5 * a], s = gmem(g.atab)[5 * a + 1];
    const double hp = gmem(g.h_pix)[h];
    p2x = c * g.D - s * hp;
    p2y = s * g.D + c * hp;
    ix = 1.0 / c;
    iy = 1.0 / s;
    ap = 0.0;
    on = false;
    l = -1.0f;
    x = y = sx = sy = 0;
    if (fabs(c) < kEps) {
      if (fabs(s) >= kEps) {  // line parallel to y (p2D.cpp:233-260)
        x = (int)floor((p2x - g.ox) / g.dx);
        y = s < 0.0 ? ny - 1 : 0;
        sy = s < 0.0 ? -1 : 1;
        l = (float)g.dy;
        on = x >= 0 && x < nx;
      }
    } else if (fabs(s) < kEps) {  // line parallel to x (p2D.cpp:261-283)
      y = (int)floor((p2y - g.oy) / g.dy);
      x = c < 0.0 ? nx - 1 : 0;
      sx = c < 0.0 ? -1 : 1;
      l = (float)g.dx;
      on = y >= 0 && y < ny;
    } else {  // general line (p2D.cpp:284-458)
      const double ax0 = (g.ox - p2x) * ix, ay0 = (g.oy - p2y) * iy;
      const double axn = (g.ox + (double)nx * g.dx - p2x) * ix;
      const double ayn = (g.oy + (double)ny * g.dy - p2y) * iy;
      const double amin = fmax(fmax(fmin(ax0, axn), fmin(ay0, ayn)), -g.dconv);
      const double amax = fmin(fmin(fmax(ax0, axn), fmax(ay0, ayn)), 0.0);
      if (amin < amax - kEps) {
        sx = c > 0.0 ? 1 : -1;
        sy = s > 0.0 ? 1 : -1;
        const double xface = sx > 0 ? ax0 : axn, yface = sy > 0 ? ay0 : ayn;
        const int xin = sx > 0 ? 0 : nx - 1, yin = sy > 0 ? 0 : ny - 1;
        bool on_x = amin == xface, on_y = amin == yface;
        if (sx > 0 && sy < 0) {
          if (on_y) on_x = false;
        } else if (!(sx < 0 && sy < 0)) {
          if (on_x) on_y = false;
        }
        if (on_x) {
          x = xin;
          y = on_y ? yin : (int)floor((p2y + amin * s - g.oy) / g.dy);
        } else if (on_y) {
          y = yin;
          x = (int)floor((p2x + amin * c - g.ox) / g.dx);
        }
        x = min(max(x, 0), nx - 1);
        y = min(max(y, 0), ny - 1);
        ap = amin;
        on = true;
      }
    }
  }
  // The next cell: its column index and length, or a column of -1 past the
  // walk's end.
  __device__ inline int step(const ParArgs &g, float &len) {
    on = on && (unsigned)x < (unsigned)g.nx && (unsigned)y < (unsigned)g.ny;
    len = 0.0f;
    if (!on) return -1;
    const int cid = x * g.ny + y;
    if (l >= 0.0f) {
      len = l;
      x += sx;
      y += sy;
      return cid;
    }
    const double nxa = (g.ox + (double)(x + (sx > 0 ? 1 : 0)) * g.dx - p2x) * ix;
    const double nya = (g.oy + (double)(y + (sy > 0 ? 1 : 0)) * g.dy - p2y) * iy;
    const bool go_x = nxa < nya - kEps, go_y = nya < nxa - kEps;
    const double nap = go_x ? nxa : (go_y ? nya : fmax(nxa, nya));
    x += go_y ? 0 : sx;
    y += go_x ? 0 : sy;
    len = (float)(nap - ap);
    ap = nap;
    return cid;
  }
};

inline bool par_share_fits(const ParArgs &g) {
  return g.map_type == 1 && sizeof(float) * (size_t)g.nx * g.ny * g.nz <= kParShareBytes;
}
// Waves per SIMD that the gathering wavefronts' registers allow (72 VGPRs).
constexpr int kParShareWavesPerSimd = 7;

// Adjacent angles that one XCD's consecutive workgroups take (16 / 32 / 64:
// 512 x 512 x 32, 360 angles 0.739 / 0.720 / 0.720 ms, 383 x 383 x 29, 180
// angles 0.263 / 0.262 / 0.276).
constexpr int kParTileA = 32;

// Workgroup `id` -> its rays and rows: ids go to the 8 XCDs in turn, each
// XCD's in tiles of kParTileA angles of the same 64 columns (par_tile_column);
// row blocks slowest.  index: the workgroup's place among the live ones (ids past the
// last tile are not live).
struct ParShareItem {
  int a, h0, v0;
  bool live;
  size_t index;
};
__host__ __device__ inline long long par_share_items(const ParArgs &g, int lr) {
  const long long nb = (g.nh + 63) / 64, nta = (g.na + kParTileA - 1) / kParTileA;
  const long long tiles = (long long)((g.nv + 4 * lr - 1) / (4 * lr)) * nta * nb;
  return (tiles + 7) / 8 * 8 * kParTileA;
}
__host__ __device__ inline size_t par_share_parts(const ParArgs &g, int lr) {
  return (size_t)((g.nv + 4 * lr - 1) / (4 * lr)) * g.na * ((g.nh + 63) / 64);
}
__device__ inline ParShareItem par_share_item(const ParArgs &g, int lr, int id) {
  const int nb = (g.nh + 63) / 64, nta = (g.na + kParTileA - 1) / kParTileA;
  const int local = id >> 3;
  const int tile = (local / kParTileA) * 8 + (id & 7);
  const int rb = tile / (nb * nta), tab = tile - rb * (nb * nta);
  ParShareItem it;
  // uniform: the rays' and rows' addresses stay in scalar registers
  const int ta = tab / nb, c = par_tile_column(nb, ta, tab % nb);
  it.a = __builtin_amdgcn_readfirstlane(ta * kParTileA + local % kParTileA);
  it.h0 = __builtin_amdgcn_readfirstlane(c * 64);
  it.v0 = __builtin_amdgcn_readfirstlane(rb * 4 * lr);
  it.live = it.a < g.na && it.v0 < g.nv;
  it.index = ((size_t)rb * g.na + it.a) * nb + c;
  return it;
}

// LDS of a workgroup of par_fp_shared: two rounds of 8 cells of 64 rays.
struct ParShare {
  uint2 ent[2][8][64];   // byte offset of the cell's column, float bits of its length
  int more[2];           // the round holds cells
};

// Rows [v0, v0 + 4 lr) of rays h0 .. h0 + 63 of angle a, by a workgroup of
// 1 + lr / NS wavefronts or more.  One row per slice, volumes below kParShareBytes
// (32-bit byte offsets; the reads past the volume that a walk's end asks for
// return 0).  VEC: nz >= 4, a lane's 4 slices in one 16-byte read that ends
// inside the column; otherwise single reads.  Every thread of the workgroup
// calls it (it synchronises).  Returns the thread's sum of squares of the
// rows it wrote.
template <int NS, bool VEC, class Acc>
__device__ inline double par_fp_shared(const ParArgs &g, int a, int h0, int v0, int lr,
                                       const float *__restrict__ vol,
                                       float *__restrict__ sino, bool acc_in, ParShare &sh) {
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const uint32_t bytes = 4u * (uint32_t)g.nz;
  if (wave == 0) {
    ParWalker W;
    W.on = false;
    if (h0 + lane < g.nh) W.start(g, a, h0 + lane);
    for (int buf = 0;; buf ^= 1) {
      bool more = false;
#pragma unroll
      for (int q = 0; q < 8; q++) {
        float len;
        const int cid = W.step(g, len);
        more |= cid >= 0;
        // an ended walk's cells read past the volume (0) with length 0
        sh.ent[buf][q][lane] =
            make_uint2(cid >= 0 ? bytes * (uint32_t)cid : 0xf0000000u, __float_as_uint(len));
      }
      const bool any = __ballot(more) != 0;
      if (lane == 0) sh.more[buf] = any ? 1 : 0;
      __syncthreads();
      if (!any) break;
    }
    return 0.0;
  }
  const int per = 64 / lr;              // rays of one wavefront at a time
  const int ray0 = (wave - 1) * NS * per;
  if (ray0 >= 64) {
    // a wavefront more than the rays need: only the barriers
    for (int buf = 0;; buf ^= 1) {
      __syncthreads();
      if (!__builtin_amdgcn_readfirstlane(sh.more[buf])) return 0.0;
    }
  }
  const int rl = lane & (lr - 1), rr = lane / lr;
  const int v = v0 + 4 * rl;            // the lane's first row
  const int nrow = max(0, min(4, g.nv - v)), nval = max(0, min(nrow, g.nz - v));
  // its slices vs .. vs + 3 all exist (VEC); rows v .. take those from `off` on
  const int vs = VEC ? min(v, g.nz - 4) : v;
  const int off = v - vs;
  const uint32_t voff = 4u * (uint32_t)vs;
  const __amdgpu_buffer_rsrc_t rv = __builtin_amdgcn_make_buffer_rsrc(
      (void *)vol, (short)0, (int)(bytes * (uint32_t)(g.nx * g.ny)), 0x00020000);
  // acc[s][q + off] is row v + q of the s-th ray
  Acc acc[NS][4];
#pragma unroll
  for (int s = 0; s < NS; s++) {
    const int h = h0 + ray0 + s * per + rr;
    const CCPI_GLOBAL float *in = gmem(sino) + ((size_t)a * g.nh + h) * g.nv + v;
#pragma unroll
    for (int k = 0; k < 4; k++)
      acc[s][k] = (acc_in && h < g.nh && k >= off && k - off < nrow) ? (Acc)in[k - off] : (Acc)0;
  }
  for (int buf = 0;; buf ^= 1) {
    __syncthreads();
    if (!__builtin_amdgcn_readfirstlane(sh.more[buf])) break;
#pragma unroll
    for (int s = 0; s < NS; s++) {
      float f[8][4], l[8];
#pragma unroll
      for (int q = 0; q < 8; q++) {
        const uint2 e = sh.ent[buf][q][ray0 + s * per + rr];
        l[q] = __uint_as_float(e.y);
        const int at = (int)(e.x + voff);
        if constexpr (VEC) {
          typedef unsigned u4 __attribute__((ext_vector_type(4)));
          const u4 t = __builtin_amdgcn_raw_buffer_load_b128(rv, at, 0, 0);
#pragma unroll
          for (int k = 0; k < 4; k++) f[q][k] = __uint_as_float(t[k]);
        } else {
#pragma unroll
          for (int k = 0; k < 4; k++)
            f[q][k] = k < 3 ? __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(
                                  rv, k < nval ? at + 4 * k : (int)0xf0000000u, 0, 0))
                            : 0.0f;
        }
      }
#pragma unroll
      for (int q = 0; q < 8; q++)
#pragma unroll
        for (int k = 0; k < 4; k++) acc[s][k] = acc[s][k] + (Acc)(f[q][k] * l[q]);
    }
  }
  double ss = 0.0;
#pragma unroll
  for (int s = 0; s < NS; s++) {
    const int h = h0 + ray0 + s * per + rr;
    if (h < g.nh) {
      CCPI_GLOBAL float *out = gmem(sino) + ((size_t)a * g.nh + h) * g.nv + v;
#pragma unroll
      for (int q = 0; q < 4; q++)
        if (q < nrow) {
          // a row without a slice keeps what it holds
          float o = (acc_in && q >= nval) ? out[q] : 0.0f;
#pragma unroll
          for (int k = 0; k < 4; k++)
            if (q + off == k && q < nval) o = (float)acc[s][k];
          out[q] = o;
          ss += (double)o * (double)o;
        }
    }
  }
  return ss;
}

// FP, ray-shared layout: `lr` lanes (a power of two, at most 16) share one
// ray, each taking 4 consecutive detector rows, so the lanes of a ray read
// one contiguous run of every crossed column.  Block bx holds rays
// [bx * 256 / lr, ...), row block by the rows [by * 4 lr, (by + 1) * 4 lr).
template <class Acc = float>
__device__ inline double par_fp_lanes(const ParArgs &g, int bx, int by, int tid, int lr,
                                      const float *__restrict__ vol,
                                      float *__restrict__ sino, bool acc_in) {
  const int r = bx * (256 / lr) + tid / lr;
  if (r >= g.na * g.nh) return 0.0;
  const int v0 = (by * lr + (tid & (lr - 1))) * 4;
  if (v0 >= g.nv) return 0.0;
  return par_fp_rows<4, Acc>(g, r, v0, vol, sino, acc_in);
}

// Footprint of the voxel column [x0, xn] x [y0, yn] on the detector at the
// angle whose table row is t (p2D.cpp:808-915): detector columns [lo, hi],
// kind 0 (general: trapezoid over [ymin, ymax]), 1 or 2 (axis-aligned:
// columns whose +-h lies in [lim0, lim1)).
struct ParFoot {
  int lo, hi, kind;
  double ymin, ymax, lim0, lim1;
};

template <class TabPtr>
__device__ inline ParFoot par_footprint(const ParArgs &g, TabPtr t, double x0, double xn,
                                        double y0, double yn) {
  const double c = t[0], s = t[1];
  ParFoot f;
  f.ymin = f.ymax = f.lim0 = f.lim1 = 0.0;
  if (fabs(c) < kEps) {  // p2D.cpp:808-844
    f.kind = s < 0.0 ? 1 : 2;
    f.lim0 = x0;
    f.lim1 = xn;
    if (s < 0.0) {
      f.lo = (int)floor(x0 * g.ihp - g.hp0);
      f.hi = (int)floor((xn - kEps) * g.ihp - g.hp0);
    } else {
      f.lo = (int)ceil((-xn + kEps) * g.ihp - g.hp0);
      f.hi = (int)ceil(-x0 * g.ihp - g.hp0);
    }
    f.lo = max(f.lo, 0);
    f.hi = min(f.hi, g.nh - 1);
  } else if (fabs(s) < kEps) {  // p2D.cpp:845-880
    f.kind = c < 0.0 ? 2 : 1;
    f.lim0 = y0;
    f.lim1 = yn;
    if (c < 0.0) {
      f.lo = (int)ceil((-yn + kEps) * g.ihp - g.hp0);
      f.hi = (int)ceil(-y0 * g.ihp - g.hp0);
    } else {
      f.lo = (int)floor(y0 * g.ihp - g.hp0);
      f.hi = (int)floor((yn - kEps) * g.ihp - g.hp0);
    }
    f.lo = max(f.lo, 0);
    f.hi = min(f.hi, g.nh - 1);
  } else {  // p2D.cpp:881-915
    f.kind = 0;
    if (c > 0.0) {
      if (s > 0.0) { f.ymin = y0 * c - xn * s; f.ymax = yn * c - x0 * s; }
      else         { f.ymin = y0 * c - x0 * s; f.ymax = yn * c - xn * s; }
    } else {
      if (s > 0.0) { f.ymin = yn * c - xn * s; f.ymax = y0 * c - x0 * s; }
      else         { f.ymin = yn * c - x0 * s; f.ymax = y0 * c - xn * s; }
    }
    // clamp at 0: the floor can round to -1 when ymin ~ h_pix[0]
    f.lo = f.ymin < cmem(g.h_pix)[0] ? 0 : max((int)floor(f.ymin * g.ihp - g.hp0), 0);
    f.hi = min((int)floor(f.ymax * g.ihp - g.hp0), g.nh - 1);
  }
  return f;
}

// Weight of detector column position hp in footprint f (p2D.cpp:916-938):
// 1 with w set, 0 to skip the column, -1 past the footprint's far edge.
template <class TabPtr>
__device__ inline int par_weight(const ParArgs &g, TabPtr t, const ParFoot &f, double hp,
                                 double &w) {
  if (f.kind != 0) {
    const double tt = f.kind == 1 ? hp : -hp;
    if (!(tt >= f.lim0 && tt < f.lim1)) return 0;
    w = fabs(t[0]) < kEps ? g.dy : g.dx;
    return 1;
  }
  const double ybot = f.ymin + t[2], ytop = f.ymax - t[2], l = t[4];
  if (!(hp > f.ymin + kEps)) return 0;
  if (hp < ybot)
    w = l * (hp - f.ymin) * t[3];
  else if (hp <= ytop)
    w = l;
  else if (hp < f.ymax - kEps)
    w = l * (f.ymax - hp) * t[3];
  else
    return -1;
  return 1;
}

// One thread of the BP: column bx * 256 + tid, slices [by * RC, by * RC +
// RC).  `acc_in` selects x += A^T y (reference b2D) or x = A^T y.  Returns
// the sum of squares of the slices written.
template <int RC, class Acc = float>
__device__ inline double par_bp_thread(const ParArgs &g, int bx, int by, int tid,
                                       const float *__restrict__ sino,
                                       float *__restrict__ vol, bool acc_in) {
  static_assert(RC % 4 == 0, "rows are read in groups of four");
  const int colid = bx * 256 + tid;
  if (colid >= g.nx * g.ny) return 0.0;
  const int i = colid / g.ny, j = colid - (colid / g.ny) * g.ny;
  const int k0 = by * RC;
  const int nz = g.nz, nv = g.nv, nh = g.nh;
  const int nk = min(RC, nz - k0);
  CCPI_GLOBAL float *__restrict__ vcol = gmem(vol) + (size_t)colid * nz + k0;
  Acc acc[RC];
#pragma unroll
  for (int q = 0; q < RC; q++) acc[q] = (acc_in && q < nk) ? (Acc)vcol[q] : (Acc)0;
  const double x0 = g.ox + (double)i * g.dx, xn = g.ox + (double)(i + 1) * g.dx;
  const double y0 = g.oy + (double)j * g.dy, yn = g.oy + (double)(j + 1) * g.dy;
  const int T = g.map_type;
  const int nvalid = max(0, min(nk, nv - k0));  // rows of the slices (T == 1)

  for (int a = 0; a < g.na; a++) {
    const CCPI_GLOBAL double *t = gmem(g.atab) + 5 * a;
    const double c = t[0], s = t[1];
    int lo, hi, kind;
    double ymin = 0, ymax = 0, lim0 = 0, lim1 = 0;
    if (fabs(c) < kEps) {  // p2D.cpp:808-844
      kind = s < 0.0 ? 1 : 2;
      lim0 = x0;
      lim1 = xn;
      if (s < 0.0) {
        lo = (int)floor(x0 * g.ihp - g.hp0);
        hi = (int)floor((xn - kEps) * g.ihp - g.hp0);
      } else {
        lo = (int)ceil((-xn + kEps) * g.ihp - g.hp0);
        hi = (int)ceil(-x0 * g.ihp - g.hp0);
      }
      lo = max(lo, 0);
      hi = min(hi, nh - 1);
    } else if (fabs(s) < kEps) {  // p2D.cpp:845-880
      kind = c < 0.0 ? 2 : 1;
      lim0 = y0;
      lim1 = yn;
      if (c < 0.0) {
        lo = (int)ceil((-yn + kEps) * g.ihp - g.hp0);
        hi = (int)ceil(-y0 * g.ihp - g.hp0);
      } else {
        lo = (int)floor(y0 * g.ihp - g.hp0);
        hi = (int)floor((yn - kEps) * g.ihp - g.hp0);
      }
      lo = max(lo, 0);
      hi = min(hi, nh - 1);
    } else {  // p2D.cpp:881-915
      kind = 0;
      if (c > 0.0) {
        if (s > 0.0) { ymin = y0 * c - xn * s; ymax = yn * c - x0 * s; }
        else         { ymin = y0 * c - x0 * s; ymax = yn * c - xn * s; }
      } else {
        if (s > 0.0) { ymin = yn * c - xn * s; ymax = y0 * c - x0 * s; }
        else         { ymin = yn * c - x0 * s; ymax = y0 * c - xn * s; }
      }
      // clamp at 0: the floor can round to -1 when ymin ~ h_pix[0]
      lo = ymin < gmem(g.h_pix)[0] ? 0 : max((int)floor(ymin * g.ihp - g.hp0), 0);
      hi = min((int)floor(ymax * g.ihp - g.hp0), nh - 1);
    }
    for (int h = lo; h <= hi; h++) {
      const double hp = gmem(g.h_pix)[h];
      double w;
      if (kind != 0) {
        const double tt = kind == 1 ? hp : -hp;
        if (!(tt >= lim0 && tt < lim1)) continue;
        w = fabs(c) < kEps ? g.dy : g.dx;
      } else {  // trapezoid (p2D.cpp:916-938)
        const double ybot = ymin + t[2], ytop = ymax - t[2], l = t[4];
        if (!(hp > ymin + kEps)) continue;
        if (hp < ybot)
          w = l * (hp - ymin) * t[3];
        else if (hp <= ytop)
          w = l;
        else if (hp < ymax - kEps)
          w = l * (ymax - hp) * t[3];
        else
          break;
      }
      const float wf = (float)w;
      const CCPI_GLOBAL float *__restrict__ p = gmem(sino) + ((size_t)a * nh + h) * nv;
      if (T == 1) {
        // rows k0 .. k0 + nvalid - 1 of the ray, read 16 bytes at a time
        const CCPI_GLOBAL float *__restrict__ pr = p + k0;
#pragma unroll
        for (int q4 = 0; q4 < RC / 4; q4++) {
          if (4 * q4 + 3 < nvalid) {
            const float4 f = load_f4(pr + 4 * q4);
            acc[4 * q4] = acc[4 * q4] + (Acc)(f.x * wf);
            acc[4 * q4 + 1] = acc[4 * q4 + 1] + (Acc)(f.y * wf);
            acc[4 * q4 + 2] = acc[4 * q4 + 2] + (Acc)(f.z * wf);
            acc[4 * q4 + 3] = acc[4 * q4 + 3] + (Acc)(f.w * wf);
          } else {
#pragma unroll
            for (int q = 4 * q4; q < 4 * q4 + 4; q++)
              if (q < nvalid) acc[q] = acc[q] + (Acc)(pr[q] * wf);
          }
        }
      } else if (T == 2 || T == 4) {  // rows summed before scaling (p2D.cpp:694-761)
#pragma unroll
        for (int q = 0; q < RC; q++) {
          const int k = k0 + q;
          if (q < nk && (k + 1) * T <= nv) {
            float sum = p[k * T];
            for (int u = 1; u < T; u++) sum = sum + p[k * T + u];
            acc[q] = acc[q] + (Acc)(sum * wf);
          }
        }
      } else {
#pragma unroll
        for (int q = 0; q < RC; q++) {
          if (q < nk) {
            const int k = k0 + q;
            const int vlo = gmem(g.rlo)[k], vhi = gmem(g.rhi)[k];
            for (int v = vlo; v < vhi; v++) acc[q] = acc[q] + (Acc)(p[v] * wf);
          }
        }
      }
    }
  }
  double ss = 0.0;
#pragma unroll
  for (int q = 0; q < RC; q++)
    if (q < nk) {
      const float o = (float)acc[q];
      vcol[q] = o;
      ss += (double)o * (double)o;
    }
  return ss;
}

// Tiled BP (one row per slice): a workgroup owns a 16 x 16 tile of voxel
// columns, one column per lane and R consecutive slices per lane.  Angles go
// in blocks of `ab`: for each angle of the block, the detector columns that
// the tile's square can reach (its corners' span plus a margin of 2) are
// staged in LDS with the R rows of the lane's slices (hmax columns at most),
// one coalesced copy per tile instead of each lane re-reading its columns'
// rows, and with the columns' positions; every lane then weighs its own
// column's footprint (the reference's FP64 arithmetic) on the staged rows.
// Bound by vector issue (at 512 x 512 x 32 up to 89 % of the cycles, LDS 63 %,
// half of it bank conflicts), 123 instructions per wavefront and angle of which
// 64 are the 16 slices' products and sums.  So there are two blocks of LDS and the next one's reads go
// straight there while this one is summed (one barrier a block, no register
// in between), spans are found 256 angles at a time, tables are scalar loads,
// and where a voxel's shadow is under two columns wide (pixels about as wide
// as a voxel or wider) two columns are weighed without a loop, a last column
// or tests that even columns answer.  With the rows staged through registers
// between two barriers and a loop over positions in global memory it took:
// 512 x 512 x 32, 360 angles 1.40 ms, now 0.66; 383 x 383 x 29, 180 angles
// 0.43, now 0.23; 256 x 256 x 16, 180 angles 0.116, now 0.061; 64 x 64 x 1, 90
// angles 0.027, now 0.019; with the staging alone 0.89, 0.31, 0.081 and
// 0.021.  Of few angles the sums are the least part: there the set-up, whose
// code each launch fetches anew, and the writes count, so an accumulating
// call's reads are behind one test, and four slices that all have a row are
// written at once.  Slice by slice, each under its own tests, 55 x 358 x 59, 11
// angles took 0.060 ms (0.043 before there was a two-column form), now 0.025;
// 200 x 200 x 64, 20 angles 0.075, now 0.035; 256 x 256 x 16, 180 angles 0.067,
// now 0.061.  Angles are visited in order, so with
// one angle group the result is bit-identical to par_bp_kernel; with G
// groups (blockIdx.z) each group writes its partial sums of its angle range
// to part[group] and par_bp_sum_kernel adds them in group order.
//
// One tile item of the tiled BP, run by all 256 threads of a workgroup
// (it synchronises the workgroup): tile `tile` (16 x 16 columns, row-major
// over the column grid), slices [zc * R, zc * R + R), angles [a_begin,
// a_end).  The result goes to `dst` (a volume-layout array), added to its
// contents when acc_in.  norm: returns the thread's sum of squares of the
// values it wrote (0 for threads outside the volume).  smem: par_bp_tile_bytes,
// 16-byte aligned; a caller with another item to do synchronises first.
// FOLD (the batched kernel's tiled items; acc_in must be false): the
// angles are split into `groups` ranges as par_bp_lds_kernel splits them,
// each summed from zero, and the running sum of the groups is kept in
// `dst` (each lane re-reads only its own writes), so one item gives bit for
// bit what the grouped launch and par_bp_sum_kernel give into a zeroed
// volume, without registers for a second set of sums.
constexpr int kParBpSpans = 256;   // one per thread
constexpr int kParBpNarrow = 1 << 30;
template <int R, class Acc, bool FOLD = false>
__device__ double par_bp_tile(const ParArgs &g, int tile, int zc, int a_begin, int a_end,
                              int hmax, int ab, bool acc_in, const float *__restrict__ sino,
                              float *__restrict__ dst_vol, float *smem, bool norm,
                              int groups = 1) {
  static_assert(R % 4 == 0, "rows are read 4 at a time");
  constexpr int Q4 = R / 4;
  // two buffers of a block's rows, column positions and spans
  float *s_rows = smem;                                                        // [2][ab][hmax][R]
  double *s_hp = reinterpret_cast<double *>(smem + 2 * (size_t)ab * hmax * R);   // [2][ab][hmax]
  int2 *s_cur = reinterpret_cast<int2 *>(s_hp + 2 * (size_t)ab * hmax);          // [2][ab]
  int2 *s_span = s_cur + 2 * ab;                                               // [kParBpSpans]
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int ntj = (g.ny + 15) >> 4;
  const int ti0 = (tile / ntj) * 16, tj0 = (tile % ntj) * 16;
  const int i = ti0 + (tid >> 4), j = tj0 + (tid & 15);
  const bool active = i < g.nx && j < g.ny;
  const int k0 = zc * R;
  const int nz = g.nz, nv = g.nv, nh = g.nh;
  const int nk = min(R, nz - k0);
  const size_t colid = (size_t)(active ? i : 0) * g.ny + (active ? j : 0);
  Acc acc[R];
  CCPI_GLOBAL float *__restrict__ vcol = gmem(dst_vol) + colid * nz + k0;
#pragma unroll
  for (int q = 0; q < R; q++) acc[q] = (Acc)0;
  if (!FOLD && acc_in && active) {
#pragma unroll
    for (int q = 0; q < R; q++)
      if (q < nk) acc[q] = (Acc)vcol[q];
  }
  const double x0 = g.ox + (double)i * g.dx, xn = g.ox + (double)(i + 1) * g.dx;
  const double y0 = g.oy + (double)j * g.dy, yn = g.oy + (double)(j + 1) * g.dy;
  // rows of the lane's slices that exist (one row per slice)
  const int nrow = max(0, min(R, min(nv, nz) - k0));

  // Detector columns that the tile's square can reach at angles sb ..
  // sb + kParBpSpans - 1: its corners' span and 2 columns on each side (the
  // footprints' own rounding), one angle per thread.  Every column of the
  // tile projects inside its square, and the index floor(y * ihp - hp0) grows
  // with y, so the footprints stay inside the span.
  auto spans = [&](int sb) {
    const int a = sb + tid;
    if (a >= a_end) return;
    const double X0 = g.ox + (double)ti0 * g.dx, XN = g.ox + (double)min(ti0 + 16, g.nx) * g.dx;
    const double Y0 = g.oy + (double)tj0 * g.dy, YN = g.oy + (double)min(tj0 + 16, g.ny) * g.dy;
    const CCPI_GLOBAL double *tab = gmem(g.atab) + 5 * a;
    const double c = tab[0], s = tab[1];
    const double p0 = Y0 * c - X0 * s, p1 = YN * c - X0 * s;
    const double p2 = Y0 * c - XN * s, p3 = YN * c - XN * s;
    const double tmin = fmin(fmin(p0, p1), fmin(p2, p3));
    const double tmax = fmax(fmax(p0, p1), fmax(p2, p3));
    const int lo = max((int)floor(tmin * g.ihp - g.hp0) - 2, 0);
    const int hi = min((int)floor(tmax * g.ihp - g.hp0) + 2, nh - 1);
    // a voxel's shadow under two columns wide, on even columns and a general
    // line: see the two-column form below
    const bool narrow = g.h_even != 0 && !(fabs(c) < kEps || fabs(s) < kEps) &&
                        (fabs(c) * g.dy + fabs(s) * g.dx) * g.ihp < 1.99;
    s_span[tid] =
        make_int2(lo, max(0, min(hi - lo + 1, hmax)) | (narrow ? kParBpNarrow : 0));
  };
  // Starts the reads of angles [a0, a0 + n) into buffer `buf`: per wavefront
  // one angle at a time, straight into LDS.  Rows of 16-byte aligned start go
  // 16 bytes at a time, others one float at a time.  Rows past nrow are not
  // read or not added in the end.
  const bool aligned = ((nv & 3) | (int)((uintptr_t)sino & 15)) == 0;
  const int have = nv - k0;             // rows of a ray from the first slice on
  auto start = [&](int a0, int n, int buf, int sb) {
    for (int t = wave; t < n; t += 4) {
      const int2 sp = s_span[a0 + t - sb];
      const int lo = __builtin_amdgcn_readfirstlane(sp.x);
      const int cnt = __builtin_amdgcn_readfirstlane(sp.y) & ~kParBpNarrow;
      const int slot = buf * ab + t;
      if (lane == 0) s_cur[slot] = sp;
      const uint32_t row_lds = lds_byte(s_rows + (size_t)slot * hmax * R);
      const CCPI_GLOBAL float *p = gmem(sino) + ((size_t)(a0 + t) * nh + lo) * nv + k0;
      if (aligned) {
        for (int hh = 0; hh < cnt; hh += 64 / Q4) {
          const int r = hh + lane / Q4, q = 4 * (lane % Q4);
          if (r < cnt && q < have) lds_load16(row_lds + hh * (4 * R), p + (size_t)r * nv + q);
        }
      } else {
        for (int hh = 0; hh < cnt; hh += 64 / R) {
          const int r = hh + lane / R, q = lane % R;
          if (r < cnt && q < have) lds_load4(row_lds + hh * (4 * R), p + (size_t)r * nv + q);
        }
      }
      const uint32_t hp_lds = lds_byte(s_hp + (size_t)slot * hmax);
      const CCPI_GLOBAL float *hp = (const CCPI_GLOBAL float *)(gmem(g.h_pix) + lo);
      for (int e = 0; e < 2 * cnt; e += 64)
        if (e + lane < 2 * cnt) lds_load4(hp_lds + 4 * e, hp + e + lane);
    }
  };
  // angle range of group `grp` (one group: all)
  const int ngrp = FOLD ? groups : 1;
  auto group_begin = [&](int grp) {
    return FOLD ? a_begin + (int)((long long)(a_end - a_begin) * grp / groups) : a_begin;
  };
  int grp = 0, a0 = a_begin, gb = FOLD ? group_begin(1) : a_end, buf = 0;
  int sb = a0;
  spans(sb);
  __syncthreads();
  start(a0, min(ab, gb - a0), 0, sb);
  for (;;) {
    const int nblk = min(ab, gb - a0);
    const bool group_ends = a0 + ab >= gb;
    const int next = group_ends ? gb : a0 + ab;
    const int next_gb = group_ends && grp + 1 < ngrp ? group_begin(grp + 2) : gb;
    // the block's reads have landed, and everybody is done with the other buffer
    lds_loads_done();
    __syncthreads();
    if (next < next_gb) {
      if (next + ab > sb + kParBpSpans) {
        sb = next;
        spans(sb);
        __syncthreads();
      }
      start(next, min(ab, next_gb - next), buf ^ 1, sb);
    }
    if (active) {
      int2 cur = s_cur[buf * ab];
      for (int t = 0; t < nblk; t++) {
        const CCPI_CONST double *tab = cmem(g.atab) + 5 * (a0 + t);
        const double c = tab[0], s = tab[1], t2 = tab[2], t3 = tab[3], l = tab[4];
        const int slot = buf * ab + t;
        const int slo = __builtin_amdgcn_readfirstlane(cur.x);
        const int sy = __builtin_amdgcn_readfirstlane(cur.y);
        cur = s_cur[slot + 1];   // the next angle's (the last one's is not used)
        const int scnt = sy & ~kParBpNarrow;
        const float *rows_t = s_rows + (size_t)slot * hmax * R;
        const double *hp_t = s_hp + (size_t)slot * hmax;
        auto add = [&](const float *pr, float wf) {
#pragma unroll
          for (int q4 = 0; q4 < Q4; q4++) {
            const float4 v = *reinterpret_cast<const float4 *>(pr + 4 * q4);
            acc[4 * q4] = acc[4 * q4] + (Acc)(v.x * wf);
            acc[4 * q4 + 1] = acc[4 * q4 + 1] + (Acc)(v.y * wf);
            acc[4 * q4 + 2] = acc[4 * q4 + 2] + (Acc)(v.z * wf);
            acc[4 * q4 + 3] = acc[4 * q4 + 3] + (Acc)(v.w * wf);
          }
        };
        // The two-column form: par_footprint's and par_weight's values
        // (p2D.cpp:881-938) for the columns lo + 1 and lo + 2, lo the one at
        // or before ymin.  On even columns lo itself is not hit, a shadow
        // under two columns wide ends before lo + 3, and the columns past it
        // fail the weight's own limits, so neither a last column nor a loop
        // is needed.  The signs of c and s choose which of the products is
        // which: their minimum and maximum.
        bool two = false, use1 = false, use2 = false;
        float w1 = 0.0f, w2 = 0.0f;
        const float *pr = rows_t;
        if (sy & kParBpNarrow) {
          const double yc0 = y0 * c, yc1 = yn * c, xs0 = x0 * s, xs1 = xn * s;
          const double ymin = min_f64(yc0, yc1) - max_f64(xs0, xs1);
          const int hh = (int)floor(ymin * g.ihp - g.hp0) - slo;
          // both staged; a footprint from before the first column goes below
          two = __builtin_amdgcn_ballot_w64((unsigned)hh >= (unsigned)max(scnt - 2, 0)) == 0;
          if (two) {
            const double ymax = max_f64(yc0, yc1) - min_f64(xs0, xs1);
            const double e0 = ymin + kEps, ybot = ymin + t2, ytop = ymax - t2;
            const double e1 = max_f64(ymax - kEps, ytop);
            const float lf = (float)l;
            auto weigh = [&](double hp, bool &use, float &w) {
              const double d = min_f64(hp - ymin, ymax - hp);
              w = hp >= ybot && hp <= ytop ? lf : (float)(l * d * t3);
              use = hp > e0 && hp < e1;
            };
            weigh(hp_t[hh + 1], use1, w1);
            weigh(hp_t[hh + 2], use2, w2);
            pr = rows_t + (hh + 1) * R;
          }
        }
        if (!two) {
          const ParFoot f = par_footprint(g, tab, x0, xn, y0, yn);
          for (int h = f.lo; h <= f.hi; h++) {
            // inside the staged span (see above); the clamp keeps the reads there
            const int hh = max(min(h - slo, scnt - 1), 0);
            double w;
            const int use = par_weight(g, tab, f, hp_t[hh], w);
            if (use == 0) continue;
            if (use < 0) break;
            add(rows_t + (size_t)hh * R, (float)w);
          }
        }
        // after both forms: in one of them alone, the sums would be copied
        // between two register sets for each angle
        if (use1) add(pr, w1);
        if (use2) add(pr + R, w2);
      }
    }
    if (FOLD && group_ends && grp + 1 < ngrp) {
      // running sum of the groups so far (the last group's is added below)
      if (active) {
#pragma unroll
        for (int q = 0; q < R; q++)
          if (q < nk) {
            const Acc t = q < nrow ? acc[q] : (Acc)0;
            vcol[q] = grp == 0 ? (float)t : (float)((Acc)vcol[q] + t);
          }
      }
#pragma unroll
      for (int q = 0; q < R; q++) acc[q] = (Acc)0;
    }
    if (!(next < next_gb)) break;
    if (group_ends) grp++;
    a0 = next;
    gb = next_gb;
    buf ^= 1;
  }
  if (!active) return 0.0;
  double ss = 0.0;
#pragma unroll
  for (int q4 = 0; q4 < R; q4 += 4) {
    if (q4 + 4 <= nrow && !(FOLD && groups > 1)) {
#pragma unroll
      for (int q = q4; q < q4 + 4; q++) vcol[q] = (float)acc[q];
      if (norm) {
#pragma unroll
        for (int q = q4; q < q4 + 4; q++) {
          const float o = (float)acc[q];
          ss += (double)o * (double)o;
        }
      }
      continue;
    }
#pragma unroll
    for (int q = q4; q < q4 + 4; q++)
      if (q < nk) {
        // slices without a row keep what they hold
        float o;
        if (FOLD && groups > 1)
          o = (float)((Acc)vcol[q] + (q < nrow ? acc[q] : (Acc)0));
        else
          o = q < nrow ? (float)acc[q] : (!FOLD && acc_in ? vcol[q] : 0.0f);
        vcol[q] = o;
        ss += (double)o * (double)o;
      }
  }
  return ss;
}

}  // namespace ccpi
