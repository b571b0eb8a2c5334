// common.hpp -- field views, periodic wrapping and launch helpers shared by
// the HTR hot-path kernels.
//
// Device-side addressing.  The host rebases every view to the low corner of
// Fluid_bounds (kernel coordinates run over [0, bsz) in each direction) and
// checks that the spatial strides of every view are an integer multiple k of
// one common triple (cx, cy, cz): that covers structure-of-arrays fields
// (k = 1, components sc = N apart) as well as the reference's per-point
// arrays (VecNEq, VecNSp, Vec3: k = number of components, sc = 1).  A point
// carries one 32-bit offset o = x cx + y cy + z cz, and an access is
//   field base + comp*sc*sizeof(T)  (uniform)  +  o * k*sizeof(T)  (32-bit),
// so the backend uses a scalar base and one VGPR of offset per access instead
// of a 64-bit address per (point, field).  In the kernels' copy of a view,
// sx holds k*sizeof(T) in bytes; sy and sz are unused.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>
#include <algorithm>
#include "../../include/htr_amd.h"
#include "mix.hpp"
#include "stencil.hpp"

namespace htr {

// Box geometry relative to the low corner of Fluid_bounds.
struct Geo {
   int32_t  bsz[3];   // Fluid_bounds extent
   int32_t  elo[3];   // execution rect, low corner
   int32_t  esz[3];   // execution rect, extent
   uint32_t cb[3];    // common stride triple (cx, cy, cz)
   int32_t  soa;      // every view has k = 1
};

// Time step of a launch: the host value dt, or, when radius is set, the
// ConstantCFL step (cfl / max spectral radius) read on the device from the
// result of a device-side reduction and multiplied by scale, in the
// reference's rounding order: dt = cfl/radius, then dt*scale
// (src/prometeo.rg:1165, :1419).
struct DtArg {
   double dt;
   const double *radius;
   double cfl, scale;
   __device__ double get() const { return radius ? (cfl/(*radius))*scale : dt; }
};

inline DtArg host_dt(double dt) { DtArg a; a.dt = dt; a.radius = nullptr; a.cfl = 0.0; a.scale = 0.0; return a; }

struct P3 {
   int32_t  c[3];
   uint32_t o;        // x cx + y cy + z cz
};

__device__ inline P3 mkp(const Geo &g, int x, int y, int z)
{
   P3 p;
   p.c[0] = x; p.c[1] = y; p.c[2] = z;
   p.o = (uint32_t)x*g.cb[0] + (uint32_t)y*g.cb[1] + (uint32_t)z*g.cb[2];
   return p;
}

__device__ inline void setc(const Geo &g, P3 &p, int d, int v)
{
   p.o += (uint32_t)(v - p.c[d])*g.cb[d];
   p.c[d] = v;
}

template<typename T>
__device__ inline const T *lp(const htr_view &v, const P3 &p, int comp)
{
   return reinterpret_cast<const T*>(reinterpret_cast<const char*>(v.ptr) + comp*v.sc*(int64_t)sizeof(T) +
                                     p.o*(uint32_t)v.sx);
}

template<typename T>
__device__ inline T ld(const htr_view &v, const P3 &p, int comp = 0) { return *lp<T>(v, p, comp); }

template<typename T>
__device__ inline T &at(const htr_view &v, const P3 &p, int comp = 0) { return *const_cast<T*>(lp<T>(v, p, comp)); }

// Access at the offset o of a point.  SOA: the caller guarantees that every
// view is structure-of-arrays (k = 1), and the byte offset is then o times the
// element size, the same register for every field of a type; otherwise it is
// a product per field (v_mul_lo_u32, four times the issue of an addition).
template<typename T, bool SOA>
__device__ __forceinline__ T *ptr_o(const htr_view &v, uint32_t o, int comp = 0)
{
   char *base = reinterpret_cast<char*>(v.ptr) + comp*v.sc*(int64_t)sizeof(T);
   return reinterpret_cast<T*>(base + (SOA ? o*(uint32_t)sizeof(T) : o*(uint32_t)v.sx));
}

template<typename T, bool SOA>
__device__ __forceinline__ T ldo(const htr_view &v, uint32_t o, int comp = 0) { return *ptr_o<T, SOA>(v, o, comp); }

// keeps the formation of a value, and the memory accesses around it, in
// program order
#ifdef __HIP_DEVICE_COMPILE__
#define HTR_PIN(x) asm volatile("" : "+v"(x) :: "memory")
#else
#define HTR_PIN(x) (void)(x)
#endif

// true when the predicate holds on every active lane of the wave (each lane
// for itself where there are no waves): chooses a path, never a result
__device__ __forceinline__ bool wave_all(bool p)
{
#ifdef __HIP_DEVICE_COMPILE__
   return __ballot(!p) == 0;
#else
   return p;
#endif
}

// warpPeriodic (src/Utils/PointDomain_helper.hpp:157-188): the point moved by
// off along d, wrapped into Fluid_bounds
__device__ inline P3 wplus(const Geo &g, int d, P3 p, int off)
{
   int c = p.c[d] + off;
   while (c >= g.bsz[d]) c -= g.bsz[d];
   while (c < 0) c += g.bsz[d];
   setc(g, p, d, c);
   return p;
}

__device__ inline P3 wminus(const Geo &g, int d, P3 p, int off) { return wplus(g, d, p, off); }

inline int64_t exec_cells(const Geo &g) { return (int64_t)g.esz[0]*g.esz[1]*g.esz[2]; }

// XCD-aware block order: the dispatcher hands workgroups to the eight XCDs
// round robin (block b runs on XCD b % 8), and each XCD has its own L2.  The
// logical index makes blocks with consecutive logical indices share an XCD
// (XCD x holds logical blocks [x n/8, (x+1) n/8)), so work items that touch
// the same cache lines -- neighbouring chunks of a face list -- meet in one
// L2.  Identity when n is not a multiple of 8.
__device__ inline uint32_t xcd_block(uint32_t b, uint32_t n)
{
   if (n & 7u) return b;
   return (b & 7u)*(n >> 3) + (b >> 3);
}

// point of the execution rect for a flat index, x fastest (the host keeps
// the cell count below 2^31)
__device__ inline P3 exec_point(const Geo &g, int64_t i64)
{
   uint32_t i = (uint32_t)i64;
   const int x = g.elo[0] + (int)(i % (uint32_t)g.esz[0]);
   i /= (uint32_t)g.esz[0];
   const int y = g.elo[1] + (int)(i % (uint32_t)g.esz[1]);
   const int z = g.elo[2] + (int)(i / (uint32_t)g.esz[1]);
   return mkp(g, x, y, z);
}

// offset of the neighbouring cell along d, one step up or down with the
// periodic wrap; c is its coordinate
__device__ __forceinline__ void step_up(const Geo &g, int d, int &c, uint32_t &o)
{
   const bool w = c + 1 == g.bsz[d];
   o += w ? -(uint32_t)(g.bsz[d] - 1)*g.cb[d] : g.cb[d];
   c = w ? 0 : c + 1;
}
__device__ __forceinline__ void step_down(const Geo &g, int d, int &c, uint32_t &o)
{
   const bool w = c == 0;
   o += w ? (uint32_t)(g.bsz[d] - 1)*g.cb[d] : -g.cb[d];
   c = w ? g.bsz[d] - 1 : c - 1;
}

// Cells of a launch whose threads read neighbours in y and z: the execution
// rect in strips of kStripRows rows, one after the other, each flattened (x
// fastest, then the rows of the strip, then z) into blocks of 256 cells, the
// blocks in XCD-aware order, so that what an XCD has in flight is a strip of a
// few planes.  (Strips cut in x as well, 32 to 128 cells wide, were no faster:
// euler_kg_kernel on 256^3 air 3.87-4.04 against 3.90 ms.)
constexpr int kStripRows = 16;

struct StripGrid {
   uint32_t per, blocks;                             // blocks of a full strip, blocks of the launch
   explicit StripGrid(const Geo &g)
   {
      const int rows = std::min<int>(kStripRows, g.esz[1]);
      per = (uint32_t)(((int64_t)g.esz[0]*rows*g.esz[2] + 255)/256);
      blocks = ((uint32_t)((g.esz[1] + rows - 1)/rows)*per + 7u) & ~7u;
   }
};

// the cell of a thread; false past the strip's end
__device__ inline bool strip_cell(const Geo &g, uint32_t per, P3 &p)
{
   const uint32_t ex = (uint32_t)g.esz[0], ey = (uint32_t)g.esz[1];
   const uint32_t b = xcd_block(blockIdx.x, gridDim.x);
   const uint32_t rows = min((uint32_t)kStripRows, ey);
   const uint32_t s = b/per, y0 = s*rows;
   if (y0 >= ey) return false;
   const uint32_t h = min(rows, ey - y0);
   const uint32_t i = (b - s*per)*256u + threadIdx.x;
   const uint32_t r = i/ex, z = r/h;
   if (z >= (uint32_t)g.esz[2]) return false;
   p = mkp(g, g.elo[0] + (int)(i - r*ex), g.elo[1] + (int)(y0 + r - z*h), g.elo[2] + (int)z);
   return true;
}

} // namespace htr
