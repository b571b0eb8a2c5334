// diffusion.hip -- viscous, heat and multicomponent (Fick + correction
// velocity) flux divergence.
//
// Reference: src/prometeo_rhs.inl:1058-1282 (GetSigma, GetDiffusionFlux,
// updateRHSSpan), src/prometeo_rhs.cu:461-622.  Two kernels, the same
// operations in the same order for every face:
//   diffusion_kernel      all three directions of a right-hand side: a thread
//                         per cell forms both its faces along each and adds
//                         (F+ - F-) m_d to Conserved_t once for all of them;
//   diffusion_line_kernel one direction: a thread per cell of a few lines, cell
//                         values and fluxes handed on through LDS.
#include "common.hpp"
#include "kernels.hpp"
#include <type_traits>

namespace htr {

// weights of the left and right cell of a face (Interp2Staggered)
struct FaceW {
   double a, b;
   __device__ double operator()(double l, double r) const { return a*l + b*r; }
};

template<class MX, bool SOA>
struct DiffCell {
   static constexpr int NS = MX::NS;
   // what the species part of a face reads of a cell
   double X[NS], Di[NS], rY[NS];
   double rho, T, lam, W;      // W: molar weight of the mixture from X
   static constexpr bool LAZY = false;
   __device__ __forceinline__ double x(int i) const { return X[i]; }
   __device__ __forceinline__ double di(int i) const { return Di[i]; }
   __device__ __forceinline__ double ry(int i) const { return rY[i]; }
   __device__ __forceinline__ void load(const htr_fields &f, const DMix &m, uint32_t o)
   {
#pragma unroll
      for (int i = 0; i < NS; i++) {
         X[i] = ldo<double, SOA>(f.MolarFracs, o, i);
         Di[i] = ldo<double, SOA>(f.Di, o, i);
         rY[i] = ldo<double, SOA>(f.Conserved, o, i);
      }
      rho = ldo<double, SOA>(f.rho, o);
      T = ldo<double, SOA>(f.temperature, o);
      lam = ldo<double, SOA>(f.lam, o);
      W = MX::MolarWeightFromX(m, X);
   }
};

// The same values in LDS, a cell's as a column of the block's: the species'
// are read after the enthalpies have been formed, and take no registers before
template<class MX>
struct LdsCell {
   static constexpr int NS = MX::NS, N = 3*NS + 4;
   static constexpr bool LAZY = true;
   const double *q;
   double rho, T, lam, W;
   template<class Cell> __device__ __forceinline__ static void put(double *q, const Cell &C)
   {
#pragma unroll
      for (int i = 0; i < NS; i++) { q[i*256] = C.X[i]; q[(NS + i)*256] = C.Di[i]; q[(2*NS + i)*256] = C.rY[i]; }
      q[3*NS*256] = C.rho; q[(3*NS + 1)*256] = C.T; q[(3*NS + 2)*256] = C.lam; q[(3*NS + 3)*256] = C.W;
   }
   __device__ __forceinline__ explicit LdsCell(const double *q_)
      : q(q_), rho(q[3*NS*256]), T(q[(3*NS + 1)*256]), lam(q[(3*NS + 2)*256]), W(q[(3*NS + 3)*256]) {}
   __device__ __forceinline__ double x(int i) const { return q[i*256]; }
   __device__ __forceinline__ double di(int i) const { return q[(NS + i)*256]; }
   __device__ __forceinline__ double ry(int i) const { return q[(2*NS + i)*256]; }
};

// GetDiffusionFlux (rhs.inl:1140-1218) at the face between cells P and Q,
// species part: the species fluxes into Flux[0..NS-1] and the heat flux
// (conduction + species enthalpy transport) returned
template<class MX, class Cell>
__device__ __forceinline__ double species_face(double *Flux, const DMix &m, const FaceW &w, double m_s,
                                               const Cell &P, const Cell &Q, const double *tab)
{
   constexpr int NS = MX::NS;
   const double rho_s = w(P.rho, Q.rho);
   const double iMixW_s = 1.0/w(P.W, Q.W);
   const double T_s = w(P.T, Q.T);
   double heatFlux = w(P.lam, Q.lam)*m_s*(P.T - Q.T);
   double ViCorr = 0.0;
   double hs[NS];
   MX::SpeciesEnthalpies(m, hs, T_s, tab);
   if constexpr (Cell::LAZY) {
#pragma unroll
      for (int i = 0; i < NS; i++) HTR_PIN(hs[i]);
   }
#pragma unroll
   for (int i = 0; i < NS; i++) {
      const double YiVi = w(P.di(i), Q.di(i))*m_s*(P.x(i) - Q.x(i))*MX::SpeciesW(m, i)*iMixW_s;
      Flux[i] = -rho_s*YiVi;
      heatFlux += rho_s*YiVi*hs[i];
      ViCorr += YiVi;
   }
#pragma unroll
   for (int i = 0; i < NS; i++) {
      const double corr = w(P.ry(i), Q.ry(i))*ViCorr;
      Flux[i] += corr;
      heatFlux -= corr*hs[i];
   }
   return heatFlux;
}

// The transverse gradients that the stress of a face along DIR takes from one
// of its cells: along D1 of velocity components (A1, B1), along D2 of (A2, B2)
template<int DIR>
struct Transverse {
   static constexpr int D1 = (DIR == 0) ? 1 : 0;   // getT1
   static constexpr int D2 = (DIR == 2) ? 1 : 2;   // getT2
   static constexpr int A1 = 0, B1 = (DIR == 2) ? 2 : 1;
   static constexpr int A2 = (DIR == 0) ? 0 : 1, B2 = 2;
   double a1, b1, a2, b2;
};

// momentum part of a face: the viscous stress into s and u.sigma returned
// (GetSigma, rhs.inl:1058-1137)
template<int DIR>
__device__ __forceinline__ double stress_face(double *s, const FaceW &w, double m_s, const double *vp, const double *vq,
                                              double muP, double muQ, const Transverse<DIR> &L, const Transverse<DIR> &R)
{
   const double mu_s = w(muP, muQ);
   double dn[3];
#pragma unroll
   for (int i = 0; i < 3; i++) dn[i] = m_s*(vq[i] - vp[i]);
   const double a1 = w(L.a1, R.a1), b1 = w(L.b1, R.b1), a2 = w(L.a2, R.a2), b2 = w(L.b2, R.b2);
   if (DIR == 0) {             // dU/dy, dV/dy, dU/dz, dW/dz
      s[0] = mu_s*(4*dn[0] - 2*b1 - 2*b2)/3;
      s[1] = mu_s*(dn[1] + a1);
      s[2] = mu_s*(dn[2] + a2);
   } else if (DIR == 1) {      // dU/dx, dV/dx, dV/dz, dW/dz
      s[0] = mu_s*(dn[0] + b1);
      s[1] = mu_s*(4*dn[1] - 2*a1 - 2*b2)/3;
      s[2] = mu_s*(dn[2] + a2);
   } else {                    // dU/dx, dW/dx, dV/dy, dW/dy
      s[0] = mu_s*(dn[0] + b1);
      s[1] = mu_s*(dn[1] + b2);
      s[2] = mu_s*(4*dn[2] - 2*a1 - 2*a2)/3;
   }
   double uSigma = 0.0;
#pragma unroll
   for (int i = 0; i < 3; i++) uSigma += w(vp[i], vq[i])*s[i];
   return uSigma;
}

__device__ __forceinline__ bool left_node(int t) { return t == L_S_node || t == L_C_node; }

// The thread's cell, its neighbours and the faces' node types and metrics
template<class MX, bool SOA>
struct Diffusion {
   static constexpr int NS = MX::NS, NEQ = MX::NEQ;
   using Cell = DiffCell<MX, SOA>;
   const htr_fields &f;
   const DMix &m;
   const Geo &g;
   const P3 &p;
   const double *tab;          // the species' polynomial coefficients in LDS
   uint32_t up[3], dn[3];      // offsets to the next and the previous cell along a direction

   __device__ __forceinline__ Diffusion(const htr_fields &f_, const DMix &m_, const Geo &g_, const P3 &p_,
                                        const double *tab_)
      : f(f_), m(m_), g(g_), p(p_), tab(tab_)
   {
#pragma unroll
      for (int d = 0; d < 3; d++) {
         int c = p.c[d];
         uint32_t o = p.o;
         step_up(g, d, c, o);
         up[d] = o - p.o;
         c = p.c[d];
         o = p.o;
         step_down(g, d, c, o);
         dn[d] = o - p.o;
      }
   }

   // the two faces of the cell along DIR: interpolation weights and staggered
   // metric of their left cells.  The minus face of a line's first cell is
   // that of p + offM1(nType) (rhs.inl:1253-1254): the previous cell's, but the
   // cell's own (plus) face at a left boundary node.
   // next: the cell after such a first cell, whose minus face is that plus face.
   struct Faces2 { FaceW wp, wm; double msp, msm, md; bool own, next; };
   template<int DIR>
   __device__ __forceinline__ Faces2 faces() const
   {
      const uint32_t om = p.o + dn[DIR];
      const int t = ldo<int, SOA>(f.nType[DIR], p.o), tm = ldo<int, SOA>(f.nType[DIR], om);
      Faces2 F;
      F.wp = F.wm = { 0.5, 0.5 };
      if (!wave_all(t == Std_node && tm == Std_node)) {
         F.wp = { (double)c_st.Interp[t][0], (double)c_st.Interp[t][1] };
         F.wm = { (double)c_st.Interp[tm][0], (double)c_st.Interp[tm][1] };
      }
      F.msp = ldo<double, SOA>(f.m_s[DIR], p.o);
      F.msm = ldo<double, SOA>(f.m_s[DIR], om);
      F.md = ldo<double, SOA>(f.m_d[DIR], p.o);
      F.own = p.c[DIR] == g.elo[DIR] && left_node(t);
      F.next = p.c[DIR] == g.elo[DIR] + 1 && left_node(tm);
      return F;
   }

   // weights of the plus face of a cell of node type t
   __device__ __forceinline__ static FaceW weights(int t)
   {
      if (wave_all(t == Std_node)) return { 0.5, 0.5 };
      return { (double)c_st.Interp[t][0], (double)c_st.Interp[t][1] };
   }

   // species fluxes along DIR into ct[0..NS-1]; the heat fluxes of the plus and
   // minus face into hp, hm
   template<int DIR>
   __device__ __forceinline__ void species(double *ct, const Cell &C0, double &hp, double &hm) const
   {
      const Faces2 F = faces<DIR>();
      double Fp[NS], Fm[NS];
      Cell C;
      C.load(f, m, p.o + up[DIR]);
      hp = species_face<MX>(Fp, m, F.wp, F.msp, C0, C, tab);
#pragma unroll
      for (int i = 0; i < NS; i++) HTR_PIN(Fp[i]);
      HTR_PIN(hp);
      C.load(f, m, p.o + dn[DIR]);
      hm = species_face<MX>(Fm, m, F.wm, F.msm, C, C0, tab);
      if (F.own) hm = hp;
#pragma unroll
      for (int i = 0; i < NS; i++) {
         if (F.own) Fm[i] = Fp[i];
         ct[i] += (Fp[i] - Fm[i])*F.md;
         HTR_PIN(ct[i]);
      }
      HTR_PIN(hm);
   }

   __device__ double vel(uint32_t o, int i) const { return ldo<double, SOA>(f.velocity, o, i); }

   // getDeriv of velocity component i along DD at the cell of offset o, whose
   // coordinate along DD is the thread's own
   struct Node { bool lo, hi; double g0, g1, mm; };
   template<int DD>
   __device__ __forceinline__ Node node(uint32_t o) const
   {
      Node n;
      const int t = ldo<int, SOA>(f.nType[DD], o);
      n.mm = ldo<double, SOA>(f.m_d[DD], o);
      n.g0 = n.g1 = 0.5;
      if (!wave_all(t == Std_node)) { n.g0 = (double)c_st.Grad[t][0]; n.g1 = (double)c_st.Grad[t][1]; }
      // stencil offsets of a node type are 0 or the natural ones
      n.lo = left_node(t);
      n.hi = t == R_S_node || t == R_C_node;
      return n;
   }
   template<int DD>
   __device__ __forceinline__ double deriv(const Node &n, uint32_t o, int i, double x) const
   {
      const double a = vel(o + dn[DD], i), b = vel(o + up[DD], i);
      return (n.g0*(x - (n.lo ? x : a)) + n.g1*((n.hi ? x : b) - x))*n.mm;
   }

   template<int DIR>
   __device__ __forceinline__ Transverse<DIR> transverse(uint32_t o, const double *v) const
   {
      using T = Transverse<DIR>;
      T r;
      const Node n1 = node<T::D1>(o), n2 = node<T::D2>(o);
      r.a1 = deriv<T::D1>(n1, o, T::A1, v[T::A1]);
      r.b1 = deriv<T::D1>(n1, o, T::B1, v[T::B1]);
      r.a2 = deriv<T::D2>(n2, o, T::A2, v[T::A2]);
      r.b2 = deriv<T::D2>(n2, o, T::B2, v[T::B2]);
      HTR_PIN(r.a1); HTR_PIN(r.b1); HTR_PIN(r.a2); HTR_PIN(r.b2);
      return r;
   }

   // stress and energy fluxes along DIR into ct[0..3] (momentum, energy); v0, mu0,
   // G0: the cell's velocity, viscosity and transverse gradients.  Where the
   // minus face is the plus face, the reference takes the plus face's left
   // gradients at p + 1, handed on from the face before (rhs.inl:1212-1214);
   // that face is also the next cell's minus face.
   template<int DIR>
   __device__ __forceinline__ void stress(double *ct, const double *v0, double mu0, double hp, double hm) const
   {
      const Faces2 F = faces<DIR>();
      const Transverse<DIR> G0 = transverse<DIR>(p.o, v0);
      double Fp[4], Fm[4], v[3];
      {
         const uint32_t o = p.o + up[DIR];
#pragma unroll
         for (int i = 0; i < 3; i++) v[i] = vel(o, i);
         const double mu = ldo<double, SOA>(f.mu, o);
         const Transverse<DIR> G = transverse<DIR>(o, v);
         Fp[3] = (stress_face<DIR>(Fp, F.wp, F.msp, v0, v, mu0, mu, F.own ? G : G0, G) - hp);
         if (F.own) Fm[3] = (stress_face<DIR>(Fm, F.wp, F.msp, v0, v, mu0, mu, G0, G) - hm);
#pragma unroll
         for (int i = 0; i < 4; i++) HTR_PIN(Fp[i]);
      }
      if (!F.own) {
         const uint32_t o = p.o + dn[DIR];
#pragma unroll
         for (int i = 0; i < 3; i++) v[i] = vel(o, i);
         const double mu = ldo<double, SOA>(f.mu, o);
         const Transverse<DIR> G = transverse<DIR>(o, v);
         Fm[3] = (stress_face<DIR>(Fm, F.wm, F.msm, v, v0, mu, mu0, F.next ? G0 : G, G0) - hm);
      }
#pragma unroll
      for (int i = 0; i < 4; i++) { ct[i] += (Fp[i] - Fm[i])*F.md; HTR_PIN(ct[i]); }
   }
};

// All three directions.  Each face is formed twice, which costs 1400 FP64
// operations more per cell and saves two thirds of the passes over memory.
// Bound by the loads' address cycles (16 per 64-lane 8-byte load; a wave issues 481
// where it straddles a range of the polynomials, counted) and FP64 issue at two
// waves per SIMD.  With the walks along lines before it in brackets: 256^3 air 3.7
// (4.8) ms, 4.5 about 6000 K; 512x256x128 boundary layer 3.8 (4.8) ms; 117x93x75
// air 195 (315) us; 32^3 one species 11 (102) us.
//
// The faces of a cell lie between temperatures, so in a flow about a range
// switch of the polynomials most waves straddle it.  Their coefficients come
// from a copy in LDS instead of 90 gathers per direction through the address
// unit that the fields' loads already fill (160^3 air about 6000 K 1318 -> 1073
// us, 907-918 us at other temperatures with and without).
template<class MX, bool SOA>
__global__ void __launch_bounds__(256, 2)
diffusion_kernel(const htr_fields f, const DMix *__restrict__ mix, const Geo g, uint32_t per)
{
   constexpr int NS = MX::NS;
   constexpr bool TAB = !MX::CP && SOA;
   __shared__ double tab[TAB ? NS*36 : 1];
   if constexpr (TAB) {
      for (int k = threadIdx.x; k < NS*36; k += 256) tab[k] = mix->sp[k/36].cp[k/12 % 3][k % 12];
      __syncthreads();
   }
   P3 p;
   if (!strip_cell(g, per, p)) return;
   const Diffusion<MX, SOA> D(f, *mix, g, p, TAB ? tab : nullptr);
   // species first, then momentum and energy, so that the species' cell values
   // are not held beside the velocity gradients; only the faces' heat fluxes
   // pass from one to the other
   double hp[3], hm[3];
   {
      DiffCell<MX, SOA> C0;
      C0.load(f, *mix, p.o);
      double ct[NS];
#pragma unroll
      for (int i = 0; i < NS; i++) ct[i] = ldo<double, SOA>(f.Conserved_t, p.o, i);
      D.template species<2>(ct, C0, hp[2], hm[2]);
      D.template species<1>(ct, C0, hp[1], hm[1]);
      D.template species<0>(ct, C0, hp[0], hm[0]);
#pragma unroll
      for (int i = 0; i < NS; i++) *ptr_o<double, SOA>(f.Conserved_t, p.o, i) = ct[i];
   }
   double v0[3], ct[4];
#pragma unroll
   for (int i = 0; i < 3; i++) v0[i] = D.vel(p.o, i);
   const double mu0 = ldo<double, SOA>(f.mu, p.o);
#pragma unroll
   for (int i = 0; i < 4; i++) ct[i] = ldo<double, SOA>(f.Conserved_t, p.o, NS + i);
   D.template stress<2>(ct, v0, mu0, hp[2], hm[2]);
   D.template stress<1>(ct, v0, mu0, hp[1], hm[1]);
   D.template stress<0>(ct, v0, mu0, hp[0], hm[0]);
#pragma unroll
   for (int i = 0; i < 4; i++) *ptr_o<double, SOA>(f.Conserved_t, p.o, NS + i) = ct[i];
}

// One direction alone.  A block holds LINES lines of the direction side by side
// (a cache line of x-adjacent cells for y and z), CELLS consecutive cells of each,
// threads on the lines first; a line counts the cell before and the cell after
// its cells too.  A thread loads its own cell, takes the next one's values from
// the thread that holds it, forms the plus face and takes the minus face from
// the thread before: every face is formed once and every cell loaded once, but
// for the block's first and last cells, which only hand on (blocks overlap by
// two).  Everything is handed on through LDS, and the cell's own values are read
// back from there too, so that 120 registers suffice and four blocks share a CU
// (values in registers: three blocks, 140^3 along y and z 10 % slower).  All loads
// go out before the first barrier; loaded where they are used, some after three
// barriers, a 200^2 box of one species took 8.8-9.0 us, now 7.5, and 140^3 air
// 5 to 12 % more.  Per-point arrays share a CU three blocks at a time: with four,
// or with two, the vector cache loses the records that a thread reads component by
// component (139x67x101 along x 124 us, two blocks 138).
// Bound by memory: 140^3 air has 0.98 GB that the pass cannot do without.  Its
// time with the clearing of Conserved_t before it, along x, y and z; in brackets
// with a thread per cell that forms both its faces, then with the walks along
// lines before that, which formed each face once but passed twice over the cells:
//   140^3, 2700 K                     251 280 260  (320 314 312; 333 385 369) us
//   140^3, 6000 K, where waves straddle
//     a range of the polynomials      260 296 269  (384 388 393; 331 384 371)
//   139x67x101, 6000 K                 93 103  98  (143 142 142; 117 126 124)
//   the same as per-point arrays      135 136 134  (229 229 227; 179 170 167)
//   700x500, 2700 K                    36  42      ( 43  43; 49 78)
template<int DIR> struct Lines {
   static constexpr int LINES = (DIR == 0) ? 1 : 16, CELLS = 256/LINES, MINE = CELLS - 2;
   static constexpr int B = (DIR == 2) ? 1 : 2;      // the other cross direction of y and z
};

// blocks of a launch: x takes the rows of a strip of kStripRows in y, the strips
// one after the other, y inside z; y and z take groups of LINES lines, x inside
// the other direction
template<int DIR>
struct LineGrid {
   uint32_t per, blocks;                             // blocks of a full strip, blocks of the launch
   explicit LineGrid(const Geo &g)
   {
      using S = Lines<DIR>;
      const int rows = std::min<int>(kStripRows, g.esz[1]);
      const int64_t lines = (DIR == 0) ? (int64_t)rows*g.esz[2] : ((int64_t)g.esz[0]*g.esz[S::B] + S::LINES - 1)/S::LINES;
      per = (uint32_t)((((int64_t)g.esz[DIR] + 2)*lines - 2 + S::MINE - 1)/S::MINE);
      blocks = ((DIR == 0 ? (uint32_t)((g.esz[1] + rows - 1)/rows) : 1u)*per + 7u) & ~7u;
   }
};

// the thread's cell p, i its place in the line (-1: the cell before the line,
// esz: the one after it), mine: the thread updates it; false past the end (the
// whole block)
template<int DIR>
__device__ __forceinline__ bool line_cell(const Geo &g, uint32_t per, P3 &p, int &i, bool &mine)
{
   using S = Lines<DIR>;
   const uint32_t b = xcd_block(blockIdx.x, gridDim.x);
   const uint32_t rows = min((uint32_t)kStripRows, (uint32_t)g.esz[1]);
   const uint32_t strip = DIR == 0 ? b/per : 0u, y0 = strip*rows;
   if (DIR == 0 && y0 >= (uint32_t)g.esz[1]) return false;
   const uint32_t h = min(rows, (uint32_t)g.esz[1] - y0);
   const uint32_t nl = (uint32_t)g.esz[0]*(uint32_t)g.esz[S::B];
   const uint32_t len = (uint32_t)g.esz[DIR] + 2u;
   const uint32_t ids = len*(DIR == 0 ? h*(uint32_t)g.esz[2] : (nl + S::LINES - 1u)/S::LINES);
   const uint32_t first = (b - strip*per)*S::MINE;
   if (first + 2u >= ids) return false;
   const uint32_t k = threadIdx.x/S::LINES;
   const uint32_t id = min(first + k, ids - 1u), r = id/len;
   i = (int)(id - r*len) - 1;
   mine = k >= 1u && k <= (uint32_t)S::MINE && first + k == id && i >= 0 && i < g.esz[DIR];
   int c[3];
   if (DIR == 0) {
      const uint32_t z = r/h;
      c[1] = g.elo[1] + (int)(y0 + r - z*h);
      c[2] = g.elo[2] + (int)z;
   } else {
      const uint32_t at = r*S::LINES + threadIdx.x % S::LINES, line = min(at, nl - 1u), q = line/(uint32_t)g.esz[0];
      mine = mine && at == line;
      c[0] = g.elo[0] + (int)(line - q*(uint32_t)g.esz[0]);
      c[S::B] = g.elo[S::B] + (int)q;
   }
   c[DIR] = g.elo[DIR] + min(max(i, 0), g.esz[DIR] - 1);
   p = mkp(g, c[0], c[1], c[2]);
   if (i < 0) step_down(g, DIR, p.c[DIR], p.o);
   if (i == g.esz[DIR]) step_up(g, DIR, p.c[DIR], p.o);
   return true;
}

// y: the x of thread q, by every thread of the block.  The first barrier: what
// was handed on before has been read
template<int N>
__device__ __forceinline__ void hand_on(double *buf, int q, const double *x, double *y)
{
   __syncthreads();
#pragma unroll
   for (int k = 0; k < N; k++) buf[k*256 + threadIdx.x] = x[k];
   __syncthreads();
#pragma unroll
   for (int k = 0; k < N; k++) y[k] = buf[k*256 + q];
}

template<class MX, int DIR, bool SOA>
__global__ void __launch_bounds__(256, 3)
diffusion_line_kernel(const htr_fields f, const DMix *__restrict__ mix, const Geo g, uint32_t per)
{
   constexpr int NS = MX::NS, NV = LdsCell<MX>::N;
   // per-point arrays of several species: LDS for three blocks per CU, not more
   constexpr int COLS = (!SOA && NV < 26 && NS > 1) ? 26 : (NV > 8) ? NV : 8;
   __shared__ double buf[COLS*256];
   P3 p;
   int i;
   bool mine;
   if (!line_cell<DIR>(g, per, p, i, mine)) return;
   const int me = (int)threadIdx.x, next = (me + Lines<DIR>::LINES) & 255, prev = (me - Lines<DIR>::LINES) & 255;
   const Diffusion<MX, SOA> D(f, *mix, g, p, nullptr);
   const int t = ldo<int, SOA>(f.nType[DIR], p.o);
   const bool own = i == 0 && left_node(t);          // as in Diffusion::faces
   // everything that is loaded, before the first barrier: velocity, viscosity and
   // transverse gradients are for the second part
   const double ms = ldo<double, SOA>(f.m_s[DIR], p.o), md = ldo<double, SOA>(f.m_d[DIR], p.o);
   DiffCell<MX, SOA> C;
   C.load(f, *mix, p.o);
   double v0[8], ct[NS + 4];
#pragma unroll
   for (int k = 0; k < 3; k++) v0[k] = D.vel(p.o, k);
   v0[3] = ldo<double, SOA>(f.mu, p.o);
   const Transverse<DIR> G0 = D.template transverse<DIR>(p.o, v0);
   v0[4] = G0.a1; v0[5] = G0.b1; v0[6] = G0.a2; v0[7] = G0.b2;
#pragma unroll
   for (int k = 0; k < NS + 4; k++) ct[k] = ldo<double, SOA>(f.Conserved_t, p.o, k);
   double hp, hm;
   {
      double Fp[NS + 1], Fm[NS + 1];
      LdsCell<MX>::put(buf + me, C);
      __syncthreads();
      const LdsCell<MX> P(buf + me), Q(buf + next);
      Fp[NS] = species_face<MX>(Fp, *mix, D.weights(t), ms, P, Q, nullptr);
      hand_on<NS + 1>(buf, prev, Fp, Fm);
      hp = Fp[NS];
      hm = own ? hp : Fm[NS];
#pragma unroll
      for (int k = 0; k < NS; k++) {
         if (own) Fm[k] = Fp[k];
         ct[k] += (Fp[k] - Fm[k])*md;
      }
   }
   double v1[8], Fp[4], Fm[4];
   hand_on<8>(buf, next, v0, v1);
   const Transverse<DIR> G1 = { v1[4], v1[5], v1[6], v1[7] };
   const FaceW w = D.weights(t);
   // the plus face of an own cell takes its left gradients at the next cell
   // (Diffusion::stress), its minus face the cell's own
   Fp[3] = stress_face<DIR>(Fp, w, ms, v0, v1, v0[3], v1[3], own ? G1 : G0, G1) - hp;
   hand_on<4>(buf, prev, Fp, Fm);
   if (own) Fm[3] = stress_face<DIR>(Fm, w, ms, v0, v1, v0[3], v1[3], G0, G1) - hm;
#pragma unroll
   for (int k = 0; k < 4; k++) ct[NS + k] += (Fp[k] - Fm[k])*md;
   if (mine) {
#pragma unroll
      for (int k = 0; k < NS + 4; k++) *ptr_o<double, SOA>(f.Conserved_t, p.o, k) = ct[k];
   }
}

template<class MX, bool SOA>
static int launch_diff(int dirs, const htr_fields &f, const DMix *mix, const Geo &g, hipStream_t s)
{
   if (exec_cells(g) == 0) return HTR_OK;
   auto line = [&](auto dir) {
      constexpr int DIR = decltype(dir)::value;
      const LineGrid<DIR> lg(g);
      HTR_LAUNCH(HTR_DIR_NAME("diffusion", DIR), (diffusion_line_kernel<MX, DIR, SOA>), dim3(lg.blocks), dim3(256), 0, s,
                 f, mix, g, lg.per);
   };
   switch (dirs) {
      case 1: line(std::integral_constant<int, 0>()); break;
      case 2: line(std::integral_constant<int, 1>()); break;
      case 4: line(std::integral_constant<int, 2>()); break;
      case 7: {
         const StripGrid sg(g);
         HTR_LAUNCH("diffusion", (diffusion_kernel<MX, SOA>), dim3(sg.blocks), dim3(256), 0, s, f, mix, g, sg.per);
         break;
      }
      default: return set_error(HTR_E_ARG, "diffusion: bad directions %d", dirs);
   }
   return check_launch("diffusion_kernel");
}

// dirs: one direction's bit, or 7 for all three (in the order z, y, x)
template<class MX>
int diffusion_dispatch(int dirs, const htr_fields &f, const DMix *mix, const Geo &g, hipStream_t s)
{
   return g.soa ? launch_diff<MX, true>(dirs, f, mix, g, s) : launch_diff<MX, false>(dirs, f, mix, g, s);
}

template int diffusion_dispatch<MixCP>(int, const htr_fields &, const DMix *, const Geo &, hipStream_t);
template int diffusion_dispatch<MixAir>(int, const htr_fields &, const DMix *, const Geo &, hipStream_t);

} // namespace htr
