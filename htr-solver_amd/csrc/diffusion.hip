// diffusion.hip -- viscous, heat and multicomponent (Fick + correction
// velocity) flux divergence.
//
// Reference: src/prometeo_rhs.inl:1058-1282 (GetSigma, GetDiffusionFlux,
// updateRHSSpan), src/prometeo_rhs.cu:461-622.  One thread per cell forms both
// its faces along every direction of the launch and adds (F+ - F-) m_d to
// Conserved_t, which is read and written once for all directions.
//
// Each face is thus formed twice, which costs 1400 FP64 operations more per
// cell and saves two thirds of the passes over memory: the walks along the
// lines that this replaces took a pass per direction and component group
// (species; momentum and energy, with the heat flux handed over through a
// buffer), each reading its fields and reading and writing Conserved_t.  Bound
// by the loads' address cycles (16 per 64-lane 8-byte load, 270 loads per
// cell) and FP64 issue at two waves per SIMD.  All three directions, with the
// walks in brackets: 256^3 air 3.8 (4.8) ms, 512x256x128 boundary layer 3.8
// (4.8) ms, 117x93x75 air 195 (315) us, 32^3 one species 13 (102) us.
#include "common.hpp"
#include "kernels.hpp"

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

// GetDiffusionFlux (rhs.inl:1140-1218) at the face between cells P and Q,
// species part: the species fluxes into Flux[0..NS-1] and the heat flux
// (conduction + species enthalpy transport) returned
template<class MX, bool SOA>
__device__ __forceinline__ double species_face(double *Flux, const DMix &m, const FaceW &w, double m_s,
                                               const DiffCell<MX, SOA> &P, const DiffCell<MX, SOA> &Q,
                                               const double *tab)
{
   constexpr int NS = MX::NS;
   const double rho_s = w(P.rho, Q.rho);
   const double iMixW_s = 1.0/w(P.W, Q.W);
   const double T_s = w(P.T, Q.T);
   double heatFlux = w(P.lam, Q.lam)*m_s*(P.T - Q.T);
   double ViCorr = 0.0;
   double hs[NS];
   MX::SpeciesEnthalpies(m, hs, T_s, tab);
#pragma unroll
   for (int i = 0; i < NS; i++) {
      const double YiVi = w(P.Di[i], Q.Di[i])*m_s*(P.X[i] - Q.X[i])*MX::SpeciesW(m, i)*iMixW_s;
      Flux[i] = -rho_s*YiVi;
      heatFlux += rho_s*YiVi*hs[i];
      ViCorr += YiVi;
   }
#pragma unroll
   for (int i = 0; i < NS; i++) {
      const double corr = w(P.rY[i], Q.rY[i])*ViCorr;
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

// The thread's cell, its neighbours and the faces' node types and metrics
template<class MX, int DIRS, bool SOA>
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
      F.own = p.c[DIR] == g.elo[DIR] && (t == L_S_node || t == L_C_node);
      F.next = p.c[DIR] == g.elo[DIR] + 1 && (tm == L_S_node || tm == L_C_node);
      return F;
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
      hp = species_face<MX, SOA>(Fp, m, F.wp, F.msp, C0, C, tab);
#pragma unroll
      for (int i = 0; i < NS; i++) HTR_PIN(Fp[i]);
      HTR_PIN(hp);
      C.load(f, m, p.o + dn[DIR]);
      hm = species_face<MX, SOA>(Fm, m, F.wm, F.msm, C, C0, tab);
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
      n.lo = t == L_S_node || t == L_C_node;
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

// The faces of a cell lie between temperatures, so in a flow about a range
// switch of the polynomials most waves straddle it.  Their coefficients come
// from a copy in LDS instead of 90 gathers per direction through the address
// unit that the fields' loads already fill, where the registers allow it: at
// two waves per SIMD, which all three directions at once have anyway (160^3 air
// about 6000 K 1318 -> 1073 us, 907-918 us at other temperatures with and
// without).  One direction alone fits three waves without the copy and would
// spill with it; along x, 140^3, at 2700 K and about 6000 K: 336 and 388 us, with
// the copy at two waves 358 and 378.
template<class MX, int DIRS, bool SOA>
__global__ void __launch_bounds__(256, DIRS == 7 ? 2 : 3)
diffusion_kernel(const htr_fields f, const DMix *__restrict__ mix, const Geo g, uint32_t per)
{
   constexpr int NS = MX::NS;
   constexpr bool TAB = !MX::CP && SOA && DIRS == 7;
   __shared__ double tab[TAB ? NS*36 : 1];
   if constexpr (TAB) {
      for (int k = threadIdx.x; k < NS*36; k += 256) tab[k] = mix->sp[k/36].cp[k/12 % 3][k % 12];
      __syncthreads();
   }
   P3 p;
   if (!strip_cell(g, per, p)) return;
   const Diffusion<MX, DIRS, SOA> D(f, *mix, g, p, TAB ? tab : nullptr);
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
      if constexpr ((DIRS & 4) != 0) D.template species<2>(ct, C0, hp[2], hm[2]);
      if constexpr ((DIRS & 2) != 0) D.template species<1>(ct, C0, hp[1], hm[1]);
      if constexpr ((DIRS & 1) != 0) D.template species<0>(ct, C0, hp[0], hm[0]);
#pragma unroll
      for (int i = 0; i < NS; i++) *ptr_o<double, SOA>(f.Conserved_t, p.o, i) = ct[i];
   }
   double v0[3], ct[4];
#pragma unroll
   for (int i = 0; i < 3; i++) v0[i] = D.vel(p.o, i);
   const double mu0 = ldo<double, SOA>(f.mu, p.o);
#pragma unroll
   for (int i = 0; i < 4; i++) ct[i] = ldo<double, SOA>(f.Conserved_t, p.o, NS + i);
   if constexpr ((DIRS & 4) != 0) D.template stress<2>(ct, v0, mu0, hp[2], hm[2]);
   if constexpr ((DIRS & 2) != 0) D.template stress<1>(ct, v0, mu0, hp[1], hm[1]);
   if constexpr ((DIRS & 1) != 0) D.template stress<0>(ct, v0, mu0, hp[0], hm[0]);
#pragma unroll
   for (int i = 0; i < 4; i++) *ptr_o<double, SOA>(f.Conserved_t, p.o, NS + i) = ct[i];
}

template<class MX, int DIRS>
static int launch_diff(const htr_fields &f, const DMix *mix, const Geo &g, hipStream_t s)
{
   if (exec_cells(g) == 0) return HTR_OK;
   const StripGrid sg(g);
   const char *name = (DIRS == 7) ? "diffusion" : (DIRS == 1) ? "diffusion_x" : (DIRS == 2) ? "diffusion_y" : "diffusion_z";
   if (g.soa) {
      HTR_LAUNCH(name, (diffusion_kernel<MX, DIRS, true>), dim3(sg.blocks), dim3(256), 0, s, f, mix, g, sg.per);
   } else {
      HTR_LAUNCH(name, (diffusion_kernel<MX, DIRS, false>), dim3(sg.blocks), dim3(256), 0, s, f, mix, g, sg.per);
   }
   return check_launch("diffusion_kernel");
}

// dirs: one direction's bit, or 7 for all three (in the order z, y, x)
template<class MX>
int diffusion_dispatch(int dirs, const htr_fields &f, const DMix *mix, const Geo &g, hipStream_t s)
{
   switch (dirs) {
      case 1: return launch_diff<MX, 1>(f, mix, g, s);
      case 2: return launch_diff<MX, 2>(f, mix, g, s);
      case 4: return launch_diff<MX, 4>(f, mix, g, s);
      case 7: return launch_diff<MX, 7>(f, mix, g, s);
      default: return set_error(HTR_E_ARG, "diffusion: bad directions %d", dirs);
   }
}

template int diffusion_dispatch<MixCP>(int, const htr_fields &, const DMix *, const Geo &, hipStream_t);
template int diffusion_dispatch<MixAir>(int, const htr_fields &, const DMix *, const Geo &, hipStream_t);

} // namespace htr
