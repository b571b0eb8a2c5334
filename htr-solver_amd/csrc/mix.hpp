// mix.hpp -- device image of a mixture and its thermodynamic, transport and
// kinetic functions, templated on the species count NS (NS == 1 with
// constprop set is the calorically perfect gas).
//
// Every function keeps the association order of the reference (so that the
// GPU and the reference CPU tasks round the same way up to libm ulps and FMA
// contraction):
//   src/Mixtures/MultiComponent.inl:45-436, src/Mixtures/Species.inl:35-357,
//   src/Mixtures/Reaction.inl:34-338, src/Mixtures/ConstPropMix.inl:65-168.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace htr {

constexpr int MAX_SP   = 40;
constexpr int MAX_REAC = 256;
constexpr int MAX_ED   = 4;
constexpr int MAX_PD   = 4;
constexpr int MAX_TB   = 8;

constexpr double PI    = 3.1415926535898;
constexpr double PI15  = 5.5683279968317265;     // PI^1.5
constexpr double RGAS  = 8.3144598;
constexpr double NA    = 6.02214086e23;
constexpr double KB    = 1.38064852e-23;
constexpr double EPS0  = 8.8541878128e-12;
constexpr double ECRG  = 1.60217662e-19;

enum { GEOM_ATOM = 0, GEOM_LINEAR = 1, GEOM_NONLINEAR = 3 };
enum { REAC_STD = 0, REAC_THIRDB = 1 };
enum { VISC_CONSTANT = 0, VISC_POWERLAW = 1, VISC_SUTHERLAND = 2 };

struct DSpec {
   double W;
   float  TSwitch1, TSwitch2, TMin, TMax;
   int    nPoly;
   int    geom;
   // NASA coefficients per range ([0] high, [1] mid, [2] low), then three
   // quotients of them the polynomials use, formed once at upload (the same
   // correctly rounded divisions, so every value is unchanged):
   // [9] c4/3, [10] c5/6, [11] c6/5
   double cp[3][12];
   double rOvW;                // R/W, formed once at upload
   double iW;                  // 1/W (correctly rounded, for quot())
   double tHi, tLo;            // range switches: T > tHi takes cp[0] (infinite with two ranges), T > tLo cp[1]
   double sigma, kbOveps, mu, alpha, Z298;
};

struct DReac {
   int    kind, has_backward, Ne, Np, Ntb, pad;
   double A;
   float  n, EovR;
   int    ed_ind[MAX_ED];
   float  ed_nu[MAX_ED];
   int    pd_ind[MAX_PD];
   float  pd_nu[MAX_PD];
   int    tb_ind[MAX_TB];
   float  tb_eff[MAX_TB];
};

constexpr int MAX_SPR  = MAX_REAC*(MAX_ED + MAX_PD);

// An entry of the species rows of the stoichiometry, for the lane-per-species
// passes of the implicit chemistry: reaction, signed coefficient, and the
// reaction's species (a byte each), so that a row's reads depend on nothing.
struct alignas(16) DRow { float nu; uint32_t info, eid, pid; };   // info: reaction | rc_info
// A reaction as the lane-per-reaction passes read it.  info: rc_info, and in
// the low byte the educts (bits 0-3) and products (4-7) of coefficient 2
struct alignas(16) DRate { double A, sumNu; float n, EovR; uint32_t info, eid, pid, pad[3]; };

// temperature-independent transport factors of a species and of a pair (i, j)
struct DTran { double mu, fV, zrot, isk; };
struct DPair { double w4, iw8, kT, iD; };

struct DMix {
   int    constprop, nSpec, nReac, viscModel;
   double R, gamma, Prandtl;
   double constVisc, plTRef, plVRef, suSRef, suTRef, suVRef;
   double PRef, TRef, MixWRef, iMixWRef, rhoRef, ieRef, iuRef, iCpRef, imuRef, ilamRef,
          iDiRef, iwiRef, iKiRef, Eps0, TMax, TMin;
   double XiRef[MAX_SP];
   DSpec  sp[MAX_SP];
   DReac  rc[MAX_REAC];
   DTran  tr[MAX_SP];
   DPair  pr[MAX_SP][MAX_SP];
   // Species-major image of the stoichiometry, for the lane-per-species
   // accumulation of the production rates: the entries of species s are
   // [spr_ptr[s], spr_ptr[s+1]), in the order the reaction loop of
   // GetProductionRates adds them (reaction order; educt entries, then
   // product entries), with the signed coefficient (-nu educt, +nu product).
   int     spr_ptr[MAX_SP + 1];
   int16_t spr_reac[MAX_SPR];
   float   spr_nu[MAX_SPR];
   // The same rows and the reactions field by field, so that the lanes of a
   // wave (a lane per species, a lane per reaction) read consecutive words:
   // entry k of species s is rows()[k*nSpec + s], k < spr_ptr[s+1] - spr_ptr[s]
   // <= nRows (behind the mixture, in its allocation); coefficients of a
   // species' polynomials are cpT[range][c][s].
   int     nRows, maxEd, maxPd, maxTb;
   int     unitNu;             // every stoichiometric coefficient is 1 or 2
   // with unitNu, two entries of a species' row in a word: reaction, doubled
   // (0x2000), negative (0x4000); past the row's end the reaction is nReac
   uint32_t prow[MAX_SPR/2 + 16][MAX_SP];
   double  cpT[3][12][MAX_SP];
   DRate   rate[MAX_REAC];
   float   kEnu[MAX_ED][MAX_REAC], kPnu[MAX_PD][MAX_REAC];
   int     kTid[MAX_TB][MAX_REAC];
   float   kTeff[MAX_TB][MAX_REAC];
   __host__ __device__ static size_t rows_at();
   __device__ const DRow *rows() const { return reinterpret_cast<const DRow*>(reinterpret_cast<const char*>(this) + rows_at()); }
};
__host__ __device__ inline size_t DMix::rows_at() { return (sizeof(DMix) + 255) & ~(size_t)255; }

// arity of a reaction in the upper half of a word: educts, products, third
// bodies that act (4 bits each), reversible
inline uint32_t rc_info(const DReac &r)
{
   const int tb = (r.kind == REAC_THIRDB) ? r.Ntb : 0;
   return ((uint32_t)r.Ne << 16) | ((uint32_t)r.Np << 20) | ((uint32_t)tb << 24) | (r.has_backward ? 1u << 28 : 0u);
}

#define HD __host__ __device__ inline

// x/b given rb, the correctly rounded 1/b: the quotient of the product is
// corrected twice by its exact residual, which makes it the correctly rounded
// one (Markstein's theorem: the first correction brings it within one ulp, the
// second rounds it correctly), and div_fixup restores the special values.  For
// |x| and |x/b| between 1e-290 and 1e300, where no step over- or underflows.
// 6 FP64 operations against the 11 of a division; worth it wherever a divisor
// is a constant of the mixture or serves several numerators.
HD double quot(double x, double b, double rb)
{
#ifdef __HIP_DEVICE_COMPILE__
   double q = x*rb;
   q = fma(fma(-b, q, x), rb, q);
   q = fma(fma(-b, q, x), rb, q);
   return __builtin_amdgcn_div_fixup(q, b, x);
#else
   (void)rb;
   return x/b;
#endif
}

// One thread's column of a shared species-major array: element i at
// p[i*stride] (stride = threads of the block, so a wave's lanes touch
// consecutive words).  The reaction loops index species arrays by runtime
// species ids; held in registers, each such access becomes a select over
// every entry, in LDS one address add.
struct SpeciesCol {
   double *p;
   int stride;
   HD double &operator[](int i) const { return p[i*stride]; }
};

HD double dmax(double a, double b) { return (a < b) ? b : a; }
HD double dmin(double a, double b) { return (b < a) ? b : a; }

// C^nu of a rate of progress: Reaction.inl:112-137 multiplies C for nu = 1
// and takes pow(C, nu) otherwise; nu = 2 (the dissociation products) is
// formed as C*C, the value pow gives to within its last bit, at the cost of a
// product in place of a pow
HD double conc_pow(double c, float nu)
{
   if (nu == 1.0f) return c;
   if (nu == 2.0f) return c*c;
   return pow(c, (double)nu);
}

// ---------------------------------------------------------------- species --
HD const double *cp_range(const DSpec &s, double T)
{
   return s.cp[T > s.tHi ? 0 : T > s.tLo ? 1 : 2];
}

// f(i, species i, its coefficients at T) for every species.  The range of a
// polynomial is a lane's own, so its nine coefficients would be nine gathers
// per species and evaluation, and the kernels that evaluate the polynomials
// several times (temperature Newton, Roe state, face enthalpies) were bound by
// them; nearly every wave has all its lanes in one range, and then the
// coefficients come through scalar loads and enter as scalar operands.  A wave
// that straddles a switch (and a mixture too large to hold its species'
// ranges) gathers, from tab where the kernel has copied the coefficients to
// LDS ([species][range][12], see diffusion_kernel).  (Selecting between the
// ranges' scalar coefficients, or taking the ranges one after another, was
// slower: 40 registers more, or the scalar loads' latency twice.)  256^3 air: Roe pass 0.79 -> 0.71 ms per direction (233 ->
// 147 VGPRs).  The chemistry source evaluates them once per cell and keeps the
// gathers (0.78 ms; 0.87 ms this way, for a wave less per SIMD).
template<int NS, class M, class F>
HD void species_loop(const M &m, double T, F f, const double *tab = nullptr)
{
#ifdef __HIP_DEVICE_COMPILE__
   if constexpr (NS <= 8) {
      const uint64_t all = __ballot(1);
      int r[NS];
      bool one = true;
#pragma unroll
      for (int i = 0; i < NS; i++) {
         const uint64_t hi = __ballot(T > m.sp[i].tHi), lo = __ballot(T > m.sp[i].tLo);
         one = one && (hi == 0 || hi == all) && (lo == 0 || lo == all);
         r[i] = hi ? 0 : lo ? 1 : 2;
      }
      // one species' coefficients at a time, in scalar or vector registers
      if (one) {
#pragma unroll
         for (int i = 0; i < NS; i++) {
            f(i, m.sp[i], m.sp[i].cp[r[i]]);
            __builtin_amdgcn_sched_barrier(0);
         }
      } else {
#pragma unroll
         for (int i = 0; i < NS; i++) {
            const DSpec &s = m.sp[i];
            f(i, s, tab ? tab + (i*3 + (T > s.tHi ? 0 : T > s.tLo ? 1 : 2))*12 : cp_range(s, T));
            __builtin_amdgcn_sched_barrier(0);
         }
      }
      return;
   }
#endif
#pragma unroll
   for (int i = 0; i < NS; i++) f(i, m.sp[i], cp_range(m.sp[i], T));
}

// the quotients of DSpec formed at upload
inline void derive_species(DSpec &s)
{
   for (int r = 0; r < 3; r++) {
      s.cp[r][9] = s.cp[r][4]/3;
      s.cp[r][10] = s.cp[r][5]/6;
      s.cp[r][11] = s.cp[r][6]/5;
   }
   s.rOvW = RGAS/s.W;
   s.iW = 1.0/s.W;
   s.tHi = (s.nPoly == 3) ? (double)s.TSwitch2 : HUGE_VAL;
   s.tLo = (double)s.TSwitch1;
}

// polynomials on the coefficients c of a range (Species.inl:35-160); S holds rOvW
template<class S>
HD double poly_cp(const S &s, const double *c, double T, double Tinv)
{
   const double poly = c[3] + T*(c[4] + T*(c[5] + T*c[6]));
   return s.rOvW*(c[0]*Tinv*Tinv + c[1]*Tinv + c[2] + T*poly);
}

HD double poly_free_enthalpy(const double *c, double T, double Tinv, double logT)
{
   const double G = -0.5*c[0]*Tinv*Tinv + c[1]*Tinv*(1.0 + logT) + c[2]*(1.0 - logT) + c[7]*Tinv - c[8];
   return G - 0.5*T*(c[3] + T*(c[9] + T*(c[10] + 0.1*T*c[6])));
}

template<class S>
HD double poly_enthalpy(const S &s, const double *c, double T, double Tinv, double logT)
{
   const double E = -c[0]*Tinv + c[1]*logT + c[7] + T*(c[2] + T*(c[3]*0.50 + T*(c[9] + T*(c[5]*0.25 + c[11]*T))));
   return E*s.rOvW;
}

HD double sp_cp(const DSpec &s, double T) { return poly_cp(s, cp_range(s, T), T, 1.0/T); }
HD double sp_free_enthalpy(const DSpec &s, double T) { return poly_free_enthalpy(cp_range(s, T), T, 1.0/T, log(T)); }
HD double sp_enthalpy(const DSpec &s, double T) { return poly_enthalpy(s, cp_range(s, T), T, 1.0/T, log(T)); }

// Collision integrals (Species.inl:163-190) as numerator and denominator: the
// transport properties divide by them, so a quotient of theirs is formed once
// with the other factors
HD double omega_mu_num(double T) { return 3.3530622607 + T*(2.53272006 + T*(2.9024238575 + T*0.11186138893)); }
HD double omega_mu_den(double T)
{ return 0.8662326188 + T*(1.3913958626 + T*(3.158490576 + T*(0.18973411754 + T*0.00018682962894))); }
HD double omega_D_num(double T) { return 6.8728271691 + T*(9.4122316321 + T*(7.7442359037 + T*0.23424661229)); }
HD double omega_D_den(double T)
{ return 1.45337701568 + T*(5.2269794238 + T*(9.7108519575 + T*(0.46539437353 + T*0.00041908394781))); }

// Rotational relaxation factor (Species.inl:290-295) of T* = kbOveps T
inline double sp_fzrot(double kbOveps, double T)
{
   const double tmp = 1.0/(kbOveps*T);
   return 1 + 0.5*pow(PI, 1.5)*sqrt(tmp) + (2 + 0.25*PI*PI)*tmp + pow(PI, 1.5)*pow(tmp, 1.5);
}

// The temperature-independent factors of the species' and pairs' transport
// properties, formed once when a mixture is uploaded
inline void derive_transport(DMix &m)
{
   for (int i = 0; i < m.nSpec; i++) {
      const DSpec &s = m.sp[i];
      DTran &t = m.tr[i];
      // Species.inl:193-199: mu = 5 sqrt(PI W/NA KB T)/(16 PI sigma^2 omega)
      t.mu = 5*sqrt(PI*s.W/NA*KB)/(16*PI*pow(s.sigma, 2.0));
      // Species.inl:310-357: the self-diffusion factor over mu
      t.fV = 3*sqrt(PI*KB*s.W/NA)/(8*PI*pow(s.sigma, 2.0))/t.mu;
      t.zrot = s.Z298*sp_fzrot(s.kbOveps, 298);
      t.isk = 1.0/sqrt(s.kbOveps);
      for (int j = 0; j < m.nSpec; j++) {
         const DSpec &o = m.sp[j];
         DPair &p = m.pr[i][j];
         // Wilke's rule: Phi = (1 + sqrt(mu_i/mu_j) (W_j/W_i)^(1/4))^2/sqrt(8 (1 + W_i/W_j))
         p.w4 = pow(o.W/s.W, 0.25);
         p.iw8 = 1.0/sqrt(8*(1 + s.W/o.W));
         // Species.inl:225-288: binary diffusivity D = 3 sqrt(2 PI KB^3 T^3 NA/W_ij)/(16 PI P sigma_ij^2 omega)
         double xi = 1.0;
         if ((s.mu*o.mu == 0.0) && (s.mu + o.mu != 0.0)) {
            const DSpec &a = (s.mu != 0.0) ? s : o, &b = (s.mu != 0.0) ? o : s;   // polar, non-polar
            const double mup = a.mu/sqrt(4*PI*EPS0*KB*pow(a.sigma, 3.0)/a.kbOveps);
            const double alp = b.alpha/pow(b.sigma, 3.0);
            xi = 1 + 0.25*mup*alp*sqrt(b.kbOveps/a.kbOveps);
         }
         const double sigmaij = 0.5*(s.sigma + o.sigma)*pow(xi, -1./6);
         const double invWij = (s.W + o.W)/(s.W*o.W);
         p.kT = sqrt(s.kbOveps*o.kbOveps)/(xi*xi);
         p.iD = 16*PI*sigmaij*sigmaij/(3*sqrt(2*PI*pow(KB, 3.0)*NA*invWij));
      }
   }
}

// ---------------------------------------------------------------- mixture --
// The mixture policy: NS species, CP = calorically perfect gas (NS == 1).
template<int NS_, bool CP_>
struct Mix {
   static constexpr int  NS  = NS_;
   static constexpr int  NEQ = NS_ + 4;
   static constexpr bool CP  = CP_;

   HD static double MolarWeightFromY(const DMix &m, const double *Y)
   {
      if (CP) return RGAS/m.R;
      double W = 0.0;
      for (int i = 0; i < NS; i++) W += quot(Y[i], m.sp[i].W, m.sp[i].iW);
      return 1.0/W;
   }
   HD static double MolarWeightFromX(const DMix &m, const double *X)
   {
      if (CP) return RGAS/m.R;
      double W = 0.0;
      for (int i = 0; i < NS; i++) W += X[i]*m.sp[i].W;
      return W;
   }
   HD static void MolarFractions(const DMix &m, double *X, double MixW, const double *Y)
   {
      if (CP) { X[0] = Y[0]; return; }
      for (int i = 0; i < NS; i++) X[i] = quot(Y[i]*MixW, m.sp[i].W, m.sp[i].iW);
   }
   HD static void MassFractions(const DMix &m, double *Y, double MixW, const double *X)
   {
      if (CP) { Y[0] = X[0]; return; }
      const double iMixW = 1.0/MixW;
      for (int i = 0; i < NS; i++) Y[i] = quot(X[i]*m.sp[i].W, MixW, iMixW);
   }
   HD static double SpeciesW(const DMix &m, int i) { return CP ? RGAS/m.R : m.sp[i].W; }
   HD static double Rho(const DMix &m, double P, double T, double MixW)
   {
      if (CP) return P/(m.R*T);
      return P*MixW*m.iMixWRef/T;
   }
   HD static double HeatCapacity(const DMix &m, double Tn, const double *Y)
   {
      if (CP) return m.gamma/(m.gamma - 1)*m.R;
      const double T = Tn*m.TRef;
      const double Tinv = 1.0/T;
      double cp = 0.0;
      species_loop<NS>(m, T, [&](int i, const DSpec &s, const double *c) { cp += Y[i]*poly_cp(s, c, T, Tinv); });
      return cp*m.iCpRef;
   }
   HD static double SpeciesEnthalpy(const DMix &m, int i, double T)
   {
      if (CP) return m.gamma/(m.gamma - 1)*m.R*T;
      return sp_enthalpy(m.sp[i], T*m.TRef)*m.ieRef;
   }
   // all species at once (the face enthalpies of the diffusion)
   HD static void SpeciesEnthalpies(const DMix &m, double *h, double Tn, const double *tab = nullptr)
   {
      if (CP) { h[0] = m.gamma/(m.gamma - 1)*m.R*Tn; return; }
      const double T = Tn*m.TRef, Tinv = 1.0/T, logT = log(T);
      species_loop<NS>(m, T, [&](int i, const DSpec &s, const double *c) { h[i] = poly_enthalpy(s, c, T, Tinv, logT)*m.ieRef; }, tab);
   }
   HD static double InternalEnergy(const DMix &m, double Tn, const double *Y)
   {
      if (CP) return Tn*m.R/(m.gamma - 1.0);
      const double T = Tn*m.TRef;
      const double Tinv = 1.0/T, logT = log(T), RT = RGAS*T;
      double e = 0.0;
      species_loop<NS>(m, T, [&](int i, const DSpec &s, const double *c) {
         e += Y[i]*(poly_enthalpy(s, c, T, Tinv, logT) - quot(RT, s.W, s.iW));
      });
      return e*m.ieRef;
   }
   // MultiComponent.inl:187-210; iters (optional) receives the Newton count
   HD static double TFromInternalEnergy(const DMix &m, double e0, double T, const double *Y, int *iters = nullptr)
   {
      if (CP) { if (iters) *iters = 0; return e0*(m.gamma - 1.0)/m.R; }
      double dfdT = 1.0;
      int j = 0;
      while (j < 1000) {
         const double f = e0 - InternalEnergy(m, T, Y);
         if (fabs(f/dfdT) < 1e-8) break;
         const double Td = T*m.TRef, Tinv = 1.0/Td;
         dfdT = 0.0;
         species_loop<NS>(m, Td, [&](int i, const DSpec &s, const double *c) {
            dfdT += Y[i]*(poly_cp(s, c, Td, Tinv) - s.rOvW)*m.iCpRef;
         });
         T += f/dfdT;
         j++;
      }
      if (iters) *iters = j;
      return T;
   }
   HD static double TFromRhoAndP(const DMix &m, double rho, double MixW, double P)
   {
      if (CP) return P*MixW/(rho*RGAS);
      return P*MixW*m.iMixWRef/rho;
   }
   HD static double PFromRhoAndT(const DMix &m, double rho, double MixW, double T)
   {
      if (CP) return rho*RGAS*T/MixW;
      return rho*T/(MixW*m.iMixWRef);
   }
   HD static double ConstVisc(const DMix &m, double T)
   {
      if (m.viscModel == VISC_CONSTANT) return m.constVisc;
      if (m.viscModel == VISC_POWERLAW) return m.plVRef*pow((T/m.plTRef), 0.7);
      return (m.suVRef*pow((T/m.suTRef), 1.5))*((m.suTRef + m.suSRef)/(T + m.suSRef));
   }
   // Viscosity (Wilke), heat conductivity, diffusivities and the speed of
   // sound of one cell (MultiComponent.inl:215-330, Species.inl:193-357).  Formed
   // together they share sqrt(T), the species viscosities (which the
   // conductivities need too), the heat capacities (which the speed of sound
   // needs too) and the factors of derive_transport: one quotient per pair and
   // collision integral, no pow, and one square root per species.  Bound by
   // FP64 issue when each property formed its own factors with pow and sqrt
   // (4200 FP64 instructions per cell); the fused stage update of 160^3 air
   // went from 2.14 to 0.52 ms, 3.8 TB/s of its 480 B per cell, with Newton
   // and properties together.
   HD static void Transport(const DMix &m, double Pn, double Tn, double MixW, const double *X, const double *Y,
                            double &muOut, double &lamOut, double *Di, double &SoS)
   {
      if (CP) {
         const double cp = m.gamma/(m.gamma - 1)*m.R;
         const double visc = ConstVisc(m, Tn);
         muOut = visc;
         lamOut = cp/m.Prandtl*visc;
         Di[0] = 0.0;
         SoS = sqrt(m.gamma*m.R*Tn);
         return;
      }
      const double T = Tn*m.TRef, P = Pn*m.PRef;
      const double sT = sqrt(T), Tinv = 1.0/T, isT = sT*Tinv;
      double sk[NS], isk[NS], cpm = 0.0, la = 0.0, lb = 0.0;
      species_loop<NS>(m, T, [&](int i, const DSpec &s, const double *c) {
         const DTran &tr = m.tr[i];
         const double Ts = T*s.kbOveps;
         const double on = omega_mu_num(Ts), od = omega_mu_den(Ts);
         const double mu = tr.mu*sT*od/on;
         sk[i] = sqrt(mu);
         isk[i] = 1.0/sk[i];
         const double cp = poly_cp(s, c, T, Tinv);
         cpm += Y[i]*cp;
         double lam;
         if (s.geom == GEOM_ATOM) {
            lam = 15.0/4*mu*s.rOvW;
         } else {
            const bool lin = (s.geom == GEOM_LINEAR);
            const double CvROvR = lin ? 1.0 : 1.5;
            const double CvT = 1.5*RGAS, CvR = CvROvR*RGAS;
            const double CvV = cp*s.W - (lin ? 3.5 : 4.0)*RGAS;
            const double fV = tr.fV*omega_D_den(Ts)*on/(omega_D_num(Ts)*od);
            const double r1 = tr.isk*isT, r2 = r1*r1;      // sqrt(1/T*), 1/T*
            const double fz = 1 + 0.5*PI15*r1 + (2 + 0.25*PI*PI)*r2 + PI15*(r2*r1);
            const double A = 2.5 - fV;
            // A/B with B = zrot/fz + 2/PI (5/3 CvR/R + fV)
            const double AB = A*fz/(tr.zrot + fz*(2/PI*(5./3*CvROvR + fV)));
            const double fT = 2.5*(1. - 2*CvR/(PI*CvT)*AB);
            const double fR = fV*(1. + 2/PI*AB);
            lam = mu*s.iW*(fT*CvT + fR*CvR + fV*CvV);
         }
         la += X[i]*lam;
         lb += X[i]/lam;
      });
      lamOut = 0.5*(la + 1.0/lb)*m.ilamRef;
      double mu = 0.0;
#pragma unroll
      for (int i = 0; i < NS; i++) {
         double den = 0.0;
#pragma unroll
         for (int j = 0; j < NS; j++) {
            if (j == i) { den += X[j]; continue; }         // Phi = 1
            const double phi = 1 + sk[i]*isk[j]*m.pr[i][j].w4;
            den += X[j]*(phi*phi*m.pr[i][j].iw8);
         }
         mu += X[i]*(sk[i]*sk[i])/den;
      }
      muOut = mu*m.imuRef;
#pragma unroll
      for (int i = 0; i < NS; i++) Di[i] = 0.0;
      const double PT = P*(Tinv*isT);                      // P/T^(3/2)
#pragma unroll
      for (int i = 0; i < NS; i++)
#pragma unroll
         for (int j = 0; j < i; j++) {
            const DPair &p = m.pr[i][j];
            const double Ts = T*p.kT;
            const double invDij = p.iD*PT*omega_D_num(Ts)/omega_D_den(Ts);
            Di[i] += X[j]*invDij;
            Di[j] += X[i]*invDij;
         }
#pragma unroll
      for (int i = 0; i < NS; i++) {
         double num = 0.0;
#pragma unroll
         for (int j = 0; j < NS; j++)
            if (j != i) num += X[j]*m.sp[j].W;
         Di[i] = num/(MixW*Di[i])*m.iDiRef;
      }
      const double cp = cpm*m.iCpRef, Wr = MixW*m.iMixWRef;
      SoS = SpeedOfSound(m, Tn, cp/(cp - 1.0/Wr), MixW);
   }
   HD static double Gamma(const DMix &m, double T, double MixW, const double *Y)
   {
      if (CP) return m.gamma;
      const double cp = HeatCapacity(m, T, Y);
      const double Wr = MixW*m.iMixWRef;
      return cp/(cp - 1.0/Wr);
   }
   HD static double SpeedOfSound(const DMix &m, double T, double gamma, double MixW)
   {
      if (CP) return sqrt(gamma*m.R*T);
      return sqrt(gamma*T/(MixW*m.iMixWRef));
   }
   HD static double dpde(double rho, double gamma) { return rho*(gamma - 1); }
   HD static void dpdrhoi(const DMix &m, double *d, double gamma, double Tn, const double *Y)
   {
      if (CP) { d[0] = m.R*Tn; return; }
      const double T = Tn*m.TRef;
      const double Tinv = 1.0/T, logT = log(T), RT = RGAS*T;
      double e = 0.0;
      species_loop<NS>(m, T, [&](int i, const DSpec &s, const double *c) {
         d[i] = poly_enthalpy(s, c, T, Tinv, logT) - quot(RT, s.W, s.iW);
         e += Y[i]*d[i];
      });
      for (int i = 0; i < NS; i++) d[i] = (quot(RT, m.sp[i].W, m.sp[i].iW) + (gamma - 1)*(e - d[i]))*m.ieRef;
   }

   // Reaction.inl:34-42: Kf = A T^n exp(-EovR/T), formed as
   // A exp(n ln T - EovR/T) from logT = ln T: one exponential in place of
   // pow and exp, the same function up to rounding
   HD static double RateCoeff(double A, float n, float EovR, double T, double logT)
   {
      double arg = 0.0;
      if (n != 0.0) arg = (double)n*logT;
      if (fabs((double)EovR) > 1e-5) arg -= (double)EovR/T;
      return A*exp(arg);
   }
   // MultiComponent.inl:371-417 with Reaction.inl:82-228 (no fall-off), on
   // species arrays w (rates), C (concentrations) and G (Gibbs energies) of
   // type A: per-thread arrays, or SpeciesCol columns of a shared array
   template<class A>
   HD static void ProductionRatesIn(const DMix &m, A w, A C, A G, double rhon, double Pn, double Tn, const double *Y)
   {
      const double T = Tn*m.TRef;
      const double P = Pn*m.PRef;
      const double rho = rhon*m.rhoRef;
      const double logT = log(T), Tinv = 1.0/T;
      for (int i = 0; i < NS; i++) {
         w[i] = 0.0;
         C[i] = Y[i]*rho/m.sp[i].W;
         G[i] = poly_free_enthalpy(cp_range(m.sp[i], T), T, Tinv, logT);
      }
      const double logRP = log(RGAS/P);
      for (int k = 0; k < m.nReac; k++) {
         const DReac &r = m.rc[k];
         const double Kf = RateCoeff(r.A, r.n, r.EovR, T, logT);
         double a = 1.0;
         for (int i = 0; i < r.Ne; i++) {
            const int ind = r.ed_ind[i];
            a *= conc_pow(C[ind], r.ed_nu[i]);
         }
         double Kb = 0.0, b = 1.0;
         if (r.has_backward) {
            double sumNu = 0.0, sumNuG = 0.0;
            for (int i = 0; i < r.Ne; i++) { sumNu -= r.ed_nu[i]; sumNuG -= r.ed_nu[i]*G[r.ed_ind[i]]; }
            for (int i = 0; i < r.Np; i++) { sumNu += r.pd_nu[i]; sumNuG += r.pd_nu[i]*G[r.pd_ind[i]]; }
            const double lnKc = -sumNuG - sumNu*(logT + logRP);
            Kb = Kf*exp(-lnKc);
            for (int i = 0; i < r.Np; i++) {
               const int ind = r.pd_ind[i];
               b *= conc_pow(C[ind], r.pd_nu[i]);
            }
         }
         double R = Kf*a - Kb*b;
         if (r.kind == REAC_THIRDB) {
            double c = 1.0;
            if (r.Ntb > 0) {
               c = P/(RGAS*T);
               for (int i = 0; i < r.Ntb; i++) c += C[r.tb_ind[i]]*(r.tb_eff[i] - 1.0);
            }
            R = c*(Kf*a - Kb*b);
         }
         for (int i = 0; i < r.Ne; i++) w[r.ed_ind[i]] -= r.ed_nu[i]*R;
         for (int i = 0; i < r.Np; i++) w[r.pd_ind[i]] += r.pd_nu[i]*R;
      }
      for (int i = 0; i < NS; i++) w[i] *= m.sp[i].W*m.iwiRef;
   }
   HD static void ProductionRates(const DMix &m, double *w, double rhon, double Pn, double Tn, const double *Y)
   {
      if (CP) { w[0] = 0.0; return; }
      double G[NS], C[NS];
      ProductionRatesIn<double *>(m, w, C, G, rhon, Pn, Tn, Y);
   }
};

} // namespace htr
