// chem_wave.hpp -- implicit chemistry with a wave per cell: the integration of
// chem.hip (same operations, same order, same results to the bit) for 64 lanes
// per cell.
//
// What bounds a cell's integration is latency: a step is a chain of small
// dependent pieces (right-hand sides, factorisation, four solves), a cell
// takes 100 to 800 steps, and a launch ends with its slowest cell.  So
//   - the solver vectors live in registers, lane i holding component i; sums
//     over species are formed in order from v_readlane operands, not from LDS;
//   - the mechanism is read field by field with consecutive lanes on
//     consecutive words (DMix::k*, rows, cpT); no read depends on another;
//   - the matrix rows are loaded into registers before they are used, with
//     the row interchanges folded into one permutation;
//   - the central-difference Jacobian, 2 nEq right-hand sides, is shared by
//     the four waves of the block.  The only thing one right-hand side hands
//     to the next is the temperature its Newton ends at, so the first wave
//     runs the Newtons, in the reference's order, six at a time, while the
//     other three form the production rates of the columns before, each the
//     pair of one column at once.
// 30 species, 180 reactions, against 64 lanes of the group kernel before:
// 12^3 cells, FP64, central differences 1033 -> 197 ms; 20^3 cells, FP32 and
// refinement, analytic Jacobian 576 -> 155 ms; 32^3 cells over 1e-5 s 5153 -> 1686
// ms (FP64, differences), 1435 -> 374 ms (FP64, analytic), 1298 -> 349 ms (refined,
// analytic: the refinement's own share of that is 7 %).  Still bound by latency: of 220000 cycles of a step with the
// analytic Jacobian the factorisation takes 45000, the solves 73000, the
// Jacobian 40000; with differences the Newtons' chain takes 184000 of 475000.
#pragma once
#include "common.hpp"
#include "kernels.hpp"

namespace htr {

// LDS synchronisation of a lane group inside one wave: LDS operations of a
// wave complete in order; the fences keep the compiler from moving them
// across and wait for the outstanding ones.
__device__ __forceinline__ void gsync()
{
   __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
   __builtin_amdgcn_wave_barrier();
   __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
}

// value of lane l (uniform) of the wave
__device__ __forceinline__ double rdlane(double x, int l)
{
   const long long b = __double_as_longlong(x);
   const int lo = __builtin_amdgcn_readlane((int)b, l);
   const int hi = __builtin_amdgcn_readlane((int)(b >> 32), l);
   return __longlong_as_double(((long long)hi << 32) | (long long)(unsigned)lo);
}

__device__ __forceinline__ float rdlane(float x, int l)
{
   return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(x), l));
}

// maximum over the wave, in every lane (NaN lanes do not count)
__device__ __forceinline__ double wave_dmax(double x)
{
#ifdef __HIP_DEVICE_COMPILE__
   // row shifts, then the row broadcasts: lane 63 ends with the maximum; a lane
   // with no source keeps its own value
#define HTR_DPP_MAX(ctrl)                                                                        \
   {                                                                                             \
      const long long b = __double_as_longlong(x);                                               \
      const int lo = __builtin_amdgcn_update_dpp((int)b, (int)b, ctrl, 0xf, 0xf, false);         \
      const int hi = __builtin_amdgcn_update_dpp((int)(b >> 32), (int)(b >> 32), ctrl, 0xf, 0xf, false); \
      x = fmax(x, __longlong_as_double(((long long)hi << 32) | (long long)(unsigned)lo));        \
   }
   HTR_DPP_MAX(0x111) HTR_DPP_MAX(0x112) HTR_DPP_MAX(0x114) HTR_DPP_MAX(0x118)
   HTR_DPP_MAX(0x142) HTR_DPP_MAX(0x143)
#undef HTR_DPP_MAX
#else
   for (int o = 32; o > 0; o >>= 1) x = dmax(x, __shfl_xor(x, o, 64));
#endif
   return rdlane(x, 63);
}

// maximum of a 32-bit key: one instruction a step
__device__ __forceinline__ uint32_t wave_umax(uint32_t x)
{
#ifdef __HIP_DEVICE_COMPILE__
#define HTR_DPP_MAX(ctrl) x = max(x, (uint32_t)__builtin_amdgcn_update_dpp((int)x, (int)x, ctrl, 0xf, 0xf, false));
   HTR_DPP_MAX(0x111) HTR_DPP_MAX(0x112) HTR_DPP_MAX(0x114) HTR_DPP_MAX(0x118)
   HTR_DPP_MAX(0x142) HTR_DPP_MAX(0x143)
#undef HTR_DPP_MAX
#else
   for (int o = 32; o > 0; o >>= 1) x = max(x, __shfl_xor(x, o, 64));
#endif
   return (uint32_t)__builtin_amdgcn_readlane((int)x, 63);
}

// upper word of a number >= 0: ordered as the numbers, but for equal words
__device__ __forceinline__ uint32_t upper_word(double x) { return (uint32_t)(__double_as_longlong(x) >> 32); }
__device__ __forceinline__ uint32_t upper_word(float x) { return (uint32_t)__float_as_int(x); }

// lane t: x of lane t - 1, and x0 in lane 0
__device__ __forceinline__ double wave_shift(double x, double x0)
{
#ifdef __HIP_DEVICE_COMPILE__
   const long long b = __double_as_longlong(x), f = __double_as_longlong(x0);
   const int lo = __builtin_amdgcn_update_dpp((int)f, (int)b, 0x138, 0xf, 0xf, false);            // wave_shr:1
   const int hi = __builtin_amdgcn_update_dpp((int)(f >> 32), (int)(b >> 32), 0x138, 0xf, 0xf, false);
   return __longlong_as_double(((long long)hi << 32) | (long long)(unsigned)lo);
#else
   const double up = __shfl_up(x, 1, 64);
   return (threadIdx.x & 63) == 0 ? x0 : up;
#endif
}

// LDS add without a result: the LDS unit takes a wave's operations in order, so
// several to one address add up in program order without waiting for each other
__device__ __forceinline__ void lds_add(double *p, double v)
{
#ifdef __HIP_DEVICE_COMPILE__
   __hip_atomic_fetch_add(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
#else
   *p += v;
#endif
}

// power of two nearest to 1/a (exact scaling)
__device__ __forceinline__ double pow2_inv(double a)
{
   if (!(a > 0.0) || !(a < 1.0e308)) return 1.0;
   // a = m 2^e with m in [0.5, 1): e from the biased exponent (normal a)
   const int be = (int)((__double_as_longlong(a) >> 52) & 0x7ff);
   if (be == 0) return 1.0;
   return ldexp(1.0, -(be - 1022));
}

constexpr int CHEM_FD_WAVES = 4;               // waves of a block with the central-difference Jacobian

// LDS of one cell, in doubles from its base
template<class MX, int PREC, bool AJ>
struct WaveLayout {
   static constexpr int NS = MX::NS, N = MX::NEQ;
   int CG, RR, EV, IND, MISC, U, total;        // J at 0
   __host__ __device__ WaveLayout(int nR, int maxEd, int maxPd)
   {
      int o = N*N;
      CG = o;   o += 2*NS;                     // concentrations and Gibbs energies
      RR = o;   o += nR + 1;                   // rates of progress, and a 0
      EV = o;   o += AJ ? 3*NS : 5*2*N + 2*N;  // analytic: dG/dT, rhoRef/W, Y; differences: rho, 1/rho, W, e, T of each
                                               // evaluation, x, Conserved_t
      IND = o;  o += (N + 1)/2;                // row permutation of the factors (int)
      MISC = o; o += 2;                        // queue slot, command (int)
      U = o;                                   // the factors; while the Jacobian is formed, its scratch
      const int fac = (PREC == HTR_CHEM_FP64) ? N*N : (N*N + 1)/2;
      const int scr = AJ ? (2 + maxEd + maxPd)*(nR + 1) : (CHEM_FD_WAVES - 1)*2*(2*NS + nR + 1);
      total = U + (fac > scr ? fac : scr);
   }
};

template<class MX, int PREC, bool AJ>
struct ChemWave {
   static constexpr int NS = MX::NS, N = MX::NEQ;
   static_assert(NS <= 32 && N <= 64, "a species per lane of half a wave, a matrix row per lane");
   using Lay = WaveLayout<MX, PREC, AJ>;
   using R = typename std::conditional<PREC == HTR_CHEM_FP64, double, float>::type;

   const DMix &m;
   const Lay  &L;
   double     *S;             // LDS of the cell
   const int   lane, sp;      // the lane's species, in both halves of the wave
   const int   nR;
   // the lane's species
   double W, iW, rOvW, tHi, tLo;
   int    nrow, range;
   double c[12];              // its coefficients in the range of Tc (or of the last sel())
   // enthalpy minus R T/W of the lane's species at the temperature guess Tc
   double E, Tc, Trc, iTrc, logTc;
   double T;                  // temperature guess (uniform)
   double ct;                 // component `lane` of Conserved_t
   bool   jac_valid, lu64;    // FP32_IR: a fallback factorises in the Jacobian's place

   __device__ __forceinline__ ChemWave(const DMix &m_, const Lay &L_, double *S_, int lane_)
      : m(m_), L(L_), S(S_), lane(lane_), sp((lane_ & 31) < NS ? (lane_ & 31) : NS - 1), nR(m_.nReac)
   {
      const DSpec &q = m.sp[sp];
      W = q.W; iW = q.iW; rOvW = q.rOvW; tHi = q.tHi; tLo = q.tLo;
      nrow = m.spr_ptr[sp + 1] - m.spr_ptr[sp];
      range = -1;
      E = Trc = iTrc = logTc = T = ct = 0.0;
      Tc = -1.0;
      jac_valid = lu64 = false;
   }

   __device__ __forceinline__ double *Jm() const { return S; }
   __device__ __forceinline__ int *ind() const { return reinterpret_cast<int*>(S + L.IND); }
   // a component of the momentum or energy of the lane-held vector x, of every lane
   __device__ __forceinline__ static double comp(double x, int i) { return rdlane(x, i); }

   // t of species 0, 1, .. added up in order.  The operands are read eight
   // ahead of their use, in program order: left alone the compiler reads each
   // right before its addition, through one pair of scalar registers, and the
   // wave waits for every one of them (25 instead of 12 cycles a term)
   __device__ __forceinline__ static double lane_sum(double t)
   {
      constexpr int D = NS < 8 ? NS : 8;
      double u[NS], a = 0.0;
#pragma unroll
      for (int i = 0; i < D; i++) u[i] = rdlane(t, i);
#pragma unroll
      for (int i = 0; i < NS; i++) {
         a += u[i];
         if (i + D < NS) u[i + D] = rdlane(t, i + D);
         __builtin_amdgcn_sched_barrier(0);
      }
      return a;
   }

   __device__ __forceinline__ static double clip_y(double y) { y = dmax(y, 1e-60); return dmin(y, 1.0); }

   // coefficients of the lane's species at Tr
   __device__ __forceinline__ void sel(double Tr)
   {
      const int r = Tr > tHi ? 0 : Tr > tLo ? 1 : 2;
      if (r != range) {
         range = r;
#pragma unroll
         for (int k = 0; k < 12; k++) c[k] = m.cpT[r][k][sp];
      }
   }

   __device__ __forceinline__ void thermo(double Tn)
   {
      Tc = Tn;
      Trc = Tn*m.TRef;
      iTrc = 1.0/Trc;
      logTc = log(Trc);
      sel(Trc);
      E = poly_enthalpy(*this, c, Trc, iTrc, logTc) - quot(RGAS*Trc, W, iW);
   }

   // MultiComponent.inl:187-210 from the guess T; Y of the lane's species
   __device__ __forceinline__ void newton(double e0, double Y)
   {
      double dfdT = 1.0;
      for (int j = 0; ; j++) {
         if (Tc != T) thermo(T);       // the last right-hand side ended at this T
         if (j == 1000) break;
         const double f = e0 - lane_sum(Y*E)*m.ieRef;
         if (fabs(f/dfdT) < 1e-8) break;
         dfdT = lane_sum(Y*(poly_cp(*this, c, Trc, iTrc) - rOvW)*m.iCpRef);
         T += f/dfdT;
      }
   }

   // what the reactions need of one evaluation (uniform)
   struct Eval { double Tr, iTr, logT, lRP, ctot; };

   // Concentrations and Gibbs energies of NE evaluations into CG; with two, the
   // halves of the wave take one each and T, rho, MixW, Y are of the lane's half
   template<int NE>
   __device__ __forceinline__ void species(double *CG, Eval *ev, double Tn, double Tr, double iTr, double logT,
                                           double rho, double MixW, double Y)
   {
      const double P = MX::PFromRhoAndT(m, rho, MixW, Tn);
      const double Pr = P*m.PRef, rr = rho*m.rhoRef;
      const double lRP = logT + log(RGAS/Pr);
      const double ctot = Pr/(RGAS*Tr);
      sel(Tr);
      if ((lane & 31) < NS && (NE == 2 || lane < 32)) {
         double *q = CG + (NE == 2 ? (lane >> 5)*2*NS : 0);
         q[sp] = quot(Y*rr, W, iW);
         q[NS + sp] = poly_free_enthalpy(c, Tr, iTr, logT);
      }
#pragma unroll
      for (int e = 0; e < NE; e++) {
         ev[e].Tr = rdlane(Tr, 32*e); ev[e].iTr = rdlane(iTr, 32*e); ev[e].logT = rdlane(logT, 32*e);
         ev[e].lRP = rdlane(lRP, 32*e); ev[e].ctot = rdlane(ctot, 32*e);
      }
      gsync();
   }

   // Rates of progress (Reaction.inl:34-228) of NE evaluations, a lane per
   // reaction, both evaluations in the lane
   template<int NE>
   __device__ __forceinline__ void progress(double *RR, const double *CG, const Eval *ev)
   {
      const bool unit = m.unitNu != 0;
      const int mE = m.maxEd, mP = m.maxPd, mT = m.maxTb;
      DRate nx = m.rate[min(lane, max(nR - 1, 0))];
      for (int k0 = 0; k0 < nR; k0 += 64) {
         const int k = min(k0 + lane, nR - 1);
         const DRate rt = nx;
         nx = m.rate[min(k0 + 64 + lane, nR - 1)];             // the next round's, in flight
         const uint32_t info = rt.info, eid = rt.eid, pid = rt.pid;
         const double A = rt.A, sumNu = rt.sumNu, rn = (double)rt.n, eR = (double)rt.EovR;
         const int ne = (info >> 16) & 15, np = (info >> 20) & 15, nt = (info >> 24) & 15;
         const bool hasE = fabs(eR) > 1e-5, back = (info >> 28) & 1;
         double a[NE], b[NE], g[NE];
#pragma unroll
         for (int e = 0; e < NE; e++) { a[e] = b[e] = 1.0; g[e] = 0.0; }
         auto term = [&](bool educt, int i) {
            const int id = ((educt ? eid : pid) >> 8*i) & 255;
            const bool in = i < (educt ? ne : np);
            if (unit) {                // info has the coefficients of 2
               const bool two = (info >> (educt ? i : 4 + i)) & 1;
#pragma unroll
               for (int e = 0; e < NE; e++) {
                  const double C = CG[e*2*NS + id], G = CG[e*2*NS + NS + id];
                  const double p = two ? C*C : C, nG = two ? G + G : G;
                  double &ab = educt ? a[e] : b[e];
                  ab = in ? ab*p : ab;
                  g[e] = in ? (educt ? g[e] - nG : g[e] + nG) : g[e];
               }
            } else if (in) {
               const float nu = educt ? m.kEnu[i][k] : m.kPnu[i][k];
#pragma unroll
               for (int e = 0; e < NE; e++) {
                  const double C = CG[e*2*NS + id], G = CG[e*2*NS + NS + id];
                  const double p = conc_pow(C, nu);
                  if (educt) { a[e] *= p; g[e] -= nu*G; }
                  else       { b[e] *= p; g[e] += nu*G; }
               }
            }
         };
         if (unit) {
#pragma unroll
            for (int i = 0; i < MAX_ED; i++) if (i < mE) term(true, i);
#pragma unroll
            for (int i = 0; i < MAX_PD; i++) if (i < mP) term(false, i);
         } else {
#pragma unroll 1
            for (int i = 0; i < mE; i++) term(true, i);
#pragma unroll 1
            for (int i = 0; i < mP; i++) term(false, i);
         }
#pragma unroll
         for (int e = 0; e < NE; e++) {
            double arg = rn*ev[e].logT;
            if (hasE) arg -= quot(eR, ev[e].Tr, ev[e].iTr);
            const double Kf = A*exp(arg);
            const double lnKc = -g[e] - sumNu*ev[e].lRP;
            double Kbb = 0.0;
            if (back) { const double Kb = Kf*exp(-lnKc); Kbb = Kb*b[e]; }
            double q = Kf*a[e] - Kbb;
            if (mT > 0) {
               double x = ev[e].ctot;
               for (int i = 0; i < mT; i++)
                  if (i < nt) x += CG[e*2*NS + m.kTid[i][k]]*(m.kTeff[i][k] - 1.0);
               if (nt > 0) q = x*q;
            }
            if (k0 + lane < nR) RR[e*(nR + 1) + k] = q;
         }
      }
      if (lane < NE) RR[lane*(nR + 1) + nR] = 0.0;             // what the padding of the rows reads
      gsync();
   }

   // production rate of the lane's species; with two evaluations, of the lane's half
   template<int NE>
   __device__ __forceinline__ double production(const double *RR)
   {
      const double *q = RR + (NE == 2 ? (lane >> 5)*(nR + 1) : 0);
      const int n = m.nRows;
      double w = 0.0;
      if (m.unitNu) {
         // eight words of two entries a batch, the next batch in flight: 2.4 KB
         // for the 30-species mechanism, which stays in the vector cache (16
         // bytes an entry did not)
         uint32_t r[8], nx[8];
#pragma unroll
         for (int k = 0; k < 8; k++) nx[k] = m.prow[k][sp];
         for (int k0 = 0; k0 < n; k0 += 16) {
#pragma unroll
            for (int k = 0; k < 8; k++) { r[k] = nx[k]; nx[k] = m.prow[k0/2 + 8 + k][sp]; }
            double t[16];
#pragma unroll
            for (int k = 0; k < 16; k++) {
               const uint32_t v = r[k/2] >> 16*(k & 1);
               const double a = q[v & 0x1ff], b = (v & 0x2000) ? a + a : a;
               t[k] = (v & 0x4000) ? -b : b;
            }
#pragma unroll
            for (int k = 0; k < 16; k++) w += t[k];
         }
      } else {
         const DRow *row = m.rows() + sp;
         for (int k = 0; k < n; k++) {
            const DRow r = row[k*NS];
            const double t = w + r.nu*q[r.info & 0xffff];
            w = (k < nrow) ? t : w;
         }
      }
      return w*(W*m.iwiRef);
   }

   // ImplicitSolver::rhs (chem.hpp:53-93) of the lane-held x; the lane's component
   __device__ __forceinline__ double rhs(double x)
   {
      const double rho = lane_sum(x);
      const double irho = 1.0/rho;
      const double Y = clip_y(irho*x);
      const double MixW = 1.0/lane_sum(quot(Y, W, iW));
      double k2 = 0.0;
#pragma unroll
      for (int i = 0; i < 3; i++) { const double v = comp(x, NS + i)*irho; k2 += v*v; }
      const double e = comp(x, NS + 3)*irho - 0.5*k2;
      newton(e, Y);
      Eval ev[1];
      species<1>(S + L.CG, ev, T, Trc, iTrc, logTc, rho, MixW, Y);
      progress<1>(S + L.RR, S + L.CG, ev);
      const double w = production<1>(S + L.RR);
      return (lane < NS) ? w + ct : ct;
   }

   // ---- central-difference Jacobian (math_utils.hpp:249-269) --------------------
   // Column j by evaluations 2 j (x_j + h) and 2 j + 1 (x_j - h).  Called by
   // every wave of the block between the same barriers; x and Conserved_t of
   // the cell in LDS.  wv: the wave.
   __device__ __forceinline__ static double moved(double xj, int sign)
   {
      const double h = xj*1.0e-6 + 1.0e-14;
      return sign ? xj - h : xj + h;
   }

   __device__ __forceinline__ void jacobian_columns(int wv)
   {
      constexpr int NE2 = 2*N, COLS = CHEM_FD_WAVES - 1;
      double *erho = S + L.EV, *eirho = erho + NE2, *eW = eirho + NE2, *ee = eW + NE2, *eT = ee + NE2;
      const double *X = eT + NE2, *CT = X + N;
      // density, mixture weight and internal energy of every evaluation, which
      // no temperature enters: a lane each
      for (int e = wv*64 + lane; e < NE2; e += CHEM_FD_WAVES*64) {
         const int j = e >> 1;
         const double xj = moved(X[j], e & 1);
         double rho = 0.0, sW = 0.0, k2 = 0.0;
#pragma unroll
         for (int i = 0; i < NS; i++) rho += (i == j) ? xj : X[i];
         const double irho = 1.0/rho;
#pragma unroll 2
         for (int i = 0; i < NS; i++) sW += quot(clip_y(irho*((i == j) ? xj : X[i])), m.sp[i].W, m.sp[i].iW);
#pragma unroll
         for (int i = 0; i < 3; i++) { const double v = ((NS + i == j) ? xj : X[NS + i])*irho; k2 += v*v; }
         erho[e] = rho;
         eirho[e] = irho;
         eW[e] = 1.0/sW;
         ee[e] = ((NS + 3 == j) ? xj : X[NS + 3])*irho - 0.5*k2;
      }
      __syncthreads();
      const double xs = X[sp];
      for (int g = 0; g <= (N + COLS - 1)/COLS; g++) {
         if (wv == 0) {
#pragma unroll 1
            for (int e = 2*COLS*g; e < min(2*COLS*(g + 1), NE2); e++) {
               const double x = (sp == (e >> 1)) ? moved(xs, e & 1) : xs;
               newton(ee[e], clip_y(eirho[e]*x));
               if (lane == 0) eT[e] = T;
            }
         } else {
            const int j = COLS*(g - 1) + wv - 1;
            if (g > 0 && j < N) {
               double *CG = S + L.U + (wv - 1)*2*(2*NS + nR + 1), *RR = CG + 4*NS;
               const int e = 2*j + (lane >> 5);
               const double x = (sp == j) ? moved(xs, e & 1) : xs;
               const double Tn = eT[e], Tr = Tn*m.TRef;
               Eval ev[2];
               species<2>(CG, ev, Tn, Tr, 1.0/Tr, log(Tr), erho[e], eW[e], clip_y(eirho[e]*x));
               progress<2>(RR, CG, ev);
               const double w = production<2>(RR) + CT[sp];
               const double wm = __shfl_xor(w, 32, 64);
               const double xj = X[j], h = xj*1.0e-6 + 1.0e-14;
               const double hp = (xj + h) - xj, hm = xj - (xj - h);
               if (lane < NS) S[lane + j*N] = (w - wm)/(hp + hm);
               if (lane < 4) S[NS + lane + j*N] = (CT[NS + lane] - CT[NS + lane])/(hp + hm);
               gsync();                // CG and RR are rewritten by the next column
            }
         }
         __syncthreads();
      }
   }

   // by the first wave; the others wait in helper()
   __device__ __forceinline__ void jacobian(double x)
   {
      double *X = S + L.EV + 5*2*N, *CT = X + N;
      if (lane < N) { X[lane] = x; CT[lane] = ct; }
      if (lane == 0) reinterpret_cast<int*>(S + L.MISC)[1] = 1;
      __syncthreads();
      jacobian_columns(0);
      jac_valid = true;
   }

   __device__ __forceinline__ void dismiss()
   {
      if (lane == 0) reinterpret_cast<int*>(S + L.MISC)[1] = 0;
      __syncthreads();
   }

   __device__ __forceinline__ void helper(int wv)
   {
      for (;;) {
         __syncthreads();
         if (reinterpret_cast<const int*>(S + L.MISC)[1] == 0) break;
         jacobian_columns(wv);
      }
   }

   // ---- analytic Jacobian (ChemGroup::jacobian_analytic) --------------------------
   // right after rhs(x): T is the temperature of x, and its concentrations and
   // Gibbs energies are in LDS
   __device__ __forceinline__ void jacobian_analytic(double x)
   {
      double *J = Jm();
      const double *C = S + L.CG, *Gk = C + NS;
      double *dG = S + L.EV, *rw = dG + NS, *Yf = rw + NS;
      const int st = nR + 1;           // element nR of each is 0: what the padding of the rows reads
      double *QT = S + L.U, *QC = QT + st, *V = QC + st, *Dq = S + L.RR;
      const int mE = m.maxEd, mP = m.maxPd, mT = m.maxTb;
      const bool unit = m.unitNu != 0;
      const double Tr = Trc;
      const double rho = lane_sum(x), irho = 1.0/rho;
      double vel[3];
#pragma unroll
      for (int i = 0; i < 3; i++) vel[i] = comp(x, NS + i)*irho;
      const double k2 = vel[0]*vel[0] + vel[1]*vel[1] + vel[2]*vel[2];
      const double e = comp(x, NS + 3)*irho - 0.5*k2;
      for (int k = lane; k < N*N; k += 64) J[k] = 0.0;
      // species terms: f, the mass fraction is not clipped
      const double y = irho*x, yc = dmin(dmax(y, 1e-60), 1.0);
      const bool f = (yc == y);
      const double h = poly_enthalpy(*this, c, Tr, iTrc, logTc);
      const double ek = E*m.ieRef;
      const double myC = (lane < NS) ? C[lane] : 0.0;
      if (lane < NS) {
         dG[lane] = -(h*W/RGAS)/(Tr*Tr);
         rw[lane] = m.rhoRef/W;
         Yf[lane] = f ? -1.0 : yc;     // negative: moves with its own density
      }
      const bool clipped = __ballot(lane < NS && !f) != 0;
      const double icv = irho/lane_sum(yc*(poly_cp(*this, c, Tr, iTrc) - rOvW)*m.iCpRef);
      const double sfe = lane_sum(f ? ek*yc : 0.0), clampW = lane_sum(f ? 0.0 : yc/W), ctot = lane_sum(myC);
      const double lct = log(ctot), logT = logTc;
      double dT, dct = 0.0;            // of column `lane`
      if (lane < NS) {
         dT = ((0.5*k2 - e) - ((f ? ek : 0.0) - sfe))*icv;
         dct = m.rhoRef*((f ? 1.0/W : 0.0) + clampW);
      } else if (lane < NS + 3) dT = -((lane == NS) ? vel[0] : (lane == NS + 1) ? vel[1] : vel[2])*icv;
      else dT = icv;
      gsync();
      // a lane per reaction: the derivatives of its rate of progress by T, by
      // ctot, and by the density of each of its species
      for (int k0 = 0; k0 < nR; k0 += 64) {
         const int k = min(k0 + lane, nR - 1);
         const bool mine = k0 + lane < nR;
         const DRate rt = m.rate[k];
         const uint32_t info = rt.info, eid = rt.eid, pid = rt.pid;
         const double A = rt.A, sumNu = rt.sumNu, rn = (double)rt.n, eR = (double)rt.EovR;
         const int ne = (info >> 16) & 15, np = (info >> 20) & 15, nt = (info >> 24) & 15;
         const bool hasE = fabs(eR) > 1e-5, back = (info >> 28) & 1;
         double arg = rn*logT, dlKf = 0.0;
         if (hasE) arg -= quot(eR, Tr, iTrc);
         const double Kf = A*exp(arg);
         if (rn != 0.0) dlKf += rn/Tr;
         if (hasE) dlKf += eR/(Tr*Tr);
         auto pw = [&](double cc, float nu) { return unit ? (nu == 1.0f ? cc : cc*cc) : conc_pow(cc, nu); };
         double a = 1.0, b = 1.0, g = 0.0, sd = 0.0;
#pragma unroll
         for (int i = 0; i < MAX_ED; i++)
            if (i < mE) {
               const int id = (eid >> 8*i) & 255;
               const float nu = m.kEnu[i][k];
               if (i < ne) { a *= pw(C[id], nu); g -= nu*Gk[id]; sd -= nu*dG[id]; }
            }
#pragma unroll
         for (int i = 0; i < MAX_PD; i++)
            if (i < mP) {
               const int id = (pid >> 8*i) & 255;
               const float nu = m.kPnu[i][k];
               if (i < np) { b *= pw(C[id], nu); g += nu*Gk[id]; sd += nu*dG[id]; }
            }
         double Kb = 0.0, dlKb = 0.0;
         if (back) { Kb = Kf*exp(g - sumNu*lct); dlKb = dlKf + sd; }
         else b = 1.0;
         const double D = Kf*a - Kb*b;
         double cc = 1.0;
         if (nt > 0) {
            cc = ctot;
            for (int i = 0; i < nt; i++) cc += C[m.kTid[i][k]]*(m.kTeff[i][k] - 1.0);
         }
         if (mine) {
            QT[k] = cc*(Kf*dlKf*a - Kb*dlKb*b)*m.TRef;
            QC[k] = cc*Kb*b*(back ? sumNu : 0.0)/ctot + (nt > 0 ? D : 0.0);
            Dq[k] = nt > 0 ? D : 0.0;
         }
         auto part = [&](bool educt, int q, double cK) {
            const uint32_t ids = educt ? eid : pid;
            const int n = educt ? ne : np, id = (ids >> 8*q) & 255;
            const float nq = educt ? m.kEnu[q][k] : m.kPnu[q][k];
            double p = (nq == 1.0f) ? 1.0 : (double)nq*(unit ? C[id] : conc_pow(C[id], nq - 1.0f));
            const int mx = educt ? mE : mP;
#pragma unroll
            for (int l = 0; l < (MAX_ED > MAX_PD ? MAX_ED : MAX_PD); l++)
               if (l < mx && l != q) {
                  const double c1 = C[(ids >> 8*l) & 255];
                  const float nu = educt ? m.kEnu[l][k] : m.kPnu[l][k];
                  const double t = p*pw(c1, nu);
                  p = (l < n) ? t : p;
               }
            if (mine) V[((educt ? 0 : mE) + q)*st + k] = (q < n && (educt || back)) ? cK*p*rw[id] : 0.0;
         };
         if (unit) {
#pragma unroll
            for (int q = 0; q < MAX_ED; q++) if (q < mE) part(true, q, cc*Kf);
#pragma unroll
            for (int q = 0; q < MAX_PD; q++) if (q < mP) part(false, q, cc*Kb);
         } else {
#pragma unroll 1
            for (int q = 0; q < mE; q++) part(true, q, cc*Kf);
#pragma unroll 1
            for (int q = 0; q < mP; q++) part(false, q, cc*Kb);
         }
      }
      for (int k = lane; k < 2 + mE + mP; k += 64) QT[k*st + nR] = 0.0;
      gsync();
      // a lane per row: the sparse entries added up in the row, in the order of
      // its reactions, and the row's sums by T and ctot
      double aT = 0.0, aC = 0.0, scl = 0.0;
      if (lane < NS) {
         auto add = [&](int id, double val) {
            if (clipped) {
               const double yf = Yf[id];
               if (yf >= 0.0) { scl += val*yf; return; }
            }
            lds_add(&J[lane + id*N], val);
         };
         const DRow *row = m.rows() + lane;
         const int n = m.nRows;
         if (!clipped && mT == 0 && mE == 2 && mP == 2) {
            // two educts, two products at most: past a reaction's arity V is 0,
            // past the row's end the entries are those of reaction nR
            DRow r[4], nx[4];
#pragma unroll
            for (int k = 0; k < 4; k++) nx[k] = row[min(k, n - 1)*NS];
            for (int k0 = 0; k0 < n; k0 += 4) {
               double qt[4], qc[4], v[4][4];
#pragma unroll
               for (int k = 0; k < 4; k++) { r[k] = nx[k]; nx[k] = row[min(k0 + 4 + k, n - 1)*NS]; }
#pragma unroll
               for (int k = 0; k < 4; k++) {
                  const int q = (k0 + k < n) ? r[k].info & 0xffff : nR;
                  qt[k] = QT[q];
                  qc[k] = QC[q];
#pragma unroll
                  for (int i = 0; i < 4; i++) v[k][i] = V[i*st + q];
               }
#pragma unroll
               for (int k = 0; k < 4; k++) {
                  const double nu = r[k].nu;
                  aT += nu*qt[k];
                  aC += nu*qc[k];
#pragma unroll
                  for (int i = 0; i < 4; i++)
                     lds_add(&J[lane + (((i < 2 ? r[k].eid : r[k].pid) >> 8*(i & 1)) & 255)*N], (i < 2 ? nu : -nu)*v[k][i]);
               }
            }
         } else {
            for (int k = 0; k < nrow; k++) {
               const DRow r = row[k*NS];
               const int q = r.info & 0xffff, ne = (r.info >> 16) & 15, np = ((r.info >> 28) & 1) ? (r.info >> 20) & 15 : 0;
               const double nu = r.nu;
               aT += nu*QT[q];
               aC += nu*QC[q];
               for (int i = 0; i < ne; i++) add((r.eid >> 8*i) & 255, nu*V[i*st + q]);
               for (int i = 0; i < np; i++) add((r.pid >> 8*i) & 255, -nu*V[(mE + i)*st + q]);
               for (int i = 0, nt = (r.info >> 24) & 15; i < nt; i++) {
                  const int id = m.kTid[i][q];
                  add(id, nu*Dq[q]*(m.kTeff[i][q] - 1.0)*rw[id]);
               }
            }
         }
      }
      gsync();
      const double wr = W*m.iwiRef;
      {
         const int l = lane < NS ? lane : 0;
         double v[N];
#pragma unroll
         for (int j = 0; j < N; j++) v[j] = J[l + j*N];
#pragma unroll
         for (int j = 0; j < N; j++)
            v[j] = wr*(v[j] + aT*rdlane(dT, j) + aC*rdlane(dct, j) + ((j < NS) ? scl : 0.0));
         if (lane < NS) {
#pragma unroll
            for (int j = 0; j < N; j++) J[lane + j*N] = v[j];
         }
      }
      gsync();
      jac_valid = true;
   }

   // LUdec::ludcmp (math_utils.hpp:87-155): lane i holds row i (a(k), k < N,
   // called by every lane) in registers and keeps it; its position after the
   // interchanges so far is tracked instead of moving the row.  Per column the
   // candidates are the rows at positions >= j, the pivot the last position
   // attaining the maximum scaled magnitude (the reference's `>=' scan), the
   // pivot row is broadcast by readlane, and every entry receives the same
   // products in the same order as ChemGroup::ludcmp, so the factors are the
   // same.  The current column is row[0]: the update of an entry writes it one
   // place down, so the loop over the columns stays a loop (unrolled, the
   // factorisation alone was 45 KB of code, and with the other unrolled pieces
   // a step missed the instruction cache throughout).  The factors go to M by
   // row, the row of each position to ind().
   template<int LEN, typename T_>
   __device__ __forceinline__ void lu_columns(T_ *M, T_ *row, T_ vvi, int &pos, int j0, int j1)
   {
      const bool act = lane < N;
#pragma unroll 1
      for (int j = j0; j < j1; j++) {
         const T_ dum = vvi*fabs(row[0]);
         const bool cand = act && pos >= j && dum >= (T_)0;       // not a NaN
         const T_ inv = (T_)1/row[0];                             // of every row: does not wait for the pivot
         const uint32_t key = cand ? upper_word(dum) + 1u : 0u;
         const uint32_t top = wave_umax(key);
         unsigned long long hit = __ballot(cand && key == top);
         if (sizeof(T_) == 8 && (hit & (hit - 1))) {              // equal upper words: the numbers themselves
            const double best = wave_dmax((cand && key == top) ? (double)dum : -1.0);
            hit = __ballot(cand && key == top && (double)dum == best);
         }
         if (!hit) hit = __ballot(act && pos == j);
         int P = __ffsll(hit) - 1;
         int imax = __builtin_amdgcn_readlane(pos, P);
         while (hit &= hit - 1) {                                 // equal magnitudes: the last position
            const int l = __ffsll(hit) - 1, o = __builtin_amdgcn_readlane(pos, l);
            if (o > imax) { imax = o; P = l; }
         }
         if (lane == P) pos = j;
         else if (act && pos == j) pos = imax;
         T_ pv = rdlane(row[0], P);
         T_ dv = rdlane(inv, P);
         if (pv == (T_)0) { pv = (T_)1.0e-20; dv = (T_)1/pv; }
         const T_ lij = row[0]*dv;
         const bool below = act && pos > j;
         const T_ w = below ? lij : (T_)0;
         if (act) M[lane + j*N] = (lane == P) ? pv : below ? lij : row[0];
         // operands eight ahead, products two ahead (lane_sum)
         T_ u[LEN + 8], t[LEN + 2];
#pragma unroll
         for (int k = 1; k < 9 && k < LEN; k++) u[k] = rdlane(row[k], P);
#pragma unroll
         for (int k = 1; k < 3 && k < LEN; k++) t[k] = w*u[k];
#pragma unroll
         for (int k = 1; k < LEN; k++) {
            if (k + 8 < LEN) u[k + 8] = rdlane(row[k + 8], P);
            if (k + 2 < LEN) t[k + 2] = w*u[k + 2];
            row[k - 1] = row[k] - t[k];
            __builtin_amdgcn_sched_barrier(0);
         }
      }
   }

   template<typename T_, typename F_>
   __device__ __forceinline__ void ludcmp(T_ *M, F_ a)
   {
      T_ row[N];
#pragma unroll
      for (int k = 0; k < N; k++) { const T_ x = a(k); row[k] = (lane < N) ? x : (T_)0; }
      T_ big = 0;
#pragma unroll
      for (int k = 0; k < N; k++) { const T_ x = fabs(row[k]); big = (big < x) ? x : big; }
      const T_ vvi = (T_)1/big;
      int pos = lane;
      constexpr int H = N/2;           // the second half of the columns on half the entries
      lu_columns<N>(M, row, vvi, pos, 0, H);
      lu_columns<N - H>(M, row, vvi, pos, H, N);
      if (lane < N) ind()[pos] = lane;
      gsync();
   }

   // LUdec::lubksb (math_utils.hpp:157-188) of the lane-held b: permutation,
   // forward substitution column by column (each entry receives its products
   // in the reference's order), back substitution row by row in its order: the
   // products of row i by a lane each (lane t: column i + 1 + t), their
   // subtraction one after another in every lane
   // Rows with n of LO < n <= HI products: the loop over the terms is HI long
   // (past the row: 0)
   template<int LO, int HI>
   __device__ __forceinline__ void back_rows(const double *M, int perm, double x, double dg, double idg, double &xs,
                                             double &next)
   {
#pragma unroll 1
      for (int n = LO + 1; n <= HI; n++) {
         const int i = N - 1 - n;
         const double p = (lane < n) ? next*xs : 0.0;
         next = M[__builtin_amdgcn_readlane(perm, max(i - 1, 0)) + min(i + lane, N - 1)*N];
         const double b = rdlane(dg, i), rb = rdlane(idg, i);
         double sum = rdlane(x, i), u[HI];
#pragma unroll
         for (int c0 = 0; c0 < 8 && c0 < HI; c0++) u[c0] = rdlane(p, c0);
#pragma unroll
         for (int c0 = 0; c0 < HI; c0++) {
            sum -= u[c0];
            if (c0 + 8 < HI) u[c0 + 8] = rdlane(p, c0 + 8);
            __builtin_amdgcn_sched_barrier(0);
         }
         xs = wave_shift(xs, quot(sum, b, rb));
      }
   }

   __device__ __forceinline__ double lubksb(const double *M, double b)
   {
      const int l = lane < N ? lane : N - 1;
      const int perm = ind()[l];
      const double *row = M + perm;
      double x = __shfl(b, perm, 64);
      const double dg = row[l*N], idg = 1.0/dg;
      {
         double lo[N];
#pragma unroll
         for (int k = 0; k < N - 1; k++) { const double t = row[k*N]; lo[k] = (lane > k) ? t : 0.0; }
#pragma unroll
         for (int k = 0; k < N - 1; k++) x -= lo[k]*rdlane(x, k);
      }
      // lane t of xs: the solution of column i + 1 + t
      double xs = wave_shift(0.0, quot(rdlane(x, N - 1), rdlane(dg, N - 1), rdlane(idg, N - 1)));
      double next = M[__builtin_amdgcn_readlane(perm, N - 2) + min(N - 1 + lane, N - 1)*N];
      constexpr int A1 = (N - 1)/4, A2 = (N - 1)/2, A3 = 3*(N - 1)/4;
      back_rows<0, A1>(M, perm, x, dg, idg, xs, next);
      back_rows<A1, A2>(M, perm, x, dg, idg, xs, next);
      back_rows<A2, A3>(M, perm, x, dg, idg, xs, next);
      back_rows<A3, N - 1>(M, perm, x, dg, idg, xs, next);
      return xs;
   }

   // A = I/(gam dt) - J, factorised (Rosenbrock::step, math_utils.hpp:282-291)
   __device__ __forceinline__ double entry(const double *J, int i, int k, double d) const
   {
      const double x = -J[i + k*N];
      return (k == i) ? x + d : x;
   }

   __device__ __forceinline__ void factor(double d)
   {
      const int i = lane < N ? lane : N - 1;
      const double *J = Jm();
      if constexpr (PREC == HTR_CHEM_FP64) {
         ludcmp<double>(S + L.U, [&](int k) { return entry(J, i, k, d); });
      } else {
         ludcmp<float>(reinterpret_cast<float*>(S + L.U), [&](int k) { return (float)(rs*entry(J, i, k, d)*rdlane(cs, k)); });
         lu64 = false;
      }
   }

   // FP32_IR: equilibration by powers of two (rows, then columns)
   double rs, cs;
   __device__ __forceinline__ void equilibrate(double d)
   {
      const int i = lane < N ? lane : N - 1;
      const double *J = Jm();
      double big = 0.0;
#pragma unroll
      for (int k = 0; k < N; k++) big = dmax(big, fabs(entry(J, i, k, d)));
      rs = pow2_inv(big);
      big = 0.0;
#pragma unroll
      for (int k = 0; k < N; k++) big = dmax(big, fabs(rdlane(rs, k)*entry(J, k, i, d)));
      cs = pow2_inv(big);
   }

   // FP32_IR solve: the FP64 matrix row and the FP32 factors of the lane's
   // position in registers, refined until the correction is below 1e-15 of the
   // solution; false (b unchanged) when the refinement stalls
   __device__ __forceinline__ bool refine(double &b, double d)
   {
      const int l = lane < N ? lane : N - 1;
      const bool act = lane < N;
      const float *M = reinterpret_cast<const float*>(S + L.U);
      const int perm = ind()[l];
      float lu[N];
#pragma unroll
      for (int k = 0; k < N; k++) lu[k] = M[perm + k*N];
      const float ud = 1.0f/M[perm + l*N];
      // the matrix is read from LDS in every sweep, a few entries ahead: held in
      // registers beside the factors it spilled.  r - (d - J) x is formed as
      // r + (J - d) x, the same to the bit
      const double *Jr = Jm() + l;
      const double jd = Jr[l*N] - d;
      double xk = 0.0, prev = 0.0;
      bool done = false;
#pragma unroll 1
      for (int it = 0; it < 9 && !done; it++) {
         double r = b;
         if (it > 0) {
            double u[N + 8], a[N + 8], t[N + 2];
#pragma unroll
            for (int j = 0; j < 8 && j < N; j++) { a[j] = Jr[j*N]; u[j] = rdlane(xk, j); }
#pragma unroll
            for (int j = 0; j < 2; j++) t[j] = ((l == j) ? jd : a[j])*u[j];
#pragma unroll
            for (int j = 0; j < N; j++) {
               if (j + 8 < N) { a[j + 8] = Jr[(j + 8)*N]; u[j + 8] = rdlane(xk, j + 8); }
               if (j + 2 < N) t[j + 2] = ((l == j + 2) ? jd : a[j + 2])*u[j + 2];
               r += t[j];
               __builtin_amdgcn_sched_barrier(0);
            }
         }
         float rf = (float)(r*rs);
         rf = __shfl(rf, perm, 64);
#pragma unroll
         for (int k = 0; k < N - 1; k++) {
            HTR_PIN(lu[k]);           // the triangle is cut out here, not kept as two
            rf -= ((lane > k) ? lu[k] : 0.0f)*rdlane(rf, k);
         }
#pragma unroll
         for (int k = N - 1; k > 0; k--) {
            HTR_PIN(lu[k]);
            rf -= ((lane < k) ? lu[k] : 0.0f)*rdlane(rf*ud, k);
         }
         rf *= ud;
         const double ci = act ? cs*(double)rf : 0.0;
         xk += ci;
         const double nc = wave_dmax(fabs(ci)), nx = wave_dmax(fabs(xk));
         if (it > 0) {
            if (!(nc > 1e-15*nx)) done = true;
            else if (!(nc < 0.5*prev)) break;
         }
         prev = nc;
      }
      if (done) b = xk;
      return done;
   }

   // A^-1 b
   __device__ __forceinline__ double solve(double b, double d)
   {
      if constexpr (PREC == HTR_CHEM_FP64) {
         return lubksb(S + L.U, b);
      } else {
         if (!lu64) {
            if (refine(b, d)) return b;
            // refinement stalled: FP64 LU of the same matrix for this step, in
            // the Jacobian's place (formed again if the step is retried)
            const int i = lane < N ? lane : N - 1;
            double *M = Jm();
            ludcmp<double>(M, [&](int k) { return entry(M, i, k, d); });   // (reads M before it writes)
            jac_valid = false;
            lu64 = true;
         }
         return lubksb(Jm(), b);
      }
   }

   // Rosenbrock::solve (math_utils.hpp:195-386): Kaps-Rentrop, gamma = 1/2;
   // returns accepted steps, or -1 if a reference cap was hit
   __device__ __forceinline__ int solve_cell(double &x, double dtTry, double DelT)
   {
      bool finish = false;
      double time = 0.0, dt = dtTry, dx = 0.0;
      for (int st = 0; st < 100000; st++) {
         const double t0 = time;
         double dtNext = 0.0, xs = x, dxs = 0.0;
         bool first = true;
         jac_valid = false;
         int jtry;
         for (jtry = 0; jtry < 100; jtry++) {
            const double d = 1.0/((1.0/2.0)*dt);
            double g1 = 0.0, g2 = 0.0, g3 = 0.0, g4 = 0.0;
            // s = -1: Jacobian (if it is not there) and factors at the step's
            // start point; s = 0 .. 3: the stages.  One loop, so that the
            // right-hand side is there once.
            if constexpr (!AJ) { if (!jac_valid) jacobian(xs); }
#pragma unroll 1
            for (int s = -1; s < 4; s++) {
               if (s >= 0) {
                  double g;
                  if (s == 0)      g = dxs + dt*(1.0/2.0)*dx;
                  else if (s == 1) g = dx + dt*(-3.0/2.0)*dx + (-8.0)*g1/dt;
                  else if (s == 2) g = dx + dt*(121.0/50.0)*dx + ((372.0/25.0)*g1 + (12.0/5.0)*g2)/dt;
                  else             g = dx + dt*(29.0/250.0)*dx + ((-112.0/125.0)*g1 + (-54.0/125.0)*g2 + (-2.0/5.0)*g3)/dt;
                  g = solve(g, d);
                  if (s == 0)      { g1 = g; x = xs + 2.0*g1; }
                  else if (s == 1) { g2 = g; x = xs + (48.0/25.0)*g1 + (6.0/25.0)*g2; }
                  else if (s == 2) g3 = g;
                  else             g4 = g;
               }
               // the analytic Jacobian needs T(x); the right-hand side of the
               // start point is kept from the first attempt
               const bool form = AJ ? !jac_valid : first;
               if (s < 0 ? form : s < 2) {
                  const double d0 = rhs(s < 0 ? xs : x);
                  if (s >= 0 || first) dx = d0;
                  if (first) { dxs = d0; first = false; }
               }
               if (s < 0) {
                  if constexpr (AJ) { if (form) jacobian_analytic(xs); }
                  if constexpr (PREC != HTR_CHEM_FP64) equilibrate(d);
                  factor(d);
               }
            }
            x = xs + (19.0/9.0)*g1 + (1.0/2.0)*g2 + (25.0/108.0)*g3 + (125.0/108.0)*g4;
            const double err = (17.0/54.0)*g1 + (7.0/36.0)*g2 + 0.0*g3 + (125.0/108.0)*g4;
            time = t0 + dt;
            // Rosenbrock::itercheck (math_utils.hpp:337-360)
            const double errmax = wave_dmax(dmax(0.0, lane < N ? fabs(err) : 0.0))*(1.0/1e-10);
            const bool accept = (errmax < 1.0) || finish;
            double grow = 1.5;
            if (!accept || errmax > 0.1296) grow = pow(errmax, accept ? -0.25 : -1.0/3.0);
            if (accept) {
               dtNext = (errmax > 0.1296) ? 0.9*dt*grow : 1.5*dt;
               break;
            }
            dtNext = 0.9*dt*grow;
            dt = (dt > 0.0) ? dmax(dtNext, 0.5*dt) : dmin(dtNext, 0.5*dt);
         }
         if (jtry == 100) return -1;
         const double Remainder = DelT - time;
         if (finish || (Remainder < 1e-12*DelT)) return st + 1;
         if (dtNext*1.5 > Remainder) { dt = Remainder; finish = true; }
         else                        { dt = dtNext;    finish = false; }
      }
      return -1;
   }
};

// A block per cell in flight: the first wave takes cells from the queue counter
// until it passes n; with the central-difference Jacobian three more waves help.
// Waves per SIMD: with differences three, although the registers then spill 300 to
// 384 B a lane (12^3 cells FP64 274 ms, 20^3 686; two 303 and 814, one 398 and 1276,
// four 309 and 726): what waits for the Newton chain of one cell is filled by other
// cells.  With the analytic Jacobian two (36 to 68 B; 20^3 refined 174 ms, 32^3 540;
// one 221 and 745, three 204 and 613, four 243 and 793): a wave is busy 46 % of its
// cycles there, and spills cost more than a third wave brings.
template<class MX, int PREC, bool AJ>
__global__ void __launch_bounds__(AJ ? 64 : 64*CHEM_FD_WAVES, AJ ? 2 : 3)
chem_wave_kernel(const htr_fields f, const DMix *__restrict__ mix, const Geo g, double dt, htr_view nsteps,
                 int *__restrict__ fails, int *__restrict__ queue, int64_t n)
{
   HIP_DYNAMIC_SHARED(double, lds)
   constexpr int N = MX::NEQ;
   const WaveLayout<MX, PREC, AJ> L(mix->nReac, mix->maxEd, mix->maxPd);
   const int lane = threadIdx.x & 63;
   const int wv = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
   ChemWave<MX, PREC, AJ> G(*mix, L, lds, lane);
   if (!AJ && wv > 0) { G.helper(wv); return; }
   for (;;) {
      int q = 0;
      if (lane == 0) q = atomicAdd(queue, 1);
      const int64_t cell = __builtin_amdgcn_readlane(q, 0);
      if (cell >= n) break;
      const P3 p = exec_point(g, cell);
      double x = 0.0;
      G.ct = 0.0;
      if (lane < N) {
         G.ct = ld<double>(f.Conserved_t, p, lane);
         at<double>(f.Conserved_t_old, p, lane) = G.ct;
         x = ld<double>(f.Conserved, p, lane);
      }
      G.T = ld<double>(f.temperature, p);
      const int st = G.solve_cell(x, dt, dt);
      if (lane < N) at<double>(f.Conserved, p, lane) = x;
      if (lane == 0) {
         at<double>(f.temperature, p) = G.T;
         if (nsteps.ptr) at<int32_t>(nsteps, p) = st;
         if (st < 0) atomicAdd(fails, 1);
      }
   }
   if (!AJ) G.dismiss();
}

} // namespace htr
