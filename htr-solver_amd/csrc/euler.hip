// euler.hip -- Euler flux divergence along one direction: hybrid KG/TENO,
// pure TENO/TENO-A/TENO-LAD and pure Kennedy-Gruber (skew-symmetric).
//
// Reference: src/prometeo_rhs.inl:40-1052 (ComputeKGSums, KGFluxReconstruction,
// ComputeRoeAverages, characteristic projections, FluxReconstruction<Op>,
// the three updateRHSSpan loops), src/prometeo_rhs.cu:37-459 (GPU variants).
//
// The face flux is a function of its left cell only: the reference's
// Kennedy-Gruber ring buffer holds pair sums S(a,b) of two cells, and its
// "first minus inter-cell location" is the face of the cell before the first
// one (or of the first cell itself at a staggered left boundary).  Passes per
// direction, all with consecutive lanes on x-adjacent cells:
//   hybrid: classify faces (sensor) into a compacted TENO list; TENO faces in
//     two passes (Roe record; characteristic components and back-projection)
//     and the limiter into a face buffer; then the KG pass: one thread per
//     cell forms both its faces and differences them into Conserved_t, reading
//     TENO faces back (for all directions at once in a full right-hand side);
//   pure TENO family: the TENO passes over every face, then a divergence pass
//     over the face buffer;
//   pure KG: the KG pass alone.
// The TENO passes evaluate the characteristic projection one component at a
// time (left-eigenvector rows of rhs.inl:436-505 with the per-point sums
// hoisted), so no 6 x nEq split-flux arrays are held in registers.
#include "common.hpp"
#include "kernels.hpp"

namespace htr {

// hybrid sensor of the face of cell p: KG when the shock sensor is clear at
// pM1, p and pP1 (rhs.inl:818-820)
template<int DIR>
__device__ __forceinline__ bool hybrid_kg(const htr_fields &f, const Geo &g, const P3 &p, int t)
{
   const P3 pM1 = wminus(g, DIR, p, c_st.Cp[t][1]);
   const P3 pP1 = wplus(g, DIR, p, c_st.Cp[t][2]);
   return ld<uint8_t>(f.shockSensor[DIR], pM1) && ld<uint8_t>(f.shockSensor[DIR], p) &&
          ld<uint8_t>(f.shockSensor[DIR], pP1);
}

template<class MX, int DIR>
struct Euler {
   static constexpr int NS = MX::NS, NEQ = MX::NEQ;
   static constexpr int iN = DIR, iT1 = (DIR == 0) ? 1 : 0, iT2 = (DIR == 2) ? 1 : 2;

   const htr_fields &f;
   const DMix &m;
   const Geo &g;
   const htr_view hv;     // total enthalpy (rhoE + p)/rho per cell, from enthalpy_kernel

   __device__ double cons(const P3 &p, int i) const { return ld<double>(f.Conserved, p, i); }
   __device__ double vel(const P3 &p, int i) const { return ld<double>(f.velocity, p, i); }

   // ---- Roe state (rhs.inl:200-279) ----------------------------------------
   struct Roe { double a, e, H, a2, rho, v[3], Y[NS], dpde, dpdrhoi[NS]; };

   __device__ __forceinline__ static double mod2(const double *v) { double r = 0.0; r += v[0]*v[0]; r += v[1]*v[1]; r += v[2]*v[2]; return r; }

   __device__ void roe(Roe &R, const P3 &L, const P3 &Rp) const
   {
      double vL[3], vR[3];
#pragma unroll
      for (int i = 0; i < 3; i++) { vL[i] = vel(L, i); vR[i] = vel(Rp, i); }
      const double rhoL = ld<double>(f.rho, L), rhoR = ld<double>(f.rho, Rp);
      const double pL = ld<double>(f.pressure, L), pR = ld<double>(f.pressure, Rp);
      const double IeL = cons(L, NS+3)/rhoL - 0.5*mod2(vL);
      const double IeR = cons(Rp, NS+3)/rhoR - 0.5*mod2(vR);
      const double HL = ld<double>(hv, L);
      const double HR = ld<double>(hv, Rp);
      const double fL = sqrt(rhoL)/(sqrt(rhoL) + sqrt(rhoR));
      const double fR = sqrt(rhoR)/(sqrt(rhoL) + sqrt(rhoR));
      R.rho = sqrt(rhoL*rhoR);
#pragma unroll
      for (int i = 0; i < NS; i++) R.Y[i] = ld<double>(f.MassFracs, L, i)*fL + ld<double>(f.MassFracs, Rp, i)*fR;
#pragma unroll
      for (int i = 0; i < 3; i++) R.v[i] = vL[i]*fL + vR[i]*fR;
      R.H = HL*fL + HR*fR;
      R.e = IeL*fL + IeR*fR;
      const double PovRho = R.H - R.e - 0.5*mod2(R.v);
      const double MixW = MX::MolarWeightFromY(m, R.Y);
      const double Teos = MX::TFromRhoAndP(m, R.rho, MixW, PovRho*R.rho);
      const double T = MX::TFromInternalEnergy(m, R.e, Teos, R.Y);
      const double gam = MX::Gamma(m, T, MixW, R.Y);
      R.dpde = MX::dpde(R.rho, gam);
      MX::dpdrhoi(m, R.dpdrhoi, gam, T, R.Y);
      const double dp = pR - pL;
      const double de = IeR - IeL;
      double dpError = dp - de*R.dpde;
      double fact = de*R.dpde; fact *= fact;
      double drhoi[NS];
#pragma unroll
      for (int i = 0; i < NS; i++) {
         drhoi[i] = rhoR*ld<double>(f.MassFracs, Rp, i) - rhoL*ld<double>(f.MassFracs, L, i);
         const double dpi = drhoi[i]*R.dpdrhoi[i];
         dpError -= dpi;
         fact += dpi*dpi;
      }
      fact = dpError/dmax(fact, 1e-6);
#pragma unroll
      for (int i = 0; i < NS; i++) R.dpdrhoi[i] = R.dpdrhoi[i]*(1.0 + R.dpdrhoi[i]*drhoi[i]*fact);
      R.dpde = R.dpde*(1.0 + R.dpde*de*fact);
      R.a2 = PovRho/R.rho*R.dpde;
#pragma unroll
      for (int i = 0; i < NS; i++) R.a2 += R.Y[i]*R.dpdrhoi[i];
      R.a = sqrt(R.a2);
   }

   // Constants of the left-eigenvector rows (rhs.inl:443-455)
   struct Proj { double iaRoe, Coeff, d, cv[3], iaRoe2; };

   // Row i of projectToCharacteristicSpace applied to the vector w, with
   // sum1 = sum_j (Coeff - dpdrhoi_j) iaRoe2 w_j and sumQsp = sum_j w_j
   // precomputed; wm[0..3] are w[NS..NS+3]; for species rows ws = w[i-1] and
   // Y = Yi[i-1] of the Roe state (passed in, so that no per-lane array is
   // indexed by the runtime row).
   __device__ __forceinline__ static double char_row(int i, const Roe &R, const Proj &P, double sum1, double sumQsp,
                                     double ws, const double *wm, double Y)
   {
      if (i == 0 || i == NEQ-1) {
         const double sg = (i == 0) ? 1.0 : -1.0;
         double r = (i == 0) ? sumQsp*R.v[iN]*P.iaRoe - sum1 : -sumQsp*R.v[iN]*P.iaRoe - sum1;
         r -= (P.cv[iN] + sg*P.iaRoe)*wm[iN];
         r -= P.cv[iT1]*wm[iT1];
         r -= P.cv[iT2]*wm[iT2];
         r += P.d*wm[3];
         return r*0.5;
      }
      if (i <= NS) {
         double r = Y*sum1;
         r += ws;
         r += Y*P.cv[0]*wm[0];
         r += Y*P.cv[1]*wm[1];
         r += Y*P.cv[2]*wm[2];
         r += -Y*P.d*wm[3];
         return r;
      }
      if (i == NS+1) { double r = -R.v[iT1]*sumQsp; r += wm[iT1]; return r; }
      double r = -R.v[iT2]*sumQsp; r += wm[iT2]; return r;
   }

   // Column i of projectFromCharacteristicSpace (rhs.inl:510-572) applied to
   // the scalar q and added to r.  Called for i = 0..NEQ-1 in order, it sums
   // every component in the reference's order: sumQsp collects the species
   // rows and enters the momentum rows where the reference adds it.
   __device__ __forceinline__ static void add_column(double *r, double &sumQsp, int i, double q, const Roe &R,
                                     double ERoe, double dedp)
   {
      if (i == 0) {
#pragma unroll
         for (int s = 0; s < NS; s++) r[s] = R.Y[s]*q;
         r[NS+iN] = (R.v[iN] - R.a)*q;
         r[NS+iT1] = R.v[iT1]*q;
         r[NS+iT2] = R.v[iT2]*q;
         r[NS+3] = (R.H - R.v[iN]*R.a)*q;
         sumQsp = 0.0;
      } else if (i <= NS) {
#pragma unroll
         for (int s = 0; s < NS; s++) if (s == i-1) {
            r[s] += q;
            r[NS+3] += (ERoe - R.rho*R.dpdrhoi[s]*dedp)*q;
         }
         sumQsp += q;
      } else if (i == NS+1) {
         r[NS+iN] += R.v[iN]*sumQsp;
         r[NS+iT1] += R.v[iT1]*sumQsp;
         r[NS+iT1] += q;
         r[NS+3] += R.v[iT1]*q;
      } else if (i == NS+2) {
         r[NS+iT2] += R.v[iT2]*sumQsp;
         r[NS+iT2] += q;
         r[NS+3] += R.v[iT2]*q;
      } else {
#pragma unroll
         for (int s = 0; s < NS; s++) r[s] += R.Y[s]*q;
         r[NS+iN] += (R.v[iN] + R.a)*q;
         r[NS+iT1] += R.v[iT1]*q;
         r[NS+iT2] += R.v[iT2]*q;
         r[NS+3] += (R.H + R.v[iN]*R.a)*q;
      }
   }

   // ---- FluxReconstruction<Op> (rhs.inl:625-759) in three passes ----------
   // face record: Roe state and the Lax-Friedrichs eigenvalue maxima.  The
   // per-point species sums of the left-eigenvector products (point_sums)
   // are formed where the point values are staged (the component pass) or,
   // on the limiter path, in the back-projection pass.
   static constexpr int NREC = 2*NS + 12;

   // stencil points pM2..pP3 of the face at p (rhs.inl:640-655)
   __device__ __forceinline__ void points(P3 *P, const P3 &p, int t) const
   {
      P[0] = wminus(g, DIR, p, c_st.Cp[t][0]);
      P[1] = wminus(g, DIR, p, c_st.Cp[t][1]);
      P[2] = p;
      P[3] = wplus(g, DIR, p, c_st.Cp[t][2]);
      P[4] = wplus(g, DIR, p, c_st.Cp[t][3]);
      P[5] = wplus(g, DIR, p, c_st.Cp[t][4]);
   }

   // eigenvalue maxima over the six points (rhs.inl:656-678)
   __device__ void lam_max(const P3 *P, double &Lam1, double &Lam, double &LamN) const
   {
#pragma unroll
      for (int k = 0; k < 6; k++) {
         const double un = vel(P[k], iN);
         const double c = ld<double>(f.SoS, P[k]);
         const double l1 = fabs(un - c), l = fabs(un), lN = fabs(un + c);
         if (k == 0) { Lam1 = l1; Lam = l; LamN = lN; }
         else { Lam1 = dmax(Lam1, l1); Lam = dmax(Lam, l); LamN = dmax(LamN, lN); }
      }
   }

   __device__ static void put_rec(double *__restrict__ rec, int64_t cap, int64_t w, const Roe &R,
                                  double Lam1, double Lam, double LamN)
   {
#pragma unroll
      for (int s = 0; s < NS; s++) { rec[s*cap + w] = R.Y[s]; rec[(NS+8+s)*cap + w] = R.dpdrhoi[s]; }
#pragma unroll
      for (int j = 0; j < 3; j++) rec[(NS+j)*cap + w] = R.v[j];
      rec[(NS+3)*cap + w] = R.a;
      rec[(NS+4)*cap + w] = R.H;
      rec[(NS+5)*cap + w] = R.e;
      rec[(NS+6)*cap + w] = R.rho;
      rec[(NS+7)*cap + w] = R.dpde;
      rec[(2*NS+8)*cap + w] = R.a2;
      rec[(2*NS+9)*cap + w] = Lam1;
      rec[(2*NS+10)*cap + w] = Lam;
      rec[(2*NS+11)*cap + w] = LamN;
   }

   __device__ __forceinline__ static void get_rec(const double *__restrict__ rec, int64_t cap, int64_t w, Roe &R)
   {
#pragma unroll
      for (int s = 0; s < NS; s++) { R.Y[s] = rec[s*cap + w]; R.dpdrhoi[s] = rec[(NS+8+s)*cap + w]; }
#pragma unroll
      for (int j = 0; j < 3; j++) R.v[j] = rec[(NS+j)*cap + w];
      R.a = rec[(NS+3)*cap + w];
      R.H = rec[(NS+4)*cap + w];
      R.e = rec[(NS+5)*cap + w];
      R.rho = rec[(NS+6)*cap + w];
      R.dpde = rec[(NS+7)*cap + w];
      R.a2 = rec[(2*NS+8)*cap + w];
   }

   // constants of the left-eigenvector rows (rhs.inl:443-455)
   __device__ __forceinline__ static void proj(Proj &J, const Roe &R)
   {
      J.iaRoe = 1.0/R.a;
      J.iaRoe2 = 1.0/R.a2;
      J.Coeff = (R.e - 0.5*mod2(R.v))*R.dpde/R.rho;
      J.d = R.dpde/(R.rho*R.a2);
#pragma unroll
      for (int j = 0; j < 3; j++) J.cv[j] = R.v[j]*J.d;
   }

   // species sums of point P for the face's Roe state (the per-point part of
   // projectToCharacteristicSpace, rhs.inl:443-451)
   __device__ __forceinline__ void point_sums(const P3 &P, const Roe &R, const Proj &J, double *sums) const
   {
      const double un = vel(P, iN);
      double s1q = 0.0, sqq = 0.0, s1f = 0.0, sqf = 0.0;
#pragma unroll
      for (int j = 0; j < NS; j++) {
         const double q = cons(P, j);
         const double w = (J.Coeff - R.dpdrhoi[j])*J.iaRoe2;
         s1q += w*q;
         sqq += q;
         const double fq = q*un;
         s1f += w*fq;
         sqf += fq;
      }
      sums[0] = s1q; sums[1] = sqq; sums[2] = s1f; sums[3] = sqf;
   }

   // ± split flux of component i at point P (getPlusMinusFlux,
   // rhs.inl:586-620): row i of the left-eigenvector product of the conserved
   // vector and of the Euler flux, given the point's species sums
   __device__ __forceinline__ void split(double &vp, double &vm, int i, const P3 &P, double lam, const Roe &R,
                         const Proj &J, double Ysel, const double *sums) const
   {
      const double un = vel(P, iN);
      const double pr = ld<double>(f.pressure, P);
      const double qs = (i >= 1 && i <= NS) ? cons(P, i-1) : 0.0;
      double qm[4], fm[4];
#pragma unroll
      for (int j = 0; j < 4; j++) { qm[j] = cons(P, NS+j); fm[j] = qm[j]*un; }
      fm[iN] += pr;
      fm[3] += pr*un;
      const double Q = char_row(i, R, J, sums[0], sums[1], qs, qm, Ysel);
      const double F = char_row(i, R, J, sums[2], sums[3], qs*un, fm, Ysel);
      vp = F + lam*Q;
      vm = F - lam*Q;
   }

   // pass A: Roe state and eigenvalue maxima of face p
   __device__ void face_record(double *__restrict__ rec, int64_t cap, int64_t w, const P3 &p, int t) const
   {
      P3 P[6];
      points(P, p, t);
      double Lam1, Lam, LamN;
      lam_max(P, Lam1, Lam, LamN);
      Roe R;
      roe(R, p, P[3]);
      put_rec(rec, cap, w, R, Lam1, Lam, LamN);
   }

   // pass D, on the faces the test flagged: the first-order flux
   // -0.5*(FluxP(p) + FluxM(p+1)) back-projected and blended with the
   // high-order Flux (rhs.inl:721-758)
   __device__ void face_limit(double *Flux, const double *__restrict__ rec, int64_t cap, int64_t w, const P3 &p,
                              int t, double RK0, double RK1, double dt) const
   {
      Roe R;
      get_rec(rec, cap, w, R);
      const double dedp = 1.0/R.dpde;
      const double ERoe = R.e + 0.5*mod2(R.v);
      const P3 pP1 = wplus(g, DIR, p, c_st.Cp[t][2]);
      const double lim_f = dt*(ld<double>(f.m_e[DIR], p) + ld<double>(f.m_e[DIR], pP1));
      Proj J;
      proj(J, R);
      double FLO[NEQ];
      double sq = 0.0, s2[4], s3[4];
      point_sums(p, R, J, s2);
      point_sums(pP1, R, J, s3);
#pragma unroll
      for (int i = 0; i < NEQ; i++) {
         const double lam = rec[((i == 0) ? 2*NS+9 : (i == NEQ-1) ? 2*NS+11 : 2*NS+10)*cap + w];
         const double Ysel = (i >= 1 && i <= NS) ? R.Y[i-1] : 0.0;
         double ap, am, bp, bm;
         split(ap, am, i, p, lam, R, J, Ysel, s2);
         split(bp, bm, i, pP1, lam, R, J, Ysel, s3);
         add_column(FLO, sq, i, -0.5*(ap + bm), R, ERoe, dedp);
      }
      const double eps = 1e-60;
      double theta = 1.0;
#pragma unroll
      for (int i = 0; i < NS; i++) {
         const double dRhoi = lim_f*Flux[i];
         const double dRhoi_lo = lim_f*FLO[i];
         double theta_p = 1.0;
         const double rhoi_p = RK0*ld<double>(f.Conserved_old, p, i) + RK1*cons(p, i);
         const double rhoHO_p = rhoi_p + dRhoi;
         if (rhoHO_p < eps) {
            const double rhoLO = rhoi_p + dRhoi_lo;
            theta_p = (fabs(rhoHO_p - rhoLO) > eps) ? dmax(0.0, (eps - rhoLO)/(rhoHO_p - rhoLO)) : 1.0;
         }
         double theta_pp1 = 1.0;
         const double rhoi_pp1 = RK0*ld<double>(f.Conserved_old, pP1, i) + RK1*cons(pP1, i);
         const double rhoHO_pp1 = rhoi_pp1 - dRhoi;
         if (rhoHO_pp1 < eps) {
            const double rhoLO = rhoi_pp1 - dRhoi_lo;
            theta_pp1 = (fabs(rhoHO_pp1 - rhoLO) > eps) ? dmax(0.0, (eps - rhoLO)/(rhoHO_pp1 - rhoLO)) : 1.0;
         }
         theta = dmin(dmin(theta_p, theta_pp1), theta);
      }
#pragma unroll
      for (int i = 0; i < NEQ; i++) Flux[i] = Flux[i]*theta + FLO[i]*(1 - theta);
   }

   __device__ bool sensor_kg(const P3 &p, int t) const { return hybrid_kg<DIR>(f, g, p, t); }

};

// Total enthalpy H = (rhoE + p)/rho of every cell of Fluid_bounds (the pair
// sums and the Roe average read it at stencil points), in a workspace array
// addressed like the FP64 fields; the same expression the reference evaluates
// inline (rhs.inl:55, :226-227).
template<class MX>
__global__ void __launch_bounds__(256)
enthalpy_kernel(const htr_fields f, const Geo g, htr_view hv, int64_t ncells)
{
   const int64_t i = (int64_t)blockIdx.x*blockDim.x + threadIdx.x;
   if (i >= ncells) return;
   uint32_t r = (uint32_t)i;
   const int x = (int)(r % (uint32_t)g.bsz[0]); r /= (uint32_t)g.bsz[0];
   const int y = (int)(r % (uint32_t)g.bsz[1]);
   const int z = (int)(r / (uint32_t)g.bsz[1]);
   const P3 p = mkp(g, x, y, z);
   at<double>(hv, p) = (ld<double>(f.Conserved, p, MX::NS+3) + ld<double>(f.pressure, p))/ld<double>(f.rho, p);
}

// ---- face enumeration --------------------------------------------------------
// A sweep along DIR over the execution rect has (esz[DIR] + 1) faces per line:
// face j = 0 is the minus face of the first cell, taken at the cell
// p0 + offM1(nType[p0]) as the reference primes FluxM (rhs.inl:800-817), and
// face j >= 1 is the plus face of cell elo[DIR] + j - 1.  Face ids put the
// x index fastest, so consecutive lanes touch consecutive cells: for the x
// sweep id = line*(esz0 + 1) + j, for y and z id = j*nlines + line with the
// line index x-fastest.
template<int DIR>
struct Faces {
   static constexpr int A = (DIR == 0) ? 1 : 0;     // fastest cross direction
   static constexpr int B = (DIR == 2) ? 1 : 2;
   __device__ static void split(const Geo &g, uint32_t fid, uint32_t &line, int &j)
   {
      if (DIR == 0) { const uint32_t n = (uint32_t)g.esz[0] + 1; line = fid/n; j = (int)(fid - line*n); }
      else { const uint32_t nl = (uint32_t)g.esz[A]*(uint32_t)g.esz[B]; j = (int)(fid/nl); line = fid - (uint32_t)j*nl; }
   }
   __device__ static uint32_t id(const Geo &g, uint32_t line, int j)
   {
      if (DIR == 0) return line*((uint32_t)g.esz[0] + 1) + (uint32_t)j;
      return (uint32_t)j*((uint32_t)g.esz[A]*(uint32_t)g.esz[B]) + line;
   }
   // the cell whose plus face is face fid
   __device__ static P3 cell(const Geo &g, const htr_fields &f, uint32_t fid)
   {
      uint32_t line; int j;
      split(g, fid, line, j);
      int c[3];
      c[A] = g.elo[A] + (int)(line % (uint32_t)g.esz[A]);
      c[B] = g.elo[B] + (int)(line / (uint32_t)g.esz[A]);
      c[DIR] = g.elo[DIR] + (j > 0 ? j - 1 : 0);
      P3 p = mkp(g, c[0], c[1], c[2]);
      if (j == 0) p = wminus(g, DIR, p, c_st.Cp[ld<int>(f.nType[DIR], p)][1]);
      return p;
   }
   __host__ __device__ static int64_t count(const Geo &g) { return ((int64_t)g.esz[DIR] + 1)*g.esz[A]*g.esz[B]; }
};

// Face buffer, face-major: the nEq components of face fid are F[fid*nEq ..
// fid*nEq + nEq - 1], so the scattered TENO faces write and read one
// cache-line run each instead of nEq separate lines.
template<int NEQ>
__device__ inline double &face_at(double *__restrict__ F, uint32_t fid, int i) { return F[(int64_t)fid*NEQ + i]; }

template<int NEQ>
__device__ inline double face_ld(const double *__restrict__ F, uint32_t fid, int i) { return F[(int64_t)fid*NEQ + i]; }

template<int NEQ>
__device__ inline void store_face(double *__restrict__ F, int64_t nfaces, uint32_t fid, const double *v)
{
   (void)nfaces;
#pragma unroll
   for (int i = 0; i < NEQ; i++) face_at<NEQ>(F, fid, i) = v[i];
}

// Pass 1 of the hybrid scheme: the hybrid sensor of every face; faces that
// need TENO are appended to a compacted list.  A block takes 256 PT faces (4096)
// and reserves its list range with one atomic (one per wave would serialise some
// 10^5 atomics on one address).  The TENO passes gather the six stencil
// points of every listed face, so the list keeps faces that share stencil
// rows together: for the y and z sweeps a block's faces are a tile of TX = 16
// x-cells x TJ = 2 PT faces along the sweep x 8 cells of the remaining direction
// (a wave takes four x-rows of the tile); for the x sweep, whose stencil runs
// along the row, 256 PT consecutive face ids.  A box too small to give every CU
// a block of 4096 faces takes PT = 4 or 1 in place of 16 (a block's atomic costs 12
// ns in line with the others', a round of dependent loads 1 us): ten blocks of
// sixteen rounds took 19.8 us for the x faces of a 200^2 box, in tiles of 256 it
// takes 4.0; 5001-cell tube 16.8 -> 3.5 us.

template<int DIR, int PT, int TX = 16, int TJ = 2*PT>
struct ClsTiles {
   static constexpr int B = Faces<DIR>::B;
   static constexpr uint32_t FACES = 256*PT;
   static constexpr int TB = FACES/(TX*TJ);
   static_assert(TX*TJ*TB == FACES && (TX & (TX - 1)) == 0 && (TJ & (TJ - 1)) == 0, "tile of 256 PT faces");
   static constexpr int LX = (TX == 64) ? 6 : (TX == 32) ? 5 : (TX == 16) ? 4 : 3;
   static constexpr int LJ = (TJ == 64) ? 6 : (TJ == 32) ? 5 : (TJ == 16) ? 4 : (TJ == 8) ? 3 : (TJ == 4) ? 2 : 1;
   __host__ __device__ static uint32_t ntx(const Geo &g) { return ((uint32_t)g.esz[0] + TX - 1u)/TX; }
   __host__ __device__ static uint32_t ntj(const Geo &g) { return ((uint32_t)g.esz[DIR] + TJ)/TJ; }
   __host__ __device__ static uint32_t ntb(const Geo &g) { return ((uint32_t)g.esz[B] + TB - 1u)/TB; }
   static int64_t blocks(const Geo &g, int64_t nfaces)
   {
      if (DIR == 0) return (nfaces + FACES - 1)/FACES;
      return (int64_t)ntx(g)*ntj(g)*ntb(g);
   }
   // face id of element e (0..FACES - 1) of block b; false past the rect
   __device__ static bool face(const Geo &g, int64_t nfaces, uint32_t b, uint32_t e, uint32_t &fid)
   {
      if (DIR == 0) {
         const int64_t id = (int64_t)b*FACES + e;
         fid = (uint32_t)id;
         return id < nfaces;
      }
      const uint32_t nx = ntx(g), nj = ntj(g);
      const uint32_t tx = b % nx, r = b/nx, tj = r % nj, tb = r/nj;
      const uint32_t x = tx*TX + (e & (TX - 1u)), j = tj*TJ + ((e >> LX) & (TJ - 1u)), c = tb*TB + (e >> (LX + LJ));
      if (x >= (uint32_t)g.esz[0] || j > (uint32_t)g.esz[DIR] || c >= (uint32_t)g.esz[B]) return false;
      fid = j*((uint32_t)g.esz[0]*(uint32_t)g.esz[B]) + x + c*(uint32_t)g.esz[0];
      return true;
   }
};

template<class MX, int DIR, int PT>
__global__ void __launch_bounds__(256)
euler_classify_kernel(const htr_fields f, const Geo g, int64_t nfaces, int32_t *__restrict__ list,
                      int *__restrict__ counter)
{
   __shared__ int wave_count[4];
   __shared__ int block_base;
   const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
   uint32_t flags = 0;
   int before = 0;                    // TENO faces of this wave in earlier rounds
   uint64_t masks[PT];
#pragma unroll
   for (int k = 0; k < PT; k++) {
      uint32_t fid;
      bool teno = false;
      if (ClsTiles<DIR, PT>::face(g, nfaces, blockIdx.x, k*256 + threadIdx.x, fid)) {
         const P3 q = Faces<DIR>::cell(g, f, fid);
         teno = !hybrid_kg<DIR>(f, g, q, ld<int>(f.nType[DIR], q));
      }
      masks[k] = __ballot(teno);
      if (teno) flags |= 1u << k;
      before += __popcll(masks[k]);
   }
   if (lane == 0) wave_count[wv] = before;
   __syncthreads();
   if (threadIdx.x == 0) {
      const int total = wave_count[0] + wave_count[1] + wave_count[2] + wave_count[3];
      block_base = total ? atomicAdd(counter, total) : 0;
   }
   __syncthreads();
   int base = block_base;
   for (int w = 0; w < wv; w++) base += wave_count[w];
   const uint64_t lt = (1ull << lane) - 1ull;
#pragma unroll
   for (int k = 0; k < PT; k++) {
      if (flags & (1u << k)) {
         uint32_t fid = 0;
         ClsTiles<DIR, PT>::face(g, nfaces, blockIdx.x, k*256 + threadIdx.x, fid);
         list[base + __popcll(masks[k] & lt)] = (int32_t)fid;
      }
      base += __popcll(masks[k]);
   }
}

// ---- Kennedy-Gruber faces of a cell, divergence fused ------------------------
// KGFluxReconstruction (rhs.inl:79-135) of the face on the plus side of cell p
// is the sum over spans l+1 = 1..3 and shifts m <= l of the pair sums
// S(p-m, p-m+l+1), l outer, m inner.  A thread forms both faces of its cell
// along every direction of the launch from the seven cells p-3..p+3 of the
// line, in the reference's order (nine distinct pairs serve the two faces),
// and adds (F+ - F-) m_e to Conserved_t, which it reads and writes once for
// all directions; TENO faces of the hybrid scheme come from the face buffers
// the TENO passes wrote.
//
// Forming every face twice costs 1000 FP64 operations per cell instead of
// 500, which is little beside what it removes.  The walks along the lines
// that this replaces (a pass per direction and component group, the ring of
// pair sums carried in registers) read and wrote Conserved_t three times and
// the stencil fields six times, and each thread took the faces of its segment
// one after another, node type -> table -> sensor -> flux -> Conserved_t, as
// a chain of dependent loads: they waited 88 % of their cycles.  Here the
// loads of a component are independent of each other, no thread waits for
// another, and a small box has a thread per cell instead of one per eight.
// Bound by the number of loads: a 64-lane 8-byte load takes the CU's address
// unit 16 cycles (measured, from L1, contiguous or not), and a wave of 64 cells
// issues 335 (counted, 256^3 air), 5400 of the 8700 cycles that a CU has for them;
// the rest is L2 latency at three waves per SIMD.
// All three directions, measured with the walks in brackets: 256^3 air 3.9
// (5.0) ms, 512x256x128 boundary layer 2.9 (4.6) ms, 32^3 one species 15 (155)
// us; one direction of 256^3 air without TENO faces 1.2 (1.66) ms.
struct KGFaces { const double *f[3]; };      // face buffers of the directions' TENO faces

// hybrid sensor of a face (rhs.inl:818-820) from the sensors of the cells
// before, at and after its left cell, whose node type is t: the stencil
// offsets of a node type are 0 or the natural ones
__device__ __forceinline__ bool face_is_kg(int t, bool sm, bool s0, bool sp)
{
   return (t == L_S_node || t == L_C_node || sm) && s0 && (t == R_S_node || t == R_C_node || sp);
}

template<class MX, int DIR, bool ALL_KG, bool SOA>
__device__ __forceinline__ void kg_dir(const htr_fields &f, const Geo &g, const htr_view &hv,
                                       const double *__restrict__ F, const P3 &p, double *ct, const htr_view &dec)
{
   constexpr int NS = MX::NS, NEQ = MX::NEQ;
   constexpr int Z = 3;                              // index of the cell itself
   uint32_t o[7];
   {
      int c = p.c[DIR];
      o[Z] = p.o;
#pragma unroll
      for (int k = 1; k <= 3; k++) { o[Z+k] = o[Z+k-1]; step_up(g, DIR, c, o[Z+k]); }
      c = p.c[DIR];
#pragma unroll
      for (int k = 1; k <= 3; k++) { o[Z-k] = o[Z-k+1]; step_down(g, DIR, c, o[Z-k]); }
   }
   const int t = ldo<int, SOA>(f.nType[DIR], o[Z]), tm = ldo<int, SOA>(f.nType[DIR], o[Z-1]);
   const double m = ldo<double, SOA>(f.m_e[DIR], o[Z]);
   // the minus face of a line's first cell is the face of p + offM1(nType)
   // (rhs.inl:800-817): the previous cell's, but the cell's own at a left
   // boundary node
   const bool first = p.c[DIR] == g.elo[DIR];
   const bool own = first && (t == L_S_node || t == L_C_node);
   bool kgp = true, kgm = true;
   if constexpr (!ALL_KG) {
      const bool s2 = ldo<uint8_t, SOA>(f.shockSensor[DIR], o[Z-2]), s1 = ldo<uint8_t, SOA>(f.shockSensor[DIR], o[Z-1]),
                 s0 = ldo<uint8_t, SOA>(f.shockSensor[DIR], o[Z]), sp = ldo<uint8_t, SOA>(f.shockSensor[DIR], o[Z+1]);
      kgp = face_is_kg(t, s1, s0, sp);
      kgm = own ? kgp : face_is_kg(tm, s2, s1, s0);
   }
   if (dec.ptr) {
      if (kgp) *ptr_o<uint32_t, SOA>(dec, o[Z]) = 1;
      if (first && kgm) *ptr_o<uint32_t, SOA>(dec, own ? o[Z] : o[Z-1]) = 1;
   }
   // span sums of a face: sixth order inside, a boundary node type has fewer
   // spans and the coefficients of that order
   const bool std = wave_all(t == Std_node && tm == Std_node);
   int op = 3, om = 3;
   if (!std) { op = c_st.KOrder[t]; om = c_st.KOrder[tm]; }
   auto spans = [&](int order, double a, double b, double c) {
      if (std) {
         double l = (3.0/4.0)*a;
         l += (-3.0/20.0)*b;
         l += (1.0/60.0)*c;
         return l;
      }
      double l = (order > 0) ? (order > 2 ? 3.0/4.0 : order > 1 ? 2.0/3.0 : 0.5)*a : 0.0;
      if (order > 1) l += (order > 2 ? -3.0/20.0 : -1.0/12.0)*b;
      if (order > 2) l += (1.0/60.0)*c;
      return l;
   };
   // faces whose flux is not the split form's: TENO faces, from the face
   // buffer, and those of staggered nodes (rhs.inl:92-110), from the cell they
   // lie on
   const bool sgp = kgp && (t == L_S_node || t == Rm1_S_node), sgm = kgm && (tm == L_S_node || tm == Rm1_S_node);
   const bool others = !wave_all(kgp && kgm && !sgp && !sgm);
   uint32_t fid = 0;
   if constexpr (!ALL_KG) {
      constexpr int A = Faces<DIR>::A, B = Faces<DIR>::B;
      const uint32_t line = (uint32_t)(p.c[A] - g.elo[A]) + (uint32_t)(p.c[B] - g.elo[B])*(uint32_t)g.esz[A];
      fid = Faces<DIR>::id(g, line, p.c[DIR] - g.elo[DIR] + 1);
   }
   auto take = [&](bool kg, bool stag, uint32_t id, uint32_t q, int i, double &fl) {
      if (!kg) {
         fl = face_ld<NEQ>(F, id, i);
      } else if (stag) {
         const double u = ldo<double, SOA>(f.velocity, q, DIR);
         fl = -(ldo<double, SOA>(f.Conserved, q, i)*u);
         if (i == NS + DIR) fl -= ldo<double, SOA>(f.pressure, q);
         if (i == NS + 3) fl -= ldo<double, SOA>(f.pressure, q)*u;
      }
   };
   // (rho_a + rho_b)(-(u_a + u_b)) of the pairs: plus face (0,1) (0,2) (-1,1)
   // (0,3) (-1,2) (-2,1), minus face (-1,0) (-1,1) (-2,0) (-1,2) (-2,1) (-3,0)
   double rv[9];
   {
      double r[7], u[7];
#pragma unroll
      for (int k = 0; k < 7; k++) { r[k] = ldo<double, SOA>(f.rho, o[k]); u[k] = ldo<double, SOA>(f.velocity, o[k], DIR); }
      auto prod = [&](int a, int b) { return (r[Z+a] + r[Z+b])*(-(u[Z+a] + u[Z+b])); };
      rv[0] = prod(0, 1);  rv[1] = prod(0, 2);  rv[2] = prod(-1, 1);
      rv[3] = prod(0, 3);  rv[4] = prod(-1, 2); rv[5] = prod(-2, 1);
      rv[6] = prod(-1, 0); rv[7] = prod(-2, 0); rv[8] = prod(-3, 0);
   }
   // the two faces' span sums of one component: S(a, b) = rv(a, b) (v_a + v_b),
   // or v_a + v_b alone for the pressure
   auto faces = [&](const double *v, bool weighted, double &lp, double &lm) {
      auto S = [&](int k, int a, int b) { const double s = v[Z+a] + v[Z+b]; return weighted ? rv[k]*s : s; };
      const double p1 = S(0, 0, 1), p2 = S(1, 0, 2), q = S(2, -1, 1), p3 = S(3, 0, 3), a4 = S(4, -1, 2), a5 = S(5, -2, 1);
      const double m1 = S(6, -1, 0), m2 = S(7, -2, 0), m3 = S(8, -3, 0);
      lp = spans(op, p1, p2 + q, (p3 + a4) + a5);
      lm = spans(om, m1, q + m2, (a4 + a5) + m3);
   };
#pragma unroll
   for (int i = 0; i < NEQ; i++) {
      double v[7], lp, lm;
#pragma unroll
      for (int k = 0; k < 7; k++)
         v[k] = (i < NS) ? ldo<double, SOA>(f.MassFracs, o[k], i)
              : (i < NS + 3) ? ldo<double, SOA>(f.velocity, o[k], i - NS) : ldo<double, SOA>(hv, o[k]);
      faces(v, true, lp, lm);
      double gp = 0.25*lp, gm = 0.25*lm;
      if (i == NS + DIR) {
#pragma unroll
         for (int k = 0; k < 7; k++) v[k] = ldo<double, SOA>(f.pressure, o[k]);
         faces(v, false, lp, lm);
         gp -= lp;
         gm -= lm;
      }
      if (others) {
         take(kgp, sgp, fid, t == L_S_node ? o[Z] : o[Z+1], i, gp);
         take(kgm, sgm, fid - Faces<DIR>::id(g, 0, 1), tm == L_S_node ? o[Z-1] : o[Z], i, gm);
      }
      if (own) gm = gp;
      ct[i] += (gp - gm)*m;
      // the sums are formed here, component by component: left to itself the
      // compiler issues the loads of all components and directions first and
      // holds 220 registers
      HTR_PIN(ct[i]);
   }
}

template<class MX, int DIRS, bool ALL_KG, bool SOA>
__global__ void __launch_bounds__(256)
euler_kg_kernel(const htr_fields f, const Geo g, const htr_view hv, const KGFaces F, uint32_t per, htr_view dec)
{
   P3 p;
   if (!strip_cell(g, per, p)) return;
   double ct[MX::NEQ];
#pragma unroll
   for (int i = 0; i < MX::NEQ; i++) ct[i] = ldo<double, SOA>(f.Conserved_t, p.o, i);
   if constexpr ((DIRS & 4) != 0) kg_dir<MX, 2, ALL_KG, SOA>(f, g, hv, F.f[2], p, ct, dec);
   if constexpr ((DIRS & 2) != 0) kg_dir<MX, 1, ALL_KG, SOA>(f, g, hv, F.f[1], p, ct, dec);
   if constexpr ((DIRS & 1) != 0) kg_dir<MX, 0, ALL_KG, SOA>(f, g, hv, F.f[0], p, ct, dec);
#pragma unroll
   for (int i = 0; i < MX::NEQ; i++) *ptr_o<double, SOA>(f.Conserved_t, p.o, i) = ct[i];
}

// Pass 2: TENO-family faces, either all faces or the compacted list:
//   2a  lane per face: Roe state + eigenvalue maxima -> record
//   2b  a block per 64 faces, face data staged in LDS: split fluxes, TENO +/-,
//       back-projection, limiter test -> face flux, decision word
//   2c  lane per listed face: limiter blend
// Records: NREC*cap doubles, component-major (capacity cap = number of faces).
struct TenoBufs {
   double *rec;
   int64_t cap;
};

template<class MX>
__host__ __device__ inline int64_t teno_doubles(int64_t cap) { return Euler<MX, 0>::NREC*cap; }

template<class MX, int DIR, bool LISTED>
__global__ void __launch_bounds__(256)
euler_roe_kernel(const htr_fields f, const DMix *__restrict__ mix, const Geo g, const htr_view hv, TenoBufs b, int64_t nfaces,
                 const int32_t *__restrict__ list, const int *__restrict__ counter)
{
   const int64_t n = LISTED ? (int64_t)counter[1] : nfaces;
   const int64_t stride = (int64_t)gridDim.x*blockDim.x;
   Euler<MX, DIR> E{f, *mix, g, hv};
   for (int64_t w = (int64_t)blockIdx.x*blockDim.x + threadIdx.x; w < n; w += stride) {
      const uint32_t fid = LISTED ? (uint32_t)list[w] : (uint32_t)w;
      const P3 q = Faces<DIR>::cell(g, f, fid);
      E.face_record(b.rec, b.cap, w, q, ld<int>(f.nType[DIR], q));
   }
}

// Pass 2b.  A block of four waves takes chunks of 64
// listed TENO faces, a lane per face, in three steps between barriers:
//   stage       the six stencil points, dealt to the waves: the point's
//               values (conserved vector, u_n, p) are gathered and left in
//               LDS with its four species sums of the left-eigenvector
//               products (rhs.inl:443-451), formed once and not again for
//               each of the nine components that use them;
//   components  the nEq components, dealt to the waves (the component index
//               is wave-uniform, so every branch on it is): split fluxes of
//               the six points on row i, TENO+ and TENO-, -(F+ + F-)/2 and
//               the stencil-selection bits into LDS;
//   finish      the last wave, before it stages the next chunk:
//               back-projection (add_column, the reference's summation
//               order), limiter test, face fluxes, decision words, and the
//               list of the faces that need the limiter blend.
// The steps of a block do not overlap; the three blocks of a CU (52 KB of LDS
// each) do, and no wave is kept for loading alone.  Bound by the latency of
// the gathers: its waves wait 74 % of their cycles.  256^3 air, per y or z
// sweep (3.36 M TENO faces): 2.17 ms, against 2.38 ms with the sums formed per
// component and the gathers of a loading wave overlapped; 128^3 with 85 % TENO
// faces 0.81 against 0.97 ms.
constexpr int TENO_WAVES = 4;

template<class MX>
struct TenoStage {
   static constexpr int NS = MX::NS, NEQ = MX::NEQ;
   // per point: rhoY_0..NS-1, rhou 3, rhoE, u_n, p, then the species sums of
   // the conserved vector (weighted, plain) and of the flux
   static constexpr int UN = NS + 4, PR = NS + 5, S1Q = NS + 6, SQQ = NS + 7, S1F = NS + 8, SQF = NS + 9;
   static constexpr int NPV = NS + 10;
   double  pt[6*NPV][64];
   double  fc[NEQ][64];
   double  w[16][4];                                // StdWeights
   uint8_t bits[NEQ][64];
};

template<class MX, int DIR, int SCHEME, bool LISTED>
__global__ void __launch_bounds__(64*TENO_WAVES)
euler_teno_kernel(const htr_fields f, const DMix *__restrict__ mix, const Geo g, const htr_view hv, TenoBufs b,
                  double RK0, double RK1, DtArg dta, double *__restrict__ F, int64_t nfaces,
                  const int32_t *__restrict__ list, const int *__restrict__ counter, htr_view dec,
                  int32_t *__restrict__ llist, int *__restrict__ lcount)
{
   using E_t = Euler<MX, DIR>;
   using St = TenoStage<MX>;
   constexpr int NS = MX::NS, NEQ = MX::NEQ, NPV = St::NPV;
   constexpr int OP = (SCHEME == HTR_EULER_TENOA) ? 1 : (SCHEME == HTR_EULER_TENOLAD) ? 2 : 0;
   constexpr int iN = E_t::iN;
   constexpr int LAST = TENO_WAVES - 1;
   __shared__ St S;
   const uint32_t n = (uint32_t)(LISTED ? (int64_t)counter[1] : nfaces);
   const uint32_t nchunks = (n + 63u)/64u;
   const int lane = threadIdx.x & 63;
   const int wv = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
   const int64_t cap = b.cap;
   E_t E{f, *mix, g, hv};
   // chunks of this block: L + k gridDim.x, with L the XCD-aware logical block
   // index (the chunks in flight on one XCD are neighbours in the list and
   // share stencil cache lines)
   const uint32_t L = xcd_block(blockIdx.x, gridDim.x);
   if (L >= nchunks) return;                         // uniform over the block
   const double dt = dta.get();
   if (threadIdx.x < 64) S.w[lane >> 2][lane & 3] = c_stdw.w[lane >> 2][lane & 3];

   // face id, left cell and node type of the lane's face of chunk c; past the
   // list's end the first cell stands in (its values are not used)
   uint32_t fid = 0;
   P3 q;
   int t = 0;
   auto face = [&](uint32_t c) {
      const uint32_t w = c*64u + (uint32_t)lane;
      fid = 0;
      t = Std_node;
      q = mkp(g, 0, 0, 0);
      if (w < n) {
         fid = LISTED ? (uint32_t)list[w] : w;
         q = Faces<DIR>::cell(g, f, fid);
         t = ld<int>(f.nType[DIR], q);
      }
   };

   // back-projection, limiter test, face flux and decision word of the lane's
   // face of chunk c (rhs.inl:708-721)
   auto finish = [&](uint32_t c) {
      const uint32_t w = c*64u + (uint32_t)lane;
      bool limit = false;
      if (w < n) {
         typename E_t::Roe R;
         E_t::get_rec(b.rec, cap, w, R);
         const double dedp = 1.0/R.dpde;
         const double ERoe = R.e + 0.5*E_t::mod2(R.v);
         double Flux[NEQ];
         double sumQsp = 0.0;
         uint32_t h = 0;
#pragma unroll
         for (int i = 0; i < NEQ; i++) {
            E_t::add_column(Flux, sumQsp, i, S.fc[i][lane], R, ERoe, dedp);
            const uint32_t bt = S.bits[i][lane];
            h = fold_bits(fold_bits(h, bt & 15u), bt >> 4);
         }
         if (NS > 1) {
            const P3 pP1 = wplus(g, DIR, q, c_st.Cp[t][2]);
            const double lim_f = dt*(ld<double>(f.m_e[DIR], q) + ld<double>(f.m_e[DIR], pP1));
#pragma unroll
            for (int i = 0; i < NS; i++) {
               const double dRhoi = lim_f*Flux[i];
               if (((RK0*ld<double>(f.Conserved_old, q, i) + RK1*ld<double>(f.Conserved, q, i) + dRhoi) < -1e-8) ||
                   ((RK0*ld<double>(f.Conserved_old, pP1, i) + RK1*ld<double>(f.Conserved, pP1, i) - dRhoi) < -1e-8))
                  limit = true;
            }
         }
         store_face<NEQ>(F, nfaces, fid, Flux);
         if (dec.ptr) at<uint32_t>(dec, q) = h << 2;
      }
      const uint64_t mask = __ballot(limit);
      if (mask) {
         const int leader = __ffsll((unsigned long long)mask) - 1;
         int base = 0;
         if (lane == leader) base = atomicAdd(lcount, __popcll(mask));
         base = __shfl(base, leader, 64);
         if (limit) llist[base + __popcll(mask & ((1ull << lane) - 1ull))] = (int32_t)w;
      }
   };

   for (uint32_t c = L; c < nchunks; c += gridDim.x) {
      if (wv == LAST && c != L) finish(c - gridDim.x);
      face(c);
      const uint32_t w = c*64u + (uint32_t)lane;
      const uint32_t wr = w < n ? w : n - 1u;        // a record that exists
      typename E_t::Roe R;
      typename E_t::Proj J;
#pragma unroll
      for (int j = 0; j < 3; j++) R.v[j] = b.rec[(int64_t)(NS + j)*cap + wr];
      R.a = b.rec[(int64_t)(NS + 3)*cap + wr];
      R.e = b.rec[(int64_t)(NS + 5)*cap + wr];
      R.rho = b.rec[(int64_t)(NS + 6)*cap + wr];
      R.dpde = b.rec[(int64_t)(NS + 7)*cap + wr];
      R.a2 = b.rec[(int64_t)(2*NS + 8)*cap + wr];
      double dpdrhoi[NS];
#pragma unroll
      for (int j = 0; j < NS; j++) dpdrhoi[j] = b.rec[(int64_t)(NS + 8 + j)*cap + wr];
      for (int k = wv; k < 6; k += TENO_WAVES) {
         const int off = (k == 2) ? 0 : c_st.Cp[t][k - (k > 2 ? 1 : 0)];
         const P3 P = wplus(g, DIR, q, off);
         double pv[NS + 6];
#pragma unroll
         for (int v = 0; v < NS + 6; v++)
            pv[v] = (v < NS + 4) ? ld<double>(f.Conserved, P, v)
                  : (v == NS + 4) ? ld<double>(f.velocity, P, iN) : ld<double>(f.pressure, P);
         if (k == wv) E_t::proj(J, R);
         double (*pt)[64] = &S.pt[k*NPV];
         double s1q = 0.0, sqq = 0.0, s1f = 0.0, sqf = 0.0;
#pragma unroll
         for (int j = 0; j < NS; j++) {
            const double wj = (J.Coeff - dpdrhoi[j])*J.iaRoe2;
            s1q += wj*pv[j];
            sqq += pv[j];
            const double fq = pv[j]*pv[St::UN];
            s1f += wj*fq;
            sqf += fq;
         }
#pragma unroll
         for (int v = 0; v < NS + 6; v++) pt[v][lane] = pv[v];
         pt[St::S1Q][lane] = s1q;
         pt[St::SQQ][lane] = sqq;
         pt[St::S1F][lane] = s1f;
         pt[St::SQF][lane] = sqf;
      }
      __syncthreads();
      const bool all_std = __ballot(t != Std_node) == 0ull;
      for (int i = wv; i < NEQ; i += TENO_WAVES) {
         // the point values are re-read from LDS for every component
         asm volatile("" ::: "memory");
         const double lam = b.rec[(int64_t)(2*NS + ((i == 0) ? 9 : (i == NEQ-1) ? 11 : 10))*cap + wr];
         const double Ysel = (i >= 1 && i <= NS) ? b.rec[(int64_t)(i - 1)*cap + wr] : 0.0;
         double vp[6], vm[6];
#pragma unroll
         for (int k = 0; k < 6; k++) {
            const double (*pt)[64] = &S.pt[k*NPV];
            const double un = pt[St::UN][lane], pr = pt[St::PR][lane];
            const double qs = (i >= 1 && i <= NS) ? pt[i - 1][lane] : 0.0;
            double qm[4], fm[4];
#pragma unroll
            for (int j = 0; j < 4; j++) { qm[j] = pt[NS + j][lane]; fm[j] = qm[j]*un; }
            fm[iN] += pr;
            fm[3] += pr*un;
            const double Q = E_t::char_row(i, R, J, pt[St::S1Q][lane], pt[St::SQQ][lane], qs, qm, Ysel);
            const double Fv = E_t::char_row(i, R, J, pt[St::S1F][lane], pt[St::SQF][lane], qs*un, fm, Ysel);
            vp[k] = Fv + lam*Q;
            vm[k] = Fv - lam*Q;
         }
         uint32_t bp, bm;
         double FPlus, FMinus;
         if (all_std) {
            FPlus  = teno_reconstruct<OP, 0, true>(vp, t, &bp, S.w);
            FMinus = teno_reconstruct<OP, 1, true>(vm, t, &bm, S.w);
         } else {
            FPlus  = teno_reconstruct<OP, 0>(vp, t, &bp, S.w);
            FMinus = teno_reconstruct<OP, 1>(vm, t, &bm, S.w);
         }
         S.fc[i][lane] = -0.5*(FPlus + FMinus);
         S.bits[i][lane] = (uint8_t)(bp | (bm << 4));
      }
      __syncthreads();
   }
   if (wv == LAST) finish(L + (nchunks - 1u - L)/gridDim.x*gridDim.x);
}

template<class MX, int DIR, bool LISTED>
__global__ void __launch_bounds__(256)
euler_limit_kernel(const htr_fields f, const DMix *__restrict__ mix, const Geo g, const htr_view hv,
                   double RK0, double RK1, DtArg dta, TenoBufs b, double *__restrict__ F, int64_t nfaces,
                   const int32_t *__restrict__ list, const int32_t *__restrict__ llist,
                   const int *__restrict__ lcount, htr_view dec)
{
   const int64_t n = *lcount;
   const int64_t stride = (int64_t)gridDim.x*blockDim.x;
   Euler<MX, DIR> E{f, *mix, g, hv};
   for (int64_t k = (int64_t)blockIdx.x*blockDim.x + threadIdx.x; k < n; k += stride) {
      const int64_t w = llist[k];
      const uint32_t fid = LISTED ? (uint32_t)list[w] : (uint32_t)w;
      const P3 q = Faces<DIR>::cell(g, f, fid);
      double Flux[MX::NEQ];
#pragma unroll
      for (int i = 0; i < MX::NEQ; i++) Flux[i] = face_ld<MX::NEQ>(F, fid, i);
      E.face_limit(Flux, b.rec, b.cap, w, q, ld<int>(f.nType[DIR], q), RK0, RK1, dta.get());
      store_face<MX::NEQ>(F, nfaces, fid, Flux);
      if (dec.ptr) at<uint32_t>(dec, q) |= 2u;
   }
}

// Pass 3: Conserved_t[p] += (F(p) - F(p - 1))*m_e[p] (rhs.inl:876-887), one
// lane per cell of the execution rect.
template<int NEQ, int DIR>
__global__ void __launch_bounds__(256)
face_divergence_kernel(const htr_fields f, const Geo g, const double *__restrict__ F, int64_t nfaces,
                       const htr_view metric, int64_t ncells)
{
   const int64_t i = (int64_t)blockIdx.x*blockDim.x + threadIdx.x;
   if (i >= ncells) return;
   const P3 p = exec_point(g, i);
   constexpr int A = Faces<DIR>::A, B = Faces<DIR>::B;
   const uint32_t line = (uint32_t)(p.c[A] - g.elo[A]) + (uint32_t)(p.c[B] - g.elo[B])*(uint32_t)g.esz[A];
   const int j = p.c[DIR] - g.elo[DIR] + 1;
   const uint32_t fp = Faces<DIR>::id(g, line, j);
   const uint32_t fm = Faces<DIR>::id(g, line, j - 1);
   const double m = ld<double>(metric, p);
#pragma unroll
   for (int c = 0; c < NEQ; c++)
      at<double>(f.Conserved_t, p, c) += (face_ld<NEQ>(F, fp, c) - face_ld<NEQ>(F, fm, c))*m;
}

// Blocks of the TENO component kernel: persistent, three per CU (what the LDS
// and registers of one block allow), each looping over chunks.
// HTR_TENO_BLOCKS=n caps the grid at n blocks (tuning; a small cap makes
// every block take many chunks).
static int teno_blocks()
{
   static int cap = -1;
   if (cap < 0) {
      int v = 256*3;
      if (const char *e = getenv("HTR_TENO_BLOCKS")) { const int x = atoi(e); if (x > 0) v = x; }
      cap = v;
   }
   return cap;
}

template<class MX, int DIR, int SCHEME, bool LISTED>
static int launch_teno(const htr_fields &f, const DMix *mix, const Geo &g, const htr_view &hv, double RK0,
                       double RK1, const DtArg &dt, Workspace &w, int64_t nfaces, double *F, const htr_view &dec,
                       hipStream_t s)
{
   constexpr int kMaxBlocks = 256*16;
   const TenoBufs b{ w.teno, nfaces };
   const unsigned nb = (unsigned)std::min<int64_t>(grid_for(nfaces, 256), kMaxBlocks);
   HTR_LAUNCH(HTR_DIR_NAME("euler_roe", DIR), (euler_roe_kernel<MX, DIR, LISTED>), dim3(nb), dim3(256), 0, s,
                      f, mix, g, hv, b, nfaces, w.list, w.counter);
   int rc = check_launch("euler_roe_kernel"); if (rc) return rc;
   int32_t *llist = w.list + nfaces;                  // limiter list after the TENO list
   const unsigned nchunk = (unsigned)std::min<int64_t>((nfaces + 63)/64, teno_blocks());
   HTR_LAUNCH(HTR_DIR_NAME("euler_teno", DIR), (euler_teno_kernel<MX, DIR, SCHEME, LISTED>), dim3(nchunk),
              dim3(64*TENO_WAVES), 0, s, f, mix, g, hv, b, RK0, RK1, dt, F, nfaces, w.list, w.counter, dec,
              llist, w.counter + 2);
   if ((rc = check_launch("euler_teno_kernel"))) return rc;
   if (MX::NS == 1) return HTR_OK;                   // single species: no positivity limiter
   HTR_LAUNCH(HTR_DIR_NAME("euler_limit", DIR), (euler_limit_kernel<MX, DIR, LISTED>), dim3(256), dim3(256), 0, s,
              f, mix, g, hv, RK0, RK1, dt, b, F, nfaces, w.list, llist, w.counter + 2, dec);
   return check_launch("euler_limit_kernel");
}

// The TENO faces of the hybrid sweep along DIR into the face buffer F:
// classification into the compacted list, Roe records, components and
// back-projection, limiter blend (the KG faces are left to the caller).
template<class MX, int DIR>
static int teno_faces(const htr_fields &f, const DMix *mix, const Geo &g, const htr_view &hv, double RK0, double RK1,
                      const DtArg &dt, Workspace &w, int64_t nfaces, double *F, const htr_view &dec, hipStream_t s)
{
   int rc = zero_counters(w.counter, s);        // TENO list and limiter list counts
   if (rc) return rc;
   auto classify = [&](auto pt) {
      constexpr int PT = decltype(pt)::value;
      HTR_LAUNCH(HTR_DIR_NAME("euler_classify", DIR), (euler_classify_kernel<MX, DIR, PT>),
                 dim3((unsigned)ClsTiles<DIR, PT>::blocks(g, nfaces)), dim3(256), 0, s, f, g, nfaces, w.list, w.counter + 1);
   };
   if (nfaces >= 256*4096)      classify(std::integral_constant<int, 16>());
   else if (nfaces >= 256*1024) classify(std::integral_constant<int, 4>());
   else                         classify(std::integral_constant<int, 1>());
   if ((rc = check_launch("euler_classify_kernel"))) return rc;
   return launch_teno<MX, DIR, HTR_EULER_TENO, true>(f, mix, g, hv, RK0, RK1, dt, w, nfaces, F, dec, s);
}

// The KG faces and the fused divergence of the sweeps DIRS (bit d: direction
// d) of a hybrid (or pure KG, ALL) scheme, in the order z, y, x; the listed TENO
// faces are read back from F
template<class MX, int DIRS, bool ALL>
static int kg_cells(const htr_fields &f, const Geo &g, const htr_view &hv, const KGFaces &F, const htr_view &dec,
                    hipStream_t s)
{
   const StripGrid sg(g);
   const char *name = (DIRS == 7) ? "euler_kg" : (DIRS == 1) ? "euler_kg_x" : (DIRS == 2) ? "euler_kg_y" : "euler_kg_z";
   if (g.soa) {
      HTR_LAUNCH(name, (euler_kg_kernel<MX, DIRS, ALL, true>), dim3(sg.blocks), dim3(256), 0, s, f, g, hv, F, sg.per, dec);
   } else {
      HTR_LAUNCH(name, (euler_kg_kernel<MX, DIRS, ALL, false>), dim3(sg.blocks), dim3(256), 0, s, f, g, hv, F, sg.per, dec);
   }
   return check_launch("euler_kg_kernel");
}

// the caller's total-enthalpy array (workspace of stream s) as a view
static int enthalpy_view(const Geo &g, Workspace &w, htr_view &hv)
{
   const int64_t span = ((int64_t)g.bsz[0] - 1)*g.cb[0] + ((int64_t)g.bsz[1] - 1)*g.cb[1] +
                        ((int64_t)g.bsz[2] - 1)*g.cb[2] + 1;
   int rc = workspace_enthalpy(w, span);
   if (rc) return rc;
   hv = {};
   hv.ptr = w.hbuf;
   hv.sx = 8;                                  // one double per base element (k = 1)
   return HTR_OK;
}

template<class MX, int DIR, int SCHEME>
static int launch_dir(const htr_fields &f, const DMix *mix, const Geo &g, double RK0, double RK1,
                      const DtArg &dt, const htr_view &dec, hipStream_t s, bool enthalpy_ready)
{
   const int64_t ncells = exec_cells(g);
   if (ncells == 0) return HTR_OK;
   const int64_t nfaces = Faces<DIR>::count(g);
   if (nfaces*MX::NEQ >= (1ll << 31)) return set_error(HTR_E_UNSUPPORTED, "euler: too many faces");
   Workspace *wp = workspace(s);
   if (!wp) return HTR_E_DEVICE;
   Workspace &w = *wp;
   int rc = workspace_faces(w, SCHEME == HTR_EULER_KG ? 0 : nfaces*MX::NEQ, SCHEME == HTR_EULER_KG ? 0 : 2*nfaces,
                            SCHEME == HTR_EULER_KG ? 0 : teno_doubles<MX>(nfaces));
   if (rc) return rc;
   // total enthalpy of every cell of the bounds
   const int64_t nb_cells = (int64_t)g.bsz[0]*g.bsz[1]*g.bsz[2];
   htr_view hv;
   if ((rc = enthalpy_view(g, w, hv))) return rc;
   if (!enthalpy_ready) {
      HTR_LAUNCH("enthalpy", (enthalpy_kernel<MX>), dim3(grid_for(nb_cells, 256)), dim3(256), 0, s, f, g, hv, nb_cells);
      if ((rc = check_launch("enthalpy_kernel"))) return rc;
   }
   if constexpr (SCHEME != HTR_EULER_KG && SCHEME != HTR_EULER_HYBRID) {
      if ((rc = zero_counters(w.counter, s))) return rc;    // limiter list count
   }
   if constexpr (SCHEME == HTR_EULER_HYBRID) {
      if ((rc = teno_faces<MX, DIR>(f, mix, g, hv, RK0, RK1, dt, w, nfaces, w.faces, dec, s))) return rc;
   }
   if constexpr (SCHEME == HTR_EULER_HYBRID || SCHEME == HTR_EULER_KG) {
      KGFaces F = {};
      F.f[DIR] = w.faces;
      return kg_cells<MX, 1 << DIR, SCHEME == HTR_EULER_KG>(f, g, hv, F, dec, s);
   } else {
      if ((rc = launch_teno<MX, DIR, SCHEME, false>(f, mix, g, hv, RK0, RK1, dt, w, nfaces, w.faces, dec, s))) return rc;
      HTR_LAUNCH(HTR_DIR_NAME("euler_divergence", DIR), (face_divergence_kernel<MX::NEQ, DIR>), dim3(grid_for(ncells, 256)),
                 dim3(256), 0, s, f, g, w.faces, nfaces, f.m_e[DIR], ncells);
      return check_launch("face_divergence_kernel");
   }
}

// Face buffers of the three sweeps of a full right-hand side, one after the
// other in one workspace
template<class MX>
static int64_t rhs_face_base(const Geo &g, int d)
{
   int64_t n = 0;
   if (d < 2) n += Faces<2>::count(g);
   if (d < 1) n += Faces<1>::count(g);
   if (d < 0) n += Faces<0>::count(g);
   return n*MX::NEQ;
}

template<class MX, int DIR>
static int rhs_teno(const htr_fields &f, const DMix *mix, const Geo &g, double RK0, double RK1, const DtArg &dt,
                    const htr_view &dec, hipStream_t ts, hipStream_t hs, double *F)
{
   Workspace *tw = workspace(ts), *hw = workspace(hs);
   if (!tw || !hw) return HTR_E_DEVICE;
   const int64_t nfaces = Faces<DIR>::count(g);
   htr_view hv;
   int rc = enthalpy_view(g, *hw, hv);
   if (!rc) rc = workspace_faces(*tw, 0, 2*nfaces, teno_doubles<MX>(nfaces));
   if (rc) return rc;
   return teno_faces<MX, DIR>(f, mix, g, hv, RK0, RK1, dt, *tw, nfaces, F, dec, ts);
}

// The Euler sweeps of a full right-hand side (hybrid or KG), total enthalpy
// formed before.  part 0: the TENO faces of direction dir, on stream ts (the
// list and the records in its workspace), into the face buffer of the
// workspace of s; part 1: KG faces and divergence of the three directions in
// one pass on s.
template<class MX>
int rhs_euler_part(int dir, int part, int scheme, const htr_fields &f, const DMix *mix, const Geo &g, double RK0,
                   double RK1, const DtArg &dt, const htr_view &dec, hipStream_t ts, hipStream_t s)
{
   if (exec_cells(g) == 0) return HTR_OK;
   for (int64_t n : { Faces<0>::count(g), Faces<1>::count(g), Faces<2>::count(g) })
      if (n*MX::NEQ >= (1ll << 31)) return set_error(HTR_E_UNSUPPORTED, "euler: too many faces");
   Workspace *w = workspace(s);
   if (!w) return HTR_E_DEVICE;
   int rc = workspace_faces(*w, scheme == HTR_EULER_KG ? 0 : rhs_face_base<MX>(g, -1), 0, 0);
   if (rc) return rc;
   KGFaces F;
   for (int d = 0; d < 3; d++) F.f[d] = w->faces ? w->faces + rhs_face_base<MX>(g, d) : nullptr;
   if (part == 0) {
      double *Fd = const_cast<double*>(F.f[dir]);
      switch (dir) {
         case 0: return rhs_teno<MX, 0>(f, mix, g, RK0, RK1, dt, dec, ts, s, Fd);
         case 1: return rhs_teno<MX, 1>(f, mix, g, RK0, RK1, dt, dec, ts, s, Fd);
         default: return rhs_teno<MX, 2>(f, mix, g, RK0, RK1, dt, dec, ts, s, Fd);
      }
   }
   htr_view hv;
   if ((rc = enthalpy_view(g, *w, hv))) return rc;
   if (scheme == HTR_EULER_KG) return kg_cells<MX, 7, true>(f, g, hv, F, dec, s);
   return kg_cells<MX, 7, false>(f, g, hv, F, dec, s);
}

template<class MX>
bool rhs_faces_fit(const Geo &g, hipStream_t s)
{
   for (int64_t n : { Faces<0>::count(g), Faces<1>::count(g), Faces<2>::count(g) })
      if (n*MX::NEQ >= (1ll << 31)) return true;      // refused by the sweeps
   Workspace *w = workspace(s);
   return !w || workspace_faces_fit(*w, rhs_face_base<MX>(g, -1));
}

template bool rhs_faces_fit<MixCP>(const Geo &, hipStream_t);
template bool rhs_faces_fit<MixAir>(const Geo &, hipStream_t);

template int rhs_euler_part<MixCP>(int, int, int, const htr_fields &, const DMix *, const Geo &, double, double,
                                   const DtArg &, const htr_view &, hipStream_t, hipStream_t);
template int rhs_euler_part<MixAir>(int, int, int, const htr_fields &, const DMix *, const Geo &, double, double,
                                    const DtArg &, const htr_view &, hipStream_t, hipStream_t);

// Total enthalpy of every cell of the bounds into the stream's workspace
// (once per RHS; the three sweeps then skip it)
template<class MX>
int enthalpy_launch(const htr_fields &f, const Geo &g, hipStream_t s)
{
   Workspace *wp = workspace(s);
   if (!wp) return HTR_E_DEVICE;
   const int64_t nb_cells = (int64_t)g.bsz[0]*g.bsz[1]*g.bsz[2];
   const int64_t span = ((int64_t)g.bsz[0] - 1)*g.cb[0] + ((int64_t)g.bsz[1] - 1)*g.cb[1] +
                        ((int64_t)g.bsz[2] - 1)*g.cb[2] + 1;
   int rc = workspace_enthalpy(*wp, span);
   if (rc) return rc;
   htr_view hv = {};
   hv.ptr = wp->hbuf;
   hv.sx = 8;
   HTR_LAUNCH("enthalpy", (enthalpy_kernel<MX>), dim3(grid_for(nb_cells, 256)), dim3(256), 0, s, f, g, hv, nb_cells);
   return check_launch("enthalpy_kernel");
}

template int enthalpy_launch<MixCP>(const htr_fields &, const Geo &, hipStream_t);
template int enthalpy_launch<MixAir>(const htr_fields &, const Geo &, hipStream_t);

// Workspace sizes of the Euler sweeps (every scheme, every direction) over the
// rect of g.
template<class MX>
WorkspaceNeed euler_workspace_need(const Geo &g)
{
   WorkspaceNeed n;
   auto dir = [&](int64_t nfaces) {
      n.faces += nfaces*MX::NEQ;               // the full right-hand side holds all three
      n.faces_one = std::max(n.faces_one, nfaces*MX::NEQ);
      n.list = std::max(n.list, 2*nfaces);
      n.teno = std::max(n.teno, teno_doubles<MX>(nfaces));
   };
   if (exec_cells(g) == 0) return n;
   dir(Faces<0>::count(g));
   dir(Faces<1>::count(g));
   dir(Faces<2>::count(g));
   n.hbuf = ((int64_t)g.bsz[0] - 1)*g.cb[0] + ((int64_t)g.bsz[1] - 1)*g.cb[1] + ((int64_t)g.bsz[2] - 1)*g.cb[2] + 1;
   return n;
}

template WorkspaceNeed euler_workspace_need<MixCP>(const Geo &);
template WorkspaceNeed euler_workspace_need<MixAir>(const Geo &);
template WorkspaceNeed euler_workspace_need<Mix30>(const Geo &);

template<class MX>
int euler_dispatch(int dir, int scheme, const htr_fields &f, const DMix *mix, const Geo &g,
                   double RK0, double RK1, const DtArg &dt, const htr_view &dec, hipStream_t s,
                   bool enthalpy_ready)
{
#define HTR_E_CASE(D, S) if (dir == D && scheme == S) return launch_dir<MX, D, S>(f, mix, g, RK0, RK1, dt, dec, s, enthalpy_ready);
#define HTR_E_DIRS(S) HTR_E_CASE(0, S) HTR_E_CASE(1, S) HTR_E_CASE(2, S)
   HTR_E_DIRS(HTR_EULER_HYBRID)
   HTR_E_DIRS(HTR_EULER_TENO)
   HTR_E_DIRS(HTR_EULER_TENOA)
   HTR_E_DIRS(HTR_EULER_TENOLAD)
   HTR_E_DIRS(HTR_EULER_KG)
#undef HTR_E_DIRS
#undef HTR_E_CASE
   return set_error(HTR_E_ARG, "euler: bad direction or scheme");
}

template int euler_dispatch<MixCP>(int, int, const htr_fields &, const DMix *, const Geo &, double, double, const DtArg &, const htr_view &, hipStream_t, bool);
template int euler_dispatch<MixAir>(int, int, const htr_fields &, const DMix *, const Geo &, double, double, const DtArg &, const htr_view &, hipStream_t, bool);

} // namespace htr
