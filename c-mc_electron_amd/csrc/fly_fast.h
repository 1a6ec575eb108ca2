// The fast pass of the flight: one particle whose step holds only tetrahedron and
// plain cell crossings (device code, included by kernels.hip).
//
// A step of most particles is a few crossings and the end of the step.  The pass
// follows Flight::fly() for those events and gives the same bits: every value that
// reaches memory is formed by the operations of Flight::next_event and
// Flight::advance in their order.  What differs is what is left out:
//
//  * A scattering is not flown here, so its time is not needed, only that it lies
//    beyond the next crossing.  Each exponent (-log of a uniform) is replaced by a
//    lower bound from the 32-bit hardware logarithm and each rate by an upper
//    bound; where the bounds do not settle it the particle goes to the slow kernel,
//    which redoes it from its stored state with the same random numbers.
//  * Of the seven faces (four of the tetrahedron, three of the cell) only the
//    nearest one's time is divided out.  Quotients from the hardware reciprocal
//    (relative error up to 2^-23, 1.2e-7) find it; a particle with two of them within 1e-6
//    of each other, or of the end of the step, goes to the slow kernel.
//
// What bounds it: the vector-memory return path (texture data unit busy 96 % of the
// kernel, waves waiting 39 % of their life to issue), since each lane gathers its own
// tetrahedron's and cell's records.  With Flight's code a wave also waited for 75 % of
// its life on some dozen dependent reads per event; here every read of an event (the
// tetrahedron's record, the cell's fields, planes and rules) is issued before the
// first use, one round trip an event, and what two reads held alike is read once: 230
// -> 100 loads and 2593 -> 1850 vector instructions a wave, 869 -> 668 us for the 3.0 M
// particles of the 80x160x48-cell step.  Records staged through LDS by direct loads:
// 772 us, a dozen lines per instruction all the same and registers spilled.
#pragma once
#include "fly_core.h"

namespace emc {

typedef double fd2 __attribute__((ext_vector_type(2)));
typedef int fi4 __attribute__((ext_vector_type(4)));

struct FastFlight {
  const EMC_CST BandDev& B;
  const EMC_CST MeshDev& M;
  const EMC_CST FieldsDev& F;
  double x, y, z, kx, ky, kz, energy, left;
  int icell, jcell, kcell, itet, isym, type;
  uint32_t k0, k1, c1, c2;  // the particle's random stream (Rng)
  int n_events, pend_kind, pend_j;

  __device__ FastFlight(const EMC_CST BandDev& b, const EMC_CST MeshDev& m, const EMC_CST FieldsDev& f)
      : B(b), M(m), F(f) {}

  static constexpr int EVENTS = 16;  // crossings and the end of the step
  enum { DONE = 1, BAIL = 2 };

  __device__ static __forceinline__ double flip(double v, uint32_t s) {  // v * (s ? -1 : 1)
    return __builtin_bit_cast(double, __builtin_bit_cast(uint64_t, v) ^ ((uint64_t)s << 63));
  }
  __device__ static __forceinline__ double sel3(uint32_t p, double a, double b, double c) {
    return p == 0 ? a : p == 1 ? b : c;
  }
  // Flight::out_wedge / in_wedge by the packed operation
  __device__ static __forceinline__ void out_wedge(uint32_t w, double& xo, double& yo, double& zo, double a, double b,
                                                   double c) {
    xo = flip(sel3(w & 3u, a, b, c), (w >> 6) & 1u);
    yo = flip(sel3((w >> 2) & 3u, a, b, c), (w >> 7) & 1u);
    zo = flip(sel3((w >> 4) & 3u, a, b, c), (w >> 8) & 1u);
  }
  __device__ static __forceinline__ void in_wedge(uint32_t w, double& xo, double& yo, double& zo, double a, double b,
                                                  double c) {
    const uint32_t p0 = w & 3u, p1 = (w >> 2) & 3u;
    a = flip(a, (w >> 6) & 1u);
    b = flip(b, (w >> 7) & 1u);
    c = flip(c, (w >> 8) & 1u);
    xo = p0 == 0 ? a : p1 == 0 ? b : c;
    yo = p0 == 1 ? a : p1 == 1 ? b : c;
    zo = p0 == 2 ? a : p1 == 2 ? b : c;
  }
  // A lower bound of -log(u) for the draw whose high word is h: u < (h + 1) 2^-32,
  // widened for the rounding of the conversion, the logarithm taken as good to 1e-5.
  __device__ static __forceinline__ double log_bound(uint32_t h) {
    const float u = ((float)h + 1.0f) * 2.3283071e-10f;  // 2^-32 (1 + 3e-7)
    const float l = -0.69314718f * __builtin_amdgcn_logf(u);
    return (double)(l * 0.99999f - 1e-6f);
  }
  // the electrons' or the holes' of two wave-wide words.  The empty asm keeps them
  // in scalar registers: the compiler otherwise selects between their addresses and
  // loads the word per lane, a read that the table read then waits for.
  template <class T>
  __device__ __forceinline__ T pick(T e, T h) const {
    asm("" : "+s"(e));
    asm("" : "+s"(h));
    return type == 0 ? e : h;
  }
  __device__ __forceinline__ void draws(uint32_t block, uint32_t& a, uint32_t& b) const {
    uint32_t c[4] = {block, c1, c2, 0u};
    philox4x32_10(c, k0, k1);
    a = c[1];
    b = c[3];
  }
  // an upper bound of Flight::GetImpScGamma(); nimp: the cell has impurity scattering
  __device__ __forceinline__ double imp_bound(double Rho, double DA, double e0, double e3, bool nimp) const {
    const double lo = __builtin_amdgcn_rcp(M.scrt0) * 1.000001;
    if (!nimp) return lo;
    const double frr = M.frickel * 4 * PI * Rho * __builtin_amdgcn_rcp(M.eps_si);
    const double em = frr * __builtin_amdgcn_rcp(8.0 * B.melt);
    const double e = em < e0 ? e0 : em > e3 ? e3 : em;
    if (e * M.eV0 >= 0.1200001) return lo;
    const double fr2 = (M.frickel * Rho) * (M.frickel * Rho);
    // eebeta * meld = frr / 2
    const double den = PI * fr2 * (1.0 + 8.0 * e * B.melt * __builtin_amdgcn_rcp(frr));
    const double r = DA * B.meld * __builtin_amdgcn_sqrt(2.0 * B.meld * e) * __builtin_amdgcn_rcp(den) * 1.00001;
    return r <= lo ? lo : r;  // a NaN stays: no comparison with it settles anything
  }

  // DONE: the step ended here and the state is final; BAIL: the slow kernel's.
  __device__ __forceinline__ int run() {
    uint32_t sw = B.symw[isym];
    double ph, im, ss = 0, ssg = 0;
    uint32_t d1;
    bool have_ss = false;
    int iband = -1;
    {
      uint32_t d0;
      draws(0u, d0, d1);
      ph = log_bound(d0);
      im = log_bound(d1);  // of the impurity draw, where there is one
    }
    n_events = 0;
    pend_kind = pend_j = 0;
#pragma clang loop unroll(disable)
    for (;;) {
      if (++n_events > EVENTS) return BAIL;
      // every read of the event
      const EMC_GLB TetRec* R = B.tr + itet;
      const EMC_GLB fd2* RN = (const EMC_GLB fd2*)&R->n[0][0];
      fd2 n[8];
#pragma unroll
      for (int q = 0; q < 8; ++q) n[q] = RN[q];
      const fd2 vt01 = ((const EMC_GLB fd2*)&R->vt[0])[0], vt23 = ((const EMC_GLB fd2*)&R->vt[0])[1];
      const fd2 ge = *(const EMC_GLB fd2*)&R->gam;  // gam, e3
      const fi4 nb = *(const EMC_GLB fi4*)&R->neib[0];
      iband = n_events == 1 ? R->ibt : iband;
      const size_t c = ((size_t)jcell * M.cnx + icell) * M.cnz + kcell;
      const EMC_GLB double *fx = pick(F.ex, F.hx), *fy = pick(F.ey, F.hy), *fz = pick(F.ez, F.hz);
      const EMC_GLB double *fr = pick(F.e_rough, F.h_rough), *fs = pick(F.e_sph, F.h_sph);
      double Ex = fx[c], Ey = fy[c], Ez = fz[c];
      const double Rho = F.rho[c], DA = M.da[c], rough = fr[c], sph = fs[c];
      const uint64_t info = M.minfo[c];
      const double px0 = M.lx[icell], px1 = M.lx[icell + 1], py0 = M.ly[jcell], py1 = M.ly[jcell + 1],
                   pz0 = M.lz[kcell], pz1 = M.lz[kcell + 1];
      asm volatile("" ::: "memory");  // the reads above stay above their uses
      const double sg = pick(M.charge_sign[0], M.charge_sign[1]);
      Ex = sg * Ex; Ey = sg * Ey; Ez = sg * Ez;
      double vx, vy, vz, xk, yk, zk, xf, yf, zf;
      out_wedge(sw, vx, vy, vz, vt01.x, vt01.y, vt23.x);
      in_wedge(sw, xk, yk, zk, kx, ky, kz);
      in_wedge(sw, xf, yf, zf, Ex, Ey, Ez);
      // the nearest face and the next nearest quotient
      double qmin = 1e99, q2 = 1e99, num = 0, den = 1;
      int face = 0;
      bool odd = false;  // a quotient that is no number
      auto cand = [&](double nu, double de, int id, bool on) {
        double q = nu * __builtin_amdgcn_rcp(de);
        q = on ? q : 1e99;
        odd |= !(q == q);
        const bool lt = q < qmin;
        q2 = fmax(qmin, fmin(q2, q));
        qmin = lt ? q : qmin;
        num = lt ? nu : num;
        den = lt ? de : den;
        face = lt ? id : face;
      };
#pragma unroll
      for (int f = 0; f < 4; ++f) {
        const double nf = n[2 * f].x * xf + n[2 * f].y * yf + n[2 * f + 1].x * zf;
        const double nu = n[2 * f + 1].y - (n[2 * f].x * xk + n[2 * f].y * yk + n[2 * f + 1].x * zk);
        cand(nu, nf, f, nf < 0);
      }
      cand(vx > 0 ? px1 - x : -(x - px0), vx, vx > 0 ? 4 + DOWN : 4 + UP, vx != 0);
      cand(vy > 0 ? py1 - y : -(y - py0), vy, vy > 0 ? 4 + RIGHT : 4 + LEFT, vy != 0);
      cand(vz > 0 ? pz1 - z : -(z - pz0), vz, vz > 0 ? 4 + BACK : 4 + FRONT, vz != 0);
      const bool later = qmin > left * 1.000001;
      if (odd || !(qmin > 1e-12) || !(later || (qmin < left * 0.999999 && q2 > qmin * 1.000001))) return BAIL;
      const double Tf = later ? left : num / den;
      // scattering before that?
      const double gam = ge.x;
      if (!(ph > gam * Tf)) return BAIL;
      const bool insurf = M.flag_surface && ((info >> 48) & 255u);
      double gi = 0;
      if (iband == B.bandofE) {
        gi = imp_bound(Rho, DA, vt23.y, ge.y, DA * M.conc0 >= 1e22 && !(insurf && M.flag_simp));
        if (!(im > gi * Tf)) return BAIL;
      }
      if (insurf) {
        if (!have_ss) {
          // the next draw: the second of block 0, or the first of block 1 after the
          // impurity's
          uint32_t a = d1, b;
          if (iband == B.bandofE) draws(1u, a, b);
          ss = log_bound(a);
          have_ss = true;
        }
        ssg = rough + sph;
        if (ssg > 0 ? !(ss > ssg * Tf) : !(ssg <= 0)) return BAIL;
      }
      if (Tf < MY_ZERO) return BAIL;
      // Flight::advance
      left -= Tf;
      ph -= gam * Tf;
      im -= gi * Tf;
      ss -= ssg * Tf;
      kx += Ex * Tf; ky += Ey * Tf; kz += Ez * Tf;
      energy += (vx * Ex + vy * Ey + vz * Ez) * Tf;
      x += vx * Tf; y += vy * Tf; z += vz * Tf;
      if (energy < 0) return BAIL;
      if (later) return DONE;
      if (face < 4) {
        // HitTet without the Brillouin-zone fold
        const int t = face == 0 ? nb.x : face == 1 ? nb.y : face == 2 ? nb.z : nb.w;
        if (t == -5 || t == -6) return BAIL;
        if (t >= 0) itet = t;
        else {
          isym = B.newisym[(-t - 2) * 48 + isym];
          sw = B.symw[isym];
        }
      } else {
        face -= 4;
        const int rule = (int)((info >> (8 * face)) & 255u);
        if (rule == PASS) {
          if (face == UP) { if (icell == 0) return BAIL; x = px0; --icell; }
          else if (face == DOWN) { if (icell + 1 >= M.cnx) return BAIL; x = px1; ++icell; }
          else if (face == FRONT) { if (kcell == 0) return BAIL; z = pz0; --kcell; }
          else if (face == BACK) { if (kcell + 1 >= M.cnz) return BAIL; z = pz1; ++kcell; }
          else {
            // the current of a y crossing is held back until the particle is done
            if (pend_kind) return BAIL;
            if (face == RIGHT) {
              if (jcell + 1 >= M.cny) return BAIL;
              y = py1;
              pend_kind = 1; pend_j = ++jcell;
            } else {
              if (jcell == 0) return BAIL;
              y = py0;
              pend_kind = 2; pend_j = jcell--;
            }
          }
        } else if (rule == REFLECT || (rule == SCATTOX && M.flag_surface)) {
          // Flight::mirror
          const int ax = face >> 1;  // UP, DOWN: x; LEFT, RIGHT: y; FRONT, BACK: z
          if (ax == 0) kx = -kx;
          else if (ax == 1) ky = -ky;
          else kz = -kz;
          const uint32_t w = sw ^ (64u << ax);
          const int s0 = (w & 64u) ? 0 : 2, s1 = (w & 128u) ? 0 : 2, s2 = (w & 256u) ? 0 : 2;
          isym = B.indmat[((s0 * 3 + s1) * 3 + s2) * 27 + (int)(w & 3u) * 9 + (int)((w >> 2) & 3u) * 3 +
                          (int)((w >> 4) & 3u)];
          sw = B.symw[isym];
        } else if (rule == PERIOD) {
          if (face == UP) x = px1;
          else if (face == DOWN) x = px0;
          else if (face == LEFT) y = py1;
          else if (face == RIGHT) y = py0;
          else if (face == FRONT) z = pz1;
          else z = pz0;
        } else
          return BAIL;
      }
      if (!(left > 0)) return DONE;
    }
  }
};

}  // namespace emc
