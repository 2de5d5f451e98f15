// redigm.hip -- the grid-space part of dogcm's Redi/GM isopycnal mixing of the tracers
// (LPhys_RediGM_hspm_vfvm_AddMixingTerm, model/dogcm/src/physics/lphys/
// LPhys_RediGM_hspm_vfvm_mod.f90:218-372) on device grids.
//
// k_redigm_scan finds the two LDD95 tapering depths of each column (the surface and bottom scans
// of TaperingFunc_LDD95, LPhys_RediGMHelper_mod.f90:392-428; one thread a column and direction):
// it evaluates the slopes of the top layers down to the first layer deeper than the eddy
// displacement and of the bottom layers up to the first one higher than it above the bottom, and
// stops there, as the reference's scans exit.  k_redigm_col then walks the layers, one thread a
// column and segment of layers (with few layers a thread scans and walks its whole column in one
// launch), with a one-layer window: vertical differences on the half levels
// (calc_GradTRC :412-424), the JM95 expansion coefficients and the slopes (calc_IsoNeutralSlope_new
// :745-775), the taper (DM95 or GKW91 times LDD95), the Redi and skew fluxes of both tracers
// on the layer and on the half level above it (calc_IsopycDiffFlux :497-553, calc_SkewFlux
// :607-676), and writes per tracer (FLonRedi + FLonGM) cos(lat), (FLatRedi + FLatGM)
// cos(lat) and the vertical flux divergence (FSig above - FSig below) RCDK / H of the layer
// above (append_Redi_GM_RHS :340-366).  Every expression keeps the reference's order of
// operations and no multiply-add is contracted, so the results equal the reference loops in
// FP64 up to the last bit of tanh and sin.
//
// Bound: HBM and, close to it, the vector issue (about 410 instructions a layer, 285 of them FP64).
// Algorithmic bytes per call: the 8 input layer fields (ptemp, salt, h, z, the four gradients)
// and the 6 output layer fields once: (14 km + 1) I J 8 bytes; the scans reread a few layers.
// 512 x 256 x 60: scan 46 us, walk 189 us (4.9 TB/s); an earlier kernel of one thread a column took
// 284 us.  What the difference was: the layer thicknesses' reciprocals were loaded from memory
// behind the next layer's loads, and so waited for them (rfdk is in LDS now); 13 full divisions a
// layer (now 4 reciprocals and corrected quotients); tanh (now one exp); 208 registers.

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <type_traits>

#include "dsht_internal.hpp"

#pragma clang fp contract(off)

namespace dsht {

namespace {

// EOS_JM95_alpha_beta (EOS_JM95_mod.f90:284-330): the McDougall (1987) polynomials of
// alpha/beta and beta in theta [degC], S - 35 [psu] and p [dbar]
constexpr double AB000 = 0.665157e-1, AB100 = 0.170907e-1, AB200 = -0.203814e-3, AB300 = 0.298357e-5,
                 AB400 = -0.255019e-7, AB010 = 0.378110e-2, AB110 = -0.846960e-4, AB011 = -0.164759e-6,
                 AB012 = -0.251520e-11, AB020 = -0.678662e-5, AB001 = 0.380374e-4, AB101 = -0.933746e-6,
                 AB201 = 0.791325e-8, AB202 = 0.512857e-12, AB003 = -0.302285e-13;
constexpr double B000 = 0.785567e-3, B100 = -0.301985e-5, B200 = 0.555579e-7, B300 = -0.415613e-9,
                 B010 = -0.356603e-6, B110 = 0.788212e-8, B011 = 0.408195e-10, B012 = -0.602281e-15,
                 B020 = 0.515032e-8, B001 = -0.121555e-7, B101 = 0.192867e-9, B201 = -0.213127e-11,
                 B002 = 0.176621e-12, B102 = -0.175379e-14, B003 = 0.121551e-17;
constexpr double PI_REF = 3.1415926535897932;  // DOGCM_Admin_Constants_mod PI

struct RediArgs {
  const double *pt, *sa, *h, *z, *topo, *cdk, *rfdk, *glon, *glat, *lat_cs;
  double *flon, *flat, *vdiv;
  long ldg, ldgr, ldo, npts;  // pitches: inputs, gradients, outputs
  int km, I, J, gkw91, seg;  // seg: layers a thread of the walk writes
  double R, rR, rg, kr, kg, smax, sd, two_omega;  // rR: 1/R, or 0 where R is outside recip_ok
};

// Quotients by one divisor d from its reciprocal: two Newton steps on the hardware estimate, and a
// quotient corrected by its exact remainder (Markstein, IBM J. Res. Dev. 34, 1990), which rounds as
// the division does where no intermediate leaves the normal range.  Where the quotient overflows the
// correction is NaN, and v_div_fixup_f64 makes the infinity of it that the division gives.  A divisor
// outside (2^-900, 2^900), 0, an infinity or NaN is divided by as such.
__device__ inline bool recip_ok(double d) {
  const double m = fabs(d);
  return m > 0x1p-900 && m < 0x1p900;
}
__device__ inline double recip(double d) {
  double r = __builtin_amdgcn_rcp(d);
  r = __builtin_fma(__builtin_fma(-d, r, 1.0), r, r);
  return __builtin_fma(__builtin_fma(-d, r, 1.0), r, r);
}
__device__ inline double quot(double n, double d, double r) {
  const double q = n * r;
  return __builtin_amdgcn_div_fixup(__builtin_fma(__builtin_fma(-d, q, n), r, q), d, n);
}
__device__ inline void div2(double n0, double n1, double d, double r, double& q0, double& q1) {
  if (__builtin_expect(recip_ok(d), 1)) {
    q0 = quot(n0, d, r);
    q1 = quot(n1, d, r);
  } else {
    q0 = n0 / d;
    q1 = n1 / d;
  }
}

// tanh(x): 1 - 2 / (exp(2|x|) + 1) with x's sign where |x| >= 1, whose subtrahend is below 0.24,
// so that its rounding stays under that of the difference
__device__ inline double taper_tanh(double x) {
  const double y = fabs(x);
  if (!(y >= 1.0)) return tanh(x);  // and NaN
  const double d = exp(y > 25.0 ? 50.0 : 2.0 * y) + 1.0;
  const double r = recip(d), q = 2.0 * r;
  return copysign(1.0 - __builtin_fma(__builtin_fma(-d, q, 2.0), r, q), x);
}

// EOSDriver_alpha_beta with p = -RefDens*Grav*z [Pa] (calc_IsoNeutralSlope_new :740-743):
// K2degC(theta), Pa2bar(p)*10 (EOSDriver_mod.f90), then the JM95 polynomials
__device__ inline void jm95_alpha_beta(double theta, double s, double z, double rg, double& al, double& be) {
  const double t = theta - 273.15;
  const double p = (1e-05 * (-(rg * z))) * 10.0;
  const double sm = s - 35.0;
  const double adb = ((AB000 + t * (AB100 + t * (AB200 + t * (AB300 + t * AB400)))) +
                      sm * (((AB010 + AB110 * t) + p * (AB011 + AB012 * p)) + sm * AB020)) +
                     p * ((AB001 + t * (AB101 + t * (AB201 + p * AB202))) + (p * p) * AB003);
  be = ((B000 + t * (B100 + t * (B200 + t * B300))) + sm * (((B010 + B110 * t) + p * (B011 + B012 * p)) + sm * B020)) +
       p * ((B001 + t * ((B101 + t * B201) + p * B102)) + p * (B002 + p * B003));
  al = adb * be;
}

// DSig of x on the half levels above (da) and below (db) layer k, from x at k-1, k, k+1
// (the top and bottom half levels copy their neighbours, calc_GradTRC :420-424)
__device__ inline void dsig_pair(int k, int km, const double* rfdk, double xm, double xc, double xp, double& da,
                                 double& db) {
  const double up = k > 0 ? (xm - xc) * rfdk[k] : 0.0;
  const double dn = k + 1 < km ? (xc - xp) * rfdk[k + 1] : 0.0;
  da = k > 0 ? up : dn;
  db = k + 1 < km ? dn : up;
}

// everything of one layer that the fluxes of the layer and of the half level above need
struct Lay {
  double h, tap, slon, slat;
  double gl[2], ga[2];  // horizontal gradients / RPlanet (temperature, salinity)
  double da[2], db[2];  // DSig above and below the layer
};

// the slopes of layer k (calc_IsoNeutralSlope_new :745-775)
__device__ inline void layer_slopes(const RediArgs& a, const double* rfdk, int k, double tm, double tc, double tp, double sm, double sc,
                                    double sp, double z, Lay& L) {
  dsig_pair(k, a.km, rfdk, tm, tc, tp, L.da[0], L.db[0]);
  dsig_pair(k, a.km, rfdk, sm, sc, sp, L.da[1], L.db[1]);
  double al, be;
  jm95_alpha_beta(tc, sc, z, a.rg, al, be);
  const double den = (1e-10 + (al * 0.5) * (L.da[0] + L.db[0])) - (be * 0.5) * (L.da[1] + L.db[1]);
  const double fac = -(L.h / den);
  L.slon = fac * (al * L.gl[0] - be * L.gl[1]);
  L.slat = fac * (al * L.ga[0] - be * L.ga[1]);
}

// the loads of one layer: h, z and the four gradients of layer k, and ptemp/salt of the next
// layer in the walk's direction (k+1 down, k-1 up; unused past the end)
struct Pre {
  double h, z, g0, a0, g1, a1, tn, sn;
};

constexpr int SRING = 2;  // layers whose loads the scans have in flight ahead of the one being computed

constexpr int REDI_LDS_LAYERS = 1024;  // layers whose half-level weights the block keeps in LDS

// a uniform layer base and the point's byte offset (I J < 2^29)
__device__ inline double ld(const double* base, unsigned qb) { return *(const double*)((const char*)base + qb); }
__device__ inline void st(double* base, unsigned qb, double v) { *(double*)((char*)base + qb) = v; }

// dir = +1: the next layer is k+1 (downward walk); -1: k-1 (upward)
__device__ inline void fetch_layer(const RediArgs& a, unsigned qb, int k, int dir, Pre& f) {
  const long g = (long)k * a.ldg, gr = (long)k * a.ldgr, TS = (long)a.km * a.ldgr;
  f.h = ld(a.h + g, qb);
  f.z = ld(a.z + g, qb);
  f.g0 = ld(a.glon + gr, qb);
  f.a0 = ld(a.glat + gr, qb);
  f.g1 = ld(a.glon + TS + gr, qb);
  f.a1 = ld(a.glat + TS + gr, qb);
  const int kn = k + dir;
  const bool in = kn >= 0 && kn < a.km;
  f.tn = in ? ld(a.pt + g + dir * a.ldg, qb) : 0.0;
  f.sn = in ? ld(a.sa + g + dir * a.ldg, qb) : 0.0;
}

// layer k's slopes from its loads and ptemp/salt at k-1, k, k+1
__device__ inline void slopes_of(const RediArgs& a, const double* rfdk, int k, const Pre& f, double tm, double tc,
                                 double tp, double sm, double sc, double sp, Lay& L) {
  L.h = f.h;
  if (a.rR != 0.0) {
    L.gl[0] = quot(f.g0, a.R, a.rR);
    L.ga[0] = quot(f.a0, a.R, a.rR);
    L.gl[1] = quot(f.g1, a.R, a.rR);
    L.ga[1] = quot(f.a1, a.R, a.rR);
  } else {
    L.gl[0] = f.g0 / a.R;
    L.ga[0] = f.a0 / a.R;
    L.gl[1] = f.g1 / a.R;
    L.ga[1] = f.a1 / a.R;
  }
  layer_slopes(a, rfdk, k, tm, tc, tp, sm, sc, sp, f.z, L);
}

// One LDD95 scan of a column (TaperingFunc_LDD95 :392-428), stopping at its first hit: from the
// surface (DIR > 0) or from the bottom up.  found(depth, hit): the depth and layer (0 and none).
template <int DIR, typename F>
__device__ __forceinline__ void redigm_scan(const RediArgs& a, const double* wfd, long q, unsigned qb, double disph,
                                            F found) {
  const int km = a.km;
  const double dzmax = a.smax * disph;
  const int k0 = DIR > 0 ? 0 : km - 1;
  const double topo = DIR > 0 ? 0.0 : a.topo[q];
  double depth = 0.0;
  int hit = DIR > 0 ? -1 : km;
  Pre ring[SRING];
#pragma unroll
  for (int u = 0; u < SRING; u++)
    if (u < km) fetch_layer(a, qb, k0 + DIR * u, DIR, ring[u]);
  double xc = ld(a.pt + (long)k0 * a.ldg, qb), yc = ld(a.sa + (long)k0 * a.ldg, qb);
  double xb = xc, yb = yc;  // the layer behind in the walk (k0 itself at the start)
  double mx = 0.0;
  bool done = false;
  for (int i0 = 0; i0 < km && !done; i0 += SRING) {
#pragma unroll
    for (int u = 0; u < SRING; u++) {
      const int i = i0 + u;
      if (done || i >= km) continue;
      const int k = k0 + DIR * i;
      const Pre c = ring[u];
      if (i + SRING < km) fetch_layer(a, qb, k + DIR * SRING, DIR, ring[u]);
      const bool end = i + 1 == km;
      const double xn = end ? xc : c.tn, yn = end ? yc : c.sn;
      Lay L;
      if (DIR > 0)
        slopes_of(a, wfd, k, c, xb, xc, xn, yb, yc, yn, L);
      else
        slopes_of(a, wfd, k, c, xn, xc, xb, yn, yc, yb, L);
      const double sab = sqrt(L.slon * L.slon + L.slat * L.slat);
      if (sab > mx) mx = sab;
      if (DIR > 0 ? (0.0 - c.z) > dzmax : (c.z - (-topo)) > dzmax) {
        hit = k;
        depth = fmin(mx, a.smax) * disph;
        done = true;
      }
      xb = xc, yb = yc, xc = xn, yc = yn;
    }
  }
  found(depth, hit);
}

// the eddy displacement at a point's latitude (TaperingFunc_LDD95 :392-396)
__device__ __forceinline__ double eddy_displacement(const RediArgs& a, long q) {
  const double asn = a.lat_cs[a.J + q / a.I];
  return fmin(fmax(15e3, 2.0 / (a.two_omega * asn)), 100e3);
}

// Both scans, blockIdx.y = 0 from the surface, 1 from the bottom.  The pair (depth, layer) goes to
// the first layer of each segment of the walk, where the segment's own thread reads it before it
// stores its fluxes there: temperature and salinity planes of flon (surface) or flat (bottom).
__global__ __launch_bounds__(256) void k_redigm_scan(RediArgs a) {
  __shared__ double wfd[REDI_LDS_LAYERS];
  for (int k = threadIdx.x; k < a.km; k += 256) wfd[k] = a.rfdk[k];
  __syncthreads();
  const long q = (long)blockIdx.x * 256 + threadIdx.x;
  if (q >= a.npts) return;
  const unsigned qb = (unsigned)q * 8u;
  const double disph = eddy_displacement(a, q);
  auto keep = [&](double* o) {
    return [=](double depth, int hit) {
      const long oS = (long)a.km * a.ldo;
      for (int k = 0; k < a.km; k += a.seg) {
        st(o + (long)k * a.ldo, qb, depth);
        st(o + oS + (long)k * a.ldo, qb, (double)hit);
      }
    };
  };
  if (blockIdx.y == 0)
    redigm_scan<1>(a, wfd, q, qb, disph, keep(a.flon));
  else
    redigm_scan<-1>(a, wfd, q, qb, disph, keep(a.flat));
}

// Segment blockIdx.y of the walk: layers k0 .. k1-1, with the layer above (its half-level terms)
// and the layer below (the flux into the segment's last layer) computed again.  SCAN: the whole
// column, after its own scans.
template <bool SCAN>
__global__ __launch_bounds__(256, SCAN ? 2 : 3) void k_redigm_col(RediArgs a) {
  // per layer k: m1 = cdk[k]/(cdk[k-1]+cdk[k]), m2 = cdk[k-1]/(cdk[k-1]+cdk[k]) (r_m1, r_m2 of
  // the half level on top of layer k, calc_IsopycDiffFlux :491-494) and z_RCDK = 1/cdk[k]
  // (DOGCM_Admin_Grid_mod.f90:315), each the same IEEE division as in the loop
  __shared__ double wm1[REDI_LDS_LAYERS], wm2[REDI_LDS_LAYERS], wrc[REDI_LDS_LAYERS];
  __shared__ double wfd[REDI_LDS_LAYERS];
  const int km = a.km;
  const int k0 = blockIdx.y * a.seg, k1 = min(k0 + a.seg, km);
  const int ka = max(k0 - 1, 0), kz = min(k1 + 1, km);
  for (int k = ka + threadIdx.x; k < min(kz + 1, km); k += 256) {
    const double c1 = a.cdk[k];
    wrc[k] = 1.0 / c1;
    wfd[k] = a.rfdk[k];
    if (k > 0) {
      const double c0 = a.cdk[k - 1];
      wm1[k] = c1 / (c0 + c1);
      wm2[k] = c0 / (c0 + c1);
    }
  }
  __syncthreads();
  const long q = (long)blockIdx.x * 256 + threadIdx.x;
  if (q >= a.npts) return;
  const unsigned qb = (unsigned)q * 8u;
  const double cs = a.lat_cs[q / a.I];
  const double topo = a.topo[q];
  const long oS = (long)km * a.ldo, o0 = (long)k0 * a.ldo;
  double tmps, tmpb;
  int ks, kb;
  if constexpr (SCAN) {
    const double disph = eddy_displacement(a, q);
    redigm_scan<1>(a, wfd, q, qb, disph, [&](double depth, int hit) { tmps = depth, ks = hit; });
    redigm_scan<-1>(a, wfd, q, qb, disph, [&](double depth, int hit) { tmpb = depth, kb = hit; });
  } else {
    tmps = ld(a.flon + o0, qb), tmpb = ld(a.flat + o0, qb);
    ks = (int)ld(a.flon + oS + o0, qb), kb = (int)ld(a.flat + oS + o0, qb);
  }
  const double kr = a.kr, kg = a.kg;
  Lay P;                         // layer k-1
  double rPh = 0.0;              // 1 / P.h
  double fs_up[2] = {0.0, 0.0};  // FSig on the half level above layer k-1
  double tc = ld(a.pt + (long)ka * a.ldg, qb), sc = ld(a.sa + (long)ka * a.ldg, qb), tm = tc, sm = sc;
  if (ka > 0) tm = ld(a.pt + (long)(ka - 1) * a.ldg, qb), sm = ld(a.sa + (long)(ka - 1) * a.ldg, qb);
  auto body = [&](int k, const Pre& f) {
    const bool last = k + 1 == km;
    const double tp = last ? tc : f.tn, sp = last ? sc : f.sn;
    Lay C;
    slopes_of(a, wfd, k, f, tm, tc, tp, sm, sc, sp, C);
    const double rCh = recip(C.h);
    const double z = f.z;
    // taper (prepare_SlopeTapering: T1 T2)
    const double mag2 = C.slon * C.slon + C.slat * C.slat;
    const double t1 =
        a.gkw91 ? fmin(1.0, (a.smax * a.smax) / mag2) : 0.5 * (1.0 + taper_tanh((a.smax - sqrt(mag2)) / a.sd));
    double r = 1.0;
    if (k <= ks) r = fmin((0.0 - z) / (tmps + 1e-13), 1.0);
    if (k >= kb) r = fmin((z - (-topo)) / (tmpb + 1e-13), 1.0);
    // r = 1 gives 0.5 (1 + sin(pi/2)) = 1 exactly; sin only where the ratio is below 1
    const double t2 = r == 1.0 ? 1.0 : 0.5 * (1.0 + sin(PI_REF * (r - 0.5)));
    C.tap = t1 * t2;
    if (k >= k0 && k < k1) {
      double dz[2];
      div2(0.5 * (C.da[0] + C.db[0]), 0.5 * (C.da[1] + C.db[1]), C.h, rCh, dz[0], dz[1]);
      const long o = (long)k * a.ldo;
#pragma unroll
      for (int x = 0; x < 2; x++) {
        const double flr = kr * (C.gl[x] + (C.tap * C.slon) * dz[x]);
        const double far_ = kr * (C.ga[x] + (C.tap * C.slat) * dz[x]);
        const double flg = -(((kg * C.tap) * C.slon) * dz[x]);  // -Psi(LAT) dz
        const double fag = -((kg * C.tap) * C.slat) * dz[x];    // Psi(LON) dz
        st(a.flon + x * oS + o, qb, (flr + flg) * cs);
        st(a.flat + x * oS + o, qb, (far_ + fag) * cs);
      }
    }
    if (k > ka) {  // the half level between layers k-1 (up) and k (lo)
      const double m1 = wm1[k], m2 = wm2[k];
      const double sl = (m1 * P.tap) * P.slon + (m2 * C.tap) * C.slon;
      const double sa_ = (m1 * P.tap) * P.slat + (m2 * C.tap) * C.slat;
      const double hden = m1 * P.h + m2 * C.h;
      const double rc = wrc[k - 1], ss = sl * sl + sa_ * sa_;
      // Psi(LON) and Psi(LAT) of both layers
      const double pln = m1 * -((kg * P.tap) * P.slat) + m2 * -((kg * C.tap) * C.slat);
      const double pat = m1 * ((kg * P.tap) * P.slon) + m2 * ((kg * C.tap) * C.slon);
      double dv[2], fs[2];
      div2(ss * C.da[0], ss * C.da[1], hden, recip(hden), dv[0], dv[1]);
#pragma unroll
      for (int x = 0; x < 2; x++) {
        const double glon = m1 * P.gl[x] + m2 * C.gl[x];
        const double glat = m1 * P.ga[x] + m2 * C.ga[x];
        const double fr = kr * ((sl * glon + sa_ * glat) + dv[x]);
        const double fg = pat * glon - pln * glat;
        fs[x] = fr + fg;
      }
      if (k > k0) {
        div2((fs_up[0] - fs[0]) * rc, (fs_up[1] - fs[1]) * rc, P.h, rPh, dv[0], dv[1]);
        st(a.vdiv + (long)(k - 1) * a.ldo, qb, dv[0]);
        st(a.vdiv + oS + (long)(k - 1) * a.ldo, qb, dv[1]);
      }
      fs_up[0] = fs[0], fs_up[1] = fs[1];
    }
    P = C;
    rPh = rCh;
    tm = tc, sm = sc, tc = tp, sc = sp;
  };
  Pre nx;
  fetch_layer(a, qb, ka, 1, nx);
  for (int k = ka; k < kz; k++) {
    const Pre c = nx;
    if (k + 1 < kz) fetch_layer(a, qb, k + 1, 1, nx);
    body(k, c);
  }
  if (k1 == km) {  // the bottom layer: FSig below it is zero
    const double rc = wrc[km - 1];
    for (int x = 0; x < 2; x++)
      st(a.vdiv + x * oS + (long)(km - 1) * a.ldo, qb, ((fs_up[x] - 0.0) * rc) / P.h);
  }
}

// rhs[c] = (rhs[c] + hdiv[c]) + vdiv[c] over the 2 km layer grids of both tracers
__global__ __launch_bounds__(256) void k_redigm_rhs(double* __restrict__ rt, double* __restrict__ rs, long ldo,
                                                    const double* __restrict__ hdiv, const double* __restrict__ vdiv,
                                                    long ldw, int km, long npts) {
  const long q = (long)blockIdx.x * 256 + threadIdx.x;
  const int c = blockIdx.y;
  if (q >= npts) return;
  double* r = c < km ? rt + (long)c * ldo : rs + (long)(c - km) * ldo;
  const long w = (long)c * ldw + q;
  r[q] = (r[q] + hdiv[w]) + vdiv[w];
}

}  // namespace

int launch_redigm_col(const dsht_plan* p, const RediParams& c, const double* pt, const double* sa, const double* h,
                      const double* z, long ldg, int km, const double* topo, const double* cdk, const double* rfdk,
                      const double* glon, const double* glat, long ldgr, double* flon, double* flat, double* vdiv,
                      long ldo, bool alone, hipStream_t s) {
  RediArgs a;
  a.pt = pt, a.sa = sa, a.h = h, a.z = z, a.topo = topo, a.cdk = cdk, a.rfdk = rfdk, a.glon = glon, a.glat = glat;
  a.lat_cs = p->d_lat_cs;
  a.flon = flon, a.flat = flat, a.vdiv = vdiv;
  a.ldg = ldg, a.ldgr = ldgr, a.ldo = ldo, a.npts = (long)p->I * p->J;
  a.km = km, a.I = p->I, a.J = p->J, a.gkw91 = c.gkw91;
  a.R = p->R, a.rg = c.ref_dens * c.grav, a.kr = c.kappa_redi, a.kg = c.kappa_gm, a.smax = c.slope_max, a.sd = c.sd;
  a.rR = fabs(p->R) > 0x1p-900 && fabs(p->R) < 0x1p900 ? 1.0 / p->R : 0.0;
  a.two_omega = 2.0 * c.omega;
  const double bytes = (14.0 * km + 1.0) * (double)a.npts * 8.0;
  ProfScope prof("redigm_col", s, bytes, 0.0);
  const unsigned nb = (unsigned)((a.npts + 255) / 256);
  // One launch, a thread a whole column, where segments give little or nothing: 2 and 3 layers (a
  // second launch and the halo layers cost more: 64 x 32 x 2 8.4 and 9.2 us), more on grids that give
  // every SIMD one wave (400 x 200 x 12 43 and 45 us, x 24 69 and 64; 384 x 192 x 14 45 and 45) or
  // one and a half (512 x 256 x 10 41 and 51 us, x 20 73 and 83; 540 x 270 x 24 109 and 106).  A call
  // of its own up to 9 layers on any grid, which waits for the host's launches (64 x 32 x 5 20.8 and
  // 23.4 us a call, though 15.2 and 13.2 on the device; x 10 23.4 and 23.4)
  if (km <= (a.npts < 65536 ? (alone ? 9 : 3) : a.npts < 98304 ? 14 : 20)) {
    a.seg = km;
    hipLaunchKernelGGL(k_redigm_col<true>, dim3(nb), dim3(256), 0, s, a);
    DSHT_HIP(hipGetLastError());
    return 0;
  }
  // Segments: at least 5120 waves (3 a SIMD on 1024 SIMDs run at once) of 3 layers or more (of 4
  // layers 2) but for the last.  Whole column (one segment) against this rule: 512 x 256 x 60 (3
  // segments) 229 and 227 us, 256 x 128 x 60 (10) 133 and 76 us, 128 x 64 x 20 (7) 49 and 25 us
  const long nseg = std::max(1l, std::min((5120l * 64 + a.npts - 1) / a.npts, (km + 2l) / 3));
  a.seg = (int)((km + nseg - 1) / nseg);
  hipLaunchKernelGGL(k_redigm_scan, dim3(nb, 2), dim3(256), 0, s, a);
  hipLaunchKernelGGL(k_redigm_col<false>, dim3(nb, (unsigned)((km + a.seg - 1) / a.seg)), dim3(256), 0, s, a);
  DSHT_HIP(hipGetLastError());
  return 0;
}

int launch_redigm_rhs(const dsht_plan* p, double* rt, double* rs, long ldo, const double* hdiv, const double* vdiv,
                      long ldw, int km, hipStream_t s) {
  const long npts = (long)p->I * p->J;
  const double bytes = 4.0 * 2.0 * km * (double)npts * 8.0;
  ProfScope prof("redigm_rhs", s, bytes, 0.0);
  hipLaunchKernelGGL(k_redigm_rhs, dim3((unsigned)((npts + 255) / 256), 2 * km), dim3(256), 0, s, rt, rs, ldo, hdiv,
                     vdiv, ldw, km, npts);
  DSHT_HIP(hipGetLastError());
  return 0;
}

}  // namespace dsht
