// lfam3.hip -- a device-resident LF-AM3 dynamics step of dogcm for many independent runs of
// one truncation and layer count (DOGCM_TInt_LFAM3_advance_Dyn,
// model/dogcm/src/tint/DOGCM_TInt_LFAM3_mod.f90:281-880).
//
// Configuration: hydrostatic Boussinesq dynamics on the hspm_vfvm grid with a rigid lid
// (one barotropic iteration, :147-170, 685-774), a flat bottom (xyz_H = D, xyz_Z = D z_CK,
// DOGCM_Admin_Grid_mod.f90:376-388), the linear equation of state (EOS_Linear_mod.f90) and
// no physics forcing.  Per layer a step stands for the reference's 42 forward and 28 inverse
// transform units (VorDivDiag x3, MOMBarocRHS x2, HTRCRHS x2 over two tracers, ImplUV,
// ImplTRC) and per run 9 forward and 9 inverse 2-D units of the barotropic mode; every
// transform runs over all layers of all active runs in one library call.  It makes fewer: the
// constant geopotential's gradient is computed once a step, the vorticity that only the divergence
// is wanted with is not, and in the FP64 form the implicit solves work on spectra.  The grid-space
// work between the transforms is fused into the kernels below; the column work (omega,
// hydrostatic pressure, barotropic velocity, QUICK flux, the implicit vertical solves) is
// done in them too, a thread walking a column.
//
// Layout (FP64 device memory): run r, layer k of a layered field is grid column r*K + k;
// tracers are run-major with temperature then salinity: column (2r + t)*K + k; 2-D fields
// one column per run; half-level fields (K+1) levels per run (per run and tracer for the
// vertical fluxes).  Spectra of internal transforms use the fast "LC" layout.
#include <algorithm>
#include <cmath>
#include <cstring>
#include <vector>

#include "dsht_internal.hpp"

namespace dsht {
namespace {

constexpr int LF_THREADS = 256;

inline dim3 lf_grid(long n) {
  long b = (n + LF_THREADS - 1) / LF_THREADS;
  if (b > 1l << 20) b = 1l << 20;
  if (b < 1) b = 1;
  return dim3((unsigned)b);
}

#define LF_LOOP(n) for (long g = (long)blockIdx.x * blockDim.x + threadIdx.x; g < (n); g += (long)gridDim.x * blockDim.x)
// 2-D walk over (column c, point p) of ncols columns of npts points, g = c npts + p: the column
// is uniform over a block (grid y), so its layer and run come from scalar arithmetic, and
// the latitude row of p is one 32-bit division
#define LF_CP(ncols, npts)                                                                                \
  for (long c = blockIdx.y; c < (ncols); c += gridDim.y)                                                 \
    for (long p = (long)blockIdx.x * blockDim.x + threadIdx.x; p < (npts); p += (long)gridDim.x * blockDim.x)
#define LF_ROW(p, I) ((int)((unsigned)(p) / (unsigned)(I)))

inline dim3 lf_grid2(long ncols, long npts) {
  long bx = (npts + LF_THREADS - 1) / LF_THREADS;
  if (bx > 4096) bx = 4096;
  long by = ncols < 65535 ? ncols : 65535;
  return dim3((unsigned)(bx < 1 ? 1 : bx), (unsigned)(by < 1 ? 1 : by));
}

// x*cos(phi_j), y*cos(phi_j) (the calc_UVCosLat2VorDiv inputs, HBEDiagnose_hspm_vfvm_mod.f90:278-281)
__global__ void k_lf_uvcos(const double* __restrict__ u, const double* __restrict__ v, const double* __restrict__ cs,
                           long npts, int I, long ncols, double* __restrict__ ucos, double* __restrict__ vcos) {
  LF_CP(ncols, npts) {
    const long g = c * npts + p;
    const double w = cs[LF_ROW(p, I)];
    ucos[g] = u[g] * w;
    vcos[g] = v[g] * w;
  }
}

// GeoPot = Grav * D * z_CK(k) (DOGCM_TInt_LFAM3_mod.f90:460)
__global__ void k_lf_geo(double* __restrict__ geo, long npts, int K, const double* __restrict__ zck, double depth,
                         double grav, long ncols) {
  LF_CP(ncols, npts) {
    const int k = (int)(c % K);
    geo[c * npts + p] = grav * (depth * zck[k]);
  }
}

__global__ void k_lf_fill(double* __restrict__ x, double v, long n) {
  LF_LOOP(n) x[g] = v;
}

// Column walks: one thread per grid point of a run (grid y) goes through the layers, G of them
// per round with their loads issued together.  The layers' running sums (pressure from the
// top, omega from the bottom) stay in registers, so a field that is only a step between two
// others (omega, the vertical fluxes) is never written.  The next round's loads go out before
// this round is worked on and stored, so that a round waits neither for its own loads nor for
// the stores before it.  Bound by HBM on large grids: every layer field in and out is touched
// once.

__device__ __forceinline__ double lf_ld(const double* x) { return __builtin_nontemporal_load(x); }

inline dim3 lf_gridc(long npts, int nr, int threads) { return dim3((unsigned)((npts + threads - 1) / threads), (unsigned)nr); }
// blocks of 64 where there are fewer waves than SIMDs, to spread the columns over the chip
inline int lf_threads(long npts, int nr) { return npts * nr >= 65536 ? 256 : 64; }

constexpr int LF_NONE[16] = {};
// layers k = first, first + dir, ... (K of them): body(k, values) with the values of NF fields
// (above: layers nearer the end of the walk, clamped to it), G layers a round
template <int NF, int G, bool NT = true, typename Body>
__device__ __forceinline__ void lf_walk(const double* const (&f)[NF], long npts, int K, int first, int dir, Body body,
                                        const int* above = LF_NONE) {
  double cur[G][NF], nxt[G][NF];
  auto load = [&](double (&x)[G][NF], int n0) {
#pragma unroll
    for (int q = 0; q < G; q++)
#pragma unroll
      for (int i = 0; i < NF; i++) {
        const int n = n0 + q + above[i] < K ? n0 + q + above[i] : K - 1;
        const double* at = f[i] + (long)(first + dir * n) * npts;
        x[q][i] = NT ? lf_ld(at) : *at;
      }
  };
  load(cur, 0);
  int n0 = 0;
  for (; n0 + G <= K; n0 += G) {
    load(nxt, n0 + G);
#pragma unroll
    for (int q = 0; q < G; q++) body(first + dir * (n0 + q), cur[q]);
#pragma unroll
    for (int q = 0; q < G; q++)
#pragma unroll
      for (int i = 0; i < NF; i++) cur[q][i] = nxt[q][i];
  }
#pragma unroll
  for (int q = 0; q < G; q++)
    if (n0 + q < K) body(first + dir * (n0 + q), cur[q]);
}

// EOS_Linear_Eval(theta, S, p = -RefDens GeoPot) and the hydrostatic pressure of its density
// (HBEDiagnose_HydPres, HBEDiagnose_hspm_vfvm_mod.f90:315-321) for every layer of every run
struct EosArgs {
  double ref_dens, ptemp_dep, press_dep, salt_dep, ref_temp, ref_salt, depth, grav;
};
__global__ __launch_bounds__(256) void k_lf_eos_hyd(const double* __restrict__ ts, long npts, int K,
                                                    const double* __restrict__ zck, const double* __restrict__ cdk,
                                                    EosArgs e, double* __restrict__ dens, double* __restrict__ hyd) {
#pragma clang fp contract(off)
  const long p = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= npts) return;
  const long r = blockIdx.y;
  const double* tp = ts + 2 * r * K * npts + p;
  const double* sp = tp + (long)K * npts;
  const long o = r * K * npts + p;
  const double gh = e.grav * e.depth;
  double sum = 0.0;
  auto layer = [&](int k, double t, double s) {
    const double geo = e.grav * (e.depth * zck[k]);
    const double pr = -e.ref_dens * geo;
    const double d = e.ref_dens * (e.ptemp_dep * (t - e.ref_temp) + e.press_dep * pr + e.salt_dep * (s - e.ref_salt));
    const double next = sum + (gh * d) * cdk[k];
    dens[o + k * npts] = d;
    hyd[o + k * npts] = 0.5 * (sum + next);
    sum = next;
  };
  const double* f[2] = {tp, sp};
  lf_walk<2, 8>(f, npts, K, 0, 1, [&](int k, const double (&x)[2]) { layer(k, x[0], x[1]); });
}

// The grid-space part of HBEBaroc_MOMRHS_VorDivForm (HBEBaroc_hspm_vfvm_mod.f90:366-420):
// omega from the divergence (HBEDiagnose_OMG, HBEDiagnose_hspm_vfvm_mod.f90:123-131), the
// vertical advection of momentum at the half levels, the absolute-vorticity fluxes A and B
// (times cos phi) and the Bernoulli function C, from the bottom layer up.  Writes -A (so that
// one calc_UVCosLat2VorDiv call with (U cos, V cos) = (B, -A) gives -H(A, B) and H(B, -A)), B
// and C.  The Coriolis terms (:474-481, 565-570): PRED f (cn x + cb xb) of the advected winds
// and (xa, xb) of the time level before; else f times the winds (xa, xb) of the present level.
struct MomArgs {
  double ref_dens, radius, depth, cn, cb;
  long npts;
  int I, K;
};
template <bool PRED>
__global__ __launch_bounds__(256) void k_lf_mom(
    MomArgs a, const double* __restrict__ u, const double* __restrict__ v, const double* __restrict__ xa,
    const double* __restrict__ xb, const double* __restrict__ div, const double* __restrict__ vor,
    const double* __restrict__ hyd, const double* __restrict__ dens, const double* __restrict__ glon,
    const double* __restrict__ glat, const double* __restrict__ sp, const double* __restrict__ two_omega,
    const double* __restrict__ mu, const double* __restrict__ cosj, const double* __restrict__ cdk,
    const double* __restrict__ rfdk, double* __restrict__ am, double* __restrict__ bg, double* __restrict__ cg) {
  const long p = (long)blockIdx.x * blockDim.x + threadIdx.x, np = a.npts;
  if (p >= np) return;
  const long r = blockIdx.y, o = r * a.K * np + p;
  const int j = LF_ROW(p, a.I);
  const double f = two_omega[r] * mu[j], cs = cosj[j], rr = a.ref_dens * a.radius;
  const double sfc = sp[r * np + p];
  double om = 0.0, vau_b = 0.0, vav_b = 0.0;  // omega and vertical advection at the layer's lower half level
  double uk = lf_ld(u + o + (a.K - 1) * np), vk = lf_ld(v + o + (a.K - 1) * np);
  // the winds one layer ahead (above); the top layer's are not used
  const double* fld[10] = {u + o, v + o, xa + o, xb + o, div + o, vor + o, hyd + o, dens + o, glon + o, glat + o};
  const int above[10] = {1, 1, 0, 0, 0, 0, 0, 0, 0, 0};
  lf_walk<10, 4>(fld, np, a.K, a.K - 1, -1, [&](int k, const double (&x)[10]) {
    const long g = o + k * np;
    om = om - x[4] * (a.depth * cdk[k]);
    double vau_a = 0.0, vav_a = 0.0;
    if (k > 0) {
      vau_a = om * (x[0] - uk) * rfdk[k];
      vav_a = om * (x[1] - vk) * rfdk[k];
    }
    const double coru = PRED ? f * (a.cn * uk + a.cb * x[2]) : f * x[2];
    const double corv = PRED ? f * (a.cn * vk + a.cb * x[3]) : f * x[3];
    double A = x[5] * uk + coru + 0.5 * (vav_b + vav_a) / a.depth;
    A = cs * (A + x[7] * x[9] / rr);
    double B = x[5] * vk + corv - 0.5 * (vau_b + vau_a) / a.depth;
    B = cs * (B + x[7] * x[8] / rr);
    am[g] = -A;
    bg[g] = B;
    cg[g] = (0.5 * (uk * uk + vk * vk) + (x[6] + sfc) / a.ref_dens) / (a.radius * a.radius);
    vau_b = vau_a;
    vav_b = vav_a;
    uk = x[0];
    vk = x[1];
  }, above);
}

// w_out[l, c] += w_in[l, c]
__global__ void k_lf_spec_add(double* __restrict__ wout, long slo, const double* __restrict__ win, long sli, int L,
                              int ncols) {
  LF_CP(L, ncols) wout[c * slo + p] += win[c * sli + p];
}

// The thickness-weighted layer means of U and V (HBEDiagnose_UVBarot, HBEDiagnose_hspm_vfvm_mod.f90:
// 246-251) of the time levels N (grid z 0) and B (z 1), one walk each
struct BarotArgs {
  const double *u[2], *v[2];
  double *ub[2], *vb[2];
};
__global__ __launch_bounds__(256) void k_lf_uvbarot(BarotArgs a, double depth, const double* __restrict__ cdk, long npts,
                                                    int K) {
#pragma clang fp contract(off)
  const long p = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= npts) return;
  const long o = (long)blockIdx.y * K * npts + p;
  const double* __restrict__ u = a.u[blockIdx.z] + o;
  const double* __restrict__ v = a.v[blockIdx.z] + o;
  double dep = 0.0, su = 0.0, sv = 0.0;
  const double* fld[2] = {u, v};
  lf_walk<2, 8>(fld, npts, K, 0, 1, [&](int k, const double (&x)[2]) {
    const double f = depth * cdk[k];
    dep = dep + f;
    su = su + x[0] * f;
    sv = sv + x[1] * f;
  });
  a.ub[blockIdx.z][blockIdx.y * npts + p] = su / dep;
  a.vb[blockIdx.z][blockIdx.y * npts + p] = sv / dep;
}

// predictor momentum (DOGCM_TInt_LFAM3_mod.f90:495-528): optional implicit Coriolis with
// CoriImplFac = 0.5 (2 dt) f, U = 5/6 dt U_RHS + (2 U_N + U_B)/3, and U's barotropic part
// replaced by that of level N.  U's layer mean follows from the means of U_RHS (a first walk)
// and of U_N and U_B (known), so U itself is written once.
__global__ __launch_bounds__(256) void k_lf_pred_uv(
    const double* __restrict__ urhs, const double* __restrict__ vrhs, const double* __restrict__ un,
    const double* __restrict__ ub, const double* __restrict__ vn, const double* __restrict__ vb,
    const double* __restrict__ ubn, const double* __restrict__ vbn, const double* __restrict__ ubb,
    const double* __restrict__ vbb, const double* __restrict__ two_omega, const double* __restrict__ mu, double depth,
    const double* __restrict__ cdk, long npts, int I, int K, double half2dt, double c56dt, int implicit,
    double* __restrict__ uo, double* __restrict__ vo) {
  const long p = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= npts) return;
  const long r = blockIdx.y, o = r * K * npts + p, q2 = r * npts + p;
  const double cif = implicit ? half2dt * (two_omega[r] * mu[LF_ROW(p, I)]) : 0.0, den = 1.0 + cif * cif;
  double dep = 0.0, su = 0.0, sv = 0.0;
  const double* rhs[2] = {urhs + o, vrhs + o};
  lf_walk<2, 8, false>(rhs, npts, K, 0, 1, [&](int k, const double (&x)[2]) {
    const double f = depth * cdk[k];
    dep = dep + f;
    su = su + x[0] * f;
    sv = sv + x[1] * f;
  });
  su /= dep;
  sv /= dep;
  const double ubr = ubn[q2], vbr = vbn[q2];
  // barotropic part of level N minus that of U, V
  const double du = ubr - (c56dt * ((su + cif * sv) / den) + (2.0 * ubr + ubb[q2]) / 3.0);
  const double dv = vbr - (c56dt * ((sv - cif * su) / den) + (2.0 * vbr + vbb[q2]) / 3.0);
  const double* fld[6] = {urhs + o, vrhs + o, un + o, ub + o, vn + o, vb + o};
  lf_walk<6, 4>(fld, npts, K, 0, 1, [&](int k, const double (&x)[6]) {
    const long g = o + k * npts;
    uo[g] = (c56dt * ((x[0] + cif * x[1]) / den) + (2.0 * x[2] + x[3]) / 3.0) + du;
    vo[g] = (c56dt * ((x[1] - cif * x[0]) / den) + (2.0 * x[4] + x[5]) / 3.0) + dv;
  });
}

// The grid-space part of HBEBaroc_HTRCRHS (HBEBaroc_hspm_vfvm_mod.f90:162-172) for both tracers
// of every run, from the bottom layer up: omega from the divergence (HBEDiagnose_OMG), the QUICK
// flux at the half levels (calc_ADVFlxZ_QUICK, :233-317: 0 at the surface and the bottom,
// centred at half levels 1 and K-1, else with the curvature terms D of the two layers), the
// horizontal flux (U, V) H cos(phi) T and the vertical flux divergence
// -(F(k) - F(k+1)) / z_CDK(k).  m1, m2, dfac: the interpolation weights per half level.
__device__ __forceinline__ double lf_curvature(double ta, double tb, double tc, double ra, double rb) {
#pragma clang fp contract(off)
  const double x = (ta - tb) * ra;
  const double y = (tb - tc) * rb;
  return (x - y) * (ra + rb);
}
__global__ __launch_bounds__(256) void k_lf_htrc(const double* __restrict__ ts, const double* __restrict__ u,
                                                 const double* __restrict__ v, const double* __restrict__ div,
                                                 double depth, double h, const double* __restrict__ cosj,
                                                 const double* __restrict__ cdk, const double* __restrict__ rcdk,
                                                 const double* __restrict__ rfdk, const double* __restrict__ m1,
                                                 const double* __restrict__ m2, const double* __restrict__ dfac,
                                                 long npts, int I, int K, double* __restrict__ fu,
                                                 double* __restrict__ fv, double* __restrict__ vf) {
#pragma clang fp contract(off)
  const long p = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= npts) return;
  const long r = blockIdx.y, o = r * K * npts + p, ot = 2 * r * K * npts + p, sec = (long)K * npts;
  const double hc = h * cosj[LF_ROW(p, I)];
  auto T = [&](int tr, int k) { return lf_ld(ts + ot + tr * sec + (long)(k > 0 ? k : 0) * npts); };
  double om = 0.0;
  double t0[2], t1[2], fb[2] = {0.0, 0.0}, db[2] = {0.0, 0.0};  // T[k], T[k-1], F(k+1), D[k]
#pragma unroll
  for (int tr = 0; tr < 2; tr++) {
    t0[tr] = T(tr, K - 1);
    t1[tr] = T(tr, K - 2);
  }
  // the tracers two layers ahead (above)
  const double* fld[5] = {ts + ot, ts + ot + sec, u + o, v + o, div + o};
  const int above[5] = {2, 2, 0, 0, 0};
  lf_walk<5, 4>(fld, npts, K, K - 1, -1, [&](int k, const double (&x)[5]) {
    const double dz = depth * cdk[k];
    om = om - x[4] * dz;
#pragma unroll
    for (int tr = 0; tr < 2; tr++) {
      const double t2 = x[tr];  // T[k-2]
      double da = 0.0, fl = 0.0;
      if (k > 0) {
        const double mid = m1[k] * t1[tr] + m2[k] * t0[tr];
        if (k >= 2) da = lf_curvature(t2, t1[tr], t0[tr], rfdk[k - 1], rfdk[k]);
        if (k >= 2 && k <= K - 2)
          fl = om * (mid - dfac[k] * (da + db[tr])) + (fabs(om) * dfac[k]) * (da - db[tr]);
        else
          fl = om * mid;
      }
      const double tmp = hc * t0[tr];
      const long g = ot + tr * sec + k * npts;
      fu[g] = x[2] * tmp;
      fv[g] = x[3] * tmp;
      vf[g] = -(fl - fb[tr]) * rcdk[k];
      fb[tr] = fl;
      db[tr] = da;
      t0[tr] = t1[tr];
      t1[tr] = t2;
    }
  }, above);
}

// w = AdvFilter (-w_alpha + w_vert) (HBEBaroc_hspm_vfvm_mod.f90:163-171), in place over w_alpha
__global__ void k_lf_htrc_spec(double* __restrict__ wa, const double* __restrict__ wv, const double* __restrict__ filt,
                               int L, int ncols) {
  LF_CP(L, ncols) {
    const long g = c * ncols + p;
    wa[g] = filt[c] * (-wa[g] + wv[g]);
  }
}

// predictor tracers (:535-541): ((H (2 T_N + T_B))/3 + 5/6 dt HTRC_RHS) / H
__global__ void k_lf_pred_trc(const double* __restrict__ tn, const double* __restrict__ tb,
                              const double* __restrict__ ht, double h, double c56dt, long n, double* __restrict__ to) {
  LF_LOOP(n) to[g] = (h * (2.0 * tn[g] + tb[g]) / 3.0 + c56dt * ht[g]) / h;
}

// After the implicit solves (:615-646) and up to the barotropic forcing (HBEBarot_MOMRHS grid
// part, HBEBarot_hspm_vfvm_mod.f90:197-201), one walk: U_RHS = (U_A - U_N)/dt and its layer
// mean, the forcing UBarocForce - CoriVBarot, VBarocForce + CoriUBarot with CoriXBarot = f x_N
// (:626-630), implicit Coriolis with CoriImplFac = alpha_ dt f, U_A = U_N + dt U_RHS and the
// layer mean of that; -A and B of A = cos (f U - VBarocForce), B = cos (f V + UBarocForce); and
// SfcPres - SfcPres_N, which is 0 in the one iteration of a rigid lid.
__global__ __launch_bounds__(256) void k_lf_impl(
    double* __restrict__ ua, double* __restrict__ va, const double* __restrict__ un, const double* __restrict__ vn,
    const double* __restrict__ ubn, const double* __restrict__ vbn, const double* __restrict__ pn,
    const double* __restrict__ two_omega, const double* __restrict__ mu, const double* __restrict__ cosj, double depth,
    const double* __restrict__ cdk, long npts, int I, int K, double adt, double dt, double* __restrict__ ubt,
    double* __restrict__ vbt, double* __restrict__ am, double* __restrict__ bg, double* __restrict__ spm) {
  const long p = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= npts) return;
  const long r = blockIdx.y, o = r * K * npts + p, q2 = r * npts + p;
  const int j = LF_ROW(p, I);
  const double f = two_omega[r] * mu[j], cif = adt * f, den = 1.0 + cif * cif;
  double dep = 0.0, fu = 0.0, fv = 0.0, su = 0.0, sv = 0.0;
  const double* fld[4] = {ua + o, va + o, un + o, vn + o};
  lf_walk<4, 4>(fld, npts, K, 0, 1, [&](int k, const double (&x)[4]) {
    const long g = o + k * npts;
    const double w = depth * cdk[k];
    const double ur = (x[0] - x[2]) / dt, vr = (x[1] - x[3]) / dt;
    dep += w;
    fu += ur * w;
    fv += vr * w;
    const double u1 = x[2] + dt * ((ur + cif * vr) / den), v1 = x[3] + dt * ((vr - cif * ur) / den);
    su += u1 * w;
    sv += v1 * w;
    ua[g] = u1;
    va[g] = v1;
  });
  ubt[q2] = su / dep;
  vbt[q2] = sv / dep;
  const double coru = f * ubn[q2], corv = f * vbn[q2];
  const double ubf = fu / dep - corv, vbf = fv / dep + coru;
  am[q2] = -(cosj[j] * (coru - vbf));
  bg[q2] = cosj[j] * (corv + ubf);
  spm[q2] = pn[q2] - pn[q2];
}

// The barotropic velocity step of the sub-cycle (:712-721), U + dts (U_RHS + c V_RHS)/(1 + c^2),
// and the result times cos phi
__global__ void k_lf_barot_step(const double* __restrict__ ur_in, const double* __restrict__ vr_in,
                                const double* __restrict__ u0, const double* __restrict__ v0,
                                const double* __restrict__ two_omega, const double* __restrict__ mu,
                                const double* __restrict__ cosj, long npts, int I, double adt, double dt, long nruns,
                                double* __restrict__ uo, double* __restrict__ vo, double* __restrict__ uc,
                                double* __restrict__ vc) {
  LF_CP(nruns, npts) {
    const long g = c * npts + p;
    const int j = LF_ROW(p, I);
    const double cif = adt * (two_omega[c] * mu[j]), ur = ur_in[g], vr = vr_in[g];
    const double u = u0[g] + dt * (ur + cif * vr) / (1.0 + cif * cif);
    const double v = v0[g] + dt * (vr - cif * ur) / (1.0 + cif * cif);
    uo[g] = u;
    vo[g] = v;
    uc[g] = u * cosj[j];
    vc[g] = v * cosj[j];
  }
}

// HBEBarot_Update_LinFreeSfc spectral part with vareps1 = 0 (:283-297): w_Tmp = -w_Div,
// w_DSfcPres = RefDens w_Coef w_Tmp / (PresTAvgCoefA dts), w_DDiv = n(n+1)/R^2 w_Coef w_Tmp
__global__ void k_lf_barot_proj(const double* __restrict__ wdiv, long sld, const double* __restrict__ coef,
                                const double* __restrict__ e, double ref_dens, double den, int L, int ncols,
                                double* __restrict__ wdsp, double* __restrict__ wddiv) {
  LF_CP(L, ncols) {
    const long g = c * ncols + p;
    const double wt = -wdiv[c * sld + p];
    wdsp[g] = ref_dens * coef[c] * wt / den;
    wddiv[g] = e[c] * coef[c] * wt;
  }
}

// The barotropic correction (UBarot + dUBarot, SfcPres + dSfcPres), the full velocity and the
// time-centred winds of the tracer update (:783-795), U_A = U_A - UBarot + UBarot_A,
// U = (5 U_A + 8 U_N - U_B)/12, and the time levels of momentum and pressure (B <- N, N <- A),
// which nothing later in the step reads
struct FinalArgs {
  double *ua, *un, *ub, *uo;              // U: levels A, N, B; the time-centred wind
  double *va, *vn, *vb, *vo;
  const double *ubt, *vbt;                // layer means to take out
  const double *ubar, *du, *vbar, *dv;    // barotropic velocity and its correction
  const double* dsp;
  double *pa, *pn, *pb;                   // surface pressure: levels A, N, B
};
__global__ void k_lf_final_uv(FinalArgs a, long npts, int K, long ncols) {
  LF_CP(ncols, npts) {
    const long g = c * npts + p;
    const long q = (c / K) * npts + p;
    const double u0 = a.un[g], v0 = a.vn[g];
    const double u = a.ua[g] - a.ubt[q] + (a.ubar[q] + a.du[q]);
    const double v = a.va[g] - a.vbt[q] + (a.vbar[q] + a.dv[q]);
    a.uo[g] = (5.0 * u + 8.0 * u0 - a.ub[g]) / 12.0;
    a.vo[g] = (5.0 * v + 8.0 * v0 - a.vb[g]) / 12.0;
    a.ua[g] = u;
    a.va[g] = v;
    a.ub[g] = u0;
    a.vb[g] = v0;
    a.un[g] = u;
    a.vn[g] = v;
    if (c % K == 0) {
      const double s0 = a.pn[q], s = s0 + a.dsp[q];
      a.pa[q] = s;
      a.pb[q] = s0;
      a.pn[q] = s;
    }
  }
}

// T_A = H_0 T_A / H_A (DOGCM_Phys_hspm_vfvm_mod.f90:641) and the tracers' time levels
__global__ void k_lf_trc_final(double* __restrict__ ta, double* __restrict__ tn, double* __restrict__ tb, double h,
                               long n) {
  LF_LOOP(n) {
    const double t = h * ta[g] / h;
    tb[g] = tn[g];
    ta[g] = t;
    tn[g] = t;
  }
}

// The implicit vertical diffusion of a tracer (calc_VDiffTRCEq, DOGCM_Phys_hspm_vfvm_mod.f90:
// 752-861) or of momentum (MOM; calc_VDiffMOMEq, :865-975) with the pool's constant
// viscosities, thickness factor and bottom friction: every grid point has the same matrix, so
// its DGTSV elimination (factors, interchanges, finished rows) is done once on the host
// (lf_vfactor) and a thread only carries its column's right-hand side through it, in DGTSV's
// order of operations: qa = q0 + x.  The right-hand side waits for the backward sweep in
// registers (K <= KM), or in qa (KM = 0).  Bound by HBM: three layer fields, against the five
// and a workspace of the general k_col_vdiff: at T170L60 two fields take 67 us (5.6 TB/s), there
// 163; loading each group only when it is worked on took 111.  Grid y: sections of K layers,
// grid z: field pairs.
constexpr int VL = 8;  // layers whose loads are in flight together
struct VSolve {
  const double *q0[2], *rhs[2];
  double* qa[2];
};
template <int KM, bool MOM>
__global__ __launch_bounds__(256) void k_lf_vsolve(VSolve a, const double* __restrict__ fact,
                                                   const double* __restrict__ dd, const double* __restrict__ du,
                                                   const double* __restrict__ du2, const int* __restrict__ swapped,
                                                   double dt, double e3, long npts, int K) {
#pragma clang fp contract(off)
  const long p = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= npts) return;
  const long o = (long)blockIdx.y * K * npts + p;
  const double* __restrict__ q0 = a.q0[blockIdx.z] + o;
  const double* __restrict__ rhs = a.rhs[blockIdx.z] + o;
  double* __restrict__ qa = a.qa[blockIdx.z] + o;
  double xa = 0.0, xb = 0.0;  // x[k+1], x[k+2]
  auto right = [&](double x) {
    const double bt = dt * x;
    return MOM ? bt : bt / e3;
  };
  auto back = [&](int k, double b, double q) {
    const double t = b - du[k] * xa;
    const double x = (t - du2[k] * xb) / dd[k];
    __builtin_nontemporal_store(q + x, qa + (long)k * npts);
    xb = xa;
    xa = x;
  };
  // rows k-1 and k after elimination step k-1
  auto step = [&](int k, double& up, double& lo) {
    if (swapped[k - 1]) {
      const double t = up;
      up = lo;
      lo = t - fact[k - 1] * lo;
    } else {
      lo = lo - fact[k - 1] * up;
    }
  };
  if constexpr (KM > 0) {
    // the next group's loads go out before this group is worked on
    double b[KM], x[2][VL];
    auto load = [&](const double* __restrict__ f, int k0, double (&to)[VL]) {
#pragma unroll
      for (int u = 0; u < VL; u++) to[u] = lf_ld(f + (long)(k0 + u < K ? k0 + u : K - 1) * npts);
    };
    load(rhs, 0, x[0]);
#pragma unroll
    for (int k0 = 0; k0 < KM; k0 += VL) {
      if (k0 >= K) break;
      if (k0 + VL < KM && k0 + VL < K) load(rhs, k0 + VL, x[(k0 / VL + 1) & 1]);
#pragma unroll
      for (int u = 0; u < VL; u++) {
        const int k = k0 + u;
        if (k >= K) break;
        b[k] = right(x[(k0 / VL) & 1][u]);
        if (k > 0) step(k, b[k > 0 ? k - 1 : 0], b[k]);
      }
    }
    const int last = (K - 1) / VL * VL;
#pragma unroll
    for (int k0 = KM - VL; k0 >= 0; k0 -= VL) {
      if (k0 > last) continue;
      if (k0 == last) load(q0, k0, x[(k0 / VL) & 1]);
      if (k0 > 0) load(q0, k0 - VL, x[(k0 / VL + 1) & 1]);
#pragma unroll
      for (int u = VL - 1; u >= 0; u--)
        if (k0 + u < K) back(k0 + u, b[k0 + u], x[(k0 / VL) & 1][u]);
    }
  } else {
    double up = right(lf_ld(rhs));
    for (int k = 1; k < K; k++) {
      double lo = right(lf_ld(rhs + (long)k * npts));
      step(k, up, lo);
      qa[(long)(k - 1) * npts] = up;
      up = lo;
    }
    for (int k = K - 1; k >= 0; k--) back(k, k == K - 1 ? up : qa[(long)k * npts], lf_ld(q0 + (long)k * npts));
  }
}

// The same solve on spectra: the matrix is the same at every point, so it commutes with the
// horizontal transform, and w = diag (q0 + x) from the spectra q0 of the field and w of its
// tendency takes the place of an inverse of the tendency, the solve on the grid (which has 4.5
// times the values of a T170 spectrum at 512 x 256) and a forward transform.  The columns of one
// coefficient are contiguous, K to a system: SB systems a block go through LDS (an odd row of
// doubles each, so that a wave's rows start in different banks), loaded and stored by the whole
// block, solved by a thread each.  The factors are padded to KP layers, a multiple of VL, with rows
// that leave zeros, so that a group's reads of LDS and factors all come before its first store.
// Elimination as k_lf_vsolve.  Bound by latency: a wave's solve takes 11 us of T170L60's 30, and
// loads and stores go out in one burst each; up to 64 layers (REG) a thread's loads, q0's too, all
// go out first (rows of more in rounds: 41 us there).  32 or 16 systems a block: 38 and 45 us.
constexpr int WS_SB = 64;  // most systems a block of k_lf_wsolve holds
template <bool MOM, bool REG>
__global__ __launch_bounds__(256) void k_lf_wsolve(const double* __restrict__ q0, double* __restrict__ w,
                                                   const double* __restrict__ diag, const double* __restrict__ fac,
                                                   const int* __restrict__ swapped, double dt, double e3,
                                                   unsigned nsys, unsigned per, int K, int KP, int SB) {
#pragma clang fp contract(off)
  extern __shared__ double sh[];
  const int P = KP + 1;
  const double *__restrict__ dd = fac + KP, *__restrict__ du = dd + KP, *__restrict__ du2 = du + KP;
  const unsigned s0 = blockIdx.x * SB;
  const int ns = (int)(nsys - s0 < (unsigned)SB ? nsys - s0 : (unsigned)SB);
  const long g0 = (long)s0 * K;
  const int l16 = threadIdx.x % 16, row0 = threadIdx.x / 16;
  auto right = [&](double x) {
    const double bt = dt * x;
    return MOM ? bt : bt / e3;
  };
  double qv[REG ? WS_SB / 16 : 1][4];
  if constexpr (REG) {
    double wv[WS_SB / 16][4];
    auto load = [&](const double* __restrict__ f, double (&to)[WS_SB / 16][4]) {
#pragma unroll
      for (int r = 0; r < WS_SB / 16; r++)
#pragma unroll
        for (int u = 0; u < 4; u++) {
          const int q = row0 + 16 * r, k = l16 + 16 * u;
          if (16 * u < K) to[r][u] = f[g0 + (q < ns ? q : 0) * K + (k < K ? k : 0)];
        }
    };
    load(w, wv);
    load(q0, qv);
#pragma unroll
    for (int r = 0; r < WS_SB / 16; r++)
#pragma unroll
      for (int u = 0; u < 4; u++) {
        const int q = row0 + 16 * r, k = l16 + 16 * u;
        if (q < ns && k < KP) sh[q * P + k] = k < K ? right(wv[r][u]) : 0.0;
      }
  } else {
    for (int q = row0; q < ns; q += 16) {
#pragma unroll 4
      for (int k = l16; k < KP; k += 16) sh[q * P + k] = k < K ? right(w[g0 + (long)q * K + k]) : 0.0;
    }
  }
  __syncthreads();
  if ((int)threadIdx.x < ns) {
    double* x = sh + threadIdx.x * P;
    double up = 0.0;  // row k-1; the step into row 0 (fac 0, not swapped) takes row 0 as it is
    for (int k0 = 0; k0 < KP; k0 += VL) {
      double v[VL + 1], f[VL];
      bool sw[VL];
#pragma unroll
      for (int u = 0; u < VL; u++) {
        v[u] = x[k0 + u];
        f[u] = u + k0 > 0 ? fac[k0 + u - 1] : 0.0;
        sw[u] = u + k0 > 0 ? swapped[k0 + u - 1] != 0 : false;
      }
#pragma unroll
      for (int u = 0; u < VL; u++) {
        const double a = sw[u] ? up : v[u], b = sw[u] ? v[u] : up;
        v[u] = b;
        up = k0 + u < K ? a - f[u] * b : 0.0;
      }
#pragma unroll
      for (int u = 0; u < VL; u++)
        if (k0 + u > 0) x[k0 + u - 1] = v[u];
    }
    if (K == KP) x[K - 1] = up;
    double xa = 0.0, xb = 0.0;  // x[k+1], x[k+2]
    for (int k0 = KP - VL; k0 >= 0; k0 -= VL) {
      double v[VL], d[VL], e[VL], e2[VL];
#pragma unroll
      for (int u = 0; u < VL; u++) {
        v[u] = x[k0 + u];
        d[u] = dd[k0 + u], e[u] = du[k0 + u], e2[u] = du2[k0 + u];
      }
#pragma unroll
      for (int u = VL - 1; u >= 0; u--) {
        const double t = v[u] - e[u] * xa;
        v[u] = (t - e2[u] * xb) / d[u];
        xb = xa;
        xa = v[u];
      }
#pragma unroll
      for (int u = 0; u < VL; u++) x[k0 + u] = v[u];
    }
  }
  __syncthreads();
#pragma unroll
  for (int r = 0; r < WS_SB / 16; r++) {
    const int q = row0 + 16 * r;
    if (q >= ns) break;
    const double dg = diag[(s0 + q) / per];
    if constexpr (REG) {
#pragma unroll
      for (int u = 0; u < 4; u++) {
        const int k = l16 + 16 * u;
        if (k < K) w[g0 + q * K + k] = (qv[r][u] + sh[q * P + k]) * dg;
      }
    } else {
#pragma unroll 4
      for (int k = l16; k < K; k += 16) {
        const long g = g0 + (long)q * K + k;
        w[g] = (q0[g] + sh[q * P + k]) * dg;
      }
    }
  }
}

}  // namespace
}  // namespace dsht

using namespace dsht;

struct dsht_lfam3 {
  dsht_plan* p = nullptr;
  dsht_lfam3_config cfg;
  int K = 0, R = 0, L = 0, I = 0, J = 0;
  long np = 0;
  std::vector<double> cdk, fdk, rcdk, rfdk, zck;
  std::vector<double*> allocs;
  // constants
  double *d_cdk = nullptr, *d_rcdk = nullptr, *d_rfdk = nullptr, *d_zck = nullptr;
  double *d_mu = nullptr, *d_cs = nullptr, *d_two_omega = nullptr;
  double *d_m1 = nullptr, *d_m2 = nullptr, *d_dfac = nullptr;  // QUICK weights per half level
  double *d_dmom = nullptr, *d_dtrc = nullptr, *d_advf = nullptr, *d_nn1 = nullptr, *d_nn1p = nullptr, *d_hcoef = nullptr,
         *d_e = nullptr;
  // state: levels B (0), N (1), A (2)
  double *U[3] = {}, *V[3] = {}, *TS[3] = {}, *SP[3] = {};
  // work
  double *VD = nullptr, *Dens = nullptr, *Hyd = nullptr;
  double *Geo = nullptr, *GLon = nullptr, *GLat = nullptr, *Am = nullptr, *Bg = nullptr, *Cg = nullptr;
  double *URHS = nullptr, *VRHS = nullptr, *Upr = nullptr, *Vpr = nullptr;
  // FU, FV: the tracers' horizontal fluxes, dead once transformed; the tracers' tendency grids (HT)
  // and the winds times cos(lat) (ucos, vcos) of the forms that need those share their memory
  double *TSpr = nullptr, *FU = nullptr, *FV = nullptr, *VF = nullptr;
  double *HT = nullptr, *ucos = nullptr, *vcos = nullptr;
  double* b2[16] = {};  // 2-D barotropic work, one grid per run each
  double *wVD = nullptr, *wGeo = nullptr, *wC = nullptr, *w1 = nullptr, *w2 = nullptr;
  double *wB = nullptr, *wC2 = nullptr, *wDSP = nullptr, *wDDiv = nullptr, *wZero = nullptr;
  // the elimination of the constant vertical systems (momentum, tracers): fact, d, du, du2 and
  // the interchanges, lf_kp(K) each
  double* d_vf[2] = {};
  int* d_vs[2] = {};
};

namespace {

enum B2 { UBN, VBN, UBB, VBB, UBT, VBT, UBR, VBR, UBAR, VBAR, DU, DV, DSP, SPM, AM2, BG2, B2_COUNT };

int lf_alloc(dsht_lfam3* s, double** out, size_t n) {
  void* ptr = nullptr;
  if (hipMalloc(&ptr, sizeof(double) * (n ? n : 1)) != hipSuccess) {
    (void)hipGetLastError();
    return fail(DSHT_ENOMEM, "LF-AM3 pool: device allocation of %zu doubles failed", n);
  }
  s->allocs.push_back((double*)ptr);
  *out = (double*)ptr;
  return 0;
}

int lf_upload(dsht_lfam3* s, double** out, const std::vector<double>& v) {
  if (int rc = lf_alloc(s, out, v.size())) return rc;
  DSHT_HIP(hipMemcpy(*out, v.data(), sizeof(double) * v.size(), hipMemcpyHostToDevice));
  return 0;
}

void lf_free(dsht_lfam3* s) {
  (void)hipDeviceSynchronize();
  for (double* d : s->allocs) (void)hipFree(d);
  s->allocs.clear();
}

#define LF_LAUNCH(kernel, n, s, ...)                                                     \
  do {                                                                                   \
    hipLaunchKernelGGL(kernel, lf_grid(n), dim3(LF_THREADS), 0, s, __VA_ARGS__);         \
    DSHT_HIP(hipGetLastError());                                                         \
  } while (0)
// kernels walking (column, point) pairs with LF_CP
#define LF_LAUNCH2(kernel, ncols, npts, s, ...)                                          \
  do {                                                                                   \
    hipLaunchKernelGGL(kernel, lf_grid2(ncols, npts), dim3(LF_THREADS), 0, s, __VA_ARGS__); \
    DSHT_HIP(hipGetLastError());                                                         \
  } while (0)

// column walks over the points of nr runs and nz field sets
#define LF_LAUNCHC(kernel, npts, nr, nz, s, ...)                                              \
  do {                                                                                        \
    const int th_ = lf_threads(npts, (nr) * (nz));                                            \
    dim3 grid_ = lf_gridc(npts, nr, th_);                                                     \
    grid_.z = nz;                                                                             \
    hipLaunchKernelGGL(kernel, grid_, dim3(th_), 0, s, __VA_ARGS__);                          \
    DSHT_HIP(hipGetLastError());                                                              \
  } while (0)

// layers of a padded factor array
int lf_kp(int K) { return (K + VL - 1) / VL * VL; }

// DGTSV's elimination (LAPACK 3.x SRC/dgtsv.f, partial pivoting by row interchange) of the
// constant vertical system of momentum or of the tracers (rows as k_col_vdiff builds them):
// fac = fact, d, du, du2 (lf_kp(K) each, rows of the identity behind K), swapped = 1 where a step interchanged its rows
void lf_vfactor(const dsht_lfam3* s, bool mom, std::vector<double>& fac, std::vector<int>& swapped) {
#pragma clang fp contract(off)
  const dsht_lfam3_config& c = s->cfg;
  const int K = s->K;
  const double kv = mom ? c.vvisc : c.vdiff, e3 = c.depth, alpha = c.lambda;
  const bool sfc = (mom ? c.mom_sfc_bc : c.trc_sfc_bc) == 'D', btm = (mom ? c.mom_btm_bc : c.trc_btm_bc) == 'D';
  std::vector<double> r(K + 1), al(K, 0.0), ad(K), au(K, 0.0);
  r[0] = kv / (s->fdk[0] * e3);
  r[K] = kv / (s->fdk[K] * e3);
  for (int h = 1; h < K; h++) {
    const double sum = s->cdk[h - 1] + s->cdk[h];
    const double m1 = s->cdk[h] / sum, m2 = s->cdk[h - 1] / sum;
    r[h] = (m1 * kv + m2 * kv) / (s->fdk[h] * (m1 * e3 + m2 * e3));
  }
  for (int k = 0; k < K; k++) {
    const double ac = alpha * (c.dt / (e3 * s->cdk[k]));
    if (k > 0) al[k] = -(ac * r[k]);
    if (k < K - 1) au[k] = -(ac * r[k + 1]);
    if (k == 0)
      ad[k] = sfc ? 1.0 + ac * (r[1] + 2.0 * r[0]) : 1.0 + ac * r[1];
    else if (k == K - 1)
      ad[k] = !btm ? 1.0 + ac * r[k] : mom ? 1.0 + ac * (c.btm_frict + r[k]) : 1.0 + ac * (2.0 * r[K] + r[k]);
    else
      ad[k] = 1.0 + ac * (r[k] + r[k + 1]);
  }
  const int KP = lf_kp(K);
  fac.assign(4 * (size_t)KP, 0.0);
  swapped.assign(KP, 0);
  double *fact = fac.data(), *d = fact + KP, *du = d + KP, *du2 = du + KP;
  for (int k = 0; k < KP; k++) d[k] = k < K ? ad[k] : 1.0, du[k] = k < K ? au[k] : 0.0;
  for (int j = 0; j < K - 1; j++) {
    const double dl = al[j + 1];
    if (std::fabs(d[j]) >= std::fabs(dl)) {
      fact[j] = dl / d[j];
      d[j + 1] = d[j + 1] - fact[j] * du[j];
    } else {
      swapped[j] = 1;
      fact[j] = d[j] / dl;
      d[j] = dl;
      const double temp = d[j + 1];
      d[j + 1] = du[j] - fact[j] * temp;
      if (j < K - 2) {
        du2[j] = du[j + 1];
        du[j + 1] = -fact[j] * du2[j];
      }
      du[j] = temp;
    }
  }
}

// one or two fields (z) of ny sections through the constant solve
int lf_vsolve(dsht_lfam3* s, bool mom, const VSolve& a, int ny, int nz, hipStream_t st) {
  const int K = s->K, KP = lf_kp(K), w = mom ? 0 : 1, th = lf_threads(s->np, ny * nz);
  auto k = mom ? (K <= 32 ? k_lf_vsolve<32, true> : K <= 64 ? k_lf_vsolve<64, true> : k_lf_vsolve<0, true>)
               : (K <= 32 ? k_lf_vsolve<32, false> : K <= 64 ? k_lf_vsolve<64, false> : k_lf_vsolve<0, false>);
  dim3 grid = lf_gridc(s->np, ny, th);
  grid.z = nz;
  const double* f = s->d_vf[w];
  hipLaunchKernelGGL(k, grid, dim3(th), 0, st, a, f, f + KP, f + 2 * KP, f + 3 * KP, s->d_vs[w], s->cfg.dt, s->cfg.depth,
                     s->np, K);
  DSHT_HIP(hipGetLastError());
  return 0;
}

// systems a block of k_lf_wsolve holds: 64, fewer where K is large (64 KB of LDS) or where that
// leaves fewer than 1024 blocks
int lf_wsolve_sb(long nsys, int K) {
  const long fit = 8192 / (lf_kp(K) + 1), spread = nsys / 1024;
  return (int)std::min({(long)WS_SB, fit, std::max(8l, spread)});
}

// w = diag (q0 + x) for the spectra of per sections of K layers, where the solve fits
// k_lf_wsolve and the form's transforms return a spectrum to FP64 rounding
bool lf_wsolve_ok(const dsht_lfam3* s) { return fwd_fused_ok(s->p) && lf_wsolve_sb(1 << 20, s->K) >= 8; }
int lf_wsolve(dsht_lfam3* s, bool mom, const double* q0, double* w, const double* diag, int per, hipStream_t st) {
  const int K = s->K, f = mom ? 0 : 1;
  const long nsys = (long)s->L * per;
  const int sb = lf_wsolve_sb(nsys, K);
  auto k = lf_kp(K) <= 64 ? (mom ? k_lf_wsolve<true, true> : k_lf_wsolve<false, true>)
                          : (mom ? k_lf_wsolve<true, false> : k_lf_wsolve<false, false>);
  hipLaunchKernelGGL(k, dim3((unsigned)((nsys + sb - 1) / sb)), dim3(256),
                     sizeof(double) * sb * (lf_kp(K) + 1), st, q0, w, diag, s->d_vf[f], s->d_vs[f],
                     s->cfg.dt, s->cfg.depth, (unsigned)nsys, (unsigned)per, K, lf_kp(K), sb);
  DSHT_HIP(hipGetLastError());
  return 0;
}

// calc_UVCosLat2VorDiv of (U cos phi, V cos phi), the vorticity in w's columns [0, nc) and the
// divergence in [nc, 2 nc): cos phi is applied as the FFT reads the winds, or, where that form
// has no such kernel, by a pass over them
int lf_uv2vordiv(dsht_lfam3* s, const double* u, const double* v, double* w, int nc, const double* diag,
                 hipStream_t st) {
  dsht_plan* p = s->p;
  if (uv_scaled_ok(p))
    return uv2vordiv_scaled(p, u, v, s->d_cs, s->np, w, w + nc, 2l * nc, 1, nc, diag, st);
  LF_LAUNCH2(k_lf_uvcos, nc, s->np, st, u, v, s->d_cs, s->np, s->I, (long)nc, s->ucos, s->vcos);
  return dsht_uv2vordiv_d(p, s->ucos, s->vcos, s->np, w, w + nc, 2l * nc, 1, nc, diag, st);
}

// w += diag w_xy(x) over nc columns of pitch sl (tmp: spectra for forms that do not add)
int lf_fwd_add(dsht_lfam3* s, const double* x, double* w, long sl, double* tmp, int nc, const double* diag,
               hipStream_t st) {
  if (fwd_fused_ok(s->p)) return fwd_add(s->p, x, s->np, w, sl, 1, nc, diag, st);
  if (int rc = dsht_fwd_d(s->p, DSHT_VAL, x, s->np, tmp, nc, 1, nc, diag, st)) return rc;
  LF_LAUNCH2(k_lf_spec_add, s->L, nc, st, w, sl, tmp, (long)nc, s->L, nc);
  return 0;
}

// HBEDiagnose_VorDiv (HBEDiagnose_hspm_vfvm_mod.f90:259-286) over every layer of the active
// runs: vorticity into VD[0, nc), divergence into VD[nc, 2 nc), their spectra in w
int lf_vordiv(dsht_lfam3* s, const double* u, const double* v, double* w, int nc, hipStream_t st) {
  if (int rc = lf_uv2vordiv(s, u, v, w, nc, nullptr, st)) return rc;
  return dsht_inv_d(s->p, DSHT_VAL, w, 2l * nc, 1, s->VD, s->np, 2 * nc, nullptr, st);
}

// its divergence alone, all that the tracers' right-hand side reads
int lf_div(dsht_lfam3* s, const double* u, const double* v, int nc, hipStream_t st) {
  if (!uv_scaled_ok(s->p)) return lf_vordiv(s, u, v, s->wVD, nc, st);
  if (int rc = div_scaled(s->p, u, v, s->d_cs, s->np, s->wVD, nc, 1, nc, st)) return rc;
  return dsht_inv_d(s->p, DSHT_VAL, s->wVD, nc, 1, s->VD + (long)nc * s->np, s->np, nc, nullptr, st);
}

// HBEBaroc_MOMRHS_VorDivForm (HBEBaroc_hspm_vfvm_mod.f90:321-443), the spectra in wVD, with the
// vorticity and divergence of (u, v) in VD.  pred: the Coriolis terms f (cn (u, v) + cb (xa, xb)),
// else f (xa, xb).  The geopotential's gradient is that of the whole step: the predictor, which
// comes first, computes it
int lf_mom_rhs(dsht_lfam3* s, const double* u, const double* v, const double* xa, const double* xb, bool pred, double cn,
               double cb, const double* sp, int nr, hipStream_t st) {
  dsht_plan* p = s->p;
  const int nc = nr * s->K;
  if (pred) {  // w_GeoPot = w_xy(GeoPot); xy_GradLat_w, xy_GradLon_w of it
    if (int rc = dsht_fwd_d(p, DSHT_VAL, s->Geo, s->np, s->wGeo, nc, 1, nc, nullptr, st)) return rc;
    if (int rc = dsht_inv_vgrad_d(p, s->wGeo, nc, 1, nullptr, s->GLon, s->GLat, s->np, nc, nullptr, st)) return rc;
  }
  const MomArgs a{s->cfg.ref_dens, p->R, s->cfg.depth, cn, cb, s->np, s->I, s->K};
  auto k = pred ? k_lf_mom<true> : k_lf_mom<false>;
  LF_LAUNCHC(k, s->np, nr, 1, st, a, u, v, xa, xb, s->VD + (long)nc * s->np, s->VD, s->Hyd, s->Dens, s->GLon, s->GLat,
             sp, s->d_two_omega, s->d_mu, s->d_cs, s->d_cdk, s->d_rfdk, s->Am, s->Bg, s->Cg);
  // (w_Vor_RHS, w_Div_RHS) = (-H(A, B), H(B, -A)) = calc_UVCosLat2VorDiv(B, -A); then
  // w_Div_RHS - w_Lapla_w(w_xy(C)) = + n(n+1) w_xy(C)
  if (int rc = dsht_uv2vordiv_d(p, s->Bg, s->Am, s->np, s->wVD, s->wVD + nc, 2l * nc, 1, nc, nullptr, st)) return rc;
  return lf_fwd_add(s, s->Cg, s->wVD + nc, 2l * nc, s->wC, nc, s->d_nn1, st);
}

// HBEBaroc_HTRCRHS (HBEBaroc_hspm_vfvm_mod.f90:119-202) for both tracers of the active runs, the
// spectra in w1, with the divergence of (u, v) in VD and the thickness factor h
int lf_htrc(dsht_lfam3* s, const double* ts, const double* u, const double* v, double h, int nr, hipStream_t st) {
  dsht_plan* p = s->p;
  const long np = s->np;
  const int nc = nr * s->K, nt = 2 * nc;
  LF_LAUNCHC(k_lf_htrc, np, nr, 1, st, ts, u, v, s->VD + (long)nc * np, s->cfg.depth, h, s->d_cs, s->d_cdk, s->d_rcdk,
             s->d_rfdk, s->d_m1, s->d_m2, s->d_dfac, np, s->I, s->K, s->FU, s->FV, s->VF);
  // w = AdvFilter (-w_AlphaOptr_xy(fluxes) + w_xy(divergence)) (:163-171)
  if (fwd_fused_ok(p)) {
    if (int rc = val_sub_alpha(p, s->FU, s->FV, s->VF, np, s->w1, nt, 1, nt, s->d_advf, st)) return rc;
  } else {
    if (int rc = dsht_alpha_fwd_d(p, s->FU, s->FV, np, s->w1, nt, 1, nt, nullptr, st)) return rc;
    if (int rc = dsht_fwd_d(p, DSHT_VAL, s->VF, np, s->w2, nt, 1, nt, nullptr, st)) return rc;
    LF_LAUNCH2(k_lf_htrc_spec, s->L, nt, st, s->w1, s->w2, s->d_advf, s->L, nt);
  }
  return 0;
}

// the grids of lf_mom_rhs and lf_htrc
int lf_mom_grid(dsht_lfam3* s, int nc, hipStream_t st) {
  return dsht_vordiv2uv_d(s->p, s->wVD, s->wVD + nc, 2l * nc, 1, s->URHS, s->VRHS, s->np, nc, st);
}
int lf_htrc_grid(dsht_lfam3* s, int nt, hipStream_t st) {
  return dsht_inv_d(s->p, DSHT_VAL, s->w1, nt, 1, s->HT, s->np, nt, nullptr, st);
}

}  // namespace

extern "C" {

int dsht_lfam3_default_config(dsht_lfam3_config* c) {
  if (!c) return fail(DSHT_EARG, "dsht_lfam3_default_config: NULL");
  std::memset(c, 0, sizeof(*c));
  c->km = 20;
  c->max_runs = 1;
  c->sub_cycles = 1;
  c->numdiff_ord = 4;
  c->dt = 3600.0;
  c->depth = 5000.0;
  c->grav = 9.79764;
  c->ref_dens = 1027.0;
  c->alpha = 0.51;
  c->lambda = 0.5;
  c->hvisc = 3e5;
  c->hdiff = 0.0;
  c->numdiff = 1e12;
  c->vvisc = 1e-3;
  c->vdiff = 3e-5;
  c->btm_frict = 0.0;
  c->mom_sfc_bc = 'N';
  c->mom_btm_bc = 'D';
  c->trc_sfc_bc = 'N';
  c->trc_btm_bc = 'N';
  c->ref_temp = 283.0;
  c->ref_salt = 35.0;
  c->beta_t = 1.67e-4;
  c->beta_s = 0.78e-3;
  c->cp0 = 3986.0;
  c->cs0 = 1490.0;
  return 0;
}

int dsht_lfam3_create(dsht_plan* p, const dsht_lfam3_config* cfg, dsht_lfam3** out) {
  if (!out) return fail(DSHT_EARG, "dsht_lfam3_create: NULL output");
  *out = nullptr;
  if (!p || p->N < 0) return fail(DSHT_ESTATE, "plan is NULL or destroyed");
  if (!cfg) return fail(DSHT_EARG, "dsht_lfam3_create: NULL config");
  const dsht_lfam3_config& c = *cfg;
  if (c.km < 2 || c.max_runs < 1) return fail(DSHT_EARG, "LF-AM3 pool needs km >= 2 and max_runs >= 1");
  if (!(c.dt > 0) || !(c.depth > 0) || !(c.lambda > 0) || c.sub_cycles < 1)
    return fail(DSHT_EARG, "LF-AM3 pool needs dt, depth, lambda > 0 and sub_cycles >= 1");
  auto bc_ok = [](int b) { return b == 'D' || b == 'N'; };
  if (!bc_ok(c.mom_sfc_bc) || !bc_ok(c.mom_btm_bc) || !bc_ok(c.trc_sfc_bc) || !bc_ok(c.trc_btm_bc))
    return fail(DSHT_EARG, "boundary types must be 'D' or 'N'");
  if (c.km % 2) return fail(DSHT_EARG, "km = %d must be even (the Chebyshev-Lobatto vertical grid)", c.km);
  dsht_lfam3* s = new dsht_lfam3();
  s->p = p;
  s->cfg = c;
  s->K = c.km;
  s->R = c.max_runs;
  s->L = p->L;
  s->I = p->I;
  s->J = p->J;
  s->np = (long)p->I * p->J;
  const int K = s->K, R = s->R, L = s->L, J = s->J;
  const long np = s->np, NC = (long)R * K;
  // vertical grid: faces g_Sig (at_module_omp.f90:598-601 on [-1, 0]), centres, thicknesses
  // and centre spacings (DOGCM_GaussSpmVFvmGrid_mod.f90:392-410)
  std::vector<double> fk(K + 1), ck(K + 2);
  if (int rc = dsht_sig_grid(K, K, -1.0, 0.0, fk.data(), nullptr)) {
    delete s;
    return rc;
  }
  s->cdk.resize(K);
  s->zck.resize(K);
  s->rcdk.resize(K);
  s->fdk.resize(K + 1);
  s->rfdk.resize(K + 1);
  for (int k = 0; k < K; k++) {
    s->cdk[k] = fk[k] - fk[k + 1];
    ck[k + 1] = 0.5 * (fk[k] + fk[k + 1]);
  }
  ck[0] = fk[0] + 0.5 * s->cdk[0];
  ck[K + 1] = fk[K] - 0.5 * s->cdk[K - 1];
  for (int k = 0; k <= K; k++) {
    s->fdk[k] = ck[k] - ck[k + 1];
    s->rfdk[k] = 1.0 / s->fdk[k];
  }
  for (int k = 0; k < K; k++) {
    s->zck[k] = ck[k + 1];
    s->rcdk[k] = 1.0 / s->cdk[k];
  }
  std::vector<double> m1(K + 1, 0.0), m2(K + 1, 0.0), dfac(K + 1, 0.0);  // HBEBaroc_hspm_vfvm_mod.f90:264-266
  for (int h = 1; h < K; h++) {
    const double sum = s->cdk[h - 1] + s->cdk[h];
    m1[h] = s->cdk[h] / sum;
    m2[h] = s->cdk[h - 1] / sum;
    dfac[h] = (0.125 * s->cdk[h]) * s->cdk[h - 1];
  }
  std::vector<double> cs(J), nn1(L), nn1p(L), e(L), hcoef(L);
  for (int j = 0; j < J; j++) cs[j] = std::sqrt((1.0 - p->mu[j]) * (1.0 + p->mu[j]));
  for (int n = 0; n <= p->N; n++)
    for (int m = -n; m <= n; m++) {
      const int l = n * (n + 1) + m;
      nn1[l] = (double)n * (n + 1.0);
      nn1p[l] = nn1[l] / (c.ref_dens * (p->R * p->R));  // of the barotropic pressure term
      e[l] = (double)n * (n + 1.0) / (p->R * p->R);
      hcoef[l] = l == 0 ? 0.0 : 1.0 / (e[l] + 0.0);  // w_Coef, HBEBarot_hspm_vfvm_mod.f90:281-290
    }
  int rc = 0;
  auto A = [&](double** d, size_t n) {
    if (!rc) rc = lf_alloc(s, d, n);
  };
  auto U = [&](double** d, const std::vector<double>& v) {
    if (!rc) rc = lf_upload(s, d, v);
  };
  U(&s->d_cdk, s->cdk);
  U(&s->d_rcdk, s->rcdk);
  U(&s->d_rfdk, s->rfdk);
  U(&s->d_zck, s->zck);
  U(&s->d_m1, m1);
  U(&s->d_m2, m2);
  U(&s->d_dfac, dfac);
  U(&s->d_mu, p->mu);
  U(&s->d_cs, cs);
  U(&s->d_nn1, nn1);
  U(&s->d_nn1p, nn1p);
  U(&s->d_e, e);
  U(&s->d_hcoef, hcoef);
  U(&s->d_two_omega, std::vector<double>(R, 2.0 * 7.292115e-5));
  A(&s->d_dmom, L);
  A(&s->d_dtrc, L);
  A(&s->d_advf, L);
  for (int lv = 0; lv < 3; lv++) {
    A(&s->U[lv], NC * np);
    A(&s->V[lv], NC * np);
    A(&s->TS[lv], 2 * NC * np);
    A(&s->SP[lv], R * np);
  }
  A(&s->VD, 2 * NC * np);
  A(&s->Dens, NC * np);
  A(&s->Hyd, NC * np);
  A(&s->Geo, NC * np);
  A(&s->GLon, NC * np);
  A(&s->GLat, NC * np);
  A(&s->Am, NC * np);
  A(&s->Bg, NC * np);
  A(&s->Cg, NC * np);
  A(&s->URHS, NC * np);
  A(&s->VRHS, NC * np);
  A(&s->Upr, NC * np);
  A(&s->Vpr, NC * np);
  A(&s->TSpr, 2 * NC * np);
  A(&s->FU, 2 * NC * np);
  A(&s->FV, 2 * NC * np);
  A(&s->VF, 2 * NC * np);
  s->HT = s->ucos = s->FU;
  s->vcos = s->FV;
  for (auto& b : s->b2) A(&b, R * np);
  A(&s->wVD, (size_t)L * 2 * NC);
  A(&s->wGeo, (size_t)L * NC);
  A(&s->wC, (size_t)L * NC);
  A(&s->w1, (size_t)L * 2 * NC);
  A(&s->w2, (size_t)L * 2 * NC);
  A(&s->wB, (size_t)L * 2 * R);
  A(&s->wC2, (size_t)L * R);
  A(&s->wDSP, (size_t)L * R);
  A(&s->wDDiv, (size_t)L * R);
  A(&s->wZero, (size_t)L * R);
  for (int w = 0; w < 2; w++) {
    std::vector<double> vf;
    std::vector<int> vs;
    lf_vfactor(s, w == 0, vf, vs);
    U(&s->d_vf[w], vf);
    double* d = nullptr;
    A(&d, (vs.size() + 1) / 2);
    s->d_vs[w] = (int*)d;
    if (!rc && hipMemcpy(d, vs.data(), sizeof(int) * vs.size(), hipMemcpyHostToDevice) != hipSuccess)
      rc = fail(DSHT_EDEVICE, "LF-AM3 pool: upload failed");
  }
  if (rc) {
    lf_free(s);
    delete s;
    return rc;
  }
  hipStream_t st = nullptr;
  auto fill = [&](double* d, double v, long n) -> int {
    hipLaunchKernelGGL(k_lf_fill, lf_grid(n), dim3(LF_THREADS), 0, st, d, v, n);
    DSHT_HIP(hipGetLastError());
    return 0;
  };
  // the state starts at zero
  if (!rc) rc = fill(s->wZero, 0.0, (long)L * R);
  for (int lv = 0; lv < 3 && !rc; lv++) {
    rc = fill(s->U[lv], 0.0, NC * np);
    if (!rc) rc = fill(s->V[lv], 0.0, NC * np);
    if (!rc) rc = fill(s->TS[lv], 0.0, 2 * NC * np);
    if (!rc) rc = fill(s->SP[lv], 0.0, R * np);
  }
  if (!rc) {
    hipLaunchKernelGGL(k_lf_geo, lf_grid2(NC, np), dim3(LF_THREADS), 0, st, s->Geo, np, K, s->d_zck, c.depth, c.grav,
                       (long)NC);
    if (hipGetLastError() != hipSuccess) rc = fail(DSHT_EDEVICE, "LF-AM3 pool: geopotential fill failed");
  }
  // lateral viscosity / diffusion factors 1/(1 - dt w_HViscCoefH), 1/(1 - dt w_HDiffCoefH)
  // (LPhys_DIFF_spm_mod.f90:148-154) and the advection filter (HBEBaroc_hspm_vfvm_mod.f90:83-95)
  const double pm[5] = {c.dt, c.hvisc, c.numdiff, (double)c.numdiff_ord, 1.0};
  const double pt[5] = {c.dt, c.hdiff, c.numdiff, (double)c.numdiff_ord, 0.0};
  if (!rc) rc = dsht_coef_d(p, DSHT_COEF_BEDIFF, pm, 5, s->d_dmom, st);
  if (!rc) rc = dsht_coef_d(p, DSHT_COEF_BEDIFF, pt, 5, s->d_dtrc, st);
  if (!rc) rc = dsht_coef_d(p, DSHT_COEF_ADVFILTER, nullptr, 0, s->d_advf, st);
  if (!rc && hipDeviceSynchronize() != hipSuccess) rc = fail(DSHT_EDEVICE, "LF-AM3 pool: set-up failed");
  if (rc) {
    lf_free(s);
    delete s;
    return rc;
  }
  *out = s;
  return 0;
}

int dsht_lfam3_destroy(dsht_lfam3* s) {
  if (!s) return 0;
  lf_free(s);
  delete s;
  return 0;
}

int dsht_lfam3_set_rotation(dsht_lfam3* s, int run, double omega) {
  if (!s) return fail(DSHT_ESTATE, "LF-AM3 pool is NULL");
  if (run < 0 || run >= s->R) return fail(DSHT_EARG, "run %d out of range [0, %d)", run, s->R);
  const double two = 2.0 * omega;
  DSHT_HIP(hipMemcpy(s->d_two_omega + run, &two, sizeof(double), hipMemcpyHostToDevice));
  return 0;
}

int dsht_lfam3_state(dsht_lfam3* s, int field, int level, double** ptr, long* ncols) {
  if (!s) return fail(DSHT_ESTATE, "LF-AM3 pool is NULL");
  if (level < DSHT_LF_B || level > DSHT_LF_A) return fail(DSHT_EARG, "bad time level %d", level);
  if (!ptr) return fail(DSHT_EARG, "NULL output");
  const long NC = (long)s->R * s->K;
  double* d = nullptr;
  long n = 0;
  switch (field) {
    case DSHT_LF_U: d = s->U[level]; n = NC; break;
    case DSHT_LF_V: d = s->V[level]; n = NC; break;
    case DSHT_LF_TRC: d = s->TS[level]; n = 2 * NC; break;
    case DSHT_LF_SFCPRES: d = s->SP[level]; n = s->R; break;
    default: return fail(DSHT_EARG, "bad field %d", field);
  }
  *ptr = d;
  if (ncols) *ncols = n;
  return 0;
}

int dsht_lfam3_units(const dsht_lfam3* s, int nruns, long* fwd_units, long* inv_units) {
  if (!s) return fail(DSHT_ESTATE, "LF-AM3 pool is NULL");
  if (fwd_units) *fwd_units = (42l * s->K + 9) * nruns;
  if (inv_units) *inv_units = (28l * s->K + 9) * nruns;
  return 0;
}

int dsht_lfam3_copy_run(dsht_lfam3* s, int dst, int src, void* stream) {
  if (!s) return fail(DSHT_ESTATE, "LF-AM3 pool is NULL");
  if (dst < 0 || src < 0 || dst >= s->R || src >= s->R) return fail(DSHT_EARG, "run index out of range");
  if (dst == src) return 0;
  hipStream_t st = (hipStream_t)stream;
  const size_t lay = (size_t)s->K * s->np * sizeof(double), two = (size_t)s->np * sizeof(double);
  for (int lv = 0; lv < 2; lv++) {
    DSHT_HIP(hipMemcpyAsync((char*)s->U[lv] + dst * lay, (char*)s->U[lv] + src * lay, lay, hipMemcpyDeviceToDevice, st));
    DSHT_HIP(hipMemcpyAsync((char*)s->V[lv] + dst * lay, (char*)s->V[lv] + src * lay, lay, hipMemcpyDeviceToDevice, st));
    DSHT_HIP(hipMemcpyAsync((char*)s->TS[lv] + 2 * dst * lay, (char*)s->TS[lv] + 2 * src * lay, 2 * lay,
                            hipMemcpyDeviceToDevice, st));
    DSHT_HIP(hipMemcpyAsync((char*)s->SP[lv] + dst * two, (char*)s->SP[lv] + src * two, two, hipMemcpyDeviceToDevice,
                            st));
  }
  DSHT_HIP(hipMemcpyAsync(s->d_two_omega + dst, s->d_two_omega + src, sizeof(double), hipMemcpyDeviceToDevice, st));
  return 0;
}

int dsht_lfam3_step(dsht_lfam3* s, int nr, void* stream) {
  if (!s) return fail(DSHT_ESTATE, "LF-AM3 pool is NULL");
  if (nr < 0 || nr > s->R) return fail(DSHT_EARG, "nruns = %d out of range [0, %d]", nr, s->R);
  if (nr == 0) return 0;
  hipStream_t st = (hipStream_t)stream;
  dsht_plan* p = s->p;
  const dsht_lfam3_config& c = s->cfg;
  const int K = s->K, I = s->I, L = s->L;
  const long np = s->np;
  const int nc = nr * K, nt = 2 * nc;
  const long ntr = (long)nt * np;
  const double dt = c.dt;
  const double gamma = 1.0 - 2.0 * c.alpha;
  const double c56dt = 5.0 / 6.0 * dt;
  double* const* b2 = s->b2;
  double *UB = s->U[0], *UN = s->U[1], *UA = s->U[2];
  double *VB = s->V[0], *VN = s->V[1], *VA = s->V[2];
  double *TB = s->TS[0], *TN = s->TS[1], *TA = s->TS[2];
  double *PN = s->SP[1], *PA = s->SP[2];
  int rc;
  // val_sub_alpha takes the most scratch: allocated at once, the first step of a plan at T42L20
  // takes 0.47 ms; three allocations and two frees within it made that 1.25
  if (fwd_fused_ok(p) && (rc = workspace_reserve(p, 3, nt, st))) return rc;
  // ---- preparation: barotropic velocities of levels N and B
  const BarotArgs ba{{UN, UB}, {VN, VB}, {b2[UBN], b2[UBB]}, {b2[VBN], b2[VBB]}};
  LF_LAUNCHC(k_lf_uvbarot, np, nr, 2, st, ba, c.depth, s->d_cdk, np, K);
  // ---- predictor; the spectra of (UN, VN) wait in w2, which the fused forms use for nothing else
  const bool spec = lf_wsolve_ok(s);
  if ((rc = lf_vordiv(s, UN, VN, spec ? s->w2 : s->wVD, nc, st))) return rc;
  EosArgs ea;
  ea.ref_dens = c.ref_dens;
  ea.ptemp_dep = -c.beta_t;
  ea.press_dep = 1.0 / (c.ref_dens * (c.cs0 * c.cs0)) - c.ref_temp * (c.beta_t * c.beta_t) / (c.ref_dens * c.cp0);
  ea.salt_dep = c.beta_s;
  ea.ref_temp = c.ref_temp;
  ea.ref_salt = c.ref_salt;
  ea.depth = c.depth;
  ea.grav = c.grav;
  LF_LAUNCHC(k_lf_eos_hyd, np, nr, 1, st, TN, np, K, s->d_zck, s->d_cdk, ea, s->Dens, s->Hyd);
  if ((rc = lf_mom_rhs(s, UN, VN, UB, VB, true, gamma, 1.0 - gamma, PN, nr, st))) return rc;
  if ((rc = lf_mom_grid(s, nc, st))) return rc;
  LF_LAUNCHC(k_lf_pred_uv, np, nr, 1, st, s->URHS, s->VRHS, UN, UB, VN, VB, b2[UBN], b2[VBN], b2[UBB], b2[VBB],
             s->d_two_omega, s->d_mu, c.depth, s->d_cdk, np, I, K, 0.5 * (2.0 * dt), c56dt, c.alpha > 0.0 ? 1 : 0,
             s->Upr, s->Vpr);
  if ((rc = lf_htrc(s, TN, UN, VN, c.depth, nr, st))) return rc;
  // the tracers' updates as the FFT stores their grids, or in a pass after it: T170L60 133 -> 85 (this)
  // and 134 -> 100 us.  Not where a latitude row is no whole number of 128-byte lines, whose store
  // runs share lines with their neighbours': the step at 540 x 270 x 30 2.54 -> 2.55 ms, at
  // 270 x 136 x 30 816 -> 833 us, while 384 x 192 x 30 gains 2 %
  const bool epi = uv_scaled_ok(p) && I % 16 == 0;
  if (epi) {
    InvEpi e;
    e.kind = E_PRED;
    e.in0 = TN;
    e.in1 = TB;
    e.ld = np;
    e.h = c.depth;
    e.c = c56dt;
    if ((rc = inv_epi(p, s->w1, nt, 1, s->TSpr, np, nt, e, st))) return rc;
  } else {
    if ((rc = lf_htrc_grid(s, nt, st))) return rc;
    LF_LAUNCH(k_lf_pred_trc, ntr, st, TN, TB, s->HT, c.depth + 0.0, c56dt, ntr, s->TSpr);
  }
  // ---- corrector
  if ((rc = lf_vordiv(s, s->Upr, s->Vpr, s->wVD, nc, st))) return rc;
  LF_LAUNCHC(k_lf_eos_hyd, np, nr, 1, st, s->TSpr, np, K, s->d_zck, s->d_cdk, ea, s->Dens, s->Hyd);
  const double alpha_ = 0.5, gamma_ = 0.5;
  const double cn = gamma_ + alpha_, cb = 1.0 - alpha_ - gamma_;  // 1 and 0: the present level alone
  if ((rc = lf_mom_rhs(s, s->Upr, s->Vpr, UN, VN, false, cn, cb, PN, nr, st))) return rc;
  // ImplUV (DOGCM_Phys_hspm_vfvm_mod.f90:666-748): implicit vertical viscosity, then
  // backward-Euler lateral viscosity on vorticity and divergence.  On spectra (see k_lf_wsolve), or
  // on the grid for forms whose transforms round more than FP64 does
  if (spec) {
    if ((rc = lf_wsolve(s, true, s->w2, s->wVD, s->d_dmom, 2 * nr, st))) return rc;
  } else {
    if ((rc = lf_mom_grid(s, nc, st))) return rc;
    if ((rc = lf_vsolve(s, true, VSolve{{UN, VN}, {s->URHS, s->VRHS}, {UA, VA}}, nr, 2, st))) return rc;
    if ((rc = lf_uv2vordiv(s, UA, VA, s->wVD, nc, s->d_dmom, st))) return rc;
  }
  if ((rc = dsht_vordiv2uv_d(p, s->wVD, s->wVD + nc, 2l * nc, 1, UA, VA, np, nc, st))) return rc;
  LF_LAUNCHC(k_lf_impl, np, nr, 1, st, UA, VA, UN, VN, b2[UBN], b2[VBN], PN, s->d_two_omega, s->d_mu, s->d_cs, c.depth,
             s->d_cdk, np, I, K, alpha_ * dt, dt, b2[UBT], b2[VBT], b2[AM2], b2[BG2], b2[SPM]);
  // ---- barotropic mode: one iteration with dts = dt / SubCycleNum (rigid lid)
  const double dts = dt / c.sub_cycles;
  if ((rc = dsht_uv2vordiv_d(p, b2[BG2], b2[AM2], np, s->wB, s->wB + nr, 2l * nr, 1, nr, nullptr, st))) return rc;
  if ((rc = lf_fwd_add(s, b2[SPM], s->wB + nr, 2l * nr, s->wC2, nr, s->d_nn1p, st))) return rc;
  if ((rc = dsht_vordiv2uv_d(p, s->wB, s->wB + nr, 2l * nr, 1, b2[UBR], b2[VBR], np, nr, st))) return rc;
  LF_LAUNCH2(k_lf_barot_step, nr, np, st, b2[UBR], b2[VBR], b2[UBN], b2[VBN], s->d_two_omega, s->d_mu, s->d_cs, np, I,
             alpha_ * dts, dts, (long)nr, b2[UBAR], b2[VBAR], b2[AM2], b2[BG2]);
  // HBEBarot_Update_LinFreeSfc, rigid lid: project onto the divergence-free part
  if ((rc = dsht_uv2vordiv_d(p, b2[AM2], b2[BG2], np, s->wB, s->wB + nr, 2l * nr, 1, nr, nullptr, st))) return rc;
  LF_LAUNCH2(k_lf_barot_proj, L, nr, st, s->wB + nr, 2l * nr, s->d_hcoef, s->d_e, c.ref_dens, alpha_ * dts, L, nr,
             s->wDSP, s->wDDiv);
  if ((rc = dsht_inv_d(p, DSHT_VAL, s->wDSP, nr, 1, b2[DSP], np, nr, nullptr, st))) return rc;
  if ((rc = dsht_vordiv2uv_d(p, s->wZero, s->wDDiv, nr, 1, b2[DU], b2[DV], np, nr, st))) return rc;
  // ---- full velocity, time-centred fields, momentum's time levels
  const FinalArgs fa{UA, UN, UB, s->Upr, VA, VN, VB, s->Vpr, b2[UBT], b2[VBT], b2[UBAR], b2[DU], b2[VBAR], b2[DV],
                     b2[DSP], PA, PN, s->SP[0]};
  LF_LAUNCH2(k_lf_final_uv, nc, np, st, fa, np, K, (long)nc);
  // ---- tracers
  if ((rc = lf_div(s, s->Upr, s->Vpr, nc, st))) return rc;
  const double hm = (5.0 * c.depth + 8.0 * c.depth - c.depth) / 12.0;  // the time-centred thickness factor
  if ((rc = lf_htrc(s, s->TSpr, s->Upr, s->Vpr, hm, nr, st))) return rc;
  // ImplTRC (DOGCM_Phys_hspm_vfvm_mod.f90:544-662)
  if (spec) {
    if ((rc = dsht_fwd_d(p, DSHT_VAL, TN, np, s->w2, nt, 1, nt, nullptr, st))) return rc;
    if ((rc = lf_wsolve(s, false, s->w2, s->w1, s->d_dtrc, 2 * nr, st))) return rc;
  } else {
    if ((rc = lf_htrc_grid(s, nt, st))) return rc;
    if ((rc = lf_vsolve(s, false, VSolve{{TN, nullptr}, {s->HT, nullptr}, {TA, nullptr}}, 2 * nr, 1, st))) return rc;
    if ((rc = dsht_fwd_d(p, DSHT_VAL, TA, np, s->w1, nt, 1, nt, s->d_dtrc, st))) return rc;
  }
  if (epi) {
    InvEpi e;
    e.kind = E_TRC;
    e.o1 = TN;
    e.o2 = TB;
    e.ld = np;
    e.h = c.depth;
    return inv_epi(p, s->w1, nt, 1, TA, np, nt, e, st);
  }
  if ((rc = dsht_inv_d(p, DSHT_VAL, s->w1, nt, 1, TA, np, nt, nullptr, st))) return rc;
  LF_LAUNCH(k_lf_trc_final, ntr, st, TA, TN, TB, c.depth, ntr);
  return 0;
}

}  // extern "C"
