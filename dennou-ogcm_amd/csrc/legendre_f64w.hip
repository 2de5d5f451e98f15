// legendre_f64w.hip -- FP64 Legendre contractions with the whole K extent staged in LDS.
//
// Same operators and tables as legendre_f64.hip (the Legendre half of SPMODEL w_xy / xy_w
// and their derivative forms, doc/description/ogcm/space_discretization.tex:199-268), on
// v_mfma_f64_16x16x4f64.  A block owns one zonal wavenumber m and 8 NCT complex columns,
// taken as 16 NCT real ones (re, im of a column side by side, as the Fourier arrays hold
// them), so one MFMA tile covers 8 complex columns and both parts of a value come out in
// neighbouring lanes.  The block requests all of its data at once, puts it into LDS behind
// one barrier, and then every wave runs barrier-free MFMA chains over the row tiles it
// owns, streaming table fragments from L2 one chunk ahead.  The data of one block load
// while the waves of the CU's other blocks multiply.
#include <type_traits>

#include "dsht_internal.hpp"

namespace dsht {

namespace {

__device__ __forceinline__ double4_t mfma64(double a, double b, double4_t c) {
  return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}

// the value of the neighbouring lane (lane ^ 1): the other part (re/im) of the same column
__device__ __forceinline__ double other_part(double x) {
  int lo = __double2loint(x), hi = __double2hiint(x);
  lo = __builtin_amdgcn_mov_dpp(lo, 0xB1, 0xF, 0xF, true);  // quad_perm [1, 0, 3, 2]
  hi = __builtin_amdgcn_mov_dpp(hi, 0xB1, 0xF, 0xF, true);
  return __hiloint2double(hi, lo);
}

// block b runs wavenumber m = b mod 8 + 8 * (b / 8 / nsub) (XCD = b mod 8) and sub-block
// (b / 8) mod nsub: the blocks of one m share an XCD's L2 copy of its tables, and low m
// (long contractions) come first
__device__ __forceinline__ bool xcd_decode_wk(int N, int nsub, int& m, int& sub) {
  const int b = blockIdx.x, idx = b >> 3;
  m = (b & 7) + 8 * (idx / nsub);
  sub = idx % nsub;
  return m <= N;
}

extern __shared__ __attribute__((aligned(16))) double wk_lds[];

// ---------------------------------------------------------------- inverse
// LDS: [input][column tile][row][16], rows = the total wavenumbers of parity 0, padded to
// whole K steps of 4, then those of parity 1.  Wave w owns latitude tiles t = rg WAVES + w,
// + RG WAVES, ...  P products of parity p accumulate into sym (p = 0) or anti (p = 1), H
// products the other way round; the factor i m is applied to the sums.
template <int OP, int NCT, int WAVES>
__global__ __launch_bounds__(WAVES * 64, 2) void k_f64_inv_wk(LegInvArgs a, int CB, int RG) {
  using Tr = InvTraits<OP>;
  constexpr int NIN = Tr::NIN, NTH = WAVES * 64, C8 = 8 * NCT;
  constexpr bool UP = Tr::USE_P, UH = Tr::USE_H;
  constexpr int NTB = (UP ? 1 : 0) + (UH ? 1 : 0);
  constexpr int U = 4;                  // K steps of table fragments per chunk
  constexpr int NP = OP == I_VORDIV2UV ? 2 : 1;  // inputs multiplied by each table
  constexpr int UB = 4;                 // staged elements per thread and round
  int m, sub;
  if (!xcd_decode_wk(a.N, CB * RG, m, sub)) return;
  const int cb = sub % CB, rg = sub / CB;
  const int tid = threadIdx.x, w = tid >> 6, lane = tid & 63, krow = lane >> 4, col = lane & 15;
  const int N = a.N, J2 = a.J2, RT = a.J2pad / TILE;
  const int nE = n_par(N, m, 0), nO = n_par(N, m, 1);
  const int kp0 = cdiv(nE, KCH) * KCH, kp1 = cdiv(nO, KCH) * KCH;
  const int ks0n = cdiv(nE, 4), ks1n = cdiv(nO, 4);
  const int KR = 4 * (ks0n + ks1n);
  const int c0 = cb * C8;
  const double* Win[2] = {a.W0, a.W1};
  const double dm = (double)m;

  // ---- stage: a thread stays in one column and takes every RS-th row; every load of a round is
  // issued (padding reads element 0) before any is used
  constexpr int RS = NTH / C8;
  const int cc = tid % C8;
  const bool cok = c0 + cc < a.ncols;
  const long co = cok ? (long)(c0 + cc) * a.sc : 0;
  double* put = wk_lds + (cc / 8) * KR * 16 + 2 * (cc % 8);
  for (int r0 = tid / C8; r0 < KR; r0 += RS * UB) {
    double re[NIN][UB], im[NIN][UB], pr[UB];
    bool ok[UB];
#pragma unroll
    for (int q = 0; q < UB; q++) {
      const int r = r0 + q * RS;
      const int n = r < 4 * ks0n ? m + 2 * r : m + 1 + 2 * (r - 4 * ks0n);
      ok[q] = r < KR && n <= N && cok;
      const int l = ok[q] ? n * (n + 1) + m : 0, li = ok[q] ? l - 2 * m : 0;
      pr[q] = a.pro ? a.pro[l] : 1.0;
#pragma unroll
      for (int i = 0; i < NIN; i++) {
        re[i][q] = __builtin_nontemporal_load(Win[i] + l * a.sl + co);
        im[i][q] = __builtin_nontemporal_load(Win[i] + li * a.sl + co);
      }
    }
#pragma unroll
    for (int q = 0; q < UB; q++) {
      const int r = r0 + q * RS;
      if (r < KR) {
#pragma unroll
        for (int i = 0; i < NIN; i++) {
          double2 v;
          v.x = ok[q] ? pr[q] * re[i][q] : 0.0;
          v.y = ok[q] && m > 0 ? pr[q] * im[i][q] : 0.0;
          *(double2*)(put + i * NCT * KR * 16 + r * 16) = v;
        }
      }
    }
  }
  __syncthreads();

  const double* tabP = a.tabP + a.offI[m] + lane;
  const double* tabH = a.tabH + a.offI[m] + lane;
  for (int t = rg * WAVES + w; t < RT; t += RG * WAVES) {
    // [P/H][input][column tile][sym/anti]
    double4_t acc[NTB][NP][NCT][2];
#pragma unroll
    for (int x = 0; x < NTB; x++)
#pragma unroll
      for (int i = 0; i < NP; i++)
#pragma unroll
        for (int ct = 0; ct < NCT; ct++) acc[x][i][ct][0] = acc[x][i][ct][1] = double4_t{0, 0, 0, 0};
    const long b0 = (long)t * kp0 * 16, b1 = (long)a.J2pad * kp0 + (long)t * kp1 * 16;
    double cur[NTB][U], nxt[NTB][U];
    // whole chunks: a tile's steps are padded to them in the table (steps past the last one that
    // is needed are not multiplied)
    static_assert(KCH % (4 * U) == 0, "chunks of the padded table");
    auto fetch = [&](double (&x)[NTB][U], long at) {
      const double *P = tabP + at, *H = tabH + at;
#pragma unroll
      for (int u = 0; u < U; u++) {
        if constexpr (UP) x[0][u] = P[u * 64];
        if constexpr (UH) x[NTB - 1][u] = H[u * 64];
      }
    };
    // the row scales are in registers by the time the products are done
    const int jr0 = t * TILE + krow;
    double sN[4], sS[4];
#pragma unroll
    for (int i = 0; i < 4; i++) {
      const int jr = jr0 + 4 * i < J2 ? jr0 + 4 * i : 0;
      sN[i] = a.rs ? a.rs[J2 + jr] : 1.0;
      sS[i] = a.rs ? a.rs[J2 - 1 - jr] : 1.0;
    }
    auto chain = [&](auto PAR) {
      constexpr int par = decltype(PAR)::value, sP = par, sH = 1 - par;
      const int nks = par ? ks1n : ks0n;
      const double* B = wk_lds + (par ? 4 * ks0n * 16 : 0) + krow * 16 + col;
      for (int ks = 0; ks < nks; ks += U) {
        // the next chunk's fragments: of this parity, or the other one's first
        const bool more = ks + U < nks;
        if (more || (par == 0 && ks1n > 0)) fetch(nxt, more ? (par ? b1 : b0) + (ks + U) * 64l : b1);
#pragma unroll
        for (int u = 0; u < U; u++) {
          if (ks + u < nks) {
            double bv[NIN][NCT];
#pragma unroll
            for (int i = 0; i < NIN; i++)
#pragma unroll
              for (int ct = 0; ct < NCT; ct++) bv[i][ct] = B[(i * NCT + ct) * KR * 16 + (ks + u) * 64];
#pragma unroll
            for (int ct = 0; ct < NCT; ct++) {
              // ALPHA: P with input 0, H with input 1; VORDIV2UV: both with both; else with the one
#pragma unroll
              for (int i = 0; i < NP; i++) {
                if constexpr (UP) acc[0][i][ct][sP] = mfma64(cur[0][u], bv[i][ct], acc[0][i][ct][sP]);
                if constexpr (UH)
                  acc[NTB - 1][i][ct][sH] = mfma64(cur[NTB - 1][u], bv[OP == I_ALPHA ? NIN - 1 : i][ct], acc[NTB - 1][i][ct][sH]);
              }
            }
          }
        }
        // the copies (and their wait for the fragments) stay behind the products
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int x = 0; x < NTB; x++)
#pragma unroll
          for (int u = 0; u < U; u++) cur[x][u] = nxt[x][u];
      }
    };
    fetch(cur, b0);
    // vmcnt(0): with nothing in flight at its entry, the loop waits only for its own loads (the
    // wait counts that the compiler merges over the loop's two entries would otherwise also
    // cover the chunk just requested)
    __builtin_amdgcn_s_waitcnt(0x0F70);
    chain(std::integral_constant<int, 0>());
    chain(std::integral_constant<int, 1>());

    // ---- epilogue: north = sym + anti, south = sym - anti, i m, row scale
    const int part = col & 1;
    const double im = part ? dm : -dm;  // (i m z) = (-m z.im, m z.re)
    const bool zero = m == 0 && part;
    const long at = ((long)m * a.gmst + c0) * 2 + col, rowN = (long)(J2 + jr0) * a.gld * 2,
               rowS = (long)(J2 - 1 - jr0) * a.gld * 2, step = 8 * a.gld;
#pragma unroll
    for (int ct = 0; ct < NCT; ct++) {
      if (c0 + ct * 8 + (col >> 1) >= a.ncols) continue;
#pragma unroll
      for (int i = 0; i < 4; i++) {
        if (jr0 + 4 * i >= J2) continue;
        auto put = [&](double2* G, double n, double s) {
          double* g = (double*)G + at + ct * 16;
          g[rowN + i * step] = zero ? 0.0 : n;
          g[rowS - i * step] = zero ? 0.0 : s;
        };
        auto north = [&](int x, int in) { return acc[x][in][ct][0][i] + acc[x][in][ct][1][i]; };
        auto south = [&](int x, int in) { return acc[x][in][ct][0][i] - acc[x][in][ct][1][i]; };
        if constexpr (OP == I_VAL || OP == I_GRADMU) {
          put(a.G0, north(0, 0) * sN[i], south(0, 0) * sS[i]);
        } else if constexpr (OP == I_GRADLAMBDA) {
          put(a.G0, im * other_part(north(0, 0)) * sN[i], im * other_part(south(0, 0)) * sS[i]);
        } else if constexpr (OP == I_VGRAD) {  // no row scale on the value
          const double n = north(0, 0), s = south(0, 0);
          if (a.G0) put(a.G0, n, s);
          if (a.G1) put(a.G1, im * other_part(n) * sN[i], im * other_part(s) * sS[i]);
          if (a.G2) put(a.G2, north(NTB - 1, 0) * sN[i], south(NTB - 1, 0) * sS[i]);
        } else if constexpr (OP == I_ALPHA) {  // i m P.A + H.B
          put(a.G0, (im * other_part(north(0, 0)) + north(NTB - 1, 0)) * sN[i],
              (im * other_part(south(0, 0)) + south(NTB - 1, 0)) * sS[i]);
        } else {  // U = i m P.chi - H.psi, V = i m P.psi + H.chi
          put(a.G0, (im * other_part(north(0, NP - 1)) - north(NTB - 1, 0)) * sN[i],
              (im * other_part(south(0, NP - 1)) - south(NTB - 1, 0)) * sS[i]);
          put(a.G1, (im * other_part(north(0, 0)) + north(NTB - 1, NP - 1)) * sN[i],
              (im * other_part(south(0, 0)) + south(NTB - 1, NP - 1)) * sS[i]);
        }
      }
    }
  }
}

// ---------------------------------------------------------------- forward
// LDS: [input][sym/anti][column tile][latitude][16]: c_j (G_N + G_S) and c_j (G_N - G_S) of
// the north latitudes, padded to whole K steps of 4.  Wave w owns row tiles t = rg WAVES + w,
// + RG WAVES, ...; rows of parity p pair P with sym (p = 0) or anti (p = 1), H with the other.
template <int OP, int NCT, int WAVES>
__global__ __launch_bounds__(WAVES * 64, 2) void k_f64_fwd_wk(LegFwdArgs a, int CB, int RG) {
  using Tr = FwdTraits<OP>;
  constexpr int NIN = Tr::NIN, NOUT = Tr::NOUT, NTH = WAVES * 64, C8 = 8 * NCT;
  constexpr bool UP = Tr::USE_P, UH = Tr::USE_H;
  constexpr int NTB = (UP ? 1 : 0) + (UH ? 1 : 0);
  constexpr int U = 4;                  // K steps of table fragments per chunk
  constexpr int NP = NOUT;              // inputs multiplied by each table
  constexpr int NLD = OP == F_VALSUBALPHA ? 3 : NIN;  // Fourier arrays read
  constexpr int UB = NIN == 2 ? 2 : 4;  // staged latitude pairs per thread and round
  int m, sub;
  if (!xcd_decode_wk(a.N, CB * RG, m, sub)) return;
  const int cb = sub % CB, rg = sub / CB;
  const int tid = threadIdx.x, w = tid >> 6, lane = tid & 63, krow = lane >> 4, col = lane & 15;
  const int N = a.N, J2 = a.J2;
  const int nE = n_par(N, m, 0), nO = n_par(N, m, 1);
  const int tE = cdiv(nE, TILE), RT = tE + cdiv(nO, TILE);
  const int nks = a.J2pad / 4, KR = a.J2pad;  // whole chunks: J2pad is a multiple of 16
  const int c0 = cb * C8;
  const double2* Gm[3] = {a.G0 + (long)m * a.gmst, NLD > 1 ? a.G1 + (long)m * a.gmst : nullptr,
                          NLD > 2 ? a.G2 + (long)m * a.gmst : nullptr};
  const double dm = (double)m;

  // ---- stage: a thread stays in one column and takes every RS-th latitude pair; every load of a
  // round is issued (padding reads the first pair) before any is used
  constexpr int RS = NTH / C8;
  const int cc = tid % C8;
  const bool cok = c0 + cc < a.ncols;
  const long co = cok ? c0 + cc : 0;
  double* put = wk_lds + (cc / 8) * KR * 16 + 2 * (cc % 8);
  for (int j0 = tid / C8; j0 < KR; j0 += RS * UB) {
    double2 gn[NLD][UB], gs[NLD][UB];
    double cw[UB], cw2[UB];
    bool ok[UB];
#pragma unroll
    for (int q = 0; q < UB; q++) {
      const int j = j0 + q * RS;
      ok[q] = j < J2 && cok;
      const int jj = ok[q] ? j : 0;
      cw[q] = a.cw[jj];
      if constexpr (NLD == 3) cw2[q] = a.cw2[jj];
      const long n = (J2 + jj) * a.gld + co, s = (J2 - 1 - jj) * a.gld + co;
#pragma unroll
      for (int i = 0; i < NLD; i++) {
        gn[i][q] = Gm[i][n];
        gs[i][q] = Gm[i][s];
      }
    }
#pragma unroll
    for (int q = 0; q < UB; q++) {
      const int j = j0 + q * RS;
      if (j < KR) {
#pragma unroll
        for (int i = 0; i < NIN; i++) {
          double2 s = make_double2(gn[i][q].x + gs[i][q].x, gn[i][q].y + gs[i][q].y);
          double2 d = make_double2(gn[i][q].x - gs[i][q].x, gn[i][q].y - gs[i][q].y);
          if constexpr (OP == F_VALSUBALPHA) {
            const double f = cw[q] * a.ralpha;
            if (i == 0) {  // with P: c' C - c i m A / R
              const double2 sa = s, da = d;
              s.x = cw2[q] * (gn[2][q].x + gs[2][q].x) + f * (dm * sa.y);
              s.y = cw2[q] * (gn[2][q].y + gs[2][q].y) - f * (dm * sa.x);
              d.x = cw2[q] * (gn[2][q].x - gs[2][q].x) + f * (dm * da.y);
              d.y = cw2[q] * (gn[2][q].y - gs[2][q].y) - f * (dm * da.x);
            } else {  // with H: c B / R
              s = make_double2(f * s.x, f * s.y);
              d = make_double2(f * d.x, f * d.y);
            }
          } else {
            s = make_double2(cw[q] * s.x, cw[q] * s.y);
            d = make_double2(cw[q] * d.x, cw[q] * d.y);
          }
          if (!ok[q]) s = d = make_double2(0.0, 0.0);
          double* at = put + i * 2 * NCT * KR * 16 + j * 16;
          *(double2*)at = s;
          *(double2*)(at + NCT * KR * 16) = d;
        }
      }
    }
  }
  __syncthreads();

  const double* tabP = a.tabP + a.offF[m] + lane;
  const double* tabH = a.tabH + a.offF[m] + lane;
  const long tstride = (long)a.J2pad * 16;  // a row tile's fragments
  double cur[NTB][U], nxt[NTB][U];
  auto fetch = [&](double (&x)[NTB][U], int t, int ks) {
#pragma unroll
    for (int u = 0; u < U; u++) {
      const long o = t * tstride + (long)(ks + u) * 64;
      if constexpr (UP) x[0][u] = tabP[o];
      if constexpr (UH) x[NTB - 1][u] = tabH[o];
    }
  };
  for (int t = rg * WAVES + w; t < RT; t += RG * WAVES) {
    const int par = t < tE ? 0 : 1;
    // [P/H][input][column tile]
    double4_t acc[NTB][NP][NCT];
#pragma unroll
    for (int x = 0; x < NTB; x++)
#pragma unroll
      for (int i = 0; i < NP; i++)
#pragma unroll
        for (int ct = 0; ct < NCT; ct++) acc[x][i][ct] = double4_t{0, 0, 0, 0};
    const double* BP = wk_lds + par * NCT * KR * 16 + krow * 16 + col;
    const double* BH = wk_lds + (1 - par) * NCT * KR * 16 + krow * 16 + col;
    fetch(cur, t, 0);
    // vmcnt(0): with nothing in flight at its entry, the loop waits only for its own loads (the
    // wait counts that the compiler merges over the loop's two entries would otherwise also
    // cover the chunk just requested)
    __builtin_amdgcn_s_waitcnt(0x0F70);
    for (int ks = 0; ks < nks; ks += U) {
      if (ks + U < nks) fetch(nxt, t, ks + U);
#pragma unroll
      for (int u = 0; u < U; u++)
#pragma unroll
        for (int ct = 0; ct < NCT; ct++)
#pragma unroll
          for (int i = 0; i < NP; i++) {
            const int o = ct * KR * 16 + (ks + u) * 64, in = 2 * NCT * KR * 16;
            // ALPHA, VALSUBALPHA: P with input 0, H with input 1; UV2VORDIV: both with both
            if constexpr (UP) acc[0][i][ct] = mfma64(cur[0][u], BP[o + i * in], acc[0][i][ct]);
            if constexpr (UH)
              acc[NTB - 1][i][ct] = mfma64(cur[NTB - 1][u], BH[o + (NIN == 2 && NOUT == 1 ? 1 : i) * in], acc[NTB - 1][i][ct]);
          }
      // the copies (and their wait for the fragments) stay behind the products
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int x = 0; x < NTB; x++)
#pragma unroll
        for (int u = 0; u < U; u++) cur[x][u] = nxt[x][u];
    }

    // ---- epilogue: i m and signs, scale, diagonal, scatter to SPMODEL order
    const int part = col & 1;
    const double im = part ? dm : -dm;  // (i m z) = (-m z.im, m z.re)
#pragma unroll
    for (int ct = 0; ct < NCT; ct++) {
      const int c = c0 + ct * 8 + (col >> 1);
      if (c >= a.ncols) continue;
      // the four rows' diagonals, and the values to add to, in one round of loads
      double dv[NOUT][4], old[NOUT][4];
#pragma unroll
      for (int o = 0; o < NOUT; o++) {
        const double* dg = o == 0 ? a.diag0 : a.diag1;
#pragma unroll
        for (int i = 0; i < 4; i++) {
          const int n = m + par + 2 * ((par ? t - tE : t) * TILE + krow + 4 * i);
          const bool mine = n <= N && !(m == 0 && part);  // a coefficient that this lane stores
          const int l = mine ? n * (n + 1) + (part ? -m : m) : 0;
          dv[o][i] = dg ? dg[l] : 1.0;
          // other coefficients are being stored by other lanes
          if constexpr (OP == F_VAL) old[o][i] = a.add && mine ? a.W0[l * a.sl + (long)c * a.sc] : 0.0;
        }
      }
#pragma unroll
      for (int i = 0; i < 4; i++) {
        const int n = m + par + 2 * ((par ? t - tE : t) * TILE + krow + 4 * i);
        double v[NOUT];
        if constexpr (OP == F_VAL) {
          v[0] = acc[0][0][ct][i];
        } else if constexpr (OP == F_DIVLAMBDA) {
          v[0] = im * other_part(acc[0][0][ct][i]);
        } else if constexpr (OP == F_DIVMU) {
          v[0] = -acc[0][0][ct][i];
        } else if constexpr (OP == F_ALPHA) {  // i m P.A - H.B
          v[0] = im * other_part(acc[0][0][ct][i]) - acc[NTB - 1][0][ct][i];
        } else if constexpr (OP == F_VALSUBALPHA) {
          v[0] = acc[0][0][ct][i] + acc[NTB - 1][0][ct][i];
        } else {  // inputs U cos (0), V cos (1): vor = i m P.V + H.U, div = i m P.U - H.V
          v[0] = im * other_part(acc[0][NP - 1][ct][i]) + acc[NTB - 1][0][ct][i];
          v[NOUT - 1] = im * other_part(acc[0][0][ct][i]) - acc[NTB - 1][NP - 1][ct][i];
        }
        if (n > N || (m == 0 && part)) continue;
        const long at = (n * (n + 1) + (part ? -m : m)) * a.sl + (long)c * a.sc;
#pragma unroll
        for (int o = 0; o < NOUT; o++) {
          double* W = (o == 0 ? a.W0 : a.W1) + at;
          const double x = v[o] * a.scale * dv[o][i];
          *W = OP == F_VAL && a.add ? old[o][i] + x : x;
        }
      }
    }
  }
}

// a block's LDS: two blocks share a CU's 160 KB
constexpr size_t WK_LDS_MAX = 80u << 10;

template <int OP, int NCT>
size_t inv_lds(const dsht_plan* p) {
  return (size_t)InvTraits<OP>::NIN * NCT * 16 * 4 * (cdiv(n_par(p->N, 0, 0), 4) + cdiv(n_par(p->N, 0, 1), 4)) * sizeof(double);
}
template <int OP, int NCT>
size_t fwd_lds(const dsht_plan* p) {
  return (size_t)FwdTraits<OP>::NIN * 2 * NCT * 16 * p->J2pad * sizeof(double);
}

// row groups per (m, column block): enough blocks to fill the chip where the columns alone
// give few, at most one tile per wave
int row_groups(int nblocks, int tiles, int waves) {
  const int most = cdiv(tiles, waves), want = cdiv(1024, nblocks);
  return want < 1 ? 1 : (want < most ? want : most);
}

template <int OP, int NCT, int WAVES>
int inv_go(const dsht_plan* p, const LegInvArgs& a, hipStream_t s) {
  const size_t lds = inv_lds<OP, NCT>(p);
  auto k = k_f64_inv_wk<OP, NCT, WAVES>;
  static const hipError_t attr =
      hipFuncSetAttribute((const void*)k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)WK_LDS_MAX);
  DSHT_HIP(attr);
  const int CB = cdiv(a.ncols, 8 * NCT), m8 = 8 * cdiv(p->N + 1, 8);
  const int RG = row_groups(m8 * CB, a.J2pad / TILE, WAVES);
  hipLaunchKernelGGL(k, dim3((unsigned)m8 * CB * RG), dim3(WAVES * 64), lds, s, a, CB, RG);
  DSHT_HIP(hipGetLastError());
  return 0;
}

template <int OP, int NCT, int WAVES>
int fwd_go(const dsht_plan* p, const LegFwdArgs& a, hipStream_t s) {
  const size_t lds = fwd_lds<OP, NCT>(p);
  auto k = k_f64_fwd_wk<OP, NCT, WAVES>;
  static const hipError_t attr =
      hipFuncSetAttribute((const void*)k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)WK_LDS_MAX);
  DSHT_HIP(attr);
  const int CB = cdiv(a.ncols, 8 * NCT), m8 = 8 * cdiv(p->N + 1, 8);
  const int RT0 = cdiv(n_par(p->N, 0, 0), TILE) + cdiv(n_par(p->N, 0, 1), TILE);
  const int RG = row_groups(m8 * CB, RT0, WAVES);
  hipLaunchKernelGGL(k, dim3((unsigned)m8 * CB * RG), dim3(WAVES * 64), lds, s, a, CB, RG);
  DSHT_HIP(hipGetLastError());
  return 0;
}

// Inverse: two-input operators 8 complex columns per block (their accumulators and data
// double); the others 16 from 4 latitude tiles on, where the spectra's 128-byte runs and the
// tables' reuse win (T170 x 240 fused: 142 us against 158; T85 x 240: 36 against 39), 8 below,
// where more blocks do (T42 x 80: 10.7 against 12.6 us).  Four waves: with eight only one
// block fits the registers of a CU (fused T170 x 240: 164 us).
template <int OP>
int inv_op(const dsht_plan* p, const LegInvArgs& a, hipStream_t s) {
  if constexpr (InvTraits<OP>::NIN == 1) {
    const bool wide = p->leg_cb ? p->leg_cb == 32 : a.ncols > 8 && a.J2pad >= 4 * TILE;
    if (wide && inv_lds<OP, 2>(p) <= WK_LDS_MAX) return inv_go<OP, 2, 4>(p, a, s);
  }
  return inv_go<OP, 1, 4>(p, a, s);
}

// Forward: past 64 north latitudes a block is long (up to 12 row tiles at T170), so eight
// waves share it, and one-input operators take 16 complex columns (F_VAL T170 x 360: 137 us
// against 145 with four waves and 8 columns; UV2VORDIV T170 x 60: 68 against 72); below, four
// waves and 8 columns give more blocks (T85 x 360: 25 us against 27; T42 x 120: 7.0 against 7.9).
template <int OP>
int fwd_op(const dsht_plan* p, const LegFwdArgs& a, hipStream_t s) {
  const bool large = a.ncols > 8 && a.J2pad > 64;
  if constexpr (FwdTraits<OP>::NIN == 1) {
    const bool wide = p->leg_cb ? p->leg_cb == 32 : large;
    if (wide && fwd_lds<OP, 2>(p) <= WK_LDS_MAX) return fwd_go<OP, 2, 8>(p, a, s);
  }
  return large ? fwd_go<OP, 1, 8>(p, a, s) : fwd_go<OP, 1, 4>(p, a, s);
}

}  // namespace

bool leg_inv_staged_ok(const dsht_plan* p, int op) {
  return (inv_nin(op) == 2 ? inv_lds<I_ALPHA, 1>(p) : inv_lds<I_VAL, 1>(p)) <= WK_LDS_MAX;
}
bool leg_fwd_staged_ok(const dsht_plan* p, int op) {
  return (op >= F_ALPHA ? fwd_lds<F_ALPHA, 1>(p) : fwd_lds<F_VAL, 1>(p)) <= WK_LDS_MAX;
}

int launch_leg_inv_staged(const dsht_plan* p, int op, const LegInvArgs& a, hipStream_t s) {
  switch (op) {
    case I_VAL: return inv_op<I_VAL>(p, a, s);
    case I_GRADLAMBDA: return inv_op<I_GRADLAMBDA>(p, a, s);
    case I_GRADMU: return inv_op<I_GRADMU>(p, a, s);
    case I_ALPHA: return inv_op<I_ALPHA>(p, a, s);
    case I_VORDIV2UV: return inv_op<I_VORDIV2UV>(p, a, s);
    case I_VGRAD: return inv_op<I_VGRAD>(p, a, s);
  }
  return fail(DSHT_EARG, "launch_leg_inv_staged: bad op %d", op);
}

int launch_leg_fwd_staged(const dsht_plan* p, int op, const LegFwdArgs& a, hipStream_t s) {
  switch (op) {
    case F_VAL: return fwd_op<F_VAL>(p, a, s);
    case F_DIVLAMBDA: return fwd_op<F_DIVLAMBDA>(p, a, s);
    case F_DIVMU: return fwd_op<F_DIVMU>(p, a, s);
    case F_ALPHA: return fwd_op<F_ALPHA>(p, a, s);
    case F_UV2VORDIV: return fwd_op<F_UV2VORDIV>(p, a, s);
    case F_VALSUBALPHA: return fwd_op<F_VALSUBALPHA>(p, a, s);
  }
  return fail(DSHT_EARG, "launch_leg_fwd_staged: bad op %d", op);
}

}  // namespace dsht
