// s2dw_kernels.hip -- gfx950 kernels of the S2DW analysis and synthesis.
//
// Analysis (one request, all scales), reference s2dw_core_mod.f90:572-775:
//   k_flm_to_fT       flm(l,m) -> fT[l][m] (m fastest, zero for m>l)
//   k_ana_contract    l-contraction T(m,m',n) with the Wigner Delta^l_{m'm}
//                     generated on the fly by a three-term recursion in l per
//                     (m',m) lane, gamma-DFT fused into the per-scale epilogue
//                     -> Tg_j[g][m'][m]                        (618-705)
//   k_beta_ana        beta sum as two length-2hi FFTs per (m,g)  (707-743)
//   k_alpha_c2r       alpha c2r FFT, two real rows per complex FFT (745-768)
// Synthesis, reference 1060-1266:
//   k_alpha_r2c       alpha r2c FFT and scaling                   (1104-1130)
//   k_beta_syn        gamma-DFT + Driscoll-Healy beta quadrature as one
//                     length-2hi FFT per (m,n), +-m' fold      (1132-1198)
//   k_syn_contract    Wigner contraction and f_lm accumulation with
//                     Delta^l_{m'm} generated by a three-term recursion in m'
//                     per (l,m) lane                              (1200-1253)
//   k_flm_final       f_lm in the caller layout + Phi^2 scoeff    (1257-1261)
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <complex>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <vector>

#include "s2dw_dev.h"
#include "s2dw_fft.h"
#include "s2dw_internal.h"
#include "s2dw_moments.h"

namespace s2dw {

// synthesis row (l, m'), m' <= l
__host__ __device__ __forceinline__ long long rowS(long long l, long long mp) { return tri0(l) + mp; }

// ---------------------------------------------------------------------------
// Wigner recursion coefficients at beta = pi/2.
// l-recursion for fixed (m', m):
//   d^{l+1} = u_m * ( A(m',l) * m * d^l + Bc(m',l) * r_m(l) * d^{l-1} )
//   u_m = 1/sqrt((l+1)^2 - m^2), r_m(l) = sqrt(l^2 - m^2),
//   A(m',l) = -(2l+1) m' u_{m'} / l,  Bc(m',l) = -(l+1) r_{m'}(l) u_{m'} / l.
// m'-recursion for fixed (l, m), descending from m' = l:
//   d_{m'-1} = c1 * 2m * d_{m'} - c2 * d_{m'+1},
//   c1 = 1/sqrt((l+m')(l-m'+1)),  c2 = sqrt((l-m')(l+m'+1)) * c1.
// ---------------------------------------------------------------------------
__host__ __device__ __forceinline__ void lrec_coefs(int mp, int l, double *A, double *Bc) {
  if (l == 0) {
    *A = 0.0;
    *Bc = 0.0;
    return;
  }
  const double ld = l, mpd = mp;
  const double a = (ld + 1.0) * (ld + 1.0) - mpd * mpd;
  const double ub = 1.0 / sqrt(a);
  const double rb = sqrt(ld * ld - mpd * mpd);
  *A = -(2.0 * ld + 1.0) * mpd * ub / ld;
  *Bc = -(ld + 1.0) * rb * ub / ld;
}

__host__ __device__ __forceinline__ void mrec_coefs(int l, int mp, double *c1, double *c2) {
  const double a = (double)(l + mp) * (double)(l - mp + 1);
  if (a <= 0.0) {
    *c1 = 0.0;
    *c2 = 0.0;
    return;
  }
  const double c = 1.0 / sqrt(a);
  *c1 = c;
  *c2 = sqrt((double)(l - mp) * (double)(l + mp + 1)) * c;
}

// ---------------------------------------------------------------------------
// Plan-time table kernels.
// ---------------------------------------------------------------------------
// Thin chains Delta^l_{m'k}, k < nk, all l in [m', L).  One thread per (m',k).
__global__ void k_thin_chains(int L, int nk, const double *__restrict__ S0, double *__restrict__ thin) {
  const int id = blockIdx.x * blockDim.x + threadIdx.x;
  if (id >= L * nk) return;
  const int mp = id / nk, k = id % nk;
  const int l0 = mp > k ? mp : k;
  for (int l = mp; l < l0 && l < L; ++l) thin[rowA(mp, l, L) * nk + k] = 0.0;
  if (l0 >= L) return;
  double d = lchain_start(S0, mp, k), dp = 0.0;
  const double md = k;
  double rm = sqrt((double)l0 * l0 - md * md);
  for (int l = l0; l < L; ++l) {
    thin[rowA(mp, l, L) * nk + k] = d;
    double A, Bc;
    lrec_coefs(mp, l, &A, &Bc);
    const double a2 = (double)(l + 1) * (l + 1) - md * md;
    const double u = a2 > 0.5 ? rsqrt(a2) : 0.0;
    const double dn = u * (A * md * d + Bc * rm * dp);
    dp = d;
    d = dn;
    rm = a2 * u;
  }
}

struct RowArgs {
  int L, nk, NCa, NCs, nsc;
  const double *thin;
  const double *thinneg;  // exact Delta^l_{m',-k} (table form), or NULL: sign symmetry
  const double *K;       // K[j + (J+1) l]
  const double *sA;      // [l][c] analysis S parts
  const double *sS;      // [l][c] synthesis weights eps*(2l+1)/(8pi^2)*S part
  const int *slotj;      // [l][2]: scale in slot 0/1 active at l (-1 none)
  int colA_n[kMaxCol];
  int colS_n[kMaxCol];
  int Jp1;
  double *Ba;            // rows (m',l): A, Bc, B[2][NCa]
  double *Bs;            // rows (l,m'): c1, c2, Bs[2][NCs]
};

__global__ void k_build_rows(const RowArgs a) {
  const int L = a.L;
  const long long nrows = (long long)L * (L + 1) / 2;
  const long long id = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (id >= nrows) return;
  // analysis row id -> (m', l)
  {
    // invert rowA: find m' with rowA(m',m') <= id
    int lo = 0, hi = L - 1;
    while (lo < hi) {
      const int mid = (lo + hi + 1) / 2;
      if (rowA(mid, mid, L) <= id) lo = mid;
      else hi = mid - 1;
    }
    const int mp = lo;
    const int l = mp + (int)(id - rowA(mp, mp, L));
    double *row = a.Ba + id * (2 + 2 * a.NCa);
    double A, Bc;
    lrec_coefs(mp, l, &A, &Bc);
    row[0] = A;
    row[1] = Bc;
    for (int s = 0; s < 2; ++s) {
      const int j = a.slotj[2 * l + s];
      for (int c = 0; c < a.NCa; ++c) {
        double v = 0.0;
        if (j >= 0) {
          const int n = a.colA_n[c];
          const int an = n < 0 ? -n : n;
          if (an < a.nk && an <= l) {
            double dl = a.thin[rowA(mp, l, L) * a.nk + an];
            if (n < 0 && a.thinneg) dl = a.thinneg[rowA(mp, l, L) * a.nk + an];
            else if (n < 0 && ((l + mp) & 1)) dl = -dl;
            v = a.K[j + (long long)a.Jp1 * l] * a.sA[(long long)l * a.NCa + c] * dl;
          }
        }
        row[2 + s * a.NCa + c] = v;
      }
    }
  }
  // synthesis row id -> (l, m')
  {
    int lo = 0, hi = L - 1;
    while (lo < hi) {
      const int mid = (lo + hi + 1) / 2;
      if (tri0(mid) <= id) lo = mid;
      else hi = mid - 1;
    }
    const int l = lo;
    const int mp = (int)(id - tri0(l));
    double *row = a.Bs + id * (2 + 2 * a.NCs);
    double c1, c2;
    mrec_coefs(l, mp, &c1, &c2);
    row[0] = c1;
    row[1] = c2;
    for (int s = 0; s < 2; ++s) {
      const int j = a.slotj[2 * l + s];
      for (int c = 0; c < a.NCs; ++c) {
        double v = 0.0;
        if (j >= 0) {
          const int n = a.colS_n[c];
          if (n < a.nk && n <= l) {
            const double dl = a.thin[rowA(mp, l, L) * a.nk + n];
            v = a.K[j + (long long)a.Jp1 * l] * a.sS[(long long)l * a.NCs + c] * dl;
          }
        }
        row[2 + s * a.NCs + c] = v;
      }
    }
  }
}

// ---------------------------------------------------------------------------
// Analysis l-contraction.
// Block (m'-block of P chains per lane, 256 lanes of m).  Each lane carries
// P recursions Delta^l_{m'_p m} over l and accumulates, for the two scales
// active at l (slot j%2), sum_l Delta^l_{m'm} f(l,m) B_j(l,m',c).  When scale
// j ends (l = hi_j - 1) the slot is turned into
//   Tg_j(m,m',g) = i^{-m} sum_c G(g,c) acc_c
// and written to Tg_j[g][m'][m].
// ---------------------------------------------------------------------------
struct AnaArgs {
  int L, N, NCtot, RA, c0, accumulate;
  const double2 *fT;
  const double *Ba;
  const double *S0;
  const int2 *lflush;  // per l: scale ending at l in slot 0 / slot 1 (-1 none)
  const double2 *G;    // [g][c]
  double2 *Tg;
  int hi[kMaxSc];
  long long tgoff[kMaxSc];
};

template <int NC, int P>
__device__ __forceinline__ void ana_flush(const AnaArgs &a, double (&acc)[P][2][NC][2], int s, int j, int mpb, int m) {
  const int hi = a.hi[j];
  if (m < hi) {
    const int rot = m & 3;  // multiply by i^{-m}
#pragma unroll
    for (int p = 0; p < P; ++p) {
      const int mp = mpb + p;
      if (mp < hi) {
        double2 *dst = a.Tg + a.tgoff[j] + (long long)mp * hi + m;
        for (int g = 0; g < a.N; ++g) {
          double xr = 0.0, xi = 0.0;
#pragma unroll
          for (int c = 0; c < NC; ++c) {
            const double2 gc = a.G[g * a.NCtot + a.c0 + c];
            xr += gc.x * acc[p][s][c][0] - gc.y * acc[p][s][c][1];
            xi += gc.x * acc[p][s][c][1] + gc.y * acc[p][s][c][0];
          }
          double yr, yi;
          if (rot == 0) { yr = xr; yi = xi; }
          else if (rot == 1) { yr = xi; yi = -xr; }   // * (-i)
          else if (rot == 2) { yr = -xr; yi = -xi; }
          else { yr = -xi; yi = xr; }                 // * (+i)
          double2 *q = dst + (long long)g * hi * hi;
          if (a.accumulate) {
            const double2 o = *q;
            *q = make_double2(o.x + yr, o.y + yi);
          } else {
            *q = make_double2(yr, yi);
          }
        }
      }
    }
  }
#pragma unroll
  for (int p = 0; p < P; ++p)
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      acc[p][s][c][0] = 0.0;
      acc[p][s][c][1] = 0.0;
    }
}

template <int NC, int P>
__global__ __launch_bounds__(256) void k_ana_contract(const AnaArgs a) {
  const int L = a.L;
  const int mpb = blockIdx.x * P;
  const int wave = threadIdx.x >> 6;
  const int m = blockIdx.y * 256 + threadIdx.x;
  const int mw0 = uniform(blockIdx.y * 256 + wave * 64);
  if (mw0 >= L) return;
  const int lstart = uniform(mpb > mw0 ? mpb : mw0);
  if (lstart >= L) return;
  const bool mval = m < L;
  const double md = (double)m;
  double d[P], dp[P], st[P];
  int l0[P];
#pragma unroll
  for (int p = 0; p < P; ++p) {
    const int mp = mpb + p;
    l0[p] = mp > m ? mp : m;
    st[p] = (mval && mp < L) ? lchain_start(a.S0, mp, m) : 0.0;
    d[p] = 0.0;
    dp[p] = 0.0;
  }
  double rm = (mval && m <= lstart) ? sqrt((double)lstart * lstart - md * md) : 0.0;
  double acc[P][2][NC][2];
#pragma unroll
  for (int p = 0; p < P; ++p)
#pragma unroll
    for (int s = 0; s < 2; ++s)
#pragma unroll
      for (int c = 0; c < NC; ++c) {
        acc[p][s][c][0] = 0.0;
        acc[p][s][c][1] = 0.0;
      }
  for (int l = lstart; l < L; ++l) {
    const double2 f = mval ? a.fT[(long long)l * L + m] : make_double2(0.0, 0.0);
    const double a2 = (double)(l + 1) * (double)(l + 1) - md * md;
    const double u = a2 > 0.5 ? rsqrt(a2) : 0.0;
#pragma unroll
    for (int p = 0; p < P; ++p) {
      const int mp = mpb + p;
      if (mp <= l) {
        const cdptr row = as_const(a.Ba) + rowA(mp, l, L) * a.RA;
        if (l == l0[p]) {
          d[p] = st[p];
          dp[p] = 0.0;
        }
        const double afx = d[p] * f.x, afy = d[p] * f.y;
#pragma unroll
        for (int s = 0; s < 2; ++s)
#pragma unroll
          for (int c = 0; c < NC; ++c) {
            const double bv = row[2 + s * a.NCtot + a.c0 + c];
            acc[p][s][c][0] = fma(afx, bv, acc[p][s][c][0]);
            acc[p][s][c][1] = fma(afy, bv, acc[p][s][c][1]);
          }
        const double dn = u * (row[0] * md * d[p] + row[1] * rm * dp[p]);
        dp[p] = d[p];
        d[p] = dn;
      }
    }
    rm = a2 * u;
    const int2 fl = make_int2(uniform(a.lflush[l].x), uniform(a.lflush[l].y));
    if (fl.x >= 0) ana_flush<NC, P>(a, acc, 0, fl.x, mpb, m);
    if (fl.y >= 0) ana_flush<NC, P>(a, acc, 1, fl.y, mpb, m);
  }
}

// ---------------------------------------------------------------------------
// Analysis l-contraction on FP64 MFMA (v_mfma_f64_16x16x4f64).
//
// Workgroup = 4 consecutive m' (one per wave) x 64 consecutive m.  For a
// group of up to 4 consecutive l, the workgroup stages f(l,m) once in LDS
// (shared by its 4 waves), and each lane advances its recursion
// Delta^l_{m'm} (one (m',m) chain per lane), staging the values in a
// wave-private LDS tile X[k][m].  The A operand of each 16-row m-tile is read
// back in MFMA layout (row = lane%16, k = lane/16) and multiplied by f; the B
// operand holds the 16 columns (2 scale slots x 8 S-columns) of the analysis
// table for the same 4 l, one element per lane (k = lane/16, col = lane%16).
// Eight MFMAs (4 m-tiles x re/im) accumulate C[m][(slot,c)].  Groups never
// cross a scale end, so at a flush each slot column holds exactly one scale;
// the flush stages one m-tile of the slot through LDS, applies the gamma-DFT
// and i^{-m}, and writes Tg_j[g][m'][m].
// Accumulator layout: C[row = lane/16 + 4r][col = lane%16] in element r.
// ---------------------------------------------------------------------------
typedef double v4d __attribute__((ext_vector_type(4)));

struct AnaMfmaArgs {
  AnaArgs a;
  const int *gev;         // per aligned group of 4 l: bit k = a scale ends at 4q + k
  const double *lcoef;    // [m'][l] (A, Bc) of the l-recursion, rows of L + 4 pairs
  long long ba_bytes;     // size of the analysis row table
  const double *uinv;     // [l][m] 1/sqrt((l+1)^2 - m^2), 0 where that is <= 0
  const double *Sa;       // reference Wigner planes [off(l) + m'(l+1) + m] (table form), or NULL
  long long sa_bytes;     // their size in bytes (below 2^32)
  const double2 *phref;   // reference-rounding form: e^{i k pi/2} as the reference rounds it
                          // (k = n - m, index k + phoff), or NULL for exact i^{n-m}
  int phoff;
  int coln[kChunk];       // n of each column of the launch
};

// Groups are the aligned l-ranges [4q, 4q+3]; gev[q] has bit k set when a
// scale ends at l = 4q + k.  Per group the workgroup stages, for its 64 m and
// the 4 l of the group, f(l,m), u_m(l) = 1/sqrt((l+1)^2 - m^2) and
// r_m(l) = sqrt(l^2 - m^2) in LDS (each computed once for the 4 waves); the
// f values of the next kDa - 1 groups are in flight in registers.  The
// l-recursion coefficients of the workgroup's four m' rows sit in LDS.
constexpr int kDa = 4;
constexpr int kAnaMaxN = 32;  // N the MFMA analysis kernel stages the gamma matrix for

__global__ __launch_bounds__(256) void k_ana_contract_mfma(const AnaMfmaArgs args) {
  const AnaArgs &a = args.a;
  __shared__ double Xs[4][4][64];   // per wave: chain values [k][m]
  __shared__ double2 Ff[2][4][64];  // per workgroup: f(l+k, m0+m), double-buffered
  __shared__ double Uf[2][4][64];   // u_m(l+k)
  __shared__ double Rf[2][4][64];   // r_m(l+k)
  __shared__ double2 Fs[4][16][9];  // per wave: flush staging [m][c] of one m-tile (row padded)
  __shared__ double2 Gs[kAnaMaxN][8]; // gamma matrix columns c0..c0+7
  extern __shared__ double2 coef[]; // [4][L]: (A, Bc) of the wave's m' row
  const int L = a.L;
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int mp = uniform(blockIdx.x * 4 + wave);
  const int m0 = blockIdx.y * 64;
  const int lstart = uniform(max((int)blockIdx.x * 4, m0));
  if (lstart >= L) return;  // uniform over the workgroup
  const bool wact = mp < L;
  const int m = m0 + lane;
  const bool mval = m < L;
  const double md = (double)m;
  const int l0 = mp > m ? mp : m;
  const double st = (mval && wact) ? lchain_start(a.S0, mp, m) : 0.0;
  double d = 0.0, dp = 0.0;
  const int kq = lane >> 4, cl = lane & 15;
  const int nc = min(8, a.NCtot - a.c0);
  const int bslot = cl >> 3, bc = cl & 7;
  const bool bcol = bc < nc;
  const int fk = threadIdx.x >> 6, fm = threadIdx.x & 63;  // staged element of this thread
  const double fmd = (double)(m0 + fm);
  // gamma matrix chunk (the flush reads it from LDS: a global load there
  // would wait for the prefetches in flight)
  for (int i = threadIdx.x; i < a.N * 8; i += 256) {
    const int gg = i >> 3, c = i & 7;
    Gs[gg][c] = c < nc ? a.G[gg * a.NCtot + a.c0 + c] : make_double2(0.0, 0.0);
  }
  // coefficient rows of the four m' of this workgroup
  for (int i = threadIdx.x; i < 4 * L; i += 256) {
    const int w = i / L, ll = i - w * L, mpw = blockIdx.x * 4 + w;
    coef[i] = mpw < L ? make_double2(args.lcoef[2 * ((long long)mpw * (L + 4) + ll)],
                                     args.lcoef[2 * ((long long)mpw * (L + 4) + ll) + 1])
                      : make_double2(0.0, 0.0);
  }
  const double2 *crow = coef + wave * L;
  v4d acc_re[4], acc_im[4];
#pragma unroll
  for (int t = 0; t < 4; ++t) {
    acc_re[t] = (v4d){0.0, 0.0, 0.0, 0.0};
    acc_im[t] = (v4d){0.0, 0.0, 0.0, 0.0};
  }
  double(*X)[64] = Xs[wave];
  // f(lg + fk, m0 + fm) through a running pointer; B(m', lg + kq, column) likewise
  // rowA(m', l) is linear in l, so row (m', l0 + 4g) sits 4g rows after row
  // (m', l0); indices are formed as integers and used only where valid
  const bool fval = m0 + fm < L;
  const long long fidx0 = (long long)(lstart + fk) * L + m0 + fm, fstep = 4LL * L;
  const int lbq = lstart + kq;
  const long long bidx0 = (wact ? rowA(mp, lbq, L) * a.RA : 0) + 2 + bslot * a.NCtot + a.c0 + bc;
  const long long bstep = 4LL * a.RA;
  auto loadF = [&](int g) {
    const int lr = lstart + 4 * g + fk;
    return (fval && lr < L) ? a.fT[fidx0 + g * fstep] : make_double2(0.0, 0.0);
  };
  auto loadB = [&](int g) {
    const int lk = lbq + 4 * g;
    return (wact && bcol && lk < L && lk >= mp) ? a.Ba[bidx0 + g * bstep] : 0.0;
  };
  auto stage = [&](int g, double2 f) {
    const int b = g & 1;
    const int lr = lstart + 4 * g + fk;
    const double a2 = (double)(lr + 1) * (double)(lr + 1) - fmd * fmd;
    const double r2 = (double)lr * (double)lr - fmd * fmd;
    Ff[b][fk][fm] = f;
    Uf[b][fk][fm] = a2 > 0.5 ? rsqrt(a2) : 0.0;
    Rf[b][fk][fm] = r2 > 0.5 ? sqrt(r2) : 0.0;
  };
  const int ng = (L - lstart + 3) >> 2;  // groups of this workgroup
  // batches of kDa groups: fa/ba hold the current batch, fb/bb the next one
  // (its loads were issued a whole batch earlier)
  double2 fa[kDa], fb[kDa];
  double ba[kDa], bb[kDa];
#pragma unroll
  for (int u = 0; u < kDa; ++u) {
    fa[u] = loadF(u);
    ba[u] = loadB(u);
    fb[u] = loadF(kDa + u);
    bb[u] = loadB(kDa + u);
  }
  stage(0, fa[0]);
  lds_barrier();
  for (int g0 = 0; g0 < ng; g0 += kDa) {
#pragma unroll
    for (int u = 0; u < kDa; ++u) {
      const int g = g0 + u;
      if (g >= ng) break;  // uniform
      const int l = lstart + 4 * g, buf = g & 1;
      // recursions: values for l..l+3
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const int lk = l + k;
        if (lk == l0) {
          d = st;
          dp = 0.0;
        }
        X[k][lane] = d;  // zero before the chain starts
        const double2 cf = crow[lk < L ? lk : 0];
        const double dn = Uf[buf][k][lane] * (cf.x * md * d + cf.y * Rf[buf][k][lane] * dp);
        dp = d;
        d = dn;
      }
      __builtin_amdgcn_wave_barrier();
      const int ev = as_const(args.gev)[l >> 2];  // scalar load: waits only on lgkmcnt
      const double bfull = ba[u];
      // segments of the group split after each scale end
      int kb = 0;
      while (true) {
        int ke = 3;
        if (ev) {
          const int rest = ev >> kb;
          ke = rest ? kb + __builtin_ctz(rest) : 3;
        }
        const double bval = (kq >= kb && kq <= ke) ? bfull : 0.0;
#pragma unroll
        for (int t = 0; t < 4; ++t) {
          const double dv = X[kq][16 * t + cl];
          const double2 f = Ff[buf][kq][16 * t + cl];
          acc_re[t] = __builtin_amdgcn_mfma_f64_16x16x4f64(dv * f.x, bval, acc_re[t], 0, 0, 0);
          acc_im[t] = __builtin_amdgcn_mfma_f64_16x16x4f64(dv * f.y, bval, acc_im[t], 0, 0, 0);
        }
        if (!((ev >> ke) & 1)) break;
        const int lev = l + ke;
        const ciptr flp = as_const(reinterpret_cast<const int *>(a.lflush)) + 2 * lev;
        const int2 fl = make_int2(flp[0], flp[1]);
        if (wact) {
#pragma unroll
          for (int s = 0; s < 2; ++s) {
            const int j = s == 0 ? fl.x : fl.y;
            if (j < 0) continue;
            const int hj = a.hi[j];
            // one 16-row m-tile at a time: stage C[m][c] of slot s, then lane
            // (row = lane%16, g = lane/16 + 4i) applies the gamma-DFT and i^{-m}
#pragma unroll
            for (int t = 0; t < 4; ++t) {
              __builtin_amdgcn_wave_barrier();
              const bool mine = bslot == s;
              if (mine) {
#pragma unroll
                for (int r = 0; r < 4; ++r) Fs[wave][kq + 4 * r][bc] = make_double2(acc_re[t][r], acc_im[t][r]);
              }
              // zero the slot's columns: every element of a lane lies in its
              // column lane%16, so the lanes of slot s clear all four (the
              // accumulators are VGPRs, so this is a select per element)
#pragma unroll
              for (int r = 0; r < 4; ++r) {
                acc_re[t][r] = mine ? 0.0 : acc_re[t][r];
                acc_im[t][r] = mine ? 0.0 : acc_im[t][r];
              }
              __builtin_amdgcn_wave_barrier();
              const int mm = m0 + 16 * t + cl;
              if (mm < hj && mp < hj) {
                double2 *dst = a.Tg + a.tgoff[j] + (long long)mp * hj + mm;
                const int rot = mm & 3;
                for (int gg = kq; gg < a.N; gg += 4) {
                  double xr2 = 0.0, xi2 = 0.0;
                  for (int c = 0; c < nc; ++c) {
                    const double2 gc = Gs[gg][c];
                    const double2 v = Fs[wave][cl][c];
                    xr2 += gc.x * v.x - gc.y * v.y;
                    xi2 += gc.x * v.y + gc.y * v.x;
                  }
                  double yr, yi;
                  if (rot == 0) { yr = xr2; yi = xi2; }
                  else if (rot == 1) { yr = xi2; yi = -xr2; }
                  else if (rot == 2) { yr = -xr2; yi = -xi2; }
                  else { yr = -xi2; yi = xr2; }
                  double2 *q = dst + (long long)gg * hj * hj;
                  if (a.accumulate) {
                    const double2 o = *q;
                    *q = make_double2(o.x + yr, o.y + yi);
                  } else {
                    *q = make_double2(yr, yi);
                  }
                }
              }
            }
          }
        }
        kb = ke + 1;
        if (kb > 3) break;
      }
      // next group's tile to LDS; at the end of a batch rotate the batches
      // and issue the loads of the batch after the next
      if (u + 1 < kDa) {
        if (g + 1 < ng) stage(g + 1, fa[u + 1]);
      } else {
#pragma unroll
        for (int q = 0; q < kDa; ++q) {
          fa[q] = fb[q];
          ba[q] = bb[q];
        }
        if (g + 1 < ng) stage(g + 1, fa[0]);
#pragma unroll
        for (int q = 0; q < kDa; ++q) {
          fb[q] = loadF(g0 + 2 * kDa + q);
          bb[q] = loadB(g0 + 2 * kDa + q);
        }
      }
      lds_barrier();
    }
  }
}

// Same contraction with every wave independent inside the l loop: the wave
// loads f(l + k, m) for its four m-tiles straight into the MFMA A layout
// (row = lane%16, k = lane/16), computes u_m(l) = 1/sqrt((l+1)^2 - m^2) in
// its own lanes and carries r_m(l+1) = ((l+1)^2 - m^2) u_m(l), and keeps
// the f and B operands of the next kRing - 1 groups in flight in a register
// ring.  The workgroup shares only read-only LDS (coefficient rows, the
// gamma matrix), so the l loop has no workgroup barrier.  One column chunk
// (at most kChunk columns) per launch: Tg is written, never accumulated.
constexpr int kRing = 3;
// s_waitcnt immediate for vmcnt(0) with expcnt and lgkmcnt left at their
// maxima (gfx9 encoding: vmcnt bits 3:0 and 15:14, expcnt 6:4, lgkmcnt 11:8)
constexpr int kWaitVmcnt0 = 0x0F70;

// TAB = true: the Wigner values come from the plan's reference-rounding
// planes (one b64 load per m-tile and group, straight into the MFMA layout)
// instead of the l-recursion; no chain state, no LDS transpose.
// REFPH = true (table form only): the reference-rounding form's phases.
template <bool TAB, bool REFPH = false>
__global__ __launch_bounds__(256, 2) void k_ana_contract_mfma_w(const AnaMfmaArgs args) {
  const AnaArgs &a = args.a;
  __shared__ double Xs[TAB ? 1 : 4][4][64];  // per wave: chain values [k][m]
  __shared__ double2 Fs[4][16][9];    // per wave: flush staging [m][c] of one m-tile (row padded)
  __shared__ double Gb[kAnaMaxN / 8][4][64];  // gamma-DFT B operands: [g block][k-step][lane]
  extern __shared__ double2 coef[];   // [4][L]: (A, Bc) of the wave's m' row
  const int L = a.L;
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int mp = uniform(blockIdx.x * 4 + wave);
  const int m0 = blockIdx.y * 64;
  const int lstart = uniform(max((int)blockIdx.x * 4, m0));
  if (lstart >= L) return;  // uniform over the workgroup
  const bool wact = mp < L;
  const int m = m0 + lane;
  const bool mval = m < L;
  const double md = (double)m, m2 = md * md;
  const int l0 = mp > m ? mp : m;
  const double st = (mval && wact) ? lchain_start(a.S0, mp, m) : 0.0;
  double d = 0.0, dp = 0.0;
  double rm = (double)lstart * lstart - m2;
  rm = rm > 0.5 ? sqrt(rm) : 0.0;  // r_m(lstart)
  (void)m2;
  const int kq = lane >> 4, cl = lane & 15;
  const int nc = min(8, a.NCtot - a.c0);
  const int bslot = cl >> 3, bc = cl & 7;
  const bool bcol = bc < nc;
  // B[k][j] of the gamma-DFT product for g = 8 b + (j & 7), c = k & 7:
  // k < 8 (Re F): Gr (j < 8), Gi (j >= 8); k >= 8 (Im F): -Gi, Gr
  for (int i = threadIdx.x; i < kAnaMaxN / 8 * 4 * 64; i += 256) {
    const int ln = i & 63, stp = (i >> 6) & 3, b = i >> 8;
    const int k = 4 * stp + (ln >> 4), jj = ln & 15, c = k & 7, gg = 8 * b + (jj & 7);
    const double2 gv = gg < a.N && c < nc ? a.G[gg * a.NCtot + a.c0 + c] : make_double2(0.0, 0.0);
    Gb[b][stp][ln] = k < 8 ? (jj < 8 ? gv.x : gv.y) : (jj < 8 ? -gv.y : gv.x);
  }
  // rows of L + 4 pairs, the last 4 zero as in the global table: a group's
  // rows l..l+3 (l <= L-1) are read without a range select
  const int W = L + 4;
  for (int i = threadIdx.x; i < (TAB ? 0 : 4 * W); i += 256) {
    const int w = i / W, ll = i - w * W, mpw = blockIdx.x * 4 + w;
    coef[i] = mpw < L ? make_double2(args.lcoef[2 * ((long long)mpw * W + ll)],
                                     args.lcoef[2 * ((long long)mpw * W + ll) + 1])
                      : make_double2(0.0, 0.0);
  }
  lds_barrier();  // read-only tables from here on
  const double2 *crow = coef + wave * W;
  v4d acc_re[4], acc_im[4];
#pragma unroll
  for (int t = 0; t < 4; ++t) {
    acc_re[t] = (v4d){0.0, 0.0, 0.0, 0.0};
    acc_im[t] = (v4d){0.0, 0.0, 0.0, 0.0};
  }
  double(*X)[64] = Xs[TAB ? 0 : wave];
  // operands of group g: f(lstart + 4g + kq, m0 + 16t + cl) for t < 4 and
  // B(m', lstart + 4g + kq, column cl); indices formed as integers, used
  // only where valid
  const long long fidx0 = (long long)(lstart + kq) * L + m0 + cl, fstep = 4LL * L;
  const int lbq = lstart + kq;
  const long long bidx0 = (wact ? rowA(mp, lbq, L) * a.RA : 0) + 2 + bslot * a.NCtot + a.c0 + bc;
  const long long bstep = 4LL * a.RA;
  const int ng = (L - lstart + 3) >> 2;
  double2 rf[kRing][4];
  double rb[kRing];
  double ru[kRing][4];
  // Operand loads go through buffer descriptors with range checking and are
  // issued for every lane, unconditionally (no branch, exact waits).  No
  // lane needs a validity test: offsets past a buffer (l >= L, or negative
  // row indices, which wrap past 2^31) read zeros, and every other element
  // a lane may read is finite and meets a zero factor or lands in a
  // discarded accumulator: f and B of an l below the chain start multiply
  // A = Delta f = 0 (fT holds zeros for m > l); rows m >= L and columns
  // c >= nc are never flushed; ring slots past the last group are never used.
  const __amdgpu_buffer_rsrc_t fres =
      __builtin_amdgcn_make_buffer_rsrc((void *)a.fT, 0, (int)((long long)L * L * sizeof(double2)), kBufWord3);
  const __amdgpu_buffer_rsrc_t bres = __builtin_amdgcn_make_buffer_rsrc((void *)a.Ba, 0, (int)args.ba_bytes, kBufWord3);
  const __amdgpu_buffer_rsrc_t ures =
      __builtin_amdgcn_make_buffer_rsrc((void *)args.uinv, 0, (int)((long long)L * L * sizeof(double)), kBufWord3);
  const unsigned foff0 = (unsigned)(fidx0 * 16), fstep_b = (unsigned)(fstep * 16);
  const unsigned boff0 = (unsigned)(bidx0 * 8), bstep_b = (unsigned)(bstep * 8);
  const unsigned uoff0 = (unsigned)(((long long)lstart * L + m) * 8), ustep_b = (unsigned)(L * 8);
  // table form: element off(lk) + m'(lk+1) + m, lk = lstart + 4g + kq, as a
  // byte offset carried across groups by second differences (off(l) =
  // sum_{l'<l} (l'+1)^2; the offsets stay below 2^32 for L <= 1024, and reads
  // past the table are range-checked to zero)
  const __amdgpu_buffer_rsrc_t sres =
      __builtin_amdgcn_make_buffer_rsrc((void *)args.Sa, 0, (int)(unsigned)args.sa_bytes, kBufWord3);
  unsigned soff = 0u, sd1 = 0u, sd2 = 0u;
  if (TAB) {
    const unsigned lk = (unsigned)(lstart + kq), mpu = (unsigned)mp;
    soff = 8u * ((lk * (lk + 1u) * (2u * lk + 1u)) / 6u + mpu * (lk + 1u) + (unsigned)(m0 + cl));
    // off(lk + 4) - off(lk) + 4 m' and its change per group
    sd1 = 8u * ((lk + 1u) * (lk + 1u) + (lk + 2u) * (lk + 2u) + (lk + 3u) * (lk + 3u) + (lk + 4u) * (lk + 4u) + 4u * mpu);
    sd2 = 8u * (32u * lk + 144u);
  }
  auto load = [&](int g, double2 (&f)[4], double &b, double (&uv)[4]) {
    const unsigned fo = foff0 + (unsigned)g * fstep_b;
#pragma unroll
    for (int t = 0; t < 4; ++t)
      f[t] = __builtin_bit_cast(double2, __builtin_amdgcn_raw_buffer_load_b128(fres, fo + 256u * t, 0, 0));
    b = __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(bres, boff0 + (unsigned)g * bstep_b, 0, 0));
    if (TAB) {
      // Delta(m', m0 + 16t + cl, lk) for the 4 m-tiles; groups are loaded in
      // order.  Only the first group can have lk < m' (lstart <= m' <=
      // lstart + 3): there the B rows belong to another m' (rowA wraps), so
      // those lanes read zeros instead of a neighbouring plane's values.
      const unsigned so = (g == 0 && lstart + kq < mp) ? 0xFFFFF000u : soff;
#pragma unroll
      for (int t = 0; t < 4; ++t)
        uv[t] = __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(sres, so + 128u * t, 0, 0));
      soff += sd1;
      sd1 += sd2;
      sd2 += 8u * 128u;
    } else {
      const unsigned uo = uoff0 + (unsigned)(4 * g) * ustep_b;
#pragma unroll
      for (int k = 0; k < 4; ++k)
        uv[k] = __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(ures, uo + (unsigned)k * ustep_b, 0, 0));
    }
  };
#pragma unroll
  for (int u = 0; u < kRing; ++u) load(u, rf[u], rb[u], ru[u]);
  for (int g0 = 0; g0 < ng; g0 += kRing) {
#pragma unroll
    for (int u = 0; u < kRing; ++u) {
      const int g = g0 + u;
      if (g >= ng) break;  // uniform
      const int l = lstart + 4 * g;
      // recursions: values for l..l+3
#pragma unroll
      for (int k = 0; k < (TAB ? 0 : 4); ++k) {
        const int lk = l + k;
        // before the chain start d and dp are exactly 0 (every step scales
        // zeros), so the start only sets d
        if (lk == l0) d = st;
        X[k][lane] = d;  // zero before the chain starts
        const double2 cf = crow[lk];  // lk <= L + 2
        const double a2 = (double)(lk + 1) * (double)(lk + 1) - m2;
        const double uu = ru[u][k];  // u_m(lk), 0 where (lk+1)^2 - m^2 <= 0
        const double dn = uu * (cf.x * md * d + cf.y * rm * dp);
        dp = d;
        d = dn;
        rm = a2 * uu;
      }
      __builtin_amdgcn_wave_barrier();
      const int ev = as_const(args.gev)[l >> 2];  // scalar load
      const double bfull = rb[u];
      // A operands of the group, formed in straight-line code before the
      // segment loop so that the waits for the ring stay partial
      double ar[4], ai[4];
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        const double dv = TAB ? ru[u][t] : X[kq][16 * t + cl];
        ar[t] = dv * rf[u][t].x;
        ai[t] = dv * rf[u][t].y;
      }
      int kb = 0;
      while (true) {
        int ke = 3;
        if (ev) {
          const int rest = ev >> kb;
          ke = rest ? kb + __builtin_ctz(rest) : 3;
        }
        const double bval = (kq >= kb && kq <= ke) ? bfull : 0.0;
#pragma unroll
        for (int t = 0; t < 4; ++t) {
          acc_re[t] = __builtin_amdgcn_mfma_f64_16x16x4f64(ar[t], bval, acc_re[t], 0, 0, 0);
          acc_im[t] = __builtin_amdgcn_mfma_f64_16x16x4f64(ai[t], bval, acc_im[t], 0, 0, 0);
        }
        if (!((ev >> ke) & 1)) break;
        const int lev = l + ke;
        const ciptr flp = as_const(reinterpret_cast<const int *>(a.lflush)) + 2 * lev;
        const int2 fl = make_int2(flp[0], flp[1]);
        if (wact) {
#pragma unroll
          for (int s = 0; s < 2; ++s) {
            const int j = s == 0 ? fl.x : fl.y;
            if (j < 0) continue;
            const int hj = a.hi[j];
#pragma unroll
            for (int t = 0; t < 4; ++t) {
              __builtin_amdgcn_wave_barrier();
              const bool mine = bslot == s;
              if (mine) {
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                  double2 x = make_double2(acc_re[t][r], acc_im[t][r]);
                  if (TAB && REFPH) {
                    // the reference-rounding form's e^{i(n-m)pi/2}, applied as staged
                    // (it replaces i^n in gamma and the rotation below)
                    const double2 ph = args.phref[args.coln[bc] - (m0 + 16 * t + kq + 4 * r) + args.phoff];
                    x = make_double2(ph.x * x.x - ph.y * x.y, ph.x * x.y + ph.y * x.x);
                  } else {
                    // i^{-m}: row m = m0 + 16 t + kq + 4 r, so m & 3 = kq
                    x = kq == 0 ? x : kq == 1 ? make_double2(x.y, -x.x) : kq == 2 ? make_double2(-x.x, -x.y)
                                                                                    : make_double2(-x.y, x.x);
                  }
                  Fs[wave][kq + 4 * r][bc] = x;
                }
              }
#pragma unroll
              for (int r = 0; r < 4; ++r) {
                acc_re[t][r] = mine ? 0.0 : acc_re[t][r];
                acc_im[t][r] = mine ? 0.0 : acc_im[t][r];
              }
              __builtin_amdgcn_wave_barrier();
              // gamma-DFT of the tile on MFMA: Y[m][g] = sum_c F[m][c] G[g][c]
              // as a real 16 x 16 x 16 product, A = (Re F | Im F) (row m =
              // lane % 16, k = 4 s + lane / 16), B = [[Gr, Gi], [-Gi, Gr]] in
              // MFMA layout (staged in LDS), D columns j < 8: Re Y(g = 8 b + j),
              // j >= 8: Im Y(g = 8 b + j - 8); the i^{-m} rotation was applied
              // to F when staged
              const double2 fa = Fs[wave][cl][kq], fb = Fs[wave][cl][4 + kq];
              const double av[4] = {fa.x, fb.x, fa.y, fb.y};
              const int mt = m0 + 16 * t + kq;  // rows kq + 4r of the tile
              for (int b = 0; 8 * b < a.N; ++b) {  // uniform trip count
                v4d y = (v4d){0.0, 0.0, 0.0, 0.0};
#pragma unroll
                for (int st = 0; st < 4; ++st)
                  y = __builtin_amdgcn_mfma_f64_16x16x4f64(av[st], Gb[b][st][lane], y, 0, 0, 0);
                const int gg = 8 * b + cl;
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                  const double yi = __shfl_xor(y[r], 8);  // Im Y from the lane 8 columns over
                  const int mm = mt + 4 * r;
                  if (cl < 8 && gg < a.N && mm < hj && mp < hj)
                    a.Tg[a.tgoff[j] + (long long)gg * hj * hj + (long long)mp * hj + mm] = make_double2(y[r], yi);
                }
              }
            }
          }
          // the stores complete here, on this rare path, so that no store
          // is outstanding where the loop reuses their registers (which
          // would otherwise put a full vmcnt wait, draining the operand
          // ring, at the top of every group)
          __builtin_amdgcn_s_waitcnt(kWaitVmcnt0);
        }
        kb = ke + 1;
        if (kb > 3) break;
      }
      __builtin_amdgcn_wave_barrier();  // X reads done before the next group's writes
      // unconditional: groups past the end read zeros, and the same number
      // of loads follows every use, which keeps the waits partial
      load(g + kRing, rf[u], rb[u], ru[u]);
    }
  }
}

// ---------------------------------------------------------------------------
// Split-precision analysis contraction (S2DW_PREC_SPLIT), on int8 MFMA.
//
// T(m, c) = sum_l A(m, l) B(l, c), A = Delta^l_{m'm} f(l, m) (complex),
// B = the real analysis columns, as exact products of fixed-point slices
// (Ozaki's error-free splitting, with integer slices):
//  - each row m of A is scaled by 2^{8D-2-e_m}, 2^{e_m} > max_l |Re, Im f(l,m)|
//    (|Delta| <= 1), rounded to an integer y_A, |y_A| < 2^{8D-2}, and split
//    into D balanced base-256 digits (int8, y = sum_i d_i 256^i); B (|B| <= 1)
//    likewise with scale 2^{8D-2}, its digits precomputed per plan;
//  - v_mfma_i32_16x16x64_i8 sums digit products exactly in int32: for the
//    shift s = i + j (weight 256^s) the K slots of a lane hold A's digits
//    d_0..d_{D-1} of its (m, l) and B's digits e_{s-i} of its (l, c); one
//    MFMA per shift and part (re/im) covers 4 l (K group = lane/16);
//  - the D highest shifts s = D-1 .. 2D-2 are kept; the dropped ones weigh
//    below 256^{D-1} against 256^{2D-2} (relative 2^{-8D+10} per product);
//  - at a scale end the int32 sums are recombined in FP64,
//    T = sum_s C_s 2^{8s + e_m - 16D + 4}, and the flush (gamma-DFT, i^{-m},
//    store) is the FP64 kernel's.
// Quantisation: |A - A~| <= 2^{e_m - 8D + 1}, |B - B~| <= 2^{-8D+1}, relative
// to the row's largest |f| (the scale is per row, over all l).  The products
// of a row at large l are far below that maximum for red spectra, and the
// FFT stages sum ~hi^2 of them: 5 digits measured ~1e-7 on the wavelet
// coefficients at L = 128, 7 digits (2^-54 per product) keep 1e-10.
// Wave = one m' x 16 m (the chains' values come from the plan's Wigner table),
// lane (k = lane/16, row = lane%16); accumulator layout of the i32 MFMA:
// C[row = 4(lane/16) + r][col = lane%16].  Columns: 2 scale slots x 8.
// ---------------------------------------------------------------------------
typedef int v4i __attribute__((ext_vector_type(4)));
constexpr int kSplitD = 7;  // digits per operand

struct AnaSplitArgs {
  AnaArgs a;
  const int *gev;
  const double *Sa;
  long long sa_bytes;
  const uint4 *Bq;   // [rowA(m',l)][16 columns]: bytes 8..8+D-1 = B's digits, most significant first
  long long bq_bytes;
  const int *erow;   // [m]: e_m
};

// balanced base-256 digits of the integer y (|y| < 2^{8D-2}), least
// significant first: w0 = digits 0..3, w1 = digits 4..D-1
template <int D>
__device__ __forceinline__ void split_digits(double y, unsigned &w0, unsigned &w1) {
  static_assert(D >= 5 && D <= 7, "5 to 7 digits");
  const double yh = floor(y * 0x1p-32);
  const double ylo = y - yh * 0x1p32;  // exact, in [0, 2^32)
  const unsigned lo = (unsigned)ylo;
  const unsigned lo2 = lo + 0x80808080u;
  const unsigned cy = lo2 < lo ? 1u : 0u;
  constexpr unsigned hb = D == 5 ? 0x80u : D == 6 ? 0x8080u : 0x808080u;
  constexpr unsigned hm = D == 5 ? 0xFFu : D == 6 ? 0xFFFFu : 0xFFFFFFu;
  const unsigned hi2 = (unsigned)(int)yh + hb + cy;
  w0 = lo2 ^ 0x80808080u;
  w1 = (hi2 ^ hb) & hm;
}

template <int D>
__global__ __launch_bounds__(256) void k_ana_contract_split(const AnaSplitArgs args) {
  const AnaArgs &a = args.a;
  __shared__ double2 Fs[4][16][9];     // per wave: flush staging [m][c]
  __shared__ double2 Gs[kAnaMaxN][8];  // gamma matrix columns c0..c0+7
  __shared__ int Es[16];               // row exponents of the tile
  const int L = a.L;
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int mp = uniform(blockIdx.x * 4 + wave);
  const int m0 = blockIdx.y * 16;
  const int lstart = uniform(max((int)blockIdx.x * 4, m0));
  if (lstart >= L) return;  // uniform over the workgroup
  const bool wact = mp < L;
  const int kq = lane >> 4, cl = lane & 15;
  const int m = m0 + cl;
  const int nc = min(8, a.NCtot - a.c0);
  const int bslot = cl >> 3, bc = cl & 7;
  for (int i = threadIdx.x; i < a.N * 8; i += 256) {
    const int gg = i >> 3, c = i & 7;
    Gs[gg][c] = c < nc ? a.G[gg * a.NCtot + a.c0 + c] : make_double2(0.0, 0.0);
  }
  if (threadIdx.x < 16) Es[threadIdx.x] = m0 + (int)threadIdx.x < L ? args.erow[m0 + threadIdx.x] : 0;
  lds_barrier();
  const double ascale = ldexp(1.0, 8 * D - 2 - Es[cl]);
  v4i cre[D], cim[D];
#pragma unroll
  for (int s = 0; s < D; ++s) {
    cre[s] = (v4i){0, 0, 0, 0};
    cim[s] = (v4i){0, 0, 0, 0};
  }
  // operand loads (range-checked buffer loads, issued unconditionally; see
  // the FP64 kernel): f(lk, m), Delta(m', m, lk) from the table and the B
  // digits of (m', lk, column cl), lk = lstart + 4g + kq
  const __amdgpu_buffer_rsrc_t fres =
      __builtin_amdgcn_make_buffer_rsrc((void *)a.fT, 0, (int)((long long)L * L * sizeof(double2)), kBufWord3);
  const __amdgpu_buffer_rsrc_t sres =
      __builtin_amdgcn_make_buffer_rsrc((void *)args.Sa, 0, (int)(unsigned)args.sa_bytes, kBufWord3);
  const __amdgpu_buffer_rsrc_t qres =
      __builtin_amdgcn_make_buffer_rsrc((void *)args.Bq, 0, (int)args.bq_bytes, kBufWord3);
  const unsigned foff0 = (unsigned)((((long long)(lstart + kq)) * L + m) * 16), fstep_b = (unsigned)(4LL * L * 16);
  const long long qrow0 = wact ? rowA(mp, lstart + kq, L) : 0;
  const unsigned qoff0 = (unsigned)((qrow0 * 16 + cl) * 16), qstep_b = 4u * 16u * 16u;
  unsigned soff, sd1, sd2;
  {
    const unsigned lk = (unsigned)(lstart + kq), mpu = (unsigned)mp;
    soff = 8u * ((lk * (lk + 1u) * (2u * lk + 1u)) / 6u + mpu * (lk + 1u) + (unsigned)m);
    sd1 = 8u * ((lk + 1u) * (lk + 1u) + (lk + 2u) * (lk + 2u) + (lk + 3u) * (lk + 3u) + (lk + 4u) * (lk + 4u) + 4u * mpu);
    sd2 = 8u * (32u * lk + 144u);
  }
  const int ng = (L - lstart + 3) >> 2;
  double2 rf[kRing];
  double rd[kRing];
  uint4 rq[kRing];
  auto load = [&](int g, double2 &f, double &d, uint4 &q) {
    f = __builtin_bit_cast(double2, __builtin_amdgcn_raw_buffer_load_b128(fres, foff0 + (unsigned)g * fstep_b, 0, 0));
    // lk < m' only in the first group: those B rows belong to another m'
    const unsigned so = (g == 0 && lstart + kq < mp) ? 0xFFFFF000u : soff;
    d = __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(sres, so, 0, 0));
    soff += sd1;
    sd1 += sd2;
    sd2 += 8u * 128u;
    q = __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(qres, qoff0 + (unsigned)g * qstep_b, 0, 0));
  };
#pragma unroll
  for (int u = 0; u < kRing; ++u) load(u, rf[u], rd[u], rq[u]);
  for (int g0 = 0; g0 < ng; g0 += kRing) {
#pragma unroll
    for (int u = 0; u < kRing; ++u) {
      const int g = g0 + u;
      if (g >= ng) break;  // uniform
      const int l = lstart + 4 * g;
      const int ev = as_const(args.gev)[l >> 2];  // scalar load
      // A digits of (m, l + kq): bytes 0-7 the real part, 8-15 the imaginary
      unsigned r0, r1, i0, i1;
      split_digits<D>(rint(rd[u] * rf[u].x * ascale), r0, r1);
      split_digits<D>(rint(rd[u] * rf[u].y * ascale), i0, i1);
      const v4i aop = (v4i){(int)r0, (int)r1, (int)i0, (int)i1};
      const uint4 q = rq[u];
      int kb = 0;
      while (true) {
        int ke = 3;
        if (ev) {
          const int rest = ev >> kb;
          ke = rest ? kb + __builtin_ctz(rest) : 3;
        }
        const bool on = kq >= kb && kq <= ke;
        const unsigned q0 = on ? q.x : 0u, q1 = on ? q.y : 0u, q2 = on ? q.z : 0u, q3 = on ? q.w : 0u;
#pragma unroll
        for (int sg = 0; sg < D; ++sg) {
          // B digits e_{s-i} at slot i, s = D - 1 + sg: bytes 8 - sg .. 15 - sg of q
          const int o = 8 - sg, k = o >> 2, r = o & 3;
          const unsigned qa[4] = {q0, q1, q2, q3};
          const unsigned wlo = r ? __builtin_amdgcn_alignbyte(qa[k + 1], qa[k], r) : qa[k];
          const unsigned whi = r ? __builtin_amdgcn_alignbyte(k + 2 < 4 ? qa[k + 2] : 0u, qa[k + 1], r) : qa[k + 1];
          const v4i bre = (v4i){(int)wlo, (int)whi, 0, 0};
          const v4i bim = (v4i){0, 0, (int)wlo, (int)whi};
          cre[sg] = __builtin_amdgcn_mfma_i32_16x16x64_i8(aop, bre, cre[sg], 0, 0, 0);
          cim[sg] = __builtin_amdgcn_mfma_i32_16x16x64_i8(aop, bim, cim[sg], 0, 0, 0);
        }
        if (!((ev >> ke) & 1)) break;
        const int lev = l + ke;
        const ciptr flp = as_const(reinterpret_cast<const int *>(a.lflush)) + 2 * lev;
        const int2 fl = make_int2(flp[0], flp[1]);
        if (wact) {
#pragma unroll
          for (int s = 0; s < 2; ++s) {
            const int j = s == 0 ? fl.x : fl.y;
            if (j < 0) continue;
            const int hj = a.hi[j];
            __builtin_amdgcn_wave_barrier();
            const bool mine = bslot == s;
            if (mine) {
#pragma unroll
              for (int r = 0; r < 4; ++r) {
                const int row = 4 * kq + r;
                double tr = 0.0, ti = 0.0;
#pragma unroll
                for (int sg = D - 1; sg >= 0; --sg) {
                  const int ex = 8 * sg - 8 * D - 4 + Es[row];
                  tr += ldexp((double)cre[sg][r], ex);
                  ti += ldexp((double)cim[sg][r], ex);
                }
                Fs[wave][row][bc] = make_double2(tr, ti);
              }
            }
#pragma unroll
            for (int sg = 0; sg < D; ++sg)
#pragma unroll
              for (int r = 0; r < 4; ++r) {
                cre[sg][r] = mine ? 0 : cre[sg][r];
                cim[sg][r] = mine ? 0 : cim[sg][r];
              }
            __builtin_amdgcn_wave_barrier();
            const int mm = m;
            if (mm < hj && mp < hj) {
              double2 *dst = a.Tg + a.tgoff[j] + (long long)mp * hj + mm;
              const int rot = mm & 3;
              double2 v[8];
#pragma unroll
              for (int c = 0; c < 8; ++c) v[c] = Fs[wave][cl][c];
              for (int i = 0; 4 * i < a.N; ++i) {  // uniform trip count
                const int gg = kq + 4 * i;
                if (gg < a.N) {
                  double xr2 = 0.0, xi2 = 0.0;
#pragma unroll
                  for (int c = 0; c < 8; ++c) {
                    const double2 gc = Gs[gg][c];
                    xr2 += gc.x * v[c].x - gc.y * v[c].y;
                    xi2 += gc.x * v[c].y + gc.y * v[c].x;
                  }
                  double yr, yi;
                  if (rot == 0) { yr = xr2; yi = xi2; }
                  else if (rot == 1) { yr = xi2; yi = -xr2; }
                  else if (rot == 2) { yr = -xr2; yi = -xi2; }
                  else { yr = -xi2; yi = xr2; }
                  dst[(long long)gg * hj * hj] = make_double2(yr, yi);
                }
              }
            }
          }
          __builtin_amdgcn_s_waitcnt(kWaitVmcnt0);
        }
        kb = ke + 1;
        if (kb > 3) break;
      }
      load(g + kRing, rf[u], rd[u], rq[u]);
    }
  }
}

// Plan-time digits of the analysis columns for the split kernel: Bq[row][c]
// (16 bytes) = zeros except bytes 8..8+D-1 = the balanced base-256 digits of
// rint(B 2^{8D-2}), most significant first, B = Ba[row][2 + s NCa + c'] for
// column c = 8 s + c' (zero for c' >= NCa).
template <int D>
__global__ void k_build_bq(long long nrows, int NCa, const double *__restrict__ Ba, uint4 *__restrict__ Bq) {
  const long long id = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (id >= nrows * 16) return;
  const long long row = id >> 4;
  const int c = (int)(id & 15), s = c >> 3, cc = c & 7;
  const double b = cc < NCa ? Ba[row * (2 + 2 * NCa) + 2 + s * NCa + cc] : 0.0;
  unsigned w0, w1;
  split_digits<D>(rint(b * ldexp(1.0, 8 * D - 2)), w0, w1);
  unsigned char dg[8] = {(unsigned char)w0, (unsigned char)(w0 >> 8), (unsigned char)(w0 >> 16),
                         (unsigned char)(w0 >> 24), (unsigned char)w1, (unsigned char)(w1 >> 8), (unsigned char)(w1 >> 16), 0};
  unsigned char out[16] = {};
  for (int k = 0; k < D; ++k) out[8 + k] = dg[D - 1 - k];
  uint4 v;
  v.x = out[0] | out[1] << 8 | out[2] << 16 | (unsigned)out[3] << 24;
  v.y = out[4] | out[5] << 8 | out[6] << 16 | (unsigned)out[7] << 24;
  v.z = out[8] | out[9] << 8 | out[10] << 16 | (unsigned)out[11] << 24;
  v.w = out[12] | out[13] << 8 | out[14] << 16 | (unsigned)out[15] << 24;
  Bq[id] = v;
}

// Row exponents of the split kernel, per transform: e_m with
// 2^{e_m} > max_{l} max(|Re f(l,m)|, |Im f(l,m)|) (0 for an all-zero row).
// One workgroup per m over f_lm as the caller holds it, l fastest: the
// reads are contiguous (L = 512: 3 us, against 145 us for one thread per m
// walking down the columns of the transposed copy).
__global__ __launch_bounds__(256) void k_row_exp(int L, const double2 *__restrict__ flm, int *__restrict__ erow) {
  __shared__ double sh[4];
  const int m = blockIdx.x;
  double mx = 0.0;
  for (int l = m + threadIdx.x; l < L; l += 256) {
    const double2 v = flm[(long long)m * L + l];
    mx = fmax(mx, fmax(fabs(v.x), fabs(v.y)));
  }
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) mx = fmax(mx, __shfl_xor(mx, o));
  if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = mx;
  __syncthreads();
  if (threadIdx.x == 0) {
    mx = fmax(fmax(sh[0], sh[1]), fmax(sh[2], sh[3]));
    int e = 0;
    if (mx > 0.0) (void)frexp(mx, &e);  // mx < 2^e
    erow[m] = e;
  }
}

// u_m(l) = 1/sqrt((l+1)^2 - m^2) table [l][m] (0 where (l+1)^2 - m^2 <= 0).
__global__ void k_uinv(int L, double *__restrict__ u) {
  const long long id = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (id >= (long long)L * L) return;
  const int l = (int)(id / L), m = (int)(id % L);
  const double a2 = (double)(l + 1) * (double)(l + 1) - (double)m * (double)m;
  u[id] = a2 > 0.5 ? 1.0 / sqrt(a2) : 0.0;
}

// l-recursion coefficient table [m'][l] (A, Bc), L + 4 pairs per row (the
// last 4 zero so that a group of 4 rows never reads past a row).
__global__ void k_lcoef(int L, double *__restrict__ lc) {
  const long long id = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  const int W = L + 4;
  if (id >= (long long)L * W) return;
  const int mp = (int)(id / W), l = (int)(id % W);
  double A = 0.0, Bc = 0.0;
  if (l < L && l >= mp) lrec_coefs(mp, l, &A, &Bc);
  lc[2 * id] = A;
  lc[2 * id + 1] = Bc;
}

// ---------------------------------------------------------------------------
// Synthesis Wigner contraction.
// Block (Q consecutive l of one segment, 256 lanes of m).  Each lane runs Q
// recursions Delta^{l_q}_{m'm} downwards in m' from m' = l_q and accumulates
//   f(l_q, m) = sum_{m'} Delta^{l_q}_{m'm} sum_{s,c} Bs(l_q,m',c) Vt_{j_s}(m,m',c)
// ---------------------------------------------------------------------------
struct SynArgs {
  int L, NCtot, RS, c0, accumulate;
  const double *Bs;
  const double *S0;
  const int4 *blocks;  // (l_first, count, scale in slot 0, scale in slot 1)
  const double2 *Vt;
  double2 *fo;
  int hi[kMaxSc];
  long long vtoff[kMaxSc];
};

template <int NC, int Q>
__global__ __launch_bounds__(256) void k_syn_contract(const SynArgs a) {
  const int4 blk = a.blocks[blockIdx.x];
  const int lf = blk.x, cnt = blk.y;
  const int js[2] = {blk.z, blk.w};
  const int L = a.L;
  const int m = blockIdx.y * 256 + threadIdx.x;
  const int wave = threadIdx.x >> 6;
  const int mw0 = uniform(blockIdx.y * 256 + wave * 64);
  const int ltop = uniform(lf + cnt - 1);
  if (mw0 > ltop) return;
  const bool mval = m <= ltop;
  const double two_m = 2.0 * m;
  double d[Q], dn[Q], acc[Q][2];
#pragma unroll
  for (int q = 0; q < Q; ++q) {
    d[q] = 0.0;
    dn[q] = 0.0;
    acc[q][0] = 0.0;
    acc[q][1] = 0.0;
  }
  for (int mp = ltop; mp >= 0; --mp) {
    double2 v[2][NC];
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      const int j = js[s];
      if (j >= 0 && mval) {
        const int hj = a.hi[j];
        const double2 *base = a.Vt + a.vtoff[j] + (long long)mp * hj + m;
        const long long cs = (long long)hj * hj;
#pragma unroll
        for (int c = 0; c < NC; ++c) v[s][c] = base[(a.c0 + c) * cs];
      } else {
#pragma unroll
        for (int c = 0; c < NC; ++c) v[s][c] = make_double2(0.0, 0.0);
      }
    }
#pragma unroll
    for (int q = 0; q < Q; ++q) {
      const int lq = lf + q;
      if (q < cnt && mp <= lq) {
        if (mp == lq) {
          double s0 = 0.0;
          if (m <= lq) {
            s0 = a.S0[tri0(lq) + m];
            if ((lq - m) & 1) s0 = -s0;
          }
          d[q] = s0;
          dn[q] = 0.0;
        }
        const cdptr row = as_const(a.Bs) + rowS(lq, mp) * a.RS;
        double yx = 0.0, yy = 0.0;
#pragma unroll
        for (int s = 0; s < 2; ++s)
#pragma unroll
          for (int c = 0; c < NC; ++c) {
            const double bv = row[2 + s * a.NCtot + a.c0 + c];
            yx = fma(bv, v[s][c].x, yx);
            yy = fma(bv, v[s][c].y, yy);
          }
        acc[q][0] = fma(d[q], yx, acc[q][0]);
        acc[q][1] = fma(d[q], yy, acc[q][1]);
        const double nd = row[0] * two_m * d[q] - row[1] * dn[q];
        dn[q] = d[q];
        d[q] = nd;
      }
    }
  }
#pragma unroll
  for (int q = 0; q < Q; ++q) {
    const int lq = lf + q;
    if (q < cnt && m <= lq && m < L) {
      double2 *dst = a.fo + (long long)lq * L + m;
      if (a.accumulate) {
        const double2 o = *dst;
        *dst = make_double2(o.x + acc[q][0], o.y + acc[q][1]);
      } else {
        *dst = make_double2(acc[q][0], acc[q][1]);
      }
    }
  }
}

// ---------------------------------------------------------------------------
// Synthesis Wigner contraction on FP64 MFMA (v_mfma_f64_16x16x4f64).
//
//   f(l,m) = sum_{m'} Delta^l_{m'm} Y(l,m',m),
//   Y(l,m',m) = sum_{j,c} B_j(m',c,l) Vt_j(c,m',m),
//   B_j(m',c,l) = eps_n (2l+1)/(8 pi^2) K_j(l) S(l,n_c) Delta^l_{m'n_c}.
//
// Workgroup = 64 l (one 16-l column tile per wave) x 16*TM m x one chunk of
// CW consecutive m'.  For each m' (descending) the workgroup stages
// Vt_j(c, m', m-range) of the scales active in its l-range in LDS
// (double-buffered, one barrier per m'); each wave forms Y for its 16 l x
// 16*TM m with MFMAs: A = Vt^T in MFMA layout (row = m = lane%16, k = lane/16)
// read from LDS, B = B_j(m', c, l) (k = lane/16, col = l = lane%16) from the
// per-scale table, one k-step of 4 columns per MFMA, re and im separately.
// The accumulator layout (row = m = lane/16 + 4r, col = l = lane%16) puts
// Y(l, m', m) in the lane that owns the chain Delta^l_{m'm}: each lane owns
// one l and 4*TM values of m, multiplies element-wise, accumulates, and steps
// its chains down to m'-1 (m'-recursion).  Chains with l above the chunk
// start from checkpoint planes (Delta at the chunk's top m' and top m' + 1,
// computed at plan time by the l-recursion); chains with l inside the chunk
// start at m' = l.  The workgroup writes its chunk's partial sums to
// fpart[chunk][m][l]; the assembly kernel adds the chunks.
// ---------------------------------------------------------------------------
constexpr int kSynWgSc = 8;  // scales per workgroup
constexpr int kSynTM = 1;    // 16-row m-tiles per wave

struct SynMfmaArgs {
  int L, NC, NCp, CW, nsc, work0;
  int xcd;              // 1: consecutive work items on one XCD (xcd_tile)
  const int4 *work;     // per workgroup: (l0, m0, chunk, k-steps)
  const double2 *cc;    // [m'][l] (c1, c2)
  const double *S0;
  const double *cp;     // [chunk][2][m][l]
  const double2 *Vt;
  const double *BT;     // per scale: [m' <= ub][NCp][l - lb]
  double2 *fpart;       // [chunk][m][l]
  int lb[kMaxSc], ub[kMaxSc], hi[kMaxSc];
  long long vtoff[kMaxSc], btoff[kMaxSc];
  long long vt_bytes, bt_bytes;  // sizes of Vt and BT (range of the buffer loads)
  const double *Sa;     // reference Wigner planes [off(l) + m'(l+1) + m] (table form), or NULL
  long long sa_bytes;   // their size in bytes (below 2^32)
};

template <int TM, int KSMAX>
__global__ __launch_bounds__(256, KSMAX <= 2 ? 3 : KSMAX <= 4 ? 2 : 1) void k_syn_contract_mfma(const SynMfmaArgs a) {
  constexpr int MW = 16 * TM;                        // m per workgroup
  constexpr int VPT = (KSMAX * 4 * MW + 255) / 256;  // staged V elements per thread (max)
  constexpr int DS = 3;                              // register slots: steps in flight
  extern __shared__ double2 vs[];                    // [2][4 * KSMAX][MW]
  __shared__ int s_j[kSynWgSc];
  const int4 wk = a.work[a.work0 + (a.xcd ? xcd_tile(blockIdx.x, gridDim.x) : (int)blockIdx.x)];
  const int l0 = wk.x, m0 = wk.y, ch = wk.z;
  const int L = a.L, NCp = a.NCp;
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  // scales active anywhere in [l0, l0 + 63]
  int nsw = 0;
  for (int j = 0; j < a.nsc; ++j) {
    if (a.lb[j] <= a.ub[j] && a.lb[j] <= l0 + 63 && a.ub[j] >= l0) {
      if (threadIdx.x == 0) s_j[nsw] = j;
      ++nsw;
    }
  }
  const int K = nsw * NCp, KS = K >> 2, kpc = NCp >> 2;
  const int top = min((ch + 1) * a.CW, L) - 1, bot = ch * a.CW;
  const int nst = top - bot + 1;  // m' steps, m' = top - i
  const int l = l0 + 16 * wave + (lane & 15);
  const bool lval = l < L;
  const int mq = m0 + (lane >> 4);  // chain (t, r) has m = mq + 16t + 4r
  // chains, checkpoint or start values
  double d[TM][4], dn[TM][4], fr[TM][4], fi[TM][4], s0v[TM][4];
#pragma unroll
  for (int t = 0; t < TM; ++t)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int m = mq + 16 * t + 4 * r;
      d[t][r] = dn[t][r] = fr[t][r] = fi[t][r] = s0v[t][r] = 0.0;
      if (lval && m < L && l > top) {
        const double *c0 = a.cp + ((long long)ch * 2 * L + m) * L + l;
        d[t][r] = c0[0];
        dn[t][r] = c0[(long long)L * L];
      }
      if (lval && l >= bot && l <= top && m <= l) {
        const double v = a.S0[tri0(l) + m];
        s0v[t][r] = ((l - m) & 1) ? -v : v;
      }
    }
  lds_barrier();  // s_j
  // V staging: element e = threadIdx.x + 256 i -> (kk = e / MW, mm = e % MW),
  // kk = slot * NCp + c; index of step 0 and the index step per m' (-hj)
  const int nel = K * MW;
  long long vidx[VPT];
  int vh[VPT];
#pragma unroll
  for (int i = 0; i < VPT; ++i) {
    const int e = threadIdx.x + 256 * i;
    vh[i] = 0;  // 0: element unused or outside the scale's block
    vidx[i] = 0;
    if (e < nel) {
      const int kk = e / MW, mm = e - kk * MW;
      const int slot = kk / NCp, c = kk - slot * NCp;
      const int j = s_j[slot];
      const int m = m0 + mm, hj = a.hi[j];
      if (c < a.NC && m < hj) {
        vh[i] = hj;
        vidx[i] = a.vtoff[j] + ((long long)c * hj + top) * hj + m;
      }
    }
  }
  // B operand of k-step ks: B_j(m', c, l), c = 4 (ks mod kpc) + lane/16; index
  // at m' = top, step per m' = NCp * W_j, valid for m' <= ub_j
  long long bidx[KSMAX];
  int bstep[KSMAX], bub[KSMAX];
#pragma unroll
  for (int ks = 0; ks < KSMAX; ++ks) {
    bidx[ks] = 0;
    bstep[ks] = 0;
    bub[ks] = -1;  // no m' valid
    if (ks < KS) {
      const int slot = ks / kpc;
      const int j = s_j[slot];
      const int c = 4 * (ks - slot * kpc) + (lane >> 4);
      const int lb = a.lb[j], ub = a.ub[j], W = ub - lb + 1;
      if (lval && l >= lb && l <= ub) {
        bub[ks] = ub;
        bstep[ks] = NCp * W;
        bidx[ks] = a.btoff[j] + ((long long)top * NCp + c) * W + (l - lb);
      }
    }
  }
  const long long ccidx = (long long)top * L + l;
  double2 sv[DS][VPT];
  double bq[DS][KSMAX];
  double2 cq[DS];
  // V, B and cc go through range-checked buffer loads: lanes and steps with
  // nothing to read (outside a scale's block, or m' below the chunk) use an
  // offset past the end and read zeros, so every load is issued
  // unconditionally and the waits for them stay partial
  const __amdgpu_buffer_rsrc_t vres = __builtin_amdgcn_make_buffer_rsrc((void *)a.Vt, 0, (int)a.vt_bytes, kBufWord3);
  const __amdgpu_buffer_rsrc_t bres = __builtin_amdgcn_make_buffer_rsrc((void *)a.BT, 0, (int)a.bt_bytes, kBufWord3);
  const __amdgpu_buffer_rsrc_t cres =
      __builtin_amdgcn_make_buffer_rsrc((void *)a.cc, 0, (int)((long long)L * L * sizeof(double2)), kBufWord3);
  auto load_step = [&](int i, double2 (&v)[VPT], double (&b)[KSMAX], double2 &c) {
    const int mp = top - i;
    const bool mok = mp >= bot;
#pragma unroll
    for (int q = 0; q < VPT; ++q) {
      const bool ok = mok & (mp < vh[q]);
      const unsigned off = ok ? (unsigned)((vidx[q] - (long long)i * vh[q]) * 16) : kBufOut;
      v[q] = __builtin_bit_cast(double2, __builtin_amdgcn_raw_buffer_load_b128(vres, off, 0, 0));
    }
#pragma unroll
    for (int ks = 0; ks < KSMAX; ++ks) {
      const bool ok = mok & (mp <= bub[ks]);
      const unsigned off = ok ? (unsigned)((bidx[ks] - (long long)i * bstep[ks]) * 8) : kBufOut;
      b[ks] = __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(bres, off, 0, 0));
    }
    const unsigned coff = (mok & lval) ? (unsigned)((ccidx - (long long)i * L) * 16) : kBufOut;
    c = __builtin_bit_cast(double2, __builtin_amdgcn_raw_buffer_load_b128(cres, coff, 0, 0));
  };
  auto commit = [&](int buf, const double2 (&v)[VPT]) {
#pragma unroll
    for (int q = 0; q < VPT; ++q) {
      const int e = threadIdx.x + 256 * q;
      if (e < nel) vs[buf * (KSMAX * 4 * MW) + e] = v[q];
    }
  };
#pragma unroll
  for (int u = 0; u < DS; ++u)
    if (u < nst) load_step(u, sv[u], bq[u], cq[u]);
  commit(0, sv[0]);
  lds_barrier();
  for (int i0 = 0; i0 < nst; i0 += DS) {
#pragma unroll
    for (int u = 0; u < DS; ++u) {
      const int i = i0 + u;
      if (i >= nst) break;  // uniform
      const int mp = top - i, buf = i & 1;
      if (mp == l) {
#pragma unroll
        for (int t = 0; t < TM; ++t)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            d[t][r] = s0v[t][r];
            dn[t][r] = 0.0;
          }
      }
      // Y(l, m', m) for the wave's 16 l x MW m
      v4d yr[TM], yi[TM];
#pragma unroll
      for (int t = 0; t < TM; ++t) {
        yr[t] = (v4d){0.0, 0.0, 0.0, 0.0};
        yi[t] = (v4d){0.0, 0.0, 0.0, 0.0};
      }
      const double2 *V = vs + buf * (KSMAX * 4 * MW);
#pragma unroll
      for (int ks = 0; ks < KSMAX; ++ks) {
        if (ks < KS) {
#pragma unroll
          for (int t = 0; t < TM; ++t) {
            const double2 v = V[(4 * ks + (lane >> 4)) * MW + 16 * t + (lane & 15)];
            yr[t] = __builtin_amdgcn_mfma_f64_16x16x4f64(v.x, bq[u][ks], yr[t], 0, 0, 0);
            yi[t] = __builtin_amdgcn_mfma_f64_16x16x4f64(v.y, bq[u][ks], yi[t], 0, 0, 0);
          }
        }
      }
      // accumulate and step the chains to m' - 1
      const double c1 = 2.0 * cq[u].x, c2 = cq[u].y;
#pragma unroll
      for (int t = 0; t < TM; ++t)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          fr[t][r] = fma(d[t][r], yr[t][r], fr[t][r]);
          fi[t][r] = fma(d[t][r], yi[t][r], fi[t][r]);
          const double md = (double)(mq + 16 * t + 4 * r);
          const double nd = (c1 * md) * d[t][r] - c2 * dn[t][r];
          dn[t][r] = d[t][r];
          d[t][r] = nd;
        }
      if (i + 1 < nst) commit(buf ^ 1, sv[(u + 1) % DS]);
      load_step(i + DS, sv[u], bq[u], cq[u]);  // past the chunk: zeros (no tail branch)
      lds_barrier();
    }
  }
  if (lval) {
#pragma unroll
    for (int t = 0; t < TM; ++t)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int m = mq + 16 * t + 4 * r;
        if (m < L) a.fpart[((long long)ch * L + m) * L + l] = make_double2(fr[t][r], fi[t][r]);
      }
  }
}

// A wave of 16 l from lw with m-tile m0 and a chunk from m' = bot up.
__host__ __device__ __forceinline__ bool syn_wave_idle(int lw, int m0, int bot, int L) {
  return lw >= L || lw + 15 < m0 || lw + 15 < bot;
}

// Same contraction with every wave independent inside the m' loop: each
// lane loads its V operand (Vt_j(c, m', m) for its k = c and row m) straight
// into the MFMA A layout in the register ring, so no V tile is staged in LDS
// and the m' loop has no workgroup barrier.
// TAB = true: Delta^l_{m'm} comes from the plan's reference-rounding planes
// (4 b64 loads per lane and m' step, in flight in the ring with V and B)
// instead of checkpoints and the m'-recursion.  Elements with m > l are read
// from neighbouring rows (finite) and land in partial sums the assembly
// never reads; elements with m' > l meet Y = 0 (B is zero there).
template <int TM, int KSMAX, bool TAB>
__global__ __launch_bounds__(256, KSMAX <= 2 ? 3 : KSMAX <= 4 ? 2 : 1) void k_syn_contract_mfma_w(const SynMfmaArgs a) {
  static_assert(TM == 1, "one 16-row m-tile per wave");
  constexpr int MW = 16 * TM;                        // m per workgroup
  constexpr int DS = 3;                              // register slots: steps in flight
  __shared__ int s_jw[4][kSynWgSc];
  const int4 wk = a.work[a.work0 + (a.xcd ? xcd_tile(blockIdx.x, gridDim.x) : (int)blockIdx.x)];
  const int l0 = wk.x, m0 = wk.y, ch = wk.z;
  const int L = a.L, NCp = a.NCp;
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  // scales active anywhere in the wave's own 16 l: a tile of 64 l that spans
  // more scales costs each wave only its own (two at dilation 2)
  const int lw = uniform(l0 + 16 * wave);
  int *s_j = s_jw[wave];
  int nsw = 0;
  for (int j = 0; j < a.nsc; ++j) {
    if (a.lb[j] <= a.ub[j] && a.lb[j] <= lw + 15 && a.ub[j] >= lw) {
      if (lane == 0) s_j[nsw] = j;
      ++nsw;
    }
  }
  const int K = nsw * NCp, KS = K >> 2, kpc = NCp >> 2;
  // the wave's m' <= l ends at lw + 15
  const int top = min(min((ch + 1) * a.CW, L) - 1, lw + 15), bot = ch * a.CW;
  const int nst = top - bot + 1;  // m' steps, m' = top - i
  const int l = l0 + 16 * wave + (lane & 15);
  const bool lval = l < L;
  const int mq = m0 + (lane >> 4);  // chain (t, r) has m = mq + 16t + 4r
  // chains, checkpoint or start values
  double d[TM][4], dn[TM][4], fr[TM][4], fi[TM][4], s0v[TM][4];
#pragma unroll
  for (int t = 0; t < TM; ++t)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int m = mq + 16 * t + 4 * r;
      d[t][r] = dn[t][r] = fr[t][r] = fi[t][r] = s0v[t][r] = 0.0;
      if (!TAB && lval && m < L && l > top) {
        const double *c0 = a.cp + ((long long)ch * 2 * L + m) * L + l;
        d[t][r] = c0[0];
        dn[t][r] = c0[(long long)L * L];
      }
      if (!TAB && lval && l >= bot && l <= top && m <= l) {
        const double v = a.S0[tri0(l) + m];
        s0v[t][r] = ((l - m) & 1) ? -v : v;
      }
    }
  lds_barrier();  // s_j
  // nothing of the wave's l reaches this m-tile (m <= l) or chunk (m' <= l):
  // the assembly never reads its partial sums
  if (syn_wave_idle(lw, m0, bot, L)) return;
  // only a chunk that some l of the wave lies in or below starts chains
  // inside the loop; below the wave's l they start at the checkpoint
  const bool starts = top >= lw;
  // table form: element off(l) + m'(l+1) + mq + 4r as a byte offset, from
  // m' = top down by l+1 per step (lanes past L use row L-1; offsets that
  // wrap below zero or pass the table read zeros)
  const __amdgpu_buffer_rsrc_t sres =
      __builtin_amdgcn_make_buffer_rsrc((void *)a.Sa, 0, (int)(unsigned)a.sa_bytes, kBufWord3);
  unsigned soff = 0u, sst = 0u;
  if (TAB) {
    const unsigned lc = (unsigned)min(l, L - 1);
    soff = 8u * ((lc * (lc + 1u) * (2u * lc + 1u)) / 6u + (unsigned)top * (lc + 1u) + (unsigned)mq);
    sst = 8u * (lc + 1u);
  }
  // V operand of k-step ks, loaded by each lane in the MFMA A layout
  // (row m = m0 + lane%16, k = lane/16): Vt_j(c, m', m), c = 4 (ks mod kpc)
  // + lane/16; index at m' = top and the step per m' (-hj); vh = 0 where the
  // element is outside the scale's block
  // Offsets are byte offsets below 2^31 (the plan keeps Vt, BT below that);
  // the per-step strides depend on the scale only, so they stay uniform and
  // the step products are scalar.
  unsigned vof[KSMAX], vst[KSMAX];
  int vh[KSMAX];
#pragma unroll
  for (int ks = 0; ks < KSMAX; ++ks) {
    vh[ks] = 0;
    vof[ks] = 0u;
    vst[ks] = 0u;
    if (ks < KS) {
      const int slot = ks / kpc;
      const int j = __builtin_amdgcn_readfirstlane(s_j[slot]);
      const int c = 4 * (ks - slot * kpc) + (lane >> 4);
      const int m = m0 + (lane & 15), hj = a.hi[j];
      vst[ks] = (unsigned)hj * 16u;
      if (c < a.NC && m < hj) {
        vh[ks] = hj;
        vof[ks] = (unsigned)((a.vtoff[j] + ((long long)c * hj + top) * hj + m) * 16);
      }
    }
  }
  // B operand of k-step ks: B_j(m', c, l), c = 4 (ks mod kpc) + lane/16; index
  // at m' = top, step per m' = NCp * W_j, valid for m' <= ub_j
  unsigned bof[KSMAX], bst[KSMAX];
  int bub[KSMAX];
#pragma unroll
  for (int ks = 0; ks < KSMAX; ++ks) {
    bof[ks] = 0u;
    bst[ks] = 0u;
    bub[ks] = -1;  // no m' valid
    if (ks < KS) {
      const int slot = ks / kpc;
      const int j = __builtin_amdgcn_readfirstlane(s_j[slot]);
      const int c = 4 * (ks - slot * kpc) + (lane >> 4);
      const int lb = a.lb[j], ub = a.ub[j], W = ub - lb + 1;
      bst[ks] = (unsigned)(NCp * W) * 8u;
      if (lval && l >= lb && l <= ub) {
        bub[ks] = ub;
        bof[ks] = (unsigned)((a.btoff[j] + ((long long)top * NCp + c) * W + (l - lb)) * 8);
      }
    }
  }
  const unsigned cof = (unsigned)(((long long)top * L + l) * 16), cst = (unsigned)L * 16u;
  double2 sv[DS][KSMAX];
  double bq[DS][KSMAX];
  double2 cq[DS];
  double dq[TAB ? DS : 1][4];
  // V, B and cc go through range-checked buffer loads: lanes and steps with
  // nothing to read (outside a scale's block, or m' below the chunk) use an
  // offset past the end and read zeros, so every load is issued
  // unconditionally and the waits for them stay partial
  const __amdgpu_buffer_rsrc_t vres = __builtin_amdgcn_make_buffer_rsrc((void *)a.Vt, 0, (int)a.vt_bytes, kBufWord3);
  const __amdgpu_buffer_rsrc_t bres = __builtin_amdgcn_make_buffer_rsrc((void *)a.BT, 0, (int)a.bt_bytes, kBufWord3);
  const __amdgpu_buffer_rsrc_t cres =
      __builtin_amdgcn_make_buffer_rsrc((void *)a.cc, 0, (int)((long long)L * L * sizeof(double2)), kBufWord3);
  auto load_step = [&](int i, double2 (&v)[KSMAX], double (&b)[KSMAX], double2 &c) {
    const int mp = top - i;
    const bool mok = mp >= bot;
#pragma unroll
    for (int q = 0; q < KSMAX; ++q) {
      const bool ok = mok & (mp < vh[q]);
      const unsigned off = ok ? vof[q] - (unsigned)i * vst[q] : kBufOut;
      v[q] = __builtin_bit_cast(double2, __builtin_amdgcn_raw_buffer_load_b128(vres, off, 0, 0));
    }
#pragma unroll
    for (int ks = 0; ks < KSMAX; ++ks) {
      const bool ok = mok & (mp <= bub[ks]);
      const unsigned off = ok ? bof[ks] - (unsigned)i * bst[ks] : kBufOut;
      b[ks] = __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(bres, off, 0, 0));
    }
    if (!TAB) {
      const unsigned coff = (mok & lval) ? cof - (unsigned)i * cst : kBufOut;
      c = __builtin_bit_cast(double2, __builtin_amdgcn_raw_buffer_load_b128(cres, coff, 0, 0));
    }
  };
  // table form: the 4 Delta values of step i (steps are loaded in order)
  auto load_d = [&](double (&dv)[4]) {
#pragma unroll
    for (int r = 0; r < 4; ++r)
      dv[r] = __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(sres, soff + 32u * r, 0, 0));
    soff -= sst;
  };
#pragma unroll
  for (int u = 0; u < DS; ++u) {
    load_step(u, sv[u], bq[u], cq[u]);  // steps past the chunk read zeros
    if (TAB) load_d(dq[TAB ? u : 0]);
  }
  for (int i0 = 0; i0 < nst; i0 += DS) {
#pragma unroll
    for (int u = 0; u < DS; ++u) {
      const int i = i0 + u;
      if (i >= nst) break;  // uniform
      const int mp = top - i;
      if (!TAB && starts && mp == l) {
#pragma unroll
        for (int t = 0; t < TM; ++t)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            d[t][r] = s0v[t][r];
            dn[t][r] = 0.0;
          }
      }
      if (TAB) {
#pragma unroll
        for (int r = 0; r < 4; ++r) d[0][r] = dq[TAB ? u : 0][r];
      }
      // Y(l, m', m) for the wave's 16 l x MW m
      v4d yr[TM], yi[TM];
#pragma unroll
      for (int t = 0; t < TM; ++t) {
        yr[t] = (v4d){0.0, 0.0, 0.0, 0.0};
        yi[t] = (v4d){0.0, 0.0, 0.0, 0.0};
      }
#pragma unroll
      for (int ks = 0; ks < KSMAX; ++ks) {
        if (ks < KS) {
          yr[0] = __builtin_amdgcn_mfma_f64_16x16x4f64(sv[u][ks].x, bq[u][ks], yr[0], 0, 0, 0);
          yi[0] = __builtin_amdgcn_mfma_f64_16x16x4f64(sv[u][ks].y, bq[u][ks], yi[0], 0, 0, 0);
        }
      }
      // accumulate and step the chains to m' - 1
      const double c1 = 2.0 * cq[u].x, c2 = cq[u].y;
#pragma unroll
      for (int t = 0; t < TM; ++t)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          fr[t][r] = fma(d[t][r], yr[t][r], fr[t][r]);
          fi[t][r] = fma(d[t][r], yi[t][r], fi[t][r]);
          if (!TAB) {
            const double md = (double)(mq + 16 * t + 4 * r);
            const double nd = (c1 * md) * d[t][r] - c2 * dn[t][r];
            dn[t][r] = d[t][r];
            d[t][r] = nd;
          }
        }
      load_step(i + DS, sv[u], bq[u], cq[u]);  // past the chunk: zeros (no tail branch)
      if (TAB) load_d(dq[TAB ? u : 0]);
    }
  }
  if (lval) {
#pragma unroll
    for (int t = 0; t < TM; ++t)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int m = mq + 16 * t + 4 * r;
        if (m < L) a.fpart[((long long)ch * L + m) * L + l] = make_double2(fr[t][r], fi[t][r]);
      }
  }
}

// Checkpoint planes for the chunked synthesis: for chunk c (top m' = T_c),
// cp[c][p][m][l] = Delta^l_{T_c + p, m} for l > T_c (0 otherwise), p = 0, 1,
// from the l-recursion.  One thread per (c, p, m).
__global__ void k_syn_checkpoints(int L, int CW, int nck, const double *__restrict__ S0, double *__restrict__ cp) {
  const int id = blockIdx.x * blockDim.x + threadIdx.x;
  if (id >= nck * 2 * L) return;
  const int m = id % L, p = (id / L) & 1, c = id / (2 * L);
  const int T = (c + 1) * CW - 1;
  const int mp = T + p;
  double *out = cp + ((long long)(c * 2 + p) * L + m) * L;
  const int l0 = mp > m ? mp : m;
  for (int l = 0; l < L; ++l)
    if (l <= T || l < l0) out[l] = 0.0;
  if (l0 >= L) return;
  double dd = lchain_start(S0, mp, m), dp = 0.0;
  const double md = m;
  double rm = sqrt((double)l0 * l0 - md * md);
  for (int l = l0; l < L; ++l) {
    if (l > T) out[l] = dd;
    double A, Bc;
    lrec_coefs(mp, l, &A, &Bc);
    const double a2 = (double)(l + 1) * (l + 1) - md * md;
    const double u = a2 > 0.5 ? rsqrt(a2) : 0.0;
    const double dnx = u * (A * md * dd + Bc * rm * dp);
    dp = dd;
    dd = dnx;
    rm = a2 * u;
  }
}

// Synthesis tables for the MFMA contraction: m'-recursion coefficients
// cc[m'][l] and per-scale B_j[m'][c][l - lb_j].
struct SynTabArgs {
  int L, nk, NC, NCp, nsc, Jp1;
  const double *thin;
  const double *K;
  const double *sS;     // [l][c]
  int colS_n[kMaxCol];
  int lb[kMaxSc], ub[kMaxSc];
  long long btoff[kMaxSc];
  double *BT;
  double2 *cc;
};

__global__ void k_syn_cc(int L, double2 *__restrict__ cc) {
  const long long id = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (id >= (long long)L * L) return;
  const int mp = (int)(id / L), l = (int)(id % L);
  double c1 = 0.0, c2 = 0.0;
  if (mp <= l) mrec_coefs(l, mp, &c1, &c2);
  cc[id] = make_double2(c1, c2);
}

__global__ void k_syn_btab(const SynTabArgs a, int j, long long count) {
  const long long id = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (id >= count) return;
  const int W = a.ub[j] - a.lb[j] + 1;
  const int l = a.lb[j] + (int)(id % W);
  const long long r = id / W;
  const int c = (int)(r % a.NCp), mp = (int)(r / a.NCp);
  double v = 0.0;
  if (c < a.NC && mp <= l) {
    const int n = a.colS_n[c];
    if (n < a.nk && n <= l) {
      const double dl = a.thin[rowA(mp, l, a.L) * a.nk + n];
      v = a.K[j + (long long)a.Jp1 * l] * a.sS[(long long)l * a.NC + c] * dl;
    }
  }
  a.BT[a.btoff[j] + id] = v;
}

// flm(l,m) = sum over chunks c <= l/CW of fpart[c][m][l] (covered l, m <= l)
//          + Phi2(l) scoeff(l,m) (l,m < bl).
__global__ void k_flm_final_chunks(int L, int bl, int CW, const double2 *__restrict__ fpart,
                                   const unsigned char *__restrict__ covered, const double *__restrict__ Phi2,
                                   const double2 *__restrict__ scoeff, double2 *__restrict__ flm) {
  const long long id = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (id >= (long long)L * L) return;
  const int m = (int)((unsigned)id / (unsigned)L), l = (int)id - m * L;  // id < L^2 < 2^31
  double2 v = make_double2(0.0, 0.0);
  if (m <= l && covered[l]) {
    const int nc = l / CW;
    for (int c = 0; c <= nc; ++c) {
      const double2 x = fpart[((long long)c * L + m) * L + l];
      v.x += x.x;
      v.y += x.y;
    }
  }
  if (l < bl && m < bl) {
    const double2 s = scoeff[l + (long long)bl * m];
    v.x += Phi2[l] * s.x;
    v.y += Phi2[l] * s.y;
  }
  flm[id] = v;
}

// ---------------------------------------------------------------------------
// Layout kernels.
// ---------------------------------------------------------------------------
// fT[l][m] = flm(l,m) for m <= l, 0 otherwise (32x32 tiles through LDS).
// With sc: also the scaling coefficients (k_scoeff), from the first bl^2
// threads of the grid (L^2 >= bl^2 of them): one launch fewer for plans that
// run on one stream.  rot >= 0: times i^{rot - m} (exact), which the
// contraction by parity would apply to every output otherwise.
__global__ void k_flm_to_fT(int L, const double2 *__restrict__ flm, double2 *__restrict__ fT, int bl,
                            double2 *__restrict__ sc, int rot) {
  __shared__ double2 tile[32][33];
  const int l0 = blockIdx.x * 32, m0 = blockIdx.y * 32;
  const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;  // 256 threads: 32 x 8
  if (sc) {
    const int id = (blockIdx.y * gridDim.x + blockIdx.x) * 256 + threadIdx.x;
    if (id < bl * bl) sc[id] = flm[id % bl + (long long)L * (id / bl)];
  }
  for (int r = ty; r < 32; r += 8) {
    const int l = l0 + tx, m = m0 + r;  // read flm[l + L m]: l fastest
    tile[r][tx] = (l < L && m < L) ? flm[l + (long long)L * m] : make_double2(0.0, 0.0);
  }
  __syncthreads();
  for (int r = ty; r < 32; r += 8) {
    const int l = l0 + r, m = m0 + tx;
    double2 x = (m <= l) ? tile[tx][r] : make_double2(0.0, 0.0);
    const int k = rot < 0 ? 0 : (rot - m) & 3;
    if (k & 1) x = make_double2(-x.y, x.x);
    if (k & 2) x = make_double2(-x.x, -x.y);
    if (l < L && m < L) fT[(long long)l * L + m] = x;
  }
}

// flm(l,m) = fo[l][m] (m <= l, l covered) + Phi2(l) scoeff(l,m) (l,m < bl).
__global__ void k_flm_final(int L, int bl, const double2 *__restrict__ fo, const unsigned char *__restrict__ covered,
                            const double *__restrict__ Phi2, const double2 *__restrict__ scoeff,
                            double2 *__restrict__ flm) {
  __shared__ double2 tile[32][33];
  const int l0 = blockIdx.x * 32, m0 = blockIdx.y * 32;
  const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;
  for (int r = ty; r < 32; r += 8) {
    const int l = l0 + r, m = m0 + tx;  // read fo[l][m]: m fastest
    double2 v = make_double2(0.0, 0.0);
    if (l < L && m <= l && covered[l]) v = fo[(long long)l * L + m];
    tile[r][tx] = v;
  }
  __syncthreads();
  for (int r = ty; r < 32; r += 8) {
    const int l = l0 + tx, m = m0 + r;  // write flm[l + L m]: l fastest
    if (l < L && m < L) {
      double2 v = tile[tx][r];
      if (l < bl && m < bl) {
        const double2 s = scoeff[l + (long long)bl * m];
        v.x += Phi2[l] * s.x;
        v.y += Phi2[l] * s.y;
      }
      flm[l + (long long)L * m] = v;
    }
  }
}

__global__ void k_scoeff(int L, int bl, const double2 *__restrict__ flm, double2 *__restrict__ sc) {
  const int id = blockIdx.x * blockDim.x + threadIdx.x;
  if (id >= bl * bl) return;
  const int l = id % bl, m = id / bl;
  sc[id] = flm[l + (long long)L * m];
}

__global__ void k_fill(double *__restrict__ p, long long n) {
  const long long id = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (id < n) p[id] = 0.0;
}

// ---------------------------------------------------------------------------
// Analysis beta stage.  For (m, g) and r in {0,1}:
//   Tb(m, 2b'+r, g) = sum_{k=-(hi-1)}^{hi-1} y(k) w^{k(1+2r)} e^{2 pi i k b'/(2hi)}
// with y(k) = Tg(m,|k|,g) (k >= 0), sigma_m Tg(m,-k,g) (k < 0), w = e^{2 pi i/(8hi)},
// sigma_m = +1 when m+N-1 is even (cosine case), -1 otherwise (sine case).
// This equals sum_{m'} Tg(m,m',g) eta(m,m',b), eta as in s2dw_core_mod.f90:725-731.
// ---------------------------------------------------------------------------
struct BetaAnaArgs {
  FftSpec f;
  int hi, N, logT;
  const double2 *Tg;
  double2 *Tb;        // [g][m][b], or [g][b][m] in the reference-rounding form: strides tbb, tbm
  int tbb, tbm;
  const double2 *tw8;
};

__global__ __launch_bounds__(256) void k_beta_ana(const BetaAnaArgs a) {
  extern __shared__ double2 lds[];
  const int T = 1 << a.logT, hi = a.hi, n = 2 * hi;
  double2 *A = lds, *Bf = lds + ((long long)a.f.M << a.logT);
  const int m0 = blockIdx.x * T, g = blockIdx.y, r = blockIdx.z;
  const int e8 = 8 * hi;
  for (int idx = threadIdx.x; idx < (n << a.logT); idx += blockDim.x) {
    const int t = idx & (T - 1), k = idx >> a.logT, m = m0 + t;
    double2 z = make_double2(0.0, 0.0);
    if (m < hi && k != hi) {
      const int kk = k < hi ? k : k - n;
      const int ak = kk < 0 ? -kk : kk;
      double2 x = a.Tg[((long long)g * hi + ak) * hi + m];
      if (kk < 0 && ((m + a.N - 1) & 1)) x = make_double2(-x.x, -x.y);
      int e = (kk * (1 + 2 * r)) % e8;
      if (e < 0) e += e8;
      z = cmul(x, a.tw8[e]);
    }
    A[idx] = z;
  }
  __syncthreads();
  const double2 *out = fft_exec<+1>(a.f, A, Bf, a.logT);
  for (int idx = threadIdx.x; idx < (hi << a.logT); idx += blockDim.x) {
    const int t = idx & (T - 1), bp = idx >> a.logT, m = m0 + t;
    if (m < hi) a.Tb[(long long)g * n * hi + (long long)(2 * bp + r) * a.tbb + (long long)m * a.tbm] = out[idx];
  }
}

// ---------------------------------------------------------------------------
// Analysis alpha stage: FFTW-style c2r of length n = 2hi-1 (unnormalised,
// e^{+}, Im X_0 ignored) of rows b and b+1 packed as one complex transform.
// ---------------------------------------------------------------------------
struct AlphaArgs {
  FftSpec f;
  int hi, logT;
  const double2 *Tb;  // analysis input, [g][m][b] (BetaAnaArgs): strides tbb, tbm
  int tbb, tbm;
  double *W;          // per-scale wav [g][b][a]
  double2 *V;         // synthesis output
  double scale;       // synthesis scaling
  const double2 *eg;  // synthesis: [ni][g] e^{-i n_ni pi g / N}
  const double *wq;   // synthesis: 2hi quadrature weights
  int N, nn, z0;      // synthesis: gamma samples, n-indices, the index of n = 0 (-1: none)
  long long woff;     // offset of W in the packed wavelet coefficients (grouped launches)
  double *mp;         // analysis reducing to moments: this scale's records (8 doubles per workgroup)
  long long moff;     // offset of mp in the plan's record buffer (grouped launches)
};

__global__ __launch_bounds__(256) void k_alpha_c2r(const AlphaArgs a) {
  extern __shared__ double2 lds[];
  const int T = 1 << a.logT, hi = a.hi, n = 2 * hi - 1;
  double2 *A = lds, *Bf = lds + ((long long)a.f.M << a.logT);
  const int g = blockIdx.y;
  for (int t = 0; t < T; ++t) {
    const int pidx = blockIdx.x * T + t;
    const double2 *rb = a.Tb + (long long)g * 2 * hi * hi + (long long)(2 * pidx) * a.tbb;
    const double2 *rb1 = rb + a.tbb;
    const long long sm = a.tbm;
    for (int k = threadIdx.x; k < n; k += blockDim.x) {
      double2 z = make_double2(0.0, 0.0);
      if (pidx < hi) {
        if (k == 0) {
          z = make_double2(rb[0].x, rb1[0].x);
        } else if (k < hi) {
          const double2 p = rb[k * sm], q = rb1[k * sm];
          z = make_double2(p.x - q.y, p.y + q.x);
        } else {
          const double2 p = rb[(n - k) * sm], q = rb1[(n - k) * sm];
          z = make_double2(p.x + q.y, -p.y + q.x);
        }
      }
      A[(k << a.logT) + t] = z;
    }
  }
  __syncthreads();
  const double2 *out = fft_exec<+1>(a.f, A, Bf, a.logT);
  for (int t = 0; t < T; ++t) {
    const int pidx = blockIdx.x * T + t;
    if (pidx >= hi) break;
    double *w0 = a.W + ((long long)g * 2 * hi + 2 * pidx) * n;
    double *w1 = w0 + n;
    for (int k = threadIdx.x; k < n; k += blockDim.x) {
      const double2 z = out[(k << a.logT) + t];
      w0[k] = z.x;
      w1[k] = z.y;
    }
  }
}

// Synthesis alpha stage: FFTW-style r2c of rows b, b+1 (packed), times scale.
__global__ __launch_bounds__(256) void k_alpha_r2c(const AlphaArgs a) {
  extern __shared__ double2 lds[];
  const int T = 1 << a.logT, hi = a.hi, n = 2 * hi - 1;
  double2 *A = lds, *Bf = lds + ((long long)a.f.M << a.logT);
  const int g = blockIdx.y;
  for (int t = 0; t < T; ++t) {
    const int pidx = blockIdx.x * T + t;
    const double *w0 = a.W + ((long long)g * 2 * hi + 2 * pidx) * n;
    const double *w1 = w0 + n;
    for (int k = threadIdx.x; k < n; k += blockDim.x)
      A[(k << a.logT) + t] = pidx < hi ? make_double2(w0[k], w1[k]) : make_double2(0.0, 0.0);
  }
  __syncthreads();
  const double2 *out = fft_exec<-1>(a.f, A, Bf, a.logT);
  const double h = 0.5 * a.scale;
  for (int t = 0; t < T; ++t) {
    const int pidx = blockIdx.x * T + t;
    if (pidx >= hi) break;
    double2 *v0 = a.V + ((long long)g * 2 * hi + 2 * pidx) * hi;
    double2 *v1 = v0 + hi;
    for (int k = threadIdx.x; k < hi; k += blockDim.x) {
      const double2 zp = out[(k << a.logT) + t];
      const double2 zm = out[((k ? n - k : 0) << a.logT) + t];  // conj taken below
      // V_b = (Z_k + conj Z_{n-k})/2,  V_{b+1} = (Z_k - conj Z_{n-k})/(2i)
      v0[k] = make_double2(h * (zp.x + zm.x), h * (zp.y - zm.y));
      v1[k] = make_double2(h * (zp.y + zm.y), -h * (zp.x - zm.x));
    }
  }
}

// ---------------------------------------------------------------------------
// Synthesis beta stage.  For (m, n):
//   u(b) = w_b sum_g V(m,b,g) e^{-i n pi g/N},   b in [0, 2hi)
//   V2(m,m') = sum_b u(b) e^{-i m' beta_b} = e^{-i pi m'/(4hi)} sum_b u(b) e^{-2 pi i m' b/(4hi)},
// a zero-padded length-4hi DFT.  Split by r = m' mod 2 (m' = 2q + r mod 4hi):
//   V2 = e^{-i pi m'/(4hi)} FFT_{2hi}(u(b) e^{-2 pi i r b/(4hi)})(q).
// m' and -m' have the same parity, so each r-half also does the fold
//   V3(m,m') = V2(m,m') + (-1)^{m+n} V2(m,-m')  (m' >= 1)
// and writes Vt_j(m,m',c) = u_c i^{m-n} V3(m,m') for m' = r mod 2.
// ---------------------------------------------------------------------------
struct BetaSynArgs {
  FftSpec f;
  int hi, N, logT, NCtot;
  const double2 *V;
  const double *wq;     // 2hi weights
  const double2 *tw8;
  const double2 *eg;    // [nidx][g] e^{-i n pi g / N}
  int nval[kMaxCol];    // n of each n-index
  int ncol[kMaxCol];    // number of columns of each n-index
  int col0[kMaxCol][2]; // column ids
  int cpart[kMaxCol][2];
  double2 *Vt;          // [c][m'][m]
};

__global__ __launch_bounds__(256) void k_beta_syn(const BetaSynArgs a) {
  extern __shared__ double2 lds[];
  const int T = 1 << a.logT, hi = a.hi, n2 = 2 * hi, e8 = 8 * hi;
  double2 *A = lds, *Bf = lds + ((long long)a.f.M << a.logT);
  const int m0 = blockIdx.x * T, ni = blockIdx.y, r = blockIdx.z;
  const int nv = a.nval[ni];
  for (int idx = threadIdx.x; idx < (n2 << a.logT); idx += blockDim.x) {
    const int t = idx & (T - 1), b = idx >> a.logT, m = m0 + t;
    double2 u = make_double2(0.0, 0.0);
    if (m < hi) {
      for (int g = 0; g < a.N; ++g) {
        const double2 v = a.V[((long long)g * n2 + b) * hi + m];
        const double2 e = a.eg[ni * a.N + g];
        u.x += v.x * e.x - v.y * e.y;
        u.y += v.x * e.y + v.y * e.x;
      }
      const double w = a.wq[b];
      u.x *= w;
      u.y *= w;
      if (r) u = cmulw<-1>(u, a.tw8[(2 * b) % e8]);  // e^{-2 pi i b/(4hi)}
    }
    A[idx] = u;
  }
  __syncthreads();
  const double2 *out = fft_exec<-1>(a.f, A, Bf, a.logT);
  const int nq = (hi - r + 1) / 2;  // number of m' in [0,hi) with m' = r mod 2
  for (int idx = threadIdx.x; idx < (nq << a.logT); idx += blockDim.x) {
    const int t = idx & (T - 1), q = idx >> a.logT, m = m0 + t;
    const int mp = 2 * q + r;
    if (m >= hi) continue;
    const double2 w = a.tw8[mp];
    double2 v3 = cmulw<-1>(out[(q << a.logT) + t], w);  // e^{-i pi m'/(4hi)} X(q)
    if (mp >= 1) {
      const int qm = (4 * hi - mp) >> 1;                  // -m' mod 4hi = 2 qm + r
      double2 v2m = cmul(out[(qm << a.logT) + t], w);     // e^{+i pi m'/(4hi)} X(qm)
      if ((m + nv) & 1) v2m = make_double2(-v2m.x, -v2m.y);
      v3 = cadd(v3, v2m);
    }
    // i^{m-n}
    const int rot = ((m - nv) % 4 + 4) % 4;
    double2 z;
    if (rot == 0) z = v3;
    else if (rot == 1) z = make_double2(-v3.y, v3.x);
    else if (rot == 2) z = make_double2(-v3.x, -v3.y);
    else z = make_double2(v3.y, -v3.x);
    for (int k = 0; k < a.ncol[ni]; ++k) {
      const int c = a.col0[ni][k];
      const double2 o = a.cpart[ni][k] ? make_double2(-z.y, z.x) : z;  // u_p: 1 or i
      a.Vt[((long long)c * hi + mp) * hi + m] = o;
    }
  }
}

// ---------------------------------------------------------------------------
// Wave-engine versions of the four transform stages, used when the work length
// M is a power of two with M <= 64*E.  Each wave owns a 64*E-element LDS
// region holding Tw = 64E/M sequences; loads and stores are cooperative across
// the workgroup so that rows are read and written in wide contiguous runs.
// ---------------------------------------------------------------------------
__device__ __forceinline__ int wave_id() { return __builtin_amdgcn_readfirstlane(threadIdx.x >> 6); }

// beta (analysis): workgroup = TMW = WPB*Tw consecutive m, one g, one r.
template <int E>
__global__ __launch_bounds__(512 / (E / 16)) void k_beta_ana_w(const BetaAnaArgs a) {
  extern __shared__ double2 lds[];
  const int hi = a.hi, n = 2 * hi, e8 = 8 * hi;
  const int logTw = a.logT;  // log2 of sequences per wave
  const int Tw = 1 << logTw, WPB = blockDim.x >> 6, TMW = WPB * Tw;
  const int m0 = blockIdx.x * TMW, g = blockIdx.y, r = blockIdx.z;
  for (int idx = threadIdx.x; idx < n * TMW; idx += blockDim.x) {
    const int t = idx % TMW, k = idx / TMW, m = m0 + t;
    double2 z = make_double2(0.0, 0.0);
    if (m < hi && k != hi) {
      const int kk = k < hi ? k : k - n;
      const int ak = kk < 0 ? -kk : kk;
      double2 x = a.Tg[((long long)g * hi + ak) * hi + m];
      if (kk < 0 && ((m + a.N - 1) & 1)) x = make_double2(-x.x, -x.y);
      int e = (kk * (1 + 2 * r)) % e8;
      if (e < 0) e += e8;
      z = cmul(x, a.tw8[e]);
    }
    lds[(t >> logTw) * (64 * E) + (k << logTw) + (t & (Tw - 1))] = z;
  }
  __syncthreads();
  wave_fft_exec<E, +1>(a.f, lds + wave_id() * (64 * E), logTw);
  __syncthreads();
  for (int idx = threadIdx.x; idx < hi * TMW; idx += blockDim.x) {
    const int t = idx % TMW, bp = idx / TMW, m = m0 + t;
    if (m < hi)
      a.Tb[(long long)g * n * hi + (long long)(2 * bp + r) * a.tbb + (long long)m * a.tbm] = lds[(t >> logTw) * (64 * E) + (bp << logTw) + (t & (Tw - 1))];
  }
}

// alpha c2r (analysis): each wave transforms Tw row pairs.
template <int E>
__global__ __launch_bounds__(512 / (E / 16)) void k_alpha_c2r_w(const AlphaArgs a) {
  extern __shared__ double2 lds[];
  const int hi = a.hi, n = 2 * hi - 1;
  const int logTw = a.logT, Tw = 1 << logTw, WPB = blockDim.x >> 6;
  const int w = wave_id(), lane = threadIdx.x & 63;
  double2 *buf = lds + w * (64 * E);
  const int g = blockIdx.y;
  const int p0 = (blockIdx.x * WPB + w) * Tw;
  for (int t = 0; t < Tw; ++t) {
    const int pidx = p0 + t;
    const double2 *rb = a.Tb + (long long)g * 2 * hi * hi + (long long)(2 * pidx) * a.tbb;
    const double2 *rb1 = rb + a.tbb;
    const long long sm = a.tbm;
    for (int k = lane; k < n; k += 64) {
      double2 z = make_double2(0.0, 0.0);
      if (pidx < hi) {
        if (k == 0) {
          z = make_double2(rb[0].x, rb1[0].x);
        } else if (k < hi) {
          const double2 p = rb[k * sm], q = rb1[k * sm];
          z = make_double2(p.x - q.y, p.y + q.x);
        } else {
          const double2 p = rb[(n - k) * sm], q = rb1[(n - k) * sm];
          z = make_double2(p.x + q.y, -p.y + q.x);
        }
      }
      buf[(k << logTw) + t] = z;
    }
  }
  __builtin_amdgcn_wave_barrier();
  wave_fft_exec<E, +1>(a.f, buf, logTw);
  for (int t = 0; t < Tw; ++t) {
    const int pidx = p0 + t;
    if (pidx >= hi) break;
    double *w0 = a.W + ((long long)g * 2 * hi + 2 * pidx) * n;
    double *w1 = w0 + n;
    for (int k = lane; k < n; k += 64) {
      const double2 z = buf[(k << logTw) + t];
      w0[k] = z.x;
      w1[k] = z.y;
    }
  }
}

// alpha r2c (synthesis): each wave transforms Tw row pairs.
template <int E>
__global__ __launch_bounds__(512 / (E / 16)) void k_alpha_r2c_w(const AlphaArgs a) {
  extern __shared__ double2 lds[];
  const int hi = a.hi, n = 2 * hi - 1;
  const int logTw = a.logT, Tw = 1 << logTw, WPB = blockDim.x >> 6;
  const int w = wave_id(), lane = threadIdx.x & 63;
  double2 *buf = lds + w * (64 * E);
  const int g = blockIdx.y;
  const int p0 = (blockIdx.x * WPB + w) * Tw;
  for (int t = 0; t < Tw; ++t) {
    const int pidx = p0 + t;
    const double *w0 = a.W + ((long long)g * 2 * hi + 2 * pidx) * n;
    const double *w1 = w0 + n;
    for (int k = lane; k < n; k += 64) buf[(k << logTw) + t] = pidx < hi ? make_double2(w0[k], w1[k]) : make_double2(0.0, 0.0);
  }
  __builtin_amdgcn_wave_barrier();
  wave_fft_exec<E, -1>(a.f, buf, logTw);
  const double h = 0.5 * a.scale;
  for (int t = 0; t < Tw; ++t) {
    const int pidx = p0 + t;
    if (pidx >= hi) break;
    double2 *v0 = a.V + ((long long)g * 2 * hi + 2 * pidx) * hi;
    double2 *v1 = v0 + hi;
    for (int k = lane; k < hi; k += 64) {
      const double2 zp = buf[(k << logTw) + t];
      const double2 zm = buf[((k ? n - k : 0) << logTw) + t];
      v0[k] = make_double2(h * (zp.x + zm.x), h * (zp.y - zm.y));
      v1[k] = make_double2(h * (zp.y + zm.y), -h * (zp.x - zm.x));
    }
  }
}

// beta (synthesis): workgroup = TMW consecutive m, one n-index, one r.
template <int E>
__global__ __launch_bounds__(512 / (E / 16)) void k_beta_syn_w(const BetaSynArgs a) {
  extern __shared__ double2 lds[];
  const int hi = a.hi, n2 = 2 * hi, e8 = 8 * hi;
  const int logTw = a.logT, Tw = 1 << logTw, WPB = blockDim.x >> 6, TMW = WPB * Tw;
  const int m0 = blockIdx.x * TMW, ni = blockIdx.y, r = blockIdx.z;
  const int nv = a.nval[ni];
  for (int idx = threadIdx.x; idx < n2 * TMW; idx += blockDim.x) {
    const int t = idx % TMW, b = idx / TMW, m = m0 + t;
    double2 u = make_double2(0.0, 0.0);
    if (m < hi) {
      for (int g = 0; g < a.N; ++g) {
        const double2 v = a.V[((long long)g * n2 + b) * hi + m];
        const double2 e = a.eg[ni * a.N + g];
        u.x += v.x * e.x - v.y * e.y;
        u.y += v.x * e.y + v.y * e.x;
      }
      const double wq = a.wq[b];
      u.x *= wq;
      u.y *= wq;
      if (r) u = cmulw<-1>(u, a.tw8[(2 * b) % e8]);
    }
    lds[(t >> logTw) * (64 * E) + (b << logTw) + (t & (Tw - 1))] = u;
  }
  __syncthreads();
  wave_fft_exec<E, -1>(a.f, lds + wave_id() * (64 * E), logTw);
  __syncthreads();
  const int nq = (hi - r + 1) / 2;
  for (int idx = threadIdx.x; idx < nq * TMW; idx += blockDim.x) {
    const int t = idx % TMW, q = idx / TMW, m = m0 + t;
    if (m >= hi) continue;
    const double2 *buf = lds + (t >> logTw) * (64 * E);
    const int tt = t & (Tw - 1);
    const int mp = 2 * q + r;
    const double2 w = a.tw8[mp];
    double2 v3 = cmulw<-1>(buf[(q << logTw) + tt], w);
    if (mp >= 1) {
      const int qm = (4 * hi - mp) >> 1;
      double2 v2m = cmul(buf[(qm << logTw) + tt], w);
      if ((m + nv) & 1) v2m = make_double2(-v2m.x, -v2m.y);
      v3 = cadd(v3, v2m);
    }
    const int rot = ((m - nv) % 4 + 4) % 4;
    double2 z;
    if (rot == 0) z = v3;
    else if (rot == 1) z = make_double2(-v3.y, v3.x);
    else if (rot == 2) z = make_double2(-v3.x, -v3.y);
    else z = make_double2(v3.y, -v3.x);
    for (int kc = 0; kc < a.ncol[ni]; ++kc) {
      const int c = a.col0[ni][kc];
      const double2 o = a.cpart[ni][kc] ? make_double2(-z.y, z.x) : z;
      a.Vt[((long long)c * hi + mp) * hi + m] = o;
    }
  }
}

// ---------------------------------------------------------------------------
// Transform stages on the workgroup FFT engine: kTN threads x kTE slots per
// workgroup, power-of-two work length M <= kTS (direct, or Bluestein for a
// length n whose work length is M).  Every global load of a load phase is
// issued before the first LDS store, so one workgroup keeps kTE loads per
// thread in flight.  Workgroups are numbered along a 1-D grid remapped per
// XCD (xcd_tile) so that neighbouring column tiles share an L2.
// ---------------------------------------------------------------------------
constexpr int kTE = 8, kTN = 256, kTS = kTE * kTN, kLogTS = 11;
__host__ __device__ constexpr int clog2(int x) { return x <= 1 ? 0 : 1 + clog2(x / 2); }
static_assert(kTS == 1 << kLogTS, "slots per workgroup");

__device__ __forceinline__ int ilog2(int x) { return 31 - __clz(x); }

// Chirp premultiplier of element k (Bluestein) or 1.
template <int DIR>
__device__ __forceinline__ double2 chirp_in(const FftSpec &f, double2 x, int k) {
  return f.bluestein ? cmulw<DIR>(x, f.chirp[k]) : x;
}

// beta (analysis): sequence t = 2*mc + r holds column m = m0 + mc and output
// parity r; the workgroup reads each Tg element once for both parities.
__device__ __forceinline__ void beta_ana_body(const BetaAnaArgs &a, int nmt, double2 *lds, int bid, int nb) {
  const FftSpec &f = a.f;
  const bool bluestein = f.bluestein != 0;
  const int hi = a.hi, n = 2 * hi, e8 = 8 * hi, M = f.M;
  const int logTw = a.logT, Tw = 1 << logTw, logMC = logTw - 1, MC = Tw >> 1;
  const int tile = xcd_tile(bid, nb);
  const int g = tile / nmt, m0 = (tile - g * nmt) * MC;
  {
    double2 x[kTE / 2], w0[kTE / 2], w1[kTE / 2], c[kTE / 2];
#pragma unroll
    for (int e = 0; e < kTE / 2; ++e) {
      const int s = threadIdx.x + kTN * e;
      const int kq = s >> logMC, mc = s & (MC - 1), m = m0 + mc;
      x[e] = make_double2(0.0, 0.0);
      w0[e] = w1[e] = c[e] = make_double2(1.0, 0.0);
      if (m < hi && kq < n && kq != hi) {
        const int kk = kq < hi ? kq : kq - n;
        const int ak = kk < 0 ? -kk : kk;
        x[e] = a.Tg[((long long)g * hi + ak) * hi + m];
        if (kk < 0 && ((m + a.N - 1) & 1)) x[e] = make_double2(-x[e].x, -x[e].y);
        // kk mod 8hi and 3 kk mod 8hi: |kk| < hi, so one conditional add each
        const int e0 = kk < 0 ? kk + e8 : kk, e1 = kk < 0 ? 3 * kk + e8 : 3 * kk;
        w0[e] = a.tw8[e0];
        w1[e] = a.tw8[e1];
        if (bluestein) c[e] = f.chirp[kq];
      }
    }
#pragma unroll
    for (int e = 0; e < kTE / 2; ++e) {
      const int s = threadIdx.x + kTN * e;
      const int kq = s >> logMC, mc = s & (MC - 1);
      double2 z0 = cmul(x[e], w0[e]), z1 = cmul(x[e], w1[e]);
      if (bluestein) {
        z0 = cmulw<+1>(z0, c[e]);
        z1 = cmulw<+1>(z1, c[e]);
      }
      lds[lpad((kq << logTw) + 2 * mc)] = z0;
      lds[lpad((kq << logTw) + 2 * mc + 1)] = z1;
    }
  }
  lds_barrier();
  team_fft_core<kTE, kTN, +1>(f, lds, M, logTw, bluestein);
  // outputs bp < hi of sequence (mc, r) -> Tb[g][2bp + r][m]
#pragma unroll
  for (int e = 0; e < kTE / 2; ++e) {
    const int s = threadIdx.x + kTN * e;  // < M*Tw/2
    const int mc = s & (MC - 1), r = (s >> logMC) & 1, bp = s >> logTw;
    const int m = m0 + mc;
    if (m < hi && bp < hi) {
      double2 y = lds[lpad((bp << logTw) + 2 * mc + r)];
      if (bluestein) y = cmulw<+1>(y, f.chirp[bp]);
      a.Tb[(long long)g * n * hi + (2 * bp + r) * a.tbb + m * a.tbm] = y;
    }
  }
}

// Rows p = rb, q = rb + sb of a packed pair at the lane's own k: lanes 2i and
// 2i + 1 (both active) load p and q of the even lane's k = ke and then of the
// odd lane's k = ko, side by side in memory where sb = 1, and swap halves.
__device__ __forceinline__ double swap1(double v) {  // the value of lane ^ 1
  int2 x = __builtin_bit_cast(int2, v);
  x.x = __builtin_amdgcn_update_dpp(0, x.x, 0xB1, 0xF, 0xF, true);
  x.y = __builtin_amdgcn_update_dpp(0, x.y, 0xB1, 0xF, 0xF, true);
  return __builtin_bit_cast(double, x);
}
__device__ __forceinline__ void load_pair(const double2 *rb, int sb, int sm, int ke, int ko, double2 &p, double2 &q) {
  const bool odd = threadIdx.x & 1;
  const double2 *c = rb + (odd ? sb : 0);
  const double2 r1 = c[ke * sm], r2 = c[ko * sm];  // < 2 hi^2 < 2^31
  const double2 snd = odd ? r1 : r2;
  const double2 rcv = make_double2(swap1(snd.x), swap1(snd.y));
  p = odd ? rcv : r1;
  q = odd ? r2 : rcv;
}

// alpha c2r (analysis): sequence t = row pair pidx = p0 + t of one g.
// MOM: instead of storing W, the workgroup reduces its values to one moments
// record (s2dw_moments.h) at a.mp + 8 tile.
template <int LOGM, int BL, bool MOM = false, int NT = kTN>
__device__ __forceinline__ void alpha_c2r_body(const AlphaArgs &a, int npt, double2 *lds, int bid, int nb) {
  constexpr int LOGTS = clog2(NT * kTE);  // log2 of the workgroup's slots
  const FftSpec &f = a.f;
  const bool bluestein = BL >= 0 ? BL != 0 : f.bluestein != 0;
  const int hi = a.hi, n = 2 * hi - 1, logM = LOGM > 0 ? LOGM : ilog2(f.M), M = 1 << logM;
  const int logTw = LOGM > 0 ? LOGTS - LOGM : a.logT;
  const int tile = xcd_tile(bid, nb);
  const int g = tile / npt, p0 = (tile - g * npt) << logTw;
  // Bluestein with a radix-4 first stage (log2 M = 2 mod 3): that stage is
  // done here, in registers, from the loaded coefficients.  Butterfly jj of
  // sequence t takes slots jj, jj + M/4, jj + M/2, jj + 3M/4; slots >= n are
  // zero and n <= M/2, so only the first two can be non-zero.  Slot k < hi is
  // p_k + i q_k, slot hi <= k < n is conj(p_{n-k}) + i conj(q_{n-k}) (rows p,
  // q of the packed pair), each times chirp_k.
  if constexpr (LOGM > 0 && LOGM % 3 == 2 && BL == 1) {
    constexpr int Q = 1 << (LOGM - 2), NB = kTE / 4;
    double2 pk[NB][2], qk[NB][2], ck[NB][2];
    int kv[NB][2];
#pragma unroll
    for (int q = 0; q < NB; ++q) {
      // rows of one k are adjacent in memory: sequences run along the lanes
      const int b = threadIdx.x + NT * q, t = b & ((1 << logTw) - 1), jj = b >> logTw, pidx = p0 + t;
      const double2 *rb = a.Tb + (long long)g * 2 * hi * hi + 2 * pidx * a.tbb;
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const int k = jj + h * Q;
        auto at = [=](int i) { return i < hi ? i : i < n ? n - i : 0; };
        kv[q][h] = pidx < hi && k < n ? k : -1;
        pk[q][h] = qk[q][h] = make_double2(0.0, 0.0);
        ck[q][h] = make_double2(0.0, 0.0);
        if constexpr (LOGM == LOGTS) {
          load_pair(rb, a.tbb, a.tbm, at(k & ~1), at(k | 1), pk[q][h], qk[q][h]);
          ck[q][h] = f.chirp[k];
        } else if (kv[q][h] >= 0) {
          pk[q][h] = rb[at(k) * a.tbm];
          qk[q][h] = rb[at(k) * a.tbm + a.tbb];
          ck[q][h] = f.chirp[k];
        }
      }
    }
#pragma unroll
    for (int q = 0; q < NB; ++q) {
      const int b = threadIdx.x + NT * q, t = b & ((1 << logTw) - 1), jj = b >> logTw;
      double2 v[4];
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const int k = kv[q][h];
        const double2 p = pk[q][h], qq = qk[q][h];
        double2 z = k == 0 ? make_double2(p.x, qq.x)
                  : k < hi  ? make_double2(p.x - qq.y, p.y + qq.x)
                            : make_double2(p.x + qq.y, -p.y + qq.x);
        v[h] = k >= 0 ? cmulw<+1>(z, ck[q][h]) : make_double2(0.0, 0.0);
      }
      v[2] = v[3] = make_double2(0.0, 0.0);
      dft_pow2<4, -1>(v);
#pragma unroll
      for (int r = 0; r < 4; ++r) lds[lpad(((4 * jj + r) << logTw) + t)] = v[r];
    }
    lds_barrier();
    if constexpr (LOGM != LOGTS) {
      team_fft_core<kTE, NT, +1, true>(f, lds, M, logTw, true);
    } else {
    // one sequence per team: the backward transform's last stage hands
    // outputs k = jj + r M/4 < M/2 (n <= M/2) to the registers, lanes along
    // k; no slot write, barrier or re-read
    double2 yl[NB][2];
    team_bluestein_x<kTE, NT, +1, true, true>(f, lds, M, logTw, nullptr, yl);
    const int Tw = 1 << logTw;
    if constexpr (MOM) {
      double v[4 * NB], wt[4 * NB];
#pragma unroll
      for (int q = 0; q < NB; ++q) {
        const int b = threadIdx.x + NT * q, t = b & (Tw - 1), jj = b >> logTw, pidx = p0 + t;
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const int k = jj + h * Q;  // < M/2 < M: the chirp read stays in its table
          const bool ok = pidx < hi && k < n;
          const double2 z = cmulw<+1>(yl[q][h], f.chirp[k]);
          v[4 * q + 2 * h] = z.x;
          v[4 * q + 2 * h + 1] = z.y;
          wt[4 * q + 2 * h] = wt[4 * q + 2 * h + 1] = ok ? 1.0 : 0.0;
        }
      }
      mom_record<4 * NB, NT>(v, wt, 0.0, a.mp + 8LL * tile);
      return;
    }
#pragma unroll
    for (int q = 0; q < NB; ++q) {
      const int b = threadIdx.x + NT * q, t = b & (Tw - 1), jj = b >> logTw, pidx = p0 + t;
      double *w0 = a.W + ((long long)g * 2 * hi + 2 * pidx) * n;
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const int k = jj + h * Q;
        if (pidx < hi && k < n) {
          const double2 z = cmulw<+1>(yl[q][h], f.chirp[k]);
          w0[k] = z.x;
          w0[n + k] = z.y;
        }
      }
    }
    return;
    }
  } else {
  // slots k >= n are zero
#pragma unroll
  for (int e = 0; e < kTE; ++e) {
    const int s = threadIdx.x + NT * e;
    if ((s >> logTw) >= n) lds[lpad(s)] = make_double2(0.0, 0.0);
  }
  // each Tb element (k < hi) is read once and gives slot k and slot n - k:
  // z_k = p + i q, z_{n-k} = conj(p) + i conj(q) for the packed rows p, q;
  // two rounds of kTE/4 elements per thread keep the loads in flight within
  // the register budget of three waves per SIMD
#pragma unroll
  for (int half = 0; half < 2; ++half) {
    constexpr int HE = kTE / 4;
    double2 pv[HE], qv[HE], c0[HE], c1[HE];
#pragma unroll
    for (int e = 0; e < HE; ++e) {
      // M/2 >= hi positions per sequence, sequences along the lanes
      const int u = threadIdx.x + NT * (e + half * HE);
      const int t = u & ((1 << logTw) - 1), kk = u >> logTw, pidx = p0 + t;
      const double2 *rb = a.Tb + (long long)g * 2 * hi * hi + 2 * pidx * a.tbb;
      pv[e] = qv[e] = make_double2(0.0, 0.0);
      c0[e] = c1[e] = make_double2(1.0, 0.0);
      if constexpr (LOGM == LOGTS)
        load_pair(rb, a.tbb, a.tbm, (kk & ~1) < hi ? kk & ~1 : 0, (kk | 1) < hi ? kk | 1 : 0, pv[e], qv[e]);
      if (pidx < hi && kk < hi) {
        if constexpr (LOGM != LOGTS) {
          pv[e] = rb[kk * a.tbm];
          qv[e] = rb[kk * a.tbm + a.tbb];
        }
        if (bluestein) {
          c0[e] = f.chirp[kk];
          c1[e] = f.chirp[kk ? n - kk : 0];
        }
      }
    }
#pragma unroll
    for (int e = 0; e < HE; ++e) {
      const int u = threadIdx.x + NT * (e + half * HE);
      const int t = u & ((1 << logTw) - 1), kk = u >> logTw, pidx = p0 + t;
      if (kk >= hi) continue;
      const double2 p = pv[e], q = qv[e];
      double2 z = kk == 0 ? make_double2(p.x, q.x) : make_double2(p.x - q.y, p.y + q.x);
      if (pidx >= hi) z = make_double2(0.0, 0.0);
      if (bluestein) z = cmulw<+1>(z, c0[e]);
      lds[lpad((kk << logTw) + t)] = z;
      if (kk) {
        double2 zm = pidx < hi ? make_double2(p.x + q.y, -p.y + q.x) : make_double2(0.0, 0.0);
        if (bluestein) zm = cmulw<+1>(zm, c1[e]);
        lds[lpad(((n - kk) << logTw) + t)] = zm;
      }
    }
  }
  lds_barrier();
  team_fft_core<kTE, NT, +1>(f, lds, M, logTw, bluestein);
  }
  if constexpr (MOM) {
    double v[2 * kTE], wt[2 * kTE];
#pragma unroll
    for (int e = 0; e < kTE; ++e) {
      const int s = threadIdx.x + NT * e;
      const int t = s >> logM, kk = s & (M - 1), pidx = p0 + t;
      const bool ok = pidx < hi && kk < n;
      double2 z = lds[lpad((kk << logTw) + t)];
      if (bluestein) z = cmulw<+1>(z, f.chirp[kk]);
      v[2 * e] = z.x;
      v[2 * e + 1] = z.y;
      wt[2 * e] = wt[2 * e + 1] = ok ? 1.0 : 0.0;
    }
    mom_record<2 * kTE, NT>(v, wt, 0.0, a.mp + 8LL * tile);
    return;
  }
#pragma unroll
  for (int e = 0; e < kTE; ++e) {
    const int s = threadIdx.x + NT * e;
    const int t = s >> logM, kk = s & (M - 1), pidx = p0 + t;
    if (pidx < hi && kk < n) {
      double2 z = lds[lpad((kk << logTw) + t)];
      if (bluestein) z = cmulw<+1>(z, f.chirp[kk]);
      double *w0 = a.W + ((long long)g * 2 * hi + 2 * pidx) * n;
      w0[kk] = z.x;
      w0[n + kk] = z.y;
    }
  }
}

template <int LOGM, int BL>
__device__ __forceinline__ void alpha_c2r_body_m(const AlphaArgs &a, int npt, double2 *lds, int bid, int nb) {
  alpha_c2r_body<LOGM, BL, true>(a, npt, lds, bid, nb);
}

// alpha r2c (synthesis) of packed real rows, without the gamma-DFT: sequence
// t = row pair pidx = p0 + t of one g.
template <int LOGM, int BL, int NT = kTN>
__device__ __forceinline__ void alpha_r2c_body(const AlphaArgs &a, int npt, double2 *lds, int bid, int nb) {
  constexpr int LOGTS = clog2(NT * kTE);  // log2 of the workgroup's slots
  const FftSpec &f = a.f;
  const bool bluestein = BL >= 0 ? BL != 0 : f.bluestein != 0;
  const int hi = a.hi, n = 2 * hi - 1, logM = LOGM > 0 ? LOGM : ilog2(f.M), M = 1 << logM;
  const int logTw = LOGM > 0 ? LOGTS - LOGM : a.logT;
  const int tile = xcd_tile(bid, nb);
  const int g = tile / npt, p0 = (tile - g * npt) << logTw;
  {
    double x0[kTE], x1[kTE];
    double2 c[kTE];
#pragma unroll
    for (int e = 0; e < kTE; ++e) {
      const int s = threadIdx.x + NT * e;
      const int t = s >> logM, kk = s & (M - 1), pidx = p0 + t;
      x0[e] = x1[e] = 0.0;
      c[e] = make_double2(1.0, 0.0);
      if (pidx < hi && kk < n) {
        const double *w0 = a.W + ((long long)g * 2 * hi + 2 * pidx) * n;
        x0[e] = w0[kk];
        x1[e] = w0[n + kk];
        if (bluestein) c[e] = f.chirp[kk];
      }
    }
#pragma unroll
    for (int e = 0; e < kTE; ++e) {
      const int s = threadIdx.x + NT * e;
      const int t = s >> logM, kk = s & (M - 1);
      double2 z = make_double2(x0[e], x1[e]);
      if (bluestein) z = cmulw<-1>(z, c[e]);
      lds[lpad((kk << logTw) + t)] = z;
    }
  }
  lds_barrier();
  // Bluestein: the final chirp multiply (by conj(chirp) for this direction)
  // is folded into the last stage through a conjugated copy
  team_fft_core<kTE, NT, -1>(f, lds, M, logTw, bluestein, bluestein ? f.chirp_c : nullptr);
  const double h = 0.5 * a.scale;
  const int logH = logM - 1;  // outputs k < hi <= M/2: slots (t, k) with k < M/2
#pragma unroll
  for (int e = 0; e < kTE / 2; ++e) {
    const int s = threadIdx.x + NT * e;
    const int t = s >> logH, kk = s & ((1 << logH) - 1), pidx = p0 + t;
    if (pidx < hi && kk < hi) {
      const double2 zp = lds[lpad((kk << logTw) + t)];
      const double2 zm = lds[lpad(((kk ? n - kk : 0) << logTw) + t)];
      double2 *v0 = a.V + ((long long)g * 2 * hi + 2 * pidx) * hi;
      v0[kk] = make_double2(h * (zp.x + zm.x), h * (zp.y - zm.y));
      v0[hi + kk] = make_double2(h * (zp.y + zm.y), -h * (zp.x - zm.x));
    }
  }
}

// ---------------------------------------------------------------------------
// Synthesis alpha stage with the gamma-DFT and the quadrature weights in it.
// The gamma-DFT commutes with the alpha transform, so it is taken first, on
// the real wavelet rows while they are loaded:
//   u_n(b, a) = sum_g w(g, b, a) e^{-i n pi g/N},
//   U[ni][b][m] = scale wq[b] sum_a u_n(b, a) e^{-2 pi i m a/(2hi - 1)},  m < hi.
// For n != 0 a row u_n(b, .) is complex and is one sequence whose outputs
// m < hi are stored as they are; for n = 0 it is real and rows b, b + 1 are
// packed into one sequence, unpacked by Hermitian symmetry.  With the n of
// one parity that is N sequences per row pair, as many as the packed real rows
// took, without the N planes V(g, b, m) being written and read again by a
// gamma pass (L = 512, N = 8: 400 MB of 740 MB for the full-band pair); the
// rows of a pair are read once per n-index, the repeats from L2 (the sequences
// of a row pair are consecutive and so run on one XCD).
// Sequence id q = (row pair) nseq + s, nseq = 2 nn - (z0 >= 0).
// ---------------------------------------------------------------------------
struct SynSeq {
  int ni, b;    // n-index and row (the first row of the pair if packed)
  bool packed;  // n = 0: rows b and b + 1
};
__device__ __forceinline__ int syn_nseq(const AlphaArgs &a) { return 2 * a.nn - (a.z0 >= 0 ? 1 : 0); }
__device__ __forceinline__ SynSeq syn_seq(const AlphaArgs &a, int q) {
  const int nseq = syn_nseq(a), p = (int)((unsigned)q / (unsigned)nseq);
  int s = q - p * nseq;
  if (a.z0 >= 0) {
    if (s == 0) return {a.z0, 2 * p, true};
    --s;
  }
  int ni = s >> 1;
  if (a.z0 >= 0 && ni >= a.z0) ++ni;
  return {ni, 2 * p + (s & 1), false};
}

// G consecutive gamma samples g0.. of the E samples at offsets o: every load
// is issued before the first use.
template <int E, int G>
__device__ __forceinline__ void syn_gather_g(const double *__restrict__ W, const int (&o)[E], int gs, int g0, bool packed,
                                             int n, const double2 *__restrict__ eg, double2 (&z)[E]) {
  double w[G][E], w1[G][E];
  double2 c[G];
#pragma unroll
  for (int i = 0; i < G; ++i) {
#pragma unroll
    for (int e = 0; e < E; ++e) w[i][e] = W[o[e] + (g0 + i) * gs];
    if (packed) {
#pragma unroll
      for (int e = 0; e < E; ++e) w1[i][e] = W[o[e] + n + (g0 + i) * gs];
    } else {
      c[i] = eg[g0 + i];
    }
  }
#pragma unroll
  for (int i = 0; i < G; ++i)
#pragma unroll
    for (int e = 0; e < E; ++e) {
      if (packed) {
        z[e].x += w[i][e];
        z[e].y += w1[i][e];
      } else {
        z[e].x += w[i][e] * c[i].x;
        z[e].y += w[i][e] * c[i].y;
      }
    }
}

// z[e] = u(sequence sq, sample k[e]), 0 for k[e] >= n or !on.  Up to four
// gamma samples (4 E loads) in flight: with one at a time the loads' latency
// was a third of the stage.
template <int E>
__device__ __forceinline__ void syn_gather(const AlphaArgs &a, const SynSeq &sq, bool on, const int (&k)[E],
                                           double2 (&z)[E]) {
  const int n = 2 * a.hi - 1, gs = 2 * a.hi * n, N = a.N;  // N gs <= 32 4096 4095 < 2^31
  int o[E];
#pragma unroll
  for (int e = 0; e < E; ++e) {
    z[e] = make_double2(0.0, 0.0);
    o[e] = sq.b * n + (k[e] < n ? k[e] : 0);
  }
  const double2 *eg = a.eg + sq.ni * N;
  if (sq.packed) {
    int g = 0;
    for (; g + 2 <= N; g += 2) syn_gather_g<E, 2>(a.W, o, gs, g, true, n, eg, z);
    if (g < N) syn_gather_g<E, 1>(a.W, o, gs, g, true, n, eg, z);
  } else {
    int g = 0;
    for (; g + 4 <= N; g += 4) syn_gather_g<E, 4>(a.W, o, gs, g, false, n, eg, z);
    if (g + 2 <= N) {
      syn_gather_g<E, 2>(a.W, o, gs, g, false, n, eg, z);
      g += 2;
    }
    if (g < N) syn_gather_g<E, 1>(a.W, o, gs, g, false, n, eg, z);
  }
#pragma unroll
  for (int e = 0; e < E; ++e)
    if (!on || k[e] >= n) z[e] = make_double2(0.0, 0.0);
}

// stores output kk of a sequence (zp = Z(kk), zm = Z(n - kk), used for a
// packed sequence only)
__device__ __forceinline__ void syn_store(const AlphaArgs &a, const SynSeq &sq, int kk, double2 zp, double2 zm) {
  double2 *u = a.V + ((long long)sq.ni * 2 * a.hi + sq.b) * a.hi;
  if (sq.packed) {
    const double h0 = 0.5 * a.scale * a.wq[sq.b], h1 = 0.5 * a.scale * a.wq[sq.b + 1];
    u[kk] = make_double2(h0 * (zp.x + zm.x), h0 * (zp.y - zm.y));
    u[a.hi + kk] = make_double2(h1 * (zp.y + zm.y), -h1 * (zp.x - zm.x));
  } else {
    const double h = a.scale * a.wq[sq.b];
    u[kk] = make_double2(h * zp.x, h * zp.y);
  }
}

// A thread works on one sequence: M/8 consecutive threads per sequence.  The
// length 2hi - 1 is odd, so this is always Bluestein, n <= M/2, M >= 8.
template <int LOGM, int NT = kTN>
__device__ __forceinline__ void alpha_syn_body(const AlphaArgs &a, double2 *lds, int bid, int nb) {
  constexpr int LOGTS = clog2(NT * kTE);
  const FftSpec &f = a.f;
  const int hi = a.hi, n = 2 * hi - 1, logM = LOGM > 0 ? LOGM : ilog2(f.M), M = 1 << logM;
  const int logTw = LOGM > 0 ? LOGTS - LOGM : a.logT;
  const int Q = hi * syn_nseq(a);
  const int t0 = threadIdx.x >> (logM - 3), j0 = threadIdx.x & ((M >> 3) - 1);
  const int tile0 = xcd_tile(bid, nb) << logTw;
  const int q0 = tile0 + t0;
  const bool on = q0 < Q;
  SynSeq sq = syn_seq(a, on ? q0 : 0);
  if constexpr (LOGM >= 9) {  // whole waves per sequence
    sq.ni = uniform(sq.ni);
    sq.b = uniform(sq.b);
    sq.packed = uniform((int)sq.packed) != 0;
  }
  // samples k < M/2 only: slots k >= n are zero
  int k[kTE / 2];
  double2 z[kTE / 2];
  if constexpr (LOGM > 0 && LOGM % 3 == 2) {
    // the radix-4 first stage from the gathered rows: butterfly jj (slots
    // jj + r M/4) has non-zero inputs for r < 2 only; the thread has
    // butterflies j0 + i M/8, i < 2
#pragma unroll
    for (int i = 0; i < 4; ++i) k[i] = j0 + (M >> 3) * (i >> 1) + (M >> 2) * (i & 1);
    syn_gather<4>(a, sq, on, k, z);
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      double2 v[4];
      v[0] = cmulw<-1>(z[2 * i], f.chirp[k[2 * i]]);  // the chirp table is zero for n <= k < M
      v[1] = cmulw<-1>(z[2 * i + 1], f.chirp[k[2 * i + 1]]);
      v[2] = v[3] = make_double2(0.0, 0.0);
      dft_pow2<4, -1>(v);
#pragma unroll
      for (int r = 0; r < 4; ++r) lds[lpad(((4 * k[2 * i] + r) << logTw) + t0)] = v[r];
    }
    lds_barrier();
    team_fft_core<kTE, NT, -1, true>(f, lds, M, logTw, true, f.chirp_c);
  } else {
#pragma unroll
    for (int e = 0; e < kTE / 2; ++e) k[e] = j0 + (M >> 3) * e;
    syn_gather<kTE / 2>(a, sq, on, k, z);
#pragma unroll
    for (int e = 0; e < kTE / 2; ++e) {
      lds[lpad((k[e] << logTw) + t0)] = cmulw<-1>(z[e], f.chirp[k[e]]);
      lds[lpad(((k[e] + (M >> 1)) << logTw) + t0)] = make_double2(0.0, 0.0);
    }
    lds_barrier();
    team_fft_core<kTE, NT, -1>(f, lds, M, logTw, true, f.chirp_c);
  }
  // outputs k < hi <= M/2
  if (on)
#pragma unroll
    for (int e = 0; e < kTE / 2; ++e) {
      const int kk = j0 + (M >> 3) * e;
      if (kk < hi) {
        const double2 zp = lds[lpad((kk << logTw) + t0)];
        const double2 zm = sq.packed ? lds[lpad(((kk ? n - kk : 0) << logTw) + t0)] : zp;
        syn_store(a, sq, kk, zp, zm);
      }
    }
}

// gamma-DFT and quadrature weights (synthesis) as a pass of its own, for large
// N (gamma_first) and for the stages whose beta kernels are not on the
// workgroup engine; in place per (b, m):
// U[ni][b][m] = wq[b] sum_g V[g][b][m] e^{-i n_ni pi g/N}; ni < nn <= N <= NMAX.
template <int NMAX>
__device__ __forceinline__ void gamma_syn_body(double2 *V, int hi, int N, int nn, const double *__restrict__ wq,
                                               const double2 *__restrict__ eg, long long id) {
  const long long plane = 2LL * hi * hi;
  if (id >= plane) return;
  const int b = (int)((unsigned)id / (unsigned)hi);  // id < 2 hi^2 < 2^31: a 32-bit division
  double2 v[NMAX];
#pragma unroll
  for (int g = 0; g < NMAX; ++g) v[g] = g < N ? V[g * plane + id] : make_double2(0.0, 0.0);
  const double w = wq[b];
#pragma unroll
  for (int i = 0; i < NMAX; ++i) {
    if (i >= nn) break;
    double ur = 0.0, ui = 0.0;
#pragma unroll
    for (int g = 0; g < NMAX; ++g) {
      if (g < N) {
        const double2 e = eg[i * N + g];
        ur += v[g].x * e.x - v[g].y * e.y;
        ui += v[g].x * e.y + v[g].y * e.x;
      }
    }
    V[i * plane + id] = make_double2(w * ur, w * ui);
  }
}

// the scales of a launch: segment s owns workgroups [first[s], first[s+1])
struct GammaSeg {
  double2 *V;
  const double *wq;
  int hi;
};
struct GammaTab {
  int nseg;
  int first[kMaxSc + 1];
  GammaSeg g[kMaxSc];
};
template <int NMAX>
__global__ __launch_bounds__(256) void k_gamma_syn(const GammaTab t, int N, int nn, const double2 *__restrict__ eg) {
  int s = 0;
  for (int i = 1; i < t.nseg; ++i) s = (int)blockIdx.x >= t.first[i] ? i : s;
  const GammaSeg &g = t.g[s];
  gamma_syn_body<NMAX>(g.V, g.hi, N, nn, g.wq, eg, (long long)(blockIdx.x - t.first[s]) * blockDim.x + threadIdx.x);
}

// beta (synthesis) for one n-index: sequence t = 2*mc + r holds column
// m = m0 + mc and m' parity r; input U from k_gamma_syn.
__device__ __forceinline__ void beta_syn_body(const BetaSynArgs &a, const double2 *V, double2 *Vt, const double2 *tw8,
                                              int nmt, double2 *lds, int bid, int nb) {
  const FftSpec &f = a.f;
  const bool bluestein = f.bluestein != 0;
  const int hi = a.hi, n2 = 2 * hi, M = f.M;
  const int logTw = a.logT, Tw = 1 << logTw, logMC = logTw - 1, MC = Tw >> 1;
  const int tile = xcd_tile(bid, nb);
  const int ni = tile / nmt, m0 = (tile - ni * nmt) * MC;
  const double2 *U = V + (long long)ni * n2 * hi;
  {
    double2 x[kTE / 2], w[kTE / 2], c[kTE / 2];
#pragma unroll
    for (int e = 0; e < kTE / 2; ++e) {
      const int s = threadIdx.x + kTN * e;
      const int b = s >> logMC, mc = s & (MC - 1), m = m0 + mc;
      x[e] = make_double2(0.0, 0.0);
      w[e] = c[e] = make_double2(1.0, 0.0);
      if (m < hi && b < n2) {
        x[e] = U[(long long)b * hi + m];
        w[e] = tw8[2 * b];  // 2b < 4hi < 8hi: no reduction needed
        if (bluestein) c[e] = f.chirp[b];
      }
    }
#pragma unroll
    for (int e = 0; e < kTE / 2; ++e) {
      const int s = threadIdx.x + kTN * e;
      const int b = s >> logMC, mc = s & (MC - 1);
      double2 z0 = x[e], z1 = cmulw<-1>(x[e], w[e]);
      if (bluestein) {
        z0 = cmulw<-1>(z0, c[e]);
        z1 = cmulw<-1>(z1, c[e]);
      }
      lds[lpad((b << logTw) + 2 * mc)] = z0;
      lds[lpad((b << logTw) + 2 * mc + 1)] = z1;
    }
  }
  lds_barrier();
  team_fft_core<kTE, kTN, -1>(f, lds, M, logTw, bluestein, bluestein ? f.chirp_c : nullptr);
  const int nv = a.nval[ni], ncol = a.ncol[ni];
  const int QH = (hi + 1) >> 1;
#pragma unroll
  for (int e = 0; e < kTE / 2; ++e) {
    const int s = threadIdx.x + kTN * e;
    const int mc = s & (MC - 1), r = (s >> logMC) & 1, q = s >> logTw;
    const int m = m0 + mc, mp = 2 * q + r;
    if (q >= QH || m >= hi || mp >= hi) continue;
    const int t = 2 * mc + r;
    const double2 w = tw8[mp];
    double2 v3 = cmulw<-1>(lds[lpad((q << logTw) + t)], w);
    if (mp >= 1) {
      const int qm = (4 * hi - mp) >> 1;
      double2 v2m = cmul(lds[lpad((qm << logTw) + t)], w);
      if ((m + nv) & 1) v2m = make_double2(-v2m.x, -v2m.y);
      v3 = cadd(v3, v2m);
    }
    const int rot = ((m - nv) % 4 + 4) % 4;
    double2 z;
    if (rot == 0) z = v3;
    else if (rot == 1) z = make_double2(-v3.y, v3.x);
    else if (rot == 2) z = make_double2(-v3.x, -v3.y);
    else z = make_double2(v3.y, -v3.x);
    for (int kc = 0; kc < ncol; ++kc) {
      const int c = a.col0[ni][kc];
      const double2 o = a.cpart[ni][kc] ? make_double2(-z.y, z.x) : z;
      Vt[((long long)c * hi + mp) * hi + m] = o;
    }
  }
}

// Kernels over one scale or over two scales of the same shape (the full-band
// scales 0 and 1: only their data pointers differ): workgroups below `half`
// run the first argument set, the others the second; one scale has half =
// gridDim.x.  The workgroup holds nt_of(LOGM) threads with kTE slots each:
// kTN threads up to M = kTS, and one sequence of M = 2^LOGM slots beyond
// (512 threads for 4096: band limits 513..1024; 1024 threads for 8192: band
// limits above 1024; their slots are dynamic LDS).
__host__ __device__ constexpr int nt_of(int logm) { return logm > kLogTS ? (1 << logm) / kTE : kTN; }
__host__ __device__ constexpr int lds_of(int logm) { return logm > kLogTS ? (1 << logm) * (int)sizeof(double2) : 0; }
// waves per SIMD: three of the kTN-thread engine (168 VGPRs), four beyond
// (two 512-thread workgroups or one of 1024 share a CU, 128 VGPRs)
__host__ __device__ constexpr int occ_of(int logm) { return logm > kLogTS ? 4 : 3; }
// largest work length, and the LDS the beta stage's column sums add to the slots
constexpr int kBigLogM = 13, kCsumLds = nt_of(kBigLogM) * (int)sizeof(double2) + 64;
inline bool big_fft(const FftSpec &f) { return f.bluestein && f.M > kTS && f.M <= 1 << kBigLogM; }
#define S2DW_SLOTS(LOGM)                                            \
  extern __shared__ double2 dyn_lds[];                              \
  __shared__ double2 fix_lds[(LOGM) > kLogTS ? 1 : lpad_size(kTS)]; \
  double2 *lds = (LOGM) > kLogTS ? dyn_lds : fix_lds;

__global__ __launch_bounds__(kTN, 3) void k_beta_ana_t2(const BetaAnaArgs a0, const BetaAnaArgs a1, int nmt, int half) {
  __shared__ double2 lds[lpad_size(kTS)];
  const bool second = (int)blockIdx.x >= half;
  beta_ana_body(second ? a1 : a0, nmt, lds, blockIdx.x - (second ? half : 0), half);
}
template <int LOGM, int BL>
__global__ __launch_bounds__(nt_of(LOGM), occ_of(LOGM)) void k_alpha_c2r_t2(const AlphaArgs a0, const AlphaArgs a1,
                                                                           int npt, int half) {
  S2DW_SLOTS(LOGM)
  const bool second = (int)blockIdx.x >= half;
  alpha_c2r_body<LOGM, BL, false, nt_of(LOGM)>(second ? a1 : a0, npt, lds, blockIdx.x - (second ? half : 0), half);
}
template <int LOGM, int BL>
__global__ __launch_bounds__(nt_of(LOGM), occ_of(LOGM)) void k_alpha_c2r_t2m(const AlphaArgs a0, const AlphaArgs a1,
                                                                            int npt, int half) {
  S2DW_SLOTS(LOGM)
  const bool second = (int)blockIdx.x >= half;
  alpha_c2r_body<LOGM, BL, true, nt_of(LOGM)>(second ? a1 : a0, npt, lds, blockIdx.x - (second ? half : 0), half);
}
template <int LOGM, int BL>
__global__ __launch_bounds__(nt_of(LOGM), occ_of(LOGM)) void k_alpha_r2c_t2(const AlphaArgs a0, const AlphaArgs a1,
                                                                           int npt, int half) {
  S2DW_SLOTS(LOGM)
  const bool second = (int)blockIdx.x >= half;
  alpha_r2c_body<LOGM, BL, nt_of(LOGM)>(second ? a1 : a0, npt, lds, blockIdx.x - (second ? half : 0), half);
}

template <int LOGM, int BL>
__global__ __launch_bounds__(nt_of(LOGM), occ_of(LOGM)) void k_alpha_syn_t2(const AlphaArgs a0, const AlphaArgs a1,
                                                                           int npt, int half) {
  S2DW_SLOTS(LOGM)
  const bool second = (int)blockIdx.x >= half;
  alpha_syn_body<LOGM, nt_of(LOGM)>(second ? a1 : a0, lds, blockIdx.x - (second ? half : 0), half);
}

// Alpha stages of the full-band pair on the odd-length engine, length
// n = 2hi - 1 = R0 R1 R2 (no Bluestein).  A workgroup holds kOddT row pairs
// (each one packed complex sequence, as in alpha_c2r_body / alpha_r2c_body)
// of one g; tile = g * npt + pair group.  otw: e^{+2 pi i k/n}, k < n.
// launch shape from a sweep: 128 threads, one row pair per workgroup, the
// radix-31 stage's output pairs shared by the two waves
constexpr int kOddT = 1, kOddNT = 128, kOddSplit = 2, kOddHi = 512;
// MOM: instead of storing W, the workgroup reduces its values to one moments
// record (s2dw_moments.h) at a.mp + 8 tile, as alpha_c2r_body<..., true>.
template <int R0, int R1, int R2, int NT = kOddNT, int T = kOddT, int SPLIT = kOddSplit, bool MOM = false>
__global__ __launch_bounds__(NT, 3) void k_alpha_c2r_o2(const AlphaArgs a0, const AlphaArgs a1, int npt,
                                                     const double2 *__restrict__ otw) {
  constexpr int n = R0 * R1 * R2, hi = (n + 1) / 2;
  __shared__ double2 lds[n * T];
  const int half = gridDim.x >> 1, second = blockIdx.x >= (unsigned)half;
  const AlphaArgs &a = second ? a1 : a0;
  const int tile = xcd_tile(blockIdx.x - (second ? half : 0), half);
  const int g = tile / npt, p0 = (tile - g * npt) * T;
  // slot k < hi: p_k + i q_k (k = 0: Re p_0 + i Re q_0), slot n - k:
  // conj(p_k) + i conj(q_k), for the packed rows p = 2 pidx, q = 2 pidx + 1
  static_assert(T == 1 && hi % NT == 0 && NT % 2 == 0, "load_pair: one row pair, whole rounds of lane pairs");
#pragma unroll
  for (int i = 0; i < hi / NT; ++i) {
    const int t = 0, kk = threadIdx.x + NT * i;
    double2 p, q;
    load_pair(a.Tb + (long long)g * 2 * hi * hi + 2 * p0 * a.tbb, a.tbb, a.tbm, kk & ~1, kk | 1, p, q);
    lds[kk * T + t] = kk == 0 ? make_double2(p.x, q.x) : make_double2(p.x - q.y, p.y + q.x);
    if (kk) lds[(n - kk) * T + t] = make_double2(p.x + q.y, -p.y + q.x);
  }
  lds_barrier();
  odd_fft<R0, R1, R2, +1, NT, T, SPLIT>(lds, otw);
  if constexpr (MOM) {
    constexpr int E = 2 * ((n * T + NT - 1) / NT);
    double v[E], wt[E];
#pragma unroll
    for (int i = 0; i < E / 2; ++i) {
      const int idx = threadIdx.x + NT * i;
      const bool ok = idx < n * T && p0 + idx % T < hi;
      const double2 z = lds[ok ? idx : 0];  // slot k T + t = idx
      v[2 * i] = z.x;
      v[2 * i + 1] = z.y;
      wt[2 * i] = wt[2 * i + 1] = ok ? 1.0 : 0.0;
    }
    mom_record<E, NT>(v, wt, 0.0, a.mp + 8LL * tile);
    return;
  }
  for (int idx = threadIdx.x; idx < n * T; idx += NT) {
    const int t = idx % T, k = idx / T, pidx = p0 + t;
    if (pidx < hi) {
      const double2 z = lds[k * T + t];
      double *w0 = a.W + ((long long)g * 2 * hi + 2 * pidx) * n;
      w0[k] = z.x;
      w0[n + k] = z.y;
    }
  }
}

// One sequence per workgroup (alpha_syn_body's ids and outputs).
template <int R0, int R1, int R2, int NT = kOddNT, int SPLIT = kOddSplit>
__global__ __launch_bounds__(NT, 3) void k_alpha_syn_o2(const AlphaArgs a0, const AlphaArgs a1,
                                                     const double2 *__restrict__ otw) {
  constexpr int n = R0 * R1 * R2, hi = (n + 1) / 2, E = (n + NT - 1) / NT;
  __shared__ double2 lds[n];
  const int half = gridDim.x >> 1, second = blockIdx.x >= (unsigned)half;
  const AlphaArgs &a = second ? a1 : a0;
  const SynSeq us = syn_seq(a, xcd_tile(blockIdx.x - (second ? half : 0), half));
  {
    int k[E];
    double2 z[E];
#pragma unroll
    for (int e = 0; e < E; ++e) k[e] = threadIdx.x + NT * e;
    syn_gather<E>(a, us, true, k, z);
#pragma unroll
    for (int e = 0; e < E; ++e)
      if (k[e] < n) lds[k[e]] = z[e];
  }
  lds_barrier();
  odd_fft<R0, R1, R2, -1, NT, 1, SPLIT>(lds, otw);
  for (int kk = threadIdx.x; kk < hi; kk += NT) {
    const double2 zp = lds[kk];
    const double2 zm = us.packed ? lds[kk ? n - kk : 0] : zp;
    syn_store(a, us, kk, zp, zm);
  }
}

// The same lengths without the gamma-DFT (gamma_first false): one packed row
// pair of one g per workgroup, alpha_r2c_body's outputs.
template <int R0, int R1, int R2, int NT = kOddNT, int SPLIT = kOddSplit>
__global__ __launch_bounds__(NT, 3) void k_alpha_r2c_o2(const AlphaArgs a0, const AlphaArgs a1,
                                                     const double2 *__restrict__ otw) {
  constexpr int n = R0 * R1 * R2, hi = (n + 1) / 2;
  __shared__ double2 lds[n];
  const int half = gridDim.x >> 1, second = blockIdx.x >= (unsigned)half;
  const AlphaArgs &a = second ? a1 : a0;
  const int row = 2 * xcd_tile(blockIdx.x - (second ? half : 0), half);  // 2 hi g + 2 pidx
  const double *w0 = a.W + (long long)row * n;
  for (int k = threadIdx.x; k < n; k += NT) lds[k] = make_double2(w0[k], w0[n + k]);
  lds_barrier();
  odd_fft<R0, R1, R2, -1, NT, 1, SPLIT>(lds, otw);
  const double h = 0.5 * a.scale;
  double2 *v0 = a.V + (long long)row * hi;
  for (int kk = threadIdx.x; kk < hi; kk += NT) {
    const double2 zp = lds[kk];
    const double2 zm = lds[kk ? n - kk : 0];
    v0[kk] = make_double2(h * (zp.x + zm.x), h * (zp.y - zm.y));
    v0[hi + kk] = make_double2(h * (zp.y + zm.y), -h * (zp.x - zm.x));
  }
}

// ---------------------------------------------------------------------------
// Alpha stages and one-FFT-per-column beta stages on the three-stage engine
// (Bluestein, M = 2^LOGM, M/16 threads, one sequence or column per
// workgroup): inputs go straight into the first stage's registers and outputs
// leave from the last stage's; the slots carry only what another thread needs
// (the mirrored halves of the packed rows and of the beta columns).
// ---------------------------------------------------------------------------
// SEQ = 1: the workgroup is one sequence; SEQ > 1 (grouped launches): SEQ
// sequences of NT threads, row pairs p0 + i of one g.
template <int LOGM, bool MOM, int SEQ>
__device__ __forceinline__ void alpha_c2r16_body(const AlphaArgs &a, int npt, double2 *lds, int bid, int nb) {
  constexpr int NT = (1 << LOGM) / 16;
  static_assert(!MOM || SEQ == 1, "one record per workgroup");
  const int tid = SEQ > 1 ? threadIdx.x & (NT - 1) : threadIdx.x, sub = SEQ > 1 ? threadIdx.x / NT : 0;
  const int hi = a.hi, n = 2 * hi - 1, tile = xcd_tile(bid, nb);
  const int g = tile / npt, pidx0 = (tile - g * npt) * SEQ + sub;
  const bool on = SEQ == 1 || pidx0 < hi;
  const int pidx = on ? pidx0 : hi - 1;
  double *buf = (double *)lds + sub * lpad16(1 << LOGM);
  double2 *mir = (double2 *)buf;
  double2 v[16];
  {
    const double2 *rb = a.Tb + (long long)g * 2 * hi * hi + 2 * pidx * a.tbb;
    // slots k < hi <= M/4 in registers, slot n - k through LDS: reading the
    // rows a second time from L2 for it costs more
    double2 p[4], q[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int k = tid + NT * r;
      load_pair(rb, a.tbb, a.tbm, min(k & ~1, hi - 1), min(k | 1, hi - 1), p[r], q[r]);
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int k = tid + NT * r;
      v[r] = k == 0 ? make_double2(p[r].x, q[r].x) : make_double2(p[r].x - q[r].y, p[r].y + q[r].x);
      if (k >= 1 && k < hi) mir[hi - 1 - k] = make_double2(p[r].x + q[r].y, -p[r].y + q[r].x);
    }
    lds_barrier();
#pragma unroll
    for (int r = 0; r < 8; ++r) {
      const int k = tid + NT * r;
      double2 z = make_double2(0.0, 0.0);
      if (k < hi) {
        if (r < 4) z = v[r & 3];
      } else if (k < n) {
        z = mir[k - hi];
      }
      v[r] = cmulw<+1>(z, a.f.chirp[k]);  // the chirp table is zero for n <= k < M
    }
    lds_barrier();
  }
  team16_bluestein<LOGM, +1, (SEQ > 1)>(a.f, buf, v);
  if constexpr (MOM) {
    double x[16], wt[16];
#pragma unroll
    for (int r = 0; r < 8; ++r) {
      const int k = tid + NT * r;
      const double2 z = cmulw<+1>(v[r], a.f.chirp[k]);
      x[2 * r] = z.x;
      x[2 * r + 1] = z.y;
      wt[2 * r] = wt[2 * r + 1] = k < n ? 1.0 : 0.0;
    }
    mom_record<16, NT>(x, wt, 0.0, a.mp + 8LL * tile);
    return;
  }
  double *w0 = a.W + ((long long)g * 2 * hi + 2 * pidx) * n;
#pragma unroll
  for (int r = 0; r < 8; ++r) {
    const int k = tid + NT * r;
    if (on && k < n) {
      const double2 z = cmulw<+1>(v[r], a.f.chirp[k]);
      w0[k] = z.x;
      w0[n + k] = z.y;
    }
  }
}

template <int LOGM, bool MOM>
__global__ __launch_bounds__((1 << LOGM) / 16, MOM && LOGM == 12 ? 2 : 3) void k_alpha_c2r16(const AlphaArgs a0, const AlphaArgs a1, int npt,
                                                                    int half) {
  extern __shared__ double2 dyn_lds[];
  const bool second = (int)blockIdx.x >= half;
  alpha_c2r16_body<LOGM, MOM, 1>(second ? a1 : a0, npt, dyn_lds, blockIdx.x - (second ? half : 0), half);
}

template <int LOGM>
__global__ __launch_bounds__((1 << LOGM) / 16, 3) void k_alpha_syn16(const AlphaArgs a0, const AlphaArgs a1, int half) {
  constexpr int NT = (1 << LOGM) / 16;
  extern __shared__ double2 dyn_lds[];
  const bool second = (int)blockIdx.x >= half;
  const AlphaArgs &a = second ? a1 : a0;
  const int hi = a.hi, n = 2 * hi - 1;
  const SynSeq us = syn_seq(a, xcd_tile(blockIdx.x - (second ? half : 0), half));
  double2 v[16];
  {
    int k[8];
    double2 z[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) k[e] = threadIdx.x + NT * e;
    syn_gather<8>(a, us, true, k, z);
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = cmulw<-1>(z[e], a.f.chirp[k[e]]);  // chirp: zero for n <= k < M
  }
  team16_bluestein<LOGM, -1>(a.f, (double *)dyn_lds, v);
#pragma unroll
  for (int r = 0; r < 8; ++r) v[r] = cmulw<-1>(v[r], a.f.chirp[threadIdx.x + NT * r]);
  if (us.packed) {  // uniform: Z(n - k), n - k >= hi, from the thread that holds it
    lds_barrier();
#pragma unroll
    for (int r = 0; r < 8; ++r) {
      const int k = threadIdx.x + NT * r;
      if (k >= hi && k < n) dyn_lds[k - hi] = v[r];
    }
    lds_barrier();
  }
#pragma unroll
  for (int r = 0; r < 8; ++r) {
    const int kk = threadIdx.x + NT * r;
    if (kk < hi) syn_store(a, us, kk, v[r], us.packed && kk ? dyn_lds[n - kk - hi] : v[r]);
  }
}

// ... without the gamma-DFT: one packed row pair of one g per workgroup
template <int LOGM>
__global__ __launch_bounds__((1 << LOGM) / 16, 3) void k_alpha_r2c16(const AlphaArgs a0, const AlphaArgs a1, int half) {
  constexpr int NT = (1 << LOGM) / 16;
  extern __shared__ double2 dyn_lds[];
  const bool second = (int)blockIdx.x >= half;
  const AlphaArgs &a = second ? a1 : a0;
  const int hi = a.hi, n = 2 * hi - 1;
  const int row = 2 * xcd_tile(blockIdx.x - (second ? half : 0), half);  // 2 hi g + 2 pidx
  const double *w0 = a.W + (long long)row * n;
  double2 v[16];
#pragma unroll
  for (int r = 0; r < 8; ++r) {
    const int k = threadIdx.x + NT * r, kk = k < n ? k : 0;
    v[r] = cmulw<-1>(make_double2(w0[kk], w0[n + kk]), a.f.chirp[k]);  // chirp: zero for n <= k < M
  }
  team16_bluestein<LOGM, -1>(a.f, (double *)dyn_lds, v);
#pragma unroll
  for (int r = 0; r < 8; ++r) v[r] = cmulw<-1>(v[r], a.f.chirp[threadIdx.x + NT * r]);
  lds_barrier();
#pragma unroll
  for (int r = 0; r < 8; ++r) {  // Z(n - k), n - k >= hi, from the thread that holds it
    const int k = threadIdx.x + NT * r;
    if (k >= hi && k < n) dyn_lds[k - hi] = v[r];
  }
  lds_barrier();
  const double h = 0.5 * a.scale;
  double2 *v0 = a.V + (long long)row * hi;
#pragma unroll
  for (int r = 0; r < 8; ++r) {
    const int kk = threadIdx.x + NT * r;
    if (kk >= hi) continue;
    const double2 zp = v[r], zm = kk ? dyn_lds[n - kk - hi] : v[r];
    v0[kk] = make_double2(h * (zp.x + zm.x), h * (zp.y - zm.y));
    v0[hi + kk] = make_double2(h * (zp.y + zm.y), -h * (zp.x - zm.x));
  }
}

__global__ __launch_bounds__(kTN, 3) void k_beta_syn_t2(const BetaSynArgs a, const double2 *V1, double2 *Vt1,
                                                        const double2 *tw81, int nmt, int half) {
  __shared__ double2 lds[lpad_size(kTS)];
  const bool second = (int)blockIdx.x >= half;
  beta_syn_body(a, second ? V1 : a.V, second ? Vt1 : a.Vt, second ? tw81 : a.tw8, nmt, lds,
                          blockIdx.x - (second ? half : 0), half);
}

// ---------------------------------------------------------------------------
// Beta stages of the full-band pair with one FFT of length L = 2hi = 2^LOGM
// per column, instead of one per column and output parity (the kernels
// above transform each column twice and keep half of each result).  A
// workgroup holds Tw = kTS / L columns, so its loads and stores move Tw
// adjacent m at a time.  theta_k = pi k / (4hi), e^{i theta_k} = tw8[k].
//
// Analysis, x_k = Tg[g][k][m] (k < hi), the reference's sum
// (s2dw_core_mod.f90:707-743)
//   Tb(b) = x_0 + sum_{k>=1} x_k 2cos(k beta_b)     (m + N - 1 even)
//   Tb(b) = x_0 + sum_{k>=1} x_k 2i sin(k beta_b)   (odd),  beta_b = (2b+1) theta_1,
// is a DCT-III (DST-III) of length L, computed as the transpose of
// Makhoul's DCT-II algorithm: V_k = s e^{-i theta_k} x_k and
// V_{L-k} = e^{i theta_k} x_k for 1 <= k < hi (s = +1 even, -1 odd),
// V_0 = x_0 (even) or 0 (odd), V_hi = 0; forward FFT v = F_L V; then
// Tb(2n) = v_n, Tb(2n+1) = v_{L-1-n} (even), and Tb(2n) = x_0 + v_n,
// Tb(2n+1) = x_0 - v_{L-1-n} (odd: the DST-III outputs carry (-1)^b).
//
// Synthesis, U_b (b < L) of one n-index and column: with a_b = U_b (m + n
// even) or (-1)^b U_b (odd), v_n = a_{2n}, v_{L-1-n} = a_{2n+1}, V = F_L v,
//   sum_b U_b (e^{-i m' beta_b} +- e^{i m' beta_b})
//     = e^{-i theta_m'} V_m' +- e^{i theta_m'} V_{L-m'}          (m' >= 1)
// (Makhoul's DCT-II for complex data, DST-II through the sign-alternated
// input), and sum_b U_b for m' = 0 (a column sum, reduced while the columns
// are loaded).  The rotation and column fan-out follow beta_syn_body.
// ---------------------------------------------------------------------------
// BL = true: the transform length L = 2hi is not a power of two and runs
// through Bluestein on the work length M = 2^LOGM >= 2L - 1 (slots L..M-1
// zero, inputs times conj(chirp_k), outputs times conj(chirp_k) in the last
// stage); otherwise L = M.
template <int LOGM, int NT = kTN, bool BL = false>
__device__ __forceinline__ void beta_ana_h2_body(const BetaAnaArgs &a, int nmt, double2 *lds, int bid, int nb) {
  constexpr int M = 1 << LOGM, logTw = clog2(NT * kTE) - LOGM, Tw = 1 << logTw;
  const int hi = BL ? a.hi : M / 2, L = 2 * hi;
  const int tile = xcd_tile(bid, nb);
  const int g = tile / nmt, m0 = (tile - g * nmt) * Tw, N = a.N;
  if constexpr (BL) {
#pragma unroll
    for (int e = 0; e < kTE; ++e) {
      const int i = threadIdx.x + NT * e;  // < Tw M
      if ((i >> logTw) >= L) lds[lpad(i)] = make_double2(0.0, 0.0);
    }
  }
  {
    double2 x[kTE / 2], w[kTE / 2];
#pragma unroll
    for (int e = 0; e < kTE / 2; ++e) {
      const int s = threadIdx.x + NT * e;  // < Tw M/2
      const int t = s & (Tw - 1), k = s >> logTw, m = m0 + t;
      x[e] = m < hi && k < hi ? a.Tg[((long long)g * hi + k) * hi + m] : make_double2(0.0, 0.0);
      w[e] = a.tw8[k < hi ? k : 0];
    }
#pragma unroll
    for (int e = 0; e < kTE / 2; ++e) {
      const int s = threadIdx.x + NT * e;
      const int t = s & (Tw - 1), k = s >> logTw, m = m0 + t;
      if (BL && k >= hi) continue;
      const bool odd = (m + N - 1) & 1;
      double2 v0, v1;  // slots k and L - k (k = 0: slots 0 and hi)
      int k1;
      if (k == 0) {
        v0 = odd ? make_double2(0.0, 0.0) : x[e];
        v1 = make_double2(0.0, 0.0);
        k1 = hi;
      } else {
        const double2 lo = cmulw<-1>(x[e], w[e]);
        v0 = odd ? make_double2(-lo.x, -lo.y) : lo;
        v1 = cmul(x[e], w[e]);
        k1 = L - k;
      }
      if constexpr (BL) {
        v0 = cmulw<-1>(v0, a.f.chirp[k]);
        v1 = cmulw<-1>(v1, a.f.chirp[k1]);
      }
      lds[lpad((k << logTw) + t)] = v0;
      lds[lpad((k1 << logTw) + t)] = v1;
    }
  }
  lds_barrier();
  team_fft_core<kTE, NT, -1>(a.f, lds, M, logTw, BL, BL ? a.f.chirp_c : nullptr);
  // lanes along b, so that the stores of a column are contiguous where tbb = 1
#pragma unroll
  for (int e = 0; e < kTE; ++e) {
    const int s = threadIdx.x + NT * e;  // < Tw M
    const int t = s >> LOGM, b = s & (M - 1), m = m0 + t;
    if (m < hi && (!BL || b < L)) {
      const bool up = b & 1;
      double2 y = lds[lpad(((up ? L - 1 - (b >> 1) : b >> 1) << logTw) + t)];
      if ((m + N - 1) & 1) {
        const double2 x0 = a.Tg[(long long)g * hi * hi + m];
        y = up ? csub(x0, y) : cadd(x0, y);
      }
      a.Tb[(long long)g * L * hi + b * a.tbb + m * a.tbm] = y;
    }
  }
}

// csum: NT entries of LDS for the column sums (m' = 0)
template <int LOGM, int NT = kTN, bool BL = false>
__device__ __forceinline__ void beta_syn_h2_body(const BetaSynArgs &a, const double2 *V, double2 *Vt,
                                                 const double2 *tw8, int nmt, double2 *lds, double2 *csum, int bid,
                                                 int nb) {
  constexpr int M = 1 << LOGM, logTw = clog2(NT * kTE) - LOGM, Tw = 1 << logTw;
  static_assert(Tw <= NT, "each thread loads one column");
  static_assert(NT % 64 == 0, "whole waves");
  constexpr int stride = Tw < 64 ? 64 : Tw;  // csum entries of one column: t + stride i
  const int hi = BL ? a.hi : M / 2, L = 2 * hi;
  const int tile = xcd_tile(bid, nb);
  const int ni = tile / nmt, m0 = (tile - ni * nmt) * Tw;
  const int nv = a.nval[ni], ncol = a.ncol[ni];
  const double2 *U = V + (long long)ni * L * hi;
  {
    double2 x[kTE];
    double2 cs = make_double2(0.0, 0.0);
    const int t = threadIdx.x & (Tw - 1), m = m0 + t;  // the thread's column
#pragma unroll
    for (int e = 0; e < kTE; ++e) {
      const int b = (threadIdx.x + NT * e) >> logTw;  // < M
      x[e] = m < hi && b < L ? U[(long long)b * hi + m] : make_double2(0.0, 0.0);
    }
#pragma unroll
    for (int e = 0; e < kTE; ++e) {
      const int b = (threadIdx.x + NT * e) >> logTw;
      cs = cadd(cs, x[e]);
      const bool flip = ((m + nv) & 1) && (b & 1);
      // b >= L (Bluestein only): slot b itself, zero
      const int slot = b >= L ? b : (b & 1) ? L - 1 - (b >> 1) : b >> 1;
      double2 v = flip ? make_double2(-x[e].x, -x[e].y) : x[e];
      if constexpr (BL) {
        if (b < L) v = cmulw<-1>(v, a.f.chirp[slot]);
      }
      lds[lpad((slot << logTw) + t)] = v;
    }
    if constexpr (Tw < 64) {
      // lanes with equal lane mod Tw hold the same column
#pragma unroll
      for (int o = Tw; o < 64; o <<= 1) {
        cs.x += __shfl_xor(cs.x, o);
        cs.y += __shfl_xor(cs.y, o);
      }
      if ((threadIdx.x & 63) < Tw) csum[threadIdx.x] = cs;
    } else {
      csum[threadIdx.x] = cs;
    }
  }
  lds_barrier();
  team_fft_core<kTE, NT, -1>(a.f, lds, M, logTw, BL, BL ? a.f.chirp_c : nullptr);
#pragma unroll
  for (int e = 0; e < kTE / 2; ++e) {
    const int s = threadIdx.x + NT * e;  // < Tw M/2
    const int t = s & (Tw - 1), mp = s >> logTw, m = m0 + t;
    if (m >= hi || (BL && mp >= hi)) continue;
    double2 v3;
    if (mp == 0) {
      v3 = csum[t];
#pragma unroll
      for (int j = t + stride; j < NT; j += stride) v3 = cadd(v3, csum[j]);
    } else {
      const double2 w = tw8[mp];
      v3 = cmulw<-1>(lds[lpad((mp << logTw) + t)], w);
      const double2 v2m = cmul(lds[lpad(((L - mp) << logTw) + t)], w);
      v3 = ((m + nv) & 1) ? csub(v3, v2m) : cadd(v3, v2m);
    }
    const int rot = ((m - nv) % 4 + 4) % 4;
    double2 z;
    if (rot == 0) z = v3;
    else if (rot == 1) z = make_double2(-v3.y, v3.x);
    else if (rot == 2) z = make_double2(-v3.x, -v3.y);
    else z = make_double2(v3.y, -v3.x);
    for (int kc = 0; kc < ncol; ++kc) {
      const int c = a.col0[ni][kc];
      const double2 o = a.cpart[ni][kc] ? make_double2(-z.y, z.x) : z;
      Vt[((long long)c * hi + mp) * hi + m] = o;
    }
  }
}

template <int LOGM, bool BL>
__global__ __launch_bounds__(nt_of(LOGM), occ_of(LOGM)) void k_beta_ana_h2(const BetaAnaArgs a0, const BetaAnaArgs a1,
                                                                          int nmt, int half) {
  S2DW_SLOTS(LOGM)
  const bool second = (int)blockIdx.x >= half;
  beta_ana_h2_body<LOGM, nt_of(LOGM), BL>(second ? a1 : a0, nmt, lds, blockIdx.x - (second ? half : 0), half);
}

template <int LOGM, bool BL>
__global__ __launch_bounds__(nt_of(LOGM), occ_of(LOGM)) void k_beta_syn_h2(const BetaSynArgs a, const double2 *V1,
                                                                          double2 *Vt1, const double2 *tw81, int nmt,
                                                                          int half) {
  S2DW_SLOTS(LOGM)
  __shared__ double2 csum[nt_of(LOGM)];
  const bool second = (int)blockIdx.x >= half;
  beta_syn_h2_body<LOGM, nt_of(LOGM), BL>(a, second ? V1 : a.V, second ? Vt1 : a.Vt, second ? tw81 : a.tw8, nmt, lds,
                                          csum, blockIdx.x - (second ? half : 0), half);
}
#undef S2DW_SLOTS

// The same two beta stages (Bluestein, L = 2hi <= M/2) on the three-stage
// engine, one column per workgroup.
template <int LOGM>
__global__ __launch_bounds__((1 << LOGM) / 16, 3) void k_beta_ana16(const BetaAnaArgs a0, const BetaAnaArgs a1, int nmt,
                                                                   int half) {
  constexpr int NT = (1 << LOGM) / 16;
  extern __shared__ double2 dyn_lds[];
  const bool second = (int)blockIdx.x >= half;
  const BetaAnaArgs &a = second ? a1 : a0;
  const int hi = a.hi, L = 2 * hi, tile = xcd_tile(blockIdx.x - (second ? half : 0), half);
  const int g = tile / nmt, m = tile - g * nmt;  // nmt = hi
  const bool odd = (m + a.N - 1) & 1;
  const double2 *T = a.Tg + (long long)g * hi * hi + m;
  double2 v[16];
  {
    // slots k < hi in registers, slot L - k through the slots
    double2 x[4], w[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int k = threadIdx.x + NT * r;  // < M/4, hi <= M/4
      x[r] = T[(long long)(k < hi ? k : 0) * hi];
      w[r] = a.tw8[k < hi ? k : 0];
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int k = threadIdx.x + NT * r;
      const double2 lo = cmulw<-1>(x[r], w[r]);
      v[r] = odd ? make_double2(-lo.x, -lo.y) : lo;
      if (k == 0 && odd) v[r] = make_double2(0.0, 0.0);
      if (k < hi) dyn_lds[k ? hi - k : 0] = k ? cmul(x[r], w[r]) : make_double2(0.0, 0.0);
    }
    lds_barrier();
#pragma unroll
    for (int r = 0; r < 8; ++r) {
      const int k = threadIdx.x + NT * r;
      double2 z = make_double2(0.0, 0.0);
      if (k < hi) {
        if (r < 4) z = v[r & 3];
      } else if (k < L) {
        z = dyn_lds[k - hi];
      }
      v[r] = cmulw<-1>(z, a.f.chirp[k]);
    }
    lds_barrier();
  }
  team16_bluestein<LOGM, -1>(a.f, (double *)dyn_lds, v);
  const double2 x0 = odd ? T[0] : make_double2(0.0, 0.0);
  double2 *o = a.Tb + (long long)g * L * hi + m * a.tbm;
#pragma unroll
  for (int r = 0; r < 8; ++r) {
    const int k = threadIdx.x + NT * r;
    if (k < L) {
      const double2 y = cmulw<-1>(v[r], a.f.chirp[k]);
      const bool up = k >= hi;  // Tb(2n) = [x0 +] v_n, Tb(2n+1) = [x0 -] v_{L-1-n}
      o[(up ? 2 * (L - 1 - k) + 1 : 2 * k) * a.tbb] = up && odd ? csub(x0, y) : cadd(x0, y);
    }
  }
}

template <int LOGM>
__global__ __launch_bounds__((1 << LOGM) / 16, 3) void k_beta_syn16(const BetaSynArgs a, const double2 *V1, double2 *Vt1,
                                                                   const double2 *tw81, int nmt, int half) {
  constexpr int NT = (1 << LOGM) / 16;
  extern __shared__ double2 dyn_lds[];
  __shared__ double2 csum[NT / 64];
  const bool second = (int)blockIdx.x >= half;
  const double2 *tw8 = second ? tw81 : a.tw8;
  const int hi = a.hi, L = 2 * hi, tile = xcd_tile(blockIdx.x - (second ? half : 0), half);
  const int ni = tile / nmt, m = tile - ni * nmt;  // nmt = hi
  const int nv = a.nval[ni], ncol = a.ncol[ni];
  const bool odd = (m + nv) & 1;
  const double2 *U = (second ? V1 : a.V) + (long long)ni * L * hi + m;
  double2 v[16];
  {
    double2 c[8];
#pragma unroll
    for (int r = 0; r < 8; ++r) {
      const int k = threadIdx.x + NT * r;
      const int b = k < hi ? 2 * k : 2 * (L - 1 - k) + 1;
      v[r] = k < L ? U[(long long)b * hi] : make_double2(0.0, 0.0);
      c[r] = a.f.chirp[k];  // zero for L <= k < M
    }
    double2 cs = make_double2(0.0, 0.0);
#pragma unroll
    for (int r = 0; r < 8; ++r) {
      cs = cadd(cs, v[r]);
      const bool flip = odd && threadIdx.x + NT * r >= (unsigned)hi;  // odd b
      v[r] = cmulw<-1>(flip ? make_double2(-v[r].x, -v[r].y) : v[r], c[r]);
    }
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      cs.x += __shfl_xor(cs.x, o);
      cs.y += __shfl_xor(cs.y, o);
    }
    if ((threadIdx.x & 63) == 0) csum[threadIdx.x >> 6] = cs;
  }
  team16_bluestein<LOGM, -1>(a.f, (double *)dyn_lds, v);  // its barriers also publish csum
#pragma unroll
  for (int r = 0; r < 8; ++r) v[r] = cmulw<-1>(v[r], a.f.chirp[threadIdx.x + NT * r]);
  lds_barrier();
#pragma unroll
  for (int r = 0; r < 8; ++r) {
    const int k = threadIdx.x + NT * r;
    if (k >= hi && k < L) dyn_lds[k - hi] = v[r];
  }
  lds_barrier();
  double2 *Vt = second ? Vt1 : a.Vt;
  const int rot = ((m - nv) % 4 + 4) % 4;
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int mp = threadIdx.x + NT * r;  // hi <= M/4
    if (mp >= hi) continue;
    double2 v3;
    if (mp == 0) {
      v3 = csum[0];
#pragma unroll
      for (int j = 1; j < NT / 64; ++j) v3 = cadd(v3, csum[j]);
    } else {
      const double2 w = tw8[mp];
      v3 = cmulw<-1>(v[r], w);
      const double2 v2m = cmul(dyn_lds[hi - mp], w);
      v3 = odd ? csub(v3, v2m) : cadd(v3, v2m);
    }
    double2 z;
    if (rot == 0) z = v3;
    else if (rot == 1) z = make_double2(-v3.y, v3.x);
    else if (rot == 2) z = make_double2(-v3.x, -v3.y);
    else z = make_double2(v3.y, -v3.x);
    for (int kc = 0; kc < ncol; ++kc) {
      const int c = a.col0[ni][kc];
      const double2 o = a.cpart[ni][kc] ? make_double2(-z.y, z.x) : z;
      Vt[((long long)c * hi + mp) * hi + m] = o;
    }
  }
}

// ---------------------------------------------------------------------------
// Grouped launches: several scales of one stage in a single grid (the two
// full-band scales together; the small scales together).  Scale (segment) s
// owns workgroups [first[s], first[s+1]); its arguments sit in a device
// table built with the plan, its body is chosen per workgroup by
// sel[s] = 2 log2(M) + bluestein for the specialised work lengths, 0 for the
// generic body.  One launch instead of one per scale saves launch and
// completion latency and shortens the relative tail of the grid.
// ---------------------------------------------------------------------------
struct SegTab {
  int nseg;
  int first[kMaxSc + 1];
  int sel[kMaxSc];
  int par[kMaxSc];  // workgroups per g (alpha) or per n-index (beta)
};

__device__ __forceinline__ int seg_of(const SegTab &t, int b) {
  int s = 0;
  for (int i = 1; i < t.nseg; ++i) s = b >= t.first[i] ? i : s;
  return s;
}

#define S2DW_SEL(BODY, LM, B, ...) \
  case 2 * (LM) + (B):             \
    BODY<LM, B>(__VA_ARGS__);      \
    break;
// three-stage engine in a grouped launch: 4096 >> log2(M) sequences per
// workgroup, selector kSel16 + log2(M)
constexpr int kSel16 = 200, kLds16g = (lpad16(4096) + 1) / 2;
#define S2DW_SEL16(LM, ...)                        \
  case kSel16 + (LM):                              \
    __VA_ARGS__;                                   \
    break;
// one-FFT-per-column beta bodies: selector kSelH2 + 2 log2(M) + bluestein
constexpr int kSelH2 = 100;
#define S2DW_SEL_H2(BODY, LM, B, ...)     \
  case kSelH2 + 2 * (LM) + (B):           \
    BODY<LM, kTN, (B) != 0>(__VA_ARGS__); \
    break;
#define S2DW_SEL_H2_ALL(BODY, ...)      \
  S2DW_SEL_H2(BODY, 4, 0, __VA_ARGS__)  \
  S2DW_SEL_H2(BODY, 5, 0, __VA_ARGS__)  \
  S2DW_SEL_H2(BODY, 6, 0, __VA_ARGS__)  \
  S2DW_SEL_H2(BODY, 7, 0, __VA_ARGS__)  \
  S2DW_SEL_H2(BODY, 8, 0, __VA_ARGS__)  \
  S2DW_SEL_H2(BODY, 9, 0, __VA_ARGS__)  \
  S2DW_SEL_H2(BODY, 10, 0, __VA_ARGS__) \
  S2DW_SEL_H2(BODY, 4, 1, __VA_ARGS__)  \
  S2DW_SEL_H2(BODY, 5, 1, __VA_ARGS__)  \
  S2DW_SEL_H2(BODY, 6, 1, __VA_ARGS__)  \
  S2DW_SEL_H2(BODY, 7, 1, __VA_ARGS__)  \
  S2DW_SEL_H2(BODY, 8, 1, __VA_ARGS__)  \
  S2DW_SEL_H2(BODY, 9, 1, __VA_ARGS__)  \
  S2DW_SEL_H2(BODY, 10, 1, __VA_ARGS__) \
  S2DW_SEL_H2(BODY, 11, 1, __VA_ARGS__)

__global__ __launch_bounds__(kTN, 3) void k_beta_ana_g(const SegTab t, const BetaAnaArgs *__restrict__ args) {
  __shared__ double2 lds[lpad_size(kTS)];
  const int s = seg_of(t, blockIdx.x), bid = blockIdx.x - t.first[s], nb = t.first[s + 1] - t.first[s];
  const BetaAnaArgs a = args[s];
  switch (t.sel[s]) {
    S2DW_SEL_H2_ALL(beta_ana_h2_body, a, t.par[s], lds, bid, nb)
    default: beta_ana_body(a, t.par[s], lds, bid, nb); break;
  }
}

__global__ __launch_bounds__(kTN, 3) void k_alpha_c2r_g(const SegTab t, const AlphaArgs *__restrict__ args,
                                                         double *wbase) {
  __shared__ double2 lds[kLds16g];
  const int s = seg_of(t, blockIdx.x), bid = blockIdx.x - t.first[s], nb = t.first[s + 1] - t.first[s];
  AlphaArgs a = args[s];
  a.W = wbase + a.woff;
  switch (t.sel[s]) {
    S2DW_SEL(alpha_c2r_body, 5, 1, a, t.par[s], lds, bid, nb)
    S2DW_SEL(alpha_c2r_body, 6, 1, a, t.par[s], lds, bid, nb)
    S2DW_SEL(alpha_c2r_body, 7, 1, a, t.par[s], lds, bid, nb)
    S2DW_SEL(alpha_c2r_body, 8, 1, a, t.par[s], lds, bid, nb)
    S2DW_SEL(alpha_c2r_body, 9, 1, a, t.par[s], lds, bid, nb)
    S2DW_SEL(alpha_c2r_body, 10, 1, a, t.par[s], lds, bid, nb)
    S2DW_SEL16(10, alpha_c2r16_body<10, false, (4096 >> 10)>(a, t.par[s], lds, bid, nb))
    S2DW_SEL16(11, alpha_c2r16_body<11, false, (4096 >> 11)>(a, t.par[s], lds, bid, nb))
    default: alpha_c2r_body<0, -1>(a, t.par[s], lds, bid, nb); break;
  }
}

__global__ __launch_bounds__(kTN, 3) void k_alpha_c2r_gm(const SegTab t, const AlphaArgs *__restrict__ args,
                                                          double *pbase) {
  __shared__ double2 lds[lpad_size(kTS)];
  const int s = seg_of(t, blockIdx.x), bid = blockIdx.x - t.first[s], nb = t.first[s + 1] - t.first[s];
  AlphaArgs a = args[s];
  a.mp = pbase + a.moff;
  switch (t.sel[s]) {
    S2DW_SEL(alpha_c2r_body_m, 5, 1, a, t.par[s], lds, bid, nb)
    S2DW_SEL(alpha_c2r_body_m, 6, 1, a, t.par[s], lds, bid, nb)
    S2DW_SEL(alpha_c2r_body_m, 7, 1, a, t.par[s], lds, bid, nb)
    S2DW_SEL(alpha_c2r_body_m, 8, 1, a, t.par[s], lds, bid, nb)
    S2DW_SEL(alpha_c2r_body_m, 9, 1, a, t.par[s], lds, bid, nb)
    S2DW_SEL(alpha_c2r_body_m, 10, 1, a, t.par[s], lds, bid, nb)
    S2DW_SEL(alpha_c2r_body_m, 11, 1, a, t.par[s], lds, bid, nb)
    default: alpha_c2r_body<0, -1, true>(a, t.par[s], lds, bid, nb); break;
  }
}

__global__ __launch_bounds__(kTN, 3) void k_alpha_syn_g(const SegTab t, const AlphaArgs *__restrict__ args,
                                                         const double *wbase) {
  __shared__ double2 lds[lpad_size(kTS)];
  const int s = seg_of(t, blockIdx.x), bid = blockIdx.x - t.first[s], nb = t.first[s + 1] - t.first[s];
  AlphaArgs a = args[s];
  a.W = const_cast<double *>(wbase) + a.woff;
  switch (t.sel[s]) {
#define S2DW_X(LM) \
  case 2 * (LM) + 1: alpha_syn_body<LM>(a, lds, bid, nb); break;
    S2DW_X(5) S2DW_X(6) S2DW_X(7) S2DW_X(8) S2DW_X(9) S2DW_X(10) S2DW_X(11)
#undef S2DW_X
    default: alpha_syn_body<0>(a, lds, bid, nb); break;
  }
}

__global__ __launch_bounds__(kTN, 3) void k_alpha_r2c_g(const SegTab t, const AlphaArgs *__restrict__ args,
                                                         const double *wbase) {
  __shared__ double2 lds[lpad_size(kTS)];
  const int s = seg_of(t, blockIdx.x), bid = blockIdx.x - t.first[s], nb = t.first[s + 1] - t.first[s];
  AlphaArgs a = args[s];
  a.W = const_cast<double *>(wbase) + a.woff;
  switch (t.sel[s]) {
    S2DW_SEL(alpha_r2c_body, 5, 1, a, t.par[s], lds, bid, nb)
    S2DW_SEL(alpha_r2c_body, 6, 1, a, t.par[s], lds, bid, nb)
    S2DW_SEL(alpha_r2c_body, 7, 1, a, t.par[s], lds, bid, nb)
    S2DW_SEL(alpha_r2c_body, 8, 1, a, t.par[s], lds, bid, nb)
    S2DW_SEL(alpha_r2c_body, 9, 1, a, t.par[s], lds, bid, nb)
    S2DW_SEL(alpha_r2c_body, 10, 1, a, t.par[s], lds, bid, nb)
    S2DW_SEL(alpha_r2c_body, 11, 1, a, t.par[s], lds, bid, nb)
    default: alpha_r2c_body<0, -1>(a, t.par[s], lds, bid, nb); break;
  }
}

__global__ __launch_bounds__(kTN, 3) void k_beta_syn_g(const SegTab t, const BetaSynArgs *__restrict__ args) {
  __shared__ double2 lds[lpad_size(kTS)];
  __shared__ double2 csum[kTN];
  const int s = seg_of(t, blockIdx.x), bid = blockIdx.x - t.first[s], nb = t.first[s + 1] - t.first[s];
  const BetaSynArgs &a = args[s];
  switch (t.sel[s]) {
    S2DW_SEL_H2_ALL(beta_syn_h2_body, a, a.V, a.Vt, a.tw8, t.par[s], lds, csum, bid, nb)
    default: beta_syn_body(a, a.V, a.Vt, a.tw8, t.par[s], lds, bid, nb); break;
  }
}
#undef S2DW_SEL
#undef S2DW_SEL16
#undef S2DW_SEL_H2
#undef S2DW_SEL_H2_ALL

// Static layout wav(0:J,0:2B-2,0:2B-1,0:N-1) (jj fastest) <-> packed scales.
// A workgroup covers 256 consecutive (jj, aa) entries of one row (b, g) of
// the static array, so every index is formed with 32-bit divisions (the
// linear index of the whole array needs 64 bits, whose divisions are
// emulated in software).
__global__ void k_pack_static(int Jp1, int B, int N, const int *__restrict__ his, const long long *__restrict__ offs,
                              const double *__restrict__ packed, double *__restrict__ stat, int to_static,
                              int nchunk) {
  const int row = (int)blockIdx.x / nchunk, chunk = (int)blockIdx.x - row * nchunk;  // row = b + 2B g
  const int per_row = Jp1 * (2 * B - 1);
  const int idr = chunk * 256 + (int)threadIdx.x;  // jj + Jp1 aa
  if (idr >= per_row) return;
  const int j = idr % Jp1, aa = idr / Jp1;
  const int b = row % (2 * B), g = row / (2 * B);
  const long long id = (long long)row * per_row + idr;
  const int hi = his[j];
  const bool in = aa < 2 * hi - 1 && b < 2 * hi;
  const long long pidx = offs[j] + aa + (long long)(2 * hi - 1) * (b + (long long)2 * hi * g);
  if (to_static) {
    stat[id] = in ? packed[pidx] : 0.0;
  } else if (in) {
    ((double *)packed)[pidx] = stat[id];
  }
}

// Diagnostic Wigner planes from the two device recursions.
__global__ void k_wigner_plane(int l, const double *__restrict__ S0, double *__restrict__ outA,
                               double *__restrict__ outS) {
  const int id = blockIdx.x * blockDim.x + threadIdx.x;
  const int n = l + 1;
  if (id < n * n && outA) {
    const int mp = id % n, m = id / n;
    const int l0 = mp > m ? mp : m;
    double d = lchain_start(S0, mp, m), dp = 0.0;
    const double md = m;
    double rm = sqrt((double)l0 * l0 - md * md);
    for (int k = l0; k < l; ++k) {
      double A, Bc;
      lrec_coefs(mp, k, &A, &Bc);
      const double a2 = (double)(k + 1) * (k + 1) - md * md;
      const double u = a2 > 0.5 ? rsqrt(a2) : 0.0;
      const double dn = u * (A * md * d + Bc * rm * dp);
      dp = d;
      d = dn;
      rm = a2 * u;
    }
    outA[mp + (long long)n * m] = d;
  }
  if (id < n && outS) {
    const int m = id;
    double d = S0[tri0(l) + m];
    if ((l - m) & 1) d = -d;
    double dn = 0.0;
    for (int mp = l; mp >= 0; --mp) {
      outS[mp + (long long)n * m] = d;
      double c1, c2;
      mrec_coefs(l, mp, &c1, &c2);
      const double nd = c1 * 2.0 * m * d - c2 * dn;
      dn = d;
      d = nd;
    }
  }
}

// ===========================================================================
// Host side: plan construction and stage drivers.
// ===========================================================================
namespace {

struct DevAlloc {
  Plan *p;
  template <class T>
  int alloc(T **ptr, size_t count) {
    void *q = nullptr;
    const size_t bytes = count * sizeof(T) > 0 ? count * sizeof(T) : 16;
    hipError_t e = hipMalloc(&q, bytes);
    if (e != hipSuccess) return hip_error(e, "hipMalloc");
    p->allocs.push_back(q);
    p->device_bytes += (long long)bytes;
    *ptr = static_cast<T *>(q);
    return kErrNone;
  }
};

int upload(void *dst, const void *src, size_t bytes, hipStream_t s) {
  S2DW_HIP_CHECK(hipMemcpyAsync(dst, src, bytes, hipMemcpyHostToDevice, s));
  return kErrNone;
}

// In-place radix-2 complex FFT in long double (host, plan time only).  Its n/2
// twiddles are computed once: with the cosine and sine of every butterfly in
// its place a plan that needs two filters of 2048 points takes 29.8 ms instead
// of 17.3 (L = 300, N = 8).
void host_fft_pow2(std::vector<std::complex<long double>> &x, int sign) {
  const size_t n = x.size();
  for (size_t i = 1, j = 0; i < n; ++i) {
    size_t bit = n >> 1;
    for (; j & bit; bit >>= 1) j ^= bit;
    j ^= bit;
    if (i < j) std::swap(x[i], x[j]);
  }
  const long double pi = 3.141592653589793238462643383279502884L;
  std::vector<std::complex<long double>> w(n / 2);
  for (size_t k = 0; k < n / 2; ++k) {
    const long double ang = sign * 2.0L * pi * (long double)k / (long double)n;
    w[k] = std::complex<long double>(cosl(ang), sinl(ang));
  }
  for (size_t len = 2; len <= n; len <<= 1) {
    for (size_t i = 0; i < n; i += len) {
      for (size_t k = 0; k < len / 2; ++k) {
        const auto u = x[i + k], v = x[i + k + len / 2] * w[k * (n / len)];
        x[i + k] = u + v;
        x[i + k + len / 2] = u - v;
      }
    }
  }
}

bool factor_smooth(int n, std::vector<int> &rad) {
  rad.clear();
  int m = n;
  while (m % 8 == 0) { rad.push_back(8); m /= 8; }
  while (m % 4 == 0) { rad.push_back(4); m /= 4; }
  while (m % 2 == 0) { rad.push_back(2); m /= 2; }
  for (int r : {7, 5, 3})
    while (m % r == 0) { rad.push_back(r); m /= r; }
  return m == 1 && (int)rad.size() <= kMaxStages;
}

// max_bluestein_M > 0: a length that is not a power of two runs through
// Bluestein whenever its work length is at most max_bluestein_M (so that it
// stays on the power-of-two workgroup engine), even if it is 7-smooth.
int make_fft(Plan *p, int n, FftSpec *out, int max_bluestein_M = 0) {
  DevAlloc da{p};
  FftSpec s{};
  s.n = n;
  std::vector<int> rad;
  const long double pi = 3.141592653589793238462643383279502884L;
  int Mb = 1;
  while (Mb < 2 * n - 1) Mb <<= 1;
  const bool pow2 = (n & (n - 1)) == 0;
  const bool force = !pow2 && max_bluestein_M > 0 && Mb <= max_bluestein_M;
  if (!force && factor_smooth(n, rad)) {
    s.M = n;
    s.bluestein = 0;
  } else {
    int M = 1;
    while (M < 2 * n - 1) M <<= 1;
    s.M = M;
    s.bluestein = 1;
    factor_smooth(M, rad);
  }
  s.nst = (int)rad.size();
  for (int i = 0; i < s.nst; ++i) s.radix[i] = rad[i];
  std::vector<double2> tw(s.M);
  for (int k = 0; k < s.M; ++k) {
    const long double a = 2.0L * pi * (long double)k / (long double)s.M;
    tw[k] = make_double2((double)cosl(a), (double)sinl(a));
  }
  double2 *dtw;
  if (int e = da.alloc(&dtw, tw.size())) return e;
  if (int e = upload(dtw, tw.data(), tw.size() * sizeof(double2), p->stream)) return e;
  s.tw = dtw;
  if (s.bluestein) {
    std::vector<std::complex<long double>> ch(n);
    std::vector<double2> chd(s.M, make_double2(0.0, 0.0));  // zero beyond n
    for (int k = 0; k < n; ++k) {
      const long long q = ((long long)k * k) % (2LL * n);
      const long double a = pi * (long double)q / (long double)n;
      ch[k] = std::complex<long double>(cosl(a), sinl(a));
      chd[k] = make_double2((double)ch[k].real(), (double)ch[k].imag());
    }
    std::vector<std::complex<long double>> hb(s.M, 0.0L), hf(s.M, 0.0L);
    for (int k = 0; k < n; ++k) {
      hb[k] = std::conj(ch[k]);
      hf[k] = ch[k];
      if (k > 0) {
        hb[s.M - k] = std::conj(ch[k]);
        hf[s.M - k] = ch[k];
      }
    }
    host_fft_pow2(hb, -1);
    host_fft_pow2(hf, -1);
    std::vector<double2> fb(s.M), ff(s.M);
    for (int k = 0; k < s.M; ++k) {
      fb[k] = make_double2((double)(hb[k].real() / s.M), (double)(hb[k].imag() / s.M));
      ff[k] = make_double2((double)(hf[k].real() / s.M), (double)(hf[k].imag() / s.M));
    }
    double2 *dch, *dfb, *dff;
    if (int e = da.alloc(&dch, s.M)) return e;
    if (int e = da.alloc(&dfb, s.M)) return e;
    if (int e = da.alloc(&dff, s.M)) return e;
    if (int e = upload(dch, chd.data(), s.M * sizeof(double2), p->stream)) return e;
    if (int e = upload(dfb, fb.data(), s.M * sizeof(double2), p->stream)) return e;
    if (int e = upload(dff, ff.data(), s.M * sizeof(double2), p->stream)) return e;
    s.chirp = dch;
    s.filt_b = dfb;
    s.filt_f = dff;
    // conj(chirp), zero beyond n: the post-multiplier of the forward direction
    std::vector<double2> chc(s.M, make_double2(0.0, 0.0));
    for (int k2 = 0; k2 < n; ++k2) chc[k2] = make_double2(chd[k2].x, -chd[k2].y);
    double2 *dchc;
    if (int e = da.alloc(&dchc, s.M)) return e;
    if (int e = upload(dchc, chc.data(), s.M * sizeof(double2), p->stream)) return e;
    s.chirp_c = dchc;
  }
  *out = s;
  return kErrNone;
}

// sequences per workgroup so that two LDS buffers fit in 64 KB
int fft_logT(const FftSpec &f, int cap) {
  int logT = 0;
  while ((2 * (f.M << (logT + 1))) * (int)sizeof(double2) <= 65536 && (1 << (logT + 1)) <= cap) ++logT;
  return logT;
}

size_t fft_lds(const FftSpec &f, int logT) { return 2 * ((size_t)f.M << logT) * sizeof(double2); }

// Wave-engine eligibility and launch shape for an FFT work length M.
struct WaveShape {
  bool ok;
  int E, logTw, WPB;
  size_t lds;
};
WaveShape wave_shape(const Plan *p, const FftSpec &f) {
  WaveShape w{false, 0, 0, 0, 0};
  const int M = f.M;
  if (p->fft_engine == 2 || M < 2 || (M & (M - 1)) || M > 2048) return w;
  w.E = M <= 1024 ? 16 : 32;
  int tw = 64 * w.E / M, lg = 0;
  while ((1 << lg) < tw) ++lg;
  w.logTw = lg;
  const size_t per_wave = (size_t)64 * w.E * sizeof(double2);
  int wpb = (int)(p->max_lds / per_wave);
  const int wpb_max = w.E == 16 ? 8 : 4;  // launch bounds of the E=16 / E=32 kernels
  if (wpb > wpb_max) wpb = wpb_max;
  if (wpb < 1) return w;
  w.WPB = wpb;
  w.lds = per_wave * wpb;
  w.ok = true;
  return w;
}

// Workgroup engine: power-of-two work length 2 <= M <= kTS (kTS/2 when the
// kernel holds both parities of a column); returns log2 of the sequences per
// workgroup, or -1.
int team_logTw(const Plan *p, const FftSpec &f, bool pairs) {
  if (p->fft_engine != 0) return -1;
  const int M = f.M;
  if (M < 2 || (M & (M - 1)) || M > (pairs ? kTS / 2 : kTS)) return -1;
  int lg = 0;
  while ((M << lg) < kTS) ++lg;
  return lg;
}

int log2_of(int M) { return 31 - __builtin_clz((unsigned)M); }

// Launch shape of a transform stage on the workgroup engine: work length
// 2^lg, sequences (columns or row pairs) per workgroup, and whether the
// one-FFT-per-column beta bodies run it.  lg < 0: the stage is not on the
// engine (another engine was asked for, or a smooth length above 2048 that
// runs directly).
struct TeamShape {
  int lg = -1, bl = 0, per = 0;
  bool h2 = false;
};

// beta: one FFT per column for every Bluestein length (M from 16 to 8192)
// and every power of two 2hi from 16 to kTS; the two-FFT bodies keep 2hi =
// 2, 4, 8 (fewer columns than the engine's minimum) and plans that ask for
// them.  Measured per full-band pair, synthesis: L = 397 (M = 2048) 52 us
// against 492 us for two FFTs per column on the wave engine, L = 899
// (M = 4096) 370 us against 2983 us on the two-buffer generic kernel;
// analysis L = 1024 (2048 points, direct) 488 us against 1434 us.  The alpha
// stage on M = 4096 in place: L = 1024 853 us against 1932 us (generic).
TeamShape beta_shape(const Plan *p, const FftSpec &f, int hi) {
  TeamShape r;
  if (p->fft_engine != 0 || f.M < 2 || (f.M & (f.M - 1))) return r;
  const int lg = log2_of(f.M);
  r.bl = f.bluestein ? 1 : 0;
  if ((p->beta_one || lg > kLogTS) && lg >= 4 && (f.bluestein ? lg <= kBigLogM && lds_of(lg) + kCsumLds <= p->max_lds : lg <= kLogTS)) {
    r.lg = lg;
    r.per = std::max(1, kTS >> lg);
    r.h2 = true;
    return r;
  }
  const int tl = team_logTw(p, f, true);
  if (tl >= 0) {
    r.lg = lg;
    r.per = 1 << (tl - 1);
  }
  return r;
}

TeamShape alpha_shape(const Plan *p, const FftSpec &f) {
  TeamShape r;
  if (p->fft_engine != 0 || f.M < 2 || (f.M & (f.M - 1))) return r;
  const int lg = log2_of(f.M);
  if (lg > kLogTS && !(f.bluestein && lg <= kBigLogM && lds_of(lg) <= p->max_lds)) return r;
  r.lg = lg;
  r.bl = f.bluestein ? 1 : 0;
  r.per = std::max(1, kTS >> lg);
  return r;
}

// Launches of one scale (second set equal to the first, half = all
// workgroups) or of the full-band pair.  The kernels are specialised on the
// work length (compile-time M folds the engine's LDS addressing into
// immediate offsets) and on Bluestein vs direct; lengths below 32 (alpha)
// run the generic instantiation <0, -1>, which reads both from the FftSpec.
// Lengths of one sequence per workgroup up to 4096 slots (M = 2048: M/16 = 128
// threads; M = 4096: 256) run on the three-stage engine.
#define S2DW_ALPHA_CASE16(KERN, LM, ...)                                                                       \
  case LM:                                                                                                     \
    hipLaunchKernelGGL((KERN), g, dim3((1 << LM) / 16), lds16_of(LM), st, a0, a1, __VA_ARGS__);                \
    break;
#define S2DW_ALPHA_CASE(KERN, LM)                                                                              \
  case LM:                                                                                                     \
    hipLaunchKernelGGL((KERN<LM, 1>), g, dim3(nt_of(LM)), lds_of(LM), st, a0, a1, npt, half);                  \
    break;
#define S2DW_ALPHA_LAUNCH(NAME, KERN, ...)                                                                     \
  void NAME(const TeamShape &t, const AlphaArgs &a0, const AlphaArgs &a1, int npt, int half, int blocks,       \
            hipStream_t st) {                                                                                  \
    const dim3 g(blocks);                                                                                      \
    switch (t.bl ? t.lg : 0) {                                                                                 \
      S2DW_ALPHA_CASE(KERN, 5) S2DW_ALPHA_CASE(KERN, 6) S2DW_ALPHA_CASE(KERN, 7) S2DW_ALPHA_CASE(KERN, 8)      \
      S2DW_ALPHA_CASE(KERN, 9) S2DW_ALPHA_CASE(KERN, 10) __VA_ARGS__ S2DW_ALPHA_CASE(KERN, 13)                 \
      default: hipLaunchKernelGGL((KERN<0, -1>), g, dim3(kTN), 0, st, a0, a1, npt, half); break;               \
    }                                                                                                          \
  }
#define S2DW_C(...) __VA_ARGS__
constexpr int lds16_of(int lg) { return lpad16(1 << lg) * (int)sizeof(double); }
S2DW_ALPHA_LAUNCH(launch_alpha_c2r, k_alpha_c2r_t2, S2DW_ALPHA_CASE16(S2DW_C(k_alpha_c2r16<11, false>), 11, npt, half)
                  S2DW_ALPHA_CASE16(S2DW_C(k_alpha_c2r16<12, false>), 12, npt, half))
S2DW_ALPHA_LAUNCH(launch_alpha_c2r_mom, k_alpha_c2r_t2m,
                  S2DW_ALPHA_CASE16(S2DW_C(k_alpha_c2r16<11, true>), 11, npt, half)
                  S2DW_ALPHA_CASE16(S2DW_C(k_alpha_c2r16<12, true>), 12, npt, half))
S2DW_ALPHA_LAUNCH(launch_alpha_syn, k_alpha_syn_t2, S2DW_ALPHA_CASE16(k_alpha_syn16<11>, 11, half)
                  S2DW_ALPHA_CASE16(k_alpha_syn16<12>, 12, half))
#undef S2DW_C
#undef S2DW_ALPHA_CASE16
#undef S2DW_ALPHA_LAUNCH
#undef S2DW_ALPHA_CASE

#define S2DW_H2_CASES(X) \
  X(4, 0) X(5, 0) X(6, 0) X(7, 0) X(8, 0) X(9, 0) X(10, 0) X(11, 0) X(4, 1) X(5, 1) X(6, 1) X(7, 1) X(8, 1) X(9, 1) \
  X(10, 1) X(13, 1)
void launch_beta_ana(const TeamShape &t, const BetaAnaArgs &b0, const BetaAnaArgs &b1, int nmt, int half, int blocks,
                     hipStream_t st) {
  const dim3 g(blocks);
  switch (t.h2 ? 2 * t.lg + t.bl : 0) {
#define S2DW_X(LM, B)                                                                                               \
  case 2 * (LM) + (B):                                                                                              \
    hipLaunchKernelGGL((k_beta_ana_h2<LM, (B) != 0>), g, dim3(nt_of(LM)), lds_of(LM), st, b0, b1, nmt, half);       \
    break;
    S2DW_H2_CASES(S2DW_X)
#undef S2DW_X
    case 2 * 11 + 1:
      hipLaunchKernelGGL((k_beta_ana16<11>), g, dim3(128), lds16_of(11), st, b0, b1, nmt, half);
      break;
    case 2 * 12 + 1:
      hipLaunchKernelGGL((k_beta_ana16<12>), g, dim3(256), lds16_of(12), st, b0, b1, nmt, half);
      break;
    default: hipLaunchKernelGGL(k_beta_ana_t2, g, dim3(kTN), 0, st, b0, b1, nmt, half); break;
  }
}
void launch_beta_syn(const TeamShape &t, const BetaSynArgs &y0, const BetaSynArgs &y1, int nmt, int half, int blocks,
                     hipStream_t st) {
  const dim3 g(blocks);
  switch (t.h2 ? 2 * t.lg + t.bl : 0) {
#define S2DW_X(LM, B)                                                                                                 \
  case 2 * (LM) + (B):                                                                                                \
    hipLaunchKernelGGL((k_beta_syn_h2<LM, (B) != 0>), g, dim3(nt_of(LM)), lds_of(LM), st, y0, y1.V, y1.Vt, y1.tw8, nmt, \
                       half);                                                                                         \
    break;
    S2DW_H2_CASES(S2DW_X)
#undef S2DW_X
    case 2 * 11 + 1:
      hipLaunchKernelGGL((k_beta_syn16<11>), g, dim3(128), lds16_of(11), st, y0, y1.V, y1.Vt, y1.tw8, nmt, half);
      break;
    case 2 * 12 + 1:
      hipLaunchKernelGGL((k_beta_syn16<12>), g, dim3(256), lds16_of(12), st, y0, y1.V, y1.Vt, y1.tw8, nmt, half);
      break;
    default: hipLaunchKernelGGL(k_beta_syn_t2, g, dim3(kTN), 0, st, y0, y1.V, y1.Vt, y1.tw8, nmt, half); break;
  }
}
#undef S2DW_H2_CASES
// packed real rows without the gamma-DFT
void launch_alpha_r2c(const TeamShape &t, const AlphaArgs &a0, const AlphaArgs &a1, int npt, int half, int blocks,
                      hipStream_t st) {
  const dim3 g(blocks);
  switch (t.bl ? t.lg : 0) {
#define S2DW_X(LM)                                                                                        \
  case LM:                                                                                                \
    hipLaunchKernelGGL((k_alpha_r2c_t2<LM, 1>), g, dim3(nt_of(LM)), lds_of(LM), st, a0, a1, npt, half);   \
    break;
    S2DW_X(5) S2DW_X(6) S2DW_X(7) S2DW_X(8) S2DW_X(9) S2DW_X(10) S2DW_X(13)
#undef S2DW_X
    case 11: hipLaunchKernelGGL((k_alpha_r2c16<11>), g, dim3(128), lds16_of(11), st, a0, a1, half); break;
    case 12: hipLaunchKernelGGL((k_alpha_r2c16<12>), g, dim3(256), lds16_of(12), st, a0, a1, half); break;
    default: hipLaunchKernelGGL((k_alpha_r2c_t2<0, -1>), g, dim3(kTN), 0, st, a0, a1, npt, half); break;
  }
}

void add_gamma(const Plan *p, GammaTab &t, int j) {
  const Scale &s = p->sc[j];
  t.first[t.nseg + 1] = t.first[t.nseg] + (int)((2LL * s.hi * s.hi + 255) / 256);
  t.g[t.nseg++] = GammaSeg{p->d_tb + s.tb_off, p->d_wq + p->wq_off[j], s.hi};
}
void launch_gamma_syn(const Plan *p, const GammaTab &t, hipStream_t st) {
  const int N = p->N, nn = (int)p->nlist.size();
  const dim3 g(t.first[t.nseg]);
  if (N <= 8) hipLaunchKernelGGL(k_gamma_syn<8>, g, dim3(256), 0, st, t, N, nn, p->eg);
  else if (N <= 16) hipLaunchKernelGGL(k_gamma_syn<16>, g, dim3(256), 0, st, t, N, nn, p->eg);
  else hipLaunchKernelGGL(k_gamma_syn<32>, g, dim3(256), 0, st, t, N, nn, p->eg);
}

// Whether the synthesis of a scale takes the gamma-DFT before the alpha
// transform (alpha_syn_body) where both its FFT stages are on the workgroup
// engine; a grouped launch takes the form of its largest scale.  The gather
// reads every wavelet row once per n, N^2/2 reads per row pair, the pass on
// its own moves N planes of f64 pairs twice.  FFT stages of a synthesis, us, before /
// on its own: L = 128, N = 32 99 / 115; L = 256, N = 12 101 / 105, 16 133 / 130,
// 32 347 / 310; L = 300, N = 12 189 / 187, 16 275 / 254, 32 717 / 582; L = 700,
// N = 16 1296 / 1186; L = 512, N = 16 386 / 394, 20 522 / 518, 32 1043 / 909;
// L = 1024, N = 16 1821 / 1849.  Scales of hi = 150 are even at N = 32.
// Between 1.8 and 2.4 million N hi^2 the N planes of the pass on its own (60 to
// 77 MB a scale) push the contraction's input out of the last-level cache and
// the N/2 of the other do not: whole synthesis, us, L = 240, N = 32 1914 /
// 2220, L = 256, N = 28 1837 / 2132; beyond, L = 300, N = 28 2687 / 2535.
bool gamma_first(const Plan *p, int hi) {
  const bool pow2 = hi > 256 && (hi & (hi - 1)) == 0;
  const double planes = (double)p->N * hi * hi;
  return hi < 200 || p->N < (pow2 ? 20 : 16) || (planes > 1.82e6 && planes < 2.4e6);
}

}  // namespace

namespace {
int build_groups(Plan *p);
void free_groups(Plan *p);
}  // namespace

void plan_free(Plan *p) {
  free_groups(p);
  refbeta_free(p);
  for (auto &e : p->ev_live) {
    (void)hipEventDestroy(e.a);
    (void)hipEventDestroy(e.b);
  }
  for (hipEvent_t e : p->ev_pool) (void)hipEventDestroy(e);
  p->ev_live.clear();
  p->ev_pool.clear();
  for (void *q : p->allocs) (void)hipFree(q);
  p->allocs.clear();
  if (p->own_stream && p->stream) (void)hipStreamDestroy(p->stream);
  p->stream = nullptr;
  plan_drop_graphs(p);
  if (p->cap) (void)hipStreamDestroy(p->cap);
  p->cap = nullptr;
  if (p->aux) (void)hipStreamDestroy(p->aux);
  if (p->fork) (void)hipEventDestroy(p->fork);
  if (p->join) (void)hipEventDestroy(p->join);
  p->aux = nullptr;
  p->fork = p->join = nullptr;
}

int plan_build(Plan *p, int B, int N, int J, double alpha, const double *K, const double *Phi2, const double *S,
               int precision, hipStream_t stream, bool own_stream) {
  if (B < 1 || N < 1 || N > B || !params_valid(J, B, alpha, N)) {
    set_error("invalid sizes B=%d N=%d J=%d alpha=%g", B, N, J, alpha);
    return kErrSizeInvalid;
  }
  if (J + 1 > kMaxSc) {
    set_error("J=%d exceeds the supported %d scales", J, kMaxSc - 1);
    return kErrSizeInvalid;
  }
  p->B = B;
  p->N = N;
  p->J = J;
  p->alpha = alpha;
  p->precision = precision & 0xF;
  // S2DW_WIGNER_TABLE (16): reference-rounding Wigner planes; S2DW_ROUNDING_REFERENCE
  // (48): the planes plus the reference's rounded phase factors and beta-sum basis
  const bool want_ref = (precision & 0x20) != 0;
  const bool want_table = want_ref || (precision & 0x10) != 0;
  // kernel choice for the analysis contraction: MFMA unless S2DW_HIP_ANA_KERNEL=valu
  if (const char *ev = std::getenv("S2DW_HIP_ANA_KERNEL")) p->ana_mfma = std::strcmp(ev, "valu") != 0;
  if (B > 1024) p->ana_mfma = false;  // the MFMA kernel keeps 4 coefficient rows of B pairs in LDS
  if (N > kAnaMaxN) p->ana_mfma = false;  // and the gamma matrix chunk, N x 8
  if (const char *ev = std::getenv("S2DW_HIP_ANA_MFMA")) p->ana_wave_indep = std::strcmp(ev, "staged") != 0;
  p->ana_mfma_ok = p->ana_mfma;
  if (const char *ev = std::getenv("S2DW_HIP_SYN_KERNEL")) p->syn_mfma = std::strcmp(ev, "valu") != 0;
  if (const char *ev = std::getenv("S2DW_HIP_SYN_MFMA")) p->syn_wave = std::strcmp(ev, "staged") != 0;
  // FFT engine for the beta/alpha stages: workgroup (default), wave, generic
  if (const char *ev = std::getenv("S2DW_HIP_FFT")) p->fft_engine = !std::strcmp(ev, "wave") ? 1 : !std::strcmp(ev, "generic") ? 2 : 0;
  if (const char *ev = std::getenv("S2DW_HIP_ODD_FFT")) p->odd_alpha = std::strcmp(ev, "0") != 0;
  if (const char *ev = std::getenv("S2DW_HIP_BETA_ONE")) p->beta_one = std::strcmp(ev, "0") != 0;
  if (const char *ev = std::getenv("S2DW_HIP_SYN_CW")) p->syn_cw_min = std::max(4, std::min(64, std::atoi(ev)));
  // plans up to B = 256 keep every launch on one stream, with every scale in
  // the grouped FFT launches: the helper stream's fork and join cost more
  // than the overlap gains there (B = 256: 96 us per transform against 106
  // eager and 100 replayed on two streams); S2DW_HIP_STREAMS=1|2 forces either
  p->single_stream = B <= 256;
  if (const char *ev = std::getenv("S2DW_HIP_STREAMS")) p->single_stream = std::strcmp(ev, "1") == 0;
  if (const char *ev = std::getenv("S2DW_HIP_SYN_XCD")) p->syn_xcd = std::strcmp(ev, "0") != 0;
  S2DW_HIP_CHECK(hipGetDevice(&p->device));
  if (own_stream) {
    S2DW_HIP_CHECK(hipStreamCreateWithFlags(&p->stream, hipStreamNonBlocking));
    p->own_stream = true;
  } else {
    p->stream = stream;  // NULL is the device's null stream
  }
  // default-priority helper stream and fork/join events (no timing)
  S2DW_HIP_CHECK(hipStreamCreateWithFlags(&p->aux, hipStreamNonBlocking));
  S2DW_HIP_CHECK(hipEventCreateWithFlags(&p->fork, hipEventDisableTiming));
  S2DW_HIP_CHECK(hipEventCreateWithFlags(&p->join, hipEventDisableTiming));
  const int L = B;
  const int Jp1 = J + 1;
  p->K.assign(K, K + (size_t)Jp1 * L);
  p->Phi2.assign(Phi2, Phi2 + L);
  p->S.assign(S, S + 2 * (size_t)L * N);
  // bl_scoeff: band limit of scale J+1, s2dw_core_mod.f90:116-152
  {
    int bw;
    const double xb = B / powi(alpha, J);
    if (!assimilate_int(xb, &bw)) bw = (int)std::ceil(xb);
    p->bl_scoeff = bw;
  }
  // scales
  p->sc.assign(Jp1, Scale{});
  // the contraction buffer starts with 4 zero entries: the synthesis
  // contraction reads out-of-range elements from index 0
  long long woff = 0, tgoff = 4, tboff = 0;
  for (int j = 0; j < Jp1; ++j) {
    Scale &s = p->sc[j];
    band_limits(j, B, alpha, &s.hi, &s.lo);
    s.wav_off = woff;
    woff += (long long)(2 * s.hi - 1) * 2 * s.hi * N;
  }
  p->wav_doubles = woff;
  // columns
  auto Spart = [&](int l, int n, int part) { return S[2 * ((size_t)l + (size_t)L * n) + part]; };
  p->cols_a.clear();
  p->cols_s.clear();
  for (int n = -(N - 1); n <= N - 1; ++n) {
    if (((N + n) % 2 + 2) % 2 == 0) continue;
    const int an = n < 0 ? -n : n;
    for (int part = 0; part < 2; ++part) {
      bool nz = false;
      for (int l = 0; l < L && !nz; ++l) nz = Spart(l, an, part) != 0.0;
      if (nz) {
        p->cols_a.push_back({n, part});
        if (n >= 0) p->cols_s.push_back({n, part});
      }
    }
  }
  const int NCa = (int)p->cols_a.size(), NCs = (int)p->cols_s.size();
  if (NCa > kMaxCol || NCs > kMaxCol) {
    set_error("N=%d gives %d columns, more than the supported %d", N, NCa, kMaxCol);
    return kErrSizeInvalid;
  }
  int nk = 1;
  for (auto &c : p->cols_a) nk = std::max(nk, (c.n < 0 ? -c.n : c.n) + 1);
  p->nk = nk;
  // table form: the MFMA contraction kernels with independent waves read the
  // Wigner values from reference-rounding planes (N <= 8 analysis columns;
  // the table's byte offsets must stay below 2^32)
  const bool split = p->precision == 1;  // S2DW_PREC_SPLIT: the split kernel reads the Wigner table
  if (split && !(p->ana_mfma && NCa <= kChunk && ref_plane_doubles(L) * 8 < 0xFFFF0000LL)) {
    set_error("the split-precision contraction needs N <= 8 (at most 8 analysis columns) and B <= 1024");
    return kErrArgInvalid;
  }
  const bool use_table = (want_table || split) && p->ana_mfma && NCa <= kChunk && (p->syn_mfma || split) &&
                         ref_plane_doubles(L) * 8 < 0xFFFF0000LL;
  // per-l active slots and flushes (non-empty scales only)
  std::vector<int> slotj(2 * L, -1);
  std::vector<int2> lflush(L, make_int2(-1, -1));
  std::vector<unsigned char> covered(L, 0);
  for (int j = 0; j < Jp1; ++j) {
    const Scale &s = p->sc[j];
    if (s.lo + 1 > s.hi - 1) continue;
    for (int l = s.lo + 1; l <= s.hi - 1; ++l) {
      if (slotj[2 * l + (j & 1)] != -1) {
        set_error("internal: two scales in one slot at l=%d", l);
        return kErrInitFail;
      }
      slotj[2 * l + (j & 1)] = j;
      covered[l] = 1;
    }
    if (j & 1) lflush[s.hi - 1].y = j;
    else lflush[s.hi - 1].x = j;
  }
  // device allocations
  DevAlloc da{p};
  const int NCmax = std::max(N, NCs);
  for (int j = 0; j < Jp1; ++j) {
    Scale &s = p->sc[j];
    s.tg_off = tgoff;
    tgoff += (long long)NCmax * s.hi * s.hi;
    s.tb_off = tboff;
    tboff += (long long)N * 2 * s.hi * s.hi;
  }
  if (int e = da.alloc(&p->d_fT, (size_t)L * L)) return e;
  if (int e = da.alloc(&p->d_fo, (size_t)L * L)) return e;
  if (int e = da.alloc(&p->d_tg, (size_t)tgoff)) return e;
  p->tg_doubles = 2 * tgoff;
  S2DW_HIP_CHECK(hipMemsetAsync(p->d_tg, 0, 4 * sizeof(double2), p->stream));
  if (int e = da.alloc(&p->d_tb, (size_t)tboff)) return e;
  // chain start values S0[l0][k] = sqrt(C(2 l0, l0+k)) / 2^l0
  {
    std::vector<double> s0(tri0(L));
    for (int l0 = 0; l0 < L; ++l0) {
      const long double lg2l = lgammal(2.0L * l0 + 1.0L);
      for (int k = 0; k <= l0; ++k) {
        const long double lv =
            0.5L * (lg2l - lgammal((long double)(l0 + k) + 1.0L) - lgammal((long double)(l0 - k) + 1.0L)) -
            (long double)l0 * logl(2.0L);
        s0[tri0(l0) + k] = (double)expl(lv);
      }
    }
    if (int e = da.alloc(&p->d_S0, s0.size())) return e;
    if (int e = upload(p->d_S0, s0.data(), s0.size() * sizeof(double), p->stream)) return e;
  }
  // S parts and K on device
  std::vector<double> sA((size_t)L * NCa), sS((size_t)L * NCs);
  const long double pi = 3.141592653589793238462643383279502884L;
  for (int l = 0; l < L; ++l) {
    for (int c = 0; c < NCa; ++c) {
      const int n = p->cols_a[c].n, part = p->cols_a[c].part, an = n < 0 ? -n : n;
      double v = Spart(l, an, part);
      if (n >= 0) {
        if (part == 1) v = -v;  // conj(S)
      } else if (an & 1) {
        v = -v;  // (-1)^n S(l,|n|)
      }
      sA[(size_t)l * NCa + c] = v;
    }
    for (int c = 0; c < NCs; ++c) {
      const int n = p->cols_s[c].n, part = p->cols_s[c].part;
      const double eps = n == 0 ? 1.0 : 2.0;
      sS[(size_t)l * NCs + c] = eps * ((double)(2.0 * l + 1) / (8.0 * (double)(pi * pi))) * Spart(l, n, part);
    }
  }
  double *d_sA, *d_sS, *d_K;
  int *d_slotj;
  if (int e = da.alloc(&d_sA, sA.size())) return e;
  if (int e = da.alloc(&d_sS, sS.size())) return e;
  if (int e = da.alloc(&d_K, p->K.size())) return e;
  if (int e = da.alloc(&d_slotj, slotj.size())) return e;
  // per aligned group of 4 l: bit k set when a scale ends at 4q + k
  std::vector<int> gev((L + 3) / 4 + 1, 0);
  for (int l = 0; l < L; ++l)
    if (lflush[l].x >= 0 || lflush[l].y >= 0) gev[l >> 2] |= 1 << (l & 3);
  if (int e = da.alloc(&p->d_lmeta, 2 * (size_t)L + gev.size())) return e;
  p->d_gev = p->d_lmeta + 2 * (size_t)L;
  unsigned char *d_cov;
  if (int e = da.alloc(&d_cov, (size_t)L)) return e;
  p->d_wq_off = nullptr;
  if (int e = upload(d_sA, sA.data(), sA.size() * sizeof(double), p->stream)) return e;
  if (int e = upload(d_sS, sS.data(), sS.size() * sizeof(double), p->stream)) return e;
  if (int e = upload(d_K, p->K.data(), p->K.size() * sizeof(double), p->stream)) return e;
  if (int e = upload(d_slotj, slotj.data(), slotj.size() * sizeof(int), p->stream)) return e;
  if (int e = upload(p->d_lmeta, lflush.data(), lflush.size() * sizeof(int2), p->stream)) return e;
  if (int e = upload(p->d_gev, gev.data(), gev.size() * sizeof(int), p->stream)) return e;
  if (int e = upload(d_cov, covered.data(), covered.size(), p->stream)) return e;
  // thin chains and rows
  const long long nrows = tri0(L);
  if (int e = da.alloc(&p->d_thin, (size_t)nrows * nk)) return e;
  if (int e = da.alloc(&p->d_Ba, (size_t)nrows * (2 + 2 * NCa))) return e;
  p->ba_bytes = (long long)nrows * (2 + 2 * NCa) * (long long)sizeof(double);
  if (int e = da.alloc(&p->d_lcoef, (size_t)L * (L + 4) * 2)) return e;
  {
    const long long n = (long long)L * (L + 4);
    hipLaunchKernelGGL(k_lcoef, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, p->stream, L, p->d_lcoef);
    S2DW_HIP_CHECK(hipGetLastError());
  }
  if (int e = da.alloc(&p->d_uinv, (size_t)L * L)) return e;
  {
    const long long n = (long long)L * L;
    hipLaunchKernelGGL(k_uinv, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, p->stream, L, p->d_uinv);
    S2DW_HIP_CHECK(hipGetLastError());
  }
  if (int e = da.alloc(&p->d_Bs, (size_t)nrows * (2 + 2 * NCs))) return e;
  if (use_table) {
    p->sa_doubles = ref_plane_doubles(L);
    if (int e = da.alloc(&p->d_Sa, (size_t)p->sa_doubles)) return e;
    if (int e = da.alloc(&p->d_thinneg, (size_t)nrows * nk)) return e;
    if (int e = build_ref_planes(L, nk, p->d_Sa, p->d_thin, p->d_thinneg, p->stream)) return e;
    p->refround = want_ref;
    p->tab_syn = want_table;  // the split form alone keeps the streamed synthesis
  }
  {
    const int nth = L * nk;
    if (!use_table)
      hipLaunchKernelGGL(k_thin_chains, dim3((nth + 127) / 128), dim3(128), 0, p->stream, L, nk, p->d_S0, p->d_thin);
    S2DW_HIP_CHECK(hipGetLastError());
    RowArgs ra{};
    ra.L = L;
    ra.nk = nk;
    ra.NCa = NCa;
    ra.NCs = NCs;
    ra.nsc = Jp1;
    ra.thin = p->d_thin;
    ra.thinneg = p->d_thinneg;
    ra.K = d_K;
    ra.sA = d_sA;
    ra.sS = d_sS;
    ra.slotj = d_slotj;
    for (int c = 0; c < NCa; ++c) ra.colA_n[c] = p->cols_a[c].n;
    for (int c = 0; c < NCs; ++c) ra.colS_n[c] = p->cols_s[c].n;
    ra.Jp1 = Jp1;
    ra.Ba = p->d_Ba;
    ra.Bs = p->d_Bs;
    hipLaunchKernelGGL(k_build_rows, dim3((unsigned)((nrows + 255) / 256)), dim3(256), 0, p->stream, ra);
    S2DW_HIP_CHECK(hipGetLastError());
  }
  // contraction by parity of l (s2dw_anapar.hip): the streamed form with one
  // real column per n (S all real or all imaginary, so that T_{-n} follows
  // from T_n; an imaginary S(l,0) breaks the symmetry) and at most 4 columns
  // n >= 0.  S2DW_HIP_ANA_KERNEL / S2DW_HIP_ANA_MFMA select another kernel.
  if (!use_table && !split && NCa > 0) {
    const int part = p->cols_a[0].part;
    bool ok = NCa <= 8;
    int nh = 0;
    for (const Column &c : p->cols_a) {
      ok = ok && c.part == part && !(c.n == 0 && part == 1);
      nh += c.n >= 0;
    }
    ok = ok && nh <= 4 && N / 2 <= nh && 16LL * (L + 16) * L <= kBufMaxBytes &&
         nrows * (2 + 2 * nh) * 8 + 4096 <= kBufMaxBytes;
    if (ok) {
      p->rows_bytes = nrows * (2 + 2 * nh) * (long long)sizeof(double);
      p->ana_nh = nh;
      p->ana_urot = part;
      p->ana_par = !std::getenv("S2DW_HIP_ANA_KERNEL") && !std::getenv("S2DW_HIP_ANA_MFMA");
      if (int e = da.alloc(&p->d_rows, (size_t)nrows * (2 + 2 * nh))) return e;
      if (int e = par_rows(nrows, NCa, nh, NCa - nh, p->d_Ba, p->d_rows, p->stream)) return e;
      // H(g, n) = i^n e^{i n pi g / N}: twice its real and imaginary part for
      // n > 0 (the columns n and -n together), 1 and 0 for n = 0; the two
      // orders put the real parts on the even-l or the odd-l sums
      std::vector<double> cg((size_t)2 * (nh + 1) * 2 * nh, 0.0);
      for (int g = 0; g <= nh; ++g)
        for (int h = 0; h < nh; ++h) {
          const int n = p->cols_a[NCa - nh + h].n;
          const long double ang = pi * (long double)n * (0.5L + (long double)g / (long double)N);
          const double cr = n == 0 ? 1.0 : (double)(2.0L * cosl(ang)), ci = n == 0 ? 0.0 : (double)(2.0L * sinl(ang));
          double *c0 = cg.data() + (size_t)g * 2 * nh + h, *c1 = c0 + (size_t)(nh + 1) * 2 * nh;
          c0[0] = c1[nh] = cr;
          c0[nh] = c1[0] = ci;
        }
      if (int e = da.alloc(&p->d_cg, cg.size())) return e;
      if (int e = upload(p->d_cg, cg.data(), cg.size() * sizeof(double), p->stream)) return e;
      const int WV = kParWv, G = kParG, ngr = (L + G - 1) / G;
      std::vector<int> ends((size_t)8 * L + 2 * (size_t)ngr, 0);
      int *pev = ends.data() + 8 * (size_t)L, *pnx = pev + ngr;
      for (int l = 0; l < L; ++l)
        for (int sl = 0; sl < 2; ++sl) {
          const int j = sl ? lflush[l].y : lflush[l].x;
          if (j < 0) continue;
          ends[8 * (size_t)l + sl] = p->sc[j].hi;
          ends[8 * (size_t)l + 2 + 2 * sl] = (int)(unsigned)p->sc[j].tg_off;
          ends[8 * (size_t)l + 3 + 2 * sl] = (int)(p->sc[j].tg_off >> 32);
          pev[l / G] |= 1 << (l % G);
        }
      for (int q = ngr - 1; q >= 0; --q) pnx[q] = pev[q] ? G * q : q + 1 < ngr ? pnx[q + 1] : G * ngr;
      // work list (WV m' x 64 m, L - max(m', m) values of l).  Workgroup i runs
      // on XCD i % 8 and, while the grid is resident, on CU (i / 8) % 32 of
      // it: every m-tile of an m'-block goes to one XCD, whose L2 then holds
      // the block's rows; there longest first, every second run of 32
      // reversed, so that a CU gets long and short ones
      std::vector<int> cls[8], wk;
      for (int y = 0; 64 * y < L; ++y)
        for (int x = 0; WV * x < L; ++x) cls[x % 8].push_back(x | y << 16);
      size_t pos[8] = {0};
      for (auto &c : cls) {
        std::stable_sort(c.begin(), c.end(), [WV](int u, int v) {
          return std::max(WV * (u & 0xffff), 64 * (u >> 16)) < std::max(WV * (v & 0xffff), 64 * (v >> 16));
        });
        for (size_t i = 32; i < c.size(); i += 64)
          std::reverse(c.begin() + (long)i, c.begin() + (long)std::min(i + 32, c.size()));
      }
      const size_t nwk = (size_t)((L + WV - 1) / WV) * ((L + 63) / 64);
      for (size_t i = 0; wk.size() < nwk; ++i) {
        int k = (int)(i % 8);
        if (pos[k] >= cls[k].size())  // this class is used up: the fullest one
          for (int q = 0; q < 8; ++q)
            if (cls[q].size() - pos[q] > cls[k].size() - pos[k]) k = q;
        wk.push_back(cls[k][pos[k]++]);
      }
      if (int e = da.alloc(&p->d_ends, ends.size())) return e;
      p->d_pgev = p->d_ends + 8 * (size_t)L;
      p->d_pgnext = p->d_pgev + ngr;
      if (int e = upload(p->d_ends, ends.data(), ends.size() * sizeof(int), p->stream)) return e;
      if (int e = da.alloc(&p->d_awork, wk.size())) return e;
      if (int e = upload(p->d_awork, wk.data(), wk.size() * sizeof(int), p->stream)) return e;
      S2DW_HIP_CHECK(hipStreamSynchronize(p->stream));  // the vectors are locals
    }
  }
  if (split) {
    if (int e = da.alloc(&p->d_Bq, (size_t)nrows * 16)) return e;
    p->bq_bytes = (long long)nrows * 16 * (long long)sizeof(uint4);
    if (int e = da.alloc(&p->d_erow, (size_t)L)) return e;
    hipLaunchKernelGGL(k_build_bq<kSplitD>, dim3((unsigned)((nrows * 16 + 255) / 256)), dim3(256), 0, p->stream,
                       nrows, NCa, p->d_Ba, p->d_Bq);
    S2DW_HIP_CHECK(hipGetLastError());
  }
  // synthesis l-blocks: segments of constant active-scale set, Q per block
  {
    std::vector<int4> blocks;
    const int Q = p->syn_q;
    int l = 0;
    while (l < L) {
      if (!covered[l]) {
        ++l;
        continue;
      }
      int e = l;
      while (e + 1 < L && covered[e + 1] && slotj[2 * (e + 1)] == slotj[2 * l] &&
             slotj[2 * (e + 1) + 1] == slotj[2 * l + 1])
        ++e;
      for (int b = l; b <= e; b += Q) blocks.push_back(make_int4(b, std::min(Q, e - b + 1), slotj[2 * l], slotj[2 * l + 1]));
      l = e + 1;
    }
    std::sort(blocks.begin(), blocks.end(), [](const int4 &x, const int4 &y) { return x.x + x.y > y.x + y.y; });
    p->n_sblk = (int)blocks.size();
    if (int e = da.alloc(&p->d_sblk, blocks.size())) return e;
    if (int e = upload(p->d_sblk, blocks.data(), blocks.size() * sizeof(int4), p->stream)) return e;
  }
  // MFMA synthesis: per-scale B tables, m'-recursion coefficients,
  // checkpoint planes, chunk partials and the work list
  if (p->syn_mfma && NCs > 0) {
    const int NCp = (NCs + 3) & ~3;
    // m' chunk width L/16, at least 4: 16 chunks of work items at every band
    // limit (small plans get as many workgroups per l-block as large ones, and
    // the tiles of the lowest l, a few workgroups whose steps wait on memory,
    // stay short).  Synthesis at widths 16, 20, 25, 32, 40 of L = 397: 206, 203,
    // 200, 205, 213 us; 16, 24, 32, 36 of L = 512: 242, 233, 230, 229 us;
    // 2, 3, 4, 6, 8 of L = 64: 35, 33, 32, 32, 33 us.
    const int CW = std::max(p->syn_cw_min, (L + 15) / 16);
    const int nch = (L + CW - 1) / CW;
    const int MW = 16 * kSynTM;
    bool ok = NCp <= 4 * kSynWgSc;
    std::vector<int> lb(Jp1), ub(Jp1);
    for (int j = 0; j < Jp1; ++j) {
      lb[j] = p->sc[j].lo + 1;
      ub[j] = p->sc[j].hi - 1;
    }
    // work items (l0, m0, chunk, k-steps), grouped by the k-step class
    // {<=2, <=4, <=8} of the kernel that runs them: by the most scales that
    // one of its waves sees (independent waves), and by those of its 64 l
    // (the kernel with a shared V tile; its list follows the other)
    std::vector<int4> wcls[2][3];
    bool side_small[2] = {true, true};
    for (int l0 = ((L - 1) / 64) * 64; l0 >= 0 && ok; l0 -= 64) {
      auto scales = [&](int la, int lz, int *jmin) {
        int n = 0;
        for (int j = Jp1 - 1; j >= 0; --j)
          if (lb[j] <= ub[j] && lb[j] <= lz && ub[j] >= la) {
            ++n;
            *jmin = j;
          }
        return n;
      };
      auto cls_of = [](int ks) { return ks <= 2 ? 0 : ks <= 4 ? 1 : 2; };
      int jmin = Jp1;
      const int nsw = scales(l0, l0 + 63, &jmin);
      if (nsw > kSynWgSc || nsw * NCp > 4 * kSynWgSc) ok = false;
      const int lmax = std::min(l0 + 63, L - 1), ks = nsw * NCp / 4;
      if (cls_of(ks) > 0 && jmin < 2) side_small[1] = false;
      for (int c = 0; c * CW <= lmax; ++c)
        for (int m0 = 0; m0 <= lmax; m0 += MW) {
          wcls[1][cls_of(ks)].push_back(make_int4(l0, m0, c, ks));
          int kw = 0, jw = Jp1;
          for (int w = 0; w < 4; ++w) {
            const int lw = l0 + 16 * w;
            if (!syn_wave_idle(lw, m0, c * CW, L)) kw = std::max(kw, scales(lw, lw + 15, &jw) * NCp / 4);
          }
          if (cls_of(kw) > 0 && jw < 2) side_small[0] = false;
          wcls[0][cls_of(kw)].push_back(make_int4(l0, m0, c, kw));
        }
    }
    // at most one item per CU: one launch of the largest class, whose
    // registers cost nothing there
    if (wcls[0][0].size() + wcls[0][1].size() + wcls[0][2].size() <= 256) {
      const int top = !wcls[0][2].empty() ? 2 : !wcls[0][1].empty() ? 1 : 0;
      for (int c = 0; c < top; ++c) {
        wcls[0][top].insert(wcls[0][top].end(), wcls[0][c].begin(), wcls[0][c].end());
        wcls[0][c].clear();
      }
    }
    std::vector<int4> work;
    for (int k = 0; k < 2; ++k)
      for (int c = 0; c < 3; ++c) {
        p->smf_wcount[k][c] = (int)wcls[k][c].size();
        work.insert(work.end(), wcls[k][c].begin(), wcls[k][c].end());
      }
    {
      // the kernel reads Vt, BT and cc through buffer loads with 32-bit offsets
      long long bt = 4;
      for (int j = 0; j < Jp1; ++j)
        if (lb[j] <= ub[j]) bt += (long long)(ub[j] + 1) * NCp * (ub[j] - lb[j] + 1);
      ok = ok && p->tg_doubles * 8 <= kBufMaxBytes && bt * 8 <= kBufMaxBytes && 16LL * L * L <= kBufMaxBytes;
    }
    if (ok) {
      for (int k = 0; k < 2; ++k) p->smf_side_small[k] = side_small[k];
      p->smf_NCp = NCp;
      p->smf_CW = CW;
      p->smf_nch = nch;
      p->smf_lb = lb;
      p->smf_ub = ub;
      p->smf_btoff.assign(Jp1, 0);
      long long bt = 4;  // 4 zero entries first (out-of-range reads use index 0)
      for (int j = 0; j < Jp1; ++j) {
        p->smf_btoff[j] = bt;
        if (lb[j] <= ub[j]) bt += (long long)(ub[j] + 1) * NCp * (ub[j] - lb[j] + 1);
      }
      if (int e = da.alloc(&p->d_BT, (size_t)bt)) return e;
      p->bt_doubles = bt;
      S2DW_HIP_CHECK(hipMemsetAsync(p->d_BT, 0, 4 * sizeof(double), p->stream));
      if (int e = da.alloc(&p->d_cc, (size_t)L * L)) return e;
      if (nch > 1 && !p->tab_syn)
        if (int e = da.alloc(&p->d_cp, (size_t)(nch - 1) * 2 * L * L)) return e;
      if (int e = da.alloc(&p->d_fpart, (size_t)nch * L * L)) return e;
      if (int e = da.alloc(&p->d_swork, work.size())) return e;
      p->n_swork = (int)work.size();
      if (int e = upload(p->d_swork, work.data(), work.size() * sizeof(int4), p->stream)) return e;
      hipLaunchKernelGGL(k_syn_cc, dim3((unsigned)(((long long)L * L + 255) / 256)), dim3(256), 0, p->stream, L, p->d_cc);
      S2DW_HIP_CHECK(hipGetLastError());
      if (nch > 1 && !p->tab_syn) {
        const int nth = (nch - 1) * 2 * L;
        hipLaunchKernelGGL(k_syn_checkpoints, dim3((nth + 127) / 128), dim3(128), 0, p->stream, L, CW, nch - 1, p->d_S0,
                           p->d_cp);
        S2DW_HIP_CHECK(hipGetLastError());
      }
      SynTabArgs ta{};
      ta.L = L;
      ta.nk = nk;
      ta.NC = NCs;
      ta.NCp = NCp;
      ta.nsc = Jp1;
      ta.Jp1 = Jp1;
      ta.thin = p->d_thin;
      ta.K = d_K;
      ta.sS = d_sS;
      for (int c = 0; c < NCs; ++c) ta.colS_n[c] = p->cols_s[c].n;
      for (int j = 0; j < Jp1; ++j) {
        ta.lb[j] = lb[j];
        ta.ub[j] = ub[j];
        ta.btoff[j] = p->smf_btoff[j];
      }
      ta.BT = p->d_BT;
      for (int j = 0; j < Jp1; ++j) {
        if (lb[j] > ub[j]) continue;
        const long long cnt = (long long)(ub[j] + 1) * NCp * (ub[j] - lb[j] + 1);
        hipLaunchKernelGGL(k_syn_btab, dim3((unsigned)((cnt + 255) / 256)), dim3(256), 0, p->stream, ta, j, cnt);
        S2DW_HIP_CHECK(hipGetLastError());
      }
    } else {
      p->syn_mfma = false;
    }
  } else {
    p->syn_mfma = false;
  }
  // gamma matrices
  {
    std::vector<double2> G((size_t)N * NCa);
    for (int g = 0; g < N; ++g)
      for (int c = 0; c < NCa; ++c) {
        const int n = p->cols_a[c].n;
        // i^n e^{i n pi g / N} u_part
        const long double ang = pi * (long double)n * (0.5L + (long double)g / (long double)N);
        std::complex<long double> z(cosl(ang), sinl(ang));
        if (p->cols_a[c].part) z *= std::complex<long double>(0.0L, 1.0L);
        G[(size_t)g * NCa + c] = make_double2((double)z.real(), (double)z.imag());
      }
    if (int e = da.alloc(&p->d_G, G.size())) return e;
    if (int e = upload(p->d_G, G.data(), G.size() * sizeof(double2), p->stream)) return e;
    if (p->refround) {
      // the reference's rounding of its phase factors: exp(I*(n-m)*PION2) and
      // the gamma-DFT factor exp(I*(n*gamma_g)), gamma_g = PI*g/N
      // (s2dw_core_mod.f90:666, 676-705)
      const double PION2 = 1.570796326794896619231321691639751442099, PI = 3.141592653589793238462643383279502884197;
      std::vector<double2> Gr((size_t)N * NCa);
      for (int g = 0; g < N; ++g) {
        const double gamma_g = PI * g / (double)N;
        for (int c = 0; c < NCa; ++c) {
          const std::complex<double> z = std::exp(std::complex<double>(0.0, p->cols_a[c].n * gamma_g));
          const std::complex<double> u = p->cols_a[c].part ? std::complex<double>(0.0, 1.0) * z : z;
          Gr[(size_t)g * NCa + c] = make_double2(u.real(), u.imag());
        }
      }
      // k = n - m in [-(L-1) - (N-1), N-1]
      p->phoff = (L - 1) + (N - 1);
      std::vector<double2> ph((size_t)p->phoff + N);
      for (int k = -p->phoff; k <= N - 1; ++k) {
        const std::complex<double> z = std::exp(std::complex<double>(0.0, 1.0) * (double)k * PION2);
        ph[(size_t)(k + p->phoff)] = make_double2(z.real(), z.imag());
      }
      if (int e = da.alloc(&p->d_Gref, Gr.size())) return e;
      if (int e = upload(p->d_Gref, Gr.data(), Gr.size() * sizeof(double2), p->stream)) return e;
      if (int e = da.alloc(&p->d_phref, ph.size())) return e;
      if (int e = upload(p->d_phref, ph.data(), ph.size() * sizeof(double2), p->stream)) return e;
      if (int e = refbeta_build(p)) return e;
    }
  }
  // FFT specs (alpha 2hi-1, beta 2hi) and per-scale tables
  {
    std::map<int, int> slot;
    p->tw8_off.assign(Jp1, 0);
    p->wq_off.assign(Jp1, 0);
    long long t8 = 0, wq = 0;
    for (int j = 0; j < Jp1; ++j) {
      Scale &s = p->sc[j];
      for (int which = 0; which < 2; ++which) {
        const int n = which == 0 ? 2 * s.hi - 1 : 2 * s.hi;
        auto it = slot.find(n);
        if (it == slot.end()) {
          FftSpec f{};
          // lengths that are no power of two: Bluestein on the workgroup engine
          // up to M = 4096 (2hi <= 2048), also where the length is smooth
          // (L = 300: the beta stage of 600 points takes 45 us per scale as
          // mixed-radix stages of the generic kernel)
          const int maxM = p->fft_engine == 0 && (which == 0 || p->beta_one) ? 2 * kTS : p->fft_engine == 0 ? kTS / 2 : 0;
          if (int e = make_fft(p, n, &f, maxM)) return e;
          slot[n] = (int)p->ffts.size();
          p->ffts.push_back(f);
          it = slot.find(n);
        }
        if (which == 0) s.fa = it->second;
        else s.fb = it->second;
      }
      p->tw8_off[j] = t8;
      t8 += 8LL * s.hi;
      p->wq_off[j] = wq;
      wq += 2LL * s.hi;
    }
    // odd-length alpha engine for the full-band pair at 2hi - 1 = 1023
    // (31 * 11 * 3): its twiddle table e^{+2 pi i k/1023}
    if (p->fft_engine == 0 && p->odd_alpha && Jp1 >= 2 && p->sc[0].hi == kOddHi && p->sc[1].hi == kOddHi) {
      const int n = 2 * kOddHi - 1;
      std::vector<double2> otw(n);
      for (int k = 0; k < n; ++k) {
        const long double a = 2.0L * pi * (long double)k / (long double)n;
        otw[k] = make_double2((double)cosl(a), (double)sinl(a));
      }
      if (int e = da.alloc(&p->d_otw, otw.size())) return e;
      if (int e = upload(p->d_otw, otw.data(), otw.size() * sizeof(double2), p->stream)) return e;
    }
    std::vector<double2> tw8(t8);
    std::vector<double> wqv(wq);
    for (int j = 0; j < Jp1; ++j) {
      const int hi = p->sc[j].hi;
      for (int k = 0; k < 8 * hi; ++k) {
        const long double a = 2.0L * pi * (long double)k / (8.0L * hi);
        tw8[p->tw8_off[j] + k] = make_double2((double)cosl(a), (double)sinl(a));
      }
      for (int b = 0; b < 2 * hi; ++b) wqv[p->wq_off[j] + b] = quad_weight(M_PI * (2.0 * b + 1.0) / (4.0 * hi), hi);
    }
    if (int e = da.alloc(&p->d_tw8, tw8.size())) return e;
    if (int e = upload(p->d_tw8, tw8.data(), tw8.size() * sizeof(double2), p->stream)) return e;
    if (int e = da.alloc(&p->d_wq, wqv.size())) return e;
    if (int e = upload(p->d_wq, wqv.data(), wqv.size() * sizeof(double), p->stream)) return e;
    // synthesis gamma table e^{-i n pi g/N} per synthesis n-index
    std::vector<int> nlist;
    for (auto &c : p->cols_s)
      if (std::find(nlist.begin(), nlist.end(), c.n) == nlist.end()) nlist.push_back(c.n);
    std::vector<double2> eg(std::max<size_t>(1, nlist.size() * N));
    for (size_t i = 0; i < nlist.size(); ++i)
      for (int g = 0; g < N; ++g) {
        const long double a = -pi * (long double)nlist[i] * (long double)g / (long double)N;
        eg[i * N + g] = make_double2((double)cosl(a), (double)sinl(a));
      }
    double2 *d_eg;
    if (int e = da.alloc(&d_eg, eg.size())) return e;
    if (int e = upload(d_eg, eg.data(), eg.size() * sizeof(double2), p->stream)) return e;
    p->eg = d_eg;
    p->nlist = nlist;
    const auto z0 = std::find(nlist.begin(), nlist.end(), 0);
    p->z0 = z0 == nlist.end() ? -1 : (int)(z0 - nlist.begin());
  }
  // LDS: the generic FFT kernels need two buffers of the work length, the
  // wave-engine kernels one 64*E region per wave.
  {
    int maxlds = 65536;
    (void)hipDeviceGetAttribute(&maxlds, hipDeviceAttributeMaxSharedMemoryPerBlock, p->device);
    p->max_lds = maxlds;
    size_t need = 0;
    for (const FftSpec &f : p->ffts)
      if (!wave_shape(p, f).ok && !(big_fft(f) && p->fft_engine == 0 && maxlds >= lds_of(log2_of(f.M)) + kCsumLds))
        need = std::max(need, fft_lds(f, 0));
    if (need > (size_t)maxlds) {
      set_error("FFT work length needs %zu bytes of LDS, the device allows %d", need, maxlds);
      return kErrSizeInvalid;
    }
    if (maxlds > 65536) {
      const void *fns[] = {(const void *)k_beta_ana, (const void *)k_alpha_c2r, (const void *)k_alpha_r2c,
                           (const void *)k_beta_syn, (const void *)k_beta_ana_w<16>, (const void *)k_beta_ana_w<32>,
                           (const void *)k_alpha_c2r_w<16>, (const void *)k_alpha_c2r_w<32>,
                           (const void *)k_alpha_r2c_w<16>, (const void *)k_alpha_r2c_w<32>,
                           (const void *)k_beta_syn_w<16>, (const void *)k_beta_syn_w<32>};
      for (const void *fn : fns) S2DW_HIP_CHECK(hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, maxlds));
    }
    const struct { const void *fn; int lds; } big[] = {
        {(const void *)k_beta_ana16<12>, lds16_of(12)},         {(const void *)k_beta_ana_h2<13, true>, lds_of(13)},
        {(const void *)k_beta_syn16<12>, lds16_of(12)},         {(const void *)k_beta_syn_h2<13, true>, lds_of(13)},
        {(const void *)k_alpha_c2r16<12, false>, lds16_of(12)}, {(const void *)k_alpha_c2r_t2<13, 1>, lds_of(13)},
        {(const void *)k_alpha_c2r16<12, true>, lds16_of(12)},  {(const void *)k_alpha_c2r_t2m<13, 1>, lds_of(13)},
        {(const void *)k_alpha_syn16<12>, lds16_of(12)},        {(const void *)k_alpha_syn_t2<13, 1>, lds_of(13)},
        {(const void *)k_alpha_r2c16<12>, lds16_of(12)},        {(const void *)k_alpha_r2c_t2<13, 1>, lds_of(13)}};
    for (const auto &b : big)
      if (b.lds + kCsumLds <= maxlds)
        S2DW_HIP_CHECK(hipFuncSetAttribute(b.fn, hipFuncAttributeMaxDynamicSharedMemorySize, b.lds));
  }
  p->d_cov = d_cov;
  p->d_Phi2 = nullptr;
  if (int e = da.alloc(&p->d_Phi2, (size_t)L)) return e;
  if (int e = upload(p->d_Phi2, Phi2, L * sizeof(double), p->stream)) return e;
  {
    std::vector<int> his(Jp1);
    std::vector<long long> offs(Jp1);
    for (int j = 0; j < Jp1; ++j) {
      his[j] = p->sc[j].hi;
      offs[j] = p->sc[j].wav_off;
    }
    if (int e = da.alloc(&p->d_his, his.size())) return e;
    if (int e = da.alloc(&p->d_woffs, offs.size())) return e;
    if (int e = upload(p->d_his, his.data(), his.size() * sizeof(int), p->stream)) return e;
    if (int e = upload(p->d_woffs, offs.data(), offs.size() * sizeof(long long), p->stream)) return e;
    // partials of the per-scale moments (s2dw_hip_stat_moments_device)
    std::vector<long long> cnt(Jp1);
    for (int j = 0; j < Jp1; ++j) cnt[j] = (long long)(2 * p->sc[j].hi - 1) * 2 * p->sc[j].hi * N;
    p->mom_doubles = moments_partial_doubles(cnt.data(), Jp1);
    if (int e = da.alloc(&p->d_mom, (size_t)p->mom_doubles)) return e;
  }
  if (int e = build_groups(p)) return e;
  p->syn_mfma_ok = p->syn_mfma;
  S2DW_HIP_CHECK(hipStreamSynchronize(p->stream));
  return kErrNone;
}

// ---------------------------------------------------------------------------
// Stage drivers.
// ---------------------------------------------------------------------------
namespace {

hipEvent_t pool_event(Plan *p) {
  if (!p->ev_pool.empty()) {
    hipEvent_t e = p->ev_pool.back();
    p->ev_pool.pop_back();
    return e;
  }
  hipEvent_t e = nullptr;
  (void)hipEventCreate(&e);
  return e;
}

// Records a pair of events around the launches of one stage when timing is on.
struct StageTimer {
  Plan *p;
  int stage;
  hipEvent_t a = nullptr;
  StageTimer(Plan *pp, int s) : p(pp), stage(s) {
    if (p->timing) {
      a = pool_event(p);
      (void)hipEventRecord(a, p->stream);
    }
  }
  ~StageTimer() {
    if (p->timing && a) {
      hipEvent_t b = pool_event(p);
      (void)hipEventRecord(b, p->stream);
      p->ev_live.push_back({stage, a, b});
    }
  }
};

template <int P>
int launch_ana_nc(int nc, dim3 grid, hipStream_t s, const AnaArgs &a) {
  switch (nc) {
#define S2DW_CASE(K)                                                             \
  case K:                                                                        \
    hipLaunchKernelGGL((k_ana_contract<K, P>), grid, dim3(256), 0, s, a);        \
    break;
    S2DW_CASE(1) S2DW_CASE(2) S2DW_CASE(3) S2DW_CASE(4) S2DW_CASE(5) S2DW_CASE(6) S2DW_CASE(7) S2DW_CASE(8)
#undef S2DW_CASE
    default: return kErrArgInvalid;
  }
  S2DW_HIP_CHECK(hipGetLastError());
  return kErrNone;
}

template <int Q>
int launch_syn_nc(int nc, dim3 grid, hipStream_t s, const SynArgs &a) {
  switch (nc) {
#define S2DW_CASE(K)                                                             \
  case K:                                                                        \
    hipLaunchKernelGGL((k_syn_contract<K, Q>), grid, dim3(256), 0, s, a);        \
    break;
    S2DW_CASE(1) S2DW_CASE(2) S2DW_CASE(3) S2DW_CASE(4) S2DW_CASE(5) S2DW_CASE(6) S2DW_CASE(7) S2DW_CASE(8)
#undef S2DW_CASE
    default: return kErrArgInvalid;
  }
  S2DW_HIP_CHECK(hipGetLastError());
  return kErrNone;
}

bool scale_empty(const Scale &s) { return s.lo + 1 > s.hi - 1; }

// Layout of the analysis's beta output Tb of one g: [m][b], so that the beta
// kernels, one column m per FFT, store whole cache lines; the alpha kernels
// read the two adjacent b of a row pair, 32 bytes per m, with the other pairs
// of a line on the same XCD.  At L = 1024, N = 8 (805 MB in and out) columns
// stored 16 bytes at a time took 447 us by themselves against 287 us whole,
// and the 32-byte reads of the alpha stage no more than contiguous ones (227
// us).  The reference-rounding form's GEMM writes [b][m].
int tb_stride_b(const Plan *p, int hi) { return p->refround ? hi : 1; }
int tb_stride_m(const Plan *p, int hi) { return p->refround ? 1 : 2 * hi; }

// Stage arguments of scale j (the launch shape fields are set by the caller).
BetaAnaArgs make_beta_ana(const Plan *p, int j) {
  const Scale &s = p->sc[j];
  BetaAnaArgs b{};
  b.f = p->ffts[s.fb];
  b.logT = fft_logT(b.f, 4);
  b.hi = s.hi;
  b.N = p->N;
  b.Tg = p->d_tg + s.tg_off;
  b.Tb = p->d_tb + s.tb_off;
  b.tbb = tb_stride_b(p, s.hi);
  b.tbm = tb_stride_m(p, s.hi);
  b.tw8 = p->d_tw8 + p->tw8_off[j];
  return b;
}

AlphaArgs make_alpha(const Plan *p, int j, bool synthesis) {
  const Scale &s = p->sc[j];
  AlphaArgs al{};
  al.f = p->ffts[s.fa];
  al.logT = fft_logT(al.f, 4);
  al.hi = s.hi;
  al.Tb = p->d_tb + s.tb_off;
  al.tbb = tb_stride_b(p, s.hi);
  al.tbm = tb_stride_m(p, s.hi);
  al.woff = s.wav_off;
  if (synthesis) {
    al.V = p->d_tb + s.tb_off;
    al.scale = (4.0 * (M_PI * M_PI) / (double)p->N) / (2.0 * s.hi - 1.0);
    al.eg = p->eg;
    al.wq = p->d_wq + p->wq_off[j];
    al.N = p->N;
    al.nn = (int)p->nlist.size();
    al.z0 = p->z0;
  }
  return al;
}

// workgroups of a synthesis alpha launch over one scale (alpha_syn_body)
int syn_blocks(const Plan *p, int hi, int per) {
  const int q = hi * (2 * (int)p->nlist.size() - (p->z0 >= 0));
  return (q + per - 1) / per;
}

BetaSynArgs make_beta_syn(const Plan *p, int j) {
  const Scale &s = p->sc[j];
  const int NCs = (int)p->cols_s.size();
  BetaSynArgs b{};
  b.f = p->ffts[s.fb];
  b.logT = fft_logT(b.f, 4);
  b.hi = s.hi;
  b.N = p->N;
  b.NCtot = NCs;
  b.V = p->d_tb + s.tb_off;
  b.wq = p->d_wq + p->wq_off[j];
  b.tw8 = p->d_tw8 + p->tw8_off[j];
  b.eg = p->eg;
  b.Vt = p->d_tg + s.tg_off;
  const int nn = (int)p->nlist.size();
  for (int i = 0; i < nn; ++i) {
    b.nval[i] = p->nlist[i];
    b.ncol[i] = 0;
    for (int c = 0; c < NCs; ++c)
      if (p->cols_s[c].n == p->nlist[i]) {
        b.col0[i][b.ncol[i]] = c;
        b.cpart[i][b.ncol[i]] = p->cols_s[c].part;
        ++b.ncol[i];
      }
  }
  return b;
}

// Body selector of a grouped alpha launch: 2 log2(M) + bluestein for the
// specialised work lengths (Bluestein, log2 M in [5, 11]; k_alpha_c2r_g has no
// 11, which always runs on its three-stage engine), else 0 (generic).
int alpha_sel(const TeamShape &t) { return t.bl && t.lg >= 5 && t.lg <= kLogTS ? 2 * t.lg + 1 : 0; }
// ... of a grouped beta launch
int beta_sel(const TeamShape &t) { return t.h2 ? kSelH2 + 2 * t.lg + t.bl : 0; }

// Grouped launches (all on the workgroup FFT engine): the two full-band
// scales j = 0, 1 (same shapes) in one launch per stage on the main stream,
// and the small scales j >= 2 in one launch per stage on the helper stream:
// analysis beta + alpha c2r, synthesis alpha (with the gamma-DFT, or its pass
// after it) + beta.  Segment tables go in the kernel arguments, the stage arguments in device tables.
struct Group {
  bool ana = false, syn = false;
  bool first = true;  // synthesis: gamma-DFT before the alpha transform
  GammaTab gm{};      // else its pass
  SegTab ba{}, ac{}, am{}, ar{}, bs{};  // am: alpha c2r reducing to moments
  BetaAnaArgs *d_ba = nullptr;
  AlphaArgs *d_ac = nullptr, *d_ar = nullptr;
  BetaSynArgs *d_bs = nullptr;
};

struct GroupState {
  Group g[2];                        // 1: scales 2..J, or 0..J on one stream (0 unused)
  std::vector<char> in_ana, in_syn;  // per scale: runs in a group
  bool pair = false;                 // scales 0 and 1 run as pair launches in the analysis
  bool pair_syn = false;             // ... and in the synthesis
};

void free_groups(Plan *p) {
  delete static_cast<GroupState *>(p->groups);
  p->groups = nullptr;
}

// Builds group gi from the scales [j0, j1).  Empty scales are left out (they
// are filled one by one).  In a group of the scales from 2 on, so are scales
// beyond the kTN-thread engine (they launch one by one); a group that starts
// at scale 0 stays off if it has one.
int build_group(Plan *p, GroupState *gs, int gi, int j0, int j1) {
  const int N = p->N, nn = (int)p->nlist.size();
  Group &G = gs->g[gi];
  std::vector<BetaAnaArgs> ba;
  std::vector<AlphaArgs> ac, ar;
  std::vector<BetaSynArgs> bs;
  std::vector<int> taken;
  bool ok = j1 - j0 >= 2 || (gi == 1 && j1 > j0);
  // workgroups that the three-stage engine would take of the analysis alpha launch
  auto wg16_of = [&](const Scale &s, const TeamShape &t) { return (s.hi + (4096 >> t.lg) - 1) / (4096 >> t.lg) * N; };
  int wg16 = 0, hmax = 0;
  for (int j = j0; j < j1; ++j) {
    const TeamShape t = scale_empty(p->sc[j]) ? TeamShape{} : alpha_shape(p, p->ffts[p->sc[j].fa]);
    if (t.bl && (t.lg == 10 || t.lg == 11)) wg16 += wg16_of(p->sc[j], t);
    if (t.lg >= 0 && t.lg <= kLogTS) hmax = std::max(hmax, p->sc[j].hi);
  }
  const bool syn_ok = !p->nlist.empty() && N <= kMaxCol;
  G.first = gamma_first(p, hmax);
  for (int j = j0; j < j1 && ok; ++j) {
    const Scale &s = p->sc[j];
    if (scale_empty(s)) {
      ok = gi == 1;  // empty small scales are filled one by one
      continue;
    }
    BetaAnaArgs b = make_beta_ana(p, j);
    AlphaArgs a = make_alpha(p, j, false), r = make_alpha(p, j, true);
    BetaSynArgs y = make_beta_syn(p, j);
    // scales beyond the kTN-thread engine's slots launch one by one
    const TeamShape tb = beta_shape(p, b.f, s.hi), ta = alpha_shape(p, a.f);
    if (tb.lg < 0 || ta.lg < 0 || tb.lg > kLogTS || ta.lg > kLogTS || (tb.h2 && !tb.bl && tb.lg == kLogTS)) {
      ok = gi == 1 && j0 > 0;
      continue;
    }
    b.logT = y.logT = team_logTw(p, b.f, true);
    a.logT = r.logT = team_logTw(p, a.f, false);
    const int nmt = (s.hi + tb.per - 1) / tb.per, npt = (s.hi + ta.per - 1) / ta.per;
    auto add = [](SegTab &t, int blocks, int sel, int par) {
      const int i = t.nseg++;
      t.first[i + 1] = t.first[i] + blocks;
      t.sel[i] = sel;
      t.par[i] = par;
    };
    add(G.ba, nmt * N, beta_sel(tb), nmt);
    // analysis, work length 2048, and 1024 where the launch has a workgroup per
    // CU of these: the three-stage engine; it holds twice the sequences per
    // workgroup.  This launch, on it and on the radix-8 body, us: L = 256, N = 2
    // (256 workgroups) 28.7 and 30.0, N = 4 (512) 38.2 and 41.7; L = 512, N = 2
    // (128) 27.2 and 25.9, L = 201, N = 1 (102) 28.1 and 25.2.  In the synthesis
    // launch, whose gather needs the registers, it spills and small plans lose
    // 5%.
    const bool e16 = ta.bl && (ta.lg == 11 || (ta.lg == 10 && wg16 >= 256));
    const int np16 = e16 ? wg16_of(s, ta) / N : 0;
    if (e16) add(G.ac, np16 * N, kSel16 + ta.lg, np16);
    else add(G.ac, npt * N, alpha_sel(ta), npt);
    add(G.am, npt * N, alpha_sel(ta), npt);
    taken.push_back(j);
    ba.push_back(b);
    a.moff = 8 * p->momf_rec0[j];
    ac.push_back(a);
    if (G.first) add(G.ar, syn_blocks(p, s.hi, ta.per), alpha_sel(ta), 0);
    else add(G.ar, npt * N, alpha_sel(ta), npt);
    add_gamma(p, G.gm, j);
    add(G.bs, nmt * nn, beta_sel(tb), nmt);
    ar.push_back(r);
    bs.push_back(y);
  }
  if (ba.empty()) ok = false;
  G.ana = ok;
  G.syn = ok && syn_ok;
  if (!ok) return kErrNone;
  for (int j : taken) {
    gs->in_ana[j] = 1;
    gs->in_syn[j] = G.syn;
  }
  DevAlloc da{p};
  if (int e = da.alloc(&G.d_ba, ba.size())) return e;
  if (int e = da.alloc(&G.d_ac, ac.size())) return e;
  if (int e = upload(G.d_ba, ba.data(), ba.size() * sizeof(BetaAnaArgs), p->stream)) return e;
  if (int e = upload(G.d_ac, ac.data(), ac.size() * sizeof(AlphaArgs), p->stream)) return e;
  if (G.syn) {
    if (int e = da.alloc(&G.d_ar, ar.size())) return e;
    if (int e = da.alloc(&G.d_bs, bs.size())) return e;
    if (int e = upload(G.d_ar, ar.data(), ar.size() * sizeof(AlphaArgs), p->stream)) return e;
    if (int e = upload(G.d_bs, bs.data(), bs.size() * sizeof(BetaSynArgs), p->stream)) return e;
  }
  // the host vectors must outlive the copies
  S2DW_HIP_CHECK(hipStreamSynchronize(p->stream));
  return kErrNone;
}

int build_groups(Plan *p) {
  const int Jp1 = p->J + 1, N = p->N;
  if (p->fft_engine != 0) return kErrNone;
  auto *gs = new (std::nothrow) GroupState;
  if (!gs) return kErrMemAlloc;
  p->groups = gs;
  gs->in_ana.assign(Jp1, 0);
  gs->in_syn.assign(Jp1, 0);
  // moments records of the analysis that reduces instead of storing: one
  // per alpha-c2r workgroup, scales in order
  p->momf_rec0.assign(Jp1 + 1, 0);
  bool mok = true;
  for (int j = 0; j < Jp1; ++j) {
    const Scale &s = p->sc[j];
    long long r = 0;
    if (!scale_empty(s)) {
      const TeamShape ta = alpha_shape(p, p->ffts[s.fa]);
      if (ta.lg < 0) mok = false;
      else r = (long long)((s.hi + ta.per - 1) / ta.per) * N;
    }
    p->momf_rec0[j + 1] = p->momf_rec0[j] + r;
  }
  // plans on one stream up to B = 256 put every scale in the group (one
  // launch per stage instead of a pair launch and a group launch), where the
  // workgroup engine takes scales 0 and 1 too; else the group holds scales
  // 2..J (at B = 512 the pair's odd-length and one-FFT-per-column kernels
  // are much faster than the group's engine: 186 against 241 us per transform)
  bool all_in = false;
  if (p->single_stream && p->B <= 256 && Jp1 >= 2) {
    if (int e = build_group(p, gs, 1, 0, Jp1)) return e;
    all_in = gs->g[1].ana;
    if (!all_in) {
      gs->g[1] = Group{};
      gs->in_ana.assign(Jp1, 0);
      gs->in_syn.assign(Jp1, 0);
    }
  }
  if (!all_in && Jp1 > 2)
    if (int e = build_group(p, gs, 1, 2, Jp1)) return e;
  // scales 0 and 1 as one pair launch per stage when they have the same
  // FFT specs and run on the workgroup engine
  if (Jp1 >= 2 && !scale_empty(p->sc[0]) && !scale_empty(p->sc[1]) && p->sc[0].fa == p->sc[1].fa &&
      p->sc[0].fb == p->sc[1].fb && p->sc[0].hi == p->sc[1].hi &&
      beta_shape(p, p->ffts[p->sc[0].fb], p->sc[0].hi).lg >= 0 && alpha_shape(p, p->ffts[p->sc[0].fa]).lg >= 0) {
    gs->pair = !gs->in_ana[0];
    gs->pair_syn = !gs->in_syn[0] && !p->nlist.empty() && N <= kMaxCol;
  }
  for (int j = 0; j < Jp1; ++j)
    if (!scale_empty(p->sc[j]) && !gs->in_ana[j] && !(gs->pair && j < 2)) mok = false;
  p->momf_ok = mok;
  if (mok) {
    DevAlloc da{p};
    if (int e = da.alloc(&p->d_momf, (size_t)(8 * p->momf_rec0[Jp1]))) return e;
  }
  return kErrNone;
}

}  // namespace

void plan_drop_graphs(Plan *p) {
  for (auto &g : p->gcache) (void)hipGraphExecDestroy(g.exec);
  p->gcache.clear();
}

int run_graphed(Plan *p, int kind, void *out0, void *out1, const void *in) {
  auto eager = [&]() {
    if (kind == 2)
      return run_analysis(p, nullptr, static_cast<double2 *>(out1), static_cast<const double2 *>(in),
                          static_cast<double *>(out0));
    return kind == 0 ? run_analysis(p, static_cast<double *>(out0), static_cast<double2 *>(out1),
                                    static_cast<const double2 *>(in))
                     : run_synthesis(p, static_cast<double2 *>(out0), static_cast<const double *>(out1),
                                     static_cast<const double2 *>(in));
  };
  // the reference-rounding form's beta sums call rocBLAS, which stays out of
  // captured graphs: that form always runs eagerly
  if (!p->graphs || p->timing || p->refround) return eager();
  constexpr size_t kMaxGraphs = 8;
  for (auto &g : p->gcache) {
    if (g.kind == kind && g.b0 == out0 && g.b1 == out1 && g.b2 == in) {
      g.last = ++p->gtick;
      S2DW_HIP_CHECK(hipGraphLaunch(g.exec, p->stream));
      return kErrNone;
    }
  }
  if (!p->cap) S2DW_HIP_CHECK(hipStreamCreateWithFlags(&p->cap, hipStreamNonBlocking));
  // capture on the private stream (the caller's may be the null stream,
  // which cannot be captured); the replay runs on the caller's stream
  const hipStream_t user = p->stream;
  p->stream = p->cap;
  hipError_t ce = hipStreamBeginCapture(p->cap, hipStreamCaptureModeThreadLocal);
  int e = ce == hipSuccess ? eager() : kErrInitFail;
  hipGraph_t graph = nullptr;
  const hipError_t ee = ce == hipSuccess ? hipStreamEndCapture(p->cap, &graph) : ce;
  p->stream = user;
  if (ce != hipSuccess || ee != hipSuccess) {
    if (graph) (void)hipGraphDestroy(graph);
    set_error("HIP graph capture failed: %s", hipGetErrorString(ce != hipSuccess ? ce : ee));
    return kErrInitFail;
  }
  if (e) {
    (void)hipGraphDestroy(graph);
    return e;
  }
  hipGraphExec_t exec = nullptr;
  const hipError_t ie = hipGraphInstantiate(&exec, graph, nullptr, nullptr, 0);
  (void)hipGraphDestroy(graph);
  S2DW_HIP_CHECK(ie);
  if (p->gcache.size() >= kMaxGraphs) {
    size_t lru = 0;
    for (size_t i = 1; i < p->gcache.size(); ++i)
      if (p->gcache[i].last < p->gcache[lru].last) lru = i;
    (void)hipGraphExecDestroy(p->gcache[lru].exec);
    p->gcache.erase(p->gcache.begin() + (long)lru);
  }
  p->gcache.push_back({kind, out0, out1, in, exec, ++p->gtick});
  S2DW_HIP_CHECK(hipGraphLaunch(exec, p->stream));
  return kErrNone;
}

int run_analysis(Plan *p, double *d_wav, double2 *d_scoeff, const double2 *d_flm, double *d_mom) {
  const int L = p->B, N = p->N, Jp1 = p->J + 1;
  if (d_mom && !p->momf_ok) {
    set_error("this plan cannot reduce the analysis to moments (a scale runs outside the grouped launches)");
    return kErrArgInvalid;
  }
  hipStream_t st = p->stream;
  // plans on one stream write the scaling coefficients with the relayout;
  // with the helper stream they follow its join (a captured analysis that
  // ends on the join, with two final nodes, replays ~7 us slower)
  const bool sc_early = p->single_stream;
  {
    StageTimer tm(p, 0);
    hipLaunchKernelGGL(k_flm_to_fT, dim3((L + 31) / 32, (L + 31) / 32), dim3(256), 0, st, L, d_flm, p->d_fT,
                       p->bl_scoeff, sc_early ? d_scoeff : nullptr, p->ana_par ? p->ana_urot : -1);
    S2DW_HIP_CHECK(hipGetLastError());
  }
  // l-contraction, column chunks of kChunk
  AnaArgs a{};
  a.L = L;
  a.N = N;
  a.NCtot = (int)p->cols_a.size();
  a.RA = 2 + 2 * a.NCtot;
  a.fT = p->d_fT;
  a.Ba = p->d_Ba;
  a.S0 = p->d_S0;
  a.lflush = reinterpret_cast<const int2 *>(p->d_lmeta);
  a.G = p->d_G;
  a.Tg = p->d_tg;
  for (int j = 0; j < Jp1; ++j) {
    a.hi[j] = p->sc[j].hi;
    a.tgoff[j] = p->sc[j].tg_off;
  }
  const int P = p->ana_p;
  if (a.NCtot == 0) {
    const long long n = p->tg_doubles;
    hipLaunchKernelGGL(k_fill, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, (double *)p->d_tg, n);
    S2DW_HIP_CHECK(hipGetLastError());
  }
  if (p->ana_par) {
    StageTimer tm(p, 1);
    AnaParArgs ap{};
    ap.L = L;
    ap.N = N;
    ap.rho = (p->cols_a[0].n & 1) ^ p->ana_urot;
    ap.fT = p->d_fT;
    ap.uinv = p->d_uinv;
    ap.rows = p->d_rows;
    ap.S0 = p->d_S0;
    ap.ends = p->d_ends;
    ap.work = p->d_awork;
    ap.gev = p->d_pgev;
    ap.gnext = p->d_pgnext;
    ap.rows_bytes = p->rows_bytes;
    ap.cg = p->d_cg;
    ap.Tg = p->d_tg;
    if (int e = par_contract(ap, p->ana_nh, st)) return e;
  }
  for (int c0 = 0; c0 < (p->ana_par ? 0 : a.NCtot); c0 += kChunk) {
    StageTimer tm(p, 1);
    a.c0 = c0;
    a.accumulate = c0 > 0;
    const int nc = std::min(kChunk, a.NCtot - c0);
    if (p->precision == 1 && p->d_Bq) {
      hipLaunchKernelGGL(k_row_exp, dim3(L), dim3(256), 0, st, L, d_flm, p->d_erow);
      AnaSplitArgs as{a, p->d_gev, p->d_Sa, p->sa_doubles * 8, p->d_Bq, p->bq_bytes, p->d_erow};
      hipLaunchKernelGGL(k_ana_contract_split<kSplitD>, dim3((L + 3) / 4, (L + 15) / 16), dim3(256), 0, st, as);
      S2DW_HIP_CHECK(hipGetLastError());
      continue;
    }
    if (p->ana_mfma) {
      AnaMfmaArgs am{a, p->d_gev, p->d_lcoef, p->ba_bytes, p->d_uinv, p->d_Sa, p->sa_doubles * 8, nullptr, 0, {}};
      if (p->refround) {
        am.phref = p->d_phref;
        am.phoff = p->phoff;
        am.a.G = p->d_Gref;
      }
      for (int c = 0; c < kChunk; ++c) am.coln[c] = c0 + c < a.NCtot ? p->cols_a[c0 + c].n : 0;
      if (p->d_Sa && p->refround)
        hipLaunchKernelGGL((k_ana_contract_mfma_w<true, true>), dim3((L + 3) / 4, (L + 63) / 64), dim3(256), 0, st, am);
      else if (p->d_Sa)
        hipLaunchKernelGGL((k_ana_contract_mfma_w<true, false>), dim3((L + 3) / 4, (L + 63) / 64), dim3(256), 0, st,
                           am);
      else if (p->ana_wave_indep && a.NCtot <= kChunk)
        hipLaunchKernelGGL(k_ana_contract_mfma_w<false>, dim3((L + 3) / 4, (L + 63) / 64), dim3(256),
                           (size_t)4 * (L + 4) * sizeof(double2), st, am);
      else
        hipLaunchKernelGGL(k_ana_contract_mfma, dim3((L + 3) / 4, (L + 63) / 64), dim3(256),
                           (size_t)4 * L * sizeof(double2), st, am);
      S2DW_HIP_CHECK(hipGetLastError());
      continue;
    }
    const dim3 grid((L + P - 1) / P, (L + 255) / 256);
    int e = P == 1 ? launch_ana_nc<1>(nc, grid, st, a) : launch_ana_nc<2>(nc, grid, st, a);
    if (e) return e;
  }
  // reference-rounding form: the beta sums of every scale as the reference
  // forms them (direct sums with its basis values), before the alpha stage
  const bool refb = p->refround;
  if (refb) {
    StageTimer tm(p, 2);
    if (int e = refbeta_run(p, st)) return e;
  }
  // scales j >= 2 (small transforms, latency-bound launches) run on the
  // helper stream beside j = 0, 1; per-stage timing keeps one stream
  const bool conc = !p->timing && !p->single_stream && Jp1 > 2;
  if (conc) {
    S2DW_HIP_CHECK(hipEventRecord(p->fork, st));
    S2DW_HIP_CHECK(hipStreamWaitEvent(p->aux, p->fork, 0));
  }
  const GroupState *grp = static_cast<const GroupState *>(p->groups);
  // grouped scales: the small ones on the helper stream, scales 0 and 1 on
  // the main stream
  for (int gi = 1; gi >= 0; --gi) {
    if (!grp || !grp->g[gi].ana) continue;
    const Group &G = grp->g[gi];
    hipStream_t sg = (conc && gi == 1) ? p->aux : st;
    if (!refb) {
      StageTimer tm(p, 9);
      hipLaunchKernelGGL(k_beta_ana_g, dim3(G.ba.first[G.ba.nseg]), dim3(kTN), 0, sg, G.ba, G.d_ba);
      S2DW_HIP_CHECK(hipGetLastError());
    }
    StageTimer tm(p, 9);
    if (d_mom)
      hipLaunchKernelGGL(k_alpha_c2r_gm, dim3(G.am.first[G.am.nseg]), dim3(kTN), 0, sg, G.am, G.d_ac, p->d_momf);
    else
      hipLaunchKernelGGL(k_alpha_c2r_g, dim3(G.ac.first[G.ac.nseg]), dim3(kTN), 0, sg, G.ac, G.d_ac, d_wav);
    S2DW_HIP_CHECK(hipGetLastError());
  }
  const bool pair = grp && grp->pair;
  if (pair) {
    BetaAnaArgs b0 = make_beta_ana(p, 0), b1 = make_beta_ana(p, 1);
    b0.logT = b1.logT = team_logTw(p, b0.f, true);
    if (!refb) {
      StageTimer tm(p, 2);
      const TeamShape tb = beta_shape(p, b0.f, b0.hi);
      const int nmt = (b0.hi + tb.per - 1) / tb.per;
      launch_beta_ana(tb, b0, b1, nmt, nmt * N, 2 * nmt * N, st);
      S2DW_HIP_CHECK(hipGetLastError());
    }
    AlphaArgs a0 = make_alpha(p, 0, false), a1 = make_alpha(p, 1, false);
    const TeamShape ta = alpha_shape(p, a0.f);
    a0.logT = a1.logT = team_logTw(p, a0.f, false);
    const int npt = (a0.hi + ta.per - 1) / ta.per;
    StageTimer tm(p, 3);
    if (d_mom) {
      a0.mp = p->d_momf + 8 * p->momf_rec0[0];
      a1.mp = p->d_momf + 8 * p->momf_rec0[1];
      // the odd engine's workgroups hold one row pair each, like the
      // Bluestein pair kernel's, so the record layout is the same
      const int npo = (kOddHi + kOddT - 1) / kOddT;
      if (p->d_otw && npo == npt)
        hipLaunchKernelGGL((k_alpha_c2r_o2<31, 11, 3, kOddNT, kOddT, kOddSplit, true>), dim3(2 * npo * N),
                           dim3(kOddNT), 0, st, a0, a1, npo, p->d_otw);
      else
        launch_alpha_c2r_mom(ta, a0, a1, npt, npt * N, 2 * npt * N, st);
    } else {
      a0.W = d_wav + p->sc[0].wav_off;
      a1.W = d_wav + p->sc[1].wav_off;
      if (p->d_otw) {
        const int npo = (kOddHi + kOddT - 1) / kOddT;
        hipLaunchKernelGGL((k_alpha_c2r_o2<31, 11, 3>), dim3(2 * npo * N), dim3(kOddNT), 0, st, a0, a1, npo, p->d_otw);
      } else {
        launch_alpha_c2r(ta, a0, a1, npt, npt * N, 2 * npt * N, st);
      }
    }
    S2DW_HIP_CHECK(hipGetLastError());
  }
  for (int j = 0; j < Jp1; ++j) {
    const Scale &s = p->sc[j];
    if ((grp && grp->in_ana[j]) || (pair && j < 2)) continue;
    if (d_mom) continue;  // only empty scales get here: no records, zero moments
    hipStream_t sj = (conc && j >= 2) ? p->aux : st;
    double *wj = d_wav + s.wav_off;
    const long long nw = (long long)(2 * s.hi - 1) * 2 * s.hi * N;
    if (scale_empty(s)) {
      hipLaunchKernelGGL(k_fill, dim3((unsigned)((nw + 255) / 256)), dim3(256), 0, sj, wj, nw);
      S2DW_HIP_CHECK(hipGetLastError());
      continue;
    }
    // beta
    if (!refb) {
      StageTimer tm(p, 2);
      BetaAnaArgs b = make_beta_ana(p, j);
      const WaveShape ws = wave_shape(p, b.f);
      const TeamShape ts = beta_shape(p, b.f, s.hi);
      if (ts.lg >= 0) {
        b.logT = team_logTw(p, b.f, true);
        const int nmt = (s.hi + ts.per - 1) / ts.per;
        launch_beta_ana(ts, b, b, nmt, nmt * N, nmt * N, sj);
      } else if (ws.ok) {
        b.logT = ws.logTw;
        const int TMW = ws.WPB << ws.logTw;
        const dim3 grid((s.hi + TMW - 1) / TMW, N, 2), block(64 * ws.WPB);
        if (ws.E == 16) hipLaunchKernelGGL(k_beta_ana_w<16>, grid, block, ws.lds, sj, b);
        else hipLaunchKernelGGL(k_beta_ana_w<32>, grid, block, ws.lds, sj, b);
      } else {
        const int T = 1 << b.logT;
        const size_t lds = fft_lds(b.f, b.logT);
        hipLaunchKernelGGL(k_beta_ana, dim3((s.hi + T - 1) / T, N, 2), dim3(256), lds, sj, b);
      }
      S2DW_HIP_CHECK(hipGetLastError());
    }
    // alpha
    {
      StageTimer tm(p, 3);
      AlphaArgs al = make_alpha(p, j, false);
      al.W = wj;
      const WaveShape ws = wave_shape(p, al.f);
      const TeamShape ts = alpha_shape(p, al.f);
      if (ts.lg >= 0) {
        al.logT = team_logTw(p, al.f, false);
        const int npt = (s.hi + ts.per - 1) / ts.per;
        launch_alpha_c2r(ts, al, al, npt, npt * N, npt * N, sj);
      } else if (ws.ok) {
        al.logT = ws.logTw;
        const int per = ws.WPB << ws.logTw;
        const dim3 grid((s.hi + per - 1) / per, N), block(64 * ws.WPB);
        if (ws.E == 16) hipLaunchKernelGGL(k_alpha_c2r_w<16>, grid, block, ws.lds, sj, al);
        else hipLaunchKernelGGL(k_alpha_c2r_w<32>, grid, block, ws.lds, sj, al);
      } else {
        const int T = 1 << al.logT;
        const size_t lds = fft_lds(al.f, al.logT);
        hipLaunchKernelGGL(k_alpha_c2r, dim3((s.hi + T - 1) / T, N), dim3(256), lds, sj, al);
      }
      S2DW_HIP_CHECK(hipGetLastError());
    }
  }
  if (conc) {
    S2DW_HIP_CHECK(hipEventRecord(p->join, p->aux));
    S2DW_HIP_CHECK(hipStreamWaitEvent(st, p->join, 0));
  }
  if (d_mom) {
    StageTimer tm(p, 3);
    std::vector<long long> cnt(Jp1);
    for (int j = 0; j < Jp1; ++j) cnt[j] = (long long)(2 * p->sc[j].hi - 1) * 2 * p->sc[j].hi * N;
    if (int e = moments_finish(st, cnt.data(), p->momf_rec0.data(), Jp1, p->d_momf, d_mom)) return e;
  }
  if (!sc_early) {
    const int bl = p->bl_scoeff;
    StageTimer tm(p, 4);
    hipLaunchKernelGGL(k_scoeff, dim3((bl * bl + 255) / 256), dim3(256), 0, st, L, bl, d_flm, d_scoeff);
    S2DW_HIP_CHECK(hipGetLastError());
  }
  return kErrNone;
}

int run_synthesis(Plan *p, double2 *d_flm, const double *d_wav, const double2 *d_scoeff) {
  const int L = p->B, N = p->N, Jp1 = p->J + 1;
  hipStream_t st = p->stream;
  const int NCs = (int)p->cols_s.size();
  const bool conc = !p->timing && !p->single_stream && Jp1 > 2;
  if (conc) {
    S2DW_HIP_CHECK(hipEventRecord(p->fork, st));
    S2DW_HIP_CHECK(hipStreamWaitEvent(p->aux, p->fork, 0));
  }
  const GroupState *grp = static_cast<const GroupState *>(p->groups);
  const int nn_all = (int)p->nlist.size();
  const bool pair = grp && grp->pair_syn;
  for (int gi = 1; gi >= 0; --gi) {
    if (!grp || !grp->g[gi].syn) continue;
    const Group &G = grp->g[gi];
    hipStream_t sg = (conc && gi == 1) ? p->aux : st;
    {
      StageTimer tm(p, 10);
      if (G.first)
        hipLaunchKernelGGL(k_alpha_syn_g, dim3(G.ar.first[G.ar.nseg]), dim3(kTN), 0, sg, G.ar, G.d_ar, d_wav);
      else
        hipLaunchKernelGGL(k_alpha_r2c_g, dim3(G.ar.first[G.ar.nseg]), dim3(kTN), 0, sg, G.ar, G.d_ar, d_wav);
      S2DW_HIP_CHECK(hipGetLastError());
    }
    if (!G.first) {
      StageTimer tm(p, 10);
      launch_gamma_syn(p, G.gm, sg);
      S2DW_HIP_CHECK(hipGetLastError());
    }
    StageTimer tm(p, 10);
    hipLaunchKernelGGL(k_beta_syn_g, dim3(G.bs.first[G.bs.nseg]), dim3(kTN), 0, sg, G.bs, G.d_bs);
    S2DW_HIP_CHECK(hipGetLastError());
  }
  if (pair) {
    const bool first = gamma_first(p, p->sc[0].hi);
    AlphaArgs a0 = make_alpha(p, 0, true), a1 = make_alpha(p, 1, true);
    const TeamShape ta = alpha_shape(p, a0.f);
    a0.logT = a1.logT = team_logTw(p, a0.f, false);
    a0.W = const_cast<double *>(d_wav + p->sc[0].wav_off);
    a1.W = const_cast<double *>(d_wav + p->sc[1].wav_off);
    {
      StageTimer tm(p, 5);
      const int nb = syn_blocks(p, a0.hi, p->d_otw ? 1 : ta.per), npt = (a0.hi + ta.per - 1) / ta.per;
      if (first && p->d_otw)
        hipLaunchKernelGGL((k_alpha_syn_o2<31, 11, 3>), dim3(2 * nb), dim3(kOddNT), 0, st, a0, a1, p->d_otw);
      else if (first)
        launch_alpha_syn(ta, a0, a1, 0, nb, 2 * nb, st);
      else if (p->d_otw)
        hipLaunchKernelGGL((k_alpha_r2c_o2<31, 11, 3>), dim3(2 * a0.hi * N), dim3(kOddNT), 0, st, a0, a1, p->d_otw);
      else
        launch_alpha_r2c(ta, a0, a1, npt, npt * N, 2 * npt * N, st);
      S2DW_HIP_CHECK(hipGetLastError());
    }
    StageTimer tm(p, 6);
    if (!first) {
      GammaTab gt{};
      for (int j : {0, 1}) add_gamma(p, gt, j);
      launch_gamma_syn(p, gt, st);
      S2DW_HIP_CHECK(hipGetLastError());
    }
    BetaSynArgs y0 = make_beta_syn(p, 0), y1 = make_beta_syn(p, 1);
    const TeamShape tb = beta_shape(p, y0.f, y0.hi);
    y0.logT = y1.logT = team_logTw(p, y0.f, true);
    const int nmt = (y0.hi + tb.per - 1) / tb.per;
    launch_beta_syn(tb, y0, y1, nmt, nmt * nn_all, 2 * nmt * nn_all, st);
    S2DW_HIP_CHECK(hipGetLastError());
  }
  for (int j = 0; j < Jp1; ++j) {
    const Scale &s = p->sc[j];
    if ((grp && grp->in_syn[j]) || (pair && j < 2)) continue;
    hipStream_t sj = (conc && j >= 2) ? p->aux : st;
    if (scale_empty(s)) continue;
    BetaSynArgs b = make_beta_syn(p, j);
    const TeamShape tb = beta_shape(p, b.f, s.hi);
    const bool team_beta = nn_all > 0 && tb.lg >= 0 && N <= kMaxCol;
    bool gamma_done = false;
    // alpha r2c -> V, or with the gamma-DFT -> U (tb buffer)
    {
      StageTimer tm(p, 5);
      AlphaArgs al = make_alpha(p, j, true);
      al.W = const_cast<double *>(d_wav + s.wav_off);
      const WaveShape ws = wave_shape(p, al.f);
      const TeamShape ts = alpha_shape(p, al.f);
      if (ts.lg >= 0) {
        al.logT = team_logTw(p, al.f, false);
        gamma_done = team_beta && gamma_first(p, s.hi);
        const int npt = (s.hi + ts.per - 1) / ts.per, nb = syn_blocks(p, s.hi, ts.per);
        if (gamma_done) launch_alpha_syn(ts, al, al, 0, nb, nb, sj);
        else launch_alpha_r2c(ts, al, al, npt, npt * N, npt * N, sj);
      } else if (ws.ok) {
        al.logT = ws.logTw;
        const int per = ws.WPB << ws.logTw;
        const dim3 grid((s.hi + per - 1) / per, N), block(64 * ws.WPB);
        if (ws.E == 16) hipLaunchKernelGGL(k_alpha_r2c_w<16>, grid, block, ws.lds, sj, al);
        else hipLaunchKernelGGL(k_alpha_r2c_w<32>, grid, block, ws.lds, sj, al);
      } else {
        const int T = 1 << al.logT;
        const size_t lds = fft_lds(al.f, al.logT);
        hipLaunchKernelGGL(k_alpha_r2c, dim3((s.hi + T - 1) / T, N), dim3(256), lds, sj, al);
      }
      S2DW_HIP_CHECK(hipGetLastError());
    }
    // beta -> Vt (tg buffer)
    {
      StageTimer tm(p, 6);
      const int nn = nn_all;
      const WaveShape ws = wave_shape(p, b.f);
      if (team_beta) {
        if (!gamma_done) {
          GammaTab gt{};
          add_gamma(p, gt, j);
          launch_gamma_syn(p, gt, sj);
          S2DW_HIP_CHECK(hipGetLastError());
        }
        b.logT = team_logTw(p, b.f, true);
        const int nmt = (s.hi + tb.per - 1) / tb.per;
        launch_beta_syn(tb, b, b, nmt, nmt * nn, nmt * nn, sj);
        S2DW_HIP_CHECK(hipGetLastError());
      } else if (nn > 0 && ws.ok) {
        b.logT = ws.logTw;
        const int TMW = ws.WPB << ws.logTw;
        const dim3 grid((s.hi + TMW - 1) / TMW, nn, 2), block(64 * ws.WPB);
        if (ws.E == 16) hipLaunchKernelGGL(k_beta_syn_w<16>, grid, block, ws.lds, sj, b);
        else hipLaunchKernelGGL(k_beta_syn_w<32>, grid, block, ws.lds, sj, b);
        S2DW_HIP_CHECK(hipGetLastError());
      } else if (nn > 0) {
        const int T = 1 << b.logT;
        const size_t lds = fft_lds(b.f, b.logT);
        hipLaunchKernelGGL(k_beta_syn, dim3((s.hi + T - 1) / T, nn, 2), dim3(256), lds, sj, b);
        S2DW_HIP_CHECK(hipGetLastError());
      }
    }
  }
  // the contraction classes with more scales per tile read only scales
  // j >= 2 when smf_side_small holds: they then run on the helper stream
  // right after those scales' transforms, beside the full-band scales'
  // transforms on the main stream, and the main class needs no fork
  const int wk = p->tab_syn || p->syn_wave ? 0 : 1;  // work list of the kernel that runs
  const int *wcount = p->smf_wcount[wk];
  const bool early = conc && p->syn_mfma && p->smf_side_small[wk] && wcount[0] > 0 && (wcount[1] + wcount[2]) > 0;
  if (conc) {
    S2DW_HIP_CHECK(hipEventRecord(p->join, p->aux));
    S2DW_HIP_CHECK(hipStreamWaitEvent(st, p->join, 0));
  }
  if (p->syn_mfma) {
    {
      StageTimer tm(p, 7);
      SynMfmaArgs a{};
      a.L = L;
      a.NC = NCs;
      a.NCp = p->smf_NCp;
      a.CW = p->smf_CW;
      a.nsc = Jp1;
      a.work = p->d_swork;
      a.xcd = p->syn_xcd ? 1 : 0;
      a.cc = p->d_cc;
      a.S0 = p->d_S0;
      a.cp = p->d_cp;
      a.Vt = p->d_tg;
      a.BT = p->d_BT;
      a.fpart = p->d_fpart;
      a.vt_bytes = p->tg_doubles * (long long)sizeof(double);
      a.bt_bytes = p->bt_doubles * (long long)sizeof(double);
      a.Sa = p->d_Sa;
      a.sa_bytes = p->sa_doubles * (long long)sizeof(double);
      for (int j = 0; j < Jp1; ++j) {
        a.lb[j] = p->smf_lb[j];
        a.ub[j] = p->smf_ub[j];
        a.hi[j] = p->sc[j].hi;
        a.vtoff[j] = p->sc[j].tg_off;
        a.btoff[j] = p->smf_btoff[j];
      }
      constexpr int TM = kSynTM;
      // the classes with more scales per tile are few, long-running
      // workgroups with more registers per wave than the main class leaves
      // free on a CU: they are launched first, on the main stream, so that
      // they take their CUs before the main class (on the helper stream)
      // fills the rest
      const bool side = !early && !p->single_stream && wcount[0] > 0 && (wcount[1] + wcount[2]) > 0;
      if (side) {
        S2DW_HIP_CHECK(hipEventRecord(p->fork, st));
        S2DW_HIP_CHECK(hipStreamWaitEvent(p->aux, p->fork, 0));
      }
      const int wb = wk ? p->smf_wcount[0][0] + p->smf_wcount[0][1] + p->smf_wcount[0][2] : 0;
      const int w0[3] = {wb, wb + wcount[0], wb + wcount[0] + wcount[1]};
      for (int c : {2, 1, 0}) {
        const int n = wcount[c];
        if (n > 0) {
          const int ksm = 2 << c;
          const size_t lds = 2 * (size_t)ksm * 4 * 16 * TM * sizeof(double2);
          // early: classes 2, 1 on the helper stream (after the join above
          // was recorded there, so the main stream does not wait for them)
          hipStream_t sc = early ? (c == 0 ? st : p->aux) : (side && c == 0) ? p->aux : st;
          a.work0 = w0[c];
          if (p->tab_syn) {
            if (c == 0) hipLaunchKernelGGL((k_syn_contract_mfma_w<TM, 2, true>), dim3(n), dim3(256), 0, sc, a);
            else if (c == 1) hipLaunchKernelGGL((k_syn_contract_mfma_w<TM, 4, true>), dim3(n), dim3(256), 0, sc, a);
            else hipLaunchKernelGGL((k_syn_contract_mfma_w<TM, 8, true>), dim3(n), dim3(256), 0, sc, a);
          } else if (p->syn_wave) {
            if (c == 0) hipLaunchKernelGGL((k_syn_contract_mfma_w<TM, 2, false>), dim3(n), dim3(256), 0, sc, a);
            else if (c == 1) hipLaunchKernelGGL((k_syn_contract_mfma_w<TM, 4, false>), dim3(n), dim3(256), 0, sc, a);
            else hipLaunchKernelGGL((k_syn_contract_mfma_w<TM, 8, false>), dim3(n), dim3(256), 0, sc, a);
          } else if (c == 0) {
            hipLaunchKernelGGL((k_syn_contract_mfma<TM, 2>), dim3(n), dim3(256), lds, sc, a);
          } else if (c == 1) {
            hipLaunchKernelGGL((k_syn_contract_mfma<TM, 4>), dim3(n), dim3(256), lds, sc, a);
          } else {
            hipLaunchKernelGGL((k_syn_contract_mfma<TM, 8>), dim3(n), dim3(256), lds, sc, a);
          }
          S2DW_HIP_CHECK(hipGetLastError());
        }
      }
      if (side || early) {
        S2DW_HIP_CHECK(hipEventRecord(p->join, p->aux));
        S2DW_HIP_CHECK(hipStreamWaitEvent(st, p->join, 0));
      }
    }
    StageTimer tm(p, 8);
    hipLaunchKernelGGL(k_flm_final_chunks, dim3((unsigned)(((long long)L * L + 255) / 256)), dim3(256), 0, st, L,
                       p->bl_scoeff, p->smf_CW, p->d_fpart, p->d_cov, p->d_Phi2, d_scoeff, d_flm);
    S2DW_HIP_CHECK(hipGetLastError());
    return kErrNone;
  }
  // Wigner contraction
  SynArgs a{};
  a.L = L;
  a.NCtot = NCs;
  a.RS = 2 + 2 * NCs;
  a.Bs = p->d_Bs;
  a.S0 = p->d_S0;
  a.blocks = p->d_sblk;
  a.Vt = p->d_tg;
  a.fo = p->d_fo;
  for (int j = 0; j < Jp1; ++j) {
    a.hi[j] = p->sc[j].hi;
    a.vtoff[j] = p->sc[j].tg_off;
  }
  if (NCs == 0) {
    const long long n = 2LL * L * L;
    hipLaunchKernelGGL(k_fill, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, (double *)p->d_fo, n);
    S2DW_HIP_CHECK(hipGetLastError());
  }
  for (int c0 = 0; c0 < NCs; c0 += kChunk) {
    StageTimer tm(p, 7);
    a.c0 = c0;
    a.accumulate = c0 > 0;
    const int nc = std::min(kChunk, NCs - c0);
    const dim3 grid(p->n_sblk, (L + 255) / 256);
    int e = p->syn_q == 4 ? launch_syn_nc<4>(nc, grid, st, a) : launch_syn_nc<8>(nc, grid, st, a);
    if (e) return e;
  }
  StageTimer tm(p, 8);
  hipLaunchKernelGGL(k_flm_final, dim3((L + 31) / 32, (L + 31) / 32), dim3(256), 0, st, L, p->bl_scoeff, p->d_fo,
                     p->d_cov, p->d_Phi2, d_scoeff, d_flm);
  S2DW_HIP_CHECK(hipGetLastError());
  return kErrNone;
}

// Autotuner: times the alternatives that can be switched on a built plan
// and keeps the fastest.  Analysis contraction: MFMA with independent waves,
// MFMA with workgroup-staged operands, VALU with 2 or 1 chains per lane;
// synthesis contraction: MFMA with independent waves, MFMA with a staged V
// tile, VALU with 4 or 8 chains per lane; then the
// helper stream for the small scales on or off, timed on whole round trips.
// Each candidate runs once untimed and `reps` times between HIP events on
// the plan's stream, on zero-filled buffers of the plan's sizes (the kernels'
// running time does not depend on the values).
int plan_autotune(Plan *p, int reps, std::string *report) {
  if (reps < 1) reps = 1;
  const int L = p->B;
  const hipStream_t st = p->stream;
  const bool timing = p->timing, graphs = p->graphs;
  p->timing = false;
  p->graphs = false;
  double2 *d_f = nullptr, *d_g = nullptr, *d_sc = nullptr;
  double *d_w = nullptr;
  hipEvent_t e0 = nullptr, e1 = nullptr;
  int err = kErrNone;
  auto cleanup = [&]() {
    (void)hipFree(d_f);
    (void)hipFree(d_g);
    (void)hipFree(d_sc);
    (void)hipFree(d_w);
    if (e0) (void)hipEventDestroy(e0);
    if (e1) (void)hipEventDestroy(e1);
    p->timing = timing;
    p->graphs = graphs;
  };
  const size_t nf = (size_t)L * L * sizeof(double2), nsc = (size_t)p->bl_scoeff * p->bl_scoeff * sizeof(double2);
  const size_t nw = (size_t)std::max(1LL, p->wav_doubles) * sizeof(double);
  if (hipMalloc(&d_f, nf) != hipSuccess || hipMalloc(&d_g, nf) != hipSuccess ||
      hipMalloc(&d_sc, std::max<size_t>(nsc, 16)) != hipSuccess || hipMalloc(&d_w, nw) != hipSuccess) {
    cleanup();
    set_error("autotune: device buffers of %zu bytes", 2 * nf + nsc + nw);
    return kErrMemAlloc;
  }
  auto chk = [&](hipError_t e, const char *what) {
    if (e != hipSuccess && !err) err = hip_error(e, what);
  };
  chk(hipMemsetAsync(d_f, 0, nf, st), "autotune memset");
  chk(hipMemsetAsync(d_w, 0, nw, st), "autotune memset");
  chk(hipMemsetAsync(d_sc, 0, std::max<size_t>(nsc, 16), st), "autotune memset");
  chk(hipEventCreate(&e0), "autotune event");
  chk(hipEventCreate(&e1), "autotune event");
  if (err) {
    cleanup();
    return err;
  }
  // ms per call of fn(), or a negative value on failure
  auto time_ms = [&](auto fn) -> double {
    if (fn()) return -1.0;
    if (hipEventRecord(e0, st) != hipSuccess) return -1.0;
    for (int r = 0; r < reps; ++r)
      if (fn()) return -1.0;
    if (hipEventRecord(e1, st) != hipSuccess || hipEventSynchronize(e1) != hipSuccess) return -1.0;
    float ms = 0.f;
    if (hipEventElapsedTime(&ms, e0, e1) != hipSuccess) return -1.0;
    return ms / reps;
  };
  auto ana = [&]() { return run_analysis(p, d_w, d_sc, d_f); };
  auto syn = [&]() { return run_synthesis(p, d_g, d_w, d_sc); };
  auto both = [&]() {
    const int e = ana();
    return e ? e : syn();
  };
  char buf[160];
  // analysis contraction
  struct AnaC {
    const char *name;
    bool mfma, wave;
    int P;
    bool par = false;
  };
  std::vector<AnaC> ac;
  // table form: the contraction kernels are fixed (only their table variants
  // reproduce the reference's Wigner values); the helper-stream choice stays
  const bool fixed = p->d_Sa != nullptr, syn_fixed = p->tab_syn;
  if (fixed) *report += p->precision == 1 ? "analysis contraction: split (fixed);" : "analysis contraction: Wigner table form (fixed);";
  if (syn_fixed) *report += " synthesis contraction: Wigner table form (fixed);";
  if (p->ana_nh > 0 && !fixed) ac.push_back({"parity", p->ana_mfma_ok, true, 2, true});
  if (p->ana_mfma_ok && !fixed) {
    ac.push_back({"mfma-wave", true, true, 2});
    ac.push_back({"mfma-staged", true, false, 2});
  }
  ac.push_back({"valu-p2", false, false, 2});
  ac.push_back({"valu-p1", false, false, 1});
  if (fixed) ac.clear();
  double best = 1e30;
  size_t bi = 0;
  if (!fixed) *report += "analysis contraction:";
  for (size_t i = 0; i < ac.size(); ++i) {
    p->ana_par = ac[i].par;
    p->ana_mfma = ac[i].mfma;
    p->ana_wave_indep = ac[i].wave;
    p->ana_p = ac[i].P;
    const double t = time_ms(ana);
    std::snprintf(buf, sizeof buf, " %s %.3f ms%s", ac[i].name, t, i + 1 < ac.size() ? "," : ";");
    *report += buf;
    if (t > 0 && t < best) {
      best = t;
      bi = i;
    }
  }
  if (!fixed) {
    p->ana_par = ac[bi].par;
    p->ana_mfma = ac[bi].mfma;
    p->ana_wave_indep = ac[bi].wave;
    p->ana_p = ac[bi].P;
  }
  // synthesis contraction
  struct SynC {
    const char *name;
    bool mfma;
    int Q;
    bool wave;
  };
  std::vector<SynC> sc;
  if (p->syn_mfma_ok && !syn_fixed) {
    sc.push_back({"mfma-wave", true, 4, true});
    sc.push_back({"mfma-staged", true, 4, false});
  }
  sc.push_back({"valu-q4", false, 4, false});
  sc.push_back({"valu-q8", false, 8, false});
  if (syn_fixed) sc.clear();
  best = 1e30;
  bi = 0;
  if (!syn_fixed) *report += " synthesis contraction:";
  for (size_t i = 0; i < sc.size(); ++i) {
    p->syn_mfma = sc[i].mfma;
    p->syn_q = sc[i].Q;
    p->syn_wave = sc[i].wave;
    const double t = time_ms(syn);
    std::snprintf(buf, sizeof buf, " %s %.3f ms%s", sc[i].name, t, i + 1 < sc.size() ? "," : ";");
    *report += buf;
    if (t > 0 && t < best) {
      best = t;
      bi = i;
    }
  }
  if (!syn_fixed) {
    p->syn_mfma = sc[bi].mfma;
    p->syn_q = sc[bi].Q;
    p->syn_wave = sc[bi].wave;
  }
  // helper stream for the small scales
  const bool single = p->single_stream;
  p->single_stream = false;
  const double t_two = time_ms(both);
  p->single_stream = true;
  const double t_one = time_ms(both);
  p->single_stream = single || (t_one > 0 && (t_two <= 0 || t_one < t_two));
  std::snprintf(buf, sizeof buf, " round trip: two streams %.3f ms, one stream %.3f ms; chosen: %s", t_two, t_one,
                p->single_stream ? "one stream" : "two streams");
  *report += buf;
  plan_drop_graphs(p);  // captured with the old choices
  chk(hipStreamSynchronize(st), "autotune");
  cleanup();
  return err;
}

int stage_times(Plan *p, double *ms, int *count) {
  for (int s = 0; s < kNumStages; ++s) {
    ms[s] = 0.0;
    count[s] = 0;
  }
  if (!p->ev_live.empty()) S2DW_HIP_CHECK(hipEventSynchronize(p->ev_live.back().b));
  for (auto &e : p->ev_live) {
    float t = 0.f;
    S2DW_HIP_CHECK(hipEventElapsedTime(&t, e.a, e.b));
    ms[e.stage] += t;
    count[e.stage] += 1;
    p->ev_pool.push_back(e.a);
    p->ev_pool.push_back(e.b);
  }
  p->ev_live.clear();
  return kErrNone;
}

int pack_static(Plan *p, const double *d_packed, double *d_static, bool to_static) {
  const int Jp1 = p->J + 1, B = p->B, N = p->N;
  const int nchunk = (Jp1 * (2 * B - 1) + 255) / 256;
  const long long blocks = (long long)2 * B * N * nchunk;
  if (blocks > 0x7FFFFFFFLL) {
    set_error("static layout of B=%d N=%d J=%d exceeds one launch", B, N, Jp1 - 1);
    return kErrSizeInvalid;
  }
  hipLaunchKernelGGL(k_pack_static, dim3((unsigned)blocks), dim3(256), 0, p->stream, Jp1, B, N, p->d_his, p->d_woffs,
                     d_packed, d_static, to_static ? 1 : 0, nchunk);
  S2DW_HIP_CHECK(hipGetLastError());
  return kErrNone;
}

int wigner_plane(int l, double *out, double *out2) {
  if (l < 0 || l > 4096) return kErrSizeInvalid;
  const int n = l + 1;
  std::vector<double> s0(tri0(n));
  for (int l0 = 0; l0 < n; ++l0) {
    const long double lg2l = lgammal(2.0L * l0 + 1.0L);
    for (int k = 0; k <= l0; ++k) {
      const long double lv = 0.5L * (lg2l - lgammal((long double)(l0 + k) + 1.0L) - lgammal((long double)(l0 - k) + 1.0L)) -
                             (long double)l0 * logl(2.0L);
      s0[tri0(l0) + k] = (double)expl(lv);
    }
  }
  double *dS0 = nullptr, *dA = nullptr, *dS = nullptr;
  S2DW_HIP_CHECK(hipMalloc(&dS0, s0.size() * sizeof(double)));
  S2DW_HIP_CHECK(hipMalloc(&dA, (size_t)n * n * sizeof(double)));
  S2DW_HIP_CHECK(hipMalloc(&dS, (size_t)n * n * sizeof(double)));
  S2DW_HIP_CHECK(hipMemcpy(dS0, s0.data(), s0.size() * sizeof(double), hipMemcpyHostToDevice));
  hipLaunchKernelGGL(k_wigner_plane, dim3((n * n + 255) / 256), dim3(256), 0, 0, l, dS0, out ? dA : nullptr,
                     out2 ? dS : nullptr);
  S2DW_HIP_CHECK(hipGetLastError());
  S2DW_HIP_CHECK(hipDeviceSynchronize());
  if (out) S2DW_HIP_CHECK(hipMemcpy(out, dA, (size_t)n * n * sizeof(double), hipMemcpyDeviceToHost));
  if (out2) S2DW_HIP_CHECK(hipMemcpy(out2, dS, (size_t)n * n * sizeof(double), hipMemcpyDeviceToHost));
  (void)hipFree(dS0);
  (void)hipFree(dA);
  (void)hipFree(dS);
  return kErrNone;
}

}  // namespace s2dw
