// s2dw_anapar.hip -- analysis l-contraction by parity of l, on the FP64 VALU.
//
// T(m', m, n) = sum_l Delta^l_{m'm} f(l,m) B_n(m',l),
// B_n = K_j(l) S(l,n) Delta^l_{m'n} (s2dw_core_mod.f90:618-674).  At pi/2
// Delta^l_{m',-n} = (-1)^{l+m'} Delta^l_{m'n}, so the columns n and -n share
// their products: with E (O) the sum over even (odd) l of the column n >= 0,
// T_n = E + O and T_{-n} = rho (E - O), rho = +-(-1)^{n+m'}.  Only the columns
// n >= 0 are accumulated, into the accumulators of the parity of l: half the
// multiply-adds of one column per n.
//
// What bounds it: FP64 instruction issue.  FP64 FMAs and FP64 MFMAs have the
// same peak on this GPU (128 flop/clk/CU) and share the unit, so a matrix
// tile pays for padding (16 columns where 2 slots x 4 columns are needed)
// and for moving the chain values into its operand layout, while the VALU
// form pays for neither: a lane is one m, and the column values B, uniform
// over the wave, sit in one register pair (lane % 16 = column) that the FMAs
// read through a DPP row broadcast.  Per l and 64 m: 4 FMAs per column (two
// scales, re and im), 2 products Delta f, 9 for the recursion.
#include <type_traits>

#include "s2dw_dev.h"
#include "s2dw_fft.h"
#include "s2dw_internal.h"

namespace s2dw {

namespace {

// acc[h] += (x, y) * element K0 + h of each lane row's 16 values b.  The DPP
// source must not be written by a VALU instruction less than two wait states
// before; b comes from a load (or a select), and the s_nop covers the select.
#define S2DW_BC(D, K, X) "v_fmac_f64_dpp %" #D ", %[b], %[" #X "] row_newbcast:" K " row_mask:0xf bank_mask:0xf\n"
template <int K0, int NH>
__device__ __forceinline__ void fma_row(double2 (&c)[NH], double b, double x, double y) {
  if constexpr (NH == 1)
    asm("s_nop 1\n" S2DW_BC(0, "%c[k]", x) S2DW_BC(1, "%c[k]", y)
        : "+v"(c[0].x), "+v"(c[0].y)
        : [b] "v"(b), [x] "v"(x), [y] "v"(y), [k] "i"(K0));
  else if constexpr (NH == 2)
    asm("s_nop 1\n" S2DW_BC(0, "%c[k]", x) S2DW_BC(1, "%c[k]", y) S2DW_BC(2, "%c[k1]", x) S2DW_BC(3, "%c[k1]", y)
        : "+v"(c[0].x), "+v"(c[0].y), "+v"(c[1].x), "+v"(c[1].y)
        : [b] "v"(b), [x] "v"(x), [y] "v"(y), [k] "i"(K0), [k1] "i"(K0 + 1));
  else if constexpr (NH == 3)
    asm("s_nop 1\n" S2DW_BC(0, "%c[k]", x) S2DW_BC(1, "%c[k]", y) S2DW_BC(2, "%c[k1]", x) S2DW_BC(3, "%c[k1]", y)
            S2DW_BC(4, "%c[k2]", x) S2DW_BC(5, "%c[k2]", y)
        : "+v"(c[0].x), "+v"(c[0].y), "+v"(c[1].x), "+v"(c[1].y), "+v"(c[2].x), "+v"(c[2].y)
        : [b] "v"(b), [x] "v"(x), [y] "v"(y), [k] "i"(K0), [k1] "i"(K0 + 1), [k2] "i"(K0 + 2));
  else
    asm("s_nop 1\n" S2DW_BC(0, "%c[k]", x) S2DW_BC(1, "%c[k]", y) S2DW_BC(2, "%c[k1]", x) S2DW_BC(3, "%c[k1]", y)
            S2DW_BC(4, "%c[k2]", x) S2DW_BC(5, "%c[k2]", y) S2DW_BC(6, "%c[k3]", x) S2DW_BC(7, "%c[k3]", y)
        : "+v"(c[0].x), "+v"(c[0].y), "+v"(c[1].x), "+v"(c[1].y), "+v"(c[2].x), "+v"(c[2].y), "+v"(c[3].x),
          "+v"(c[3].y)
        : [b] "v"(b), [x] "v"(x), [y] "v"(y), [k] "i"(K0), [k1] "i"(K0 + 1), [k2] "i"(K0 + 2), [k3] "i"(K0 + 3));
}
// A x + Bc y, the row's elements 0 and 1
__device__ __forceinline__ double row_rec(double b, double x, double y) {
  double s = 0.0;
  asm("s_nop 1\n" S2DW_BC(0, "0", x) S2DW_BC(0, "1", y) : "+v"(s) : [b] "v"(b), [x] "v"(x), [y] "v"(y));
  return s;
}
#undef S2DW_BC

// One wave: one m', 64 m, every l.  Workgroup: WV consecutive m' of one
// m-tile.  Its f and u go through LDS, G values of l at a time and double
// buffered (every wave reads them: from L2 they would be 1.5 KB per wave and
// l, 32 bytes per clock and CU, which bounded a form that loaded them into
// registers: 640 us at L = 1024), the waves' rows beside them; one LDS-only
// barrier per G values of l.  WV = 8 measures the same at L = 1024 (447 us)
// and is slower below (115 against 98 us at L = 512, 71 against 59 at 300:
// fewer workgroups to balance over the CUs).
//
// Measured (N = 8, device time of the kernel; before: the FP64 MFMA kernel
// with independent waves): L = 1024 1252 -> 447 us, 512 157 -> 98, 300 92 -> 59;
// N = 4, L = 181 53 -> 28; N = 3, L = 64 35 -> 16.  At L = 1024 FP64 issues
// in 69% of the cycles (FMAs 53%, products 16%); at L <= 512 the longest chains (m', m ~ 0: L steps) end
// alone on their SIMDs and their latency bounds the kernel.
constexpr int G = kParG, WV = kParWv;
template <int NH>
struct ParLds {
  static constexpr int W = 2 * NH + 2;  // A, Bc, slot 0 columns, slot 1 columns
  static constexpr int RP = G * W + 16;  // a wave's rows; lanes past the last row's columns read the padding
  double2 f[2][G][64];
  double u[2][G][64];
  double r[2][WV][RP];
  double cg[2][NH + 1][2 * NH];  // gamma coefficients [order][g][E columns, O columns], g = 0 .. N/2 <= NH
};

template <int NH>
__global__ __launch_bounds__(64 * WV, 4) void k_ana_contract_par(const AnaParArgs a) {
  typedef ParLds<NH> Lds;
  constexpr int W = Lds::W, NT = 64 * WV, NF = G * 64 / NT, NR = (G * W + 63) / 64;
  __shared__ Lds S;
  const int L = a.L;
  const int lane = threadIdx.x & 63, wave = uniform(threadIdx.x >> 6);
  for (int i = threadIdx.x; i < 2 * (NH + 1) * 2 * NH; i += NT) (&S.cg[0][0][0])[i] = a.cg[i];
  const int wk = as_const(a.work)[blockIdx.x];  // m'-block | m-tile << 16
  const int mpb = (wk & 0xffff) * WV, m0 = (wk >> 16) * 64;
  const int mp = uniform(mpb + wave), m = m0 + lane;
  const int lb = max(mpb, m0) & ~(G - 1);  // < L
  const int l0 = mp > m ? mp : m;
  // range-checked loads, issued for every lane: past the buffers they read
  // zeros, and lanes m >= L read the next row's (finite) elements times a
  // chain value of zero
  const __amdgpu_buffer_rsrc_t fres =
      __builtin_amdgcn_make_buffer_rsrc((void *)a.fT, 0, (int)((long long)L * L * sizeof(double2)), kBufWord3);
  const __amdgpu_buffer_rsrc_t ures =
      __builtin_amdgcn_make_buffer_rsrc((void *)a.uinv, 0, (int)((long long)L * L * sizeof(double)), kBufWord3);
  const __amdgpu_buffer_rsrc_t rres =
      __builtin_amdgcn_make_buffer_rsrc((void *)a.rows, 0, (int)a.rows_bytes, kBufWord3);
  // staging: thread (wave, lane) loads f and u of l + wave + WV i, and the
  // wave's G rows as one run of doubles (m' >= L, and l < m' before the
  // table: zeros; l < m' else: rows of m' - 1, finite, met by a chain value
  // of zero)
  unsigned so = (unsigned)((lb + wave) * L + m);
  unsigned ro = mp < L ? (unsigned)((int)(rowA(mp, mp, L) + (lb - mp)) * W + lane) * 8u : kBufOut;
  double2 gf[NF];
  double gu[NF], gr[NR];
  auto fetch = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < NF; ++i) {
      const unsigned e = so + (unsigned)(WV * i * L);
      gf[i] = __builtin_bit_cast(double2, __builtin_amdgcn_raw_buffer_load_b128(fres, e * 16u, 0, 0));
      gu[i] = __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(ures, e * 8u, 0, 0));
    }
#pragma unroll
    for (int i = 0; i < NR; ++i)
      gr[i] = __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(rres, ro + 512u * i, 0, 0));
    so += (unsigned)(G * L);
    ro += mp < L ? G * W * 8u : 0u;
  };
  int bf = 0;  // buffer being read
  auto put = [&](int b) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < NF; ++i) {
      S.f[b][wave + WV * i][lane] = gf[i];
      S.u[b][wave + WV * i][lane] = gu[i];
    }
#pragma unroll
    for (int i = 0; i < NR; ++i)
      if (64 * i + 64 <= G * W || lane < G * W - 64 * i) S.r[b][wave][64 * i + lane] = gr[i];
  };
  fetch();
  const double st = m < L && mp < L ? lchain_start(a.S0, mp, m) : 0.0;
  const double md = (double)m, m2 = md * md;
  double d = 0.0, dp = 0.0;
  double rm = (double)lb * lb - m2;
  rm = rm > 0.5 ? sqrt(rm) : 0.0;  // r_m(lb)
  // E, O sums [parity of l][slot][column]
  double2 acc[2][2][NH];
#pragma unroll
  for (int q = 0; q < 2; ++q)
#pragma unroll
    for (int s = 0; s < 2; ++s)
#pragma unroll
      for (int h = 0; h < NH; ++h) acc[q][s][h] = make_double2(0.0, 0.0);
  const int sgn = ((mp & 1) ^ a.rho) & 1;  // 0: X = E, Z = O; 1: X = O, Z = E
  put(0);
  lds_barrier();

  auto chain = [&](double uu, double r, int l) __attribute__((always_inline)) {
    const double l1 = (double)(l + 1);
    const double a2 = l1 * l1 - m2;
    const double dn = uu * row_rec(r, md * d, rm * dp);
    dp = d;
    d = dn;
    rm = a2 * uu;
  };
  // G values of l in which no scale ends; START while a chain of the wave may
  // start in them.  The operands of the next l are read one l ahead.
  auto group = [&](auto start, int l) __attribute__((always_inline)) {
    fetch();
    double2 f = S.f[bf][0][lane];
    double uu = S.u[bf][0][lane], r = S.r[bf][wave][lane & 15];
#pragma unroll
    for (int u = 0; u < G; ++u) {
      double2 fn = f;
      double un = uu, rn = r;
      if (u + 1 < G) {
        fn = S.f[bf][u + 1][lane];
        un = S.u[bf][u + 1][lane];
        rn = S.r[bf][wave][(u + 1) * W + (lane & 15)];
      }
      if constexpr (decltype(start)::value) {
        if (l + u == l0) d = st;
      }
      const double ar = d * f.x, ai = d * f.y;
      fma_row<2>(acc[u & 1][0], r, ar, ai);
      fma_row<2 + NH>(acc[u & 1][1], r, ar, ai);
      chain(uu, r, l + u);
      f = fn;
      uu = un;
      r = rn;
      __builtin_amdgcn_sched_barrier(0);
    }
    put(bf ^ 1);
    bf ^= 1;
    lds_barrier();
  };
  // G values of l in which a scale ends, one l at a time (both parities' sums
  // take the column, one of them times zero), with the only copy of the flush
  auto group_end = [&](int lg, int ev) __attribute__((always_inline)) {
    fetch();
    // the arguments that only this path needs are read again here, through a
    // pointer the compiler cannot trace, so that the l loop holds no scalar
    // register for them
    auto *ka = (const AnaParArgs __attribute__((address_space(4))) *)__builtin_amdgcn_kernarg_segment_ptr();
    asm volatile("" : "+s"(ka));
#pragma unroll 1
    for (int u = 0; u < G; ++u) {
      const int l = lg + u;
      const bool end = (ev >> u) & 1;
      // the scales ending here: hi and plane offset of slots 0, 1 (hi = 0: none)
      const ciptr er = as_const(ka->ends) + 8 * l;
      int e[6] = {0, 0, 0, 0, 0, 0};
      if (end) {
#pragma unroll
        for (int i = 0; i < 6; ++i) e[i] = er[i];
      }
      const double2 f = S.f[bf][u][lane];
      const double uu = S.u[bf][u][lane], r = S.r[bf][wave][u * W + (lane & 15)];
      if (l == l0) d = st;
      const double ar = d * f.x, ai = d * f.y;
      const double re = (u & 1) ? 0.0 : r, ro1 = (u & 1) ? r : 0.0;
      fma_row<2>(acc[0][0], re, ar, ai);
      fma_row<2 + NH>(acc[0][1], re, ar, ai);
      fma_row<2>(acc[1][0], ro1, ar, ai);
      fma_row<2 + NH>(acc[1][1], ro1, ar, ai);
      chain(uu, r, l);
      if (!end) continue;
#pragma unroll
      for (int s = 0; s < 2; ++s) {
        const int hj = e[s];
        if (hj == 0) continue;
        if (mp < hj) {
          const long long plane = (long long)hj * hj;
          double2 *dst =
              ka->Tg + (((long long)e[3 + 2 * s] << 32) | (unsigned)e[2 + 2 * s]) + (long long)mp * hj + m;
          const double *cg = &S.cg[0][0][0] + sgn * (NH + 1) * 2 * NH;
          const int N = ka->N, gn = N >> 1;
#pragma unroll 1
          for (int g = 0; g <= gn; ++g, cg += 2 * NH) {
            double2 X = make_double2(0.0, 0.0), Y = make_double2(0.0, 0.0);
#pragma unroll
            for (int h = 0; h < NH; ++h) {
              const double ce = cg[h], co = cg[NH + h];
              X.x = fma(ce, acc[0][s][h].x, X.x);
              X.y = fma(ce, acc[0][s][h].y, X.y);
              Y.x = fma(co, acc[1][s][h].x, Y.x);
              Y.y = fma(co, acc[1][s][h].y, Y.y);
            }
            // Y_g = R + i I, Y_{N-g} = R - i I
            const double2 R = sgn ? Y : X, I = sgn ? X : Y;
            if (m < hj) {
              dst[g * plane] = make_double2(R.x - I.y, R.y + I.x);
              if (g > 0 && 2 * g < N) dst[(N - g) * plane] = make_double2(R.x + I.y, R.y - I.x);
            }
          }
        }
#pragma unroll
        for (int q = 0; q < 2; ++q)
#pragma unroll
          for (int h = 0; h < NH; ++h) acc[q][s][h] = make_double2(0.0, 0.0);
      }
    }
    put(bf ^ 1);
    bf ^= 1;
    lds_barrier();
  };
  const int lst = (max(mpb + WV - 1, m0 + 63) & ~(G - 1)) + G;  // no chain starts from here on
  for (int l = lb; l < L;) {
    const int ln = as_const(a.gnext)[l / G];  // next group in which a scale ends
    const int la = min(ln, lst);
    for (; l < la; l += G) group(std::true_type(), l);
    for (; l < ln; l += G) group(std::false_type(), l);
    if (l >= L) break;
    group_end(l, as_const(a.gev)[l / G]);
    l += G;
  }
}

// rows of the kernel above from the general analysis rows: A, Bc and the
// columns n >= 0 of both slots
__global__ void k_par_rows(long long nrows, int NCa, int NH, int c0, const double *__restrict__ Ba,
                           double *__restrict__ out) {
  const long long id = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  const int W = 2 * NH + 2;
  const long long r = id / W;
  const int i = (int)(id - r * W);
  if (r >= nrows) return;
  const double *row = Ba + r * (2 + 2 * NCa);
  out[id] = i < 2 ? row[i] : i < 2 + NH ? row[2 + c0 + i - 2] : row[2 + NCa + c0 + i - 2 - NH];
}

}  // namespace

int par_rows(long long nrows, int NCa, int NH, int c0, const double *Ba, double *out, hipStream_t st) {
  const long long n = nrows * (2 * NH + 2);
  hipLaunchKernelGGL(k_par_rows, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, nrows, NCa, NH, c0, Ba, out);
  S2DW_HIP_CHECK(hipGetLastError());
  return kErrNone;
}

int par_contract(const AnaParArgs &a, int NH, hipStream_t st) {
  const dim3 grid(((a.L + WV - 1) / WV) * ((a.L + 63) / 64)), block(64 * WV);
  switch (NH) {
    case 1: hipLaunchKernelGGL(k_ana_contract_par<1>, grid, block, 0, st, a); break;
    case 2: hipLaunchKernelGGL(k_ana_contract_par<2>, grid, block, 0, st, a); break;
    case 3: hipLaunchKernelGGL(k_ana_contract_par<3>, grid, block, 0, st, a); break;
    case 4: hipLaunchKernelGGL(k_ana_contract_par<4>, grid, block, 0, st, a); break;
    default: return kErrArgInvalid;
  }
  S2DW_HIP_CHECK(hipGetLastError());
  return kErrNone;
}

}  // namespace s2dw
