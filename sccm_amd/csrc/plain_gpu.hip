// plain_gpu.hip -- the plain-form mesh-point kernels of the PNAMP path for
// MI355X (gfx950): states of any kind (proton-neutron mixing included), FP64.
//
// One mesh point = (pair, Euler point, gauge angles phi_p, phi_n).  With
// A = diag(e^{i phi_p} R, e^{i phi_n} R) (UVphiomega, Codes/PNAMP/PNAMP_Proj.f90:396-455)
// and D = diag(e^{i phi_s(a)}) every gauge-dependent matrix is a phase
// rescaling of a gauge-independent one:
//   A Z1 A^T          = D M0 D,              M0 = R~ Z1 R~^T
//   T = V0^T A V1 + U0^T A* U1 = sum_s e^{i phi_s} X_s + e^{-i phi_s} Y_s,
//                     X_s = V0^T P_s R~ V1,  Y_s = U0^T P_s R~* U1
//   A V1 = D (R~ V1), A* U1 = D* (R~* U1)
// (R~ = diag(R, R), P_s the projector on species s).  k_plain_setup forms
// M0, X_p, X_n, Y_p, Y_n, R~ V1, R~* U1 once per (pair, Euler point);
// k_plain_gauge then needs only O(n^2) phase work per gauge point before the
// Pfaffian and the inverse.
//
// k_plain_pf: the Pfaffian of the 2n x 2n skew matrix (ZPfaffianF,
// Codes/PNAMP/PNAMP_Proj.f90:218-350), see there.
// k_plain_gauge, one workgroup per gauge point:
//   * T^{-1}: W = [A V1; A* U1] T^{-1} by Gauss-Jordan column operations on the
//     stacked 3n x n matrix [T; A V1; A* U1] (pivot: largest |re|+|im| in the
//     current row of T among unused columns, as IZAMAX; the solution columns
//     come out permuted);
//   * rho = W1 V0^T, kappa10 = W1 U0^T, kappa01 = -W2 V0^T
//     (ROKAPPAphiomega, PNAMP_Proj.f90:459-551) on the FP64 matrix units; rho
//     to LDS, kappa only as A01 = kappa01 - kappa01^T (strict upper) and A10 /
//     4 = (kappa10 - kappa10^T) / 4 (strict lower) of one n x n LDS block, each
//     entry the sum of exactly two LDS atomic adds onto zero (so the result
//     does not depend on their order).
//   * the energy (HFB_Energy_COMPLEX, PNAMP_Energy_OpenMP.f90:5-100) from the
//     regrouped list: (1/4) V [r_ijkl - r_jikl - r_ijlk + r_jilk + d (...)] =
//     V [rho_ki rho_lj - rho_li rho_kj + A01_ij A10_kl / 4] + d (kl <-> ij),
//     exact algebra; entries with a = b or c = d add exactly zero;
//   * <J^2> (ZJ2_0, PNAMP_ME2B.f90:1-152) in the ladder form
//     J.J = Jz Jz + (J+ J- + J- J+)/2, E_kin, Tr rho per species (ZN_0).
#include <hip/hip_runtime.h>

#include <cstdint>
#include <type_traits>

#include "../../include/pnamp_gpu.h"
#include "pnamp_dev.h"
#include "plain_gpu.h"

namespace {

using namespace pnamp_dev;

typedef double d4 __attribute__((ext_vector_type(4)));

constexpr int NOBS = PNAMP_NOBS;
constexpr int NOG_E2 = NOBS + 10;  // per gauge point: observables, then tr_s(Q_mu rho), then orbit traces

// k_plain_gauge's grid of GR x GC threads (see there) and its tiles.
template <int N>
struct PlainCfg {
  static constexpr int GC = N <= 24 ? 8 : 16, GR = N == 64 ? 32 : 16;
  static constexpr int NTH = GR * GC, NW = NTH / 64;
  static constexpr int TR = (3 * N + GR - 1) / GR, TC = (N + GC - 1) / GC, TP = (N + GR - 1) / GR;
  // 16 x 16 output tiles of the densities: [W1; W2] V0^T and W1 U0^T
  static constexpr int MT2 = (2 * N + 15) / 16, MT1 = (N + 15) / 16, NT = (N + 15) / 16;
  static constexpr int JOBS = (MT2 + MT1) * NT, JW = (JOBS + NW - 1) / NW;
  // waves per SIMD the registers are fitted to (LDS: 3 workgroups per CU at n =
  // 40, 2 at n = 44, 1 at n = 64)
  static constexpr int GAUGE_WAVES = N <= 32 ? 4 : (N <= 40 ? 3 : 2);
};

// ------------------------------------------------------------------ setup
struct PSetup {
  int n, h, nalp, ngam, npack, NE, u0;  // NE here and below: Euler points evaluated
  const int2 *ecan;
  const double *alp, *gam, *rtab;
  const int *pk_a, *pk_b, *blk_off, *blk_sz, *blk_base, *twom;
  const int *q0, *q1;
  const double *U, *V, *Z;
  double2 *hoist;  // [unit - u0][7][n*n]: X_p, X_n, Y_p, Y_n, R~V1, R~*U1 (column-major), M0 (row-major)
};

constexpr int RPK = 256;  // packed rotation entries (per species) held in LDS

// One workgroup per (unit, 16 columns): R~ V1, R~* U1 and X, Y of its columns, M0
// of the rows of the same numbers, so a few units still fill the card.  X_s =
// V0^T P_s (R~ V1) and Y_s run on v_mfma_f64_16x16x4, a wave per 16 rows (a V0
// element is read once per 16 columns instead of once per column, the columns
// from LDS).  With one workgroup per unit and a thread per element, 45 units of
// n = 64 took 224 us and 432 units of n = 40 83 us; now 28 and 46 us.
constexpr int SC = 16, SLD = SC + 1;
__host__ __device__ constexpr size_t setup_lds(int n) { return sizeof(double2) * (2 * (size_t)n * SLD + SC * ((size_t)n + 1)); }

__global__ __launch_bounds__(256) void k_plain_setup(PSetup p) {
  extern __shared__ double2 lds[];
  __shared__ double2 sR[RPK], ea[32], eg[32];
  __shared__ short m_off[32], m_sz[32], m_base[32];
  const int tid = threadIdx.x, n = p.n, h = p.h, nn = n * n;
  const int ul = blockIdx.x, u = p.u0 + ul, ip = u / p.NE, iang = p.ecan[u - ip * p.NE].x;
  const int c0 = blockIdx.y * SC, cw = min(SC, n - c0);
  const int ig = iang % p.ngam, ia = (iang / p.ngam) % p.nalp, ib = iang / (p.ngam * p.nalp);
  const double alp = p.alp[ia], gam = p.gam[ig];
  const int q0 = p.q0[ip], q1 = p.q1[ip];
  const double *V0 = p.V + (size_t)q0 * nn, *U0 = p.U + (size_t)q0 * nn;
  const double *V1 = p.V + (size_t)q1 * nn, *U1 = p.U + (size_t)q1 * nn, *Z1 = p.Z + (size_t)q1 * nn;
  double2 *out = p.hoist + (size_t)ul * 7 * nn;
  double2 *const sA = lds, *const sB = lds + n * SLD, *const sZ = lds + 2 * n * SLD;  // R~V1, R~*U1 (row * SLD + column), rows of R~ Z1
  // R(a, b) = exp(-i alp m_a) d(beta)_{ab} exp(-i gam m_b) (ROTATION_MAT, PNAMP_Proj.f90:83-136)
  for (int i = tid; i < h; i += 256) {
    m_off[i] = (short)p.blk_off[i];
    m_sz[i] = (short)p.blk_sz[i];
    m_base[i] = (short)p.blk_base[i];
    ea[i] = cexpi(-alp * 0.5 * p.twom[i]);
    eg[i] = cexpi(-gam * 0.5 * p.twom[i]);
  }
  __syncthreads();
  for (int e = tid; e < p.npack; e += 256)
    sR[e] = cscale(p.rtab[(size_t)ib * p.npack + e], cmul(ea[p.pk_a[e]], eg[p.pk_b[e]]));
  __syncthreads();
  // R~ V1, R~* U1 (block-sparse rows), 16 columns
  for (int e = tid; e < n * cw; e += 256) {
    const int jl = e / n, i = e - jl * n, j = c0 + jl;
    const int sp = i >= h, il = i - sp * h;
    const int off = m_off[il], sz = m_sz[il], base = m_base[il];
    double2 a = cz(), b = cz();
    for (int k = 0; k < sz; ++k) {
      const double2 r = sR[base + (il - off) + k * sz];
      const int row = sp * h + off + k;
      rfma(a, V1[row + j * n], r);
      rfma(b, U1[row + j * n], cconj(r));
    }
    sA[i * SLD + jl] = a;
    sB[i * SLD + jl] = b;
    out[4 * nn + i + j * n] = a;
    out[5 * nn + i + j * n] = b;
  }
  // rows c0 .. of R~ Z1
  for (int e = tid; e < n * SC; e += 256) {
    const int il0 = e & (SC - 1), j = e >> 4, i = c0 + il0;
    if (il0 >= cw) continue;
    const int sp = i >= h, il = i - sp * h;
    const int off = m_off[il], sz = m_sz[il], base = m_base[il];
    double2 a = cz();
    for (int k = 0; k < sz; ++k) rfma(a, Z1[(sp * h + off + k) + j * n], sR[base + (il - off) + k * sz]);
    sZ[il0 * (n + 1) + j] = a;
  }
  __syncthreads();
  // M0 = (R~ Z1) R~^T, row-major output: consecutive threads, consecutive j
  for (int e = tid; e < n * cw; e += 256) {
    const int il0 = e / n, j = e - il0 * n;
    const int sp = j >= h, jl = j - sp * h;
    const int off = m_off[jl], sz = m_sz[jl], base = m_base[jl];
    double2 a = cz();
    for (int k = 0; k < sz; ++k) cfma(a, sZ[il0 * (n + 1) + sp * h + off + k], sR[base + (jl - off) + k * sz]);
    out[6 * nn + (size_t)(c0 + il0) * n + j] = a;
  }
  // X_s(a, c) = sum_{i in s} V0(i, a) (R~V1)(i, c), Y_s likewise with U0, R~*U1:
  // lane l: A row a = l % 16, B column c = l % 16, both i = l / 16 of the step
  const int lane = tid & 63, l16 = lane & 15, lk = lane >> 4;
  for (int m = tid >> 6; m < (n + 15) / 16; m += 4) {
    const int ar = min(16 * m + l16, n - 1);
    for (int s = 0; s < 2; ++s) {
      d4 xr = {0.0, 0.0, 0.0, 0.0}, xi = xr, yr = xr, yi = xr;
      for (int k0 = 0; k0 < h; k0 += 4) {
        const int k = k0 + lk, i = s * h + min(k, h - 1);
        const double z = (k < h) ? 1.0 : 0.0;
        const double av = z * V0[i + ar * n], au = z * U0[i + ar * n];
        const double2 bv = sA[i * SLD + min(l16, cw - 1)], bu = sB[i * SLD + min(l16, cw - 1)];
        xr = __builtin_amdgcn_mfma_f64_16x16x4f64(av, bv.x, xr, 0, 0, 0);
        xi = __builtin_amdgcn_mfma_f64_16x16x4f64(av, bv.y, xi, 0, 0, 0);
        yr = __builtin_amdgcn_mfma_f64_16x16x4f64(au, bu.x, yr, 0, 0, 0);
        yi = __builtin_amdgcn_mfma_f64_16x16x4f64(au, bu.y, yi, 0, 0, 0);
      }
#pragma unroll
      for (int v = 0; v < 4; ++v) {  // D: row 4 v + l / 16, column l % 16
        const int r = 16 * m + 4 * v + lk;
        if (r < n && l16 < cw) {
          out[s * nn + r + (c0 + l16) * n] = make_double2(xr[v], xi[v]);
          out[(2 + s) * nn + r + (c0 + l16) * n] = make_double2(yr[v], yi[v]);
        }
      }
    }
  }
}

// ------------------------------------------------------------------ gauge point
struct PGauge {
  int n, h, nphi, NE, ngc, nl, lbytes, nob2, nog, u0, nwg;
  const int2 *gcls;  // [ngc]: gauge indices of the pairs evaluated
  double cscale, e0;
  const int *q0, *q1;
  const double *U, *V, *Z;
  const double2 *hoist;
  const double *mtab, *t1b;
  const uint4 *lofs;
  const double *lme;
  const double *q2;
  const int4 *orbp;
  double2 *gout;  // [unit - u0][ngc][nog]: observables per gauge point, not yet norm-weighted
  int *gst;       // [unit - u0][ngc]
  double2 *gpf;   // [unit - u0][ngc]: Pfaffian of the gauge point's skew matrix
};

template <int N>
__host__ __device__ constexpr size_t gauge_misc_bytes() {
  // pivots [2] (16 B), reductions [NW][20], ladder table [N] (8 B), pivot
  // columns [2] and the solution order [N] (4 B): 1,160 B at N = 40, so three
  // workgroups of n = 40 (53,640 B) share a CU's 160 KB
  return 32 + 160 * PlainCfg<N>::NW + 8 * N + 8 + 4 * N;
}

template <int CTRL>
__device__ __forceinline__ double dpp_quad_f64(double v) {  // DPP move of a double
  const long long b = __double_as_longlong(v);
  const int lo = __builtin_amdgcn_update_dpp(0, (int)b, CTRL, 0xF, 0xF, false);
  const int hi = __builtin_amdgcn_update_dpp(0, (int)(b >> 32), CTRL, 0xF, 0xF, false);
  return __longlong_as_double(((long long)hi << 32) | (long long)(unsigned)lo);
}

// Pfaffian per gauge point: S = cscale [[D M0 D, -1], [1, -Z0]] (Pfaf_Over, 2n x
// 2n skew) by Parlett-Reid elimination, the pivot of row r = 2k the largest
// |S(r, c)|, c > r; index c exchanged with r + 1 (sign -1), rank-2 Schur update.
// The zero rule is ZPfaffianF's: Pf = 0 where no entry left exceeds 1e-13 in
// modulus.  ZPfaffianF pivots on the largest entry of the whole remaining
// matrix, a search of every entry in every step; a pivot that is the largest
// of its row bounds the multipliers S(j, r) / s by one as well.
//
// 2D block-cyclic layout over a G x G grid of threads (one wave for 2n <= 48,
// four above): thread (a, b) holds S(a + G p, b + G q) in slot (p, q), p <= q < T
// = ceil(2N / G); the diagonal slots hold the whole block (both triangles), so
// a row or column of the matrix is T slots of one row or column of threads and
// nothing is indexed at run time but the slot column of c (a uniform switch).
// Step r: the wave that holds rows r, r + 1 finds c, and writes R = row r / s
// and A = row r + 1; then every wave knows c and writes column c (C, below the
// diagonal block from row c with the sign); then row and column c take the
// place of r + 1 and the trailing slots get S(i, j) += R_i C_j - C_i R_j.  Two
// barriers per step (none for one wave): R and A of the next step go to the
// other half of their buffers while slow waves still update.  Entries that
// left the trailing matrix are updated on with values nobody reads.
// Bound by VALU issue (G = 8) and the wait of each step for its pivot chain (G =
// 16, hidden by the other workgroups of the CU: n = 40 at three waves per SIMD
// 77 ns, at four, spilling 20 bytes, 64 ns).  Against full pivoting with the
// triangle spread entry by entry over 3n / 32 waves, per gauge point on the whole
// card: n = 24 41 -> 15 ns, n = 40 168 -> 64 ns, n = 44 570 -> 97 ns, n = 64 1,230 ->
// 300 ns.
template <int N>
struct PfCfg {
  static constexpr int G = (2 * N <= 48) ? 8 : 16;
  static constexpr int NT = G * G;
  static constexpr int T = (2 * N + G - 1) / G, NS = T * (T + 1) / 2;
  // slots, held R and C, addresses: the waves per SIMD that fit (512 / waves
  // registers).  Of the size classes only N = 40 lies between four waves' 128 and
  // the line's 136: 128 registers and 20 bytes spilled, faster than three waves
  // (above); the others take 103 (16, 32: 4 waves), 166 (24, 48: 3), 248 (64: 2)
  // and spill nothing
  static constexpr int REGS = 4 * NS + 8 * T + 36;
  static constexpr int WV = REGS <= 102 ? 5 : (REGS <= 136 ? 4 : (REGS <= 168 ? 3 : 2));
};

template <int N>
__global__ __launch_bounds__(PfCfg<N>::NT) __attribute__((amdgpu_waves_per_eu(PfCfg<N>::WV))) void k_plain_pf(PGauge p) {
  using C_ = PfCfg<N>;
  constexpr int G = C_::G, T = C_::T, NS = C_::NS, KB = (2 * N <= 64) ? 6 : 7;
  __shared__ double2 vR[2][G * T], vA[2][G * T], vC[G * T], sS[2];
  __shared__ int sC[2];
  const int n = p.n, h = p.h, nn = n * n, N2 = 2 * n;
  const int tid = threadIdx.x, wave = tid >> 6;
  const int a = tid / G, b = tid % G;
  const unsigned L = (blockIdx.x & 7u) * (gridDim.x >> 3) + (blockIdx.x >> 3);
  if (L >= (unsigned)p.nwg) return;
  const int ng = p.ngc;
  const int g = (int)(L % (unsigned)ng), ul = (int)(L / (unsigned)ng), u = p.u0 + ul;
  const int q0 = p.q0[u / p.NE];
  const int2 gl = p.gcls[g];
  const double2 ep = cexpi((2.0 * M_PI / p.nphi) * gl.x), en = cexpi((2.0 * M_PI / p.nphi) * gl.y);
  const double2 *const M0 = p.hoist + (size_t)ul * 7 * nn + 6 * nn;  // row-major
  const double *const Z0 = p.Z + (size_t)q0 * nn;
  auto SI = [](int pp, int qq) { return pp * T - pp * (pp - 1) / 2 + (qq - pp); };
  double2 sv[NS];
  {
    // every load unconditional (indices clamped into the blocks), the block chosen by selects
    const double2 e2p = cmul(ep, ep), epn = cmul(ep, en), e2n = cmul(en, en);
#pragma unroll
    for (int pp = 0; pp < T; ++pp)
#pragma unroll
      for (int qq = pp; qq < T; ++qq) {
        const int i = a + G * pp, j = b + G * qq, lo = min(i, j), hi = max(i, j);
        const int ml = min(lo, n - 1), mh = min(hi, n - 1);
        const double2 m0v = M0[(size_t)ml * n + mh];
        const double z0v = Z0[min(max(lo - n, 0), n - 1) + (size_t)min(max(hi - n, 0), n - 1) * n];
        const int sidx = (ml >= h) + (mh >= h);
        double2 up = cmul(sidx == 0 ? e2p : (sidx == 1 ? epn : e2n), m0v);
        if (hi >= n) up = (lo < n) ? make_double2((hi - n == lo) ? -1.0 : 0.0, 0.0) : make_double2(-z0v, 0.0);
        up = (hi < N2 && lo != hi) ? cscale(p.cscale, up) : cz();
        sv[SI(pp, qq)] = (i < j) ? up : cneg(up);
      }
  }
  double2 pf = make_double2(1.0, 0.0);
  bool zero = false;
#pragma unroll
  for (int P = 0; P < T; ++P) {
    if (zero || G * P >= N2 - 2) break;
    for (int t = 0; t < G / 2 && G * P + 2 * t < N2 - 2; ++t) {
      const int r = G * P + 2 * t, par = t & 1;  // (G / 2 is even: the halves alternate across P too)
      double2 *const R = vR[par], *const A = vA[par];
      if (wave == (2 * t * G) >> 6) {  // rows r (a = 2t) and r + 1 are this wave's
        const int base = (2 * t * G) & 63;  // its lane of thread (2t, 0)
        unsigned key = 0u;
#pragma unroll
        for (int q = P; q < T; ++q) {
          const int j = b + G * q;
          const double2 v = sv[SI(P, q)];
          const unsigned kk = pivot_key_hi<KB>(v.x * v.x + v.y * v.y, j);
          key = (j > r && j < N2) ? max(key, kk) : key;
        }
        key = oct_umax(key);
        if (G == 16) key = dpp_umax<0x140, 0xF>(key);  // row_mirror
        key = (unsigned)__builtin_amdgcn_readlane((int)key, base);
        const int c = (1 << KB) - 1 - (int)(key & ((1u << KB) - 1u));
        const int Q = c / G, src = base + c % G;
        double2 s = cz();
#pragma unroll
        for (int qq = P; qq < T; ++qq) {
          if (qq == Q) {
            const double2 v = sv[SI(P, qq)];
            const long long bx = __double_as_longlong(v.x), by = __double_as_longlong(v.y);
            s.x = __longlong_as_double(((long long)__builtin_amdgcn_readlane((int)(bx >> 32), src) << 32) |
                                       (unsigned)__builtin_amdgcn_readlane((int)bx, src));
            s.y = __longlong_as_double(((long long)__builtin_amdgcn_readlane((int)(by >> 32), src) << 32) |
                                       (unsigned)__builtin_amdgcn_readlane((int)by, src));
          }
        }
        const double2 inv = crecip_nr(s);
        if (a == 2 * t) {
#pragma unroll
          for (int q = P; q < T; ++q) {
            const double2 v = cmul(sv[SI(P, q)], inv);
            R[b + G * q] = v;
          }
          // position c takes index r + 1 (thread (2t, 2t + 1) holds it; after the row's own stores)
          if (b == 2 * t + 1) R[c] = cmul(sv[SI(P, P)], inv);
        }
        if (a == 2 * t + 1) {
#pragma unroll
          for (int q = P; q < T; ++q) A[b + G * q] = sv[SI(P, q)];
        }
        if (a == 2 * t && b == 0) {
          sC[par] = c;
          sS[par] = s;
        }
      }
      __syncthreads();
      const int c = __builtin_amdgcn_readfirstlane(sC[par]);
      const double2 s = sS[par];
      const double s2 = s.x * s.x + s.y * s.y;
      if (__builtin_amdgcn_readfirstlane((int)!(s2 > 1.0e-26))) {
        // |pivot| <= 1e-13: Pf = 0 if no entry left is larger (or the row is zero)
        bool big = false;
#pragma unroll
        for (int pp = P; pp < T; ++pp)
#pragma unroll
          for (int q = pp; q < T; ++q) {
            const int i = a + G * pp, j = b + G * q;
            const double2 v = sv[SI(pp, q)];
            big = big || (i >= r && j > i && j < N2 && v.x * v.x + v.y * v.y > 1.0e-26);
          }
        const int any = __syncthreads_or(big ? 1 : 0);
        if (!any || !(s2 > 1.0e-290)) {
          zero = true;
          break;
        }
      }
      const bool swap = c != r + 1;
      pf = cmul(pf, swap ? cneg(s) : s);
      const int Q = c / G, cg = c % G;
      // column c of the trailing matrix -> C (position c: the exchanged S(r + 1, c))
      const double2 ac = A[c];
#pragma unroll
      for (int qq = P; qq < T; ++qq) {
        if (qq == Q) {
          if (b == cg) {
#pragma unroll
            for (int pp = P; pp <= qq; ++pp) {
              double2 v = sv[SI(pp, qq)];
              v.x = (a + G * pp == c) ? ac.x : v.x;
              v.y = (a + G * pp == c) ? ac.y : v.y;
              vC[a + G * pp] = v;
            }
          }
          if (a == cg) {
#pragma unroll
            for (int q = qq + 1; q < T; ++q) vC[b + G * q] = cneg(sv[SI(qq, q)]);
          }
          // exchange: S'(x, c) = S(x, r + 1) = -A[x], S'(c, y) = A[y]
          if (swap) {
            if (b == cg) {
#pragma unroll
              for (int pp = P; pp <= qq; ++pp) sv[SI(pp, qq)] = cneg(A[a + G * pp]);
            }
            if (a == cg) {
#pragma unroll
              for (int q = qq; q < T; ++q) sv[SI(qq, q)] = A[b + G * q];
            }
          }
        }
      }
      __syncthreads();
      double2 Rj[T], Cj[T];
#pragma unroll
      for (int q = P; q < T; ++q) {
        Rj[q] = R[b + G * q];
        Cj[q] = vC[b + G * q];
      }
#pragma unroll
      for (int pp = P; pp < T; ++pp) {
        const double2 Ri = R[a + G * pp], Ci = vC[a + G * pp];
#pragma unroll
        for (int q = pp; q < T; ++q) {
          cfms(sv[SI(pp, q)], Ci, Rj[q]);
          cfma(sv[SI(pp, q)], Ri, Cj[q]);
        }
      }
    }
  }
  // the last 2 x 2 block: S(2n - 2, 2n - 1)
  const int lt = ((N2 - 2) % G) * G + (N2 - 1) % G;
  if (tid == lt) {
    double2 v = cz();
#pragma unroll
    for (int q = 0; q < T; ++q)
      if (q == (N2 - 2) / G) v = sv[SI(q, q)];
    p.gpf[L] = zero ? cz() : cmul(pf, v);
  }
}

// The stacked matrix [T; A V1; A* U1] is block-cyclic over the GR x GC threads:
// thread (a, b) holds rows a + GR p, columns b + GC q in slot (p, q).  Step k
// (row k of T: thread row k % GR, a compile-time slot row): the wave that holds
// row k finds the pivot column c and writes R = row k / pivot (R_c = -1 /
// pivot); then every wave knows c and writes column c (C), which starts again
// from zero; then slot (p, q) -= C R, from TR + TC LDS reads for TR TC products.
// Two barriers per step; R has two halves for the waves still updating.  Slot
// rows of T above row k are left out.  (With a row per two lanes and its
// columns in registers the pivot column was picked by selects over all register
// columns and every lane read the whole of row k.)
// The densities are products with the real V0, U0: W goes to LDS in solution
// order and 16 x 16 tiles of [W1; W2] V0^T and W1 U0^T run on
// v_mfma_f64_16x16x4 (its rate equals the vector units', but an operand is read
// once per 16 results: the vector form read V0 once per result pair and thread).
// Per gauge point on the whole card, with the list (a row per two lanes, vector
// densities -> this): n = 24 70 -> 34 ns, n = 40 292 -> 163 ns, n = 44 688 -> 211
// ns, n = 64 1,960 -> 785 ns; of n = 40's, loads 15 %, Gauss-Jordan 38 % (VALU
// issue, half of it multiply-adds, and the barriers), densities 12 %, the list
// and the sums 27 % (LDS gathers).
template <int N, bool E2>
__global__ __launch_bounds__(PlainCfg<N>::NTH) __attribute__((amdgpu_waves_per_eu(PlainCfg<N>::GAUGE_WAVES))) void k_plain_gauge(PGauge p) {
  using C = PlainCfg<N>;
  constexpr int NTH = C::NTH, NW = C::NW, GR = C::GR, GC = C::GC, TR = C::TR, TC = C::TC, TP = C::TP, JW = C::JW;
  extern __shared__ double2 lds[];
  const int n = p.n, h = p.h, nn = n * n, ld = n + 1;
  double2 *const R = lds;              // rho, column-major with leading dimension n + 1
  double2 *const AB = lds + n * ld;    // A01 (i < j at i + j (n + 1)), A10 / 4 (i < j at j + i (n + 1))
  char *const misc = (char *)(AB + n * ld);
  double2 *const sS = (double2 *)misc;             // pivots [2]
  double *const red = (double *)(misc + 32);
  double *const mt = red + 20 * NW;                // [2][N / 2]: m, <m+1|J+|m> per species-local state
  int *const sC = (int *)(mt + N);                 // pivot columns [2]
  int *const kinv = sC + 2;                        // [N]: solution index of each column
  // Gauss-Jordan vectors, then W, at the front (rho and the A-block come later)
  double2 *const vR = lds, *const vC = lds + 2 * GC * TC, *const W = lds;

  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  // XCD-aware order: the ngc workgroups of one unit stay on one XCD (and
  // its L2, where the unit's setup matrices are); gridDim.x is a multiple of 8
  const unsigned L = (blockIdx.x & 7u) * (gridDim.x >> 3) + (blockIdx.x >> 3);
  if (L >= (unsigned)p.nwg) return;
  const int ng = p.ngc;
  const int g = (int)(L % (unsigned)ng), ul = (int)(L / (unsigned)ng), u = p.u0 + ul;
  const int ip = u / p.NE;
  const int q0 = p.q0[ip];
  const int2 gl = p.gcls[g];
  const double2 ep = cexpi((2.0 * M_PI / p.nphi) * gl.x), en = cexpi((2.0 * M_PI / p.nphi) * gl.y);
  const double2 *const H = p.hoist + (size_t)ul * 7 * nn;

  for (int i = tid; i < 2 * h; i += NTH) mt[i] = p.mtab[i];
  // ---------------------------------------------------------------- Gauss-Jordan
  const int a = tid / GC, b = tid % GC;
  double2 sv[TR][TC];
  {
    const double2 *Xp = H, *Xn = H + nn, *Yp = H + 2 * nn, *Yn = H + 3 * nn, *RV1 = H + 4 * nn;  // (R~* U1 after R~ V1)
    // unconditional loads (indices clamped, the value chosen by selects), so a
    // slot row's loads are in flight together; slot rows below n / GR hold rows
    // of T only, those from (n - 1) / GR + 1 on none
#pragma unroll
    for (int pp = 0; pp < TR; ++pp) {
      const int r = a + GR * pp;
      const int kind = (r < n) ? 0 : (r < 2 * n) ? 1 : 2;
      const int ri = min(r - kind * n, n - 1);
      const bool ok = r < 3 * n;
      const double2 es = (ri >= h) ? en : ep;
      const double2 ph = (kind == 1) ? es : cconj(es);
#pragma unroll
      for (int q = 0; q < TC; ++q) {
        const int c = b + GC * q;
        const unsigned o = (unsigned)(ri + min(c, n - 1) * n) * 16u;  // (a 32-bit offset to uniform bases)
        auto at = [&](const double2 *m) { return *(const double2 *)((const char *)m + o); };
        auto atw = [&](unsigned x) { return *(const double2 *)((const char *)RV1 + (o + x)); };
        double2 t = cz(), w = cz();
        if (GR * pp < n) {  // (uniform)
          t = cmul(ep, at(Xp));
          cfma(t, en, at(Xn));
          cfma(t, cconj(ep), at(Yp));
          cfma(t, cconj(en), at(Yn));
        }
        if (GR * pp + GR > n) w = cmul(ph, atw(kind == 2 ? 16u * (unsigned)nn : 0u));
        const bool in = ok && c < n;
        sv[pp][q].x = in ? (kind == 0 ? t.x : w.x) : 0.0;
        sv[pp][q].y = in ? (kind == 0 ? t.y : w.y) : 0.0;
      }
      // a row's values are made before the next row's loads are issued (the
      // scheduler would otherwise issue all loads first and spill)
#pragma unroll
      for (int q = 0; q < TC; ++q) __asm__ volatile("" : "+v"(sv[pp][q].x), "+v"(sv[pp][q].y) : : "memory");
    }
  }
  int info = 0;
  unsigned long long used = 0ull;
#pragma unroll
  for (int P = 0; P < TP; ++P) {
    for (int t = 0; t < GR && GR * P + t < n; ++t) {
      const int k = GR * P + t, par = t & 1;  // (GR is even: the halves alternate across P too)
      double2 *const Rk = vR + par * GC * TC;
      if (wave == (t * GC) >> 6) {
        const int base = (t * GC) & 63;
        // pivot: largest |re| + |im| among unused columns, ties to the smaller
        // column (a NaN entry wins)
        unsigned key = 0u;
#pragma unroll
        for (int q = 0; q < TC; ++q) {
          const int j = b + GC * q;
          const unsigned kk = pivot_key_hi<6>(cabs1(sv[P][q]), j);
          key = (j < n && !((used >> j) & 1ull)) ? max(key, kk) : key;
        }
        key = oct_umax(key);
        if (GC == 16) key = dpp_umax<0x140, 0xF>(key);  // row_mirror
        key = (unsigned)__builtin_amdgcn_readlane((int)key, base);
        const int c = 63 - (int)(key & 63u), Q = c / GC, src = base + c % GC;
        double2 s = cz();
#pragma unroll
        for (int qq = 0; qq < TC; ++qq) {
          if (qq == Q) {
            const double2 v = sv[P][qq];
            const long long bx = __double_as_longlong(v.x), by = __double_as_longlong(v.y);
            s.x = __longlong_as_double(((long long)__builtin_amdgcn_readlane((int)(bx >> 32), src) << 32) |
                                       (unsigned)__builtin_amdgcn_readlane((int)bx, src));
            s.y = __longlong_as_double(((long long)__builtin_amdgcn_readlane((int)(by >> 32), src) << 32) |
                                       (unsigned)__builtin_amdgcn_readlane((int)by, src));
          }
        }
        const double2 inv = crecip_nr(s);
        if (a == t) {
#pragma unroll
          for (int q = 0; q < TC; ++q) Rk[b + GC * q] = cmul(sv[P][q], inv);
          if (b == 0) {  // (after the row's own stores)
            Rk[c] = cneg(inv);
            sC[par] = c;
            sS[par] = s;
          }
        }
      }
      __syncthreads();
      const int c = __builtin_amdgcn_readfirstlane(sC[par]), Q = c / GC, cg = c % GC;
      used |= 1ull << c;
      if (tid == 0) {
        const double2 s = sS[par];
        if (s.x == 0.0 && s.y == 0.0 && !info) info = k + 1;
        kinv[c] = k;
      }
#pragma unroll
      for (int qq = 0; qq < TC; ++qq) {
        if (qq == Q && b == cg) {
#pragma unroll
          for (int pp = P; pp < TR; ++pp) {
            vC[a + GR * pp] = sv[pp][qq];
            sv[pp][qq] = cz();
          }
        }
      }
      __syncthreads();
      double2 Rj[TC];
#pragma unroll
      for (int q = 0; q < TC; ++q) Rj[q] = Rk[b + GC * q];
#pragma unroll
      for (int pp = P; pp < TR; ++pp) {
        const double2 Ci = vC[a + GR * pp];
#pragma unroll
        for (int q = 0; q < TC; ++q) cfms(sv[pp][q], Ci, Rj[q]);
      }
    }
  }
  __syncthreads();
  // W(row, k) in solution order, rows of W1 then W2, column-major with an odd
  // leading dimension (a row of threads writes 16 columns at once)
#pragma unroll
  for (int pp = 0; pp < TR; ++pp) {
    const int r = a + GR * pp - n;
#pragma unroll
    for (int q = 0; q < TC; ++q) {
      const int c = b + GC * q;
      if (r >= 0 && r < 2 * n && c < n) W[r + kinv[c] * (2 * n + 1)] = sv[pp][q];
    }
  }
  __syncthreads();

  // ---------------------------------------------------------------- densities
  // tile jobs of this wave; lane l: A row l % 16, k = l / 16; B column l % 16
  d4 tre[JW], tim[JW];
  {
    const double *V0 = p.V + (size_t)q0 * nn, *U0 = p.U + (size_t)q0 * nn;
    const double *bp[JW];
    int ar[JW];
#pragma unroll
    for (int w = 0; w < JW; ++w) {
      const int jb = min(wave * JW + w, C::JOBS - 1), j2 = jb - C::MT2 * C::NT;
      const int m = j2 < 0 ? jb % C::MT2 : j2 % C::MT1, nt = j2 < 0 ? jb / C::MT2 : j2 / C::MT1;
      ar[w] = min(16 * m + (lane & 15), 2 * n - 1);
      bp[w] = (j2 < 0 ? V0 : U0) + min(16 * nt + (lane & 15), n - 1);
      tre[w] = tim[w] = d4{0.0, 0.0, 0.0, 0.0};
    }
    for (int k0 = 0; k0 < n; k0 += 4) {  // (n is a multiple of 4: every species has an even number of states)
      const int k = k0 + (lane >> 4);
#pragma unroll
      for (int w = 0; w < JW; ++w) {
        const double bv = bp[w][(size_t)k * n];
        const double2 av = W[ar[w] + k * (2 * n + 1)];
        tre[w] = __builtin_amdgcn_mfma_f64_16x16x4f64(av.x, bv, tre[w], 0, 0, 0);
        tim[w] = __builtin_amdgcn_mfma_f64_16x16x4f64(av.y, bv, tim[w], 0, 0, 0);
      }
    }
  }
  __syncthreads();  // W is read no more
  for (int e = tid; e < n * ld; e += NTH) AB[e] = cz();
  __syncthreads();
#pragma unroll
  for (int w = 0; w < JW; ++w) {
    const int jb = wave * JW + w, j2 = jb - C::MT2 * C::NT;
    const int m = j2 < 0 ? jb % C::MT2 : j2 % C::MT1, nt = j2 < 0 ? jb / C::MT2 : j2 / C::MT1;
    const int j = 16 * nt + (lane & 15);
    if (jb >= C::JOBS || j >= n) continue;
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int r = 16 * m + 4 * v + (lane >> 4);  // D: row 4 v + l / 16, column l % 16
      const double2 x = make_double2(tre[w][v], tim[w][v]);
      if (j2 < 0) {
        if (r < n) {
          R[r + j * ld] = x;  // rho
        } else if (r < 2 * n && r - n != j) {  // kappa01 = -x -> A01
          const int i = r - n;
          const double sg = (i < j) ? -1.0 : 1.0;
          double *dst = (double *)&AB[min(i, j) + max(i, j) * ld];
          atomicAdd(dst, sg * x.x);
          atomicAdd(dst + 1, sg * x.y);
        }
      } else if (r < n && r != j) {  // kappa10 -> A10 / 4
        const double sg = (r < j) ? 0.25 : -0.25;
        double *dst = (double *)&AB[max(r, j) + min(r, j) * ld];
        atomicAdd(dst, sg * x.x);
        atomicAdd(dst + 1, sg * x.y);
      }
    }
  }
  __syncthreads();

  // ---------------------------------------------------------------- observables
  // per element rho(a, b): E_kin t1(b, a); <J^2> rho part -m_a m_b rho(a,b) rho(b,a)
  // - c_a c_b rho(a,b) rho(b-1,a-1) + j_a(j_a+1) d_ab; kappa part
  // (A10/4)(a,b) [m_a m_b A01(a,b) + c_a c_{b+1}/2 A01(a-1,b+1) + c_{a+1} c_b/2 A01(a+1,b-1)]
  // (c_a = <m_a+1|J+|m_a>, 0 for the first state of an orbit, m = j .. -j);
  // traces t_z = sum m_a rho_aa, t_+ = sum c_a rho(a, a-1), t_- = sum c_{a+1} rho(a, a+1)
  double2 ek = cz(), aj = cz(), tz = cz(), tpl = cz(), tmi = cz(), zp = cz(), zn = cz();
  auto a01 = [&](int x, int y) -> double2 {  // branch-free: the stored triangle with the sign, 0 on the diagonal
    const double2 v = AB[min(x, y) + max(x, y) * ld];
    const double sg = (x < y) ? 1.0 : (x > y ? -1.0 : 0.0);
    return cscale(sg, v);
  };
  // b fastest (t1(b, a) contiguous, rho at an odd leading dimension)
  for (int e = tid, x = tid / n, y = tid - x * n; e < nn; e += NTH) {
    const int a = x, b = y;
    const double2 rab = R[a + b * ld], rba = R[b + a * ld];
    const int al = a >= h ? a - h : a, bl = b >= h ? b - h : b;
    const double ma = mt[al], mb = mt[bl], ca = mt[h + al], cb = mt[h + bl];  // c = 0 at the first state of an orbit
    const double ca1 = (a + 1 < n) ? mt[h + (a + 1 >= h ? a + 1 - h : a + 1)] : 0.0;
    const double cb1 = (b + 1 < n) ? mt[h + (b + 1 >= h ? b + 1 - h : b + 1)] : 0.0;
    rfma(ek, p.t1b[b + (size_t)a * n], rab);
    double2 q = cscale(ma * mb, rba);
    rfma(q, ca * cb, R[max(b - 1, 0) + max(a - 1, 0) * ld]);
    cfms(aj, rab, q);
    if (a == b) {
      rfma(aj, p.mtab[2 * h + al], rab);
      rfma(tz, ma, rab);
      if (a < h) zp = cadd(zp, rab);
      else zn = cadd(zn, rab);
    }
    if (a == b + 1) rfma(tpl, ca, rab);
    if (b == a + 1) rfma(tmi, cb, rab);
    {
      double2 l4 = AB[max(a, b) + min(a, b) * ld];  // (A10 / 4)(a, b) up to the sign; a = b: never used
      l4 = cscale((a < b) ? 1.0 : (a > b ? -1.0 : 0.0), l4);
      double2 w = cscale(ma * mb, a01(a, b));
      rfma(w, 0.5 * ca * cb1, a01(max(a - 1, 0), min(b + 1, n - 1)));
      rfma(w, 0.5 * ca1 * cb, a01(min(a + 1, n - 1), max(b - 1, 0)));
      cfma(aj, l4, w);
    }
    x += NTH / n;
    y += NTH % n;
    if (y >= n) {
      y -= n;
      ++x;
    }
  }
  // two-body energy, regrouped list
  double2 e2 = cz();
  {
    const char *lb = (const char *)lds;
    const int shift = p.lbytes ? 0 : 4;
    auto at = [&](unsigned o) { return *(const double2 *)(lb + (o << shift)); };
    for (int q = tid; q < p.nl; q += NTH) {
      const uint4 o = p.lofs[q];
      const double me = p.lme[q];
      double2 t = cmul(at(o.x & 0xffffu), at(o.x >> 16));
      cfms(t, at(o.y & 0xffffu), at(o.y >> 16));
      cfma(t, at(o.z & 0xffffu), at(o.z >> 16));
      rfma(e2, me, t);
    }
  }
  // the 16 sums: quad sums by DPP, those of each value through LDS (the A-block
  // is free after the list), thread k < 16 adds value k's
  double v[16] = {e2.x, e2.y, ek.x, ek.y, aj.x, aj.y, tz.x, tz.y, tpl.x, tpl.y, tmi.x, tmi.y, zp.x, zp.y, zn.x, zn.y};
#pragma unroll
  for (int k = 0; k < 16; ++k) {
    v[k] += dpp_quad_f64<0xB1>(v[k]);  // quad_perm [1,0,3,2]
    v[k] += dpp_quad_f64<0x4E>(v[k]);  // quad_perm [2,3,0,1]
  }
  __syncthreads();
  double *const qs = (double *)AB;
  int NQ = NTH / 4 < 64 ? NTH / 4 : 64;  // quads through LDS at a time: 17 doubles each in the A-block's 16 n (n + 1) bytes
  while (NQ * 17 * 8 > 16 * n * ld) NQ >>= 1;
  double tot = 0.0;
#pragma unroll 1
  for (int q0 = 0; q0 < NTH / 4; q0 += NQ) {
    const int qd = (tid >> 2) - q0;
    if ((tid & 3) == 0 && qd >= 0 && qd < NQ) {
#pragma unroll
      for (int k = 0; k < 16; ++k) qs[qd * 17 + k] = v[k];
    }
    __syncthreads();
    if (tid < 16)
      for (int i = 0; i < NQ; ++i) tot += qs[i * 17 + tid];
    __syncthreads();
  }
  if (tid < 16) red[tid] = tot;
  __syncthreads();
  double2 *const go = p.gout + (size_t)L * p.nog;
  if (tid == 0) {
    const double *t = red;
    const double2 E2v = make_double2(t[0], t[1]), EK = make_double2(t[2], t[3]), A = make_double2(t[4], t[5]);
    const double2 TZ = make_double2(t[6], t[7]), TP = make_double2(t[8], t[9]), TM = make_double2(t[10], t[11]);
    const double2 ZP = make_double2(t[12], t[13]), ZN = make_double2(t[14], t[15]);
    const double2 J2 = cadd(A, cadd(cmul(TZ, TZ), cmul(TP, TM)));
    go[0] = make_double2(1.0, 0.0);
    go[1] = ZP;
    go[2] = ZN;
    go[3] = EK;
    go[4] = cadd(cadd(E2v, EK), make_double2(p.e0, 0.0));
    go[5] = J2;
    p.gst[L] = info;
  }
  if (E2) {
    // tr_s(Q_mu rho) = sum_{i, j in s} Q_mu(i, j) rho(j, i) (ZQ2, PNAMP_ME1B.f90:52-75)
    __syncthreads();
    double q[20];
#pragma unroll
    for (int k = 0; k < 20; ++k) q[k] = 0.0;
#pragma unroll
    for (int sp = 0; sp < 2; ++sp)
      for (int rr = tid; rr < h * h; rr += NTH) {
        const int i = sp * h + rr % h, j = sp * h + rr / h;
        const double2 rji = R[j + i * ld];
#pragma unroll
        for (int mu = 0; mu < 5; ++mu) {
          const double qv = p.q2[(size_t)mu * nn + i + (size_t)j * n];
          q[sp * 10 + 2 * mu] = fma(qv, rji.x, q[sp * 10 + 2 * mu]);
          q[sp * 10 + 2 * mu + 1] = fma(qv, rji.y, q[sp * 10 + 2 * mu + 1]);
        }
      }
#pragma unroll
    for (int k = 0; k < 20; ++k)
      for (int off = 32; off > 0; off >>= 1) q[k] += __shfl_xor(q[k], off);
    if (lane == 0)
#pragma unroll
      for (int k = 0; k < 20; ++k) red[wave * 20 + k] = q[k];
    __syncthreads();
    if (tid < 10) {
      double re = 0.0, im = 0.0;
      for (int w = 0; w < NW; ++w) {
        re += red[w * 20 + 2 * tid];
        im += red[w * 20 + 2 * tid + 1];
      }
      go[NOBS + tid] = make_double2(re, im);
    }
    // orbit-pair traces sum_m rho(k_a(m), k_b(m)) (ZRho1B_Angles, PNAMP_Rho1B.f90:13-33)
    for (int o = tid; o < p.nob2; o += NTH) {
      const int4 op = p.orbp[o];
      double2 t = cz();
      for (int m = 0; m < op.w; ++m) t = cadd(t, R[(op.y + m) + (op.z + m) * ld]);
      go[NOG_E2 + o] = t;
    }
  }
}

// ------------------------------------------------------------------ gauge sum
struct PSum {
  int ng, ngc, nog, nob2, u0, NE, nefull, nphi, zval, nval;
  const int2 *ecan;
  const int *gmap;  // [nphi^2]: the gauge pair evaluated, | 1 << 16 as its conjugate
  double vac_scale, snpfaf;
  const int *q0, *q1, *pz, *pn;
  const double *det;
  const double2 *gout, *gpf;
  const int *gst;
  double2 *zres, *ze2, *zrho;
  int *status;
};

// Fomenko sum over the gauge points of one unit: the norm weight
// znorm = <0|Phi0><0|Phi1> Pf e^{-i (phi_p Z + phi_n N)} times each observable
// (PNAMP_Kernel3D.f90:262-387), divided by nphi^2; a mirrored Euler point
// takes the conjugate sums.
__global__ __launch_bounds__(64) void k_plain_sum(PSum p) {
  __shared__ double2 zn[256];
  __shared__ int gm[256];
  const int ul = blockIdx.x, u = p.u0 + ul, ip = u / p.NE;
  const int2 en = p.ecan[u - ip * p.NE];
  const size_t ue = (size_t)ip * p.nefull + en.x, um = (size_t)ip * p.nefull + (en.y >= 0 ? en.y : en.x);
  const double inv = 1.0 / (double)p.ng;
  const double vac = p.snpfaf * (p.det[p.q0[ip]] * p.vac_scale) * (p.det[p.q1[ip]] * p.vac_scale);
  const double zv = p.pz ? p.pz[ip] : p.zval, nv = p.pn ? p.pn[ip] : p.nval;
  for (int g = threadIdx.x; g < p.ng; g += 64) {
    const int lp = g / p.nphi, ln = g - lp * p.nphi;
    const double phip = (2.0 * M_PI / p.nphi) * lp;
    const double phin = (2.0 * M_PI / p.nphi) * ln;
    const int m = p.gmap[g];
    gm[g] = m;
    double2 pf = p.gpf[(size_t)ul * p.ngc + (m & 0xffff)];
    if (m >> 16) pf = cconj(pf);
    zn[g] = cmul(cscale(vac, pf), cexpi(-phip * zv - phin * nv));
  }
  __syncthreads();
  const double2 *gi = p.gout + (size_t)ul * p.ngc * p.nog;
  for (int o = threadIdx.x; o < p.nog; o += 64) {
    double2 s = cz();
    for (int g = 0; g < p.ng; ++g) {
      if (o == 0) s = cadd(s, zn[g]);
      else {
        double2 v = gi[(size_t)(gm[g] & 0xffff) * p.nog + o];
        if (gm[g] >> 16) v = cconj(v);
        cfma(s, zn[g], v);
      }
    }
    s = cscale(inv, s);
    const double2 sc = (en.y >= 0) ? cconj(s) : s;
    if (o < NOBS) p.zres[um * NOBS + o] = sc, p.zres[ue * NOBS + o] = s;
    else if (o < NOG_E2) p.ze2[um * 10 + (o - NOBS)] = sc, p.ze2[ue * 10 + (o - NOBS)] = s;
    else p.zrho[um * p.nob2 + (o - NOG_E2)] = sc, p.zrho[ue * p.nob2 + (o - NOG_E2)] = s;
  }
  if (threadIdx.x == 0) {
    int st = 0;
    for (int g = 0; g < p.ngc && !st; ++g) st = p.gst[(size_t)ul * p.ngc + g];
    p.status[um] = st;
    p.status[ue] = st;
  }
}

// ------------------------------------------------------------------ host
// Size classes of the kernels (n <= N): sd 24, pf 40, f5pg9 44 -> 48,
// sdpf 64.  The gauge kernel's LDS is 32 n (n + 1) bytes plus ~1 KB:
// 53.6 KB at n = 40 (three workgroups per CU), 64.6 KB at n = 44 (two),
// 136 KB at n = 64 (one).
constexpr int NCLASS = 6;
constexpr int CLASSES[NCLASS] = {16, 24, 32, 40, 48, 64};

int class_of(int n) {
  for (int c : CLASSES)
    if (n <= c) return c;
  return 0;
}

template <int N>
size_t gauge_lds(int n) {
  return sizeof(double2) * 2 * (size_t)n * (n + 1) + gauge_misc_bytes<N>();
}

template <int N, bool E2>
hipError_t prepare_nc(int n) {
  return hipFuncSetAttribute((const void *)k_plain_gauge<N, E2>, hipFuncAttributeMaxDynamicSharedMemorySize,
                             (int)gauge_lds<N>(n));
}

template <int N>
hipError_t launch_gauge(bool e2, unsigned grid, hipStream_t s, const PGauge &gp) {
  hipLaunchKernelGGL((k_plain_pf<N>), dim3(grid), dim3(PfCfg<N>::NT), 0, s, gp);
  const size_t lds = gauge_lds<N>(gp.n);
  if (e2) hipLaunchKernelGGL((k_plain_gauge<N, true>), dim3(grid), dim3(PlainCfg<N>::NTH), lds, s, gp);
  else hipLaunchKernelGGL((k_plain_gauge<N, false>), dim3(grid), dim3(PlainCfg<N>::NTH), lds, s, gp);
  return hipGetLastError();
}

size_t align256(size_t b) { return (b + 255) & ~(size_t)255; }

}  // namespace

bool plain_supported(int n) { return n >= 8 && !(n & 1) && class_of(n) != 0; }

size_t plain_unit_bytes(const PlainArgs &a) {
  const size_t nn = (size_t)a.n * a.n, ng = (size_t)a.ngc;
  const size_t nog = a.q2 ? (size_t)NOG_E2 + a.nob2 : (size_t)NOBS;
  return align256(sizeof(double2) * 7 * nn) + align256(sizeof(double2) * ng * nog) + align256(sizeof(int) * ng) +
         align256(sizeof(double2) * ng);
}

hipError_t plain_prepare(int n, bool e2) {
  const hipError_t e = hipFuncSetAttribute((const void *)k_plain_setup, hipFuncAttributeMaxDynamicSharedMemorySize,
                                           (int)setup_lds(n));
  if (e != hipSuccess) return e;
  switch (class_of(n)) {
    case 16: return e2 ? prepare_nc<16, true>(n) : prepare_nc<16, false>(n);
    case 24: return e2 ? prepare_nc<24, true>(n) : prepare_nc<24, false>(n);
    case 32: return e2 ? prepare_nc<32, true>(n) : prepare_nc<32, false>(n);
    case 40: return e2 ? prepare_nc<40, true>(n) : prepare_nc<40, false>(n);
    case 48: return e2 ? prepare_nc<48, true>(n) : prepare_nc<48, false>(n);
    case 64: return e2 ? prepare_nc<64, true>(n) : prepare_nc<64, false>(n);
    default: return hipErrorInvalidValue;
  }
}

hipError_t plain_run(const PlainArgs &a, int u0, int nu, void *work, hipStream_t s) {
  const int N = class_of(a.n);
  if (!N || nu <= 0) return hipErrorInvalidValue;
  const size_t nn = (size_t)a.n * a.n, ng = (size_t)a.ngc;
  const bool e2 = a.q2 != nullptr;
  const int nog = e2 ? NOG_E2 + a.nob2 : NOBS;
  // work buffer: all units' setup matrices, then all gauge outputs, then all gauge status
  char *w = (char *)work;
  double2 *hoist = (double2 *)w;
  double2 *gout = (double2 *)(w + align256(sizeof(double2) * 7 * nn * nu));
  int *gst = (int *)((char *)gout + align256(sizeof(double2) * ng * nog * nu));
  double2 *gpf = (double2 *)((char *)gst + align256(sizeof(int) * ng * nu));
  if (a.nphi > 16) return hipErrorInvalidValue;  // nphi <= 16

  PSetup sp;
  sp.n = a.n; sp.h = a.h; sp.nalp = a.nalp; sp.ngam = a.ngam; sp.npack = a.npack; sp.NE = a.nec; sp.ecan = a.ecan; sp.u0 = u0;
  sp.alp = a.alp; sp.gam = a.gam; sp.rtab = a.rtab; sp.pk_a = a.pk_a; sp.pk_b = a.pk_b;
  sp.blk_off = a.blk_off; sp.blk_sz = a.blk_sz; sp.blk_base = a.blk_base; sp.twom = a.twom;
  sp.q0 = a.q0; sp.q1 = a.q1; sp.U = a.U; sp.V = a.V; sp.Z = a.Z; sp.hoist = hoist;
  hipLaunchKernelGGL(k_plain_setup, dim3(nu, (a.n + SC - 1) / SC), dim3(256), setup_lds(a.n), s, sp);
  hipError_t err = hipGetLastError();
  if (err != hipSuccess) return err;

  PGauge gp;
  gp.n = a.n; gp.h = a.h; gp.nphi = a.nphi; gp.NE = a.nec; gp.ngc = a.ngc; gp.gcls = a.gcls;
  gp.nl = a.nl; gp.lbytes = a.lbytes; gp.nob2 = a.nob2; gp.nog = nog; gp.u0 = u0;
  gp.nwg = (int)(ng * nu);
  gp.cscale = a.cscale; gp.e0 = a.e0;
  gp.q0 = a.q0; gp.q1 = a.q1;
  gp.U = a.U; gp.V = a.V; gp.Z = a.Z; gp.hoist = hoist;
  gp.mtab = a.mtab; gp.t1b = a.t1b; gp.lofs = a.lofs; gp.lme = a.lme; gp.q2 = a.q2; gp.orbp = a.orbp;
  gp.gout = gout; gp.gst = gst; gp.gpf = gpf;
  const unsigned grid = (unsigned)((ng * nu + 7) / 8 * 8);
  switch (N) {
    case 16: err = launch_gauge<16>(e2, grid, s, gp); break;
    case 24: err = launch_gauge<24>(e2, grid, s, gp); break;
    case 32: err = launch_gauge<32>(e2, grid, s, gp); break;
    case 40: err = launch_gauge<40>(e2, grid, s, gp); break;
    case 48: err = launch_gauge<48>(e2, grid, s, gp); break;
    default: err = launch_gauge<64>(e2, grid, s, gp); break;
  }
  if (err != hipSuccess) return err;

  PSum sm;
  sm.ng = a.nphi * a.nphi; sm.ngc = a.ngc; sm.nog = nog; sm.nob2 = a.nob2; sm.u0 = u0;
  sm.NE = a.nec; sm.nefull = a.NE; sm.ecan = a.ecan; sm.gmap = a.gmap; sm.nphi = a.nphi;
  sm.zval = a.zval; sm.nval = a.nval; sm.vac_scale = a.vac_scale; sm.snpfaf = a.snpfaf;
  sm.q0 = a.q0; sm.q1 = a.q1; sm.pz = a.pz; sm.pn = a.pn; sm.det = a.det;
  sm.gout = gout; sm.gpf = gpf; sm.gst = gst; sm.zres = a.zres; sm.ze2 = a.ze2; sm.zrho = a.zrho; sm.status = a.status;
  hipLaunchKernelGGL(k_plain_sum, dim3(nu), dim3(64), 0, s, sm);
  return hipGetLastError();
}
