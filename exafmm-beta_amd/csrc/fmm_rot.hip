// fmm_rot.hip -- M2L on target tiles, M2M and L2L as rotate, shift along z,
// rotate back.
//
// The translation of one offset class as a dense real P^2 x P^2 operator costs
// 2 P^4 flop a pair (41.5 kflop at P = 12).  Turned so that the offset lies on
// the z axis it factors (M~, L^ as in fmm_device.hpp, s = sqrt((n-m)!(n+m)!)):
//   u[n,m]  = s M~[n,m] e^{i m phi}                           (z rotation)
//   v[n,.]  = Q_n(beta) u[n,.]      Re and Im parts apart     (y rotation)
//   w[j,m]  = sum_n T_m[j,n] v[n,m] (Re and Im alike)         (shift by r)
//   L^[j,.] = s e^{-i m phi} (S Q_j S) w[j,.],  S = (-1)^m    (back)
// with Q_n built from the Wigner matrix d^n(beta) (columns m and -m folded),
// T_m[j,n] = (-1)^(j+m) (j+n)! / (r^(j+n+1) s(j,m) s(n,m)), and S Q S the
// inverse rotation: one set of matrices serves both rotations.  All blocks
// have at most P rows: about 6 P^3 multiply-adds a pair in place of P^4.
//
// The blocks run on v_mfma_f64_4x4x4f64 (four independent 4x4 products an
// instruction; A[r][k] of block b in lane 16k + 4b + r, B[k][c] in lane
// 16k + 4b + c, D[r][c] in lane 16r + 4b + c, so a result is the next
// product's B operand).  Block b holds one degree n (rotations) or one order
// m (shift), columns c are four pairs:
//   layout 1 (rotations): tile (i, j), lane (r, b, c): n = 4i + b, m = 4j + r
//   layout 2 (shift):     level k, tile i, lane (r, b, c): m = m0(k) + b,
//                         n = m0(k) + 4i + r
// and 4 P^2 doubles go through LDS between them (twice a slice).  When the
// last row of tiles holds only one or two degrees (P = 9, 10, 5, 6) their Re
// and Im parts share it (b = part, degree), and the orders of the same size
// likewise: 57 instead of 84 products a slice at P = 10.  Of a single degree
// (P = 5, 9) both blocks of a part hold the values and compute different tiles:
// 12 instead of 18 products at P = 5, 45 instead of 57 at P = 9 (M2L of the 10^6
// cube 0.50 -> 0.45 ms and 1.27 -> 1.13).
//
// M2M and L2L factor the same way with T_m[j,n] = (-r)^(j-n) / (j-n)! (n <= j)
// and r^(n-j) / (n-j)! (n >= j); as both sides are in one normalisation, s is
// folded into Q (s^-1 Q s, s Q s^-1) instead of the z rotation.  A level's 8
// child offsets are reflections of (h, h, h), so a level has one record each.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <vector>

#include "fmm_device.hpp"

namespace fmmdev {

namespace {

constexpr int kRotMaxP = 12;
__host__ __device__ constexpr int tri(int i, int j) { return i * (i + 1) / 2 + j; }
__host__ __device__ constexpr int sq_sum(int n) { return n * (n + 1) * (2 * n + 1) / 6; }

template <int P> struct RotCfg {
  static constexpr int NT = P * (P + 1) / 2;
  static constexpr int G = (P + 3) / 4;         // tiles of 4 along a degree
  static constexpr int REM = P - 4 * (G - 1);   // degrees in the last row of tiles
  static constexpr bool COMB = REM <= 2;        // their Re and Im share the blocks
  static constexpr int NL = COMB ? G - 1 : G;   // full rows of tiles
  static constexpr int NF = tri(NL, 0);         // full tiles (of each part)
  static constexpr int NX = COMB ? G : 0;       // tiles of the shared row
  // one degree in it: its values sit in both blocks of a part, which compute
  // different tiles (2 p and 2 p + 1); the four blocks of m = 0 (Re) likewise
  static constexpr bool ONE = COMB && REM == 1;
  static constexpr int NXO = ONE ? (NX + 1) / 2 : NX, NXS = ONE ? (NX + 3) / 4 : NX;
  // products: rotations of the full rows (Re, Im), of the shared row; shifts
  static constexpr int NQ = sq_sum(NL), NQX = NXO * NX;
  static constexpr int NFRAG = 3 * NQ + NQX + NXS * NX;
  static constexpr int QRE = 0, QIM = NQ, QX = 2 * NQ, TF = 2 * NQ + NQX, TX = 3 * NQ + NQX;
  static constexpr int NCS = NF + NX;           // (s cos m phi, s sin m phi) of every tile
  static constexpr int NREC = NFRAG + 2 * NCS;  // doubles a lane of one class's record
  static constexpr int NREC2 = (NREC + 1) / 2;  // stored [NREC2][64 lanes][2]
  // shift levels: orders m0(k) .. m0(k) + 3 with tiles(k) tiles of degrees
  static __host__ __device__ constexpr int m0(int k) { return (COMB ? REM : 0) + 4 * k; }
  static __host__ __device__ constexpr int tiles(int k) { return NL - k; }
  static __host__ __device__ constexpr int off2(int k) { return NF - tri(NL - k, 0); }     // first tile of level k
  static __host__ __device__ constexpr int offT(int k) { return NQ - sq_sum(NL - k); }     // its products
  // exchange buffer (doubles): element (n, m, c) at n AST + 4 m + c; AST = 4 x
  // odd keeps the four blocks of both layouts on distinct banks
  static constexpr int AST = 16 * G + 4;
  static constexpr int ROWS = COMB ? P : 4 * G;
  static constexpr int PART = COMB ? (ROWS * AST + 7) / 16 * 16 + 8 : 0;  // Im part (Re and Im in turn otherwise)
  static constexpr int XSZ = COMB ? PART + ROWS * AST : ROWS * AST;
};

// Delta_n = d^n(pi/2), n < kRotMaxP, orders k, a >= 0: (n+1)^2 each, row-major,
// as unevaluated sums hi + lo
__device__ double2 g_delta[sq_sum(kRotMaxP)];

// Double-double arithmetic for the records: an operator entry is applied three
// times in a row to every pair, so it is rounded once, not once per step of
// its recurrences (measured: up to 9e-16 off at n = 11 in plain FP64).
struct dd {
  double h, l;
};
#pragma clang fp contract(off)
__device__ __forceinline__ dd dd_norm(double a, double b) {  // |a| >= |b|
  const double s = a + b;
  return {s, b - (s - a)};
}
__device__ __forceinline__ dd dd_add(dd a, dd b) {
  const double s = a.h + b.h, t = s - a.h;
  const double e = (a.h - (s - t)) + (b.h - t);
  return dd_norm(s, e + (a.l + b.l));
}
__device__ __forceinline__ dd dd_mul(dd a, dd b) {
  const double p = a.h * b.h;
  return dd_norm(p, __builtin_fma(a.h, b.h, -p) + (a.h * b.l + a.l * b.h));
}
__device__ __forceinline__ dd dd_neg(dd a) { return {-a.h, -a.l}; }
__device__ __forceinline__ dd dd_div(dd a, dd b) {
  const double q = a.h / b.h;
  const dd r = dd_add(a, dd_neg(dd_mul(b, {q, 0.0})));
  return dd_norm(q, r.h / b.h);
}
__device__ __forceinline__ dd dd_sqrt(dd a) {
  const double x = sqrt(a.h);
  if (!(x > 0.0)) return {x, 0.0};
  const dd r = dd_add(a, dd_neg(dd_mul({x, 0.0}, {x, 0.0})));
  return dd_norm(x, r.h / (2.0 * x));
}
#pragma clang fp contract(fast)

// The record of every offset (components >= 0): the A operands of all products
// and the z rotation factors, one block each.  With W[a][b] = d^n(beta)[a][b] =
// sum_k Delta[k][a] Delta[k][b] Re(i^(b-a) e^{-i k beta}) -- no cancelling
// terms -- the folded matrix Q[a][m] = W[a][m] +- (-1)^m W[a][-m] keeps, by the
// symmetries of Delta, the orders k >= 0 of n's parity (Re) or the other (Im).
// kind: 0 M2L, 1 M2M, 2 L2L.
template <int P>
__global__ __launch_bounds__(256) void rot_ops_kernel(int kind, const double *__restrict__ cdx, int nrep,
                                                      double *__restrict__ ops) {
  using C = RotCfg<P>;
  __shared__ dd ck[2][P], rp[2 * P];  // cos, sin k beta; r^-(k+1) (M2L), r^k
  __shared__ double zc[2][P], fac[2 * P];
  const int g = blockIdx.x, tid = threadIdx.x;
  if (g >= nrep) return;
  if (tid % 64 == 0 && tid < 192) {  // three short recurrences, one wavefront each
    const dd x = {cdx[3 * g], 0.0}, y = {cdx[3 * g + 1], 0.0}, z = {cdx[3 * g + 2], 0.0};
    const dd rho2 = dd_add(dd_mul(x, x), dd_mul(y, y));
    const dd rho = dd_sqrt(rho2), r = dd_sqrt(dd_add(rho2, dd_mul(z, z)));
    if (tid < 128) {
      const bool polar = tid == 0;
      dd c1 = {1.0, 0.0}, s1 = {0.0, 0.0};
      if (polar) {
        c1 = dd_div(z, r);
        s1 = dd_div(rho, r);
      } else if (rho.h > 0.0) {
        c1 = dd_div(x, rho);
        s1 = dd_div(y, rho);
      }
      dd c = {1.0, 0.0}, sn = {0.0, 0.0};
      for (int k = 0; k < P; k++) {
        if (polar) {
          ck[0][k] = c;
          ck[1][k] = sn;
        } else {
          zc[0][k] = c.h;
          zc[1][k] = sn.h;
        }
        const dd cn = dd_add(dd_mul(c, c1), dd_neg(dd_mul(sn, s1)));
        sn = dd_add(dd_mul(sn, c1), dd_mul(c, s1));
        c = cn;
      }
    } else {
      const dd step = kind == 0 ? dd_div({1.0, 0.0}, r) : r;
      dd v = {1.0, 0.0};
      if (kind == 0) v = step;
      double f = 1.0;
      for (int k = 0; k < 2 * P; k++) {
        rp[k] = v;
        v = dd_mul(v, step);
        fac[k] = f;
        f *= k + 1;
      }
    }
  }
  __syncthreads();
  auto rot = [&](int n, int a, int m, int part) {  // Q_n[a][m] of the part
    if (n >= P || a > n || m > n || (part && (a == 0 || m == 0))) return 0.0;
    const double2 *D = g_delta + n * (n + 1) * (2 * n + 1) / 6;
    const int q = (m - a) & 3;
    dd v = {0.0, 0.0};
    for (int k = (n + part) & 1; k <= n; k += 2) {
      const double2 da = D[k * (n + 1) + a], db = D[k * (n + 1) + m];
      const dd t = dd_mul(dd_mul({da.x, da.y}, {db.x, db.y}), ck[q & 1][k]);
      v = dd_add(v, k == 0 ? t : dd{2.0 * t.h, 2.0 * t.l});  // orders k and -k
    }
    double w = m == 0 ? v.h : 2.0 * v.h;  // columns m and -m
    if (q & 2) w = -w;
    if (kind != 0 && a != m) {  // s folded in: s^-1 Q s (M2M), s Q s^-1 (L2L)
      const double u = sqrt((fac[n - m] / fac[n - a]) * (fac[n + m] / fac[n + a]));
      w = kind == 1 ? w * u : w / u;
    }
    return w;
  };
  auto shift = [&](int m, int j, int n) {  // T_m[j][n], times the inner S of the back rotation
    if (j >= P || n >= P || j < m || n < m) return 0.0;
    if (kind == 0) {
      const double t = rp[j + n].h * (fac[j + n] / sqrt((fac[j - m] * fac[n - m]) * (fac[j + m] * fac[n + m])));
      return (j & 1) ? -t : t;
    }
    const int d = kind == 1 ? j - n : n - j;
    if (d < 0) return 0.0;
    const double t = rp[d].h / fac[d];
    return ((kind == 1 ? d + m : m) & 1) ? -t : t;
  };
  double *rec = ops + (size_t)g * C::NREC2 * 128;
  for (int e = tid; e < C::NREC2 * 128; e += 256) {
    const int f = e >> 6, lane = e & 63;
    const int k = lane >> 4, b = (lane >> 2) & 3, r = lane & 3;
    double v = 0.0;
    if (f < C::QX) {  // full rows
      const int part = f >= C::QIM;
      int h = f - (part ? C::QIM : 0), i = 0;
      while (h >= (i + 1) * (i + 1)) {
        h -= (i + 1) * (i + 1);
        i++;
      }
      v = rot(4 * i + b, 4 * (h / (i + 1)) + r, 4 * (h % (i + 1)) + k, part);
    } else if (f < C::TF) {  // shared row
      const int h = f - C::QX;
      const int jo = C::ONE ? 2 * (h / C::G) + (b & 1) : h / C::G;
      v = rot(C::ONE ? P - 1 : 4 * (C::G - 1) + (b & 1), 4 * jo + r, 4 * (h % C::G) + k, b >> 1);
    } else if (f < C::TX) {  // shift levels
      int h = f - C::TF, lev = 0;
      while (h >= C::tiles(lev) * C::tiles(lev)) {
        h -= C::tiles(lev) * C::tiles(lev);
        lev++;
      }
      const int t = C::tiles(lev), mm = C::m0(lev);
      v = shift(mm + b, mm + 4 * (h / t) + r, mm + 4 * (h % t) + k);
    } else if (f < C::NFRAG) {  // shared orders m < REM
      const int h = f - C::TX, m = C::ONE ? 0 : b & 1, jo = C::ONE ? 4 * (h / C::G) + b : h / C::G;
      v = m < C::REM ? shift(m, 4 * jo + r, 4 * (h % C::G) + k) : 0.0;
    } else if (f < C::NREC) {  // z rotation factors, lane (r = lane / 16, b, c)
      const int h = (f - C::NFRAG) >> 1, sn = (f - C::NFRAG) & 1, rr = lane >> 4;
      int n, m;
      bool neg = false;
      if (h < C::NF) {
        int i = 0, j = h;
        while (j > i) {
          j -= i + 1;
          i++;
        }
        n = 4 * i + b;
        m = 4 * j + rr;
      } else {  // own factor cos, partner factor -sin (Re) or +sin (Im)
        n = C::ONE ? P - 1 : 4 * (C::G - 1) + (b & 1);
        m = 4 * (h - C::NF) + rr;
        neg = !(b >> 1);
      }
      if (n < P && m <= n)
        v = (neg && sn ? -1.0 : 1.0) * (kind == 0 ? sqrt(fac[n - m] * fac[n + m]) : 1.0) * zc[sn][m];
    }
    rec[(size_t)(f >> 1) * 128 + lane * 2 + (f & 1)] = v;
  }
}

// v of lane l ^ 8 (the other part of a shared-row lane)
__device__ __forceinline__ double partner(double v) {
  const long long x = __double_as_longlong(v);
  const int lo = __builtin_amdgcn_mov_dpp((int)x, 0x128, 0xf, 0xf, true);  // row_ror:8
  const int hi = __builtin_amdgcn_mov_dpp((int)(x >> 32), 0x128, 0xf, 0xf, true);
  return __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}
__device__ __forceinline__ double flip(double v, unsigned mask) {
  return __longlong_as_double(__double_as_longlong(v) ^ ((long long)mask << 32));
}
__device__ __forceinline__ double mm(double a, double b, double c) {
  return __builtin_amdgcn_mfma_f64_4x4x4f64(a, b, c, 0, 0, 0);
}
// the exchange buffer is written and read by one wavefront, whose LDS
// operations complete in order: the compiler only must not reorder them
__device__ __forceinline__ void lds_order() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

// One wavefront's share of a translation: lane geometry, the record in
// registers, and the exchange buffer sX (XSZ doubles, zeroed, the
// wavefront's own).
template <int P> struct Rot {
  using C = RotCfg<P>;
  static constexpr int NT = C::NT, G = C::G, NL = C::NL, NF = C::NF, NX = C::NX, AST = C::AST, PART = C::PART;
  static constexpr int NF1 = NF > 0 ? NF : 1, NX1 = NX > 0 ? NX : 1;
  static constexpr int NXO = C::NXO, NXO1 = NXO > 0 ? NXO : 1;  // results of the shared row
  int r, b, c;
  int row[G], last;  // term of this lane's element of tile (i, 0), of tile (G-1, G-1)
  int w1, w2, x1, x2, x2l;
  double *sX;
  double A[C::NFRAG];
  double2 cs[C::NCS];

  __device__ __forceinline__ void init(int l, double *buf) {
    r = l >> 4;
    b = (l >> 2) & 3;
    c = l & 3;
    // lanes past the order or above the diagonal read a stand-in inside the
    // cell (their operator columns are zero)
#pragma unroll
    for (int i = 0; i < G; i++) {
      const int n = min(4 * i + (C::COMB && i == G - 1 ? b & 1 : b), P - 1);
      row[i] = n * (n + 1) / 2 + r;
    }
    last = min(row[G - 1] + 4 * (G - 1), NT - 1);
    w1 = b * AST + 4 * r + c;
    w2 = r * AST + 4 * b + c;
    x1 = min(b & 1, C::REM - 1) * AST + (b >> 1) * PART + 4 * r + c;
    const int xo = C::ONE ? c : (b >> 1) * PART + 4 * (b & 1) + c;
    x2 = r * AST + xo;
    x2l = min(4 * (G - 1) + r, C::ROWS - 1) * AST + xo;
    sX = buf;
  }
  __device__ __forceinline__ int term(int i, int j) const { return i == G - 1 && j == G - 1 ? last : row[i] + 4 * j; }
  __device__ __forceinline__ bool valid(int i, int j) const {  // this lane's element of tile (i, j) exists
    const int n = 4 * i + (C::COMB && i == G - 1 ? b & 1 : b);
    return n < P && 4 * j + r <= n;
  }
  __device__ __forceinline__ void load(const double2 *ops, int g, int l) {
    const double2 *rec = ops + (size_t)g * C::NREC2 * 64 + l;
#pragma unroll
    for (int f = 0; f < C::NREC2; f++) {
      const double2 v = rec[(size_t)f * 64];
#pragma unroll
      for (int h = 0; h < 2; h++) {
        const int u = 2 * f + h;
        const double x = h ? v.y : v.x;
        if (u < C::NFRAG)
          A[u] = x;
        else if (u < C::NREC) {
          if ((u - C::NFRAG) & 1)
            cs[(u - C::NFRAG) / 2].y = x;
          else
            cs[(u - C::NFRAG) / 2].x = x;
        }
      }
    }
  }
  // results of the shared row: tile, its term (a stand-in past the order), whether it exists
  __device__ __forceinline__ int xtile(int p) const { return C::ONE ? 2 * p + (b & 1) : p; }
  __device__ __forceinline__ int xterm(int p) const {
    return C::ONE ? min(row[G - 1] + 4 * xtile(p), NT - 1) : term(G - 1, p);
  }
  __device__ __forceinline__ bool xvalid(int p) const {
    return C::ONE ? 4 * xtile(p) + r < P : valid(G - 1, p);
  }
  // an expansion's terms as this lane holds them
  __device__ __forceinline__ void gather(const double2 *m, double2 (&pf)[NF1], double (&px)[NX1]) const {
#pragma unroll
    for (int i = 0; i < NL; i++)
#pragma unroll
      for (int j = 0; j <= i; j++) pf[tri(i, j)] = m[term(i, j)];
#pragma unroll
    for (int j = 0; j < NX; j++) px[j] = reinterpret_cast<const double *>(m + term(G - 1, j))[b >> 1];
  }
  // an expansion that results are added to, as this lane holds those
  __device__ __forceinline__ void gather_out(const double2 *m, double2 (&av)[NF1], double (&ax)[NXO1]) const {
#pragma unroll
    for (int i = 0; i < NL; i++)
#pragma unroll
      for (int j = 0; j <= i; j++) av[tri(i, j)] = m[term(i, j)];
#pragma unroll
    for (int p = 0; p < NXO; p++) ax[p] = reinterpret_cast<const double *>(m + xterm(p))[b >> 1];
  }
  // z rotation factors of the class's offset reflected by the bits rf (x, y,
  // z): the operator changes by the sign (-1)^(x m + z (n + m)) on both sides,
  // and phi -> -phi when one of x and y is reflected
  __device__ __forceinline__ void zfactors(int rf, double2 (&z)[C::NCS]) const {
    const unsigned mc = (unsigned)((rf & r) ^ ((rf >> 2) & (b ^ r))) << 31, sc = (unsigned)(rf ^ (rf >> 1)) << 31;
    const unsigned mx = C::ONE ? (unsigned)((rf & r) ^ ((rf >> 2) & r)) << 31 : mc;  // n = P - 1 is even
#pragma unroll
    for (int t = 0; t < C::NCS; t++) {
      const unsigned m = t < NF ? mc : mx;
      z[t] = make_double2(flip(cs[t].x, m), flip(cs[t].y, m ^ sc));
    }
  }
  __device__ __forceinline__ void zrot(const double2 (&z)[C::NCS], const double2 (&pf)[NF1], const double (&px)[NX1],
                                       double (&re)[NF1], double (&im)[NF1], double (&xv)[NX1]) const {
#pragma unroll
    for (int t = 0; t < NF; t++) {
      re[t] = fma(z[t].x, pf[t].x, -z[t].y * pf[t].y);
      im[t] = fma(z[t].x, pf[t].y, z[t].y * pf[t].x);
    }
#pragma unroll
    for (int t = 0; t < NX; t++) xv[t] = fma(z[NF + t].x, px[t], z[NF + t].y * partner(px[t]));
  }
  // z rotation back, added to av, ax
  __device__ __forceinline__ void zback(const double2 (&z)[C::NCS], const double (&re)[NF1], const double (&im)[NF1],
                                        const double (&xv)[NXO1], double2 (&av)[NF1], double (&ax)[NXO1]) const {
#pragma unroll
    for (int t = 0; t < NF; t++) {
      av[t].x = fma(z[t].x, re[t], fma(z[t].y, im[t], av[t].x));
      av[t].y = fma(z[t].x, im[t], fma(-z[t].y, re[t], av[t].y));
    }
#pragma unroll
    for (int p = 0; p < NXO; p++) {
      const double2 z0 = z[NF + (C::ONE ? 2 * p : p)];
      double cx = z0.x, cy = z0.y;
      if constexpr (C::ONE) {
        const double2 z1 = z[NF + (2 * p + 1 < NX ? 2 * p + 1 : 2 * p)];
        cx = b & 1 ? z1.x : cx;
        cy = b & 1 ? z1.y : cy;
      }
      ax[p] = fma(cx, xv[p], fma(-cy, partner(xv[p]), ax[p]));
    }
  }
  // this lane's terms stored into an expansion
  __device__ __forceinline__ void scatter(double2 *acc, const double2 (&av)[NF1], const double (&ax)[NXO1]) const {
#pragma unroll
    for (int i = 0; i < NL; i++)
#pragma unroll
      for (int j = 0; j < i; j++)
        if (4 * i + 3 < P || valid(i, j)) acc[row[i] + 4 * j] = av[tri(i, j)];
#pragma unroll
    for (int i = 0; i < NL; i++)
      if (4 * i + 3 < P ? r <= b : valid(i, i)) acc[row[i] + 4 * i] = av[tri(i, i)];
#pragma unroll
    for (int p = 0; p < NXO; p++)
      if (xvalid(p)) reinterpret_cast<double *>(acc + row[G - 1] + 4 * xtile(p))[b >> 1] = ax[p];
  }
  // products of one part: rotation of the full rows, of the shared row, shift
  __device__ __forceinline__ void rot_part(int q, double (&v)[NF1]) const {
    double o[NF1];
#pragma unroll
    for (int t = 0; t < NF; t++) o[t] = 0.0;
#pragma unroll
    for (int i = 0; i < NL; i++)
#pragma unroll
      for (int ji = 0; ji <= i; ji++)
#pragma unroll
        for (int jo = 0; jo <= i; jo++)
          o[tri(i, jo)] = mm(A[q + sq_sum(i) + jo * (i + 1) + ji], v[tri(i, ji)], o[tri(i, jo)]);
#pragma unroll
    for (int t = 0; t < NF; t++) v[t] = o[t];
  }
  template <int NO, int NO1> __device__ __forceinline__ void mul_shared(int q, const double (&v)[NX1],
                                                                        double (&o)[NO1]) const {
#pragma unroll
    for (int t = 0; t < NO; t++) o[t] = 0.0;
#pragma unroll
    for (int ji = 0; ji < NX; ji++)
#pragma unroll
      for (int jo = 0; jo < NO; jo++) o[jo] = mm(A[q + jo * G + ji], v[ji], o[jo]);
  }
  __device__ __forceinline__ void shift_part(double (&v)[NF1]) const {
    double o[NF1];
#pragma unroll
    for (int t = 0; t < NF; t++) o[t] = 0.0;
#pragma unroll
    for (int k = 0; k < NL; k++)
#pragma unroll
      for (int ii = 0; ii < C::tiles(k); ii++)
#pragma unroll
        for (int io = 0; io < C::tiles(k); io++)
          o[C::off2(k) + io] =
              mm(A[C::TF + C::offT(k) + io * C::tiles(k) + ii], v[C::off2(k) + ii], o[C::off2(k) + io]);
#pragma unroll
    for (int t = 0; t < NF; t++) v[t] = o[t];
  }
  // exchange buffer, layout 1 and 2 of one part, and of the shared tiles
  __device__ __forceinline__ void put1(const double (&v)[NF1], int off) const {
#pragma unroll
    for (int i = 0; i < NL; i++)
#pragma unroll
      for (int j = 0; j <= i; j++) sX[w1 + off + 4 * i * AST + 16 * j] = v[tri(i, j)];
  }
  __device__ __forceinline__ void get1(double (&v)[NF1], int off) const {
#pragma unroll
    for (int i = 0; i < NL; i++)
#pragma unroll
      for (int j = 0; j <= i; j++) v[tri(i, j)] = sX[w1 + off + 4 * i * AST + 16 * j];
  }
  __device__ __forceinline__ void put2(const double (&v)[NF1], int off) const {
#pragma unroll
    for (int k = 0; k < NL; k++)
#pragma unroll
      for (int i = 0; i < C::tiles(k); i++)
        sX[w2 + off + (C::m0(k) + 4 * i) * AST + 4 * C::m0(k)] = v[C::off2(k) + i];
  }
  __device__ __forceinline__ void get2(double (&v)[NF1], int off) const {
#pragma unroll
    for (int k = 0; k < NL; k++)
#pragma unroll
      for (int i = 0; i < C::tiles(k); i++)
        v[C::off2(k) + i] = sX[w2 + off + (C::m0(k) + 4 * i) * AST + 4 * C::m0(k)];
  }
  __device__ __forceinline__ void put1x(const double (&v)[NXO1]) const {
#pragma unroll
    for (int p = 0; p < NXO; p++)
      if (C::ONE ? xtile(p) < NX : (b & 1) < C::REM) sX[x1 + 4 * (G - 1) * AST + 16 * xtile(p)] = v[p];
  }
  __device__ __forceinline__ void get1x(double (&v)[NX1]) const {
#pragma unroll
    for (int j = 0; j < NX; j++) v[j] = sX[x1 + 4 * (G - 1) * AST + 16 * j];
  }
  static constexpr int NXS1 = C::NXS > 0 ? C::NXS : 1;
  __device__ __forceinline__ void put2x(const double (&v)[NXS1]) const {
#pragma unroll
    for (int i = 0; i < C::NXS; i++) {
      if constexpr (C::ONE) {
        if (4 * (4 * i + b) + r < P) sX[x2 + 4 * (4 * i + b) * AST] = v[i];
      } else {
        if ((i < G - 1 || 4 * i + r < P) && (b & 1) < C::REM) sX[x2 + 4 * i * AST] = v[i];
      }
    }
  }
  __device__ __forceinline__ void get2x(double (&v)[NX1]) const {
#pragma unroll
    for (int i = 0; i < NX; i++) v[i] = sX[i == G - 1 ? x2l : x2 + 4 * i * AST];
  }
  // rotation and shift, results in layout 1; each part's exchange runs beside
  // the other part's products
  __device__ __forceinline__ void turn_shift(double (&re)[NF1], double (&im)[NF1], double (&xv)[NX1]) const {
    if constexpr (C::COMB) {
      double xo[NXO1], xs[NXS1];
      mul_shared<NXO>(C::QX, xv, xo);
      rot_part(C::QRE, re);
      put1x(xo);
      put1(re, 0);
      rot_part(C::QIM, im);
      lds_order();
      get2(re, 0);
      put1(im, PART);
      lds_order();
      get2x(xv);
      get2(im, PART);
      lds_order();
      shift_part(re);
      put2(re, 0);
      mul_shared<C::NXS>(C::TX, xv, xs);
      put2x(xs);
      shift_part(im);
      lds_order();
      get1(re, 0);
      put2(im, PART);
      lds_order();
      get1x(xv);
      get1(im, PART);
      lds_order();
    } else {
      rot_part(C::QRE, re);
      put1(re, 0);
      lds_order();
      get2(re, 0);
      lds_order();
      rot_part(C::QIM, im);
      put1(im, 0);
      lds_order();
      get2(im, 0);
      lds_order();
      shift_part(re);
      put2(re, 0);
      lds_order();
      get1(re, 0);
      lds_order();
      shift_part(im);
      put2(im, 0);
      lds_order();
      get1(im, 0);
      lds_order();
    }
  }
  __device__ __forceinline__ void turn_back(double (&re)[NF1], double (&im)[NF1], const double (&xv)[NX1],
                                            double (&xo)[NXO1]) const {
    rot_part(C::QRE, re);
    if constexpr (C::COMB) mul_shared<NXO>(C::QX, xv, xo);
    rot_part(C::QIM, im);
  }
};

// One wavefront per work item: the slices (<= 4 pairs of one class with
// distinct targets) of a tile of TT targets, whose local expansions are held
// in LDS (times (-1)^m: the outer S of the back rotation) and stored, or
// added atomically when the tile is split over items, at the end.  The class's
// record stays in registers while consecutive slices share it.  No barriers:
// a wavefront owns its tile and its exchange buffer.
//
// Bound: issue.  A slice at P = 12 issues 84 products (16 cycles each) and
// about 110 other vector instructions, which do not overlap FP64 products on
// a SIMD; the rest is latency of the LDS round trips, hidden by the other
// part's products and by the second wavefront of the SIMD (registers: the
// record alone takes 108 at P = 12).  Measured on MI355X against one dense
// operator per class on v_mfma_f64_16x16x4 (same lists), M2L in ms: 8M cube,
// P = 12: 155 -> 42.5; 1M Plummer, P = 10: 6.7 -> 3.0; 10^6 cube, P = 8: 3.7 ->
// 2.1, P = 4: 1.10 -> 0.66; also against FP32 (P = 12 10.4 ms, P = 8 2.65) and
// split-FP16 (8.4, 2.27) dense operators on that cube (4.6, 2.1 here).
// TT: what LDS leaves room for with 8 wavefronts a CU (P >= 9), 16 below.
template <int P, int TT>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(2))) void m2l_rot_kernel(
    const int *__restrict__ ttgt, const int4 *__restrict__ items, const int4 *__restrict__ slices,
    const int *__restrict__ psrc, const unsigned short *__restrict__ plt, const double2 *__restrict__ ops,
    const double2 *__restrict__ M, double *__restrict__ L) {
  using C = RotCfg<P>;
  using R = Rot<P>;
  constexpr int NT = C::NT, G = C::G;
  __shared__ double2 sAcc[TT * NT];
  __shared__ double sX[C::XSZ];
  const int l = threadIdx.x;
  const int4 item = items[blockIdx.x];
  const int s0 = item.y, s1 = item.z;
  if (s0 >= s1) return;
  for (int e = l; e < TT * NT; e += 64) sAcc[e] = make_double2(0.0, 0.0);
  for (int e = l; e < C::XSZ; e += 64) sX[e] = 0.0;
  R rot;
  rot.init(l, sX);
  const int c = rot.c;
  // a slice's pairs: lanes past its count read its last pair as a stand-in
  auto desc = [&](int s) { return slices[min(s, s1 - 1)]; };
  auto pair_of = [&](const int4 &d) { return d.y + min(c, d.z - 1); };
  auto cell = [&](int src) { return M + (size_t)(src & ((1 << 26) - 1)) * NT; };
  double2 pf[R::NF1];
  double px[R::NX1];
  // pipeline: slice s computes, s + 1's multipoles load, s + 2's pair indices
  // load, s + 3's descriptor loads
  int4 d = desc(s0), d1 = desc(s0 + 1), d2 = desc(s0 + 2);
  rot.load(ops, d.x, l);
  rot.gather(cell(psrc[pair_of(d)]), pf, px);
  int lt = plt[pair_of(d)], lt1 = plt[pair_of(d1)], src1 = psrc[pair_of(d1)];
  for (int s = s0; s < s1; s++) {
    const int4 d3 = desc(s + 3);
    double2 z[C::NCS];
    rot.zfactors(lt >> 8, z);
    double re[R::NF1], im[R::NF1], xv[R::NX1];
    rot.zrot(z, pf, px, re, im, xv);
    rot.gather(cell(src1), pf, px);
    const int p2 = pair_of(d2);
    src1 = psrc[p2];
    const int lt2 = plt[p2];
    rot.turn_shift(re, im, xv);
    // the targets' local expansions are read while the back rotation runs
    double2 *acc = sAcc + (lt & 255) * NT;
    double2 av[R::NF1];
    double ax[R::NXO1], xo[R::NXO1];
    rot.gather_out(acc, av, ax);
    rot.turn_back(re, im, xv, xo);
    if (d1.x != d.x) rot.load(ops, d1.x, l);
    rot.zback(z, re, im, xo, av, ax);
    if (c < d.z) rot.scatter(acc, av, ax);
    lds_order();
    d = d1;
    d1 = d2;
    d2 = d3;
    lt = lt1;
    lt1 = lt2;
  }
  // store (or add) the tile's local expansions
  for (int t0 = 0; t0 < TT; t0 += 4) {
    const int t = t0 + c;
    const int tc = t < TT ? ttgt[(size_t)item.x * TT + t] : -1;
    if (tc < 0) continue;
    double *Lc = L + (size_t)tc * NT * 2;
#pragma unroll
    for (int i = 0; i < G; i++)
#pragma unroll
      for (int j = 0; j <= i; j++) {
        const int u = rot.row[i] + 4 * j;
        if (!rot.valid(i, j) || (C::COMB && i == G - 1 && (rot.b >> 1))) continue;
        double2 v = sAcc[t * NT + u];
        if (rot.r & 1) v = make_double2(-v.x, -v.y);
        if (item.w) {
          unsafeAtomicAdd(Lc + 2 * u, v.x);
          unsafeAtomicAdd(Lc + 2 * u + 1, v.y);
        } else {
          reinterpret_cast<double2 *>(Lc)[u] = v;
        }
      }
  }
}

// M2M of one level: blocks of 8 wavefronts, wavefront w the children of octant
// w of 4 parents; the 8 results are added in octant order through LDS and
// stored.  child8[8 i + o]: child of parent i in octant o (-1: none).  A block
// takes groups of 4 parents in turn, so that the record is loaded once.
// Bound: latency of the children's gather and the LDS round trips on the small
// levels, issue on the large ones.  Measured against a dense P^2 x P^2 operator
// per octant (16 parents a block, each reading 8 operators of 166 KB at P =
// 12), all levels: alone, 8M cube, P = 12, 1.78 -> 0.36 ms, 1M Plummer, P = 10,
// 0.32 -> 0.10; in a solve, beside P2P, 4.0 -> 2.4 and 0.83 -> 0.56; 4096 bodies, P
// = 8: 13 -> 7 us a level.
template <int P>
__global__ __launch_bounds__(512) void m2m_rot_kernel(const int *__restrict__ parents, const int *__restrict__ child8,
                                                      int np, const double2 *__restrict__ rec,
                                                      double2 *__restrict__ M) {
  using C = RotCfg<P>;
  using R = Rot<P>;
  constexpr int NT = C::NT;
  __shared__ double sX[8][C::XSZ];
  __shared__ double2 sO[8][4 * NT];
  const int w = threadIdx.x >> 6, l = threadIdx.x & 63;
  for (int e = l; e < C::XSZ; e += 64) sX[w][e] = 0.0;
  R rot;
  rot.init(l, sX[w]);
  rot.load(rec, 0, l);
  double2 z[C::NCS];
  rot.zfactors(w, z);  // X_parent - X_child: negative along d when octant bit d is set
  for (int g = blockIdx.x * 4; g < np; g += gridDim.x * 4) {
    const int i = g + rot.c;
    const int ch = i < np ? child8[8 * (size_t)i + w] : -1;
    double2 pf[R::NF1], av[R::NF1];
    double px[R::NX1], ax[R::NXO1], xo[R::NXO1];
    rot.gather(M + (size_t)max(ch, 0) * NT, pf, px);
#pragma unroll
    for (int t = 0; t < R::NF1; t++) {
      if (ch < 0) pf[t] = make_double2(0.0, 0.0);
      av[t] = make_double2(0.0, 0.0);
    }
#pragma unroll
    for (int t = 0; t < R::NX1; t++)
      if (ch < 0) px[t] = 0.0;
#pragma unroll
    for (int t = 0; t < R::NXO1; t++) ax[t] = 0.0;
    double re[R::NF1], im[R::NF1], xv[R::NX1];
    rot.zrot(z, pf, px, re, im, xv);
    rot.turn_shift(re, im, xv);
    rot.turn_back(re, im, xv, xo);
    rot.zback(z, re, im, xo, av, ax);
    rot.scatter(sO[w] + rot.c * NT, av, ax);
    __syncthreads();
    for (int e = threadIdx.x; e < 4 * NT; e += 512) {
      const int k = e / NT, u = e - k * NT;
      double2 v = sO[0][e];
#pragma unroll
      for (int o = 1; o < 8; o++) {
        v.x += sO[o][e].x;
        v.y += sO[o][e].y;
      }
      int n = 0;
      while ((n + 1) * (n + 2) / 2 <= u) n++;
      if ((u - n * (n + 1) / 2) & 1) v = make_double2(-v.x, -v.y);  // the outer S
      if (g + k < np) M[(size_t)parents[g + k] * NT + u] = v;
    }
    __syncthreads();
  }
}

// L2L of one level: a wavefront takes 4 children at a time, each from its
// parent: kids[k] = {child, parent | octant << 27}.  Adds into the children's
// local expansions.  Bound: reading and writing L and the record's load.  8M
// cube, P = 12, 13 levels: 2.85 -> 0.58 ms (dense operators per octant before).
template <int P>
__global__ __launch_bounds__(64) void l2l_rot_kernel(const int2 *__restrict__ kids, int nk,
                                                     const double2 *__restrict__ rec, double2 *__restrict__ L) {
  using C = RotCfg<P>;
  using R = Rot<P>;
  constexpr int NT = C::NT;
  __shared__ double sX[C::XSZ];
  const int l = threadIdx.x;
  for (int e = l; e < C::XSZ; e += 64) sX[e] = 0.0;
  R rot;
  rot.init(l, sX);
  rot.load(rec, 0, l);
  const unsigned odd = (unsigned)(rot.r & 1) << 31;  // the outer S
  for (int g = blockIdx.x * 4; g < nk; g += gridDim.x * 4) {
    const int2 kd = kids[min(g + rot.c, nk - 1)];
    double2 z[C::NCS];
    rot.zfactors(~(kd.y >> 27) & 7, z);  // X_child - X_parent: negative along d when octant bit d is clear
    double2 pf[R::NF1], av[R::NF1];
    double px[R::NX1], ax[R::NXO1], xo[R::NXO1];
    rot.gather(L + (size_t)(kd.y & ((1 << 27) - 1)) * NT, pf, px);
    double re[R::NF1], im[R::NF1], xv[R::NX1];
    rot.zrot(z, pf, px, re, im, xv);
    rot.turn_shift(re, im, xv);
    double2 *Lc = L + (size_t)kd.x * NT;
    rot.gather_out(Lc, av, ax);
    rot.turn_back(re, im, xv, xo);
#pragma unroll
    for (int t = 0; t < C::NCS; t++) z[t] = make_double2(flip(z[t].x, odd), flip(z[t].y, odd));
    rot.zback(z, re, im, xo, av, ax);
    if (g + rot.c < nk) rot.scatter(Lc, av, ax);
  }
}

template <int P> constexpr int rot_tt() { return P >= 9 ? 12 : 16; }

template <template <int> class F, typename... A> hipError_t rot_dispatch(int P, A... a) {
  switch (P) {
    case 2: return F<2>::run(a...);
    case 3: return F<3>::run(a...);
    case 4: return F<4>::run(a...);
    case 5: return F<5>::run(a...);
    case 6: return F<6>::run(a...);
    case 7: return F<7>::run(a...);
    case 8: return F<8>::run(a...);
    case 9: return F<9>::run(a...);
    case 10: return F<10>::run(a...);
    case 11: return F<11>::run(a...);
    case 12: return F<12>::run(a...);
    default: return hipErrorInvalidValue;
  }
}
template <int P> struct RotBytes {
  static hipError_t run(size_t *b, int *tt) {
    *b = sizeof(double) * 128 * RotCfg<P>::NREC2;
    *tt = rot_tt<P>();
    return hipSuccess;
  }
};
template <int P> struct RunRotOps {
  static hipError_t run(int kind, const double *cdx, int nrep, void *ops, hipStream_t s) {
    hipLaunchKernelGGL((rot_ops_kernel<P>), dim3(nrep), dim3(256), 0, s, kind, cdx, nrep, static_cast<double *>(ops));
    return hipGetLastError();
  }
};
template <int P> struct RunM2MRot {
  static hipError_t run(const int *parents, const int *child8, int np, const void *rec, double2 *M, hipStream_t s) {
    hipLaunchKernelGGL((m2m_rot_kernel<P>), dim3(std::min((np + 3) / 4, 512)), dim3(512), 0, s, parents, child8, np,
                       static_cast<const double2 *>(rec), M);
    return hipGetLastError();
  }
};
template <int P> struct RunL2LRot {
  static hipError_t run(const int2 *kids, int nk, const void *rec, double2 *L, hipStream_t s) {
    hipLaunchKernelGGL((l2l_rot_kernel<P>), dim3(std::min((nk + 3) / 4, 4096)), dim3(64), 0, s, kids, nk,
                       static_cast<const double2 *>(rec), L);
    return hipGetLastError();
  }
};
template <int P> struct RunM2LRot {
  static hipError_t run(int nitem, const int *ttgt, const int4 *items, const int4 *slices, const int *psrc,
                        const unsigned short *plt, const void *ops, const double2 *M, double2 *L, hipStream_t s) {
    hipLaunchKernelGGL((m2l_rot_kernel<P, rot_tt<P>()>), dim3(nitem), dim3(64), 0, s, ttgt, items, slices, psrc, plt,
                       static_cast<const double2 *>(ops), M, reinterpret_cast<double *>(L));
    return hipGetLastError();
  }
};

}  // namespace

hipError_t init_rot_constants() {
  // d^n(pi/2)[a][b] = 2^-n sqrt((n+a)!(n-a)! / ((n+b)!(n-b)!)) x an integer sum
  std::vector<double> h(2 * sq_sum(kRotMaxP));
  auto binom = [](int n, int k) {
    long long v = 1;
    for (int i = 1; i <= k; i++) v = v * (n - k + i) / i;
    return v;
  };
  long double f[2 * kRotMaxP];
  f[0] = 1.0L;
  for (int i = 1; i < 2 * kRotMaxP; i++) f[i] = f[i - 1] * i;
  for (int n = 0; n < kRotMaxP; n++)
    for (int a = 0; a <= n; a++)
      for (int b = 0; b <= n; b++) {
        long long t = 0;
        for (int k = std::max(0, b - a); k <= std::min(n + b, n - a); k++) {
          const long long v = binom(n + b, k) * binom(n - b, n - a - k);
          t += (a - b + k) & 1 ? -v : v;
        }
        const long double d =
            std::ldexp((long double)t, -n) * sqrtl(f[n + a] * f[n - a] / (f[n + b] * f[n - b]));
        double *o = h.data() + 2 * (sq_sum(n) + a * (n + 1) + b);
        o[0] = (double)d;
        o[1] = (double)(d - o[0]);
      }
  return hipMemcpyToSymbol(HIP_SYMBOL(g_delta), h.data(), h.size() * sizeof(double));
}

bool rot_supported(int P) { return P >= 2 && P <= kRotMaxP; }

size_t rot_ops_bytes(int P) {
  size_t b = 0;
  int tt = 0;
  (void)rot_dispatch<RotBytes>(P, &b, &tt);
  return b;
}

int m2l_tile_targets(int P) {
  size_t b = 0;
  int tt = 0;
  (void)rot_dispatch<RotBytes>(P, &b, &tt);
  return tt;
}

hipError_t launch_rot_ops(int P, int kind, const double *cdx, int nrep, void *ops, hipStream_t s) {
  return nrep > 0 ? rot_dispatch<RunRotOps>(P, kind, cdx, nrep, ops, s) : hipSuccess;
}
hipError_t launch_m2m_rot(int P, const int *parents, const int *child8, int np, const void *rec, double2 *M,
                          hipStream_t s) {
  return np > 0 ? rot_dispatch<RunM2MRot>(P, parents, child8, np, rec, M, s) : hipSuccess;
}
hipError_t launch_l2l_rot(int P, const int2 *kids, int nk, const void *rec, double2 *L, hipStream_t s) {
  return nk > 0 ? rot_dispatch<RunL2LRot>(P, kids, nk, rec, L, s) : hipSuccess;
}

hipError_t launch_m2l_rot(int P, int nitem, const int *ttgt, const int4 *items, const int4 *slices, const int *psrc,
                          const unsigned short *plt, const void *ops, const double2 *M, double2 *L, hipStream_t s) {
  return nitem > 0 ? rot_dispatch<RunM2LRot>(P, nitem, ttgt, items, slices, psrc, plt, ops, M, L, s) : hipSuccess;
}

}  // namespace fmmdev
