// fmm_kernels.hip -- gfx950 kernels of the Laplace FMM evaluator (FP64 path).
//
// Harmonics are generated by recurrences on Cartesian offsets (no acos,
// atan2 or complex exp):
//   regular  R[n][m] = r^n P_n^m(cos a) e^{i m b} / (n+m)!
//     R[m][m] = -(x+iy)/(2m) R[m-1][m-1],
//     R[n][m] = ((2n-1) z R[n-1][m] - r^2 R[n-2][m]) / (n^2 - m^2)
//   singular S[n][m] = (n-m)! r^{-n-1} P_n^m(cos a) e^{i m b}
//     S[m][m] = -(2m-1)(x+iy)/r^2 S[m-1][m-1],
//     S[n][m] = ((2n-1) z S[n-1][m] - ((n-1)^2 - m^2) S[n-2][m]) / r^2
// (P_n^m with the Condon-Shortley sign, as produced by the Legendre recurrence
// of kernels/laplace.h:48-113).  With M~ = M/s and L^ = L*s (s(n,m) =
// sqrt((n-m)!(n+m)!)) the reference operators become:
//   P2M  M~[n,m] = sum_b q_b conj(R[n][m](x_b - X_c))
//   M2L  L^[j,k] = (-1)^j i^{-k} sum_{n,m} Mh[n,m] Yh[j+n][m-k]
//        Mh[n,m] = i^{-|m|} M~c[n,m],  Yh[a][b] = i^{|b|} S[a][|b|] (conj for b<0)
//   M2M, L2L: the index patterns of laplace.h:254-290 and :324-357 with the
//        Anm ratios folded into the normalisation.
//   L2P: local expansion shifted to the body, read off at degrees 0 and 1.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <type_traits>

#include "fmm_device.hpp"
#include "fmm_p2m_lanes.hpp"

namespace fmmdev {

__constant__ double c_rcp[1024];  // c_rcp[k] = 1/k
// row r < kMaxP^2 of a real expansion vector: n | m << 8 | im << 16
__constant__ int c_vdec[kMaxP * kMaxP];
// triangular term u -> rows of its real and imaginary parts: re | im << 16
__constant__ int c_urow[kMaxP * (kMaxP + 1) / 2];

hipError_t init_constants() {
  double h[1024];
  h[0] = 0.0;
  for (int k = 1; k < 1024; k++) h[k] = 1.0 / k;
  hipError_t e = hipMemcpyToSymbol(HIP_SYMBOL(c_rcp), h, sizeof h);
  if (e != hipSuccess) return e;
  int vd[kMaxP * kMaxP], ur[kMaxP * (kMaxP + 1) / 2];
  for (int n = 0; n < kMaxP; n++) {
    vd[n * n] = n;
    for (int m = 1; m <= n; m++) {
      vd[n * n + 2 * m - 1] = n | (m << 8);
      vd[n * n + 2 * m] = n | (m << 8) | (1 << 16);
    }
    for (int m = 0; m <= n; m++)
      ur[n * (n + 1) / 2 + m] = (n * n + (m ? 2 * m - 1 : 0)) | ((n * n + 2 * m) << 16);
  }
  e = hipMemcpyToSymbol(HIP_SYMBOL(c_vdec), vd, sizeof vd);
  if (e != hipSuccess) return e;
  return hipMemcpyToSymbol(HIP_SYMBOL(c_urow), ur, sizeof ur);
}

bool order_supported(int P) { return P >= 2 && P <= kMaxP; }

// ---------------------------------------------------------------- helpers
__device__ __forceinline__ double2 cmul(double2 a, double2 b) {
  return make_double2(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x);
}
__device__ __forceinline__ double2 cmac(double2 acc, double2 a, double2 b) {
  acc.x = fma(a.x, b.x, acc.x);
  acc.x = fma(-a.y, b.y, acc.x);
  acc.y = fma(a.x, b.y, acc.y);
  acc.y = fma(a.y, b.x, acc.y);
  return acc;
}
__device__ __forceinline__ double2 cconj(double2 a) { return make_double2(a.x, -a.y); }
__device__ __forceinline__ double2 cscale(double2 a, double s) { return make_double2(a.x * s, a.y * s); }
__device__ __forceinline__ double2 cadd(double2 a, double2 b) { return make_double2(a.x + b.x, a.y + b.y); }
__device__ __forceinline__ double2 csub(double2 a, double2 b) { return make_double2(a.x - b.x, a.y - b.y); }
// a * i^e
__device__ __forceinline__ double2 cmul_ipow(double2 a, int e) {
  switch (e & 3) {
    case 0: return a;
    case 1: return make_double2(-a.y, a.x);
    case 2: return make_double2(-a.x, -a.y);
    default: return make_double2(a.y, -a.x);
  }
}
// a * i^e without divergent branches (e may differ across lanes)
__device__ __forceinline__ double2 cmul_ipow_sel(double2 a, int e) {
  e &= 3;
  const bool sw = e & 1;
  const double u = sw ? a.y : a.x, v = sw ? a.x : a.y;
  return make_double2((e == 1 || e == 2) ? -u : u, (e >= 2) ? -v : v);
}
__host__ __device__ constexpr int nterm(int P) { return P * (P + 1) / 2; }
typedef double dbl4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ int tidx(int n, int m) { return n * (n + 1) / 2 + m; }
// source codes of the lists: cell in the low 26 bits, periodic image above
// (image i = shift (i/9 - 1, i/3 % 3 - 1, i % 3 - 1) * cycle; cycle = 0
// without images)
__device__ __forceinline__ int cell_of(int code) { return code & ((1 << 26) - 1); }
__device__ __forceinline__ double3 image_shift(int code, double3 cyc) {
  const int i = code >> 26;
  return make_double3((i / 9 - 1) * cyc.x, (i / 3 % 3 - 1) * cyc.y, (i % 3 - 1) * cyc.z);
}
__device__ __forceinline__ double sgn(int e) { return (e & 1) ? -1.0 : 1.0; }

// decode a triangular index u = n(n+1)/2 + m (0 <= m <= n)
__device__ __forceinline__ void tdecode(int u, int &n, int &m) {
  int j = (int)((sqrtf(8.0f * u + 1.0f) - 1.0f) * 0.5f);
  while (j * (j + 1) / 2 > u) j--;
  while ((j + 1) * (j + 2) / 2 <= u) j++;
  n = j;
  m = u - j * (j + 1) / 2;
}

// Column m of the regular harmonics R[n][m], n = m..P-1, of (dx,dy,dz) into
// tab[n*P + m] (used for the M2M / L2L translation tables).
template <int P>
__device__ void regular_column(double dx, double dy, double dz, int m, double2 *tab) {
  double r2 = dx * dx + dy * dy + dz * dz;
  double2 rmm = make_double2(1.0, 0.0);
  for (int i = 1; i <= m; i++) rmm = cscale(cmul(rmm, make_double2(dx, dy)), -0.5 * c_rcp[i]);
  double2 r0 = make_double2(0.0, 0.0), r1 = rmm;
  tab[m * P + m] = rmm;
  for (int n = m + 1; n < P; n++) {
    double2 rn = cscale(csub(cscale(r1, (2 * n - 1) * dz), cscale(r0, r2)), c_rcp[n * n - m * m]);
    tab[n * P + m] = rn;
    r0 = r1;
    r1 = rn;
  }
}

// ---------------------------------------------------------------- P2M
// H = ceil(P / 2) lanes share a leaf: lane h runs the columns m = h and m' =
// P - 1 - h of the regular harmonics one after the other, P + 1 steps in all,
// so that every lane has the same number of steps and step t adds into the
// register acc[t] whatever its (n, m); the recurrence's constants sit in
// registers.  With S > 1 the bodies of a leaf are dealt to S such groups whose
// sums are added in order through LDS; a wavefront takes 64 / (H S) leaves.
// Bound: FP64 VALU (about 180 instructions a body and lane) and the serial
// steps of each body.  A lane per (body slot, m) left half its steps masked off
// and loaded a constant from memory in every step: alone, 8M cube, P = 12, 1.85 ->
// 0.67 ms, 1M Plummer, P = 10, 0.17 -> 0.09; in a solve, where P2P runs beside it
// and has most of the SIMDs, 8.0 -> 5.4 and 1.37 -> 0.86.
template <int P, int S>
__global__ __launch_bounds__(64) void p2m_kernel(DevBodies B, DevCells C, const int *__restrict__ leaves,
                                                 int nleaf, double2 *__restrict__ M) {
  using Ln = P2MLanes<P, S>;
  static_assert(Ln::sound(), "a group's sums are read from its own row and leaf");
  constexpr int NT = nterm(P);
  __shared__ double2 sRed[S > 1 ? 64 * (P + 1) : 1];
  const int lane = threadIdx.x;
  const int h = Ln::column(lane), slot = Ln::slot(lane);
  const int li = blockIdx.x * Ln::LW + Ln::leaf(lane);
  const bool act = Ln::holds(lane) && li < nleaf;
  const int c = act ? leaves[li] : 0;
  const double Xc = C.cx[c], Yc = C.cy[c], Zc = C.cz[c];
  const int b1 = act ? C.ibody[c] + C.nbody[c] : 0;
  int b = act ? C.ibody[c] + slot : 0;
  const int m1 = h, m2 = P - 1 - h, n1 = P - m1;  // steps of the first column
  // step t: degree n of its column m; r_n = (2n-1)/(n^2-m^2) z r_(n-1) - r^2/(n^2-m^2) r_(n-2),
  // started (k1 = k2 = 0 here) at n = m
  double k1[P + 1], k2[P + 1];
#pragma unroll
  for (int t = 0; t <= P; t++) {
    const bool second = t >= n1;
    const int m = second ? m2 : m1, n = m + (second ? t - n1 : t);
    const double inv = n > m ? 1.0 / (double)(n * n - m * m) : 0.0;
    k1[t] = (2 * n - 1) * inv;
    k2[t] = inv;
  }
  // (-1/2)^m / m! of the two columns
  double f1 = 1.0, f2 = 1.0;
  for (int i = 1; i <= m2; i++) {
    f2 *= -0.5 / i;
    if (i <= m1) f1 = f2;
  }
  double2 acc[P + 1];
#pragma unroll
  for (int t = 0; t <= P; t++) acc[t] = make_double2(0.0, 0.0);
  double bx = 0.0, by = 0.0, bz = 0.0, bq = 0.0;
  if (b < b1) {
    bx = B.x[b];
    by = B.y[b];
    bz = B.z[b];
    bq = B.q[b];
  }
  while (b < b1) {
    const double dx = bx - Xc, dy = by - Yc, dz = bz - Zc, q = bq;
    b += S;
    if (b < b1) {  // the next body loads during this one's recurrences
      bx = B.x[b];
      by = B.y[b];
      bz = B.z[b];
      bq = B.q[b];
    }
    const double r2 = dx * dx + dy * dy + dz * dz;
    // q (x + i y)^m of both columns from the squares
    double2 z = make_double2(dx, dy), p1 = make_double2(q * f1, 0.0), p2 = make_double2(q * f2, 0.0);
#pragma unroll
    for (int bit = 0; (1 << bit) < P; bit++) {
      if (bit > 0) z = make_double2(z.x * z.x - z.y * z.y, 2.0 * z.x * z.y);
      const double2 w1 = cmul(p1, z), w2 = cmul(p2, z);
      if ((m1 >> bit) & 1) p1 = w1;
      if ((m2 >> bit) & 1) p2 = w2;
    }
    double2 r0 = make_double2(0.0, 0.0), r1 = p1;
#pragma unroll
    for (int t = 0; t <= P; t++) {
      if (t > 0) {
        const double u = k1[t] * dz, v = k2[t] * r2;
        double2 rn = make_double2(u * r1.x - v * r0.x, u * r1.y - v * r0.y);
        const bool start = t == n1;
        r0 = start ? make_double2(0.0, 0.0) : r1;
        r1 = start ? p2 : rn;
      }
      acc[t].x += r1.x;
      acc[t].y -= r1.y;
    }
  }
  if constexpr (S > 1) {
#pragma unroll
    for (int t = 0; t <= P; t++) sRed[t * 64 + lane] = acc[t];
    __syncthreads();
    if (Ln::adds(lane)) {
#pragma unroll
      for (int t = 0; t <= P; t++)
        for (int k = 1; k < S; k++) acc[t] = cadd(acc[t], sRed[Ln::entry(t, lane, k)]);
    }
  }
  if (!act || slot > 0) return;
  double2 *Mc = M + (size_t)c * NT;
#pragma unroll
  for (int t = 0; t <= P; t++) {
    const bool second = t >= n1;
    const int m = second ? m2 : m1, n = m + (second ? t - n1 : t);
    if (!second || m2 != m1) Mc[n * (n + 1) / 2 + m] = acc[t];
  }
}

// ---------------------------------------------------------------- M2M
// One block per parent cell; children processed one after another, the
// translation table R(X_parent - X_child) staged in LDS.  Overwrites M[parent].
template <int P>
__global__ __launch_bounds__(64) void m2m_kernel(DevCells C, const int *__restrict__ cells, int ncell,
                                                 double2 *__restrict__ M) {
  constexpr int NT = nterm(P);
  constexpr int TPT = (NT + 63) / 64;
  __shared__ double2 T[P * P];
  __shared__ double2 Mc[NT];
  const int p = cells[blockIdx.x];
  const int tid = threadIdx.x;
  double2 acc[TPT];
#pragma unroll
  for (int u = 0; u < TPT; u++) acc[u] = make_double2(0.0, 0.0);
  const int c0 = C.ichild[p], nc = C.nchild[p];
  for (int c = c0; c < c0 + nc; c++) {
    const double dx = C.cx[p] - C.cx[c], dy = C.cy[p] - C.cy[c], dz = C.cz[p] - C.cz[c];
    if (tid < P) regular_column<P>(dx, dy, dz, tid, T);
    for (int u = tid; u < NT; u += 64) Mc[u] = M[(size_t)c * NT + u];
    __syncthreads();
#pragma unroll
    for (int uu = 0; uu < TPT; uu++) {
      const int u = tid + 64 * uu;
      if (u < NT) {
        int j, k;
        tdecode(u, j, k);
        double2 a = acc[uu];
        for (int n = 0; n <= j; n++) {
          const double sn = sgn(n);
          const int mlo = -n, mhi = min(k - 1, n);
          for (int m = mlo; m <= mhi; m++) {
            if (j - n >= k - m) {
              // Rc = conj(R[n][m]) (m >= 0) or R[n][-m] (m < 0); i^{m-|m|} = (-1)^m for m < 0
              double2 Rc = (m >= 0) ? cconj(T[n * P + m]) : T[n * P - m];
              double f = (m >= 0) ? sn : sn * sgn(m);
              a = cmac(a, cscale(Rc, f), Mc[tidx(j - n, k - m)]);
            }
          }
          for (int m = k; m <= n; m++) {
            if (j - n >= m - k) {
              double2 Rc = cconj(T[n * P + m]);
              a = cmac(a, cscale(Rc, sgn(k + n + m)), cconj(Mc[tidx(j - n, m - k)]));
            }
          }
        }
        acc[uu] = a;
      }
    }
    __syncthreads();
  }
#pragma unroll
  for (int uu = 0; uu < TPT; uu++) {
    const int u = tid + 64 * uu;
    if (u < NT) M[(size_t)p * NT + u] = acc[uu];
  }
}

// ---------------------------------------------------------------- L2L
// One block per child cell; pulls from its parent with R(X_child - X_parent).
template <int P>
__global__ __launch_bounds__(64) void l2l_kernel(DevCells C, const int *__restrict__ cells, int ncell,
                                                 double2 *__restrict__ L) {
  constexpr int NT = nterm(P);
  constexpr int TPT = (NT + 63) / 64;
  __shared__ double2 T[P * P];
  __shared__ double2 Lp[NT];
  const int c = cells[blockIdx.x];
  const int p = C.iparent[c];
  const int tid = threadIdx.x;
  const double dx = C.cx[c] - C.cx[p], dy = C.cy[c] - C.cy[p], dz = C.cz[c] - C.cz[p];
  if (tid < P) regular_column<P>(dx, dy, dz, tid, T);
  for (int u = tid; u < NT; u += 64) Lp[u] = L[(size_t)p * NT + u];
  __syncthreads();
#pragma unroll
  for (int uu = 0; uu < TPT; uu++) {
    const int u = tid + 64 * uu;
    if (u < NT) {
      int j, k;
      tdecode(u, j, k);
      double2 a = make_double2(0.0, 0.0);
      const double sk = sgn(k);
      for (int n = j; n < P; n++) {
        for (int m = j + k - n; m < 0; m++) {
          // (-1)^k conj(L^[n,-m]) * conj(R[n-j][k-m])
          double2 Rx = cconj(T[(n - j) * P + (k - m)]);
          a = cmac(a, cscale(cconj(Lp[tidx(n, -m)]), sk), Rx);
        }
        for (int m = 0; m <= n; m++) {
          const int d = m - k;
          if (n - j >= abs(d)) {
            double2 Rx = (d >= 0) ? T[(n - j) * P + d] : cconj(T[(n - j) * P - d]);
            double f = (d >= 0) ? 1.0 : sgn(d);
            a = cmac(a, cscale(Lp[tidx(n, m)], f), Rx);
          }
        }
      }
      double2 *Lc = L + (size_t)c * NT + u;
      *Lc = cadd(*Lc, a);
    }
  }
}

// ---------------------------------------------------------------- L2P
// One thread per body: regular harmonics of (x_b - X_leaf) streamed column by
// column; the potential and the degree-1 coefficients of the local expansion
// shifted to the body give phi and grad phi.
template <int P>
__global__ __launch_bounds__(256) void l2p_kernel(DevBodies B, DevCells C,
                                                  const int *__restrict__ body_leaf, int n,
                                                  const double2 *__restrict__ L) {
  constexpr int NT = nterm(P);
  const int b = blockIdx.x * blockDim.x + threadIdx.x;
  if (b >= n) return;
  const int c = body_leaf[b];
  const double2 *Lc = L + (size_t)c * NT;
  // kernels/laplace.h:362 offsets dX by EPS = 1e-16 in every component
  const double dx = B.x[b] - C.cx[c] + 1e-16, dy = B.y[b] - C.cy[c] + 1e-16,
               dz = B.z[b] - C.cz[c] + 1e-16;
  const double r2 = dx * dx + dy * dy + dz * dz;
  double phi = 0.0, l10 = 0.0;
  double2 l11 = make_double2(0.0, 0.0);
  double2 rbb = make_double2(1.0, 0.0);
#pragma unroll
  for (int bb = 0; bb < P; bb++) {
    if (bb > 0) rbb = cscale(cmul(rbb, make_double2(dx, dy)), -0.5 / bb);
    double2 r0 = make_double2(0.0, 0.0), r1 = make_double2(0.0, 0.0);
    const double w = bb == 0 ? 1.0 : 2.0;
#pragma unroll
    for (int a = bb; a < P; a++) {
      double2 rn = (a == bb) ? rbb
                             : cscale(csub(cscale(r1, (2 * a - 1) * dz), cscale(r0, r2)),
                                      1.0 / (a * a - bb * bb));
      const double2 La = Lc[a * (a + 1) / 2 + bb];
      phi += w * (La.x * rn.x - La.y * rn.y);
      if (a + 1 < P) {
        const double2 L1 = Lc[(a + 1) * (a + 2) / 2 + bb];
        l10 += w * (L1.x * rn.x - L1.y * rn.y);
        l11 = cmac(l11, Lc[(a + 1) * (a + 2) / 2 + bb + 1], rn);
        if (bb == 1) l11 = csub(l11, cmul(Lc[(a + 1) * (a + 2) / 2], cconj(rn)));
        if (bb >= 2) l11 = csub(l11, cconj(cmul(Lc[(a + 1) * (a + 2) / 2 + bb - 1], rn)));
      }
      r0 = r1;
      r1 = rn;
    }
  }
  B.pot[b] += phi;
  B.ax[b] += -l11.x;
  B.ay[b] += l11.y;
  B.az[b] += l10;
}

// ---------------------------------------------------------------- M2L
// Lane layout per order P: J local terms (j0..j0+J-1, fixed k) per lane, LPS
// lanes per source, SPW = 64/LPS sources in flight per wavefront.
template <int P> struct M2LCfg;
#define FMM_M2L_CFG(P_, J_, LPS_) \
  template <> struct M2LCfg<P_> { static constexpr int J = J_, LPS = LPS_; };
FMM_M2L_CFG(2, 4, 2)
FMM_M2L_CFG(3, 2, 4)
FMM_M2L_CFG(4, 4, 4)
FMM_M2L_CFG(5, 1, 16)
FMM_M2L_CFG(6, 4, 8)
FMM_M2L_CFG(7, 2, 16)
FMM_M2L_CFG(8, 3, 16)
FMM_M2L_CFG(9, 4, 16)
FMM_M2L_CFG(10, 2, 32)
FMM_M2L_CFG(11, 3, 32)
FMM_M2L_CFG(12, 3, 32)
FMM_M2L_CFG(13, 4, 32)
FMM_M2L_CFG(14, 4, 32)
FMM_M2L_CFG(15, 2, 64)
FMM_M2L_CFG(16, 3, 64)
FMM_M2L_CFG(17, 3, 64)
FMM_M2L_CFG(18, 3, 64)
FMM_M2L_CFG(19, 4, 64)
FMM_M2L_CFG(20, 4, 64)
#undef FMM_M2L_CFG

// One wavefront per target cell.  Each slot (LPS lanes) takes one source of
// the target's list per step: it stages Mh (P x (2P-1)) and generates Yh
// (rows a < 2P-1, columns b+2P-2) in LDS, then every lane accumulates its J
// terms.  Partial sums of the slots are combined in a fixed order at the end.
template <int P>
__global__ __launch_bounds__(64) void m2l_kernel(DevCells C, const int *__restrict__ targets,
                                                 int ntarget, const int *__restrict__ ptr,
                                                 const int *__restrict__ src, double3 xper,
                                                 const double2 *__restrict__ M,
                                                 double2 *__restrict__ L, int accumulate) {
  constexpr int NT = nterm(P);
  constexpr int J = M2LCfg<P>::J, LPS = M2LCfg<P>::LPS, SPW = 64 / LPS;
  constexpr int YR = 2 * P + J - 2, YC = 3 * P - 2, MC = 2 * P - 1;
  constexpr int OFF = 2 * P - 2;  // column of b = 0
  __shared__ double2 sY[SPW][YR * YC];
  __shared__ double2 sM[SPW][P * MC];

  const int lane = threadIdx.x;
  const int slot = lane / LPS, gl = lane % LPS;
  const int t = targets[blockIdx.x];
  const double Xt = C.cx[t], Yt = C.cy[t], Zt = C.cz[t];

  // lane -> (j0, k)
  int j0 = 0, k = 0;
  bool valid = false;
  {
    int g = gl;
    for (int kk = 0; kk < P; kk++) {
      const int cnt = (P - kk + J - 1) / J;
      if (g < cnt) {
        j0 = kk + g * J;
        k = kk;
        valid = true;
        break;
      }
      g -= cnt;
    }
    if (!valid) {
      j0 = 0;
      k = 0;
    }
  }

  // zero the Yh tiles once: entries never written stay finite
  for (int u = lane; u < SPW * YR * YC; u += 64) (&sY[0][0])[u] = make_double2(0.0, 0.0);
  __syncthreads();

  double2 acc[J];
#pragma unroll
  for (int tt = 0; tt < J; tt++) acc[tt] = make_double2(0.0, 0.0);

  const int beg = ptr[t], end = ptr[t + 1];
  for (int base = beg; base < end; base += SPW) {
    const int si = base + slot;
    const bool has = si < end;
    const int code = has ? src[si] : t;
    const int s = cell_of(code);
    const double3 sh = image_shift(code, xper);  // xper: the periodic cycle
    // stage Mh[n][m] = i^{-|m|} M~c[n,m]
    for (int u = gl; u < NT; u += LPS) {
      int n, m;
      tdecode(u, n, m);
      double2 v = has ? M[(size_t)s * NT + u] : make_double2(0.0, 0.0);
      sM[slot][n * MC + m + P - 1] = cmul_ipow(v, -m);
      if (m > 0) sM[slot][n * MC - m + P - 1] = cmul_ipow(cconj(v), -m);
    }
    // generate Yh[a][b] for the offset X_t - X_s - shift
    {
      double dx = Xt - C.cx[s] - sh.x, dy = Yt - C.cy[s] - sh.y, dz = Zt - C.cz[s] - sh.z;
      if (!has) {
        dx = 1.0;
        dy = 0.0;
        dz = 0.0;
      }
      const double r2 = dx * dx + dy * dy + dz * dz;
      const double inv_r = 1.0 / sqrt(r2);
      const double inv_r2 = inv_r * inv_r;
      for (int cc = gl; cc <= 2 * P - 2; cc += LPS) {
        double2 smm = make_double2(inv_r, 0.0);
        for (int i = 1; i <= cc; i++)
          smm = cscale(cmul(smm, make_double2(dx, dy)), -(2 * i - 1) * inv_r2);
        double2 sp = make_double2(0.0, 0.0), sc = smm;
        for (int a = cc; a <= 2 * P - 2; a++) {
          if (cc <= P - 1) sY[slot][a * YC + OFF + cc] = cmul_ipow(sc, cc);
          if (cc > 0) sY[slot][a * YC + OFF - cc] = cmul_ipow(cconj(sc), cc);
          double2 nx = cscale(csub(cscale(sc, (2 * a + 1) * dz), cscale(sp, (double)(a * a - cc * cc))),
                              inv_r2);
          sp = sc;
          sc = nx;
        }
      }
    }
    __syncthreads();
    const double2 *yb = &sY[slot][j0 * YC + OFF - k];
    const double2 *mb = &sM[slot][P - 1];
#pragma unroll
    for (int m = -(P - 1); m <= P - 1; m++) {
      const int am = m < 0 ? -m : m;
      double2 mc[P];
#pragma unroll
      for (int n = 0; n < P; n++)
        if (n >= am) mc[n] = mb[n * MC + m];
#pragma unroll
      for (int n = 0; n <= P + J - 2; n++) {
        if (n >= am) {
          const double2 y = yb[n * YC + m];
#pragma unroll
          for (int tt = 0; tt < J; tt++) {
            const int np = n - tt;
            if (np >= am && np <= P - 1) acc[tt] = cmac(acc[tt], mc[np], y);
          }
        }
      }
    }
    __syncthreads();
  }

  // L^[j,k] = (-1)^j i^{-k} acc; combine slots; slot 0 writes
#pragma unroll
  for (int tt = 0; tt < J; tt++) {
    const int j = j0 + tt;
    double2 v = cmul_ipow(cscale(acc[tt], sgn(j)), -k);
#pragma unroll
    for (int off = LPS; off < 64; off <<= 1) {
      v.x += __shfl_xor(v.x, off);
      v.y += __shfl_xor(v.y, off);
    }
    if (slot == 0 && valid && j <= P - 1) {
      double2 *dst = L + (size_t)t * NT + j * (j + 1) / 2 + k;
      *dst = accumulate ? cadd(*dst, v) : v;
    }
  }
}


// ---------------------------------------------------------------- M2L on MFMA
// M2L is linear in M and depends only on the offset X_t - X_s.  For one offset
// the map from M~ to L^ is a dense real P^2 x P^2 matrix T acting on
//   v(M~) = [Re M~[n,0]; Re M~[n,m], Im M~[n,m] (m>0)]  (row n^2 + (m? 2m-1 : 0), +1 for Im)
// and producing v(L^) the same way (Im L^[n,0] is identically zero and dropped):
//   A = (-1)^j i^{-(k+m)} Yh[j+n][m-k],  B = (-1)^j i^{-(k+m)} Yh[j+n][-m-k]  (m > 0)
//   Re L += (Ar+Br) Re M + (Bi-Ai) Im M,   Im L += (Ai+Bi) Re M + (Ar-Br) Im M.
// One block per chunk of <= kM2LChunkPairs pairs of one offset group, one wavefront per
// 16-row block of T (RB = ceil(P^2/16) wavefronts).  Each wavefront builds its
// rows of T once per chunk directly as MFMA A operands (registers), from the
// singular harmonics of the group's offset in LDS.  The chunk is processed in
// 16-pair slices: the block gathers v(M~) of 16 source cells into a double
// buffered B tile in LDS (the next slice is loaded into registers while the
// current one runs), every wavefront runs KP/4 v_mfma_f64_16x16x4 over it,
// and scatters its 16x16 result tile into L^ with FP64 atomic adds (the pairs
// of a group have distinct targets; the order of additions across groups is
// not fixed).
template <int P> struct MfmaCfg {
  static constexpr int PP = P * P;
  static constexpr int KP = (PP + 3) / 4 * 4;  // K padded to the MFMA depth
  static constexpr int KT = KP / 4;            // k steps
  static constexpr int RB = (PP + 15) / 16;    // 16-row blocks of T = wavefronts
  static constexpr int NTH = 64 * RB;
  static constexpr int YSZ = (2 * P - 1) * (3 * P - 2);  // complex Yh entries
  // register budget (no spills at 2-3 waves/SIMD): above P = 10 the A operands
  // grow to 36 doubles, so one slice in flight and shorter B read groups
  static constexpr int CT = 2;                 // 16-pair column tiles per slice
  static constexpr int D = P <= 10 ? 2 : 1;    // slices of multipoles in flight per thread
  static constexpr int KG = P <= 10 ? 5 : 3;   // MFMA k-steps per group of B operand reads
  static constexpr bool ok = P <= 12;
};

bool m2l_mfma_supported(int P) { return P >= 2 && P <= 12; }

constexpr int kM2LChunk = kM2LChunkPairs;

template <int P>
__global__ __launch_bounds__(MfmaCfg<P>::NTH) void m2l_mfma_kernel(const int4 *__restrict__ chunks,
                                                                   const double *__restrict__ gdx,
                                                                   const int *__restrict__ ptgt,
                                                                   const int *__restrict__ psrc,
                                                                   const double2 *__restrict__ M,
                                                                   double *__restrict__ L) {
  using Cfg = MfmaCfg<P>;
  constexpr int NT = nterm(P), PP = Cfg::PP, KP = Cfg::KP, KT = Cfg::KT, NTH = Cfg::NTH;
  constexpr int YC = 3 * P - 2, OFF = 2 * P - 2, D = Cfg::D, CT = Cfg::CT;
  constexpr int SW = 16 * CT;                     // pairs per slice
  constexpr int IT = (SW * NT + NTH - 1) / NTH;   // gathered elements per thread per slice
  __shared__ double2 sY[Cfg::YSZ];
  __shared__ double sB[2][KP * SW];
  __shared__ double sO[Cfg::RB][16 * 17];
  __shared__ int sSrc[kM2LChunk], sTgt[kM2LChunk];
  const int tid = threadIdx.x, w = tid >> 6, l = tid & 63;
  const int4 ch = chunks[blockIdx.x];
  const int g = ch.x, p0 = ch.y, cnt = ch.z;
  const int nsub = (cnt + SW - 1) / SW;
  if (cnt == 0) return;  // padding block (whole block exits before any barrier)

  for (int e = tid; e < cnt; e += NTH) {
    sSrc[e] = psrc[p0 + e];
    sTgt[e] = ptgt[p0 + e];
  }
  // singular harmonics Yh of the group offset
  {
    const double dx = gdx[3 * g], dy = gdx[3 * g + 1], dz = gdx[3 * g + 2];
    const double r2 = dx * dx + dy * dy + dz * dz;
    const double inv_r = 1.0 / sqrt(r2), inv_r2 = inv_r * inv_r;
    for (int cc = tid; cc <= 2 * P - 2; cc += NTH) {
      double2 smm = make_double2(inv_r, 0.0);
      for (int i = 1; i <= cc; i++) smm = cscale(cmul(smm, make_double2(dx, dy)), -(2 * i - 1) * inv_r2);
      double2 sp = make_double2(0.0, 0.0), sc = smm;
      for (int a = cc; a <= 2 * P - 2; a++) {
        if (cc <= P - 1) sY[a * YC + OFF + cc] = cmul_ipow(sc, cc);
        if (cc > 0) sY[a * YC + OFF - cc] = cmul_ipow(cconj(sc), cc);
        double2 nx = cscale(csub(cscale(sc, (2 * a + 1) * dz), cscale(sp, (double)(a * a - cc * cc))), inv_r2);
        sp = sc;
        sc = nx;
      }
    }
    for (int e = tid; e < (KP - PP) * SW; e += NTH) {
      sB[0][PP * SW + e] = 0.0;
      sB[1][PP * SW + e] = 0.0;
    }
  }
  __syncthreads();

  // gather v(M~) of slice sc into registers (column-fastest: conflict-free
  // staging); stage them into a B tile Bt[row * SW + col]
  double2 pre[D][IT];
  auto gather = [&](int sc, double2 *buf) {
#pragma unroll
    for (int it = 0; it < IT; it++) {
      const int e = tid + NTH * it;
      const int c = e % SW, u = e / SW;
      const int q = sc * SW + c;
      const bool ok = e < SW * NT && q < cnt;
      buf[it] = ok ? M[(size_t)cell_of(sSrc[ok ? q : 0]) * NT + u] : make_double2(0.0, 0.0);
    }
  };
  auto stage = [&](const double2 *buf, double *Bt) {
#pragma unroll
    for (int it = 0; it < IT; it++) {
      const int e = tid + NTH * it;
      if (e < SW * NT) {
        const int c = e % SW, u = e / SW;
        const int rr = c_urow[u];
        Bt[(rr & 0xffff) * SW + c] = buf[it].x;
        if ((rr >> 16) != (rr & 0xffff)) Bt[(rr >> 16) * SW + c] = buf[it].y;
      }
    }
  };
#pragma unroll
  for (int d = 0; d < D; d++) gather(d, pre[d]);

  // A operands: rows w*16 + l%16 of T, columns kt*4 + l/16
  double A[KT];
  {
    const int i = w * 16 + (l & 15);
    const int di = c_vdec[i < PP ? i : 0];
    const int j = di & 255, k = (di >> 8) & 255, io = di >> 16;
    const double sj = (j & 1) ? -1.0 : 1.0;
#pragma unroll
    for (int kt = 0; kt < KT; kt++) {
      const int kk = kt * 4 + (l >> 4);
      double val = 0.0;
      if (i < PP && kk < PP) {
        const int dk = c_vdec[kk];
        const int n = dk & 255, m = (dk >> 8) & 255, ii = dk >> 16;
        const double2 Av = cscale(cmul_ipow_sel(sY[(j + n) * YC + OFF + m - k], -(k + m)), sj);
        double2 Bv = cscale(cmul_ipow_sel(sY[(j + n) * YC + OFF - m - k], -(k + m)), sj);
        if (m == 0) Bv = make_double2(0.0, 0.0);
        const double re = ii ? (Bv.y - Av.y) : (Av.x + Bv.x);
        const double im = ii ? (Av.x - Bv.x) : (Av.y + Bv.y);
        val = io ? im : re;
      }
      A[kt] = val;
    }
  }
  // output row of this lane in the transposed store: row = w*16 + l%16
  const int orow = w * 16 + (l & 15);
  int ooff = 0;
  if (orow < PP) {
    const int dr = c_vdec[orow];
    ooff = (dr & 255) * ((dr & 255) + 1) + 2 * ((dr >> 8) & 255) + (dr >> 16);
  }
  stage(pre[0], sB[0]);
  __syncthreads();

  for (int sc0 = 0; sc0 < nsub; sc0 += D) {
#pragma unroll
    for (int d = 0; d < D; d++) {
      const int sc = sc0 + d;
      if (sc < nsub) {  // uniform across the block
        gather(sc + D, pre[d]);  // pre[d] held slice sc, already staged
        const double *Bt = sB[sc & 1];
        dbl4 acc[CT];
#pragma unroll
        for (int ct = 0; ct < CT; ct++) acc[ct] = dbl4{0.0, 0.0, 0.0, 0.0};
        // B operands are read from LDS one group of KG k-steps ahead, so the
        // MFMA chain waits on partial LDS counts instead of a full round trip
        // before every instruction.
        constexpr int KG = Cfg::KG, NKG = (KT + KG - 1) / KG;
        const double *bp = Bt + (l >> 4) * SW + (l & 15);
        double bv[2][KG][CT];
#pragma unroll
        for (int k = 0; k < KG; k++)
#pragma unroll
          for (int ct = 0; ct < CT; ct++) bv[0][k][ct] = k < KT ? bp[(k * 4) * SW + ct * 16] : 0.0;
#pragma unroll
        for (int kg = 0; kg < NKG; kg++) {
          if (kg + 1 < NKG) {
#pragma unroll
            for (int k = 0; k < KG; k++) {
              const int kt = (kg + 1) * KG + k;
#pragma unroll
              for (int ct = 0; ct < CT; ct++)
                bv[(kg + 1) & 1][k][ct] = kt < KT ? bp[(kt * 4) * SW + ct * 16] : 0.0;
            }
          }
          // keep the reads of the next group ahead of this group's MFMAs
          __builtin_amdgcn_sched_barrier(0);
#pragma unroll
          for (int k = 0; k < KG; k++) {
            const int kt = kg * KG + k;
            if (kt < KT) {
#pragma unroll
              for (int ct = 0; ct < CT; ct++)
                acc[ct] = __builtin_amdgcn_mfma_f64_16x16x4f64(A[kt], bv[kg & 1][k][ct], acc[ct], 0, 0, 0);
            }
          }
          __builtin_amdgcn_sched_barrier(0);
        }
        // D layout of v_mfma_f64_16x16x4: lane l, element v -> row (l/16) + 4v, column l%16;
        // transpose through LDS so consecutive lanes write consecutive terms of one target
        double *O = sO[w];
#pragma unroll
        for (int ct = 0; ct < CT; ct++) {
#pragma unroll
          for (int v = 0; v < 4; v++) O[(l & 15) * 17 + (l >> 4) + 4 * v] = acc[ct][v];
          __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0): this wavefront's LDS writes done
          __builtin_amdgcn_wave_barrier();
          if (orow < PP) {
#pragma unroll
            for (int cq = 0; cq < 4; cq++) {
              const int c = cq * 4 + (l >> 4);
              const int q = sc * SW + ct * 16 + c;
              if (q < cnt) unsafeAtomicAdd(&L[(size_t)sTgt[q] * 2 * NT + ooff], O[c * 17 + (l & 15)]);
            }
          }
          __builtin_amdgcn_s_waitcnt(0xc07f);
          __builtin_amdgcn_wave_barrier();
        }
        stage(pre[(d + 1) % D], sB[(sc + 1) & 1]);
        __syncthreads();
      }
    }
  }
}

// ---------------------------------------------------------------- P2P
// One wavefront per target leaf.  Lanes are (target body, source slice): the
// leaf's nt bodies (chunks of 64) take S = 64/nt slices of the sources, which
// are staged in LDS in chunks of CH bodies as {x, y, z, q}; the S partial sums
// of each body are combined through LDS in slice order.
// 1/sqrt(r2) in FP64: the hardware v_rsq_f64 estimate and one Newton step.
// Measured on MI355X against the oracle's IEEE 1/sqrt over a whole P2P
// phase (100k Plummer bodies): rel-L2 1.2e-15 (potential), 1.4e-15
// (acceleration); the reference's own SIMD rsqrt (float estimate + two Newton
// steps, vec.h:1456-1461) is at about 6e-14 per pair.  An FP32 estimate with
// one step was 3% slower and 4x less accurate, with two steps 12% slower.
__device__ __forceinline__ double rsqrt_f64(double r2) {
  const double y = __builtin_amdgcn_rsq(r2);
  return y * fma(-0.5 * r2, y * y, 1.5);
}

// Source staging of the P2P kernels.  A leaf's list is read in windows of up
// to 64 entries: lane e loads entry e's cell, image shift and body range at
// once, a wave scan turns the body counts into offsets, and the window's
// bodies, flattened, are staged CH at a time with every lane loading its own
// slots (slot f belongs to the entry e with off[e] <= f < off[e + 1], found by
// a 6-step binary search over the offsets in LDS).  The FP64 kernel leaves
// the leaf's own entry out (count 0) for its masked pass after the list.
// LDS arrays of one wavefront: its operations complete in order, the compiler
// only must not reorder them
__device__ __forceinline__ void wave_lds_order() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

struct P2PWindow {
  int off[65];
  int ib[64];
  double sx[64], sy[64], sz[64];
};

__device__ __forceinline__ int wave_incl_scan(int v) {
  const int lane = threadIdx.x & 63;
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const int t = __shfl_up(v, d, 64);
    if (lane >= d) v += t;
  }
  return v;
}

// Loads the window of entries [w0, min(w0 + 64, k1)) of leaf c's list into W;
// returns the window's body count.  With skip_own the leaf's own entry (no
// image shift) counts no bodies and sets *self.
__device__ __forceinline__ int p2p_window(P2PWindow &W, DevCells C, const int *__restrict__ src, int c, int w0,
                                          int k1, double3 xper, bool skip_own, bool *self) {
  const int lane = threadIdx.x & 63;
  const int e = w0 + lane;
  int cnt = 0, ib = 0;
  double3 sh = make_double3(0.0, 0.0, 0.0);
  bool own = false;
  if (e < k1) {
    const int code = src[e];
    const int sc = cell_of(code);
    sh = image_shift(code, xper);
    own = skip_own && sc == c && sh.x == 0.0 && sh.y == 0.0 && sh.z == 0.0;
    if (!own) {
      ib = C.ibody[sc];
      cnt = C.nbody[sc];
    }
  }
  if (__any(own)) *self = true;
  const int incl = wave_incl_scan(cnt);
  W.off[lane + 1] = incl;
  if (lane == 0) W.off[0] = 0;
  W.ib[lane] = ib;
  W.sx[lane] = sh.x;
  W.sy[lane] = sh.y;
  W.sz[lane] = sh.z;
  return __shfl(incl, 63, 64);
}

// the entry of flattened slot f of the window: the largest e with off[e] <= f
__device__ __forceinline__ int p2p_entry(const P2PWindow &W, int f) {
  int lo = 0;
#pragma unroll
  for (int step = 32; step > 0; step >>= 1)
    if (W.off[lo + step] <= f) lo += step;
  return lo;
}

// W wavefronts per target leaf (one where the leaves fill the GPU), each
// with its own staging: the list's chunks of CH bodies are dealt to them in
// turn and their sums added in order at the end.  Each lane holds K target bodies (t,
// t + nk, ... of the leaf's nk = ceil(nt / K) groups), so one LDS read of a
// source feeds K interactions, and the leaf's target groups take
// S = 64 / nk slices of the sources.
// Only pairs of bodies of one leaf can coincide in trees built here (equal
// positions fall in the same octant at every level), so the r^2 = 0 mask of
// laplace.h:192 is applied to the leaf's own entry alone, taken after the
// others; with mask_all (caller-built trees) every pair is masked.  The order
// of the sums is the same either way.
// Targets per lane by leaf size: 4 for leaves of kP2PWideLeaf bodies or more,
// 1 below (the host lists the wide leaves first; two launches).  Measured:
// 1M Plummer, P = 10 (18.7 bodies per leaf), all leaves with K = 1 / 2 / 3 / 4:
// solve 9.84 / 9.57 / 9.50 / 9.49 ms; 8M uniform cube (10.5 bodies per leaf),
// all leaves with K = 4: P2P 4% (FP64) and 20% (FP32) slower than K = 1 (a
// fifth of the lanes' targets empty, occupancy lost to registers).
template <int K, int W>
__global__ __launch_bounds__(64 * W) void p2p_kernel(DevBodies B, DevCells C, const int *__restrict__ targets,
                                                 int ntarget, const int *__restrict__ ptr,
                                                 const int *__restrict__ src, double3 xper, double eps2,
                                                 int mask_all) {
  constexpr int CH = 256;
  static_assert(64 * K <= CH, "the partial sums reuse the staging buffer");
  __shared__ double4 sball[W][CH];
  __shared__ P2PWindow win[W];
  const int lane = threadIdx.x & 63, wave = W > 1 ? __builtin_amdgcn_readfirstlane(threadIdx.x >> 6) : 0;
  double4 *sb = sball[wave];
  P2PWindow &Q = win[wave];
  const int c = targets[blockIdx.x];
  const int ib = C.ibody[c], ni = C.nbody[c];
  const int k0 = ptr[c], k1 = ptr[c + 1];
  for (int tb = 0; tb < ni; tb += 64 * K) {
    const int nt = min(ni - tb, 64 * K);
    const int nk = (nt + K - 1) / K;
    const int S = 64 / nk;
    const int tg = lane % nk, sl = lane / nk;
    const bool active = sl < S;
    int bt[K];
    double tx[K], ty[K], tz[K], ap[K], ax[K], ay[K], az[K];
#pragma unroll
    for (int h = 0; h < K; h++) {
      const int t = tg + h * nk;
      bt[h] = ib + tb + (t < nt ? t : tg);  // past the leaf: a stand-in, not stored
      tx[h] = B.x[bt[h]];
      ty[h] = B.y[bt[h]];
      tz[h] = B.z[bt[h]];
      ap[h] = ax[h] = ay[h] = az[h] = 0.0;
    }
    auto accumulate = [&](int cnt, bool mask) {
      if (!active) return;
      for (int j = sl; j < cnt; j += S) {
        const double4 s4 = sb[j];
#pragma unroll
        for (int h = 0; h < K; h++) {
          const double dx = s4.x - tx[h], dy = s4.y - ty[h], dz = s4.z - tz[h];
          const double r2 = fma(dx, dx, fma(dy, dy, fma(dz, dz, eps2)));
          const double invr = mask ? (r2 > 0.0 ? rsqrt_f64(r2) : 0.0) : rsqrt_f64(r2);
          const double qr = s4.w * invr;
          ap[h] += qr;
          const double q3 = qr * invr * invr;
          ax[h] = fma(dx, q3, ax[h]);
          ay[h] = fma(dy, q3, ay[h]);
          az[h] = fma(dz, q3, az[h]);
        }
      }
    };
    bool self = false;  // the leaf's own entry was met (and left for the masked pass)
    int turn = 0;       // of the chunks, over the wavefronts
    for (int w0 = k0; w0 < k1; w0 += 64) {
      wave_lds_order();  // the last window's readers
      const int total = p2p_window(Q, C, src, c, w0, k1, xper, true, &self);
      wave_lds_order();
      for (int base = 0; base < total; base += CH, turn++) {
        if (W > 1 && turn % W != wave) continue;
        const int cnt = min(CH, total - base);
        for (int u = lane; u < cnt; u += 64) {
          const int f = base + u, e = p2p_entry(Q, f);
          const int j = Q.ib[e] + (f - Q.off[e]);
          sb[u] = make_double4(B.x[j] + Q.sx[e], B.y[j] + Q.sy[e], B.z[j] + Q.sz[e], B.q[j]);
        }
        wave_lds_order();
        if (mask_all)
          accumulate(cnt, true);
        else
          accumulate(cnt, false);
        wave_lds_order();
      }
    }
    for (int j0 = 0; self && j0 < ni; j0 += CH, turn++) {  // the own leaf, masked
      if (W > 1 && turn % W != wave) continue;
      const int cnt = min(ni - j0, CH);
      for (int u = lane; u < cnt; u += 64) {
        const int j = ib + j0 + u;
        sb[u] = make_double4(B.x[j], B.y[j], B.z[j], B.q[j]);
      }
      wave_lds_order();
      accumulate(cnt, true);
      wave_lds_order();
    }
#pragma unroll
    for (int h = 0; h < K; h++) sb[64 * h + lane] = make_double4(ap[h], ax[h], ay[h], az[h]);
    __syncthreads();
    for (int t = threadIdx.x; t < nt; t += 64 * W) {  // target t = tg + h nk: its wavefronts and slices, in order
      const int h = t / nk, tg = t - h * nk;
      double4 acc = make_double4(0.0, 0.0, 0.0, 0.0);
#pragma unroll
      for (int w = 0; w < W; w++)
        for (int k = 0; k < S; k++) {
          const double4 v = sball[w][64 * h + tg + k * nk];
          acc.x += v.x;
          acc.y += v.y;
          acc.z += v.z;
          acc.w += v.w;
        }
      const int bi = ib + tb + t;
      B.pot[bi] = acc.x;
      B.ax[bi] = acc.y;
      B.ay[bi] = acc.z;
      B.az[bi] = acc.w;
    }
    __syncthreads();
  }
}

// ---------------------------------------------------------------- mixed precision
// FP32 arithmetic for the two list-driven phases, FP64 everywhere else (P2M,
// M2M, the harmonics of every offset, the accumulation of L, L2L, L2P).
//
// M2L in FP32 on MFMA.  Multipoles are rescaled per cell before conversion,
//   M32[c][n,m] = M~[c][n,m] / R_c^n,
// and the operator of a group (offset dX, target level lt, source level ls)
// absorbs the scales: T'[j,n] = T[j,n] R_s^n R_t^j, built in FP64 and rounded
// to FP32, so that L^[j] = R_t^-j sum_n T'[j,n] M32[n].  With R_s/|dX| and
// R_t/|dX| below the acceptance ratio every factor stays far inside the FP32
// range at any depth.  Each 16x16 FP32 tile of one group is scaled by R_t^-j
// and added into the FP64 L^ with FP64 atomics.

// M32 = M~ / R^n for every cell (one thread per coefficient)
template <int P>
__global__ __launch_bounds__(256) void m_to_f32_kernel(const double2 *__restrict__ M,
                                                       const double *__restrict__ R, int ncell,
                                                       float2 *__restrict__ M32) {
  constexpr int NT = nterm(P);
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i >= ncell * NT) return;
  const int c = i / NT, u = i - c * NT;
  const int n = c_vdec[c_urow[u] & 0xffff] & 255;
  const double inv = 1.0 / R[c];
  double f = 1.0;
  for (int k = 0; k < n; k++) f *= inv;
  const double2 v = M[i];
  M32[i] = make_float2((float)(v.x * f), (float)(v.y * f));
}

typedef float flt4 __attribute__((ext_vector_type(4)));

template <int P> struct Mfma32Cfg {
  static constexpr int PP = P * P;
  static constexpr int KP = (PP + 3) / 4 * 4;
  static constexpr int KT = KP / 4;
  static constexpr int RB = (PP + 15) / 16;
  static constexpr int NTH = 64 * RB;
  static constexpr int YSZ = (2 * P - 1) * (3 * P - 2);
  static constexpr int CT = 2, D = 2, KG = 5;
  static constexpr bool ok = P <= 12;
};

bool m2l_mixed_supported(int P) { return P >= 2 && P <= 12; }

// gscale: per group (R_s, R_t)
template <int P>
__global__ __launch_bounds__(Mfma32Cfg<P>::NTH) void m2l_mfma32_kernel(
    const int4 *__restrict__ chunks, const double *__restrict__ gdx, const double2 *__restrict__ gscale,
    const int *__restrict__ ptgt, const int *__restrict__ psrc, const float2 *__restrict__ M32,
    double *__restrict__ L) {
  using Cfg = Mfma32Cfg<P>;
  constexpr int NT = nterm(P), PP = Cfg::PP, KP = Cfg::KP, KT = Cfg::KT, NTH = Cfg::NTH;
  constexpr int YC = 3 * P - 2, OFF = 2 * P - 2, D = Cfg::D, CT = Cfg::CT;
  constexpr int SW = 16 * CT;
  constexpr int IT = (SW * NT + NTH - 1) / NTH;
  __shared__ double2 sY[Cfg::YSZ];
  __shared__ double sPow[2][P];  // R_s^n, R_t^j
  __shared__ float sB[2][KP * SW];
  __shared__ float sO[Cfg::RB][16 * 17];
  __shared__ int sSrc[kM2LChunkPairs], sTgt[kM2LChunkPairs];
  const int tid = threadIdx.x, w = tid >> 6, l = tid & 63;
  const int4 ch = chunks[blockIdx.x];
  const int g = ch.x, p0 = ch.y, cnt = ch.z;
  const int nsub = (cnt + SW - 1) / SW;
  if (cnt == 0) return;  // padding block (whole block exits before any barrier)

  for (int e = tid; e < cnt; e += NTH) {
    sSrc[e] = psrc[p0 + e];
    sTgt[e] = ptgt[p0 + e];
  }
  {
    const double dx = gdx[3 * g], dy = gdx[3 * g + 1], dz = gdx[3 * g + 2];
    const double r2 = dx * dx + dy * dy + dz * dz;
    const double inv_r = 1.0 / sqrt(r2), inv_r2 = inv_r * inv_r;
    for (int cc = tid; cc <= 2 * P - 2; cc += NTH) {
      double2 smm = make_double2(inv_r, 0.0);
      for (int i = 1; i <= cc; i++) smm = cscale(cmul(smm, make_double2(dx, dy)), -(2 * i - 1) * inv_r2);
      double2 sp = make_double2(0.0, 0.0), sc = smm;
      for (int a = cc; a <= 2 * P - 2; a++) {
        if (cc <= P - 1) sY[a * YC + OFF + cc] = cmul_ipow(sc, cc);
        if (cc > 0) sY[a * YC + OFF - cc] = cmul_ipow(cconj(sc), cc);
        double2 nx = cscale(csub(cscale(sc, (2 * a + 1) * dz), cscale(sp, (double)(a * a - cc * cc))), inv_r2);
        sp = sc;
        sc = nx;
      }
    }
    if (tid < 2) {
      const double2 rs = gscale[g];
      const double base = tid == 0 ? rs.x : rs.y;
      double pw = 1.0;
      for (int n = 0; n < P; n++) {
        sPow[tid][n] = pw;
        pw *= base;
      }
    }
    for (int e = tid; e < (KP - PP) * SW; e += NTH) {
      sB[0][PP * SW + e] = 0.0f;
      sB[1][PP * SW + e] = 0.0f;
    }
  }
  __syncthreads();

  float2 pre[D][IT];
  auto gather = [&](int sc, float2 *buf) {
#pragma unroll
    for (int it = 0; it < IT; it++) {
      const int e = tid + NTH * it;
      const int c = e % SW, u = e / SW;
      const int q = sc * SW + c;
      const bool ok = e < SW * NT && q < cnt;
      buf[it] = ok ? M32[(size_t)cell_of(sSrc[ok ? q : 0]) * NT + u] : make_float2(0.0f, 0.0f);
    }
  };
  auto stage = [&](const float2 *buf, float *Bt) {
#pragma unroll
    for (int it = 0; it < IT; it++) {
      const int e = tid + NTH * it;
      if (e < SW * NT) {
        const int c = e % SW, u = e / SW;
        const int rr = c_urow[u];
        Bt[(rr & 0xffff) * SW + c] = buf[it].x;
        if ((rr >> 16) != (rr & 0xffff)) Bt[(rr >> 16) * SW + c] = buf[it].y;
      }
    }
  };
#pragma unroll
  for (int d = 0; d < D; d++) gather(d, pre[d]);

  // A operands: rows w*16 + l%16 of T', columns kt*4 + l/16, rounded to FP32
  float A[KT];
  {
    const int i = w * 16 + (l & 15);
    const int di = c_vdec[i < PP ? i : 0];
    const int j = di & 255, k = (di >> 8) & 255, io = di >> 16;
    const double sj = ((j & 1) ? -1.0 : 1.0) * sPow[1][j];
#pragma unroll
    for (int kt = 0; kt < KT; kt++) {
      const int kk = kt * 4 + (l >> 4);
      double val = 0.0;
      if (i < PP && kk < PP) {
        const int dk = c_vdec[kk];
        const int n = dk & 255, m = (dk >> 8) & 255, ii = dk >> 16;
        const double s = sj * sPow[0][n];
        const double2 Av = cscale(cmul_ipow_sel(sY[(j + n) * YC + OFF + m - k], -(k + m)), s);
        double2 Bv = cscale(cmul_ipow_sel(sY[(j + n) * YC + OFF - m - k], -(k + m)), s);
        if (m == 0) Bv = make_double2(0.0, 0.0);
        const double re = ii ? (Bv.y - Av.y) : (Av.x + Bv.x);
        const double im = ii ? (Av.x - Bv.x) : (Av.y + Bv.y);
        val = io ? im : re;
      }
      A[kt] = (float)val;
    }
  }
  // output row of this lane in the transposed store, and its R_t^-j
  const int orow = w * 16 + (l & 15);
  int ooff = 0;
  double oscale = 0.0;
  if (orow < PP) {
    const int dr = c_vdec[orow];
    const int j = dr & 255;
    ooff = j * (j + 1) + 2 * ((dr >> 8) & 255) + (dr >> 16);
    oscale = 1.0 / sPow[1][j];
  }
  stage(pre[0], sB[0]);
  __syncthreads();

  for (int sc0 = 0; sc0 < nsub; sc0 += D) {
#pragma unroll
    for (int d = 0; d < D; d++) {
      const int sc = sc0 + d;
      if (sc < nsub) {  // uniform across the block
        gather(sc + D, pre[d]);
        const float *Bt = sB[sc & 1];
        flt4 acc[CT];
#pragma unroll
        for (int ct = 0; ct < CT; ct++) acc[ct] = flt4{0.0f, 0.0f, 0.0f, 0.0f};
        constexpr int KG = Cfg::KG, NKG = (KT + KG - 1) / KG;
        const float *bp = Bt + (l >> 4) * SW + (l & 15);
        float bv[2][KG][CT];
#pragma unroll
        for (int k = 0; k < KG; k++)
#pragma unroll
          for (int ct = 0; ct < CT; ct++) bv[0][k][ct] = k < KT ? bp[(k * 4) * SW + ct * 16] : 0.0f;
#pragma unroll
        for (int kg = 0; kg < NKG; kg++) {
          if (kg + 1 < NKG) {
#pragma unroll
            for (int k = 0; k < KG; k++) {
              const int kt = (kg + 1) * KG + k;
#pragma unroll
              for (int ct = 0; ct < CT; ct++)
                bv[(kg + 1) & 1][k][ct] = kt < KT ? bp[(kt * 4) * SW + ct * 16] : 0.0f;
            }
          }
          __builtin_amdgcn_sched_barrier(0);
#pragma unroll
          for (int k = 0; k < KG; k++) {
            const int kt = kg * KG + k;
            if (kt < KT) {
#pragma unroll
              for (int ct = 0; ct < CT; ct++)
                acc[ct] = __builtin_amdgcn_mfma_f32_16x16x4f32(A[kt], bv[kg & 1][k][ct], acc[ct], 0, 0, 0);
            }
          }
          __builtin_amdgcn_sched_barrier(0);
        }
        // D layout of v_mfma_f32_16x16x4f32: lane l, element v -> row 4(l/16) + v, column l%16
        float *O = sO[w];
#pragma unroll
        for (int ct = 0; ct < CT; ct++) {
#pragma unroll
          for (int v = 0; v < 4; v++) O[(l & 15) * 17 + 4 * (l >> 4) + v] = acc[ct][v];
          __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0): this wavefront's LDS writes done
          __builtin_amdgcn_wave_barrier();
          if (orow < PP) {
#pragma unroll
            for (int cq = 0; cq < 4; cq++) {
              const int c = cq * 4 + (l >> 4);
              const int q = sc * SW + ct * 16 + c;
              if (q < cnt)
                unsafeAtomicAdd(&L[(size_t)sTgt[q] * 2 * NT + ooff], (double)O[c * 17 + (l & 15)] * oscale);
            }
          }
          __builtin_amdgcn_s_waitcnt(0xc07f);
          __builtin_amdgcn_wave_barrier();
        }
        stage(pre[(d + 1) % D], sB[(sc + 1) & 1]);
        __syncthreads();
      }
    }
  }
}

// P2P in FP32.  Positions are taken relative to the target leaf's centre in
// FP64 and then rounded, so the FP32 differences carry the leaf-scale
// precision, not the domain-scale one.  1/r is v_rsq_f32.  Each lane sums at
// most 32 sources in FP32 before adding the partial sums into FP64
// accumulators (cascaded summation: the FP32 rounding of a partial covers 32
// terms, never the whole list).
// Each lane holds K target bodies, as in p2p_kernel.
template <int K, int W>
__global__ __launch_bounds__(64 * W) void p2p32_kernel(DevBodies B, DevCells C, const int *__restrict__ targets,
                                                   int ntarget, const int *__restrict__ ptr,
                                                   const int *__restrict__ src, double3 xper, double eps2) {
  constexpr int CH = 256, RUN = 32;
  constexpr int NRED = 64 * K > CH / 2 ? 64 * K : CH / 2;  // holds the CH FP32 staging slots too
  __shared__ double4 sball[W][NRED];  // the FP32 staging buffer lives in the same bytes
  __shared__ P2PWindow win[W];
  const int lane = threadIdx.x & 63, wave = W > 1 ? __builtin_amdgcn_readfirstlane(threadIdx.x >> 6) : 0;
  float4 *sb = reinterpret_cast<float4 *>(sball[wave]);
  P2PWindow &Q = win[wave];
  const int c = targets[blockIdx.x];
  const int ib = C.ibody[c], ni = C.nbody[c];
  const int k0 = ptr[c], k1 = ptr[c + 1];
  const double Xc = C.cx[c], Yc = C.cy[c], Zc = C.cz[c];
  const float e2 = (float)eps2;
  for (int tb = 0; tb < ni; tb += 64 * K) {
    const int nt = min(ni - tb, 64 * K);
    const int nk = (nt + K - 1) / K;
    const int S = 64 / nk;
    const int tg = lane % nk, sl = lane / nk;
    const bool active = sl < S;
    float tx[K], ty[K], tz[K];
    double ap[K], ax[K], ay[K], az[K];
#pragma unroll
    for (int h = 0; h < K; h++) {
      const int t = tg + h * nk;
      const int bi = ib + tb + (t < nt ? t : tg);  // past the leaf: a stand-in, not stored
      tx[h] = (float)(B.x[bi] - Xc);
      ty[h] = (float)(B.y[bi] - Yc);
      tz[h] = (float)(B.z[bi] - Zc);
      ap[h] = ax[h] = ay[h] = az[h] = 0.0;
    }
    int turn = 0;  // of the chunks, over the wavefronts (a chunk's FP32 partial sums do not depend on W)
    for (int w0 = k0; w0 < k1; w0 += 64) {
      bool unused = false;
      wave_lds_order();  // the last window's readers
      const int total = p2p_window(Q, C, src, c, w0, k1, xper, false, &unused);
      wave_lds_order();
      for (int base = 0; base < total; base += CH, turn++) {
        if (W > 1 && turn % W != wave) continue;
        const int cnt = min(CH, total - base);
        for (int u = lane; u < cnt; u += 64) {
          const int f = base + u, e = p2p_entry(Q, f);
          const int j = Q.ib[e] + (f - Q.off[e]);
          sb[u] = make_float4((float)(B.x[j] + Q.sx[e] - Xc), (float)(B.y[j] + Q.sy[e] - Yc),
                              (float)(B.z[j] + Q.sz[e] - Zc), (float)B.q[j]);
        }
        wave_lds_order();
        if (active) {
          for (int j0 = sl; j0 < cnt; j0 += RUN * S) {
            const int jend = min(cnt, j0 + RUN * S);
            float p[K], fx[K], fy[K], fz[K];
#pragma unroll
            for (int h = 0; h < K; h++) p[h] = fx[h] = fy[h] = fz[h] = 0.0f;
            for (int j = j0; j < jend; j += S) {
              const float4 s4 = sb[j];
#pragma unroll
              for (int h = 0; h < K; h++) {
                const float dx = s4.x - tx[h], dy = s4.y - ty[h], dz = s4.z - tz[h];
                const float r2 = fmaf(dx, dx, fmaf(dy, dy, fmaf(dz, dz, e2)));
                const float invr = r2 > 0.0f ? __builtin_amdgcn_rsqf(r2) : 0.0f;
                const float qr = s4.w * invr;
                p[h] += qr;
                const float q3 = qr * invr * invr;
                fx[h] = fmaf(dx, q3, fx[h]);
                fy[h] = fmaf(dy, q3, fy[h]);
                fz[h] = fmaf(dz, q3, fz[h]);
              }
            }
#pragma unroll
            for (int h = 0; h < K; h++) {
              ap[h] += p[h];
              ax[h] += fx[h];
              ay[h] += fy[h];
              az[h] += fz[h];
            }
          }
        }
        wave_lds_order();
      }
    }
#pragma unroll
    for (int h = 0; h < K; h++) sball[wave][64 * h + lane] = make_double4(ap[h], ax[h], ay[h], az[h]);
    __syncthreads();
    for (int t = threadIdx.x; t < nt; t += 64 * W) {  // target t = tg + h nk: its wavefronts and slices, in order
      const int h = t / nk, tg = t - h * nk;
      double4 acc = make_double4(0.0, 0.0, 0.0, 0.0);
#pragma unroll
      for (int w = 0; w < W; w++)
        for (int k = 0; k < S; k++) {
          const double4 v = sball[w][64 * h + tg + k * nk];
          acc.x += v.x;
          acc.y += v.y;
          acc.z += v.z;
          acc.w += v.w;
        }
      const int bi = ib + tb + t;
      B.pot[bi] = acc.x;
      B.ax[bi] = acc.y;
      B.ay[bi] = acc.z;
      B.az[bi] = acc.w;
    }
    __syncthreads();
  }
}

// ---------------------------------------------------------------- periodic far images
// Traversal::traversePeriodic (include/traversal.h:233-287) translates the
// root multipole to the root local expansion through images - 1 levels of
// ever larger supercells.  Every step is linear in the root multipole and
// fixed by the geometry, so the whole far field is one real P^2 x P^2
// operator F on the expansion vectors, built once per plan:
//   F = sum_l T_l S_(l-1) ... S_0,  T_l = sum of the level's M2L operators,
//   S_l = I + sum of the level's supercell M2M operators,
// and applied each evaluation with one matrix-vector product.

// Both operators are linear in the harmonics of their offset, so a level needs
// only the harmonics' sums over its offsets (M2L: w cycle for the integer w of
// the cube |w| <= prange nb + prange without |w| <= prange; M2M: |i| <= prange
// without 0; nb = 2 prange + 1) and one operator of each: summing the 15500
// operators themselves (prange = 2) took 1.1 ms a level at P = 10.  Blocks 0 ..
// kFarBlocks - 1: part[block][a][b] = sums of the singular harmonics; block
// kFarBlocks: rsum[n P + m] = sums of the regular ones.  Fixed order.
constexpr int kFarBlocks = 48;
template <int P>
__global__ __launch_bounds__(256) void far_sums_kernel(int prange, double3 cyc, double2 *__restrict__ part,
                                                       double2 *__restrict__ rsum) {
  constexpr int NC = 2 * P - 1;
  __shared__ double2 sum[NC * NC];
  const int tid = threadIdx.x, nb = 2 * prange + 1;
  double2 acc[NC];
#pragma unroll
  for (int a = 0; a < NC; a++) acc[a] = make_double2(0.0, 0.0);
  for (int e = tid; e < NC * NC; e += 256) sum[e] = make_double2(0.0, 0.0);
  const bool reg = blockIdx.x == kFarBlocks;
  const int ncol = reg ? P : NC, SL = 256 / ncol;
  const int col = tid % ncol, slot = tid / ncol;
  if (slot < SL) {
    static_assert((2 * kFarMaxRange + 1) <= 35, "side^3 and the last step past it fit an int up to 35^6 + 48 * 256");
    const int side = reg ? nb : nb * nb, half = side / 2;
    const int first = reg ? slot : blockIdx.x * SL + slot, step = reg ? SL : kFarBlocks * SL;
    for (int e = first; e < side * side * side; e += step) {
      const int wx = e / (side * side) - half, wy = e / side % side - half, wz = e % side - half;
      if (max(abs(wx), max(abs(wy), abs(wz))) <= (reg ? 0 : prange)) continue;
      const double dx = -wx * cyc.x, dy = -wy * cyc.y, dz = -wz * cyc.z;
      const double r2 = dx * dx + dy * dy + dz * dz;
      double2 c0 = make_double2(0.0, 0.0), c1;
      if (reg) {
        c1 = make_double2(1.0, 0.0);
        for (int i = 1; i <= col; i++) c1 = cscale(cmul(c1, make_double2(dx, dy)), -0.5 * c_rcp[i]);
#pragma unroll
        for (int n = 0; n < P; n++)
          if (n >= col) {
            if (n > col) {
              const double2 cn = cscale(csub(cscale(c1, (2 * n - 1) * dz), cscale(c0, r2)), c_rcp[n * n - col * col]);
              c0 = c1;
              c1 = cn;
            }
            acc[n] = cadd(acc[n], c1);
          }
      } else {
        const double inv_r = 1.0 / sqrt(r2), inv_r2 = inv_r * inv_r;
        c1 = make_double2(inv_r, 0.0);
        for (int i = 1; i <= col; i++) c1 = cscale(cmul(c1, make_double2(dx, dy)), -(2 * i - 1) * inv_r2);
#pragma unroll
        for (int a = 0; a < NC; a++)
          if (a >= col) {
            acc[a] = cadd(acc[a], c1);
            const double2 cn =
                cscale(csub(cscale(c1, (2 * a + 1) * dz), cscale(c0, (double)(a * a - col * col))), inv_r2);
            c0 = c1;
            c1 = cn;
          }
      }
    }
  }
  for (int k = 0; k < SL; k++) {
    __syncthreads();
    if (slot == k)
#pragma unroll
      for (int a = 0; a < NC; a++) sum[a * NC + col] = cadd(sum[a * NC + col], acc[a]);
  }
  __syncthreads();
  if (reg)
    for (int e = tid; e < P * P; e += 256) rsum[e] = sum[(e / P) * NC + e % P];
  else
    for (int e = tid; e < NC * NC; e += 256) part[(size_t)blockIdx.x * NC * NC + e] = sum[e];
}

// The level's operators from the sums (row-major P^2 x P^2, rows and columns
// n^2 + (m ? 2m-1 : 0), +1 for imaginary parts): blocks 0 .. nt - 1 T (v(L^) =
// T v(M~)), the rest S = I + the supercell M2M operators.
template <int P>
__global__ __launch_bounds__(256) void far_ops_kernel(const double2 *__restrict__ part,
                                                      const double2 *__restrict__ rsum, int nt,
                                                      double *__restrict__ T, double *__restrict__ S) {
  constexpr int PP = P * P, NT = nterm(P), NC = 2 * P - 1, YC = 3 * P - 2, OFF = 2 * P - 2;
  __shared__ double2 sY[NC * YC];
  const int tid = threadIdx.x;
  if ((int)blockIdx.x < nt) {
    for (int e = tid; e < NC * NC; e += 256) {
      const int a = e / NC, cc = e - a * NC;
      if (cc > a) continue;
      double2 v = make_double2(0.0, 0.0);
      for (int k = 0; k < kFarBlocks; k++) v = cadd(v, part[(size_t)k * NC * NC + e]);
      if (cc <= P - 1) sY[a * YC + OFF + cc] = cmul_ipow(v, cc);
      if (cc > 0) sY[a * YC + OFF - cc] = cmul_ipow(cconj(v), cc);
    }
    __syncthreads();
    const int e = blockIdx.x * 256 + tid;
    if (e >= PP * PP) return;
    const int row = e / PP, col = e - row * PP;
    const int di = c_vdec[row], dk = c_vdec[col];
    const int j = di & 255, k = (di >> 8) & 255, io = di >> 16;
    const int nn = dk & 255, m = (dk >> 8) & 255, ii = dk >> 16;
    const double sj = (j & 1) ? -1.0 : 1.0;
    const double2 Av = cscale(cmul_ipow_sel(sY[(j + nn) * YC + OFF + m - k], -(k + m)), sj);
    double2 Bv = cscale(cmul_ipow_sel(sY[(j + nn) * YC + OFF - m - k], -(k + m)), sj);
    if (m == 0) Bv = make_double2(0.0, 0.0);
    const double re = ii ? (Bv.y - Av.y) : (Av.x + Bv.x);
    const double im = ii ? (Av.x - Bv.x) : (Av.y + Bv.y);
    T[e] = io ? im : re;
    return;
  }
  for (int e = tid; e < PP; e += 256) sY[e] = rsum[e];
  __syncthreads();
  const int e = (blockIdx.x - nt) * 256 + tid;
  if (e >= PP * NT) return;
  const int col = e / NT, u = e - col * NT;
  const int dc = c_vdec[col];
  const int ia = dc & 255, ib = (dc >> 8) & 255;
  const double2 v = (dc >> 16) ? make_double2(0.0, 1.0) : make_double2(1.0, 0.0);
  int j, k;
  tdecode(u, j, k);
  // the scalar M2M of m2m_kernel with a unit child multipole at (ia, ib): its
  // terms (n, m) with (j - n, |k - m|) = (ia, ib)
  double2 a = make_double2(0.0, 0.0);
  const int n = j - ia;
  if (n >= 0) {
    const double sn = sgn(n);
    const int m = k - ib;  // k - m = ib >= 0, m <= k - 1 or (ib = 0) m = k
    if (ib > 0 && m >= -n && m <= n) {
      const double2 Rc = (m >= 0) ? cconj(sY[n * P + m]) : sY[n * P - m];
      a = cmac(a, cscale(Rc, (m >= 0) ? sn : sn * sgn(m)), v);
    }
    const int m2 = k + ib;  // m - k = ib >= 0
    if (m2 <= n) a = cmac(a, cscale(cconj(sY[n * P + m2]), sgn(k + n + m2)), cconj(v));
  }
  const int row = j * j + (k ? 2 * k - 1 : 0);
  S[row * PP + col] = a.x + (row == col ? 1.0 : 0.0);
  if (k) S[(row + 1) * PP + col] = a.y + (row + 1 == col ? 1.0 : 0.0);
}

// C = A B (+ C when acc), n x n, row-major with leading dimension n
__global__ __launch_bounds__(256) void matmul_kernel(const double *__restrict__ A, const double *__restrict__ B,
                                                     double *__restrict__ C, int n, int acc) {
  const int e = blockIdx.x * 256 + threadIdx.x;
  if (e >= n * n) return;
  const int i = e / n, j = e - i * n;
  double s = acc ? C[e] : 0.0;
  for (int k = 0; k < n; k++) s = fma(A[i * n + k], B[k * n + j], s);
  C[e] = s;
}

// L^(root) += F v(M~(root))
template <int P>
__global__ __launch_bounds__(256) void periodic_far_kernel(const double *__restrict__ F, const double2 *__restrict__ M,
                                                           double2 *__restrict__ L) {
  constexpr int PP = P * P, NT = nterm(P);
  __shared__ double v[PP];
  const int tid = threadIdx.x;
  for (int c = tid; c < PP; c += 256) {
    const int dc = c_vdec[c];
    const double2 m = M[tidx(dc & 255, (dc >> 8) & 255)];
    v[c] = (dc >> 16) ? m.y : m.x;
  }
  __syncthreads();
  for (int r = tid; r < PP; r += 256) {
    double s = 0.0;
    for (int c = 0; c < PP; c++) s = fma(F[r * PP + c], v[c], s);
    const int dr = c_vdec[r];
    const int j = dr & 255;
    double *dst = reinterpret_cast<double *>(L) + j * (j + 1) + 2 * ((dr >> 8) & 255) + (dr >> 16);
    *dst += s;
  }
  (void)NT;
}

// ---------------------------------------------------------------- direct
// Verification sum.  Uses IEEE sqrt and division (not the P2P rsqrt path) so it
// checks the P2P kernel independently.  A block holds 64 targets and a run of
// `chunk` sources, staged 256 at a time through LDS, a quarter of them (of the
// images, where there are any) to each of its 4 wavefronts; the quarters are
// added in order through LDS and the runs by direct_sum_kernel (part: [run][pot, ax, ay, az][nt]; one run writes
// the result itself).  Bound: FP64 VALU (about 45 instructions a pair).
// Accuracy checks sum a thousand targets over all bodies: with one thread per
// target over every source, 1000 targets of 2^20 bodies ran on 4 blocks.
// Measured there: 190 -> 1.7 ms a call.
__global__ __launch_bounds__(256) void direct_kernel(DevBodies B, int n, const double *__restrict__ tx,
                                                     const double *__restrict__ ty,
                                                     const double *__restrict__ tz, int nt, int chunk,
                                                     double *__restrict__ part, double eps2, int prange,
                                                     double3 cyc) {
  __shared__ double4 sb[256];
  __shared__ double sr[4][4][64];  // [wavefront][component][target]
  const int l = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int i = blockIdx.x * 64 + l;
  const bool act = i < nt;
  const double xi = act ? tx[i] : 0.0, yi = act ? ty[i] : 0.0, zi = act ? tz[i] : 0.0;
  const long long first = (long long)blockIdx.y * chunk;
  const int j0 = (int)min((long long)n, first), j1 = (int)min((long long)n, first + chunk);
  double pot = 0.0, ax = 0.0, ay = 0.0, az = 0.0;
  for (int base = j0; base < j1; base += 256) {
    const int j = base + threadIdx.x;
    if (j < j1) sb[threadIdx.x] = make_double4(B.x[j], B.y[j], B.z[j], B.q[j]);
    __syncthreads();
    const int cnt = min(256, j1 - base);
    auto add = [&](double px, double py, double pz, int k0, int k1) {
      for (int k = k0; k < k1; k++) {
        const double4 s4 = sb[k];
        const double dx = px - s4.x, dy = py - s4.y, dz = pz - s4.z;
        const double r2 = dx * dx + dy * dy + dz * dz + eps2;
        if (r2 != 0.0) {
          const double inv2 = 1.0 / r2;
          const double qr = s4.w * sqrt(inv2);
          const double q3 = inv2 * qr;
          pot += qr;
          ax -= dx * q3;
          ay -= dy * q3;
          az -= dz * q3;
        }
      }
    };
    if (prange == 0) {
      add(xi, yi, zi, 64 * w, min(64 * w + 64, cnt));
    } else {
      // periodic images (Traversal::direct, include/traversal.h:355-377): sources
      // shifted by (ix, iy, iz) * cycle, |ix|, |iy|, |iz| <= prange, dealt to the
      // wavefronts; an image's sources stay together (a neutral system's terms
      // cancel image by image: quarters of them summed apart lost two digits)
      const int m = 2 * prange + 1;
      for (long long e = w; e < (long long)m * m * m; e += 4) {
        const int ix = (int)(e / ((long long)m * m)) - prange, iy = (int)(e / m % m) - prange, iz = (int)(e % m) - prange;
        add(xi - ix * cyc.x, yi - iy * cyc.y, zi - iz * cyc.z, 0, cnt);
      }
    }
    __syncthreads();
  }
  sr[w][0][l] = pot;
  sr[w][1][l] = ax;
  sr[w][2][l] = ay;
  sr[w][3][l] = az;
  __syncthreads();
  // wavefront w adds component w
  if (act)
    part[((size_t)blockIdx.y * 4 + w) * nt + i] = ((sr[0][w][l] + sr[1][w][l]) + sr[2][w][l]) + sr[3][w][l];
}

__global__ __launch_bounds__(256) void direct_sum_kernel(const double *__restrict__ part, int runs, int n4,
                                                         double *__restrict__ out) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i >= n4) return;
  double v = 0.0;
  for (int r = 0; r < runs; r++) v += part[(size_t)r * n4 + i];
  out[i] = v;
}

// sources per run: about 2048 blocks (8 a CU) in all, whole staging buffers
static int direct_chunk(int n, int nt) {
  const long long groups = (nt + 63) / 64, runs = std::max(1LL, 2048 / std::max(1LL, groups));
  const long long c = ((n + runs - 1) / runs + 255) / 256 * 256;
  return (int)std::max(256LL, std::min(c, 1LL << 30));
}
int direct_runs(int n, int nt) {
  const int c = direct_chunk(n, nt);
  return n <= 0 ? 1 : (n - 1) / c + 1;
}

// UpDownPass::getDipole(bodies, X0 = 0) (include/up_down_pass.h:77-86): per-block
// partial sums of q x, fixed order, no atomics
__global__ __launch_bounds__(256) void dipole_partial_kernel(DevBodies B, int n, double *__restrict__ part) {
  __shared__ double s[3][256];
  double d0 = 0.0, d1 = 0.0, d2 = 0.0;
  for (int i = blockIdx.x * 256 + threadIdx.x; i < n; i += gridDim.x * 256) {
    const double q = B.q[i];
    d0 += B.x[i] * q;
    d1 += B.y[i] * q;
    d2 += B.z[i] * q;
  }
  s[0][threadIdx.x] = d0;
  s[1][threadIdx.x] = d1;
  s[2][threadIdx.x] = d2;
  __syncthreads();
  for (int w = 128; w > 0; w >>= 1) {
    if (threadIdx.x < w)
      for (int d = 0; d < 3; d++) s[d][threadIdx.x] += s[d][threadIdx.x + w];
    __syncthreads();
  }
  if (threadIdx.x < 3) part[3 * blockIdx.x + threadIdx.x] = s[threadIdx.x][0];
}

// UpDownPass::dipoleCorrection (include/up_down_pass.h:89-99): every block sums
// the nb partials in the same order, so all bodies see the same dipole D;
// pot -= coef |D|^2 / (n q), grad -= coef D
__global__ __launch_bounds__(256) void dipole_apply_kernel(DevBodies B, int n, const double *__restrict__ part,
                                                           int nb, double coef) {
  __shared__ double D[3];
  if (threadIdx.x < 3) {
    double a = 0.0;
    for (int b = 0; b < nb; b++) a += part[3 * b + threadIdx.x];
    D[threadIdx.x] = a;
  }
  __syncthreads();
  const double dd = D[0] * D[0] + D[1] * D[1] + D[2] * D[2];
  for (int i = blockIdx.x * 256 + threadIdx.x; i < n; i += gridDim.x * 256) {
    B.pot[i] -= coef * dd / n / B.q[i];
    B.ax[i] -= coef * D[0];
    B.ay[i] -= coef * D[1];
    B.az[i] -= coef * D[2];
  }
}

int dipole_partials(int n) { return n <= 0 ? 0 : min(256, (n + 255) / 256); }

hipError_t launch_dipole_correction(DevBodies B, int n, double *part, double coef, hipStream_t s) {
  const int nb = dipole_partials(n);
  if (nb == 0) return hipSuccess;
  hipLaunchKernelGGL(dipole_partial_kernel, dim3(nb), dim3(256), 0, s, B, n, part);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(dipole_apply_kernel, dim3(min(2048, (n + 255) / 256)), dim3(256), 0, s, B, n, part, nb, coef);
  return hipGetLastError();
}

// ---------------------------------------------------------------- Ewald sum
// Ewald (include/ewald.h), the validator of the periodic path, on the device.
// Bodies are read through EwBodies: positions and forces with a stride (1 for
// structure-of-arrays buffers, 3 for a caller's n x 3 arrays), each position
// wrapped once into [-cycle/2, cycle/2] as it is loaded (vec.h:217-230, as
// FMM_Ewald does before its sum, md_distributed.cxx:329).
// Wave part: S(k) = sum_j q_j e^{i k.x_j} per wave vector (one block per wave,
// fixed-order reduction), scaled by 2/(sigma V) e^{-K^2/4 alpha^2}/K^2
// (ewald.h:163-180), then every body sums its waves (ewald.h:43-60).
__device__ __forceinline__ double wrap1(double v, double L) {
  if (v < -L / 2) v += L;
  if (v > L / 2) v -= L;
  return v;
}
__device__ __forceinline__ double3 ew_pos(const EwBodies &B, int i, double3 cyc) {
  const size_t o = (size_t)i * B.xs;
  return make_double3(wrap1(B.x[o], cyc.x), wrap1(B.y[o], cyc.y), wrap1(B.z[o], cyc.z));
}
__device__ __forceinline__ void ew_add(const EwBodies &B, int i, double p, double gx, double gy, double gz) {
  const size_t o = (size_t)i * B.fs;
  B.pot[i] += p;
  B.ax[o] += gx;
  B.ay[o] += gy;
  B.az[o] += gz;
}

// Ewald::initWaves (include/ewald.h:64-88): the wave vectors (l, m, k) of the
// half space, |k| <= ksize, in the order of its loops (l outer, k inner), one
// block: rows (l, m) in runs of 256, each row's count of k, a prefix sum over
// the run, then each row writes its own k.
__device__ __forceinline__ int isqrt_floor(int v) {  // floor(sqrt(v)), v >= 0
  int r = (int)sqrt((double)v);
  while (r * r > v) r--;
  while ((r + 1) * (r + 1) <= v) r++;
  return r;
}
__global__ __launch_bounds__(256) void ewald_waves_kernel(int ksize, int *__restrict__ kv) {
  __shared__ int off[257];
  const int W = 2 * ksize + 1, nrow = (ksize + 1) * W, tid = threadIdx.x;
  int base = 0;
  for (int r0 = 0; r0 < nrow; r0 += 256) {
    const int r = r0 + tid;
    int cnt = 0, kmin = 0, kmax = -1, l = 0, m = 0;
    if (r < nrow) {
      l = r / W;
      m = r % W - ksize;
      const int rem = ksize * ksize - l * l - m * m;
      if (rem >= 0 && !(l == 0 && m < 0)) {
        kmax = isqrt_floor(rem);
        kmin = (l == 0 && m == 0) ? 1 : -kmax;
        cnt = kmax >= kmin ? kmax - kmin + 1 : 0;
      }
    }
    off[tid + 1] = cnt;
    __syncthreads();
    if (tid == 0) {
      off[0] = base;
      for (int t = 1; t <= 256; t++) off[t] += off[t - 1];
    }
    __syncthreads();
    for (int k = kmin, o = off[tid]; k <= kmax && cnt > 0; k++, o++) {
      kv[3 * o] = l;
      kv[3 * o + 1] = m;
      kv[3 * o + 2] = k;
    }
    base = off[256];
    __syncthreads();
  }
}

int ewald_nwaves(int ksize) {
  if (ksize < 0) return 0;
  int nw = 0;
  for (int l = 0; l <= ksize; l++)
    for (int m = l == 0 ? 0 : -ksize; m <= ksize; m++) {
      const int rem = ksize * ksize - l * l - m * m;
      if (rem < 0) continue;
      int kmax = (int)std::sqrt((double)rem);
      while (kmax * kmax > rem) kmax--;
      while ((kmax + 1) * (kmax + 1) <= rem) kmax++;
      nw += (l == 0 && m == 0) ? kmax : 2 * kmax + 1;
    }
  return nw;
}

__global__ __launch_bounds__(256) void ewald_dft_kernel(EwBodies B, int n, const int *__restrict__ kv, int nw,
                                                        double3 cyc, double3 scale, double coef, double coef2,
                                                        double2 *__restrict__ S) {
  __shared__ double sre[256], sim[256];
  const int w = blockIdx.x, tid = threadIdx.x;
  if (w >= nw) return;
  const double kx = kv[3 * w] * scale.x, ky = kv[3 * w + 1] * scale.y, kz = kv[3 * w + 2] * scale.z;
  double re = 0.0, im = 0.0;
  for (int j = tid; j < n; j += 256) {
    const double3 xj = ew_pos(B, j, cyc);
    double sn, cs;
    sincos(kx * xj.x + ky * xj.y + kz * xj.z, &sn, &cs);
    re += B.q[j] * cs;
    im += B.q[j] * sn;
  }
  sre[tid] = re;
  sim[tid] = im;
  __syncthreads();
  for (int h = 128; h > 0; h >>= 1) {
    if (tid < h) {
      sre[tid] += sre[tid + h];
      sim[tid] += sim[tid + h];
    }
    __syncthreads();
  }
  if (tid == 0) {
    const double K2 = kx * kx + ky * ky + kz * kz;
    const double factor = coef * exp(-K2 * coef2) / K2;
    S[w] = make_double2(sre[0] * factor, sim[0] * factor);
  }
}

// The sum over the waves runs kEwT bodies a block, every body's terms dealt to
// kEwS lanes (slices) and their partial sums added in slice order through LDS:
// with a thread per body, 24573 bodies filled 96 of the 256 CUs with one
// wavefront per SIMD (that system, 1500 wave vectors: 370 -> 110 us).
constexpr int kEwT = 16, kEwS = 256 / kEwT;
__device__ __forceinline__ double4 ew_reduce(double4 v, double4 *sr) {  // the total in slice 0's lanes
  __syncthreads();
  sr[threadIdx.x] = v;
  __syncthreads();
  if (threadIdx.x < kEwT)
    for (int k = 1; k < kEwS; k++) {
      const double4 u = sr[threadIdx.x + kEwT * k];
      v.x += u.x;
      v.y += u.y;
      v.z += u.z;
      v.w += u.w;
    }
  return v;
}

__global__ __launch_bounds__(256) void ewald_idft_kernel(EwBodies B, int n, const int *__restrict__ kv,
                                                         const double2 *__restrict__ S, int nw, double3 cyc,
                                                         double3 scale) {
  __shared__ double4 sw[256];  // kx, ky, kz scaled; re
  __shared__ double si[256];   // im
  const int i = blockIdx.x * kEwT + threadIdx.x % kEwT, slice = threadIdx.x / kEwT;
  const bool act = i < n;
  const double3 xi = act ? ew_pos(B, i, cyc) : make_double3(0.0, 0.0, 0.0);
  double p = 0.0, gx = 0.0, gy = 0.0, gz = 0.0;
  for (int w0 = 0; w0 < nw; w0 += 256) {
    const int w = w0 + threadIdx.x;
    if (w < nw) {
      sw[threadIdx.x] = make_double4(kv[3 * w] * scale.x, kv[3 * w + 1] * scale.y, kv[3 * w + 2] * scale.z, S[w].x);
      si[threadIdx.x] = S[w].y;
    }
    __syncthreads();
    const int cnt = min(256, nw - w0);
    for (int k = slice; k < cnt; k += kEwS) {
      const double4 kw = sw[k];
      double sn, cs;
      sincos(kw.x * xi.x + kw.y * xi.y + kw.z * xi.z, &sn, &cs);
      const double re = kw.w, im = si[k];
      p += re * cs + im * sn;
      const double dt = re * sn - im * cs;
      gx -= dt * kw.x;
      gy -= dt * kw.y;
      gz -= dt * kw.z;
    }
    __syncthreads();
  }
  const double4 v = ew_reduce(make_double4(p, gx, gy, gz), sw);
  if (act && slice == 0) ew_add(B, i, v.x, v.y, v.z, v.w);
}

// (x + K) e^{x^2} erfc(x), K = 3.75, x >= 0, as a polynomial in
// t = (x - K) / (x + K): the transform of Shepherd and Laframboise (Math. Comp.
// 36, 1981) on a factor that keeps the function finite at both ends, its
// Chebyshev series in 60-digit arithmetic cut after t^23 (next term 4e-18).
// e^{x^2} erfc(x) by it: 1.9e-16 rms, 6.6e-16 at most over [0, 3000].
struct Erfcx {
  double c[24];
};
constexpr Erfcx kErfcx = {{
    1.0919229095627891,     -0.95874157665290949,    0.73631892522175368,     -0.49047029120768826,
    0.2790620490336852,     -0.13195540117824336,    0.049118778617206059,    -0.012535880044978472,
    0.00098633806014572696, 0.0007948231282476774,   -0.00034864674071764747, 1.0593866720431546e-05,
    3.7471310663113975e-05, -8.9036267414649746e-06, -3.288570958593065e-06,  1.6555849395166649e-06,
    2.7865722181858276e-07, -2.6337499684119528e-07, -2.5922843337984979e-08, 4.0207875133061638e-08,
    2.774844499122888e-09,  -5.3688142939511958e-09, -2.2991140565077379e-10, 4.4046755782598165e-10}};

// a separation wrapped to its minimum image (vec.h:217-230)
__device__ __forceinline__ double ew_wrap(double d, double L) {
  return d - (fabs(d) > 0.5 * L ? copysign(L, d) : 0.0);
}
// the same up to its sign
__device__ __forceinline__ double ew_least(double d, double L) { return fmin(fabs(d), L - fabs(d)); }

// Real part (ewald.h:90-110) over every pair within the cutoff at its minimum
// image (the sum ewald.h's cell search aims at), and the self term
// (ewald.h:156-160).  Bound: FP64 VALU issue, the distances of all pairs and
// erfc and exp of those within the cutoff.  A wavefront a body, tiles of
// sources in LDS: the lanes test 64 sources at a time and list those within
// the cutoff, then evaluate the list, so that the long part runs on full
// wavefronts (at a cutoff of half the box, 52% of the pairs, every wavefront
// of a lane per body had one to evaluate); erfc and exp share one exponential
// and no branch.  24573 bodies: 3.2 -> 2.0 ms.  Two or four bodies a wavefront
// are no faster below 30000 bodies (registers), 4% at 36000.
constexpr int kEwTile = 1024;
__global__ __launch_bounds__(256) void ewald_real_kernel(EwBodies B, int n, double3 cyc, double alpha,
                                                         double cutoff2, Erfcx coef) {
  __shared__ double sx[kEwTile], sy[kEwTile], sz[kEwTile], sq[kEwTile];
  __shared__ unsigned short list[4][kEwTile];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int i = blockIdx.x * 4 + wave;
  const double alpha2 = alpha * alpha, a3 = alpha2 * alpha;
  const double3 xi = ew_pos(B, min(i, n - 1), cyc);
  double p = 0.0, gx = 0.0, gy = 0.0, gz = 0.0;
  for (int j0 = 0; j0 < n; j0 += kEwTile) {
    const int cnt = min(kEwTile, n - j0);
    __syncthreads();  // the last tile's readers
    for (int k = threadIdx.x; k < cnt; k += 256) {
      const double3 xj = ew_pos(B, j0 + k, cyc);
      sx[k] = xj.x;
      sy[k] = xj.y;
      sz[k] = xj.z;
      sq[k] = B.q[j0 + k];
    }
    if (threadIdx.x < 64 && cnt + threadIdx.x < kEwTile) sx[cnt + threadIdx.x] = NAN;  // never within the cutoff
    __syncthreads();
    int m = 0;  // sources listed
    for (int k0 = 0; k0 < cnt; k0 += 64) {
      const int k = k0 + lane;
      const double dx = ew_least(xi.x - sx[k], cyc.x), dy = ew_least(xi.y - sy[k], cyc.y),
                   dz = ew_least(xi.z - sz[k], cyc.z);
      const double R2 = dx * dx + dy * dy + dz * dz;
      const bool in = 0.0 < R2 && R2 < cutoff2;
      const unsigned long long b = __ballot(in);
      if (in) list[wave][m + __popcll(b & ((1ull << lane) - 1))] = (unsigned short)k;
      m += __popcll(b);
    }
    wave_lds_order();
    for (int e = lane; e < m; e += 64) {
      const int k = list[wave][e];
      const double dx = ew_wrap(xi.x - sx[k], cyc.x), dy = ew_wrap(xi.y - sy[k], cyc.y),
                   dz = ew_wrap(xi.z - sz[k], cyc.z), q = sq[k];
      const double s = (dx * dx + dy * dy + dz * dz) * alpha2;
      // 1/sqrt(s), 1/(x + K): the hardware estimates corrected to the last bit or two
      double y = __builtin_amdgcn_rsq(s);
      const double r = fma(-(s * y), y, 1.0);
      y = fma(y * r, fma(0.375, r, 0.5), y);
      const double x = s * y, xk = x + 3.75;
      double v = __builtin_amdgcn_rcp(xk);
      v = fma(v, fma(-xk, v, 1.0), v);
      v = fma(v, fma(-xk, v, 1.0), v);
      const double t = (x - 3.75) * v, t2 = t * t;
      double ge = coef.c[22], go = coef.c[23];
#pragma unroll
      for (int c = 20; c >= 0; c -= 2) {
        ge = fma(ge, t2, coef.c[c]);
        go = fma(go, t2, coef.c[c + 1]);
      }
      const double ex = exp(-s), ec = ex * fma(go, t, ge) * v * y;  // erfc(x) / x
      const double w = q * (M_2_SQRTPI * ex + ec) * (y * y) * a3;
      p += q * ec * alpha;
      gx -= dx * w;
      gy -= dy * w;
      gz -= dz * w;
    }
    wave_lds_order();  // the list's readers
  }
  for (int h = 32; h > 0; h >>= 1) {
    p += __shfl_xor(p, h);
    gx += __shfl_xor(gx, h);
    gy += __shfl_xor(gy, h);
    gz += __shfl_xor(gz, h);
  }
  if (i < n && lane == 0) ew_add(B, i, p - M_2_SQRTPI * B.q[i] * alpha, gx, gy, gz);
}

hipError_t launch_ewald(EwBodies B, int n, int ksize, int *kv, double2 *S, double3 cyc, double alpha,
                        double sigma, double cutoff, hipStream_t s) {
  if (n <= 0) return hipSuccess;
  const int nw = ewald_nwaves(ksize);
  const double3 scale = make_double3(2 * M_PI / cyc.x, 2 * M_PI / cyc.y, 2 * M_PI / cyc.z);
  const double coef = 2 / sigma / cyc.x / cyc.y / cyc.z, coef2 = 1 / (4 * alpha * alpha);
  if (nw > 0) {
    hipLaunchKernelGGL(ewald_waves_kernel, dim3(1), dim3(256), 0, s, ksize, kv);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(ewald_dft_kernel, dim3(nw), dim3(256), 0, s, B, n, kv, nw, cyc, scale, coef, coef2, S);
    e = hipGetLastError();
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(ewald_idft_kernel, dim3((n + kEwT - 1) / kEwT), dim3(256), 0, s, B, n, kv, S, nw, cyc, scale);
    e = hipGetLastError();
    if (e != hipSuccess) return e;
  }
  hipLaunchKernelGGL(ewald_real_kernel, dim3((n + 3) / 4), dim3(256), 0, s, B, n, cyc, alpha, cutoff * cutoff, kErfcx);
  return hipGetLastError();
}

// Per-device scratch of the allocation-free Ewald entry point: the structure
// factors S (double2 per wave) followed by the wave table (3 ints per wave)
// for ksize <= kEwaldScratchMaxK.  Host code never passes `scratch` itself to
// a kernel (on the host the name is not a device address): init_scratch()
// looks up each device's address of it once, with that device current.
constexpr size_t kEwaldScratchWaves = 70000;  // >= ewald_nwaves(kEwaldScratchMaxK) = 68,633
constexpr size_t kEwaldScratchBytes = kEwaldScratchWaves * (sizeof(double2) + 3 * sizeof(int));
static __device__ __align__(256) unsigned char scratch[kEwaldScratchBytes];
static void *g_scratch[kMaxDevices];

hipError_t init_scratch(int device) {
  if (device < 0 || device >= kMaxDevices) return hipErrorInvalidDevice;
  void *ptr = nullptr;
  hipError_t e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
  if (e != hipSuccess) return e;
  g_scratch[device] = ptr;
  return hipSuccess;
}

hipError_t launch_ewald_scratch(int device, EwBodies B, int n, int ksize, double3 cyc, double alpha, double sigma,
                                double cutoff, hipStream_t s) {
  if (device < 0 || device >= kMaxDevices || !g_scratch[device]) return hipErrorNotInitialized;
  if (ksize < 0 || ksize > kEwaldScratchMaxK || (size_t)ewald_nwaves(ksize) > kEwaldScratchWaves)
    return hipErrorInvalidValue;
  unsigned char *base = static_cast<unsigned char *>(g_scratch[device]);
  double2 *S = reinterpret_cast<double2 *>(base);
  int *kv = reinterpret_cast<int *>(base + kEwaldScratchWaves * sizeof(double2));
  return launch_ewald(B, n, ksize, kv, S, cyc, alpha, sigma, cutoff, s);
}

hipError_t launch_direct(DevBodies B, int n, const double *tx, const double *ty, const double *tz,
                         int nt, double *part, double *out, double eps2, int prange, double3 cyc, hipStream_t s) {
  if (nt <= 0) return hipSuccess;
  const int runs = direct_runs(n, nt);
  hipLaunchKernelGGL(direct_kernel, dim3((nt + 63) / 64, runs), dim3(256), 0, s, B, n, tx, ty, tz, nt,
                     direct_chunk(n, nt), runs > 1 ? part : out, eps2, prange, cyc);
  if (runs > 1)
    hipLaunchKernelGGL(direct_sum_kernel, dim3((unsigned)(((size_t)nt * 4 + 255) / 256)), dim3(256), 0, s, part, runs,
                       4 * nt, out);
  return hipGetLastError();
}

// ---------------------------------------------------------------- zero fill
// Clears n doubles with a kernel (the solve's phases use it instead of
// hipMemsetAsync so that a captured solve graph holds kernel nodes only).
__global__ __launch_bounds__(256) void zero_kernel(double *__restrict__ p, size_t n) {
  for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (size_t)gridDim.x * 256) p[i] = 0.0;
}

hipError_t launch_zero(double *p, size_t n, hipStream_t s) {
  if (n == 0) return hipSuccess;
  const size_t blocks = std::min<size_t>((n + 255) / 256, 8192);
  hipLaunchKernelGGL(zero_kernel, dim3((unsigned)blocks), dim3(256), 0, s, p, n);
  return hipGetLastError();
}

// a solve's four target arrays in one launch (four of them led a solve of 4096
// bodies by 12 of its 210 us)
__global__ __launch_bounds__(256) void zero_targets_kernel(double *__restrict__ p, double *__restrict__ x,
                                                           double *__restrict__ y, double *__restrict__ z, size_t n) {
  for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (size_t)gridDim.x * 256)
    p[i] = x[i] = y[i] = z[i] = 0.0;
}

hipError_t launch_zero_targets(double *p, double *x, double *y, double *z, size_t n, hipStream_t s) {
  if (n == 0) return hipSuccess;
  const size_t blocks = std::min<size_t>((n + 255) / 256, 8192);
  hipLaunchKernelGGL(zero_targets_kernel, dim3((unsigned)blocks), dim3(256), 0, s, p, x, y, z, n);
  return hipGetLastError();
}

// bodies into tree order (SoA): body i of the tree is input body perm[i]
__global__ void gather_bodies_kernel(int n, const int *__restrict__ perm, const double *__restrict__ xin,
                                     const double *__restrict__ qin, double *__restrict__ x,
                                     double *__restrict__ y, double *__restrict__ z, double *__restrict__ q) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const size_t b = (size_t)perm[i];
  x[i] = xin[3 * b];
  y[i] = xin[3 * b + 1];
  z[i] = xin[3 * b + 2];
  q[i] = qin[b];
}

hipError_t launch_gather_bodies(int n, const int *perm, const double *xin, const double *qin, double *x, double *y,
                                double *z, double *q, hipStream_t s) {
  if (n == 0) return hipSuccess;
  hipLaunchKernelGGL(gather_bodies_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, n, perm, xin, qin,
                     x, y, z, q);
  return hipGetLastError();
}

__global__ void gather_charges_kernel(int n, const int *__restrict__ perm, const double *__restrict__ qin,
                                      double *__restrict__ q) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i < n) q[i] = qin[perm[i]];
}
hipError_t launch_gather_charges(int n, const int *perm, const double *qin, double *q, hipStream_t s) {
  if (n > 0) hipLaunchKernelGGL(gather_charges_kernel, dim3((n - 1) / 256 + 1), dim3(256), 0, s, n, perm, qin, q);
  return hipGetLastError();
}

// targets in the caller's order and layout: the random 32-byte writes go to
// device memory, and the host only copies
__global__ void pack_targets_kernel(int n, const int *__restrict__ perm, DevBodies B, double2 *__restrict__ trg) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  const size_t o = perm ? perm[i] : i;
  trg[2 * o] = make_double2(B.pot[i], B.ax[i]);
  trg[2 * o + 1] = make_double2(B.ay[i], B.az[i]);
}
hipError_t launch_pack_targets(int n, const int *perm, DevBodies B, double *trg, hipStream_t s) {
  if (n > 0)
    hipLaunchKernelGGL(pack_targets_kernel, dim3((n - 1) / 256 + 1), dim3(256), 0, s, n, perm, B,
                       reinterpret_cast<double2 *>(trg));
  return hipGetLastError();
}

// every body's leaf: one thread per leaf over its bodies
__global__ void body_leaf_kernel(int nleaf, const int *__restrict__ leaves, const int *__restrict__ ibody,
                                 const int *__restrict__ nbody, int *__restrict__ body_leaf) {
  const int k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= nleaf) return;
  const int leaf = leaves[k], b0 = ibody[leaf], nb = nbody[leaf];
  for (int i = b0; i < b0 + nb; i++) body_leaf[i] = leaf;
}

hipError_t launch_body_leaf(int nleaf, const int *leaves, const int *ibody, const int *nbody, int *body_leaf,
                            hipStream_t s) {
  if (nleaf == 0) return hipSuccess;
  hipLaunchKernelGGL(body_leaf_kernel, dim3((unsigned)((nleaf + 255) / 256)), dim3(256), 0, s, nleaf, leaves,
                     ibody, nbody, body_leaf);
  return hipGetLastError();
}

// ---------------------------------------------------------------- dispatch
template <template <int> class F, typename... A>
static hipError_t dispatch(int P, A... a) {
  switch (P) {
#define FMM_CASE(p) \
  case p: return F<p>::run(a...);
    FMM_CASE(2) FMM_CASE(3) FMM_CASE(4) FMM_CASE(5) FMM_CASE(6) FMM_CASE(7) FMM_CASE(8)
    FMM_CASE(9) FMM_CASE(10) FMM_CASE(11) FMM_CASE(12) FMM_CASE(13) FMM_CASE(14)
    FMM_CASE(15) FMM_CASE(16) FMM_CASE(17) FMM_CASE(18) FMM_CASE(19) FMM_CASE(20)
#undef FMM_CASE
    default: return hipErrorInvalidValue;
  }
}

template <int P> struct RunP2M {
  template <int S> static void go(DevBodies B, DevCells C, const int *leaves, int nleaf, double2 *M, hipStream_t s) {
    constexpr int LW = P2MLanes<P, S>::LW;
    hipLaunchKernelGGL((p2m_kernel<P, S>), dim3((nleaf + LW - 1) / LW), dim3(64), 0, s, B, C, leaves, nleaf, M);
  }
  static hipError_t run(DevBodies B, DevCells C, const int *leaves, int nfew, int nmany, double2 *M, hipStream_t s) {
    constexpr int SM = 64 / ((P + 1) / 2);  // one leaf a wavefront
    // few leaves: a leaf's bodies over the whole wavefront, else over two groups
    // of lanes.  Upward pass with SM / 2 / 1 groups: 253 leaves, P = 8, 29 / 38 /
    // 46 us; 3229, P = 8, 52 / 55 / 66; 13003, P = 10, 101 / 101 / 116; 56095, P =
    // 10, 244 / 177 / 195; 797144, P = 12, 3032 / 1530 / 1487
    if (nfew > 0) go<SM>(B, C, leaves, nfew, M, s);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    if (nmany > 0) go<2>(B, C, leaves + nfew, nmany, M, s);
    return hipGetLastError();
  }
};
template <int P> struct RunM2M {
  static hipError_t run(DevCells C, const int *cells, int ncell, double2 *M, hipStream_t s) {
    if (ncell > 0) hipLaunchKernelGGL(m2m_kernel<P>, dim3(ncell), dim3(64), 0, s, C, cells, ncell, M);
    return hipGetLastError();
  }
};
template <int P> struct RunL2L {
  static hipError_t run(DevCells C, const int *cells, int ncell, double2 *L, hipStream_t s) {
    if (ncell > 0) hipLaunchKernelGGL(l2l_kernel<P>, dim3(ncell), dim3(64), 0, s, C, cells, ncell, L);
    return hipGetLastError();
  }
};
template <int P> struct RunL2P {
  static hipError_t run(DevBodies B, DevCells C, const int *body_leaf, int n, const double2 *L,
                        hipStream_t s) {
    const int grid = (n + 255) / 256;
    if (grid > 0) hipLaunchKernelGGL(l2p_kernel<P>, dim3(grid), dim3(256), 0, s, B, C, body_leaf, n, L);
    return hipGetLastError();
  }
};
template <int P> struct RunM2L {
  static hipError_t run(DevCells C, const int *targets, int ntarget, const int *ptr, const int *src,
                        double3 xper, const double2 *M, double2 *L, int accumulate, hipStream_t s) {
    if (ntarget > 0)
      hipLaunchKernelGGL(m2l_kernel<P>, dim3(ntarget), dim3(64), 0, s, C, targets, ntarget, ptr, src, xper,
                         M, L, accumulate);
    return hipGetLastError();
  }
};
template <int P> struct RunM2LMfma {
  static hipError_t run(const int4 *chunks, int nchunk, const double *gdx, const int *ptgt, const int *psrc,
                        const double2 *M, double2 *L, hipStream_t s) {
    if constexpr (MfmaCfg<P>::ok) {
      if (nchunk > 0)
        hipLaunchKernelGGL(m2l_mfma_kernel<P>, dim3(nchunk), dim3(MfmaCfg<P>::NTH), 0, s, chunks, gdx, ptgt,
                           psrc, M, reinterpret_cast<double *>(L));
      return hipGetLastError();
    } else {
      return hipErrorInvalidValue;
    }
  }
};

hipError_t launch_p2m(int P, DevBodies B, DevCells C, const int *leaves, int nfew, int nmany, double2 *M,
                      hipStream_t s) {
  return dispatch<RunP2M>(P, B, C, leaves, nfew, nmany, M, s);
}
hipError_t launch_m2m(int P, DevCells C, const int *cells, int ncell, double2 *M, hipStream_t s) {
  return dispatch<RunM2M>(P, C, cells, ncell, M, s);
}
hipError_t launch_l2l(int P, DevCells C, const int *cells, int ncell, double2 *L, hipStream_t s) {
  return dispatch<RunL2L>(P, C, cells, ncell, L, s);
}
hipError_t launch_l2p(int P, DevBodies B, DevCells C, const int *body_leaf, int n, const double2 *L,
                      hipStream_t s) {
  return dispatch<RunL2P>(P, B, C, body_leaf, n, L, s);
}
hipError_t launch_m2l(int P, DevCells C, const int *targets, int ntarget, const int *ptr, const int *src,
                      double3 xper, const double2 *M, double2 *L, int accumulate, hipStream_t s) {
  return dispatch<RunM2L>(P, C, targets, ntarget, ptr, src, xper, M, L, accumulate, s);
}
hipError_t launch_m2l_mfma(int P, const int4 *chunks, int nchunk, const double *gdx, const int *ptgt,
                           const int *psrc, const double2 *M, double2 *L, hipStream_t s) {
  return dispatch<RunM2LMfma>(P, chunks, nchunk, gdx, ptgt, psrc, M, L, s);
}
template <int P> struct RunMToF32 {
  static hipError_t run(const double2 *M, const double *R, int ncell, float2 *M32, hipStream_t s) {
    const int n = ncell * nterm(P);
    if (n > 0) hipLaunchKernelGGL(m_to_f32_kernel<P>, dim3((n + 255) / 256), dim3(256), 0, s, M, R, ncell, M32);
    return hipGetLastError();
  }
};
template <int P> struct RunM2LMfma32 {
  static hipError_t run(const int4 *chunks, int nchunk, const double *gdx, const double2 *gscale,
                        const int *ptgt, const int *psrc, const float2 *M32, double2 *L, hipStream_t s) {
    if constexpr (Mfma32Cfg<P>::ok) {
      if (nchunk > 0)
        hipLaunchKernelGGL(m2l_mfma32_kernel<P>, dim3(nchunk), dim3(Mfma32Cfg<P>::NTH), 0, s, chunks, gdx,
                           gscale, ptgt, psrc, M32, reinterpret_cast<double *>(L));
      return hipGetLastError();
    } else {
      return hipErrorInvalidValue;
    }
  }
};
template <int P> struct RunFarOps {
  static hipError_t run(int prange, double3 cyc, double2 *sums, double *T, double *S, hipStream_t s) {
    constexpr int NC = 2 * P - 1, PP = P * P, nt = (PP * PP + 255) / 256, ns = (PP * nterm(P) + 255) / 256;
    double2 *rsum = sums + (size_t)kFarBlocks * NC * NC;
    hipLaunchKernelGGL(far_sums_kernel<P>, dim3(kFarBlocks + (S ? 1 : 0)), dim3(256), 0, s, prange, cyc, sums, rsum);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(far_ops_kernel<P>, dim3(nt + (S ? ns : 0)), dim3(256), 0, s, sums, rsum, nt, T, S);
    return hipGetLastError();
  }
};
size_t far_sums_bytes(int P) { return sizeof(double2) * ((size_t)kFarBlocks * (2 * P - 1) * (2 * P - 1) + P * P); }
hipError_t launch_far_ops(int P, int prange, double3 cyc, void *sums, double *T, double *S, hipStream_t s) {
  if (prange < 1 || prange > kFarMaxRange) return hipErrorInvalidValue;
  return dispatch<RunFarOps>(P, prange, cyc, static_cast<double2 *>(sums), T, S, s);
}
template <int P> struct RunPeriodicFar {
  static hipError_t run(const double *F, const double2 *M, double2 *L, hipStream_t s) {
    hipLaunchKernelGGL(periodic_far_kernel<P>, dim3(1), dim3(256), 0, s, F, M, L);
    return hipGetLastError();
  }
};
hipError_t launch_matmul(const double *A, const double *B, double *C, int n, int acc, hipStream_t s) {
  hipLaunchKernelGGL(matmul_kernel, dim3((n * n + 255) / 256), dim3(256), 0, s, A, B, C, n, acc);
  return hipGetLastError();
}
hipError_t launch_periodic_far(int P, const double *F, const double2 *M, double2 *L, hipStream_t s) {
  return dispatch<RunPeriodicFar>(P, F, M, L, s);
}
hipError_t launch_m_to_f32(int P, const double2 *M, const double *R, int ncell, float2 *M32, hipStream_t s) {
  return dispatch<RunMToF32>(P, M, R, ncell, M32, s);
}
hipError_t launch_m2l_mfma32(int P, const int4 *chunks, int nchunk, const double *gdx, const double2 *gscale,
                             const int *ptgt, const int *psrc, const float2 *M32, double2 *L, hipStream_t s) {
  return dispatch<RunM2LMfma32>(P, chunks, nchunk, gdx, gscale, ptgt, psrc, M32, L, s);
}
// Wavefronts per leaf: four while the leaves fill the GPU's wavefront slots
// (about 15 of this kernel a CU) less than about three times over, as the
// longest lists then set the time.  Solve of 1 / 4 wavefronts a leaf, P = 8:
// 239 leaves 0.262 / 0.146 ms, 3037 0.705 / 0.550, 4118 (ragged) 2.05 / 0.74,
// 7229 0.685 / 0.665, 10047 0.854 / 0.826, 13003 1.080 / 1.093, 13248 0.687 /
// 0.759, 21300 1.611 / 1.697; a mixed-precision solve of 3037 0.526 / 0.420.
// The leaves counted are the system's own: see P2PCounts.
template <template <int, int> class F, typename... A> static hipError_t p2p_dispatch(P2PCounts n, A... a) {
  int first = 0;
  hipError_t e = hipSuccess;
  auto go = [&](auto run, int m) {
    if (m <= 0 || e != hipSuccess) return;
    run(first, m, a...);
    first += m;
    e = hipGetLastError();
  };
  go(F<4, 4>::run, n.wide_few);
  go(F<4, 1>::run, n.wide_many);
  go(F<1, 4>::run, n.few);
  go(F<1, 1>::run, n.many);
  return e;
}
template <int K, int W> struct RunP2P {
  static void run(int first, int n, DevBodies B, DevCells C, const int *targets, const int *ptr, const int *src,
                  double3 xper, double eps2, int mask_all, hipStream_t s) {
    hipLaunchKernelGGL((p2p_kernel<K, W>), dim3(n), dim3(64 * W), 0, s, B, C, targets + first, n, ptr, src, xper, eps2,
                       mask_all);
  }
};
template <int K, int W> struct RunP2P32 {
  static void run(int first, int n, DevBodies B, DevCells C, const int *targets, const int *ptr, const int *src,
                  double3 xper, double eps2, hipStream_t s) {
    hipLaunchKernelGGL((p2p32_kernel<K, W>), dim3(n), dim3(64 * W), 0, s, B, C, targets + first, n, ptr, src, xper,
                       eps2);
  }
};
hipError_t launch_p2p32(DevBodies B, DevCells C, const int *targets, P2PCounts n, const int *ptr,
                        const int *src, double3 xper, double eps2, int /*mask_all: every pair is masked*/,
                        hipStream_t s) {
  return p2p_dispatch<RunP2P32>(n, B, C, targets, ptr, src, xper, eps2, s);
}
hipError_t launch_p2p(DevBodies B, DevCells C, const int *targets, P2PCounts n, const int *ptr,
                      const int *src, double3 xper, double eps2, int mask_all, hipStream_t s) {
  return p2p_dispatch<RunP2P>(n, B, C, targets, ptr, src, xper, eps2, mask_all, s);
}

}  // namespace fmmdev
