// fmm_traverse.hip -- the octree and the interaction lists built on the device.
//
// The dual tree traversal of include/traversal.h:117-177 (dualTreeTraversal)
// and :90-114 (splitCell) run breadth first: every round takes the frontier
// of cell pairs, applies the multipole acceptance test and the split rules to
// each pair independently, appends accepted pairs to the M2L list, leaf pairs
// to the P2P list (or to M2L when the source leaf is empty) and the split
// pairs to the next frontier.  The rules are local to a pair, so the pairs
// found are exactly those of the recursive walk; only their order differs,
// and the lists are sorted by (target, source) at the end.  The acceptance
// test rounds exactly like the host walker's: no contraction into FMAs.
// device_visit_lists keeps the recursive walk's order instead: see there.
#include <hip/hip_runtime.h>
#include <hipcub/hipcub.hpp>

#include <algorithm>
#include <cstdint>
#include <cstring>
#include <deque>
#include <functional>
#include <map>
#include <mutex>
#include <utility>
#include <vector>

#include "fmm_device.hpp"

namespace fmmdev {

namespace {

struct TravCells {
  const double *X;  // 3 per cell
  const double *R;
  const int *nchild, *ichild, *nbody;
};

enum { kM2L = 0, kP2P = 1, kNext = 2 };

// classify pair (Ci, Cj): what it emits and how many frontier pairs it splits into
__device__ __forceinline__ void classify(const TravCells &t, int Ci, int Cj, double theta, double xp0, double xp1,
                                         double xp2, int nspawn, int &kind, int &na, int &nb, int &sa, int &sb) {
#pragma clang fp contract(off)
  const double dx = t.X[3 * (size_t)Ci] - t.X[3 * (size_t)Cj] - xp0;
  const double dy = t.X[3 * (size_t)Ci + 1] - t.X[3 * (size_t)Cj + 1] - xp1;
  const double dz = t.X[3 * (size_t)Ci + 2] - t.X[3 * (size_t)Cj + 2] - xp2;
  const double RT2 = (dx * dx + dy * dy + dz * dz) * theta * theta;
  const double Ri = t.R[Ci], Rj = t.R[Cj];
  const double Rs = Ri + Rj;
  const bool accept = RT2 > Rs * Rs * (1 - 1e-3);
  const int nci = t.nchild[Ci], ncj = t.nchild[Cj];
  // na x nb frontier pairs: a over Ci's children (or Ci itself), b over Cj's
  na = nb = 0;
  sa = Ci;
  sb = Cj;
  if (accept) {
    kind = kM2L;
  } else if (nci == 0 && ncj == 0) {
    kind = t.nbody[Cj] == 0 ? kM2L : kP2P;
  } else {
    kind = kNext;
    const int ci0 = t.ichild[Ci], cj0 = t.ichild[Cj];
    if (ncj == 0) {
      na = nci; sa = ci0; nb = 1;
    } else if (nci == 0) {
      na = 1; nb = ncj; sb = cj0;
    } else if (t.nbody[Ci] + t.nbody[Cj] >= nspawn || Ci == Cj) {
      na = nci; sa = ci0; nb = ncj; sb = cj0;
    } else if (Ri >= Rj) {
      na = nci; sa = ci0; nb = 1;
    } else {
      na = 1; nb = ncj; sb = cj0;
    }
  }
}

// count (write = false) or emit (write = true) one round; cnt[0..2]: M2L,
// P2P and next-frontier totals (running offsets while writing).  The count
// leaves what every pair becomes for the emission (0 M2L, 1 P2P, 1 + its
// children if split), which tests only the split ones again.  Bound by the
// blocks' additions to the three counters, some 3 ns each: a thread takes
// kTravPairs pairs and a block adds once for 2048 of them (the
// largest round of a 1M-body tree: 232 us counting and 237 emitting with an
// addition for 256 pairs, 51 and 92 now).
constexpr int kTravPairs = 8;
template <bool WRITE>
__global__ __launch_bounds__(256) void trav_round_kernel(const int2 *__restrict__ F, int nf, TravCells t, double theta,
                                                         double xp0, double xp1, double xp2, int nspawn,
                                                         unsigned char *__restrict__ kinds,
                                                         unsigned long long *__restrict__ cnt, int2 *__restrict__ m2l,
                                                         int2 *__restrict__ p2p, int2 *__restrict__ next) {
  const int i0 = blockIdx.x * (256 * kTravPairs) + threadIdx.x;
  int na, nb, sa, sb, cm = 0, cp = 0, cn = 0, kd[kTravPairs];
#pragma unroll
  for (int k = 0; k < kTravPairs; k++) {
    const int i = i0 + 256 * k;
    kd[k] = -1;
    if (i < nf) {
      if (WRITE) {
        kd[k] = kinds[i];
      } else {
        const int2 pr = F[i];
        classify(t, pr.x, pr.y, theta, xp0, xp1, xp2, nspawn, kd[k], na, nb, sa, sb);
        if (kd[k] == kNext) kd[k] = 1 + na * nb;
        kinds[i] = (unsigned char)kd[k];
      }
    }
    cm += kd[k] == kM2L;
    cp += kd[k] == kP2P;
    cn += kd[k] >= kNext ? kd[k] - 1 : 0;
  }
  // offsets within the wavefront (the three counts packed), then in the block
  const unsigned long long mine = (unsigned long long)cn << 32 | (unsigned)(cm | cp << 16);
  unsigned long long off = mine;
  const int lane = threadIdx.x & 63;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const unsigned long long y = __shfl_up(off, o, 64);
    if (lane >= o) off += y;
  }
  __shared__ unsigned long long wtot[4], bbase[3];
  const int wv = threadIdx.x >> 6;
  if (lane == 63) wtot[wv] = off;
  off -= mine;
  __syncthreads();
  if (threadIdx.x < 3) {
    const unsigned long long sum = wtot[0] + wtot[1] + wtot[2] + wtot[3];
    const unsigned long long v =
        threadIdx.x == 0 ? sum & 0xffff : threadIdx.x == 1 ? sum >> 16 & 0xffff : sum >> 32;
    bbase[threadIdx.x] = v ? atomicAdd(&cnt[threadIdx.x], v) : 0ull;
  }
  if (!WRITE) return;
  __syncthreads();
  for (int k = 0; k < wv; k++) off += wtot[k];  // the earlier wavefronts' counts
  int2 *om = m2l + bbase[0] + (off & 0xffff), *op = p2p + bbase[1] + (off >> 16 & 0xffff),
       *on = next + bbase[2] + (off >> 32);
#pragma unroll
  for (int k = 0; k < kTravPairs; k++) {
    if (kd[k] < 0) continue;
    const int2 pr = F[i0 + 256 * k];
    if (kd[k] == kM2L) {
      *om++ = pr;
    } else if (kd[k] == kP2P) {
      *op++ = pr;
    } else {
      int kind;
      classify(t, pr.x, pr.y, theta, xp0, xp1, xp2, nspawn, kind, na, nb, sa, sb);
      for (int a = 0; a < na; a++)
        for (int b = 0; b < nb; b++) *on++ = make_int2(sa + a, sb + b);
    }
  }
}

// sort keys (target, source)
__global__ void pair_keys_kernel(const int2 *__restrict__ pr, size_t n, int bits,
                                 unsigned long long *__restrict__ key) {
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const int2 p = pr[i];
  key[i] = ((unsigned long long)(unsigned)p.x << bits) | (unsigned)p.y;
}

// sorted keys below k
template <typename K>
__device__ __forceinline__ int keys_below(const K *__restrict__ key, int n, K k) {
  int lo = 0, hi = n;
  while (lo < hi) {
    const int m = (lo + hi) >> 1;
    if (key[m] < k)
      lo = m + 1;
    else
      hi = m;
  }
  return lo;
}

// ptr[c] = first pair of target c in the sorted keys, c = 0 .. ncell (counts
// by atomics while the keys are made took 86 us for 12M pairs in the order of
// their targets and 478 us otherwise; this takes 10)
__global__ void pair_ptr_kernel(int ncell, const unsigned long long *__restrict__ key, int n, int bits,
                                int *__restrict__ ptr) {
  const int c = blockIdx.x * blockDim.x + threadIdx.x;
  if (c <= ncell) ptr[c] = keys_below(key, n, (unsigned long long)c << bits);
}

__global__ void key_src_kernel(const unsigned long long *__restrict__ key, size_t n, int bits,
                               int *__restrict__ src) {
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) src[i] = (int)(key[i] & ((1ull << bits) - 1));
}

// grid-stride over the pairs, one atomic per block (256 threads)
__global__ void body_pairs_kernel(const int2 *__restrict__ pr, size_t n, const int *__restrict__ nbody,
                                  unsigned long long *__restrict__ out) {
  __shared__ unsigned long long part[4];
  unsigned long long v = 0;
  for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x)
    v += (unsigned long long)nbody[pr[i].x] * (unsigned long long)nbody[pr[i].y];
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = v;
  __syncthreads();
  if (threadIdx.x == 0) {
    const unsigned long long t = part[0] + part[1] + part[2] + part[3];
    if (t) atomicAdd(out, t);
  }
}

// device scratch from the plan builders' per-stream cache (plan_scratch_get)
struct Buf {
  hipStream_t s;
  void *p = nullptr;
  size_t bytes = 0;  // capacity
  explicit Buf(hipStream_t st) : s(st) {}
  Buf(const Buf &) = delete;
  ~Buf() {
    if (p) plan_scratch_put(p, bytes, s);
  }
  hipError_t need(size_t b) {
    if (b <= bytes) return hipSuccess;
    if (p) plan_scratch_put(p, bytes, s);
    p = nullptr;
    bytes = 0;
    return plan_scratch_get(&p, &bytes, b, s);
  }
  void swap(Buf &o) {
    std::swap(p, o.p);
    std::swap(bytes, o.bytes);
  }
  template <class T> T *as() const { return static_cast<T *>(p); }
};

#define TCHK(expr)                          \
  do {                                      \
    hipError_t e_ = (expr);                 \
    if (e_ != hipSuccess) return e_;        \
  } while (0)

// sorted CSR of a pair list on the device: ptr (ncell + 1) and the sources,
// copied to the host, or, with keep, left on the device in keep (src empty)
hipError_t pairs_to_csr(const int2 *pr, size_t n, int ncell, std::vector<int> &ptr, std::vector<int> &src,
                        hipStream_t s, DevArray *keep) {
  ptr.assign((size_t)ncell + 1, 0);
  src.clear();
  if (!keep) src.resize(n);
  Buf keys(s), keys2(s), dptr(s), tmp(s), out(s);
  if (n > 0) {
    TCHK(keys.need(8 * n));
    TCHK(keys2.need(8 * n));
    int bits = 1;  // the cell indices' bits: the sort takes a pass for every 8 of the two
    while ((1ll << bits) < (long long)ncell) bits++;
    pair_keys_kernel<<<(unsigned)((n + 255) / 256), 256, 0, s>>>(pr, n, bits, keys.as<unsigned long long>());
    TCHK(hipGetLastError());
    hipcub::DoubleBuffer<unsigned long long> db(keys.as<unsigned long long>(), keys2.as<unsigned long long>());
    size_t tb = 0;
    TCHK(hipcub::DeviceRadixSort::SortKeys(nullptr, tb, db, (int)n, 0, 2 * bits, s));
    TCHK(tmp.need(tb));
    TCHK(hipcub::DeviceRadixSort::SortKeys(tmp.p, tb, db, (int)n, 0, 2 * bits, s));
    int *dst;
    if (keep) {
      int dev = 0;
      TCHK(hipGetDevice(&dev));
      TCHK(keep->alloc(sizeof(int) * n, dev));
      dst = keep->as<int>();
    } else {
      TCHK(out.need(sizeof(int) * n));
      dst = out.as<int>();
    }
    key_src_kernel<<<(unsigned)((n + 255) / 256), 256, 0, s>>>(db.Current(), n, bits, dst);
    TCHK(hipGetLastError());
    if (!keep) TCHK(hipMemcpyAsync(src.data(), out.p, sizeof(int) * n, hipMemcpyDeviceToHost, s));
    TCHK(dptr.need(sizeof(int) * ((size_t)ncell + 1)));
    pair_ptr_kernel<<<(unsigned)(ncell / 256 + 1), 256, 0, s>>>(ncell, db.Current(), (int)n, bits, dptr.as<int>());
    TCHK(hipGetLastError());
    TCHK(hipMemcpyAsync(ptr.data(), dptr.p, sizeof(int) * ((size_t)ncell + 1), hipMemcpyDeviceToHost, s));
  } else if (keep) {
    keep->bytes = 0;
  }
  return hipStreamSynchronize(s);
}

// ---- the octree (include/build_tree.h:77-209, as fmm_host.cpp builds it) ----
//
// Each body's octant path to level 30 is computed with the host builder's
// centre arithmetic (octant o = (x > X) + 2 (y > Y) + 4 (z > Z), child centre
// X + r (+-1), r = R0 / 2^(level + 1)), and the bodies are sorted stably by
// it.  A node of level d is then a run of bodies sharing d octants; a body's
// leaf is its first run of at most ncrit bodies (or its level-30 run).  The
// runs come from lcp[j], the octants shared by sorted bodies j - 1 and j,
// with a sparse table of its minima: the run of level d around j ends at the
// first k > j with lcp[k] < d and starts at the last k <= j with lcp[k] < d.
// Cells are enumerated in pre-order (position, level); the cell numbering of
// nodes2cells (children contiguous, each child's descendants after all
// children, in child order) follows top-down from the subtree sizes.  Bodies
// keep their input order within a leaf, as the host's stable partitions do.

__global__ void tree_keys_kernel(int n, const double *__restrict__ x, double X0, double X1, double X2, double R0,
                                 unsigned long long *__restrict__ hi, unsigned long long *__restrict__ lo,
                                 int *__restrict__ idx) {
#pragma clang fp contract(off)
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const double b0 = x[3 * (size_t)i], b1 = x[3 * (size_t)i + 1], b2 = x[3 * (size_t)i + 2];
  double c0 = X0, c1 = X1, c2 = X2;
  unsigned long long h = 0, w = 0;
  for (int lev = 0; lev < 30; lev++) {
    const int o = (b0 > c0) + ((b1 > c1) << 1) + ((b2 > c2) << 2);
    if (lev < 21)
      h |= (unsigned long long)o << (3 * (20 - lev));
    else
      w |= (unsigned long long)o << (3 * (29 - lev));
    const double r = R0 / (1 << (lev + 1));
    c0 += r * ((o & 1) * 2 - 1);
    c1 += r * (((o >> 1) & 1) * 2 - 1);
    c2 += r * (((o >> 2) & 1) * 2 - 1);
  }
  hi[i] = h;
  lo[i] = w;
  idx[i] = i;
}

__global__ void gather_u64_kernel(int n, const unsigned long long *__restrict__ src, const int *__restrict__ idx,
                                  unsigned long long *__restrict__ dst) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) dst[i] = src[idx[i]];
}

// lcp[j] (j = 0..n): octants shared by sorted bodies j - 1 and j; -1 at both ends
__global__ void tree_lcp_kernel(int n, const unsigned long long *__restrict__ hi,
                                const unsigned long long *__restrict__ lo, signed char *__restrict__ lcp) {
  const int j = blockIdx.x * blockDim.x + threadIdx.x;
  if (j > n) return;
  int v = -1;
  if (j > 0 && j < n) {
    const unsigned long long a = hi[j] ^ hi[j - 1];
    if (a) {
      v = (__clzll(a) - 1) / 3;
    } else {
      const unsigned long long b = lo[j] ^ lo[j - 1];
      v = b ? 21 + (__clzll(b) - 37) / 3 : 30;
    }
  }
  lcp[j] = (signed char)v;
}

// table level lv: minimum of lcp over [p, p + 2^lv) (positions past n count as 127)
__global__ void tree_table_kernel(int m, const signed char *__restrict__ prev, int half,
                                  signed char *__restrict__ cur) {
  const int p = blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= m) return;
  const signed char a = prev[p];
  const signed char b = p + half < m ? prev[p + half] : (signed char)127;
  cur[p] = a < b ? a : b;
}

struct Runs {
  const signed char *tbl;  // (LG + 1) levels of m = n + 1 entries
  int m, LG;
  // first k > j with lcp[k] < d (at most n)
  __device__ int next(int j, int d) const {
    int pos = j + 1;
    if (tbl[pos] < d) return pos;
    for (int lv = LG; lv >= 0; lv--)
      if (pos + (1 << lv) <= m && tbl[(size_t)lv * m + pos] >= d) pos += 1 << lv;
    return pos;
  }
  // last k <= j with lcp[k] < d (at least 0)
  __device__ int prev(int j, int d) const {
    int pos = j;
    if (tbl[pos] < d) return pos;
    for (int lv = LG; lv >= 0; lv--)
      if (pos - (1 << lv) >= 0 && tbl[(size_t)lv * m + pos - (1 << lv)] >= d) pos -= 1 << lv;
    return pos - 1;
  }
};

// leaf level L[j] of every sorted body, the start of its leaf, and the number
// of cells starting at position j (levels lcp[j] + 1 .. L[j])
__global__ void tree_leaf_kernel(int n, Runs R, int ncrit, signed char *__restrict__ L, int *__restrict__ lstart,
                                 int *__restrict__ cnt) {
  const int j = blockIdx.x * blockDim.x + threadIdx.x;
  if (j > n) return;
  if (j == n) {
    cnt[j] = 0;
    return;
  }
  int lo = 0, hi = 30;  // the first level whose run holds <= ncrit bodies, else 30
  while (lo < hi) {
    const int d = (lo + hi) >> 1;
    if (R.next(j, d) - R.prev(j, d) <= ncrit)
      hi = d;
    else
      lo = d + 1;
  }
  L[j] = (signed char)lo;
  lstart[j] = R.prev(j, lo);
  const int c = lo - R.tbl[j];
  cnt[j] = c > 0 ? c : 0;
}

struct PreCells {
  int *pos, *level, *nbody, *nnode, *nchild;
};

// every cell (pre-order id cstart[j] + d - lcp[j] - 1 for level d at position j)
__global__ void tree_cells_kernel(int n, Runs R, const signed char *__restrict__ L, const int *__restrict__ cstart,
                                  PreCells C) {
  const int j = blockIdx.x * blockDim.x + threadIdx.x;
  if (j >= n) return;
  const int d0 = R.tbl[j] + 1, d1 = L[j];
  for (int d = d0; d <= d1; d++) {
    const int p = cstart[j] + (d - d0);
    const int e = R.next(j, d);
    int nc = 0;
    if (d < d1)
      for (int k = j; k < e; k = R.next(k, d + 1)) nc++;
    C.pos[p] = j;
    C.level[p] = d;
    C.nbody[p] = e - j;
    C.nnode[p] = cstart[e] - p;
    C.nchild[p] = nc;
  }
}

// nodes2cells numbering, one level: every cell of level d numbers its children
__global__ void tree_number_kernel(int ncell, int d, Runs R, const int *__restrict__ cstart, PreCells C,
                                   int *__restrict__ fidx, int *__restrict__ fbase, int *__restrict__ fpar) {
  const int p = blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= ncell || C.level[p] != d || C.nchild[p] == 0) return;
  const int j = C.pos[p], e = j + C.nbody[p], base = fbase[p], nc = C.nchild[p];
  int i = 0, off = base + nc;
  for (int k = j; k < e; k = R.next(k, d + 1), i++) {
    const int pc = cstart[k] + (d + 1) - (R.tbl[k] + 1);  // the child's pre-order id (level d + 1 at k)
    fidx[pc] = base + i;
    fbase[pc] = off;
    fpar[pc] = fidx[p];
    off += C.nnode[pc] - 1;
  }
}

// the cell arrays in nodes2cells order
__global__ void tree_scatter_kernel(int ncell, PreCells C, const int *__restrict__ fidx, const int *__restrict__ fbase,
                                    const int *__restrict__ fpar, const unsigned long long *__restrict__ hi,
                                    const unsigned long long *__restrict__ lo, double X0, double X1, double X2,
                                    double R0, int *__restrict__ iparent, int *__restrict__ ichild,
                                    int *__restrict__ nchild, int *__restrict__ ibody, int *__restrict__ nbody,
                                    int *__restrict__ level, double *__restrict__ X, double *__restrict__ Rc) {
#pragma clang fp contract(off)
  const int p = blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= ncell) return;
  const int f = fidx[p], j = C.pos[p], d = C.level[p];
  iparent[f] = fpar[p];
  nchild[f] = C.nchild[p];
  ichild[f] = C.nchild[p] ? fbase[p] : 0;
  ibody[f] = j;
  nbody[f] = C.nbody[p];
  level[f] = d;
  double c0 = X0, c1 = X1, c2 = X2;
  const unsigned long long h = hi[j], w = lo[j];
  for (int lev = 0; lev < d; lev++) {
    const int o = lev < 21 ? (int)((h >> (3 * (20 - lev))) & 7) : (int)((w >> (3 * (29 - lev))) & 7);
    const double r = R0 / (1 << (lev + 1));
    c0 += r * ((o & 1) * 2 - 1);
    c1 += r * (((o >> 1) & 1) * 2 - 1);
    c2 += r * (((o >> 2) & 1) * 2 - 1);
  }
  X[3 * (size_t)f] = c0;
  X[3 * (size_t)f + 1] = c1;
  X[3 * (size_t)f + 2] = c2;
  Rc[f] = R0 / (1 << d);
}

// the leaf start of every body, by input index
__global__ void tree_leafkey_kernel(int n, const int *__restrict__ idx, const int *__restrict__ lstart,
                                    unsigned *__restrict__ key, int *__restrict__ iota) {
  const int j = blockIdx.x * blockDim.x + threadIdx.x;
  if (j >= n) return;
  key[idx[j]] = (unsigned)lstart[j];
  iota[j] = j;
}
}  // namespace

hipError_t device_lists(int ncell, const double *X, const double *R, const int *nchild, const int *ichild,
                        const int *nbody, double theta, int nspawn, const double xper[3], int root_i, int root_j,
                        std::vector<int> &m2l_ptr, std::vector<int> &m2l_src, std::vector<int> &p2p_ptr,
                        std::vector<int> &p2p_src, int64_t &body_pairs, hipStream_t s, PlanArrays *keep) {
  if (keep) {
    keep->lists = false;
    keep->m2l_src.bytes = 0;
    keep->p2p_src.bytes = 0;
    TCHK(hipGetDevice(&keep->device));
  }
  m2l_ptr.assign((size_t)ncell + 1, 0);
  p2p_ptr.assign((size_t)ncell + 1, 0);
  m2l_src.clear();
  p2p_src.clear();
  body_pairs = 0;
  if (ncell == 0) return hipSuccess;
  Buf dX(s), dR(s), dnc(s), dic(s), dnb(s), cnt(s), F0(s), F1(s), M(s), Pp(s), bp(s), kinds(s);
  TCHK(dX.need(sizeof(double) * 3 * (size_t)ncell));
  TCHK(dR.need(sizeof(double) * (size_t)ncell));
  TCHK(dnc.need(sizeof(int) * (size_t)ncell));
  TCHK(dic.need(sizeof(int) * (size_t)ncell));
  TCHK(dnb.need(sizeof(int) * (size_t)ncell));
  TCHK(hipMemcpyAsync(dX.p, X, sizeof(double) * 3 * (size_t)ncell, hipMemcpyHostToDevice, s));
  TCHK(hipMemcpyAsync(dR.p, R, sizeof(double) * (size_t)ncell, hipMemcpyHostToDevice, s));
  TCHK(hipMemcpyAsync(dnc.p, nchild, sizeof(int) * (size_t)ncell, hipMemcpyHostToDevice, s));
  TCHK(hipMemcpyAsync(dic.p, ichild, sizeof(int) * (size_t)ncell, hipMemcpyHostToDevice, s));
  TCHK(hipMemcpyAsync(dnb.p, nbody, sizeof(int) * (size_t)ncell, hipMemcpyHostToDevice, s));
  TravCells t{dX.as<double>(), dR.as<double>(), dnc.as<int>(), dic.as<int>(), dnb.as<int>()};
  TCHK(cnt.need(sizeof(unsigned long long) * 3));
  const int2 root = make_int2(root_i, root_j);
  // first sizes from the tree (a cell has tens of M2L and P2P partners), grown by half again when short
  TCHK(F0.need(sizeof(int2) * 8 * (size_t)ncell));
  TCHK(M.need(sizeof(int2) * 64 * (size_t)ncell));
  TCHK(Pp.need(sizeof(int2) * 16 * (size_t)ncell));
  TCHK(hipMemcpyAsync(F0.p, &root, sizeof(int2), hipMemcpyHostToDevice, s));
  size_t nf = 1, nm = 0, np = 0;
  unsigned long long h[3];
  while (nf > 0) {
    if (nf > 0x7fffffff) return hipErrorInvalidValue;  // frontier beyond one launch's index range
    // count: the M2L, P2P and next-frontier pairs of this traversal round
    TCHK(hipMemsetAsync(cnt.p, 0, sizeof(h), s));
    const unsigned nb = (unsigned)((nf + 256 * kTravPairs - 1) / (256 * kTravPairs));
    TCHK(kinds.need(nf));
    trav_round_kernel<false><<<nb, 256, 0, s>>>(F0.as<int2>(), (int)nf, t, theta, xper[0], xper[1], xper[2], nspawn,
                                                kinds.as<unsigned char>(), cnt.as<unsigned long long>(), nullptr, nullptr, nullptr);
    TCHK(hipGetLastError());
    TCHK(hipMemcpyAsync(h, cnt.p, sizeof(h), hipMemcpyDeviceToHost, s));
    TCHK(hipStreamSynchronize(s));
    // room for the appended pairs (grown by half again when short), then emit
    auto grow = [&](Buf &b, size_t used, size_t add) -> hipError_t {
      const size_t want = sizeof(int2) * (used + add);
      if (want <= b.bytes) return hipSuccess;
      Buf nbuf(s);
      TCHK(nbuf.need(want + want / 2));
      if (used) TCHK(hipMemcpyAsync(nbuf.p, b.p, sizeof(int2) * used, hipMemcpyDeviceToDevice, s));
      b.swap(nbuf);  // the old buffer is released on the stream after the copy
      return hipSuccess;
    };
    TCHK(grow(M, nm, h[0]));
    TCHK(grow(Pp, np, h[1]));
    if (sizeof(int2) * h[2] > F1.bytes) TCHK(F1.need(sizeof(int2) * (h[2] + h[2] / 2)));
    const unsigned long long base[3] = {nm, np, 0};
    TCHK(hipMemcpyAsync(cnt.p, base, sizeof(base), hipMemcpyHostToDevice, s));
    trav_round_kernel<true><<<nb, 256, 0, s>>>(F0.as<int2>(), (int)nf, t, theta, xper[0], xper[1], xper[2], nspawn,
                                               kinds.as<unsigned char>(), cnt.as<unsigned long long>(), M.as<int2>(), Pp.as<int2>(),
                                               F1.as<int2>());
    TCHK(hipGetLastError());
    nm += h[0];
    np += h[1];
    nf = h[2];
    F0.swap(F1);
  }
  if (np > 0) {
    TCHK(bp.need(sizeof(unsigned long long)));
    TCHK(hipMemsetAsync(bp.p, 0, sizeof(unsigned long long), s));
    body_pairs_kernel<<<(unsigned)std::min<size_t>((np + 255) / 256, 2048), 256, 0, s>>>(
        Pp.as<int2>(), np, dnb.as<int>(), bp.as<unsigned long long>());
    TCHK(hipGetLastError());
    unsigned long long v = 0;
    TCHK(hipMemcpyAsync(&v, bp.p, sizeof v, hipMemcpyDeviceToHost, s));
    TCHK(hipStreamSynchronize(s));
    body_pairs = (int64_t)v;
  }
  TCHK(pairs_to_csr(M.as<int2>(), nm, ncell, m2l_ptr, m2l_src, s, keep ? &keep->m2l_src : nullptr));
  TCHK(pairs_to_csr(Pp.as<int2>(), np, ncell, p2p_ptr, p2p_src, s, keep ? &keep->p2p_src : nullptr));
  if (keep) keep->lists = true;
  return hipSuccess;
}

// ---- the lists in the recursive walk's order ----
//
// The rounds keep the visiting order: a round's pairs stand in it, and a
// split pair writes its children, in the order the recursion takes them, to
// the slots that an exclusive sum over the round gives it.  A pair's place
// among all emitted pairs is its parent's plus the emitted pairs below its
// earlier siblings: emitted pairs are counted bottom-up (a round's counts are
// differences of the next round's running sum), places handed out top-down,
// and one stable radix sort of the pairs so placed by (list, target) gives
// both lists, every target's sources in visiting order as the host's.
// Periodic images are 27 roots in image order, as the host walks them.
// Bound by latency: per round three launches and one size read back by the
// host, and as many launches again on the way back.
namespace {
struct VisitOrder {
  unsigned char o[8][8][64];  // [na - 1][nb - 1][k] = 8 a + b of the k-th child pair
};
// TraverseRange::operator() (traversal.h:196-229) over the children a, b
constexpr void visit_range(unsigned char *o, int &k, int ib, int ie, int jb, int je) {
  if (ie - ib == 1 || je - jb == 1) {
    for (int i = ib; i < ie; i++)
      for (int j = jb; j < je; j++) o[k++] = (unsigned char)(8 * i + j);
  } else {
    const int im = ib + (ie - ib) / 2, jm = jb + (je - jb) / 2;
    visit_range(o, k, ib, im, jb, jm);
    visit_range(o, k, im, ie, jm, je);
    visit_range(o, k, ib, im, jm, je);
    visit_range(o, k, im, ie, jb, jm);
  }
}
constexpr VisitOrder visit_order() {
  VisitOrder v{};
  for (int na = 1; na <= 8; na++)
    for (int nb = 1; nb <= 8; nb++) {
      int k = 0;
      visit_range(v.o[na - 1][nb - 1], k, 0, na, 0, nb);
    }
  return v;
}
__device__ constexpr VisitOrder kVisit = visit_order();

struct Shifts {
  double s[27][3];
};

__device__ __forceinline__ int visit_kind(const TravCells &t, int2 pr, double theta, const Shifts &sh, int nspawn,
                                          int &na, int &nb, int &sa, int &sb) {
  const int img = pr.y >> fmm::kImageShift;
  int kind;
  classify(t, pr.x, pr.y & fmm::kCellMask, theta, sh.s[img][0], sh.s[img][1], sh.s[img][2], nspawn, kind, na, nb, sa,
           sb);
  return kind;
}

// kind[i] and the number of children cn[i] of every pair of a round; cn[nf] = 0
__global__ __launch_bounds__(256) void visit_count_kernel(const int2 *__restrict__ F, int nf, TravCells t, double theta,
                                                          Shifts sh, int nspawn, unsigned char *__restrict__ kind,
                                                          int *__restrict__ cn) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i > nf) return;
  int na = 0, nb = 0, sa, sb;
  if (i < nf) kind[i] = (unsigned char)visit_kind(t, F[i], theta, sh, nspawn, na, nb, sa, sb);
  cn[i] = na * nb;
}

// *out += cn[0] + ... + cn[n - 1], one atomic per block
__global__ __launch_bounds__(256) void children_total_kernel(const int *__restrict__ cn, int n,
                                                             unsigned long long *__restrict__ out) {
  __shared__ unsigned long long part[4];
  unsigned long long v = 0;
  for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < (size_t)n; i += (size_t)gridDim.x * 256) v += cn[i];
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = v;
  __syncthreads();
  if (threadIdx.x == 0) atomicAdd(out, part[0] + part[1] + part[2] + part[3]);
}

// the next round: the children of every split pair from slot co[i] on.  A
// wavefront takes 64 pairs and its lanes their children, each finding its pair
// by a search in the pairs' slots (pair by pair, a lane a child, the rounds of
// a 62k-body tree took 16 us each, most of it for pairs of a few children;
// 8 us now)
__global__ __launch_bounds__(256) void visit_expand_kernel(const int2 *__restrict__ F, int nf, TravCells t,
                                                           double theta, Shifts sh, int nspawn,
                                                           const unsigned char *__restrict__ kind,
                                                           const int *__restrict__ co, int2 *__restrict__ next,
                                                           int *__restrict__ par) {
  __shared__ int soff[4][65], sa0[4][64], sb0[4][64], snn[4][64];
  const int w = threadIdx.x >> 6, lane = threadIdx.x & 63, i0 = (blockIdx.x * 4 + w) * 64, i = i0 + lane;
  int *off = soff[w];
  off[lane] = co[min(i, nf)];
  if (lane == 63) off[64] = co[min(i0 + 64, nf)];
  if (i < nf && kind[i] == kNext) {
    int na, nb, sa, sb;
    visit_kind(t, F[i], theta, sh, nspawn, na, nb, sa, sb);
    sa0[w][lane] = sa;
    sb0[w][lane] = sb | (F[i].y & ~fmm::kCellMask);
    snn[w][lane] = 8 * (na - 1) + nb - 1;
  }
  __syncthreads();
  for (int c = off[0] + lane; c < off[64]; c += 64) {
    int l = 0;  // the last pair with off[l] <= c: the one that has child c
#pragma unroll
    for (int d = 32; d > 0; d >>= 1)
      if (off[l + d] <= c) l += d;
    const int k = (&kVisit.o[0][0][0])[64 * snn[w][l] + c - off[l]];
    next[c] = make_int2(sa0[w][l] + (k >> 3), sb0[w][l] + (k & 7));
    par[c] = i0 + l;
  }
}

// emitted pairs at or below every pair of a round; sub[nf] = 0
__global__ __launch_bounds__(256) void visit_below_kernel(int nf, const unsigned char *__restrict__ kind,
                                                          const int *__restrict__ co, const int *__restrict__ nsum,
                                                          int *__restrict__ sub) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i > nf) return;
  sub[i] = i == nf ? 0 : kind[i] == kNext ? nsum[co[i + 1]] - nsum[co[i]] : 1;
}

// the places of a round's pairs among the emitted ones, the emitted ones
// written there, and the body pairs of the P2P ones added up
__global__ __launch_bounds__(256) void visit_place_kernel(const int2 *__restrict__ F, int nf,
                                                          const unsigned char *__restrict__ kind,
                                                          const int *__restrict__ sum, const int *__restrict__ par,
                                                          const int *__restrict__ pplace, const int *__restrict__ pco,
                                                          const int *__restrict__ nbody, int tbits,
                                                          int *__restrict__ place, unsigned *__restrict__ key,
                                                          int *__restrict__ src, unsigned long long *__restrict__ bp) {
  __shared__ unsigned long long part[4];
  unsigned long long v = 0;
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i < nf) {
    int at = sum[i];
    if (par) {
      const int p = par[i];
      at += pplace[p] - sum[pco[p]];
    }
    place[i] = at;
    const int kd = kind[i];
    if (kd != kNext) {
      const int2 pr = F[i];
      key[at] = (unsigned)kd << tbits | (unsigned)pr.x;
      src[at] = pr.y;
      if (kd == kP2P) v = (unsigned long long)nbody[pr.x] * (unsigned long long)nbody[pr.y & fmm::kCellMask];
    }
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = v;
  __syncthreads();
  if (threadIdx.x == 0) {
    const unsigned long long tot = part[0] + part[1] + part[2] + part[3];
    if (tot) atomicAdd(bp, tot);
  }
}

// ptr[c] of both lists (M2L: [0, ncell], P2P behind it) in the sorted keys
__global__ void visit_ptr_kernel(int ncell, int n, const unsigned *__restrict__ key, int tbits, int *__restrict__ ptr) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= 2 * (ncell + 1)) return;
  const bool p2p = i > ncell;
  const unsigned list = (unsigned)kP2P << tbits;
  ptr[i] = p2p ? keys_below(key, n, list + (unsigned)(i - ncell - 1)) - keys_below(key, n, list)
               : keys_below(key, n, (unsigned)i);
}
}  // namespace

hipError_t device_visit_lists(const fmm::Tree &t, double theta, int nspawn, int images, const double *cycle,
                              fmm::Lists &L, const std::function<int *(bool p2p, int64_t n)> &dst, bool &done,
                              hipStream_t s) {
  done = false;
  const int nc = t.ncell;
  if (nc == 0) return hipSuccess;
  // the cells in one copy: X, R, then nchild, ichild, nbody
  std::vector<double> h((size_t)nc * 4 + ((size_t)nc * 3 + 1) / 2);
  std::memcpy(h.data(), t.X.data(), sizeof(double) * 3 * (size_t)nc);
  std::memcpy(h.data() + 3 * (size_t)nc, t.R.data(), sizeof(double) * (size_t)nc);
  int *hi = reinterpret_cast<int *>(h.data() + 4 * (size_t)nc);
  for (int c = 0; c < nc; c++) {
    if (t.nchild[c] > 8) return hipSuccess;
    hi[c] = t.nchild[c];
    hi[nc + c] = t.ichild[c];
    hi[2 * (size_t)nc + c] = t.nbody[c];
  }
  Buf dcell(s), tmp(s), dbp(s), key(s), key2(s), src(s), src2(s), dptr(s);
  TCHK(dcell.need(8 * h.size()));
  TCHK(hipMemcpyAsync(dcell.p, h.data(), 8 * h.size(), hipMemcpyHostToDevice, s));
  const double *dX = dcell.as<double>();
  const int *di = reinterpret_cast<const int *>(dX + 4 * (size_t)nc);
  const TravCells cells{dX, dX + 3 * (size_t)nc, di, di + nc, di + 2 * (size_t)nc};
  Shifts sh{};
  const int nimg = images > 0 ? 27 : 1;
  for (int m = 0; images > 0 && m < nimg; m++) fmm::image_shift(m, cycle, sh.s[m]);
  struct Round {
    Buf F, par, kind, co, sum, place;
    int n = 0;
    explicit Round(hipStream_t st) : F(st), par(st), kind(st), co(st), sum(st), place(st) {}
  };
  std::deque<Round> R;
  auto scan = [&](const Buf &in, Buf &out, int n) -> hipError_t {
    size_t tb = 0;
    TCHK(hipcub::DeviceScan::ExclusiveSum(nullptr, tb, in.as<int>(), out.as<int>(), n, s));
    TCHK(tmp.need(tb));
    return hipcub::DeviceScan::ExclusiveSum(tmp.p, tb, in.as<int>(), out.as<int>(), n, s);
  };
  int2 root[27];
  for (int m = 0; m < nimg; m++) root[m] = make_int2(0, m << fmm::kImageShift);
  R.emplace_back(s);
  R.back().n = nimg;
  TCHK(R.back().F.need(sizeof(int2) * nimg));
  TCHK(hipMemcpyAsync(R.back().F.p, root, sizeof(int2) * nimg, hipMemcpyHostToDevice, s));
  Buf cn(s);
  int64_t total = nimg;  // pairs of all rounds
  for (;;) {
    Round &r = R.back();
    const size_t n = (size_t)r.n;
    const unsigned nb = (unsigned)(n / 256 + 1);
    TCHK(r.kind.need(n));
    TCHK(cn.need(4 * (n + 1)));
    TCHK(r.co.need(4 * (n + 1)));
    visit_count_kernel<<<nb, 256, 0, s>>>(r.F.as<int2>(), r.n, cells, theta, sh, nspawn, r.kind.as<unsigned char>(),
                                          cn.as<int>());
    TCHK(hipGetLastError());
    TCHK(scan(cn, r.co, r.n + 1));
    int n32 = 0;
    int64_t nn = 0;
    if (fmm::visit_sum_wraps(r.n)) {  // the sum in 32 bits may have wrapped: added up in 64
      TCHK(dbp.need(8));
      TCHK(hipMemsetAsync(dbp.p, 0, 8, s));
      children_total_kernel<<<(unsigned)std::min<size_t>(nb, 2048), 256, 0, s>>>(cn.as<int>(), r.n,
                                                                              dbp.as<unsigned long long>());
      TCHK(hipGetLastError());
      TCHK(hipMemcpyAsync(&nn, dbp.p, 8, hipMemcpyDeviceToHost, s));
      TCHK(hipStreamSynchronize(s));
    } else {
      TCHK(hipMemcpyAsync(&n32, r.co.as<int>() + n, 4, hipMemcpyDeviceToHost, s));
      TCHK(hipStreamSynchronize(s));
      nn = n32;
    }
    if (!fmm::visit_fits(total, nn)) return hipSuccess;  // beyond the 32-bit sums: the host walks this tree
    if (nn == 0) break;
    R.emplace_back(s);
    Round &q = R.back();
    q.n = (int)nn;
    total += nn;
    TCHK(q.F.need(sizeof(int2) * (size_t)nn));
    TCHK(q.par.need(4 * (size_t)nn));
    visit_expand_kernel<<<(unsigned)((n + 255) / 256), 256, 0, s>>>(
        r.F.as<int2>(), r.n, cells, theta, sh, nspawn, r.kind.as<unsigned char>(), r.co.as<int>(), q.F.as<int2>(),
        q.par.as<int>());
    TCHK(hipGetLastError());
  }
  // emitted pairs below, bottom-up (cn: this round's counts)
  for (size_t k = R.size(); k-- > 0;) {
    Round &r = R[k];
    TCHK(cn.need(4 * ((size_t)r.n + 1)));
    TCHK(r.sum.need(4 * ((size_t)r.n + 1)));
    visit_below_kernel<<<(unsigned)(r.n / 256 + 1), 256, 0, s>>>(
        r.n, r.kind.as<unsigned char>(), r.co.as<int>(), k + 1 < R.size() ? R[k + 1].sum.as<int>() : nullptr,
        cn.as<int>());
    TCHK(hipGetLastError());
    TCHK(scan(cn, r.sum, r.n + 1));
  }
  int ne = 0;  // emitted pairs
  TCHK(hipMemcpyAsync(&ne, R[0].sum.as<int>() + R[0].n, 4, hipMemcpyDeviceToHost, s));
  TCHK(dbp.need(8));
  TCHK(hipMemsetAsync(dbp.p, 0, 8, s));
  TCHK(hipStreamSynchronize(s));
  int tbits = 1;
  while ((1ll << tbits) < nc) tbits++;
  for (Buf *b : {&key, &key2, &src, &src2}) TCHK(b->need(4 * (size_t)ne));
  for (size_t k = 0; k < R.size(); k++) {
    Round &r = R[k];
    TCHK(r.place.need(4 * (size_t)r.n));
    visit_place_kernel<<<(unsigned)((r.n + 255) / 256), 256, 0, s>>>(
        r.F.as<int2>(), r.n, r.kind.as<unsigned char>(), r.sum.as<int>(), k ? r.par.as<int>() : nullptr,
        k ? R[k - 1].place.as<int>() : nullptr, k ? R[k - 1].co.as<int>() : nullptr, cells.nbody, tbits,
        r.place.as<int>(), key.as<unsigned>(), src.as<int>(), dbp.as<unsigned long long>());
    TCHK(hipGetLastError());
  }
  size_t tb = 0;
  TCHK(hipcub::DeviceRadixSort::SortPairs(nullptr, tb, key.as<unsigned>(), key2.as<unsigned>(), src.as<int>(),
                                          src2.as<int>(), ne, 0, tbits + 1, s));
  TCHK(tmp.need(tb));
  TCHK(hipcub::DeviceRadixSort::SortPairs(tmp.p, tb, key.as<unsigned>(), key2.as<unsigned>(), src.as<int>(),
                                          src2.as<int>(), ne, 0, tbits + 1, s));
  const size_t np = 2 * ((size_t)nc + 1);
  TCHK(dptr.need(4 * np));
  visit_ptr_kernel<<<(unsigned)((np + 255) / 256), 256, 0, s>>>(nc, ne, key2.as<unsigned>(), tbits, dptr.as<int>());
  TCHK(hipGetLastError());
  std::vector<int> ptr(np);
  unsigned long long bp = 0;
  TCHK(hipMemcpyAsync(ptr.data(), dptr.p, 4 * np, hipMemcpyDeviceToHost, s));
  TCHK(hipMemcpyAsync(&bp, dbp.p, 8, hipMemcpyDeviceToHost, s));
  TCHK(hipStreamSynchronize(s));
  L = fmm::Lists();
  L.m2l_ptr.assign(ptr.begin(), ptr.begin() + nc + 1);
  L.p2p_ptr.assign(ptr.begin() + nc + 1, ptr.end());
  L.nm2l = L.m2l_ptr[nc];
  L.np2p = L.p2p_ptr[nc];
  L.p2p_body_pairs = (int64_t)bp;
  for (int c = 0; c < nc; c++) {
    if (L.m2l_ptr[c + 1] > L.m2l_ptr[c]) L.m2l_targets.push_back(c);
    if (L.p2p_ptr[c + 1] > L.p2p_ptr[c]) L.p2p_targets.push_back(c);
  }
  for (bool p2p : {false, true}) {
    const int64_t n = p2p ? L.np2p : L.nm2l;
    int *d = dst(p2p, n);
    if (!d) return hipErrorOutOfMemory;
    if (n)
      TCHK(hipMemcpyAsync(d, src2.as<int>() + (p2p ? L.nm2l : 0), 4 * (size_t)n, hipMemcpyDeviceToDevice, s));
  }
  done = true;
  return hipSuccess;
}

namespace {
struct ScratchCache {
  std::multimap<size_t, void *> blocks;  // capacity -> block
  size_t total = 0;
};
std::mutex g_scratch_mu;
std::map<hipStream_t, ScratchCache> g_scratch;
constexpr size_t kScratchKeep = (size_t)12 << 30;
}  // namespace

hipError_t plan_scratch_get(void **p, size_t *cap, size_t bytes, hipStream_t s, size_t spare) {
  *p = nullptr;
  *cap = 0;
  if (bytes == 0) bytes = 1;
  {
    std::lock_guard<std::mutex> lk(g_scratch_mu);
    auto f = g_scratch.find(s);
    if (f != g_scratch.end()) {
      auto it = f->second.blocks.lower_bound(bytes);
      if (it != f->second.blocks.end() && it->first <= 2 * bytes + ((size_t)1 << 20)) {
        *p = it->second;
        *cap = it->first;
        f->second.total -= it->first;
        f->second.blocks.erase(it);
        return hipSuccess;
      }
    }
  }
  hipError_t e = device_alloc(p, bytes + spare);
  if (e == hipErrorOutOfMemory && spare > 0) e = device_alloc(p, bytes), spare = 0;
  if (e != hipSuccess) return e;
  *cap = bytes + spare;
  return hipSuccess;
}

void plan_scratch_put(void *p, size_t cap, hipStream_t s) {
  if (!p) return;
  {
    std::lock_guard<std::mutex> lk(g_scratch_mu);
    ScratchCache &c = g_scratch[s];
    if (c.total + cap <= kScratchKeep) {
      c.blocks.emplace(cap, p);
      c.total += cap;
      return;
    }
  }
  (void)hipFree(p);  // waits for the device's work, the stream's included
}

void plan_scratch_release(hipStream_t s) {
  ScratchCache c;
  {
    std::lock_guard<std::mutex> lk(g_scratch_mu);
    auto f = g_scratch.find(s);
    if (f == g_scratch.end()) return;
    c = std::move(f->second);
    g_scratch.erase(f);
  }
  if (c.blocks.empty()) return;
  (void)hipStreamSynchronize(s);
  for (auto &b : c.blocks) (void)hipFree(b.second);
}

// every stream's idle blocks
static bool plan_scratch_release_all() {
  std::vector<void *> idle;
  {
    std::lock_guard<std::mutex> lk(g_scratch_mu);
    for (auto &c : g_scratch) {
      for (auto &b : c.second.blocks) idle.push_back(b.second);
      c.second = ScratchCache();
    }
  }
  for (void *p : idle) (void)hipFree(p);  // waits for the device's work
  return !idle.empty();
}

hipError_t device_alloc(void **p, size_t bytes) {
  hipError_t e = hipMalloc(p, bytes);
  if (e == hipErrorOutOfMemory) {
    (void)hipGetLastError();
    if (plan_scratch_release_all()) e = hipMalloc(p, bytes);
    if (e == hipErrorOutOfMemory) (void)hipGetLastError();
  }
  if (e != hipSuccess) *p = nullptr;
  return e;
}

hipError_t DevArray::alloc(size_t b, int dev) {
  if (p && device == dev && cap >= b) {
    bytes = b;
    return hipSuccess;
  }
  // a context's array that was too small grows by a quarter more, as its other
  // buffers do, where there is room
  size_t want = cap ? b + b / 4 : b;
  reset();
  if (b == 0) return hipSuccess;
  if (pool) {
    const hipError_t e = plan_scratch_get(&p, &cap, b, pool, b / 4);
    if (e != hipSuccess) return e;
    bytes = b;
    device = dev;
    return hipSuccess;
  }
  hipError_t e = device_alloc(&p, want);
  if (e == hipErrorOutOfMemory && want > b) e = device_alloc(&p, want = b);
  if (e != hipSuccess) return e;
  bytes = b;
  cap = want;
  device = dev;
  return hipSuccess;
}

void DevArray::reset() {
  if (p && pool) {
    plan_scratch_put(p, cap, pool);
  } else if (p) {
    int cur = -1;
    const bool same = hipGetDevice(&cur) == hipSuccess && cur == device;
    if (!same) (void)hipSetDevice(device);
    (void)hipFree(p);
    if (!same && cur >= 0) (void)hipSetDevice(cur);
  }
  p = nullptr;
  bytes = cap = 0;
  device = -1;
}

hipError_t fetch_lists(const PlanArrays &d, fmm::Lists &L, hipStream_t s) {
  if (!d.lists) return hipSuccess;
  if ((int64_t)L.m2l_src.size() != L.nm2l) {
    L.m2l_src.resize(L.nm2l);
    if (L.nm2l) TCHK(hipMemcpyAsync(L.m2l_src.data(), d.m2l_src.p, 4 * (size_t)L.nm2l, hipMemcpyDeviceToHost, s));
  }
  if ((int64_t)L.p2p_src.size() != L.np2p) {
    L.p2p_src.resize(L.np2p);
    if (L.np2p) TCHK(hipMemcpyAsync(L.p2p_src.data(), d.p2p_src.p, 4 * (size_t)L.np2p, hipMemcpyDeviceToHost, s));
  }
  return hipStreamSynchronize(s);
}

hipError_t fetch_tiles(const PlanArrays &d, fmm::M2LTiles &T, hipStream_t s) {
  if (!d.tiles) return hipSuccess;
  const size_t np = d.t_src.bytes / 4;
  if (T.src.size() != np) {
    T.slice.resize(4 * (size_t)d.nslice);
    T.src.resize(np);
    T.lt.resize(np);
    if (d.nslice) TCHK(hipMemcpyAsync(T.slice.data(), d.t_slice.p, 16 * (size_t)d.nslice, hipMemcpyDeviceToHost, s));
    if (np) {
      TCHK(hipMemcpyAsync(T.src.data(), d.t_src.p, 4 * np, hipMemcpyDeviceToHost, s));
      TCHK(hipMemcpyAsync(T.lt.data(), d.t_lt.p, 2 * np, hipMemcpyDeviceToHost, s));
    }
  }
  return hipStreamSynchronize(s);
}

hipError_t device_tree(int n, const double *x, int ncrit, const double X0[3], double R0, std::vector<int> &perm,
                       std::vector<int> &iparent, std::vector<int> &ichild, std::vector<int> &nchild,
                       std::vector<int> &ibody, std::vector<int> &nbody, std::vector<int> &level,
                       std::vector<double> &X, std::vector<double> &R, hipStream_t s, const double *dx_in) {
  perm.resize(n);
  if (n == 0) {
    for (auto *v : {&iparent, &ichild, &nchild, &ibody, &nbody, &level}) v->clear();
    X.clear();
    R.clear();
    return hipSuccess;
  }
  const unsigned nb = (unsigned)((n + 255) / 256);
  using u64 = unsigned long long;
  Buf dx(s), kh(s), kl(s), ka(s), kb(s), idx(s), idx2(s), tmp(s);
  const double *xd = dx_in;
  if (!xd) {
    TCHK(dx.need(sizeof(double) * 3 * (size_t)n));
    TCHK(hipMemcpyAsync(dx.p, x, sizeof(double) * 3 * (size_t)n, hipMemcpyHostToDevice, s));
    xd = dx.as<double>();
  }
  for (Buf *b : {&kh, &kl, &ka, &kb}) TCHK(b->need(8 * (size_t)n));
  TCHK(idx.need(4 * (size_t)n));
  TCHK(idx2.need(4 * (size_t)n));
  tree_keys_kernel<<<nb, 256, 0, s>>>(n, xd, X0[0], X0[1], X0[2], R0, kh.as<u64>(), kl.as<u64>(),
                                      idx.as<int>());
  TCHK(hipGetLastError());
  // stable sort by the path, least significant part first: by levels 21-29
  // (kl), then by levels 0-20 (kh, gathered into the first sort's order)
  size_t tb = 0, tb2 = 0;
  TCHK(hipcub::DeviceRadixSort::SortPairs(nullptr, tb, kl.as<u64>(), ka.as<u64>(), idx.as<int>(), idx2.as<int>(), n,
                                          0, 27, s));
  TCHK(hipcub::DeviceRadixSort::SortPairs(nullptr, tb2, ka.as<u64>(), kb.as<u64>(), idx2.as<int>(), idx.as<int>(), n,
                                          0, 63, s));
  TCHK(tmp.need(std::max(tb, tb2)));
  TCHK(hipcub::DeviceRadixSort::SortPairs(tmp.p, tb, kl.as<u64>(), ka.as<u64>(), idx.as<int>(), idx2.as<int>(), n,
                                          0, 27, s));
  gather_u64_kernel<<<nb, 256, 0, s>>>(n, kh.as<u64>(), idx2.as<int>(), ka.as<u64>());
  TCHK(hipGetLastError());
  TCHK(hipcub::DeviceRadixSort::SortPairs(tmp.p, tb2, ka.as<u64>(), kb.as<u64>(), idx2.as<int>(), idx.as<int>(), n,
                                          0, 63, s));
  gather_u64_kernel<<<nb, 256, 0, s>>>(n, kl.as<u64>(), idx.as<int>(), ka.as<u64>());
  TCHK(hipGetLastError());
  // sorted paths: levels 0-20 in kb, 21-29 in ka; idx: input index of every sorted body
  const u64 *hiS = kb.as<u64>(), *loS = ka.as<u64>();
  const int m = n + 1;
  int LG = 0;
  while ((1 << (LG + 1)) <= m) LG++;
  Buf tbl(s), Lv(s), lst(s), cnt(s), cst(s);
  TCHK(tbl.need((size_t)(LG + 1) * m));
  tree_lcp_kernel<<<(unsigned)((m + 255) / 256), 256, 0, s>>>(n, hiS, loS, tbl.as<signed char>());
  TCHK(hipGetLastError());
  for (int lv = 1; lv <= LG; lv++) {
    tree_table_kernel<<<(unsigned)((m + 255) / 256), 256, 0, s>>>(
        m, tbl.as<signed char>() + (size_t)(lv - 1) * m, 1 << (lv - 1), tbl.as<signed char>() + (size_t)lv * m);
    TCHK(hipGetLastError());
  }
  Runs RR{tbl.as<signed char>(), m, LG};
  TCHK(Lv.need(m));
  TCHK(lst.need(4 * (size_t)m));
  TCHK(cnt.need(4 * (size_t)m));
  TCHK(cst.need(4 * (size_t)m));
  tree_leaf_kernel<<<(unsigned)((m + 255) / 256), 256, 0, s>>>(n, RR, ncrit, Lv.as<signed char>(), lst.as<int>(),
                                                               cnt.as<int>());
  TCHK(hipGetLastError());
  size_t ts = 0;
  TCHK(hipcub::DeviceScan::ExclusiveSum(nullptr, ts, cnt.as<int>(), cst.as<int>(), m, s));
  Buf tmp2(s);
  TCHK(tmp2.need(ts));
  TCHK(hipcub::DeviceScan::ExclusiveSum(tmp2.p, ts, cnt.as<int>(), cst.as<int>(), m, s));
  int ncell = 0;
  TCHK(hipMemcpyAsync(&ncell, cst.as<int>() + n, sizeof(int), hipMemcpyDeviceToHost, s));
  TCHK(hipStreamSynchronize(s));
  Buf cpos(s), clev(s), cnb(s), cnn(s), cnc(s), fidx(s), fbase(s), fpar(s);
  for (Buf *b : {&cpos, &clev, &cnb, &cnn, &cnc, &fidx, &fbase, &fpar}) TCHK(b->need(4 * (size_t)ncell));
  PreCells C{cpos.as<int>(), clev.as<int>(), cnb.as<int>(), cnn.as<int>(), cnc.as<int>()};
  tree_cells_kernel<<<nb, 256, 0, s>>>(n, RR, Lv.as<signed char>(), cst.as<int>(), C);
  TCHK(hipGetLastError());
  // the root: index 0, children from 1, parent 0
  const int root[3] = {0, 1, 0};
  TCHK(hipMemcpyAsync(fidx.p, &root[0], sizeof(int), hipMemcpyHostToDevice, s));
  TCHK(hipMemcpyAsync(fbase.p, &root[1], sizeof(int), hipMemcpyHostToDevice, s));
  TCHK(hipMemcpyAsync(fpar.p, &root[2], sizeof(int), hipMemcpyHostToDevice, s));
  const unsigned nbc = (unsigned)((ncell + 255) / 256);
  for (int d = 0; d < 30; d++) {
    tree_number_kernel<<<nbc, 256, 0, s>>>(ncell, d, RR, cst.as<int>(), C, fidx.as<int>(), fbase.as<int>(),
                                           fpar.as<int>());
    TCHK(hipGetLastError());
  }
  Buf oip(s), oic(s), onc(s), oib(s), onb(s), olv(s), oX(s), oR(s);
  for (Buf *b : {&oip, &oic, &onc, &oib, &onb, &olv}) TCHK(b->need(4 * (size_t)ncell));
  TCHK(oX.need(24 * (size_t)ncell));
  TCHK(oR.need(8 * (size_t)ncell));
  tree_scatter_kernel<<<nbc, 256, 0, s>>>(ncell, C, fidx.as<int>(), fbase.as<int>(), fpar.as<int>(),
                                          hiS, loS, X0[0], X0[1], X0[2], R0, oip.as<int>(), oic.as<int>(), onc.as<int>(), oib.as<int>(),
                                          onb.as<int>(), olv.as<int>(), oX.as<double>(), oR.as<double>());
  TCHK(hipGetLastError());
  // bodies: by leaf, input order within a leaf
  Buf key(s), key2(s), io(s), io2(s);
  TCHK(key.need(4 * (size_t)n));
  TCHK(key2.need(4 * (size_t)n));
  TCHK(io.need(4 * (size_t)n));
  TCHK(io2.need(4 * (size_t)n));
  tree_leafkey_kernel<<<nb, 256, 0, s>>>(n, idx.as<int>(), lst.as<int>(), key.as<unsigned>(), io.as<int>());
  TCHK(hipGetLastError());
  int nbits = 1;
  while ((1ll << nbits) < (long long)n) nbits++;
  size_t tk = 0;
  TCHK(hipcub::DeviceRadixSort::SortPairs(nullptr, tk, key.as<unsigned>(), key2.as<unsigned>(), io.as<int>(),
                                          io2.as<int>(), n, 0, nbits, s));
  Buf tmp3(s);
  TCHK(tmp3.need(tk));
  TCHK(hipcub::DeviceRadixSort::SortPairs(tmp3.p, tk, key.as<unsigned>(), key2.as<unsigned>(), io.as<int>(),
                                          io2.as<int>(), n, 0, nbits, s));
  for (auto *v : {&iparent, &ichild, &nchild, &ibody, &nbody, &level}) v->resize(ncell);
  X.resize(3 * (size_t)ncell);
  R.resize(ncell);
  TCHK(hipMemcpyAsync(perm.data(), io2.p, 4 * (size_t)n, hipMemcpyDeviceToHost, s));
  TCHK(hipMemcpyAsync(iparent.data(), oip.p, 4 * (size_t)ncell, hipMemcpyDeviceToHost, s));
  TCHK(hipMemcpyAsync(ichild.data(), oic.p, 4 * (size_t)ncell, hipMemcpyDeviceToHost, s));
  TCHK(hipMemcpyAsync(nchild.data(), onc.p, 4 * (size_t)ncell, hipMemcpyDeviceToHost, s));
  TCHK(hipMemcpyAsync(ibody.data(), oib.p, 4 * (size_t)ncell, hipMemcpyDeviceToHost, s));
  TCHK(hipMemcpyAsync(nbody.data(), onb.p, 4 * (size_t)ncell, hipMemcpyDeviceToHost, s));
  TCHK(hipMemcpyAsync(level.data(), olv.p, 4 * (size_t)ncell, hipMemcpyDeviceToHost, s));
  TCHK(hipMemcpyAsync(X.data(), oX.p, 24 * (size_t)ncell, hipMemcpyDeviceToHost, s));
  TCHK(hipMemcpyAsync(R.data(), oR.p, 8 * (size_t)ncell, hipMemcpyDeviceToHost, s));
  TCHK(hipStreamSynchronize(s));
  return hipSuccess;
}

}  // namespace fmmdev
