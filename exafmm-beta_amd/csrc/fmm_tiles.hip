// fmm_tiles.hip -- the M2L offset groups and target tiles built on the device.
//
// The same partition as fmm::build_m2l_groups and the same tiles, slices and
// work items as fmm::build_m2l_tiles (fmm_host.cpp), for trees whose cells all
// have the radius of their level (trees built by fmm::build_tree or
// fmmdev::device_tree):
//
//  * every M2L pair's offset, in units of its finer cell's size, reduced by
//    common factors of two (the host's lattice key), packed into one 64-bit
//    key; a hash table gives each pair its key's slot;
//  * over the distinct keys only (thousands): group numbers in key order,
//    reflection classes and their representatives' offsets -- the host's
//    numbering is first-appearance order, which only permutes the groups and
//    classes;
//  * tiles: the targets sorted by (level, cell), TT per tile -- the host's
//    order, so the same tiles; each tile's pairs sorted by (class, target) and
//    every (tile, class) run of m pairs dealt into S = max(ceil(m / SW), most
//    pairs of one target) slices of distinct targets, pair i of the run to
//    slice i mod S, as the host does.
//
// Periodic lists: the image is part of the key, and the reflection class is
// that of the whole translation vector.  Keys that do not fit (an offset
// component of 2^13 or more after the reduction, an offset off the lattice)
// make the whole plan fall back to the host.
#include <hip/hip_runtime.h>
#include <hipcub/hipcub.hpp>

#include <algorithm>
#include <cmath>
#include <cstdint>
#include <utility>
#include <vector>

#include "fmm_device.hpp"
#include "fmm_host.hpp"

namespace fmmdev {

namespace {

constexpr unsigned long long kEmptyKey = ~0ull;
constexpr int kKBits = 14, kKOff = 1 << (kKBits - 1);  // offset components in [-2^13, 2^13)
constexpr int kImgBits = 5;  // periodic image 0..26
constexpr int kHashBits = 20;

struct DBufT {  // device scratch from the plan builders' per-stream cache
  hipStream_t s;
  void *p = nullptr;
  size_t bytes = 0;  // capacity
  explicit DBufT(hipStream_t st) : s(st) {}
  DBufT(const DBufT &) = delete;
  ~DBufT() {
    if (p) plan_scratch_put(p, bytes, s);
  }
  hipError_t need(size_t b) {
    if (b <= bytes) return hipSuccess;
    if (p) plan_scratch_put(p, bytes, s);
    p = nullptr;
    bytes = 0;
    return plan_scratch_get(&p, &bytes, b, s);
  }
  template <class T> T *as() const { return static_cast<T *>(p); }
};

#define TCHK(expr)                   \
  do {                               \
    hipError_t e_ = (expr);          \
    if (e_ != hipSuccess) return e_; \
  } while (0)

__device__ __forceinline__ unsigned long long mix64(unsigned long long k) {
  k ^= k >> 33;
  k *= 0xff51afd7ed558ccdull;
  k ^= k >> 33;
  k *= 0xc4ceb9fe1a85ec53ull;
  k ^= k >> 33;
  return k;
}

// the target cell of every pair; a wavefront a cell, its lanes the cell's
// pairs (a thread a cell wrote one pair after the other: 30 us for 3700 cells
// of some 160 pairs, 3 us now)
__global__ void __launch_bounds__(256) pair_target_kernel(int ncell, const int *__restrict__ ptr,
                                                          int *__restrict__ ptgt) {
  const int c = blockIdx.x * 4 + threadIdx.x / 64;
  if (c >= ncell) return;
  for (int p = ptr[c] + threadIdx.x % 64; p < ptr[c + 1]; p += 64) ptgt[p] = c;
}

// every pair's key (host: build_m2l_groups), inserted into the hash table;
// slot[p] its slot, *bad set when a key does not fit
__global__ void pair_key_kernel(int64_t np, const int *__restrict__ ptgt, const int *__restrict__ psrc,
                                const double *__restrict__ X, const int *__restrict__ level, double R0,
                                unsigned long long *__restrict__ table, int *__restrict__ slot,
                                int *__restrict__ bad) {
#pragma clang fp contract(off)
  const int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= np) return;
  const int c = ptgt[p], sc = psrc[p] & fmm::kCellMask;
  const int lt = level[c], ls = level[sc];
  int e = lt > ls ? lt : ls;
  const double scale = ldexp(1.0, e) / R0;
  long long k[3];
  bool ok = true;
  for (int d = 0; d < 3; d++) {
    const double v = (X[3 * (size_t)c + d] - X[3 * (size_t)sc + d]) * scale;
    const double rv = rint(v);
    if (!(fabs(v - rv) < 1e-6) || fabs(rv) >= (double)(1 << 26)) ok = false;
    k[d] = (long long)rv;
  }
  if (ok) {
    while (e > 0 && ((k[0] | k[1] | k[2]) & 1) == 0) {
      k[0] /= 2;
      k[1] /= 2;
      k[2] /= 2;
      e--;
    }
    for (int d = 0; d < 3; d++)
      if (k[d] <= -kKOff || k[d] >= kKOff) ok = false;
  }
  if (!ok) {
    atomicOr(bad, 1);
    slot[p] = -1;
    return;
  }
  const unsigned long long img = (unsigned long long)(psrc[p] >> fmm::kImageShift);
  const unsigned long long key = ((unsigned long long)e << (3 * kKBits + kImgBits)) | (img << (3 * kKBits)) |
                                 ((unsigned long long)(k[0] + kKOff) << (2 * kKBits)) |
                                 ((unsigned long long)(k[1] + kKOff) << kKBits) | (unsigned long long)(k[2] + kKOff);
  const unsigned long long mask = (1ull << kHashBits) - 1;
  unsigned long long h = mix64(key) & mask;
  for (int probe = 0; probe <= (int)mask; probe++) {
    // a slot changes once, empty -> key: a plain read that shows a key is
    // final (most pairs find theirs so, without an atomic on a hot slot);
    // one that shows empty may be stale, and the CAS decides
    unsigned long long prev = table[h];
    if (prev == kEmptyKey) prev = atomicCAS(&table[h], kEmptyKey, key);
    if (prev == kEmptyKey || prev == key) {
      slot[p] = (int)h;
      return;
    }
    h = (h + 1) & mask;
  }
  atomicOr(bad, 2);  // table full
  slot[p] = -1;
}

// The filled slots of the hash table (any order: they are sorted next). Bound
// by the additions to the one counter, about 8 ns each, so a block counts its
// kCompact * 256 slots in LDS and adds once: 104 us at 13k keys when every
// wavefront that held a key added for itself, 7 us now.
constexpr int kCompact = 16;
__global__ void __launch_bounds__(256) table_compact_kernel(int tsize, const unsigned long long *__restrict__ table,
                                                            unsigned long long *__restrict__ okey,
                                                            int *__restrict__ oslot, int *__restrict__ count) {
  __shared__ int nblk, base;
  if (threadIdx.x == 0) nblk = 0;
  __syncthreads();
  const int h0 = blockIdx.x * (256 * kCompact) + threadIdx.x;
  unsigned long long k[kCompact];
  int at[kCompact];
#pragma unroll
  for (int i = 0; i < kCompact; i++) {
    const int h = h0 + 256 * i;
    k[i] = h < tsize ? table[h] : kEmptyKey;
  }
#pragma unroll
  for (int i = 0; i < kCompact; i++) at[i] = k[i] != kEmptyKey ? atomicAdd(&nblk, 1) : 0;
  __syncthreads();
  if (threadIdx.x == 0) base = nblk ? atomicAdd(count, nblk) : 0;
  __syncthreads();
#pragma unroll
  for (int i = 0; i < kCompact; i++)
    if (k[i] != kEmptyKey) {
      okey[base + at[i]] = k[i];
      oslot[base + at[i]] = h0 + 256 * i;
    }
}

// group g (keys in order) of slot gslot[g]: slot2grp, its reflections and the
// key of its class: the offset and image of the translation vector (offset
// minus image shift) reflected into non-negative components
__global__ void group_class_kernel(int ng, const unsigned long long *__restrict__ gkey, const int *__restrict__ gslot,
                                   double R0, double3 cycle, int periodic, int *__restrict__ slot2grp,
                                   unsigned char *__restrict__ grefl, unsigned long long *__restrict__ ckey,
                                   int *__restrict__ gid, double *__restrict__ adx) {
#pragma clang fp contract(off)
  const int g = blockIdx.x * blockDim.x + threadIdx.x;
  if (g >= ng) return;
  slot2grp[gslot[g]] = g;
  const unsigned long long key = gkey[g], kmask = (1ull << kKBits) - 1;
  const int e = (int)(key >> (3 * kKBits + kImgBits));
  const int img = (int)((key >> (3 * kKBits)) & ((1u << kImgBits) - 1));
  const double u = R0 / ldexp(1.0, e);
  const double cyc[3] = {cycle.x, cycle.y, cycle.z};
  int ic[3] = {img / 9 - 1, img / 3 % 3 - 1, img % 3 - 1};
  unsigned char r = 0;
  unsigned long long ck = (unsigned long long)e << kImgBits;
  long long k[3];
  for (int d = 0; d < 3; d++) {
    k[d] = (long long)((key >> (kKBits * (2 - d))) & kmask) - kKOff;
    const double sh = periodic ? ic[d] * cyc[d] : 0.0;
    const double tv = (double)k[d] * u - sh;
    adx[3 * (size_t)g + d] = fabs(tv);
    if (periodic ? tv < 0.0 : k[d] < 0) {
      r |= (unsigned char)(1 << d);
      k[d] = -k[d];
      ic[d] = -ic[d];
    }
  }
  if (periodic) ck |= (unsigned long long)((ic[0] + 1) * 9 + (ic[1] + 1) * 3 + ic[2] + 1);
  for (int d = 0; d < 3; d++) ck = ck << kKBits | (unsigned long long)(k[d] + kKOff);
  grefl[g] = r;
  ckey[g] = ck;
  gid[g] = g;
}

// class keys in order: 1 where a class starts
__global__ void class_flag_kernel(int ng, const unsigned long long *__restrict__ ckey, int *__restrict__ flag) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < ng) flag[i] = i == 0 || ckey[i] != ckey[i - 1];
}

// every group's class (cid: inclusive sum of the flags), every class's offset
__global__ void class_number_kernel(int ng, const unsigned long long *__restrict__ ckey, const int *__restrict__ cid,
                                    const int *__restrict__ gid, const double *__restrict__ adx,
                                    int *__restrict__ gcanon, double *__restrict__ cdx) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= ng) return;
  const int g = gid[i], c = cid[i] - 1;
  gcanon[g] = c;
  if (i == 0 || ckey[i] != ckey[i - 1])
    for (int d = 0; d < 3; d++) cdx[3 * (size_t)c + d] = adx[3 * (size_t)g + d];
}

// the cells' sort keys: (level, cell) of a target -- siblings are adjacent --
// and behind them the cells without pairs
__global__ void target_key_kernel(int ncell, const int *__restrict__ ptr, const int *__restrict__ level,
                                  unsigned long long *__restrict__ key, int *__restrict__ cell) {
  const int c = blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= ncell) return;
  key[c] = ptr[c + 1] == ptr[c] ? 1ull << 39 : ((unsigned long long)level[c] << 32) | (unsigned)c;
  cell[c] = c;
}

__global__ void tile_of_kernel(int nt, const int *__restrict__ cells, int TT, int *__restrict__ tile_of,
                               int *__restrict__ local) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= nt) return;
  tile_of[cells[i]] = i / TT;
  local[cells[i]] = i % TT;
}

// pair sort keys (tile, class, target in the tile), the pair's source with
// them; the reflections ride in the key above the sorted bits.  A tile's
// pairs are sorted on as many bits as tiles, classes and targets take: 31 for
// 12M pairs of a 1M-body tree, four passes of 0.1 ms where fixed fields of 32
// and 8 bits took seven
struct TileKey {
  int lb, cb;  // bits of the target in the tile, of the class
  __device__ unsigned long long body(unsigned long long k) const { return k & ((1ull << 61) - 1); }
  __device__ unsigned long long segment(unsigned long long k) const { return body(k) >> lb; }
  __device__ int local(unsigned long long k) const { return (int)(k & ((1ull << lb) - 1)); }
  __device__ int rep(unsigned long long k) const { return (int)((k >> lb) & ((1ull << cb) - 1)); }
  __device__ int tile(unsigned long long k) const { return (int)(body(k) >> (lb + cb)); }
  __device__ int refl(unsigned long long k) const { return (int)(k >> 61); }
};
__global__ void pair_tile_key_kernel(int64_t np, const int *__restrict__ ptgt, const int *__restrict__ slot,
                                     const int *__restrict__ slot2grp, const int *__restrict__ gcanon,
                                     const unsigned char *__restrict__ grefl, const int *__restrict__ tile_of,
                                     const int *__restrict__ local, TileKey K, unsigned long long *__restrict__ key) {
  const int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= np) return;
  const int c = ptgt[p], g = slot2grp[slot[p]];
  key[p] = (unsigned long long)grefl[g] << 61 | (unsigned long long)tile_of[c] << (K.lb + K.cb) |
           (unsigned long long)gcanon[g] << K.lb | (unsigned)local[c];
}

// sorted position i: flags of run starts (segment = (tile, class), run = target)
__global__ void seg_flags_kernel(int64_t np, TileKey K, const unsigned long long *__restrict__ key, int *__restrict__ segf,
                                 int *__restrict__ runs) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= np) return;
  const bool segb = i == 0 || K.segment(key[i]) != K.segment(key[i - 1]);
  const bool runb = i == 0 || K.body(key[i]) != K.body(key[i - 1]);
  segf[i] = segb ? 1 : 0;
  runs[i] = runb ? (int)i : 0;  // max-scanned into the run start
}

// per segment: start, length and the longest run of one target
__global__ void seg_stats_kernel(int64_t np, TileKey K, const unsigned long long *__restrict__ key,
                                 const int *__restrict__ segid, const int *__restrict__ runstart,
                                 int *__restrict__ sstart, int *__restrict__ slen, int *__restrict__ smost) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= np) return;
  const int sg = segid[i] - 1;
  if (i == 0 || K.segment(key[i]) != K.segment(key[i - 1])) sstart[sg] = (int)i;
  if (i + 1 == np || K.segment(key[i + 1]) != K.segment(key[i])) slen[sg] = (int)(i + 1);  // end, made a length below
  // the longest run of one target; runs of one pair cannot raise the slice
  // count max(ceil(m / SW), longest run) above ceil(m / SW) >= 1, so only
  // longer runs (a target's several reflections of one class) take an atomic
  if (i + 1 == np || K.body(key[i + 1]) != K.body(key[i])) {
    const int len = (int)(i - runstart[i] + 1);
    if (len > 1) atomicMax(&smost[sg], len);
  }
}

__global__ void seg_slices_kernel(int nseg, const int *__restrict__ sstart, int *__restrict__ slen,
                                  const int *__restrict__ smost, int SW, int *__restrict__ nsl) {
  const int g = blockIdx.x * blockDim.x + threadIdx.x;
  if (g >= nseg) return;
  const int m = slen[g] - sstart[g];
  slen[g] = m;
  const int a = (m + SW - 1) / SW;
  nsl[g] = a > smost[g] ? a : smost[g];
}

// deal every sorted pair into its slice: the tile's source and (target | reflection << 8)
__global__ void deal_kernel(int64_t np, TileKey K, const unsigned long long *__restrict__ key,
                            const int *__restrict__ src, const int *__restrict__ segid,
                            const int *__restrict__ sstart, const int *__restrict__ slen, const int *__restrict__ nsl,
                            int *__restrict__ tsrc, unsigned short *__restrict__ tlt) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= np) return;
  const int sg = segid[i] - 1, s0 = sstart[sg], m = slen[sg], S = nsl[sg];
  const int r = (int)(i - s0), j = r % S, q = r / S;
  const int out = s0 + j * (m / S) + min(j, m % S) + q;
  tsrc[out] = src[i];
  tlt[out] = (unsigned short)(K.local(key[i]) | K.refl(key[i]) << 8);
}

// the slice descriptors of every segment, and each tile's first slice
__global__ void slice_desc_kernel(int nseg, TileKey K, const unsigned long long *__restrict__ key, const int *__restrict__ sstart,
                                  const int *__restrict__ slen, const int *__restrict__ nsl,
                                  const int *__restrict__ sbase, int *__restrict__ slice, int *__restrict__ tptr) {
  const int g = blockIdx.x * blockDim.x + threadIdx.x;
  if (g >= nseg) return;
  const int s0 = sstart[g], m = slen[g], S = nsl[g];
  const unsigned long long k = key[s0];
  const int rep = K.rep(k), tile = K.tile(k);
  if (g == 0 || K.tile(key[sstart[g - 1]]) != tile) tptr[tile] = sbase[g];
  for (int j = 0; j < S; j++) {
    int *o = slice + 4 * (size_t)(sbase[g] + j);
    o[0] = rep;
    o[1] = s0 + j * (m / S) + min(j, m % S);
    o[2] = m / S + (j < m % S ? 1 : 0);
    o[3] = 0;
  }
}

}  // namespace

hipError_t device_groups_tiles(const fmm::Tree &t, const fmm::Lists &L, int TT, int SW, int seg,
                               fmm::M2LGroups &G, fmm::M2LTiles &T, bool &done, hipStream_t s,
                               PlanArrays *keep, const int *dsrc_in, const double *cycle) {
  done = false;
  if (keep) {
    keep->tiles = false;
    keep->t_slice.bytes = 0;
    keep->t_src.bytes = 0;
    keep->t_lt.bytes = 0;
    keep->nslice = 0;
  }
  const int nc = t.ncell;
  const int64_t np = L.nm2l;
  if (nc == 0 || np == 0 || np > 0x7fffffff || TT > 255) return hipSuccess;
  int ntg = 0;  // cells with pairs
  for (int c = 0; c < nc; c++) {
    if (t.R[c] != t.R[0] / (1 << t.level[c])) return hipSuccess;  // regular tree: every radius R0 / 2^level
    ntg += L.m2l_ptr[c + 1] > L.m2l_ptr[c];
  }
  const double R0 = t.R[0];
  DBufT dX(s), dlev(s), dptr(s), dsrc(s), dtgt(s), dtab(s), dslot(s), dbad(s);
  TCHK(dX.need(sizeof(double) * 3 * (size_t)nc));
  TCHK(dlev.need(4 * (size_t)nc));
  TCHK(dptr.need(4 * ((size_t)nc + 1)));
  // the pair sources: given on the device, or the lists' device column when
  // the plan keeps one, else uploaded from L
  const bool dev_src = dsrc_in || (keep && keep->lists && keep->m2l_src.bytes == 4 * (size_t)np);
  if (!dev_src) TCHK(dsrc.need(4 * (size_t)np));
  const int *psrc = dsrc_in ? dsrc_in : dev_src ? keep->m2l_src.as<int>() : dsrc.as<int>();
  TCHK(dtgt.need(4 * (size_t)np));
  TCHK(hipMemcpyAsync(dX.p, t.X.data(), sizeof(double) * 3 * (size_t)nc, hipMemcpyHostToDevice, s));
  TCHK(hipMemcpyAsync(dlev.p, t.level.data(), 4 * (size_t)nc, hipMemcpyHostToDevice, s));
  TCHK(hipMemcpyAsync(dptr.p, L.m2l_ptr.data(), 4 * ((size_t)nc + 1), hipMemcpyHostToDevice, s));
  if (!dev_src) TCHK(hipMemcpyAsync(dsrc.p, L.m2l_src.data(), 4 * (size_t)np, hipMemcpyHostToDevice, s));
  const unsigned nbc = (unsigned)((nc + 255) / 256), nbp = (unsigned)((np + 255) / 256);
  pair_target_kernel<<<(unsigned)((nc + 3) / 4), 256, 0, s>>>(nc, dptr.as<int>(), dtgt.as<int>());
  TCHK(hipGetLastError());
  // keys and the hash table
  const size_t tsize = (size_t)1 << kHashBits;
  TCHK(dtab.need(8 * tsize));
  TCHK(dslot.need(4 * (size_t)np));
  TCHK(dbad.need(4));
  TCHK(hipMemsetAsync(dtab.p, 0xff, 8 * tsize, s));
  TCHK(hipMemsetAsync(dbad.p, 0, 4, s));
  pair_key_kernel<<<nbp, 256, 0, s>>>(np, dtgt.as<int>(), psrc, dX.as<double>(), dlev.as<int>(), R0,
                                       dtab.as<unsigned long long>(), dslot.as<int>(),
                                       dbad.as<int>());
  TCHK(hipGetLastError());
  // the filled slots come back (key, slot), not the whole table
  DBufT dfk(s), dfs(s), dcn(s);
  TCHK(dfk.need(8 * tsize));
  TCHK(dfs.need(4 * tsize));
  TCHK(dcn.need(4));
  TCHK(hipMemsetAsync(dcn.p, 0, 4, s));
  table_compact_kernel<<<(unsigned)((tsize + 256 * kCompact - 1) / (256 * kCompact)), 256, 0, s>>>(
      (int)tsize, dtab.as<unsigned long long>(), dfk.as<unsigned long long>(), dfs.as<int>(), dcn.as<int>());
  TCHK(hipGetLastError());
  int bad = 0, nfill = 0;
  TCHK(hipMemcpyAsync(&bad, dbad.p, 4, hipMemcpyDeviceToHost, s));
  TCHK(hipMemcpyAsync(&nfill, dcn.p, 4, hipMemcpyDeviceToHost, s));
  TCHK(hipStreamSynchronize(s));
  if (bad) return hipSuccess;  // the host groups this plan
  // groups in key order, classes in the order of their representatives' keys
  const int ng = nfill;
  const unsigned nbg = (unsigned)((ng + 255) / 256);
  DBufT dgk(s), dgs(s), ds2g(s), dgc(s), dgr(s), dck(s), dck2(s), dgi(s), dgi2(s), dadx(s), dcf(s), dcid(s), dcdx(s),
      tmp(s);
  TCHK(dgk.need(8 * (size_t)ng));
  TCHK(dgs.need(4 * (size_t)ng));
  TCHK(ds2g.need(4 * tsize));
  TCHK(dgc.need(4 * (size_t)ng));
  TCHK(dgr.need((size_t)ng));
  for (DBufT *d : {&dck, &dck2}) TCHK(d->need(8 * (size_t)ng));
  for (DBufT *d : {&dgi, &dgi2, &dcf, &dcid}) TCHK(d->need(4 * (size_t)ng));
  for (DBufT *d : {&dadx, &dcdx}) TCHK(d->need(24 * (size_t)ng));
  constexpr int kKeyBits = 3 * kKBits + kImgBits + 6;
  auto sort_u64 = [&](const DBufT &k, const DBufT &ko, const int *v, const DBufT &vo, int n, int bits) -> hipError_t {
    size_t bytes = 0;
    TCHK(hipcub::DeviceRadixSort::SortPairs(nullptr, bytes, k.as<unsigned long long>(), ko.as<unsigned long long>(),
                                            v, vo.as<int>(), n, 0, bits, s));
    TCHK(tmp.need(bytes));
    return hipcub::DeviceRadixSort::SortPairs(tmp.p, bytes, k.as<unsigned long long>(), ko.as<unsigned long long>(),
                                              v, vo.as<int>(), n, 0, bits, s);
  };
  TCHK(sort_u64(dfk, dgk, dfs.as<int>(), dgs, ng, kKeyBits));
  group_class_kernel<<<nbg, 256, 0, s>>>(ng, dgk.as<unsigned long long>(), dgs.as<int>(), R0,
                                         cycle ? make_double3(cycle[0], cycle[1], cycle[2]) : make_double3(0, 0, 0),
                                         cycle ? 1 : 0, ds2g.as<int>(), dgr.as<unsigned char>(),
                                         dck.as<unsigned long long>(), dgi.as<int>(), dadx.as<double>());
  TCHK(hipGetLastError());
  TCHK(sort_u64(dck, dck2, dgi.as<int>(), dgi2, ng, kKeyBits));
  class_flag_kernel<<<nbg, 256, 0, s>>>(ng, dck2.as<unsigned long long>(), dcf.as<int>());
  TCHK(hipGetLastError());
  size_t tbc = 0;
  TCHK(hipcub::DeviceScan::InclusiveSum(nullptr, tbc, dcf.as<int>(), dcid.as<int>(), ng, s));
  TCHK(tmp.need(tbc));
  TCHK(hipcub::DeviceScan::InclusiveSum(tmp.p, tbc, dcf.as<int>(), dcid.as<int>(), ng, s));
  class_number_kernel<<<nbg, 256, 0, s>>>(ng, dck2.as<unsigned long long>(), dcid.as<int>(), dgi2.as<int>(),
                                          dadx.as<double>(), dgc.as<int>(), dcdx.as<double>());
  TCHK(hipGetLastError());
  // the tile path reads the counts and the classes' offsets only
  G = fmm::M2LGroups();
  G.ngroup = ng;
  G.rest_ptr.assign((size_t)nc + 1, 0);
  G.grp_ptr.assign(1, 0);
  // tiles: targets in (level, cell) order
  DBufT dtk(s), dtk2(s), dtc(s), dtc2(s), dtof(s), dloc(s);
  TCHK(dtk.need(8 * (size_t)nc));
  TCHK(dtk2.need(8 * (size_t)nc));
  TCHK(dtc.need(4 * (size_t)nc));
  TCHK(dtc2.need(4 * (size_t)nc));
  TCHK(dtof.need(4 * (size_t)nc));
  TCHK(dloc.need(4 * (size_t)nc));
  target_key_kernel<<<nbc, 256, 0, s>>>(nc, dptr.as<int>(), dlev.as<int>(), dtk.as<unsigned long long>(),
                                        dtc.as<int>());
  TCHK(hipGetLastError());
  TCHK(sort_u64(dtk, dtk2, dtc.as<int>(), dtc2, nc, 40));
  tile_of_kernel<<<(unsigned)((ntg + 255) / 256), 256, 0, s>>>(ntg, dtc2.as<int>(), TT, dtof.as<int>(),
                                                                dloc.as<int>());
  TCHK(hipGetLastError());
  T = fmm::M2LTiles();
  T.TT = TT;
  T.ntile = (ntg + TT - 1) / TT;
  T.tgt.assign((size_t)T.ntile * TT, -1);
  // pairs sorted by (tile, class, target)
  DBufT dpk(s), dpk2(s), dpv2(s);
  TCHK(dpk.need(8 * (size_t)np));
  TCHK(dpk2.need(8 * (size_t)np));
  TCHK(dpv2.need(4 * (size_t)np));
  auto bits = [](int64_t n) {  // of 0 .. n - 1
    int b = 1;
    while ((1ll << b) < n) b++;
    return b;
  };
  const TileKey K{bits(TT), bits(ng)};
  const int kbits = K.lb + K.cb + bits(T.ntile);
  if (kbits > 61) return hipSuccess;
  pair_tile_key_kernel<<<nbp, 256, 0, s>>>(np, dtgt.as<int>(), dslot.as<int>(), ds2g.as<int>(), dgc.as<int>(),
                                           dgr.as<unsigned char>(), dtof.as<int>(), dloc.as<int>(), K,
                                           dpk.as<unsigned long long>());
  TCHK(hipGetLastError());
  TCHK(sort_u64(dpk, dpk2, psrc, dpv2, (int)np, kbits));
  // segments (tile, class) and runs (target)
  DBufT dsegf(s), dsegid(s), druns(s), drs(s);
  TCHK(dsegf.need(4 * (size_t)np));
  TCHK(dsegid.need(4 * (size_t)np));
  TCHK(druns.need(4 * (size_t)np));
  TCHK(drs.need(4 * (size_t)np));
  seg_flags_kernel<<<nbp, 256, 0, s>>>(np, K, dpk2.as<unsigned long long>(), dsegf.as<int>(), druns.as<int>());
  TCHK(hipGetLastError());
  size_t ts1 = 0, ts2 = 0;
  TCHK(hipcub::DeviceScan::InclusiveSum(nullptr, ts1, dsegf.as<int>(), dsegid.as<int>(), (int)np, s));
  TCHK(hipcub::DeviceScan::InclusiveScan(nullptr, ts2, druns.as<int>(), drs.as<int>(), hipcub::Max(), (int)np, s));
  TCHK(tmp.need(std::max(ts1, ts2)));
  TCHK(hipcub::DeviceScan::InclusiveSum(tmp.p, ts1, dsegf.as<int>(), dsegid.as<int>(), (int)np, s));
  TCHK(hipcub::DeviceScan::InclusiveScan(tmp.p, ts2, druns.as<int>(), drs.as<int>(), hipcub::Max(), (int)np, s));
  int nseg = 0;
  TCHK(hipMemcpyAsync(&nseg, dsegid.as<int>() + (np - 1), 4, hipMemcpyDeviceToHost, s));
  TCHK(hipMemcpyAsync(&G.ncanon, dcid.as<int>() + (ng - 1), 4, hipMemcpyDeviceToHost, s));
  TCHK(hipStreamSynchronize(s));
  DBufT dss(s), dsl(s), dsm(s), dns(s), dsb(s);
  for (DBufT *b : {&dss, &dsl, &dsm, &dns, &dsb}) TCHK(b->need(4 * ((size_t)nseg + 1)));
  TCHK(hipMemsetAsync(dsm.p, 0, 4 * (size_t)nseg, s));
  seg_stats_kernel<<<nbp, 256, 0, s>>>(np, K, dpk2.as<unsigned long long>(), dsegid.as<int>(), drs.as<int>(),
                                       dss.as<int>(), dsl.as<int>(), dsm.as<int>());
  TCHK(hipGetLastError());
  const unsigned nbs = (unsigned)((nseg + 255) / 256);
  seg_slices_kernel<<<nbs, 256, 0, s>>>(nseg, dss.as<int>(), dsl.as<int>(), dsm.as<int>(), SW, dns.as<int>());
  TCHK(hipGetLastError());
  size_t ts3 = 0;
  TCHK(hipcub::DeviceScan::ExclusiveSum(nullptr, ts3, dns.as<int>(), dsb.as<int>(), nseg + 1, s));
  TCHK(tmp.need(ts3));
  TCHK(hipMemsetAsync(dns.as<int>() + nseg, 0, 4, s));
  TCHK(hipcub::DeviceScan::ExclusiveSum(tmp.p, ts3, dns.as<int>(), dsb.as<int>(), nseg + 1, s));
  int nslice = 0;
  TCHK(hipMemcpyAsync(&nslice, dsb.as<int>() + nseg, 4, hipMemcpyDeviceToHost, s));
  TCHK(hipStreamSynchronize(s));
  // the tiles' pair sources, pair targets and slices: on the device in keep,
  // else staged here and copied to T
  DBufT dts(s), dtl(s), dsd(s), dtp(s);
  int *osrc, *osd;
  unsigned short *olt;
  if (keep) {
    int dev = 0;
    TCHK(hipGetDevice(&dev));
    TCHK(keep->t_src.alloc(4 * (size_t)np, dev));
    TCHK(keep->t_lt.alloc(2 * (size_t)np, dev));
    TCHK(keep->t_slice.alloc(16 * (size_t)nslice, dev));
    osrc = keep->t_src.as<int>();
    olt = keep->t_lt.as<unsigned short>();
    osd = keep->t_slice.as<int>();
  } else {
    TCHK(dts.need(4 * (size_t)np));
    TCHK(dtl.need(2 * (size_t)np));
    TCHK(dsd.need(16 * (size_t)nslice));
    osrc = dts.as<int>();
    olt = dtl.as<unsigned short>();
    osd = dsd.as<int>();
  }
  TCHK(dtp.need(4 * ((size_t)T.ntile + 1)));
  deal_kernel<<<nbp, 256, 0, s>>>(np, K, dpk2.as<unsigned long long>(), dpv2.as<int>(), dsegid.as<int>(),
                                  dss.as<int>(), dsl.as<int>(), dns.as<int>(), osrc, olt);
  TCHK(hipGetLastError());
  slice_desc_kernel<<<nbs, 256, 0, s>>>(nseg, K, dpk2.as<unsigned long long>(), dss.as<int>(), dsl.as<int>(),
                                        dns.as<int>(), dsb.as<int>(), osd, dtp.as<int>());
  TCHK(hipGetLastError());
  G.cdx.resize(3 * (size_t)G.ncanon);
  TCHK(hipMemcpyAsync(G.cdx.data(), dcdx.p, 24 * (size_t)G.ncanon, hipMemcpyDeviceToHost, s));
  TCHK(hipMemcpyAsync(T.tgt.data(), dtc2.p, 4 * (size_t)ntg, hipMemcpyDeviceToHost, s));
  T.ptr.resize((size_t)T.ntile + 1);
  TCHK(hipMemcpyAsync(T.ptr.data(), dtp.p, 4 * (size_t)T.ntile, hipMemcpyDeviceToHost, s));
  if (keep) {
    T.slice.clear();
    T.src.clear();
    T.lt.clear();
  } else {
    T.slice.resize(4 * (size_t)nslice);
    T.src.resize(np);
    T.lt.resize(np);
    TCHK(hipMemcpyAsync(T.slice.data(), dsd.p, 16 * (size_t)nslice, hipMemcpyDeviceToHost, s));
    TCHK(hipMemcpyAsync(T.src.data(), dts.p, 4 * (size_t)np, hipMemcpyDeviceToHost, s));
    TCHK(hipMemcpyAsync(T.lt.data(), dtl.p, 2 * (size_t)np, hipMemcpyDeviceToHost, s));
  }
  TCHK(hipStreamSynchronize(s));
  T.ptr[T.ntile] = nslice;
  if (keep) {
    TCHK(hipGetDevice(&keep->device));
    keep->nslice = nslice;
    keep->tiles = true;
  }
  fmm::split_m2l_tiles(T, seg);
  done = true;
  return hipSuccess;
}

}  // namespace fmmdev
