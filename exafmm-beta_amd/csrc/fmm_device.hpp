// fmm_device.hpp -- launchers for the gfx950 Laplace FMM kernels.
//
// Device data layout (all in HBM, tree order):
//   bodies: SoA x, y, z, q and targets pot, ax, ay, az (double)
//   cells : SoA centres cx, cy, cz; int ibody, nbody, ichild, nchild, iparent
//   M     : [ncell][NTERM] complex, M~[n,m] = M[n,m] / s(n,m)
//   L     : [ncell][NTERM] complex, L^[n,m] = L[n,m] * s(n,m)
// with NTERM = P(P+1)/2, index n(n+1)/2+m, and s(n,m) = sqrt((n-m)!(n+m)!);
// M and L are exafmm-beta's coefficients (kernels/laplace.h) rescaled so every
// operator becomes a plain sum over regular / singular solid harmonics.
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>
#include <functional>
#include <vector>

#include "fmm_host.hpp"

namespace fmmdev {

struct DevBodies {
  const double *x, *y, *z, *q;
  double *pot, *ax, *ay, *az;
};

struct DevCells {
  const double *cx, *cy, *cz;
  const int *ibody, *nbody, *ichild, *nchild, *iparent;
};

constexpr int kMaxP = 20;

// p[0, n) = 0 with a kernel (no memset node when the stream is being captured)
hipError_t launch_zero(double *p, size_t n, hipStream_t s);
// p, x, y, z[0, n) = 0 likewise
hipError_t launch_zero_targets(double *p, double *x, double *y, double *z, size_t n, hipStream_t s);
// bodies into tree order: x/y/z/q[i] from input body perm[i] of xin (AoS)
// and qin
hipError_t launch_gather_bodies(int n, const int *perm, const double *xin, const double *qin, double *x, double *y,
                                double *z, double *q, hipStream_t s);
// q[i] = qin[perm[i]]; trg[4 o .. 4 o + 3] = body i's potential and gradient, o =
// perm[i] (i when perm is null)
hipError_t launch_gather_charges(int n, const int *perm, const double *qin, double *q, hipStream_t s);
hipError_t launch_pack_targets(int n, const int *perm, DevBodies B, double *trg, hipStream_t s);
// body_leaf[i] = the leaf holding body i (tree order)
hipError_t launch_body_leaf(int nleaf, const int *leaves, const int *ibody, const int *nbody, int *body_leaf,
                            hipStream_t s);

bool order_supported(int P);
hipError_t init_constants();

// P2M for every leaf in `leaves` (kernels/laplace.h:237-252)
// P2M and P2P deal a leaf's bodies or list to more lanes while the leaves do not
// fill the GPU.  The sums' order follows, so it is decided for each system of a
// forest by its own leaves: leaves[0, nfew) are of systems of less than
// kP2MFillLeaves leaves, the other nmany of larger ones
constexpr int kP2MFillLeaves = 8192, kP2PFillLeaves = 12000;
hipError_t launch_p2m(int P, DevBodies B, DevCells C, const int *leaves, int nfew, int nmany, double2 *M,
                      hipStream_t s);
// M2M into every parent listed in `cells` from its children (laplace.h:254-290)
hipError_t launch_m2m(int P, DevCells C, const int *cells, int ncell, double2 *M, hipStream_t s);
// M2L: L[t] (=|+=) sum over the CSR list of t (laplace.h:292-322), one
// wavefront per target, harmonics generated per pair (deterministic order)
hipError_t launch_m2l(int P, DevCells C, const int *targets, int ntarget, const int *ptr,
                      const int *src, double3 xper, const double2 *M, double2 *L, int accumulate,
                      hipStream_t s);
// M2L over offset groups on FP64 MFMA: chunks are (group, begin, count, 0) over
// the grouped pair arrays; adds into L with atomics (L must hold its initial
// value).  Available for the orders where m2l_mfma_supported(P).
bool m2l_mfma_supported(int P);
constexpr int kM2LChunkPairs = 512;  // pairs per M2L chunk (one block)
hipError_t launch_m2l_mfma(int P, const int4 *chunks, int nchunk, const double *gdx, const int *ptgt,
                           const int *psrc, const double2 *M, double2 *L, hipStream_t s);
// L2L into every cell in `cells` from its parent (laplace.h:324-357); accumulates
hipError_t launch_l2l(int P, DevCells C, const int *cells, int ncell, double2 *L, hipStream_t s);
// L2P for every body (laplace.h:359-388); accumulates into the targets
hipError_t launch_l2p(int P, DevBodies B, DevCells C, const int *body_leaf, int n,
                      const double2 *L, hipStream_t s);
// Target-tile M2L (fmm_rot.hip, 2 <= P <= 12): tiles of m2l_tile_targets(P)
// targets, slices of at most kM2LSlicePairs pairs of one offset class, one
// wavefront per work item of a tile.  ops: every class's record
// (rot_ops_bytes(P) each) from its offset with non-negative components.  A
// tile in one item stores its targets' L, a split tile adds into L (which
// must start at zero).
bool rot_supported(int P);
int m2l_tile_targets(int P);
constexpr int kM2LSlicePairs = 4;
size_t rot_ops_bytes(int P);
hipError_t init_rot_constants();
hipError_t launch_rot_ops(int P, int kind, const double *cdx, int nrep, void *ops, hipStream_t s);
hipError_t launch_m2l_rot(int P, int nitem, const int *ttgt, const int4 *items, const int4 *slices, const int *psrc,
                          const unsigned short *plt, const void *ops, const double2 *M, double2 *L, hipStream_t s);
// M2M and L2L of one level the same way, on one record of the level's child
// offset (h, h, h) (launch_rot_ops kind 1 M2M, 2 L2L; kind 0 M2L).  child8[8 i +
// octant]: children of parents[i] (-1: none); kids[k] = {child, parent | octant << 27}
hipError_t launch_m2m_rot(int P, const int *parents, const int *child8, int np, const void *rec, double2 *M,
                          hipStream_t s);
hipError_t launch_l2l_rot(int P, const int2 *kids, int nk, const void *rec, double2 *L, hipStream_t s);
// periodic far images, one level of supercells of period cyc: T = sum of its
// M2L operators, S = I + its M2M operators (dense P^2 x P^2, row-major; S may be
// null); prange <= kFarMaxRange; sums: far_sums_bytes(P) of scratch
constexpr int kFarMaxRange = 17;
size_t far_sums_bytes(int P);
hipError_t launch_far_ops(int P, int prange, double3 cyc, void *sums, double *T, double *S, hipStream_t s);
hipError_t launch_matmul(const double *A, const double *B, double *C, int n, int acc, hipStream_t s);
hipError_t launch_periodic_far(int P, const double *F, const double2 *M, double2 *L, hipStream_t s);
// mixed precision (FP32 list phases): M32 = M~ / R^n per cell; grouped FP32-MFMA
// M2L with per-group scales (R_s, R_t) accumulating into the FP64 L; FP32 P2P
bool m2l_mixed_supported(int P);
hipError_t launch_m_to_f32(int P, const double2 *M, const double *R, int ncell, float2 *M32, hipStream_t s);
hipError_t launch_m2l_mfma32(int P, const int4 *chunks, int nchunk, const double *gdx, const double2 *gscale,
                             const int *ptgt, const int *psrc, const float2 *M32, double2 *L, hipStream_t s);
// P2P for every target leaf over its CSR list (laplace.h:150-235); overwrites
// the targets of each listed leaf.  targets: wide leaves (at least kP2PWideLeaf
// bodies, run with four targets per lane, the rest with one) of systems with
// less than kP2PFillLeaves targets, then of larger ones, then the rest likewise
constexpr int kP2PWideLeaf = 16;
struct P2PCounts {
  int wide_few = 0, wide_many = 0, few = 0, many = 0;
};
hipError_t launch_p2p32(DevBodies B, DevCells C, const int *targets, P2PCounts n, const int *ptr,
                        const int *src, double3 xper, double eps2, int mask_all, hipStream_t s);
hipError_t launch_p2p(DevBodies B, DevCells C, const int *targets, P2PCounts n, const int *ptr,
                      const int *src, double3 xper, double eps2, int mask_all, hipStream_t s);

// Direct sum (include/traversal.h:355-377) of all n sources at nt targets
// (SoA txyz); writes tpot/tax/tay/taz.
// getDipole + dipoleCorrection on the bodies' targets; part: 3 * dipole_partials(n) doubles
int dipole_partials(int n);
hipError_t launch_dipole_correction(DevBodies B, int n, double *part, double coef, hipStream_t s);
// Ewald sum (include/ewald.h): bodies with positions x[i*xs], y[i*xs],
// z[i*xs] (each wrapped once into the box as it is read), charges q[i]; the
// results are added into pot[i] and ax/ay/az[i*fs]
struct EwBodies {
  const double *x, *y, *z, *q;
  double *pot, *ax, *ay, *az;
  int xs, fs;
};
// number of wave vectors of Ewald::initWaves for ksize
int ewald_nwaves(int ksize);
// wave part over the ewald_nwaves(ksize) wave vectors (table kv: 3 ints each,
// S: one double2 each, both written here), real part over minimum-image pairs
// within the cutoff, self term
hipError_t launch_ewald(EwBodies B, int n, int ksize, int *kv, double2 *S, double3 cyc, double alpha,
                        double sigma, double cutoff, hipStream_t s);
// The same on the device's static scratch array (no allocation): ksize up to
// kEwaldScratchMaxK; init_scratch(device) must have run once with that device
// current.  Calls that overlap on one device share the array and race.
constexpr int kMaxDevices = 64;
constexpr int kEwaldScratchMaxK = 32;
hipError_t init_scratch(int device);
// Scratch of the plan builders (device tree, lists, groups), cached per
// stream: a block given back on stream s is handed to a later request on s
// (the stream's order makes the reuse safe), the smallest cached block that
// fits and is at most twice the request plus 1 MiB, else a new hipMalloc'd
// one (current device).  A stream keeps at most 12 GiB cached (a block beyond
// that is freed: with 8 the 60M M2L pairs of 8M bodies, whose pair arrays change
// places with cached ones, took 53 ms to set in place of 50); plan_scratch_release(s) frees the stream's blocks after
// its work (the owner calls it before destroying s).  Replaces a
// hipMallocAsync / hipFreeAsync pair per buffer, about 0.2 ms of host time
// each on this runtime.
// (spare: a new block gets that much more, where there is room)
hipError_t plan_scratch_get(void **p, size_t *cap, size_t bytes, hipStream_t s, size_t spare = 0);
void plan_scratch_put(void *p, size_t cap, hipStream_t s);
void plan_scratch_release(hipStream_t s);
// hipMalloc on the current device; out of memory, the blocks cached for any
// stream are given back and it is tried once more (*p null after a failure)
hipError_t device_alloc(void **p, size_t bytes);
// One device allocation (hipMalloc on `device`), freed on that device when
// its owner goes; move-only.  With a pool it is taken from and given back to
// that stream's cached blocks.
struct DevArray {
  void *p = nullptr;
  size_t bytes = 0;  // in use
  size_t cap = 0;    // allocated
  int device = -1;
  hipStream_t pool = nullptr;
  DevArray() = default;
  DevArray(const DevArray &) = delete;
  DevArray &operator=(const DevArray &) = delete;
  ~DevArray() { reset(); }
  hipError_t alloc(size_t b, int dev);  // keeps an allocation that is large enough; the device must be current
  void reset();
  template <class T> T *as() const { return static_cast<T *>(p); }
};
// The large arrays of a plan built on the device, left there for the upload
// into a context on the same device: the lists' source columns (the host
// Lists keep the row pointers and counts, their m2l_src and p2p_src stay
// empty) and the M2L tiles' slices, pair sources and pair targets (the host
// M2LTiles keep the tiles, items and target cells).  Written on the
// builder's stream, complete when the build returns.
struct PlanArrays {
  int device = -1;
  bool lists = false, tiles = false;
  DevArray m2l_src, p2p_src;    // int per pair
  DevArray t_slice, t_src, t_lt;  // 4 ints per slice, int and uint16 per pair
  int64_t nslice = 0;
};
// Copy the device-held parts into the host structures (synchronous on s).
hipError_t fetch_lists(const PlanArrays &d, fmm::Lists &L, hipStream_t s);
hipError_t fetch_tiles(const PlanArrays &d, fmm::M2LTiles &T, hipStream_t s);
// The M2L groups and tiles of a regular tree (cycle: of periodic lists) built on the device
// (fmm_tiles.hip): the same partition into groups and classes as
// fmm::build_m2l_groups (numbered in key order), the same tiles, slices and
// work items as fmm::build_m2l_tiles; done = false (no error) when the plan
// does not fit (the caller then builds them on the host).  Only the fields
// the tile path reads are filled (no chunks).  With keep, the pair sources
// are read from keep->m2l_src when keep->lists (else from L.m2l_src), and
// the tiles' slices, pair sources and pair targets are left in keep instead
// of T (keep->tiles).  dsrc_in: the lists' source column already on the
// device (stream s), read instead of L.m2l_src.
hipError_t device_groups_tiles(const fmm::Tree &t, const fmm::Lists &L, int TT, int SW, int seg,
                               fmm::M2LGroups &G, fmm::M2LTiles &T, bool &done, hipStream_t s,
                               PlanArrays *keep = nullptr, const int *dsrc_in = nullptr,
                               const double *cycle = nullptr);
// The octree of n bodies (host array x, AoS) built on the device: the same
// cells, numbering and body order as fmm::build_tree for the root box (X0,
// R0) (fmm_traverse.hip); outputs are host arrays.  dx_in: the same bodies
// already on the device (then x is not read), written on stream s.
hipError_t device_tree(int n, const double *x, int ncrit, const double X0[3], double R0, std::vector<int> &perm,
                       std::vector<int> &iparent, std::vector<int> &ichild, std::vector<int> &nchild,
                       std::vector<int> &ibody, std::vector<int> &nbody, std::vector<int> &level,
                       std::vector<double> &X, std::vector<double> &R, hipStream_t s,
                       const double *dx_in = nullptr);
// The interaction lists of a free-space tree built on the device (the dual
// traversal breadth first, fmm_traverse.hip): CSR lists sorted by (target,
// source), the P2P body-pair count; the cell arrays are host arrays.  With
// keep, the source columns stay on the device in keep->m2l_src and
// keep->p2p_src (keep->lists) and m2l_src, p2p_src are left empty.
hipError_t device_lists(int ncell, const double *X, const double *R, const int *nchild, const int *ichild,
                        const int *nbody, double theta, int nspawn, const double xper[3], int root_i, int root_j,
                        std::vector<int> &m2l_ptr, std::vector<int> &m2l_src, std::vector<int> &p2p_ptr,
                        std::vector<int> &p2p_src, int64_t &body_pairs, hipStream_t s,
                        PlanArrays *keep = nullptr);
// The interaction lists of a tree with the host walker's order
// (fmm::build_lists of the root with itself), the source columns copied to
// the device arrays that dst gives for their lengths (m2l_src and p2p_src are
// left empty); done = false (no error) when the host has to walk the tree.
hipError_t device_visit_lists(const fmm::Tree &t, double theta, int nspawn, int images, const double *cycle,
                              fmm::Lists &L, const std::function<int *(bool p2p, int64_t n)> &dst, bool &done,
                              hipStream_t s);
hipError_t launch_ewald_scratch(int device, EwBodies B, int n, int ksize, double3 cyc, double alpha, double sigma,
                                double cutoff, hipStream_t s);
// part: 4 nt direct_runs(n, nt) doubles (not read when that is one run), out: [4][nt]
int direct_runs(int n, int nt);
hipError_t launch_direct(DevBodies B, int n, const double *tx, const double *ty, const double *tz, int nt,
                         double *part, double *out, double eps2, int prange, double3 cyc, hipStream_t s);

}  // namespace fmmdev
