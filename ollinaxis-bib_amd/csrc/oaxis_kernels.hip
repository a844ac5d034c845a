// HIP kernels of the evolution hot path (gfx950, FP64 throughout).
//
// One launch of k_rhs_table (or k_rhs_phases) performs, for every point of a level, what the
// reference does in one internal iteration of onestep.f90:129-342:
//   the derivative stencils and algebra of auxiliary_geometry.f90,
//   sources_geometry/lapse/shift/scalar, Kreiss-Oliger dissipation,
//   radiative boundaries on level 0, RK4 accumulate / update,
//   the axis (and equator) parity images, and the pointwise part of the
//   next auxiliary call (factordet, phi/chi, KT_H / lambda are implicit).
// The state stays projected in memory, as in the reference.
//
// Layout: a level holds each evolved field as one z-fastest plane; point
// (i, j) of the reference's (1-g:Nr, 1-g:Nz) range sits at
// (i+g-1)*ld + (j+g-1).  Ghost columns i <= 0 (axis) and, with equatorial
// symmetry, ghost rows j <= 0 are stored and kept equal to the parity images
// of the interior, so every centred stencil reads them directly.
#include <hip/hip_runtime.h>

#include <cmath>
#include <mutex>
#include <string>

#include "oa_internal.h"

#define OA_HD __device__ __forceinline__
#define OA_HHD __host__ __device__ inline
#include "oaxis_device.h"
#include "oaxis_rhs.h"

namespace oax {

#define RC_K(call)                \
  do {                            \
    const int rc_ = (call);       \
    if (rc_ != OA_OK) return rc_; \
  } while (0)

// ------------------------------------------------------------ RHS kernel
// Each block stages a 16 x 16 tile of every field, with a 3-point halo, in
// LDS and reads all stencils from there.  Centred stencils reach 3 points.
// The one-sided closures at i = Nr-1..Nr, j = Nz-1..Nz and (without
// equatorial symmetry) j = 1-ghost..2-ghost reach up to 5 points, always
// towards the interior; the first and the last tile of each direction are
// anchored to the ends of the computed range, so those reads stay inside the
// tile.  The last tile of a direction may overlap the one before it; its
// points already covered there are skipped (the RK accumulator is
// read-modify-write).
constexpr int kTile = 16, kHalo = 3;
constexpr int kTileW = kTile + 2 * kHalo;                 // staged extent per direction
constexpr int kTileSize = kTileW * kTileW;                // values per field
constexpr int kRhsBlock = 512;                            // two waves per 64 points
constexpr int kResidentBlocks = 512;                      // RHS blocks resident at once (256 CUs x 2)

// first point of tile b of nb along [lo, hi] (extent >= kTile)
__host__ __device__ inline int tile_start(int b, int nb, int lo, int hi) {
  return (b < nb - 1) ? lo + b * kTile : hi - (kTile - 1);
}

// A tile wholly inside i in [1, Nr-3], j in [1, Nz-3]: every stencil there
// takes its centred form, so the closure branches compile out (IN).
__device__ __forceinline__ bool interior_tile(const KGrid& G, int i0, int j0) {
  return i0 >= 1 && i0 + kTile - 1 <= G.Nr - 3 && j0 >= 1 && j0 + kTile - 1 <= G.Nz - 3;
}

// Staging an RHS input tile into LDS: each of the first 484 threads owns one
// point of every staged plane, so its offset in a plane is worked out once.
// Points of the tile outside the level, which no stencil reads, take the
// value of the nearest point inside it, so that every load is in bounds and
// none needs a branch.
__device__ __forceinline__ long stage_offset(const KGrid& G, int ib, int jb, int tw, int q) {
  const int lo = 1 - G.g;
  const int ii = min(max(ib + q / tw, lo), G.Nr), jj = min(max(jb + q % tw, lo), G.Nz);
  return IDX(G, ii, jj);
}

// Stage NST planes, plane f from src(f), into tile slots first .. first +
// NST - 1.  Every load of the batch is issued before the first LDS store, so
// their latencies overlap instead of adding up (a load-wait-store loop per
// plane waits out one memory round trip per plane and point).
template <int NST, class Src>
__device__ __forceinline__ void stage_planes(double* tile, int first, int q, long off, Src src) {
  double v[NST];
#pragma unroll
  for (int f = 0; f < NST; ++f) v[f] = src(f)[off];
#pragma unroll
  for (int f = 0; f < NST; ++f) tile[(first + f) * kTileSize + q] = v[f];
}

// Pointers read from a work item are generic; every one of them addresses
// device (global) memory and is uniform across the block.  Passing each
// through the global address space, behind an empty asm so the two casts do
// not fold away, lets the compiler emit global loads and stores instead of
// flat ones (flat accesses also count against the LDS wait counter, so every
// LDS wait would also wait for outstanding global traffic).
template <class T>
__device__ __forceinline__ T* gmem(T* p) {
  __attribute__((address_space(1))) T* g = (__attribute__((address_space(1))) T*)p;
  asm volatile("" : "+s"(g));
  return (T*)g;
}

// The tile address a thread's stencils are read relative to: its point's
// value, kHalo rows and columns back (di, dj: the point's position in the
// staged tile).  The centred stencils then reach offsets 0 .. 6 rows and
// columns from it, all non-negative, so every read is one LDS instruction
// with an immediate offset; the empty asm keeps the compiler from splitting
// the address back into a tile base and a signed per-read offset.
__device__ __forceinline__ const double* corner_of(const double* tile, int di, int dj) {
  auto l = (__attribute__((address_space(3))) const double*)(tile + (di - kHalo) * kTileW + (dj - kHalo));
  asm volatile("" : "+v"(l));
  return (const double*)l;
}

// the item of block b in a table launch: the last one whose block0 (STRIP:
// strip0) <= b (they ascend; the loads are uniform across the block)
template <bool STRIP = false, class Item>
__device__ __forceinline__ const Item& find_item(const Item* __restrict__ items, int n, int b) {
  int lo = 0, hi = n - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    int first;
    if constexpr (STRIP) first = items[mid].strip0;
    else first = items[mid].block0;
    if (first <= b) lo = mid;
    else hi = mid - 1;
  }
  return items[lo];
}

// the 1/r table of a tile's columns, in LDS after its planes
constexpr int kInvR = 72;
__device__ __forceinline__ void stage_inv_r(const KGrid& G, double* rinv, int ib, int q) {
  if (q < kInvR) rinv[q] = 1.0 / ((static_cast<double>(ib + q) - 0.5) * G.dr);
}

// The boundary work that rides on a substep's launch, in units of one wave:
// 64 records of one field group of finebound, or 64 points of one field's
// strips of saveold.  Finebound reads the coarse level, the step's start at
// its own points and the strips of time level t-1, and writes only the zone,
// which the substep leaves alone; on the last substep, whose output is the
// step's start, each of its groups reads only what it overwrites itself
// (finebound_point).  Saveold rides on the first substep, whose output is never
// the step's start that it reads.  So both run beside the tiles, and a level
// step is one launch per substep instead of two and a saveold (each a few us
// that leave most of the GPU idle).
__device__ __forceinline__ int edge_fb_units(long n, int groups) { return groups * static_cast<int>((n + 63) / 64); }

template <bool SHIFT, bool SCALAR>
__device__ __forceinline__ void edge_work(const RhsItem& it, int v, int nv) {
  constexpr int groups = finebound_groups(SHIFT, SCALAR), nf = nslots(SHIFT, SCALAR);
  const KGrid& G = it.G;
  const int lane = static_cast<int>(threadIdx.x & 63u);
  const long n = it.E.n;
  const int ufb = edge_fb_units(n, groups), chunks = static_cast<int>((n + 63) / 64);
  const int nrt = G.Nr + G.g, nzt = G.Nz + G.g, per = G.g * max(nrt, nzt), schunks = (per + 63) / 64;
  const int usave = it.E.rR ? nf * schunks : 0;
  for (int u = v; u < ufb + usave; u += nv) {
    if (u < ufb) {
      const int grp = u / chunks;
      const long q = static_cast<long>(u % chunks) * 64 + lane;
      if (q >= n) continue;
      const double* const yp = gmem(it.yp);
      const FbPoint* const rec = gmem(it.E.table) + q;
      const long k = IDX(G, rec->i, rec->j);
      finebound_point<SHIFT, SCALAR>(G, it.E.Gc, it.P, it.E.T, it.E.time0, gmem(it.E.yc), gmem(it.yout),
                                     gmem(it.E.rR1), gmem(it.E.zL1), gmem(it.E.zR1), *rec, grp,
                                     [&](int s) { return yp[s * G.plane + k]; });
    } else {
      const int s = u - ufb, f = s / schunks, q = (s % schunks) * 64 + lane;
      if (q < per) saveold_point(G, gmem(it.yp), gmem(it.E.rR), gmem(it.E.zL), gmem(it.E.zR), f, q);
    }
  }
}

// this wave's share of the edge work of an item with nt tiles: block t of its
// nt + xtra, wave w of W; its own blocks come first, then wave after wave of
// the tiles' blocks
template <bool SHIFT, bool SCALAR>
__device__ __forceinline__ void edge_share(const RhsItem& it, int nt, int t, int w, int W) {
  if (it.E.n == 0 && !it.E.rR) return;
  const int v = t >= nt ? (t - nt) * W + w : it.xtra * W + w * nt + t;
  edge_work<SHIFT, SCALAR>(it, __builtin_amdgcn_readfirstlane(v), (nt + it.xtra) * W);
}

// the point is left to finebound (depth < 0: none is)
__device__ __forceinline__ bool finebound_zone(const KGrid& G, int depth, int i, int j) {
  return depth >= 0 && (i >= G.Nr - depth || j >= G.Nz - depth || (!G.eqsym && j <= 1 - G.g + depth));
}

// One RK substep of a level.  A block stages its tile once and eight waves
// work on it: waves 0-3 form one half of the sources of the tile's points,
// waves 4-7 the other half (rhs_roles), so the LDS of a tile serves twice the
// waves that one thread per point would give.  The halves are about equal in
// instructions per point.
template <bool SHIFT, bool SCALAR>
constexpr int kRole0 = ROLE_K | (SHIFT && SCALAR ? ROLE_SCALAR : SHIFT || SCALAR ? ROLE_LAPSE : 0);
template <bool SHIFT, bool SCALAR>
constexpr int kRole1 = (ROLE_DELTA | ROLE_LAPSE | ROLE_METRIC | ROLE_SCALAR) & ~kRole0<SHIFT, SCALAR>;

// What a block computes: the 16 x 16 tiles of the item's range, or a strip of
// the frame around it, the outer 3 rows where some stencils are one-sided:
//   rho strips  i = Nr-2 .. Nr, 64 points along z; wave w holds row Nr-2+w
//   z strips    j = Nz-2 .. Nz or j = 1-ghost .. 3-ghost, 62 points along
//               rho with i <= Nr-3; wave w holds one j
// so a wave's points share their distance from the edge and take one branch
// of every closure.  (In square tiles along the edges, each wave ran most
// branches, three to four times the work of a tile inside.)  Strips stage 6
// rows or columns: the closures reach 5 points inward.
constexpr int kStripR = 64, kStripZ = 62;
constexpr int kStripRW = kStripR + 2 * kHalo, kStripZW = 7;
static_assert(6 * kStripRW <= kTileSize && (kStripZ + 2 * kHalo) * kStripZW <= kTileSize, "a strip fits the tile's LDS");
static_assert(kStripZ + 2 * kHalo <= kInvR && kTileW <= kInvR, "1/r table");

template <bool SHIFT, bool SCALAR, bool PHIMODE>
__device__ __forceinline__ void rhs_block(const RhsItem& it, bool strip, int t, double* tile) {
  constexpr int nf = nslots(SHIFT, SCALAR);
  const KGrid& G = it.G;
  KStep S = it.S;
  S.dtb_pre = gmem(S.dtb_pre);            // null stays null
  const int tid = static_cast<int>(threadIdx.x);
  const int lane = tid & 63, w = (tid >> 6) & 3;
  int ib, jb, tw = kTileW, size = kTileSize;   // staged corner, pitch and values
  int i, j;                                    // this thread's point
  bool mine = true, inside = false;
  if (strip) {
    if (t < it.nstr) {
      const int js = (t > 0 && t == it.nstr - 1) ? G.Nz - (kStripR - 1) : G.jlo + t * kStripR;
      ib = G.Nr - 5;
      jb = js - kHalo;
      tw = kStripRW;
      size = 6 * kStripRW;
      i = G.Nr - 2 + w;
      j = js + lane;
      mine = w < 3 && j <= G.Nz && !(t == it.nstr - 1 && j < G.jlo + t * kStripR);
    } else {
      const int q = t - it.nstr, side = q / it.nstz, is = 1 + (q % it.nstz) * kStripZ;
      ib = is - kHalo;
      jb = side == 0 ? G.Nz - 5 : G.jlo;
      tw = kStripZW;
      size = (kStripZ + 2 * kHalo) * kStripZW;
      i = is + lane;
      j = (side == 0 ? G.Nz - 2 : G.jlo) + w;
      mine = w < 3 && lane < kStripZ && i <= G.Nr - 3;
    }
  } else if (t >= it.nbi * it.nbj) {
    edge_share<SHIFT, SCALAR>(it, it.nbi * it.nbj, t, tid >> 6, kRhsBlock / 64);
    return;
  } else {
    const int bi = t / it.nbj, bj = t % it.nbj;
    const int i0 = tile_start(bi, it.nbi, 1, it.ihi), j0 = tile_start(bj, it.nbj, it.jlo, it.jhi);
    ib = i0 - kHalo;
    jb = j0 - kHalo;
    i = i0 + 4 * w + lane / kTile;
    j = j0 + lane % kTile;
    inside = interior_tile(G, i0, j0);
    // points of the last tile that the tile before it covers
    mine = !(bi == it.nbi - 1 && i < 1 + bi * kTile) && !(bj == it.nbj - 1 && j < it.jlo + bj * kTile) &&
           !finebound_zone(G, it.depth, i, j);
  }
  // the evolved fields, then (first substep only) the dtbeta planes it
  // differentiates, then the 1/r table
  const double* __restrict__ yin = gmem(it.yin);
  double* const rinv = tile + (nf + (SHIFT && S.dtb_pre ? 2 : 0)) * kTileSize;
  if (tid < size) {
    const long off = stage_offset(G, ib, jb, tw, tid);
    stage_planes<nf>(tile, 0, tid, off, [&](int f) { return yin + f * G.plane; });
    if (SHIFT && S.dtb_pre) stage_planes<2>(tile, nf, tid, off, [&](int f) { return S.dtb_pre + f * G.plane; });
  }
  stage_inv_r(G, rinv, ib, tid);
  __syncthreads();
  const bool second = __builtin_amdgcn_readfirstlane(tid >> 8) != 0;
  if (mine) {
    const double* const yp = gmem(it.yp);
    double* const acc = gmem(it.acc);
    double* const yout = gmem(it.yout);
    constexpr int R0 = kRole0<SHIFT, SCALAR>, R1 = kRole1<SHIFT, SCALAR>;
    constexpr int ndtb = SHIFT ? shift_slot(SH_dtbeta_r) : 0;
    const double* const ri = rinv + (i - ib);
    if (inside) {
      const RoleView V{corner_of(tile, i - ib, j - jb), i - kHalo, j - kHalo, kTileW, kTileSize, ri, ndtb, nf};
      if (!second) rhs_roles<SHIFT, SCALAR, PHIMODE, true, R0>(G, it.P, S, it.W, V, yp, acc, yout, i, j);
      else rhs_roles<SHIFT, SCALAR, PHIMODE, true, R1>(G, it.P, S, it.W, V, yp, acc, yout, i, j);
    } else {
      const RoleView V{tile + (i - ib) * tw + (j - jb), i, j, tw, kTileSize, ri, ndtb, nf};
      if (!second) rhs_roles<SHIFT, SCALAR, PHIMODE, false, R0>(G, it.P, S, it.W, V, yp, acc, yout, i, j);
      else rhs_roles<SHIFT, SCALAR, PHIMODE, false, R1>(G, it.P, S, it.W, V, yp, acc, yout, i, j);
    }
  }
  if (!strip) edge_share<SHIFT, SCALAR>(it, it.nbi * it.nbj, t, 7 - (tid >> 6), kRhsBlock / 64);
}

// Workgroups are dispatched to the 8 XCDs round robin (block b to XCD b % 8),
// and each XCD has its own L2.  Renumbering the blocks so that every XCD
// receives one contiguous range of tiles keeps neighbouring tiles, whose
// halos overlap, in the same L2.  A bijection of [0, total).
constexpr int kXcds = 8;
__device__ __forceinline__ int xcd_block(int b, int total) {
  const int q = total / kXcds, r = total % kXcds;
  const int x = b % kXcds, l = b / kXcds;
  return x * q + (x < r ? x : r) + l;
}

// The first `strips` blocks are the items' frame strips, which take longer than
// a tile inside: they start first and are spread over the XCDs.  Four waves on a
// SIMD hide the stencils' LDS latency, which bounded the sources in two phases
// of four waves: 512 x 1024 in vacuum 80.4 -> 55 us a launch (its bytes take 44
// at the rate of a large copy); a fine level of 128 x 256 with Gamma-driver and
// scalar field 17 us with its finebound, 20 with its saveold too, which were
// launches of their own.
template <bool SHIFT, bool SCALAR, bool PHIMODE>
__global__ void __launch_bounds__(kRhsBlock, 4) k_rhs_table(const RhsItem* __restrict__ items, int n, int strips,
                                                            int xcd_remap) {
  extern __shared__ double tile[];
  const int b = static_cast<int>(blockIdx.x);
  const bool strip = b < strips;
  int t = b;
  if (!strip) {
    t = b - strips;
    if (xcd_remap) t = xcd_block(t, static_cast<int>(gridDim.x) - strips);
  }
  const RhsItem& it = strip ? find_item<true>(items, n, t) : find_item<false>(items, n, t);
  rhs_block<SHIFT, SCALAR, PHIMODE>(it, strip, t - (strip ? it.strip0 : it.block0), tile);
}

// The tile points of a block of 256 threads: each owns q0 = tid and q1 = tid
// + 256 of the tile's 484.
struct PhaseSlots {
  long o0, o1;          // plane offsets of the two points
  int q0, q1;           // their tile positions
  bool two;             // q1 lies inside the tile
};

__device__ __forceinline__ PhaseSlots phase_slots(const KGrid& G, int ib, int jb) {
  PhaseSlots s;
  const int tid = static_cast<int>(threadIdx.y * blockDim.x + threadIdx.x);
  const int lo = 1 - G.g;
  s.q0 = tid;
  s.q1 = tid + kTile * kTile;
  s.two = s.q1 < kTileSize;
  auto offset = [&](int q) {
    const int ii = min(max(ib + q / kTileW, lo), G.Nr), jj = min(max(jb + q % kTileW, lo), G.Nz);
    return IDX(G, ii, jj);
  };
  s.o0 = offset(s.q0);
  s.o1 = s.two ? offset(s.q1) : s.o0;
  return s;
}

// the same staging with two points per thread
template <int NST, class Src>
__device__ __forceinline__ void stage_planes(double* tile, int first, const PhaseSlots& s, Src src) {
  double v0[NST], v1[NST];
#pragma unroll
  for (int f = 0; f < NST; ++f) {
    const double* __restrict__ p = src(f);
    v0[f] = p[s.o0];
    v1[f] = p[s.o1];
  }
#pragma unroll
  for (int f = 0; f < NST; ++f) {
    double* dst = tile + (first + f) * kTileSize;
    dst[s.q0] = v0[f];
    if (s.two) dst[s.q1] = v1[f];
  }
}

// Whether the point lies in an interior tile of the level's whole tile grid.
// The two forms of phase 1 contract their sums differently, so a point keeps
// one form whichever range of the level an item computes.
__device__ __forceinline__ bool interior_point(const KGrid& G, int i, int j) {
  const int nbi = (G.Nr + kTile - 1) / kTile, nbj = (G.Nz - G.jlo + kTile) / kTile;
  const int bi = min((i - 1) / kTile, nbi - 1), bj = min((j - G.jlo) / kTile, nbj - 1);
  return interior_tile(G, tile_start(bi, nbi, 1, G.Nr), tile_start(bj, nbj, G.jlo, G.Nz));
}

// The Gamma-driver in vacuum: one thread per point in two phases.  Phase 1
// forms the geometric auxiliaries (the Ricci tensor and div KT: the longest
// expressions, which need only the vacuum fields) and passes them through the
// per-level buffer gaux; phase 2 forms D_i D_j alpha, every source, the
// dissipation, the radiative boundaries and the RK update.  Kept apart, the
// phases need at most the registers of the larger one: 242 VGPRs, two waves
// per SIMD, and the staged tile (17 fields, 66 KB) allows two blocks per CU.
//
// The form by parts would be faster here too, and nothing shows it less accurate.
// But other sums have other last bits, and the constraints of such data, residuals
// that amplify the last bit of the state by 1/h^2, move with them by 1e-10 to 3e-9
// of their size.  That this configuration keeps its bits is a choice.
template <bool PHIMODE>
__device__ __forceinline__ void rhs_phases_tile(const RhsItem& it, int t, double* tile) {
  constexpr int nf = nslots(true, false);
  const KGrid& G = it.G;
  const int nt = it.nbi * it.nbj, wave = static_cast<int>(threadIdx.x >> 6);
  if (t >= nt) {
    edge_share<true, false>(it, nt, t, wave, kTile * kTile / 64);
    return;
  }
  const int bi = t / it.nbj, bj = t % it.nbj;
  const int ti = static_cast<int>(threadIdx.x) / kTile, tj = static_cast<int>(threadIdx.x) % kTile;
  KStep S = it.S;
  S.dtb_pre = gmem(S.dtb_pre);            // null stays null
  const int nbj = it.nbj, nbi = it.nbi;
  const int j0 = tile_start(bj, nbj, it.jlo, it.jhi);
  const int i0 = tile_start(bi, nbi, 1, it.ihi);
  const int ib = i0 - kHalo, jb = j0 - kHalo;
  if (it.skip && i0 + kTile - 1 <= it.sihi && j0 >= it.sjlo && j0 + kTile - 1 <= it.sjhi) return;
  // the evolved fields, then (first substep only) the dtbeta planes it differentiates
  const double* __restrict__ yin = gmem(it.yin);
  double* const gaux = gmem(it.gaux);
  {
    const PhaseSlots ss = phase_slots(G, ib, jb);
    stage_planes<nf>(tile, 0, ss, [&](int f) { return yin + f * G.plane; });
    if (S.dtb_pre) stage_planes<2>(tile, nf, ss, [&](int f) { return S.dtb_pre + f * G.plane; });
    __syncthreads();
  }
  const int i = i0 + ti, j = j0 + tj;
  // not the points done by the tile before, outside the item's frame or left
  // to finebound
  if (!(bi == nbi - 1 && i < 1 + (nbi - 1) * kTile) && !(bj == nbj - 1 && j < it.jlo + (nbj - 1) * kTile) &&
      !(it.skip && i <= it.sihi && j >= it.sjlo && j <= it.sjhi) && !finebound_zone(G, it.depth, i, j)) {
    const TileView V{corner_of(tile, i - ib, j - jb), i - kHalo, j - kHalo, kTileW, kTileSize, nf};
    // phase 1: the geometric auxiliaries of this point, through gaux (own point
    // only, so no synchronisation); the memory barrier keeps the compiler from
    // carrying phase-1 values or loads into phase 2, so the two phases do not
    // add up in registers
    if (interior_point(G, i, j))
      rhs_point<false, PHIMODE, true, 1>(G, it.P, S, V, nullptr, nullptr, nullptr, gaux, i, j);
    else
      rhs_point<false, PHIMODE, false, 1>(G, it.P, S, V, nullptr, nullptr, nullptr, gaux, i, j);
    asm volatile("" ::: "memory");
    rhs_point<true, PHIMODE, false, 2>(G, it.P, S, V, gmem(it.yp), gmem(it.acc), gmem(it.yout), gaux, i, j);
  }
  edge_share<true, false>(it, nt, t, wave, kTile * kTile / 64);
}

// Two waves on a SIMD, bound by the latency of its LDS reads (half of a wave's
// life is waits).  A level of 256 x 512 with its finebound and saveold takes 39
// us; over all rows, without them, it took 62.
template <bool PHIMODE>
__global__ void __launch_bounds__(kTile * kTile, 2) k_rhs_phases(const RhsItem* __restrict__ items, int n,
                                                                 int xcd_remap) {
  extern __shared__ double tile[];
  const int b = xcd_remap ? xcd_block(static_cast<int>(blockIdx.x), static_cast<int>(gridDim.x))
                          : static_cast<int>(blockIdx.x);
  const RhsItem& it = find_item(items, n, b);
  const int t = b - it.block0;
  rhs_phases_tile<PHIMODE>(it, t, tile);
}

// ------------------------------------------------------ constraints
// The geometric auxiliaries of the current state (phase 1 of the two-phase
// kernel alone, on the vacuum fields), for the constraints.
template <bool PHIMODE>
__global__ void __launch_bounds__(kTile * kTile, 2) k_aux(RhsItem it) {
  extern __shared__ double tile[];
  const KGrid& G = it.G;
  const int bi = static_cast<int>(blockIdx.y), bj = static_cast<int>(blockIdx.x);
  const int j0 = tile_start(bj, it.nbj, G.jlo, G.Nz);
  const int i0 = tile_start(bi, it.nbi, 1, G.Nr);
  const int ib = i0 - kHalo, jb = j0 - kHalo;
  const double* __restrict__ yin = it.yin;
  stage_planes<NBASE>(tile, 0, phase_slots(G, ib, jb), [&](int f) { return yin + f * G.plane; });
  __syncthreads();
  const int i = i0 + static_cast<int>(threadIdx.y), j = j0 + static_cast<int>(threadIdx.x);
  if (bi == it.nbi - 1 && i < 1 + (it.nbi - 1) * kTile) return;     // done by the tile before
  if (bj == it.nbj - 1 && j < G.jlo + (it.nbj - 1) * kTile) return;
  const TileView V{corner_of(tile, i - ib, j - jb), i - kHalo, j - kHalo, kTileW, kTileSize, NBASE};
  if (interior_tile(G, i0, j0))
    rhs_point<false, PHIMODE, true, 1>(G, it.P, it.S, V, nullptr, nullptr, nullptr, it.gaux, i, j);
  else
    rhs_point<false, PHIMODE, false, 1>(G, it.P, it.S, V, nullptr, nullptr, nullptr, it.gaux, i, j);
}

struct ConsArgs {
  KGrid G; KPhys P; int sc0;
  const double* y; const double* gaux; double* out;
};

template <bool PHIMODE, bool SCALAR>
__global__ void __launch_bounds__(256) k_constraints(ConsArgs c) {
  const int j = c.G.jlo + static_cast<int>(blockIdx.x * blockDim.x + threadIdx.x);
  const int i = 1 + static_cast<int>(blockIdx.y * blockDim.y + threadIdx.y);
  if (j > c.G.Nz || i > c.G.Nr) return;
  constraints_point<PHIMODE, SCALAR>(c.G, c.P, c.sc0, c.y, c.gaux, c.out, i, j);
}

// constraints.f90:68-93, in the reference's order: ham copied from the
// neighbouring row at i = 1-ghost, i = Nr, j = 1-ghost, j = Nz, then the
// axis images and (equatorial symmetry) the equator images.  One block;
// each step sees the previous one's writes.
__global__ void __launch_bounds__(256) k_ham_fix(KGrid G, double* __restrict__ ham) {
  const int t = static_cast<int>(threadIdx.x), nt = static_cast<int>(blockDim.x);
  const int g = G.g;
  for (int j = 1 - g + t; j <= G.Nz; j += nt) ham[IDX(G, 1 - g, j)] = ham[IDX(G, 2 - g, j)];
  __syncthreads();
  for (int j = 1 - g + t; j <= G.Nz; j += nt) ham[IDX(G, G.Nr, j)] = ham[IDX(G, G.Nr - 1, j)];
  __syncthreads();
  for (int i = 1 - g + t; i <= G.Nr; i += nt) ham[IDX(G, i, 1 - g)] = ham[IDX(G, i, 2 - g)];
  __syncthreads();
  for (int i = 1 - g + t; i <= G.Nr; i += nt) ham[IDX(G, i, G.Nz)] = ham[IDX(G, i, G.Nz - 1)];
  __syncthreads();
  for (int q = t; q < g * (G.Nz + g); q += nt) {
    const int i = 1 + q / (G.Nz + g), j = 1 - g + q % (G.Nz + g);
    ham[IDX(G, 1 - i, j)] = ham[IDX(G, i, j)];
  }
  __syncthreads();
  if (G.eqsym)
    for (int q = t; q < g * (G.Nr + g); q += nt) {
      const int j = 1 + q / (G.Nr + g), i = 1 - g + q % (G.Nr + g);
      ham[IDX(G, i, 1 - j)] = ham[IDX(G, i, j)];
    }
}

// ----------------------------------------------- pointwise kernels
// One thread per point (or record) of an item, 256 threads per block; q is
// the thread's index within its item.
constexpr int kPtBlock = 256;

__device__ __forceinline__ bool level_point(const KGrid& G, long q, int& i, int& j) {
  const int nj = G.Nz - G.jlo + 1;
  i = 1 + static_cast<int>(q / nj);
  j = G.jlo + static_cast<int>(q % nj);
  return i <= G.Nr;
}

template <bool SHIFT, bool SCALAR>
__device__ __forceinline__ void project_body(const ProjItem& it, long q) {
  int i, j;
  if (level_point(it.G, q, i, j)) project_point<SHIFT, SCALAR>(it.G, it.P, it.time0, gmem(it.y), i, j);
}

__device__ __forceinline__ void deldef_body(const DelItem& it, long q) {
  int i, j;
  if (level_point(it.G, q, i, j)) deldef_point(it.G, gmem(it.y), i, j);
}

// saveold for the fine-boundary strips: blocks of one field, then the next
__device__ __forceinline__ int save_per_field(const KGrid& G) {
  const int nrt = G.Nr + G.g, nzt = G.Nz + G.g;
  return G.g * (nrt > nzt ? nrt : nzt);
}
__device__ __forceinline__ void saveold_body(const SaveItem& it, int blk) {
  const int per = save_per_field(it.G);
  const int bpf = (per + kPtBlock - 1) / kPtBlock;
  const int f = blk / bpf;
  const int q = (blk % bpf) * kPtBlock + static_cast<int>(threadIdx.x);
  if (f < it.nf && q < per) saveold_point(it.G, gmem(it.y), gmem(it.rR), gmem(it.zL), gmem(it.zR), f, q);
}

// finebound: blocks of one field group, then the next (the group stays
// uniform within a block)
template <bool SHIFT, bool SCALAR>
__device__ __forceinline__ void finebound_body(const FbItem& it, int blk) {
  const int bpg = static_cast<int>((it.n + kPtBlock - 1) / kPtBlock);
  const int grp = blk / bpg;
  const long q = static_cast<long>(blk % bpg) * kPtBlock + threadIdx.x;
  if (grp >= finebound_groups(SHIFT, SCALAR) || q >= it.n) return;
  const FbPoint& rec = gmem(it.table)[q];
  // the strip of time level t0 this point belongs to
  const double *const r0 = gmem(it.rR0), *const zL0 = gmem(it.zL0), *const zR0 = gmem(it.zR0);
  const double* const s0 = (rec.which == 0) ? r0 : (rec.which == 1) ? zR0 : zL0;
  const long sper = static_cast<long>(it.Gf.g) * ((rec.which == 0) ? (it.Gf.Nz + it.Gf.g) : (it.Gf.Nr + it.Gf.g));
  const long sidx = rec.sidx;
  finebound_point<SHIFT, SCALAR>(it.Gf, it.Gc, it.P, it.T, it.time0, gmem(it.yc), gmem(it.yf), gmem(it.rR1),
                                 gmem(it.zL1), gmem(it.zR1), rec, grp,
                                 [&](int s) { return s0[s * sper + sidx]; });
}

// restrict: blocks of one field, then the next; one thread per coarse point
// of the item's box (the points of the coarse level the fine level may
// restrict onto; restrict_point tests each against the exact bounds)
__device__ __forceinline__ void restrict_body(const RsItem& it, int blk) {
  const long per = static_cast<long>(it.nic) * it.njc;
  const int bpf = static_cast<int>((per + kPtBlock - 1) / kPtBlock);
  const int s = blk / bpf;
  const long q = static_cast<long>(blk % bpf) * kPtBlock + threadIdx.x;
  if (s >= it.nf || q >= per) return;
  const int ic = it.ic0 + static_cast<int>(q / it.njc), jc = it.jc0 + static_cast<int>(q % it.njc);
  restrict_point(it.Gf, it.Gc, s, it.interporder, gmem(it.yf), gmem(it.yc), ic, jc);
}

template <bool SHIFT, bool SCALAR>
__global__ void __launch_bounds__(kPtBlock) k_project_table(const ProjItem* __restrict__ items, int n) {
  const ProjItem& it = find_item(items, n, static_cast<int>(blockIdx.x));
  project_body<SHIFT, SCALAR>(it, static_cast<long>(blockIdx.x - it.block0) * kPtBlock + threadIdx.x);
}

__global__ void __launch_bounds__(kPtBlock) k_deldef_table(const DelItem* __restrict__ items, int n) {
  const DelItem& it = find_item(items, n, static_cast<int>(blockIdx.x));
  deldef_body(it, static_cast<long>(blockIdx.x - it.block0) * kPtBlock + threadIdx.x);
}

__global__ void __launch_bounds__(kPtBlock) k_saveold_table(const SaveItem* __restrict__ items, int n) {
  const SaveItem& it = find_item(items, n, static_cast<int>(blockIdx.x));
  saveold_body(it, static_cast<int>(blockIdx.x) - it.block0);
}

template <bool SHIFT, bool SCALAR>
__global__ void __launch_bounds__(kPtBlock) k_finebound_table(const FbItem* __restrict__ items, int n) {
  const FbItem& it = find_item(items, n, static_cast<int>(blockIdx.x));
  finebound_body<SHIFT, SCALAR>(it, static_cast<int>(blockIdx.x) - it.block0);
}

__global__ void __launch_bounds__(kPtBlock) k_restrict_table(const RsItem* __restrict__ items, int n) {
  const RsItem& it = find_item(items, n, static_cast<int>(blockIdx.x));
  restrict_body(it, static_cast<int>(blockIdx.x) - it.block0);
}

// 0D norms of one field over i in [1, Nr-g], j in [1, Nz-g] (the range
// save0Ddata.f90:221-246 reduces): per block max, min, max|f|, sum f^2,
// point count and a NaN flag, in a fixed tree order; the host combines the
// blocks in block order.
constexpr int kNormBlocks = 256;
// partial record b of one field: a grid-stride pass of block b of nb
__device__ __forceinline__ void norms_block(const KGrid& G, const double* __restrict__ f, double* __restrict__ part,
                                            int b, int nb) {
  __shared__ double smax[kPtBlock], smin[kPtBlock], sabs[kPtBlock], ssq[kPtBlock], scnt[kPtBlock], snan[kPtBlock];
  const int ni = G.Nr - G.g, nj = G.Nz - G.g;
  const long n = static_cast<long>(ni) * nj;
  double vmax = -1.0e300, vmin = 1.0e300, vabs = 0.0, sq = 0.0, cnt = 0.0, nan = 0.0;
  for (long q = static_cast<long>(b) * kPtBlock + threadIdx.x; q < n; q += static_cast<long>(nb) * kPtBlock) {
    const int i = 1 + static_cast<int>(q / nj), j = 1 + static_cast<int>(q % nj);
    const double v = f[IDX(G, i, j)];
    if (v != v) nan = 1.0;
    vmax = fmax(vmax, v);
    vmin = fmin(vmin, v);
    vabs = fmax(vabs, fabs(v));
    sq += v * v;
    cnt += 1.0;
  }
  const int t = static_cast<int>(threadIdx.x);
  smax[t] = vmax; smin[t] = vmin; sabs[t] = vabs; ssq[t] = sq; scnt[t] = cnt; snan[t] = nan;
  __syncthreads();
  for (int h = kPtBlock / 2; h > 0; h >>= 1) {
    if (t < h) {
      smax[t] = fmax(smax[t], smax[t + h]);
      smin[t] = fmin(smin[t], smin[t + h]);
      sabs[t] = fmax(sabs[t], sabs[t + h]);
      ssq[t] += ssq[t + h];
      scnt[t] += scnt[t + h];
      snan[t] = fmax(snan[t], snan[t + h]);
    }
    __syncthreads();
  }
  if (t == 0) {
    double* o = part + 6 * b;
    o[0] = smax[0]; o[1] = smin[0]; o[2] = sabs[0]; o[3] = ssq[0]; o[4] = scnt[0]; o[5] = snan[0];
  }
}

__global__ void __launch_bounds__(kPtBlock) k_norms_partial(KGrid G, const double* __restrict__ f,
                                                            double* __restrict__ part) {
  norms_block(G, f, part, static_cast<int>(blockIdx.x), kNormBlocks);
}

// The norms of several fields of one level: blockIdx.y picks the field,
// whose kNormBlocks partial records start at part + y * 6 * kNormBlocks.
constexpr int kNormsMaxFields = 32;
struct NormsFields {
  KGrid G;
  int n;
  const double* f[kNormsMaxFields];
};

__global__ void __launch_bounds__(kPtBlock) k_norms_fields(NormsFields a, double* __restrict__ part) {
  const int y = static_cast<int>(blockIdx.y);
  norms_block(a.G, a.f[y], part + static_cast<long>(6) * kNormBlocks * y, static_cast<int>(blockIdx.x),
              kNormBlocks);
}

// Thread y combines the partial records of field y in block order, as the
// host does for oa_norms0d: out[5y..5y+4] = max, min, max|f|, rms, NaN flag.
__global__ void __launch_bounds__(64) k_norms_combine(int n, const double* __restrict__ part,
                                                      double* __restrict__ out) {
  const int y = static_cast<int>(threadIdx.x);
  if (y >= n) return;
  const double* p = part + static_cast<long>(6) * kNormBlocks * y;
  double vmax = -1.0e300, vmin = 1.0e300, vabs = 0.0, sq = 0.0, cnt = 0.0, nan = 0.0;
  for (int b = 0; b < kNormBlocks; ++b) {
    const double* o = p + 6 * b;
    vmax = fmax(vmax, o[0]);
    vmin = fmin(vmin, o[1]);
    vabs = fmax(vabs, o[2]);
    sq += o[3];
    cnt += o[4];
    nan = fmax(nan, o[5]);
  }
  double* r = out + 5 * y;
  r[0] = vmax;
  r[1] = vmin;
  r[2] = vabs;
  r[3] = (cnt > 0.0) ? sqrt(sq / cnt) : 0.0;
  r[4] = nan;
}

// dtbeta = drivercsi * Delta (evolve.f90:174-195), whole arrays incl. images
__global__ void k_dtbeta_init(long n, double csi, const double* __restrict__ dr, const double* __restrict__ dz,
                              double* __restrict__ tr, double* __restrict__ tz) {
  const long q = static_cast<long>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (q >= n) return;
  tr[q] = csi * dr[q];
  tz[q] = csi * dz[q];
}

// the fixed geometry of the fine boundary zone of depth D (once per level)
__global__ void __launch_bounds__(256) k_fb_table(KGrid Gf, KGrid Gc, int D, int interporder, long n,
                                                  FbPoint* __restrict__ table) {
  const long q = static_cast<long>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (q >= n) return;
  FbPoint fp{};               // a record of no point holds zeros: its i and j are read before its kind is looked at
  fb_geometry(Gf, Gc, D, interporder, q, fp);
  table[q] = fp;
}

// ------------------------------------------------------------- launchers
static int check_launch() {
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) {
    oa_set_error(std::string("kernel launch failed: ") + hipGetErrorString(e));
    return OA_ERR_HIP;
  }
  return OA_OK;
}

static int blocks_for(long threads) { return static_cast<int>((threads + kPtBlock - 1) / kPtBlock); }

static void set_tiles(RhsItem* it) {
  it->nbi = (it->ihi + kTile - 1) / kTile;
  it->nbj = (it->jhi - it->jlo + 1 + kTile - 1) / kTile;
}

static void set_strips(RhsItem* it) {
  const KGrid& G = it->G;
  it->nstr = (G.Nz - G.jlo + 1 + kStripR - 1) / kStripR;
  it->nstz = (G.Nr - G.g + kStripZ - 1) / kStripZ;
}

bool rhs_by_parts(bool shift, bool scalar) { return !shift || scalar; }

int rhs_strips(const RhsItem& it) { return it.nstr + it.nstz * (it.G.eqsym ? 1 : 2); }

int rhs_tiles(RhsItem* it, bool strips, bool* inner) {
  const KGrid& G = it->G;
  if (G.Nr < kTile || G.Nz - G.jlo + 1 < kTile) {
    oa_set_error("RHS kernel: a level needs at least 16 points in each direction");
    return OA_ERR_ARG;
  }
  it->ihi = G.Nr;
  it->jlo = G.jlo;
  it->jhi = G.Nz;
  it->skip = 0;
  it->nstr = it->nstz = 0;
  it->depth = -1;
  if (*inner || strips) {
    const int jlo = G.eqsym ? G.jlo : G.jlo + G.g;
    if (G.Nr - G.g >= kTile && G.Nz - G.g - jlo + 1 >= kTile) {
      it->ihi = G.Nr - G.g;
      it->jlo = jlo;
      it->jhi = G.Nz - G.g;
      if (!*inner) set_strips(it);
    } else {
      *inner = false;
    }
  }
  set_tiles(it);
  return OA_OK;
}

void rhs_add_frame(std::vector<RhsItem>* items, bool strips) {
  RhsItem& it = items->front();
  if (strips) {
    set_strips(&it);
    return;
  }
  RhsItem f = it;
  f.skip = 1;
  f.sihi = it.ihi;
  f.sjlo = it.jlo;
  f.sjhi = it.jhi;
  f.ihi = it.G.Nr;
  f.jlo = it.G.jlo;
  f.jhi = it.G.Nz;
  set_tiles(&f);
  items->push_back(f);
}

void rhs_stencil(const KGrid& G, const KPhys& P, KStencil* W) {
  W->r12 = G.idr / 12.0;
  W->z12 = G.idz / 12.0;
  W->rr12 = G.idr * G.idr / 12.0;
  W->zz12 = G.idz * G.idz / 12.0;
  W->rz3 = G.idr * G.idz / 3.0;
  W->rz48 = G.idr * G.idz / 48.0;
  const double up[3] = {10.5, -3.0, 0.5}, cen[3] = {8.0, -1.0, 0.0};
  for (int k = 0; k < 3; ++k) {
    W->ar[k] = (P.shiftadvect ? up[k] : cen[k]) * G.idr / 12.0;
    W->az[k] = (P.shiftadvect ? up[k] : cen[k]) * G.idz / 12.0;
  }
  W->ur = P.shiftadvect ? 0.5 * G.idr / 12.0 : 0.0;
  W->uz = P.shiftadvect ? 0.5 * G.idz / 12.0 : 0.0;
  W->ko_g = P.geodiss / G.dt * 0.05;
  W->ko_s = P.scalardiss / G.dt * 0.05;
}

int rhs_blocks(const RhsItem& it) { return it.nbi * it.nbj + it.xtra; }

// Blocks of their own for the edge work, only if the whole launch is then
// resident at once (two blocks per CU): they end before the tiles, whose
// blocks would take several units each on a small level.  A launch that fills
// the GPU spreads the units over its tiles' blocks instead, one or two waves
// of each.  The deeper zone is counted whichever is filled, so that the grid
// does not depend on whether the clocks meet (a floating comparison).
void rhs_plan_edges(std::vector<RhsItem>* items, bool shift, bool scalar) {
  const int waves = (rhs_by_parts(shift, scalar) ? kRhsBlock : kTile * kTile) / 64;
  auto own = [&](const RhsItem& it) {
    const int nrt = it.G.Nr + it.G.g, nzt = it.G.Nz + it.G.g;
    int u = it.E.n > 0 ? finebound_groups(shift, scalar) * static_cast<int>((fb_count(it.G, it.G.g + 2) + 63) / 64) : 0;
    if (it.E.rR) u += nslots(shift, scalar) * ((it.G.g * (nrt > nzt ? nrt : nzt) + 63) / 64);
    return (u + waves - 1) / waves;
  };
  int total = 0;
  for (RhsItem& it : *items) {
    it.xtra = 0;
    total += rhs_blocks(it) + rhs_strips(it) + own(it);
  }
  if (total > kResidentBlocks) return;
  for (RhsItem& it : *items) it.xtra = own(it);
}
int proj_blocks(const ProjItem& it) { return blocks_for(static_cast<long>(it.G.Nr) * (it.G.Nz - it.G.jlo + 1)); }
int del_blocks(const DelItem& it) { return blocks_for(static_cast<long>(it.G.Nr) * (it.G.Nz - it.G.jlo + 1)); }
int save_blocks(const SaveItem& it) {
  const int nrt = it.G.Nr + it.G.g, nzt = it.G.Nz + it.G.g;
  return it.nf * blocks_for(static_cast<long>(it.G.g) * (nrt > nzt ? nrt : nzt));
}
// Sized for the deeper of the two zones whichever this call fills, so that
// the grid of a finebound launch does not depend on whether the clocks meet
// (a floating comparison); the blocks past the item's own records exit.
int fb_blocks(const FbItem& it, bool shift, bool scalar) {
  return finebound_groups(shift, scalar) * blocks_for(fb_count(it.Gf, it.Gf.g + 2));
}
int rs_blocks(const RsItem& it) { return it.nf * blocks_for(static_cast<long>(it.nic) * it.njc); }

template <class K>
static int raise_lds_limit(K* kernel, size_t bytes) {
  if (hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize,
                          static_cast<int>(bytes)) != hipSuccess) {
    oa_set_error("hipFuncSetAttribute(MaxDynamicSharedMemorySize) failed for an RHS kernel");
    return OA_ERR_HIP;
  }
  return OA_OK;
}

// the dynamic LDS of one RHS block exceeds the 64 KiB default; two more
// planes on a level's first substep (KStep::dtb_pre)
template <bool SH, bool SC, bool PM>
static int rhs_lds(bool dtb_pre, size_t* lds) {
  const size_t per = sizeof(double) * kTileSize, col = (SH && !SC) ? 0 : sizeof(double) * kInvR;
  static bool attr_set = false;
  if (!attr_set) {
    const size_t most = per * static_cast<size_t>(nslots(SH, SC) + 2) + col;
    if constexpr (SH && !SC) RC_K(raise_lds_limit(&k_rhs_phases<PM>, most));
    else RC_K(raise_lds_limit(&k_rhs_table<SH, SC, PM>, most));
    attr_set = true;
  }
  *lds = per * static_cast<size_t>(nslots(SH, SC) + (dtb_pre ? 2 : 0)) + col;
  return OA_OK;
}

template <bool SH, bool SC, bool PM>
static int launch_rhs_table_t(const RhsItem* items, int n, int blocks, int strips, bool any_pre, bool xcd,
                              hipStream_t st) {
  size_t lds = 0;
  RC_K((rhs_lds<SH, SC, PM>(any_pre, &lds)));
  if constexpr (SH && !SC) {
    (void)strips;
    hipLaunchKernelGGL((k_rhs_phases<PM>), dim3(blocks), dim3(kTile * kTile), lds, st, items, n, xcd ? 1 : 0);
    return check_launch();
  } else {
    hipLaunchKernelGGL((k_rhs_table<SH, SC, PM>), dim3(blocks), dim3(kRhsBlock), lds, st, items, n, strips, xcd ? 1 : 0);
    return check_launch();
  }
}

// The LDS limits of every RHS variant, raised once before any launch (and so
// outside any graph capture).
int prepare_rhs_kernels() {
  static int rc = -1;
  if (rc >= 0) return rc;
  size_t lds = 0;
  rc = OA_OK;
  if (rc == OA_OK) rc = rhs_lds<false, false, false>(false, &lds);
  if (rc == OA_OK) rc = rhs_lds<false, false, true>(false, &lds);
  if (rc == OA_OK) rc = rhs_lds<false, true, false>(false, &lds);
  if (rc == OA_OK) rc = rhs_lds<false, true, true>(false, &lds);
  if (rc == OA_OK) rc = rhs_lds<true, false, false>(false, &lds);
  if (rc == OA_OK) rc = rhs_lds<true, false, true>(false, &lds);
  if (rc == OA_OK) rc = rhs_lds<true, true, false>(false, &lds);
  if (rc == OA_OK) rc = rhs_lds<true, true, true>(false, &lds);
  return rc;
}

#define RHS_DISPATCH(FN, ...)                                   \
  switch ((shift ? 4 : 0) + (scalar ? 2 : 0) + (phimode ? 1 : 0)) { \
    case 0: return FN<false, false, false>(__VA_ARGS__);        \
    case 1: return FN<false, false, true>(__VA_ARGS__);         \
    case 2: return FN<false, true, false>(__VA_ARGS__);         \
    case 3: return FN<false, true, true>(__VA_ARGS__);          \
    case 4: return FN<true, false, false>(__VA_ARGS__);         \
    case 5: return FN<true, false, true>(__VA_ARGS__);          \
    case 6: return FN<true, true, false>(__VA_ARGS__);          \
    default: return FN<true, true, true>(__VA_ARGS__);          \
  }

int launch_rhs_table(const RhsItem* items, int n, int blocks, int strips, bool shift, bool scalar, bool phimode,
                     bool any_dtb_pre, bool xcd_remap, void* stream) {
  hipStream_t st = static_cast<hipStream_t>(stream);
  RHS_DISPATCH(launch_rhs_table_t, items, n, blocks, strips, any_dtb_pre, xcd_remap, st)
}

#define SC_DISPATCH(K, GRID, ...)                                                                  \
  do {                                                                                             \
    if (shift && scalar) hipLaunchKernelGGL((K<true, true>), GRID, dim3(kPtBlock), 0, st, __VA_ARGS__);   \
    else if (shift) hipLaunchKernelGGL((K<true, false>), GRID, dim3(kPtBlock), 0, st, __VA_ARGS__);       \
    else if (scalar) hipLaunchKernelGGL((K<false, true>), GRID, dim3(kPtBlock), 0, st, __VA_ARGS__);      \
    else hipLaunchKernelGGL((K<false, false>), GRID, dim3(kPtBlock), 0, st, __VA_ARGS__);                 \
  } while (0)

int launch_project_table(const ProjItem* items, int n, int blocks, bool shift, bool scalar, void* stream) {
  hipStream_t st = static_cast<hipStream_t>(stream);
  SC_DISPATCH(k_project_table, dim3(blocks), items, n);
  return check_launch();
}

int launch_finebound_table(const FbItem* items, int n, int blocks, bool shift, bool scalar, void* stream) {
  hipStream_t st = static_cast<hipStream_t>(stream);
  SC_DISPATCH(k_finebound_table, dim3(blocks), items, n);
  return check_launch();
}

int launch_deldef_table(const DelItem* items, int n, int blocks, void* stream) {
  hipLaunchKernelGGL(k_deldef_table, dim3(blocks), dim3(kPtBlock), 0, static_cast<hipStream_t>(stream), items, n);
  return check_launch();
}

int launch_saveold_table(const SaveItem* items, int n, int blocks, void* stream) {
  hipLaunchKernelGGL(k_saveold_table, dim3(blocks), dim3(kPtBlock), 0, static_cast<hipStream_t>(stream), items, n);
  return check_launch();
}

int launch_restrict_table(const RsItem* items, int n, int blocks, void* stream) {
  hipLaunchKernelGGL(k_restrict_table, dim3(blocks), dim3(kPtBlock), 0, static_cast<hipStream_t>(stream), items,
                     n);
  return check_launch();
}

int launch_dtbeta_init(const KGrid& G, double csi, bool scalar, double* y, void* stream) {
  (void)scalar;
  const long n = G.plane;
  const long pl = G.plane;
  hipLaunchKernelGGL(k_dtbeta_init, dim3(blocks_for(n)), dim3(kPtBlock), 0, static_cast<hipStream_t>(stream), n,
                     csi, y + S_Delta_r * pl, y + S_Delta_z * pl, y + shift_slot(SH_dtbeta_r) * pl,
                     y + shift_slot(SH_dtbeta_z) * pl);
  return check_launch();
}

int norms_blocks() { return kNormBlocks; }

// An array on its way to the caller: transposed from the device's layout (z
// fastest) through LDS and written straight into pinned host memory.  Bound by
// the link to the host; 256 x 512 took 298 us as a copy to pageable memory and
// a transposition there, and takes 103 us with the copy out of the pinned buffer.
constexpr int kOutTile = 32, kOutRows = 8;

__global__ void __launch_bounds__(kOutTile * kOutRows) k_plane_out(KGrid G, const double* __restrict__ src,
                                                                    double* __restrict__ host) {
  __shared__ double tile[kOutTile][kOutTile + 1];
  const int nrt = G.Nr + G.g, nzt = G.Nz + G.g, x = static_cast<int>(threadIdx.x), y = static_cast<int>(threadIdx.y);
  const int i0 = static_cast<int>(blockIdx.x) * kOutTile, j0 = static_cast<int>(blockIdx.y) * kOutTile;
  for (int r = y; r < kOutTile; r += kOutRows)
    if (i0 + r < nrt && j0 + x < nzt) tile[r][x] = src[static_cast<long>(i0 + r) * G.ld + j0 + x];
  __syncthreads();
  for (int r = y; r < kOutTile; r += kOutRows)
    if (j0 + r < nzt && i0 + x < nrt) host[static_cast<long>(j0 + r) * nrt + i0 + x] = tile[x][r];
}

int launch_plane_out(const KGrid& G, const double* src, double* host, void* stream) {
  const dim3 grd((G.Nr + G.g + kOutTile - 1) / kOutTile, (G.Nz + G.g + kOutTile - 1) / kOutTile);
  hipLaunchKernelGGL(k_plane_out, grd, dim3(kOutTile, kOutRows), 0, static_cast<hipStream_t>(stream), G, src, host);
  return check_launch();
}

int launch_norms_partial(const KGrid& G, const double* f, double* part, void* stream) {
  hipLaunchKernelGGL(k_norms_partial, dim3(kNormBlocks), dim3(kPtBlock), 0, static_cast<hipStream_t>(stream), G, f,
                     part);
  return check_launch();
}

// Partial records of oa_norms0d_noalloc: kNormsMaxFields fields of
// kNormBlocks records of 6 doubles (384 KiB).  Each GPU holds its own copy for
// the life of the process.  Host code never uses this name as an address: it
// uses the device address hipGetSymbolAddress returns for the current device.
static __device__ __align__(256) double scratch[kNormsMaxFields * kNormBlocks * 6];

namespace {
constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
double* g_scratch_ptr[kMaxDevices] = {};

// the address of `scratch` on device dev, looked up once per device with that
// device current
int scratch_on(int dev, double** out) {
  if (dev < 0 || dev >= kMaxDevices) {
    oa_set_error("oa_norms0d_noalloc: device index out of range");
    return OA_ERR_HIP;
  }
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (!g_scratch_ptr[dev]) {
    int prev = -1;
    if (hipGetDevice(&prev) != hipSuccess) {
      oa_set_error("oa_norms0d_noalloc: hipGetDevice failed");
      return OA_ERR_HIP;
    }
    if (prev != dev && hipSetDevice(dev) != hipSuccess) {
      oa_set_error("oa_norms0d_noalloc: hipSetDevice failed");
      return OA_ERR_HIP;
    }
    void* ptr = nullptr;
    const hipError_t e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
    if (prev != dev) (void)hipSetDevice(prev);
    if (e != hipSuccess || !ptr) {
      oa_set_error(std::string("oa_norms0d_noalloc: hipGetSymbolAddress(scratch) failed: ") + hipGetErrorString(e));
      return OA_ERR_HIP;
    }
    g_scratch_ptr[dev] = static_cast<double*>(ptr);
  }
  *out = g_scratch_ptr[dev];
  return OA_OK;
}
}  // namespace

int norms_max_fields() { return kNormsMaxFields; }

int launch_norms_fields_noalloc(int dev, const KGrid& G, int n, const double* const* planes, double* out,
                                void* stream) {
  if (n < 1 || n > kNormsMaxFields) {
    oa_set_error("oa_norms0d_noalloc: " + std::to_string(n) + " arrays requested; one call takes 1 to " +
                 std::to_string(kNormsMaxFields));
    return OA_ERR_ARG;
  }
  double* part = nullptr;
  RC_K(scratch_on(dev, &part));
  NormsFields a{};
  a.G = G;
  a.n = n;
  for (int k = 0; k < n; ++k) a.f[k] = planes[k];
  const hipStream_t st = static_cast<hipStream_t>(stream);
  hipLaunchKernelGGL(k_norms_fields, dim3(kNormBlocks, static_cast<unsigned>(n)), dim3(kPtBlock), 0, st, a, part);
  RC_K(check_launch());
  hipLaunchKernelGGL(k_norms_combine, dim3(1), dim3(64), 0, st, n, part, out);
  return check_launch();
}

int launch_constraints(const KGrid& G, const KPhys& P, const KStep& S, bool phimode, bool scalar, int sc0,
                       const double* y, double* gaux, double* out, void* stream) {
  hipStream_t st = static_cast<hipStream_t>(stream);
  RhsItem it{};
  it.G = G;
  it.P = P;
  bool inner = false;
  RC_K(rhs_tiles(&it, false, &inner));
  it.S = S;
  it.S.dtb_pre = nullptr;
  it.yin = y;
  it.gaux = gaux;
  const size_t lds = sizeof(double) * kTileSize * NBASE;
  static bool attr = false;
  if (!attr) {
    RC_K(raise_lds_limit(&k_aux<false>, lds));
    RC_K(raise_lds_limit(&k_aux<true>, lds));
    attr = true;
  }
  const dim3 tg(static_cast<unsigned>(it.nbj), static_cast<unsigned>(it.nbi), 1);
  if (phimode) hipLaunchKernelGGL(k_aux<true>, tg, dim3(kTile, kTile, 1), lds, st, it);
  else hipLaunchKernelGGL(k_aux<false>, tg, dim3(kTile, kTile, 1), lds, st, it);
  RC_K(check_launch());
  const ConsArgs c{G, P, sc0, y, gaux, out};
  const dim3 blk(64, 4, 1);
  const dim3 grd((G.Nz - G.jlo + 1 + 63) / 64, (G.Nr + 3) / 4, 1);
  const int code = (phimode ? 2 : 0) + (scalar ? 1 : 0);
  if (code == 0) hipLaunchKernelGGL((k_constraints<false, false>), grd, blk, 0, st, c);
  else if (code == 1) hipLaunchKernelGGL((k_constraints<false, true>), grd, blk, 0, st, c);
  else if (code == 2) hipLaunchKernelGGL((k_constraints<true, false>), grd, blk, 0, st, c);
  else hipLaunchKernelGGL((k_constraints<true, true>), grd, blk, 0, st, c);
  RC_K(check_launch());
  hipLaunchKernelGGL(k_ham_fix, dim3(1), dim3(256), 0, st, G, out + CN_ham * G.plane);
  return check_launch();
}

long fb_points(const KGrid& Gf, int depth) { return fb_count(Gf, depth); }
size_t fb_record_bytes() { return sizeof(FbPoint); }

int launch_fb_table(const KGrid& Gf, const KGrid& Gc, int depth, int interporder, FbPoint* table, long n,
                    void* stream) {
  hipLaunchKernelGGL(k_fb_table, dim3(blocks_for(n)), dim3(kPtBlock), 0, static_cast<hipStream_t>(stream), Gf, Gc,
                     depth, interporder, n, table);
  return check_launch();
}

}  // namespace oax
