// build_kernels.hpp -- pair-list construction on gfx950: periodic wrap,
// counting-sort cell binning (atomics + prefix scan, then each cell's members
// put back in input order, so the result does not depend on atomic ordering)
// and the ghost images of the single-domain halo, for every replica of a
// domain at once (each particle carries its replica index).
//
// Reference semantics (kaityo256/mdacp): AdjustPeriodicBoundary
// (variables.cc:59-79), MakeMesh (meshlist.cc:153-205), FindBorderParticles
// and MakeBufferForBorderParticles (mdunit.cc:125-176, mdrect.cc:24-47),
// SearchMesh (meshlist.cc:220-271).  The distance test is evaluated without
// fused multiply-adds (the library is compiled with -ffp-contract=off), so the
// pair set is bit-exact with the reference's default build.
#pragma once
#include "device_common.hpp"

namespace mdgpu {

// MeshList's cell of a position (meshlist.cc:164-182): int((q - s) * (1/w)) + 1
// per axis with s the box origin (0 for a periodic box, where q - 0.0 is q), as
// a global cell index.
__device__ __forceinline__ int cell_of(double x, double y, double z, const Replica &R) {
  int ix = (int)((x - R.o[0]) * R.im[0]) + 1;
  int iy = (int)((y - R.o[1]) * R.im[1]) + 1;
  int iz = (int)((z - R.o[2]) * R.im[2]) + 1;
  if (ix < 0) ix = R.m[0] - 1; else if (ix >= R.m[0]) ix = 0;
  if (iy < 0) iy = R.m[1] - 1; else if (iy >= R.m[1]) iy = 0;
  if (iz < 0) iz = R.m[2] - 1; else if (iz >= R.m[2]) iz = 0;
  return R.cell0 + R.m[0] * R.m[1] * iz + R.m[0] * iy + ix;
}

// A slot in cell c's counter for each active lane of the wavefront: one
// atomic add per distinct cell among the active lanes, whose lanes take
// consecutive slots in lane order.  The lanes are first grouped by cell with
// ballots (no memory traffic); then the first lane of every group adds its
// group's size in the same instruction, so the wavefront waits for one atomic
// round trip however many cells it meets (rows sorted by list length put many
// cells in one wavefront).  Per-particle atomics on one counter would
// serialise.  The order within a cell is settled later by particle id.
__device__ __forceinline__ int cell_slot(int *__restrict__ counts, int c) {
  unsigned long long todo = __ballot(1);
  const int lane = __lane_id();
  int leader_of = lane, rank = 0, size = 0;
  while (todo) {
    const int leader = __ffsll((long long)todo) - 1;
    const int cl = __shfl(c, leader, kWave);
    const unsigned long long same = __ballot(c == cl) & todo;
    if (c == cl) {
      leader_of = leader;
      rank = __popcll(same & ((1ull << lane) - 1ull));
    }
    if (lane == leader) size = __popcll(same);
    todo &= ~same;
  }
  int base = 0;
  if (lane == leader_of) base = atomicAdd(&counts[c], size);
  return __shfl(base, leader_of, kWave) + rank;
}

// Wrap owned particles into their replica's box (one +-L per component), flag
// positions still outside, bin, and take a slot in the cell (cell_slot).
__global__ void k_wrap_bin(double4 *__restrict__ pos, int n, const int *__restrict__ rep,
                           const Replica *__restrict__ reps, int *__restrict__ cell, int *__restrict__ slot,
                           int *__restrict__ ccount, int *__restrict__ err, int wrap) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const Replica &R = reps[rep[i]];
  double4 q = pos[i];
  if (wrap) {
    const double Lx = R.L[0], Ly = R.L[1], Lz = R.L[2];
    if (q.x < 0.0) q.x += Lx; else if (q.x > Lx) q.x -= Lx;
    if (q.y < 0.0) q.y += Ly; else if (q.y > Ly) q.y -= Ly;
    if (q.z < 0.0) q.z += Lz; else if (q.z > Lz) q.z -= Lz;
    pos[i] = q;
    // the reference lets NaN through this test; a NaN is refused here
    if (!(q.x >= 0.0 && q.x <= Lx && q.y >= 0.0 && q.y <= Ly && q.z >= 0.0 && q.z <= Lz))
      atomicOr(err, kErrInvalidPosition);
  }
  const int c = cell_of(q.x, q.y, q.z, R);
  // 0 <= q <= L bins into cells 1 .. m - 1, which bricks cover; the lower
  // ghost layer is refused like a position outside the box
  const int l = c - R.cell0;
  if (l % R.m[0] == 0 || (l / R.m[0]) % R.m[1] == 0 || l / (R.m[0] * R.m[1]) == 0)
    atomicOr(err, kErrInvalidPosition);
  cell[i] = c;
  slot[i] = cell_slot(ccount, c);
}

// Zeroes a construction's state and its two cell counters.
__global__ void k_build_begin(BuildState *__restrict__ bs, int *__restrict__ ocount, int *__restrict__ gcount,
                              int ncell) {
  const int c = blockIdx.x * blockDim.x + threadIdx.x;
  if (c == 0) *bs = BuildState{};
  if (c < ncell) {
    ocount[c] = 0;
    gcount[c] = 0;
  }
}

// First particle of each cell: the cells taken in storage order (order[k] =
// the k-th cell, brick by brick), also by that order in start_r.
struct ScanCells {
  const int *count, *order;
  int *start, *start_r;
  __device__ __forceinline__ long long in(long long k) const { return count[order[k]]; }
  __device__ __forceinline__ void out(long long k, long long x, long long) const {
    start[order[k]] = (int)x;
    start_r[k] = (int)x;
  }
  __device__ __forceinline__ void total(long long) const {}
};

// Order of a cell's members: by (key, input index) when `key` is given, else
// by input index.  Keys are unique, so this is a permutation, and with the
// slots taken by atomics it makes the order deterministic.  Owned particles
// are keyed by particle id, so the order after a construction depends only on
// the particles and their ids, not on the order an earlier one left.
__device__ __forceinline__ unsigned long long sort_key(const int *__restrict__ key, int i) {
  const unsigned long long k = key ? (unsigned long long)((unsigned)key[i] ^ 0x80000000u) : 0ull;
  return (k << 32) | (unsigned)i;
}

// Items grouped by cell, in atomic order, as their sort keys (the item in the
// low word).  n items, or bs->ng.
__global__ void k_scatter_keys(const int *__restrict__ cell, const int *__restrict__ slot,
                               const int *__restrict__ cstart, int n, const int *__restrict__ key,
                               unsigned long long *__restrict__ keys, const BuildState *__restrict__ bs) {
  if (bs->err) return;
  const int m = n >= 0 ? n : (int)bs->ng;
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < m; i += gridDim.x * blockDim.x)
    keys[cstart[cell[i]] + slot[i]] = sort_key(key, i);
}

// The place of grouped item p in its cell [s0, s0 + m): s0 and the members
// that sort before it, read four at a time (a chain of single reads took 20 us
// at any size).
__device__ __forceinline__ int sorted_place(const unsigned long long *__restrict__ keys, unsigned long long mine,
                                            int s0, int m) {
  int rank = 0, q = 0;
  for (; q + 4 <= m; q += 4) {
    const unsigned long long a = keys[s0 + q], b = keys[s0 + q + 1], c = keys[s0 + q + 2], d = keys[s0 + q + 3];
    rank += (a < mine) + (b < mine) + (c < mine) + (d < mine);
  }
  for (; q < m; q++) rank += keys[s0 + q] < mine;
  return s0 + rank;
}

struct OwnedArrays {
  double4 *pos, *mom;
  int *id, *cell, *rep;
};

// The owned particles in brick order, each cell's by id, and (nimg) the ghost
// images each will have (face_options).
__global__ void k_sort_owned(const unsigned long long *__restrict__ keys, const int *__restrict__ cstart,
                             const int *__restrict__ ccount, int n, OwnedArrays in, OwnedArrays out,
                             int *__restrict__ nimg, const Replica *__restrict__ reps, double SL,
                             const BuildState *__restrict__ bs) {
  const int p = blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= n || bs->err) return;
  const unsigned long long mine = keys[p];
  const int i = (int)(unsigned)mine;
  const int c = in.cell[i];
  const double4 q = in.pos[i], mo = in.mom[i];
  const int id = in.id[i], r = in.rep[i];
  const int k = sorted_place(keys, mine, cstart[c], ccount[c]);
  out.pos[k] = q;
  out.mom[k] = mo;
  out.id[k] = id;
  out.cell[k] = c;
  out.rep[k] = r;
  if (nimg) {
    int lo[3], hi[3];
    face_options(q, reps[r], SL, lo, hi);
    nimg[k] = (1 + lo[0] + hi[0]) * (1 + lo[1] + hi[1]) * (1 + lo[2] + hi[2]) - 1;
  }
}

// First image of each owned particle; the construction stops when there are
// more images than room.
struct ScanImages {
  const int *nimg;
  int *goff;
  BuildState *bs;
  long long cap;
  __device__ __forceinline__ long long in(long long i) const { return nimg[i]; }
  __device__ __forceinline__ void out(long long i, long long x, long long) const { goff[i] = (int)x; }
  __device__ __forceinline__ void total(long long t) const {
    bs->ng = t;
    if (t > cap) atomicOr(&bs->err, kErrGhostCap);
  }
};

// Halo of one domain (MDManager::MakePairList's six sequential
// FindBorderParticles/SendBorderParticlesSub passes, mdmanager.cc:269-275):
// along each axis a particle strictly within SL of the low face gets an image
// at +L, strictly within SL of the high face an image at -L; images of images
// make the edges and corners.  Equivalently, one image per non-zero shift
// vector whose every non-zero component passes its face test.  The box is
// [s, e) = [0, L) (MDRect::IsInsideEdge, mdrect.cc:24-47: s < q < s + SL and
// e - SL < q < e).
struct GhostArrays {
  int *src, *code;
  double4 *pos;
  int *cell, *slot, *count;
};

__device__ __forceinline__ void put_image(const GhostArrays &G, int k, int i, int code, int r, const double3 y,
                                          int cl, int slot) {
  G.src[k] = i;
  G.code[k] = ghost_word(code, r);
  G.pos[k] = make_double4(y.x, y.y, y.z, 0.0);
  G.cell[k] = cl;
  G.slot[k] = slot;
}

// The images of each particle from goff[i], in the order of the shifts 0, +1,
// -1 along x, then y, then z.  A particle near one face of an axis at most has
// up to seven; their cells' counters are asked for together (one after
// another, each waiting for its slot, they took 19 us).  One near both faces
// (a box of two search lengths, to a rounding) takes the general loop.
__global__ void k_emit_images(const double4 *__restrict__ pos, int n, const int *__restrict__ rep,
                              const Replica *__restrict__ reps, double SL, const int *__restrict__ goff,
                              const BuildState *__restrict__ bs, GhostArrays G) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n || bs->err) return;
  const int r = rep[i];
  const Replica &R = reps[r];
  const double4 q = pos[i];
  int lo[3], hi[3];
  face_options(q, R, SL, lo, hi);
  if (!(lo[0] | lo[1] | lo[2] | hi[0] | hi[1] | hi[2])) return;
  const int ng = (int)bs->ng;
  int k = goff[i];
  if ((lo[0] & hi[0]) | (lo[1] & hi[1]) | (lo[2] & hi[2])) {
    const int sxs[3] = {0, 1, -1};
    for (int a = 0; a < 3; a++)
      for (int b = 0; b < 3; b++)
        for (int c = 0; c < 3; c++) {
          const int s[3] = {sxs[a], sxs[b], sxs[c]};
          bool image = (s[0] | s[1] | s[2]) != 0;
          for (int x = 0; x < 3; x++) image = image && (s[x] == 0 || (s[x] > 0 ? lo[x] : hi[x]));
          if (!image || k >= ng) continue;  // goff is the scan of the images' count: k < ng
          const int code = (s[0] + 1) + 3 * (s[1] + 1) + 9 * (s[2] + 1);
          const double3 y = image_of(q, code, R.L);
          const int cl = cell_of(y.x, y.y, y.z, R);
          put_image(G, k, i, code, r, y, cl, atomicAdd(&G.count[cl], 1));
          k++;
        }
    return;
  }
  const int s[3] = {lo[0] - hi[0], lo[1] - hi[1], lo[2] - hi[2]};
  int cl[8], slot[8];
#pragma unroll
  for (int j = 1; j < 8; j++) {
    const int sx = (j & 4) ? s[0] : 0, sy = (j & 2) ? s[1] : 0, sz = (j & 1) ? s[2] : 0;
    const bool image = (!(j & 4) || s[0]) && (!(j & 2) || s[1]) && (!(j & 1) || s[2]);
    cl[j] = -1;
    slot[j] = 0;
    if (image) {
      const double3 y = image_of(q, (sx + 1) + 3 * (sy + 1) + 9 * (sz + 1), R.L);
      cl[j] = cell_of(y.x, y.y, y.z, R);
      slot[j] = atomicAdd(&G.count[cl[j]], 1);
    }
  }
#pragma unroll
  for (int j = 1; j < 8; j++) {
    if (cl[j] < 0 || k >= ng) continue;
    const int sx = (j & 4) ? s[0] : 0, sy = (j & 2) ? s[1] : 0, sz = (j & 1) ? s[2] : 0;
    const int code = (sx + 1) + 3 * (sy + 1) + 9 * (sz + 1);
    put_image(G, k, i, code, r, image_of(q, code, R.L), cl[j], slot[j]);
    k++;
  }
}

// The ghosts in cell order, each cell's in the order they were emitted, after
// the pn owned particles.  gunit (a unit of a group): the source unit, taken
// out of the code word.
__global__ void k_sort_ghosts(const unsigned long long *__restrict__ keys, const int *__restrict__ gstart,
                              const int *__restrict__ gcount, int pn, const int *__restrict__ src_in,
                              const int *__restrict__ code_in, const double4 *__restrict__ gpos_in,
                              const int *__restrict__ gcell_in, int *__restrict__ gsrc, int *__restrict__ gcode,
                              int *__restrict__ gunit, double4 *__restrict__ pos, int *__restrict__ cell,
                              const BuildState *__restrict__ bs) {
  if (bs->err) return;
  const int ng = (int)bs->ng;
  for (int p = blockIdx.x * blockDim.x + threadIdx.x; p < ng; p += gridDim.x * blockDim.x) {
    const unsigned long long mine = keys[p];
    const int g = (int)(unsigned)mine;
    const int c = gcell_in[g], src = src_in[g], w = code_in[g];
    const double4 q = gpos_in[g];
    const int k = sorted_place(keys, mine, gstart[c], gcount[c]);
    gsrc[k] = src;
    gcode[k] = gunit ? ghost_shift(w) : w;
    if (gunit) gunit[k] = ghost_rep(w);
    pos[pn + k] = q;
    cell[pn + k] = c;
  }
}

// ---- units of a process grid: MDManager with several MDUnits in one process
// (mdmanager.cc:194-348), each unit a box [s, e) of the grid on the same device.

// Variables::AdjustPeriodicBoundary (variables.cc:59-79) with the whole box's
// edges: one +-L per component, then a position still outside [0, L] (or NaN)
// is flagged.
__global__ void k_unit_wrap(double4 *__restrict__ pos, int n, double Lx, double Ly, double Lz,
                            int *__restrict__ err) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  double4 q = pos[i];
  if (q.x < 0.0) q.x += Lx; else if (q.x > Lx) q.x -= Lx;
  if (q.y < 0.0) q.y += Ly; else if (q.y > Ly) q.y -= Ly;
  if (q.z < 0.0) q.z += Lz; else if (q.z > Lz) q.z -= Lz;
  pos[i] = q;
  if (!(q.x >= 0.0 && q.x <= Lx && q.y >= 0.0 && q.y <= Ly && q.z >= 0.0 && q.z <= Lz))
    atomicOr(err, kErrInvalidPosition);
}

// MDRect::IsOverBoundary (mdrect.cc:4-21) of direction dir (D_LEFT, D_RIGHT,
// D_BACK, D_FORWARD, D_DOWN, D_UP = 0..5: axis dir / 2, the low face for even
// dir) for a unit whose box spans [s, e) along that axis.
__global__ void k_leave_flags(const double4 *__restrict__ pos, int n, int dir, double s, double e,
                              int *__restrict__ flag) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const double4 q = pos[i];
  const int a = dir >> 1;
  const double v = a == 0 ? q.x : (a == 1 ? q.y : q.z);
  flag[i] = (dir & 1) ? (v >= e) : (v < s);
}

// MDUnit::MakeBufferForSendingParticle (mdunit.cc:78-101): the particles that
// leave go to the send buffer in their order (off = exclusive scan of the
// flags, from any value), the others are compacted in theirs.
__global__ void k_partition(const int *__restrict__ flag, const int *__restrict__ off, int n,
                            const double4 *__restrict__ pos, const double4 *__restrict__ mom,
                            const int *__restrict__ id, double4 *__restrict__ pos_keep,
                            double4 *__restrict__ mom_keep, int *__restrict__ id_keep,
                            double4 *__restrict__ pos_send, double4 *__restrict__ mom_send,
                            int *__restrict__ id_send) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const int o = off[i] - off[0];
  if (flag[i]) {
    pos_send[o] = pos[i];
    mom_send[o] = mom[i];
    id_send[o] = id[i];
  } else {
    pos_keep[i - o] = pos[i];
    mom_keep[i - o] = mom[i];
    id_keep[i - o] = id[i];
  }
}

// One unit of the group as a source of another unit's ghosts.  Along each
// axis the source is in the receiver's slab (same grid coordinate), or its
// left or right neighbour, or several of these at once (a grid of one or two
// units along the axis).  What the reference relays through six sequential
// FindBorderParticles / SendBorderParticlesSub passes (mdmanager.cc:269-275,
// mdunit.cc:125-191) is then, per axis and independently: the position
// itself from the same slab; from the left neighbour, a particle strictly
// within SL of that neighbour's high face (MDRect::IsInsideEdge D_RIGHT,
// mdrect.cc:30-31), shifted by -L when the neighbour's D_RIGHT crosses the
// periodic boundary (ParaInfo::IsOverBoundary, parainfo.cc:256-275); from the
// right neighbour, strictly within SL of its low face (D_LEFT), shifted by +L
// when that crosses.  The ghosts are every combination of one option per axis
// except the particle itself; a ghost relayed through other units carries the
// same position, since each relay adds 0 or +-L to one component only.
struct SrcUnit {
  const double4 *pos;     // the source's owned particles
  int n, base;            // their number and first entry in the concatenation
  int same[3];            // same grid coordinate as the receiver along the axis
  int left[3], right[3];  // the source is the receiver's left / right neighbour
  int lsh[3], rsh[3];     // image shift of what comes from the left / right: -1, 0, +1
  double s[3], e[3];      // the source's box, for its border tests
};
constexpr int kMaxUnits = 64;  // units in one group

// The options of one axis in the order k_emit_images takes its shifts (0,
// +1, -1 for a unit that is its own neighbour), so that a grid of one unit
// places its ghosts exactly as a periodic domain does.
__device__ __forceinline__ int unit_axis_options(const SrcUnit &S, int a, double v, double SL, int sh[3]) {
  int k = 0;
  if (S.same[a]) sh[k++] = 0;
  if (S.right[a] && v < S.s[a] + SL && v > S.s[a]) sh[k++] = S.rsh[a];
  if (S.left[a] && v > S.e[a] - SL && v < S.e[a]) sh[k++] = S.lsh[a];
  return k;
}

__device__ __forceinline__ int unit_source(const SrcUnit *__restrict__ tab, int nsrc, int t) {
  int w = nsrc - 1;
  while (w > 0 && t < tab[w].base) w--;
  return w;
}

__global__ void k_unit_count(const SrcUnit *__restrict__ tab, int nsrc, int total, int self, double SL,
                             int *__restrict__ cnt) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= total) return;
  const int w = unit_source(tab, nsrc, t);
  const SrcUnit &S = tab[w];
  const double4 q = S.pos[t - S.base];
  int sh[3];
  const int nx = unit_axis_options(S, 0, q.x, SL, sh);
  const int ny = unit_axis_options(S, 1, q.y, SL, sh);
  const int nz = unit_axis_options(S, 2, q.z, SL, sh);
  cnt[t] = nx * ny * nz - (w == self ? 1 : 0);
}

// The images of k_unit_count's count, at off[t]: source index and a word
// holding the shift code and the source unit (ghost_word), the position, the
// Owned positions of every unit of a group, by unit slot.
struct UnitPos {
  const double4 *pos[kMaxUnits];
};

// receiver's cell and a slot in it.  The shift is added as image_of adds it.
// The positions come in the arguments, not from the table: making room for the
// ghosts may have moved them since it was copied, and the pinned table is free
// to be written again as soon as this is queued.
__global__ void k_unit_emit(const SrcUnit *__restrict__ tab, UnitPos P, int nsrc, int total, int self, double SL,
                            const int *__restrict__ off, int ng, double Lx, double Ly, double Lz,
                            const Replica *__restrict__ reps, int *__restrict__ gsrc, int *__restrict__ gword,
                            double4 *__restrict__ gpos, int *__restrict__ gcell, int *__restrict__ gslot,
                            int *__restrict__ gcount) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= total) return;
  const int w = unit_source(tab, nsrc, t);
  const SrcUnit &S = tab[w];
  const int i = t - S.base;
  const double4 q = P.pos[w][i];
  int ox[3], oy[3], oz[3];
  const int nx = unit_axis_options(S, 0, q.x, SL, ox);
  const int ny = unit_axis_options(S, 1, q.y, SL, oy);
  const int nz = unit_axis_options(S, 2, q.z, SL, oz);
  const Replica &R = reps[0];
  const double L[3] = {Lx, Ly, Lz};
  int k = off[t];
  for (int a = 0; a < nx; a++)
    for (int b = 0; b < ny; b++)
      for (int c = 0; c < nz; c++) {
        const int sx = ox[a], sy = oy[b], sz = oz[c];
        if (w == self && !sx && !sy && !sz) continue;  // the particle itself
        if (k >= ng) return;  // cannot happen: off is the scan of k_unit_count
        const int code = (sx + 1) + 3 * (sy + 1) + 9 * (sz + 1);
        const double3 y = image_of(q, code, L);
        gsrc[k] = i;
        gword[k] = ghost_word(code, w);
        gpos[k] = make_double4(y.x, y.y, y.z, 0.0);
        const int cl = cell_of(y.x, y.y, y.z, R);
        gcell[k] = cl;
        gslot[k] = cell_slot(gcount, cl);
        k++;
      }
}

// The row order each unit of a group gave its owned particles at its last
// construction (old index -> new), by unit slot.
struct UnitRowInv {
  const int *inv[kMaxUnits];
};

// Every unit of a group in one launch: the flat index t of a launch over all
// units' items (owned particles, ghosts or blocks) belongs to the last unit u
// with base[u] <= t (units without items share their successor's base).
__device__ __forceinline__ int group_unit_of(const int *base, int n, int t) {
  int lo = 0, hi = n - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (base[mid] <= t) lo = mid; else hi = mid - 1;
  }
  return lo;
}

// The owned particles of every unit (UpdatePositionHalf, fcalculator.cc:22-32,
// with k_drift's operations).
struct GroupDrift {
  double4 *pos[kMaxUnits];
  const double4 *mom[kMaxUnits];
  int base[kMaxUnits + 1];
  int n;
};

__global__ void k_group_drift(GroupDrift G, double dt2) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= G.base[G.n]) return;
  const int u = group_unit_of(G.base, G.n, t);
  const int i = t - G.base[u];
  double4 q = G.pos[u][i];
  const double4 p = G.mom[u][i];
  q.x += p.x * dt2;
  q.y += p.y * dt2;
  q.z += p.z * dt2;
  G.pos[u][i] = q;
}

// The first half drift of the units' owned particles into tmp, the start of a
// run of fused steps.
struct GroupStart {
  const double4 *pos[kMaxUnits];
  const double4 *mom[kMaxUnits];
  double4 *tmp[kMaxUnits];
  int base[kMaxUnits + 1];
  int n;
};

__global__ void k_group_start(GroupStart G, double dt2, RunGate *__restrict__ gate) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t == 0) *gate = RunGate{0, 0, 0};
  if (t >= G.base[G.n]) return;
  const int u = group_unit_of(G.base, G.n, t);
  const int i = t - G.base[u];
  double4 q = G.pos[u][i];
  const double4 p = G.mom[u][i];
  q.x += p.x * dt2;
  q.y += p.y * dt2;
  q.z += p.z * dt2;
  G.tmp[u][i] = q;
}

// The ghosts of every unit from their sources' current positions (k_unit_refresh
// for the whole group); in a run (gate), from the half-drifted ones in src.
struct GroupHalo {
  double4 *pos[kMaxUnits];
  const double4 *src[kMaxUnits];
  const int *gsrc[kMaxUnits];
  const int *gcode[kMaxUnits];
  const int *gunit[kMaxUnits];
  int pn[kMaxUnits];
  int base[kMaxUnits + 1];
  int n;
};

__global__ void k_group_refresh(GroupHalo G, double Lx, double Ly, double Lz, const RunGate *__restrict__ gate) {
  if (run_halted(gate)) return;
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= G.base[G.n]) return;
  const int u = group_unit_of(G.base, G.n, t);
  const int k = t - G.base[u];
  const double L[3] = {Lx, Ly, Lz};
  const double3 y = image_of(G.src[G.gunit[u][k]][G.gsrc[u][k]], G.gcode[u][k], L);
  G.pos[u][G.pn[u] + k] = make_double4(y.x, y.y, y.z, 0.0);
}

// max |p|^2 of every unit: blocks aligned to units (bbase: first block of each
// unit), a partial maximum per block, then one workgroup per unit.
struct GroupMomenta {
  const double4 *mom[kMaxUnits];
  int pn[kMaxUnits];
  int bbase[kMaxUnits + 1];
  int n;
};

__global__ void k_group_max_p2(GroupMomenta G, double *__restrict__ partial) {
  const int b = blockIdx.x;
  const int u = group_unit_of(G.bbase, G.n, b);
  const int i = (b - G.bbase[u]) * blockDim.x + threadIdx.x;
  double v = 0.0;
  if (i < G.pn[u]) {
    const double4 p = G.mom[u][i];
    v = p.x * p.x + p.y * p.y + p.z * p.z;
  }
  block_max_to_partial(v, partial, b);
}

template <class T>
__global__ void k_group_reduce_max(T G, const double *__restrict__ partial,
                                   unsigned long long *__restrict__ out) {
  __shared__ double red[kBlock];
  const int u = blockIdx.x;
  double m = 0.0;
  for (int k = G.bbase[u] + threadIdx.x; k < G.bbase[u + 1]; k += blockDim.x) m = fmax(m, partial[k]);
  red[threadIdx.x] = m;
  __syncthreads();
  for (int o = blockDim.x / 2; o > 0; o >>= 1) {
    if ((int)threadIdx.x < o) red[threadIdx.x] = fmax(red[threadIdx.x], red[threadIdx.x + o]);
    __syncthreads();
  }
  if (threadIdx.x == 0) out[u] = (unsigned long long)__double_as_longlong(red[0]);
}

// PairList::CheckByDisplacement (pairlist.cc:68-121) of the units whose budget
// is spent, all of them in each launch (k_displacement, k_candidates and
// k_candidate_pairs unit by unit otherwise): blocks aligned to units, the
// maxima by k_group_reduce_max.  A check is launches and a wait: 50 steps of
// 500k particles in 2x2x2 units, seven checks among them, took 11.5 ms with
// eight launches, clears and copies per unit and take 10.1 with these four and
// one copy.
constexpr int kCheckUnits = 16;      // units per launch
constexpr int kCheckPairBlocks = 64; // blocks over a unit's candidate pairs
struct GroupCheck {
  const double4 *pos[kCheckUnits], *old[kCheckUnits];
  double *disp[kCheckUnits];
  int *cand[kCheckUnits];
  double margin[kCheckUnits], SL2[kCheckUnits], CL2[kCheckUnits];
  int tn[kCheckUnits], cap[kCheckUnits];
  int bbase[kCheckUnits + 1];
  int n;
};
struct UnitCheck {  // a unit's outcome
  int count, flag;
};

__global__ void k_group_displacement(GroupCheck G, double *__restrict__ partial, UnitCheck *__restrict__ out) {
  const int b = blockIdx.x;
  const int u = group_unit_of(G.bbase, G.n, b);
  const int i = (b - G.bbase[u]) * blockDim.x + threadIdx.x;
  if (i == 0) out[u] = UnitCheck{0, 0};
  double v = 0.0;
  if (i < G.tn[u]) {
    const double4 o = G.old[u][i], q = G.pos[u][i];
    const double dx = o.x - q.x, dy = o.y - q.y, dz = o.z - q.z;
    v = dx * dx + dy * dy + dz * dz;
    G.disp[u][i] = v;
  }
  block_max_to_partial(v, partial, b);
}

__global__ void k_group_candidates(GroupCheck G, const unsigned long long *__restrict__ dmax,
                                   UnitCheck *__restrict__ out) {
  const int b = blockIdx.x;
  const int u = group_unit_of(G.bbase, G.n, b);
  const int i = (b - G.bbase[u]) * blockDim.x + threadIdx.x;
  if (i >= G.tn[u]) return;
  const double c_distance = G.margin[u] - sqrt(__longlong_as_double((long long)dmax[u]));
  if (G.disp[u][i] > c_distance * c_distance) {
    const int k = atomicAdd(&out[u].count, 1);
    if (k < G.cap[u]) G.cand[u][k] = i;
  }
}

__global__ void k_group_candidate_pairs(GroupCheck G, UnitCheck *__restrict__ out) {
  const int u = blockIdx.x / kCheckPairBlocks;
  const int l = out[u].count;
  if (l <= 1 || l >= min(G.tn[u], G.cap[u])) return;
  const double4 *pos = G.pos[u], *old = G.old[u];
  const int *list = G.cand[u];
  const long long total = (long long)l * l;
  for (long long t = (long long)(blockIdx.x % kCheckPairBlocks) * blockDim.x + threadIdx.x; t < total;
       t += (long long)kCheckPairBlocks * blockDim.x) {
    const int a = (int)(t / l), b = (int)(t % l);
    if (b <= a) continue;
    const int i1 = list[a], i2 = list[b];
    const double4 o1 = old[i1], o2 = old[i2];
    double dx = o1.x - o2.x, dy = o1.y - o2.y, dz = o1.z - o2.z;
    if (dx * dx + dy * dy + dz * dz < G.SL2[u]) continue;
    const double4 q1 = pos[i1], q2 = pos[i2];
    dx = q1.x - q2.x;
    dy = q1.y - q2.y;
    dz = q1.z - q2.z;
    if (dx * dx + dy * dy + dz * dz < G.CL2[u]) atomicOr(&out[u].flag, 1);
  }
}

// k_leave_flags for every unit of a group in one launch, the flags of the units
// one after another; after their scan, how many of each unit leave.
struct GroupLeave {
  const double4 *pos[kMaxUnits];
  double s[kMaxUnits], e[kMaxUnits];  // the units' boxes along the direction's axis
  int base[kMaxUnits + 1];
  int n;
};

__global__ void k_group_leave_flags(GroupLeave G, int dir, int *__restrict__ flag) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= G.base[G.n]) return;
  const int u = group_unit_of(G.base, G.n, t);
  const double4 q = G.pos[u][t - G.base[u]];
  const int a = dir >> 1;
  const double v = a == 0 ? q.x : (a == 1 ? q.y : q.z);
  flag[t] = (dir & 1) ? (v >= G.e[u]) : (v < G.s[u]);
}

// off: the exclusive scan of the flags, total[0] their sum; count is in pinned memory
__global__ void k_group_leaving(GroupLeave G, const int *__restrict__ off, const long long *__restrict__ total,
                                int *__restrict__ count) {
  const int u = threadIdx.x;
  if (u >= G.n) return;
  const int all = G.base[G.n];
  auto at = [&](int t) { return t < all ? off[t] : (int)total[0]; };
  count[u] = at(G.base[u + 1]) - at(G.base[u]);
}

// MDUnit::ReceiveParticles (mdunit.cc:104-122): n particles from a send buffer
// appended to a unit's pn.
__global__ void k_receive(double4 *__restrict__ pos, double4 *__restrict__ mom, int *__restrict__ id,
                          int *__restrict__ rep, int pn, int n, const double4 *__restrict__ spos,
                          const double4 *__restrict__ smom, const int *__restrict__ sid) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  pos[pn + i] = spos[i];
  mom[pn + i] = smom[i];
  id[pn + i] = sid[i];
  rep[pn + i] = 0;
}

// A unit's ghost sources follow their source units' row orders: the indices
// were taken before the sources ordered their rows.
__global__ void k_remap_unit_ghosts(int *__restrict__ gsrc, const int *__restrict__ gunit, int ng, UnitRowInv R) {
  const int k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= ng) return;
  gsrc[k] = R.inv[gunit[k]][gsrc[k]];
}

// MDManager::SendBorderParticles for a unit (mdmanager.cc:283-348): every
// ghost from its source unit's current position plus its shift.
__global__ void k_unit_refresh(double4 *__restrict__ pos, const int *__restrict__ gsrc,
                               const int *__restrict__ gcode, const int *__restrict__ gunit, int pn, int ng,
                               UnitPos P, double Lx, double Ly, double Lz) {
  const int k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= ng) return;
  const double L[3] = {Lx, Ly, Lz};
  const double3 y = image_of(P.pos[gunit[k]][gsrc[k]], gcode[k], L);
  pos[pn + k] = make_double4(y.x, y.y, y.z, 0.0);
}

}  // namespace mdgpu
