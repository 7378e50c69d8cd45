// k_block.hip -- cell-block (LDS-staged) neighbour list and EAM passes.
//
// The cell grid is cut into bricks of bx*by*bz cells.  One workgroup owns one
// brick: it stages the brick's halo -- the brick plus one cell on every side,
// periodic images applied once at staging -- into LDS as arrays of doubles
// (x, y, z, and w = F'(rho) in the force pass), then two lanes walk the list of
// each central atom.  List entries are 16-bit halo-local slots, so a pair costs
// three 8-byte LDS reads instead of a global gather, and the list is half the
// size of the global one.
//
// The halo of a brick is an (ex+2)x(ey+2)x(ez+2) box of cells enumerated z-major,
// x fastest.  Atoms of one cell are contiguous in HBM (cell-sorted order) and are
// staged contiguously, cells in enumeration order, so ascending slot order equals
// the visit order of the global build.  The build finds the same pairs as the
// global build and orders short lists by distance; k_block_to_global restores slot
// order, so a converted block list equals the global list entry for entry.
#include "pair_math.hpp"

#include <algorithm>
#include <cmath>
#include <type_traits>

namespace xsmd {
namespace {

struct HaloCell {
  int gstart;  // first atom of the cell in HBM
  int lstart;  // first slot in LDS
  int count;
  int img;     // periodic image, 2 bits per axis as in list entries (bits 26..31 >> 26)
};

struct BlockShape {
  int r;                 // replica
  int cx0, cy0, cz0;     // first central cell
  int ex, ey, ez;        // central cells along each axis (clipped at the grid edge)
  int hx, hy, hz;        // halo dims = e + 2
};

__device__ __forceinline__ BlockShape block_shape(const BlockGeom& g, int64_t b)
{
  BlockShape s;
  // full bricks first (fx fy fz of each replica), then those the grid's edge cuts: the
  // slab of the last brick along x, then along y and z of what is left
  const int64_t full = (int64_t)g.fx * g.fy * g.fz;
  const bool whole = b < g.nfull;
  const int64_t per = whole ? full : (int64_t)g.nbx * g.nby * g.nbz - full;
  int64_t q = whole ? b : b - g.nfull;
  s.r = (int)(q / per);
  q -= (int64_t)s.r * per;
  int wx = g.fx, wy = g.fy, x0 = 0, y0 = 0, z0 = 0;  // extents of the part q counts in, and its origin
  if (!whole) {
    const int64_t sx = (int64_t)(g.nbx - g.fx) * g.nby * g.nbz, sy = (int64_t)(g.nby - g.fy) * g.fx * g.nbz;
    if (q < sx) {
      wx = g.nbx - g.fx;
      wy = g.nby;
      x0 = g.fx;
    } else if (q < sx + sy) {
      q -= sx;
      wy = g.nby - g.fy;
      y0 = g.fy;
    } else {
      q -= sx + sy;
      z0 = g.fz;
    }
  }
  const int ibx = x0 + (int)(q % wx);
  q /= wx;
  const int iby = y0 + (int)(q % wy);
  const int ibz = z0 + (int)(q / wy);
  s.cx0 = ibx * g.bx;
  s.cy0 = iby * g.by;
  s.cz0 = ibz * g.bz;
  s.ex = min(g.bx, g.nx - s.cx0);
  s.ey = min(g.by, g.ny - s.cy0);
  s.ez = min(g.bz, g.nz - s.cz0);
  s.hx = s.ex + 2;
  s.hy = s.ey + 2;
  s.hz = s.ez + 2;
  return s;
}

__device__ __forceinline__ bool wrap_axis(int c, int n, int periodic, int& w, int& k)
{
  k = 0;
  w = c;
  if (c < 0) {
    if (!periodic) return false;
    w = c + n;
    k = -1;
  } else if (c >= n) {
    if (!periodic) return false;
    w = c - n;
    k = 1;
  }
  return true;
}

// Staged halo records in LDS: {x, y, z} of slot c as three doubles at 24 c (one
// address and immediate offsets per neighbour) and, for the passes that read it, w[c]
// in an array of its own.  Random 8-byte reads at a 24-byte stride spread over the
// same 32 bank pairs as reads of 8-byte arrays (6 c mod 64 covers the even banks),
// while 16-byte reads conflict more: the passes measured faster with 8-byte reads
// per component than with the two 16-byte reads of {x, y}, {z, w} records.  Passes
// without w alias w to the x of the records (never read).
struct LRec {
  double* xyz;
  double* w;
  bool has_w;
  __device__ __forceinline__ Pos4 get(int c) const
  {
    const double* r = xyz + 3 * c;
    return {r[0], r[1], r[2], w[has_w ? c : 3 * c]};
  }
  __device__ __forceinline__ void put(int c, const Pos4& p) const
  {
    double* r = xyz + 3 * c;
    r[0] = p.x;
    r[1] = p.y;
    r[2] = p.z;
    if (has_w) w[c] = p.w;
  }
};

// records at p for cap slots plus the far record at slot cap (see stage); returns
// the bytes they take
__device__ __forceinline__ size_t lrec_at(unsigned char* p, int cap, bool with_w, LRec& r)
{
  r.xyz = reinterpret_cast<double*>(p);
  r.w = with_w ? r.xyz + 3 * (size_t)(cap + 1) : r.xyz;
  r.has_w = with_w;
  return (size_t)(cap + 1) * sizeof(double) * (with_w ? 4 : 3);
}

// Halo table of block b in LDS (hc[0..nh)), filled by all threads; returns the
// number of halo atoms.  Ends with __syncthreads().
__device__ int build_halo(const BlockGeom& g, const BlockShape& s, const int* __restrict__ cell_off,
                          HaloCell* hc, int* total_out)
{
  const int nh = s.hx * s.hy * s.hz;
  for (int h = threadIdx.x; h < nh; h += blockDim.x) {
    const int ix = h % s.hx, iy = (h / s.hx) % s.hy, iz = h / (s.hx * s.hy);
    int wx, wy, wz, kx, ky, kz;
    HaloCell e{0, 0, 0, 0};
    if (wrap_axis(s.cx0 - 1 + ix, g.nx, g.px, wx, kx) && wrap_axis(s.cy0 - 1 + iy, g.ny, g.py, wy, ky) &&
        wrap_axis(s.cz0 - 1 + iz, g.nz, g.pz, wz, kz)) {
      const int64_t c = (int64_t)s.r * g.ncell_rep + ((int64_t)wz * g.ny + wy) * g.nx + wx;
      e.gstart = cell_off[c];
      e.count = cell_off[c + 1] - e.gstart;
      e.img = (int)(xsmd_nbr_encode(0u, kx, ky, kz) >> XSMD_NBR_INDEX_BITS);
    }
    hc[h] = e;
  }
  __syncthreads();
  // exclusive prefix sum of the counts in the first wave, 64 cells at a time
  if (threadIdx.x < 64) {
    const int lane = threadIdx.x;
    int carry = 0;
    for (int base = 0; base < nh; base += 64) {
      const int h = base + lane;
      const int cnt = (h < nh) ? hc[h].count : 0;
      int v = cnt;
#pragma unroll
      for (int off = 1; off < 64; off <<= 1) {
        const int t = __shfl_up(v, off);
        if (lane >= off) v += t;
      }
      if (h < nh) hc[h].lstart = carry + v - cnt;
      carry += __shfl(v, 63);
    }
    if (lane == 0) *total_out = carry;
  }
  __syncthreads();
  return *total_out;
}

// Halo atoms of a brick for the list build: f(c, p, e) for slot c, position p (+ image
// shift) and staging entry e (global index and image, encoded like a neighbour entry);
// ends with __syncthreads().  slot_cell (total <= its capacity) first receives the halo
// cell of every slot, so that a thread finds the cell of a slot with one LDS read
// instead of a binary search over the halo table.
template <class F>
__device__ void stage_cells(const BlockShape& s, const HaloCell* hc, int total, const Pos4* __restrict__ pos,
                            const double* L, uint16_t* slot_cell, F f)
{
  const int nh = s.hx * s.hy * s.hz;
  for (int h = threadIdx.x; h < nh; h += blockDim.x) {
    const HaloCell e = hc[h];
    for (int k = 0; k < e.count; k++) slot_cell[e.lstart + k] = (uint16_t)h;
  }
  __syncthreads();
  for (int c = threadIdx.x; c < total; c += blockDim.x) {
    const HaloCell e = hc[slot_cell[c]];
    const uint32_t j = (uint32_t)(e.gstart + (c - e.lstart));
    const double* q = reinterpret_cast<const double*>(pos + j);
    const double2 xy = *reinterpret_cast<const double2*>(q);
    Pos4 p = {xy.x, xy.y, q[2], 0.0};
    const uint32_t code = (uint32_t)e.img << XSMD_NBR_INDEX_BITS;
    if (e.img) {
      p.x = xsmd_image(p.x, xsmd_nbr_img_x(code), L[0]);
      p.y = xsmd_image(p.y, xsmd_nbr_img_y(code), L[1]);
      p.z = xsmd_image(p.z, xsmd_nbr_img_z(code), L[2]);
    }
    f(c, p, j | code);
  }
  __syncthreads();
}

// Brick of this workgroup.  Hardware hands workgroup b to XCD b % 8: each XCD takes a
// contiguous eighth of the full bricks (one contiguous piece of space for its L2), then
// an eighth of the cut ones.  The cut ones last: started among the others they leave a
// last round of full bricks on a mostly idle GPU.  500 k EAM atoms: 2057 full bricks of
// 768 resident workgroups, 391 cut ones.
__device__ __forceinline__ int64_t brick_of_block(int64_t nfull, int64_t nblocks)
{
  const int64_t k = blockIdx.x & 7u, p = blockIdx.x >> 3;
  const int64_t f0 = nfull * k >> 3, nf = (nfull * (k + 1) >> 3) - f0;
  if (p < nf) return f0 + p;
  const int64_t cut = nblocks - nfull, c0 = cut * k >> 3, c = c0 + p - nf;
  return c < (cut * (k + 1) >> 3) ? nfull + c : nblocks;
}

// Two lanes per central atom: the two halves of a wave take the same 32 atoms
// (list build: alternate candidates; EAM passes: even and odd list entries).
constexpr int kPassThreads = 512;
constexpr int kPassAtoms = kPassThreads / 2;

// What the block kernels read.  The build leaves each brick's halo as a staging table, so
// that a pass reaches the positions with one table read instead of rebuilding the halo
// from the cells (cell ranges, a prefix sum, a slot table, three barriers), and holds
// nothing but the records in LDS.  The table costs 4 bytes per halo atom (about 24 per
// atom at 220-atom bricks) written at the build and read by each pass; the chain of
// waits it removes was longer: 8.39 M EAM atoms, mixed: density pass 0.907 -> 0.761 ms,
// force pass 1.350 -> 1.258 ms; 1.05 M argon atoms 0.171 -> 0.141 ms per pass.
// Where the bricks are filled alike, each has room for the densest one; where that would
// more than double the tables (a cluster in a large vacuum box: gigabytes), the bricks'
// parts follow one another as the build's workgroups take them, one atomic each (the
// build of 136 k atoms, whose 700 workgroups start together, takes 86 us so against 80; at
// 1.05 M atoms there is no difference).
constexpr uint32_t kStageAlign = 16;  // a brick's staging entries start on 64 bytes
struct BlockArgs {
  const uint4* __restrict__ head;      // per brick: BrickHead
  const uint32_t* __restrict__ stage;  // global index and image of each halo slot
  const uint32_t* __restrict__ cen;    // central atoms (global index)
  const uint16_t* __restrict__ cen_slot;  // and their slots
  const Pos4* __restrict__ pos;
  const uint8_t* __restrict__ type;
  const BoxDev* __restrict__ box;
  const uint16_t* __restrict__ nbr16;
  const int* __restrict__ nnb;
  int64_t npad;
  int64_t nblocks, nfull;
  int cap;  // halo slots (LDS records)
  double rc2;
  int nmax;            // list capacity
  int split;           // SPLIT passes: log2 of the parts an atom's list is walked in
  const XformDev* xf;  // the staging maps positions to physical space when not NULL
  StepGate gate;       // MD loop
};

// What a brick holds and where its parts of the tables start
struct BrickHead {
  int halo, central, replica;
  uint32_t stage, cen;
  __device__ __forceinline__ static uint4 pack(int halo, int central, int replica, uint32_t stage16, uint32_t cen)
  {
    return make_uint4((uint32_t)halo | (uint32_t)central << 16, (uint32_t)replica, stage16, cen);
  }
  __device__ __forceinline__ explicit BrickHead(const uint4& h)
      : halo((int)(h.x & 0xffffu)), central((int)(h.x >> 16)), replica((int)h.y), stage(h.z * kStageAlign), cen(h.w)
  {
  }
};

// LDS of the block passes: records, then per-record types (block_lds_bytes on the host
// adds up the same sizes)
__device__ __forceinline__ LRec pass_lds(const BlockArgs& a, bool with_type, bool with_w, uint8_t*& ltype)
{
  extern __shared__ __align__(32) unsigned char smem[];
  LRec rec;
  const size_t rb = lrec_at(smem, a.cap, with_w, rec);
  ltype = with_type ? smem + rb : nullptr;
  return rec;
}

// Stages the halo of brick b (head hd) into the records (and types when asked for):
// position + image shift, under a non-identity xform mapped to physical space, so that
// the passes' displacements are physical; w with WITH_W (else the 24 bytes of x, y, z
// are read, not the whole record).  The far record goes to slot cap: list entries past
// an atom's count point there (lslots), so their displacement is finite and longer than
// any cutoff, and the passes mask them by d2 <= rc2 alone.  It lies at least 10^4 A from
// every staged position (which are within the box and its images) and close enough that
// its knot index fits an int.  The caller's __syncthreads() follows.
template <bool WITH_W>
__device__ __forceinline__ void stage(const BlockArgs& a, const BrickHead& hd, const LRec& rec, uint8_t* ltype)
{
  const BoxDev& box = a.box[hd.replica];
  const double* L = box.L;
  if (threadIdx.x == 0) {
    const double far = 4.0 * (fabs(box.lo[0]) + fabs(box.lo[1]) + fabs(box.lo[2]) + L[0] + L[1] + L[2]) + 1e4;
    Pos4 f = {far, far, far, 0.0};
    if (a.xf) {
      xsmd_xform_apply(a.xf->m, &f.x, &f.y, &f.z);
      const double g = 1e4 + 4.0 * fabs(f.x - far) + 4.0 * fabs(f.y - far) + 4.0 * fabs(f.z - far);
      f = {f.x + g, f.y + g, f.z + g, 0.0};  // still far in physical space
    }
    rec.put(a.cap, f);
    if (ltype) ltype[a.cap] = 0;
  }
  const uint32_t* st = a.stage + hd.stage;
  int c = threadIdx.x;
  uint32_t ahead = c < hd.halo ? st[c] : 0u;  // the next entry is on its way while a record is staged
  while (c < hd.halo) {
    const uint32_t e = ahead;
    if (c + kPassThreads < hd.halo) ahead = st[c + kPassThreads];
    const uint32_t j = xsmd_nbr_index(e);
    Pos4 p;
    if constexpr (WITH_W) {
      p = load_pos(a.pos, j);
    } else {
      const double* q = reinterpret_cast<const double*>(a.pos + j);
      const double2 xy = *reinterpret_cast<const double2*>(q);
      p = {xy.x, xy.y, q[2], 0.0};
    }
    if (e >> XSMD_NBR_INDEX_BITS) {
      p.x = xsmd_image(p.x, xsmd_nbr_img_x(e), L[0]);
      p.y = xsmd_image(p.y, xsmd_nbr_img_y(e), L[1]);
      p.z = xsmd_image(p.z, xsmd_nbr_img_z(e), L[2]);
    }
    if (a.xf) xsmd_xform_apply(a.xf->m, &p.x, &p.y, &p.z);
    rec.put(c, p);
    if (ltype) ltype[c] = a.type[j];
    c += kPassThreads;
  }
}

// sum of v over the two halves of the wave (lanes l and l ^ 32)
__device__ __forceinline__ double half_sum(double v)
{
  double a = v, b = v;
  swap_halves<false>(a, b);
  return a + b;
}

// The lanes of a pass.  Two lanes take an atom, the even and the odd entries of its
// list.  SPLIT (bricks of at most 128 atoms, which small systems are cut into): 2 parts
// lanes, each taking every parts-th group of 8 entries, so that a workgroup's 512 lanes
// are busy whatever its atom count.  4000 argon atoms: 27 bricks of 148 atoms, 9.2 us a
// pass -> 125 bricks of 32 atoms, 16 lanes each, 7.0 us.
template <bool SPLIT>
struct PassLanes {
  int half, slot, part, log;
  __device__ __forceinline__ explicit PassLanes(const BlockArgs& a)
  {
    const int l = threadIdx.x & 31, w = threadIdx.x >> 6;
    half = (threadIdx.x >> 5) & 1;
    log = SPLIT ? a.split : 0;
    slot = (w << (5 - log)) + (SPLIT ? l & ((32 >> log) - 1) : l);
    part = SPLIT ? l >> (5 - log) : 0;
  }
  __device__ __forceinline__ int atoms() const { return kPassAtoms >> log; }
  __device__ __forceinline__ int first() const { return half + 8 * part; }  // first entry
  __device__ __forceinline__ int step() const { return 8 << log; }          // to the next group
  __device__ __forceinline__ bool writes() const { return half == 0 && part == 0; }
  // sum over the atom's lanes
  __device__ __forceinline__ double sum(double v) const
  {
    v = half_sum(v);
    if constexpr (SPLIT)
      for (int off = 16; off >= (32 >> log); off >>= 1) v += __shfl_xor(v, off);
    return v;
  }
};

// ---------------------------------------------------------------------------
// list build
// ---------------------------------------------------------------------------
// Destination lane of this lane's key in one stable split pass: keys with a 0 bit
// first (in lane order), then those with a 1.  zeros = ballot of the 0 keys; mbcnt
// counts the 0 keys below this lane, so the 1 keys below it are lane minus that.
// Both candidates are formed and one is selected, so the pass has no branch.
__device__ __forceinline__ int split_dest(bool one, unsigned long long zeros, int lane)
{
  const int zb = (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(zeros >> 32),
                                                __builtin_amdgcn_mbcnt_lo((uint32_t)zeros, 0u));
  const int nz = __popcll(zeros);
  const int d1 = nz + lane - zb;
  return one ? d1 : zb;
}

// Stable sort of one 32-bit key per lane over the 64 lanes of a wave by key bits
// [lo, lo + nbits): least-significant-digit radix sort, one bit per pass (ballot,
// prefix counts, forward permute).  Keys whose sort bits are all ones go last.
__device__ __forceinline__ uint32_t wave_radix_sort(uint32_t key, int lo, int nbits)
{
  const int lane = threadIdx.x & 63;
  for (int bit = lo; bit < lo + nbits; bit++) {
    const bool one = (key >> bit) & 1u;
    const int dest = split_dest(one, __ballot(!one), lane);
    key = (uint32_t)__builtin_amdgcn_ds_permute(dest << 2, (int)key);
  }
  return key;
}

// Lists of at most 64 entries are kept sorted by distance (see k_block_build).
constexpr int kSortRows = 64;

// list order (0, 1), (2, 3), (4, 5), (6, 7) -> the bl_index order (0, 2), (4, 6),
// (1, 3), (5, 7)
__device__ __forceinline__ uint4 group_interleave(const uint32_t (&o)[4])
{
  return make_uint4((o[0] & 0xffffu) | (o[1] << 16), (o[2] & 0xffffu) | (o[3] << 16),
                    (o[0] >> 16) | (o[1] & 0xffff0000u), (o[2] >> 16) | (o[3] & 0xffff0000u));
}

// Smallest value over the 16 lanes of a row (lane order reversed in ever larger
// groups, so four steps reach every lane).
__device__ __forceinline__ double row16_min(double v)
{
  v = fmin(v, dpp_double<kDppXor1>(v));
  v = fmin(v, dpp_double<kDppXor2>(v));
  v = fmin(v, dpp_double<kDppHalfMirror>(v));
  v = fmin(v, dpp_double<kDppMirror>(v));
  return v;
}

// Sorts, ascending, the 64 values that each group of 8 consecutive lanes holds, 8 per
// lane; lane j of the group ends with places 8 j .. 8 j + 7.  A sorting network in
// registers: each lane sorts its own 8 (19 exchanges), then lists of 8, 16 and 32 merge
// pairwise -- the first exchange of a merge pairs mirrored places, the later ones places
// at a fixed distance -- with the partner lane's values as DPP operands.  A wave sorts
// eight lists at once, about 260 instructions; a bitwise radix sort of one list per wave
// needs about 60 for each list and a pass through LDS for every bit.
template <int CTRL>
__device__ __forceinline__ uint32_t lane_swap(uint32_t v)
{
  return (uint32_t)__builtin_amdgcn_mov_dpp((int)v, CTRL, 0xf, 0xf, true);
}
__device__ __forceinline__ void order2(uint32_t& a, uint32_t& b)
{
  const uint32_t lo = min(a, b), hi = max(a, b);
  a = lo;
  b = hi;
}
// the lower places of both partners keep the smaller values; MIRROR: place r against 7 - r
template <int CTRL, bool MIRROR>
__device__ __forceinline__ void order_lanes(uint32_t (&v)[8], bool lower)
{
  uint32_t o[8];
#pragma unroll
  for (int r = 0; r < 8; r++) {
    const uint32_t t = lane_swap<CTRL>(v[MIRROR ? 7 - r : r]);
    o[r] = lower ? min(v[r], t) : max(v[r], t);
  }
#pragma unroll
  for (int r = 0; r < 8; r++) v[r] = o[r];
}
__device__ __forceinline__ void merge8(uint32_t (&v)[8])
{
#pragma unroll
  for (int d = 4; d >= 1; d >>= 1)
#pragma unroll
    for (int r = 0; r < 8; r++)
      if ((r & d) == 0) order2(v[r], v[r + d]);
}
__device__ __forceinline__ void sort64(uint32_t (&v)[8])
{
  const int net[19][2] = {{0, 2}, {1, 3}, {4, 6}, {5, 7}, {0, 4}, {1, 5}, {2, 6}, {3, 7}, {0, 1}, {2, 3},
                          {4, 5}, {6, 7}, {2, 4}, {3, 5}, {1, 4}, {3, 6}, {1, 2}, {3, 4}, {5, 6}};
#pragma unroll
  for (int k = 0; k < 19; k++) order2(v[net[k][0]], v[net[k][1]]);
  const int j = threadIdx.x & 7;
  order_lanes<kDppXor1, true>(v, (j & 1) == 0);  // lanes 0-1
  merge8(v);
  order_lanes<0x1B, true>(v, (j & 2) == 0);      // lanes 0-3 mirrored, quad_perm [3, 2, 1, 0]
  order_lanes<kDppXor1, false>(v, (j & 1) == 0);
  merge8(v);
  order_lanes<kDppHalfMirror, true>(v, (j & 4) == 0);  // lanes 0-7 mirrored
  order_lanes<kDppXor2, false>(v, (j & 2) == 0);
  order_lanes<kDppXor1, false>(v, (j & 1) == 0);
  merge8(v);
}

// base plus the number of set bits of m below this lane
__device__ __forceinline__ int wave_rank(unsigned long long m, int base)
{
  return (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, (uint32_t)base));
}

// LDS written by some lanes of a wave and read by others of the same wave
__device__ __forceinline__ void wave_lds_sync()
{
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Block list: stencil order dz, dy, dx, in-cell order ascending (the order of the
// global build, ascending halo slot), then ordered by distance.
//
// One wave takes one central cell.  All its atoms share the candidates of the 27
// cells around it, so the wave collects them once -- dropping those farther than rl
// from the bounding box of the cell's atoms -- holds them in registers, up to kBuildTile
// at a time, and tests each central atom (the same
// for every lane) against 64 candidates at a time.  A ballot gives each hit its place
// in the atom's list, so no lane waits for another's trip count and only hits are
// stored.  The lists of kBuildAtoms atoms are collected in LDS, sorted together in
// registers and written as whole 8-entry groups, 128 contiguous bytes per group.
//
// The dropped candidates would fail the exact test: for an atom inside the box every
// component of its displacement is at least the gap to the box in magnitude, and
// rounding (subtraction, fma) is monotonic, so d2 >= the box's d2 >= rl2 in floating
// point as well.
//
// The sort orders lists of at most kSortRows entries by d^2 (FP32, cut to 8 significant
// bits), then slot.  At a given list position the atoms of a wave then look up nearby
// spline rows, which cuts the cache lines each table gather of the EAM passes touches
// by about 40 %.
//
// Bound by vector instruction issue (about 130 vector instructions per atom at 53
// entries, the tests of 197 candidates, the sort and the candidate search in equal
// parts) at the three 4-wave workgroups per CU its LDS leaves.  One lane per atom
// walking its own candidates, with the sort as a second kernel, issued twice as many on
// diverging lanes.  8.39 M EAM atoms (53 entries): 4.04 -> 2.65 ms, 1.05 M argon atoms
// (79 entries, unsorted) 0.79 -> 0.42 ms, 4000 argon atoms 112 -> 15 us, the staging
// tables included.  Workgroups of
// 5, 6 or 8 waves measured slower (4.86, 2.84 and 3.70 ms: their waves share the SIMDs
// unevenly or leave LDS for two workgroups).
//
// XF: a non-identity domain xform.  The halo stays in grid space and each candidate's
// displacement is mapped by xf->m before the test, in the operation order of the
// global build (so the lists stay bit-identical); grid-space boxes do not bound
// physical distances, so no candidate is dropped.
constexpr int kBuildThreads = 256;
constexpr int kBuildWaves = kBuildThreads / 64;
constexpr int kBuildAtoms = 8;
constexpr int kBuildTile = 512;  // candidates held in registers

// LDS of the list build: cap + 1 position records of 24 bytes, 16-byte aligned
__host__ __device__ inline size_t build_rec_bytes(int cap) { return ((size_t)(cap + 1) * 24 + 15) / 16 * 16; }

struct BuildArgs {
  BlockGeom g;
  const int* __restrict__ cell_off;
  const Pos4* __restrict__ pos;
  const BoxDev* __restrict__ box;
  const XformDev* __restrict__ xf;
  double rl2;
  uint16_t* __restrict__ nbr16;
  int* __restrict__ nnb;
  int64_t npad;
  int nmax;      // list capacity (a multiple of 8)
  int cap;       // halo slots
  int cand_cap;  // most atoms in the 27 cells of a central cell
  int atoms;     // lists collected per wave, at most kBuildAtoms
  bool sort;     // false: lists stay in stencil order
  // what the passes read instead of the cells (see BlockArgs)
  uint4* __restrict__ head;
  uint32_t* __restrict__ stage;
  uint32_t* __restrict__ cen;
  uint16_t* __restrict__ cen_slot;
  uint32_t* __restrict__ base;  // per atom: start of its brick's staging entries
  int stage_step, cen_step;     // entries per brick; 0: parts handed out through flags[2]
  // [0] longest list beyond nmax, [1] halo beyond cap, [2] table space taken (staging
  // entries in units of kStageAlign, central atoms in the lower half)
  unsigned long long* __restrict__ flags;
  uint32_t* __restrict__ over;  // host memory: set when [0] or [1] is
};

// candidate slots of each wave (the staging uses the same bytes first) and the list rows
__host__ __device__ inline size_t build_cand_bytes(int cap, int cand_cap)
{
  const size_t a = (size_t)cap, b = (size_t)kBuildWaves * cand_cap;
  return ((a > b ? a : b) * sizeof(uint16_t) + 3) / 4 * 4;
}

template <bool XF>
__global__ void __launch_bounds__(kBuildThreads) k_block_build(BuildArgs a)
{
  const int64_t b = brick_of_block(a.g.nfull, a.g.nblocks);
  if (b >= a.g.nblocks) return;
  extern __shared__ __align__(32) unsigned char smem[];
  double3* P = reinterpret_cast<double3*>(smem);
  HaloCell* hc = reinterpret_cast<HaloCell*>(smem + build_rec_bytes(a.cap));
  // [0] halo atoms, [1] next central cell, [2] the brick's staging entries / kStageAlign,
  // (-1: no central atoms), [3] its central atoms in the tables
  int* total_p = reinterpret_cast<int*>(hc + a.g.nh_max);
  int* cell_q = total_p + 4;                                // first central atom of each central cell
  uint16_t* cand_all = reinterpret_cast<uint16_t*>(cell_q + a.g.bx * a.g.by * a.g.bz);
  uint32_t* rows_all = reinterpret_cast<uint32_t*>(reinterpret_cast<unsigned char*>(cand_all) +
                                                   build_cand_bytes(a.cap, a.cand_cap));
  const BlockShape s = block_shape(a.g, b);
  const int total = build_halo(a.g, s, a.cell_off, hc, total_p);
  if (total > a.cap) {  // cannot happen when cap = measured maximum; never write past LDS
    if (threadIdx.x == 0) {
      atomicMax(a.flags + 1, (unsigned long long)total);
      *a.over = 1;
    }
    return;
  }
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int ncell = s.ex * s.ey * s.ez;
  const auto central_cell = [&](int cc) {
    return ((1 + cc / (s.ex * s.ey)) * s.hy + 1 + (cc / s.ex) % s.ey) * s.hx + 1 + cc % s.ex;
  };
  if (wave == 0) {  // central atoms before each central cell
    int carry = 0;
    for (int c0 = 0; c0 < ncell; c0 += 64) {
      const int cc = c0 + lane;
      const int n = cc < ncell ? hc[central_cell(cc)].count : 0;
      int v = n;
#pragma unroll
      for (int off = 1; off < 64; off <<= 1) {
        const int t = __shfl_up(v, off);
        if (lane >= off) v += t;
      }
      if (cc < ncell) cell_q[cc] = carry + v - n;
      carry += __shfl(v, 63);
    }
    if (lane == 0) {
      total_p[1] = 0;
      total_p[2] = -1;
      uint4 head = BrickHead::pack(0, 0, s.r, 0, 0);  // no central atom: nothing to stage
      if (carry > 0) {
        uint32_t at_stage = (uint32_t)b * ((uint32_t)a.stage_step / kStageAlign);
        uint32_t at_cen = (uint32_t)b * (uint32_t)a.cen_step;
        if (a.stage_step == 0) {
          const unsigned long long need = (unsigned long long)((total + kStageAlign - 1) / kStageAlign) << 32;
          const unsigned long long at = atomicAdd(a.flags + 2, need | (unsigned long long)carry);
          at_stage = (uint32_t)(at >> 32);
          at_cen = (uint32_t)at;
        }
        total_p[2] = (int)at_stage;
        total_p[3] = (int)at_cen;
        head = BrickHead::pack(total, carry, s.r, at_stage, at_cen);
      }
      a.head[b] = head;
    }
  }
  const BoxDev bx = a.box[s.r];
  stage_cells(s, hc, total, a.pos, bx.L, cand_all, [&](int c, const Pos4& p, uint32_t e) {
    P[c] = double3{p.x, p.y, p.z};
    if (total_p[2] >= 0) a.stage[(uint32_t)total_p[2] * kStageAlign + (uint32_t)c] = e;
  });
  const uint32_t stage0 = (uint32_t)__builtin_amdgcn_readfirstlane(total_p[2]) * kStageAlign;
  const uint32_t cen0 = (uint32_t)__builtin_amdgcn_readfirstlane(total_p[3]);

  uint16_t* cand = cand_all + (size_t)wave * a.cand_cap;
  const int stride = a.nmax + 1;  // odd, so the group loads of 8 rows start in distinct banks
  uint32_t* rows = rows_all + (size_t)wave * a.atoms * stride;
  // bricks of fewer cells than waves: several waves share a cell's atoms
  const int parts = ncell >= kBuildWaves ? 1 : kBuildWaves / ncell;
  int nrow = 0;         // lists in the rows
  int cnt = 0, gi = 0;  // lane k: entries and atom of row k
  // the collected lists out: counts, then whole groups, 8 lanes per atom and one group
  // each (places past the count hold whatever the row held; readers stop at the count)
  const auto flush = [&]() {
    wave_lds_sync();
    if (lane < nrow) {
      a.nnb[gi] = cnt;
      if (cnt > a.nmax) {
        atomicMax(a.flags, (unsigned long long)cnt);
        *a.over = 1;
      }
    }
    const int la = lane >> 3, j = lane & 7;
    const int ca = la < nrow ? min(__shfl(cnt, la), a.nmax) : 0;
    const int64_t ga = __shfl(gi, la);
    const uint32_t* row = rows + (la < nrow ? la : 0) * stride;
    const auto put = [&](int grp, const uint32_t (&e)[8]) {
      uint32_t o[4];
#pragma unroll
      for (int k = 0; k < 4; k++) o[k] = (e[2 * k] & 0xffffu) | (e[2 * k + 1] << 16);
      *reinterpret_cast<uint4*>(a.nbr16 + bl_index(a.npad, ga, 8 * grp)) = group_interleave(o);
    };
    const bool sorts = a.sort && ca <= kSortRows;
    if (__any(sorts)) {
      uint32_t v[8];
#pragma unroll
      for (int r = 0; r < 8; r++) v[r] = j + 8 * r < (sorts ? ca : 0) ? row[j + 8 * r] : 0xffffffffu;
      sort64(v);
      if (sorts && 8 * j < ca) put(j, v);
    }
    if (!sorts)
      for (int grp = j; 8 * grp < ca; grp += 8) {
        uint32_t v[8];
#pragma unroll
        for (int r = 0; r < 8; r++) v[r] = row[8 * grp + r];
        put(grp, v);
      }
    wave_lds_sync();
    nrow = 0;
    cnt = 0;
  };
  for (;;) {
    int cc = 0;
    if (lane == 0) cc = atomicAdd(total_p + 1, 1);
    cc = __builtin_amdgcn_readfirstlane(cc);
    if (cc >= ncell * parts) break;
    const int part = cc % parts;
    cc /= parts;
    const int h = central_cell(cc);
    const int all = __builtin_amdgcn_readfirstlane(hc[h].count);
    const int skip = all * part / parts, nat = all * (part + 1) / parts - skip;
    if (nat == 0) continue;
    const int l0 = __builtin_amdgcn_readfirstlane(hc[h].lstart) + skip;
    const int g0 = __builtin_amdgcn_readfirstlane(hc[h].gstart) + skip;
    const uint32_t q0 = cen0 + (uint32_t)(cell_q[cc] + skip);
    for (int k = lane; k < nat; k += 64) {
      a.cen[q0 + k] = (uint32_t)(g0 + k);
      a.cen_slot[q0 + k] = (uint16_t)(l0 + k);
      a.base[g0 + k] = stage0;
    }
    double lx = 1e300, ly = 1e300, lz = 1e300, ux = -1e300, uy = -1e300, uz = -1e300;
    if constexpr (!XF) {
      for (int k = lane & 15; k < nat; k += 16) {
        const double3 p = P[l0 + k];
        lx = fmin(lx, p.x);
        ly = fmin(ly, p.y);
        lz = fmin(lz, p.z);
        ux = fmax(ux, p.x);
        uy = fmax(uy, p.y);
        uz = fmax(uz, p.z);
      }
      lx = row16_min(lx);
      ly = row16_min(ly);
      lz = row16_min(lz);
      ux = -row16_min(-ux);
      uy = -row16_min(-uy);
      uz = -row16_min(-uz);
    }
    // candidates, in ascending slot order; lane k < 9 holds the slots of stencil row k
    const int rk = min(lane, 8);
    const int rh = h + ((rk / 3 - 1) * s.hy + (rk % 3 - 1)) * s.hx - 1;
    const int row_beg = hc[rh].lstart, row_end = hc[rh + 2].lstart + hc[rh + 2].count;
    int nc = 0;
    for (int row = 0; row < 9; row++) {
      const int beg = __builtin_amdgcn_readlane(row_beg, row), end = __builtin_amdgcn_readlane(row_end, row);
      for (int c0 = beg; c0 < end; c0 += 64) {
        const int c = c0 + lane;
        bool keep = c < end;
        if constexpr (!XF) {
          const double3 p = P[min(c, a.cap)];
          const double gx = fmax(fmax(lx - p.x, p.x - ux), 0.0);
          const double gy = fmax(fmax(ly - p.y, p.y - uy), 0.0);
          const double gz = fmax(fmax(lz - p.z, p.z - uz), 0.0);
          keep = keep && xsmd_d2(gx, gy, gz) < a.rl2;
        }
        const unsigned long long m = __builtin_amdgcn_ballot_w64(keep);
        const int at = wave_rank(m, nc);
        if (keep) cand[at] = (uint16_t)c;
        nc += __popcll(m);
      }
    }
    wave_lds_sync();
    // T x 64 candidates from t0 on against atoms a0 .. a0 + nb - 1, lists into rows nrow,
    // nrow + 1, ...; with ALL (every candidate of the cell fits) the full rows go out
    // between atoms, so the candidates are loaded once per cell
    const auto test = [&](auto tiles, auto all, int t0, int a0, int nb) {
      constexpr int T = decltype(tiles)::value;
      constexpr bool ALL = decltype(all)::value;
      double cx[T], cy[T], cz[T];
      int cs[T];
#pragma unroll
      for (int t = 0; t < T; t++) {
        const int k = t0 + 64 * t + lane;
        cs[t] = k < nc ? (int)cand[k] : a.cap;
        const double3 p = P[cs[t]];
        cx[t] = k < nc ? p.x : 1e200;  // no candidate: its d2 is infinite
        cy[t] = p.y;
        cz[t] = p.z;
      }
      for (int k = 0; k < nb; k++) {
        const int local = l0 + a0 + k, to_row = ALL ? nrow : nrow + k;
        const double3 pi = P[local];
        uint32_t* row = rows + to_row * stride;
        int base = ALL ? 0 : __builtin_amdgcn_readlane(cnt, to_row);
        double d2[T];
        bool in[T];
        uint32_t* to[T];
#pragma unroll
        for (int t = 0; t < T; t++) {
          double dx = cx[t] - pi.x, dy = cy[t] - pi.y, dz = cz[t] - pi.z;
          if constexpr (XF) xsmd_xform_apply(a.xf->m, &dx, &dy, &dz);
          d2[t] = xsmd_d2(dx, dy, dz);
          in[t] = d2[t] < a.rl2 && cs[t] != local;
          const unsigned long long m = __builtin_amdgcn_ballot_w64(d2[t] < a.rl2) &
                                       ~__builtin_amdgcn_ballot_w64(cs[t] == local);
          to[t] = row + base + min(wave_rank(m, 0), a.nmax - base);  // past the capacity: the row's spare word
          base += __popcll(m);
        }
#pragma unroll
        for (int t = 0; t < T; t++)
          if (in[t]) *to[t] = (__float_as_uint((float)d2[t]) & 0xffff0000u) | (uint32_t)cs[t];
        cnt = lane == to_row ? base : cnt;
        if constexpr (ALL) {
          gi = lane == to_row ? g0 + k : gi;
          if (++nrow == a.atoms) flush();
        }
      }
    };
    const auto pick = [&](int t0, auto all, int a0, int nb) {
      const int left = nc - t0;
      if (left > 384) test(std::integral_constant<int, 8>{}, all, t0, a0, nb);
      else if (left > 256) test(std::integral_constant<int, 6>{}, all, t0, a0, nb);
      else if (left > 192) test(std::integral_constant<int, 4>{}, all, t0, a0, nb);
      else if (left > 128) test(std::integral_constant<int, 3>{}, all, t0, a0, nb);
      else test(std::integral_constant<int, 2>{}, all, t0, a0, nb);
    };
    if (nc <= kBuildTile) {
      pick(0, std::true_type{}, 0, nat);
      continue;
    }
    for (int a0 = 0; a0 < nat;) {
      const int nb = min(a.atoms - nrow, nat - a0);
      for (int t0 = 0; t0 < nc; t0 += kBuildTile) pick(t0, std::false_type{}, a0, nb);
      if (lane >= nrow && lane < nrow + nb) gi = g0 + a0 + lane - nrow;
      nrow += nb;
      a0 += nb;
      if (nrow == a.atoms) flush();
    }
  }
  if (nrow > 0) flush();
}

// Block-local entries -> global (index, image) entries of the same list, in the
// stencil order of the global build: a distance-sorted list goes back to ascending
// halo slot order (the stencil order) first.  A slot's staging entry is its global
// entry.  One wave per central atom.
__global__ void __launch_bounds__(256) k_block_to_global(BlockArgs a, uint32_t* __restrict__ nbr)
{
  const int64_t b = brick_of_block(a.nfull, a.nblocks);
  if (b >= a.nblocks) return;
  const BrickHead hd(a.head[b]);
  const uint32_t* stage = a.stage + hd.stage;
  const int lane = threadIdx.x & 63;
  for (int q = threadIdx.x >> 6; q < hd.central; q += blockDim.x >> 6) {
    const int64_t i = a.cen[hd.cen + (uint32_t)q];
    const int cnt = a.nnb[i];
    if (cnt <= kSortRows) {
      uint32_t key = 0xffffu;
      if (lane < cnt) key = a.nbr16[bl_index(a.npad, i, lane)];
      key = wave_radix_sort(key, 0, 16);
      if (lane < cnt) nbr[(int64_t)lane * a.npad + i] = stage[key];
    } else {
      for (int k = lane; k < cnt; k += 64) nbr[(int64_t)k * a.npad + i] = stage[a.nbr16[bl_index(a.npad, i, k)]];
    }
  }
}

// Sizes the LDS of the block kernels and the staging table: the most halo atoms and
// central atoms of a brick, the most atoms in the 27 cells of a central cell, and the
// staging entries of the bricks that hold atoms, in units of kStageAlign.  Each workgroup
// writes its four to host memory, where they are put together (atomics on four words
// took 20 us of the kernel's 25 at 700 bricks).  One wave per brick, one lane
// per halo cell (a thread per brick reads its cells one after the other: 33 us for a
// single brick of 125 cells, against 4 us).  Clears the build's flags, which follows.
constexpr int kHaloMaxWaves = 4;
__global__ void __launch_bounds__(64 * kHaloMaxWaves) k_block_halo_max(BlockGeom g, const int* __restrict__ cell_off,
                                                                       uint32_t* __restrict__ out,
                                                                       unsigned long long* __restrict__ flags)
{
  if (blockIdx.x == 0 && threadIdx.x < 3) flags[threadIdx.x] = 0;
  __shared__ int cnt_all[kHaloMaxWaves][kMaxHaloCells];
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  int* cnt = cnt_all[wave];
  int m_total = 0, m_central = 0, m_cand = 0;
  uint32_t entries = 0;
  for (int64_t b = (int64_t)blockIdx.x * kHaloMaxWaves + wave; b < g.nblocks; b += (int64_t)gridDim.x * kHaloMaxWaves) {
    const BlockShape s = block_shape(g, b);
    const int nh = s.hx * s.hy * s.hz;
    int total = 0, central = 0;
    for (int h = lane; h < nh; h += 64) {
      const int ix = h % s.hx, iy = (h / s.hx) % s.hy, iz = h / (s.hx * s.hy);
      int wx, wy, wz, kx, ky, kz, n = 0;
      if (wrap_axis(s.cx0 - 1 + ix, g.nx, g.px, wx, kx) && wrap_axis(s.cy0 - 1 + iy, g.ny, g.py, wy, ky) &&
          wrap_axis(s.cz0 - 1 + iz, g.nz, g.pz, wz, kz)) {
        const int64_t c = (int64_t)s.r * g.ncell_rep + ((int64_t)wz * g.ny + wy) * g.nx + wx;
        n = cell_off[c + 1] - cell_off[c];
      }
      cnt[h] = n;
      total += n;
      if (ix >= 1 && ix <= s.ex && iy >= 1 && iy <= s.ey && iz >= 1 && iz <= s.ez) central += n;
    }
    wave_lds_sync();
    const int ncell = s.ex * s.ey * s.ez;
    for (int cc = lane; cc < ncell; cc += 64) {
      const int h = ((1 + cc / (s.ex * s.ey)) * s.hy + 1 + (cc / s.ex) % s.ey) * s.hx + 1 + cc % s.ex;
      int n = 0;
      for (int row = 0; row < 9; row++) {
        const int h0 = h + ((row / 3 - 1) * s.hy + (row % 3 - 1)) * s.hx;
        n += cnt[h0 - 1] + cnt[h0] + cnt[h0 + 1];
      }
      m_cand = max(m_cand, n);
    }
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) {
      total += __shfl_xor(total, off);
      central += __shfl_xor(central, off);
    }
    m_total = max(m_total, total);
    if (central > 0) entries += (uint32_t)(total + kStageAlign - 1) / kStageAlign;
    m_central = max(m_central, central);
    wave_lds_sync();
  }
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) m_cand = max(m_cand, __shfl_xor(m_cand, off));
  __shared__ uint32_t best[kHaloMaxWaves][4];
  if (lane == 0) {
    best[wave][3] = entries;
    best[wave][0] = m_total;
    best[wave][1] = m_central;
    best[wave][2] = m_cand;
  }
  __syncthreads();
  if (threadIdx.x < 4) {
    uint32_t v = best[0][threadIdx.x];
    for (int w = 1; w < kHaloMaxWaves; w++)
      v = threadIdx.x == 3 ? v + best[w][3] : max(v, best[w][threadIdx.x]);
    out[4 * blockIdx.x + threadIdx.x] = v;
  }
}

// ---------------------------------------------------------------------------
// EAM passes on the block list
// ---------------------------------------------------------------------------
constexpr int kBBatch = 4;
// EAM passes run two lanes per central atom: the two halves of a wave take the
// even and odd list entries of the same 32 atoms and combine their sums with one
// cross-half exchange, doubling the waves that hide the table-gather latency for
// the LDS a brick needs.
// Minimum waves per SIMD the register allocation must allow: three 8-wave
// workgroups per CU (what the LDS of a ~200-atom brick permits) need 6; the
// virial form of the force pass carries 9 more sums and is held to 4.
template <bool VIRIAL>
constexpr int kPassWaves = VIRIAL ? 4 : 6;

// FP64 displacement to the staged record of slot c (image already applied)
struct LNb {
  double x, y, z, d2, w;
  int c;
  bool in;
};

// List slots of entries k0, k0 + 2, k0 + 4, k0 + 6 of atom gi (this lane's parity of
// the list).  k0 = half + 8 q, so one 8-byte word brings the four entries of group q
// (in bounds for k0 < nmax); lslots turns entries past this atom's count into the far
// record (a pair longer than any cutoff).  The passes load the next group's word one
// iteration ahead (none at the end of the list).  In the bl_index layout the word of
// (gi, half + 8 q) is word 2 gi + half of group q, whose words start q * 2 npad words
// into the array; a lane steps its own pointer, one 64-bit add (from the group's number,
// which the compiler cannot know to be the same in every lane, it took eight
// instructions of the 40 to 80 per list word).
template <bool SPLIT>
struct LWords {
  const uint2* at;  // this lane's word of its current group
  int64_t step;     // words to its next group
  __device__ __forceinline__ LWords(const BlockArgs& a, int64_t gi, const PassLanes<SPLIT>& ln)
      : at(reinterpret_cast<const uint2*>(a.nbr16) + 2 * gi + ln.half), step(2 * a.npad)
  {
    if constexpr (SPLIT) {
      at += ln.part * step;
      step <<= ln.log;
    }
  }
  __device__ __forceinline__ uint2 first() const { return *at; }
  __device__ __forceinline__ uint2 next()
  {
    at += step;
    return *at;
  }
};
// A central atom on its way: its index and slot, then the length of its list and the
// lane's first list word.  The first atom of each lane is fetched while the halo is
// staged, so that the passes do not wait for these loads one after the other behind the
// barrier.
template <bool SPLIT>
struct PassAtom {
  int64_t gi = 0;
  int slot = 0, cnt = 0;
  uint2 w = {0u, 0u};
  __device__ __forceinline__ void index(const BlockArgs& a, const BrickHead& hd, int q)
  {
    gi = a.cen[hd.cen + (uint32_t)q];
    slot = a.cen_slot[hd.cen + (uint32_t)q];
  }
  __device__ __forceinline__ void list(const BlockArgs& a, const PassLanes<SPLIT>& ln)
  {
    cnt = a.nnb[gi];
    // a part's first group may lie beyond the lists' capacity
    if (!SPLIT || 8 * ln.part < a.nmax) w = LWords<SPLIT>(a, gi, ln).first();
  }
  __device__ __forceinline__ void fetch(const BlockArgs& a, const BrickHead& hd, int q, const PassLanes<SPLIT>& ln)
  {
    cnt = 0;
    if (q >= hd.central) return;
    index(a, hd, q);
    list(a, ln);
  }
};
__device__ __forceinline__ void lslots(uint2 w, int far_slot, int k0, int cnt, int (&c)[4])
{
  const int raw[4] = {(int)(w.x & 0xffffu), (int)(w.x >> 16), (int)(w.y & 0xffffu), (int)(w.y >> 16)};
  // slots are 16-bit: saying so of the far slot too keeps the record addresses 24-bit
  // multiplies instead of 64-bit ones
  const int fs = far_slot & 0xffff;
#pragma unroll
  for (int u = 0; u < 4; u++) c[u] = (k0 + 2 * u < cnt) ? raw[u] : fs;
}

// FP64 table rows are loaded by pairs of neighbouring lanes (pm::RowPair), which hold
// consecutive atoms: both stay to the end of the longer list, and a lane whose neighbour
// has the brick's last atom runs along with an empty one.
template <class Real>
constexpr bool kPaired = sizeof(Real) == 8;
template <class Real>
__device__ __forceinline__ int pair_end(int cnt)
{
  if constexpr (kPaired<Real>) return max(cnt, (int)pm::dpp_xor1((uint32_t)cnt));
  return cnt;
}

// neighbour records of slots c[0..U-1] (entries k0, k0 + 2, ...)
template <int U>
__device__ __forceinline__ void lgather(const BlockArgs& a, const LRec& rec, const int* c, int k0, int cnt,
                                        const Pos4& pi, LNb (&nb)[U])
{
#pragma unroll
  for (int u = 0; u < U; u++) {
    const Pos4 pj = rec.get(c[u]);
    nb[u].x = pj.x - pi.x;
    nb[u].y = pj.y - pi.y;
    nb[u].z = pj.z - pi.z;
    nb[u].d2 = xsmd_d2(nb[u].x, nb[u].y, nb[u].z);
    nb[u].w = pj.w;
    nb[u].c = c[u];
    nb[u].in = nb[u].d2 <= a.rc2;  // entries past the count read the far record
  }
}

// rho_i, then (EMB) F(rho_i) and F'(rho_i) for the central atoms of one brick
template <class Real, bool MULTI, bool EMB, bool ENERGY, bool SET_EP, bool SPLIT>
__global__ void __launch_bounds__(kPassThreads, kPassWaves<SPLIT>) k_block_eam_rho(BlockArgs a, EamTabDev<Real> t,
                                                                const Real* __restrict__ pair,
                                                                double* __restrict__ rho_io,
                                                                double* __restrict__ pos_w, double* __restrict__ ep)
{
  const int64_t b = brick_of_block(a.nfull, a.nblocks);
  if (b >= a.nblocks || a.gate.closed()) return;
  uint8_t* ltype;
  const LRec rec = pass_lds(a, MULTI, false, ltype);
  const BrickHead hd(a.head[b]);
  const PassLanes<SPLIT> ln(a);
  PassAtom<SPLIT> at;
  if (ln.slot < hd.central) at.index(a, hd, ln.slot);
  stage<false>(a, hd, rec, ltype);
  if (ln.slot < hd.central) at.list(a, ln);
  __syncthreads();
  for (int q = ln.slot; (kPaired<Real> ? q & ~1 : q) < hd.central; q += ln.atoms(), at.fetch(a, hd, q, ln)) {
    const int64_t gi = at.gi;
    const int slot = at.slot;
    const Pos4 pi = rec.get(slot);
    const int ti = MULTI ? ltype[slot] : 0;
    const bool oni = !MULTI || pm::eam_on(t, ti);
    const int cnt = oni ? at.cnt : 0;
    double rho = 0.0;
    LWords<SPLIT> lw(a, gi, ln);
    uint2 wnext = at.w;
    const int end = pair_end<Real>(cnt);
    for (int k0 = ln.first(); k0 < end; k0 += ln.step()) {
      const uint2 w = wnext;
      if (k0 + ln.step() < end) wnext = lw.next();
      int c[kBBatch];
      lslots(w, a.cap, k0, cnt, c);
      LNb nb[kBBatch];
      lgather<kBBatch>(a, rec, c, k0, cnt, pi, nb);
      if constexpr (MULTI) {
#pragma unroll
        for (int u = 0; u < kBBatch; u++) nb[u].in = nb[u].in && pm::eam_on(t, ltype[nb[u].c]);
      }
      // a batch with no pair inside rc on any lane of the wave (the tails of the
      // distance-sorted lists) skips the table reads; skipped terms would add 0
      bool any = false;
#pragma unroll
      for (int u = 0; u < kBBatch; u++) any |= nb[u].in;
      if (!__any(any)) continue;
#pragma unroll
      for (int u = 0; u < kBBatch; u++) {
        const int tj = MULTI ? ltype[nb[u].c] : 0;
        // every d2 here is finite and positive (entries past the count read the far
        // record), so the knot index needs no guard value; the sum masks by `in`
        const Real val = pm::eam_rho_knot<Real, MULTI, kPaired<Real>>(t, pair, ti, tj, nb[u].d2, true);
        rho += (double)(nb[u].in ? val : Real(0));
      }
    }
    rho = ln.sum(rho);
    if (ln.writes() && (!kPaired<Real> || q < hd.central)) {
      rho_io[gi] = rho;
      if constexpr (EMB) {
        Real F, Fp;
        pm::embed(t, ti, rho, F, Fp);
        if (!oni) F = Fp = Real(0);  // a disabled species keeps rho_dEmb = 0 and adds no F
        pos_w[4 * gi + 3] = (double)Fp;
        if constexpr (ENERGY) {
          if constexpr (SET_EP) ep[gi] = (double)F;
          else ep[gi] += (double)F;
        }
      }
    }
  }
}

template <class Real, bool MULTI, bool ENERGY, bool VIRIAL, bool FUSED, bool DRIFT, bool SPLIT>
__global__ void __launch_bounds__(kPassThreads, kPassWaves<VIRIAL || SPLIT>) k_block_eam_force(BlockArgs a, EamTabDev<Real> t,
                                                                  const Real* __restrict__ pair, pm::Outputs o,
                                                                  pm::Drift dr)
{
  static_assert(!DRIFT || (FUSED && !ENERGY && !VIRIAL), "the drift epilogue is the plain MD-loop step");
  const int64_t b = brick_of_block(a.nfull, a.nblocks);
  if (b >= a.nblocks || a.gate.closed()) return;
  uint8_t* ltype;
  const LRec rec = pass_lds(a, MULTI, true, ltype);
  const BrickHead hd(a.head[b]);
  const PassLanes<SPLIT> ln(a);
  PassAtom<SPLIT> at;
  if (ln.slot < hd.central) at.index(a, hd, ln.slot);
  stage<true>(a, hd, rec, ltype);
  if (ln.slot < hd.central) at.list(a, ln);
  __syncthreads();
  for (int q = ln.slot; (kPaired<Real> ? q & ~1 : q) < hd.central; q += ln.atoms(), at.fetch(a, hd, q, ln)) {
    const int64_t gi = at.gi;
    const int slot = at.slot;
    const Pos4 pi = rec.get(slot);
    const int ti = MULTI ? ltype[slot] : 0;
    const Real fpi = (Real)pi.w;
    const int cnt = (!MULTI || pm::eam_on(t, ti)) ? at.cnt : 0;
    double fx = 0.0, fy = 0.0, fz = 0.0, e = 0.0;
    double v[9] = {0, 0, 0, 0, 0, 0, 0, 0, 0};
    LWords<SPLIT> lw(a, gi, ln);
    uint2 wnext = at.w;
    const int end = pair_end<Real>(cnt);
    for (int k0 = ln.first(); k0 < end; k0 += ln.step()) {
      const uint2 w = wnext;
      if (k0 + ln.step() < end) wnext = lw.next();
      int c[kBBatch];
      lslots(w, a.cap, k0, cnt, c);
      // two entries at a time: their four table rows stay in flight together within
      // the register budget of six waves per SIMD (the barrier keeps the compiler
      // from hoisting the second pair's gathers above the first pair's rows)
#pragma unroll
      for (int sub = 0; sub < kBBatch; sub += 2) {
        LNb nb[2];
        lgather<2>(a, rec, c + sub, k0 + 2 * sub, cnt, pi, nb);
        if constexpr (MULTI) {
          nb[0].in = nb[0].in && pm::eam_on(t, ltype[nb[0].c]);
          nb[1].in = nb[1].in && pm::eam_on(t, ltype[nb[1].c]);
        }
        if (!__any(nb[0].in || nb[1].in)) continue;  // as in the density pass
        auto add = [&](const LNb& q, bool in, Real fp, Real ph) {
          const double fpair = in ? (double)fp : 0.0;
          const double fe0 = q.x * fpair, fe1 = q.y * fpair, fe2 = q.z * fpair;
          fx += fe0;
          fy += fe1;
          fz += fe2;
          if constexpr (ENERGY) e += in ? 0.5 * (double)ph : 0.0;
          if constexpr (VIRIAL) pm::add_virial(v, fe0, fe1, fe2, q.x, q.y, q.z);
        };
        if constexpr (pm::kSTable<Real, MULTI>) {
          // FP32 single element: the s-table; the knot rows for pairs outside its range
          const int tj[2] = {0, 0};
          Real fp_r[2], phi[2] = {Real(0), Real(0)};
          bool slow[2];
          pm::eam_pair_batch<Real, MULTI, ENERGY, 2>(t, pair, ti, tj, fpi, nb, fp_r, phi, slow);
#pragma unroll
          for (int u = 0; u < 2; u++) add(nb[u], nb[u].in && !slow[u], fp_r[u], phi[u]);
          if (__builtin_expect(__any(slow[0] || slow[1]), 0)) {
#pragma unroll
            for (int u = 0; u < 2; u++)
              if (slow[u]) {
                Real fp, ph = Real(0);
                pm::eam_pair_knot<Real, false>(t, pair, 0, 0, fpi, (Real)nb[u].w, nb[u].d2, true, fp, ph);
                add(nb[u], true, fp, ph);
              }
          }
        } else {
#pragma unroll
          for (int u = 0; u < 2; u++) {
            const int tj = MULTI ? ltype[nb[u].c] : 0;
            Real fp_r, phi;
            pm::eam_pair_knot<Real, MULTI, kPaired<Real>>(t, pair, ti, tj, fpi, (Real)nb[u].w, nb[u].d2, true, fp_r, phi);
            add(nb[u], nb[u].in, fp_r, phi);
          }
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    fx = ln.sum(fx);
    fy = ln.sum(fy);
    fz = ln.sum(fz);
    if constexpr (ENERGY) e = ln.sum(e);
    if constexpr (VIRIAL) {
#pragma unroll
      for (int k = 0; k < 9; k++) v[k] = ln.sum(v[k]);
    }
    if (ln.writes() && (!kPaired<Real> || q < hd.central)) {
      if constexpr (DRIFT) pm::write_outputs_drift(o, dr, gi, pi, fx, fy, fz);
      else pm::write_outputs<ENERGY, VIRIAL, FUSED>(o, gi, fx, fy, fz, e, v);
    }
  }
}

// First sweep of the EAM adjoint (formulas in k_adjoint.hip): drho_i = sum_j rho'_tj(r_ij) s_ij
// with s_ij = u_ij . (g_i - g_j), then lambda_i = F''(rho_i) drho_i into the w of g_i's
// record.  The density pass with the neighbours' loss gradients staged beside their
// positions (48 bytes a slot, two workgroups per CU at 220-atom bricks); distances, knot
// fractions and sums FP64, Real is the table's storage.
struct AdjB1Args {
  Pos4* gvec;         // g_i (dL/dF_i) in cell order; lambda_i into w
  double* drho;
  const double* rho;  // checkpointed rho_i
  const void* frho;   // rows [c3 c4 c5 c6 | c0 c1 c2 0]
  int nrho;
  double rdrho, conv;
};

template <class Real, bool MULTI, bool SPLIT>
__global__ void __launch_bounds__(kPassThreads, 4) k_block_adj_b1(BlockArgs a, EamTabDev<Real> t, AdjB1Args g)
{
  const int64_t b = brick_of_block(a.nfull, a.nblocks);
  if (b >= a.nblocks) return;
  extern __shared__ __align__(32) unsigned char smem[];
  LRec rec;
  const size_t rb = lrec_at(smem, a.cap, false, rec);
  double* gl = reinterpret_cast<double*>(smem + rb);  // g of slot c at 3 c
  uint8_t* ltype = MULTI ? smem + 2 * rb : nullptr;
  const BrickHead hd(a.head[b]);
  const PassLanes<SPLIT> ln(a);
  PassAtom<SPLIT> at;
  if (ln.slot < hd.central) at.index(a, hd, ln.slot);
  stage<false>(a, hd, rec, ltype);
  for (int c = threadIdx.x; c < hd.halo; c += kPassThreads) {
    const double* q = reinterpret_cast<const double*>(g.gvec + xsmd_nbr_index(a.stage[hd.stage + (uint32_t)c]));
    const double2 xy = *reinterpret_cast<const double2*>(q);
    gl[3 * c] = xy.x;
    gl[3 * c + 1] = xy.y;
    gl[3 * c + 2] = q[2];
  }
  if (threadIdx.x < 3) gl[3 * a.cap + threadIdx.x] = 0.0;  // the far record
  if (ln.slot < hd.central) at.list(a, ln);
  __syncthreads();
  for (int q = ln.slot; q < hd.central; q += ln.atoms(), at.fetch(a, hd, q, ln)) {
    const int64_t gi = at.gi;
    const int slot = at.slot;
    const Pos4 pi = rec.get(slot);
    const double g0 = gl[3 * slot], g1 = gl[3 * slot + 1], g2 = gl[3 * slot + 2];
    const int ti = MULTI ? ltype[slot] : 0;
    const bool oni = !MULTI || pm::eam_on(t, ti);
    const int cnt = oni ? at.cnt : 0;
    double drho = 0.0;
    LWords<SPLIT> lw(a, gi, ln);
    uint2 wnext = at.w;
    for (int k0 = ln.first(); k0 < cnt; k0 += ln.step()) {
      const uint2 w = wnext;
      if (k0 + ln.step() < cnt) wnext = lw.next();
      int c[kBBatch];
      lslots(w, a.cap, k0, cnt, c);
      LNb nb[kBBatch];
      lgather<kBBatch>(a, rec, c, k0, cnt, pi, nb);
      bool any = false;
#pragma unroll
      for (int u = 0; u < kBBatch; u++) {
        if constexpr (MULTI) nb[u].in = nb[u].in && pm::eam_on(t, ltype[nb[u].c]);
        any |= nb[u].in;
      }
      if (!__any(any)) continue;
#pragma unroll
      for (int u = 0; u < kBBatch; u++) {
        const int tj = MULTI ? ltype[nb[u].c] : 0;
        const double* gj = gl + 3 * nb[u].c;
        double r, rinv;
        pm::dist(nb[u].d2, r, rinv);
        const double s = (nb[u].x * (gj[0] - g0) + nb[u].y * (gj[1] - g1) + nb[u].z * (gj[2] - g2)) * rinv;
        double p = fma(r, t.rdr_d, 1.0);
        const int m = max(0, min((int)p, t.nr - 1));
        p = fmin(p - (double)m, 1.0);
        const int plane = MULTI && max(ti, tj) < t.nel ? tj : 0;
        const pm::Q4<Real> row = pm::load4(pm::pair_row(t.slope, t, plane, m));
        const double dr = ((double)row.a * p + (double)row.b) * p + (double)row.c;
        drho += nb[u].in ? dr * s : 0.0;
      }
    }
    drho = ln.sum(drho);
    if (ln.writes()) {
      // F'' = d/drho of (c0 p + c1) p + c2, zero where p was clamped
      double p = g.rho[gi] * g.rdrho + 1.0;
      const int m = max(1, min((int)p, g.nrho - 1));
      p -= (double)m;
      const Real* row = static_cast<const Real*>(g.frho) + ((int64_t)t.t2frho[ti + 1] * (g.nrho + 1) + m) * 8;
      const double fpp = p > 1.0 ? 0.0 : (2.0 * (double)row[4] * p + (double)row[5]) * g.rdrho * g.conv;
      g.drho[gi] = drho;
      reinterpret_cast<double*>(g.gvec + gi)[3] = oni ? fpp * drho : 0.0;
    }
  }
}

// Gather ceiling of the mixed single-element EAM passes (a measurement, not an
// operator): the staging, list walk, LDS neighbour reads, FP64 displacement, cutoff
// test and table-row index of the density pass (knot rows, FORCE = false) or of the
// force pass (s-table rows, FORCE = true), with the same table gathers, but none of
// the spline or pair arithmetic: every gathered row is summed into a per-atom sink,
// so no load is dead, and the sink is the only output.  Its time against the pass's
// own is the fraction of the pass that its data movement accounts for.  LEVEL takes
// parts away to split that time: 0 everything above; 1 without the table-row
// gathers (the row index still computed and summed); 2 the list words only (no
// neighbour records, no displacement); 3 the staging only.
template <bool FORCE, int LEVEL>
__global__ void __launch_bounds__(kPassThreads, kPassWaves<false>) k_block_gather_ceiling(BlockArgs a,
                                                                                            EamTabDev<float> t,
                                                                                            const float* __restrict__ pair,
                                                                                            double* __restrict__ sink)
{
  const int64_t b = brick_of_block(a.nfull, a.nblocks);
  if (b >= a.nblocks) return;
  uint8_t* ltype;
  const LRec rec = pass_lds(a, false, FORCE, ltype);
  const BrickHead hd(a.head[b]);
  const PassLanes<false> ln(a);
  PassAtom<false> at;
  if (ln.slot < hd.central) at.index(a, hd, ln.slot);
  stage<FORCE>(a, hd, rec, ltype);
  if (ln.slot < hd.central) at.list(a, ln);
  __syncthreads();
  for (int q = ln.slot; q < hd.central; q += ln.atoms(), at.fetch(a, hd, q, ln)) {
    const int64_t gi = at.gi;
    const int slot = at.slot;
    const Pos4 pi = rec.get(slot);
    const int cnt = at.cnt;
    float acc = 0.0f;
    if constexpr (LEVEL == 3) {
      if (ln.writes()) sink[gi] = pi.x + cnt;
      continue;
    }
    LWords<false> lw(a, gi, ln);
    uint2 wnext = at.w;
    for (int k0 = ln.first(); k0 < cnt; k0 += ln.step()) {
      const uint2 w = wnext;
      if (k0 + ln.step() < cnt) wnext = lw.next();
      int c[kBBatch];
      lslots(w, a.cap, k0, cnt, c);
      if constexpr (LEVEL == 2) {
        acc += (float)((c[0] + c[1]) + (c[2] + c[3]));
        continue;
      }
      LNb nb[kBBatch];
      lgather<kBBatch>(a, rec, c, k0, cnt, pi, nb);
      bool any = false;
#pragma unroll
      for (int u = 0; u < kBBatch; u++) any |= nb[u].in;
      if (!__any(any)) continue;
#pragma unroll
      for (int u = 0; u < kBBatch; u++) {
        int m;
        float pp;
        if constexpr (FORCE) {
          bool out;
          pm::s_knot(t, nb[u].d2, m, pp, out);
          float v;
          if constexpr (LEVEL == 0) {
            const float* row = pm::at32(pair + t.s_force, (uint32_t)m * 8u);
            const pm::Q3 gr = pm::load3(row);
            const pm::Q3 gz = pm::load3(row + 4);
            v = ((gr.a + gr.b) + (gr.c + gz.a)) + ((gz.b + gz.c) + pp) + (float)nb[u].w;
          } else {
            v = (pp + (float)m) + (float)nb[u].w;
          }
          acc += nb[u].in ? v : 0.0f;
        } else {
          float rinv;
          pm::knot_dist(t, nb[u].d2, m, pp, rinv);
          float v;
          if constexpr (LEVEL == 0) {
            const pm::Q4<float> r = pm::load4(pm::pair_rho_row(pair, m));
            v = ((r.a + r.b) + (r.c + r.d)) + (pp + rinv);
          } else {
            v = (pp + rinv) + (float)m;
          }
          acc += nb[u].in ? v : 0.0f;
        }
      }
    }
    const double sum = ln.sum((double)acc);
    if (ln.writes()) sink[gi] = sum;
  }
}

// LJ forces (lj_compute_force, pair_potential_force_op_singlemat.h:45-218) on the
// block list: the staging, list walk and epilogues of k_block_eam_force with the
// pair math of the global-list kernel (pm::lj_pair).
// MULTI (lj_multi_force): types staged with the records; each pair takes the
// parameters and cutoff of its two species.
template <class Real, bool ENERGY, bool VIRIAL, bool FUSED, bool DRIFT, bool SPLIT, bool MULTI = false>
__global__ void __launch_bounds__(kPassThreads, kPassWaves<VIRIAL || SPLIT>) k_block_lj(BlockArgs a, pm::LJ<Real> lp,
                                                                           pm::Outputs o, pm::Drift dr,
                                                                           pm::LJMultiDev lm = {})
{
  static_assert(!DRIFT || (FUSED && !ENERGY && !VIRIAL), "the drift epilogue is the plain MD-loop step");
  const int64_t b = brick_of_block(a.nfull, a.nblocks);
  if (b >= a.nblocks || a.gate.closed()) return;
  uint8_t* ltype;
  const LRec rec = pass_lds(a, MULTI, false, ltype);
  const BrickHead hd(a.head[b]);
  // MULTI: the pairs' parameters and squared cutoffs (at most 28 pairs of 7 species), so
  // that a pair's lookup is an LDS read rather than two gathers through the texture path
  // (136 k atoms, FP64, energy and virial: 90 -> 66 us)
  __shared__ pm::LJ<Real> lrow[MULTI ? 28 : 1];
  __shared__ double lrc2[MULTI ? 28 : 1];
  if constexpr (MULTI) {
    if ((int)threadIdx.x < lm.npair) {
      lrow[threadIdx.x] = pm::lj_multi_row<Real>(lm, threadIdx.x);
      lrc2[threadIdx.x] = lm.rcut2[threadIdx.x];
    }
  }
  const PassLanes<SPLIT> ln(a);
  PassAtom<SPLIT> at;
  if (ln.slot < hd.central) at.index(a, hd, ln.slot);
  stage<false>(a, hd, rec, ltype);
  if (ln.slot < hd.central) at.list(a, ln);
  __syncthreads();
  for (int q = ln.slot; q < hd.central; q += ln.atoms(), at.fetch(a, hd, q, ln)) {
    const int64_t gi = at.gi;
    const int slot = at.slot;
    const Pos4 pi = rec.get(slot);
    const int ti = MULTI ? ltype[slot] : 0;
    const int cnt = at.cnt;
    double fx = 0.0, fy = 0.0, fz = 0.0, e = 0.0;
    double v[9] = {0, 0, 0, 0, 0, 0, 0, 0, 0};
    LWords<SPLIT> lw(a, gi, ln);
    uint2 wnext = at.w;
    for (int k0 = ln.first(); k0 < cnt; k0 += ln.step()) {
      const uint2 w = wnext;
      if (k0 + ln.step() < cnt) wnext = lw.next();
      int c[kBBatch];
      lslots(w, a.cap, k0, cnt, c);
      LNb nb[kBBatch];
      lgather<kBBatch>(a, rec, c, k0, cnt, pi, nb);
#pragma unroll
      for (int u = 0; u < kBBatch; u++) {
        double de_r, eh;
        if constexpr (MULTI) {
          const int pid = pm::type_pair(ti, ltype[nb[u].c]);
          pm::lj_pair(lrow[pid], nb[u].d2, nb[u].in && nb[u].d2 <= lrc2[pid], de_r, eh);
        } else {
          pm::lj_pair(lp, nb[u].d2, nb[u].in, de_r, eh);
        }
        fx = fma(nb[u].x, de_r, fx);
        fy = fma(nb[u].y, de_r, fy);
        fz = fma(nb[u].z, de_r, fz);
        if constexpr (ENERGY) e += eh;
        if constexpr (VIRIAL)
          pm::add_virial(v, nb[u].x * de_r, nb[u].y * de_r, nb[u].z * de_r, nb[u].x, nb[u].y, nb[u].z);
      }
    }
    fx = ln.sum(fx);
    fy = ln.sum(fy);
    fz = ln.sum(fz);
    if constexpr (ENERGY) e = ln.sum(e);
    if constexpr (VIRIAL) {
#pragma unroll
      for (int k = 0; k < 9; k++) v[k] = ln.sum(v[k]);
    }
    if (ln.writes()) {
      if constexpr (DRIFT) pm::write_outputs_drift(o, dr, gi, pi, fx, fy, fz);
      else pm::write_outputs<ENERGY, VIRIAL, FUSED>(o, gi, fx, fy, fz, e, v);
    }
  }
}

// Analytic Johnson EAM on the block list (FP64): pass 1 (EmbOp, eam_force_op_singlemat.h:39-171),
// rho_i, F'(rho_i) into the position record's w and F(rho_i) added to ep.
// Bound by the FP64 arithmetic of the pairs (one or two exponentials, divisions and a
// square root each).  128 k Ta atoms (83 entries, 53 in rc), both passes with energy and
// virial: 121 us, against 338 us, and 115 us to convert the list, on the global list with
// the general power function and every term evaluated for itself.
template <bool SPLIT>
__global__ void __launch_bounds__(kPassThreads, 4) k_block_johnson_rho(BlockArgs a, JohnsonParams jp,
                                                                       double* __restrict__ rho_out,
                                                                       double* __restrict__ pos_w,
                                                                       double* __restrict__ ep)
{
  const int64_t b = brick_of_block(a.nfull, a.nblocks);
  if (b >= a.nblocks) return;
  uint8_t* ltype;
  const LRec rec = pass_lds(a, false, false, ltype);
  const BrickHead hd(a.head[b]);
  const PassLanes<SPLIT> ln(a);
  PassAtom<SPLIT> at;
  if (ln.slot < hd.central) at.index(a, hd, ln.slot);
  stage<false>(a, hd, rec, ltype);
  if (ln.slot < hd.central) at.list(a, ln);
  __syncthreads();
  for (int q = ln.slot; q < hd.central; q += ln.atoms(), at.fetch(a, hd, q, ln)) {
    const int64_t gi = at.gi;
    const int slot = at.slot;
    const Pos4 pi = rec.get(slot);
    const int cnt = at.cnt;
    double rho = 0.0;
    LWords<SPLIT> lw(a, gi, ln);
    uint2 wnext = at.w;
    for (int k0 = ln.first(); k0 < cnt; k0 += ln.step()) {
      const uint2 w = wnext;
      if (k0 + ln.step() < cnt) wnext = lw.next();
      int c[kBBatch];
      lslots(w, a.cap, k0, cnt, c);
#pragma unroll
      for (int u = 0; u < kBBatch; u++) {
        LNb nb[1];
        lgather<1>(a, rec, c + u, k0 + 2 * u, cnt, pi, nb);
        if (!__any(nb[0].in)) continue;
        const double v = pm::johnson_rho(jp, nb[0].in ? nb[0].d2 : jp.re * jp.re);
        rho += nb[0].in ? v : 0.0;
      }
    }
    rho = ln.sum(rho);
    if (ln.writes()) {
      rho_out[gi] = rho;
      double F, Fp;
      pm::johnson_embed(jp, rho, F, Fp);
      pos_w[4 * gi + 3] = Fp;
      ep[gi] += F;
    }
  }
}

// Pass 2 (ForceOp): f_i += (rho'(r) (F'_i + F'_j) + phi'(r)) / r (r_j - r_i), ep += phi / 2,
// virial -1/2 f (x) dr.
template <bool VIRIAL, bool SPLIT>
__global__ void __launch_bounds__(kPassThreads, 4) k_block_johnson_force(BlockArgs a, JohnsonParams jp, pm::Outputs o)
{
  const int64_t b = brick_of_block(a.nfull, a.nblocks);
  if (b >= a.nblocks) return;
  uint8_t* ltype;
  const LRec rec = pass_lds(a, false, true, ltype);
  const BrickHead hd(a.head[b]);
  const PassLanes<SPLIT> ln(a);
  PassAtom<SPLIT> at;
  if (ln.slot < hd.central) at.index(a, hd, ln.slot);
  stage<true>(a, hd, rec, ltype);
  if (ln.slot < hd.central) at.list(a, ln);
  __syncthreads();
  for (int q = ln.slot; q < hd.central; q += ln.atoms(), at.fetch(a, hd, q, ln)) {
    const int64_t gi = at.gi;
    const int slot = at.slot;
    const Pos4 pi = rec.get(slot);
    const int cnt = at.cnt;
    double fx = 0.0, fy = 0.0, fz = 0.0, e = 0.0;
    double v[9] = {0, 0, 0, 0, 0, 0, 0, 0, 0};
    LWords<SPLIT> lw(a, gi, ln);
    uint2 wnext = at.w;
    for (int k0 = ln.first(); k0 < cnt; k0 += ln.step()) {
      const uint2 w = wnext;
      if (k0 + ln.step() < cnt) wnext = lw.next();
      int c[kBBatch];
      lslots(w, a.cap, k0, cnt, c);
#pragma unroll
      for (int u = 0; u < kBBatch; u++) {
        LNb nb[1];
        lgather<1>(a, rec, c + u, k0 + 2 * u, cnt, pi, nb);
        if (!__any(nb[0].in)) continue;
        double de, phi;
        pm::johnson_pair(jp, nb[0].in ? nb[0].d2 : jp.re * jp.re, pi.w + nb[0].w, de, phi);
        de = nb[0].in ? de : 0.0;
        const double fe0 = de * nb[0].x, fe1 = de * nb[0].y, fe2 = de * nb[0].z;
        fx += fe0;
        fy += fe1;
        fz += fe2;
        e += nb[0].in ? 0.5 * phi : 0.0;
        if constexpr (VIRIAL) pm::add_virial(v, fe0, fe1, fe2, nb[0].x, nb[0].y, nb[0].z);
      }
    }
    fx = ln.sum(fx);
    fy = ln.sum(fy);
    fz = ln.sum(fz);
    e = ln.sum(e);
    if constexpr (VIRIAL) {
#pragma unroll
      for (int k = 0; k < 9; k++) v[k] = ln.sum(v[k]);
    }
    if (ln.writes()) pm::write_outputs<true, VIRIAL, false>(o, gi, fx, fy, fz, e, v);
  }
}

BlockArgs block_args(const Ctx& c, double rcut, const StepGate& gate = {})
{
  BlockArgs a;
  a.gate = gate;
  a.head = c.brick_head.p;
  a.stage = c.brick_stage.p;
  a.cen = c.brick_cen.p;
  a.cen_slot = c.brick_cen_slot.p;
  a.pos = c.pos.p;
  a.type = c.type.p;
  a.box = c.box_d.p;
  a.nbr16 = c.nbr16.p;
  a.nnb = c.nnb.p;
  a.npad = c.npad;
  a.nblocks = c.bgeom.nblocks;
  a.nfull = c.bgeom.nfull;
  a.cap = c.bcap;
  a.rc2 = rcut * rcut;
  a.xf = c.xf_dev();
  a.nmax = c.nmax;
  a.split = 0;
  while (a.split < 3 && (c.bcentral << (a.split + 1)) <= kPassAtoms) a.split++;
  return a;
}

// Fused next-step drift of the MD loop (ForceEpilogue::drift) for a force launch
// with the plain MD-loop epilogue; false when it does not apply.
bool drift_setup(Ctx& c, const ForceEpilogue& epi, unsigned flags, pm::Drift& dr)
{
  // under a non-identity xform the loop's own drift kernel (which maps the step by the
  // inverse xform) runs instead: the epilogue drifts from the staged record, which is
  // then a physical position, and it keeps the identity form's code
  if (!(epi.fused && epi.drift) || (flags & (XS_ENERGY | XS_VIRIAL)) || c.xf_dev()) return false;
  c.pos2.reserve(c.npad);
  dr.pos_out = c.pos2.p;
  dr.rrx = c.rrx.p;
  dr.rry = c.rry.p;
  dr.rrz = c.rrz.p;
  dr.dt = epi.drift_dt;
  dr.dt2 = epi.drift_dt * epi.drift_dt * 0.5;
  dr.hdt = epi.drift_dt * 0.5;
  dr.thr2 = epi.drift_thr2;
  dr.over = StepFlag{c.dscalar.p + 6, c.hflag, epi.step + 1};
  return true;
}

// after the launch: the next step's positions (pos2) become current
void drift_commit(Ctx& c)
{
  c.pos.swap(c.pos2);
  c.rho_ckpt = false;
  c.drift_done = true;
}

template <class Real, bool MULTI>
void block_eam_dispatch(Ctx& c, double rcut, bool do_rho, bool do_emb, bool do_force, unsigned flags,
                        const ForceEpilogue& epi)
{
  const EamTabDev<Real> t = make_eam_tab<Real>(c);
  const Real* pair = eam_pair_table<Real>(c);
  const BlockArgs a = block_args(c, rcut, step_gate(c, epi));
  const size_t lds_rho = block_lds_bytes(c, MULTI, false);
  const size_t lds = block_lds_bytes(c, MULTI, true);
  const unsigned g = block_grid(c);
  const bool energy = flags & XS_ENERGY;
  double* pos_w = reinterpret_cast<double*>(c.pos.p);
  if (do_rho) {
    ProfScope prof(c.prof, c.stream, XS_PROF_EAM_RHO);
#define XS_BRHO(EMB, EN, SET) \
  (a.split ? k_block_eam_rho<Real, MULTI, EMB, EN, SET, true> : k_block_eam_rho<Real, MULTI, EMB, EN, SET, false>) \
      <<<g, kPassThreads, lds_rho, c.stream>>>(a, t, pair, c.rho.p, pos_w, c.ep.p)
    if (!do_emb) XS_BRHO(false, false, false);
    else if (energy && epi.fused) XS_BRHO(true, true, true);
    else if (energy) XS_BRHO(true, true, false);
    else XS_BRHO(true, false, false);
#undef XS_BRHO
    XS_HIP(hipGetLastError());
  }
  if (do_force) {
    const pm::Outputs o = make_outputs(c, epi);
    const bool vir = flags & XS_VIRIAL;
    pm::Drift dr{};
    const bool drift = drift_setup(c, epi, flags, dr);
    ProfScope prof(c.prof, c.stream, XS_PROF_EAM_FORCE);
#define XS_BF(EN, VI, FU, DR) \
  (a.split ? k_block_eam_force<Real, MULTI, EN, VI, FU, DR, true>                                       \
           : k_block_eam_force<Real, MULTI, EN, VI, FU, DR, false>)<<<g, kPassThreads, lds, c.stream>>>(a, t, pair, o, dr)
    if (drift) {
      XS_BF(false, false, true, true);
    } else if (epi.fused) {
      if (energy && vir) XS_BF(true, true, true, false);
      else if (energy) XS_BF(true, false, true, false);
      else if (vir) XS_BF(false, true, true, false);
      else XS_BF(false, false, true, false);
    } else {
      if (energy && vir) XS_BF(true, true, false, false);
      else if (energy) XS_BF(true, false, false, false);
      else if (vir) XS_BF(false, true, false, false);
      else XS_BF(false, false, false, false);
    }
#undef XS_BF
    XS_HIP(hipGetLastError());
    if (drift) drift_commit(c);
  }
}

}  // namespace

// Average time (ms) of `reps` launches of the gather-ceiling kernel of one pass at
// one level (see k_block_gather_ceiling) on the current block list and FP32
// single-element tables.
double gather_ceiling(Ctx& c, double rcut, bool force, int level, int reps)
{
  if (level < 0 || level > 3) throw Error(XS_E_ARG, "gather ceiling level must be 0..3");
  if (c.list_kind != ListKind::Block) throw Error(XS_E_STATE, "gather ceiling needs the cell-block list");
  if (!c.has_eam || eam_multi(c)) throw Error(XS_E_STATE, "gather ceiling needs single-element EAM tables");
  if (reps < 1) throw Error(XS_E_ARG, "reps must be >= 1");
  const EamTabDev<float> t = make_eam_tab<float>(c);
  if (force && c.eam.s_pieces == 0) throw Error(XS_E_STATE, "gather ceiling of the force pass needs the s-table");
  const BlockArgs a = block_args(c, rcut);
  DBuf<double> sink;
  sink.reserve(c.npad);
  const unsigned g = block_grid(c);
  const size_t lds = block_lds_bytes(c, false, force);
  hipEvent_t e0, e1;
  XS_HIP(hipEventCreate(&e0));
  XS_HIP(hipEventCreate(&e1));
  XS_HIP(hipEventRecord(e0, c.stream));
  using K = void (*)(BlockArgs, EamTabDev<float>, const float*, double*);
  const K ks[2][4] = {{k_block_gather_ceiling<false, 0>, k_block_gather_ceiling<false, 1>,
                       k_block_gather_ceiling<false, 2>, k_block_gather_ceiling<false, 3>},
                      {k_block_gather_ceiling<true, 0>, k_block_gather_ceiling<true, 1>,
                       k_block_gather_ceiling<true, 2>, k_block_gather_ceiling<true, 3>}};
  const K k = ks[force ? 1 : 0][level];
  for (int r = 0; r < reps; r++) k<<<g, kPassThreads, lds, c.stream>>>(a, t, c.eam.pair_f.p, sink.p);
  XS_HIP(hipGetLastError());
  XS_HIP(hipEventRecord(e1, c.stream));
  XS_HIP(hipEventSynchronize(e1));
  float ms = 0.f;
  XS_HIP(hipEventElapsedTime(&ms, e0, e1));
  (void)hipEventDestroy(e0);
  (void)hipEventDestroy(e1);
  return ms / reps;
}

// ---------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------
// Brick shape: the one that stages the fewest halo cells per grid cell (partial
// bricks at the grid edge count as whole ones) among the shapes whose expected
// central atoms stay within `bound` (one round of the 256 atom slots of a pass
// workgroup, with headroom for density fluctuations) and, unless XSMD_BLOCK_ATOMS
// set the bound, whose expected halo leaves LDS for three pass workgroups per CU
// (32-byte records, 15 % headroom).
void block_shape_choose(const Ctx& c, BlockGeom& g, double bound, double per_cell)
{
  const double lds_halo_cells = (double)(kLdsPerCu / 3 - 2048) / (32.0 * 1.15 * per_cell);
  int bx = 1, by = 1, bz = 1;
  double best = 1e300;
  for (int z = 1; z <= std::min(g.nz, 8); z++)
    for (int y = 1; y <= std::min(g.ny, 8); y++)
      for (int x = 1; x <= std::min(g.nx, 8); x++) {
        const int halo = (x + 2) * (y + 2) * (z + 2);
        if (x * y * z > 1 && (x * y * z * per_cell > bound || halo > kMaxHaloCells ||
                              (!c.block_atoms_set && halo > lds_halo_cells)))
          continue;
        const double nb = (double)((g.nx + x - 1) / x) * ((g.ny + y - 1) / y) * ((g.nz + z - 1) / z);
        const double cost = nb * halo / ((double)g.nx * g.ny * g.nz);
        if (cost < best * (1.0 - 1e-9)) {
          best = cost;
          bx = x;
          by = y;
          bz = z;
        }
      }
  g.bx = bx;
  g.by = by;
  g.bz = bz;
  g.nbx = (g.nx + bx - 1) / bx;
  g.nby = (g.ny + by - 1) / by;
  g.nbz = (g.nz + bz - 1) / bz;
  g.nblocks = (int64_t)g.nbx * g.nby * g.nbz * c.nrep;
  g.fx = g.nx / bx;
  g.fy = g.ny / by;
  g.fz = g.nz / bz;
  g.nfull = (int64_t)g.fx * g.fy * g.fz * c.nrep;
  g.nh_max = (bx + 2) * (by + 2) * (bz + 2);
}

void block_setup(Ctx& c)
{
  BlockGeom& g = c.bgeom;
  g.nx = c.nc[0];
  g.ny = c.nc[1];
  g.nz = c.nc[2];
  g.px = c.periodic[0];
  g.py = c.periodic[1];
  g.pz = c.periodic[2];
  g.ncell_rep = c.ncell_rep;
  // The shape is chosen from the mean atoms per cell; where atoms crowd into part
  // of the grid (slabs, clusters) the measured halo can exceed the LDS budget, and
  // the bound shrinks until it fits (or the bricks are single cells).
  double per_cell = std::max((double)c.n / (double)c.ncell_tot, 1e-3);
  // Systems that 230-atom bricks would not spread over the CUs are cut into smaller ones,
  // whose passes walk each list with more lanes (PassLanes).  One and a half workgroups
  // per CU measured best at 50 k EAM atoms (density and force pass, mixed: bricks of at
  // most 60 atoms 11.4 + 15.8 us, 85: 10.6 + 16.0, 128: 11.0 + 12.8, 170: 12.3 + 14.6,
  // 230: 12.9 + 18.2); 4000 argon atoms end at one cell per brick either way.
  double bound = c.block_atoms;
  if (!c.block_atoms_set) bound = std::min(bound, std::max(8.0, (double)c.n / (1.5 * std::max(c.num_cu, 1))));
  for (int attempt = 0;; attempt++) {
    block_shape_choose(c, g, bound, per_cell);
    const unsigned groups = (unsigned)std::min<int64_t>(kHaloGroups, (g.nblocks + kHaloMaxWaves - 1) / kHaloMaxWaves);
    k_block_halo_max<<<groups, 64 * kHaloMaxWaves, 0, c.stream>>>(g, c.cell_off.p, c.hhalo, c.dscalar.p);
    XS_HIP(hipGetLastError());
    XS_HIP(hipStreamSynchronize(c.stream));
    uint32_t halo = 0, central = 0, cand = 0;
    size_t entries = 0;
    for (unsigned k = 0; k < groups; k++) {
      const uint32_t* h = c.hhalo + 4 * k;
      halo = std::max(halo, h[0]);
      central = std::max(central, h[1]);
      cand = std::max(cand, h[2]);
      entries += h[3];
    }
    c.bcap = (int)((halo + 63) / 64 * 64);
    c.bcentral = (int)central;
    c.bcand = (int)cand;
    c.bstage = entries * kStageAlign;
    const size_t budget = c.block_atoms_set ? kBlockLdsLimit : std::min(kBlockLdsLimit, kLdsPerCu / 3);
    if (block_lds_bytes(c, true, true) <= budget || g.nh_max == 27 || attempt == 6) break;
    // the densest halo set the capacity: size the next shape for that density
    per_cell = std::max(per_cell, (double)halo / g.nh_max);
    bound *= 0.75;
  }
}

size_t block_lds_bytes(const Ctx& c, bool with_type, bool with_w)
{
  // bcap records and the far record, and their types (pass_lds)
  return ((size_t)c.bcap + 1) * (sizeof(double) * (with_w ? 4 : 3) + (with_type ? 1 : 0));
}

bool block_feasible(const Ctx& c)
{
  return c.bcap > 0 && c.bcap < 65536 && c.bstage < (size_t)1 << 32 && block_lds_bytes(c, true, true) <= kBlockLdsLimit;
}

unsigned block_grid(const Ctx& c)
{
  // every XCD's share of the full and of the cut bricks (brick_of_block)
  return (unsigned)(8 * ((c.bgeom.nfull + 7) / 8 + (c.bgeom.nblocks - c.bgeom.nfull + 7) / 8));
}

// LDS of a build launch that collects `atoms` lists per wave
static size_t build_lds_bytes(const Ctx& c, int atoms)
{
  return build_rec_bytes(c.bcap) + (size_t)c.bgeom.nh_max * sizeof(HaloCell) +
         (4 + (size_t)c.bgeom.bx * c.bgeom.by * c.bgeom.bz) * sizeof(int) + build_cand_bytes(c.bcap, c.bcand) +
         (size_t)kBuildWaves * atoms * (c.nmax + 1) * sizeof(uint32_t);
}

// Block list build; false when its LDS does not fit a workgroup (then nothing was
// built).  The lists of fewer atoms are collected at once where long lists need it.
bool block_build(Ctx& c, double rl2)
{
  BuildArgs a;
  a.g = c.bgeom;
  a.cell_off = c.cell_off.p;
  a.pos = c.pos.p;
  a.box = c.box_d.p;
  a.xf = c.xf_dev();
  a.rl2 = rl2;
  a.npad = c.npad;
  a.cap = c.bcap;
  a.cand_cap = c.bcand;
  a.sort = !c.list_sort_disabled;
  a.flags = c.dscalar.p;
  a.over = c.hhalo + 4 * kHaloGroups;
  c.brick_head.reserve(c.bgeom.nblocks);
  // bcap is a multiple of kStageAlign
  const size_t step_total = (size_t)c.bgeom.nblocks * c.bcap;
  const bool step = step_total <= 2 * c.bstage && step_total < (size_t)1 << 32;
  a.stage_step = step ? c.bcap : 0;
  a.cen_step = step ? c.bcentral : 0;
  c.brick_stage.reserve(step ? step_total : c.bstage);
  const size_t cen = step ? (size_t)c.bgeom.nblocks * c.bcentral : (size_t)c.n;
  c.brick_cen.reserve(cen);
  c.brick_cen_slot.reserve(cen);
  c.atom_stage.reserve(c.n);
  a.head = c.brick_head.p;
  a.stage = c.brick_stage.p;
  a.cen = c.brick_cen.p;
  a.cen_slot = c.brick_cen_slot.p;
  a.base = c.atom_stage.p;
  for (int attempt = 0; attempt < 2; attempt++) {
    a.atoms = kBuildAtoms;
    while (a.atoms > 1 && build_lds_bytes(c, a.atoms) > kBlockLdsLimit) a.atoms /= 2;
    const size_t lds = build_lds_bytes(c, a.atoms);
    if (lds > c.lds_max) return false;
    c.nbr16.reserve((size_t)c.nmax * c.npad);
    c.nnb.reserve(c.npad);
    a.nbr16 = c.nbr16.p;
    a.nnb = c.nnb.p;
    a.nmax = c.nmax;
    const auto k = a.xf ? k_block_build<true> : k_block_build<false>;
    if (lds > kBlockLdsLimit)
      XS_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(k), hipFuncAttributeMaxDynamicSharedMemorySize,
                                 (int)lds));
    // block_setup's kernel cleared the flags
    if (attempt > 0) XS_HIP(hipMemsetAsync(c.dscalar.p, 0, 3 * sizeof(unsigned long long), c.stream));
    *a.over = 0;
    k<<<block_grid(c), kBuildThreads, lds, c.stream>>>(a);
    XS_HIP(hipGetLastError());
    XS_HIP(hipStreamSynchronize(c.stream));
    if (*a.over == 0) return true;
    XS_HIP(hipMemcpyAsync(c.hscalar, c.dscalar.p, 2 * sizeof(unsigned long long), hipMemcpyDeviceToHost,
                          c.stream));
    XS_HIP(hipStreamSynchronize(c.stream));
    if (c.hscalar[1] != 0) throw Error(XS_E_STATE, "block halo exceeds its measured capacity");
    const unsigned long long need = c.hscalar[0];
    if (attempt == 1) throw Error(XS_E_STATE, "neighbour list overflow after resize");
    c.nmax = (int)((need + 7) / 8 * 8 + 8);
  }
  return false;
}

void block_to_global(Ctx& c)
{
  c.nbr.reserve((size_t)c.nmax * c.npad);
  k_block_to_global<<<block_grid(c), kBlock, 0, c.stream>>>(block_args(c, 0.0), c.nbr.p);
  XS_HIP(hipGetLastError());
}

}  // namespace xsmd

namespace xsmd {

// EAM on the block list.  The embedding step alone (eam_rho2emb after a separate
// eam_rho, as in the split-pass deck) reads no list and runs the per-atom kernel of
// the global path; its arithmetic is the same as the fused block pass.
void launch_eam_block(Ctx& c, double rcut, bool do_rho, bool do_emb, bool do_force, unsigned flags,
                      const ForceEpilogue& epi)
{
  const bool mixed = (flags & XS_MIXED) != 0;
  const bool multi = eam_multi(c);
  if (do_emb && !do_rho) {
    const ListKind keep = c.list_kind;
    c.list_kind = ListKind::Global;
    try {
      launch_eam(c, rcut, false, true, false, flags, epi);
    } catch (...) {
      c.list_kind = keep;
      throw;
    }
    c.list_kind = keep;
    if (!do_force) return;
    do_emb = false;
  }
  if (mixed) {
    if (multi) block_eam_dispatch<float, true>(c, rcut, do_rho, do_emb, do_force, flags, epi);
    else block_eam_dispatch<float, false>(c, rcut, do_rho, do_emb, do_force, flags, epi);
  } else {
    if (multi) block_eam_dispatch<double, true>(c, rcut, do_rho, do_emb, do_force, flags, epi);
    else block_eam_dispatch<double, false>(c, rcut, do_rho, do_emb, do_force, flags, epi);
  }
}

void launch_lj_block(Ctx& c, double eps, double sigma, double rcut, unsigned flags, const ForceEpilogue& epi)
{
  const double ecut = lj_energy_cutoff(eps, sigma, rcut);
  const BlockArgs a = block_args(c, rcut, step_gate(c, epi));
  const size_t lds = block_lds_bytes(c, false, false);
  const unsigned g = block_grid(c);
  pm::Outputs o = make_outputs(c, epi);
  o.set_ep = epi.fused;
  const bool energy = flags & XS_ENERGY, vir = flags & XS_VIRIAL;
  pm::Drift dr{};
  const bool drift = drift_setup(c, epi, flags, dr);
  ProfScope prof(c.prof, c.stream, XS_PROF_LJ);
  auto run = [&](auto zero) {
    using Real = decltype(zero);
    const pm::LJ<Real> lp{(Real)(sigma * sigma), (Real)(4.0 * eps), (Real)(24.0 * eps), (Real)ecut};
#define XS_BL(EN, VI, FU, DR)                                                                                \
  (a.split ? k_block_lj<Real, EN, VI, FU, DR, true> : k_block_lj<Real, EN, VI, FU, DR, false>)               \
      <<<g, kPassThreads, lds, c.stream>>>(a, lp, o, dr, pm::LJMultiDev{})
    if (drift) {
      XS_BL(false, false, true, true);
    } else if (epi.fused) {
      if (energy && vir) XS_BL(true, true, true, false);
      else if (energy) XS_BL(true, false, true, false);
      else if (vir) XS_BL(false, true, true, false);
      else XS_BL(false, false, true, false);
    } else {
      if (energy && vir) XS_BL(true, true, false, false);
      else if (energy) XS_BL(true, false, false, false);
      else if (vir) XS_BL(false, true, false, false);
      else XS_BL(false, false, false, false);
    }
#undef XS_BL
  };
  if (flags & XS_MIXED) run(0.0f);
  else run(0.0);
  XS_HIP(hipGetLastError());
  if (drift) drift_commit(c);
}

void launch_lj_multi_block(Ctx& c, unsigned flags)
{
  BlockArgs a = block_args(c, 0.0);
  a.rc2 = c.ljm_rc2;
  const size_t lds = block_lds_bytes(c, true, false);
  const unsigned g = block_grid(c);
  const pm::Outputs o = make_outputs(c, ForceEpilogue{});
  const bool energy = flags & XS_ENERGY, vir = flags & XS_VIRIAL;
  const pm::Drift dr{};
  ProfScope prof(c.prof, c.stream, XS_PROF_LJ);
  auto run = [&](auto zero) {
    using Real = decltype(zero);
    const pm::LJ<Real> none{};
    const pm::LJMultiDev lm = ljm_dev<Real>(c);
#define XS_BLM(EN, VI) \
  (a.split ? k_block_lj<Real, EN, VI, false, false, true, true>                                              \
           : k_block_lj<Real, EN, VI, false, false, false, true>)<<<g, kPassThreads, lds, c.stream>>>(a, none, o, dr, lm)
    if (energy && vir) XS_BLM(true, true);
    else if (energy) XS_BLM(true, false);
    else if (vir) XS_BLM(false, true);
    else XS_BLM(false, false);
#undef XS_BLM
  };
  if (flags & XS_MIXED) run(0.0f);
  else run(0.0);
  XS_HIP(hipGetLastError());
}

void launch_johnson_block(Ctx& c, const JohnsonParams& p, double rcut, bool do_emb, bool do_force, unsigned flags)
{
  const BlockArgs a = block_args(c, rcut);
  const unsigned g = block_grid(c);
  if (do_emb) {
    ProfScope prof(c.prof, c.stream, XS_PROF_EAM_RHO);
    (a.split ? k_block_johnson_rho<true> : k_block_johnson_rho<false>)
        <<<g, kPassThreads, block_lds_bytes(c, false, false), c.stream>>>(a, p, c.rho.p, reinterpret_cast<double*>(c.pos.p), c.ep.p);
    XS_HIP(hipGetLastError());
  }
  if (!do_force) return;
  const pm::Outputs o = make_outputs(c, ForceEpilogue{});
  ProfScope prof(c.prof, c.stream, XS_PROF_EAM_FORCE);
  const size_t lds = block_lds_bytes(c, false, true);
  const bool vir = flags & XS_VIRIAL;
  const auto k = a.split ? (vir ? k_block_johnson_force<true, true> : k_block_johnson_force<false, true>)
                         : (vir ? k_block_johnson_force<true, false> : k_block_johnson_force<false, false>);
  k<<<g, kPassThreads, lds, c.stream>>>(a, p, o);
  XS_HIP(hipGetLastError());
}

void launch_adj_b1_block(Ctx& c, double rcut, bool mixed)
{
  const BlockArgs a = block_args(c, rcut);
  const bool multi = eam_multi(c);
  // at most 97 KB for the largest halo the brick list allows (kBlockLdsLimit)
  const size_t lds = ((size_t)c.bcap + 1) * (6 * sizeof(double) + (multi ? 1 : 0));
  AdjB1Args g;
  g.gvec = c.adj_gvec.p;
  g.drho = c.adj_drho.p;
  g.rho = c.rho.p;
  g.nrho = c.eam.nrho;
  g.rdrho = c.eam.rdrho;
  g.conv = kEV;
  const auto run = [&](auto zero, auto k) {
    using Real = decltype(zero);
    if constexpr (sizeof(Real) == 4) g.frho = c.eam.frho_f.p;
    else g.frho = c.eam.frho_d.p;
    if (lds > kBlockLdsLimit)
      XS_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(k), hipFuncAttributeMaxDynamicSharedMemorySize,
                                 (int)lds));
    k<<<block_grid(c), kPassThreads, lds, c.stream>>>(a, make_eam_tab<Real>(c), g);
    XS_HIP(hipGetLastError());
  };
  const auto pick = [&](auto zero) {
    using Real = decltype(zero);
    if (multi) run(zero, a.split ? k_block_adj_b1<Real, true, true> : k_block_adj_b1<Real, true, false>);
    else run(zero, a.split ? k_block_adj_b1<Real, false, true> : k_block_adj_b1<Real, false, false>);
  };
  if (mixed) pick(0.0f);
  else pick(0.0);
}

void ensure_global_list(Ctx& c)
{
  if (c.list_kind == ListKind::Global || c.global_from_block) return;
  block_to_global(c);
  c.global_from_block = true;
}

}  // namespace xsmd
