// k_neighbors.hip -- cell binning, atom re-sort and full neighbour-list build.
//
// A rebuild is: wrap atoms into their periodic box, compute each atom's cell,
// stable counting sort by cell (so the in-cell order is deterministic and equal to
// a stable CPU sort), gather every per-atom array into the new order, find the
// cell ranges, then one thread per atom scans the 27 surrounding cells and
// writes the (atom, image) entries within rcut+skin into an ELL list stored
// column-major (entry k of atom i at nbr[k*npad + i]) so the force kernels read
// it with coalesced loads.
#include "xsmd_internal.hpp"

#include <algorithm>
#include <cmath>

namespace xsmd {
namespace {

// Re-sort by cell.  A counting sort: the atoms of each cell are counted and numbered in
// the order the counting happened to take them (k_cell_count), an exclusive sum over the
// cells gives each cell its range (k_cell_sums, k_cell_offsets), k_cell_place writes the
// atom indices into the ranges, and k_cell_order puts each at the number of smaller
// indices in its cell, so the result is the stable sort by cell whatever order the
// counts were taken in.  That last step reads a cell's members once per atom, which is a
// small part of the list build's own work per cell.  Four or five launches; a library
// radix sort of (cell, index) pairs took 8 launches at 4 k atoms and 20 at 1 M
// (about 150 us there against 57, and 90 against 17 at 4 k).  Up to kFusedOrder atoms
// k_order_permute also moves each atom to its place, which saves a launch; above, its
// writes lose more by their scatter (340 us against 237 + 75 at 8.39 M atoms, 48 against
// 34 + 16 at 1.05 M).

// Wraps atom i into its box, finds its cell, counts it there: num[i] = its number among
// the atoms of the cell so far.  Consecutive atoms mostly share a cell (they were sorted
// at the last build), so a run of equal cells in a wave takes one atomic.
__global__ void __launch_bounds__(256) k_cell_count(int64_t n, Pos4* __restrict__ pos, const uint16_t* __restrict__ rep,
                                                    const BoxDev* __restrict__ box, int px, int py, int pz, int nx,
                                                    int ny, int nz, int64_t ncell_rep, uint32_t* __restrict__ keys,
                                                    uint32_t* __restrict__ num, uint32_t* __restrict__ count)
{
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const bool live = i < n;
  uint32_t key = 0xffffffffu;  // no cell has it (fewer than 2^32 cells)
  if (live) {
    const int r = rep ? rep[i] : 0;
    const BoxDev& b = box[r];
    Pos4 p = load_pos(pos, i);
    if (px || py || pz) {
      if (px) p.x = xsmd_wrap(p.x, b.lo[0], b.L[0]);
      if (py) p.y = xsmd_wrap(p.y, b.lo[1], b.L[1]);
      if (pz) p.z = xsmd_wrap(p.z, b.lo[2], b.L[2]);
      store_pos(pos, i, p);
    }
    const int cx = xsmd_cell_coord(p.x, b.lo[0], b.inv_cs[0], nx);
    const int cy = xsmd_cell_coord(p.y, b.lo[1], b.inv_cs[1], ny);
    const int cz = xsmd_cell_coord(p.z, b.lo[2], b.inv_cs[2], nz);
    key = (uint32_t)((int64_t)r * ncell_rep + ((int64_t)cz * ny + cy) * nx + cx);
    keys[i] = key;
  }
  const int lane = threadIdx.x & 63;
  const uint32_t before = __shfl_up(key, 1);
  const unsigned long long heads = __ballot(lane == 0 || key != before);
  const unsigned long long upto = heads & (~0ull >> (63 - lane));
  const int head = 63 - __clzll((long long)upto);
  const unsigned long long after = lane == 63 ? 0ull : heads >> (lane + 1) << (lane + 1);
  uint32_t base = 0;
  if (live && lane == head) {
    const int end = after ? __ffsll((unsigned long long)after) - 1 : 64;
    base = atomicAdd(count + key, (uint32_t)(end - lane));
  }
  base = __shfl(base, head);
  if (live) num[i] = base + (uint32_t)(lane - head);
}

constexpr int kScanThreads = 256;

// sum of v over the threads below this one (and the workgroup's total)
__device__ __forceinline__ uint32_t block_exclusive(uint32_t v, uint32_t& total)
{
  __shared__ uint32_t wsum[kScanThreads / 64];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  uint32_t s = v;
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const uint32_t t = __shfl_up(s, off);
    if (lane >= off) s += t;
  }
  __syncthreads();  // the sums of an earlier call are read
  if (lane == 63) wsum[w] = s;
  __syncthreads();
  uint32_t before = 0;
  total = 0;
#pragma unroll
  for (int k = 0; k < kScanThreads / 64; k++) {
    if (k < w) before += wsum[k];
    total += wsum[k];
  }
  return before + s - v;
}

// atoms in each run of `items` cells
__global__ void __launch_bounds__(kScanThreads) k_cell_sums(int64_t ncell, int64_t items,
                                                            const uint32_t* __restrict__ count,
                                                            uint32_t* __restrict__ sums)
{
  const int64_t c0 = (int64_t)blockIdx.x * items, c1 = min(c0 + items, ncell);
  uint32_t v = 0, total;
  for (int64_t c = c0 + threadIdx.x; c < c1; c += kScanThreads) v += count[c];
  block_exclusive(v, total);
  if (threadIdx.x == 0) sums[blockIdx.x] = total;
}

// first atom of each cell, off[ncell] = n; clears the counts for the next sort
__global__ void __launch_bounds__(kScanThreads) k_cell_offsets(int64_t ncell, int64_t items,
                                                               uint32_t* __restrict__ count,
                                                               const uint32_t* __restrict__ sums,
                                                               int* __restrict__ off)
{
  const int64_t c0 = (int64_t)blockIdx.x * items, c1 = min(c0 + items, ncell);
  uint32_t v = 0, base, total;
  for (int b = threadIdx.x; b < (int)blockIdx.x; b += kScanThreads) v += sums[b];
  block_exclusive(v, base);
  for (int64_t c = c0; c < c1; c += kScanThreads) {
    const int64_t k = c + threadIdx.x;
    v = 0;
    if (k < c1) {
      v = count[k];
      count[k] = 0;
    }
    const uint32_t ex = block_exclusive(v, total);
    if (k < c1) off[k] = (int)(base + ex);
    base += total;
  }
  if (c1 == ncell && threadIdx.x == 0) off[ncell] = (int)base;
}

__global__ void k_cell_place(int64_t n, const uint32_t* __restrict__ keys, const uint32_t* __restrict__ num,
                             const int* __restrict__ off, uint32_t* __restrict__ members)
{
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) members[off[keys[i]] + num[i]] = (uint32_t)i;
}

// the atom p at place k of `members`, and its place in the stable order; its cell to keys_out
__device__ __forceinline__ int64_t stable_place(int64_t k, const uint32_t* __restrict__ members,
                                                const uint32_t* __restrict__ keys, const int* __restrict__ off,
                                                uint32_t* __restrict__ keys_out, uint32_t& p)
{
  p = members[k];
  const uint32_t key = keys[p];
  const int o0 = off[key], o1 = off[key + 1];
  int64_t i = o0;
  for (int o = o0; o < o1; o++) i += members[o] < p;
  keys_out[k] = key;  // places k and i are in the same cell
  return i;
}

// perm[i] = atom at place i of the stable order
__global__ void k_cell_order(int64_t n, const uint32_t* __restrict__ members, const uint32_t* __restrict__ keys,
                             const int* __restrict__ off, uint32_t* __restrict__ perm,
                             uint32_t* __restrict__ keys_out)
{
  const int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= n) return;
  uint32_t p;
  const int64_t i = stable_place(k, members, keys, off, keys_out, p);
  perm[i] = p;
}

struct PermuteArgs {
  const Pos4* pos_src;
  Pos4* pos_dst;
  double* rrx;
  double* rry;
  double* rrz;
  const double* src[6];
  double* dst[6];
  const uint8_t* type_src;
  uint8_t* type_dst;
  const int64_t* id_src;
  int64_t* id_dst;
  const uint16_t* rep_src;
  uint16_t* rep_dst;
};

// Gather every per-atom array into the new order (ND of the six velocity and
// acceleration components; a caller about to overwrite the accelerations leaves them
// out); the new positions also become the reference positions of the displacement check.
template <int ND>
__device__ __forceinline__ void move_atom(const PermuteArgs& a, uint32_t p, int64_t i)
{
  const Pos4 q = load_pos(a.pos_src, p);
  store_pos(a.pos_dst, i, q);
  a.rrx[i] = q.x;
  a.rry[i] = q.y;
  a.rrz[i] = q.z;
#pragma unroll
  for (int d = 0; d < ND; d++) a.dst[d][i] = a.src[d][p];
  a.type_dst[i] = a.type_src[p];
  a.id_dst[i] = a.id_src[p];
  if (a.rep_src) a.rep_dst[i] = a.rep_src[p];
}
template <int ND>
__global__ void __launch_bounds__(256) k_permute(int64_t n, const uint32_t* __restrict__ perm, PermuteArgs a)
{
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) move_atom<ND>(a, perm[i], i);
}

// k_cell_order and k_permute in one
constexpr int64_t kFusedOrder = 1 << 19;
template <int ND>
__global__ void __launch_bounds__(256) k_order_permute(int64_t n, const uint32_t* __restrict__ members,
                                                       const uint32_t* __restrict__ keys, const int* __restrict__ off,
                                                       uint32_t* __restrict__ keys_out, PermuteArgs a)
{
  const int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= n) return;
  uint32_t p;
  const int64_t i = stable_place(k, members, keys, off, keys_out, p);
  move_atom<ND>(a, p, i);
}

// One thread per atom; stencil order dz, dy, dx (outer to inner), in-cell order
// ascending -- the same visit order as the oracle, so lists match entry by entry.
__global__ void __launch_bounds__(256) k_build(
    int64_t n, const Pos4* __restrict__ pos, const uint32_t* __restrict__ keys,
    const BoxDev* __restrict__ box, int px, int py, int pz, int nx, int ny, int nz,
    int64_t ncell_rep, const int* __restrict__ cell_off, double rl2,
    uint32_t* __restrict__ nbr, int* __restrict__ nnb, int nmax, int64_t npad,
    unsigned long long* __restrict__ maxcnt, const XformDev* __restrict__ xf)
{
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const uint32_t key = keys[i];
  const int64_t r = key / ncell_rep;
  const int64_t cl = key - r * ncell_rep;
  const int cx = (int)(cl % nx);
  const int cy = (int)((cl / nx) % ny);
  const int cz = (int)(cl / ((int64_t)nx * ny));
  const BoxDev& b = box[r];
  const Pos4 pi = load_pos(pos, i);
  int cnt = 0;
  for (int dz = -1; dz <= 1; dz++) {
    int z = cz + dz, kz = 0;
    if (z < 0) { if (!pz) continue; z += nz; kz = -1; }
    else if (z >= nz) { if (!pz) continue; z -= nz; kz = 1; }
    for (int dy = -1; dy <= 1; dy++) {
      int y = cy + dy, ky = 0;
      if (y < 0) { if (!py) continue; y += ny; ky = -1; }
      else if (y >= ny) { if (!py) continue; y -= ny; ky = 1; }
      for (int dx = -1; dx <= 1; dx++) {
        int x = cx + dx, kx = 0;
        if (x < 0) { if (!px) continue; x += nx; kx = -1; }
        else if (x >= nx) { if (!px) continue; x -= nx; kx = 1; }
        const int64_t cell = r * ncell_rep + ((int64_t)z * ny + y) * nx + x;
        const int j0 = cell_off[cell], j1 = cell_off[cell + 1];
        const bool self_img = (kx == 0 && ky == 0 && kz == 0);
        for (int j = j0; j < j1; j++) {
          if (self_img && j == (int)i) continue;
          const Pos4 pj = load_pos(pos, j);
          double ddx = xsmd_image(pj.x, kx, b.L[0]) - pi.x;
          double ddy = xsmd_image(pj.y, ky, b.L[1]) - pi.y;
          double ddz = xsmd_image(pj.z, kz, b.L[2]) - pi.z;
          if (xf) xsmd_xform_apply(xf->m, &ddx, &ddy, &ddz);
          if (xsmd_d2(ddx, ddy, ddz) < rl2) {
            if (cnt < nmax) nbr[(int64_t)cnt * npad + i] = xsmd_nbr_encode((uint32_t)j, kx, ky, kz);
            cnt++;
          }
        }
      }
    }
  }
  nnb[i] = cnt;
  if (cnt > nmax) atomicMax(maxcnt, (unsigned long long)cnt);
}

// block-wide max of a non-negative double
__device__ __forceinline__ void block_max_to(double v, double* out)
{
  for (int off = 32; off > 0; off >>= 1) v = fmax(v, __shfl_xor(v, off));
  __shared__ double sh[kBlock / 64];
  if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = v;
  __syncthreads();
  if (threadIdx.x == 0) {
    double m = sh[0];
    for (int w = 1; w < (int)(blockDim.x >> 6); w++) m = fmax(m, sh[w]);
    *out = m;
  }
}

// Largest squared displacement since the last build: each workgroup's maximum goes to host
// memory (out, kDisplGroups values), where they are put together; a clear, an atomic per
// workgroup on one word and a copy back took as long as the sweep at 130 k atoms.
__global__ void __launch_bounds__(256) k_max_displ2(int64_t n, const Pos4* __restrict__ pos,
                                                    const double* __restrict__ rrx,
                                                    const double* __restrict__ rry,
                                                    const double* __restrict__ rrz, double* __restrict__ out,
                                                    const XformDev* __restrict__ xf)
{
  double m = 0.0;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x) {
    const Pos4 p = load_pos(pos, i);
    double ux = p.x - rrx[i], uy = p.y - rry[i], uz = p.z - rrz[i];
    if (xf) xsmd_xform_apply(xf->m, &ux, &uy, &uz);  // the threshold is a physical distance
    m = fmax(m, xsmd_d2(ux, uy, uz));
  }
  block_max_to(m, out + blockIdx.x);
}

__global__ void k_pair_count(int64_t n, int64_t npad, const Pos4* __restrict__ pos,
                             const uint16_t* __restrict__ rep, const BoxDev* __restrict__ box,
                             const uint32_t* __restrict__ nbr, const int* __restrict__ nnb, double rc2,
                             unsigned long long* __restrict__ out, const XformDev* __restrict__ xf)
{
  unsigned long long e = 0, w = 0;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x) {
    const double* L = box[rep ? rep[i] : 0].L;
    const Pos4 pi = load_pos(pos, i);
    const int cnt = nnb[i];
    e += cnt;
    for (int k = 0; k < cnt; k++) {
      const uint32_t en = nbr[(int64_t)k * npad + i];
      const Pos4 pj = load_pos(pos, xsmd_nbr_index(en));
      double dx = xsmd_image(pj.x, xsmd_nbr_img_x(en), L[0]) - pi.x;
      double dy = xsmd_image(pj.y, xsmd_nbr_img_y(en), L[1]) - pi.y;
      double dz = xsmd_image(pj.z, xsmd_nbr_img_z(en), L[2]) - pi.z;
      if (xf) xsmd_xform_apply(xf->m, &dx, &dy, &dz);
      if (xsmd_d2(dx, dy, dz) <= rc2) w++;
    }
  }
  for (int off = 32; off > 0; off >>= 1) {
    e += __shfl_xor(e, off);
    w += __shfl_xor(w, off);
  }
  if ((threadIdx.x & 63) == 0) {
    atomicAdd(out, e);
    atomicAdd(out + 1, w);
  }
}

}  // namespace

void build_neighbor_list(Ctx& c, double rcut, double skin, bool prefer_block, bool keep_accel)
{
  ProfScope prof(c.prof, c.stream, XS_PROF_NEIGHBORS);
  const int64_t n = c.n;
  if (n == 0) {
    c.list_valid = true;
    c.list_rcut = rcut;
    c.list_skin = skin;
    c.list_kind = ListKind::Global;
    c.global_from_block = false;
    return;
  }
  c.list_valid = false;  // until the new list is complete
  const double rl = rcut + skin;
  if (!(rl > 0)) throw Error(XS_E_ARG, "rcut + skin must be positive");

  // cell grid: common dims for all replicas (from the smallest box), each
  // replica with its own n/L so every cell is at least rl wide (in grid space,
  // rl times the xform's reach along the axis)
  for (int a = 0; a < 3; a++) {
    const double rla = c.xf.on ? rl * xsmd_xform_reach(c.xf.mi, a) : rl;
    int nmin = 1 << 30;
    for (const BoxDev& b : c.box_h) nmin = std::min(nmin, xsmd_cells_along(b.L[a], rla));
    c.nc[a] = nmin;
  }
  for (BoxDev& b : c.box_h)
    for (int a = 0; a < 3; a++) b.inv_cs[a] = c.nc[a] / b.L[a];
  // the device's copy, when a box or the cell grid is another than at the last build
  const size_t box_bytes = sizeof(BoxDev) * c.box_h.size();
  if (c.box_up.size() != c.box_h.size() || std::memcmp(c.box_up.data(), c.box_h.data(), box_bytes) != 0) {
    c.box_up.clear();
    XS_HIP(hipMemcpyAsync(c.box_d.p, c.box_h.data(), box_bytes, hipMemcpyHostToDevice, c.stream));
    c.box_up = c.box_h;
  }
  c.ncell_rep = (int64_t)c.nc[0] * c.nc[1] * c.nc[2];
  c.ncell_tot = c.ncell_rep * c.nrep;
  if (c.ncell_tot >= (int64_t)1 << 32) throw Error(XS_E_LIMIT, "too many cells");

  const unsigned g = grid_for(n);
  c.cell_off.reserve(c.ncell_tot + 1);
  if (c.cell_count.n < (size_t)c.ncell_tot || !c.counts_clear) {
    c.cell_count.reserve(c.ncell_tot);
    XS_HIP(hipMemsetAsync(c.cell_count.p, 0, sizeof(uint32_t) * c.cell_count.n, c.stream));
  }
  c.counts_clear = false;  // until k_cell_offsets, which clears them, is queued
  k_cell_count<<<g, kBlock, 0, c.stream>>>(n, c.pos.p, c.has_rep ? c.rep.p : nullptr, c.box_d.p, c.periodic[0],
                                           c.periodic[1], c.periodic[2], c.nc[0], c.nc[1], c.nc[2], c.ncell_rep,
                                           c.keys.p, c.vals.p, c.cell_count.p);
  XS_HIP(hipGetLastError());
  // runs of at least 2048 cells, at most 1024 of them (each workgroup adds up the sums
  // of the runs before its own)
  const int64_t items = std::max<int64_t>(2048, (c.ncell_tot + 1023) / 1024);
  const unsigned runs = (unsigned)((c.ncell_tot + items - 1) / items);
  c.cell_sums.reserve(1024);
  if (runs > 1) {
    k_cell_sums<<<runs, kScanThreads, 0, c.stream>>>(c.ncell_tot, items, c.cell_count.p, c.cell_sums.p);
    XS_HIP(hipGetLastError());
  }
  k_cell_offsets<<<runs, kScanThreads, 0, c.stream>>>(c.ncell_tot, items, c.cell_count.p, c.cell_sums.p, c.cell_off.p);
  XS_HIP(hipGetLastError());
  c.counts_clear = true;
  k_cell_place<<<g, kBlock, 0, c.stream>>>(n, c.keys.p, c.vals.p, c.cell_off.p, c.vals2.p);
  XS_HIP(hipGetLastError());

  PermuteArgs pa{};
  pa.pos_src = c.pos.p;
  pa.pos_dst = c.pos2.p;
  pa.rrx = c.rrx.p;
  pa.rry = c.rry.p;
  pa.rrz = c.rrz.p;
  const double* src[6] = {c.vx.p, c.vy.p, c.vz.p, c.ax.p, c.ay.p, c.az.p};
  double* dst[6] = {c.vx2.p, c.vy2.p, c.vz2.p, c.ax2.p, c.ay2.p, c.az2.p};
  for (int d = 0; d < 6; d++) {
    pa.src[d] = src[d];
    pa.dst[d] = dst[d];
  }
  pa.type_src = c.type.p;
  pa.type_dst = c.type2.p;
  pa.id_src = c.id.p;
  pa.id_dst = c.id2.p;
  pa.rep_src = c.has_rep ? c.rep.p : nullptr;
  pa.rep_dst = c.has_rep ? c.rep2.p : nullptr;
  if (n <= kFusedOrder) {
    (keep_accel ? k_order_permute<6> : k_order_permute<3>)<<<g, kBlock, 0, c.stream>>>(n, c.vals2.p, c.keys.p,
                                                                                       c.cell_off.p, c.keys2.p, pa);
  } else {
    k_cell_order<<<g, kBlock, 0, c.stream>>>(n, c.vals2.p, c.keys.p, c.cell_off.p, c.vals.p, c.keys2.p);
    XS_HIP(hipGetLastError());
    (keep_accel ? k_permute<6> : k_permute<3>)<<<g, kBlock, 0, c.stream>>>(n, c.vals.p, pa);
  }
  XS_HIP(hipGetLastError());
  c.pos.swap(c.pos2);
  c.vx.swap(c.vx2);
  c.vy.swap(c.vy2);
  c.vz.swap(c.vz2);
  if (keep_accel) {
    c.ax.swap(c.ax2);
    c.ay.swap(c.ay2);
    c.az.swap(c.az2);
  }
  c.type.swap(c.type2);
  c.id.swap(c.id2);
  if (c.has_rep) c.rep.swap(c.rep2);
  c.rho_state = RhoState::None;  // per-atom EAM state is in the old order
  c.rho_ckpt = false;

  // list capacity: estimate from the density, grow to the measured maximum on overflow
  if (c.nmax == 0) {
    double vol = 0;
    for (const BoxDev& b : c.box_h) vol += b.L[0] * b.L[1] * b.L[2] * xform_det(c.xf);
    const double dens = (double)n / vol;
    const double est = dens * 4.18879020478639 * rl * rl * rl;  // 4/3 pi rl^3
    c.nmax = std::max(16, (int)std::ceil(est * 1.25 / 8.0) * 8);
  }
  const double rl2 = rl * rl;
  c.global_from_block = false;
  c.list_kind = ListKind::Global;
  if (prefer_block && !c.block_disabled) {
    block_setup(c);
    if (block_feasible(c) && block_build(c, rl2)) c.list_kind = ListKind::Block;
  }
  for (int attempt = 0; c.list_kind == ListKind::Global && attempt < 2; attempt++) {
    c.nbr.reserve((size_t)c.nmax * c.npad);
    c.nnb.reserve(c.npad);
    XS_HIP(hipMemsetAsync(c.dscalar.p, 0, sizeof(unsigned long long), c.stream));
    k_build<<<g, kBlock, 0, c.stream>>>(n, c.pos.p, c.keys2.p, c.box_d.p, c.periodic[0], c.periodic[1],
                                        c.periodic[2], c.nc[0], c.nc[1], c.nc[2], c.ncell_rep, c.cell_off.p, rl2,
                                        c.nbr.p, c.nnb.p, c.nmax, c.npad, c.dscalar.p, c.xf_dev());
    XS_HIP(hipGetLastError());
    XS_HIP(hipMemcpyAsync(c.hscalar, c.dscalar.p, sizeof(unsigned long long), hipMemcpyDeviceToHost,
                          c.stream));
    XS_HIP(hipStreamSynchronize(c.stream));
    const unsigned long long need = c.hscalar[0];
    if (need == 0) break;
    if (attempt == 1) throw Error(XS_E_STATE, "neighbour list overflow after resize");
    c.nmax = (int)((need + 7) / 8 * 8 + 8);
  }
  c.list_valid = true;
  c.list_rcut = rcut;
  c.list_skin = skin;
}

void pair_count(Ctx& c, double rcut, int64_t& entries, int64_t& within)
{
  entries = within = 0;
  if (c.n == 0) return;
  ensure_global_list(c);
  XS_HIP(hipMemsetAsync(c.dscalar.p + 2, 0, 2 * sizeof(unsigned long long), c.stream));
  const unsigned g = std::min<unsigned>(grid_for(c.n), 4096);
  k_pair_count<<<g, kBlock, 0, c.stream>>>(c.n, c.npad, c.pos.p, c.has_rep ? c.rep.p : nullptr, c.box_d.p,
                                           c.nbr.p, c.nnb.p, rcut * rcut, c.dscalar.p + 2, c.xf_dev());
  XS_HIP(hipGetLastError());
  XS_HIP(hipMemcpyAsync(c.hscalar + 2, c.dscalar.p + 2, 2 * sizeof(unsigned long long), hipMemcpyDeviceToHost,
                        c.stream));
  XS_HIP(hipStreamSynchronize(c.stream));
  entries = (int64_t)c.hscalar[2];
  within = (int64_t)c.hscalar[3];
}

double max_displacement2(Ctx& c)
{
  if (c.n == 0) return 0.0;
  const unsigned g = std::min<unsigned>(grid_for(c.n), kDisplGroups);
  k_max_displ2<<<g, kBlock, 0, c.stream>>>(c.n, c.pos.p, c.rrx.p, c.rry.p, c.rrz.p, c.hdispl, c.xf_dev());
  XS_HIP(hipGetLastError());
  XS_HIP(hipStreamSynchronize(c.stream));
  return *std::max_element(c.hdispl, c.hdispl + g);
}

}  // namespace xsmd
