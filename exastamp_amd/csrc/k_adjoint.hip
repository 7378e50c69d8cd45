// k_adjoint.hip -- reverse mode of the EAM force/energy with respect to the
// tabulated knots (no counterpart in exaStamp; the fitting capability built on
// its eam_alloy tables).
//
// For a loss L(F, E) with g_i = dL/dF_i and per-replica gE = dL/dE:
//   dL/dtheta = sum_i gE_i dE/dtheta - dD/dtheta,   D = sum_i g_i . dE/dx_i,
// because F_i = -dE/dx_i.  With u_ij = (x_i - x_j)/r and s_ij = u_ij . (g_i - g_j),
//   D = sum_i F'_i drho_i + 1/2 sum_i sum_j phi'_ij s_ij,   drho_i = sum_j rho'_tj(r_ij) s_ij.
// Differentiating through both EAM passes (rho_i inside F'_i is the mixed second
// derivative) gives, per atom and per pair of the full list,
//   F table at rho_i : value weight  gE_i conv,
//                      slope weight  conv (gE_i (rho_i - rhomax)^+ - drho_i)
//   rho table at r_ij: value weight  gE_i F'_i - lambda_i,  slope weight  -F'_i s_ij,
//                      lambda_i = F''(rho_i) drho_i
//   z2r table at r_ij: value weight  conv (gE_i / (2r) + s_ij / (2r^2)),
//                      slope weight  -conv s_ij / (2r)
// where "slope" multiplies the derivative of the spline with respect to r (or rho).
// rho_i and F'_i come from the forward pass (checkpointed, not recomputed).
//
// Every undirected pair is taken once, from its atom with the smaller index: the two
// list entries of a pair share r, the knot and s_ij, their z2r weights are equal, and
// for atoms of one species so are their rho rows, so the second one costs two adds.
//
// A spline row is the Hermite cubic of the values f and slopes s at its two knots, so the
// weights of a pair go to f and s of knots m and m + 1 (FP64); a last kernel applies the
// transpose of the knot -> slope map.
//
// Accumulation.  All pairs of a shell fall on a few hundred rows, and all atoms on
// a few F rows, so atomics on the gradient rows in HBM serialise.  Instead a
// launch covers a set of row windows (one per table) that fit in LDS: persistent
// workgroups walk all atoms (or pairs), add the contributions that fall in a window
// into their LDS copy (LDS FP64 atomics), and write it out as a partial; a second
// kernel sums the partials over the workgroups in a fixed order.  Windows cover
// every row of every table, one launch per group of windows.  Two sums per knot (16
// bytes, against 32 for four coefficients per row) let the five pair tables of two
// species at 2000 knots share one launch's 160 KB.
//
// The first sweep (drho_i, lambda_i) needs no accumulators and runs on the brick lists
// like the density pass (k_block_adj_b1); the second gathers positions and loss gradients
// through the list, since the accumulators take the LDS a brick's halo would need.
// Bound by the LDS atomics (8 to 12 per pair) and the gathers (64 bytes per pair).
// 1.04 M Cu/Ni atoms, 2000 knots: first sweep 201 us, second 473 us, F rows 12 us; walking
// every list entry on the global list, with four coefficients per row and so three
// launches, took 1107 + 2 x 645 us.  55 k atoms, 500 knots: 13 + 35 us against 80.
#include "pair_math.hpp"

#include <algorithm>

namespace xsmd {
namespace {

__device__ __forceinline__ int64_t lblock()
{
  const unsigned b = blockIdx.x, g = gridDim.x;
  if (g & 7u) return b;
  return (int64_t)(b & 7u) * (g >> 3) + (b >> 3);
}

struct AdjArgs {
  int64_t n, npad;
  const Pos4* pos;        // x y z F'_i
  Pos4* gvec;             // g_i (dL/dF_i) in cell order, w = lambda_i (first sweep out)
  const double* rho;      // checkpointed rho_i
  double* drho;           // first sweep out
  const uint8_t* type;
  const uint16_t* rep;
  const BoxDev* box;
  const uint32_t* nbr;    // global list, or
  const uint16_t* nbr16;  // brick list: slots,
  const uint32_t* stage;  // the global entry of each slot,
  const uint32_t* base;   // and where the slots of atom i's brick start
  const int* nnb;
  const double* gE;       // per replica
  double rc2;
  int nel, nr, nrho;      // table ids: F 0..nel-1, rho nel..2nel-1, z2r 2nel..
  double rdr, rdrho, rhomax, conv;
  uint32_t types;         // types slot of eam_alloy_force: bit t set = species t takes part
  const XformDev* xf;     // physical displacements m * (r_j(image) - r_i) when not NULL
};

__device__ __forceinline__ bool adj_on(const AdjArgs& a, int type) { return (a.types >> type) & 1u; }
__device__ __forceinline__ int f_table(const AdjArgs& a, int type) { return type < a.nel ? type : 0; }

// LDS row windows of one launch: of table T the knots lo + 1 .. lo + rows at LDS rows
// off .. off + rows - 1 (rows = 0: none)
struct AdjWin {
  int lo, rows, off;
};
constexpr int kAdjTables = 7 + 7 + 28;
constexpr int kAdjThreads = 1024;
struct AdjWindows {
  int total;  // rows of the launch: as many values, then as many slopes
  AdjWin w[kAdjTables];
};
__host__ __device__ inline size_t adj_lds_bytes(int total)
{
  return (size_t)total * 2 * sizeof(double) + (kAdjTables * sizeof(AdjWin) + 7) / 8 * 8;
}

// the accumulators of a workgroup, and the windows beside them: their lookup by table is
// per lane
struct AdjAcc {
  double* f;
  double* s;
  const AdjWin* win;
  int total;
  __device__ __forceinline__ AdjAcc(double* lds, const AdjWindows& W)
      : f(lds), s(lds + W.total), win(reinterpret_cast<const AdjWin*>(lds + 2 * W.total)), total(W.total)
  {
    AdjWin* w = reinterpret_cast<AdjWin*>(lds + 2 * W.total);
    for (int k = threadIdx.x; k < kAdjTables; k += blockDim.x) w[k] = W.w[k];
    for (int q = threadIdx.x; q < 2 * total; q += blockDim.x) lds[q] = 0.0;
    __syncthreads();
  }
  __device__ __forceinline__ void out(double* __restrict__ part) const
  {
    __syncthreads();
    double* dst = part + (int64_t)blockIdx.x * 2 * total;
    for (int q = threadIdx.x; q < 2 * total; q += blockDim.x) dst[q] = f[q];
  }
};

// Hermite basis at fraction p of knots m, m + 1: of a value weight and of the weight of
// the derivative with respect to p
struct Hermite {
  double h01, h10, h11, d01, d10, d11;
  __device__ __forceinline__ explicit Hermite(double p)
  {
    const double q = 1.0 - p, pq = p * q;
    h01 = p * p * (3.0 - 2.0 * p);
    h10 = pq * q;
    h11 = -pq * p;
    d01 = 6.0 * pq;
    d10 = q * (1.0 - 3.0 * p);
    d11 = p * (3.0 * p - 2.0);
  }
};

// value weight wv and p-derivative weight ws at knot m (1-based) of table T; WHOLE: the
// launch holds every row of its tables
template <bool WHOLE>
__device__ __forceinline__ void adj_add(const AdjAcc& A, int T, int m, const Hermite& h, double wv, double ws)
{
  if constexpr (WHOLE) {
    const double f = wv * h.h01 + ws * h.d01;
    const int at = A.win[T].off + m - 1;
    atomicAdd(A.f + at, wv - f);
    atomicAdd(A.f + at + 1, f);
    atomicAdd(A.s + at, wv * h.h10 + ws * h.d10);
    atomicAdd(A.s + at + 1, wv * h.h11 + ws * h.d11);
    return;
  }
  const AdjWin w = A.win[T];
  const int row = m - 1 - w.lo;
  const double f1 = wv * h.h01 + ws * h.d01;
  if ((unsigned)row < (unsigned)w.rows) {
    atomicAdd(A.f + w.off + row, wv - f1);
    atomicAdd(A.s + w.off + row, wv * h.h10 + ws * h.d10);
  }
  if ((unsigned)(row + 1) < (unsigned)w.rows) {
    atomicAdd(A.f + w.off + row + 1, f1);
    atomicAdd(A.s + w.off + row + 1, wv * h.h11 + ws * h.d11);
  }
}

// knot and fraction of x as the spline evaluation finds them (knots 1 .. n - 1)
__device__ __forceinline__ void adj_knot(double x, double rscale, int n, int& m, double& p)
{
  p = x * rscale + 1.0;
  m = max(1, min((int)p, n - 1));
  p = fmin(p - (double)m, 1.0);
}

// First sweep on the global list: kB1Lanes lanes per atom gather through it.
constexpr int kB1Lanes = 4;
template <class Real, bool MULTI>
__global__ void __launch_bounds__(256) k_adj_b1(AdjArgs a, EamTabDev<Real> t)
{
  const int sub = threadIdx.x % kB1Lanes;
  const int64_t i = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) / kB1Lanes;
  if (i >= a.n) return;  // the lanes of an atom leave together (their shuffles)
  const int ti = MULTI ? a.type[i] : 0;
  const double* Lb = a.box[a.rep ? a.rep[i] : 0].L;
  const Pos4 pi = load_pos(a.pos, i);
  const double* gi = reinterpret_cast<const double*>(a.gvec + i);
  const bool oni = !MULTI || adj_on(a, ti);
  const int cnt = oni ? a.nnb[i] : 0;
  double drho = 0.0;
  for (int k = sub; k < cnt; k += kB1Lanes) {
    const uint32_t e = a.nbr[(int64_t)k * a.npad + i];
    const uint32_t j = xsmd_nbr_index(e);
    const Pos4 pj = load_pos(a.pos, j);
    double dx = xsmd_image(pj.x, xsmd_nbr_img_x(e), Lb[0]) - pi.x;
    double dy = xsmd_image(pj.y, xsmd_nbr_img_y(e), Lb[1]) - pi.y;
    double dz = xsmd_image(pj.z, xsmd_nbr_img_z(e), Lb[2]) - pi.z;
    if (a.xf) xsmd_xform_apply(a.xf->m, &dx, &dy, &dz);
    const double d2 = xsmd_d2(dx, dy, dz);
    if (d2 > a.rc2) continue;
    const int tj = MULTI ? a.type[j] : 0;
    if (MULTI && !adj_on(a, tj)) continue;
    const double* gj = reinterpret_cast<const double*>(a.gvec + j);
    double r, rinv;
    pm::dist(d2, r, rinv);
    const double s = (dx * (gj[0] - gi[0]) + dy * (gj[1] - gi[1]) + dz * (gj[2] - gi[2])) * rinv;
    int m;
    double p;
    adj_knot(r, a.rdr, a.nr, m, p);
    const pm::Q4<Real> row = pm::load4(pm::pair_row(t.slope, t, MULTI && max(ti, tj) < a.nel ? tj : 0, m));
    drho += (((double)row.a * p + (double)row.b) * p + (double)row.c) * s;
  }
#pragma unroll
  for (int off = 1; off < kB1Lanes; off <<= 1) drho += __shfl_xor(drho, off);
  if (sub != 0) return;
  // F'' = d/drho of (c0 p + c1) p + c2, zero where p was clamped
  double p = a.rho[i] * a.rdrho + 1.0;
  const int m = max(1, min((int)p, a.nrho - 1));
  p -= (double)m;
  const Real* row = t.frho + ((int64_t)f_table(a, ti) * (a.nrho + 1) + m) * 8;
  const double fpp = p > 1.0 ? 0.0 : (2.0 * (double)row[4] * p + (double)row[5]) * a.rdrho * a.conv;
  a.drho[i] = drho;
  reinterpret_cast<double*>(a.gvec + i)[3] = oni ? fpp * drho : 0.0;
}

// The F-table weights of atom i (a disabled species has no embedding term)
template <bool MULTI, bool WHOLE>
__device__ __forceinline__ void adj_embed_add(const AdjArgs& a, const AdjAcc& acc, int64_t i)
{
  const int ti = MULTI ? a.type[i] : 0;
  if (MULTI && !adj_on(a, ti)) return;
  const double rho = a.rho[i], ge = a.gE[a.rep ? a.rep[i] : 0];
  int m;
  double p;
  adj_knot(rho, a.rdrho, a.nrho, m, p);
  const double over = rho > a.rhomax ? rho - a.rhomax : 0.0;
  adj_add<WHOLE>(acc, f_table(a, ti), m, Hermite(p), ge * a.conv, a.conv * (ge * over - a.drho[i]) * a.rdrho);
}

// F-table rows where they have launches of their own
template <bool MULTI>
__global__ void __launch_bounds__(kAdjThreads) k_adj_fsum(AdjArgs a, AdjWindows W, double* __restrict__ part)
{
  extern __shared__ double lds[];
  const AdjAcc acc(lds, W);
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < a.n; i += (int64_t)gridDim.x * blockDim.x)
    adj_embed_add<MULTI, false>(a, acc, i);
  acc.out(part);
}

// Second sweep: the rho and z2r rows of every pair, from its atom with the smaller index
// (an atom's own images come as two entries, which take half each), and with FSUM the
// F-table rows.  1 << lanes_log lanes per atom.  A lane first marks which of its entries
// are its to take, up to 64 of them, then walks the marked ones, so that lanes whose
// neighbour had the larger index do not idle through the pair's arithmetic; the next pair's
// records are fetched while one is evaluated (1.04 M atoms: 521 -> 473 us with the rows'
// window tests left out where the launch holds whole tables).
template <bool MULTI, bool BLOCK, bool FSUM, bool WHOLE>
__global__ void __launch_bounds__(kAdjThreads) k_adj_pairs(AdjArgs a, AdjWindows W, int lanes_log,
                                                           double* __restrict__ part)
{
  extern __shared__ double lds[];
  const AdjAcc acc(lds, W);
  const int lanes = 1 << lanes_log, sub = threadIdx.x & (lanes - 1);
  // a contiguous range of atoms per workgroup, neighbouring ranges on one XCD
  const int64_t per = (a.n + gridDim.x - 1) / gridDim.x;
  const int64_t first = lblock() * per, end = min(first + per, a.n);
  for (int64_t i = first + (threadIdx.x >> lanes_log); i < end; i += blockDim.x >> lanes_log) {
    if (FSUM && sub == 0) adj_embed_add<MULTI, WHOLE>(a, acc, i);
    const int ti = MULTI ? a.type[i] : 0;
    const int rep = a.rep ? a.rep[i] : 0;
    const double* Lb = a.box[rep].L;
    const Pos4 pi = load_pos(a.pos, i);
    const Pos4 gi = load_pos(a.gvec, i);
    const double ge = a.gE[rep];
    const int cnt = (!MULTI || adj_on(a, ti)) ? a.nnb[i] : 0;
    const uint32_t base = BLOCK ? a.base[i] : 0;
    const uint32_t iu = (uint32_t)i;
    // bit 8 t + u of a lane's mask: place u of its t-th group (BLOCK), or its (8 t + u)-th entry
    for (int k0 = 0; k0 < cnt; k0 += 64 * lanes) {
      unsigned long long mask = 0;
      for (int t = 0; t < 8; t++) {
        uint32_t m8 = 0;
        if constexpr (BLOCK) {
          const int g = (k0 >> 3) + sub + lanes * t;
          if (8 * g >= cnt) break;
          const uint4 w = *reinterpret_cast<const uint4*>(a.nbr16 + (((int64_t)g * a.npad + i) << 3));
          const uint32_t ws[4] = {w.x, w.y, w.z, w.w};
#pragma unroll
          for (int u = 0; u < 8; u++) {
            const int k = 8 * g + (u < 4 ? 2 * u : 2 * u - 7);
            const uint32_t slot = u & 1 ? ws[u >> 1] >> 16 : ws[u >> 1] & 0xffffu;
            const uint32_t j = xsmd_nbr_index(a.stage[base + (k < cnt ? slot : 0u)]);
            m8 |= (k < cnt && j >= iu ? 1u : 0u) << u;
          }
        } else {
          for (int u = 0; u < 8; u++) {
            const int k = k0 + sub + lanes * (8 * t + u);
            m8 |= (k < cnt && xsmd_nbr_index(a.nbr[(int64_t)k * a.npad + i]) >= iu ? 1u : 0u) << u;
          }
        }
        mask |= (unsigned long long)m8 << (8 * t);
      }
      // the marked entry with the smallest bit, and the mask without it
      const auto pop = [&]() {
        const int bit = __ffsll(mask) - 1;
        mask &= mask - 1;
        if constexpr (BLOCK) {
          const int g = (k0 >> 3) + sub + lanes * (bit >> 3);
          return a.stage[base + a.nbr16[(((int64_t)g * a.npad + i) << 3) + (bit & 7)]];
        } else {
          return a.nbr[(int64_t)(k0 + sub + lanes * bit) * a.npad + i];
        }
      };
      // each pair's records are on their way while the pair before it is evaluated
      bool more = mask != 0;
      uint32_t e_next = 0;
      Pos4 pj_next{}, gj_next{};
      int tj_next = 0;
      const auto fetch = [&]() {
        e_next = pop();
        const uint32_t j = xsmd_nbr_index(e_next);
        pj_next = load_pos(a.pos, j);
        gj_next = load_pos(a.gvec, j);
        if (MULTI) tj_next = a.type[j];
      };
      if (more) fetch();
      while (more) {
        const uint32_t e = e_next, j = xsmd_nbr_index(e);
        const Pos4 pj = pj_next, gj = gj_next;
        const int tj = tj_next;
        more = mask != 0;
        if (more) fetch();
        if (MULTI && !adj_on(a, tj)) continue;
        double dx = pj.x - pi.x, dy = pj.y - pi.y, dz = pj.z - pi.z;
        const bool image = e >> XSMD_NBR_INDEX_BITS;
        if (image) {
          dx = xsmd_image(pj.x, xsmd_nbr_img_x(e), Lb[0]) - pi.x;
          dy = xsmd_image(pj.y, xsmd_nbr_img_y(e), Lb[1]) - pi.y;
          dz = xsmd_image(pj.z, xsmd_nbr_img_z(e), Lb[2]) - pi.z;
        }
        if (a.xf) xsmd_xform_apply(a.xf->m, &dx, &dy, &dz);
        const double d2 = xsmd_d2(dx, dy, dz);
        // wi, wj: which of the pair's two entries count; through an image the distance
        // from j rounds by itself, so a pair at the cutoff may count from one side only
        double wi = d2 <= a.rc2 ? 1.0 : 0.0, wj = wi;
        if (image) {
          double ux = xsmd_image(pi.x, -xsmd_nbr_img_x(e), Lb[0]) - pj.x;
          double uy = xsmd_image(pi.y, -xsmd_nbr_img_y(e), Lb[1]) - pj.y;
          double uz = xsmd_image(pi.z, -xsmd_nbr_img_z(e), Lb[2]) - pj.z;
          if (a.xf) xsmd_xform_apply(a.xf->m, &ux, &uy, &uz);
          wj = xsmd_d2(ux, uy, uz) <= a.rc2 ? 1.0 : 0.0;
          if (j == iu) {
            wi *= 0.5;
            wj *= 0.5;
          }
        }
        const double both = wi + wj;
        if (both == 0.0) continue;
        double r, ir;
        pm::dist(d2, r, ir);
        // s_ij = u_ij . (g_i - g_j), u_ij = -(dx,dy,dz)/r
        const double s = (dx * (gj.x - gi.x) + dy * (gj.y - gi.y) + dz * (gj.z - gi.z)) * ir;
        int m;
        double p;
        adj_knot(r, a.rdr, a.nr, m, p);
        const Hermite h(p);
        int ri = 0, rj = 0, z = a.nel;
        if constexpr (MULTI) pm::pair_planes(a.nel, ti, tj, ri, rj, z);
        const double srdr = s * a.rdr;
        const double vi = wi * (ge * pi.w - gi.w), vj = wj * (ge * pj.w - gj.w);
        const double si = -wi * pi.w * srdr, sj = -wj * pj.w * srdr;
        if (!MULTI || ri == rj) {
          adj_add<WHOLE>(acc, a.nel + ri, m, h, vi + vj, si + sj);
        } else {
          adj_add<WHOLE>(acc, a.nel + rj, m, h, vi, si);  // rho_j's table at atom i
          adj_add<WHOLE>(acc, a.nel + ri, m, h, vj, sj);
        }
        const double c = 0.5 * both * a.conv * ir;
        adj_add<WHOLE>(acc, a.nel + z, m, h, c * (ge + s * ir), -c * srdr);
      }
    }
  }
  acc.out(part);
}

// Sum of the partials of `groups` workgroups into the gradient rows of this launch's
// windows (each row belongs to exactly one window of one launch).  A workgroup takes
// 64 consecutive values; its 16 waves sum the partials w = wave, wave + 16, ...
// (coalesced), and the 16 sums are added in wave order, so the result does not
// depend on scheduling.
constexpr int kRedThreads = 1024;
__global__ void __launch_bounds__(kRedThreads) k_adj_reduce(AdjWindows W, int nel, int nz, int nrho, int nr, int groups,
                                                            const double* __restrict__ part, double* __restrict__ g)
{
  __shared__ double red[kRedThreads];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int q = blockIdx.x * 64 + lane;
  const bool in = q < 2 * W.total;
  double v = 0.0;
  if (in)
    for (int w = wave; w < groups; w += kRedThreads / 64) v += part[(int64_t)w * 2 * W.total + q];
  red[threadIdx.x] = v;
  __syncthreads();
  if (wave != 0 || !in) return;
  v = red[lane];
  for (int k = 1; k < kRedThreads / 64; k++) v += red[k * 64 + lane];
  const bool slope = q >= W.total;
  const int row = slope ? q - W.total : q;
  const int64_t knots = (int64_t)nel * nrho + (int64_t)(nel + nz) * nr;
  for (int T = 0; T < 2 * nel + nz; T++) {
    const AdjWin w = W.w[T];
    if (row < w.off || row >= w.off + w.rows) continue;
    const int64_t g0 = T < nel ? (int64_t)T * nrho : (int64_t)nel * nrho + (int64_t)(T - nel) * nr;
    g[(slope ? knots : 0) + g0 + w.lo + row - w.off] = v;
  }
}

// g (dL/dF) from id order into cell order as position-like records
// (and times `scale`); the first nrep threads scale the per-replica dL/dE
__global__ void k_gather_g(int64_t n, const int64_t* __restrict__ id, const double* __restrict__ g_id,
                           Pos4* __restrict__ gvec, double scale, const double* __restrict__ gE_in,
                           double* __restrict__ gE, int nrep)
{
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < nrep) gE[i] = gE_in[i] * scale;
  if (i >= n) return;
  const int64_t q = id[i];
  store_pos(gvec, i, Pos4{g_id[3 * q] * scale, g_id[3 * q + 1] * scale, g_id[3 * q + 2] * scale, 0.0});
}

// ---------------------------------------------------------------------------
// Lennard-Jones adjoint with respect to (epsilon, sigma).
// With w(r) = e'(r)/r (the force factor, F_i = sum_j w(r_ij) (x_j - x_i)) and the
// pair energy 1/2 (e(r) - e(rc)) per list entry (pair_potential_impl.hxx:487-498,
// lennard_jones.h:40-50), for theta in {epsilon, sigma}:
//   dL/dtheta = sum over list entries (i, j), r_ij <= rc, of
//               1/2 gE_rep(i) (de/dtheta(r) - de/dtheta(rc)) + dw/dtheta(r) g_i.(x_j - x_i)
// with s6 = (sigma/r)^6, s12 = s6^2:
//   de/deps = 4 (s12 - s6),             de/dsigma = 4 eps (12 s12 - 6 s6) / sigma,
//   dw/deps = -24 (2 s12 - s6) / r^2,   dw/dsigma = -24 eps (24 s12 - 6 s6) / (sigma r^2).
// One thread per atom walks the global list in FP64; each workgroup writes its two
// sums, and one workgroup adds the partials in a fixed order (no atomics, so the
// result does not depend on scheduling).
// ---------------------------------------------------------------------------
struct LjAdjArgs {
  int64_t n, npad;
  const Pos4* pos;
  const Pos4* gvec;       // dL/dF_i in cell order
  const uint16_t* rep;
  const BoxDev* box;
  const uint32_t* nbr;
  const int* nnb;
  const double* gE;       // per replica
  double rc2, eps, sigma, sigma2;
  double decut_eps, decut_sigma;  // de/deps and de/dsigma at r = rc
  const XformDev* xf;
};

constexpr int kLjAdjThreads = 256;

// a and b summed over the workgroup in a fixed order (shuffle tree within each wave,
// then the waves in index order through red); every thread calls it and gets both sums
__device__ __forceinline__ void block_sum2(double a, double b, double* red, double& ra, double& rb)
{
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) {
    a += __shfl_xor(a, off);
    b += __shfl_xor(b, off);
  }
  const int w = threadIdx.x >> 6, nw = blockDim.x >> 6;
  if ((threadIdx.x & 63) == 0) {
    red[2 * w] = a;
    red[2 * w + 1] = b;
  }
  __syncthreads();
  ra = rb = 0.0;
  for (int k = 0; k < nw; k++) {
    ra += red[2 * k];
    rb += red[2 * k + 1];
  }
}

__global__ void __launch_bounds__(kLjAdjThreads) k_lj_adjoint(LjAdjArgs a, double* __restrict__ part)
{
  __shared__ double red[2 * (kLjAdjThreads / 64)];
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  double ge = 0.0, gs = 0.0;
  if (i < a.n) {
    const int rep = a.rep ? a.rep[i] : 0;
    const double* L = a.box[rep].L;
    const Pos4 pi = load_pos(a.pos, i);
    const Pos4 gi = load_pos(a.gvec, i);
    const double hE = 0.5 * a.gE[rep];
    const int cnt = a.nnb[i];
    for (int k = 0; k < cnt; k++) {
      const uint32_t e = a.nbr[(int64_t)k * a.npad + i];
      const Pos4 pj = load_pos(a.pos, xsmd_nbr_index(e));
      double dx = xsmd_image(pj.x, xsmd_nbr_img_x(e), L[0]) - pi.x;
      double dy = xsmd_image(pj.y, xsmd_nbr_img_y(e), L[1]) - pi.y;
      double dz = xsmd_image(pj.z, xsmd_nbr_img_z(e), L[2]) - pi.z;
      if (a.xf) xsmd_xform_apply(a.xf->m, &dx, &dy, &dz);
      const double d2 = xsmd_d2(dx, dy, dz);
      if (d2 > a.rc2) continue;
      const double ir2 = 1.0 / d2;
      const double s2 = a.sigma2 * ir2;
      const double s6 = s2 * s2 * s2;
      const double s12 = s6 * s6;
      const double gd = gi.x * dx + gi.y * dy + gi.z * dz;
      ge += hE * (4.0 * (s12 - s6) - a.decut_eps) - 24.0 * (2.0 * s12 - s6) * ir2 * gd;
      gs += hE * (4.0 * a.eps * (12.0 * s12 - 6.0 * s6) / a.sigma - a.decut_sigma) -
            24.0 * a.eps * (24.0 * s12 - 6.0 * s6) / a.sigma * ir2 * gd;
    }
  }
  double ra, rb;
  block_sum2(ge, gs, red, ra, rb);
  if (threadIdx.x == 0) {
    part[2 * blockIdx.x] = ra;
    part[2 * blockIdx.x + 1] = rb;
  }
}

// out[0..1] = sum of the nparts partials, each thread a fixed stride of them
__global__ void __launch_bounds__(kLjAdjThreads) k_lj_adjoint_reduce(int64_t nparts, const double* __restrict__ part,
                                                                     double* __restrict__ out)
{
  __shared__ double red[2 * (kLjAdjThreads / 64)];
  double a = 0.0, b = 0.0;
  for (int64_t k = threadIdx.x; k < nparts; k += blockDim.x) {
    a += part[2 * k];
    b += part[2 * k + 1];
  }
  double ra, rb;
  block_sum2(a, b, red, ra, rb);
  if (threadIdx.x == 0) {
    out[0] = ra;
    out[1] = rb;
  }
}

// Row windows of every table (F tables have nrho knots, rho and z2r tables nr), packed
// into launches of at most `limit` LDS rows; `what` selects the F tables (0), the rho and
// z2r tables (1) or all of them (2).
std::vector<AdjWindows> adj_launches(int nel, int nz, int nrho, int nr, int what, int limit)
{
  std::vector<AdjWindows> out;
  AdjWindows cur{};
  const auto add = [&](int T, int rows) {
    for (int lo = 0; lo < rows;) {
      if (cur.total == limit) {
        out.push_back(cur);
        cur = AdjWindows{};
      }
      const int w = std::min(limit - cur.total, rows - lo);
      cur.w[T] = AdjWin{lo, w, cur.total};
      cur.total += w;
      lo += w;
    }
  };
  if (what != 1)
    for (int t = 0; t < nel; t++) add(t, nrho);
  if (what != 0)
    for (int t = 0; t < nel + nz; t++) add(nel + t, nr);
  if (cur.total) out.push_back(cur);
  return out;
}

template <class Real>
void adj_first_sweep(Ctx& c, const AdjArgs& a)
{
  const auto k = eam_multi(c) ? k_adj_b1<Real, true> : k_adj_b1<Real, false>;
  k<<<grid_for(a.n * kB1Lanes), 256, 0, c.stream>>>(a, make_eam_tab<Real>(c));
  XS_HIP(hipGetLastError());
}

void adj_run(Ctx& c, const AdjArgs& a, double rcut, bool mixed)
{
  EamHost& e = c.eam;
  const int nel = e.nel, nz = nel * (nel + 1) / 2;
  const bool multi = eam_multi(c), block = a.nbr16 != nullptr;
  if (block) launch_adj_b1_block(c, rcut, mixed);
  else if (mixed) adj_first_sweep<float>(c, a);
  else adj_first_sweep<double>(c, a);
  // LDS windows as large as one workgroup may hold; one persistent workgroup per CU, of
  // 256 to 1024 threads as the atoms fill them: more of them would each write and have
  // summed a copy of the rows (864 workgroups of 256 threads at 55 k atoms and 1500 rows
  // made the sum of the partials 17 us)
  const int limit = (int)((c.lds_max - adj_lds_bytes(0)) / (2 * sizeof(double)));
  const int64_t cus = std::max(c.num_cu, 1);
  const auto shape = [&](int64_t items, int& groups, int& threads) {
    threads = 256;
    while (threads < kAdjThreads && items > cus * threads) threads *= 2;
    groups = (int)std::max<int64_t>(1, std::min<int64_t>(cus, (items + threads - 1) / threads));
  };
  const auto reduce = [&](const AdjWindows& W, int groups) {
    XS_HIP(hipGetLastError());
    k_adj_reduce<<<(unsigned)((2 * W.total + 63) / 64), kRedThreads, 0, c.stream>>>(
        W, nel, nz, e.nrho, e.nr, groups, c.adj_part.p, c.adj_g.p);
    XS_HIP(hipGetLastError());
  };
  const auto launch = [&](auto k, const AdjWindows& W, int64_t items, auto... args) {
    int groups, threads;
    shape(items, groups, threads);
    const size_t lds = adj_lds_bytes(W.total);
    c.adj_part.reserve((size_t)groups * 2 * W.total);
    XS_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(k), hipFuncAttributeMaxDynamicSharedMemorySize,
                               (int)lds));
    k<<<groups, threads, lds, c.stream>>>(a, W, args..., c.adj_part.p);
    reduce(W, groups);
  };
  // lanes per atom: 2, up to 8 where the atoms do not fill the CUs (1.04 M atoms: 589 us
  // with 1, 473 with 2, 503 with 4, 558 with 8; 55 k: 39.7 with 2, 36.7 with 4, 34.8 with 8)
  int lanes_log = 1;
  while (lanes_log < 3 && (a.n << lanes_log) < cus * kAdjThreads) lanes_log++;
  const auto pairs = [&](const AdjWindows& W, bool fsum) {
    const auto pick = [&](auto m, auto b) {
      constexpr bool M = decltype(m)::value, B = decltype(b)::value;
      bool whole = true;
      for (int T = fsum ? 0 : nel; T < 2 * nel + nz; T++) whole = whole && W.w[T].rows == (T < nel ? e.nrho : e.nr);
      const auto k = whole ? (fsum ? k_adj_pairs<M, B, true, true> : k_adj_pairs<M, B, false, true>)
                           : (fsum ? k_adj_pairs<M, B, true, false> : k_adj_pairs<M, B, false, false>);
      launch(k, W, a.n << lanes_log, lanes_log);
    };
    if (multi && block) pick(std::true_type{}, std::true_type{});
    else if (multi) pick(std::true_type{}, std::false_type{});
    else if (block) pick(std::false_type{}, std::true_type{});
    else pick(std::false_type{}, std::false_type{});
  };
  const std::vector<AdjWindows> all = adj_launches(nel, nz, e.nrho, e.nr, 2, limit);
  if (all.size() == 1) {  // every row fits: one launch
    pairs(all[0], true);
    return;
  }
  for (const AdjWindows& W : adj_launches(nel, nz, e.nrho, e.nr, 1, limit)) pairs(W, false);
  for (const AdjWindows& W : adj_launches(nel, nz, e.nrho, e.nr, 0, limit))
    launch(multi ? k_adj_fsum<true> : k_adj_fsum<false>, W, a.n);
}

}  // namespace

// Transpose of the knot -> value cubic map of spline_interpolate for one table, on the
// host (xs_spline_adjoint, for programs that hold gradients of the coefficients; the
// adjoint's own sweeps sum values and slopes, whose transpose is k_spline_adjoint):
// G holds dL/d(c3,c4,c5,c6) per row (rows 0..n), out receives dL/df for the n knots.
void spline_interpolate_adjoint(int n, double delta, const double* G, double* out)
{
  std::vector<double> gf(n + 2, 0.0), gs(n + 2, 0.0);
  (void)delta;  // the value cubics are in units of the knot spacing
  for (int m = 1; m <= n; m++) {
    const double* g = G + 4 * (size_t)m;
    gf[m] += g[3];  // c6 = f
    gs[m] += g[2];  // c5 = s
    if (m <= n - 1) {
      // c4 = 3 (f[m+1] - f[m]) - 2 s[m] - s[m+1]
      gf[m + 1] += 3.0 * g[1];
      gf[m] -= 3.0 * g[1];
      gs[m] -= 2.0 * g[1];
      gs[m + 1] -= g[1];
      // c3 = s[m] + s[m+1] - 2 (f[m+1] - f[m])
      gs[m] += g[0];
      gs[m + 1] += g[0];
      gf[m + 1] -= 2.0 * g[0];
      gf[m] += 2.0 * g[0];
    }
  }
  // slopes
  gf[2] += gs[1];
  gf[1] -= gs[1];
  gf[3] += 0.5 * gs[2];
  gf[1] -= 0.5 * gs[2];
  gf[n] += 0.5 * gs[n - 1];
  gf[n - 2] -= 0.5 * gs[n - 1];
  gf[n] += gs[n];
  gf[n - 1] -= gs[n];
  for (int m = 3; m <= n - 2; m++) {
    const double w = gs[m] / 12.0;
    gf[m - 2] += w;
    gf[m + 2] -= w;
    gf[m + 1] += 8.0 * w;
    gf[m - 1] -= 8.0 * w;
  }
  for (int m = 1; m <= n; m++) out[m - 1] = gf[m];
}

namespace {

// dL/dknots of every table from the sums over the pairs and atoms: G holds dL/df then
// dL/ds of every knot.  One thread per knot k (1-based) of its table: f[k] itself, and
// through the slopes s[m] of the knots m = k - 2 .. k + 2 (the transpose of
// spline_interpolate's slope map).
__global__ void k_spline_adjoint(int nel, int nz, int nrho, int nr, const double* __restrict__ G,
                                 double* __restrict__ grad)
{
  const int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int64_t kf = (int64_t)nel * nrho, knots = kf + (int64_t)(nel + nz) * nr;
  if (q >= knots) return;
  const int n = q < kf ? nrho : nr;
  const int64_t t0 = q < kf ? q / nrho * nrho : kf + (q - kf) / nr * nr;  // the table's first knot
  const int k = (int)(q - t0) + 1;
  const double* gs = G + knots + t0 - 1;  // slopes, 1-based
  double v = G[q];
  if (k == 2) v += gs[1];
  if (k == 1) v -= gs[1] + 0.5 * gs[2];
  if (k == 3) v += 0.5 * gs[2];
  if (k == n) v += 0.5 * gs[n - 1] + gs[n];
  if (k == n - 2) v -= 0.5 * gs[n - 1];
  if (k == n - 1) v -= gs[n];
  // interior slopes m in [3, n - 2]: f[m - 2] +w, f[m + 2] -w, f[m + 1] +8w, f[m - 1] -8w
  const auto interior = [&](int m) { return m >= 3 && m <= n - 2; };
  if (interior(k + 2)) v += gs[k + 2] / 12.0;
  if (interior(k - 2)) v -= gs[k - 2] / 12.0;
  if (interior(k - 1)) v += 8.0 * (gs[k - 1] / 12.0);
  if (interior(k + 1)) v -= 8.0 * (gs[k + 1] / 12.0);
  grad[q] = v;
}

}  // namespace

void eam_adjoint(Ctx& c, double rcut, const double* dLdF_id, const double* dLdE, double scale, double* grad,
                 bool mixed, bool device)
{
  EamHost& e = c.eam;
  const int nel = e.nel, nz = nel * (nel + 1) / 2;
  const size_t nknots = (size_t)nel * e.nrho + (size_t)(nel + nz) * e.nr;
  c.adj_g.reserve(2 * nknots);
  c.adj_gvec.reserve(c.npad);
  c.adj_drho.reserve(c.npad);
  c.adj_gE.reserve(c.nrep);
  if (!device) c.adj_grad.reserve(nknots);
  const double *gF = dLdF_id, *gE = dLdE;  // on the device
  if (!device) {
    c.adj_in.reserve(3 * (size_t)c.n + c.nrep);
    XS_HIP(hipMemcpyAsync(c.adj_in.p, dLdF_id, sizeof(double) * 3 * c.n, hipMemcpyHostToDevice, c.stream));
    XS_HIP(hipMemcpyAsync(c.adj_in.p + 3 * c.n, dLdE, sizeof(double) * c.nrep, hipMemcpyHostToDevice, c.stream));
    gF = c.adj_in.p;
    gE = c.adj_in.p + 3 * c.n;
  }
  if (c.n > 0) {
    k_gather_g<<<grid_for(std::max<int64_t>(c.n, c.nrep)), kBlock, 0, c.stream>>>(
        c.n, c.id.p, gF, c.adj_gvec.p, scale, gE, c.adj_gE.p, c.nrep);
    XS_HIP(hipGetLastError());
    const bool block = c.list_kind == ListKind::Block;
    AdjArgs a;
    a.n = c.n;
    a.npad = c.npad;
    a.pos = c.pos.p;
    a.gvec = c.adj_gvec.p;
    a.rho = c.rho.p;
    a.drho = c.adj_drho.p;
    a.type = c.type.p;
    a.rep = c.has_rep ? c.rep.p : nullptr;
    a.box = c.box_d.p;
    a.nbr = block ? nullptr : c.nbr.p;
    a.nbr16 = block ? c.nbr16.p : nullptr;
    a.stage = c.brick_stage.p;
    a.base = c.atom_stage.p;
    a.nnb = c.nnb.p;
    a.gE = c.adj_gE.p;
    a.rc2 = rcut * rcut;
    a.nel = nel;
    a.nr = e.nr;
    a.nrho = e.nrho;
    a.rdr = e.rdr;
    a.rdrho = e.rdrho;
    a.rhomax = e.rhomax;
    a.conv = kEV;
    a.types = c.eam_types;
    a.xf = c.xf_dev();
    ProfScope prof(c.prof, c.stream, XS_PROF_ADJOINT);
    adj_run(c, a, rcut, mixed);
  } else {
    XS_HIP(hipMemsetAsync(c.adj_g.p, 0, sizeof(double) * 2 * nknots, c.stream));
  }
  // dL/dtheta: the transpose of the knot -> slope map, on the device
  double* out = device ? grad : c.adj_grad.p;
  k_spline_adjoint<<<grid_for((int64_t)nknots), kBlock, 0, c.stream>>>(nel, nz, e.nrho, e.nr, c.adj_g.p, out);
  XS_HIP(hipGetLastError());
  if (!device) {
    XS_HIP(hipMemcpyAsync(grad, out, sizeof(double) * nknots, hipMemcpyDeviceToHost, c.stream));
    XS_HIP(hipStreamSynchronize(c.stream));
  }
}

void lj_adjoint(Ctx& c, double eps, double sigma, double rcut, const double* dLdF_id, const double* dLdE,
                double grad[2])
{
  ensure_global_list(c);
  const unsigned g = grid_for(c.n, kLjAdjThreads);
  c.adj_gvec.reserve(c.npad);
  c.adj_in.reserve(3 * (size_t)c.n + c.nrep);
  c.adj_part.reserve(2 * (size_t)std::max(g, 1u) + 2);
  XS_HIP(hipMemcpyAsync(c.adj_in.p, dLdF_id, sizeof(double) * 3 * c.n, hipMemcpyHostToDevice, c.stream));
  XS_HIP(hipMemcpyAsync(c.adj_in.p + 3 * c.n, dLdE, sizeof(double) * c.nrep, hipMemcpyHostToDevice, c.stream));
  double* out = c.adj_part.p + 2 * (size_t)std::max(g, 1u);
  if (c.n > 0) {
    k_gather_g<<<grid_for(c.n), kBlock, 0, c.stream>>>(c.n, c.id.p, c.adj_in.p, c.adj_gvec.p, 1.0, nullptr, nullptr, 0);
    XS_HIP(hipGetLastError());
    LjAdjArgs a;
    a.n = c.n;
    a.npad = c.npad;
    a.pos = c.pos.p;
    a.gvec = c.adj_gvec.p;
    a.rep = c.has_rep ? c.rep.p : nullptr;
    a.box = c.box_d.p;
    a.nbr = c.nbr.p;
    a.nnb = c.nnb.p;
    a.gE = c.adj_in.p + 3 * c.n;
    a.rc2 = rcut * rcut;
    a.eps = eps;
    a.sigma = sigma;
    a.sigma2 = sigma * sigma;
    a.xf = c.xf_dev();
    // the derivatives of energy_cutoff = e(rc) (pair_potential_impl.hxx:487-498)
    const double sc2 = a.sigma2 / a.rc2, sc6 = sc2 * sc2 * sc2, sc12 = sc6 * sc6;
    a.decut_eps = 4.0 * (sc12 - sc6);
    a.decut_sigma = 4.0 * eps * (12.0 * sc12 - 6.0 * sc6) / sigma;
    ProfScope prof(c.prof, c.stream, XS_PROF_ADJOINT);
    k_lj_adjoint<<<g, kLjAdjThreads, 0, c.stream>>>(a, c.adj_part.p);
    XS_HIP(hipGetLastError());
    k_lj_adjoint_reduce<<<1, kLjAdjThreads, 0, c.stream>>>(g, c.adj_part.p, out);
    XS_HIP(hipGetLastError());
    XS_HIP(hipMemcpyAsync(grad, out, 2 * sizeof(double), hipMemcpyDeviceToHost, c.stream));
  } else {
    grad[0] = grad[1] = 0.0;
  }
  XS_HIP(hipStreamSynchronize(c.stream));
}

}  // namespace xsmd
