// pair_math.hpp -- device arithmetic shared by the global-list kernels (k_pair.hip)
// and the cell-block kernels (k_block.hip): spline evaluation (eam_alloy.h:198-313),
// the EAM pair scalars (eam_alloy_mm_force), the per-atom output epilogue.
//
// Real is the type of the pair and spline arithmetic: double for the plain FP64
// form, float for the mixed form (FP64 displacement, d^2, cutoff test and all
// accumulations in either case).
#pragma once

#include "xsmd_internal.hpp"

namespace xsmd {
namespace pm {

template <class Real>
struct Q4 {
  Real a, b, c, d;
};

__device__ __forceinline__ Q4<float> load4(const float* __restrict__ p)
{
  const float4 v = *reinterpret_cast<const float4*>(p);
  return {v.x, v.y, v.z, v.w};
}
__device__ __forceinline__ Q4<double> load4(const double* __restrict__ p)
{
  const double2 u = reinterpret_cast<const double2*>(p)[0];
  const double2 w = reinterpret_cast<const double2*>(p)[1];
  return {u.x, u.y, w.x, w.y};
}

// Distance from its square, and the reciprocal distance, in FP64.  The compiler's square
// root and division scale for the ends of the exponent range and fix up special cases: 29
// instructions of the 79 per list entry of the FP64 force pass.  Squared distances need
// none of that, so both come from the hardware's reciprocal square root y (about 2^-23) by
// Goldschmidt's iteration: g -> sqrt, h -> 1 / (2 sqrt), then one residual step each,
// 12 instructions with the minimum.  On 8.4 M values from 0.01 to 1e12 r equals sqrt(d2) in every one and
// rinv is as far from the exact reciprocal as 1 / r (1.50 ulp at most, 0.36 on average);
// recip equals 1 / x.  For d2 = 0 (coincident atoms) the steps give NaN: the minimum makes
// rinv the infinity that the division gives, r stays NaN (knot_r takes it as 0).
__device__ __forceinline__ void dist_steps(double d2, double y, double& g, double& h)
{
  g = d2 * y;
  h = 0.5 * y;
  const double e = fma(-h, g, 0.5);
  g = fma(g, e, g);
  h = fma(h, e, h);
  g = fma(fma(-g, g, d2), h, g);
}
__device__ __forceinline__ void dist(double d2, double& r, double& rinv)
{
  double h;
  dist_steps(d2, __builtin_amdgcn_rsq(d2), r, h);
  const double y = h + h;
  rinv = fmin(fma(fma(-y, r, 1.0), y, y), HUGE_VAL);
}
// the distance alone; finite at d2 = 0 (1e-145, the table's first knot)
__device__ __forceinline__ double dist(double d2)
{
  double r, h;
  // the larger of the two by their upper halves (fmax first quiets NaNs, an instruction more)
  const unsigned long long b = (unsigned long long)__double_as_longlong(d2);
  const uint32_t hi = (uint32_t)max((int)(b >> 32), 0x03b90000);
  const double x = __longlong_as_double((long long)((unsigned long long)hi << 32 | (uint32_t)b));
  dist_steps(x, __builtin_amdgcn_rsq(x), r, h);
  return r;
}
__device__ __forceinline__ float recip(float x) { return __builtin_amdgcn_rcpf(x); }
// Newton's iteration on the hardware's reciprocal, without the division's scaling
__device__ __forceinline__ double recip(double x)
{
  double y = __builtin_amdgcn_rcp(x);
  y = fma(fma(-x, y, 1.0), y, y);
  return fma(fma(-x, y, 1.0), y, y);
}
__device__ __forceinline__ float fma_r(float a, float b, float c) { return fmaf(a, b, c); }
__device__ __forceinline__ double fma_r(double a, double b, double c) { return fma(a, b, c); }

// XCD-aware block order: hardware hands workgroup b to XCD b % 8, so map it to
// logical block (b % 8) * (G/8) + b / 8 and each XCD's L2 sees one contiguous
// (hence spatially compact) range of atoms.  G is padded to a multiple of 8.
__device__ __forceinline__ int64_t logical_block()
{
  const unsigned b = blockIdx.x, g = gridDim.x;
  return (int64_t)(b & 7u) * (g >> 3) + (b >> 3);
}

struct Outputs {
  double* ax;
  double* ay;
  double* az;
  double* ep;
  double* vir;
  const double* mass;  // fused epilogue
  const uint8_t* type;
  double* vx;
  double* vy;
  double* vz;
  double kick_dt;
  int64_t npad;
  bool set_ep;  // ep is written, not added to
};

// Per-atom epilogue: add the force (operator form) or write a = f/m and kick v
// (fused MD form); energy and virial when requested.
template <bool ENERGY, bool VIRIAL, bool FUSED>
__device__ __forceinline__ void write_outputs(const Outputs& o, int64_t i, double fx, double fy, double fz,
                                              double e, const double* v)
{
  if constexpr (FUSED) {
    const double m = o.mass[o.type[i]];
    const double a0 = fx / m, a1 = fy / m, a2 = fz / m;
    o.ax[i] = a0;
    o.ay[i] = a1;
    o.az[i] = a2;
    o.vx[i] = fma(a0, o.kick_dt, o.vx[i]);
    o.vy[i] = fma(a1, o.kick_dt, o.vy[i]);
    o.vz[i] = fma(a2, o.kick_dt, o.vz[i]);
  } else {
    o.ax[i] += fx;
    o.ay[i] += fy;
    o.az[i] += fz;
  }
  if constexpr (ENERGY) o.ep[i] = o.set_ep ? e : o.ep[i] + e;
  if constexpr (VIRIAL) {
#pragma unroll
    for (int q = 0; q < 9; q++) {
      if constexpr (FUSED) o.vir[q * o.npad + i] = v[q];
      else o.vir[q * o.npad + i] += v[q];
    }
  }
}

// Next-step drift fused into the MD-loop epilogue: the arithmetic of k_drift_kick
// applied to the velocity this step's kick produced.  The loop only needs to know
// whether some atom moved more than the rebuild threshold, so an atom past it raises
// the loop's flag (see StepGate).
struct Drift {
  Pos4* pos_out;
  const double* rrx;
  const double* rry;
  const double* rrz;
  double dt, dt2, hdt;
  double thr2;
  StepFlag over;
};

// Fused epilogue with drift: a = f/m, v += a*kick_dt (this step), then
// push_f_v_r(dt) and push_f_v(dt/2) of the next step from the record p of atom i,
// and the rebuild test on the displacement since the last list build.
__device__ __forceinline__ void write_outputs_drift(const Outputs& o, const Drift& d, int64_t i, const Pos4& p,
                                                    double fx, double fy, double fz)
{
  const double m = o.mass[o.type[i]];
  const double a0 = fx / m, a1 = fy / m, a2 = fz / m;
  o.ax[i] = a0;
  o.ay[i] = a1;
  o.az[i] = a2;
  const double v0 = fma(a0, o.kick_dt, o.vx[i]);
  const double v1 = fma(a1, o.kick_dt, o.vy[i]);
  const double v2 = fma(a2, o.kick_dt, o.vz[i]);
  Pos4 q = p;
  q.x += fma(v0, d.dt, a0 * d.dt2);
  q.y += fma(v1, d.dt, a1 * d.dt2);
  q.z += fma(v2, d.dt, a2 * d.dt2);
  q.w = 0.0;
  store_pos(d.pos_out, i, q);
  o.vx[i] = fma(a0, d.hdt, v0);
  o.vy[i] = fma(a1, d.hdt, v1);
  o.vz[i] = fma(a2, d.hdt, v2);
  if (xsmd_d2(q.x - d.rrx[i], q.y - d.rry[i], q.z - d.rrz[i]) > d.thr2) d.over.raise();
}

// onika tensor(fe, dr) * -0.5 added to v (row-major m11 m12 ... m33)
__device__ __forceinline__ void add_virial(double* v, double fe0, double fe1, double fe2, double dx, double dy,
                                           double dz)
{
  const double fe[3] = {fe0, fe1, fe2};
  const double dr[3] = {dx, dy, dz};
#pragma unroll
  for (int a = 0; a < 3; a++)
#pragma unroll
    for (int b = 0; b < 3; b++) v[3 * a + b] = fma(fe[a] * dr[b], -0.5, v[3 * a + b]);
}

template <class Real>
__device__ __forceinline__ void knot_r(const EamTabDev<Real>& t, Real r, int& m, Real& p)
{
  p = r * t.rdr + Real(1);
  m = max(1, min((int)p, t.nr - 1));  // NaN, the distance of coincident atoms, converts to 0
  p -= (Real)m;
  p = fmin(fmax(p, Real(0)), Real(1));  // one instruction's clamp, which takes NaN as 0
}

// Distance, 1/r and spline knot of a pair from its FP64 d^2 (the first steps of
// eam_alloy_rho_noderiv / eam_alloy_mm_force, eam_alloy.h:198-265: p = r rdr + 1,
// m = min(int p, nr - 1), p -= m, p = min(p, 1)).
// Mixed form: the knot fraction of r ~ 5 A at 1000 knots per A needs more than FP32
// (its ulp at p ~ 5000 is 5e-4 of a knot, which puts ~1e-5 of relative error on the
// forces of atoms whose pair forces nearly cancel), so 1/sqrt(d2) is the FP32
// hardware rsq refined by one FP64 Newton step (relative error ~1e-14), r and p are
// formed in FP64, and only the fraction (in [0, 1]) and 1/r are rounded to FP32 for
// the spline arithmetic.
__device__ __forceinline__ void knot_dist(const EamTabDev<double>& t, double d2, int& m, double& p, double& rinv)
{
  double r;
  dist(d2, r, rinv);
  knot_r(t, r, m, p);
}
// the knot alone
__device__ __forceinline__ void knot_dist(const EamTabDev<double>& t, double d2, int& m, double& p)
{
  knot_r(t, dist(d2), m, p);
}
__device__ __forceinline__ void knot_dist(const EamTabDev<float>& t, double d2, int& m, float& p, float& rinv)
{
  const double y0 = (double)__builtin_amdgcn_rsqf((float)d2);
  const double y = y0 * fma(-0.5 * d2 * y0, y0, 1.5);
  double q = fma(d2 * y, t.rdr_d, 1.0);
  m = min((int)q, t.nr - 1);
  q -= (double)m;
  p = (float)fmin(q, 1.0);
  rinv = (float)y;
}
__device__ __forceinline__ void knot_dist(const EamTabDev<float>& t, double d2, int& m, float& p)
{
  float rinv;
  knot_dist(t, d2, m, p, rinv);
}

// Element `i` of a table whose base is the same for every lane: the byte offset is
// formed in 32 bits (every table here is far below 4 GiB and its indices are
// non-negative), so the loads take the scalar-base form with one 32-bit offset per
// lane instead of 64-bit address arithmetic.
template <class T>
__device__ __forceinline__ const T* at32(const T* base, uint32_t i)
{
  return reinterpret_cast<const T*>(reinterpret_cast<const char*>(base) + (i * (uint32_t)sizeof(T)));
}

// A 32-byte row of a table, loaded together with the neighbouring lane's (lane ^ 1, which
// must be active and do the same): one load takes the two halves of the even lane's row,
// the next those of the odd lane's, and the halves change lanes in registers.  A lane's load
// of 16 bytes looks up the cache line of each row it touches; two loads of 64 scattered rows
// look up about 100 lines, two of 32 rows each, whole, little more than half, and the FP64
// passes are bound by those lookups (texture address and data units busy 80 % of the time).
// 500 k EAM atoms, FP64: lookups of the force pass 84 -> 48 million, 118 -> 102 us, density
// pass 65 -> 56.  The mixed force pass, whose rows are 32 bytes too, pays more for
// the exchange than it gains (8.39 M atoms: 1139 -> 1346 us).
__device__ __forceinline__ uint32_t dpp_xor1(uint32_t v)
{
  return (uint32_t)__builtin_amdgcn_mov_dpp((int)v, kDppXor1, 0xf, 0xf, true);
}
// the rows of a pair of lanes: byte offsets, within a table, of this lane's halves of the
// even and of the odd lane's row
struct RowPair {
  uint32_t even, odd;
  __device__ __forceinline__ explicit RowPair(uint32_t row)
  {
    const bool is_odd = threadIdx.x & 1;
    const uint32_t half = is_odd ? 16u : 0u, other = dpp_xor1(row);
    even = (is_odd ? other : row) << 5 | half;
    odd = (is_odd ? row : other) << 5 | half;
  }
};
__device__ __forceinline__ Q4<double> load_row(const double* base, const RowPair& r)
{
  const bool is_odd = threadIdx.x & 1;
  const uint4 e = *reinterpret_cast<const uint4*>(reinterpret_cast<const char*>(base) + r.even);
  const uint4 o = *reinterpret_cast<const uint4*>(reinterpret_cast<const char*>(base) + r.odd);
  // both lanes take part in the exchanges, so they come before the selections
  const uint4 xe = make_uint4(dpp_xor1(e.x), dpp_xor1(e.y), dpp_xor1(e.z), dpp_xor1(e.w));
  const uint4 xo = make_uint4(dpp_xor1(o.x), dpp_xor1(o.y), dpp_xor1(o.z), dpp_xor1(o.w));
  const uint4 lo = is_odd ? xo : e, hi = is_odd ? o : xe;
  return {__hiloint2double((int)lo.y, (int)lo.x), __hiloint2double((int)lo.w, (int)lo.z),
          __hiloint2double((int)hi.y, (int)hi.x), __hiloint2double((int)hi.w, (int)hi.z)};
}
// Row `row` of four values; PAIRED: with the neighbouring lane (FP64 rows)
template <bool PAIRED, class Real>
__device__ __forceinline__ Q4<Real> load_row(const Real* base, uint32_t row)
{
  if constexpr (PAIRED && sizeof(Real) == 8) return load_row(base, RowPair(row));
  else return load4(at32(base, row * 4u));
}

template <class Real>
__device__ __forceinline__ Real cubic(const Q4<Real>& c, Real p)
{
  return ((c.a * p + c.b) * p + c.c) * p + c.d;
}
template <class Real>
__device__ __forceinline__ Real quad(const Q4<Real>& c, Real p)
{
  return (c.a * p + c.b) * p + c.c;
}
// derivative of the value cubic with respect to p
template <class Real>
__device__ __forceinline__ Real dcubic(const Q4<Real>& c, Real p)
{
  return (Real(3) * c.a * p + Real(2) * c.b) * p + c.c;
}
// The FP32 forms spell out their fused multiply-adds, so every kernel that shares
// them (block and global lists) rounds them alike whatever the
// compiler's contraction choices around them.
__device__ __forceinline__ float cubic(const Q4<float>& c, float p) { return fmaf(fmaf(fmaf(c.a, p, c.b), p, c.c), p, c.d); }
__device__ __forceinline__ float quad(const Q4<float>& c, float p) { return fmaf(fmaf(c.a, p, c.b), p, c.c); }
__device__ __forceinline__ float dcubic(const Q4<float>& c, float p)
{
  return fmaf(fmaf(3.0f * c.a, p, 2.0f * c.b), p, c.c);
}

// types slot of eam_alloy_force (m_pair_enabled, eam_potential_multimat.cu:154-166):
// species `type` takes part when its bit is set; a pair counts when both species do,
// and an atom of a disabled species keeps rho = 0, F' = 0 and gets no force.
template <class Real>
__device__ __forceinline__ bool eam_on(const EamTabDev<Real>& t, int type)
{
  return (t.types >> type) & 1u;
}

// F(rho), F'(rho) in eV-converted internal units, with the linear extrapolation
// of F above rhomax (eam_alloy.h:289-313).
template <class Real>
__device__ __forceinline__ void embed(const EamTabDev<Real>& t, int ti, double rho, Real& F, Real& Fp)
{
  const Real rr = (Real)rho;
  Real p;
  if constexpr (sizeof(Real) == 4) p = fmaf(rr, t.rdrho, 1.0f);
  else p = rr * t.rdrho + Real(1);
  int m = (int)p;
  m = max(1, min(m, t.nrho - 1));
  p -= (Real)m;
  p = fmin(p, Real(1));
  const Real* row = t.frho + ((int64_t)t.t2frho[ti + 1] * (t.nrho + 1) + m) * 8;
  const Q4<Real> v = load4(row);
  const Q4<Real> dv = load4(row + 4);
  Fp = quad(dv, p);
  F = cubic(v, p);
  if (rr > t.rhomax) {
    if constexpr (sizeof(Real) == 4) F = fmaf(Fp, rr - t.rhomax, F);
    else F += Fp * (rr - t.rhomax);
  }
  F *= t.conv;
  Fp *= t.conv;
}

// Pair table: planes of (nr + 1) rows of 4 values, the value cubic [c3 c4 c5 c6] of knot
// m at row m; nel planes of rho, then the nel (nel + 1) / 2 planes of z2r (one of each
// for a single element).  Rows of 4 values keep 8 (FP32) or 4 (FP64) knots per 128-byte
// line, so the clustered knots that the lanes of a wave look up touch few lines; the
// derivative quadratics follow from the value cubics.
template <class Real>
__device__ __forceinline__ uint32_t row_index(const EamTabDev<Real>& t, int plane, int m)
{
  return (uint32_t)plane * (uint32_t)(t.nr + 1) + (uint32_t)m;
}
template <class Real>
__device__ __forceinline__ const Real* pair_row(const Real* __restrict__ pair, const EamTabDev<Real>& t, int plane,
                                                int m)
{
  return at32(pair, row_index(t, plane, m) * 4u);
}
// Planes of the pair of types ti, tj (type t is element t; initialize_types_table,
// eam_alloy.h:70-133): rho of each and their z2r, in arithmetic.  A type map is one more
// gather ahead of every row's, and rows that also hold the derivative quadratic cost four
// 32-byte gathers per pair instead of three: the alloy force pass of 130 k atoms (FP64,
// energy and virial) took 134 us with both, 80 us without (73 with rows loaded in pairs),
// the density pass 42 and 35 (32).  Types past the last element take the first planes.
__device__ __forceinline__ void pair_planes(int nel, int ti, int tj, int& rho_i, int& rho_j, int& z2r)
{
  const int hi = max(ti, tj), lo = min(ti, tj);
  const bool known = hi < nel;
  rho_i = known ? ti : 0;
  rho_j = known ? tj : 0;
  z2r = nel + (known ? ((hi * (hi + 1)) >> 1) + lo : 0);
}
template <class Real>
__device__ __forceinline__ const Real* pair_rho_row(const Real* __restrict__ pair, int m)
{
  return at32(pair, (uint32_t)m * 4u);
}
// Single-element psi'(r)/r and phi(r) from the two rows of knot m:
// rc = rho value cubic, zc = z2r value cubic; the derivative quadratics follow
// from the value cubics (times 1/dr).
template <class Real>
__device__ __forceinline__ void eam_pair_rows(const EamTabDev<Real>& t, const Q4<Real>& rc, const Q4<Real>& zc, Real p,
                                              Real rinv, Real fpi, Real fpj, Real& fpair, Real& phi)
{
  const Real rhop = dcubic(rc, p) * t.rdr;
  const Real z2p = dcubic(zc, p) * t.rdr;
  const Real z2 = cubic(zc, p);
  phi = z2 * rinv;
  Real phip, psip;
  if constexpr (sizeof(Real) == 4) {
    phip = fmaf(z2p, rinv, -(phi * rinv)) * t.conv;
    psip = fmaf(fpi + fpj, rhop, phip);
  } else {
    phip = (z2p * rinv - phi * rinv) * t.conv;
    psip = (fpi + fpj) * rhop + phip;
  }
  phi *= t.conv;
  fpair = psip * rinv;
}

// ---------------------------------------------------------------------------
// FP32 tables in s = r^2 (single element, mixed form, force pass)
// ---------------------------------------------------------------------------
// The mixed force pass of one element reads, instead of the knot rows, cubic pieces
// in s = r^2 over [s_lo, s_hi] = [(0.3 rmax)^2, rmax^2] (rmax = (nr - 1) dr), uniform
// in s: piece k covers [s_lo + k ds, s_lo + (k+1) ds] in the local coordinate
// p = (s - s_lo) / ds - k.  Each piece is the Hermite cubic through the reference
// spline's FP64 values and s-slopes at its two ends (value and slope continuous from
// piece to piece), of
//   force plane: rho'(r)/r | phi'(r) conv / r   [A B C 0 | A B C 0]: the s-derivative
//                quadratics times 2/ds, so (A p + B) p + C is the function itself
//   phi plane:   phi(r) conv = z2r(r) conv / r  [a b c d]  (energy)
// so a pair needs no square root and no division: its index comes from the FP64
// d^2 (p formed in FP64, rounded to FP32 in [0, 1]), and
// psi'(r)/r = (F'_i + F'_j) rho'(r)/r + phi'(r)/r is one FMA of two quadratics.
// The host takes the fewest pieces (256 .. 8192, doubling) whose FP32 evaluation stays
// within 8 FP32 ulps of the largest |rho'/r|, |phi'/r| and 4 of the largest |phi| of
// the FP64 spline over [s_lo, s_hi] (the FP32 knot rows are at about 1-4 of each), or
// no s-table (then every pair reads the knot rows).  A pair with d^2 outside
// [s_lo, s_hi] (closer than 0.3 rmax, or past the table's end) takes the knot rows:
// the reference evaluates r beyond rmax at the table's end, which the s-table cannot
// express.  An FP64 cubic in s could not reproduce the spline to FP64 precision, so
// the FP64 form keeps the knot rows; the density pass, a single cubic per pair, keeps
// them too (its FP32 s-table form measured no faster: the pass is bound by its
// gathers, which the s-table does not reduce).

// row and local coordinate of d^2 in the s-table; `out` = d^2 outside [s_lo, s_hi]
// (with no s-table the host sets a range no d^2 falls in, so every pair is `out`)
__device__ __forceinline__ void s_knot(const EamTabDev<float>& t, double d2, int& m, float& p, bool& out)
{
  const double x0 = fma(d2, t.s_rds, t.s_off);
  const double x = fmin(fmax(x0, 0.0), t.s_xmax);
  out = x != x0;
  m = min((int)x, t.sprows - 1);
  p = (float)(x - (double)m);
}

// the slope quadratic [A B C] of an s-table force row (its fourth value is padding)
struct Q3 {
  float a, b, c;
};
__device__ __forceinline__ Q3 load3(const float* __restrict__ p)
{
  const float3 v = *reinterpret_cast<const float3*>(p);
  return {v.x, v.y, v.z};
}
__device__ __forceinline__ float quad3(const Q3& c, float p) { return fmaf(fmaf(c.a, p, c.b), p, c.c); }

// The FP32 single-element form reads the s-table; every other form the knot rows.
template <class Real, bool MULTI>
constexpr bool kSTable = !MULTI && sizeof(Real) == 4;

// rho_{type_j}(r) contribution to atom i (SymRhoOp, eam_force_op_multimat.h:142-171)
// from the knot rows (single element: plane 0 of the pair table).  `in` false
// evaluates at d2 = 1 instead (a guard for list padding whose d2 may be 0); the value
// of a pair that does not count is arbitrary and callers mask it.  Callers whose d2 is
// always finite and positive pass true.
template <class Real, bool MULTI, bool PAIRED = false>
__device__ __forceinline__ Real eam_rho_knot(const EamTabDev<Real>& t, const Real* __restrict__ pair, int ti, int tj,
                                             double d2, bool in)
{
  Real p;
  int m;
  knot_dist(t, in ? d2 : 1.0, m, p);
  const int plane = MULTI && max(ti, tj) < t.nel ? tj : 0;
  return cubic(load_row<PAIRED>(pair, row_index(t, plane, m)), p);
}

// psi'(r)/r and phi(r) of eam_alloy_mm_force (eam_alloy.h:222-265) from the knot
// rows: psi' = F'_i rho'_j + F'_j rho'_i + phi', phi = z2r / r.
template <class Real, bool MULTI, bool PAIRED = false>
__device__ __forceinline__ void eam_pair_knot(const EamTabDev<Real>& t, const Real* __restrict__ pair, int ti, int tj,
                                              Real fpi, Real fpj, double d2, bool in, Real& fpair, Real& phi)
{
  Real p, rinv;
  int m;
  knot_dist(t, in ? d2 : 1.0, m, p, rinv);
  if constexpr (MULTI) {
    int pi, pj, pz;
    pair_planes(t.nel, ti, tj, pi, pj, pz);
    const Q4<Real> zc = load_row<PAIRED>(pair, row_index(t, pz, m));
    // FP32: derivative rows of their own; 1/dr and the cubic's coefficients each rounded
    // would add to the forces' error (2.27e-7 of their rms against 2.45e-7)
    Real rhoip, rhojp, z2p;
    if constexpr (sizeof(Real) == 4) {
      rhoip = quad(load4(pair_row(t.slope, t, pi, m)), p);
      rhojp = quad(load4(pair_row(t.slope, t, pj, m)), p);
      z2p = quad(load4(pair_row(t.slope, t, pz, m)), p);
    } else {
      rhoip = dcubic(load_row<PAIRED>(pair, row_index(t, pi, m)), p) * t.rdr;
      rhojp = dcubic(load_row<PAIRED>(pair, row_index(t, pj, m)), p) * t.rdr;
      z2p = dcubic(zc, p) * t.rdr;
    }
    const Real z2 = cubic(zc, p);
    phi = z2 * rinv;
    // half of phi' to each embedding term: the sum of the two is the same from either atom,
    // so the forces of a pair are opposite to the last bit
    const Real hp = fma_r(z2p, rinv, -(phi * rinv)) * (Real(0.5) * t.conv);
    const Real psip = fma_r(fpi, rhojp, hp) + fma_r(fpj, rhoip, hp);
    phi *= t.conv;
    fpair = psip * rinv;
  } else {
    const Real* z2r = pair + 4 * (t.nr + 1);  // the second plane, at the same offset
    if constexpr (PAIRED && sizeof(Real) == 8) {
      const RowPair r((uint32_t)m);
      eam_pair_rows(t, load_row(pair, r), load_row(z2r, r), p, rinv, fpi, fpj, fpair, phi);
    } else {
      eam_pair_rows(t, load4(at32(pair, (uint32_t)m * 4u)), load4(at32(z2r, (uint32_t)m * 4u)), p, rinv, fpi, fpj,
                    fpair, phi);
    }
  }
}

// Pair scalars psi'(r)/r (and, with PHI, phi(r)) of U pairs (nb[u].d2, nb[u].in,
// nb[u].w = F'_j; neighbour species tj[u]).  The s-table form evaluates all U from
// the s-table (their row loads in flight together: psi'/r = (F'_i + F'_j) rho'(r)/r +
// phi'(r)/r from the two slope quadratics of one 32-byte row) and flags slow[u] = a
// counted pair outside the s-table's range, which the caller evaluates with
// eam_pair_knot, only in the rare wave where some slow[u] is set.  Every other form
// reads the knot rows and leaves slow[] false.
template <class Real, bool MULTI, bool PHI, int U, class Nb>
__device__ __forceinline__ void eam_pair_batch(const EamTabDev<Real>& t, const Real* __restrict__ pair, int ti,
                                               const int (&tj)[U], Real fpi, const Nb (&nb)[U], Real (&fpair)[U],
                                               Real (&phi)[U], bool (&slow)[U])
{
  if constexpr (kSTable<Real, MULTI>) {
#pragma unroll
    for (int u = 0; u < U; u++) {
      int m;
      float p;
      bool out;
      s_knot(t, nb[u].d2, m, p, out);
      const Real* row = at32(pair + t.s_force, (uint32_t)m * 8u);
      const Q3 gr = load3(row), gz = load3(row + 4);
      fpair[u] = fmaf(fpi + (Real)nb[u].w, quad3(gr, p), quad3(gz, p));
      if constexpr (PHI) phi[u] = cubic(load4(at32(pair + t.s_phi, (uint32_t)m * 4u)), p);
      slow[u] = nb[u].in && out;
    }
  } else {
#pragma unroll
    for (int u = 0; u < U; u++) {
      eam_pair_knot<Real, MULTI>(t, pair, ti, tj[u], fpi, (Real)nb[u].w, nb[u].d2, nb[u].in, fpair[u], phi[u]);
      slow[u] = false;
    }
  }
}

// ---------------------------------------------------------------------------
// Analytic Johnson EAM (johnson.h:59-167), FP64
// ---------------------------------------------------------------------------
// Its functions of r are sums of screened exponentials t(x) = exp(-a (x - 1)) / (1 + (x - k)^20)
// of x = r / re (johnson.h:59-124); t and its x-derivative -t (a + 20 (x - k)^19 / (1 + (x - k)^20)).
// The power is five squarings and products (the general power function cost more than
// the two exponentials of a pair), and rho and the second term of phi share one t.
__device__ __forceinline__ void johnson_term(double a, double k, double x, double& t, double& dt)
{
  const double s = x - k, s2 = s * s, s4 = s2 * s2, s8 = s4 * s4;
  const double s19 = s8 * s8 * (s2 * s);
  const double inv = 1.0 / fma(s19, s, 1.0);
  t = exp(-a * (x - 1.0)) * inv;
  dt = -t * fma(20.0 * s19, inv, a);
}

// rho(r) at d2 = r^2
__device__ __forceinline__ double johnson_rho(const JohnsonParams& p, double d2)
{
  double t, dt;
  johnson_term(p.beta, p.lambda, dist(d2) / p.re, t, dt);
  return p.fe * t;
}

// (rho'(r) fsum + phi'(r)) / r and phi(r) at d2 = r^2, fsum = F'_i + F'_j
__device__ __forceinline__ void johnson_pair(const JohnsonParams& p, double d2, double fsum, double& de_r,
                                             double& phi)
{
  const double ire = 1.0 / p.re;
  double r, rinv;
  dist(d2, r, rinv);
  const double x = fmax(r, 0.0) * ire;  // coincident atoms: 0
  double t1, d1, t2, d2x;
  johnson_term(p.alpha, p.kappa, x, t1, d1);
  johnson_term(p.beta, p.lambda, x, t2, d2x);
  phi = p.A * t1 - p.B * t2;
  de_r = (fma(p.fe, fsum, -p.B) * d2x + p.A * d1) * ire * rinv;
}

// F(rho) and F'(rho) (johnson.h:131-167): cubic in rho / (0.85 rhoe) - 1 below
// 0.85 rhoe, cubic in rho / rhoe - 1 below 1.15 rhoe, Fo (1 - ln q^eta) q^eta above.
__device__ __forceinline__ void johnson_embed(const JohnsonParams& p, double rho, double& f, double& df)
{
  const double rhon = 0.85 * p.rhoe, rho0 = 1.15 * p.rhoe;
  const double irhoe = 1.0 / p.rhoe;
  if (rho < rhon) {
    const double t = rho / rhon - 1.0, t2 = t * t, t3 = t * t2;
    f = p.Fn0 + p.Fn1 * t + p.Fn2 * t2 + p.Fn3 * t3;
    df = (p.Fn1 + 2.0 * p.Fn2 * t + 3.0 * p.Fn3 * t2) * (1.0 / rhon);
  } else if (rho < rho0) {
    const double t = rho * irhoe - 1.0, t2 = t * t, t3 = t * t2;
    f = p.F0 + p.F1 * t + p.F2 * t2 + p.F3 * t3;
    df = (p.F1 + 2.0 * p.F2 * t + 3.0 * p.F3 * t2) * irhoe;
  } else {
    const double q = rho * irhoe;
    const double qe = pow(q, p.eta);
    const double lq = log(qe);
    f = p.Fo * (1.0 - lq) * qe;
    df = (-p.eta * qe + (1.0 - lq) * p.eta * qe) * (p.Fo * irhoe / q);
  }
}

// Lennard-Jones pair (lennard_jones.h:40-50, force_op_impl2.hxx:33-78) written in
// r^2 only: (sigma/r)^2 = sigma^2 / d2, de/r = -24 eps (2 s^12 - s^6) / d2, e shifted
// by E(rcut) (pair_potential_impl.hxx:487-498).  Pair math in Real, FP64 out.
template <class Real>
struct LJ {
  Real sigma2, eps4, eps24, ecut;
};

// lj_multi_force: parameters per unordered pair of species (packed triangle,
// entry b*(b+1)/2 + a for a <= b) and each pair's squared cutoff; a pair counts when
// r <= its rcut (pair_potential_force_op_multiparam.h:82-84), i.e. when d2 is at most the
// largest number whose square root is (the host's rcut2; below 0: no interaction).
struct LJMultiDev {
  const void* rows;          // LJ<Real> per type pair
  const double* __restrict__ rcut2;
  int npair;
};
__device__ __forceinline__ int type_pair(int a, int b)
{
  const int lo = min(a, b), hi = max(a, b);
  return hi * (hi + 1) / 2 + lo;
}
template <class Real>
__device__ __forceinline__ LJ<Real> lj_multi_row(const LJMultiDev& m, int pid)
{
  return reinterpret_cast<const LJ<Real>*>(m.rows)[pid];
}

template <class Real>
__device__ __forceinline__ void lj_pair(const LJ<Real>& lp, double d2, bool in, double& de_r, double& e)
{
  const Real ir2 = recip((Real)(in ? d2 : 1.0));
  const Real s2 = lp.sigma2 * ir2;
  const Real s6 = s2 * s2 * s2;
  const Real s12 = s6 * s6;
  // fused multiply-adds spelled out, so that every kernel rounds a pair alike
  de_r = in ? (double)(-lp.eps24 * fma_r(Real(2), s12, -s6) * ir2) : 0.0;
  e = in ? 0.5 * (double)fma_r(lp.eps4, s12 - s6, -lp.ecut) : 0.0;
}

}  // namespace pm

pm::Outputs make_outputs(Ctx& c, const ForceEpilogue& ep);

// device view of the lj_multi_force tables in the precision Real
template <class Real>
inline pm::LJMultiDev ljm_dev(const Ctx& c)
{
  pm::LJMultiDev m;
  if constexpr (sizeof(Real) == 4) m.rows = c.ljm_f.p;
  else m.rows = c.ljm_d.p;
  m.rcut2 = c.ljm_rcut2.p;
  m.npair = c.ljm_ntypes * (c.ljm_ntypes + 1) / 2;
  return m;
}

}  // namespace xsmd
