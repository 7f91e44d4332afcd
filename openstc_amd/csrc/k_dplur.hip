// DPLUR sweeps (DPLUR_inner_iteration, src/DPLURHPP.cuh:78-249, EPI_for_dqk
// src/FiniteRateChem.cu:255-284): one Jacobi sweep of the split implicit
// linearisation, din -> dout, and the per-cell scalars it gathers.
//
// Every cell takes from each of its six neighbours inside the block
//   +-1/2 (A_dir(q) d(q) +- rho_dir(q) d(q)),
// with the convective Jacobian A applied to the neighbour's increment d.  In a
// mixture one thread owns one cell and gathers the six terms from memory, with
// no barrier and 3-8 waves per SIMD to hide the loads behind (53-132 vector
// registers on the 9-species kernels; the variant that solves the reduced
// species block re-orders its rows through 9 KB of LDS a workgroup, 18 KB in
// FP64).  Air marches tiles through k instead (below).  A term is
// two multiply-adds a row once three numbers of the neighbour are known: the
// contravariant velocity, b1 = k.d(rho V) - U d(rho), and the pressure
// increment s(q) (b2 + b3 - b4 of the reference), which for a mixture needs
// the enthalpies of all species; it and the total enthalpy h are therefore
// formed once per cell by whoever writes d (s) or once per iteration (h) and
// gathered like any other field.
#include <algorithm>

#include "ostc_kernels.h"
#include "ostc_thermo.h"

namespace ostc {

namespace {

// Workgroup coordinates ordered for the caches: after the XCD remap, bands of
// `jb` workgroup rows, inside a band plane after plane.  The planes above and
// below a band's plane then pass through the same L2 within a few workgroups
// of each other (in row-major order over whole planes they are one plane,
// megabytes, apart).
__device__ __forceinline__ uint3 band_block(unsigned jb) {
  const unsigned gx = gridDim.x, gy = gridDim.y, gz = gridDim.z;
  const unsigned b = blockIdx.x + gx * (blockIdx.y + gy * blockIdx.z);
  unsigned r = xcd_remap(b, gx * gy * gz);
  const unsigned full = gy / jb, size = gx * jb * gz;
  unsigned band = r / size, width = jb;
  if (band >= full) {
    band = full;
    width = gy - full * jb;
  }
  r -= band * size;
  const unsigned plane = gx * width, k = r / plane;
  r -= k * plane;
  return make_uint3(r % gx, band * jb + r / gx, k);
}

// the pressure increment s of an increment d of a mixture (src/DPLURHPP.cuh:
// 127-191: b2 + b3 - b4) at speed |V| = vel; h0: the total enthalpy
template <typename R, int NS>
__device__ __forceinline__ R pressure_increment(const ostc_param *__restrict__ p, R u, R v, R w, R vel, R t,
                                                R gamma, const R *d, const R *y, R *h0) {
  const R e = (R)0.5 * vel * vel;
  R hk[NS];
  enthalpy<R>(t, hk, p, NS);
  R b3 = 0, b4 = 0, h = 0;
#pragma unroll
  for (int l = 0; l < NS; ++l) {
    b3 += t * r_over_mw<R>(p, l) * d[5 + l];
    b4 += hk[l] * d[5 + l];
    if (h0) h += y[l] * hk[l];
  }
  if (h0) *h0 = h + e;
  return (gamma - (R)1) * (e * d[0] - u * d[1] - v * d[2] - w * d[3] + d[4]) + gamma * b3 - (gamma - (R)1) * b4;
}

// h and s of the stored increment d (mixtures whose d was written by a kernel
// that does not form them)
template <typename R, int NS, bool H>
__global__ __launch_bounds__(256) void k_dplur_scalars(ZoneView<R> z, const ostc_param *__restrict__ p,
                                                       const R *__restrict__ din, R *__restrict__ s_out) {
  const uint3 b = xcd_block();
  const int i = (int)(b.x * 64 + threadIdx.x), j = (int)(b.y * 4 + threadIdx.y), k = (int)b.z;
  if (i >= z.mx || j >= z.my) return;
  const int64_t id = z.idx(i, j, k), P = z.plane;
  R d[5 + NS], y[NS], h0;
#pragma unroll
  for (int l = 0; l < 5 + NS; ++l) d[l] = din[l * P + id];
#pragma unroll
  for (int l = 0; l < NS; ++l) y[l] = H ? z.sv[l * P + id] : (R)0;
  s_out[id] = pressure_increment<R, NS>(p, z.bv[P + id], z.bv[2 * P + id], z.bv[3 * P + id], z.vel[id],
                                        z.bv[5 * P + id], z.gamma[id], d, y, H ? &h0 : nullptr);
  if (H) z.imp[id] = h0;
}

// One neighbour's term added to acc.  SIDE +1: the neighbour on the minus
// side, acc += 1/2 (A d + rho d); -1: on the plus side, acc -= 1/2 (A d - rho
// d).
template <typename R, int NS, int NT, int DIR, int SIDE>
__device__ __forceinline__ void gather(const ZoneView<R> &z, const R *__restrict__ din, const R *__restrict__ s_in,
                                       unsigned o, R *acc) {
  constexpr int NV = 5 + NS + NT;
  const int64_t P = z.plane;
  R d[NV];
#pragma unroll
  for (int l = 0; l < NV; ++l) d[l] = at(din + l * P, o);
  const R *m = z.metric + DIR * 3 * P;
  const R kx = at(m, o), ky = at(m + P, o), kz = at(m + 2 * P, o);
  const R u = at(z.bv + P, o), v = at(z.bv + 2 * P, o), w = at(z.bv + 3 * P, o);
  const R rad = at(z.spectr + DIR * P, o), h = at(z.imp, o), s = at(s_in, o);
  const R U = kx * u + ky * v + kz * w;
  constexpr R half = (R)(0.5 * SIDE);
  const R f = half * (U + (R)SIDE * rad), b1 = half * (kx * d[1] + ky * d[2] + kz * d[3] - U * d[0]), hs = half * s;
  acc[0] += f * d[0] + b1;
  acc[1] += f * d[1] + (u * b1 + kx * hs);
  acc[2] += f * d[2] + (v * b1 + ky * hs);
  acc[3] += f * d[3] + (w * b1 + kz * hs);
  acc[4] += f * d[4] + (h * b1 + U * hs);
#pragma unroll
  for (int l = 0; l < NS + NT; ++l) acc[5 + l] += f * d[5 + l] + at(z.sv + l * P, o) * b1;
}

// How a sweep treats the species rows of a mixture.
enum { ROWS_DIAGONAL = 0, ROWS_REDUCED, ROWS_SUMS, ROWS_DA };

// ROWS_REDUCED: EPI block of k_chem_dq0_red, solved here from its 48 numbers;
// ROWS_SUMS: the off-diagonal sums are left in dout for k_dplur_chem; ROWS_DA:
// the diagonal approximation.  s_out (mixtures, not ROWS_SUMS): the new
// increment's s, null in the last sweep.
template <typename R, int NS, int NT, int ROWS>
__global__ __launch_bounds__(256) void k_dplur(ZoneView<R> z, const ostc_param *__restrict__ p,
                                               const R *__restrict__ din, R *__restrict__ dout,
                                               const R *__restrict__ s_in, R *__restrict__ s_out, unsigned jb) {
  constexpr int NV = 5 + NS + NT;
  const uint3 b = band_block(jb);
  const int i = (int)(b.x * 64 + threadIdx.x), j = (int)(b.y * 4 + threadIdx.y), k = (int)b.z;
  if (i >= z.mx || j >= z.my) return;
  const int64_t P = z.plane, id = z.idx(i, j, k);
  const unsigned o = (unsigned)id * (unsigned)sizeof(R);
  const unsigned sj = (unsigned)z.nx * (unsigned)sizeof(R), sk = sj * (unsigned)z.ny;
  R acc[NV];
#pragma unroll
  for (int l = 0; l < NV; ++l) acc[l] = 0;
  // in the reference's order
  if (i > 0) gather<R, NS, NT, 0, 1>(z, din, s_in, o - (unsigned)sizeof(R), acc);
  if (j > 0) gather<R, NS, NT, 1, 1>(z, din, s_in, o - sj, acc);
  if (k > 0) gather<R, NS, NT, 2, 1>(z, din, s_in, o - sk, acc);
  if (i + 1 < z.mx) gather<R, NS, NT, 0, -1>(z, din, s_in, o + (unsigned)sizeof(R), acc);
  if (j + 1 < z.my) gather<R, NS, NT, 1, -1>(z, din, s_in, o + sj, acc);
  if (k + 1 < z.mz) gather<R, NS, NT, 2, -1>(z, din, s_in, o + sk, acc);
  // diagonal solve (src/DPLURHPP.cuh:193-249)
  const R dt = at(z.dt, o);
  const R diag = (R)1 + dt * (at(z.spectr, o) + at(z.spectr + P, o) + at(z.spectr + 2 * P, o));
  const R dti = dt / diag;
  R d[NV];
#pragma unroll
  for (int l = 0; l < 5; ++l) d[l] = at(z.dq0 + l * P, o) + dti * acc[l];
  if constexpr (NT > 0) {
    R t0 = dti, t1 = dti;
    if (p->turb_implicit == 1) {
      t0 = dt / (diag - dt * at(z.turb_jac, o));
      t1 = dt / (diag - dt * at(z.turb_jac + P, o));
    }
    d[5 + NS] = at(z.dq0 + (5 + NS) * P, o) + t0 * acc[5 + NS];
    d[6 + NS] = at(z.dq0 + (6 + NS) * P, o) + t1 * acc[6 + NS];
  }
  if constexpr (ROWS == ROWS_DIAGONAL) {
#pragma unroll
    for (int l = 5; l < 5 + NS; ++l) d[l] = at(z.dq0 + l * P, o) + dti * acc[l];
  } else if constexpr (ROWS == ROWS_DA) {
#pragma unroll
    for (int l = 5; l < 5 + NS; ++l)
      d[l] = (R)((double)at(z.dq0 + l * P, o) +
                 (double)dt * (double)acc[l] / ((double)diag - (double)dt * z.chem_jac[(l - 5) * P + id]));
  } else {
#pragma unroll
    for (int l = 5; l < 5 + NS; ++l) d[l] = acc[l];
  }
#pragma unroll
  for (int l = 0; l < NV; ++l)
    if (ROWS != ROWS_REDUCED || l < 5 || l >= 5 + NS) put(dout + l * P, o, d[l]);
  if constexpr (ROWS == ROWS_REDUCED) {
    static_assert(NS == kRedSpec, "the reduced tables are for 9 species");
    constexpr int K = kRedKept;
    const ChemRed *ct = chem_red(p);
    double a[K * K], cc[K * kRedDep], x[kRedSlots];
    int piv[K];
    const double *tile = z.chem_lu + (id & ~(int64_t)63) * kRedFactors + (id & 63);
#pragma unroll
    for (int q = 0; q < K * K; ++q) a[q] = tile[q * 64];
#pragma unroll
    for (int q = 0; q < K * kRedDep; ++q) cc[q] = tile[(K * K + q) * 64];
    const unsigned pw = (unsigned)z.chem_piv[id];
#pragma unroll
    for (int q = 0; q < K; ++q) piv[q] = (int)(pw >> (4 * q) & 15u);
    const double dtd = (double)dt, dinv = 1.0 / (double)diag;
    // species order <-> slot order (run-time numbers) through this thread's
    // column of LDS
    constexpr int T = 256;
    __shared__ R row[kRedSpec * T];
    R *mine = row + threadIdx.x + 64 * threadIdx.y;
#pragma unroll
    for (int l = 0; l < NS; ++l) mine[l * T] = acc[5 + l];
#pragma unroll
    for (int m = 0; m < kRedSlots; ++m) x[m] = (double)mine[ct->slot[m] * T] * dtd;
    const double rest = (double)mine[ct->slot[kRedSlots] * T] * dtd * dinv;
    chem_red_solve(ct, a, cc, piv, dinv, x);
#pragma unroll
    for (int m = 0; m < kRedSlots; ++m) mine[ct->slot[m] * T] = (R)((double)at(z.dq0 + (5 + ct->slot[m]) * P, o) + x[m]);
    mine[ct->slot[kRedSlots] * T] = (R)((double)at(z.dq0 + (5 + ct->slot[kRedSlots]) * P, o) + rest);
#pragma unroll
    for (int l = 0; l < NS; ++l) {
      d[5 + l] = mine[l * T];
      put(dout + (5 + l) * P, o, d[5 + l]);
    }
  }
  if constexpr (ROWS != ROWS_SUMS) {
    if (s_out)
      put(s_out, o, pressure_increment<R, NS>(p, at(z.bv + P, o), at(z.bv + 2 * P, o), at(z.bv + 3 * P, o),
                                              at(z.vel, o), at(z.bv + 5 * P, o), at(z.gamma, o), d,
                                              (const R *)nullptr, (R *)nullptr));
  }
}

// Chemistry block of one DPLUR sweep of a reacting zone with EPI
// (EPI_for_dqk, src/FiniteRateChem.cu:255-284) where the mechanism has no
// reduced tables: the sweep kernel leaves the species rows' off-diagonal sums
// in dout; each cell solves its block with the LU factors k_dq0 kept,
// dout_s = dq0_s + (diag I - dt J)^-1 (dt acc_s), in place.
template <typename R, int NS, int NA, bool TILED = false>
__global__ __launch_bounds__(256) void k_dplur_chem(ZoneView<R> z, const ostc_param *__restrict__ p,
                                                    R *__restrict__ dout) {
  const uint3 b3 = xcd_block();
  const int i = (int)(b3.x * 64 + threadIdx.x), j = (int)(b3.y * 4 + threadIdx.y), k = (int)b3.z;
  if (i >= z.mx || j >= z.my) return;
  const int64_t id = z.idx(i, j, k), P = z.plane;
  const ChemF64 *ct = chem64(p);
  const R dt = z.dt[id];
  const double dtd = (double)dt;
  double a[NA * NA], b[NA];
  int piv[NA];
  unsigned w[PivPack<NA>::words];
#pragma unroll
  for (int q = 0; q < NA * NA; ++q) a[q] = z.chem_lu[TILED ? lu_tiled(id, q, NA * NA) : q * P + id];
#pragma unroll
  for (int q = 0; q < PivPack<NA>::words; ++q) w[q] = (unsigned)z.chem_piv[q * P + id];
  piv_unpack<NA>(w, piv);
#pragma unroll
  for (int r = 0; r < NA; ++r) b[r] = (double)dout[(5 + block_species<NS, NA>(ct, r)) * P + id] * dtd;
  lu_solve_any<NA>(a, piv, b);
#pragma unroll
  for (int r = 0; r < NA; ++r) {
    const int m = block_species<NS, NA>(ct, r);
    dout[(5 + m) * P + id] = (R)((double)z.dq0[(5 + m) * P + id] + b[r]);
  }
  if constexpr (NA < NS) {
    // species that react in no reaction: their block row is diag, as k_dq0
    // formed it
    const double dg = (double)((R)1 + dt * (z.spectr[id] + z.spectr[P + id] + z.spectr[2 * P + id]));
    for (int m = 0; m < NS; ++m)
      if (ct->rank[m] < 0)
        dout[(5 + m) * P + id] = (R)((double)z.dq0[(5 + m) * P + id] + (double)dout[(5 + m) * P + id] * dtd / dg);
  }
}

// ------------------------------------------------------------------ air

// Per-cell inputs of the convective-Jacobian products of one DPLUR sweep
// (the neighbour part of src/DPLURHPP.cuh:127-191), loaded once per cell.
template <typename R, int NT>
struct JdCell {
  static constexpr int NV = 5 + NT;
  R d[NV];
  R sv[NT > 0 ? NT : 1];
  R u, v, w, e, h, s;
  R dt, diag, tj0, tj1;  // first sweep only: the cell's dq0 scaling
};

// compute_DQ_0's diagonal scaling without a chemistry block
// (src/DPLURHPP.cuh:13-76, SST rows src/SST.cu:196-204): d = dq / diag, the
// same operations k_dq0 performs.  The first sweep of a non-reacting zone
// applies it to every dq it loads instead of reading a stored dq0, and keeps
// dt, diag and the SST Jacobian diagonal for the cell's own diagonal solve.
template <typename R, int NT>
__device__ __forceinline__ void dq0_scale(const ZoneView<R> &z, const ostc_param *__restrict__ p, int64_t q,
                                          JdCell<R, NT> &c) {
  const int64_t P = z.plane;
  c.dt = z.dt[q];
  c.diag = (R)1 + c.dt * (z.spectr[q] + z.spectr[P + q] + z.spectr[2 * P + q]);
  c.tj0 = c.tj1 = 0;
#pragma unroll
  for (int l = 0; l < 5; ++l) c.d[l] = c.d[l] / c.diag;
  if constexpr (NT > 0) {
    if (p->turb_implicit == 1) {
      c.tj0 = z.turb_jac[q];
      c.tj1 = z.turb_jac[P + q];
      c.d[5] = c.d[5] / (c.diag - c.dt * c.tj0);
      c.d[6] = c.d[6] / (c.diag - c.dt * c.tj1);
    } else {
      c.d[5] = c.d[5] / c.diag;
      c.d[6] = c.d[6] / c.diag;
    }
  }
}

// FIRST: din is the right-hand side dq, scaled to dq0 on load
template <typename R, int NT, bool FIRST>
__device__ __forceinline__ void jd_load(const ZoneView<R> &z, const ostc_param *__restrict__ p,
                                        const R *__restrict__ din, int64_t q, JdCell<R, NT> &c) {
  constexpr int NV = 5 + NT;
  const int64_t P = z.plane;
#pragma unroll
  for (int l = 0; l < NV; ++l) c.d[l] = din[l * P + q];
  if constexpr (FIRST) dq0_scale<R, NT>(z, p, q, c);
#pragma unroll
  for (int l = 0; l < NT; ++l) c.sv[l] = z.sv[l * P + q];
  c.u = z.bv[P + q];
  c.v = z.bv[2 * P + q];
  c.w = z.bv[3 * P + q];
  const R vel = z.vel[q];
  c.e = (R)0.5 * vel * vel;
  const R gamma = (R)kGammaAir;
  c.h = gamma / (gamma - (R)1) * z.bv[4 * P + q] / z.bv[q] + c.e;
  c.s = (gamma - (R)1) * (c.e * c.d[0] - c.u * c.d[1] - c.v * c.d[2] - c.w * c.d[3] + c.d[4]);
}

// Contribution of cell q, seen as a neighbour across direction `dir`:
// w * (A_dir(q) dq(q) + pm_sr dq(q)); out = 0.5 * (JD + sr*d) (sign +1, the
// minus-side neighbour) or 0.5 * (JD - sr*d) (sign -1, the plus-side one).
template <typename R, int NT>
__device__ __forceinline__ void jd_dir(const ZoneView<R> &z, int64_t q, int dir, const JdCell<R, NT> &c,
                                       R sr, R *plus, R *minus) {
  constexpr int NV = 5 + NT;
  const int64_t P = z.plane;
  const R xi_x = z.metric[(dir * 3) * P + q], xi_y = z.metric[(dir * 3 + 1) * P + q],
          xi_z = z.metric[(dir * 3 + 2) * P + q];
  const R U = xi_x * c.u + xi_y * c.v + xi_z * c.w;
  const R b1 = xi_x * c.d[1] + xi_y * c.d[2] + xi_z * c.d[3] - U * c.d[0];
  R jd[NV];
  jd[0] = b1 + U * c.d[0];
  jd[1] = c.u * b1 + xi_x * c.s + U * c.d[1];
  jd[2] = c.v * b1 + xi_y * c.s + U * c.d[2];
  jd[3] = c.w * b1 + xi_z * c.s + U * c.d[3];
  jd[4] = c.h * b1 + U * c.s + U * c.d[4];
#pragma unroll
  for (int l = 0; l < NT; ++l) jd[5 + l] = U * c.d[5 + l] + c.sv[l] * b1;
#pragma unroll
  for (int l = 0; l < NV; ++l) {
    if (plus) plus[l] = (R)0.5 * (jd[l] + sr * c.d[l]);
    if (minus) minus[l] = (R)0.5 * (jd[l] - sr * c.d[l]);
  }
}

// Diagonal solve and write of one cell after a sweep has gathered its
// off-diagonal sum acc (src/DPLURHPP.cuh:193-249).  FIRST: the cell's dq0
// comes in dq0v[0..NV) and is stored for the later sweeps; dq0v[NV],
// dq0v[NV+1] hold its SST Jacobian diagonal.
template <typename R, int NT, bool FIRST>
__device__ __forceinline__ void dplur_finish(const ZoneView<R> &z, const ostc_param *__restrict__ p, int64_t id,
                                             const R *acc, R dt, R diag, R *__restrict__ dout, const R *dq0v) {
  const int64_t P = z.plane;
  auto q0 = [&](int l) -> R {
    if constexpr (FIRST) {
      z.dq0[l * P + id] = dq0v[l];
      return dq0v[l];
    } else {
      return z.dq0[l * P + id];
    }
  };
  const R dti = dt / diag;
#pragma unroll
  for (int l = 0; l < 5; ++l) dout[l * P + id] = q0(l) + dti * acc[l];
  if constexpr (NT > 0) {
    R t0 = dti, t1 = dti;
    if (p->turb_implicit == 1) {
      t0 = dt / (diag - dt * (FIRST ? dq0v[5 + NT] : z.turb_jac[id]));
      t1 = dt / (diag - dt * (FIRST ? dq0v[6 + NT] : z.turb_jac[P + id]));
    }
    dout[5 * P + id] = q0(5) + t0 * acc[5];
    dout[6 * P + id] = q0(6) + t1 * acc[6];
  }
}

// The sweep of air (no species).  A workgroup owns a 64 x 4 (i, j) tile and marches through a chunk of
// k planes: each cell's Jacobian products are formed once per direction and
// handed to its neighbours -- along i by lane shuffles inside the wave (one
// wave = one i row), along j through LDS, along k in registers from the
// previous plane.  Tile-edge neighbours outside the tile: the rows above and
// below by the edge rows themselves (whole-wave loads); the cells left and
// right of every row by 2*TJ lanes of an inner row's wave in one pass, handed
// over through LDS (single-lane halo loads per row would double the tile's vector
// memory instructions, which bound this kernel).  Off-diagonal sums are
// accumulated in the reference's order (i-, j-, k-, i+, j+, k+).  FIRST
// (first sweep): din is the right-hand side dq, scaled
// to dq0 as it is loaded, and each cell's dq0 is stored for the later sweeps
// (no separate dq0 pass).
template <typename R, int NT, int TJ, bool FIRST>
__global__ __launch_bounds__(64 * TJ) void k_dplur_air(ZoneView<R> z, const ostc_param *__restrict__ p,
                                               const R *__restrict__ din, R *__restrict__ dout, int kc) {
  constexpr int NV = 5 + NT;
  __shared__ R sj[2][TJ][NV][64];  // [plus/minus][row][var][lane]
  __shared__ R si[2][TJ][NV];      // [left P_i / right M_i][row][var]
  const int tx = threadIdx.x, ty = threadIdx.y;
  const uint3 bk = xcd_block();
  const int i = (int)bk.x * 64 + tx, j = (int)bk.y * TJ + ty;
  const int k0 = (int)bk.z * kc, k1 = min(k0 + kc, z.mz);
  const bool ok = i < z.mx && j < z.my;
  const int ii = min(i, z.mx - 1), jj = min(j, z.my - 1);  // clamped (loads of idle lanes stay in bounds)
  const int64_t P = z.plane;
  const int64_t sk = (int64_t)z.nx * z.ny;
  const R *sr = z.spectr;
  JdCell<R, NT> c;
  R pk[NV], acc[NV], accp[NV];
  R dq0p[FIRST ? NV + 2 : 1];  // FIRST: dq0 (+ SST diagonal) of the cell below, finished with the next plane
  R dtp = 0, diagp = 1;
  // P_k of the plane below the chunk
  if (k0 > 0) {
    const int64_t q = z.idx(ii, jj, k0 - 1);
    jd_load<R, NT, FIRST>(z, p, din, q, c);
    jd_dir<R, NT>(z, q, 2, c, sr[2 * P + q], pk, nullptr);
  }
  for (int k = k0; k < k1; ++k) {
    const int64_t id = z.idx(ii, jj, k);
    jd_load<R, NT, FIRST>(z, p, din, id, c);
    R mk[NV], pnext[NV];
    jd_dir<R, NT>(z, id, 2, c, sr[2 * P + id], pnext, mk);
    // finish the cell below: its plus-side k neighbour is this cell
    if (k > k0) {
#pragma unroll
      for (int l = 0; l < NV; ++l) accp[l] -= mk[l];
      if (ok) dplur_finish<R, NT, FIRST>(z, p, id - sk, accp, dtp, diagp, dout, dq0p);
    }
    // minus-side terms in the reference order: i-, j-, k-
    R pi[NV], mi[NV];
    jd_dir<R, NT>(z, id, 0, c, sr[id], pi, mi);
    R pj[NV], mj[NV];
    jd_dir<R, NT>(z, id, 1, c, sr[P + id], pj, mj);
    __syncthreads();  // previous plane's j exchange is consumed
#pragma unroll
    for (int l = 0; l < NV; ++l) {
      sj[0][ty][l][tx] = pj[l];
      sj[1][ty][l][tx] = mj[l];
    }
    // i: neighbours' P_i / M_i from the adjacent lanes
    R ip[NV], im[NV];
#pragma unroll
    for (int l = 0; l < NV; ++l) {
      ip[l] = lane_prev(pi[l]);
      im[l] = lane_next(mi[l]);
    }
    if (ty == (TJ > 2 ? 1 : 0) && tx < 2 * TJ) {
      // lane 2r: the cell left of row r's segment (its P_i); lane 2r+1: the
      // cell right of it (its M_i).  An inner row does this (rows 0 and TJ-1
      // also evaluate the rows outside the tile), so that no wave carries
      // more than two cells' loads per plane.
      const int r = tx >> 1, side = tx & 1;
      const int ih = side ? (int)bk.x * 64 + 64 : (int)bk.x * 64 - 1;
      const int jr = min((int)bk.y * TJ + r, z.my - 1);
      if (ih >= 0 && ih < z.mx) {
        const int64_t q = z.idx(ih, jr, k);
        JdCell<R, NT> e;
        R hp[NV], hm[NV];
        jd_load<R, NT, FIRST>(z, p, din, q, e);
        jd_dir<R, NT>(z, q, 0, e, sr[q], hp, hm);
#pragma unroll
        for (int l = 0; l < NV; ++l) si[side][r][l] = side ? hm[l] : hp[l];
      }
    }
    // j: rows at the tile edge evaluate the neighbour row themselves
    R jp[NV], jm[NV];
    if (ty == 0 && j > 0) {
      const int64_t q = z.idx(ii, j - 1, k);
      JdCell<R, NT> e;
      jd_load<R, NT, FIRST>(z, p, din, q, e);
      jd_dir<R, NT>(z, q, 1, e, sr[P + q], jp, nullptr);
    }
    if (ty == TJ - 1 && j + 1 < z.my) {
      const int64_t q = z.idx(ii, j + 1, k);
      JdCell<R, NT> e;
      jd_load<R, NT, FIRST>(z, p, din, q, e);
      jd_dir<R, NT>(z, q, 1, e, sr[P + q], nullptr, jm);
    }
    __syncthreads();
    if (tx == 0 && i > 0 && i - 1 < z.mx)
#pragma unroll
      for (int l = 0; l < NV; ++l) ip[l] = si[0][ty][l];
    if (tx == 63 && i + 1 < z.mx)
#pragma unroll
      for (int l = 0; l < NV; ++l) im[l] = si[1][ty][l];
    if (ty > 0)
#pragma unroll
      for (int l = 0; l < NV; ++l) jp[l] = sj[0][ty - 1][l][tx];
    if (ty < TJ - 1)
#pragma unroll
      for (int l = 0; l < NV; ++l) jm[l] = sj[1][ty + 1][l][tx];
    const bool hi = i > 0, hj = j > 0, hk = k > 0;
    const bool lo_i = i + 1 < z.mx, lo_j = j + 1 < z.my;
#pragma unroll
    for (int l = 0; l < NV; ++l) {
      R a = 0;
      if (hi) a += ip[l];
      if (hj) a += jp[l];
      if (hk) a += pk[l];
      if (lo_i) a -= im[l];
      if (lo_j) a -= jm[l];
      acc[l] = a;
    }
    // this plane's plus-side k term arrives with the next plane
#pragma unroll
    for (int l = 0; l < NV; ++l) {
      accp[l] = acc[l];
      pk[l] = pnext[l];
    }
    if constexpr (FIRST) {
      dtp = c.dt;
      diagp = c.diag;
#pragma unroll
      for (int l = 0; l < NV; ++l) dq0p[l] = c.d[l];
      dq0p[NV] = c.tj0;
      dq0p[NV + 1] = c.tj1;
    } else {
      dtp = z.dt[id];
      diagp = (R)1 + dtp * (sr[id] + sr[P + id] + sr[2 * P + id]);
    }
  }
  // last plane of the chunk: plus-side k neighbour from the plane above
  if (k1 > k0) {
    const int kl = k1 - 1;
    if (k1 < z.mz) {
      const int64_t q = z.idx(ii, jj, k1);
      jd_load<R, NT, FIRST>(z, p, din, q, c);
      R mk[NV];
      jd_dir<R, NT>(z, q, 2, c, sr[2 * P + q], nullptr, mk);
#pragma unroll
      for (int l = 0; l < NV; ++l) accp[l] -= mk[l];
    }
    if (ok) dplur_finish<R, NT, FIRST>(z, p, z.idx(ii, jj, kl), accp, dtp, diagp, dout, dq0p);
  }
}

// Workgroups of a DPLUR sweep kernel resident on the whole current device at
// once (registers and LDS decide it), cached per device.
template <typename R, int NT, int TJ, bool FIRST>
int dplur_resident() {
  static int cached[64] = {};
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 0;
  if (cached[dev] > 0) return cached[dev];
  int per_cu = 0, cus = 0;
  if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, k_dplur_air<R, NT, TJ, FIRST>, 64 * TJ, 0) !=
          hipSuccess ||
      hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess)
    return 0;
  cached[dev] = per_cu * cus;
  return cached[dev];
}

// Planes per k chunk of a sweep over `tiles` (i, j) tiles.  The chunks run in
// rounds of `resident` workgroups and a round lasts one chunk's march and the
// two boundary planes it evaluates besides (about 1.5 plane steps), so the
// sweep takes about rounds x (planes per chunk + 1.5) steps: the count
// minimising that is taken (ties: fewer chunks).  resident <= 0 (unknown)
// counts as 1024.
inline int dplur_chunk_planes(int tiles, int mz, int resident) {
  if (resident <= 0) resident = 1024;
  int best = mz;
  long long best_cost = -1;
  for (int n = 1; n <= mz; ++n) {
    const int kc = (mz + n - 1) / n;
    const long long chunks = (mz + kc - 1) / kc;
    const long long rounds = ((long long)tiles * chunks + resident - 1) / resident;
    const long long cost = rounds * (2 * kc + 3);
    if (best_cost < 0 || cost < best_cost) {
      best_cost = cost;
      best = kc;
    }
  }
  return best;
}

inline int last_err() { return hipGetLastError() == hipSuccess ? OSTC_OK : OSTC_ERR_HIP; }

// the EPI block solve of a mechanism without reduced tables
template <typename R, int NS>
int chem_solve(const ZoneView<R> &z, const ostc_param *dp, const CellOpts &o, bool tiled, R *out, hipStream_t st) {
  const auto g = cell_grid(z.mx, z.my, z.mz);
  if constexpr (NS == 9) {
    if (tiled)
      OSTC_DISPATCH_NA(o, hipLaunchKernelGGL((k_dplur_chem<R, 9, NA_, true>), g.grid, g.block, 0, st, z, dp, out));
    else
      OSTC_DISPATCH_NA(o, hipLaunchKernelGGL((k_dplur_chem<R, 9, NA_>), g.grid, g.block, 0, st, z, dp, out));
  } else {
    hipLaunchKernelGGL((k_dplur_chem<R, 20, 20>), g.grid, g.block, 0, st, z, dp, out);
  }
  return last_err();
}

// air: dq -> dq0 and the first increment in one sweep, then dqk -> dq -> dqk
template <typename R, int NT>
int sweeps_air(const ZoneView<R> &z, const ostc_param *dp, const CellOpts &o, hipStream_t st, R **result) {
  constexpr int tj = 4;
  const int tiles = ((z.mx + 63) / 64) * ((z.my + tj - 1) / tj);
  const int kc = dplur_chunk_planes(tiles, z.mz, o.dplur_wg > 0 ? o.dplur_wg : dplur_resident<R, NT, tj, false>());
  const dim3 grid((unsigned)((z.mx + 63) / 64), (unsigned)((z.my + tj - 1) / tj), (unsigned)((z.mz + kc - 1) / kc));
  const dim3 block(64, tj, 1);
  R *in = z.dq, *out = z.dqk;
  for (int q = 0; q < o.dplur_steps; ++q) {
    const int stage = q == 0 ? P_DPLUR_FIRST : P_DPLUR;
    prof_mark(stage, st, true);
    if (q == 0)
      hipLaunchKernelGGL((k_dplur_air<R, NT, tj, true>), grid, block, 0, st, z, dp, (const R *)in, out, kc);
    else
      hipLaunchKernelGGL((k_dplur_air<R, NT, tj, false>), grid, block, 0, st, z, dp, (const R *)in, out, kc);
    prof_mark(stage, st, false);
    if (last_err()) return OSTC_ERR_HIP;
    in = out;
    out = (out == z.dqk) ? z.dq : z.dqk;
  }
  *result = in;
  return OSTC_OK;
}

// mixtures: dq0 stays, dqk and dq take the increments in turn
template <typename R, int NS, int NT>
int sweeps(const ZoneView<R> &z, const ostc_param *dp, const CellOpts &o, hipStream_t st, bool chem_late,
           R **result) {
  const bool chem = o.mix_model == OSTC_FR, epi = chem && o.chem == 1;
  const bool reduced = epi && chem_late && o.red;
  const auto g = cell_grid(z.mx, z.my, z.mz);
  // bands of about 24 workgroups a plane
  const unsigned jb = std::max(1u, 24u / g.grid.x);
  R *in = z.dq0, *out = z.dqk;
  R *s_in = z.imp + z.plane, *s_out = s_in + z.plane;
  for (int q = 0; q < o.dplur_steps; ++q) {
    const bool last = q + 1 == o.dplur_steps;
    R *so = last ? nullptr : s_out;
    prof_mark(P_DPLUR, st, true);
#define OSTC_SWEEP(ROWS)                                                                                \
  hipLaunchKernelGGL((k_dplur<R, NS, NT, ROWS>), g.grid, g.block, 0, st, z, dp, (const R *)in, out, \
                     (const R *)s_in, so, jb)
    if (!epi) {
      if (chem && o.chem == 2)
        OSTC_SWEEP(ROWS_DA);
      else
        OSTC_SWEEP(ROWS_DIAGONAL);
    } else if constexpr (NS == kRedSpec) {
      if (reduced)
        OSTC_SWEEP(ROWS_REDUCED);
      else
        OSTC_SWEEP(ROWS_SUMS);
    } else {
      OSTC_SWEEP(ROWS_SUMS);
    }
#undef OSTC_SWEEP
    prof_mark(P_DPLUR, st, false);
    if (last_err()) return OSTC_ERR_HIP;
    if (epi && !reduced) {
      prof_mark(P_DPLUR_CHEM, st, true);
      int r = chem_solve<R, NS>(z, dp, o, chem_late, out, st);
      if (r == OSTC_OK && !last) {
        hipLaunchKernelGGL((k_dplur_scalars<R, NS, false>), g.grid, g.block, 0, st, z, dp, (const R *)out, s_out);
        r = last_err();
      }
      prof_mark(P_DPLUR_CHEM, st, false);
      if (r) return r;
    }
    std::swap(s_in, s_out);
    in = out;
    out = (out == z.dqk) ? z.dq : z.dqk;
  }
  *result = in;
  return OSTC_OK;
}

}  // namespace

template <typename R>
int dplur_scalars(const ZoneView<R> &z, const ostc_param *dp, const CellOpts &o, hipStream_t st) {
  const auto g = cell_grid(z.mx, z.my, z.mz);
  R *s = z.imp + z.plane;
  if (o.ns == 9)
    hipLaunchKernelGGL((k_dplur_scalars<R, 9, true>), g.grid, g.block, 0, st, z, dp, (const R *)z.dq0, s);
  else if (o.ns == 20)
    hipLaunchKernelGGL((k_dplur_scalars<R, 20, true>), g.grid, g.block, 0, st, z, dp, (const R *)z.dq0, s);
  else
    return OSTC_ERR_ARG;
  return last_err();
}

template <typename R>
int dplur_sweeps(const ZoneView<R> &z, const ostc_param *dp, const CellOpts &o, hipStream_t st, bool chem_late,
                 R **result) {
  if (o.ns == 0) return o.nt == 2 ? sweeps_air<R, 2>(z, dp, o, st, result) : sweeps_air<R, 0>(z, dp, o, st, result);
  if (o.ns == 9 && o.nt == 2) return sweeps<R, 9, 2>(z, dp, o, st, chem_late, result);
  if (o.ns == 9 && o.nt == 0) return sweeps<R, 9, 0>(z, dp, o, st, chem_late, result);
  if (o.ns == 20 && o.nt == 2) return sweeps<R, 20, 2>(z, dp, o, st, chem_late, result);
  if (o.ns == 20 && o.nt == 0) return sweeps<R, 20, 0>(z, dp, o, st, chem_late, result);
  return OSTC_ERR_ARG;
}

template int dplur_scalars<float>(const ZoneView<float> &, const ostc_param *, const CellOpts &, hipStream_t);
template int dplur_scalars<double>(const ZoneView<double> &, const ostc_param *, const CellOpts &, hipStream_t);
template int dplur_sweeps<float>(const ZoneView<float> &, const ostc_param *, const CellOpts &, hipStream_t, bool,
                                 float **);
template int dplur_sweeps<double>(const ZoneView<double> &, const ostc_param *, const CellOpts &, hipStream_t, bool,
                                  double **);

}  // namespace ostc
