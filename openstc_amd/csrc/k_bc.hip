// Boundary conditions (src/BoundCond.cuh:45-412) and the on-device inner-face
// halo exchange (src/DataCommunication.cuh:27-98): one thread per (face point,
// layer), faces that touch no common point in one launch.
#include <algorithm>

#include "ostc_kernels.h"
#include "ostc_thermo.h"

namespace ostc {

namespace {

// Thread -> (face point, layer g): g = 0 is the face point itself, 1..ngg the
// ghost layers outside it.  Every (point, layer) pair is independent, so the
// layers run in parallel and each thread issues all its loads before its
// stores.  On an i-face four adjacent lanes take the layers of one row (the
// layers are adjacent in memory there); on j/k faces i varies fastest.  id:
// the face point's index; step: the index distance of one layer outward.
template <typename R, int FACE>
__device__ __forceinline__ bool face_layer(const ZoneView<R> &z, const FaceLaunch &f, uint3 blk, int64_t &id,
                                           int64_t &step, int &g) {
  constexpr int A = FACE == 0 ? 1 : 0, B = FACE == 2 ? 1 : 2;
  const int il = FACE == 0 ? (int)(threadIdx.x & 3) : (int)blk.z;
  const int ia = FACE == 0 ? (int)(blk.x * 16 + (threadIdx.x >> 2)) : (int)(blk.x * 64 + threadIdx.x);
  const int a = f.rs[A] + ia, b = f.rs[B] + (int)(blk.y * 4 + threadIdx.y), n = f.rs[FACE];
  g = f.g0 + il;
  id = FACE == 0 ? z.idx(n, a, b) : (FACE == 1 ? z.idx(a, n, b) : z.idx(a, b, n));
  step = (FACE == 0 ? (int64_t)1 : (FACE == 1 ? (int64_t)z.nx : (int64_t)z.nx * z.ny)) * f.direction;
  return g <= z.g && a <= f.re[A] && b <= f.re[B];
}

// compute_total_energy (src/FieldOperation.cuh:15-35) of a point whose bv and
// species cv are in registers
template <typename R, int NS>
__device__ __forceinline__ R total_energy_reg(const ostc_param *__restrict__ p, R rho, R u, R v, R w, R pr, R t,
                                              const R *cvs, R &vel) {
  const R vel2 = u * u + v * v + w * w;
  R e = (R)0.5 * rho * vel2;
  if constexpr (NS > 0) {
    R h[NS];
    enthalpy<R>(t, h, p, NS);
#pragma unroll
    for (int l = 0; l < NS; ++l) e += h[l] * cvs[l];
    e -= pr;
  } else {
    e += pr / (R)(kGammaAir - 1);
  }
  vel = sqrt(vel2);
  return e;
}

// apply_outflow (src/BoundCond.cuh:127-154): ghost layer g copies the face point
template <typename R, int NSC, bool RANS, int FACE>
__device__ __forceinline__ void outflow_face(const ZoneView<R> &z, const FaceLaunch &f, uint3 blk) {
  int64_t id, step;
  int g;
  if (!face_layer<R, FACE>(z, f, blk, id, step, g)) return;
  const int64_t P = z.plane;
  const int64_t gi = id + g * step;
  R bv[6], sv[NSC > 0 ? NSC : 1], mut = 0;
#pragma unroll
  for (int l = 0; l < 6; ++l) bv[l] = z.bv[l * P + id];
#pragma unroll
  for (int l = 0; l < NSC; ++l) sv[l] = z.sv[l * P + id];
  if (RANS) mut = z.mut[id];
#pragma unroll
  for (int l = 0; l < 6; ++l) z.bv[l * P + gi] = bv[l];
#pragma unroll
  for (int l = 0; l < NSC; ++l) z.sv[l * P + gi] = sv[l];
  if (RANS) z.mut[gi] = mut;
}

// apply_inflow (src/BoundCond.cuh:156-194): ghost layers take the inflow state
template <typename R, int NSC, bool RANS, int FACE>
__device__ __forceinline__ void inflow_face(const ZoneView<R> &z, const FaceLaunch &f, uint3 blk,
                                            const ostc_inflow *__restrict__ in) {
  int64_t id, step;
  int g;
  if (!face_layer<R, FACE>(z, f, blk, id, step, g)) return;
  const int64_t P = z.plane;
  const int64_t gi = id + g * step;
  z.bv[gi] = (R)in->density;
  z.bv[P + gi] = (R)in->u;
  z.bv[2 * P + gi] = (R)in->v;
  z.bv[3 * P + gi] = (R)in->w;
  z.bv[4 * P + gi] = (R)in->pressure;
  z.bv[5 * P + gi] = (R)in->temperature;
#pragma unroll
  for (int l = 0; l < NSC; ++l) z.sv[l * P + gi] = (R)in->sv[l];
  if (RANS) z.mut[gi] = (R)in->mut;
}

// apply_symmetry (src/BoundCond.cuh:45-125): layer 0 = the face point (the
// interior neighbour's state with its normal velocity removed), layer g = the
// mirror of interior point -g with the normal velocity reversed
template <typename R, int NSC, bool RANS, int FACE>
__device__ __forceinline__ void symmetry_face(const ZoneView<R> &z, const FaceLaunch &f, uint3 blk) {
  int64_t id, step;
  int g;
  if (!face_layer<R, FACE>(z, f, blk, id, step, g)) return;
  const int64_t P = z.plane;
  R kx = z.metric[(FACE * 3) * P + id], ky = z.metric[(FACE * 3 + 1) * P + id],
    kz = z.metric[(FACE * 3 + 2) * P + id];
  const R km = sqrt(kx * kx + ky * ky + kz * kz);
  kx /= km;
  ky /= km;
  kz /= km;
  if (g == 0) {
    const int64_t in = id - step;
    const R u1 = z.bv[P + in], v1 = z.bv[2 * P + in], w1 = z.bv[3 * P + in];
    const R rho = z.bv[in], pr = z.bv[4 * P + in], tt = z.bv[5 * P + in], e1 = z.cv[4 * P + in];
    R sv[NSC > 0 ? NSC : 1];
#pragma unroll
    for (int l = 0; l < NSC; ++l) sv[l] = z.sv[l * P + in];
    const R uk = kx * u1 + ky * v1 + kz * w1;
    const R ut = u1 - kx * uk, vt = v1 - ky * uk, wt = w1 - kz * uk;
    z.bv[P + id] = ut;
    z.bv[2 * P + id] = vt;
    z.bv[3 * P + id] = wt;
    z.vel[id] = sqrt(ut * ut + vt * vt + wt * wt);
    z.bv[id] = rho;
    z.bv[4 * P + id] = pr;
    z.bv[5 * P + id] = tt;
#pragma unroll
    for (int l = 0; l < NSC; ++l) z.sv[l * P + id] = sv[l];
    z.cv[id] = rho;
    z.cv[P + id] = rho * ut;
    z.cv[2 * P + id] = rho * vt;
    z.cv[3 * P + id] = rho * wt;
    z.cv[4 * P + id] = e1 - (R)0.5 * rho * (u1 * u1 + v1 * v1 + w1 * w1) + (R)0.5 * rho * (ut * ut + vt * vt + wt * wt);
#pragma unroll
    for (int l = 0; l < NSC; ++l) z.cv[(5 + l) * P + id] = rho * sv[l];
    return;
  }
  const int64_t gi = id + g * step;
  const int64_t si = id - g * step;
  const R rho = z.bv[si], u = z.bv[P + si], v = z.bv[2 * P + si], w = z.bv[3 * P + si];
  const R pr = z.bv[4 * P + si], tt = z.bv[5 * P + si];
  R sv[NSC > 0 ? NSC : 1], mut = 0;
#pragma unroll
  for (int l = 0; l < NSC; ++l) sv[l] = z.sv[l * P + si];
  if (RANS) mut = z.mut[si];
  const R uk = kx * u + ky * v + kz * w;
  const R ug = u - (R)2 * uk * kx, vg = v - (R)2 * uk * ky, wg = w - (R)2 * uk * kz;
  z.bv[gi] = rho;
  z.bv[P + gi] = ug;
  z.bv[2 * P + gi] = vg;
  z.bv[3 * P + gi] = wg;
  z.vel[gi] = sqrt(ug * ug + vg * vg + wg * wg);
  z.bv[4 * P + gi] = pr;
  z.bv[5 * P + gi] = tt;
#pragma unroll
  for (int l = 0; l < NSC; ++l) z.sv[l * P + gi] = sv[l];
  if (RANS) z.mut[gi] = mut;
}

// apply_wall (src/BoundCond.cuh:196-319): layer 0 = the wall point (no slip,
// pressure of the interior neighbour, wall or interior temperature, SST omega
// at the wall), layer g = the reflection of interior point -g; a ghost thread
// recomputes the wall omega it copies
template <typename R, int NS, bool RANS, int FACE>
__device__ __forceinline__ void wall_face(const ZoneView<R> &z, const FaceLaunch &f, uint3 blk,
                                          const ostc_param *__restrict__ p, int isothermal, double tw_in) {
  int64_t id, step;
  int g;
  if (!face_layer<R, FACE>(z, f, blk, id, step, g)) return;
  const int64_t P = z.plane;
  const int64_t in = id - step;
  R t_wall = (R)tw_in;
  if (!isothermal) t_wall = z.bv[5 * P + in];
  const R pw = z.bv[4 * P + in];
  R mw = (R)kMwAir;
  R yw[NS > 0 ? NS : 1];
  if constexpr (NS > 0) {
    mw = 0;
#pragma unroll
    for (int l = 0; l < NS; ++l) {
      yw[l] = z.sv[l * P + in];
      mw += yw[l] * inv_mw<R>(p, l);
    }
    mw = (R)1 / mw;
  }
  const R rho_w = pw * mw / (t_wall * (R)kRu);
  R om = 0;
  if constexpr (RANS) {
    R mu_w;
    if constexpr (NS > 0) {
      mixture_transport<R>(p, NS, t_wall, mw, yw, (const R *)nullptr, &mu_w, (R *)nullptr, (R *)nullptr);
    } else {
      mu_w = sutherland<R>(t_wall);
    }
    const R dy = z.wall_dist[in];
    if (dy > (R)1e-25)
      om = (R)60 * mu_w / (rho_w * (R)sst::beta_1 * dy * dy);
    else
      om = z.sv[(NS + 1) * P + in];
  }
  if (g == 0) {
    R cvs[NS > 0 ? NS : 1];
#pragma unroll
    for (int l = 0; l < NS; ++l) cvs[l] = yw[l] * rho_w;
    R vel;
    const R e = total_energy_reg<R, NS>(p, rho_w, (R)0, (R)0, (R)0, pw, t_wall, cvs, vel);
#pragma unroll
    for (int l = 0; l < NS; ++l) z.sv[l * P + id] = yw[l];
    z.bv[id] = rho_w;
    z.bv[P + id] = 0;
    z.bv[2 * P + id] = 0;
    z.bv[3 * P + id] = 0;
    z.bv[4 * P + id] = pw;
    z.bv[5 * P + id] = t_wall;
    z.cv[id] = rho_w;
    z.cv[P + id] = 0;
    z.cv[2 * P + id] = 0;
    z.cv[3 * P + id] = 0;
#pragma unroll
    for (int l = 0; l < NS; ++l) z.cv[(5 + l) * P + id] = cvs[l];
    z.cv[4 * P + id] = e;
    z.vel[id] = vel;
    if constexpr (RANS) {
      z.sv[NS * P + id] = 0;
      z.cv[(NS + 5) * P + id] = 0;
      z.sv[(NS + 1) * P + id] = om;
      z.cv[(NS + 6) * P + id] = rho_w * om;
    }
    return;
  }
  const int64_t si = id - g * step;
  const int64_t gi = id + g * step;
  const R ui = z.bv[P + si], vi = z.bv[2 * P + si], wi = z.bv[3 * P + si];
  const R pi = z.bv[4 * P + si], ti = z.bv[5 * P + si];
  R ys[NS > 0 ? NS : 1];
  R mg = (R)kMwAir;
  if constexpr (NS > 0) {
    mg = 0;
#pragma unroll
    for (int l = 0; l < NS; ++l) {
      ys[l] = z.sv[l * P + si];
      mg += ys[l] * inv_mw<R>(p, l);
    }
    mg = (R)1 / mg;
  }
  R tg = ti;
  if (isothermal) {
    tg = (R)2 * t_wall - ti;
    if (tg <= (R)0.1 * t_wall) tg = t_wall;
  }
#pragma unroll
  for (int l = 0; l < NS; ++l) z.sv[l * P + gi] = ys[l];
  z.bv[gi] = pi * mg / (tg * (R)kRu);
  z.bv[P + gi] = -ui;
  z.bv[2 * P + gi] = -vi;
  z.bv[3 * P + gi] = -wi;
  z.bv[4 * P + gi] = pi;
  z.bv[5 * P + gi] = tg;
  if constexpr (RANS) {
    z.sv[NS * P + gi] = 0;
    z.sv[(NS + 1) * P + gi] = om;
    z.mut[gi] = 0;
  }
}

template <typename R, int NS, int NT, int FACE>
__device__ __forceinline__ void one_face(const ZoneView<R> &z, const BatchFace &b, uint3 blk,
                                         const ostc_param *__restrict__ p, const ostc_inflow *__restrict__ in) {
  constexpr int NSC = NS + NT;
  constexpr bool RANS = NT > 0;
  switch (b.kind) {
    case 6: outflow_face<R, NSC, RANS, FACE>(z, b.f, blk); break;
    case 5: inflow_face<R, NSC, RANS, FACE>(z, b.f, blk, in + b.slot); break;
    case 3: symmetry_face<R, NSC, RANS, FACE>(z, b.f, blk); break;
    default: wall_face<R, NS, RANS, FACE>(z, b.f, blk, p, b.isothermal, b.temperature); break;
  }
}

// One launch over the faces of a batch.  The batch travels with the launch, as
// the grid does, so that a launch that is queued or captured keeps the faces,
// wall flags and wall temperatures it was made for.  What a launch costs is
// latency: the workgroup's face follows from the grid's z (no divisions), and
// the face direction is a template argument (no indexed registers): the code
// a wave walks through once, uncached, is the time.
template <typename R, int NS, int NT>
__global__ __launch_bounds__(256) void k_faces(ZoneView<R> z, const FaceBatch batch,
                                               const ostc_param *__restrict__ p,
                                               const ostc_inflow *__restrict__ in) {
  int q = 0;
#pragma unroll
  for (int k = 1; k < kBatchFaces; ++k) q += (int)blockIdx.z >= batch.first[k];
  const BatchFace &b = batch.face[q];
  if ((int)blockIdx.x >= b.gx || (int)blockIdx.y >= b.gy) return;
  const uint3 blk = make_uint3(blockIdx.x, blockIdx.y, blockIdx.z - (unsigned)b.first);
  if (b.f.face == 0)
    one_face<R, NS, NT, 0>(z, b, blk, p, in);
  else if (b.f.face == 1)
    one_face<R, NS, NT, 1>(z, b, blk, p, in);
  else
    one_face<R, NS, NT, 2>(z, b, blk, p, in);
}

// update_bv_1_point (src/FieldOperation.cuh:185-215) incl. the Newton solve
template <typename R, int NS, int NT>
__device__ __forceinline__ void update_bv_point(const ZoneView<R> &z, const ostc_param *__restrict__ p, int64_t id) {
  const int64_t P = z.plane;
  const R rho = z.cv[id];
  const R rinv = (R)1.0 / rho;
  z.bv[id] = rho;
  const R u = z.cv[P + id] * rinv, v = z.cv[2 * P + id] * rinv, w = z.cv[3 * P + id] * rinv;
  z.bv[P + id] = u;
  z.bv[2 * P + id] = v;
  z.bv[3 * P + id] = w;
  const R vel2 = u * u + v * v + w * w;
#pragma unroll
  for (int l = 0; l < NS + NT; ++l) z.sv[l * P + id] = z.cv[(5 + l) * P + id] * rinv;
  if constexpr (NS > 0) {
    double y[NS], mw = 0;
#pragma unroll
    for (int l = 0; l < NS; ++l) {
      y[l] = (double)z.sv[l * P + id];
      mw += y[l] / p->mw[l];
    }
    mw = 1 / mw;
    const double gc = kRu / mw;
    const double e = (double)z.cv[4 * P + id] / (double)rho -
                     0.5 * ((double)u * u + (double)v * v + (double)w * w);
    double t = (double)z.bv[5 * P + id];
    double err = 1;
    int iter = 0;
    while (err > 1e-3 && iter++ < 1000) {
      double h[NS], cp[NS];
      enthalpy_cp<double>(t, h, cp, p, NS);
      double cpt = 0, hm = 0;
#pragma unroll
      for (int l = 0; l < NS; ++l) {
        cpt += cp[l] * y[l];
        hm += h[l] * y[l];
      }
      const double t1 = t - (hm - gc * t - e) / (cpt - gc);
      err = fabs(1 - t1 / t);
      t = t1;
    }
    z.bv[5 * P + id] = (R)t;
    z.bv[4 * P + id] = (R)((double)rho * t * gc);
  } else {
    const R pr = (R)(kGammaAir - 1) * (z.cv[4 * P + id] - (R)0.5 * rho * vel2);
    z.bv[4 * P + id] = pr;
    z.bv[5 * P + id] = pr * (R)kMwAir * rinv / (R)kRu;
  }
  z.vel[id] = sqrt(vel2);
}

// inner_communication (src/DataCommunication.cuh:58-98)
template <typename R, int NS, int NT>
__global__ void k_inner(ZoneView<R> z, ZoneView<R> t, const ostc_param *__restrict__ p, ostc_inner_face f) {
  constexpr int NV = 5 + NS + NT;
  const int n[3] = {(int)(blockIdx.x * blockDim.x + threadIdx.x), (int)(blockIdx.y * blockDim.y + threadIdx.y),
                    (int)(blockIdx.z * blockDim.z + threadIdx.z)};
  if (n[0] >= f.n_point[0] || n[1] >= f.n_point[1] || n[2] >= f.n_point[2]) return;
  int idx[3], it[3], d[3];
#pragma unroll
  for (int q = 0; q < 3; ++q) {
    d[q] = f.loop_dir[q] * n[q];
    idx[q] = f.range_start[q] + d[q];
  }
#pragma unroll
  for (int q = 0; q < 3; ++q) it[q] = f.target_start[q] + f.target_loop_dir[q] * d[f.src_tar[q]];
  const int face_dir = f.direction > 0 ? f.range_start[f.face] : f.range_end[f.face];
  const int64_t a = z.idx(idx[0], idx[1], idx[2]), b = t.idx(it[0], it[1], it[2]);
  if (idx[f.face] == face_dir) {
#pragma unroll
    for (int l = 0; l < NV; ++l) {
      const R ave = (R)0.5 * (t.cv[l * t.plane + b] + z.cv[l * z.plane + a]);
      z.cv[l * z.plane + a] = ave;
      t.cv[l * t.plane + b] = ave;
    }
    update_bv_point<R, NS, NT>(z, p, a);
  } else {
#pragma unroll
    for (int l = 0; l < 6; ++l) z.bv[l * z.plane + a] = t.bv[l * t.plane + b];
#pragma unroll
    for (int l = 0; l < NS + NT; ++l) z.sv[l * z.plane + a] = t.sv[l * t.plane + b];
  }
}

// launch shape of face_layer: layers g0..ngg of every face point
dim3 face_grid(const FaceLaunch &f, int ngg, dim3 &block) {
  const int a = f.face == 0 ? 1 : 0, b = f.face == 2 ? 1 : 2;
  const int na = f.re[a] - f.rs[a] + 1, nb = f.re[b] - f.rs[b] + 1;
  const int nl = ngg + 1 - f.g0;
  block = dim3(64, 4, 1);
  if (f.face == 0) return dim3((na + 15) / 16, (nb + 3) / 4, 1);  // 4 lanes (layers) per point
  return dim3((na + 63) / 64, (nb + 3) / 4, nl);
}

// Wall friction coefficient and heat flux along the j = 0 wall of the k = 0
// line (wall_friction_heatFlux_2d, src/PostProcess.cu:49-70): per i,
//   u_par = (xi_x u + xi_y v) / |(xi_x, xi_y)|  at j = 1,
//   cf    = mu_l(i,0,0) u_par |(eta_x, eta_y)| / q_dyn,
//   qw    = lambda(i,0,0) (T(i,1,0) - T(i,0,0)) |(eta_x, eta_y)|,
// evaluated in FP64 from the stored fields (metrics at the wall point).
template <typename R>
__global__ __launch_bounds__(128) void k_wall_cf_qw(ZoneView<R> z, double dyn_pressure, double *__restrict__ cf,
                                                    double *__restrict__ qw) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= z.mx) return;
  const int64_t w = z.idx(i, 0, 0), a = z.idx(i, 1, 0);
  const double xi_x = z.m(w, 1, 1), xi_y = z.m(w, 1, 2);
  const double eta_x = z.m(w, 2, 1), eta_y = z.m(w, 2, 2);
  const double u = z.bv[a + z.plane], v = z.bv[a + 2 * z.plane];
  const double u_par = (xi_x * u + xi_y * v) / sqrt(xi_x * xi_x + xi_y * xi_y);
  const double grad_eta = sqrt(eta_x * eta_x + eta_y * eta_y);
  cf[i] = (double)z.mul[w] * (u_par * grad_eta) / dyn_pressure;
  const double t1 = z.bv[a + 5 * z.plane], t0 = z.bv[w + 5 * z.plane];
  qw[i] = (double)z.lambda[w] * (t1 - t0) * grad_eta;
}

}  // namespace

namespace {

// Points a face reads and writes: its ranges, and along its normal the
// offsets lo..hi outward from the face point.
struct FaceBox {
  int lo[3], hi[3];
};
FaceBox face_box(const FaceLaunch &f, int from, int to) {
  FaceBox b;
  for (int q = 0; q < 3; ++q) {
    b.lo[q] = f.rs[q];
    b.hi[q] = f.re[q];
  }
  const int x = f.rs[f.face] + f.direction * from, y = f.rs[f.face] + f.direction * to;
  b.lo[f.face] = std::min(x, y);
  b.hi[f.face] = std::max(x, y);
  return b;
}
bool meet(const FaceBox &a, const FaceBox &b) {
  for (int q = 0; q < 3; ++q)
    if (a.hi[q] < b.lo[q] || b.hi[q] < a.lo[q]) return false;
  return true;
}
// neither face writes a point the other reads or writes
bool independent(const FaceLaunch &a, const FaceLaunch &b, int ngg) {
  const FaceBox wa = face_box(a, 0, ngg), wb = face_box(b, 0, ngg);
  const FaceBox ra = face_box(a, -ngg, 0), rb = face_box(b, -ngg, 0);
  return !meet(wa, wb) && !meet(wa, rb) && !meet(ra, wb);
}

}  // namespace

int plan_bc(const ostc_bc &bc, int ngg, std::vector<FaceBatch> &batches) {
  batches.clear();
  if (ngg > 3) return OSTC_ERR_ARG;  // four lanes per point on i-faces
  for (int fi = 0; fi < bc.n_face; ++fi) {
    const ostc_face &bf = bc.face[fi];
    BatchFace q{};
    FaceLaunch &f = q.f;
    for (int d = 0; d < 3; ++d) {
      f.rs[d] = bf.range_start[d];
      f.re[d] = bf.range_end[d];
    }
    f.face = bf.face;
    f.direction = bf.direction;
    f.g0 = (bf.kind == 5 || bf.kind == 6) ? 1 : 0;  // inflow/outflow write only the ghost layers
    for (int d = 0; d < 3; ++d)
      if (d != f.face && f.re[d] < f.rs[d]) return OSTC_ERR_ARG;  // an empty face
    dim3 block;
    const dim3 grid = face_grid(f, ngg, block);
    q.kind = bf.kind;
    q.slot = bf.slot;
    q.gx = (int)grid.x;
    q.gy = (int)grid.y;
    if (bf.kind == 2) {
      q.isothermal = bc.wall[bf.slot].isothermal;
      q.temperature = bc.wall[bf.slot].temperature;
    }
    bool joins = !batches.empty() && batches.back().n < kBatchFaces;
    if (joins)
      for (int k = 0; k < batches.back().n && joins; ++k) joins = independent(batches.back().face[k].f, f, ngg);
    if (!joins) batches.emplace_back();
    FaceBatch &b = batches.back();
    q.first = b.gz;
    b.first[b.n] = b.gz;
    b.face[b.n++] = q;
    b.gx = std::max(b.gx, q.gx);
    b.gy = std::max(b.gy, q.gy);
    b.gz += (int)grid.z;
  }
  for (auto &b : batches)
    for (int k = b.n; k < kBatchFaces; ++k) b.first[k] = b.gz;
  return OSTC_OK;
}

template <typename R>
int apply_bc(const ZoneView<R> &z, const ostc_param *dp, const CellOpts &o, const std::vector<FaceBatch> &plan,
             const ostc_inflow *d_inflow, hipStream_t st) {
  for (const FaceBatch &b : plan) {
    const dim3 grid((unsigned)b.gx, (unsigned)b.gy, (unsigned)b.gz), block(64, 4, 1);
    OSTC_DISPATCH_NSNT(o, hipLaunchKernelGGL((k_faces<R, NS_, NT_>), grid, block, 0, st, z, b, dp, d_inflow));
    if (hipGetLastError() != hipSuccess) return OSTC_ERR_HIP;
  }
  return OSTC_OK;
}

template <typename R>
int inner_halo(const ZoneView<R> &z, const ZoneView<R> &t, const ostc_param *dp, const CellOpts &o,
               const ostc_inner_face &f, hipStream_t st) {
  unsigned tpb[3], bpg[3];
  const int fd = f.face;
  if (fd >= 0 && fd < 3 && f.n_point[fd] <= 2 * z.g + 1) {
    // all layers of a face point in one workgroup, on adjacent lanes: along
    // i (an i face) a row's layers then share their cache lines; i first
    // among the other two directions, where it is one of them
    tpb[fd] = f.n_point[fd];
    int budget = 256 / (int)tpb[fd];
    for (int q = 0; q < 3; ++q) {
      if (q == fd) continue;
      const int want = q == 0 ? 64 : 16;
      tpb[q] = (unsigned)std::max(1, std::min(std::min(want, budget), f.n_point[q]));
      budget = std::max(1, budget / (int)tpb[q]);
    }
  } else {
    for (int q = 0; q < 3; ++q) tpb[q] = f.n_point[q] <= 2 * z.g + 1 ? 1 : 16;
  }
  for (int q = 0; q < 3; ++q) bpg[q] = (f.n_point[q] - 1) / tpb[q] + 1;
  const dim3 grid(bpg[0], bpg[1], bpg[2]), block(tpb[0], tpb[1], tpb[2]);
  if (o.ns == 0 && o.nt == 0)
    hipLaunchKernelGGL((k_inner<R, 0, 0>), grid, block, 0, st, z, t, dp, f);
  else if (o.ns == 0 && o.nt == 2)
    hipLaunchKernelGGL((k_inner<R, 0, 2>), grid, block, 0, st, z, t, dp, f);
  else if (o.ns == 9 && o.nt == 0)
    hipLaunchKernelGGL((k_inner<R, 9, 0>), grid, block, 0, st, z, t, dp, f);
  else if (o.ns == 9 && o.nt == 2)
    hipLaunchKernelGGL((k_inner<R, 9, 2>), grid, block, 0, st, z, t, dp, f);
  else if (o.ns == 20 && o.nt == 0)
    hipLaunchKernelGGL((k_inner<R, 20, 0>), grid, block, 0, st, z, t, dp, f);
  else if (o.ns == 20 && o.nt == 2)
    hipLaunchKernelGGL((k_inner<R, 20, 2>), grid, block, 0, st, z, t, dp, f);
  else
    return OSTC_ERR_ARG;
  return hipGetLastError() == hipSuccess ? OSTC_OK : OSTC_ERR_HIP;
}

template <typename R>
int wall_friction_heatflux(const ZoneView<R> &z, double dyn_pressure, double *cf, double *qw, hipStream_t st) {
  hipLaunchKernelGGL((k_wall_cf_qw<R>), dim3((z.mx + 127) / 128), dim3(128), 0, st, z, dyn_pressure, cf, qw);
  return hipGetLastError() == hipSuccess ? OSTC_OK : OSTC_ERR_HIP;
}

template int apply_bc<float>(const ZoneView<float> &, const ostc_param *, const CellOpts &,
                             const std::vector<FaceBatch> &, const ostc_inflow *, hipStream_t);
template int apply_bc<double>(const ZoneView<double> &, const ostc_param *, const CellOpts &,
                              const std::vector<FaceBatch> &, const ostc_inflow *, hipStream_t);
template int inner_halo<float>(const ZoneView<float> &, const ZoneView<float> &, const ostc_param *,
                               const CellOpts &, const ostc_inner_face &, hipStream_t);
template int inner_halo<double>(const ZoneView<double> &, const ZoneView<double> &, const ostc_param *,
                                const CellOpts &, const ostc_inner_face &, hipStream_t);
template int wall_friction_heatflux<float>(const ZoneView<float> &, double, double *, double *, hipStream_t);
template int wall_friction_heatflux<double>(const ZoneView<double> &, double, double *, double *, hipStream_t);

}  // namespace ostc
