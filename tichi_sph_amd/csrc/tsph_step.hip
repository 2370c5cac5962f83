// Fused per-step kernels of the DFSPH / VFSPH step (main.py:175-256).
//
// Storage is in cell order (tsph_grid.hip).  The 27 (3D) / 9 (2D) cells of a
// particle's neighbourhood are visited as 9 / 3 contiguous row runs: cells
// (x-R .. x+R) of one (y, z) row have consecutive codes and therefore
// consecutive slots, in the reference's template order (x fastest,
// sph_config.py:219-224) and in-cell order.  Pass A walks the runs once per
// step, testing every candidate, and records the in-range neighbours
// (0 < r < h, exact f32 test) of each fluid particle in reference order;
// every later sweep iterates only those lists.  Terms beyond h are exact
// zeros in the reference, so skipping them changes no value.
#include <cstring>
#include <type_traits>

#include "tsph_sweep.h"

namespace tsph {

// Pair terms of pass A for one in-range candidate (strict arithmetic, the
// order of sph.py:61-64, 81, 97).
template <class T>
struct PassAAcc {
  T w = 0, cp = 0, dn = 0, ax = 0, ay = 0, az = 0, a2 = 0;
  T bx = 0, by = 0, bz = 0;  // the boundary neighbours' share of alpha_1
  // XM: the solver alias X is the mass (DFSPH), so X_j = m_j
  template <bool FQ, bool XM>
  __device__ __forceinline__ bool add(const KP<T>& k, const V4<T>& p, const V4<T>& q, T mj, T vj,
                                      bool fluid) {
    T dx = p.x - q.x, dy = p.y - q.y, dz = p.z - q.z;
    T r2, r, qh;
    {
      TSPH_STRICT
      r2 = s_r2(dx, dy, dz);
      r = pa_sqrt<FQ>(r2);
      qh = pa_quot<FQ>(k, r);
      T Wr = s_W_q_sel(k, qh);
      w = w + Wr;
      cp = cp + Wr * vj;
      dn = dn + Wr * mj;
      if (!(r > T(0))) return false;
    }
    // W'(q) / r from the r and q just formed: 6 sig/h^2 (3q - 2) for q <= 1/2
    // (no division), -6 sig/h (1 - q)^2 / r above
    const T u = T(1) - qh;
    const T g = qh <= T(0.5) ? k.wg_a * (T(3) * qh - T(2)) : -k.wg_b * (u * u) * f_rcp(r);
    T Xj = q.w;
    T xg = Xj * g;
    ax += xg * dx;
    ay += xg * dy;
    az += xg * dz;
    if (fluid) {
      // W'^2 X_j^2 / m_j; for DFSPH X_j is m_j and the quotient is X_j
      const T x2m = XM ? Xj : (Xj * Xj) * f_rcp(mj);
      a2 += (g * g) * r2 * x2m;
    } else {
      bx += xg * dx;
      by += xg * dy;
      bz += xg * dz;
    }
    return true;
  }
  // add() for one list slot per lane of a quad: the sums take the quad's terms
  // in lane order (a lane without one adds an exact zero).
  template <bool FQ, bool XM>
  __device__ __forceinline__ void add_quad(const KP<T>& k, const V4<T>& p, const V4<T>& q, T mj,
                                           T vj, bool valid, bool apart, bool fluid) {
    const T dx = p.x - q.x, dy = p.y - q.y, dz = p.z - q.z;
    T r2, r, qh;
    {
      TSPH_STRICT
      r2 = s_r2(dx, dy, dz);
      r = pa_sqrt<FQ>(r2);
      qh = pa_quot<FQ>(k, r);
      // (a lane without a slot holds another's: its products are dropped, since
      // zero times an infinite mass is a NaN)
      const T Wr = s_W_q_sel(k, qh);
      w = quad_add(w, valid ? Wr : T(0));
      cp = quad_add(cp, valid ? Wr * vj : T(0));
      dn = quad_add(dn, valid ? Wr * mj : T(0));
    }
    const T u = T(1) - qh;
    T g = qh <= T(0.5) ? k.wg_a * (T(3) * qh - T(2)) : -k.wg_b * (u * u) * f_rcp(r);
    const T Xj = q.w;
    const T xg = valid && apart ? Xj * g : T(0);
    // both factors: a massless or infinite particle at r = 0 has no term
    const T x2m = !(valid && apart) ? T(0) : XM ? Xj : (Xj * Xj) * f_rcp(mj);
    const T t2 = valid && apart ? (g * g) * r2 : T(0);
    add_lane<0>(xg, dx, dy, dz, t2, x2m, fluid);
    add_lane<1>(xg, dx, dy, dz, t2, x2m, fluid);
    add_lane<2>(xg, dx, dy, dz, t2, x2m, fluid);
    add_lane<3>(xg, dx, dy, dz, t2, x2m, fluid);
  }
  template <int K>
  __device__ __forceinline__ void add_lane(T xg_, T dx_, T dy_, T dz_, T t2, T x2m, bool fluid) {
    const T xg = quad_lane<K>(xg_), dx = quad_lane<K>(dx_), dy = quad_lane<K>(dy_),
            dz = quad_lane<K>(dz_);
    ax += xg * dx;
    ay += xg * dy;
    az += xg * dz;
    if (fluid) {
      a2 += quad_lane<K>(t2) * quad_lane<K>(x2m);
    } else {
      bx += xg * dx;
      by += xg * dy;
      bz += xg * dz;
    }
  }
};

// List slots per particle staged in LDS by pass A (kPassAK x kBlock ints per
// block; 22 KB keeps the kernel at its register-bound occupancy).
constexpr int kPassAK = 22;

// ---------------------------------------------------------------------------
// Pass A, fluid particles: SPH_prepare_attr (f,f)(f,b), SPH_prepare_alpha_1
// (f,f)(f,b), SPH_prepare_alpha_2 (f,f), SPH_prepare_alpha, SPH_vel_2_vel_adv,
// neighbour lists.  Strict arithmetic: bit-for-bit the reference's order.
// ---------------------------------------------------------------------------
template <class T>
__device__ __forceinline__ void pass_a_epilogue(const KP<T>& k, int i, const V4<T>& p, T mi,
                                                const PassAAcc<T>& a, int nf, int nbb,
                                                T* W, T* comp, T* dens, V4<T>* alpha_1,
                                                T* alpha_2, T* alpha, T* vol, const V4<T>* vel,
                                                V4<T>* vel_adv, int* nbr_nf, int* nbr_nb,
                                                TsphControl* ctrl) {
  TSPH_STRICT
  W[i] = a.w;
  comp[i] = a.cp;
  dens[i] = a.dn;
  alpha_1[i] = V4<T>{a.ax, a.ay, a.az, T(0)};
  alpha_2[i] = a.a2;
  T dot = s_r2(a.ax, a.ay, a.az);
  T al = dot / mi + a.a2;  // SPH_prepare_alpha, sph.py:103-105
  if (al < T(1e-4)) al = T(1e-4);
  alpha[i] = al;
  T psi = k.solver == TSPH_VFSPH ? a.cp : a.dn;
  const T Vi = p.w / psi;  // X / sph_psi, reused by the viscosity and normal sweeps
  vol[i] = Vi;
  // SPH_vel_2_vel_adv, sph.py:253-256.  The unused 4th lane carries V_i until
  // the advection sweep, so that sweep gathers one record less per pair; the
  // Jacobi sweeps only update x, y, z.
  const V4<T> v = vel[i];
  vel_adv[i] = V4<T>{v.x, v.y, v.z, Vi};
  if (nf > k.list_cap_f) {
    atomicAdd(&ctrl->overflow_f, 1);
    nf = k.list_cap_f + 1;
  }
  if (nbb > k.list_cap_b) {
    atomicAdd(&ctrl->overflow_b, 1);
    nbb = k.list_cap_b + 1;
  }
  nbr_nf[i] = nf;
  nbr_nb[i] = nbb;
}

template <class T, bool FQ, bool XM>
__device__ __forceinline__ void k_pass_a_fluid_body(Blk blk, const KP<T>& k, int n, int cap, const V4<T>* __restrict__ fpos,
                   const T* __restrict__ fmass, const T* __restrict__ frvol,
                   const int* __restrict__ fstart, int nb, const V4<T>* __restrict__ bpos,
                   const T* __restrict__ bmass, const T* __restrict__ brvol,
                   const int* __restrict__ bstart, T* __restrict__ W, T* __restrict__ comp,
                   T* __restrict__ dens, V4<T>* __restrict__ alpha_1, T* __restrict__ alpha_2,
                   T* __restrict__ alpha, T* __restrict__ vol, const V4<T>* __restrict__ vel,
                   V4<T>* __restrict__ vel_adv, int* __restrict__ nbr_f, int* __restrict__ nbr_b,
                   int* __restrict__ nbr_nf, int* __restrict__ nbr_nb, int* __restrict__ flag,
                   V4<T>* __restrict__ a1b, TsphControl* ctrl, int* __restrict__ stage) {
  const int i = xcd_block(blk.b, blk.nb) * kBlock + threadIdx.x;
  if (i >= n) return;
  const int capf = k.list_cap_f, capb = k.list_cap_b;
  // the first kPassAK slots of each list go to this lane's column of the
  // block's LDS stage; the rest are appended to the list directly
  const int nstage = capf < kPassAK ? capf : kPassAK;
  const int nstage_b = capb < kPassAK ? capb : kPassAK;
  flag[i] = 0;  // SPH_clean_value, sph.py:30
  const V4<T> p = fpos[i];
  const T mi = fmass[i];
  int c[3];
  node_encode(k, p.x, p.y, p.z, c);
  PassAAcc<T> acc;
  int nf = 0, nbb = 0;
  // pos.w is the solver alias X (mass for DFSPH, rest volume for VFSPH), so
  // only the other of the two fields is loaded
  const T* __restrict__ fo = XM ? frvol : fmass;
  const T* __restrict__ bo = XM ? brvol : bmass;
  walk_cells_batched<kPassAU>(k, fstart, c, fpos, [&](int j, const V4<T>& q) {
    if (s_r2(p.x - q.x, p.y - q.y, p.z - q.z) <= k.r2max) {
      const T o = fo[j];
      if (acc.template add<FQ, XM>(k, p, q, XM ? q.w : o, XM ? o : q.w, true)) {
        if (nf < nstage)
          stage[nf * kBlock + threadIdx.x] = j;
        else if (nf < capf)
          nbr_f[(long)nf * cap + i] = j;
        ++nf;
      }
    }
  });
  // the staged slots, row by row: the wave's lanes store consecutive
  // entries of one slot row together, whole lines at a time, instead of one
  // scattered entry per lane whenever a lane finds a neighbour
  const int ns = nf < nstage ? nf : nstage;
  for (int s = 0; s < ns; ++s) nbr_f[(long)s * cap + i] = stage[s * kBlock + threadIdx.x];
  walk_cells_batched<kPassAU>(k, bstart, c, bpos, [&](int j, const V4<T>& q) {
    if (s_r2(p.x - q.x, p.y - q.y, p.z - q.z) <= k.r2max) {
      const T o = bo[j];
      if (acc.template add<FQ, XM>(k, p, q, XM ? q.w : o, XM ? o : q.w, false)) {
        if (nbb < nstage_b)
          stage[nbb * kBlock + threadIdx.x] = j;
        else if (nbb < capb)
          nbr_b[(long)nbb * cap + i] = j;
        ++nbb;
      }
    }
  });
  const int nsb = nbb < nstage_b ? nbb : nstage_b;
  for (int s = 0; s < nsb; ++s) nbr_b[(long)s * cap + i] = stage[s * kBlock + threadIdx.x];
  a1b[i] = V4<T>{acc.bx, acc.by, acc.bz, T(0)};
  pass_a_epilogue(k, i, p, mi, acc, nf, nbb, W, comp, dens, alpha_1, alpha_2, alpha, vol, vel,
                  vel_adv, nbr_nf, nbr_nb, ctrl);
}

// Pass A of the fluid, a quad of lanes per particle (walk_quad).  Every sum
// takes the quad's terms in walk order, so all of them are those of
// k_pass_a_fluid_body, bit for bit.
template <class T>
struct PassARec {
  V4<T> q;
  T o;  // mass or rest volume, whichever is not the alias in q.w
};
template <class T, bool FQ, bool XM>
__device__ __forceinline__ void pass_a_quad_fluid(
    int sub, const KP<T>& k, const TsphObject& f, const TsphObject& b, V4<T>* __restrict__ a1b,
    TsphControl* ctrl, WalkLds& lds) {
  const int i = coop_particle<kQuad>(sub), c = coop_lane<kQuad>();
  if (i >= f.n) return;
  const V4<T>* __restrict__ fpos = (const V4<T>*)f.pos;
  const V4<T> p = fpos[i];
  const T mi = ((const T*)f.mass)[i];
  const unsigned below = (1u << c) - 1;
  PassAAcc<T> acc;
  int cnt[2] = {0, 0};
#pragma unroll
  for (int ob = 0; ob < 2; ++ob) {
    const TsphObject& o = ob == 0 ? f : b;
    const V4<T>* __restrict__ opos = (const V4<T>*)o.pos;
    const T* __restrict__ oo = (const T*)(XM ? o.rest_volume : o.mass);
    int* __restrict__ list = ob == 0 ? f.nbr_f : f.nbr_b;
    const int lcap = ob == 0 ? k.list_cap_f : k.list_cap_b;
    int nl = 0;
    if (ob == 0 || b.n > 0)
      walk_quad(k, o.cell_start, opos, p, lds,
                [&](int j) { return PassARec<T>{opos[j], oo[j]}; },
                [&](const PassARec<T>& r, int j, bool valid, bool apart) {
                  acc.template add_quad<FQ, XM>(k, p, r.q, XM ? r.q.w : r.o, XM ? r.o : r.q.w,
                                                valid, apart, ob == 0);
                  const unsigned v = quad_vote(valid && apart);
                  const int slot = nl + __popc(v & below);
                  if (valid && apart && slot < lcap) list[(long)slot * f.capacity + i] = j;
                  nl += __popc(v);
                });
    cnt[ob] = nl;
  }
  if (c != 0) return;
  f.flag[i] = 0;  // SPH_clean_value, sph.py:30
  a1b[i] = V4<T>{acc.bx, acc.by, acc.bz, T(0)};
  pass_a_epilogue(k, i, p, mi, acc, cnt[0], cnt[1], (T*)f.W, (T*)f.sph_compression,
                  (T*)f.sph_density, (V4<T>*)f.alpha_1, (T*)f.alpha_2, (T*)f.alpha, (T*)f.vol,
                  (const V4<T>*)f.vel, (V4<T>*)f.vel_adv, f.nbr_nf, f.nbr_nb, ctrl);
}

// Runs f(fq, xm) with the fluid body's compile-time variant for these
// constants: the verified fast quotient, and whether X is the mass.
template <class T, class F>
__device__ __forceinline__ void pass_a_fluid_variant(const KP<T>& k, F&& f) {
  using Y = std::true_type;
  using N = std::false_type;
  const bool xm = k.solver != TSPH_VFSPH;
  if (k.fastq) {
    if (xm) f(Y{}, Y{});
    else f(Y{}, N{});
  } else {
    if (xm) f(N{}, Y{});
    else f(N{}, N{});
  }
}

template <class T>
__global__ void __launch_bounds__(kBlock)
    k_pass_a_fluid(KP<T> k, int n, int cap, const V4<T>* __restrict__ fpos,
                   const T* __restrict__ fmass, const T* __restrict__ frvol,
                   const int* __restrict__ fstart, int nb, const V4<T>* __restrict__ bpos,
                   const T* __restrict__ bmass, const T* __restrict__ brvol,
                   const int* __restrict__ bstart, T* __restrict__ W, T* __restrict__ comp,
                   T* __restrict__ dens, V4<T>* __restrict__ alpha_1, T* __restrict__ alpha_2,
                   T* __restrict__ alpha, T* __restrict__ vol, const V4<T>* __restrict__ vel,
                   V4<T>* __restrict__ vel_adv, int* __restrict__ nbr_f, int* __restrict__ nbr_b,
                   int* __restrict__ nbr_nf, int* __restrict__ nbr_nb, int* __restrict__ flag,
                   V4<T>* __restrict__ a1b, TsphControl* ctrl) {
  __shared__ int stage[kPassAK * kBlock];
  const Blk blk{(int)blockIdx.x, (int)gridDim.x};
  pass_a_fluid_variant(k, [&](auto fq, auto xm) {
    k_pass_a_fluid_body<T, decltype(fq)::value, decltype(xm)::value>(blk, k, n, cap, fpos, fmass, frvol, fstart, nb, bpos, bmass, brvol, bstart, W, comp, dens, alpha_1, alpha_2, alpha, vol, vel, vel_adv, nbr_f, nbr_b, nbr_nf, nbr_nb, flag, a1b, ctrl, stage);
  });
}

template <class T>
struct BoundRec {
  V4<T> q;
  T v, m;  // rest volume, mass
};

// Pass A, boundary particles: SPH_prepare_attr (b,b)(b,f), SPH_prepare_alpha_2
// (b,f), SPH_prepare_alpha (alpha_1 of the boundary is never accumulated).
// The reference adds all (b,b) pairs before the (b,f) ones (main.py:189-190),
// and the boundary never moves, so the (b,b) partial sums are kept in ss
// (when given): with `kept` they are read instead of summed, otherwise summed
// and stored.
template <class T, bool FQ>
__device__ __forceinline__ void k_pass_a_bound_body(Blk blk, const KP<T>& k, int nb, const V4<T>* __restrict__ bpos, const T* __restrict__ bmass,
                   const T* __restrict__ brvol, const int* __restrict__ bstart,
                   const V4<T>* __restrict__ fpos, const T* __restrict__ fmass,
                   const T* __restrict__ frvol, const int* __restrict__ fstart,
                   T* __restrict__ W, T* __restrict__ comp, T* __restrict__ dens,
                   V4<T>* __restrict__ alpha_1, T* __restrict__ alpha_2, T* __restrict__ alpha,
                   T* __restrict__ vol, V4<T>* __restrict__ ss, bool kept) {
  TSPH_STRICT
  int i = xcd_block(blk.b, blk.nb) * kBlock + threadIdx.x;
  if (i >= nb) return;
  V4<T> p = bpos[i];
  int c[3];
  node_encode(k, p.x, p.y, p.z, c);
  T w = 0, cp = 0, dn = 0, a2 = 0;
  if (ss != nullptr && kept) {
    const V4<T> s0 = ss[i];
    w = s0.x;
    cp = s0.y;
    dn = s0.z;
  } else {
    walk_cells_batched<kPassAU>(k, bstart, c, bpos, [&](int j, const V4<T>& q) {
      T r2 = s_r2(p.x - q.x, p.y - q.y, p.z - q.z);
      if (r2 <= k.r2max) {
        T Wr = s_W_q(k, pa_quot<FQ>(k, pa_sqrt<FQ>(r2)));
        w = w + Wr;
        cp = cp + Wr * brvol[j];
        dn = dn + Wr * bmass[j];
      }
    });
    if (ss != nullptr) ss[i] = V4<T>{w, cp, dn, T(0)};
  }
  walk_cells_batched<kPassAU>(k, fstart, c, fpos, [&](int j, const V4<T>& q) {
    T r2 = s_r2(p.x - q.x, p.y - q.y, p.z - q.z);
    if (r2 <= k.r2max) {
      T r = pa_sqrt<FQ>(r2);
      T qh = pa_quot<FQ>(k, r);
      T Wr = s_W_q(k, qh);
      w = w + Wr;
      cp = cp + Wr * frvol[j];
      dn = dn + Wr * fmass[j];
      if (r > T(0)) {
        T wg = s_Wg_q(k, qh);
        T Xj = q.w;
        T wg2 = wg * wg;
        a2 = a2 + wg2 * (Xj * Xj) / fmass[j];
      }
    }
  });
  W[i] = w;
  comp[i] = cp;
  dens[i] = dn;
  alpha_1[i] = V4<T>{T(0), T(0), T(0), T(0)};
  alpha_2[i] = a2;
  T al = T(0) / bmass[i] + a2;
  if (al < T(1e-4)) al = T(1e-4);
  alpha[i] = al;
  T psi = k.solver == TSPH_VFSPH ? cp : dn;
  vol[i] = p.w / psi;
}

template <class T>
__global__ void __launch_bounds__(kBlock)
    k_pass_a_bound(KP<T> k, int nb, const V4<T>* __restrict__ bpos, const T* __restrict__ bmass,
                   const T* __restrict__ brvol, const int* __restrict__ bstart,
                   const V4<T>* __restrict__ fpos, const T* __restrict__ fmass,
                   const T* __restrict__ frvol, const int* __restrict__ fstart,
                   T* __restrict__ W, T* __restrict__ comp, T* __restrict__ dens,
                   V4<T>* __restrict__ alpha_1, T* __restrict__ alpha_2, T* __restrict__ alpha,
                   T* __restrict__ vol, V4<T>* __restrict__ ss, int kept) {
  k_pass_a_bound_body<T, false>(Blk{(int)blockIdx.x, (int)gridDim.x}, k, nb, bpos, bmass, brvol, bstart, fpos, fmass, frvol, fstart, W, comp, dens, alpha_1, alpha_2, alpha, vol, ss, kept != 0);
}

// Pass A of the boundary, a quad of lanes per particle (walk_quad): the sums
// of k_pass_a_bound_body, each in walk order.
template <class T>
__device__ __forceinline__ void pass_a_quad_bound(int sub, const KP<T>& k, const TsphObject& f,
                                                  const TsphObject& b, bool kept, WalkLds& lds) {
  TSPH_STRICT
  const int i = coop_particle<kQuad>(sub), c = coop_lane<kQuad>();
  if (i >= b.n) return;
  const V4<T>* __restrict__ bpos = (const V4<T>*)b.pos;
  const V4<T>* __restrict__ fpos = (const V4<T>*)f.pos;
  V4<T>* ss = (V4<T>*)b.static_sums;
  const V4<T> p = bpos[i];
  const T mi = ((const T*)b.mass)[i];
  T w = 0, cp = 0, dn = 0, a2 = 0;
  if (ss != nullptr && kept) {
    const V4<T> s0 = ss[i];
    w = s0.x;
    cp = s0.y;
    dn = s0.z;
  } else {
    const T* __restrict__ bm = (const T*)b.mass;
    const T* __restrict__ bv = (const T*)b.rest_volume;
    walk_quad(k, b.cell_start, bpos, p, lds,
              [&](int j) { return BoundRec<T>{bpos[j], bv[j], bm[j]}; },
              [&](const BoundRec<T>& r, int, bool valid, bool) {
                TSPH_STRICT
                const T d = s_sqrt(s_r2(p.x - r.q.x, p.y - r.q.y, p.z - r.q.z));
                const T Wr = s_W_q_sel(k, d / k.h);
                w = quad_add(w, valid ? Wr : T(0));
                cp = quad_add(cp, valid ? Wr * r.v : T(0));
                dn = quad_add(dn, valid ? Wr * r.m : T(0));
              });
    if (ss != nullptr && c == 0) ss[i] = V4<T>{w, cp, dn, T(0)};
  }
  if (f.n > 0) {
    const T* __restrict__ fm = (const T*)f.mass;
    const T* __restrict__ fv = (const T*)f.rest_volume;
    walk_quad(k, f.cell_start, fpos, p, lds,
              [&](int j) { return BoundRec<T>{fpos[j], fv[j], fm[j]}; },
              [&](const BoundRec<T>& r, int, bool valid, bool apart) {
                TSPH_STRICT
                const T d = s_sqrt(s_r2(p.x - r.q.x, p.y - r.q.y, p.z - r.q.z));
                const T qh = d / k.h;
                const T Wr = s_W_q_sel(k, qh);
                w = quad_add(w, valid ? Wr : T(0));
                cp = quad_add(cp, valid ? Wr * r.v : T(0));
                dn = quad_add(dn, valid ? Wr * r.m : T(0));
                const T wg = s_Wg_q(k, qh);
                const T Xj = r.q.w;
                const T wg2 = wg * wg;
                a2 = quad_add(a2, valid && apart ? wg2 * (Xj * Xj) / r.m : T(0));
              });
  }
  if (c != 0) return;
  ((T*)b.W)[i] = w;
  ((T*)b.sph_compression)[i] = cp;
  ((T*)b.sph_density)[i] = dn;
  ((V4<T>*)b.alpha_1)[i] = V4<T>{T(0), T(0), T(0), T(0)};
  ((T*)b.alpha_2)[i] = a2;
  T al = T(0) / mi + a2;
  if (al < T(1e-4)) al = T(1e-4);
  ((T*)b.alpha)[i] = al;
  const T psi = k.solver == TSPH_VFSPH ? cp : dn;
  ((T*)b.vol)[i] = p.w / psi;
}

// Pass A of both objects by quads, for small scenes.  One lane per particle
// walks its 200 or so candidates one trip after the other: that chain takes
// 65 us however few the particles (8,000: 125 waves on 1,024 SIMDs), and the
// quads cut it to a quarter.  They spend more instructions per candidate (the
// votes and the list in LDS), so once the chip is full the single lanes win.
// us per launch, one lane / quads: 3D FP32 8k 71 / 30, 64k 72 / 39, 133k 78 /
// 67, 149k 80 / 73, 195k 82 / 85, 1M 238 / 368; FP64 8k 87 / 32, 64k 91 / 66,
// 97k 105 / 89, 195k 130 / 156; 2D FP32 8k 24 / 17, 78k 24.8 / 23.1, 102k
// 25.5 / 26, FP64 70k 26.8 / 25.6.
// A boundary particle counts by a half: its walk over its own object, which the
// sums kept from an earlier step replace (then by a sixteenth).  Fluid + boundary,
// us, one lane / quads, sums formed and kept: 3D FP32 8k + 213k 72 / 53 and 67 /
// 25, 8k + 283k 72 / 67, 64k + 166k 69 / 70 and 66 / 41, 64k + 283k 71 / 88 and
// 68 / 46, 97k + 94k 69 / 66 and 69 / 51, 97k + 596k 105 / 157 and 72 / 69, 125k +
// 283k 87 / 110 and 71 / 68; FP64 8k + 124k 83 / 64 and 84 / 28, 64k + 94k 87 / 96
// and 86 / 67, 64k + 387k 127 / 197 and 91 / 89, 64k + 596k 167 / 268 and 92 / 104.
// 2D FP32 8k + 134k 21.3 / 21.8 and 16.1 / 10.2, 40k + 134k 22.5 / 26.1 and 17.9 /
// 14.4.  In 2D with FP64 the single lanes' short chain counts least: 8k + 42k
// 20.9 / 17.2 and 18.7 / 12.0, 8k + 86k 23.6 / 26.9, 40k + 42k 26.0 / 28.6 and 21.0 /
// 19.0, 40k + 86k 25.9 / 36.7 and 21.5 / 21.0, 40k + 134k 29 / 48 and 22.4 / 24.4.
template <class T>
static bool pass_a_by_quads(int dim, const TsphObject& f, const TsphObject& b) {
  const bool kept = b.static_sums != nullptr && (b.flags & TSPH_OBJ_STATIC_SUMS);
  const bool flat64 = dim == 2 && sizeof(T) == 8;
  const long most = flat64 ? 70 * 1024 : dim == 2 ? 80 * 1024 : sizeof(T) == 4 ? 144 * 1024 : 96 * 1024;
  const int share = kept ? (flat64 ? 4 : 16) : (flat64 ? 1 : 2);
  return f.n > 0 && f.n + (long)b.n / share <= most;
}
template <class T>
__global__ void __launch_bounds__(kBlock)
    k_pass_a_quad(KP<T> k, TsphObject f, TsphObject b, int nbf, V4<T>* a1b, TsphControl* ctrl) {
  __shared__ WalkLds lds;
  if ((int)blockIdx.x < nbf) {
    const int sub = coop_sub(Blk{(int)blockIdx.x, nbf});
    pass_a_fluid_variant(k, [&](auto fq, auto xm) {
      pass_a_quad_fluid<T, decltype(fq)::value, decltype(xm)::value>(sub, k, f, b, a1b, ctrl, lds);
    });
  } else {
    pass_a_quad_bound<T>(coop_sub(Blk{(int)blockIdx.x - nbf, (int)gridDim.x - nbf}), k, f, b,
                         (b.flags & TSPH_OBJ_STATIC_SUMS) != 0, lds);
  }
}

__global__ void k_step_reset(TsphControl* ctrl) { step_reset_body(ctrl); }

// Pass A of both objects in one launch: blocks [0, nbf) run the fluid body,
// the rest the boundary body.  The two halves are independent (each writes
// only its own object's fields), so the boundary blocks fill the tail of the
// fluid's grid instead of waiting for it.
template <class T>
__device__ __forceinline__ void pass_a_both_body(const KP<T>& k, const TsphObject& f,
                                                 const TsphObject& b, int nbf, V4<T>* a1b,
                                                 TsphControl* ctrl, int* stage) {
  if ((int)blockIdx.x < nbf) {
    pass_a_fluid_variant(k, [&](auto fq, auto xm) {
      k_pass_a_fluid_body<T, decltype(fq)::value, decltype(xm)::value>(
          Blk{(int)blockIdx.x, nbf}, k, f.n, f.capacity, (const V4<T>*)f.pos, (const T*)f.mass,
          (const T*)f.rest_volume, f.cell_start, b.n, (const V4<T>*)b.pos, (const T*)b.mass,
          (const T*)b.rest_volume, b.cell_start, (T*)f.W, (T*)f.sph_compression,
          (T*)f.sph_density, (V4<T>*)f.alpha_1, (T*)f.alpha_2, (T*)f.alpha, (T*)f.vol,
          (const V4<T>*)f.vel, (V4<T>*)f.vel_adv, f.nbr_f, f.nbr_b, f.nbr_nf, f.nbr_nb, f.flag,
          a1b, ctrl, stage);
    });
  } else {
    k_pass_a_bound_body<T, false>(Blk{(int)blockIdx.x - nbf, (int)gridDim.x - nbf}, k, b.n,
                               (const V4<T>*)b.pos, (const T*)b.mass, (const T*)b.rest_volume,
                               b.cell_start, (const V4<T>*)f.pos, (const T*)f.mass,
                               (const T*)f.rest_volume, f.cell_start, (T*)b.W,
                               (T*)b.sph_compression, (T*)b.sph_density, (V4<T>*)b.alpha_1,
                               (T*)b.alpha_2, (T*)b.alpha, (T*)b.vol, (V4<T>*)b.static_sums,
                               (b.flags & TSPH_OBJ_STATIC_SUMS) != 0);
  }
}
template <class T>
__global__ void __launch_bounds__(kBlock)
    k_pass_a_both(KP<T> k, TsphObject f, TsphObject b, int nbf, V4<T>* a1b, TsphControl* ctrl) {
  __shared__ int stage[kPassAK * kBlock];
  pass_a_both_body<T>(k, f, b, nbf, a1b, ctrl, stage);
}

// The check behind TSPH_FLAG_FAST_QUOTIENT: for every FP32 r^2 in
// [0, r2_max] (bit patterns 0 .. umax), the reduced and the IEEE sequences
// are compared on W(q) and r > 0 (out[0]: inputs that differ, out[2]: the
// largest such bit pattern) and on W'(q) (out[1]).  Each wave adds its
// counts once.
__global__ void __launch_bounds__(kBlock) k_verify_fast_quotient(KP<float> k, uint32_t umax, int* out) {
  int bad = 0, badg = 0;
  uint32_t last = 0;
  const uint32_t stride = gridDim.x * kBlock;
  for (uint32_t u = blockIdx.x * kBlock + threadIdx.x; u <= umax; u += stride) {
    const float x = __uint_as_float(u);
    float rs, ws, gs;
    {
      TSPH_STRICT
      rs = s_sqrt(x);
      const float qs = rs / k.h;
      ws = s_W_q(k, qs);
      gs = s_Wg_q(k, qs);
    }
    const float rf = f_sqrt_cr(x);
    const float qf = f_quot_h(rf, k.h, k.inv_h);
    const float wf = s_W_q(k, qf), gf = s_Wg_q(k, qf);
    const bool dw = (__float_as_uint(ws) != __float_as_uint(wf)) || ((rs > 0.0f) != (rf > 0.0f));
    bad += dw;
    badg += __float_as_uint(gs) != __float_as_uint(gf);
    if (dw) last = u;
  }
  for (int o = 32; o > 0; o >>= 1) {
    bad += __shfl_xor(bad, o, 64);
    badg += __shfl_xor(badg, o, 64);
    last = max(last, (uint32_t)__shfl_xor((int)last, o, 64));
  }
  if ((threadIdx.x & 63) == 0) {
    if (bad) atomicAdd(out, bad);
    if (badg) atomicAdd(out + 1, badg);
    if (last) atomicMax((unsigned int*)(out + 2), last);
  }
}

__global__ void k_fill3_i32(int* p, int v0, int v1, int v2) {
  p[0] = v0;
  p[1] = v1;
  p[2] = v2;
}

int verify_fast_quotient(const TsphParams& prm, int* out, hipStream_t st) {
  if (prm.precision != 4) {
    hipLaunchKernelGGL(k_fill3_i32, dim3(1), dim3(1), 0, st, out, 1, 1, 0);
    TSPH_LAUNCH_CHECK("verify_fast_quotient");
    return 0;
  }
  KP<float> k = make_kp<float>(prm);
  uint32_t umax;
  std::memcpy(&umax, &k.r2max, sizeof(umax));
  TSPH_REQUIRE(k.r2max >= 0.0f && umax < 0x7f800000u, TSPH_EINVAL,
               "tsph_verify_fast_quotient: r2_max is not a finite non-negative value");
  hipLaunchKernelGGL(k_fill3_i32, dim3(1), dim3(1), 0, st, out, 0, 0, 0);
  hipLaunchKernelGGL(k_verify_fast_quotient, dim3(8192), dim3(kBlock), 0, st, k, umax, out);
  TSPH_LAUNCH_CHECK("verify_fast_quotient");
  return 0;
}

template <class T>
__global__ void k_solver_begin(KP<T> k, TsphControl* ctrl, int solve, int* signal, int token) {
  solver_begin_body(k, ctrl, solve, signal, token);
}

// Jacobi half-step P: IPPE_adv_psi_init + IPPE_adv_psi (f,f)(f,b) +
// IPPE_psi_adv_non_negative (sph.py:196-226) for iteration kk of the solve.
template <class T, int R = 1, bool GROUP = false>
__device__ __forceinline__ void k_solver_psi_body(Blk blk, const KP<T>& k, int n, int cap, int kk, const V4<T>* __restrict__ fpos,
                 const V4<T>* __restrict__ vadv, const T* __restrict__ psi_rho,
                 const T* __restrict__ rdens, const T* __restrict__ alpha,
                 const int* __restrict__ fstart, const V4<T>* __restrict__ bpos,
                 const int* __restrict__ bstart, const int* __restrict__ nbr_f,
                 const int* __restrict__ nbr_b, const int* __restrict__ nbr_nf,
                 const int* __restrict__ nbr_nb, T* __restrict__ psi_adv, T* __restrict__ kappa,
                 V4<T>* __restrict__ krec, const V4<T>* __restrict__ a1b,
                 V4<T>* __restrict__ tape_v, T* __restrict__ tape_k,
                 const T* __restrict__ clamp_ref,
                 double* __restrict__ partial, TsphControl* ctrl) {
  __shared__ double lds[R][kWaves];
  if (!ctrl->run_u[kk]) return;
  const int c = coop_lane<kCoop>();
  const T dt = (T)ctrl->dt;
#pragma unroll 1
  for (int r = 0; r < R; ++r) {
    const int i = coop_particle<kCoop>(coop_sub<R>(blk, r));
    double err = 0;
    if (i < n) {
      const V4<T> p = fpos[i];
      const V4<T> va = vadv[i];
      // the particle's own fields, requested before the walk so that their
      // latency hides behind it
      const V4<T> B = a1b[i];
      const T rp = rest_psi_of(k, rdens, i);
      const T pr = psi_rho[i];
      const T al = alpha[i];
      T sum = 0;  // this lane's share of sum_j X_j (v_i - v_j) . grad W_ij
      auto term = [&](const Rec2<T>& d, bool ok) {
        const V4<T>& q = d.a;
        const V4<T>& vj = d.b;
        T dx = p.x - q.x, dy = p.y - q.y, dz = p.z - q.z;
        T r2 = dx * dx + dy * dy + dz * dz, r;
        T g = f_grad(k, r2, &r);
        T dot = (dx * (va.x - vj.x) + dy * (va.y - vj.y) + dz * (va.z - vj.z)) * g;
        const T with = sum + dot * q.w;
        sum = ok ? with : sum;  // (no zero times X_j: it may be infinite)
      };
      // (f,f) pairs from the list; the (f,b) pairs have v_j = 0 (boundary
      // vel_adv is never written), so their sum is v_i . sum_b X_j grad W_ij,
      // the boundary share of alpha_1 that pass A recorded
      sweep_lists_coop<kCoop, T, Rec2<T>, GROUP ? group_nb<T, Rec2<T>, R>(3) : kCoopNb,
                     GROUP ? group_nb<T, Rec2<T>, R>(2) : kCoopNb>(
          k, cap, i, c, p, fstart, bstart, fpos, bpos, nbr_f, nullptr, nbr_nf[i], 0,
          [&](int j) { return Rec2<T>{fpos[j], vadv[j]}; },
          [&](int) { return Rec2<T>{}; }, term, [&](const Rec2<T>&, bool) {});
      sum = group_sum<kCoop>(sum);
      if (c == 0) {
        sum += va.x * B.x + va.y * B.y + va.z * B.z;
        T psi = (pr - rp) + sum * dt;
        // IPPE_psi_adv_non_negative (sph.py:219-226); with a clamp reference, the
        // clamp set of a recorded iteration instead (psi clamped exactly where the
        // recorded kappa is 0): the path whose derivative the adjoint takes
        if (clamp_ref ? clamp_ref[i] == T(0) : psi < T(0)) psi = T(0);
        psi_adv[i] = psi;
        const T kap = psi / al;
        kappa[i] = kap;
        krec[i] = V4<T>{p.x, p.y, p.z, kap};  // the record the update sweep gathers
        if (tape_v) {  // record the iteration for the adjoint
          tape_v[i] = va;
          tape_k[i] = kap;
        }
        err += (double)(psi / rp);
      }
    }
    err = wave_sum(err);
    if ((threadIdx.x & 63) == 0) lds[r][threadIdx.x >> 6] = err;
  }
  // one partial per sub-tile, in storage order
  __syncthreads();
  if (threadIdx.x < R) {
    double s = 0;
    for (int w = 0; w < kWaves; ++w) s += lds[threadIdx.x][w];
    partial[coop_sub<R>(blk, threadIdx.x)] = s;
  }
  __syncthreads();  // lds is free again for a grid-stride block's next tile
}

template <class T>
__global__ void __launch_bounds__(kBlock)
    k_solver_psi(KP<T> k, int n, int cap, int kk, const V4<T>* __restrict__ fpos,
                 const V4<T>* __restrict__ vadv, const T* __restrict__ psi_rho,
                 const T* __restrict__ rdens, const T* __restrict__ alpha,
                 const int* __restrict__ fstart, const V4<T>* __restrict__ bpos,
                 const int* __restrict__ bstart, const int* __restrict__ nbr_f,
                 const int* __restrict__ nbr_b, const int* __restrict__ nbr_nf,
                 const int* __restrict__ nbr_nb, T* __restrict__ psi_adv, T* __restrict__ kappa,
                 V4<T>* __restrict__ krec, const V4<T>* __restrict__ a1b,
                 V4<T>* __restrict__ tape_v, T* __restrict__ tape_k,
                 const T* __restrict__ clamp_ref,
                 double* __restrict__ partial, TsphControl* ctrl, int ahead) {
  const int run = ctrl->run_u[kk], go = ctrl->go;  // in flight together
  if (!run || (ahead && !go)) return;
  k_solver_psi_body<T>(Blk{(int)blockIdx.x, (int)gridDim.x}, k, n, cap, kk, fpos, vadv, psi_rho, rdens, alpha, fstart, bpos, bstart, nbr_f, nbr_b, nbr_nf, nbr_nb, psi_adv, kappa, krec, a1b, tape_v, tape_k, clamp_ref, partial, ctrl);
}

// Jacobi half-step U: IPPE_update_vel_adv (f,f)(f,b) (sph.py:229-244), with
// kappa = psi_adv / alpha formed once per particle.  Block 0 also finishes
// iteration kk's compression and takes the loop decision for iteration kk+1.
//
// The pair coefficient of a fluid neighbour is kappa_i X_j + kappa_j X_i, of
// a boundary neighbour kappa_i X_j (boundary kappa is never written: 0).
// Summed over all neighbours, the kappa_i X_j halves are kappa_i times
// alpha_1 = sum_j X_j grad W_ij of pass A (positions and X do not change
// within the step), so the sweep only visits the fluid list, gathering the
// one record (x_j, kappa_j) that the psi half-step wrote.
template <class T, int R = 1, bool GROUP = false>
__device__ __forceinline__ void k_solver_update_body(Blk blk, const KP<T>& k, int n, int cap, int kk, const V4<T>* __restrict__ fpos,
                    const T* __restrict__ fmass, const T* __restrict__ kappa,
                    const V4<T>* __restrict__ krec, const V4<T>* __restrict__ alpha_1,
                    const int* __restrict__ fstart, const V4<T>* __restrict__ bpos,
                    const int* __restrict__ bstart, const int* __restrict__ nbr_f,
                    const int* __restrict__ nbr_b, const int* __restrict__ nbr_nf,
                    const int* __restrict__ nbr_nb, V4<T>* __restrict__ vadv,
                    const double* __restrict__ partial, TsphControl* ctrl) {
  __shared__ double lds[kWaves];
  if (!ctrl->run_u[kk]) return;
  if (blk.b == 0) {
    // IPPE_psi_adv_non_negative's 0-D reduction (sph.py:221-226) and the loop
    // test of main.py:201-213 / 222-234
    double tot = sum_partials(partial, coop_blocks<kCoop>(n), lds);
    if (threadIdx.x == 0) {
      TSPH_STRICT
      T comp = (T)tot / (T)n;
      ctrl->compression = (double)comp;
      int solve = ctrl->solve;
      if (solve == 0) ctrl->err_div[kk] = (double)comp;
      else ctrl->err_incom[kk] = (double)comp;
      int it = kk + 1;
      ctrl->it = it;
      if (solve == 0) ctrl->div_iter = it;
      else ctrl->incom_iter = it;
      T thr = solve == 0 ? k.div_thr : k.comp_thr;
      bool cont = (it < k.iter_min) || (comp > thr);
      bool run = it <= k.iter_max && cont && it < TSPH_MAX_ITER_LOG;
      if (it < TSPH_MAX_ITER_LOG) ctrl->run_u[it] = run ? 1 : 0;
      ctrl->stop = run ? 0 : 1;
      if (ctrl->signal) {  // early stop signal to the host: one 64-bit system-scope store
        const uint64_t w = ((uint64_t)(uint32_t)ctrl->token << 32) | (uint32_t)(2 * it + (run ? 0 : 1));
        __hip_atomic_store((uint64_t*)(uintptr_t)ctrl->signal, w, __ATOMIC_RELAXED,
                           __HIP_MEMORY_SCOPE_SYSTEM);
      }
    }
  }
  const int cl = coop_lane<kCoopU>();
  const T dt = (T)ctrl->dt;
#pragma unroll 1
  for (int r = 0; r < R; ++r) {
    const int i = coop_particle<kCoopU>(coop_sub<R>(blk, r));
    if (i >= n) break;
    const V4<T> p = fpos[i];
    const T Xi = p.w;
    T sx = 0, sy = 0, sz = 0;  // this lane's share of sum_j kappa_j grad W_ij
    auto term = [&](const V4<T>& q, bool ok) {  // q = (x_j, kappa_j)
      T dx = p.x - q.x, dy = p.y - q.y, dz = p.z - q.z;
      T r2 = dx * dx + dy * dy + dz * dz, r;
      T g = f_grad(k, r2, &r);
      T s = ok ? q.w * g : T(0);
      sx += s * dx;
      sy += s * dy;
      sz += s * dz;
    };
    sweep_lists_coop<kCoopU, T, V4<T>, GROUP ? group_nb<T, V4<T>, R>(3) : kCoopNb,
                     GROUP ? group_nb<T, V4<T>, R>(2) : kCoopNb>(
        k, cap, i, cl, p, fstart, bstart, fpos, bpos, nbr_f, nullptr, nbr_nf[i], 0,
        [&](int j) { return krec[j]; }, [&](int) { return V4<T>{}; }, term,
        [&](const V4<T>&, bool) {});
    sx = group_sum<kCoopU>(sx);
    sy = group_sum<kCoopU>(sy);
    sz = group_sum<kCoopU>(sz);
    if (cl != 0) continue;
    V4<T> va = vadv[i];
    const T ki = kappa[i];
    const T c = -(T(1) / dt) / fmass[i];
    const V4<T> A = alpha_1[i];
    const T cA = c * ki, cX = c * Xi;
    va.x += cA * A.x + cX * sx;
    va.y += cA * A.y + cX * sy;
    va.z += cA * A.z + cX * sz;
    vadv[i] = va;
  }
}

template <class T>
__global__ void __launch_bounds__(kBlock)
    k_solver_update(KP<T> k, int n, int cap, int kk, const V4<T>* __restrict__ fpos,
                    const T* __restrict__ fmass, const T* __restrict__ kappa,
                    const V4<T>* __restrict__ krec, const V4<T>* __restrict__ alpha_1,
                    const int* __restrict__ fstart, const V4<T>* __restrict__ bpos,
                    const int* __restrict__ bstart, const int* __restrict__ nbr_f,
                    const int* __restrict__ nbr_b, const int* __restrict__ nbr_nf,
                    const int* __restrict__ nbr_nb, V4<T>* __restrict__ vadv,
                    const double* __restrict__ partial, TsphControl* ctrl, int ahead) {
  const int run = ctrl->run_u[kk], go = ctrl->go;  // in flight together
  if (!run || (ahead && !go)) return;
  k_solver_update_body<T>(Blk{(int)blockIdx.x, (int)gridDim.x}, k, n, cap, kk, fpos, fmass, kappa, krec, alpha_1, fstart, bpos, bstart, nbr_f, nbr_b, nbr_nf, nbr_nb, vadv, partial, ctrl);
}

// ---------------------------------------------------------------------------
// Advection: SPH_vel_adv_2_vel, gravity, viscosity (f,f), surface-tension
// normals (f,f).  Neighbour velocities are read from vel_adv, so this sweep
// must not write vel_adv: the update vel_adv = vel + dt * acce_adv happens in
// the next kernel (k_surface_tension).
// ---------------------------------------------------------------------------
template <class T, bool GROUP = false>
__device__ __forceinline__ void k_advect_body(Blk blk, const KP<T>& k, int n, int cap, const V4<T>* __restrict__ fpos, const T* __restrict__ vf,
             const T* __restrict__ rdens, const int* __restrict__ fstart,
             const int* __restrict__ bstart, const V4<T>* __restrict__ bpos,
             const int* __restrict__ nbr_f, const int* __restrict__ nbr_nf,
             V4<T>* __restrict__ vadv, V4<T>* __restrict__ vel, V4<T>* __restrict__ acce_adv,
             V4<T>* __restrict__ normal, const T* __restrict__ fmass,
             const T* __restrict__ psi_rho, V4<T>* __restrict__ strec) {
  const int c = coop_lane<kCoop>();
  const int i = coop_particle<kCoop>(coop_sub(blk));
  if (i >= n) return;
  const V4<T> p = fpos[i];
  const V4<T> vi = vadv[i];
  const T fvis = k.two_d2 * mu_of(k, vf, i) / rdens[i];
  T ax = 0, ay = 0, az = 0, nx = 0, ny = 0, nz = 0;  // this lane's share
  auto term = [&](const Rec2<T>& d, bool ok) {
    const V4<T>& q = d.a;
    const V4<T>& vj = d.b;
    T Vj = vj.w;  // V_j = X_j / sph_psi_j rides in vel_adv's 4th lane (pass A)
    T dx = p.x - q.x, dy = p.y - q.y, dz = p.z - q.z;
    T r2 = dx * dx + dy * dy + dz * dz, r;
    T g = f_grad(k, r2, &r);
    T Ax = (vi.x - vj.x) * dx + (vi.y - vj.y) * dy + (vi.z - vj.z) * dz;
    T s = fvis * Vj * g * Ax * f_rcp(k.eps + r2);  // W_lap, sph_util.py:40-43 (fast quotient)
    s = ok ? s : T(0);
    ax += s * dx;
    ay += s * dy;
    az += s * dz;
    T t = ok ? -Vj * g : T(0);  // normal, sph.py:149
    nx += t * dx;
    ny += t * dy;
    nz += t * dz;
  };
  // viscosity and normals are (f,f) only: the boundary list is not visited
  sweep_lists_coop<kCoop, T, Rec2<T>, GROUP ? group_nb<T, Rec2<T>, 1>(3) : kCoopNb,
                     GROUP ? group_nb<T, Rec2<T>, 1>(2) : kCoopNb>(
      k, cap, i, c, p, fstart, bstart, fpos, bpos, nbr_f, nullptr, nbr_nf[i], 0,
      [&](int j) { return Rec2<T>{fpos[j], vadv[j]}; },
      [&](int j) { return Rec2<T>{}; }, term, [&](const Rec2<T>&, bool) {});
  ax = group_sum<kCoop>(ax);
  ay = group_sum<kCoop>(ay);
  az = group_sum<kCoop>(az);
  nx = group_sum<kCoop>(nx);
  ny = group_sum<kCoop>(ny);
  nz = group_sum<kCoop>(nz);
  if (c != 0) return;
  // SPH_vel_adv_2_vel; the spare lane keeps V_i until the tail writes 0:
  // the adjoint's tape of this velocity carries it to the reverse sweep
  vel[i] = vi;
  acce_adv[i] = V4<T>{k.g[0] + ax, k.g[1] + ay, k.g[2] + az, T(0)};
  if (k.gamma != T(0) || k.st_rec) {
    // the records the surface-tension walks gather per candidate j: the
    // normal's spare lane carries +-psi_j, negative where j's 0.99 gate
    // fails (psi_j > 0 for every particle in a cell: its own W(0) term),
    // and the forward walk's (x_j, m_j) goes to strec, so that it loads two
    // records instead of five
    const T psi = psi_rho[i];
    normal[i] = V4<T>{nx * k.h, ny * k.h, nz * k.h, vf[(long)i * k.P] > T(0.99) ? psi : -psi};
    strec[i] = V4<T>{p.x, p.y, p.z, fmass[i]};
  } else {
    normal[i] = V4<T>{nx * k.h, ny * k.h, nz * k.h, T(0)};
  }
}

template <class T>
__global__ void __launch_bounds__(kBlock)
    k_advect(KP<T> k, int n, int cap, const V4<T>* __restrict__ fpos, const T* __restrict__ vf,
             const T* __restrict__ rdens, const int* __restrict__ fstart,
             const int* __restrict__ bstart, const V4<T>* __restrict__ bpos,
             const int* __restrict__ nbr_f, const int* __restrict__ nbr_nf,
             V4<T>* __restrict__ vadv, V4<T>* __restrict__ vel, V4<T>* __restrict__ acce_adv,
             V4<T>* __restrict__ normal, const T* __restrict__ fmass,
             const T* __restrict__ psi_rho, V4<T>* __restrict__ strec, TsphControl* ctrl, int after) {
  const bool go = may_go(ctrl, after);
  if (blockIdx.x == 0 && threadIdx.x == 0) ctrl->go = go;
  if (!go) return;
  k_advect_body<T>(Blk{(int)blockIdx.x, (int)gridDim.x}, k, n, cap, fpos, vf, rdens, fstart, bstart, bpos, nbr_f, nbr_nf, vadv, vel, acce_adv, normal, fmass, psi_rho, strec);
}

// Surface tension loop 2 (sph.py:151-166) + SPH_advection_update_vel_adv
// (sph.py:247-250).  The curvature term carries no kernel weight, so every
// candidate of the neighbouring cells contributes to it: that part walks the
// cells, gathering only the normal record.  Its r > 0 test is j != i: two
// distinct particles at one position have bit-equal normals (their neighbour
// sums run over the same particles in the same order), so their curvature
// term is an exact zero either way.  The cohesion term's C(r) vanishes
// beyond h, so it is summed over the in-range list.  Both terms share the
// factor 2 psi_0 / (psi_i + psi_j) and gamma.  With gamma == 0 every term is
// an exact zero and only the update runs.
// A quad of lanes per particle, kStFwdU gathers in flight per lane: a row run
// holds about 24 candidates, one trip of six.  us, one lane with 8 in flight /
// quads with 2, 3, 4, 6, 7, 8: 4k 29 / 14.3, 12.4, 13.4, 11.8, 12.5, 12.3; 200k
// 50 / 52, 50, 57, 46, 49, 54; 2M 246 / 259, 244, 276, 229, 245, 266.
// (Dropping the terms of a candidate that is left out, instead of multiplying
// them by zero, costs 1 us at 200k and 8 at 2M.)
constexpr int kStFwdU = 6;
// One lane per particle (st_one_lane) has kStOneU in flight; eight of the walk and the
// list raise the registers of the grouped kernel.
constexpr int kStOneU = 4;
// One particle, by L lanes: a quad, or one lane in a quad's order (the same sums
// bit for bit, so that a scene's own launch and a grouped one may differ in it).
template <class T, int L>
__device__ __forceinline__ void st_particle(int i, const KP<T>& k, int cap,
                      const V4<T>* __restrict__ fpos, const T* __restrict__ psi_rho,
                      const T* __restrict__ rdens, const T* __restrict__ vf,
                      const int* __restrict__ fstart, const V4<T>* __restrict__ normal,
                      const V4<T>* __restrict__ strec, const int* __restrict__ nbr_f,
                      const int* __restrict__ nbr_nf, const V4<T>* __restrict__ vel,
                      V4<T>* __restrict__ acce_adv, V4<T>* __restrict__ vadv, T dt) {
  const int cl = coop_lane<L>();
  V4<T> a = acce_adv[i];
  if (vf[(long)i * k.P] > T(0.99)) {
    V4<T> p = fpos[i];
    V4<T> ni = normal[i];
    T rp = rest_psi_of(k, rdens, i);
    T psi_i = psi_rho[i];
    int c[3];
    node_encode(k, p.x, p.y, p.z, c);
    // the normal record's spare lane holds +-psi_j, negative where j's 0.99
    // gate fails (the advection sweep writes it).  Reciprocal square root
    // and reciprocals instead of the IEEE forms: the pair terms of these
    // sums are not part of the bit-exact sums.
    constexpr int S = L == 1 ? kQuad : 1;  // partial sums per lane
    T ux[S], uy[S], uz[S];                 // sums of (n_i - n_j) / (psi_i + psi_j)
#pragma unroll
    for (int u = 0; u < S; ++u) ux[u] = uy[u] = uz[u] = T(0);
    auto curv = [&](int u, int j, const V4<T>& nj, bool valid) {
      // a candidate left out may hold anything: its terms are dropped, not
      // multiplied by zero
      const bool on = valid && j != i && nj.w > T(0);
      const T w = f_rcp(psi_i + nj.w);
      ux[u] += on ? w * (ni.x - nj.x) : T(0);
      uy[u] += on ? w * (ni.y - nj.y) : T(0);
      uz[u] += on ? w * (ni.z - nj.z) : T(0);
    };
    auto loadn = [&](int j) { return normal[j]; };
    // per in-range neighbour: (x_j, m_j) and the normal record
    auto load = [&](int j) { return Rec2<T>{strec[j], normal[j]}; };
    auto coh = [&](int u, const Rec2<T>& d, bool ok) {  // - m_j C(r) x_ij / r / (psi_i + psi_j)
      const V4<T>& q = d.a;
      const T dx = p.x - q.x, dy = p.y - q.y, dz = p.z - q.z;
      const T r2 = dx * dx + dy * dy + dz * dz;
      const T rinv = f_rsqrt(r2);
      T s = q.w * f_coh(k, r2 * rinv * k.inv_h) * rinv * f_rcp(psi_i + d.b.w);
      s = ok && d.b.w > T(0) ? s : T(0);
      ux[u] -= s * dx;
      uy[u] -= s * dy;
      uz[u] -= s * dz;
    };
    T sx, sy, sz;
    if constexpr (L == 1) {
      walk_as_quad<kStOneU>(k, fstart, c, loadn, curv);
      sweep_list_as_quad<Rec2<T>, kQuad>(k, cap, i, p, c, fstart, fpos, nbr_f, nbr_nf[i], load,
                                         coh);
      sx = (ux[0] + ux[1]) + (ux[2] + ux[3]);
      sy = (uy[0] + uy[1]) + (uy[2] + uy[3]);
      sz = (uz[0] + uz[1]) + (uz[2] + uz[3]);
    } else {
      walk_quad_all<kStFwdU>(k, fstart, c, loadn, [&](int j, const V4<T>& nj, bool valid) {
        curv(0, j, nj, valid);
      });
      sweep_lists_coop<kQuad, T, Rec2<T>>(
          k, cap, i, cl, p, fstart, nullptr, fpos, nullptr, nbr_f, nullptr, nbr_nf[i], 0, load,
          load, [&](const Rec2<T>& d, bool ok) { coh(0, d, ok); }, [&](const Rec2<T>&, bool) {});
      sx = group_sum<kQuad>(ux[0]);
      sy = group_sum<kQuad>(uy[0]);
      sz = group_sum<kQuad>(uz[0]);
    }
    // 2 psi_0 / (psi_i + psi_j) (cohesion + curvature), cohesion =
    // -gamma m_j C(r) x_ij / r, curvature = gamma (n_i - n_j)
    const T f = T(2) * rp * k.gamma;
    a.x += f * sx;
    a.y += f * sy;
    a.z += f * sz;
    if (cl == 0) acce_adv[i] = a;
  }
  if (cl != 0) return;
  {
    TSPH_STRICT  // SPH_advection_update_vel_adv, sph.py:247-250
    const V4<T> v = vel[i];
    vadv[i] = V4<T>{v.x + a.x * dt, v.y + a.y * dt, v.z + a.z * dt, T(0)};
  }
}

// A block's particles: with a quad each the sub-tile of 64 (blk counts sub-tiles),
// with one lane each the tile of 256 (blk counts tiles).
template <class T, int L>
__device__ __forceinline__ void k_surface_tension_body(Blk blk, const KP<T>& k, int n, int cap,
                      const V4<T>* __restrict__ fpos, const T* __restrict__ psi_rho,
                      const T* __restrict__ rdens, const T* __restrict__ vf,
                      const int* __restrict__ fstart, const V4<T>* __restrict__ normal,
                      const V4<T>* __restrict__ strec, const int* __restrict__ nbr_f,
                      const int* __restrict__ nbr_nf, const V4<T>* __restrict__ vel,
                      V4<T>* __restrict__ acce_adv, V4<T>* __restrict__ vadv,
                      const TsphControl* ctrl) {
  const T dt = (T)ctrl->dt;
  const int i = coop_particle<L>(coop_sub(blk));
  if (i < n)
    st_particle<T, L>(i, k, cap, fpos, psi_rho, rdens, vf, fstart, normal, strec, nbr_f, nbr_nf,
                      vel, acce_adv, vadv, dt);
}
// vel_adv = vel + dt acce_adv alone, of a scene without surface tension in a grouped
// launch: a tile of 256 particles.
template <class T>
__device__ __forceinline__ void st_update_only(Blk blk, int n, const V4<T>* __restrict__ vel,
                                               const V4<T>* __restrict__ acce_adv,
                                               V4<T>* __restrict__ vadv, const TsphControl* ctrl) {
  TSPH_STRICT
  const int i = xcd_block(blk.b, blk.nb) * kBlock + (int)threadIdx.x;
  if (i >= n) return;
  const T dt = (T)ctrl->dt;
  const V4<T> v = vel[i], a = acce_adv[i];
  vadv[i] = V4<T>{v.x + a.x * dt, v.y + a.y * dt, v.z + a.z * dt, T(0)};
}

// SPH_advection_update_vel_adv alone (sph.py:247-250), for gamma = 0: a
// separate kernel, so that it runs at the occupancy of an elementwise kernel
// rather than at that of the surface-tension walk.
template <class T>
__global__ void __launch_bounds__(kBlock)
    k_vel_adv_update(KP<T> k, int n, const V4<T>* __restrict__ vel,
                     const V4<T>* __restrict__ acce_adv, V4<T>* __restrict__ vadv,
                     TsphControl* ctrl, SolveOpen open) {
  TSPH_STRICT
  if (open.ahead && !ctrl->go) return;
  if (open.on && blockIdx.x == 0) solver_begin_body(k, ctrl, 1, (int*)open.signal, open.token);
  const int i = xcd_block(blockIdx.x, gridDim.x) * kBlock + threadIdx.x;
  if (i >= n) return;
  const T dt = (T)ctrl->dt;
  const V4<T> a = acce_adv[i], v = vel[i];
  vadv[i] = V4<T>{v.x + a.x * dt, v.y + a.y * dt, v.z + a.z * dt, T(0)};
}

template <class T, int L>
__global__ void __launch_bounds__(kBlock, sizeof(T) == 4 ? 7 : 1)  // 72 registers, not 75
    k_surface_tension(KP<T> k, int n, int cap, const V4<T>* __restrict__ fpos,
                      const T* __restrict__ psi_rho,
                      const T* __restrict__ rdens, const T* __restrict__ vf,
                      const int* __restrict__ fstart, const V4<T>* __restrict__ normal,
                      const V4<T>* __restrict__ strec, const int* __restrict__ nbr_f,
                      const int* __restrict__ nbr_nf, const V4<T>* __restrict__ vel,
                      V4<T>* __restrict__ acce_adv, V4<T>* __restrict__ vadv,
                      TsphControl* ctrl, SolveOpen open) {
  if (open.ahead && !ctrl->go) return;
  if (open.on && blockIdx.x == 0) solver_begin_body(k, ctrl, 1, (int*)open.signal, open.token);
  k_surface_tension_body<T, L>(Blk{(int)blockIdx.x, (int)gridDim.x}, k, n, cap, fpos, psi_rho, rdens, vf, fstart, normal, strec, nbr_f, nbr_nf, vel, acce_adv, vadv, ctrl);
}

// ---------------------------------------------------------------------------
// FBM round (sph.py:301-372), predicated on ctrl->general_flag.
// ---------------------------------------------------------------------------
template <class T>
__global__ void __launch_bounds__(kBlock)
    k_fbm_drift(KP<T> k, int n, const V4<T>* __restrict__ vadv, const V4<T>* __restrict__ vel,
                const T* __restrict__ rdens, const T* __restrict__ vf, V4<T>* __restrict__ acce_adv,
                V4<T>* __restrict__ acce, T* __restrict__ zeta, V4<T>* __restrict__ drift,
                T* __restrict__ tmp, const int* __restrict__ flag, TsphControl* ctrl, int after) {
  TSPH_STRICT
  if (!fbm_may_go(ctrl, after)) return;
  if (blockIdx.x == 0 && threadIdx.x == 0) ctrl->fbm_rounds += 1;
  int i = xcd_block(blockIdx.x, gridDim.x) * kBlock + threadIdx.x;
  if (i >= n) return;
  const T dt = (T)ctrl->dt;
  const int P = k.P;
  for (int q = 0; q < P; ++q) tmp[(long)i * P + q] = T(0);  // SPH_FBM_clean_tmp
  V4<T> va = vadv[i], v = vel[i];
  T aa[3] = {(va.x - v.x) / dt, (va.y - v.y) / dt, (va.z - v.z) / dt};
  T rd = rdens[i];
  T z = T(0);
  for (int q = 0; q < P; ++q) z = z + vf[(long)i * P + q] * (k.rho[q] - rd) / k.rho[q];
  T fa[3];
  for (int d = 0; d < 3; ++d) fa[d] = (aa[d] - z * k.g[d]) / (T(1) - z);
  acce_adv[i] = V4<T>{aa[0], aa[1], aa[2], T(0)};
  acce[i] = V4<T>{fa[0], fa[1], fa[2], T(0)};
  zeta[i] = z;
  for (int q = 0; q < P; ++q) {
    T phi = vf[(long)i * P + q];
    T s = phi * (k.rho[q] - rd);
    T u[3];
    for (int d = 0; d < 3; ++d) u[d] = s * (k.g[d] - fa[d]);
    T wgt = phi * k.rho[q];
    if (wgt > T(1e-6)) {
      for (int d = 0; d < 3; ++d) u[d] = u[d] / wgt;
    } else {
      for (int d = 0; d < 3; ++d) u[d] = u[d] * T(0);
    }
    for (int d = 0; d < 3; ++d) u[d] = (u[d] + (fa[d] - aa[d])) * dt;
    if (k.dim == 2) u[2] = T(0);
    // the spare lane carries what the cooperative flux sweep gathers of this
    // particle besides its drift: phi_q, or -1 once the particle is flagged
    // (sph.py:366-372; the flags of this round are those of the last check)
    drift[(long)i * P + q] = V4<T>{u[0], u[1], u[2], flag[i] != 0 ? T(-1) : phi};
  }
}

template <class T>
__global__ void __launch_bounds__(kBlock)
    k_fbm_flux(KP<T> k, int n, int cap, const V4<T>* __restrict__ fpos,
               const T* __restrict__ rvol, const T* __restrict__ vf,
               const V4<T>* __restrict__ drift, const int* __restrict__ flag,
               const int* __restrict__ fstart, const int* __restrict__ nbr_f_in,
               const int* __restrict__ nbr_nf, T* __restrict__ tmp, const TsphControl* ctrl, int after) {
  TSPH_STRICT
  if (!fbm_may_go(ctrl, after)) return;
  int i = xcd_block(blockIdx.x, gridDim.x) * kBlock + threadIdx.x;
  if (i >= n || flag[i] != 0) return;
  const int* nbr_f = nbr_f_in;
  const T dt = (T)ctrl->dt;
  const int P = k.P;
  V4<T> p = fpos[i];
  T acc[kMaxP];
  for (int q = 0; q < P; ++q) acc[q] = tmp[(long)i * P + q];
  const T pre_c = k.fbmC * dt;
  const T pre_d = dt * k.fbmD;
  int nf = nbr_nf[i];
  // SPH_FBM_convect loop 2 (sph.py:346-363)
  for_fluid_nbrs(k, i, cap, nf, nbr_f, fstart, fpos, p, [&](int j) {
    if (flag[j] != 0) return;
    V4<T> q = fpos[j];
    T dx = p.x - q.x, dy = p.y - q.y, dz = p.z - q.z;
    T r = s_sqrt(s_r2(dx, dy, dz));
    T wg = s_Wg(k, r);
    T ex = dx / r, ey = dy / r, ez = dz / r;
    T Vj = rvol[j];
    for (int s = 0; s < P; ++s) {
      V4<T> ui = drift[(long)i * P + s], uj = drift[(long)j * P + s];
      T pi = vf[(long)i * P + s], pj = vf[(long)j * P + s];
      T fx = pi * ui.x + pj * uj.x, fy = pi * ui.y + pj * uj.y, fz = pi * ui.z + pj * uj.z;
      T dot = fx * ex;
      dot = dot + fy * ey;
      dot = dot + fz * ez;
      T t = pre_c * Vj * dot * wg;
      acc[s] = acc[s] - t;
    }
  });
  // SPH_FBM_diffuse (sph.py:308-326)
  for_fluid_nbrs(k, i, cap, nf, nbr_f, fstart, fpos, p, [&](int j) {
    if (flag[j] != 0) return;
    V4<T> q = fpos[j];
    T dx = p.x - q.x, dy = p.y - q.y, dz = p.z - q.z;
    T r2 = s_r2(dx, dy, dz);
    T r = s_sqrt(r2);
    T wg = s_Wg(k, r);
    T den = r * r + k.eps;
    T Vj = rvol[j];
    for (int s = 0; s < P; ++s) {
      T dphi = vf[(long)i * P + s] - vf[(long)j * P + s];
      T t = pre_d * dphi * Vj * r * wg / den;
      acc[s] = acc[s] + t;
    }
  });
  for (int q = 0; q < P; ++q) tmp[(long)i * P + q] = acc[q];
}

// The same sweep for NP phases as one cooperative list sweep (kCoop lanes
// per particle, gathers in flight as in the solver sweeps).  The pair terms
// of SPH_FBM_convect and SPH_FBM_diffuse share the neighbour's record and
// W'/r (fast arithmetic); their sums are added to tmp in the reference's
// order, convection first.  With W'(r) e = (W'/r) x and r W'(r) = r^2 W'/r,
// the terms are pre_c V_j (f . x) W'/r and pre_d dphi V_j r^2 (W'/r) / (r^2 + eps).
template <class T, int NP>
struct FbmRec {
  V4<T> x;
  V4<T> u[NP];  // drift of each phase, (u, phi) or (u, -1) when flagged (k_fbm_drift)
  T V;
};

template <class T, int NP>
__global__ void __launch_bounds__(kBlock)
    k_fbm_flux_coop(KP<T> k, int n, int cap, const V4<T>* __restrict__ fpos,
                    const T* __restrict__ rvol, const T* __restrict__ vf,
                    const V4<T>* __restrict__ drift, const int* __restrict__ flag,
                    const int* __restrict__ fstart, const int* __restrict__ nbr_f,
                    const int* __restrict__ nbr_nf, T* __restrict__ tmp,
                    const TsphControl* ctrl, int after) {
  if (!fbm_may_go(ctrl, after)) return;
  const int i = coop_particle<kCoop>(coop_sub(Blk{(int)blockIdx.x, (int)gridDim.x}));
  if (i >= n) return;
  const int c = coop_lane<kCoop>();
  const T dt = (T)ctrl->dt;
  if (flag[i] != 0) return;  // the whole group: one particle
  const V4<T> p = fpos[i];
  V4<T> ui[NP];
  T pi[NP], conv[NP], diff[NP];
#pragma unroll
  for (int s = 0; s < NP; ++s) {
    ui[s] = drift[(long)i * NP + s];
    pi[s] = vf[(long)i * NP + s];
    conv[s] = T(0);
    diff[s] = T(0);
  }
  // VFSPH: the position's alias lane is the rest volume (no extra gather)
  const bool vx = k.solver == TSPH_VFSPH;
  auto load = [&](int j) {
    FbmRec<T, NP> d;
    d.x = fpos[j];
#pragma unroll
    for (int s = 0; s < NP; ++s) d.u[s] = drift[(long)j * NP + s];
    d.V = vx ? d.x.w : rvol[j];
    return d;
  };
  auto pair = [&](const FbmRec<T, NP>& d, bool ok) {
    if (!ok || d.u[0].w < T(0)) return;  // no neighbour, or a flagged one
    const T dx = p.x - d.x.x, dy = p.y - d.x.y, dz = p.z - d.x.z;
    const T r2 = dx * dx + dy * dy + dz * dz;
    T r;
    const T g = f_grad(k, r2, &r);
    const T gv = g * d.V;
    const T gd = gv * r2 * f_rcp(r2 + k.eps);
#pragma unroll
    for (int s = 0; s < NP; ++s) {
      const T pj = d.u[s].w;
      const T fx = pi[s] * ui[s].x + pj * d.u[s].x;
      const T fy = pi[s] * ui[s].y + pj * d.u[s].y;
      const T fz = pi[s] * ui[s].z + pj * d.u[s].z;
      conv[s] += (fx * dx + fy * dy + fz * dz) * gv;
      diff[s] += (pi[s] - pj) * gd;
    }
  };
  sweep_lists_coop<kCoop, T, FbmRec<T, NP>>(
      k, cap, i, c, p, fstart, fstart, fpos, fpos, nbr_f, nullptr, nbr_nf[i], 0, load, load,
      pair, [&](const FbmRec<T, NP>&, bool) {});
#pragma unroll
  for (int s = 0; s < NP; ++s) {
    conv[s] = group_sum<kCoop>(conv[s]);
    diff[s] = group_sum<kCoop>(diff[s]);
  }
  if (c != 0) return;
  const T pre_c = k.fbmC * dt, pre_d = dt * k.fbmD;
#pragma unroll
  for (int s = 0; s < NP; ++s) {
    T a = tmp[(long)i * NP + s];
    a = a - pre_c * conv[s];
    a = a + pre_d * diff[s];
    tmp[(long)i * NP + s] = a;
  }
}

template <class T>
__global__ void __launch_bounds__(kBlock)
    k_fbm_check(KP<T> k, int n, const T* __restrict__ vf, const T* __restrict__ tmp,
                int* __restrict__ flag, double* __restrict__ partial, TsphControl* ctrl, int after) {
  TSPH_STRICT
  __shared__ double lds[kWaves];
  if (!fbm_may_go(ctrl, after)) return;
  int nblk = gridDim.x;
  int i = xcd_block(blockIdx.x, nblk) * kBlock + threadIdx.x;
  double any = 0;
  if (i < n) {
    bool neg = false;  // has_negative, sph_util.py:56-62
    for (int q = 0; q < k.P; ++q)
      if (vf[(long)i * k.P + q] + tmp[(long)i * k.P + q] < T(0)) neg = true;
    if (neg) {
      flag[i] = 1;
      any = 1;
    }
  }
  double s = block_sum(any, lds);
  if (threadIdx.x == 0) partial[blockIdx.x] = s;
}

// general_flag = any particle flagged this round (sph.py:368-372); skipped,
// like the round itself, once the flag is clear.
// With a signal, the flag and the rounds that ran also go to the host:
// (token << 32) | (2 rounds + flag).
__global__ void __launch_bounds__(kBlock)
    k_fbm_check_finish(const double* __restrict__ partial, int nblk, TsphControl* ctrl,
                       uint64_t* signal, int token, int after) {
  __shared__ double lds[kWaves];
  int flag = 0;
  if (after && !(ctrl->go && may_go(ctrl, after))) return;
  if (ctrl->general_flag) {
    double a = sum_partials(partial, nblk, lds);
    if (threadIdx.x == 0) ctrl->general_flag = flag = a > 0 ? 1 : 0;
  }
  if (signal && threadIdx.x == 0)
    __hip_atomic_store(signal, ((uint64_t)(uint32_t)token << 32) | (uint32_t)(2 * ctrl->fbm_rounds + flag),
                       __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

// ---------------------------------------------------------------------------
// Tail: [SPH_update_volume_frac], SPH_update_mass, SPH_update_pos,
// SPH_update_energy (sph.py:265-286, 375-379).
// ---------------------------------------------------------------------------
template <class T>
__device__ __forceinline__ void k_tail_body(Blk blk, const KP<T>& k, int n, int fbm, V4<T>* __restrict__ pos, V4<T>* __restrict__ vel,
           const V4<T>* __restrict__ vadv, T* __restrict__ mass, T* __restrict__ rdens,
           const T* __restrict__ rvol, T* __restrict__ vf, const T* __restrict__ tmp,
           const int* __restrict__ flag, double* __restrict__ partial, TsphControl* ctrl) {
  TSPH_STRICT
  __shared__ double lds[kWaves];
  int nblk = blk.nb;
  int i = xcd_block(blk.b, nblk) * kBlock + threadIdx.x;
  const T dt = (T)ctrl->dt;
  double ke = 0, pe = 0;
  if (i < n) {
    const int P = k.P;
    if (fbm && !(flag[i] > 0))
      for (int q = 0; q < P; ++q) vf[(long)i * P + q] = vf[(long)i * P + q] + tmp[(long)i * P + q];
    T rd = k.rho[0] * vf[(long)i * P];
    for (int q = 1; q < P; ++q) rd = rd + k.rho[q] * vf[(long)i * P + q];
    T m = rd * rvol[i];
    rdens[i] = rd;
    mass[i] = m;
    V4<T> v = vadv[i];
    V4<T> p = pos[i];
    p.x = p.x + v.x * dt;
    p.y = p.y + v.y * dt;
    p.z = p.z + v.z * dt;
    p.w = k.solver == TSPH_VFSPH ? rvol[i] : m;
    pos[i] = p;
    vel[i] = V4<T>{v.x, v.y, v.z, T(0)};
    T n2 = s_r2(v.x, v.y, v.z);
    ke = (double)(T(0.5) * m * n2);
    pe = (double)(-m * k.g[1] * (p.y - k.lb[1]));
  }
  double s1 = block_sum(ke, lds);
  double s2 = block_sum(pe, lds);
  if (threadIdx.x == 0) {
    partial[blk.b] = s1;
    partial[nblk + blk.b] = s2;
  }
}

template <class T>
__global__ void __launch_bounds__(kBlock)
    k_tail(KP<T> k, int n, int fbm, V4<T>* __restrict__ pos, V4<T>* __restrict__ vel,
           const V4<T>* __restrict__ vadv, T* __restrict__ mass, T* __restrict__ rdens,
           const T* __restrict__ rvol, T* __restrict__ vf, const T* __restrict__ tmp,
           const int* __restrict__ flag, double* __restrict__ partial, TsphControl* ctrl, int after) {
  if (!tail_may_go(ctrl, after, fbm)) return;
  k_tail_body<T>(Blk{(int)blockIdx.x, (int)gridDim.x}, k, n, fbm, pos, vel, vadv, mass, rdens, rvol, vf, tmp, flag, partial, ctrl);
}

// ---------------------------------------------------------------------------
// Host launchers.
// ---------------------------------------------------------------------------
template <class T>
static int pass_a(const TsphParams& prm, TsphObject* f, TsphObject* b, TsphControl* ctrl,
                  bool with_bound, const WsLayout& L, bool opened, hipStream_t st) {
  KP<T> k = make_kp<T>(prm);
  if (!opened) hipLaunchKernelGGL(k_step_reset, dim3(1), dim3(64), 0, st, ctrl);
  if (with_bound && pass_a_by_quads<T>(prm.dim, *f, *b)) {
    const int nbf = coop_blocks<kQuad>(f->n);
    hipLaunchKernelGGL(k_pass_a_quad<T>, dim3(nbf + (b->n > 0 ? coop_blocks<kQuad>(b->n) : 0)),
                       dim3(kBlock), 0, st, k, *f, *b, nbf, (V4<T>*)L.a1b, ctrl);
    TSPH_LAUNCH_CHECK("density_alpha");
    if (b->n > 0 && b->static_sums) b->flags |= TSPH_OBJ_STATIC_SUMS;
    return 0;
  }
  if (with_bound && f->n > 0 && b->n > 0) {
    const int nbf = blocks_for(f->n);
    hipLaunchKernelGGL(k_pass_a_both<T>, dim3(nbf + blocks_for(b->n)), dim3(kBlock), 0, st, k, *f,
                       *b, nbf, (V4<T>*)L.a1b, ctrl);
    TSPH_LAUNCH_CHECK("density_alpha");
    if (b->static_sums) b->flags |= TSPH_OBJ_STATIC_SUMS;  // stream order: later launches read them
    return 0;
  }
  if (f->n > 0)
    hipLaunchKernelGGL(k_pass_a_fluid<T>, dim3(blocks_for(f->n)), dim3(kBlock), 0, st, k, f->n,
                       f->capacity, (const V4<T>*)f->pos, (const T*)f->mass,
                       (const T*)f->rest_volume, f->cell_start, b->n, (const V4<T>*)b->pos,
                       (const T*)b->mass, (const T*)b->rest_volume, b->cell_start, (T*)f->W,
                       (T*)f->sph_compression, (T*)f->sph_density, (V4<T>*)f->alpha_1,
                       (T*)f->alpha_2, (T*)f->alpha, (T*)f->vol, (const V4<T>*)f->vel,
                       (V4<T>*)f->vel_adv, f->nbr_f, f->nbr_b, f->nbr_nf, f->nbr_nb, f->flag,
                       (V4<T>*)L.a1b, ctrl);
  if (with_bound && b->n > 0)
    hipLaunchKernelGGL(k_pass_a_bound<T>, dim3(blocks_for(b->n)), dim3(kBlock), 0, st, k, b->n,
                       (const V4<T>*)b->pos, (const T*)b->mass, (const T*)b->rest_volume,
                       b->cell_start, (const V4<T>*)f->pos, (const T*)f->mass,
                       (const T*)f->rest_volume, f->cell_start, (T*)b->W, (T*)b->sph_compression,
                       (T*)b->sph_density, (V4<T>*)b->alpha_1, (T*)b->alpha_2, (T*)b->alpha,
                       (T*)b->vol, (V4<T>*)b->static_sums, b->flags & TSPH_OBJ_STATIC_SUMS);
  TSPH_LAUNCH_CHECK("density_alpha");
  if (with_bound && b->n > 0 && b->static_sums) b->flags |= TSPH_OBJ_STATIC_SUMS;
  return 0;
}

template <class T>
int density_alpha(const TsphParams& prm, TsphObject* f, TsphObject* b, TsphControl* ctrl,
                  void* ws, size_t wsb, bool opened, hipStream_t st) {
  WsLayout L;
  TSPH_REQUIRE(carve_ws(ws, wsb, f->capacity, prm.node_num, &L), TSPH_ECAPACITY,
               "tsph_density_alpha: workspace too small");
  return pass_a<T>(prm, f, b, ctrl, true, L, opened, st);
}

// The fluid's neighbour lists alone, as pass A builds them (8 candidates in
// flight: without pass A's pair math the walk is bound by the gathers): in-range
// candidates with r > 0 (r^2 > 0) in walk order.  The counters are updated
// without branches (per-branch increments get merged into an indexed
// increment of a stack array).
constexpr int kListsU = 8;
template <class T>
__global__ void __launch_bounds__(kBlock)
    k_lists(KP<T> k, int n, int cap, const V4<T>* __restrict__ fpos, const int* __restrict__ fstart,
            const V4<T>* __restrict__ bpos, const int* __restrict__ bstart, int* __restrict__ nbr_f,
            int* __restrict__ nbr_b, int* __restrict__ nbr_nf, int* __restrict__ nbr_nb,
            TsphControl* ctrl) {
  const int i = xcd_block(blockIdx.x, gridDim.x) * kBlock + threadIdx.x;
  if (i >= n) return;
  const int capf = k.list_cap_f, capb = k.list_cap_b;
  const V4<T> p = fpos[i];
  int c[3];
  node_encode(k, p.x, p.y, p.z, c);
  int nf = 0, nbb = 0;
  walk_cells_batched<kListsU>(k, fstart, c, fpos, [&](int j, const V4<T>& q) {
    const T r2 = s_r2(p.x - q.x, p.y - q.y, p.z - q.z);
    const bool take = r2 <= k.r2max && r2 > T(0);
    if (take && nf < capf) nbr_f[(long)nf * cap + i] = j;
    nf += take ? 1 : 0;
  });
  walk_cells_batched<kListsU>(k, bstart, c, bpos, [&](int j, const V4<T>& q) {
    const T r2 = s_r2(p.x - q.x, p.y - q.y, p.z - q.z);
    const bool take = r2 <= k.r2max && r2 > T(0);
    if (take && nbb < capb) nbr_b[(long)nbb * cap + i] = j;
    nbb += take ? 1 : 0;
  });
  if (nf > capf) {
    atomicAdd(&ctrl->overflow_f, 1);
    nf = capf + 1;
  }
  if (nbb > capb) {
    atomicAdd(&ctrl->overflow_b, 1);
    nbb = capb + 1;
  }
  nbr_nf[i] = nf;
  nbr_nb[i] = nbb;
}

// Rebuilds the fluid's neighbour lists from recorded sorted positions and
// cell table.  The adjoint recomputes per-step lists this way when it does
// not store them (it stores the step's densities and alpha factors).
template <class T>
int relist(const TsphParams& prm, TsphObject* f, TsphObject* b, TsphControl* ctrl, void* ws,
           size_t wsb, hipStream_t st) {
  (void)ws;
  (void)wsb;
  KP<T> k = make_kp<T>(prm);
  if (f->n == 0) return 0;
  hipLaunchKernelGGL(k_lists<T>, dim3(blocks_for(f->n)), dim3(kBlock), 0, st, k, f->n, f->capacity,
                     (const V4<T>*)f->pos, f->cell_start, (const V4<T>*)b->pos, b->cell_start,
                     f->nbr_f, f->nbr_b, f->nbr_nf, f->nbr_nb, ctrl);
  TSPH_LAUNCH_CHECK("relist");
  return 0;
}

template <class T>
int solver_begin(const TsphParams& prm, TsphControl* ctrl, int solve, int* signal, int token,
                 hipStream_t st) {
  KP<T> k = make_kp<T>(prm);
  hipLaunchKernelGGL(k_solver_begin<T>, dim3(1), dim3(kBlock), 0, st, k, ctrl, solve, signal,
                     token);
  TSPH_LAUNCH_CHECK("solver_begin");
  return 0;
}

template <class T>
int solver_half(const TsphParams& prm, TsphObject* f, TsphObject* b, TsphControl* ctrl, int kk,
                int half, void* tape_v, void* tape_k, const void* clamp_ref, void* ws, size_t wsb,
                int ahead, hipStream_t st) {
  KP<T> k = make_kp<T>(prm);
  WsLayout L;
  TSPH_REQUIRE(carve_ws(ws, wsb, f->capacity, prm.node_num, &L), TSPH_ECAPACITY,
               "tsph_solver_iteration: workspace too small");
  // With no fluid particles one block still runs the stop rule: the mean of
  // an empty sum is 0/0 = NaN, as in the reference (sph.py:221-226), so the
  // solve runs its minimum iteration count.
  const T* psi = (const T*)(prm.solver_type == TSPH_VFSPH ? f->sph_compression : f->sph_density);
  if (half & 1)
    hipLaunchKernelGGL(k_solver_psi<T>, dim3(coop_blocks<kCoop>(f->n)), dim3(kBlock), 0, st, k,
                       f->n, f->capacity, kk, (const V4<T>*)f->pos, (const V4<T>*)f->vel_adv, psi,
                       (const T*)f->rest_density, (const T*)f->alpha, f->cell_start,
                       (const V4<T>*)b->pos, b->cell_start, f->nbr_f, f->nbr_b, f->nbr_nf,
                       f->nbr_nb, (T*)f->psi_adv, (T*)f->kappa, (V4<T>*)L.krec,
                       (const V4<T>*)L.a1b, (V4<T>*)tape_v, (T*)tape_k, (const T*)clamp_ref,
                       L.partial, ctrl, ahead);
  if (half & 2)
    hipLaunchKernelGGL(k_solver_update<T>, dim3(coop_blocks<kCoopU>(f->n)), dim3(kBlock), 0, st,
                       k, f->n, f->capacity, kk, (const V4<T>*)f->pos, (const T*)f->mass, (const T*)f->kappa,
                       (const V4<T>*)L.krec, (const V4<T>*)f->alpha_1, f->cell_start, (const V4<T>*)b->pos, b->cell_start, f->nbr_f, f->nbr_b,
                       f->nbr_nf, f->nbr_nb, (V4<T>*)f->vel_adv, L.partial, ctrl, ahead);
  TSPH_LAUNCH_CHECK("solver_iteration");
  return 0;
}

template <class T>
int advect(const TsphParams& prm, TsphObject* f, TsphObject* b, TsphControl* ctrl, void* ws,
           size_t wsb, SolveOpen open, hipStream_t st) {
  KP<T> k = make_kp<T>(prm);
  WsLayout L;
  TSPH_REQUIRE(carve_ws(ws, wsb, f->capacity, prm.node_num, &L), TSPH_ECAPACITY,
               "tsph_advect: workspace too small");
  if (f->n == 0) return 0;
  int nb = blocks_for(f->n);
  const T* psi = (const T*)(prm.solver_type == TSPH_VFSPH ? f->sph_compression : f->sph_density);
  hipLaunchKernelGGL(k_advect<T>, dim3(coop_blocks<kCoop>(f->n)), dim3(kBlock), 0, st, k, f->n,
                     f->capacity, (const V4<T>*)f->pos, (const T*)f->volume_frac, (const T*)f->rest_density,
                     f->cell_start, b->cell_start, (const V4<T>*)b->pos, f->nbr_f, f->nbr_nf,
                     (V4<T>*)f->vel_adv, (V4<T>*)f->vel, (V4<T>*)f->acce_adv,
                     (V4<T>*)f->normal, (const T*)f->mass, psi, (V4<T>*)L.krec, ctrl, open.ahead);
  if (k.gamma == T(0))
    hipLaunchKernelGGL(k_vel_adv_update<T>, dim3(nb), dim3(kBlock), 0, st, k, f->n,
                       (const V4<T>*)f->vel, (const V4<T>*)f->acce_adv, (V4<T>*)f->vel_adv, ctrl,
                       open);
  else {
    auto tension = [&](auto kern, int blocks) {
      hipLaunchKernelGGL(kern, dim3(blocks), dim3(kBlock), 0, st, k, f->n, f->capacity,
                         (const V4<T>*)f->pos, psi, (const T*)f->rest_density,
                         (const T*)f->volume_frac, f->cell_start, (const V4<T>*)f->normal,
                         (const V4<T>*)L.krec, f->nbr_f, f->nbr_nf, (const V4<T>*)f->vel,
                         (V4<T>*)f->acce_adv, (V4<T>*)f->vel_adv, ctrl, open);
    };
    if (st_one_lane(prm.dim, f->n))
      tension(k_surface_tension<T, 1>, nb);
    else
      tension(k_surface_tension<T, kQuad>, coop_blocks<kQuad>(f->n));
  }
  TSPH_LAUNCH_CHECK("advect");
  return 0;
}

template <class T>
int fbm_round(const TsphParams& prm, TsphObject* f, TsphControl* ctrl, void* ws, size_t wsb,
              uint64_t* signal, int token, int after, hipStream_t st) {
  KP<T> k = make_kp<T>(prm);
  WsLayout L;
  TSPH_REQUIRE(carve_ws(ws, wsb, f->capacity, prm.node_num, &L), TSPH_ECAPACITY,
               "tsph_fbm_round: workspace too small");
  if (f->n == 0) return 0;
  int nb = blocks_for(f->n);
  hipLaunchKernelGGL(k_fbm_drift<T>, dim3(nb), dim3(kBlock), 0, st, k, f->n,
                     (const V4<T>*)f->vel_adv, (const V4<T>*)f->vel, (const T*)f->rest_density,
                     (const T*)f->volume_frac, (V4<T>*)f->acce_adv, (V4<T>*)f->acce,
                     (T*)f->fbm_zeta, (V4<T>*)f->drift_vel, (T*)f->volume_frac_tmp, f->flag, ctrl,
                     after);
  auto flux = [&](auto kern, int nbk) {
    hipLaunchKernelGGL(kern, dim3(nbk), dim3(kBlock), 0, st, k, f->n, f->capacity,
                       (const V4<T>*)f->pos, (const T*)f->rest_volume, (const T*)f->volume_frac,
                       (const V4<T>*)f->drift_vel, f->flag, f->cell_start, f->nbr_f, f->nbr_nf,
                       (T*)f->volume_frac_tmp, ctrl, after);
  };
  switch (prm.phase_num) {  // the cooperative sweep keeps NP phases' records in registers
    case 1: flux(k_fbm_flux_coop<T, 1>, coop_blocks<kCoop>(f->n)); break;
    case 2: flux(k_fbm_flux_coop<T, 2>, coop_blocks<kCoop>(f->n)); break;
    case 3: flux(k_fbm_flux_coop<T, 3>, coop_blocks<kCoop>(f->n)); break;
    default: flux(k_fbm_flux<T>, nb); break;
  }
  hipLaunchKernelGGL(k_fbm_check<T>, dim3(nb), dim3(kBlock), 0, st, k, f->n,
                     (const T*)f->volume_frac, (const T*)f->volume_frac_tmp, f->flag, L.partial,
                     ctrl, after);
  hipLaunchKernelGGL(k_fbm_check_finish, dim3(1), dim3(kBlock), 0, st, L.partial, nb, ctrl,
                     signal, token, after);
  TSPH_LAUNCH_CHECK("fbm_round");
  return 0;
}

template <class T>
int tail(const TsphParams& prm, TsphObject* f, TsphControl* ctrl, int fbm, void* ws, size_t wsb,
         int after, hipStream_t st) {
  KP<T> k = make_kp<T>(prm);
  WsLayout L;
  TSPH_REQUIRE(carve_ws(ws, wsb, f->capacity, prm.node_num, &L), TSPH_ECAPACITY,
               "tsph_tail: workspace too small");
  int nb = blocks_for(f->n > 0 ? f->n : 1);
  hipLaunchKernelGGL(k_tail<T>, dim3(nb), dim3(kBlock), 0, st, k, f->n, fbm, (V4<T>*)f->pos,
                     (V4<T>*)f->vel, (const V4<T>*)f->vel_adv, (T*)f->mass,
                     (T*)f->rest_density, (const T*)f->rest_volume, (T*)f->volume_frac,
                     (const T*)f->volume_frac_tmp, f->flag, L.partial, ctrl, after);
  hipLaunchKernelGGL(k_finalize<T>, dim3(1), dim3(kBlock), 0, st, k, (int)kFinEnergy, L.partial, nb,
                     f->n, ctrl, after, fbm);
  TSPH_LAUNCH_CHECK("tail");
  return 0;
}

// ---------------------------------------------------------------------------
// WCSPH block (main.py:236-240, commented in the reference's sph_step):
// WC_pressure_val (fluid), WC_pressure_acce (f,f)(f,b) and
// SPH_advection_update_vel_adv.  Boundary pressure is never set by the
// reference (WC_pressure_val runs for the fluid only), so it reads 0.
// Strict arithmetic, the reference's order.
// ---------------------------------------------------------------------------
template <class T>
__global__ void __launch_bounds__(kBlock)
    k_wc_pressure(KP<T> k, int n, const T* __restrict__ dens, const T* __restrict__ rdens,
                  T* __restrict__ pressure) {
  TSPH_STRICT
  int i = xcd_block(blockIdx.x, gridDim.x) * kBlock + threadIdx.x;
  if (i >= n) return;
  // (rho0 * cs^2 / gamma) * ((rho / rho0)^7 - 1), clamped at 0 (sph.py:169-175);
  // the integer power by repeated squaring
  T cs2 = (T)(k.cs * k.cs);
  T ratio = dens[i] / rdens[i];
  T res = T(1), b = ratio;
  int e = 7;
  while (e > 0) {
    if (e & 1) res = res * b;
    b = b * b;
    e >>= 1;
  }
  T pr = (rdens[i] * cs2 / (T)k.wc_gamma) * (res - T(1));
  if (pr < T(0)) pr = T(0);
  pressure[i] = pr;
}

template <class T>
__global__ void __launch_bounds__(kBlock)
    k_wc_acce(KP<T> k, int n, int cap, const V4<T>* __restrict__ fpos, const T* __restrict__ fmass,
              const T* __restrict__ fdens, const T* __restrict__ fpress, const int* __restrict__ fstart,
              const V4<T>* __restrict__ bpos, const T* __restrict__ bmass,
              const T* __restrict__ bdens, const T* __restrict__ bpress,
              const int* __restrict__ bstart, const int* __restrict__ nbr_f,
              const int* __restrict__ nbr_b, const int* __restrict__ nbr_nf,
              const int* __restrict__ nbr_nb, const V4<T>* __restrict__ vel,
              V4<T>* __restrict__ acce_adv, V4<T>* __restrict__ vel_adv,
              const TsphControl* ctrl) {
  TSPH_STRICT
  int i = xcd_block(blockIdx.x, gridDim.x) * kBlock + threadIdx.x;
  if (i >= n) return;
  const V4<T> p = fpos[i];
  V4<T> a = acce_adv[i];
  const T pi = fpress[i], di = fdens[i];
  auto term = [&](const V4<T>& q, T mj, T dj, T pj) {
    T dx = p.x - q.x, dy = p.y - q.y, dz = p.z - q.z;
    T r = s_sqrt(s_r2(dx, dy, dz));
    T pt = pi / (di * di) + pj / (dj * dj);
    T wg = s_Wg(k, r);
    a.x = a.x + -pt * mj * dx / r * wg;
    a.y = a.y + -pt * mj * dy / r * wg;
    if (k.dim == 3) a.z = a.z + -pt * mj * dz / r * wg;
  };
  for_fluid_nbrs(k, i, cap, nbr_nf[i], nbr_f, fstart, fpos, p,
                 [&](int j) { term(fpos[j], fmass[j], fdens[j], fpress[j]); });
  for_bound_nbrs(k, i, cap, nbr_nb[i], nbr_b, bstart, bpos, p,
                 [&](int j) { term(bpos[j], bmass[j], bdens[j], bpress[j]); });
  acce_adv[i] = a;
  const T dt = (T)ctrl->dt;
  const V4<T> v = vel[i];
  vel_adv[i] = V4<T>{v.x + dt * a.x, v.y + dt * a.y, v.z + dt * a.z, T(0)};
}

template <class T>
int wcsph(const TsphParams& prm, TsphObject* f, TsphObject* b, TsphControl* ctrl,
          hipStream_t st) {
  KP<T> k = make_kp<T>(prm);
  if (f->n == 0) return 0;
  int nb = blocks_for(f->n);
  hipLaunchKernelGGL(k_wc_pressure<T>, dim3(nb), dim3(kBlock), 0, st, k, f->n,
                     (const T*)f->sph_density, (const T*)f->rest_density, (T*)f->pressure);
  hipLaunchKernelGGL(k_wc_acce<T>, dim3(nb), dim3(kBlock), 0, st, k, f->n, f->capacity,
                     (const V4<T>*)f->pos, (const T*)f->mass, (const T*)f->sph_density,
                     (const T*)f->pressure, f->cell_start, (const V4<T>*)b->pos,
                     (const T*)b->mass, (const T*)b->sph_density, (const T*)b->pressure,
                     b->cell_start, f->nbr_f, f->nbr_b, f->nbr_nf, f->nbr_nb,
                     (const V4<T>*)f->vel, (V4<T>*)f->acce_adv, (V4<T>*)f->vel_adv, ctrl);
  TSPH_LAUNCH_CHECK("wcsph");
  return 0;
}
template int wcsph<float>(const TsphParams&, TsphObject*, TsphObject*, TsphControl*, hipStream_t);
template int wcsph<double>(const TsphParams&, TsphObject*, TsphObject*, TsphControl*, hipStream_t);

// ---------------------------------------------------------------------------
// map_velocity (sph.py:382-397) over a Grid (sph_obj.py:328-344): one thread
// per grid node (row-major, last axis fastest) at lb + I * dist; the node's
// velocity sums X_j / psi_j * vel_j * W(|x_I - x_j|) over the object's
// candidates in the cells around the node's cell, in template and in-cell
// order (the object's cell table from this step's sort).  Strict arithmetic.
// ---------------------------------------------------------------------------
template <class T>
__global__ void __launch_bounds__(kBlock)
    k_map_velocity(KP<T> k, long total, int g0, int g1, int g2, T dist,
                   const V4<T>* __restrict__ pos, const V4<T>* __restrict__ vel,
                   const T* __restrict__ psi, const int* __restrict__ cstart,
                   V4<T>* __restrict__ out) {
  TSPH_STRICT
  const long idx = (long)blockIdx.x * kBlock + threadIdx.x;
  if (idx >= total) return;
  int I[3] = {0, 0, 0};
  if (k.dim == 3) {
    I[2] = (int)(idx % g2);
    long r = idx / g2;
    I[1] = (int)(r % g1);
    I[0] = (int)(r / g1);
  } else {
    I[1] = (int)(idx % g1);
    I[0] = (int)(idx / g1);
  }
  T gp[3] = {T(0), T(0), T(0)};
  for (int d = 0; d < k.dim; ++d) gp[d] = k.lb[d] + T(I[d]) * dist;
  int c[3];
  node_encode(k, gp[0], gp[1], gp[2], c);
  T vx = 0, vy = 0, vz = 0;
  walk_cells(k, cstart, c, [&](int j) {
    const V4<T> q = pos[j];
    const T w = s_W(k, s_sqrt(s_r2(gp[0] - q.x, gp[1] - q.y, gp[2] - q.z)));
    const T sc = q.w / psi[j];
    const V4<T> v = vel[j];
    vx = vx + (sc * v.x) * w;
    vy = vy + (sc * v.y) * w;
    vz = vz + (sc * v.z) * w;
  });
  out[idx] = V4<T>{vx, vy, vz, T(0)};
}

template <class T>
int map_velocity(const TsphParams& prm, const TsphObject* o, const int* shape, double dist,
                 void* out, hipStream_t st) {
  KP<T> k = make_kp<T>(prm);
  long total = 1;
  for (int d = 0; d < prm.dim; ++d) total *= shape[d];
  if (total <= 0) return 0;
  const T* psi = (const T*)(prm.solver_type == TSPH_VFSPH ? o->sph_compression : o->sph_density);
  hipLaunchKernelGGL(k_map_velocity<T>, dim3((unsigned)((total + kBlock - 1) / kBlock)), dim3(kBlock), 0,
                     st, k, total, shape[0], shape[1], prm.dim == 3 ? shape[2] : 1, (T)dist,
                     (const V4<T>*)o->pos, (const V4<T>*)o->vel, psi, o->cell_start, (V4<T>*)out);
  TSPH_LAUNCH_CHECK("map_velocity");
  return 0;
}
template int map_velocity<float>(const TsphParams&, const TsphObject*, const int*, double, void*, hipStream_t);
template int map_velocity<double>(const TsphParams&, const TsphObject*, const int*, double, void*, hipStream_t);

// ---------------------------------------------------------------------------
// Grouped (batched) launches: the kernels above over every scene of a table
// (tsph_host.h:SceneEntry), with the single-scene launchers' arguments.
// ---------------------------------------------------------------------------
template <class T>
__device__ __forceinline__ const T* psi_of(const SceneEntry<T>& e) {
  return (const T*)(e.k.solver == TSPH_VFSPH ? e.f.sph_compression : e.f.sph_density);
}

template <class T>
__global__ void __launch_bounds__(kBlock) kb_step_reset(const char* __restrict__ tab, int ns) {
  for_tiles<T, kTileScene>(tab, ns, [&](const SceneEntry<T>& e, int, Blk) { step_reset_body(e.ctrl); });
}

// After the grouped boundary pass A: every scene whose boundary has a kept-sum
// buffer now holds its (b,b) sums, so later steps read them (the table's copy
// of TSPH_OBJ_STATIC_SUMS, as tsph_density_alpha sets it in the caller's
// descriptor).  One thread per scene, a vector store into the table; the
// grouped kernels read the table at their next launch.
template <class T>
__global__ void kb_mark_static_sums(char* tab, int ns) {
  const int s = blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= ns) return;
  TsphObject& b = ((SceneEntry<T>*)tab)[s].b;
  if (b.static_sums != nullptr && b.n > 0) b.flags |= TSPH_OBJ_STATIC_SUMS;
}

// Pass A of one fluid tile / one boundary tile of a scene.
template <class T>
__device__ __forceinline__ void pass_a_fluid_tile(const SceneEntry<T>& e, Blk blk, int* stage) {
  const TsphObject& f = e.f;
  const TsphObject& b = e.b;
  pass_a_fluid_variant(e.k, [&](auto fq, auto xm) {
    k_pass_a_fluid_body<T, decltype(fq)::value, decltype(xm)::value>(
        blk, e.k, f.n, f.capacity, (const V4<T>*)f.pos, (const T*)f.mass,
        (const T*)f.rest_volume, f.cell_start, b.n, (const V4<T>*)b.pos, (const T*)b.mass,
        (const T*)b.rest_volume, b.cell_start, (T*)f.W, (T*)f.sph_compression,
        (T*)f.sph_density, (V4<T>*)f.alpha_1, (T*)f.alpha_2, (T*)f.alpha, (T*)f.vol,
        (const V4<T>*)f.vel, (V4<T>*)f.vel_adv, f.nbr_f, f.nbr_b, f.nbr_nf, f.nbr_nb, f.flag,
        (V4<T>*)e.L.a1b, e.ctrl, stage);
  });
}
template <class T>
__device__ __forceinline__ void pass_a_bound_tile(const SceneEntry<T>& e, Blk blk) {
  const TsphObject& f = e.f;
  const TsphObject& b = e.b;
  k_pass_a_bound_body<T, false>(
      blk, e.k, b.n, (const V4<T>*)b.pos, (const T*)b.mass, (const T*)b.rest_volume,
      b.cell_start, (const V4<T>*)f.pos, (const T*)f.mass, (const T*)f.rest_volume,
      f.cell_start, (T*)b.W, (T*)b.sph_compression, (T*)b.sph_density, (V4<T>*)b.alpha_1,
      (T*)b.alpha_2, (T*)b.alpha, (T*)b.vol, (V4<T>*)b.static_sums,
      (b.flags & TSPH_OBJ_STATIC_SUMS) != 0);
}

// Pass A of every scene's fluid and boundary in one grouped launch: tiles
// [0, fluid tiles) are fluid tiles, the rest boundary tiles.  The two
// halves write only their own object's fields, so the boundary tiles fill
// the tail of the fluid tiles' launch instead of waiting for it.
template <class T>
__global__ void __launch_bounds__(kBlock) kb_pass_a_both(const char* __restrict__ tab, int ns) {
  __shared__ int stage[kPassAK * kBlock];
  const int tf = tile_prefix<T, kTileFluid>(tab, ns)[ns];
  const int total = tf + tile_prefix<T, kTileBound>(tab, ns)[ns];
  for (int t = blockIdx.x; t < total; t += gridDim.x) {
    if (t < tf)
      on_tile<T, kTileFluid>(tab, ns, t, [&](const SceneEntry<T>& e, int, Blk blk) {
        pass_a_fluid_tile(e, blk, stage);
      });
    else
      on_tile<T, kTileBound>(tab, ns, t - tf, [&](const SceneEntry<T>& e, int, Blk blk) {
        pass_a_bound_tile(e, blk);
      });
  }
}

template <class T>
__global__ void __launch_bounds__(kBlock)
    kb_solver_begin(const char* __restrict__ tab, int ns, int solve, uint64_t* signal, int token) {
  // scene s's early stop signal goes to signal[s] (no signal when null)
  for_tiles<T, kTileScene>(tab, ns, [&](const SceneEntry<T>& e, int s, Blk) {
    solver_begin_body(e.k, e.ctrl, solve, signal ? (int*)(signal + s) : nullptr, token);
  });
}

template <class T, int R>
__global__ void __launch_bounds__(kBlock, sizeof(T) == 4 ? 5 : 1)  // R = 4: 96 registers, not 99
    kb_solver_psi(const char* __restrict__ tab, int ns, int kk) {
  for_coop_tiles<T, kCoop, R>(tab, ns, [&](const SceneEntry<T>& e, Blk blk) {
    const TsphObject& f = e.f;
    k_solver_psi_body<T, R, true>(blk, e.k, f.n, f.capacity, kk, (const V4<T>*)f.pos,
                         (const V4<T>*)f.vel_adv, psi_of(e), (const T*)f.rest_density,
                         (const T*)f.alpha, f.cell_start, (const V4<T>*)e.b.pos, e.b.cell_start,
                         f.nbr_f, f.nbr_b, f.nbr_nf, f.nbr_nb, (T*)f.psi_adv, (T*)f.kappa,
                         (V4<T>*)e.L.krec, (const V4<T>*)e.L.a1b, (V4<T>*)nullptr, (T*)nullptr,
                         (const T*)nullptr, e.L.partial, e.ctrl);
  });
}

template <class T, int R>
__global__ void __launch_bounds__(kBlock)
    kb_solver_update(const char* __restrict__ tab, int ns, int kk) {
  for_coop_tiles<T, kCoopU, R>(tab, ns, [&](const SceneEntry<T>& e, Blk blk) {
    const TsphObject& f = e.f;
    k_solver_update_body<T, R, true>(blk, e.k, f.n, f.capacity, kk, (const V4<T>*)f.pos,
                            (const T*)f.mass, (const T*)f.kappa, (const V4<T>*)e.L.krec,
                            (const V4<T>*)f.alpha_1, f.cell_start,
                            (const V4<T>*)e.b.pos, e.b.cell_start, f.nbr_f, f.nbr_b, f.nbr_nf,
                            f.nbr_nb, (V4<T>*)f.vel_adv, e.L.partial, e.ctrl);
  });
}

template <class T>
__global__ void __launch_bounds__(kBlock) kb_advect(const char* __restrict__ tab, int ns) {
  for_coop_tiles<T, kCoop, 1>(tab, ns, [&](const SceneEntry<T>& e, Blk blk) {
    const TsphObject& f = e.f;
    k_advect_body<T, true>(blk, e.k, f.n, f.capacity, (const V4<T>*)f.pos, (const T*)f.volume_frac,
                     (const T*)f.rest_density, f.cell_start, e.b.cell_start,
                     (const V4<T>*)e.b.pos, f.nbr_f, f.nbr_nf, (V4<T>*)f.vel_adv, (V4<T>*)f.vel,
                     (V4<T>*)f.acce_adv, (V4<T>*)f.normal, (const T*)f.mass, psi_of(e),
                     (V4<T>*)e.L.krec);
  });
}

// Tiles [0, whole tiles) are whole ones (one lane per particle, or the update alone),
// the rest sub-tiles of a quad each.  Each kind has its own tiles: blocks of a scene's
// sub-tiles that leave its work to every fourth one fill a quarter of the shader engines
// (2D, 2880 tiles: 146 us, and 48).  FP64 is held to 128 registers for four waves per
// SIMD: 3D, 768 tiles 94 us, with 132 registers and three 103; 4608 tiles 531 and 592.
template <class T>
__global__ void __launch_bounds__(kBlock, sizeof(T) == 4 ? 6 : 4)
    kb_surface_tension(const char* __restrict__ tab, int ns) {
  const int tw = tile_prefix<T, kTileWhole>(tab, ns)[ns];
  const int total = tw + tile_prefix<T, kTileQuads>(tab, ns)[ns] * kQuad;
  auto scene = [&](const SceneEntry<T>& e, Blk blk, auto lanes) {
    const TsphObject& f = e.f;
    k_surface_tension_body<T, decltype(lanes)::value>(
        blk, e.k, f.n, f.capacity, (const V4<T>*)f.pos, psi_of(e), (const T*)f.rest_density,
        (const T*)f.volume_frac, f.cell_start, (const V4<T>*)f.normal, (const V4<T>*)e.L.krec,
        f.nbr_f, f.nbr_nf, (const V4<T>*)f.vel, (V4<T>*)f.acce_adv, (V4<T>*)f.vel_adv, e.ctrl);
  };
  for (int t = blockIdx.x; t < total; t += gridDim.x) {
    if (t < tw)
      on_tile<T, kTileWhole>(tab, ns, t, [&](const SceneEntry<T>& e, int, Blk tile) {
        const TsphObject& f = e.f;
        if (e.k.gamma == T(0))
          st_update_only<T>(tile, f.n, (const V4<T>*)f.vel, (const V4<T>*)f.acce_adv,
                            (V4<T>*)f.vel_adv, e.ctrl);
        else
          scene(e, tile, std::integral_constant<int, 1>{});
      });
    else
      on_tile<T, kTileQuads>(tab, ns, (t - tw) / kQuad, [&](const SceneEntry<T>& e, int, Blk tile) {
        scene(e, Blk{tile.b * kQuad + (t - tw) % kQuad, tile.nb * kQuad},
              std::integral_constant<int, kQuad>{});
      });
  }
}

template <class T>
__global__ void __launch_bounds__(kBlock) kb_tail(const char* __restrict__ tab, int ns) {
  for_tiles<T, kTileFluid>(tab, ns, [&](const SceneEntry<T>& e, int, Blk blk) {
    const TsphObject& f = e.f;
    k_tail_body<T>(blk, e.k, f.n, 0, (V4<T>*)f.pos, (V4<T>*)f.vel, (const V4<T>*)f.vel_adv,
                   (T*)f.mass, (T*)f.rest_density, (const T*)f.rest_volume, (T*)f.volume_frac,
                   (const T*)f.volume_frac_tmp, f.flag, e.L.partial, e.ctrl);
  });
}

template <class T>
__global__ void __launch_bounds__(kBlock) kb_finalize_energy(const char* __restrict__ tab, int ns) {
  const int* firstf = (const int*)(tab + batch_entries_bytes<T>(ns)) + kTileFluid * (ns + 1);
  for_tiles<T, kTileScene>(tab, ns, [&](const SceneEntry<T>& e, int s, Blk blk) {
    k_finalize_body<T>(blk, e.k, (int)kFinEnergy, e.L.partial, firstf[s + 1] - firstf[s], e.f.n,
                       e.ctrl);
  });
}

template <class T>
__global__ void kb_stop_state(const char* __restrict__ tab, int ns, int* out) {
  int s = blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= ns) return;
  const TsphControl* c = ((SceneEntry<T>*)tab)[s].ctrl;
  out[2 * s] = c->it;
  out[2 * s + 1] = c->stop;
}

template <class T>
int batch_density_alpha(const TsphBatchInfo& bi, char* tab, int grid, hipStream_t st) {
  const int ns = bi.nscenes;
  hipLaunchKernelGGL(kb_step_reset<T>, dim3(ns), dim3(kBlock), 0, st, tab, ns);
  if (int g = grid_for(bi.tiles[kTileFluid] + bi.tiles[kTileBound], grid))
    hipLaunchKernelGGL(kb_pass_a_both<T>, dim3(g), dim3(kBlock), 0, st, tab, ns);
  if (bi.tiles[kTileBound] > 0)
    hipLaunchKernelGGL(kb_mark_static_sums<T>, dim3((ns + 63) / 64), dim3(64), 0, st, tab, ns);
  TSPH_LAUNCH_CHECK("batch_density_alpha");
  return 0;
}

template <class T>
int batch_solver_begin(const TsphBatchInfo& bi, char* tab, int solve, uint64_t* signal, int token,
                       hipStream_t st) {
  hipLaunchKernelGGL(kb_solver_begin<T>, dim3(bi.nscenes), dim3(kBlock), 0, st, tab, bi.nscenes,
                     solve, signal, token);
  TSPH_LAUNCH_CHECK("batch_solver_begin");
  return 0;
}

template <class T>
int batch_solver_half(const TsphBatchInfo& bi, char* tab, int kk, int half, int grid,
                      hipStream_t st) {
  const int tiles = bi.tiles[kTileFluid];
  if (tiles <= 0) return 0;
  auto launch = [&](auto kern, int blocks) {
    hipLaunchKernelGGL(kern, dim3(grid_for(blocks, grid)), dim3(kBlock), 0, st, tab, bi.nscenes, kk);
  };
  if (half & 1) {
    if (psi_split<T>(tiles)) launch(kb_solver_psi<T, 1>, tiles * kCoop);
    else launch(kb_solver_psi<T, kCoop>, tiles);
  }
  if (half & 2) {
    if (update_split<T>(tiles)) launch(kb_solver_update<T, 1>, tiles * kCoopU);
    else launch(kb_solver_update<T, kCoopU>, tiles);
  }
  TSPH_LAUNCH_CHECK("batch_solver_iteration");
  return 0;
}

template <class T>
int batch_advect(const TsphBatchInfo& bi, char* tab, int grid, hipStream_t st) {
  const int tiles = bi.tiles[kTileFluid];
  if (tiles <= 0) return 0;
  hipLaunchKernelGGL(kb_advect<T>, dim3(grid_for(tiles * kCoop, grid)), dim3(kBlock), 0, st, tab,
                     bi.nscenes);
  hipLaunchKernelGGL(kb_surface_tension<T>, dim3(grid_for(tiles * kQuad, grid)), dim3(kBlock), 0, st,
                     tab, bi.nscenes);
  TSPH_LAUNCH_CHECK("batch_advect");
  return 0;
}

template <class T>
int batch_tail(const TsphBatchInfo& bi, char* tab, int grid, hipStream_t st) {
  const int g = grid_for(bi.tiles[kTileFluid], grid);
  if (g) hipLaunchKernelGGL(kb_tail<T>, dim3(g), dim3(kBlock), 0, st, tab, bi.nscenes);
  hipLaunchKernelGGL(kb_finalize_energy<T>, dim3(bi.nscenes), dim3(kBlock), 0, st, tab, bi.nscenes);
  TSPH_LAUNCH_CHECK("batch_tail");
  return 0;
}

template <class T>
int batch_stop_state(const TsphBatchInfo& bi, char* tab, int* out, hipStream_t st) {
  hipLaunchKernelGGL(kb_stop_state<T>, dim3((bi.nscenes + 63) / 64), dim3(64), 0, st, tab,
                     bi.nscenes, out);
  TSPH_LAUNCH_CHECK("batch_stop_state");
  return 0;
}

#define TSPH_BATCH_INST(T)                                                                  \
  template int batch_density_alpha<T>(const TsphBatchInfo&, char*, int, hipStream_t);      \
  template int batch_solver_begin<T>(const TsphBatchInfo&, char*, int, uint64_t*, int, hipStream_t); \
  template int batch_solver_half<T>(const TsphBatchInfo&, char*, int, int, int, hipStream_t); \
  template int batch_advect<T>(const TsphBatchInfo&, char*, int, hipStream_t);             \
  template int batch_tail<T>(const TsphBatchInfo&, char*, int, hipStream_t);               \
  template int batch_stop_state<T>(const TsphBatchInfo&, char*, int*, hipStream_t);
TSPH_BATCH_INST(float)
TSPH_BATCH_INST(double)
#undef TSPH_BATCH_INST

template int relist<float>(const TsphParams&, TsphObject*, TsphObject*, TsphControl*, void*, size_t, hipStream_t);
template int relist<double>(const TsphParams&, TsphObject*, TsphObject*, TsphControl*, void*, size_t, hipStream_t);
template int density_alpha<float>(const TsphParams&, TsphObject*, TsphObject*, TsphControl*, void*, size_t, bool, hipStream_t);
template int density_alpha<double>(const TsphParams&, TsphObject*, TsphObject*, TsphControl*, void*, size_t, bool, hipStream_t);
template int solver_begin<float>(const TsphParams&, TsphControl*, int, int*, int, hipStream_t);
template int solver_begin<double>(const TsphParams&, TsphControl*, int, int*, int, hipStream_t);
template int solver_half<float>(const TsphParams&, TsphObject*, TsphObject*, TsphControl*, int, int, void*, void*, const void*, void*, size_t, int, hipStream_t);
template int solver_half<double>(const TsphParams&, TsphObject*, TsphObject*, TsphControl*, int, int, void*, void*, const void*, void*, size_t, int, hipStream_t);
template int advect<float>(const TsphParams&, TsphObject*, TsphObject*, TsphControl*, void*, size_t, SolveOpen, hipStream_t);
template int advect<double>(const TsphParams&, TsphObject*, TsphObject*, TsphControl*, void*, size_t, SolveOpen, hipStream_t);
template int fbm_round<float>(const TsphParams&, TsphObject*, TsphControl*, void*, size_t, uint64_t*, int, int, hipStream_t);
template int fbm_round<double>(const TsphParams&, TsphObject*, TsphControl*, void*, size_t, uint64_t*, int, int, hipStream_t);
template int tail<float>(const TsphParams&, TsphObject*, TsphControl*, int, void*, size_t, int, hipStream_t);
template int tail<double>(const TsphParams&, TsphObject*, TsphControl*, int, void*, size_t, int, hipStream_t);

}  // namespace tsph
