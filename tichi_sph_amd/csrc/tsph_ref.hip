// The reference's kernel surface on the GPU: each sph.py kernel with its
// (ngrid, obj, nobj) signature, walking the shared Ngrid
// (node_part_count / node_part_shift / part_pid_in_node / part_uid_in_node,
// sph_obj.py:280-323) with the uid filter, in the reference's order
// (sph.py:9-19).  Strict arithmetic in the reference's evaluation order,
// accumulation into the existing field values.
// These kernels are the drop-in for callers that drive the solver kernel by
// kernel; the fused step (tsph_step.hip) is the fast path.
#include <algorithm>

#include "tsph_sweep.h"

namespace tsph {

struct RefGrid {
  const int *npc, *nps, *pin, *uin;
};

template <class T>
struct RefObj {
  int n, uid;
  V4<T>*pos, *vel, *vel_adv, *acce_adv, *acce, *normal, *alpha_1;
  T *mass, *rest_density, *rest_volume, *vf, *vf_tmp;
  V4<T>* drift;
  T *W, *comp, *dens, *psi_adv, *alpha, *alpha_2, *zeta, *pressure;
  int *flag, *cs;
};

template <class T>
RefObj<T> ref_obj(const TsphObject* o) {
  RefObj<T> r;
  r.n = o->n;
  r.uid = o->uid;
  r.pos = (V4<T>*)o->pos;
  r.vel = (V4<T>*)o->vel;
  r.vel_adv = (V4<T>*)o->vel_adv;
  r.acce_adv = (V4<T>*)o->acce_adv;
  r.acce = (V4<T>*)o->acce;
  r.normal = (V4<T>*)o->normal;
  r.alpha_1 = (V4<T>*)o->alpha_1;
  r.mass = (T*)o->mass;
  r.rest_density = (T*)o->rest_density;
  r.rest_volume = (T*)o->rest_volume;
  r.vf = (T*)o->volume_frac;
  r.vf_tmp = (T*)o->volume_frac_tmp;
  r.drift = (V4<T>*)o->drift_vel;
  r.W = (T*)o->W;
  r.comp = (T*)o->sph_compression;
  r.dens = (T*)o->sph_density;
  r.psi_adv = (T*)o->psi_adv;
  r.alpha = (T*)o->alpha;
  r.alpha_2 = (T*)o->alpha_2;
  r.zeta = (T*)o->fbm_zeta;
  r.pressure = (T*)o->pressure;
  r.flag = o->flag;
  r.cs = o->cell_structured;
  return r;
}

// DFSPH/VFSPH aliases, sph_obj.py:65-73
template <class T>
__device__ __forceinline__ T Xof(const KP<T>& k, const RefObj<T>& o, int i) {
  return k.solver == TSPH_VFSPH ? o.rest_volume[i] : o.mass[i];
}
template <class T>
__device__ __forceinline__ T psiof(const KP<T>& k, const RefObj<T>& o, int i) {
  return k.solver == TSPH_VFSPH ? o.comp[i] : o.dens[i];
}
template <class T>
__device__ __forceinline__ T rpsiof(const KP<T>& k, const RefObj<T>& o, int i) {
  return k.solver == TSPH_VFSPH ? T(1) : o.rest_density[i];
}

// sph.py:11-19
template <class T, class F>
__device__ __forceinline__ void ref_walk(const KP<T>& k, const RefGrid& g, const int* cs, int nuid,
                                         F&& f) {
  const int side = 2 * k.R + 1;
  for (int t = 0; t < k.ntemp; ++t) {
    int ox = t % side - k.R;
    int oy = (t / side) % side - k.R;
    int oz = k.dim == 3 ? t / (side * side) - k.R : 0;
    int code = dim_encode(k, wadd(cs[0], ox), wadd(cs[1], oy), wadd(cs[2], oz));
    if (0 < code && code < k.node_num) {
      int cnt = g.npc[code];
      for (int j = 0; j < cnt; ++j) {
        int shift = g.nps[code] + j;
        if (g.uin[shift] == nuid) f(g.pin[shift]);
      }
    }
  }
}

template <class T>
__device__ __forceinline__ T ref_norm(T x, T y, T z) {
  return s_sqrt(s_r2(x, y, z));
}

// ---------------------------------------------------------------------------
// Candidates beyond h.  W, W' and C vanish there, so a pair's term is an exact
// zero and leaving the pair out changes no sum, as long as what the zero is
// multiplied with is finite: an infinity, a NaN or an overflow makes the term a
// NaN, which the reference adds.  ref_plain_other(j) and ref_plain_own(i) hold
// where the other's and the particle's own share of a term cannot do that:
// magnitudes up to 1e9 and divisors from 1e-9 on, so that no product of a term
// leaves FP32.  k_ref_plain asks it of every particle of nobj before a pair
// kernel runs; a block of the pair kernel that meets one that is not plain, on
// either side, takes all candidates of its walks instead of those in range.
// ---------------------------------------------------------------------------
constexpr int kRefNormal = 100, kRefForce = 101;  // surface tension's two loops

template <class T>
__device__ __forceinline__ bool small(T v) {
  return fabs(v) <= T(1e9);
}
template <class T>
__device__ __forceinline__ bool small(const V4<T>& v) {
  return small(v.x) && small(v.y) && small(v.z);
}
template <class T>
__device__ __forceinline__ bool divides(T v) {
  return fabs(v) >= T(1e-9);
}

template <int KID, class T>
__device__ __forceinline__ bool ref_plain_other(const KP<T>& k, const RefObj<T>& no, int j) {
  bool ok = small(no.pos[j]);
  if constexpr (KID == TSPH_K_SPH_prepare_attr)
    ok = ok && small(no.rest_volume[j]) && small(no.mass[j]);
  if constexpr (KID == TSPH_K_SPH_prepare_alpha_1) ok = ok && small(Xof(k, no, j));
  if constexpr (KID == TSPH_K_SPH_prepare_alpha_2)
    ok = ok && small(Xof(k, no, j)) && divides(no.mass[j]);
  if constexpr (KID == TSPH_K_SPH_advection_viscosity_acc)
    ok = ok && small(no.vel[j]) && small(Xof(k, no, j) / psiof(k, no, j));
  if constexpr (KID == TSPH_K_WC_pressure_acce)
    ok = ok && small(no.mass[j]) && small(no.pressure[j] / (no.dens[j] * no.dens[j]));
  if constexpr (KID == TSPH_K_IPPE_adv_psi)
    ok = ok && small(no.vel_adv[j]) && small(Xof(k, no, j));
  if constexpr (KID == TSPH_K_IPPE_update_vel_adv)
    ok = ok && small(Xof(k, no, j)) && small(no.psi_adv[j]) && divides(no.alpha[j]);
  if constexpr (KID == kRefNormal) ok = ok && small(Xof(k, no, j) / psiof(k, no, j));
  if constexpr (KID == kRefForce)
    ok = ok && small(no.mass[j]) && small(no.normal[j]) && psiof(k, no, j) >= T(1e-9);
  if constexpr (KID == TSPH_K_SPH_FBM_diffuse || KID == TSPH_K_SPH_FBM_convect) {
    ok = ok && small(no.rest_volume[j]);
    for (int q = 0; q < k.P; ++q) {
      ok = ok && small(no.vf[(long)j * k.P + q]);
      if constexpr (KID == TSPH_K_SPH_FBM_convect) ok = ok && small(no.drift[(long)j * k.P + q]);
    }
  }
  return ok;
}

template <int KID, class T>
__device__ __forceinline__ bool ref_plain_own(const KP<T>& k, const RefObj<T>& o, int i, T dt) {
  bool ok = small(o.pos[i]) && small(dt);
  if constexpr (KID == TSPH_K_SPH_advection_viscosity_acc)
    ok = ok && small(o.vel[i]) && divides(o.rest_density[i]) && small(mu_of(k, o.vf, i));
  if constexpr (KID == TSPH_K_WC_pressure_acce)
    ok = ok && small(o.pressure[i] / (o.dens[i] * o.dens[i]));
  if constexpr (KID == TSPH_K_IPPE_adv_psi) ok = ok && small(o.vel_adv[i]);
  if constexpr (KID == TSPH_K_IPPE_update_vel_adv)
    ok = ok && small(Xof(k, o, i)) && small(o.psi_adv[i]) && divides(o.alpha[i]) &&
         divides(o.mass[i]) && divides(dt);
  if constexpr (KID == kRefForce)
    ok = ok && small(o.normal[i]) && small(rpsiof(k, o, i)) && psiof(k, o, i) >= T(1e-9);
  if constexpr (KID == TSPH_K_SPH_FBM_diffuse || KID == TSPH_K_SPH_FBM_convect) {
    ok = ok && small(KID == TSPH_K_SPH_FBM_diffuse ? dt * k.fbmD : k.fbmC * dt);
    for (int q = 0; q < k.P; ++q) {
      ok = ok && small(o.vf[(long)i * k.P + q]);
      if constexpr (KID == TSPH_K_SPH_FBM_convect) ok = ok && small(o.drift[(long)i * k.P + q]);
    }
  }
  return ok;
}

// flags[block]: a particle of the block's share is not plain.  At most kBlock
// blocks, as a pair kernel's block reads one flag per thread: 4.6-5.1 us a call at
// 100k particles.
constexpr int kPlainThreads = 1024;
inline int plain_blocks(int n, long room) {
  const long want = ((long)n + kPlainThreads - 1) / kPlainThreads;
  return (int)std::min({want, (long)kBlock, room});
}
template <class T, int KID>
__global__ void __launch_bounds__(kPlainThreads) k_ref_plain(KP<T> k, RefObj<T> no, int* flags) {
  bool ok = true;
  for (int j = blockIdx.x * kPlainThreads + threadIdx.x; j < no.n; j += gridDim.x * kPlainThreads)
    ok = ok && ref_plain_other<KID>(k, no, j);
  const int odd = __syncthreads_or(!ok);
  if (threadIdx.x == 0) flags[blockIdx.x] = odd;
}
// Whether this block has to take all candidates (every thread of the block asks).
template <int KID, class T>
__device__ __forceinline__ bool ref_take_all(const KP<T>& k, const RefObj<T>& o, int i, T dt,
                                             const int* flags, int nflag) {
  const bool other = (int)threadIdx.x < nflag && flags[threadIdx.x] != 0;
  return __syncthreads_or(other || (i < o.n && !ref_plain_own<KID>(k, o, i, dt))) != 0;
}

template <class T>
__global__ void __launch_bounds__(kBlock)
    k_ref(int kid, KP<T> k, RefGrid g, RefObj<T> o, RefObj<T> no, double* partial,
          TsphControl* ctrl, const int* flags, int nflag) {
  TSPH_STRICT
  __shared__ double lds[kWaves];
  const int nblk = gridDim.x;
  const int i = blockIdx.x * kBlock + threadIdx.x;
  const bool act = i < o.n;
  const T dt = (T)ctrl->dt;
  const int P = k.P;
  double red0 = 0, red1 = 0;
  double redmin = 1e300;
  const int* cs = act ? o.cs + 4 * i : nullptr;
  switch (kid) {
    case TSPH_K_SPH_clean_value:  // sph.py:22-38
      if (blockIdx.x == 0 && threadIdx.x == 0) ctrl->general_flag = 1;
      if (act) {
        o.W[i] = 0; o.comp[i] = 0; o.dens[i] = 0; o.alpha_2[i] = 0; o.flag[i] = 0;
        V4<T> z{T(0), T(0), T(0), T(0)};
        o.acce[i] = z; o.acce_adv[i] = z; o.alpha_1[i] = z;
        for (int q = 0; q < P; ++q) o.drift[(long)i * P + q] = z;
      }
      return;
    case TSPH_K_cfl_condition:  // sph.py:41-47
      if (act) {
        V4<T> v = o.vel[i];
        T vn = ref_norm(v.x, v.y, v.z);
        if (vn > T(1e-4)) {
          T q = k.gps / vn;
          redmin = (double)(q * k.cfl);
        }
      }
      break;
    case TSPH_K_SPH_prepare_alpha:  // sph.py:100-105
      if (act) {
        V4<T> a = o.alpha_1[i];
        T al = s_r2(a.x, a.y, a.z) / o.mass[i] + o.alpha_2[i];
        if (al < T(1e-4)) al = T(1e-4);
        o.alpha[i] = al;
      }
      return;
    case TSPH_K_SPH_advection_gravity_acc:  // sph.py:108-111
      if (act) {
        V4<T> a = o.acce_adv[i];
        o.acce_adv[i] = V4<T>{a.x + k.g[0], a.y + k.g[1], a.z + k.g[2], a.w};
      }
      return;
    case TSPH_K_WC_pressure_val:  // sph.py:169-175
      if (act) {
        T cs2 = (T)(k.cs * k.cs);
        T ratio = o.dens[i] / o.rest_density[i];
        T res = T(1), b = ratio;
        int e = 7;
        while (e > 0) {
          if (e & 1) res = res * b;
          b = b * b;
          e >>= 1;
        }
        T pr = (o.rest_density[i] * cs2 / (T)k.wc_gamma) * (res - T(1));
        if (pr < T(0)) pr = T(0);
        o.pressure[i] = pr;
      }
      return;
    case TSPH_K_IPPE_adv_psi_init:  // sph.py:196-199
      if (act) o.psi_adv[i] = psiof(k, o, i) - rpsiof(k, o, i);
      return;
    case TSPH_K_IPPE_psi_adv_non_negative:  // sph.py:219-226
      if (act) {
        T psi = o.psi_adv[i];
        if (psi < T(0)) psi = T(0);
        o.psi_adv[i] = psi;
        red0 = (double)(psi / rpsiof(k, o, i));
      }
      break;
    case TSPH_K_SPH_advection_update_vel_adv:  // sph.py:247-250
      if (act) {
        V4<T> v = o.vel[i], a = o.acce_adv[i];
        o.vel_adv[i] = V4<T>{v.x + a.x * dt, v.y + a.y * dt, v.z + a.z * dt, T(0)};
      }
      return;
    case TSPH_K_SPH_vel_2_vel_adv:  // sph.py:253-256
      if (act) o.vel_adv[i] = o.vel[i];
      return;
    case TSPH_K_SPH_vel_adv_2_vel:  // sph.py:259-262
      if (act) o.vel[i] = o.vel_adv[i];
      return;
    case TSPH_K_SPH_update_pos:  // sph.py:265-269
      if (act) {
        V4<T> v = o.vel_adv[i], p = o.pos[i];
        o.vel[i] = v;
        o.pos[i] = V4<T>{p.x + v.x * dt, p.y + v.y * dt, p.z + v.z * dt, p.w};
      }
      return;
    case TSPH_K_SPH_update_energy:  // sph.py:272-279
      if (act) {
        V4<T> v = o.vel[i], p = o.pos[i];
        T m = o.mass[i];
        red0 = (double)(T(0.5) * m * s_r2(v.x, v.y, v.z));
        red1 = (double)(-m * k.g[1] * (p.y - k.lb[1]));
      }
      break;
    case TSPH_K_SPH_update_mass:  // sph.py:282-286
      if (act) {
        T rd = k.rho[0] * o.vf[(long)i * P];
        for (int q = 1; q < P; ++q) rd = rd + k.rho[q] * o.vf[(long)i * P + q];
        o.rest_density[i] = rd;
        T m = rd * o.rest_volume[i];
        o.mass[i] = m;
        V4<T> p = o.pos[i];
        p.w = k.solver == TSPH_VFSPH ? o.rest_volume[i] : m;
        o.pos[i] = p;
      }
      return;
    case TSPH_K_SPH_FBM_clean_tmp:  // sph.py:301-305
      if (act)
        for (int q = 0; q < P; ++q) o.vf_tmp[(long)i * P + q] = T(0);
      return;
    case TSPH_K_SPH_FBM_diffuse: {  // sph.py:308-326
      const bool all = ref_take_all<TSPH_K_SPH_FBM_diffuse>(k, o, i, dt, flags, nflag);
      if (act && o.flag[i] == 0) {
        V4<T> p = o.pos[i];
        T acc[kMaxP];
        for (int q = 0; q < P; ++q) acc[q] = o.vf_tmp[(long)i * P + q];
        T pre = dt * k.fbmD;
        ref_walk(k, g, cs, no.uid, [&](int j) {
          V4<T> q = no.pos[j];
          if (!all && !(s_r2(p.x - q.x, p.y - q.y, p.z - q.z) <= k.r2max)) return;
          if (no.flag[j] != 0) return;
          T r = ref_norm(p.x - q.x, p.y - q.y, p.z - q.z);
          if (r > T(0)) {
            T wg = s_Wg(k, r);
            T den = r * r + k.eps;
            for (int s = 0; s < P; ++s) {
              T dphi = o.vf[(long)i * P + s] - no.vf[(long)j * P + s];
              acc[s] = acc[s] + pre * dphi * no.rest_volume[j] * r * wg / den;
            }
          }
        });
        for (int q = 0; q < P; ++q) o.vf_tmp[(long)i * P + q] = acc[q];
      }
      return;
    }
    case TSPH_K_SPH_FBM_check_tmp:  // sph.py:366-372
      if (act) {
        bool neg = false;
        for (int q = 0; q < P; ++q)
          if (o.vf[(long)i * P + q] + o.vf_tmp[(long)i * P + q] < T(0)) neg = true;
        if (neg) {
          o.flag[i] = 1;
          red0 = 1;
        }
      }
      break;
    case TSPH_K_SPH_update_volume_frac:  // sph.py:375-379
      if (act && !(o.flag[i] > 0))
        for (int q = 0; q < P; ++q)
          o.vf[(long)i * P + q] = o.vf[(long)i * P + q] + o.vf_tmp[(long)i * P + q];
      return;
    default:
      return;
  }
  // reductions: block partials, finished by k_finalize in stream order
  double s0 = block_sum(red0, lds);
  double s1 = block_sum(red1, lds);
  double mn = block_min(redmin, lds);
  if (threadIdx.x == 0) {
    partial[blockIdx.x] = kid == TSPH_K_cfl_condition ? mn : s0;
    partial[nblk + blockIdx.x] = s1;
  }
}

// ---------------------------------------------------------------------------
// The pair kernels, one instance per kernel id, a quad of lanes per particle
// (tsph_sweep.h: walk_quad_cells): the quad tests the candidates of the Ngrid
// four at a time and works off those in range, and every sum takes its terms
// in the reference's order.  One kernel with a switch over all ids, one lane per
// particle and the whole pair math on each of the 200 or so candidates took
// 130-170 us per call at 100k particles; these take 39-72 us there, bound by the
// dependent loads of the walk (entry, then position).  A whole reference step at
// 4k / 100k / 1M: 3.5 / 4.0 / 15.5 ms, now 1.09 / 1.65 / 9.5 (0.96 / 1.46 / 8.7
// without k_ref_plain's calls and the row check below).
// ---------------------------------------------------------------------------

// The walk around cell cs[] of particle p over nuid's candidates up to r2lim
// (those at a NaN distance among them).  A row of cells is one range where the
// Ngrid holds them one after the other, as tsph_ngrid_build does; where it does
// not (the reference's mem_shift, sph_obj.py:308-314, hands the ranges out in
// whatever order its threads reach the cells) every cell is read by itself.
// Asking whether it does costs 1-2 us of a call's 39-72 at 100k particles.
template <class T, class Load, class Term>
__device__ __forceinline__ void ref_quad(const KP<T>& k, const RefGrid& g, const int* cs, int nuid,
                                         const V4<T>* __restrict__ npos, const V4<T>& p, T r2lim,
                                         WalkLds& lds, Load&& load, Term&& term) {
  walk_quad_cells<true>(
      k, cs, lds,
      [&](int lo, int hi, bool* split) {
        int s0, end;
        if (hi - lo == 2) {  // a row of the default range (R = 1): two loads
          int s[3], n[3];
          __builtin_memcpy(s, g.nps + lo, sizeof(s));
          __builtin_memcpy(n, g.npc + lo, sizeof(n));
          s0 = s[0];
          end = s[2] + n[2];
          *split |= s[1] != s0 + n[0] || s[2] != s[1] + n[1];
        } else {
          s0 = g.nps[lo];
          end = s0 + g.npc[lo];
          for (int q = lo + 1; q <= hi; ++q) {
            const int s = g.nps[q];
            *split |= s != end;
            end = s + g.npc[q];
          }
        }
        return make_int2(s0, end);
      },
      [&](int s) {
        Cand<T> d;
        d.j = g.uin[s] == nuid ? g.pin[s] : -1;
        d.q = d.j >= 0 ? npos[d.j] : p;
        return d;
      },
      [&](const Cand<T>& d, bool* apart) {
        const T r2 = s_r2(p.x - d.q.x, p.y - d.q.y, p.z - d.q.z);
        *apart = r2 > T(0);  // as r > 0: the square root of a positive value is positive
        return !(r2 > r2lim);
      },
      load, term);
}

template <class T>
struct RefRec {
  V4<T> q, v;
  T a, b, c;
};

// These two keep 7 waves per SIMD in FP32 (the update by a spill at its entry, for
// the address of its result, instead of 76 registers): 54 us a call of the update
// at 100k with 6, 47 with 7.
template <class T>
constexpr int ref_waves(int kid) {
  return sizeof(T) == 4 && (kid == TSPH_K_IPPE_update_vel_adv || kid == TSPH_K_SPH_prepare_attr) ? 7 : 1;
}
template <class T, int KID>
__global__ void __launch_bounds__(kBlock, ref_waves<T>(KID))
    k_ref_pair(KP<T> k, RefGrid g, RefObj<T> o, RefObj<T> no, const TsphControl* ctrl,
               const int* flags, int nflag) {
  TSPH_STRICT
  __shared__ WalkLds lds;
  const int i = coop_particle<kQuad>(coop_sub(Blk{(int)blockIdx.x, (int)gridDim.x}));
  const T dt = (T)ctrl->dt;
  bool all = ref_take_all<KID>(k, o, i, dt, flags, nflag);
  if constexpr (KID == kRefForce) {
    if (!all && k.gamma == T(0)) return;  // every term is an exact zero
    all = true;                           // else (n_i - n_j) counts at any distance
  }
  const T r2lim = all ? T(INFINITY) : k.r2max;
  if (i >= o.n) return;
  const bool lead = coop_lane<kQuad>() == 0;
  const bool d3 = k.dim == 3;
  const int* cs = o.cs + 4 * i;
  const V4<T> p = o.pos[i];
  // add(load, pair): pair(record, dx, dy, dz, r, on) with on = the lane holds
  // a candidate (r > 0, except for W(0) in prepare_attr)
  auto add = [&](auto&& load, auto&& pair) {
    ref_quad(k, g, cs, no.uid, no.pos, p, r2lim, lds, load,
             [&](const RefRec<T>& d, int, bool valid, bool apart) {
               TSPH_STRICT
               const T dx = p.x - d.q.x, dy = p.y - d.q.y, dz = p.z - d.q.z;
               pair(d, dx, dy, dz, ref_norm(dx, dy, dz),
                    valid && (apart || KID == TSPH_K_SPH_prepare_attr));
             });
  };
  // acc + the quad's terms, component by component
  auto add3 = [&](V4<T>& acc, T x, T y, T z, bool on) {
    acc.x = quad_add(acc.x, on ? x : T(0));
    acc.y = quad_add(acc.y, on ? y : T(0));
    acc.z = quad_add(acc.z, on ? z : T(0));
  };
  if constexpr (KID == TSPH_K_SPH_prepare_attr) {  // sph.py:50-64
    T w = o.W[i], cp = o.comp[i], dn = o.dens[i];
    add([&](int j) { return RefRec<T>{no.pos[j], V4<T>{}, no.rest_volume[j], no.mass[j], T(0)}; },
        [&](const RefRec<T>& d, T, T, T, T r, bool on) {
          TSPH_STRICT
          const T Wr = s_W(k, r);
          w = quad_add(w, on ? Wr : T(0));
          cp = quad_add(cp, on ? Wr * d.a : T(0));
          dn = quad_add(dn, on ? Wr * d.b : T(0));
        });
    if (lead) {
      o.W[i] = w;
      o.comp[i] = cp;
      o.dens[i] = dn;
    }
  } else if constexpr (KID == TSPH_K_SPH_prepare_alpha_1) {  // sph.py:67-81
    V4<T> a = o.alpha_1[i];
    add([&](int j) { return RefRec<T>{no.pos[j], V4<T>{}, Xof(k, no, j), T(0), T(0)}; },
        [&](const RefRec<T>& d, T dx, T dy, T dz, T r, bool on) {
          TSPH_STRICT
          const T wg = s_Wg(k, r);
          add3(a, d.a * dx / r * wg, d.a * dy / r * wg, d.a * dz / r * wg, on);
        });
    if (lead) o.alpha_1[i] = a;
  } else if constexpr (KID == TSPH_K_SPH_prepare_alpha_2) {  // sph.py:84-97
    T a2 = o.alpha_2[i];
    add([&](int j) { return RefRec<T>{no.pos[j], V4<T>{}, Xof(k, no, j), no.mass[j], T(0)}; },
        [&](const RefRec<T>& d, T, T, T, T r, bool on) {
          TSPH_STRICT
          const T wg = s_Wg(k, r);
          const T wg2 = wg * wg;
          a2 = quad_add(a2, on ? wg2 * (d.a * d.a) / d.b : T(0));
        });
    if (lead) o.alpha_2[i] = a2;
  } else if constexpr (KID == TSPH_K_SPH_advection_viscosity_acc) {  // sph.py:114-129
    const V4<T> vi = o.vel[i];
    V4<T> a = o.acce_adv[i];
    const T rd = o.rest_density[i];
    const T mu = mu_of(k, o.vf, i);  // the global mu, or the per-phase extension
    add([&](int j) { return RefRec<T>{no.pos[j], no.vel[j], Xof(k, no, j), psiof(k, no, j), T(0)}; },
        [&](const RefRec<T>& d, T dx, T dy, T dz, T r, bool on) {
          TSPH_STRICT
          const T Vj = d.a / d.b;
          const T s = k.two_d2 * Vj * s_Wg(k, r);
          const T inv = T(1) / ref_norm(dx, dy, dz);
          T Ax = (vi.x - d.v.x) * dx;
          Ax = Ax + (vi.y - d.v.y) * dy;
          if (d3) Ax = Ax + (vi.z - d.v.z) * dz;
          const T den = k.eps + r * r;
          add3(a, s * (inv * dx) * Ax / den * mu / rd, s * (inv * dy) * Ax / den * mu / rd,
               d3 ? s * (inv * dz) * Ax / den * mu / rd : T(0), on);
        });
    if (lead) o.acce_adv[i] = a;
  } else if constexpr (KID == TSPH_K_WC_pressure_acce) {  // sph.py:178-193
    V4<T> a = o.acce_adv[i];
    const T pi = o.pressure[i], di = o.dens[i];
    add([&](int j) { return RefRec<T>{no.pos[j], V4<T>{}, no.dens[j], no.pressure[j], no.mass[j]}; },
        [&](const RefRec<T>& d, T dx, T dy, T dz, T r, bool on) {
          TSPH_STRICT
          const T pt = pi / (di * di) + d.b / (d.a * d.a);
          const T wg = s_Wg(k, r);
          add3(a, -pt * d.c * dx / r * wg, -pt * d.c * dy / r * wg,
               d3 ? -pt * d.c * dz / r * wg : T(0), on);
        });
    if (lead) o.acce_adv[i] = a;
  } else if constexpr (KID == TSPH_K_IPPE_adv_psi) {  // sph.py:202-216
    const V4<T> va = o.vel_adv[i];
    T psi = o.psi_adv[i];
    add([&](int j) { return RefRec<T>{no.pos[j], no.vel_adv[j], Xof(k, no, j), T(0), T(0)}; },
        [&](const RefRec<T>& d, T dx, T dy, T dz, T r, bool on) {
          TSPH_STRICT
          const T wg = s_Wg(k, r);
          T dot = (dx / r * wg) * (va.x - d.v.x);
          dot = dot + (dy / r * wg) * (va.y - d.v.y);
          if (d3) dot = dot + (dz / r * wg) * (va.z - d.v.z);
          psi = quad_add(psi, on ? dot * d.a * dt : T(0));
        });
    if (lead) o.psi_adv[i] = psi;
  } else if constexpr (KID == TSPH_K_IPPE_update_vel_adv) {  // sph.py:229-244
    V4<T> va = o.vel_adv[i];
    const T pi = o.psi_adv[i], ai = o.alpha[i], Xi = Xof(k, o, i), mi = o.mass[i];
    const T c = -(T(1) / dt);
    add([&](int j) { return RefRec<T>{no.pos[j], V4<T>{}, Xof(k, no, j), no.psi_adv[j], no.alpha[j]}; },
        [&](const RefRec<T>& d, T dx, T dy, T dz, T r, bool on) {
          TSPH_STRICT
          const T a = pi * d.a / ai;
          const T b = d.b * Xi / d.c;
          const T s = c * (a + b);
          const T wg = s_Wg(k, r);
          add3(va, s * (dx / r * wg) / mi, s * (dy / r * wg) / mi,
               d3 ? s * (dz / r * wg) / mi : T(0), on);
        });
    if (lead) o.vel_adv[i] = va;
  } else if constexpr (KID == kRefNormal) {  // sph.py:141-149
    V4<T> n{};
    add([&](int j) { return RefRec<T>{no.pos[j], V4<T>{}, Xof(k, no, j), psiof(k, no, j), T(0)}; },
        [&](const RefRec<T>& d, T dx, T dy, T dz, T r, bool on) {
          TSPH_STRICT
          const T s = -d.a / d.b * s_Wg(k, r);
          add3(n, s * dx / r, s * dy / r, s * dz / r, on);
        });
    if (lead) o.normal[i] = V4<T>{n.x * k.h, n.y * k.h, n.z * k.h, T(0)};
  } else {  // kRefForce, sph.py:151-166: over all candidates with r > 0
    if (!(o.vf[(long)i * k.P] > T(0.99))) return;  // the whole quad: one particle
    V4<T> a = o.acce_adv[i];
    const V4<T> ni = o.normal[i];
    const T ri = rpsiof(k, o, i), pi = psiof(k, o, i);
    add([&](int j) {
          return RefRec<T>{no.pos[j], no.normal[j], no.mass[j], psiof(k, no, j), no.vf[(long)j * k.P]};
        },
        [&](const RefRec<T>& d, T dx, T dy, T dz, T r, bool on) {
          TSPH_STRICT
          const T cs2 = -k.gamma * d.a * s_C(k, r);
          const T f = T(2) * ri / (pi + d.b);
          add3(a, f * (cs2 * dx / r + k.gamma * (ni.x - d.v.x)),
               f * (cs2 * dy / r + k.gamma * (ni.y - d.v.y)),
               d3 ? f * (cs2 * dz / r + k.gamma * (ni.z - d.v.z)) : T(0), on && d.c > T(0.99));
        });
    if (lead) o.acce_adv[i] = a;
  }
}

// SPH_FBM_convect loop 1 (drift velocities) and loop 2 (flux), sph.py:329-363.
template <class T>
__global__ void __launch_bounds__(kBlock)
    k_ref_convect(int pass, KP<T> k, RefGrid g, RefObj<T> o, RefObj<T> no,
                  const TsphControl* ctrl, const int* flags, int nflag) {
  TSPH_STRICT
  int i = blockIdx.x * kBlock + threadIdx.x;
  const T dt = (T)ctrl->dt;
  const bool all =
      pass == 1 && ref_take_all<TSPH_K_SPH_FBM_convect>(k, o, i, dt, flags, nflag);
  if (i >= o.n) return;
  const int P = k.P;
  if (pass == 0) {
    V4<T> va = o.vel_adv[i], v = o.vel[i];
    T aa[3] = {(va.x - v.x) / dt, (va.y - v.y) / dt, (va.z - v.z) / dt};
    T rd = o.rest_density[i];
    T z = T(0);
    for (int q = 0; q < P; ++q) z = z + o.vf[(long)i * P + q] * (k.rho[q] - rd) / k.rho[q];
    T fa[3];
    for (int d = 0; d < 3; ++d) fa[d] = (aa[d] - z * k.g[d]) / (T(1) - z);
    o.acce_adv[i] = V4<T>{aa[0], aa[1], aa[2], T(0)};
    o.acce[i] = V4<T>{fa[0], fa[1], fa[2], T(0)};
    o.zeta[i] = z;
    for (int q = 0; q < P; ++q) {
      T phi = o.vf[(long)i * P + q];
      T s = phi * (k.rho[q] - rd);
      T u[3];
      for (int d = 0; d < 3; ++d) u[d] = s * (k.g[d] - fa[d]);
      T wgt = phi * k.rho[q];
      if (wgt > T(1e-6)) {
        for (int d = 0; d < 3; ++d) u[d] = u[d] / wgt;
      } else {
        for (int d = 0; d < 3; ++d) u[d] = u[d] * T(0);
      }
      for (int d = 0; d < 3; ++d) u[d] = u[d] + (fa[d] - aa[d]);
      for (int d = 0; d < 3; ++d) u[d] = u[d] * dt;
      if (k.dim == 2) u[2] = T(0);
      o.drift[(long)i * P + q] = V4<T>{u[0], u[1], u[2], T(0)};
    }
    return;
  }
  if (o.flag[i] != 0) return;
  const int* cs = o.cs + 4 * i;
  V4<T> p = o.pos[i];
  T acc[kMaxP];
  for (int q = 0; q < P; ++q) acc[q] = o.vf_tmp[(long)i * P + q];
  T pre = k.fbmC * dt;
  ref_walk(k, g, cs, no.uid, [&](int j) {
    V4<T> q = no.pos[j];
    T dx = p.x - q.x, dy = p.y - q.y, dz = p.z - q.z;
    if (!all && !(s_r2(dx, dy, dz) <= k.r2max)) return;
    if (no.flag[j] != 0) return;
    T r = ref_norm(dx, dy, dz);
    if (r > T(0)) {
      T wg = s_Wg(k, r);
      for (int s = 0; s < P; ++s) {
        V4<T> ui = o.drift[(long)i * P + s], uj = no.drift[(long)j * P + s];
        T pi = o.vf[(long)i * P + s], pj = no.vf[(long)j * P + s];
        T dot = (pi * ui.x + pj * uj.x) * (dx / r);
        dot = dot + (pi * ui.y + pj * uj.y) * (dy / r);
        if (k.dim == 3) dot = dot + (pi * ui.z + pj * uj.z) * (dz / r);
        acc[s] = acc[s] - pre * no.rest_volume[j] * dot * wg;
      }
    }
  });
  for (int q = 0; q < P; ++q) o.vf_tmp[(long)i * P + q] = acc[q];
}

template <class T>
int ref_kernel(const TsphParams& prm, int kid, TsphObject* obj, const TsphObject* nobj,
               const int* npc, const int* nps, const int* pin, const int* uin, TsphControl* ctrl,
               void* ws, size_t wsb, hipStream_t st) {
  TSPH_REQUIRE(kid >= 0 && kid < TSPH_K_COUNT, TSPH_EINVAL, "tsph_ref_kernel: bad kernel id %d",
               kid);
  KP<T> k = make_kp<T>(prm);
  WsLayout L;
  TSPH_REQUIRE(carve_ws(ws, wsb, obj->capacity, prm.node_num, &L), TSPH_ECAPACITY,
               "tsph_ref_kernel: workspace too small");
  RefGrid g{npc, nps, pin, uin};
  RefObj<T> o = ref_obj<T>(obj);
  RefObj<T> no = ref_obj<T>(nobj ? nobj : obj);
  int nb = blocks_for(obj->n > 0 ? obj->n : 1);
  int* flags = (int*)L.partial;  // unused by the pair kernels otherwise
  const int nflag = plain_blocks(no.n, partial_doubles(obj->capacity) * 2);
  auto plain = [&](auto kern) {
    if (nflag > 0)
      hipLaunchKernelGGL(kern, dim3(nflag), dim3(kPlainThreads), 0, st, k, no, flags);
  };
  auto pair = [&](auto ask, auto kern) {
    if (o.n <= 0) return;
    plain(ask);
    hipLaunchKernelGGL(kern, dim3(coop_blocks<kQuad>(o.n)), dim3(kBlock), 0, st, k, g, o, no, ctrl,
                       flags, nflag);
  };
  if (kid == TSPH_K_SPH_prepare_attr) {
    pair(k_ref_plain<T, TSPH_K_SPH_prepare_attr>, k_ref_pair<T, TSPH_K_SPH_prepare_attr>);
  } else if (kid == TSPH_K_SPH_prepare_alpha_1) {
    pair(k_ref_plain<T, TSPH_K_SPH_prepare_alpha_1>, k_ref_pair<T, TSPH_K_SPH_prepare_alpha_1>);
  } else if (kid == TSPH_K_SPH_prepare_alpha_2) {
    pair(k_ref_plain<T, TSPH_K_SPH_prepare_alpha_2>, k_ref_pair<T, TSPH_K_SPH_prepare_alpha_2>);
  } else if (kid == TSPH_K_SPH_advection_viscosity_acc) {
    pair(k_ref_plain<T, TSPH_K_SPH_advection_viscosity_acc>, k_ref_pair<T, TSPH_K_SPH_advection_viscosity_acc>);
  } else if (kid == TSPH_K_WC_pressure_acce) {
    pair(k_ref_plain<T, TSPH_K_WC_pressure_acce>, k_ref_pair<T, TSPH_K_WC_pressure_acce>);
  } else if (kid == TSPH_K_IPPE_adv_psi) {
    pair(k_ref_plain<T, TSPH_K_IPPE_adv_psi>, k_ref_pair<T, TSPH_K_IPPE_adv_psi>);
  } else if (kid == TSPH_K_IPPE_update_vel_adv) {
    pair(k_ref_plain<T, TSPH_K_IPPE_update_vel_adv>, k_ref_pair<T, TSPH_K_IPPE_update_vel_adv>);
  } else if (kid == TSPH_K_SPH_advection_surface_tension_acc) {
    pair(k_ref_plain<T, kRefNormal>, k_ref_pair<T, kRefNormal>);
    if (k.gamma == T(0))  // whether any term can be other than zero
      pair(k_ref_plain<T, kRefForce>, k_ref_pair<T, kRefForce>);
    else if (o.n > 0)
      hipLaunchKernelGGL((k_ref_pair<T, kRefForce>), dim3(coop_blocks<kQuad>(o.n)), dim3(kBlock), 0,
                         st, k, g, o, no, ctrl, flags, 0);
  } else if (kid == TSPH_K_SPH_FBM_convect) {
    hipLaunchKernelGGL(k_ref_convect<T>, dim3(nb), dim3(kBlock), 0, st, 0, k, g, o, no, ctrl,
                       flags, 0);
    plain(k_ref_plain<T, TSPH_K_SPH_FBM_convect>);  // the drifts are there now
    hipLaunchKernelGGL(k_ref_convect<T>, dim3(nb), dim3(kBlock), 0, st, 1, k, g, o, no, ctrl,
                       flags, nflag);
  } else {
    if (kid == TSPH_K_SPH_FBM_diffuse) plain(k_ref_plain<T, TSPH_K_SPH_FBM_diffuse>);
    hipLaunchKernelGGL(k_ref<T>, dim3(nb), dim3(kBlock), 0, st, kid, k, g, o, no, L.partial, ctrl,
                       flags, nflag);
    int mode = kid == TSPH_K_cfl_condition ? kFinCfl
               : kid == TSPH_K_SPH_update_energy ? kFinEnergy
               : kid == TSPH_K_SPH_FBM_check_tmp ? kFinFlag
               : kid == TSPH_K_IPPE_psi_adv_non_negative ? kFinCompression : -1;
    if (mode >= 0)
      hipLaunchKernelGGL(k_finalize<T>, dim3(1), dim3(kBlock), 0, st, k, mode, L.partial, nb,
                         obj->n, ctrl, 0, 0);
  }
  TSPH_LAUNCH_CHECK("ref_kernel");
  return 0;
}

template int ref_kernel<float>(const TsphParams&, int, TsphObject*, const TsphObject*, const int*, const int*, const int*, const int*, TsphControl*, void*, size_t, hipStream_t);
template int ref_kernel<double>(const TsphParams&, int, TsphObject*, const TsphObject*, const int*, const int*, const int*, const int*, TsphControl*, void*, size_t, hipStream_t);

}  // namespace tsph
