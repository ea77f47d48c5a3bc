// kernels_dfsph.hip -- DFSPH sweeps over the cell-sorted particles
// (DFSPHSolver, SPH/main.py:1519-1848; SPHBase, :908-1093).
//
// 1, 4 or 16 lanes per particle (Batch::lanes) share its neighbor list and add
// their terms in list order (for_pairs), so every per-particle sum is formed in
// the reference's serial order.  The source sweeps leave FP64 partials of the
// average density error per scene; k_scene_finish adds them and decides
// termination, clearing the scene's active flag; later launches of a finished
// scene return at once.
#include <algorithm>

#include "device_common.h"

namespace nn {

// alpha as the pressure solve sees it: the reference scales the stored factor by
// 1/dt and dt around the divergence solve and then by 1/dt^2 (:1688,1713,1771).
__device__ __forceinline__ float alpha_div(const SceneDev& sc, float a) { return a * sc.inv_dt; }
__device__ __forceinline__ float alpha_press(const SceneDev& sc, float a) {
  return (sc.flags & SF_DIVERGENCE) ? ((a * sc.inv_dt) * sc.dt) * sc.inv_dt2 : a * sc.inv_dt2;
}

// Before a search: the cell counts to zero and the scenes' state as `begin`
// says: BEGIN_STATUS (a search by itself), BEGIN_STEP (also the three solvers'),
// BEGIN_CG (only the CG's, before a solve is repeated; no cells).  One launch
// for what were five: 1.5 to 3 us each, and the gaps between them.
__global__ void k_begin(Dev d, int begin, long cells) {
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < cells) d.cell_count[i] = 0;
  if (i < d.nscenes && begin != BEGIN_CELLS) {
    const SceneDev& sc = d.scenes[i];
    SceneState& st = d.state[i];
    if (begin != BEGIN_CG) st.status = 0;
    if (begin == BEGIN_STEP) {
      st.active_v = (sc.flags & SF_HAS_FLUID) && (sc.flags & SF_DIVERGENCE) ? 1 : 0;
      st.iter_v = 0;
      st.err_v = 0.0;
      st.active_p = (sc.flags & SF_HAS_FLUID) ? 1 : 0;
      st.iter_p = 0;
      st.err_p = 0.0;
    }
    if (begin != BEGIN_STATUS) {  // cg_init activates scenes
      st.active_cg = 0;
      st.cg_stop_at = 0;
      st.iter_cg = 0;
      st.cg_rr = 0.0;
      st.cg_bb = 0.0;
    }
  }
  if (i == 0 && begin >= BEGIN_STEP) {
    d.cg_list_n[0] = d.cg_list_n[1] = d.cg_list_n[2] = 0;
    d.n_active[0] = d.n_active[1] = 0;
  }
}

// compute_densities (:962-984), compute_DFSPH_factor (:1569-1608) and the first
// compute_density_change of the divergence solve (:1610-1645), fused: all three
// read the same neighbors and none reads what another writes.
template <int G, int B>
__global__ void k_density_alpha(Dev d) {
  const Ahead<G, B> own(d);
  int i, q, s;
  if (!lane_slot_scene<G>(d, i, q, s)) return;
  const SceneDev& sc = d.scenes[s];
  if (!(sc.flags & SF_HAS_FLUID)) return;
  float rho_out = 0.0f;
  if (i < sc.p_begin + sc.n && kind_of(own.info(d, i)) == KIND_FLUID) {
    const KernH kh(sc);
    const float4 xi = own.pos(d, i);
    const float4 vi = d.vel[i];
    const int cnt = own.count(d, i);
    const bool comp = (sc.flags & SF_COMPENSATED) != 0;
    KSum den{0.0f, 0.0f};
    float gix = 0.f, giy = 0.f, giz = 0.f, sk = 0.f, rd = 0.f;
    for_pairs<G, B, 6>(
        d, i, q, cnt, [&](int j) { return PosVel{d.pos[j], d.vel[j]}; },
        [&](int, const PosVel& nj, bool live, float (&t)[6]) {
          const float4 xj = nj.x, vj = nj.v;
          const float rx = xi.x - xj.x, ry = xi.y - xj.y, rz = xi.z - xj.z;
          const float Vj = fabsf(xj.w);
          float rn, w;
          const float3 g = pair_grad<true, false>(kh, sc, rx, ry, rz, live, rn, w);
          const float gpx = -Vj * g.x, gpy = -Vj * g.y, gpz = -Vj * g.z;
          const float dvx = vi.x - vj.x, dvy = vi.y - vj.y, dvz = vi.z - vj.z;
          t[0] = Vj * w;
          t[1] = live && xj.w > 0.0f ? gpx * gpx + gpy * gpy + gpz * gpz : NEUTRAL;
          t[2] = live ? -gpx : NEUTRAL;
          t[3] = live ? -gpy : NEUTRAL;
          t[4] = live ? -gpz : NEUTRAL;
          t[5] = live ? Vj * (dvx * g.x + dvy * g.y + dvz * g.z) : NEUTRAL;
        },
        [&](const float (&t)[6], bool ok) {
          KSum n = den;
          if (comp) n.add(t[0]);
          else n.s += t[0];
          den.s = ok ? n.s : den.s;
          den.c = ok ? n.c : den.c;
          sk += t[1];
          gix += t[2];
          giy += t[3];
          giz += t[4];
          rd += t[5];
        },
        &own);
    float rho = xi.w * sc.W0;
    rho += den.s;
    rho *= sc.rho0;
    rho_out = rho;
    sk += gix * gix + giy * giy + giz * giz;
    const float al = sk > 1e-6f ? -1.0f / sk : 0.0f;
    rd = rd > 0.0f ? rd : 0.0f;
    if (cnt < 20) rd = 0.0f;
    if (q == 0) {
      d.rho[i] = rho;
      d.sa[i] = make_float2(rd, al);
    }
  }
  const float m = wave_max(rho_out);
  if ((threadIdx.x & 63) == 0) d.wave_rho[i / (64 / G)] = m;
}

// A report to the host: one word of its pinned memory, which it polls, with the
// ticket it waits for in the high half.
__device__ __forceinline__ void report_word(unsigned long long* word, unsigned ticket, unsigned bits) {
  __hip_atomic_store(word, ((unsigned long long)ticket << 32) | bits, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}
// (a launch of its own: the end of the launches before it is what it reports)
__global__ void k_report_active(Dev d, int which, unsigned long long* report, unsigned ticket) {
  if (threadIdx.x == 0) report_word(report, ticket, which >= 0 && d.n_active[which] > 0);
}

// End of a step: per scene, the pair counts and the largest density of its
// wavefronts (list_lanes and rho_lanes entries per 64 slots), then its state
// into the host's pinned copy.  (With an atomic per wavefront on the scene's
// words, the density sweep of 131,072 particles took 45 us instead of 22: each
// atomic of one address costs about 13 ns.)  1,024 threads: 4.7 us at 138,304
// particles, 10.0 with 256.
constexpr int PUBLISH_THREADS = 1024;
__global__ __launch_bounds__(PUBLISH_THREADS) void k_publish(Dev d, int list_lanes, int rho_lanes, SceneState* host,
                                                             unsigned long long* report, unsigned ticket) {
  __shared__ long long red[2][PUBLISH_THREADS / 64];
  __shared__ float rmax[PUBLISH_THREADS / 64];
  const int s = blockIdx.x, t = threadIdx.x;
  const SceneDev& sc = d.scenes[s];
  long long tot = 0, cf = 0;
  float m = 0.0f;
  for (int k = list_lanes * sc.wave_begin + t; k < list_lanes * sc.wave_end; k += PUBLISH_THREADS) {
    const int2 c = d.wave_pairs[k];
    tot += c.x;
    cf += c.y;
  }
  if (sc.flags & SF_HAS_FLUID)
    for (int k = rho_lanes * sc.wave_begin + t; k < rho_lanes * sc.wave_end; k += PUBLISH_THREADS) m = fmaxf(m, d.wave_rho[k]);
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) {
    tot += __shfl_xor(tot, off, 64);
    cf += __shfl_xor(cf, off, 64);
  }
  m = wave_max(m);
  if ((t & 63) == 0) {
    red[0][t >> 6] = tot;
    red[1][t >> 6] = cf;
    rmax[t >> 6] = m;
  }
  __syncthreads();
  if (t != 0) return;
  unsigned long long pairs = 0, pairs_fluid = 0;
  m = 0.0f;
  for (int w = 0; w < PUBLISH_THREADS / 64; w++) {
    pairs += (unsigned long long)red[0][w];
    pairs_fluid += (unsigned long long)red[1][w];
    m = fmaxf(m, rmax[w]);
  }
  // copied first and completed in place: completed as a local copy, it lay in
  // scratch, for which every queue of a step would have to keep memory
  host[s] = d.state[s];
  host[s].pairs = pairs;
  host[s].pairs_fluid = pairs_fluid;
  host[s].max_rho_bits = __float_as_uint(m);
  // after the state: released to the host
  __hip_atomic_store(report + s, (unsigned long long)ticket << 32, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

// sum_j of the velocity changes both solvers' updates make (:1721-1760,
// :1799-1841): dt (k_i + k_j) V_j gradW_ij for a fluid neighbor, dt k_i V_j
// gradW_ij for a solid one, each where the factor exceeds eps; kj(nj) is the
// neighbor's factor.  SIGNED where the sums start at a velocity, which may be
// -0, and not at +0.
template <int G, int B, bool SIGNED, typename KJ>
__device__ __forceinline__ void velocity_push(const Dev& d, const SceneDev& sc, const KernH& kh, int i, int q,
                                              const Ahead<G, B>& own, float ki, KJ kj, float& ax, float& ay, float& az) {
  const float4 xi = own.pos(d, i);
  const bool solid_on = fabsf(ki) > sc.eps;
  for_pairs<G, B, 3>(
      d, i, q, own.count(d, i), [&](int j) { const float2 t = d.sa[j]; return PosSrc{d.pos[j], t.x, t.y}; },
      [&](int, const PosSrc& nj, bool live, float (&t)[3]) {
        const float4 xj = nj.x;
        const bool fluid = xj.w > 0.0f;
        const float ksum = ki + kj(nj);
        const bool on = live && (fluid ? fabsf(ksum) > sc.eps : solid_on);
        t[0] = t[1] = t[2] = NEUTRAL;
        if (on) {
          const float3 g = pair_grad<SIGNED>(kh, sc, xi.x - xj.x, xi.y - xj.y, xi.z - xj.z, true);
          // v -= f (-V g) with f = dt ksum, v += f (-V g) with f = -dt ki
          const float f = fluid ? -(sc.dt * ksum) : -sc.dt * ki;
          const float Vj = fabsf(xj.w);
          t[0] = f * (-Vj * g.x);
          t[1] = f * (-Vj * g.y);
          t[2] = f * (-Vj * g.z);
        }
      },
      [&](const float (&t)[3], bool) {
        ax += t[0];
        ay += t[1];
        az += t[2];
      },
      &own);
}

// divergence_solver_iteration_kernel, :1721-1760 (Jacobi: reads rho-dot and
// alpha, writes v).  Reactions on dynamic solids are not formed: the second
// clear_accelerations (:1552) erases them.
template <int G, int B>
__global__ void k_div_update(Dev d) {
  const Ahead<G, B> own(d);
  int i, q, s;
  if (!lane_slot_scene<G>(d, i, q, s)) return;
  const SceneDev& sc = d.scenes[s];
  if (!d.state[s].active_v) return;
  if (i >= sc.p_begin + sc.n || kind_of(own.info(d, i)) != KIND_FLUID) return;
  const KernH kh(sc);
  const float2 sai = d.sa[i];
  const float ki = sai.x * alpha_div(sc, sai.y);
  float dvx = 0.f, dvy = 0.f, dvz = 0.f;
  velocity_push<G, B, false>(d, sc, kh, i, q, own, ki, [&](const PosSrc& nj) { return nj.src * alpha_div(sc, nj.alpha); },
                             dvx, dvy, dvz);
  if (q != 0) return;
  float4 v = d.vel[i];
  v.x += dvx;
  v.y += dvy;
  v.z += dvz;
  d.vel[i] = v;
}

// sum_j V_j (v_i - v_j) . gradW_ij over all neighbors
template <int G, int B>
__device__ __forceinline__ float velocity_divergence(const Dev& d, const SceneDev& sc, int i, int q, const Ahead<G, B>& own) {
  const KernH kh(sc);
  const float4 xi = own.pos(d, i), vi = d.vel[i];
  const int cnt = own.count(d, i);
  float acc = 0.f;
  for_pairs<G, B, 1>(
      d, i, q, cnt, [&](int j) { return PosVel{d.pos[j], d.vel[j]}; },
      [&](int, const PosVel& nj, bool live, float (&t)[1]) {
        const float4 xj = nj.x, vj = nj.v;
        const float3 g = pair_grad(kh, sc, xi.x - xj.x, xi.y - xj.y, xi.z - xj.z, live);
        const float dvx = vi.x - vj.x, dvy = vi.y - vj.y, dvz = vi.z - vj.z;
        t[0] = live ? fabsf(xj.w) * (dvx * g.x + dvy * g.y + dvz * g.z) : NEUTRAL;
      },
      [&](const float (&t)[1], bool) { acc += t[0]; }, &own);
  return acc;
}

// compute_density_change (:1610-1645) + compute_density_error(0) (:1669-1675)
// and the loop test of divergence_solve (:1695-1703)
template <int G, int B>
__global__ void k_div_source(Dev d) {
  const Ahead<G, B> own(d);
  int i, q, s;
  if (!lane_slot_scene<G>(d, i, q, s)) return;
  const SceneDev& sc = d.scenes[s];
  SceneState* st = d.state + s;
  if (!st->active_v) return;
  double v[1] = {0.0};
  if (i < sc.p_begin + sc.n && kind_of(own.info(d, i)) == KIND_FLUID) {
    float rd = velocity_divergence<G, B>(d, sc, i, q, own);
    rd = rd > 0.0f ? rd : 0.0f;
    if (own.count(d, i) < 20) rd = 0.0f;
    if (q == 0) d.sa[i].x = rd;
    v[0] = (double)sc.rho0 * (double)rd - 0.0;
  }
  lane_partials<G, 1>(d, i, v, 0);
}

// non-pressure forces (:1557-1567): surface tension (:1378-1414) and the
// explicit viscosity (:1417-1468) in one neighbor walk, the Weiler result when
// the implicit solver ran, then non_pressure_advect (:1843-1848).  The second
// clear_accelerations (:1552) is folded in.  v is double-buffered: the sweep
// reads vel and writes vel_alt.
template <int G, int B>
__global__ void k_nonpressure(Dev d) {
  const Ahead<G, B> own(d);
  int i, q, s;
  if (!lane_slot_scene<G>(d, i, q, s)) return;
  const SceneDev& sc = d.scenes[s];
  if (i >= sc.p_begin + sc.n) return;
  const int kind = kind_of(own.info(d, i));
  const float4 vi = d.vel[i];
  if (!(sc.flags & SF_HAS_FLUID)) {
    if (q == 0) d.vel_alt[i] = vi;
    return;
  }
  const bool vis_on = (sc.flags & SF_VISCOSITY) != 0;
  const bool weiler = vis_on && (sc.flags & SF_WEILER);
  // one lane per particle: only for batches without velocity terms (Batch::lanes)
  const bool expl = G != 1 && vis_on && !weiler;
  const bool bnu_on = G != 1 && vis_on && sc.bnu != 0.0f;
  if (kind == KIND_FLUID) {
    const KernH kh(sc);
    const float4 xi = own.pos(d, i);
    const bool st_on = (sc.flags & SF_SURFACE_TENSION) != 0;
    const float rhoi = d.rho[i];
    float sx = 0.f, sy = 0.f, sz = 0.f, wvx = 0.f, wvy = 0.f, wvz = 0.f;
    // surface tension reads positions only: the velocities and densities are
    // gathered only for a viscosity term formed here (two loops, so that the
    // position-only one holds no velocity registers)
    if (expl || bnu_on) {
      struct NJ {
        float4 x, v;
        float rho;
      };
      const int cnt = own.count(d, i);
      for_pairs<G, B, 6>(
          d, i, q, cnt, [&](int j) { return NJ{d.pos[j], d.vel[j], d.rho[j]}; },
          [&](int, const NJ& nj, bool live, float (&t)[6]) {
            const float4 xj = nj.x, vj = nj.v;
            const float rx = xi.x - xj.x, ry = xi.y - xj.y, rz = xi.z - xj.z;
            const bool fluid = xj.w > 0.0f;
            float rn, w;
            const float3 g = pair_grad<true, false>(kh, sc, rx, ry, rz, live, rn, w);
#pragma unroll
            for (int n = 0; n < 6; n++) t[n] = NEUTRAL;
            if (live && fluid && st_on) {
              const float r2 = rx * rx + ry * ry + rz * rz;
              w = r2 > sc.diam2 ? w : sc.Wd;
              t[0] = -(sc.sig_m * rx * w);
              t[1] = -(sc.sig_m * ry * w);
              t[2] = -(sc.sig_m * rz * w);
            }
            if (live && (fluid ? expl : bnu_on)) {
              const float vxy = (vi.x - vj.x) * rx + (vi.y - vj.y) * ry + (vi.z - vj.z) * rz;
              const float num = fluid ? sc.mass : sc.rho0 * (-xj.w);
              const float f = (fluid ? sc.ten_nu : sc.ten_bnu) * (num / (fluid ? nj.rho : rhoi)) * vxy / (rn * rn + sc.visc_eps);
              t[3] = f * g.x;
              t[4] = f * g.y;
              t[5] = f * g.z;
            }
          },
          [&](const float (&t)[6], bool) {
            sx += t[0];
            sy += t[1];
            sz += t[2];
            wvx += t[3];
            wvy += t[4];
            wvz += t[5];
          },
          &own);
    } else if (st_on) {
      const int cnt = own.count(d, i);
      for_pairs<G, B, 3>(
          d, i, q, cnt, [&](int j) { return d.pos[j]; },
          [&](int, const float4& xj, bool live, float (&t)[3]) {
            const float rx = xi.x - xj.x, ry = xi.y - xj.y, rz = xi.z - xj.z;
            const float r2 = rx * rx + ry * ry + rz * rz;
            const float far = pair_w(kh, sc, rx, ry, rz, live && r2 > sc.diam2);
            const float w = r2 > sc.diam2 ? far : sc.Wd;
            const bool on = live && xj.w > 0.0f;
            t[0] = on ? -(sc.sig_m * rx * w) : NEUTRAL;
            t[1] = on ? -(sc.sig_m * ry * w) : NEUTRAL;
            t[2] = on ? -(sc.sig_m * rz * w) : NEUTRAL;
          },
          [&](const float (&t)[3], bool) {
            sx += t[0];
            sy += t[1];
            sz += t[2];
          },
          &own);
    }
    if (q != 0) return;
    float ax = sc.gx, ay = sc.gy, az = sc.gz;
    if (st_on) {
      ax += sx;
      ay += sy;
      az += sz;
    }
    if (expl) {
      ax += wvx;
      ay += wvy;
      az += wvz;
    } else if (weiler) {
      const float3 x = d.wx[i];
      const float dx = x.x - vi.x, dy = x.y - vi.y, dz = x.z - vi.z;
      ax += dx / sc.dt;
      ay += dy / sc.dt;
      az += dz / sc.dt;
      if (sc.flags & SF_WARM_CG) d.vdiff[i] = make_float4(dx, dy, dz, 0.f);
      if (bnu_on) {
        ax += wvx;
        ay += wvy;
        az += wvz;
      }
    }
    d.acc[i] = make_float4(ax, ay, az, 0.f);
    d.vel_alt[i] = make_float4(vi.x + sc.dt * ax, vi.y + sc.dt * ay, vi.z + sc.dt * az, vi.w);
    return;
  }
  float4 acc = make_float4(0.f, 0.f, 0.f, 0.f);
  if (dyn_solid(kind)) {
    float ax = sc.gx, ay = sc.gy, az = sc.gz;
    if (bnu_on) {  // reaction of the boundary viscosity (:1458-1460), gathered
      struct NF {
        float4 x, v;
        float rho;
      };
      const KernH kh(sc);
      const float4 xi = d.pos[i];
      const float Vi = -xi.w;
      for_pairs<G, B, 3>(
          d, i, q, d.nnbr[i], [&](int j) { return NF{d.pos[j], d.vel[j], d.rho[j]}; },
          [&](int, const NF& nf, bool live, float (&t)[3]) {
            const float4 xf = nf.x, vf = nf.v;
            t[0] = t[1] = t[2] = NEUTRAL;
            if (live && xf.w > 0.0f) {
              const float rx = xf.x - xi.x, ry = xf.y - xi.y, rz = xf.z - xi.z;
              const float vxy = (vf.x - vi.x) * rx + (vf.y - vi.y) * ry + (vf.z - vi.z) * rz;
              float rn, w;
              const float3 g = pair_grad<false, true>(kh, sc, rx, ry, rz, true, rn, w);
              const float ff = sc.ten_bnu * (sc.rho0 * Vi / nf.rho) * vxy / (rn * rn + sc.visc_eps);
              t[0] = -(ff * g.x);
              t[1] = -(ff * g.y);
              t[2] = -(ff * g.z);
            }
          },
          [&](const float (&t)[3], bool) {
            ax += t[0];
            ay += t[1];
            az += t[2];
          });
    }
    acc = make_float4(ax, ay, az, 0.f);
  }
  if (q != 0) return;
  d.acc[i] = acc;
  d.vel_alt[i] = vi;
}

// compute_density_adv (:1647-1667) + compute_density_error(rho0) and the loop
// test of pressure_solve (:1778-1784)
template <int G, int B>
__global__ void k_press_source(Dev d, int reduce) {
  const Ahead<G, B> own(d);
  int i, q, s;
  if (!lane_slot_scene<G>(d, i, q, s)) return;
  const SceneDev& sc = d.scenes[s];
  SceneState* st = d.state + s;
  if (!st->active_p) return;
  double v[1] = {0.0};
  if (i < sc.p_begin + sc.n && kind_of(own.info(d, i)) == KIND_FLUID) {
    const float delta = velocity_divergence<G, B>(d, sc, i, q, own);
    float da = d.rho[i] / sc.rho0 + sc.dt * delta;
    da = da > 1.0f ? da : 1.0f;
    if (q == 0) d.sa[i].x = da;
    v[0] = (double)sc.rho0 * (double)da - sc.rho0_d;
  }
  if (reduce) lane_partials<G, 1>(d, i, v, 0);
}

// Second stage of the per-scene reductions: one FINISH_THREADS-thread workgroup
// per scene adds the partials of its waves and applies the loop test of the
// solver.
//   which 0: divergence solve (:1695-1703), 1: pressure solve (:1778-1784),
//         2: CG start (after cg_guess and the first matvec),
//         4: scale of the initial guess (after cg_init, SF_WARM_CG scenes).
// (The CG's per-iteration reduction is done inside k_cg_update.)
// Thread t adds entries t, t + FINISH_THREADS, ... in order (two interleaved
// chains); the wavefront sums are combined by a fixed pairwise tree: a fixed
// order, the same bits every run.  A sweep with several lanes per particle
// leaves that many partials per 64 particles (`lanes` of the solvers' sweeps),
// which are first added by the tree that sweep's wavefront would have
// continued, so an entry has the same bits for every number of lanes.
constexpr int FINISH_THREADS = NN_FINISH_THREADS;
constexpr int FINISH_WAVES = FINISH_THREADS / 64;

__global__ __launch_bounds__(FINISH_THREADS) void k_scene_finish(Dev d, int which, int lanes, unsigned long long* report,
                                                                unsigned ticket) {
  __shared__ double red[4][FINISH_WAVES];
  const int s = blockIdx.x;
  const int t = threadIdx.x;
  const SceneDev& sc = d.scenes[s];
  SceneState* st = d.state + s;
  const bool weiler = (sc.flags & SF_HAS_FLUID) && (sc.flags & SF_VISCOSITY) && (sc.flags & SF_WEILER);
  bool part;
  switch (which) {
    case 0: part = st->active_v != 0; break;
    case 1: part = st->active_p != 0; break;
    case 2: part = weiler; break;
    default: part = weiler && (sc.flags & SF_WARM_CG); break;  // 4
  }
  if (!part) {  // uniform over the workgroup
    if (report && t == 0) report_word(report + s, ticket, 0);
    return;
  }
  // partial arrays read, and the entries each has per 64 particles (cg_init
  // and the first matvec, array 3, run four lanes per particle)
  const int nr = which == 2 ? 4 : (which == 4 ? 2 : 1);
  double tot[4] = {0.0, 0.0, 0.0, 0.0};
  for (int r = 0; r < nr; r++) {
    const int per = which < 2 ? lanes : (which == 4 || r == 3 ? 4 : 1);
    const double* src = d.partials + (long)r * 4 * d.W;
    const int lo = sc.wave_begin, hi = sc.wave_end;
    auto entry = [&](int k) {
      if (per == 1) return src[k];
      if (per == 4) return (src[4 * k] + src[4 * k + 1]) + (src[4 * k + 2] + src[4 * k + 3]);
      double v[16];
#pragma unroll
      for (int e = 0; e < 16; e++) v[e] = src[16 * k + e];
#pragma unroll
      for (int off = 1; off < 16; off <<= 1)
#pragma unroll
        for (int e = 0; e < 16; e += 2 * off) v[e] += v[e + off];
      return v[0];
    };
    double a0 = 0.0, a1 = 0.0;
    int k = lo + t;
    for (; k + FINISH_THREADS < hi; k += 2 * FINISH_THREADS) {
      a0 += entry(k);
      a1 += entry(k + FINISH_THREADS);
    }
    if (k < hi) a0 += entry(k);
    const double w = wave_sum(a0 + a1);
    if ((t & 63) == 0) red[r][t >> 6] = w;
  }
  __syncthreads();
  for (int r = 0; r < nr; r++) {  // fixed pairwise tree over the wave sums
    double w[FINISH_WAVES];
#pragma unroll
    for (int q = 0; q < FINISH_WAVES; q++) w[q] = red[r][q];
#pragma unroll
    for (int span = 1; span < FINISH_WAVES; span *= 2)
#pragma unroll
      for (int q = 0; q + span < FINISH_WAVES; q += 2 * span) w[q] += w[q + span];
    tot[r] = w[0];
  }
  if (which == 2) {  // the waves that the CG's iterations go over
    __shared__ int fluid[FINISH_WAVES];
    int n = 0;
    for (int j0 = sc.wave_begin; j0 < sc.wave_end; j0 += FINISH_THREADS) {
      const bool f = j0 + t < sc.wave_end && d.cg_list[j0 + t];
      const unsigned long long m = __ballot(f);
      if ((t & 63) == 0) fluid[t >> 6] = __popcll(m);
      __syncthreads();
      int at = n + __popcll(m & ((1ull << (t & 63)) - 1ull));
      for (int q = 0; q < FINISH_WAVES; q++) {
        if (q < t >> 6) at += fluid[q];
        n += fluid[q];
      }
      if (f) d.cg_waves[sc.wave_begin + at] = j0 + t;
      __syncthreads();
    }
    // the rest names some wave, for lanes that request one before they know n
    for (int j = sc.wave_begin + n + t; j < sc.wave_end; j += FINISH_THREADS) d.cg_waves[j] = sc.wave_begin;
    if (t == 0) st->cg_nw = n;
  }
  if (t != 0) return;
  if (which == 0) {
    const double err = tot[0] / sc.nf_d;
    const int ran = st->iter_v + 1;
    st->iter_v = ran;
    st->err_v = err;
    if (err <= sc.eta_v || ran >= sc.max_iter_v) {
      st->active_v = 0;
      if (!(err <= sc.eta_v)) st->status |= ST_NOCONV;
    }
    if (report) report_word(report + s, ticket, !(err <= sc.eta_v || ran >= sc.max_iter_v));
  } else if (which == 1) {
    const double err = tot[0] / sc.nf_d;
    const int ran = st->iter_p + 1;
    st->iter_p = ran;
    st->err_p = err;
    if (err <= sc.eta_p || ran >= sc.max_iter_p) {
      st->active_p = 0;
      if (!(err <= sc.eta_p)) st->status |= ST_NOCONV;
    }
    if (report) report_word(report + s, ticket, !(err <= sc.eta_p || ran >= sc.max_iter_p));
  } else if (which == 4) {
    // tot: e.r0, e.Ae
    st->cg_theta = tot[1] > 0.0 ? tot[0] / tot[1] : 0.0;
  } else {
    // which 2, tot: b.b, r.r, r.u, u.w of the initial residual; the CG's
    // iteration 1 reads alpha and gamma from parity slot 1
    st->cg_bb = tot[0];
    st->cg_rr = tot[1];
    st->cg_gamma2[1] = tot[2];
    st->cg_alpha2[1] = tot[2] / tot[3];
    st->iter_cg = 0;
    const int act = (tot[0] > 0.0 && tot[1] > sc.cg_tol2 * tot[0]) ? 1 : 0;
    st->active_cg = act;
    st->cg_stop_at = 0;
    if (act) atomicAdd(&d.n_active[0], 1);
  }
}

// pressure_solve_iteration_kernel, :1799-1841.  Fluid lanes update v in place
// (nothing in the sweep reads v); dynamic-solid lanes gather the reaction
// -vel_change/dt of every fluid neighbor (:1835-1841) into their acceleration.
template <int G, int B>
__global__ void k_press_update(Dev d) {
  const Ahead<G, B> own(d);
  int i, q, s;
  if (!lane_slot_scene<G>(d, i, q, s)) return;
  const SceneDev& sc = d.scenes[s];
  if (!d.state[s].active_p) return;
  if (i >= sc.p_begin + sc.n) return;
  const int kind = kind_of(own.info(d, i));
  if (kind == KIND_FLUID) {
    const KernH kh(sc);
    const float2 sai = d.sa[i];
    const float ki = (sai.x - 1.0f) * alpha_press(sc, sai.y);
    float4 v = d.vel[i];
    velocity_push<G, B, true>(d, sc, kh, i, q, own, ki,
                              [&](const PosSrc& nj) { return (nj.src - 1.0f) * alpha_press(sc, nj.alpha); }, v.x, v.y, v.z);
    if (q == 0) d.vel[i] = v;
  } else if (dyn_solid(kind)) {
    const KernH kh(sc);
    const float4 xi = d.pos[i];
    const float Vi = -xi.w;
    float4 a = d.acc[i];
    for_pairs<G, B, 3>(
        d, i, q, d.nnbr[i], [&](int f) { const float2 t = d.sa[f]; return PosSrc{d.pos[f], t.x, t.y}; },
        [&](int, const PosSrc& nf, bool live, float (&t)[3]) {
          const float4 xf = nf.x;
          const float kf = (nf.src - 1.0f) * alpha_press(sc, nf.alpha);
          t[0] = t[1] = t[2] = NEUTRAL;
          if (live && xf.w > 0.0f && fabsf(kf) > sc.eps) {
            const float3 g = pair_grad<true>(kh, sc, xf.x - xi.x, xf.y - xi.y, xf.z - xi.z, true);
            const float fk = -sc.dt * kf;
            t[0] = -(fk * (-Vi * g.x)) * 1.0f / sc.dt;
            t[1] = -(fk * (-Vi * g.y)) * 1.0f / sc.dt;
            t[2] = -(fk * (-Vi * g.z)) * 1.0f / sc.dt;
          }
        },
        [&](const float (&t)[3], bool) {
          a.x += t[0];
          a.y += t[1];
          a.z += t[2];
        });
    if (q == 0) d.acc[i] = a;
  }
}

// advect (:1086-1093) then enforce_boundary_3D for FLUID and SOLID (:1044-1080,
// :936-937), fused: each dynamic particle is touched once.
// New positions go to pos_alt (the host swaps the pair afterwards), so the
// positions the step's search used stay available until the next search.
__global__ void k_advect(Dev d) {
  int i, s;
  if (!slot_scene(d, i, s)) return;
  const SceneDev& sc = d.scenes[s];
  if (i >= sc.p_begin + sc.n) return;
  const int kind = kind_of(d.info[i]);
  float4 x = d.pos[i];
  if (kind == KIND_STATIC) {
    d.pos_alt[i] = x;
    return;
  }
  float4 v = d.vel[i];
  if (dyn_solid(kind)) {
    const float4 a = d.acc[i];
    v.x += sc.dt * a.x;
    v.y += sc.dt * a.y;
    v.z += sc.dt * a.z;
  }
  x.x += sc.dt * v.x;
  x.y += sc.dt * v.y;
  x.z += sc.dt * v.z;
  const float px = x.x, py = x.y, pz = x.z;
  float nx = 0.f, ny = 0.f, nz = 0.f;
  if (px > sc.hi0) { nx += 1.0f; x.x = sc.hi0; }
  if (px <= sc.lo0) { nx += -1.0f; x.x = sc.lo0; }
  if (py > sc.hi1) { ny += 1.0f; x.y = sc.hi1; }
  if (py <= sc.lo1) { ny += -1.0f; x.y = sc.lo1; }
  if (pz > sc.hi2) { nz += 1.0f; x.z = sc.hi2; }
  if (pz <= sc.lo2) { nz += -1.0f; x.z = sc.lo2; }
  const float nl = norm3(nx, ny, nz);
  if (nl > 1e-6f) {
    const float hx = nx / nl, hy = ny / nl, hz = nz / nl;
    const float f = sc.opc * (v.x * hx + v.y * hy + v.z * hz);
    v.x -= f * hx;
    v.y -= f * hy;
    v.z -= f * hz;
    v.x *= sc.sticky;
    v.y *= sc.sticky;
    v.z *= sc.sticky;
  }
  if (!(isfinite(x.x) && isfinite(x.y) && isfinite(x.z) && isfinite(v.x) && isfinite(v.y) && isfinite(v.z)))
    atomicOr(&d.state[s].status, ST_NAN);
  d.pos_alt[i] = x;
  d.vel[i] = v;
}

static inline dim3 grid_of(const DevRef& d, int block) { return dim3((d.h.Pn + block - 1) / block); }

void launch_begin(const DevRef& d, int begin, long cells, hipStream_t st) {
  const long n = std::max(cells, (long)d.h.nscenes);
  if (n > 0) NN_LAUNCH(k_begin, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, d.h, begin, cells);
}
void launch_publish(const DevRef& d, int list_lanes, int rho_lanes, SceneState* host, unsigned long long* report,
                    unsigned ticket, hipStream_t st) {
  if (d.h.nscenes > 0)
    NN_LAUNCH(k_publish, dim3(d.h.nscenes), dim3(PUBLISH_THREADS), 0, st, d.h, list_lanes, rho_lanes, host, report, ticket);
}
void launch_report_active(const DevRef& d, int which, unsigned long long* report, unsigned ticket, hipStream_t st) {
  NN_LAUNCH(k_report_active, dim3(1), dim3(64), 0, st, d.h, which, report, ticket);
}
void launch_density_alpha(const DevRef& d, int block, int lanes, int depth, hipStream_t st) {
  SWEEP_LAUNCH(k_density_alpha, lanes, depth, d.h.Pn, block, st, d.h);
}
void launch_div_update(const DevRef& d, int block, int lanes, int depth, hipStream_t st) {
  SWEEP_LAUNCH_4(k_div_update, lanes, depth, d.h.Pn, block, st, d.h);
}
void launch_div_source(const DevRef& d, int block, int lanes, int depth, hipStream_t st) {
  SWEEP_LAUNCH_4(k_div_source, lanes, depth, d.h.Pn, block, st, d.h);
}
void launch_nonpressure(const DevRef& d, int block, int lanes, int depth, hipStream_t st) {
  SWEEP_LAUNCH(k_nonpressure, lanes, depth, d.h.Pn, block, st, d.h);
}
void launch_press_source(const DevRef& d, int block, int lanes, int depth, int reduce, hipStream_t st) {
  SWEEP_LAUNCH_4(k_press_source, lanes, depth, d.h.Pn, block, st, d.h, reduce);
}
void launch_press_update(const DevRef& d, int block, int lanes, int depth, hipStream_t st) {
  SWEEP_LAUNCH_4(k_press_update, lanes, depth, d.h.Pn, block, st, d.h);
}
void launch_advect(const DevRef& d, int block, hipStream_t st) {
  NN_LAUNCH(k_advect, grid_of(d, block), dim3(block), 0, st, d.h);
}
void launch_scene_finish(const DevRef& d, int which, int lanes, unsigned long long* report, unsigned ticket, hipStream_t st) {
  if (d.h.nscenes > 0)
    NN_LAUNCH(k_scene_finish, dim3(d.h.nscenes), dim3(FINISH_THREADS), 0, st, d.h, which, lanes, report, ticket);
}

}  // namespace nn
