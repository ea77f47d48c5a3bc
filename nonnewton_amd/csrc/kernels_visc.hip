// kernels_visc.hip -- non-Newtonian viscosity and the Weiler 2018 implicit
// viscosity solver.
//
// The reference computes a per-particle non-Newtonian viscosity that no force
// reads (NonNewton, SPH/main.py:332-492) and declares an implicit solver whose
// operator is empty (Viscosity_Weiler2018, :1471-1513).  Here the strain rate
// feeds the model, the model feeds the implicit solve:
//   D_i   = (0.5 / rho_i) sum_j m_j (v_ji (x) gradW_ij + gradW_ij (x) v_ji)
//   eta_i = model(||D_i||_F)                        (kinematic, :404-459)
//   mu_i  = rho0 * eta_i   (rho0 * viscosity when the model is off)
//   (A x)_i = x_i - (dt / rho_i) sum_{fluid j} (s_ij ((x_i - x_j) . r_ij)) r_ij
//   s_ij  = c_ij F(|r_ij|) / (|r_ij| h)   (gradW_ij = F r_ij / (|r_ij| h))
//   c_ij  = 10 mu_ij (m / rho_j) / (|r_ij|^2 + 0.01 h^2),  mu_ij = (mu_i + mu_j) / 2
// Weiler et al. 2018, "A Physically Consistent Implicit Viscosity Solver for
// SPH Fluids", solved by preconditioned conjugate gradients: block-Jacobi 3x3
// preconditioner M, FP64 dot products, stop when ||r|| <= tol ||b|| with b = v.
// A is symmetric (f_i s_ij = 10 dt mu_ij m F / (rho_i rho_j |r| h (|r|^2 +
// 0.01 h^2)) with mu_ij the mean), so CG applies; it runs in the
// Chronopoulos-Gear arrangement, which needs one reduction per iteration, and
// an iteration is two launches (or, for one small scene, a pass of the loop in
// k_cg_solve):
//   update sweep:  the scene's sums of the previous iteration -> test r.r,
//                  gamma = r.u, delta = u.w, beta = gamma / gamma_old,
//                  alpha = gamma / (delta - beta gamma / alpha_old); then
//                  p = u + beta p, s = w + beta s, x += alpha p, r -= alpha s,
//                  u = M r; partials (r.r, r.u)
//   matvec sweep:  w = A u (gathers u of the neighbors); partial u.w
// The pair scalars s_ij are formed once per solve (cg_init) and stored next to
// the neighbor lists, so a CG matvec needs no sqrt or division.  cg_init and
// cg_matvec run four lanes per particle, each lane over every fourth list
// position; list sums are (S0 + S1) + (S2 + S3).
#include "device_common.h"

namespace nn {

__device__ __forceinline__ bool weiler_scene(const SceneDev& sc) {
  return (sc.flags & SF_HAS_FLUID) && (sc.flags & SF_VISCOSITY) && (sc.flags & SF_WEILER);
}

// NonNewton.calcStrainRate (:461-492, with the accumulation the reference
// omits) + the viscosity model; mu for the implicit solver.
template <int G, int B>
__global__ void k_strain(Dev d) {
  int i, q, s;
  if (!lane_slot_scene<G>(d, i, q, s)) return;
  const SceneDev& sc = d.scenes[s];
  if (!(sc.flags & SF_HAS_FLUID)) return;
  const bool nn_on = (sc.flags & SF_NON_NEWTONIAN) != 0;
  const bool weiler = weiler_scene(sc);
  if (!nn_on && !weiler) return;
  if (i >= sc.p_begin + sc.n || kind_of(d.info[i]) != KIND_FLUID) return;
  float eta = 0.0f;
  if (nn_on) {
    const KernH kh(sc);
    const float4 xi = d.pos[i];
    const float4 vi = d.vel[i];
    const int cnt = d.nnbr[i];
    // the tensor is symmetric, its two halves equal bit for bit (a sum of two
    // products does not depend on their order): six sums
    float S[6];
#pragma unroll
    for (int n = 0; n < 6; n++) S[n] = 0.0f;
    for_pairs<G, B, 6>(
        d, i, q, cnt, [&](int j) { return PosVel{d.pos[j], d.vel[j]}; },
        [&](int, const PosVel& nj, bool live, float (&t)[6]) {
          const float4 xj = nj.x, vj = nj.v;
          const float3 g3 = pair_grad(kh, sc, xi.x - xj.x, xi.y - xj.y, xi.z - xj.z, live);
          const float g[3] = {g3.x, g3.y, g3.z};
          const float vji[3] = {vj.x - vi.x, vj.y - vi.y, vj.z - vi.z};
          int n = 0;
#pragma unroll
          for (int a = 0; a < 3; a++)
#pragma unroll
            for (int b = a; b < 3; b++) t[n++] = live ? sc.mass * (vji[a] * g[b] + vji[b] * g[a]) : NEUTRAL;
        },
        [&](const float (&t)[6], bool) {
#pragma unroll
          for (int n = 0; n < 6; n++) S[n] += t[n];
        });
    const float f = 0.5f / d.rho[i];
    const float M[9] = {S[0], S[1], S[2], S[1], S[3], S[4], S[2], S[4], S[5]};
    float n2 = 0.0f;
#pragma unroll
    for (int e = 0; e < 9; e++) {
      const float t = f * M[e];
      n2 += t * t;
    }
    const float gam = sqrtf(n2);
    eta = nn_model(sc, gam);
    if (q == 0) {
      d.gam[i] = gam;
      d.eta[i] = eta;
    }
  }
  if (weiler && q == 0) d.mu[i] = (nn_on ? eta : sc.nu) * sc.rho0;
}

// Start of a solve, b = v.  Pair scalars s_ij (stored), the inverse diagonal
// block M, r0 = b - A b (into wr).  With SF_WARM_CG also A e for the previous
// solve's e = x - v (into ww) and partial sums of (e.r0, e.Ae), from which the
// scene finish forms theta = (e.r0) / (e.Ae); k_cg_guess then starts CG from
// u = M r
__device__ __forceinline__ float3 precondition(float4 w0, float2 w1, float3 r) {
  return make_float3(w0.x * r.x + w0.y * r.y + w0.z * r.z, w0.y * r.x + w0.w * r.y + w1.x * r.z,
                     w0.z * r.x + w1.x * r.y + w1.y * r.z);
}

// Partial arrays of iteration k, one entry per 64 slots: (r.r, r.u), by parity,
// since update k + 1 reads them while writing its own, and u.w (in words that
// neither those arrays nor k_cg_solve's use).
__device__ __forceinline__ int cg_rr(int k) { return 4 + 2 * (k & 1); }
constexpr long CG_UW = 31;  // times d.W

// x0 = b + theta e, r = r0 - theta A e.
__global__ void k_cg_init(Dev d) {
  int i, q, s, hw;
  if (!quad_slot_scene(d, i, q, s, hw)) return;
  const SceneDev& sc = d.scenes[s];
  if (!weiler_scene(sc)) return;
  double v[2] = {0.0, 0.0};
  const bool valid = i < sc.p_begin + sc.n && kind_of(d.info[i]) == KIND_FLUID;
  const bool warm = (sc.flags & SF_WARM_CG) != 0;
  float ax = 0.f, ay = 0.f, az = 0.f;  // sum for A v
  float bx = 0.f, by = 0.f, bz = 0.f;  // sum for A e
  float m0 = 0.f, m1 = 0.f, m2 = 0.f, m3 = 0.f, m4 = 0.f, m5 = 0.f;
  float4 xi = make_float4(0.f, 0.f, 0.f, 0.f), vi = xi, ei = xi;
  if (valid) {
    xi = d.pos[i];
    vi = d.vel[i];
    if (warm) ei = d.vdiff[i];
    const float mui = d.mu[i];
    const int cnt = d.nnbr[i];
    const long P = d.P;
    // one neighbor's contribution, in list order
    auto pair_term = [&](int k, const float4& xj, const float4& vj, const float4& ej, float muj, float rhoj) {
      float sij = 0.0f;
      if (xj.w > 0.0f) {
        const float rx = xi.x - xj.x, ry = xi.y - xj.y, rz = xi.z - xj.z;
        sij = weiler_pair(sc, rx, ry, rz, mui, muj, rhoj);
        const float t = sij * ((vi.x - vj.x) * rx + (vi.y - vj.y) * ry + (vi.z - vj.z) * rz);
        ax += t * rx;
        ay += t * ry;
        az += t * rz;
        if (warm) {
          const float te = sij * ((ei.x - ej.x) * rx + (ei.y - ej.y) * ry + (ei.z - ej.z) * rz);
          bx += te * rx;
          by += te * ry;
          bz += te * rz;
        }
        m0 += sij * rx * rx;
        m1 += sij * rx * ry;
        m2 += sij * rx * rz;
        m3 += sij * ry * ry;
        m4 += sij * ry * rz;
        m5 += sij * rz * rz;
      }
      d.spair[nb_word(P, i, k)] = sij;
    };
    const float4 zero4 = make_float4(0.f, 0.f, 0.f, 0.f);
    // two list positions of this lane per batch, their loads issued together
    for (int k = q; k < cnt; k += 8) {
      const bool two = k + 4 < cnt;
      const int j0 = d.nbr[nb_word(P, i, k)];
      const int j1 = two ? d.nbr[nb_word(P, i, k + 4)] : i;
      const float4 x0 = d.pos[j0], x1 = d.pos[j1];
      const float4 v0 = d.vel[j0], v1 = d.vel[j1];
      const float mu0 = d.mu[j0], mu1 = d.mu[j1];
      const float r0 = d.rho[j0], r1 = d.rho[j1];
      const float4 e0 = warm ? d.vdiff[j0] : zero4;
      const float4 e1 = warm ? d.vdiff[j1] : zero4;
      pair_term(k, x0, v0, e0, mu0, r0);
      if (two) pair_term(k + 4, x1, v1, e1, mu1, r1);
    }
  }
  ax = quad_sum(ax);
  ay = quad_sum(ay);
  az = quad_sum(az);
  if (warm) {
    bx = quad_sum(bx);
    by = quad_sum(by);
    bz = quad_sum(bz);
  }
  m0 = quad_sum(m0);
  m1 = quad_sum(m1);
  m2 = quad_sum(m2);
  m3 = quad_sum(m3);
  m4 = quad_sum(m4);
  m5 = quad_sum(m5);
  // the positions the CG gathers, for every particle of the scene
  if (q == 0 && i < sc.p_begin + sc.n) {
    const float4 p = valid ? xi : d.pos[i];
    d.xu[i].p = make_float3(p.x, p.y, p.z);
  }
  if (valid && q == 0) {
    const float f = sc.dt / d.rho[i];
    const float qx = vi.x - f * ax, qy = vi.y - f * ay, qz = vi.z - f * az;
    const float rrx = vi.x - qx, rry = vi.y - qy, rrz = vi.z - qz;
    const float d00 = 1.0f - f * m0, d01 = -f * m1, d02 = -f * m2;
    const float d11 = 1.0f - f * m3, d12 = -f * m4, d22 = 1.0f - f * m5;
    const float c00 = d11 * d22 - d12 * d12, c01 = d02 * d12 - d01 * d22, c02 = d01 * d12 - d02 * d11;
    const float c11 = d00 * d22 - d02 * d02, c12 = d01 * d02 - d00 * d12, c22 = d00 * d11 - d01 * d01;
    const float det = d00 * c00 + d01 * c01 + d02 * c02;
    float4 w0;
    float2 w1;
    if (det > 0.0f && det == det) {
      const float id = 1.0f / det;
      w0 = make_float4(c00 * id, c01 * id, c02 * id, c11 * id);
      w1 = make_float2(c12 * id, c22 * id);
    } else {
      w0 = make_float4(1.f, 0.f, 0.f, 1.f);
      w1 = make_float2(0.f, 1.f);
    }
    d.wd0[i] = w0;
    d.wd1[i] = w1;
    d.wr[i] = make_float3(rrx, rry, rrz);
    if (warm) {
      const float zx = ei.x - f * bx, zy = ei.y - f * by, zz = ei.z - f * bz;
      d.ww[i] = make_float3(zx, zy, zz);
      v[0] = (double)ei.x * (double)rrx + (double)ei.y * (double)rry + (double)ei.z * (double)rrz;
      v[1] = (double)ei.x * (double)zx + (double)ei.y * (double)zy + (double)ei.z * (double)zz;
    }
  }
  lane_partials<4, 2>(d, i, v, 0);
}

// x0 = b + theta e, r = r0 - theta A e (x0 = b, r = r0 without SF_WARM_CG),
// u = M r; partials (b.b, r.r, r.u).
__global__ void k_cg_guess(Dev d) {
  int i, s;
  if (!slot_scene(d, i, s)) return;
  const SceneDev& sc = d.scenes[s];
  if (!weiler_scene(sc)) return;
  double v[3] = {0.0, 0.0, 0.0};
  if (i < sc.p_begin + sc.n && kind_of(d.info[i]) == KIND_FLUID) {
    const float4 b = d.vel[i];
    float3 r = d.wr[i];
    float3 x = make_float3(b.x, b.y, b.z);
    if (sc.flags & SF_WARM_CG) {
      const float th = (float)d.state[s].cg_theta;
      const float4 e = d.vdiff[i];
      const float3 z = d.ww[i];
      x = make_float3(b.x + th * e.x, b.y + th * e.y, b.z + th * e.z);
      r = make_float3(r.x - th * z.x, r.y - th * z.y, r.z - th * z.z);
    }
    const float3 u = precondition(d.wd0[i], d.wd1[i], r);
    d.wx[i] = x;
    d.wr[i] = r;
    d.xu[i].u = u;
    v[0] = (double)b.x * (double)b.x + (double)b.y * (double)b.y + (double)b.z * (double)b.z;
    v[1] = (double)r.x * (double)r.x + (double)r.y * (double)r.y + (double)r.z * (double)r.z;
    v[2] = (double)r.x * (double)u.x + (double)r.y * (double)u.y + (double)r.z * (double)u.z;
  }
  lane_partials<1, 3>(d, i, v, 0);
  // the partials of the iterations, of k_cg_solve's words or of waves that
  // k_cg_update and k_cg_matvec pass by; the waves that they go over
  const bool fluid = __any(kind_of(d.info[i]) == KIND_FLUID && i < sc.p_begin + sc.n);
  if ((threadIdx.x & 63) < 16)
    reinterpret_cast<unsigned long long*>(d.partials)[(16L + (threadIdx.x & 63)) * d.W + (i >> 6)] = 0ull;
  if ((threadIdx.x & 63) == 0) d.cg_list[i >> 6] = fluid;
}

// w = A u of particle i by its four lanes (u gathered from the neighbors, in
// the 24-byte records with the positions).  D list positions of a lane per
// batch: their list words and pair scalars, then their neighbors' records, are
// loaded before any of them is used (a shorter chain of dependent loads), and
// the next batch's list words and pair scalars are requested right after this
// batch's records, so that they arrive while this batch is summed; the terms
// are added in list order whatever D is.  A pair with s_ij = 0 -- every
// neighbor that is not fluid -- adds nothing and is skipped, so the neighbor's
// u is never read there.  Returns u.w of the particle (lane 0; else 0).
// (Slots without a particle are of no kind, so validity needs no scene word.)
template <int D>
__device__ __forceinline__ double matvec_row(const Dev& d, const SceneDev& sc, int i, int q) {
  const long P = d.P;
  // one round of loads: the particle's own data and its lanes' first positions
  // (every slot has room for MAX_NB; those past the list's end are replaced)
  static_assert(4 * D <= MAX_NB, "list positions of the first batch");
  int jn[D];
  float sn[D];
#pragma unroll
  for (int e = 0; e < D; e++) {
    jn[e] = d.nbr[nb_word(P, i, q + 4 * e)];
    sn[e] = d.spair[nb_word(P, i, q + 4 * e)];
  }
  const XU own = d.xu[i];
  const int cnt = d.nnbr[i];
  const float rho = d.rho[i];
  const bool valid = kind_of(d.info[i]) == KIND_FLUID;
  float ax = 0.f, ay = 0.f, az = 0.f;
  const float3 xi = own.p, ui = own.u;
  if (valid) {
#pragma unroll
    for (int e = 0; e < D; e++) {
      const bool in = q + 4 * e < cnt;
      jn[e] = in ? jn[e] : i;
      sn[e] = in ? sn[e] : 0.0f;
    }
    for (int k = q; k < cnt; k += 4 * D) {
      int j[D];
      float sp[D];
      float3 xj[D], uj[D];
#pragma unroll
      for (int e = 0; e < D; e++) {
        j[e] = jn[e];
        sp[e] = sn[e];
      }
#pragma unroll
      for (int e = 0; e < D; e++) {
        const XU nb = d.xu[j[e]];
        xj[e] = nb.p;
        uj[e] = nb.u;
      }
      // the next batch's list words and pair scalars, in flight while this
      // batch's records arrive
#pragma unroll
      for (int e = 0; e < D; e++) {
        const int kk = k + 4 * D + 4 * e;
        const bool in = kk < cnt;
        jn[e] = in ? d.nbr[nb_word(P, i, kk)] : i;
        sn[e] = in ? d.spair[nb_word(P, i, kk)] : 0.0f;
      }
#pragma unroll
      for (int e = 0; e < D; e++) {
        if (sp[e] != 0.0f) {
          const float rx = xi.x - xj[e].x, ry = xi.y - xj[e].y, rz = xi.z - xj[e].z;
          const float t = sp[e] * ((ui.x - uj[e].x) * rx + (ui.y - uj[e].y) * ry + (ui.z - uj[e].z) * rz);
          ax += t * rx;
          ay += t * ry;
          az += t * rz;
        }
      }
    }
  }
  ax = quad_sum(ax);
  ay = quad_sum(ay);
  az = quad_sum(az);
  if (!valid || q != 0) return 0.0;
  const float f = sc.dt / rho;
  const float wx = ui.x - f * ax, wy = ui.y - f * ay, wz = ui.z - f * az;
  d.ww[i] = make_float3(wx, wy, wz);
  return (double)ui.x * (double)wx + (double)ui.y * (double)wy + (double)ui.z * (double)wz;
}

// The start product (after cg_guess): every Weiler scene; partial u.w into
// array 3, per 16 particles.
template <int D>
__global__ void k_cg_matvec_start(Dev d) {
  int i, q, s, hw;
  if (!quad_slot_scene(d, i, q, s, hw)) return;
  const SceneDev& sc = d.scenes[s];
  if (!weiler_scene(sc)) return;
  double v[1] = {matvec_row<D>(d, sc, i, q)};
  lane_partials<4, 1>(d, i, v, 3);
}

// Matvec k over the waves that update k listed (the scenes still iterating):
// workgroup = 256 threads = the four lanes of one wave's 64 particles, looping
// over the list; partial u.w per 64 particles into array CG_UW.
constexpr int MVL_THREADS = 256;

template <int D>
__global__ __launch_bounds__(MVL_THREADS) void k_cg_matvec(Dev d, int k) {
  __shared__ double red[2][MVL_THREADS / 64];
  const int count = d.cg_list_n[k % 3];
  const int* list = d.cg_list + (long)(k % 3) * d.W;
  const int q = threadIdx.x & 3;
  int flip = 0;
  for (int u = blockIdx.x; u < count; u += gridDim.x, flip ^= 1) {
    const int w = list[u];
    const int s = uniform(d.wave_scene[w]);
    const double v = tree_sum<4>(matvec_row<D>(d, d.scenes[s], w * 64 + (threadIdx.x >> 2), q));
    if ((threadIdx.x & 63) == 0) red[flip][threadIdx.x >> 6] = v;
    __syncthreads();
    if (threadIdx.x == 0)
      d.partials[CG_UW * d.W + w] = (red[flip][0] + red[flip][1]) + (red[flip][2] + red[flip][3]);
  }
}

// The scene's sums of iteration k - 1 -- r.r, r.u (arrays cg_rr(k - 1) and the
// next) and u.w (CG_UW) -- by every workgroup of the scene in one fixed
// order, so that all obtain the same bits: the 512 threads add the
// 64-particle entries t, t + 512, ... in two interleaved chains, then the
// wavefront sums and a fixed pairwise tree.
constexpr int SUM_THREADS = 512;
__device__ __forceinline__ void scene_sums(const Dev& d, const SceneDev& sc, int k, double (*red)[SUM_THREADS / 64],
                                           double (&tot)[3]) {
  const int t = threadIdx.x;
  const double* src[3] = {d.partials + (long)cg_rr(k - 1) * 4 * d.W, d.partials + (long)(cg_rr(k - 1) + 1) * 4 * d.W,
                          d.partials + CG_UW * d.W};
  const int lo = sc.wave_begin, hi = sc.wave_end;
  double a[3][2] = {};
  for (int j = lo + t; j < hi; j += 2 * SUM_THREADS) {  // six loads in flight
    double e[3][2];
#pragma unroll
    for (int c = 0; c < 2; c++)
#pragma unroll
      for (int r = 0; r < 3; r++) e[r][c] = j + c * SUM_THREADS < hi ? src[r][j + c * SUM_THREADS] : 0.0;
#pragma unroll
    for (int c = 0; c < 2; c++)
#pragma unroll
      for (int r = 0; r < 3; r++) a[r][c] += e[r][c];
  }
#pragma unroll
  for (int r = 0; r < 3; r++) {
    const double w = wave_sum(a[r][0] + a[r][1]);
    if ((t & 63) == 0) red[r][t >> 6] = w;
  }
  __syncthreads();
#pragma unroll
  for (int r = 0; r < 3; r++) {
    double w[SUM_THREADS / 64];
#pragma unroll
    for (int v = 0; v < SUM_THREADS / 64; v++) w[v] = red[r][v];
#pragma unroll
    for (int span = 1; span < SUM_THREADS / 64; span *= 2)
#pragma unroll
      for (int v = 0; v + span < SUM_THREADS / 64; v += 2 * span) w[v] += w[v + span];
    tot[r] = w[0];
  }
}

// The decision of iteration k for a scene, from its sums of iteration k - 1:
//   converged (r.r <= tol^2 b.b) or k - 1 iterations reached the limit: the
//     scene leaves the solve (`lead` records it); returns false
//   otherwise beta = gamma / gamma_old, alpha = gamma / (delta - beta gamma /
//     alpha_old) (iteration 1 takes alpha from the start reduction, beta = 0)
__device__ __forceinline__ bool cg_decide(const Dev& d, const SceneDev& sc, SceneState* st, int k, bool lead,
                                          double (*red)[SUM_THREADS / 64], double& al, double& be) {
  if (k == 1) {
    al = st->cg_alpha2[1];
    be = 0.0;
    return true;
  }
  const int q = (k - 1) & 1;
  const double bb = st->cg_bb, ga_old = st->cg_gamma2[q], al_old = st->cg_alpha2[q];
  double tot[3];
  scene_sums(d, sc, k, red, tot);
  const double rr = tot[0], ga = tot[1], de = tot[2];
  const int it = k - 1;
  const bool conv = rr <= sc.cg_tol2 * bb;
  if (conv || it >= sc.max_iter_cg) {
    if (lead) {
      st->iter_cg = it;
      st->cg_rr = rr;
      st->cg_stop_at = k;
      if (!conv) st->status |= ST_NOCONV;
      atomicSub(&d.n_active[0], 1);
    }
    return false;
  }
  be = ga / ga_old;
  al = ga / (de - be * ga / al_old);
  if (lead) {
    st->iter_cg = it;
    st->cg_rr = rr;
    st->cg_gamma2[k & 1] = ga;
    st->cg_alpha2[k & 1] = al;
  }
  return true;
}

// a scene that iterates on lists its waves for what follows in iteration k
__device__ __forceinline__ void cg_list_scene(const Dev& d, const SceneDev& sc, int k) {
  __shared__ int base;
  const int nw = d.state[&sc - d.scenes].cg_nw;
  if (threadIdx.x == 0) base = atomicAdd(&d.cg_list_n[k % 3], nw);
  __syncthreads();
  int* out = d.cg_list + (long)(k % 3) * d.W + base;
  for (int m = threadIdx.x; m < nw; m += SUM_THREADS) out[m] = d.cg_waves[sc.wave_begin + m];
}

// Iteration k of the CG with the scene's reduction of iteration k - 1 done in
// the same launch (no separate reduction kernel per iteration).  Workgroup =
// up to CG_UPD_WAVES of the scene's waves with fluid (cg_waves; d.cg_blocks has
// room for all its waves).  Every workgroup takes the scene's decision
// (cg_decide) and then p = u + beta p, s = w + beta s, x += alpha p,
// r -= alpha s, u = M r, with partials (r.r, r.u) into arrays cg_rr(k) and the
// next.
//
// 20 MB in and out at 131,072 particles: 4.3 us at the rate of a large copy,
// and a chain of loads through the tables and the sums before it.  Requested
// after the decision, with the sums' loads four at a time, the vectors made the
// update take 11.8 us; requested before it, with the sums' loads together, 10.6;
// with the wave's number requested beside the tables' words as well, 10.5
// (workgroups of 4 or 16 waves: 10.9, 10.1).  Waves without fluid, a fifth
// there and half of a small scene's, made up a tenth of a 64-scene pool's tick.
constexpr int UPD_THREADS = 64 * CG_UPD_WAVES;
static_assert(UPD_THREADS == SUM_THREADS, "scene_sums runs in k_cg_update's workgroups");

// Which scenes take part is read from state that no workgroup of this launch
// changes in a way that matters to the others: active_cg is set by the start
// reduction, and cg_stop_at by an earlier update -- or by this one's first
// workgroup of the scene, as k, which reads the same as 0 here.  (Had that
// workgroup cleared a flag that the others read, a workgroup whose waves read
// it on both sides of the store would split at the barrier below, some waves
// leaving and the rest reducing with wave sums never written.)  A workgroup of
// a scene stopping now reaches the same decision from the same sums and
// leaves without writing.
__global__ __launch_bounds__(UPD_THREADS) void k_cg_update(Dev d, int k) {
  __shared__ double red[3][SUM_THREADS / 64];
  const int2 e = d.cg_blocks[blockIdx.x];
  const int s = e.x;
  const SceneDev& sc = d.scenes[s];
  SceneState* st = d.state + s;
  const int t = threadIdx.x;
  const int w = d.cg_waves[min(e.y + (t >> 6), d.W - 1)];  // with the tables' words, not after them
  if (blockIdx.x == 0 && t == 0) d.cg_list_n[(k + 1) % 3] = 0;  // for iteration k + 1
  const int stop = st->cg_stop_at;
  if (!st->active_cg || (stop != 0 && stop < k)) return;  // uniform over the workgroup
  // waves [m0, m0 + CG_UPD_WAVES) of the scene's waves with fluid
  const int m0 = e.y - sc.wave_begin, m = m0 + (t >> 6), nw = st->cg_nw;
  if (m0 != 0 && m0 >= nw) return;
  // the particle's vectors are requested before the decision that scales them
  const int i = (m < nw ? w : sc.wave_begin) * 64 + (t & 63);
  const int inf = d.info[i];
  const float3 ww = d.ww[i], po = d.wp[i], so = d.ws[i];
  float3 x = d.wx[i], r = d.wr[i];
  const float4 w0 = d.wd0[i];
  const float2 w1 = d.wd1[i];
  double al, be;
  if (!cg_decide(d, sc, st, k, e.y == sc.wave_begin && t == 0, red, al, be)) return;
  if (e.y == sc.wave_begin) cg_list_scene(d, sc, k);
  const float alf = (float)al, bef = (float)be;
  if (m >= nw) return;  // whole waves past the list
  double v[2] = {0.0, 0.0};
  if (i < sc.p_begin + sc.n && kind_of(inf) == KIND_FLUID) {
    const float3 u = precondition(w0, w1, r);  // as the last update stored it for the matvec
    float3 p, sv;
    if (k == 1) {
      p = u;
      sv = ww;
    } else {
      p = make_float3(u.x + bef * po.x, u.y + bef * po.y, u.z + bef * po.z);
      sv = make_float3(ww.x + bef * so.x, ww.y + bef * so.y, ww.z + bef * so.z);
    }
    x.x += alf * p.x;
    x.y += alf * p.y;
    x.z += alf * p.z;
    r.x -= alf * sv.x;
    r.y -= alf * sv.y;
    r.z -= alf * sv.z;
    const float3 z = precondition(w0, w1, r);
    d.wp[i] = p;
    d.ws[i] = sv;
    d.wx[i] = x;
    d.wr[i] = r;
    d.xu[i].u = z;
    v[0] = (double)r.x * (double)r.x + (double)r.y * (double)r.y + (double)r.z * (double)r.z;
    v[1] = (double)r.x * (double)z.x + (double)r.y * (double)z.y + (double)r.z * (double)z.z;
  }
  lane_partials<1, 2>(d, i, v, cg_rr(k));
}

// The whole solve of a batch of one scene of at most CG_SOLVE_WAVES waves in
// one launch: a workgroup of 1,024 threads per wave of 64 slots, 16 lanes per
// particle, all resident at once, each keeping its particles' vectors, list
// words, pair scalars and the neighbors' positions and preconditioners in
// registers through the iterations.  An iteration has one exchange: every
// workgroup stores its particles' r, w and s and its partials of (r.r, r.u,
// u.w) as 64-bit words of half a partial under the iteration's number; every
// workgroup reads all workgroups' words until they are the iteration's, adds
// the partials in the order of scene_sums, and forms the neighbors' updated u
// again from their r, w and s.  Two copies of r, w, s and of the words: a
// workgroup may be one iteration ahead of another's reads, and cannot be two
// (it waits for that one's words).
//
// What bounds an iteration is the latency of that exchange: a store's way to
// memory, the words' to the other XCDs, the neighbors' data back, about 1 us
// each.  6.3 us at 27 workgroups, 7.0 at 102, 8.0 at 222; as an update and a
// matvec launch an iteration takes 13 to 15 us at these sizes, as one launch
// that recomputes the neighbors' updates 9 to 11.
//
// The wait is bounded (CG_SOLVE_POLLS polls, and none after `patience`
// exchanges, which is for the tests of what follows a wait in vain): should a workgroup not have been
// scheduled by then -- the device held by other work -- the waiting ones set
// n_active[1] and leave, a workgroup that comes later finds it at its 64th poll
// (about 60 us) instead of waiting as long again, and the host repeats the solve with k_cg_update and k_cg_matvec.  Nothing that
// such a repetition starts from is written here.
//
// Order: lane 4 q + a takes list positions q + 4 a + 16 b, so the four lanes of
// q together hold the positions of lane q of k_cg_matvec and add them in its
// order.
constexpr int SOLVE_THREADS = 1024;
constexpr int SOLVE_B = (MAX_NB + 15) / 16;  // list positions per lane
constexpr int SOLVE_KEEP = 2;                // of which this many stay in registers
constexpr int CG_SOLVE_POLLS = 1 << 14;  // about 15 ms

// The exchanged data goes past the L2 of an XCD, which does not see another
// XCD's: stores and loads of device scope (buffer accesses with SC1; the
// partials' words as relaxed atomics of agent scope, which are the same).
// A store of device scope is done, for the wait on the store counter, when it
// has reached memory.  (With plain accesses between release and acquire
// fences, whose write-backs and invalidations of a whole L2 queue up, an
// iteration of 222 workgroups took 13 us.)
constexpr int DEVICE_SCOPE = 16;
typedef unsigned u32x4 __attribute__((ext_vector_type(4)));

// three arrays of 16 bytes a slot: (r, w.x), (w.y, w.z, s.x, s.y), (s.z)
struct CgExchange {
  __amdgpu_buffer_rsrc_t a, b, c;
  __device__ __forceinline__ CgExchange(float4* pa, float4* pb, float4* pc, int slots)
      : a(__builtin_amdgcn_make_buffer_rsrc(pa, 0, slots * 16, 0x00027000)),
        b(__builtin_amdgcn_make_buffer_rsrc(pb, 0, slots * 16, 0x00027000)),
        c(__builtin_amdgcn_make_buffer_rsrc(pc, 0, slots * 16, 0x00027000)) {}
  __device__ __forceinline__ void load(int j, float3& r, float3& w, float3& s) const {
    const u32x4 e = __builtin_amdgcn_raw_buffer_load_b128(a, 16 * j, 0, DEVICE_SCOPE);
    const u32x4 f = __builtin_amdgcn_raw_buffer_load_b128(b, 16 * j, 0, DEVICE_SCOPE);
    const unsigned g = __builtin_amdgcn_raw_buffer_load_b32(c, 16 * j, 0, DEVICE_SCOPE);
    r = make_float3(__uint_as_float(e.x), __uint_as_float(e.y), __uint_as_float(e.z));
    w = make_float3(__uint_as_float(e.w), __uint_as_float(f.x), __uint_as_float(f.y));
    s = make_float3(__uint_as_float(f.z), __uint_as_float(f.w), __uint_as_float(g));
  }
  __device__ __forceinline__ void store(int i, float3 r, float3 w, float3 s) const {
    const u32x4 e = {__float_as_uint(r.x), __float_as_uint(r.y), __float_as_uint(r.z), __float_as_uint(w.x)};
    const u32x4 f = {__float_as_uint(w.y), __float_as_uint(w.z), __float_as_uint(s.x), __float_as_uint(s.y)};
    __builtin_amdgcn_raw_buffer_store_b128(e, a, 16 * i, 0, DEVICE_SCOPE);
    __builtin_amdgcn_raw_buffer_store_b128(f, b, 16 * i, 0, DEVICE_SCOPE);
    __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(s.z), c, 16 * i, 0, DEVICE_SCOPE);
  }
};

__global__ __launch_bounds__(SOLVE_THREADS) void k_cg_solve(Dev d, int patience) {
  __shared__ double red[3][SUM_THREADS / 64];
  __shared__ double part[3][SOLVE_THREADS / 64];
  __shared__ float fixed[SOLVE_KEEP][9][SOLVE_THREADS];  // a lane's neighbors' position and M
  SceneState* st = d.state;
  if (!st->active_cg) return;  // the same for every workgroup: set by an earlier launch
  const SceneDev& sc = d.scenes[0];
  const int t = threadIdx.x, w = blockIdx.x, nw = gridDim.x;
  const int g = t & 15, q = g >> 2, a = g & 3;
  const long P = d.P;
  const int i = w * 64 + (t >> 4);
  const bool valid = i < sc.n && kind_of(d.info[i]) == KIND_FLUID;
  const int cnt = valid ? d.nnbr[i] : 0;
  // word e of a workgroup: half e & 1 of partial e / 2, under its iteration
  unsigned long long* words = reinterpret_cast<unsigned long long*>(d.partials + 16L * d.W);
  // copy 1 (first written in iteration 1) in arrays that the non-pressure
  // forces and the advection write before anything reads them; copy 0
  // (iteration 2, when every workgroup has read its pair scalars) in theirs
  float4* sp4 = reinterpret_cast<float4*>(d.spair);
  const CgExchange ex0(sp4, sp4 + P, sp4 + 2 * P, nw * 64);
  const CgExchange ex1(d.pos_alt, d.vel_alt, d.acc, nw * 64);
  // what does not change through the solve
  int j[SOLVE_KEEP];
  float sp[SOLVE_B];
#pragma unroll
  for (int b = 0; b < SOLVE_B; b++) {
    const int m = q + 4 * a + 16 * b;
    if (b < SOLVE_KEEP) j[b] = m < cnt ? d.nbr[nb_word(P, i, m)] : i;
    sp[b] = m < cnt ? d.spair[nb_word(P, i, m)] : 0.0f;
  }
#pragma unroll
  for (int b = 0; b < SOLVE_KEEP; b++) {  // (read back by the same thread)
    const float3 pb = d.xu[j[b]].p;
    const float4 mj0 = d.wd0[j[b]];
    const float2 mj1 = d.wd1[j[b]];
    const float e[9] = {pb.x, pb.y, pb.z, mj0.x, mj0.y, mj0.z, mj0.w, mj1.x, mj1.y};
#pragma unroll
    for (int m = 0; m < 9; m++) fixed[b][m][t] = e[m];
  }
  const float3 pi = d.xu[i].p;
  const float4 mi0 = d.wd0[i];
  const float2 mi1 = d.wd1[i];
  const float f = valid ? sc.dt / d.rho[i] : 0.0f;
  float3 r = d.wr[i], ww = d.ww[i], x = d.wx[i], u = d.xu[i].u, p = u, sv = ww;
  const double bb = st->cg_bb;
  double alpha = st->cg_alpha2[1], gamma_old = st->cg_gamma2[1], rr = 0.0;
  int k = 1;
  for (;; k++) {
    double al = alpha, be = 0.0;
    const bool first = k == 1;
    float3 rn[SOLVE_KEEP], wn[SOLVE_KEEP], sn[SOLVE_KEEP];  // the kept neighbors' r, w, s
    auto neighbor = [&](int m, float3& rj, float3& wj, float3& sj) {
      if (k & 1) ex0.load(m, rj, wj, sj);
      else ex1.load(m, rj, wj, sj);
    };
    if (first) {
#pragma unroll
      for (int b = 0; b < SOLVE_KEEP; b++) {
        rn[b] = d.wr[j[b]];
        wn[b] = sn[b] = d.ww[j[b]];
      }
    } else {
      // every workgroup's r, w, s and partials of iteration k - 1 are there
      bool late = false;
      const auto gave_up = [&] { return __any(__hip_atomic_load(&d.n_active[1], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0); };
      double mine[3] = {0.0, 0.0, 0.0};
      if (t < CG_SOLVE_WAVES) {
        const unsigned long long* from = words + 6L * ((k - 1) & 1) * d.W + t;
        bool there = t >= nw;  // the words of workgroup t are in
        const int limit = k - 1 > patience ? 0 : CG_SOLVE_POLLS;
        for (int polls = 0; !__all(there); polls++) {
          if (polls >= limit || ((polls & 63) == 63 && gave_up())) {
            late = true;
            break;
          }
          if (there) continue;
          // the first word alone is polled; the others are seldom later
          const unsigned long long e0 = __hip_atomic_load(from, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
          if ((int)(e0 >> 32) != k - 1) continue;
          unsigned long long e[5];
          there = true;
#pragma unroll
          for (int m = 0; m < 5; m++) e[m] = __hip_atomic_load(from + (m + 1L) * d.W, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
          for (int m = 0; m < 5; m++) there = there && (int)(e[m] >> 32) == k - 1;
          mine[0] = __hiloint2double((int)(unsigned)e[0], (int)(unsigned)e0);
          mine[1] = __hiloint2double((int)(unsigned)e[2], (int)(unsigned)e[1]);
          mine[2] = __hiloint2double((int)(unsigned)e[4], (int)(unsigned)e[3]);
        }
      }
      if (t < SUM_THREADS) {
#pragma unroll
        for (int e = 0; e < 3; e++) mine[e] = wave_sum(mine[e]);
        if ((t & 63) == 0) {
#pragma unroll
          for (int e = 0; e < 3; e++) red[e][t >> 6] = mine[e];
        }
      }
      if (__syncthreads_or(late)) {
        if (t == 0) atomicOr(&d.n_active[1], 1);
        return;
      }
#pragma unroll
      for (int b = 0; b < SOLVE_KEEP; b++) neighbor(j[b], rn[b], wn[b], sn[b]);
      double tot[3];
#pragma unroll
      for (int e = 0; e < 3; e++) {
        double v[SUM_THREADS / 64];
#pragma unroll
        for (int m = 0; m < SUM_THREADS / 64; m++) v[m] = red[e][m];
#pragma unroll
        for (int span = 1; span < SUM_THREADS / 64; span *= 2)
#pragma unroll
          for (int m = 0; m + span < SUM_THREADS / 64; m += 2 * span) v[m] += v[m + span];
        tot[e] = v[0];
      }
      rr = tot[0];
      if (rr <= sc.cg_tol2 * bb || k - 1 >= sc.max_iter_cg) break;
      be = tot[1] / gamma_old;
      al = tot[1] / (tot[2] - be * tot[1] / alpha);
      gamma_old = tot[1];
      alpha = al;
    }
    const float alf = (float)al, bef = (float)be;
    double v[3] = {0.0, 0.0, 0.0};
    if (valid) {
      if (first) {
        p = u;
        sv = ww;
      } else {
        p = make_float3(u.x + bef * p.x, u.y + bef * p.y, u.z + bef * p.z);
        sv = make_float3(ww.x + bef * sv.x, ww.y + bef * sv.y, ww.z + bef * sv.z);
      }
      x.x += alf * p.x;
      x.y += alf * p.y;
      x.z += alf * p.z;
      r.x -= alf * sv.x;
      r.y -= alf * sv.y;
      r.z -= alf * sv.z;
      u = precondition(mi0, mi1, r);
      float ax = 0.f, ay = 0.f, az = 0.f;
#pragma unroll
      for (int b = 0; b < SOLVE_B; b++) {
        if (16 * b < cnt) {
          float tt[3] = {NEUTRAL, NEUTRAL, NEUTRAL};
          if (sp[b] != 0.0f) {  // (0 for every neighbor that is not fluid)
            float3 rj, wj, so, pb;
            float4 mj0;
            float2 mj1;
            if (b < SOLVE_KEEP) {
              rj = rn[b];
              wj = wn[b];
              so = sn[b];
              const float(*e)[SOLVE_THREADS] = fixed[b];
              pb = make_float3(e[0][t], e[1][t], e[2][t]);
              mj0 = make_float4(e[3][t], e[4][t], e[5][t], e[6][t]);
              mj1 = make_float2(e[7][t], e[8][t]);
            } else {
              const int m = d.nbr[nb_word(P, i, q + 4 * a + 16 * b)];
              if (first) {
                rj = d.wr[m];
                wj = so = d.ww[m];
              } else {
                neighbor(m, rj, wj, so);
              }
              pb = d.xu[m].p;
              mj0 = d.wd0[m];
              mj1 = d.wd1[m];
            }
            const float3 sj = first ? wj : make_float3(wj.x + bef * so.x, wj.y + bef * so.y, wj.z + bef * so.z);
            rj.x -= alf * sj.x;
            rj.y -= alf * sj.y;
            rj.z -= alf * sj.z;
            const float3 uj = precondition(mj0, mj1, rj);
            const float rx = pi.x - pb.x, ry = pi.y - pb.y, rz = pi.z - pb.z;
            const float e = sp[b] * ((u.x - uj.x) * rx + (u.y - uj.y) * ry + (u.z - uj.z) * rz);
            tt[0] = e * rx;
            tt[1] = e * ry;
            tt[2] = e * rz;
          }
          auto add = [&](const float (&e)[3], bool) {
            ax += e[0];
            ay += e[1];
            az += e[2];
          };
          add_in_order<4, 3, 0>(tt, 4, add);
        }
      }
      auto quads = [](float e) {  // (S0 + S1) + (S2 + S3) over the quads of the row
        return (lane_bcast<16, 0>(e) + lane_bcast<16, 4>(e)) + (lane_bcast<16, 8>(e) + lane_bcast<16, 12>(e));
      };
      ax = quads(ax);
      ay = quads(ay);
      az = quads(az);
      ww = make_float3(u.x - f * ax, u.y - f * ay, u.z - f * az);
      v[0] = (double)r.x * (double)r.x + (double)r.y * (double)r.y + (double)r.z * (double)r.z;
      v[1] = (double)r.x * (double)u.x + (double)r.y * (double)u.y + (double)r.z * (double)u.z;
      v[2] = (double)u.x * (double)ww.x + (double)u.y * (double)ww.y + (double)u.z * (double)ww.z;
      if (g == 0) {
        if (k & 1) ex1.store(i, r, ww, sv);
        else ex0.store(i, r, ww, sv);
      }
    }
#pragma unroll
    for (int e = 0; e < 3; e++) {
      v[e] = tree_sum<16>(v[e]);
      if ((t & 63) == 0) part[e][t >> 6] = v[e];
    }
    __builtin_amdgcn_s_waitcnt(0);  // this wavefront's stores are done
    __syncthreads();
    if (t < 64) {
      if (t < 6) {
        double e[SOLVE_THREADS / 64];
#pragma unroll
        for (int m = 0; m < SOLVE_THREADS / 64; m++) e[m] = part[t >> 1][m];
#pragma unroll
        for (int off = 1; off < SOLVE_THREADS / 64; off <<= 1)
#pragma unroll
          for (int m = 0; m < SOLVE_THREADS / 64; m += 2 * off) e[m] += e[m + off];
        const unsigned half = (unsigned)((t & 1) ? __double2hiint(e[0]) : __double2loint(e[0]));
        __hip_atomic_store(words + (6L * (k & 1) + t) * d.W + w, ((unsigned long long)(unsigned)k << 32) | half,
                           __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
    }
  }
  if (valid && g == 0) d.wx[i] = x;
  if (w == 0 && t == 0) {
    st->iter_cg = k - 1;
    st->cg_rr = rr;
    if (!(rr <= sc.cg_tol2 * bb)) st->status |= ST_NOCONV;
    d.n_active[0] = 0;
  }
}

static inline dim3 grid_of(const DevRef& d, int block) { return dim3((d.h.Pn + block - 1) / block); }
// four-lane sweeps: a workgroup covers the particles of a one-lane workgroup
// (fewer workgroups to dispatch when most scenes have left the solve)
static inline int quad_block(int block) { return block * 4 <= 1024 ? block * 4 : 1024; }
static inline dim3 grid4_of(const DevRef& d, int block) {
  const int qb = quad_block(block);
  return dim3((4 * d.h.Pn + qb - 1) / qb);
}

void launch_strain(const DevRef& d, int block, int lanes, int depth, hipStream_t st) {
  SWEEP_LAUNCH(k_strain, lanes, depth, d.h.Pn, block, st, d.h);
}
void launch_cg_init(const DevRef& d, int block, hipStream_t st) {
  NN_LAUNCH(k_cg_init, grid4_of(d, block), dim3(quad_block(block)), 0, st, d.h);
}
void launch_cg_guess(const DevRef& d, int block, hipStream_t st) {
  NN_LAUNCH(k_cg_guess, grid_of(d, block), dim3(block), 0, st, d.h);
}
#define CG_DEPTH_LAUNCH(kern, depth, g, b, st, ...)                    \
  do {                                                                \
    switch (depth) {                                                  \
      case 1: NN_LAUNCH(kern<1>, g, b, 0, st, __VA_ARGS__); break;     \
      case 4: NN_LAUNCH(kern<4>, g, b, 0, st, __VA_ARGS__); break;     \
      case 8: NN_LAUNCH(kern<8>, g, b, 0, st, __VA_ARGS__); break;     \
      default: NN_LAUNCH(kern<2>, g, b, 0, st, __VA_ARGS__); break;    \
    }                                                                 \
  } while (0)
void launch_cg_matvec_start(const DevRef& d, int block, int depth, hipStream_t st) {
  CG_DEPTH_LAUNCH(k_cg_matvec_start, depth, grid4_of(d, block), dim3(quad_block(block)), st, d.h);
}
void launch_cg_matvec(const DevRef& d, int depth, int k, int grid, hipStream_t st) {
  CG_DEPTH_LAUNCH(k_cg_matvec, depth, dim3(grid > 0 ? grid : 1), dim3(MVL_THREADS), st, d.h, k);
}
void launch_cg_update(const DevRef& d, int nblocks, int k, hipStream_t st) {
  if (nblocks > 0) NN_LAUNCH(k_cg_update, dim3(nblocks), dim3(UPD_THREADS), 0, st, d.h, k);
}
void launch_cg_solve(const DevRef& d, int waves, int patience, hipStream_t st) {
  NN_LAUNCH(k_cg_solve, dim3(waves), dim3(SOLVE_THREADS), 0, st, d.h, patience);
}

}  // namespace nn
