// kernels_elastic.hip -- Becker et al. 2009 corotated SPH elasticity on frozen
// rest-state neighbor lists (Elasticity, SPH/main.py:1182-1375).
//
// The stress set S holds every elastic particle and every rest neighbor of one
// (the reference forms rotations and stresses for all particles, :1191, but the
// forces of elastic particles read only those of their rest neighbors).  S is
// padded per scene to 64 so a wavefront never spans two scenes.  Rest data live
// in original-index space; the current slot of particle `id` of scene s is
// p_begin + inv[p_begin + id].
#include "device_common.h"

namespace nn {

// Elasticity.initValues_kernel, :1220-1236: x_0 and the rest volume
// V0_i = m_i / (m_i W0 + sum_j m_j W_ij) on the lists of the first search.
__global__ void k_elastic_init(Dev d) {
  int i, s;
  if (!slot_scene(d, i, s)) return;
  const SceneDev& sc = d.scenes[s];
  if (i >= sc.p_begin + sc.n) return;
  const float4 xi = d.pos[i];
  const int cnt = d.nnbr[i];
  const int P = d.P;
  float den = sc.mass * sc.W0;
  for (int k = 0; k < cnt; k++) {
    const int j = d.nbr[nb_word(P, i, k)];
    const float4 xj = d.pos[j];
    const float rx = xi.x - xj.x, ry = xi.y - xj.y, rz = xi.z - xj.z;
    den += sc.mass * kern_w(sc.h, sc.kW, norm3(rx, ry, rz));
  }
  d.x0[sc.p_begin + id_of(d.info[i])] = make_float4(xi.x, xi.y, xi.z, sc.mass / den);
}

// The stress set's sweeps: 64 members per workgroup, G lanes per member (4 or
// 16, as the list sweeps), so that every wavefront of a workgroup belongs to one
// scene.
template <int G>
__device__ __forceinline__ bool member(const Dev& d, int& m, int& q, int& lane, int& s) {
  m = threadIdx.x / G;
  lane = threadIdx.x % G;
  q = blockIdx.x * 64 + m;
  s = uniform(d.s_wave_scene[blockIdx.x]);
  return s >= 0;  // the same for the whole workgroup
}

// B positions per lane and batch over the rest list of member q: load(id),
// term(data, live, t), add(t), as for_pairs
template <int G, int B, int N, typename Load, typename Term, typename Add>
__device__ __forceinline__ void for_rest(const Dev& d, int q, int lane, int cnt, int own, Load load, Term term, Add add) {
  using T = decltype(load(0));
  const long NS = d.NS;
  for (int k0 = 0; k0 < cnt; k0 += G * B) {
    int id[B];
    T v[B];
#pragma unroll
    for (int b = 0; b < B; b++) {
      const int k = k0 + b * G + lane;
      id[b] = k < cnt ? d.rest[k * NS + q] : own;
    }
#pragma unroll
    for (int b = 0; b < B; b++) v[b] = load(id[b]);
#pragma unroll
    for (int b = 0; b < B; b++) {
      const int left = cnt - (k0 + b * G);
      if (left > 0) {
        float t[N];
        term(v[b], lane < left, t);
        add_in_order<G, N, 0>(t, left, add);
      }
    }
  }
}

struct RestPair {
  float4 x, x0;
};

// computeRotations_kernel (:1249-1274) and computeStress_kernel (:1285-1323),
// fused: the stress of particle i uses only its own rotation.
//
// With one lane per member this was bound by latency: three dependent gathers
// per rest neighbor, a serial chain of 18 Jacobi rotations, and 1.5 wavefronts
// a SIMD to hide them (98,304 members).  The lanes share the gathers of both
// passes; the rotations are formed once per member, by the workgroup's first
// wavefront (64 members, all lanes busy), through LDS.  36.4 -> 30.0 us, now
// bound by its instructions (about 2,400 a wavefront, six wavefronts a SIMD: 23
// us); workgroups placed so that each XCD has one part of the set took 33.0.
template <int G>
__global__ __launch_bounds__(64 * G) void k_elastic_rot_stress(Dev d) {
  __shared__ float M[9][64];
  int m, q, lane, s;
  if (!member<G>(d, m, q, lane, s)) return;
  const SceneDev& sc = d.scenes[s];
  const KernH kh(sc);
  const int pb = sc.p_begin;
  const int pid = d.s_pid[q];
  const int own = pid < 0 ? 0 : pid;
  const int cnt = pid < 0 ? 0 : d.rest_cnt[q];
  const float4 xi = d.pos[pb + d.inv[pb + own]];
  const float4 xi0 = d.x0[pb + own];
  const auto load = [&](int id) { return RestPair{d.pos[pb + d.inv[pb + id]], d.x0[pb + id]}; };
  float A[9];
#pragma unroll
  for (int k = 0; k < 9; k++) A[k] = 0.0f;
  for_rest<G, 2, 9>(
      d, q, lane, cnt, own, load,
      [&](const RestPair& p, bool live, float* t) {
        const float dd[3] = {p.x.x - xi.x, p.x.y - xi.y, p.x.z - xi.z};
        const float d0[3] = {p.x0.x - xi0.x, p.x0.y - xi0.y, p.x0.z - xi0.z};
        const float w = sc.mass * pair_w(kh, sc, d0[0], d0[1], d0[2], live);
#pragma unroll
        for (int a = 0; a < 3; a++)
#pragma unroll
          for (int b = 0; b < 3; b++) t[3 * a + b] = live ? w * (dd[a] * d0[b]) : NEUTRAL;
      },
      [&](const float* t, bool) {
#pragma unroll
        for (int k = 0; k < 9; k++) A[k] += t[k];
      });
  if (lane == 0) {
#pragma unroll
    for (int k = 0; k < 9; k++) M[k][m] = A[k];
  }
  __syncthreads();
  float R[9];
  if (threadIdx.x < 64) {
#pragma unroll
    for (int k = 0; k < 9; k++) A[k] = M[k][threadIdx.x];
    polar3(A, R);
#pragma unroll
    for (int k = 0; k < 9; k++) M[k][threadIdx.x] = R[k];
  }
  __syncthreads();
#pragma unroll
  for (int k = 0; k < 9; k++) R[k] = M[k][m];
  float U[9];
#pragma unroll
  for (int k = 0; k < 9; k++) U[k] = 0.0f;
  for_rest<G, 2, 9>(
      d, q, lane, cnt, own, load,
      [&](const RestPair& p, bool live, float* t) {
        const float dd[3] = {p.x.x - xi.x, p.x.y - xi.y, p.x.z - xi.z};
        const float d0[3] = {p.x0.x - xi0.x, p.x0.y - xi0.y, p.x0.z - xi0.z};
        float u[3];
#pragma unroll
        for (int a = 0; a < 3; a++) u[a] = R[a] * dd[0] + R[3 + a] * dd[1] + R[6 + a] * dd[2] - d0[a];
        const float3 g3 = pair_grad(kh, sc, d0[0], d0[1], d0[2], live);
        const float g[3] = {g3.x, g3.y, g3.z};
        const float vj0 = p.x0.w;
#pragma unroll
        for (int a = 0; a < 3; a++)
#pragma unroll
          for (int b = 0; b < 3; b++) t[3 * a + b] = live ? -((vj0 * u[a]) * g[b]) : NEUTRAL;
      },
      [&](const float* t, bool) {
#pragma unroll
        for (int k = 0; k < 9; k++) U[k] += t[k];
      });
  if (lane != 0 || pid < 0) return;
  const float e[6] = {U[0], U[4], U[8], 0.5f * (U[1] + U[3]), 0.5f * (U[2] + U[6]), 0.5f * (U[5] + U[7])};
  const float Cd = sc.C_diag, Co = sc.C_off, Cs = sc.C_shear;
  const float C[6][6] = {{Cd, Co, Co, 0.f, 0.f, 0.f}, {Co, Cd, Co, 0.f, 0.f, 0.f}, {Co, Co, Cd, 0.f, 0.f, 0.f},
                         {0.f, 0.f, 0.f, Cs, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f, Cs, 0.f}, {0.f, 0.f, 0.f, 0.f, 0.f, Cs}};
  float sg[6];
#pragma unroll
  for (int a = 0; a < 6; a++) {
    float t = 0.0f;
#pragma unroll
    for (int b = 0; b < 6; b++) t += C[a][b] * e[b];
    sg[a] = t;
  }
  float4* o = d.rs + 4L * q;
  o[0] = make_float4(R[0], R[1], R[2], sg[0]);
  o[1] = make_float4(R[3], R[4], R[5], sg[1]);
  o[2] = make_float4(R[6], R[7], R[8], sg[2]);
  o[3] = make_float4(sg[3], sg[4], sg[5], 0.f);
}

__device__ __forceinline__ void sym_mat_vec(const float* M, const float* v, float* out) {
  out[0] = M[0] * v[0] + M[3] * v[1] + M[4] * v[2];
  out[1] = M[3] * v[0] + M[1] * v[1] + M[5] * v[2];
  out[2] = M[4] * v[0] + M[5] * v[1] + M[2] * v[2];
}

struct RestStress {
  float4 x0, b0, b1, b2, b3;
};

// computeForces_kernel, :1334-1375, for elastic particles: a += f / m.
// Bound by the gather of 80 bytes per rest neighbor (98,304 members: 0.26 GB in
// 21.4 us; with one lane per member 23.3).
template <int G>
__global__ __launch_bounds__(64 * G) void k_elastic_force(Dev d) {
  int m, q, lane, s;
  if (!member<G>(d, m, q, lane, s)) return;
  const SceneDev& sc = d.scenes[s];
  const KernH kh(sc);
  const int pb = sc.p_begin;
  const int pid = d.s_pid[q];
  if (pid < 0) return;
  const int i = pb + d.inv[pb + pid];
  if (kind_of(d.info[i]) != KIND_ELASTIC) return;
  const float4 xi0 = d.x0[pb + pid];
  const float vi0 = xi0.w;
  const float4* ri = d.rs + 4L * q;
  const float4 a0 = ri[0], a1 = ri[1], a2 = ri[2], a3 = ri[3];
  const float Ri[9] = {a0.x, a0.y, a0.z, a1.x, a1.y, a1.z, a2.x, a2.y, a2.z};
  const float si[6] = {a0.w, a1.w, a2.w, a3.x, a3.y, a3.z};
  float fi[3] = {0.f, 0.f, 0.f};
  for_rest<G, 1, 3>(
      d, q, lane, d.rest_cnt[q], pid,
      [&](int id) {
        const float4* rj = d.rs + 4L * (sc.s_begin + d.s_of[pb + id]);
        return RestStress{d.x0[pb + id], rj[0], rj[1], rj[2], rj[3]};
      },
      [&](const RestStress& p, bool live, float* t) {
        const float Rj[9] = {p.b0.x, p.b0.y, p.b0.z, p.b1.x, p.b1.y, p.b1.z, p.b2.x, p.b2.y, p.b2.z};
        const float sj[6] = {p.b0.w, p.b1.w, p.b2.w, p.b3.x, p.b3.y, p.b3.z};
        const float d0[3] = {p.x0.x - xi0.x, p.x0.y - xi0.y, p.x0.z - xi0.z};
        const float3 g3 = pair_grad(kh, sc, d0[0], d0[1], d0[2], live);
        const float g[3] = {g3.x, g3.y, g3.z};
        const float vj0 = p.x0.w;
        float dji[3], dij[3], sdji[3], sdij[3], fij[3], fji[3];
#pragma unroll
        for (int c = 0; c < 3; c++) {
          dji[c] = vi0 * g[c];
          dij[c] = -vj0 * g[c];
        }
        sym_mat_vec(sj, dji, sdji);
        sym_mat_vec(si, dij, sdij);
#pragma unroll
        for (int c = 0; c < 3; c++) {
          fij[c] = -vj0 * sdji[c];
          fji[c] = -vi0 * sdij[c];
        }
#pragma unroll
        for (int a = 0; a < 3; a++) {
          const float t1 = Rj[3 * a] * fij[0] + Rj[3 * a + 1] * fij[1] + Rj[3 * a + 2] * fij[2];
          const float t2 = Ri[3 * a] * fji[0] + Ri[3 * a + 1] * fji[1] + Ri[3 * a + 2] * fji[2];
          t[a] = live ? t1 - t2 : NEUTRAL;
        }
      },
      [&](const float* t, bool) {
#pragma unroll
        for (int a = 0; a < 3; a++) fi[a] += t[a];
      });
  if (lane != 0) return;
  float4 acc = d.acc[i];
  fi[0] = 0.5f * fi[0];
  fi[1] = 0.5f * fi[1];
  fi[2] = 0.5f * fi[2];
  acc.x += fi[0] / sc.mass;
  acc.y += fi[1] / sc.mass;
  acc.z += fi[2] / sc.mass;
  d.acc[i] = acc;
}

void launch_elastic_init(const DevRef& d, int block, hipStream_t st) {
  NN_LAUNCH(k_elastic_init, dim3((d.h.Pn + block - 1) / block), dim3(block), 0, st, d.h);
}
void launch_elastic_rot_stress(const DevRef& d, int lanes, hipStream_t st) {
  if (d.h.NSn <= 0) return;
  const dim3 g((d.h.NSn + 63) / 64);
  if (lanes == 16) NN_LAUNCH(k_elastic_rot_stress<16>, g, dim3(1024), 0, st, d.h);
  else NN_LAUNCH(k_elastic_rot_stress<4>, g, dim3(256), 0, st, d.h);
}
void launch_elastic_force(const DevRef& d, int lanes, hipStream_t st) {
  if (d.h.NSn <= 0) return;
  const dim3 g((d.h.NSn + 63) / 64);
  if (lanes == 16) NN_LAUNCH(k_elastic_force<16>, g, dim3(1024), 0, st, d.h);
  else NN_LAUNCH(k_elastic_force<4>, g, dim3(256), 0, st, d.h);
}

}  // namespace nn
