// device_common.h -- device helpers shared by the kernels of libnnsph.
//
// Every floating-point expression here is written in the operation order of the
// reference's Taichi code (cited per function) and compiled with
// -ffp-contract=off, so a result is rounded exactly as the reference's FP32
// expression would be.  Division and sqrt are IEEE correctly rounded (hipcc's
// default for single precision).
#pragma once
#include "engine.h"

namespace nn {

__device__ __forceinline__ int uniform(int v) { return __builtin_amdgcn_readfirstlane(v); }

// Slot of this thread and the scene of its wavefront; returns false for waves
// past the batch (the whole wave leaves together).
__device__ __forceinline__ bool slot_scene(const Dev& d, int& i, int& s) {
  i = blockIdx.x * blockDim.x + threadIdx.x;
  int w = uniform(i >> 6);
  if (w >= d.W) return false;
  s = uniform(d.wave_scene[w]);
  return s >= 0;
}

__device__ __forceinline__ int kind_of(int info) { return info >> 28; }
__device__ __forceinline__ int id_of(int info) { return info & 0x0FFFFFFF; }
// dynamic solids (SOLID and is_dynamic, SPH/main.py:281-282): elastic and rigid particles
__device__ __forceinline__ bool dyn_solid(int kind) { return kind == KIND_ELASTIC || kind == KIND_RIGID; }

// ---------------------------------------------------------------------------
// SPH kernel, SPH/main.py:859-880 (cubic_kernel) and :883-905 (derivative)
// ---------------------------------------------------------------------------
__device__ __forceinline__ float norm3(float x, float y, float z) { return sqrtf(x * x + y * y + z * z); }

__device__ __forceinline__ float kern_w(float h, float kW, float rn) {
  float res = 0.0f;
  float q = rn / h;
  if (q <= 1.0f) {
    if (q <= 0.5f) {
      float q2 = q * q;
      float q3 = q2 * q;
      res = kW * (6.0f * q3 - 6.0f * q2 + 1.0f);
    } else {
      float t = 1.0f - q;
      res = (kW * 2.0f) * (t * t * t);
    }
  }
  return res;
}

// gradient of W at r with |r| = rn already known (rn = norm3(r) bit for bit)
__device__ __forceinline__ float3 kern_grad(float h, float kG, float rx, float ry, float rz, float rn) {
  float3 g = make_float3(0.0f, 0.0f, 0.0f);
  float q = rn / h;
  if (rn > 1e-5f && q <= 1.0f) {
    float den = rn * h;
    float f;
    if (q <= 0.5f) {
      f = (kG * q) * (3.0f * q - 2.0f);
    } else {
      float fa = 1.0f - q;
      f = kG * ((-fa) * fa);
    }
    g.x = f * (rx / den);
    g.y = f * (ry / den);
    g.z = f * (rz / den);
  }
  return g;
}

// Word of list position k of particle i in nbr (and of its pair scalar in
// spair): groups of four positions, one int4 per particle and group.
__device__ __forceinline__ long nb_word(long P, int i, int k) { return 4 * ((long)(k >> 2) * P + i) + (k & 3); }

// ---------------------------------------------------------------------------
// The same roundings with fewer instructions.  hipcc's FP32 square root and
// division are correctly rounded over the whole range; what they spend on
// scaling (operands near overflow or underflow) a pair of particles never
// needs.  Where a scene's h lies in [2^-20, 2^20] (SF_MIDRANGE) and a pair's
// squared distance is above 1e-10 with no component in (0, 2^-100), the
// sequences below give the same bits (nn_check_roundings compares them on the
// device at hand, a root for every float of the range):
//   sqrt_mid   x rsq(x) and one residual correction
//   recip_mid  v_rcp_f32 and one Newton step, shared by every quotient of one
//              denominator
//   div_mid    a y, then two residual corrections q + (a - b q) y (Markstein,
//              IBM J. R&D 34, 1990), for quotients in the normal range (a
//              component's below it, which takes h > 2^13, is multiplied by the
//              kernel's factor of less than 2^-35 and gives 0 in either form);
//              -0 / b comes out as +0, which only a sum
//              that may itself be -0 can tell (pair_grad's SIGNED)
// A gradient has one square root and four quotients of two denominators (h
// and r h), about half of its instructions.
// ---------------------------------------------------------------------------
__device__ __forceinline__ float sqrt_mid(float x) {
  const float y = __builtin_amdgcn_rsqf(x);
  const float g = x * y;
  return __builtin_fmaf(__builtin_fmaf(-g, g, x), 0.5f * y, g);
}
__device__ __forceinline__ float recip_mid(float b) {
  const float y = __builtin_amdgcn_rcpf(b);
  return __builtin_fmaf(__builtin_fmaf(-b, y, 1.0f), y, y);
}
__device__ __forceinline__ float div_mid(float a, float b, float y) {
  float q = a * y;
  q = __builtin_fmaf(__builtin_fmaf(-b, q, a), y, q);
  return __builtin_fmaf(__builtin_fmaf(-b, q, a), y, q);
}
// some component nonzero and below 2^-100 in magnitude
__device__ __forceinline__ bool any_tiny(float x, float y, float z) {
  const unsigned tx = (__float_as_uint(x) << 1) - 1u, ty = (__float_as_uint(y) << 1) - 1u, tz = (__float_as_uint(z) << 1) - 1u;
  return min(tx, min(ty, tz)) < (27u << 24) - 1u;  // 2^-100 has biased exponent 27
}

// The kernel's radius in the form the pairs use.
struct KernH {
  float h, yh;
  bool mid;
  __device__ __forceinline__ explicit KernH(const SceneDev& sc)
      : h(sc.h), yh(recip_mid(sc.h)), mid((sc.flags & SF_MIDRANGE) != 0) {}
};

// kern_w and kern_grad's radial factor at q = |r| / h <= 1, both branches
// formed and one selected
__device__ __forceinline__ float w_of(float kW, float q) {
  const float q2 = q * q, q3 = q2 * q, t = 1.0f - q;
  const float in = kW * (6.0f * q3 - 6.0f * q2 + 1.0f), out = (kW * 2.0f) * (t * t * t);
  const float w = q <= 0.5f ? in : out;
  return q <= 1.0f ? w : 0.0f;
}
__device__ __forceinline__ float radial_of(float kG, float q) {
  const float fa = 1.0f - q;
  const float in = (kG * q) * (3.0f * q - 2.0f), out = kG * ((-fa) * fa);
  const float f = q <= 0.5f ? in : out;
  return q <= 1.0f ? f : 0.0f;
}

// One pair's |r| and gradient (kern_grad), and W (kern_w) where asked for;
// `live` lanes get kern_grad's and kern_w's bits, others anything.  Without
// SIGNED a zero component may have the other sign.
template <bool WANT_W, bool SIGNED>
__device__ __forceinline__ float3 pair_grad(const KernH& k, const SceneDev& sc, float rx, float ry, float rz, bool live,
                                            float& rn, float& w) {
  const float ss = rx * rx + ry * ry + rz * rz;
  rn = sqrt_mid(ss);
  const float q = div_mid(rn, k.h, k.yh);
  const float den = rn * k.h;
  const float y = recip_mid(den);
  const float f = radial_of(sc.kG, q);
  float ux = div_mid(rx, den, y), uy = div_mid(ry, den, y), uz = div_mid(rz, den, y);
  if (SIGNED) {
    ux = __builtin_copysignf(ux, rx);
    uy = __builtin_copysignf(uy, ry);
    uz = __builtin_copysignf(uz, rz);
  }
  float3 g = make_float3(f * ux, f * uy, f * uz);
  if (WANT_W) w = w_of(sc.kW, q);
  // 1e-10 < ss: |r| > 1e-5, so the gradient's own cut-off needs no test here;
  // a pair past q = 1 (|r| rounds below h and |r| / h above 1) takes the plain form
  if (__builtin_expect(live && (!k.mid || !(ss > 1.01e-10f) || !(q <= 1.0f) || any_tiny(rx, ry, rz)), 0)) {
    rn = norm3(rx, ry, rz);
    g = kern_grad(sc.h, sc.kG, rx, ry, rz, rn);
    if (WANT_W) w = kern_w(sc.h, sc.kW, rn);
  }
  return g;
}
template <bool SIGNED = false>
__device__ __forceinline__ float3 pair_grad(const KernH& k, const SceneDev& sc, float rx, float ry, float rz, bool live) {
  float rn, w;
  return pair_grad<false, SIGNED>(k, sc, rx, ry, rz, live, rn, w);
}
// W of one pair alone (kern_w of norm3)
__device__ __forceinline__ float pair_w(const KernH& k, const SceneDev& sc, float rx, float ry, float rz, bool live) {
  const float ss = rx * rx + ry * ry + rz * rz;
  float w = w_of(sc.kW, div_mid(sqrt_mid(ss), k.h, k.yh));
  if (__builtin_expect(live && (!k.mid || !(ss > 1.01e-10f)), 0)) w = kern_w(sc.h, sc.kW, norm3(rx, ry, rz));
  return w;
}

// ---------------------------------------------------------------------------
// Sweeps over a particle's list with G lanes per particle (1, 4 or 16, equal
// to lane groups that DPP can broadcast in).  Lane q takes list positions q,
// q + G, ...; each lane forms its own pair's terms and the group adds them in
// list order, every lane reading the owning lane's term, so the sums are the
// serial ones bit for bit whatever G is.
// ---------------------------------------------------------------------------
template <int G, int U>
__device__ __forceinline__ float lane_bcast(float v) {
  static_assert(G == 1 || G == 4 || G == 16, "lane groups");
  if constexpr (G == 1) return v;
  else if constexpr (G == 4)  // quad_perm [U, U, U, U]
    return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), U * 0x55, 0xf, 0xf, true));
  else  // row_newbcast:U
    return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0x150 + U, 0xf, 0xf, true));
}

template <int G>
__device__ __forceinline__ bool lane_slot_scene(const Dev& d, int& i, int& q, int& s) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  i = t / G;
  q = t % G;
  const int w = uniform(i >> 6);
  if (w >= d.W) return false;
  s = uniform(d.wave_scene[w]);
  return s >= 0;
}

// x + NEUTRAL == x for every x, signed zeros included: what a lane without a
// term contributes
constexpr float NEUTRAL = -0.0f;

template <int G, int N, int U, typename Add>
__device__ __forceinline__ void add_in_order(const float (&t)[N], int left, Add& add) {
  if constexpr (U < G) {
    float b[N];
#pragma unroll
    for (int n = 0; n < N; n++) b[n] = lane_bcast<G, U>(t[n]);
    add(b, U < left);
    add_in_order<G, N, U + 1>(t, left, add);
  }
}

// What a sweep of 16 lanes per particle needs of its particle, requested before
// the wave's scene is known (slots past the last read the last one's): kind,
// position, list length and the first batch's list words, whether or not the
// list is that long.  In a small scene a sweep is largely the chain of its
// loads: arguments, scene, its state, kind, length, words and neighbors were
// seven trips, and are four.  At 13,824 particles press_source went from 5.4 to
// 5.0 us, div_update from 5.8 to 4.8, nonpressure from 9.7 to 8.9, density_alpha
// from 9.8 to 9.2.  Larger scenes hide the chain behind other waves (and would
// read it for static particles in vain): there each value is loaded where it
// is used.
template <int G, int B>
struct Ahead {
  int inf, cnt, w[B];
  float4 x;
  __device__ __forceinline__ explicit Ahead(const Dev& d) {
    if constexpr (G == 16) {
      const int t = blockIdx.x * blockDim.x + threadIdx.x;
      const int i = min(t / G, d.Pn - 1), q = t % G;
      inf = d.info[i];
      cnt = d.nnbr[i];
      x = d.pos[i];
#pragma unroll
      for (int b = 0; b < B; b++) w[b] = d.nbr[nb_word(d.P, i, b * G + q)];
      __builtin_amdgcn_sched_barrier(0);  // the loads are not moved down to their first use
    }
  }
  __device__ __forceinline__ int info(const Dev& d, int i) const { return G == 16 ? inf : d.info[i]; }
  __device__ __forceinline__ int count(const Dev& d, int i) const { return G == 16 ? cnt : d.nnbr[i]; }
  __device__ __forceinline__ float4 pos(const Dev& d, int i) const { return G == 16 ? x : d.pos[i]; }
};

// B positions per lane and batch: their list words are loaded together, then
// the neighbors' data (load(j)), then term(j, data, live, t) forms the N terms
// of each (a lane past the end of the list loads its own particle and is not
// live) and add(t, ok) is called for every position in list order.
template <int G, int B, int N, typename Load, typename Term, typename Add>
__device__ __forceinline__ void for_pairs(const Dev& d, int i, int q, int cnt, Load load, Term term, Add add,
                                          const Ahead<G, B>* ahead = nullptr) {
  using T = decltype(load(0));
  const long P = d.P;
  int w[B];  // 16 lanes: the batch's list words, requested a batch ahead
  if constexpr (G == 16) {
#pragma unroll
    for (int b = 0; b < B; b++) w[b] = ahead ? ahead->w[b] : d.nbr[nb_word(P, i, b * G + q)];
  }
  for (int k0 = 0; k0 < cnt; k0 += G * B) {
    int j[B];
    T v[B];
    if constexpr (G == 1) {
      static_assert(B % 4 == 0, "whole groups of four list positions");
      const int4* groups = reinterpret_cast<const int4*>(d.nbr);
#pragma unroll
      for (int g = 0; g < B / 4; g++) {
        const int k = k0 + 4 * g;
        const int4 w = k < cnt ? groups[(long)(k >> 2) * P + i] : make_int4(i, i, i, i);
        j[4 * g + 0] = w.x;
        j[4 * g + 1] = k + 1 < cnt ? w.y : i;
        j[4 * g + 2] = k + 2 < cnt ? w.z : i;
        j[4 * g + 3] = k + 3 < cnt ? w.w : i;
      }
    } else {
#pragma unroll
      for (int b = 0; b < B; b++) {
        const int k = k0 + b * G + q;
        if constexpr (G == 16) j[b] = k < cnt ? w[b] : i;
        else j[b] = k < cnt ? d.nbr[nb_word(P, i, k)] : i;
      }
    }
#pragma unroll
    for (int b = 0; b < B; b++) v[b] = load(j[b]);
    if constexpr (G == 16) {
#pragma unroll
      for (int b = 0; b < B; b++) {
        const int k = k0 + (B + b) * G + q;
        if (k < cnt) w[b] = d.nbr[nb_word(P, i, k)];
      }
    }
#pragma unroll
    for (int b = 0; b < B; b++) {
      const int left = cnt - (k0 + b * G);
      if (left > 0) {
        float t[N];
        term(j[b], v[b], q < left, t);
        add_in_order<G, N, 0>(t, left, add);
      }
    }
  }
}

// Launch a sweep templated on its lanes per particle and positions per lane and
// batch.  `depth` (4, 8 or 16; anything else is the default 8) is the list
// positions a particle has in flight per batch, at least one per lane (one lane:
// 4 or 8; 16 took 148 us against 91 in density and 135 against 93 in strain, with
// 80 bytes of scratch a lane).  Neither changes the order of a sum.
#define SWEEP_LAUNCH_4(kern, lanes, depth, slots, block, st, ...)                                   \
  do {                                                                                             \
    const dim3 _g((unsigned)(((long)(slots) * (lanes) + (block) - 1) / (block))), _b(block);       \
    switch ((lanes) * 100 + ((depth) == 4 || (depth) == 16 ? (depth) : 8)) {                       \
      case 404: NN_LAUNCH((kern<4, 1>), _g, _b, 0, st, __VA_ARGS__); break;                        \
      case 408: NN_LAUNCH((kern<4, 2>), _g, _b, 0, st, __VA_ARGS__); break;                        \
      case 416: NN_LAUNCH((kern<4, 4>), _g, _b, 0, st, __VA_ARGS__); break;                        \
      default: NN_LAUNCH((kern<16, 2>), _g, _b, 0, st, __VA_ARGS__); break;                        \
    }                                                                                              \
  } while (0)
#define SWEEP_LAUNCH(kern, lanes, depth, slots, block, st, ...)                                     \
  do {                                                                                             \
    const dim3 _g1((unsigned)(((long)(slots) + (block) - 1) / (block))), _b1(block);               \
    if ((lanes) != 1) SWEEP_LAUNCH_4(kern, lanes, depth, slots, block, st, __VA_ARGS__);           \
    else if ((depth) == 4) NN_LAUNCH((kern<1, 4>), _g1, _b1, 0, st, __VA_ARGS__);                  \
    else NN_LAUNCH((kern<1, 8>), _g1, _b1, 0, st, __VA_ARGS__);                                    \
  } while (0)

struct PosVel {
  float4 x, v;
};
struct PosSrc {
  float4 x;
  float src, alpha;
};

// Kahan (compensated) summation
struct KSum {
  float s, c;
  __device__ __forceinline__ void add(float y) {
    float t = y - c;
    float u = s + t;
    c = (u - s) - t;
    s = u;
  }
};

// ---------------------------------------------------------------------------
// wavefront reductions (fixed butterfly order: every lane ends with the same
// bits, and the result is the same on every run)
// ---------------------------------------------------------------------------
__device__ __forceinline__ double wave_sum(double v) {
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) v += __shfl_xor(v, off, 64);
  return v;
}

// The same over values held once per G lanes, neighbors first: partials of
// fewer particles (sweeps with several lanes per particle) combine further by
// the same tree, so the sum over 64 particles has the same bits for every G.
template <int G>
__device__ __forceinline__ double tree_sum(double v) {
#pragma unroll
  for (int off = G; off <= 32; off <<= 1) v += __shfl_xor(v, off, 64);
  return v;
}

__device__ __forceinline__ float wave_max(float v) {
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) v = fmaxf(v, __shfl_xor(v, off, 64));
  return v;
}

// Per-scene FP64 reductions, first stage: every wavefront of a participating
// scene stores the sums of its particles' NR values (each held by the lane 0,
// or by all, of a particle's G lanes) in partial arrays base..base+NR-1, G
// entries per 64 particles (plain stores, no fences).  A later launch adds
// them in a fixed order: the totals are the same on every run and do not
// depend on the order in which wavefronts ran.
template <int G, int NR>
__device__ __forceinline__ void lane_partials(const Dev& d, int i, double (&v)[NR], int base) {
#pragma unroll
  for (int r = 0; r < NR; r++) v[r] = tree_sum<G>(v[r]);
  if ((threadIdx.x & 63) == 0) {
#pragma unroll
    for (int r = 0; r < NR; r++) d.partials[(long)(base + r) * 4 * d.W + i / (64 / G)] = v[r];
  }
}

// Entries of list[b, e) below `id`, eight loads in flight (one at a time, each
// member of a cell costs a trip to the L2).
__device__ __forceinline__ int lower_ids(const int* list, int b, int e, int id) {
  int n = 0;
  for (int k = b; k < e; k += 8) {
    int v[8];
#pragma unroll
    for (int u = 0; u < 8; u++) v[u] = list[min(k + u, e - 1)];
#pragma unroll
    for (int u = 0; u < 8; u++) n += k + u < e && v[u] < id ? 1 : 0;
  }
  return n;
}

// Four-lane sweeps: lanes 4i..4i+3 share particle slot i, lane q walks list
// positions k = q, q+4, ...; a wavefront covers 16 particles.  `hw` is the
// hardware wavefront index used for the partial sums.
__device__ __forceinline__ bool quad_slot_scene(const Dev& d, int& i, int& q, int& s, int& hw) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  hw = uniform(t >> 6);
  i = t >> 2;
  q = t & 3;
  const int w = hw >> 2;
  if (w >= d.W) return false;
  s = uniform(d.wave_scene[w]);
  return s >= 0;
}

// (S0 + S1) + (S2 + S3) over the four lanes of a particle; all four lanes end
// with the same bits.
__device__ __forceinline__ float quad_sum(float v) {
  v += __shfl_xor(v, 1, 64);
  v += __shfl_xor(v, 2, 64);
  return v;
}

// Weiler operator pair scalar s_ij = c_ij F(|r|) / (|r| h), c_ij =
// 10 mu_ij (m / rho_j) / (|r|^2 + 0.01 h^2); 0 where the kernel gradient is 0.
__device__ __forceinline__ float weiler_pair(const SceneDev& sc, float rx, float ry, float rz, float mui, float muj,
                                             float rhoj) {
  const float rn = norm3(rx, ry, rz);
  const float q = rn / sc.h;
  if (!(rn > 1e-5f && q <= 1.0f)) return 0.0f;
  float F;
  if (q <= 0.5f) {
    F = (sc.kG * q) * (3.0f * q - 2.0f);
  } else {
    const float fa = 1.0f - q;
    F = sc.kG * ((-fa) * fa);
  }
  const float den = rn * sc.h;
  const float muij = 0.5f * (mui + muj);
  const float c = 10.0f * muij * (sc.mass / rhoj) / ((rx * rx + ry * ry + rz * rz) + sc.visc_eps);
  return c * F / den;
}

// ---------------------------------------------------------------------------
// Polar decomposition A = R S with det R = +1 (the factor ti.polar_decompose
// returns through its SVD, SPH/main.py:1273).  Cyclic Jacobi eigen-decomposition
// of A^T A (Golub & Van Loan, Matrix Computations, Alg. 8.5.3), columns sorted by
// decreasing eigenvalue with det V kept +1, then a Givens QR of A V (the
// structure of McAdams et al. 2011); R = U V^T.  A is row-major a[3*r + c].
// ---------------------------------------------------------------------------
__device__ __forceinline__ void jacobi_rot(float* S, float* V, int p, int q) {
  float apq = S[3 * p + q];
  if (apq == 0.0f) return;
  float theta = (S[3 * q + q] - S[3 * p + p]) / (2.0f * apq);
  const float sg = theta >= 0.0f ? 1.0f : -1.0f;
  float tt;
  if (fabsf(theta) < 0x1p49f) {  // operands within the shorter forms' range
    const float den = fabsf(theta) + sqrt_mid(theta * theta + 1.0f);
    tt = div_mid(sg, den, recip_mid(den));
  } else {
    tt = sg / (fabsf(theta) + sqrtf(theta * theta + 1.0f));
  }
  const float den = sqrt_mid(tt * tt + 1.0f);  // |tt| <= 1
  float c = div_mid(1.0f, den, recip_mid(den));
  float sn = tt * c;
#pragma unroll
  for (int k = 0; k < 3; k++) {
    float skp = S[3 * k + p], skq = S[3 * k + q];
    S[3 * k + p] = c * skp - sn * skq;
    S[3 * k + q] = sn * skp + c * skq;
  }
#pragma unroll
  for (int k = 0; k < 3; k++) {
    float spk = S[3 * p + k], sqk = S[3 * q + k];
    S[3 * p + k] = c * spk - sn * sqk;
    S[3 * q + k] = sn * spk + c * sqk;
  }
#pragma unroll
  for (int k = 0; k < 3; k++) {
    float vkp = V[3 * k + p], vkq = V[3 * k + q];
    V[3 * k + p] = c * vkp - sn * vkq;
    V[3 * k + q] = sn * vkp + c * vkq;
  }
}

__device__ __forceinline__ void givens_rows(float* B, float* U, int p, int q, int col) {
  float x = B[3 * p + col], y = B[3 * q + col];
  float rn = sqrtf(x * x + y * y);
  float c = 1.0f, sn = 0.0f;
  if (rn > 0.0f) {
    c = x / rn;
    sn = y / rn;
  }
#pragma unroll
  for (int k = 0; k < 3; k++) {
    float bp = B[3 * p + k], bq = B[3 * q + k];
    B[3 * p + k] = c * bp + sn * bq;
    B[3 * q + k] = -sn * bp + c * bq;
  }
#pragma unroll
  for (int k = 0; k < 3; k++) {
    float up = U[3 * k + p], uq = U[3 * k + q];
    U[3 * k + p] = c * up + sn * uq;
    U[3 * k + q] = -sn * up + c * uq;
  }
}

__device__ __forceinline__ void polar3(const float* A, float* R) {
  float S[9];
#pragma unroll
  for (int a = 0; a < 3; a++)
#pragma unroll
    for (int b = 0; b < 3; b++) S[3 * a + b] = A[a] * A[b] + A[3 + a] * A[3 + b] + A[6 + a] * A[6 + b];
  float V[9] = {1, 0, 0, 0, 1, 0, 0, 0, 1};
  for (int sweep = 0; sweep < 6; sweep++) {
    jacobi_rot(S, V, 0, 1);
    jacobi_rot(S, V, 0, 2);
    jacobi_rot(S, V, 1, 2);
  }
  float ev[3] = {S[0], S[4], S[8]};
#pragma unroll
  for (int a = 0; a < 2; a++)
#pragma unroll
    for (int b = 0; b < 2 - a; b++)
      if (ev[b] < ev[b + 1]) {
        float t = ev[b];
        ev[b] = ev[b + 1];
        ev[b + 1] = t;
#pragma unroll
        for (int k = 0; k < 3; k++) {
          float x = V[3 * k + b];
          V[3 * k + b] = V[3 * k + b + 1];
          V[3 * k + b + 1] = -x;
        }
      }
  float B[9];
#pragma unroll
  for (int a = 0; a < 3; a++)
#pragma unroll
    for (int b = 0; b < 3; b++) B[3 * a + b] = A[3 * a] * V[b] + A[3 * a + 1] * V[3 + b] + A[3 * a + 2] * V[6 + b];
  float U[9] = {1, 0, 0, 0, 1, 0, 0, 0, 1};
  givens_rows(B, U, 0, 1, 0);
  givens_rows(B, U, 0, 2, 0);
  givens_rows(B, U, 1, 2, 1);
#pragma unroll
  for (int a = 0; a < 3; a++)
#pragma unroll
    for (int b = 0; b < 3; b++) R[3 * a + b] = U[3 * a] * V[3 * b] + U[3 * a + 1] * V[3 * b + 1] + U[3 * a + 2] * V[3 * b + 2];
}

// NonNewton viscosity models, SPH/main.py:404-459, clamped to [0, max].
__device__ __forceinline__ float nn_model(const SceneDev& c, float gam) {
  float eta;
  const float n = c.nn_n, K = c.nn_K, e0 = c.nn_e0, einf = c.nn_einf, gc = c.nn_gc;
  switch (c.nn_method) {
    case 1:
      eta = K * powf(gam, n - 1.0f);
      break;
    case 2:
      eta = einf + (e0 - einf) / (1.0f + powf(K * gam, n));
      break;
    case 3: {
      float t = sqrtf(c.nn_muc) + sqrtf(c.nn_tauy / gam);
      eta = t * t;
      break;
    }
    case 4:
      eta = einf + (e0 - einf) / (1.0f + powf(K * gam * gam, (1.0f - n) / 2.0f));
      break;
    case 5:
      if (gam < gc) eta = e0;
      else eta = gc * (e0 - einf) / gam + einf;
      break;
    case 6:
      if (gam < gc) eta = e0;
      else {
        float tau0 = e0 * gc - K * powf(gc, n);
        eta = tau0 / gam + K * powf(gam, n - 1.0f);
      }
      break;
    default:
      eta = e0;
      break;
  }
  const float mx = c.nn_max;
  if (!(eta >= 0.0f)) eta = (eta != eta) ? mx : 0.0f;
  if (eta > mx) eta = mx;
  return eta;
}

// The 9 runs' bounds from the lanes that loaded them, to every lane.
template <int G, int R>
__device__ __forceinline__ void run_table(const int* lo, const int* len, int base, int* first, int* shift, int& total) {
  if constexpr (R < 9) {
    const int b = __float_as_int(lane_bcast<G, R % G>(__int_as_float(lo[R / G])));
    const int n = __float_as_int(lane_bcast<G, R % G>(__int_as_float(len[R / G])));
    first[R] = total;
    shift[R] = b + base - total;
    total += n;
    run_table<G, R + 1>(lo, len, base, first, shift, total);
  }
}

}  // namespace nn
