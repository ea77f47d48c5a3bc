// surface.hip -- particle surface reconstruction on the GPU: the path
// SRTool.dual_contouring runs (SPH/surf_recon/srtool.py:1264-1304), behind the
// nn_surface_* entry points of include/nnsph.h.
//
// Stages (one or more launches each, all on the object's stream):
//   bounds      voxel range of the particles (integer min/max atomics)
//   hash        per-voxel particle lists, <= 64 each, sorted by particle index
//               (update_particles / add_particle, :1193-1196, :820-823)
//   aniso       x_bar, C_i, G_i per particle (pre_process_data, :1007-1112)
//   field       the blocks the particles' boxes write are marked; then one
//               workgroup per 8^3 vertex tile sums, per vertex, the poly6 values
//               (generate_fluid_field, :1239-1251) and the anisotropic values
//               (generate_smooth_fluid_field_impl, :1136-1157) of the particles
//               whose boxes reach it
//   stats       FP64 mean and sd of the negative values (density_field_stats, :1437-1456)
//   smooth      bilateral 27-point pass(es) (smooth_sdf_impl, :1459-1484)
//   contour     cubes with a crossing numbered by a scan, their dual-contouring
//               points (dual_contouring_impl, :1532-1596) and triangle counts,
//               a scan, the triangles (dual_contouring_polygen, :1708-1763)
//   normals     per mesh vertex (process_normal, :1384-1410)
//
// Layout in HBM: a dense vertex grid over the 32^3 blocks that can be written
// (vertex (x, y, z) at origin + (x, y, z) * voxel_size, z fastest), one byte per
// block for "written" (the reference's sparse leaf blocks: its loops visit
// exactly those, and an unwritten vertex reads 0).  The field is accumulated in
// 2^-32 fixed point (FP64 sums of each tile where they are exact, int64 sums
// elsewhere), so its value does not depend on the order in which the particles'
// contributions are added (a gather per tile here, a scatter per particle in the
// reference), then rounded once to FP32.  The
// reference adds FP32 with atomics in no defined order.  Every other
// expression is FP32 in the reference's operation order (-ffp-contract=off).
#include <hip/hip_runtime.h>

#include <chrono>
#include <cmath>
#include <cstdint>
#include <cstring>
#include <initializer_list>
#include <string>
#include <vector>

#include "batch.h"
#include "device_common.h"

namespace nn {
namespace sr {

constexpr int BLOCK = 32;
constexpr int MAX_PER_VOXEL = 64;  // max_num_particle_per_voxel, srtool.py:685
constexpr double FIX_SCALE = 4294967296.0;
constexpr double FIX_INV = 1.0 / 4294967296.0;
constexpr float MAX_CONTRIB = 1048576.0f;  // |contribution| bound keeping the int64 sums exact

enum { ERR_OUT_OF_GRID = 1, ERR_VOXEL_OVERFLOW = 2, ERR_RANGE = 4 };

struct K {
  float o[3], vs, sr, iso, vol, acoef, c48, c16, lam, lam1, kr, ks, kn, c2pi;
  int R, off, aniso, n;
  int vlo[3], vdim[3];
  int glo[3], gdim[3], bdim[3];
  long nvox, nvert, nblock;
  const float* pos;  // 3 per particle, caller order
  const float* vel;  // 3 per particle when the velocity channels are on, else null
  float *vfield, *mvel;  // 3 per vertex, 3 per mesh vertex
  int mid;                   // the smooth radius lies where sqrt_mid and div_mid hold
  float cvs3;                // voxel_size^3 (contribution_coeff, :1165)
  int* pvox;         // 3 per particle: its voxel
  int *vcount, *vstart, *vslot, *vlist;
  float *G, *xbar;
  unsigned char* active;
  float4* sorted;  // per entry of vlist: position, particle
  float4* rec;     // REC_QUADS per entry of vlist
  float *field0, *field, *tmp;
  int *flag, *cube_id;      // per vertex of the grid: its cube's code and mesh vertex + 1
  int *cubes, *tcount, *tstart;  // per mesh vertex: its cube, its triangles
  float *verts, *normals;
  int* faces;
  int* err;
  int* bounds;     // min xyz, max xyz
  double* stats;   // sum, count, mean (as float), sd (as float)
};

// ------------------------------------------------------------------ helpers

__device__ __forceinline__ float norm3f(float x, float y, float z) { return sqrtf(x * x + y * y + z * z); }
// exp for the bilateral weights (x <= 0 there).  Cody-Waite reduction
// x = k ln2 + r with ln2 split into a 16-bit high part (k ln2_hi exact) and a
// low part, the degree-7 Taylor polynomial of e^r in Horner form, exact
// scaling by 2^k; below 2^-125 the result is 0.
__device__ __forceinline__ float sr_expf(float x) {
  if (x != x) return x;
  if (x < -87.0f) return 0.0f;
  if (x > 88.0f) return INFINITY;
  const float k = rintf(x * 1.44269504f);
  const float r = (x - k * 0.693145751953125f) - k * 1.428606765330187e-06f;
  float p = 1.98412698e-4f;
  p = p * r + 1.38888889e-3f;
  p = p * r + 8.33333333e-3f;
  p = p * r + 4.16666667e-2f;
  p = p * r + 1.66666667e-1f;
  p = p * r + 0.5f;
  p = p * r + 1.0f;
  p = p * r + 1.0f;
  return ldexpf(p, (int)k);
}

// cyclic Jacobi eigen-decomposition of a symmetric 3x3 (Golub & Van Loan,
// Alg. 8.5.2), 6 sweeps; ev = the diagonal, V = the accumulated rotations
__device__ __forceinline__ void eig3(const float* A, float* ev, float* V) {
  float S[9];
#pragma unroll
  for (int k = 0; k < 9; k++) S[k] = A[k];
#pragma unroll
  for (int k = 0; k < 9; k++) V[k] = (k % 4) == 0 ? 1.0f : 0.0f;
  for (int sweep = 0; sweep < 6; sweep++) {
    jacobi_rot(S, V, 0, 1);
    jacobi_rot(S, V, 0, 2);
    jacobi_rot(S, V, 1, 2);
  }
  ev[0] = S[0];
  ev[1] = S[4];
  ev[2] = S[8];
}

__device__ __forceinline__ long gidx(const K& k, int gx, int gy, int gz) {
  return ((long)gx * k.gdim[1] + gy) * k.gdim[2] + gz;
}
__device__ __forceinline__ long bidx(const K& k, int gx, int gy, int gz) {
  return ((long)(gx / BLOCK) * k.bdim[1] + gy / BLOCK) * k.bdim[2] + gz / BLOCK;
}
// value at vertex (x, y, z) (absolute vertex coordinates); 0 if unwritten (the
// fields hold 0 in blocks that no box touches)
__device__ __forceinline__ float val_at(const K& k, const float* f, int x, int y, int z) {
  const int gx = x - k.glo[0], gy = y - k.glo[1], gz = z - k.glo[2];
  if (gx < 0 || gy < 0 || gz < 0 || gx >= k.gdim[0] || gy >= k.gdim[1] || gz >= k.gdim[2]) return 0.0f;
  return f[gidx(k, gx, gy, gz)];
}
// get_mapped_position (:795-796)
__device__ __forceinline__ void vpos(const K& k, int x, int y, int z, float* p) {
  p[0] = (float)x * k.vs + k.o[0];
  p[1] = (float)y * k.vs + k.o[1];
  p[2] = (float)z * k.vs + k.o[2];
}
// get_voxel_index (:799-803): truncation toward zero
__device__ __forceinline__ void voxel_of(const K& k, const float* p, int* v) {
  v[0] = (int)((p[0] - k.o[0]) / k.vs);
  v[1] = (int)((p[1] - k.o[1]) / k.vs);
  v[2] = (int)((p[2] - k.o[2]) / k.vs);
}
// poly6_weight (:1213-1227)
__device__ __forceinline__ float poly6(const K& k, float rx, float ry, float rz, float h) {
  const float rn = norm3f(rx, ry, rz);
  float res = 0.0f;
  if (rn <= h) {
    float tmp = h * h;
    res = tmp - rn * rn;
    res = res * res * res;
    tmp = tmp * tmp * tmp * tmp * h;
    res = k.acoef * res / tmp;
  }
  return res;
}
__device__ __forceinline__ unsigned long long fix_of(float v) {
  return (unsigned long long)(long long)rint((double)v * FIX_SCALE);
}
__device__ __forceinline__ int mult_axis(int v, int c, int off, int R) {
  const int lo = c - off, hi = c - off + R - 1;
  return (v >= lo && v <= hi) + (v - 1 >= lo && v - 1 <= hi);
}

// ------------------------------------------------------------------ stages

__global__ void k_fill_i32(int* p, int v, long n) {
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = v;
}
__global__ void k_fill_u8(unsigned char* p, long n) {
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = 0;
}

__global__ void k_start(K k) {
  const int t = threadIdx.x;
  if (t < 6) k.bounds[t] = t < 3 ? INT32_MAX : INT32_MIN;
  if (t == 6) *k.err = 0;
}

// voxel range of the particles: a workgroup min/max in LDS, then one atomic
// per bound per workgroup (integers: the order does not matter)
constexpr int BOUNDS_THREADS = 256;
__global__ __launch_bounds__(BOUNDS_THREADS) void k_bounds(K k) {
  __shared__ int red[6][BOUNDS_THREADS];
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  const int t = threadIdx.x;
  int v[3] = {INT32_MAX, INT32_MAX, INT32_MAX}, u[3] = {INT32_MIN, INT32_MIN, INT32_MIN};
  if (i < k.n) {
    const float* p = k.pos + 3 * (long)i;
    bool ok = true;
    for (int a = 0; a < 3; a++) {
      const float tt = (p[a] - k.o[a]) / k.vs;
      if (!(tt > -1.0f && tt < 1.0e8f)) ok = false;
    }
    if (ok) {
      int w[3];
      voxel_of(k, p, w);
      for (int a = 0; a < 3; a++)
        if (w[a] < 0) ok = false;
      if (ok)
        for (int a = 0; a < 3; a++) v[a] = u[a] = w[a];
    }
    if (!ok) atomicOr(k.err, ERR_OUT_OF_GRID);
  }
  for (int a = 0; a < 3; a++) {
    red[a][t] = v[a];
    red[3 + a][t] = u[a];
  }
  __syncthreads();
  for (int span = BOUNDS_THREADS / 2; span > 0; span >>= 1) {
    if (t < span)
      for (int a = 0; a < 3; a++) {
        red[a][t] = min(red[a][t], red[a][t + span]);
        red[3 + a][t] = max(red[3 + a][t], red[3 + a][t + span]);
      }
    __syncthreads();
  }
  if (t < 3 && red[t][0] != INT32_MAX) {
    atomicMin(k.bounds + t, red[t][0]);
    atomicMax(k.bounds + 3 + t, red[3 + t][0]);
  }
}

__device__ __forceinline__ long vkey(const K& k, const int* v) {
  return ((long)(v[0] - k.vlo[0]) * k.vdim[1] + (v[1] - k.vlo[1])) * k.vdim[2] + (v[2] - k.vlo[2]);
}

__global__ void k_vcount(K k) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= k.n) return;
  int v[3];
  voxel_of(k, k.pos + 3 * (long)i, v);
  k.pvox[3 * (long)i] = v[0];
  k.pvox[3 * (long)i + 1] = v[1];
  k.pvox[3 * (long)i + 2] = v[2];
  const int slot = atomicAdd(k.vcount + vkey(k, v), 1);
  if (slot >= MAX_PER_VOXEL) atomicOr(k.err, ERR_VOXEL_OVERFLOW);
  k.vslot[i] = slot;
}

__global__ void k_vplace(K k, int* bucket) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= k.n) return;
  int v[3];
  voxel_of(k, k.pos + 3 * (long)i, v);
  bucket[k.vstart[vkey(k, v)] + k.vslot[i]] = i;
}

// a voxel's particles in increasing index (a particle's place is the number of
// lower indices there; a voxel with too many is reported, k_vcount): vlist, and
// their positions in the same order
__global__ void k_vsort(K k, const int* bucket) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= k.n) return;
  const int i = bucket[t];
  const float* x = k.pos + 3 * (long)i;
  int v[3];
  voxel_of(k, x, v);
  const long key = vkey(k, v);
  const int b = k.vstart[key], e = k.vstart[key + 1];
  int dest = t;
  if (e - b <= MAX_PER_VOXEL) {
    dest = b + lower_ids(bucket, b, e, i);
  }
  k.vlist[dest] = i;
  k.sorted[dest] = make_float4(x[0], x[1], x[2], __int_as_float(i));
}

// Record of list entry m (particle j = vlist[m]), for the field's tiles:
//   (x_bar, det G), (G row 0, support radius), (G row 1, voxel x), (G row 2,
//   voxel y), (voxel z, position)
// Beyond the support radius the anisotropic value is exactly 0: there
// |G d| > 1.  G = V diag(1 / (h s)) V^T with V orthonormal to FP32 rounding,
// so |G d| >= |d| / (h max |s|) less a few ulp; 1% covers them.
constexpr int REC_QUADS = 5;
// Lists and sums of k_aniso, a workgroup of one wavefront with 16 lanes per
// particle.  Data crosses lanes of a group through LDS, which a wavefront's
// accesses reach in order; wave_order() keeps the compiler to that order.
constexpr int AN_GROUPS = 4;   // particles of a workgroup
constexpr int AN_CAND = 128;   // candidates laid out at a time
constexpr int AN_LIST = 1024;  // neighbors held for the second pass
constexpr int AN_BATCH = 32;   // neighbors whose terms are formed together
struct AnisoLds {
  int cand[AN_GROUPS][AN_CAND];
  unsigned short list[AN_GROUPS][AN_LIST];  // less a base
  float term[AN_GROUPS][6][AN_BATCH + 4];
};
__device__ __forceinline__ void wave_order() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// The particles within r2 (to 1e-5) of one at x in the order of pre_process_data
// (voxel dx, dy, dz nested, z fastest, then the voxel's list), as entries of
// vlist less `base`, into the group's list; full(count) takes the list whenever
// it may not hold the next 64.  Returns the entries left in the list.
//
// A voxel's particles are contiguous in vlist and the voxels of one (x, y)
// column are consecutive, so a column is one range: the lanes find those of 32
// columns at a time, restricted to the voxels that can hold a particle closer
// than r2 (rows and column ends are trimmed with a margin of 1e-3 voxel around
// each voxel and 1e-4 of r2), lay their entries end to end, and test 16 a round.
// Particles left out have weight 0 and would add +0 to every sum.
template <typename Full>
__device__ __forceinline__ int find_neighbors(const K& k, AnisoLds& lds, int g, int q, const int* v, float4 x, float r2,
                                              int& base, Full full) {
  const int R = k.R, off = k.off;
  const float reach = r2 * 1.0001f;
  const float reach2 = reach * reach;
  const float m = 1e-3f * k.vs;
  int* cand = lds.cand[g];
  unsigned short* list = lds.list[g];
  const int base_lane = threadIdx.x & 48;
  const float within = r2 * 1.00001f, within2 = within * within;
  int cnt = 0;
  for (int col0 = 0; col0 < R * R; col0 += 32) {
    int b[2], len[2];
#pragma unroll
    for (int s = 0; s < 2; s++) {
      const int col = col0 + 2 * q + s;
      b[s] = len[s] = 0;
      const int cx = v[0] + col / R - off, cy = v[1] + col % R - off;
      if (col < R * R && cx >= max(0, k.vlo[0]) && cx < k.vlo[0] + k.vdim[0] && cy >= max(0, k.vlo[1]) &&
          cy < k.vlo[1] + k.vdim[1]) {
        const float lx = (float)cx * k.vs + k.o[0] - m, hx = lx + k.vs + 2.0f * m;
        const float gx = fmaxf(0.0f, fmaxf(lx - x.x, x.x - hx));
        const float ly = (float)cy * k.vs + k.o[1] - m, hy = ly + k.vs + 2.0f * m;
        const float gy = fmaxf(0.0f, fmaxf(ly - x.y, x.y - hy));
        const float rest = reach2 - (gx * gx + gy * gy);
        if (rest > 0.0f) {
          const float zr = sqrtf(rest);
          int z0 = (int)floorf((x.z - zr - k.o[2]) / k.vs) - 1;
          int z1 = (int)floorf((x.z + zr - k.o[2]) / k.vs) + 1;
          z0 = max(max(z0, v[2] - off), max(0, k.vlo[2]));
          z1 = min(min(z1, v[2] - off + R - 1), k.vlo[2] + k.vdim[2] - 1);
          if (z0 <= z1) {
            const long at = ((long)(cx - k.vlo[0]) * k.vdim[1] + (cy - k.vlo[1])) * k.vdim[2] - k.vlo[2];
            b[s] = k.vstart[at + z0];
            len[s] = k.vstart[at + z1 + 1] - b[s];
          }
        }
      }
    }
    int incl = len[0] + len[1];  // scanned over the group
#pragma unroll
    for (int d = 1; d < 16; d <<= 1) {
      const int u = __shfl_up(incl, d, 16);
      if (q >= d) incl += u;
    }
    const int total = __float_as_int(lane_bcast<16, 15>(__int_as_float(incl)));
    const int first[2] = {incl - len[0] - len[1], incl - len[1]};
    for (int c0 = 0; c0 < total; c0 += AN_CAND) {
#pragma unroll
      for (int s = 0; s < 2; s++)
        for (int t = max(0, c0 - first[s]); t < min(len[s], c0 + AN_CAND - first[s]); t++) cand[first[s] + t - c0] = b[s] + t;
      wave_order();
      const int n = min(AN_CAND, total - c0);
      for (int r = 0, lim; r < n; r = lim) {
        lim = min(r + 64, n);  // entries increase along the sequence
        if (cnt + 64 > AN_LIST || cand[lim - 1] - base > 0xFFFF) {
          if (cnt) full(cnt);
          cnt = 0;
          base = cand[r];
          while (cand[lim - 1] - base > 0xFFFF) lim--;
        }
        int e[4];
        float4 p[4];
#pragma unroll
        for (int u = 0; u < 4; u++) {
          const int c = r + 16 * u + q;
          e[u] = cand[c < lim ? c : r];
          p[u] = k.sorted[e[u]];
        }
#pragma unroll
        for (int u = 0; u < 4; u++) {
          const float dx = x.x - p[u].x, dy = x.y - p[u].y, dz = x.z - p[u].z;
          const bool hit = r + 16 * u + q < lim && dx * dx + dy * dy + dz * dz < within2;
          const int hits = (int)(__ballot(hit) >> base_lane) & 0xFFFF;
          if (hit) list[cnt + __popc(hits & ((1 << q) - 1))] = (unsigned short)(e[u] - base);
          cnt += __popc(hits);
        }
      }
      wave_order();  // cand is written again
    }
  }
  return cnt;
}

// N sums over `cnt` entries of the group's list, in order: every lane forms the
// terms of its entries, lane n < N adds up sum n.
template <int N, typename Term>
__device__ __forceinline__ void add_neighbors(const K& k, AnisoLds& lds, int g, int q, int base, int cnt, float& acc,
                                              Term term) {
  const unsigned short* list = lds.list[g];
  for (int c0 = 0; c0 < cnt; c0 += AN_BATCH) {
    float4 p[AN_BATCH / 16];
#pragma unroll
    for (int u = 0; u < AN_BATCH / 16; u++) {
      const int c = c0 + 16 * u + q;
      p[u] = k.sorted[base + list[c < cnt ? c : 0]];
    }
#pragma unroll
    for (int u = 0; u < AN_BATCH / 16; u++) {
      float t[N];
      const bool on = c0 + 16 * u + q < cnt;
      term(p[u], on, t);
#pragma unroll
      for (int n = 0; n < N; n++) lds.term[g][n][16 * u + q] = on ? t[n] : NEUTRAL;
    }
    wave_order();
    if (q < N) {
      const float4* row = reinterpret_cast<const float4*>(lds.term[g][q]);
#pragma unroll
      for (int h = 0; h < AN_BATCH / 4; h++) {
        const float4 t = row[h];
        acc += t.x;
        acc += t.y;
        acc += t.z;
        acc += t.w;
      }
    }
    wave_order();  // the terms are written again
  }
}

// pre_process_data (:1007-1112) for particle i >= 1 (particle 0 keeps G = 0,
// x_bar = 0: the reference's loop starts at 1 and reset() zeroes both), in
// the order of the voxel lists.  16 lanes per particle find its neighbors once
// into LDS and walk them twice; a sum's additions, serial by their order, are
// one lane's.  What bounds it is issue, and at 2,000 particles the chain of
// loads.  Milliseconds at 2,000 / 30,011 / 128,000 particles: 0.067 / 0.145 /
// 1.19; with the columns searched twice and every lane of a group repeating its
// additions 0.140 / 0.312 / 1.77; lists of 4-byte entries leave six workgroups
// to a CU instead of eleven and take 0.066 / 0.211 / 1.89.
__global__ __launch_bounds__(16 * AN_GROUPS) void k_aniso(K k) {
  __shared__ __align__(16) AnisoLds lds;
  const int grp = threadIdx.x >> 4, q = threadIdx.x & 15;
  const int m = blockIdx.x * AN_GROUPS + grp;
  if (m >= k.n) return;  // whole groups leave together
  const float4 own = k.sorted[m];
  const int i = __float_as_int(own.w);
  float* G = k.G + 9 * (long)i;
  float* xb = k.xbar + 3 * (long)i;
  float4* rec = k.rec + (long)REC_QUADS * m;
  const float x0 = own.x, x1 = own.y, x2 = own.z;
  int v[3];
  {
    const float xi[3] = {x0, x1, x2};
    voxel_of(k, xi, v);
  }
  if (i == 0) {
    if (q == 0) {
      for (int a = 0; a < 9; a++) G[a] = 0.0f;
      for (int a = 0; a < 3; a++) xb[a] = 0.0f;
      rec[0] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
      rec[1] = make_float4(0.0f, 0.0f, 0.0f, -1.0f);  // q = 0 everywhere: no value anywhere
      rec[2] = make_float4(0.0f, 0.0f, 0.0f, __int_as_float(v[0]));
      rec[3] = make_float4(0.0f, 0.0f, 0.0f, __int_as_float(v[1]));
      rec[4] = make_float4(__int_as_float(v[2]), x0, x1, x2);
    }
    return;
  }
  const float r2 = 2.0f * k.sr;
  const float r2y = recip_mid(r2);
  const auto weight = [&](const float4& y) {
    const float dx = x0 - y.x, dy = x1 - y.y, dz = x2 - y.z;
    const float ss = dx * dx + dy * dy + dz * dz;
    float nr = sqrt_mid(ss);
    float t = div_mid(nr, r2, r2y);
    if (__builtin_expect(!(ss > 1e-30f) || !k.mid, 0)) {
      nr = sqrtf(ss);
      t = nr / r2;
    }
    return nr < r2 ? 1.0f - t * t * t : 0.0f;
  };
  float sum = 0.0f;
  int nn = 0;  // neighbors: w > 0
  bool whole = true;  // the list has held them all
  constexpr int NO_BASE = -0x10000;  // farther below every entry than the list reaches
  int base = NO_BASE;
  const auto first_pass = [&](int cnt) {
    add_neighbors<4>(k, lds, grp, q, base, cnt, sum, [&](const float4& y, bool on, float (&t)[4]) {
      const float w = weight(y);
      nn += on && w > 0.0f;
      t[0] = w;
      t[1] = w * y.x;
      t[2] = w * y.y;
      t[3] = w * y.z;
    });
  };
  const int left = find_neighbors(k, lds, grp, q, v, own, r2, base, [&](int cnt) {
    wave_order();
    first_pass(cnt);
    whole = false;
  });
  wave_order();
  first_pass(left);
  const float sw[4] = {lane_bcast<16, 0>(sum), lane_bcast<16, 1>(sum), lane_bcast<16, 2>(sum), lane_bcast<16, 3>(sum)};
  const float tw = sw[0];
  float w0 = sw[1], w1 = sw[2], w2 = sw[3];
  if (tw != 0.0f) {
    w0 /= tw;
    w1 /= tw;
    w2 /= tw;
  }
  const float b0 = k.lam1 * x0 + k.lam * w0, b1 = k.lam1 * x1 + k.lam * w1, b2 = k.lam1 * x2 + k.lam * w2;
  // C is symmetric bit for bit (w (a b) and w (b a)): six sums
  sum = 0.0f;
  const auto second_pass = [&](int cnt) {
    add_neighbors<6>(k, lds, grp, q, base, cnt, sum, [&](const float4& y, bool, float (&t)[6]) {
      const float w = weight(y);
      const float dp[3] = {y.x - w0, y.y - w1, y.z - w2};
      int n = 0;
#pragma unroll
      for (int a = 0; a < 3; a++)
#pragma unroll
        for (int c = a; c < 3; c++) t[n++] = w * (dp[a] * dp[c]);
    });
  };
  if (whole) {
    second_pass(left);
  } else {
    base = NO_BASE;
    const int rest = find_neighbors(k, lds, grp, q, v, own, r2, base, [&](int cnt) {
      wave_order();
      second_pass(cnt);
    });
    wave_order();
    second_pass(rest);
  }
  // the lanes' counts
#pragma unroll
  for (int d = 1; d < 16; d <<= 1) nn += __shfl_xor(nn, d, 16);
  const float cs[6] = {lane_bcast<16, 0>(sum), lane_bcast<16, 1>(sum), lane_bcast<16, 2>(sum),
                       lane_bcast<16, 3>(sum), lane_bcast<16, 4>(sum), lane_bcast<16, 5>(sum)};
  float C[9] = {cs[0], cs[1], cs[2], cs[1], cs[3], cs[4], cs[2], cs[4], cs[5]};
  if (tw != 0.0f)
#pragma unroll
    for (int a = 0; a < 9; a++) C[a] /= tw;
  float ev[3], V[9];
  eig3(C, ev, V);
#pragma unroll
  for (int a = 0; a < 2; a++)
#pragma unroll
    for (int b = 0; b < 2 - a; b++)
      if (ev[b] < ev[b + 1]) {
        const float t = ev[b];
        ev[b] = ev[b + 1];
        ev[b + 1] = t;
#pragma unroll
        for (int c = 0; c < 3; c++) {
          const float x = V[3 * c + b];
          V[3 * c + b] = V[3 * c + b + 1];
          V[3 * c + b + 1] = x;
        }
      }
  float g[9];
  float radius = 1.01f;
  if (tw == 0.0f) {
#pragma unroll
    for (int a = 0; a < 9; a++) g[a] = (a % 4) == 0 ? 1.0f : 0.0f;
  } else {
    float sg[3];
    if (nn > 25) {  // Nvep
      sg[0] = ev[0];
      sg[1] = fmaxf(ev[1], ev[0] / k.kr);
      sg[2] = fmaxf(ev[2], ev[0] / k.kr);
#pragma unroll
      for (int a = 0; a < 3; a++) sg[a] *= k.ks;
    } else {
      sg[0] = sg[1] = sg[2] = k.kn;
    }
    radius = 1.01f * k.sr * fmaxf(fabsf(sg[0]), fmaxf(fabsf(sg[1]), fabsf(sg[2])));
    const float ih = 1.0f / k.sr;
    float P[9];
#pragma unroll
    for (int a = 0; a < 3; a++)
#pragma unroll
      for (int c = 0; c < 3; c++) P[3 * a + c] = (ih * V[3 * a + c]) * (1.0f / sg[c]);
#pragma unroll
    for (int a = 0; a < 3; a++)
#pragma unroll
      for (int b = 0; b < 3; b++) g[3 * a + b] = P[3 * a] * V[3 * b] + P[3 * a + 1] * V[3 * b + 1] + P[3 * a + 2] * V[3 * b + 2];
    // a support radius is only trusted where V came out orthonormal
    float e = 0.0f;
#pragma unroll
    for (int a = 0; a < 3; a++)
#pragma unroll
      for (int b = 0; b < 3; b++)
        e = fmaxf(e, fabsf(V[a] * V[b] + V[3 + a] * V[3 + b] + V[6 + a] * V[6 + b] - (a == b ? 1.0f : 0.0f)));
    if (!(e < 1e-3f)) radius = INFINITY;
  }
  if (q != 0) return;
#pragma unroll
  for (int a = 0; a < 9; a++) G[a] = g[a];
  xb[0] = b0;
  xb[1] = b1;
  xb[2] = b2;
  const float det = g[0] * (g[4] * g[8] - g[7] * g[5]) - g[3] * (g[1] * g[8] - g[7] * g[2]) + g[6] * (g[1] * g[5] - g[4] * g[2]);
  rec[0] = make_float4(b0, b1, b2, det);
  rec[1] = make_float4(g[0], g[1], g[2], radius);
  rec[2] = make_float4(g[3], g[4], g[5], __int_as_float(v[0]));
  rec[3] = make_float4(g[6], g[7], g[8], __int_as_float(v[1]));
  rec[4] = make_float4(__int_as_float(v[2]), x0, x1, x2);
}

// The blocks the two field passes write: every vertex >= 0 of the particle's
// 27-vertex poly6 box and of its anisotropic box [c - off, c - off + R]^3
// (the reference writes them all, zeros included).  Each box spans at most two
// blocks per axis (R + 1 <= 32 is checked on the host), so its 8 corners name
// every block it touches.
__global__ void k_mark(K k) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= k.n) return;
  const int* v = k.pvox + 3 * (long)i;
  int lo[3], hi[3];
  for (int a = 0; a < 3; a++) {
    lo[a] = v[a] - 1;
    hi[a] = v[a] + 1;
    if (k.aniso) {
      lo[a] = min(lo[a], v[a] - k.off);
      hi[a] = max(hi[a], v[a] - k.off + k.R);
    }
    lo[a] = max(lo[a], 0);
  }
  for (int c = 0; c < 8; c++) {
    const int x = (c >> 2) ? hi[0] : lo[0], y = ((c >> 1) & 1) ? hi[1] : lo[1], z = (c & 1) ? hi[2] : lo[2];
    k.active[bidx(k, x - k.glo[0], y - k.glo[1], z - k.glo[2])] = 1;
  }
}

// The field at the vertices of one 8^3 tile, one workgroup of 8 wavefronts per
// tile.  All contributions are 2^-32 fixed-point integers, so their sum is the
// one any order of the reference's atomics would give exactly.
//
// FIELD_ANISO: the anisotropic values of the particles whose boxes reach the
// tile (voxels c in [T - R + off, T + 7 + off] per axis, T the tile's first
// vertex).  The workgroup lists the candidate voxel columns and their particle
// counts, stages the candidates' records in LDS 512 at a time, dropping those
// whose support radius ends before the tile, and each wavefront takes every
// eighth of them: a lane holds the 8 vertices of one (x, y) column, so the
// x and y parts of G d are formed once for 8 values, a vertex plane outside
// the particle's box is skipped by the whole wavefront, and the multiplicity
// of the reference's voxel-corner loop is a factor (1, 2, 4 or 8).  The
// wavefronts' sums meet in LDS.  What bounds it is VALU issue: about 36
// instructions a value, in 26 of every 33 planes and 26^2 of every 33^2
// columns; 128,000 particles take 3.3 ms (4.1 with int64 sums, 45 instructions
// a value; 10.7 with one vertex per lane and every candidate evaluated at all
// 512).
// The fixed-point form of v: the double v + 1.5 2^20 has an ulp of 2^-32, so
// (v + 1.5 2^20) - 1.5 2^20 is v rounded to a multiple of 2^-32, and sums of such
// below 2^21 are exact in FP64.  Each staged particle adds a bound of its values
// to a total; only if that reaches 2^18 (a value counts up to 8 times) or is not
// a number is the tile summed again in the general form (fix_of in int64, with
// its error flag).
//
// FIELD_VELOCITY: the poly6-weighted velocity of the particles within h
// (generate_smooth_fluid_field_with_velocity_impl, :1160-1190), same layout:
// 30,011 particles take 0.235 ms, 0.35 with int64 sums and the full-range root
// and division.
//
// Every tile then has the isotropic poly6 values added (in FIELD_ANISO or, for
// the isotropic field, FIELD_ISO), one thread per vertex over the 27 voxels
// around it.  Tiles of unwritten blocks store 0.
enum { FIELD_ISO = 0, FIELD_ANISO = 1, FIELD_VELOCITY = 2 };
constexpr int TILE = 8;
constexpr int FIELD_THREADS = TILE * TILE * TILE;
constexpr int FIELD_WAVES = FIELD_THREADS / 64;
constexpr int MAX_COLS = 1536;  // (TILE + R)^2 columns, R + 1 <= 32
constexpr float FIX_ROOM = 262144.0f;  // 2^18

// acc + mult v (half of that where not `whole`, which is uniform), v rounded to a
// multiple of 2^-32, where that is exact; acc holds a double
__device__ __forceinline__ unsigned long long fix_fast(unsigned long long acc, float v, double mult, bool whole) {
  double r = ((double)v + 1572864.0) - 1572864.0;  // 1.5 2^20
  if (__builtin_expect(!whole, 0)) r *= 0.5;
  return (unsigned long long)__double_as_longlong(__builtin_fma(r, mult, __longlong_as_double((long long)acc)));
}
__device__ __forceinline__ unsigned long long fix_done(unsigned long long acc) {
  return (unsigned long long)(long long)(__longlong_as_double((long long)acc) * FIX_SCALE);
}

// multiplicity of axis position v for a particle of voxel c, as a shift: 0, 1, or -1 for none
__device__ __forceinline__ int mult_shift(int v, int c, int off, int R) { return mult_axis(v, c, off, R) - 1; }

// cubic_spline_kernel (:1115-1124) at q = |G d|, "+ 1" where the reference puts it
__device__ __forceinline__ float aniso_of(float c48d, float c16d, float q) {
  const float in = c48d * (q * q * q - q * q) + 1.0f;
  const float out = c16d * (1.0f - q) * (1.0f - q) * (1.0f - q);
  const float r = q <= 0.5f ? in : out;
  return 0.0f < q && q <= 1.0f ? r : 0.0f;
}
// the same for q > 0: past 1 (or not a number) 1 - q is clamped to 0, and the value is +-0
// (the inner form under a wavefront's branch instead: 3.30 -> 3.47 ms)
__device__ __forceinline__ float aniso_mid(float c48d, float c16d, float q) {
  const float in = c48d * (q * q * q - q * q) + 1.0f;
  const float u = __builtin_amdgcn_fmed3f(1.0f - q, 0.0f, 1.0f);
  const float out = c16d * u * u * u;
  return q <= 0.5f ? in : out;
}

// one staged particle's values at the 8 vertices of each lane's column
template <bool GENERAL>
__device__ __forceinline__ void aniso_column(const K& k, const float4 (&r)[REC_QUADS], const int* T, int vx, int vy, float px,
                                             float py, unsigned long long (&acc)[TILE], float& total, bool& bad) {
  const int c0 = uniform(__float_as_int(r[2].w)), c1 = uniform(__float_as_int(r[3].w)), c2 = uniform(__float_as_int(r[4].x));
  const int sx = mult_shift(vx, c0, k.off, k.R), sy = mult_shift(vy, c1, k.off, k.R);
  const float c48d = k.c48 * r[0].w, c16d = k.c16 * r[0].w;
  // |q^3 - q^2| <= 1/8 up to q = 1/2, (1 - q)^3 <= 1/8 from there on
  if (!GENERAL) total += fmaxf(fabsf(c48d), fabsf(c16d)) * 0.1251f + 1.001f;
  if (sx < 0 || sy < 0) return;
  const int sxy = sx + sy;
  const double mult = (double)(2 << sxy);  // inside the box along z; half of it in its first and last plane
  const float dx = r[0].x - px, dy = r[0].y - py;
  const float ta = r[1].x * dx + r[1].y * dy, tb = r[2].x * dx + r[2].y * dy, tc = r[3].x * dx + r[3].y * dy;
#pragma unroll
  for (int z = 0; z < TILE; z++) {
    const unsigned rel = (unsigned)(T[2] + z - c2 + k.off);  // mult_shift, uniform: 0 .. R, 1 .. R - 1
    if (rel > (unsigned)k.R) continue;
    const bool inner = rel - 1u < (unsigned)k.R - 1u;
    const float dz = r[0].z - ((float)(T[2] + z) * k.vs + k.o[2]);
    const float a = ta + r[1].z * dz, b = tb + r[2].z * dz, c = tc + r[3].z * dz;
    const float ss = a * a + b * b + c * c;
    if (GENERAL) {
      const float w = k.vol * aniso_of(c48d, c16d, sqrtf(ss));
      if (!(fabsf(w) <= MAX_CONTRIB)) bad = true;
      else acc[z] += fix_of(w) << (sxy + inner);
    } else {
      if (__all(ss > 1.0f)) continue;  // q = 1 gives 0 too
      float f = aniso_mid(c48d, c16d, sqrt_mid(ss));
      if (__builtin_expect(ss < 1e-30f, 0)) f = aniso_of(c48d, c16d, sqrtf(ss));
      acc[z] = fix_fast(acc[z], k.vol * f, mult, inner);
    }
  }
}

// poly6's constants, with the shorter exact root and division where they hold: a
// numerator below 2^-103 may round differently, but gives less than 2^-40 there
// (den >= 2^-63), which times a velocity and voxel_size^3 of less than 2^6
// rounds to 0 in either form
struct Poly6 {
  float h, h2, den, y;
  bool mid;
  __device__ __forceinline__ explicit Poly6(const K& k) : h(k.sr), h2(k.sr * k.sr) {
    den = h2 * h2 * h2 * h2 * h;
    y = recip_mid(den);
    mid = k.mid && den > 0x1p-63f && den < 0x1p30f;
  }
};

// one staged particle's poly6-weighted velocity at the 8 vertices of each lane's column
// (GENERAL: into the tile's sums at once)
template <bool GENERAL>
__device__ __forceinline__ void velocity_column(const K& k, const Poly6& w6, const float4& p4, const float4& v4, int c0, int c1,
                                                const int* T, int vx, int vy, float px, float py,
                                                unsigned long long (&acc)[3][TILE], unsigned long long (*sum)[FIELD_THREADS],
                                                float& total, bool& bad) {
  const int sx = mult_shift(vx, c0, k.off, k.R), sy = mult_shift(vy, c1, k.off, k.R);
  if (!GENERAL) total += fmaxf(fabsf(v4.x), fmaxf(fabsf(v4.y), fabsf(v4.z)));
  if (sx < 0 || sy < 0) return;
  const double mult = (double)(2 << (sx + sy));
  const int c2 = uniform(__float_as_int(p4.x));
  const float rx = p4.y - px, ry = p4.z - py;
  if (__all(rx * rx + ry * ry > 1.0001f * k.sr * k.sr)) return;
  const auto plane = [&](int z) {
    const unsigned rel = (unsigned)(T[2] + z - c2 + k.off);  // as in aniso_column
    if (rel > (unsigned)k.R) return;
    const bool inner = rel - 1u < (unsigned)k.R - 1u;
    const float rz = p4.w - ((float)(T[2] + z) * k.vs + k.o[2]);
    if (fabsf(rz) > 1.0001f * k.sr) return;  // uniform; poly6 is 0 there
    if (GENERAL) {
      const float f = poly6(k, rx, ry, rz, k.sr) * k.cvs3;
      const float u[3] = {v4.x * f, v4.y * f, v4.z * f};
      for (int c = 0; c < 3; c++) {
        if (!(fabsf(u[c]) <= MAX_CONTRIB)) bad = true;
        else atomicAdd(&sum[c][((threadIdx.x & 63) << 3) + z], fix_of(u[c]) << (sx + sy + inner));
      }
      return;
    }
    const float ss = rx * rx + ry * ry + rz * rz;
    const float rn = sqrt_mid(ss);
    float res = w6.h2 - rn * rn;
    res = res * res * res;
    float f = rn <= w6.h ? div_mid(k.acoef * res, w6.den, w6.y) : 0.0f;
    if (__builtin_expect(ss < 1e-30f, 0)) f = poly6(k, rx, ry, rz, k.sr);
    f *= k.cvs3;
    acc[0][z] = fix_fast(acc[0][z], v4.x * f, mult, inner);
    acc[1][z] = fix_fast(acc[1][z], v4.y * f, mult, inner);
    acc[2][z] = fix_fast(acc[2][z], v4.z * f, mult, inner);
  };
  if constexpr (GENERAL) {
#pragma unroll 1
    for (int z = 0; z < TILE; z++) plane(z);
  } else {
#pragma unroll
    for (int z = 0; z < TILE; z++) plane(z);
  }
}

template <int MODE>
__global__ __launch_bounds__(FIELD_THREADS) __attribute__((amdgpu_waves_per_eu(4))) void k_field(K k) {
  constexpr int QUADS = MODE == FIELD_VELOCITY ? 3 : REC_QUADS;
  __shared__ int col_off[MODE == FIELD_ISO ? 1 : MAX_COLS + 1];
  __shared__ int col_begin[MODE == FIELD_ISO ? 1 : MAX_COLS];
  __shared__ float4 stage[MODE == FIELD_ISO ? 1 : QUADS * FIELD_THREADS];
  __shared__ unsigned long long sum[MODE == FIELD_VELOCITY ? 3 : 1][FIELD_THREADS];
  __shared__ int wave_tot[FIELD_WAVES];
  __shared__ int kept;
  const int tb = blockIdx.x;
  const int tdy = k.gdim[1] / TILE, tdz = k.gdim[2] / TILE;
  const int tx = tb / (tdy * tdz), ty = (tb / tdz) % tdy, tz = tb % tdz;
  const int t = threadIdx.x;
  const long q = gidx(k, tx * TILE + (t >> 6), ty * TILE + ((t >> 3) & 7), tz * TILE + (t & 7));
  if (!k.active[bidx(k, tx * TILE, ty * TILE, tz * TILE)]) {  // a tile lies in one block
    if (MODE == FIELD_VELOCITY) {
      for (int c = 0; c < 3; c++) k.vfield[3 * q + c] = 0.0f;
    } else {
      k.field0[q] = 0.0f;
      k.field[q] = 0.0f;
    }
    return;
  }
  const int T[3] = {tx * TILE + k.glo[0], ty * TILE + k.glo[1], tz * TILE + k.glo[2]};
  const int R = k.R, off = k.off;
  bool bad = false;
  if (MODE == FIELD_VELOCITY)
    for (int c = 0; c < 3; c++) sum[c][t] = 0ull;
  if (MODE != FIELD_VELOCITY) {  // the isotropic part, one vertex per thread
    const int vx = T[0] + (t >> 6), vy = T[1] + ((t >> 3) & 7), vz = T[2] + (t & 7);
    float p[3];
    vpos(k, vx, vy, vz, p);
    const int z0 = max(vz - 1, k.vlo[2]), z1 = min(vz + 1, k.vlo[2] + k.vdim[2] - 1);
    unsigned long long acc = 0ull;
    if (z0 <= z1)
      for (int x = max(vx - 1, k.vlo[0]); x <= min(vx + 1, k.vlo[0] + k.vdim[0] - 1); x++)
        for (int y = max(vy - 1, k.vlo[1]); y <= min(vy + 1, k.vlo[1] + k.vdim[1] - 1); y++) {
          const long base = ((long)(x - k.vlo[0]) * k.vdim[1] + (y - k.vlo[1])) * k.vdim[2] - k.vlo[2];
          for (int m = k.vstart[base + z0]; m < k.vstart[base + z1 + 1]; m++) {
            const float4 xj = k.sorted[m];
            const float w = k.vol * poly6(k, xj.x - p[0], xj.y - p[1], xj.z - p[2], k.sr);
            if (!(fabsf(w) <= MAX_CONTRIB)) bad = true;
            else acc += fix_of(w);
          }
        }
    sum[0][t] = acc;
  }
  if constexpr (MODE != FIELD_ISO) {
    // candidate columns: the voxels whose boxes (or, for the velocities, whose
    // spheres of h) can reach the tile
    const int near = (int)(k.sr / k.vs) + 2;
    int clo[3], chi[3];
    for (int a = 0; a < 3; a++) {
      clo[a] = T[a] - R + off;
      chi[a] = T[a] + TILE - 1 + off;
      if (MODE == FIELD_VELOCITY) {
        clo[a] = max(clo[a], T[a] - near);
        chi[a] = min(chi[a], T[a] + TILE - 1 + near);
      }
      clo[a] = max(clo[a], k.vlo[a]);
      chi[a] = min(chi[a], k.vlo[a] + k.vdim[a] - 1);
    }
    const int ncx = max(0, chi[0] - clo[0] + 1), ncy = max(0, chi[1] - clo[1] + 1);
    const int ncol = clo[2] <= chi[2] ? ncx * ncy : 0;  // <= MAX_COLS (checked on the host)
    // their particle counts, scanned: wavefront scans, then the wavefronts' totals
    int carry = 0;
    if (t == 0) col_off[0] = 0;
    for (int c0 = 0; c0 < ncol; c0 += FIELD_THREADS) {
      const int c = c0 + t;
      int cnt = 0;
      if (c < ncol) {
        const int cx = clo[0] + c / ncy, cy = clo[1] + c % ncy;
        const long base = ((long)(cx - k.vlo[0]) * k.vdim[1] + (cy - k.vlo[1])) * k.vdim[2] - k.vlo[2];
        const int b = k.vstart[base + clo[2]];
        col_begin[c] = b;
        cnt = k.vstart[base + chi[2] + 1] - b;
      }
      int incl = cnt;
#pragma unroll
      for (int d = 1; d < 64; d <<= 1) {
        const int u = __shfl_up(incl, d, 64);
        if ((t & 63) >= d) incl += u;
      }
      __syncthreads();  // the previous round's totals are read
      if ((t & 63) == 63) wave_tot[t >> 6] = incl;
      __syncthreads();
      int before = carry, all = 0;
      for (int w = 0; w < FIELD_WAVES; w++) {
        if (w < (t >> 6)) before += wave_tot[w];
        all += wave_tot[w];
      }
      if (c < ncol) col_off[c + 1] = before + incl;
      carry += all;
    }
    __syncthreads();
    const int total = carry;
    const int lane = t & 63, wave = uniform(t >> 6);
    const int vx = T[0] + (lane >> 3), vy = T[1] + (lane & 7);
    const float px = (float)vx * k.vs + k.o[0], py = (float)vy * k.vs + k.o[1];
    // the tile's box of vertices
    float tlo[3], thi[3];
    for (int a = 0; a < 3; a++) {
      tlo[a] = (float)T[a] * k.vs + k.o[a];
      thi[a] = (float)(T[a] + TILE - 1) * k.vs + k.o[a];
    }
    unsigned long long acc[MODE == FIELD_VELOCITY ? 3 : 1][TILE];
    const Poly6 w6(k);
    // a second round, in the general form, only where the first was out of range
    for (int round = 0; round < 2; round++) {
      for (int c = 0; c < (MODE == FIELD_VELOCITY ? 3 : 1); c++)
#pragma unroll
        for (int z = 0; z < TILE; z++) acc[c][z] = 0ull;
      float bound = 0.0f;
      for (int s0 = 0; s0 < total; s0 += FIELD_THREADS) {
        if (t == 0) kept = 0;
        __syncthreads();
        const int idx = s0 + t;
        if (idx < total) {
          int lo = 0, hi = ncol - 1;  // the column c with col_off[c] <= idx < col_off[c + 1]
          while (lo < hi) {
            const int mid = (lo + hi + 1) >> 1;
            if (col_off[mid] <= idx) lo = mid;
            else hi = mid - 1;
          }
          const int m = col_begin[lo] + (idx - col_off[lo]);
          const float4* rec = k.rec + (long)REC_QUADS * m;
          if (MODE == FIELD_ANISO) {
            const float4 r0 = rec[0], r1 = rec[1];
            const float gx = fmaxf(0.0f, fmaxf(tlo[0] - r0.x, r0.x - thi[0]));
            const float gy = fmaxf(0.0f, fmaxf(tlo[1] - r0.y, r0.y - thi[1]));
            const float gz = fmaxf(0.0f, fmaxf(tlo[2] - r0.z, r0.z - thi[2]));
            const bool out = r1.w < 0.0f || gx * gx + gy * gy + gz * gz > 1.001f * r1.w * r1.w;
            if (!out) {
              const int at = atomicAdd(&kept, 1);
              stage[at] = r0;
              stage[FIELD_THREADS + at] = r1;
              stage[2 * FIELD_THREADS + at] = rec[2];
              stage[3 * FIELD_THREADS + at] = rec[3];
              stage[4 * FIELD_THREADS + at] = rec[4];
            }
          } else {
            const int at = atomicAdd(&kept, 1);
            const float* u = k.vel + 3 * (long)k.vlist[m];
            stage[at] = rec[4];
            stage[FIELD_THREADS + at] = make_float4(u[0], u[1], u[2], 0.0f);
            stage[2 * FIELD_THREADS + at] = make_float4(rec[2].w, rec[3].w, 0.0f, 0.0f);
          }
        }
        __syncthreads();
        const int nst = kept;
        for (int r = wave; r < nst; r += FIELD_WAVES) {
          if constexpr (MODE == FIELD_ANISO) {
            float4 rr[REC_QUADS];
#pragma unroll
            for (int e = 0; e < REC_QUADS; e++) rr[e] = stage[e * FIELD_THREADS + r];
            if (round == 0) aniso_column<false>(k, rr, T, vx, vy, px, py, acc[0], bound, bad);
            else aniso_column<true>(k, rr, T, vx, vy, px, py, acc[0], bound, bad);
          } else {
            const float4 c4 = stage[2 * FIELD_THREADS + r];
            const int v0 = uniform(__float_as_int(c4.x)), v1 = uniform(__float_as_int(c4.y));
            if (round == 0)
              velocity_column<false>(k, w6, stage[r], stage[FIELD_THREADS + r], v0, v1, T, vx, vy, px, py, acc, sum, bound, bad);
            else
              velocity_column<true>(k, w6, stage[r], stage[FIELD_THREADS + r], v0, v1, T, vx, vy, px, py, acc, sum, bound, bad);
          }
        }
        __syncthreads();
      }
      if (round == 1) break;
      // poly6 <= acoef h^6 / h^9
      const bool fits = MODE == FIELD_ANISO ? fabsf(k.vol) * bound < FIX_ROOM
                                            : w6.mid && fabsf(k.acoef * k.cvs3 / (w6.h2 * w6.h)) * 1.001f * bound < FIX_ROOM &&
                                                  bound * k.cvs3 < 64.0f;
      if (!__syncthreads_or(!fits)) {
        for (int c = 0; c < (MODE == FIELD_VELOCITY ? 3 : 1); c++)
#pragma unroll
          for (int z = 0; z < TILE; z++) acc[c][z] = fix_done(acc[c][z]);
        break;
      }
    }
    for (int c = 0; c < (MODE == FIELD_VELOCITY ? 3 : 1); c++)
#pragma unroll
      for (int z = 0; z < TILE; z++) atomicAdd(&sum[c][(lane << 3) + z], acc[c][z]);
    __syncthreads();
  }
  if (MODE == FIELD_VELOCITY) {
    for (int c = 0; c < 3; c++) k.vfield[3 * q + c] = (float)((double)(long long)sum[c][t] * FIX_INV);
  } else {
    const float v = (float)((double)(long long)sum[0][t] * FIX_INV);
    k.field0[q] = v;
    k.field[q] = v;
  }
  if (bad) atomicOr(k.err, ERR_RANGE);
}

// a velocity that is not finite gives no finite contribution anywhere in its particle's box
__global__ void k_check_velocities(K k) {
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < 3L * k.n && !isfinite(k.vel[i])) atomicOr(k.err, ERR_RANGE);
}

// Blocked FP64 statistic of the negative values, one workgroup per block in
// block order (inactive blocks add 0): lane t adds vertices l = t + 256 j of
// the block (l = (lx * 32 + ly) * 32 + lz) in order, then a pairwise tree.
// which 0: sum of v, count; which 1: sum of (v - mean)^2 (v - mean in FP32).
constexpr int ST_THREADS = 256;
__global__ __launch_bounds__(ST_THREADS) void k_stats(K k, int which, double* part, long long* pcount) {
  __shared__ double lane[ST_THREADS];
  __shared__ int cnt;
  const long b = blockIdx.x;
  const int t = threadIdx.x;
  if (t == 0) cnt = 0;
  __syncthreads();
  if (!k.active[b]) {
    if (t == 0) {
      part[b] = 0.0;
      pcount[b] = 0;
    }
    return;
  }
  const int bz = (int)(b % k.bdim[2]), by = (int)((b / k.bdim[2]) % k.bdim[1]), bx = (int)(b / ((long)k.bdim[1] * k.bdim[2]));
  const float mean = (float)k.stats[2];
  double a = 0.0;
  int c = 0;
  // few blocks, so few wavefronts: 32 loads in flight each, 11 to 14 us (a
  // block's 128 a lane one after the other took 34 to 37)
  constexpr int DEEP = 32;
  const float* f = k.field + gidx(k, bx * BLOCK, by * BLOCK + (t >> 5), bz * BLOCK + (t & 31));
  for (int j0 = 0; j0 < BLOCK * BLOCK * BLOCK / ST_THREADS; j0 += DEEP) {
    float v[DEEP];
#pragma unroll
    for (int j = 0; j < DEEP; j++) {  // vertex l = t + 256 (j0 + j)
      const int row = (j0 + j) * (ST_THREADS / BLOCK);
      v[j] = f[((long)(row >> 5) * k.gdim[1] + (row & 31)) * k.gdim[2]];
    }
#pragma unroll
    for (int j = 0; j < DEEP; j++) {
      if (v[j] < 0.0f) {
        if (which == 0) {
          a += (double)v[j];
          c++;
        } else {
          const double d = (double)(v[j] - mean);
          a += d * d;
        }
      }
    }
  }
  lane[t] = a;
  if (c) atomicAdd(&cnt, c);
  __syncthreads();
  for (int span = ST_THREADS / 2; span > 0; span >>= 1) {
    if (t < span) lane[t] += lane[t + span];
    __syncthreads();
  }
  if (t == 0) {
    part[b] = lane[0];
    pcount[b] = cnt;
  }
}

// blocks added in block order; which 0 sets the mean, which 1 the sd
__global__ __launch_bounds__(ST_THREADS) void k_stats_final(K k, int which, const double* part, const long long* pcount) {
  __shared__ double ps[ST_THREADS];
  __shared__ long long pc[ST_THREADS];
  const int t = threadIdx.x;
  double s = 0.0;
  long long c = 0;
  for (long b0 = 0; b0 < k.nblock; b0 += ST_THREADS) {
    const int n = (int)min((long)ST_THREADS, k.nblock - b0);
    if (t < n) {
      ps[t] = part[b0 + t];
      pc[t] = pcount[b0 + t];
    }
    __syncthreads();
    if (t == 0)
      for (int b = 0; b < n; b++) {
        s += ps[b];
        c += pc[b];
      }
    __syncthreads();
  }
  if (t != 0) return;
  if (which == 0) {
    k.stats[0] = s;
    k.stats[1] = (double)c;
    k.stats[2] = c > 0 ? (double)(float)(s / (double)c) : 0.0;
    if (c == 0) k.stats[3] = (double)NAN;
  } else if (k.stats[1] > 0.0) {
    k.stats[3] = (double)(float)sqrt(s / k.stats[1]);
  }
}

// smooth_sdf_impl (:1459-1484), radius 1.  Bound by issue: 27 exponentials and as
// many pairs of quotients a vertex; 2.5 million vertices take 87 us, 95 with
// full-range divisions.
__global__ void k_smooth(K k, const float* in, float* out) {
  const long q = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (q >= k.nvert) return;
  const int gz = (int)(q % k.gdim[2]), gy = (int)((q / k.gdim[2]) % k.gdim[1]), gx = (int)(q / ((long)k.gdim[1] * k.gdim[2]));
  if (!k.active[bidx(k, gx, gy, gz)]) {
    out[q] = 0.0f;
    return;
  }
  const float sd = (float)k.stats[3];
  const int i = gx + k.glo[0], j = gy + k.glo[1], l = gz + k.glo[2];
  const float vc = in[q];
  const float den = 2.0f * sd * sd, tt = k.c2pi * sd * sd, scale = tt * sqrtf(tt);
  // the shorter exact quotients where the denominators let them be used.  A
  // numerator so small that they may round differently gives an exponent whose
  // e^x is 1 in either form; one too large, or a weight too small, takes the
  // full-range division.
  const bool mid = den > 0x1p-40f && den < 0x1p40f && scale > 0x1p-40f && scale < 0x1p40f;
  const float yd = recip_mid(den), ys = recip_mid(scale);
  float avg = 0.0f, weight = 0.0f;
#pragma unroll
  for (int dx = -1; dx <= 1; dx++) {  // nine loads in flight
    float vn[9];
    bool on[9];
#pragma unroll
    for (int e = 0; e < 9; e++) {
      const int dy = e / 3 - 1, dz = e % 3 - 1;
      on[e] = min(i + dx, min(j + dy, l + dz)) >= 0;
      vn[e] = val_at(k, in, i + dx, j + dy, l + dz);
    }
#pragma unroll
    for (int e = 0; e < 9; e++) {
      const float d = fabsf(vc - vn[e]);
      const float dd = -d * d;
      float ex = sr_expf(div_mid(dd, den, yd));
      float gw = div_mid(ex, scale, ys);
      if (__builtin_expect(!mid || !(dd > -0x1p60f) || (ex < 0x1p-60f && ex > 0.0f), 0)) {
        ex = sr_expf(dd / den);
        gw = ex / scale;
      }
      gw = on[e] ? gw : 0.0f;
      avg += gw * vn[e];
      weight += gw;
    }
  }
  if (weight != 0.0f) avg /= weight;
  out[q] = avg;
}

// corner offsets (voxel_vertex_offset_map, :772-779) and edge corner pairs
// (interpolation_table, :925-936)
__constant__ int CORNER[8][3] = {{0, 1, 0}, {1, 1, 0}, {1, 0, 0}, {0, 0, 0}, {0, 1, 1}, {1, 1, 1}, {1, 0, 1}, {0, 0, 1}};
__constant__ int EDGE[12][2] = {{0, 1}, {1, 2}, {2, 3}, {3, 0}, {4, 5}, {5, 6}, {6, 7}, {7, 4}, {0, 4}, {1, 5}, {2, 6}, {3, 7}};
// cubes sharing edges 2, 3, 11 of a cube (get_edge_adjacent_cubes, :1613-1705)
__constant__ int ADJ_W[3] = {2, 3, 11};
__constant__ int ADJ[3][3][3] = {
    {{0, 0, -1}, {0, -1, -1}, {0, -1, 0}},
    {{0, 0, -1}, {-1, 0, -1}, {-1, 0, 0}},
    {{0, -1, 0}, {-1, -1, 0}, {-1, 0, 0}},
};

// Code of every cube (its vertex of the grid): 0 without a crossing, else the
// bits (corner value < isolevel) << 12 | crossed-edge mask (the marching-cubes
// edge table, derived: an edge is crossed when its corners differ).
__global__ void k_cube_flag(K k) {
  const long q = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (q >= k.nvert) return;
  const int gz = (int)(q % k.gdim[2]), gy = (int)((q / k.gdim[2]) % k.gdim[1]), gx = (int)(q / ((long)k.gdim[1] * k.gdim[2]));
  int code = 0;
  if (k.active[bidx(k, gx, gy, gz)]) {
    int ci = 0;
#pragma unroll
    for (int j = 0; j < 8; j++)
      if (val_at(k, k.field, gx + k.glo[0] + CORNER[j][0], gy + k.glo[1] + CORNER[j][1], gz + k.glo[2] + CORNER[j][2]) < k.iso)
        ci |= 1 << j;
    int mask = 0;
#pragma unroll
    for (int w = 0; w < 12; w++)
      if (((ci >> EDGE[w][0]) & 1) != ((ci >> EDGE[w][1]) & 1)) mask |= 1 << w;
    if (mask) code = (ci << 12) | mask;
  }
  k.flag[q] = code;
}

// cube_id held the number of crossing cubes before each cube: a crossing cube's
// vertex number + 1 (0 for the others), and the cubes by vertex number
__global__ void k_cube_id(K k) {
  const long q = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (q >= k.nvert) return;
  const bool on = k.flag[q] != 0;
  const int m = k.cube_id[q];
  if (on) k.cubes[m] = (int)q;
  k.cube_id[q] = on ? m + 1 : 0;
}

// calc_vertex_normal (:1307-1321) with normalize (:1413-1417)
__device__ __forceinline__ void unit_or_zero(float* n) {
  const float nr = norm3f(n[0], n[1], n[2]);
  if (nr != 0.0f) {
    n[0] /= nr;
    n[1] /= nr;
    n[2] /= nr;
  } else {
    n[0] = n[1] = n[2] = 0.0f;
  }
}
__device__ __forceinline__ void vertex_normal(const K& k, int x, int y, int z, float* n) {
  const float* f = k.field;
  n[0] = x == 0 ? -val_at(k, f, x + 1, y, z) : val_at(k, f, x - 1, y, z) - val_at(k, f, x + 1, y, z);
  n[1] = y == 0 ? -val_at(k, f, x, y + 1, z) : val_at(k, f, x, y - 1, z) - val_at(k, f, x, y + 1, z);
  n[2] = z == 0 ? -val_at(k, f, x, y, z + 1) : val_at(k, f, x, y, z - 1) - val_at(k, f, x, y, z + 1);
  unit_or_zero(n);
}
// process_normal_at (:1336-1349)
__device__ __forceinline__ void normal_at(const K& k, const float* p, float* out) {
  int v[3];
  voxel_of(k, p, v);
  float base[3];
  vpos(k, v[0], v[1], v[2], base);
  const float xd = (p[0] - base[0]) / k.vs, yd = (p[1] - base[1]) / k.vs, zd = (p[2] - base[2]) / k.vs;
  float c[8][3];
  const int gx = v[0] - k.glo[0], gy = v[1] - k.glo[1], gz = v[2] - k.glo[2];
  // the 4^3 vertices around the voxel lie in the grid
  if (min(gx, min(gy, gz)) >= 1 && gx + 2 < k.gdim[0] && gy + 2 < k.gdim[1] && gz + 2 < k.gdim[2]) {
    const long sy = k.gdim[2], sx = (long)k.gdim[1] * k.gdim[2];
    const float* f = k.field + gidx(k, gx, gy, gz);
#pragma unroll
    for (int j = 0; j < 8; j++) {
      const float* at = f + (j >> 2) * sx + ((j >> 1) & 1) * sy + (j & 1);
      c[j][0] = at[-sx] - at[sx];
      c[j][1] = at[-sy] - at[sy];
      c[j][2] = at[-1] - at[1];
    }
#pragma unroll
    for (int j = 0; j < 8; j++) unit_or_zero(c[j]);
  } else {
#pragma unroll
    for (int j = 0; j < 8; j++) vertex_normal(k, v[0] + (j >> 2), v[1] + ((j >> 1) & 1), v[2] + (j & 1), c[j]);
  }
  float r[3];
#pragma unroll
  for (int a = 0; a < 3; a++) {
    const float c00 = c[0][a] * (1.0f - xd) + c[4][a] * xd;
    const float c01 = c[1][a] * (1.0f - xd) + c[5][a] * xd;
    const float c10 = c[2][a] * (1.0f - xd) + c[6][a] * xd;
    const float c11 = c[3][a] * (1.0f - xd) + c[7][a] * xd;
    const float c0 = c00 * (1.0f - yd) + c10 * yd;
    const float c1 = c01 * (1.0f - yd) + c11 * yd;
    r[a] = c0 * (1.0f - zd) + c1 * zd;
  }
  const float nr = norm3f(r[0], r[1], r[2]);
  if (nr != 0.0f) {
    out[0] = r[0] / nr;
    out[1] = r[1] / nr;
    out[2] = r[2] / nr;
  } else {
    out[0] = out[1] = out[2] = 0.0f;
  }
}
// vertex_interpolate (:1254-1262)
__device__ __forceinline__ void vinterp(float iso, const float* p1, const float* p2, float v1, float v2, float* out) {
  const float delta = v2 - v1;
  const float off = fabsf(delta) < 0.00001f ? 0.5f : (iso - v1) / delta;
#pragma unroll
  for (int a = 0; a < 3; a++) out[a] = p1[a] + off * (p2[a] - p1[a]);
}

// the QEF: rows folded into a 4x4 triangle by Givens rotations (incremental QR,
// Ju et al. 2002; the reference's Householder form holds 4 rows), the 3x3 block
// solved through its SVD with singular values clamped to sign(s) max(0.1, |s|)
// (solve_qef, :70-80), x = V diag(1 / s') U^T b; singular values up to 1e-6 of
// the largest count as 0 (the null space, where U is arbitrary, is dropped)
__device__ __forceinline__ void qef_add(float* R, float a0, float a1, float a2, float a3) {
  float a[4] = {a0, a1, a2, a3};
#pragma unroll
  for (int kk = 0; kk < 4; kk++) {
    const float xk = a[kk];
    if (xk == 0.0f) continue;
    const float rk = R[5 * kk];
    const float rho = sqrtf(rk * rk + xk * xk);
    const float c = rk / rho, sn = xk / rho;
#pragma unroll
    for (int j = kk; j < 4; j++) {
      const float u = R[4 * kk + j], w = a[j];
      R[4 * kk + j] = c * u + sn * w;
      a[j] = -sn * u + c * w;
    }
    a[kk] = 0.0f;
  }
}
__device__ __forceinline__ void givens_rows3(float* B, float* U, int p, int q, int col) {
  const float x = B[3 * p + col], y = B[3 * q + col];
  const float rn = sqrtf(x * x + y * y);
  float c = 1.0f, sn = 0.0f;
  if (rn > 0.0f) {
    c = x / rn;
    sn = y / rn;
  }
#pragma unroll
  for (int kk = 0; kk < 3; kk++) {
    const float bp = B[3 * p + kk], bq = B[3 * q + kk];
    B[3 * p + kk] = c * bp + sn * bq;
    B[3 * q + kk] = -sn * bp + c * bq;
  }
#pragma unroll
  for (int kk = 0; kk < 3; kk++) {
    const float up = U[3 * kk + p], uq = U[3 * kk + q];
    U[3 * kk + p] = c * up + sn * uq;
    U[3 * kk + q] = -sn * up + c * uq;
  }
}
// A = U diag(s) V^T: V = Jacobi eigenvectors of A^T A by decreasing
// eigenvalue, then a Givens QR of A V = U B, s = diag(B) (McAdams et al. 2011)
__device__ __forceinline__ void svd3(const float* A, float* U, float* sg, float* V) {
  float M[9], ev[3];
#pragma unroll
  for (int a = 0; a < 3; a++)
#pragma unroll
    for (int b = 0; b < 3; b++) M[3 * a + b] = A[a] * A[b] + A[3 + a] * A[3 + b] + A[6 + a] * A[6 + b];
  eig3(M, ev, V);
#pragma unroll
  for (int a = 0; a < 2; a++)
#pragma unroll
    for (int b = 0; b < 2 - a; b++)
      if (ev[b] < ev[b + 1]) {
        const float t = ev[b];
        ev[b] = ev[b + 1];
        ev[b + 1] = t;
#pragma unroll
        for (int kk = 0; kk < 3; kk++) {
          const float x = V[3 * kk + b];
          V[3 * kk + b] = V[3 * kk + b + 1];
          V[3 * kk + b + 1] = x;
        }
      }
  float B[9];
#pragma unroll
  for (int a = 0; a < 3; a++)
#pragma unroll
    for (int b = 0; b < 3; b++) B[3 * a + b] = A[3 * a] * V[b] + A[3 * a + 1] * V[3 + b] + A[3 * a + 2] * V[6 + b];
#pragma unroll
  for (int kk = 0; kk < 9; kk++) U[kk] = (kk % 4) == 0 ? 1.0f : 0.0f;
  givens_rows3(B, U, 0, 1, 0);
  givens_rows3(B, U, 0, 2, 0);
  givens_rows3(B, U, 1, 2, 1);
  sg[0] = B[0];
  sg[1] = B[4];
  sg[2] = B[8];
}
__device__ __forceinline__ void qef_solve(const float* R, float* x) {
  float A[9];
#pragma unroll
  for (int a = 0; a < 3; a++)
#pragma unroll
    for (int b = 0; b < 3; b++) A[3 * a + b] = R[4 * a + b];
  float Us[9], sg[3], V[9];
  svd3(A, Us, sg, V);
  const float bb[3] = {R[3], R[7], R[11]};
  const float tiny = 1e-6f * fmaxf(fabsf(sg[0]), fmaxf(fabsf(sg[1]), fabsf(sg[2])));
  float z[3];
#pragma unroll
  for (int kk = 0; kk < 3; kk++) {
    const float bk = Us[kk] * bb[0] + Us[3 + kk] * bb[1] + Us[6 + kk] * bb[2];
    const float sc = (sg[kk] < 0.0f ? -1.0f : 1.0f) * fmaxf(0.1f, fabsf(sg[kk]));
    z[kk] = fabsf(sg[kk]) > tiny ? bk / sc : 0.0f;
  }
#pragma unroll
  for (int a = 0; a < 3; a++) x[a] = V[3 * a] * z[0] + V[3 * a + 1] * z[1] + V[3 * a + 2] * z[2];
}

__device__ __forceinline__ int cube_vertex(const K& k, int x, int y, int z) {
  const int gx = x - k.glo[0], gy = y - k.glo[1], gz = z - k.glo[2];
  if (gx < 0 || gy < 0 || gz < 0 || gx >= k.gdim[0] || gy >= k.gdim[1] || gz >= k.gdim[2]) return 0;
  return k.cube_id[gidx(k, gx, gy, gz)];
}

// dual_contouring_impl (:1532-1596) for the cubes with a crossing, and the
// number of triangles each emits (dual_contouring_polygen, :1708-1763).
//
// A lane per edge of a cube (16 lanes, three of the others for the faces) forms
// the crossing point and its normal, the longest part (64 field values), into
// LDS; then a lane per cube folds them in edge order and solves, the
// workgroup's first wavefront for its 64 cubes.  Microseconds at 5,013, 46,166
// and 66,148 cubes: 26, 71 and 101; with a thread per vertex of the grid, few of
// a wavefront's lanes on a cube, 248, 530 and 450.
constexpr int DC_CUBES = 64;
constexpr int DC_THREADS = 16 * DC_CUBES;
__global__ __launch_bounds__(DC_THREADS) __attribute__((amdgpu_waves_per_eu(4, 4))) void k_dc_point(K k, int nv) {
  __shared__ float pn[12][6][DC_CUBES + 1];  // crossing point and normal of an edge
  const int e = threadIdx.x & 15, c = threadIdx.x >> 4;
  const int m = blockIdx.x * DC_CUBES + c;
  if (m < nv) {
    const int q = k.cubes[m];
    const int mask = k.flag[q] & 0xFFF;
    const int gz = q % k.gdim[2], gy = (q / k.gdim[2]) % k.gdim[1], gx = q / (k.gdim[1] * k.gdim[2]);
    const int x = gx + k.glo[0], y = gy + k.glo[1], z = gz + k.glo[2];
    bool quad = false;
    if (e < 12) {
      if (mask & (1 << e)) {
        float cv[2], cp[2][3], p[3], n[3];
#pragma unroll
        for (int s = 0; s < 2; s++) {
          const int* o = CORNER[EDGE[e][s]];
          cv[s] = val_at(k, k.field, x + o[0], y + o[1], z + o[2]);
          vpos(k, x + o[0], y + o[1], z + o[2], cp[s]);
        }
        vinterp(k.iso, cp[0], cp[1], cv[0], cv[1], p);
        normal_at(k, p, n);
#pragma unroll
        for (int a = 0; a < 3; a++) {
          pn[e][a][c] = p[a];
          pn[e][3 + a][c] = n[a];
        }
      }
    } else if (e < 15) {
      const int (&adj)[3][3] = ADJ[e - 12];
      quad = (mask & (1 << ADJ_W[e - 12])) && cube_vertex(k, x + adj[0][0], y + adj[0][1], z + adj[0][2]) &&
             cube_vertex(k, x + adj[1][0], y + adj[1][1], z + adj[1][2]) &&
             cube_vertex(k, x + adj[2][0], y + adj[2][1], z + adj[2][2]);
    }
    const int quads = __popcll(__ballot(quad) >> (threadIdx.x & 48) & 0x7000ull);
    if (e == 0) k.tcount[m] = 2 * quads;
  }
  __syncthreads();
  if (threadIdx.x >= DC_CUBES) return;
  const int t = threadIdx.x, mt = blockIdx.x * DC_CUBES + t;
  if (mt >= nv) return;
  const int q = k.cubes[mt];
  const int mask = k.flag[q] & 0xFFF;
  float mean[3] = {0.0f, 0.0f, 0.0f};
  int cnt = 0;
  for (int w = 0; w < 12; w++) {
    if (!(mask & (1 << w))) continue;
    mean[0] += pn[w][0][t];
    mean[1] += pn[w][1][t];
    mean[2] += pn[w][2][t];
    cnt++;
  }
  const float fc = (float)cnt;
  mean[0] /= fc;
  mean[1] /= fc;
  mean[2] /= fc;
  float R[16];
#pragma unroll
  for (int a = 0; a < 16; a++) R[a] = 0.0f;
  for (int w = 0; w < 12; w++) {
    if (!(mask & (1 << w))) continue;
    const float d0 = pn[w][0][t] - mean[0], d1 = pn[w][1][t] - mean[1], d2 = pn[w][2][t] - mean[2];
    const float n0 = pn[w][3][t], n1 = pn[w][4][t], n2 = pn[w][5][t];
    qef_add(R, n0, n1, n2, n0 * d0 + n1 * d1 + n2 * d2);
  }
  float r[3];
  qef_solve(R, r);
  const float pt[3] = {r[0] + mean[0], r[1] + mean[1], r[2] + mean[2]};
  int v[3];
  voxel_of(k, pt, v);
  const int gz = q % k.gdim[2], gy = (q / k.gdim[2]) % k.gdim[1], gx = q / (k.gdim[1] * k.gdim[2]);
  const bool in = v[0] == gx + k.glo[0] && v[1] == gy + k.glo[1] && v[2] == gz + k.glo[2];
  float* out = k.verts + 3 * (long)mt;
#pragma unroll
  for (int a = 0; a < 3; a++) out[a] = in ? pt[a] : mean[a];
}

__global__ void k_faces(K k, int nv) {
  const int m = blockIdx.x * blockDim.x + threadIdx.x;
  if (m >= nv || !k.tcount[m]) return;
  const int q = k.cubes[m];
  const int gz = q % k.gdim[2], gy = (q / k.gdim[2]) % k.gdim[1], gx = q / (k.gdim[1] * k.gdim[2]);
  const int x = gx + k.glo[0], y = gy + k.glo[1], z = gz + k.glo[2];
  const int mask = k.flag[q] & 0xFFF, ci = k.flag[q] >> 12;
  int* f = k.faces + 3 * (long)k.tstart[m];
  for (int e = 0; e < 3; e++) {
    const int w = ADJ_W[e];
    if (!(mask & (1 << w))) continue;
    const int i1 = m + 1;
    const int i2 = cube_vertex(k, x + ADJ[e][0][0], y + ADJ[e][0][1], z + ADJ[e][0][2]);
    const int i3 = cube_vertex(k, x + ADJ[e][1][0], y + ADJ[e][1][1], z + ADJ[e][1][2]);
    const int i4 = cube_vertex(k, x + ADJ[e][2][0], y + ADJ[e][2][1], z + ADJ[e][2][2]);
    if (!(i2 && i3 && i4)) continue;
    const int flip = ((ci >> EDGE[w][0]) & 1) != (w == 11);
    if (!flip) {
      f[0] = i3 - 1; f[1] = i2 - 1; f[2] = i1 - 1;
      f[3] = i4 - 1; f[4] = i3 - 1; f[5] = i1 - 1;
    } else {
      f[0] = i1 - 1; f[1] = i2 - 1; f[2] = i3 - 1;
      f[3] = i1 - 1; f[4] = i3 - 1; f[5] = i4 - 1;
    }
    f += 6;
  }
}

// get_velocity_at (:1352-1359): 0 outside written blocks
__device__ __forceinline__ void vel_at(const K& k, int x, int y, int z, float* out) {
  const int gx = x - k.glo[0], gy = y - k.glo[1], gz = z - k.glo[2];
  if (gx < 0 || gy < 0 || gz < 0 || gx >= k.gdim[0] || gy >= k.gdim[1] || gz >= k.gdim[2]) {
    out[0] = out[1] = out[2] = 0.0f;
    return;
  }
  const long q = gidx(k, gx, gy, gz);
  for (int c = 0; c < 3; c++) out[c] = k.vfield[3 * q + c];
}

// per mesh vertex: the normal (process_normal, :1384-1410) and the velocity
// (process_velocity_at with trilinear_interpolate, :1362-1375, :1324-1333)
__global__ void k_vertex_attrs(K k, long nv, int want_normals, int want_vel) {
  const long v = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (v >= nv) return;
  float p[3] = {k.verts[3 * v], k.verts[3 * v + 1], k.verts[3 * v + 2]};
  if (want_normals) normal_at(k, p, k.normals + 3 * v);
  if (!want_vel) return;
  float* out = k.mvel + 3 * v;
  if (!k.vel) {
    out[0] = out[1] = out[2] = 0.0f;
    return;
  }
  int c3[3];
  voxel_of(k, p, c3);
  float base[3];
  vpos(k, c3[0], c3[1], c3[2], base);
  const float xd = (p[0] - base[0]) / k.vs, yd = (p[1] - base[1]) / k.vs, zd = (p[2] - base[2]) / k.vs;
  float c[8][3];
#pragma unroll
  for (int j = 0; j < 8; j++) vel_at(k, c3[0] + (j >> 2), c3[1] + ((j >> 1) & 1), c3[2] + (j & 1), c[j]);
#pragma unroll
  for (int a = 0; a < 3; a++) {
    const float c00 = c[0][a] * (1.0f - xd) + c[4][a] * xd;
    const float c01 = c[1][a] * (1.0f - xd) + c[5][a] * xd;
    const float c10 = c[2][a] * (1.0f - xd) + c[6][a] * xd;
    const float c11 = c[3][a] * (1.0f - xd) + c[7][a] * xd;
    const float c0 = c00 * (1.0f - yd) + c10 * yd;
    const float c1 = c01 * (1.0f - yd) + c11 * yd;
    out[a] = c0 * (1.0f - zd) + c1 * zd;
  }
}

// ------------------------------------------------------------------ host

template <typename T>
struct DBuf {
  T* p = nullptr;
  size_t cap = 0;
  hipError_t ensure(size_t n) {
    if (n <= cap && p) return hipSuccess;
    if (p) (void)hipFree(p);
    p = nullptr;
    cap = 0;
    const size_t c = n > 0 ? n : 1;
    hipError_t e = hipMalloc(&p, c * sizeof(T));
    if (e == hipErrorOutOfMemory && free_kept()) {
      (void)hipGetLastError();
      e = hipMalloc(&p, c * sizeof(T));
    }
    if (e == hipSuccess) cap = c;
    return e;
  }
  void release() {
    if (p) (void)hipFree(p);
    p = nullptr;
    cap = 0;
  }
};

// What the host reads between the launches, written by k_report into pinned
// memory: the ticket last.
struct Report {
  unsigned long long ticket;
  double stats[4];
  int err, count, bounds[6];
  long long active;
};
__global__ __launch_bounds__(256) void k_report(K k, const int* count, int active, Report* host, unsigned long long ticket) {
  __shared__ int red[4];
  const int t = threadIdx.x;
  int na = 0;
  if (active)
    for (long b = t; b < k.nblock; b += 256) na += k.active[b];
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) na += __shfl_xor(na, off, 64);
  if ((t & 63) == 0) red[t >> 6] = na;
  __syncthreads();
  if (t != 0) return;
  host->err = *k.err;
  host->count = count ? *count : 0;
  host->active = (long long)red[0] + red[1] + red[2] + red[3];
  for (int a = 0; a < 6; a++) host->bounds[a] = k.bounds[a];
  for (int a = 0; a < 4; a++) host->stats[a] = k.stats[a];
  __hip_atomic_store(&host->ticket, ticket, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

struct Surface {
  nn_surface_params prm{};
  K k{};
  hipStream_t st = nullptr;
  DBuf<float> pos, vel, G, xbar, field0, field, tmp, verts, normals, vfield, mvel;
  DBuf<int> vcount, vstart, vslot, vlist, pvox, flag, cube_id, cubes, tcount, tstart, faces, err, bounds, scratch;
  DBuf<unsigned char> active;
  DBuf<float4> rec, sorted;
  DBuf<double> stats, part;
  DBuf<long long> pcount;
  long nverts = 0, ntris = 0, nactive = 0;
  double sd = 0.0;
  bool have = false;
  int64_t budget = 0;  // device bytes a run may use (0 = no limit)
  Report *report = nullptr, *report_dev = nullptr;  // pinned, and its device address
  unsigned long long ticket = 0;
  int *stage = nullptr, *stage_dev = nullptr;  // pinned, STAGE_BYTES
  bool stage_read = false;                     // a kernel may still read it

  ~Surface() {
    for (auto* b : {&pos, &vel, &G, &xbar, &field0, &field, &tmp, &verts, &normals, &vfield, &mvel}) b->release();
    for (auto* b : {&vcount, &vstart, &vslot, &vlist, &pvox, &flag, &cube_id, &cubes, &tcount, &tstart, &faces, &err, &bounds, &scratch})
      b->release();
    active.release();
    rec.release();
    sorted.release();
    stats.release();
    part.release();
    pcount.release();
    if (report) (void)hipHostFree(report);
    if (stage) (void)hipHostFree(stage);
    if (st) (void)hipStreamDestroy(st);
  }
};

static inline unsigned grid1(long n, int b) { return (unsigned)((n + b - 1) / b); }

// exclusive scan of in[0, L) (nz: of in[i] != 0) into out[0, L], total in out[L]
static hipError_t scan(Surface& S, const int* in, int* out, long L, int nz = 0) {
  if (L <= 0) {
    hipLaunchKernelGGL(k_fill_i32, dim3(1), dim3(64), 0, S.st, out, 0, 1L);
    return hipGetLastError();
  }
  hipError_t e = S.scratch.ensure((size_t)scan_tmp_ints(L));
  if (e != hipSuccess) return e;
  launch_scan_i32(in, (int)L, S.scratch.p, out, S.st, nz, 1);
  return hipGetLastError();
}

// Caller's arrays of up to STAGE_BYTES together cross through pinned memory that
// kernels read and write: a copy of 60 to 130 KB to or from pageable memory takes
// 40 to 80 us, this 11 to 17 (fields of that size).
constexpr size_t STAGE_BYTES = 1 << 20;
struct Piece {
  void* p;     // device side
  void* host;  // caller's side
  size_t bytes;
};
struct Pieces {
  int* dev[3];
  long end[3];  // words of the pieces up to this one
};
__global__ void k_stage(Pieces c, int* stage, int in) {
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= c.end[2]) return;
  const int a = i < c.end[0] ? 0 : i < c.end[1] ? 1 : 2;
  int* d = c.dev[a] + (i - (a ? c.end[a - 1] : 0));
  if (in) *d = stage[i];
  else stage[i] = *d;
}

static int fail(hipError_t e, const char* what) { return hip_fail(e, what); }

#define SR_HIP(expr, what)                      \
  do {                                          \
    hipError_t e__ = (expr);                    \
    if (e__ != hipSuccess) return fail(e__, what); \
  } while (0)

// Launches k_report and waits for it (as Batch::await: polled, a long wait left to
// the stream's); report() then returns the error the launches so far have flagged.
static int wait_report(Surface& S, const int* count, bool active) {
  if (!S.report) {
    SR_HIP(hipHostMalloc((void**)&S.report, sizeof(Report), hipHostMallocDefault), "nn_surface_run: alloc");
    S.report->ticket = 0;
    SR_HIP(hipHostGetDevicePointer((void**)&S.report_dev, S.report, 0), "nn_surface_run");
  }
  hipLaunchKernelGGL(k_report, dim3(1), dim3(256), 0, S.st, S.k, count, active ? 1 : 0, S.report_dev, ++S.ticket);
  SR_HIP(hipGetLastError(), "nn_surface_run: launch");
  const auto start = std::chrono::steady_clock::now();
  for (int polls = 1; __atomic_load_n(&S.report->ticket, __ATOMIC_ACQUIRE) != S.ticket; polls++) {
    if (polls % 64 == 0 && std::chrono::steady_clock::now() - start > std::chrono::microseconds(300)) {
      SR_HIP(hipStreamSynchronize(S.st), "nn_surface_run");
      if (__atomic_load_n(&S.report->ticket, __ATOMIC_ACQUIRE) == S.ticket) break;
      set_error("nn_surface_run: a launch did not report its end");
      return NN_E_HIP;
    }
    __builtin_ia32_pause();
  }
  S.stage_read = false;
  return NN_OK;
}

static int report(Surface& S, const int* count = nullptr, bool active = false) {
  const int rc = wait_report(S, count, active);
  if (rc) return rc;
  const int err = S.report->err;
  if (err & ERR_OUT_OF_GRID) {
    set_error("nn_surface_run: a particle lies below the bounding box's first voxel, or its position is not finite");
    return NN_E_OUT_OF_GRID;
  }
  if (err & ERR_VOXEL_OVERFLOW) {
    set_error("nn_surface_run: more than 64 particles in one voxel (max_num_particle_per_voxel)");
    return NN_E_CELL_OVERFLOW;
  }
  if (err & ERR_RANGE) {
    set_error("nn_surface_run: a field contribution is not finite or exceeds 2^20");
    return NN_E_NAN;
  }
  return NN_OK;
}

// Copies pieces in (before a run) or out (after one); in: the run waits for it.
static int transfer(Surface& S, bool in, std::initializer_list<Piece> pieces, const char* what) {
  (void)hipGetLastError();  // what another call left on this thread is not this one's error
  size_t total = 0;
  bool host = true;  // memory that the CPU can use
  for (const Piece& q : pieces) {
    total += q.bytes;
    hipPointerAttribute_t at{};
    if (q.bytes == 0) continue;
    if (hipPointerGetAttributes(&at, q.host) != hipSuccess) (void)hipGetLastError();
    else host = host && at.type != hipMemoryTypeDevice;
  }
  if (total == 0) return NN_OK;
  if (!host || total > STAGE_BYTES) {
    for (const Piece& q : pieces) {
      if (q.bytes == 0) continue;
      if (in) SR_HIP(hipMemcpyAsync(q.p, q.host, q.bytes, hipMemcpyHostToDevice, S.st), what);
      else SR_HIP(hipMemcpy(q.host, q.p, q.bytes, hipMemcpyDeviceToHost), what);
    }
    return NN_OK;
  }
  if (!S.stage) {
    SR_HIP(hipHostMalloc((void**)&S.stage, STAGE_BYTES, hipHostMallocDefault), what);
    SR_HIP(hipHostGetDevicePointer((void**)&S.stage_dev, S.stage, 0), what);
  }
  if (S.stage_read) SR_HIP(hipStreamSynchronize(S.st), what);  // by a run that ended before its first report
  S.stage_read = in;
  Pieces c{};
  long words = 0;
  int a = 0;
  for (const Piece& q : pieces) {
    if (in && q.bytes) std::memcpy(S.stage + words, q.host, q.bytes);
    words += (long)(q.bytes / 4);
    c.dev[a] = static_cast<int*>(q.p);
    c.end[a++] = words;
  }
  for (; a < 3; a++) c.end[a] = words;
  hipLaunchKernelGGL(k_stage, dim3(grid1(words, 256)), dim3(256), 0, S.st, c, S.stage_dev, in ? 1 : 0);
  SR_HIP(hipGetLastError(), what);
  if (in) return NN_OK;
  const int rc = wait_report(S, nullptr, false);
  if (rc) return rc;
  words = 0;
  for (const Piece& q : pieces) {
    if (q.bytes) std::memcpy(q.host, S.stage + words, q.bytes);
    words += (long)(q.bytes / 4);
  }
  return NN_OK;
}

static int run(Surface& S, const float* dpos, const float* dvel, long n) {
  K& k = S.k;
  S.have = false;
  k.n = (int)n;
  k.pos = dpos;
  k.vel = (S.prm.velocity && k.aniso) ? dvel : nullptr;  // the reference samples velocity in the smooth field only
  SR_HIP(S.err.ensure(1), "nn_surface_run: alloc");
  SR_HIP(S.bounds.ensure(6), "nn_surface_run: alloc");
  SR_HIP(S.stats.ensure(4), "nn_surface_run: alloc");
  k.err = S.err.p;
  k.bounds = S.bounds.p;
  k.stats = S.stats.p;
  hipLaunchKernelGGL(k_start, dim3(1), dim3(64), 0, S.st, k);
  hipLaunchKernelGGL(k_bounds, dim3(grid1(n, BOUNDS_THREADS)), dim3(BOUNDS_THREADS), 0, S.st, k);
  int rc = report(S);
  if (rc) return rc;
  const int* hb = S.report->bounds;
  // voxel range and the vertex grid (blocks that the field passes can write)
  long nvox = 1;
  for (int a = 0; a < 3; a++) {
    k.vlo[a] = hb[a];
    k.vdim[a] = hb[3 + a] - hb[a] + 1;
    nvox *= k.vdim[a];
  }
  long nvert = 1, nblock = 1;
  for (int a = 0; a < 3; a++) {
    const int vmin = k.vlo[a], vmax = k.vlo[a] + k.vdim[a] - 1;
    long lo = vmin - 1, hi = (long)vmax + 1;
    if (k.aniso) {
      lo = std::min<long>(lo, vmin - k.off);
      hi = std::max<long>(hi, (long)vmax - k.off + k.R);
    }
    if (lo < 0) lo = 0;
    const long glo = (lo / BLOCK) * BLOCK, ghi = (hi / BLOCK) * BLOCK + BLOCK - 1;
    k.glo[a] = (int)glo;
    k.gdim[a] = (int)(ghi - glo + 1);
    k.bdim[a] = k.gdim[a] / BLOCK;
    nvert *= k.gdim[a];
    nblock *= k.bdim[a];
  }
  k.nvox = nvox;
  k.nvert = nvert;
  k.nblock = nblock;
  // the device bytes of the buffers below, the inputs' copies (pos, vel) and the
  // scans' partials; the mesh's are added once its size is known
  double need = (double)nvox * 8 + (double)nvert * (k.vel ? 32 : 20) + (double)nblock * 17 +
                (double)n * (84 + (k.aniso ? 16 * REC_QUADS : 0)) + 4.0 * (double)scan_tmp_ints(std::max(nvox, nvert));
  if (dpos == S.pos.p) need += 12.0 * (double)n;
  if (dvel) need += 12.0 * (double)n;
  // int32 scans: up to 6 triangles per cube must stay below 2^31
  if (nvert > (1L << 28) || nvox > (1L << 30) || (S.budget > 0 && need > (double)S.budget)) {
    set_error("nn_surface_run: the vertex grid over the particles' extent exceeds the device budget (" +
              std::to_string(nvert) + " vertices, " + std::to_string(n) + " particles)");
    return NN_E_OOM;
  }
  const auto mesh_fits = [&](double bytes) {
    need += bytes;
    if (!(S.budget > 0 && need > (double)S.budget)) return true;
    set_error("nn_surface_run: the mesh exceeds the device budget");
    return false;
  };
  SR_HIP(S.vcount.ensure(nvox), "nn_surface_run: alloc");
  SR_HIP(S.vstart.ensure(nvox + 1), "nn_surface_run: alloc");
  SR_HIP(S.vslot.ensure(n), "nn_surface_run: alloc");
  SR_HIP(S.vlist.ensure(n), "nn_surface_run: alloc");
  SR_HIP(S.sorted.ensure(n), "nn_surface_run: alloc");
  SR_HIP(S.pvox.ensure(3 * n), "nn_surface_run: alloc");
  SR_HIP(S.G.ensure(9 * n), "nn_surface_run: alloc");
  SR_HIP(S.xbar.ensure(3 * n), "nn_surface_run: alloc");
  if (k.aniso) SR_HIP(S.rec.ensure(REC_QUADS * (size_t)n), "nn_surface_run: alloc");
  SR_HIP(S.active.ensure(nblock), "nn_surface_run: alloc");
  SR_HIP(S.field0.ensure(nvert), "nn_surface_run: alloc");
  SR_HIP(S.field.ensure(nvert), "nn_surface_run: alloc");
  SR_HIP(S.tmp.ensure(nvert), "nn_surface_run: alloc");
  SR_HIP(S.flag.ensure(nvert), "nn_surface_run: alloc");
  SR_HIP(S.cube_id.ensure(nvert + 1), "nn_surface_run: alloc");
  SR_HIP(S.part.ensure(nblock), "nn_surface_run: alloc");
  SR_HIP(S.pcount.ensure(nblock), "nn_surface_run: alloc");
  if (k.vel) {
    SR_HIP(S.vfield.ensure(3 * nvert), "nn_surface_run: alloc");
    k.vfield = S.vfield.p;
  }
  k.vcount = S.vcount.p;
  k.vstart = S.vstart.p;
  k.vslot = S.vslot.p;
  k.vlist = S.vlist.p;
  k.pvox = S.pvox.p;
  k.G = S.G.p;
  k.xbar = S.xbar.p;
  k.rec = S.rec.p;
  k.sorted = S.sorted.p;
  k.active = S.active.p;
  k.field0 = S.field0.p;
  k.field = S.field.p;
  k.tmp = S.tmp.p;
  k.flag = S.flag.p;
  k.cube_id = S.cube_id.p;
  // hash
  hipLaunchKernelGGL(k_fill_i32, dim3(grid1(nvox, 256)), dim3(256), 0, S.st, k.vcount, 0, nvox);
  hipLaunchKernelGGL(k_vcount, dim3(grid1(n, 256)), dim3(256), 0, S.st, k);
  SR_HIP(scan(S, k.vcount, k.vstart, nvox), "nn_surface_run: scan");
  int* bucket = reinterpret_cast<int*>(k.xbar);  // written by k_aniso, after this
  hipLaunchKernelGGL(k_vplace, dim3(grid1(n, 256)), dim3(256), 0, S.st, k, bucket);
  hipLaunchKernelGGL(k_vsort, dim3(grid1(n, 256)), dim3(256), 0, S.st, k, bucket);
  if ((rc = report(S))) return rc;  // before sweeps over voxels that may hold any number
  // anisotropic kernel and field
  if (k.aniso) hipLaunchKernelGGL(k_aniso, dim3(grid1(n, AN_GROUPS)), dim3(16 * AN_GROUPS), 0, S.st, k);
  hipLaunchKernelGGL(k_fill_u8, dim3(grid1(nblock, 256)), dim3(256), 0, S.st, k.active, nblock);
  hipLaunchKernelGGL(k_mark, dim3(grid1(n, 256)), dim3(256), 0, S.st, k);
  const dim3 tiles((unsigned)(nvert / FIELD_THREADS)), ft(FIELD_THREADS);
  if (k.aniso) hipLaunchKernelGGL(k_field<FIELD_ANISO>, tiles, ft, 0, S.st, k);
  else hipLaunchKernelGGL(k_field<FIELD_ISO>, tiles, ft, 0, S.st, k);
  if (k.vel) {
    hipLaunchKernelGGL(k_check_velocities, dim3(grid1(3 * n, 256)), dim3(256), 0, S.st, k);
    hipLaunchKernelGGL(k_field<FIELD_VELOCITY>, tiles, ft, 0, S.st, k);
  }
  // smoothing
  hipLaunchKernelGGL(k_stats, dim3((unsigned)nblock), dim3(ST_THREADS), 0, S.st, k, 0, S.part.p, S.pcount.p);
  hipLaunchKernelGGL(k_stats_final, dim3(1), dim3(ST_THREADS), 0, S.st, k, 0, S.part.p, S.pcount.p);
  hipLaunchKernelGGL(k_stats, dim3((unsigned)nblock), dim3(ST_THREADS), 0, S.st, k, 1, S.part.p, S.pcount.p);
  hipLaunchKernelGGL(k_stats_final, dim3(1), dim3(ST_THREADS), 0, S.st, k, 1, S.part.p, S.pcount.p);
  for (int it = 0; it < S.prm.smooth_iterations; it++) {
    hipLaunchKernelGGL(k_smooth, dim3(grid1(nvert, 256)), dim3(256), 0, S.st, k, k.field, k.tmp);
    std::swap(k.field, k.tmp);
  }
  // contour
  hipLaunchKernelGGL(k_cube_flag, dim3(grid1(nvert, 256)), dim3(256), 0, S.st, k);
  SR_HIP(scan(S, k.flag, k.cube_id, nvert, 1), "nn_surface_run: scan");
  if ((rc = report(S, k.cube_id + nvert))) return rc;
  const int nv = S.report->count;
  // verts, cubes, tcount, tstart; normals and velocities
  if (!mesh_fits((double)nv * (24 + (S.prm.normals ? 12 : 0) + (S.prm.velocity ? 12 : 0)))) return NN_E_OOM;
  SR_HIP(S.verts.ensure(3 * (size_t)nv), "nn_surface_run: alloc");
  SR_HIP(S.cubes.ensure(nv), "nn_surface_run: alloc");
  SR_HIP(S.tcount.ensure(nv), "nn_surface_run: alloc");
  SR_HIP(S.tstart.ensure((size_t)nv + 1), "nn_surface_run: alloc");
  k.verts = S.verts.p;
  k.cubes = S.cubes.p;
  k.tcount = S.tcount.p;
  k.tstart = S.tstart.p;
  hipLaunchKernelGGL(k_cube_id, dim3(grid1(nvert, 256)), dim3(256), 0, S.st, k);
  if (nv > 0) hipLaunchKernelGGL(k_dc_point, dim3(grid1(nv, DC_CUBES)), dim3(DC_THREADS), 0, S.st, k, nv);
  SR_HIP(scan(S, k.tcount, k.tstart, nv), "nn_surface_run: scan");
  if ((rc = report(S, k.tstart + nv, true))) return rc;
  const int nt = S.report->count;
  S.nactive = (long)S.report->active;  // the written blocks and the deviation, for the caller's statistics
  S.sd = S.report->stats[3];
  if (!mesh_fits(12.0 * (double)nt)) return NN_E_OOM;
  SR_HIP(S.faces.ensure(3 * (size_t)nt), "nn_surface_run: alloc");
  k.faces = S.faces.p;
  if (nv > 0) hipLaunchKernelGGL(k_faces, dim3(grid1(nv, 128)), dim3(128), 0, S.st, k, nv);
  const int want_n = S.prm.normals ? 1 : 0, want_v = S.prm.velocity ? 1 : 0;
  if ((want_n || want_v) && nv > 0) {
    if (want_n) {
      SR_HIP(S.normals.ensure(3 * (size_t)nv), "nn_surface_run: alloc");
      k.normals = S.normals.p;
    }
    if (want_v) {
      SR_HIP(S.mvel.ensure(3 * (size_t)nv), "nn_surface_run: alloc");
      k.mvel = S.mvel.p;
    }
    hipLaunchKernelGGL(k_vertex_attrs, dim3(grid1(nv, 128)), dim3(128), 0, S.st, k, (long)nv, want_n, want_v);
  }
  SR_HIP(hipGetLastError(), "nn_surface_run: launch");
  if ((rc = report(S))) return rc;
  S.nverts = nv;
  S.ntris = nt;
  S.have = true;
  return NN_OK;
}

// a scene's fluid positions, from the batch's cell order into original-index
// order (the reference numbers the fluid first, so ids are 0 .. n_fluid - 1)
__global__ void k_fluid_positions(const float4* pos, const float4* vel, const int* info, int pb, int n, int nf, float* out,
                                  float* vout, int* err) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= n) return;
  const int inf = info[pb + t];
  if ((inf >> 28) != KIND_FLUID) return;
  const int id = inf & 0x0FFFFFFF;
  if (id >= nf) {
    atomicOr(err, 1);
    return;
  }
  const float4 p = pos[pb + t];
  out[3 * (long)id] = p.x;
  out[3 * (long)id + 1] = p.y;
  out[3 * (long)id + 2] = p.z;
  if (vout) {
    const float4 v = vel[pb + t];
    vout[3 * (long)id] = v.x;
    vout[3 * (long)id + 1] = v.y;
    vout[3 * (long)id + 2] = v.z;
  }
}

}  // namespace sr
}  // namespace nn

using nn::sr::Surface;

struct nn_surface {
  Surface impl;
};

int nn::surface_run_scene(nn_surface* h, Batch& b, int k) {
  Surface& S = h->impl;
  const SceneHost& sc = *b.scenes[k];
  const int nf = sc.n_fluid;
  if (nf <= 0) {
    set_error("nn_surface_run_context: the scene has no fluid particles");
    return NN_E_ARG;
  }
  hipError_t e = hipStreamSynchronize(b.stream);  // the step's positions are complete
  if (e == hipSuccess) e = S.pos.ensure(3 * (size_t)nf);
  if (e == hipSuccess) e = S.err.ensure(1);
  const bool with_vel = S.prm.velocity != 0;
  if (e == hipSuccess && with_vel) e = S.vel.ensure(3 * (size_t)nf);
  if (e != hipSuccess) return hip_fail(e, "nn_surface_run_context");
  hipLaunchKernelGGL(sr::k_fill_i32, dim3(1), dim3(64), 0, S.st, S.err.p, 0, 1L);
  hipLaunchKernelGGL(sr::k_fluid_positions, dim3((sc.n + 255) / 256), dim3(256), 0, S.st, b.d.pos, b.d.vel, b.d.info,
                     sc.p_begin, sc.n, nf, S.pos.p, with_vel ? S.vel.p : nullptr, S.err.p);
  int err = 0;
  e = hipMemcpyAsync(&err, S.err.p, sizeof(int), hipMemcpyDeviceToHost, S.st);
  if (e == hipSuccess) e = hipStreamSynchronize(S.st);
  if (e != hipSuccess) return hip_fail(e, "nn_surface_run_context");
  if (err) {
    set_error("nn_surface_run_context: fluid particles must be numbered 0 .. n_fluid - 1 (the reference numbers them first)");
    return NN_E_UNSUPPORTED;
  }
  return sr::run(S, S.pos.p, with_vel ? S.vel.p : nullptr, nf);
}

extern "C" {

int32_t nn_surface_create(const nn_surface_params* p, nn_surface** out) {
  if (!p || !out) {
    nn::set_error("nn_surface_create: bad arguments");
    return NN_E_ARG;
  }
  *out = nullptr;
  if (!(p->voxel_size > 0.0) || !(p->particle_radius > 0.0) || !(p->smooth_radius > 0.0) ||
      p->smooth_iterations < 0 || p->smooth_iterations > 64) {
    nn::set_error("nn_surface_create: voxel_size, particle_radius and smooth_radius must be positive, "
                  "smooth_iterations in [0, 64]");
    return NN_E_ARG;
  }
  nn_surface* H = new nn_surface();
  Surface* S = &H->impl;
  S->prm = *p;
  nn::sr::K& k = S->k;
  for (int a = 0; a < 3; a++) k.o[a] = (float)p->origin[a];
  k.vs = (float)p->voxel_size;
  const double r = p->particle_radius;
  k.sr = (float)p->smooth_radius;
  k.iso = (float)p->isolevel;
  k.vol = (float)(r * r * r * M_PI * 4 / 3);  // srtool.py:945
  k.acoef = (float)(315 / (64 * M_PI));        // :946
  k.c48 = (float)(48 / M_PI);
  k.c16 = (float)(16 / M_PI);
  k.lam = (float)0.9;  // akLambda, :929
  k.lam1 = (float)(1 - 0.9);
  k.kr = 4.0f;  // kr, ks, kn, :925-928
  k.ks = 1400.0f;
  k.kn = 0.5f;
  k.c2pi = (float)(2 * M_PI);
  k.cvs3 = (float)(p->voxel_size * p->voxel_size * p->voxel_size);
  k.aniso = p->anisotropic ? 1 : 0;
  k.mid = k.sr >= 0x1p-20f && k.sr <= 0x1p20f ? 1 : 0;
  k.R = (int)ceilf(4.0f * k.sr / k.vs) + 1;  // smooth_range, :1137
  k.off = k.R / 2;
  if (k.aniso && (k.R < 1 || k.R + 1 > nn::sr::BLOCK)) {
    nn::set_error("nn_surface_create: 4 * smooth_radius / voxel_size must be below 30 (the anisotropic box "
                  "spans at most two 32-vertex blocks per axis)");
    delete H;
    return NN_E_UNSUPPORTED;
  }
  hipError_t e = hipStreamCreateWithFlags(&S->st, hipStreamNonBlocking);
  if (e != hipSuccess) {
    delete H;
    return nn::hip_fail(e, "nn_surface_create: stream");
  }
  *out = H;
  return NN_OK;
}

int32_t nn_surface_destroy(nn_surface* s) {
  delete s;
  return NN_OK;
}

int32_t nn_surface_set_budget(nn_surface* s, int64_t bytes) {
  if (!s || bytes < 0) {
    nn::set_error("nn_surface_set_budget: bad arguments");
    return NN_E_ARG;
  }
  s->impl.budget = bytes;
  return NN_OK;
}

int32_t nn_surface_run_device(nn_surface* s, const float* dpos, int64_t n) {
  Surface* S = s ? &s->impl : nullptr;
  if (!S || !dpos || n <= 0 || n > (1L << 30)) {
    nn::set_error("nn_surface_run_device: bad arguments (n must be in [1, 2^30])");
    return NN_E_ARG;
  }
  return nn::sr::run(*S, dpos, nullptr, (long)n);
}

int32_t nn_surface_run(nn_surface* s, const float* pos, int64_t n) {
  Surface* S = s ? &s->impl : nullptr;
  if (!S || !pos || n <= 0 || n > (1L << 30)) {
    nn::set_error("nn_surface_run: bad arguments (n must be in [1, 2^30])");
    return NN_E_ARG;
  }
  hipError_t e = S->pos.ensure(3 * (size_t)n);
  if (e != hipSuccess) return nn::hip_fail(e, "nn_surface_run: alloc");
  const int rc = nn::sr::transfer(*S, true, {{S->pos.p, const_cast<float*>(pos), sizeof(float) * 3 * (size_t)n}}, "nn_surface_run: upload");
  if (rc) return rc;
  return nn::sr::run(*S, S->pos.p, nullptr, (long)n);
}

int32_t nn_surface_run_velocity(nn_surface* s, const float* pos, const float* vel, int64_t n) {
  Surface* S = s ? &s->impl : nullptr;
  if (!S || !pos || !vel || n <= 0 || n > (1L << 30)) {
    nn::set_error("nn_surface_run_velocity: bad arguments (n must be in [1, 2^30])");
    return NN_E_ARG;
  }
  if (!S->prm.velocity) {
    nn::set_error("nn_surface_run_velocity: the velocity channels were not requested (nn_surface_params.velocity)");
    return NN_E_STATE;
  }
  hipError_t e = S->pos.ensure(3 * (size_t)n);
  if (e == hipSuccess) e = S->vel.ensure(3 * (size_t)n);
  if (e != hipSuccess) return nn::hip_fail(e, "nn_surface_run_velocity: alloc");
  const size_t bytes = sizeof(float) * 3 * (size_t)n;
  const int rc = nn::sr::transfer(*S, true, {{S->pos.p, const_cast<float*>(pos), bytes}, {S->vel.p, const_cast<float*>(vel), bytes}},
                                  "nn_surface_run_velocity: upload");
  if (rc) return rc;
  return nn::sr::run(*S, S->pos.p, S->vel.p, (long)n);
}

int32_t nn_surface_mesh_velocity(nn_surface* s, float* out) {
  Surface* S = s ? &s->impl : nullptr;
  if (!S || (!out && S->nverts)) {
    nn::set_error("nn_surface_mesh_velocity: bad arguments");
    return NN_E_ARG;
  }
  if (!S->have || !S->prm.velocity) {
    nn::set_error("nn_surface_mesh_velocity: no completed run with the velocity channels");
    return NN_E_STATE;
  }
  return nn::sr::transfer(*S, false, {{S->k.mvel, out, sizeof(float) * 3 * S->nverts}}, "nn_surface_mesh_velocity");
}

int32_t nn_surface_info(nn_surface* s, int64_t* out, double* sd) {
  Surface* S = s ? &s->impl : nullptr;
  if (!S || !out) {
    nn::set_error("nn_surface_info: bad arguments");
    return NN_E_ARG;
  }
  if (!S->have) {
    nn::set_error("nn_surface_info: no completed run");
    return NN_E_STATE;
  }
  const nn::sr::K& k = S->k;
  for (int a = 0; a < 3; a++) {
    out[a] = k.glo[a];
    out[3 + a] = k.gdim[a];
    out[9 + a] = k.vlo[a];
    out[12 + a] = k.vdim[a];
  }
  out[6] = S->nverts;
  out[7] = S->ntris;
  out[8] = S->nactive;
  out[15] = k.n;
  if (sd) *sd = S->sd;
  return NN_OK;
}

int32_t nn_surface_mesh(nn_surface* s, float* vertices, int32_t* faces, float* normals) {
  Surface* S = s ? &s->impl : nullptr;
  if (!S || (!vertices && S->nverts) || (!faces && S->ntris)) {
    nn::set_error("nn_surface_mesh: bad arguments");
    return NN_E_ARG;
  }
  if (!S->have) {
    nn::set_error("nn_surface_mesh: no completed run");
    return NN_E_STATE;
  }
  if (normals && !S->prm.normals) {
    nn::set_error("nn_surface_mesh: normals were not requested (nn_surface_params.normals)");
    return NN_E_STATE;
  }
  return nn::sr::transfer(*S, false,
                          {{S->k.verts, vertices, sizeof(float) * 3 * S->nverts},
                           {S->k.faces, faces, sizeof(int) * 3 * S->ntris},
                           {S->k.normals, normals, normals ? sizeof(float) * 3 * S->nverts : 0}},
                          "nn_surface_mesh");
}

int32_t nn_surface_field(nn_surface* s, int32_t which, float* out, size_t count) {
  Surface* S = s ? &s->impl : nullptr;
  if (!S || !out || (which != 0 && which != 1)) {
    nn::set_error("nn_surface_field: bad arguments");
    return NN_E_ARG;
  }
  if (!S->have) {
    nn::set_error("nn_surface_field: no completed run");
    return NN_E_STATE;
  }
  if (count < (size_t)S->k.nvert) {
    nn::set_error("nn_surface_field: count below the grid's vertex count");
    return NN_E_ARG;
  }
  const float* src = which == 0 ? S->k.field0 : S->k.field;
  hipError_t e = hipMemcpy(out, src, sizeof(float) * S->k.nvert, hipMemcpyDeviceToHost);
  if (e != hipSuccess) return nn::hip_fail(e, "nn_surface_field");
  return NN_OK;
}

int32_t nn_surface_aniso(nn_surface* s, float* G, float* xbar, int64_t n) {
  Surface* S = s ? &s->impl : nullptr;
  if (!S || !G || !xbar) {
    nn::set_error("nn_surface_aniso: bad arguments");
    return NN_E_ARG;
  }
  if (!S->have || !S->k.aniso) {
    nn::set_error("nn_surface_aniso: no completed anisotropic run");
    return NN_E_STATE;
  }
  if (n != S->k.n) {
    nn::set_error("nn_surface_aniso: n differs from the last run's particle count");
    return NN_E_ARG;
  }
  hipError_t e = hipMemcpy(G, S->k.G, sizeof(float) * 9 * n, hipMemcpyDeviceToHost);
  if (e == hipSuccess) e = hipMemcpy(xbar, S->k.xbar, sizeof(float) * 3 * n, hipMemcpyDeviceToHost);
  if (e != hipSuccess) return nn::hip_fail(e, "nn_surface_aniso");
  return NN_OK;
}

}  // extern "C"
