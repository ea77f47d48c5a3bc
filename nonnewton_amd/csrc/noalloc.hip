// noalloc.hip -- nn_neighbors_noalloc: the neighbor lists of nn_neighbors
// (meta.ns.run_search() + meta.ns.neighbors, SPH/main.py:815-847) for
// positions already in device memory, written to device memory, with no
// device allocation: the search's scratch (cell counts, cell starts, scan
// partials, cell keys, the particles by cell and in cell order) lives in one
// file-scope __device__ array per device, at a fixed maximum size.
//
// Order and test are those of the context's search: cell = truncation of x / h
// (pos_to_index, :805-807), the 27 cells visited dx slowest and dz fastest,
// inside a cell increasing particle index (the serial fill order of
// update_grid, :815-820), and |x_i - x_j| < h evaluated as the FP32
// sqrt_rn(s) < h (s < the least float whose rounded square root is >= h).
#include <cmath>
#include <mutex>

#include "batch.h"
#include "device_common.h"

namespace nn {

constexpr long NA_MAX_PARTICLES = 1L << 20;
constexpr long NA_MAX_CELLS = 1L << 22;
constexpr int NA_WIDE = 131072;  // up to here 16 lanes per particle (Batch::lanes of the search)
constexpr long na_round(long w) { return (w + 63) / 64 * 64; }  // 256-byte sections
constexpr long NA_COUNTS = 0;                                                  // NA_MAX_CELLS + 1 ints
constexpr long NA_STARTS = NA_COUNTS + na_round(NA_MAX_CELLS + 1);             // NA_MAX_CELLS + 1 ints
constexpr long NA_SUMS = NA_STARTS + na_round(NA_MAX_CELLS + 1);               // scan partials
constexpr long NA_KEY = NA_SUMS + na_round((NA_MAX_CELLS + 1 + SCAN_TILE_ITEMS - 1) / SCAN_TILE_ITEMS);
constexpr long NA_BUCKET = NA_KEY + na_round(NA_MAX_PARTICLES);                // particles by cell, in arrival order
constexpr long NA_SORTED = NA_BUCKET + na_round(NA_MAX_PARTICLES);             // float4 (x, index) in cell order
constexpr long NA_WORDS = NA_SORTED + 4 * na_round(NA_MAX_PARTICLES);          // 14.7M ints = 59 MB

// The scratch of nn_neighbors_noalloc.  Host code never names it directly:
// scratch_base() returns the device's address from hipGetSymbolAddress.
static __device__ __align__(256) int scratch[NA_WORDS];

__global__ void k_na_zero(int* p, long n, int* status) {
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = 0;
  if (status && i == 0) *status = 0;
}

// cell_of of the context's search on caller-layout positions
__device__ __forceinline__ int na_key(const float* x, int i, float h, int g0, int g1, int g2) {
  const float fx = x[3 * (long)i] / h, fy = x[3 * (long)i + 1] / h, fz = x[3 * (long)i + 2] / h;
  if (!(fabsf(fx) < 1.0e9f && fabsf(fy) < 1.0e9f && fabsf(fz) < 1.0e9f)) return -1;
  const int cx = (int)fx, cy = (int)fy, cz = (int)fz;
  if (cx < 0 || cx >= g0 || cy < 0 || cy >= g1 || cz < 0 || cz >= g2) return -1;
  return (cx * g1 + cy) * g2 + cz;
}

// Cell key and arrival rank in the cell (kept in the sorted section, which is
// written only after the ranks were read).  A particle outside the grid is in
// no cell: its list is empty.
__global__ void k_na_count(const float* x, int n, float h, int g0, int g1, int g2, int* key, int* counts, int* arrival,
                           int* nbr, int* count, int cap, int* status) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const int k = na_key(x, i, h, g0, g1, g2);
  key[i] = k;
  if (k >= 0) {
    arrival[i] = atomicAdd(&counts[k], 1);
    return;
  }
  atomicOr(status, ST_OUT_OF_GRID);
  for (int m = 0; m < cap; m++) nbr[(long)i * cap + m] = -1;
  count[i] = 0;
}

// every particle into its cell's range, in arrival order
__global__ void k_na_bucket(const int* key, int n, const int* starts, const int* arrival, int* bucket) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const int k = key[i];
  if (k >= 0) bucket[starts[k] + arrival[i]] = i;
}

// Position and index into cell order: a particle's place in its cell is the
// number of lower indices there (a cell with more than MAX_PIC particles is
// reported and left in arrival order).  One thread per cell sorting its range
// by insertion took 27 us for 200,000 particles, a serial chain through memory
// per cell, and left the lists to gather each position through its index; this
// and the arrival order take 6.7 + 3.7 us (7.5 with one member read at a time).
__global__ void k_na_place(const float* x, const int* starts, int ncells, const int* key, const int* bucket,
                           float4* sorted, int* status) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= starts[ncells]) return;
  const int i = bucket[t];
  const int k = key[i];
  const int b = starts[k], e = starts[k + 1];
  int dest = t;
  if (e - b > MAX_PIC) {
    atomicOr(status, ST_CELL_OVERFLOW);
  } else {
    dest = b + lower_ids(bucket, b, e, i);
  }
  sorted[dest] = make_float4(x[3 * (long)i], x[3 * (long)i + 1], x[3 * (long)i + 2], __int_as_float(i));
}

// store_neighbors (:836-847) for the particle in place t of the cell order: the
// 9 runs of (cx+dx, cy+dy, cz-1..cz+1) cells, -1 padding up to cap.  G lanes
// per particle share the runs as in the context's search (k_build_lists).  With
// one thread per particle in caller order each candidate was a dependent index
// load and a gather of 3 floats: 198 us for 200,000 particles, now 59, of
// which writing the 48 MB of rows is 11.
template <int G, int B>
__global__ void k_na_lists(float thr2, int g0, int g1, int g2, const int* key, const int* starts,
                           const float4* sorted, int* nbr, int* count, int cap, int* status) {
  const long tid = (long)blockIdx.x * blockDim.x + threadIdx.x;
  const int t = (int)(tid / G), q = (int)(tid % G);
  if (t >= starts[g0 * g1 * g2]) return;
  const float4 xi = sorted[t];
  const int i = __float_as_int(xi.w);
  int* row = nbr + (long)i * cap;
  const int k = key[i];
  const int cz = k % g2, cy = (k / g2) % g1, cx = k / (g1 * g2);
  const int z0 = cz > 0 ? cz - 1 : 0;
  const int z1 = cz + 1 < g2 ? cz + 1 : g2 - 1;
  constexpr int RL = (9 + G - 1) / G;  // runs whose bounds a lane loads
  int lo[RL], len[RL];
#pragma unroll
  for (int e = 0; e < RL; e++) {
    const int r = q + e * G;
    const int a = cx + r / 3 - 1, b = cy + r % 3 - 1;
    lo[e] = len[e] = 0;
    if (r < 9 && a >= 0 && a < g0 && b >= 0 && b < g1) {
      const int base = (a * g1 + b) * g2;
      lo[e] = starts[base + z0];
      len[e] = starts[base + z1 + 1] - lo[e];
    }
  }
  int first[9], shift[9], total = 0;
  run_table<G, 0>(lo, len, 0, first, shift, total);
  const int lane = threadIdx.x & 63;
  const int below = (1 << q) - 1;
  int cnt = 0;
  for (int c0 = 0; c0 < total; c0 += G * B) {
    int p[B];
    float4 xj[B];
#pragma unroll
    for (int u = 0; u < B; u++) {
      const int c = c0 + u * G + q;
      int sh = shift[0];
#pragma unroll
      for (int r = 1; r < 9; r++) sh = c >= first[r] ? shift[r] : sh;
      p[u] = c < total ? c + sh : t;
    }
#pragma unroll
    for (int u = 0; u < B; u++) xj[u] = sorted[p[u]];
#pragma unroll
    for (int u = 0; u < B; u++) {
      const float ex = xi.x - xj[u].x, ey = xi.y - xj[u].y, ez = xi.z - xj[u].z;
      const float ss = ex * ex + ey * ey + ez * ez;
      const bool hit = ss < thr2 && p[u] != t;
      const int hits = (int)(__ballot(hit) >> (lane & ~(G - 1))) & ((1 << G) - 1);
      const int at = cnt + __popc(hits & below);
      cnt += __popc(hits);
      if (hit && at < MAX_NB) row[at] = __float_as_int(xj[u].w);
    }
  }
  if (cnt > MAX_NB) {
    if (q == 0) atomicOr(status, ST_NEIGHBOR_OVERFLOW);
    cnt = MAX_NB;
  }
  for (int m = cnt + q; m < cap; m += G) row[m] = -1;
  if (q == 0) count[i] = cnt;
}

// Address of this device's scratch, looked up once per device with the device
// current (each GPU holds its own copy of the array).
constexpr int NA_MAX_DEVICES = 64;
static std::mutex na_mu;
static int* na_base[NA_MAX_DEVICES] = {};

static int scratch_base(int** out) {
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return hip_fail(e, "hipGetDevice");
  if (dev < 0 || dev >= NA_MAX_DEVICES) {
    set_error("nn_neighbors_noalloc: device index beyond 63");
    return NN_E_UNSUPPORTED;
  }
  std::lock_guard<std::mutex> lk(na_mu);
  if (!na_base[dev]) {
    void* p = nullptr;
    e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !p) return hip_fail(e != hipSuccess ? e : hipErrorInvalidSymbol, "hipGetSymbolAddress");
    na_base[dev] = static_cast<int*>(p);
  }
  *out = na_base[dev];
  return NN_OK;
}

}  // namespace nn

extern "C" int32_t nn_neighbors_noalloc(const nn_params* params, const float* x, int64_t n, int32_t* nbr,
                                        int32_t* count, int32_t cap, int32_t* status, void* stream) {
  using namespace nn;
  if (!params || !status || n < 0 || (n > 0 && (!x || !nbr || !count))) {
    set_error("nn_neighbors_noalloc: bad arguments");
    return NN_E_ARG;
  }
  if (cap < MAX_NB) {
    set_error("nn_neighbors_noalloc: cap must be at least 60");
    return NN_E_ARG;
  }
  if (n > NA_MAX_PARTICLES) {
    set_error("nn_neighbors_noalloc: more than 1048576 particles (the fixed scratch's maximum)");
    return NN_E_ARG;
  }
  if (!(params->particle_radius > 0.0)) {
    set_error("nn_neighbors_noalloc: particle_radius must be positive");
    return NN_E_ARG;
  }
  const double h = 4.0 * params->particle_radius;  // Parameter.support_radius, :606
  long g[3];
  long cells = 1;
  for (int k = 0; k < 3; k++) {
    const double gk = std::ceil((params->domain_end[k] - params->domain_start[k]) / h);  // :773-775
    if (!(gk >= 1.0) || gk > (double)NA_MAX_CELLS) {
      set_error("nn_neighbors_noalloc: the domain must span 1 .. 4194304 cells per axis");
      return NN_E_ARG;
    }
    g[k] = (long)gk;
    cells *= g[k];
    if (cells > NA_MAX_CELLS) {
      set_error("nn_neighbors_noalloc: more than 4194304 grid cells (the fixed scratch's maximum)");
      return NN_E_ARG;
    }
  }
  int* base = nullptr;
  int rc = scratch_base(&base);
  if (rc < 0) return rc;
  hipStream_t st = static_cast<hipStream_t>(stream);
  const float hf = (float)h;
  const float thr2 = neighbor_threshold(hf);
  int* counts = base + NA_COUNTS;
  int* starts = base + NA_STARTS;
  int* sums = base + NA_SUMS;
  int* key = base + NA_KEY;
  int* bucket = base + NA_BUCKET;
  float4* sorted = reinterpret_cast<float4*>(base + NA_SORTED);
  int* arrival = base + NA_SORTED;
  const int nc = (int)cells;
  const int ni = (int)n;
  const int T = 256;
  // the scratch keeps the last call's contents: counts (and the status) start at zero
  hipLaunchKernelGGL(k_na_zero, dim3((unsigned)((nc + 1 + T - 1) / T)), dim3(T), 0, st, counts, (long)nc + 1, status);
  if (ni > 0) {
    hipLaunchKernelGGL(k_na_count, dim3((ni + T - 1) / T), dim3(T), 0, st, x, ni, hf, (int)g[0], (int)g[1], (int)g[2],
                       key, counts, arrival, nbr, count, cap, status);
  }
  launch_scan_i32(counts, nc + 1, sums, starts, st);
  if (ni > 0) {
    const dim3 per_particle((ni + T - 1) / T);
    hipLaunchKernelGGL(k_na_bucket, per_particle, dim3(T), 0, st, key, ni, starts, arrival, bucket);
    hipLaunchKernelGGL(k_na_place, per_particle, dim3(T), 0, st, x, starts, nc, key, bucket, sorted, status);
    const auto lists = [&](auto kern, int lanes) {
      hipLaunchKernelGGL(kern, dim3((unsigned)(((long)ni * lanes + T - 1) / T)), dim3(T), 0, st, thr2, (int)g[0],
                         (int)g[1], (int)g[2], key, starts, sorted, nbr, count, cap, status);
    };
    if (ni <= NA_WIDE) lists(k_na_lists<16, 4>, 16);
    else lists(k_na_lists<4, 4>, 4);
  }
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return hip_fail(e, "nn_neighbors_noalloc launch");
  return NN_OK;
}
