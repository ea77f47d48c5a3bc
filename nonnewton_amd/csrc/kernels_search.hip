// kernels_search.hip -- neighbor search as a counting sort into cell order plus
// compact neighbor lists (replaces NeighborhoodSearchSparse.run_search,
// SPH/main.py:815-847).
//
// Pipeline per step:
//   cell_count  : cell key of every particle, per-cell arrival counter (atomic)
//   scan        : exclusive prefix sum of the cell counts (block sums, then block
//                 scans with wavefront shuffles over the sums before theirs)
//   bucket      : every particle into its cell's range of a bucket array
//   place       : final slot = cell start + number of cell-mates with a smaller
//                 original index; state is moved into the new order
//   build_lists : for every particle the 9 contiguous runs of (cx+dx, cy+dy,
//                 cz-1..cz+1) cells are scanned with the reference's FP32
//                 distance test, which yields the reference's serial list order
//                 (SPH/main.py:840-847: dx slowest, dz fastest, then slot order =
//                 original index order, :815-820)
#include "device_common.h"

namespace nn {

__global__ void k_fill_i32(int* p, long n, int v) {
  long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = v;
}

__global__ void k_fill_f4(float4* p, long n, float4 v) {
  long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = v;
}

void launch_fill_i32(int* p, long n, int v, hipStream_t st) {
  if (n <= 0) return;
  NN_LAUNCH(k_fill_i32, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, p, n, v);
}

void launch_fill_f4(float4* p, long n, float4 v, hipStream_t st) {
  if (n <= 0) return;
  NN_LAUNCH(k_fill_f4, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, p, n, v);
}

// Fields of float[n][3] in original order (inv: slot of an id); `ordered` is pinned
// host memory.  (Reordered by the host, particle by particle over two arrays
// copied each way, an upload of 168,218 particles took 402 us and a download 360.)
__global__ void k_gather3(const float4* slots, const int* inv, int n, float* ordered) {
  const int id = blockIdx.x * blockDim.x + threadIdx.x;
  if (id >= n) return;
  const float4 v = slots[inv[id]];
  ordered[3 * (long)id] = v.x;
  ordered[3 * (long)id + 1] = v.y;
  ordered[3 * (long)id + 2] = v.z;
}
__global__ void k_scatter3(const float* ordered, const int* inv, int n, float4* slots) {
  const int id = blockIdx.x * blockDim.x + threadIdx.x;
  if (id >= n) return;
  float4* p = slots + inv[id];
  p->x = ordered[3 * (long)id];
  p->y = ordered[3 * (long)id + 1];
  p->z = ordered[3 * (long)id + 2];
}
__global__ void k_expand(Dev d, int pb, int n, float V0, const float* x, const int* kind, const float* v) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const int kd = min(kind[i], (int)KIND_RIGID);  // a rigid particle's kind holds its body
  const float* xi = x + 3 * (long)i;
  d.pos[pb + i] = make_float4(xi[0], xi[1], xi[2], kd == KIND_FLUID ? V0 : -V0);  // :607, :741
  float4 vi = make_float4(0.f, 0.f, 0.f, 0.f);
  if (v) vi = make_float4(v[3 * (long)i], v[3 * (long)i + 1], v[3 * (long)i + 2], 0.f);
  d.vel[pb + i] = vi;
  d.vdiff[pb + i] = make_float4(0.f, 0.f, 0.f, 0.f);
  d.info[pb + i] = (kd << 28) | i;
  d.inv[pb + i] = i;
}
void launch_expand(const DevRef& d, int pb, int n, float V0, const float* x, const int* kind, const float* v, hipStream_t st) {
  if (n > 0) NN_LAUNCH(k_expand, dim3((n + 255) / 256), dim3(256), 0, st, d.h, pb, n, V0, x, kind, v);
}
void launch_gather3(const float4* slots, const int* inv, int n, float* ordered, hipStream_t st) {
  if (n > 0) NN_LAUNCH(k_gather3, dim3((n + 255) / 256), dim3(256), 0, st, slots, inv, n, ordered);
}
void launch_scatter3(const float* ordered, const int* inv, int n, float4* slots, hipStream_t st) {
  if (n > 0) NN_LAUNCH(k_scatter3, dim3((n + 255) / 256), dim3(256), 0, st, ordered, inv, n, slots);
}

// ---------------------------------------------------------------------------
// exclusive scan over n ints: 256 threads x 8 items per block
// ---------------------------------------------------------------------------
constexpr int SCAN_T = 256;
constexpr int SCAN_I = 8;
constexpr int SCAN_TILE = SCAN_T * SCAN_I;

__device__ __forceinline__ int wave_incl_scan(int v) {
  const int lane = threadIdx.x & 63;
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    int t = __shfl_up(v, off, 64);
    if (lane >= off) v += t;
  }
  return v;
}

__device__ __forceinline__ int block_excl_scan(int v, int* lds, int& total) {
  const int wid = threadIdx.x >> 6, lane = threadIdx.x & 63;
  int incl = wave_incl_scan(v);
  if (lane == 63) lds[wid] = incl;
  __syncthreads();
  int off = 0;
  total = 0;
#pragma unroll
  for (int w = 0; w < SCAN_T / 64; w++) {
    int t = lds[w];
    if (w < wid) off += t;
    total += t;
  }
  __syncthreads();
  return off + incl - v;
}

// a thread's SCAN_I items from `base` on (16-byte loads where they may be);
// nz: 1 for an item that is not zero
__device__ __forceinline__ void scan_items(const int* in, int n, long base, int nz, int* v) {
  if (base + SCAN_I <= n && ((uintptr_t)in & 15) == 0) {
    const int4* q = reinterpret_cast<const int4*>(in + base);
#pragma unroll
    for (int k = 0; k < SCAN_I / 4; k++) {
      const int4 t = q[k];
      v[4 * k] = t.x;
      v[4 * k + 1] = t.y;
      v[4 * k + 2] = t.z;
      v[4 * k + 3] = t.w;
    }
  } else {
#pragma unroll
    for (int k = 0; k < SCAN_I; k++) v[k] = base + k < n ? in[base + k] : 0;
  }
#pragma unroll
  for (int k = 0; k < SCAN_I; k++) v[k] = nz ? v[k] != 0 : v[k];
}

__global__ __launch_bounds__(SCAN_T) void k_scan_reduce(const int* in, int n, int nz, int* sums) {
  __shared__ int lds[SCAN_T / 64];
  int v[SCAN_I], s = 0;
  scan_items(in, n, (long)blockIdx.x * SCAN_TILE + threadIdx.x * SCAN_I, nz, v);
#pragma unroll
  for (int k = 0; k < SCAN_I; k++) s += v[k];
  int total;
  block_excl_scan(s, lds, total);
  if (threadIdx.x == 0) sums[blockIdx.x] = total;
}

// scanned: sums holds the blocks' offsets; else each block adds the sums of
// those before it (one block scanning them first was a launch of 3 us)
__global__ __launch_bounds__(SCAN_T) void k_scan_down(const int* in, int n, int nz, const int* sums, int scanned, int total_out,
                                                      int* out) {
  __shared__ int lds[SCAN_T / 64];
  const long base = (long)blockIdx.x * SCAN_TILE + threadIdx.x * SCAN_I;
  int v[SCAN_I], s = 0;
  scan_items(in, n, base, nz, v);
#pragma unroll
  for (int k = 0; k < SCAN_I; k++) s += v[k];
  int total, offset;
  if (scanned) {
    offset = sums[blockIdx.x];
  } else {
    int before = 0;
    for (int k = threadIdx.x; k < (int)blockIdx.x; k += SCAN_T) before += sums[k];
    block_excl_scan(before, lds, offset);
  }
  int ex = block_excl_scan(s, lds, total) + offset;
#pragma unroll
  for (int k = 0; k < SCAN_I; k++) {
    if (base + k < n) out[base + k] = ex;
    ex += v[k];
  }
  if (total_out && blockIdx.x == gridDim.x - 1 && threadIdx.x == SCAN_T - 1) out[n] = ex;
}

// Exclusive scan of in[0..n) -- with nz of (in[i] != 0) -- into out[0..n), which
// may be in; with total also out[n].  scan_tmp_ints(n) ints of tmp.  Up to
// SCAN_DIRECT blocks add the sums before theirs, 32 loads a thread on average;
// beyond that the sums are scanned by this first.
constexpr int SCAN_DIRECT = 16384;
long scan_tmp_ints(long n) {
  const long nb = (n + SCAN_TILE - 1) / SCAN_TILE;
  return (nb + 63) / 64 * 64 + (nb > SCAN_DIRECT ? scan_tmp_ints(nb) : 0);
}
void launch_scan_i32(const int* in, int n, int* tmp, int* out, hipStream_t st, int nz, int total) {
  const int nb = (n + SCAN_TILE - 1) / SCAN_TILE;
  const int scanned = nb > SCAN_DIRECT;
  NN_LAUNCH(k_scan_reduce, dim3(nb), dim3(SCAN_T), 0, st, in, n, nz, tmp);
  if (scanned) launch_scan_i32(tmp, nb, tmp + (nb + 63) / 64 * 64, tmp, st, 0, 0);
  NN_LAUNCH(k_scan_down, dim3(nb), dim3(SCAN_T), 0, st, in, n, nz, tmp, scanned, total, out);
}

void launch_scan(const DevRef& d, int n, hipStream_t st) {
  launch_scan_i32(d.h.cell_count, n, d.h.scan_tmp, d.h.cell_start, st);
}

// ---------------------------------------------------------------------------
// counting sort into cell order
// ---------------------------------------------------------------------------
// pos_to_index, SPH/main.py:805-807: truncation of x / h, no domain offset.
__device__ __forceinline__ bool cell_of(const SceneDev& sc, float4 p, int& cx, int& cy, int& cz) {
  float fx = p.x / sc.h, fy = p.y / sc.h, fz = p.z / sc.h;
  if (!(fabsf(fx) < 1.0e9f && fabsf(fy) < 1.0e9f && fabsf(fz) < 1.0e9f)) return false;
  cx = (int)fx;
  cy = (int)fy;
  cz = (int)fz;
  return cx >= 0 && cx < sc.gn0 && cy >= 0 && cy < sc.gn1 && cz >= 0 && cz < sc.gn2;
}

// Cell key and a unique rank among the cell's particles.  Particles arrive in
// the previous step's cell order, so equal keys sit in runs of adjacent lanes:
// the first lane of each run adds the run length with one atomic and the run's
// lanes take consecutive ranks from it.  (Ranks only need to be unique; the
// final order inside a cell is fixed by k_place.)
__global__ void k_cell_count(Dev d) {
  int i, s;
  if (!slot_scene(d, i, s)) return;  // uniform over the wavefront
  const SceneDev& sc = d.scenes[s];
  const bool valid = i < sc.p_begin + sc.n;
  int key = -1;
  if (valid) {
    int cx, cy, cz;
    if (cell_of(sc, d.pos[i], cx, cy, cz)) {
      key = sc.cell_begin + (cx * sc.gn1 + cy) * sc.gn2 + cz;
    } else {
      // out of grid: parked in the scene's extra cell, reported, never searched
      key = sc.cell_begin + sc.gn0 * sc.gn1 * sc.gn2;
      atomicOr(&d.state[s].status, ST_OUT_OF_GRID);
    }
  }
  const int lane = threadIdx.x & 63;
  const int prev = __shfl_up(key, 1, 64);
  const bool start = lane == 0 || prev != key;
  const unsigned long long starts = __ballot(start);
  const unsigned long long upto = (2ull << lane) - 1ull;  // lanes 0..lane (all 64 for lane 63)
  const int leader = 63 - __clzll(starts & upto);
  const unsigned long long after = starts & ~upto;
  const int next = after ? __ffsll(after) - 1 : 64;
  int base = 0;
  if (start && key >= 0) base = atomicAdd(&d.cell_count[key], next - lane);
  base = __shfl(base, leader, 64);
  if (!valid) return;
  const int r = base + (lane - leader);
  if (r >= MAX_PIC) atomicOr(&d.state[s].status, ST_CELL_OVERFLOW);
  d.key[i] = key;
  d.rank[i] = r;
}

__global__ void k_bucket(Dev d) {
  int i, s;
  if (!slot_scene(d, i, s)) return;
  const SceneDev& sc = d.scenes[s];
  if (i >= sc.p_begin + sc.n) return;
  d.bucket[d.cell_start[d.key[i]] + d.rank[i]] = id_of(d.info[i]);
}

// Particles to their places: in its cell, a particle's place is the number of
// lower ids there.  clear_acc: the accelerations of a step start here
// (clear_accelerations_kernel, :945-951; a launch of its own took 3.5 to 5 us).
// Bound by the chain of its loads: key, cell, members, then the stores.  What it
// moves is requested before all of them and the members eight at a time: 6.1 us
// for 138,304 slots, 4.4 for 27,000; with one member at a time, and each load
// of what it moves behind the store before it, 9.9 and 5.7.
__global__ void k_place(Dev d, int clear_acc) {
  int i, s;
  if (!slot_scene(d, i, s)) return;
  const SceneDev& sc = d.scenes[s];
  if (i >= sc.p_begin + sc.n) return;
  const int key = d.key[i];
  const int inf = d.info[i];
  const float4 p = d.pos[i], v = d.vel[i];
  const bool warm = (sc.flags & SF_WARM_CG) != 0;
  const float4 e = warm ? d.vdiff[i] : p;
  const float4 g = kind_of(inf) == KIND_STATIC ? make_float4(0.f, 0.f, 0.f, 0.f) : make_float4(sc.gx, sc.gy, sc.gz, 0.f);
  const int my = id_of(inf), pb = sc.p_begin;
  const int cs = d.cell_start[key], ce = d.cell_start[key + 1];
  const int dest = sc.shift + cs + lower_ids(d.bucket, cs, ce, my);
  d.pos_alt[dest] = p;
  d.vel_alt[dest] = v;
  d.info_alt[dest] = inf;
  if (warm) d.vdiff_alt[dest] = e;
  if (clear_acc) d.acc[dest] = g;
  d.inv[pb + my] = dest - pb;
}

// store_neighbors, SPH/main.py:836-847, over the sorted particles.  With
// all == 0 (the search inside a step) static boundary particles get no list:
// after the boundary volumes of the first search no sweep reads one.
//
// G lanes per particle.  The bounds of the 9 runs are loaded by the group at
// once and the runs laid end to end: candidate c of the sequence is slot
// c + shift[r] of the run r that holds it.  The lanes test candidates q, q + G,
// ..., B rounds of loads in flight, and a hit's list position is the hits
// before it: those of earlier rounds plus those of lower lanes (a ballot), so
// the list keeps the reference's order.
template <int G, int B>
__global__ void k_build_lists(Dev d, int all) {
  int i, q, s;
  if (!lane_slot_scene<G>(d, i, q, s)) return;
  const SceneDev& sc = d.scenes[s];
  const bool mine = i < sc.p_begin + sc.n;
  const int kind = mine ? kind_of(d.info[i]) : KIND_STATIC;
  int cnt = 0;
  int cx, cy, cz;
  const float4 xi = d.pos[i];
  if (mine && (all || kind != KIND_STATIC) && cell_of(sc, xi, cx, cy, cz)) {
    const float thr2 = sc.thr2;
    const long P = d.P;
    const int z0 = cz > 0 ? cz - 1 : 0;
    const int z1 = cz + 1 < sc.gn2 ? cz + 1 : sc.gn2 - 1;
    constexpr int RL = (9 + G - 1) / G;  // runs whose bounds a lane loads
    int lo[RL], len[RL];
#pragma unroll
    for (int e = 0; e < RL; e++) {
      const int r = q + e * G;
      const int a = cx + r / 3 - 1, b = cy + r % 3 - 1;
      lo[e] = len[e] = 0;
      if (r < 9 && a >= 0 && a < sc.gn0 && b >= 0 && b < sc.gn1) {
        const int base = sc.cell_begin + (a * sc.gn1 + b) * sc.gn2;
        lo[e] = d.cell_start[base + z0];
        len[e] = d.cell_start[base + z1 + 1] - lo[e];
      }
    }
    int first[9], shift[9], total = 0;  // run r: candidates [first[r], first[r + 1])
    run_table<G, 0>(lo, len, sc.shift, first, shift, total);
    const int lane = threadIdx.x & 63;
    const int below = (1 << q) - 1;
    for (int c0 = 0; c0 < total; c0 += G * B) {
      int j[B];
      float4 xj[B];
#pragma unroll
      for (int u = 0; u < B; u++) {
        const int c = c0 + u * G + q;
        int sh = shift[0];
#pragma unroll
        for (int r = 1; r < 9; r++) sh = c >= first[r] ? shift[r] : sh;
        j[u] = c < total ? c + sh : i;
      }
#pragma unroll
      for (int u = 0; u < B; u++) xj[u] = d.pos[j[u]];
#pragma unroll
      for (int u = 0; u < B; u++) {
        const float ex = xi.x - xj[u].x, ey = xi.y - xj[u].y, ez = xi.z - xj[u].z;
        const float ss = ex * ex + ey * ey + ez * ez;
        // sqrt_rn(ss) < h  <=>  ss < thr2 (thr2: least float whose rounded sqrt >= h)
        const bool hit = ss < thr2 && j[u] != i;
        const int hits = (int)(__ballot(hit) >> (lane & ~(G - 1))) & ((1 << G) - 1);
        const int at = cnt + __popc(hits & below);
        cnt += __popc(hits);
        if (hit && at < MAX_NB) d.nbr[nb_word(P, i, at)] = j[u];
      }
    }
    if (cnt > MAX_NB) {
      if (q == 0) atomicOr(&d.state[s].status, ST_NEIGHBOR_OVERFLOW);
      cnt = MAX_NB;
    }
  }
  if (mine && q == 0) d.nnbr[i] = cnt;
  // the step's pair counts cover the lists a step uses: fluid and dynamic
  // solid particles (static boundary lists serve only the boundary volumes);
  // a wavefront's counts go to its own entry (k_publish adds them: thousands of
  // atomics on one word took longer than the search)
  int tot = q == 0 && kind != KIND_STATIC ? cnt : 0, cf = q == 0 && kind == KIND_FLUID ? cnt : 0;
#pragma unroll
  for (int off = 32; off >= G; off >>= 1) {
    tot += __shfl_xor(tot, off, 64);
    cf += __shfl_xor(cf, off, 64);
  }
  if ((threadIdx.x & 63) == 0) d.wave_pairs[i / (64 / G)] = make_int2(tot, cf);
}

// compute_static/moving_boundary_volume, SPH/main.py:1010-1035:
// V_b = 3 / (W0 + sum over solid neighbors of W); stored as -V (solid sign).
template <int G, int B>
__global__ void k_bvol(Dev d, int dynamic) {
  int i, q, s;
  if (!lane_slot_scene<G>(d, i, q, s)) return;
  const SceneDev& sc = d.scenes[s];
  if (i >= sc.p_begin + sc.n) return;
  const int kind = kind_of(d.info[i]);
  if (dynamic ? !dyn_solid(kind) : kind != KIND_STATIC) return;
  const KernH kh(sc);
  const float4 xi = d.pos[i];
  KSum ks{sc.W0, 0.0f};
  const bool comp = (sc.flags & SF_COMPENSATED) != 0;
  // (the volume of a neighbor may be rewritten meanwhile: only its sign, which
  // stays, is read)
  for_pairs<G, B, 2>(
      d, i, q, d.nnbr[i], [&](int j) { return d.pos[j]; },
      [&](int, const float4& xj, bool live, float (&t)[2]) {
        const bool on = live && xj.w < 0.0f;
        t[0] = pair_w(kh, sc, xi.x - xj.x, xi.y - xj.y, xi.z - xj.z, on);
        t[1] = on ? 1.0f : 0.0f;
      },
      [&](const float (&t)[2], bool) {
        KSum n = ks;
        if (comp) n.add(t[0]);
        else n.s += t[0];
        const bool on = t[1] != 0.0f;
        ks.s = on ? n.s : ks.s;
        ks.c = on ? n.c : ks.c;
      });
  if (q == 0) d.pos[i].w = -(1.0f / ks.s * 3.0f);
}

void launch_cell_count(const DevRef& d, int block, hipStream_t st) {
  NN_LAUNCH(k_cell_count, dim3((d.h.Pn + block - 1) / block), dim3(block), 0, st, d.h);
}
void launch_bucket(const DevRef& d, int block, hipStream_t st) {
  NN_LAUNCH(k_bucket, dim3((d.h.Pn + block - 1) / block), dim3(block), 0, st, d.h);
}
void launch_place(const DevRef& d, int block, int clear_acc, hipStream_t st) {
  NN_LAUNCH(k_place, dim3((d.h.Pn + block - 1) / block), dim3(block), 0, st, d.h, clear_acc);
}
void launch_build_lists(const DevRef& d, int block, int lanes, int all, hipStream_t st) {
  const dim3 g((unsigned)(((long)d.h.Pn * lanes + block - 1) / block)), b(block);
  if (lanes == 4) NN_LAUNCH((k_build_lists<4, 4>), g, b, 0, st, d.h, all);
  else NN_LAUNCH((k_build_lists<16, 4>), g, b, 0, st, d.h, all);
}
void launch_bvol(const DevRef& d, int block, int lanes, int dynamic, hipStream_t st) {
  SWEEP_LAUNCH_4(k_bvol, lanes, 8, d.h.Pn, block, st, d.h, dynamic);
}

}  // namespace nn
