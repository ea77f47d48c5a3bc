// batch.hip -- host driver of the SPH step: derived constants, device layout of
// one or many scenes, upload, initialization, the per-step launch sequence with
// device-side solver termination, and downloads in original particle order.
#include "batch.h"

#include <algorithm>
#include <atomic>
#include <chrono>
#include <cmath>
#include <cstring>

namespace nn {

static thread_local std::string g_err;
void set_error(const std::string& m) { g_err = m; }
const char* last_error_text() { return g_err.c_str(); }
int hip_fail(hipError_t e, const char* what) {
  set_error(std::string(what) + ": " + hipGetErrorString(e));
  return NN_E_HIP;
}

#define HIPCHK(expr)                                   \
  do {                                                 \
    hipError_t _e = (expr);                            \
    if (_e != hipSuccess) return hip_fail(_e, #expr); \
  } while (0)

#define CHK(expr)              \
  do {                         \
    int _rc = (expr);          \
    if (_rc < 0) return _rc;   \
  } while (0)

static inline int round_up64(int v) { return (v + 63) & ~63; }

// The neighbor lists of slots [pb, pb + n) into host memory (n * MAX_NB ints),
// in the device's grouped layout restricted to those slots: position m of
// slot pb + t is at host_nb(n, t, m).
static hipError_t copy_lists(int* host, const Dev& d, int pb, int n, hipStream_t st) {
  return hipMemcpy2DAsync(host, sizeof(int4) * n, d.nbr + 4L * pb, sizeof(int4) * d.P, sizeof(int4) * n, MAX_NB / 4,
                          hipMemcpyDeviceToHost, st);
}
static inline size_t host_nb(int n, int t, int m) { return 4 * ((size_t)(m >> 2) * n + t) + (m & 3); }
// After the copy has completed: list entries to scene-local slots, each
// checked to lie in [0, n).
static int lists_to_local(std::vector<int>& nb, const std::vector<int>& cnt, int pb, int n) {
  for (int t = 0; t < n; t++) {
    if (cnt[t] < 0 || cnt[t] > MAX_NB) {
      set_error("neighbor count out of range");
      return NN_E_STATE;
    }
    for (int m = 0; m < cnt[t]; m++) {
      int& j = nb[host_nb(n, t, m)];
      j -= pb;
      if (j < 0 || j >= n) {
        set_error("neighbor list entry outside its scene");
        return NN_E_STATE;
      }
    }
  }
  return NN_OK;
}

// cubic_kernel (SPH/main.py:859-880), host copy of the device function
static float host_kern_w(float h, float kW, float rn) {
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

float neighbor_threshold(float h) {
  float t = h * h;
  while (t > 0.0f && sqrtf(t) >= h) t = nextafterf(t, 0.0f);
  while (sqrtf(t) < h) t = nextafterf(t, INFINITY);
  return t;
}

int derive_scene(SceneHost& s, std::string& err) {
  const nn_params& p = s.params;
  if (!(p.particle_radius > 0.0) || !(p.dt > 0.0) || !(p.density0 > 0.0)) {
    err = "particle_radius, dt and density0 must be positive";
    return NN_E_ARG;
  }
  if (p.warm_start & ~1) {
    err = "warm_start: only bit 0 (Weiler CG initial guess) is supported";
    return NN_E_UNSUPPORTED;
  }
  if (p.non_newton_method < 0 || p.non_newton_method > 6) {
    err = "non_newton_method must be 0..6";
    return NN_E_ARG;
  }
  const double r = p.particle_radius, dd = 2.0 * r, h = 4.0 * r;
  long cells = 1;
  for (int k = 0; k < 3; k++) {
    const double g = std::ceil((p.domain_end[k] - p.domain_start[k]) / h);  // :773-775
    if (!(g >= 1.0) || g > 1.0e6) {
      err = "domain must span at least one cell per axis";
      return NN_E_ARG;
    }
    s.gn[k] = (int)g;
    cells *= s.gn[k];
  }
  if (cells > (1L << 30)) {
    err = "grid too large";
    return NN_E_ARG;
  }
  s.ncells = cells;
  SceneDev& c = s.dev;
  c.gn0 = s.gn[0];
  c.gn1 = s.gn[1];
  c.gn2 = s.gn[2];
  c.h = (float)h;
  c.thr2 = neighbor_threshold(c.h);
  c.kW = (float)(8.0 / M_PI / (h * h * h));
  c.kG = (float)(6.0 * 8.0 / M_PI / (h * h * h));
  c.W0 = host_kern_w(c.h, c.kW, 0.0f);
  c.dt = (float)p.dt;
  c.inv_dt = (float)(1.0 / (double)c.dt);
  c.inv_dt2 = (float)(1.0 / ((double)c.dt * (double)c.dt));
  c.rho0 = (float)p.density0;
  const double vol0 = 0.8 * dd * dd * dd;  // :607
  c.mass = (float)(p.particle_mass > 0.0 ? p.particle_mass : vol0 * 1000.0);  // :743
  c.nu = (float)p.viscosity;
  c.bnu = (float)p.boundary_viscosity;
  c.gx = (float)p.gravity[0];
  c.gy = (float)p.gravity[1];
  c.gz = (float)p.gravity[2];
  c.lo0 = (float)(p.domain_start[0] + h);
  c.lo1 = (float)(p.domain_start[1] + h);
  c.lo2 = (float)(p.domain_start[2] + h);
  c.hi0 = (float)(p.domain_end[0] - h);
  c.hi1 = (float)(p.domain_end[1] - h);
  c.hi2 = (float)(p.domain_end[2] - h);
  c.diam2 = (float)(dd * dd);
  const float dr = (float)dd;
  c.Wd = host_kern_w(c.h, c.kW, sqrtf(dr * dr + 0.0f * 0.0f + 0.0f * 0.0f));  // :1414
  c.visc_eps = (float)(0.01 * h * h);
  c.sigma = (float)p.surface_tension;
  c.opc = (float)(1.0 + p.collision_coeff);
  c.sticky = (float)p.sticky_coeff;
  c.eps = (float)p.eps;
  const double E = p.youngs_modulus, nu = p.poisson_ratio;
  const double factor = E / ((1.0 + nu) * (1.0 - 2.0 * nu));  // :1277-1281
  c.C_diag = (float)(factor * (1.0 - nu));
  c.C_off = (float)(factor * nu);
  c.C_shear = (float)(factor * 0.5 * (1.0 - 2.0 * nu));
  c.nn_method = p.non_newton_method;
  c.nn_n = (float)p.power_index;
  c.nn_K = (float)p.consistency_index;
  c.nn_e0 = (float)p.viscosity0;
  c.nn_einf = (float)p.viscosity_inf;
  c.nn_gc = (float)p.critical_strain_rate;
  c.nn_muc = (float)p.mu_c;
  c.nn_tauy = (float)p.yield_stress;
  c.nn_max = (float)p.max_viscosity;
  c.ten_nu = 10.0f * c.nu;
  c.ten_bnu = 10.0f * c.bnu;
  c.sig_m = c.sigma / c.mass * c.mass;
  c.eta_v = 1.0 / (double)c.dt * p.max_error_v * 0.01 * p.density0;  // :1699
  c.eta_p = p.max_error * 0.01 * p.density0;                          // :1781
  c.cg_tol2 = p.weiler_tol * p.weiler_tol;
  c.rho0_d = p.density0;
  c.max_iter_v = p.max_iterations_v;
  c.max_iter_p = p.max_iterations;
  c.max_iter_cg = p.weiler_max_iter;
  c.vol0 = (float)vol0;
  c.nbody = s.nbody;
  c.coupling = std::max(0, p.coupling_interval);
  int f = 0;
  if (p.use_surface_tension) f |= SF_SURFACE_TENSION;
  if (p.use_viscosity) f |= SF_VISCOSITY;
  if (p.use_non_newtonian) f |= SF_NON_NEWTONIAN;
  if (p.viscosity_method == 1) f |= SF_WEILER;
  else if (p.viscosity_method != 0) {
    err = "viscosity_method must be 0 (explicit) or 1 (Weiler)";
    return NN_E_ARG;
  }
  if (p.enable_divergence_solver) f |= SF_DIVERGENCE;
  if (p.warm_start & 1) f |= SF_WARM_CG;
  if (p.compensated) f |= SF_COMPENSATED;
  if (s.n_fluid > 0) f |= SF_HAS_FLUID;
  if (s.n_elastic > 0) f |= SF_HAS_ELASTIC;
  if (s.nbody > 0) f |= SF_HAS_RIGID;
  if (c.h >= 0x1p-20f && c.h <= 0x1p20f) f |= SF_MIDRANGE;
  c.flags = f;
  c.n = s.n;
  c.n_fluid = s.n_fluid;
  c.n_elastic = s.n_elastic;
  c.nf_d = (double)s.n_fluid;
  return NN_OK;
}

// Rest centres of mass of the rigid bodies (RigidBodySolver.__init__,
// :1100-1106) from the initial positions: FP64 sums of the FP32 terms m x in
// index order, rounded once.  Needs derive_scene (the mass) and the bodies of
// the kinds; runs before the scene is laid out.
void rigid_rest_centres(SceneHost& s, const float* x) {
  const float mass_r = s.dev.vol0 * s.dev.rho0;
  s.rest_cm.assign(3 * (size_t)s.nbody, 0.0f);
  for (int b = 0; b < s.nbody; b++) {
    double sm = 0.0, sx[3] = {0.0, 0.0, 0.0};
    for (int m = s.body_off[b]; m < s.body_off[b + 1]; m++) {
      const int id = s.body_ids[m];
      sm += (double)mass_r;
      for (int c = 0; c < 3; c++) sx[c] += (double)(mass_r * x[3 * id + c]);
    }
    for (int c = 0; c < 3; c++) s.rest_cm[3 * b + c] = (float)(sx[c] / sm);
  }
}

// bytes per particle slot: pos,pos_alt,vel,vel_alt,acc,wd0,x0,vdiff,vdiff_alt (9 float4),
// wx,wr,ww,wp,ws (5 float3), xu (2 float3), wd1 (float2), info,info_alt,key,rank,inv,bucket,nnbr,s_of (8 int),
// rho,mu,gam,eta (4 float), sa (float2), nbr and spair (60 int + 60 float), partials (16 doubles per 64
// slots), wave table
static constexpr long long BYTES_PER_SLOT = 9 * 16 + 7 * 12 + 8 + 8 * 4 + 6 * 4 + 2 * MAX_NB * 4 + 3;
static constexpr long long BYTES_PER_MEMBER = 4 + 4 + MAX_REST * 4 + 4 * 16 + 1;

long long scene_footprint(long long n, long long ns, long long cells) {
  const long long np = (n + 63) / 64 * 64, nsp = (ns + 63) / 64 * 64;
  return np * BYTES_PER_SLOT + nsp * BYTES_PER_MEMBER + (cells + 1) * 8 + 2048;
}

// Pinned memory through which the kernels read and write fields, larger ones in
// pieces.  Microseconds of an upload / a download by field size, this way and
// with a copy to or from device memory:
//             5 KB      134 KB    329 KB    886 KB    1.9 MB     3.4 MB      6.5 MB
//   kernels   11 / 11   15 / 17   21 / 27   41 / 51   68 / 93    111 / 157   196 / 291
//   copies    20 / 27   74 / 82   36 / 40   60 / 68   91 / 140   136 / 256   228 / 473
constexpr size_t STAGE_BYTES = 1 << 20;
static size_t state_bytes(int scenes) { return (sizeof(SceneState) + sizeof(unsigned long long)) * (size_t)scenes; }

Spares& Spares::get() {
  static Spares* s = new Spares();  // not destroyed: the runtime may be gone by then
  return *s;
}

size_t Spares::limit() const {
  int64_t most = 0;
  for (int64_t b : budgets_) most = std::max(most, b);
  return (size_t)std::max<long long>(0, std::min<long long>(most / 8, most - scenes_));
}

void Spares::evict(std::vector<Block>& dev, std::vector<Block>& host) {
  while (!dev_.empty() && held_ + excess_ > (long long)limit()) {
    held_ -= (long long)dev_.front().bytes;
    dev.push_back(dev_.front());
    dev_.erase(dev_.begin());
  }
  while (!host_.empty() && pinned_ > (budgets_.empty() ? 0 : 128 << 20)) {
    pinned_ -= (long long)host_.front().bytes;
    host.push_back(host_.front());
    host_.erase(host_.begin());
  }
}

void Spares::release(const std::vector<Block>& dev, const std::vector<Block>& host) {
  for (auto& b : dev) (void)hipFree(b.p);
  for (auto& b : host) (void)hipHostFree(b.p);
}

void Spares::pool_begins(int64_t budget) {
  std::lock_guard<std::mutex> lk(mu_);
  budgets_.push_back(budget);
}

void Spares::pool_ends(int64_t budget) {
  std::vector<Block> dev, host;
  {
    std::lock_guard<std::mutex> lk(mu_);
    budgets_.erase(std::find(budgets_.begin(), budgets_.end(), budget));
    evict(dev, host);
  }
  release(dev, host);
}

void Spares::scenes(long long bytes) {
  std::vector<Block> dev, host;
  {
    std::lock_guard<std::mutex> lk(mu_);
    scenes_ += bytes;
    evict(dev, host);
  }
  release(dev, host);
}

bool Spares::take(bool host, size_t bytes, void** p, size_t* got) {
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess) return false;
  std::lock_guard<std::mutex> lk(mu_);
  auto& v = host ? host_ : dev_;
  const size_t room = host ? 4096 : 1u << 20;  // a block may have twice the bytes asked for and twice this more
  size_t best = v.size();
  for (size_t k = 0; k < v.size(); k++)
    if (v[k].device == dev && v[k].bytes >= bytes && v[k].bytes / 2 <= bytes + room &&
        (best == v.size() || v[k].bytes < v[best].bytes))
      best = k;
  if (best == v.size()) return false;
  *p = v[best].p;
  *got = v[best].bytes;
  if (!host) {
    held_ -= (long long)*got;
    excess_ += (long long)(*got - bytes);
  } else {
    pinned_ -= (long long)*got;
  }
  v.erase(v.begin() + best);
  return true;
}

void Spares::give(bool host, void* p, size_t bytes, size_t need) {
  std::vector<Block> dev, pinned;
  hipPointerAttribute_t at{};
  int device = 0;
  if (hipPointerGetAttributes(&at, p) == hipSuccess) device = at.device;
  else (void)hipGetLastError();
  {
    std::lock_guard<std::mutex> lk(mu_);
    (host ? host_ : dev_).push_back({p, bytes, device});
    if (!host) {
      held_ += (long long)bytes;
      excess_ -= (long long)(bytes - need);
    } else {
      pinned_ += (long long)bytes;
    }
    evict(dev, pinned);
  }
  release(dev, pinned);
}

bool Spares::clear() {
  std::vector<Block> dev, host;
  {
    std::lock_guard<std::mutex> lk(mu_);
    dev.swap(dev_);
    host.swap(host_);
    held_ = pinned_ = 0;
  }
  release(dev, host);
  return !dev.empty() || !host.empty();
}

long long Spares::kept() {
  std::lock_guard<std::mutex> lk(mu_);
  return held_ + excess_;
}

Batch::Batch(hipStream_t st, bool keep) : stream(st), keep_(keep) {}

Batch::~Batch() {
  release();
  free_host(h_state_, h_state_bytes_);
  free_host(h_stage_, h_stage_bytes_);
}

int Batch::alloc_host(void** p, size_t bytes, size_t& got) {
  got = bytes;
  if (keep_ && Spares::get().take(true, bytes, p, &got)) return NN_OK;
  hipError_t e = hipHostMalloc(p, bytes, hipHostMallocDefault);
  if (e != hipSuccess && free_kept()) {
    (void)hipGetLastError();
    e = hipHostMalloc(p, bytes, hipHostMallocDefault);
  }
  return e == hipSuccess ? NN_OK : hip_fail(e, "hipHostMalloc");
}
void Batch::free_host(void* p, size_t got) {  // no work on it is pending
  if (!p) return;
  if (keep_) Spares::get().give(true, p, got, got);
  else (void)hipHostFree(p);
}
void Batch::free_arena(const Alloc& a) {  // no work on it is pending, or (not kept) hipFree waits for it
  if (keep_) Spares::get().give(false, a.p, a.bytes, a.need);
  else (void)hipFree(a.p);
}

// The arrays of a layout are carved from one device allocation (256-byte
// aligned sub-ranges): one hipMalloc and, when the batch is released or laid
// out again, one hipFree, which synchronizes the device.
int Batch::alloc_arena(std::vector<std::pair<void**, size_t>>& req) {
  size_t total = 0;
  for (auto& r : req) total += (r.second + 255) & ~(size_t)255;
  void* q = nullptr;
  size_t got = total;
  if (!(keep_ && Spares::get().take(false, total, &q, &got))) {
    hipError_t e = hipMalloc(&q, total);
    if (e == hipErrorOutOfMemory && free_kept()) {
      (void)hipGetLastError();
      e = hipMalloc(&q, total);
    }
    if (e != hipSuccess) {
      (void)hipGetLastError();
      set_error(std::string("hipMalloc failed: ") + hipGetErrorString(e));
      return NN_E_OOM;
    }
  }
  char* c = (char*)q;
  for (auto& r : req) {
    *r.first = c;
    c += (r.second + 255) & ~(size_t)255;
  }
  allocs_.push_back({q, got, total});
  bytes_ += (long long)got;
  return NN_OK;
}

// Blocks are given on only when no work on them is pending: the stream is asked,
// not waited for.  After waits that poll (await), hipStreamSynchronize leaves the
// runtime with the ends of all launches to take note of, and the calls that
// follow wait for that: a pool's life (made, one scene admitted, two ticks,
// closed) took 1.39 ms with it and takes 0.72 at 1,082 particles, 2.33 and 0.85
// at 22,530.  (A staging stream that other admissions keep busy is waited for
// after all.)
void Batch::release() {
  if (keep_ && !allocs_.empty()) {
    const auto start = std::chrono::steady_clock::now();
    hipError_t e;
    bool asked = false;
    for (; (e = hipStreamQuery(stream)) == hipErrorNotReady; asked = true) {
      if (std::chrono::steady_clock::now() - start > std::chrono::microseconds(300)) break;
      __builtin_ia32_pause();
    }
    if (asked) (void)hipGetLastError();  // hipErrorNotReady
    if (e == hipErrorNotReady) (void)hipStreamSynchronize(stream);
  }
  for (auto& a : allocs_) free_arena(a);
  allocs_.clear();
  bytes_ = 0;
}

DevRef Batch::dref() { return DevRef{d}; }

// Lanes per particle of a list sweep, by the slots in use.  A sweep is bound by
// its longest chain (a lane walking its list) until the device is full of
// wavefronts, and by instructions after that, where every lane of a group
// repeats the additions.  Microseconds a launch with 4 / 16 lanes (or 1 / 4), by
// slots (one scene; the last columns 8 and 64 mixed scenes in a pool):
//   4 / 16 lanes        11,970       19,170       28,514       36,066
//   build_lists         21 / 11      21 / 11      24 / 13      22 / 14
//   density_alpha       8.5 / 7.8    8.7 / 8.7    9.5 / 10.6   9.6 / 12.5
//   strain              11.4 / 9.5   10.8 / 11.1  12.2 / 12.3  11.6 / 14.0
//   nonpressure         10.3 / 6.9   10.6 / 7.7   12.1 / 9.4   12.1 / 10.0
//   press_source        7.3 / 6.4    6.9 / 5.9    7.4 / 5.5    7.7 / 6.1
//                       86,754       118,178      153,954      202,594
//   build_lists         31 / 26      34 / 34      42 / 44      55 / 56
//   press_source        9.6 / 9.8    12.0 / 12.8  14.1 / 16.4  18.6 / 20.6
//   1 / 4 lanes         86,754       118,178      202,594      572,130      1,288,930    248,122      1,616,737
//   density_alpha       16.7 / 15.3  18.0 / 19.3  24.0 / 28.2  58 / 67      124 / 142    24.7 / 26.6  90 / 124
//   strain              18.1 / 16.9  21.0 / 21.0  29.3 / 28.3  66 / 63      138 / 132    29.3 / 27.5  92 / 113
//   nonpressure, with velocities   (explicit or boundary viscosity)
//                       31 / 18      34 / 23      46 / 36      109 / 87     238 / 185
//   nonpressure, positions only    (surface tension beside the implicit solve)
//                       18.5 / 15.1  19.5 / 17.4  25.1 / 29.6  62 / 69      161 / 193    30.9 / 34.5  154 / 173
//                       members of the stress set, 4 / 16 lanes
//                       4,096        13,824       24,576       30,720       40,960
//   elastic_rot_stress  18.5 / 18.9  19.9 / 20.3  23 / 38      24 / 38      28 / 53
//   elastic_force       10.2 / 7.9   11.4 / 8.2   14.0 / 13.5  14.5 / 13.4  16.1 / 18.1
// The search's lanes share candidates and repeat nothing, so its limit is the
// highest; the sums of density and strain are the most, so theirs are the
// lowest, and one lane is left to them and to the position-only sweep.
int Batch::lanes(int id) const {
  const bool members = id == K_ELASTIC_ROT_STRESS || id == K_ELASTIC_FORCE;
  const int slots = members ? d.NSn : d.Pn;
  int wide = 32768, one = INT_MAX;  // 16 lanes up to, 1 lane above
  switch (id) {
    case K_BUILD_LISTS: wide = 131072; break;
    case K_DENSITY_ALPHA: wide = 16384; one = 98304; break;
    case K_STRAIN: wide = 16384; one = 1048576; break;
    case K_NONPRESSURE: one = any_velocity_terms_ ? INT_MAX : 196608; break;
    case K_ELASTIC_ROT_STRESS: wide = 16384; break;
  }
  return slots <= wide ? 16 : slots > one ? 1 : 4;
}

void Batch::swap_sort_buffers() {
  std::swap(d.pos, d.pos_alt);
  std::swap(d.vel, d.vel_alt);
  std::swap(d.info, d.info_alt);
  std::swap(d.vdiff, d.vdiff_alt);
}

// the non-pressure sweep forms viscosity terms of this scene (k_nonpressure)
static bool velocity_terms(const SceneDev& c) {
  return (c.flags & SF_HAS_FLUID) && (c.flags & SF_VISCOSITY) && (!(c.flags & SF_WEILER) || c.bnu != 0.0f);
}

// Per-scene fields that depend on the scenes' order and offsets (p_begin,
// cell_begin and s_begin must be set): the slot shift used by the sort, the
// wave range, and the batch-wide feature flags.
void Batch::derive_members() {
  long base = 0;
  any_fluid_ = any_elastic_ = any_weiler_ = any_strain_ = any_div_ = any_warm_cg_ = any_rigid_ = false;
  any_velocity_terms_ = false;
  max_body_ = max_coupling_ = max_body_waves_ = 0;
  max_iter_[0] = max_iter_[1] = max_iter_[2] = 1;
  for (auto& sp : scenes) {
    SceneHost& s = *sp;
    s.dev.p_begin = s.p_begin;
    s.dev.shift = (int)(s.p_begin - base);  // particles of the scenes before this one, in cell order
    s.dev.wave_begin = s.p_begin / 64;
    s.dev.wave_end = (s.p_begin + round_up64(s.n)) / 64;
    s.dev.cell_begin = s.cell_begin;
    s.dev.s_begin = s.s_begin;
    s.dev.ns = s.ns;
    s.dev.body_begin = s.body_begin;
    base += s.n;
    const int f = s.dev.flags;
    any_velocity_terms_ |= velocity_terms(s.dev);
    if (f & SF_HAS_FLUID) {
      any_fluid_ = true;
      if (f & SF_DIVERGENCE) any_div_ = true;
      if ((f & SF_VISCOSITY) && (f & SF_WEILER)) any_weiler_ = true;
      if ((f & SF_VISCOSITY) && (f & SF_WEILER) && (f & SF_WARM_CG)) any_warm_cg_ = true;
      if ((f & SF_NON_NEWTONIAN) || ((f & SF_VISCOSITY) && (f & SF_WEILER))) any_strain_ = true;
    }
    if (f & SF_HAS_ELASTIC) any_elastic_ = true;
    if (f & SF_HAS_RIGID) {
      any_rigid_ = true;
      max_body_ = std::max(max_body_, s.dev.nbody);
      max_coupling_ = std::max(max_coupling_, s.dev.coupling);
      for (size_t b = 0; b + 1 < s.body_off.size(); b++)
        max_body_waves_ = std::max(max_body_waves_, round_up64(s.body_off[b + 1] - s.body_off[b]) / 64);
    }
    max_iter_[0] = std::max(max_iter_[0], s.dev.max_iter_v);
    max_iter_[1] = std::max(max_iter_[1], s.dev.max_iter_p);
    max_iter_[2] = std::max(max_iter_[2], s.dev.max_iter_cg);
  }
}

// Scene table and the wave -> scene maps of `nd` for the current scenes
// (waves of no scene map to -1).
int Batch::upload_tables(const Dev& nd) {
  std::vector<int> hw(std::max(nd.W, 1), -1), hsw(std::max(nd.SW, 1), -1);
  std::vector<SceneDev> hs(scenes.size());
  std::vector<int2> cgb;
  for (size_t k = 0; k < scenes.size(); k++) {
    SceneHost& s = *scenes[k];
    for (int w = s.dev.wave_begin; w < s.dev.wave_end; w++) hw[w] = (int)k;
    for (int w = s.s_begin / 64; w < (s.s_begin + round_up64(s.ns)) / 64; w++) hsw[w] = (int)k;
    hs[k] = s.dev;
    const int f = s.dev.flags;
    if ((f & SF_HAS_FLUID) && (f & SF_VISCOSITY) && (f & SF_WEILER))  // CG update workgroups
      for (int w = s.dev.wave_begin; w < s.dev.wave_end; w += CG_UPD_WAVES) cgb.push_back(make_int2((int)k, w));
  }
  n_cg_blocks_ = (int)cgb.size();
  // rigid set and body table, rebuilt from the scenes' host data (ranges of
  // retired scenes map to no body; their table entries get rank -1)
  if (nd.NRn > 0 || nd.nbodies > 0) {
    std::vector<int> rp(std::max(nd.NRn, 1), -1), rwb(std::max(nd.NRn / 64, 1), -1);
    std::vector<BodyDev> bt(std::max(nd.nbodies, 1));
    for (auto& b : bt) {
      b = BodyDev{};
      b.rank = -1;
    }
    for (size_t k = 0; k < scenes.size(); k++) {
      const SceneHost& s = *scenes[k];
      if (s.rest_cm.size() < 3 * (size_t)s.nbody || s.body_off.size() < (size_t)s.nbody + 1) {
        set_error("rigid bodies without rest centres");
        return NN_E_STATE;
      }
      int off = s.r_begin;
      for (int b = 0; b < s.nbody; b++) {
        const int lo = s.body_off[b], hi = s.body_off[b + 1];
        for (int m = lo; m < hi; m++) rp[off + m - lo] = s.body_ids[m];
        const int len = round_up64(hi - lo);
        for (int w = off / 64; w < (off + len) / 64; w++) rwb[w] = s.body_begin + b;
        BodyDev& e = bt[s.body_begin + b];
        e.scene = (int)k;
        e.rank = b;
        e.wave_begin = off / 64;
        e.wave_end = (off + len) / 64;
        for (int c = 0; c < 3; c++) e.rest_cm[c] = e.cm[c] = s.rest_cm[3 * b + c];
        for (int q = 0; q < 9; q++) e.R[q] = (q % 4) == 0 ? 1.0f : 0.0f;
        off += len;
      }
    }
    if (nd.NRn > 0) {
      HIPCHK(hipMemcpyAsync((void*)nd.r_pid, rp.data(), sizeof(int) * nd.NRn, hipMemcpyHostToDevice, stream));
      HIPCHK(hipMemcpyAsync((void*)nd.r_wave_body, rwb.data(), sizeof(int) * (nd.NRn / 64), hipMemcpyHostToDevice, stream));
    }
    if (nd.nbodies > 0)
      HIPCHK(hipMemcpyAsync((void*)nd.bodies, bt.data(), sizeof(BodyDev) * nd.nbodies, hipMemcpyHostToDevice, stream));
    // the host vectors must outlive the copies
    HIPCHK(hipStreamSynchronize(stream));
  }
  if (!cgb.empty())
    HIPCHK(hipMemcpyAsync((void*)nd.cg_blocks, cgb.data(), sizeof(int2) * cgb.size(), hipMemcpyHostToDevice, stream));
  if (!scenes.empty())
    HIPCHK(hipMemcpyAsync((void*)nd.scenes, hs.data(), sizeof(SceneDev) * hs.size(), hipMemcpyHostToDevice, stream));
  if (nd.W) HIPCHK(hipMemcpyAsync((void*)nd.wave_scene, hw.data(), sizeof(int) * nd.W, hipMemcpyHostToDevice, stream));
  if (nd.SW) HIPCHK(hipMemcpyAsync((void*)nd.s_wave_scene, hsw.data(), sizeof(int) * nd.SW, hipMemcpyHostToDevice, stream));
  // the host vectors must outlive the copies
  HIPCHK(hipStreamSynchronize(stream));
  return NN_OK;
}

// Persistent state of scene s (at its offsets in nd) from batch `from`, where
// it sits at slot ob and stress-set slot osb with a stress set of ons members.
int Batch::copy_scene_state(const Dev& nd, const SceneHost& s, const Batch* from, int ob, int osb, int ons) {
  const Dev& od = from->d;
  const int nb = s.p_begin, n = s.n;
  auto cp = [&](void* dst, const void* sp, size_t bytes) -> hipError_t {
    return bytes ? hipMemcpyAsync(dst, sp, bytes, hipMemcpyDeviceToDevice, stream) : hipSuccess;
  };
  HIPCHK(cp(nd.pos + nb, od.pos + ob, sizeof(float4) * n));
  HIPCHK(cp(nd.vel + nb, od.vel + ob, sizeof(float4) * n));
  HIPCHK(cp(nd.info + nb, od.info + ob, sizeof(int) * n));
  HIPCHK(cp(nd.inv + nb, od.inv + ob, sizeof(int) * n));
  HIPCHK(cp(nd.x0 + nb, od.x0 + ob, sizeof(float4) * n));
  HIPCHK(cp(nd.s_of + nb, od.s_of + ob, sizeof(int) * n));
  HIPCHK(cp(nd.rho + nb, od.rho + ob, sizeof(float) * n));
  HIPCHK(cp(nd.sa + nb, od.sa + ob, sizeof(float2) * n));
  HIPCHK(cp(nd.acc + nb, od.acc + ob, sizeof(float4) * n));
  HIPCHK(cp(nd.gam + nb, od.gam + ob, sizeof(float) * n));
  HIPCHK(cp(nd.eta + nb, od.eta + ob, sizeof(float) * n));
  HIPCHK(cp(nd.vdiff + nb, od.vdiff + ob, sizeof(float4) * n));
  if (s.ns > 0 && ons == s.ns) {  // a resized stress set is uploaded afresh
    const int ns_ = s.s_begin;
    HIPCHK(cp(nd.s_pid + ns_, od.s_pid + osb, sizeof(int) * s.ns));
    HIPCHK(cp(nd.rest_cnt + ns_, od.rest_cnt + osb, sizeof(int) * s.ns));
    HIPCHK(cp(nd.rs + 4L * ns_, od.rs + 4L * osb, sizeof(float4) * 4 * s.ns));
    HIPCHK(hipMemcpy2DAsync(nd.rest + ns_, sizeof(int) * nd.NS, od.rest + osb, sizeof(int) * od.NS,
                            sizeof(int) * s.ns, MAX_REST, hipMemcpyDeviceToDevice, stream));
  }
  return NN_OK;
}

int Batch::layout(const std::vector<const Batch*>& from, double slack, int scene_capacity) {
  struct Src {
    const Batch* b;
    int pb, sb, ns;  // offsets and stress-set size in the source batch
  };
  std::vector<Src> src(scenes.size(), Src{nullptr, 0, 0, 0});
  for (size_t k = 0; k < scenes.size(); k++) {
    for (const Batch* b : from) {
      if (!b) continue;
      for (auto& t : b->scenes)
        if (t.get() == scenes[k].get()) src[k] = Src{b, scenes[k]->p_begin, scenes[k]->s_begin, scenes[k]->dev.ns};
    }
  }
  // offsets, packed in member order (committed once the arrays exist)
  int P = 0, C = 0, NS = 0, NR = 0, NB = 0;
  std::vector<int> pb(scenes.size()), cb(scenes.size()), sb(scenes.size()), rb(scenes.size()), bb(scenes.size());
  for (size_t k = 0; k < scenes.size(); k++) {
    const SceneHost& s = *scenes[k];
    pb[k] = P;
    P += round_up64(s.n);
    cb[k] = C;
    C += (int)s.ncells + 1;
    sb[k] = NS;
    NS += round_up64(s.ns);
    rb[k] = NR;
    NR += s.nr;
    bb[k] = NB;
    NB += s.nbody;
  }
  // capacities: the extents, grown by `slack` so that scenes can be appended
  // later without moving the others
  slack = slack < 1.0 ? 1.0 : slack;
  const int Pc = round_up64((int)std::ceil(P * slack));
  const int Cc = (int)std::ceil(C * slack);
  const int NSc = round_up64((int)std::ceil(NS * slack));
  const int NRc = round_up64((int)std::ceil(NR * slack));
  const int NBc = (int)std::ceil(NB * slack);
  const int Sc = std::max<int>((int)scenes.size(), scene_capacity);
  // new arrays
  Dev nd{};
  std::vector<Alloc> old_allocs;
  old_allocs.swap(allocs_);
  long long old_bytes = bytes_;
  bytes_ = 0;
  nd.P = Pc;
  nd.W = Pc / 64;
  nd.Pn = P;
  nd.C = C;
  nd.NS = NSc;
  nd.SW = NSc / 64;
  nd.NSn = NS;
  nd.NR = NRc;
  nd.NRn = NR;
  nd.nbodies = NB;
  nd.nscenes = (int)scenes.size();
  const int ncell_entries = Cc + 1;
  const size_t nscan = (size_t)scan_tmp_ints(ncell_entries);
  std::vector<std::pair<void**, size_t>> req;
  auto A = [&](auto*& p, size_t count) {
    using T = std::remove_reference_t<decltype(*p)>;
    req.push_back({(void**)&p, (count ? count : 1) * sizeof(T)});
  };
  // arrays that start at zero, arrays that start at -1, and the others
  A(nd.state, Sc);
  A(nd.pos, Pc);
  A(nd.pos_alt, Pc);
  A(nd.vel, Pc);
  A(nd.vel_alt, Pc);
  A(nd.acc, Pc);
  A(nd.rho, Pc);
  A(nd.sa, Pc);
  A(nd.gam, Pc);
  A(nd.eta, Pc);
  A(nd.x0, Pc);
  A(nd.vdiff, Pc);
  A(nd.vdiff_alt, Pc);  // swapped with vdiff also where the sort does not copy it
  A(nd.nnbr, Pc);
  A(nd.rest_cnt, NSc);
  A(nd.info, Pc);
  A(nd.info_alt, Pc);
  A(nd.s_of, Pc);
  A(nd.s_pid, NSc);
  SceneDev* scenes_dev = nullptr;
  A(scenes_dev, Sc);
  int* ws = nullptr;
  A(ws, nd.W);
  int* sws = nullptr;
  A(sws, nd.SW);
  A(nd.nbr, (size_t)Pc * MAX_NB);
  A(nd.key, Pc);
  A(nd.rank, Pc);
  A(nd.inv, Pc);
  A(nd.bucket, Pc);
  A(nd.cell_count, ncell_entries);
  A(nd.cell_start, ncell_entries);
  A(nd.scan_tmp, nscan);
  A(nd.partials, 32 * (size_t)nd.W);
  int2* cgb = nullptr;
  A(cgb, (size_t)nd.W / CG_UPD_WAVES + Sc + 1);
  A(nd.cg_list, 3 * (size_t)nd.W);
  A(nd.cg_list_n, 3);
  A(nd.n_active, 4);
  A(nd.wx, Pc);
  A(nd.wr, Pc);
  A(nd.ww, Pc);
  A(nd.wp, Pc);
  A(nd.ws, Pc);
  A(nd.xu, Pc);
  A(nd.wd0, Pc);
  A(nd.wd1, Pc);
  A(nd.spair, (size_t)Pc * MAX_NB);
  A(nd.mu, Pc);
  A(nd.rest, (size_t)NSc * MAX_REST);
  A(nd.rs, 4 * (size_t)NSc);
  int* rpid = nullptr;
  A(rpid, NRc);
  int* rwb = nullptr;
  A(rwb, NRc / 64);
  A(nd.rpartials, 9 * (size_t)(NRc / 64));
  A(nd.bodies, NBc);
  const int rc = alloc_arena(req);
  if (rc != NN_OK) {
    release();
    allocs_.swap(old_allocs);
    bytes_ = old_bytes;
    return rc;
  }
  // the sort's keys and ranks are dead once the lists are being built: 16 W of
  // the wavefronts' counts and densities fit in each (64 W words)
  nd.wave_pairs = reinterpret_cast<int2*>(nd.rank);
  nd.wave_rho = reinterpret_cast<float*>(nd.key);
  nd.cg_waves = nd.bucket;  // the search's, dead after it
  nd.scenes = scenes_dev;
  nd.wave_scene = ws;
  nd.s_wave_scene = sws;
  nd.cg_blocks = cgb;
  nd.r_pid = rpid;
  nd.r_wave_body = rwb;
  for (size_t k = 0; k < scenes.size(); k++) {
    scenes[k]->p_begin = pb[k];
    scenes[k]->cell_begin = cb[k];
    scenes[k]->s_begin = sb[k];
    scenes[k]->r_begin = rb[k];
    scenes[k]->body_begin = bb[k];
  }
  derive_members();
  C_total_ = C;
  C_cap_ = Cc;
  NB_cap_ = NBc;
  scene_cap_ = Sc;
  // pinned host copies of the scene states and their report words, for as many
  // scenes as the layout holds (a staging batch holds one; hipHostFree
  // synchronizes the device)
  if (!h_state_ || h_state_cap_ < Sc) {
    if (h_state_) HIPCHK(hipStreamSynchronize(stream));
    free_host(h_state_, h_state_bytes_);
    h_state_ = nullptr;
    const size_t cap = (size_t)std::max(Sc, 1);
    CHK(alloc_host((void**)&h_state_, state_bytes((int)cap), h_state_bytes_));
    h_report_ = reinterpret_cast<unsigned long long*>(h_state_ + cap);
    std::fill(h_report_, h_report_ + cap, 0ull);
    h_state_cap_ = (int)cap;
    HIPCHK(hipHostGetDevicePointer((void**)&state_dev_, h_state_, 0));
    report_dev_ = reinterpret_cast<unsigned long long*>(state_dev_ + cap);
  }
  // nothing else is read before it is written (device memory comes as it was
  // left, new or used again; every GPU test gives the same with the rest filled
  // with NaN and, where it holds indices, with 1)
  launch_fill_f4(reinterpret_cast<float4*>(nd.state), (long)((char*)nd.info - (char*)nd.state) / 16,
                 make_float4(0.f, 0.f, 0.f, 0.f), stream);
  launch_fill_i32(nd.info, (long)((char*)scenes_dev - (char*)nd.info) / 4, -1, stream);
  CHK(upload_tables(nd));
  // copy persistent state of relocated scenes
  for (size_t k = 0; k < scenes.size(); k++)
    if (src[k].b) CHK(copy_scene_state(nd, *scenes[k], src[k].b, src[k].pb, src[k].sb, src[k].ns));
  HIPCHK(hipStreamSynchronize(stream));
  // the old arrays are freed by the caller's choice: now, or later (off the
  // thread that steps the batch; hipFree waits for the device)
  if (defer_free_) {
    for (auto& al : old_allocs) deferred_.push_back(al);
  } else {
    for (auto& al : old_allocs) free_arena(al);
  }
  d = nd;
  lists_state_ = 0;
  return NN_OK;
}

int Batch::append_in_place(const std::vector<std::shared_ptr<SceneHost>>& members, const std::vector<const Batch*>& from) {
  // the scenes kept must come first, in their present order
  std::vector<SceneHost*> cur;
  for (auto& sp : scenes) cur.push_back(sp.get());
  size_t nk = 0, pos = 0;
  for (; nk < members.size(); nk++) {
    auto it = std::find(cur.begin() + pos, cur.end(), members[nk].get());
    if (it == cur.end()) break;
    pos = (size_t)(it - cur.begin()) + 1;
  }
  for (size_t k = nk; k < members.size(); k++)
    if (std::find(cur.begin(), cur.end(), members[k].get()) != cur.end()) return LAYOUT_NEEDED;
  if ((int)members.size() > scene_cap_) return LAYOUT_NEEDED;
  // offsets of the new scenes, after the last slot, cell and stress slot used
  int P = d.Pn, C = C_total_, NS = d.NSn, NR = d.NRn, NB = d.nbodies;
  std::vector<std::pair<int, int>> place(members.size(), {0, 0});  // (p_begin, s_begin) of new scenes
  std::vector<int> cells(members.size(), 0), rb(members.size(), 0), bb(members.size(), 0);
  for (size_t k = nk; k < members.size(); k++) {
    const SceneHost& s = *members[k];
    place[k] = {P, NS};
    cells[k] = C;
    rb[k] = NR;
    bb[k] = NB;
    P += round_up64(s.n);
    C += (int)s.ncells + 1;
    NS += round_up64(s.ns);
    NR += s.nr;
    NB += s.nbody;
  }
  if (P > d.P || C > C_cap_ || NS > d.NS || NR > d.NR || NB > NB_cap_) return LAYOUT_NEEDED;
  // sources of the new scenes
  struct Src {
    const Batch* b;
    int pb, sb, ns;
  };
  std::vector<Src> src(members.size(), Src{nullptr, 0, 0, 0});
  for (size_t k = nk; k < members.size(); k++)
    for (const Batch* b : from) {
      if (!b || b == this) continue;
      for (auto& t : b->scenes)
        if (t.get() == members[k].get()) src[k] = Src{b, t->p_begin, t->s_begin, t->dev.ns};
    }
  for (size_t k = nk; k < members.size(); k++) {
    SceneHost& s = *members[k];
    s.p_begin = place[k].first;
    s.s_begin = place[k].second;
    s.cell_begin = cells[k];
    s.r_begin = rb[k];
    s.body_begin = bb[k];
  }
  scenes = members;
  derive_members();
  d.Pn = P;
  d.NSn = NS;
  d.NRn = NR;
  d.nbodies = NB;
  d.nscenes = (int)scenes.size();
  C_total_ = C;
  d.C = C;
  CHK(upload_tables(d));
  for (size_t k = nk; k < members.size(); k++)
    if (src[k].b) CHK(copy_scene_state(d, *members[k], src[k].b, src[k].pb, src[k].sb, src[k].ns));
  HIPCHK(hipStreamSynchronize(stream));
  if (nk < members.size()) lists_state_ = 0;  // the new scenes have no lists here yet
  return NN_OK;
}

void Batch::take_deferred(std::vector<Alloc>& out) {
  out.insert(out.end(), deferred_.begin(), deferred_.end());
  deferred_.clear();
}

int Batch::refresh_scene_table() {
  std::vector<SceneDev> hs(scenes.size());
  for (size_t k = 0; k < scenes.size(); k++) hs[k] = scenes[k]->dev;
  if (!hs.empty())
    HIPCHK(hipMemcpyAsync((void*)d.scenes, hs.data(), sizeof(SceneDev) * hs.size(), hipMemcpyHostToDevice, stream));
  max_iter_[0] = max_iter_[1] = max_iter_[2] = 1;
  any_velocity_terms_ = false;
  for (auto& sp : scenes) {
    any_velocity_terms_ |= velocity_terms(sp->dev);
    max_iter_[0] = std::max(max_iter_[0], sp->dev.max_iter_v);
    max_iter_[1] = std::max(max_iter_[1], sp->dev.max_iter_p);
    max_iter_[2] = std::max(max_iter_[2], sp->dev.max_iter_cg);
  }
  HIPCHK(hipStreamSynchronize(stream));
  return NN_OK;
}

int Batch::upload(int k, const float* x, const float* v, const int* kind) {
  SceneHost& s = *scenes[k];
  const int n = s.n, pb = s.p_begin;
  // expanded on the device, from staging memory or (larger scenes) from a copy
  // in the pair scalars, which only a step uses
  const size_t words = (size_t)(v ? 7 : 4) * n;
  (void)hipGetLastError();  // what another call left on this thread is not this one's error
  float* raw = d.spair;
  if (4 * words <= STAGE_BYTES) {
    CHK(stage());
    std::memcpy(h_stage_, x, sizeof(float) * 3 * n);
    std::memcpy(h_stage_ + 3 * (size_t)n, kind, sizeof(int) * n);
    if (v) std::memcpy(h_stage_ + 4 * (size_t)n, v, sizeof(float) * 3 * n);
    raw = stage_dev_;
  } else {
    HIPCHK(hipMemcpyAsync(raw, x, sizeof(float) * 3 * n, hipMemcpyHostToDevice, stream));
    HIPCHK(hipMemcpyAsync(raw + 3 * (size_t)n, kind, sizeof(int) * n, hipMemcpyHostToDevice, stream));
    if (v) HIPCHK(hipMemcpyAsync(raw + 4 * (size_t)n, v, sizeof(float) * 3 * n, hipMemcpyHostToDevice, stream));
  }
  launch_expand(dref(), pb, n, s.dev.vol0, raw, reinterpret_cast<const int*>(raw + 3 * (size_t)n),
                v ? raw + 4 * (size_t)n : nullptr, stream);
  HIPCHK(hipGetLastError());
  HIPCHK(hipStreamSynchronize(stream));
  s.initialized = false;
  s.stepped = false;
  return NN_OK;
}

// ---------------------------------------------------------------------------
// kernel timer
// ---------------------------------------------------------------------------
static const char* const KERNEL_NAMES[K_COUNT] = {
    "cell_count", "scan", "bucket", "place", "build_lists", "bvol", "clear_acc", "density_alpha",
    "div_update", "div_source", "strain", "cg_init", "cg_matvec", "cg_update", "nonpressure",
    "press_source", "press_update", "elastic_rot_stress", "elastic_force", "advect", "cg_guess"};

const char* kernel_name(int id) { return (id >= 0 && id < K_COUNT) ? KERNEL_NAMES[id] : ""; }

KernelTimer::~KernelTimer() {
  for (auto e : events) (void)hipEventDestroy(e);
}

LaunchEvents& launch_events() {
  static thread_local LaunchEvents e;
  return e;
}

// A timed launch carries a start and a stop event (NN_LAUNCH): the dispatch
// stamps them itself, so the duration is the kernel's and the timing adds no
// packets to the stream.
int KernelTimer::begin(int id, hipStream_t st) {
  (void)st;
  open = false;
  if (!on) return NN_OK;
  const long long n = seen[id]++;  // every kernel's launches are counted while on
  if (!((mask >> id) & 1u) || n % stride != 0) return NN_OK;
  open = true;
  while (events.size() < used + 2) {
    hipEvent_t e;
    HIPCHK(hipEventCreateWithFlags(&e, TIMING_EVENT_FLAGS));
    events.push_back(e);
  }
  pending.push_back({id, used});
  LaunchEvents& le = launch_events();
  le.start = events[used];
  le.stop = events[used + 1];
  le.launched = false;
  used += 2;
  return NN_OK;
}

int KernelTimer::end(hipStream_t st) {
  (void)st;
  if (!open) return NN_OK;
  open = false;
  LaunchEvents& le = launch_events();
  if (!le.launched) pending.pop_back();  // the launcher launched nothing (no work): no sample
  le = LaunchEvents{};
  return NN_OK;
}

int KernelTimer::collect() {
  for (auto& p : pending) {
    float ms = 0.0f;
    HIPCHK(hipEventElapsedTime(&ms, events[p.second], events[p.second + 1]));
    total_ms[p.first] += ms;
    count[p.first]++;
  }
  pending.clear();
  used = 0;
  return NN_OK;
}

void KernelTimer::reset() {
  for (int k = 0; k < K_COUNT; k++) {
    total_ms[k] = 0.0;
    count[k] = 0;
    seen[k] = 0;
  }
}

#define TIMED(id, call)               \
  do {                                \
    CHK(timer.begin((id), stream));   \
    call;                             \
    CHK(timer.end(stream));           \
  } while (0)

// The counting sort and the lists.  all == 0 (inside a step) leaves static
// boundary particles without a list; lists_state_ records which kind of search
// ran last, so that list downloads can complete them first.
int Batch::search_impl(int all, int begin) {
  launch_begin(dref(), begin, (long)C_total_ + 1, stream);
  TIMED(K_CELL_COUNT, launch_cell_count(dref(), blk(K_CELL_COUNT), stream));
  TIMED(K_SCAN, launch_scan(dref(), C_total_ + 1, stream));
  TIMED(K_BUCKET, launch_bucket(dref(), blk(K_BUCKET), stream));
  TIMED(K_PLACE, launch_place(dref(), blk(K_PLACE), begin == BEGIN_STEP, stream));
  swap_sort_buffers();
  TIMED(K_BUILD_LISTS, launch_build_lists(dref(), blk(K_BUILD_LISTS), lanes(K_BUILD_LISTS), all, stream));
  lists_state_ = all ? 2 : 1;
  return NN_OK;
}

int Batch::search() {
  if (scenes.empty()) return NN_OK;
  CHK(search_impl(1, BEGIN_STATUS));
  HIPCHK(hipGetLastError());
  CHK(gather_state());
  for (size_t k = 0; k < scenes.size(); k++) {
    const int stt = h_state_[k].status;
    if (stt & ST_OUT_OF_GRID) { set_error("particle outside the grid"); return NN_E_OUT_OF_GRID; }
    if (stt & ST_CELL_OVERFLOW) { set_error("more than 50 particles in a cell"); return NN_E_CELL_OVERFLOW; }
    if (stt & ST_NEIGHBOR_OVERFLOW) { set_error("more than 60 neighbors"); return NN_E_NEIGHBOR_OVERFLOW; }
  }
  return NN_OK;
}

// Waits until each of the first n report words carries the ticket, the last one
// given out by default (later: or one after it); bits: the or of what they
// report.  Polling them costs 6 us less than a copy of the counter and a wait for
// the stream (six small launches and the wait: 19.5 us against 26); a wait that
// lasts is left to the stream's, which also returns the errors of launches that
// cannot report.
int Batch::await(int n, unsigned& bits) { return await(n, bits, ticket_, false); }
int Batch::await(int n, unsigned& bits, unsigned ticket, bool later) {
  HIPCHK(hipGetLastError());
  bits = 0;
  bool synced = false;
  const auto start = std::chrono::steady_clock::now();
  for (int k = 0, polls = 0; k < n;) {
    const unsigned long long v = __atomic_load_n(h_report_ + k, __ATOMIC_ACQUIRE);
    if ((unsigned)(v >> 32) == ticket || (later && (int)((unsigned)(v >> 32) - ticket) > 0)) {
      bits |= (unsigned)v;
      k++;
    } else if (synced) {
      set_error("a launch did not report its end");
      return NN_E_HIP;
    } else if (++polls % 64 == 0 && std::chrono::steady_clock::now() - start > std::chrono::microseconds(300)) {
      HIPCHK(hipStreamSynchronize(stream));
      synced = true;
    } else {
      __builtin_ia32_pause();
    }
  }
  return NN_OK;
}

int Batch::gather_state() {
  const size_t ns = scenes.size();
  if (ns > 4096) {
    set_error("too many scenes in one batch");
    return NN_E_ARG;
  }
  HIPCHK(hipMemcpyAsync(h_state_, d.state, sizeof(SceneState) * ns, hipMemcpyDeviceToHost, stream));
  HIPCHK(hipStreamSynchronize(stream));
  return NN_OK;
}

// stress set: elastic particles and their rest neighbors (first search), with
// rest lists capped at 50 (Elasticity.initValues_kernel, :1220-1236)
int Batch::build_stress_set(const std::vector<int>& which, bool& any) {
  any = false;
  for (int k : which) {
    SceneHost& s = *scenes[k];
    s.s_pid.clear();
    s.rest.clear();
    s.rest_cnt.clear();
    s.ns = 0;
    if (s.n_elastic == 0) continue;
    any = true;
    const int n = s.n, pb = s.p_begin;
    std::vector<int> info(n), cnt(n), nb((size_t)n * MAX_NB);
    HIPCHK(hipMemcpyAsync(info.data(), d.info + pb, sizeof(int) * n, hipMemcpyDeviceToHost, stream));
    HIPCHK(hipMemcpyAsync(cnt.data(), d.nnbr + pb, sizeof(int) * n, hipMemcpyDeviceToHost, stream));
    HIPCHK(copy_lists(nb.data(), d, pb, n, stream));
    HIPCHK(hipStreamSynchronize(stream));
    CHK(lists_to_local(nb, cnt, pb, n));
    std::vector<int> slot_of_id(n, -1);
    for (int t = 0; t < n; t++) slot_of_id[info[t] & 0x0FFFFFFF] = t;
    std::vector<char> mark(n, 0);
    for (int t = 0; t < n; t++) {
      if ((info[t] >> 28) != KIND_ELASTIC) continue;
      mark[info[t] & 0x0FFFFFFF] = 1;
      for (int m = 0; m < cnt[t]; m++) mark[info[nb[host_nb(n, t, m)]] & 0x0FFFFFFF] = 1;
    }
    std::vector<int> s_of(n, -1);
    for (int id = 0; id < n; id++)
      if (mark[id]) {
        s_of[id] = (int)s.s_pid.size();
        s.s_pid.push_back(id);
      }
    s.ns = (int)s.s_pid.size();
    s.rest.assign((size_t)s.ns * MAX_REST, -1);
    s.rest_cnt.assign(s.ns, 0);
    bool overflow = false;
    for (int q = 0; q < s.ns; q++) {
      const int t = slot_of_id[s.s_pid[q]];
      int c = cnt[t];
      if (c > MAX_REST) {
        overflow = true;
        c = MAX_REST;
      }
      s.rest_cnt[q] = c;
      for (int m = 0; m < c; m++) s.rest[(size_t)q * MAX_REST + m] = info[nb[host_nb(n, t, m)]] & 0x0FFFFFFF;
    }
    if (overflow) {
      set_error("an elastic particle has more than 50 rest neighbors");
      return NN_E_REST_OVERFLOW;
    }
    s_of.swap(s.s_of_host);  // uploaded after the relayout below
  }
  if (!any) return NN_OK;
  // re-layout with the new stress-set sizes, keeping all particle state
  CHK(layout({this}));
  for (int k : which) {
    SceneHost& s = *scenes[k];
    if (s.ns == 0) continue;
    const int sb = s.s_begin, pb = s.p_begin;
    std::vector<int> rest_t((size_t)s.ns * MAX_REST);
    for (int q = 0; q < s.ns; q++)
      for (int m = 0; m < MAX_REST; m++) rest_t[(size_t)m * s.ns + q] = s.rest[(size_t)q * MAX_REST + m];
    HIPCHK(hipMemcpyAsync(d.s_pid + sb, s.s_pid.data(), sizeof(int) * s.ns, hipMemcpyHostToDevice, stream));
    HIPCHK(hipMemcpyAsync(d.rest_cnt + sb, s.rest_cnt.data(), sizeof(int) * s.ns, hipMemcpyHostToDevice, stream));
    HIPCHK(hipMemcpy2DAsync(d.rest + sb, sizeof(int) * d.NS, rest_t.data(), sizeof(int) * s.ns, sizeof(int) * s.ns,
                            MAX_REST, hipMemcpyHostToDevice, stream));
    HIPCHK(hipMemcpyAsync(d.s_of + pb, s.s_of_host.data(), sizeof(int) * s.n, hipMemcpyHostToDevice, stream));
  }
  HIPCHK(hipStreamSynchronize(stream));
  return NN_OK;
}

int Batch::init_scenes(const std::vector<int>& which) {
  if (scenes.empty()) return NN_OK;
  CHK(search_impl(1, BEGIN_STATUS));
  launch_elastic_init(dref(), block, stream);
  HIPCHK(hipGetLastError());
  CHK(gather_state());
  for (size_t k = 0; k < scenes.size(); k++) {
    const int stt = h_state_[k].status;
    if (stt & ST_OUT_OF_GRID) { set_error("particle outside the grid"); return NN_E_OUT_OF_GRID; }
    if (stt & ST_CELL_OVERFLOW) { set_error("more than 50 particles in a cell"); return NN_E_CELL_OVERFLOW; }
    if (stt & ST_NEIGHBOR_OVERFLOW) { set_error("more than 60 neighbors"); return NN_E_NEIGHBOR_OVERFLOW; }
  }
  bool relayout = false;
  CHK(build_stress_set(which, relayout));
  // the stress-set relayout does not carry neighbor lists (they hold absolute
  // slots); search again on the unchanged positions before the volume sweeps
  if (relayout) CHK(search_impl(1, BEGIN_CELLS));
  launch_bvol(dref(), block, lanes(K_BVOL), 0, stream);
  launch_bvol(dref(), block, lanes(K_BVOL), 1, stream);
  HIPCHK(hipGetLastError());
  HIPCHK(hipStreamSynchronize(stream));
  for (int k : which) scenes[k]->initialized = true;
  return NN_OK;
}

// RigidBodySolver.substep for every scene's bodies (:929-931): body rank r
// of all scenes together, coupling_interval substeps each (a scene with fewer
// bodies or substeps sits the extra launches out); small bodies in one launch.
int Batch::rigid_step() {
  if (max_body_waves_ <= RB_WHOLE) {
    if (max_coupling_ > 0) launch_rigid_ground(dref(), 0, 0, stream);
    launch_rigid_bodies(dref(), stream);
    HIPCHK(hipGetLastError());
    return NN_OK;
  }
  for (int r = 0; r < max_body_; r++)
    for (int c = 0; c < max_coupling_; c++) {
      launch_rigid_ground(dref(), r, c, stream);
      launch_rigid_sum(dref(), 0, r, c, stream);
      launch_body_finish(dref(), 0, r, c, stream);
      launch_rigid_sum(dref(), 1, r, c, stream);
      launch_body_finish(dref(), 1, r, c, stream);
      launch_rigid_place(dref(), r, c, stream);
    }
  HIPCHK(hipGetLastError());
  return NN_OK;
}

// Runs solver iterations until no scene is active: the first chunk is the
// previous step's count, later chunks four at a time; the last scene finish of a
// chunk reports each scene's active flag to the host.
int Batch::solver_loop(int which) {
  int pred = 1;
  for (auto& sp : scenes) pred = std::max(pred, sp->last_iter[which]);
  const int maxit = std::max(1, max_iter_[which]);
  int done = 0, chunk = std::min(pred, maxit);
  for (;;) {
    ticket_++;
    const int reporting = done + chunk < maxit ? chunk - 1 : -1;  // its scene finish reports
    for (int c = 0; c < chunk; c++) {
      unsigned long long* report = c == reporting ? report_dev_ : nullptr;
      if (which == 0) {
        TIMED(K_DIV_UPDATE, launch_div_update(dref(), blk(K_DIV_UPDATE), lanes(K_DIV_UPDATE), dep(K_DIV_UPDATE), stream));
        TIMED(K_DIV_SOURCE, launch_div_source(dref(), blk(K_DIV_SOURCE), lanes(K_DIV_SOURCE), dep(K_DIV_SOURCE), stream));
        launch_scene_finish(dref(), 0, lanes(K_DIV_SOURCE), report, ticket_, stream);
      } else if (which == 1) {
        TIMED(K_PRESS_UPDATE, launch_press_update(dref(), blk(K_PRESS_UPDATE), lanes(K_PRESS_UPDATE), dep(K_PRESS_UPDATE), stream));
        TIMED(K_PRESS_SOURCE, launch_press_source(dref(), blk(K_PRESS_SOURCE), lanes(K_PRESS_SOURCE), dep(K_PRESS_SOURCE), 1, stream));
        launch_scene_finish(dref(), 1, lanes(K_PRESS_SOURCE), report, ticket_, stream);
      }
    }
    done += chunk;
    if (done >= maxit) break;
    unsigned active = 0;
    CHK(await((int)scenes.size(), active));
    if (!active) break;
    chunk = std::min(4, maxit - done);
  }
  return NN_OK;
}

// The Weiler CG.  A batch of one scene of few waves (with a workgroup for each
// and no more than the compute units): one launch, k_cg_solve, which may give
// up waiting.  An iteration then takes 6.3 us at 27 waves, 7.0 at 102 and 8.0
// at 222, against 13 to 15 as two launches.  Otherwise update k (which first forms
// the scene sums of iteration k - 1 and stops converged scenes) and matvec k,
// for k = 1 .. limit, then update limit + 1, which only tests the last
// residual.  Enqueued in chunks -- first the previous step's iteration count
// plus three, then four -- with one report of the active-scene counter per chunk;
// iterations past convergence are near-empty launches.
int Batch::cg_start() {
  TIMED(K_CG_INIT, launch_cg_init(dref(), blk(K_CG_INIT), stream));
  if (any_warm_cg_) launch_scene_finish(dref(), 4, 1, nullptr, 0, stream);
  TIMED(K_CG_GUESS, launch_cg_guess(dref(), blk(K_CG_GUESS), stream));
  TIMED(K_CG_MATVEC, launch_cg_matvec_start(dref(), blk(K_CG_MATVEC), dep(K_CG_MATVEC), stream));
  launch_scene_finish(dref(), 2, 1, nullptr, 0, stream);
  return NN_OK;
}

constexpr int SOLVE_REST = 256;
// Workgroups of the one-launch solves under way, by device.  Each holds a compute
// unit and waits for the others of its solve, so solves of several contexts run
// at once only while there is a compute unit for every workgroup: three of 200
// waves in three threads left a solve each after a wait in vain (0.68 ms for a
// step of all three over the first 60, 0.56 with this; later steps the same).
constexpr int SOLVE_DEVICES = 64;
static std::atomic<int> solving[SOLVE_DEVICES];

int Batch::cg_solve(bool& done, bool& gave_up) {
  done = gave_up = false;
  if (cus_ < 0) {
    HIPCHK(hipGetDevice(&device_));
    HIPCHK(hipDeviceGetAttribute(&cus_, hipDeviceAttributeMultiprocessorCount, device_));
  }
  if (solve_rest_ > 0 && solve_rest_-- > 0) return NN_OK;
  if (dep(K_CG_MATVEC) != 0) return NN_OK;  // a gather depth was asked for: it is k_cg_matvec's
  if (scenes.size() != 1 || scenes[0]->dev.wave_begin != 0) return NN_OK;
  const int waves = scenes[0]->dev.wave_end;
  if (waves > std::min(cus_, CG_SOLVE_WAVES) || device_ >= SOLVE_DEVICES) return NN_OK;
  struct Share {
    std::atomic<int>& all;
    const int mine;
    const bool fits;
    Share(std::atomic<int>& a, int n, int limit) : all(a), mine(n), fits(a.fetch_add(n) + n <= limit) {}
    ~Share() { all.fetch_sub(mine); }
  } share(solving[device_], waves, cus_);
  if (!share.fits) return NN_OK;
  if (timer.on) timer.seen[K_CG_UPDATE]++;  // one launch does the work of both
  TIMED(K_CG_MATVEC, launch_cg_solve(dref(), waves, cg_patience, stream));
  unsigned bits = 0;
  launch_report_active(dref(), 1, report_dev_, ++ticket_, stream);
  CHK(await(1, bits));
  gave_up = bits != 0;
  done = !gave_up;
  // the device was busy: a wait in vain takes about 15 ms, a solve in one launch
  // saves about 0.5 ms, so the next try comes after SOLVE_REST solves
  if (gave_up) solve_rest_ = SOLVE_REST;
  return NN_OK;
}

int Batch::cg_loop() {
  int pred = 1;
  long last_waves = 0;
  for (auto& sp : scenes) {
    const int f = sp->dev.flags;
    if (!((f & SF_HAS_FLUID) && (f & SF_VISCOSITY) && (f & SF_WEILER))) continue;
    if (sp->last_iter[2] > pred) last_waves = 0;
    pred = std::max(pred, sp->last_iter[2]);
    if (sp->last_iter[2] == pred) last_waves += sp->dev.wave_end - sp->dev.wave_begin;
  }
  // waves expected to still iterate at iteration k, from each scene's count
  // in the previous step (plus a margin; past every count, the scenes that had
  // the most): the matvec's grid (its list of waves holds the exact set either
  // way; a grid of 64 workgroups for a scene of 131,072 particles that iterated
  // longer than it had before took 141 us a product instead of 16)
  auto expected_waves = [&](int k) {
    long w = 0;
    for (auto& sp : scenes) {
      const int f = sp->dev.flags;
      if ((f & SF_HAS_FLUID) && (f & SF_VISCOSITY) && (f & SF_WEILER) && sp->last_iter[2] + 2 >= k)
        w += sp->dev.wave_end - sp->dev.wave_begin;
    }
    return std::max(w, last_waves);
  };
  const int maxit = std::max(1, max_iter_[2]);
  const int last = maxit + 1;
  int k = 1, chunk = std::min(pred + 3, last);
  for (;;) {
    for (int c = 0; c < chunk && k <= last; c++, k++) {
      TIMED(K_CG_UPDATE, launch_cg_update(dref(), n_cg_blocks_, k, stream));
      if (k > maxit) continue;
      TIMED(K_CG_MATVEC, launch_cg_matvec(dref(), dep(K_CG_MATVEC), k, (int)expected_waves(k), stream));
    }
    if (k > last) break;
    unsigned active = 0;
    launch_report_active(dref(), 0, report_dev_, ++ticket_, stream);
    CHK(await(1, active));
    if (!active) break;
    chunk = 4;
  }
  return NN_OK;
}

int Batch::step(std::vector<nn_step_stats>* stats) {
  if (scenes.empty()) return NN_OK;
  for (auto& sp : scenes)
    if (!sp->initialized) {
      set_error("step before init");
      return NN_E_STATE;
    }
  // static particles get no list inside a step, except in batches with rigid
  // bodies: their ground collision moves positions after the search, so the
  // search positions would not survive to build those lists on demand
  CHK(search_impl(any_rigid_ ? 1 : 0, BEGIN_STEP));  // :917, :920
  if (any_elastic_ || any_rigid_) TIMED(K_BVOL, launch_bvol(dref(), blk(K_BVOL), lanes(K_BVOL), 1, stream));  // :918
  if (any_fluid_) {  // DFSPHSolver.substep, :1546-1555
    TIMED(K_DENSITY_ALPHA, launch_density_alpha(dref(), blk(K_DENSITY_ALPHA), lanes(K_DENSITY_ALPHA), dep(K_DENSITY_ALPHA), stream));
    if (any_div_) CHK(solver_loop(0));
    if (any_strain_) TIMED(K_STRAIN, launch_strain(dref(), blk(K_STRAIN), lanes(K_STRAIN), dep(K_STRAIN), stream));
    if (any_weiler_) {
      CHK(cg_start());
      bool done = false, gave_up = false;
      CHK(cg_solve(done, gave_up));
      cg_forms[done ? 0 : 1]++;
      cg_forms[2] += gave_up;
      if (!done) {
        if (gave_up) {  // from the start again
          launch_begin(dref(), BEGIN_CG, 0, stream);
          CHK(cg_start());
        }
        CHK(cg_loop());
      }
    }
    TIMED(K_NONPRESSURE, launch_nonpressure(dref(), blk(K_NONPRESSURE), lanes(K_NONPRESSURE), dep(K_NONPRESSURE), stream));
    std::swap(d.vel, d.vel_alt);
    TIMED(K_PRESS_SOURCE, launch_press_source(dref(), blk(K_PRESS_SOURCE), lanes(K_PRESS_SOURCE), dep(K_PRESS_SOURCE), 0, stream));
    CHK(solver_loop(1));
  }
  if (any_elastic_) {  // Elasticity.substep, :1241-1244
    TIMED(K_ELASTIC_ROT_STRESS, launch_elastic_rot_stress(dref(), lanes(K_ELASTIC_ROT_STRESS), stream));
    TIMED(K_ELASTIC_FORCE, launch_elastic_force(dref(), lanes(K_ELASTIC_FORCE), stream));
  }
  if (any_rigid_) CHK(rigid_step());  // :929-931
  TIMED(K_ADVECT, launch_advect(dref(), blk(K_ADVECT), stream));  // :933, :936-937
  std::swap(d.pos, d.pos_alt);  // pos_alt keeps the positions of this step's search
  launch_publish(dref(), lanes(K_BUILD_LISTS), lanes(K_DENSITY_ALPHA), state_dev_, report_dev_, ++ticket_, stream);
  unsigned none = 0;
  CHK(await((int)scenes.size(), none));
  if (timer.on) HIPCHK(hipStreamSynchronize(stream));
  CHK(timer.collect());
  int rc = NN_OK;
  if (stats) stats->resize(scenes.size());
  for (size_t k = 0; k < scenes.size(); k++) {
    SceneHost& s = *scenes[k];
    const SceneState& st = h_state_[k];
    nn_step_stats o{};
    o.iterations_v = st.iter_v;
    o.iterations_p = st.iter_p;
    o.iterations_cg = st.iter_cg;
    o.status = st.status;
    o.avg_density_err_v = st.err_v;
    o.avg_density_err_p = st.err_p;
    o.cg_rel_residual = st.cg_bb > 0.0 ? std::sqrt(st.cg_rr / st.cg_bb) : 0.0;
    float mx;
    unsigned bits = st.max_rho_bits;
    std::memcpy(&mx, &bits, 4);
    o.max_density = mx;
    o.num_pairs = (int64_t)st.pairs;
    o.num_pairs_fluid = (int64_t)st.pairs_fluid;
    s.last = o;
    s.stepped = true;
    s.last_iter[0] = std::max(1, st.iter_v);
    s.last_iter[1] = std::max(1, st.iter_p);
    s.last_iter[2] = std::max(1, st.iter_cg);
    if (stats) (*stats)[k] = o;
    int e = NN_OK;
    if (st.status & ST_NAN) e = NN_E_NAN;
    if (st.status & ST_NEIGHBOR_OVERFLOW) e = NN_E_NEIGHBOR_OVERFLOW;
    if (st.status & ST_CELL_OVERFLOW) e = NN_E_CELL_OVERFLOW;
    if (st.status & ST_OUT_OF_GRID) e = NN_E_OUT_OF_GRID;
    if (e < 0 && (rc >= 0 || e < rc)) rc = e;
    if (e == NN_OK && (st.status & ST_NOCONV) && rc == NN_OK) rc = NN_W_NOCONV;
  }
  if (rc < 0) set_error("step reported an error status (see nn_step_stats.status)");
  return rc;
}

int Batch::synchronize() {
  HIPCHK(hipStreamSynchronize(stream));
  return NN_OK;
}

// ---------------------------------------------------------------------------
// downloads in original order
// ---------------------------------------------------------------------------
static int field_width(int field) {
  switch (field) {
    case NN_FIELD_X:
    case NN_FIELD_V:
    case NN_FIELD_ACCELERATION:
    case NN_FIELD_X0:
    case NN_FIELD_VISC_DIFF:
      return 3;
    case NN_FIELD_ROTATION:
      return 9;
    case NN_FIELD_STRESS:
      return 6;
    case NN_FIELD_VOLUME:
    case NN_FIELD_DENSITY:
    case NN_FIELD_DFSPH_FACTOR:
    case NN_FIELD_DENSITY_ADV:
    case NN_FIELD_STRAIN_NORM:
    case NN_FIELD_VISCOSITY:
    case NN_FIELD_REST_VOLUME:
    case NN_FIELD_KIND:
    case NN_FIELD_NUM_NEIGHBORS:
      return 1;
    default:
      return 0;
  }
}

int Batch::stage() {
  if (h_stage_) return NN_OK;
  CHK(alloc_host((void**)&h_stage_, STAGE_BYTES, h_stage_bytes_));
  HIPCHK(hipHostGetDevicePointer((void**)&stage_dev_, h_stage_, 0));
  return NN_OK;
}

// A three-component field of n particles through the two halves of the staging
// memory: a piece is copied by the host while the kernel of the next one runs.
// launch(first particle, particles, device address of the half) reads or writes.
template <typename Launch>
int Batch::field_pieces(int n, float* out, const float* in, Launch launch) {
  CHK(stage());
  constexpr int PIECE = (int)(STAGE_BYTES / 2 / 12);
  const int pieces = (n + PIECE - 1) / PIECE;
  const unsigned before = ticket_;  // piece c reports ticket before + 1 + c
  ticket_ += pieces;
  const auto count = [&](int c) { return std::min(PIECE, n - c * PIECE); };
  const auto half = [&](int c) { return (size_t)(c & 1) * (STAGE_BYTES / 2 / 4); };
  const auto start = [&](int c) {
    if (in) std::memcpy(h_stage_ + half(c), in + 3 * (size_t)c * PIECE, 12 * (size_t)count(c));
    launch(c * PIECE, count(c), stage_dev_ + half(c));
    launch_report_active(dref(), -1, report_dev_, before + 1 + c, stream);
  };
  for (int c = 0; c < std::min(pieces, 2); c++) start(c);
  for (int c = 0; c < pieces; c++) {
    unsigned none = 0;
    CHK(await(1, none, before + 1 + c, true));
    if (out) std::memcpy(out + 3 * (size_t)c * PIECE, h_stage_ + half(c), 12 * (size_t)count(c));
    if (c + 2 < pieces) start(c + 2);
  }
  return NN_OK;
}

int Batch::download(int k, int field, void* host, size_t bytes) {
  SceneHost& s = *scenes[k];
  const int w = field_width(field);
  if (w == 0) {
    set_error("unknown field");
    return NN_E_ARG;
  }
  const int n = s.n, pb = s.p_begin;
  if (bytes != (size_t)n * w * 4) {
    set_error("buffer size does not match n * width * 4");
    return NN_E_ARG;
  }
  (void)hipGetLastError();  // as in upload
  if (field == NN_FIELD_NUM_NEIGHBORS) CHK(complete_lists());
  // three-component fields: into original order by the kernel that writes them
  if (field == NN_FIELD_X || field == NN_FIELD_V || field == NN_FIELD_ACCELERATION || field == NN_FIELD_VISC_DIFF) {
    const float4* p = field == NN_FIELD_V ? d.vel : field == NN_FIELD_ACCELERATION ? d.acc : field == NN_FIELD_VISC_DIFF ? d.vdiff : d.pos;
    if (bytes <= STAGE_BYTES) {
      CHK(stage());
      launch_gather3(p + pb, d.inv + pb, n, stage_dev_, stream);
      launch_report_active(dref(), -1, report_dev_, ++ticket_, stream);
      unsigned none = 0;
      CHK(await(1, none));
      std::memcpy(host, h_stage_, bytes);
      return NN_OK;
    }
    return field_pieces(n, static_cast<float*>(host), nullptr,
                        [&](int at, int m, float* dev) { launch_gather3(p + pb, d.inv + pb + at, m, dev, stream); });
  }
  std::vector<int> info(n);
  HIPCHK(hipMemcpyAsync(info.data(), d.info + pb, sizeof(int) * n, hipMemcpyDeviceToHost, stream));
  float* out = (float*)host;
  int* iout = (int*)host;
  auto slot_f4 = [&](const float4* p, std::vector<float4>& v) -> hipError_t {
    v.resize(n);
    return hipMemcpyAsync(v.data(), p + pb, sizeof(float4) * n, hipMemcpyDeviceToHost, stream);
  };
  auto slot_f = [&](const float* p, std::vector<float>& v) -> hipError_t {
    v.resize(n);
    return hipMemcpyAsync(v.data(), p + pb, sizeof(float) * n, hipMemcpyDeviceToHost, stream);
  };
  // one component of the (src, alpha) pairs
  auto slot_sa = [&](int comp, std::vector<float>& v) -> hipError_t {
    std::vector<float2> t(n);
    hipError_t e = hipMemcpyAsync(t.data(), d.sa + pb, sizeof(float2) * n, hipMemcpyDeviceToHost, stream);
    if (e == hipSuccess) e = hipStreamSynchronize(stream);
    v.resize(n);
    for (int k = 0; k < n; k++) v[k] = comp ? t[k].y : t[k].x;
    return e;
  };
  std::vector<float4> f4;
  std::vector<float> f1;
  std::vector<int> i1;
  switch (field) {
    case NN_FIELD_VOLUME:
      HIPCHK(slot_f4(d.pos, f4));
      HIPCHK(hipStreamSynchronize(stream));
      for (int t = 0; t < n; t++) out[info[t] & 0x0FFFFFFF] = std::fabs(f4[t].w);
      return NN_OK;
    case NN_FIELD_X0:
    case NN_FIELD_REST_VOLUME: {
      f4.resize(n);
      HIPCHK(hipMemcpyAsync(f4.data(), d.x0 + pb, sizeof(float4) * n, hipMemcpyDeviceToHost, stream));
      HIPCHK(hipStreamSynchronize(stream));
      for (int id = 0; id < n; id++) {
        if (field == NN_FIELD_REST_VOLUME) out[id] = f4[id].w;
        else {
          out[3 * id] = f4[id].x;
          out[3 * id + 1] = f4[id].y;
          out[3 * id + 2] = f4[id].z;
        }
      }
      return NN_OK;
    }
    case NN_FIELD_DENSITY:
    case NN_FIELD_DFSPH_FACTOR:
    case NN_FIELD_DENSITY_ADV:
    case NN_FIELD_STRAIN_NORM:
    case NN_FIELD_VISCOSITY: {
      if (field == NN_FIELD_DFSPH_FACTOR || field == NN_FIELD_DENSITY_ADV) {
        HIPCHK(slot_sa(field == NN_FIELD_DFSPH_FACTOR ? 1 : 0, f1));
      } else {
        const float* p = field == NN_FIELD_DENSITY ? d.rho : field == NN_FIELD_STRAIN_NORM ? d.gam : d.eta;
        HIPCHK(slot_f(p, f1));
      }
      HIPCHK(hipStreamSynchronize(stream));
      const SceneDev& c = s.dev;
      for (int t = 0; t < n; t++) {
        const int id = info[t] & 0x0FFFFFFF;
        const bool fluid = (info[t] >> 28) == KIND_FLUID;
        float val = f1[t];
        if (field == NN_FIELD_DENSITY) val = (fluid && s.stepped) ? f1[t] : c.rho0;  // density.fill(density0), :744
        else if (!fluid || !s.stepped) val = 0.0f;
        else if (field == NN_FIELD_DFSPH_FACTOR) {
          // the value the reference holds after a step: alpha * 1/dt * dt * 1/dt^2 (:1688,1713,1771)
          val = (c.flags & SF_DIVERGENCE) ? ((f1[t] * c.inv_dt) * c.dt) * c.inv_dt2 : f1[t] * c.inv_dt2;
        }
        out[id] = val;
      }
      return NN_OK;
    }
    case NN_FIELD_KIND:
      HIPCHK(hipStreamSynchronize(stream));
      for (int t = 0; t < n; t++) iout[info[t] & 0x0FFFFFFF] = info[t] >> 28;
      for (int b = 0; b < s.nbody; b++)  // a rigid particle reads back as KIND_RIGID + its body
        for (int m = s.body_off[b]; m < s.body_off[b + 1]; m++) iout[s.body_ids[m]] = KIND_RIGID + b;
      return NN_OK;
    case NN_FIELD_NUM_NEIGHBORS: {
      i1.resize(n);
      HIPCHK(hipMemcpyAsync(i1.data(), d.nnbr + pb, sizeof(int) * n, hipMemcpyDeviceToHost, stream));
      HIPCHK(hipStreamSynchronize(stream));
      for (int t = 0; t < n; t++) iout[info[t] & 0x0FFFFFFF] = i1[t];
      return NN_OK;
    }
    case NN_FIELD_ROTATION:
    case NN_FIELD_STRESS: {
      HIPCHK(hipStreamSynchronize(stream));
      for (int id = 0; id < n; id++) {
        for (int a = 0; a < w; a++) out[(size_t)w * id + a] = (field == NN_FIELD_ROTATION && (a % 4) == 0) ? 1.0f : 0.0f;
      }
      if (s.ns > 0) {
        std::vector<float4> rs((size_t)4 * s.ns);
        HIPCHK(hipMemcpyAsync(rs.data(), d.rs + 4L * s.s_begin, sizeof(float4) * 4 * s.ns, hipMemcpyDeviceToHost, stream));
        HIPCHK(hipStreamSynchronize(stream));
        for (int q = 0; q < s.ns; q++) {
          const int id = s.s_pid[q];
          const float4* r = &rs[4 * (size_t)q];
          if (field == NN_FIELD_ROTATION) {
            const float R[9] = {r[0].x, r[0].y, r[0].z, r[1].x, r[1].y, r[1].z, r[2].x, r[2].y, r[2].z};
            if (s.stepped) std::memcpy(out + 9 * (size_t)id, R, sizeof(R));
          } else {
            const float S[6] = {r[0].w, r[1].w, r[2].w, r[3].x, r[3].y, r[3].z};
            if (s.stepped) std::memcpy(out + 6 * (size_t)id, S, sizeof(S));
          }
        }
      }
      return NN_OK;
    }
  }
  set_error("unknown field");
  return NN_E_ARG;
}

int Batch::upload_field(int k, int field, const void* host, size_t bytes) {
  SceneHost& s = *scenes[k];
  const int n = s.n, pb = s.p_begin;
  if ((field != NN_FIELD_X && field != NN_FIELD_V && field != NN_FIELD_VISC_DIFF) || bytes != (size_t)n * 12) {
    set_error("only x, v and the Weiler warm-start direction (float[n][3]) can be uploaded");
    return NN_E_ARG;
  }
  float4* p = field == NN_FIELD_X ? d.pos : field == NN_FIELD_V ? d.vel : d.vdiff;
  (void)hipGetLastError();  // as in upload
  if (bytes <= STAGE_BYTES) {
    CHK(stage());
    std::memcpy(h_stage_, host, bytes);
    launch_scatter3(stage_dev_, d.inv + pb, n, p + pb, stream);
    launch_report_active(dref(), -1, report_dev_, ++ticket_, stream);
    unsigned none = 0;
    return await(1, none);
  }
  return field_pieces(n, nullptr, static_cast<const float*>(host),
                      [&](int at, int m, float* dev) { launch_scatter3(dev, d.inv + pb + at, m, p + pb, stream); });
}

// After a step, the static particles' lists are built on demand, from the
// positions and cell order of that step's search (kept in pos_alt): the lists
// the reference holds after a step.  (A step of a batch with rigid bodies
// builds them in its search.)
int Batch::complete_lists() {
  if (lists_state_ == 2) return NN_OK;
  if (lists_state_ == 0) return search_impl(1, BEGIN_CELLS);  // laid out since: search the current positions
  Dev at_search = d;
  at_search.pos = d.pos_alt;
  launch_build_lists(DevRef{at_search}, blk(K_BUILD_LISTS), lanes(K_BUILD_LISTS), 1, stream);
  HIPCHK(hipGetLastError());
  lists_state_ = 2;
  return NN_OK;
}

int Batch::neighbors(int k, int* nbr, int* cnt, int cap) {
  CHK(complete_lists());
  SceneHost& s = *scenes[k];
  const int n = s.n, pb = s.p_begin;
  if (cap < MAX_NB) {
    set_error("cap must be at least 60");
    return NN_E_ARG;
  }
  std::vector<int> info(n), c(n), nb((size_t)n * MAX_NB);
  HIPCHK(hipMemcpyAsync(info.data(), d.info + pb, sizeof(int) * n, hipMemcpyDeviceToHost, stream));
  HIPCHK(hipMemcpyAsync(c.data(), d.nnbr + pb, sizeof(int) * n, hipMemcpyDeviceToHost, stream));
  HIPCHK(copy_lists(nb.data(), d, pb, n, stream));
  HIPCHK(hipStreamSynchronize(stream));
  CHK(lists_to_local(nb, c, pb, n));
  for (size_t t = 0; t < (size_t)n * cap; t++) nbr[t] = -1;
  for (int t = 0; t < n; t++) {
    const int id = info[t] & 0x0FFFFFFF;
    cnt[id] = c[t];
    for (int m = 0; m < c[t]; m++) nbr[(size_t)id * cap + m] = info[nb[host_nb(n, t, m)]] & 0x0FFFFFFF;
  }
  return NN_OK;
}

}  // namespace nn
