// Context, step orchestration and C ABI of the MI355X adaptive step.
#include <hip/hip_runtime.h>
#include <hip/hip_ext.h>

#include <algorithm>
#include <array>
#include <atomic>
#include <chrono>
#include <cstdlib>
#include <cmath>
#include <cstdio>
#include <cstring>
#include <map>
#include <memory>
#include <mutex>
#include <string>
#include <sys/stat.h>
#include <type_traits>
#include <vector>

#include "../../include/mwdg2.h"
#include "mw_input.hpp"
#include "mw_kernels.inc"
#include "mw_learn.inc"
#include "mw_batch.inc"

namespace mw {

namespace {

thread_local std::string g_err;

struct HipError : std::runtime_error {
  using std::runtime_error::runtime_error;
};

#define MW_HIP(x)                                                                              \
  do {                                                                                         \
    hipError_t e_ = (x);                                                                       \
    if (e_ != hipSuccess) throw ::mw::HipError(std::string(#x) + ": " + hipGetErrorString(e_));     \
  } while (0)

inline int nblk(long long n, int b = WG) { return (int)std::max(1LL, (n + b - 1) / b); }

template <typename T>
T* dalloc(size_t n) {
  void* p = nullptr;
  MW_HIP(hipMalloc(&p, std::max<size_t>(n, 1) * sizeof(T)));
  return static_cast<T*>(p);
}

// A device buffer for one call, freed on every exit path after the stream
// has drained.
template <typename T>
struct DevTmp {
  hipStream_t s;
  T* p;
  DevTmp(hipStream_t st, size_t n) : s(st), p(dalloc<T>(n)) {}
  ~DevTmp() {
    (void)hipStreamSynchronize(s);
    (void)hipFree(p);
  }
  DevTmp(const DevTmp&) = delete;
  DevTmp& operator=(const DevTmp&) = delete;
};

// Host restatement of the series cursor used once at set-up
// (PointSources constructor calls update_all_srcs(dt), PointSources.h:74).
template <typename real>
void advance_series_host(real t, int& row, const std::vector<real>& T, const std::vector<real>& V, real& out) {
  const int n = (int)T.size();
  if ((row - 1) < n && row + 1 < n) {
    real t_1 = T[row], t_2 = T[row + 1];
    if (t > t_2 && row + 2 < n) { row++; t_1 = T[row]; t_2 = T[row + 1]; }
    else if (t > t_2) { out = V[n - 1]; return; }
    const real i_1 = V[row], i_2 = V[row + 1];
    out = i_1 + (i_2 - i_1) / (t_2 - t_1) * (t - t_1);
  } else {
    out = V[n - 1];
  }
}

}  // namespace

struct CtxBase {
  virtual ~CtxBase() = default;
  // a number no other context of the process has (trace recordings tell
  // their contexts apart by it)
  const unsigned long long serial = next_serial();
  static unsigned long long next_serial() {
    static std::atomic<unsigned long long> n{0};
    return ++n;
  }
  int prec = 8;
  hipStream_t stream = nullptr;
  int profiling = 0;                // 0 off, 1 all kernels, 2 update kernels only
  struct Prof { long long n = 0; double ms = 0; };
  std::map<std::string, Prof> prof;
  std::vector<std::pair<std::string, std::pair<hipEvent_t, hipEvent_t>>> pending;
  std::vector<hipEvent_t> event_pool;

  hipEvent_t ev() {
    if (!event_pool.empty()) { hipEvent_t e = event_pool.back(); event_pool.pop_back(); return e; }
    hipEvent_t e;
    MW_HIP(hipEventCreate(&e));
    return e;
  }
  // Kernel launches go through launch_k: when a timed() section is open, the
  // dispatch itself records the section's start and stop events
  // (hipExtLaunchKernelGGL), so timing adds no packets between kernels.
  hipEvent_t ev_a = nullptr, ev_b = nullptr;
  template <typename... KArgs, typename... Args>
  void launch_k(void (*kernel)(KArgs...), dim3 grid, dim3 block, uint32_t shmem, hipStream_t s, Args... args) {
    if (ev_a) {
      hipExtLaunchKernelGGL(kernel, grid, block, shmem, s, ev_a, ev_b, 0, args...);
      ev_a = ev_b = nullptr;
    } else {
      hipLaunchKernelGGL(kernel, grid, block, shmem, s, args...);
    }
  }
  template <typename F>
  void timed(const char* name, F&& launch) {
    // mode 2 times the leaf kernels and the MRA band kernels
    const bool update = !std::strncmp(name, "stage", 5) || !std::strncmp(name, "fv1", 3) ||
                        !std::strncmp(name, "sweep", 5) || !std::strncmp(name, "wet", 3) ||
                        !std::strncmp(name, "emit_sweep", 10) || !std::strcmp(name, "emit_fv1") || !std::strcmp(name, "encode") ||
                        !std::strcmp(name, "decode") || !std::strcmp(name, "encode_scale") ||
                        !std::strcmp(name, "encode_scale_level") ||
                        !std::strcmp(name, "encode_level") || !std::strcmp(name, "decode_level");
    if (!profiling || (profiling == 2 && !update)) { launch(); return; }
    hipEvent_t a = ev(), b = ev();
    ev_a = a;
    ev_b = b;
    launch();
    if (ev_a) {                          // the section launched nothing
      MW_HIP(hipEventRecord(a, stream));
      MW_HIP(hipEventRecord(b, stream));
      ev_a = ev_b = nullptr;
    }
    pending.push_back({name, {a, b}});
  }
  // A section of several kernels, bracketed by event packets of its own.
  template <typename F>
  void timed_span(const char* name, F&& launch) {
    if (profiling != 1) { launch(); return; }
    hipEvent_t a = ev(), b = ev();
    MW_HIP(hipEventRecord(a, stream));
    launch();
    MW_HIP(hipEventRecord(b, stream));
    pending.push_back({name, {a, b}});
  }
  void drain_profile() {
    for (auto& p : pending) {
      MW_HIP(hipEventSynchronize(p.second.second));
      float ms = 0;
      MW_HIP(hipEventElapsedTime(&ms, p.second.first, p.second.second));
      Prof& q = prof[p.first];
      q.n++;
      q.ms += ms;
      event_pool.push_back(p.second.first);
      event_pool.push_back(p.second.second);
    }
    pending.clear();
  }

  virtual void step(int n) = 0;
  virtual void counters(mw_counters* c) = 0;
  virtual void stage(const std::string& s) = 0;
  virtual long long transfer(const std::string& name, void* host, long long count, bool up) = 0;
  virtual void set_scalar(const std::string& name, double v) = 0;
  virtual void set_initial(const void* const* modal) = 0;
  virtual void set_boundaries(const mw_boundary* b) = 0;
  virtual void set_sources(int n, const mw_point_source* s) = 0;
  virtual int stage_records(double* out, int max_rows, int* n_points) = 0;
  virtual const std::vector<int>& gauge_codes() const = 0;
  virtual void write_rasters(int index) = 0;
  virtual bool raster_due() = 0;
  virtual double dx() const = 0;
  virtual std::string out_path() const = 0;
  virtual bool voutput_stage() const = 0;
  virtual int cumulative_records(double* out, int max_rows) = 0;
  virtual void write_cumulative(const std::string& path) = 0;
  virtual std::string cumulative_path() const = 0;
  virtual void write_vtk(int index) = 0;
  virtual void write_c_prop() = 0;
  virtual void save_outputs(int index) = 0;
  virtual bool saveint_outputs() const = 0;
  // learned refinement
  virtual void set_learned(const MlpDev* w, int decide_every, int full_every, float threshold) = 0;
  virtual void set_trace(unsigned short* x, uint8_t* chg, int cap, int n0) = 0;
  virtual int trace_count() const = 0;
  virtual void learn_counters(long long* out) = 0;
  // ensembles
  virtual void set_sweep_groups(int g) = 0;
  virtual int sweep_groups() const = 0;
  virtual int default_sweep_groups() const = 0;
  virtual int tile_groups() const = 0;           // one work-group per 256-leaf tile of the finest level (capped)
  virtual void capture_step(hipGraph_t* g) = 0;
  virtual int parity() const = 0;
  virtual void set_parity(int c) = 0;
  virtual void check_graphable() const = 0;
  virtual void ensemble_step() = 0;               // one step of the captured sequence, launched directly
  // batched ensemble steps (mw_batch.inc)
  virtual bool batchable() const = 0;
  virtual size_t batch_args_size() const = 0;
  virtual void batch_args(void* out, int flip, BatchShape& shape) const = 0;
  virtual void batch_launch(const void* table, const BatchShape& shape, hipStream_t s) const = 0;
  virtual long long device_steps() = 0;           // steps the device has taken (drains the stream)
  virtual void resync(long long dev_steps) = 0;   // host step bookkeeping restarts from dev_steps
  bool in_ensemble = false;
  // Calls that change what an ensemble's captured steps use (buffers, grid
  // sizes, parameters, the state) are refused while the context is in one.
  void not_in_ensemble(const char* what) const {
    if (in_ensemble) throw std::logic_error(std::string(what) + ": the context belongs to an ensemble (destroy the ensemble first)");
  }
};

template <typename real>
struct Ctx : CtxBase {
  HostCase<real> hc;
  Params<real> P{};
  int L = 0, N = 0, D = 0, H = 0, md = 0;
  bool mwm = true;

  DevState<real>* st = nullptr;
  Hier<real> hier[2]{};        // MWDG2: [0] main (A), [1] stage buffer (B); HWFV1: ping-pong
  int main_h = 0;
  ZHier<real> zh{};
  uint8_t* sig[2] = {nullptr, nullptr};
  int cur = 0;
  uint8_t *xflag = nullptr, *leaflev = nullptr, *preflag = nullptr;
  int* leaf = nullptr;
  int* nbr[4] = {nullptr, nullptr, nullptr, nullptr};
  bool nbr_behind = false;                    // HWFV1: the last leaf list's neighbour lists are not written yet
  int* tile_sums = nullptr;
  int *rev_z = nullptr, *rev_rm = nullptr;
  real* uprev = nullptr;
  unsigned long long* maxh = nullptr;         // limiter: slots of the largest stage-1 depth (bit patterns), on list_n
  size_t Hp = 0;                              // node count rounded up to whole sibling groups
  real* xbuf = nullptr;                       // one coefficient as a plain array (parity transfers)
  real* red = nullptr;                        // [5][2 * leaf_grid()] next-step reduction slots
  WetList wet[2]{};                           // wet-leaf lists of the two MWDG2 stages
  int* list_n = nullptr;                      // their counters (with the limiter maxh), zeroed by each step's prologue
  int n_stage = 0;                            // gauges (stage points)
  int* stage_codes = nullptr;
  real* rec = nullptr;                        // stage-output rows: time, depths, elevations, velocities
  double* cum = nullptr;                      // cumulative rows: time, dt, leaves, mra ticks, ticks, step
  int rec_cap = 0;
  real* leafdt = nullptr;                     // per-leaf CFL time step (VTK output)
  real* lbuf = nullptr;                       // leaf-field staging for the leaf-list writers
  double* clk = nullptr;                      // k_clock output
  int cprop_writes = 0;
  std::vector<std::array<double, 6>> cprop_rows;   // cumulative rows written with the c-property files
  unsigned long long* cnt[3] = {nullptr, nullptr, nullptr};  // P_e, P_d, rescaled parents (slot arrays)
  // series and sources on the device
  int *s_off = nullptr, *s_len = nullptr;
  real *s_t = nullptr, *s_v = nullptr;
  int *src_code = nullptr, *src_type = nullptr, *src_row = nullptr;
  real* src_val = nullptr;
  int n_src = 0;
  bool issued_first = false;
  std::vector<void*> allocs;
  // learned refinement (MWDG2, eps > 0, level-6 units: 7 <= max_ref_lvl <= 12)
  bool learn = false;
  MlpDev lw{};
  int l_decide = 8, l_full = 32;
  float l_thr = 0.5f;
  long long lstep = 0, l_steps = 0;
  bool l_need = true;
  unsigned short* tr_x = nullptr;             // trace recording: features at each step's start
  uint8_t* tr_chg = nullptr;                  // ... and the step's per-unit tree change
  int tr_cap = 0, tr_n = 0;
  uint8_t *umode = nullptr, *uchg = nullptr;
  int* uage = nullptr;
  float* ustat = nullptr;
  unsigned short* ux = nullptr;
  unsigned long long* lcnt = nullptr;         // [2][CNT_SLOTS]: frozen unit-steps, parents kept (not reconstructed)
  uint8_t* dirty = nullptr;                   // parents whose children changed since their last encode
  uint8_t *uquiet = nullptr, *uwet = nullptr, *utouch = nullptr, *uborder = nullptr;
  bool quiet_off_pending = false;
  real* umx = nullptr;                        // [unit][4] maxima of a unit's leaves when last swept
  real* dm = nullptr;                         // [3][D] detail maxima of each parent's last encode
  unsigned short* lwb = nullptr;              // the network's BF16 weights (a copy)
  float* lwf = nullptr;                       // ... and its biases

  template <typename T>
  T* alloc(size_t n) {
    T* p = dalloc<T>(n);
    allocs.push_back(p);
    return p;
  }

  ~Ctx() override {
    if (stream) (void)hipStreamSynchronize(stream);
    for (void* p : allocs) (void)hipFree(p);
    for (auto& p : pending) { (void)hipEventDestroy(p.second.first); (void)hipEventDestroy(p.second.second); }
    for (hipEvent_t e : event_pool) (void)hipEventDestroy(e);
    if (stream) (void)hipStreamDestroy(stream);
  }

  Series<real> series() const { return {s_off, s_len, s_t, s_v}; }
  Sources<real> sources() const { return {n_src, src_code, src_type, src_val, src_row}; }
  LeafLists leaves() const {
    return {leaf, {nbr[0], nbr[1], nbr[2], nbr[3]}, &st->n_leaves, leaflev, {nbr[0], nbr[1], nbr[2], nbr[3]}};
  }

  void create(const mw_config& cfg) {
    prec = sizeof(real);
    read_case<real>(cfg.par_path, cfg.argc, cfg.argv, hc);
    L = hc.L;
    md = 1 << L;
    N = md * md;
    D = lvl_idx(L);
    H = lvl_idx(L + 1);
    mwm = hc.solver == MWDG2;
    MW_HIP(hipStreamCreateWithFlags(&stream, hipStreamNonBlocking));
    if (mwm && !hc.limitslopes) {
      int dev = 0, cus = 0, per_cu = 0;
      MW_HIP(hipGetDevice(&dev));
      MW_HIP(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
      MW_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, k_sweep2<real>, WG, 0));
      resident_g = std::min(RED_SLOTS, std::max(8, cus * per_cu / 8 * 8));
    }
    Hp = ((size_t)H + 3) / 4 * 4;
    for (int b = 0; b < 2; ++b) {
      hier[b].eta0 = alloc<real>(Hp);
      hier[b].rec = alloc<real>(Hp * (mwm ? REC_SLOTS<true> : REC_SLOTS<false>));
    }
    zh.z0 = alloc<real>(Hp);
    zh.rec = mwm ? alloc<real>(Hp * 2) : nullptr;
    xbuf = alloc<real>(Hp);
    clear_hierarchies();
    sig[0] = alloc<uint8_t>(D + 4);
    sig[1] = alloc<uint8_t>(D + 4);
    xflag = alloc<uint8_t>(D + 4);
    leaflev = alloc<uint8_t>(D + 4);
    preflag = alloc<uint8_t>(D + 4);
    for (uint8_t* p : {sig[0], sig[1], xflag, leaflev, preflag}) MW_HIP(hipMemsetAsync(p, 0, D + 4, stream));
    leaf = alloc<int>(N);
    for (int k = 0; k < 4; ++k) nbr[k] = alloc<int>(N);
    tile_sums = alloc<int>(nblk(std::max(1, N / 4), EMIT_TILE_MIN) + 4);   // read by fours
    st = alloc<DevState<real>>(1);
    red = alloc<real>((size_t)5 * 2 * RED_SLOTS);
    {
      // neutral slots (dt +inf, maxima 0): kernels that do not write a slot leave it neutral
      // layout [5][2 * leaf_grid()]: row 0 holds dt candidates, rows 1-4 maxima
      std::vector<real> init((size_t)5 * 2 * RED_SLOTS, real(0));
      for (int i = 0; i < 2 * leaf_grid(); ++i) init[i] = real(__builtin_inff());
      MW_HIP(hipMemcpyAsync(red, init.data(), sizeof(real) * init.size(), hipMemcpyHostToDevice, stream));
      MW_HIP(hipStreamSynchronize(stream));
    }
    if (mwm) alloc_wet_lists();
    for (int q = 0; q < 3; ++q) {
      cnt[q] = alloc<unsigned long long>(CNT_SLOTS);
      MW_HIP(hipMemsetAsync(cnt[q], 0, sizeof(unsigned long long) * CNT_SLOTS, stream));
    }
    if (hc.limitslopes && mwm) uprev = alloc<real>((size_t)9 * N);
    n_stage = (int)hc.stage_codes.size();
    if ((n_stage > 0 || hc.cumulative) && hc.massint_count0 == 0 && hc.massint > real(0)) {
      const double rows = std::floor((double)hc.sim_time / (double)hc.massint) + 3.0;
      rec_cap = (int)std::min(rows, (double)(1 << 20));
      if (n_stage > 0) {
        rec = alloc<real>((size_t)rec_cap * (1 + 4 * n_stage));
        stage_codes = alloc<int>(n_stage);
        MW_HIP(hipMemcpyAsync(stage_codes, hc.stage_codes.data(), sizeof(int) * n_stage, hipMemcpyHostToDevice,
                              stream));
      }
      if (hc.cumulative) cum = alloc<double>((size_t)rec_cap * 6);
    }
    fill_params();
    if (hc.vtk) {
      leafdt = alloc<real>(N);
      P.leaf_dt = leafdt;
    }
    upload_sources_and_series();
    build_initial();
  }

  void clear_hierarchies() {
    const size_t rs = mwm ? REC_SLOTS<true> : REC_SLOTS<false>;
    for (int b = 0; b < 2; ++b) {
      MW_HIP(hipMemsetAsync(hier[b].eta0, 0, sizeof(real) * Hp, stream));
      MW_HIP(hipMemsetAsync(hier[b].rec, 0, sizeof(real) * Hp * rs, stream));
    }
    MW_HIP(hipMemsetAsync(zh.z0, 0, sizeof(real) * Hp, stream));
    if (zh.rec) MW_HIP(hipMemsetAsync(zh.rec, 0, sizeof(real) * Hp * 2, stream));
  }

  void fill_params() {
    P.L = L; P.N = N; P.D = D; P.H = H; P.mesh_dim = md; P.xsz = hc.xsz; P.ysz = hc.ysz;
    if (umode) set_quiet_params();
    P.solver = hc.solver;
    P.eps = hc.epsilon; P.dx = hc.dx; P.g = hc.g;
    P.tol_h = real(1e-3); P.tol_q = real(0.0); P.tol_s = real(1e-9);   // classes/SolverParams.h:23-25
    P.manning = hc.manning; P.initial_tstep = hc.initial_tstep; P.wall_height = hc.wall_height;
    P.CFL = hc.CFL; P.tol_Krivo = hc.tol_Krivo;
    P.eps_extra_factor = std::pow(real(2.0), real(1.5) + 1);          // extra_significance_kernel.cu:23
    P.limitslopes = hc.limitslopes ? 1 : 0;
    P.monai = hc.monai ? 1 : 0;
    P.oregon = hc.oregon ? 1 : 0;
    P.test_case = hc.test_case;
    {
      const int tc = hc.test_case;
      P.flow = (tc >= 1 && tc <= 18) ? ((tc % 2 == 1) ? FLOW_EW : FLOW_NS) : FLOW_NONE;
    }
    P.massint = hc.massint;
    for (int k = 0; k < 4; ++k) { P.btype[k] = hc.bdy[k].type; P.bstart[k] = hc.bdy[k].start; P.bend[k] = hc.bdy[k].end; }
  }

  void upload_sources_and_series() {
    n_src = (int)hc.srcs.size();
    if (n_src > MAX_SRC) throw InputError("too many point sources");
    for (void* p : {(void*)s_off, (void*)s_len, (void*)s_t, (void*)s_v, (void*)src_code, (void*)src_type,
                    (void*)src_row, (void*)src_val})
      release(p);
    std::vector<int> off, len;
    std::vector<real> tt, vv;
    auto add = [&](const HostSeries<real>& s) {
      off.push_back((int)tt.size());
      len.push_back((int)s.t.size());
      tt.insert(tt.end(), s.t.begin(), s.t.end());
      vv.insert(vv.end(), s.v.begin(), s.v.end());
    };
    for (int k = 0; k < 4; ++k) add(hc.bdy[k].series);
    for (auto& s : hc.srcs) add(s.series);
    s_off = alloc<int>(off.size());
    s_len = alloc<int>(len.size());
    s_t = alloc<real>(tt.size() + 1);
    s_v = alloc<real>(vv.size() + 1);
    MW_HIP(hipMemcpy(s_off, off.data(), off.size() * sizeof(int), hipMemcpyHostToDevice));
    MW_HIP(hipMemcpy(s_len, len.data(), len.size() * sizeof(int), hipMemcpyHostToDevice));
    if (!tt.empty()) {
      MW_HIP(hipMemcpy(s_t, tt.data(), tt.size() * sizeof(real), hipMemcpyHostToDevice));
      MW_HIP(hipMemcpy(s_v, vv.data(), vv.size() * sizeof(real), hipMemcpyHostToDevice));
    }
    std::vector<int> code(n_src + 1), type(n_src + 1), row(n_src + 1, 0);
    std::vector<real> val(n_src + 1, real(0));
    for (int s = 0; s < n_src; ++s) {
      code[s] = hc.srcs[s].code;
      type[s] = hc.srcs[s].type;
      val[s] = hc.srcs[s].value;
      if (type[s] == HVAR || type[s] == QVAR)             // PointSources.h:74, update_all_srcs(dt)
        advance_series_host<real>(real(0.001), row[s], hc.srcs[s].series.t, hc.srcs[s].series.v, val[s]);
    }
    src_code = alloc<int>(n_src + 1);
    src_type = alloc<int>(n_src + 1);
    src_row = alloc<int>(n_src + 1);
    src_val = alloc<real>(n_src + 1);
    MW_HIP(hipMemcpy(src_code, code.data(), code.size() * sizeof(int), hipMemcpyHostToDevice));
    MW_HIP(hipMemcpy(src_type, type.data(), type.size() * sizeof(int), hipMemcpyHostToDevice));
    MW_HIP(hipMemcpy(src_row, row.data(), row.size() * sizeof(int), hipMemcpyHostToDevice));
    MW_HIP(hipMemcpy(src_val, val.data(), val.size() * sizeof(real), hipMemcpyHostToDevice));
  }

  // generate_all_morton_codes.cu:3-20 + get_sorting_indices.cu:3-62:
  // rev_z_order[m] = row-major index of the cell with Morton code m (a sort
  // of (code, index) pairs), rev_row_major its inverse (a sort of
  // (rev_z_order, index) pairs). Both key sets are below 4^L, so the sorts
  // take ceil(2L / 8) digit passes. Built on first use: only row-major
  // initial values (mw_set_initial) and the named downloads need them.
  bool zorder_ready = false;
  void zorder_build() {
    if (!rev_z) {
      rev_z = alloc<int>(N);
      rev_rm = alloc<int>(N);
    }
    DevTmp<int> codes(stream, N), idx(stream, N), k1(stream, N), tk(stream, N), tv(stream, N);
    DevTmp<int> cnt(stream, sort_table(N)), off(stream, sort_table(N)), sums(stream, sort_chunks(N));
    const SortScratch S{tk.p, tv.p, cnt.p, off.p, sums.p};
    const int passes = (2 * L + 7) / 8;
    launch_k(k_iota_morton, dim3(nblk(N)), dim3(WG), 0, stream, codes.p, idx.p, md, N);
    timed_span("zorder_sort", [&] { radix_sort_pairs(N, codes.p, idx.p, k1.p, rev_z, S, passes, stream); });
    launch_k(k_iota_morton, dim3(nblk(N)), dim3(WG), 0, stream, codes.p, idx.p, md, N);  // idx = iota again
    timed_span("zorder_sort", [&] { radix_sort_pairs(N, rev_z, idx.p, k1.p, rev_rm, S, passes, stream); });
    MW_HIP(hipGetLastError());
    MW_HIP(hipStreamSynchronize(stream));
    zorder_ready = true;
  }
  void ensure_zorder() {
    if (!zorder_ready) zorder_build();
  }

  void build_initial() {
    // finest level of A and Zh, and each cell's depth for the maxima
    real* h0 = dalloc<real>(N);
    if (!hc.modal[0].empty()) {
      ensure_zorder();
      // row-major modal values given through mw_set_initial -> Z order
      // (zorder/sort_finest_scale_coeffs_z_order.cu, copy_finest_coefficients.cu)
      std::vector<real*> dm(12, nullptr);
      for (int v = 0; v < 12; ++v)
        if (!hc.modal[v].empty()) {
          dm[v] = dalloc<real>(N);
          MW_HIP(hipMemcpyAsync(dm[v], hc.modal[v].data(), sizeof(real) * N, hipMemcpyHostToDevice, stream));
        }
      real** dtab = dalloc<real*>(12);
      MW_HIP(hipMemcpyAsync(dtab, dm.data(), sizeof(real*) * 12, hipMemcpyHostToDevice, stream));
      if (mwm)
        launch_k((k_set_finest<real, true>), dim3(nblk(N)), dim3(WG), 0, stream, (const real* const*)dtab,
                           rev_z, hier[0], zh, L, N, h0);
      else
        launch_k((k_set_finest<real, false>), dim3(nblk(N)), dim3(WG), 0, stream,
                           (const real* const*)dtab, rev_z, hier[0], zh, L, N, h0);
      MW_HIP(hipGetLastError());
      MW_HIP(hipStreamSynchronize(stream));
      for (real* p : dm) if (p) (void)hipFree(p);
      (void)hipFree(dtab);
    } else {
      // rasters (or a synthetic case) -> nodes -> modes, on the device
      InitSrc<real> S{};
      std::vector<real*> dr;
      for (int v = 0; v < 4; ++v) {
        S.r[v] = nullptr;
        if (hc.raster[v].empty()) continue;
        real* d = dalloc<real>(N);
        MW_HIP(hipMemcpyAsync(d, hc.raster[v].data(), sizeof(real) * N, hipMemcpyHostToDevice, stream));
        S.r[v] = d;
        dr.push_back(d);
      }
      if (hc.test_case == 0 && (!S.r[0] || !S.r[3])) throw InputError("no initial rasters (mw_set_initial not called)");
      S.xsz = hc.xsz; S.ysz = hc.ysz; S.test_case = hc.test_case;
      S.xmin = hc.xmin; S.ymin = hc.ymin; S.dx = hc.dx; S.hl = hc.syn_hl; S.hr = hc.syn_hr;
      S.s3 = std::sqrt(real(3.0));
      if (mwm)
        launch_k((k_init_cells<real, true>), dim3(nblk(N)), dim3(WG), 0, stream, S, hier[0], zh, L, h0);
      else
        launch_k((k_init_cells<real, false>), dim3(nblk(N)), dim3(WG), 0, stream, S, hier[0], zh, L, h0);
      MW_HIP(hipGetLastError());
      MW_HIP(hipStreamSynchronize(stream));
      for (real* p : dr) (void)hipFree(p);
    }

    // preflags from gauges, boundaries, sources, walls (mra/preflag_details.cu:15-92)
    {
      std::vector<int> codes(hc.stage_codes.begin(), hc.stage_codes.end());
      for (int k = 0; k < 4; ++k) codes.insert(codes.end(), hc.bdy[k].codes.begin(), hc.bdy[k].codes.end());
      for (auto& sr : hc.srcs) codes.push_back(sr.code);
      const int thick = hc.refine_wall ? hc.ref_thickness : 0;
      const long long work = (long long)codes.size() + (long long)thick * (hc.xsz + hc.ysz);
      int* dcodes = dalloc<int>(codes.size() + 1);
      if (!codes.empty())
        MW_HIP(hipMemcpyAsync(dcodes, codes.data(), sizeof(int) * codes.size(), hipMemcpyHostToDevice, stream));
      MW_HIP(hipMemsetAsync(preflag, 0, D + 4, stream));
      if (work > 0)
        launch_k(k_preflag_init, dim3(nblk(work)), dim3(WG), 0, stream, preflag, dcodes, (int)codes.size(), L,
                           thick, hc.xsz, hc.ysz);
      MW_HIP(hipGetLastError());
      MW_HIP(hipStreamSynchronize(stream));
      (void)hipFree(dcodes);
    }

    DevState<real> s{};
    s.time = real(0);
    s.dt = real(0.001);                                      // run_simulation.cu:37
    s.sim_time = hc.sim_time;
    s.n_leaves = N;
    s.done = 0;
    s.first = 1;
    s.steps = 0;
    for (int k = 0; k < 4; ++k) { s.inlet[k] = hc.bdy[k].inlet; s.row[k] = 0; }
    s.n_src = n_src;
    s.save_count = hc.massint_count0;
    s.n_records = 0;
    s.nonfinite = 0;
    MW_HIP(hipMemcpyAsync(st, &s, sizeof s, hipMemcpyHostToDevice, stream));

    // maxima of the initial assembled solution with the point sources
    // inserted (mra/insert_point_srcs.cu:3-29, get_max_scale_coeffs.cu)
    {
      const int nparts = std::min(nblk(N), 1024);
      real* part = dalloc<real>((size_t)4 * nparts);
      if (mwm)
        launch_k((k_init_maxima<real, true>), dim3(nparts), dim3(WG), 0, stream, h0, hier[0], zh, L,
                           sources(), real(0.001), hc.dx, part);
      else
        launch_k((k_init_maxima<real, false>), dim3(nparts), dim3(WG), 0, stream, h0, hier[0], zh, L,
                           sources(), real(0.001), hc.dx, part);
      launch_k((k_init_maxima_final<real>), dim3(1), dim3(64), 0, stream, st, part, nparts);
      MW_HIP(hipGetLastError());
      MW_HIP(hipStreamSynchronize(stream));
      (void)hipFree(part);
    }
    (void)hipFree(h0);

    // z hierarchy and topography preflags (mra/preflag_topo.cu:3-43)
    for (int level = L - 1; level >= 0; --level) {
      if (mwm)
        launch_k((k_z_encode<real, true>), dim3(nblk(1LL << (2 * level))), dim3(WG), 0, stream, zh, preflag,
                           level, L, hc.epsilon, (const DevState<real>*)st);
      else
        launch_k((k_z_encode<real, false>), dim3(nblk(1LL << (2 * level))), dim3(WG), 0, stream, zh, preflag,
                           level, L, hc.epsilon, (const DevState<real>*)st);
    }
    MW_HIP(hipGetLastError());
    // all parents significant before the first encode (mra/init_sig_details.cu)
    cur = 0;
    MW_HIP(hipMemsetAsync(sig[cur], 1, D + 4, stream));
    MW_HIP(hipStreamSynchronize(stream));
    main_h = 0;
    issued_first = false;
    issued_since_sync = 0;
    dev_steps_at_sync = 0;
  }

  // ---- step pieces ---------------------------------------------------------
  // with_sources: the prologue also applies the point sources (a step's
  // prologue; the single-stage calls launch k_point_sources on their own)
  // A step's prologue also zeroes the emission tiles' leaf counts, which the
  // decode of level L-1 adds up (counts_tiles).
  void k_prologue_launch(bool with_sources = false) {
    const bool zero = with_sources && counts_tiles();
    timed("prologue", [&] {
      launch_k((k_prologue<real>), dim3(1), dim3(PRO_WG), 0, stream, st, P, series(), sources(), red,
               2 * leaf_grid(), (with_sources && n_src) ? 1 : 0, hier[main_h], P.dirty,
               zero ? tile_sums : (int*)nullptr, zero ? emit_tiles() : 0, list_n);
    });
  }
  void k_sources_launch() {
    if (!n_src) return;
    timed("point_sources", [&] {
      launch_k((k_point_sources<real>), dim3(nblk(n_src)), dim3(WG), 0, stream, st, hier[main_h], sources(), L, hc.dx,
               P.dirty);
    });
  }
  // Levels of the encode, the decode and the stage-1 re-encode. From level 10 (4^10 nodes) on each level
  // is a flat launch, one node per thread: there a level fills the chip, and
  // a band's chain of barriers would hold most of its threads idle. Below,
  // levels mra_lo .. mra_hi are one band launch whose work-groups have at most
  // 256 nodes of the deepest level, one per thread, and levels 0 .. mra_top
  // (at most 4: 341 nodes) one work-group. max_ref_lvl 12: flat 11 and 10,
  // band 5-9, top 0-4; 10: band 5-9; 8: band 3-7, top 0-2. The learned step
  // has its own encode and decode kernels from level 6 on.
  struct Levels {
    int lo, hi, top;
    bool band() const { return lo <= hi; }
  };
  Levels levels(int deepest) const {
    const int hi = std::min(deepest, MRA_FLAT - 1), lo = std::max(hi - (MRA_BAND - 1), 3);
    return {lo, hi, std::min(lo - 1, L - 1)};
  }
  int mra_hi() const { return levels(lrn() ? UNIT_LEVEL - 1 : L - 1).hi; }
  int mra_lo() const { return levels(lrn() ? UNIT_LEVEL - 1 : L - 1).lo; }
  int mra_top() const { return levels(lrn() ? UNIT_LEVEL - 1 : L - 1).top; }
  bool mra_band() const { return mra_lo() <= mra_hi(); }
  bool counts_tiles() const { return !lrn() && mra_band(); }
  void encode_launch(bool skip_top = false) {
    uint8_t* prev = sig[cur];
    uint8_t* nw = sig[cur ^ 1];
    if (lrn()) {
      timed("encode", [&] {
        const int full = l_full_step() ? 1 : 0;
        uint8_t* ut = P.uquiet ? utouch : nullptr;
        if (l_stats())
          launch_k((k_encode_band_learn<real, true>), dim3(N_UNITS), dim3(WG), 0, stream, st, hier[main_h], prev, nw,
                   xflag, preflag, UNIT_LEVEL, L - 1, L, hc.epsilon, P.eps_extra_factor, cnt[0], ustat, P.dirty, dm,
                   D, full, ut);
        else
          launch_k((k_encode_band_learn<real, false>), dim3(N_UNITS), dim3(WG), 0, stream, st, hier[main_h], prev,
                   nw, xflag, preflag, UNIT_LEVEL, L - 1, L, hc.epsilon, P.eps_extra_factor, cnt[0], ustat, P.dirty,
                   dm, D, full, ut);
      });
    } else {
      for (int level = L - 1; level > mra_hi(); --level) {
        const int g = 1 << (2 * level);
        timed("encode_level", [&] {
          if (mwm)
            launch_k((k_encode_level<real, true>), dim3(g / WG), dim3(WG), 0, stream, st, hier[main_h], prev, nw,
                     xflag, preflag, level, L, hc.epsilon, P.eps_extra_factor, cnt[0]);
          else
            launch_k((k_encode_level<real, false>), dim3(g / WG), dim3(WG), 0, stream, st, hier[main_h], prev, nw,
                     xflag, preflag, level, L, hc.epsilon, P.eps_extra_factor, cnt[0]);
        });
      }
    }
    if (mra_band())
      timed(lrn() ? "encode_coarse" : "encode", [&] {
        const int nwg = 1 << (2 * mra_lo());
        if (mwm)
          launch_k((k_encode_band<real, true>), dim3(nwg), dim3(WG), 0, stream, st, hier[main_h], prev, nw,
                             xflag, preflag, mra_lo(), mra_hi(), L, hc.epsilon, P.eps_extra_factor, cnt[0]);
        else
          launch_k((k_encode_band<real, false>), dim3(nwg), dim3(WG), 0, stream, st, hier[main_h], prev, nw,
                             xflag, preflag, mra_lo(), mra_hi(), L, hc.epsilon, P.eps_extra_factor, cnt[0]);
      });
    if (!skip_top) top_launch(1);
  }
  // the coarse levels: mode 1 encode, 2 decode, 3 both
  void top_launch(int mode) {
    uint8_t* prev = sig[cur];
    uint8_t* nw = sig[cur ^ 1];
    timed("top_mra", [&] {
      const dim3 wg(top_threads(mra_top()));
      if (mwm)
        launch_k((k_top_mra<real, true>), dim3(1), wg, 0, stream, st, hier[main_h], (const uint8_t*)prev, nw, xflag,
                 (const uint8_t*)preflag, leaflev, mra_top(), L, hc.epsilon, P.eps_extra_factor, cnt[0], cnt[1], mode);
      else
        launch_k((k_top_mra<real, false>), dim3(1), wg, 0, stream, st, hier[main_h], (const uint8_t*)prev, nw, xflag,
                 (const uint8_t*)preflag, leaflev, mra_top(), L, hc.epsilon, P.eps_extra_factor, cnt[0], cnt[1], mode);
    });
  }
  // HWFV1's whole encode and decode in one work-group
  bool hw_tree() const { return !mwm && !lrn() && mra_band() && L <= HW_TREE_LEVELS; }
  void hw_tree_launch() {
    timed("hw_tree", [&] {
      launch_k((k_hw_tree<real>), dim3(1), dim3(1 << (2 * (L - 1))), 0, stream, st, hier[main_h],
               (const uint8_t*)sig[cur], sig[cur ^ 1], xflag, (const uint8_t*)preflag, leaflev, L, hc.epsilon,
               P.eps_extra_factor, cnt[0], cnt[1], tile_sums, emit_tile());
    });
  }
  // Returns true when the decode of level L-1 also added up the emission
  // tiles' leaf counts (count_tiles: the step's prologue zeroed them).
  bool decode_launch(bool with_encode = false, bool count_tiles = false) {
    uint8_t* prev = sig[cur];
    uint8_t* nw = sig[cur ^ 1];
    top_launch(with_encode ? 3 : 2);
    const bool counted = count_tiles && counts_tiles();
    int* tz = counted ? tile_sums : nullptr;
    if (mra_band())
      timed(lrn() ? "decode_coarse" : "decode", [&] {
        const int nwg = 1 << (2 * mra_lo());
        if (mwm)
          launch_k((k_topdown_band<real, true>), dim3(nwg), dim3(WG), 0, stream, st, hier[main_h], prev, nw,
                   xflag, leaflev, mra_lo(), mra_hi(), L, hc.epsilon, P.eps_extra_factor, cnt[1], tz, emit_tile());
        else
          launch_k((k_topdown_band<real, false>), dim3(nwg), dim3(WG), 0, stream, st, hier[main_h], prev, nw,
                   xflag, leaflev, mra_lo(), mra_hi(), L, hc.epsilon, P.eps_extra_factor, cnt[1], tz, emit_tile());
      });
    if (lrn()) {
      timed("decode", [&] {
        launch_k((k_topdown_band_learn<real>), dim3(N_UNITS), dim3(WG), 0, stream, st, hier[main_h], prev, nw,
                 (const uint8_t*)xflag, leaflev, UNIT_LEVEL, L - 1, L, hc.epsilon, P.eps_extra_factor, cnt[1],
                 (const uint8_t*)umode, lcnt, uchg, uage,
                 tr_x ? tr_chg + (size_t)tr_n * N_UNITS : (uint8_t*)nullptr, P.dirty,
                 P.uquiet ? utouch : (uint8_t*)nullptr);
      });
      return false;
    }
    for (int level = mra_hi() + 1; level < L; ++level) {
      const int g = 1 << (2 * level);
      int* t = level == L - 1 ? tz : nullptr;
      timed("decode_level", [&] {
        if (mwm)
          launch_k((k_topdown_level<real, true>), dim3(g / WG), dim3(WG), 0, stream, st, hier[main_h], prev, nw,
                   xflag, leaflev, level, L, hc.epsilon, P.eps_extra_factor, cnt[1], t, emit_tile());
        else
          launch_k((k_topdown_level<real, false>), dim3(g / WG), dim3(WG), 0, stream, st, hier[main_h], prev, nw,
                   xflag, leaflev, level, L, hc.epsilon, P.eps_extra_factor, cnt[1], t, emit_tile());
      });
    }
    return counted;
  }
  // Nodes per emission tile: small grids need small tiles to have a
  // work-group for every CU, large ones keep more of their neighbours inside
  // a tile. us per launch with 64 / 256 / 1024 nodes: dam break 256^2 FP64
  // 8.5 / 15 / 37, valley 1024^2 FP32 28 / 23 / 44, HWFV1 2048^2 (emit_write)
  // 11 / 10 / 16, urban 4096^2 FP32 329 / 161 / 156 (with 64 or 256 nodes that
  // grid has more than EMIT_SELF_SCAN tiles, whose counts take a single-group
  // scan of some 24 us first). The learned step's tiles hold whole level-6
  // units (one from max_ref_lvl 10 on).
  int emit_tile() const {
    const int t = L <= 9 ? 64 : (L <= 11 ? 256 : 1024);
    return umode && L >= 10 ? 1 << (2 * (L - 1 - UNIT_LEVEL)) : t;
  }
  int emit_tiles() const { return nblk(1 << (2 * (L - 1)), emit_tile()); }
  // f with the tile's node count as a constant
  template <typename F>
  void with_tile(F&& f) const {
    switch (emit_tile()) {
      case 64: f(std::integral_constant<int, 64>{}); break;
      case 256: f(std::integral_constant<int, 256>{}); break;
      default: f(std::integral_constant<int, 1024>{}); break;
    }
  }
  EmitScan emit_scan_args(bool scanned) const {
    return {tile_sums, scanned ? 1 : 0, &st->n_leaves, &st->clk_step, &st->mra_ticks};
  }
  bool fuse_sweep1() const { return mwm && !hc.limitslopes; }
  // HWFV1: the whole update in the leaf emission. Not with epsilon = 0, whose
  // later steps read the neighbour lists of the one emission.
  bool fuse_fv1() const { return !mwm && hc.epsilon > real(0) && emit_tile() == EMIT_TILE_MIN; }
  // Leaf emission; with `sweep` (MWDG2 without limiter) the stage-1 sweep of
  // the emitted leaves runs in the same kernel.
  // counted: the decode wrote the tiles' leaf counts already
  void emit_launch(bool sweep = false, bool counted = false) {
    const int Q = 1 << (2 * (L - 1));
    const int tiles = emit_tiles();
    int* done = &st->done;
    int* nl = &st->n_leaves;
    if (!counted)
      timed("emit_count", [&] {
        with_tile([&](auto T) {
          launch_k(k_emit_count<T.value>, dim3(tiles), dim3(WG), 0, stream, done, leaflev, L, Q, tile_sums);
        });
      });
    const bool scanned = tiles > EMIT_SELF_SCAN;
    const EmitScan E = emit_scan_args(scanned);
    if (scanned)
      timed("emit_scan", [&] { launch_k(k_emit_scan, dim3(1), dim3(1024), 0, stream, done, nl, tile_sums, tiles,
                                                  &st->clk_step, &st->mra_ticks); });
    if (sweep && !mwm) {
      timed("emit_fv1", [&] {
        launch_k((k_emit_fv1<real>), dim3(tiles), dim3(WG), 0, stream, st, P, leaflev, Q, E, leaf, hier[main_h],
                 hier[main_h ^ 1], zh, red, 2 * leaf_grid());
      });
      main_h ^= 1;
      return;
    }
    if (sweep) {
      timed("emit_sweep1", [&] {
        with_tile([&](auto T) {
          launch_k((k_emit_sweep1<real, T.value>), dim3(tiles), dim3(WG), 0, stream, st, P, leaflev, Q, E,
                   leaf, nbr[0], nbr[1], nbr[2], nbr[3], hier[main_h], hier[main_h ^ 1], zh, wet[0]);
        });
      });
      return;
    }
    timed("emit_write", [&] {
      with_tile([&](auto T) {
        launch_k(k_emit_write<T.value>, dim3(tiles), dim3(WG), 0, stream, done, leaflev, L, Q, E, leaf,
                 nbr[0], nbr[1], nbr[2], nbr[3], md, hc.xsz, hc.ysz);
      });
    });
  }
  int sweep_g = 0;                            // work-groups of the leaf sweeps (0: the default)
  // The leaf sweeps loop over tiles, so their work-group count is free. The
  // default is one resident round of the MWDG2 stage-2 sweep (CUs x its
  // occupancy, a multiple of 8): a count between one and two rounds leaves a
  // tail (urban 4096^2, FP32: 2048 groups 236 us, 1536 groups 200 us, 4096
  // groups 208 us per launch).
  int resident_g = 0;
  int tile_groups() const override { return std::min((nblk(N) + 7) / 8 * 8, RED_SLOTS); }
  int default_sweep_groups() const override {
    const int g = tile_groups();
    return resident_g ? std::min(g, resident_g) : g;
  }
  int leaf_grid() const { return sweep_g ? sweep_g : default_sweep_groups(); }
  int sweep_groups() const override { return leaf_grid(); }
  // The sweeps' work-group count (a multiple of 8, 8 .. 4096). The per-group
  // reduction slots of the last step are folded into the new layout; results
  // do not depend on it (exact min/max reductions, per-leaf updates).
  void set_sweep_groups(int g) override {
    not_in_ensemble("set_sweep_groups");
    if (!mwm || hc.limitslopes) throw std::invalid_argument("sweep groups apply to the MWDG2 sweeps without limiter");
    if (g < 8 || g > RED_SLOTS || g % 8) throw std::invalid_argument("sweep groups must be a multiple of 8 in [8, 4096]");
    MW_HIP(hipStreamSynchronize(stream));
    const int g0 = leaf_grid();
    std::vector<real> old((size_t)5 * 2 * g0);
    MW_HIP(hipMemcpy(old.data(), red, sizeof(real) * old.size(), hipMemcpyDeviceToHost));
    std::vector<real> nw((size_t)5 * 2 * RED_SLOTS, real(0));
    for (int i = 0; i < 2 * g; ++i) nw[i] = real(__builtin_inff());
    for (int r = 0; r < 5; ++r) {
      real v = old[(size_t)r * 2 * g0];
      for (int i = 1; i < 2 * g0; ++i) {
        const real x = old[(size_t)r * 2 * g0 + i];
        v = (r == 0) ? std::min(v, x) : std::max(v, x);
      }
      nw[(size_t)r * 2 * g] = v;
    }
    MW_HIP(hipMemcpy(red, nw.data(), sizeof(real) * nw.size(), hipMemcpyHostToDevice));
    sweep_g = g;
    MW_HIP(hipStreamSynchronize(stream));
  }
  void release(void* p) {
    if (!p) return;
    allocs.erase(std::remove(allocs.begin(), allocs.end(), p), allocs.end());
    (void)hipFree(p);
  }
  // The wet lists: a region holds the leaves of its share of the emission's
  // tiles (of any tile size) or of the sweeps' (256 leaves). Small grids, with
  // few appends, have 8 regions.
  static constexpr int LIST_INTS = 2 * LIST_REGIONS * LIST_PAD;
  void alloc_wet_lists() {
    list_n = alloc<int>(LIST_INTS);
    MW_HIP(hipMemsetAsync(list_n, 0, sizeof(int) * LIST_INTS, stream));
    if (hc.limitslopes) {                           // no wet lists
      maxh = reinterpret_cast<unsigned long long*>(list_n);
      return;
    }
    const int R = L <= 9 ? 8 : LIST_REGIONS;
    long long cap = 0;
    for (int t : {EMIT_TILE_MIN, 256, EMIT_TILE_MAX})             // the smallest hold 256 leaves, as the sweeps'
      cap = std::max(cap, (long long)nblk(nblk(std::max(1, N / 4), t), R) * 4 * t);
    for (int q = 0; q < 2; ++q)
      wet[q] = {alloc<int>((size_t)R * cap), list_n + q * LIST_REGIONS * LIST_PAD, &st->wet_sum[q], (int)cap, R};
  }
  // a single stage run without the prologue starts its wet list afresh
  void reset_wet_list(int q) {
    if (mwm && !hc.limitslopes) MW_HIP(hipMemsetAsync(wet[q].n, 0, sizeof(int) * LIST_REGIONS * LIST_PAD, stream));
  }
  void check_graphable() const override {
    if (!mwm || hc.limitslopes) throw std::invalid_argument("ensembles run the MWDG2 step without limiter");
    if (learn || tr_x) throw std::invalid_argument("ensembles run the plain step (no learned mode or trace)");
    if (profiling) throw std::invalid_argument("ensembles need kernel profiling off");
  }
  // One step recorded into a graph (nothing runs). The step flips the mask
  // buffers when it rebuilds the tree, so an ensemble records two
  // consecutive steps and replays them alternately.
  void capture_step(hipGraph_t* g) override {
    check_graphable();
    MW_HIP(hipStreamSynchronize(stream));
    MW_HIP(hipStreamBeginCapture(stream, hipStreamCaptureModeThreadLocal));
    try {
      one_step();
    } catch (...) {
      hipGraph_t tmp = nullptr;
      (void)hipStreamEndCapture(stream, &tmp);
      if (tmp) (void)hipGraphDestroy(tmp);
      throw;
    }
    MW_HIP(hipStreamEndCapture(stream, g));
  }
  int parity() const override { return cur; }
  void set_parity(int c) override { cur = c; }
  // swept: the stage-1 sweep already ran inside the leaf emission
  void stage1_launch(bool swept = false) {
    const int other = main_h ^ 1;
    const int G = leaf_grid();
    if (mwm && !hc.limitslopes) {
      if (!swept) {
        timed("sweep1", [&] {
          launch_k((k_sweep1<real>), dim3(G), dim3(WG), 0, stream, st, P, leaves(), hier[main_h], hier[other],
                             zh, wet[0]);
        });
      }
      timed("wet1", [&] {
        launch_k((k_wet1<real>), dim3(G), dim3(WG), 0, stream, st, P, leaves(), hier[main_h], hier[other], zh,
                           wet[0]);
      });
      return;
    }
    timed(mwm ? "stage1" : "fv1", [&] {
      if (mwm)
        launch_k((k_stage1<real, true, true>), dim3(G), dim3(WG), 0, stream, st, P, leaves(), hier[main_h],
                           hier[other], zh, uprev, red, maxh);
      else
        launch_k((k_stage1<real, false, false>), dim3(G), dim3(WG), 0, stream, st, P, leaves(),
                           hier[main_h], hier[other], zh, uprev, red, maxh);
    });
    if (!mwm) main_h = other;
  }
  // gated: the leaf emission of this step ran in k_emit_sweep1, which marks
  // leaves at levels <= TOP_LEVEL (the top re-encode is skipped without them).
  // With quiet units the bands are the level-6 units themselves where that
  // saves a flat launch (levels 6..10 at max_ref_lvl 12): quiet units and units
  // outside the tree leave at once. us a step against flat 11 and 10 and bands
  // 5..9: urban 4096^2 FP32 443 and 449 (four of five units quiet), 664 and 663
  // (few quiet), 2500 x 1500 425 and 429, 2300 x 600 FP64 276 and 282. Up to
  // max_ref_lvl 11, without a flat launch to save, they lose (2048^2 268 and
  // 265, 700 x 650 FP64 279 and 268).
  void encode_scale_launch(bool gated = false) {
    const uint8_t* q = P.uquiet;                    // quiet units keep their stage-1 parents
    const int* gate = gated ? (const int*)&st->coarse_leaves : nullptr;
    const bool units = q && L - 1 > MRA_FLAT;
    const Levels v = units ? Levels{UNIT_LEVEL, MRA_FLAT, UNIT_LEVEL - 2} : levels(L - 1);
    for (int level = L - 1; level > v.hi; --level)
      timed("encode_scale_level", [&] {
        launch_k((k_scale_level<real>), dim3((1 << (2 * level)) / WG), dim3(WG), 0, stream, st, hier[1],
                 (const uint8_t*)sig[cur], level, cnt[2], q);
      });
    if (v.band())
      timed("encode_scale", [&] {
        launch_k((k_scale_band<real>), dim3(1 << (2 * v.lo)), dim3(WG), 0, stream, st, hier[1],
                 (const uint8_t*)sig[cur], v.lo, v.hi, cnt[2], q, gate);
      });
    timed("encode_scale_top", [&] {
      if (units)
        launch_k((k_scale_top<real, true>), dim3(1), dim3(1024), 0, stream, st, hier[1],
                 (const uint8_t*)sig[cur], v.top, cnt[2], gate);
      else
        launch_k((k_scale_top<real>), dim3(1), dim3(top_threads(v.top)), 0, stream, st, hier[1],
                 (const uint8_t*)sig[cur], v.top, cnt[2], gate);
    });
  }
  // alone: not after this step's stage 1 (whose kernel leaves the limiter's
  // largest depths)
  void stage2_launch(bool alone = false) {
    const int G = leaf_grid();
    if (hc.limitslopes) {
      if (alone) {
        MW_HIP(hipMemsetAsync(list_n, 0, sizeof(int) * LIST_INTS, stream));
        timed("maxh2", [&] {
          launch_k((k_maxh_stage2<real>), dim3(G), dim3(WG), 0, stream, st, P, leaves(), hier[1], zh, maxh);
        });
      }
      timed("stage2", [&] {
        launch_k((k_stage2_limited<real>), dim3(G), dim3(WG), 0, stream, st, P, leaves(), hier[0], hier[1],
                           zh, uprev, (const unsigned long long*)maxh, red);
      });
      return;
    }
    timed("sweep2", [&] {
      launch_k((k_sweep2<real>), dim3(G), dim3(WG), 0, stream, st, P, leaves(), hier[0], hier[1], zh, wet[1],
                         red);
    });
    timed("wet2", [&] {
      launch_k((k_wet2<real>), dim3(G), dim3(WG), 0, stream, st, P, leaves(), hier[0], hier[1], zh, wet[1], red);
    });
  }

  // ---- learned refinement ----
  bool lrn() const { return (learn || tr_x) && mwm && hc.epsilon > real(0); }

  void learn_alloc() {
    if (!mwm || !(hc.epsilon > real(0)) || hc.limitslopes)
      throw std::invalid_argument("learned refinement needs the MWDG2 solver without slope limiter and epsilon > 0");
    if (L <= UNIT_LEVEL || L > 12)
      throw std::invalid_argument("learned refinement needs 7 <= max_ref_lvl <= 12");
    if (umode) return;
    umode = alloc<uint8_t>(N_UNITS);
    uchg = alloc<uint8_t>(N_UNITS);
    uage = alloc<int>(N_UNITS);
    ustat = alloc<float>((size_t)N_UNITS * USTAT);
    ux = alloc<unsigned short>((size_t)N_UNITS * NF);
    lcnt = alloc<unsigned long long>(3 * (size_t)CNT_SLOTS);
    dirty = alloc<uint8_t>(D + 4);
    dm = alloc<real>((size_t)3 * D);
    uquiet = alloc<uint8_t>(N_UNITS);
    uwet = alloc<uint8_t>(N_UNITS);
    utouch = alloc<uint8_t>(N_UNITS);
    uborder = alloc<uint8_t>(N_UNITS);
    umx = alloc<real>((size_t)4 * N_UNITS);
    set_border_units();
    MW_HIP(hipMemsetAsync(umode, 1, N_UNITS, stream));
    MW_HIP(hipMemsetAsync(uchg, 0, N_UNITS, stream));
    MW_HIP(hipMemsetAsync(uage, 0, sizeof(int) * N_UNITS, stream));
    MW_HIP(hipMemsetAsync(ustat, 0, sizeof(float) * N_UNITS * USTAT, stream));
    MW_HIP(hipMemsetAsync(lcnt, 0, sizeof(unsigned long long) * 3 * CNT_SLOTS, stream));
  }
  void features_launch(unsigned short* out) {
    launch_k((k_unit_features<real>), dim3(nblk(N_UNITS)), dim3(WG), 0, stream, (const DevState<real>*)st,
             hier[main_h], zh, (const float*)ustat, (const uint8_t*)uchg, (const int*)uage, L, out);
  }
  // At the start of a step: the unit modes for this step. Trace recording
  // runs the plain method (every unit watched) and records the features.
  // Otherwise every l_full-th step is plain, and the step after it and every
  // l_decide-th step the network re-decides (units that changed in the last
  // step stay watched).
  void learn_decide() {
    timed("learn", [&] {
      if (tr_x) {
        if (tr_n >= tr_cap) throw std::invalid_argument("trace buffer full");
        launch_k(k_fill_u8, dim3(nblk(N_UNITS)), dim3(WG), 0, stream, umode, N_UNITS, (uint8_t)1);
        features_launch(tr_x + (size_t)tr_n * N_UNITS * NF);
      } else if (lstep % l_full == 0) {
        launch_k(k_fill_u8, dim3(nblk(N_UNITS)), dim3(WG), 0, stream, umode, N_UNITS, (uint8_t)1);
        l_need = true;
      } else if (l_need || lstep % l_decide == 0) {
        features_launch(ux);
        launch_k(k_mlp_forward, dim3(N_UNITS / MLP_BLOCK), dim3(64 * MLP_WAVES), 0, stream, lw,
                 (const unsigned short*)ux, N_UNITS, (float*)nullptr, umode, (const uint8_t*)uchg, l_thr);
        l_need = false;
      }
    });
  }
  // the unit statistics are needed by the features of the next step's
  // decision (or of every step of a trace)
  bool l_stats() const {
    if (tr_x) return true;
    const long long nx = lstep + 1;
    return (nx % l_full != 0) && (l_need || nx % l_decide == 0);
  }
  // after the rebuild (the decode band recorded each unit's tree change)
  void learn_after() {
    if (tr_x) ++tr_n;
    ++lstep;
    ++l_steps;
  }
  void set_learned(const MlpDev* w, int decide_every, int full_every, float threshold) override {
    not_in_ensemble("set_learned");
    if (!w) {
      // the next prologue still adds the record of the units the last
      // learned step did not sweep; then the quiet parameters are dropped
      learn = false;
      P.dirty = nullptr;
      P.uwet = nullptr;
      quiet_off_pending = P.uquiet != nullptr;
      return;
    }
    if (decide_every < 1 || full_every < 1) throw std::invalid_argument("decide_every and full_every must be >= 1");
    learn_alloc();
    // the context keeps its own copy of the network
    if (!lwb) {
      lwb = alloc<unsigned short>(NH * NF + 2 * NH * NH + NH);
      lwf = alloc<float>(2 * NH + 1);
    }
    unsigned short* b = lwb;
    const std::pair<const void*, size_t> parts[7] = {{w->w1, 2 * NH * NF}, {w->w2, 2 * NH * NH}, {w->w2t, 2 * NH * NH},
                                                     {w->w3, 2 * NH}, {w->b1, 4 * NH}, {w->b2, 4 * NH}, {w->b3, 4}};
    char* dst[7] = {(char*)b, (char*)(b + NH * NF), (char*)(b + NH * NF + NH * NH), (char*)(b + NH * NF + 2 * NH * NH),
                    (char*)lwf, (char*)(lwf + NH), (char*)(lwf + 2 * NH)};
    for (int k = 0; k < 7; ++k)
      MW_HIP(hipMemcpyAsync(dst[k], parts[k].first, parts[k].second, hipMemcpyDeviceToDevice, stream));
    lw = {b, b + NH * NF, b + NH * NF + NH * NH, b + NH * NF + 2 * NH * NH, lwf, lwf + NH, lwf + 2 * NH};
    l_decide = decide_every;
    l_full = full_every;
    l_thr = threshold;
    lstep = 0;
    l_need = true;
    learn = true;
    MW_HIP(hipMemsetAsync(dirty, 1, D + 4, stream));      // the first learned step re-encodes everything
    quiet_off_pending = false;
    MW_HIP(hipMemsetAsync(uquiet, 0, N_UNITS, stream));
    MW_HIP(hipMemsetAsync(uwet, 1, N_UNITS, stream));      // no unit is known dry yet
    MW_HIP(hipMemsetAsync(utouch, 1, N_UNITS, stream));
    set_quiet_params();
  }
  // Units that may never be quiet: those reaching past the DEM and, unless
  // a raster case has walls on every side (a ghost cell is then a function
  // of its border cell alone, so an unchanged dry border cell stays
  // unchanged), those touching the domain border.
  void set_border_units() {
    if (!uborder) return;
    bool walls = hc.test_case == 0;
    for (int k = 0; k < 4; ++k) walls = walls && hc.bdy[k].type == CLOSED;
    std::vector<uint8_t> b(N_UNITS);
    const int side = 1 << (L - UNIT_LEVEL);
    for (int u = 0; u < N_UNITS; ++u) {
      const int x0 = compact(u) * side, y0 = compact(u >> 1) * side;
      const bool past = x0 + side > hc.xsz || y0 + side > hc.ysz;
      const bool edge = x0 == 0 || y0 == 0 || x0 + side - 1 >= hc.xsz - 1 || y0 + side - 1 >= hc.ysz - 1;
      b[u] = (walls ? past : edge) ? 1 : 0;
    }
    MW_HIP(hipMemcpy(uborder, b.data(), N_UNITS, hipMemcpyHostToDevice));
  }
  // After the state changed outside the step (new initial state, uploads):
  // every parent is re-encoded and no unit is quiet until swept again.
  void learn_invalidate() {
    if (!dirty) return;
    MW_HIP(hipMemsetAsync(dirty, 1, D + 4, stream));
    MW_HIP(hipMemsetAsync(uquiet, 0, N_UNITS, stream));
    MW_HIP(hipMemsetAsync(uwet, 1, N_UNITS, stream));
    MW_HIP(hipMemsetAsync(utouch, 1, N_UNITS, stream));
  }
  // quiet units: the emission tiles of the fused stage-1 sweep hold whole
  // units (max_ref_lvl <= 12)
  void set_quiet_params() {
    P.dirty = learn ? dirty : nullptr;
    static_assert(EMIT_TILE_MAX == 1 << (2 * (12 - 1 - UNIT_LEVEL)), "one unit per emission tile at max_ref_lvl 12");
    const bool q = learn && L <= 12 && fuse_sweep1();
    P.uquiet = q ? uquiet : nullptr;
    P.uwet = q ? uwet : nullptr;
    P.umx = q ? umx : nullptr;
    P.n_units = N_UNITS;
  }
  void set_trace(unsigned short* x, uint8_t* chg, int cap, int n0) override {
    if (!x) { tr_x = nullptr; tr_chg = nullptr; return; }
    not_in_ensemble("trace recording");
    learn_alloc();
    tr_x = x;
    tr_chg = chg;
    tr_cap = cap;
    tr_n = n0;
  }
  int trace_count() const override { return tr_n; }
  void learn_counters(long long* out) override {
    out[0] = l_steps;
    out[1] = out[2] = out[3] = 0;
    if (!lcnt) return;
    std::vector<unsigned long long> v(3 * (size_t)CNT_SLOTS);
    MW_HIP(hipMemcpyAsync(v.data(), lcnt, sizeof(unsigned long long) * v.size(), hipMemcpyDeviceToHost, stream));
    MW_HIP(hipStreamSynchronize(stream));
    for (int k = 0; k < CNT_SLOTS; ++k) {
      out[1] += (long long)v[k];
      out[2] += (long long)v[CNT_SLOTS + k];
      out[3] += (long long)v[2 * CNT_SLOTS + k];
    }
  }

  bool l_full_step() const { return tr_x || !P.dirty || lstep % l_full == 0; }
  void rebuild(bool sweep = false) {
    bool counted = hw_tree();                        // the step's prologue zeroed the tile sums
    if (counted) {
      hw_tree_launch();
    } else {
      encode_launch(true);
      counted = decode_launch(true, true);
    }
    if (lrn() && P.uquiet) {
      timed("learn", [&] {
        with_tile([&](auto T) {
          launch_k(k_quiet_and_count<T.value>, dim3(QUIET_GROUPS + emit_tiles()), dim3(WG), 0, stream,
                   (const uint8_t*)sig[cur ^ 1], (const uint8_t*)utouch, (const uint8_t*)uwet,
                   (const uint8_t*)uborder, uquiet, l_full_step() ? 1 : 0, lcnt + 2 * CNT_SLOTS,
                   (const int*)&st->done, (const uint8_t*)leaflev, L, 1 << (2 * (L - 1)), tile_sums);
        });
      });
      counted = true;
    }
    emit_launch(sweep, counted);
    cur ^= 1;
  }

  void one_step() {
    ++issued_since_sync;
    k_prologue_launch(true);
    if (quiet_off_pending) {
      P.uquiet = nullptr;
      P.umx = nullptr;
      quiet_off_pending = false;
    }
    const bool rb = hc.epsilon > real(0.0) || !issued_first;
    if (rb) {
      if (lrn()) learn_decide();
      rebuild(fuse_sweep1() || fuse_fv1());
      if (lrn()) learn_after();
    }
    if (mwm || !fuse_fv1()) stage1_launch(rb && fuse_sweep1());
    if (mwm) {
      if (hc.epsilon > real(0.0)) encode_scale_launch(rb && fuse_sweep1());
      stage2_launch();
    }
    if (rec || cum) {
      timed("stage_record", [&] {
        if (mwm)
          launch_k((k_stage_record<real, true>), dim3(1), dim3(256), 0, stream, st, P, hier[main_h], zh,
                             leaflev, stage_codes, n_stage, rec, cum, rec_cap, red, 2 * leaf_grid());
        else
          launch_k((k_stage_record<real, false>), dim3(1), dim3(256), 0, stream, st, P, hier[main_h], zh,
                             leaflev, stage_codes, n_stage, rec, cum, rec_cap, red, 2 * leaf_grid());
      });
    }
    issued_first = true;
  }

  // rows of (time, depth, bed elevation, x velocity, y velocity at each gauge)
  int stage_records(double* out, int max_rows, int* n_points) override {
    const DevState<real> s = read_state();
    *n_points = n_stage;
    const int rows = rec ? s.n_records : 0;
    if (out && rows > 0) {
      const int k = std::min(rows, max_rows);
      std::vector<real> buf((size_t)k * (1 + 4 * n_stage));
      MW_HIP(hipMemcpyAsync(buf.data(), rec, sizeof(real) * buf.size(), hipMemcpyDeviceToHost, stream));
      MW_HIP(hipStreamSynchronize(stream));
      for (size_t i = 0; i < buf.size(); ++i) out[i] = (double)buf[i];
    }
    return rows;
  }
  double dx() const override { return (double)hc.dx; }
  const std::vector<int>& gauge_codes() const override { return hc.stage_codes; }

  // output/write_all_raster_maps_{dg2,fv1}.cu + write_raster_file.cu:
  // dirroot/resroot-<index>.<elev|wd|qx|qy|vx|vy>
  real* rbuf = nullptr;
  int raster_count = -1;
  void write_rasters(int index) override {
    const int n = hc.xsz * hc.ysz;
    if (!rbuf) rbuf = alloc<real>((size_t)6 * n);
    real* o[6];
    for (int k = 0; k < 6; ++k) o[k] = rbuf + (size_t)k * n;
    if (mwm)
      launch_k((k_raster_project<real, true>), dim3(nblk(n)), dim3(WG), 0, stream, P, hier[main_h], zh, leaflev,
                         o[0], o[1], o[2], o[3], o[4], o[5]);
    else
      launch_k((k_raster_project<real, false>), dim3(nblk(n)), dim3(WG), 0, stream, P, hier[main_h], zh,
                         leaflev, o[0], o[1], o[2], o[3], o[4], o[5]);
    MW_HIP(hipGetLastError());
    std::vector<real> h((size_t)6 * n);
    MW_HIP(hipMemcpyAsync(h.data(), rbuf, sizeof(real) * h.size(), hipMemcpyDeviceToHost, stream));
    MW_HIP(hipStreamSynchronize(stream));
    const char* ext[6] = {"elev", "wd", "qx", "qy", "vx", "vy"};
    const bool on[6] = {!hc.elevoff, !hc.depthoff, hc.qoutput, hc.qoutput, hc.voutput, hc.voutput};
    mkdir(hc.dirroot.c_str(), 0755);
    for (int k = 0; k < 6; ++k) {
      if (!on[k]) continue;
      const std::string path = hc.dirroot + "/" + hc.resroot + "-" + std::to_string(index) + "." + ext[k];
      FILE* f = std::fopen(path.c_str(), "w");
      if (!f) throw InputError("cannot write " + path);
      std::fprintf(f, "ncols        %d\nnrows        %d\n", hc.xsz, hc.ysz);
      std::fprintf(f, "xllcorner    %f\nyllcorner    %f\ncellsize     %f\nNODATA_value %d\n", (double)hc.xmin,
                   (double)hc.ymin, (double)hc.dx, -9999);
      const char* fmt = sizeof(real) == 4 ? "%.8f " : "%.15f ";
      for (int j = 0; j < hc.ysz; ++j) {
        const real* row = h.data() + (size_t)k * n + (size_t)(hc.ysz - 1 - j) * hc.xsz;
        for (int i = 0; i < hc.xsz; ++i) std::fprintf(f, fmt, (double)row[i]);
        std::fprintf(f, "\n");
      }
      std::fclose(f);
    }
  }
  // classes/SaveInterval.h:47-56 with the saveint interval, checked after a step
  bool raster_due() override {
    if (raster_count < 0) raster_count = hc.saveint_count0;
    const DevState<real> s = read_state();
    if (s.time >= hc.saveint * real(raster_count)) {
      ++raster_count;
      return true;
    }
    return false;
  }
  // cumulative rows of the massint saves (device) and of the c-property saves
  // (host), as (time, dt, leaves, mra ticks, ticks, step, kind 0 c_prop / 1 massint)
  std::vector<std::array<double, 7>> cumulative_rows() {
    std::vector<std::array<double, 7>> out;
    for (const auto& r : cprop_rows) out.push_back({r[0], r[1], r[2], r[3], r[4], r[5], 0.0});
    if (cum) {
      const DevState<real> s = read_state();
      const int rows = std::min(s.n_records, rec_cap);
      std::vector<double> v((size_t)rows * 6);
      if (rows > 0) {
        MW_HIP(hipMemcpyAsync(v.data(), cum, sizeof(double) * v.size(), hipMemcpyDeviceToHost, stream));
        MW_HIP(hipStreamSynchronize(stream));
      }
      for (int i = 0; i < rows; ++i) {
        const double* r = v.data() + (size_t)i * 6;
        out.push_back({r[0], r[1], r[2], r[3], r[4], r[5], 1.0});
      }
    }
    // file order: per step the saveint block, then the massint block
    // (run_simulation.cu:656-750); both open the file with "w" on the first
    // step, so a first-step massint row replaces the c-property one
    std::stable_sort(out.begin(), out.end(), [](const auto& a, const auto& b) {
      return a[5] != b[5] ? a[5] < b[5] : a[6] < b[6];
    });
    const double first = out.empty() ? 0.0 : out.front()[5];
    bool massint_first = false;
    for (const auto& r : out) massint_first |= (r[5] == first && r[6] == 1.0);
    if (massint_first)
      out.erase(std::remove_if(out.begin(), out.end(), [&](const auto& r) { return r[5] == first && r[6] == 0.0; }),
                out.end());
    return out;
  }
  int cumulative_records(double* out, int max_rows) override {
    const auto rows = cumulative_rows();
    if (out)
      for (int i = 0; i < std::min<int>(max_rows, (int)rows.size()); ++i)
        for (int k = 0; k < 7; ++k) out[(size_t)i * 7 + k] = rows[i][k];
    return (int)rows.size();
  }
  double clock_hz() {
    int dev = 0, khz = 0;
    MW_HIP(hipGetDevice(&dev));
    MW_HIP(hipDeviceGetAttribute(&khz, hipDeviceAttributeWallClockRate, dev));
    return 1000.0 * (double)khz;
  }
  // output/write_cumulative_data.cpp:3-50
  void write_cumulative(const std::string& path) override {
    const auto rows = cumulative_rows();
    if (rows.empty()) return;
    const double hz = clock_hz();
    mkdir(hc.dirroot.c_str(), 0755);
    FILE* f = std::fopen(path.c_str(), "w");
    if (!f) throw InputError("cannot write " + path);
    std::fprintf(f, "simtime,runtime_mra,runtime_solver,runtime_total,dt,reduction\n");
    for (const auto& r : rows) {
      const real reduction = (real(100.0) - real(100.0) * real((int)r[2]) / real(hc.xsz * hc.ysz)) / real(100.0);
      const double mra = r[3] / hz, total = r[4] / hz;
      std::fprintf(f, "%f,%f,%f,%f,%f,%f\n", r[0], mra, total - mra, total, r[1], (double)reduction);
    }
    std::fclose(f);
  }
  std::string cumulative_path() const override { return hc.dirroot + "/" + hc.resroot + ".cumu"; }

  // leaf values (field ids of k_leaf_fields) of the current leaf list, field-major
  std::vector<real> leaf_fields(const std::vector<int>& ids, int n) {
    if (!lbuf) lbuf = alloc<real>((size_t)8 * N);
    FieldSel F{};
    F.n = (int)ids.size();
    for (int k = 0; k < F.n; ++k) F.v[k] = ids[k];
    if (mwm)
      launch_k((k_leaf_fields<real, true>), dim3(nblk(n)), dim3(WG), 0, stream, st, hier[main_h], zh, leaf,
                         F, lbuf, N);
    else
      launch_k((k_leaf_fields<real, false>), dim3(nblk(n)), dim3(WG), 0, stream, st, hier[main_h], zh, leaf,
                         F, lbuf, N);
    MW_HIP(hipGetLastError());
    std::vector<real> out((size_t)F.n * n);
    for (int k = 0; k < F.n; ++k)
      MW_HIP(hipMemcpyAsync(out.data() + (size_t)k * n, lbuf + (size_t)k * N, sizeof(real) * n, hipMemcpyDeviceToHost,
                            stream));
    MW_HIP(hipStreamSynchronize(stream));
    return out;
  }

  // output/write_soln_vtk.cu:3-221: dirroot/resroot-<index>.vtk, one pixel per leaf
  void write_vtk(int index) override {
    if (!leafdt) throw InputError("the VTK output needs the vtk keyword in the .par file");
    const DevState<real> s = read_state();
    const int n = s.n_leaves;
    const std::vector<real> v = leaf_fields({0, 9, 3, 6}, n);
    std::vector<int> act(n);
    std::vector<real> dtl(n);
    MW_HIP(hipMemcpyAsync(act.data(), leaf, sizeof(int) * n, hipMemcpyDeviceToHost, stream));
    MW_HIP(hipMemcpyAsync(dtl.data(), leafdt, sizeof(real) * n, hipMemcpyDeviceToHost, stream));
    MW_HIP(hipStreamSynchronize(stream));
    mkdir(hc.dirroot.c_str(), 0755);
    const std::string path = hc.dirroot + "/" + hc.resroot + "-" + std::to_string(index) + ".vtk";
    FILE* f = std::fopen(path.c_str(), "w");
    if (!f) throw InputError("cannot write " + path);
    std::fprintf(f, "# vtk DataFile Version 3.0\nMultiresolution flow and topo data\nASCII\n\n"
                    "DATASET UNSTRUCTURED_GRID\nPOINTS %d float\n", n * 4);
    for (int i = 0; i < n; ++i) {
      const int level = level_of(act[i]);
      const int code = act[i] - lvl_idx(level);
      const real cs = hc.dx * real(1 << (L - level));
      const int x = compact(code), y = compact(code >> 1);
      const real x0 = hc.xmin + real(x) * cs, x1 = hc.xmin + real(x + 1) * cs;
      const real y0 = hc.ymin + real(y) * cs, y1 = hc.ymin + real(y + 1) * cs;
      std::fprintf(f, "%f %f %f\n%f %f %f\n%f %f %f\n%f %f %f\n", (double)x0, (double)y0, 1.0, (double)x0,
                   (double)y1, 1.0, (double)x1, (double)y0, 1.0, (double)x1, (double)y1, 1.0);
    }
    std::fprintf(f, "\nCELLS %d %d\n", n, n * 5);
    for (int i = 0; i < n; ++i) std::fprintf(f, "4 %d %d %d %d\n", 4 * i, 4 * i + 1, 4 * i + 2, 4 * i + 3);
    std::fprintf(f, "\nCELL_TYPES %d\n", n);
    for (int i = 0; i < n; ++i) std::fprintf(f, "8\n");
    std::fprintf(f, "\nCELL_DATA %d\n", n);
    const real* eta = v.data();
    const real* z = v.data() + (size_t)n;
    const real* qx = v.data() + (size_t)2 * n;
    const real* qy = v.data() + (size_t)3 * n;
    auto scalars = [&](const char* name, auto value) {
      std::fprintf(f, "\nSCALARS %s float 1\nLOOKUP_TABLE default\n", name);
      for (int i = 0; i < n; ++i) std::fprintf(f, "%f\n", (double)value(i));
    };
    scalars("dt", [&](int i) { return dtl[i]; });
    scalars("h", [&](int i) { return eta[i] - z[i]; });
    scalars("qx", [&](int i) { return qx[i]; });
    scalars("qy", [&](int i) { return qy[i]; });
    scalars("z", [&](int i) { return z[i]; });
    scalars("eta", [&](int i) { return (eta[i] - z[i]) + z[i]; });
    std::fclose(f);
  }

  // output/write_c_prop_data.cu:3-84 (+ append_reals_to_file.cu): one row of
  // the leaves' discharges per save in <dirroot>qx0-c-prop.csv ... (the
  // reference joins dirroot and the name without a separator), and a row of
  // the cumulative output
  void write_c_prop() override {
    const DevState<real> s = read_state();
    const int n = s.n_leaves;
    const std::vector<int> ids = mwm ? std::vector<int>{3, 6, 4, 5, 7, 8} : std::vector<int>{3, 6};
    const char* names[6] = {"qx0-c-prop", "qy0-c-prop", "qx1x-c-prop", "qx1y-c-prop", "qy1x-c-prop", "qy1y-c-prop"};
    const std::vector<real> v = leaf_fields(ids, n);
    const char* fmt = sizeof(real) == 4 ? "%.8f," : "%.15f,";
    mkdir(hc.dirroot.c_str(), 0755);                  // classes/PlottingParams.h:48-53
    for (size_t k = 0; k < ids.size(); ++k) {
      const std::string path = hc.dirroot + names[k] + ".csv";
      FILE* f = std::fopen(path.c_str(), cprop_writes == 0 ? "w" : "a");
      if (!f) throw InputError("cannot write " + path);
      for (int i = 0; i < n; ++i) std::fprintf(f, fmt, (double)v[k * (size_t)n + i]);
      std::fprintf(f, "\n");
      std::fclose(f);
    }
    ++cprop_writes;
    if (!clk) clk = alloc<double>(2);
    launch_k((k_clock<real>), dim3(1), dim3(64), 0, stream, st, clk);
    MW_HIP(hipGetLastError());
    double c[2];
    MW_HIP(hipMemcpyAsync(c, clk, sizeof c, hipMemcpyDeviceToHost, stream));
    MW_HIP(hipStreamSynchronize(stream));
    cprop_rows.push_back({(double)s.time, (double)next_dt(), (double)n, c[0], c[1], (double)s.steps});
  }

  // the saveint block of run_simulation.cu:656-705: whatever the .par asks for
  void save_outputs(int index) override {
    if (hc.vtk) write_vtk(index);
    if (hc.raster_out) write_rasters(index);
    if (hc.c_prop) write_c_prop();
  }
  bool saveint_outputs() const override { return hc.vtk || hc.raster_out || hc.c_prop; }

  std::string out_path() const override { return hc.dirroot + "/" + hc.resroot + ".stage"; }
  bool voutput_stage() const override { return hc.voutput_stage; }

  void ensemble_step() override {
    one_step();
    MW_HIP(hipGetLastError());
  }
  // A scenario of a batched ensemble: the plain MWDG2 step without limiter,
  // epsilon > 0, 7 <= max_ref_lvl <= 12, no recording.
  bool batchable() const override {
    return mwm && !hc.limitslopes && hc.epsilon > real(0.0) && L >= 7 && L <= 12 &&
           !rec && !cum && !learn && !tr_x && !profiling;
  }
  size_t batch_args_size() const override { return sizeof(EnsArgs<real>); }
  // The table entry of a step that starts from mask parity cur ^ flip.
  void batch_args(void* out, int flip, BatchShape& shape) const override {
    EnsArgs<real> e{};
    const int c = cur ^ flip;
    e.st = st;
    e.P = P;
    e.ser = series();
    e.src = sources();
    e.red = red;
    e.nred = 2 * leaf_grid();
    e.A = hier[0];
    e.B = hier[1];
    e.Z = zh;
    e.sig_prev = sig[c];
    e.sig_new = sig[c ^ 1];
    e.xflag = xflag;
    e.preflag = preflag;
    e.leaflev = leaflev;
    e.L = L;
    e.eps = hc.epsilon;
    e.xfac = P.eps_extra_factor;
    e.dx = hc.dx;
    e.cnt_enc = cnt[0];
    e.cnt_dec = cnt[1];
    e.cnt_rescale = cnt[2];
    e.tiles = nblk(1 << (2 * (L - 1)), EMIT_TILE_BATCH);
    e.Q = 1 << (2 * (L - 1));
    e.tile_sums = tile_sums;
    e.scan = emit_scan_args(false);
    e.leaf = leaf;
    for (int k = 0; k < 4; ++k) e.nbr[k] = nbr[k];
    e.LL = leaves();
    e.W0 = wet[0];
    e.W1 = wet[1];
    e.list_n = list_n;
    e.G = leaf_grid();
    e.src_blocks = n_src ? nblk(n_src) : 0;
    e.mtop = mra_top();
    e.mlo = mra_lo();
    e.mhi = mra_hi();
    std::memcpy(out, &e, sizeof e);
    shape.max_tiles = std::max(shape.max_tiles, e.tiles);
    shape.max_g = std::max(shape.max_g, e.G);
    shape.max_src = std::max(shape.max_src, e.src_blocks);
    shape.mra_units = std::max(shape.mra_units, 1 << (2 * e.mlo));
    shape.mra_top = std::max(shape.mra_top, e.mtop);
    shape.max_level = std::max(shape.max_level, L - 1);
  }
  // One batched step of all scenarios of a table (this context only chooses
  // the precision): the pass order of one_step for the plain MWDG2 step.
  void batch_launch(const void* table, const BatchShape& sh, hipStream_t s) const override {
    const auto* E = static_cast<const EnsArgs<real>*>(table);
    const unsigned S = (unsigned)sh.scenarios;
    hipLaunchKernelGGL(kb_prologue<real>, dim3(1, S), dim3(PRO_WG), 0, s, E);
    if (sh.max_src) hipLaunchKernelGGL(kb_point_sources<real>, dim3(sh.max_src, S), dim3(WG), 0, s, E);
    // the flat levels are launched for the scenarios that have them
    for (int l = sh.max_level; l >= MRA_FLAT; --l)
      hipLaunchKernelGGL(kb_encode_level<real>, dim3((1 << (2 * l)) / WG, S), dim3(WG), 0, s, E, l);
    hipLaunchKernelGGL(kb_encode_band<real>, dim3(sh.mra_units, S), dim3(WG), 0, s, E);
    hipLaunchKernelGGL(kb_top_mra<real>, dim3(1, S), dim3(top_threads(sh.mra_top)), 0, s, E);
    hipLaunchKernelGGL(kb_topdown_band<real>, dim3(sh.mra_units, S), dim3(WG), 0, s, E);
    for (int l = MRA_FLAT; l <= sh.max_level; ++l)
      hipLaunchKernelGGL(kb_topdown_level<real>, dim3((1 << (2 * l)) / WG, S), dim3(WG), 0, s, E, l);
    hipLaunchKernelGGL(kb_emit_sweep1<real>, dim3(sh.max_tiles, S), dim3(WG), 0, s, E);
    hipLaunchKernelGGL(kb_wet1<real>, dim3(sh.max_g, S), dim3(WG), 0, s, E);
    for (int l = sh.max_level; l >= MRA_FLAT; --l)
      hipLaunchKernelGGL(kb_scale_level<real>, dim3((1 << (2 * l)) / WG, S), dim3(WG), 0, s, E, l);
    hipLaunchKernelGGL(kb_scale_band<real>, dim3(sh.mra_units, S), dim3(WG), 0, s, E);
    hipLaunchKernelGGL(kb_scale_top<real>, dim3(1, S), dim3(top_threads(sh.mra_top)), 0, s, E);
    hipLaunchKernelGGL(kb_sweep2<real>, dim3(sh.max_g, S), dim3(WG), 0, s, E);
    hipLaunchKernelGGL(kb_wet2<real>, dim3(sh.max_g, S), dim3(WG), 0, s, E);
    MW_HIP(hipGetLastError());
  }
  long long device_steps() override {
    DevState<real> s;
    MW_HIP(hipMemcpyAsync(&s, st, sizeof s, hipMemcpyDeviceToHost, stream));
    MW_HIP(hipStreamSynchronize(stream));
    return s.steps;
  }
  void resync(long long dev_steps) override {
    issued_since_sync = 0;
    dev_steps_at_sync = (int)dev_steps;
  }
  void step(int n) override {
    if (in_ensemble) throw std::invalid_argument("the context belongs to an ensemble: step the ensemble");
    for (int i = 0; i < n; ++i) one_step();
    MW_HIP(hipGetLastError());
    if (profiling) drain_profile();
  }

  DevState<real> read_state() {
    DevState<real> s;
    MW_HIP(hipMemcpyAsync(&s, st, sizeof s, hipMemcpyDeviceToHost, stream));
    MW_HIP(hipStreamSynchronize(stream));
    reconcile(s);
    return s;
  }
  // Steps enqueued after the end time do nothing on the device, but the host
  // flipped the mask parity (every rebuilding step) and, for HWFV1, the
  // ping-pong hierarchy (every step) when it enqueued them. At each state
  // read (the stream has drained) the flips of the steps the device did not
  // take are undone.
  long long issued_since_sync = 0;          // whole steps enqueued since the last state read
  int dev_steps_at_sync = 0;
  void reconcile(const DevState<real>& s) {
    const long long performed = (long long)s.steps - dev_steps_at_sync;
    const long long wasted = issued_since_sync - performed;
    if (fuse_fv1() && std::min(performed, issued_since_sync) > 0) nbr_behind = true;
    issued_since_sync = 0;
    dev_steps_at_sync = s.steps;
    if (wasted <= 0 || in_ensemble) return;
    if (hc.epsilon > real(0.0)) {
      cur ^= (int)(wasted & 1);
    } else if (s.steps == 0 && issued_first) {  // the only rebuilding step was one of them
      cur ^= 1;
      issued_first = false;
    }
    if (!mwm) main_h ^= (int)(wasted & 1);
  }

  // The fused HWFV1 update (k_emit_fv1) uses a leaf's neighbours where it
  // derives them and leaves the lists unwritten (at 512^2 the stores cost 1 us
  // of a 52 us step). They follow from the leaf list and its labels, so they
  // are written here, before a call that reads them or changes either.
  void write_nbrs() {
    if (mwm) return;
    const DevState<real> s = read_state();
    if (!nbr_behind) return;
    nbr_behind = false;
    fill_nbrs(s.n_leaves);
  }
  void fill_nbrs(int n) {
    if (n > 0)
      launch_k((k_fill_nbrs<real>), dim3(nblk(n)), dim3(WG), 0, stream, P, (const int*)&st->n_leaves,
               (const int*)leaf, (const uint8_t*)leaflev, nbr[0], nbr[1], nbr[2], nbr[3]);
    MW_HIP(hipGetLastError());
  }

  // minimum over the reduction slots written by the last update kernel
  real next_dt() {
    std::vector<real> v(2 * leaf_grid());
    MW_HIP(hipMemcpyAsync(v.data(), red, sizeof(real) * v.size(), hipMemcpyDeviceToHost, stream));
    MW_HIP(hipStreamSynchronize(stream));
    real m = v[0];
    for (real x : v) m = x < m ? x : m;
    return m;
  }
  unsigned long long slot_sum(const unsigned long long* d) {
    std::vector<unsigned long long> v(CNT_SLOTS);
    MW_HIP(hipMemcpyAsync(v.data(), d, sizeof(unsigned long long) * CNT_SLOTS, hipMemcpyDeviceToHost, stream));
    MW_HIP(hipStreamSynchronize(stream));
    unsigned long long s = 0;
    for (auto x : v) s += x;
    return s;
  }

  void counters(mw_counters* c) override {
    const DevState<real> s = read_state();
    c->time = s.time;
    c->dt = s.dt;
    c->dt_next = s.first ? (double)s.dt : (double)next_dt();
    c->sim_time = s.sim_time;
    c->steps = s.steps;
    c->n_leaves = s.n_leaves;
    c->done = s.done;
    c->max_ref_lvl = L;
    c->solver = hc.solver;
    c->precision = (int)sizeof(real);
    for (int k = 0; k < 5; ++k) c->maxes[k] = s.mx[k];
    c->leaf_updates = (long long)s.leaf_sum;
    c->parents_encoded = (long long)slot_sum(cnt[0]);
    c->parents_decoded = (long long)slot_sum(cnt[1]);
    c->parents_rescaled = (long long)slot_sum(cnt[2]);
    c->wet_updates[0] = (long long)s.wet_sum[0];
    c->wet_updates[1] = (long long)s.wet_sum[1];
    c->nonfinite = s.nonfinite;
  }

  void stage(const std::string& s) override {
    if (learn || tr_x)
      throw std::logic_error("single stages run the plain step: turn the learned step and trace recording off first");
    if (in_ensemble) throw std::logic_error("the context belongs to an ensemble: step the ensemble");
    write_nbrs();
    if (s == "prologue") k_prologue_launch();
    else if (s == "point_sources") k_sources_launch();
    else if (s == "encode") encode_launch();
    else if (s == "decode") decode_launch();
    else if (s == "emit") { emit_launch(); }
    else if (s == "swap_masks") cur ^= 1;
    else if (s == "stage1" || s == "fv1") { reset_wet_list(0); stage1_launch(); }
    else if (s == "encode_scale") encode_scale_launch();
    else if (s == "stage2") { reset_wet_list(1); stage2_launch(true); }
    else if (s == "mark_first_issued") issued_first = true;
    else throw std::invalid_argument("unknown stage " + s);
    MW_HIP(hipGetLastError());
    MW_HIP(hipStreamSynchronize(stream));
    if (profiling) drain_profile();
  }

  long long transfer(const std::string& name, void* host, long long count, bool up) override {
    if (up) not_in_ensemble("upload");
    if (!in_ensemble) (void)read_state();      // the host's mask parity and hierarchy index are current
    if (up || name.rfind("nbr", 0) == 0) write_nbrs();
    void* dev = nullptr;
    long long len = 0;
    size_t esz = 0;
    const char* fn[9] = {"eta0", "eta1x", "eta1y", "qx0", "qx1x", "qx1y", "qy0", "qy1x", "qy1y"};
    int coef_id = -1, hb = 0;                 // hierarchy coefficient through xbuf
    if (name.size() > 2 && (name[0] == 'A' || name[0] == 'B') && name[1] == '.') {
      hb = (name[0] == 'A') ? (mwm ? 0 : main_h) : (mwm ? 1 : main_h ^ 1);
      for (int v = 0; v < 9; ++v)
        if (name.substr(2) == fn[v] && (mwm || v % 3 == 0)) coef_id = v;
    } else if (name == "z0" || (mwm && (name == "z1x" || name == "z1y"))) {
      coef_id = 9 + (name == "z0" ? 0 : (name == "z1x" ? 1 : 2));
    }
    if (coef_id >= 0) {
      dev = xbuf; len = H; esz = sizeof(real);
      if (host && count > 0) {
        const int n = (int)std::min<long long>(count, len);
        if (up) {
          learn_invalidate();
          MW_HIP(hipMemcpyAsync(xbuf, host, sizeof(real) * n, hipMemcpyHostToDevice, stream));
          coef_io_launch(hb, coef_id, n, false);
        } else {
          coef_io_launch(hb, coef_id, n, true);
          MW_HIP(hipMemcpyAsync(host, xbuf, sizeof(real) * n, hipMemcpyDeviceToHost, stream));
        }
        MW_HIP(hipStreamSynchronize(stream));
      }
      return len;
    }
    if (name == "sig") { dev = sig[cur]; len = D; esz = 1; }
    else if (name == "sig_next") { dev = sig[cur ^ 1]; len = D; esz = 1; }
    else if (name == "xflag") { dev = xflag; len = D; esz = 1; }
    else if (name == "leaflev") { dev = leaflev; len = D; esz = 1; }
    else if (name == "preflag") { dev = preflag; len = D; esz = 1; }
    else if (name == "leaves" || name.rfind("nbr", 0) == 0) {
      const DevState<real> s = read_state();
      len = s.n_leaves;
      esz = sizeof(int);
      if (name != "leaves") {
        const int k = name.size() == 4 ? name[3] - '0' : -1;
        if (k < 0 || k > 3) throw std::invalid_argument("unknown array " + name);
        // the MWDG2 sweeps derive neighbours from the labels: materialise them
        if (mwm && !hc.limitslopes) fill_nbrs(len);
        dev = nbr[k];
      } else {
        dev = leaf;
      }
    } else if (name == "leaf_dt" && leafdt) {
      len = read_state().n_leaves; esz = sizeof(real); dev = leafdt;
    } else if (name == "ustat" && ustat) { dev = ustat; len = (long long)N_UNITS * USTAT; esz = sizeof(float); }
    else if (name == "uchg" && uchg) { dev = uchg; len = N_UNITS; esz = 1; }
    else if (name == "uage" && uage) { dev = uage; len = N_UNITS; esz = sizeof(int); }
    else if (name == "umode" && umode) { dev = umode; len = N_UNITS; esz = 1; }
    else if (name == "ufeat" && ux && !up) {      // features of the current state, BF16 bits
      features_launch(ux);
      dev = ux; len = (long long)N_UNITS * NF; esz = 2;
    }
    else if (name == "rev_z_order" || name == "rev_row_major") {
      if (up) throw std::invalid_argument("the sorted orders are derived arrays (download only)");
      ensure_zorder();
      dev = name == "rev_z_order" ? rev_z : rev_rm;
      len = N;
      esz = sizeof(int);
    }
    if (!dev) throw std::invalid_argument("unknown or absent array " + name);
    if (host && count > 0) {
      const size_t bytes = (size_t)std::min(count, len) * esz;
      if (up) {
        learn_invalidate();
        MW_HIP(hipMemcpyAsync(dev, host, bytes, hipMemcpyHostToDevice, stream));
      } else {
        MW_HIP(hipMemcpyAsync(host, dev, bytes, hipMemcpyDeviceToHost, stream));
      }
      MW_HIP(hipStreamSynchronize(stream));
    }
    return len;
  }

  void coef_io_launch(int b, int which, int n, bool to_buf) {
    if (mwm)
      launch_k((k_coef_io<real, true>), dim3(nblk(n)), dim3(WG), 0, stream, hier[b], zh, which, xbuf, n,
                         to_buf ? 1 : 0);
    else
      launch_k((k_coef_io<real, false>), dim3(nblk(n)), dim3(WG), 0, stream, hier[b], zh, which, xbuf, n,
                         to_buf ? 1 : 0);
    MW_HIP(hipGetLastError());
  }

  void set_scalar(const std::string& name, double v) override {
    not_in_ensemble("set_scalar");
    write_nbrs();
    DevState<real> s = read_state();
    if (name == "time") s.time = (real)v;
    else if (name == "dt") s.dt = (real)v;
    else if (name == "dt_next") {
      std::vector<real> slots(2 * leaf_grid(), real(__builtin_inff()));
      slots[0] = (real)v;
      MW_HIP(hipMemcpyAsync(red, slots.data(), sizeof(real) * slots.size(), hipMemcpyHostToDevice, stream));
    }
    else if (name == "n_leaves") s.n_leaves = (int)v;
    else if (name == "first") s.first = (int)v;
    else if (name == "mx_eta") s.mx[0] = (real)v;
    else if (name == "mx_h") s.mx[1] = (real)v;
    else if (name == "mx_qx") s.mx[2] = (real)v;
    else if (name == "mx_qy") s.mx[3] = (real)v;
    else if (name == "mx_z") s.mx[4] = (real)v;
    else if (name == "issued_first") { issued_first = v != 0; return; }
    else if (name == "cur") { cur = (int)v & 1; return; }
    else throw std::invalid_argument("unknown scalar " + name);
    MW_HIP(hipMemcpyAsync(st, &s, sizeof s, hipMemcpyHostToDevice, stream));
    MW_HIP(hipStreamSynchronize(stream));
  }

  void set_initial(const void* const* modal) override {
    not_in_ensemble("set_initial");
    for (int v = 0; v < 12; ++v) {
      const bool used = mwm || (v % 3 == 0);
      if (!used) continue;
      if (!modal[v]) throw std::invalid_argument("missing modal array");
      hc.modal[v].assign((const real*)modal[v], (const real*)modal[v] + N);
    }
    rebuild_all();
  }
  void set_boundaries(const mw_boundary* b) override {
    not_in_ensemble("set_boundaries");
    for (int k = 0; k < 4; ++k) {
      HostBoundary<real>& d = hc.bdy[k];
      d = HostBoundary<real>();
      d.type = b[k].type; d.start = b[k].start; d.end = b[k].end; d.inlet = (real)b[k].inlet;
      if ((d.type == HVAR || d.type == QVAR) && (b[k].n_series < 1 || !b[k].series_t || !b[k].series_v))
        throw std::invalid_argument("HVAR/QVAR boundary needs a time series");
      if (d.type != CLOSED && d.type != FREE && d.type != HFIX && d.type != HVAR && d.type != QFIX && d.type != QVAR)
        throw std::invalid_argument("unknown boundary type");
      for (int i = 0; i < b[k].n_series; ++i) { d.series.t.push_back((real)b[k].series_t[i]); d.series.v.push_back((real)b[k].series_v[i]); }
      for (int i = 0; i < d.end - d.start + 1; ++i) {
        const int c = d.start + i;
        const int x = (k == 0 || k == 2) ? c : (k == 1 ? hc.xsz - 1 : 0);
        const int y = (k == 0) ? hc.ysz - 1 : (k == 2 ? 0 : c);
        if (x < 0 || y < 0 || x >= md || y >= md) throw InputError("boundary span leaves the mesh");
        d.codes.push_back(morton(x, y));
      }
    }
    rebuild_all();
  }
  void set_sources(int n, const mw_point_source* s) override {
    not_in_ensemble("set_point_sources");
    hc.srcs.clear();
    for (int i = 0; i < n; ++i) {
      if (s[i].x < 0 || s[i].y < 0 || s[i].x >= md || s[i].y >= md) throw InputError("point source outside the mesh");
      HostSource<real> d;
      d.code = morton(s[i].x, s[i].y); d.type = s[i].type; d.value = (real)s[i].value;
      if ((d.type == HVAR || d.type == QVAR) && (s[i].n_series < 1 || !s[i].series_t || !s[i].series_v))
        throw std::invalid_argument("HVAR/QVAR point source needs a time series");
      if (d.type != HFIX && d.type != HVAR && d.type != QFIX && d.type != QVAR)
        throw std::invalid_argument("unknown point source type");
      for (int j = 0; j < s[i].n_series; ++j) { d.series.t.push_back((real)s[i].series_t[j]); d.series.v.push_back((real)s[i].series_v[j]); }
      hc.srcs.push_back(d);
    }
    rebuild_all();
  }
  void rebuild_all() {
    write_nbrs();
    MW_HIP(hipStreamSynchronize(stream));
    learn_invalidate();
    set_border_units();
    clear_hierarchies();
    for (uint8_t* p : {sig[0], sig[1], xflag, leaflev, preflag}) MW_HIP(hipMemsetAsync(p, 0, D + 4, stream));
    fill_params();
    upload_sources_and_series();
    build_initial();
  }
};

// ----------------------------------------------------------------------------
// The refinement network: FP32 master parameters with Adam moments, BF16
// copies for the MFMA kernels, and a device-resident dataset of recorded
// unit features and tree changes.
// ----------------------------------------------------------------------------
struct Mlp {
  hipStream_t stream = nullptr;
  float *prm = nullptr, *m1 = nullptr, *m2 = nullptr, *grad = nullptr;
  unsigned short *w1 = nullptr, *w2 = nullptr, *w2t = nullptr, *w3 = nullptr;
  unsigned short* x = nullptr;      // recorded features, steps x units x 48 (BF16)
  std::vector<int> seg_start;       // first recorded step of each recording (one context's consecutive steps)
  unsigned long long last_serial = 0;   // context and step count where the last recording ended
  long long last_steps = -1;
  unsigned short* xl = nullptr;     // features of the labelled samples (rows of x whose window fits its recording)
  uint8_t* chg = nullptr;           // recorded tree changes, steps x units
  uint8_t* y = nullptr;             // labels of the first n_samples rows of x
  int cap_steps = 0, n_steps = 0;
  long long n_samples = 0;
  float* part = nullptr;            // per-wave gradient partials
  int part_waves = 0;
  float* lossb = nullptr;           // per-batch mean losses of an epoch
  long long lossb_n = 0;
  int adam_t = 0;
  std::vector<void*> allocs;

  template <typename T>
  T* alloc(size_t n) {
    T* p = dalloc<T>(n);
    allocs.push_back(p);
    return p;
  }
  void release(void* p) {
    if (!p) return;
    allocs.erase(std::remove(allocs.begin(), allocs.end(), p), allocs.end());
    (void)hipFree(p);
  }
  ~Mlp() {
    if (stream) (void)hipStreamSynchronize(stream);
    for (void* p : allocs) (void)hipFree(p);
    if (stream) (void)hipStreamDestroy(stream);
  }
  MlpDev dev() const { return {w1, w2, w2t, w3, prm + P_B1, prm + P_B2, prm + P_B3}; }

  // Glorot-uniform weights from SplitMix64, zero biases
  void create(unsigned long long seed) {
    MW_HIP(hipStreamCreateWithFlags(&stream, hipStreamNonBlocking));
    prm = alloc<float>(N_PARAM);
    m1 = alloc<float>(N_PARAM);
    m2 = alloc<float>(N_PARAM);
    grad = alloc<float>(N_PARAM);
    w1 = alloc<unsigned short>(NH * NF);
    w2 = alloc<unsigned short>(NH * NH);
    w2t = alloc<unsigned short>(NH * NH);
    w3 = alloc<unsigned short>(NH);
    std::vector<float> h(N_PARAM, 0.f);
    unsigned long long z = seed;
    auto next = [&]() {
      z += 0x9E3779B97F4A7C15ull;
      unsigned long long r = z;
      r = (r ^ (r >> 30)) * 0xBF58476D1CE4E5B9ull;
      r = (r ^ (r >> 27)) * 0x94D049BB133111EBull;
      r ^= r >> 31;
      return (double)(r >> 11) * (1.0 / 9007199254740992.0);
    };
    auto fill = [&](int off, int n, int fan_in, int fan_out) {
      const double a = std::sqrt(6.0 / (fan_in + fan_out));
      for (int i = 0; i < n; ++i) h[off + i] = (float)((2.0 * next() - 1.0) * a);
    };
    fill(P_W1, NH * NF, NF, NH);
    fill(P_W2, NH * NH, NH, NH);
    fill(P_W3, NH, NH, 1);
    set_params(h.data());
  }
  void set_params(const float* h) {
    MW_HIP(hipMemcpyAsync(prm, h, sizeof(float) * N_PARAM, hipMemcpyHostToDevice, stream));
    MW_HIP(hipMemsetAsync(m1, 0, sizeof(float) * N_PARAM, stream));
    MW_HIP(hipMemsetAsync(m2, 0, sizeof(float) * N_PARAM, stream));
    hipLaunchKernelGGL(k_mlp_refresh, dim3(nblk(N_PARAM)), dim3(WG), 0, stream, (const float*)prm, w1, w2, w2t, w3);
    MW_HIP(hipGetLastError());
    MW_HIP(hipStreamSynchronize(stream));
    adam_t = 0;
  }
  void get_params(float* h) {
    MW_HIP(hipMemcpyAsync(h, prm, sizeof(float) * N_PARAM, hipMemcpyDeviceToHost, stream));
    MW_HIP(hipStreamSynchronize(stream));
  }
  void ensure_part(int waves) {
    if (waves <= part_waves) return;
    release(part);
    part = alloc<float>((size_t)waves * (N_PARAM + 1));
    part_waves = waves;
  }
  static int grad_grid(long long nb) { return (int)std::min<long long>(64, (nb + MLP_BLOCK - 1) / MLP_BLOCK); }

  // host rows -> device BF16
  void upload_x(const float* xh, long long n, unsigned short* d) {
    std::vector<unsigned short> b((size_t)n * NF);
    for (size_t i = 0; i < b.size(); ++i) b[i] = f2bf(xh[i]);
    MW_HIP(hipMemcpyAsync(d, b.data(), 2 * b.size(), hipMemcpyHostToDevice, stream));
    MW_HIP(hipStreamSynchronize(stream));
  }
  void forward(const float* xh, int n, float* prob) {
    DevTmp<unsigned short> d(stream, (size_t)n * NF);
    DevTmp<float> pd(stream, n);
    upload_x(xh, n, d.p);
    hipLaunchKernelGGL(k_mlp_forward, dim3(std::max(1, std::min(1024, (n + MLP_BLOCK - 1) / MLP_BLOCK))),
                       dim3(64 * MLP_WAVES), 0, stream, dev(), (const unsigned short*)d.p, n, pd.p,
                       (uint8_t*)nullptr, (const uint8_t*)nullptr, 0.f);
    MW_HIP(hipGetLastError());
    MW_HIP(hipMemcpyAsync(prob, pd.p, sizeof(float) * n, hipMemcpyDeviceToHost, stream));
    MW_HIP(hipStreamSynchronize(stream));
  }
  // batch gradient and mean loss of host samples, without an update
  void gradient(const float* xh, const float* yh, int n, float pos_weight, float* loss, float* g) {
    DevTmp<unsigned short> d(stream, (size_t)n * NF);
    DevTmp<uint8_t> yd(stream, n);
    DevTmp<float> ld(stream, 1);
    upload_x(xh, n, d.p);
    std::vector<uint8_t> yb(n);
    for (int i = 0; i < n; ++i) yb[i] = yh[i] >= 0.5f ? 1 : 0;
    MW_HIP(hipMemcpyAsync(yd.p, yb.data(), n, hipMemcpyHostToDevice, stream));
    const int grid = grad_grid(n);
    ensure_part(grid * MLP_WAVES);
    hipLaunchKernelGGL(k_mlp_grad, dim3(grid), dim3(64 * MLP_WAVES), 0, stream, dev(), (const unsigned short*)d.p,
                       (const uint8_t*)yd.p, (long long)n, 1LL, 0LL, 0LL, n, pos_weight, part);
    hipLaunchKernelGGL(k_mlp_reduce_adam, dim3(nblk(N_PARAM + 1)), dim3(WG), 0, stream, (const float*)part,
                       grid * MLP_WAVES, 1.f / (float)n, prm, m1, m2, 0.f, 0, grad, ld.p, w1, w2, w2t, w3);
    MW_HIP(hipGetLastError());
    MW_HIP(hipMemcpyAsync(g, grad, sizeof(float) * N_PARAM, hipMemcpyDeviceToHost, stream));
    MW_HIP(hipMemcpyAsync(loss, ld.p, sizeof(float), hipMemcpyDeviceToHost, stream));
    MW_HIP(hipStreamSynchronize(stream));
  }
  // trace of `steps` plain steps of ctx appended to the dataset
  void record(CtxBase& c, int steps) {
    if (steps <= 0) return;
    const int need = n_steps + steps;
    if (need > cap_steps) {
      const int cap = std::max(need, 2 * cap_steps);
      unsigned short* nx = alloc<unsigned short>((size_t)cap * N_UNITS * NF);
      uint8_t* nc = alloc<uint8_t>((size_t)cap * N_UNITS);
      if (n_steps) {
        MW_HIP(hipMemcpyAsync(nx, x, (size_t)n_steps * N_UNITS * NF * 2, hipMemcpyDeviceToDevice, stream));
        MW_HIP(hipMemcpyAsync(nc, chg, (size_t)n_steps * N_UNITS, hipMemcpyDeviceToDevice, stream));
      }
      MW_HIP(hipStreamSynchronize(stream));
      release(x);
      release(chg);
      x = nx;
      chg = nc;
      cap_steps = cap;
    }
    mw_counters cc{};
    c.counters(&cc);
    if (n_steps == 0 || c.serial != last_serial || cc.steps != last_steps) seg_start.push_back(n_steps);
    c.set_trace(x, chg, cap_steps, n_steps);
    try {
      c.step(steps);
    } catch (...) {
      c.set_trace(nullptr, nullptr, 0, 0);
      throw;
    }
    MW_HIP(hipStreamSynchronize(c.stream));
    n_steps = c.trace_count();
    c.set_trace(nullptr, nullptr, 0, 0);
    c.counters(&cc);
    last_serial = c.serial;
    last_steps = cc.steps;
  }
  // A sample (step t, unit u) takes the steps t .. t+horizon-1 of t's own
  // recording (the consecutive steps of one context, over one or more
  // mw_mlp_record calls): steps whose window would run past the end of their
  // recording (into the next, unrelated one) are left out, and the features
  // of the others are packed into xl in step order.
  long long build_labels(int horizon) {
    if (horizon < 1) throw std::invalid_argument("horizon must be >= 1");
    std::vector<std::pair<int, int>> segs;            // (first step, labelled steps)
    long long rows = 0;
    for (size_t k = 0; k < seg_start.size(); ++k) {
      const int s0 = seg_start[k], s1 = (k + 1 < seg_start.size()) ? seg_start[k + 1] : n_steps;
      const int valid = s1 - s0 - horizon + 1;
      if (valid > 0) {
        segs.push_back({s0, valid});
        rows += valid;
      }
    }
    if (rows == 0) throw std::invalid_argument("not enough recorded steps for the horizon");
    const long long n = rows * N_UNITS;
    release(y);
    release(xl);
    y = alloc<uint8_t>(n);
    xl = alloc<unsigned short>((size_t)n * NF);
    long long r0 = 0;
    for (const auto& sg : segs) {
      const size_t at = (size_t)r0 * N_UNITS;
      MW_HIP(hipMemcpyAsync(xl + at * NF, x + (size_t)sg.first * N_UNITS * NF, (size_t)sg.second * N_UNITS * NF * 2,
                            hipMemcpyDeviceToDevice, stream));
      const long long m = (long long)sg.second * N_UNITS;
      hipLaunchKernelGGL(k_unit_labels, dim3(nblk(m)), dim3(WG), 0, stream, (const uint8_t*)(chg + (size_t)sg.first * N_UNITS),
                         sg.second + horizon - 1, horizon, y + at);
      r0 += sg.second;
    }
    MW_HIP(hipGetLastError());
    MW_HIP(hipStreamSynchronize(stream));
    n_samples = n;
    return n;
  }
  // Adam over the dataset, one affine permutation of the samples per epoch
  void fit(int epochs, int batch, float lr, float pos_weight, float* epoch_loss) {
    if (!y || n_samples <= 0) throw std::invalid_argument("no labelled samples: record and build labels first");
    if (batch < MLP_BLOCK) throw std::invalid_argument("batch must be at least 64 samples");
    const long long n = n_samples;
    const long long nbatch = (n + batch - 1) / batch;
    if (nbatch > lossb_n) {
      release(lossb);
      lossb = alloc<float>(nbatch);
      lossb_n = nbatch;
    }
    ensure_part(grad_grid(batch) * MLP_WAVES);
    static const long long primes[] = {1000003, 998244353, 1000000007, 2147483647, 104729, 7919};
    for (int e = 0; e < epochs; ++e) {
      long long a = 1;
      for (long long pcand : primes) {
        const long long p = pcand + 2 * e;           // odd, different per epoch
        long long g = p, h = n;
        while (h) { const long long t = g % h; g = h; h = t; }
        if (g == 1) { a = p % n; break; }
      }
      if (a == 0) a = 1;
      const long long c = ((long long)e * 7919 + 13) % n;
      for (long long b = 0; b < nbatch; ++b) {
        const long long base = b * batch;
        const int nb = (int)std::min<long long>(batch, n - base);
        const int grid = grad_grid(nb);
        hipLaunchKernelGGL(k_mlp_grad, dim3(grid), dim3(64 * MLP_WAVES), 0, stream, dev(), (const unsigned short*)xl,
                           (const uint8_t*)y, n, a, c, base, nb, pos_weight, part);
        ++adam_t;
        hipLaunchKernelGGL(k_mlp_reduce_adam, dim3(nblk(N_PARAM + 1)), dim3(WG), 0, stream, (const float*)part,
                           grid * MLP_WAVES, 1.f / (float)nb, prm, m1, m2, lr, adam_t, (float*)nullptr, lossb + b,
                           w1, w2, w2t, w3);
      }
      MW_HIP(hipGetLastError());
      std::vector<float> lb(nbatch);
      MW_HIP(hipMemcpyAsync(lb.data(), lossb, sizeof(float) * nbatch, hipMemcpyDeviceToHost, stream));
      MW_HIP(hipStreamSynchronize(stream));
      double sum = 0;
      for (float v : lb) sum += v;
      if (epoch_loss) epoch_loss[e] = (float)(sum / nbatch);
    }
  }
  // confusion counts (tp, fp, fn, tn) of the dataset at a threshold
  void eval(float thr, long long* out) {
    if (!y || n_samples <= 0) throw std::invalid_argument("no labelled samples");
    if (n_samples > INT32_MAX) throw std::invalid_argument("more than 2^31 samples");
    const long long n = n_samples;
    DevTmp<float> pd(stream, n);
    hipLaunchKernelGGL(k_mlp_forward, dim3((unsigned)std::min<long long>(4096, (n + MLP_BLOCK - 1) / MLP_BLOCK)),
                       dim3(64 * MLP_WAVES), 0, stream, dev(), (const unsigned short*)xl, (int)n, pd.p,
                       (uint8_t*)nullptr, (const uint8_t*)nullptr, 0.f);
    MW_HIP(hipGetLastError());
    std::vector<float> p(n);
    std::vector<uint8_t> yy(n);
    MW_HIP(hipMemcpyAsync(p.data(), pd.p, sizeof(float) * n, hipMemcpyDeviceToHost, stream));
    MW_HIP(hipMemcpyAsync(yy.data(), y, n, hipMemcpyDeviceToHost, stream));
    MW_HIP(hipStreamSynchronize(stream));
    out[0] = out[1] = out[2] = out[3] = 0;
    for (long long i = 0; i < n; ++i) {
      const bool pp = p[i] >= thr, t = yy[i] != 0;
      out[pp ? (t ? 0 : 1) : (t ? 2 : 3)]++;
    }
  }
  long long dataset(float* xo, uint8_t* yo, long long max) {
    const long long n = std::min(max, n_samples);
    if (n <= 0) return n_samples;
    std::vector<unsigned short> b((size_t)n * NF);
    MW_HIP(hipMemcpyAsync(b.data(), xl, 2 * b.size(), hipMemcpyDeviceToHost, stream));
    if (yo) MW_HIP(hipMemcpyAsync(yo, y, n, hipMemcpyDeviceToHost, stream));
    MW_HIP(hipStreamSynchronize(stream));
    if (xo)
      for (size_t i = 0; i < b.size(); ++i) xo[i] = bf2f(b[i]);
    return n_samples;
  }
};

// ----------------------------------------------------------------------------
// Ensemble: scenarios of any sizes advanced together. Each scenario's step is
// recorded as two graphs (consecutive steps: the tree rebuild flips the mask
// buffers), the graphs of all scenarios become child nodes without
// dependencies of two parent graphs, and one ensemble step is one launch of a
// parent graph (alternating). Every scenario keeps its own time step on the
// device. The optional autotuner picks each scenario's sweep work-group count
// by timing a few steps at each candidate, then the launch shape: the one
// parent graph on one stream, or each scenario's graph on its own stream.
// ----------------------------------------------------------------------------
struct Ensemble {
  std::vector<CtxBase*> ctx;
  std::vector<int> par0, par1;                   // host mask parity after even / odd replays
  std::vector<int> groups;
  std::vector<double> tune_ms;                   // per scenario: ms per step at the chosen count
  hipStream_t stream = nullptr;
  hipGraph_t parent[2] = {nullptr, nullptr};
  hipGraphExec_t exec[2] = {nullptr, nullptr};
  std::vector<hipGraph_t> child;
  std::vector<hipGraphExec_t> own;               // [scenario][2]: each scenario's graphs, instantiated
  // 0: parent graph, 1: a graph per scenario stream, 2: the captured
  // sequence launched directly on each scenario's stream
  // 3: every pass of all scenarios in one batched launch (mw_batch.inc),
  // the step's passes captured as one graph per mask parity
  int mode = 0;
  double mode_ms[4] = {0.0, 0.0, 0.0, 0.0};
  bool batched = false;
  BatchShape bshape;
  void* btab[2] = {nullptr, nullptr};
  hipGraph_t bgraph[2] = {nullptr, nullptr};
  hipGraphExec_t bexec[2] = {nullptr, nullptr};
  long long k = 0;

  ~Ensemble() {
    if (stream) (void)hipStreamSynchronize(stream);
    try {
      restore();
    } catch (...) {
    }
    for (int p = 0; p < 2; ++p) {
      if (exec[p]) (void)hipGraphExecDestroy(exec[p]);
      if (parent[p]) (void)hipGraphDestroy(parent[p]);
    }
    for (hipGraphExec_t x : own) (void)hipGraphExecDestroy(x);
    for (hipGraph_t g : child) (void)hipGraphDestroy(g);
    for (int p = 0; p < 2; ++p) {
      if (bexec[p]) (void)hipGraphExecDestroy(bexec[p]);
      if (bgraph[p]) (void)hipGraphDestroy(bgraph[p]);
      if (btab[p]) (void)hipFree(btab[p]);
    }
    for (CtxBase* c : ctx) c->in_ensemble = false;
    if (stream) (void)hipStreamDestroy(stream);
  }
  // The host mask parity of each scenario after the steps its device took
  // (a scenario past its end time takes no more, whatever the replays).
  std::vector<long long> steps0;                 // device steps when the replays started
  void restore() {
    const size_t n = std::min(par0.size(), par1.size());
    for (size_t i = 0; i < n; ++i) {
      const long long d = ctx[i]->device_steps();
      const long long r = i < steps0.size() ? d - steps0[i] : k;
      ctx[i]->set_parity((r & 1) ? par1[i] : par0[i]);
      ctx[i]->resync(d);
    }
  }
  static double time_steps(CtxBase& c, int n) {
    struct Ev {
      hipEvent_t e = nullptr;
      Ev() { MW_HIP(hipEventCreate(&e)); }
      ~Ev() { (void)hipEventDestroy(e); }
    } a, b;
    MW_HIP(hipEventRecord(a.e, c.stream));
    c.step(n);
    MW_HIP(hipEventRecord(b.e, c.stream));
    MW_HIP(hipEventSynchronize(b.e));
    float ms = 0.f;
    MW_HIP(hipEventElapsedTime(&ms, a.e, b.e));
    return ms / n;
  }
  // ms per step of all scenarios stepped one after another on their own
  // streams (before capture)
  double time_together(int n) {
    for (CtxBase* c : ctx) c->step(1);
    for (CtxBase* c : ctx) MW_HIP(hipStreamSynchronize(c->stream));
    const auto t0 = std::chrono::steady_clock::now();
    for (int i = 0; i < n; ++i)
      for (CtxBase* c : ctx) c->step(1);
    for (CtxBase* c : ctx) MW_HIP(hipStreamSynchronize(c->stream));
    return std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - t0).count() / n;
  }
  void create(const std::vector<CtxBase*>& cs, int autotune) {
    ctx = cs;
    for (CtxBase* c : ctx) {
      if (c->in_ensemble) throw std::invalid_argument("a context is in another ensemble");
      c->check_graphable();
    }
    MW_HIP(hipStreamCreateWithFlags(&stream, hipStreamNonBlocking));
    for (CtxBase* c : ctx) {
      c->step(1);                                   // the first step builds the tree from the initial state
      int g = c->sweep_groups();
      double best = 0.0;
      if (autotune > 0) {
        // one resident round of the sweep and fewer (room for the other
        // scenarios' kernels), and two rounds
        const int g0 = c->default_sweep_groups();
        for (int cand : {g0, g0 / 2, g0 / 4, g0 / 8, 2 * g0}) {
          if (cand < 8 || cand % 8 || cand > c->tile_groups()) continue;
          c->set_sweep_groups(cand);
          c->step(1);
          const double ms = time_steps(*c, autotune);
          if (best == 0.0 || ms < best) { best = ms; g = cand; }
        }
        c->set_sweep_groups(g);
      }
      groups.push_back(g);
      tune_ms.push_back(best);
      MW_HIP(hipStreamSynchronize(c->stream));
    }
    if (autotune > 0) {
      // each count above was timed with its scenario alone: keep the choice
      // only if the scenarios stepped together run at least 2% faster with it
      // than with the default counts
      std::vector<int> def;
      for (CtxBase* c : ctx) def.push_back(c->default_sweep_groups());
      if (def != groups) {
        const double t_tuned = time_together(std::max(8, 2 * autotune));
        for (size_t i = 0; i < ctx.size(); ++i) ctx[i]->set_sweep_groups(def[i]);
        const double t_def = time_together(std::max(8, 2 * autotune));
        if (t_tuned < 0.98 * t_def) {
          for (size_t i = 0; i < ctx.size(); ++i) ctx[i]->set_sweep_groups(groups[i]);
        } else {
          groups = def;
        }
      }
    }
    for (int p = 0; p < 2; ++p) {
      MW_HIP(hipGraphCreate(&parent[p], 0));
    }
    for (CtxBase* c : ctx) {
      par0.push_back(c->parity());
      hipGraph_t g[2];
      c->capture_step(&g[0]);
      par1.push_back(c->parity());
      c->capture_step(&g[1]);
      c->set_parity(par0.back());
      for (int p = 0; p < 2; ++p) {
        child.push_back(g[p]);
        hipGraphNode_t node;
        MW_HIP(hipGraphAddChildGraphNode(&node, parent[p], nullptr, 0, g[p]));
      }
      c->in_ensemble = true;
    }
    for (CtxBase* c : ctx) steps0.push_back(c->device_steps());
    build_batched();
    for (int p = 0; p < 2; ++p) MW_HIP(hipGraphInstantiate(&exec[p], parent[p], nullptr, nullptr, 0));
    for (hipGraph_t g : child) {
      hipGraphExec_t x;
      MW_HIP(hipGraphInstantiate(&x, g, nullptr, nullptr, 0));
      own.push_back(x);
    }
    if (batched) mode = 3;
    if (autotune > 0) {
      const int nm = batched ? 4 : 3;
      for (int m = 0; m < nm; ++m) {
        mode = m;
        step(1);
        wait();
        const int n = std::max(8, 2 * autotune);
        const auto t0 = std::chrono::steady_clock::now();
        step(n);
        wait();
        mode_ms[m] = std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - t0).count() / n;
      }
      mode = 0;
      for (int m = 1; m < nm; ++m)
        if (mode_ms[m] < mode_ms[mode]) mode = m;
    }
  }
  // The batched step when every scenario allows it and all share one
  // precision: argument tables for the two mask parities (the scenarios'
  // parities at the first replay and after it) and one graph of the step's
  // batched passes for each.
  void build_batched() {
    for (CtxBase* c : ctx)
      if (!c->batchable() || c->prec != ctx[0]->prec) return;
    const size_t esz = ctx[0]->batch_args_size();
    bshape = BatchShape{};
    bshape.scenarios = (int)ctx.size();
    std::vector<char> host(esz * ctx.size());
    for (int p = 0; p < 2; ++p) {
      for (size_t i = 0; i < ctx.size(); ++i) ctx[i]->batch_args(host.data() + i * esz, p, bshape);
      MW_HIP(hipMalloc(&btab[p], host.size()));
      MW_HIP(hipMemcpy(btab[p], host.data(), host.size(), hipMemcpyHostToDevice));
    }
    for (int p = 0; p < 2; ++p) {
      MW_HIP(hipStreamBeginCapture(stream, hipStreamCaptureModeThreadLocal));
      try {
        ctx[0]->batch_launch(btab[p], bshape, stream);
      } catch (...) {
        hipGraph_t tmp = nullptr;
        (void)hipStreamEndCapture(stream, &tmp);
        if (tmp) (void)hipGraphDestroy(tmp);
        throw;
      }
      MW_HIP(hipStreamEndCapture(stream, &bgraph[p]));
      MW_HIP(hipGraphInstantiate(&bexec[p], bgraph[p], nullptr, nullptr, 0));
    }
    batched = true;
  }
  void step(int n) {
    for (int i = 0; i < n; ++i) {
      if (mode == 0) {
        MW_HIP(hipGraphLaunch(exec[k & 1], stream));
      } else if (mode == 1) {
        for (size_t j = 0; j < ctx.size(); ++j) MW_HIP(hipGraphLaunch(own[2 * j + (k & 1)], ctx[j]->stream));
      } else if (mode == 3) {
        MW_HIP(hipGraphLaunch(bexec[k & 1], stream));
      } else {
        // the host mask parity of step k, as the graph of that parity starts from
        for (size_t j = 0; j < ctx.size(); ++j) {
          ctx[j]->set_parity((k & 1) ? par1[j] : par0[j]);
          ctx[j]->ensemble_step();
        }
      }
      ++k;
    }
  }
  void wait() {
    MW_HIP(hipStreamSynchronize(stream));
    for (CtxBase* c : ctx) MW_HIP(hipStreamSynchronize(c->stream));
  }
  void sync() {
    wait();
    restore();
  }
};

}  // namespace mw

// ============================================================================
// C ABI
// ============================================================================
struct mw_ctx {
  std::unique_ptr<mw::CtxBase> impl;
};
struct mw_mlp {
  mw::Mlp impl;
};
struct mw_ensemble {
  mw::Ensemble impl;
};

// Scratch of mw_sort_pairs_noalloc: the radix sort's alternate key/value
// pair and its count tables for up to MW_SORT_NOALLOC_MAX pairs (8.7 MB),
// one copy per GPU for the life of the process. Host code never uses the
// array's name as an address: each device's copy is found once with
// hipGetSymbolAddress (with that device current) and that address is what
// the kernels receive.
namespace mw {
constexpr long long NA_N = MW_SORT_NOALLOC_MAX;
constexpr long long NA_TK = 0, NA_TV = NA_N, NA_CNT = 2 * NA_N;
constexpr long long NA_OFF = NA_CNT + sort_table(NA_N), NA_SUMS = NA_OFF + sort_table(NA_N);
constexpr long long NA_INTS = NA_SUMS + sort_chunks(NA_N);
static_assert(NA_CNT % 64 == 0 && NA_OFF % 64 == 0 && NA_SUMS % 64 == 0, "256-byte aligned parts");
}  // namespace mw
static __device__ __align__(256) int scratch[mw::NA_INTS];

namespace mw {
constexpr int NA_MAX_DEVICES = 64;
int* sort_scratch_ptr() {
  static std::mutex mu;
  static std::array<int*, NA_MAX_DEVICES> ptr{};
  int dev = 0;
  MW_HIP(hipGetDevice(&dev));
  if (dev < 0 || dev >= NA_MAX_DEVICES) throw std::invalid_argument("device ordinal out of range");
  std::lock_guard<std::mutex> lock(mu);
  if (!ptr[dev]) {
    void* p = nullptr;
    MW_HIP(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
    if (!p) throw HipError("hipGetSymbolAddress(scratch) returned a null address");
    ptr[dev] = static_cast<int*>(p);
  }
  return ptr[dev];
}
}  // namespace mw

namespace {

template <typename F>
int guarded(F&& f) {
  try {
    f();
    return MW_OK;
  } catch (const mw::InputError& e) {
    mw::g_err = e.what();
    return MW_ERR_INPUT;
  } catch (const mw::HipError& e) {
    mw::g_err = e.what();
    return MW_ERR_HIP;
  } catch (const std::invalid_argument& e) {
    mw::g_err = e.what();
    return MW_ERR_ARG;
  } catch (const std::exception& e) {
    mw::g_err = e.what();
    return MW_ERR_STATE;
  }
}

#define MW_NEED(c) \
  if (!(c)) { mw::g_err = "invalid argument: " #c; return MW_ERR_ARG; }

}  // namespace

extern "C" {

const char* mw_version(void) { return "mwdg2-mi355x 0.1"; }
const char* mw_last_error(void) { return mw::g_err.c_str(); }

int mw_create(const mw_config* cfg, mw_ctx** out) {
  MW_NEED(cfg && out && cfg->par_path);
  MW_NEED(cfg->precision == 4 || cfg->precision == 8);
  *out = nullptr;
  return guarded([&] {
    auto c = std::make_unique<mw_ctx>();
    if (cfg->precision == 4) {
      auto p = std::make_unique<mw::Ctx<float>>();
      p->create(*cfg);
      c->impl = std::move(p);
    } else {
      auto p = std::make_unique<mw::Ctx<double>>();
      p->create(*cfg);
      c->impl = std::move(p);
    }
    *out = c.release();
  });
}

int mw_destroy(mw_ctx* ctx) {
  if (ctx && ctx->impl && ctx->impl->in_ensemble) {
    mw::g_err = "mw_destroy: the context belongs to an ensemble (destroy the ensemble first)";
    return MW_ERR_STATE;
  }
  delete ctx;
  return MW_OK;
}

int mw_set_initial(mw_ctx* ctx, const void* const* modal) {
  MW_NEED(ctx && modal);
  return guarded([&] { ctx->impl->set_initial(modal); });
}
int mw_set_boundaries(mw_ctx* ctx, const mw_boundary* b4) {
  MW_NEED(ctx && b4);
  return guarded([&] { ctx->impl->set_boundaries(b4); });
}
int mw_set_point_sources(mw_ctx* ctx, int n, const mw_point_source* src) {
  MW_NEED(ctx && n >= 0 && (n == 0 || src));
  return guarded([&] { ctx->impl->set_sources(n, src); });
}

int mw_step(mw_ctx* ctx, int n) {
  MW_NEED(ctx && n >= 0);
  return guarded([&] { ctx->impl->step(n); });
}

int mw_mlp_create(unsigned long long seed, mw_mlp** out) {
  MW_NEED(out);
  *out = nullptr;
  return guarded([&] {
    auto m = std::make_unique<mw_mlp>();
    m->impl.create(seed);
    *out = m.release();
  });
}

int mw_mlp_destroy(mw_mlp* m) {
  delete m;
  return MW_OK;
}

int mw_mlp_param_count(void) { return mw::N_PARAM; }

int mw_mlp_get_params(mw_mlp* m, float* out) {
  MW_NEED(m && out);
  return guarded([&] { m->impl.get_params(out); });
}

int mw_mlp_set_params(mw_mlp* m, const float* in) {
  MW_NEED(m && in);
  return guarded([&] { m->impl.set_params(in); });
}

int mw_mlp_forward(mw_mlp* m, const float* x, int n, float* prob) {
  MW_NEED(m && x && prob && n > 0);
  return guarded([&] { m->impl.forward(x, n, prob); });
}

int mw_mlp_gradient(mw_mlp* m, const float* x, const float* y, int n, float pos_weight, float* loss, float* grad) {
  MW_NEED(m && x && y && loss && grad && n > 0 && pos_weight > 0.f);
  return guarded([&] { m->impl.gradient(x, y, n, pos_weight, loss, grad); });
}

int mw_mlp_record(mw_mlp* m, mw_ctx* ctx, int steps) {
  MW_NEED(m && ctx && steps >= 0);
  return guarded([&] { m->impl.record(*ctx->impl, steps); });
}

int mw_mlp_build_labels(mw_mlp* m, int horizon, long long* n_samples) {
  MW_NEED(m && horizon >= 1);
  return guarded([&] {
    const long long n = m->impl.build_labels(horizon);
    if (n_samples) *n_samples = n;
  });
}

int mw_mlp_fit(mw_mlp* m, int epochs, int batch, float lr, float pos_weight, float* epoch_loss) {
  MW_NEED(m && epochs >= 0 && batch > 0 && lr > 0.f && pos_weight > 0.f);
  return guarded([&] { m->impl.fit(epochs, batch, lr, pos_weight, epoch_loss); });
}

int mw_mlp_eval(mw_mlp* m, float threshold, long long* counts) {
  MW_NEED(m && counts);
  return guarded([&] { m->impl.eval(threshold, counts); });
}

int mw_mlp_dataset(mw_mlp* m, float* x, unsigned char* y, long long max_samples, long long* n_samples) {
  MW_NEED(m && max_samples >= 0);
  return guarded([&] {
    const long long n = m->impl.dataset(x, y, max_samples);
    if (n_samples) *n_samples = n;
  });
}

int mw_set_learned(mw_ctx* ctx, mw_mlp* m, int decide_every, int full_every, float threshold) {
  MW_NEED(ctx);
  return guarded([&] {
    if (!m) {
      ctx->impl->set_learned(nullptr, 0, 0, 0.f);
      return;
    }
    MW_HIP(hipStreamSynchronize(m->impl.stream));
    const mw::MlpDev w = m->impl.dev();
    ctx->impl->set_learned(&w, decide_every, full_every, threshold);
  });
}

int mw_learn_counters(mw_ctx* ctx, long long* out) {
  MW_NEED(ctx && out);
  return guarded([&] { ctx->impl->learn_counters(out); });
}

int mw_set_sweep_groups(mw_ctx* ctx, int groups) {
  MW_NEED(ctx);
  return guarded([&] { ctx->impl->set_sweep_groups(groups); });
}

int mw_get_sweep_groups(mw_ctx* ctx, int* groups) {
  MW_NEED(ctx);
  MW_NEED(groups);
  return guarded([&] { *groups = ctx->impl->sweep_groups(); });
}

int mw_ensemble_create(mw_ctx* const* ctxs, int n, int autotune_steps, mw_ensemble** out) {
  MW_NEED(ctxs && n > 0 && out && autotune_steps >= 0);
  *out = nullptr;
  return guarded([&] {
    std::vector<mw::CtxBase*> cs;
    for (int i = 0; i < n; ++i) {
      if (!ctxs[i]) throw std::invalid_argument("null context");
      for (mw::CtxBase* c : cs)
        if (c == ctxs[i]->impl.get()) throw std::invalid_argument("a context is listed twice");
      cs.push_back(ctxs[i]->impl.get());
    }
    auto e = std::make_unique<mw_ensemble>();
    e->impl.create(cs, autotune_steps);
    *out = e.release();
  });
}

int mw_ensemble_step(mw_ensemble* e, int steps) {
  MW_NEED(e && steps >= 0);
  return guarded([&] { e->impl.step(steps); });
}

int mw_ensemble_sync(mw_ensemble* e) {
  MW_NEED(e);
  return guarded([&] { e->impl.sync(); });
}

int mw_ensemble_groups(mw_ensemble* e, int* groups, double* ms_per_step) {
  MW_NEED(e);
  for (size_t i = 0; i < e->impl.groups.size(); ++i) {
    if (groups) groups[i] = e->impl.groups[i];
    if (ms_per_step) ms_per_step[i] = e->impl.tune_ms[i];
  }
  return MW_OK;
}

int mw_ensemble_launch_mode(mw_ensemble* e, int* mode, double* ms_per_step) {
  MW_NEED(e && mode);
  *mode = e->impl.mode;
  if (ms_per_step)
    for (int m = 0; m < 4; ++m) ms_per_step[m] = e->impl.mode_ms[m];
  return MW_OK;
}

int mw_ensemble_set_launch_mode(mw_ensemble* e, int mode) {
  MW_NEED(e && mode >= 0 && mode <= 3);
  if (mode == 3 && !e->impl.batched) {
    mw::g_err = "the batched launch needs every scenario to be MWDG2 without limiter, epsilon > 0, "
                "7 <= max_ref_lvl <= 12, no gauge or cumulative output, one precision";
    return MW_ERR_STATE;
  }
  return guarded([&] {
    e->impl.wait();
    e->impl.mode = mode;
  });
}

int mw_ensemble_destroy(mw_ensemble* e) {
  delete e;
  return MW_OK;
}

int mw_sync(mw_ctx* ctx) {
  MW_NEED(ctx);
  return guarded([&] {
    hipError_t e = hipStreamSynchronize(ctx->impl->stream);
    if (e != hipSuccess) throw mw::HipError(hipGetErrorString(e));
  });
}

int mw_counters_get(mw_ctx* ctx, mw_counters* out) {
  MW_NEED(ctx && out);
  return guarded([&] { ctx->impl->counters(out); });
}

int mw_run_until(mw_ctx* ctx, long long max_steps, int batch, mw_counters* out) {
  MW_NEED(ctx && batch > 0);
  mw_counters c{};
  int rc = MW_OK;
  long long taken = 0;
  while (true) {
    rc = mw_counters_get(ctx, &c);
    if (rc != MW_OK) return rc;
    if (c.done || (max_steps >= 0 && c.steps >= max_steps)) break;
    if (c.steps > 0 && !(c.dt_next > 0.0)) {
      mw::g_err = "time step collapsed to " + std::to_string(c.dt_next) + " at t = " + std::to_string(c.time);
      if (out) *out = c;
      return MW_ERR_NUMERIC;
    }
    if (c.nonfinite) {
      mw::g_err = "an update produced a non-finite depth, discharge or time step by t = " + std::to_string(c.time);
      if (out) *out = c;
      return MW_ERR_NUMERIC;
    }
    int n = batch;
    if (max_steps >= 0) n = (int)std::min<long long>(batch, max_steps - c.steps);
    rc = mw_step(ctx, n);
    if (rc != MW_OK) return rc;
    taken += n;
  }
  if (out) *out = c;
  return MW_OK;
}

static int stage(mw_ctx* ctx, const char* s) {
  MW_NEED(ctx);
  return guarded([&] { ctx->impl->stage(s); });
}
int mw_zorder_build(mw_ctx* ctx) {
  MW_NEED(ctx);
  return guarded([&] {
    if (auto* f = dynamic_cast<mw::Ctx<float>*>(ctx->impl.get())) f->zorder_build();
    else dynamic_cast<mw::Ctx<double>*>(ctx->impl.get())->zorder_build();
  });
}
int mw_prologue(mw_ctx* ctx) { return stage(ctx, "prologue"); }
int mw_point_sources(mw_ctx* ctx) { return stage(ctx, "point_sources"); }
int mw_encode(mw_ctx* ctx) { return stage(ctx, "encode"); }
int mw_decode(mw_ctx* ctx) { return stage(ctx, "decode"); }
int mw_extract_leaves(mw_ctx* ctx) { return stage(ctx, "emit"); }
int mw_update_stage(mw_ctx* ctx, int s) {
  MW_NEED(s >= 0 && s <= 2);
  return stage(ctx, s == 0 ? "fv1" : (s == 1 ? "stage1" : "stage2"));
}
int mw_encode_scale(mw_ctx* ctx) { return stage(ctx, "encode_scale"); }
int mw_cfl_min(mw_ctx* ctx, double* dt_next) {
  MW_NEED(ctx && dt_next);
  mw_counters c{};
  const int rc = mw_counters_get(ctx, &c);
  if (rc == MW_OK) *dt_next = c.dt_next;
  return rc;
}
int mw_stage_named(mw_ctx* ctx, const char* name) {
  MW_NEED(name);
  return stage(ctx, name);
}

int mw_download(mw_ctx* ctx, const char* name, void* host, long long count, long long* len) {
  MW_NEED(ctx && name);
  return guarded([&] {
    const long long l = ctx->impl->transfer(name, host, count, false);
    if (len) *len = l;
  });
}
int mw_upload(mw_ctx* ctx, const char* name, const void* host, long long count) {
  MW_NEED(ctx && name && host);
  return guarded([&] { ctx->impl->transfer(name, const_cast<void*>(host), count, true); });
}
int mw_set_scalar(mw_ctx* ctx, const char* name, double v) {
  MW_NEED(ctx && name);
  return guarded([&] { ctx->impl->set_scalar(name, v); });
}

int mw_sort_pairs(int n, const int* keys, const int* vals, int* keys_out, int* vals_out) {
  MW_NEED(n >= 0 && (n == 0 || (keys && vals && keys_out && vals_out)));
  if (n == 0) return MW_OK;
  return guarded([&] {
    struct Stream {
      hipStream_t s = nullptr;
      ~Stream() { if (s) (void)hipStreamDestroy(s); }
    } st;
    MW_HIP(hipStreamCreateWithFlags(&st.s, hipStreamNonBlocking));
    mw::DevTmp<int> k0(st.s, n), v0(st.s, n), k1(st.s, n), v1(st.s, n), tk(st.s, n), tv(st.s, n);
    mw::DevTmp<int> cnt(st.s, mw::sort_table(n)), off(st.s, mw::sort_table(n)), sums(st.s, mw::sort_chunks(n));
    MW_HIP(hipMemcpyAsync(k0.p, keys, sizeof(int) * n, hipMemcpyHostToDevice, st.s));
    MW_HIP(hipMemcpyAsync(v0.p, vals, sizeof(int) * n, hipMemcpyHostToDevice, st.s));
    mw::radix_sort_pairs(n, k0.p, v0.p, k1.p, v1.p, mw::SortScratch{tk.p, tv.p, cnt.p, off.p, sums.p}, 4, st.s);
    MW_HIP(hipGetLastError());
    MW_HIP(hipMemcpyAsync(keys_out, k1.p, sizeof(int) * n, hipMemcpyDeviceToHost, st.s));
    MW_HIP(hipMemcpyAsync(vals_out, v1.p, sizeof(int) * n, hipMemcpyDeviceToHost, st.s));
    MW_HIP(hipStreamSynchronize(st.s));
  });
}

int mw_sort_pairs_noalloc(int n, const int* keys, const int* vals, int* keys_out, int* vals_out, void* stream) {
  if (n > MW_SORT_NOALLOC_MAX) {
    mw::g_err = "mw_sort_pairs_noalloc: n = " + std::to_string(n) + " exceeds the static scratch capacity of " +
                std::to_string(MW_SORT_NOALLOC_MAX) + " pairs";
    return MW_ERR_ARG;
  }
  MW_NEED(n >= 0 && (n == 0 || (keys && vals && keys_out && vals_out)));
  if (n == 0) return MW_OK;
  return guarded([&] {
    int* s = mw::sort_scratch_ptr();
    const mw::SortScratch S{s + mw::NA_TK, s + mw::NA_TV, s + mw::NA_CNT, s + mw::NA_OFF, s + mw::NA_SUMS};
    mw::radix_sort_pairs(n, keys, vals, keys_out, vals_out, S, 4, static_cast<hipStream_t>(stream));
    MW_HIP(hipGetLastError());
  });
}

int mw_device_name(char* buf, int len) {
  MW_NEED(buf && len > 0);
  return guarded([&] {
    int dev = 0;
    MW_HIP(hipGetDevice(&dev));
    hipDeviceProp_t p;
    MW_HIP(hipGetDeviceProperties(&p, dev));
    const double gib = (double)p.totalGlobalMem / (1024.0 * 1024.0 * 1024.0);
    if (p.name[0])
      std::snprintf(buf, (size_t)len, "%s (%s), %d CUs, %.0f GiB", p.name, p.gcnArchName, p.multiProcessorCount, gib);
    else                                           // some runtimes leave the marketing name empty
      std::snprintf(buf, (size_t)len, "%s, %d CUs, %.0f GiB", p.gcnArchName, p.multiProcessorCount, gib);
  });
}

int mw_stream_copy(long long bytes, int reps, double* gbs) {
  MW_NEED(bytes >= 16 && reps > 0 && gbs);
  return guarded([&] {
    const long long n = bytes / 16;
    mw::Ctx<float> tmp;
    MW_HIP(hipStreamCreateWithFlags(&tmp.stream, hipStreamNonBlocking));
    float4* a = tmp.alloc<float4>(n);
    float4* b = tmp.alloc<float4>(n);
    MW_HIP(hipMemsetAsync(a, 0, n * 16, tmp.stream));
    const int grid = 256 * 32;
    hipLaunchKernelGGL(mw::k_stream_copy, dim3(grid), dim3(mw::WG), 0, tmp.stream, a, b, n);   // warm-up
    hipEvent_t e0, e1;
    MW_HIP(hipEventCreate(&e0));
    MW_HIP(hipEventCreate(&e1));
    MW_HIP(hipEventRecord(e0, tmp.stream));
    for (int r = 0; r < reps; ++r) hipLaunchKernelGGL(mw::k_stream_copy, dim3(grid), dim3(mw::WG), 0, tmp.stream, a, b, n);
    MW_HIP(hipEventRecord(e1, tmp.stream));
    MW_HIP(hipEventSynchronize(e1));
    float ms = 0;
    MW_HIP(hipEventElapsedTime(&ms, e0, e1));
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    *gbs = 2.0 * (double)n * 16.0 * reps / (ms * 1e-3) / 1e9;
  });
}

int mw_profile(mw_ctx* ctx, int enable) {
  MW_NEED(ctx);
  return guarded([&] {
    ctx->impl->not_in_ensemble("mw_profile");
    ctx->impl->drain_profile();
    ctx->impl->profiling = enable;
    if (enable) ctx->impl->prof.clear();
  });
}

int mw_profile_read(mw_ctx* ctx, mw_kernel_time* out, int max_entries, int* n_entries) {
  MW_NEED(ctx && n_entries);
  return guarded([&] {
    ctx->impl->drain_profile();
    int i = 0;
    for (auto& kv : ctx->impl->prof) {
      if (out && i < max_entries) {
        std::snprintf(out[i].name, sizeof out[i].name, "%s", kv.first.c_str());
        out[i].launches = kv.second.n;
        out[i].total_ms = kv.second.ms;
      }
      ++i;
    }
    *n_entries = i;
  });
}

int mw_filter_table(int precision, void* out144) {
  MW_NEED(out144 && (precision == 4 || precision == 8));
  for (int f = 0; f < 4; ++f)
    for (int k = 0; k < 4; ++k)
      for (int i = 0; i < 3; ++i)
        for (int j = 0; j < 3; ++j) {
          const int o = ((f * 4 + k) * 3 + i) * 3 + j;
          if (precision == 8) static_cast<double*>(out144)[o] = mw::FB[f][k][i][j].d;
          else static_cast<float*>(out144)[o] = mw::FB[f][k][i][j].f;
        }
  return MW_OK;
}

// Drop-in for the reference binary (MAIN.cu:16-22, run_simulation.cu:3-800).
int mw_stage_records(mw_ctx* ctx, double* out, int max_rows, int* n_rows, int* n_points) {
  MW_NEED(ctx && n_rows && n_points && max_rows >= 0 && (max_rows == 0 || out));
  return guarded([&] { *n_rows = ctx->impl->stage_records(out, max_rows, n_points); });
}

int mw_write_stage_file(mw_ctx* ctx, const char* path) {
  MW_NEED(ctx);
  return guarded([&] {
    int np = 0;
    const int rows = ctx->impl->stage_records(nullptr, 0, &np);
    if (np == 0) return;
    const size_t w = 1 + 4 * (size_t)np;
    std::vector<double> r((size_t)std::max(rows, 1) * w);
    if (rows > 0) ctx->impl->stage_records(r.data(), rows, &np);
    const std::string p = path ? std::string(path) : ctx->impl->out_path();
    const size_t slash = p.rfind('/');
    if (slash != std::string::npos && slash > 0) mkdir(p.substr(0, slash).c_str(), 0755);   // dirroot
    const std::vector<int>& codes = ctx->impl->gauge_codes();
    const double dx = ctx->impl->dx();
    // output/write_stage_point_data.cu:37-190: the depth file, and with
    // voutput_stage the x and y velocity files beside it
    struct Out { std::string path, title, label; int col; };
    std::vector<Out> outs{{p, "depth (m)", "depths", 0}};
    if (ctx->impl->voutput_stage()) {
      const std::string base = (p.size() > 6 && p.compare(p.size() - 6, 6, ".stage") == 0) ? p.substr(0, p.size() - 6) : p;
      outs.push_back({base + ".xvelocity", "x velocity (m/s)", "x velocities", 2});
      outs.push_back({base + ".yvelocity", "y velocity (m/s)", "y velocities", 3});
    }
    for (const Out& o : outs) {
      FILE* f = std::fopen(o.path.c_str(), "w");
      if (!f) throw mw::InputError("cannot write " + o.path);
      std::fprintf(f, "Stage output, %s.\n\nStage information (stage,x,y,elev):\n", o.title.c_str());
      for (int k = 0; k < np; ++k) {
        const int i = mw::compact(codes[k]), j = mw::compact(codes[k] >> 1);
        std::fprintf(f, "%d %f %f %f\n", k + 1, i * dx + dx / 2.0, j * dx + dx / 2.0, rows > 0 ? r[1 + np + k] : 0.0);
      }
      std::fprintf(f, "\nOutput, %s:\nTime; stages 1 to %d\n", o.label.c_str(), np);
      for (int row = 0; row < rows; ++row) {
        const double* x = r.data() + (size_t)row * w;
        std::fprintf(f, "%f ", x[0]);
        for (int k = 0; k < np; ++k) std::fprintf(f, (k + 1 == np) ? "%f" : "%f ", x[1 + o.col * np + k]);
        std::fprintf(f, "\n");
      }
      std::fclose(f);
    }
  });
}

int mw_write_rasters(mw_ctx* ctx, int index) {
  MW_NEED(ctx && index >= 0);
  return guarded([&] { ctx->impl->write_rasters(index); });
}

int mw_write_vtk(mw_ctx* ctx, int index) {
  MW_NEED(ctx && index >= 0);
  return guarded([&] { ctx->impl->write_vtk(index); });
}

int mw_write_c_prop(mw_ctx* ctx) {
  MW_NEED(ctx);
  return guarded([&] { ctx->impl->write_c_prop(); });
}

int mw_save_outputs(mw_ctx* ctx, int index) {
  MW_NEED(ctx && index >= 0);
  return guarded([&] { ctx->impl->save_outputs(index); });
}

int mw_cumulative_records(mw_ctx* ctx, double* out, int max_rows, int* n_rows) {
  MW_NEED(ctx && n_rows && max_rows >= 0 && (out || max_rows == 0));
  return guarded([&] { *n_rows = ctx->impl->cumulative_records(out, max_rows); });
}

int mw_write_cumulative_file(mw_ctx* ctx, const char* path) {
  MW_NEED(ctx);
  return guarded([&] { ctx->impl->write_cumulative(path ? std::string(path) : ctx->impl->cumulative_path()); });
}

int mw_run_simulation(int argc, const char* const* argv) {
  MW_NEED(argc >= 2 && argv);
  const char* par = argv[argc - 1];
  // FP32 unless MW_PRECISION=8, as the reference build's default (options.cmake:2)
  const bool f64 = std::getenv("MW_PRECISION") && std::string(std::getenv("MW_PRECISION")) == "8";
  mw_config cfg{par, f64 ? 8 : 4, argc, argv};
  mw_ctx* ctx = nullptr;
  int rc = mw_create(&cfg, &ctx);
  if (rc != MW_OK) { std::fprintf(stderr, "mwdg2: %s\n", mw_last_error()); return rc; }
  mw_counters c{};
  const auto t0 = std::chrono::steady_clock::now();
  mw_counters_get(ctx, &c);
  double n = (double)(1 << c.max_ref_lvl);
  long long last_print = -1;
  const bool saves = ctx->impl->saveint_outputs();
  int saved = 0;
  while (true) {
    if (saves) {            // the save check needs the time after every step (run_simulation.cu:656-705)
      rc = mw_run_until(ctx, c.steps + 1, 1, &c);
      if (rc == MW_OK && !c.done) {
        bool due = false;
        rc = guarded([&] { due = ctx->impl->raster_due(); });
        if (rc == MW_OK && due) rc = mw_save_outputs(ctx, saved++);
      }
    } else {
      rc = mw_run_until(ctx, c.steps + 10000, 64, &c);
    }
    if (rc != MW_OK) break;
    if (c.steps / 10000 != last_print) {            // run_simulation.cu:753-762
      last_print = c.steps / 10000;
      std::printf("Elements: %lld, compression: %f%%, time step: %f, timestep: %lld, sim time: %f\n", c.n_leaves,
                  100.0 - 100.0 * c.n_leaves / (n * n), c.dt_next, c.steps, c.time);
    }
    if (c.done) break;
  }
  const double secs = std::chrono::duration<double>(std::chrono::steady_clock::now() - t0).count();
  if (rc == MW_OK) {
    std::printf("Elements: %lld, compression: %f%%, time step: %f, timestep: %lld, sim time: %f\n", c.n_leaves,
                100.0 - 100.0 * c.n_leaves / (n * n), c.dt_next, c.steps + 1, c.time);
    std::printf("Loop time: %f s\n", secs);
    if (mw_write_stage_file(ctx, nullptr) != MW_OK) std::fprintf(stderr, "mwdg2: %s\n", mw_last_error());
    if (mw_write_cumulative_file(ctx, nullptr) != MW_OK) std::fprintf(stderr, "mwdg2: %s\n", mw_last_error());
  } else {
    std::fprintf(stderr, "mwdg2: %s\n", mw_last_error());
  }
  mw_destroy(ctx);
  return rc;
}

}  // extern "C"
