// Device-side data structures and kernel declarations of the MI355X step.
#pragma once

#include "mw_math.hpp"

namespace mw {

constexpr int WG = 256;          // work-group size (4 wave64s)
// Minimum waves per SIMD asked of a latency-bound kernel's FP32 build (the
// register cap that allows them); FP64 builds keep their registers (a cap
// makes them spill).
#define WAVES32(n) (sizeof(real) == 4 ? (n) : 1)
// Levels of the tree passes from this one on are flat launches, one node per
// thread: they move their bytes at the rate of memory, a launch of 4 us is
// little beside them, and a band unit leaves lanes idle on its inner levels.
// Encode + decode of levels 5..11 at 4096^2 FP32 240 us against 256 us with
// levels 6..10 in a band. Below it the launch counts: at 1024^2 FP32 the band
// with level 9 takes 17 + 27 us, against 31 + 51 us as band and flat launch.
constexpr int MRA_FLAT = 10;
// Level-(L-1) nodes of a leaf-emission tile (one work-group): the smallest and
// the largest tile, and the tile of a batched ensemble pass.
constexpr int EMIT_TILE_MIN = 64, EMIT_TILE_MAX = 1024, EMIT_TILE_BATCH = 1024;
// Wet lists: regions at most, and ints between two regions' counters (a
// 128-byte line each).
constexpr int LIST_REGIONS = 64, LIST_PAD = 32;
// Tiles whose leaf counts each emission work-group adds up itself.
constexpr int EMIT_SELF_SCAN = 4096;
// Most level-6 units of the learned step that a tile of T nodes covers.
template <int T>
constexpr int EMIT_UNITS = T == EMIT_TILE_MIN ? 64 : 1;
constexpr int MAX_SRC = 4096;
constexpr int RED_SLOTS = 4096;  // max work-groups of a leaf kernel (one reduction slot each)
// Units of the learned step: level-6 nodes and their subtrees.
constexpr int UNIT_LEVEL = 6;
constexpr int N_UNITS = 1 << (2 * UNIT_LEVEL);

// Scalars that live on the device for the whole run, so that a step needs no
// host round trip (the reference reads dt, N_a and the maxima back every step).
template <typename real>
struct DevState {
  real time, dt, sim_time;
  real mx[5];                     // eta, h, qx, qy(=qx), z used by this step's encode
  int n_leaves;
  int done;                       // set once time >= sim_time at the top of a step
  int first;                      // 1 until the first step's prologue ran
  int steps;
  real inlet[4];                  // N, E, S, W boundary inlet values
  int row[4];                     // time-series cursors
  int n_src;
  unsigned long long leaf_sum;    // leaves updated, summed over steps
  unsigned long long wet_sum[2];  // leaves of the wet lists of stage 1 and 2, summed over steps
  alignas(128) int coarse_leaves; // set by the leaf emission when a leaf lies at a level <= TOP_LEVEL
  int save_count;                 // stage-output counter (classes/SaveInterval.h:47-56)
  int n_records;                  // stage-output rows written
  unsigned long long clk0;        // device wall clock at the first step's start
  unsigned long long clk_step;    // ... at this step's start
  unsigned long long mra_ticks;   // summed step start -> leaf list (the reference's time_mra)
  int nonfinite;                  // set once an update produced a non-finite h0, qx0, qy0 or time step
};

// Time series of the boundaries (entries 0..3) and point sources (4..).
template <typename real>
struct Series {
  const int* off;
  const int* len;
  const real* t;
  const real* v;
};

template <typename real>
struct Params {
  int L, N, D, H, mesh_dim, xsz, ysz;
  int solver;
  real eps, dx, g, tol_h, tol_q, tol_s, manning, initial_tstep, wall_height, CFL, tol_Krivo;
  real eps_extra_factor;          // 2^(M_BAR+1), evaluated on the host
  int limitslopes;
  int btype[4];                   // N, E, S, W boundary type
  int bstart[4], bend[4];
  int monai;                      // west HFIX/HVAR is the Monai non-reflective wavemaker
  int oregon;                     // west HFIX/HVAR is the Oregon Seaside wavemaker (if not monai)
  real massint;                   // stage-output interval
  real* leaf_dt;                  // per-leaf CFL time step of the last update (VTK output), or null
  uint8_t* dirty;                 // learned step: parents whose children changed since their last encode, or null
  // learned step, max_ref_lvl 12: level-6 units whose two sweeps are skipped
  // this step (all leaves dry and unchanged, neighbour units dry), or null
  const uint8_t* uquiet;
  uint8_t* uwet;                  // units holding a leaf with h >= tol_h after the last stage 2
  real* umx;                      // [unit][4] maxima of the unit's leaves when it was last swept
  int n_units;
  int test_case;                  // 0: raster case; else the built-in synthetic case
  int flow;                       // synthetic cases: FLOW_EW, FLOW_NS or FLOW_NONE
};

// Flow direction of the synthetic cases (neighbours/add_ghost_cells.cu:36-62).
enum { FLOW_NONE = 0, FLOW_EW = 1, FLOW_NS = 2 };

// Flow scale coefficients of every node of the hierarchy, eta form. Coefficient
// v = 3 * var + mode: eta0 eta1x eta1y qx0 qx1x qx1y qy0 qy1x qy1y.
// eta0 is a plain array over the nodes (read alone by the wet/dry probes and
// the point sources). The other coefficients of a node form its record
// rec[node][slot]: 8 slots for MWDG2 (eta1x ... qy1y, 32 bytes in FP32) and 2
// for HWFV1 (qx0, qy0). A leaf's coefficients are then one record read with
// two vector loads (a lane's load costs one cache access whatever its width,
// and the leaf sweeps gather one leaf per lane), and the 4 children of a
// parent, nodes 4g .. 4g+3, fill one 128-byte line.
template <typename real>
struct Hier {
  real* eta0;
  real* rec;
};

// Bed coefficients: z0 a plain array, z1x and z1y in a 2-slot node record
// (MWDG2 only).
template <typename real>
struct ZHier {
  real* z0;
  real* rec;
};

template <bool MWm>
constexpr int REC_SLOTS = MWm ? 8 : 2;

template <bool MWm>
__host__ __device__ constexpr int rec_slot(int v) { return MWm ? v - 1 : (v == 3 ? 0 : 1); }

// Node-major records: the REC_SLOTS coefficients of node h other than eta0
// are contiguous at rec + h * REC_SLOTS (32 bytes per node in FP32 MWDG2), so
// a leaf's record is two vector accesses and a sibling group's four records
// fill one 128-byte line; eta0 is a plain array (4 siblings: 16 bytes).
template <typename real, bool MWm>
__host__ __device__ __forceinline__ real* rec_of(const Hier<real>& S, int h) {
  return S.rec + (size_t)h * REC_SLOTS<MWm>;
}
template <typename real, bool MWm>
__host__ __device__ __forceinline__ real& coef(const Hier<real>& S, int v, int idx) {
  return v == 0 ? S.eta0[idx] : rec_of<real, MWm>(S, idx)[rec_slot<MWm>(v)];
}
// bed: z0 a plain array, z1x and z1y a 2-slot node-major record
template <typename real>
__host__ __device__ __forceinline__ real& zcoef(const ZHier<real>& Z, int m, int idx) {
  return m == 0 ? Z.z0[idx] : Z.rec[(size_t)idx * 2 + (m - 1)];
}

template <typename real>
struct Sources {
  int n;
  const int* code;
  const int* type;
  real* value;                    // updated in place by the prologue for HVAR/QVAR
  int* row;
};

}  // namespace mw
