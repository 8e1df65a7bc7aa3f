// Host side of libsph_hip.so: context, step sequencing and the C-ABI
// declared in include/sph_hip.h.
//
// sph_step follows iterate() (iterator.f90:44-179): for the process/ics chosen
// at context creation it wraps escaped particles, builds the neighbour lists
// (virtual periodic images instead of ghost copies), runs loop 1 (c1advanced
// Newton sweeps or c1simple), the EOS and loop 2.  All particle data stay in
// device memory between calls; the host only sizes the cell grid (one small
// read-back), watches the Newton convergence count and reads error bits.
#include <hip/hip_runtime.h>
#include <hipcub/hipcub.hpp>

#include <algorithm>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <mutex>
#include <type_traits>
#include <unordered_map>
#include <vector>

#include "../../include/sph_hip.h"
#include "sph_kernels.h"

using namespace sph;

namespace sph {
// kernels (sph_kernels.hip)
__global__ void k_wrap_reduce(Fields, const int64_t *, int, int64_t, Box, int, long long *);
__global__ void k_keys(Fields, int, Grid, uint32_t *, uint32_t *, int *, int *, long long *);
__global__ void k_cell_list(const uint32_t *, const uint32_t *, const int *, int, uint32_t *);
__global__ void k_move(Fields, Fields, const double *, double *, int, int, const uint32_t *, const int *, const uint32_t *,
                       int *, const int64_t *, int64_t *, int, int *);
__global__ void k_check_sorted(const uint32_t *, int, int *);
__global__ void k_reorder(Fields, Fields, const uint32_t *, const int64_t *, int64_t *, int, int);
__global__ void k_cell_start(const uint32_t *, int, uint32_t, int *);
__global__ void k_prep(Fields, const int64_t *, int, int64_t, Box, Grid, int, double4 *, double *, float4 *,
                       uint8_t *, double4 *, double *, uint3 *, FixFrame, float2 *, double *, long long *,
                       long long *, int, long long *, int, long long *, int);
template <int DIM, bool EXT>
__global__ void k_neigh(NeighArgs, const double4 *__restrict__, const float4 *__restrict__, uint32_t *__restrict__,
                        int *__restrict__);
template <int DIM, int KT, typename PT, typename V4, int G>
__global__ void k_loop2_fab(Loop2Args<V4>);
template <int DIM, int KT, int GRAD, typename PT, int G>
__global__ void k_loop1(Loop1Args<double4>);
template <int DIM, int KT, int GRAD, typename PT, int G>
__global__ void k_loop1_simple(Loop1Args<double4>, Fields);
template <typename V4>
__global__ void k_post1(Fields, PostSel, const uint8_t *, int, int, int, int, double, double, V4 *, V4 *,
                        V4 *, V4 *, V4 *, double4 *, double *, float2 *, long long *, long long *);
template <int DIM, int KT, typename PT, typename V4, int MODE, int G>
__global__ void k_loop2(Loop2Args<V4>);
__global__ void k_aos_to_soa(const double *, int64_t, int, const uint32_t *, Fields, int64_t *);
__global__ void k_load_cols(const double *, int64_t, int, Fields, int64_t *);
__global__ void k_step_close(const double *, int, const int *, const long long *, long long *);
__global__ void k_soa_to_aos(Fields, const int64_t *, int, double *, int64_t);
__global__ void k_ext_count(Grid, ExtGrid, const int *, int, int *, long long *);
__global__ void k_ext_fill(Grid, ExtGrid, const int *, int *, const float4 *, int, int, float4 *, int *, long long *);
__global__ void k_neigh_export(const uint32_t *, const int *, const int64_t *, const uint8_t *, int, int,
                               const int64_t *, int32_t *, int8_t *, int64_t);
__global__ void k_set_i64(int64_t *, int64_t);
__global__ void k_zero_ll(long long *, int);
__global__ void k_prerun_check(Fields, int, int *);
__global__ void k_counts_by_orig(const int *, const int64_t *, const uint8_t *, int, int64_t *);
__global__ void k_find_orig(const int64_t *, int, int64_t, int *);
__global__ void k_predict(Fields, int, DtArgs, double *, int);
__global__ void k_correct(Fields, int, const double *, const double *, int, const int *, const int *);
__global__ void k_rad_exchange(Fields, int, double, double, double, double, int *);
__global__ void k_dt_reduce(Fields, const uint8_t *, int, long long *);
__global__ void k_gravity(Fields, const uint8_t *, int, int);
__global__ void k_sts_stage(double *, const double *, double *, double *, double *, int, int, double, double, double,
                            double, const int *, const int *);
template <int DIM, int KT>
__global__ void k_diff_weights(DiffOpArgs, double *, double *);
template <int DIM, int KT>
__global__ void k_diff_rweights(DiffOpArgs, const double *, double *);
template <int DIM, int KT>
__global__ void k_diff_gcontract(DiffOpArgs, const double *, const double *, const double *, const double *, double *);
__global__ void k_diff_spmv(DiffOpArgs, const double *, const double *, double *);
__global__ void k_adj_stage(AdjStage);
__global__ void k_adj_pack(int, AdjRecs, int, int, int, const double *, double2 *);
__global__ void k_diff_coef(const uint32_t *, const int *, const double2 *, double *, int, int, int);
__global__ void k_gk_accum(const double *, int, double, double, double *);
__global__ void k_zrho(int, const double *, const double4 *, double *);
__global__ void k_diff_pack(int, const double4 *, const double4 *, double4 *, double *, double *);
__global__ void k_rev_fill(const uint8_t *, const uint32_t *, const int *, int, int, int, int *, uint32_t *);
__global__ void k_rev_sort(int, int, const int *, uint32_t *);
__global__ void k_rev_count(const uint8_t *, const uint32_t *, const int *, int, int, int *);
__global__ void k_rev_chunk(const int *, const uint32_t *, int, int, int *, uint32_t *);
__global__ void k_pair_enum(const uint8_t *, const uint32_t *, const int *, int, int, const int *, uint32_t *,
                            uint32_t *);
__global__ void k_to_sorted(const double *, const int64_t *, int, double *);
__global__ void k_from_sorted(const double *, const int64_t *, int, double *);
__global__ void k_batch_merge(int, int, int64_t, int, const int *, const uint32_t *, const double *, const double4 *,
                              const int64_t *, int, int *, uint32_t *, double *, float *, double *, int64_t *, int *);
template <bool FIRST, typename WT, bool ONE>
__global__ void k_batch_stage(BatchStage);
__global__ void k_batch_in(const double *, const int64_t *, const double *, int, double *, double *);
template <int DIM, int KT, int MODE, int G>
__global__ void k_nl_grad(DiffOpArgs, const double *, double4 *, double4 *, double *, double *, double *);
template <int DIM, int KT, int OP, int G>
__global__ void k_nl_apply(DiffOpArgs, const double *, const double4 *, const double *, NlStage);
template <int DIM, int KT, int OP, int G>
__global__ void k_nl_nu(DiffOpArgs, const double *, const double4 *, double4 *);
__global__ void k_nl_mu(DiffOpArgs, const double4 *, const double4 *, const double4 *, double4 *, double *);
template <int DIM, int KT, int MODE, int G>
__global__ void k_nl_gT(DiffOpArgs, const double4 *, const double4 *, const double *, NlAdjStage);
template <int DIM, int KT, int G>
__global__ void k_fld_adj(DiffOpArgs, const double *, const double *, const double *, const double *, const double *,
                          const double4 *, double *, double4 *);
}  // namespace sph

namespace {

constexpr int kBlock = 256;
// Per-step counters in d_stripes (long long slots, kStripes per value): the
// search's pair counts and list lengths, k_step_close's record (energy bits,
// loop 2's error bits, h_max), k_post1's h_max, the error words (ints),
// k_prep's v / B flags; loop 1's per-sweep regions follow at kStepLL.
// k_prep zeroes [0, kZeroLL) as it starts a step, so the step's first
// search, first sweep, k_post1 and loop 2 find their counters cleared
// without a fill of their own.
constexpr int kSearchLL = 0;
constexpr int kCloseRec = 2 * kStripes;
constexpr int kHmaxLL = 4 * kStripes;
constexpr int kErrLL = 5 * kStripes;      // ints: 0 search, 1 loop 1, 2 loop 2
constexpr int kExtLL = kErrLL + 4;        // where the extended grid was built: its records
constexpr int kFullLL = kErrLL + 8;       // and its fullest cell (kFullStripes)
constexpr int kZeroLL = kFullLL + kFullStripes;
constexpr int kFlagSlots = 6 * kStripes;
constexpr int kDtLL = 7 * kStripes;       // the leapfrog pass's time step (not cleared)
constexpr int kMovedLL = kDtLL + 1;       // an int: the order of the particles broke (cleared by k_keys)
constexpr int kDtBlocks = 256;            // k_dt_reduce's blocks at most
// particles of the fullest cell up to which a step orders them by counting
// (k_move): a particle looks through its whole cell there, which stays a few
// percent of the pass at 256, and is then still a small part of what the
// search reads for it; beyond, one cell's atomics also follow one another
constexpr long long kCountedCell = 256;
constexpr int kStepLL = 9 * kStripes;     // the counters before the sweep regions
enum { kErrSearch = 0, kErrLoop1 = 1, kErrLoop2 = 2 };
constexpr int kMaxLanes = 8;  // lanes per particle of a pair loop, at most
constexpr int kAux = 16;  // auxiliary per-particle arrays permuted with the fields

// statevars slots (0-based), const.f90:14-66
enum { S_DIM = 0, S_EQS = 1, S_DDW = 2, S_ICS = 3, S_ADDEN = 4, S_ARTTS = 5, S_COORD = 6, S_DISO = 7,
       S_DCOND = 8, S_MUZERO = 9, S_HFAC = 12, S_XMIN = 16, S_BORD = 22, S_PAD = 23, S_REALPN = 24,
       S_FIXEDPN = 25, S_GAMMA = 26, S_PROCESS = 30, S_AU = 31, S_EQONHYDRO = 33, S_EQONDIFF = 34,
       S_EQONFLD = 35, S_MOLMASS = 46 };

inline unsigned grid_for(int64_t n) { return (unsigned)std::max<int64_t>(1, (n + kBlock - 1) / kBlock); }

// blocks of the store's transposes: tiles of 64 particles
inline unsigned tiles_for(int64_t n) { return (unsigned)std::max<int64_t>(1, (n + 63) / 64); }

inline double ord2d(long long v) {
  long long b = v >= 0 ? v : (v ^ 0x7FFFFFFFFFFFFFFFLL);
  double d;
  memcpy(&d, &b, 8);
  return d;
}
inline long long d2ord_h(double d) {
  long long b;
  memcpy(&b, &d, 8);
  return b >= 0 ? b : (b ^ 0x7FFFFFFFFFFFFFFFLL);
}

}  // namespace

struct sph_ctx {
  int device = 0;
  hipStream_t stream = nullptr;
  int kt = 1;
  sph_options opt{};
  // SPH_NEIGH_TRAVERSAL=lane at creation: the search takes the per-lane
  // traversal and builds no extended grid (the lists are the same; tests
  // compare the two)
  bool lane_search = false;
  // SPH_LOOP2_GENERIC=1 at creation: loop 2 takes the kernel with every term
  // under its run-time flag, never a compile-time equation set (tests compare
  // the two)
  bool loop2_generic = false;
  // the search's extended grid (ghost cells of the imaged axes): cell counts,
  // cell starts, records; valid for the positions, order and grid it was
  // built from
  int *ext_count = nullptr, *ecs = nullptr;
  float4 *erec = nullptr;
  void *ext_tmp = nullptr;
  size_t ext_cells_cap = 0, ext_rec_cap = 0, ext_tmp_bytes = 0;
  ExtGrid ext_g{};
  uint64_t ext_version = 0;  // pos_version it was built from (0: none)
  int64_t ext_total = 0;
  int ext_cur = -1, ext_n = -1;
  Grid ext_grid{};
  Phys frozen{};
  Box box{};
  int process = 0, ics = 0, do_eos = 1, eos_iso = 0, gravity = 0;
  int maxneib = 150;
  // particles
  int64_t n = 0, n_real = 0, n_fixed = 0, cap = 0, npad = 0;
  double *fbuf[2] = {nullptr, nullptr};  // (32 + kAux) * npad doubles each
  int cur = 0;
  int naux = 0;
  int64_t *orig[2] = {nullptr, nullptr};
  uint32_t *keys = nullptr, *keys2 = nullptr, *vals = nullptr, *vals2 = nullptr;
  void *sort_tmp = nullptr;
  size_t sort_tmp_bytes = 0;
  int *cstart = nullptr;   // first sorted index of every cell key
  int *ccount = nullptr;   // particles per cell key while they are counted, else zero (behind cstart)
  int64_t ncell_cap = 0;
  long long fullest = 0;   // particles in the fullest search cell last seen (0: not known)
  int breaks = 2;          // how often the particles' moves broke their order lately (see note_order)
  bool counted = false;    // this step ordered them by counting: whether it had to comes with the search's counts
  bool red_ready = false;  // d_red holds k_wrap_reduce's start values
  bool load_moved = false;   // the load before this step reordered the rows
  bool flags_clear = false;  // the v / B flags' stripes are zero since load_order's k_keys
  bool ext_exact = false;  // the next extended grid waits for its size
  bool ext_built = false;  // this step built one: its counts come with the search's
  bool correct = false;    // this step's tail ends with the leapfrog corrector
  int sts_j = 0;           // or with stage sts_j of sts_s of an RKL2 super-step
  int sts_s = 0;
  double sts_dt = 0.0;
  long long *d_dtpart = nullptr;  // k_dt_reduce's block partials (in d_red's allocation)
  double4 *pm = nullptr, *st[2] = {nullptr, nullptr};
  double *tr[2] = {nullptr, nullptr};  // T den of the loop-1 sweep state st[k]
  // mixed path: position records (31-bit fractions, `ff` their frame),
  // (m, T den) of sweep state st[k] and (m/den, T den) for loop 2
  uint3 *pfix = nullptr;
  FixFrame ff{};
  float2 *s1[2] = {nullptr, nullptr};
  float2 *s2 = nullptr;
  double4 *pd = nullptr;                // loop 2, diffusion mode: x, y, z, m/den
  double *trd = nullptr;                // loop 2, diffusion mode: T den
  double *h0 = nullptr, *eps = nullptr;
  float4 *pf = nullptr;   // FP32 search records (relative coordinates + band bits)
  uint8_t *real = nullptr;
  uint32_t *nb = nullptr;
  int nb_cap = 0;
  int last_maxcnt = 0;  // longest neighbour list of the last search
  int even = -1;        // how even its lists were (lists_evenness; -1: none since the load)
  long long step_flags = 0;       // k_prep's v / B flags of this step
  bool loop2_pending = false;     // loop 2's read-back still to be taken
  bool neigh_pending = false;     // the search's read-back still to be taken (loop 1's first sync brings it)
  int *cnt = nullptr;
  void *q[5] = {nullptr, nullptr, nullptr, nullptr, nullptr};
  double *energy_part = nullptr;
  int64_t energy_cap = 0;
  // small device scratch: [0..7] long long reductions, then ints
  long long *d_red = nullptr;
  int *d_int = nullptr;  // 0 err, 1 maxcnt, 2 sorted flag, 3 pos, 8.. sweep counters (max_sweeps+2)
  long long *d_stripes = nullptr;         // striped counters (kStripes slots per value), sweep regions
  long long *h_rec = nullptr;             // pinned mirror of d_stripes and the sweep regions
  int *h_int = nullptr;                   // pinned mirror of d_int
  long long *h_ll = nullptr;              // pinned scratch for small host<->device values (2048)
  double *d_staging = nullptr;
  int64_t staging_bytes = 0;
  double4 *final_st = nullptr;
  Grid grid{};
  // cell keys kept from an earlier step: valid while the positions they were
  // computed from are unchanged (pos_version) and the grid is the same
  uint64_t pos_version = 1;       // bumped by every write of positions (load, leapfrog, wrap)
  bool keep_q0 = false;           // the step writes the FP64 q0 pack for sph_diff_prepare
  uint64_t vb_version = 1;        // bumped by every write of v or B (load, leapfrog)
  uint64_t flags_version = 0;     // vb_version step_flags were computed from
  bool flags_pending = false;     // this step's k_prep computes them (read with the search)
  // the bounding box and h_max the next grid needs, when nothing but the
  // library's own step changed the positions (bbox_version) or h (hmax_version)
  uint64_t h_version = 1;         // bumped by every write of h other than the step's own (load, leapfrog)
  uint64_t bbox_version = 0, hmax_version = 0;
  double last_lo[3] = {0, 0, 0}, last_hi[3] = {0, 0, 0}, next_hmax = 0.0;
  uint64_t keys_version = 0;      // pos_version the keys and cell starts belong to
  // the position records k_prep last wrote (pm, real, pf): for which
  // positions, buffer, count and grid
  uint64_t prep_version = 0;
  int prep_cur = -1;
  int64_t prep_n = -1;
  Grid prep_grid{};
  Grid keys_grid{};
  int64_t keys_n = -1, keys_nkeys = -1;
  // per-sweep counters of loop 1 (still-active stripes, pair stripes, a
  // ran flag), one region per sweep of a step, and their pinned mirror: the
  // parts of d_stripes and h_rec from kStepLL on
  long long *d_sweep = nullptr, *h_sweep = nullptr;
  int sweep_hint = 4;             // sweeps this step launches before it synchronises
  int sweep_hints[2] = {4, 4};    // for a step on the last one's results, and for the first on a loaded state
  int fresh = 1;                  // which of the two this step is
  int sweeps_zeroed = 0;          // k_prep cleared the regions of sweeps 1..this for the next batch
  sph_stats stats{};
  bool have_step = false;
  // the resident store holds the derivatives of the last successful iterate
  // of this state (nothing loaded since): a leapfrog pass then starts at its
  // predictor, as every pass after main.f90:219's initial iterate does
  bool derivs_ready = false;
  hipEvent_t ev[11]{};            // the stats' phase and kernel times (8 unused; 9, 10: a batch of sweeps)
  bool timing = false;            // record them (sph_set_timing)
  // differentiable diffusion (sph_diff_*)
  bool diff_ready = false;
  Phys diff_phys{};
  uint32_t *rent = nullptr;      // reverse entries (owner, image), list layout, rcnt per particle
  double4 *dpxh = nullptr;       // x, y, z, 1 / h of the frozen geometry
  double *dirho = nullptr;       // 1 / rho of the frozen geometry
  double *dW = nullptr, *ddW = nullptr;  // forward pair weights (list layout) and their row sums
  double *dR = nullptr, *dS = nullptr;   // reverse weights and gradient coefficients (reverse order)
  double *dZ = nullptr;
  double *drho = nullptr;        // rho of the frozen geometry
  double2 *dRec = nullptr;       // (lam, Zt) of kRecs adjoint stages per particle
  AdjRecs recs{};                // stages not yet added to the pair coefficients
  int rec_pend = 0;              // their number
  int rec_packed = 0;            // those whose records are written already
  bool coef_set = false;         // dS holds a sum (else the next records start it)
  int stage_rev = 0;             // the direction the next product runs its rows in
  bool fw_tail = false;          // the forward kept its last checkpoint segment's stage states
  int *rcnt = nullptr;           // reverse-list lengths
  int rcap = 0;                  // reverse-list capacity (list layout, multiple of 8)
  bool w_valid = false;          // dW/dR hold the weights of w_K
  double w_K[6] = {0, 0, 0, 0, 0, 0};
  double *gkdev = nullptr;       // 12 tensor-gradient accumulators
  double *dvec = nullptr;        // work vectors of npad
  double *gpart = nullptr;       // 12 partial sums per block
  double *ckpt = nullptr;        // checkpoints of T, (nsteps / every + 1) x npad
  int64_t ckpt_cap = 0;
  int fw_s = 0, fw_steps = 0, fw_every = 0;
  double fw_dt = 0.0, fw_K[6] = {0, 0, 0, 0, 0, 0};
  // operators that read grad T (2nw-+ 3, 2nw+- 4, flux-limited diffusion 5;
  // 0 = the Hessian operators of the assembled path)
  int diff_op = 0;
  double4 *nlF = nullptr, *nlU = nullptr, *nlUB = nullptr, *nlNu = nullptr, *nlMu = nullptr;
  double *nlD = nullptr, *nlDD = nullptr, *nlR = nullptr;

  // capacity in bytes of the buffers sph_diff_prepare keeps between calls, by
  // the address of their pointer
  std::unordered_map<void *, size_t> kept;

  Fields fields() const {
    Fields F;
    for (int f = 0; f < F_TOTAL; f++) F.f[f] = fbuf[cur] + (size_t)f * npad;
    return F;
  }
  double *aux(int k) const { return fbuf[cur] + (size_t)(F_TOTAL + k) * npad; }
};

#define HIPCHK(x)                                                                  \
  do {                                                                             \
    hipError_t e_ = (x);                                                           \
    if (e_ != hipSuccess) {                                                        \
      fprintf(stderr, "sph_hip: %s failed: %s\n", #x, hipGetErrorString(e_));      \
      return SPH_ERR_HIP;                                                          \
    }                                                                              \
  } while (0)

#define RCHK(x)             \
  do {                      \
    int r_ = (x);           \
    if (r_ != SPH_OK) return r_; \
  } while (0)

static int dev_alloc(void **p, size_t bytes) {
  if (*p) { (void)hipFree(*p); *p = nullptr; }
  if (bytes == 0) bytes = 16;
  if (hipMalloc(p, bytes) != hipSuccess) { *p = nullptr; return SPH_ERR_NOMEM; }
  return SPH_OK;
}

template <typename T>
static int dalloc(T **p, size_t count) { return dev_alloc((void **)p, count * sizeof(T)); }

// A buffer of the prepared operator, kept from one preparation to the next
// and made anew only to grow (its contents are then gone): allocating and
// freeing them took 1 ms of a preparation of 40^3 particles.
template <typename T>
static int keep(sph_ctx *c, T **p, size_t count) {
  size_t &cap = c->kept[(void *)p];
  const size_t bytes = std::max<size_t>(count * sizeof(T), 16);
  if (*p && bytes <= cap) return SPH_OK;
  cap = 0;
  RCHK(dev_alloc((void **)p, bytes));
  cap = bytes;
  return SPH_OK;
}

// --------------------------------------------------------------- kernel base
static double knorm(int kt, int dim) {
  const double pi = kPi;
  if (kt == KT_M4) { const double k[3] = {2. / 3., 10. / (7. * pi), 1. / pi}; return k[dim - 1]; }
  if (kt == KT_M6) { const double k[3] = {1. / 120., 7. / (478. * pi), 1. / (120. * pi)}; return k[dim - 1]; }
  const double k[3] = {1. / sqrt(pi), 1. / pi, 1. / pow(pi, 1.5)};
  return k[dim - 1];
}
static double fwc_of(int kt, int dim) {
  if (kt == KT_M4) { const double f[3] = {6., 6.3226, 6.66400}; return f[dim - 1]; }
  if (kt == KT_M6) { const double f[3] = {4., 9.31505 / 2.25, 9.6429 / 2.25}; return f[dim - 1]; }
  return 4.0;
}
static int maxneib_of(int kt, int dim) {
  static const int t[3][3] = {{35, 250, 150}, {50, 10000, 150}, {100, 5000, 50000}};
  return t[kt][dim - 1];
}
// CFL numbers cnarr (base_m6.f90:30-33, base_m4.f90:127-130, base_gauss.f90:222-225)
static void cn_of(int kt, int ddw, double *cnhydro, double *cnd2) {
  static const double t[3][4] = {{0.1, 0.96, 0.15, 0.2}, {0.3, 1.1, 0.2, 0.4}, {0.55, 1.25, 0.24, 0.50}};
  *cnhydro = t[kt][0];
  if (ddw == 401) *cnd2 = t[kt][3];                        // n2w
  else if (ddw == 403 || ddw == 404) *cnd2 = t[kt][1];     // 2nw
  else *cnd2 = t[kt][2];                                   // fab, fw, default
}

// getEqComponent, state.f90:117-149
static void eq_components(const double *s, Phys *P) {
  P->hydro = P->magneto = P->diff = P->fld = 0;
  switch ((int)s[S_EQS]) {
    case 300: P->hydro = 1; break;
    case 302: P->hydro = P->magneto = 1; break;
    case 301: P->diff = 1; break;
    case 306: P->fld = P->hydro = 1; break;
    case 303: P->hydro = P->magneto = P->diff = 1; break;
    case 304: P->hydro = P->diff = 1; break;
    case 307:
      P->diff = (int)s[S_EQONDIFF] == 1;
      P->hydro = (int)s[S_EQONHYDRO] == 1;
      P->fld = (int)s[S_EQONFLD] == 1;
      break;
    default: break;
  }
}

// ------------------------------------------------------------------ buffers
static int ensure_particles(sph_ctx *c, int64_t n) {
  if (n <= c->cap) return SPH_OK;
  int64_t cap = std::max<int64_t>(n, 1024);
  int64_t npad = (cap + 63) / 64 * 64;
  const size_t nf = F_TOTAL + kAux;
  for (int b = 0; b < 2; b++) {
    RCHK(dalloc(&c->fbuf[b], nf * npad));
    RCHK(dalloc(&c->orig[b], npad));
    RCHK(dalloc(&c->st[b], npad));
    RCHK(dalloc(&c->tr[b], npad));
    if (c->opt.precision == 1) RCHK(dalloc(&c->s1[b], npad));
  }
  if (c->opt.precision == 1) {
    RCHK(dalloc(&c->pfix, npad));
    RCHK(dalloc(&c->s2, npad));
  }
  RCHK(dalloc(&c->pd, npad));
  RCHK(dalloc(&c->trd, npad));
  RCHK(dalloc(&c->keys, npad));
  RCHK(dalloc(&c->keys2, npad));
  RCHK(dalloc(&c->vals, npad));
  RCHK(dalloc(&c->vals2, npad));
  RCHK(dalloc(&c->pm, npad));
  RCHK(dalloc(&c->h0, npad));
  RCHK(dalloc(&c->eps, npad));
  RCHK(dalloc(&c->pf, npad + 4));  // + 4 records read past the last cell by k_neigh
  HIPCHK(hipMemset(c->pf, 0, sizeof(float4) * (npad + 4)));
  RCHK(dalloc(&c->real, npad));
  RCHK(dalloc(&c->cnt, npad));
  size_t v4 = c->opt.precision == 1 ? sizeof(float4) : sizeof(double4);
  for (int k = 0; k < 5; k++) RCHK(dev_alloc(&c->q[k], v4 * npad));
  c->energy_cap = (npad * kMaxLanes + kBlock - 1) / kBlock;
  RCHK(dalloc(&c->energy_part, c->energy_cap));
  // radix-sort scratch for n keys
  size_t bytes = 0;
  (void)hipcub::DeviceRadixSort::SortPairs(nullptr, bytes, c->keys, c->keys2, c->vals, c->vals2, (int)npad, 0, 32,
                                     c->stream);
  RCHK(dev_alloc(&c->sort_tmp, bytes));
  c->sort_tmp_bytes = bytes;
  c->cap = cap;
  c->npad = npad;
  c->nb_cap = 0;
  if (c->nb) { (void)hipFree(c->nb); c->nb = nullptr; }
  return SPH_OK;
}

static int ensure_nb(sph_ctx *c, int cap) {
  if (cap <= c->nb_cap && c->nb) return SPH_OK;
  cap = (std::max(cap, 16) + 7) / 8 * 8;  // whole chunks of 8 (nb_slot)
  RCHK(dalloc(&c->nb, (size_t)cap * c->npad));
  c->nb_cap = cap;
  return SPH_OK;
}

static int ensure_cells(sph_ctx *c, int64_t nkeys) {
  if (nkeys + 1 <= c->ncell_cap) return SPH_OK;
  int64_t cap = std::max<int64_t>(nkeys + 1, 1024);
  c->ncell_cap = 0;
  RCHK(dalloc(&c->cstart, 2 * cap));
  c->ccount = c->cstart + cap;
  HIPCHK(hipMemsetAsync(c->ccount, 0, sizeof(int) * cap, c->stream));
  c->ncell_cap = cap;
  return SPH_OK;
}

// A HIP call whose failure is tolerated (timings of events a failed step never
// recorded, best-effort clean-up) still leaves the thread's last error set,
// and hipcub reports that error as its own after its next launch: clear it.
static void tolerate(hipError_t e) {
  if (e != hipSuccess) (void)hipGetLastError();
}

// The events around a step's phases and kernels, recorded only with timing
// on: every record leaves the stream idle for a few microseconds between the
// two kernels it separates (about 40 us over a 128^3 step's ten of them).
static hipError_t mark(sph_ctx *c, int k) {
  return c->timing ? hipEventRecord(c->ev[k], c->stream) : hipSuccess;
}

static float elapsed(sph_ctx *c, hipEvent_t a, hipEvent_t b) {
  if (!c->timing) return 0.f;
  float ms = 0.f;
  hipError_t e = hipEventSynchronize(b);
  if (e == hipSuccess) e = hipEventElapsedTime(&ms, a, b);
  if (e != hipSuccess) {
    tolerate(e);
    return 0.f;
  }
  return ms;
}

static int map_err(int bits) {
  if (bits & EB_Q) return SPH_ERR_Q_NAN_OR_NEG;
  if (bits & EB_NEG_H) return SPH_ERR_NEG_H;
  if (bits & EB_TRUNC) return SPH_ERR_NEIGH_TRUNCATED;
  if (bits & EB_OUTSIDE) return SPH_ERR_UNSUPPORTED;
  return SPH_OK;
}

// The short waits inside a step poll the stream until its work is done:
// the runtime's blocking wait adds its wake-up to every host round trip of
// the step, and an event recorded to wait on adds the processing of its own
// marker (a few microseconds after the last copy).
static hipError_t wait_stream(sph_ctx *c) {
  hipError_t r;
  while ((r = hipStreamQuery(c->stream)) == hipErrorNotReady) {
  }
  return r;
}

static int read_ints(sph_ctx *c, int first, int count) {
  HIPCHK(hipMemcpyAsync(c->h_int + first, c->d_int + first, sizeof(int) * count, hipMemcpyDeviceToHost, c->stream));
  HIPCHK(wait_stream(c));
  return SPH_OK;
}

// ------------------------------------------------------- step: neighbours
// Sum / max / or of the kStripes slots of value v in a pinned copy.
static long long stripe_sum(const long long *h, int v) {
  long long t = 0;
  for (int k = 0; k < kStripes; k++) t += h[v * kStripes + k];
  return t;
}
static long long stripe_max(const long long *h, int v) {
  long long t = h[v * kStripes];
  for (int k = 1; k < kStripes; k++) t = std::max(t, h[v * kStripes + k]);
  return t;
}
static long long stripe_min(const long long *h, int v) {
  long long t = h[v * kStripes];
  for (int k = 1; k < kStripes; k++) t = std::min(t, h[v * kStripes + k]);
  return t;
}

// Stencil half-width of the neighbour search in cells (cells rmax/RS wide).
#ifndef SPH_NEIGH_RS
#define SPH_NEIGH_RS 3
#endif
static const int kNeighRS = SPH_NEIGH_RS;

// The mixed path's position-record frame: an imaged axis maps its box length
// L onto 2^(31-k), k the least with 2^k L beyond any listed separation along
// it (the stencil's reach), so wrap-around differences of the fractions stay
// exact; other axes map the grid span onto 2^31.
static FixFrame fix_frame(const sph_ctx *c, const Grid &g, int dim, const int rc[3], double rmax) {
  FixFrame f{};
  for (int a = 0; a < dim; a++) {
    if (g.periodic[a]) {
      const double L = c->box.emax[a] - c->box.emin[a];
      const double reach = std::max(rc[a] * g.cs[a], rmax) + g.cs[a];
      int k = 0;
      while (k < 24 && std::ldexp(L, k) <= reach) k++;
      const double m = std::ldexp(1.0, 31 - k);
      f.base[a] = c->box.emin[a];
      f.mul[a] = m / L;
      f.scale[a] = (float)(L / m);
      f.step[a] = (uint32_t)m;
    } else {
      const double span = g.nc[a] * g.cs[a];
      const double m = std::ldexp(1.0, 31);
      f.base[a] = g.lo[a];
      f.mul[a] = span > 0.0 ? m / span : 0.0;
      f.scale[a] = (float)(span / m);
      f.step[a] = 0;
    }
  }
  return f;
}

static bool same_grid(const Grid &a, const Grid &b) {
  for (int d = 0; d < 3; d++)
    if (a.lo[d] != b.lo[d] || a.inv_cs[d] != b.inv_cs[d] || a.cs[d] != b.cs[d] || a.nc[d] != b.nc[d] ||
        a.periodic[d] != b.periodic[d])
      return false;
  return a.mdim == b.mdim && a.ty == b.ty;
}

// loop 1's per-sweep counter regions: [0, kStripes) still active,
// [kStripes, 2 kStripes) pairs, [2 kStripes] ran; region k for sweep k
constexpr int kSweepRegion = 2 * kStripes + 8;
constexpr int kSweepRegions = 242;  // sweeps 1..240 (the cap on max_sweeps) and slack
constexpr int kRecLL = kStepLL + kSweepRegions * kSweepRegion;  // d_stripes and h_rec size

// The step's read-back, one copy into the pinned mirror h_rec: d_stripes'
// counters (the search's pair counts and list lengths, k_prep's flags, the
// error words, k_step_close's record) and the regions of sweeps 1..last_sweep
// (none for 0).  The search's part can wait for a later synchronisation (the
// step's last), as loop 1 and loop 2 write only their own words of it.
static hipError_t copy_record(sph_ctx *c, int last_sweep) {
  const size_t ll = kStepLL + (last_sweep > 0 ? (size_t)(last_sweep + 1) * kSweepRegion : 0);
  return hipMemcpyAsync(c->h_rec, c->d_stripes, sizeof(long long) * ll, hipMemcpyDeviceToHost, c->stream);
}

// The Newton sweeps cap, and the last sweep of a step's first batch (the
// sweeps launched before its first synchronisation).
static int sweep_cap(const sph_ctx *c) { return c->opt.max_sweeps > 0 ? c->opt.max_sweeps : 100; }
static int first_batch_last(const sph_ctx *c) { return std::min(sweep_cap(c), std::max(1, c->sweep_hint)); }
constexpr int kWhichInt = 6;        // d_int slot: parity of the last sweep that ran
constexpr int kGoInt = 7;           // d_int slot: the queued tail runs (k_post1 decides)
constexpr int kExtTotalInt = 16;    // h_int slot: records of the extended grid
constexpr int kRedoNeigh = 1000; // internal: the lists overflowed, search again (not an SPH_ERR code)

// the error words of the step (ints in d_stripes), and the same words in a
// pinned copy of d_stripes starting at slot `base`
static int *step_err(sph_ctx *c) { return reinterpret_cast<int *>(c->d_stripes + kErrLL); }
static int copied_err(const long long *copy, int base, int word) {
  return reinterpret_cast<const int *>(copy + (kErrLL - base))[word];
}

// A move of the particles broke their order or left it: `breaks` climbs where
// more than a third of them did.
static void note_order(sph_ctx *c, bool broke) { c->breaks = std::clamp(c->breaks + (broke ? 2 : -1), 0, 6); }

static int finish_neighbours(sph_ctx *c, const long long *ll, int bits) {
  bool ext_short = false;
  if (c->ext_built) {
    c->ext_built = false;
    c->fullest = *std::max_element(ll + kFullLL, ll + kFullLL + kFullStripes);
    c->ext_total = ll[kExtLL];
    c->stats.ext_records = c->ext_total;
    ext_short = (size_t)c->ext_total + 8 > c->ext_rec_cap;
    // the grid is kept only now that it is known to be whole; where records
    // were left out it is built again with room
    c->ext_version = ext_short ? 0 : c->pos_version;
    c->ext_exact = ext_short;
  }
  if (c->counted) {
    c->counted = false;
    const bool broke = *reinterpret_cast<const int *>(ll + kMovedLL) != 0;
    note_order(c, broke);
    c->stats.sorted = broke ? 1 : 0;
  }
  if (c->flags_pending) {  // k_prep's v / B flags of this step
    c->step_flags = 0;
    for (int k = 0; k < kStripes; k++) c->step_flags |= ll[kFlagSlots + k];
    c->flags_version = c->vb_version;
    c->flags_pending = false;
  }
  c->stats.n_pairs = stripe_sum(ll, 0);
  int maxcnt = (int)stripe_max(ll, 1);
  c->last_maxcnt = maxcnt;
  c->even = lists_evenness(maxcnt, c->n_real, c->stats.n_pairs);
  c->stats.ms_k_neigh = elapsed(c, c->ev[4], c->ev[7]);
  if (bits & EB_TRUNC) return SPH_ERR_NEIGH_TRUNCATED;
  if (!(bits & EB_OVERFLOW)) return SPH_OK;
  if (ext_short) return kRedoNeigh;  // the lists' lengths are not the real ones
  RCHK(ensure_nb(c, maxcnt + 8));
  return kRedoNeigh;
}

// The deferred read-back after a synchronisation the caller made.
static int take_neighbours_now(sph_ctx *c) {
  const long long *ll = c->h_rec;
  return finish_neighbours(c, ll, copied_err(ll, 0, kErrSearch));
}

// A deferred read-back, once the stream has passed its copies.
static int take_neighbours(sph_ctx *c) {
  if (!c->neigh_pending) return SPH_OK;
  c->neigh_pending = false;
  const long long *ll = c->h_rec;
  return finish_neighbours(c, ll, copied_err(ll, 0, kErrSearch));
}

// out = exclusive prefix sums of count ints.
static int prefix_sum(sph_ctx *c, const int *in, int *out, int count) {
  size_t tb = 0;
  HIPCHK(hipcub::DeviceScan::ExclusiveSum(nullptr, tb, in, out, count, c->stream));
  if (tb > c->ext_tmp_bytes) {
    if (c->ext_tmp) { (void)hipFree(c->ext_tmp); c->ext_tmp = nullptr; }
    c->ext_tmp_bytes = 0;
    RCHK(dev_alloc(&c->ext_tmp, tb));
    c->ext_tmp_bytes = tb;
  }
  tb = c->ext_tmp_bytes;
  HIPCHK(hipcub::DeviceScan::ExclusiveSum(c->ext_tmp, tb, in, out, count, c->stream));
  return SPH_OK;
}

// Escaped real particles wrapped back into the box, the bounding box of all and
// the largest h of the real ones (F's x, y, z and h in `orig`'s order).
static int wrap_pass(sph_ctx *c, Fields F, const int64_t *orig, double lo[3], double hi[3], double *hmax,
                     bool *wrapped) {
  const long long BIG = 0x7FFFFFFFFFFFFFFFLL, SMALL = -0x7FFFFFFFFFFFFFFFLL - 1;
  if (!c->red_ready) {  // else the last step's k_prep set the start values
    long long *init = c->h_ll;
    for (int k = 0; k < kRedLL; k++) init[k] = k < 3 * kStripes ? BIG : (k < 7 * kStripes ? SMALL : 0);
    HIPCHK(hipMemcpyAsync(c->d_red, init, sizeof(long long) * kRedLL, hipMemcpyHostToDevice, c->stream));
    HIPCHK(hipMemsetAsync(c->d_int, 0, sizeof(int) * 8, c->stream));
  }
  c->red_ready = false;
  // at most 1024 blocks (four per CU), each striding over the particles
  hipLaunchKernelGGL(k_wrap_reduce, dim3(std::min(grid_for(c->n), 1024u)), dim3(kBlock), 0, c->stream, F, orig,
                     (int)c->n, c->n_real, c->box, c->frozen.dim, c->d_red);
  long long *red = c->h_ll + 512;
  HIPCHK(hipMemcpyAsync(red, c->d_red, sizeof(long long) * kRedLL, hipMemcpyDeviceToHost, c->stream));
  HIPCHK(wait_stream(c));
  if (red[7 * kStripes] & EB_OUTSIDE) return SPH_ERR_UNSUPPORTED;
  *wrapped = red[7 * kStripes + 1] != 0;
  for (int a = 0; a < 3; a++) { lo[a] = ord2d(stripe_min(red, a)); hi[a] = ord2d(stripe_max(red, 3 + a)); }
  *hmax = c->n_real > 0 ? ord2d(stripe_max(red, 6)) : 0.0;
  return SPH_OK;
}

// The cell grid: cells at least rmax/RS wide; imaged axes tile
// [emin, emax] and need 2 RS + 1 cells, else RS drops to 1.  The search
// reads each (y, z) row as whole ranges along x, so thin rows follow the
// sphere closely at a few more row ranges, and they order the particles
// so that adjacent lanes gather adjacent neighbours in the loops.  Cells
// of a third of the radius measured fastest for the whole step (a half
// and a quarter were slower in the loops and in the search).
static Grid search_grid(const sph_ctx *c, const double lo[3], const double hi[3], double hmax, double *rmax_out,
                        double cs[3], int64_t *nkeys) {
  const int dim = c->frozen.dim;
  double rmax = c->frozen.krad * hmax * (1.0 + 1e-9);
  if (!(rmax > 0.0)) rmax = 1.0;
  *rmax_out = rmax;
  const int axis_cap = dim == 3 ? 1024 : (dim == 2 ? 32768 : (1 << 30));
  Grid g{};
  int RS = c->opt.cell_div > 0 ? c->opt.cell_div : kNeighRS;
  for (int attempt = 0; attempt < 2; attempt++) {
    g = Grid{};
    g.mdim = dim;
    const double cw = rmax / RS;
    bool ok = true;
    for (int a = 0; a < 3; a++) {
      g.periodic[a] = 0;
      if (a >= dim) { g.lo[a] = lo[a]; g.nc[a] = 1; cs[a] = 0; continue; }
      if ((c->box.ghost_mask >> a) & 1) {
        double L = c->box.emax[a] - c->box.emin[a];
        int64_t nc = (int64_t)std::floor(L / cw);
        nc = std::max<int64_t>(1, std::min<int64_t>(nc, axis_cap));
        g.nc[a] = (int)nc;
        g.lo[a] = c->box.emin[a];
        cs[a] = L / (double)nc;
        g.periodic[a] = 1;
        if (RS > 1 && nc < 2 * RS + 1) ok = false;
      } else {
        double ext = hi[a] - lo[a];
        cs[a] = cw;
        if (ext / cs[a] + 1 > axis_cap) cs[a] = ext / (axis_cap - 1) * (1.0 + 1e-9);
        g.nc[a] = (int)std::min<int64_t>((int64_t)std::floor(ext / cs[a]) + 1, axis_cap);
        g.lo[a] = lo[a];
      }
      if (RS > 1 && cs[a] * RS < rmax) ok = false;  // capped axis: cells too small for the stencil
    }
    if (ok || RS == 1) break;
    RS = 1;
  }
  // bound the cell count (sparse sets): coarsen the largest axis
  while ((int64_t)g.nc[0] * g.nc[1] * g.nc[2] > (int64_t)1 << 26) {
    int a = g.nc[0] >= g.nc[1] ? (g.nc[0] >= g.nc[2] ? 0 : 2) : (g.nc[1] >= g.nc[2] ? 1 : 2);
    if (g.periodic[a]) {
      g.nc[a] = std::max(1, g.nc[a] / 2);
      cs[a] = (c->box.emax[a] - c->box.emin[a]) / g.nc[a];
      if (RS > 1 && g.nc[a] < 2 * RS + 1) RS = 1;
    } else {
      cs[a] *= 2;
      g.nc[a] = (int)std::floor((hi[a] - lo[a]) / cs[a]) + 1;
    }
  }
  for (int a = 0; a < 3; a++) {
    g.cs[a] = cs[a];
    g.inv_cs[a] = cs[a] > 0 ? 1.0 / cs[a] : 0.0;
  }
  // sort keys: row (y, z) times nx plus x; 3D rows in tiles of (y, z)
  int64_t nrow = 1;
  if (dim == 3) {
    g.ty = (g.nc[1] + kRowTile - 1) / kRowTile;
    nrow = (int64_t)g.ty * ((g.nc[2] + kRowTile - 1) / kRowTile) * kRowTile * kRowTile;
  } else if (dim == 2) {
    nrow = g.nc[1];
  }
  *nkeys = nrow * g.nc[0];
  return g;
}

// The bits a sort by keys below nkeys has to look at.
static int bits_of(int64_t nkeys) {
  int b = 1;
  while (b < 32 && ((int64_t)1 << b) < nkeys) b++;
  return b;
}

// defer: launch the search without waiting for its read-back (a later
// copy_record brings it); the lists then hold at most nb_cap entries per
// particle, so what runs on them before take_neighbours stays in bounds.
static int build_neighbours(sph_ctx *c, bool defer = false) {
  const int n = (int)c->n;
  const int dim = c->frozen.dim;
  Fields F = c->fields();
  unsigned G = grid_for(n);
  c->ext_built = c->counted = false;
  // 1. wrap escaped real particles, bounding box, max h (striped reductions).
  //    Positions unchanged since the last pass (so none escaped) and h last
  //    set by the previous step (whose k_post1 reduced h_max): nothing to do.
  double lo[3], hi[3], hmax;
  if (c->bbox_version == c->pos_version && c->hmax_version == c->h_version && c->n_real > 0) {
    for (int a = 0; a < 3; a++) { lo[a] = c->last_lo[a]; hi[a] = c->last_hi[a]; }
    hmax = c->next_hmax;
  } else {
    bool wrapped;
    RCHK(wrap_pass(c, F, c->orig[c->cur], lo, hi, &hmax, &wrapped));
    if (wrapped) c->pos_version++;  // keys, records and lists are made anew
    for (int a = 0; a < 3; a++) { c->last_lo[a] = lo[a]; c->last_hi[a] = hi[a]; }
    c->bbox_version = c->pos_version;
  }
  if (!(hmax > 0.0) && c->n_real > 0) return SPH_ERR_Q_NAN_OR_NEG;
  double rmax, cs[3];
  int64_t nkeys;
  const Grid g = search_grid(c, lo, hi, hmax, &rmax, cs, &nkeys);
  c->grid = g;
  RCHK(ensure_cells(c, nkeys));
  // 3. cell keys, sortedness, radix sort + reorder when needed; keys and
  //    cell starts of the same positions on the same grid are still valid
  c->stats.sorted = c->load_moved ? 1 : 0;
  c->load_moved = false;
  const bool keys_kept = c->keys_version == c->pos_version && c->keys_n == n && c->keys_nkeys == nkeys &&
                         same_grid(g, c->keys_grid);
  if (!keys_kept) {
    // Particles that moved since the keys were made are ordered by counting,
    // without asking the host whether their order broke, unless the last
    // fullest cell was crowded; others are checked first and sorted if they
    // must be.  Counting reads and writes every column, which large sets whose
    // moves mostly leave the order pay for each pass: they are checked too
    // (diffusion at rest, 128^3 in FP32, a pass 2.23 ms, counted 2.57; 1M
    // particles in 1D 0.60 and 0.73; at 262k 0.51 and 0.52, at 90k 0.21 and
    // 0.20; 1000^2 hydro, where the grid's changes break it every other pass,
    // counted 1.00, checked and sorted 1.14).
    const bool moves = c->keys_version != c->pos_version;
    const bool counted = moves && (n < 200000 || c->breaks >= 2) && c->fullest > 0 && c->fullest <= kCountedCell &&
                         nkeys < INT32_MAX;
    c->counted = counted;
    int *order_flag = reinterpret_cast<int *>(c->d_stripes + kMovedLL);
    hipLaunchKernelGGL(k_keys, dim3(G), dim3(kBlock), 0, c->stream, F, n, g, c->keys, c->vals, order_flag,
                       counted ? c->ccount : nullptr, c->d_stripes + kFlagSlots);
    const int nxt = 1 - c->cur;
    Fields src = c->fields();
    Fields dst;
    for (int f = 0; f < F_TOTAL; f++) dst.f[f] = c->fbuf[nxt] + (size_t)f * c->npad;
    const double *aux_src = c->aux(0);
    double *aux_dst = c->fbuf[nxt] + (size_t)F_TOTAL * c->npad;
    bool moved = counted;
    if (counted) {
      const int rs = prefix_sum(c, c->ccount, c->cstart, (int)nkeys + 1);
      if (rs != SPH_OK) {  // no room for the scan: the counts are not left behind
        HIPCHK(hipMemsetAsync(c->ccount, 0, sizeof(int) * c->ncell_cap, c->stream));
        return rs;
      }
      hipLaunchKernelGGL(k_cell_list, dim3(G), dim3(kBlock), 0, c->stream, c->keys, c->vals, c->cstart, n, c->vals2);
      hipLaunchKernelGGL(k_move, dim3(G), dim3(kBlock), 0, c->stream, src, dst, aux_src, aux_dst, c->naux,
                         (int)c->npad, c->keys, c->cstart, c->vals2, c->ccount, c->orig[c->cur], c->orig[nxt], n,
                         order_flag);
    } else {
      hipLaunchKernelGGL(k_check_sorted, dim3(std::min(G, 256u)), dim3(kBlock), 0, c->stream, c->keys, n, order_flag);
      HIPCHK(hipMemcpyAsync(c->h_int + 2, order_flag, sizeof(int), hipMemcpyDeviceToHost, c->stream));
      HIPCHK(wait_stream(c));
      moved = c->h_int[2] != 0;
      if (moves) note_order(c, moved);
    }
    if (moved && !counted) {
      size_t bytes = c->sort_tmp_bytes;
      HIPCHK(hipcub::DeviceRadixSort::SortPairs(c->sort_tmp, bytes, c->keys, c->keys2, c->vals, c->vals2, n, 0,
                                                bits_of(nkeys), c->stream));
      hipLaunchKernelGGL(k_reorder, dim3(G), dim3(kBlock), 0, c->stream, src, dst, c->vals2, c->orig[c->cur],
                         c->orig[nxt], n, (int)F_TOTAL);
      // auxiliary arrays ride along in groups of up to 32
      for (int k0 = 0; k0 < c->naux; k0 += F_TOTAL) {
        Fields as{}, ad{};
        const int m = std::min((int)F_TOTAL, c->naux - k0);
        for (int f = 0; f < m; f++) {
          as.f[f] = c->fbuf[c->cur] + (size_t)(F_TOTAL + k0 + f) * c->npad;
          ad.f[f] = c->fbuf[nxt] + (size_t)(F_TOTAL + k0 + f) * c->npad;
        }
        hipLaunchKernelGGL(k_reorder, dim3(G), dim3(kBlock), 0, c->stream, as, ad, c->vals2, c->orig[c->cur],
                           (int64_t *)nullptr, n, m);
      }
      std::swap(c->keys, c->keys2);
    }
    if (moved) {
      c->cur = nxt;
      F = c->fields();
      c->stats.sorted = 1;
    }
    if (!counted)
      hipLaunchKernelGGL(k_cell_start, dim3(grid_for(n + 1)), dim3(kBlock), 0, c->stream, c->keys, n, (uint32_t)nkeys,
                         c->cstart);
    c->keys_version = c->pos_version;
    c->keys_grid = g;
    c->keys_n = n;
    c->keys_nkeys = nkeys;
  }
  // the v / B flags are computed again only when v or B may have changed
  c->flags_pending = c->flags_version != c->vb_version;
  if (c->flags_pending && keys_kept && !c->flags_clear)  // else k_keys cleared them
    HIPCHK(hipMemsetAsync(c->d_stripes + kFlagSlots, 0, sizeof(long long) * kStripes, c->stream));
  // rows and cells within r_max (1 + 1e-6) of a cell; imaged axes at most
  // one wrap away
  int rc[3];
  for (int d = 0; d < 3; d++) {
    rc[d] = d < dim && cs[d] > 0 ? (int)std::ceil(rmax * (1.0 + 1e-6) / cs[d]) : 0;
    if (g.periodic[d]) rc[d] = std::min(rc[d], g.nc[d]);
  }
  const FixFrame ff = fix_frame(c, g, dim, rc, rmax);
  const bool pos_kept = keys_kept && c->prep_version == c->pos_version && c->prep_cur == c->cur &&
                        c->prep_n == n && same_grid(g, c->prep_grid) &&
                        std::memcmp(&ff, &c->ff, sizeof(ff)) == 0;
  c->ff = ff;
  // the start-state copy only for c1simple (a deferred search is
  // c1advanced's, whose first sweep reads the fields); the counters cleared
  // with the regions of the first batch of Newton sweeps when they follow
  // this search (c1advanced)
  const int zlast = defer ? first_batch_last(c) : 0;
  hipLaunchKernelGGL(k_prep, dim3(G), dim3(kBlock), 0, c->stream, F, c->orig[c->cur], n, c->n_real, c->box, g, dim,
                     c->pm, c->h0, c->pf, c->real, defer ? nullptr : c->st[0], c->tr[0], c->pfix, ff, c->s1[0],
                     c->eps,
                     c->flags_pending ? c->d_stripes + kFlagSlots : nullptr, c->d_stripes, kZeroLL,
                     c->d_sweep + kSweepRegion, zlast * kSweepRegion, c->d_red, pos_kept ? 0 : 1);
  c->red_ready = true;
  c->flags_clear = false;
  c->sweeps_zeroed = zlast;
  c->prep_version = c->pos_version;
  c->prep_cur = c->cur;
  c->prep_n = n;
  c->prep_grid = g;
  // 4. the extended grid: rc ghost cells on each side of every axis (the
  //    periodic images on an imaged axis, empty on a walled one), so every
  //    stencil row of the search is one range of records and no row or cell
  //    needs a bounds test; rebuilt when the positions, their order, the
  //    grid or the stencil change
  bool use_ext = !c->lane_search;
  ExtGrid xg{};
  int64_t ncells = 1;
  for (int d = 0; d < 3; d++) {
    xg.gh[d] = rc[d];
    xg.ne[d] = g.nc[d] + 2 * xg.gh[d];
    xg.lenf[d] = g.periodic[d] ? (float)(c->box.emax[d] - c->box.emin[d]) : 0.f;
    ncells *= xg.ne[d];
  }
  // offsets are ints (every record has at most 27 copies) and the search
  // addresses the cell starts with 32-bit byte offsets
  if (ncells + 1 > INT32_MAX / 4 || (int64_t)n * 27 > INT32_MAX) use_ext = false;
  if (use_ext) {
    const bool ext_kept = c->ext_version == c->pos_version && c->ext_cur == c->cur && c->ext_n == n &&
                          same_grid(g, c->ext_grid) && std::memcmp(&xg, &c->ext_g, sizeof(xg)) == 0;
    if (!ext_kept) {
      const int E = (int)ncells;
      if ((size_t)E + 1 > c->ext_cells_cap) {
        if (c->ext_count) { (void)hipFree(c->ext_count); c->ext_count = nullptr; }
        if (c->ecs) { (void)hipFree(c->ecs); c->ecs = nullptr; }
        c->ext_cells_cap = 0;
        RCHK(dev_alloc((void **)&c->ext_count, sizeof(int) * ((size_t)E + 1)));
        RCHK(dev_alloc((void **)&c->ecs, sizeof(int) * ((size_t)E + 1)));
        c->ext_cells_cap = (size_t)E + 1;
      }
      hipLaunchKernelGGL(k_ext_count, dim3(grid_for(E + 1)), dim3(kBlock), 0, c->stream, g, xg, c->cstart, E,
                         c->ext_count, c->d_stripes + kFullLL);
      RCHK(prefix_sum(c, c->ext_count, c->ecs, E + 1));
      // With records already held (an eighth more than the last grid's) the
      // step does not wait for their number: what does not fit is left out, and
      // the search's error word then has it done again with the exact room.
      int64_t total = c->ext_total;
      const bool waits = !defer || c->ext_exact || c->ext_rec_cap == 0 || c->ext_total < 0;
      c->ext_exact = false;
      if (waits) {
        HIPCHK(hipMemcpyAsync(c->h_int + kExtTotalInt, c->ecs + E, sizeof(int), hipMemcpyDeviceToHost, c->stream));
        HIPCHK(wait_stream(c));
        total = c->h_int[kExtTotalInt];
      }
      // 8 records of padding: the search reads whole batches past a row's
      // end.  The search addresses records with 32-bit byte offsets, so a
      // larger set (over 2^28 records) takes the per-lane traversal.
      if (waits && (total + 8) * (int64_t)sizeof(float4) > (int64_t)UINT32_MAX) {
        total = -1;
      } else {
        if (waits && (size_t)total + 8 > c->ext_rec_cap) {
          if (c->erec) { (void)hipFree(c->erec); c->erec = nullptr; }
          c->ext_rec_cap = 0;
          const size_t cap = std::min<size_t>((size_t)total + 8 + (size_t)total / 8, UINT32_MAX / sizeof(float4));
          RCHK(dev_alloc((void **)&c->erec, sizeof(float4) * cap));
          c->ext_rec_cap = cap;
        }
        total = std::max<int64_t>(total, 0);
        hipLaunchKernelGGL(k_ext_fill, dim3(grid_for(E + 1)), dim3(kBlock), 0, c->stream, g, xg, c->cstart, c->ecs,
                           c->pf, E, (int)(c->ext_rec_cap - 8), c->erec, step_err(c) + kErrSearch,
                           c->d_stripes + kExtLL);
        c->ext_built = true;
      }
      c->ext_total = total;
      // a grid being filled counts as kept once its size is read back
      // (finish_neighbours): a step that ends before that leaves none
      c->ext_version = c->ext_built ? 0 : c->pos_version;
      c->ext_cur = c->cur;
      c->ext_n = n;
      c->ext_grid = g;
      c->ext_g = xg;
    }
    if (c->ext_total < 0) use_ext = false;
  }
  c->stats.ext_records = use_ext ? c->ext_total : 0;
  // 5. neighbour lists; grow the storage and redo if any list overflowed
  if (c->nb_cap == 0) RCHK(ensure_nb(c, std::min(c->maxneib, dim == 3 ? 160 : (dim == 2 ? 48 : 16))));
  for (int attempt = 0; attempt < 2; attempt++) {
    if (attempt > 0) {  // k_prep cleared the first search's counters
      HIPCHK(hipMemsetAsync(c->d_stripes + kSearchLL, 0, sizeof(long long) * 2 * kStripes, c->stream));
      HIPCHK(hipMemsetAsync(step_err(c) + kErrSearch, 0, sizeof(int), c->stream));
    }
    NeighArgs a;
    a.hs = c->h0; a.real = c->real; a.cstart = c->cstart;
    a.rx = rc[0]; a.ry = rc[1]; a.rz = rc[2];
    a.ecs = use_ext ? c->ecs : nullptr;
    a.erec = use_ext ? c->erec : nullptr;
    for (int d = 0; d < 3; d++) { a.ne[d] = xg.ne[d]; a.gh[d] = xg.gh[d]; }
    // a position in cell units is FP32: its rounding stays below 2^-23 of the
    // cell count along the axis
    for (int d = 0; d < 3; d++) a.mcell[d] = (float)(1e-4 + 1e-6 * g.nc[d]);
    a.g = g; a.b = c->box; a.krad = c->frozen.krad; a.n = n; a.npad = (int)c->npad; a.cap = c->nb_cap;
    // FP32 search records: coordinates relative to the grid origin lie within
    // the grid span S (imaged axes: the box), images within 2 S; each of the
    // roundings involved is at most 2^-24 S, six of them at most, so
    // 2^-21 S bounds the error of an FP32 separation component.
    double span = 0.0;
    for (int d = 0; d < dim; d++) span = std::max(span, g.nc[d] * cs[d]);
    a.delta = std::ldexp(span, -21);
    for (int d = 0; d < 3; d++)  // only imaged axes shift (elsewhere the shift is 0, keep 0 * lenf finite)
      a.lenf[d] = g.periodic[d] ? (float)(c->box.emax[d] - c->box.emin[d]) : 0.f;
    a.maxneib = c->maxneib; a.err = step_err(c) + kErrSearch; a.stripes = c->d_stripes + kSearchLL;
    // the search's own events (loop 1 reuses 5 and 6 before a deferred read-back is taken)
    HIPCHK(mark(c, 4));
#define NEIGH(D)                                                                                              \
  if (use_ext) hipLaunchKernelGGL((k_neigh<D, true>), dim3(G), dim3(kBlock), 0, c->stream, a, c->pm, c->pf, c->nb, c->cnt); \
  else hipLaunchKernelGGL((k_neigh<D, false>), dim3(G), dim3(kBlock), 0, c->stream, a, c->pm, c->pf, c->nb, c->cnt)
    if (dim == 1) { NEIGH(1); }
    else if (dim == 2) { NEIGH(2); }
    else { NEIGH(3); }
#undef NEIGH
    HIPCHK(mark(c, 7));
    // pair counts, list lengths, error words and k_prep's flags: deferred,
    // they come back with the step's next record copy
    if (defer) {
      c->neigh_pending = true;
      return SPH_OK;
    }
    HIPCHK(copy_record(c, 0));
    HIPCHK(wait_stream(c));
    const long long *ll = c->h_rec;
    const int fin = finish_neighbours(c, ll, copied_err(ll, 0, kErrSearch));
    if (fin != kRedoNeigh) return fin;
  }
  return SPH_ERR_HIP;
}

// ------------------------------------------------------------ step: loops
// The equation set of loop 2 where one is fixed at compile time (2D and 3D:
// hydro, magnetohydro, hydro with FLD), else -1.
static int loop2_terms(const sph_ctx *c, const Phys &P) {
  if (c->loop2_generic || P.dim < 2) return -1;
  const int terms = (P.hydro ? 1 : 0) | (P.magneto ? 2 : 0) | (P.diff ? 4 : 0) | (P.fld ? 8 : 0);
  return terms == kSpecHydro || terms == kSpecMhd || terms == kSpecHydroFld ? terms : -1;
}

// Whether loop 2 runs its general form (k_loop2 with every term, or a fixed
// equation set): all but diffusion alone with a Hessian operator.
static bool loop2_general(const Phys &P) {
  return !(P.diff && !P.hydro && !P.artts && !P.magneto && !P.fld &&
           (P.ddw == 400 || P.ddw == 401 || P.ddw == 402));
}

// Whether loop 2 is k_loop2_fab: fab with one tensor for every pair and no
// velocity term, by the v and B flags last read.
static bool loop2_fab(const sph_ctx *c, const Phys &P) {
  if (loop2_general(P) || P.ddw != 400) return false;
  const bool reads_v = P.adden && (c->step_flags & 1) != 0;
  const bool reads_b = P.diso == 0 && (c->step_flags & 2) != 0;
  return !reads_v && !reads_b;
}

// Lanes per particle of the pair loops (1, 4 or 8).  One lane walks a list
// alone: on a lattice in row order the wave's 64 k-th neighbours lie side by
// side and every list is as long, and the loop is bound by its arithmetic.
// Where lists differ the wave waits for its longest and its k-th neighbours
// drift apart; several lanes of one particle read runs of its cell rows
// instead, and few particles then still fill the chip.  Short lists leave a lane
// little more to do than what every lane repeats.  So the lines lie by the
// particles (1D: always one lane), by the length of a list as kernel and hfac
// give it (short: M4 at hfac 1.0, 33 in 3D; medium: M4 at 1.2, 58; long: M6, 113
// and more; 2D: M4 13 to 18, M6 28) and by how even the lists are.  Measured,
// one lane against several, loop 2 where nothing else is said (us):
//   3D below 40k particles: 8 (2nw FP64 at 30^3 108 against 49).
//   Particles that move (hydro, MHD, FLD): 8 (FP32 MHD tube of 1M 3440 against
//     1640, sweeps 2650 against 1570; FP64 hydro tube of 300k 1118 against
//     515).  FP32 takes 1 for even lists from 170k (lattice, hydro: 56^3 127 and
//     135, 64^3 154 and 192, 128^3 1207 and 1500; sweeps with grad T 64^3 69 and
//     92), medium ones from 110k (56^3 60 and 76), short ones, also disordered,
//     from 90k (46^3 32 and 34, 56^3 jittered 45 and 57); its sweeps with grad T
//     sooner (medium, jittered 56^3 37 and 48; short, a glass 31 and 38).  FP64
//     loop 1: short, disordered from 90k (56^3 28 and 32, 80^3 53 and 74), medium,
//     even from 200k (64^3 44 and 53); a fixed set's loop 2: the short ones (80^3
//     lattice 138 and 171, jittered 166 and 175).  FP64 sets that are not fixed
//     at compile time: even from 110k (hydro with diffusion 46^3 208 and 194, 58^3
//     338 and 364, 100^3 1522 and 1862), a glass from 500k, medium 200k, short
//     100k (100^3 jittered 1609 and 1738; medium 64^3 266 and 304; short 131 and
//     187), random particles 8 (tube of 300k 1480 and 1022).
//   General form without hydro: 4.  FP64: even 1 from 110k (2nw: 48^3 141 and
//     159, 64^3 272 and 337; FLD 46^3 200 and 179, 64^3 387 and 436), medium and
//     disordered too from 200k (2nw 64^3 174 and 204), short ones from 75k (46^3
//     46 and 51).  FP32: even 1 from 150k (2nw: 52^3 124 and 114, 54^3 127 and 135,
//     100^3 722 and 823; FLD 58^3 152 and 173; jittered 64^3 320 and 222), medium
//     and short 120k (short, jittered 56^3 43 and 55).  The 2nw operators 1 from
//     300k on also where lists are uneven (FP64 80^3 616 and 661).
//   fab (and FP64 n2w, fw): 4, even 1 from 700k (FP32 lattice 88^3 172 and 174,
//     100^3 236 and 254; jittered 100^3 330 and 243; FP64 lattice 100^3 366 and
//     361, 128^3 666 and 731; jittered 128^3 1025 and 741), medium from 150k in
//     FP32 and 200k in FP64 (64^3 36 and 43, 50 and 57), short and disordered ones
//     from 100k and 150k (56^3 22 and 25; 80^3 61 and 75; FP64 n2w a glass too,
//     80^3 122 and 135).
//   n2w and fw in FP32: 4 below 225k (medium 200k, short 150k), then 1 (60^3 102
//     and 99, 64^3 104 and 113, 100^3 393 and 431, jittered 387 and 409; short
//     64^3 37 and 46); fab there with velocities or a B of its own per particle 4,
//     even lists 1 from the same lines (with velocities 58^3 131 and 124, 64^3 142
//     and 160, 80^3 315 and 356; jittered 390 and 346).
//   Loop 1 in FP64 without hydro: as fab (128^3 677 and 723, jittered 1015 and
//     733; medium 64^3 50 and 55; short 64^3 jittered 37 and 41).
//   2D: 8 below 40k particles (M6 64^2: sweeps 0.056 -> 0.025 ms, loop 2 0.029 ->
//     0.011), 4 below 150k (256^2 0.051 -> 0.041 and 0.032 -> 0.025), then 1 (512^2
//     0.078 against 0.089, 0.069 against 0.071); M4 90k (387^2 30 and 35).
// FP32: loop 1 keeps its sums in list order on 8 lanes (k_loop1), which pays
// below 100k particles in 3D diffusion (46^3 45.8 against 43, 58^3 58 against
// 75; medium 50k, short 36k: 40^3 20 and 22, 15 and 18) and below 40k in 2D;
// loop 2 of 2D stays on one lane, since
// the accelerations of a 2D set at rest are the small remainder of large terms
// and another order's rounding moves them by 4e-5.  The same for loop 2 of
// particles that move where the equation set is not fixed (k_loop2).
// `even` is of the step's own lists wherever it changes how a sum is rounded
// (run_advanced), so that a step's bits depend on nothing before it.
static int loop_lanes(const sph_ctx *c, const Phys &P, bool loop2, int even) {
  const int64_t n = c->n;
  const bool mixed = c->opt.precision == 1;
  if (P.dim == 1 || (mixed && loop2 && P.dim == 2)) return 1;
  const double reach = P.krad * P.hfac;
  if (P.dim == 2) {
    if (n < 40000) return 8;
    return !mixed && n < (kPi * reach * reach < 22.0 ? 90000 : 150000) ? 4 : 1;
  }
  const double near = 4.0 / 3.0 * kPi * reach * reach * reach;
  const int len = near < 45.0 ? 0 : (near < 90.0 ? 1 : 2);
  // n at or past the line of its list length (short, medium, long)
  auto past = [&](int64_t s, int64_t m, int64_t l) { return n >= (len == 0 ? s : (len == 1 ? m : l)); };
  const int64_t never = INT64_MAX;
  const bool grad_t = P.diff || P.fld;
  if (P.hydro) {
    const bool fixed_set = loop2_terms(c, P) >= 0;
    if (mixed) {
      if (loop2 && !fixed_set) return 1;
      if (!loop2 && grad_t && even >= (len == 0 ? kGlass : kNearEven) && past(90000, 100000, never)) return 1;
      return even >= (len == 0 ? kNearEven : kEven) && past(90000, 110000, 170000) ? 1 : 8;
    }
    if (loop2 && !fixed_set)
      return (even >= kEven && past(90000, 110000, 110000)) || (even >= kGlass && past(100000, 200000, 500000)) ? 1 : 8;
    if (even >= kNearEven && past(90000, never, never)) return 1;
    return !loop2 && even >= kEven && past(never, 200000, never) ? 1 : 8;
  }
  if (mixed && !loop2) return past(36000, 50000, 100000) ? 1 : 8;
  if (n < 40000) return 8;
  if (loop2 && loop2_general(P)) {
    if (even >= (len == 0 ? kNearEven : kEven) && (mixed ? past(120000, 120000, 150000) : past(75000, 90000, 110000)))
      return 1;
    if (!mixed && even >= kGlass && past(200000, 200000, never)) return 1;
    return !P.fld && (P.ddw == 403 || P.ddw == 404) && P.diff && n >= 300000 ? 1 : 4;
  }
  if (mixed && !loop2_fab(c, P)) return past(150000, 200000, 225000) && (P.ddw != 400 || even >= kEven) ? 1 : 4;
  if (len == 0) {
    const int enough = loop2 && !mixed && P.ddw != 400 ? kGlass : kNearEven;
    return even >= enough && n >= (mixed ? 100000 : 150000) ? 1 : 4;
  }
  return even >= kEven && (mixed ? past(never, 150000, 700000) : past(never, 200000, 700000)) ? 1 : 4;
}

// The evennesses (a bit each) whose lanes round the sums as those of `even` do:
// FP32 sums of loop 1, and of loop 2 of a fixed equation set, are in the list's
// order on any lanes.
static int same_rounding(const sph_ctx *c, const Phys &P, int even) {
  const bool mixed = c->opt.precision == 1;
  int same = 0;
  for (int e = kRandom; e <= kEven; e++) {
    bool eq = (mixed && loop2_terms(c, P) >= 0) || loop_lanes(c, P, true, e) == loop_lanes(c, P, true, even);
    eq = eq && (mixed || loop_lanes(c, P, false, e) == loop_lanes(c, P, false, even));
    if (eq) same |= 1 << e;
  }
  return same;
}
constexpr int kAnyLists = (1 << (kEven + 1)) - 1;

// fn(constant G) for lanes = 1, 4 (where HAS4) or 8 (HAS8): the counts
// loop_lanes can give a kernel
template <bool HAS4, bool HAS8, typename Fn>
static void with_lanes(int lanes, Fn fn) {
  if constexpr (HAS8) {
    if (lanes == 8) return fn(std::integral_constant<int, 8>{});
  }
  if constexpr (HAS4) {
    if (lanes == 4) return fn(std::integral_constant<int, 4>{});
  }
  fn(std::integral_constant<int, 1>{});
}

template <int DIM, int KT>
static void launch_loop1(sph_ctx *c, Loop1Args<double4> &a, int grad, bool simple, Fields F) {
  bool mixed = c->opt.precision == 1;
  if (simple) {
    // FP32 sums keep the list order: one lane.  FP64: loop 1's lanes (1M
    // particles in 1D, us: one lane 32, eight 76; 1000^2 82, 122), of uneven lists
    // where they are long (100^3 lattice 302, four 267, jittered 403, 279)
    const double reach = a.p.krad * a.p.hfac;
    const bool long_lists = 4.0 / 3.0 * kPi * reach * reach * reach >= 90.0;
    const int lanes = mixed ? 1 : loop_lanes(c, a.p, false, long_lists ? kRandom : std::max(c->even, 0));
#define L1S(GR, PT)                                                                                          \
  with_lanes<DIM != 1 && std::is_same_v<PT, double>, DIM != 1 && std::is_same_v<PT, double>>(lanes, [&](auto l) { \
    constexpr int G = decltype(l)::value;                                                                    \
    hipLaunchKernelGGL((k_loop1_simple<DIM, KT, GR, PT, G>), dim3(grid_for((int64_t)a.n * G)), dim3(kBlock), 0, \
                       c->stream, a, F);                                                                     \
  })
    if (mixed) {
      if (grad == 0) { L1S(0, float); } else if (grad == 1) { L1S(1, float); } else { L1S(2, float); }
    } else {
      if (grad == 0) { L1S(0, double); } else if (grad == 1) { L1S(1, double); } else { L1S(2, double); }
    }
#undef L1S
    return;
  }
  const int lanes = loop_lanes(c, a.p, false, std::max(c->even, 0));
#define L1(GR, PT)                                                                                           \
  with_lanes<DIM != 1 && std::is_same_v<PT, double>, DIM != 1>(lanes, [&](auto l) {                          \
    constexpr int G = decltype(l)::value;                                                                    \
    hipLaunchKernelGGL((k_loop1<DIM, KT, GR, PT, G>), dim3(grid_for((int64_t)a.n * G)), dim3(kBlock), 0, c->stream, a); \
  })
  if (mixed) {
    if (grad == 0) { L1(0, float); } else if (grad == 1) { L1(1, float); } else { L1(2, float); }
  } else {
    if (grad == 0) { L1(0, double); } else if (grad == 1) { L1(1, double); } else { L1(2, double); }
  }
#undef L1
}

template <int DIM>
static void launch_loop1_k(sph_ctx *c, Loop1Args<double4> &a, int grad, bool simple, Fields F) {
  if (c->kt == KT_M4) launch_loop1<DIM, KT_M4>(c, a, grad, simple, F);
  else if (c->kt == KT_M6) launch_loop1<DIM, KT_M6>(c, a, grad, simple, F);
  else launch_loop1<DIM, KT_GAUSS>(c, a, grad, simple, F);
}

// c1simple (circuit1.f90:227-305): one pass, grad T only with diffusion and
// the 2nw operators; the search is checked first (it writes h, rho, om in
// place), so this waits for the pass.
static int run_loop1_simple(sph_ctx *c, const Phys &P) {
  const int n = (int)c->n;
  Fields F = c->fields();
  Loop1Args<double4> a{};
  a.pm = c->pm; a.h0 = c->h0; a.real = c->real; a.nb = c->nb; a.cnt = c->cnt; a.eps = c->eps;
  a.dtdx = F.f[F_DTDX]; a.dtdy = F.f[F_DTDY]; a.dtdz = F.f[F_DTDZ]; a.err = step_err(c) + kErrLoop1;
  a.b = c->box; a.p = P; a.n = n; a.npad = (int)c->npad;
  const int grad = (P.diff && P.ddw == 403) ? 1 : ((P.diff && P.ddw == 404) ? 2 : 0);
  a.cur = c->st[0];
  a.next = c->st[1];
  HIPCHK(mark(c, 5));
  if (P.dim == 1) launch_loop1_k<1>(c, a, grad, true, F);
  else if (P.dim == 2) launch_loop1_k<2>(c, a, grad, true, F);
  else launch_loop1_k<3>(c, a, grad, true, F);
  HIPCHK(mark(c, 6));
  c->final_st = c->st[0];
  c->stats.sweeps = 0;
  HIPCHK(hipMemcpyAsync(c->h_ll, c->d_stripes + kErrLL, sizeof(long long) * 4, hipMemcpyDeviceToHost, c->stream));
  HIPCHK(wait_stream(c));
  RCHK(take_neighbours(c));
  c->stats.ms_k_loop1 = elapsed(c, c->ev[5], c->ev[6]);
  c->stats.loop1_pairs = c->stats.n_pairs;
  return map_err(copied_err(c->h_ll, kErrLL, kErrLoop1));
}

// Sweeps first..last of c1advanced (circuit1.f90:104-211) on the stream with
// no host round trip: each sweep runs only if the one before left a particle
// active (while maxval(eps) > tol, circuit1.f90:114) and no error stopped the
// search or loop 1 (k_loop1 decides on the device); their counters go to
// the sweep regions, zeroed here first (by k_prep for a step's first batch).
static void launch_sweeps(sph_ctx *c, const Phys &P, int first, int last) {
  const int n = (int)c->n;
  Fields F = c->fields();
  Loop1Args<double4> a{};
  a.pm = c->pm; a.h0 = c->h0; a.real = c->real; a.nb = c->nb; a.cnt = c->cnt; a.eps = c->eps;
  a.dtdx = F.f[F_DTDX]; a.dtdy = F.f[F_DTDY]; a.dtdz = F.f[F_DTDZ]; a.err = step_err(c) + kErrLoop1;
  a.b = c->box; a.p = P; a.n = n; a.npad = (int)c->npad;
  a.tol = c->opt.newton_tol > 0 ? c->opt.newton_tol : (c->opt.precision == 1 ? 1e-6 : 1e-8);
  a.serr = step_err(c) + kErrSearch;
  a.which = c->d_int + kWhichInt;
  const int grad = (P.diff || P.fld) ? (P.ddw == 404 ? 2 : 1) : 0;
  const int nreg = (last - first + 1) * kSweepRegion;
  if (!(first == 1 && last <= c->sweeps_zeroed))
    hipLaunchKernelGGL(k_zero_ll, dim3((nreg + 255) / 256), dim3(256), 0, c->stream,
                       c->d_sweep + (size_t)first * kSweepRegion, nreg);
  c->sweeps_zeroed = 0;
  tolerate(mark(c, 9));
  for (int it = first; it <= last; it++) {
    a.cur = c->st[(it - 1) & 1];
    a.next = c->st[it & 1];
    // the first sweep reads its start state from the fields (unchanged until
    // the tail's k_post1, which a redone search leaves idle)
    const bool s1st = it == 1;
    a.f_h = s1st ? F.f[F_H] : nullptr;
    a.f_den = s1st ? F.f[F_DEN] : nullptr;
    a.f_om = s1st ? F.f[F_OM] : nullptr;
    a.f_t = s1st ? F.f[F_T] : nullptr;
    a.trc = c->tr[(it - 1) & 1];
    a.trn = c->tr[it & 1];
    a.s1c = c->s1[(it - 1) & 1];
    a.s1n = c->s1[it & 1];
    a.pfix = c->pfix;
    a.ff = c->ff;
    a.stripes = c->d_sweep + (size_t)it * kSweepRegion;
    a.prev = it > 1 ? c->d_sweep + (size_t)(it - 1) * kSweepRegion : nullptr;
    a.sweep = it;
    if (P.dim == 1) launch_loop1_k<1>(c, a, grad, false, F);
    else if (P.dim == 2) launch_loop1_k<2>(c, a, grad, false, F);
    else launch_loop1_k<3>(c, a, grad, false, F);
  }
  tolerate(mark(c, 10));
}

template <int DIM, int KT, int MODE, typename PT, typename V4>
static void launch_loop2_p(sph_ctx *c, int lanes, const Loop2Args<V4> &a) {
  constexpr bool F64 = std::is_same_v<PT, double>, MANY = DIM == 3 || (DIM == 2 && F64);
  constexpr bool MOVING3 = DIM == 3 && MODE >= MODE_SPEC;  // one lane or eight
  with_lanes<MANY && !MOVING3, MANY>(lanes, [&](auto l) {
    constexpr int G = decltype(l)::value;
    const dim3 B(grid_for(c->n * G)), T(kBlock);
    if constexpr (MODE == MODE_FAB) hipLaunchKernelGGL((k_loop2_fab<DIM, KT, PT, V4, G>), B, T, 0, c->stream, a);
    else hipLaunchKernelGGL((k_loop2<DIM, KT, PT, V4, MODE, G>), B, T, 0, c->stream, a);
  });
}
template <int DIM, int KT, int MODE>
static void launch_loop2(sph_ctx *c, int lanes, void *args) {
  if (c->opt.precision == 1)
    launch_loop2_p<DIM, KT, MODE, float, float4>(c, lanes, *(Loop2Args<float4> *)args);
  else
    launch_loop2_p<DIM, KT, MODE, double, double4>(c, lanes, *(Loop2Args<double4> *)args);
}
template <int DIM, int MODE>
static void launch_loop2_k(sph_ctx *c, int lanes, void *args) {
  if (c->kt == KT_M4) launch_loop2<DIM, KT_M4, MODE>(c, lanes, args);
  else if (c->kt == KT_M6) launch_loop2<DIM, KT_M6, MODE>(c, lanes, args);
  else launch_loop2<DIM, KT_GAUSS, MODE>(c, lanes, args);
}
template <int MODE>
static void launch_loop2_d(sph_ctx *c, int dim, int lanes, void *args) {
  if (dim == 1) launch_loop2_k<1, MODE>(c, lanes, args);
  else if (dim == 2) launch_loop2_k<2, MODE>(c, lanes, args);
  else launch_loop2_k<3, MODE>(c, lanes, args);
}
// modes built in 2D and 3D only
template <int MODE>
static void launch_loop2_d23(sph_ctx *c, int dim, int lanes, void *args) {
  if (dim == 2) launch_loop2_k<2, MODE>(c, lanes, args);
  else launch_loop2_k<3, MODE>(c, lanes, args);
}

template <typename V4>
static int run_post_and_loop2(sph_ctx *c, const Phys &P, const long long *pending, int even) {
  const int n = (int)c->n;
  Fields F = c->fields();
  unsigned G = grid_for(n);
  // reference c1 for isothermal EOS reads particle 1's sound speed (eos.f90:43)
  double c1 = 0.0;
  if (c->do_eos && c->eos_iso && n > 0) {
    HIPCHK(hipMemsetAsync(c->d_int + 3, 0, sizeof(int), c->stream));
    hipLaunchKernelGGL(k_find_orig, dim3(G), dim3(kBlock), 0, c->stream, c->orig[c->cur], n, (int64_t)0,
                       c->d_int + 3);
    RCHK(read_ints(c, 3, 1));
    HIPCHK(hipMemcpyAsync(c->h_ll + 4, F.f[F_C] + c->h_int[3], sizeof(double), hipMemcpyDeviceToHost, c->stream));
    HIPCHK(hipStreamSynchronize(c->stream));
    memcpy(&c1, c->h_ll + 4, sizeof(double));
  }
  // which j-side packs loop 2 may gather (must match k_loop2)
  const bool generic = loop2_general(P);
  const bool want_v = P.adden || P.artts || P.hydro || P.magneto;
  const bool want_q2 = generic && ((P.diff && P.fld) || P.artts);
  const bool want_q3 = generic && P.diff && (P.fld || P.ddw == 403 || P.ddw == 404);
  const bool want_q4 = P.magneto || (P.diff && !P.fld && P.diso == 0);
  // k_prep's flags (v and B are what they were there): the diffusion-only
  // loop 2 reads v only where it is non-zero and B only where it varies
  const long long fl = c->step_flags;
  // q0 feeds the generic loop, and in FP64 also the adjoint and batched
  // operators sph_diff_prepare builds after its step; the diffusion loops
  // read pd alone
  V4 *q0 = !generic && (std::is_same_v<V4, float4> || !c->keep_q0) ? nullptr : (V4 *)c->q[0];
  V4 *q1 = want_v && (generic || (fl & 1)) ? (V4 *)c->q[1] : nullptr;
  V4 *q2 = want_q2 ? (V4 *)c->q[2] : nullptr;
  V4 *q3 = want_q3 ? (V4 *)c->q[3] : nullptr;
  V4 *q4 = want_q4 && (generic || (fl & 2)) ? (V4 *)c->q[4] : nullptr;
  long long *none = nullptr;
  PostSel sel{};
  sel.fin0 = P.adden ? c->st[0] : c->final_st;
  sel.fin1 = c->st[1];
  sel.which = P.adden ? c->d_int + kWhichInt : nullptr;
  sel.serr = step_err(c) + kErrSearch;
  sel.err1 = step_err(c) + kErrLoop1;
  sel.pending = pending;
  sel.lists = c->d_stripes + kSearchLL;
  sel.n_real = c->n_real;
  sel.even = even == kAnyLists ? 0 : even;
  sel.go = c->d_int + kGoInt;
  hipLaunchKernelGGL(k_post1<V4>, dim3(G), dim3(kBlock), 0, c->stream, F, sel, c->real, n, P.adden ? 1 : 0,
                     c->do_eos, c->eos_iso, c1, P.gamma, q0, q1, q2, q3, q4,
                     generic || std::is_same_v<V4, float4> ? nullptr : c->pd,
                     generic ? nullptr : c->trd, generic || !std::is_same_v<V4, float4> ? nullptr : c->s2, none,
                     c->d_stripes + kHmaxLL);
  if (P.diff && P.fld && P.diso != 1) return SPH_ERR_FLD_ANISO;
  if (P.diff && !(P.ddw >= 400 && P.ddw <= 404)) return SPH_ERR_BAD_DDW;
  Loop2Args<V4> a{};
  a.pm = c->pm; a.real = c->real; a.nb = c->nb; a.cnt = c->cnt;
  a.q0 = q0; a.q1 = q1; a.q2 = q2; a.q3 = q3; a.q4 = q4;
  a.pd = generic ? nullptr : c->pd;
  a.trd = generic ? nullptr : c->trd;
  a.pfix = c->pfix;
  a.s2 = c->s2;
  a.ff = c->ff;
  a.v_nonzero = (fl & 1) ? 1 : 0;
  a.b_uniform = (fl & 2) ? 0 : 1;
  // loop 2's error word and k_post1's h_max stripes: cleared by this step's k_prep
  a.go = c->d_int + kGoInt;
  a.out = F; a.energy_part = c->energy_part; a.err = step_err(c) + kErrLoop2; a.b = c->box; a.p = P; a.n = n;
  a.npad = (int)c->npad;
  HIPCHK(mark(c, 5));
  const bool fab = loop2_fab(c, P);  // the loop without run-time choices
  const int terms = generic ? loop2_terms(c, P) : -1;
  const int lanes = loop_lanes(c, P, true, std::max(c->even, 0));
  if (terms == kSpecHydro) launch_loop2_d23<MODE_SPEC + kSpecHydro>(c, P.dim, lanes, &a);
  else if (terms == kSpecMhd) launch_loop2_d23<MODE_SPEC + kSpecMhd>(c, P.dim, lanes, &a);
  else if (terms == kSpecHydroFld) launch_loop2_d23<MODE_SPEC + kSpecHydroFld>(c, P.dim, lanes, &a);
  else if (generic) launch_loop2_d<MODE_GENERIC>(c, P.dim, lanes, &a);
  else if (fab) launch_loop2_d<MODE_FAB>(c, P.dim, lanes, &a);
  else launch_loop2_d<MODE_DIFF>(c, P.dim, lanes, &a);
  HIPCHK(mark(c, 6));
  // energy, error bits and h_max in one record of d_stripes, which the
  // caller's copy_record brings back with the step's closing sync
  hipLaunchKernelGGL(k_step_close, dim3(1), dim3(256), 0, c->stream, c->energy_part, (int)grid_for((int64_t)n * lanes),
                     step_err(c) + kErrLoop2, c->d_stripes + kHmaxLL, c->d_stripes + kCloseRec);
  c->loop2_pending = true;
  return SPH_OK;
}

// After the step's closing copy_record and sync: loop 2's energy sum (block
// partials summed in block order) and its error bits.
static int finish_loop2(sph_ctx *c) {
  if (!c->loop2_pending) return SPH_OK;
  c->loop2_pending = false;
  double e;
  std::memcpy(&e, c->h_rec + kCloseRec, sizeof e);
  c->stats.energy = e;
  // h_max after the step's own h update: the next step's grid needs no
  // bounding-box pass while positions and h change no other way
  const double hm = ord2d(c->h_rec[kCloseRec + 2]);
  if (hm > 0.0 && std::isfinite(hm)) {
    c->next_hmax = hm;
    c->hmax_version = c->h_version;
  }
  c->stats.ms_k_loop2 = elapsed(c, c->ev[5], c->ev[6]);
  return map_err((int)c->h_rec[kCloseRec + 1]);
}

static Phys call_phys(const sph_ctx *c, const double *state) {
  Phys P = c->frozen;
  // read at every call by the reference (circuit1.f90:96, circuit2.f90:86-90)
  P.hfac = state[S_HFAC];
  P.dcond = state[S_DCOND];
  P.diso = (int)state[S_DISO];
  P.muzero = state[S_MUZERO];
  P.gamma = state[S_GAMMA];
  return P;
}

// The tail of a step after loop 1: Newton bookkeeping, EOS and packs
// (k_post1), loop 2, mti gravity, and a leapfrog pass's corrector or an RKL2 stage.  pending: the
// still-active stripes of the last sweep queued, when more could follow it;
// even: the evennesses of the step's own lists, while they are not known, for
// which the loops' lanes are right (kAnyLists: they are known, or no matter).
static int enqueue_tail(sph_ctx *c, const Phys &P, const long long *pending = nullptr, int even = kAnyLists) {
  HIPCHK(mark(c, 2));
  int rc = c->opt.precision == 1 ? run_post_and_loop2<float4>(c, P, pending, even)
                                   : run_post_and_loop2<double4>(c, P, pending, even);
  if (rc == SPH_OK && c->gravity)
    hipLaunchKernelGGL(k_gravity, dim3(grid_for(c->n)), dim3(kBlock), 0, c->stream, c->fields(), c->real, (int)c->n,
                       c->gravity);
  if (rc == SPH_OK && c->correct)
    hipLaunchKernelGGL(k_correct, dim3(grid_for(c->n)), dim3(kBlock), 0, c->stream, c->fields(), (int)c->n,
                       reinterpret_cast<const double *>(c->d_stripes + kDtLL), c->aux(0), (int)c->npad,
                       c->d_int + kGoInt, step_err(c));
  if (rc == SPH_OK && c->sts_j > 0) {
    double co[4];
    RCHK(sph_sts_coeffs(c->sts_j, c->sts_s, co));
    Fields F = c->fields();
    hipLaunchKernelGGL(k_sts_stage, dim3(grid_for(c->n)), dim3(kBlock), 0, c->stream, F.f[F_T], F.f[F_DDT], c->aux(0),
                       c->aux(1), c->aux(2), (int)c->n, c->sts_j == 1 ? 1 : 0, co[0], co[1], co[2] * c->sts_dt,
                       co[3] * c->sts_dt, c->d_int + kGoInt, step_err(c));
  }
  HIPCHK(mark(c, 3));
  return rc;
}

// Whether loop 2's packs or terms depend on k_prep's v / B flags (the
// "every velocity 0" and "one B for every particle" bits): the diffusion-only
// loops skip v and B by them; the general loop reads v for every pair unless
// no term needs it always (hydro, MHD, artificial conductivity), and B by
// them only for a diffusion tensor from B (k_loop2).  Otherwise a step need
// not wait for the flags before its tail: they come back at its end.
static bool loop2_reads_flags(const Phys &P) {
  const bool generic = loop2_general(P);
  if (!generic) return true;
  const bool v_always = P.hydro || P.magneto || P.artts;
  const bool tensor_b = P.diff && !P.fld && P.diso == 0;
  return !v_always || tensor_b;
}

// c1advanced steps: the search (its read-back left pending), a batch of
// sweeps, the tail, then one synchronisation.  Only when k_prep's v / B
// flags must come back before the tail picks loop 2's packs (after a load or
// a leapfrog change of v or B, for a loop 2 that reads them) does the step
// wait after the sweeps.  Lists
// that overflowed leave loop 1 and k_post1 idle (device-side checks), so the
// step searches again with room and starts over; a batch that ends with
// particles still active leaves its tail idle and is followed by more sweeps
// and another tail.  Where the evenness of the lists decides over the lanes
// and so over the sums' rounding, the step is queued for lists like the last
// ones' and done again if its own are not (the tail then stayed idle); the first
// after a load waits for its own.
static int run_advanced(sph_ctx *c, const Phys &P) {
  const int maxsw = sweep_cap(c);
  int first = 1, sweeps = 0, bits = 0;
  long long pairs = 0;
  float ms1 = 0.f;
  if (c->n_real <= 0) {  // no sweep, no active particle (circuit1.f90:114)
    if (c->neigh_pending) HIPCHK(copy_record(c, 0));
    HIPCHK(hipStreamSynchronize(c->stream));
    const int fin = take_neighbours(c);
    if (fin == kRedoNeigh) RCHK(build_neighbours(c));
    else RCHK(fin);
    c->stats.sweeps = 0;
    c->stats.loop1_pairs = 0;
    const int rc = enqueue_tail(c, P);
    HIPCHK(copy_record(c, 0));
    HIPCHK(wait_stream(c));
    const int rc2 = finish_loop2(c);
    return rc != SPH_OK ? rc : rc2;
  }
  int even = kAnyLists;
  if (c->neigh_pending && same_rounding(c, P, kRandom) != kAnyLists) {
    if (c->even >= 0) {
      even = same_rounding(c, P, c->even);
    } else {
      HIPCHK(copy_record(c, 0));
      HIPCHK(wait_stream(c));
      const int fin = take_neighbours(c);
      if (fin == kRedoNeigh) RCHK(build_neighbours(c));
      else RCHK(fin);
    }
  }
  auto start_over = [&] {
    first = 1; sweeps = 0; pairs = 0; ms1 = 0.f;
    even = kAnyLists;
  };
  // the step's own lists are known: were the loops queued for such?
  auto other_lists = [&] { return (even >> c->even & 1) == 0; };
  for (;;) {
    const int last = std::min(maxsw, first + std::max(1, c->sweep_hint) - 1);
    launch_sweeps(c, P, first, last);
    if (c->neigh_pending && c->flags_pending && loop2_reads_flags(P)) {
      HIPCHK(copy_record(c, 0));
      HIPCHK(wait_stream(c));
      c->neigh_pending = false;
      const int fin = take_neighbours_now(c);
      if (fin == kRedoNeigh) {
        RCHK(build_neighbours(c));
        start_over();
        continue;
      }
      RCHK(fin);
      if (other_lists()) {
        HIPCHK(hipMemsetAsync(step_err(c) + kErrLoop1, 0, 2 * sizeof(int), c->stream));
        start_over();
        continue;
      }
      even = kAnyLists;
    }
    const int rc = enqueue_tail(c, P, last < maxsw ? c->d_sweep + (size_t)last * kSweepRegion : nullptr, even);
    // the search's read-back if still pending, error words, the tail's record
    // and the sweep regions: one copy
    HIPCHK(copy_record(c, last));
    HIPCHK(wait_stream(c));
    ms1 += elapsed(c, c->ev[9], c->ev[10]);
    if (rc != SPH_OK) return rc;
    if (c->neigh_pending) {
      c->neigh_pending = false;
      const int fin = take_neighbours_now(c);
      if (fin == kRedoNeigh) {
        RCHK(build_neighbours(c));
        start_over();
        continue;
      }
      RCHK(fin);
      if (other_lists()) {
        HIPCHK(hipMemsetAsync(step_err(c) + kErrLoop1, 0, 2 * sizeof(int), c->stream));
        start_over();
        continue;
      }
      even = kAnyLists;
    }
    for (int it = first; it <= last; it++) {
      const long long *r = c->h_sweep + (size_t)it * kSweepRegion;
      if (!r[2 * kStripes]) break;
      sweeps = it;
      pairs += stripe_sum(r, 1);
    }
    bits = copied_err(c->h_rec, 0, kErrLoop1);
    if (bits) break;  // circuit1.f90:202-204 stops inside the sweep
    if (sweeps == last && last < maxsw && stripe_sum(c->h_sweep + (size_t)last * kSweepRegion, 0) > 0) {
      first = last + 1;  // still active: more sweeps, then the tail again
      continue;
    }
    break;
  }
  c->stats.sweeps = sweeps;
  c->stats.loop1_pairs = pairs;
  c->stats.ms_k_loop1 = ms1;
  // one sweep more than this step took: a sweep past convergence exits at
  // once (its launch costs about 16 us at 2M particles), while a step that
  // needs more sweeps than launched waits for one more round trip
  c->sweep_hint = std::min(maxsw, std::max(2, sweeps + 1));
  c->sweep_hints[c->fresh] = c->sweep_hint;
  const int rc2 = finish_loop2(c);
  const int r1 = map_err(bits);
  return r1 != SPH_OK ? r1 : rc2;
}

static int run_step(sph_ctx *c, const double *state) {
  if (c->n <= 0) return SPH_ERR_BAD_ARG;
  // a new step changes the geometry the differentiable operator was prepared on
  c->diff_ready = false;
  c->w_valid = false;
  c->fw_steps = 0;
  c->fw_tail = false;
  c->fresh = c->derivs_ready ? 0 : 1;
  c->sweep_hint = c->sweep_hints[c->fresh];
  c->derivs_ready = false;
  Phys P = call_phys(c, state);
  c->stats.ms_k_neigh = c->stats.ms_k_loop1 = c->stats.ms_k_loop2 = 0.0;
  HIPCHK(mark(c, 0));
  // the search's read-back is taken with the step's closing synchronisation
  // (c1advanced); c1simple writes h, rho and om in place, so its search is
  // checked before it runs
  RCHK(build_neighbours(c, P.adden != 0));
  c->hmax_version = 0;  // h changes from here; this step's k_post1 reports the new h_max
  HIPCHK(mark(c, 1));
  int rc;
  if (P.adden) {
    rc = run_advanced(c, P);
  } else {
    int r1 = run_loop1_simple(c, P);
    c->neigh_pending = false;
    RCHK(r1);
    rc = enqueue_tail(c, P);
    HIPCHK(copy_record(c, 0));
    HIPCHK(wait_stream(c));
    const int rc2 = finish_loop2(c);
    if (rc == SPH_OK) rc = rc2;
  }
  c->neigh_pending = false;
  float t01 = 0, t12 = 0, t23 = 0;
  if (c->timing) {
    tolerate(hipEventElapsedTime(&t01, c->ev[0], c->ev[1]));
    tolerate(hipEventElapsedTime(&t12, c->ev[1], c->ev[2]));
    tolerate(hipEventElapsedTime(&t23, c->ev[2], c->ev[3]));
  }
  c->stats.ms_neigh = t01;
  c->stats.ms_loop1 = t12;
  c->stats.ms_loop2 = t23;
  c->stats.ms_total = t01 + t12 + t23;
  c->have_step = true;
  c->derivs_ready = rc == SPH_OK;
  return rc;
}

// ----------------------------------------------------------------- loading
// The order of a new store's rows by cell key, as the first step's sort would
// make it, so that the fields are read in that order once: *perm gets it, or
// null where the rows are in order already or cannot be ordered (the step then
// says why).  A first step after it has bounding box, keys and cell starts, and
// sorts nothing: the gather of 32 columns over 1.1M random particles was 0.62
// ms, the rows of 256 bytes are read in any order in 0.15.
static int load_order(sph_ctx *c, const double *src, int64_t ld, const uint32_t **perm) {
  const int n = (int)c->n;
  const unsigned G = grid_for(n);
  *perm = nullptr;
  c->load_moved = false;
  if (c->n_real <= 0) return SPH_OK;
  Fields F;
  for (int f = 0; f < F_TOTAL; f++) F.f[f] = c->fbuf[1] + (size_t)f * c->npad;
  hipLaunchKernelGGL(k_load_cols, dim3(G), dim3(kBlock), 0, c->stream, src, ld, n, F, c->orig[1]);
  double lo[3], hi[3], hmax, rmax, cs[3];
  int64_t nkeys;
  bool wrapped;
  const int rc = wrap_pass(c, F, c->orig[1], lo, hi, &hmax, &wrapped);
  if (rc == SPH_ERR_UNSUPPORTED) return SPH_OK;
  RCHK(rc);
  bool finite = hmax > 0.0 && std::isfinite(hmax);
  for (int a = 0; a < 3; a++) finite = finite && std::isfinite(lo[a]) && std::isfinite(hi[a]);
  if (!finite) return SPH_OK;
  const Grid g = search_grid(c, lo, hi, hmax, &rmax, cs, &nkeys);
  const int rk = ensure_cells(c, nkeys);
  if (rk == SPH_ERR_NOMEM) return SPH_OK;
  RCHK(rk);
  hipLaunchKernelGGL(k_keys, dim3(G), dim3(kBlock), 0, c->stream, F, n, g, c->keys, c->vals, c->d_int + 2,
                     (int *)nullptr, c->d_stripes + kFlagSlots);
  hipLaunchKernelGGL(k_check_sorted, dim3(std::min(G, 256u)), dim3(kBlock), 0, c->stream, c->keys, n, c->d_int + 2);
  RCHK(read_ints(c, 2, 1));
  if (c->h_int[2] != 0) {
    size_t bytes = c->sort_tmp_bytes;
    HIPCHK(hipcub::DeviceRadixSort::SortPairs(c->sort_tmp, bytes, c->keys, c->keys2, c->vals, c->vals2, n, 0,
                                              bits_of(nkeys), c->stream));
    std::swap(c->keys, c->keys2);
    *perm = c->vals2;
    c->load_moved = true;
  }
  hipLaunchKernelGGL(k_cell_start, dim3(grid_for(n + 1)), dim3(kBlock), 0, c->stream, c->keys, n, (uint32_t)nkeys,
                     c->cstart);
  c->flags_clear = true;
  if (wrapped) return SPH_OK;  // the step wraps them, and makes the keys of the new positions
  for (int a = 0; a < 3; a++) { c->last_lo[a] = lo[a]; c->last_hi[a] = hi[a]; }
  c->next_hmax = hmax;
  c->bbox_version = c->keys_version = c->pos_version;
  c->hmax_version = c->h_version;
  c->keys_grid = g;
  c->keys_n = n;
  c->keys_nkeys = nkeys;
  return SPH_OK;
}

static int load_impl(sph_ctx *c, int64_t n, const double *store, int64_t ld, int on_device) {
  if (n <= 0 || ld < F_TOTAL || !store) return SPH_ERR_BAD_ARG;
  if (n > ((int64_t)1 << 27) - 1) return SPH_ERR_UNSUPPORTED;
  if (n < c->n_real) return SPH_ERR_BAD_ARG;
  RCHK(ensure_particles(c, n));
  c->n = n;
  c->n_fixed = n - c->n_real;
  const double *src = store;
  int64_t bytes = n * ld * (int64_t)sizeof(double);
  if (!on_device) {
    if (bytes > c->staging_bytes) {
      RCHK(dev_alloc((void **)&c->d_staging, bytes));
      c->staging_bytes = bytes;
    }
    HIPCHK(hipMemcpyAsync(c->d_staging, store, bytes, hipMemcpyHostToDevice, c->stream));
    src = c->d_staging;
  }
  c->cur = 0;
  c->fullest = 0;
  c->even = -1;
  c->breaks = 2;
  c->pos_version++;
  c->vb_version++;
  c->h_version++;
  // the particles (and their order) are new: lists, the prepared operator,
  // its weights and the recorded forward belong to the old ones
  c->have_step = false;
  c->derivs_ready = false;
  c->diff_ready = false;
  c->w_valid = false;
  c->fw_steps = 0;
  c->fw_tail = false;
  const uint32_t *perm;
  RCHK(load_order(c, src, ld, &perm));
  hipLaunchKernelGGL(k_aos_to_soa, dim3(tiles_for(n)), dim3(kBlock), 0, c->stream, src, ld, (int)n, perm, c->fields(),
                     c->orig[0]);
  HIPCHK(wait_stream(c));
  return SPH_OK;
}

static int save_impl(sph_ctx *c, double *store, int64_t ld, int on_device) {
  if (!store || ld < F_TOTAL || c->n <= 0) return SPH_ERR_BAD_ARG;
  int64_t bytes = c->n * ld * (int64_t)sizeof(double);
  double *dst = store;
  if (!on_device) {
    if (bytes > c->staging_bytes) {
      RCHK(dev_alloc((void **)&c->d_staging, bytes));
      c->staging_bytes = bytes;
    }
    dst = c->d_staging;
    if (ld > F_TOTAL) HIPCHK(hipMemcpyAsync(dst, store, bytes, hipMemcpyHostToDevice, c->stream));
  }
  hipLaunchKernelGGL(k_soa_to_aos, dim3(tiles_for(c->n)), dim3(kBlock), 0, c->stream, c->fields(), c->orig[c->cur],
                     (int)c->n, dst, ld);
  if (!on_device) HIPCHK(hipMemcpyAsync(store, dst, bytes, hipMemcpyDeviceToHost, c->stream));
  HIPCHK(hipStreamSynchronize(c->stream));
  return SPH_OK;
}

// ================================================================== C-ABI
extern "C" {

int sph_default_options(sph_options *o) {
  if (!o) return SPH_ERR_BAD_ARG;
  memset(o, 0, sizeof(*o));
  o->precision = 0;
  o->tensor_mode = 0;
  o->kappa_perp = 0.0;
  o->max_sweeps = 100;
  o->newton_tol = 0.0;
  o->neigh_cap = 0;
  o->device = 0;
  o->cell_div = 0;
  return SPH_OK;
}

int sph_ctx_create(const double state[49], int kernel_id, const sph_options *opt, sph_ctx **out) {
  if (!state || !out || kernel_id < 0 || kernel_id > 2) return SPH_ERR_BAD_ARG;
  *out = nullptr;
  int dim = (int)state[S_DIM];
  if (dim < 1 || dim > 3) return SPH_ERR_BAD_ARG;
  if ((int)state[S_COORD] == 2) return SPH_ERR_UNSUPPORTED;  // cylindrical, kernel.f90:135-148
  sph_ctx *c = new sph_ctx();
  if (opt) c->opt = *opt;
  else sph_default_options(&c->opt);
  {
    const char *t = std::getenv("SPH_NEIGH_TRAVERSAL");
    c->lane_search = t && std::strcmp(t, "lane") == 0;
    const char *g = std::getenv("SPH_LOOP2_GENERIC");
    c->loop2_generic = g && std::strcmp(g, "1") == 0;
  }
  if (c->opt.precision < 0 || c->opt.precision > 1 || c->opt.tensor_mode < 0 || c->opt.tensor_mode > 1 ||
      c->opt.cell_div < 0 || c->opt.cell_div > 4 || c->opt.neigh_cap < 0 || c->opt.neigh_cap > (1 << 20)) {
    delete c;
    return SPH_ERR_BAD_ARG;
  }
  c->device = c->opt.device;
  if (hipSetDevice(c->device) != hipSuccess || hipStreamCreate(&c->stream) != hipSuccess) {
    delete c;
    return SPH_ERR_HIP;
  }
  for (auto &e : c->ev) (void)hipEventCreate(&e);
  c->kt = kernel_id;
  Phys &P = c->frozen;
  P.dim = dim;
  P.kt = kernel_id;
  P.ddw = (int)state[S_DDW];
  P.adden = (int)state[S_ADDEN] == 1;
  P.artts = (int)state[S_ARTTS] == 1;
  P.au = state[S_AU];
  P.tensor_mode = c->opt.tensor_mode;
  P.kappa_perp = c->opt.kappa_perp;
  eq_components(state, &P);
  P.wcv = knorm(kernel_id, dim);
  P.fwc = fwc_of(kernel_id, dim);
  P.krad = krad_of(kernel_id);
  c->maxneib = c->opt.neigh_cap > 0 ? c->opt.neigh_cap : maxneib_of(kernel_id, dim);
  // process / legacy-setup branch of iterate (iterator.f90:60-178)
  c->process = (int)state[S_PROCESS];
  c->ics = (int)state[S_ICS];
  int wrap = 0, ghost = 0;
  c->do_eos = 1;
  c->eos_iso = 0;
  if (c->process == 601) { wrap = ghost = 7; }
  else if (c->process == 602) { }
  else if (c->process == 600) {
    switch (c->ics) {
      case 102: ghost = 2; break;
      case 103: case 104: case 111: c->do_eos = 0; break;
      case 105: wrap = ghost = 7; c->eos_iso = 1; break;
      case 106: wrap = ghost = 6; break;
      case 108: wrap = ghost = 7; break;
      case 101: wrap = ghost = 1; c->gravity = 1; break;  // mti
      case 110: wrap = ghost = 1; c->gravity = 2; break;  // mtilowres
      default: delete c; return SPH_ERR_UNSUPPORTED;
    }
  } else {
    delete c;
    return SPH_ERR_BAD_ARG;
  }
  // box and ghost bands, BC.f90:46-68,210-223
  Box &b = c->box;
  double bs = state[S_BORD], pad = state[S_PAD];
  for (int a = 0; a < 3; a++) {
    b.emin[a] = state[S_XMIN + 2 * a];
    b.emax[a] = state[S_XMIN + 2 * a + 1];
    b.boxmax[a] = b.emax[a] - bs;
    b.boxmin[a] = b.emin[a] + bs;
    b.pmin[a] = b.emin[a];
    b.pmax[a] = b.emax[a];
    if (pad == 0) { b.pmin[a] = b.emin[a] + pad / 10; b.pmax[a] = b.emax[a] - pad / 10; }
  }
  int dmask = (1 << dim) - 1;
  b.wrap_mask = wrap & dmask;
  b.ghost_mask = ghost & dmask;
  c->n_real = (int64_t)state[S_REALPN];
  c->n_fixed = (int64_t)state[S_FIXEDPN];
  if (c->n_real < 0) { delete c; return SPH_ERR_BAD_ARG; }
  if (dev_alloc((void **)&c->d_red, (16 * kStripes + 8 * kDtBlocks) * sizeof(long long)) != SPH_OK ||
      dev_alloc((void **)&c->d_int, 256 * sizeof(int)) != SPH_OK ||
      dev_alloc((void **)&c->d_stripes, kRecLL * sizeof(long long)) != SPH_OK ||
      hipHostMalloc((void **)&c->h_int, 256 * sizeof(int)) != hipSuccess ||
      hipHostMalloc((void **)&c->h_ll, 2048 * sizeof(long long)) != hipSuccess ||
      hipHostMalloc((void **)&c->h_rec, kRecLL * sizeof(long long)) != hipSuccess) {
    sph_ctx_destroy(c);
    return SPH_ERR_NOMEM;
  }
  c->d_dtpart = c->d_red + 16 * kStripes;
  c->d_sweep = c->d_stripes + kStepLL;
  c->h_sweep = c->h_rec + kStepLL;
  if (c->opt.max_sweeps > 240) c->opt.max_sweeps = 240;
  *out = c;
  return SPH_OK;
}

int sph_ctx_destroy(sph_ctx *c) {
  if (!c) return SPH_ERR_BAD_ARG;
  (void)hipSetDevice(c->device);
  if (c->stream) (void)hipStreamSynchronize(c->stream);
  void *ptrs[] = {c->fbuf[0], c->fbuf[1], c->orig[0], c->orig[1], c->keys, c->keys2, c->vals, c->vals2,
                  c->sort_tmp, c->cstart, c->pm, c->st[0], c->st[1], c->tr[0], c->tr[1], c->s1[0], c->s1[1], c->pfix, c->s2, c->pd, c->trd,
                  c->h0, c->eps, c->pf,
                  c->real, c->nb, c->cnt, c->q[0], c->q[1], c->q[2], c->q[3], c->q[4], c->energy_part,
                  c->d_red, c->d_int, c->d_stripes, c->d_staging, c->rent,
                  c->dvec, c->gpart, c->ckpt, c->rcnt, c->dpxh, c->dirho, c->dW, c->ddW, c->dR, c->dS, c->dZ, c->drho, c->dRec,
                  c->gkdev, c->nlF, c->nlU, c->nlUB, c->nlNu, c->nlMu, c->nlD, c->nlDD, c->nlR,
                  c->ext_count, c->ecs, c->erec, c->ext_tmp};
  for (void *p : ptrs)
    if (p) (void)hipFree(p);
  if (c->h_int) (void)hipHostFree(c->h_int);
  if (c->h_ll) (void)hipHostFree(c->h_ll);
  if (c->h_rec) (void)hipHostFree(c->h_rec);
  for (auto &e : c->ev)
    if (e) (void)hipEventDestroy(e);
  if (c->stream) (void)hipStreamDestroy(c->stream);
  delete c;
  (void)hipGetLastError();  // clean-up failures are not the next call's
  return SPH_OK;
}

static int check_counts(sph_ctx *c, int64_t n, const double *state) {
  if (!state) return SPH_ERR_BAD_ARG;
  int64_t nr = (int64_t)state[S_REALPN];
  if (nr != c->n_real || n < nr) return SPH_ERR_BAD_ARG;
  return SPH_OK;
}

int sph_load(sph_ctx *c, int64_t n, const double *store, int64_t ld, int on_device) {
  if (!c) return SPH_ERR_BAD_ARG;
  (void)hipSetDevice(c->device);
  return load_impl(c, n, store, ld, on_device);
}

int sph_save(sph_ctx *c, double *store, int64_t ld, int on_device) {
  if (!c) return SPH_ERR_BAD_ARG;
  (void)hipSetDevice(c->device);
  return save_impl(c, store, ld, on_device);
}

int sph_step(sph_ctx *c, const double state[49], double *maxconsenrg) {
  if (!c || !state) return SPH_ERR_BAD_ARG;
  (void)hipSetDevice(c->device);
  int rc = run_step(c, state);
  if (maxconsenrg) *maxconsenrg = 0.0;  // circuit2.f90:101
  return rc;
}

int sph_iterate(sph_ctx *c, int64_t n, double *store, int64_t ld, const double state[49], double *maxconsenrg) {
  if (!c) return SPH_ERR_BAD_ARG;
  RCHK(check_counts(c, n, state));
  RCHK(sph_load(c, n, store, ld, 0));
  int rc = sph_step(c, state, maxconsenrg);
  int rs = save_impl(c, store, ld, 0);
  return rc != SPH_OK ? rc : rs;
}

int sph_iterate_device(sph_ctx *c, int64_t n, double *d_store, int64_t ld, const double state[49],
                       double *maxconsenrg) {
  if (!c) return SPH_ERR_BAD_ARG;
  RCHK(check_counts(c, n, state));
  RCHK(sph_load(c, n, d_store, ld, 1));
  int rc = sph_step(c, state, maxconsenrg);
  int rs = save_impl(c, d_store, ld, 1);
  return rc != SPH_OK ? rc : rs;
}

int sph_neighbours(sph_ctx *c, int64_t *off, int32_t *j, int8_t *code, int64_t cap_pairs, int64_t *n_pairs) {
  if (!c || !off || !c->have_step) return SPH_ERR_BAD_ARG;
  (void)hipSetDevice(c->device);
  const int n = (int)c->n;
  int64_t nr = c->n_real;
  int64_t *d_cnt = nullptr;
  RCHK(dalloc(&d_cnt, nr + 1));
  HIPCHK(hipMemsetAsync(d_cnt, 0, sizeof(int64_t) * (nr + 1), c->stream));
  hipLaunchKernelGGL(k_counts_by_orig, dim3(grid_for(n)), dim3(kBlock), 0, c->stream, c->cnt, c->orig[c->cur],
                     c->real, n, d_cnt);
  std::vector<int64_t> h(nr + 1);
  HIPCHK(hipMemcpyAsync(h.data(), d_cnt, sizeof(int64_t) * nr, hipMemcpyDeviceToHost, c->stream));
  HIPCHK(hipStreamSynchronize(c->stream));
  off[0] = 0;
  for (int64_t i = 0; i < nr; i++) off[i + 1] = off[i] + h[i];
  int64_t total = off[nr];
  if (n_pairs) *n_pairs = total;
  int rc = SPH_OK;
  if (j && code) {
    if (total > cap_pairs) rc = SPH_ERR_BAD_ARG;
    else {
      int32_t *dj = nullptr;
      int8_t *dc = nullptr;
      if (dalloc(&dj, total + 1) != SPH_OK || dalloc(&dc, total + 1) != SPH_OK) rc = SPH_ERR_NOMEM;
      else {
        HIPCHK(hipMemcpyAsync(d_cnt, off, sizeof(int64_t) * nr, hipMemcpyHostToDevice, c->stream));
        hipLaunchKernelGGL(k_neigh_export, dim3(grid_for(n)), dim3(kBlock), 0, c->stream, c->nb, c->cnt,
                           c->orig[c->cur], c->real, n, (int)c->npad, d_cnt, dj, dc, total);
        HIPCHK(hipMemcpyAsync(j, dj, sizeof(int32_t) * total, hipMemcpyDeviceToHost, c->stream));
        HIPCHK(hipMemcpyAsync(code, dc, total, hipMemcpyDeviceToHost, c->stream));
        HIPCHK(hipStreamSynchronize(c->stream));
      }
      if (dj) (void)hipFree(dj);
      if (dc) (void)hipFree(dc);
    }
  }
  (void)hipFree(d_cnt);
  return rc;
}

}  // extern "C"

// ------------------------------------------- allocation-free list export
// Scratch of sph_neighbours_device_noalloc, in device memory the library
// never allocates: the list lengths in original order (int64, at most
// kNoAllocMaxReal + 1 of them) and the prefix sum's temporary storage.  Each
// GPU the library runs on holds its own copy (about 33 MiB) until the process
// ends, and every call on that GPU shares it.
constexpr int64_t kNoAllocMaxReal = (int64_t)1 << 22;
constexpr size_t kNoAllocCountBytes = ((size_t)(kNoAllocMaxReal + 1) * sizeof(int64_t) + 255) / 256 * 256;
constexpr size_t kNoAllocTempBytes = (size_t)1 << 20;
static __device__ __align__(256) unsigned char scratch[kNoAllocCountBytes + kNoAllocTempBytes];
constexpr int kExportLL = 1600;  // h_ll slot of the pair-count read-back

// The device address of this device's `scratch`, looked up once per device
// (the device must be current).  Host code uses only this address: the
// array's own name is a host-side stand-in.
static std::mutex g_scratch_mu;
static unsigned char *g_scratch[64] = {};
static int scratch_on_device(int device, unsigned char **out) {
  if (device < 0 || device >= 64) return SPH_ERR_BAD_ARG;
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (!g_scratch[device]) {
    void *p = nullptr;
    const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !p) {
      fprintf(stderr, "sph_hip: hipGetSymbolAddress(scratch) failed on device %d: %s\n", device,
              hipGetErrorString(e));
      return SPH_ERR_HIP;
    }
    g_scratch[device] = static_cast<unsigned char *>(p);
  }
  *out = g_scratch[device];
  return SPH_OK;
}

extern "C" {

int sph_neighbours_device_noalloc(sph_ctx *c, int64_t *d_off, int32_t *d_j, int8_t *d_code, int64_t cap_pairs,
                                  int64_t *n_pairs) {
  if (!c || !d_off || !c->have_step || cap_pairs < 0 || (cap_pairs > 0 && (!d_j || !d_code)))
    return SPH_ERR_BAD_ARG;
  HIPCHK(hipSetDevice(c->device));
  const int64_t nr = c->n_real;
  if (nr > kNoAllocMaxReal) {
    fprintf(stderr, "sph_neighbours_device_noalloc: %lld real particles, at most %lld\n", (long long)nr,
            (long long)kNoAllocMaxReal);
    return SPH_ERR_BAD_ARG;
  }
  unsigned char *base = nullptr;
  RCHK(scratch_on_device(c->device, &base));
  int64_t *counts = reinterpret_cast<int64_t *>(base);
  void *temp = base + kNoAllocCountBytes;
  size_t temp_bytes = 0;
  HIPCHK(hipcub::DeviceScan::ExclusiveSum(nullptr, temp_bytes, counts, d_off, (int)(nr + 1), c->stream));
  if (temp_bytes > kNoAllocTempBytes) {
    fprintf(stderr, "sph_neighbours_device_noalloc: the prefix sum needs %zu bytes of scratch, %zu held\n",
            temp_bytes, kNoAllocTempBytes);
    return SPH_ERR_BAD_ARG;
  }
  const int n = (int)c->n;
  // every real particle writes its own slot; the slot after them (the
  // total) is the only one the last call's contents could leave stale
  hipLaunchKernelGGL(k_counts_by_orig, dim3(grid_for(n)), dim3(kBlock), 0, c->stream, c->cnt, c->orig[c->cur],
                     c->real, n, counts);
  hipLaunchKernelGGL(k_set_i64, dim3(1), dim3(64), 0, c->stream, counts + nr, (int64_t)0);
  HIPCHK(hipcub::DeviceScan::ExclusiveSum(temp, temp_bytes, counts, d_off, (int)(nr + 1), c->stream));
  if (cap_pairs > 0)
    hipLaunchKernelGGL(k_neigh_export, dim3(grid_for(n)), dim3(kBlock), 0, c->stream, c->nb, c->cnt,
                       c->orig[c->cur], c->real, n, (int)c->npad, d_off, d_j, d_code, cap_pairs);
  HIPCHK(hipMemcpyAsync(c->h_ll + kExportLL, d_off + nr, sizeof(int64_t), hipMemcpyDeviceToHost, c->stream));
  HIPCHK(hipStreamSynchronize(c->stream));
  const int64_t total = (int64_t)c->h_ll[kExportLL];
  if (n_pairs) *n_pairs = total;
  return (cap_pairs > 0 && total > cap_pairs) ? SPH_ERR_BAD_ARG : SPH_OK;
}

// checkVarsReady (preruncheck.f90:13-60) on the resident store; *what gets
// the failed test: 32 mu0 <= 0 with MHD, 64 isotropic conductivity <= 0,
// else the per-particle bits of k_prerun_check.
static int prerun_check(sph_ctx *c, const double *state, int *what) {
  *what = 0;
  const int eqs = (int)state[S_EQS];
  if (state[S_MUZERO] <= 0.0 && (eqs == 302 || eqs == 303)) *what = 32;
  else if ((int)state[S_DISO] > 0 && state[S_DCOND] <= 0.0) *what = 64;
  if (*what) return SPH_ERR_PRECONDITION;
  if (c->n <= 0) return SPH_ERR_BAD_ARG;
  HIPCHK(hipMemsetAsync(c->d_int + 5, 0, sizeof(int), c->stream));
  hipLaunchKernelGGL(k_prerun_check, dim3(grid_for(c->n)), dim3(kBlock), 0, c->stream, c->fields(), (int)c->n,
                     c->d_int + 5);
  RCHK(read_ints(c, 5, 1));
  const int b = c->h_int[5];
  // the reference stops at the first failing test, in this order
  for (int bit : {1, 2, 4, 8, 16})
    if (b & bit) { *what = bit; return SPH_ERR_PRECONDITION; }
  return SPH_OK;
}

int sph_prerun_check(sph_ctx *c, const double state[49], int *what) {
  if (!c || !state) return SPH_ERR_BAD_ARG;
  (void)hipSetDevice(c->device);
  int w = 0;
  const int rc = prerun_check(c, state, &w);
  if (what) *what = w;
  return rc;
}

int sph_leapfrog(sph_ctx *c, const double state[49], double dtcap, double *dt_used) {
  if (!c || !state || c->n <= 0) return SPH_ERR_BAD_ARG;
  (void)hipSetDevice(c->device);
  Phys P = call_phys(c, state);
  // main.f90:216-219: the pre-run checks and the initial iterate, once;
  // later passes take the derivatives the previous pass's iterate left
  // (main.f90:323-329)
  if (!c->derivs_ready) {
    int what = 0;
    RCHK(prerun_check(c, state, &what));
    RCHK(run_step(c, state));
  }
  // the time step, the predictor, the iterate and the corrector are queued
  // one behind the other: the host learns the step with the iterate's record
  const unsigned G = grid_for(c->n);
  DtArgs d{};
  d.part = c->d_dtpart;
  d.nblk = (int)std::min(G, (unsigned)kDtBlocks);
  d.hydro = P.hydro; d.magneto = P.magneto; d.diff = P.diff; d.fld = P.fld;
  cn_of(c->kt, P.ddw, &d.cnhydro, &d.cnd2);
  d.cap = dtcap;
  d.out = reinterpret_cast<double *>(c->d_stripes + kDtLL);
  hipLaunchKernelGGL(k_dt_reduce, dim3((unsigned)d.nblk), dim3(kBlock), 0, c->stream, c->fields(), c->real, (int)c->n,
                     c->d_dtpart);
  c->naux = 9;
  hipLaunchKernelGGL(k_predict, dim3(G), dim3(kBlock), 0, c->stream, c->fields(), (int)c->n, d, c->aux(0),
                     (int)c->npad);
  c->pos_version++;
  c->vb_version++;
  c->h_version++;
  c->correct = true;
  const int rc = run_step(c, state);
  c->correct = false;
  c->pos_version++;
  c->vb_version++;
  c->h_version++;
  c->naux = 0;
  if (rc != SPH_OK)  // the record may not hold the time step
    HIPCHK(hipMemcpyAsync(c->h_rec + kDtLL, c->d_stripes + kDtLL, sizeof(double), hipMemcpyDeviceToHost, c->stream));
  HIPCHK(wait_stream(c));
  if (dt_used) memcpy(dt_used, c->h_rec + kDtLL, sizeof(double));
  return rc;
}

// update_radenergy(n, store, dt), rad_exchange.f90:9-66, on every loaded
// particle (rows 1..n = real + fixed, as main.f90:367-369 passes n).
int sph_rad_exchange(sph_ctx *c, const double state[49], double dt) {
  if (!c || !state || c->n <= 0 || !(dt > 0.0)) return SPH_ERR_BAD_ARG;
  (void)hipSetDevice(c->device);
  const double a = 4. * kSigmaB / kLightspeed;                 // rad_exchange.f90:25
  const double cv1 = (state[S_GAMMA] - 1.) * state[S_MOLMASS] / kRg;  // :26
  HIPCHK(hipMemsetAsync(c->d_int, 0, sizeof(int), c->stream));
  hipLaunchKernelGGL(k_rad_exchange, dim3(grid_for(c->n)), dim3(kBlock), 0, c->stream, c->fields(), (int)c->n, dt, a,
                     cv1, kSigmaB, c->d_int);
  RCHK(read_ints(c, 0, 1));
  return (c->h_int[0] & EB_RAD) ? SPH_ERR_RAD_NEGATIVE : SPH_OK;
}

// sts_integrator.f90:10-51
static double sts_b(int j) { return j <= 2 ? 1. / 3. : (j * j + j - 2.) / (2. * j * (j + 1.)); }
static double sts_a(int j) { return 1 - sts_b(j); }
static double sts_mu(int j) { return (2. * j - 1.) / j * sts_b(j) / sts_b(j - 1); }
static double sts_nu(int j) { return -(j - 1.) / j * sts_b(j) / sts_b(j - 2); }
static double sts_w(int s) { return 4. / (s * s + s - 2.); }
static double sts_mu_hat(int j, int s) { return j == 1 ? sts_b(1) * sts_w(s) : sts_mu(j) * sts_w(s); }
static double sts_gm_hat(int j, int s) { return -sts_a(j - 1) * sts_mu_hat(j, s); }

int sph_sts_coeffs(int j, int s, double out[4]) {
  if (!out || j < 1 || s < 2) return SPH_ERR_BAD_ARG;
  out[0] = j >= 2 ? sts_mu(j) : 0.0;
  out[1] = j >= 2 ? sts_nu(j) : 0.0;
  out[2] = sts_mu_hat(j, s);
  out[3] = j >= 2 ? sts_gm_hat(j, s) : 0.0;
  return SPH_OK;
}

// sts_integrate, sts_integrator.f90:87-124: s steps, each with its stage behind
// it (k_sts_stage); aux arrays 0 Y_0, 1 dY_0, 2 Y_{j-2} (permuted with the
// particles at every re-sort).
int sph_sts(sph_ctx *c, const double state[49], int s, double dt) {
  if (!c || !state || c->n <= 0 || s < 2) return SPH_ERR_BAD_ARG;
  (void)hipSetDevice(c->device);
  c->sts_s = s;
  c->sts_dt = dt;
  int rc = SPH_OK;
  for (int j = 1; j <= s && rc == SPH_OK; j++) {
    c->naux = j == 1 ? 0 : 3;
    c->sts_j = j;
    rc = run_step(c, state);
  }
  c->sts_j = 0;
  c->naux = 0;
  return rc;
}

int sph_set_timing(sph_ctx *c, int on) {
  if (!c || (on != 0 && on != 1)) return SPH_ERR_BAD_ARG;
  c->timing = on != 0;
  return SPH_OK;
}

int sph_get_stats(sph_ctx *c, sph_stats *s) {
  if (!c || !s) return SPH_ERR_BAD_ARG;
  *s = c->stats;
  s->n_real = c->n_real;
  s->n_fixed = c->n_fixed;
  return SPH_OK;
}

const char *sph_error_string(int code) {
  switch (code) {
    case SPH_OK: return "ok";
    case SPH_ERR_NEIGH_TRUNCATED: return "# <!> KDTree neibsearch result was truncated.";
    case SPH_ERR_NEG_H: return "Negative smoothing length in c1 advanced";
    case SPH_ERR_Q_NAN_OR_NEG: return "q is nan or negative";
    case SPH_ERR_FLD_ANISO: return "There is no anisotropic for FLD";
    case SPH_ERR_BAD_DDW: return "# <!> second deriv id not found";
    case SPH_ERR_PRECONDITION: return "pre-run check failed";
    case SPH_ERR_BAD_ARG: return "invalid argument";
    case SPH_ERR_HIP: return "HIP runtime error";
    case SPH_ERR_NOMEM: return "device allocation failed";
    case SPH_ERR_UNSUPPORTED: return "unsupported configuration";
    case SPH_ERR_RAD_NEGATIVE: return "radiation or thermal energy is negative after exchange";
    default: return "unknown error";
  }
}

}  // extern "C"

// ------------------------------------------------- differentiable diffusion
// Set-up, operator applications and the checkpointed RKL2 forward/backward of
// the STS super-steps (sts_integrator.f90:87-124) with a global tensor K.
static DiffOpArgs diff_args(sph_ctx *c, const double K[6]) {
  DiffOpArgs a{};
  a.pm = c->pm; a.q0 = (const double4 *)c->q[0]; a.real = c->real; a.nb = c->nb; a.cnt = c->cnt;
  a.rcnt = c->rcnt; a.rent = c->rent; a.pxh = c->dpxh; a.b = c->box;
  for (int k = 0; k < 6; k++) a.K[k] = K[k];
  a.wcv = c->diff_phys.wcv; a.fwc = c->diff_phys.fwc; a.ddw = c->diff_phys.ddw;
  a.n = (int)c->n; a.npad = (int)c->npad;
  a.kap = c->fields().f[F_KAPPA];
  a.rho = c->drho;
  return a;
}

// ---- operators that read grad T (frozen geometry; see sph_adjoint.hip)
// Lanes per particle of these operators: 8 below 40k particles, else 4, in
// every dimension and whatever the lists are.
#define COMMA ,
#define NL_LAUNCH(KERNEL, ...)                                                                                      \
  do {                                                                                                              \
    if (c->n < 40000)                                                                                               \
      hipLaunchKernelGGL((KERNEL, 8>), dim3(grid_for(c->n * 8)), dim3(kBlock), 0, c->stream, __VA_ARGS__);          \
    else                                                                                                            \
      hipLaunchKernelGGL((KERNEL, 4>), dim3(grid_for(c->n * 4)), dim3(kBlock), 0, c->stream, __VA_ARGS__);          \
  } while (0)
// U = G(Y) and, for FLD with a state, its conductivity
template <int DIM, int KT>
static void nl_grad_k(sph_ctx *c, const DiffOpArgs &a, const double *Y, double4 *U, double4 *F) {
  double *D = c->diff_op == 5 && Y ? c->nlD : nullptr;
  if (c->diff_op == 4) NL_LAUNCH(k_nl_grad<DIM COMMA KT COMMA 2, a, Y, U, F, D, c->nlDD, c->nlR);
  else NL_LAUNCH(k_nl_grad<DIM COMMA KT COMMA 1, a, Y, U, F, D, c->nlDD, c->nlR);
}
// f(Y), Y sorted, to where `o` says
template <int DIM, int KT>
static void nl_apply_k(sph_ctx *c, const DiffOpArgs &a, const double *Y, const NlStage &o) {
  nl_grad_k<DIM, KT>(c, a, Y, c->nlU, nullptr);
  if (c->diff_op == 5) NL_LAUNCH(k_nl_apply<DIM COMMA KT COMMA 5, a, Y, c->nlU, c->nlD, o);
  else if (c->diff_op == 3) NL_LAUNCH(k_nl_apply<DIM COMMA KT COMMA 3, a, Y, c->nlU, c->nlD, o);
  else NL_LAUNCH(k_nl_apply<DIM COMMA KT COMMA 4, a, Y, c->nlU, c->nlD, o);
}
// A^T lam (2nw: A linear; FLD: the Jacobian of f at Ya, transposed) to where `o`
// says, `work` a sorted vector; for 2nw the tensor gradients gw lam^T dA/dK Ya
// -> gkdev[0..5] and, with Yb (which may be Ya), the same of Yb -> [6..11]
template <int DIM, int KT>
static void nl_adjoint_k(sph_ctx *c, const DiffOpArgs &a, const double *lam, const double *Ya, const double *Yb,
                         double *work, double gw, const NlAdjStage &o) {
  const unsigned G = grid_for(c->n);
  const double *none = nullptr;
  nl_grad_k<DIM, KT>(c, a, Ya, c->nlU, nullptr);
  if (c->diff_op == 5) {
    NL_LAUNCH(k_fld_adj<DIM COMMA KT, a, lam, Ya, c->nlD, c->nlDD, c->nlR, c->nlU, work, c->nlMu);
    const double *base = work;
    NL_LAUNCH(k_nl_gT<DIM COMMA KT COMMA 1, a, c->nlMu, c->nlF, base, o);
    return;
  }
  const double4 *UB = Yb ? c->nlU : nullptr;
  if (Yb && Yb != Ya) {
    nl_grad_k<DIM, KT>(c, a, Yb, c->nlUB, nullptr);
    UB = c->nlUB;
  }
  if (c->diff_op == 3) NL_LAUNCH(k_nl_nu<DIM COMMA KT COMMA 3, a, lam, c->nlF, c->nlNu);
  else NL_LAUNCH(k_nl_nu<DIM COMMA KT COMMA 4, a, lam, c->nlF, c->nlNu);
  hipLaunchKernelGGL(k_nl_mu, dim3(G), dim3(kBlock), 0, c->stream, a, c->nlNu, c->nlU, UB, c->nlMu, c->gpart);
  hipLaunchKernelGGL(k_gk_accum, dim3(1), dim3(256), 0, c->stream, c->gpart, (int)G, gw, 0.0, c->gkdev);
  if (Yb)
    hipLaunchKernelGGL(k_gk_accum, dim3(1), dim3(256), 0, c->stream, c->gpart, (int)G, 0.0, gw, c->gkdev + 6);
  if (c->diff_op == 4) NL_LAUNCH(k_nl_gT<DIM COMMA KT COMMA 2, a, c->nlMu, c->nlF, none, o);
  else NL_LAUNCH(k_nl_gT<DIM COMMA KT COMMA 1, a, c->nlMu, c->nlF, none, o);
}
#undef NL_LAUNCH
#undef COMMA
#define NL_DISPATCH(FN, ...)                                                                       \
  do {                                                                                            \
    const int d_ = c->diff_phys.dim, k_ = c->kt;                                                  \
    if (d_ == 1) { if (k_ == KT_M4) FN<1, KT_M4>(__VA_ARGS__); else if (k_ == KT_M6) FN<1, KT_M6>(__VA_ARGS__); else FN<1, KT_GAUSS>(__VA_ARGS__); } \
    else if (d_ == 2) { if (k_ == KT_M4) FN<2, KT_M4>(__VA_ARGS__); else if (k_ == KT_M6) FN<2, KT_M6>(__VA_ARGS__); else FN<2, KT_GAUSS>(__VA_ARGS__); } \
    else { if (k_ == KT_M4) FN<3, KT_M4>(__VA_ARGS__); else if (k_ == KT_M6) FN<3, KT_M6>(__VA_ARGS__); else FN<3, KT_GAUSS>(__VA_ARGS__); } \
  } while (0)

template <int DIM>
static void launch_weights_d(sph_ctx *c, const DiffOpArgs &a) {
  unsigned G = grid_for(c->n);
#define WTS(KT)                                                                                                  \
  do {                                                                                                           \
    hipLaunchKernelGGL((k_diff_weights<DIM, KT>), dim3(G), dim3(kBlock), 0, c->stream, a, c->dW, c->ddW);       \
    hipLaunchKernelGGL((k_diff_rweights<DIM, KT>), dim3(G), dim3(kBlock), 0, c->stream, a, c->dirho, c->dR);    \
  } while (0)
  if (c->kt == KT_M4) WTS(KT_M4);
  else if (c->kt == KT_M6) WTS(KT_M6);
  else WTS(KT_GAUSS);
#undef WTS
}
// Pair weights of A(K), assembled once per K (list order and reverse order).
static void ensure_weights(sph_ctx *c, const double K[6]) {
  if (c->w_valid && std::equal(K, K + 6, c->w_K)) return;
  DiffOpArgs a = diff_args(c, K);
  if (c->diff_phys.dim == 1) launch_weights_d<1>(c, a);
  else if (c->diff_phys.dim == 2) launch_weights_d<2>(c, a);
  else launch_weights_d<3>(c, a);
  std::copy(K, K + 6, c->w_K);
  c->w_valid = true;
}
// out = A(K) Y (sorted vectors).
static void diff_apply(sph_ctx *c, const double K[6], const double *Y, double *out) {
  ensure_weights(c, K);
  DiffOpArgs a = diff_args(c, K);
  const unsigned G = grid_for(c->n);
  hipLaunchKernelGGL(k_zrho, dim3(G), dim3(kBlock), 0, c->stream, (int)c->n, Y, a.q0, c->dZ);
  hipLaunchKernelGGL(k_diff_spmv, dim3(G), dim3(kBlock), 0, c->stream, a, c->dW, c->dZ, out);
}
// Successive products run their rows in alternating directions (stage_row).
static int next_rev(sph_ctx *c) { return c->stage_rev ^= 1; }

// The records of the pending stages, before their vectors change (fill: and
// empty ones behind them).
static void adj_pack(sph_ctx *c, bool fill) {
  if (c->rec_packed < (fill ? kRecs : c->rec_pend))
    hipLaunchKernelGGL(k_adj_pack, dim3(grid_for(c->n * kRecs)), dim3(kBlock), 0, c->stream, (int)c->n, c->recs,
                       c->rec_packed, c->rec_pend, fill ? 1 : 0, c->drho, c->dRec);
  c->rec_packed = c->rec_pend;
}
// The pending stages into the pair coefficients.
static void coef_flush(sph_ctx *c) {
  if (c->rec_pend == 0) return;
  adj_pack(c, true);
  hipLaunchKernelGGL(k_diff_coef, dim3(grid_for(c->n * 4)), dim3(kBlock), 0, c->stream, c->rent, c->rcnt, c->dRec,
                     c->dS, c->coef_set ? 1 : 0, (int)c->n, (int)c->npad);
  c->coef_set = true;
  c->rec_pend = c->rec_packed = 0;
}
// A stage's record: lam and Zt = (wa Ya + wb Yb) rho (Yb may be null).  The
// vectors stay as they are until adj_pack.
static void adj_record(sph_ctx *c, const double *lam, const double *Ya, const double *Yb, double wa, double wb) {
  const int q = c->rec_pend++;
  c->recs.lam[q] = lam; c->recs.Ya[q] = Ya; c->recs.Yb[q] = Yb; c->recs.wa[q] = wa; c->recs.wb[q] = wb;
  if (c->rec_pend == kRecs) coef_flush(c);
}
static AdjStage adj_args(sph_ctx *c) {
  AdjStage a{};
  a.rent = c->rent; a.rcnt = c->rcnt; a.R = c->dR; a.dW = c->ddW;
  a.n = (int)c->n; a.npad = (int)c->npad; a.rev = next_rev(c);
  return a;
}
template <int DIM>
static void launch_gcontract_d(sph_ctx *c, const DiffOpArgs &a, const double *S, const double *lam) {
  const dim3 G(grid_for(c->n)), T(kBlock);
  const double *Z = c->dZ;
  if (c->kt == KT_M4) hipLaunchKernelGGL((k_diff_gcontract<DIM, KT_M4>), G, T, 0, c->stream, a, c->dirho, S, lam, Z, c->gpart);
  else if (c->kt == KT_M6) hipLaunchKernelGGL((k_diff_gcontract<DIM, KT_M6>), G, T, 0, c->stream, a, c->dirho, S, lam, Z, c->gpart);
  else hipLaunchKernelGGL((k_diff_gcontract<DIM, KT_GAUSS>), G, T, 0, c->stream, a, c->dirho, S, lam, Z, c->gpart);
}
static void launch_gcontract(sph_ctx *c, const double K[6], const double *S, const double *lam, double *gk) {
  DiffOpArgs a = diff_args(c, K);
  if (c->diff_phys.dim == 1) launch_gcontract_d<1>(c, a, S, lam);
  else if (c->diff_phys.dim == 2) launch_gcontract_d<2>(c, a, S, lam);
  else launch_gcontract_d<3>(c, a, S, lam);
  hipLaunchKernelGGL(k_gk_accum, dim3(1), dim3(256), 0, c->stream, c->gpart, (int)grid_for(c->n), 1.0, 0.0, gk);
}
// gk[0..5] += sum over pairs of the accumulated coefficients times G (fixed
// reduction order); the next record starts new coefficients.
static void diff_gcontract(sph_ctx *c, const double K[6], double *gk) {
  coef_flush(c);
  launch_gcontract(c, K, c->dS, nullptr, gk);
  c->coef_set = false;
}
// The same for one stage: lam^T dA/dK Y.
static void stage_gcontract(sph_ctx *c, const double K[6], const double *lam, const double *Y, double *gk) {
  hipLaunchKernelGGL(k_zrho, dim3(grid_for(c->n)), dim3(kBlock), 0, c->stream, (int)c->n, Y, (const double4 *)c->q[0],
                     c->dZ);
  launch_gcontract(c, K, nullptr, lam, gk);
}

static int ensure_dvec(sph_ctx *c, int nvec) { return keep(c, &c->dvec, (size_t)nvec * c->npad); }
static double *dv(sph_ctx *c, int k) { return c->dvec + (size_t)k * c->npad; }

// Work vectors of the super-steps: rotating stage states, the first stage's
// rate, Z = Y rho of the last and the next state, the state between steps,
// what the adjoint's L_0 collects, and the adjoint's L in rotation (those of
// the pending records, the one before them and the next); then the stage
// states of a checkpoint segment, s per step.
constexpr int kLams = kRecs + 2;
enum { V_STATE = 0, V_DY0 = 3, V_Z = 4, V_Y = 6, V_A0 = 7, V_L = 8, V_SEG = V_L + kLams };

// One RKL2 super-step (sts_integrator.f90:100-123) of s stages from Y[0], whose
// Z is in the Z vector *z (left at the result's): stage states into Y[1..s]
// (Y[s] may be Y[0]).  keep_last false: the last stage is not needed.
static void sts_forward_step(sph_ctx *c, int s, double dt, double *const *Y, int *z, bool keep_last = true) {
  BatchStage a{};
  a.cnt = c->cnt; a.nb = c->nb; a.W = c->dW; a.rho = c->drho; a.h = dt; a.Y0 = Y[0]; a.DY0 = dv(c, V_DY0);
  a.n = (int)c->n; a.npad = (int)c->npad;
  const dim3 B(grid_for(c->n)), T(kBlock);
  for (int j = 1; j <= (keep_last ? s : s - 1); j++) {
    a.Yjm1 = Y[j - 1]; a.Yjm2 = j > 1 ? Y[j - 2] : Y[0]; a.Yj = Y[j];
    a.Zjm1 = dv(c, V_Z + *z); a.Zj = dv(c, V_Z + (*z ^= 1));
    a.mhat = sts_mu_hat(j, s);
    a.rev = next_rev(c);
    if (j == 1) {
      hipLaunchKernelGGL((k_batch_stage<true, double, true>), B, T, 0, c->stream, a);
    } else {
      a.mu = sts_mu(j); a.nu = sts_nu(j); a.c0 = 1. - a.mu - a.nu; a.ghat = sts_gm_hat(j, s);
      hipLaunchKernelGGL((k_batch_stage<false, double, true>), B, T, 0, c->stream, a);
    }
  }
}

// Adjoint of one super-step with the stage states Y[0..s-1]: L (V_L + *l) holds
// dL/dY_s on entry and dL/dY_0 on return.  The tensor-gradient coefficients
// accumulate per pair (dS).
static void sts_backward_step(sph_ctx *c, int s, double dt, double *const *Y, int *l) {
  auto L = [&](int k) { return dv(c, V_L + (*l + k + kLams) % kLams); };
  for (int j = s; j >= 1; j--) {
    AdjStage a = adj_args(c);
    a.lam = L(0);
    a.lam1 = j < s ? L(-1) : nullptr;
    a.out = L(1);
    a.A0 = dv(c, V_A0);
    a.mh = sts_mu_hat(j, s) * dt;
    if (j > 1) {
      a.mu = sts_mu(j); a.gh = sts_gm_hat(j, s) * dt;
      a.c0 = 1. - a.mu - sts_nu(j);
      a.nu0 = j == 2 ? sts_nu(j) : 0.;
      a.nu1 = j < s ? sts_nu(j + 1) : 0.;
      a.a0_add = j < s;
    } else {
      a.last = 1;
    }
    hipLaunchKernelGGL(k_adj_stage, dim3(grid_for(c->n)), dim3(kBlock), 0, c->stream, a);
    adj_record(c, L(0), Y[j - 1], j > 1 ? Y[0] : nullptr, a.mh, a.gh);
    *l = (*l + 1) % kLams;
  }
}

// Reverse lists of more than kRevSort entries: stable radix sort of the
// owner-major pairs on the neighbour index, then into the list layout.
static int reverse_lists_radix(sph_ctx *c, int64_t npairs) {
  const int n = (int)c->n, npad = (int)c->npad;
  const unsigned G = grid_for(n);
  int *foff = nullptr, *roff = nullptr;
  uint32_t *keys = nullptr, *keys2 = nullptr, *vals = nullptr, *flat = nullptr;
  void *tmp = nullptr;
  auto run = [&]() -> int {
    const size_t np = (size_t)std::max<int64_t>(npairs, 1);
    RCHK(dalloc(&foff, c->npad + 1));
    RCHK(dalloc(&roff, c->npad + 1));
    RCHK(dalloc(&keys, np));
    RCHK(dalloc(&keys2, np));
    RCHK(dalloc(&vals, np));
    RCHK(dalloc(&flat, np));
    size_t b1 = 0, b2 = 0, b3 = 0;
    int bits = 1;
    while (bits < 32 && ((int64_t)1 << bits) < (int64_t)n) bits++;
    HIPCHK(hipcub::DeviceScan::ExclusiveSum(nullptr, b1, c->rcnt, roff, n + 1, c->stream));
    HIPCHK(hipcub::DeviceScan::ExclusiveSum(nullptr, b2, c->cnt, foff, n, c->stream));
    HIPCHK(hipcub::DeviceRadixSort::SortPairs(nullptr, b3, keys, keys2, vals, flat, (int)npairs, 0, bits, c->stream));
    size_t bytes = std::max(b1, std::max(b2, b3));
    RCHK(dev_alloc(&tmp, bytes));
    // how often each particle is someone's neighbour, and where its segment starts
    HIPCHK(hipMemsetAsync(c->rcnt, 0, sizeof(int) * (c->npad + 1), c->stream));
    hipLaunchKernelGGL(k_rev_count, dim3(G), dim3(kBlock), 0, c->stream, c->real, c->nb, c->cnt, n, npad, c->rcnt);
    HIPCHK(hipcub::DeviceScan::ExclusiveSum(tmp, bytes, c->rcnt, roff, n + 1, c->stream));
    HIPCHK(hipcub::DeviceScan::ExclusiveSum(tmp, bytes, c->cnt, foff, n, c->stream));
    hipLaunchKernelGGL(k_pair_enum, dim3(G), dim3(kBlock), 0, c->stream, c->real, c->nb, c->cnt, n, npad, foff, keys,
                       vals);
    if (npairs > 0)
      HIPCHK(hipcub::DeviceRadixSort::SortPairs(tmp, bytes, keys, keys2, vals, flat, (int)npairs, 0, bits, c->stream));
    hipLaunchKernelGGL(k_rev_chunk, dim3(G), dim3(kBlock), 0, c->stream, roff, flat, n, npad, c->rcnt, c->rent);
    HIPCHK(hipStreamSynchronize(c->stream));
    return SPH_OK;
  };
  const int rc = run();
  void *t[] = {foff, roff, keys, keys2, vals, flat, tmp};
  for (void *q : t)
    if (q) (void)hipFree(q);
  return rc;
}

// The reverse lists (rent, rcnt) of the last search, capacity rcap.
static int reverse_lists(sph_ctx *c, int64_t npairs) {
  const int n = (int)c->n, npad = (int)c->npad;
  // room for an eighth more than the longest forward list
  int cap = (c->last_maxcnt + c->last_maxcnt / 8 + 8) / 8 * 8;
  for (;;) {
    RCHK(keep(c, &c->rent, (size_t)npad * cap));
    HIPCHK(hipMemsetAsync(c->rcnt, 0, sizeof(int) * ((size_t)npad + 1), c->stream));
    hipLaunchKernelGGL(k_rev_fill, dim3(grid_for(c->n * 8)), dim3(kBlock), 0, c->stream, c->real, c->nb, c->cnt, n,
                       npad, cap, c->rcnt, c->rent);
    HIPCHK(hipMemcpyAsync(c->h_int, c->rcnt + npad, sizeof(int), hipMemcpyDeviceToHost, c->stream));
    HIPCHK(wait_stream(c));
    const int longest = c->h_int[0];
    c->rcap = std::max(8, (longest + 7) / 8 * 8);
    if (longest <= cap) break;
    cap = c->rcap;
  }
  if (c->rcap > kRevSort) return reverse_lists_radix(c, npairs);
  hipLaunchKernelGGL(k_rev_sort, dim3((unsigned)((n + 3) / 4)), dim3(kBlock), 0, c->stream, n, npad, c->rcnt, c->rent);
  return SPH_OK;
}

extern "C" {

int sph_diff_prepare(sph_ctx *c, const double state[49]) {
  if (!c || !state || c->n <= 0) return SPH_ERR_BAD_ARG;
  (void)hipSetDevice(c->device);
  if (c->opt.precision != 0 || c->n_fixed != 0) return SPH_ERR_UNSUPPORTED;
  Phys P = call_phys(c, state);
  const bool hess = P.ddw == 400 || P.ddw == 401 || P.ddw == 402;
  int op;
  if (!P.diff) return SPH_ERR_UNSUPPORTED;
  if (P.fld) {
    // FLD: isotropic (circuit2.f90:189), one of the Hessian operators
    if (!hess || P.diso != 1) return SPH_ERR_UNSUPPORTED;
    op = 5;
  } else if (P.ddw == 403 || P.ddw == 404) {
    // the 2nw operators with one tensor K for every particle
    op = P.ddw == 403 ? 3 : 4;
  } else if (hess) {
    op = 0;
  } else {
    return SPH_ERR_UNSUPPORTED;
  }
  c->keep_q0 = true;
  const int step_rc = run_step(c, state);  // neighbours, Newton h, EOS, loop 2: h, rho, q0 now frozen
  c->keep_q0 = false;
  RCHK(step_rc);
  c->diff_phys = P;
  c->diff_op = op;
  const int n = (int)c->n;
  unsigned G = grid_for(n);
  const int64_t npairs = c->stats.n_pairs;
  if (npairs >= ((int64_t)1 << 31)) return SPH_ERR_UNSUPPORTED;  // 32-bit pair counts
  // rcnt: the reverse-list lengths, then the longest of them
  RCHK(keep(c, &c->rcnt, c->npad + 1));
  RCHK(keep(c, &c->dpxh, c->npad));
  RCHK(keep(c, &c->dirho, c->npad));
  if (op == 0) RCHK(keep(c, &c->dW, (size_t)c->npad * c->nb_cap));
  RCHK(keep(c, &c->ddW, c->npad));
  RCHK(keep(c, &c->dZ, c->npad));
  RCHK(keep(c, &c->drho, c->npad));
  if (op == 0) RCHK(keep(c, &c->dRec, (size_t)c->npad * kRecs));
  c->rec_pend = c->rec_packed = 0;
  c->coef_set = false;
  RCHK(keep(c, &c->gkdev, 12));
  RCHK(keep(c, &c->gpart, (size_t)G * 12));
  c->w_valid = false;
  hipLaunchKernelGGL(k_diff_pack, dim3(G), dim3(kBlock), 0, c->stream, n, c->pm, (const double4 *)c->q[0], c->dpxh,
                     c->drho, c->dirho);
  RCHK(reverse_lists(c, npairs));
  if (op == 0) {
    const size_t rslots = (size_t)c->npad * c->rcap;
    RCHK(keep(c, &c->dR, rslots));
    RCHK(keep(c, &c->dS, rslots));
  }
  if (op != 0) {
    RCHK(keep(c, &c->nlF, c->npad));
    RCHK(keep(c, &c->nlU, c->npad));
    RCHK(keep(c, &c->nlUB, c->npad));
    RCHK(keep(c, &c->nlNu, c->npad));
    RCHK(keep(c, &c->nlMu, c->npad));
    RCHK(keep(c, &c->nlD, c->npad));
    RCHK(keep(c, &c->nlDD, c->npad));
    RCHK(keep(c, &c->nlR, c->npad));
    const double K0[6] = {0, 0, 0, 0, 0, 0};
    DiffOpArgs a = diff_args(c, K0);
    NL_DISPATCH(nl_grad_k, c, a, nullptr, nullptr, c->nlF);  // F_s = sum_b m_b nw(r_sb, h_s)
  }
  HIPCHK(hipStreamSynchronize(c->stream));
  c->fw_tail = false;
  c->diff_ready = true;
  return SPH_OK;
}

int sph_diff_apply(sph_ctx *c, const double K[6], const double *d_T, double *d_out) {
  if (!c || !c->diff_ready || !d_T || !d_out || (!K && c->diff_op != 5)) return SPH_ERR_BAD_ARG;
  (void)hipSetDevice(c->device);
  RCHK(ensure_dvec(c, 2));
  const int n = (int)c->n;
  unsigned G = grid_for(n);
  hipLaunchKernelGGL(k_to_sorted, dim3(G), dim3(kBlock), 0, c->stream, d_T, c->orig[c->cur], n, dv(c, 0));
  if (c->diff_op != 0) {
    const double K0[6] = {0, 0, 0, 0, 0, 0};
    DiffOpArgs a = diff_args(c, K ? K : K0);
    NlStage st{};
    st.orig = c->orig[c->cur];
    st.out = d_out;
    NL_DISPATCH(nl_apply_k, c, a, dv(c, 0), st);
  } else {
    diff_apply(c, K, dv(c, 0), dv(c, 1));
    hipLaunchKernelGGL(k_from_sorted, dim3(G), dim3(kBlock), 0, c->stream, dv(c, 1), c->orig[c->cur], n, d_out);
  }
  HIPCHK(hipStreamSynchronize(c->stream));
  return SPH_OK;
}

int sph_diff_apply_adjoint(sph_ctx *c, const double K[6], const double *d_lam, const double *d_Ya,
                           const double *d_Yb, double *d_out, double gA[6], double gB[6]) {
  if (!c || !c->diff_ready || !d_lam || !d_Ya || !d_out || !gA || !gB) return SPH_ERR_BAD_ARG;
  if (c->diff_op != 5 && (!K || !d_Yb)) return SPH_ERR_BAD_ARG;
  (void)hipSetDevice(c->device);
  RCHK(ensure_dvec(c, 4));
  const int n = (int)c->n;
  unsigned G = grid_for(n);
  const int64_t *o = c->orig[c->cur];
  hipLaunchKernelGGL(k_to_sorted, dim3(G), dim3(kBlock), 0, c->stream, d_lam, o, n, dv(c, 0));
  hipLaunchKernelGGL(k_to_sorted, dim3(G), dim3(kBlock), 0, c->stream, d_Ya, o, n, dv(c, 1));
  const bool yb = d_Yb && d_Yb != d_Ya;
  if (yb) hipLaunchKernelGGL(k_to_sorted, dim3(G), dim3(kBlock), 0, c->stream, d_Yb, o, n, dv(c, 2));
  HIPCHK(hipMemsetAsync(c->gkdev, 0, sizeof(double) * 12, c->stream));
  if (c->diff_op != 0) {
    const double K0[6] = {0, 0, 0, 0, 0, 0};
    DiffOpArgs a = diff_args(c, K ? K : K0);
    NlAdjStage st{};
    st.orig = o;
    st.out = d_out;
    NL_DISPATCH(nl_adjoint_k, c, a, dv(c, 0), dv(c, 1), dv(c, yb ? 2 : 1), dv(c, 3), 1.0, st);
  } else {
    ensure_weights(c, K);
    AdjStage a = adj_args(c);  // A^T lam alone
    a.lam = dv(c, 0); a.out = dv(c, 3); a.mh = 1.0; a.last = 1;
    hipLaunchKernelGGL(k_adj_stage, dim3(G), dim3(kBlock), 0, c->stream, a);
    for (int k = 0; k < (yb ? 2 : 1); k++) stage_gcontract(c, K, dv(c, 0), dv(c, 1 + k), c->gkdev + 6 * k);
    hipLaunchKernelGGL(k_from_sorted, dim3(G), dim3(kBlock), 0, c->stream, dv(c, 3), o, n, d_out);
  }
  double g12[12];
  HIPCHK(hipMemcpyAsync(g12, c->gkdev, sizeof(double) * 12, hipMemcpyDeviceToHost, c->stream));
  HIPCHK(hipStreamSynchronize(c->stream));
  for (int k = 0; k < 6; k++) { gA[k] = g12[k]; gB[k] = yb || c->diff_op != 0 ? g12[6 + k] : g12[k]; }
  return SPH_OK;
}

// A checkpoint segment's stage states: Y[j] of its step k, the first step's
// Y[0] being the checkpoint itself.
static void segment_states(sph_ctx *c, int sg, int k, int s, std::vector<double *> &Y) {
  for (int j = 0; j < s; j++) Y[j] = dv(c, V_SEG + k * s + j);
  if (k == 0) Y[0] = c->ckpt + (size_t)sg * c->npad;
}

int sph_diff_forward(sph_ctx *c, const double K[6], int s, double dt, int nsteps, int every, const double *d_T0,
                     double *d_T) {
  if (!c || !c->diff_ready || !K || !d_T0 || !d_T || s < 2 || nsteps < 1 || every < 1) return SPH_ERR_BAD_ARG;
  if (c->diff_op != 0) return SPH_ERR_UNSUPPORTED;  // stepped stage by stage by the caller (autograd.py)
  (void)hipSetDevice(c->device);
  const int n = (int)c->n;
  unsigned G = grid_for(n);
  int nck = nsteps / every + 1;
  if ((int64_t)nck * c->npad > c->ckpt_cap) {
    RCHK(dalloc(&c->ckpt, (size_t)nck * c->npad));
    c->ckpt_cap = (int64_t)nck * c->npad;
  }
  RCHK(ensure_dvec(c, V_SEG + std::min(every, nsteps) * s));
  ensure_weights(c, K);
  // a step's last stage writes where the next step's Y_0 is kept: the next
  // checkpoint, its place in the last segment (whose stage states the
  // backward pass then need not recompute), or the state between steps
  const int last_sg = (nsteps - 1) / every;
  std::vector<double *> Y(s + 1);
  double *y0 = c->ckpt;
  int z = 0;
  hipLaunchKernelGGL(k_batch_in, dim3(G), dim3(kBlock), 0, c->stream, d_T0, c->orig[c->cur], c->drho, n, y0,
                     dv(c, V_Z));
  for (int st = 0; st < nsteps; st++) {
    const int sg = st / every, k = st % every;
    if (sg == last_sg) {
      segment_states(c, sg, k, s, Y);
    } else {
      for (int j = 1; j < s; j++) Y[j] = dv(c, V_STATE + j % 3);
    }
    Y[0] = y0;
    if (st == nsteps - 1) y0 = dv(c, V_Y);
    else if (k == every - 1) y0 = c->ckpt + (size_t)(sg + 1) * c->npad;
    else y0 = sg == last_sg ? dv(c, V_SEG + (k + 1) * s) : dv(c, V_Y);
    Y[s] = y0;
    sts_forward_step(c, s, dt, Y.data(), &z);
  }
  hipLaunchKernelGGL(k_from_sorted, dim3(G), dim3(kBlock), 0, c->stream, y0, c->orig[c->cur], n, d_T);
  HIPCHK(hipStreamSynchronize(c->stream));
  c->fw_s = s; c->fw_steps = nsteps; c->fw_every = every; c->fw_dt = dt;
  for (int k = 0; k < 6; k++) c->fw_K[k] = K[k];
  c->fw_tail = true;
  return SPH_OK;
}

int sph_diff_backward(sph_ctx *c, const double *d_gT, double *d_gT0, double gK[6]) {
  if (!c || !c->diff_ready || c->fw_steps < 1 || !d_gT || !d_gT0 || !gK) return SPH_ERR_BAD_ARG;
  (void)hipSetDevice(c->device);
  const int n = (int)c->n, s = c->fw_s, every = c->fw_every, nsteps = c->fw_steps;
  const double dt = c->fw_dt;
  const double *K = c->fw_K;
  unsigned G = grid_for(n);
  ensure_weights(c, K);
  HIPCHK(hipMemsetAsync(c->gkdev, 0, sizeof(double) * 12, c->stream));
  c->rec_pend = c->rec_packed = 0;
  c->coef_set = false;
  int l = 0;  // the vector of the running L
  hipLaunchKernelGGL(k_to_sorted, dim3(G), dim3(kBlock), 0, c->stream, d_gT, c->orig[c->cur], n, dv(c, V_L));
  const int nseg = (nsteps + every - 1) / every;
  std::vector<double *> Y(s + 1);
  for (int sg = nseg - 1; sg >= 0; sg--) {
    const int steps = std::min(nsteps, (sg + 1) * every) - sg * every;
    // the segment's stage states from its checkpoint (the last segment's are
    // still there from the forward pass)
    if (!(sg == nseg - 1 && c->fw_tail)) {
      adj_pack(c, false);  // the last segment's stages, before their states go
      double *ck = c->ckpt + (size_t)sg * c->npad;
      int z = 0;
      hipLaunchKernelGGL(k_batch_in, dim3(G), dim3(kBlock), 0, c->stream, ck, (const int64_t *)nullptr, c->drho, n, ck,
                         dv(c, V_Z));
      for (int k = 0; k < steps; k++) {
        segment_states(c, sg, k, s, Y);
        Y[s] = k + 1 < steps ? dv(c, V_SEG + (k + 1) * s) : nullptr;
        sts_forward_step(c, s, dt, Y.data(), &z, k + 1 < steps);
      }
    }
    for (int k = steps - 1; k >= 0; k--) {
      segment_states(c, sg, k, s, Y);
      sts_backward_step(c, s, dt, Y.data(), &l);
    }
  }
  hipLaunchKernelGGL(k_from_sorted, dim3(G), dim3(kBlock), 0, c->stream, dv(c, V_L + l), c->orig[c->cur], n, d_gT0);
  diff_gcontract(c, K, c->gkdev);
  c->fw_tail = false;  // segment buffers now hold the first segment
  HIPCHK(hipMemcpyAsync(gK, c->gkdev, sizeof(double) * 6, hipMemcpyDeviceToHost, c->stream));
  HIPCHK(hipStreamSynchronize(c->stream));
  return SPH_OK;
}

// Super-steps of the operators that read grad T.  Work vectors: the adjoint's
// L, what is pending for the next, L_0 and the first rate's, a scratch vector,
// the first stage's rate, four states in rotation; then the stage states of a
// checkpoint segment, s per step.
enum { W_L = 0, W_PEND, W_L0, W_LDY0, W_WORK, W_DY0, W_STATE, W_SEG = W_STATE + 4 };

// One super-step (sts_integrator.f90:100-123) over Y[0..s]; with a null Y[s]
// its last stage is left out (the states of a segment's last step).
static int staged_step(sph_ctx *c, const DiffOpArgs &a, int s, double dt, double *const *Y) {
  for (int j = 1; j <= s && Y[j]; j++) {
    double co[4];
    RCHK(sph_sts_coeffs(j, s, co));
    NlStage st{};
    st.out = Y[j];
    st.y0 = Y[0];
    st.dy0 = dv(c, W_DY0);
    st.first = j == 1;
    st.cf = co[2] * dt;
    if (j > 1) {
      st.y1 = Y[j - 1];
      st.y2 = Y[j - 2];
      st.c1 = co[0]; st.c2 = co[1]; st.c0 = 1 - co[0] - co[1]; st.cd = co[3] * dt;
    }
    NL_DISPATCH(nl_apply_k, c, a, Y[j - 1], st);
  }
  return SPH_OK;
}

// dL/dY_0 of one super-step from dL/dY_s, both in W_L; dL/dK added into gkdev.
static int staged_step_adjoint(sph_ctx *c, const DiffOpArgs &a, int s, double dt, double *const *Y) {
  const double *none = nullptr;
  double co[4];
  RCHK(sph_sts_coeffs(1, s, co));
  NlAdjStage st{};
  st.lam = dv(c, W_L); st.pend = dv(c, W_PEND); st.l0 = dv(c, W_L0); st.ldy0 = dv(c, W_LDY0);
  st.c_1 = co[2] * dt;
  for (int j = s; j >= 2; j--) {
    RCHK(sph_sts_coeffs(j, s, co));
    st.c1 = co[0]; st.c2 = co[1]; st.c0 = 1 - co[0] - co[1]; st.cf = co[2] * dt; st.cd = co[3] * dt;
    st.first = j == s;
    st.last = j == 2;
    NL_DISPATCH(nl_adjoint_k, c, a, dv(c, W_L), Y[j - 1], none, dv(c, W_WORK), co[2] * dt, st);
  }
  st.close = 1;
  NL_DISPATCH(nl_adjoint_k, c, a, dv(c, W_LDY0), Y[0], none, dv(c, W_WORK), 1.0, st);
  return SPH_OK;
}

int sph_diff_staged_forward(sph_ctx *c, const double K[6], int s, double dt, int nsteps, int every, const double *d_T0,
                            double *d_T, double *d_ckpt) {
  if (!c || !c->diff_ready || !d_T0 || !d_T || !d_ckpt || s < 2 || nsteps < 1 || every < 1) return SPH_ERR_BAD_ARG;
  if (c->diff_op == 0) return SPH_ERR_UNSUPPORTED;  // sph_diff_forward
  if (!K && c->diff_op != 5) return SPH_ERR_BAD_ARG;
  (void)hipSetDevice(c->device);
  RCHK(ensure_dvec(c, W_SEG));
  const int n = (int)c->n;
  const unsigned G = grid_for(n);
  const int64_t *o = c->orig[c->cur];
  const double K0[6] = {0, 0, 0, 0, 0, 0};
  const DiffOpArgs a = diff_args(c, K ? K : K0);
  double *ring[4];
  for (int k = 0; k < 4; k++) ring[k] = dv(c, W_STATE + k);
  std::vector<double *> Y(s + 1);
  hipLaunchKernelGGL(k_to_sorted, dim3(G), dim3(kBlock), 0, c->stream, d_T0, o, n, ring[0]);
  for (int st = 0; st < nsteps; st++) {
    if (st % every == 0)
      hipLaunchKernelGGL(k_from_sorted, dim3(G), dim3(kBlock), 0, c->stream, ring[0], o, n,
                         d_ckpt + (size_t)(st / every) * n);
    Y[0] = ring[0];
    for (int j = 1; j <= s; j++) Y[j] = ring[1 + (j - 1) % 3];
    RCHK(staged_step(c, a, s, dt, Y.data()));
    std::swap(ring[0], ring[1 + (s - 1) % 3]);
  }
  hipLaunchKernelGGL(k_from_sorted, dim3(G), dim3(kBlock), 0, c->stream, ring[0], o, n, d_T);
  HIPCHK(hipStreamSynchronize(c->stream));
  return SPH_OK;
}

int sph_diff_staged_backward(sph_ctx *c, const double K[6], int s, double dt, int nsteps, int every,
                             const double *d_ckpt, const double *d_gT, double *d_gT0, double gK[6]) {
  if (!c || !c->diff_ready || !d_ckpt || !d_gT || !d_gT0 || !gK || s < 2 || nsteps < 1 || every < 1)
    return SPH_ERR_BAD_ARG;
  if (c->diff_op == 0) return SPH_ERR_UNSUPPORTED;
  if (!K && c->diff_op != 5) return SPH_ERR_BAD_ARG;
  (void)hipSetDevice(c->device);
  RCHK(ensure_dvec(c, W_SEG + std::min(every, nsteps) * s));
  const int n = (int)c->n;
  const unsigned G = grid_for(n);
  const int64_t *o = c->orig[c->cur];
  const double K0[6] = {0, 0, 0, 0, 0, 0};
  const DiffOpArgs a = diff_args(c, K ? K : K0);
  HIPCHK(hipMemsetAsync(c->gkdev, 0, sizeof(double) * 12, c->stream));
  hipLaunchKernelGGL(k_to_sorted, dim3(G), dim3(kBlock), 0, c->stream, d_gT, o, n, dv(c, W_L));
  std::vector<double *> Y(s + 1);
  for (int sg = (nsteps - 1) / every; sg >= 0; sg--) {
    const int steps = std::min(nsteps, (sg + 1) * every) - sg * every;
    auto states = [&](int k) {
      for (int j = 0; j < s; j++) Y[j] = dv(c, W_SEG + k * s + j);
      Y[s] = k + 1 < steps ? dv(c, W_SEG + (k + 1) * s) : nullptr;
    };
    hipLaunchKernelGGL(k_to_sorted, dim3(G), dim3(kBlock), 0, c->stream, d_ckpt + (size_t)sg * n, o, n,
                       dv(c, W_SEG));
    for (int k = 0; k < steps; k++) {
      states(k);
      RCHK(staged_step(c, a, s, dt, Y.data()));
    }
    for (int k = steps - 1; k >= 0; k--) {
      states(k);
      RCHK(staged_step_adjoint(c, a, s, dt, Y.data()));
    }
  }
  hipLaunchKernelGGL(k_from_sorted, dim3(G), dim3(kBlock), 0, c->stream, dv(c, W_L), o, n, d_gT0);
  double g[6];
  HIPCHK(hipMemcpyAsync(g, c->gkdev, sizeof(g), hipMemcpyDeviceToHost, c->stream));
  HIPCHK(hipStreamSynchronize(c->stream));
  std::copy(g, g + 6, gK);
  return SPH_OK;
}

}  // extern "C"

// ------------------------------------------------------- batched problems
// Independent prepared diffusion problems merged into one operator: one
// launch per RKL2 stage covers every particle of every problem, a super-step
// is captured once as a hipGraph and replayed, and the stage kernel's block
// size is picked by timing the candidates on the merged operator.
struct sph_batch {
  int device = 0;
  hipStream_t stream = nullptr;
  int nprob = 0;
  int64_t n = 0, npad = 0, n_pairs = 0;
  int cap = 0;
  std::vector<int64_t> off;            // nprob + 1 offsets of the problems' rows
  int *cnt = nullptr, *pid = nullptr;  // list lengths, problem of each row
  uint32_t *nb = nullptr;              // merged neighbour indices (list layout)
  double *W = nullptr, *rho = nullptr; // merged pair weights, densities
  float *W32 = nullptr;                // merged pair weights in FP32 (precision 1)
  int precision = 0;
  double *dt = nullptr;                // per-problem time steps
  int64_t *orig = nullptr;             // merged row -> position in the concatenated vectors
  double *vec = nullptr;               // Y0, three stage states, DY0, three Z (npad each)
  int block = 256;
  float tune_ms[4] = {0, 0, 0, 0};
  hipGraph_t graph = nullptr;
  hipGraphExec_t gexec = nullptr;
  int graph_s = 0, graph_block = 0;
};

namespace {
constexpr int kBatchBlocks[4] = {64, 128, 256, 512};
constexpr int kBatchVecs = 8;

double *bvec(sph_batch *b, int k) { return b->vec + (size_t)k * b->npad; }

// The launches of one RKL2 super-step of s stages (sts_integrator.f90:87-124)
// from Y_0 (buffer 0, its Z in buffer 5) back into buffers 0 and 5; stage
// states rotate over buffers 1-3, their Z over 6-7.
void batch_super_step(sph_batch *b, int s, int block) {
  double *Y0 = bvec(b, 0), *DY0 = bvec(b, 4), *Z0 = bvec(b, 5);
  double *R[3] = {bvec(b, 1), bvec(b, 2), bvec(b, 3)};
  double *ZR[2] = {bvec(b, 6), bvec(b, 7)};
  auto Y = [&](int j) -> double * { return (j == 0 || j == s) ? Y0 : R[j % 3]; };
  auto Z = [&](int j) -> double * { return (j == 0 || j == s) ? Z0 : ZR[j & 1]; };
  const unsigned G = (unsigned)((b->n + block - 1) / block);
  BatchStage a{};
  a.cnt = b->cnt; a.nb = b->nb; a.W = b->W; a.W32 = b->W32; a.rho = b->rho; a.pid = b->pid; a.dt = b->dt;
  a.Y0 = Y0; a.DY0 = DY0; a.n = (int)b->n; a.npad = (int)b->npad;
  a.Yjm1 = Y0; a.Yjm2 = Y0; a.Zjm1 = Z0; a.Yj = Y(1); a.Zj = Z(1);
  a.mhat = sts_mu_hat(1, s);
  const bool f32 = b->precision == 1;
  if (f32) hipLaunchKernelGGL((k_batch_stage<true, float, false>), dim3(G), dim3(block), 0, b->stream, a);
  else hipLaunchKernelGGL((k_batch_stage<true, double, false>), dim3(G), dim3(block), 0, b->stream, a);
  for (int j = 2; j <= s; j++) {
    a.Yjm1 = Y(j - 1); a.Yjm2 = Y(j - 2); a.Zjm1 = Z(j - 1); a.Yj = Y(j); a.Zj = Z(j);
    a.mu = sts_mu(j); a.nu = sts_nu(j); a.c0 = 1. - a.mu - a.nu;
    a.mhat = sts_mu_hat(j, s); a.ghat = sts_gm_hat(j, s);
    a.rev = (j - 1) & 1;
    if (f32) hipLaunchKernelGGL((k_batch_stage<false, float, false>), dim3(G), dim3(block), 0, b->stream, a);
    else hipLaunchKernelGGL((k_batch_stage<false, double, false>), dim3(G), dim3(block), 0, b->stream, a);
  }
}

void batch_free(sph_batch *b) {
  if (b->gexec) (void)hipGraphExecDestroy(b->gexec);
  if (b->graph) (void)hipGraphDestroy(b->graph);
  void *p[] = {b->cnt, b->pid, b->nb, b->W, b->W32, b->rho, b->dt, b->orig, b->vec};
  for (void *q : p)
    if (q) (void)hipFree(q);
  if (b->stream) (void)hipStreamDestroy(b->stream);
  delete b;
}

// Time one 4-stage super-step per candidate block size (on the zeroed work
// vectors: the stage kernels' work does not depend on the values) and keep
// the fastest.
int batch_autotune(sph_batch *b) {
  hipEvent_t e0, e1;
  HIPCHK(hipEventCreate(&e0));
  HIPCHK(hipEventCreate(&e1));
  float best = 1e30f;
  for (int k = 0; k < 4; k++) {
    const int blk = kBatchBlocks[k];
    batch_super_step(b, 4, blk);  // warm-up
    float t = 1e30f;
    for (int r = 0; r < 3; r++) {
      tolerate(hipEventRecord(e0, b->stream));
      batch_super_step(b, 4, blk);
      tolerate(hipEventRecord(e1, b->stream));
      tolerate(hipEventSynchronize(e1));
      float ms = 0.f;
      tolerate(hipEventElapsedTime(&ms, e0, e1));
      t = std::min(t, ms);
    }
    b->tune_ms[k] = t;
    if (t < best) { best = t; b->block = blk; }
  }
  (void)hipEventDestroy(e0);
  (void)hipEventDestroy(e1);
  HIPCHK(hipGetLastError());
  HIPCHK(hipMemsetAsync(b->vec, 0, sizeof(double) * kBatchVecs * b->npad, b->stream));
  HIPCHK(hipStreamSynchronize(b->stream));
  return SPH_OK;
}
}  // namespace

extern "C" {

int sph_batch_create(sph_ctx *const *ctxs, int nprob, const double *K, int precision, sph_batch **out) {
  if (!ctxs || nprob < 1 || !K || !out || (precision != 0 && precision != 1)) return SPH_ERR_BAD_ARG;
  *out = nullptr;
  int64_t n = 0, np = 0;
  int maxc = 0;
  for (int p = 0; p < nprob; p++) {
    const sph_ctx *c = ctxs[p];
    if (!c || !c->diff_ready || c->device != ctxs[0]->device) return SPH_ERR_BAD_ARG;
    if (c->diff_op != 0) return SPH_ERR_UNSUPPORTED;  // the assembled Hessian operators only
    n += c->n;
    np += c->stats.n_pairs;
    maxc = std::max(maxc, c->last_maxcnt);
  }
  if (n >= ((int64_t)1 << 31) - 64) return SPH_ERR_UNSUPPORTED;  // 32-bit merged row indices
  sph_batch *b = new sph_batch();
  b->device = ctxs[0]->device;
  (void)hipSetDevice(b->device);
  b->nprob = nprob;
  b->precision = precision;
  b->n = n;
  b->n_pairs = np;
  b->npad = (n + 63) / 64 * 64;
  b->cap = std::max(8, (maxc + 7) / 8 * 8);
  b->off.assign(nprob + 1, 0);
  int rc = SPH_OK;
  auto fail = [&](int r) { batch_free(b); return r; };
  if (hipStreamCreateWithFlags(&b->stream, hipStreamNonBlocking) != hipSuccess) return fail(SPH_ERR_HIP);
  const size_t slots = (size_t)b->npad * b->cap;
  if ((rc = dalloc(&b->cnt, b->npad)) || (rc = dalloc(&b->pid, b->npad)) || (rc = dalloc(&b->nb, slots)) ||
      (rc = precision == 1 ? dalloc(&b->W32, slots) : dalloc(&b->W, slots)) || (rc = dalloc(&b->rho, b->npad)) ||
      (rc = dalloc(&b->dt, nprob)) ||
      (rc = dalloc(&b->orig, b->npad)) || (rc = dalloc(&b->vec, kBatchVecs * (size_t)b->npad)))
    return fail(rc);
  if (hipMemset(b->cnt, 0, sizeof(int) * b->npad) != hipSuccess ||
      hipMemset(b->dt, 0, sizeof(double) * nprob) != hipSuccess ||
      hipMemset(b->vec, 0, sizeof(double) * kBatchVecs * b->npad) != hipSuccess || hipDeviceSynchronize() != hipSuccess)
    return fail(SPH_ERR_HIP);
  // each problem's weights for its tensor, then into the merged layout
  for (int p = 0; p < nprob; p++) {
    sph_ctx *c = ctxs[p];
    ensure_weights(c, K + 6 * p);
    hipLaunchKernelGGL(k_batch_merge, dim3(grid_for(c->n)), dim3(kBlock), 0, c->stream, (int)c->n, (int)c->npad,
                       b->off[p], p, c->cnt, c->nb, c->dW, (const double4 *)c->q[0], c->orig[c->cur],
                       (int)b->npad, b->cnt, b->nb, b->W, b->W32, b->rho, b->orig, b->pid);
    if (hipStreamSynchronize(c->stream) != hipSuccess) return fail(SPH_ERR_HIP);
    b->off[p + 1] = b->off[p] + c->n;
  }
  if ((rc = batch_autotune(b))) return fail(rc);
  *out = b;
  return SPH_OK;
}

int sph_batch_destroy(sph_batch *b) {
  if (!b) return SPH_ERR_BAD_ARG;
  (void)hipSetDevice(b->device);
  (void)hipStreamSynchronize(b->stream);
  batch_free(b);
  return SPH_OK;
}

int sph_batch_sts(sph_batch *b, int s, const double *dt, int nsteps, const double *d_T0, double *d_T,
                  int use_graph) {
  if (!b || !dt || !d_T0 || !d_T || s < 2 || nsteps < 0) return SPH_ERR_BAD_ARG;
  (void)hipSetDevice(b->device);
  const unsigned G = grid_for(b->n);
  HIPCHK(hipMemcpyAsync(b->dt, dt, sizeof(double) * b->nprob, hipMemcpyHostToDevice, b->stream));
  hipLaunchKernelGGL(k_batch_in, dim3(G), dim3(kBlock), 0, b->stream, d_T0, b->orig, b->rho, (int)b->n, bvec(b, 0),
                     bvec(b, 5));
  if (use_graph && nsteps > 0) {
    if (!b->gexec || b->graph_s != s || b->graph_block != b->block) {
      if (b->gexec) { (void)hipGraphExecDestroy(b->gexec); b->gexec = nullptr; }
      if (b->graph) { (void)hipGraphDestroy(b->graph); b->graph = nullptr; }
      HIPCHK(hipStreamBeginCapture(b->stream, hipStreamCaptureModeThreadLocal));
      batch_super_step(b, s, b->block);
      HIPCHK(hipStreamEndCapture(b->stream, &b->graph));
      HIPCHK(hipGraphInstantiate(&b->gexec, b->graph, nullptr, nullptr, 0));
      b->graph_s = s;
      b->graph_block = b->block;
    }
    for (int st = 0; st < nsteps; st++) HIPCHK(hipGraphLaunch(b->gexec, b->stream));
  } else {
    for (int st = 0; st < nsteps; st++) batch_super_step(b, s, b->block);
  }
  HIPCHK(hipGetLastError());
  hipLaunchKernelGGL(k_from_sorted, dim3(G), dim3(kBlock), 0, b->stream, bvec(b, 0), b->orig, (int)b->n, d_T);
  HIPCHK(hipStreamSynchronize(b->stream));
  return SPH_OK;
}

int sph_batch_get_info(sph_batch *b, sph_batch_info *info) {
  if (!b || !info) return SPH_ERR_BAD_ARG;
  info->n_problems = b->nprob;
  info->n_total = b->n;
  info->n_pairs = b->n_pairs;
  info->list_cap = b->cap;
  info->block = b->block;
  for (int k = 0; k < 4; k++) {
    info->tune_block[k] = kBatchBlocks[k];
    info->tune_ms[k] = b->tune_ms[k];
  }
  return SPH_OK;
}

int sph_batch_offsets(sph_batch *b, int64_t *off) {
  if (!b || !off) return SPH_ERR_BAD_ARG;
  for (int p = 0; p <= b->nprob; p++) off[p] = b->off[p];
  return SPH_OK;
}

}  // extern "C"
