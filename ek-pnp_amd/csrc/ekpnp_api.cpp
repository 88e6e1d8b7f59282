// ekpnp_api.cpp -- host side of the C ABI declared in include/ekpnp.h.
//
// The context owns every device allocation for all channels; per-channel
// sub-arrays are addressed through ChanDesc offsets.  Nothing here computes
// on the host except parameter bookkeeping, input generation (the seeded cold
// start) and the D2H formatting of outputs.
#include <hip/hip_runtime.h>
#include <sys/mman.h>

#include <algorithm>
#include <atomic>
#include <cerrno>
#include <chrono>
#include <cmath>
#include <condition_variable>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <exception>
#include <string>
#include <thread>
#include <tuple>
#include <vector>

#include "../../include/ekpnp.h"
#include "../../include/ekpnp_seed.h"
#include "ekpnp_internal.h"

#include <rocprofiler-sdk-roctx/roctx.h>

using namespace ekpnp;

namespace {

// A roctx range over one call of an entry point: the host-side span of the
// call (kernel launches, graph replays, copies) as a named range under
// rocprofv3 --marker-trace; with no tool attached a push/pop pair is two
// calls that return at once.
struct ApiRange {
  explicit ApiRange(const char* name) { roctxRangePushA(name); }
  ~ApiRange() { roctxRangePop(); }
  ApiRange(const ApiRange&) = delete;
  ApiRange& operator=(const ApiRange&) = delete;
};

const double W[9] = {4.0 / 9.0, 1.0 / 9.0, 1.0 / 9.0, 1.0 / 9.0, 1.0 / 9.0,
                     1.0 / 36.0, 1.0 / 36.0, 1.0 / 36.0, 1.0 / 36.0};
const int CXH[9] = {0, 1, 0, -1, 0, 1, -1, -1, 1};
// storage references: one record of 8 doubles per row, X (rho, c+, c-) row
// means, J (their x-fluxes), 2 unused; and per row nb block records of
// BLK_STRIDE floats, X over each 64-node block of the row
constexpr int kRefStride = 8;
constexpr int kDftLds = 32768;             // LDS bytes of a narrow rows' direct-DFT tile
constexpr int kMaxTriChunks = TRI_WG / 2;  // the plan keeps G = TRI_WG / C >= 2 modes per work-group

// stored value + ref[d][y][x] = population (FP32 storage; 0 for FP64)
std::vector<double> ref_offsets(ekpnp_ctx* c, int channel, int species, hipError_t* err);

thread_local std::string g_create_error;

bool is_pow2(int n) { return n > 0 && (n & (n - 1)) == 0; }
int pow2_ceil(int v) {
  int p = 1;
  while (p < v) p <<= 1;
  return p;
}

// copy_to_host: bytes per staged piece, pieces in flight, copying threads,
// the size from which it uses several pieces and threads, the size from which it
// asks what the destination is, and how long a thread spins for the next piece
// before it sleeps (a piece's DMA takes 20 to 170 us)
constexpr size_t STAGE_CHUNK = 8u << 20, STAGE_PARALLEL_MIN = 2u << 20, STAGE_ASK_MIN = 64u << 10;
constexpr int STAGE_SLOTS = 3, STAGE_THREADS = 4, STAGE_SPIN_US = 500;

struct ChannelTiles {
  int fft_first, fft_count;  // range in the FFT tile table
  int tri_first, tri_count;  // range in the tridiagonal tile table
  int row_first;             // first of its ny entries in the row table
};

}  // namespace

struct ekpnp_ctx {
  std::vector<ekpnp_channel_params> params;
  ekpnp_options opt{};
  int nchan = 0;
  int elem = 4;  // bytes per population value
  std::vector<ChanDesc> desc;
  std::vector<ChannelTiles> ctiles;
  long long total_nodes = 0, total_spec = 0, total_pops = 0, total_refs = 0, total_blocks = 0;
  int total_nx = 0;
  // host copies
  std::vector<int2> lbm_tiles;
  std::vector<int4> fft_tiles;
  std::vector<int2> tri_tiles;
  std::vector<int> first_tile;
  std::vector<int2> row_tiles;
  int n_row_narrow = 0;          // its first rows, of channels of at most ROW_WAVE_NX nodes a row
  std::vector<double> walls;  // 6 planes x total_nx
  // device
  void* lat[2] = {nullptr, nullptr};
  ChanDesc* d_desc = nullptr;
  int2* d_lbm_tiles = nullptr;
  int2* d_lbm_split = nullptr;   // lbm_split on the device
  std::vector<int2> lbm_split;   // LBM tiles for the step: row-kernel interior, row-kernel wall, others
  int n_lbm_row = 0, n_lbm_wall = 0;
  std::vector<int2> lbm_fwd;     // k_lbm_fwd tiles; empty: the context is too wide or too large for it
  int2* d_lbm_fwd = nullptr;
  int lbm_fwd_kind = FWD_GENERAL;
  bool lbm_inv = false;          // k_lbm_fwd does the step before's inverse x-transforms too
  bool lbm_fuse = false;         // the step takes k_lbm_fwd (the Poisson plan's x-transform is the one it holds)
  int lbm_wrows = 0;             // interior tile shape of the row kernel (0: consecutive blocks)
  size_t lbm_split_cap = 0;      // capacity of d_lbm_split (the largest shape)
  // the coupled step updates the row kernel's wall tiles inside the
  // tridiagonal launch (set with the Poisson plan)
  bool walls_in_tri = false;
  int4* d_fft_tiles = nullptr;
  int2* d_tri_tiles = nullptr;
  int* d_first_tile = nullptr;
  double* d_rho_e = nullptr;
  double* d_psi = nullptr;
  double* d_macro = nullptr;
  double* d_walls = nullptr;
  double2* d_tw = nullptr;
  double2* d_spec = nullptr;
  double2* d_spec2 = nullptr;    // every other step's spectrum (lbm_inv)
  double* d_ux_prev = nullptr;
  double* d_refs = nullptr;      // storage references in use, [ny][8] per channel
  double* d_refs_new = nullptr;  // staging for a change of reference
  float* d_blocks = nullptr;     // block references in use, [ny][nb][BLK_STRIDE] per channel
  float* d_blocks_new = nullptr; // staging for a change of reference
  int2* d_row_tiles = nullptr;
  double* d_partials = nullptr;
  double* d_red = nullptr;
  double* d_diag = nullptr;      // diagnostics: 2 x DIAG_MAX_WG partials, then umax and the current sum
  double* d_cprime = nullptr;    // chunk-entry Thomas coefficients (Poisson plan)
  long long total_cprime = 0;    // its capacity: kMaxTriChunks x nk per channel
  size_t dev_bytes = 0;
  int max_lds = 65536;
  hipStream_t stream = nullptr;
  StepBuffers sb{};
  // state
  int cur = 0;          // lattice holding the current state
  bool state_q = false; // current lattice holds unshifted pre-collision populations
  bool has_fields = false, has_pops = false;
  long long steps = 0;
  long long snapshot_step = -1;
  long long rebase_step = 0;  // step count at the last change of storage reference
  long long origin_step = 0;  // step count when init_equilibrium last set the populations
  // Poisson work decomposition (see build_poisson_plan)
  int fft_elems = 2048, tri_rows = 16, fft_persist = 1;
  int n_cu = 256;
  size_t fft_tiles_cap = 0, tri_tiles_cap = 0;
  unsigned max_lds_needed = 0;
  // pinned staging of copy_to_host, allocated on first use and grown to the
  // largest field read (at most STAGE_SLOTS x STAGE_CHUNK bytes)
  char* stage = nullptr;
  size_t stage_bytes = 0;
  hipEvent_t stage_ev[STAGE_SLOTS + 1] = {};  // a piece has come; the work before the copy is done
  std::map<std::tuple<int, int, int, int>, hipGraphExec_t> graphs;
  std::string err;
};

namespace {

int fail(ekpnp_ctx* c, int code, const std::string& msg) {
  if (c) c->err = msg;
  return code;
}

#define HIP_OR_FAIL(ctx, call)                                                     \
  do {                                                                             \
    hipError_t e_ = (call);                                                        \
    if (e_ != hipSuccess)                                                          \
      return fail((ctx), EKPNP_ERR_HIP,                                            \
                  std::string(#call) + ": " + hipGetErrorString(e_));              \
  } while (0)

std::string validate(const ekpnp_channel_params& p, int ch) {
  char buf[256];
  auto bad = [&](const char* what) {
    snprintf(buf, sizeof buf, "channel %d: %s", ch, what);
    return std::string(buf);
  };
  if (p.nx < 2) return bad("nx < 2");
  if (p.ny < 4) return bad("ny < 4");
  if (is_pow2(p.nx) && p.nx > MAX_NX) return bad("power-of-two nx above 8192");
  if (!is_pow2(p.nx) && p.nx > MAX_NX_DFT) return bad("non-power-of-two nx above 2048");
  if (p.ny - 2 > MAX_INTERIOR_ROWS) return bad("ny above 2050");
  if (!(p.dx > 0 && p.dy > 0 && p.dt > 0 && p.cfl > 0 && p.cs2 > 0)) return bad("non-positive dx/dy/dt/cfl/cs2");
  if (!(p.nu > 0 && p.diff_pos > 0 && p.diff_neg > 0)) return bad("non-positive viscosity or diffusivity");
  if (!(p.magic_f > 0 && p.magic_pos > 0 && p.magic_neg > 0)) return bad("non-positive TRT magic parameter");
  if (!(p.rho0 > 0)) return bad("non-positive rho0");
  if (!(p.lx > 0)) return bad("non-positive lx");
  // the x length sets the x-FFT wavenumbers, dx the lattice: LX = NX dx
  // (LBM.h:35-42)
  if (std::fabs(p.lx - p.nx * p.dx) > 1e-9 * p.lx) return bad("lx differs from nx * dx");
  if (!std::isfinite(p.poisson_coef) || !std::isfinite(p.force_coef)) return bad("non-finite coefficient");
  return std::string();
}

// EKPNP_CHECK_* flags of one channel (ekpnp_check_params)
uint32_t check_flags(const ekpnp_channel_params& p, double* kappa_dy, double* drift, double* flow) {
  const double kappa = std::sqrt(std::max(0.0, 2.0 * p.poisson_coef * p.c_bulk * p.inv_thermal_voltage));
  const double zw = std::max(std::fabs(p.psi_lo), std::fabs(p.psi_hi));
  const double kmax = std::max(std::fabs(p.mob_pos), std::fabs(p.mob_neg));
  const double ivt = p.inv_thermal_voltage;
  const double ew = ivt > 0.0 ? 2.0 * kappa / ivt * std::sinh(0.5 * ivt * zw) : 0.0;  // wall field
  *kappa_dy = kappa * p.dy;
  *drift = kmax * ew * p.dt / p.dx;
  // the bulk electro-osmotic velocity: nu rho0 u'' = -force_coef rho_e E_x
  // and psi'' = -poisson_coef rho_e give u = force_coef E_x (psi - zeta) /
  // (poisson_coef nu rho0), in dx/dt units
  const double den = p.poisson_coef * p.nu * p.rho0;
  *flow = den != 0.0 ? std::fabs(p.force_coef * p.e_applied * zw / den) * p.dt / p.dx : 0.0;
  uint32_t f = 0;
  if (!(*kappa_dy <= 0.4)) f |= EKPNP_CHECK_DEBYE_UNRESOLVED;
  if (!(*drift <= 0.05)) f |= EKPNP_CHECK_WALL_DRIFT;
  if (!(*flow <= 0.1)) f |= EKPNP_CHECK_FLOW_FAST;
  return f;
}

ChanDesc make_desc(const ekpnp_channel_params& p, int precision) {
  ChanDesc d{};
  d.nx = p.nx;
  d.ny = p.ny;
  d.nk = p.nx / 2 + 1;
  d.nk_stride = (d.nk + 7) / 8 * 8;  // modes rounded up to whole blocks of 8
  d.active = 1;
  d.swap = 0;
  d.flags = (int)p.flags;
  d.pow2 = (is_pow2(p.nx) && p.nx >= 8) ? 1 : 0;
  d.nb = (p.nx + REF_BLOCK - 1) / REF_BLOCK;
  const double cs2 = p.cs2, dt = p.dt;
  // relaxation rates, LBM.cu:336-341
  const double omega_plus = 1.0 / (p.nu / cs2 / dt + 1.0 / 2.0) / dt;
  const double omega_minus = 1.0 / (p.magic_f / (p.nu / cs2 / dt) + 1.0 / 2.0) / dt;
  const double omega_c_minus = 1.0 / (p.diff_pos / cs2 / dt + 1.0 / 2.0) / dt;
  const double omega_c_plus = 1.0 / (p.magic_pos / (p.diff_pos / cs2 / dt) + 1.0 / 2.0) / dt;
  const double omega_T_minus = 1.0 / (p.diff_neg / cs2 / dt + 1.0 / 2.0) / dt;
  const double omega_T_plus = 1.0 / (p.magic_neg / (p.diff_neg / cs2 / dt) + 1.0 / 2.0) / dt;
  d.inv_cfl = 1.0 / p.cfl;
  d.inv_cs2 = 1.0 / cs2;
  d.om_pf = omega_plus * dt;
  d.om_mf = omega_minus * dt;
  d.om_pp = omega_c_plus * dt;
  d.om_mp = omega_c_minus * dt;
  d.om_pn = omega_T_plus * dt;
  d.om_mn = omega_T_minus * dt;
  d.src_p = 1.0 - 0.5 * dt * omega_plus;  // LBM.cu:745-746
  d.src_m = 1.0 - 0.5 * dt * omega_minus;
  d.dt = dt;
  d.half_dt = 0.5 * dt;
  d.kp = p.mob_pos;
  d.kn = p.mob_neg;
  d.fcoef = p.force_coef;
  d.e_app = p.e_applied;
  d.exf = p.exf;
  d.drift_app = (p.flags & EKPNP_FLAG_ION_DRIFT_APPLIED) ? p.e_applied : 0.0;
  d.inv2dx = 0.5 / p.dx;
  d.inv2dy = 0.5 / p.dy;
  d.multis = 2.0 * p.rho0 * p.uw / cs2 * (1.0 / 9.0) / p.cfl;  // LBM.cu:812-813
  d.multid = 2.0 * p.rho0 * p.uw / cs2 * (1.0 / 36.0) / p.cfl;
  d.pc_dy2 = p.poisson_coef * p.dy * p.dy;
  d.kdy_scale = 2.0 * M_PI / p.lx * p.dy;
  d.c_bulk = p.c_bulk;
  d.inv_vt = p.inv_thermal_voltage;
  d.pb_omega = p.pb_omega;
  return d;
}

// How many of the 27 population planes go through the caches (an index into
// LBM_CACHED).  A streamed plane is read from and written to HBM every step; a
// cached one is found in the 256 MB Infinity Cache if both its lattices still
// lie there a step later, and one that does not evicts psi and the spectrum for
// nothing.  So as many planes as fit LBM_CACHE_BYTES: the largest count of
// LBM_CACHED whose planes, both lattices of them (bytes: all 27), stay within
// it (FP64 storage without narrow channels: LBM_CACHE_BYTES_FP64, but for the first
// two planes).  k_lbm (the widths the row kernel does not take, FP64 storage) gains from
// whole lattices a little longer, up to LBM_CACHE_BYTES_WHOLE, and with FP32
// storage and narrow channels only from whole ones; the row kernel and FP64
// storage stream what is below LBM_CACHE_BYTES_MIN, which the L2 caches serve
// better so.  Step in us, nothing cached -> the rule's count [another count]:
//   32 channels fp32   33 MB  34.9 (0)                 [37.7 with 27]
//   512x256     fp64   57 MB  30.6 (0)                 [31.8 with 27]
//   64x128 x32  fp32   57 MB  33.9 (0)                 [34.7 with 27]
//   128x128 x24 fp32   85 MB  43.0 -> 41.2 (27)
//   512x400     fp64   88 MB  41.1 -> 37.8 (27)
//   1024x514    fp32  114 MB  54.1 -> 49.7 (27)
//   1024x1026   fp32  227 MB  82.2 -> 75.7 (18)        [80.6 with 27]
//   1024x514    fp64  227 MB  80.1 -> 60.3 (27)        [63.8 with 18]
//   1024x800    fp64  354 MB  100.7 -> 86.9 (13)       [89.4 with 9, 87.8 with 18, 103 with 27]
//   512x1800    fp64  398 MB  98.4 (13)                [105.8 with 9]
//   1024x1300   fp64  575 MB  140.9 (9)                [146.0 with 6, 147.6 with 13]
//   1000x1300   fp64  562 MB  332.7 (9)                [340.5 with 6]
//   64x128 x150 fp64  531 MB  121.3 (6)                [121.9 with 9]
//   4x200 x700  fp64  242 MB  79.5 (13)                [81.2 with 18]
//   1024x2000   fp64  885 MB  191.3 (6)                [205.8 with 4, 218.9 with 9]
//   4096x640    fp64 1132 MB  282.1 -> 256.6 (4)       [262.4 with 2, 269.1 with 6]
//   4096x1330   fp64 2353 MB  531.9 (0)                [540.0 with 2]
//   2048x1024   fp32  453 MB  139.6 -> 131.8 (9)       [136.8 with 13]
//   4096x700    fp32  619 MB  181.5 -> 169.0 (6)       [170.9 with 9]
//   2048x1024   fp64  906 MB  210.3 -> 195.2 (4)       [214.7 with 9]
//   4096x1024   fp32  906 MB  230.3 -> 220.1 (4)       [235.1 with 6]
//   4096x1400   fp32 1239 MB  335.6 -> 326.8 (2)       [342.4 with 4]
//   4096x1024   fp64 1812 MB  393.2 -> 369.7 (2)       [396.7 with 4]
//   8192x2048   fp32 3624 MB  955.1 (0)                [956.9 with 2]
// and k_lbm with FP32 storage:
//   n_x = 8 x200       62 MB  42.1 -> 36.6 (27)        [40.9 with 13]
//   n_x = 32 x300     213 MB  75.7 -> 68.0 (27)        [75.0 with 13]
//   1000x1001         216 MB  214.1 -> 201.0 (27)      [207.1 with 13]
//   1000x1251         270 MB  272.3 -> 264.1 (13)      [269.9 with 27]
//   1500x1201         389 MB  528.0 -> 517.5 (9)       [523.0 with 18]
//   n_x = 8 x1000     294 MB  120.6 (0)                [120.3 with 13, 125.8 with 27]
//   n_x = 8 x4000    1178 MB  418.6 (0)                [433.1 with 2]
constexpr double LBM_CACHE_BYTES = 160e6, LBM_CACHE_BYTES_FP64 = 200e6, LBM_CACHE_BYTES_WHOLE = 230e6,
                 LBM_CACHE_BYTES_MIN = 80e6;
// narrowest channel of k_lbm with a part (FP64 storage: a larger part) of the planes cached
constexpr int LBM_CACHE_PART_NX = 256;

int lbm_cached_planes(double bytes, bool fp64, bool rows, int min_nx) {
  if (!rows && bytes <= LBM_CACHE_BYTES_WHOLE && (!fp64 || bytes >= LBM_CACHE_BYTES_MIN)) return LBM_CACHED_ALL;
  if ((!rows && !fp64 && min_nx < LBM_CACHE_PART_NX) || bytes < LBM_CACHE_BYTES_MIN) return 0;
  const double most = fp64 && min_nx >= LBM_CACHE_PART_NX ? LBM_CACHE_BYTES_FP64 : LBM_CACHE_BYTES;
  int i = 0;
  while (i < LBM_CACHED_ALL && LBM_CACHED[i + 1] / 27.0 * bytes <= (i > 0 ? most : LBM_CACHE_BYTES)) ++i;
  return i;
}

StepBuffers make_buffers(ekpnp_ctx* c) {
  StepBuffers b{};
  b.chans = c->d_desc;
  b.lbm_tiles = c->d_lbm_tiles;
  b.n_lbm_tiles = (int)c->lbm_tiles.size();
  b.fft_tiles = c->d_fft_tiles;
  b.n_fft_tiles = (int)c->fft_tiles.size();
  b.tri_tiles = c->d_tri_tiles;
  b.n_tri_tiles = (int)c->tri_tiles.size();
  b.rho_e = c->d_rho_e;
  b.psi = c->d_psi;
  b.macro = c->d_macro;
  b.macro_stride = c->total_nodes;
  b.walls = c->d_walls;
  b.walls_stride = c->total_nx;
  b.tw = c->d_tw;
  b.spec = c->d_spec;
  b.spec_prev = c->d_spec;
  b.ux_prev = c->d_ux_prev;
  b.partials = c->d_partials;
  b.red_out = c->d_red;
  b.red_first_tile = c->d_first_tile;
  b.n_channels = c->nchan;
  b.refs = c->d_refs;
  b.blocks = c->d_blocks;
  b.row_tiles = c->d_row_tiles;
  b.n_row_tiles = (int)c->row_tiles.size();
  b.n_row_narrow = c->n_row_narrow;
  b.cprime = c->d_cprime;
  b.lbm_row_tiles = c->d_lbm_split;
  b.n_lbm_row_tiles = c->n_lbm_row;
  b.lbm_wall_tiles = c->d_lbm_split + c->n_lbm_row;
  b.n_lbm_wall_tiles = c->n_lbm_wall;
  b.lbm_gen_tiles = c->d_lbm_split + c->n_lbm_row + c->n_lbm_wall;
  b.n_lbm_gen_tiles = (int)c->lbm_split.size() - c->n_lbm_row - c->n_lbm_wall;
  b.lbm_wrows = c->lbm_wrows;
  b.lbm_fwd_tiles = c->d_lbm_fwd;
  b.n_lbm_fwd_tiles = (int)c->lbm_fwd.size();
  b.lbm_fwd_kind = c->lbm_fwd_kind;
  const bool fp64 = c->opt.precision == EKPNP_POP_FP64;
  const double pop_bytes = 2.0 * (double)c->total_pops * (fp64 ? 8 : 4);
  int min_nx = MAX_NX;
  for (const auto& d : c->desc) min_nx = std::min(min_nx, d.nx);
  b.lbm_cached = lbm_cached_planes(pop_bytes, fp64, false, min_nx);
  b.lbm_rows_cached = lbm_cached_planes(pop_bytes, fp64, true, min_nx);
  return b;
}

template <typename T>
hipError_t dalloc(ekpnp_ctx* c, T** p, size_t count) {
  size_t bytes = std::max<size_t>(count * sizeof(T), 16);
  hipError_t e = hipMalloc((void**)p, bytes);
  if (e == hipSuccess) c->dev_bytes += bytes;
  return e;
}

void drop_graphs(ekpnp_ctx* c);

void release(ekpnp_ctx* c) {
  drop_graphs(c);
  void* ptrs[] = {c->lat[0], c->lat[1], c->d_desc, c->d_lbm_tiles, c->d_fft_tiles,
                  c->d_tri_tiles, c->d_first_tile, c->d_rho_e, c->d_psi, c->d_macro,
                  c->d_walls, c->d_tw, c->d_spec, c->d_spec2, c->d_ux_prev, c->d_partials, c->d_red,
                  c->d_refs, c->d_refs_new, c->d_row_tiles, c->d_cprime, c->d_lbm_split,
                  c->d_blocks, c->d_blocks_new, c->d_diag, c->d_lbm_fwd};
  for (void* p : ptrs)
    if (p) (void)hipFree(p);
  if (c->stage) (void)hipHostFree(c->stage);
  for (auto e : c->stage_ev)
    if (e) (void)hipEventDestroy(e);
  if (c->stream) (void)hipStreamDestroy(c->stream);
  c->stream = nullptr;
}

void drop_graphs(ekpnp_ctx* c) {
  for (auto& kv : c->graphs) (void)hipGraphExecDestroy(kv.second);
  c->graphs.clear();
}

// The step's split of the LBM tiles (FP32 storage, FP64 arithmetic):
// channels with nx a multiple of 64 run on the row kernel, the others on
// k_lbm.  The row kernel's wall launch takes the tiles of consecutive 64-node
// blocks that hold a wall row; its interior launch those that hold an
// interior row (wrows = 0) or tiles of wrows interior rows x 4 / wrows
// blocks (wrows = 2, 4).  EKPNP_LBM_ROWS=0 in the environment keeps every
// tile on k_lbm.
void build_lbm_split(ekpnp_ctx* c, int wrows) {
  const char* env = std::getenv("EKPNP_LBM_ROWS");
  const bool use_rows = !(env && env[0] == '0');
  std::vector<int2> wall, gen;
  c->lbm_split.clear();
  for (const int2& t : c->lbm_tiles) {
    const ChanDesc& d = c->desc[t.x];
    if (!use_rows || d.nx % 64 != 0) {
      gen.push_back(t);
      continue;
    }
    const int last = std::min(t.y + LBM_WG, d.nx * d.ny) - 1;  // last node of the tile
    const int ya = t.y / d.nx, yb = last / d.nx;
    if (ya == 0 || yb == d.ny - 1) wall.push_back(t);
    if (wrows == 0 && !(ya == yb && (ya == 0 || ya == d.ny - 1))) c->lbm_split.push_back(t);
  }
  if (wrows > 0 && use_rows)
    for (int i = 0; i < c->nchan; ++i) {
      const ChanDesc& d = c->desc[i];
      if (d.nx % 64 != 0) continue;
      const int nblk = d.nx / 64, bpt = (LBM_WG / 64) / wrows;
      for (int y0 = 1; y0 <= d.ny - 2; y0 += wrows)
        for (int k0 = 0; k0 < nblk; k0 += bpt) c->lbm_split.push_back(make_int2(i, y0 * d.nx + 64 * k0));
    }
  c->n_lbm_row = (int)c->lbm_split.size();
  c->n_lbm_wall = (int)wall.size();
  c->lbm_split.insert(c->lbm_split.end(), wall.begin(), wall.end());
  c->lbm_split.insert(c->lbm_split.end(), gen.begin(), gen.end());
  c->lbm_wrows = wrows;
}

// x-transform of a channel, in the order of the FFT tile table: 0 power-of-two
// FFT, 1 matrix-core direct DFT, 2 direct DFT of narrow rows
int x_family(const ChanDesc& d) { return d.pow2 ? 0 : d.nx >= DFT_MIN_NX ? 1 : 2; }

// Tiles of k_lbm_fwd: contexts of FP64 arithmetic whose every channel has rows
// of at most LBM_WG nodes, of a power of two or of the narrow rows' direct DFT,
// as long as the chip is not full: the transform holds every work-group for
// some us longer, which is less than the launches it saves only while there are
// few work-groups a CU (n_cu = 256).  Step in us, launches apart -> this one,
// with the inverse transforms where the rule below puts them in:
//   10x101 fp64              4 tiles  18.4 -> 13.5
//   64x128 fp64             32        21.7 -> 16.3
//   256x256 fp32           256        26.0 -> 18.6
//   32 channels (32, 64)   576        35.2 -> 23.4
//   64x128 x48 fp32       1536        41.5 -> 38.7    64x128 x56 fp32  1792  44.0 -> 44.7
//   64x128 x40 fp64       1280        42.7 -> 40.4    64x128 x64 fp64  2048  56.4 -> 58.7
//   32 wide x90           1040        33.2 -> 32.0    32 wide x120     1448  37.2 -> 36.9, 36.4
// (two draws of heights 64 and 128) and with rows below 24 nodes, FP32 storage:
//   n_x = 4 x1100         2750        70.4 -> 63.1    n_x = 4 x1300    3250  89.3 -> 89.4
//   n_x = 8 x450          2800        51.4 -> 50.6    12, 20 x400      4000  99.5 -> 100.6
// 16 nodes are not narrow: their transforms apart are the pipelined kernels'
// (n_y = 128, and 60: the last tile of a channel partly empty):
//   n_x = 16 x192         1536        38.2 -> 35.9    n_x = 16 x208    1664  39.0 -> 40.3
//   n_x = 16, 60 x384     1536        38.5 -> 37.6    n_x = 16, 60 x416 1664 40.0 -> 43.7, x768 3072 54.9 -> 64.1
constexpr int LBM_FWD_TILES_PER_CU = 6, LBM_FWD_TILES_PER_CU_NARROW = 12, LBM_FWD_NARROW_POW2 = 8;
// The inverse x-transforms of the step before are in that launch too, with FP64
// storage while it is emptier still (each work-group transforms a row to either
// side as well: half as much again at 4 rows a tile, three times at one).  Step
// in us, inverse apart -> in it:
//   10x101 fp64     4 tiles  15.5 -> 13.5    32 channels (32, 64)  576  29.6 -> 23.4
//   64x128 fp64    32        18.7 -> 16.3    n_x = 4 x512 fp32    1280  38.7 -> 35.2
//   256x256 fp32  256        21.8 -> 18.6    64x128 x48 fp32      1536  41.0 -> 38.7
//   256x512 fp64  512        29.1 -> 25.4    256x96 x15 fp32      1440  40.5 -> 40.1
//   256x1000 fp64 1000       37.6 -> 38.4
//   64x128 x32 fp64 1024     35.4 -> 36.4
// Narrow rows with FP32 storage: past LBM_FWD_TILES_PER_CU only with rows that hold whole
// groups of 4 nodes (or at most 4), of 8 nodes up to LBM_FWD_INV_TILES_PER_CU_8; the others'
// spectra, of an even number of modes a row or ragged tiles, lose:
//   n_x = 4 x597         1791  44.9 -> 43.6    x939  2817  61.1 -> 59.3
//   n_x = 12 x358        1790  41.3 -> 41.1    x614  3070  59.4 -> 58.9    x409  2045  46.4 -> 44.1
//   n_x = 20 x138        1794  39.6 -> 39.0    x177  2301  45.9 -> 44.6    x217  2821  51.0 -> 52.2
//   n_x = 8 x299         1794  41.8 -> 41.4    x384  2304  47.2 -> 47.4    x512  3072  55.3 -> 58.2
//   n_x = 6 x384         1536  38.4 -> 37.7    x512  2048  45.4 -> 48.3    x704  2816  57.1 -> 61.5
//   n_x = 7 x384         1536  37.8 -> 37.7    x448  1792  42.3 -> 43.9    x768  3072  58.2 -> 63.4
//   n_x = 10 x307        1535  37.3 -> 35.9    x358  1790  39.6 -> 40.6    x614  3070  54.3 -> 58.1
//   n_x = 18 x192        1536  36.6 -> 35.8    x224  1792  39.9 -> 41.2    x384  3072  56.6 -> 60.3
constexpr int LBM_FWD_INV_TILES_PER_CU_FP64 = 3, LBM_FWD_INV_TILES_PER_CU_8 = 9;
void build_lbm_fwd(ekpnp_ctx* c) {
  c->lbm_fwd.clear();
  for (auto& d : c->desc) d.lbm_span = d.nx <= LBM_WG ? LBM_WG / d.nx * d.nx : LBM_WG;
  if (c->opt.precision == EKPNP_POP_FP32 && !c->opt.compute_fp64) return;
  for (const auto& d : c->desc)
    if (d.nx > LBM_WG || x_family(d) == 1) return;
  const char* env = std::getenv("EKPNP_LBM_ROWS");
  const bool use_rows = c->opt.precision == EKPNP_POP_FP32 && !(env && env[0] == '0');
  int n_rows = 0;
  for (int i = 0; i < c->nchan; ++i) {
    const ChanDesc& d = c->desc[i];
    n_rows += use_rows && d.nx % 64 == 0;
    for (int n = 0; n < d.nx * d.ny; n += d.lbm_span) c->lbm_fwd.push_back(make_int2(i, n));
  }
  c->lbm_fwd_kind = n_rows == 0 ? FWD_GENERAL : n_rows == c->nchan ? FWD_ROWS : FWD_MIXED;
  const bool fp64 = c->opt.precision == EKPNP_POP_FP64;
  bool narrow = !fp64, groups = true, eight = false;
  for (const auto& d : c->desc) {
    narrow = narrow && d.nx < DFT_MIN_NX && (!d.pow2 || d.nx <= LBM_FWD_NARROW_POW2);
    groups = groups && (d.nx <= 4 || d.nx % 4 == 0);
    eight = eight || d.nx == LBM_FWD_NARROW_POW2;
  }
  const int most = narrow ? LBM_FWD_TILES_PER_CU_NARROW : LBM_FWD_TILES_PER_CU;
  const int most_inv = fp64 ? LBM_FWD_INV_TILES_PER_CU_FP64
                       : !(narrow && groups) ? LBM_FWD_TILES_PER_CU
                       : eight ? LBM_FWD_INV_TILES_PER_CU_8 : most;
  if (c->lbm_fwd.size() > (size_t)most * c->n_cu) c->lbm_fwd.clear();
  c->lbm_inv = !c->lbm_fwd.empty() && c->lbm_fwd.size() <= (size_t)most_inv * c->n_cu;
}

// a new interior tile shape for the row kernel: table, buffers, graphs
hipError_t apply_lbm_tiles(ekpnp_ctx* c, int wrows) {
  hipError_t e = hipStreamSynchronize(c->stream);  // no launch still reads the table
  if (e != hipSuccess) return e;
  build_lbm_split(c, wrows);
  if (c->lbm_split.size() > c->lbm_split_cap) return hipErrorInvalidValue;
  e = hipMemcpy(c->d_lbm_split, c->lbm_split.data(), c->lbm_split.size() * sizeof(int2), hipMemcpyHostToDevice);
  if (e != hipSuccess) return e;
  const StepBuffers nb = make_buffers(c);
  c->sb.lbm_row_tiles = nb.lbm_row_tiles;
  c->sb.n_lbm_row_tiles = nb.n_lbm_row_tiles;
  c->sb.lbm_wall_tiles = nb.lbm_wall_tiles;
  c->sb.n_lbm_wall_tiles = nb.n_lbm_wall_tiles;
  c->sb.lbm_gen_tiles = nb.lbm_gen_tiles;
  c->sb.n_lbm_gen_tiles = nb.n_lbm_gen_tiles;
  c->sb.lbm_wrows = wrows;
  drop_graphs(c);
  return hipSuccess;
}

// Poisson work decomposition.  x-FFT: a work-group transforms whole rows,
// up to fft_elems complex values (power-of-two channels and narrow others; the
// matrix-core direct DFT takes 16 or 32 rows per work-group); the tiles are
// sorted by family (x_family).  Tridiagonal: each column is cut into C = 2^k chunks of at
// most about tri_rows rows (8 <= C <= 128), G = TRI_WG / C modes per
// work-group.  Rebuilding drops the cached graphs (their grids change).
hipError_t build_poisson_plan(ekpnp_ctx* c, int fft_elems, int tri_rows, int fft_persist) {
  c->fft_tiles.clear();
  c->tri_tiles.clear();
  unsigned lds_pow2 = 16, lds_dft = 16, lds_pow2_tw = 16;  // rows; rows + quadrant table
  unsigned lds_pow2_t2 = 16;                                 // rows + two-level table
  int n_fft_pow2 = 0, n_fft_dft = 0, groups_fwd = 1, groups_inv = 1;
  unsigned dft_lds = 16;
  // wide row-pair kernels: every power-of-two channel has rows of
  // N = FFT_PAIR_WIDE_S * FFT_WG_ROWS complex values (nx = 8192), asked for
  // as fft_elems = N with the row-pair family; tiles of two rows, one row
  // buffer and the two-level twiddle table in LDS
  constexpr int kWideN = FFT_PAIR_WIDE_S * FFT_WG_ROWS;
  bool wide = fft_persist == 2 && fft_elems == kWideN;
  int n_pow2_chan = 0;
  for (const auto& d : c->desc)
    if (d.pow2) {
      ++n_pow2_chan;
      wide = wide && d.nx == 2 * kWideN;
    }
  wide = wide && n_pow2_chan > 0;
  const unsigned wide_lds = (unsigned)((kWideN + tw2_count(2 * kWideN)) * sizeof(double2));
  wide = wide && wide_lds <= (unsigned)c->max_lds;
  for (int pass = 0; pass < 3; ++pass) {
    for (int i = 0; i < c->nchan; ++i) {
      ChanDesc& d = c->desc[i];
      if (pass != x_family(d)) continue;
      const int M = d.ny - 2;
      int rows = 1, dft_wr = 0;
      if (d.pow2) {
        const int N = d.nx / 2;
        rows = wide ? 2 : std::max(1, std::min(std::min(M, FFT_MAX_ROWS), fft_elems / N));
        // rows are padded to whole 16-element groups (LDS swizzle)
        const int padded = (rows * N + 15) & ~15;
        lds_pow2 = std::max<unsigned>(lds_pow2, (unsigned)(padded * sizeof(double2)));
        lds_pow2_tw = std::max<unsigned>(lds_pow2_tw, (unsigned)((padded + d.nx / 4) * sizeof(double2)));
        const int t2 = tw2_count(d.nx);  // the kernels' two-level twiddle table
        lds_pow2_t2 = std::max<unsigned>(lds_pow2_t2, (unsigned)((padded + t2) * sizeof(double2)));
      } else if (d.nx >= DFT_MIN_NX) {
        // matrix-core direct DFT: 16 rows per row tile, the four waves of a
        // work-group split between rows and columns by the width (k_dft_fwd)
        dft_wr = d.nx <= 32 ? 2 : 1;
        rows = 16 * dft_wr;
        dft_lds = std::max(dft_lds, dft_lds_bytes(d.nx));
        const int cols = 64 / dft_wr;
        groups_fwd = std::max(groups_fwd, (d.nk + cols - 1) / cols);
        groups_inv = std::max(groups_inv, (d.nx + cols - 1) / cols);
      } else {
        // narrow rows: as many whole rows as fit fft_elems values and
        // kDftLds bytes of LDS (a row of nx | 1 right-hand-side values, or
        // its nk spectrum values)
        const int per_row = (int)std::max((d.nx | 1) * sizeof(double), d.nk * sizeof(double2));
        rows = std::max(1, std::min({M, fft_elems / d.nx, kDftLds / per_row}));
        lds_dft = std::max<unsigned>(lds_dft, (unsigned)(rows * per_row));
      }
      d.fft_rows = rows;
      c->ctiles[i].fft_first = (int)c->fft_tiles.size();
      for (int y0 = 1; y0 <= M; y0 += rows)
        c->fft_tiles.push_back(make_int4(i, y0, std::min(rows, M + 1 - y0), dft_wr));
      c->ctiles[i].fft_count = (int)c->fft_tiles.size() - c->ctiles[i].fft_first;
    }
    if (pass == 0) n_fft_pow2 = (int)c->fft_tiles.size();
    if (pass == 1) n_fft_dft = (int)c->fft_tiles.size() - n_fft_pow2;
  }
  int tri_lmax = 1;
  for (int i = 0; i < c->nchan; ++i) {
    ChanDesc& d = c->desc[i];
    const int M = d.ny - 2;
    int C = pow2_ceil((M + tri_rows - 1) / tri_rows);
    C = std::max(8, std::min(kMaxTriChunks, C));
    d.tri_C = C;
    d.tri_L = (M + C - 1) / C;
    d.tri_G = TRI_WG / C;
    c->ctiles[i].tri_first = (int)c->tri_tiles.size();
    for (int k0 = 0; k0 < d.nk; k0 += d.tri_G) c->tri_tiles.push_back(make_int2(i, k0));
    c->ctiles[i].tri_count = (int)c->tri_tiles.size() - c->ctiles[i].tri_first;
    tri_lmax = std::max(tri_lmax, d.tri_L);
  }
  if (tri_lmax > TRI_LMAX) return hipErrorInvalidValue;  // ny is validated against MAX_INTERIOR_ROWS
  if (c->fft_tiles.size() > c->fft_tiles_cap || c->tri_tiles.size() > c->tri_tiles_cap) return hipErrorInvalidValue;
  hipError_t e = hipMemcpy(c->d_fft_tiles, c->fft_tiles.data(), c->fft_tiles.size() * sizeof(int4),
                           hipMemcpyHostToDevice);
  if (e != hipSuccess) return e;
  e = hipMemcpy(c->d_tri_tiles, c->tri_tiles.data(), c->tri_tiles.size() * sizeof(int2), hipMemcpyHostToDevice);
  if (e != hipSuccess) return e;
  e = hipMemcpy(c->d_desc, c->desc.data(), c->nchan * sizeof(ChanDesc), hipMemcpyHostToDevice);
  if (e != hipSuccess) return e;
  // chunk-entry Thomas coefficients of the new chunking (one launch)
  long long max_entries = 0;
  for (const auto& d : c->desc) max_entries = std::max(max_entries, (long long)d.tri_C * d.nk);
  e = launch_cprime_tables(c->sb, c->nchan, max_entries, c->stream);
  if (e != hipSuccess) return e;
  c->sb.fft_tiles = c->d_fft_tiles;
  c->sb.n_fft_tiles = (int)c->fft_tiles.size();
  c->sb.n_fft_pow2 = n_fft_pow2;
  c->sb.tri_tiles = c->d_tri_tiles;
  c->sb.n_tri_tiles = (int)c->tri_tiles.size();
  // rows + quadrant twiddle table in LDS when the device allows that much
  // dynamic LDS per work-group and the table costs no resident work-group per
  // CU (nx = 8192: 96 KB with the table, one work-group per CU); otherwise
  // rows + the two-level table (nx = 8192: 67 KB, two work-groups per CU),
  // whose twiddles are products of two quadrant-table values
  c->sb.fft_tw_lds = (lds_pow2_tw <= (unsigned)c->max_lds &&
                      fft_one_tile_blocks_per_cu(true, lds_pow2_tw) >= fft_one_tile_blocks_per_cu(false, lds_pow2_t2))
                         ? 1 : 0;
  c->sb.fft_lds_pow2 = c->sb.fft_tw_lds ? lds_pow2_tw : lds_pow2_t2;
  c->sb.n_fft_dft = n_fft_dft;
  c->sb.dft_lds = dft_lds;
  c->sb.fft_lds_dft = lds_dft;
  c->sb.dft_groups_fwd = groups_fwd;
  c->sb.dft_groups_inv = groups_inv;
  c->sb.tri_lmax = tri_lmax;
  // the persistent kernels take tiles of <= FFT_PERSIST_ELEMS values and keep
  // twiddles in LDS
  bool persist_ok = fft_persist == 1 && fft_elems <= FFT_PERSIST_ELEMS && fft_lds_persist(FFT_PF) <= (unsigned)c->max_lds;
  for (const auto& d : c->desc) {
    if (!d.pow2) continue;
    const int N = d.nx / 2;
    // the rows of a tile must fit the persistent kernels' prefetch registers
    // (FFT_PF values or their spectrum pairs per lane) and LDS
    if (N * d.fft_rows > FFT_PERSIST_ELEMS || d.fft_rows > FFT_MAX_ROWS) persist_ok = false;
  }
  c->sb.fft_persist = persist_ok ? 1 : 0;
  int max_tile = 0;
  for (const auto& d : c->desc)
    if (d.pow2) max_tile = std::max(max_tile, d.nx / 2 * d.fft_rows);
  c->sb.fft_pf = max_tile <= 4 * FFT_WG ? 4 : FFT_PF;
  c->sb.fft_grid = std::max(1, std::min(n_fft_pow2, (c->sb.fft_pf == 4 ? 3 : 2) * c->n_cu));
  // row-pair kernels: every power-of-two channel of one width nx = 2 N with
  // N = S * FFT_WG_ROWS, S in {2, 4}, two rows per tile (fft_elems = 2 N),
  // rows and twiddles in LDS
  c->sb.fft_pair_s = 0;
  if (wide) {
    c->sb.fft_pair_s = FFT_PAIR_WIDE_S;
    c->sb.fft_tw_lds = 0;
    c->sb.fft_lds_pow2 = wide_lds;
  } else if (fft_persist == 2 && n_fft_pow2 > 0 && c->sb.fft_tw_lds) {
    int n_common = -1;
    bool ok = true;
    for (const auto& d : c->desc) {
      if (!d.pow2) continue;
      const int N = d.nx / 2;
      if (n_common < 0) n_common = N;
      ok = ok && N == n_common;
    }
    const int S = n_common / FFT_WG_ROWS;
    ok = ok && n_common % FFT_WG_ROWS == 0 && (S == 2 || S == 4) && fft_elems == 2 * n_common;
    // two row regions and the quadrant table, also when no tile holds two rows
    const unsigned lds = (unsigned)((2 * n_common + n_common / 2) * sizeof(double2));
    ok = ok && lds <= (unsigned)c->max_lds;
    if (ok) {
      c->sb.fft_pair_s = S;
      c->sb.fft_lds_pow2 = std::max(c->sb.fft_lds_pow2, lds);
    }
  }
  // Wall tiles on the tridiagonal launch when they fit the slots its tiles
  // leave free (256-lane work-groups, as many per CU as its registers allow,
  // three on gfx950): the launch then keeps its number of rounds.
  // EKPNP_WALLS_IN_TRI=0 in the environment keeps them on a launch of their
  // own.
  {
    const char* env = std::getenv("EKPNP_WALLS_IN_TRI");
    const int per_cu = tridiag_walls_blocks_per_cu();
    const long long slots = (long long)(per_cu > 0 ? per_cu : 3) * c->n_cu;
    const long long nt = (long long)c->tri_tiles.size(), nw = (c->n_lbm_wall + 7) & ~7;
    c->walls_in_tri = !(env && env[0] == '0') && nw > 0 && (nt + nw + slots - 1) / slots == (nt + slots - 1) / slots;
  }
  c->lbm_fuse = !c->lbm_fwd.empty() && (n_fft_pow2 == 0 || c->sb.fft_persist == 1);
  if (c->lbm_fuse) c->walls_in_tri = false;
  c->fft_elems = fft_elems;
  c->tri_rows = tri_rows;
  c->fft_persist = c->sb.fft_pair_s > 0 ? 2 : c->sb.fft_persist;
  drop_graphs(c);
  return hipSuccess;
}

// Poisson stages for all channels, or for one channel's tile ranges.
hipError_t enqueue_poisson(ekpnp_ctx* c, int only_channel) {
  StepBuffers b = c->sb;
  if (only_channel >= 0) {
    const ChannelTiles& t = c->ctiles[only_channel];
    b.fft_tiles = c->d_fft_tiles + t.fft_first;
    b.n_fft_tiles = t.fft_count;
    b.n_fft_pow2 = x_family(c->desc[only_channel]) == 0 ? t.fft_count : 0;
    b.n_fft_dft = x_family(c->desc[only_channel]) == 1 ? t.fft_count : 0;
    b.tri_tiles = c->d_tri_tiles + t.tri_first;
    b.n_tri_tiles = t.tri_count;
  }
  hipError_t e = launch_poisson_fwd(b, c->stream);
  if (e != hipSuccess) return e;
  e = launch_poisson_tri(b, c->stream);
  if (e != hipSuccess) return e;
  return launch_poisson_inv(b, c->stream);
}

hipError_t enqueue_lbm(ekpnp_ctx* c, bool macro, bool walls = true) {
  hipError_t e = launch_lbm(c->opt.precision, c->opt.compute_fp64 != 0, c->state_q, macro, c->sb,
                            c->lat[c->cur],
                            c->lat[c->cur ^ 1], c->stream, walls);
  c->cur ^= 1;
  c->state_q = false;
  return e;
}

// whether the next step's wall tiles go on its tridiagonal launch: row-kernel
// steps only (FP32 storage, FP64 arithmetic, populations not in the
// pre-collision form of a restart)
bool defer_walls(const ekpnp_ctx* c) {
  return c->walls_in_tri && !c->state_q && c->opt.precision == 0 && c->opt.compute_fp64 != 0;
}

// one coupled step: collide-stream, then the Poisson stages; ev (optional)
// receives an event after each of the four stages
hipError_t enqueue_step(ekpnp_ctx* c, bool macro, hipEvent_t* ev = nullptr) {
  const bool fuse = c->lbm_fuse && !c->state_q;
  const bool defer = !fuse && defer_walls(c);
  const void* src = c->lat[c->cur];
  void* dst = c->lat[c->cur ^ 1];
  hipError_t e;
  if (fuse) {
    e = launch_lbm_fwd(c->opt.precision, macro, false, c->sb, src, dst, c->stream);
    c->cur ^= 1;
  } else {
    e = enqueue_lbm(c, macro, !defer);
  }
  if (e == hipSuccess && ev) e = hipEventRecord(ev[0], c->stream);
  if (e == hipSuccess && !fuse) e = launch_poisson_fwd(c->sb, c->stream);
  if (e == hipSuccess && ev) e = hipEventRecord(ev[1], c->stream);
  if (e == hipSuccess)
    e = defer ? launch_poisson_tri_walls(macro, c->sb, src, dst, c->stream) : launch_poisson_tri(c->sb, c->stream);
  if (e == hipSuccess && ev) e = hipEventRecord(ev[2], c->stream);
  if (e == hipSuccess) e = launch_poisson_inv(c->sb, c->stream);
  if (e == hipSuccess && ev) e = hipEventRecord(ev[3], c->stream);
  return e;
}

// n steps.  With lbm_inv a step's inverse x-transforms are the next one's
// first work (psi goes to memory after the last step only): the
// spectrum alternates between two buffers, because a work-group transforms the
// rows beside its own too, whose owners may already be writing the new ones.
hipError_t enqueue_steps(ekpnp_ctx* c, int n, bool macro_last) {
  if (c->lbm_fuse && c->lbm_inv && !c->state_q && n > 1) {
    StepBuffers b = c->sb;
    for (int i = 0; i < n; ++i) {
      hipError_t e = launch_lbm_fwd(c->opt.precision, macro_last && i == n - 1, i > 0, b, c->lat[c->cur],
                                    c->lat[c->cur ^ 1], c->stream);
      c->cur ^= 1;
      if (e == hipSuccess) e = launch_poisson_tri(b, c->stream);
      if (e == hipSuccess && i == n - 1) e = launch_poisson_inv(b, c->stream);
      if (e != hipSuccess) return e;
      b.spec_prev = b.spec;
      b.spec = b.spec == c->d_spec ? c->d_spec2 : c->d_spec;
    }
    return hipSuccess;
  }
  for (int i = 0; i < n; ++i) {
    hipError_t e = enqueue_step(c, macro_last && i == n - 1);
    if (e != hipSuccess) return e;
  }
  return hipSuccess;
}

// n steps from the P' state through a cached hipGraph
int graph_steps(ekpnp_ctx* c, int n, bool macro_last) {
  auto key = std::make_tuple(n, c->cur, macro_last ? 1 : 0, 0);
  auto it = c->graphs.find(key);
  if (it == c->graphs.end()) {
    const int cur0 = c->cur;
    HIP_OR_FAIL(c, hipStreamBeginCapture(c->stream, hipStreamCaptureModeThreadLocal));
    hipError_t e = enqueue_steps(c, n, macro_last);
    hipGraph_t g = nullptr;
    hipError_t e2 = hipStreamEndCapture(c->stream, &g);
    c->cur = cur0;
    if (e != hipSuccess) return fail(c, EKPNP_ERR_HIP, std::string("capture: ") + hipGetErrorString(e));
    if (e2 != hipSuccess) return fail(c, EKPNP_ERR_HIP, std::string("end capture: ") + hipGetErrorString(e2));
    hipGraphExec_t ex = nullptr;
    hipError_t e3 = hipGraphInstantiate(&ex, g, nullptr, nullptr, 0);
    (void)hipGraphDestroy(g);
    if (e3 != hipSuccess) return fail(c, EKPNP_ERR_HIP, std::string("instantiate: ") + hipGetErrorString(e3));
    it = c->graphs.emplace(key, ex).first;
  }
  HIP_OR_FAIL(c, hipGraphLaunch(it->second, c->stream));
  c->cur ^= (n & 1);
  return EKPNP_OK;
}

int check_channel(ekpnp_ctx* c, int ch) {
  if (!c) return EKPNP_ERR_INVALID;
  if (ch < 0 || ch >= c->nchan) return fail(c, EKPNP_ERR_INVALID, "channel index out of range");
  return EKPNP_OK;
}

// push the host copy of the channel descriptors (active/swap flags) to the device
hipError_t sync_desc(ekpnp_ctx* c) {
  hipError_t e = hipMemcpyAsync(c->d_desc, c->desc.data(), c->nchan * sizeof(ChanDesc), hipMemcpyHostToDevice,
                                c->stream);
  if (e != hipSuccess) return e;
  return hipStreamSynchronize(c->stream);
}

// lattice index holding channel ch's current state
int chan_lattice(const ekpnp_ctx* c, int ch) { return c->cur ^ c->desc[ch].swap; }

// [9][ny][nx]: w_d (X(x, y) + c_dx J(y) / (cs^2 CFL)) of one species
std::vector<double> ref_offsets(ekpnp_ctx* c, int channel, int species, hipError_t* err) {
  const ChanDesc& d = c->desc[channel];
  const size_t nn = (size_t)d.nx * d.ny;
  std::vector<double> rec(kRefStride * (size_t)d.ny), out(9 * nn);
  std::vector<float> kn(BLK_STRIDE * (size_t)d.nb * d.ny);
  *err = hipMemcpy(rec.data(), c->d_refs + d.ref_off, rec.size() * sizeof(double), hipMemcpyDeviceToHost);
  if (*err == hipSuccess)
    *err = hipMemcpy(kn.data(), c->d_blocks + d.blk_off, kn.size() * sizeof(float), hipMemcpyDeviceToHost);
  const double tc = d.inv_cs2 * d.inv_cfl;
  for (int y = 0; y < d.ny; ++y) {
    const double J = rec[kRefStride * (size_t)y + 3 + species];
    const float* Br = &kn[BLK_STRIDE * (size_t)d.nb * y];
    for (int x = 0; x < d.nx; ++x) {
      const double X = Br[BLK_STRIDE * (x / REF_BLOCK) + species];  // the block's reference
      for (int dd = 0; dd < 9; ++dd) out[dd * nn + (size_t)y * d.nx + x] = W[dd] * (X + CXH[dd] * tc * J);
    }
  }
  return out;
}

// Have the whole pages of a destination that is about to be overwritten mapped
// in one call: memory fresh from the allocator costs a fault per 4 KB page
// otherwise (256 MB in 1 MB fields: 55 ms with the copy, 28 ms this way, 4 ms
// once mapped).  Nothing is lost where the kernel does not know the request.
void map_pages(char* p, size_t bytes) {
#ifdef MADV_POPULATE_WRITE
  const uintptr_t a = ((uintptr_t)p + 4095) & ~(uintptr_t)4095, e = ((uintptr_t)p + bytes) & ~(uintptr_t)4095;
  if (e > a) {
    const int err = errno;
    (void)madvise(reinterpret_cast<void*>(a), e - a, MADV_POPULATE_WRITE);
    errno = err;
  }
#else
  (void)p;
  (void)bytes;
#endif
}

// A condition that another thread makes true with set()
struct Gate {
  std::mutex m;
  std::condition_variable cv;
  template <typename F>
  void set(F change) {
    {
      std::lock_guard<std::mutex> lock(m);
      change();
    }
    cv.notify_all();
  }
  // spins for spin_us, then sleeps
  template <typename F>
  void wait(int spin_us, F ready) {
    const auto until = std::chrono::steady_clock::now() + std::chrono::microseconds(spin_us);
    do {
      if (ready()) return;
    } while (std::chrono::steady_clock::now() < until);
    std::unique_lock<std::mutex> lock(m);
    cv.wait(lock, ready);
  }
};

// dst = bytes of device memory at src, once the stream's earlier work is done.
// The runtime's copy to pageable memory moves a field at 10 GB/s (13 ms for the
// 134 MB of 8192 x 2048): it copies and first touches the caller's pages on one
// thread.  Here pieces go to pinned memory by DMA, the next ones under way
// while STAGE_THREADS threads copy a piece on (3.5 ms); a small field takes
// one pinned copy (64 KB: 37 -> 11 us).
// Memory that the runtime knows (pinned, managed) needs no staging: it is copied
// to directly (67 MB: 1.2 ms of CPU time instead of 5.7).  Asking takes half a
// microsecond, as much as copying 8 KB on, so small fields are staged unasked.
hipError_t copy_to_host(ekpnp_ctx* c, void* dst, const void* src, size_t bytes) {
  const auto direct = [&] {
    const hipError_t e = hipStreamSynchronize(c->stream);
    return e == hipSuccess ? hipMemcpy(dst, src, bytes, hipMemcpyDeviceToHost) : e;
  };
  if (bytes >= STAGE_ASK_MIN) {
    hipPointerAttribute_t attr{};
    if (hipPointerGetAttributes(&attr, dst) != hipSuccess) (void)hipGetLastError();  // unknown: pageable
    else if (attr.type != hipMemoryTypeUnregistered) return direct();
  }
  const bool parallel = bytes >= STAGE_PARALLEL_MIN;
  const size_t chunk = parallel ? std::min(STAGE_CHUNK, (bytes / 4 + 4095) & ~(size_t)4095) : bytes;
  const size_t pieces = (bytes + chunk - 1) / chunk, slots = std::min<size_t>(STAGE_SLOTS, pieces);
  if (c->stage_bytes < slots * chunk) {
    if (c->stage) (void)hipHostFree(c->stage);
    c->stage = nullptr;
    c->stage_bytes = 0;
    void* p = nullptr;
    if (hipHostMalloc(&p, slots * chunk, hipHostMallocDefault) == hipSuccess) {
      c->stage = static_cast<char*>(p);
      c->stage_bytes = slots * chunk;
    } else {
      (void)hipGetLastError();
    }
  }
  for (size_t i = 0; i <= STAGE_SLOTS && pieces > 1 && c->stage; ++i)
    if (!c->stage_ev[i] && hipEventCreateWithFlags(&c->stage_ev[i], hipEventDisableTiming) != hipSuccess) {
      (void)hipGetLastError();
      c->stage_ev[i] = nullptr;
      (void)hipHostFree(c->stage);
      c->stage = nullptr;
      c->stage_bytes = 0;
    }
  if (!c->stage) return direct();  // no pinned memory for the staging
  if (pieces == 1) {
    hipError_t e = hipMemcpyAsync(c->stage, src, bytes, hipMemcpyDeviceToHost, c->stream);
    map_pages(static_cast<char*>(dst), bytes);
    const hipError_t e2 = hipStreamSynchronize(c->stream);
    if (e == hipSuccess) e = e2;
    if (e == hipSuccess) std::memcpy(dst, c->stage, bytes);
    return e;
  }
  char* out = static_cast<char*>(dst);
  auto size_of = [&](size_t i) { return std::min(chunk, bytes - i * chunk); };
  auto issue = [&](size_t i) {
    hipError_t e = hipMemcpyAsync(c->stage + (i % slots) * chunk, static_cast<const char*>(src) + i * chunk, size_of(i),
                                  hipMemcpyDeviceToHost, c->stream);
    return e == hipSuccess ? hipEventRecord(c->stage_ev[i % slots], c->stream) : e;
  };
  // The helpers sleep while the stream works off what is in front of the copy,
  // wake when that is done, with the first piece's DMA under way, and copy their
  // share of each piece the main thread announces in `ready`.
  std::atomic<size_t> ready{0};
  std::atomic<int> left{0};
  std::atomic<bool> stop{false};
  const hipEvent_t begin = c->stage_ev[STAGE_SLOTS];
  const bool idle = hipStreamQuery(c->stream) == hipSuccess;
  if (!idle) (void)hipGetLastError();
  std::atomic<bool> begun{idle};
  Gate wake, announced, copied;
  const int threads = STAGE_THREADS;
  auto share = [&](int t, size_t i, bool map_only) {
    const size_t n = size_of(i), part = (n / threads + 4095) & ~(size_t)4095, a = std::min(n, part * t);
    if (map_only) map_pages(out + i * chunk + a, std::min(part, n - a));
    else std::memcpy(out + i * chunk + a, c->stage + (i % slots) * chunk + a, std::min(part, n - a));
  };
  std::vector<std::thread> helpers;
  try {
    for (int t = 1; t < STAGE_THREADS; ++t)
      helpers.emplace_back([&, t] {
        for (size_t i = 0; i < pieces; ++i) {
          share(t, i, true);
          if (i == 0) wake.wait(0, [&] { return begun.load() || stop.load(); });
          announced.wait(STAGE_SPIN_US, [&] { return ready.load() > i || stop.load(); });
          if (ready.load() <= i) return;
          share(t, i, false);
          if (left.fetch_sub(1) == 1) copied.set([] {});
        }
      });
  } catch (const std::exception&) {
    // fewer threads than asked for: the caller's thread takes their shares
  }
  const int helping = (int)helpers.size();
  hipError_t e = idle ? hipSuccess : hipEventRecord(begin, c->stream);
  for (size_t i = 0; i < slots && e == hipSuccess; ++i) e = issue(i);
  for (size_t i = 0; i < pieces && e == hipSuccess; ++i) {
    share(0, i, true);
    if (i == 0 && !idle) {
      e = hipEventSynchronize(begin);
      wake.set([&] { begun.store(true); });
      if (e != hipSuccess) break;
    }
    e = hipEventSynchronize(c->stage_ev[i % slots]);
    if (e != hipSuccess) break;
    left.store(helping);
    announced.set([&] { ready.store(i + 1); });
    for (int t = 0; t < threads; t = t == 0 ? helping + 1 : t + 1) share(t, i, false);
    copied.wait(STAGE_SPIN_US, [&] { return left.load() == 0; });
    if (i + slots < pieces) e = issue(i + slots);
  }
  wake.set([&] { stop.store(true); });
  announced.set([] {});
  for (auto& t : helpers) t.join();
  if (e != hipSuccess) (void)hipStreamSynchronize(c->stream);  // no copy into the staging buffer stays in flight
  return e;
}

// psi wall rows of one channel from the wall planes
hipError_t upload_psi_walls(ekpnp_ctx* c, int ch) {
  const ChanDesc& d = c->desc[ch];
  const double* lo = &c->walls[W_PSI_LO * (size_t)c->total_nx + d.wall_off];
  const double* hi = &c->walls[W_PSI_HI * (size_t)c->total_nx + d.wall_off];
  hipError_t e = hipMemcpyAsync(c->d_psi + d.fld_off, lo, d.nx * sizeof(double),
                                hipMemcpyHostToDevice, c->stream);
  if (e != hipSuccess) return e;
  e = hipMemcpyAsync(c->d_psi + d.fld_off + (long long)(d.ny - 1) * d.nx, hi, d.nx * sizeof(double),
                     hipMemcpyHostToDevice, c->stream);
  if (e != hipSuccess) return e;
  return hipStreamSynchronize(c->stream);
}

// Step count at which FP32 storage next re-centres its references: 8, 16,
// ..., EKPNP_REBASE_INTERVAL steps after init_equilibrium (the fields change
// fastest while a cold start's double layer and flow form, and the
// references must follow them to keep the stored deviations small), then
// every EKPNP_REBASE_INTERVAL steps.  A function of the step counts only, so
// a run re-centres at the same steps however it is cut into calls.
long long next_rebase(const ekpnp_ctx* c) {
  const long long last = c->rebase_step - c->origin_step;
  const long long next = last < EKPNP_REBASE_INTERVAL ? std::max<long long>(8, 2 * last)
                                                      : last + EKPNP_REBASE_INTERVAL;
  return c->origin_step + next;
}

}  // namespace

extern "C" {

void ekpnp_reference_params(ekpnp_channel_params* p) {
  if (!p) return;
  std::memset(p, 0, sizeof(*p));
  p->nx = 10;              // LBM.h:35
  p->ny = 101;             // LBM.h:36
  p->flags = EKPNP_FLAG_G0_FLUID_U;  // LBM.cu:493 as shipped
  p->dx = 1.0e-6 / 100.0;  // LBM.h:42
  p->dy = 1.0e-6 / 100.0;  // LBM.h:43
  p->cfl = 0.01;           // LBM.h:50
  p->dt = 0.01 * 1.0e-6 / 100.0;            // LBM.h:51
  p->cs2 = 1.0 / 3.0 / (0.01 * 0.01);       // LBM.h:52
  p->rho0 = 1000.0;        // LBM.h:53
  p->nu = 0.889e-6;        // LBM.h:65
  p->diff_pos = 1.0e-8;    // LBM.h:64
  p->diff_neg = 1.0e-8;    // LBM.h:71
  p->mob_pos = 4.245e-7;   // LBM.h:67
  p->mob_neg = -4.245e-7;  // LBM.h:74
  p->magic_f = 1.0e-6;     // LBM.h:110-112
  p->magic_pos = 1.0e-6;
  p->magic_neg = 1.0e-6;
  p->psi_lo = -5.2574e-3;  // LBM.h:58
  p->psi_hi = -5.2574e-3;  // LBM.h:60
  p->cpos_lo = 1.2364549e-2;  // LBM.h:55-56
  p->cpos_hi = 1.2364549e-2;
  p->cneg_lo = 8.087639e-3;   // LBM.h:81-83
  p->cneg_hi = 8.087639e-3;
  p->c_bulk = 0.01;           // chargeinf, LBM.h:54
  p->poisson_coef = 9.64e4 / 6.95e-10;  // convertCtoCharge/eps, LBM.h:63, 90
  p->force_coef = 0.0;        // LBM.cu:388-389 as shipped
  p->e_applied = 1.0e3;       // LBM.h:62
  p->exf = 0.0;
  p->uw = 0.0;
  p->lx = 1.0e-7;             // LBM.h:40
  p->init_noise = 0.0;
  p->inv_thermal_voltage = 1.6e-19 / 1.38e-23 / 273.0;  // electron/kB/roomT, LBM.h:87-89
  p->pb_omega = 0.05;         // LBM.h:91
  p->pb_iterations = 501.0;   // LBM.cu:116
}

int ekpnp_lattice_params(ekpnp_channel_params* p, int nx, int ny, double tau, double zeta,
                         double kappa_h, double e_x, double diff) {
  if (!p || nx < 2 || ny < 4 || !(tau > 0.5) || !(diff > 0)) return EKPNP_ERR_INVALID;
  std::memset(p, 0, sizeof(*p));
  p->nx = nx;
  p->ny = ny;
  p->flags = 0;
  p->dx = p->dy = p->dt = p->cfl = 1.0;
  p->cs2 = 1.0 / 3.0;
  p->rho0 = 1.0;
  p->nu = (tau - 0.5) / 3.0;
  p->diff_pos = p->diff_neg = diff;
  p->mob_pos = diff;
  p->mob_neg = -diff;
  p->magic_f = p->magic_pos = p->magic_neg = 0.25;
  p->psi_lo = p->psi_hi = zeta;
  p->cpos_lo = p->cpos_hi = std::exp(-zeta);
  p->cneg_lo = p->cneg_hi = std::exp(zeta);
  p->c_bulk = 1.0;
  const double h = 0.5 * (ny - 1);
  const double kappa = kappa_h / h;
  p->poisson_coef = 0.5 * kappa * kappa;
  p->force_coef = p->poisson_coef;
  p->e_applied = e_x;
  p->exf = 0.0;
  p->uw = 0.0;
  p->lx = (double)nx;
  p->init_noise = 1.0e-3;
  p->inv_thermal_voltage = 1.0;
  p->pb_omega = 0.05;
  p->pb_iterations = 501.0;
  return EKPNP_OK;
}

void ekpnp_default_options(ekpnp_options* o) {
  if (!o) return;
  o->precision = EKPNP_POP_FP32;
  o->device = 0;
  o->use_graph = 1;
  o->compute_fp64 = 1;
  o->reject_unresolved = 0;
}

int ekpnp_check_params(const ekpnp_channel_params* channels, int n_channels, uint32_t* flags_out) {
  if (!channels || n_channels <= 0) return EKPNP_ERR_INVALID;
  int flagged = 0;
  for (int i = 0; i < n_channels; ++i) {
    double kdy = 0.0, drift = 0.0, flow = 0.0;
    const uint32_t f = check_flags(channels[i], &kdy, &drift, &flow);
    if (flags_out) flags_out[i] = f;
    flagged += f != 0;
  }
  return flagged;
}

const char* ekpnp_create_error(void) { return g_create_error.c_str(); }

const char* ekpnp_last_error(const ekpnp_ctx* ctx) { return ctx ? ctx->err.c_str() : "null context"; }

int ekpnp_create(const ekpnp_channel_params* channels, int n_channels, const ekpnp_options* opt,
                 ekpnp_ctx** out) {
  const ApiRange range_("ekpnp_create");
  g_create_error.clear();
  if (!out) return EKPNP_ERR_INVALID;
  *out = nullptr;
  if (!channels || n_channels <= 0) {
    g_create_error = "no channels";
    return EKPNP_ERR_INVALID;
  }
  ekpnp_options o;
  ekpnp_default_options(&o);
  if (opt) o = *opt;
  if (o.precision != EKPNP_POP_FP32 && o.precision != EKPNP_POP_FP64) {
    g_create_error = "unknown precision";
    return EKPNP_ERR_INVALID;
  }
  for (int i = 0; i < n_channels; ++i) {
    std::string m = validate(channels[i], i);
    if (!m.empty()) {
      g_create_error = m;
      return (m.find("above") != std::string::npos) ? EKPNP_ERR_UNSUPPORTED : EKPNP_ERR_INVALID;
    }
    double kdy = 0.0, drift = 0.0, flow = 0.0;
    const uint32_t f = check_flags(channels[i], &kdy, &drift, &flow);
    if (o.reject_unresolved && f) {
      std::string why;
      if (f & EKPNP_CHECK_DEBYE_UNRESOLVED) why += "Debye length unresolved";
      if (f & EKPNP_CHECK_WALL_DRIFT) why += std::string(why.empty() ? "" : ", ") + "wall drift too fast";
      if (f & EKPNP_CHECK_FLOW_FAST) why += std::string(why.empty() ? "" : ", ") + "electro-osmotic flow too fast";
      char buf[320];
      snprintf(buf, sizeof buf,
               "channel %d: %s (kappa dy = %.3g, limit 0.4; wall drift = %.3g, limit 0.05; flow = %.3g, limit 0.1)", i,
               why.c_str(), kdy, drift, flow);
      g_create_error = buf;
      return EKPNP_ERR_UNSTABLE;
    }
  }
  hipError_t he = hipSetDevice(o.device);
  if (he != hipSuccess) {
    g_create_error = std::string("hipSetDevice: ") + hipGetErrorString(he);
    return EKPNP_ERR_HIP;
  }
  // the device's copy of the allocation-free reductions' scratch array
  he = noalloc_scratch_init(o.device);
  if (he != hipSuccess) {
    g_create_error = std::string("scratch address: ") + hipGetErrorString(he);
    return EKPNP_ERR_HIP;
  }
  ekpnp_ctx* c = new ekpnp_ctx();
  c->opt = o;
  c->nchan = n_channels;
  c->elem = (o.precision == EKPNP_POP_FP32) ? 4 : 8;
  // the device's sizes, before anything is planned by them
  int max_lds = 65536;
  if (hipDeviceGetAttribute(&max_lds, hipDeviceAttributeMaxSharedMemoryPerBlock, o.device) != hipSuccess)
    max_lds = 65536;
  c->max_lds = max_lds;
  int n_cu = 256;
  if (hipDeviceGetAttribute(&n_cu, hipDeviceAttributeMultiprocessorCount, o.device) == hipSuccess && n_cu > 0)
    c->n_cu = n_cu;
  c->params.assign(channels, channels + n_channels);
  c->desc.resize(n_channels);
  c->ctiles.resize(n_channels);

  // layout
  long long pop = 0, fld = 0, spec = 0, refs = 0, cprime = 0, blocks = 0;
  int wall = 0;
  // every per-channel block starts on a 64-element boundary
  auto pad64 = [](long long v) { return (v + 63) / 64 * 64; };
  for (int i = 0; i < n_channels; ++i) {
    ChanDesc d = make_desc(channels[i], o.precision);
    const long long nn = (long long)d.nx * d.ny;
    d.plane = pad64(nn);
    d.pop_off = pop;
    d.fld_off = fld;
    d.spec_off = spec;
    d.ref_off = refs;
    d.blk_off = blocks;
    d.cp_off = cprime;
    d.wall_off = wall;
    d.tw_off = wall;
    pop += 27 * d.plane;
    fld += pad64(nn);
    spec += pad64((long long)d.ny * d.nk_stride);
    refs += pad64((long long)kRefStride * d.ny);
    blocks += pad64((long long)BLK_STRIDE * d.nb * d.ny);
    cprime += pad64((long long)kMaxTriChunks * d.nk);
    wall += (int)pad64(d.nx);
    c->desc[i] = d;
  }
  build_lbm_fwd(c);
  c->total_pops = pop;
  c->total_nodes = fld;
  c->total_spec = spec;
  c->total_refs = refs;
  c->total_blocks = blocks;
  c->total_cprime = cprime;
  c->total_nx = wall;
  // rows of narrow channels first (k_row_means_narrow)
  for (const bool narrow : {true, false}) {
    for (int i = 0; i < n_channels; ++i) {
      if ((c->desc[i].nx <= ROW_WAVE_NX) != narrow) continue;
      c->ctiles[i].row_first = (int)c->row_tiles.size();
      for (int y = 0; y < c->desc[i].ny; ++y) c->row_tiles.push_back(make_int2(i, y));
    }
    if (narrow) c->n_row_narrow = (int)c->row_tiles.size();
  }

  // LBM tiles, channel-major
  c->first_tile.resize(n_channels + 1);
  for (int i = 0; i < n_channels; ++i) {
    c->first_tile[i] = (int)c->lbm_tiles.size();
    const long long nn = (long long)c->desc[i].nx * c->desc[i].ny;
    for (long long s = 0; s < nn; s += LBM_WG) c->lbm_tiles.push_back(make_int2(i, (int)s));
  }
  c->first_tile[n_channels] = (int)c->lbm_tiles.size();
  // the step's split for every interior tile shape (the device table holds
  // the largest), the default shape last
  for (int w : {2, 4, 0}) {
    build_lbm_split(c, w);
    c->lbm_split_cap = std::max(c->lbm_split_cap, c->lbm_split.size());
  }
  // Poisson tile tables: capacity for the finest decomposition (one row per
  // FFT tile, two modes per tridiagonal work-group)
  for (int i = 0; i < n_channels; ++i) {
    c->fft_tiles_cap += (size_t)(c->desc[i].ny - 2);
    c->tri_tiles_cap += (size_t)((c->desc[i].nk + 1) / 2);
  }

  // wall planes and twiddles
  c->walls.assign(6 * (size_t)wall, 0.0);
  std::vector<double2> tw((size_t)wall);
  for (int i = 0; i < n_channels; ++i) {
    const ekpnp_channel_params& p = channels[i];
    const ChanDesc& d = c->desc[i];
    for (int x = 0; x < d.nx; ++x) {
      c->walls[W_PSI_LO * (size_t)wall + d.wall_off + x] = p.psi_lo;
      c->walls[W_PSI_HI * (size_t)wall + d.wall_off + x] = p.psi_hi;
      c->walls[W_CP_LO * (size_t)wall + d.wall_off + x] = p.cpos_lo;
      c->walls[W_CP_HI * (size_t)wall + d.wall_off + x] = p.cpos_hi;
      c->walls[W_CN_LO * (size_t)wall + d.wall_off + x] = p.cneg_lo;
      c->walls[W_CN_HI * (size_t)wall + d.wall_off + x] = p.cneg_hi;
      const double a = 2.0 * M_PI * (double)x / (double)d.nx;
      tw[d.tw_off + x] = make_double2(std::cos(a), -std::sin(a));
    }
  }

  // device allocations
  auto alloc_all = [&]() -> hipError_t {
    hipError_t e;
    const size_t npop = (size_t)c->total_pops;
    for (int k = 0; k < 2; ++k) {
      e = hipMalloc(&c->lat[k], std::max<size_t>(npop * c->elem, 16));
      if (e != hipSuccess) return e;
      c->dev_bytes += npop * c->elem;
    }
    if ((e = dalloc(c, &c->d_desc, n_channels)) != hipSuccess) return e;
    if ((e = dalloc(c, &c->d_lbm_tiles, c->lbm_tiles.size())) != hipSuccess) return e;
    if ((e = dalloc(c, &c->d_lbm_split, c->lbm_split_cap)) != hipSuccess) return e;
    if ((e = dalloc(c, &c->d_lbm_fwd, c->lbm_fwd.size())) != hipSuccess) return e;
    if ((e = dalloc(c, &c->d_fft_tiles, c->fft_tiles_cap)) != hipSuccess) return e;
    if ((e = dalloc(c, &c->d_tri_tiles, c->tri_tiles_cap)) != hipSuccess) return e;
    if ((e = dalloc(c, &c->d_first_tile, c->first_tile.size())) != hipSuccess) return e;
    if ((e = dalloc(c, &c->d_rho_e, c->total_nodes)) != hipSuccess) return e;
    if ((e = dalloc(c, &c->d_psi, c->total_nodes)) != hipSuccess) return e;
    if ((e = dalloc(c, &c->d_macro, M_COUNT * (size_t)c->total_nodes)) != hipSuccess) return e;
    if ((e = dalloc(c, &c->d_walls, c->walls.size())) != hipSuccess) return e;
    if ((e = dalloc(c, &c->d_tw, tw.size())) != hipSuccess) return e;
    if ((e = dalloc(c, &c->d_spec, c->total_spec)) != hipSuccess) return e;
    if (c->lbm_inv && (e = dalloc(c, &c->d_spec2, c->total_spec)) != hipSuccess) return e;
    if ((e = dalloc(c, &c->d_ux_prev, c->total_nodes)) != hipSuccess) return e;
    if ((e = dalloc(c, &c->d_refs, c->total_refs)) != hipSuccess) return e;
    if ((e = dalloc(c, &c->d_refs_new, c->total_refs)) != hipSuccess) return e;
    if ((e = dalloc(c, &c->d_blocks, c->total_blocks)) != hipSuccess) return e;
    if ((e = dalloc(c, &c->d_blocks_new, c->total_blocks)) != hipSuccess) return e;
    if ((e = dalloc(c, &c->d_row_tiles, c->row_tiles.size())) != hipSuccess) return e;
    if ((e = dalloc(c, &c->d_partials, 8 * c->lbm_tiles.size())) != hipSuccess) return e;
    if ((e = dalloc(c, &c->d_red, 8 * (size_t)n_channels)) != hipSuccess) return e;
    if ((e = dalloc(c, &c->d_diag, 2 * (size_t)DIAG_MAX_WG + 2)) != hipSuccess) return e;
    if ((e = dalloc(c, &c->d_cprime, c->total_cprime)) != hipSuccess) return e;
    if ((e = hipStreamCreateWithFlags(&c->stream, hipStreamNonBlocking)) != hipSuccess) return e;
    return hipSuccess;
  };
  he = alloc_all();
  if (he != hipSuccess) {
    g_create_error = std::string("allocation: ") + hipGetErrorString(he);
    release(c);
    delete c;
    return (he == hipErrorOutOfMemory) ? EKPNP_ERR_NOMEM : EKPNP_ERR_HIP;
  }
  auto upload = [&]() -> hipError_t {
    hipError_t e;
    if ((e = hipMemcpy(c->d_desc, c->desc.data(), n_channels * sizeof(ChanDesc), hipMemcpyHostToDevice)) != hipSuccess) return e;
    if ((e = hipMemcpy(c->d_lbm_tiles, c->lbm_tiles.data(), c->lbm_tiles.size() * sizeof(int2), hipMemcpyHostToDevice)) != hipSuccess) return e;
    if ((e = hipMemcpy(c->d_lbm_split, c->lbm_split.data(), c->lbm_split.size() * sizeof(int2), hipMemcpyHostToDevice)) != hipSuccess) return e;
    if (!c->lbm_fwd.empty() &&
        (e = hipMemcpy(c->d_lbm_fwd, c->lbm_fwd.data(), c->lbm_fwd.size() * sizeof(int2), hipMemcpyHostToDevice)) != hipSuccess)
      return e;
    if ((e = hipMemcpy(c->d_first_tile, c->first_tile.data(), c->first_tile.size() * sizeof(int), hipMemcpyHostToDevice)) != hipSuccess) return e;
    if ((e = hipMemcpy(c->d_walls, c->walls.data(), c->walls.size() * sizeof(double), hipMemcpyHostToDevice)) != hipSuccess) return e;
    if ((e = hipMemcpy(c->d_tw, tw.data(), tw.size() * sizeof(double2), hipMemcpyHostToDevice)) != hipSuccess) return e;
    if ((e = hipMemcpy(c->d_row_tiles, c->row_tiles.data(), c->row_tiles.size() * sizeof(int2), hipMemcpyHostToDevice)) != hipSuccess) return e;
    if ((e = hipMemset(c->d_refs, 0, c->total_refs * sizeof(double))) != hipSuccess) return e;
    if ((e = hipMemset(c->d_refs_new, 0, c->total_refs * sizeof(double))) != hipSuccess) return e;
    if ((e = hipMemset(c->d_blocks, 0, c->total_blocks * sizeof(float))) != hipSuccess) return e;
    if ((e = hipMemset(c->d_blocks_new, 0, c->total_blocks * sizeof(float))) != hipSuccess) return e;
    const size_t npop = (size_t)c->total_pops;
    if ((e = hipMemset(c->lat[0], 0, npop * c->elem)) != hipSuccess) return e;
    if ((e = hipMemset(c->lat[1], 0, npop * c->elem)) != hipSuccess) return e;
    if ((e = hipMemset(c->d_rho_e, 0, c->total_nodes * sizeof(double))) != hipSuccess) return e;
    if ((e = hipMemset(c->d_psi, 0, c->total_nodes * sizeof(double))) != hipSuccess) return e;
    if ((e = hipMemset(c->d_macro, 0, M_COUNT * c->total_nodes * sizeof(double))) != hipSuccess) return e;
    if ((e = hipMemset(c->d_ux_prev, 0, c->total_nodes * sizeof(double))) != hipSuccess) return e;
    if ((e = hipMemset(c->d_spec, 0, c->total_spec * sizeof(double2))) != hipSuccess) return e;
    if (c->d_spec2 && (e = hipMemset(c->d_spec2, 0, c->total_spec * sizeof(double2))) != hipSuccess) return e;
    return hipDeviceSynchronize();
  };
  he = upload();
  if (he != hipSuccess) {
    g_create_error = std::string("upload: ") + hipGetErrorString(he);
    release(c);
    delete c;
    return EKPNP_ERR_HIP;
  }
  c->sb = make_buffers(c);
  // default plan (ekpnp_autotune refines it): rows of nx = 4096 and 8192
  // run fastest in the row-pair kernels (two rows per work-group; when the
  // channels' widths differ, the one-tile kernels with as many rows as fit
  // 4096 values), narrower rows in the persistent pipelined kernels with up
  // to 1024 values per tile
  int max_n = 0;
  for (const auto& d : c->desc)
    if (d.pow2) max_n = std::max(max_n, d.nx / 2);
  if (max_n >= 2048) {
    c->fft_elems = 4096;
    c->fft_persist = 2;
  } else {
    c->fft_elems = 1024;
    c->fft_persist = 1;
  }
  he = build_poisson_plan(c, c->fft_elems, c->tri_rows, c->fft_persist);
  if (he != hipSuccess) {
    g_create_error = std::string("Poisson plan: ") + hipGetErrorString(he);
    release(c);
    delete c;
    return EKPNP_ERR_HIP;
  }
  for (int i = 0; i < n_channels; ++i) {
    if (upload_psi_walls(c, i) != hipSuccess) {
      g_create_error = "psi wall upload failed";
      release(c);
      delete c;
      return EKPNP_ERR_HIP;
    }
  }
  *out = c;
  return EKPNP_OK;
}

void ekpnp_destroy(ekpnp_ctx* ctx) {
  const ApiRange range_("ekpnp_destroy");
  if (!ctx) return;
  (void)hipSetDevice(ctx->opt.device);
  if (ctx->stream) (void)hipStreamSynchronize(ctx->stream);
  release(ctx);
  delete ctx;
}

int ekpnp_set_wall_profile(ekpnp_ctx* ctx, int channel, const double* psi_lo, const double* psi_hi,
                           const double* cpos_lo, const double* cpos_hi, const double* cneg_lo,
                           const double* cneg_hi) {
  int rc = check_channel(ctx, channel);
  if (rc) return rc;
  HIP_OR_FAIL(ctx, hipSetDevice(ctx->opt.device));
  const ChanDesc& d = ctx->desc[channel];
  const double* src[6] = {psi_lo, psi_hi, cpos_lo, cpos_hi, cneg_lo, cneg_hi};
  for (int a = 0; a < 6; ++a) {
    if (!src[a]) continue;
    double* dst = &ctx->walls[a * (size_t)ctx->total_nx + d.wall_off];
    std::memcpy(dst, src[a], d.nx * sizeof(double));
    HIP_OR_FAIL(ctx, hipMemcpyAsync(ctx->d_walls + a * (size_t)ctx->total_nx + d.wall_off, dst,
                                    d.nx * sizeof(double), hipMemcpyHostToDevice, ctx->stream));
  }
  // graphs read the wall planes through device pointers: nothing to rebuild
  HIP_OR_FAIL(ctx, upload_psi_walls(ctx, channel));
  return EKPNP_OK;
}

int ekpnp_set_fields(ekpnp_ctx* ctx, int channel, const double* rho, const double* ux,
                     const double* uy, const double* cpos, const double* cneg, const double* psi) {
  const ApiRange range_("ekpnp_set_fields");
  int rc = check_channel(ctx, channel);
  if (rc) return rc;
  if (!rho || !ux || !uy || !cpos || !cneg) return fail(ctx, EKPNP_ERR_INVALID, "null field");
  HIP_OR_FAIL(ctx, hipSetDevice(ctx->opt.device));
  const ChanDesc& d = ctx->desc[channel];
  const size_t nn = (size_t)d.nx * d.ny;
  const double* f[M_COUNT] = {rho, ux, uy, cpos, cneg};
  for (int k = 0; k < M_COUNT; ++k)
    HIP_OR_FAIL(ctx, hipMemcpyAsync(ctx->d_macro + k * ctx->total_nodes + d.fld_off, f[k],
                                    nn * sizeof(double), hipMemcpyHostToDevice, ctx->stream));
  HIP_OR_FAIL(ctx, launch_charge(ctx->sb, channel, (long long)nn, ctx->stream));
  if (psi) {
    HIP_OR_FAIL(ctx, hipMemcpyAsync(ctx->d_psi + d.fld_off, psi, nn * sizeof(double),
                                    hipMemcpyHostToDevice, ctx->stream));
  } else {
    HIP_OR_FAIL(ctx, enqueue_poisson(ctx, channel));
  }
  HIP_OR_FAIL(ctx, hipStreamSynchronize(ctx->stream));
  ctx->has_fields = true;
  return EKPNP_OK;
}

}  // extern "C"

namespace {
// One channel's starting fields: the reference's gpu_initialization
// (LBM.cu:147-160: rho0, u = 0, c+- = 0, psi = the wall potential) for the
// reference and PB-Picard modes, or uniform c_bulk with seeded noise and the
// wall concentrations on the wall rows for the cold start
int initial_fields(ekpnp_ctx* ctx, int ch, int mode, uint64_t seed) {
  const ekpnp_channel_params& p = ctx->params[ch];
  const ChanDesc& d = ctx->desc[ch];
  const size_t nn = (size_t)d.nx * d.ny;
  std::vector<double> rho(nn, p.rho0), zero(nn, 0.0), cp(nn), cn(nn);
  if (mode == EKPNP_INIT_REFERENCE || mode == EKPNP_INIT_PB_PICARD) {
    std::vector<double> psi(nn, p.psi_lo);
    return ekpnp_set_fields(ctx, ch, rho.data(), zero.data(), zero.data(), zero.data(), zero.data(), psi.data());
  }
  const size_t T = ctx->total_nx;
  ekpnp_cold_field(cp.data(), d.nx, d.ny, p.c_bulk, p.init_noise, &ctx->walls[W_CP_LO * T + d.wall_off],
                   &ctx->walls[W_CP_HI * T + d.wall_off], seed, ch, 0);
  ekpnp_cold_field(cn.data(), d.nx, d.ny, p.c_bulk, p.init_noise, &ctx->walls[W_CN_LO * T + d.wall_off],
                   &ctx->walls[W_CN_HI * T + d.wall_off], seed, ch, 1);
  return ekpnp_set_fields(ctx, ch, rho.data(), zero.data(), zero.data(), cp.data(), cn.data(), nullptr);
}
}  // namespace

extern "C" {

int ekpnp_initialization(ekpnp_ctx* ctx, int mode, uint64_t seed) {
  const ApiRange range_("ekpnp_initialization");
  if (!ctx) return EKPNP_ERR_INVALID;
  if (mode != EKPNP_INIT_COLD_NOISE && mode != EKPNP_INIT_REFERENCE && mode != EKPNP_INIT_PB_PICARD)
    return fail(ctx, EKPNP_ERR_INVALID, "unknown initialization mode");
  HIP_OR_FAIL(ctx, hipSetDevice(ctx->opt.device));
  for (int ch = 0; ch < ctx->nchan; ++ch) {
    int rc = initial_fields(ctx, ch, mode, seed);
    if (rc) return rc;
  }
  if (mode == EKPNP_INIT_PB_PICARD) {
    // LBM.cu:106-127: psi_old = psi; iterate {Boltzmann c+-, Poisson, relax};
    // the ux snapshot buffer holds psi_old (the residual snapshot restarts)
    int iters = 0;
    for (const auto& p : ctx->params) iters = std::max(iters, (int)p.pb_iterations);
    HIP_OR_FAIL(ctx, hipMemcpyAsync(ctx->d_ux_prev, ctx->d_psi, ctx->total_nodes * sizeof(double),
                                    hipMemcpyDeviceToDevice, ctx->stream));
    for (int it = 0; it < iters; ++it) {
      HIP_OR_FAIL(ctx, launch_pb_fields(ctx->sb, ctx->stream));
      HIP_OR_FAIL(ctx, enqueue_poisson(ctx, -1));
      HIP_OR_FAIL(ctx, launch_pb_relax(ctx->sb, ctx->d_ux_prev, ctx->stream));
    }
    HIP_OR_FAIL(ctx, hipMemsetAsync(ctx->d_ux_prev, 0, ctx->total_nodes * sizeof(double), ctx->stream));
    HIP_OR_FAIL(ctx, hipStreamSynchronize(ctx->stream));
  }
  ctx->has_pops = false;
  ctx->steps = 0;
  ctx->snapshot_step = -1;
  return EKPNP_OK;
}

int ekpnp_init_equilibrium(ekpnp_ctx* ctx) {
  const ApiRange range_("ekpnp_init_equilibrium");
  if (!ctx) return EKPNP_ERR_INVALID;
  if (!ctx->has_fields) return fail(ctx, EKPNP_ERR_STATE, "init_equilibrium before initialization/set_fields");
  HIP_OR_FAIL(ctx, hipSetDevice(ctx->opt.device));
  bool reset = false;
  for (auto& d : ctx->desc) {
    reset |= (d.swap != 0 || d.active != 1);
    d.swap = 0;
    d.active = 1;
  }
  if (reset) HIP_OR_FAIL(ctx, sync_desc(ctx));
  // FP32 storage: populations are stored as deviations from w_i times the
  // references (block means along x, row-mean fluxes) of the fields they start from
  if (ctx->opt.precision == EKPNP_POP_FP32)
    HIP_OR_FAIL(ctx, launch_row_means(ctx->sb, ctx->d_refs, ctx->d_blocks, ctx->stream));
  HIP_OR_FAIL(ctx, launch_init_equilibrium(ctx->opt.precision, ctx->sb, ctx->lat[ctx->cur], ctx->stream));
  HIP_OR_FAIL(ctx, hipStreamSynchronize(ctx->stream));
  ctx->state_q = true;
  ctx->has_pops = true;
  ctx->rebase_step = ctx->steps;
  ctx->origin_step = ctx->steps;
  return EKPNP_OK;
}

int ekpnp_restart_channel(ekpnp_ctx* ctx, int channel, int mode, uint64_t seed) {
  const ApiRange range_("ekpnp_restart_channel");
  int rc = check_channel(ctx, channel);
  if (rc) return rc;
  if (mode != EKPNP_INIT_COLD_NOISE && mode != EKPNP_INIT_REFERENCE)
    return fail(ctx, EKPNP_ERR_UNSUPPORTED, "restart_channel: cold-noise or reference start only");
  if (!ctx->has_pops) return fail(ctx, EKPNP_ERR_STATE, "restart_channel: no populations (use init_equilibrium)");
  HIP_OR_FAIL(ctx, hipSetDevice(ctx->opt.device));
  const ChanDesc& d = ctx->desc[channel];
  if (!d.active || d.swap) return fail(ctx, EKPNP_ERR_STATE, "restart_channel: channel frozen");
  // the channel's fields (macroscopic planes, charge, its own Poisson solve)
  rc = initial_fields(ctx, channel, mode, seed);
  if (rc) return rc;
  // every other channel keeps its state: the lattice goes to the unshifted
  // pre-collision form (a copy of the values, as for set_populations), then
  // only this channel's work-groups re-derive its references and write its
  // equilibrium populations
  if (!ctx->state_q) {
    HIP_OR_FAIL(ctx, launch_to_q(ctx->opt.precision, ctx->sb, ctx->lat[ctx->cur], ctx->lat[ctx->cur ^ 1], ctx->stream));
    ctx->cur ^= 1;
    ctx->state_q = true;
  }
  StepBuffers b = ctx->sb;
  const int t0 = ctx->first_tile[channel];
  const int t1 = channel + 1 < ctx->nchan ? ctx->first_tile[channel + 1] : (int)ctx->lbm_tiles.size();
  b.lbm_tiles = ctx->d_lbm_tiles + t0;
  b.n_lbm_tiles = t1 - t0;
  b.row_tiles = ctx->d_row_tiles + ctx->ctiles[channel].row_first;
  b.n_row_tiles = d.ny;
  b.n_row_narrow = d.nx <= ROW_WAVE_NX ? d.ny : 0;
  if (ctx->opt.precision == EKPNP_POP_FP32)
    HIP_OR_FAIL(ctx, launch_row_means(b, ctx->d_refs, ctx->d_blocks, ctx->stream));
  HIP_OR_FAIL(ctx, launch_init_equilibrium(ctx->opt.precision, b, ctx->lat[ctx->cur], ctx->stream));
  // the residual snapshot of this channel restarts from its new u_x
  const size_t nn = (size_t)d.nx * d.ny;
  HIP_OR_FAIL(ctx, hipMemcpyAsync(ctx->d_ux_prev + d.fld_off, ctx->d_macro + M_UX * ctx->total_nodes + d.fld_off,
                                  nn * sizeof(double), hipMemcpyDeviceToDevice, ctx->stream));
  HIP_OR_FAIL(ctx, hipStreamSynchronize(ctx->stream));
  return EKPNP_OK;
}

int ekpnp_stream_collide_save(ekpnp_ctx* ctx) {
  const ApiRange range_("ekpnp_stream_collide_save");
  if (!ctx) return EKPNP_ERR_INVALID;
  if (!ctx->has_pops) return fail(ctx, EKPNP_ERR_STATE, "no populations: call init_equilibrium first");
  HIP_OR_FAIL(ctx, hipSetDevice(ctx->opt.device));
  HIP_OR_FAIL(ctx, enqueue_lbm(ctx, true));
  ctx->steps++;
  return EKPNP_OK;
}

int ekpnp_fast_poisson(ekpnp_ctx* ctx) {
  const ApiRange range_("ekpnp_fast_poisson");
  if (!ctx) return EKPNP_ERR_INVALID;
  if (!ctx->has_fields) return fail(ctx, EKPNP_ERR_STATE, "no fields");
  HIP_OR_FAIL(ctx, hipSetDevice(ctx->opt.device));
  HIP_OR_FAIL(ctx, enqueue_poisson(ctx, -1));
  return EKPNP_OK;
}

int ekpnp_poisson_iterative(ekpnp_ctx* ctx, int channel, double omega, double tol, int max_iter, int check_every,
                            int* iters_out, double* change_out) {
  const ApiRange range_("ekpnp_poisson_iterative");
  if (!ctx || !iters_out || !change_out) return EKPNP_ERR_INVALID;
  if (channel < 0 || channel >= ctx->nchan) return fail(ctx, EKPNP_ERR_INVALID, "channel out of range");
  if (!(omega > 0.0 && omega < 2.0)) return fail(ctx, EKPNP_ERR_INVALID, "omega must lie in (0, 2)");
  if (!(tol >= 0.0) || max_iter < 1 || check_every < 1)
    return fail(ctx, EKPNP_ERR_INVALID, "need tol >= 0, max_iter >= 1, check_every >= 1");
  if (!ctx->has_fields) return fail(ctx, EKPNP_ERR_STATE, "no fields");
  const ChanDesc& d = ctx->desc[channel];
  if (d.nx & 1)
    return fail(ctx, EKPNP_ERR_UNSUPPORTED, "the iterative Poisson solve needs an even nx (red-black colouring)");
  HIP_OR_FAIL(ctx, hipSetDevice(ctx->opt.device));
  const ekpnp_channel_params& p = ctx->params[channel];
  const double r = (p.dy / p.dx) * (p.dy / p.dx);
  const double inv = 1.0 / (2.0 * (1.0 + r));
  const int nwg = ((d.nx / 2) * (d.ny - 2) + LBM_WG - 1) / LBM_WG;  // per colour; 2 nwg <= LBM tiles
  double* part = ctx->d_partials;
  HIP_OR_FAIL(ctx, launch_psi_wall_rows(ctx->sb, channel, d.nx, ctx->stream));
  int it = 0;
  double change = INFINITY;
  while (it < max_iter) {
    HIP_OR_FAIL(ctx, launch_sor_sweep(ctx->sb, channel, d.nx, d.ny, 0, omega, r, inv, part, ctx->stream));
    HIP_OR_FAIL(ctx, launch_sor_sweep(ctx->sb, channel, d.nx, d.ny, 1, omega, r, inv, part + nwg, ctx->stream));
    ++it;
    if (it % check_every == 0 || it == max_iter) {
      HIP_OR_FAIL(ctx, launch_max_final(part, 2 * nwg, ctx->d_red, ctx->stream));
      HIP_OR_FAIL(ctx, hipMemcpyAsync(&change, ctx->d_red, sizeof(double), hipMemcpyDeviceToHost, ctx->stream));
      HIP_OR_FAIL(ctx, hipStreamSynchronize(ctx->stream));
      if (change < tol) break;  // poisson.cu:57
    }
  }
  *iters_out = it;
  *change_out = change;
  return EKPNP_OK;
}

int ekpnp_rebase(ekpnp_ctx* ctx) {
  const ApiRange range_("ekpnp_rebase");
  if (!ctx) return EKPNP_ERR_INVALID;
  if (!ctx->has_pops) return fail(ctx, EKPNP_ERR_STATE, "no populations: call init_equilibrium first");
  ctx->rebase_step = ctx->steps;
  if (ctx->opt.precision != EKPNP_POP_FP32) return EKPNP_OK;
  HIP_OR_FAIL(ctx, hipSetDevice(ctx->opt.device));
  // the macroscopic planes hold the moments of the last step (or the fields
  // the populations were initialised from)
  // (frozen channels of run_to_residual keep their references and state)
  HIP_OR_FAIL(ctx, launch_row_means(ctx->sb, ctx->d_refs_new, ctx->d_blocks_new, ctx->stream));
  HIP_OR_FAIL(ctx, launch_rebase(ctx->opt.precision, ctx->sb, ctx->lat[ctx->cur], ctx->lat[ctx->cur ^ 1],
                                 ctx->d_refs_new, ctx->d_blocks_new, ctx->stream));
  HIP_OR_FAIL(ctx, hipMemcpyAsync(ctx->d_refs, ctx->d_refs_new, ctx->total_refs * sizeof(double),
                                  hipMemcpyDeviceToDevice, ctx->stream));
  HIP_OR_FAIL(ctx, hipMemcpyAsync(ctx->d_blocks, ctx->d_blocks_new, ctx->total_blocks * sizeof(float),
                                  hipMemcpyDeviceToDevice, ctx->stream));
  return EKPNP_OK;
}

int ekpnp_step(ekpnp_ctx* ctx, int nsteps) {
  const ApiRange range_("ekpnp_step");
  if (!ctx) return EKPNP_ERR_INVALID;
  if (nsteps < 0) return fail(ctx, EKPNP_ERR_INVALID, "negative step count");
  if (nsteps == 0) return EKPNP_OK;
  if (!ctx->has_pops) return fail(ctx, EKPNP_ERR_STATE, "no populations: call init_equilibrium first");
  HIP_OR_FAIL(ctx, hipSetDevice(ctx->opt.device));
  // FP32 storage follows the drifting row means so that the stored
  // deviations stay small: a long call is cut into segments that end where
  // a re-centring is due (the last step of each segment writes the
  // macroscopic planes the re-centring reads)
  const bool fp32 = ctx->opt.precision == EKPNP_POP_FP32;
  int left = nsteps;
  while (left > 0) {
    int n = left;
    if (fp32) {
      // overdue (steps taken by other entry points): re-centre first; the
      // change of representation is exact whatever the references
      if (ctx->steps >= next_rebase(ctx)) {
        int rc = ekpnp_rebase(ctx);
        if (rc) return rc;
      }
      const long long until = next_rebase(ctx) - ctx->steps;
      if (until < n) n = (int)until;
    }
    const int seg = n;
    if (ctx->state_q) {
      HIP_OR_FAIL(ctx, enqueue_steps(ctx, 1, n == 1));
      n -= 1;
    }
    if (!ctx->opt.use_graph) {
      HIP_OR_FAIL(ctx, enqueue_steps(ctx, n, true));
    } else {
      const int CHUNK = 64;
      while (n > 0) {
        const int k = n > CHUNK ? CHUNK : n;
        const bool last = (k == n);
        int rc = graph_steps(ctx, k, last);
        if (rc) return rc;
        n -= k;
      }
    }
    ctx->steps += seg;
    left -= seg;
    if (fp32 && ctx->steps >= next_rebase(ctx)) {
      int rc = ekpnp_rebase(ctx);
      if (rc) return rc;
    }
  }
  return EKPNP_OK;
}

int ekpnp_synchronize(ekpnp_ctx* ctx) {
  if (!ctx) return EKPNP_ERR_INVALID;
  HIP_OR_FAIL(ctx, hipSetDevice(ctx->opt.device));
  HIP_OR_FAIL(ctx, hipStreamSynchronize(ctx->stream));
  return EKPNP_OK;
}

int ekpnp_get_field(ekpnp_ctx* ctx, int channel, int field, double* host_out) {
  const ApiRange range_("ekpnp_get_field");
  int rc = check_channel(ctx, channel);
  if (rc) return rc;
  if (!host_out) return fail(ctx, EKPNP_ERR_INVALID, "null output");
  if (field < 0 || field >= EKPNP_FIELD_COUNT) return fail(ctx, EKPNP_ERR_INVALID, "unknown field");
  HIP_OR_FAIL(ctx, hipSetDevice(ctx->opt.device));
  const ChanDesc& d = ctx->desc[channel];
  const ekpnp_channel_params& p = ctx->params[channel];
  const size_t nn = (size_t)d.nx * d.ny;
  if (field <= EKPNP_FIELD_CNEG) {
    HIP_OR_FAIL(ctx, copy_to_host(ctx, host_out, ctx->d_macro + field * ctx->total_nodes + d.fld_off,
                                  nn * sizeof(double)));
    return EKPNP_OK;
  }
  if (field == EKPNP_FIELD_PSI) {
    HIP_OR_FAIL(ctx, copy_to_host(ctx, host_out, ctx->d_psi + d.fld_off, nn * sizeof(double)));
    return EKPNP_OK;
  }
  std::vector<double> psi(nn);
  HIP_OR_FAIL(ctx, copy_to_host(ctx, psi.data(), ctx->d_psi + d.fld_off, nn * sizeof(double)));
  // E = -grad(psi), poisson.cu:145-174
  const int nx = d.nx, ny = d.ny;
  for (int y = 0; y < ny; ++y) {
    for (int x = 0; x < nx; ++x) {
      const int xm = (x + nx - 1) % nx, xp = (x + 1) % nx;
      if (field == EKPNP_FIELD_EX) {
        host_out[(size_t)y * nx + x] = (psi[(size_t)y * nx + xm] - psi[(size_t)y * nx + xp]) * (0.5 / p.dx);
      } else {
        int ya = y - 1, yb = y + 1;
        if (y == 0) { ya = 0; yb = 2; }
        if (y == ny - 1) { ya = ny - 3; yb = ny - 1; }
        host_out[(size_t)y * nx + x] = (psi[(size_t)ya * nx + x] - psi[(size_t)yb * nx + x]) * (0.5 / p.dy);
      }
    }
  }
  return EKPNP_OK;
}

int ekpnp_get_populations(ekpnp_ctx* ctx, int channel, int species, double* host_out) {
  const ApiRange range_("ekpnp_get_populations");
  int rc = check_channel(ctx, channel);
  if (rc) return rc;
  if (species < 0 || species > 2 || !host_out) return fail(ctx, EKPNP_ERR_INVALID, "bad species or output");
  if (!ctx->has_pops) return fail(ctx, EKPNP_ERR_STATE, "no populations");
  HIP_OR_FAIL(ctx, hipSetDevice(ctx->opt.device));
  const int L = chan_lattice(ctx, channel);
  const void* src = ctx->lat[L];
  if (!ctx->state_q) {
    // every channel's pre-collision state lands in the lattice its state is not in
    HIP_OR_FAIL(ctx, launch_to_q(ctx->opt.precision, ctx->sb, ctx->lat[ctx->cur], ctx->lat[ctx->cur ^ 1], ctx->stream));
    src = ctx->lat[L ^ 1];
  }
  HIP_OR_FAIL(ctx, hipStreamSynchronize(ctx->stream));
  const ChanDesc& d = ctx->desc[channel];
  const size_t nn = (size_t)d.nx * d.ny;
  hipError_t re = hipSuccess;
  const std::vector<double> ref = ref_offsets(ctx, channel, species, &re);
  HIP_OR_FAIL(ctx, re);
  const size_t off = (size_t)d.pop_off + (size_t)(9 * species) * (size_t)d.plane;
  const char* base = (const char*)src + off * ctx->elem;
  if (ctx->elem == 8) {
    HIP_OR_FAIL(ctx, hipMemcpy2D(host_out, nn * 8, base, (size_t)d.plane * 8, nn * 8, 9, hipMemcpyDeviceToHost));
  } else {
    std::vector<float> tmp(9 * nn);
    HIP_OR_FAIL(ctx, hipMemcpy2D(tmp.data(), nn * 4, base, (size_t)d.plane * 4, nn * 4, 9, hipMemcpyDeviceToHost));
    for (size_t i = 0; i < 9 * nn; ++i) host_out[i] = (double)tmp[i];
  }
  for (size_t i = 0; i < 9 * nn; ++i) host_out[i] += ref[i];
  return EKPNP_OK;
}

int ekpnp_set_populations(ekpnp_ctx* ctx, int channel, int species, const double* host_in) {
  const ApiRange range_("ekpnp_set_populations");
  int rc = check_channel(ctx, channel);
  if (rc) return rc;
  if (species < 0 || species > 2 || !host_in) return fail(ctx, EKPNP_ERR_INVALID, "bad species or input");
  HIP_OR_FAIL(ctx, hipSetDevice(ctx->opt.device));
  if (ctx->has_pops && !ctx->state_q) {
    // bring every channel to the unshifted pre-collision form first
    HIP_OR_FAIL(ctx, launch_to_q(ctx->opt.precision, ctx->sb, ctx->lat[ctx->cur], ctx->lat[ctx->cur ^ 1], ctx->stream));
    ctx->cur ^= 1;
  }
  ctx->state_q = true;
  const ChanDesc& d = ctx->desc[channel];
  const size_t nn = (size_t)d.nx * d.ny;
  const size_t off = (size_t)d.pop_off + (size_t)(9 * species) * (size_t)d.plane;
  char* base = (char*)ctx->lat[chan_lattice(ctx, channel)] + off * ctx->elem;
  HIP_OR_FAIL(ctx, hipStreamSynchronize(ctx->stream));
  hipError_t re = hipSuccess;
  const std::vector<double> ref = ref_offsets(ctx, channel, species, &re);
  HIP_OR_FAIL(ctx, re);
  if (ctx->elem == 8) {
    std::vector<double> tmp(9 * nn);
    for (int dd = 0; dd < 9; ++dd)
      for (size_t i = 0; i < nn; ++i) tmp[dd * nn + i] = host_in[dd * nn + i] - ref[dd * nn + i];
    HIP_OR_FAIL(ctx, hipMemcpy2D(base, (size_t)d.plane * 8, tmp.data(), nn * 8, nn * 8, 9, hipMemcpyHostToDevice));
  } else {
    std::vector<float> tmp(9 * nn);
    for (int dd = 0; dd < 9; ++dd)
      for (size_t i = 0; i < nn; ++i) tmp[dd * nn + i] = (float)(host_in[dd * nn + i] - ref[dd * nn + i]);
    HIP_OR_FAIL(ctx, hipMemcpy2D(base, (size_t)d.plane * 4, tmp.data(), nn * 4, nn * 4, 9, hipMemcpyHostToDevice));
  }
  ctx->has_pops = true;
  return EKPNP_OK;
}

// residuals from the copied records (DUX2 and UX2 over the interval since
// the last snapshot), and the new snapshot's step
static void finish_reductions(ekpnp_ctx* ctx, double* out) {
  const long long interval = ctx->snapshot_step >= 0 ? ctx->steps - ctx->snapshot_step : 0;
  for (int ch = 0; ch < ctx->nchan; ++ch) {
    double* r = out + 8 * ch;
    double res = 0.0;
    if (interval > 0) {
      res = (r[EKPNP_RED_UX2] > 0.0) ? std::sqrt(r[EKPNP_RED_DUX2] / r[EKPNP_RED_UX2]) / (double)interval
                                     : (r[EKPNP_RED_DUX2] > 0.0 ? INFINITY : 0.0);
    }
    r[EKPNP_RED_RESIDUAL] = res;
  }
  ctx->snapshot_step = ctx->steps;
}

int ekpnp_reductions(ekpnp_ctx* ctx, double* out) {
  const ApiRange range_("ekpnp_reductions");
  if (!ctx || !out) return EKPNP_ERR_INVALID;
  HIP_OR_FAIL(ctx, hipSetDevice(ctx->opt.device));
  HIP_OR_FAIL(ctx, launch_reductions(ctx->sb, 1, ctx->stream));
  HIP_OR_FAIL(ctx, hipMemcpyAsync(out, ctx->d_red, 8 * (size_t)ctx->nchan * sizeof(double),
                                  hipMemcpyDeviceToHost, ctx->stream));
  HIP_OR_FAIL(ctx, hipStreamSynchronize(ctx->stream));
  finish_reductions(ctx, out);
  return EKPNP_OK;
}

int ekpnp_reductions_noalloc(ekpnp_ctx* ctx, double* out) {
  const ApiRange range_("ekpnp_reductions_noalloc");
  if (!ctx || !out) return EKPNP_ERR_INVALID;
  const long long need = 8LL * ((long long)ctx->lbm_tiles.size() + ctx->nchan);
  if (need > NOALLOC_SCRATCH_DOUBLES)
    return fail(ctx, EKPNP_ERR_UNSUPPORTED,
                "ekpnp_reductions_noalloc: 8 x (LBM tiles + channels) = " + std::to_string(need) +
                    " doubles exceed its scratch of " + std::to_string(NOALLOC_SCRATCH_DOUBLES) +
                    " (contexts of up to about 33 million nodes)");
  HIP_OR_FAIL(ctx, hipSetDevice(ctx->opt.device));
  double* ptr = noalloc_scratch(ctx->opt.device);
  if (!ptr) return fail(ctx, EKPNP_ERR_STATE, "ekpnp_reductions_noalloc: scratch address not set up");
  // partial sums of every tile, then the per-channel records, in the
  // scratch array; both kernels write every slot they later read, so
  // nothing is cleared first
  StepBuffers b = ctx->sb;
  b.partials = ptr;
  b.red_out = ptr + 8LL * (long long)ctx->lbm_tiles.size();
  HIP_OR_FAIL(ctx, launch_reductions(b, 1, ctx->stream));
  HIP_OR_FAIL(ctx, hipMemcpyAsync(out, b.red_out, 8 * (size_t)ctx->nchan * sizeof(double), hipMemcpyDeviceToHost,
                                  ctx->stream));
  HIP_OR_FAIL(ctx, hipStreamSynchronize(ctx->stream));
  finish_reductions(ctx, out);
  return EKPNP_OK;
}

}  // extern "C"

int ekpnp::channel_diagnostics(ekpnp_ctx* ctx, int channel, double* umax, double* current_sum) {
  int rc = check_channel(ctx, channel);
  if (rc) return rc;
  HIP_OR_FAIL(ctx, hipSetDevice(ctx->opt.device));
  const ChanDesc& d = ctx->desc[channel];
  const ekpnp_channel_params& p = ctx->params[channel];
  const long long nn = (long long)d.nx * d.ny;
  const int grid = (int)std::min<long long>(DIAG_MAX_WG, std::max<long long>(1, (nn + 4095) / 4096));
  const double* uy = ctx->d_macro + M_UY * ctx->total_nodes + d.fld_off;
  const double* cp = ctx->d_macro + M_CP * ctx->total_nodes + d.fld_off;
  double* out = ctx->d_diag + 2 * DIAG_MAX_WG;
  HIP_OR_FAIL(ctx, launch_diagnostics(uy, cp, ctx->d_psi + d.fld_off, d.nx, d.ny, 0.5 / p.dy, ctx->d_diag, grid,
                                      out, ctx->stream));
  double host[2];
  HIP_OR_FAIL(ctx, hipMemcpyAsync(host, out, sizeof(host), hipMemcpyDeviceToHost, ctx->stream));
  HIP_OR_FAIL(ctx, hipStreamSynchronize(ctx->stream));
  if (umax) *umax = host[0];
  if (current_sum) *current_sum = host[1];
  return EKPNP_OK;
}

extern "C" {

int ekpnp_run_to_residual(ekpnp_ctx* ctx, double tol, int check_every, int max_steps, int* steps_out) {
  const ApiRange range_("ekpnp_run_to_residual");
  if (!ctx) return EKPNP_ERR_INVALID;
  if (check_every < 2 || (check_every & 1)) return fail(ctx, EKPNP_ERR_INVALID, "check_every must be even and >= 2");
  if (!ctx->has_pops) return fail(ctx, EKPNP_ERR_STATE, "no populations");
  std::vector<double> red(8 * (size_t)ctx->nchan);
  std::vector<int> done(ctx->nchan, -1);
  // converged channels are frozen (their kernels return at once) until the
  // call ends; frozen_lat remembers which lattice holds each frozen state
  std::vector<int> frozen_lat(ctx->nchan, -1);
  auto thaw = [&]() -> int {
    bool any = false;
    for (int ch = 0; ch < ctx->nchan; ++ch) {
      if (frozen_lat[ch] < 0) continue;
      ctx->desc[ch].swap = ctx->cur ^ frozen_lat[ch];
      ctx->desc[ch].active = 1;
      frozen_lat[ch] = -1;
      any = true;
    }
    if (any) HIP_OR_FAIL(ctx, sync_desc(ctx));
    if (steps_out)
      for (int k = 0; k < ctx->nchan; ++k) steps_out[k] = done[k];
    return EKPNP_OK;
  };
  int rc = ekpnp_reductions(ctx, red.data());  // snapshot
  if (rc) return rc;
  long long start = ctx->steps;
  int remaining = ctx->nchan;
  while (remaining > 0 && ctx->steps - start < max_steps) {
    rc = ekpnp_step(ctx, check_every);
    if (rc) {
      thaw();
      return rc;
    }
    rc = ekpnp_reductions(ctx, red.data());
    if (rc) {
      thaw();
      return rc;
    }
    bool froze = false;
    for (int ch = 0; ch < ctx->nchan; ++ch) {
      if (red[8 * ch + EKPNP_RED_NONFINITE] > 0.0) {
        char buf[128];
        snprintf(buf, sizeof buf, "channel %d: non-finite values after %lld steps", ch, ctx->steps - start);
        std::string msg = buf;
        thaw();
        return fail(ctx, EKPNP_ERR_UNSTABLE, msg);
      }
      if (done[ch] < 0 && red[8 * ch + EKPNP_RED_RESIDUAL] <= tol) {
        done[ch] = (int)(ctx->steps - start);
        --remaining;
        frozen_lat[ch] = chan_lattice(ctx, ch);
        ctx->desc[ch].active = 0;
        froze = true;
      }
    }
    if (froze && remaining > 0) {
      hipError_t e = sync_desc(ctx);
      if (e != hipSuccess) {
        thaw();
        return fail(ctx, EKPNP_ERR_HIP, std::string("sync_desc: ") + hipGetErrorString(e));
      }
    }
  }
  return thaw();
}

int ekpnp_autotune(ekpnp_ctx* ctx, int reps, double* out) {
  const ApiRange range_("ekpnp_autotune");
  if (!ctx || reps <= 0) return EKPNP_ERR_INVALID;
  HIP_OR_FAIL(ctx, hipSetDevice(ctx->opt.device));
  HIP_OR_FAIL(ctx, hipStreamSynchronize(ctx->stream));
  // every trial recomputes psi from rho_e; the current psi is put back after
  double* keep = nullptr;
  HIP_OR_FAIL(ctx, hipMalloc((void**)&keep, ctx->total_nodes * sizeof(double)));
  hipEvent_t ev[2] = {nullptr, nullptr};
  auto finish = [&](int rc) {
    for (auto e : ev)
      if (e) (void)hipEventDestroy(e);
    (void)hipFree(keep);
    return rc;
  };
  if (hipMemcpyAsync(keep, ctx->d_psi, ctx->total_nodes * sizeof(double), hipMemcpyDeviceToDevice, ctx->stream) !=
          hipSuccess ||
      hipEventCreate(&ev[0]) != hipSuccess || hipEventCreate(&ev[1]) != hipSuccess)
    return finish(fail(ctx, EKPNP_ERR_HIP, "autotune set-up failed"));
  const int elems[3] = {1024, 2048, 4096};
  const int rows[2] = {8, 16};
  int best_e = ctx->fft_elems, best_r = ctx->tri_rows, best_p = ctx->fft_persist;
  double best = 1e30;
  // three passes over the candidates, each candidate's fastest pass counting:
  // one timing of `reps` solves can be off by a transient (seen under a
  // profiler, which then picked a plan 10 % slower)
  for (int ic = 0; ic < 27; ++ic) {
    // one-tile kernels for every size, persistent up to 2048, row pairs
    // where the channels allow them
    const int ie = ic % 3, ip = (ic / 3) % 3;
    if (ip == 1 && elems[ie] > FFT_PERSIST_ELEMS) continue;
    // a step by k_lbm_fwd holds the persistent family's transforms, and saves more
    // than another family could (64x128 with FP64 storage: 16.3 against 21.7 us)
    if (ip != 1 && !ctx->lbm_fwd.empty()) continue;
    for (int ir = 0; ir < 2; ++ir) {
      hipError_t e = build_poisson_plan(ctx, elems[ie], rows[ir], ip);
      if (e == hipSuccess && ip == 2 && ctx->fft_persist != 2) break;  // not eligible
      for (int w = 0; w < 2 && e == hipSuccess; ++w) e = enqueue_poisson(ctx, -1);
      if (e == hipSuccess) e = hipEventRecord(ev[0], ctx->stream);
      for (int k = 0; k < reps && e == hipSuccess; ++k) e = enqueue_poisson(ctx, -1);
      if (e == hipSuccess) e = hipEventRecord(ev[1], ctx->stream);
      if (e == hipSuccess) e = hipEventSynchronize(ev[1]);
      float ms = 0.0f;
      if (e == hipSuccess) e = hipEventElapsedTime(&ms, ev[0], ev[1]);
      if (e != hipSuccess) return finish(fail(ctx, EKPNP_ERR_HIP, std::string("autotune: ") + hipGetErrorString(e)));
      const double per = (double)ms / reps;
      if (per < best) {
        best = per;
        best_e = elems[ie];
        best_r = rows[ir];
        best_p = ctx->fft_persist;
      }
    }
  }
  hipError_t e = build_poisson_plan(ctx, best_e, best_r, best_p);
  if (e == hipSuccess)
    e = hipMemcpyAsync(ctx->d_psi, keep, ctx->total_nodes * sizeof(double), hipMemcpyDeviceToDevice, ctx->stream);
  if (e == hipSuccess) e = hipStreamSynchronize(ctx->stream);
  if (e != hipSuccess) return finish(fail(ctx, EKPNP_ERR_HIP, std::string("autotune: ") + hipGetErrorString(e)));
  if (out) {
    out[0] = best_e;
    out[1] = best_r;
    out[2] = best;
    out[3] = ctx->fft_persist;
  }
  return finish(EKPNP_OK);
}

int ekpnp_set_poisson_plan(ekpnp_ctx* ctx, int fft_elems, int tri_rows, int fft_persistent) {
  if (!ctx) return EKPNP_ERR_INVALID;
  if (fft_elems < 1 || fft_elems > FFT_MAX_ELEMS || tri_rows < 1 || tri_rows > 16 || fft_persistent < 0 ||
      fft_persistent > 2)
    return fail(ctx, EKPNP_ERR_INVALID,
                "fft_elems must be in [1, 4096], tri_rows in [1, 16] and fft_persistent in [0, 2]");
  HIP_OR_FAIL(ctx, hipSetDevice(ctx->opt.device));
  HIP_OR_FAIL(ctx, hipStreamSynchronize(ctx->stream));
  HIP_OR_FAIL(ctx, build_poisson_plan(ctx, fft_elems, tri_rows, fft_persistent));
  return EKPNP_OK;
}

int ekpnp_get_poisson_plan(const ekpnp_ctx* ctx, int* out) {
  if (!ctx || !out) return EKPNP_ERR_INVALID;
  out[0] = ctx->fft_elems;
  out[1] = ctx->tri_rows;
  out[2] = ctx->fft_persist;
  out[3] = (ctx->walls_in_tri && ctx->opt.precision == 0 && ctx->opt.compute_fp64 != 0) ? 1 : 0;
  return EKPNP_OK;
}

int ekpnp_set_lbm_tiles(ekpnp_ctx* ctx, int wrows) {
  if (!ctx) return EKPNP_ERR_INVALID;
  if (wrows != 0 && wrows != 2 && wrows != 4) return fail(ctx, EKPNP_ERR_INVALID, "wrows must be 0, 2 or 4");
  HIP_OR_FAIL(ctx, hipSetDevice(ctx->opt.device));
  HIP_OR_FAIL(ctx, apply_lbm_tiles(ctx, wrows));
  return EKPNP_OK;
}

int ekpnp_get_lbm_tiles(const ekpnp_ctx* ctx, int* wrows) {
  if (!ctx || !wrows) return EKPNP_ERR_INVALID;
  *wrows = ctx->lbm_wrows;
  return EKPNP_OK;
}

// Times the row kernel's interior launch for each tile shape on the current
// state without advancing it: a trial reads the current lattice and writes
// the other one (the next step overwrites it) and the charge density, which
// is saved and put back; no macroscopic planes.
int ekpnp_autotune_lbm(ekpnp_ctx* ctx, int reps, double* out) {
  const ApiRange range_("ekpnp_autotune_lbm");
  if (!ctx || reps <= 0) return EKPNP_ERR_INVALID;
  if (!ctx->has_pops) return fail(ctx, EKPNP_ERR_STATE, "autotune_lbm: no populations (call init_equilibrium first)");
  HIP_OR_FAIL(ctx, hipSetDevice(ctx->opt.device));
  HIP_OR_FAIL(ctx, hipStreamSynchronize(ctx->stream));
  const bool rows = ctx->opt.precision == EKPNP_POP_FP32 && ctx->opt.compute_fp64 != 0 && ctx->n_lbm_row > 0;
  if (!rows) {  // no channel on the row kernel: nothing to choose
    if (out) {
      out[0] = ctx->lbm_wrows;
      out[1] = 0.0;
    }
    return EKPNP_OK;
  }
  double* keep = nullptr;
  HIP_OR_FAIL(ctx, hipMalloc((void**)&keep, ctx->total_nodes * sizeof(double)));
  hipEvent_t ev[2] = {nullptr, nullptr};
  auto finish = [&](int rc) {
    for (auto e : ev)
      if (e) (void)hipEventDestroy(e);
    (void)hipFree(keep);
    return rc;
  };
  if (hipMemcpyAsync(keep, ctx->d_rho_e, ctx->total_nodes * sizeof(double), hipMemcpyDeviceToDevice, ctx->stream) !=
          hipSuccess ||
      hipEventCreate(&ev[0]) != hipSuccess || hipEventCreate(&ev[1]) != hipSuccess)
    return finish(fail(ctx, EKPNP_ERR_HIP, "autotune_lbm set-up failed"));
  const int shapes[3] = {0, 2, 4};
  double best_ms[3] = {1e30, 1e30, 1e30};
  // three passes over the shapes, each shape's fastest pass counting
  for (int pass = 0; pass < 3; ++pass)
    for (int is = 0; is < 3; ++is) {
      hipError_t e = apply_lbm_tiles(ctx, shapes[is]);
      const void* src = ctx->lat[ctx->cur];
      void* dst = ctx->lat[ctx->cur ^ 1];
      for (int w = 0; w < 2 && e == hipSuccess; ++w) e = launch_lbm_rows_interior(ctx->sb, src, dst, ctx->stream);
      if (e == hipSuccess) e = hipEventRecord(ev[0], ctx->stream);
      for (int k = 0; k < reps && e == hipSuccess; ++k) e = launch_lbm_rows_interior(ctx->sb, src, dst, ctx->stream);
      if (e == hipSuccess) e = hipEventRecord(ev[1], ctx->stream);
      if (e == hipSuccess) e = hipEventSynchronize(ev[1]);
      float ms = 0.0f;
      if (e == hipSuccess) e = hipEventElapsedTime(&ms, ev[0], ev[1]);
      if (e != hipSuccess)
        return finish(fail(ctx, EKPNP_ERR_HIP, std::string("autotune_lbm: ") + hipGetErrorString(e)));
      best_ms[is] = std::min(best_ms[is], (double)ms / reps);
    }
  // another shape replaces the default (consecutive blocks, the least HBM
  // traffic) only when it is at least 1 % faster: the shapes often time
  // within the run-to-run spread of each other
  int best = 0;
  for (int is = 1; is < 3; ++is)
    if (best_ms[is] < 0.99 * best_ms[0] && best_ms[is] < best_ms[best]) best = is;
  hipError_t e = apply_lbm_tiles(ctx, shapes[best]);
  if (e == hipSuccess)
    e = hipMemcpyAsync(ctx->d_rho_e, keep, ctx->total_nodes * sizeof(double), hipMemcpyDeviceToDevice, ctx->stream);
  if (e == hipSuccess) e = hipStreamSynchronize(ctx->stream);
  if (e != hipSuccess) return finish(fail(ctx, EKPNP_ERR_HIP, std::string("autotune_lbm: ") + hipGetErrorString(e)));
  if (out) {
    out[0] = shapes[best];
    out[1] = best_ms[best];
  }
  return finish(EKPNP_OK);
}

int ekpnp_get_params(ekpnp_ctx* ctx, int channel, ekpnp_channel_params* out) {
  int rc = check_channel(ctx, channel);
  if (rc) return rc;
  if (!out) return fail(ctx, EKPNP_ERR_INVALID, "null output");
  *out = ctx->params[channel];
  return EKPNP_OK;
}

// ---------------------------------------------------------------------------
// Binary checkpoint.  Layout (native byte order):
//   char[8] "EKPNPCK2"; int32 nchan, precision, state_q, has_pops;
//   int64 steps, snapshot_step, rebase_step, origin_step;
//   per channel: int32 nx, ny;
//   per channel: populations [27][ny][nx] in the storage type, references
//   [ny][8], block references [ny][nb][4] (FP32, nb = ceil(nx/64)), psi, rho, ux,
//   uy, c+, c- [ny][nx], wall planes [6][nx],
//   residual snapshot [ny][nx] (FP64 unless stated).
// ---------------------------------------------------------------------------
namespace {
const char kCkptMagic[8] = {'E', 'K', 'P', 'N', 'P', 'C', 'K', '2'};

struct FileCloser {
  FILE* f;
  ~FileCloser() {
    if (f) std::fclose(f);
  }
};
}  // namespace

int ekpnp_save_checkpoint(ekpnp_ctx* ctx, const char* path) {
  const ApiRange range_("ekpnp_save_checkpoint");
  if (!ctx || !path) return EKPNP_ERR_INVALID;
  if (!ctx->has_fields) return fail(ctx, EKPNP_ERR_STATE, "nothing to save: no fields");
  HIP_OR_FAIL(ctx, hipSetDevice(ctx->opt.device));
  HIP_OR_FAIL(ctx, hipStreamSynchronize(ctx->stream));
  FILE* fp = std::fopen(path, "wb");
  if (!fp) return fail(ctx, EKPNP_ERR_IO, std::string("cannot open ") + path);
  FileCloser closer{fp};
  bool ok = true;
  auto put = [&](const void* p, size_t n) { ok = ok && std::fwrite(p, 1, n, fp) == n; };
  const int32_t hdr[4] = {ctx->nchan, ctx->opt.precision, ctx->state_q ? 1 : 0, ctx->has_pops ? 1 : 0};
  const int64_t cnt[4] = {ctx->steps, ctx->snapshot_step, ctx->rebase_step, ctx->origin_step};
  put(kCkptMagic, 8);
  put(hdr, sizeof hdr);
  put(cnt, sizeof cnt);
  for (const auto& d : ctx->desc) {
    const int32_t sh[2] = {d.nx, d.ny};
    put(sh, sizeof sh);
  }
  std::vector<char> buf;
  for (int ch = 0; ch < ctx->nchan && ok; ++ch) {
    const ChanDesc& d = ctx->desc[ch];
    const size_t nn = (size_t)d.nx * d.ny, e = ctx->elem;
    buf.resize(std::max<size_t>(27 * nn * e, (M_COUNT + 1) * nn * sizeof(double)));
    const char* lat = (const char*)ctx->lat[chan_lattice(ctx, ch)] + (size_t)d.pop_off * e;
    HIP_OR_FAIL(ctx, hipMemcpy2D(buf.data(), nn * e, lat, (size_t)d.plane * e, nn * e, 27, hipMemcpyDeviceToHost));
    put(buf.data(), 27 * nn * e);
    std::vector<double> refs(kRefStride * (size_t)d.ny);
    HIP_OR_FAIL(ctx, hipMemcpy(refs.data(), ctx->d_refs + d.ref_off, refs.size() * sizeof(double),
                               hipMemcpyDeviceToHost));
    put(refs.data(), refs.size() * sizeof(double));
    std::vector<float> kn(BLK_STRIDE * (size_t)d.nb * d.ny);
    HIP_OR_FAIL(ctx, hipMemcpy(kn.data(), ctx->d_blocks + d.blk_off, kn.size() * sizeof(float),
                               hipMemcpyDeviceToHost));
    put(kn.data(), kn.size() * sizeof(float));
    double* fb = reinterpret_cast<double*>(buf.data());
    HIP_OR_FAIL(ctx, hipMemcpy(fb, ctx->d_psi + d.fld_off, nn * sizeof(double), hipMemcpyDeviceToHost));
    for (int k = 0; k < M_COUNT; ++k)
      HIP_OR_FAIL(ctx, hipMemcpy(fb + (k + 1) * nn, ctx->d_macro + k * ctx->total_nodes + d.fld_off,
                                 nn * sizeof(double), hipMemcpyDeviceToHost));
    put(fb, (M_COUNT + 1) * nn * sizeof(double));
    for (int a = 0; a < 6; ++a) put(&ctx->walls[a * (size_t)ctx->total_nx + d.wall_off], d.nx * sizeof(double));
    HIP_OR_FAIL(ctx, hipMemcpy(fb, ctx->d_ux_prev + d.fld_off, nn * sizeof(double), hipMemcpyDeviceToHost));
    put(fb, nn * sizeof(double));
  }
  if (!ok) return fail(ctx, EKPNP_ERR_IO, std::string("short write to ") + path);
  return EKPNP_OK;
}

int ekpnp_load_checkpoint(ekpnp_ctx* ctx, const char* path) {
  const ApiRange range_("ekpnp_load_checkpoint");
  if (!ctx || !path) return EKPNP_ERR_INVALID;
  HIP_OR_FAIL(ctx, hipSetDevice(ctx->opt.device));
  HIP_OR_FAIL(ctx, hipStreamSynchronize(ctx->stream));
  FILE* fp = std::fopen(path, "rb");
  if (!fp) return fail(ctx, EKPNP_ERR_IO, std::string("cannot open ") + path);
  FileCloser closer{fp};
  auto get = [&](void* p, size_t n) { return std::fread(p, 1, n, fp) == n; };
  char magic[8];
  int32_t hdr[4];
  int64_t cnt[4];
  if (!get(magic, 8) || std::memcmp(magic, kCkptMagic, 8) != 0 || !get(hdr, sizeof hdr) || !get(cnt, sizeof cnt))
    return fail(ctx, EKPNP_ERR_IO, "not a checkpoint file");
  if (hdr[0] != ctx->nchan || hdr[1] != ctx->opt.precision)
    return fail(ctx, EKPNP_ERR_INVALID, "checkpoint channel count or precision differs from the context");
  for (const auto& d : ctx->desc) {
    int32_t sh[2];
    if (!get(sh, sizeof sh)) return fail(ctx, EKPNP_ERR_IO, "truncated checkpoint");
    if (sh[0] != d.nx || sh[1] != d.ny) return fail(ctx, EKPNP_ERR_INVALID, "checkpoint channel shape differs");
  }
  // every channel's state goes to lattice cur
  for (auto& d : ctx->desc) {
    d.swap = 0;
    d.active = 1;
  }
  HIP_OR_FAIL(ctx, sync_desc(ctx));
  std::vector<char> buf;
  for (int ch = 0; ch < ctx->nchan; ++ch) {
    const ChanDesc& d = ctx->desc[ch];
    const size_t nn = (size_t)d.nx * d.ny, e = ctx->elem;
    buf.resize(std::max<size_t>(27 * nn * e, (M_COUNT + 1) * nn * sizeof(double)));
    if (!get(buf.data(), 27 * nn * e)) return fail(ctx, EKPNP_ERR_IO, "truncated checkpoint");
    char* lat = (char*)ctx->lat[ctx->cur] + (size_t)d.pop_off * e;
    HIP_OR_FAIL(ctx, hipMemcpy2D(lat, (size_t)d.plane * e, buf.data(), nn * e, nn * e, 27, hipMemcpyHostToDevice));
    std::vector<double> refs(kRefStride * (size_t)d.ny);
    if (!get(refs.data(), refs.size() * sizeof(double))) return fail(ctx, EKPNP_ERR_IO, "truncated checkpoint");
    HIP_OR_FAIL(ctx, hipMemcpy(ctx->d_refs + d.ref_off, refs.data(), refs.size() * sizeof(double),
                               hipMemcpyHostToDevice));
    std::vector<float> kn(BLK_STRIDE * (size_t)d.nb * d.ny);
    if (!get(kn.data(), kn.size() * sizeof(float))) return fail(ctx, EKPNP_ERR_IO, "truncated checkpoint");
    HIP_OR_FAIL(ctx, hipMemcpy(ctx->d_blocks + d.blk_off, kn.data(), kn.size() * sizeof(float),
                               hipMemcpyHostToDevice));
    double* fb = reinterpret_cast<double*>(buf.data());
    if (!get(fb, (M_COUNT + 1) * nn * sizeof(double))) return fail(ctx, EKPNP_ERR_IO, "truncated checkpoint");
    HIP_OR_FAIL(ctx, hipMemcpy(ctx->d_psi + d.fld_off, fb, nn * sizeof(double), hipMemcpyHostToDevice));
    for (int k = 0; k < M_COUNT; ++k)
      HIP_OR_FAIL(ctx, hipMemcpy(ctx->d_macro + k * ctx->total_nodes + d.fld_off, fb + (k + 1) * nn,
                                 nn * sizeof(double), hipMemcpyHostToDevice));
    for (int a = 0; a < 6; ++a) {
      double* w = &ctx->walls[a * (size_t)ctx->total_nx + d.wall_off];
      if (!get(w, d.nx * sizeof(double))) return fail(ctx, EKPNP_ERR_IO, "truncated checkpoint");
      HIP_OR_FAIL(ctx, hipMemcpy(ctx->d_walls + a * (size_t)ctx->total_nx + d.wall_off, w, d.nx * sizeof(double),
                                 hipMemcpyHostToDevice));
    }
    if (!get(fb, nn * sizeof(double))) return fail(ctx, EKPNP_ERR_IO, "truncated checkpoint");
    HIP_OR_FAIL(ctx, hipMemcpy(ctx->d_ux_prev + d.fld_off, fb, nn * sizeof(double), hipMemcpyHostToDevice));
  }
  ctx->state_q = hdr[2] != 0;
  ctx->has_pops = hdr[3] != 0;
  ctx->has_fields = true;
  ctx->steps = cnt[0];
  ctx->snapshot_step = cnt[1];
  ctx->rebase_step = cnt[2];
  ctx->origin_step = cnt[3];
  return EKPNP_OK;
}

int ekpnp_copy_bandwidth(int device, size_t bytes, int reps, int grid, double* gbps_out, double* ms_out) {
  const ApiRange range_("ekpnp_copy_bandwidth");
  if (!gbps_out || reps < 1 || grid < 1 || bytes < 16 || bytes % 16 != 0) return EKPNP_ERR_INVALID;
  if (hipSetDevice(device) != hipSuccess) return EKPNP_ERR_HIP;
  void* a = nullptr;
  void* b = nullptr;
  hipStream_t st = nullptr;
  hipEvent_t ev[2] = {nullptr, nullptr};
  int rc = EKPNP_OK;
  if (hipMalloc(&a, bytes) != hipSuccess || hipMalloc(&b, bytes) != hipSuccess) rc = EKPNP_ERR_NOMEM;
  if (rc == EKPNP_OK && (hipStreamCreateWithFlags(&st, hipStreamNonBlocking) != hipSuccess ||
                         hipEventCreate(&ev[0]) != hipSuccess || hipEventCreate(&ev[1]) != hipSuccess ||
                         hipMemsetAsync(a, 0, bytes, st) != hipSuccess))
    rc = EKPNP_ERR_HIP;
  const long long n = (long long)(bytes / 16);
  float ms = 0.0f;
  if (rc == EKPNP_OK) {
    // one untimed copy, then reps timed ones
    hipError_t e = launch_copy_nt(a, b, n, grid, st);
    if (e == hipSuccess) e = hipEventRecord(ev[0], st);
    for (int r = 0; r < reps && e == hipSuccess; ++r) e = launch_copy_nt(a, b, n, grid, st);
    if (e == hipSuccess) e = hipEventRecord(ev[1], st);
    if (e == hipSuccess) e = hipEventSynchronize(ev[1]);
    if (e == hipSuccess) e = hipEventElapsedTime(&ms, ev[0], ev[1]);
    if (e != hipSuccess) rc = EKPNP_ERR_HIP;
  }
  if (rc == EKPNP_OK) {
    const double per = (double)ms / reps;
    *gbps_out = 2.0 * (double)bytes / (per * 1e-3) / 1e9;
    if (ms_out) *ms_out = per;
  }
  for (auto e : ev)
    if (e) (void)hipEventDestroy(e);
  if (st) (void)hipStreamDestroy(st);
  if (a) (void)hipFree(a);
  if (b) (void)hipFree(b);
  return rc;
}

int ekpnp_num_channels(const ekpnp_ctx* ctx) { return ctx ? ctx->nchan : 0; }
long long ekpnp_steps_done(const ekpnp_ctx* ctx) { return ctx ? ctx->steps : 0; }
size_t ekpnp_device_bytes(const ekpnp_ctx* ctx) { return ctx ? ctx->dev_bytes : 0; }

int ekpnp_time_stages(ekpnp_ctx* ctx, int nsteps, double* ms_out) {
  const ApiRange range_("ekpnp_time_stages");
  if (!ctx || !ms_out || nsteps <= 0) return EKPNP_ERR_INVALID;
  if (!ctx->has_pops) return fail(ctx, EKPNP_ERR_STATE, "no populations");
  HIP_OR_FAIL(ctx, hipSetDevice(ctx->opt.device));
  if (ctx->state_q) {
    int rc = ekpnp_step(ctx, 1);
    if (rc) return rc;
  }
  hipEvent_t ev[5];
  for (int i = 0; i < 5; ++i) HIP_OR_FAIL(ctx, hipEventCreate(&ev[i]));
  double acc[4] = {0, 0, 0, 0};
  int rc = EKPNP_OK;
  for (int it = 0; it < nsteps && rc == EKPNP_OK; ++it) {
    // the step as the graphs enqueue it (wall tiles on the tridiagonal
    // launch when the plan puts them there)
    hipError_t e = hipEventRecord(ev[0], ctx->stream);
    if (e == hipSuccess) e = enqueue_step(ctx, false, ev + 1);
    if (e == hipSuccess) e = hipEventSynchronize(ev[4]);
    if (e != hipSuccess) {
      rc = fail(ctx, EKPNP_ERR_HIP, std::string("time_stages: ") + hipGetErrorString(e));
      break;
    }
    for (int k = 0; k < 4; ++k) {
      float ms = 0.f;
      (void)hipEventElapsedTime(&ms, ev[k], ev[k + 1]);
      acc[k] += ms;
    }
    ctx->steps++;
  }
  if (rc == EKPNP_OK) {
    for (int k = 0; k < 4; ++k) ms_out[k] = acc[k] / nsteps;
    // graph replay: untimed first (twice for odd nsteps, which ends on the
    // other lattice parity) so that capture and instantiation of these
    // graphs stay out of the timed replay
    for (int w = 0; w < 1 + (nsteps & 1) && rc == EKPNP_OK; ++w) rc = ekpnp_step(ctx, nsteps);
  }
  if (rc == EKPNP_OK) {
    hipError_t e = hipEventRecord(ev[0], ctx->stream);
    long long s0 = ctx->steps;
    if (e == hipSuccess) rc = ekpnp_step(ctx, nsteps);
    ctx->steps = s0 + nsteps;
    if (rc == EKPNP_OK) {
      e = hipEventRecord(ev[1], ctx->stream);
      if (e == hipSuccess) e = hipEventSynchronize(ev[1]);
      float ms = 0.f;
      if (e == hipSuccess) e = hipEventElapsedTime(&ms, ev[0], ev[1]);
      if (e != hipSuccess) rc = fail(ctx, EKPNP_ERR_HIP, std::string("time_stages: ") + hipGetErrorString(e));
      ms_out[4] = ms / nsteps;
    }
  }
  for (int i = 0; i < 5; ++i) (void)hipEventDestroy(ev[i]);
  return rc;
}

}  // extern "C"
