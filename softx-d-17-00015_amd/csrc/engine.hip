// Host orchestration and the C ABI (include/opf.h).
//
// One opf_ctx holds a resolution class: the host mesh, FFT plans, and the
// device arrays of `capacity` slots.  The time loop of main.f90:18-46 runs as
// a sequence of "iterations", each one nonlinear evaluation plus one
// predictor or corrector (per slot, as the slot's control block says):
//   k_zfwd -> k_theta -> k_zbwd -> k_step
// (k_step ends with the curl for the next evaluation).  The corrector test
// (tim_check_cgce) runs in k_step's last workgroup on the device, so the host only enqueues
// iterations and checks progress between chunks.
#include <hip/hip_runtime.h>
#include <dlfcn.h>

#include <algorithm>
#include <cmath>
#include <cstdlib>
#include <cstdio>
#include <cstring>
#include <fstream>
#include <map>
#include <mutex>
#include <sstream>
#include <stdexcept>
#include <string>
#include <vector>

#include "../../include/opf.h"
#include "kernels.hpp"
#include "engine_internal.hpp"

using namespace opf;

namespace {

thread_local std::string g_err;

struct OpfError : std::runtime_error {
  int code;
  OpfError(int c, const std::string& m) : std::runtime_error(m), code(c) {}
};

#define HIPCHK(x)                                                                        \
  do {                                                                                   \
    hipError_t e_ = (x);                                                                 \
    if (e_ != hipSuccess)                                                                \
      throw OpfError(OPF_ERR_HIP, std::string(#x) + ": " + hipGetErrorString(e_));       \
  } while (0)

template <typename F> int guard(F&& f) {
  try {
    f();
    return OPF_OK;
  } catch (const OpfError& e) {
    g_err = e.what();
    return e.code;
  } catch (const std::exception& e) {
    g_err = e.what();
    return OPF_ERR_ARG;
  }
}

size_t round_up(size_t v, size_t a) { return (v + a - 1) / a * a; }

struct Timing {
  bool on = false;
  struct Rec { std::string name; hipEvent_t a, b; };
  std::vector<Rec> recs;
  std::vector<hipEvent_t> pool;
  hipEvent_t get() {
    if (!pool.empty()) { hipEvent_t e = pool.back(); pool.pop_back(); return e; }
    hipEvent_t e;
    HIPCHK(hipEventCreate(&e));
    return e;
  }
};

}  // namespace

struct opf_ctx {
  int N, K, M, Mp, H, Hp, P, Z, T, cap;
  int diag_cap = 256;
  HostMesh mesh;
  hipStream_t stream = nullptr;
  double* d_mesh = nullptr;
  Bufs B{};
  Geo G{};
  FftTiles tiles{};
  StepTiles st{};              // launches of several slots
  StepTiles st1{};             // and of one, which leaves the chip emptier

  FftKerns fk{};
  PlaneKern plane = nullptr;   // whole-plane evaluation, where the grid has one
  size_t smem_plane = 0;
  std::vector<void*> allocs;
  size_t bytes = 0;
  std::vector<int> occupied;   // slot holds a state
  std::vector<int> setup;      // slot matrices built
  struct Adapt { int on = 0; double maxdt = 1e99, courant = 0.5; };
  std::vector<Adapt> adapt;    // d_timestep < 0, d_maxdt, d_courant per slot
  int n_adaptive = 0;          // slots with the adaptive time step on
  std::vector<int> symm;       // symmetry bits per slot (SlotParams::symm)
  int n_symm = 0;              // slots with a symmetry imposed
  std::vector<double> alpha_h; // d_alpha per slot (host copy of SlotParams::alpha)
  struct Cor { int on = 0; double Ek0 = 0.0, phi = 0.0; };
  std::vector<Cor> cor;        // coriolis.in per slot (Coriolis.f90:36-39)
  struct NN { int on = 0; double rho = 0, radius = 0, mu0 = 0, muinf = 0, lam = 0, n = 0, a = 0; };
  std::vector<NN> nn;          // params_model.in per slot (nonnewtonian.f90:67-86)
  int n_nn = 0;                // slots with the non-Newtonian viscosity on
  std::vector<double> Re_h;    // d_Re per slot (host copy of SlotParams::Re)
  struct LES { int on = 0, model = 1, filter = 1; double Cs = 0, Aplus = 0; };
  std::vector<LES> les;        // params_model.in per slot (LES.f90:70-95)
  int n_les = 0;               // slots with the LES eddy viscosity on
  double* lesD = nullptr;      // per slot [Delta, Delta_r, L_theta, coef] x N
  unsigned long long* lesMax = nullptr;   // per slot nu_max (bit pattern)
  double* nnP = nullptr;       // non-Newtonian physical fields (16 of N*Z*T), first use
  double2* nnC = nullptr;      // non-Newtonian coll temporaries (9 of coll), first use
  double2* nnY = nullptr;      // their z-transform intermediates (9 fields), first use
  // granular transform temporaries (allocated on first use)
  double2* tY = nullptr;
  double* tP = nullptr;
  double2* tC = nullptr;
  double2* shiftTab = nullptr;   // var_coll_shift tables, (2K + M) per slot (first use)
  double* normBuf = nullptr;     // opf_var_coll_norm: field, partials and sums (first use)
  double* stage[2] = {nullptr, nullptr};   // pinned pieces of fields on their way to or from the host (first use)
  hipEvent_t stage_ev[2] = {nullptr, nullptr};
  double* dterrHost = nullptr;   // pinned: tim_dterr of the last host-driven call (first use)
  SlotParams* prmHost = nullptr; // pinned parameters of asynchronous admissions (first use)
  std::vector<LuFactors> lu;     // LAPACK-form factors [slot][4] (first use)
  long mat_gen = 1;              // counts the launches that may change a factor set
  std::vector<long> lu_gen;      // its value when the factors of a set [slot][4] were last asked for
  int* luVerdict = nullptr;      // tim_lumesh_init: a zero pivot; blocks that cannot represent the set (pinned, first use)
  std::vector<int> lu_unsafe;    // the latter per factor set [slot][4]
  int n_unsafe = 0;              // and how many
  std::vector<int> lu_bc;        // BC of each factor set [slot][4] (tim_lumesh_invert's (0,0) rule)
  int device = 0;                // HIP device of the context
  // launch modes of the time loop: one iteration captured as a HIP graph
  // and replayed; iterations of a run's tail over the list of slots still
  // active (compaction)
  int use_graph = 0, use_compact = 1;   // use_graph: iterations per captured graph (0: eager)
  int use_streams = 2;           // streams a run's slots are split over (1 or 2; table or choose_streams)
  hipStream_t stream2 = nullptr; // the second stream of a split run (first use)
  hipEvent_t ev_fork = nullptr, ev_join = nullptr;
  int* smapDev = nullptr;        // compacted slot list on the device [cap]
  std::vector<int> smapHost;     // its host copy (what the device holds)
  struct GraphKey {
    int s0 = -1, ns = 0, symm = 0, adapt = 0, banded = 0, iters = 0;
    const int* smap = nullptr;
    bool operator==(const GraphKey& o) const {
      return s0 == o.s0 && ns == o.ns && symm == o.symm && adapt == o.adapt && banded == o.banded &&
             iters == o.iters && smap == o.smap;
    }
  } gkey;
  hipGraphExec_t gexec = nullptr;
  long graph_launches = 0, graph_captures = 0, compact_iterations = 0;
  Timing tm;

  template <typename T> T* alloc(size_t n) {
    void* p = nullptr;
    const size_t b = round_up(std::max<size_t>(n, 1) * sizeof(T), 256);
    HIPCHK(hipMalloc(&p, b));
    // the context's streams are non-blocking: they do not wait for this fill,
    // which runs on the null stream and may outlast the call
    HIPCHK(hipMemset(p, 0, b));
    HIPCHK(hipStreamSynchronize(nullptr));
    allocs.push_back(p);
    bytes += b;
    return (T*)p;
  }
};

namespace {

// -------------------------------------------------------------------------
// shapes
// -------------------------------------------------------------------------
struct Shape {
  int H, Hp, P, Z, T;
  size_t coll;
};
Shape shape_of(int N, int K, int M) {
  Shape s;
  s.H = (2 * K - 1) * M - (K - 1);
  s.Hp = (int)round_up((size_t)s.H, 64);
  s.P = K * M;
  s.Z = 3 * K;
  s.T = 3 * M;
  s.coll = (size_t)N * s.Hp;
  return s;
}

size_t bytes_needed(int N, int K, int M, int cap, int diag_cap) {
  const Shape s = shape_of(N, K, M);
  size_t b = 0;
  const size_t c3 = (size_t)cap * 3 * s.coll * sizeof(double2);
  b += c3 * 6;                                               // U[3], Nraw[2], om
  b += (size_t)cap * 4 * s.P * blk_count(N) * 16 * sizeof(double);   // SE
  b += (size_t)cap * 6 * N * s.P * sizeof(double);           // Uinf
  b += (size_t)cap * 16 * s.H * sizeof(double);              // Ainv
  b += (size_t)cap * 3 * s.Hp * sizeof(double);              // diagb
  b += (size_t)cap * 3 * N * sizeof(unsigned long long);     // cflmax
  b += (size_t)cap * arrive_words(s.P) * sizeof(unsigned long long);
  b += (size_t)cap * diag_cap * sizeof(DiagRec);
  b += (size_t)cap * N * ((s.Z + 3) / 4 * 4) * 9 * M * sizeof(double2);   // Yf + Yb
  return b;
}

FftTiles choose_tiles(int Z, int T, int M) {
  FftTiles t{};
  t.pz = make_plan(Z);
  t.pt = make_plan(T);
  // a workgroup transforms at most FFT_TILE complex values: tm columns of
  // length Z, or 3*tz packed lines of length T
  if (Z > FFT_TILE || T > THETA_MAX) throw OpfError(OPF_ERR_ARG, "transform length too large for the FFT tiles");
  t.tm = std::max(1, std::min(M, tile_m(Z)));
  t.tz = std::max(1, std::min(Z, FFT_TILE / (3 * T)));
  if (t.tz == 1 && Z >= 2 && 2 * T <= THETA_ITEMS) t.tz = 2;   // long theta lines
  return t;
}

// Tuned launch shapes.  The autotuner (opf/autotune.py) times the fused step
// kernel's pairs per workgroup and the transforms' tile widths per (N, K, M,
// capacity) on the device and writes the fastest into a table, tuning.tsv
// beside libopf.so, or the file OPF_TUNING names (OPF_TUNING=none: no table).
// Rows: N K M min_capacity pairs tm tz graph [measured figures]; '#' starts
// a comment; graph = iterations per captured HIP graph (0: eager launches).
// A context takes the row of its (N, K, M) with the largest min_capacity not
// above its capacity; a zero leaves that shape to the built-in choice.  The tuner
// lets a row hold below twice the capacity it was measured at and follows it
// with one of zeros from there: the shapes depend on how full the slots make the
// chip.
struct Tuned {
  int gp = 0, tm = 0, tz = 0, graph = 0, streams = 0;
};
std::string tuning_path() {
  if (const char* e = std::getenv("OPF_TUNING")) return std::string(e);
  Dl_info info;
  if (dladdr((void*)&tuning_path, &info) && info.dli_fname) {
    const std::string lib(info.dli_fname);
    const size_t k = lib.rfind('/');
    return (k == std::string::npos ? std::string(".") : lib.substr(0, k)) + "/tuning.tsv";
  }
  return std::string();
}
Tuned lookup_tuning(int N, int K, int M, int cap) {
  Tuned t;
  const std::string path = tuning_path();
  if (path.empty() || path == "none") return t;
  std::ifstream f(path);
  std::string line;
  int best = -1;
  while (std::getline(f, line)) {
    if (line.empty() || line[0] == '#') continue;
    std::istringstream is(line);
    int n, k, m, cmin, gp, tm, tz, graph;
    if (!(is >> n >> k >> m >> cmin >> gp >> tm >> tz >> graph)) continue;
    // an optional ninth integer column: streams (a token with a '.' is the
    // first timing column of a row without it)
    std::string tok;
    int streams = 0;
    if (is >> tok && tok.find('.') == std::string::npos) streams = std::atoi(tok.c_str());
    if (n == N && k == K && m == M && cmin <= cap && cmin > best) {
      best = cmin;
      t.gp = gp;
      t.tm = tm;
      t.tz = tz;
      t.graph = std::max(0, std::min(64, graph));
      t.streams = streams == 1 || streams == 2 ? streams : 0;
    }
  }
  return t;
}

size_t step_smem(int N, int gp) { return round_up(step_lds_doubles(N, gp) * sizeof(double), 16); }

// Pairs per workgroup of the fused step kernel.  Two pairs where their
// workgroups are all resident at once (three per CU; up to N = 32, where the
// kernel is short, one per CU), otherwise four (N <= 96), which write longer
// runs of each field's rows and need half the rounds.  us per launch with two
// and four, and workgroups of two per CU: (48,48,32) 23.6 24.8, 3; (64,48,32)
// 27.8 28.1, 3; (64,64,36) 42.9 35.0, 4.5; (64,64,48) 48.9 37.1, 6; (80,48,32)
// 32.5 35.0, 3; (96,64,48) 84.9 77.4, 6; (32,24,12) 13.1 13.8, 0.6; (32,32,24)
// 16.6 15.9, 1.5.
StepTiles choose_step_tiles(int N, int P, int cap, int ncu, int gp_req, size_t lds_max) {
  StepTiles t{};
  int gp = gp_req;
  if (gp <= 0)
    gp = (N <= 96 && step_smem(N, 4) <= lds_max && (long long)((P + 1) / 2) * cap > (N <= 32 ? 1LL : 3LL) * ncu) ? 4 : 2;
  if (gp != 1 && gp != 2 && gp != 4) throw OpfError(OPF_ERR_ARG, "step pairs per workgroup must be 1, 2 or 4");
  if (gp == 4 && N > 96) throw OpfError(OPF_ERR_ARG, "four pairs per workgroup need N <= 96");
  t.gp = gp;
  t.ngroups = (P + gp - 1) / gp;
  t.smem = step_smem(N, gp);
  if (t.smem > lds_max) throw OpfError(OPF_ERR_ARG, "step kernel tiles do not fit in LDS");
  return t;
}

// Streams of a run over many slots: two where the slots have more than four step
// workgroups per CU, so that either half fills the chip; one where the halves
// would only leave it emptier.  Time with one stream over two, and workgroups per
// CU: (16,6,4) 16 and 256 slots 0.67, 0.75 and 1.03, 6; (24,16,8) 16, 32 and 64
// slots 0.85, 2; 0.94, 4 and 1.02, 8; (32,24,12) 8 and 16 slots 0.93, 2.3 and
// 1.13, 4.5; (64,32,24) 4 and 8 slots 0.98, 3 and 1.04, 6; (48,48,24) 4 slots 1.05,
// 4.5; (64,64,48) 4 slots 1.04, 12.
int choose_streams(const StepTiles& st, int cap, int ncu) { return (long long)st.ngroups * cap > 4LL * ncu ? 2 : 1; }

void check_slot(opf_ctx* c, int slot) {
  if (!c) throw OpfError(OPF_ERR_ARG, "null context");
  if (slot < 0 || slot >= c->cap) throw OpfError(OPF_ERR_ARG, "slot out of range");
}

std::vector<SlotCtl> read_ctl(opf_ctx* c) {
  std::vector<SlotCtl> v(c->cap);
  HIPCHK(hipStreamSynchronize(c->stream));
  HIPCHK(hipMemcpy(v.data(), c->B.ctl, sizeof(SlotCtl) * c->cap, hipMemcpyDeviceToHost));
  return v;
}
void write_ctl(opf_ctx* c, const std::vector<SlotCtl>& v) {
  HIPCHK(hipMemcpy(c->B.ctl, v.data(), sizeof(SlotCtl) * c->cap, hipMemcpyHostToDevice));
}

// Launch helper with optional event timing.
template <typename Kern, typename... Args>
void launch(opf_ctx* c, const char* name, Kern k, dim3 grid, dim3 block, size_t smem, Args... args) {
  hipEvent_t a = nullptr, b = nullptr;
  if (c->tm.on) {
    a = c->tm.get();
    b = c->tm.get();
    HIPCHK(hipEventRecord(a, c->stream));
  }
  hipLaunchKernelGGL(k, grid, block, smem, c->stream, args...);
  HIPCHK(hipGetLastError());
  if (c->tm.on) {
    HIPCHK(hipEventRecord(b, c->stream));
    c->tm.recs.push_back({name, a, b});
  }
}

dim3 grid_h(opf_ctx* c, int nslots) { return dim3((c->H + 63) / 64, 1, nslots); }
// k_curl's blocks: (64-harmonic block, n) tiles rounded up to 8 XCDs
dim3 grid_hn(opf_ctx* c, int nslots) {
  const int ntile = ((c->H + 63) / 64) * c->N;
  return dim3(8 * ((ntile + 7) / 8), 1, nslots);
}
// blocks of k_zfwd_t / k_zbwd_t: their (m tile, n, field) tiles, 6 or 3
// fields, rounded up to 8 XCDs
unsigned ztile_blocks(const opf_ctx* c, int nfield) {
  const int gx = (c->M + c->fk.t.tm - 1) / c->fk.t.tm;
  return (unsigned)(8 * ((gx * nfield * c->N + 7) / 8));
}

// vel_transform's z transforms; the theta transforms, products and the way back
void launch_zfwd(opf_ctx* c, int s0, int ns) {
  launch(c, "zfwd", c->fk.zfwd, dim3(ztile_blocks(c, 6), 1, ns), dim3(c->fk.zn), c->fk.zfs, c->G, c->B, c->fk.t, s0);
}
void launch_back(opf_ctx* c, int s0, int ns) {
  const int gz = (c->Z + c->fk.t.tz - 1) / c->fk.t.tz;
  launch(c, "theta", c->fk.theta, dim3(8 * ((gz * c->N + 7) / 8), 1, ns), dim3(c->fk.tn), c->fk.ts, c->G,
         c->B, c->fk.t, s0);
  launch(c, "zbwd", c->fk.zbwd, dim3(ztile_blocks(c, 3), 1, ns), dim3(c->fk.zn), c->fk.zbs, c->G, c->B, c->fk.t, s0);
}

// One evaluation (vel_transform + vel_nonlinear without the base-flow
// terms) for slots [s0, s0+ns).
void launch_eval(opf_ctx* c, int s0, int ns) {
  if (c->plane) {   // one workgroup per radial plane, the intermediates in LDS
    launch(c, "plane", c->plane, dim3(c->N, 1, ns), dim3(PLANE_THREADS), c->smem_plane, c->G, c->B, c->fk.t, s0);
    return;
  }
  launch_zfwd(c, s0, ns);
  launch_back(c, s0, ns);
}

void set_unsafe(opf_ctx* c, int slot, int which, int unsafe) {
  int& u = c->lu_unsafe[(size_t)slot * 4 + which];
  c->n_unsafe += unsafe - u;
  u = unsafe;
}
void launch_step(opf_ctx* c, int s0, int ns) {
  if (c->n_unsafe > 0) {   // a slot holds a set that needs the banded LU
    const StepTiles st{1, c->P, step_smem(c->N, 1)};
    launch(c, "step", step_kernel_banded(), dim3(8 * ((c->P + 7) / 8), 1, ns), dim3(step_threads(1)), st.smem, c->G, c->B,
           st, s0);
    return;
  }
  const StepTiles& st = ns == 1 ? c->st1 : c->st;
  const int per = (st.ngroups + 7) / 8;   // XCD-aware order inside the kernel
  launch(c, "step", step_kernel(c->N, st.gp), dim3(8 * per, 1, ns), dim3(step_threads(st.gp)), st.smem, c->G, c->B, st, s0);
}

// vel_matrices for slots s0 .. s0+ns-1 of B, c->B unless the launch is of a slot
// whatever list c->B.smap holds (gate: k_matrices_t)
void launch_matrices(opf_ctx* c, int s0, int ns, int gate, const Bufs& B) {
  ++c->mat_gen;
  launch(c, "matrices", matrices_kernel(c->N), dim3((c->P + 7) / 8, 1, ns), dim3(256), matrices_smem(c->N), c->G, B,
         s0, gate);
}
void launch_matrices(opf_ctx* c, int s0, int ns, int gate) { launch_matrices(c, s0, ns, gate, c->B); }

// One iteration.  With adaptive slots, the predictor's evaluation is
// followed by vel_maxtstep + tim_new_tstep and, where dt changed,
// vel_matrices (main.f90:24-29), all decided on the device.
void launch_nonnewtonian(opf_ctx* c, int slot);
void launch_les(opf_ctx* c, int slot);

// slots [s0, s0 + ns) of the launch, or, in a compacted launch, entries
// s0 .. s0 + ns - 1 of the host copy of the slot list
void launch_iteration(opf_ctx* c, int s0, int ns) {
  if (c->n_symm > 0) {   // vel_imposesym at the start of a step (main.f90:21), then the new curl
    launch(c, "symmetry", k_symmetry, dim3((3 * c->N * c->H + 255) / 256, 1, ns), dim3(256), 0, c->G, c->B, s0, 1);
    launch(c, "curl", k_curl, grid_hn(c, ns), dim3(64), 0, c->G, c->B, s0, 1);
  }
  launch_eval(c, s0, ns);
  if (c->n_nn > 0 || c->n_les > 0)   // var_null(2) after vel_nonlinear (main.f90:23,38)
    for (int i = s0; i < s0 + ns; ++i) {
      const int s = c->B.smap ? c->smapHost[i] : i;
      if (c->nn[s].on) launch_nonnewtonian(c, s);
      if (c->les[s].on) launch_les(c, s);
    }
  if (c->n_adaptive > 0) {
    launch_matrices(c, s0, ns, 2);
  }
  launch_step(c, s0, ns);
}

int* lu_verdict(opf_ctx* c) {
  if (!c->luVerdict) {
    HIPCHK(hipHostMalloc((void**)&c->luVerdict, 2 * sizeof(int), hipHostMallocDefault));
    c->luVerdict[0] = c->luVerdict[1] = 0;
  }
  return c->luVerdict;
}

// The LAPACK-form factors of one factor set, for tim_lumesh_get and
// tim_lumesh_invert: built from the matrix the set holds when they are asked
// for (the time step does not read them), where they are not there yet.  Buffers
// per set on first use.  A zero pivot is left in luVerdict, which only
// tim_lumesh_init looks at.
const LuFactors& lapack_factors(opf_ctx* c, int slot, int which) {
  LuFactors& L = c->lu[(size_t)slot * 4 + which];
  const size_t cols = (size_t)c->P * c->N, groups = (c->P + 15) / 16;
  if (!L.F) {   // one buffer: the factors, the versions, the pivots
    L.F = c->alloc<double>(cols * LUS + (groups + 1) / 2 + (cols + 7) / 8);
    L.built = (unsigned*)(L.F + cols * LUS);
    L.pv = (unsigned char*)(L.F + cols * LUS + (groups + 1) / 2);
    HIPCHK(hipMemcpy(&c->B.sets[(size_t)slot * 4 + which].lu, &L, sizeof L, hipMemcpyHostToDevice));
  }
  long& gen = c->lu_gen[(size_t)slot * 4 + which];
  if (gen != c->mat_gen) {   // no launch since then may have changed the set
    launch(c, "lapack_factor", k_lu_factor, dim3((unsigned)groups), dim3(64), 0, c->G, c->B, L, slot, which,
           lu_verdict(c));
    gen = c->mat_gen;
  }
  return L;
}

// n doubles per plane between the host's planes (null: skipped or zeros) and
// device memory, where they follow each other, in pieces through two pinned
// buffers: the copy of one piece runs beside the host's of the next (300 MB in
// 11 to 12 ms; straight into pageable memory they take 17, and each plane of a
// small state 70 us).
constexpr size_t STAGE = (size_t)4 << 20;
template <typename Seg>
void each_segment(size_t off, size_t len, size_t n, Seg seg) {   // doubles [off, off + len) of the planes
  while (len > 0) {
    const size_t i = off / n, o = off - i * n, m = std::min(len, n - o);
    seg(i, o, m);
    off += m;
    len -= m;
  }
}
void stage_init(opf_ctx* c) {
  for (int b = 0; b < 2; ++b) {
    if (!c->stage[b]) HIPCHK(hipHostMalloc((void**)&c->stage[b], STAGE, hipHostMallocDefault));
    if (!c->stage_ev[b]) HIPCHK(hipEventCreateWithFlags(&c->stage_ev[b], hipEventDisableTiming));
  }
}
void planes_to_host(opf_ctx* c, const double* dev, double* const* host, int np, size_t n) {
  stage_init(c);
  constexpr size_t P = STAGE / sizeof(double);
  const size_t total = (size_t)np * n;
  auto drain = [&](size_t off, int b) {
    HIPCHK(hipEventSynchronize(c->stage_ev[b]));
    const double* s = c->stage[b];
    each_segment(off, std::min(P, total - off), n, [&](size_t i, size_t o, size_t m) {
      if (host[i]) std::memcpy(host[i] + o, s, m * sizeof(double));
      s += m;
    });
  };
  int b = 0;
  for (size_t off = 0; off < total; off += P, b ^= 1) {
    HIPCHK(hipMemcpyAsync(c->stage[b], dev + off, std::min(P, total - off) * sizeof(double), hipMemcpyDeviceToHost,
                          c->stream));
    HIPCHK(hipEventRecord(c->stage_ev[b], c->stream));
    if (off > 0) drain(off - P, b ^ 1);
  }
  drain((total - 1) / P * P, b ^ 1);
}
void planes_to_dev(opf_ctx* c, double* dev, const double* const* host, int np, size_t n) {
  stage_init(c);
  constexpr size_t P = STAGE / sizeof(double);
  const size_t total = (size_t)np * n;
  int b = 0;
  for (size_t off = 0; off < total; off += P, b ^= 1) {
    if (off >= 2 * P) HIPCHK(hipEventSynchronize(c->stage_ev[b]));
    double* s = c->stage[b];
    each_segment(off, std::min(P, total - off), n, [&](size_t i, size_t o, size_t m) {
      if (host[i]) std::memcpy(s, host[i] + o, m * sizeof(double));
      else std::memset(s, 0, m * sizeof(double));
      s += m;
    });
    HIPCHK(hipMemcpyAsync(dev + off, c->stage[b], std::min(P, total - off) * sizeof(double), hipMemcpyHostToDevice,
                          c->stream));
    HIPCHK(hipEventRecord(c->stage_ev[b], c->stream));
  }
}
// nf coll fields (reference layout, planes re, im of each) <-> device rows.  The
// planes pass through slot 0's backward intermediates, which only hold values
// between two kernels of an evaluation.  Fields of up to one pinned piece stay
// there, and the kernels read and write it themselves, without a copy beside
// them: a state of (16,6,4) in 25 us instead of 40, of (32,24,12) in 56 instead
// of 74, one component of it in 49 instead of 65, of (48,48,24) in 119 instead of
// 133 (and still no slower at 9 MB).
bool direct_planes(const opf_ctx* c, int nf) { return (size_t)2 * nf * c->N * c->H * sizeof(double) <= STAGE; }
dim3 grid_planes(const opf_ctx* c, int nf) { return dim3((c->Hp + 31) / 32, (c->N + 31) / 32, nf); }
void coll_to_dev(opf_ctx* c, const double* const* planes, int nf, double2* dst, bool add) {
  const size_t n = (size_t)c->N * c->H;
  double* dev = (double*)c->B.Yb;
  if (direct_planes(c, nf)) {
    stage_init(c);
    dev = c->stage[0];
    for (int i = 0; i < 2 * nf; ++i)
      if (planes[i]) std::memcpy(dev + i * n, planes[i], n * sizeof(double));
      else std::memset(dev + i * n, 0, n * sizeof(double));
  } else {
    planes_to_dev(c, dev, planes, 2 * nf, n);
  }
  launch(c, add ? "add_rows" : "to_rows", add ? k_planes_to_rows<true> : k_planes_to_rows<false>, grid_planes(c, nf),
         dim3(256), 0, c->G, (const double*)dev, dst);
  HIPCHK(hipStreamSynchronize(c->stream));
}
void coll_to_dev(opf_ctx* c, const double* const* planes, int nf, double2* dst) { coll_to_dev(c, planes, nf, dst, false); }
void dev_to_coll(opf_ctx* c, const double2* src, int nf, double* const* planes) {
  const size_t n = (size_t)c->N * c->H;
  const bool direct = direct_planes(c, nf);
  if (direct) stage_init(c);
  double* dev = direct ? c->stage[0] : (double*)c->B.Yb;
  launch(c, "to_planes", k_rows_to_planes, grid_planes(c, nf), dim3(256), 0, c->G, src, dev);
  if (!direct) {
    planes_to_host(c, dev, planes, 2 * nf, n);
    return;
  }
  HIPCHK(hipStreamSynchronize(c->stream));
  for (int i = 0; i < 2 * nf; ++i)
    if (planes[i]) std::memcpy(planes[i], dev + i * n, n * sizeof(double));
}
void coll_to_dev(opf_ctx* c, const double* re, const double* im, double2* dst) {
  const double* planes[2] = {re, im};
  coll_to_dev(c, planes, 1, dst);
}
void dev_to_coll(opf_ctx* c, const double2* src, double* re, double* im) {
  double* planes[2] = {re, im};
  dev_to_coll(c, src, 1, planes);
}

size_t y_one(const opf_ctx* c) { return (size_t)c->N * c->G.ZQ * c->M; }   // z-transformed planes of one field
void ensure_temps(opf_ctx* c) {
  if (c->tY) return;
  c->tY = c->alloc<double2>(y_one(c));
  c->tP = c->alloc<double>((size_t)c->N * c->Z * c->T);
  c->tC = c->alloc<double2>(c->G.coll);
}

// one coll field to / from the planes Y of its z transform (nf fields)
void launch_zfwd_one(opf_ctx* c, const double2* src, double2* Y, int nf) {
  launch(c, "zfwd1", c->fk.zfwd1, dim3(ztile_blocks(c, 1), 1, nf), dim3(c->fk.zn), c->fk.zfs, c->G, c->B, c->fk.t, src,
         Y, (size_t)c->G.coll, y_one(c));
}
void launch_zbwd_one(opf_ctx* c, const double2* Y, double2* dst, int nf) {
  launch(c, "zbwd1", c->fk.zbwd1, dim3(ztile_blocks(c, 1), 1, nf), dim3(c->fk.zn), c->fk.zbs, c->G, c->B, c->fk.t, Y,
         dst, y_one(c), (size_t)c->G.coll);
}
// Transforms of nf coll fields (stride coll) to / from physical fields
// (stride N*Z*T) on device buffers for the plugins (tra_spec2phys /
// tra_phys2spec, transform.fftw3.f90:65-147), one launch per stage with the
// field as grid z; physical fields in the plugins' layout [n][z][theta].  The
// padding of the coll rows is left as it is (no kernel reads it).
dim3 grid_lines(const opf_ctx* c, int nf) { return dim3((c->Z + 2 * c->fk.bt - 1) / (2 * c->fk.bt), c->N, nf); }
void coll2phys_dev(opf_ctx* c, const double2* src, double* dst, int nf) {
  launch_zfwd_one(c, src, c->nnY, nf);
  launch(c, "c2r_lines", c->fk.c2r, grid_lines(c, nf), dim3(c->fk.ln), c->fk.c2rs, c->G, c->B, c->fk.t, c->fk.bt,
         (const double2*)c->nnY, dst, y_one(c), (size_t)c->N * c->Z * c->T);
}
void phys2coll_dev(opf_ctx* c, const double* src, double2* dst, int nf) {
  launch(c, "r2c_lines", c->fk.r2c, grid_lines(c, nf), dim3(c->fk.ln), c->fk.r2cs, c->G, c->B, c->fk.t, c->fk.bt, src,
         c->nnY, (size_t)c->N * c->Z * c->T, y_one(c));
  launch_zbwd_one(c, c->nnY, dst, nf);
}

// The variable-viscosity plugins share their transforms: the gradient
// tensor of u + U on the physical grid (into P.S), then, once nu is known on
// the grid, grad(nu) (P.g) and curl curl (u + U) (P.q), and finally the
// forcing in P.q added to the slot's raw N.
NnPhys visc_fields(opf_ctx* c) {
  ensure_temps(c);
  const size_t np = (size_t)c->N * c->Z * c->T;
  if (!c->nnP) c->nnP = c->alloc<double>(16 * np);
  if (!c->nnC) c->nnC = c->alloc<double2>(9 * c->G.coll);
  if (!c->nnY) c->nnY = c->alloc<double2>(9 * y_one(c));
  NnPhys P{};
  for (int i = 0; i < 9; ++i) P.S[i] = c->nnP + (size_t)i * np;
  P.nu = c->nnP + 9 * np;
  for (int i = 0; i < 3; ++i) P.g[i] = c->nnP + (size_t)(10 + i) * np;
  for (int i = 0; i < 3; ++i) P.q[i] = c->nnP + (size_t)(13 + i) * np;
  return P;
}
void visc_gradient(opf_ctx* c, int slot, const NnPhys& P) {
  launch(c, "nn_grad", k_nn_grad, dim3((c->H + 63) / 64, c->N, 3), dim3(64), 0, c->G, c->B, slot, c->nnC);
  coll2phys_dev(c, c->nnC, P.S[0], 9);   // A(row, j), S[0..8] one after another
}
void visc_derivatives(opf_ctx* c, int slot, const NnPhys& P) {
  double2* c6 = c->nnC;
  double2* nuc = c->nnC + 6 * c->G.coll;
  const dim3 gh((c->H + 63) / 64, c->N), b64(64);
  phys2coll_dev(c, P.nu, nuc, 1);
  launch(c, "nn_gradp", k_nn_gradp, gh, b64, 0, c->G, c->B, slot, (const double2*)nuc, c6);
  launch(c, "nn_curlcurl", k_nn_curlcurl, gh, b64, 0, c->G, c->B, slot, c6 + 3 * c->G.coll);
  coll2phys_dev(c, c6, P.g[0], 6);   // g[0..2] and q[0..2] one after another
}
void visc_add(opf_ctx* c, int slot, const NnPhys& P) {
  double2* c3 = c->nnC;
  phys2coll_dev(c, P.q[0], c3, 3);
  launch(c, "nn_addN", k_nn_addN, dim3((c->H + 63) / 64, c->N, 3), dim3(64), 0, c->G, c->B, slot, (const double2*)c3);
}

// util(2) of the non-Newtonian plugin for one slot: get_nu and
// update_nonlin_terms (nonnewtonian.f90:93-244) on the slot's current
// evaluation, vel_nu = 1.
void launch_nonnewtonian(opf_ctx* c, int slot) {
  const NnPhys P = visc_fields(c);
  const size_t np = (size_t)c->N * c->Z * c->T;
  visc_gradient(c, slot, P);
  const opf_ctx::NN& q = c->nn[slot];
  const double lam = c->Re_h[slot] * q.lam * q.mu0 / (q.rho * (q.radius * q.radius));   // lam_ (:77)
  const dim3 gp((unsigned)((np + 255) / 256)), b256(256);
  launch(c, "nn_visc", k_nn_visc, gp, b256, 0, P, np, lam, q.muinf / q.mu0, -q.n / q.a, q.a);
  visc_derivatives(c, slot, P);
  launch(c, "nn_force", k_nn_force, gp, b256, 0, P, np, 1.0, c->Re_h[slot]);
  visc_add(c, slot, P);
}

// util(2) of the LES plugin for one slot (LES.f90:100-320): get_nu with the
// slot's eddy-viscosity model, update_nu_r before a predictor (vel_matrices
// on the device where vel_nu changed), update_nonlin_terms.
void launch_les(opf_ctx* c, int slot) {
  const NnPhys P = visc_fields(c);
  const size_t np = (size_t)c->N * c->Z * c->T;
  if (!c->lesD) c->lesD = c->alloc<double>((size_t)c->cap * 4 * c->N);
  if (!c->lesMax) c->lesMax = c->alloc<unsigned long long>(c->cap);
  double* D = c->lesD + (size_t)slot * 4 * c->N;
  const opf_ctx::LES& q = c->les[slot];
  visc_gradient(c, slot, P);
  launch(c, "les_prep", k_les_prep, dim3(1), dim3(64), 0, c->G, c->B, slot, q.model, q.Cs, q.Aplus, D, c->lesMax);
  const double dz = (2.0 * D_PI / (c->alpha_h[slot] * (double)c->Z)) * (3.0 / 2.0);
  const dim3 gp((unsigned)((np + 255) / 256)), b256(256);
  launch(c, "les_visc", k_les_visc, gp, b256, 0, P, np, c->N, c->Z * c->T, q.model, q.Cs, dz, (const double*)D,
         c->lesMax + slot);
  launch(c, "les_nur", k_les_nur, dim3(1), dim3(1), 0, c->B, slot, (const unsigned long long*)c->lesMax);
  Bufs B = c->B;
  B.smap = nullptr;   // `slot` is a slot, also in a compacted iteration
  launch_matrices(c, slot, 1, 1, B);
  visc_derivatives(c, slot, P);
  launch(c, "les_force", k_les_force, gp, b256, 0, P, np, c->B, slot);
  visc_add(c, slot, P);
}

// The filter lengths of init_params_model and Smagorinsky (LES.f90:81-89,
// 199-206) for the slot's alpha, uploaded once.
void les_geometry(opf_ctx* c, int slot) {
  if (!c->lesD) c->lesD = c->alloc<double>((size_t)c->cap * 4 * c->N);
  const int N = c->N;
  const std::vector<double>& r = c->mesh.r;
  const opf_ctx::LES& q = c->les[slot];
  const double Rdth = (2.0 * D_PI / (double)(c->Mp * c->T)) * (3.0 / 2.0);
  const double dz = (2.0 * D_PI / (c->alpha_h[slot] * (double)c->Z)) * (3.0 / 2.0);
  std::vector<double> h((size_t)4 * N, 0.0);
  double* Delta = h.data();
  double* Dr = h.data() + N;
  double* Lt = h.data() + 2 * N;
  Dr[0] = (r[1] - 0.0) / 2.0;
  for (int n = 1; n < N - 1; ++n) Dr[n] = (r[n + 1] - r[n - 1]) / 2.0;
  Dr[N - 1] = 1.0 - r[N - 2];
  for (int n = 0; n < N; ++n) {
    if (q.filter == 1) Delta[n] = std::pow(Dr[n] * Rdth * dz, 1.0 / 3.0);
    else if (q.filter == 2) Delta[n] = std::pow(Dr[n] * r[n] * Rdth * dz, 1.0 / 3.0);
    else Delta[n] = std::sqrt((Dr[n] * Dr[n] + (r[n] * Rdth) * (r[n] * Rdth) + dz * dz) / 3.0);
    Lt[n] = q.filter == 2 ? r[n] * Rdth : Rdth;   // Vreman's azimuthal length (:229-230)
  }
  HIPCHK(hipMemcpy(c->lesD + (size_t)slot * 4 * N, h.data(), h.size() * sizeof(double), hipMemcpyHostToDevice));
}

std::vector<double2> twiddles(int L) {
  std::vector<double2> tw(L);
  const long double pi = 3.141592653589793238462643383279502884L;
  for (int q = 0; q < L; ++q) {
    const long double a = 2.0L * pi * (long double)q / (long double)L;
    tw[q] = make_double2((double)cosl(a), (double)sinl(a));
  }
  return tw;
}

// gp_req, tm_req, tz_req > 0 fix the launch shapes (the autotuner's
// candidates); 0 takes OPF_STEP_GP, then the tuning table, then the defaults.
void create(opf_ctx* c, int N, int K, int M, int Mp, int cap, const double* r, int gp_req, int tm_req,
            int tz_req) {
  if (N < 9 || N > MAXN) throw OpfError(OPF_ERR_ARG, "N must be in [9, 128]");
  if (K < 2 || M < 1 || Mp < 1 || cap < 1) throw OpfError(OPF_ERR_ARG, "bad K, M, Mp or capacity");
  if (M > 256) throw OpfError(OPF_ERR_ARG, "M must be <= 256");
  int ndev = 0;
  if (hipGetDeviceCount(&ndev) != hipSuccess || ndev < 1) throw OpfError(OPF_ERR_HIP, "no HIP device");
  c->N = N; c->K = K; c->M = M; c->Mp = Mp; c->cap = cap;
  const Shape s = shape_of(N, K, M);
  c->H = s.H; c->Hp = s.Hp; c->P = s.P; c->Z = s.Z; c->T = s.T;
  build_mesh(N, r, c->mesh);
  c->tiles = choose_tiles(c->Z, c->T, M);
  const Tuned tuned = lookup_tuning(N, K, M, cap);
  c->use_graph = tuned.graph;
  {
    // narrower transform tiles than the defaults (the kernels hold at most
    // the default width) from the caller or the table
    const int tm = tm_req > 0 ? tm_req : tuned.tm;
    const int tz = tz_req > 0 ? tz_req : tuned.tz;
    const int tz_run = fft_kernels(c->tiles.pz, c->tiles.pt, c->tiles, M).t.tz;   // the width that runs by default
    if (tm > 0) {
      if (tm > c->tiles.tm) throw OpfError(OPF_ERR_ARG, "z tile wider than the kernels hold");
      c->tiles.tm = tm;
    }
    if (tz > 0 && tz != c->tiles.tz && tz == tz_run) {
      c->tiles.tz = tz;
    } else if (tz > 0 && tz != c->tiles.tz) {
      // the theta kernel transforms N_z of z-lines 2q and 2q + 1 together; an
      // even tile keeps those partners (and so the rounding) of the default
      if (tz > c->tiles.tz) throw OpfError(OPF_ERR_ARG, "theta tile wider than the kernels hold");
      if (tz % 2 != 0 || c->tiles.tz % 2 != 0) throw OpfError(OPF_ERR_ARG, "theta tile must be even");
      c->tiles.tz = tz;
    }
  }
  {
    const char* e1 = std::getenv("OPF_STEP_GP");
    int dev = 0, ncu = 0, lds = 0;
    HIPCHK(hipGetDevice(&dev));
    c->device = dev;
    HIPCHK(hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, dev));
    HIPCHK(hipDeviceGetAttribute(&lds, hipDeviceAttributeMaxSharedMemoryPerBlock, dev));
    const int gp = gp_req > 0 ? gp_req : e1 ? std::atoi(e1) : 0;
    c->st = choose_step_tiles(N, c->P, cap, ncu, gp > 0 ? gp : tuned.gp, (size_t)lds);
    c->st1 = choose_step_tiles(N, c->P, 1, ncu, gp > 0 ? gp : lookup_tuning(N, K, M, 1).gp, (size_t)lds);
    c->use_streams = tuned.streams > 0 ? tuned.streams : choose_streams(c->st, cap, ncu);
    for (const StepTiles* t : {&c->st, &c->st1})
      if (t->smem > 64 * 1024)   // dynamic LDS beyond 64 KiB is requested per kernel
        HIPCHK(hipFuncSetAttribute((const void*)step_kernel(N, t->gp), hipFuncAttributeMaxDynamicSharedMemorySize,
                                   (int)t->smem));
    // the whole-plane evaluation where the grid has one and its LDS fits
    // (OPF_PLANE=0: the three transform kernels instead)
    const char* e2 = std::getenv("OPF_PLANE");
    c->plane = plane_kernel(c->Z, c->T, &c->smem_plane);
    if (c->plane && ((e2 && std::atoi(e2) == 0) || c->smem_plane > (size_t)lds)) c->plane = nullptr;
    if (c->plane && c->smem_plane > 64 * 1024)
      HIPCHK(hipFuncSetAttribute((const void*)c->plane, hipFuncAttributeMaxDynamicSharedMemorySize,
                                 (int)c->smem_plane));
  }
  c->fk = fft_kernels(c->tiles.pz, c->tiles.pt, c->tiles, M);
  const std::pair<const void*, size_t> lds_of[] = {
      {(const void*)c->fk.zfwd, c->fk.zfs},  {(const void*)c->fk.zfwd1, c->fk.zfs}, {(const void*)c->fk.zbwd, c->fk.zbs},
      {(const void*)c->fk.zbwd1, c->fk.zbs}, {(const void*)c->fk.theta, c->fk.ts},  {(const void*)c->fk.c2r, c->fk.c2rs},
      {(const void*)c->fk.r2c, c->fk.r2cs}};
  for (const auto& k : lds_of)
    if (k.second > 64 * 1024)
      HIPCHK(hipFuncSetAttribute(k.first, hipFuncAttributeMaxDynamicSharedMemorySize, (int)k.second));
  HIPCHK(hipStreamCreateWithFlags(&c->stream, hipStreamNonBlocking));
  // device mesh block
  const MeshOff mo = MeshOff::make(N);
  std::vector<double> hm(mo.total, 0.0);
  const HostMesh& me = c->mesh;
  for (int n = 0; n < N; ++n) {
    hm[mo.r + n] = me.r[n];
    hm[mo.rinv + n] = me.rinv[n];
    hm[mo.rinv2 + n] = me.rinv2[n];
    hm[mo.Ubase + n] = 1.0 - me.r2[n];        // vel_U = 1 - r^2 (velocity.f90:53)
    hm[mo.twor + n] = -(-2.0 * me.r[n]);      // -vel_Up, vel_Up = -2r (velocity.f90:54, 342)
    hm[mo.intrdr + n] = me.intrdr[n];
  }
  std::copy(me.dr1b.begin(), me.dr1b.end(), hm.begin() + mo.dr1b);
  std::copy(me.lapb.begin(), me.lapb.end(), hm.begin() + mo.lapb);
  std::copy(me.dr0.begin(), me.dr0.end(), hm.begin() + mo.dr0);
  std::copy(me.dr1.begin(), me.dr1.end(), hm.begin() + mo.dr1);
  for (int n = 0; n < N; ++n) {
    for (int dd = -KL; dd <= KL; ++dd)
      if (n + dd >= 0 && n + dd < N) {
        hm[mo.lapT + 10 * n + dd + KL] = me.lapb[(size_t)(KL - dd) * N + n + dd];
        hm[mo.d1T + 10 * n + dd + KL] = me.dr1b[(size_t)(KL - dd) * N + n + dd];
      }
    hm[mo.d1T + 10 * n + 9] = me.rinv[n];
    hm[mo.rowv + n] = hm[mo.Ubase + n];
    hm[mo.rowv + N + n] = hm[mo.twor + n];
    hm[mo.rowv + 2 * N + n] = hm[mo.rinv2 + n];
  }
  c->d_mesh = c->alloc<double>(mo.total);
  HIPCHK(hipMemcpy(c->d_mesh, hm.data(), hm.size() * sizeof(double), hipMemcpyHostToDevice));

  Bufs& B = c->B;
  const size_t c3 = (size_t)cap * 3 * s.coll;
  for (int i = 0; i < 3; ++i) B.U[i] = c->alloc<double2>(c3);
  for (int i = 0; i < 2; ++i) B.Nraw[i] = c->alloc<double2>(c3);
  B.om = c->alloc<double2>(c3);
  B.SE = c->alloc<double>((size_t)cap * 4 * s.P * blk_count(N) * 16);
  struct SlotSets {   // one buffer: an allocation takes about 0.1 ms
    FactorSet sets[4];
    LuSpec spec[4];
  };
  B.sets = (FactorSet*)c->alloc<SlotSets>(cap);
  B.spec = (LuSpec*)(B.sets + (size_t)cap * 4);
  B.Uinf = c->alloc<double>((size_t)cap * 6 * N * s.P);
  B.Ainv = c->alloc<double>((size_t)cap * 16 * s.H);
  B.Ui = c->alloc<double>((size_t)cap * N);
  B.diagb = c->alloc<double>((size_t)cap * 3 * s.Hp);
  B.cflmax = c->alloc<unsigned long long>((size_t)cap * 3 * N);
  B.arrive = c->alloc<unsigned long long>((size_t)cap * arrive_words(s.P));
  B.diag = c->alloc<DiagRec>((size_t)cap * c->diag_cap);
  B.prm = c->alloc<SlotParams>(cap);
  B.ctl = c->alloc<SlotCtl>(cap);
  B.Yf = c->alloc<double2>((size_t)cap * N * ((s.Z + 3) / 4 * 4) * 6 * M);
  B.Yb = c->alloc<double2>((size_t)cap * N * ((s.Z + 3) / 4 * 4) * 3 * M);
  B.twZ = c->alloc<double2>(s.Z);
  B.twT = c->alloc<double2>(s.T);
  B.smap = nullptr;
  c->smapDev = c->alloc<int>(cap);
  auto tz = twiddles(s.Z), tt = twiddles(s.T);
  HIPCHK(hipMemcpy(B.twZ, tz.data(), tz.size() * sizeof(double2), hipMemcpyHostToDevice));
  HIPCHK(hipMemcpy(B.twT, tt.data(), tt.size() * sizeof(double2), hipMemcpyHostToDevice));

  Geo& G = c->G;
  G.N = N; G.K = K; G.M = M; G.Mp = Mp; G.H = s.H; G.Hp = s.Hp; G.P = s.P; G.Z = s.Z; G.T = s.T; G.ZQ = (s.Z + 3) / 4 * 4;
  G.coll = s.coll;
  G.mesh = c->d_mesh;

  std::vector<SlotCtl> ctl(cap);
  for (int i = 0; i < cap; ++i) {
    SlotCtl& k = ctl[i];
    std::memset(&k, 0, sizeof(k));
    k.ubase = 2; k.ucur = 0; k.unext = 1;
    k.ncur = 0; k.npred = 1;
    k.target_steps = -1;
    k.diag_cap = c->diag_cap;
    k.lasterr = 1e99;
  }
  write_ctl(c, ctl);
  c->occupied.assign(cap, 0);
  c->setup.assign(cap, 0);
  c->lu.assign((size_t)cap * 4, LuFactors{});
  c->lu_gen.assign((size_t)cap * 4, 0);
  c->lu_unsafe.assign((size_t)cap * 4, 0);
  c->lu_bc.assign((size_t)cap * 4, 0);
  for (int i = 0; i < cap; ++i) c->lu_bc[(size_t)i * 4 + MAT_LNP] = 1;
  c->adapt.assign(cap, opf_ctx::Adapt{});
  c->symm.assign(cap, 0);
  c->alpha_h.assign(cap, 0.0);
  c->cor.assign(cap, opf_ctx::Cor{});
  c->nn.assign(cap, opf_ctx::NN{});
  c->les.assign(cap, opf_ctx::LES{});
  c->Re_h.assign(cap, 0.0);
}

// The Coriolis parameters of Coriolis.f90:49-50, 58: Ro = Re Ek0, d1 = -1/(4 Ro).
void set_coriolis(SlotParams& p, const opf_ctx::Cor& k) {
  p.coriolis = k.on;
  p.cor_d1 = k.on ? -1.0 / (4.0 * (p.Re * k.Ek0)) : 0.0;
  p.cor_sphi = k.on ? std::sin(k.phi) : 0.0;
  p.cor_cphi = k.on ? std::cos(k.phi) : 0.0;
}

void slot_setup(opf_ctx* c, int slot, double Re, double alpha, double dt, double implicit, int cf) {
  check_slot(c, slot);
  if (!(dt > 0.0) || !(Re > 0.0) || alpha == 0.0) throw OpfError(OPF_ERR_ARG, "Re, dt must be > 0 and alpha != 0");
  SlotParams p{};
  p.Re = Re; p.alpha = alpha; p.dt = dt; p.implicit = implicit; p.nu = 1.0;   // vel_nu (velocity.f90:51)
  if (c->setup[slot] && c->les[slot].on) {   // vel_nu as update_nu_r left it
    HIPCHK(hipStreamSynchronize(c->stream));
    SlotParams old{};
    HIPCHK(hipMemcpy(&old, c->B.prm + slot, sizeof(old), hipMemcpyDeviceToHost));
    p.nu = old.nu;
  }
  p.dterr_tol = 1e-5;   // d_dterr (parameters.f90:40)
  p.courant = c->adapt[slot].courant;   // d_courant (parameters.f90:41)
  p.const_flux = cf;
  p.adaptive = c->adapt[slot].on;        // d_timestep < 0 (parameters.f90:38)
  p.maxdt = c->adapt[slot].maxdt;        // d_maxdt (parameters.f90:39)
  p.symm = c->symm[slot];                // b_mirrorsym, b_shiftrefl, b_shiftrott
  set_coriolis(p, c->cor[slot]);
  HIPCHK(hipMemcpy(c->B.prm + slot, &p, sizeof(p), hipMemcpyHostToDevice));
  c->alpha_h[slot] = alpha;
  c->Re_h[slot] = Re;
  if (c->les[slot].on) les_geometry(c, slot);
  auto ctl = read_ctl(c);
  ctl[slot].status = 0;
  write_ctl(c, ctl);
  launch_matrices(c, slot, 1, 0);
  for (int q = 0; q < 4; ++q) set_unsafe(c, slot, q, 0);
  ctl = read_ctl(c);
  if (ctl[slot].status != 0) {
    const int st = ctl[slot].status;
    ctl[slot].status = 0;
    write_ctl(c, ctl);
    throw OpfError(OPF_ERR_SINGULAR, st < 110 ? "tim_lumesh_init: singular factor"
                                              : (st == 110 ? "vel_adjustFlux: err 2" : "matrix inversion error"));
  }
  c->setup[slot] = 1;
}

void put_state(opf_ctx* c, int slot, const double* const* f, double t) {
  check_slot(c, slot);
  if (!c->setup[slot]) throw OpfError(OPF_ERR_STATE, "slot not set up (opf_slot_setup)");
  auto ctl = read_ctl(c);
  SlotCtl& k = ctl[slot];
  double2* u = c->B.U[k.ucur] + (size_t)slot * 3 * c->G.coll;
  coll_to_dev(c, f, 3, u);
  k.step = 0;
  k.t = t;
  k.mode = MODE_PRED;
  k.it = 0;
  k.ncorr = 0;
  k.status = 0;
  k.ndiag = 0;
  k.active = 1;
  k.corr_dt = 0.0;   // tim_corr_dt, tim_cfl_dt and tim_new_tstep's counter of a fresh run
  k.cfl_dt = 0.0;
  k.cfl_dir = 0;
  k.ntc = 0;
  k.refactor = 0;
  write_ctl(c, ctl);
  launch(c, "imposesym", k_imposesym, dim3((c->N + 63) / 64, 1, 1), dim3(64), 0, c->G, c->B, slot);
  launch(c, "curl0", k_curl, grid_hn(c, 1), dim3(64), 0, c->G, c->B, slot, 0);
  HIPCHK(hipStreamSynchronize(c->stream));
  ctl = read_ctl(c);
  ctl[slot].active = 0;
  write_ctl(c, ctl);
  c->occupied[slot] = 1;
}

}  // namespace

// ---- the device-resident loop in phases (also used by the server) --------
namespace opf {

RunPlan run_begin(opf_ctx* c, const std::vector<int>& slots, const std::vector<int>& nsteps,
                  const std::vector<int>& corr_fixed, int diag_every, bool strict) {
  if (slots.size() != nsteps.size() || slots.size() != corr_fixed.size())
    throw OpfError(OPF_ERR_ARG, "run plan: size mismatch");
  auto ctl = read_ctl(c);
  RunPlan p;
  int lo = c->cap, hi = -1;
  for (size_t i = 0; i < slots.size(); ++i) {
    const int s = slots[i];
    check_slot(c, s);
    if (!c->occupied[s]) throw OpfError(OPF_ERR_STATE, "slot holds no state");
    if (nsteps[i] < 0) throw OpfError(OPF_ERR_ARG, "nsteps < 0");
    SlotCtl& k = ctl[s];
    if (k.status != 0) {
      if (strict) throw OpfError(OPF_ERR_CORRECTOR, "slot failed earlier");
      continue;
    }
    if (nsteps[i] == 0) continue;
    k.active = 1;
    k.mode = MODE_PRED;
    k.target_steps = k.step + nsteps[i];
    // the variable-viscosity plugins set tim_pcn = 1 (nonnewtonian.f90:70, LES.f90:76)
    k.corr_fixed = (c->nn[s].on || c->les[s].on) ? 1 : corr_fixed[i];
    k.diag_every = diag_every;
    k.host_driven = 0;
    p.slots.push_back(s);
    p.max_steps = std::max(p.max_steps, nsteps[i]);
    lo = std::min(lo, s);
    hi = std::max(hi, s);
  }
  if (hi < 0) return p;
  write_ctl(c, ctl);
  p.lo = lo;
  p.ns = hi - lo + 1;
  return p;
}

// Iterations over [s0, s0 + ns) (of the slot list when c->B.smap is set):
// replays of one captured iteration where the launch sequence allows it
// (no per-slot plugin launches, no event timing), else eager launches.
void enqueue_iterations(opf_ctx* c, int s0, int ns, long iterations) {
  if (iterations <= 0 || ns <= 0) return;
  const int gi = c->use_graph;   // iterations per captured graph (0: eager launches)
  const bool graph = gi > 0 && iterations >= gi && !c->tm.on && c->n_nn == 0 && c->n_les == 0;
  if (!graph) {
    for (long i = 0; i < iterations; ++i) launch_iteration(c, s0, ns);
    return;
  }
  opf_ctx::GraphKey key;
  key.s0 = s0;
  key.ns = ns;
  key.symm = c->n_symm > 0;
  key.adapt = c->n_adaptive > 0;
  key.banded = c->n_unsafe > 0;
  key.smap = c->B.smap;
  key.iters = gi;
  if (!c->gexec || !(key == c->gkey)) {
    if (c->gexec) {
      HIPCHK(hipGraphExecDestroy(c->gexec));
      c->gexec = nullptr;
    }
    hipGraph_t g = nullptr;
    HIPCHK(hipStreamBeginCapture(c->stream, hipStreamCaptureModeThreadLocal));
    try {
      for (int i = 0; i < gi; ++i) launch_iteration(c, s0, ns);
    } catch (...) {
      (void)hipStreamEndCapture(c->stream, &g);
      if (g) (void)hipGraphDestroy(g);
      throw;
    }
    HIPCHK(hipStreamEndCapture(c->stream, &g));
    const hipError_t e = hipGraphInstantiate(&c->gexec, g, nullptr, nullptr, 0);
    (void)hipGraphDestroy(g);
    if (e != hipSuccess) {
      c->gexec = nullptr;
      throw OpfError(OPF_ERR_HIP, std::string("hipGraphInstantiate: ") + hipGetErrorString(e));
    }
    c->gkey = key;
    ++c->graph_captures;
  }
  const long reps = iterations / gi;
  ++c->mat_gen;   // replays launch what their capture did
  for (long i = 0; i < reps; ++i) HIPCHK(hipGraphLaunch(c->gexec, c->stream));
  for (long i = reps * gi; i < iterations; ++i) launch_iteration(c, s0, ns);
  c->graph_launches += reps;
}

// Iterations over two halves of [s0, s0 + ns) on two streams, so that one
// half's step kernels overlap the other half's transforms (the slots are
// independent).  The second stream first waits for the context stream's
// earlier work, and the context stream waits for the second stream's at the
// end, so every later call on the context sees both.
void enqueue_split(opf_ctx* c, int s0, int ns, long iterations) {
  if (!c->stream2) {
    HIPCHK(hipStreamCreateWithFlags(&c->stream2, hipStreamNonBlocking));
    HIPCHK(hipEventCreateWithFlags(&c->ev_fork, hipEventDisableTiming));
    HIPCHK(hipEventCreateWithFlags(&c->ev_join, hipEventDisableTiming));
  }
  const int na = ns / 2;
  HIPCHK(hipEventRecord(c->ev_fork, c->stream));
  HIPCHK(hipStreamWaitEvent(c->stream2, c->ev_fork, 0));
  hipStream_t main = c->stream;
  c->stream = c->stream2;
  try {
    for (long i = 0; i < iterations; ++i) launch_iteration(c, s0 + na, ns - na);
  } catch (...) {
    c->stream = main;
    throw;
  }
  c->stream = main;
  for (long i = 0; i < iterations; ++i) launch_iteration(c, s0, na);
  HIPCHK(hipEventRecord(c->ev_join, c->stream2));
  HIPCHK(hipStreamWaitEvent(c->stream, c->ev_join, 0));
}

void run_enqueue(opf_ctx* c, const RunPlan& p, long iterations) {
  if (p.ns == 0 || iterations <= 0) return;
  const int nl = (int)p.live.size();
  if (c->use_compact && nl > 0 && 2 * nl <= p.ns) {
    // the run's tail: only the listed slots are still active
    if (c->smapHost != p.live) {
      c->smapHost = p.live;
      HIPCHK(hipMemcpyAsync(c->smapDev, c->smapHost.data(), sizeof(int) * nl, hipMemcpyHostToDevice, c->stream));
    }
    c->B.smap = c->smapDev;
    try {
      enqueue_iterations(c, 0, nl, iterations);
    } catch (...) {
      c->B.smap = nullptr;
      throw;
    }
    c->B.smap = nullptr;
    c->compact_iterations += iterations;
    return;
  }
  // two streams for runs over many slots without per-slot plugin launches
  if (c->use_streams > 1 && p.ns >= 4 && !c->tm.on && c->n_nn == 0 && c->n_les == 0) {
    enqueue_split(c, p.lo, p.ns, iterations);
    return;
  }
  enqueue_iterations(c, p.lo, p.ns, iterations);
}

hipStream_t ctx_stream(opf_ctx* c) { return c->stream; }

// slot's part of the backward intermediates: the planes of an idle slot pass
// through it
static double* slot_planes(opf_ctx* c, int slot) { return (double*)(c->B.Yb + (size_t)slot * c->N * c->G.ZQ * 3 * c->M); }

void admit_async(opf_ctx* c, int slot, double Re, double alpha, double dt, int ucur, const double* planes,
                 int nsteps, int corr_fixed) {
  check_slot(c, slot);
  if (!(dt > 0.0) || !(Re > 0.0) || alpha == 0.0) throw OpfError(OPF_ERR_ARG, "Re, dt must be > 0 and alpha != 0");
  if (ucur < 0 || ucur > 2 || nsteps < 1 || corr_fixed < 0) throw OpfError(OPF_ERR_ARG, "bad admission");
  if (c->n_nn || c->n_les || c->n_adaptive || c->n_symm) throw OpfError(OPF_ERR_STATE, "plain slots only");
  if (!c->prmHost) HIPCHK(hipHostMalloc((void**)&c->prmHost, sizeof(SlotParams) * c->cap, hipHostMallocDefault));
  SlotParams& p = c->prmHost[slot];
  std::memset(&p, 0, sizeof p);
  p.Re = Re; p.alpha = alpha; p.dt = dt; p.implicit = 0.51; p.nu = 1.0;   // velocity.f90:51
  p.dterr_tol = 1e-5;
  p.courant = 0.5;
  p.const_flux = 1;
  p.maxdt = 1e99;
  c->alpha_h[slot] = alpha;
  c->Re_h[slot] = Re;
  hipLaunchKernelGGL(k_admit, dim3(1), dim3(1), 0, c->stream, c->B, slot, 0, 0, 0);
  HIPCHK(hipGetLastError());
  HIPCHK(hipMemcpyAsync(c->B.prm + slot, &p, sizeof p, hipMemcpyHostToDevice, c->stream));
  launch_matrices(c, slot, 1, 0);
  double* dev = slot_planes(c, slot);
  HIPCHK(hipMemcpyAsync(dev, planes, sizeof(double) * 6 * c->N * c->H, hipMemcpyHostToDevice, c->stream));
  launch(c, "to_rows", k_planes_to_rows<false>, grid_planes(c, 3), dim3(256), 0, c->G, (const double*)dev,
         c->B.U[ucur] + (size_t)slot * 3 * c->G.coll);
  launch(c, "imposesym", k_imposesym, dim3((c->N + 63) / 64, 1, 1), dim3(64), 0, c->G, c->B, slot);
  hipLaunchKernelGGL(k_admit, dim3(1), dim3(1), 0, c->stream, c->B, slot, 1, nsteps, corr_fixed);
  HIPCHK(hipGetLastError());
  launch(c, "curl0", k_curl, grid_hn(c, 1), dim3(64), 0, c->G, c->B, slot, 0);
  c->setup[slot] = 1;
  c->occupied[slot] = 1;
}

void enqueue_iteration_range(opf_ctx* c, int s0, int ns) { launch_iteration(c, s0, ns); }

void ctl_snapshot_async(opf_ctx* c, SlotCtl* out) {
  HIPCHK(hipMemcpyAsync(out, c->B.ctl, sizeof(SlotCtl) * c->cap, hipMemcpyDeviceToHost, c->stream));
}

void fetch_async(opf_ctx* c, int slot, int ucur, double* planes) {
  check_slot(c, slot);
  double* dev = slot_planes(c, slot);
  launch(c, "to_planes", k_rows_to_planes, grid_planes(c, 3), dim3(256), 0, c->G,
         (const double2*)(c->B.U[ucur] + (size_t)slot * 3 * c->G.coll), dev);
  HIPCHK(hipMemcpyAsync(planes, dev, sizeof(double) * 6 * c->N * c->H, hipMemcpyDeviceToHost, c->stream));
}

int run_remaining(opf_ctx* c, RunPlan& p) {
  p.live.clear();
  if (p.ns == 0) return 0;
  auto ctl = read_ctl(c);
  int remaining = 0;
  for (int s : p.slots)
    if (ctl[s].active) {
      remaining = std::max(remaining, std::max(1, ctl[s].target_steps - ctl[s].step));
      p.live.push_back(s);
    }
  return remaining;
}

}  // namespace opf

namespace {

void run_plan(opf_ctx* c, const std::vector<int>& slots, const std::vector<int>& nsteps,
              const std::vector<int>& corr_fixed, int diag_every) {
  RunPlan p = run_begin(c, slots, nsteps, corr_fixed, diag_every, true);
  if (p.ns == 0) return;
  // Most steps take one corrector; enqueue 2 iterations per step, then top
  // up until every slot has reached its target.  A step takes at most 11
  // iterations (a predictor and tim_check_cgce's 10 correctors), or fails.
  const long budget = 11L * p.max_steps + 2;
  long enqueued = 0;
  long chunk = std::min(budget, 2L * p.max_steps);
  int remaining = 1;
  while (chunk > 0) {
    run_enqueue(c, p, chunk);
    enqueued += chunk;
    remaining = run_remaining(c, p);
    chunk = remaining > 0 ? std::min(budget - enqueued, std::max(2L, 2L * remaining)) : 0;
  }
  auto ctl = read_ctl(c);
  for (int s : slots)
    if (ctl[s].status != 0) {
      char msg[128];
      std::snprintf(msg, sizeof msg, "tim_check_cgce failure %d in slot %d at step %d", ctl[s].status, s, ctl[s].step);
      throw OpfError(OPF_ERR_CORRECTOR, msg);
    }
  if (remaining > 0) {   // cannot happen while control_decide keeps its corrector limit; never leave slots running
    for (int s : p.slots) ctl[s].active = 0;
    write_ctl(c, ctl);
    throw OpfError(OPF_ERR_CORRECTOR, "time loop: steps left after the iteration budget");
  }
}

void run_slots(opf_ctx* c, const std::vector<int>& slots, int nsteps, int corr_fixed, int diag_every) {
  if (nsteps < 0) throw OpfError(OPF_ERR_ARG, "nsteps < 0");
  run_plan(c, slots, std::vector<int>(slots.size(), nsteps), std::vector<int>(slots.size(), corr_fixed),
           diag_every);
}

// var_coll_shift tables of slots [s0, s0 + ns) (k_shift's layout); a slot
// not in `sel` gets none.  The host's cos / sin stand for dcos / dsin.
void launch_shift(opf_ctx* c, int s0, int ns, const std::vector<int>& sel, const std::vector<double>& dth,
                  const std::vector<double>& dz) {
  const int per = 2 * c->K + c->M;
  if (!c->shiftTab) c->shiftTab = c->alloc<double2>((size_t)c->cap * per);
  std::vector<double2> tab((size_t)ns * per, make_double2(0.0, 0.0));
  bool any = false;
  for (size_t i = 0; i < sel.size(); ++i) {
    const int j = sel[i] - s0;
    double2* t = &tab[(size_t)j * per];
    t[0] = make_double2(dz[i] != 0.0 ? 1.0 : 0.0, dth[i] != 0.0 ? 1.0 : 0.0);
    any = any || dz[i] != 0.0 || dth[i] != 0.0;
    for (int k = -(c->K - 1); k <= c->K - 1; ++k) {
      const double a = dz[i] * (double)k * c->alpha_h[sel[i]];
      t[k + c->K] = make_double2(std::cos(a), std::sin(a));
    }
    for (int m = 0; m < c->M; ++m) {
      const double a = dth[i] * (double)m * (double)c->Mp;
      t[2 * c->K + m] = make_double2(std::cos(a), std::sin(a));
    }
  }
  if (!any) return;
  HIPCHK(hipStreamSynchronize(c->stream));   // no kernel still reads the previous tables
  HIPCHK(hipMemcpy(c->shiftTab, tab.data(), tab.size() * sizeof(double2), hipMemcpyHostToDevice));
  launch(c, "shift", k_shift, dim3((3 * c->N * c->H + 255) / 256, 1, ns), dim3(256), 0, c->G, c->B, s0,
         (const double2*)c->shiftTab);
}

// The end of steporbit (newton.f90:721-775) for slots `sel`: vel_imposesym
// after the last corrector, var_coll_shift by (dth, dz), and the vorticity
// of the result for the next evaluation.
void orbit_finish(opf_ctx* c, const std::vector<int>& sel, const std::vector<double>& dth,
                  const std::vector<double>& dz) {
  if (sel.empty()) return;
  int lo = c->cap, hi = -1;
  for (int s : sel) { lo = std::min(lo, s); hi = std::max(hi, s); }
  const int ns = hi - lo + 1;
  auto ctl = read_ctl(c);
  for (int s : sel) {
    ctl[s].active = 1;
    ctl[s].target_steps = -1;
  }
  write_ctl(c, ctl);
  launch(c, "symmetry", k_symmetry, dim3((3 * c->N * c->H + 255) / 256, 1, ns), dim3(256), 0, c->G, c->B, lo, 0);
  launch_shift(c, lo, ns, sel, dth, dz);
  launch(c, "curl0", k_curl, grid_hn(c, ns), dim3(64), 0, c->G, c->B, lo, 0);
  HIPCHK(hipStreamSynchronize(c->stream));
  ctl = read_ctl(c);
  for (int s : sel) ctl[s].active = 0;
  write_ctl(c, ctl);
}

}  // namespace

namespace {
// run `fn` with the slot marked active (kernels skip inactive slots); returns
// tim_dterr.  The marks are kernels on the stream: reading the control block
// back and writing it, before and after, cost more than the work of most calls
// (a host's loop over (48,48,24) took 625 us per step, 110 of it in kernels).
template <typename F> double with_active(opf_ctx* c, int slot, int mode, F&& fn) {
  check_slot(c, slot);
  if (!c->occupied[slot]) throw OpfError(OPF_ERR_STATE, "slot holds no state");
  if (!c->dterrHost) HIPCHK(hipHostMalloc((void**)&c->dterrHost, sizeof(double), hipHostMallocDefault));
  launch(c, "host_call", k_host_call, dim3(1), dim3(1), 0, c->B, slot, 1, mode, c->dterrHost);
  fn();
  launch(c, "host_call", k_host_call, dim3(1), dim3(1), 0, c->B, slot, 0, mode, c->dterrHost);
  HIPCHK(hipStreamSynchronize(c->stream));
  return *c->dterrHost;
}
}  // namespace

// =========================================================================
// C ABI
// =========================================================================
extern "C" {

const char* opf_last_error(void) { return g_err.c_str(); }
int opf_version(void) { return 100; }

static double* scratch_on(int dev);

int opf_ctx_create_tiles(opf_ctx** out, int N, int K, int M, int Mp, int capacity, const double* r, int pairs,
                         int tm, int tz) {
  return guard([&] {
    if (!out) throw OpfError(OPF_ERR_ARG, "null out");
    *out = nullptr;
    if (pairs < 0 || tm < 0 || tz < 0) throw OpfError(OPF_ERR_ARG, "negative tile size");
    auto* c = new opf_ctx();
    try {
      create(c, N, K, M, Mp, capacity, r, pairs, tm, tz);
      (void)scratch_on(c->device);   // opf_var_coll_norm_noalloc's buffer on this device
    } catch (...) {
      opf_ctx_destroy(c);
      throw;
    }
    *out = c;
  });
}

int opf_ctx_create(opf_ctx** out, int N, int K, int M, int Mp, int capacity, const double* r) {
  return opf_ctx_create_tiles(out, N, K, M, Mp, capacity, r, 0, 0, 0);
}

int opf_ctx_destroy(opf_ctx* c) {
  if (!c) return OPF_OK;
  if (c->stream) (void)hipStreamSynchronize(c->stream);
  if (c->gexec) (void)hipGraphExecDestroy(c->gexec);
  if (c->stream2) (void)hipStreamSynchronize(c->stream2);
  if (c->ev_fork) (void)hipEventDestroy(c->ev_fork);
  if (c->ev_join) (void)hipEventDestroy(c->ev_join);
  if (c->stream2) (void)hipStreamDestroy(c->stream2);
  if (c->prmHost) (void)hipHostFree(c->prmHost);
  if (c->dterrHost) (void)hipHostFree(c->dterrHost);
  if (c->luVerdict) (void)hipHostFree(c->luVerdict);
  for (int b = 0; b < 2; ++b) {
    if (c->stage[b]) (void)hipHostFree(c->stage[b]);
    if (c->stage_ev[b]) (void)hipEventDestroy(c->stage_ev[b]);
  }
  for (void* p : c->allocs) (void)hipFree(p);
  for (auto& r : c->tm.recs) { (void)hipEventDestroy(r.a); (void)hipEventDestroy(r.b); }
  for (auto e : c->tm.pool) (void)hipEventDestroy(e);
  if (c->stream) (void)hipStreamDestroy(c->stream);
  delete c;
  return OPF_OK;
}

int opf_ctx_dims(const opf_ctx* c, int* N, int* K, int* M, int* Mp, int* H, int* cap, size_t* bytes) {
  return guard([&] {
    if (!c) throw OpfError(OPF_ERR_ARG, "null context");
    if (N) *N = c->N;
    if (K) *K = c->K;
    if (M) *M = c->M;
    if (Mp) *Mp = c->Mp;
    if (H) *H = c->H;
    if (cap) *cap = c->cap;
    if (bytes) *bytes = c->bytes;
  });
}

size_t opf_ctx_bytes_needed(int N, int K, int M, int capacity) { return bytes_needed(N, K, M, capacity, 256); }

namespace {
void mesh_out(const HostMesh& me, double* r, double* intrdr, double* dr0, double* dr1, double* dr1band,
              double* radlap) {
  const int N = me.N;
    if (r) std::copy(me.r.begin(), me.r.end(), r);
    if (intrdr) std::copy(me.intrdr.begin(), me.intrdr.end(), intrdr);
    if (dr0) std::copy(me.dr0.begin(), me.dr0.end(), dr0);
    if (dr1) std::copy(me.dr1.begin(), me.dr1.end(), dr1);
    // band [row][col] -> Fortran M(row+1, col+1) column-major: M[row + 9*col]
    for (int row = 0; row < LDA; ++row)
      for (int col = 0; col < N; ++col) {
        if (dr1band) dr1band[row + LDA * col] = me.dr1b[(size_t)row * N + col];
        if (radlap) radlap[row + LDA * col] = me.lapb[(size_t)row * N + col];
      }
}
}  // namespace

extern "C" int opf_mesh_get(const opf_ctx* c, double* r, double* intrdr, double* dr0, double* dr1,
                            double* dr1band, double* radlap) {
  return guard([&] {
    if (!c) throw OpfError(OPF_ERR_ARG, "null context");
    mesh_out(c->mesh, r, intrdr, dr0, dr1, dr1band, radlap);
  });
}

extern "C" int opf_mesh_build(int N, const double* r_in, double* r, double* intrdr, double* dr0, double* dr1,
                              double* dr1band, double* radlap) {
  return guard([&] {
    HostMesh me;
    try {
      build_mesh(N, r_in, me);
    } catch (const std::runtime_error& e) {
      throw OpfError(OPF_ERR_ARG, e.what());
    }
    mesh_out(me, r, intrdr, dr0, dr1, dr1band, radlap);
  });
}

int opf_slot_setup(opf_ctx* c, int slot, double Re, double alpha, double dt, double implicit, int cf) {
  return guard([&] { slot_setup(c, slot, Re, alpha, dt, implicit, cf); });
}

int opf_slot_adaptive(opf_ctx* c, int slot, int enable, double maxdt, double courant) {
  return guard([&] {
    check_slot(c, slot);
    if (enable && !(maxdt > 0.0 && courant > 0.0)) throw OpfError(OPF_ERR_ARG, "maxdt and courant must be > 0");
    opf_ctx::Adapt& a = c->adapt[slot];
    c->n_adaptive += (enable ? 1 : 0) - a.on;
    a.on = enable ? 1 : 0;
    if (enable) {
      a.maxdt = maxdt;
      a.courant = courant;
    }
    if (c->setup[slot]) {   // the slot's parameters on the device follow at once
      SlotParams p{};
      HIPCHK(hipMemcpy(&p, c->B.prm + slot, sizeof(p), hipMemcpyDeviceToHost));
      p.adaptive = a.on;
      p.maxdt = a.maxdt;
      p.courant = a.courant;
      HIPCHK(hipMemcpy(c->B.prm + slot, &p, sizeof(p), hipMemcpyHostToDevice));
    }
  });
}

int opf_slot_symmetry(opf_ctx* c, int slot, int mirror, int shiftrefl, int shiftrott) {
  return guard([&] {
    check_slot(c, slot);
    const int bits = (mirror ? 1 : 0) | (shiftrefl ? 2 : 0) | (shiftrott ? 4 : 0);
    c->n_symm += (bits != 0) - (c->symm[slot] != 0);
    c->symm[slot] = bits;
    if (c->setup[slot]) {
      SlotParams p{};
      HIPCHK(hipMemcpy(&p, c->B.prm + slot, sizeof(p), hipMemcpyDeviceToHost));
      p.symm = bits;
      HIPCHK(hipMemcpy(c->B.prm + slot, &p, sizeof(p), hipMemcpyHostToDevice));
    }
  });
}

int opf_slot_coriolis(opf_ctx* c, int slot, int enable, double Ek0, double phi) {
  return guard([&] {
    check_slot(c, slot);
    if (enable && c->Mp != 1) throw OpfError(OPF_ERR_ARG, "add_coriolis: i_Mp/=1");
    if (enable && !(Ek0 > 0.0)) throw OpfError(OPF_ERR_ARG, "Ek0 must be > 0");
    opf_ctx::Cor& k = c->cor[slot];
    k.on = enable ? 1 : 0;
    k.Ek0 = enable ? Ek0 : 0.0;
    k.phi = enable ? phi : 0.0;
    if (c->setup[slot]) {
      SlotParams p{};
      HIPCHK(hipMemcpy(&p, c->B.prm + slot, sizeof(p), hipMemcpyDeviceToHost));
      set_coriolis(p, k);
      HIPCHK(hipMemcpy(c->B.prm + slot, &p, sizeof(p), hipMemcpyHostToDevice));
    }
  });
}

int opf_slot_les(opf_ctx* c, int slot, int enable, int model, double C_s, int filter, double A_plus) {
  return guard([&] {
    check_slot(c, slot);
    if (enable && model != 1 && model != 2) throw OpfError(OPF_ERR_ARG, "load_params_model: unknown model");
    if (enable && (filter < 1 || filter > (model == 1 ? 3 : 2))) throw OpfError(OPF_ERR_ARG, "bad LES filter");
    if (enable && !(C_s > 0.0)) throw OpfError(OPF_ERR_ARG, "C_s must be > 0");
    opf_ctx::LES& q = c->les[slot];
    c->n_les += (enable ? 1 : 0) - q.on;
    q = opf_ctx::LES{};
    if (enable) q = opf_ctx::LES{1, model, filter, C_s, A_plus};
    if (enable && c->setup[slot]) les_geometry(c, slot);
    if (!enable && c->setup[slot]) {   // vel_nu back to 1 and the matrices with it
      SlotParams p{};
      HIPCHK(hipMemcpy(&p, c->B.prm + slot, sizeof(p), hipMemcpyDeviceToHost));
      if (p.nu != 1.0) slot_setup(c, slot, p.Re, p.alpha, p.dt, p.implicit, p.const_flux);
    }
  });
}

int opf_slot_nonnewtonian(opf_ctx* c, int slot, int enable, double rho, double radius, double mu_0,
                          double mu_inf, double lam_CY, double n_CY, double a_CY) {
  return guard([&] {
    check_slot(c, slot);
    if (enable && !(rho > 0.0 && radius > 0.0 && mu_0 > 0.0 && mu_inf >= 0.0 && lam_CY >= 0.0 && a_CY > 0.0))
      throw OpfError(OPF_ERR_ARG, "bad Carreau-Yasuda parameters");
    opf_ctx::NN& q = c->nn[slot];
    c->n_nn += (enable ? 1 : 0) - q.on;
    q = opf_ctx::NN{};
    if (enable) q = opf_ctx::NN{1, rho, radius, mu_0, mu_inf, lam_CY, n_CY, a_CY};
  });
}

int opf_slot_timestep(opf_ctx* c, int slot, double* dt, double* corr_dt, double* cfl_dt, int* cfl_dir) {
  return guard([&] {
    check_slot(c, slot);
    HIPCHK(hipStreamSynchronize(c->stream));
    SlotParams p{};
    HIPCHK(hipMemcpy(&p, c->B.prm + slot, sizeof(p), hipMemcpyDeviceToHost));
    auto ctl = read_ctl(c);
    if (dt) *dt = p.dt;
    if (corr_dt) *corr_dt = ctl[slot].corr_dt;
    if (cfl_dt) *cfl_dt = ctl[slot].cfl_dt;
    if (cfl_dir) *cfl_dir = ctl[slot].cfl_dir;
  });
}

int opf_vel_maxtstep(opf_ctx* c, int slot, double* cfl_dt, int* cfl_dir) {
  return guard([&] {
    check_slot(c, slot);
    if (!c->occupied[slot]) throw OpfError(OPF_ERR_STATE, "slot holds no state");
    launch(c, "maxtstep", k_maxtstep, dim3(1), dim3(64), 0, c->G, c->B, slot);
    HIPCHK(hipStreamSynchronize(c->stream));
    auto ctl = read_ctl(c);
    if (cfl_dt) *cfl_dt = ctl[slot].cfl_dt;
    if (cfl_dir) *cfl_dir = ctl[slot].cfl_dir;
  });
}

int opf_vel_matrices(opf_ctx* c, int slot, double dt) {
  return guard([&] {
    check_slot(c, slot);
    if (!c->setup[slot]) throw OpfError(OPF_ERR_STATE, "slot not set up (opf_slot_setup)");
    if (!(dt > 0.0)) throw OpfError(OPF_ERR_ARG, "dt must be > 0");
    SlotParams p{};
    HIPCHK(hipMemcpy(&p, c->B.prm + slot, sizeof(p), hipMemcpyDeviceToHost));
    slot_setup(c, slot, p.Re, p.alpha, dt, p.implicit, p.const_flux);
  });
}

int opf_put_state(opf_ctx* c, int slot, const double* urr, const double* uri, const double* utr,
                  const double* uti, const double* uzr, const double* uzi, double t) {
  return guard([&] {
    const double* f[6] = {urr, uri, utr, uti, uzr, uzi};
    for (auto p : f)
      if (!p) throw OpfError(OPF_ERR_ARG, "null field");
    put_state(c, slot, f, t);
  });
}

int opf_get_state(opf_ctx* c, int slot, double* urr, double* uri, double* utr, double* uti, double* uzr,
                  double* uzi, double* t) {
  return guard([&] {
    check_slot(c, slot);
    auto ctl = read_ctl(c);
    const double2* u = c->B.U[ctl[slot].ucur] + (size_t)slot * 3 * c->G.coll;
    double* f[6] = {urr, uri, utr, uti, uzr, uzi};
    dev_to_coll(c, u, 3, f);
    if (t) *t = ctl[slot].t;
  });
}

int opf_run(opf_ctx* c, int nsteps, int corr_fixed, int diag_every) {
  return guard([&] {
    if (!c) throw OpfError(OPF_ERR_ARG, "null context");
    std::vector<int> slots;
    for (int s = 0; s < c->cap; ++s)
      if (c->occupied[s]) slots.push_back(s);
    run_slots(c, slots, nsteps, corr_fixed, diag_every);
  });
}

int opf_run_slots(opf_ctx* c, const int* slots, int nslots, int nsteps, int corr_fixed, int diag_every) {
  return guard([&] {
    if (!c || (!slots && nslots > 0)) throw OpfError(OPF_ERR_ARG, "null argument");
    run_slots(c, std::vector<int>(slots, slots + nslots), nsteps, corr_fixed, diag_every);
  });
}

int opf_slot_status(opf_ctx* c, int slot, int* step, double* t, int* status, int* last_ncorr, double* last_dterr,
                    double* Pr0) {
  return guard([&] {
    check_slot(c, slot);
    auto ctl = read_ctl(c);
    const SlotCtl& k = ctl[slot];
    if (step) *step = k.step;
    if (t) *t = k.t;
    if (status) *status = k.status;
    if (last_ncorr) *last_ncorr = k.last_ncorr;
    if (last_dterr) *last_dterr = k.last_dterr;
    if (Pr0) *Pr0 = k.Pr0;
  });
}

int opf_diag_get(opf_ctx* c, int slot, double* recs, int maxrec, int* nrec) {
  return guard([&] {
    check_slot(c, slot);
    auto ctl = read_ctl(c);
    const int nd = ctl[slot].ndiag;
    const int have = std::min(nd, c->diag_cap);
    std::vector<DiagRec> all(c->diag_cap);
    HIPCHK(hipMemcpy(all.data(), c->B.diag + (size_t)slot * c->diag_cap, sizeof(DiagRec) * c->diag_cap,
                     hipMemcpyDeviceToHost));
    const int n = std::min(have, maxrec);
    const int first = nd - have + (have - n);
    for (int i = 0; i < n; ++i) {
      const DiagRec& r = all[(first + i) % c->diag_cap];
      std::memcpy(recs + 10 * i, &r, sizeof(DiagRec));
    }
    if (nrec) *nrec = n;
  });
}

// ---- granular reference procedures -----------------------------------------

int opf_vel_imposesym(opf_ctx* c, int slot) {
  return guard([&] {
    check_slot(c, slot);
    if (!c->occupied[slot]) throw OpfError(OPF_ERR_STATE, "slot holds no state");
    with_active(c, slot, -1, [&] {
      launch(c, "symmetry", k_symmetry, dim3((3 * c->N * c->H + 255) / 256, 1, 1), dim3(256), 0, c->G, c->B, slot,
             0);
      launch(c, "curl", k_curl, grid_hn(c, 1), dim3(64), 0, c->G, c->B, slot, 0);
    });
  });
}


int opf_vel_transform(opf_ctx* c, int slot) {
  return guard([&] {
    with_active(c, slot, -1, [&] {
      launch_zfwd(c, slot, 1);
    });
  });
}

int opf_vel_nonlinear(opf_ctx* c, int slot) {
  return guard([&] {
    with_active(c, slot, -1, [&] {
      launch_back(c, slot, 1);
      if (c->nn[slot].on) launch_nonnewtonian(c, slot);   // var_null(2)
      if (c->les[slot].on) launch_les(c, slot);
    });
  });
}

int opf_vel_predictor(opf_ctx* c, int slot) {
  return guard([&] { with_active(c, slot, MODE_PRED, [&] { launch_step(c, slot, 1); }); });
}

int opf_vel_corrector(opf_ctx* c, int slot, double* dterr) {
  return guard([&] {
    const double d = with_active(c, slot, MODE_CORR, [&] { launch_step(c, slot, 1); });
    if (dterr) *dterr = d;
  });
}

int opf_get_nonlinear(opf_ctx* c, int slot, double* nrr, double* nri, double* ntr, double* nti, double* nzr,
                      double* nzi) {
  // Nraw of the last evaluation plus the base-flow terms of vel_addHPF,
  // added on the host from the current iterate (velocity.f90:338-361).
  return guard([&] {
    check_slot(c, slot);
    auto ctl = read_ctl(c);
    SlotParams prm;
    HIPCHK(hipMemcpy(&prm, c->B.prm + slot, sizeof prm, hipMemcpyDeviceToHost));
    const int N = c->N, H = c->H;
    std::vector<double> f[12];
    for (auto& v : f) v.assign((size_t)N * H, 0.0);
    const double2* nr = c->B.Nraw[ctl[slot].ncur] + (size_t)slot * 3 * c->G.coll;
    const double2* u = c->B.U[ctl[slot].ucur] + (size_t)slot * 3 * c->G.coll;
    double* planes[12];
    for (int i = 0; i < 12; ++i) planes[i] = f[i].data();
    dev_to_coll(c, nr, 3, planes);
    dev_to_coll(c, u, 3, planes + 6);
    const HostMesh& me = c->mesh;
    double Pr0 = 0.0;
    for (int hh = 0; hh < H; ++hh) {
      int k, m;
      if (hh < c->K) { m = 0; k = hh; }
      else { const int q = hh - c->K; m = 1 + q / (2 * c->K - 1); k = q % (2 * c->K - 1) - (c->K - 1); }
      (void)m;
      for (int n = 0; n < N; ++n) {
        const size_t o = (size_t)hh * N + n;
        const double a = (prm.alpha * (double)k) * (1.0 - me.r2[n]);
        const double b = 2.0 * me.r[n];
        f[0][o] = f[0][o] + a * f[7][o];
        f[1][o] = f[1][o] - a * f[6][o];
        f[2][o] = f[2][o] + a * f[9][o];
        f[3][o] = f[3][o] - a * f[8][o];
        f[4][o] = (f[4][o] + a * f[11][o]) + b * f[6][o];
        f[5][o] = (f[5][o] - a * f[10][o]) + b * f[7][o];
      }
    }
    if (prm.const_flux) {
      double s = 0.0;
      for (int i = 0; i <= KL; ++i) s = s + f[10][(size_t)(N - 1 - KL + i)] * me.dr1[i + (KL + 1)];
      Pr0 = s / (-2.0);
      for (int n = 0; n < N; ++n) f[4][n] = f[4][n] + (4.0 * Pr0) / prm.Re;
    }
    double* outs[6] = {nrr, nri, ntr, nti, nzr, nzi};
    for (int i = 0; i < 6; ++i)
      if (outs[i]) std::copy(f[i].begin(), f[i].end(), outs[i]);
  });
}

// the slot's current iterate, one component, on the host (coll planes)
static void slot_field_to_host(opf_ctx* c, int slot, int comp, std::vector<double>& re, std::vector<double>& im) {
  auto ctl = read_ctl(c);
  re.assign((size_t)c->N * c->H, 0.0);
  im.assign((size_t)c->N * c->H, 0.0);
  const double2* u = c->B.U[ctl[slot].ucur] + (size_t)slot * 3 * c->G.coll + (size_t)comp * c->G.coll;
  dev_to_coll(c, u, re.data(), im.data());
}

int opf_var_norm(opf_ctx* c, int slot, int comp, double* E, double* Ek, double* Em) {
  // var_coll_norm (variables.f90:718-751): per harmonic b = (w f) . intrdr,
  // halved for (0,0); Em(m) and Ek(|k|) accumulate in harmonic order;
  // E = sum(Em)
  return guard([&] {
    check_slot(c, slot);
    if (comp < 0 || comp > 2) throw OpfError(OPF_ERR_ARG, "component must be 0, 1 or 2");
    if (!c->occupied[slot]) throw OpfError(OPF_ERR_STATE, "slot holds no state");
    SlotParams prm;
    HIPCHK(hipMemcpy(&prm, c->B.prm + slot, sizeof prm, hipMemcpyDeviceToHost));
    std::vector<double> re, im;
    slot_field_to_host(c, slot, comp, re, im);
    const int N = c->N;
    std::vector<double> ek(c->K, 0.0), em(c->M, 0.0);
    const double w = 4.0 * D_PI * D_PI / prm.alpha;
    for (int hh = 0; hh < c->H; ++hh) {
      int k, m;
      if (hh < c->K) { m = 0; k = hh; }
      else { const int q = hh - c->K; m = 1 + q / (2 * c->K - 1); k = q % (2 * c->K - 1) - (c->K - 1); }
      double b = 0.0;
      for (int n = 0; n < N; ++n) {
        const size_t o = (size_t)hh * N + n;
        const double f = w * (re[o] * re[o] + im[o] * im[o]);
        b = b + f * c->mesh.intrdr[n];
      }
      if (k == 0 && m == 0) b = 0.5 * b;
      em[m] = em[m] + b;
      ek[k < 0 ? -k : k] = ek[k < 0 ? -k : k] + b;
    }
    double e = 0.0;
    for (double v : em) e = e + v;
    if (E) *E = e;
    if (Ek) std::copy(ek.begin(), ek.end(), Ek);
    if (Em) std::copy(em.begin(), em.end(), Em);
  });
}

// var_coll_norm's two passes (k_norm_harm, k_norm_sum) on device arrays:
// the field (re, im in the coll layout), partials b[H], out[1 + K + M].
static void launch_norm(opf_ctx* c, int slot, const double* re, const double* im, double* b, double* out,
                 hipStream_t stream) {
  hipLaunchKernelGGL(k_norm_harm, dim3((c->H + 255) / 256), dim3(256), 0, stream, c->G,
                     (const SlotParams*)(c->B.prm + slot), re, im, b);
  HIPCHK(hipGetLastError());
  hipLaunchKernelGGL(k_norm_sum, dim3(1), dim3(256), 0, stream, c->G, (const double*)b, out);
  HIPCHK(hipGetLastError());
}

int opf_var_coll_norm(opf_ctx* c, int slot, const double* re, const double* im, double* E, double* Ek,
                      double* Em) {
  // var_coll_norm (variables.f90:718-751) of any coll field, with d_alpha of
  // the slot's parameters, on the device
  return guard([&] {
    check_slot(c, slot);
    if (!re || !im) throw OpfError(OPF_ERR_ARG, "null field");
    if (!c->setup[slot]) throw OpfError(OPF_ERR_STATE, "slot not set up (alpha unknown)");
    const size_t nh = (size_t)c->N * c->H, nout = 1 + (size_t)c->K + c->M;
    if (!c->normBuf) c->normBuf = c->alloc<double>(2 * nh + c->H + nout);
    double* dre = c->normBuf;
    double* dim = dre + nh;
    double* b = dim + nh;
    double* out = b + c->H;
    HIPCHK(hipMemcpyAsync(dre, re, nh * sizeof(double), hipMemcpyHostToDevice, c->stream));
    HIPCHK(hipMemcpyAsync(dim, im, nh * sizeof(double), hipMemcpyHostToDevice, c->stream));
    launch_norm(c, slot, dre, dim, b, out, c->stream);
    std::vector<double> h(nout);
    HIPCHK(hipMemcpyAsync(h.data(), out, nout * sizeof(double), hipMemcpyDeviceToHost, c->stream));
    HIPCHK(hipStreamSynchronize(c->stream));
    if (E) *E = h[0];
    if (Ek) std::copy(h.begin() + 1, h.begin() + 1 + c->K, Ek);
    if (Em) std::copy(h.begin() + 1 + c->K, h.end(), Em);
  });
}

// ---- var_coll_norm without allocation --------------------------------------
// The per-harmonic partials of opf_var_coll_norm_noalloc live in a file-scope
// device array, one copy per GPU, held until the process ends.  Host code
// never passes `scratch` itself to a kernel: its device address, looked up
// once per device with hipGetSymbolAddress (at context creation), is kept in
// g_scratch and used instead.
constexpr int NORM_SCRATCH_MAX = 65536;   // harmonics (512 KiB of doubles)
static __device__ __align__(256) double scratch[NORM_SCRATCH_MAX];

static std::mutex g_scratch_mu;
static std::map<int, double*> g_scratch;   // device -> address of its scratch

// Address of `scratch` on device `dev` (looked up with dev current).
static double* scratch_on(int dev) {
  std::lock_guard<std::mutex> lk(g_scratch_mu);
  auto it = g_scratch.find(dev);
  if (it != g_scratch.end()) return it->second;
  int cur = 0;
  HIPCHK(hipGetDevice(&cur));
  if (cur != dev) HIPCHK(hipSetDevice(dev));
  void* ptr = nullptr;
  const hipError_t e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
  if (cur != dev) (void)hipSetDevice(cur);
  if (e != hipSuccess || !ptr)
    throw OpfError(OPF_ERR_HIP, std::string("hipGetSymbolAddress(scratch): ") + hipGetErrorString(e));
  g_scratch[dev] = (double*)ptr;
  return (double*)ptr;
}

int opf_var_coll_norm_noalloc(opf_ctx* c, int slot, const double* re, const double* im, double* out,
                              void* stream) {
  // opf_var_coll_norm on device arrays; no device memory is allocated
  return guard([&] {
    check_slot(c, slot);
    if (!re || !im || !out) throw OpfError(OPF_ERR_ARG, "null device pointer");
    if (c->H > NORM_SCRATCH_MAX)
      throw OpfError(OPF_ERR_ARG, "H = " + std::to_string(c->H) + " exceeds the " +
                                      std::to_string(NORM_SCRATCH_MAX) + " harmonics of the norm scratch buffer");
    if (!c->setup[slot]) throw OpfError(OPF_ERR_STATE, "slot not set up (alpha unknown)");
    double* b = scratch_on(c->device);
    hipStream_t s = stream ? (hipStream_t)stream : c->stream;
    launch_norm(c, slot, re, im, b, out, s);
    if (!stream) HIPCHK(hipStreamSynchronize(c->stream));
  });
}

int opf_friction(opf_ctx* c, int slot, double* Ub, double* Uc, double* Ufr) {
  // io_write_friction (io.f90:627-639) on the (0,0) mode of u_z; with
  // constant flux Ub is vel_Pr0 of the current state (velocity.f90:356-357)
  return guard([&] {
    check_slot(c, slot);
    if (!c->occupied[slot]) throw OpfError(OPF_ERR_STATE, "slot holds no state");
    SlotParams prm;
    HIPCHK(hipMemcpy(&prm, c->B.prm + slot, sizeof prm, hipMemcpyDeviceToHost));
    std::vector<double> re, im;
    slot_field_to_host(c, slot, 2, re, im);
    const int N = c->N;
    const HostMesh& me = c->mesh;
    const double* uz = re.data();   // harmonic 0 occupies the first N values
    double ub = 0.0;
    if (prm.const_flux) {
      double s = 0.0;
      for (int i = 0; i <= KL; ++i) s = s + uz[N - 1 - KL + i] * me.dr1[i + (KL + 1) * 1];
      ub = s / (-2.0);
    } else {
      double s = 0.0;
      for (int n = 0; n < N; ++n) s = s + uz[n] * me.intrdr[n];
      ub = 0.5 + 2.0 * s;
    }
    double uc = 0.0;
    for (int i = 0; i <= KL; ++i) uc = uc + uz[i] * me.dr0[i];
    double f = 0.0;
    for (int i = 0; i <= KL; ++i) f = f + uz[N - 1 - KL + i] * me.dr1[i + (KL + 1) * 1];
    if (Ub) *Ub = ub;
    if (Uc) *Uc = 1.0 + uc;
    if (Ufr) *Ufr = std::sqrt(std::fabs((f - 2.0) / prm.Re));
  });
}

int opf_get_phys(opf_ctx* c, int slot, int which, double* phys) {
  // vel_r/t/z (which 0..2) and vel_curlr/t/z (3..5) of vel_transform
  // (velocity.f90:304-317) for the slot's current iterate, phys layout
  return guard([&] {
    check_slot(c, slot);
    if (which < 0 || which > 5 || !phys) throw OpfError(OPF_ERR_ARG, "which must be 0..5");
    if (!c->occupied[slot]) throw OpfError(OPF_ERR_STATE, "slot holds no state");
    ensure_temps(c);
    auto ctl = read_ctl(c);
    const double2* src = which < 3 ? c->B.U[ctl[slot].ucur] + (size_t)slot * 3 * c->G.coll + (size_t)which * c->G.coll
                                   : c->B.om + (size_t)slot * 3 * c->G.coll + (size_t)(which - 3) * c->G.coll;
    const FftTiles& t = c->tiles;
    launch_zfwd_one(c, src, c->tY, 1);
    launch(c, "c2r", k_theta_c2r, dim3((c->Z + 1) / 2, c->N, 1), dim3(FFT_THREADS),
           (padded_len(c->T) + c->T) * sizeof(double2), c->G, c->B, t, (const double2*)c->tY, c->tP);
    planes_to_host(c, c->tP, &phys, 1, (size_t)c->N * c->Z * c->T);
  });
}

int opf_add_nonlinear(opf_ctx* c, int slot, const double* nrr, const double* nri, const double* ntr,
                      const double* nti, const double* nzr, const double* nzi) {
  // var_null(2) hooks add forcing to vel_N* after vel_nonlinear
  // (Coriolis.f90:54-71); added here to the slot's current evaluation
  return guard([&] {
    check_slot(c, slot);
    if (!nrr || !ntr || !nzr) throw OpfError(OPF_ERR_ARG, "null argument");
    auto ctl = read_ctl(c);
    const double* planes[6] = {nrr, nri, ntr, nti, nzr, nzi};
    coll_to_dev(c, planes, 3, c->B.Nraw[ctl[slot].ncur] + (size_t)slot * 3 * c->G.coll, true);
  });
}

int opf_tra_coll2phys(opf_ctx* c, const double* cre, const double* cim, double* phys) {
  return guard([&] {
    if (!c || !cre || !phys) throw OpfError(OPF_ERR_ARG, "null argument");
    ensure_temps(c);
    coll_to_dev(c, cre, cim, c->tC);
    const FftTiles& t = c->tiles;
    launch_zfwd_one(c, c->tC, c->tY, 1);
    launch(c, "c2r", k_theta_c2r, dim3((c->Z + 1) / 2, c->N, 1), dim3(FFT_THREADS), (padded_len(c->T) + c->T) * sizeof(double2), c->G,
           c->B, t, (const double2*)c->tY, c->tP);
    planes_to_host(c, c->tP, &phys, 1, (size_t)c->N * c->Z * c->T);
  });
}

int opf_tra_phys2coll(opf_ctx* c, const double* phys, double* cre, double* cim) {
  return guard([&] {
    if (!c || !phys) throw OpfError(OPF_ERR_ARG, "null argument");
    ensure_temps(c);
    planes_to_dev(c, c->tP, &phys, 1, (size_t)c->N * c->Z * c->T);
    const FftTiles& t = c->tiles;
    HIPCHK(hipMemsetAsync(c->tC, 0, sizeof(double2) * c->G.coll, c->stream));
    launch(c, "r2c", k_theta_r2c, dim3((c->Z + 1) / 2, c->N, 1), dim3(FFT_THREADS), (padded_len(c->T) + c->T) * sizeof(double2), c->G,
           c->B, t, (const double*)c->tP, c->tY);
    launch_zbwd_one(c, c->tY, c->tC, 1);
    dev_to_coll(c, c->tC, cre, cim);
  });
}

int opf_tim_lumesh_get(opf_ctx* c, int slot, int which, double* ab, int* ipiv) {
  return guard([&] {
    check_slot(c, slot);
    if (which < 0 || which > 3) throw OpfError(OPF_ERR_ARG, "which must be 0..3");
    if (!c->setup[slot]) throw OpfError(OPF_ERR_STATE, "slot not set up");
    const int N = c->N, P = c->P, H = c->H;
    const LuFactors& L = lapack_factors(c, slot, which);
    // per-pair blocks [pair][n][LUS] and [pair][n]
    std::vector<double> F((size_t)P * N * LUS);
    std::vector<unsigned char> pv((size_t)P * N);
    HIPCHK(hipMemcpyAsync(F.data(), L.F, F.size() * sizeof(double), hipMemcpyDeviceToHost, c->stream));
    HIPCHK(hipMemcpyAsync(pv.data(), L.pv, pv.size(), hipMemcpyDeviceToHost, c->stream));
    HIPCHK(hipStreamSynchronize(c->stream));
    for (int hh = 0; hh < H; ++hh) {
      int k, m;
      if (hh < c->K) { m = 0; k = hh; }
      else { const int q = hh - c->K; m = 1 + q / (2 * c->K - 1); k = q % (2 * c->K - 1) - (c->K - 1); }
      const int p = m * c->K + std::abs(k);
      for (int n = 0; n < N; ++n) {
        for (int row = 0; row < NLU; ++row)
          if (ab) ab[((size_t)hh * N + n) * NLU + row] = F[((size_t)p * N + n) * LUS + row];
        if (ipiv) ipiv[(size_t)hh * N + n] = n + 1 + pv[(size_t)p * N + n];
      }
    }
  });
}

}  // extern "C"

// tim_lumesh_invert on a host field: solved on the device, lane per harmonic.
namespace opf {
__global__ void k_lumesh_invert(Geo G, LuFactors L, int bc, double2* x);
}

extern "C" int opf_tim_lumesh_invert(opf_ctx* c, int slot, int which, int BC, double* bre, double* bim) {
  return guard([&] {
    check_slot(c, slot);
    if (which < 0 || which > 3) throw OpfError(OPF_ERR_ARG, "which must be 0..3");
    if (BC > 1) throw OpfError(OPF_ERR_ARG, "BC must be 0 or 1 (negative: the matrix's own)");
    if (!c->setup[slot]) throw OpfError(OPF_ERR_STATE, "slot not set up");
    if (!bre || !bim) throw OpfError(OPF_ERR_ARG, "null field");
    const int bc = BC >= 0 ? BC : c->lu_bc[(size_t)slot * 4 + which];
    ensure_temps(c);
    const LuFactors& L = lapack_factors(c, slot, which);
    coll_to_dev(c, bre, bim, c->tC);
    launch(c, "lumesh_invert", k_lumesh_invert, grid_h(c, 1), dim3(64), 0, c->G, L, bc, c->tC);
    dev_to_coll(c, c->tC, bre, bim);
  });
}

extern "C" int opf_tim_lumesh_init(opf_ctx* c, int slot, int which, int PM, int BC, double c1, double c2) {
  // tim_lumesh_init (timestep.f90:67-96): c1 I + c2 Lap (PM = +-1: the
  // modified Laplacian of u+-), the axis parity row and the BC row, then
  // DGBTF2, for every (|k|, m) pair, into factor set `which` of the slot
  return guard([&] {
    check_slot(c, slot);
    if (which < 0 || which > 3) throw OpfError(OPF_ERR_ARG, "which must be 0..3");
    if (PM < -1 || PM > 1 || BC < 0 || BC > 1) throw OpfError(OPF_ERR_ARG, "PM must be -1, 0, 1 and BC 0 or 1");
    if (!c->setup[slot]) throw OpfError(OPF_ERR_STATE, "slot not set up (alpha unknown)");
    auto ctl = read_ctl(c);
    if (ctl[slot].status != 0) {
      ctl[slot].status = 0;
      write_ctl(c, ctl);
    }
    ++c->mat_gen;
    int* verdict = lu_verdict(c);
    verdict[0] = verdict[1] = 0;
    launch(c, "factor", k_block_factor, dim3((c->P + 31) / 32), dim3(64), 0, c->G, c->B, slot,
           LuSpec{which, PM, BC, c1, c2}, verdict + 1);
    lapack_factors(c, slot, which);   // DGBTF2's own verdict on a singular matrix
    HIPCHK(hipStreamSynchronize(c->stream));
    c->lu_bc[(size_t)slot * 4 + which] = BC;
    if (verdict[0]) throw OpfError(OPF_ERR_SINGULAR, "tim_lumesh_init");
    // a set that needs row interchanges across blocks: the slot's steps solve
    // with the LAPACK-form factors of all four sets
    const int* unsafe = &c->lu_unsafe[(size_t)slot * 4];
    const int before = unsafe[0] | unsafe[1] | unsafe[2] | unsafe[3];
    set_unsafe(c, slot, which, verdict[1]);
    const int banded = unsafe[0] | unsafe[1] | unsafe[2] | unsafe[3];
    if (!banded && !before) return;
    if (banded)
      for (int q = 0; q < 4; ++q) lapack_factors(c, slot, q);
    HIPCHK(hipStreamSynchronize(c->stream));
    HIPCHK(hipMemcpy(&c->B.sets[(size_t)slot * 4].banded, &banded, sizeof banded, hipMemcpyHostToDevice));
  });
}

extern "C" int opf_kernel_timing(opf_ctx* c, int enable) {
  return guard([&] {
    if (!c) throw OpfError(OPF_ERR_ARG, "null context");
    HIPCHK(hipStreamSynchronize(c->stream));
    for (auto& r : c->tm.recs) { c->tm.pool.push_back(r.a); c->tm.pool.push_back(r.b); }
    c->tm.recs.clear();
    c->tm.on = enable != 0;
  });
}

extern "C" int opf_launch_mode(opf_ctx* c, int graph, int compact, int streams, int* graph_now, int* compact_now,
                               int* streams_now, long long* graph_launches, long long* graph_captures,
                               long long* compact_iterations) {
  return guard([&] {
    if (!c) throw OpfError(OPF_ERR_ARG, "null context");
    if (graph > 64) throw OpfError(OPF_ERR_ARG, "at most 64 iterations per captured graph");
    if (streams > 2) throw OpfError(OPF_ERR_ARG, "at most 2 streams");
    if (graph >= 0) c->use_graph = graph;
    if (compact >= 0) c->use_compact = compact != 0;
    if (streams >= 1) c->use_streams = streams;
    if (graph_now) *graph_now = c->use_graph;
    if (compact_now) *compact_now = c->use_compact;
    if (streams_now) *streams_now = c->use_streams;
    if (graph_launches) *graph_launches = c->graph_launches;
    if (graph_captures) *graph_captures = c->graph_captures;
    if (compact_iterations) *compact_iterations = c->compact_iterations;
  });
}

extern "C" int opf_tile_config(const opf_ctx* c, int* pairs, int* tm, int* tz) {
  return guard([&] {
    if (!c) throw OpfError(OPF_ERR_ARG, "null context");
    if (pairs) *pairs = c->st.gp;
    if (tm) *tm = c->fk.t.tm;   // what the launches use: at most what the kernels of the length hold
    if (tz) *tz = c->fk.t.tz;
  });
}

extern "C" int opf_step_config(const opf_ctx* c, int* gp, int* threads, long long* lds) {
  return guard([&] {
    if (!c || !gp || !threads || !lds) throw OpfError(OPF_ERR_ARG, "null argument");
    *gp = c->st.gp;
    *threads = step_threads(c->st.gp);
    *lds = (long long)c->st.smem;
  });
}

extern "C" int opf_kernel_time(opf_ctx* c, const char* name, double* ms, int* launches) {
  return guard([&] {
    if (!c || !name) throw OpfError(OPF_ERR_ARG, "null argument");
    HIPCHK(hipStreamSynchronize(c->stream));
    double tot = 0.0;
    int cnt = 0;
    for (auto& r : c->tm.recs)
      if (r.name == name) {
        float t = 0.f;
        HIPCHK(hipEventElapsedTime(&t, r.a, r.b));
        tot += t;
        ++cnt;
      }
    if (ms) *ms = tot;
    if (launches) *launches = cnt;
  });
}

// ---- state files (io.f90) -------------------------------------------------
extern "C" int opf_state_file_info(const char* path, int* N, int* K, int* M, int* Mp, double* t, double* Re,
                                   double* alpha, double* dt) {
  return guard([&] {
    if (!path) throw OpfError(OPF_ERR_ARG, "null path");
    StateInfo s = read_state_info(path);
    if (N) *N = s.N;
    if (K) *K = s.K;
    if (M) *M = s.M;
    if (Mp) *Mp = s.Mp;
    if (t) *t = s.t;
    if (Re) *Re = s.Re;
    if (alpha) *alpha = s.alpha;
    if (dt) *dt = s.dt;
  });
}

extern "C" int opf_state_file_write(const char* path, int N, int K, int M, int Mp, const double* r, double t,
                                    double Re, double alpha, double dt, double dtcor, double dtcfl,
                                    const double* urr, const double* uri, const double* utr, const double* uti,
                                    const double* uzr, const double* uzi) {
  return guard([&] {
    const double* f[6] = {urr, uri, utr, uti, uzr, uzi};
    if (!path || !r) throw OpfError(OPF_ERR_ARG, "null argument");
    for (auto p : f)
      if (!p) throw OpfError(OPF_ERR_ARG, "null field");
    if (N <= KL || N > MAXN || K < 1 || M < 1 || Mp < 1) throw OpfError(OPF_ERR_ARG, "bad N, K, M or Mp");
    write_state_file(path, N, K, M, Mp, t, Re, alpha, dt, dtcor, dtcfl, r, f);
  });
}

extern "C" int opf_state_file_read(const char* path, int N, int K, int M, int Mp, const double* r, double* t,
                                   double* Re, double* alpha, double* dt, double* dtcor, double* dtcfl, double* urr,
                                   double* uri, double* utr, double* uti, double* uzr, double* uzi) {
  return guard([&] {
    double* f[6] = {urr, uri, utr, uti, uzr, uzi};
    if (!path) throw OpfError(OPF_ERR_ARG, "null path");
    for (auto p : f)
      if (!p) throw OpfError(OPF_ERR_ARG, "null field");
    if (N <= KL || N > MAXN || K < 1 || M < 1 || Mp < 1) throw OpfError(OPF_ERR_ARG, "bad N, K, M or Mp");
    HostMesh me;
    if (!r) build_mesh(N, nullptr, me);   // the default mesh of mes_precompute
    read_state_file(path, N, K, M, Mp, r ? r : me.r.data(), t, Re, alpha, dt, dtcor, dtcfl, f);
  });
}

extern "C" int opf_state_save(opf_ctx* c, int slot, const char* path) {
  return guard([&] {
    check_slot(c, slot);
    if (!path) throw OpfError(OPF_ERR_ARG, "null path");
    if (!c->occupied[slot]) throw OpfError(OPF_ERR_STATE, "slot holds no state");
    HIPCHK(hipStreamSynchronize(c->stream));
    SlotParams p{};
    HIPCHK(hipMemcpy(&p, c->B.prm + slot, sizeof(p), hipMemcpyDeviceToHost));
    auto ctl = read_ctl(c);
    const SlotCtl& k = ctl[slot];
    const size_t nh = (size_t)c->N * c->H;
    std::vector<double> buf(6 * nh);
    const double2* u = c->B.U[k.ucur] + (size_t)slot * 3 * c->G.coll;
    double* out[6];
    const double* f[6];
    for (int i = 0; i < 6; ++i) f[i] = out[i] = &buf[i * nh];
    dev_to_coll(c, u, 3, out);
    write_state_file(path, c->N, c->K, c->M, c->Mp, k.t, p.Re, p.alpha, p.dt, k.corr_dt, k.cfl_dt,
                     c->mesh.r.data(), f);
  });
}

extern "C" int opf_state_load(opf_ctx* c, int slot, const char* path, double t) {
  return guard([&] {
    check_slot(c, slot);
    if (!path) throw OpfError(OPF_ERR_ARG, "null path");
    if (!c->setup[slot]) throw OpfError(OPF_ERR_STATE, "slot not set up (opf_slot_setup)");
    const size_t nh = (size_t)c->N * c->H;
    std::vector<double> buf(6 * nh);
    double* f[6];
    for (int i = 0; i < 6; ++i) f[i] = &buf[i * nh];
    double tf = 0.0, dtf = 0.0, dtcor = 0.0, dtcfl = 0.0;
    read_state_file(path, c->N, c->K, c->M, c->Mp, c->mesh.r.data(), &tf, nullptr, nullptr, &dtf, &dtcor, &dtcfl,
                    f);
    if (c->adapt[slot].on && dtf > 0.0) {   // d_timestep < 0: tim_dt from the file (io.f90:145)
      SlotParams p{};
      HIPCHK(hipMemcpy(&p, c->B.prm + slot, sizeof(p), hipMemcpyDeviceToHost));
      if (p.dt != dtf) slot_setup(c, slot, p.Re, p.alpha, dtf, p.implicit, p.const_flux);
    }
    const double* cf[6] = {f[0], f[1], f[2], f[3], f[4], f[5]};
    put_state(c, slot, cf, t < 0.0 ? tf : t);   // d_time < 0: tim_t from the file (io.f90:120)
    auto ctl = read_ctl(c);
    ctl[slot].corr_dt = dtcor;   // tim_corr_dt, tim_cfl_dt (io.f90:147-150)
    ctl[slot].cfl_dt = dtcfl;
    write_ctl(c, ctl);
  });
}

// ---- Newton-Krylov clients (newton.f90) ------------------------------------
extern "C" int opf_vel_shift(opf_ctx* c, int slot, double dth, double dz) {
  return guard([&] {
    check_slot(c, slot);
    if (!c->occupied[slot]) throw OpfError(OPF_ERR_STATE, "slot holds no state");
    HIPCHK(hipStreamSynchronize(c->stream));
    auto ctl = read_ctl(c);
    ctl[slot].active = 1;
    write_ctl(c, ctl);
    launch_shift(c, slot, 1, {slot}, {dth}, {dz});
    launch(c, "curl0", k_curl, grid_hn(c, 1), dim3(64), 0, c->G, c->B, slot, 0);
    HIPCHK(hipStreamSynchronize(c->stream));
    ctl = read_ctl(c);
    ctl[slot].active = 0;
    write_ctl(c, ctl);
  });
}

extern "C" int opf_steporbit(opf_ctx* c, int nslots, const int* slots, const int* ndts, const double* T,
                             const double* sth, const double* sz) {
  return guard([&] {
    if (!c || nslots < 0 || (nslots > 0 && (!slots || !ndts || !T || !sth || !sz)))
      throw OpfError(OPF_ERR_ARG, "null argument");
    std::vector<int> sel, steps, fixed;
    std::vector<double> dth, dz;
    std::vector<int> seen(c->cap, 0);
    for (int i = 0; i < nslots; ++i) {
      const int s = slots[i];
      check_slot(c, s);
      if (seen[s]++) throw OpfError(OPF_ERR_ARG, "slot listed twice");
      if (!c->occupied[s]) throw OpfError(OPF_ERR_STATE, "slot holds no state");
      if (c->adapt[s].on) throw OpfError(OPF_ERR_ARG, "steporbit needs a fixed time step (adaptive slot)");
      if (ndts[i] < 1) throw OpfError(OPF_ERR_ARG, "ndts must be >= 1");
      if (ndts[i] != 1) {   // tim_dt = T / ndts and vel_matrices (newton.f90:736-743)
        if (!(T[i] > 0.0)) throw OpfError(OPF_ERR_ARG, "T must be > 0");
        SlotParams p{};
        HIPCHK(hipMemcpy(&p, c->B.prm + s, sizeof(p), hipMemcpyDeviceToHost));
        const double dt = T[i] / (double)ndts[i];
        if (p.dt != dt) slot_setup(c, s, p.Re, p.alpha, dt, p.implicit, p.const_flux);
      }
      sel.push_back(s);
      steps.push_back(ndts[i]);
      fixed.push_back(1);   // predictor and one corrector per step (newton.f90:745-757)
      // the shift back by the orbit's shifts after the last step (:765-770)
      dth.push_back(ndts[i] != 1 ? -sth[i] : 0.0);
      dz.push_back(ndts[i] != 1 ? -sz[i] : 0.0);
    }
    // multJ's trajectory direction (ndts = 1) leaves tim_t and tim_step as
    // they were (newton.f90:759-762 advances them only for ndts /= 1)
    std::vector<std::pair<int, double>> keep_t;
    std::vector<int> keep_step;
    {
      const auto ctl = read_ctl(c);
      for (int i = 0; i < nslots; ++i)
        if (ndts[i] == 1) {
          keep_t.push_back({slots[i], ctl[slots[i]].t});
          keep_step.push_back(ctl[slots[i]].step);
        }
    }
    run_plan(c, sel, steps, fixed, 0);
    orbit_finish(c, sel, dth, dz);
    if (!keep_t.empty()) {
      auto ctl = read_ctl(c);
      for (size_t i = 0; i < keep_t.size(); ++i) {
        ctl[keep_t[i].first].t = keep_t[i].second;
        ctl[keep_t[i].first].step = keep_step[i];
      }
      write_ctl(c, ctl);
    }
  });
}
