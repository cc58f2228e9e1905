// Device buffers of a resolution class and the kernel entry points.
#pragma once
#include <hip/hip_runtime.h>

#include "opf_internal.hpp"

namespace opf {

// The matrix a factorisation builds for set `mat`: c1 + c2 Lap (of u+-: PM =
// +-1) with the wall row BC.
struct LuSpec {
  int mat, PM, BC;
  double c1, c2;
};

// LAPACK-form factors of one factor set (buffers on first use of
// tim_lumesh_*): column n of pair p, LAPACK band row r at F[(p N + n) LUS + r],
// pivot offset ipiv(n) - n at pv[p N + n].
struct LuFactors {
  double* F;
  unsigned char* pv;
  unsigned* built;   // per workgroup of k_lu_factor: the set's version that its factors are of
};
struct FactorSet {
  LuFactors lu;
  unsigned ver;      // counts the set's rebuilds
  int banded;        // of a slot's first set: its steps solve with the LAPACK-form factors (a set needs row interchanges)
};

// All device arrays of one resolution class (slot-major).  Passed by value.
struct Bufs {
  double2* U[3];        // velocity buffers [slot][3][N][Hp]; roles per slot in SlotCtl
  double2* Nraw[2];     // nonlinear terms without base-flow terms [slot][3][N][Hp]
  double2* om;          // curl of the current iterate [slot][3][N][Hp]
  FactorSet* sets;      // [slot][4 mats]
  double* SE;           // block inverses (block_factor, solve.hpp) [slot][4 mats][P pairs][blk_count(N)][16],
                        // element (row, column) at 4 column + row
  LuSpec* spec;         // [slot][4] the matrix each factor set holds
  double* Uinf;         // influence vectors [slot][6][N][P]
  double* Ainv;         // inverted influence matrices [slot][16][H]
  double* Ui;           // flux correction vector [slot][N]
  double* diagb;        // per-harmonic energy partials [slot][3][Hp]
  unsigned long long* cflmax;  // [slot][3][N] per-plane max of |u_r|, |u_t|, |u_z + 1 - r^2| on the
                               // physical grid of the last evaluation (bit patterns, vel_maxtstep)
  unsigned long long* arrive;  // [slot][arrive_words(P)] arrivals of the step kernel's workgroups (0 between
                        // launches), one word per 128 bytes, then each workgroup's max |du|^2 (bit pattern)
  DiagRec* diag;        // diagnostics records [slot][diag_cap]
  SlotParams* prm;      // [slot]
  SlotCtl* ctl;         // [slot]
  double2* Yf;          // forward intermediates [slot][N][ZQ/4][6][M][4] (z, field, m, z % 4)
  double2* Yb;          // backward intermediates [slot][N][ZQ/4][3][M][4]
  double2* twZ;         // twiddles exp(2 pi i q / Z), q < Z
  double2* twT;         // twiddles exp(2 pi i q / T), q < T
  const int* smap;      // null: grid z counts slots from slot0; else the slots of a
                        // compacted launch, smap[slot0 + z]
};

// The slot a workgroup serves: slot0 + blockIdx.z, or its entry of the
// compacted slot list.
__device__ __forceinline__ int slot_of(const Bufs& B, int slot0) {
  return B.smap ? B.smap[slot0 + (int)blockIdx.z] : slot0 + (int)blockIdx.z;
}

// Tile shapes of the transform kernels (chosen by the host / autotuner).
struct FftTiles {
  int tm;     // m columns per workgroup in the z kernels
  int tz;     // z lines per workgroup in the theta kernel
  FftPlan pz, pt;
};

// Block elimination: blocks of four rows, the block where the two sides meet,
// and the scale of a matrix' unknowns (solve.hpp).
__host__ __device__ constexpr int blk_count(int N) { return (N + 3) / 4; }
__host__ __device__ constexpr int blk_mid(int N) { return blk_count(N) / 2; }
// The scale is c2; without a Laplacian (c2 = 0, d_implicit = 0) a stand-in so
// small that the couplings drop out of every sum, and so far from the smallest
// double that the scaled unknowns keep their digits.
__host__ __device__ inline double blk_scale(double c2) { return c2 != 0.0 ? c2 : 1e-100; }

// curl of one harmonic at one radial point (var_coll_curl,
// variables.f90:408-436) from u, the radial derivatives d1 of u_z and d2 of
// u_theta, 1/r, m/r and alpha k: one definition for the step kernel and
// k_curl, so that a state read back and loaded again continues with the same bits.
__device__ __forceinline__ void curl_of(double2 vr, double2 vt, double2 vz, double2 d1, double2 d2, double ri,
                                        double mr, double ak, double2 (&w)[3]) {
  w[0] = make_double2(fma(vt.y, ak, -(vz.y * mr)), fma(-vt.x, ak, vz.x * mr));
  w[1] = make_double2(-fma(vr.y, ak, d1.x), fma(vr.x, ak, -d1.y));
  w[2] = make_double2(fma(vr.y, mr, fma(vt.x, ri, d2.x)), fma(-vr.x, mr, fma(vt.y, ri, d2.y)));
}

// Shape of the fused step kernel.
struct StepTiles {
  int gp;        // (|k|, m) pairs per workgroup: 1, 2 or 4
  int ngroups;   // workgroups per slot
  size_t smem;   // dynamic LDS bytes
};
constexpr int ARRIVE_WORDS = 16;
__host__ __device__ constexpr size_t arrive_words(int P) { return 16 * ARRIVE_WORDS + (size_t)P; }
inline int step_threads(int gp) { return gp == 1 ? 128 : 256; }
// LDS of a step workgroup in doubles: V[3][N + 8][2 gp] (complex, four rows of
// zeros at either end), the mesh tables (MeshOff::lapT, d1T, rowv), the
// influence coefficients and the reduction words.
__host__ __device__ constexpr size_t step_lds_doubles(int N, int gp) {
  return (size_t)12 * (N + 8) * gp + 10 * (N + 8) + 13 * N + (N & 1) + 16 * gp + 16;
}

constexpr int FFT_THREADS = 256;
constexpr int FFT_TILE = 2048;   // complex values per transform workgroup (all its lines)
constexpr int THETA_MAX = FFT_TILE / 3;   // longest theta line: its three packed transforms fill a tile
// items (line, theta point) one theta workgroup holds in registers: FFT_TILE / 3
// rounded up to whole rounds of FFT_THREADS (768).  Lines of 3M > FFT_TILE / 2
// would leave one line per workgroup under FFT_TILE; they take two lines
// when 2 * 3M fits in these items (up to 3M = 384).
constexpr int THETA_ITEMS = ((FFT_TILE / 3 + FFT_THREADS - 1) / FFT_THREADS) * FFT_THREADS;

// LDS stride of one transform of length L in the transform kernels: one pad
// slot per 16 elements, rounded up to an odd count.
// m columns per workgroup of the z transforms for length Z (as many as fit
// in FFT_TILE values; rounding down to whole 128-byte lines of the
// intermediates measured slower)
__host__ __device__ constexpr int tile_m(int Z) { return FFT_TILE / Z; }

__host__ __device__ constexpr int padded_len(int L) { return (L + (L - 1) / 16 + 1) | 1; }

__global__ void k_block_factor(Geo G, Bufs B, int slot, LuSpec A, int* unsafe);
__global__ void k_lu_factor(Geo G, Bufs B, LuFactors L, int slot, int mat, int* singular);
using MatricesKern = void (*)(Geo, Bufs, int, int);
MatricesKern matrices_kernel(int N);
inline size_t matrices_smem(int N) { return (size_t)(10 * (N + 8) + 40 * (N + 4) + 48 * (KL + 1)) * sizeof(double); }
__global__ void k_curl(Geo G, Bufs B, int slot0, int gated);
__global__ void k_symmetry(Geo G, Bufs B, int slot0, int gated);
__global__ void k_maxtstep(Geo G, Bufs B, int slot);
__global__ void k_imposesym(Geo G, Bufs B, int slot0);
__global__ void k_host_call(Bufs B, int slot, int begin, int mode, double* dterr);
__global__ void k_admit(Bufs B, int slot, int phase, int nsteps, int corr_fixed);
__global__ void k_shift(Geo G, Bufs B, int slot0, const double2* __restrict__ tab);
// non-Newtonian plugin: physical-grid fields of one slot (row-major S(i,j) at S[3i+j])
struct NnPhys {
  double* S[9];
  double* nu;
  double* g[3];
  double* q[3];
};
__global__ void k_nn_grad(Geo G, Bufs B, int slot, double2* __restrict__ out);
__global__ void k_nn_gradp(Geo G, Bufs B, int slot, const double2* __restrict__ p, double2* __restrict__ out);
__global__ void k_nn_curlcurl(Geo G, Bufs B, int slot, double2* __restrict__ out);
__global__ void k_nn_visc(NnPhys P, size_t np, double lam, double d1, double d2, double a);
__global__ void k_nn_force(NnPhys P, size_t np, double nu_r, double Re);
__global__ void k_nn_addN(Geo G, Bufs B, int slot, const double2* __restrict__ src);
__global__ void k_les_prep(Geo G, Bufs B, int slot, int model, double Cs, double Aplus, double* D,
                           unsigned long long* numax);
__global__ void k_les_visc(NnPhys P, size_t np, int N, int ZT, int model, double Cs, double dz, const double* D,
                           unsigned long long* numax_slot);
__global__ void k_les_nur(Bufs B, int slot, const unsigned long long* numax);
__global__ void k_les_force(NnPhys P, size_t np, Bufs B, int slot);
__global__ void k_rows_to_planes(Geo G, const double2* rows, double* planes);
template <bool ADD> __global__ void k_planes_to_rows(Geo G, const double* planes, double2* rows);
// var_coll_norm of a field in the coll layout: per-harmonic partials b[H], then [E, Ek, Em]
__global__ void k_norm_harm(Geo G, const SlotParams* prm, const double* re, const double* im, double* b);
__global__ void k_norm_sum(Geo G, const double* b, double* out);
// the fused step kernel for N radial points and gp pairs per workgroup
using StepKern = void (*)(Geo, Bufs, StepTiles, int);
StepKern step_kernel(int N, int gp);
StepKern step_kernel_banded();   // one pair per workgroup, any N: also for slots marked banded

// transforms: kernels specialised to the radix plans of (Z, T), chosen once
// per context by fft_kernels (run-time plans for other lengths)
using FftKern = void (*)(Geo, Bufs, FftTiles, int);
using ZOneKern = void (*)(Geo, Bufs, FftTiles, const double2*, double2*, size_t, size_t);
using C2rKern = void (*)(Geo, Bufs, FftTiles, int, const double2*, double*, size_t, size_t);
using R2cKern = void (*)(Geo, Bufs, FftTiles, int, const double*, double2*, size_t, size_t);
struct FftKerns {
  FftKern zfwd, theta, zbwd;
  ZOneKern zfwd1, zbwd1;   // one coll field to / from its z-transformed plane, a batch of fields as grid z
  C2rKern c2r;             // theta lines of such planes to / from phys[n][z][theta], two lines per transform
  R2cKern r2c;
  FftTiles t;       // the tiles asked for, at most those that the kernels hold
  int zn, tn, ln;   // threads of the z, theta and line kernels
  int bt;           // transforms per workgroup of the line kernels
  size_t zfs, zbs, ts, c2rs, r2cs;   // dynamic LDS bytes (zfwd1, zbwd1: as zfwd, zbwd)
};
FftKerns fft_kernels(const FftPlan& pz, const FftPlan& pt, const FftTiles& t, int M);
// whole-plane evaluation (z, theta, products, theta, z in one workgroup per
// radial plane) for the grids that have one; nullptr otherwise.
// smem: its dynamic LDS bytes.
constexpr int PLANE_THREADS = 1024;
using PlaneKern = FftKern;
PlaneKern plane_kernel(int Z, int T, size_t* smem);
// phys of one coll field by theta lines with z fastest (granular API), from the
// z transforms' output
__global__ void k_theta_c2r(Geo G, Bufs B, FftTiles T, const double2* Y, double* phys);
__global__ void k_theta_r2c(Geo G, Bufs B, FftTiles T, const double* phys, double2* Y);

}  // namespace opf
