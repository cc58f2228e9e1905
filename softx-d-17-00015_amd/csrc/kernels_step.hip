// Per-state set-up kernels and the small kernels around the fused step:
// block inverses of the four matrices per (|k|, m) pair (and their
// LAPACK-form factors on request), the influence vectors and 4x4 inverses of the
// influence-matrix method, the curl, imposesym, on-device corrector control
// and diagnostics sums, the granular tim_lumesh_invert, and forcing added
// to the nonlinear terms.
//
// Layout: a spectral (coll) field is stored harmonic-fastest, one complex
// double2 per (n, h): element (slot, comp, n, h) at ((slot*3+comp)*N + n)*Hp + h.
// The factors are stored once per (|k|, m) pair (the matrices depend on k
// only through (alpha k)^2, timestep.f90:76-77).
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "kernels.hpp"
#include "solve.hpp"

// Sums round as they are written: separately, as in the reference's Fortran
// (built for x86-64 without FMA), in the LAPACK-form factors, the 4x4 inverses,
// the shifts and the norms, which then agree with it to the last bit or nearly;
// fused where fma() stands, in the block elimination and the curl.
#pragma clang fp contract(off)

namespace opf {

// ---------------------------------------------------------------------------
// small helpers
// ---------------------------------------------------------------------------
__device__ __forceinline__ void harmonic_km(int h, int K, int& k, int& m) {
  // parallel.h:47-56: m = 0 holds k = 0..K-1, each m >= 1 holds k = -(K-1)..K-1
  if (h < K) {
    m = 0;
    k = h;
  } else {
    const int hh = h - K;
    m = 1 + hh / (2 * K - 1);
    k = hh % (2 * K - 1) - (K - 1);
  }
}

__device__ __forceinline__ double2 cadd(double2 a, double2 b) { return make_double2(a.x + b.x, a.y + b.y); }
__device__ __forceinline__ double2 csub(double2 a, double2 b) { return make_double2(a.x - b.x, a.y - b.y); }

// Banded matrix-vector row: sum_j A(n,j) x(j), j ascending, accumulated from
// `init` (var_coll_meshmult starts from 0, tim_meshmult from c(n)).
__device__ __forceinline__ double2 band_row(const double* band, int N, int n,
                                            const double2* x, size_t xs, double2 init) {
  double2 acc = init;
  const int j0 = n - KL < 0 ? 0 : n - KL;
  const int j1 = n + KL > N - 1 ? N - 1 : n + KL;
  for (int j = j0; j <= j1; ++j) {
    const double a = band[(KL + n - j) * N + j];
    const double2 v = x[j * xs];
    acc.x = acc.x + a * v.x;
    acc.y = acc.y + a * v.y;
  }
  return acc;
}

// ---------------------------------------------------------------------------
// wall boundary residuals of the influence method (vel_evalBC,
// velocity.f90:262-298) for one harmonic; inputs are the last KL+1 radial
// values of u+, u-, uz.
// ---------------------------------------------------------------------------
__device__ void eval_bc(const double2* up, const double2* um, const double2* uz,
                        const double* dr1c, double d, double m_, double a_,
                        double BRe[4], double BIm[4]) {
  const double2 upN = up[KL], umN = um[KL], uzN = uz[KL];
  const double urRe = 0.5 * (upN.x + umN.x);
  const double urIm = 0.5 * (upN.y + umN.y);
  const double utRe = 0.5 * (upN.y - umN.y);
  const double utIm = -0.5 * (upN.x - umN.x);
  double drRe = 0.0, drIm = 0.0;
#pragma unroll
  for (int i = 0; i <= KL; ++i) {
    drRe = drRe + dr1c[i] * (up[i].x + um[i].x);
    drIm = drIm + dr1c[i] * (up[i].y + um[i].y);
  }
  drRe = 0.5 * drRe;
  drIm = 0.5 * drIm;
  BRe[0] = upN.x;
  BIm[0] = upN.y;
  BRe[1] = umN.x;
  BIm[1] = umN.y;
  BRe[2] = -uzN.y;
  BIm[2] = uzN.x;
  BRe[3] = ((urRe * d + drRe) - (d * m_) * utIm) - a_ * uzN.y;
  BIm[3] = ((urIm * d + drIm) + (d * m_) * utRe) + a_ * uzN.x;
}

// 4x4 inverse as mes_mat_invert (meshs.f90:231-243): DGETF2 + DGETRI.
// A row-major, in place.  Returns false if singular.
__device__ bool inv4(double A[16]) {
  int ipiv[4];
  for (int j = 0; j < 4; ++j) {
    int p = j;
    double best = fabs(A[j * 4 + j]);
    for (int i = j + 1; i < 4; ++i) {
      const double v = fabs(A[i * 4 + j]);
      if (v > best) { best = v; p = i; }
    }
    ipiv[j] = p;
    if (A[p * 4 + j] == 0.0) return false;
    if (p != j)
      for (int c = 0; c < 4; ++c) { const double t = A[p * 4 + c]; A[p * 4 + c] = A[j * 4 + c]; A[j * 4 + c] = t; }
    if (j < 3) {
      const double rc = 1.0 / A[j * 4 + j];
      for (int i = j + 1; i < 4; ++i) A[i * 4 + j] = A[i * 4 + j] * rc;
      for (int i = j + 1; i < 4; ++i) {
        const double lij = A[i * 4 + j];
        for (int c = j + 1; c < 4; ++c) A[i * 4 + c] = A[i * 4 + c] - lij * A[j * 4 + c];
      }
    }
  }
  double x[4];
  for (int j = 0; j < 4; ++j) {
    A[j * 4 + j] = 1.0 / A[j * 4 + j];
    const double ajj = -A[j * 4 + j];
    for (int i = 0; i < j; ++i) x[i] = A[i * 4 + j];
    for (int jj = 0; jj < j; ++jj) {
      if (x[jj] != 0.0) {
        const double temp = x[jj];
        for (int i = 0; i < jj; ++i) x[i] = x[i] + temp * A[i * 4 + jj];
        x[jj] = x[jj] * A[jj * 4 + jj];
      }
    }
    for (int i = 0; i < j; ++i) A[i * 4 + j] = x[i] * ajj;
  }
  double work[4];
  for (int j = 3; j >= 0; --j) {
    for (int i = j + 1; i < 4; ++i) { work[i] = A[i * 4 + j]; A[i * 4 + j] = 0.0; }
    for (int jj = j + 1; jj < 4; ++jj) {
      const double temp = -work[jj];
      if (temp != 0.0)
        for (int i = 0; i < 4; ++i) A[i * 4 + j] = A[i * 4 + j] + temp * A[i * 4 + jj];
    }
  }
  for (int j = 2; j >= 0; --j) {
    const int jp = ipiv[j];
    if (jp != j)
      for (int i = 0; i < 4; ++i) { const double t = A[i * 4 + j]; A[i * 4 + j] = A[i * 4 + jp]; A[i * 4 + jp] = t; }
  }
  return true;
}

// Diagonal term d(n) of tim_mesh_init / tim_lumesh_init (timestep.f90:54-55,
// 76-77) for azimuthal index m, axial index k and PM in {-1, 0, 1}.
__device__ __forceinline__ double diag_d(double r2inv, int Mp, int m, double alpha, int k, int PM) {
  double d = -((((r2inv * (double)Mp) * (double)m) * (double)Mp) * (double)m) -
             (((alpha * (double)k) * alpha) * (double)k);
  if (PM != 0) d = (d - r2inv) - ((((2.0 * (double)PM) * (double)Mp) * (double)m) * r2inv);
  return d;
}

// ---------------------------------------------------------------------------
// The block elimination's inverses (solve.hpp) of tim_lumesh_init's matrices
// (timestep.f90:67-96), one lane per (pair, matrix, side), the sides of a
// matrix in neighbouring lanes:
//   S_t = A(t, t) - A(t, o) E_o A(o, t)   (o the block before, seen from the side)
//   E_t = inv(S_t), stored as -c2 E_t
// and, for the block where the sides meet, both sides' terms subtracted.  The
// 4 x 4 inverses interchange rows; between blocks nothing is interchanged (the
// boundary rows, whose scale differs from the interior's, sit in the outermost
// blocks; against 80-bit arithmetic the solves are about as accurate as with the
// banded LU and partial pivoting: error ratio 0.3 to 1.8 in the geometric mean
// over N = 9 .. 128, single systems 30 times better or worse).
// A lane's chain is N / 8 blocks of a few hundred instructions, which bounds it.
// T: MeshOff::lapT in LDS.
// The matrices of vel_matrices are definite and their Schur complements stay
// near their diagonal blocks (row sums of the subtracted terms up to 0.7 of the
// block's own).  A matrix that a caller gives tim_lumesh_init need not be: where
// a leading block is singular, or nearly, the elimination has nothing to divide
// by.  CHECK sets *unsafe where a subtracted term exceeds BLK_GROWTH times the
// block's own row; the step then solves that slot with the banded LU.  Why the
// line lies there: over indefinite matrices with c1 near such points, against
// 80-bit arithmetic, the block elimination's error is 0.7 to 0.9 of the banded
// LU's in the geometric mean with terms up to 10 times the row, 1.7 at 10 to 30,
// 4 at 30 to 100, 130 at 300 to 1000, and it grows with the square from there.
// ---------------------------------------------------------------------------
constexpr double BLK_GROWTH = 10.0;
// the matrices of vel_matrices (velocity.f90:85-100)
__device__ __forceinline__ LuSpec matrix_spec(int mat, const SlotParams& prm) {
  const bool pr = mat == MAT_LNP;
  return LuSpec{mat, pr || mat == MAT_LDZ ? 0 : (mat == MAT_LDP ? 1 : -1), pr ? 1 : 0, pr ? 0.0 : 1.0 / prm.dt,
                pr ? 1.0 : -prm.implicit * prm.nu / prm.Re};
}
// the factor set A.mat now holds the matrix A
__device__ __forceinline__ void hold(const Bufs& B, int slot, const LuSpec& A) {
  B.spec[slot * 4 + A.mat] = A;
  atomicAdd(&B.sets[slot * 4 + A.mat].ver, 1u);
}
template <bool CHECK>
__device__ __forceinline__ void block_factor(const Geo& G, const Bufs& B, int slot, const LuSpec& A, int mat, int p,
                                             int side, double alpha, const double* T, int* unsafe) {
  const int N = G.N, P = G.P, NB = blk_count(N);
  const MeshOff mo = MeshOff::make(N);
  const double* me = G.mesh;
  const int m = p / G.K, k = p % G.K;
  const int S1 = (m * G.Mp + (A.PM != 0)) & 1;
  const double* ax = me + mo.dr0 + (KL + 1) * (1 - S1);   // axis row, columns 0..4
  const double* wl = me + mo.dr1 + (KL + 1) * A.BC;       // wall row, columns N-5..N-1
  const bool raw = A.BC == 1 && k == 0 && m == 0;   // singular, never solved (timestep.f90:84): zero inverses
  const double sc = -blk_scale(A.c2);
  double* out = B.SE + ((size_t)(slot * 4 + mat) * P + p) * NB * 16;
  // the coupling of block t to the block after it (up = 1) or before it
  auto couple = [&](int t, int up, double (&C)[4][4]) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int n = 4 * t + i;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int q = up ? (j <= i ? 8 + j - i : 9) : (j >= i ? j - i : 9);
        C[i][j] = A.c2 * T[n * 10 + q];
      }
    }
    if (t == 0) C[0][0] = ax[KL];   // only ever coupled upwards
    if (t == NB - 1) {              // only ever coupled downwards
      const int iw = (N - 1) & 3;
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const int q = 4 * (NB - 2) + j - (N - 1 - KL);
          const double v = wl[q >= 0 ? q : 0];
          C[i][j] = i == iw ? (q >= 0 ? v : 0.0) : C[i][j];
        }
    }
  };
  auto diagonal = [&](int t, double (&D)[4][4]) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int n = 4 * t + i;
      const double dg = A.c2 * diag_d(me[mo.rinv2 + min(n, N - 1)], G.Mp, m, alpha, k, A.PM) + A.c1;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        double x = A.c2 * T[n * 10 + KL + j - i];
        x = i == j ? x + dg : x;
        if (i == 0) x = t == 0 ? ax[j] : x;
        const int q = 4 * t + j - (N - 1 - KL);
        const double v = wl[q >= 0 && q <= KL ? q : 0];
        x = n == N - 1 ? (q >= 0 && q <= KL ? v : 0.0) : x;
        x = n >= N ? (i == j ? 1.0 : 0.0) : x;   // rows past the matrix
        D[i][j] = 4 * t + j >= N && i != j ? 0.0 : x;
      }
    }
  };
  // in-place inverse, Gauss-Jordan with row interchanges
  auto invert = [&](double (&D)[4][4]) {
    double I[4][4];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j) I[i][j] = i == j ? 1.0 : 0.0;
    bool singular = false;
#pragma unroll
    for (int c = 0; c < 4; ++c) {
#pragma unroll
      for (int r = c + 1; r < 4; ++r) {   // the largest of the column to row c
        const bool sw = fabs(D[r][c]) > fabs(D[c][c]);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const double a = D[c][j], b = D[r][j], e = I[c][j], f = I[r][j];
          D[c][j] = sw ? b : a;
          D[r][j] = sw ? a : b;
          I[c][j] = sw ? f : e;
          I[r][j] = sw ? e : f;
        }
      }
      singular = singular || D[c][c] == 0.0;
      const double rp = 1.0 / D[c][c];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        D[c][j] = D[c][j] * rp;
        I[c][j] = I[c][j] * rp;
      }
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        if (r == c) continue;
        const double f = D[r][c];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          D[r][j] = fma(-f, D[c][j], D[r][j]);
          I[r][j] = fma(-f, I[c][j], I[r][j]);
        }
      }
    }
    if (singular && !raw) {
      if (CHECK) *unsafe = 1;
      else atomicMax(&B.ctl[slot].status, 100 + mat);
    }
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j) D[i][j] = I[i][j];
  };
  auto store = [&](int t, const double (&E)[4][4]) {
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int i = 0; i < 4; i += 2)
        *(double2*)(out + t * 16 + 4 * j + i) =
            raw ? make_double2(0.0, 0.0) : make_double2(sc * E[i][j], sc * E[i + 1][j]);
  };
  // D -= U; a row whose term dwarfs it loses that many digits
  auto subtract = [&](double (&D)[4][4], const double (&U)[4][4]) {
    if (CHECK && !raw) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        double u = 0.0, d = 0.0;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          u = u + fabs(U[i][j]);
          d = d + fabs(D[i][j]);
        }
        if (!(u <= BLK_GROWTH * d)) *unsafe = 1;   // a NaN, after a singular block, also
      }
    }
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j) D[i][j] = D[i][j] - U[i][j];
  };
  const int nm = blk_mid(N);
  const int steps = side ? NB - 1 - nm : nm, dt = side ? -1 : 1;
  double D[4][4], U[4][4];   // the next block's matrix; the terms to subtract from it
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) U[i][j] = 0.0;
  int t = side ? NB - 1 : 0;
#pragma unroll 1
  for (int s = 0; s < nm; ++s) {
    if (s >= steps) break;
    diagonal(t, D);
    subtract(D, U);
    invert(D);
    store(t, D);
    double C[4][4], Y[4][4];
    couple(t, side ? 0 : 1, C);   // Y = E_t A(t, u)
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        double v = 0.0;
#pragma unroll
        for (int q = 0; q < 4; ++q) v = fma(D[i][q], C[q][j], v);
        Y[i][j] = v;
      }
    t += dt;
    couple(t, side ? 1 : 0, C);   // U = A(u, t) Y
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        double v = 0.0;
#pragma unroll
        for (int q = 0; q < 4; ++q) v = fma(C[i][q], Y[q][j], v);
        U[i][j] = v;
      }
  }
  diagonal(nm, D);
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) U[i][j] = U[i][j] + __shfl_xor(U[i][j], 1);
  subtract(D, U);
  invert(D);
  if (side == 0) store(nm, D);
}

// one factor set of its own matrix (tim_lumesh_init).  grid: x = pairs / 32; 64 threads.
__global__ void __launch_bounds__(64) k_block_factor(Geo G, Bufs B, int slot, LuSpec A, int* unsafe) {
  __shared__ double T[10 * (MAXN + 8)];
  for (int i = threadIdx.x; i < 10 * (G.N + 8); i += 64) T[i] = G.mesh[MeshOff::make(G.N).lapT + i];
  if (threadIdx.x == 0 && blockIdx.x == 0) hold(B, slot, A);
  __syncthreads();
  // spare lanes repeat the last pair
  block_factor<true>(G, B, slot, A, A.mat, min((int)blockIdx.x * 32 + (int)(threadIdx.x >> 1), G.P - 1),
                     threadIdx.x & 1, B.prm[slot].alpha, T, unsafe);
}

// ---------------------------------------------------------------------------
// tim_lumesh_init (timestep.f90:67-96) + DGBTF2 of one matrix per pair in
// LAPACK band layout, for tim_lumesh_get / tim_lumesh_invert (the time step
// solves with block_factor's inverses).  Four lanes per system.  *singular is
// set where a pivot is zero.  A workgroup whose factors are of the set's present
// version has nothing to do, so a host that solves with its own sets again and
// again pays for the factors once per set; the version counts on the device,
// where the matrices change (adaptive time step, LES).
// grid: x = pairs/16; 64 threads = 16 systems x 4 lanes.
// ---------------------------------------------------------------------------
__global__ void __launch_bounds__(64) k_lu_factor(Geo G, Bufs B, LuFactors L, int slot, int mat,
                                                 int* singular) {
  constexpr int LPS = 4;              // lanes per system
  constexpr int SPW = 64 / LPS;       // systems per workgroup
  const int q = threadIdx.x % LPS, sl = threadIdx.x / LPS;
  const int p = blockIdx.x * SPW + sl;
  const unsigned ver = B.sets[slot * 4 + mat].ver;
  if (L.built[blockIdx.x] == ver) return;
  // no barriers below: a lane may leave on its own
  if (p >= G.P) return;
  const int N = G.N;
  const int m = p / G.K, k = p % G.K;  // pair (|k|, m)
  const SlotParams prm = B.prm[slot];
  const MeshOff mo = MeshOff::make(N);
  const double* me = G.mesh;
  const LuSpec spec = B.spec[slot * 4 + mat];   // the matrix that the factor set holds
  const int PM = spec.PM, BC = spec.BC;
  const double c1 = spec.c1, c2 = spec.c2;
  double* F = L.F + (size_t)p * N * LUS;
  unsigned char* pv = L.pv + (size_t)p * N;
  // The elimination at column j touches columns j .. j + KV only, so each
  // system keeps a window of KV + 1 band columns in LDS (column c in slot
  // c mod 9, the systems' values interleaved) instead of working on the
  // factor array in global memory, where every access of the serial
  // elimination waited a full cache round trip.  A column leaves the window
  // finished (stored once) and the next enters built from the mesh.  The
  // four lanes of a system share a step's work, each on its own data with
  // the same instructions: lane q takes the window columns j + c with
  // c = q, q + 4 (and 8 for lane 0), the rows q, q + 4, q + 8 (and 12) of a
  // new column, and a quarter of a finished one; all four find the pivot.
  // Lanes pass values to each other through the window: a wave's LDS
  // operations complete in the order issued, and lds_fence() keeps the
  // compiler from moving an access across a hand-over point.  The
  // arithmetic is DGBTF2's, operation for operation.
  constexpr int WC = 2 * KL + 1;   // window columns
  __shared__ double Wd[WC * NLU * SPW];
  auto W = [&](int ws, int row) -> double& { return Wd[(ws * NLU + row) * SPW + sl]; };
  auto lds_fence = [] { __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront"); };
  const int S = (m * G.Mp + (PM < 0 ? -PM : PM)) % 2;
  // column `col` of tim_lumesh_init's band (timestep.f90:67-96): the mesh
  // operator, then the boundary rows of the first and last KL + 1 columns.
  // Lane q builds rows brow(t) = q + 4t (t < 3) and row 12 (t = 3, all four
  // lanes, the same value).  fetch() reads the mesh values of a column into
  // registers a column ahead of place(), so the loads overlap an
  // elimination step.  Both run on every step (with the column clamped,
  // place() writing only when `put`): a load left pending on one path would
  // make every later step wait for all the stores before it.  Each lane
  // loads its own rows' values and reads its own rows of a finished column,
  // so no lane ever selects among values by q (the compiler turns such
  // selects into an indexed stack array).
  auto brow = [&](int t) { return t < 3 ? LPS * t + q : NLU - 1; };
  struct Src {
    double lap[4], r2, b0, b1;
  };
  auto fetch = [&](int col, Src& c) {
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      const int a = brow(t) - KL;
      c.lap[t] = me[mo.lapb + (a < 0 ? 0 : a) * N + col];
    }
    c.r2 = me[mo.rinv2 + col];
    const int i0 = col <= KL ? col : KL, i1 = col >= N - KL - 1 ? col - (N - KL - 1) : 0;
    c.b0 = me[mo.dr0 + i0 + (KL + 1) * (1 - S)];
    c.b1 = me[mo.dr1 + i1 + (KL + 1) * BC];
  };
  auto place = [&](int ws, int col, const Src& c, bool put) {
    const double d = diag_d(c.r2, G.Mp, m, prm.alpha, k, PM);
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      const int row = brow(t);
      double x = row < KL ? 0.0 : c2 * c.lap[t];
      x = row == 2 * KL ? (x + c2 * d) + c1 : x;
      x = (col <= KL && row == 2 * KL - col) ? c.b0 : x;
      x = (col >= N - KL - 1 && row == 2 * KL + N - 1 - col) ? c.b1 : x;
      if (put) W(ws, row) = x;
    }
  };
  auto rd = [&](int ws, int row) { return W(ws, row < NLU ? row : NLU - 1); };
  auto store = [&](int ws, int col, int pj) {
    // LAPACK column: rows 4q .. 4q + 3 from lane q (rows 13 .. 15 zero)
    double x[LPS];
#pragma unroll
    for (int r = 0; r < LPS; ++r) {
      const int row = LPS * q + r;
      const double v = rd(ws, row);
      x[r] = row < NLU ? v : 0.0;
    }
    reinterpret_cast<double4*>(F + (size_t)col * LUS)[q] = make_double4(x[0], x[1], x[2], x[3]);
    if (q == 0) pv[col] = (unsigned char)pj;
  };
  // the pressure matrix of (0,0) is never factored: its lanes store the
  // columns as built, in the same loop as the others
  const bool raw = BC == 1 && k == 0 && m == 0;
  for (int col = 0; col < WC && col < N; ++col) {
    Src c;
    fetch(col, c);
    place(col, col, c, true);
  }
  // DGBTF2, KL = KU = 4, KV = 8 (0-based rows).  A step touches columns
  // j .. j + 8 (the window) and rows KV - 8 .. KV + 4 of them; each lane
  // reads the elements of its columns that the step may change at once and
  // writes every one back, changed where DGBTF2 changes it and unchanged
  // elsewhere, so the step is straight-line code (selects instead of
  // branches on the run-time limits km, ju and the pivot).  Window slots
  // past the matrix's last column hold columns already stored; rewriting
  // them with their own values is harmless.
  constexpr int KV = 2 * KL;
  int ju = 0;
  Src nx;
  for (int j = 0, wj = 0; j < N; ++j, wj = wj + 1 == WC ? 0 : wj + 1) {
    const int jn = j + WC < N ? j + WC : N - 1;
    fetch(jn, nx);
    lds_fence();   // the previous step's columns and new column are written
    const int km = raw ? 0 : (N - 1 - j < KL ? N - 1 - j : KL);
    double pc[KL + 1];   // rows KV .. KV + KL of column j
#pragma unroll
    for (int i = 0; i <= KL; ++i) pc[i] = W(wj, KV + i);
    int jp = 0;
    double best = fabs(pc[0]), piv = pc[0];
#pragma unroll
    for (int i = 1; i <= KL; ++i) {
      const double v = fabs(pc[i]);
      const bool better = i <= km && v > best;
      best = better ? v : best;
      jp = better ? i : jp;
      piv = better ? pc[i] : piv;
    }
    if (!raw && piv == 0.0) {
      if (q == 0) pv[j] = (unsigned char)jp;
      if (q == 0) *singular = 1;
      return;
    }
    const int lim = j + KL + jp < N - 1 ? j + KL + jp : N - 1;
    ju = raw ? ju : (ju > lim ? ju : lim);
    const int nc = raw ? -1 : ju - j;   // columns j .. j + nc take part (nc <= KV)
    // multipliers: the pivot column below the diagonal after the
    // interchange, scaled by 1/pivot (rows 1 .. km)
    const double rc = 1.0 / (raw ? 1.0 : piv);
    double l[KL + 1];
#pragma unroll
    for (int i = 1; i <= KL; ++i) {
      const double li = (jp != 0 && i == jp) ? pc[0] : pc[i];
      l[i] = i <= km ? li * rc : li;
    }
    // this lane's columns j + c: the row interchange of rows j and j + jp,
    // then, for c = 0, the multipliers and, for c > 0, the rank-1 update of
    // the rows below the diagonal
#pragma unroll
    for (int t = 0; t < 3; ++t) {
      const int c = q + LPS * t;
      if (t == 2 && q != 0) break;   // c = 8 is lane 0's alone
      const int ws = wj + c >= WC ? wj + c - WC : wj + c;
      const double ra = W(ws, KV + jp - c), rb = W(ws, KV - c);
      const bool sw = jp != 0 && c <= nc;
      W(ws, KV + jp - c) = sw ? rb : ra;
      W(ws, KV - c) = sw ? ra : rb;
      const double temp = -(sw ? ra : rb);   // row KV - c after the interchange
      const bool col_on = c <= nc && temp != 0.0;
      double cv[KL + 1];
#pragma unroll
      for (int i = 1; i <= KL; ++i) cv[i] = W(ws, KV + i - c);
#pragma unroll
      for (int i = 1; i <= KL; ++i)
        W(ws, KV + i - c) = c == 0 ? l[i] : ((col_on && i <= km) ? cv[i] + l[i] * temp : cv[i]);
    }
    lds_fence();   // column j is final
    store(wj, j, jp);
    lds_fence();   // every lane has read column j before its slot is refilled
    place(wj, jn, nx, j + WC < N);
  }
  if (threadIdx.x == 0) L.built[blockIdx.x] = ver;
}

// ---------------------------------------------------------------------------
// Device rows u[comp][n][Hp] <-> the reference's coll planes, of a component
// re[h][n] then im[h][n] (r fastest), through LDS tiles of 32 x 32 so that both
// sides move whole lines.  The host's loops over both layouts took 100 ms for
// the 300 MB of a (96,256,128) state, whose copy needs 11.
// grid: x = 32-harmonic tiles of a row (Hp, the padding included: zeros), y =
// 32-point tiles, z = component; 256 threads.
// ---------------------------------------------------------------------------
__global__ void __launch_bounds__(256) k_rows_to_planes(Geo G, const double2* __restrict__ rows,
                                                        double* __restrict__ planes) {
  __shared__ double2 t[32][33];
  const int h0 = blockIdx.x * 32, n0 = blockIdx.y * 32, lo = threadIdx.x & 31, hi = threadIdx.x >> 5;
  const size_t nh = (size_t)G.N * G.H;
  rows += blockIdx.z * G.coll;
  planes += blockIdx.z * 2 * nh;
  for (int i = hi; i < 32; i += 8)
    if (n0 + i < G.N && h0 + lo < G.H) t[i][lo] = rows[(size_t)(n0 + i) * G.Hp + h0 + lo];
  __syncthreads();
  for (int i = hi; i < 32; i += 8)
    if (n0 + lo < G.N && h0 + i < G.H) {
      const double2 v = t[lo][i];
      const size_t o = (size_t)(h0 + i) * G.N + n0 + lo;
      planes[o] = v.x;
      planes[nh + o] = v.y;
    }
}
// ADD: onto the rows (forcing added to vel_N* by var_null(2) hooks), of the H harmonics
template <bool ADD>
__global__ void __launch_bounds__(256) k_planes_to_rows(Geo G, const double* __restrict__ planes,
                                                        double2* __restrict__ rows) {
  __shared__ double2 t[32][33];
  const int h0 = blockIdx.x * 32, n0 = blockIdx.y * 32, lo = threadIdx.x & 31, hi = threadIdx.x >> 5;
  const size_t nh = (size_t)G.N * G.H;
  rows += blockIdx.z * G.coll;
  planes += blockIdx.z * 2 * nh;
  double re[4], im[4];   // all loads in one batch: the planes may be host memory
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const size_t o = (size_t)min(h0 + hi + 8 * q, G.H - 1) * G.N + min(n0 + lo, G.N - 1);
    re[q] = planes[o];
    im[q] = planes[nh + o];
  }
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const int i = hi + 8 * q;
    t[lo][i] = n0 + lo < G.N && h0 + i < G.H ? make_double2(re[q], im[q]) : make_double2(0.0, 0.0);
  }
  __syncthreads();
  for (int i = hi; i < 32; i += 8)
    if (n0 + i < G.N && h0 + lo < (ADD ? G.H : G.Hp)) {
      double2 v = t[i][lo];
      double2* r = rows + (size_t)(n0 + i) * G.Hp + h0 + lo;
      if (ADD) v = make_double2(r->x + v.x, r->y + v.y);
      *r = v;
    }
}
template __global__ void k_planes_to_rows<false>(Geo, const double*, double2*);
template __global__ void k_planes_to_rows<true>(Geo, const double*, double2*);

// ---------------------------------------------------------------------------
// var_coll_norm (variables.f90:718-751) of a field in the reference's coll
// layout (re, im: N x H, r fastest).  Pass 1, one thread per harmonic:
// b(h) = sum_n f(n) intrdr(n) with f = w (re^2 + im^2), w = 4 pi^2 / alpha,
// in n order, halved for (0,0).  Pass 2, one workgroup: Em(m) and Ek(|k|)
// accumulate b in harmonic order (parallel.h:47-56), then E = sum(Em) in m
// order.  out = [E, Ek(0:K-1), Em(0:M-1)].
// ---------------------------------------------------------------------------
__global__ void k_norm_harm(Geo G, const SlotParams* __restrict__ prm, const double* __restrict__ re,
                            const double* __restrict__ im, double* __restrict__ b) {
  const int h = blockIdx.x * blockDim.x + threadIdx.x;
  if (h >= G.H) return;
  const double w = 4.0 * D_PI * D_PI / prm->alpha;
  const double* intrdr = G.mesh + MeshOff::make(G.N).intrdr;
  const double* a = re + (size_t)h * G.N;
  const double* c = im + (size_t)h * G.N;
  double s = 0.0;
  for (int n = 0; n < G.N; ++n) {
    const double f = w * (a[n] * a[n] + c[n] * c[n]);
    s = s + f * intrdr[n];
  }
  b[h] = h == 0 ? 0.5 * s : s;
}

__global__ void k_norm_sum(Geo G, const double* __restrict__ b, double* __restrict__ out) {
  const int t = threadIdx.x;
  const int K = G.K, M = G.M, W = 2 * G.K - 1;
  double* Ek = out + 1;
  double* Em = out + 1 + K;
  for (int m = t; m < M; m += blockDim.x) {   // the harmonics of m, k ascending
    double s = 0.0;
    if (m == 0) {
      for (int k = 0; k < K; ++k) s = s + b[k];
    } else {
      const double* bm = b + K + (size_t)(m - 1) * W;
      for (int i = 0; i < W; ++i) s = s + bm[i];
    }
    Em[m] = s;
  }
  for (int q = t; q < K; q += blockDim.x) {   // |k| = q: (q, 0), then (-q, m), (q, m) for m >= 1
    double s = b[q];
    for (int m = 1; m < M; ++m) {
      const double* bm = b + K + (size_t)(m - 1) * W + (K - 1);
      if (q > 0) s = s + bm[-q];
      s = s + bm[q];
    }
    Ek[q] = s;
  }
  __syncthreads();
  if (t == 0) {
    double e = 0.0;
    for (int m = 0; m < M; ++m) e = e + Em[m];
    out[0] = e;
  }
}

// ---------------------------------------------------------------------------
// vel_maxtstep (velocity.f90:438-481) from the per-plane maxima that the
// theta kernel recorded for the last evaluation, and tim_new_tstep
// (timestep.f90:259-278): cfl and its direction, and the new dt, nw whether
// vel_matrices follows.  Every lane of a wave takes the planes n = lane,
// lane + 64, ..; the minima are exact, so their order is free.
// ---------------------------------------------------------------------------
struct NewStep {
  double cfl, dt;
  int dir, ntc;
  bool nw;
};
__device__ __forceinline__ NewStep new_tstep(const Geo& G, const Bufs& B, int slot, const SlotCtl& c,
                                             const SlotParams& prm, int lane) {
  const int N = G.N;
  const MeshOff mo = MeshOff::make(N);
  const double* r = G.mesh + mo.r;
  const unsigned long long* mx = B.cflmax + (size_t)slot * 3 * N;
  const double dth = (2.0 * D_PI) / (double)(G.T * G.Mp);
  const double dz = (2.0 * D_PI) / (prm.alpha * (double)G.Z);
  double t1 = 1e99, t2 = 1e99, t3 = 1e99;
  for (int n = lane; n < N; n += 64) {
    double d;
    if (n == 0) d = r[1] - r[0];
    else if (n == N - 1) d = r[N - 1] - r[N - 2];
    else d = fmin(r[n] - r[n - 1], r[n + 1] - r[n]);
    const double a = __longlong_as_double((long long)mx[n]);
    const double b = __longlong_as_double((long long)mx[N + n]);
    const double e = __longlong_as_double((long long)mx[2 * N + n]);
    if (a != 0.0) t1 = fmin(t1, d / a);
    if (b != 0.0) t2 = fmin(t2, dth / b);
    if (e != 0.0) t3 = fmin(t3, dz / e);
  }
  for (int off = 32; off >= 1; off >>= 1) {
    t1 = fmin(t1, __shfl_xor(t1, off));
    t2 = fmin(t2, __shfl_xor(t2, off));
    t3 = fmin(t3, __shfl_xor(t3, off));
  }
  NewStep s;
  s.cfl = fmin(t1, fmin(t2, t3));
  s.dir = c.cfl_dir;
  if (s.cfl == t1) s.dir = 1;
  if (s.cfl == t2) s.dir = 2;
  if (s.cfl == t3) s.dir = 3;
  // tim_new_tstep
  const double dt0 = prm.dt;
  double dt = fmin(dt0 * 1.11, prm.maxdt);
  if (c.step == 0 && c.corr_dt == 0.0) dt = fmin(dt, s.cfl * 0.1);
  if (s.cfl > 0.0) dt = fmin(dt, s.cfl * prm.courant);
  if (c.corr_dt > 0.0) dt = fmin(dt, c.corr_dt * 0.95);
  const int i = c.ntc - 1;
  s.nw = dt < dt0 * 0.95 || (dt > dt0 * 1.10 && i < 0) || (dt == prm.maxdt && dt0 < dt && i < 0);
  s.ntc = (s.nw && dt >= dt0) ? 99 : i;
  s.dt = s.nw ? dt : dt0;
  return s;
}
// vel_maxtstep alone (one wave)
__global__ void k_maxtstep(Geo G, Bufs B, int slot) {
  SlotCtl* c = &B.ctl[slot];
  const NewStep s = new_tstep(G, B, slot, *c, B.prm[slot], threadIdx.x);
  if (threadIdx.x != 0) return;
  c->cfl_dt = s.cfl;
  c->cfl_dir = s.dir;
}

// ---------------------------------------------------------------------------
// vel_matrices (velocity.f90:85-100) of eight pairs per workgroup: the four
// matrices' inverses (block_factor, all 64 lanes of wave 0), the influence
// vectors of vel_adjPPE(0) (velocity.f90:191-218; wave w solves matrix w) with
// vel_adjustFlux(0) (:160-168) on pair 0, and the inverted influence matrices
// of the pairs' harmonics (:219-225).
// Uinf slots: 0 U1 (LDp), 1 U2 (LDm), 2 U3 (LDz), 3 U4, 4 U5, 5 p (U6 = p*alpha*k).
// gate: 0 always; 1 where ctl.refactor asks for it; 2 a slot of the device
// loop about to run a predictor with an adaptive time step: tim_new_tstep first,
// and the rest where it changed dt.
// One launch, since most launches find nothing to do and cost their few
// microseconds all the same (an adaptive step of (48,48,24) spent 28 of its 115
// us on four of them per evaluation; 106 now), and a set-up is a chain of
// latencies: 41 us in three launches and 29 in this one at (32,24,12), 75 and
// 57 at (64,64,48).
// grid: x = pairs/8, z = slot.  SM >= blk_mid(N).
// ---------------------------------------------------------------------------
template <int SM>
__global__ void __launch_bounds__(256) k_matrices_t(Geo G, Bufs B, int slot0, int gate) {
  constexpr int PW = 8, XS = PW + 2;   // right-hand sides: the pairs', the flux problem's, and zeros
  const int p0 = blockIdx.x * PW;
  const int slot = slot_of(B, slot0);
  const int N = G.N, P = G.P, K = G.K;
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const int np = min(PW, P - p0);
  SlotCtl* ctl = &B.ctl[slot];
  SlotParams prm = B.prm[slot];
  if (gate == 1 && !ctl->refactor) return;
  if (gate == 2) {
    const SlotCtl c = *ctl;
    if (!(c.active && c.mode == MODE_PRED && prm.adaptive)) return;
    const NewStep s = new_tstep(G, B, slot, c, prm, lane);
    __syncthreads();
    // every workgroup has read what the last one to arrive here writes
    if (tid == 0 &&
        __hip_atomic_fetch_add(&ctl->arrived, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == gridDim.x - 1) {
      ctl->arrived = 0u;
      ctl->cfl_dt = s.cfl;
      ctl->cfl_dir = s.dir;
      ctl->ntc = s.ntc;
      B.prm[slot].dt = s.dt;
    }
    if (!s.nw) return;
    prm.dt = s.dt;
  }
  const MeshOff mo = MeshOff::make(N);
  const double* me = G.mesh;
  extern __shared__ double lap[];          // the Laplacian's rows
  double* X = lap + 10 * (N + 8);          // [4][N + 4][XS]
  double* W = X + 4 * (N + 4) * XS;        // [6][PW][KL + 1]: the vectors' rows at the wall
  const int mat = wave;
  const bool flux = p0 == 0 && mat == MAT_LDZ && prm.const_flux != 0;
  double* Xi = X + mat * (N + 4) * XS;
  for (int i = tid; i < 10 * (N + 8); i += 256) lap[i] = me[mo.lapT + i];
  for (int i = lane; i < (N + 4) * XS; i += 64) {
    const int n = i / XS, r = i - n * XS;
    double v = 0.0;
    if (r < PW && n == N - 1) v = mat == MAT_LNP ? -1.0 : 1.0;
    if (r == PW && flux) v = n == 0 || n >= N - 1 ? 0.0 : 1.0;
    Xi[i] = v;
  }
  __syncthreads();
  if (wave == 0) {
    const int fm = lane >> 4, fp = (lane >> 1) & 7;
    const LuSpec A = matrix_spec(fm, prm);
    if (p0 == 0 && (lane & 15) == 0) hold(B, slot, A);
    if (p0 == 0 && lane == 0) B.sets[slot * 4].banded = 0;
    // spare lanes repeat the last pair
    block_factor<false>(G, B, slot, A, fm, p0 + min(fp, np - 1), lane & 1, prm.alpha, lap, nullptr);
  }
  __syncthreads();
  const BlkLane l = BlkLane::make(lane);
  const LuSpec A = matrix_spec(mat, prm);
#pragma unroll 1
  for (int g = 0; g < PW / 2; ++g) {
    BlkE<SM, 1> E;
    const int pl = 2 * g + l.mi;
    blk_load(E, 0, G, B, slot, A, mat, p0 + min(pl, np - 1), l);
    double* const x[1] = {Xi + (l.col == 0 ? pl : l.col == 1 && pl == 0 ? PW : PW + 1)};
    blk_solve(E, N, l, lap, x, XS);
  }
  __syncthreads();
  double* U = B.Uinf + (size_t)slot * 6 * N * P + p0;
  const size_t us = (size_t)N * P;
  for (int i = lane; i < N * PW; i += 64) {
    const int n = i / PW, ip = i % PW, wr = n - (N - 1 - KL);
    if (ip >= np) continue;
    double* u = U + (size_t)n * P + ip;
    double* w = W + ip * (KL + 1) + wr;
    auto put = [&](int f, double v) {
      u[f * us] = v;
      if (wr >= 0) w[f * PW * (KL + 1)] = v;
    };
    const double x = Xi[n * XS + ip];
    if (mat != MAT_LNP) {
      put(mat, x);
    } else {
      // grad: dr1 . p (meshmult from 0), t.Im = p * m/r; rt2pm -> U4 = gr - tIm, U5 = gr + tIm
      double gr = 0.0;
#pragma unroll
      for (int dd = -KL; dd <= KL; ++dd) {
        const int j = n + dd;
        if (j >= 0 && j <= N - 1) gr = gr + me[mo.dr1b + (KL - dd) * N + j] * Xi[j * XS + ip];
      }
      const double mr = (me[mo.rinv + n] * (double)G.Mp) * (double)((p0 + ip) / K);
      const double tIm = x * mr;
      put(5, x);
      put(3, gr - tIm);
      put(4, gr + tIm);
    }
  }
  if (p0 == 0 && mat == MAT_LDZ) {
    double* Ui = B.Ui + (size_t)slot * N;
    for (int n = lane; n < N; n += 64) Ui[n] = Xi[n * XS + PW];
    if (flux && lane == 0) {
      double s = 0.0;
      for (int n = 0; n < N; ++n) s = s + Xi[n * XS + PW] * me[mo.intrdr + n];
      ctl->flux_d1 = 2.0 * s;
      if (2.0 * s == 0.0) atomicMax(&ctl->status, 110);
    }
  }
  __syncthreads();
  // harmonics +k and -k of the pairs
  const int ip = tid & (PW - 1), p = p0 + ip, m = p / K, ka = p - m * K, k = tid & PW ? -ka : ka;
  if (tid >= 2 * PW || ip >= np || (k < 0 && m == 0) || (tid >= PW && ka == 0)) return;
  const int h = m == 0 ? k : K + (m - 1) * (2 * K - 1) + k + K - 1;
  double* Ai = B.Ainv + (size_t)slot * 16 * G.H + h;
  if (p == 0) {
    for (int q = 0; q < 16; ++q) Ai[(size_t)q * G.H] = 0.0;
    return;
  }
  const double ak = prm.alpha * (double)k;
  double M4[16];
  for (int j = 0; j < 4; ++j) {
    double2 up[KL + 1], um[KL + 1], uz[KL + 1];
    for (int i = 0; i <= KL; ++i) {
      const double* w = W + ip * (KL + 1) + i;
      constexpr int fs = PW * (KL + 1);
      up[i] = um[i] = uz[i] = make_double2(0.0, 0.0);
      if (j == 0) up[i].x = w[0];
      if (j == 1) um[i].x = w[fs];
      if (j == 2) uz[i].y = w[2 * fs];
      if (j == 3) {
        up[i].x = w[3 * fs];
        um[i].x = w[4 * fs];
        uz[i].y = w[5 * fs] * ak;
      }
    }
    double BRe[4], BIm[4];
    eval_bc(up, um, uz, me + mo.dr1 + (KL + 1), me[mo.rinv + N - 1], (double)(m * G.Mp), ak, BRe, BIm);
    for (int i = 0; i < 4; ++i) M4[i * 4 + j] = BRe[i];
  }
  if (!inv4(M4)) atomicMax(&ctl->status, 120);
  for (int q = 0; q < 16; ++q) Ai[(size_t)q * G.H] = M4[q];
}

MatricesKern matrices_kernel(int N) {
  static_assert(blk_mid(32) == 4 && blk_mid(64) == 8 && blk_mid(96) == 12 && blk_mid(MAXN) == 16, "the ranges");
  return N <= 32 ? k_matrices_t<4> : N <= 64 ? k_matrices_t<8> : N <= 96 ? k_matrices_t<12> : k_matrices_t<16>;
}

// ---------------------------------------------------------------------------
// curl (var_coll_curl, variables.f90:408-436) of the current iterate -> om
// ---------------------------------------------------------------------------
__device__ __forceinline__ void curl_point(const Geo& G, int h, int n, int k, int m, double alpha,
                                           const double2* ur, const double2* ut, const double2* uz, double2* om) {
  const int N = G.N;
  const size_t hs = G.Hp;
  const MeshOff mo = MeshOff::make(N);
  const double* me = G.mesh;
  const double ri = me[mo.rinv + n], mr = ri * ((double)G.Mp * (double)m);
  const size_t o = (size_t)n * hs + h;
  double2 d1 = make_double2(0.0, 0.0), d2 = d1;
  for (int j = max(n - KL, 0); j <= min(n + KL, N - 1); ++j) {
    const double a = me[mo.dr1b + (KL + n - j) * N + j];
    const double2 z = uz[(size_t)j * hs + h], t = ut[(size_t)j * hs + h];
    d1 = make_double2(fma(a, z.x, d1.x), fma(a, z.y, d1.y));
    d2 = make_double2(fma(a, t.x, d2.x), fma(a, t.y, d2.y));
  }
  double2 w[3];
  curl_of(ur[o], ut[o], uz[o], d1, d2, ri, mr, alpha * (double)k, w);
#pragma unroll
  for (int c = 0; c < 3; ++c) om[c * G.coll + o] = w[c];
}

// which = 0: curl of U[ucur]; used after put_state and after every step.
// One thread per (h, n).  grid: x = 8 * per blocks over the (64-harmonic
// block, n) tiles, z = slot; tiles in XCD-aware order (block b takes tile
// (b % 8) per + b / 8, tiles ordered harmonic block first), so the nine rows
// of a stencil are read by workgroups on one XCD and come from its L2.
__global__ void k_curl(Geo G, Bufs B, int slot0, int gated) {
  const int nhb = (G.H + 63) / 64, ntile = nhb * G.N, per = (ntile + 7) / 8;
  const int tile = (int)(blockIdx.x % 8) * per + (int)(blockIdx.x / 8);
  if (tile >= ntile) return;
  const int hb = tile / G.N, n = tile - hb * G.N;
  const int h = hb * 64 + threadIdx.x;
  const int slot = slot_of(B, slot0);
  const SlotCtl* c = &B.ctl[slot];
  if (!c->active || h >= G.H) return;
  if (gated && (c->mode != MODE_PRED || B.prm[slot].symm == 0)) return;
  int k, m;
  harmonic_km(h, G.K, k, m);
  const double2* u = B.U[c->ucur] + (size_t)slot * 3 * G.coll;
  curl_point(G, h, n, k, m, B.prm[slot].alpha, u, u + G.coll, u + 2 * G.coll,
             B.om + (size_t)slot * 3 * G.coll);
}

// vel_imposesym (velocity.f90:61-74) with the slot's symmetries on U[ucur]:
// var_imposesym(0), then (1) mirror, (2) shift & reflect, (3) shift &
// rotate as enabled (variables.f90:538-618; each ends with the harmonic-0
// conditions of mode 0).  Modes 1 and 2 average a harmonic (k, m) with the
// image of its partner (-k, m) (itself for m = 0): factor a = 1, or (-1)^k
// for shift & reflect; the imaginary part flips for m > 0; u_theta flips.
// Both act within a pair, mode 3 within a harmonic and every mode within a
// component, so one thread takes (n, pair, component) and applies the
// enabled modes in order in registers.  gated: only slots about to run a
// predictor (the start of a step, main.f90:21) with a symmetry enabled.
__global__ void k_symmetry(Geo G, Bufs B, int slot0, int gated) {
  const int slot = slot_of(B, slot0);
  const SlotCtl* c = &B.ctl[slot];
  const int symm = B.prm[slot].symm;
  if (!c->active || (gated && (c->mode != MODE_PRED || symm == 0))) return;
  const int idx = blockIdx.x * blockDim.x + threadIdx.x;   // (comp, n, h)
  const int h = idx % G.H, rest = idx / G.H;
  const int n = rest % G.N, comp = rest / G.N;
  if (comp >= 3) return;
  int k, m;
  harmonic_km(h, G.K, k, m);
  if (m > 0 && k < 0) return;                 // taken by the partner (k > 0)
  const int hp = m == 0 ? h : h - 2 * k;      // harmonic (-k, m)
  double2* u = B.U[c->ucur] + (size_t)slot * 3 * G.coll + (size_t)comp * G.coll + (size_t)n * G.Hp;
  double2 x = u[h], y = u[hp];
  const double b = m == 0 ? 1.0 : -1.0;
  const double sg = comp == 1 ? -1.0 : 1.0;   // u_theta changes sign
  auto fix0 = [&]() {                         // mode 0 on harmonic 0
    if (h == 0) {
      if (comp == 0) x = make_double2(0.0, 0.0);
      else x.y = 0.0;
    }
  };
  fix0();
  for (int i = 1; i <= 3; ++i) {
    if (!(symm & (1 << (i - 1)))) continue;
    if (i <= 2) {
      const double a = (i == 2 && (k & 1)) ? -1.0 : 1.0;
      const double f = sg * a;
      // image of the partner (of x for the partner's own update)
      const double2 ix = make_double2(y.x * f, y.y * (f * b));
      const double2 iy = make_double2(x.x * f, x.y * (f * b));
      x = make_double2((x.x + ix.x) / 2.0, (x.y + ix.y) / 2.0);
      if (hp != h) y = make_double2((y.x + iy.x) / 2.0, (y.y + iy.y) / 2.0);
      else y = x;
    } else if ((k + m) & 1) {
      x = make_double2(0.0, 0.0);
      y = x;
    }
    fix0();
  }
  u[h] = x;
  if (hp != h) u[hp] = y;
}

// ---------------------------------------------------------------------------
// Non-Newtonian viscosity (the plugin of nonnewtonian.f90:93-244): the
// velocity-gradient tensor of the total flow u + U(r) z^, the strain rate and
// the Carreau-Yasuda viscosity nu on the physical grid, and the forcing
// N' = [(nu - 1) Lap(u) + grad(nu) . 2S] / Re added to the raw N of the
// evaluation.  Spectral pieces run per harmonic (one thread per h, all n),
// physical pieces per grid point; the transforms between them are the
// single-field transforms of tra_coll2phys / tra_phys2coll.
// ---------------------------------------------------------------------------
// The gradient tensor A of the slot's current iterate (get_nu,
// nonnewtonian.f90:108-147): row 0 the radial derivatives by
// var_coll_meshmult with dr(1), row 1 the theta terms (1/r)(d/dtheta u -
// e_theta x u), row 2 the z derivatives; out holds the three components of each
// row.  One thread per (h, n): grid x = harmonics / 64, y = N, z = row.  The nine
// fields then pass through each transform in one launch, which for few fields
// takes little more than the launch itself ((48,48,24), z and theta: 6.1 and 7.0
// us for three fields, 8.5 and 11.2 for six and nine).
__global__ void k_nn_grad(Geo G, Bufs B, int slot, double2* __restrict__ out) {
  const int row = blockIdx.z;
  out += (size_t)row * 3 * G.coll;
  const int h = blockIdx.x * blockDim.x + threadIdx.x;
  const int n = blockIdx.y;
  if (h >= G.H) return;
  int k, m;
  harmonic_km(h, G.K, k, m);
  const double2* u = B.U[B.ctl[slot].ucur] + (size_t)slot * 3 * G.coll;
  const MeshOff mo = MeshOff::make(G.N);
  const double* me = G.mesh;
  const size_t hs = G.Hp;
  const int N = G.N;
  auto at = [&](int comp, int j) {   // u, with vel_U added to the (0, 0) mode of u_z
    double2 v = u[(size_t)comp * G.coll + (size_t)j * hs + h];
    if (comp == 2 && h == 0) v.x = v.x + me[mo.Ubase + j];
    return v;
  };
  const size_t o = (size_t)n * hs + h;
  if (row == 0) {
    const int j0 = n - KL < 0 ? 0 : n - KL;
    const int j1 = n + KL > N - 1 ? N - 1 : n + KL;
    for (int comp = 0; comp < 3; ++comp) {
      double2 acc = make_double2(0.0, 0.0);
      for (int j = j0; j <= j1; ++j) {
        const double a = me[mo.dr1b + (KL + n - j) * N + j];
        const double2 v = at(comp, j);
        acc.x = acc.x + a * v.x;
        acc.y = acc.y + a * v.y;
      }
      out[(size_t)comp * G.coll + o] = acc;
    }
  } else if (row == 1) {
    const double ri = me[mo.rinv + n];
    const double mm = (double)(m * G.Mp);
    const double2 vr = at(0, n), vt = at(1, n), vz = at(2, n);
    out[o] = make_double2(ri * (-(vr.y * mm) - vt.x), ri * (vr.x * mm - vt.y));
    out[G.coll + o] = make_double2(ri * (-(vt.y * mm) + vr.x), ri * (vt.x * mm + vr.y));
    out[2 * G.coll + o] = make_double2(ri * (-(vz.y * mm)), ri * (vz.x * mm));
  } else {
    const double d1 = B.prm[slot].alpha * (double)k;
    for (int comp = 0; comp < 3; ++comp) {
      const double2 v = at(comp, n);
      out[(size_t)comp * G.coll + o] = make_double2(-(v.y * d1), v.x * d1);
    }
  }
}

// var_coll_grad (variables.f90:442-459) of a scalar coll field p into out;
// one thread per (h, n).
__global__ void k_nn_gradp(Geo G, Bufs B, int slot, const double2* __restrict__ p, double2* __restrict__ out) {
  const int h = blockIdx.x * blockDim.x + threadIdx.x;
  const int n = blockIdx.y;
  if (h >= G.H) return;
  int k, m;
  harmonic_km(h, G.K, k, m);
  const MeshOff mo = MeshOff::make(G.N);
  const double* me = G.mesh;
  const double ak = B.prm[slot].alpha * (double)k;
  const size_t o = (size_t)n * G.Hp + h;
  out[o] = band_row(me + mo.dr1b, G.N, n, p + h, G.Hp, make_double2(0.0, 0.0));
  const double mr = (me[mo.rinv + n] * (double)G.Mp) * (double)m;
  const double2 v = p[o];
  out[G.coll + o] = make_double2(-(v.y * mr), v.x * mr);
  out[2 * G.coll + o] = make_double2(-(v.y * ak), v.x * ak);
}

// curl(curl(u + U z^)) of the current iterate: the curl (var_coll_curl,
// variables.f90:408-436) of the slot's vorticity om = curl u, plus curl curl
// (U z^) = -Lap(U) z^ = 4 z^ on the (0, 0) mode (U = 1 - r^2); one thread
// per (h, n).
__global__ void k_nn_curlcurl(Geo G, Bufs B, int slot, double2* __restrict__ out) {
  const int h = blockIdx.x * blockDim.x + threadIdx.x;
  const int n = blockIdx.y;
  if (h >= G.H) return;
  int k, m;
  harmonic_km(h, G.K, k, m);
  const int N = G.N;
  const size_t hs = G.Hp;
  const MeshOff mo = MeshOff::make(N);
  const double* me = G.mesh;
  const double ak = B.prm[slot].alpha * (double)k;
  const double2* wr = B.om + (size_t)slot * 3 * G.coll;
  const double2* wt = wr + G.coll;
  const double2* wz = wr + 2 * G.coll;
  const double mr = (me[mo.rinv + n] * (double)G.Mp) * (double)m;
  const size_t o = (size_t)n * hs + h;
  const double2 vr = wr[o], vt = wt[o], vz = wz[o];
  out[o] = make_double2(-(vz.y * mr) + vt.y * ak, vz.x * mr - vt.x * ak);
  const double2 d1 = band_row(me + mo.dr1b, N, n, wz + h, hs, make_double2(0.0, 0.0));
  out[G.coll + o] = make_double2(-(vr.y * ak) - d1.x, vr.x * ak - d1.y);
  const double2 d2 = band_row(me + mo.dr1b, N, n, wt + h, hs, make_double2(0.0, 0.0));
  const double ri = me[mo.rinv + n];
  double2 qz = make_double2((vt.x * ri + d2.x) + vr.y * mr, (vt.y * ri + d2.y) - vr.x * mr);
  if (h == 0) qz.x += 4.0;
  out[2 * G.coll + o] = qz;
}

// get_nu's algebra per grid point (nonnewtonian.f90:148-172): the upper half of
// S = (A + A^T)/2 written back over A's, strain rate sr = (2 S:S)^(1/2) and the Carreau-Yasuda
// viscosity nu = d1 + (1 - d1)(1 + (lam sr)^a)^d2.
__global__ void k_nn_visc(NnPhys P, size_t np, double lam, double d1, double d2, double a) {
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= np) return;
  double* const* S = P.S;
  const double s12 = 0.5 * (S[1][i] + S[3][i]);
  const double s13 = 0.5 * (S[2][i] + S[6][i]);
  const double s23 = 0.5 * (S[5][i] + S[7][i]);
  S[1][i] = s12;
  S[2][i] = s13;
  S[5][i] = s23;
  const double s11 = S[0][i], s22 = S[4][i], s33 = S[8][i];
  double sr = s11 * s11 + s22 * s22 + s33 * s33 + 2.0 * (s12 * s12 + s13 * s13 + s23 * s23);
  sr = sqrt(2.0 * sr);
  P.nu[i] = d1 + (1.0 - d1) * pow(1.0 + pow(lam * sr, a), d2);
}

// update_nonlin_terms' algebra per grid point (nonnewtonian.f90:227-236):
// q_i = [(nu - nu_r)(-curlcurl(u)_i) + sum_j grad(nu)_j S_ji 2 + (nu_r - 1)(-4) delta_i3] / Re.
__global__ void k_nn_force(NnPhys P, size_t np, double nu_r, double Re) {
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= np) return;
  const double nu_ = P.nu[i] - nu_r;
  const double g[3] = {P.g[0][i], P.g[1][i], P.g[2][i]};
  const double s01 = P.S[1][i], s02 = P.S[2][i], s12 = P.S[5][i];
  const double S[9] = {P.S[0][i], s01, s02, s01, P.S[4][i], s12, s02, s12, P.S[8][i]};
  for (int c = 0; c < 3; ++c) {
    double q = nu_ * (-P.q[c][i]);
    for (int j = 0; j < 3; ++j) q = q + g[j] * S[j * 3 + c] * 2.0;
    if (c == 2) q = q + (nu_r - 1.0) * (-4.0);
    P.q[c][i] = q / Re;
  }
}

// ---------------------------------------------------------------------------
// LES eddy viscosity (the plugin of LES.f90:100-395).  D holds per slot
// [Delta(N), Delta_r(N), L_theta(N), coef(N)]: the Smagorinsky filter width,
// the radial spacing, the azimuthal length of Vreman's filter and, written
// by k_les_prep, the per-plane model coefficient.
// ---------------------------------------------------------------------------
// u_tau, Re_tau, y+ (get_nu, LES.f90:170-177) and the per-plane coefficient:
// Smagorinsky vanDr (C_s Delta)^2 (:206-213), Vreman's damping
// d1 + (1 - d1) vanDr with d1 = 0.03/C_s, or 1 without damping (:247-256);
// clears the slot's nu_max.  One wave.
__global__ void k_les_prep(Geo G, Bufs B, int slot, int model, double Cs, double Aplus, double* D,
                           unsigned long long* numax) {
  const int N = G.N;
  const MeshOff mo = MeshOff::make(N);
  const double* me = G.mesh;
  const double2* uz = B.U[B.ctl[slot].ucur] + (size_t)slot * 3 * G.coll + 2 * G.coll;
  const double* w = me + mo.dr1 + (KL + 1);   // dr1(:,1)
  double d1 = 0.0;
  for (int i = 0; i <= KL; ++i) d1 = d1 + uz[(size_t)(N - 1 - KL + i) * G.Hp].x * w[i];
  const double Re = B.prm[slot].Re;
  const double utau = sqrt(fabs((d1 - 2.0) / Re));
  const double Retau = Re * utau;
  for (int n = threadIdx.x; n < N; n += blockDim.x) {
    const double yp = Retau * (1.0 - me[mo.r + n]);
    const double q = yp / Aplus;
    const double vanDr = 1.0 - exp(-(q * q));
    double c;
    if (model == 1) {
      const double cd = Cs * D[n];
      c = vanDr * (cd * cd);
    } else if (Aplus <= 0.0) {
      c = 1.0;
    } else {
      const double a = 0.03 / Cs;
      c = a + (1.0 - a) * vanDr;
    }
    D[3 * N + n] = c;
  }
  if (threadIdx.x == 0) numax[slot] = 0ull;
}

// The eddy viscosity per grid point from the gradient tensor A (row-major in
// P.S), which is then replaced by S = (A + A^T)/2: Smagorinsky nu = coef
// sr, sr = (2 S:S)^(1/2); Vreman nu = coef C_s (P/AA)^(1/2) with
// B = sum_m Delta_m^2 A_mi A_mj (:218-257).  The slot's nu_max by one
// atomic per workgroup on the bit pattern (nu >= 0).
__global__ void k_les_visc(NnPhys P, size_t np, int N, int ZT, int model, double Cs, double dz, const double* D,
                           unsigned long long* numax_slot) {
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  double nu = 0.0;
  if (i < np) {
    const int n = (int)(i / (size_t)ZT);
    double a[9];
    for (int q = 0; q < 9; ++q) a[q] = P.S[q][i];
    if (model == 2) {
      double AA = 0.0;
      for (int q = 0; q < 9; ++q) AA = AA + a[q] * a[q];
      const double dl[3] = {D[N + n], D[2 * N + n], dz};
      double Bm[9];
      for (int r = 0; r < 3; ++r)
        for (int c = 0; c < 3; ++c) {
          double b = 0.0;
          for (int m = 0; m < 3; ++m) b = b + (dl[m] * dl[m]) * a[m * 3 + r] * a[m * 3 + c];
          Bm[r * 3 + c] = b;
        }
      double Pv = Bm[0] * Bm[4] - Bm[1] * Bm[1] + Bm[0] * Bm[8] - Bm[2] * Bm[2] + Bm[4] * Bm[8] - Bm[5] * Bm[5];
      Pv = AA < 1e-12 ? 0.0 : Pv;
      Pv = fmax(Pv, 0.0);
      AA = fmax(AA, 1e-12);
      nu = Cs * sqrt(Pv / AA) * D[3 * N + n];
    }
    const double s12 = 0.5 * (a[1] + a[3]);
    const double s13 = 0.5 * (a[2] + a[6]);
    const double s23 = 0.5 * (a[5] + a[7]);
    if (model == 1) {
      double sr = a[0] * a[0] + a[4] * a[4] + a[8] * a[8] + 2.0 * (s12 * s12 + s13 * s13 + s23 * s23);
      sr = sqrt(2.0 * sr);
      nu = D[3 * N + n] * sr;
    }
    P.S[1][i] = s12; P.S[3][i] = s12;
    P.S[2][i] = s13; P.S[6][i] = s13;
    P.S[5][i] = s23; P.S[7][i] = s23;
    P.nu[i] = nu;
  }
  for (int off = 32; off >= 1; off >>= 1) nu = fmax(nu, __shfl_xor(nu, off));
  __shared__ double wm[4];
  if ((threadIdx.x & 63) == 0) wm[threadIdx.x >> 6] = nu;
  __syncthreads();
  if (threadIdx.x == 0) {
    double v = wm[0];
    for (int q = 1; q < (int)(blockDim.x >> 6); ++q) v = fmax(v, wm[q]);
    atomicMax(numax_slot, (unsigned long long)__double_as_longlong(v));
  }
}

// update_nu_r (LES.f90:264-273) before a predictor: vel_nu = 1.1 (1 + Re
// nu_max) when it has left [0.93, 1.07] of that value; the change is left in
// `refactor` for the gated vel_matrices launches that follow.
__global__ void k_les_nur(Bufs B, int slot, const unsigned long long* numax) {
  SlotCtl* c = &B.ctl[slot];
  SlotParams* prm = &B.prm[slot];
  if (!(c->active && c->mode == MODE_PRED)) {
    c->refactor = 0;
    return;
  }
  const double nm = __longlong_as_double((long long)numax[slot]);
  double d1 = 1.0 + prm->Re * nm;
  d1 = 1.10 * d1;
  const bool ch = prm->nu < 0.93 * d1 || prm->nu > 1.07 * d1;
  if (ch) prm->nu = d1;
  c->refactor = ch ? 1 : 0;
}

// The LES forcing per grid point (update_nonlin_terms, LES.f90:303-311):
// q_i = (1/Re) nu' (-curlcurl(u)_i) + nu (-4) delta_i3 + sum_j grad(nu)_j S_ji 2,
// nu' = Re nu + 1 - vel_nu.
__global__ void k_les_force(NnPhys P, size_t np, Bufs B, int slot) {
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= np) return;
  const double Re = B.prm[slot].Re, nur = B.prm[slot].nu;
  const double nu = P.nu[i];
  const double nu_ = Re * nu + (1.0 - nur);
  for (int c = 0; c < 3; ++c) {
    double q = (1.0 / Re) * nu_ * (-P.q[c][i]);
    if (c == 2) q = q + nu * (-4.0);
    for (int j = 0; j < 3; ++j) q = q + P.g[j][i] * P.S[j * 3 + c][i] * 2.0;
    P.q[c][i] = q;
  }
}

// N += N': added to the raw nonlinear terms of the slot's current evaluation.
// grid: x = H/64, y = N, z = component.
__global__ void k_nn_addN(Geo G, Bufs B, int slot, const double2* __restrict__ src) {
  const int comp = blockIdx.z;
  src += (size_t)comp * G.coll;
  const int h = blockIdx.x * blockDim.x + threadIdx.x;
  const int n = blockIdx.y;
  if (h >= G.H || n >= G.N) return;
  double2* dst = B.Nraw[B.ctl[slot].ncur] + (size_t)slot * 3 * G.coll + (size_t)comp * G.coll;
  const size_t o = (size_t)n * G.Hp + h;
  const double2 a = dst[o], b = src[o];
  dst[o] = make_double2(a.x + b.x, a.y + b.y);
}

// var_coll_shift (variables.f90:487-528) on U[ucur] of slots [slot0,
// slot0 + gridDim.z): harmonic (k, m) rotated by e^{-i alpha k dz}, then by
// e^{-i m Mp dth}, each in the reference's order of operations
// (Re' = Re c + Im s, Im' = Im c - Re s).  tab holds 2K + M entries per
// slot: [0] = (z shift on, theta shift on), [k + K] = (cos, sin)(dz k alpha)
// for k = -(K-1)..K-1, [2K + m] = (cos, sin)(dth m Mp), evaluated on the host
// with the C library's cos and sin as the reference's dcos and dsin.  One
// thread per (component, n, harmonic).
__global__ void k_shift(Geo G, Bufs B, int slot0, const double2* __restrict__ tab) {
  const int slot = slot_of(B, slot0);
  const double2* tb = tab + (size_t)blockIdx.z * (2 * G.K + G.M);
  const double2 on = tb[0];
  if (on.x == 0.0 && on.y == 0.0) return;
  const int idx = blockIdx.x * blockDim.x + threadIdx.x;
  const int h = idx % G.H, rest = idx / G.H;
  const int n = rest % G.N, comp = rest / G.N;
  if (comp >= 3) return;
  int k, m;
  harmonic_km(h, G.K, k, m);
  double2* u = B.U[B.ctl[slot].ucur] + (size_t)slot * 3 * G.coll + (size_t)comp * G.coll + (size_t)n * G.Hp + h;
  double2 x = *u;
  auto rot = [&](const double2 cs) {
    const double re = x.x;
    x.x = re * cs.x + x.y * cs.y;   // products rounded before the sum (no FMA in this file)
    x.y = x.y * cs.x - re * cs.y;
  };
  if (on.x != 0.0) rot(tb[k + G.K]);
  if (on.y != 0.0) rot(tb[2 * G.K + m]);
  *u = x;
}

// A request's admission into a free slot, in stream order between
// iterations of the other slots (one thread).  phase 0, before its factors
// are built: clear the failure status the factor kernels report into.
// phase 1, after the state is loaded: a fresh run of nsteps steps with
// corr_fixed correctors per step (put_state + run_begin of the synchronous
// path), active only if the factorisation succeeded.
__global__ void k_admit(Bufs B, int slot, int phase, int nsteps, int corr_fixed) {
  SlotCtl k = B.ctl[slot];
  if (phase == 0) {
    k.status = 0;
    k.active = 0;
  } else {
    k.step = 0;
    k.t = 0.0;
    k.mode = MODE_PRED;
    k.it = 0;
    k.ncorr = 0;
    k.ndiag = 0;
    k.corr_dt = 0.0;
    k.cfl_dt = 0.0;
    k.cfl_dir = 0;
    k.ntc = 0;
    k.refactor = 0;
    k.target_steps = nsteps;
    k.corr_fixed = corr_fixed;
    k.diag_every = 0;
    k.host_driven = 0;
    k.active = k.status == 0 ? 1 : 0;
  }
  B.ctl[slot] = k;
}

// A host-driven call on one slot, in stream order (one thread): begin marks the
// slot active, for the launches between, as a single procedure of the host's
// own loop (mode < 0: as it is); the end clears the mark and reports tim_dterr
// to host memory.
__global__ void k_host_call(Bufs B, int slot, int begin, int mode, double* dterr) {
  SlotCtl* c = &B.ctl[slot];
  if (begin) {
    c->active = 1;
    c->target_steps = -1;
    if (mode >= 0) c->mode = mode;
    c->diag_every = 0;
    c->corr_fixed = 0;
    c->host_driven = 1;
  } else {
    c->active = 0;
    *dterr = c->last_dterr;
  }
}

// var_imposesym(0) (variables.f90:611-616) on harmonic 0 of U[ucur].
__global__ void k_imposesym(Geo G, Bufs B, int slot0) {
  const int n = blockIdx.x * blockDim.x + threadIdx.x;
  const int slot = slot_of(B, slot0);
  const SlotCtl* c = &B.ctl[slot];
  if (n >= G.N) return;
  double2* u = B.U[c->ucur] + (size_t)slot * 3 * G.coll;
  const size_t o = (size_t)n * G.Hp;
  u[o] = make_double2(0.0, 0.0);
  u[G.coll + o].y = 0.0;
  u[2 * G.coll + o].y = 0.0;
}

// tim_lumesh_invert (timestep.f90:102-123) of one coll field x[n][Hp] with
// the factors L; (0,0) of the pressure matrix gives zero.
__global__ void k_lumesh_invert(Geo G, LuFactors L, int bc, double2* x) {
  const int h = blockIdx.x * blockDim.x + threadIdx.x;
  if (h >= G.H) return;
  int k, m;
  harmonic_km(h, G.K, k, m);
  const int N = G.N;
  const int p = m * G.K + (k < 0 ? -k : k);
  if (bc == 1 && k == 0 && m == 0) {   // the (0,0) pressure system is singular: b = 0
    for (int n = 0; n < N; ++n) x[(size_t)n * G.Hp + h] = make_double2(0.0, 0.0);
    return;
  }
  lu_solve<double2>(L.F + (size_t)p * N * LUS, L.pv + (size_t)p * N, x + h, G.Hp, N);
}

}  // namespace opf
