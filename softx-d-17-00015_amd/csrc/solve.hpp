// Two-sided block elimination of the banded systems on the matrix cores
// (device code shared by the fused step kernel and the influence vectors).
//
// The matrices have half bandwidth 4, so in blocks of four rows they are block
// tridiagonal: A(t, t-1), A(t, t), A(t, t+1), t < NB = ceil(N / 4) (rows past
// N are identity rows).  Side 0 eliminates the blocks 0, 1, .. and side 1 the
// blocks NB-1, NB-2, .. towards the middle block blk_mid(N), where the two
// meet:
//   z_t = E_t c_t,  c_u = b_u - A(u, t) z_t        (u the next block inwards)
//   x_m = E_m c_m
//   x_t = z_t - E_t A(t, u) x_u                    (back, outwards)
// with E_t the inverse of the block's Schur complement, the only numbers that
// are stored per matrix: 16 per four rows, read once for both sweeps, where
// a band LU has 9 to 13 per row and reads them twice.  The couplings A(t, u)
// are c2 times the radial Laplacian whatever the matrix (k, m and the time
// step enter on the diagonal only), so they come from one table of the mesh in
// LDS; scaling the unknown by c2 takes c2 out of them.  Only the boundary
// rows differ (BlkLane::bc).
//
// Every product is a v_mfma_f64_4x4x4 of four 4x4x4 blocks: block b of a wave
// is (matrix b / 2, side b % 2), its columns the matrix' four right-hand sides
// (harmonics +k and -k, real and imaginary part).  Lane l holds element
// (row or k = l / 16, column = l % 4) of block (l / 4) % 4 of B, C and D, so a
// product's result is the next one's operand as it stands, and element
// (row = l % 4, k = l / 16) of A.  A solve is four dependent products per pair
// of blocks, N / 8 pairs, and its code is short: a wave runs it once per launch,
// at the rate at which instructions arrive rather than execute.  (An
// elimination row by row took 90 to 105 ns a row in straight-line code.)
//
// lu_solve at the end is that elimination, with LAPACK's factors and row
// interchanges: tim_lumesh_invert's, and the step kernel's for a slot one of
// whose sets the blocks cannot represent (block_factor).
#pragma once
#include <hip/hip_runtime.h>

#include "kernels.hpp"

namespace opf {

__device__ __forceinline__ double mfma4(double a, double b, double c) {
  return __builtin_amdgcn_mfma_f64_4x4x4f64(a, b, c, 0, 0, 0);
}

// What a lane of a solving wave stands for.
struct BlkLane {
  int side, mi;    // side and matrix (0, 1) of its block
  int row;         // row in the block of B, C, D (and k of A)
  int col;         // right-hand side (and row of A)
  __device__ static BlkLane make(int lane) {
    return BlkLane{(lane >> 2) & 1, (lane >> 3) & 1, lane >> 4, lane & 3};
  }
};

// The sweep's geometry (uniform) and this lane's part of it.
struct BlkSweep {
  int NB, S, d;        // blocks; steps of either side; 1: side 1 has one block less (its step 0 is empty)
  int t0, dt;          // block of step i: t0 + i dt (step 0 of an empty first step clamped by the callers)
  __host__ __device__ static constexpr BlkSweep make(int N, int side) {
    BlkSweep s{};
    s.NB = blk_count(N);
    s.S = blk_mid(N);
    s.d = 1 - (s.NB & 1);
    s.t0 = side ? s.NB - 1 + s.d : 0;
    s.dt = side ? -1 : 1;
    return s;
  }
  __host__ __device__ __forceinline__ constexpr int first(int side) const { return side ? NB - 1 : 0; }
};

// The sweeps take every block once, the middle one last, and stay within the
// table (rows 0 .. N + 7) and the right-hand sides (rows 0 .. N + 3), for every N
// of a context.
constexpr bool blk_sweeps_cover() {
  for (int N = 9; N <= MAXN; ++N) {
    bool seen[blk_count(MAXN)] = {};
    const int mid = blk_mid(N);
    for (int side = 0; side < 2; ++side) {
      const BlkSweep w = BlkSweep::make(N, side);
      if (w.S != mid || 4 * w.NB + 4 > N + 8) return false;
      for (int i = 0; i < w.S; ++i) {
        const int t = w.t0 + i * w.dt;
        const int f = t + w.dt;   // table rows 4 f .. of the forward sweep, 4 t .. of the backward one
        if (f < 0 || f > w.NB || t < 0 || t > w.NB) return false;
        const bool empty = side && w.d && i == 0;
        if (empty != (t == w.NB)) return false;
        if (empty) continue;
        if (seen[t] || t == mid) return false;
        seen[t] = true;
        if (i == w.S - 1 && f != mid) return false;
      }
    }
    for (int t = 0; t < blk_count(N); ++t)
      if (seen[t] == (t == mid)) return false;
  }
  return true;
}
static_assert(blk_sweeps_cover(), "blocks of the two sides");

// The inverses of NG groups of two matrices: steps 0 .. S-1, then the middle
// block in e[g][SM].  SM >= S.
template <int SM, int NG>
struct BlkE {
  double e[NG][SM + 1];
  double bc[NG];      // the boundary row's entries in the outermost coupling
  double rs[NG];      // scale of the solution, -1 / c2
};

// Loads of group g: the set `mat` of pair p (this lane's), holding the matrix s;
// p's m gives the parity.
template <int SM, int NG>
__device__ __forceinline__ void blk_load(BlkE<SM, NG>& R, int g, const Geo& G, const Bufs& B, int slot, const LuSpec& s,
                                         int mat, int p, const BlkLane& l) {
  const int N = G.N;
  const BlkSweep sw = BlkSweep::make(N, l.side);
  const char* base = (const char*)(B.SE + (size_t)slot * 4 * G.P * sw.NB * 16);
  const unsigned o = ((unsigned)(mat * G.P + p) * (unsigned)sw.NB) * 128u + (unsigned)(l.row * 4 + l.col) * 8u;
#pragma unroll
  for (int i = 0; i < SM; ++i)
    if (i < sw.S) {
      const int t = i == 0 ? sw.first(l.side) : sw.t0 + i * sw.dt;
      R.e[g][i] = *(const double*)(base + (o + (unsigned)t * 128u));
    }
  R.e[g][SM] = *(const double*)(base + (o + (unsigned)sw.S * 128u));
  R.rs[g] = -1.0 / blk_scale(s.c2);
  // row 0 reaches one column of block 1, dr0(5, 1 - S); row N-1 the columns
  // N-5 .. of block NB-2
  const MeshOff mo = MeshOff::make(N);
  const int par = ((p / G.K) * G.Mp + (s.PM != 0)) & 1;
  const int q = 4 * (sw.NB - 2) + l.row - (N - 1 - KL);
  const bool in = l.side ? q >= 0 && q <= KL : true;
  const int src = l.side ? mo.dr1 + (KL + 1) * s.BC + (in ? q : 0) : mo.dr0 + KL + (KL + 1) * (1 - par);
  const double v = G.mesh[src];
  R.bc[g] = in ? -v * R.rs[g] : 0.0;
}

// The solve of NG groups, in place.  lap: the mesh's radial Laplacian in LDS,
// row n's nine weights at lap[10 n], then a zero, rows N .. N+7 zero.  x[g]:
// the lane's right-hand side column, row n at x[g][n * xs]; rows N .. N+3
// exist and hold zeros.  All 64 lanes take part; lanes of a repeated matrix
// write the same values.
template <int SM, int NG>
__device__ __forceinline__ void blk_solve(BlkE<SM, NG>& R, int N, const BlkLane& l, const double* lap,
                                          double* const (&x)[NG], int xs) {
  const BlkSweep sw = BlkSweep::make(N, l.side);
  const int S = sw.S;
  const bool empty0 = l.side && sw.d;   // this lane's side has no block at step 0
  const int ai = l.col, ak = l.row;     // element of A
  // weights that couple a block to the one before it / after it
  const int before = ak >= ai ? ak - ai : 9, after = ak <= ai ? 8 + ak - ai : 9;
  const double* lf = lap + (4 * (sw.t0 + sw.dt) + ai) * 10 + (l.side ? after : before);
  const double* lb = lap + (4 * sw.t0 + ai) * 10 + (l.side ? before : after);
  const int ls = sw.dt * 40;
  // the lanes whose coupling entry belongs to a boundary row
  const bool bcl = l.side ? ai == ((N - 1) & 3) : ai == 0 && ak == 0;
  auto rowof = [&](int i) { return (4 * (i == 0 ? sw.first(l.side) : sw.t0 + i * sw.dt) + l.row) * xs; };
  double z[NG][SM], c[NG];
#pragma unroll
  for (int g = 0; g < NG; ++g) {
    c[g] = x[g][rowof(0)];
    if (empty0) R.e[g][0] = 0.0;
  }
#pragma unroll
  for (int i = 0; i < SM; ++i)
    if (i < S) {
      const double a = lf[i * ls];
      double b[NG];
#pragma unroll
      for (int g = 0; g < NG; ++g) b[g] = i + 1 < SM && i + 1 < S ? x[g][rowof(i + 1)] : 0.0;
#pragma unroll
      for (int g = 0; g < NG; ++g) z[g][i] = mfma4(R.e[g][i], c[g], 0.0);
#pragma unroll
      for (int g = 0; g < NG; ++g) c[g] = mfma4(a, z[g][i], b[g]);
    }
  const int om = (4 * S + l.row) * xs;
#pragma unroll
  for (int g = 0; g < NG; ++g) {
    const double bm = x[g][om];
    c[g] = bm + (c[g] + __shfl_xor(c[g], 4));   // both sides' contributions
  }
#pragma unroll
  for (int g = 0; g < NG; ++g) c[g] = mfma4(R.e[g][SM], c[g], 0.0);
#pragma unroll
  for (int g = 0; g < NG; ++g) x[g][om] = c[g] * R.rs[g];
#pragma unroll
  for (int i = SM - 1; i >= 0; --i)
    if (i < S) {
      const double a0 = lb[i * ls];
      double y[NG];
#pragma unroll
      for (int g = 0; g < NG; ++g) {
        double a = a0;
        if (i == 0) a = bcl && !empty0 ? R.bc[g] : a;
        if (i == 1) a = bcl && empty0 ? R.bc[g] : a;
        y[g] = mfma4(a, c[g], 0.0);
      }
#pragma unroll
      for (int g = 0; g < NG; ++g) c[g] = mfma4(R.e[g][i], y[g], z[g][i]);
      if (i > 0 || !empty0) {
#pragma unroll
        for (int g = 0; g < NG; ++g) x[g][rowof(i)] = c[g] * R.rs[g];
      }
    }
}

// ---------------------------------------------------------------------------
// banded LU solve (LAPACK DGBTRS 'N', KL = KU = 4), one system per lane.
// F: factor of this lane's matrix, column n at F[n*LUS] with the 13 rows of
// LAPACK band storage AB(1:13, n) (rows 9..12 hold the multipliers); pv:
// pivot offsets ipiv(j)-j; x: vector with stride xs, solved in place.  T is
// double or double2 (real and imaginary parts solved with the same factor,
// as tim_lumesh_invert does with two dgbtrs calls).
// ---------------------------------------------------------------------------
template <typename T> struct VT;
template <> struct VT<double> {
  __device__ static double zero() { return 0.0; }
  __device__ static void axpy(double& y, double a, double t) {
#pragma clang fp contract(off)
    y = y + a * t;
  }
  __device__ static double neg(double v) { return -v; }
  __device__ static double div(double v, double d) { return v / d; }
  __device__ static void sub_mul(double& y, double t, double a) {
#pragma clang fp contract(off)
    y = y - t * a;
  }
};
template <> struct VT<double2> {
  __device__ static double2 zero() { return make_double2(0.0, 0.0); }
  __device__ static void axpy(double2& y, double a, double2 t) {
#pragma clang fp contract(off)
    y.x = y.x + a * t.x;
    y.y = y.y + a * t.y;
  }
  __device__ static double2 neg(double2 v) { return make_double2(-v.x, -v.y); }
  __device__ static double2 div(double2 v, double d) { return make_double2(v.x / d, v.y / d); }
  __device__ static void sub_mul(double2& y, double2 t, double a) {
#pragma clang fp contract(off)
    y.x = y.x - t.x * a;
    y.y = y.y - t.y * a;
  }
};

template <typename T>
__device__ void lu_solve(const double* F, const unsigned char* pv, T* x, size_t xs, int N) {
  using V = VT<T>;
  // L solve with row interchanges: window w[i] = b(j+i)
  T w[5];
#pragma unroll
  for (int i = 0; i < 5; ++i) w[i] = i < N ? x[i * xs] : V::zero();
  for (int j = 0; j < N - 1; ++j) {
    const int off = pv[j];
    const T a0 = w[0];
    T s = w[0];
    s = off == 1 ? w[1] : s;
    s = off == 2 ? w[2] : s;
    s = off == 3 ? w[3] : s;
    s = off == 4 ? w[4] : s;
    w[0] = s;
    w[1] = off == 1 ? a0 : w[1];
    w[2] = off == 2 ? a0 : w[2];
    w[3] = off == 3 ? a0 : w[3];
    w[4] = off == 4 ? a0 : w[4];
    const T t = V::neg(w[0]);
    const int lm = N - 1 - j < KL ? N - 1 - j : KL;
    const double* Fj = F + (size_t)j * LUS;
#pragma unroll
    for (int i = 1; i <= KL; ++i)
      if (i <= lm) V::axpy(w[i], Fj[8 + i], t);
    x[j * xs] = w[0];
#pragma unroll
    for (int i = 0; i < 4; ++i) w[i] = w[i + 1];
    w[4] = j + 5 < N ? x[(j + 5) * xs] : V::zero();
  }
  // U solve (DTBSV upper, 8 superdiagonals): window v[q] = x(j-8+q)
  T v[9];
  const int jN = N - 1;
#pragma unroll
  for (int q = 0; q < 8; ++q) {
    const int idx = jN - 8 + q;
    v[q] = idx >= 0 ? x[idx * xs] : V::zero();
  }
  v[8] = w[0];
  for (int j = N - 1; j >= 0; --j) {
    const double* Fj = F + (size_t)j * LUS;
    v[8] = V::div(v[8], Fj[8]);
    const T t = v[8];
    x[j * xs] = t;
#pragma unroll
    for (int d = 1; d <= 8; ++d)
      if (j - d >= 0) V::sub_mul(v[8 - d], t, Fj[8 - d]);
#pragma unroll
    for (int q = 8; q >= 1; --q) v[q] = v[q - 1];
    v[0] = j - 9 >= 0 ? x[(j - 9) * xs] : V::zero();
  }
}

}  // namespace opf
