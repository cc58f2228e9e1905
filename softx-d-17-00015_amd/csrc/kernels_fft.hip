// Dealiased spectral <-> physical transforms with the u x curl(u) products.
//
// The reference transforms each radial plane with FFTW (transform.fftw3.f90:
// 65-147): a complex length-3K transform along z for every azimuthal mode
// (exponent +1 to physical space, -1 back), and a real length-3M transform
// along theta for every z line, with the 3/2 zero padding and truncation done
// by copies.  Here the same DFTs run as LDS-resident Stockham FFTs in three
// kernels with intermediates laid out for coalesced access:
//
//   k_zfwd : 6 coll fields (u, curl u) -> Yf[slot][n][z][6][M]   (z transform)
//   k_theta: Yf -> theta transforms, products, scaling, inverse theta
//            transforms -> Yb[slot][n][z][3][M]
//   k_zbwd : Yb -> z transform, truncation -> Nraw coll fields
//
// For grids whose radial plane fits in LDS, k_plane runs the same three
// stages for one plane in one workgroup, with Yf and Yb kept in LDS.
//
// The padding, the m = 0 Hermitian fill and the coll <-> spec layout change
// (variables.f90:184-294) are folded into the loads and stores.  Two real
// theta transforms share one complex FFT (a + ib), so the three c2r
// transforms per pair of fields and the r2c transforms run as 3 + 2 complex
// FFTs per line.
//
// Every pass is one radix-R butterfly per thread (R up to 16, built from
// radix 2/3/4 DFTs in registers), so the lengths 3K, 3M of the usual grids
// take two or three passes.  The first pass reads its input straight from
// global memory and the last one hands its output on in registers, so a
// length of two passes crosses LDS once.  In the theta kernel the last pass
// towards physical space holds, for one j, the points j + r L/R of the three
// packed transforms: the products follow in registers, and those points are
// also one first-pass butterfly of the way back.
//
// The intermediates are blocked by four z: value (z, field f, m) of a plane
// with F fields lies at (((z / 4) F + f) M + m) 4 + z % 4, so that the z
// kernels, which hold runs of z for a few m, and the theta kernel, which holds
// a few z for all m, both move runs of at least 64 bytes.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <type_traits>

#include "kernels.hpp"

// no contraction by the compiler: the kernels that share a transform round alike
#pragma clang fp contract(off)

namespace opf {

extern __shared__ double2 smem[];

namespace {

// 1 - r^2 with the product rounded before the difference, as the
// reference's host arithmetic does (no fused multiply-add)
__device__ __forceinline__ double one_minus_sq(double r) {
#pragma clang fp contract(off)
  return 1.0 - r * r;
}

// a * (w.x + i SG w.y)
template <int SG>
__device__ __forceinline__ double2 cmul_tw(double2 a, double2 w) {
  return SG > 0 ? make_double2(fma(a.x, w.x, -(a.y * w.y)), fma(a.x, w.y, a.y * w.x))
                : make_double2(fma(a.x, w.x, a.y * w.y), fma(a.y, w.x, -(a.x * w.y)));
}

// a * exp(2 pi i SG D / 720), D half degrees
template <int SG, int D>
__device__ __forceinline__ double2 cmul_deg(double2 a) {
  constexpr int E = D % 720;
  if constexpr (E == 0) return a;
  else if constexpr (E >= 360) {
    const double2 b = cmul_deg<SG, E - 360>(a);
    return make_double2(-b.x, -b.y);
  } else if constexpr (E >= 180) {
    const double2 b = cmul_deg<SG, E - 180>(a);
    return SG > 0 ? make_double2(-b.y, b.x) : make_double2(b.y, -b.x);
  } else if constexpr (E == 90) {
    constexpr double c = 0.70710678118654757;   // cos(pi/4)
    return SG > 0 ? make_double2(c * (a.x - a.y), c * (a.x + a.y)) : make_double2(c * (a.x + a.y), c * (a.y - a.x));
  } else {
    // cosine and sine of 22.5, 30, 40, 60, 67.5, 70 and 80 degrees
    static_assert(E == 45 || E == 60 || E == 80 || E == 120 || E == 135 || E == 140 || E == 160,
                  "angles of the radices");
    constexpr double c = E == 45    ? 0.92387953251128674
                         : E == 60  ? 0.8660254037844386
                         : E == 80  ? 0.76604444311897801
                         : E == 120 ? 0.5
                         : E == 135 ? 0.38268343236508978
                         : E == 140 ? 0.34202014332566871
                                    : 0.17364817766693036;
    constexpr double n = E == 45    ? 0.38268343236508978
                         : E == 60  ? 0.5
                         : E == 80  ? 0.64278760968653936
                         : E == 120 ? 0.8660254037844386
                         : E == 135 ? 0.92387953251128674
                         : E == 140 ? 0.93969262078590843
                                    : 0.98480775301220802;
    return cmul_tw<SG>(a, make_double2(c, n));
  }
}

template <int R, int SG> __device__ __forceinline__ void dft(double2* v) {
  if constexpr (R == 2) {
    const double2 a = v[0], b = v[1];
    v[0] = make_double2(a.x + b.x, a.y + b.y);
    v[1] = make_double2(a.x - b.x, a.y - b.y);
  } else if constexpr (R == 3) {
    constexpr double s3 = SG * 0.8660254037844386;  // SG * sin(2 pi / 3)
    const double2 a = v[0], b = v[1], c = v[2];
    const double2 t1 = make_double2(b.x + c.x, b.y + c.y);
    const double2 t2 = make_double2(fma(-0.5, t1.x, a.x), fma(-0.5, t1.y, a.y));
    const double2 t3 = make_double2(b.x - c.x, b.y - c.y);
    v[0] = make_double2(a.x + t1.x, a.y + t1.y);
    // X1 = t2 + i s3 t3, X2 = t2 - i s3 t3
    v[1] = make_double2(fma(-s3, t3.y, t2.x), fma(s3, t3.x, t2.y));
    v[2] = make_double2(fma(s3, t3.y, t2.x), fma(-s3, t3.x, t2.y));
  } else if constexpr (R == 4) {
    const double2 a = v[0], b = v[1], c = v[2], d = v[3];
    const double2 s02 = make_double2(a.x + c.x, a.y + c.y);
    const double2 d02 = make_double2(a.x - c.x, a.y - c.y);
    const double2 s13 = make_double2(b.x + d.x, b.y + d.y);
    const double2 d13 = make_double2(b.x - d.x, b.y - d.y);
    v[0] = make_double2(s02.x + s13.x, s02.y + s13.y);
    v[2] = make_double2(s02.x - s13.x, s02.y - s13.y);
    // d02 +- SG i d13
    v[SG > 0 ? 1 : 3] = make_double2(d02.x - d13.y, d02.y + d13.x);
    v[SG > 0 ? 3 : 1] = make_double2(d02.x + d13.y, d02.y - d13.x);
  }
}

// Radix R = R1 * R2 (R1, R2 <= 4) as R2 DFTs of length R1, the internal
// twiddles W_R^(n2 k1) and R1 DFTs of length R2 (Cooley-Tukey): input n =
// R2 n1 + n2, output k = k1 + R1 k2.  Computed in place: output k is left in
// v[perm<R>(k)], perm(k1 + R1 k2) = R2 k1 + k2.
template <int R> struct Split;
template <> struct Split<1> { static constexpr int R1 = 1, R2 = 1; };
template <> struct Split<2> { static constexpr int R1 = 2, R2 = 1; };
template <> struct Split<3> { static constexpr int R1 = 3, R2 = 1; };
template <> struct Split<4> { static constexpr int R1 = 4, R2 = 1; };
template <> struct Split<6> { static constexpr int R1 = 3, R2 = 2; };
template <> struct Split<8> { static constexpr int R1 = 4, R2 = 2; };
template <> struct Split<9> { static constexpr int R1 = 3, R2 = 3; };
template <> struct Split<12> { static constexpr int R1 = 4, R2 = 3; };
template <> struct Split<16> { static constexpr int R1 = 4, R2 = 4; };

template <int R>
__host__ __device__ constexpr int perm(int k) {
  return Split<R>::R2 * (k % Split<R>::R1) + k / Split<R>::R1;
}

template <int R, int SG, int X>   // v[R2 k1 + n2] *= W_R^(n2 k1) for X = R2 k1 + n2 and up
__device__ __forceinline__ void bfly_tw(double2 (&v)[R]) {
  constexpr int R1 = Split<R>::R1, R2 = Split<R>::R2;
  if constexpr (X < R1 * R2) {
    v[X] = cmul_deg<SG, (X % R2) * (X / R2) * (720 / R)>(v[X]);
    bfly_tw<R, SG, X + 1>(v);
  }
}

template <int R, int SG>
__device__ __forceinline__ void bfly(double2 (&v)[R]) {
  constexpr int R1 = Split<R>::R1, R2 = Split<R>::R2;
  if constexpr (R2 == 1) {
    dft<R1, SG>(v);
  } else {
#pragma unroll
    for (int n2 = 0; n2 < R2; ++n2) {
      double2 a[R1];
#pragma unroll
      for (int n1 = 0; n1 < R1; ++n1) a[n1] = v[R2 * n1 + n2];
      dft<R1, SG>(a);
#pragma unroll
      for (int k1 = 0; k1 < R1; ++k1) v[R2 * k1 + n2] = a[k1];
    }
    bfly_tw<R, SG, 0>(v);
#pragma unroll
    for (int k1 = 0; k1 < R1; ++k1) {
      double2 a[R2];
#pragma unroll
      for (int n2 = 0; n2 < R2; ++n2) a[n2] = v[R2 * k1 + n2];
      dft<R2, SG>(a);
#pragma unroll
      for (int k2 = 0; k2 < R2; ++k2) v[R2 * k1 + k2] = a[k2];
    }
  }
}

// LDS layout of a batch of transforms of length L: a transform's input,
// element i of transform b, at buf[b*Lp + i] (linear), its output at
// buf[b*Lp + pidx(i)], pidx(i) = i + i/16, Lp = padded_len(L).  The pad
// spreads the stride-R writes of the first Stockham pass over the LDS
// banks; the first pass reads the linear input, whose stride-L/R reads
// fall on consecutive addresses across a wave, with constant offsets.
__host__ __device__ __forceinline__ int pidx(int i) { return i + (i >> 4); }

// One Stockham pass of radix R over B transforms of a run-time length L
// (B * L <= FFT_TILE; LIN: the first pass, reading the linear input layout
// buf[b*Lp + i]).  Ns = product of the radices of the previous passes (the
// twiddles of the first pass are all 1 and skipped); tw: the length-L twiddle
// table in LDS.  Outer twiddles are fetched four at a time to bound register
// use.
template <int R, int SG, bool LIN>
__device__ __forceinline__ void fft_pass(double2* buf, int L, int B, int Ns, const double2* tw) {
  constexpr int NT = FFT_THREADS;
  constexpr int MB = (3 * THETA_ITEMS + R * NT - 1) / (R * NT);
  const int Lp = padded_len(L);
  const int nb = L / R;
  const int total = nb * B;
  const int tid = threadIdx.x;
  const int stride_tw = L / (Ns * R);
  double2 v[MB][R];
  int dst[MB];
#pragma unroll
  for (int i = 0; i < MB; ++i) {
    const int q = tid + i * NT;
    dst[i] = -1;
    if (q < total) {
      const int b = q / nb, j = q - b * nb;
      const double2* x = buf + b * Lp;
      const int kk = j % Ns;
#pragma unroll
      for (int r = 0; r < R; ++r) v[i][r] = LIN ? x[j + r * nb] : x[pidx(j + r * nb)];
      if (Ns > 1) {
#pragma unroll
        for (int g = 1; g < R; g += 4) {
          __builtin_amdgcn_sched_barrier(0);
          double2 w[4];
#pragma unroll
          for (int u = 0; u < 4; ++u)
            if (g + u < R) w[u] = tw[kk * (g + u) * stride_tw];
#pragma unroll
          for (int u = 0; u < 4; ++u)
            if (g + u < R) v[i][g + u] = cmul_tw<SG>(v[i][g + u], w[u]);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
      bfly<R, SG>(v[i]);
      dst[i] = b * Lp + (j / Ns) * Ns * R + kk;
    }
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < MB; ++i) {
    if (dst[i] >= 0) {
      const int b = (tid + i * NT) / nb;
      const int e = dst[i] - b * Lp;          // unpadded index of output 0
      double2* x = buf + b * Lp;
#pragma unroll
      for (int r = 0; r < R; ++r) x[pidx(e + r * Ns)] = v[i][perm<R>(r)];
    }
  }
  __syncthreads();
}

// Full transform of a run-time plan: SG = +1 (to physical space) or -1,
// unnormalised (FFTW).
template <int SG>
__device__ __forceinline__ void fft_lds(double2* buf, int B, const FftPlan& pl, const double2* tw) {
  auto pass = [&](auto lin, int R, int Ns) {
    constexpr bool LN = decltype(lin)::value;
    switch (R) {
      case 16: fft_pass<16, SG, LN>(buf, pl.L, B, Ns, tw); break;
      case 12: fft_pass<12, SG, LN>(buf, pl.L, B, Ns, tw); break;
      case 9: fft_pass<9, SG, LN>(buf, pl.L, B, Ns, tw); break;
      case 8: fft_pass<8, SG, LN>(buf, pl.L, B, Ns, tw); break;
      case 6: fft_pass<6, SG, LN>(buf, pl.L, B, Ns, tw); break;
      case 4: fft_pass<4, SG, LN>(buf, pl.L, B, Ns, tw); break;
      case 3: fft_pass<3, SG, LN>(buf, pl.L, B, Ns, tw); break;
      default: fft_pass<2, SG, LN>(buf, pl.L, B, Ns, tw); break;
    }
  };
  pass(std::true_type{}, pl.rad[0], 1);
  int Ns = pl.rad[0];
  for (int p = 1; p < pl.nrad; ++p) {
    pass(std::false_type{}, pl.rad[p], Ns);
    Ns *= pl.rad[p];
  }
}

// A transform of the fixed radix sequence F, MID (1: none), LA (1: none)
// whose passes exchange through LDS.  The first pass' butterfly j takes the
// inputs j + r JF and leaves its outputs as row j of an (L/F) x F table with
// rows of odd pitch (lanes of consecutive j write without bank conflicts); a
// middle pass turns it into an LA x (F MID) table; butterfly j of the last
// pass reads column j and returns the outputs j + r JL.
template <int F_, int MID_, int LA_>
struct Seq {
  static constexpr int F = F_, MID = MID_, LA = LA_;
  static constexpr int L = F * MID * LA, JF = L / F, JM = L / MID, JL = L / LA;
  static constexpr int P1 = F | 1, P2 = (F * MID) | 1, PL = MID > 1 ? P2 : P1;
  static constexpr int SIZE = JF * P1 > (MID > 1 ? LA * P2 : 0) ? JF * P1 : LA * P2;
  static_assert(JF * P1 <= SIZE && LA * PL <= SIZE && F <= P1 && JL <= PL, "each pass' table within the transform's part");
};
// the smallest size >= n with size % 8 == r: the distance of two transforms in
// LDS, such that the lanes of a few transforms share no bank
constexpr int lds_step(int n, int r) { return n + ((r - n) % 8 + 8) % 8; }

template <class S, int SG>
__device__ __forceinline__ void fft_first(double2 (&v)[S::F], double2* x, int j) {
  bfly<S::F, SG>(v);
#pragma unroll
  for (int r = 0; r < S::F; ++r) x[j * S::P1 + r] = v[perm<S::F>(r)];
}
// W column j's inputs at distance D (double2) of W transforms that share twiddles
template <class S, int SG, int W = 1>
__device__ __forceinline__ void fft_last(double2 (&v)[W][S::LA], const double2* x, int D, int j, const double2* tw) {
#pragma unroll
  for (int p = 0; p < W; ++p)
#pragma unroll
    for (int r = 0; r < S::LA; ++r) v[p][r] = x[p * D + r * S::PL + j];
#pragma unroll
  for (int r = 1; r < S::LA; ++r) {
    const double2 w = tw[j * r];
#pragma unroll
    for (int p = 0; p < W; ++p) v[p][r] = cmul_tw<SG>(v[p][r], w);
  }
#pragma unroll
  for (int p = 0; p < W; ++p) bfly<S::LA, SG>(v[p]);
}
// the middle pass of nt <= NTR transforms at distance D, barriers included
template <class S, int SG, int NT, int NTR>
__device__ __forceinline__ void fft_mid(double2* x, int D, int nt, const double2* tw) {
  if constexpr (S::MID > 1) {
    constexpr int MB = (NTR * S::JM + NT - 1) / NT;
    double2 v[MB][S::MID];
#pragma unroll
    for (int u = 0; u < MB; ++u) {
      const int q = threadIdx.x + u * NT, t = q / S::JM, j = q - t * S::JM;
      if (t >= nt) continue;
      const int jr = j / S::F, jc = j - jr * S::F;
#pragma unroll
      for (int r = 0; r < S::MID; ++r) v[u][r] = x[t * D + (jr + r * S::LA) * S::P1 + jc];
#pragma unroll
      for (int r = 1; r < S::MID; ++r) v[u][r] = cmul_tw<SG>(v[u][r], tw[jc * r * S::LA]);
      bfly<S::MID, SG>(v[u]);
    }
    __syncthreads();
#pragma unroll
    for (int u = 0; u < MB; ++u) {
      const int q = threadIdx.x + u * NT, t = q / S::JM, j = q - t * S::JM;
      if (t >= nt) continue;
      const int jr = j / S::F, jc = j - jr * S::F;
#pragma unroll
      for (int r = 0; r < S::MID; ++r) x[t * D + jr * S::P2 + jc + r * S::F] = v[u][perm<S::MID>(r)];
    }
    __syncthreads();
  }
}

// value (z, field f, m) of a plane of the intermediates
__device__ __forceinline__ int yoff(int z, int NF, int f, int M, int m) {
  return (((z >> 2) * NF + f) * M + m) * 4 + (z & 3);
}

// twiddle table of length L into LDS
template <int NT = FFT_THREADS>
__device__ __forceinline__ void load_tw(double2* twl, const double2* tw, int L) {
  for (int i = threadIdx.x; i < L; i += NT) twl[i] = tw[i];
}

// spectral coefficient (k, m) at radial row `row` of a coll field, k in
// (-K, K); for m = 0 the k < 0 half is the conjugate of k > 0
// (transform.fftw3.f90:72-74).
__device__ __forceinline__ double2 coef(const double2* row, int K, int k, int m) {
  if (m == 0) {
    if (k >= 0) return row[k];
    const double2 c = row[-k];
    return make_double2(c.x, -c.y);
  }
  return row[K + (m - 1) * (2 * K - 1) + k + K - 1];
}

// the kernels of any length: two waves of every SIMD, at up to 256 registers
#define ANY_LENGTH __launch_bounds__(FFT_THREADS) __attribute__((amdgpu_waves_per_eu(2)))

// Padded z columns of modes m0 .. m0+tm-1 into the tile: X(j) = a(k=j)
// for j < K, X(Z+k) = a(k) for k < 0, zero in between
// (transform.fftw3.f90:72-84).  A tile holds at most FFT_TILE values, so
// every thread issues its (at most ZLD) loads in one batch.
constexpr int ZLD = FFT_TILE / FFT_THREADS;
__device__ __forceinline__ void load_zcols(double2* buf, const double2* row, int K, int Z, int Zp, int m0, int tm) {
  const int nk = 2 * K - 1;
  const int total = tm * nk;
  double2 v[ZLD];
  int d[ZLD];
#pragma unroll
  for (int u = 0; u < ZLD; ++u) {
    const int i = threadIdx.x + u * FFT_THREADS;
    const bool ok = i < total;
    const int ic = ok ? i : 0;
    const int b = ic / nk, e = ic - b * nk;
    const int k = e - (K - 1);
    v[u] = coef(row, K, k, m0 + b);
    d[u] = ok ? b * Zp + (k >= 0 ? k : k + Z) : -1;
  }
#pragma unroll
  for (int u = 0; u < ZLD; ++u)
    if (d[u] >= 0) buf[d[u]] = v[u];
  const int nzero = K + 1;   // j = K .. 2K
  for (int i = threadIdx.x; i < tm * nzero; i += FFT_THREADS) {
    const int b = i / nzero, j = K + (i - b * nzero);
    buf[b * Zp + j] = make_double2(0.0, 0.0);
  }
}

// column b of the tile (linear input layout) = Y[at(z, m0 + b)], one batch
template <typename At>
__device__ __forceinline__ void load_ycols(double2* buf, const double2* Y, At at, int Z, int Zp, int m0, int tm) {
  const int total = tm * Z;
  double2 v[ZLD];
  int d[ZLD];
#pragma unroll
  for (int u = 0; u < ZLD; ++u) {
    const int i = threadIdx.x + u * FFT_THREADS;
    const bool ok = i < total;
    const int ic = ok ? i : 0;
    const int z = ic / tm, b = ic - z * tm;
    v[u] = Y[at(z, m0 + b)];
    d[u] = ok ? b * Zp + z : -1;
  }
#pragma unroll
  for (int u = 0; u < ZLD; ++u)
    if (d[u] >= 0) buf[d[u]] = v[u];
}

// truncation of a z column to the 2K-1 retained k into a coll row
__device__ __forceinline__ void store_zcol(double2* row, const double2* buf, int K, int Z, int m, int tid, int nth) {
  if (m == 0) {
    for (int k = tid; k < K; k += nth) row[k] = buf[pidx(k)];
  } else {
    double2* blk = row + K + (m - 1) * (2 * K - 1) + (K - 1);
    for (int k = tid - (K - 1); k < K; k += nth) blk[k] = buf[pidx(k >= 0 ? k : k + Z)];
  }
}

}  // namespace

// ---------------------------------------------------------------------------
// z transforms.  grid: x = 8 * per >= (m tile, plane, field) tiles, z = slot.
// XCD-aware tiles: launch order b goes to XCD b % 8, so tile t = (b % 8) per +
// b / 8 keeps runs of neighbouring m tiles, which share cache lines of the
// coll rows, on one XCD's L2; spare blocks return.
//
// Tile widths: as many m columns as give every thread of a pass about one
// butterfly, with 128 threads for two passes and 256 for three.
// ---------------------------------------------------------------------------
template <int F, int MID, int LA>
struct ZTile {
  using S = Seq<F, MID, LA>;
  static constexpr int NT = MID > 1 ? 256 : 128;
  static constexpr int JX = S::JF > (MID > 1 ? S::JM : S::JL) ? S::JF : (MID > 1 ? S::JM : S::JL);
  static constexpr int TM = NT / JX;               // m columns
  static constexpr int D = lds_step(S::SIZE, 4);   // four lanes of a column, then the next column
  // the forward kernel of three passes copies the twiddles into LDS
  static constexpr bool LTW = MID > 1;
  static constexpr size_t smem_b = (size_t)(TM * D) * sizeof(double2);
  static constexpr size_t smem_f = smem_b + (LTW ? S::L * sizeof(double2) : 0);
  static_assert(JX <= NT, "a middle pass runs in one round");
};

struct ZWhere {
  int n, f, m0, tm;
};
// the tile of this workgroup (NF fields); false: a spare block
__device__ __forceinline__ bool ztile(const Geo& G, int tmw, int NF, ZWhere& w) {
  const int gx = (G.M + tmw - 1) / tmw, ntile = gx * NF * G.N;
  const int per = (ntile + 7) / 8;
  const int tile = (int)(blockIdx.x % 8) * per + (int)(blockIdx.x / 8);
  if (tile >= ntile) return false;
  const int ty = tile / gx, tx = tile - ty * gx;
  w.n = ty / NF;
  w.f = ty - w.n * NF;
  w.m0 = tx * tmw;
  w.tm = min(tmw, G.M - w.m0);
  return true;
}

// Padded z columns of modes m0 .. of a coll row (X(j) = a(k=j) for j < K,
// X(Z+k) = a(k) for k < 0, zero in between, transform.fftw3.f90:72-84; for
// m = 0 the k < 0 half is the conjugate of k > 0) as first-pass butterflies.
template <class S>
__device__ __forceinline__ void zcol_input(double2 (&v)[S::F], const double2* row, int m, int j) {
  constexpr int Z = S::L, K = Z / 3;
  const int base = K + (m - 1) * (2 * K - 1) + K - 1;
  // all loads in one batch: those of zeros go to the row's first value
#pragma unroll
  for (int r = 0; r < S::F; ++r) {
    v[r] = make_double2(0.0, 0.0);
    if (r * S::JF >= K && (r + 1) * S::JF - 1 <= Z - K) continue;   // zero for every j
    const int i = j + r * S::JF, k = i < K ? i : i - Z;
    v[r] = row[i < K || i > Z - K ? (m == 0 ? abs(k) : base + k) : 0];
  }
#pragma unroll
  for (int r = 0; r < S::F; ++r) {
    if (r * S::JF >= K && (r + 1) * S::JF - 1 <= Z - K) continue;
    const int i = j + r * S::JF;
    if (i >= K && i <= Z - K) v[r] = make_double2(0.0, 0.0);
    if (i >= K && m == 0) v[r].y = -v[r].y;
  }
}
// output r of last-pass butterfly j of a column of mode m, where k is retained
template <class S>
__device__ __forceinline__ void zcol_output(double2* row, const double2 (&v)[S::LA], int m, int j) {
  constexpr int Z = S::L, K = Z / 3;
  const int base = K + (m - 1) * (2 * K - 1) + K - 1;
#pragma unroll
  for (int r = 0; r < S::LA; ++r) {
    if (r * S::JL >= K && (r + 1) * S::JL - 1 <= Z - K) continue;
    const int i = j + r * S::JL, k = i < K ? i : i - Z;
    if (i < K || i > Z - K) {
      if (m > 0) row[base + k] = v[perm<S::LA>(r)];
      else if (k >= 0) row[k] = v[perm<S::LA>(r)];
    }
  }
}

// columns of a tile from a coll row to Y (F: offset of (z, m))
template <int F, int MID, int LA, typename At>
__device__ __forceinline__ void zfwd_tile(const double2* row, double2* Y, At at, int m0, int tm, const double2* tw) {
  using C = ZTile<F, MID, LA>;
  using S = typename C::S;
  double2* buf = smem;
  double2* twc = smem + C::TM * C::D;
  const double2* twl = C::LTW ? twc : tw;
  {
    const int b = threadIdx.x / S::JF, j = threadIdx.x - b * S::JF;
    double2 v[F];
    if (b < tm) zcol_input<S>(v, row, m0 + b, j);
    if (C::LTW) load_tw<C::NT>(twc, tw, S::L);
    if (b < tm) fft_first<S, 1>(v, buf + b * C::D, j);
  }
  __syncthreads();
  fft_mid<S, 1, C::NT, C::TM>(buf, C::D, tm, twl);
  constexpr int J4 = (S::JL + 3) / 4;
#pragma unroll
  for (int q0 = 0; q0 < 4 * J4 * C::TM; q0 += C::NT) {
    const int q = threadIdx.x + q0, b = (q >> 2) % C::TM, j = (q >> 2) / C::TM * 4 + (q & 3);
    if (j >= S::JL || b >= tm) continue;
    double2 v[1][LA];
    fft_last<S, 1>(v, buf + b * C::D, 0, j, twl);
#pragma unroll
    for (int r = 0; r < LA; ++r) Y[at(j + r * S::JL, m0 + b)] = v[0][perm<LA>(r)];
  }
}
template <int F, int MID, int LA, typename At>
__device__ __forceinline__ void zbwd_tile(const double2* Y, At at, double2* row, int m0, int tm, const double2* tw) {
  using C = ZTile<F, MID, LA>;
  using S = typename C::S;
  double2* buf = smem;
  constexpr int J4 = (S::JF + 3) / 4, R0 = (4 * J4 * C::TM + C::NT - 1) / C::NT;
  {
    double2 v[R0][F];
#pragma unroll
    for (int u = 0; u < R0; ++u) {
      const int q = threadIdx.x + u * C::NT, b = (q >> 2) % C::TM, j = (q >> 2) / C::TM * 4 + (q & 3);
      if (j >= S::JF || b >= tm) continue;
#pragma unroll
      for (int r = 0; r < F; ++r) v[u][r] = Y[at(j + r * S::JF, m0 + b)];
    }
#pragma unroll
    for (int u = 0; u < R0; ++u) {
      const int q = threadIdx.x + u * C::NT, b = (q >> 2) % C::TM, j = (q >> 2) / C::TM * 4 + (q & 3);
      if (j < S::JF && b < tm) fft_first<S, -1>(v[u], buf + b * C::D, j);
    }
  }
  __syncthreads();
  fft_mid<S, -1, C::NT, C::TM>(buf, C::D, tm, tw);
#pragma unroll
  for (int q0 = 0; q0 < S::JL * C::TM; q0 += C::NT) {
    const int q = threadIdx.x + q0, b = q / S::JL, j = q - b * S::JL;
    if (b >= tm) continue;
    double2 v[1][LA];
    fft_last<S, -1>(v, buf + b * C::D, 0, j, tw);
    zcol_output<S>(row, v[0], m0 + b, j);
  }
}

// u and curl u of all active slots -> Yf
template <int F, int MID, int LA>
__global__ void __launch_bounds__((ZTile<F, MID, LA>::NT)) k_zfwd_t(Geo G, Bufs B, FftTiles T, int slot0) {
  using C = ZTile<F, MID, LA>;
  const int slot = slot_of(B, slot0);
  const SlotCtl* c = &B.ctl[slot];
  if (!c->active) return;
  // a new evaluation: clear the slot's per-plane velocity maxima (the theta
  // kernel that follows records them)
  if (blockIdx.x == 0)
    for (int i = threadIdx.x; i < 3 * G.N; i += C::NT) B.cflmax[(size_t)slot * 3 * G.N + i] = 0ull;
  ZWhere w;
  if (!ztile(G, T.tm, 6, w)) return;
  const int M = G.M, f = w.f;
  const double2* row = (f < 3 ? B.U[c->ucur] : B.om) + ((size_t)slot * 3 + (f < 3 ? f : f - 3)) * G.coll + (size_t)w.n * G.Hp;
  double2* Y = B.Yf + ((size_t)slot * G.N + w.n) * G.ZQ * 6 * M;
  zfwd_tile<F, MID, LA>(row, Y, [=](int z, int m) { return yoff(z, 6, f, M, m); }, w.m0, w.tm, B.twZ);
}
// Yb -> truncated raw nonlinear terms
template <int F, int MID, int LA>
__global__ void __launch_bounds__((ZTile<F, MID, LA>::NT)) k_zbwd_t(Geo G, Bufs B, FftTiles T, int slot0) {
  const int slot = slot_of(B, slot0);
  const SlotCtl* c = &B.ctl[slot];
  if (!c->active) return;
  ZWhere w;
  if (!ztile(G, T.tm, 3, w)) return;
  const int M = G.M, f = w.f;
  const double2* Y = B.Yb + ((size_t)slot * G.N + w.n) * G.ZQ * 3 * M;
  double2* row = B.Nraw[c->ncur] + ((size_t)slot * 3 + f) * G.coll + (size_t)w.n * G.Hp;
  zbwd_tile<F, MID, LA>(Y, [=](int z, int m) { return yoff(z, 3, f, M, m); }, row, w.m0, w.tm, B.twZ);
}

// products (velocity.f90:325-329) at one physical point of radial plane n,
// scaled as tra_phys2spec (:114-117), and the running maxima of |u_r|,
// |u_t|, |u_z + 1 - r^2| for vel_maxtstep (velocity.f90:464-475).  Inputs:
// the packed transforms' values (u_r, u_t), (u_z, w_r), (w_t, w_z); outputs
// (N_r, N_t) and N_z.  One definition for every kernel that forms them, so
// they round alike.
struct NlPlane {
  double scale, ubase, cor_d1, cor_s, cor_c;
  bool cor;
  __device__ static NlPlane make(const Geo& G, const Bufs& B, int slot, int n, int TT) {
    NlPlane p;
    p.scale = 1.0 / (double)(G.Z * TT);
    p.ubase = one_minus_sq(G.mesh[MeshOff::make(G.N).r + n]);
    p.cor = B.prm[slot].coriolis != 0;
    p.cor_d1 = B.prm[slot].cor_d1;
    p.cor_s = B.prm[slot].cor_sphi;
    p.cor_c = B.prm[slot].cor_cphi;
    return p;
  }
  __device__ __forceinline__ void point(double2 w0, double2 w1, double2 w2, const double2* twl, int th, double& mr,
                                        double& mt, double& mz, double2& nrt, double& nz) const {
    const double ur = w0.x, ut = w0.y, uz = w1.x, cr = w1.y, ct = w2.x, cz = w2.y;
    mr = fmax(mr, fabs(ur));
    mt = fmax(mt, fabs(ut));
    mz = fmax(mz, fabs(uz + ubase));
    double Nr = fma(ut, cz, -(uz * ct));
    double Nt = fma(uz, cr, -(ur * cz));
    double Nz = fma(ur, ct, -(ut * cr));
    if (cor) {   // Coriolis.f90:62-68: N += -1/(4 Ro) Omega^ x (U + u)
      const double2 cs = twl[th];   // (cos, sin)(2 pi th / T)
      const double Or = cor_s * cs.x, Ot = -cor_s * cs.y;
      const double uzU = uz + ubase;
      Nr = fma(cor_d1, fma(Ot, uzU, -(cor_c * ut)), Nr);
      Nt = fma(cor_d1, fma(cor_c, ur, -(Or * uzU)), Nt);
      Nz = fma(cor_d1, fma(Or, ut, -(Ot * ur)), Nz);
    }
    nrt = make_double2(scale * Nr, scale * Nt);
    nz = scale * Nz;
  }
};

// the workgroup's velocity maxima (NT threads) into out[0], out[N], out[2N].
// Maxima are exact and order free: non-negative doubles order like their bit
// patterns, so one integer atomic max per workgroup and component, or a store
// where the workgroup has the whole plane (ALL).
template <int NT, bool ALL = false>
__device__ __forceinline__ void plane_maxima(double mr, double mt, double mz, unsigned long long* out, int N) {
  __shared__ double wmax[3][NT / 64];
  for (int off = 32; off >= 1; off >>= 1) {
    mr = fmax(mr, __shfl_xor(mr, off));
    mt = fmax(mt, __shfl_xor(mt, off));
    mz = fmax(mz, __shfl_xor(mz, off));
  }
  if ((threadIdx.x & 63) == 0) {
    wmax[0][threadIdx.x >> 6] = mr;
    wmax[1][threadIdx.x >> 6] = mt;
    wmax[2][threadIdx.x >> 6] = mz;
  }
  __syncthreads();
  if (threadIdx.x < 3) {
    double v = 0.0;
    for (int w = 0; w < NT / 64; ++w) v = fmax(v, wmax[threadIdx.x][w]);
    const unsigned long long bits = (unsigned long long)__double_as_longlong(v);
    if (ALL) out[(size_t)threadIdx.x * N] = bits;
    else atomicMax(out + (size_t)threadIdx.x * N, bits);
  }
}

// the value of the neighbouring lane (l ^ 1)
__device__ __forceinline__ double lane_pair(double x) {
  const int lo = __builtin_amdgcn_mov_dpp(__double2loint(x), 0xB1, 0xf, 0xf, true);
  const int hi = __builtin_amdgcn_mov_dpp(__double2hiint(x), 0xB1, 0xf, 0xf, true);
  return __hiloint2double(hi, lo);
}

// ---------------------------------------------------------------------------
// theta transforms and products, TZ z-lines per workgroup.  Towards physical
// space: (u_r,u_t), (u_z,w_r), (w_t,w_z) packed as a + ib into Hermitian
// spectra; back: (N_r,N_t) of each line as one transform, N_z of lines 2q and
// 2q + 1 as another (a last line without a partner pairs with zero).
// ---------------------------------------------------------------------------
template <int F, int MID, int LA>
struct ThetaTile {
  using S = Seq<F, MID, LA>;   // to physical space
  using I = Seq<LA, MID, F>;   // and back
  static constexpr int TT = S::L, M = TT / 3;
  // lines: 3 TT values each, up to about 32 KiB of LDS
  static constexpr int TZ = TT <= 72 ? 8 : TT <= 192 ? 4 : 2;
  static constexpr int NTR = TZ + TZ / 2;          // transforms back
  static constexpr int items = 3 * TZ * S::JF > TZ * S::JL ? 3 * TZ * S::JF : TZ * S::JL;
  static constexpr int NT = MID > 1 ? 256 : items > 128 ? 192 : 128;
  static constexpr int DS = lds_step(S::SIZE, 8 / TZ), DI = lds_step(I::SIZE, 8 / TZ);
  static constexpr int DO = (2 * M - 1) | 1;       // the retained bins |m| < M of a transform back
  static constexpr int OUT = NTR * DI;             // where they stand
  static constexpr int BUF = 3 * TZ * DS > OUT + NTR * DO ? 3 * TZ * DS : OUT + NTR * DO;
  static constexpr bool LTW = MID > 1;             // twiddles copied into LDS
  static constexpr size_t smem = (size_t)(BUF + (LTW ? TT : 0)) * sizeof(double2);
};
// bins m and TT - m of the packed spectra a + ib; c2r reads only the real
// part of the m = 0 bin (transform.fftw3.f90:97-98)
__device__ __forceinline__ double2 pack_bin(double2 a, double2 b, int i, int m) {
  if (m == 0) return make_double2(a.x, b.x);
  return i == m ? make_double2(a.x - b.y, a.y + b.x) : make_double2(a.x + b.y, b.x - a.y);
}
// A(m) = (X(m) + conj X(-m))/2 or B(m) = (X(m) - conj X(-m))/2i of a packed transform back
__device__ __forceinline__ double2 unpack_bin(double2 X, double2 Xc, bool first) {
  return first ? make_double2(0.5 * (X.x + Xc.x), 0.5 * (X.y - Xc.y))
               : make_double2(0.5 * (X.y + Xc.y), -0.5 * (X.x - Xc.x));
}
// products of the points j + r JL of a line, then the first pass back: w
// becomes the butterfly of (N_r, N_t) in w[0] and of N_z (of the lines of a
// lane pair, valid in the even lane) in w[1]
template <class S>
__device__ __forceinline__ void theta_middle(double2 (&w)[3][S::LA], const NlPlane& pl, const double2* twl, int j,
                                             bool live, bool pair, double& mr, double& mt, double& mz) {
  constexpr int LA = S::LA;
  double2 a[LA], b[LA];
  double lr = 0.0, lt = 0.0, lz = 0.0;
#pragma unroll
  for (int r = 0; r < LA; ++r) {
    const int k = perm<LA>(r);
    double nz;
    pl.point(w[0][k], w[1][k], w[2][k], twl, j + r * S::JL, lr, lt, lz, a[r], nz);
    const double other = lane_pair(nz);
    b[r] = make_double2(nz, pair ? other : 0.0);
  }
  if (live) {
    mr = fmax(mr, lr);
    mt = fmax(mt, lt);
    mz = fmax(mz, lz);
  }
  bfly<LA, -1>(a);
  bfly<LA, -1>(b);
#pragma unroll
  for (int r = 0; r < LA; ++r) {
    w[0][r] = a[r];
    w[1][r] = b[r];
  }
}

template <int F, int MID, int LA>
__global__ void __launch_bounds__((ThetaTile<F, MID, LA>::NT)) __attribute__((amdgpu_waves_per_eu(2)))
k_theta_t(Geo G, Bufs B, FftTiles T, int slot0) {
  using C = ThetaTile<F, MID, LA>;
  using S = typename C::S;
  using I = typename C::I;
  constexpr int TT = C::TT, M = C::M, TZ = C::TZ, NT = C::NT;
  const int slot = slot_of(B, slot0);
  const SlotCtl* c = &B.ctl[slot];
  if (!c->active) return;
  // XCD-aware tiles as in the z kernels: neighbouring tiles share cache lines
  // of the intermediates where a tile has less than four lines
  const int gz = (G.Z + T.tz - 1) / T.tz, per = (gz * G.N + 7) / 8;
  const int tile = (int)(blockIdx.x % 8) * per + (int)(blockIdx.x / 8);
  if (tile >= gz * G.N) return;
  const int n = tile / gz;
  const int z0 = (tile - n * gz) * T.tz;
  const int tz = min(T.tz, G.Z - z0);
  const double2* Yf = B.Yf + ((size_t)slot * G.N + n) * G.ZQ * 6 * M;
  double2* Yb = B.Yb + ((size_t)slot * G.N + n) * G.ZQ * 3 * M;
  double2* buf = smem;
  double2* twc = smem + C::BUF;
  const double2* twl = C::LTW ? twc : B.twT;
  // the packed spectra as first-pass butterflies, lines on neighbouring lanes
  constexpr int NA = 3 * TZ * S::JF;
#pragma unroll
  for (int q0 = 0; q0 < NA; q0 += NT) {
    const int q = threadIdx.x + q0, line = q % TZ, rest = q / TZ, j = rest % S::JF, p = rest / S::JF;
    double2 v[F], bv[F];
    const bool live = line < tz && q < NA;
    const double2* src = Yf + (live ? yoff(z0 + line, 6, 2 * p, M, 0) : 0);
    // all loads in one batch: those of zeros go to m = 0
#pragma unroll
    for (int r = 0; r < F; ++r) {
      v[r] = bv[r] = make_double2(0.0, 0.0);
      if (r * S::JF >= M && (r + 1) * S::JF - 1 <= TT - M) continue;
      const int i = j + r * S::JF, m = i < M ? i : i > TT - M ? TT - i : 0;
      v[r] = src[4 * m];
      bv[r] = src[4 * (M + m)];
    }
#pragma unroll
    for (int r = 0; r < F; ++r) {
      if (r * S::JF >= M && (r + 1) * S::JF - 1 <= TT - M) continue;
      const int i = j + r * S::JF, m = i < M ? i : TT - i;
      v[r] = live && (i < M || i > TT - M) ? pack_bin(v[r], bv[r], i, m) : make_double2(0.0, 0.0);
    }
    if (C::LTW && q0 == 0) load_tw<NT>(twc, B.twT, TT);
    if (q < NA) fft_first<S, 1>(v, buf + (p * TZ + line) * C::DS, j);
  }
  __syncthreads();
  fft_mid<S, 1, NT, 3 * TZ>(buf, C::DS, 3 * TZ, twl);
  const NlPlane pl = NlPlane::make(G, B, slot, n, TT);
  double mr = 0.0, mt = 0.0, mz = 0.0;
  constexpr int NB = TZ * S::JL, RB = (NB + NT - 1) / NT;
  double2 w[RB][3][LA];
#pragma unroll
  for (int u = 0; u < RB; ++u) {
    const int q = threadIdx.x + u * NT, line = q % TZ, j = q / TZ;
    if (q >= NB) continue;
    fft_last<S, 1, 3>(w[u], buf + line * C::DS, TZ * C::DS, j, twl);
    theta_middle<S>(w[u], pl, twl, j, line < tz, line + 1 < tz, mr, mt, mz);
  }
  __syncthreads();
#pragma unroll
  for (int u = 0; u < RB; ++u) {
    const int q = threadIdx.x + u * NT, line = q % TZ, j = q / TZ;
    if (q >= NB) continue;
#pragma unroll
    for (int r = 0; r < LA; ++r) {
      buf[line * C::DI + j * I::P1 + r] = w[u][0][perm<LA>(r)];
      if (!(line & 1)) buf[(TZ + line / 2) * C::DI + j * I::P1 + r] = w[u][1][perm<LA>(r)];
    }
  }
  __syncthreads();
  fft_mid<I, -1, NT, C::NTR>(buf, C::DI, C::NTR, twl);
  // last pass: the retained bins, m < M at m and -m at 2M - 1 - m
  double2* out = buf + C::OUT;
  constexpr int NC = C::NTR * I::JL;
#pragma unroll
  for (int q0 = 0; q0 < NC; q0 += NT) {
    const int q = threadIdx.x + q0, t = q % C::NTR, j = q / C::NTR;
    if (q >= NC) continue;
    double2 v[1][F];
    fft_last<I, -1>(v, buf + t * C::DI, 0, j, twl);
#pragma unroll
    for (int r = 0; r < F; ++r) {
      if (r * I::JL >= M && (r + 1) * I::JL - 1 <= TT - M) continue;
      const int i = j + r * I::JL;
      if (i < M) out[t * C::DO + i] = v[0][perm<F>(r)];
      else if (i > TT - M) out[t * C::DO + i - (M + 1)] = v[0][perm<F>(r)];
    }
  }
  // recorded only where they are read: an adaptive slot's predictor
  // evaluation (the device loop) and host-driven evaluations
  if ((B.prm[slot].adaptive && c->mode == MODE_PRED) || c->host_driven)
    plane_maxima<NT>(mr, mt, mz, B.cflmax + (size_t)slot * 3 * G.N + n, G.N);
  __syncthreads();
  constexpr int ND = TZ * 3 * M;
#pragma unroll
  for (int q0 = 0; q0 < ND; q0 += NT) {
    const int q = threadIdx.x + q0, line = q % TZ, rest = q / TZ, m = rest % M, f = rest / M;
    if (q >= ND || line >= tz) continue;
    const double2* o = out + (f == 2 ? TZ + line / 2 : line) * C::DO;
    Yb[yoff(z0 + line, 3, f, M, m)] =
        unpack_bin(o[m], o[m == 0 ? 0 : 2 * M - 1 - m], f == 0 || (f == 2 && (line & 1) == 0));
  }
}

// ---------------------------------------------------------------------------
// A radial plane's whole evaluation in one workgroup, for grids whose theta
// transforms (3 Z lines of T values) fit in LDS: the passes of k_zfwd_t,
// k_theta_t and k_zbwd_t in turn (the same operations, so the same bits), with
// the intermediates in LDS.  grid: x = N, z = slot.  Each pass reads all it
// needs into registers before a barrier and the next table is written over the
// last one.  One workgroup runs the plane's chain of latencies alone: one
// round of butterflies per pass (1024 threads) and ten barriers: 12.6 us for
// (K, M) = (24, 12) against 20.6 us with every pass, the packing and the
// products through LDS in chunks of lines; the three kernels take 14.5 us.
// ---------------------------------------------------------------------------
template <int ZF, int ZL, int TF, int TL>
struct PlaneTile {
  using ZS = Seq<ZF, 1, ZL>;
  using S = Seq<TF, 1, TL>;
  using I = Seq<TL, 1, TF>;
  static constexpr int Z = ZS::L, TT = S::L, K = Z / 3, M = TT / 3, NT = PLANE_THREADS;
  static_assert(Z % 2 == 0, "N_z pairs lines 2q and 2q + 1");
  static constexpr int DZ = ZS::SIZE | 1, DY = Z | 1;       // a column's exchange table, and its values
  static constexpr int DS = S::SIZE | 1, DI = I::SIZE | 1, DO = (2 * M - 1) | 1;
  static constexpr int NTR = Z + Z / 2, OUT = NTR * DI;
  static constexpr int mx(int a, int b) { return a > b ? a : b; }
  // the retained bins stand behind both the tables of the transforms back that
  // they are read from and the z columns that they are read into
  static constexpr int BINS = mx(OUT, 3 * M * DZ);
  static constexpr int BUF = mx(mx(6 * M * mx(DZ, DY), 3 * Z * DS), BINS + NTR * DO);
  static constexpr size_t smem = (size_t)(BUF + Z + TT) * sizeof(double2);
  static_assert(BINS >= NTR * DI && BINS >= 3 * M * DZ && BUF >= 3 * Z * DS && BUF >= 6 * M * DY && 2 * M - 1 <= DO,
                "the tables of a stage");
  static_assert(smem <= 160 * 1024, "the LDS of a CU");
};
template <int ZF, int ZL, int TF, int TL>
__global__ void __launch_bounds__(PLANE_THREADS) k_plane_t(Geo G, Bufs B, FftTiles, int slot0) {
  using C = PlaneTile<ZF, ZL, TF, TL>;
  using ZS = typename C::ZS;
  using S = typename C::S;
  using I = typename C::I;
  constexpr int NT = C::NT, Z = C::Z, TT = C::TT, M = C::M;
  const int slot = slot_of(B, slot0);
  const SlotCtl* c = &B.ctl[slot];
  if (!c->active) return;
  const int n = blockIdx.x;
  const int tid = threadIdx.x;
  double2* buf = smem;
  double2* twz = smem + C::BUF;
  double2* twt = twz + Z;
  // z transforms of the six fields
  constexpr int N1 = 6 * M * ZS::JF, R1 = (N1 + NT - 1) / NT;
  {
    double2 v[R1][ZF];
#pragma unroll
    for (int u = 0; u < R1; ++u) {
      const int q = tid + u * NT, col = q / ZS::JF, j = q - col * ZS::JF, f = col / M, m = col - f * M;
      if (q >= N1) continue;
      const double2* row = (f < 3 ? B.U[c->ucur] : B.om) + ((size_t)slot * 3 + (f < 3 ? f : f - 3)) * G.coll + (size_t)n * G.Hp;
      zcol_input<ZS>(v[u], row, m, j);
    }
    load_tw<NT>(twz, B.twZ, Z);
    load_tw<NT>(twt, B.twT, TT);
#pragma unroll
    for (int u = 0; u < R1; ++u) {
      const int q = tid + u * NT, col = q / ZS::JF, j = q - col * ZS::JF;
      if (q < N1) fft_first<ZS, 1>(v[u], buf + col * C::DZ, j);
    }
  }
  __syncthreads();
  constexpr int N2 = 6 * M * ZS::JL, R2 = (N2 + NT - 1) / NT;
  {
    double2 v[R2][1][ZL];
#pragma unroll
    for (int u = 0; u < R2; ++u) {
      const int q = tid + u * NT, col = q / ZS::JL, j = q - col * ZS::JL;
      if (q < N2) fft_last<ZS, 1>(v[u], buf + col * C::DZ, 0, j, twz);
    }
    __syncthreads();
#pragma unroll
    for (int u = 0; u < R2; ++u) {
      const int q = tid + u * NT, col = q / ZS::JL, j = q - col * ZS::JL;
      if (q >= N2) continue;
#pragma unroll
      for (int r = 0; r < ZL; ++r) buf[col * C::DY + j + r * ZS::JL] = v[u][0][perm<ZL>(r)];
    }
  }
  __syncthreads();
  // theta transforms, all lines at once, lines on neighbouring lanes
  constexpr int N3 = 3 * Z * S::JF, R3 = (N3 + NT - 1) / NT;
  {
    double2 v[R3][TF];
#pragma unroll
    for (int u = 0; u < R3; ++u) {
      const int q = tid + u * NT, line = q % Z, rest = q / Z, j = rest % S::JF, p = rest / S::JF;
      if (q >= N3) continue;
      const double2* src = buf + 2 * p * M * C::DY + line;
#pragma unroll
      for (int r = 0; r < TF; ++r) {
        v[u][r] = make_double2(0.0, 0.0);
        if (r * S::JF >= M && (r + 1) * S::JF - 1 <= TT - M) continue;
        const int i = j + r * S::JF, m = i < M ? i : TT - i;
        if (i < M || i > TT - M) v[u][r] = pack_bin(src[m * C::DY], src[(M + m) * C::DY], i, m);
      }
    }
    __syncthreads();
#pragma unroll
    for (int u = 0; u < R3; ++u) {
      const int q = tid + u * NT, line = q % Z, rest = q / Z, j = rest % S::JF, p = rest / S::JF;
      if (q < N3) fft_first<S, 1>(v[u], buf + (p * Z + line) * C::DS, j);
    }
  }
  __syncthreads();
  const NlPlane pl = NlPlane::make(G, B, slot, n, TT);
  double mr = 0.0, mt = 0.0, mz = 0.0;
  constexpr int N4 = Z * S::JL, R4 = (N4 + NT - 1) / NT;
  {
    double2 w[R4][3][TL];
#pragma unroll
    for (int u = 0; u < R4; ++u) {
      const int q = tid + u * NT, line = q % Z, j = q / Z;
      if (q >= N4) continue;
      fft_last<S, 1, 3>(w[u], buf + line * C::DS, Z * C::DS, j, twt);
      theta_middle<S>(w[u], pl, twt, j, true, true, mr, mt, mz);
    }
    __syncthreads();
#pragma unroll
    for (int u = 0; u < R4; ++u) {
      const int q = tid + u * NT, line = q % Z, j = q / Z;
      if (q >= N4) continue;
#pragma unroll
      for (int r = 0; r < TL; ++r) {
        buf[line * C::DI + j * I::P1 + r] = w[u][0][perm<TL>(r)];
        if (!(line & 1)) buf[(Z + line / 2) * C::DI + j * I::P1 + r] = w[u][1][perm<TL>(r)];
      }
    }
  }
  // the plane's velocity maxima where they are read (zero otherwise, as the
  // z kernel leaves them)
  unsigned long long* mx = B.cflmax + (size_t)slot * 3 * G.N + n;
  if ((B.prm[slot].adaptive && c->mode == MODE_PRED) || c->host_driven) plane_maxima<NT, true>(mr, mt, mz, mx, G.N);
  else if (tid < 3) mx[(size_t)tid * G.N] = 0ull;
  __syncthreads();
  double2* out = buf + C::BINS;
  constexpr int N5 = C::NTR * I::JL;
#pragma unroll
  for (int q0 = 0; q0 < N5; q0 += NT) {
    const int q = tid + q0, t = q % C::NTR, j = q / C::NTR;
    if (q >= N5) continue;
    double2 v[1][TF];
    fft_last<I, -1>(v, buf + t * C::DI, 0, j, twt);
#pragma unroll
    for (int r = 0; r < TF; ++r) {
      if (r * I::JL >= M && (r + 1) * I::JL - 1 <= TT - M) continue;
      const int i = j + r * I::JL;
      if (i < M) out[t * C::DO + i] = v[0][perm<TF>(r)];
      else if (i > TT - M) out[t * C::DO + i - (M + 1)] = v[0][perm<TF>(r)];
    }
  }
  __syncthreads();
  // z transforms of the nonlinear terms, unpacked as they are read
  constexpr int N6 = 3 * M * ZS::JF;
#pragma unroll
  for (int q0 = 0; q0 < N6; q0 += NT) {
    const int q = tid + q0, col = q / ZS::JF, j = q - col * ZS::JF, f = col / M, m = col - f * M;
    if (q >= N6) continue;
    double2 v[ZF];
#pragma unroll
    for (int r = 0; r < ZF; ++r) {
      const int line = j + r * ZS::JF;
      const double2* o = out + (f == 2 ? Z + line / 2 : line) * C::DO;
      v[r] = unpack_bin(o[m], o[m == 0 ? 0 : 2 * M - 1 - m], f == 0 || (f == 2 && (line & 1) == 0));
    }
    fft_first<ZS, -1>(v, buf + col * C::DZ, j);
  }
  __syncthreads();
  constexpr int N7 = 3 * M * ZS::JL;
#pragma unroll
  for (int q0 = 0; q0 < N7; q0 += NT) {
    const int q = tid + q0, col = q / ZS::JL, j = q - col * ZS::JL, f = col / M, m = col - f * M;
    if (q >= N7) continue;
    double2 v[1][ZL];
    fft_last<ZS, -1>(v, buf + col * C::DZ, 0, j, twz);
    zcol_output<ZS>(B.Nraw[c->ncur] + ((size_t)slot * 3 + f) * G.coll + (size_t)n * G.Hp, v[0], m, j);
  }
}

// ---------------------------------------------------------------------------
// The three stages for any other length, with run-time plans: whole tiles in
// LDS (linear input, padded output), every pass through it.
// ---------------------------------------------------------------------------
__global__ void ANY_LENGTH k_zfwd_any(Geo G, Bufs B, FftTiles T, int slot0) {
  const int slot = slot_of(B, slot0);
  const SlotCtl* c = &B.ctl[slot];
  if (!c->active) return;
  if (blockIdx.x == 0)
    for (int i = threadIdx.x; i < 3 * G.N; i += FFT_THREADS) B.cflmax[(size_t)slot * 3 * G.N + i] = 0ull;
  ZWhere w;
  if (!ztile(G, T.tm, 6, w)) return;
  const int Z = G.Z, K = G.K, M = G.M, f = w.f, tm = w.tm;
  const double2* src = (f < 3 ? B.U[c->ucur] : B.om) + ((size_t)slot * 3 + (f < 3 ? f : f - 3)) * G.coll + (size_t)w.n * G.Hp;
  const int Zp = padded_len(Z);
  double2* buf = smem;
  double2* twl = smem + (size_t)T.tm * Zp;
  load_tw(twl, B.twZ, Z);
  load_zcols(buf, src, K, Z, Zp, w.m0, tm);
  __syncthreads();
  fft_lds<1>(buf, tm, T.pz, twl);
  double2* Y = B.Yf + ((size_t)slot * G.N + w.n) * G.ZQ * 6 * M;
  for (int i = threadIdx.x; i < tm * Z; i += FFT_THREADS) {
    const int z = i / tm, b = i - z * tm;
    Y[yoff(z, 6, f, M, w.m0 + b)] = buf[b * Zp + pidx(z)];
  }
}

constexpr int TLD = THETA_ITEMS / FFT_THREADS;
__global__ void ANY_LENGTH k_theta_any(Geo G, Bufs B, FftTiles T, int slot0) {
  const int slot = slot_of(B, slot0);
  const SlotCtl* c = &B.ctl[slot];
  if (!c->active) return;
  const int gz = (G.Z + T.tz - 1) / T.tz, per = (gz * G.N + 7) / 8;
  const int tile = (int)(blockIdx.x % 8) * per + (int)(blockIdx.x / 8);
  if (tile >= gz * G.N) return;
  const int n = tile / gz;
  const int z0 = (tile - n * gz) * T.tz;
  const int tz = min(T.tz, G.Z - z0);
  const int TT = G.T, M = G.M;   // T = 3M
  const double2* Yf = B.Yf + ((size_t)slot * G.N + n) * G.ZQ * 6 * M;
  const int Tp = padded_len(TT);
  // transform (pair*tz + line) of the three packed pairs at stride Tp, so the
  // two forward transforms of every line are the first 2*tz transforms
  double2* buf = smem;
  double2* twl = smem + (size_t)3 * T.tz * Tp;
  load_tw(twl, B.twT, TT);
  const int total = tz * 3 * M;   // = tz * T <= THETA_ITEMS = TLD * FFT_THREADS
  double2 A[TLD], Bv[TLD];
  int it[TLD];
#pragma unroll
  for (int u = 0; u < TLD; ++u) {
    const int i = threadIdx.x + u * FFT_THREADS;
    const bool ok = i < total;
    const int ic = ok ? i : 0;
    const int line = ic / (3 * M), rem = ic - line * 3 * M;
    const int pr = rem / M, mm = rem - pr * M;
    const double2* src = Yf + yoff(z0 + line, 6, 2 * pr, M, mm);
    A[u] = src[0];
    Bv[u] = src[4 * M];
    it[u] = ok ? i : -1;
  }
#pragma unroll
  for (int u = 0; u < TLD; ++u) {
    if (it[u] < 0) continue;
    const int i = it[u];
    const int line = i / (3 * M), rem = i - line * 3 * M;
    const int pr = rem / M, mm = rem - pr * M;
    double2* L = buf + ((size_t)pr * tz + line) * Tp;
    L[mm] = pack_bin(A[u], Bv[u], mm, mm);
    if (mm > 0) L[TT - mm] = pack_bin(A[u], Bv[u], TT - mm, mm);
  }
  const int nzero = TT - 2 * M + 1;   // bins M .. T-M
  for (int i = threadIdx.x; i < 3 * tz * nzero; i += FFT_THREADS) {
    const int pl = i / nzero, mm = M + (i - pl * nzero);
    const int pr = pl / tz, line = pl - pr * tz;
    buf[((size_t)pr * tz + line) * Tp + mm] = make_double2(0.0, 0.0);
  }
  __syncthreads();
  fft_lds<1>(buf, 3 * tz, T.pt, twl);
  // products and the plane's velocity maxima
  const NlPlane pl = NlPlane::make(G, B, slot, n, TT);
  double mr = 0.0, mt = 0.0, mz = 0.0;
  // N of this thread's items, written after a barrier as the transforms
  // back's linear input (it overlaps the other transforms' output)
  double2 nrt[TLD];
  double nzv[TLD];
#pragma unroll
  for (int u = 0; u < TLD; ++u) {
    const int i = threadIdx.x + u * FFT_THREADS;
    if (i >= tz * TT) continue;
    const int line = i / TT, th = i - line * TT;
    const double2* L0 = buf + (size_t)line * Tp + pidx(th);
    pl.point(L0[0], L0[(size_t)tz * Tp], L0[(size_t)2 * tz * Tp], twl, th, mr, mt, mz, nrt[u], nzv[u]);
  }
  if ((B.prm[slot].adaptive && c->mode == MODE_PRED) || c->host_driven)
    plane_maxima<FFT_THREADS>(mr, mt, mz, B.cflmax + (size_t)slot * 3 * G.N + n, G.N);
  __syncthreads();
  const int nzt = (tz + 1) / 2;
#pragma unroll
  for (int u = 0; u < TLD; ++u) {
    const int i = threadIdx.x + u * FFT_THREADS;
    if (i >= tz * TT) continue;
    const int line = i / TT, th = i - line * TT;
    buf[(size_t)line * Tp + th] = nrt[u];
    double* d = (double*)(buf + ((size_t)tz + (line >> 1)) * Tp + th);
    d[line & 1] = nzv[u];
    if ((line & 1) == 0 && line + 1 == tz) d[1] = 0.0;
  }
  __syncthreads();
  fft_lds<-1>(buf, tz + nzt, T.pt, twl);
  double2* Yb = B.Yb + ((size_t)slot * G.N + n) * G.ZQ * 3 * M;
  for (int i = threadIdx.x; i < tz * 3 * M; i += FFT_THREADS) {
    const int line = i / (3 * M), rem = i - line * 3 * M;
    const int f = rem / M, mm = rem - f * M;
    const double2* L = buf + (f == 2 ? (size_t)tz + (line >> 1) : (size_t)line) * Tp;
    Yb[yoff(z0 + line, 3, f, M, mm)] =
        unpack_bin(L[pidx(mm)], L[pidx((TT - mm) % TT)], f == 0 || (f == 2 && (line & 1) == 0));
  }
}

__global__ void ANY_LENGTH k_zbwd_any(Geo G, Bufs B, FftTiles T, int slot0) {
  const int slot = slot_of(B, slot0);
  const SlotCtl* c = &B.ctl[slot];
  if (!c->active) return;
  ZWhere w;
  if (!ztile(G, T.tm, 3, w)) return;
  const int Z = G.Z, K = G.K, M = G.M, f = w.f, tm = w.tm;
  const double2* Y = B.Yb + ((size_t)slot * G.N + w.n) * G.ZQ * 3 * M;
  const int Zp = padded_len(Z);
  double2* buf = smem;
  double2* twl = smem + (size_t)T.tm * Zp;
  load_tw(twl, B.twZ, Z);
  load_ycols(buf, Y, [=](int z, int m) { return yoff(z, 3, f, M, m); }, Z, Zp, w.m0, tm);
  __syncthreads();
  fft_lds<-1>(buf, tm, T.pz, twl);
  double2* row = B.Nraw[c->ncur] + ((size_t)slot * 3 + f) * G.coll + (size_t)w.n * G.Hp;
  for (int b = 0; b < tm; ++b) store_zcol(row, buf + b * Zp, K, Z, w.m0 + b, threadIdx.x, FFT_THREADS);
}

// ---------------------------------------------------------------------------
// Granular transforms of one coll field (tra_coll2phys / tra_phys2coll of the
// drop-in interface): spec -> Y -> phys[n][z][th] and back, Y the intermediates
// of one field per plane (yoff with one field).
// ---------------------------------------------------------------------------
__global__ void ANY_LENGTH k_zfwd_one(Geo G, Bufs B, FftTiles T, const double2* a, double2* Y,
                                                          size_t fa, size_t fy) {
  a += blockIdx.z * fa;   // field blockIdx.z of a batch at strides fa, fy
  Y += blockIdx.z * fy;
  ZWhere w;
  if (!ztile(G, T.tm, 1, w)) return;
  const int n = w.n, m0 = w.m0, tm = w.tm;
  const int Z = G.Z, K = G.K, M = G.M;
  const double2* src = a + (size_t)n * G.Hp;
  const int Zp = padded_len(Z);
  double2* buf = smem;
  double2* twl = smem + (size_t)T.tm * Zp;
  load_tw(twl, B.twZ, Z);
  load_zcols(buf, src, K, Z, Zp, m0, tm);
  __syncthreads();
  fft_lds<1>(buf, tm, T.pz, twl);
  for (int i = threadIdx.x; i < tm * Z; i += FFT_THREADS) {
    const int z = i / tm, b = i - z * tm;
    Y[(size_t)n * G.ZQ * M + yoff(z, 1, 0, M, m0 + b)] = buf[b * Zp + pidx(z)];
  }
}

// c2r along theta of one field, lines paired as a + ib.  grid: x = z pairs, y = N.
// LDS: one padded line, then T twiddles.
__global__ void ANY_LENGTH k_theta_c2r(Geo G, Bufs B, FftTiles T, const double2* Y, double* phys) {
  const int n = blockIdx.y;
  const int z0 = blockIdx.x * 2;
  const int M = G.M, TT = G.T;
  const bool two = z0 + 1 < G.Z;
  double2* buf = smem;
  double2* twl = smem + padded_len(TT);
  load_tw(twl, B.twT, TT);
  // z0 and z0 + 1 stand side by side (z0 is even)
  const double2* A = Y + (size_t)n * G.ZQ * M + yoff(z0, 1, 0, M, 0);
  const double2* Bp = A + 1;
  for (int mm = threadIdx.x; mm < TT; mm += FFT_THREADS) {
    double2 v = make_double2(0.0, 0.0);
    if (mm == 0) v = make_double2(A[0].x, two ? Bp[0].x : 0.0);
    else if (mm < M) {
      const double2 a = A[4 * mm], b = two ? Bp[4 * mm] : make_double2(0.0, 0.0);
      v = make_double2(a.x - b.y, a.y + b.x);
    } else if (mm > TT - M) {
      const int q = TT - mm;
      const double2 a = A[4 * q], b = two ? Bp[4 * q] : make_double2(0.0, 0.0);
      v = make_double2(a.x + b.y, -a.y + b.x);
    }
    buf[mm] = v;
  }
  __syncthreads();
  fft_lds<1>(buf, 1, T.pt, twl);
  // phys layout of the reference: Re(0:3K-1, 0:3M-1, N), z fastest
  double* out = phys + (size_t)n * TT * G.Z + z0;
  for (int th = threadIdx.x; th < TT; th += FFT_THREADS) {
    out[(size_t)th * G.Z] = buf[pidx(th)].x;
    if (two) out[(size_t)th * G.Z + 1] = buf[pidx(th)].y;
  }
}

// r2c along theta (scaled by 1/(3K 3M) first, transform.fftw3.f90:114-117).
// The theta transforms of the variable-viscosity plugins: the z-lines of one
// radial plane packed two per complex transform (as k_theta_c2r does), BT
// transforms per workgroup, on physical fields in the plugins' own layout
// [n][z][theta] (theta fastest, so every line is one contiguous run).
// grid: x = blocks of 2 BT z-lines, y = N.
__global__ void ANY_LENGTH k_c2r_lines(Geo G, Bufs B, FftTiles T, int BT, const double2* Y,
                                                           double* phys, size_t fy, size_t fp) {
  Y += blockIdx.z * fy;   // field blockIdx.z of a batch at strides fy, fp
  phys += blockIdx.z * fp;
  const int n = blockIdx.y;
  const int M = G.M, TT = G.T, Z = G.Z;
  const int Tp = padded_len(TT);
  const int z0 = blockIdx.x * 2 * BT;
  const int nt = min(BT, (Z - z0 + 1) / 2);
  double2* buf = smem;
  double2* twl = smem + (size_t)BT * Tp;
  load_tw(twl, B.twT, TT);
  for (int i = threadIdx.x; i < nt * TT; i += FFT_THREADS) {
    const int b = i / TT, mm = i - b * TT;
    const int z = z0 + 2 * b;
    const bool two = z + 1 < Z;
    const double2* A = Y + (size_t)n * G.ZQ * M + yoff(z, 1, 0, M, 0);
    const double2* Bp = A + 1;
    double2 v = make_double2(0.0, 0.0);
    if (mm == 0) v = make_double2(A[0].x, two ? Bp[0].x : 0.0);
    else if (mm < M) {
      const double2 a = A[4 * mm], c = two ? Bp[4 * mm] : make_double2(0.0, 0.0);
      v = make_double2(a.x - c.y, a.y + c.x);
    } else if (mm > TT - M) {
      const int q = TT - mm;
      const double2 a = A[4 * q], c = two ? Bp[4 * q] : make_double2(0.0, 0.0);
      v = make_double2(a.x + c.y, -a.y + c.x);
    }
    buf[(size_t)b * Tp + mm] = v;
  }
  __syncthreads();
  fft_lds<1>(buf, nt, T.pt, twl);
  for (int i = threadIdx.x; i < nt * TT; i += FFT_THREADS) {
    const int b = i / TT, th = i - b * TT;
    const int z = z0 + 2 * b;
    const double2 v = buf[(size_t)b * Tp + pidx(th)];
    double* out = phys + ((size_t)n * Z + z) * TT + th;
    out[0] = v.x;
    if (z + 1 < Z) out[TT] = v.y;
  }
}

// The inverse of k_c2r_lines with the scaling of tra_phys2spec (1/(3K 3M),
// transform.fftw3.f90:114), into the z-transform intermediates Y.
__global__ void ANY_LENGTH k_r2c_lines(Geo G, Bufs B, FftTiles T, int BT, const double* phys,
                                                           double2* Y, size_t fp, size_t fy) {
  phys += blockIdx.z * fp;   // field blockIdx.z of a batch at strides fp, fy
  Y += blockIdx.z * fy;
  const int n = blockIdx.y;
  const int M = G.M, TT = G.T, Z = G.Z;
  const int Tp = padded_len(TT);
  const int z0 = blockIdx.x * 2 * BT;
  const int nt = min(BT, (Z - z0 + 1) / 2);
  const double scale = 1.0 / (double)(Z * TT);
  double2* buf = smem;
  double2* twl = smem + (size_t)BT * Tp;
  load_tw(twl, B.twT, TT);
  for (int i = threadIdx.x; i < nt * TT; i += FFT_THREADS) {
    const int b = i / TT, th = i - b * TT;
    const int z = z0 + 2 * b;
    const double* in = phys + ((size_t)n * Z + z) * TT + th;
    buf[(size_t)b * Tp + th] = make_double2(scale * in[0], z + 1 < Z ? scale * in[TT] : 0.0);
  }
  __syncthreads();
  fft_lds<-1>(buf, nt, T.pt, twl);
  for (int i = threadIdx.x; i < nt * M; i += FFT_THREADS) {
    const int b = i / M, mm = i - b * M;
    const int z = z0 + 2 * b;
    const double2* L = buf + (size_t)b * Tp;
    const double2 X = L[pidx(mm)], Xc = L[pidx((TT - mm) % TT)];
    double2* A = Y + (size_t)n * G.ZQ * M + yoff(z, 1, 0, M, mm);
    A[0] = unpack_bin(X, Xc, true);
    if (z + 1 < Z) A[1] = unpack_bin(X, Xc, false);
  }
}

__global__ void ANY_LENGTH k_theta_r2c(Geo G, Bufs B, FftTiles T, const double* phys, double2* Y) {
  const int n = blockIdx.y;
  const int z0 = blockIdx.x * 2;
  const int M = G.M, TT = G.T;
  const bool two = z0 + 1 < G.Z;
  const double scale = 1.0 / (double)(G.Z * TT);
  double2* buf = smem;
  double2* twl = smem + padded_len(TT);
  load_tw(twl, B.twT, TT);
  const double* in = phys + (size_t)n * TT * G.Z + z0;
  for (int th = threadIdx.x; th < TT; th += FFT_THREADS)
    buf[th] = make_double2(scale * in[(size_t)th * G.Z], two ? scale * in[(size_t)th * G.Z + 1] : 0.0);
  __syncthreads();
  fft_lds<-1>(buf, 1, T.pt, twl);
  double2* A = Y + (size_t)n * G.ZQ * M + yoff(z0, 1, 0, M, 0);
  for (int mm = threadIdx.x; mm < M; mm += FFT_THREADS) {
    const double2 X = buf[pidx(mm)], Xc = buf[pidx((TT - mm) % TT)];
    A[4 * mm] = unpack_bin(X, Xc, true);
    if (two) A[4 * mm + 1] = unpack_bin(X, Xc, false);
  }
}

__global__ void ANY_LENGTH k_zbwd_one(Geo G, Bufs B, FftTiles T, const double2* Y, double2* a,
                                                          size_t fy, size_t fa) {
  Y += blockIdx.z * fy;   // field blockIdx.z of a batch at strides fy, fa
  a += blockIdx.z * fa;
  ZWhere w;
  if (!ztile(G, T.tm, 1, w)) return;
  const int n = w.n, m0 = w.m0, tm = w.tm;
  const int Z = G.Z, K = G.K, M = G.M;
  const int Zp = padded_len(Z);
  double2* buf = smem;
  double2* twl = smem + (size_t)T.tm * Zp;
  load_tw(twl, B.twZ, Z);
  load_ycols(buf, Y + (size_t)n * G.ZQ * M, [=](int z, int m) { return yoff(z, 1, 0, M, m); }, Z, Zp, m0, tm);
  __syncthreads();
  fft_lds<-1>(buf, tm, T.pz, twl);
  double2* row = a + (size_t)n * G.Hp;
  for (int b = 0; b < tm; ++b) store_zcol(row, buf + b * Zp, K, Z, m0 + b, threadIdx.x, FFT_THREADS);
}

// The plugins' transforms at the lengths with fixed radix sequences: the z
// tiles of k_zfwd_t and k_zbwd_t on any coll field (grid z: field of a batch at
// strides fa, fy), and the theta lines two per complex transform.
template <int F, int MID, int LA>
__global__ void __launch_bounds__((ZTile<F, MID, LA>::NT)) k_zfwd_one_t(Geo G, Bufs B, FftTiles T, const double2* a,
                                                                       double2* Y, size_t fa, size_t fy) {
  ZWhere w;
  if (!ztile(G, T.tm, 1, w)) return;
  const int M = G.M;
  zfwd_tile<F, MID, LA>(a + blockIdx.z * fa + (size_t)w.n * G.Hp, Y + blockIdx.z * fy + (size_t)w.n * G.ZQ * M,
                        [=](int z, int m) { return yoff(z, 1, 0, M, m); }, w.m0, w.tm, B.twZ);
}
template <int F, int MID, int LA>
__global__ void __launch_bounds__((ZTile<F, MID, LA>::NT)) k_zbwd_one_t(Geo G, Bufs B, FftTiles T, const double2* Y,
                                                                       double2* a, size_t fy, size_t fa) {
  ZWhere w;
  if (!ztile(G, T.tm, 1, w)) return;
  const int M = G.M;
  zbwd_tile<F, MID, LA>(Y + blockIdx.z * fy + (size_t)w.n * G.ZQ * M, [=](int z, int m) { return yoff(z, 1, 0, M, m); },
                        a + blockIdx.z * fa + (size_t)w.n * G.Hp, w.m0, w.tm, B.twZ);
}
// BT = ZTile::TM transforms of two lines each.  grid: x = line blocks, y = N, z = field.
template <int F, int MID, int LA>
__global__ void __launch_bounds__((ZTile<F, MID, LA>::NT)) k_c2r_lines_t(Geo G, Bufs B, FftTiles, int, const double2* Y,
                                                                        double* phys, size_t fy, size_t fp) {
  using C = ZTile<F, MID, LA>;
  using S = typename C::S;
  constexpr int TT = S::L, M = TT / 3, BT = C::TM, NT = C::NT;
  const int n = blockIdx.y, Z = G.Z, z0 = blockIdx.x * 2 * BT;
  Y += blockIdx.z * fy + (size_t)n * G.ZQ * M;
  phys += blockIdx.z * fp + (size_t)n * Z * TT;
  double2* buf = smem;
  // two pairs of lines (a block of four z) on neighbouring lanes
  constexpr int NA = (BT + 1) / 2 * 2 * S::JF;
#pragma unroll
  for (int q0 = 0; q0 < NA; q0 += NT) {
    const int q = threadIdx.x + q0, j = (q >> 1) % S::JF, t = (q >> 1) / S::JF * 2 + (q & 1), z = z0 + 2 * t;
    const bool live = t < BT && z < Z, two = z + 1 < Z;
    const double2* src = Y + (live ? yoff(z, 1, 0, M, 0) : 0);
    double2 v[F], bv[F];
#pragma unroll
    for (int r = 0; r < F; ++r) {
      v[r] = bv[r] = make_double2(0.0, 0.0);
      if (r * S::JF >= M && (r + 1) * S::JF - 1 <= TT - M) continue;
      const int i = j + r * S::JF, m = i < M ? i : i > TT - M ? TT - i : 0;
      v[r] = src[4 * m];
      bv[r] = src[4 * m + 1];   // in the block of four also where Z ends before it
    }
#pragma unroll
    for (int r = 0; r < F; ++r) {
      if (r * S::JF >= M && (r + 1) * S::JF - 1 <= TT - M) continue;
      const int i = j + r * S::JF, m = i < M ? i : TT - i;
      if (!two) bv[r] = make_double2(0.0, 0.0);
      v[r] = i < M || i > TT - M ? pack_bin(v[r], bv[r], i, m) : make_double2(0.0, 0.0);
    }
    if (live) fft_first<S, 1>(v, buf + t * C::D, j);
  }
  __syncthreads();
  fft_mid<S, 1, NT, BT>(buf, C::D, BT, B.twT);
#pragma unroll
  for (int q0 = 0; q0 < BT * S::JL; q0 += NT) {
    const int q = threadIdx.x + q0, t = q / S::JL, j = q - t * S::JL, z = z0 + 2 * t;
    if (t >= BT || z >= Z) continue;
    double2 v[1][LA];
    fft_last<S, 1>(v, buf + t * C::D, 0, j, B.twT);
    double* out = phys + (size_t)z * TT + j;
#pragma unroll
    for (int r = 0; r < LA; ++r) {
      out[r * S::JL] = v[0][perm<LA>(r)].x;
      if (z + 1 < Z) out[TT + r * S::JL] = v[0][perm<LA>(r)].y;
    }
  }
}
template <int F, int MID, int LA>
__global__ void __launch_bounds__((ZTile<F, MID, LA>::NT)) k_r2c_lines_t(Geo G, Bufs B, FftTiles, int, const double* phys,
                                                                        double2* Y, size_t fp, size_t fy) {
  using C = ZTile<F, MID, LA>;
  using S = typename C::S;
  constexpr int TT = S::L, M = TT / 3, BT = C::TM, NT = C::NT, DO = (2 * M - 1) | 1;
  const int n = blockIdx.y, Z = G.Z, z0 = blockIdx.x * 2 * BT;
  const double scale = 1.0 / (double)(Z * TT);
  phys += blockIdx.z * fp + (size_t)n * Z * TT;
  Y += blockIdx.z * fy + (size_t)n * G.ZQ * M;
  double2* buf = smem;
  double2* out = smem + BT * C::D;
#pragma unroll
  for (int q0 = 0; q0 < BT * S::JF; q0 += NT) {
    const int q = threadIdx.x + q0, t = q / S::JF, j = q - t * S::JF, z = z0 + 2 * t;
    if (t >= BT || z >= Z) continue;
    const double* in = phys + (size_t)z * TT + j;
    const int second = z + 1 < Z ? TT : 0;
    double2 v[F];
#pragma unroll
    for (int r = 0; r < F; ++r) v[r] = make_double2(in[r * S::JF], in[second + r * S::JF]);
#pragma unroll
    for (int r = 0; r < F; ++r) v[r] = make_double2(scale * v[r].x, second ? scale * v[r].y : 0.0);
    fft_first<S, -1>(v, buf + t * C::D, j);
  }
  __syncthreads();
  fft_mid<S, -1, NT, BT>(buf, C::D, BT, B.twT);
#pragma unroll
  for (int q0 = 0; q0 < BT * S::JL; q0 += NT) {
    const int q = threadIdx.x + q0, t = q / S::JL, j = q - t * S::JL;
    if (t >= BT) continue;
    double2 v[1][LA];
    fft_last<S, -1>(v, buf + t * C::D, 0, j, B.twT);
#pragma unroll
    for (int r = 0; r < LA; ++r) {
      if (r * S::JL >= M && (r + 1) * S::JL - 1 <= TT - M) continue;
      const int i = j + r * S::JL;
      if (i < M) out[t * DO + i] = v[0][perm<LA>(r)];
      else if (i > TT - M) out[t * DO + i - (M + 1)] = v[0][perm<LA>(r)];
    }
  }
  __syncthreads();
  constexpr int ND = (2 * BT + 3) / 4 * 4 * M;
#pragma unroll
  for (int q0 = 0; q0 < ND; q0 += NT) {
    const int q = threadIdx.x + q0, m = (q >> 2) % M, line = (q >> 2) / M * 4 + (q & 3), z = z0 + line;
    if (line >= 2 * BT || z >= Z) continue;
    const double2* o = out + (line >> 1) * DO;
    Y[yoff(z, 1, 0, M, m)] = unpack_bin(o[m], o[m == 0 ? 0 : 2 * M - 1 - m], (line & 1) == 0);
  }
}

// Every length 3K, 3M = 2^a 3^b from 9 to 768 has kernels of its own; longer
// ones use the run-time plans (z forward and backward of (64, 32, 24), Z = 96:
// 20.5 and 14.4 us with those, 8.0 and 5.2 us with 12 x 8).
//
// Sequences: two passes where both radices can be 16 or less, three beyond.  A
// first radix divisible by 3 reads exactly the retained third at either end,
// and a last one of 4 to 9 leaves few values per thread and long runs to
// store: z forward and backward at Z = 768 take 406 and 191 us with 16 x 16 x
// 3, 420 and 169 with 16 x 12 x 4, 274 and 152 with 12 x 8 x 8.  The theta
// kernel holds three last-pass butterflies at once, so it takes a third pass
// rather than a last radix of 9 (144: 16 x 9 33 us, 12 x 4 x 3 28.9; 108: 12 x
// 9 25.6, 9 x 4 x 3 23.4; 81: 9 x 9 15.0, 9 x 3 x 3 11.8), but not instead of
// one of 6 (72: 12 x 6 11.9, 6 x 4 x 3 13.0; 54: 9 x 6 8.2, 6 x 3 x 3 8.5), and
// at 384 12 x 8 x 4 (432 us) is ahead of 16 x 12 x 2 (488) and 8 x 8 x 6 (484).
//
// Before, each pass read and wrote LDS, the input and the products with it; z
// forward, theta, z backward took (us per launch, then and now) 11.5, 14.8, 9.3
// and 8.9, 11.9, 5.6 at (N, K, M) = (48, 48, 24); 24.1, 32.4, 13.3 and 18.1,
// 28.9, 10.8 at (64, 64, 48); 461, 597, 217 and 274, 432, 152 (4.4, 3.2 and
// 5.0 TB/s of the bytes they must move) at (96, 256, 128).
namespace {
struct LenKerns {
  int L;
  FftKern zfwd, zbwd, theta;
  ZOneKern zfwd1;
  ZOneKern zbwd1;
  C2rKern c2r;
  R2cKern r2c;
  int zn, tm, tn, tz;
  int ln, bt;   // threads and transforms (two lines each) of the line kernels
  size_t zfs, zbs, ts, c2rs, r2cs;
};
// passes (first, middle or 1, last) of the z kernels and of the theta kernel (up
// to the longest theta line that contexts take)
template <int ZF, int ZM, int ZL, int TF = ZF, int TM = ZM, int TL = ZL>
LenKerns kerns_of() {
  static_assert(TF * TM * TL == ZF * ZM * ZL, "one length");
  using ZT = ZTile<ZF, ZM, ZL>;
  using TT = ThetaTile<TF, TM, TL>;
  using LT = ZTile<TF, TM, TL>;
  LenKerns k{};
  k.L = ZF * ZM * ZL;
  k.zfwd = k_zfwd_t<ZF, ZM, ZL>;
  k.zbwd = k_zbwd_t<ZF, ZM, ZL>;
  k.zfwd1 = k_zfwd_one_t<ZF, ZM, ZL>;
  k.zbwd1 = k_zbwd_one_t<ZF, ZM, ZL>;
  k.zn = ZT::NT;
  k.tm = ZT::TM;
  k.zfs = ZT::smem_f;
  k.zbs = ZT::smem_b;
  if constexpr (TF * TM * TL <= THETA_MAX) {
    k.theta = k_theta_t<TF, TM, TL>;
    k.c2r = k_c2r_lines_t<TF, TM, TL>;
    k.r2c = k_r2c_lines_t<TF, TM, TL>;
    k.tn = TT::NT;
    k.tz = TT::TZ;
    k.ln = LT::NT;
    k.bt = LT::TM;
    k.ts = TT::smem;
    k.c2rs = LT::smem_b;
    k.r2cs = LT::smem_b + (size_t)LT::TM * ((2 * (k.L / 3) - 1) | 1) * sizeof(double2);
  }
  return k;
}
}  // namespace

// Plan pairs (z, theta) with a whole-plane kernel: the grids whose theta
// transforms fit in LDS.
PlaneKern plane_kernel(int Z, int T, size_t* smem) {
  struct Entry {
    int Z, T;
    PlaneKern k;
    size_t smem;
  };
  static const Entry table[] = {
      {72, 36, k_plane_t<12, 6, 12, 3>, PlaneTile<12, 6, 12, 3>::smem},   // (K, M) = (24, 12)
  };
  for (const auto& e : table)
    if (Z == e.Z && T == e.T) {
      *smem = e.smem;
      return e.k;
    }
  *smem = 0;
  return nullptr;
}

FftKerns fft_kernels(const FftPlan& pz, const FftPlan& pt, const FftTiles& t, int M) {
  static const LenKerns table[] = {
      kerns_of<9, 1, 1>(),            kerns_of<12, 1, 1>(),             kerns_of<9, 1, 2>(),
      kerns_of<12, 1, 2>(),           kerns_of<9, 1, 3>(),              kerns_of<12, 1, 3>(),
      kerns_of<12, 1, 4>(),           kerns_of<9, 1, 6>(),              kerns_of<12, 1, 6>(),
      kerns_of<9, 1, 9, 9, 3, 3>(),   kerns_of<12, 1, 8, 16, 1, 6>(),   kerns_of<12, 1, 9, 9, 4, 3>(),
      kerns_of<16, 1, 9, 12, 4, 3>(), kerns_of<9, 3, 6, 9, 6, 3>(),     kerns_of<16, 1, 12, 12, 4, 4>(),
      kerns_of<12, 3, 6, 12, 6, 3>(), kerns_of<9, 3, 9, 9, 9, 3>(),     kerns_of<12, 4, 6, 12, 6, 4>(),
      kerns_of<12, 3, 9, 12, 9, 3>(), kerns_of<12, 4, 8, 12, 8, 4>(),   kerns_of<12, 6, 6, 12, 9, 4>(),
      kerns_of<9, 6, 9, 9, 9, 6>(),   kerns_of<12, 6, 8, 12, 12, 4>(),  kerns_of<12, 6, 9, 12, 9, 6>(),
      kerns_of<12, 8, 8>(),
  };
  auto find = [&](int L) -> const LenKerns* {
    for (const auto& e : table)
      if (e.L == L) return &e;
    return nullptr;
  };
  FftKerns k{};
  k.t = t;
  k.zfwd = k_zfwd_any;
  k.zbwd = k_zbwd_any;
  k.theta = k_theta_any;
  k.zfwd1 = k_zfwd_one;
  k.zbwd1 = k_zbwd_one;
  k.c2r = k_c2r_lines;
  k.r2c = k_r2c_lines;
  k.zn = k.tn = k.ln = FFT_THREADS;
  k.bt = std::max(1, FFT_TILE / padded_len(pt.L));
  k.c2rs = k.r2cs = ((size_t)k.bt * padded_len(pt.L) + pt.L) * sizeof(double2);
  k.zfs = k.zbs = ((size_t)t.tm * padded_len(pz.L) + pz.L) * sizeof(double2);
  k.ts = ((size_t)3 * t.tz * padded_len(pt.L) + pt.L) * sizeof(double2);
  if (const LenKerns* z = find(pz.L)) {
    k.zfwd = z->zfwd;
    k.zbwd = z->zbwd;
    k.zfwd1 = z->zfwd1;
    k.zbwd1 = z->zbwd1;
    k.zn = z->zn;
    k.zfs = z->zfs;
    k.zbs = z->zbs;
    // equal tiles: M columns over as many workgroups as the widest tile needs
    const int w = std::min(t.tm, z->tm), g = (M + w - 1) / w;
    k.t.tm = (M + g - 1) / g;
  }
  if (const LenKerns* z = find(pt.L); z && z->theta) {
    k.theta = z->theta;
    k.c2r = z->c2r;
    k.r2c = z->r2c;
    k.ln = z->ln;
    k.bt = z->bt;
    k.c2rs = z->c2rs;
    k.r2cs = z->r2cs;
    k.tn = z->tn;
    k.ts = z->ts;
    // one line is the run-time plans' tile beyond 384 points; these hold two
    // (432 points 37.4 to 24.4 us, 576 points 63.4 to 38.4, 648 points 39.4 to 25.9)
    k.t.tz = t.tz == 1 ? z->tz : std::min(t.tz, z->tz);
  }
  return k;
}

}  // namespace opf
