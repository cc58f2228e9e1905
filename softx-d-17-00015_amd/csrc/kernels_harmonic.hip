// The fused per-harmonic step kernel: vel_predictor / vel_corrector
// (velocity.f90:400-432) with vel_addHPF (:338-361), tim_nlincorr
// (timestep.f90:174-184), vel_step (velocity.f90:367-394), tim_measurecorr
// (timestep.f90:190-207) and the curl of the new velocity for the next
// nonlinear evaluation (var_coll_curl, variables.f90:408-436).
//
// One workgroup owns a group of GP consecutive (|k|, m) pairs, i.e. the
// harmonics +k and -k of each pair (2*GP "harmonic slots"): two waves for
// GP = 1, 2 and four for GP = 4.
// Everything a harmonic needs between its input and output stays in LDS:
//   V[3][N][2GP]  the right-hand sides (u+, u-, uz), with the pressure in the
//                 third field while that of uz waits in registers.
// All waves map threads to (radial point, harmonic) for the stages that are
// parallel in r (right-hand side, divergence, gradient, influence correction,
// curl).  The banded systems are solved by blocks of four rows on the matrix
// cores, wave w those of pair w (solve.hpp).
//
// What bounds the kernel is one workgroup's chain: the memory latencies in it,
// and the number of instructions, which arrive no faster than about a cache
// line per 90 ns in code that a wave runs through once.  So every global load
// is issued well before its use (the state and the mesh tables in one batch, a
// solve's inverses a stage ahead, the influence data and the iterate to compare
// with ahead of the Helmholtz solves), addresses are a uniform base plus a
// 32-bit offset, stencils run over zero rows at both ends without bounds
// checks, and the sums are fused multiply-adds.  Against the row-by-row solves
// with their LDS ring of factors, and separately rounded stencils, this took a
// launch from 69 to 41 us at (64,64,48) (148 MB, 3.6 TB/s), 1395 to 860 us at
// (96,256,128), 26.5 to 11.7 us at (32,24,12) and 21.8 to 10.9 us at (16,6,4);
// without spilled registers 37 and 723 us at the larger two, the control step
// included.
#include <hip/hip_runtime.h>

#include "kernels.hpp"
#include "solve.hpp"

// no contraction by the compiler: every instantiation rounds alike
#pragma clang fp contract(off)

namespace opf {

namespace {

struct Slot {
  bool valid;
  bool h00;
  int pl, s, p, m, ka, k, h;
};

__device__ __forceinline__ Slot slot_of(int lh, int gp, int np, int p0, int K) {
  Slot r;
  r.pl = lh % gp;
  r.s = lh / gp;
  r.p = p0 + r.pl;
  r.m = r.p / K;
  r.ka = r.p - r.m * K;
  r.k = r.s ? -r.ka : r.ka;
  r.valid = r.pl < np && (r.s == 0 || (r.ka > 0 && r.m > 0));
  r.h = r.m == 0 ? r.k : K + (r.m - 1) * (2 * K - 1) + r.k + K - 1;
  r.h00 = r.valid && r.h == 0;
  return r;
}

// wall boundary residuals (vel_evalBC, velocity.f90:262-298)
__device__ __forceinline__ void eval_bc5(const double2* up, const double2* um, double2 uzN, const double* dr1c,
                                         double d, double m_, double a_, double BRe[4], double BIm[4]) {
  const double2 upN = up[KL], umN = um[KL];
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

// max |du|^2 of a corrector as a bit pattern: the values are sums of squares, so
// their patterns order as they do, and a NaN (its sign cleared) sorts above
// them all, where fmax would drop it and count the corrector as converged
__device__ __forceinline__ unsigned long long du_bits(double d, bool nan) {
  return nan ? 0x7ff8000000000000ull : (unsigned long long)__double_as_longlong(d);
}
__device__ __forceinline__ unsigned long long du_max(unsigned long long a, unsigned long long b) { return a > b ? a : b; }

__device__ __forceinline__ double pr0_of(const double2* uz0, size_t hs, int N, const double* dr1c) {
  // vel_Pr0 = dot_product(uz%Re(N-KL:N,0), dr1(:,1)) / (-2)  (velocity.f90:356-357)
  double s = 0.0;
#pragma unroll
  for (int i = 0; i <= KL; ++i) s = s + uz0[(size_t)(N - 1 - KL + i) * hs].x * dr1c[i];
  return s / (-2.0);
}

// ---------------------------------------------------------------------------
// tim_check_cgce (timestep.f90:214-253), buffer roles, time and step counters
// of one slot: one thread, on the slot's control block, after every
// workgroup's part of the step.  Pr0 and Pr0_hpf are another workgroup's to
// write.  dt2: max |du|^2 of a corrector, a NaN if there was one; E, Ek0, Em0: var_coll_norm of a
// diagnostics step.
// ---------------------------------------------------------------------------
__device__ __forceinline__ void control_decide(SlotCtl* c, const SlotParams& prm, DiagRec* recs, bool diag_now,
                                               double dt2, double E, double Ek0, double Em0) {
  SlotCtl k = *c;
  c->arrived = 0u;
  if (k.mode == MODE_PRED) {
    if (diag_now) {
      DiagRec* rec = recs + (k.ndiag % k.diag_cap);
      rec->E = E;
      rec->Ek0 = Ek0;
      rec->Em0 = Em0;
      rec->ncorr = -1.0;
      rec->dterr = 0.0;
      c->ndiag = k.ndiag + 1;
    }
    // vel_predictor done: u_ := old current, N_ := this evaluation's raw N
    c->ubase = k.ucur;
    c->ucur = k.unext;
    c->unext = k.ubase;
    c->npred = k.ncur;
    c->ncur = 1 - k.ncur;
    c->it = 1;
    c->ncorr = 0;
    c->lasterr = 1e99;
    c->mode = MODE_CORR;
    return;
  }
  // corrector done
  const double dterr = sqrt(dt2);
  const int ncorr = k.ncorr + 1;
  c->ncorr = ncorr;
  c->ucur = k.unext;
  c->unext = k.ucur;
  c->last_dterr = dterr;
  if (k.host_driven) return;   // the caller applies tim_check_cgce itself
  int it = k.it;
  if (it == 1) {
    c->corr_dt = prm.dt * sqrt(prm.dterr_tol / dterr);
    c->lasterr = k.lasterr = 1e99;
  }
  int fail = OPF_FAIL_NONE;
  if (!(dterr == dterr)) {
    fail = OPF_FAIL_NAN;
    it = 0;
  } else if (prm.dt < 1e-9 && k.step > 30) {
    fail = OPF_FAIL_DT0;
    it = 0;
  } else if (it > 10) {
    fail = OPF_FAIL_ITS;
    it = 0;
  } else if (dterr > k.lasterr) {
    if (dterr > 2.0 * prm.dterr_tol) fail = OPF_FAIL_INCERR;
    else c->corr_dt = prm.dt / (10.0 * prm.courant);
    it = 0;
  } else if (dterr > prm.dterr_tol) {
    c->lasterr = dterr;
    it = it + 1;
  } else {
    it = 0;
  }
  if (k.corr_fixed > 0) it = ncorr >= k.corr_fixed ? 0 : (it == 0 ? 1 : it);
  if (fail != OPF_FAIL_NONE && k.corr_fixed <= 0) {
    c->status = fail;
    c->active = 0;
    return;
  }
  c->it = it;
  if (it == 0) {
    // step complete: tim_t += dt, tim_step += 1 (main.f90:43-44)
    if (k.diag_every > 0 && k.ndiag > 0) {
      DiagRec* rec = recs + ((k.ndiag - 1) % k.diag_cap);
      if ((int)rec->step == k.step) {
        rec->ncorr = ncorr;
        rec->dterr = dterr;
      }
    }
    c->last_ncorr = ncorr;
    c->t = k.t + prm.dt;
    c->step = k.step + 1;
    c->mode = MODE_PRED;
    if (k.target_steps >= 0 && k.step + 1 >= k.target_steps) c->active = 0;
  }
}

// The systems of the sets m0 .. m0 + nf - 1 of pair p with their LAPACK-form
// factors, in place, a lane per system: the fields f0 .. of V (VC double2 apart,
// V at the pair's harmonic +k; -k is gp further), rows 2 gp double2 apart.
__device__ void band_solve(const Geo& G, const Bufs& B, int slot, int f0, int nf, int m0, int p, double2* V, int VC,
                           int gp, int lane) {
  const int f = lane >> 1, N = G.N;
  if (f >= nf) return;
  double2* x = V + (f0 + f) * VC + gp * (lane & 1);
  if (B.spec[slot * 4 + m0 + f].BC == 1 && p == 0) {   // singular (timestep.f90:84): zero
    for (int n = 0; n < N; ++n) x[n * 2 * gp] = make_double2(0.0, 0.0);
    return;
  }
  const LuFactors L = B.sets[slot * 4 + m0 + f].lu;
  lu_solve<double2>(L.F + (size_t)p * N * LUS, L.pv + (size_t)p * N, x, 2 * gp, N);
}

// IT: (radial point, harmonic) items per thread in the parallel stages,
// N * 2 * GP <= IT * THR; THR: threads of the workgroup; SM >= blk_mid(N).
// BAND: slots marked banded are solved with the LAPACK-form factors.
template <int GP, int IT, int THR, int SM, bool BAND>
__device__ __forceinline__ void step_body(const Geo& G, const Bufs& B, const StepTiles& ST, int slot0) {
  const int slot = slot_of(B, slot0);
  SlotCtl* ctl = &B.ctl[slot];
  const SlotCtl ct = *ctl;              // both control blocks in one round trip
  const SlotParams prm = B.prm[slot];
  if (!ct.active) return;
  // XCD-aware group order: consecutive workgroup ids go to different XCDs,
  // so give each XCD a contiguous range of pairs (neighbouring harmonics
  // share cache lines of the spectral fields).
  const int per = (ST.ngroups + 7) / 8;
  const int grp = (blockIdx.x % 8) * per + blockIdx.x / 8;
  if (grp >= ST.ngroups) return;
  const int N = G.N, P = G.P, K = G.K;
  const int p0 = grp * GP;
  const int np = min(GP, P - p0);
  const int tid = threadIdx.x;
  const MeshOff mo = MeshOff::make(N);
  const double* __restrict__ me = G.mesh;
  const double* dr1c = me + mo.dr1 + (KL + 1);
  const bool corr = ct.mode == MODE_CORR;
  const bool want_diag = !corr && ct.diag_every > 0 && (ct.step % ct.diag_every) == 0;
  constexpr int GH = 2 * GP;
  // the fields of the slot: wave-uniform bases, 32-bit byte offsets per item.
  // Distinct buffers (the ring of velocity roles; uc and ub coincide only in
  // the predictor, where both are read-only), so restrict-qualified: loads
  // may move past the stores of un and om.
  const size_t s3 = (size_t)slot * 3 * G.coll;
  const unsigned cb = (unsigned)(G.coll * sizeof(double2)), rb = (unsigned)G.Hp * (unsigned)sizeof(double2);
  const char* __restrict__ uc = (const char*)(B.U[ct.ucur] + s3);   // current iterate
  const char* __restrict__ ub = (const char*)(B.U[corr ? ct.ubase : ct.ucur] + s3);   // u_ (vel_predictor: u_ = u)
  char* __restrict__ un = (char*)(B.U[ct.unext] + s3);
  const char* __restrict__ Nc = (const char*)(B.Nraw[ct.ncur] + s3);
  const char* __restrict__ Np = (const char*)(B.Nraw[ct.npred] + s3);
  char* __restrict__ om = (char*)(B.om + s3);

  // LDS (step_lds_doubles): V, rows -4 .. N+3; LT, the Laplacian's rows; DT,
  // the first derivative's, and Ubase, 2r, 1/r^2; the influence coefficients;
  // reduction words
  extern __shared__ double2 lds2[];
  const int VC = (N + 8) * GH;      // double2 per field
  double2* V = lds2 + KL * GH;      // V[c * VC + n * GH + lh]
  double* LT = (double*)(lds2 + 3 * VC);
  double* DT = LT + 10 * (N + 8);
  double* AC = DT + 13 * N + (N & 1);   // [GH][8]
  double* RED = AC + GH * 8;            // [16]
  double* EN = (double*)(V + 2 * VC);               // energy terms [2][N][GH] in V's third field
  const double* RV = DT + 10 * N;

  const double th = prm.implicit, th1 = 1.0 - prm.implicit;
  const double c1 = 1.0 / prm.dt;
  const double c2 = (1.0 - prm.implicit) * prm.nu / prm.Re;
  const int NI = N * GH;
  // items it = tid + q * THR of the parallel stages: radial point it / GH,
  // harmonic slot it % GH, the same slot for all of a thread's items
  static_assert(THR % GH == 0, "threads must cover whole radial rows");
  const int lh = tid % GH, n0 = tid / GH;
  constexpr int DN = THR / GH;   // a thread's items are DN rows apart
  const Slot S = slot_of(lh, GP, np, p0, K);
  const double ak = prm.alpha * (double)S.k, mm = (double)G.Mp * (double)S.m;
  const bool has00 = p0 == 0;
  const unsigned ho = (unsigned)S.h * (unsigned)sizeof(double2);

  // a row of the mesh tables: nine weights and the tenth value
  auto row10 = [](const double* src, double (&w)[10]) {
#pragma unroll
    for (int i = 0; i < 5; ++i) {
      const double2 a = ((const double2*)src)[i];
      w[2 * i] = a.x;
      w[2 * i + 1] = a.y;
    }
  };

  // ---- stage 0: loads ------------------------------------------------------
  // the mesh tables first (one batch, ahead of the state loads)
  constexpr int WMAX = DN * IT;   // N <= WMAX
  constexpr int TT = ((23 * WMAX + 81) / 2 + THR - 1) / THR;
  const int ntab = (10 * (N + 8) + 13 * N + 1) / 2;   // d1T and rowv follow lapT
  double2 tab[TT];
#pragma unroll
  for (int u = 0; u < TT; ++u) {
    const int i = tid + u * THR;
    tab[u] = ((const double2*)(me + mo.lapT))[i < ntab ? i : 0];
  }
  // u_, N and, for the corrector, the iterate and N_ of all items in one batch
  double2 vb[IT][3], vc[IT][3], vn[IT][3], vp[IT][3];
#pragma unroll
  for (int q = 0; q < IT; ++q) {
    const int n = n0 + q * DN;
    const unsigned o = n < N && S.valid ? (unsigned)n * rb + ho : 0u;
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      vb[q][c] = *(const double2*)(ub + (size_t)(c * cb) + o);
      vn[q][c] = *(const double2*)(Nc + (size_t)(c * cb) + o);
    }
  }
  auto load_np = [&]() {
#pragma unroll
    for (int q = 0; q < IT; ++q) {
      const int n = n0 + q * DN;
      const unsigned o = n < N && S.valid ? (unsigned)n * rb + ho : 0u;
#pragma unroll
      for (int c = 0; c < 3; ++c) vp[q][c] = *(const double2*)(Np + (size_t)(c * cb) + o);
    }
  };
  // Registers: with two items, a thread's loads of N_ wait for the others and
  // the influence loads stand behind the Helmholtz solve, which leaves three
  // waves a SIMD without spills (44.8 us with 21 spilled registers, 37.1 without,
  // at (64,64,48)); with three, two waves of 256 registers are better than
  // three of 168 (886 to 723 us at (96,256,128)).
  constexpr bool LATE_NP = IT == 2;
  if (corr) {
#pragma unroll
    for (int q = 0; q < IT; ++q) {
      const int n = n0 + q * DN;
      const unsigned o = n < N && S.valid ? (unsigned)n * rb + ho : 0u;
#pragma unroll
      for (int c = 0; c < 3; ++c) vc[q][c] = *(const double2*)(uc + (size_t)(c * cb) + o);
    }
    if (!LATE_NP) load_np();
  }
  // the mean flow's pressure gradients of both iterates (harmonic (0,0))
  double prc = 0.0, prb = 0.0;
  if (has00 && prm.const_flux) {
    prc = pr0_of((const double2*)(uc + (size_t)(2 * cb)), G.Hp, N, dr1c);
    prb = pr0_of((const double2*)(ub + (size_t)(2 * cb)), G.Hp, N, dr1c);
  }
#pragma unroll
  for (int u = 0; u < TT; ++u)
    if (tid + u * THR < ntab) ((double2*)LT)[tid + u * THR] = tab[u];
  // zero rows at either end of the three fields
  for (int i = tid; i < 3 * 8 * GH; i += THR) {
    const int c = i / (8 * GH), r = i - c * 8 * GH;
    V[c * VC + (r < 4 * GH ? r - 4 * GH : r + (N - 4) * GH)] = make_double2(0.0, 0.0);
  }
  // u_ as (u+, u-, uz) for the stencil
#pragma unroll
  for (int q = 0; q < IT; ++q) {
    const int n = n0 + q * DN;
    if (n >= N) continue;
    if (!S.valid) {
#pragma unroll
      for (int c = 0; c < 3; ++c) vb[q][c] = make_double2(0.0, 0.0);
    }
    if (!corr) {
#pragma unroll
      for (int c = 0; c < 3; ++c) vc[q][c] = vb[q][c];
    }
    const double2 r = vb[q][0], t = vb[q][1];
    V[n * GH + lh] = make_double2(r.x - t.y, r.y + t.x);
    V[VC + n * GH + lh] = make_double2(r.x + t.y, r.y - t.x);
    V[2 * VC + n * GH + lh] = vb[q][2];
  }
  __syncthreads();

  // ---- stage 1: effective N and RHS = Lt u_ + N (tim_meshmult) -----------
  // Results are held in registers until every thread has read its stencil
  // from u_, then written over it; the third field then takes the pressure,
  // and the right-hand side of uz stays in registers.
  double2 res[IT][3];
#pragma unroll
  for (int q = 0; q < IT; ++q) {
    const int n = n0 + q * DN;
    if (n >= N || !S.valid) continue;
    const double a = ak * RV[n];
    const double b = RV[N + n];
    const double2 ucr = vc[q][0], uct = vc[q][1], ucz = vc[q][2];
    double2 nr = vn[q][0], nt = vn[q][1], nz = vn[q][2];
    nr = make_double2(fma(a, ucr.y, nr.x), fma(-a, ucr.x, nr.y));
    nt = make_double2(fma(a, uct.y, nt.x), fma(-a, uct.x, nt.y));
    nz = make_double2(fma(b, ucr.x, fma(a, ucz.y, nz.x)), fma(b, ucr.y, fma(-a, ucz.x, nz.y)));
    if (S.h00) nz.x = nz.x + (4.0 * prc) / prm.Re;
    vn[q][0] = nr;
    vn[q][1] = nt;
    vn[q][2] = nz;
  }
  if (LATE_NP && corr) {
    __builtin_amdgcn_sched_barrier(0);
    load_np();
    __builtin_amdgcn_sched_barrier(0);
  }
#pragma unroll
  for (int q = 0; q < IT; ++q) {
    const int n = n0 + q * DN;
    res[q][0] = res[q][1] = res[q][2] = make_double2(0.0, 0.0);
    if (n >= N || !S.valid) continue;
    const double a = ak * RV[n];
    const double b = RV[N + n];
    double2 nr = vn[q][0], nt = vn[q][1], nz = vn[q][2];
    if (corr) {
      const double2 bur = vb[q][0], but = vb[q][1], buz = vb[q][2];
      double2 pr = vp[q][0], pt = vp[q][1], pz = vp[q][2];
      pr = make_double2(fma(a, bur.y, pr.x), fma(-a, bur.x, pr.y));
      pt = make_double2(fma(a, but.y, pt.x), fma(-a, but.x, pt.y));
      pz = make_double2(fma(b, bur.x, fma(a, buz.y, pz.x)), fma(b, bur.y, fma(-a, buz.x, pz.y)));
      if (S.h00) pz.x = pz.x + (4.0 * prb) / prm.Re;
      nr = make_double2(fma(th, nr.x, th1 * pr.x), fma(th, nr.y, th1 * pr.y));
      nt = make_double2(fma(th, nt.x, th1 * pt.x), fma(th, nt.y, th1 * pt.y));
      nz = make_double2(fma(th, nz.x, th1 * pz.x), fma(th, nz.y, th1 * pz.y));
    }
    // the Laplacian's radial part, sum of weight times row
    double2 sp = make_double2(0.0, 0.0), sm = sp, sz = sp;
    double w[10];
    row10(LT + 10 * n, w);
    const double2* v = V + (n - KL) * GH + lh;
#pragma unroll
    for (int dd = 0; dd < LDA; ++dd) {
      const double2 vp_ = v[dd * GH], vm_ = v[VC + dd * GH], vz_ = v[2 * VC + dd * GH];
      sp = make_double2(fma(w[dd], vp_.x, sp.x), fma(w[dd], vp_.y, sp.y));
      sm = make_double2(fma(w[dd], vm_.x, sm.x), fma(w[dd], vm_.y, sm.y));
      sz = make_double2(fma(w[dd], vz_.x, sz.x), fma(w[dd], vz_.y, sz.y));
    }
    // diagonal terms: c1 - c2 ((mm +- 1)^2 / r^2 + ak^2)
    const double r2i = RV[2 * N + n];
    const double dz = -fma(r2i * mm, mm, ak * ak);
    const double gp = fma(c2, fma(-r2i, fma(2.0, mm, 1.0), dz), c1);
    const double gm = fma(c2, fma(-r2i, fma(-2.0, mm, 1.0), dz), c1);
    const double gz = fma(c2, dz, c1);
    const double2 up = v[KL * GH], um = v[VC + KL * GH], uz = v[2 * VC + KL * GH];
    res[q][0] = make_double2((nr.x - nt.y) + fma(c2, sp.x, gp * up.x), (nr.y + nt.x) + fma(c2, sp.y, gp * up.y));
    res[q][1] = make_double2((nr.x + nt.y) + fma(c2, sm.x, gm * um.x), (nr.y - nt.x) + fma(c2, sm.y, gm * um.y));
    res[q][2] = make_double2(nz.x + fma(c2, sz.x, gz * uz.x), nz.y + fma(c2, sz.y, gz * uz.y));
  }
  // the pressure factors are in flight while the next stages run.  Wave w
  // solves pair w.
  const int wave = tid >> 6;
  const BlkLane bl = BlkLane::make(tid & 63);
  const bool solver = wave < GP;
  const int ps = p0 + min(wave, np - 1);   // a missing pair of the last group repeats a factor on zeros
  const int lhs = wave + GP * (bl.col >> 1);
  BlkE<SM, 1> EP;
  if (solver) blk_load(EP, 0, G, B, slot, B.spec[slot * 4 + MAT_LNP], MAT_LNP, ps, bl);
  __syncthreads();
#pragma unroll
  for (int q = 0; q < IT; ++q) {
    const int n = n0 + q * DN;
    if (n >= N) continue;
    V[n * GH + lh] = res[q][0];
    V[VC + n * GH + lh] = res[q][1];
  }
  if (want_diag) {
    if (S.h00 && n0 == 0) {
      const double2* uz = (const double2*)(uc + (size_t)(2 * cb));
      double s = 0.0, f = 0.0;
      for (int i = 0; i <= KL; ++i) s = s + uz[(size_t)i * G.Hp].x * me[mo.dr0 + i];
      for (int i = 0; i <= KL; ++i) f = f + uz[(size_t)(N - 1 - KL + i) * G.Hp].x * dr1c[i];
      DiagRec* rec = B.diag + (size_t)slot * ct.diag_cap + (ct.ndiag % ct.diag_cap);
      rec->step = ct.step;
      rec->t = ct.t;
      if (prm.const_flux) {
        rec->Ub = prc;
      } else {   // io.f90:630
        double q2 = 0.0;
        for (int i = 0; i < N; ++i) q2 = q2 + uz[(size_t)i * G.Hp].x * me[mo.intrdr + i];
        rec->Ub = 0.5 + 2.0 * q2;
      }
      rec->Uc = 1.0 + s;
      rec->Ufr = sqrt(fabs((f - 2.0) / prm.Re));
    }
    // energy partials (var_coll_norm, variables.f90:732-735), n ascending:
    // two components, then the third, through V's third field
    const double wnorm = 4.0 * D_PI * D_PI / prm.alpha;
    for (int cc = 0; cc < 3; cc += 2) {
#pragma unroll
      for (int q = 0; q < IT; ++q) {
        const int n = n0 + q * DN;
        if (n >= N) continue;
        const double2 a = cc == 0 ? vb[q][0] : vb[q][2], b = vb[q][1];   // the iterate of a predictor is u_
        EN[n * GH + lh] = S.valid ? wnorm * (a.x * a.x + a.y * a.y) : 0.0;
        if (cc == 0) EN[NI + n * GH + lh] = S.valid ? wnorm * (b.x * b.x + b.y * b.y) : 0.0;
      }
      __syncthreads();
      if (tid < (cc == 0 ? 2 : 1) * GH && slot_of(tid % GH, GP, np, p0, K).valid) {
        const int c = tid / GH, l = tid - c * GH;
        const Slot Sd = slot_of(l, GP, np, p0, K);
        double bsum = 0.0;
        for (int n = 0; n < N; ++n) bsum = bsum + EN[c * NI + n * GH + l] * me[mo.intrdr + n];
        if (Sd.h00) bsum = 0.5 * bsum;
        B.diagb[(size_t)slot * 3 * G.Hp + (size_t)(cc + c) * G.Hp + Sd.h] = bsum;
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");   // for the workgroup that sums them
      }
      __syncthreads();
    }
  }
  __syncthreads();

  // ---- stage 2: pressure RHS = div(pm2rt(R+, R-), Rz) (vel_adjPPE(1)) ----
#pragma unroll
  for (int q = 0; q < IT; ++q) {
    const int n = n0 + q * DN;
    if (n >= N) continue;
    double2 dv = make_double2(0.0, 0.0);
    if (S.valid && !S.h00 && n != 0 && n != N - 1) {
      double w[10];
      row10(DT + 10 * n, w);
      const double2* v = V + (n - KL) * GH + lh;
      double2 d = make_double2(0.0, 0.0);
#pragma unroll
      for (int dd = 0; dd < LDA; ++dd) {
        const double2 a = v[dd * GH], b = v[VC + dd * GH];
        d.x = fma(w[dd], a.x + b.x, d.x);
        d.y = fma(w[dd], a.y + b.y, d.y);
      }
      // u_r = (R+ + R-)/2, u_th = (R+ - R-)/2i
      const double2 a = v[KL * GH], b = v[VC + KL * GH], z = res[q][2];
      const double ri = w[9], mr = ri * mm;
      dv.x = fma(0.5, fma(a.x - b.x, mr, fma(a.x + b.x, ri, d.x)), -(z.y * ak));
      dv.y = fma(0.5, fma(a.y - b.y, mr, fma(a.y + b.y, ri, d.y)), z.x * ak);
    }
    V[2 * VC + n * GH + lh] = dv;
  }
  __syncthreads();

  // ---- stage 3: pressure solve with LNp (tim_lumesh_invert(1,...)) -------
  // (harmonics without a mode or with none to solve hold zeros and stay so)
  if (solver) {
    double* const x[1] = {(double*)(V + 2 * VC + lhs) + (bl.col & 1)};
    if (!BAND || !B.sets[slot * 4].banded) blk_solve(EP, N, bl, LT, x, 2 * GH);
    else band_solve(G, B, slot, 2, 1, MAT_LNP, ps, V + wave, VC, GP, tid & 63);
  }
  BlkE<SM, 2> EH;
  if (solver) {
    blk_load(EH, 0, G, B, slot, B.spec[slot * 4 + MAT_LDP + bl.mi], MAT_LDP + bl.mi, ps, bl);
    blk_load(EH, 1, G, B, slot, B.spec[slot * 4 + MAT_LDZ], MAT_LDZ, ps, bl);
  }
  __syncthreads();

  // ---- stage 4: subtract grad p (rt2pm), zero the BC rows ----------------
#pragma unroll
  for (int q = 0; q < IT; ++q) {
    const int n = n0 + q * DN;
    if (n >= N || !S.valid) continue;
    double2 r0 = make_double2(0.0, 0.0), r1 = r0, r2 = r0;
    if (n != 0 && n != N - 1) {
      double w[10];
      row10(DT + 10 * n, w);
      const double2* v = V + 2 * VC + (n - KL) * GH + lh;
      double2 gr = make_double2(0.0, 0.0);
#pragma unroll
      for (int dd = 0; dd < LDA; ++dd) {
        const double2 pj = v[dd * GH];
        gr.x = fma(w[dd], pj.x, gr.x);
        gr.y = fma(w[dd], pj.y, gr.y);
      }
      const double2 pv = v[KL * GH];
      const double mr = w[9] * mm;
      r0 = V[n * GH + lh];
      r1 = V[VC + n * GH + lh];
      // rt2pm(grad p) = (gr - mr p, gr + mr p)
      r0 = make_double2(r0.x - fma(-mr, pv.x, gr.x), r0.y - fma(-mr, pv.y, gr.y));
      r1 = make_double2(r1.x - fma(mr, pv.x, gr.x), r1.y - fma(mr, pv.y, gr.y));
      r2 = make_double2(fma(ak, pv.y, res[q][2].x), fma(-ak, pv.x, res[q][2].y));
    }
    V[n * GH + lh] = r0;
    V[VC + n * GH + lh] = r1;
    res[q][2] = r2;
  }
  __syncthreads();
#pragma unroll
  for (int q = 0; q < IT; ++q) {
    const int n = n0 + q * DN;
    if (n < N) V[2 * VC + n * GH + lh] = res[q][2];
  }
  __syncthreads();

  // ---- stage 5: Helmholtz solves LDp, LDm, LDz ---------------------------
  // the influence step's global inputs: the influence vectors, the iterate
  // that the corrector compares with, a row of the 4x4 inverses.  Ahead of the
  // solve, or, where the registers do not hold both, behind it.
  double uv[IT][6];
  double2 old[IT][3];
  double ai[4] = {0.0, 0.0, 0.0, 0.0};
  const int clh = tid >> 2, ci = tid & 3;   // coefficient thread: harmonic slot, row of the inverse
  const Slot CS = slot_of(clh % GH, GP, np, p0, K);
  const bool cf = tid < 4 * GH && CS.valid && !CS.h00;
  auto influence_loads = [&]() {
#pragma unroll
    for (int q = 0; q < IT; ++q) {
      const int n = n0 + q * DN;
      const bool ok = n < N && S.valid;
      const char* U = (const char*)(B.Uinf + (size_t)slot * 6 * N * P);
      const unsigned us = (unsigned)(N * P) * 8u, o = ok ? (unsigned)(n * P + S.p) * 8u : 0u;
#pragma unroll
      for (int i = 0; i < 6; ++i) uv[q][i] = *(const double*)(U + (size_t)(i * us) + o);
      if (corr) {
        const unsigned oo = ok ? (unsigned)n * rb + ho : 0u;
#pragma unroll
        for (int c = 0; c < 3; ++c) old[q][c] = *(const double2*)(uc + (size_t)(c * cb) + oo);
      }
    }
    if (cf) {
#pragma unroll
      for (int j = 0; j < 4; ++j) ai[j] = B.Ainv[(size_t)slot * 16 * G.H + (size_t)(ci * 4 + j) * G.H + CS.h];
    }
  };
  constexpr bool EARLY = IT != 2;
  if (EARLY || !solver) influence_loads();
  if (solver) {
    double* xp = (double*)(V + lhs) + (bl.col & 1);
    double* const x[2] = {xp + (bl.mi ? 2 * VC : 0), xp + 4 * VC};
    if (!BAND || !B.sets[slot * 4].banded) blk_solve(EH, N, bl, LT, x, 2 * GH);
    else band_solve(G, B, slot, 0, 3, MAT_LDP, ps, V + wave, VC, GP, tid & 63);
    if (!EARLY) influence_loads();
  }
  __syncthreads();

  // ---- stage 6: influence-matrix correction (vel_adjPPE(2)) --------------
  if (tid < 4 * GH) {
    double sR = 0.0, sI = 0.0;
    if (cf) {
      double2 wp[KL + 1], wm[KL + 1], wz = V[2 * VC + (N - 1) * GH + clh];
#pragma unroll
      for (int i = 0; i <= KL; ++i) {
        wp[i] = V[(N - 1 - KL + i) * GH + clh];
        wm[i] = V[VC + (N - 1 - KL + i) * GH + clh];
      }
      double BRe[4], BIm[4];
      eval_bc5(wp, wm, wz, dr1c, me[mo.rinv + N - 1], (double)(CS.m * G.Mp), prm.alpha * (double)CS.k, BRe, BIm);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        sR = fma(ai[j], BRe[j], sR);
        sI = fma(ai[j], BIm[j], sI);
      }
    }
    AC[clh * 8 + ci] = -sR;
    AC[clh * 8 + 4 + ci] = -sI;
  }
  __syncthreads();
  double2 nu[IT][3];
#pragma unroll
  for (int q = 0; q < IT; ++q) {
    const int n = n0 + q * DN;
    nu[q][0] = nu[q][1] = nu[q][2] = make_double2(0.0, 0.0);
    if (n >= N || !S.valid) continue;
    double2 up = V[n * GH + lh], um = V[VC + n * GH + lh], uz = V[2 * VC + n * GH + lh];
    if (!S.h00) {
      const double* aR = AC + lh * 8;
      const double* aI = aR + 4;
      const double U6 = uv[q][5] * ak;
      up = make_double2(fma(aR[3], uv[q][3], fma(aR[0], uv[q][0], up.x)), fma(aI[3], uv[q][3], fma(aI[0], uv[q][0], up.y)));
      um = make_double2(fma(aR[3], uv[q][4], fma(aR[1], uv[q][1], um.x)), fma(aI[3], uv[q][4], fma(aI[1], uv[q][1], um.y)));
      uz = make_double2(fma(-aI[3], U6, fma(-aI[2], uv[q][2], uz.x)), fma(aR[3], U6, fma(aR[2], uv[q][2], uz.y)));
    }
    // vel_pm2rt
    nu[q][0] = make_double2(0.5 * (up.x + um.x), 0.5 * (up.y + um.y));
    nu[q][1] = make_double2(0.5 * (up.y - um.y), -0.5 * (up.x - um.x));
    nu[q][2] = uz;
    V[VC + n * GH + lh] = nu[q][1];
    V[2 * VC + n * GH + lh] = uz;
  }
  // vel_adjustFlux(1) (velocity.f90:170-175) on harmonic (0,0): the radial
  // quadrature over one wave's lanes, n = lane and lane + 64
  if (has00) {
    __syncthreads();
    if (tid < 64) {
      double d3 = 0.0, s = 0.0;
      if (prm.const_flux) {
        for (int n = tid; n < N; n += 64) s = s + V[2 * VC + n * GH].x * me[mo.intrdr + n];
        for (int off = 32; off >= 1; off >>= 1) s = s + __shfl_xor(s, off);
        d3 = -(2.0 * s) / ct.flux_d1;
      }
      if (tid == 0) {
        RED[0] = d3;
        ctl->Pr0 = prc + (d3 * prm.Re) / 4.0;
        ctl->Pr0_hpf = prc;
      }
    }
    __syncthreads();
    if (S.h00) {
#pragma unroll
      for (int q = 0; q < IT; ++q) {
        const int n = n0 + q * DN;
        if (n >= N) continue;
        if (prm.const_flux) nu[q][2].x = fma(RED[0], B.Ui[(size_t)slot * N + n], nu[q][2].x);
        nu[q][0] = make_double2(0.0, 0.0);
        nu[q][1].y = 0.0;
        nu[q][2].y = 0.0;
        V[VC + n * GH + lh] = nu[q][1];
        V[2 * VC + n * GH + lh] = nu[q][2];
      }
    }
  }
  unsigned long long* WD = (unsigned long long*)(RED + 1);   // the waves' maxima
  if (corr) {
    double dmax = 0.0;
    bool nan = false;
#pragma unroll
    for (int q = 0; q < IT; ++q) {
      if (n0 + q * DN >= N || !S.valid) continue;
#pragma unroll
      for (int c = 0; c < 3; ++c) {
        const double dx = old[q][c].x - nu[q][c].x, dy = old[q][c].y - nu[q][c].y;
        const double d = fma(dx, dx, dy * dy);
        nan = nan || d != d;
        dmax = fmax(dmax, d);
      }
    }
    for (int off = 32; off >= 1; off >>= 1) dmax = fmax(dmax, __shfl_xor(dmax, off));
    nan = __any(nan);
    if ((tid & 63) == 0) WD[wave] = du_bits(dmax, nan);
  }
  __syncthreads();

  // This workgroup's maximum, and its arrival: the last one to arrive takes
  // the control step (control_decide).  An arrival follows the return of its
  // workgroup's exchange, and both round trips run behind the stores and the
  // curl.  Arrivals at one word cost about 3 ns each, so many workgroups
  // arrive at ARRIVE_WORDS words first, and the last at each of those at the
  // slot's.  A kernel of its own for the control step took 4.6 us per
  // evaluation; this takes 1.3 us at (32,24,12) and 3 us at (64,64,48).
  unsigned long long* arr = B.arrive + (size_t)slot * arrive_words(P);
  const int nsub = ST.ngroups > 2 * ARRIVE_WORDS ? ARRIVE_WORDS : 1;
  const int sub = grp % nsub;
  unsigned long long prev = 0ull, cnt = 0ull;
  if (tid == 0 && corr) {
    unsigned long long wd = WD[0];
#pragma unroll
    for (int w = 1; w < THR / 64; ++w) wd = du_max(wd, WD[w]);
    prev = __hip_atomic_exchange(arr + 16 * ARRIVE_WORDS + grp, wd, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
#pragma unroll
  for (int q = 0; q < IT; ++q) {
    const int n = n0 + q * DN;
    if (n >= N || !S.valid) continue;
    const unsigned o = (unsigned)n * rb + ho;
#pragma unroll
    for (int c = 0; c < 3; ++c) *(double2*)(un + (size_t)(c * cb) + o) = nu[q][c];
  }
  if (tid == 0) {
    asm volatile("" ::"v"(prev) : "memory");
    cnt = __hip_atomic_fetch_add(arr + 16 * sub, 1ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }

  // ---- stage 7: curl of the new velocity for the next evaluation ---------
#pragma unroll
  for (int q = 0; q < IT; ++q) {
    const int n = n0 + q * DN;
    if (n >= N || !S.valid) continue;
    double w[10];
    row10(DT + 10 * n, w);
    const double2* v = V + (n - KL) * GH + lh;
    double2 d1 = make_double2(0.0, 0.0), d2 = d1;
#pragma unroll
    for (int dd = 0; dd < LDA; ++dd) {
      const double2 tj = v[VC + dd * GH], zj = v[2 * VC + dd * GH];
      d1.x = fma(w[dd], zj.x, d1.x);
      d1.y = fma(w[dd], zj.y, d1.y);
      d2.x = fma(w[dd], tj.x, d2.x);
      d2.y = fma(w[dd], tj.y, d2.y);
    }
    const double ri = w[9], mr = ri * mm;
    const double2 vr = nu[q][0], vt = nu[q][1], vz = nu[q][2];
    const unsigned o = (unsigned)n * rb + ho;
    double2 cw[3];
    curl_of(vr, vt, vz, d1, d2, ri, mr, ak, cw);
#pragma unroll
    for (int c = 0; c < 3; ++c) *(double2*)(om + (size_t)(c * cb) + o) = cw[c];
  }
  if (tid == 0) {
    bool last = cnt == (unsigned long long)((ST.ngroups - sub + nsub - 1) / nsub - 1);
    if (last) {
      arr[16 * sub] = 0ull;
      if (nsub > 1)
        last = __hip_atomic_fetch_add(&ctl->arrived, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == nsub - 1u;
    }
    RED[0] = last ? 1.0 : 0.0;
  }
  __syncthreads();
  if (RED[0] == 0.0) return;
  DiagRec* recs = B.diag + (size_t)slot * ct.diag_cap;
  double* ws = (double*)V;   // [wave][3]
  double dt2 = 0.0;
  if (corr) {
    unsigned long long wd = 0ull;
    for (int i = tid; i < ST.ngroups; i += 4 * THR) {
      unsigned long long w4[4];
#pragma unroll
      for (int u = 0; u < 4; ++u)   // past the end: the last one again
        w4[u] = __hip_atomic_load(arr + 16 * ARRIVE_WORDS + min(i + u * THR, ST.ngroups - 1), __ATOMIC_RELAXED,
                                  __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
      for (int u = 0; u < 4; ++u) wd = du_max(wd, w4[u]);
    }
    for (int off = 32; off >= 1; off >>= 1) wd = du_max(wd, __shfl_xor(wd, off));
    unsigned long long* wsd = (unsigned long long*)V;
    if ((tid & 63) == 0) wsd[wave] = wd;
    __syncthreads();
    for (int w = 0; w < THR / 64; ++w) wd = du_max(wd, wsd[w]);
    dt2 = __longlong_as_double((long long)wd);
  }
  if (!want_diag) {
    if (tid == 0) control_decide(ctl, prm, recs, false, dt2, 0.0, 0.0, 0.0);
    return;
  }
  // var_coll_norm (variables.f90:727-749) from the harmonics' partials
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
  constexpr int DTN = 128;   // summing threads: the same sums for every THR
  double en[3] = {0.0, 0.0, 0.0};   // E, E of k = 0, E of m = 0
  for (int c = 0; c < 3 && tid < DTN; ++c) {
    const double* db = B.diagb + ((size_t)slot * 3 + c) * G.Hp;
    for (int h0 = tid; h0 < G.H; h0 += 8 * DTN) {
      double v[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) v[u] = h0 + u * DTN < G.H ? db[h0 + u * DTN] : 0.0;
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        const int h = h0 + u * DTN;
        en[0] = en[0] + v[u];
        if (h == 0 || (h >= K && (h - K) % (2 * K - 1) == K - 1)) en[1] = en[1] + v[u];
        if (h < K) en[2] = en[2] + v[u];
      }
    }
  }
  for (int i = 0; i < 3; ++i) {
    for (int off = 32; off >= 1; off >>= 1) en[i] = en[i] + __shfl_xor(en[i], off);
    if ((tid & 63) == 0) ws[wave * 3 + i] = en[i];
  }
  __syncthreads();
  if (tid == 0) {
    for (int i = 0; i < 3; ++i) en[i] = en[i] + ws[3 + i];
    control_decide(ctl, prm, recs, true, 0.0, en[0], en[1], en[2]);
  }
}

}  // namespace

template <int GP, int IT, int THR, int SM, int WPE, bool BAND = false>
__global__ void __launch_bounds__(THR) __attribute__((amdgpu_waves_per_eu(WPE)))
k_step_t(Geo G, Bufs B, StepTiles ST, int slot0) {
  step_body<GP, IT, THR, SM, BAND>(G, B, ST, slot0);
}

StepKern step_kernel(int N, int gp) {
  static_assert(blk_mid(32) == 4 && blk_mid(64) == 8 && blk_mid(96) == 12 && blk_mid(MAXN) == 16, "the ranges");
  const int r = N <= 32 ? 0 : N <= 64 ? 1 : N <= 96 ? 2 : 3;
  static const StepKern g1[] = {k_step_t<1, 1, 128, 4, 3>, k_step_t<1, 1, 128, 8, 3>, k_step_t<1, 2, 128, 12, 3>,
                                k_step_t<1, 2, 128, 16, 2>};
  static const StepKern g2[] = {k_step_t<2, 1, 256, 4, 3>, k_step_t<2, 1, 256, 8, 3>, k_step_t<2, 2, 256, 12, 3>,
                                k_step_t<2, 2, 256, 16, 2>};
  static const StepKern g4[] = {k_step_t<4, 1, 256, 4, 3>, k_step_t<4, 2, 256, 8, 3>, k_step_t<4, 3, 256, 12, 2>};
  return gp == 1 ? g1[r] : gp == 2 ? g2[r] : g4[r];
}
StepKern step_kernel_banded() { return k_step_t<1, 2, 128, 16, 2, true>; }

}  // namespace opf
