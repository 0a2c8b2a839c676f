// FP64 linear algebra of the chi-truncation chain (statevector -> chi-MPS).
//
// Step i of the right-to-left truncated projection chain works on
// Y_i = X_{i+1} viewed as a (2^i x n_i) row-major complex128 matrix:
//   rho_i = Y_i^H Y_i             gram + gram_reduce   (n_i x n_i, ld = nmax)
//   rho_i = V diag(lam) V^H       one-sided Jacobi (two-sided by option)
//   W_i   = V[:, top k_i]         select               (rsum2 cutoff, max bond chi)
//   X_i   = Y_i W_i               gemm
// and the state is contracted back with Z_{i+1} = Z_i W_i^H (gemm, conj_b).
// Shapes that depend on the cutoff live on the device (k_i, n_i per state);
// launches are sized by host upper bounds and idle blocks exit early.
#include <algorithm>

#include "qmx_device.h"
#include "qmx_internal.h"

namespace qmx {

// ------------------------------------------------------------------ gram ----
// part[b][chunk] (nmax x nmax) = sum over the chunk's rows of conj(Y)[:, p] Y[:, q]
// 16 T x 16 T entries per block, T x T per thread (every fourth of its tile's
// columns: neighbouring lanes read neighbouring LDS words), rows in steps of
// 16 fetched into registers one step ahead.  Bound by FP64 FMA at T = 4; T = 2
// reads LDS twice as often for the same products and takes the launches whose
// 64 x 64 tiles would leave CUs idle.  32 states of 2^13 x 128: 0.78 ms,
// with 32 x 32 tiles and 1 x 4 entries per thread 1.04.
constexpr int kGemmFill = 512;   // two blocks per CU
template <int T>
__global__ __launch_bounds__(256) void gram_kernel(const double2* __restrict__ y, size_t y_stride,
                                                   const int* ncols_dev, int rows_log2, int nmax,
                                                   double2* part, int nchunks) {
  constexpr int kTile = 16 * T, kStep = 16;
  __shared__ double2 ya[kStep][kTile];
  __shared__ double2 yb[kStep][kTile];
  const int b = blockIdx.z;
  const int nc = ncols_dev[b];
  const int ntile = (nmax + kTile - 1) / kTile;
  const int p0 = blockIdx.x / ntile * kTile, q0 = blockIdx.x % ntile * kTile;
  if (p0 >= nc || q0 >= nc) return;
  const size_t rows = (size_t)1 << rows_log2;
  const size_t per = (rows + nchunks - 1) / nchunks;
  const size_t r0 = per * blockIdx.y;
  const size_t r1 = (r0 + per < rows) ? r0 + per : rows;
  const double2* src = y + (size_t)b * y_stride;
  const int tx = threadIdx.x & 15, ty = threadIdx.x >> 4;
  double2 acc[T][T], fa[T], fb[T];
#pragma unroll
  for (int i = 0; i < T; ++i)
#pragma unroll
    for (int j = 0; j < T; ++j) acc[i][j] = cz();
  auto fetch = [&](size_t rb) {
#pragma unroll
    for (int u = 0; u < T; ++u) {
      const int e = threadIdx.x + 256 * u, rr = e / kTile, cc = e % kTile;
      const size_t row = rb + rr;
      fa[u] = row < r1 && p0 + cc < nc ? src[row * nc + p0 + cc] : cz();
      fb[u] = row < r1 && q0 + cc < nc ? src[row * nc + q0 + cc] : cz();
    }
  };
  fetch(r0);
  for (size_t rb = r0; rb < r1; rb += kStep) {
#pragma unroll
    for (int u = 0; u < T; ++u) {
      const int e = threadIdx.x + 256 * u;
      ya[e / kTile][e % kTile] = fa[u];
      yb[e / kTile][e % kTile] = fb[u];
    }
    __syncthreads();
    if (rb + kStep < r1) fetch(rb + kStep);
#pragma unroll 4
    for (int rr = 0; rr < kStep; ++rr) {
      double2 av[T], bv[T];
#pragma unroll
      for (int i = 0; i < T; ++i) av[i] = ya[rr][ty + 16 * i];
#pragma unroll
      for (int j = 0; j < T; ++j) bv[j] = yb[rr][tx + 16 * j];
#pragma unroll
      for (int i = 0; i < T; ++i)
#pragma unroll
        for (int j = 0; j < T; ++j) acc[i][j] = cfmac(av[i], bv[j], acc[i][j]);
    }
    __syncthreads();
  }
  double2* out = part + ((size_t)b * nchunks + blockIdx.y) * nmax * nmax;
#pragma unroll
  for (int i = 0; i < T; ++i)
#pragma unroll
    for (int j = 0; j < T; ++j) {
      const int p = p0 + ty + 16 * i, q = q0 + tx + 16 * j;
      if (p < nc && q < nc) out[(size_t)p * nmax + q] = acc[i][j];
    }
}

__global__ void gram_reduce_kernel(const double2* part, int nchunks, const int* ncols_dev, int nmax,
                                   double2* a, size_t a_stride) {
  const int b = blockIdx.y;
  const int nc = ncols_dev[b];
  int e = blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= nc * nc) return;
  int p = e / nc, q = e % nc;
  double2 s = cz();
  for (int c = 0; c < nchunks; ++c)
    s = cadd(s, part[((size_t)b * nchunks + c) * nmax * nmax + (size_t)p * nmax + q]);
  a[(size_t)b * a_stride + (size_t)p * nmax + q] = s;
}

// ---------------------------------------------------------------- jacobi ----
// QMX_OPT_TWO_SIDED_JACOBI for 129 to 512 columns.
// Parallel cyclic two-sided Jacobi for a Hermitian n x n matrix (n even,
// n <= 2 * 256), one block per state.  Round r pairs the indices by the circle
// method; all n/2 rotations of a round are disjoint, so the update
// A <- J^H A J is done blockwise: each 2x2 block (P, Q) of A becomes
// J_P^H A_PQ J_Q, independently of every other block.  V accumulates J.
constexpr int kJacobiMaxPairs = 512;

// A pair is rotated only if its off-diagonal entry exceeds kJacobiAbsTol times
// the trace (and 1e-15 of the geometric mean of its diagonal entries).  The
// Gram matrix carries rounding errors of order eps * trace from its own
// formation, and every rotation that involves a large eigenvalue leaves
// errors of that order in the entries it touches; with a floor well below
// that level the rotations inside a cluster of numerically zero eigenvalues
// (rank-deficient Gram matrices: fewer rows than columns) regenerate each
// other's entries and a sweep may never come out clean.  A quarter of eps
// ends those sweeps and leaves the kept subspace as accurate as the Gram
// matrix it comes from.
constexpr double kJacobiAbsTol = 0.25 * 2.220446049250313e-16;

__global__ __launch_bounds__(512) void jacobi_kernel(double2* a_all, double2* v_all, size_t stride,
                                                     const int* ncols_dev, int ld, int max_sweeps,
                                                     int* error) {
  __shared__ int pp[kJacobiMaxPairs], qq[kJacobiMaxPairs];
  __shared__ double jc[kJacobiMaxPairs], js[kJacobiMaxPairs];
  __shared__ double2 je[kJacobiMaxPairs];
  __shared__ int any_rot;
  __shared__ double s_scale;
  const int b = blockIdx.x;
  const int n = ncols_dev[b];
  double2* a = a_all + (size_t)b * stride;
  double2* v = v_all + (size_t)b * stride;
  const int tid = threadIdx.x, nt = blockDim.x;
  for (int e = tid; e < n * n; e += nt) {
    int i = e / n, j = e % n;
    v[(size_t)i * ld + j] = make_double2(i == j ? 1.0 : 0.0, 0.0);
  }
  if (tid == 0) {
    double tr = 0.0;
    for (int i = 0; i < n; ++i) tr += fabs(a[(size_t)i * ld + i].x);
    s_scale = tr;
  }
  __syncthreads();
  if (n < 2) return;
  const int np = n / 2;
  const double abs_tol = kJacobiAbsTol * s_scale + 1e-300;
  bool converged = false;
  for (int sweep = 0; sweep < max_sweeps; ++sweep) {
    __syncthreads();
    if (tid == 0) any_rot = 0;
    __syncthreads();
    for (int r = 0; r < n - 1; ++r) {
      if (tid < np) {
        int m = tid;
        int p = (m == 0) ? n - 1 : (r + m) % (n - 1);
        int q = (r + n - 1 - m) % (n - 1);
        if (m == 0) q = r % (n - 1);
        if (p > q) { int t = p; p = q; q = t; }
        double al = a[(size_t)p * ld + p].x, be = a[(size_t)q * ld + q].x;
        double2 g = a[(size_t)p * ld + q];
        double ag = cabs_(g);
        double c = 1.0, s = 0.0;
        double2 em = make_double2(1.0, 0.0);
        if (ag > abs_tol && ag > 1e-15 * sqrt(fabs(al * be))) {
          double tau = (be - al) / (2.0 * ag);
          double t = (tau >= 0 ? 1.0 : -1.0) / (fabs(tau) + sqrt(1.0 + tau * tau));
          c = 1.0 / sqrt(1.0 + t * t);
          s = t * c;
          em = make_double2(g.x / ag, -g.y / ag);   // e^{-i phi}
          any_rot = 1;
        }
        pp[m] = p; qq[m] = q; jc[m] = c; js[m] = s; je[m] = em;
      }
      __syncthreads();
      for (int e = tid; e < np * np; e += nt) {
        int P = e / np, Q = e % np;
        int p0 = pp[P], p1 = qq[P], q0 = pp[Q], q1 = qq[Q];
        // J = [[c, s], [-s em, c em]]
        double2 J00 = make_double2(jc[Q], 0.0), J01 = make_double2(js[Q], 0.0);
        double2 J10 = cscale(je[Q], -js[Q]), J11 = cscale(je[Q], jc[Q]);
        double2 K00 = make_double2(jc[P], 0.0), K01 = make_double2(js[P], 0.0);
        double2 K10 = cscale(je[P], -js[P]), K11 = cscale(je[P], jc[P]);
        double2 a00 = a[(size_t)p0 * ld + q0], a01 = a[(size_t)p0 * ld + q1];
        double2 a10 = a[(size_t)p1 * ld + q0], a11 = a[(size_t)p1 * ld + q1];
        double2 b00 = cadd(cmul(a00, J00), cmul(a01, J10));
        double2 b01 = cadd(cmul(a00, J01), cmul(a01, J11));
        double2 b10 = cadd(cmul(a10, J00), cmul(a11, J10));
        double2 b11 = cadd(cmul(a10, J01), cmul(a11, J11));
        double2 c00 = cadd(cmulc(K00, b00), cmulc(K10, b10));
        double2 c01 = cadd(cmulc(K00, b01), cmulc(K10, b11));
        double2 c10 = cadd(cmulc(K01, b00), cmulc(K11, b10));
        double2 c11 = cadd(cmulc(K01, b01), cmulc(K11, b11));
        if (P == Q) {
          c00.y = 0.0; c11.y = 0.0;
          c01 = cz(); c10 = cz();
        }
        a[(size_t)p0 * ld + q0] = c00; a[(size_t)p0 * ld + q1] = c01;
        a[(size_t)p1 * ld + q0] = c10; a[(size_t)p1 * ld + q1] = c11;
      }
      for (int e = tid; e < n * np; e += nt) {
        int i = e / np, Q = e % np;
        int q0 = pp[Q], q1 = qq[Q];
        double2 J00 = make_double2(jc[Q], 0.0), J01 = make_double2(js[Q], 0.0);
        double2 J10 = cscale(je[Q], -js[Q]), J11 = cscale(je[Q], jc[Q]);
        double2 x = v[(size_t)i * ld + q0], y = v[(size_t)i * ld + q1];
        v[(size_t)i * ld + q0] = cadd(cmul(x, J00), cmul(y, J10));
        v[(size_t)i * ld + q1] = cadd(cmul(x, J01), cmul(y, J11));
      }
      __syncthreads();
    }
    __syncthreads();
    if (!any_rot) { converged = true; break; }
  }
  if (!converged && tid == 0 && error) atomicOr(error, kErrEigNoConv);
}

// ------------------------------------------------ LDS-resident Jacobi -------
// QMX_OPT_TWO_SIDED_JACOBI and cutoffs near rounding (the one-sided solver below
// is the default).
// For n <= kJacobiLdsMax the upper triangle of A (n (n + 1) / 2 complex128,
// 132 KiB at n = 128) lives in LDS for a whole sweep: one block per state,
// the same parallel (circle) ordering and rotations as jacobi_kernel.  Each
// sweep logs its rotations (c, s, e^{-i phi} per pair and round); a second
// kernel applies the log to the rows of V, 16 rows per block held in LDS.
// The host launches sweep / update pairs; a state none of whose off-diagonal
// entries passes the rotation test at the start of a sweep is converged (that
// sweep would rotate nothing and is not run), as is one whose sweep rotated
// nothing, and every later launch returns at once for it.
// One round of n = 128 takes 2.8 us, most of it the FP64 and address
// instructions of 2016 blocks on one CU's four SIMDs (3.3 us with the diagonal
// blocks as a third pass over the threads and addresses formed per access); the
// rows' kernel, bound by its rounds' LDS round trips, 40 us a sweep with a wave
// per row (72 with a barrier per round).  Every product keeps the operands and
// order that fix its rounding.
constexpr int kJacobiLdsMax = 128;
constexpr int kJacobiRowsPerBlock = 16;

QMX_DEV int tri_index(int i, int j, int n) { return i * (2 * n - i + 1) / 2 + (j - i); }

// kAll: V (n x n) is in LDS too and takes the rotations of a round with A, all
// sweeps run in one launch (sweep = their limit; no log, no state).  The host
// takes it up to kJacobiAllMax columns, where two launches per sweep, most of
// them after the last one, cost more than the one CU that V then has (the chain
// of one N = 15 state: 3.6 ms against 4.8 at 32 columns, 6.1 against 6.7 at 48,
// 7.5 both at 56, 9.0 against 8.1 at 64).
constexpr int kJacobiAllMax = 48;
template <bool kAll>
__global__ __launch_bounds__(1024) void jacobi_lds_sweep_kernel(double2* a_all, double2* v_all, size_t stride,
                                                                const int* ncols_dev, int ld,
                                                                double4* log_all, size_t log_stride,
                                                                int* state, int sweep, int* error) {
  extern __shared__ double2 tri[];
  __shared__ int4 pq[kJacobiLdsMax / 2];             // p, q and their rows' places
  __shared__ double2 jcs[kJacobiLdsMax / 2], je[kJacobiLdsMax / 2];
  __shared__ int any_rot;
  __shared__ double s_scale;
  const int b = blockIdx.x;
  // state[b]: 0 = running, 1 = converged; state[batch + b] = sweeps run
  if (!kAll && state[b]) return;
  const int n = ncols_dev[b];
  double2* a = a_all + (size_t)b * stride;
  double2* v = v_all + (size_t)b * stride;
  if (n < 2) {
    if (threadIdx.x == 0) {
      if (kAll && n == 1) v[0] = make_double2(1.0, 0.0);
      if (!kAll) state[b] = 1;
    }
    return;
  }
  double4* lg = log_all + (size_t)b * log_stride;
  double2* vl = tri + ld * (ld + 1) / 2;
  const int tid = threadIdx.x, nt = blockDim.x;
  const int lane = tid & 63, wave = tid >> 6, waves = nt >> 6;
  // entry (i, j) of the triangle is at rowbase(i) + j; a wave per row
  auto rowbase = [&](int i) { return i * (2 * n - i + 1) / 2 - i; };
  for (int i = wave; i < n; i += waves)
    for (int j = i + lane; j < n; j += 64) tri[rowbase(i) + j] = a[(size_t)i * ld + j];
  if constexpr (kAll)
    for (int e = tid; e < n * n; e += nt) vl[e] = make_double2(e / n == e % n ? 1.0 : 0.0, 0.0);
  const int np = n / 2;
  // this thread's pair blocks (P, Q), P < Q, row-major over the strict upper
  // triangle of pair blocks; the same in every round (the kernel is launched
  // with 1024 threads: two blocks each cover the 2016 of n = 128).  The diagonal
  // blocks belong to the threads that find their rotations.
  constexpr int kBlkPer = (kJacobiLdsMax / 2 * (kJacobiLdsMax / 2 - 1) / 2 + 1023) / 1024;
  const int nblocks = np * (np - 1) / 2;
  int bP[kBlkPer], bQ[kBlkPer];
#pragma unroll
  for (int k = 0; k < kBlkPer; ++k) {
    const int e = tid + k * nt;
    // block (P, Q) of the strict triangle of np: entry (P, Q - 1) of the triangle of np - 1
    const int m = np - 1;
    int P = 0, Q = 0;
    if (e < nblocks) {
      P = (int)((2.0 * m + 1.0 - sqrt((2.0 * m + 1.0) * (2.0 * m + 1.0) - 8.0 * e)) * 0.5);
      while (P > 0 && tri_index(P, P, m) > e) --P;
      while (P + 1 < m && tri_index(P + 1, P + 1, m) <= e) ++P;
      Q = P + (e - tri_index(P, P, m)) + 1;
    }
    bP[k] = P;
    bQ[k] = Q;
  }
  bool converged = false, ran = false;
  for (int s = 0; s < (kAll ? sweep : 1); ++s) {
    __syncthreads();
    if (tid == 0) {
      any_rot = 0;
      double tr = 0.0;
#pragma unroll 16
      for (int i = 0; i < n; ++i) tr += fabs(tri[rowbase(i) + i].x);
      s_scale = tr;
    }
    __syncthreads();
    const double abs_tol = kJacobiAbsTol * s_scale + 1e-300;
    // a sweep would rotate nothing iff no off-diagonal entry passes the rotation
    // test now: then the state is converged and the sweep is not run
    for (int i = wave; i < n; i += waves) {
      const double al = tri[rowbase(i) + i].x;
      for (int j = i + 1 + lane; j < n; j += 64) {
        const double ag = cabs_(tri[rowbase(i) + j]);
        if (ag > abs_tol && ag > 1e-15 * sqrt(fabs(al * tri[rowbase(j) + j].x))) any_rot = 1;
      }
    }
    __syncthreads();
    const bool go = any_rot;
    __syncthreads();
    if (!go) {
      converged = true;
      break;
    }
    if (tid == 0) any_rot = 0;
    ran = true;
    __syncthreads();
    for (int r = 0; r < n - 1; ++r) {
      double c = 1.0, sn = 0.0;
      double2 em = make_double2(1.0, 0.0), g = cz(), app = cz(), aqq = cz();
      int ipp = 0, ipq = 0, iqq = 0;
      if (tid < np) {
        const int m = tid;
        int p = (m == 0) ? n - 1 : (r + m) % (n - 1);
        int q = (r + n - 1 - m) % (n - 1);
        if (m == 0) q = r % (n - 1);
        if (p > q) { int t = p; p = q; q = t; }
        const int bp = rowbase(p), bq = rowbase(q);
        ipp = bp + p;
        ipq = bp + q;
        iqq = bq + q;
        app = tri[ipp];
        aqq = tri[iqq];
        g = tri[ipq];
        const double al = app.x, be = aqq.x;
        const double ag = cabs_(g);
        // one comparison against the larger threshold: the diagonal reads are
        // issued together with the off-diagonal one
        if (ag > fmax(abs_tol, 1e-15 * sqrt(fabs(al * be)))) {
          const double tau = (be - al) / (2.0 * ag);
          const double t = (tau >= 0 ? 1.0 : -1.0) / (fabs(tau) + sqrt(1.0 + tau * tau));
          c = 1.0 / sqrt(1.0 + t * t);
          sn = t * c;
          em = make_double2(g.x / ag, -g.y / ag);   // e^{-i phi}
          any_rot = 1;
        }
        pq[m] = make_int4(p, q, bp, bq);
        jcs[m] = make_double2(c, sn);
        je[m] = em;
        if constexpr (!kAll) lg[(size_t)r * np + m] = make_double4(c, sn, em.x, em.y);
      }
      __syncthreads();
      // blocks (P, Q), P <= Q: B' = J_P^H B J_Q with B = A[{p0, p1}][{q0, q1}];
      // (Q, P) is its conjugate transpose and is never stored separately
      auto turn = [](double2 a00, double2 a01, double2 a10, double2 a11, double2 kcs, double2 ke, double2 qcs,
                     double2 qe, double2& c00, double2& c01, double2& c10, double2& c11) {
        const double2 J00 = make_double2(qcs.x, 0.0), J01 = make_double2(qcs.y, 0.0);
        const double2 J10 = cscale(qe, -qcs.y), J11 = cscale(qe, qcs.x);
        const double2 K00 = make_double2(kcs.x, 0.0), K01 = make_double2(kcs.y, 0.0);
        const double2 K10 = cscale(ke, -kcs.y), K11 = cscale(ke, kcs.x);
        const double2 b00 = cadd(cmul(a00, J00), cmul(a01, J10));
        const double2 b01 = cadd(cmul(a00, J01), cmul(a01, J11));
        const double2 b10 = cadd(cmul(a10, J00), cmul(a11, J10));
        const double2 b11 = cadd(cmul(a10, J01), cmul(a11, J11));
        c00 = cadd(cmulc(K00, b00), cmulc(K10, b10));
        c01 = cadd(cmulc(K00, b01), cmulc(K10, b11));
        c10 = cadd(cmulc(K01, b00), cmulc(K11, b10));
        c11 = cadd(cmulc(K01, b01), cmulc(K11, b11));
      };
      if (tid < np) {
        double2 c00, c01, c10, c11;
        // (the diagonal's zero imaginary parts come from memory, so that the
        // compiler cannot fold them and round these blocks otherwise)
        turn(app, g, cconj(g), aqq, make_double2(c, sn), em, make_double2(c, sn), em, c00, c01, c10, c11);
        tri[ipp] = make_double2(c00.x, 0.0);
        tri[ipq] = cz();
        tri[iqq] = make_double2(c11.x, 0.0);
      }
#pragma unroll
      for (int k = 0; k < kBlkPer; ++k) {
        if (tid + k * nt >= nblocks) break;
        const int P = bP[k], Q = bQ[k];
        const int4 u = pq[P], w = pq[Q];
        // one LDS access per entry: (i, j) with i > j is the conjugate of (j, i)
        auto at = [&](int i, int bi, int j, int bj) { return i > j ? bj + i : bi + j; };
        const int i00 = at(u.x, u.z, w.x, w.z), i01 = at(u.x, u.z, w.y, w.w);
        const int i10 = at(u.y, u.w, w.x, w.z), i11 = at(u.y, u.w, w.y, w.w);
        auto flip = [](double2 v, bool lo) { return make_double2(v.x, lo ? -v.y : v.y); };
        const double2 a00 = flip(tri[i00], u.x > w.x), a01 = flip(tri[i01], u.x > w.y);
        const double2 a10 = flip(tri[i10], u.y > w.x), a11 = flip(tri[i11], u.y > w.y);
        double2 c00, c01, c10, c11;
        turn(a00, a01, a10, a11, jcs[P], je[P], jcs[Q], je[Q], c00, c01, c10, c11);
        tri[i00] = flip(c00, u.x > w.x);
        tri[i01] = flip(c01, u.x > w.y);
        tri[i10] = flip(c10, u.y > w.x);
        tri[i11] = flip(c11, u.y > w.y);
      }
      if constexpr (kAll) {
        // V <- V J, a wave per row and a lane per pair
        if (lane < np) {
          const int4 u = pq[lane];
          const double2 cs = jcs[lane], em = je[lane];
          const double2 J00 = make_double2(cs.x, 0.0), J01 = make_double2(cs.y, 0.0);
          const double2 J10 = cscale(em, -cs.y), J11 = cscale(em, cs.x);
          for (int i = wave; i < n; i += waves) {
            const double2 x = vl[i * n + u.x], y = vl[i * n + u.y];
            vl[i * n + u.x] = cadd(cmul(x, J00), cmul(y, J10));
            vl[i * n + u.y] = cadd(cmul(x, J01), cmul(y, J11));
          }
        }
      }
      __syncthreads();
    }
    if (!any_rot) {   // a sweep that rotated nothing leaves the log at identity
      converged = true;
      break;
    }
  }
  if constexpr (kAll) {
    __syncthreads();
    for (int e = tid; e < n * n; e += nt) v[(size_t)(e / n) * ld + e % n] = vl[e];
    for (int i = tid; i < n; i += nt) a[(size_t)i * ld + i] = tri[rowbase(i) + i];
    if (tid == 0 && !converged && error) atomicOr(error, kErrEigNoConv);
  } else {
    // (a sweep that was not run has neither changed A nor a log)
    if (tid == 0 && converged) state[b] = 1;
    if (!ran) return;
    // write the triangle back (the lower part stays stale: readers use i <= j)
    for (int i = wave; i < n; i += waves)
      for (int j = i + lane; j < n; j += 64) a[(size_t)i * ld + j] = tri[rowbase(i) + j];
    if (tid == 0) state[gridDim.x + b] = sweep + 1;
  }
}

// V <- V J over one sweep's log; rows [16 blockIdx.x, +16) of state blockIdx.y
__global__ __launch_bounds__(1024) void jacobi_lds_rows_kernel(double2* v_all, size_t stride,
                                                               const int* ncols_dev, int ld,
                                                               const double4* log_all, size_t log_stride,
                                                               const int* state, int sweep) {
  __shared__ double2 rows[kJacobiRowsPerBlock][kJacobiLdsMax];
  const int b = blockIdx.y;
  // the sweep ran for this state iff its sweep counter reached sweep + 1
  if (state[gridDim.y + b] != sweep + 1) return;
  const int n = ncols_dev[b];
  const int r0 = blockIdx.x * kJacobiRowsPerBlock;
  // a wave per row, a lane per pair: the rows need no barrier between rounds
  const int i = threadIdx.x >> 6, m = threadIdx.x & 63;
  if (n < 2 || r0 + i >= n) return;
  double2* v = v_all + (size_t)b * stride + (size_t)(r0 + i) * ld;
  const int np = n / 2;
  const double4* lg = log_all + (size_t)b * log_stride + m;
  double2* row = rows[i];
  for (int e = m; e < n; e += 64) row[e] = v[e];
  __builtin_amdgcn_wave_barrier();
  // the log is read kAhead rounds before its use
  constexpr int kAhead = 4;
  double4 R[kAhead];
#pragma unroll
  for (int k = 0; k < kAhead; ++k)
    if (m < np && k < n - 1) R[k] = lg[(size_t)k * np];
  auto round = [&](int r, double4& Rr) {
    if (m >= np) return;
    const double4 w = Rr;
    if (r + kAhead < n - 1) Rr = lg[(size_t)(r + kAhead) * np];
    // p = (r + m) % (n - 1), q = (r - m) % (n - 1); pair 0 is (n - 1, r)
    int p = r + m, q = r - m;
    p = m == 0 ? n - 1 : (p >= n - 1 ? p - (n - 1) : p);
    q = q < 0 ? q + n - 1 : q;
    if (p > q) { const int t = p; p = q; q = t; }
    const double2 em = make_double2(w.z, w.w);
    const double2 J00 = make_double2(w.x, 0.0), J01 = make_double2(w.y, 0.0);
    const double2 J10 = cscale(em, -w.y), J11 = cscale(em, w.x);
    const double2 x = row[p], y = row[q];
    row[p] = cadd(cmul(x, J00), cmul(y, J10));
    row[q] = cadd(cmul(x, J01), cmul(y, J11));
  };
  int r = 0;
  for (; r + kAhead <= n - 1; r += kAhead) {
#pragma unroll
    for (int k = 0; k < kAhead; ++k) {
      round(r + k, R[k]);
      __builtin_amdgcn_wave_barrier();
    }
  }
#pragma unroll
  for (int k = 0; k < kAhead; ++k) {
    if (r + k < n - 1) round(r + k, R[k]);
    __builtin_amdgcn_wave_barrier();
  }
  for (int e = m; e < n; e += 64) v[e] = row[e];
}

__global__ void jacobi_lds_init_kernel(double2* v_all, size_t stride, const int* ncols_dev, int ld, int* state,
                                       int batch) {
  const int b = blockIdx.y;
  const int n = ncols_dev[b];
  double2* v = v_all + (size_t)b * stride;
  for (int e = blockIdx.x * blockDim.x + threadIdx.x; e < n * n; e += gridDim.x * blockDim.x) {
    const int i = e / n, j = e % n;
    v[(size_t)i * ld + j] = make_double2(i == j ? 1.0 : 0.0, 0.0);
  }
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    state[b] = 0;
    state[batch + b] = 0;
  }
}

__global__ void jacobi_lds_check_kernel(const int* state, int batch, int* error) {
  const int b = blockIdx.x * blockDim.x + threadIdx.x;
  if (b < batch && !state[b] && error) atomicOr(error, kErrEigNoConv);
}

// ------------------------------------ one-sided Jacobi on L -----------------
// Eigensolver of the chain: one-sided Jacobi on the pivoted Cholesky factor of
// the Gram matrix.
//
//   A = L L^H       pivoted Cholesky (largest remaining diagonal first), cut at
//                   eps * trace: L has as many columns as A has rank
//   L J = U S       one-sided Jacobi on L's columns (K. Veselic, V. Hari, "A
//                   note on a one-sided Jacobi algorithm", Numer. Math. 56
//                   (1989)): plane rotations from the right until every two
//                   columns are orthogonal to kOsjTol of their norms
// The columns of U = (L J) S^{-1} are A's eigenvectors and the squared column
// norms its eigenvalues; nothing has to be accumulated beside the columns
// themselves.  The factor of a pivoted Cholesky is graded, which is what makes
// the rotations converge (8 to 10 sweeps on the chain's matrices, the last of
// them only checking), and the columns that a rank-deficient Gram matrix does
// not have (fewer rows than columns left of the chain's centre) are never
// touched.  Columns dropped at eps * trace get eigenvalue 0 and a zero vector:
// the caller takes this solver where its cutoff drops them too, and the identity
// in the place of the vectors of a matrix that is not truncated.
constexpr double kEps = 2.220446049250313e-16;
// columns p, q are orthogonal when |p^H q| <= kOsjTol |p| |q|: the rounding of
// a 128-term product is about sqrt(128) eps
constexpr double kOsjTol = 2e-15;

// NR entries of one column: rows lane, lane + 64, ...
template <int NR> struct Col { double2 v[NR]; };

template <int NR> QMX_DEV double col_norm(const Col<NR>& a) {
  double s = 0.0;
#pragma unroll
  for (int r = 0; r < NR; ++r) s += cabs2(a.v[r]);
  return s;
}
template <int NR> QMX_DEV double2 col_dot(const Col<NR>& a, const Col<NR>& b) {
  double2 s = cz();
#pragma unroll
  for (int r = 0; r < NR; ++r) s = cfmac(a.v[r], b.v[r], s);
  return s;
}

// the total over each quad of lanes, on all of them
QMX_DEV double sum4(double v) {
  v += dpp<kDppSwap>(v);
  return v + dpp<kDppCol2>(v);
}

// Rotates the four disjoint pairs (p_k, q_k) to orthogonality.  al, be: squared
// norms of p_k and q_k in row k of the wave, updated.  With g = p^H q and
// d = |q|^2 - |p|^2 the smaller root of t^2 + t d / |g| - 1 = 0 gives
//   t e^{i arg g} = te = 2 g sign(d) / (|d| + sqrt(d^2 + 4 |g|^2)),
//   p' = c (p - conj(te) q),  q' = c (q + te p),  c = 1 / sqrt(1 + |te|^2),
//   |p'|^2 = |p|^2 - t |g|,  |q'|^2 = |q|^2 + t |g|.
// The four pairs' parameters are computed once, one pair per row, and read back
// as scalars.  Returns whether any pair was rotated (uniform over the wave).
struct Rotation { double2 te; double c; };
// (al, be, g: a pair per row of lanes; whether it is rotated in the result)
QMX_DEV bool rotation(double2 g, double& al, double& be, double tol, Rotation& t) {
  const double ag2 = cabs2(g);
  const bool rot = ag2 > tol * tol * al * be && ag2 > 0.0;
  const double d = be - al;
  const double q = fma(4.0, ag2, d * d);
  double f = 2.0 * rcp_newton(fma(q, rsqrt_newton(q), fabs(d)));
  f = rot ? (d >= 0.0 ? f : -f) : 0.0;
  t.te = rot ? cscale(g, f) : cz();
  t.c = rsqrt_newton(1.0 + cabs2(t.te));
  const double tg = rot ? ag2 * f : 0.0;
  al -= tg;
  be += tg;
  return rot;
}
// pair k's rotation, from row k of the wave
template <int NR> QMX_DEV void rotate_pair(Col<NR>& p, Col<NR>& q, const Rotation& t, int k) {
  const double tx = lane_value(t.te.x, 16 * k), ty = lane_value(t.te.y, 16 * k), cc = lane_value(t.c, 16 * k);
#pragma unroll
  for (int r = 0; r < NR; ++r) {
    const double2 u = p.v[r], w = q.v[r];
    p.v[r] = make_double2(cc * fma(-tx, w.x, fma(-ty, w.y, u.x)), cc * fma(-tx, w.y, fma(ty, w.x, u.y)));
    q.v[r] = make_double2(cc * fma(tx, u.x, fma(-ty, u.y, w.x)), cc * fma(tx, u.y, fma(ty, u.x, w.y)));
  }
}
template <int NR>
QMX_DEV double2 dots4(const Col<NR>& p0, const Col<NR>& q0, const Col<NR>& p1, const Col<NR>& q1, const Col<NR>& p2,
                      const Col<NR>& q2, const Col<NR>& p3, const Col<NR>& q3) {
  const double2 g0 = col_dot(p0, q0), g1 = col_dot(p1, q1), g2 = col_dot(p2, q2), g3 = col_dot(p3, q3);
  return make_double2(rows_total(g0.x, g1.x, g2.x, g3.x), rows_total(g0.y, g1.y, g2.y, g3.y));
}
template <int NR>
QMX_DEV double norms4(const Col<NR>& p0, const Col<NR>& p1, const Col<NR>& p2, const Col<NR>& p3) {
  return rows_total(col_norm(p0), col_norm(p1), col_norm(p2), col_norm(p3));
}
// (total: sums a value per row of lanes over the waves that share the columns)
template <int NR, typename F>
QMX_DEV bool rotate4(Col<NR>& p0, Col<NR>& q0, Col<NR>& p1, Col<NR>& q1, Col<NR>& p2, Col<NR>& q2, Col<NR>& p3,
                     Col<NR>& q3, double& al, double& be, double tol, F total) {
  const double2 g = total(dots4(p0, q0, p1, q1, p2, q2, p3, q3));
  if (!__any(cabs2(g) > tol * tol * al * be)) return false;
  Rotation t;
  rotation(g, al, be, tol, t);
  rotate_pair(p0, q0, t, 0);
  rotate_pair(p1, q1, t, 1);
  rotate_pair(p2, q2, t, 2);
  rotate_pair(p3, q3, t, 3);
  return true;
}

// ------------------------------------------------ up to 128 columns ---------
// One block per state, the matrix in registers: wave w holds two blocks of 4
// columns, lane l their rows l (and l + 64).  The blocks are paired by the
// circle method: nb - 1 rounds of 4 sets of 4 disjoint pairs per sweep, after
// which every wave passes its blocks on through LDS; at the start of a sweep
// the pairs inside the blocks are rotated and the norms recomputed.
// Bound by FP64 issue (per set and wave about 250 instructions, half of them
// the 12 NR + 4 NR per pair that the rotations and products need) with 3 to 4
// waves per SIMD, one CU per state.  The truncation chain of 32 states (N=20,
// chi = 64: ten matrices of 128 columns and rank 96 to 8) spends 13.2 ms here
// and 1.3 ms in the Cholesky factors; the two-sided Jacobi it replaces, which
// kept A's triangle in LDS and logged its rotations for a second kernel that
// accumulated V, spent 62.7 + 16.1 ms (up to 17 sweeps per matrix).
constexpr int kOsjMax = 128;

// Pivoted Cholesky factor of one state's Gram matrix (n <= 128): thread (row,
// g) holds columns 16 g .. 16 g + 15 of its row in registers, and every step
// subtracts the outer product of the new column.  Column k of L goes to
// a + k ld (A's own storage), L's column count to rank[b]; -1 for a matrix that
// is zero, not finite, or not truncated at all (n <= keep_all), which stays as
// it is.  Bound by the two barriers and the pivot search per step.
__global__ __launch_bounds__(1024) void chol_kernel(double2* a_all, size_t stride, const int* ncols_dev, int ld,
                                                    int keep_all, int* rank_out) {
  __shared__ double2 lcol[kOsjMax];
  __shared__ int s_p;
  __shared__ double s_d;
  const int b = blockIdx.x;
  const int n = ncols_dev[b];
  double2* a = a_all + (size_t)b * stride;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int row = tid & (kOsjMax - 1), g = wave >> 1;
  if (n <= keep_all) {
    if (tid == 0) rank_out[b] = -1;
    return;
  }
  // a column of the Hermitian matrix is its conjugated row: contiguous loads
  double2 x[16];
#pragma unroll
  for (int c = 0; c < 16; ++c) {
    const int col = 16 * g + c;
    x[c] = col < n && row < n ? cconj(a[(size_t)col * ld + row]) : cz();
  }
  // wave 0: the remaining diagonal of columns lane, lane + 64
  double d0 = lane < n ? a[(size_t)lane * ld + lane].x : 0.0;
  double d1 = lane + 64 < n ? a[(size_t)(lane + 64) * ld + lane + 64].x : 0.0;
  const double tr = wave_sum(d0 + d1);
  if (!(tr > 0.0) || !(tr < 1e300)) {
    if (tid == 0) rank_out[b] = -1;
    return;
  }
  if (lane >= n) d0 = -1.0;
  if (lane + 64 >= n) d1 = -1.0;
  __syncthreads();   // A is in registers: its storage takes L
  unsigned done = 0;
  bool used = false;
  int rank = 0;
  for (; rank < n; ++rank) {
    if (wave == 0) {
      // largest remaining diagonal entry, lowest index on ties
      double best = d1 > d0 ? d1 : d0;
      int p = d1 > d0 ? lane + 64 : lane;
#pragma unroll
      for (int m = 1; m < 64; m <<= 1) {
        const double o = __shfl_xor(best, m, 64);
        const int op = __shfl_xor(p, m, 64);
        if (o > best || (o == best && op < p)) {
          best = o;
          p = op;
        }
      }
      if (lane == 0) {
        s_p = best > kEps * tr ? p : -1;
        s_d = best;
      }
    }
    __syncthreads();
    const int p = __builtin_amdgcn_readfirstlane(s_p);
    if (p < 0) break;
    if (g == (p >> 4)) {
      double2 t = cz();
#pragma unroll
      for (int c = 0; c < 16; ++c)
        if (c == (p & 15)) t = x[c];
      const double d = s_d, inv = rsqrt_newton(d);
      t = used ? cz() : (row == p ? make_double2(d * inv, 0.0) : cscale(t, inv));
      lcol[row] = t;
      if (row < n) a[(size_t)rank * ld + row] = t;
      done |= 1u << (p & 15);
    }
    __syncthreads();
    const double2 l = lcol[row];
    if (row == p) used = true;
#pragma unroll
    for (int c = 0; c < 16; ++c)
      if (!((done >> c) & 1u)) {
        const double2 lc = lcol[16 * g + c];   // x -= l conj(l_c)
        x[c].x = fma(-l.x, lc.x, fma(-l.y, lc.y, x[c].x));
        x[c].y = fma(-l.y, lc.x, fma(l.x, lc.y, x[c].y));
      }
    if (wave == 0) {
      d0 = lane == p ? -1.0 : d0 - cabs2(lcol[lane]);
      d1 = lane + 64 == p ? -1.0 : d1 - cabs2(lcol[lane + 64]);
    }
  }
  if (tid == 0) rank_out[b] = rank;
}

template <int NR>
__global__ __launch_bounds__(NR == 2 ? 1024 : 512) void osj_kernel(double2* a_all, double2* v_all, size_t stride,
                                                                   const int* ncols_dev, int ld,
                                                                   const int* rank_in, int max_sweeps, int* error) {
  constexpr int kRows = 64 * NR;
  extern __shared__ double2 xbuf[];                   // W + 1 slots of 4 columns
  __shared__ double nbuf[17][4];
  const int b = blockIdx.x;
  const int n = ncols_dev[b], rank = rank_in[b];
  double2* a = a_all + (size_t)b * stride;
  double2* v = v_all + (size_t)b * stride;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  if (rank < 0) {   // any unitary basis will do; the diagonal stays as it is
    for (int e = tid; e < n * n; e += blockDim.x) {
      const int i = e / n, j = e % n;
      v[(size_t)i * ld + j] = make_double2(i == j ? 1.0 : 0.0, 0.0);
    }
    return;
  }
  Col<NR> x[8];
  const int nb = ((rank + 3) / 4 + 1) & ~1;   // blocks of 4, an even number
  const int m = nb / 2;                       // waves with columns
  const int tb = 4 * wave, bb = 4 * (nb - 1 - wave);   // first columns of this wave's blocks
  const bool live = wave < m;
#pragma unroll
  for (int c = 0; c < 8; ++c)
#pragma unroll
    for (int r = 0; r < NR; ++r) {
      const int k = c < 4 ? tb + c : bb + c - 4, row = lane + 64 * r;
      x[c].v[r] = live && k < rank && row < n ? a[(size_t)k * ld + row] : cz();
    }
  __syncthreads();   // L is in registers: A's storage takes the eigenvalues
  // ---- one-sided Jacobi sweeps: x[0..3] the top block, x[4..7] the bottom one
  auto slot = [&](int s) { return xbuf + (size_t)s * 4 * kRows; };
  auto put = [&](int s, int c0, double nrm) {
    double2* t = slot(s);
#pragma unroll
    for (int c = 0; c < 4; ++c)
#pragma unroll
      for (int r = 0; r < NR; ++r) t[c * kRows + lane + 64 * r] = c0 ? x[4 + c].v[r] : x[c].v[r];
    if ((lane & 15) == 0) nbuf[s][lane >> 4] = nrm;
  };
  auto get = [&](int s, int c0, double& nrm) {
    const double2* t = slot(s);
#pragma unroll
    for (int c = 0; c < 4; ++c)
#pragma unroll
      for (int r = 0; r < NR; ++r) {
        const double2 w = t[c * kRows + lane + 64 * r];
        if (c0) x[4 + c].v[r] = w;
        else x[c].v[r] = w;
      }
    nrm = nbuf[s][lane >> 4];
  };
  bool converged = false;
  auto own = [](double2 g) { return g; };   // a column is one wave's
  for (int sweep = 0; sweep < max_sweeps; ++sweep) {
    bool rot = false;
    double nt = 0.0, nq = 0.0;   // squared norms: row k of the wave, column k of the top / bottom block
    if (live) {
      auto inside = [&](Col<NR>& p0, Col<NR>& q0, Col<NR>& p1, Col<NR>& q1, Col<NR>& p2, Col<NR>& q2, Col<NR>& p3,
                        Col<NR>& q3) {
        double al = rows_total(col_norm(p0), col_norm(p1), col_norm(p2), col_norm(p3));
        double be = rows_total(col_norm(q0), col_norm(q1), col_norm(q2), col_norm(q3));
        rot |= rotate4(p0, q0, p1, q1, p2, q2, p3, q3, al, be, kOsjTol, own);
      };
      inside(x[0], x[1], x[2], x[3], x[4], x[5], x[6], x[7]);
      inside(x[0], x[2], x[1], x[3], x[4], x[6], x[5], x[7]);
      inside(x[0], x[3], x[1], x[2], x[4], x[7], x[5], x[6]);
      nt = rows_total(col_norm(x[0]), col_norm(x[1]), col_norm(x[2]), col_norm(x[3]));
      nq = rows_total(col_norm(x[4]), col_norm(x[5]), col_norm(x[6]), col_norm(x[7]));
    }
    for (int round = 0; round < nb - 1; ++round) {
      if (live) {
        // set s: pairs (top k, bottom (k + s) % 4); the bottom norms move up one row per set
        auto next = [&]() { nq = __shfl(nq, (lane + 16) & 63, 64); };
        rot |= rotate4(x[0], x[4], x[1], x[5], x[2], x[6], x[3], x[7], nt, nq, kOsjTol, own);
        next();
        rot |= rotate4(x[0], x[5], x[1], x[6], x[2], x[7], x[3], x[4], nt, nq, kOsjTol, own);
        next();
        rot |= rotate4(x[0], x[6], x[1], x[7], x[2], x[4], x[3], x[5], nt, nq, kOsjTol, own);
        next();
        rot |= rotate4(x[0], x[7], x[1], x[4], x[2], x[5], x[3], x[6], nt, nq, kOsjTol, own);
        next();
      }
      if (m == 1) continue;   // two blocks: the only pair
      // circle: top 0 stays, top w goes to top w + 1, the last top to the last
      // bottom, bottom w to bottom w - 1, bottom 0 to top 1.  Tops first, then
      // bottoms; the last top waits in its slot, so the last bottom uses slot m.
      if (live && wave > 0) put(wave, 0, nt);
      __syncthreads();
      if (live && wave > 1) get(wave - 1, 0, nt);
      __syncthreads();
      if (live) put(wave == m - 1 ? m : wave, 1, nq);
      __syncthreads();
      if (live) {
        if (wave == 1) get(0, 0, nt);
        get(wave == m - 1 ? m - 1 : (wave + 1 == m - 1 ? m : wave + 1), 1, nq);
      }
      __syncthreads();
    }
    if (!__syncthreads_or(rot ? 1 : 0)) {
      converged = true;
      break;
    }
  }
  if (!converged && tid == 0 && error) atomicOr(error, kErrEigNoConv);
  // eigenvalues to A's diagonal, eigenvectors to V; the dropped columns are zero
  const double nt = rows_total(col_norm(x[0]), col_norm(x[1]), col_norm(x[2]), col_norm(x[3]));
  const double nq = rows_total(col_norm(x[4]), col_norm(x[5]), col_norm(x[6]), col_norm(x[7]));
  if (live) {
#pragma unroll
    for (int c = 0; c < 8; ++c) {
      const int k = c < 4 ? tb + c : bb + c - 4;
      const double nn = lane_value(c < 4 ? nt : nq, 16 * (c & 3));
      const double inv = nn > 0.0 ? rsqrt_newton(nn) : 0.0;
      if (k < n) {
#pragma unroll
        for (int r = 0; r < NR; ++r)
          if (lane + 64 * r < n) v[(size_t)(lane + 64 * r) * ld + k] = cscale(x[c].v[r], inv);
        if (lane == 0) a[(size_t)k * ld + k] = make_double2(nn, 0.0);
      }
    }
  }
  for (int k = 4 * nb + wave; k < n; k += blockDim.x >> 6) {
    for (int row = lane; row < n; row += 64) v[(size_t)row * ld + k] = cz();
    if (lane == 0) a[(size_t)k * ld + k] = cz();
  }
}

// ------------------------------------------------ circle ordering --------
// Round r of the parallel (circle) ordering of n indices (n even): pair m of
// the n / 2 disjoint pairs, p < q; the n - 1 rounds of a sweep pair every
// two indices once.
QMX_DEV void circle_pair(int n, int r, int m, int& p, int& q) {
  p = (m == 0) ? n - 1 : (r + m) % (n - 1);
  q = (r + n - 1 - m) % (n - 1);
  if (m == 0) q = r % (n - 1);
  if (p > q) { const int t = p; p = q; q = t; }
}

// ------------------------------------------- 129 to 1024 columns -----------
// The same eigensolver with a state's columns spread over the chip.
//
// Cholesky: panels of kPcPanel pivots.  One block per state takes a panel's
// pivots (thread = row, its entries of the panel's columns in registers; the
// pivot search and one column of A per step, two barriers), then the whole grid
// subtracts the panel from A.  Bound by the latency of the panel's steps; each
// panel reads and writes A once, which a step by step update would do
// kPcPanel times.
// Jacobi: L's columns lie one after the other in V's storage, 4 to a block of
// columns; one launch per round of the circle method, one thread block per pair
// of column blocks: rows spread over its four waves, one to a SIMD, the columns
// in registers, each set of four pairs' products summed over the waves through
// LDS.  Blocks of 8 columns would halve the launches, but run twice the sets on
// half the CUs (21 us a round against 8.4 at 600 columns, two rows a lane).  The launches of a sweep are bound by their own latency while a
// state has at most 512 columns (7.2 us a round at 512 to
// 600 columns, 3.4 to 4 without rotations; 8 to 9 sweeps).  One state of N = 18
// at chi = 300: 16.2 ms here and 1.7 in the Cholesky factors of five matrices of
// 512 and 600 columns; the two-sided block Jacobi below 176 + 108 ms.
// L is cut at max_rank columns, the number of rows the Gram matrix was formed
// from: more are rounding errors.
constexpr int kOsjWide = 1024;
constexpr int kPcPanel = 16;

// Panel k0 of the pivoted Cholesky factor.  diag: the remaining diagonal
// (-infinity: a pivot already) and, at ld, the trace.  rank: columns of L so
// far, the result once a panel comes out short; -1 as in chol_kernel.
__global__ __launch_bounds__(kOsjWide) void pchol_panel_kernel(const double2* a_all, double2* l_all, size_t stride,
                                                               const int* ncols_dev, int ld, int keep_all, int k0,
                                                               int max_rank, int* rank_all, double* diag_all) {
  __shared__ double wbest[16];
  __shared__ int wpiv[16];
  __shared__ double2 lp[kPcPanel];
  const int b = blockIdx.x;
  const int n = ncols_dev[b];
  const double2* a = a_all + (size_t)b * stride;
  double2* l_out = l_all + (size_t)b * stride;
  double* diag = diag_all + (size_t)b * (ld + 1);
  const int row = threadIdx.x, lane = row & 63, wave = __builtin_amdgcn_readfirstlane(row >> 6);
  const double inf = __builtin_inf();
  double d, tr;
  if (row < 16) wbest[row] = k0 == 0 ? 0.0 : -inf;   // (waves that a narrow launch has not)
  __syncthreads();
  if (k0 == 0) {
    if (n <= keep_all) {
      if (row == 0) rank_all[b] = -1;
      return;
    }
    d = row < n ? a[(size_t)row * ld + row].x : 0.0;
    const double w = rows_sum(sum16(d));
    if (lane == 0) wbest[wave] = w;
    __syncthreads();
    tr = 0.0;
    for (int k = 0; k < 16; ++k) tr += wbest[k];
    __syncthreads();   // (wbest is written again below)
    if (!(tr > 0.0) || !(tr < 1e300)) {
      if (row == 0) rank_all[b] = -1;
      return;
    }
    if (row == 0) diag[ld] = tr;
    // (only for waves that are not there: the others write theirs next)
    if (row < 16 && row >= (int)(blockDim.x >> 6)) wbest[row] = -inf;
    if (row >= n) d = -inf;
  } else {
    if (rank_all[b] != k0) return;
    d = row < n ? diag[row] : -inf;
    tr = diag[ld];
  }
  double2 l[kPcPanel];
#pragma unroll
  for (int t = 0; t < kPcPanel; ++t) l[t] = cz();
  int rank = k0;
  bool run = true;
#pragma unroll
  for (int j = 0; j < kPcPanel; ++j) {
    if (run) {
      // largest remaining diagonal entry, lowest index on ties
      auto max16 = [](double v) {
        v = fmax(v, dpp<kDppRow2>(v));
        v = fmax(v, dpp<kDppRow1>(v));
        v = fmax(v, dpp<kDppCol2>(v));
        return fmax(v, dpp<kDppSwap>(v));
      };
      double m = max16(d);
      m = fmax(m, __shfl_xor(m, 16, 64));
      m = fmax(m, __shfl_xor(m, 32, 64));
      const unsigned long long at = __ballot(d == m);
      if (lane == 0) {
        wbest[wave] = m;
        wpiv[wave] = 64 * wave + __ffsll(at) - 1;
      }
      __syncthreads();
      const double wm = wbest[lane & 15], best = max16(wm);
      const int wsel = __ffsll(__ballot(wm == best)) - 1;
      const int p = __builtin_amdgcn_readfirstlane(wpiv[wsel & 15]);
      if (best > kEps * tr && rank < max_rank && rank < n) {
        // (a column of the Hermitian matrix is its conjugated row: contiguous loads)
        double2 x = row < n ? cconj(a[(size_t)p * ld + row]) : cz();
        if (row == p)
#pragma unroll
          for (int t = 0; t < kPcPanel; ++t) lp[t] = l[t];
        __syncthreads();
#pragma unroll
        for (int t = 0; t < j; ++t) {
          const double2 c = lp[t];   // x -= l conj(c)
          x.x = fma(-l[t].x, c.x, fma(-l[t].y, c.y, x.x));
          x.y = fma(-l[t].y, c.x, fma(l[t].x, c.y, x.y));
        }
        const double inv = rsqrt_newton(best);
        x = d == -inf ? cz() : (row == p ? make_double2(best * inv, 0.0) : cscale(x, inv));
        l[j] = x;
        if (row < n) l_out[(size_t)rank * ld + row] = x;
        d = row == p ? -inf : d - cabs2(x);
        ++rank;
      } else {
        run = false;
      }
    }
  }
  if (row < n) diag[row] = d;
  if (row == 0) rank_all[b] = rank;
}

// A -= L_panel L_panel^H, 64 x 64 entries per block, for the states whose panel
// k0 is full
__global__ __launch_bounds__(256) void pchol_update_kernel(double2* a_all, const double2* l_all, size_t stride,
                                                           const int* ncols_dev, int ld, int k0, int ntile,
                                                           const int* rank_all) {
  __shared__ double2 li[kPcPanel][64], lj[kPcPanel][64];
  const int b = blockIdx.y;
  const int n = ncols_dev[b], i0 = blockIdx.x / ntile * 64, j0 = blockIdx.x % ntile * 64;
  if (rank_all[b] < k0 + kPcPanel || i0 >= n || j0 >= n) return;
  double2* a = a_all + (size_t)b * stride;
  const double2* l = l_all + (size_t)b * stride + (size_t)k0 * ld;
  const int tid = threadIdx.x, tx = tid & 15, ty = tid >> 4;
  for (int e = tid; e < kPcPanel * 64; e += 256) {
    const int t = e >> 6, r = e & 63;
    li[t][r] = i0 + r < n ? l[(size_t)t * ld + i0 + r] : cz();
    lj[t][r] = j0 + r < n ? l[(size_t)t * ld + j0 + r] : cz();
  }
  __syncthreads();
  double2 acc[4][4];
#pragma unroll
  for (int u = 0; u < 4; ++u)
#pragma unroll
    for (int w = 0; w < 4; ++w) acc[u][w] = cz();
#pragma unroll 2
  for (int t = 0; t < kPcPanel; ++t) {
    double2 x[4], y[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) x[u] = li[t][ty + 16 * u];
#pragma unroll
    for (int w = 0; w < 4; ++w) y[w] = lj[t][tx + 16 * w];
#pragma unroll
    for (int u = 0; u < 4; ++u)
#pragma unroll
      for (int w = 0; w < 4; ++w) acc[u][w] = cfmac(y[w], x[u], acc[u][w]);
  }
#pragma unroll
  for (int u = 0; u < 4; ++u)
#pragma unroll
    for (int w = 0; w < 4; ++w) {
      const int i = i0 + ty + 16 * u, j = j0 + tx + 16 * w;
      if (i < n && j < n) {
        double2* e = a + (size_t)i * ld + j;
        *e = csub(*e, acc[u][w]);
      }
    }
}

// Round r of a sweep over nb blocks of four columns: pair blockIdx.x of state
// blockIdx.y.  Round 0 also rotates the pairs inside the blocks and forms the
// squared norms, which later rounds read from nrm and update.
template <int NR>
__global__ __launch_bounds__(256) void osj_round_kernel(double2* l_all, size_t stride, int ld, const int* ncols_dev,
                                                        const int* rank_all, int nb, int r, double tol,
                                                        double* nrm_all, const int* conv, int* rot_all) {
  __shared__ double2 gpart[2][4][4];
  const int b = blockIdx.y;
  const int rank = rank_all[b];
  if (conv[b]) return;
  int I, J;
  circle_pair(nb, r, blockIdx.x, I, J);
  if (4 * (r == 0 ? I : J) >= rank) return;   // I < J: nothing but zero columns to pair
  const int n = ncols_dev[b];
  double2* l = l_all + (size_t)b * stride;
  double* nrm = nrm_all + (size_t)b * (ld + 1);
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int row0 = wave * 64 * NR + lane;
  auto column = [&](int c) { return c < 4 ? 4 * I + c : 4 * J + c - 4; };
  Col<NR> x[8];   // block I, block J
#pragma unroll
  for (int c = 0; c < 8; ++c)
#pragma unroll
    for (int h = 0; h < NR; ++h) {
      const int k = column(c), row = row0 + 64 * h;
      x[c].v[h] = k < rank && row < n ? l[(size_t)k * ld + row] : cz();
    }
  int par = 0;
  auto total = [&](double2 g) {
    if ((lane & 15) == 0) gpart[par][lane >> 4][wave] = g;
    __syncthreads();
    const double2 t = gpart[par][lane >> 4][lane & 3];
    par ^= 1;   // the next sum's values go to the other half: one barrier per sum
    return make_double2(sum4(t.x), sum4(t.y));
  };
  bool rot = false;
  double nt, nq;   // squared norms: row k of the wave, column k of block I / J
  if (r == 0) {
    auto inside = [&](Col<NR>& p0, Col<NR>& q0, Col<NR>& p1, Col<NR>& q1, Col<NR>& p2, Col<NR>& q2, Col<NR>& p3,
                      Col<NR>& q3) {
      double2 t = total(make_double2(norms4(p0, p1, p2, p3), norms4(q0, q1, q2, q3)));
      rot |= rotate4(p0, q0, p1, q1, p2, q2, p3, q3, t.x, t.y, tol, total);
    };
    inside(x[0], x[1], x[2], x[3], x[4], x[5], x[6], x[7]);
    inside(x[0], x[2], x[1], x[3], x[4], x[6], x[5], x[7]);
    inside(x[0], x[3], x[1], x[2], x[4], x[7], x[5], x[6]);
    const double2 t = total(make_double2(norms4(x[0], x[1], x[2], x[3]), norms4(x[4], x[5], x[6], x[7])));
    nt = t.x;
    nq = t.y;
  } else {
    const int k = lane >> 4;
    nt = 4 * I + k < rank ? nrm[4 * I + k] : 0.0;
    nq = 4 * J + k < rank ? nrm[4 * J + k] : 0.0;
  }
  // set s: pairs (top k, bottom (k + s) % 4); the bottom norms move up one row per set
  auto next = [&]() { nq = __shfl(nq, (lane + 16) & 63, 64); };
  rot |= rotate4(x[0], x[4], x[1], x[5], x[2], x[6], x[3], x[7], nt, nq, tol, total);
  next();
  rot |= rotate4(x[0], x[5], x[1], x[6], x[2], x[7], x[3], x[4], nt, nq, tol, total);
  next();
  rot |= rotate4(x[0], x[6], x[1], x[7], x[2], x[4], x[3], x[5], nt, nq, tol, total);
  next();
  rot |= rotate4(x[0], x[7], x[1], x[4], x[2], x[5], x[3], x[6], nt, nq, tol, total);
  next();
  if (wave == 0 && (lane & 15) == 0 && (rot || r == 0)) {
    const int k = lane >> 4;
    if (4 * I + k < rank) nrm[4 * I + k] = nt;
    if (4 * J + k < rank) nrm[4 * J + k] = nq;
  }
  if (!rot) return;
  if (threadIdx.x == 0) rot_all[b] = 1;
#pragma unroll
  for (int c = 0; c < 8; ++c)
#pragma unroll
    for (int h = 0; h < NR; ++h) {
      const int k = column(c), row = row0 + 64 * h;
      if (k < rank && row < n) l[(size_t)k * ld + row] = x[c].v[h];
    }
}

__global__ void osj_wide_begin_kernel(const int* rank_all, int* conv, int* rot, int batch) {
  const int b = blockIdx.x * blockDim.x + threadIdx.x;
  if (b >= batch) return;
  conv[b] = rank_all[b] <= 1;
  rot[b] = 0;
}

// eigenvalues to A's diagonal, one wave per column
__global__ __launch_bounds__(256) void osj_values_kernel(double2* a_all, const double2* l_all, size_t stride, int ld,
                                                         const int* ncols_dev, const int* rank_all, const int* conv,
                                                         int* error) {
  const int b = blockIdx.y;
  const int n = ncols_dev[b], rank = rank_all[b];
  const int k = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
  if (k == 0 && lane == 0 && !conv[b]) atomicOr(error, kErrEigNoConv);
  if (rank < 0 || k >= n) return;
  double s = 0.0;
  if (k < rank)
    for (int row = lane; row < n; row += 64) s += cabs2(l_all[(size_t)b * stride + (size_t)k * ld + row]);
  s = rows_sum(sum16(s));
  if (lane == 0) a_all[(size_t)b * stride + (size_t)k * ld + k] = make_double2(s, 0.0);
}

// eigenvectors: V[row][k] = L[k][row] / |L_k|, transposed in place by pairs of
// 32 x 32 tiles; the identity for a state that is not truncated
__global__ __launch_bounds__(256) void osj_vectors_kernel(const double2* a_all, double2* v_all, size_t stride, int ld,
                                                          const int* ncols_dev, const int* rank_all, int ntile) {
  __shared__ double2 t0[32][33], t1[32][33];
  const int b = blockIdx.y;
  const int n = ncols_dev[b], rank = rank_all[b];
  const int ti = blockIdx.x / ntile, tj = blockIdx.x % ntile;
  if (ti > tj || 32 * ti >= n || 32 * tj >= n) return;
  const double2* a = a_all + (size_t)b * stride;
  double2* v = v_all + (size_t)b * stride;
  const int x = threadIdx.x & 31, y0 = threadIdx.x >> 5;
  auto load = [&](double2 (&t)[32][33], int tk, int tr) {   // columns of tile tk, rows of tile tr
    for (int y = y0; y < 32; y += 8) {
      const int k = 32 * tk + y, row = 32 * tr + x;
      double2 e = cz();
      if (k < n && row < n) {
        if (rank < 0) {
          e = make_double2(k == row ? 1.0 : 0.0, 0.0);
        } else if (k < rank) {
          const double nn = a[(size_t)k * ld + k].x;
          e = cscale(v[(size_t)k * ld + row], nn > 0.0 ? rsqrt_newton(nn) : 0.0);
        }
      }
      t[y][x] = e;
    }
  };
  auto store = [&](const double2 (&t)[32][33], int tk, int tr) {
    for (int y = y0; y < 32; y += 8) {
      const int row = 32 * tr + y, k = 32 * tk + x;
      if (k < n && row < n) v[(size_t)row * ld + k] = t[x][y];
    }
  };
  load(t0, ti, tj);
  if (ti != tj) load(t1, tj, ti);
  __syncthreads();
  store(t0, ti, tj);
  if (ti != tj) store(t1, tj, ti);
}

// ----------------------------------------------------- block Jacobi -------
// QMX_OPT_TWO_SIDED_JACOBI for Gram matrices too large for one workgroup (n >
// 512, chi > 256): a two-sided block Jacobi over blocks of kBjBs columns.  The matrix is copied
// into an npad x npad buffer (npad = n rounded up to 2 kBjBs, zero padding:
// padded indices are never rotated, as every off-diagonal entry they have is
// zero), and the nb = npad / kBjBs blocks are paired by the same circle
// method as the scalar solvers: nb - 1 rounds per sweep, nb / 2 disjoint block
// pairs per round.  Per round:
//   solve: each pair's 2 kBjBs x 2 kBjBs Hermitian submatrix gets one cyclic
//          Jacobi sweep in LDS (the scalar solvers' rotation test), the
//          product U of its rotations is logged;
//   A <- A J (in place), A' = (A J)^H J into the other buffer, V <- V J (in
//   place), J the block-diagonal unitary of the round's U (columns permuted).
// After each sweep a state none of whose off-diagonal entries passes the
// rotation test is converged; the diagonal and V go back to the solver's
// own layout for select_kernel.
constexpr int kBjBs = 16;
constexpr int kBjSub = 2 * kBjBs;   // subproblem size (32)
constexpr int kBjRows = 32;         // rows per block of the apply kernel (ldp is a multiple of 64)
// The update A' = (A J)^H J is Hermitian only up to rounding, and a unitary
// conjugation carries an anti-Hermitian part forward unchanged (of order eps
// times the largest eigenvalue).  The solve rotates the Hermitian part of
// each submatrix, so the convergence test measures the Hermitian part of the
// off-diagonal entries too (testing the raw entries, a sweep never comes out
// clean once they are at that level); the rotation floor is the scalar
// solvers' (kJacobiAbsTol times the trace).

// Rotation (c, s, e^{-i phi}) of a pair from its diagonal entries al, be and
// its upper off-diagonal entry g: the scalar solvers' test (|g| above tol
// and above 1e-15 sqrt|al be|) and formulas, with a short chain of dependent
// FP64 operations for the latency-bound block solve: the test compares
// squares, and one reciprocal square root of |g|^2 gives both e^{-i phi} and
// tau = (be - al) / (2 |g|); t = sign(tau) / (|tau| + sqrt(1 + tau^2)),
// c = rsqrt(1 + t^2), s = t c.
QMX_DEV double4 bj_rotation(double al, double be, double2 g, double tol) {
  const double ag2 = g.x * g.x + g.y * g.y;
  const double thr = fmax(tol * tol, 1e-30 * fabs(al * be));
  if (!(ag2 > thr)) return make_double4(1.0, 0.0, 1.0, 0.0);
  const double ri = rsqrt(ag2);   // 1 / |g|
  const double tau = 0.5 * (be - al) * ri;
  const double t = (tau >= 0 ? 1.0 : -1.0) / (fabs(tau) + sqrt(1.0 + tau * tau));
  const double c = rsqrt(1.0 + t * t);
  return make_double4(c, t * c, g.x * ri, -g.y * ri);
}

QMX_DEV int bj_col(int nb, int r, int m, int l) {
  int P, Q;
  circle_pair(nb, r, m, P, Q);
  return l < kBjBs ? P * kBjBs + l : Q * kBjBs + (l - kBjBs);
}

// padded copies: ap = A (n x n of ld) with zeros up to npad, vp = I; scale =
// trace, conv = (n < 2), rot = 0
__global__ __launch_bounds__(256) void bj_init_kernel(const double2* a_all, size_t stride, const int* ncols_dev,
                                                      int ld, double2* ap_all, double2* vp_all, size_t pstride,
                                                      int ldp, double* scale, int* conv, int* rot) {
  const int b = blockIdx.y;
  const int n = ncols_dev[b];
  const double2* a = a_all + (size_t)b * stride;
  double2* ap = ap_all + (size_t)b * pstride;
  double2* vp = vp_all + (size_t)b * pstride;
  for (size_t e = blockIdx.x * (size_t)blockDim.x + threadIdx.x; e < (size_t)ldp * ldp;
       e += (size_t)gridDim.x * blockDim.x) {
    const int i = (int)(e / ldp), j = (int)(e % ldp);
    ap[e] = (i < n && j < n) ? a[(size_t)i * ld + j] : cz();
    vp[e] = make_double2(i == j ? 1.0 : 0.0, 0.0);
  }
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    double tr = 0.0;
    for (int i = 0; i < n; ++i) tr += fabs(a[(size_t)i * ld + i].x);
    scale[b] = tr;
    conv[b] = n < 2 ? 1 : 0;
    rot[b] = 0;
  }
}

// one block per (block pair m, state b): one Jacobi sweep of the pair's
// symmetrised submatrix S in LDS; U (product of the rotations) -> log
__global__ __launch_bounds__(256) void bj_solve_kernel(const double2* ap_all, size_t pstride, int ldp, int nb,
                                                       int r, double2* log_all, const double* scale,
                                                       const int* conv) {
  __shared__ double2 S[kBjSub][kBjSub + 1];
  __shared__ double2 U[kBjSub][kBjSub + 1];
  __shared__ double4 R[kBjSub / 2];
  __shared__ int col[kBjSub];
  const int b = blockIdx.y;
  if (conv[b]) return;
  const int m = blockIdx.x;
  const double2* ap = ap_all + (size_t)b * pstride;
  if (threadIdx.x < kBjSub) col[threadIdx.x] = bj_col(nb, r, m, threadIdx.x);
  __syncthreads();
  for (int e = threadIdx.x; e < kBjSub * kBjSub; e += blockDim.x) {
    const int i = e / kBjSub, j = e % kBjSub;
    const double2 x = ap[(size_t)col[i] * ldp + col[j]], y = ap[(size_t)col[j] * ldp + col[i]];
    S[i][j] = i == j ? make_double2(x.x, 0.0) : make_double2(0.5 * (x.x + y.x), 0.5 * (x.y - y.y));
    U[i][j] = make_double2(i == j ? 1.0 : 0.0, 0.0);
  }
  __syncthreads();
  const double tol = kJacobiAbsTol * scale[b] + 1e-300;
  constexpr int np = kBjSub / 2;
  for (int ir = 0; ir < kBjSub - 1; ++ir) {
    if (threadIdx.x < np) {
      int p, q;
      circle_pair(kBjSub, ir, threadIdx.x, p, q);
      R[threadIdx.x] = bj_rotation(S[p][p].x, S[q][q].x, S[p][q], tol);
    }
    __syncthreads();
    {
      // 2x2 block (P', Q') of S: K^H S J (one block per thread, in place)
      const int Pb = threadIdx.x / np, Qb = threadIdx.x % np;
      int p0, p1, q0, q1;
      circle_pair(kBjSub, ir, Pb, p0, p1);
      circle_pair(kBjSub, ir, Qb, q0, q1);
      const double4 RP = R[Pb], RQ = R[Qb];
      const double2 K00 = make_double2(RP.x, 0.0), K01 = make_double2(RP.y, 0.0);
      const double2 K10 = cscale(make_double2(RP.z, RP.w), -RP.y);
      const double2 K11 = cscale(make_double2(RP.z, RP.w), RP.x);
      const double2 J00 = make_double2(RQ.x, 0.0), J01 = make_double2(RQ.y, 0.0);
      const double2 J10 = cscale(make_double2(RQ.z, RQ.w), -RQ.y);
      const double2 J11 = cscale(make_double2(RQ.z, RQ.w), RQ.x);
      const double2 a00 = S[p0][q0], a01 = S[p0][q1], a10 = S[p1][q0], a11 = S[p1][q1];
      const double2 b00 = cadd(cmul(a00, J00), cmul(a01, J10));
      const double2 b01 = cadd(cmul(a00, J01), cmul(a01, J11));
      const double2 b10 = cadd(cmul(a10, J00), cmul(a11, J10));
      const double2 b11 = cadd(cmul(a10, J01), cmul(a11, J11));
      double2 c00 = cadd(cmulc(K00, b00), cmulc(K10, b10));
      double2 c01 = cadd(cmulc(K00, b01), cmulc(K10, b11));
      double2 c10 = cadd(cmulc(K01, b00), cmulc(K11, b10));
      double2 c11 = cadd(cmulc(K01, b01), cmulc(K11, b11));
      if (Pb == Qb) {
        c00.y = 0.0;
        c11.y = 0.0;
        c01 = cz();
        c10 = cz();
      }
      S[p0][q0] = c00;
      S[p0][q1] = c01;
      S[p1][q0] = c10;
      S[p1][q1] = c11;
      // U <- U J: items (row i, pair k), two per thread
      for (int it = threadIdx.x; it < kBjSub * np; it += blockDim.x) {
        const int i = it / np, k = it % np;
        int p, q;
        circle_pair(kBjSub, ir, k, p, q);
        const double4 Rk = R[k];
        const double2 em = make_double2(Rk.z, Rk.w);
        const double2 x = U[i][p], y = U[i][q];
        U[i][p] = cadd(cmul(x, make_double2(Rk.x, 0.0)), cmul(y, cscale(em, -Rk.y)));
        U[i][q] = cadd(cmul(x, make_double2(Rk.y, 0.0)), cmul(y, cscale(em, Rk.x)));
      }
    }
    __syncthreads();
  }
  double2* lg = log_all + ((size_t)b * (nb / 2) + m) * kBjSub * kBjSub;
  for (int e = threadIdx.x; e < kBjSub * kBjSub; e += blockDim.x) lg[e] = U[e / kBjSub][e % kBjSub];
}

// out[i][col_m[l]] = sum_k in'[i][col_m[k]] U_m[k][l] for rows [32 blockIdx.x, +32)
// and the round's pair m = blockIdx.y; in' = in (conjt = 0) or in^H (conjt = 1).
// blockIdx.z = mat * batch + b: matrix mat (0: in0 -> out0, 1: in1 -> out1)
// of state b, so that two independent updates share one launch.  With
// conjt = 0, in == out is allowed (a block reads its whole tile first).
__global__ __launch_bounds__(256) void bj_apply_kernel(const double2* in0, double2* out0, const double2* in1,
                                                       double2* out1, size_t pstride, int ldp, int nb, int r,
                                                       const double2* log_all, int conjt, const int* conv,
                                                       int batch) {
  __shared__ double2 X[kBjRows][kBjSub + 1];
  __shared__ double2 Um[kBjSub][kBjSub + 1];
  __shared__ int col[kBjSub];
  const int mat = blockIdx.z / batch, b = blockIdx.z % batch;
  if (conv[b]) return;
  const int m = blockIdx.y, i0 = blockIdx.x * kBjRows;
  const double2* in = (mat ? in1 : in0) + (size_t)b * pstride;
  double2* out = (mat ? out1 : out0) + (size_t)b * pstride;
  const double2* lg = log_all + ((size_t)b * (nb / 2) + m) * kBjSub * kBjSub;
  if (threadIdx.x < kBjSub) col[threadIdx.x] = bj_col(nb, r, m, threadIdx.x);
  for (int e = threadIdx.x; e < kBjSub * kBjSub; e += blockDim.x) Um[e / kBjSub][e % kBjSub] = lg[e];
  __syncthreads();
  if (!conjt) {
    for (int e = threadIdx.x; e < kBjRows * kBjSub; e += blockDim.x) {
      const int ii = e / kBjSub, k = e % kBjSub;
      X[ii][k] = in[(size_t)(i0 + ii) * ldp + col[k]];
    }
  } else {
    for (int e = threadIdx.x; e < kBjRows * kBjSub; e += blockDim.x) {
      const int ii = e % kBjRows, k = e / kBjRows;
      X[ii][k] = cconj(in[(size_t)col[k] * ldp + i0 + ii]);
    }
  }
  __syncthreads();
  // thread: column l = tid % 32, rows ii = tid / 32 + 8 t (t < kBjRows / 8)
  constexpr int kPer = kBjRows / 8;
  const int l = threadIdx.x % kBjSub, ib = threadIdx.x / kBjSub;
  double2 acc[kPer];
#pragma unroll
  for (int t = 0; t < kPer; ++t) acc[t] = cz();
  for (int k = 0; k < kBjSub; ++k) {
    const double2 u = Um[k][l];
#pragma unroll
    for (int t = 0; t < kPer; ++t) acc[t] = cfma(X[ib + 8 * t][k], u, acc[t]);
  }
#pragma unroll
  for (int t = 0; t < kPer; ++t) out[(size_t)(i0 + ib + 8 * t) * ldp + col[l]] = acc[t];
}

// rot[b] = 1 if the Hermitian part of an off-diagonal entry of the current A
// passes the rotation test (rot is clear on entry)
__global__ __launch_bounds__(256) void bj_check_kernel(const double2* acur_all, size_t pstride, const int* ncols_dev,
                                                       int ldp, const double* scale, const int* conv, int* rot) {
  const int b = blockIdx.y;
  if (conv[b]) return;
  const int n = ncols_dev[b];
  const double2* a = acur_all + (size_t)b * pstride;
  const double tol = kJacobiAbsTol * scale[b] + 1e-300;
  bool pass = false;
  for (size_t e = blockIdx.x * (size_t)blockDim.x + threadIdx.x; e < (size_t)n * n;
       e += (size_t)gridDim.x * blockDim.x) {
    const int i = (int)(e / n), j = (int)(e % n);
    if (j <= i) continue;
    const double2 x = a[(size_t)i * ldp + j], y = a[(size_t)j * ldp + i];
    const double ag = 0.5 * sqrt((x.x + y.x) * (x.x + y.x) + (x.y - y.y) * (x.y - y.y));
    if (ag > tol && ag > 1e-15 * sqrt(fabs(a[(size_t)i * ldp + i].x * a[(size_t)j * ldp + j].x))) pass = true;
  }
  if (pass) rot[b] = 1;
}

// end of a sweep: a running state whose A passed no rotation test converges
__global__ void bj_sweep_end_kernel(int* conv, int* rot, int batch) {
  const int b = blockIdx.x * blockDim.x + threadIdx.x;
  if (b >= batch) return;
  if (!conv[b] && !rot[b]) conv[b] = 1;
  rot[b] = 0;
}

// eigenvalues (diagonal of the final A) and V back into the solver's layout;
// a state still running after the last sweep did not converge
__global__ __launch_bounds__(256) void bj_store_kernel(const double2* cur_all, const double2* vp_all, size_t pstride,
                                                       int ldp, double2* a_all, double2* v_all, size_t stride,
                                                       int ld, const int* ncols_dev, const int* conv, int* error) {
  const int b = blockIdx.y;
  const int n = ncols_dev[b];
  const double2* cur = cur_all + (size_t)b * pstride;
  const double2* vp = vp_all + (size_t)b * pstride;
  double2* a = a_all + (size_t)b * stride;
  double2* v = v_all + (size_t)b * stride;
  for (size_t e = blockIdx.x * (size_t)blockDim.x + threadIdx.x; e < (size_t)n * n;
       e += (size_t)gridDim.x * blockDim.x) {
    const int i = (int)(e / n), j = (int)(e % n);
    v[(size_t)i * ld + j] = vp[(size_t)i * ldp + j];
    if (i == j) a[(size_t)i * ld + i] = make_double2(cur[(size_t)i * ldp + i].x, 0.0);
  }
  if (blockIdx.x == 0 && threadIdx.x == 0 && !conv[b]) atomicOr(error, kErrEigNoConv);
}

// ---------------------------------------------------------------- select ----
// Sort eigenvalues (diag of A) in decreasing order, pick k (rsum2 cutoff and
// max bond chi; k = n when n <= chi), and write the sorted eigenvectors into
// the columns of w (same layout as v).  k_out[b] = k; spectra (optional).
// keep_as_is: w is the identity when n <= chi (the one-sided solver's vectors
// of such a matrix are not a basis where its factor has no columns).
// Every block of a state sorts for itself and copies its rows of w; the first
// one also picks k (600 columns: 36 us, in one block 192).
constexpr int kSelectRows = 16;
__global__ __launch_bounds__(512) void select_kernel(const double2* a_all, const double2* v_all,
                                                     double2* w_all, size_t stride,
                                                     const int* ncols_dev, int ld, int chi, bool keep_as_is,
                                                     double cutoff, int* k_out, int kstride,
                                                     double* spectra, size_t spec_stride) {
  __shared__ double val[2 * kJacobiMaxPairs], lam[2 * kJacobiMaxPairs];
  __shared__ int perm[2 * kJacobiMaxPairs];
  const int b = blockIdx.y;
  const int n = ncols_dev[b], row0 = blockIdx.x * kSelectRows;
  if (row0 >= n) return;
  const double2* a = a_all + (size_t)b * stride;
  const double2* v = v_all + (size_t)b * stride;
  double2* w = w_all + (size_t)b * stride;
  // (entries that are not numbers have no rank: perm stays in range for them)
  for (int j = threadIdx.x; j < n; j += blockDim.x) {
    val[j] = a[(size_t)j * ld + j].x;
    lam[j] = 0.0;
    perm[j] = j;
  }
  __syncthreads();
  for (int j = threadIdx.x; j < n; j += blockDim.x) {
    const double lj = val[j];
    int rank = 0;
#pragma unroll 8
    for (int i = 0; i < n; ++i) {
      const double li = val[i];
      rank += li > lj || (li == lj && i < j);
    }
    lam[rank] = lj;
    perm[rank] = j;
  }
  __syncthreads();
  if (row0 == 0) {
    if (threadIdx.x == 0) {
      int k;
      if (n <= chi) {
        k = n;
      } else {
        double total = 0.0;
#pragma unroll 8
        for (int i = 0; i < n; ++i) total += fmax(lam[i], 0.0);
        k = n;
        if (total > 0.0 && cutoff > 0.0) {
          double tail = 0.0;
          for (int j = n - 1; j > 0; --j) {
            tail += fmax(lam[j], 0.0);
            if (tail <= cutoff * total) k = j; else break;
          }
        }
        if (k > chi) k = chi;
        if (k < 1) k = 1;
      }
      k_out[(size_t)b * kstride] = k;
    }
    if (spectra)
      for (int j = threadIdx.x; j < n; j += blockDim.x) spectra[(size_t)b * spec_stride + j] = lam[j];
  }
  for (int i = row0; i < min(row0 + kSelectRows, n); ++i)
    for (int c = threadIdx.x; c < n; c += blockDim.x)
      w[(size_t)i * ld + c] = keep_as_is && n <= chi ? make_double2(i == c ? 1.0 : 0.0, 0.0) : v[(size_t)i * ld + perm[c]];
}

// ------------------------------------------------------------------ gemm ----
// C (m x nc, ld nc) = A (m x kd, ld kd) * op(B); B has leading dimension ldb.
// 16 T x 16 T entries per block, T x T per thread, K in chunks of 16 fetched
// into registers one chunk ahead; T as in gram_kernel.  512 x
// 600 x 300: 27 us with T = 2, 96 with 40 tiles of T = 4; 32 states of 2^13 x 128
// x 64 and smaller: 197 us on average with T = 4.
template <int T>
__global__ __launch_bounds__(256) void gemm_kernel(const double2* __restrict__ a_all, size_t a_stride,
                                                   const double2* __restrict__ b_all, size_t b_stride,
                                                   double2* c_all, size_t c_stride, int rows_log2,
                                                   const int* kdim, const int* ncols, int dim_stride,
                                                   int kmax, int nmax, int ldb, int conj_b) {
  constexpr int kTile = 16 * T;
  __shared__ double2 as[kTile][17];
  __shared__ double2 bs[16][kTile + 1];
  const int b = blockIdx.z;
  const int kd = kdim ? kdim[(size_t)b * dim_stride] : kmax;
  const int nc = ncols ? ncols[(size_t)b * dim_stride] : nmax;
  const size_t m = (size_t)1 << rows_log2;
  const size_t row0 = (size_t)blockIdx.y * kTile;
  const int col0 = blockIdx.x * kTile;
  if (col0 >= nc || row0 >= m) return;
  const double2* A = a_all + (size_t)b * a_stride;
  const double2* B = b_all + (size_t)b * b_stride;
  double2* C = c_all + (size_t)b * c_stride;
  const int tx = threadIdx.x & 15, ty = threadIdx.x >> 4;
  double2 acc[T][T], fa[T], fb[T];
#pragma unroll
  for (int i = 0; i < T; ++i)
#pragma unroll
    for (int j = 0; j < T; ++j) acc[i][j] = cz();
  // (B^H: the chunk index runs fastest, as it does in memory)
  auto b_kk = [&](int e) { return conj_b ? e & 15 : e / kTile; };
  auto b_cc = [&](int e) { return conj_b ? e >> 4 : e % kTile; };
  auto fetch = [&](int k0) {
#pragma unroll
    for (int u = 0; u < T; ++u) {
      const int e = threadIdx.x + 256 * u;
      const size_t row = row0 + (e >> 4);
      const int ka = k0 + (e & 15), kb = k0 + b_kk(e), col = col0 + b_cc(e);
      fa[u] = row < m && ka < kd ? A[row * kd + ka] : cz();
      fb[u] = cz();
      if (kb < kd && col < nc) fb[u] = conj_b ? cconj(B[(size_t)col * ldb + kb]) : B[(size_t)kb * ldb + col];
    }
  };
  fetch(0);
  for (int k0 = 0; k0 < kd; k0 += 16) {
#pragma unroll
    for (int u = 0; u < T; ++u) {
      const int e = threadIdx.x + 256 * u;
      as[e >> 4][e & 15] = fa[u];
      bs[b_kk(e)][b_cc(e)] = fb[u];
    }
    __syncthreads();
    if (k0 + 16 < kd) fetch(k0 + 16);
#pragma unroll 4
    for (int kk = 0; kk < 16; ++kk) {
      double2 av[T], bv[T];
#pragma unroll
      for (int i = 0; i < T; ++i) av[i] = as[ty + 16 * i][kk];
#pragma unroll
      for (int j = 0; j < T; ++j) bv[j] = bs[kk][tx + 16 * j];
#pragma unroll
      for (int i = 0; i < T; ++i)
#pragma unroll
        for (int j = 0; j < T; ++j) acc[i][j] = cfma(av[i], bv[j], acc[i][j]);
    }
    __syncthreads();
  }
#pragma unroll
  for (int i = 0; i < T; ++i) {
    const size_t row = row0 + ty + 16 * i;
    if (row >= m) continue;
#pragma unroll
    for (int j = 0; j < T; ++j) {
      const int col = col0 + tx + 16 * j;
      if (col < nc) C[row * nc + col] = acc[i][j];
    }
  }
}

// ------------------------------------------------------------- launchers ----
void launch_gram(const double2* y, size_t y_stride, const int* ncols_dev, int rows_log2,
                 int ncols_max, double2* part, int nchunks, int batch, hipStream_t st) {
  const long nt = (ncols_max + 63) / 64;
  if (ncols_max > 32 && nt * nt * nchunks * batch >= kGemmFill) {
    hipLaunchKernelGGL(gram_kernel<4>, dim3(nt * nt, nchunks, batch), dim3(256), 0, st, y, y_stride,
                       ncols_dev, rows_log2, ncols_max, part, nchunks);
  } else {
    const int ns = (ncols_max + 31) / 32;
    hipLaunchKernelGGL(gram_kernel<2>, dim3(ns * ns, nchunks, batch), dim3(256), 0, st, y, y_stride,
                       ncols_dev, rows_log2, ncols_max, part, nchunks);
  }
}

void launch_gram_reduce(const double2* part, int nchunks, const int* ncols_dev, int ncols_max,
                        double2* a, size_t a_stride, int batch, hipStream_t st) {
  int tot = ncols_max * ncols_max;
  hipLaunchKernelGGL(gram_reduce_kernel, dim3((tot + 255) / 256, batch), dim3(256), 0, st, part,
                     nchunks, ncols_dev, ncols_max, a, a_stride);
}

void launch_jacobi(double2* a, double2* v, size_t stride, const int* ncols_dev, int ncols_max,
                   int batch, int max_sweeps, int* error, hipStream_t st) {
  hipLaunchKernelGGL(jacobi_kernel, dim3(batch), dim3(512), 0, st, a, v, stride, ncols_dev,
                     ncols_max, max_sweeps, error);
}

// block Jacobi workspace: padded A (two buffers) and V, the round's U log,
// scale, conv, rot
int bj_ldp(int ncols_max) { return (ncols_max + 63) / 64 * 64; }

size_t jacobi_block_bytes(int ncols_max, int batch) {
  const size_t ldp = (size_t)bj_ldp(ncols_max), nb = ldp / kBjBs;
  return 3 * (size_t)batch * ldp * ldp * sizeof(double2) + 256 +
         (size_t)batch * (nb / 2) * kBjSub * kBjSub * sizeof(double2) + 256 +
         (size_t)batch * (sizeof(double) + 2 * sizeof(int)) + 256;
}

int launch_jacobi_block(double2* a, double2* v, size_t stride, const int* ncols_dev, int ncols_max, int batch,
                        void* ws, int* conv_host_buf, int max_sweeps, int* error, hipStream_t st) {
  if (stride != (size_t)ncols_max * ncols_max) return -1;
  const int ldp = bj_ldp(ncols_max), nb = ldp / kBjBs;
  const size_t pstride = (size_t)ldp * ldp;
  auto up = [](size_t x) { return (x + 255) & ~static_cast<size_t>(255); };
  char* p = static_cast<char*>(ws);
  double2* ap = reinterpret_cast<double2*>(p);
  double2* a2 = ap + (size_t)batch * pstride;
  double2* vp = a2 + (size_t)batch * pstride;
  p += up(3 * (size_t)batch * pstride * sizeof(double2));
  double2* lg = reinterpret_cast<double2*>(p);
  p += up((size_t)batch * (nb / 2) * kBjSub * kBjSub * sizeof(double2));
  double* scale = reinterpret_cast<double*>(p);
  int* conv = reinterpret_cast<int*>(scale + batch);
  int* rot = conv + batch;
  hipLaunchKernelGGL(bj_init_kernel, dim3(std::max(1, ldp * ldp / 256 / 16), batch), dim3(256), 0, st, a, stride,
                     ncols_dev, ncols_max, ap, vp, pstride, ldp, scale, conv, rot);
  double2* cur = ap;
  double2* oth = a2;
  const dim3 sgrid(nb / 2, batch), agrid2(ldp / kBjRows, nb / 2, 2 * batch), agrid(ldp / kBjRows, nb / 2, batch);
  for (int s = 0; s < max_sweeps; ++s) {
    for (int r = 0; r < nb - 1; ++r) {
      hipLaunchKernelGGL(bj_solve_kernel, sgrid, dim3(256), 0, st, cur, pstride, ldp, nb, r, lg, scale, conv);
      // A <- A J and V <- V J (in place) in one launch, then A' = (A J)^H J
      hipLaunchKernelGGL(bj_apply_kernel, agrid2, dim3(256), 0, st, cur, cur, vp, vp, pstride, ldp, nb, r, lg, 0,
                         conv, batch);
      hipLaunchKernelGGL(bj_apply_kernel, agrid, dim3(256), 0, st, cur, oth, cur, oth, pstride, ldp, nb, r, lg, 1,
                         conv, batch);
      std::swap(cur, oth);
    }
    hipLaunchKernelGGL(bj_check_kernel, dim3(256, batch), dim3(256), 0, st, cur, pstride, ncols_dev, ldp, scale,
                       conv, rot);
    hipLaunchKernelGGL(bj_sweep_end_kernel, dim3((batch + 255) / 256), dim3(256), 0, st, conv, rot, batch);
    // stop once every state has converged (one host read per sweep)
    if (hipMemcpyAsync(conv_host_buf, conv, sizeof(int) * batch, hipMemcpyDeviceToHost, st) != hipSuccess ||
        hipStreamSynchronize(st) != hipSuccess)
      return -1;
    bool all = true;
    for (int b = 0; b < batch; ++b) all = all && conv_host_buf[b];
    if (all) break;
  }
  hipLaunchKernelGGL(bj_store_kernel, dim3(std::max(1, ncols_max * ncols_max / 256 / 16), batch), dim3(256), 0, st,
                     cur, vp, pstride, ldp, a, v, stride, ncols_max, ncols_dev, conv, error);
  return 0;
}

size_t jacobi_lds_log_doubles(int ncols_max) {
  return ncols_max <= kJacobiLdsMax ? (size_t)(ncols_max - 1) * (ncols_max / 2) * 4 : 0;
}

bool jacobi_lds_fits(int ncols_max) { return ncols_max >= 2 && ncols_max <= kJacobiLdsMax; }

void launch_jacobi_lds(double2* a, double2* v, size_t stride, const int* ncols_dev, int ncols_max,
                       int batch, double* log, int* state, int max_sweeps, int* error, hipStream_t st) {
  const size_t tri_bytes = sizeof(double2) * (size_t)ncols_max * (ncols_max + 1) / 2;
  const size_t log_stride = (size_t)(ncols_max - 1) * (ncols_max / 2);
  double4* lg = reinterpret_cast<double4*>(log);
  if (ncols_max <= kJacobiAllMax) {
    hipLaunchKernelGGL(jacobi_lds_sweep_kernel<true>, dim3(batch), dim3(1024),
                       tri_bytes + sizeof(double2) * (size_t)ncols_max * ncols_max, st, a, v, stride, ncols_dev,
                       ncols_max, lg, log_stride, state, max_sweeps, error);
    return;
  }
  hipLaunchKernelGGL(jacobi_lds_init_kernel, dim3((ncols_max * ncols_max + 255) / 256, batch), dim3(256), 0,
                     st, v, stride, ncols_dev, ncols_max, state, batch);
  const int row_blocks = (ncols_max + kJacobiRowsPerBlock - 1) / kJacobiRowsPerBlock;
  for (int s = 0; s < max_sweeps; ++s) {
    hipLaunchKernelGGL(jacobi_lds_sweep_kernel<false>, dim3(batch), dim3(1024), tri_bytes, st, a, v, stride,
                       ncols_dev, ncols_max, lg, log_stride, state, s, error);
    hipLaunchKernelGGL(jacobi_lds_rows_kernel, dim3(row_blocks, batch), dim3(1024), 0, st, v, stride,
                       ncols_dev, ncols_max, lg, log_stride, state, s);
  }
  hipLaunchKernelGGL(jacobi_lds_check_kernel, dim3((batch + 255) / 256), dim3(256), 0, st, state, batch,
                     error);
}

// The dynamic-LDS limit is set to the largest triangle the kernel takes
// (kJacobiLdsMax columns), whatever ncols_max this call needs: calls from
// several host threads (one per ragged bucket) then never lower it under a
// launch that needs more.
hipError_t jacobi_lds_setup(int ncols_max) {
  if (ncols_max > kJacobiLdsMax) return hipErrorInvalidValue;
  const size_t tri_bytes = sizeof(double2) * (size_t)kJacobiLdsMax * (kJacobiLdsMax + 1) / 2;
  const size_t all_bytes = sizeof(double2) * ((size_t)kJacobiAllMax * (kJacobiAllMax + 1) / 2 +
                                              (size_t)kJacobiAllMax * kJacobiAllMax);
  const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(jacobi_lds_sweep_kernel<true>),
                                           hipFuncAttributeMaxDynamicSharedMemorySize, (int)all_bytes);
  if (e != hipSuccess) return e;
  return hipFuncSetAttribute(reinterpret_cast<const void*>(jacobi_lds_sweep_kernel<false>),
                             hipFuncAttributeMaxDynamicSharedMemorySize, (int)tri_bytes);
}

bool osj_fits(int ncols_max) { return ncols_max >= 1 && ncols_max <= kOsjMax; }

int launch_osj(double2* a, double2* v, size_t stride, const int* ncols_dev, int ncols_max, int batch, int keep_all,
               int* rank, int max_sweeps, int* error, hipStream_t st) {
  const int waves = (ncols_max + 7) / 8;
  // the dynamic-LDS limit is set to the largest need (16 waves), whatever this
  // call needs, so that launches from several host threads never lower it
  const size_t most = (size_t)17 * 4 * 128 * sizeof(double2);
  if (ncols_max > 64 && hipFuncSetAttribute(reinterpret_cast<const void*>(osj_kernel<2>),
                                            hipFuncAttributeMaxDynamicSharedMemorySize, (int)most) != hipSuccess)
    return -1;
  hipLaunchKernelGGL(chol_kernel, dim3(batch), dim3(1024), 0, st, a, stride, ncols_dev, ncols_max, keep_all, rank);
  if (ncols_max <= 64) {
    // at most 9 slots of 4 KiB: below the default limit
    const size_t shm = (size_t)(waves + 1) * 4 * 64 * sizeof(double2);
    hipLaunchKernelGGL(osj_kernel<1>, dim3(batch), dim3(64 * waves), shm, st, a, v, stride, ncols_dev, ncols_max,
                       rank, max_sweeps, error);
  } else {
    const size_t shm = (size_t)(waves + 1) * 4 * 128 * sizeof(double2);
    hipLaunchKernelGGL(osj_kernel<2>, dim3(batch), dim3(64 * waves), shm, st, a, v, stride, ncols_dev, ncols_max,
                       rank, max_sweeps, error);
  }
  return 0;
}

bool osj_wide_fits(int ncols_max) { return ncols_max > kOsjMax && ncols_max <= kOsjWide; }

// state: 3 ints per state (rank, converged, rotated); diag: ncols_max + 1
// doubles per state.  rows: of the matrix that the Gram matrices belong to.
int launch_osj_wide(double2* a, double2* v, size_t stride, const int* ncols_dev, int ncols_max, int rows, int batch,
                    int keep_all, int* state, double* diag, int* conv_host_buf, int max_sweeps, int* error,
                    hipStream_t st) {
  const int max_rank = std::min(ncols_max, rows);
  int *rank = state, *conv = state + batch, *rot = conv + batch;
  const int ut = (ncols_max + 63) / 64, vt = (ncols_max + 31) / 32;
  const int threads = (ncols_max + 63) / 64 * 64;
  for (int k0 = 0; k0 < max_rank; k0 += kPcPanel) {
    hipLaunchKernelGGL(pchol_panel_kernel, dim3(batch), dim3(threads), 0, st, a, v, stride, ncols_dev, ncols_max,
                       keep_all, k0, max_rank, rank, diag);
    if (k0 + kPcPanel < max_rank)
      hipLaunchKernelGGL(pchol_update_kernel, dim3(ut * ut, batch), dim3(256), 0, st, a, v, stride, ncols_dev,
                         ncols_max, k0, ut, rank);
  }
  hipLaunchKernelGGL(osj_wide_begin_kernel, dim3((batch + 255) / 256), dim3(256), 0, st, rank, conv, rot, batch);
  const int nb = ((max_rank + 3) / 4 + 1) & ~1;
  auto* const round = ncols_max <= 256 ? osj_round_kernel<1> : ncols_max <= 512 ? osj_round_kernel<2>
                    : ncols_max <= 768 ? osj_round_kernel<3> : osj_round_kernel<4>;
  const double tol = kOsjTol * std::sqrt(std::max(1.0, ncols_max / 128.0));
  for (int s = 0; s < max_sweeps; ++s) {
    for (int r = 0; r < nb - 1; ++r)
      hipLaunchKernelGGL(round, dim3(nb / 2, batch), dim3(256), 0, st, v, stride, ncols_max,
                         ncols_dev, rank, nb, r, tol, diag, conv, rot);
    hipLaunchKernelGGL(bj_sweep_end_kernel, dim3((batch + 255) / 256), dim3(256), 0, st, conv, rot, batch);
    // stop once every state has converged (one host read per sweep)
    if (hipMemcpyAsync(conv_host_buf, conv, sizeof(int) * batch, hipMemcpyDeviceToHost, st) != hipSuccess ||
        hipStreamSynchronize(st) != hipSuccess)
      return -1;
    bool all = true;
    for (int b = 0; b < batch; ++b) all = all && conv_host_buf[b];
    if (all) break;
  }
  hipLaunchKernelGGL(osj_values_kernel, dim3((ncols_max + 3) / 4, batch), dim3(256), 0, st, a, v, stride, ncols_max,
                     ncols_dev, rank, conv, error);
  hipLaunchKernelGGL(osj_vectors_kernel, dim3(vt * vt, batch), dim3(256), 0, st, a, v, stride, ncols_max, ncols_dev,
                     rank, vt);
  return 0;
}

void launch_select(const double2* a, const double2* v, double2* w, size_t stride,
                   const int* ncols_dev, int ncols_max, int chi, bool keep_as_is, double cutoff,
                   int* k_out, int kstride, double* spectra, size_t spec_stride, int batch, hipStream_t st) {
  hipLaunchKernelGGL(select_kernel, dim3((ncols_max + kSelectRows - 1) / kSelectRows, batch),
                     dim3(std::min(512, (ncols_max + 63) / 64 * 64)), 0, st, a, v, w, stride, ncols_dev, ncols_max, chi,
                     keep_as_is, cutoff, k_out, kstride, spectra, spec_stride);
}

// nn[b][step] = ncur[b] = first_cols (> 0) or 2 * kk[b][step + 1]
__global__ void chain_dims_kernel(int* nn, int* ncur, const int* kk, int n, int step,
                                  int first_cols, int batch) {
  int b = blockIdx.x * blockDim.x + threadIdx.x;
  if (b >= batch) return;
  int v = first_cols > 0 ? first_cols : 2 * kk[(size_t)b * (n + 1) + step + 1];
  nn[(size_t)b * (n + 1) + step] = v;
  ncur[b] = v;
}

void launch_chain_dims(int* nn, int* ncur, const int* kk, int n, int step, int first_cols,
                       int batch, hipStream_t st) {
  hipLaunchKernelGGL(chain_dims_kernel, dim3((batch + 63) / 64), dim3(64), 0, st, nn, ncur, kk, n,
                     step, first_cols, batch);
}

// Sweep early stop: skip[b] = 1 once |<psi|C|0>| >= goal[b]; active[0] counts
// the states still running, whose sweeps_done[b] is incremented.
__global__ void goal_check_kernel(const double2* dot, int dot_stride, const double* goal, int* skip,
                                  int* active, int* sweeps_done, int batch) {
  int b = blockIdx.x * blockDim.x + threadIdx.x;
  if (b >= batch) return;
  if (!skip[b]) {
    double2 d = dot[(size_t)b * dot_stride];
    double f = sqrt(d.x * d.x + d.y * d.y);
    if (f >= goal[b]) {
      skip[b] = 1;
    } else {
      atomicAdd(active, 1);
      if (sweeps_done) sweeps_done[b] += 1;
    }
  }
}

void launch_goal_check(const double2* dot, int dot_stride, const double* goal, int* skip,
                       int* active, int* sweeps_done, int batch, hipStream_t st) {
  hipLaunchKernelGGL(goal_check_kernel, dim3((batch + 63) / 64), dim3(64), 0, st, dot, dot_stride,
                     goal, skip, active, sweeps_done, batch);
}

// one block: chunks of 1024 states, each compacted by a block-wide exclusive
// scan of the live flags
__global__ __launch_bounds__(1024) void live_list_kernel(const int* skip, int batch, int* list) {
  __shared__ int sc[1024];
  int base = 0;
  for (int b0 = 0; b0 < batch; b0 += 1024) {
    const int b = b0 + (int)threadIdx.x;
    const int live = (b < batch && !skip[b]) ? 1 : 0;
    sc[threadIdx.x] = live;
    __syncthreads();
    for (int off = 1; off < 1024; off <<= 1) {
      const int v = threadIdx.x >= (unsigned)off ? sc[threadIdx.x - off] : 0;
      __syncthreads();
      sc[threadIdx.x] += v;
      __syncthreads();
    }
    if (live) list[base + sc[threadIdx.x] - 1] = b;
    const int total = sc[1023];
    __syncthreads();
    base += total;
  }
}

void launch_live_list(const int* skip, int batch, int* list, hipStream_t st) {
  hipLaunchKernelGGL(live_list_kernel, dim3(1), dim3(1024), 0, st, skip, batch, list);
}

void launch_gemm(const double2* a, size_t a_stride, const double2* bm, size_t b_stride, double2* c,
                 size_t c_stride, const GemmDims& d, int conj_b, int batch, hipStream_t st) {
  size_t m = (size_t)1 << d.rows_log2;
  const size_t big = (size_t)((d.nmax + 63) / 64) * ((m + 63) / 64) * batch;
  if (d.nmax > 32 && m > 32 && big >= (size_t)kGemmFill) {
    dim3 grid((d.nmax + 63) / 64, (unsigned)((m + 63) / 64), batch);
    hipLaunchKernelGGL(gemm_kernel<4>, grid, dim3(256), 0, st, a, a_stride, bm, b_stride, c, c_stride,
                       d.rows_log2, d.kdim, d.ncols, d.dim_stride, d.kmax, d.nmax, d.ldb, conj_b);
  } else {
    dim3 grid((d.nmax + 31) / 32, (unsigned)((m + 31) / 32), batch);
    hipLaunchKernelGGL(gemm_kernel<2>, grid, dim3(256), 0, st, a, a_stride, bm, b_stride, c, c_stride,
                       d.rows_log2, d.kdim, d.ncols, d.dim_stride, d.kmax, d.nmax, d.ldb, conj_b);
  }
}

}  // namespace qmx
