// Device-side helpers shared by the qmx kernels (gfx950, wave64).
//
// Complex numbers are double2 (re, im) in registers and LDS; dense states are
// stored either as float2 (complex64) or double2 (complex128) in HBM.
// All small linear algebra here is FP64: the matrices are tiny and the results
// feed every later step.  The 4x4 Hermitian eigensolver and the Householder
// completion run serially in one lane, the 4x4 polar factor on one wave.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#define QMX_DEV __device__ __forceinline__

// ---------------------------------------------------------------- complex --
QMX_DEV double2 cz() { return make_double2(0.0, 0.0); }
QMX_DEV double2 cadd(double2 a, double2 b) { return make_double2(a.x + b.x, a.y + b.y); }
QMX_DEV double2 csub(double2 a, double2 b) { return make_double2(a.x - b.x, a.y - b.y); }
QMX_DEV double2 cmul(double2 a, double2 b) {
  return make_double2(fma(a.x, b.x, -a.y * b.y), fma(a.x, b.y, a.y * b.x));
}
// conj(a) * b
QMX_DEV double2 cmulc(double2 a, double2 b) {
  return make_double2(fma(a.x, b.x, a.y * b.y), fma(a.x, b.y, -a.y * b.x));
}
// acc + a * b
QMX_DEV double2 cfma(double2 a, double2 b, double2 acc) {
  acc.x = fma(a.x, b.x, acc.x);
  acc.x = fma(-a.y, b.y, acc.x);
  acc.y = fma(a.x, b.y, acc.y);
  acc.y = fma(a.y, b.x, acc.y);
  return acc;
}
// acc + conj(a) * b
QMX_DEV double2 cfmac(double2 a, double2 b, double2 acc) {
  acc.x = fma(a.x, b.x, acc.x);
  acc.x = fma(a.y, b.y, acc.x);
  acc.y = fma(a.x, b.y, acc.y);
  acc.y = fma(-a.y, b.x, acc.y);
  return acc;
}
QMX_DEV double2 cconj(double2 a) { return make_double2(a.x, -a.y); }
QMX_DEV double2 cscale(double2 a, double s) { return make_double2(a.x * s, a.y * s); }
QMX_DEV double cabs2(double2 a) { return fma(a.x, a.x, a.y * a.y); }
QMX_DEV double cabs_(double2 a) { return sqrt(cabs2(a)); }

// storage <-> compute conversion
QMX_DEV double2 to_c(float2 v) { return make_double2((double)v.x, (double)v.y); }
QMX_DEV double2 to_c(double2 v) { return v; }
template <typename S> QMX_DEV S from_c(double2 v);
template <> QMX_DEV float2 from_c<float2>(double2 v) { return make_float2((float)v.x, (float)v.y); }
template <> QMX_DEV double2 from_c<double2>(double2 v) { return v; }

// ------------------------------------------------------------- reductions --
QMX_DEV double wave_sum(double v) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
  return v;
}

// ------------------------------------------------- 4x4 Hermitian Jacobi ----
// Cyclic two-sided Jacobi on a 4 x 4 Hermitian matrix a (row-major; pad a
// smaller matrix with zeros).  On return lam[] holds the eigenvalues in
// decreasing order and the columns of v the matching orthonormal eigenvectors.
// All indices are compile-time so the arrays stay in registers.
QMX_DEV void herm_eig4(double2* a, double2* v, double* lam) {
#pragma unroll
  for (int i = 0; i < 16; ++i) v[i] = make_double2((i % 5) == 0 ? 1.0 : 0.0, 0.0);
  for (int sweep = 0; sweep < 40; ++sweep) {
    double off = 0.0, diag = 0.0;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      diag += a[i * 4 + i].x * a[i * 4 + i].x;
#pragma unroll
      for (int j = i + 1; j < 4; ++j) off += cabs2(a[i * 4 + j]);
    }
    if (off <= 1e-32 * diag || off == 0.0) break;
#pragma unroll
    for (int p = 0; p < 3; ++p) {
#pragma unroll
      for (int q = p + 1; q < 4; ++q) {
        double2 g = a[p * 4 + q];
        double ag = cabs_(g);
        if (ag != 0.0) {
          double al = a[p * 4 + p].x, be = a[q * 4 + q].x;
          double2 ph = make_double2(g.x / ag, g.y / ag);  // e^{i phi}
          double tau = (be - al) / (2.0 * ag);
          double t = (tau >= 0 ? 1.0 : -1.0) / (fabs(tau) + sqrt(1.0 + tau * tau));
          double c = 1.0 / sqrt(1.0 + t * t), sn = t * c;
          // J = [[c, s], [-s e^{-i phi}, c e^{-i phi}]] acting on columns (p, q)
          double2 em = cconj(ph);
          double2 j00 = make_double2(c, 0), j01 = make_double2(sn, 0);
          double2 j10 = cscale(em, -sn), j11 = cscale(em, c);
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            double2 x = a[i * 4 + p], y = a[i * 4 + q];
            a[i * 4 + p] = cadd(cmul(x, j00), cmul(y, j10));
            a[i * 4 + q] = cadd(cmul(x, j01), cmul(y, j11));
            double2 vx = v[i * 4 + p], vy = v[i * 4 + q];
            v[i * 4 + p] = cadd(cmul(vx, j00), cmul(vy, j10));
            v[i * 4 + q] = cadd(cmul(vx, j01), cmul(vy, j11));
          }
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            double2 x = a[p * 4 + j], y = a[q * 4 + j];
            a[p * 4 + j] = cadd(cmulc(j00, x), cmulc(j10, y));
            a[q * 4 + j] = cadd(cmulc(j01, x), cmulc(j11, y));
          }
          a[p * 4 + q] = cz();
          a[q * 4 + p] = cz();
          a[p * 4 + p].y = 0.0;
          a[q * 4 + q].y = 0.0;
        }
      }
    }
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) lam[i] = a[i * 4 + i].x;
  // decreasing order by a fixed compare-exchange network (stable on ties)
#define QMX_CX(i, j)                                                        \
  if (lam[j] > lam[i]) {                                                    \
    double tl = lam[i]; lam[i] = lam[j]; lam[j] = tl;                       \
    _Pragma("unroll") for (int r = 0; r < 4; ++r) {                         \
      double2 tv = v[r * 4 + i]; v[r * 4 + i] = v[r * 4 + j]; v[r * 4 + j] = tv; \
    }                                                                       \
  }
  QMX_CX(0, 1) QMX_CX(2, 3) QMX_CX(0, 2) QMX_CX(1, 3) QMX_CX(1, 2)
#undef QMX_CX
}

// rsum2 cutoff + max_bond keep count (decreasing eigenvalues lam[0..n-1]).
QMX_DEV int keep_count(const double* lam, int n, int max_bond, double cutoff) {
  double total = 0.0;
  for (int i = 0; i < n; ++i) total += fmax(lam[i], 0.0);
  int k = n;
  if (total > 0.0 && cutoff > 0.0) {
    double tail = 0.0;
    for (int j = n - 1; j > 0; --j) {
      tail += fmax(lam[j], 0.0);
      if (tail <= cutoff * total) k = j; else break;
    }
  }
  if (max_bond > 0 && k > max_bond) k = max_bond;
  return k < 1 ? 1 : k;
}

// Canonical orthonormal basis of span(v[:, 0:k]) (columns of a 4 x 4 v;
// pad smaller problems with zero rows): two-pass Gram-Schmidt over the
// columns of the projector P = V V^H in index order, skipping residuals with
// norm <= tol.  Writes w (columns 0..found-1).  Returns found (== k unless
// the input is degenerate).  Compile-time indices only.
QMX_DEV int canonical_basis4(int k, const double2* v, double2* w, double tol) {
  double2 p[16];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      double2 s = cz();
#pragma unroll
      for (int m = 0; m < 4; ++m)
        if (m < k) s = cfma(v[i * 4 + m], cconj(v[j * 4 + m]), s);
      p[i * 4 + j] = s;
    }
#pragma unroll
  for (int i = 0; i < 16; ++i) w[i] = cz();
  int found = 0;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    if (found < k) {
      double2 x[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) x[i] = p[i * 4 + j];
#pragma unroll
      for (int pass = 0; pass < 2; ++pass) {
#pragma unroll
        for (int b = 0; b < 4; ++b) {
          if (b < found) {
            double2 d = cz();
#pragma unroll
            for (int i = 0; i < 4; ++i) d = cfmac(w[i * 4 + b], x[i], d);
#pragma unroll
            for (int i = 0; i < 4; ++i) x[i] = csub(x[i], cmul(w[i * 4 + b], d));
          }
        }
      }
      double nrm = 0.0;
#pragma unroll
      for (int i = 0; i < 4; ++i) nrm += cabs2(x[i]);
      nrm = sqrt(nrm);
      if (nrm > tol) {
#pragma unroll
        for (int c = 0; c < 4; ++c)
          if (c == found) {
#pragma unroll
            for (int i = 0; i < 4; ++i) w[i * 4 + c] = cscale(x[i], 1.0 / nrm);
          }
        ++found;
      }
    }
  }
  return found;
}

// ------------------------------------------------------- polar (d <= 4) ----
// ---- the polar factor on one wave ---------------------------------------------
// A 4 x 4 matrix lives in 16 lanes, lane l = 4 i + j holding entry (i, j); the
// wave's four rows of 16 lanes all hold the same matrix, so every branch below
// is uniform over the wave.  Neighbours are read with DPP moves (row_ror by
// multiples of 4 walks the matrix rows, quad_perm the columns), which cost
// their issue slots only; a ds_bpermute would add an LDS round trip to a chain
// that is bound by its latency.
template <int CTRL>
QMX_DEV double dpp(double v) {
  const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(v), CTRL, 0xf, 0xf, true);
  const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(v), CTRL, 0xf, 0xf, true);
  return __hiloint2double(hi, lo);
}
constexpr int kDppRow1 = 0x12c, kDppRow2 = 0x128, kDppRow3 = 0x124;   // lane + 4, 8, 12 of the 16
constexpr int kDppCol2 = 0x4e;                                         // matrix column (j + 2) % 4
constexpr int kDppSwap = 0xb1;                                         // column j ^ 1

// sum over the 16 lanes (both partners add the same two values at every
// level, so every lane holds the bitwise same sum)
QMX_DEV double sum16(double v) {
  v += dpp<kDppRow2>(v);
  v += dpp<kDppRow1>(v);
  v += dpp<kDppCol2>(v);
  v += dpp<kDppSwap>(v);
  return v;
}
QMX_DEV double lane_value(double v, int lane) {
  return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(v), lane),
                          __builtin_amdgcn_readlane(__double2loint(v), lane));
}

// Half-wave (quarter-wave) exchange and add: lanes below 32 (even rows of 16)
// get a's sum over the two halves (the row and the next), the others b's.
QMX_DEV double swap_add32(double a, double b) {
  const auto lo = __builtin_amdgcn_permlane32_swap(__double2loint(a), __double2loint(b), false, false);
  const auto hi = __builtin_amdgcn_permlane32_swap(__double2hiint(a), __double2hiint(b), false, false);
  return __hiloint2double(hi[0], lo[0]) + __hiloint2double(hi[1], lo[1]);
}
QMX_DEV double swap_add16(double a, double b) {
  const auto lo = __builtin_amdgcn_permlane16_swap(__double2loint(a), __double2loint(b), false, false);
  const auto hi = __builtin_amdgcn_permlane16_swap(__double2hiint(a), __double2hiint(b), false, false);
  return __hiloint2double(hi[0], lo[0]) + __hiloint2double(hi[1], lo[1]);
}
// the sum over the wave's four rows of 16 lanes, on every lane
QMX_DEV double rows_sum(double v) {
  v = swap_add32(v, v);
  return swap_add16(v, v);
}

template <int J> QMX_DEV double quad_bcast(double v) { return dpp<J * 0x55>(v); }
template <int J> QMX_DEV double2 quad_bcast2(double2 v) { return make_double2(quad_bcast<J>(v.x), quad_bcast<J>(v.y)); }
// The totals over the wave of four per-lane values: row k (lanes 16 k ..
// 16 k + 15) holds the total of v_k on every lane.  Two half-swaps merge the
// four registers, then four DPP steps add inside the rows.
QMX_DEV double rows_total(double v0, double v1, double v2, double v3) {
  return sum16(swap_add16(swap_add32(v0, v2), swap_add32(v1, v3)));
}

// 1 / x to rounding: the hardware estimate and two Newton steps
QMX_DEV double rcp_newton(double x) {
  double r = __builtin_amdgcn_rcp(x);
  r = fma(fma(-x, r, 1.0), r, r);
  return fma(fma(-x, r, 1.0), r, r);
}

// 1 / sqrt(x) to rounding, x in the normal range away from its ends
QMX_DEV double rsqrt_newton(double x) {
  double r = __builtin_amdgcn_rsq(x);
  const double h = 0.5 * x;
  r = fma(r, fma(-h * r, r, 0.5), r);
  return fma(r, fma(-h * r, r, 0.5), r);
}

// ---- 4 x 4 Hermitian eigenproblem on one wave -----------------------------------
// Two-sided Jacobi with entry (i, j) of A and V in lane 4 i + j: the two
// disjoint rotations of a round run side by side (rounds pair an index with
// itself ^ X, X = 1, 2, 3), every entry is updated by its own lane.  With
// d = a_qq - a_pp, g = a_pq, the rotation p' = c (p - conj(te) q), q' = c (q +
// te p) has te = 2 g sign(d) / (|d| + sqrt(d^2 + 4 |g|^2)) and c = 1 / sqrt(1 +
// |te|^2); w is the weight of an index's partner, -conj(te) or te.
// Bound by the chain of a round's dependent operations; a step of the layers'
// chain at N = 10, which is mostly this, takes 11.3 us, with the one-lane solver
// above 28.
template <int X> QMX_DEV double2 row_partner(double2 v) {   // lane ^ 4 X
  if constexpr (X == 2) return make_double2(dpp<kDppRow2>(v.x), dpp<kDppRow2>(v.y));
  // mirrored within 8 or 16 lanes, the quads turned back
  constexpr int mirror = X == 1 ? 0x141 : 0x140;
  return make_double2(dpp<mirror>(dpp<0x1b>(v.x)), dpp<mirror>(dpp<0x1b>(v.y)));
}
template <int X> QMX_DEV double2 col_partner(double2 v) {   // lane ^ X
  constexpr int perm = X == 1 ? kDppSwap : X == 2 ? kDppCol2 : 0x1b;
  return make_double2(dpp<perm>(v.x), dpp<perm>(v.y));
}
template <int X> QMX_DEV void herm_eig4_round(double2& a, double2& v, int i, int j) {
  constexpr int kP = X == 1 ? 2 : 1, kQ = kP ^ X;   // the pair beside (0, X)
  const bool jf = j == 0 || j == X, jq = j > (j ^ X), fi = i == 0 || i == X, iq = i > (i ^ X);
  const double al = jf ? lane_value(a.x, 0) : lane_value(a.x, 5 * kP);
  const double be = jf ? lane_value(a.x, 5 * X) : lane_value(a.x, 5 * kQ);
  const double2 g = make_double2(jf ? lane_value(a.x, X) : lane_value(a.x, 4 * kP + kQ),
                                 jf ? lane_value(a.y, X) : lane_value(a.y, 4 * kP + kQ));
  const double ag2 = cabs2(g), d = be - al;
  const bool rot = ag2 > 1e-280;
  const double q = fma(4.0, ag2, d * d);
  double f = 2.0 * rcp_newton(fma(q, rsqrt_newton(q), fabs(d)));
  f = rot ? (d >= 0.0 ? f : -f) : 0.0;
  const double2 te = rot ? cscale(g, f) : cz();
  const double c = rsqrt_newton(1.0 + cabs2(te));
  const double2 w = jq ? te : make_double2(-te.x, te.y);
  // the same of this lane's row index, from its quad
  const double2 w0 = quad_bcast2<0>(w), w1 = quad_bcast2<kP>(w);
  const double cr = fi ? quad_bcast<0>(c) : quad_bcast<kP>(c);
  double2 wr = fi ? w0 : w1;                      // of the pair's first index: -conj(te)
  if (iq) wr = make_double2(-wr.x, wr.y);
  const double2 ac = cscale(cfma(w, col_partner<X>(a), a), c);
  v = cscale(cfma(w, col_partner<X>(v), v), c);
  a = cscale(cfmac(wr, row_partner<X>(ac), ac), cr);
  if (i == j) a.y = 0.0;
  if (rot && i == (j ^ X)) a = cz();
}
// Eigenvalues of the matrix a (entry (i, j) in lane 4 i + j, the same in each
// row of 16 lanes) in decreasing order to lam[4] and the eigenvectors to the columns of vec[16],
// both in LDS; a matrix that is not finite gives vectors that are not.
QMX_DEV void herm_eig4_wave(double2 a, int lane, double* lam, double2* vec) {
  const int i = (lane >> 2) & 3, j = lane & 3;
  double2 v = make_double2(i == j ? 1.0 : 0.0, 0.0);
  const double all = sum16(cabs2(a));
  for (int sweep = 0; sweep < 40; ++sweep) {
    const double off = sum16(i < j ? cabs2(a) : 0.0), diag = sum16(i == j ? a.x * a.x : 0.0);
    if (off <= 1e-32 * diag || off < 1e-270) break;
    herm_eig4_round<1>(a, v, i, j);
    herm_eig4_round<2>(a, v, i, j);
    herm_eig4_round<3>(a, v, i, j);
  }
  // place of column j: stable, decreasing
  const double l0 = lane_value(a.x, 0), l1 = lane_value(a.x, 5), l2 = lane_value(a.x, 10), l3 = lane_value(a.x, 15);
  const double lj = j == 0 ? l0 : j == 1 ? l1 : j == 2 ? l2 : l3;
  const int at = (l0 > lj || (l0 == lj && 0 < j)) + (l1 > lj || (l1 == lj && 1 < j)) +
                 (l2 > lj || (l2 == lj && 2 < j)) + (l3 > lj || (l3 == lj && 3 < j));
  const double bad = 0.0 * all;
  if (lane < 16) {
    vec[4 * i + at] = make_double2(v.x + bad, v.y + bad);
    if (i == j) lam[at] = lj;
  }
}

// ---- 4 x 4 complex products on the matrix cores --------------------------------
// v_mfma_f64_4x4x4_4b: four 4 x 4 products at once, operands A[i][k] in lane
// i + 4 blk + 16 k, B[k][j] in lane j + 4 blk + 16 k, result D[i][j] in lane
// j + 4 blk + 16 i (checked on gfx950).  A complex matrix M is held in the
// result's layout, real parts in the even blocks and imaginary parts in the odd
// ones (v, the two pairs of blocks alike), with the other part beside it (o).
// As an A operand this layout reads as the transpose.
struct Mat4 {
  double v, o;
};
QMX_DEV Mat4 mat4(double v) { return {v, dpp<kDppRow3>(v)}; }   // row_ror:4: the block before
// C + M^T B, or C + M^H B with CONJ
template <bool CONJ>
QMX_DEV double mat4_tmul(Mat4 m, Mat4 b, bool even, double c = 0.0) {
  const double re = even ? m.v : m.o;
  const double im = CONJ ? (even ? m.o : -m.v) : (even ? -m.o : m.v);
  const double d = __builtin_amdgcn_mfma_f64_4x4x4f64(re, b.v, c, 0, 0, 0);
  return __builtin_amdgcn_mfma_f64_4x4x4f64(im, b.o, d, 0, 0, 0);
}
// C + M^T B with the sums of mat4_tmul<false>(b, m): the same bits, transposed
QMX_DEV double mat4_tmul_swapped(Mat4 m, Mat4 b, bool even, double c = 0.0) {
  const double d = __builtin_amdgcn_mfma_f64_4x4x4f64(m.v, even ? b.v : b.o, c, 0, 0, 0);
  return __builtin_amdgcn_mfma_f64_4x4x4f64(even ? -m.o : m.o, even ? b.o : b.v, d, 0, 0, 0);
}

QMX_DEV bool polar4_rank2(double2& x, int l, const double2* es, int h, double fro, double* nuc);
// Unitary polar factor of es 2^h (|.|_F^2 = fro, near 1) by the scaled
// Newton-Schulz iteration
//   X <- X (a - b X^H X),  a = 3 s / 2,  b = s^3 / 2,
// two products per step, on one wave.  It maps a singular value x <= 1 to
// f(s x) <= 1, f(y) = y (3 - y^2) / 2, and with s^2 = 3 / (1 + l + l^2) the
// interval [l, 1] to [f(s l), 1], the best a cubic can do (J. Chen, E. Chow, "A
// stable scaling of Newton-Schulz for improving the sign function computation
// of a Hermitian matrix", 2014).  Six steps are scaled for l = 0.05, then s = 1,
// which gains a factor of 1.5 per step on a value that is still small and ends
// quadratically: once |X^H X - 1| <= 3e-9 in every entry the next step is exact
// to rounding.  On the sweeps' environments (condition numbers 5 to 90 at the
// median, 1e3 to 1e4 at the 90th percentile) that takes 8 to 14 steps on
// average.  The transpose of X is carried along as the left operand, with the
// same sums and so the same rounding.
// The steps' roundings turn X away from E's factor, by eps over the singular
// values of the time: the first step has the matrix as it is (its norm is in
// the step's coefficients), and the last X is turned back, X <- X + X W: with
// X^H E = (1 + W) H, H Hermitian, X^H E - E^H X is H W + W H, of which 0.9 over
// E's norm is taken for W (all of it for equal singular values, less for the
// small ones, whose share the early steps decide).
// Bound by the latency of the two products, about 300 cycles per step: 4600
// cycles for a Gaussian 4 x 4 matrix, 6400 at condition number 1000 (4100 and
// 5800 without the exact start and the turn back).  The scaled Newton iteration
// took 24000 and 27000 with its pivoted inverse by ds_bpermute.  Error against
// 80-bit arithmetic, rms of the factor, and the Newton iteration's: Gaussian
// 4.4e-16 and 5.3e-16, unitary 2.3e-16 and 2.5e-16, condition numbers up to 10
// 3.4e-16 and 3.5e-16, up to 1000 2.5e-15 and 2.9e-15, up to 1e5 1.27e-13 and
// 1.29e-13 (without the exact start and the turn back 6.5e-16, 4.4e-16, 5.5e-16,
// 3.5e-15 and 1.7e-13).
// u: this lane's part of the factor in the split layout.  False after 34
// unscaled steps (a condition number above about 1e6).
QMX_DEV bool polar4_newton_schulz(const double2* es, int h, double fro, int lane, Mat4& u, double2& x2, double& nuc2,
                                  bool& rank2) {
  const int i = lane >> 4, j = lane & 3;
  const bool even = !(lane & 4);
  const double r = rsqrt_newton(fro);
  const double2 e = es[4 * i + j], t = es[4 * j + i];
  const Mat4 x0 = mat4(ldexp(even ? e.x : e.y, h));   // r x0 is the matrix to start from
  Mat4 x = x0, xt = mat4(ldexp(even ? t.x : t.y, h));
  const double one = even && i == j ? 1.0 : 0.0;
  // X <- X P, or X + X P; and its transpose, bit for bit
  auto times = [&](double pv, bool add) {
    const Mat4 p = mat4(pv);
    const double xn = mat4_tmul<false>(xt, p, even, add ? x.v : 0.0);
    const double tn = mat4_tmul_swapped(p, xt, even, add ? xt.v : 0.0);
    x = mat4(xn);
    xt = mat4(tn);
  };
  auto gram = [&]() { return mat4_tmul<true>(x, x, even); };
  auto scaled = [&](double a, double b) { times(fma(-b, gram(), a * one), false); };
  scaled(2.5324497354750872 * r, 2.406128014703171 * (r * r * r));   // l = 0.05
  scaled(2.430892812235437, 2.128107957418897);    // 0.1263
  scaled(2.200129819325986, 1.5777607537549168);   // 0.3028
  scaled(1.832672820412407, 0.9119080391587333);   // 0.6224
  scaled(1.5614350757473685, 0.5639856062462636);  // 0.9208
  scaled(1.5019149323066294, 0.5019173779907503);  // 0.9974
  for (int it = 0; it < 34; ++it) {
    const double y = gram();
    if (it == 0) {
      // Two singular values that are zero, or below 1e-4 or so, leave the trace
      // of X^H X, by now about the number of the others, no larger than 2
      const double tr = (lane_value(y, 0) + lane_value(y, 17)) + (lane_value(y, 34) + lane_value(y, 51));
      if (tr < 2.0001 && polar4_rank2(x2, lane & 15, es, h, fro, &nuc2)) {
        rank2 = true;
        return true;
      }
    }
    const bool last = __all(fabs(y - one) <= 3e-9);
    times(0.5 * (one - y), true);
    if (last) {
      times(0.9 * r * (mat4_tmul<true>(x, x0, even) - mat4_tmul<true>(x0, x, even)), true);
      u = x;
      return true;
    }
  }
  return false;
}

// Unitary polar factor of a 2 x 2 matrix (a b; c d): with e = det / |det|,
// M + e adj(M)^H has both singular values s_1 + s_2, whose square is
// |M|_F^2 + 2 |det|; so the factor is that sum over its norm.  False for a
// matrix singular to 1e-13.  |M|_F is near 1.
QMX_DEV bool polar2(double2& a, double2& b, double2& c, double2& d, double* nuc) {
  const double fro = (cabs2(a) + cabs2(b)) + (cabs2(c) + cabs2(d));
  const double2 det = csub(cmul(a, d), cmul(b, c));
  const double d2 = cabs2(det);
  if (!(d2 > 1e-26 * fro * fro)) return false;
  const double id = rsqrt_newton(d2);
  const double2 e = cscale(det, id);
  const double s2 = fma(2.0 * d2, id, fro);
  const double r = rsqrt_newton(s2);
  *nuc = s2 * r;
  // adj(M)^H = (conj d, -conj c; -conj b, conj a)
  const double2 a2 = cadd(a, cmulc(d, e)), b2 = csub(b, cmulc(c, e));
  const double2 c2 = csub(c, cmulc(b, e)), e2 = cadd(d, cmulc(a, e));
  a = cscale(a2, r); b = cscale(b2, r); c = cscale(c2, r); d = cscale(e2, r);
  return true;
}

// sum over the 4 rows i
QMX_DEV double col_total(double v) {
  v += dpp<kDppRow2>(v);
  return v + dpp<kDppRow1>(v);
}
// sum over the 4 columns j
QMX_DEV double row_total(double v) {
  v += dpp<kDppSwap>(v);
  return v + dpp<kDppCol2>(v);
}
// x - q (q^H x), x and q by the lanes' rows i: a second pass for an x that was
// e_k - sum q conj(q_k), whose rounding grows with what was taken off
QMX_DEV double2 without(double2 x, double2 q) {
  const double2 t = cmulc(q, x);
  return csub(x, cmul(q, make_double2(col_total(t.x), col_total(t.y))));
}
// Two unit vectors beside q_0, q_1 (rows in the lanes' i), as polar4_jacobi
// completes: residuals of the first e_k, in order, whose squared norm is above 1/4
QMX_DEV bool complete_two(int i, double2 q0, double2 q1, double2& q2, double2& q3) {
  // squared residual of e_i against q_0, q_1; the first above 1/4
  const double res = 1.0 - cabs2(q0) - cabs2(q1);
  const unsigned m2 = (unsigned)__ballot(res > 0.25) & 0x1111u;
  if (!m2) return false;
  const int e2 = __builtin_amdgcn_readfirstlane((__ffs(m2) - 1) >> 2);
  auto row = [&](double2 v, int k) { return make_double2(lane_value(v.x, 4 * k), lane_value(v.y, 4 * k)); };
  double2 t = cadd(cmulc(row(q0, e2), q0), cmulc(row(q1, e2), q1));
  q2 = make_double2((i == e2 ? 1.0 : 0.0) - t.x, -t.y);
  q2 = without(without(q2, q0), q1);
  q2 = cscale(q2, rsqrt_newton(col_total(cabs2(q2))));
  const unsigned m3 = (unsigned)__ballot(i > e2 && res - cabs2(q2) > 0.25) & 0x1111u;
  if (!m3) return false;
  const int e3 = __builtin_amdgcn_readfirstlane((__ffs(m3) - 1) >> 2);
  t = cadd(cadd(cmulc(row(q0, e3), q0), cmulc(row(q1, e3), q1)), cmulc(row(q2, e3), q2));
  q3 = make_double2((i == e3 ? 1.0 : 0.0) - t.x, -t.y);
  q3 = without(without(without(q3, q0), q1), q2);
  q3 = cscale(q3, rsqrt_newton(col_total(cabs2(q3))));
  return true;
}

// The environments of the gates next to a site still in |0>: two columns of E
// are zero (to 1e-14 of its norm; the Jacobi path drops singular values below
// 1e-13 of the largest).  With Q R = the two columns left (Gram-Schmidt, two
// passes), their part of the factor is Q polar(R); the zero columns z_1 < z_2,
// whose right singular vectors are e_{z_1}, e_{z_2}, take the rule's left
// completion, the first unit vectors with a residual above 1/2.  Lane 4 i + j of
// 16 works on row i and on column j of (live, live, zero, zero).  zero: the zero
// columns (bits), es 2^h: the matrix, fro: its squared norm, near 1; x: entry
// (i, j) of the factor.  False where the Jacobi path decides (30600 cycles); 2900
// cycles, against 5300 to 7500 with the whole problem in every lane.
QMX_DEV bool polar4_two_columns(double2& x, int l, const double2* es, int h, unsigned zero, double fro, double* nuc) {
  const unsigned live = ~zero & 15u;
  const int c0 = __ffs(live) - 1, c1 = 31 - __clz(live), z0 = __ffs(zero) - 1, z1 = 31 - __clz(zero);
  const int i = l >> 2, j = l & 3;
  const double2 e = es[4 * i + (j & 1 ? c1 : c0)];
  double2 y = make_double2(ldexp(e.x, h), ldexp(e.y, h));   // columns j = 0, 1 (and again at 2, 3)
  const double n0 = quad_bcast<0>(col_total(cabs2(y)));
  const double i0 = rsqrt_newton(n0);
  const double2 q0 = cscale(quad_bcast2<0>(y), i0);         // row i of q_0
  double2 p00 = make_double2(n0 * i0, 0.0), p01 = cz(), p10 = cz();
#pragma unroll
  for (int pass = 0; pass < 2; ++pass) {
    const double2 t = cmulc(q0, y);
    const double2 d = make_double2(col_total(t.x), col_total(t.y));
    p01 = cadd(p01, quad_bcast2<1>(d));
    y = csub(y, cmul(q0, d));
  }
  const double n1 = quad_bcast<1>(col_total(cabs2(y)));
  if (!(n1 > 1e-26 * fro)) return false;
  const double i1 = rsqrt_newton(n1);
  const double2 q1 = cscale(quad_bcast2<1>(y), i1);
  double2 p11 = make_double2(n1 * i1, 0.0);
  if (!polar2(p00, p01, p10, p11, nuc)) return false;
  double2 q2, q3;
  if (!complete_two(i, q0, q1, q2, q3)) return false;
  // out column z_1: q_2, z_2: q_3, the live ones: Q polar(R)
  const double2 a = j == c0 ? p00 : p01, b = j == c0 ? p10 : p11;
  x = cadd(cmul(q0, a), cmul(q1, b));
  if (j == z0) x = q2;
  if (j == z1) x = q3;
  return true;
}

// The same with three zero columns, the environment of the gate whose both
// sites are in |0>: the live column over its norm, and three completions.
QMX_DEV bool polar4_one_column(double2& x, int l, const double2* es, int h, unsigned zero, double* nuc) {
  const int c0 = __ffs(~zero & 15u) - 1;
  const int i = l >> 2, j = l & 3;
  const double2 e = es[4 * i + c0];
  const double2 y = make_double2(ldexp(e.x, h), ldexp(e.y, h));
  const double n0 = col_total(cabs2(y)), i0 = rsqrt_newton(n0);
  *nuc = n0 * i0;
  double2 q[4];
  q[0] = cscale(y, i0);
  x = q[0];
  double res = 1.0 - cabs2(q[0]);   // squared residual of e_i
  int from = 0, slot = 0;
#pragma unroll
  for (int k = 1; k < 4; ++k) {
    const unsigned m = (unsigned)__ballot(i >= from && res > 0.25) & 0x1111u;
    if (!m) return false;
    const int ek = __builtin_amdgcn_readfirstlane((__ffs(m) - 1) >> 2);
    double2 t = cz();
#pragma unroll
    for (int b = 0; b < k; ++b)
      t = cadd(t, cmulc(make_double2(lane_value(q[b].x, 4 * ek), lane_value(q[b].y, 4 * ek)), q[b]));
    double2 w = make_double2((i == ek ? 1.0 : 0.0) - t.x, -t.y);
#pragma unroll
    for (int b = 0; b < k; ++b) w = without(w, q[b]);
    q[k] = cscale(w, rsqrt_newton(col_total(cabs2(w))));
    res -= cabs2(q[k]);
    from = ek + 1;
    if (slot == c0) ++slot;
    if (j == slot) x = q[k];
    ++slot;
  }
  return true;
}

// one of four by two selects (a chain of comparisons becomes a table in memory)
QMX_DEV double2 pick4(int k, double2 a, double2 b, double2 c, double2 d) {
  const double2 lo = make_double2(k & 1 ? b.x : a.x, k & 1 ? b.y : a.y);
  const double2 hi = make_double2(k & 1 ? d.x : c.x, k & 1 ? d.y : c.y);
  return make_double2(k & 2 ? hi.x : lo.x, k & 2 ? hi.y : lo.y);
}
// A dense E of rank 2, the environment of the first site's gate above the first
// circuit layer, whose state has Schmidt rank 2 beside it: E = Q L W^H by
// column-pivoted Gram-Schmidt and again on the rows, and the factor is
// Q polar(L) W^H with both sides completed as polar4_jacobi completes them.
// Taken when nothing above 3e-14 of the norm is left beside Q (the Jacobi path
// drops singular values below 1e-13).  9500 cycles with the six steps that find
// it out; it is met once a sweep, and the Jacobi path took 64000 there.
QMX_DEV bool polar4_rank2(double2& x, int l, const double2* es, int h, double fro, double* nuc) {
  const int i = l >> 2, j = l & 3;
  auto at = [&](int c) {
    const double2 e = es[4 * i + c];
    return make_double2(ldexp(e.x, h), ldexp(e.y, h));
  };
  double2 y = at(j);
  auto largest = [&](double n) {   // the column of the largest n (the same down each column)
    const double n0 = lane_value(n, 0), n1 = lane_value(n, 1), n2 = lane_value(n, 2), n3 = lane_value(n, 3);
    const int a = n1 > n0 ? 1 : 0, b = n3 > n2 ? 3 : 2;
    return fmax(n2, n3) > fmax(n0, n1) ? b : a;
  };
  auto project = [&](double2 q, double2& r) {   // y -= q (q^H y), r += q^H y
#pragma unroll
    for (int pass = 0; pass < 2; ++pass) {
      const double2 t = cmulc(q, y);
      const double2 d = make_double2(col_total(t.x), col_total(t.y));
      r = cadd(r, d);
      y = csub(y, cmul(q, d));
    }
  };
  double n = col_total(cabs2(y));
  const int c0 = largest(n);
  double2 q0 = at(c0);
  q0 = cscale(q0, rsqrt_newton(col_total(cabs2(q0))));
  double2 r0 = cz(), r1 = cz();
  project(q0, r0);
  n = col_total(cabs2(y));
  const int c1 = largest(n);
  double2 q1 = quad_bcast2<0>(y);
  if (c1 == 1) q1 = quad_bcast2<1>(y);
  if (c1 == 2) q1 = quad_bcast2<2>(y);
  if (c1 == 3) q1 = quad_bcast2<3>(y);
  const double n1 = col_total(cabs2(q1));
  if (!(n1 > 1e-26 * fro)) return false;
  q1 = cscale(q1, rsqrt_newton(n1));
  project(q1, r1);
  if (!(sum16(cabs2(y)) < 1e-27 * fro)) return false;
  // rows r_0, r_1 = L W^H
  const double m0 = row_total(cabs2(r0)), i0 = rsqrt_newton(m0);
  double2 w0 = cscale(cconj(r0), i0), l10 = cz();
#pragma unroll
  for (int pass = 0; pass < 2; ++pass) {
    const double2 t = cmul(r1, w0);
    const double2 d = make_double2(row_total(t.x), row_total(t.y));
    l10 = cadd(l10, d);
    r1 = csub(r1, cmul(d, cconj(w0)));
  }
  const double m1 = row_total(cabs2(r1));
  if (!(m1 > 1e-26 * fro)) return false;
  const double i1 = rsqrt_newton(m1);
  double2 w1 = cscale(cconj(r1), i1);
  double2 p00 = make_double2(m0 * i0, 0.0), p01 = cz(), p10 = l10, p11 = make_double2(m1 * i1, 0.0);
  if (!polar2(p00, p01, p10, p11, nuc)) return false;
  double2 u2, u3, v2, v3;
  if (!complete_two(i, q0, q1, u2, u3)) return false;
  // W's entries by the lanes' i for its completion, and that by their j
  auto by_row = [&](double2 v) {
    const double2 a = quad_bcast2<0>(v), b = quad_bcast2<1>(v), c = quad_bcast2<2>(v), d = quad_bcast2<3>(v);
    return pick4(i, a, b, c, d);
  };
  auto by_col = [&](double2 v) {
    auto row = [&](int k) { return make_double2(lane_value(v.x, 4 * k), lane_value(v.y, 4 * k)); };
    const double2 a = row(0), b = row(1), c = row(2), d = row(3);
    return pick4(j, a, b, c, d);
  };
  if (!complete_two(i, by_row(w0), by_row(w1), v2, v3)) return false;
  v2 = by_col(v2);
  v3 = by_col(v3);
  const double2 a = cadd(cmul(q0, p00), cmul(q1, p10)), b = cadd(cmul(q0, p01), cmul(q1, p11));
  x = cadd(cadd(cmul(a, cconj(w0)), cmul(b, cconj(w1))), cadd(cmul(u2, cconj(v2)), cmul(u3, cconj(v3))));
  return true;
}

// Polar factor of the d x d matrix in es (LDS, stride 4, zero outside the
// block) on one wave, to out (LDS; imaginary parts times sgn).  *nuc: the sum of
// the singular values, if wanted.  False: the matrix is left to polar4_jacobi.
QMX_DEV bool polar4_wave(int d, const double2* es, double2* out, double sgn, int lane, bool want, double* nuc) {
  const int l = lane & 15, i = l >> 2, j = l & 3;
  const double2 e = es[l];
  const double n2 = cabs2(e);
  double fro = sum16(n2);
  if (!(fro > 1e-280) || !(fro < 1e280)) return false;
  // exact scaling by a power of two to a squared norm in [1/2, 2)
  const int h = -(__builtin_amdgcn_frexp_exp(fro) >> 1);
  double2 x;
  double s = 0.0;
  if (d == 2) {
    auto at = [&](int k) {
      const double2 v = es[k];
      return make_double2(ldexp(v.x, h), ldexp(v.y, h));
    };
    double2 a = at(0), b = at(1), c = at(4), f = at(5);
    const double n0 = cabs2(a) + cabs2(c), n1 = cabs2(b) + cabs2(f);
    if (n1 <= 1e-28 * n0) {
      // the site is still in |0>: one column, completed as in polar4_jacobi
      const double r = rsqrt_newton(n0);
      s = n0 * r;
      a = cscale(a, r);
      c = cscale(c, r);
      const bool first = cabs2(c) > 0.25;   // the residual of e_0 has norm |c|
      const double2 g = first ? a : c;
      const double2 t0 = cmulc(g, a), t1 = cmulc(g, c);
      b = make_double2((first ? 1.0 : 0.0) - t0.x, -t0.y);
      f = make_double2((first ? 0.0 : 1.0) - t1.x, -t1.y);
      const double2 again = cadd(cmulc(a, b), cmulc(c, f));
      b = csub(b, cmul(a, again));
      f = csub(f, cmul(c, again));
      const double q = rsqrt_newton(cabs2(b) + cabs2(f));
      b = cscale(b, q);
      f = cscale(f, q);
    } else if (!polar2(a, b, c, f, &s)) {
      return false;
    }
    x = i == 0 ? (j == 0 ? a : b) : (j == 0 ? c : f);
    if (i > 1 || j > 1) x = cz();
    if (lane < 16) out[l] = make_double2(x.x, sgn * x.y);
    *nuc = ldexp(s, -h);
    return true;
  }
  // columns with an entry above 1e-14 of the norm
  const unsigned long long big = __ballot(n2 > 1e-28 * fro);
  unsigned zero = 0;
#pragma unroll
  for (int k = 0; k < 4; ++k)
    if (!(big & (0x1111ull << k))) zero |= 1u << k;
  fro = ldexp(fro, 2 * h);
  if (__popc(zero) >= 2) {
    if (!(__popc(zero) == 2 ? polar4_two_columns(x, l, es, h, zero, fro, &s)
                            : polar4_one_column(x, l, es, h, zero, &s)))
      return false;
    if (lane < 16) out[l] = make_double2(x.x, sgn * x.y);
    *nuc = ldexp(s, -h);
    return true;
  }
  Mat4 u;
  bool singular = false;
  if (!polar4_newton_schulz(es, h, fro, lane, u, x, s, singular)) return false;
  if (singular) {
    if (lane < 16) out[l] = make_double2(x.x, sgn * x.y);
    *nuc = ldexp(s, -h);
    return true;
  }
  if (!(lane & 12)) out[4 * (lane >> 4) + (lane & 3)] = make_double2(u.v, sgn * u.o);
  if (want) {   // Re tr(U^H E)
    __builtin_amdgcn_wave_barrier();
    const double2 g = out[l];
    *nuc = sum16(g.x * e.x + sgn * g.y * e.y);
  }
  return true;
}

// Unitary polar factor U V^H of the d x d (d = 2 or 4) matrix e (row-major,
// stride 4, zero outside the block) for the inputs that polar4_wave leaves to
// it: a one-sided (Hestenes) Jacobi SVD on a 4 x 4 working matrix (a
// 2 x 2 problem is embedded as diag(E, |E| I), whose padded columns are
// orthogonal to E's and never rotate).  Rotations: cyclic pairs p < q, when
// |a_p^H a_q| > 1e-16 |a_p| |a_q|.  Pairs (u_j, v_j) with sigma_j >
// 1e-13 sigma_max are kept; each other column j (in increasing j) receives
// the next unit vector e_0, e_1, ... whose two-pass Gram-Schmidt residual
// against the columns already set has norm > 1/2, on both the U and V sides.
// The result then depends only on the well-determined singular subspaces.
// *nuc = sum of E's singular values.
// Lane k of a quad holds row k of both matrices, every quad the same, and the
// loops that need not be unrolled are not: with everything in one lane's
// registers this was 70 KiB of code, and a call, which found none of it in the
// instruction cache, took 64000 cycles and left the rest of the sweep to be
// fetched again.  A matrix of rank 3: 48000 cycles against 190000 (4000 blocks).
QMX_DEV void polar4_jacobi(int d, const double2* e, double2* out, double sgn, int lane, double* nuc) {
  const int i = lane & 3;
  double2 a[4], v[4];
  double fro = 0.0;
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    a[c] = e[4 * i + c];
    fro += cabs2(a[c]);
    v[c] = make_double2(i == c ? 1.0 : 0.0, 0.0);
  }
  fro = row_total(fro);
  // exact scaling to a squared norm near 1
  const int h = fro > 0.0 && fro < __builtin_inf() ? -(__builtin_amdgcn_frexp_exp(fro) >> 1) : 0;
  const double s = fro > 0.0 ? sqrt(ldexp(fro, 2 * h)) : 1.0;
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    a[c] = make_double2(ldexp(a[c].x, h), ldexp(a[c].y, h));
    if (d == 2 && (i >= 2 || c >= 2)) a[c] = make_double2(i == c ? s : 0.0, 0.0);
  }
  auto dot = [](double2 x, double2 y) {   // x^H y
    const double2 t = cmulc(x, y);
    return make_double2(row_total(t.x), row_total(t.y));
  };
#pragma unroll 1
  for (int sweep = 0; sweep < 60; ++sweep) {
    bool rotated = false;
#pragma unroll
    for (int p = 0; p < 3; ++p)
#pragma unroll
      for (int q = p + 1; q < 4; ++q) {
        const double al = row_total(cabs2(a[p])), be = row_total(cabs2(a[q]));
        const double2 g = dot(a[p], a[q]);
        const double ag2 = cabs2(g);
        if (ag2 > 0.0 && ag2 > 1e-32 * (al * be)) {
          rotated = true;
          const double dd = be - al, w = fma(4.0, ag2, dd * dd);
          double f = 2.0 * rcp_newton(fma(w, rsqrt_newton(w), fabs(dd)));
          f = dd >= 0.0 ? f : -f;
          double2 te = cscale(g, f);
          const double c = rsqrt_newton(1.0 + cabs2(te));
          te = cscale(te, c);
          const double2 tm = make_double2(-te.x, te.y);   // c te, -c conj(te)
          // (the larger term last: one rounding at its size)
          auto turn = [&](double2 t, double2 y, double2 x) {
            const double2 w = cmul(t, y);
            return make_double2(fma(c, x.x, w.x), fma(c, x.y, w.y));
          };
          const double2 x = a[p], y = a[q], vx = v[p], vy = v[q];
          a[p] = turn(tm, y, x);
          a[q] = turn(te, x, y);
          v[p] = turn(tm, vy, vx);
          v[q] = turn(te, vx, vy);
        }
      }
    if (!rotated) break;
  }
  double sig2[4], smax2 = 0.0, ssum = 0.0;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    sig2[j] = row_total(cabs2(a[j]));
    if (j < d) {
      smax2 = fmax(smax2, sig2[j]);
      ssum += sig2[j] == 0.0 ? 0.0 : sqrt(sig2[j]);
    }
  }
  *nuc = ldexp(ssum, -h);
  unsigned good = 0;
#pragma unroll
  for (int j = 0; j < 4; ++j)
    if (j >= d || (smax2 > 0.0 && sig2[j] > 1e-26 * smax2)) {
      good |= 1u << j;
      a[j] = cscale(a[j], rsqrt_newton(sig2[j]));
    }
  // canonical completion of the other columns, U side (a) then V side (v)
#pragma unroll 1
  for (int side = 0; side < 2; ++side) {
    unsigned set = good;
    int next_e = 0;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
#pragma unroll 1
      for (int e0 = next_e; e0 < 4 && !((set >> j) & 1u); ++e0) {
        double2 x = make_double2(i == e0 ? 1.0 : 0.0, 0.0);
#pragma unroll 1
        for (int pass = 0; pass < 2; ++pass)
#pragma unroll
          for (int b = 0; b < 4; ++b)
            if ((set >> b) & 1u) x = csub(x, cmul(a[b], dot(a[b], x)));
        const double nr2 = row_total(cabs2(x));
        if (nr2 > 0.25) {
          a[j] = cscale(x, rsqrt_newton(nr2));
          set |= 1u << j;
          next_e = e0 + 1;
        }
      }
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) {   // the other side's turn
      const double2 t = a[j];
      a[j] = v[j];
      v[j] = t;
    }
  }
  // out = U V^H (the d x d block)
  double2 o[4];
  auto entry = [&](auto bcast) {
    double2 t = cz();
#pragma unroll
    for (int m = 0; m < 4; ++m) t = cfma(a[m], cconj(bcast(v[m])), t);
    return t;
  };
  o[0] = entry([](double2 t) { return quad_bcast2<0>(t); });
  o[1] = entry([](double2 t) { return quad_bcast2<1>(t); });
  o[2] = entry([](double2 t) { return quad_bcast2<2>(t); });
  o[3] = entry([](double2 t) { return quad_bcast2<3>(t); });
  if (lane < 4)
#pragma unroll
    for (int j = 0; j < 4; ++j) out[4 * i + j] = i < d && j < d ? make_double2(o[j].x, sgn * o[j].y) : cz();
}

// The update of one gate on one wave: g_new = conj(polar(E)), d x d block of
// the 4 x 4 es, and zero outside it.  With omega_m1 = omega - 1 != 0 the
// over-relaxed update (no reference counterpart): g becomes
//   polar(g + omega_m1 (g - g_old)),
// a step past the local optimum along the direction of the update, projected
// back onto the unitaries.  es, g_old, rm (scratch) and g_new hold 16 entries
// each in LDS and are used by this wave alone until the caller's barrier.
// Returns the overlap after the update, the sum of E's singular values or
// |sum_{o,i} g[o][i] E[o][i]| (on every lane), if wanted.
QMX_DEV double update_gate_wave(int d, double omega_m1, const double2* g_old, const double2* es, double2* rm,
                                double2* g_new, int lane, bool want) {
  const int l = lane & 15;
  const int rounds = omega_m1 != 0.0 ? 2 : 1;
  const double2* m = es;
  double nuc = 0.0;
  for (int r = 0; r < rounds; ++r) {
    const double sgn = r == 0 ? -1.0 : 1.0;
    __builtin_amdgcn_wave_barrier();
    if (!polar4_wave(d, m, g_new, sgn, lane, want, &nuc)) {
      // zero or ill-conditioned matrices, and whatever else it declined
      polar4_jacobi(d, m, g_new, sgn, lane, &nuc);
    }
    __builtin_amdgcn_wave_barrier();
    if (r + 1 < rounds) {
      const bool in = (l >> 2) < d && (l & 3) < d;
      const double2 g = g_new[l];
      if (lane < 16) rm[l] = in ? cadd(g, cscale(csub(g, g_old[l]), omega_m1)) : cz();
      m = rm;
    }
  }
  if (rounds > 1 && want) {
    const double2 p = cmul(g_new[l], es[l]);
    const double re = sum16(p.x), im = sum16(p.y);
    nuc = sqrt(re * re + im * im);
  }
  return nuc;
}

// --------------------------------------------- Householder null space -----
// Trailing columns of the full Householder QR of rows^T (n x m, n <= 4,
// m < n), LAPACK zgeqr2 + zung2r conventions.  rows is m x n (stride 4).
// Writes q (n x n, stride 4); the null space is q[:, m:].
QMX_DEV void householder_q(int m, int n, const double2* rows, double2* q) {
  double2 a[16];
  for (int i = 0; i < n; ++i)
    for (int j = 0; j < m; ++j) a[i * 4 + j] = rows[j * 4 + i];
  double2 vs[4][4];
  double2 taus[4];
  for (int j = 0; j < m; ++j) {
    double2 alpha = a[j * 4 + j];
    double xn2 = 0.0;
    for (int i = j + 1; i < n; ++i) xn2 += cabs2(a[i * 4 + j]);
    double2 vv[4];
    for (int i = 0; i < 4; ++i) vv[i] = cz();
    vv[0] = make_double2(1.0, 0.0);
    double2 tau;
    if (xn2 == 0.0 && alpha.y == 0.0) {
      tau = cz();
    } else {
      double nrm = sqrt(alpha.x * alpha.x + alpha.y * alpha.y + xn2);
      double beta = signbit(alpha.x) ? nrm : -nrm;   // -sign(Re alpha) * norm
      tau = make_double2((beta - alpha.x) / beta, -alpha.y / beta);
      // scale = 1 / (alpha - beta)
      double2 den = make_double2(alpha.x - beta, alpha.y);
      double dd = cabs2(den);
      double2 scale = make_double2(den.x / dd, -den.y / dd);
      for (int i = j + 1; i < n; ++i) vv[i - j] = cmul(a[i * 4 + j], scale);
      a[j * 4 + j] = make_double2(beta, 0.0);
      for (int i = j + 1; i < n; ++i) a[i * 4 + j] = cz();
    }
    // apply H^H = I - conj(tau) v v^H to trailing columns
    for (int c = j + 1; c < m; ++c) {
      double2 w = cz();
      for (int i = j; i < n; ++i) w = cfmac(vv[i - j], a[i * 4 + c], w);
      double2 f = cmul(cconj(tau), w);
      for (int i = j; i < n; ++i) a[i * 4 + c] = csub(a[i * 4 + c], cmul(vv[i - j], f));
    }
    for (int i = 0; i < 4; ++i) vs[j][i] = vv[i];
    taus[j] = tau;
  }
  for (int i = 0; i < 4; ++i)
    for (int j = 0; j < 4; ++j) q[i * 4 + j] = make_double2(i == j ? 1.0 : 0.0, 0.0);
  for (int j = m - 1; j >= 0; --j) {
    // q[j:, :] -= tau v (v^H q[j:, :])
    for (int c = 0; c < n; ++c) {
      double2 w = cz();
      for (int i = j; i < n; ++i) w = cfmac(vs[j][i - j], q[i * 4 + c], w);
      double2 f = cmul(taus[j], w);
      for (int i = j; i < n; ++i) q[i * 4 + c] = csub(q[i * 4 + c], cmul(vs[j][i - j], f));
    }
  }
}

// ----------------------------------------------------------- bit helpers --
// Insert a zero bit at position pos of x.
QMX_DEV uint64_t insert_zero(uint64_t x, int pos) {
  uint64_t lo = x & ((1ull << pos) - 1ull);
  return ((x >> pos) << (pos + 1)) | lo;
}
