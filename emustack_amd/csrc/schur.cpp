// Schur form of a complex upper Hessenberg matrix on the host: the projected
// problem of the Krylov eigensolver (65 to 504 rows, once per instance and
// restart).
//
// Small-bulge multishift QR with aggressive early deflation (Braman, Byers and
// Mathias, SIAM J. Matrix Anal. Appl. 23 (2002) 929 and 948).  A train of
// single-shift bulges two rows apart moves down the active block one row per
// step.  The row pairs of one step are disjoint and contiguous in a column, so
// the step's left rotations are vectors down each column, and its right
// rotations vectors down each pair of columns.  Only the window that the train
// covers in the next kStep steps is touched step by step; the columns right of
// it, the rows above it and the Schur vectors take the recorded rotations
// afterwards, strip by strip from the first-level cache.  The deflation
// criterion, the shifts and the exchange of eigenvalues are from the papers and
// the book named at each; windows, trains and their limits are measured here.
// Measured on one core (QR iteration with vectors; zgees without its Hessenberg
// reduction in brackets): 65 rows 0.37 ms (2.0), 90 rows 0.77 (3.9), 176 rows
// 3.8 (12.5), 440 rows 36 (95).
#include "schur.h"

#include <algorithm>
#include <cmath>
#include <cstring>
#include <limits>
#include <vector>

#if defined(__x86_64__)
#include <immintrin.h>
#endif

namespace emu {

#if defined(__x86_64__)
#pragma clang attribute push(__attribute__((target("avx512f,avx512dq,avx512vl,fma"))), apply_to = function)

namespace {
typedef std::complex<double> cplx;
const double kUlp = std::numeric_limits<double>::epsilon();
const double kFloor = std::numeric_limits<double>::min() / kUlp;
const int kMaxShifts = 48;  // bulges in one train
const int kStep = 32;       // steps of a train between two far updates

inline double abs1(cplx z) { return std::fabs(z.real()) + std::fabs(z.imag()); }
inline cplx mul(cplx a, cplx b) {
  return cplx(a.real() * b.real() - a.imag() * b.imag(), a.real() * b.imag() + a.imag() * b.real());
}

// [c s; -conj(s) c] [a; b] = [r; 0]: c = |a|^2 / d, s = a conj(b) / d, r = a (|a|^2 + |b|^2) / d with
// d = |a| sqrt(|a|^2 + |b|^2), one square root and one division
inline void rotation(cplx a, cplx b, double &c, cplx &s, cplx &r) {
  double a2 = a.real() * a.real() + a.imag() * a.imag();
  double b2 = b.real() * b.real() + b.imag() * b.imag();
  double h2 = a2 + b2;
  if (a2 > 1e-140 && h2 < 1e140) {
    const double q = 1.0 / std::sqrt(a2 * h2);
    const double c0 = a2 * q, sr = (a.real() * b.real() + a.imag() * b.imag()) * q,
                 si = (a.imag() * b.real() - a.real() * b.imag()) * q;
    // a rotation meets every row and column, so the rounding of its length
    // adds up in one direction: one Newton step for c^2 + |s|^2 = 1 (backward
    // error of the Schur form at 176 rows 0.8 -> 0.2 e-14, LAPACK 0.5 e-14)
    const double e = 0.5 * std::fma(-si, si, std::fma(-sr, sr, std::fma(-c0, c0, 1.0)));
    c = c0 + c0 * e;
    s = cplx(sr + sr * e, si + si * e);
    r = a * (h2 * q);
    return;
  }
  // far from 1 in size: each phase from its number scaled by a power of two (the
  // smallest numbers have no digits left for a quotient of modulus one)
  const double ma = std::max(std::fabs(a.real()), std::fabs(a.imag()));
  const double mb = std::max(std::fabs(b.real()), std::fabs(b.imag()));
  if (!(mb > 0)) {
    c = 1;
    s = 0;
    r = a;
    return;
  }
  const int ea = ma > 0 ? std::ilogb(ma) : 0, eb = std::ilogb(mb), e0 = ma > 0 ? std::max(ea, eb) : eb;
  const cplx sa(std::ldexp(a.real(), -ea), std::ldexp(a.imag(), -ea));
  const cplx sb(std::ldexp(b.real(), -eb), std::ldexp(b.imag(), -eb));
  const double ha = std::hypot(sa.real(), sa.imag()), hb = std::hypot(sb.real(), sb.imag());
  const cplx pa = ma > 0 ? cplx(sa.real() / ha, sa.imag() / ha) : cplx(1);
  const cplx pb(sb.real() / hb, -sb.imag() / hb);
  const double ar = ma > 0 ? std::ldexp(ha, ea - e0) : 0.0, br = std::ldexp(hb, eb - e0), n = std::hypot(ar, br);
  c = ar / n;
  s = mul(pa, pb) * (br / n);
  r = pa * std::ldexp(n, e0);
}

// columns x, y (m complex values): [x y] <- [x y] [c, -s; conj(s), c]
inline void rot_cols(int m, double *x, double *y, double c, cplx s) {
  const __m512d C = _mm512_set1_pd(c), SR = _mm512_set1_pd(s.real());
  const __m512d SI = _mm512_setr_pd(s.imag(), -s.imag(), s.imag(), -s.imag(), s.imag(), -s.imag(), s.imag(),
                                    -s.imag());
  int i = 0;
  for (; i + 4 <= m; i += 4) {
    const __m512d a = _mm512_loadu_pd(x + 2 * i), b = _mm512_loadu_pd(y + 2 * i);
    const __m512d ap = _mm512_permute_pd(a, 0x55), bp = _mm512_permute_pd(b, 0x55);
    _mm512_storeu_pd(x + 2 * i, _mm512_fmadd_pd(SI, bp, _mm512_fmadd_pd(SR, b, _mm512_mul_pd(C, a))));
    _mm512_storeu_pd(y + 2 * i, _mm512_fmadd_pd(SI, ap, _mm512_fnmadd_pd(SR, a, _mm512_mul_pd(C, b))));
  }
  if (i < m) {
    const __mmask8 k = (__mmask8)((1u << (2 * (m - i))) - 1);
    const __m512d a = _mm512_maskz_loadu_pd(k, x + 2 * i), b = _mm512_maskz_loadu_pd(k, y + 2 * i);
    const __m512d ap = _mm512_permute_pd(a, 0x55), bp = _mm512_permute_pd(b, 0x55);
    _mm512_mask_storeu_pd(x + 2 * i, k, _mm512_fmadd_pd(SI, bp, _mm512_fmadd_pd(SR, b, _mm512_mul_pd(C, a))));
    _mm512_mask_storeu_pd(y + 2 * i, k, _mm512_fmadd_pd(SI, ap, _mm512_fnmadd_pd(SR, a, _mm512_mul_pd(C, b))));
  }
}

// rows p, p + 1 of columns j0..j1-1
inline void rot_rows(double *h, int ld, int p, int j0, int j1, double c, cplx s) {
  const double r = s.real(), i = s.imag();
  const __m256d C = _mm256_set1_pd(c), SR = _mm256_setr_pd(r, r, -r, -r), SI = _mm256_setr_pd(-i, i, -i, i);
  double *x = h + 2 * ((size_t)j0 * ld + p);
  for (int j = j0; j < j1; ++j, x += 2 * (size_t)ld) {
    const __m256d a = _mm256_loadu_pd(x);
    const __m256d y = _mm256_permute4x64_pd(a, 0x4e), z = _mm256_permute4x64_pd(a, 0x1b);
    _mm256_storeu_pd(x, _mm256_fmadd_pd(SI, z, _mm256_fmadd_pd(SR, y, _mm256_mul_pd(C, a))));
  }
}

// One step of a train as vectors down a column: two bulges (four complex rows)
// each, the lowest rows first.
struct Step {
  int row, cnt;  // rows row .. row + 2 cnt - 1
  double cf[(kMaxShifts / 2) * 24];  // per two bulges: C, SR, SI
  void set(int i, double c, cplx s) {  // pair i: rows row + 2 i, row + 2 i + 1
    double *q = cf + (i / 2) * 24 + (i % 2) * 4;
    q[0] = q[1] = q[2] = q[3] = c;
    q[8] = q[9] = s.real();
    q[10] = q[11] = -s.real();
    q[16] = q[18] = -s.imag();
    q[17] = q[19] = s.imag();
  }
};

const int kPath = 64;  // rotations of a path

// A chain of rotations in a window: columns p, p + 1, then p + 1, p + 2, ...
// (dir = 1, a bulge), or p - 1, p, ... (dir = -1, an eigenvalue on its way up)
struct Path {
  int p, cnt, dir;
  double c[kPath], sr[kPath], si[kPath];
  void add(double cc, cplx s) {
    c[cnt] = cc;
    sr[cnt] = s.real();
    si[cnt++] = s.imag();
  }
};

// A strip of eight values per column (buf, two vectors a column) through the
// paths of a window, path by path: a bulge never meets a column that an
// earlier one has still to reach, so the order across bulges is free, and the
// column that two successive rotations share stays in registers.
// sign = 1: right rotations; -1: left rotations on a transposed strip.
inline void strip_paths(const Path *pt, int npt, int base, double sign, double *buf) {
  const __m512d alt = _mm512_setr_pd(sign, -sign, sign, -sign, sign, -sign, sign, -sign);
  for (int b = 0; b < npt; ++b) {
    const Path &q = pt[b];
    if (q.cnt == 0) continue;
    double *x = buf + 16 * (q.p - base);
    if (q.dir < 0) {
      __m512d y = _mm512_load_pd(x + 16), f = _mm512_load_pd(x + 24);
      for (int i = 0; i < q.cnt; ++i, x -= 16) {
        const __m512d C = _mm512_set1_pd(q.c[i]), SR = _mm512_set1_pd(q.sr[i]);
        const __m512d SI = _mm512_mul_pd(alt, _mm512_set1_pd(q.si[i]));
        const __m512d a = _mm512_load_pd(x), e = _mm512_load_pd(x + 8);
        const __m512d ap = _mm512_permute_pd(a, 0x55), yp = _mm512_permute_pd(y, 0x55);
        const __m512d ep = _mm512_permute_pd(e, 0x55), fp = _mm512_permute_pd(f, 0x55);
        _mm512_store_pd(x + 16, _mm512_fmadd_pd(SI, ap, _mm512_fnmadd_pd(SR, a, _mm512_mul_pd(C, y))));
        _mm512_store_pd(x + 24, _mm512_fmadd_pd(SI, ep, _mm512_fnmadd_pd(SR, e, _mm512_mul_pd(C, f))));
        y = _mm512_fmadd_pd(SI, yp, _mm512_fmadd_pd(SR, y, _mm512_mul_pd(C, a)));
        f = _mm512_fmadd_pd(SI, fp, _mm512_fmadd_pd(SR, f, _mm512_mul_pd(C, e)));
      }
      _mm512_store_pd(x + 16, y);
      _mm512_store_pd(x + 24, f);
      continue;
    }
    __m512d a = _mm512_load_pd(x), e = _mm512_load_pd(x + 8);
    for (int i = 0; i < q.cnt; ++i, x += 16) {
      const __m512d C = _mm512_set1_pd(q.c[i]), SR = _mm512_set1_pd(q.sr[i]);
      const __m512d SI = _mm512_mul_pd(alt, _mm512_set1_pd(q.si[i]));
      const __m512d y = _mm512_load_pd(x + 16), f = _mm512_load_pd(x + 24);
      const __m512d ap = _mm512_permute_pd(a, 0x55), yp = _mm512_permute_pd(y, 0x55);
      const __m512d ep = _mm512_permute_pd(e, 0x55), fp = _mm512_permute_pd(f, 0x55);
      _mm512_store_pd(x, _mm512_fmadd_pd(SI, yp, _mm512_fmadd_pd(SR, y, _mm512_mul_pd(C, a))));
      _mm512_store_pd(x + 8, _mm512_fmadd_pd(SI, fp, _mm512_fmadd_pd(SR, f, _mm512_mul_pd(C, e))));
      a = _mm512_fmadd_pd(SI, ap, _mm512_fnmadd_pd(SR, a, _mm512_mul_pd(C, y)));
      e = _mm512_fmadd_pd(SI, ep, _mm512_fnmadd_pd(SR, e, _mm512_mul_pd(C, f)));
    }
    _mm512_store_pd(x, a);
    _mm512_store_pd(x + 8, e);
  }
}

// the window's rotations from the right on rows r0..r1-1 (columns wa..wb are theirs)
inline void far_right(const Path *pt, int npt, double *h, int ld, int wa, int wb, int r0, int r1, double *buf) {
  for (int r = r0; r < r1; r += 8) {
    const int m = std::min(8, r1 - r);
    const __mmask8 k0 = (__mmask8)(m >= 4 ? 0xff : (1u << (2 * m)) - 1);
    const __mmask8 k1 = (__mmask8)(m >= 8 ? 0xff : m > 4 ? (1u << (2 * (m - 4))) - 1 : 0);
    double *x = h + 2 * ((size_t)wa * ld + r);
    for (int j = 0; j <= wb - wa; ++j) {
      _mm512_store_pd(buf + 16 * j, _mm512_maskz_loadu_pd(k0, x + 2 * (size_t)j * ld));
      _mm512_store_pd(buf + 16 * j + 8, _mm512_maskz_loadu_pd(k1, x + 2 * (size_t)j * ld + 8));
    }
    strip_paths(pt, npt, wa, 1.0, buf);
    for (int j = 0; j <= wb - wa; ++j) {
      _mm512_mask_storeu_pd(x + 2 * (size_t)j * ld, k0, _mm512_load_pd(buf + 16 * j));
      _mm512_mask_storeu_pd(x + 2 * (size_t)j * ld + 8, k1, _mm512_load_pd(buf + 16 * j + 8));
    }
  }
}

// and from the left on columns j0..j1-1 (rows wa..wb)
inline void far_left(const Path *pt, int npt, double *h, int ld, int wa, int wb, int j0, int j1, double *buf) {
  for (int j = j0; j < j1; j += 8) {
    const int m = std::min(8, j1 - j);
    for (int k = 0; k < m; ++k) {
      const double *x = h + 2 * ((size_t)(j + k) * ld + wa);
      for (int i = 0; i <= wb - wa; ++i) _mm_store_pd(buf + 16 * i + 2 * k, _mm_loadu_pd(x + 2 * i));
    }
    strip_paths(pt, npt, wa, -1.0, buf);
    for (int k = 0; k < m; ++k) {
      double *x = h + 2 * ((size_t)(j + k) * ld + wa);
      for (int i = 0; i <= wb - wa; ++i) _mm_storeu_pd(x + 2 * i, _mm_load_pd(buf + 16 * i + 2 * k));
    }
  }
}

// x (rows x w, leading dimension ld) <- x V (w x w, leading dimension w)
void mul_right(double *x, int ld, int rows, int w, const double *v, double *tmp) {
  const __m512d one = _mm512_set1_pd(1.0);
  for (int r = 0; r < rows; r += 8) {
    const int m = std::min(8, rows - r);
    const __mmask8 k0 = (__mmask8)(m >= 4 ? 0xff : (1u << (2 * m)) - 1);
    const __mmask8 k1 = (__mmask8)(m >= 8 ? 0xff : m > 4 ? (1u << (2 * (m - 4))) - 1 : 0);
    for (int k = 0; k < w; ++k) {
      const double *q = x + 2 * ((size_t)k * ld + r);
      _mm512_storeu_pd(tmp + 16 * k, _mm512_maskz_loadu_pd(k0, q));
      _mm512_storeu_pd(tmp + 16 * k + 8, _mm512_maskz_loadu_pd(k1, q + 8));
    }
    for (int j = 0; j < w; j += 4) {
      const int nj = std::min(4, w - j);
      __m512d re[4][2], im[4][2];
      for (int b = 0; b < 4; ++b) re[b][0] = re[b][1] = im[b][0] = im[b][1] = _mm512_setzero_pd();
      const double *vj[4];
      for (int b = 0; b < 4; ++b) vj[b] = v + 2 * (size_t)(j + std::min(b, nj - 1)) * w;
      for (int k = 0; k < w; ++k) {
        const __m512d a = _mm512_loadu_pd(tmp + 16 * k), e = _mm512_loadu_pd(tmp + 16 * k + 8);
#pragma unroll
        for (int b = 0; b < 4; ++b) {
          const __m512d vr = _mm512_set1_pd(vj[b][2 * k]), vi = _mm512_set1_pd(vj[b][2 * k + 1]);
          re[b][0] = _mm512_fmadd_pd(a, vr, re[b][0]);
          re[b][1] = _mm512_fmadd_pd(e, vr, re[b][1]);
          im[b][0] = _mm512_fmadd_pd(a, vi, im[b][0]);
          im[b][1] = _mm512_fmadd_pd(e, vi, im[b][1]);
        }
      }
      for (int b = 0; b < nj; ++b) {
        double *q = x + 2 * ((size_t)(j + b) * ld + r);
        _mm512_mask_storeu_pd(q, k0, _mm512_fmaddsub_pd(one, re[b][0], _mm512_permute_pd(im[b][0], 0x55)));
        _mm512_mask_storeu_pd(q + 8, k1, _mm512_fmaddsub_pd(one, re[b][1], _mm512_permute_pd(im[b][1], 0x55)));
      }
    }
  }
}

// x (w x cols) <- V^H x; vh = V^H with leading dimension ldv (a multiple of 8, zero rows below w)
void mul_left(double *x, int ld, int cols, int w, const double *vh, int ldv) {
  const __m512d one = _mm512_set1_pd(1.0);
  double out[4][2 * 128];
  for (int c = 0; c < cols; c += 4) {
    const int nc = std::min(4, cols - c);
    const double *xc[4];
    for (int b = 0; b < 4; ++b) xc[b] = x + 2 * (size_t)(c + std::min(b, nc - 1)) * ld;
    for (int r = 0; r < w; r += 8) {
      __m512d re[4][2], im[4][2];
      for (int b = 0; b < 4; ++b) re[b][0] = re[b][1] = im[b][0] = im[b][1] = _mm512_setzero_pd();
      const double *q = vh + 2 * r;
      for (int k = 0; k < w; ++k, q += 2 * ldv) {
        const __m512d a = _mm512_loadu_pd(q), e = _mm512_loadu_pd(q + 8);
#pragma unroll
        for (int b = 0; b < 4; ++b) {
          const __m512d vr = _mm512_set1_pd(xc[b][2 * k]), vi = _mm512_set1_pd(xc[b][2 * k + 1]);
          re[b][0] = _mm512_fmadd_pd(a, vr, re[b][0]);
          re[b][1] = _mm512_fmadd_pd(e, vr, re[b][1]);
          im[b][0] = _mm512_fmadd_pd(a, vi, im[b][0]);
          im[b][1] = _mm512_fmadd_pd(e, vi, im[b][1]);
        }
      }
      for (int b = 0; b < 4; ++b) {
        _mm512_storeu_pd(out[b] + 2 * r, _mm512_fmaddsub_pd(one, re[b][0], _mm512_permute_pd(im[b][0], 0x55)));
        _mm512_storeu_pd(out[b] + 2 * r + 8, _mm512_fmaddsub_pd(one, re[b][1], _mm512_permute_pd(im[b][1], 0x55)));
      }
    }
    for (int b = 0; b < nc; ++b) std::memcpy(x + 2 * (size_t)(c + b) * ld, out[b], sizeof(double) * 2 * w);
  }
}

struct Mat {
  cplx *a;
  int ld;
  cplx &operator()(int i, int j) const { return a[i + (size_t)j * ld]; }
  double *d() const { return reinterpret_cast<double *>(a); }
  double *col(int i, int j) const { return reinterpret_cast<double *>(a + i + (size_t)j * ld); }
};

// May the subdiagonal entry c = h(k, k - 1) go?  [a b; c d] is the 2 x 2 diagonal block that it holds together.
// Beside a and d it has to be rounding, and without it the block's eigenvalues move by about b c / (a - d), which
// has to be rounding beside d: so the small eigenvalues of a graded matrix stay (the criterion of Ahues and
// Tisseur, A new deflation criterion for the QR algorithm, 1997).  Below kFloor a product with kUlp is no longer a
// normal number, and the entry goes in any case.
bool negligible(const Mat &h, int k) {
  const double c = abs1(h(k, k - 1));
  if (c <= kFloor) return true;
  const cplx a = h(k - 1, k - 1), d = h(k, k);
  return c <= kUlp * (abs1(a) + abs1(d)) && c * abs1(h(k - 1, k)) <= kUlp * abs1(d) * abs1(a - d);
}

// first row of the active block that ends at hi; the negligible entry above it becomes zero
int split(const Mat &h, int hi) {
  int lo = hi;
  while (lo > 0 && !negligible(h, lo)) --lo;
  if (lo > 0) h(lo, lo - 1) = 0;
  return lo;
}

// Wilkinson's shift: the eigenvalue of [a b; c d] nearer to d, d - b c / (x + r) with x = (a - d) / 2 and
// r = +-sqrt(x^2 + b c), the root that does not cancel
inline cplx wilkinson(cplx a, cplx bc, cplx d) {
  const cplx x = 0.5 * (a - d), r = std::sqrt(mul(x, x) + bc);
  const cplx den = x.real() * r.real() + x.imag() * r.imag() < 0 ? x - r : x + r;
  return abs1(den) > 0 ? d - bc / den : d;
}

// A shift for a block that has stalled: off the diagonal entry by the size of the two subdiagonal entries before
// it (Martin, Peters and Wilkinson, Numer. Math. 14 (1970) 219)
inline cplx stall_shift(const Mat &h, int lo, int k) {
  double t = abs1(h(k, k - 1));
  if (k - 1 > lo) t += abs1(h(k - 1, k - 2));
  return h(k, k) + t;
}

// single-shift QR of a small matrix, rotation by rotation
bool qr_small(int n, const Mat &h, const Mat &z, int nz) {
  int steps = 0;  // since the last deflation
  for (int hi = n - 1; hi >= 0;) {
    const int lo = split(h, hi);
    if (lo == hi) {
      --hi;
      steps = 0;
      continue;
    }
    if (++steps > 48) return false;
    const cplx sh = steps % 8 ? wilkinson(h(hi - 1, hi - 1), mul(h(hi - 1, hi), h(hi, hi - 1)), h(hi, hi))
                              : stall_shift(h, lo, hi);
    for (int p = lo; p < hi; ++p) {
      double c;
      cplx s, r;
      if (p == lo) {
        rotation(h(lo, lo) - sh, h(lo + 1, lo), c, s, r);
      } else {
        rotation(h(p, p - 1), h(p + 1, p - 1), c, s, r);
        h(p, p - 1) = r;
        h(p + 1, p - 1) = 0;
      }
      rot_rows(h.d(), h.ld, p, p, n, c, s);
      rot_cols(std::min(p + 2, hi) + 1, h.col(0, p), h.col(0, p + 1), c, s);
      if (nz) rot_cols(nz, z.col(0, p), z.col(0, p + 1), c, s);
    }
  }
  return true;
}

// exchange of the diagonal entries k, k + 1 of the upper triangular t, in its
// rows r0.. and columns ..n-1: the rotation that turns (t12, t22 - t11), the
// eigenvector of t22, onto the first axis (Golub and Van Loan, Matrix
// Computations, 7.6.2)
void swap_diag(int r0, int n, const Mat &t, int k, double &c, cplx &s) {
  const cplx t1 = t(k, k), t2 = t(k + 1, k + 1);
  cplx r;
  rotation(t(k, k + 1), t2 - t1, c, s, r);
  rot_rows(t.d(), t.ld, k, k + 2, n, c, s);
  rot_cols(k - r0, t.col(r0, k), t.col(r0, k + 1), c, s);
  t(k, k) = t2;
  t(k + 1, k + 1) = t1;
}

struct Work {
  std::vector<Path> paths;
  std::vector<cplx> t, v, vh, strip;
  std::vector<cplx> shifts;
};

bool qr(int n, const Mat &h, const Mat &z, int nz, std::vector<Work> &work, int depth);

// Householder vector of x[0..n-1]: (I - tau w w^H) x = beta e1, w[0] = 1
void reflector(int n, const cplx *x, cplx *w, double &tau, cplx &beta) {
  double top = 0;
  for (int i = 0; i < n; ++i) top = std::max(top, std::max(std::fabs(x[i].real()), std::fabs(x[i].imag())));
  // numbers whose squares lose digits are scaled by a power of two
  const int e = top > 0 && (top < 1e-130 || top > 1e130) ? std::ilogb(top) : 0;
  auto at = [&](int i) { return e ? cplx(std::ldexp(x[i].real(), -e), std::ldexp(x[i].imag(), -e)) : x[i]; };
  double nr = 0;
  for (int i = 1; i < n; ++i) nr += std::norm(at(i));
  w[0] = 1;
  if (nr == 0) {
    tau = 0;
    beta = x[0];
    for (int i = 1; i < n; ++i) w[i] = 0;
    return;
  }
  const cplx x0 = at(0);
  const double a0 = std::abs(x0), nm = std::sqrt(nr + a0 * a0);
  const cplx ph = a0 > 1e-280 ? x0 / a0 : cplx(1);  // smaller ones have no digits for a phase
  beta = -ph * nm;
  const cplx u0 = x0 - beta;  // |u0| = a0 + nm: no cancellation
  for (int i = 1; i < n; ++i) w[i] = at(i) / u0;
  if (e) beta = cplx(std::ldexp(beta.real(), e), std::ldexp(beta.imag(), e));
  tau = (a0 + nm) / nm;  // 2 |u0|^2 / ||u||^2
}

inline __mmask8 tail(int m) { return (__mmask8)(m >= 4 ? 0xff : (1u << (2 * m)) - 1); }
inline double sum_even_minus(__m512d v) {  // odd lanes minus even lanes
  return _mm512_reduce_add_pd(_mm512_mask_sub_pd(v, 0x55, _mm512_setzero_pd(), v));
}

// rows r0..r0+n-1, columns j0..j1-1: x <- (I - tau w w^H) x, tau real
void reflect_left(const Mat &a, int r0, int n, int j0, int j1, const cplx *wv, double tau) {
  const double *w = reinterpret_cast<const double *>(wv);
  for (int j = j0; j < j1; j += 4) {
    const int nc = std::min(4, j1 - j);
    double *x[4];
    for (int b = 0; b < 4; ++b) x[b] = a.col(r0, j + std::min(b, nc - 1));
    __m512d p[4], q[4];
    for (int b = 0; b < 4; ++b) p[b] = q[b] = _mm512_setzero_pd();
    for (int i = 0; i < n; i += 4) {
      const __mmask8 k = tail(n - i);
      const __m512d u = _mm512_maskz_loadu_pd(k, w + 2 * i), us = _mm512_permute_pd(u, 0x55);
#pragma unroll
      for (int b = 0; b < 4; ++b) {
        const __m512d v = _mm512_maskz_loadu_pd(k, x[b] + 2 * i);
        p[b] = _mm512_fmadd_pd(u, v, p[b]);
        q[b] = _mm512_fmadd_pd(us, v, q[b]);
      }
    }
    __m512d dr[4], di[4];
    for (int b = 0; b < 4; ++b) {
      const double im = tau * sum_even_minus(q[b]);
      dr[b] = _mm512_set1_pd(tau * _mm512_reduce_add_pd(p[b]));
      di[b] = _mm512_setr_pd(-im, im, -im, im, -im, im, -im, im);
    }
    for (int i = 0; i < n; i += 4) {
      const __mmask8 k = tail(n - i);
      const __m512d u = _mm512_maskz_loadu_pd(k, w + 2 * i), us = _mm512_permute_pd(u, 0x55);
#pragma unroll
      for (int b = 0; b < 4; ++b) {
        if (b >= nc) break;
        const __m512d v = _mm512_maskz_loadu_pd(k, x[b] + 2 * i);
        _mm512_mask_storeu_pd(x[b] + 2 * i, k, _mm512_fnmadd_pd(us, di[b], _mm512_fnmadd_pd(u, dr[b], v)));
      }
    }
  }
}

// columns c0..c0+n-1, rows 0..m-1: a <- a (I - tau w w^H), tau real
void reflect_right(const Mat &a, int c0, int n, int m, const cplx *wv, double tau) {
  for (int r = 0; r < m; r += 16) {  // strips of sixteen rows: y = a w
    __m512d p[4], q[4];
    __mmask8 k[4];
    for (int b = 0; b < 4; ++b) {
      p[b] = q[b] = _mm512_setzero_pd();
      k[b] = m - r - 4 * b > 0 ? tail(m - r - 4 * b) : 0;
    }
    for (int c = 0; c < n; ++c) {
      const double *x = a.col(r, c0 + c);
      const __m512d wr = _mm512_set1_pd(wv[c].real()), wi = _mm512_set1_pd(wv[c].imag());
#pragma unroll
      for (int b = 0; b < 4; ++b) {
        const __m512d v = _mm512_maskz_loadu_pd(k[b], x + 8 * b);
        p[b] = _mm512_fmadd_pd(v, wr, p[b]);
        q[b] = _mm512_fmadd_pd(v, wi, q[b]);
      }
    }
    const __m512d t = _mm512_set1_pd(tau), one = _mm512_set1_pd(1.0);
    for (int b = 0; b < 4; ++b)
      p[b] = _mm512_mul_pd(t, _mm512_fmaddsub_pd(one, p[b], _mm512_permute_pd(q[b], 0x55)));
    for (int b = 0; b < 4; ++b) q[b] = _mm512_permute_pd(p[b], 0x55);
    for (int c = 0; c < n; ++c) {  // a -= y conj(w_c)
      double *x = a.col(r, c0 + c);
      const double wi = wv[c].imag();
      const __m512d wr = _mm512_set1_pd(wv[c].real());
      const __m512d ws = _mm512_setr_pd(wi, -wi, wi, -wi, wi, -wi, wi, -wi);
#pragma unroll
      for (int b = 0; b < 4; ++b) {
        const __m512d v = _mm512_maskz_loadu_pd(k[b], x + 8 * b);
        _mm512_mask_storeu_pd(x + 8 * b, k[b], _mm512_fnmadd_pd(q[b], ws, _mm512_fnmadd_pd(p[b], wr, v)));
      }
    }
  }
}

// Aggressive early deflation in the last nw rows of the active block lo..hi
// (the second of the two papers): the window's Schur form T = V^H W V turns the
// entry s0 to its left into a spike s0 V(0, :)^H, and an eigenvalue whose spike
// entry is rounding beside it has converged.  The entry is only that while the
// eigenvalue is the last one, so each one that has not converged makes way to
// the others that have not, at the top.  Returns the number of eigenvalues
// deflated; wk.shifts takes the others'.
int deflate(int n, const Mat &h, const Mat &z, int nz, int lo, int hi, int nw, std::vector<Work> &work, int depth) {
  Work &wk = work[depth];
  const int kw = hi - nw + 1;
  const cplx s0 = kw > lo ? h(kw, kw - 1) : cplx(0);
  wk.t.assign((size_t)nw * nw, 0);
  wk.v.assign((size_t)nw * nw, 0);
  const Mat t{wk.t.data(), nw}, v{wk.v.data(), nw};
  for (int j = 0; j < nw; ++j) {
    for (int i = 0; i <= std::min(j + 1, nw - 1); ++i) t(i, j) = h(kw + i, kw + j);
    v(j, j) = 1;
  }
  wk.shifts.clear();
  if (!qr(nw, t, v, nw, work, depth + 1)) return -1;
  int ns = 0;  // rows 0..ns-1 stay
  if (kw > lo)
    for (int last = nw - 1; last >= ns;) {
      if (abs1(mul(s0, v(0, last))) <= std::max(kFloor, kUlp * abs1(t(last, last)))) {
        --last;
        continue;
      }
      for (int k = last - 1; k >= ns; --k) {
        double c;
        cplx s;
        swap_diag(0, nw, t, k, c, s);
        rot_cols(nw, v.col(0, k), v.col(0, k + 1), c, s);
      }
      ++ns;
    }
  for (int i = 0; i < ns; ++i) wk.shifts.push_back(t(i, i));
  if (ns == nw) return 0;
  if (ns > 0) {
    // the spike s0 V(0, :)^H back to its first entry, then Hessenberg form
    std::vector<cplx> x(nw), w(nw);
    double tau;
    cplx beta;
    for (int i = 0; i < ns; ++i) x[i] = std::conj(v(0, i));
    for (int k = -1; k < ns - 2; ++k) {
      const int r = k + 1, m = ns - r;
      if (k >= 0)
        for (int i = 0; i < m; ++i) x[i] = t(r + i, k);
      reflector(m, x.data(), w.data(), tau, beta);
      if (tau == 0.0) continue;
      reflect_left(t, r, m, std::max(k, 0), nw, w.data(), tau);
      if (k >= 0) {
        t(r, k) = beta;
        for (int i = 1; i < m; ++i) t(r + i, k) = 0;
      }
      reflect_right(t, r, m, ns, w.data(), tau);
      reflect_right(v, r, m, nw, w.data(), tau);
    }
    h(kw, kw - 1) = mul(s0, std::conj(v(0, 0)));
  } else if (kw > lo) {
    h(kw, kw - 1) = 0;
  }
  for (int j = 0; j < nw; ++j)
    for (int i = 0; i <= std::min(j + 1, nw - 1); ++i) h(kw + i, kw + j) = t(i, j);
  wk.strip.resize((size_t)8 * nw);
  mul_right(h.col(0, kw), h.ld, kw, nw, v.d(), reinterpret_cast<double *>(wk.strip.data()));
  if (nz) mul_right(z.col(0, kw), z.ld, nz, nw, v.d(), reinterpret_cast<double *>(wk.strip.data()));
  if (hi + 1 < n) {
    const int ldv = (nw + 7) & ~7;
    wk.vh.assign((size_t)ldv * nw, 0);
    for (int k = 0; k < nw; ++k)
      for (int j = 0; j < nw; ++j) wk.vh[j + (size_t)k * ldv] = std::conj(v(k, j));
    mul_left(h.col(kw, hi + 1), h.ld, n - hi - 1, nw, reinterpret_cast<double *>(wk.vh.data()), ldv);
  }
  return nw - ns;
}

// One train of bulges, one per shift, down the active block lo..hi.
void sweep(int n, const Mat &h, const Mat &z, int nz, int lo, int hi, const cplx *shift, int ns, Work &wk) {
  wk.paths.resize(ns);
  Path *pt = wk.paths.data();
  Step st;
  alignas(64) double buf[16 * (kStep + 2 * kMaxShifts + 2)];
  std::memset(buf, 0, sizeof buf);
  const int total = hi - lo + 2 * (ns - 1);
  for (int t0 = 0; t0 < total; t0 += kStep) {
    const int t1 = std::min(t0 + kStep, total);
    // bulge j is at row lo + t - 2 j in step t; the window is rows and columns wa..wb
    int wa = hi, wb = lo;
    for (int j = 0; j < ns; ++j) {
      const int ta = std::max(t0, 2 * j), tb = std::min(t1, hi - lo + 2 * j);
      pt[j].cnt = 0;
      pt[j].dir = 1;
      pt[j].p = lo + ta - 2 * j;
      if (ta >= tb) continue;
      wa = std::min(wa, pt[j].p);
      wb = std::max(wb, std::min(hi, lo + tb - 1 - 2 * j + 2));
    }
    for (int t = t0; t < t1; ++t) {
      const int j1 = std::min(ns - 1, t / 2), j0 = std::max(0, (t - (hi - 1 - lo) + 1) / 2);
      st.row = lo + t - 2 * j1;
      st.cnt = j1 - j0 + 1;
      for (int i = 0; i < st.cnt; ++i) {
        const int p = st.row + 2 * i;
        double c;
        cplx s, r;
        if (p == lo)
          rotation(h(lo, lo) - shift[j1 - i], h(lo + 1, lo), c, s, r);
        else
          rotation(h(p, p - 1), h(p + 1, p - 1), c, s, r);
        st.set(i, c, s);
        pt[j1 - i].add(c, s);
      }
      for (int i = 0; i < st.cnt; i += 2) {  // two bulges, from the lower one's first column
        const int p = st.row + 2 * i, c0 = std::max(lo, p - 1);
        const double *cf = st.cf + (i / 2) * 24;
        double *x = h.col(p, c0);
        if (i + 1 < st.cnt) {
          const __m512d C = _mm512_loadu_pd(cf), SR = _mm512_loadu_pd(cf + 8), SI = _mm512_loadu_pd(cf + 16);
          for (int j = c0; j <= wb; ++j, x += 2 * (size_t)h.ld) {
            const __m512d a = _mm512_loadu_pd(x);
            const __m512d y = _mm512_permutex_pd(a, 0x4e), w = _mm512_permutex_pd(a, 0x1b);
            _mm512_storeu_pd(x, _mm512_fmadd_pd(SI, w, _mm512_fmadd_pd(SR, y, _mm512_mul_pd(C, a))));
          }
        } else {
          rot_rows(h.d(), h.ld, p, c0, wb + 1, cf[0], cplx(cf[8], cf[17]));
        }
      }
      for (int i = 0; i < st.cnt; ++i) {
        const int p = st.row + 2 * i;
        const double *cf = st.cf + (i / 2) * 24 + (i % 2) * 4;
        if (p > lo) h(p + 1, p - 1) = 0;
        rot_cols(std::min(p + 2, hi) - wa + 1, h.col(wa, p), h.col(wa, p + 1), cf[0], cplx(cf[8], cf[17]));
      }
    }
    far_right(pt, ns, h.d(), h.ld, wa, wb, 0, wa, buf);
    far_left(pt, ns, h.d(), h.ld, wa, wb, wb + 1, n, buf);
    if (nz) far_right(pt, ns, z.d(), z.ld, wa, wb, 0, nz, buf);
  }
}

const int kSmall = 26;  // blocks that qr_small finishes

bool qr(int n, const Mat &h, const Mat &z, int nz, std::vector<Work> &work, int depth) {
  if (n <= kSmall) return qr_small(n, h, z, nz);
  if ((int)work.size() < depth + 2) return false;  // windows shrink from 96 rows to kSmall in two levels
  // bulges per train and rows of the deflation window: the fastest of 6 to 48
  // and 8 to 64 at 65, 90, 176 and 440 rows (flat around these)
  const int ns0 = n < 80 ? 8 : n < 160 ? 10 : n < 320 ? 20 : 40;
  const int nw0 = ns0;
  int hi = n - 1, idle = 0;  // idle: sweeps since the last deflation
  for (int budget = 40 * n; hi >= 0; --budget) {
    if (budget == 0) return false;
    const int lo = split(h, hi);
    if (lo == hi) {
      --hi;
      idle = 0;
      continue;
    }
    // twice as wide after every six sweeps that found nothing (wider sooner costs time and roundings: 28 to 176
    // rows 1.2 to 1.7 times as long with three)
    const int nh = hi - lo + 1;
    int nw = std::min(nw0 << std::min(idle / 6, 4), 96);
    if (nh <= kSmall || nw + 1 >= nh) nw = nh;
    if (nw == n) nw = n - 1;  // the recursion gets smaller
    const int nd = deflate(n, h, z, nz, lo, hi, nw, work, depth);
    if (nd < 0) return false;
    hi -= nd;
    idle = nd > 0 ? 0 : idle + 1;
    // a window that gave up more than a fifth of its rows is followed by another, which is cheaper than a sweep (the
    // time is flat from a sixteenth to a third, 30 to 504 rows)
    if (hi <= lo || 5 * nd > nw) continue;
    const std::vector<cplx> &found = work[depth].shifts;
    const int ns = std::min({ns0, (int)found.size(), std::max(1, (hi - lo + 1) / 3)});
    std::vector<cplx> use(found.end() - ns, found.end());
    if (idle % 5 == 4)
      for (int i = 0; i < ns; ++i) use[i] = stall_shift(h, lo, std::max(lo + 1, hi - i));
    sweep(n, h, z, nz, lo, hi, use.data(), ns, work[depth]);
  }
  return true;
}
}  // namespace

// The selected eigenvalues to the top, in their order, by exchanges of
// neighbours; again window by window, a window's rows and columns outside it
// and z taking the recorded rotations strip by strip.
static void reorder(int n, const Mat &t, const Mat &z, int nz, const int *sel) {
  alignas(64) double buf[16 * (kPath + 1)];
  std::vector<Path> paths(kPath / 2);
  std::vector<char> mark(n);
  for (int i = 0; i < n; ++i) mark[i] = sel[i] != 0;
  for (int top = 0; top < n; ++top) {
    if (mark[top]) continue;
    // the next selected rows, at most half a window of them; they travel together
    int last = top, cnt = 0;
    for (int k = top + 1; k < n && cnt < kPath / 2; ++k)
      if (mark[k]) {
        ++cnt;
        last = k;
      }
    if (cnt == 0) return;
    for (int wb = last; wb >= top;) {
      const int wa = std::max(top, wb - kPath + 1);
      int np = 0, to = wa;
      for (int k = wa; k <= wb; ++k) {
        if (!mark[k]) continue;
        if (k > to) {
          Path &q = paths[np++];
          q.p = k - 1;
          q.cnt = 0;
          q.dir = -1;
          for (int p = k - 1; p >= to; --p) {
            double c;
            cplx s;
            swap_diag(wa, wb + 1, t, p, c, s);
            q.add(c, s);
          }
          mark[k] = 0;
          mark[to] = 1;
        }
        ++to;
      }
      far_right(paths.data(), np, t.d(), t.ld, wa, wb, 0, wa, buf);
      far_left(paths.data(), np, t.d(), t.ld, wa, wb, wb + 1, n, buf);
      if (nz) far_right(paths.data(), np, z.d(), z.ld, wa, wb, 0, nz, buf);
      if (wa == top) break;
      wb = to - 1;
    }
  }
}

// A (n x n) <- H = Q^H A Q upper Hessenberg, by Householder vectors one column
// at a time; a and q stay in the second-level cache for the sizes it is for.
static void hessenberg(int n, const Mat &a, const Mat &q) {
  std::vector<cplx> w((size_t)n * n);
  std::vector<double> tau(n, 0);
  for (int k = 0; k + 2 < n; ++k) {
    const int m = n - k - 1;
    cplx *wk = &w[(size_t)k * n], beta;
    reflector(m, &a(k + 1, k), wk, tau[k], beta);
    a(k + 1, k) = beta;
    for (int i = k + 2; i < n; ++i) a(i, k) = 0;
    if (tau[k] == 0) continue;
    reflect_left(a, k + 1, m, k + 1, n, wk, tau[k]);
    reflect_right(a, k + 1, m, n, wk, tau[k]);
  }
  for (int j = 0; j < n; ++j)
    for (int i = 0; i < n; ++i) q(i, j) = i == j ? 1.0 : 0.0;
  for (int k = n - 3; k >= 0; --k)
    if (tau[k] != 0) reflect_left(q, k + 1, n - k - 1, k + 1, n, &w[(size_t)k * n], tau[k]);
}

static bool qr_entry(int n, cplx *H, int ldh, cplx *Z, int ldz, int nz) {
  std::vector<Work> work(8);
  return qr(n, Mat{H, ldh}, Mat{Z, ldz}, nz, work, 0);
}
#pragma clang attribute pop

bool schur_available() {
  return __builtin_cpu_supports("avx512f") && __builtin_cpu_supports("avx512dq") &&
         __builtin_cpu_supports("avx512vl") && __builtin_cpu_supports("fma");
}
void schur_reduce(int n, std::complex<double> *A, int lda, std::complex<double> *Q, int ldq) {
  hessenberg(n, Mat{A, lda}, Mat{Q, ldq});
}
void schur_reorder(int n, std::complex<double> *T, int ldt, std::complex<double> *Z, int ldz, int nz, const int *sel) {
  reorder(n, Mat{T, ldt}, Mat{Z, ldz}, nz, sel);
}
bool schur_hessenberg(int n, std::complex<double> *H, int ldh, std::complex<double> *Z, int ldz, int nz) {
  return qr_entry(n, H, ldh, Z, ldz, nz);
}
#else
bool schur_available() { return false; }
bool schur_hessenberg(int, std::complex<double> *, int, std::complex<double> *, int, int) { return false; }
void schur_reduce(int, std::complex<double> *, int, std::complex<double> *, int) {}
void schur_reorder(int, std::complex<double> *, int, std::complex<double> *, int, int, const int *) {}
#endif
}  // namespace emu
