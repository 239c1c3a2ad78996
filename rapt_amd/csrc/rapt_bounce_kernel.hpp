// rapt_bounce_kernel.hpp -- field-line kernels (half-bounce path, eye,
// surrogate labels, BounceCenter), shared by rapt_bounce.hip (the built-in
// field models) and the kernels that rapt_jit.hip compiles at run time for
// user-written fields.
//
// Half-bounce path length S_b on the device, the output
// step of GuidingCenter.advance (bounceperiod()/bounceresolution,
// rapt/GuidingCenter.py:443-446, 593-606).
//
// A pair of lanes carries one field line: lane 0 the half along +b, lane 1 the
// half along -b, which are independent traces of nearly the same length.
//  1. trace both halves as rapt/fieldline.py:37-105 does: chunks of length
//     ds = 1/(curvature * fieldlineresolution), each integrated by RKF45
//     (rapt/rkf.py) with tol 1e-3 forward and 1e-4 backward, hmax = ds,
//     hmin = 1e-6, stopping after the chunk whose end has |B| > Bm; a chunk
//     that fails the hmin test ends the half line without its points;
//  2. keep the points inside B <= Bm plus one beyond each mirror point
//     (rapt/flutils.py:282-293); three points use the reference's equatorial
//     formula pi sqrt(2 Bm / B'') (:295-305);
//  3. otherwise interpolate B(s) by the quadratic spline of scipy's
//     interp1d(kind='quadratic') (not-a-knot: the knots are the data midpoints
//     without the first and last), find the mirror points in the end
//     intervals, and integrate ds / sqrt(1 - B/Bm) between them.  The integral
//     uses the substitution s = (a+b)/2 - (b-a)/2 cos(theta), which removes
//     the inverse-square-root end-point singularities, and 32 panels of
//     16-point Gauss-Legendre; the reference calls QUADPACK with epsrel 1e-4.
//
// The arithmetic is that of one lane doing all of it in order (collocation rows
// solved from the first, quadrature terms added from the first), whatever the
// lanes share: the mirror field's neighbourhood amplifies rounding to 1e-12 of
// S_b, and a guiding centre whose output step moves by that follows, through
// its finite-difference gradients, a trajectory that is 1e-9 away.  What is
// independent is split: the collocation rows' coefficients (every other row a
// lane), the two mirror points, the quadrature terms (half a lane each).
//
// Points live in a scratch buffer laid out [wave][point][array][line of the
// wave]: pairs at the same step touch neighbouring addresses, a point's four
// arrays share one address, and a wave's scratch is one run of memory.
//
// What bounds it: the dependent chain of the trace (six field evaluations a
// step, a step a chunk for nearly every chunk, up to ~200 chunks a half line
// at fieldlineresolution 50) where few lines run, and with 65,536 lines vector
// issue (127,000 instructions a wave of 32 lines) and the points' traffic.
// Against one lane a line, with a binary search through the scratch, a cosine
// and a sine at each of the 512 nodes, a |B| evaluation beside each point's
// direction and 16,384 lanes at most: S_b of 65,536 lines 12.1 -> 0.80 ms,
// labels 17.0 -> 1.2 ms (16,384 queries with every wave; 9.9 on the 72 waves that
// dipole-type fields' are launched with, rapt_bounce.hip) and 14.8 -> 0.46 ms
// (300), five bounce centres over four
// rows 400 -> 11.1 ms, the same results bit for bit.
#pragma once
#ifndef __HIPCC_RTC__
#include <hip/hip_runtime.h>
#endif
#include <stdint.h>

#include "rapt_hip.h"
#include "rapt_fields.hpp"
#include "rapt_kargs.hpp"
#include "rapt_steppers.hpp"

namespace rapt {

static constexpr double GL16_X[8] = {0.09501250983763745, 0.2816035507792589,
                                     0.45801677765722737, 0.6178762444026438,
                                     0.755404408355003,   0.8656312023878318,
                                     0.9445750230732326,  0.9894009349916499};
static constexpr double GL16_W[8] = {0.18945061045506859, 0.1826034150449236,
                                     0.16915651939500262, 0.14959598881657676,
                                     0.12462897125553403, 0.09515851168249259,
                                     0.062253523938647706, 0.027152459411754037};

// A row of the points' scratch: 32 lines of arc length, |B|, spline coefficient
// and elimination workspace, at these byte offsets
constexpr uint32_t PT_S = 0, PT_B = 256, PT_C = 512, PT_W = 768, ROW = 1024;
// A wave's scratch: its rows, and an odd number of 256-byte pieces so that the
// waves, which move through their rows together, do not all address the same
// memory channels
__host__ __device__ constexpr uint32_t wave_bytes(int32_t cap) {
  return 2u * (uint32_t)cap * ROW + 17u * 256u;
}

enum { BST_OK = 1, BST_OVERFLOW = -20, BST_NOBRACKET = -21, BST_ROOT = -22, BST_NAN = -23 };

struct BounceArgs {
  FieldC F;
  int64_t n;
  const double* tpos;
  const double* Bm;
  double res;
  int32_t cap;   // points per half line
  int32_t what;  // k_halfbounce output: 0 S_b, 1 the second invariant I
  const int32_t* order;  // work item -> query (nullptr: identity)
  int64_t slots; // resident work items (lines; labels and bounce centres: groups)
  char* pts;     // [blocks] waves' points, wave_bytes(cap) each (below)
  double* Zs;    // [2*cap][slots] z of the centre line's points (labels only, else nullptr)
  double* Rs;    // [2*cap][slots] their cylindrical radius (labels only)
  double* out;
  int32_t* status;
};

template <int M>
struct LineRHS {
  const FieldC& F;
  double t, sign;
  __device__ __forceinline__ void operator()(double, const double* Y, double* o) {
    const V3 b = unitb<M>(F, t, Y[1], Y[2], Y[3]);
    o[0] = sign;
    o[1] = sign * b.x;
    o[2] = sign * b.y;
    o[3] = sign * b.z;
  }
};

// de Boor's BSPLVB for k = 2: the three splines that are not 0 at s in
// [ka, kb), whose neighbouring knots are kz <= ka and kb <= kc
struct Basis {
  double b0, b1, b2;
};
__device__ __forceinline__ Basis bsplines(double s, double kz, double ka, double kb, double kc) {
  const double left1 = s - ka, right1 = kb - s, left2 = s - kz, right2 = kc - s;
  double t = div_nr(1.0, right1 + left1);
  const double p0 = right1 * t, p1 = left1 * t;
  t = div_nr(p0, right1 + left2);
  const double b0 = right1 * t, sv = left2 * t;
  t = div_nr(p1, right2 + left1);
  return Basis{b0, sv + right2 * t, left1 * t};
}

// The quadratic spline on one interval between knots: the knots around it and
// its three coefficients
struct SplinePiece {
  double kz, ka, kb, kc, c0, c1, c2;
  __device__ __forceinline__ double operator()(double s) const {
    const Basis b = bsplines(s, kz, ka, kb, kc);
    return b.b0 * c0 + b.b1 * c1 + b.b2 * c2;
  }
};

// Brent's method (R. P. Brent, Algorithms for Minimization without
// Derivatives, 1973, ch. 4) with scipy.optimize.brentq's default tolerances
template <class Fn>
__device__ __forceinline__ bool brent(const Fn& f, double a, double b, double& root) {
  const double xtol = 2e-12, rtol = 8.881784197001252e-16;
  double fa = f(a), fb = f(b);
  if (fa == 0.0) { root = a; return true; }
  if (fb == 0.0) { root = b; return true; }
  if ((fa > 0.0) == (fb > 0.0)) return false;
  double c = a, fc = fa, d = b - a, e = d;
  for (int it = 0; it < 100; ++it) {
    if ((fb > 0.0) == (fc > 0.0)) { c = a; fc = fa; d = b - a; e = d; }
    if (fabs(fc) < fabs(fb)) { a = b; b = c; c = a; fa = fb; fb = fc; fc = fa; }
    const double tol1 = xtol + rtol * fabs(b);
    const double m = 0.5 * (c - b);
    if (fabs(m) <= tol1 || fb == 0.0) { root = b; return true; }
    if (fabs(e) >= tol1 && fabs(fa) > fabs(fb)) {
      double p, q, r;
      const double s = fb / fa;
      if (a == c) {
        p = 2.0 * m * s;
        q = 1.0 - s;
      } else {
        q = fa / fc;
        r = fb / fc;
        p = s * (2.0 * m * q * (q - r) - (b - a) * (r - 1.0));
        q = (q - 1.0) * (r - 1.0) * (s - 1.0);
      }
      if (p > 0.0) q = -q; else p = -p;
      if (2.0 * p < fmin(3.0 * m * q - fabs(tol1 * q), fabs(e * q))) {
        e = d;
        d = p / q;
      } else {
        d = m;
        e = m;
      }
    } else {
      d = m;
      e = m;
    }
    a = b;
    fa = fb;
    b += (fabs(d) > tol1) ? d : (m > 0.0 ? tol1 : -tol1);
    fb = f(b);
  }
  root = b;
  return true;
}

// The quadrature's nodes: cos(theta) and weight * sin(theta) of node q of
// panel p at [16 p + q].  The same for every line, so a block forms them once
// in LDS (512 cosines and sines a line otherwise).
constexpr int GL_P = 32, GL_N = 16 * GL_P;
constexpr int NODES = 2;  // between stores (line_pair)
struct QuadTab {
  double c[GL_N], ws[GL_N];
};
__device__ __forceinline__ void quad_tab(QuadTab& T) {
  const double pw = 3.141592653589793 / GL_P;
  for (int e = (int)threadIdx.x; e < GL_N; e += (int)blockDim.x) {
    const int p = e >> 4, q = e & 15;
    const double xg = (q < 8) ? -GL16_X[7 - q] : GL16_X[q - 8];
    const double wg = (q < 8) ? GL16_W[7 - q] : GL16_W[q - 8];
    const double th = (p + 0.5) * pw + 0.5 * pw * xg;
    T.c[e] = cos(th);
    T.ws[e] = wg * sin(th);
  }
  __syncthreads();
}

// the other lane of the pair's value (quad_perm [1, 0, 3, 2])
__device__ __forceinline__ double pair_swap(double v) {
  const long long b = __builtin_bit_cast(long long, v);
  const int lo = __builtin_amdgcn_update_dpp(0, (int)b, 0xB1, 0xF, 0xF, true);
  const int hi = __builtin_amdgcn_update_dpp(0, (int)(b >> 32), 0xB1, 0xF, 0xF, true);
  return __builtin_bit_cast(double, ((long long)hi << 32) | (unsigned)lo);
}

// The scratch value at a byte offset (unsigned: it reaches 2.01 GiB, and
// rapt_bounce.hip holds it below 4): the address stays in scalar registers and
// the offset is one 32-bit register.
__device__ __forceinline__ double& pt(const BounceArgs& A, uint32_t off) {
  return *(double*)(A.pts + off);
}

// Integrals over the field line through (x0, y0, z0) between the mirror
// points of B = Bm: sb = int ds / sqrt(1 - B/Bm) (flutils.halfbouncepath,
// rapt/flutils.py:254-316), eye = int sqrt(1 - B/Bm) ds (flutils.eye,
// rapt/flutils.py:65-151; 0 where the reference returns 0: Bm below the
// minimum of B on the line, or an equatorial particle to 1e-12), and lat =
// latitude (rad) of the mirror point along +b (when zq >= 0; eye when want_eye).  The eye
// integral uses the same quadratic spline and Gauss-Legendre quadrature as
// sb for every pitch angle; the reference switches to Simpson's rule on the
// trace points below 70 degrees, a rule whose discretisation error depends on
// where the trace points fall and so adds jitter to finite differences of I.
//
// Called by the two lanes of a pair (lanes 2k and 2k+1 of a wave) with the
// same arguments, in a block of one wave; both return the same values.
template <int M>
__device__ __forceinline__ int32_t line_pair(const BounceArgs& A, const QuadTab& T,
                                             int64_t zq, double t, double x0, double y0,
                                             double z0, double Bm, bool want_eye, double& sb,
                                             double& eye, double& lat) {
  const FieldC& F = A.F;
  const int g = (int)threadIdx.x & 1;
  const int32_t base = A.cap;  // array index of the start point
  // this pair's column in the wave's scratch
  const uint32_t col0 = blockIdx.x * wave_bytes(A.cap) + (threadIdx.x >> 1) * 8;
  sb = eye = lat = __builtin_nan("");
  const double ds = 1.0 / curvature<M>(F, t, x0, y0, z0) / A.res;
  // A chunk length that is not finite and positive (a NaN start point or
  // mirror field, a zero or infinite curvature such as |B| = 0 or a straight
  // line) would let a chunk end without adding a point, and the trace below
  // would never reach its mirror field.
  if (!(ds > 0.0 && ds < __builtin_inf()) || !(Bm > 0.0 && Bm < __builtin_inf()))
    return BST_NAN;
  int32_t st = BST_OK;
  int32_t np = 0;                   // points of the completed chunks of this half
  int32_t in_first = 0, in_last = 0;  // first and last of them with B <= Bm (0: none)
  double bmin = __builtin_inf();    // smallest |B| of them
  double b0;
  {
    const double sign = g ? -1.0 : 1.0, tol = g ? 1e-4 : 1e-3;
    const int32_t dir = g ? -1 : 1;
    LineRHS<M> f{F, t, sign};
    double Y[4] = {0.0, x0, y0, z0}, Y1[4], k0[4];
    uint32_t at = (uint32_t)base * ROW + col0 - (g ? ROW : 0);
    // |B| of the point just reached, and the first stage of the step from it
    auto at_point = [&](int32_t m) {
      const V3 B = fieldB<M>(F, t, Y[1], Y[2], Y[3]);
      const double bb = dot3(B, B);
      const double ib = rsqrt_nr(bb);
      const double bm = __builtin_sqrt(bb);
      k0[0] = sign;
      k0[1] = sign * (B.x * ib);
      k0[2] = sign * (B.y * ib);
      k0[3] = sign * (B.z * ib);
      if (m > 0 || g == 0) {
        const int64_t k = base + dir * m;
        pt(A, at + PT_S) = Y[0];
        pt(A, at + PT_B) = bm;
        at += g ? -ROW : ROW;
        if (zq >= 0) {
          A.Zs[k * A.slots + zq] = Y[3];
          A.Rs[k * A.slots + zq] = __builtin_sqrt(Y[1] * Y[1] + Y[2] * Y[2]);
        }
      }
      return bm;
    };
    b0 = at_point(0);
    double bm = b0;
    double tl = 0.0, h = ds;          // within the chunk
    int32_t m = 0, c_first = 0, c_last = 0;
    double c_min = __builtin_inf();   // of the chunk's points, until it completes
    for (;;) {
      if (tl + h > ds) h = ds - tl;
      const double r = rkf45_attempt_f0<4>(f, tl, h, Y, k0, Y1);
      if (r <= tol) {
        tl = tl + h;
        Y[0] = Y1[0]; Y[1] = Y1[1]; Y[2] = Y1[2]; Y[3] = Y1[3];
        if (++m >= A.cap) {
          st = BST_OVERFLOW;
          break;
        }
        bm = at_point(m);
        c_min = fmin(c_min, bm);
        if (bm <= Bm) {
          c_last = m;
          if (c_first == 0) c_first = m;
        }
      }
      const bool end = !(tl < ds);
      // the next step size: of no use at a chunk's end unless it is below
      // hmin, and it is at least a tenth of this one
      if (!end || h < 2e-5) {
        h = h * fmin(fmax(0.84 * pow(tol / r, 0.25), 0.1), 4.0);
        if (h > ds) {
          h = ds;
        } else if (h < 1e-6) {
          break;
        }
      }
      if (end) {
        np = m;
        bmin = fmin(bmin, c_min);
        if (in_first == 0) in_first = c_first;
        if (c_last != 0) in_last = c_last;
        if (bm > Bm) break;
        tl = 0.0;
        h = ds;
        c_first = c_last = 0;
        c_min = __builtin_inf();
      }
    }
  }
  // the other half's
  const int32_t np_o = __shfl_xor(np, 1), first_o = __shfl_xor(in_first, 1),
                last_o = __shfl_xor(in_last, 1), st_o = __shfl_xor(st, 1);
  bmin = fmin(fmin(bmin, __shfl_xor(bmin, 1)), b0);
  {
    const int32_t sf = g ? st_o : st, sn = g ? st : st_o;
    st = sf != BST_OK ? sf : sn;
  }
  if (st != BST_OK) return st;
  // both lanes read what the other one wrote
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup");
  // curve = array indices [base-nb, base+nf]; keep B <= Bm plus one each side
  const int32_t nf = g ? np_o : np, nb = g ? np : np_o;
  const int32_t lo = base - nb, hi = base + nf;
  const int32_t f1 = g ? first_o : in_first, f2 = g ? last_o : in_last;  // +b half
  const int32_t r1 = g ? in_first : first_o, r2 = g ? in_last : last_o;  // -b half
  const bool s_in = b0 <= Bm;
  const int32_t first = r2 ? base - r2 : (s_in ? base : (f1 ? base + f1 : -1));
  const int32_t lastin = f2 ? base + f2 : (s_in ? base : (r1 ? base - r1 : -1));
  int32_t i1, i2;
  const int32_t ncur = hi - lo + 1;
  if (first < 0) {
    i1 = lo + (ncur - 3) / 2;
    i2 = lo + (ncur + 1) / 2;
  } else {
    i1 = first - 1 < lo ? lo : first - 1;
    i2 = lastin + 1 > hi ? hi : lastin + 1;
  }
  const int32_t nt = i2 - i1 + 1;
  if (nt < 3) return BST_NOBRACKET;
  const bool eye_zero = bmin > Bm || __builtin_fabs(bmin - Bm) / Bm < 1e-12;
  if (nt == 3) {
    // equatorial: B(s) ~ B(s0) + B''/2 (s - s0)^2 from the Lagrange parabola
    auto X = [&](int32_t j) { return pt(A, (uint32_t)(i1 + j) * ROW + col0 + PT_S); };
    auto Yv = [&](int32_t j) { return pt(A, (uint32_t)(i1 + j) * ROW + col0 + PT_B); };
    const double s12 = X(0) - X(1), s23 = X(1) - X(2), s13 = X(0) - X(2);
    const double B2s = 2 * (Yv(0) * s23 - Yv(1) * s13 + Yv(2) * s12) / (s12 * s13 * s23);
    sb = 3.141592653589793 * __builtin_sqrt(2 * Bm / B2s);
    const double a2 = fmax(2.0 * (Bm - Yv(1)) / B2s, 0.0);
    eye = eye_zero ? 0.0 : 0.5 * 3.141592653589793 * a2 * __builtin_sqrt(B2s / (2.0 * Bm));
    if (zq >= 0) lat = atan(__builtin_sqrt(a2) / A.Rs[(int64_t)(i1 + 1) * A.slots + zq]);
    return BST_OK;
  }
  const int32_t nl = nt - 1;  // the last point
  const uint32_t o0 = (uint32_t)i1 * ROW + col0, ol = o0 + (uint32_t)nl * ROW;  // first, last
  const double xl = pt(A, ol + PT_S);
  // Tridiagonal collocation system (ROW j: N_{j-1}, N_j, N_{j+1} at x_j; rows
  // 0 and nl are the data), eliminated two rows an iteration: this lane forms
  // the coefficients of row jr, both lanes run the recurrence over both rows.
  {
    const double x00 = pt(A, o0 + PT_S);
    double cprev = 0.0, dprev = pt(A, o0 + PT_B);
    if (g == 0) {
      pt(A, o0 + PT_W) = 0.0;
      pt(A, o0 + PT_C) = dprev;
    }
    auto upto = [&](uint32_t o) { return o < ol ? o : ol; };
    int32_t jr = 1 + g;
    uint32_t oj = o0 + (uint32_t)jr * ROW;
    // points jr - 2 .. jr + 4 and values jr, jr + 2: two iterations' worth, the
    // next two's read while they are worked on (a read-ahead that only moves
    // from register to register each iteration would be waited for there)
    double xs[7], ys[2];
    xs[0] = x00;
#pragma unroll
    for (int k = 1; k < 7; ++k) xs[k] = pt(A, upto(oj + k * ROW - 2 * ROW) + PT_S);
    ys[0] = pt(A, upto(oj) + PT_B);
    ys[1] = pt(A, upto(oj + 2 * ROW) + PT_B);
#pragma unroll 1
    for (int32_t j = 1; j < nl; j += 4) {
      double xn[4], yn[2];
#pragma unroll
      for (int k = 0; k < 4; ++k) xn[k] = pt(A, upto(oj + (5 + k) * ROW) + PT_S);
#pragma unroll
      for (int k = 0; k < 2; ++k) yn[k] = pt(A, upto(oj + (4 + 2 * k) * ROW) + PT_B);
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const double *x = xs + 2 * h, y = ys[h];
        const int32_t q = jr + 2 * h, jh = j + 2 * h;  // this lane's row, the first of the two
        if (jh >= nl) break;
        // knots q .. q + 3 (0-2: the first point; nt and above: the last)
        const double k0 = q <= 2 ? x00 : (x[0] + x[1]) / 2;
        const double k1 = q <= 1 ? x00 : (x[1] + x[2]) / 2;
        const double k2 = q + 2 >= nt ? xl : (x[2] + x[3]) / 2;
        const double k3 = q + 3 >= nt ? xl : (x[3] + x[4]) / 2;
        const Basis b = bsplines(x[2], k0, k1, k2, k3);
        const double so = pair_swap(b.b0), to = pair_swap(b.b1), uo = pair_swap(b.b2),
                     yo = pair_swap(y);
        const double sub1 = g ? so : b.b0, dia1 = g ? to : b.b1, sup1 = g ? uo : b.b2,
                     y1 = g ? yo : y;
        double m = dia1 - sub1 * cprev, r = rcp_nr(m);
        const double ca = div_r(sup1, m, r), da = div_r(y1 - sub1 * dprev, m, r);
        cprev = ca;
        dprev = da;
        if (jh + 1 < nl) {
          const double sub2 = g ? b.b0 : so, dia2 = g ? b.b1 : to, sup2 = g ? b.b2 : uo,
                       y2 = g ? y : yo;
          m = dia2 - sub2 * cprev;
          r = rcp_nr(m);
          cprev = div_r(sup2, m, r);
          dprev = div_r(y2 - sub2 * dprev, m, r);
        }
        if (q < nl) {
          pt(A, oj + 2 * h * ROW + PT_W) = g ? cprev : ca;
          pt(A, oj + 2 * h * ROW + PT_C) = g ? dprev : da;
        }
      }
      jr += 4;
      oj += 4 * ROW;
#pragma unroll
      for (int k = 0; k < 3; ++k) xs[k] = xs[k + 4];
#pragma unroll
      for (int k = 0; k < 4; ++k) xs[3 + k] = xn[k];
      ys[0] = yn[0];
      ys[1] = yn[1];
    }
  }
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup");
  {
    // back substitution, the next eight rows read while eight are worked on
    double cn = pt(A, ol + PT_B);
    if (g == 0) pt(A, ol + PT_C) = cn;
    double w[8], c[8];
    uint32_t oj = ol - ROW;  // row j
    auto read8 = [&](uint32_t o) {
#pragma unroll
      for (int k = 0; k < 8; ++k) {
        const uint32_t ok = (int32_t)(o - o0) < k * (int32_t)ROW ? o0 : o - k * ROW;
        w[k] = pt(A, ok + PT_W);
        c[k] = pt(A, ok + PT_C);
      }
    };
    read8(oj);
#pragma unroll 1
    for (int32_t j = nl - 1; j >= 0; j -= 8) {
      double v[8];
#pragma unroll
      for (int k = 0; k < 8; ++k) v[k] = cn = j - k < 0 ? cn : c[k] - w[k] * cn;
      if (j >= 8) read8(oj - 8 * ROW);
      if (g == 0) {
#pragma unroll
        for (int k = 0; k < 8; ++k)
          if (j - k >= 0) pt(A, oj - k * ROW + PT_C) = v[k];
      }
      oj -= 8 * ROW;
    }
  }
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup");
  auto X = [&](int32_t j) { return pt(A, o0 + (uint32_t)j * ROW + PT_S); };
  auto C = [&](int32_t j) { return pt(A, o0 + (uint32_t)j * ROW + PT_C); };
  // knot i of the not-a-knot vector for k = 2
  auto knot = [&](int32_t i) {
    return i <= 2 ? X(0) : (i >= nt ? X(nl) : (X(i - 2) + X(i - 1)) / 2);
  };
  // the spline on [knot l, knot l + 1), 2 <= l <= nt - 1
  auto piece = [&](int32_t l) {
    return SplinePiece{knot(l - 1), knot(l),           knot(l + 1),      knot(l + 2),
                       C(l - 2), C(l - 1), C(l)};
  };
  // the mirror point of this lane's end, between the two outermost points
  double root = 0.0;
  {
    const SplinePiece sp = piece(g ? nt - 1 : 2);
    auto f = [&](double s) { return sp(s) - Bm; };
    const bool found = brent(f, g ? X(nl - 1) : X(0), g ? X(nl) : X(1), root);
    const int found_o = __shfl_xor((int)found, 1);
    if (!found || !found_o) return BST_ROOT;
  }
  const double ro = pair_swap(root);
  const double sm1 = g ? ro : root, sm2 = g ? root : ro;
  // s = mid - half cos(theta) removes the end-point singularities
  const double mid = 0.5 * (sm1 + sm2), half = 0.5 * (sm2 - sm1);
  double acc = 0.0, acc_i = 0.0;
  {
    // this lane's half of the nodes, from the interval of the first one to
    // the right; the next interval's data is read ahead
    const double *tc = T.c + g * (GL_N / 2), *tw = T.ws + g * (GL_N / 2);
    int32_t l = 2;
    if (g) {
      const double s = mid - half * tc[0];
      int32_t hi_l = nt - 1;  // largest l with knot(l) <= s
      while (hi_l - l > 1) {
        const int32_t ml = (l + hi_l) / 2;
        if (knot(ml) <= s) l = ml; else hi_l = ml;
      }
      if (knot(hi_l) <= s) l = hi_l;
    }
    SplinePiece sp = piece(l);
    // points l + 1 .. l + 3 and coefficients l + 1, l + 2, read ahead
    auto upto = [&](uint32_t o) { return o < ol ? o : ol; };
    uint32_t oq = o0 + (uint32_t)(l + 3) * ROW;  // of point l + 3
    double xp = pt(A, upto(oq - 2 * ROW) + PT_S), xn = pt(A, upto(oq - ROW) + PT_S),
           xm = pt(A, upto(oq) + PT_S);
    double cn = pt(A, upto(oq - 2 * ROW) + PT_C), cm = pt(A, upto(oq - ROW) + PT_C);
    const double rBm = rcp_nr(Bm);
    uint32_t ot = col0;  // the second half's terms (Wk's rows are free again)
    // NODES nodes between stores: loads and stores complete in order, so a
    // store at every node would put its latency before the next read's
#pragma unroll 1
    for (int e0 = 0; e0 < GL_N / 2; e0 += NODES) {
      double ts[NODES], ti[NODES];
#pragma unroll
      for (int k = 0; k < NODES; ++k) {
        const double s = mid - half * tc[e0 + k];
        while (l < nt - 1 && sp.kb <= s) {
          ++l;
          oq += ROW;
          sp.kz = sp.ka;
          sp.ka = sp.kb;
          sp.kb = sp.kc;
          sp.kc = l + 2 >= nt ? xl : (xp + xn) / 2;
          sp.c0 = sp.c1;
          sp.c1 = sp.c2;
          sp.c2 = cn;
          xp = xn;
          xn = xm;
          xm = pt(A, upto(oq) + PT_S);
          cn = cm;
          cm = pt(A, upto(oq - ROW) + PT_C);
        }
        const double val = 1.0 - div_r(sp(s), Bm, rBm);
        const double w = tw[e0 + k];
        const double sq = __builtin_sqrt(val);
        ts[k] = div_nr(w, sq);
        ti[k] = val > 0.0 ? w * sq : 0.0;
      }
      if (g == 0) {
#pragma unroll
        for (int k = 0; k < NODES; ++k) {
          acc += ts[k];
          acc_i += ti[k];
        }
      } else {
#pragma unroll
        for (int k = 0; k < NODES; ++k) pt(A, ot + k * ROW + PT_W) = ts[k];
        if (want_eye) {
#pragma unroll
          for (int k = 0; k < NODES; ++k) pt(A, ot + (GL_N / 2 + k) * ROW + PT_W) = ti[k];
        }
      }
      ot += NODES * ROW;
    }
    // the first half's sums, then the second half's terms in order
    // (the swaps run with both lanes of the pair active)
    const double a0 = pair_swap(acc), i0 = pair_swap(acc_i);
    if (g) {
      acc = a0;
      acc_i = i0;
      auto add = [&](double& sum, uint32_t o) {
        double v[8];
#pragma unroll
        for (int k = 0; k < 8; ++k) v[k] = pt(A, o + k * ROW + PT_W);
#pragma unroll 1
        for (int e = 8; e <= GL_N / 2; e += 8) {
          double u[8];
          o += 8 * ROW;
#pragma unroll
          for (int k = 0; k < 8; ++k) {
            u[k] = v[k];
            if (e < GL_N / 2) v[k] = pt(A, o + k * ROW + PT_W);
          }
#pragma unroll
          for (int k = 0; k < 8; ++k) sum += u[k];
        }
      };
      add(acc, col0);
      if (want_eye) add(acc_i, col0 + GL_N / 2 * ROW);
    }
    const double a1 = pair_swap(acc), i1s = pair_swap(acc_i);
    acc = g ? acc : a1;
    acc_i = g ? acc_i : i1s;
  }
  const double pw = 3.141592653589793 / GL_P;
  sb = acc * 0.5 * pw * half;
  eye = eye_zero ? 0.0 : acc_i * 0.5 * pw * half;
  if (!__builtin_isfinite(sb)) st = BST_NAN;
  if (zq >= 0) {
    // quadratic Lagrange interpolation of (z, rho) at the +b mirror point
    double zz = 0.0, rr = 0.0, xs[3];
    for (int a = 0; a < 3; ++a) xs[a] = pt(A, (uint32_t)(i2 - 2 + a) * ROW + col0 + PT_S);
    for (int a = 0; a < 3; ++a) {
      double w = 1.0;
      for (int b2 = 0; b2 < 3; ++b2)
        if (b2 != a) w *= (sm2 - xs[b2]) / (xs[a] - xs[b2]);
      zz += w * A.Zs[(int64_t)(i2 - 2 + a) * A.slots + zq];
      rr += w * A.Rs[(int64_t)(i2 - 2 + a) * A.slots + zq];
    }
    lat = atan2(zz, rr);
  }
  return st;
}

// Two waves a SIMD (256 registers) hide part of a line's dependent chain;
// gridded fields would spill 180 bytes a lane for it, the interpreter's calls
// more.
template <int M>
constexpr int line_waves() {
  return M == F_GRID || (M == F_EXPR && !EXPR_COMPILED) ? 1 : 2;
}

// Order in which a batch's lines are taken: by |B| / Bm at the start point
// (labels: sin^2 of the equatorial pitch angle), which sets how far along the
// line the mirror points lie and so how many points it has.  A wave's lines
// then end together, and read their points from the same rows of the scratch:
// taken as they come, 65,536 lines moved 3.1 GB past L2 and held a wave for the
// longest of 32 lines.  Each block sorts ORDER_CHUNK queries by counting.
constexpr int ORDER_CHUNK = 2048, ORDER_KEYS = 512, ORDER_THREADS = 512;
template <int M>
__global__ __launch_bounds__(ORDER_THREADS) void k_line_order(FieldC F, int64_t n, int labels,
                                                             const double* __restrict__ tpos,
                                                             const double* __restrict__ Bm,
                                                             int32_t* __restrict__ order) {
  __shared__ int32_t count[ORDER_KEYS];
  const int t = (int)threadIdx.x;
  const int64_t i0 = (int64_t)blockIdx.x * ORDER_CHUNK;
  constexpr int PER = ORDER_CHUNK / ORDER_THREADS;
  count[t] = 0;
  __syncthreads();
  int key[PER], rank[PER];
#pragma unroll
  for (int k = 0; k < PER; ++k) {
    const int64_t i = i0 + k * ORDER_THREADS + t;
    key[k] = -1;
    if (i >= n) continue;
    double x;
    if (labels) {
      const double sa = sin(tpos[3 * i + 1] * (3.141592653589793 / 180.0));
      x = sa * sa;
    } else {
      x = magB<M>(F, tpos[4 * i], tpos[4 * i + 1], tpos[4 * i + 2], tpos[4 * i + 3]) / Bm[i];
    }
    // longest lines first; any order is right, so a NaN may go anywhere
    key[k] = x >= 0.0 && x < 1.0 ? (int)(x * ORDER_KEYS) : ORDER_KEYS - 1;
    rank[k] = atomicAdd(&count[key[k]], 1);
  }
  __syncthreads();
  // exclusive prefix sum of the counts
  for (int d = 1; d < ORDER_KEYS; d <<= 1) {
    const int32_t v = t >= d ? count[t - d] : 0;
    __syncthreads();
    count[t] += v;
    __syncthreads();
  }
#pragma unroll
  for (int k = 0; k < PER; ++k) {
    if (key[k] < 0) continue;
    const int32_t at = (key[k] > 0 ? count[key[k] - 1] : 0) + rank[k];
    order[i0 + at] = (int32_t)(i0 + k * ORDER_THREADS + t);
  }
}

// S_b or I of a batch of start points, a pair of lanes each
template <int M>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(line_waves<M>())))
void k_halfbounce(BounceArgs A) {
  __shared__ QuadTab T;
  quad_tab(T);
  const int64_t slot = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) >> 1;
  if (slot >= A.slots) return;
  for (int64_t w = slot; w < A.n; w += A.slots) {
    const int64_t i = A.order ? A.order[w] : w;
    double sb, eye, lat;
    const int32_t st = line_pair<M>(A, T, -1, A.tpos[4 * i], A.tpos[4 * i + 1],
                                    A.tpos[4 * i + 2], A.tpos[4 * i + 3], A.Bm[i], A.what != 0,
                                    sb, eye, lat);
    if ((threadIdx.x & 1) == 0) {
      A.out[i] = A.what ? eye : sb;
      A.status[i] = st;
    }
  }
}

// The five lines of one bounce-averaged drift (flutils.gradI,
// rapt/flutils.py:153-229): the line through the point and the four at
// +-dstep across the field, one a pair of lanes, so a group is ten lanes and
// a wave holds six.
constexpr int GRP = 10;
constexpr int GRP_PER_WAVE = 6;
struct DriftLines {
  double sb, lat;     // of the centre line
  V3 gI;              // grad I across the field
  int32_t st;
};
// What a group needs again after its lines, kept in LDS meanwhile: in
// registers it costs the line integrals a wave a SIMD, or spills.
struct GroupKeep {
  V3 v1, v2;             // the directions across the field
  double v, gm, bsq, x;  // labels: speed, gamma m v^2, |B|^2 and x of the point
  V3 B;
};
// Called by the ten lanes of group gi of the wave with the same arguments.  I on the four lines is differenced
// centrally, or one-sided where an I is 0 (rapt/flutils.py:212-227); the
// status is the first failure in the order centre, +v1, -v1, +v2, -v2.
template <int M>
__device__ __forceinline__ DriftLines drift_lines(const BounceArgs& A, const QuadTab& T,
                                                  GroupKeep& keep, int gi, int64_t zq, double t,
                                                  double x, double y, double z, const V3& B,
                                                  double bsq, double Bm, double dstep) {
  // directions (rapt/flutils.py:196-207)
  const double mx = fmax(__builtin_fabs(x), __builtin_fabs(y));
  V3 r{x / mx, y / mx, 0.0};
  const double ib = 1.0 / __builtin_sqrt(bsq);
  const V3 b{B.x * ib, B.y * ib, B.z * ib};
  const double rb = dot3(r, b);
  r = V3{r.x - rb * b.x, r.y - rb * b.y, r.z - rb * b.z};
  const double rn = 1.0 / __builtin_sqrt(dot3(r, r));
  V3 v1{r.x * rn, r.y * rn, r.z * rn};
  V3 v2 = cross3(b, v1);
  const int l0 = GRP * gi, p = ((int)(threadIdx.x & 63) - l0) >> 1;
  double px = x, py = y, pz = z;
  if (p > 0) {
    const V3 w = p < 3 ? v1 : v2;
    const double d = (p & 1) ? dstep : -dstep;
    px = x + d * w.x;
    py = y + d * w.y;
    pz = z + d * w.z;
  }
  if ((int)threadIdx.x == l0) {
    keep.v1 = v1;
    keep.v2 = v2;
  }
  double sb, eye, lat;
  const int32_t st = line_pair<M>(A, T, p == 0 ? zq : -1, t, px, py, pz,
                                  Bm, true, sb, eye, lat);
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup");
  v1 = keep.v1;
  v2 = keep.v2;
  DriftLines D{__shfl(sb, l0), __shfl(lat, l0), V3{0.0, 0.0, 0.0}, __shfl(st, l0)};
  const double ic = __shfl(eye, l0);
  double dI[2];
  for (int k = 0; k < 2; ++k) {
    const double Ip = __shfl(eye, l0 + 2 + 4 * k), Imn = __shfl(eye, l0 + 4 + 4 * k);
    const int32_t sp = __shfl(st, l0 + 2 + 4 * k), sn = __shfl(st, l0 + 4 + 4 * k);
    if (D.st == BST_OK) D.st = sp;
    if (D.st == BST_OK) D.st = sn;
    if (Ip == 0.0) dI[k] = (ic - Imn) / dstep;
    else if (Imn == 0.0) dI[k] = (Ip - ic) / dstep;
    else dI[k] = (Ip - Imn) / (2.0 * dstep);
  }
  D.gI = V3{dI[0] * v1.x + dI[1] * v2.x, dI[0] * v1.y + dI[1] * v2.y,
            dI[0] * v1.z + dI[1] * v2.z};
  return D;
}

// Surrogate labels from one bounce-averaged drift evaluation per query
// (BounceCenter.advance's deriv, rapt/BounceCenter.py:235-244, at t = 0):
// query (L, equatorial pitch angle alpha [deg], log10 K [eV]) starts at the
// equatorial point (L Re, 0, 0); v from K (utils.speedfromKE), Bm =
// B_eq / sin^2 alpha, T_b = 2 S_b / v (flutils.bounceperiod), grad I by
// flutils.gradI (rapt/flutils.py:153-229: central differences of eye across
// the field, step eyegradientstep, one-sided where an I is 0), v_d =
// gamma m v^2 / (q S_b B^2) grad I x B, omega_d = v_d . phi_hat / rho.
// out[3 i + 0..2] = (T_b [s], omega_d [rad/s], mirror latitude [deg]).
struct LabelArgs {
  double mass, charge, dstep;
  double Re, eV;  // Earth radius [m] and joules per eV, as the caller's constants
};

template <int M>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(line_waves<M>())))
void k_bounce_labels(BounceArgs A, LabelArgs L) {
  __shared__ QuadTab T;
  __shared__ GroupKeep keep[GRP_PER_WAVE];
  quad_tab(T);
  const int gi = (int)threadIdx.x / GRP;
  const int64_t slot = (int64_t)blockIdx.x * GRP_PER_WAVE + gi;
  if (gi >= GRP_PER_WAVE || slot >= A.slots) return;
  const FieldC& F = A.F;
  const double Re = L.Re;
  const double mc2 = L.mass * C_LIGHT * C_LIGHT;
  for (int64_t w = slot; w < A.n; w += A.slots) {
    const int64_t i = A.order ? A.order[w] : w;
    const double Lsh = A.tpos[3 * i], alpha = A.tpos[3 * i + 1] * (3.141592653589793 / 180.0);
    const double K = pow(10.0, A.tpos[3 * i + 2]) * L.eV;
    // speedfromKE (rapt/utils.py:218-249): non-relativistic below K/mc2 = 1e-6
    double v;
    if (K / mc2 < 1e-6) {
      v = __builtin_sqrt(2.0 * K / L.mass);
    } else {
      const double g = 1.0 + K / mc2;
      v = C_LIGHT * __builtin_sqrt(1.0 - 1.0 / (g * g));
    }
    const double gamma = 1.0 / __builtin_sqrt(1.0 - (v / C_LIGHT) * (v / C_LIGHT));
    const double x0 = Lsh * Re, y0 = 0.0, z0 = 0.0, t = 0.0;
    const V3 B = fieldB<M>(F, t, x0, y0, z0);
    const double bsq = dot3(B, B);
    const double sa = sin(alpha);
    const double Bm = __builtin_sqrt(bsq) / (sa * sa);
    GroupKeep& k = keep[gi];
    if ((int)threadIdx.x == GRP * gi) {
      k.v = v;
      k.gm = gamma * L.mass * v * v;
      k.bsq = bsq;
      k.x = x0;
      k.B = B;
    }
    const DriftLines D = drift_lines<M>(A, T, k, gi, slot, t, x0, y0, z0, B, bsq, Bm, L.dstep);
    double Tb = __builtin_nan(""), wd = __builtin_nan(""), latd = __builtin_nan("");
    if (D.st == BST_OK) {
      const double coef = k.gm / (L.charge * D.sb * k.bsq);
      const V3 c = cross3(D.gI, k.B);
      const double rho = __builtin_sqrt(k.x * k.x + y0 * y0);
      // phi_hat = (-y, x, 0) / rho
      wd = coef * (c.y * k.x - c.x * y0) / (rho * rho);
      Tb = 2.0 * D.sb / k.v;
      latd = D.lat * (180.0 / 3.141592653589793);
    }
    if ((int)threadIdx.x == GRP * gi) {
      A.out[3 * i] = Tb;
      A.out[3 * i + 1] = wd;
      A.out[3 * i + 2] = latd;
      A.status[i] = D.st;
    }
  }
}

// ---- BounceCenter.advance (rapt/BounceCenter.py:206-251) -----------------------
// The drift right-hand side of the reference's deriv (:235-244, the
// non-equatorial branch): gamma m v^2 / (q S_b |B|^2) grad I x B, with S_b and
// grad I from the field-line integrals above.  A failed line integral stores
// its status and makes the derivative NaN.
template <int M>
struct DriftRHS {
  const BounceArgs& A;
  const QuadTab& T;
  GroupKeep& keep;
  int gi;  // the group in the wave
  double Bm, coef, dstep;
  int32_t st;
  int64_t nf;
  __device__ __forceinline__ void operator()(double t, const double* Y, double* out) {
    ++nf;
    const V3 B = fieldB<M>(A.F, t, Y[0], Y[1], Y[2]);
    const double bsq = dot3(B, B);
    const DriftLines D =
        drift_lines<M>(A, T, keep, gi, -1, t, Y[0], Y[1], Y[2], B, bsq, Bm, dstep);
    if (D.st != BST_OK) {
      if (st == BST_OK) st = D.st;
      out[0] = out[1] = out[2] = __builtin_nan("");
      return;
    }
    const double c = coef / (D.sb * bsq);
    const V3 x = cross3(D.gI, B);
    out[0] = c * x.x;
    out[1] = c * x.y;
    out[2] = c * x.z;
  }
};

struct BCArgs {
  int64_t n;
  double* tpos;          // [n][4] (t, x, y, z): start in, end out
  const double* Bm;      // [n] mirror field
  const double* coef;    // [n] gamma m v^2 / q
  const double* dt;      // [n] output step
  const double* tcur;    // [n] first row time (np.arange start)
  const int64_t* nrow;   // [n] rows to write
  const int64_t* row_off;
  double* rows;          // [.][4]
  int32_t* status;
  int64_t* naccpt;
  double rtol, atol, dstep;
  int32_t nmax, pad;
  CtlParams c5;
};

// The equatorial branch of deriv (rapt/BounceCenter.py:237-238): gradient
// plus inertial drift, _v_grad + _v_inert (:154-204), for bounce centres
// with no parallel motion.  _v_grad = mu (B x grad|B|) / (q gamma |B|^2);
// _v_inert = m |v_g| / (q |B|^2 2d) B x (v_g(+) - v_g(-)), the gradient drift
// differenced at +-d along its own direction, where the reference shifts the
// whole 4-vector (t, x, y, z) by d (t, v_g/|v_g|) -- the time shift included.
// The reference calls both with Y[:4], the 3-vector (x, y, z), which the
// fields' `t, x, y, z = tpos` rejects; here they take (t, x, y, z).
template <int M>
struct EqDriftRHS {
  const FieldC& F;
  double mu, mass, charge, gamma;
  int32_t st;
  int64_t nf;
  __device__ __forceinline__ V3 vgrad(double t, double x, double y, double z) const {
    const V3 B = fieldB<M>(F, t, x, y, z);
    const double bsq = dot3(B, B);
    const double d = F.gstep;
    // _Field.gradB (rapt/fields.py:111-131): central differences of |B|
    const double gx = (magB<M>(F, t, x + d, y, z) - magB<M>(F, t, x - d, y, z)) / (2.0 * d);
    const double gy = (magB<M>(F, t, x, y + d, z) - magB<M>(F, t, x, y - d, z)) / (2.0 * d);
    const double gz = (magB<M>(F, t, x, y, z + d) - magB<M>(F, t, x, y, z - d)) / (2.0 * d);
    const V3 c = cross3(B, V3{gx, gy, gz});
    const double den = charge * gamma * bsq;
    return V3{mu * c.x / den, mu * c.y / den, mu * c.z / den};
  }
  __device__ __forceinline__ void operator()(double t, const double* Y, double* out) {
    ++nf;
    const V3 vg = vgrad(t, Y[0], Y[1], Y[2]);
    const double vm = __builtin_sqrt(dot3(vg, vg));
    const double d = F.gstep;
    const double ux = vg.x / vm, uy = vg.y / vm, uz = vg.z / vm;
    const V3 v1 = vgrad(t - d * t, Y[0] - d * ux, Y[1] - d * uy, Y[2] - d * uz);
    const V3 v2 = vgrad(t + d * t, Y[0] + d * ux, Y[1] + d * uy, Y[2] + d * uz);
    const V3 B = fieldB<M>(F, t, Y[0], Y[1], Y[2]);
    const double s = mass * vm / (charge * dot3(B, B) * 2.0 * d);
    const V3 c = cross3(B, V3{v2.x - v1.x, v2.y - v1.y, v2.z - v1.z});
    out[0] = vg.x + s * c.x;
    out[1] = vg.y + s * c.y;
    out[2] = vg.z + s * c.z;
  }
};

// One lane per bounce centre: r = ode(deriv).set_integrator("dopri5", ...),
// then for each t in arange(tcur, tcur + delta, dt): integrate(r.t + dt) and
// append [t, r.y] (the row's time is the arange value, one step behind the
// state, as the reference writes it).  scipy's call semantics as in k_trace.
// writes: this lane stores the results (the lanes of a group run in step on
// the same values)
template <class RHS>
__device__ __forceinline__ void bc_run(RHS& f, const BCArgs& C, int64_t i, bool writes) {
  const CtlParams& P = C.c5;
  {
    double x = C.tpos[4 * i];
    double y[3] = {C.tpos[4 * i + 1], C.tpos[4 * i + 2], C.tpos[4 * i + 3]};
    double k1[3], y1[3], k7[3];
    f(x, y, k1);
    double h = 0.0;
    int32_t code = 1;
    int64_t acc = 0;
    const double dt = C.dt[i];
    for (int64_t r = 0; r < C.nrow[i] && code == 1; ++r) {
      const double xend = x + dt;
      const double hmax = xend - x;
      if (h == 0.0) h = hinit<3>(f, x, y, k1, 5, hmax, C.atol, C.rtol);
      double facold = 1.0e-4;
      int nstep = 0;
      bool last = false, reject = false;
      for (;;) {
        if (f.st != BST_OK) { code = f.st; break; }
        if (nstep > C.nmax) { code = RAPT_ST_NSTEPS; break; }
        if (0.1 * __builtin_fabs(h) <= __builtin_fabs(x) * UROUND) { code = RAPT_ST_HSMALL; break; }
        if (x + 1.01 * h - xend > 0.0) {
          h = xend - x;
          last = true;
        }
        ++nstep;
        const double err = dopri5_attempt<3>(f, x, h, y, k1, y1, k7, C.atol, C.rtol);
        if (f.st != BST_OK) { code = f.st; break; }
        const double fac11 = pow(err, P.expo1);
        double fac = fac11 / pow(facold, P.beta);
        fac = fmax(P.facc2, fmin(P.facc1, fac / P.safe));
        double hnew = h / fac;
        if (err <= 1.0) {
          facold = fmax(err, 1.0e-4);
          ++acc;
          for (int k = 0; k < 3; ++k) {
            k1[k] = k7[k];
            y[k] = y1[k];
          }
          x = x + h;
          if (last) {
            h = hnew;
            break;
          }
          if (__builtin_fabs(hnew) > hmax) hnew = hmax;
          if (reject) hnew = fmin(__builtin_fabs(hnew), __builtin_fabs(h));
          reject = false;
          h = hnew;
        } else {
          hnew = h / fmin(P.facc1, fac11 / P.safe);
          reject = true;
          last = false;
          h = hnew;
        }
      }
      if (writes) {
        double* row = C.rows + (C.row_off[i] + r) * 4;
        row[0] = C.tcur[i] + (double)r * dt;
        row[1] = y[0];
        row[2] = y[1];
        row[3] = y[2];
      }
    }
    if (!writes) return;
    C.tpos[4 * i] = x;
    C.tpos[4 * i + 1] = y[0];
    C.tpos[4 * i + 2] = y[1];
    C.tpos[4 * i + 3] = y[2];
    C.status[i] = code;
    C.naccpt[i] = acc;
  }
}

template <int M>
__global__ __launch_bounds__(64) void k_bounce_center(BounceArgs A, BCArgs C) {
  __shared__ QuadTab T;
  __shared__ GroupKeep keep[GRP_PER_WAVE];
  quad_tab(T);
  const int gi = (int)threadIdx.x / GRP;
  const int64_t slot = (int64_t)blockIdx.x * GRP_PER_WAVE + gi;
  if (gi >= GRP_PER_WAVE || slot >= A.slots) return;
  for (int64_t i = slot; i < C.n; i += A.slots) {
    DriftRHS<M> f{A, T, keep[gi], gi, C.Bm[i], C.coef[i], C.dstep, BST_OK, 0};
    bc_run(f, C, i, (int)threadIdx.x == GRP * gi);
  }
}

// Per-centre constants of the equatorial drift: mu, mass, charge, gamma
struct EqArgs {
  const double* k;  // [n][4]
};

template <int M>
__global__ __launch_bounds__(64) void k_bounce_center_eq(FieldC F, BCArgs C, EqArgs E) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= C.n) return;
  EqDriftRHS<M> f{F, E.k[4 * i], E.k[4 * i + 1], E.k[4 * i + 2], E.k[4 * i + 3], BST_OK, 0};
  bc_run(f, C, i, true);
}

}  // namespace rapt
