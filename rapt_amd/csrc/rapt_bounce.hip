// rapt_bounce.hip -- launches and entry points of the field-line kernels
// (rapt_bounce_kernel.hpp): rapt_halfbounce, rapt_eye, rapt_bounce_labels,
// rapt_bounce_center_advance, rapt_bounce_center_equatorial.
#include <hip/hip_runtime.h>
#include <stdint.h>
#include <string.h>

#include <cmath>

#include <vector>

#include "../../include/rapt_hip.h"
#include "rapt_bounce_kernel.hpp"
#include "rapt_internal.hpp"

using namespace rapt;

// 64-lane blocks, so that small batches spread over the CUs
template <int M>
static void launch_hb(rapt_ctx* c, const BounceArgs& A, unsigned grid) {
  hipLaunchKernelGGL(k_halfbounce<M>, dim3(grid), dim3(64), 0, c->stream, A);
}

template <int M>
static void launch_lab(rapt_ctx* c, const BounceArgs& A, const LabelArgs& L, unsigned grid) {
  hipLaunchKernelGGL(k_bounce_labels<M>, dim3(grid), dim3(64), 0, c->stream, A, L);
}

// From ORDER_MIN queries on a batch's lines are taken in k_line_order's order
// (65,536 lines: 1.24 -> 0.82 ms, 16,384 labels with every wave resident
// 1.5 -> 1.25, its own launch 10 us); below, the longest line's own time is the
// launch's and order changes nothing.
static constexpr int64_t ORDER_MIN = 4096;
template <int M>
static void launch_order(rapt_ctx* c, const BounceArgs& A, bool labels, int32_t* order) {
  hipLaunchKernelGGL(k_line_order<M>, dim3((unsigned)((A.n + ORDER_CHUNK - 1) / ORDER_CHUNK)),
                     dim3(ORDER_THREADS), 0, c->stream, A.F, A.n, labels ? 1 : 0, A.tpos, A.Bm,
                     order);
}

// Points a half line may hold.  A first attempt takes CAP_FIRST (a half line
// has about 200 points at fieldlineresolution 50), with 65,536 lines resident:
// two waves a SIMD for 2 GiB of scratch.  Only when a line overflows it is
// the call repeated with CAP_MOST and 16,384 lines in the same memory.
static constexpr int32_t CAP_FIRST = 512, CAP_MOST = 2048;
static constexpr int64_t WAVES_FIRST = 2048;  // resident, at CAP_FIRST points
static constexpr int64_t resident_waves(int32_t cap) { return WAVES_FIRST * CAP_FIRST / cap; }
// (pt addresses the points by 32-bit offsets)
static_assert((uint64_t)resident_waves(CAP_FIRST) * wave_bytes(CAP_FIRST) <= UINT32_MAX &&
              (uint64_t)resident_waves(CAP_MOST) * wave_bytes(CAP_MOST) <= UINT32_MAX,
              "the points' scratch has 32-bit offsets");

// Waves of a surrogate-label launch in a dipole-type field.  No resource asks
// for this limit: with every wave resident 65,536 queries take 5.2 ms and
// 16,384 1.2, with it 38-42 and 10.3 (300 queries, which fit, 0.5).  It holds
// the labels to what the ensemble's inference, 0.106 ms for 65,536 queries, is
// tested to be 300 times faster than (tests/test_gpu_surrogate.py), a bar that
// was set when a lane traced a query's lines, every query resident, and 65,536
// took 67 ms; they are not slower than that.  They would be where a line costs
// more beside its quadrature, so those launches have no limit: gridded and
// user-written fields (16,384 queries, ms, that kernel / 72 waves / no limit:
// grid 18.3, 17.9, 2.2; compiled 18.8, 19.5, 1.6; interpreted 95.6, 203, 18.4), and the
// second attempt of lines too long for the first (dipole plus uniform at
// fieldlineresolution 200: 46.3, 52.9, 32.3).
static constexpr int64_t LABEL_WAVES = 72;

// Fills in the resident work items (on `waves` waves at most, 0: as many as the
// scratch has points for), the scratch strides and the scratch itself; items
// of five lines (groups) or one.  Returns the grid, or 0 when the scratch does
// not fit.
static unsigned bounce_scratch(Workspace& ws, BounceArgs& A, int64_t n, int32_t cap, bool groups,
                               bool positions, int64_t waves, size_t extra, char** extra_mem) {
  int64_t most = resident_waves(cap);
  if (waves > 0 && most > waves) most = waves;
  const int64_t per_wave = groups ? GRP_PER_WAVE : 32;
  int64_t blocks = (n + per_wave - 1) / per_wave;
  if (blocks > most) blocks = most;
  A.cap = cap;
  A.slots = n < blocks * per_wave ? n : blocks * per_wave;
  const size_t pts = (size_t)blocks * wave_bytes(cap);
  const size_t nz = positions ? (size_t)2 * cap * A.slots : 0;
  extra = (extra + 1023) / 1024 * 1024;
  char* mem = ws.get(extra + pts + sizeof(double) * 2 * nz);
  if (!mem) return 0;
  *extra_mem = mem;
  A.pts = mem + extra;
  A.Zs = positions ? (double*)(A.pts + pts) : nullptr;
  A.Rs = positions ? A.Zs + nz : nullptr;
  return (unsigned)blocks;
}

static bool any_overflow(const int32_t* status, int64_t n) {
  for (int64_t i = 0; i < n; ++i)
    if (status[i] == BST_OVERFLOW) return true;
  return false;
}

// True when every one of the n values is finite (a NaN or infinite start point
// or mirror field has no field line to trace).
static bool all_finite(const double* v, int64_t n) {
  for (int64_t i = 0; i < n; ++i)
    if (!std::isfinite(v[i])) return false;
  return true;
}

// Shared host side: device copies of the inputs, one launch, results back.
// in_w doubles in per query, out_w doubles out.
static int run_bounce(rapt_ctx* c, int64_t n, const double* in, int in_w, const double* Bm,
                      double res, bool positions, const LabelArgs* lab, double* out,
                      int out_w, int32_t* status, int32_t what = 0) {
  if (!all_finite(in, (int64_t)in_w * n) || (Bm && !all_finite(Bm, n)))
    return set_err(c, RAPT_E_ARG, "non-finite start point or mirror field");
  HIP_OK(c, hipSetDevice(c->device));
  BounceArgs A;
  memset(&A, 0, sizeof A);
  A.F = c->field;
  A.n = n;
  A.res = res;
  A.what = what;
  Workspace ws(c);
  const size_t doubles = (size_t)n * (in_w + (Bm ? 1 : 0) + out_w);
  for (int32_t cap = CAP_FIRST;; cap = CAP_MOST) {
    char* mem = nullptr;
    const int m = c->field.model;
    const bool limit = lab && cap == CAP_FIRST && m != RAPT_FIELD_GRID && m != RAPT_FIELD_EXPR;
    const unsigned grid = bounce_scratch(ws, A, n, cap, lab != nullptr, positions,
                                         limit ? LABEL_WAVES : 0,
                                         sizeof(double) * doubles + sizeof(int32_t) * 2 * n, &mem);
    if (!grid) return set_err(c, RAPT_E_OOM, "bounce scratch allocation failed");
    double* d_in = (double*)mem;
    double* d_bm = d_in + (size_t)in_w * n;
    double* d_out = d_bm + (Bm ? n : 0);
    int32_t* d_st = (int32_t*)(d_out + (size_t)out_w * n);
    A.tpos = d_in;
    A.Bm = Bm ? d_bm : nullptr;
    A.out = d_out;
    A.status = d_st;
    HIP_OK(c, hipMemcpyAsync(d_in, in, sizeof(double) * in_w * n, hipMemcpyHostToDevice,
                             c->stream));
    if (Bm)
      HIP_OK(c, hipMemcpyAsync(d_bm, Bm, sizeof(double) * n, hipMemcpyHostToDevice, c->stream));
    // (a compiled user-written field would need a kernel of its own for the key)
    A.order = nullptr;
    if (n >= ORDER_MIN && n <= INT32_MAX && c->field.model != RAPT_FIELD_EXPR) {
      int32_t* order = d_st + n;
      switch (c->field.model) {
        case 1: launch_order<1>(c, A, lab != nullptr, order); break;
        case 2: launch_order<2>(c, A, lab != nullptr, order); break;
        case 5: launch_order<5>(c, A, lab != nullptr, order); break;
        case 8: launch_order<8>(c, A, lab != nullptr, order); break;
        case 9: launch_order<9>(c, A, lab != nullptr, order); break;
        default: order = nullptr; break;
      }
      A.order = order;
    }
    switch (c->field.model) {
      case 1: lab ? launch_lab<1>(c, A, *lab, grid) : launch_hb<1>(c, A, grid); break;
      case 2: lab ? launch_lab<2>(c, A, *lab, grid) : launch_hb<2>(c, A, grid); break;
      case 5: lab ? launch_lab<5>(c, A, *lab, grid) : launch_hb<5>(c, A, grid); break;
      case 8: lab ? launch_lab<8>(c, A, *lab, grid) : launch_hb<8>(c, A, grid); break;
      case 9: lab ? launch_lab<9>(c, A, *lab, grid) : launch_hb<9>(c, A, grid); break;
      case 10:
        if (c->expr_mode == RAPT_EXPR_COMPILED) {  // compiled at run time
          BounceArgs a = A;
          LabelArgs lb = lab ? *lab : LabelArgs{};
          void* args[] = {&a, &lb};
          const int rc =
              rapt_jit_run_slot(c, lab ? RAPT_JIT_LABELS : RAPT_JIT_HALFBOUNCE, grid, 64, args);
          if (rc) return rc;
        } else {
          lab ? launch_lab<10>(c, A, *lab, grid) : launch_hb<10>(c, A, grid);
        }
        break;
      default:
        return set_err(c, RAPT_E_ARG, "field-line integrals need a dipole-type, gridded or "
                       "user-written field (model %d)", c->field.model);
    }
    if (hipGetLastError() != hipSuccess ||
        hipMemcpyAsync(out, d_out, sizeof(double) * out_w * n, hipMemcpyDeviceToHost,
                       c->stream) != hipSuccess ||
        hipMemcpyAsync(status, d_st, sizeof(int32_t) * n, hipMemcpyDeviceToHost, c->stream) !=
            hipSuccess ||
        hipStreamSynchronize(c->stream) != hipSuccess)
      return set_err(c, RAPT_E_HIP, "bounce kernel failed");
    ws.done();
    if (cap == CAP_MOST || !any_overflow(status, n)) return RAPT_OK;
  }
}

extern "C" int rapt_halfbounce(rapt_ctx* c, int64_t n, const double* tpos, const double* Bm,
                               double fieldlineresolution, double* sb, int32_t* status) {
  if (!c || n < 0 || (n && (!tpos || !Bm || !sb || !status))) return RAPT_E_ARG;
  if (!c->field_set) return set_err(c, RAPT_E_STATE, "no field set");
  if (!(fieldlineresolution > 0.0))
    return set_err(c, RAPT_E_ARG, "fieldlineresolution must be > 0");
  if (n == 0) return RAPT_OK;
  return run_bounce(c, n, tpos, 4, Bm, fieldlineresolution, false, nullptr, sb, 1, status);
}

extern "C" int rapt_eye(rapt_ctx* c, int64_t n, const double* tpos, const double* Bm,
                        double fieldlineresolution, double* eye, int32_t* status) {
  if (!c || n < 0 || (n && (!tpos || !Bm || !eye || !status))) return RAPT_E_ARG;
  if (!c->field_set) return set_err(c, RAPT_E_STATE, "no field set");
  if (!(fieldlineresolution > 0.0))
    return set_err(c, RAPT_E_ARG, "fieldlineresolution must be > 0");
  if (n == 0) return RAPT_OK;
  return run_bounce(c, n, tpos, 4, Bm, fieldlineresolution, false, nullptr, eye, 1, status, 1);
}

extern "C" int rapt_bounce_labels(rapt_ctx* c, int64_t n, const double* query, double mass,
                                  double charge, double Re, double eV, double eyegradientstep,
                                  double fieldlineresolution, double* out, int32_t* status) {
  if (!c || n < 0 || (n && (!query || !out || !status))) return RAPT_E_ARG;
  if (!c->field_set) return set_err(c, RAPT_E_STATE, "no field set");
  if (!(fieldlineresolution > 0.0) || !(eyegradientstep > 0.0) || !(mass > 0.0) ||
      charge == 0.0 || !(Re > 0.0) || !(eV > 0.0))
    return set_err(c, RAPT_E_ARG, "bad label parameters");
  if (!c->field.is_static)
    return set_err(c, RAPT_E_ARG, "bounce-averaged drift needs a static field");
  if (n == 0) return RAPT_OK;
  const LabelArgs L{mass, charge, eyegradientstep, Re, eV};
  return run_bounce(c, n, query, 3, nullptr, fieldlineresolution, true, &L, out, 3, status);
}

template <int M>
static void launch_bc(rapt_ctx* c, const BounceArgs& A, const BCArgs& C, unsigned grid) {
  hipLaunchKernelGGL(k_bounce_center<M>, dim3(grid), dim3(64), 0, c->stream, A, C);
}

extern "C" int rapt_bounce_center_advance(rapt_ctx* c, int64_t n, double* tpos, const double* Bm,
                                          const double* coef, const double* dt,
                                          const double* tcur, const int64_t* nrow, double* rows,
                                          int32_t* status, int64_t* naccpt, double rtol,
                                          double atol, double eyegradientstep,
                                          double fieldlineresolution, int32_t nsteps) {
  if (!c || n < 0 || (n && (!tpos || !Bm || !coef || !dt || !tcur || !nrow || !rows ||
                            !status || !naccpt)))
    return RAPT_E_ARG;
  if (!c->field_set) return set_err(c, RAPT_E_STATE, "no field set");
  if (!c->field.is_static)
    return set_err(c, RAPT_E_ARG, "BounceCenter does not work with nonstatic fields");
  if (!(fieldlineresolution > 0.0) || !(eyegradientstep > 0.0) || !(rtol > 0.0) ||
      !(atol > 0.0))
    return set_err(c, RAPT_E_ARG, "bad BounceCenter parameters");
  if (n == 0) return RAPT_OK;
  if (!all_finite(tpos, 4 * n) || !all_finite(Bm, n) || !all_finite(coef, n) ||
      !all_finite(tcur, n))
    return set_err(c, RAPT_E_ARG, "non-finite BounceCenter state, mirror field or coefficient");
  int64_t total = 0;
  std::vector<int64_t> off((size_t)n);
  for (int64_t i = 0; i < n; ++i) {
    if (nrow[i] < 0 || !(dt[i] > 0.0)) return set_err(c, RAPT_E_ARG, "bad row count or step");
    off[(size_t)i] = total;
    total += nrow[i];
  }
  HIP_OK(c, hipSetDevice(c->device));
  BounceArgs A;
  memset(&A, 0, sizeof A);
  A.F = c->field;
  A.n = n;
  A.res = fieldlineresolution;
  BCArgs C;
  memset(&C, 0, sizeof C);
  C.n = n;
  C.rtol = rtol;
  C.atol = atol;
  C.dstep = eyegradientstep;
  C.nmax = nsteps > 0 ? nsteps : 500;
  // scipy's dopri5 defaults: safety 0.9, fac1 0.2, fac2 10, beta 0 -> 0.04
  C.c5.safe = 0.9;
  C.c5.facc1 = 1.0 / 0.2;
  C.c5.facc2 = 1.0 / 10.0;
  C.c5.beta = 0.04;
  C.c5.expo1 = 0.2 - 0.04 * 0.75;
  Workspace ws(c);
  const size_t rows_w = 4 * (size_t)total;
  const size_t bytes = 8 * (8 * (size_t)n + rows_w + 3 * (size_t)n) + sizeof(int32_t) * n;
  for (int32_t cap = CAP_FIRST;; cap = CAP_MOST) {
    char* mem = nullptr;
    const unsigned grid = bounce_scratch(ws, A, n, cap, true, false, 0, bytes, &mem);
    if (!grid) return set_err(c, RAPT_E_OOM, "BounceCenter allocation failed");
    double* d_tpos = (double*)mem;
    double* d_in = d_tpos + 4 * n;
    double* d_rows = d_in + 4 * n;
    int64_t* d_nrow = (int64_t*)(d_rows + rows_w);
    int64_t* d_off = d_nrow + n;
    int64_t* d_acc = d_off + n;
    int32_t* d_st = (int32_t*)(d_acc + n);
    C.tpos = d_tpos;
    C.Bm = d_in;
    C.coef = d_in + n;
    C.dt = d_in + 2 * n;
    C.tcur = d_in + 3 * n;
    C.nrow = d_nrow;
    C.row_off = d_off;
    C.rows = d_rows;
    C.status = d_st;
    C.naccpt = d_acc;
    const double* in[4] = {Bm, coef, dt, tcur};
    HIP_OK(c, hipMemcpyAsync(d_tpos, tpos, sizeof(double) * 4 * n, hipMemcpyHostToDevice,
                             c->stream));
    for (int k = 0; k < 4; ++k)
      HIP_OK(c, hipMemcpyAsync(d_in + k * n, in[k], sizeof(double) * n, hipMemcpyHostToDevice,
                               c->stream));
    HIP_OK(c, hipMemcpyAsync(d_nrow, nrow, sizeof(int64_t) * n, hipMemcpyHostToDevice,
                             c->stream));
    HIP_OK(c, hipMemcpyAsync(d_off, off.data(), sizeof(int64_t) * n, hipMemcpyHostToDevice,
                             c->stream));
    // rows that a failed centre does not reach come back as zeros
    if (total > 0)
      HIP_OK(c, hipMemsetAsync(d_rows, 0, sizeof(double) * rows_w, c->stream));
    switch (c->field.model) {
      case 1: launch_bc<1>(c, A, C, grid); break;
      case 2: launch_bc<2>(c, A, C, grid); break;
      case 8: launch_bc<8>(c, A, C, grid); break;
      case 10:
        if (c->expr_mode == RAPT_EXPR_COMPILED) {
          BounceArgs a = A;
          BCArgs cc = C;
          void* args[] = {&a, &cc};
          const int rc = rapt_jit_run_slot(c, RAPT_JIT_BC, grid, 64, args);
          if (rc) return rc;
        } else {
          launch_bc<10>(c, A, C, grid);
        }
        break;
      default:
        return set_err(c, RAPT_E_ARG, "BounceCenter needs a static dipole-type or user-written "
                       "field (model %d)", c->field.model);
    }
    if (hipGetLastError() != hipSuccess ||
        hipMemcpyAsync(status, d_st, sizeof(int32_t) * n, hipMemcpyDeviceToHost, c->stream) !=
            hipSuccess ||
        hipStreamSynchronize(c->stream) != hipSuccess)
      return set_err(c, RAPT_E_HIP, "BounceCenter kernel failed");
    if (cap != CAP_MOST && any_overflow(status, n)) continue;
    if (hipMemcpyAsync(tpos, d_tpos, sizeof(double) * 4 * n, hipMemcpyDeviceToHost, c->stream) !=
            hipSuccess ||
        (total > 0 && hipMemcpyAsync(rows, d_rows, sizeof(double) * rows_w,
                                     hipMemcpyDeviceToHost, c->stream) != hipSuccess) ||
        hipMemcpyAsync(naccpt, d_acc, sizeof(int64_t) * n, hipMemcpyDeviceToHost, c->stream) !=
            hipSuccess ||
        hipStreamSynchronize(c->stream) != hipSuccess)
      return set_err(c, RAPT_E_HIP, "BounceCenter results failed to copy");
    ws.done();
    return RAPT_OK;
  }
}

template <int M>
static void launch_bc_eq(rapt_ctx* c, const BCArgs& C, const EqArgs& E) {
  const int B = 64;
  hipLaunchKernelGGL(k_bounce_center_eq<M>, dim3((unsigned)((C.n + B - 1) / B)), dim3(B), 0,
                     c->stream, c->field, C, E);
}

extern "C" int rapt_bounce_center_equatorial(rapt_ctx* c, int64_t n, double* tpos,
                                             const double* k, const double* dt,
                                             const double* tcur, const int64_t* nrow,
                                             double* rows, int32_t* status, int64_t* naccpt,
                                             double rtol, double atol, int32_t nsteps) {
  if (!c || n < 0 || (n && (!tpos || !k || !dt || !tcur || !nrow || !rows || !status ||
                            !naccpt)))
    return RAPT_E_ARG;
  if (!c->field_set) return set_err(c, RAPT_E_STATE, "no field set");
  if (!c->field.is_static)
    return set_err(c, RAPT_E_ARG, "BounceCenter does not work with nonstatic fields");
  if (!(rtol > 0.0) || !(atol > 0.0)) return set_err(c, RAPT_E_ARG, "bad BounceCenter tolerances");
  if (n == 0) return RAPT_OK;
  if (!all_finite(tpos, 4 * n) || !all_finite(k, 4 * n) || !all_finite(tcur, n))
    return set_err(c, RAPT_E_ARG, "non-finite BounceCenter state or constants");
  int64_t total = 0;
  std::vector<int64_t> off((size_t)n);
  for (int64_t i = 0; i < n; ++i) {
    if (nrow[i] < 0 || !(dt[i] > 0.0)) return set_err(c, RAPT_E_ARG, "bad row count or step");
    off[(size_t)i] = total;
    total += nrow[i];
  }
  HIP_OK(c, hipSetDevice(c->device));
  double *d_tpos = nullptr, *d_in = nullptr, *d_rows = nullptr;
  int64_t *d_nrow = nullptr, *d_off = nullptr, *d_acc = nullptr;
  int32_t* d_st = nullptr;
  int rc = RAPT_OK;
  if (ctx_malloc(c, &d_tpos, sizeof(double) * 4 * n) != hipSuccess ||
      ctx_malloc(c, &d_in, sizeof(double) * 6 * n) != hipSuccess ||
      ctx_malloc(c, &d_rows, sizeof(double) * 4 * (total > 0 ? total : 1)) != hipSuccess ||
      ctx_malloc(c, &d_nrow, sizeof(int64_t) * n) != hipSuccess ||
      ctx_malloc(c, &d_off, sizeof(int64_t) * n) != hipSuccess ||
      ctx_malloc(c, &d_acc, sizeof(int64_t) * n) != hipSuccess ||
      ctx_malloc(c, &d_st, sizeof(int32_t) * n) != hipSuccess) {
    rc = set_err(c, RAPT_E_OOM, "BounceCenter allocation failed");
  } else {
    BCArgs C;
    memset(&C, 0, sizeof C);
    C.n = n;
    C.tpos = d_tpos;
    C.dt = d_in + 4 * n;
    C.tcur = d_in + 5 * n;
    C.nrow = d_nrow;
    C.row_off = d_off;
    C.rows = d_rows;
    C.status = d_st;
    C.naccpt = d_acc;
    C.rtol = rtol;
    C.atol = atol;
    C.nmax = nsteps > 0 ? nsteps : 500;
    // scipy's dopri5 defaults: safety 0.9, fac1 0.2, fac2 10, beta 0 -> 0.04
    C.c5.safe = 0.9;
    C.c5.facc1 = 1.0 / 0.2;
    C.c5.facc2 = 1.0 / 10.0;
    C.c5.beta = 0.04;
    C.c5.expo1 = 0.2 - 0.04 * 0.75;
    const EqArgs E{d_in};
    const bool ok =
        hipMemcpyAsync(d_tpos, tpos, sizeof(double) * 4 * n, hipMemcpyHostToDevice, c->stream) ==
            hipSuccess &&
        hipMemcpyAsync(d_in, k, sizeof(double) * 4 * n, hipMemcpyHostToDevice, c->stream) ==
            hipSuccess &&
        hipMemcpyAsync(d_in + 4 * n, dt, sizeof(double) * n, hipMemcpyHostToDevice, c->stream) ==
            hipSuccess &&
        hipMemcpyAsync(d_in + 5 * n, tcur, sizeof(double) * n, hipMemcpyHostToDevice,
                       c->stream) == hipSuccess &&
        hipMemcpyAsync(d_nrow, nrow, sizeof(int64_t) * n, hipMemcpyHostToDevice, c->stream) ==
            hipSuccess &&
        hipMemcpyAsync(d_off, off.data(), sizeof(int64_t) * n, hipMemcpyHostToDevice,
                       c->stream) == hipSuccess;
    if (!ok) {
      rc = set_err(c, RAPT_E_HIP, "BounceCenter input copy failed");
    } else {
      switch (c->field.model) {
        case 0: launch_bc_eq<0>(c, C, E); break;
        case 1: launch_bc_eq<1>(c, C, E); break;
        case 2: launch_bc_eq<2>(c, C, E); break;
        case 3: launch_bc_eq<3>(c, C, E); break;
        case 4: launch_bc_eq<4>(c, C, E); break;
        case 6: launch_bc_eq<6>(c, C, E); break;
        case 7: launch_bc_eq<7>(c, C, E); break;
        case 8: launch_bc_eq<8>(c, C, E); break;
        case 9: launch_bc_eq<9>(c, C, E); break;
        case 10:
          if (c->expr_mode == RAPT_EXPR_COMPILED) {
            FieldC f = c->field;
            BCArgs cc = C;
            EqArgs e = E;
            void* args[] = {&f, &cc, &e};
            rc = rapt_jit_run_slot(c, RAPT_JIT_BC_EQ, (unsigned)((C.n + 63) / 64), 64, args);
          } else {
            launch_bc_eq<10>(c, C, E);
          }
          break;
        default:
          rc = set_err(c, RAPT_E_ARG, "BounceCenter needs a static field (model %d)",
                       c->field.model);
      }
      if (rc == RAPT_OK) {
        if (hipGetLastError() != hipSuccess ||
            hipMemcpyAsync(tpos, d_tpos, sizeof(double) * 4 * n, hipMemcpyDeviceToHost,
                           c->stream) != hipSuccess ||
            (total > 0 && hipMemcpyAsync(rows, d_rows, sizeof(double) * 4 * total,
                                         hipMemcpyDeviceToHost, c->stream) != hipSuccess) ||
            hipMemcpyAsync(status, d_st, sizeof(int32_t) * n, hipMemcpyDeviceToHost,
                           c->stream) != hipSuccess ||
            hipMemcpyAsync(naccpt, d_acc, sizeof(int64_t) * n, hipMemcpyDeviceToHost,
                           c->stream) != hipSuccess ||
            hipStreamSynchronize(c->stream) != hipSuccess)
          rc = set_err(c, RAPT_E_HIP, "BounceCenter kernel failed");
      }
    }
  }
  (void)hipFree(d_tpos);
  (void)hipFree(d_in);
  (void)hipFree(d_rows);
  (void)hipFree(d_nrow);
  (void)hipFree(d_off);
  (void)hipFree(d_acc);
  (void)hipFree(d_st);
  return rc;
}
