// smaug_host.hip -- C-ABI of the engine (declared in include/smaug_hip.h):
// device state, grid set-up, stage orchestration on one HIP stream.
#include <math.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

#include <mutex>
#include <string>
#include <vector>

#include "../../include/smaug_hip.h"
#include "smaug_dev.h"
#include "smaug_ops.h"


using namespace smaug;

static thread_local std::string g_err;

#include <stdarg.h>
static int vfail(int code, const char* fmt, va_list ap) {
  char buf[512];
  vsnprintf(buf, sizeof buf, fmt, ap);
  g_err = buf;
  return code;
}

static int fail(int code, const char* fmt, ...) {
  va_list ap;
  va_start(ap, fmt);
  const int r = vfail(code, fmt, ap);
  va_end(ap);
  return r;
}

namespace smaug {
// error reporting for the file readers/writers (smaug_io.cpp)
int io_fail(int code, const char* fmt, ...) {
  va_list ap;
  va_start(ap, fmt);
  const int r = vfail(code, fmt, ap);
  va_end(ap);
  return r;
}
}  // namespace smaug

#define HIPCHK(call)                                                                   \
  do {                                                                                 \
    hipError_t e_ = (call);                                                            \
    if (e_ != hipSuccess) return fail(SMAUG_E_HIP, "%s (code %d)", hipGetErrorString(e_), (int)e_); \
  } while (0)

// A caller's device buffer of `bytes` bytes at p must lie inside one device
// allocation (a pointer torch or another allocator hands out, or one of this
// library's); otherwise the call is refused before anything is queued.
static int check_range(const void* p, size_t bytes, const char* what) {
  hipDeviceptr_t base = nullptr;
  size_t size = 0;
  const hipError_t e = hipMemGetAddressRange(&base, &size, (hipDeviceptr_t)p);
  if (e != hipSuccess) {
    (void)hipGetLastError();  // the failed query leaves no error for the next call
    return fail(SMAUG_E_ARG, "%s (%p) is not device memory: %s", what, p, hipGetErrorString(e));
  }
  const char* end = (const char*)base + size;
  if ((const char*)p + bytes > end)
    return fail(SMAUG_E_ARG, "%s: %zu bytes at %p run %zu bytes past the end of its allocation", what, bytes, p,
                (size_t)((const char*)p + bytes - end));
  return SMAUG_OK;
}

struct smaug_ctx {
  smaug_params p;
  Geo G;
  hipStream_t stream = nullptr;  // stream all work is queued on
  hipStream_t own = nullptr;     // the context's own stream
  int nd = 0, np = 0, nb = 0, npr = 0, nvar = 0;
  long long N = 0;
  double* U[4] = {nullptr, nullptr, nullptr, nullptr};  // evolved-field buffers
  double* bg = nullptr;
  void* prim = nullptr;     // double, or float when mixed
  float* shadow = nullptr;  // mixed: FP32 copy of the stage input for the stencils
  double* delx = nullptr;
  double* rdelx = nullptr;
  double* dx1 = nullptr;   // separable grid: per-coordinate spacing (n0+n1+n2)
  double* rdx1 = nullptr;
  double* pos = nullptr;
  double* dshape = nullptr;  // per-axis factors of the vertical driver (separable grid)
  unsigned long long* cmax = nullptr;  // 3 slots of 4
  double* dts = nullptr;               // dt, t
  int* flag = nullptr;
  int cur = 0;      // buffer holding the current state
  int cslot = 0;    // maxima slot of the next k_prim
  double qt = 0;
  int it = 0;
  std::vector<double> h_pos, h_delx;
  double* amap = nullptr;    // driver amplitude per (j,k) column
  double* adj = nullptr;     // adjoint work: lam_s1..3, mu, T (np*N each), gcell (N)
  double* aprim = nullptr;   // FP64 k_prim of an adjoint stage input
  // tangent-linear run (smaug_tl_*): Dual stage buffers, derived fields
  // and driver map, its own maxima slots, (dt, t), clock and host staging
  Dual* tlU[4] = {nullptr, nullptr, nullptr, nullptr};
  void* tlprim = nullptr;     // Dual, or DualF in a mixed-precision context
  void* tlshadow = nullptr;   // mixed precision: FP32 dual shadow of the stage input
  Dual* tlbg = nullptr;  // background with its tangent
  Dual* tlamap = nullptr;
  unsigned long long* tlcmax = nullptr;  // 2 slots of 4
  double* tldts = nullptr;
  double* tltmp = nullptr;  // 2 np*N doubles
  int tlcur = 0, tlslot = 0, tlit = 0;
  double tlqt = 0;
  double tldamp = 0;  // tangent of the driver amplitude drv[0]
  bool tl = false;
};

static void free_tl(smaug_t* s) {
  for (auto& u : s->tlU) {
    hipFree(u);
    u = nullptr;
  }
  hipFree(s->tlprim);
  hipFree(s->tlshadow);
  hipFree(s->tlbg);
  hipFree(s->tlamap);
  hipFree(s->tlcmax);
  hipFree(s->tldts);
  hipFree(s->tltmp);
  s->tlprim = s->tlshadow = nullptr;
  s->tlbg = s->tlamap = nullptr;
  s->tlcmax = nullptr;
  s->tldts = s->tltmp = nullptr;
  s->tl = false;
}

// ---- grid: positions extrapolated past the interior, delx (initgrid,
// src/init.cu:2502-3051, quirk Q11) -----------------------------------------
static void initgrid_host(int nd, const int* n, const double* pos, std::vector<double>& opos,
                          std::vector<double>& odelx) {
  const long long n0 = n[0], n1 = n[1], n2 = nd == 3 ? n[2] : 1;
  const long long N = n0 * n1 * n2;
  const long long P0 = n0 + 2, P1 = n1 + 2, P2 = nd == 3 ? n2 + 2 : 1;
  const long long NP2 = P0 * P1 * P2;
  auto e2 = [&](long long a, long long b, long long c) { return (c * P1 + b) * P0 + a; };
  std::vector<double> tt((size_t)3 * NP2, 0.0);
  for (int d = 0; d < nd; d++)
    for (long long k = 0; k < n2; k++)
      for (long long j = 0; j < n1; j++)
        for (long long i = 0; i < n0; i++)
          tt[d * NP2 + e2(i + 1, j + 1, nd == 3 ? k + 1 : 0)] = pos[d * N + (k * n1 + j) * n0 + i];
  const long long PP[3] = {P0, P1, P2};
  for (int dir = 0; dir < nd; dir++) {
    const int nn = n[dir];
    for (int side = 0; side < 2; side++) {
      int ixmin, ixmax, ixe, ixf;
      if (side == 0) {
        ixmax = nn + 1;
        ixmin = nn - 1;
        ixe = ixmin - 1;
        ixf = ixe - 1;
      } else {
        ixmin = 0;
        ixmax = dir == 0 ? 1 : 2;
        ixe = ixmax + 1;
        ixf = ixe + 1;
      }
      for (int d1 = 0; d1 < nd; d1++) {
        double* T = tt.data() + d1 * NP2;
        for (long long c2 = 0; c2 < PP[2]; c2++)
          for (long long c1 = 0; c1 < PP[1]; c1++)
            for (long long c0 = 0; c0 < PP[0]; c0++) {
              long long cc[3] = {c0, c1, c2};
              const int ix = (int)cc[dir];
              if (ix < ixmin || ix > ixmax) continue;
              long long e1[3] = {c0, c1, c2}, f1[3] = {c0, c1, c2};
              e1[dir] = ixe;
              f1[dir] = ixf;
              const double a = (double)(1 + abs(ixe - ix)), b = (double)abs(ixe - ix);
              T[e2(c0, c1, c2)] = a * (T[e2(e1[0], e1[1], e1[2])]) - b * (T[e2(f1[0], f1[1], f1[2])]);
            }
      }
    }
  }
  opos.assign((size_t)nd * N, 0.0);
  odelx.assign((size_t)nd * N, 0.0);
  for (int d = 0; d < nd; d++) {
    const double* T = tt.data() + d * NP2;
    const long long o0 = d == 0, o1 = d == 1, o2 = d == 2;
    for (long long k = 0; k < n2; k++)
      for (long long j = 0; j < n1; j++)
        for (long long i = 0; i < n0; i++) {
          const long long c = (k * n1 + j) * n0 + i, kp = nd == 3 ? k + 1 : 0;
          opos[d * N + c] = T[e2(i + 1, j + 1, kp)];
          odelx[d * N + c] = 0.5 * (T[e2(i + 1 + o0, j + 1 + o1, kp + o2)] - T[e2(i + 1 - o0, j + 1 - o1, kp - o2)]);
        }
  }
}

static int check_params(const smaug_params* p) {
  if (p->ndim != 2 && p->ndim != 3) return fail(SMAUG_E_ARG, "ndim must be 2 or 3");
  for (int d = 0; d < p->ndim; d++)
    if (p->n[d] < 8) return fail(SMAUG_E_ARG, "n[%d] must be >= 8 (got %d)", d, p->n[d]);
  if (p->ndim == 2 && p->n[2] != 1) return fail(SMAUG_E_ARG, "2D runs need n[2] == 1");
  {  // the stencil kernels address a field with 32-bit byte offsets
    const long long cells = (long long)p->n[0] * p->n[1] * (p->ndim == 3 ? p->n[2] : 1);
    if (cells >= (1ll << 29))
      return fail(SMAUG_E_UNSUPPORTED, "%lld cells: grids of 2^29 cells or more are not supported", cells);
  }
  if (p->divbon != 0 && p->divbon != 1) return fail(SMAUG_E_ARG, "divbon must be 0 or 1");
  if (p->rkon != 0 && p->rkon != 1) return fail(SMAUG_E_ARG, "rkon must be 0 or 1");
  if (p->precision != SMAUG_PREC_FP64 && p->precision != SMAUG_PREC_MIXED)
    return fail(SMAUG_E_ARG, "unknown precision");
  if (p->driver < SMAUG_DRIVER_NONE || p->driver > SMAUG_DRIVER_SPICULE1) return fail(SMAUG_E_ARG, "unknown driver");
  if (p->driver == SMAUG_DRIVER_VERTICAL && (p->drv[1] == 0 || p->drv[5] == 0 || p->drv[6] == 0))
    return fail(SMAUG_E_ARG, "driver needs a period and widths (drv[1], drv[5], drv[6])");
  if (p->driver == SMAUG_DRIVER_TORSIONAL) {
    if (p->ndim != 3) return fail(SMAUG_E_ARG, "the torsional driver (fluxtube1) is 3D");
    for (int q = 5; q <= 9; q++)
      if (p->drv[q] == 0) return fail(SMAUG_E_ARG, "the torsional driver needs widths and scales (drv[5..9])");
  }
  if (p->driver == SMAUG_DRIVER_SPICULE1 && (p->drv[5] == 0 || p->drv[6] == 0))
    return fail(SMAUG_E_ARG, "the spicule driver needs widths (drv[5], drv[6])");
  const int np = 2 + 2 * p->ndim;
  for (int f = 0; f < np; f++)
    for (int d = 0; d < p->ndim; d++) {
      const int bt = p->boundtype[f][d][0];
      if (bt == 0 && p->ndim == 3)
        return fail(SMAUG_E_UNSUPPORTED, "periodic boundaries are supported in 2D only");
      if (bt == 1 || bt == 2)
        return fail(SMAUG_E_UNSUPPORTED, "MPI boundary types (1, 2) need a multi-domain run");
      if (bt < 0 || bt > 7) return fail(SMAUG_E_ARG, "unknown boundary type %d", bt);
    }
  if (p->moddton == 1 && !(p->courant > 0)) return fail(SMAUG_E_ARG, "courant must be > 0");
  if (!(p->dt > 0)) return fail(SMAUG_E_ARG, "dt must be > 0");
  return SMAUG_OK;
}

static void make_geo(const smaug_params* p, Geo& G) {
  memset(&G, 0, sizeof G);
  G.nd = p->ndim;
  G.n[0] = p->n[0];
  G.n[1] = p->n[1];
  G.n[2] = p->ndim == 3 ? p->n[2] : 1;
  G.N = (long long)G.n[0] * G.n[1] * G.n[2];
  G.st[0] = 1;
  G.st[1] = G.n[0];
  G.st[2] = (long long)G.n[0] * G.n[1];
  G.np = 2 + 2 * p->ndim;
  G.gamma = p->gamma;
  for (int d = 0; d < 3; d++) G.g[d] = p->g[d];
  for (int f = 0; f < G.np; f++) G.chyp[f] = p->chyp[f];
  for (int idx = 0; idx < kMaxVar; idx++) {
    unsigned m = 0;
    for (int d = 0; d < p->ndim; d++)
      if (p->boundtype[idx][d][0] != 0) m |= 1u << d;
    G.zm[idx] = m;
  }
  G.bc_uniform = 1;
  for (int f = 0; f < G.np; f++)
    for (int d = 0; d < 3; d++) {
      G.bct[f][d] = d < p->ndim ? p->boundtype[f][d][0] : 4;
      if (G.bct[f][d] != G.bct[0][d]) G.bc_uniform = 0;
      if (d < p->ndim && G.bct[f][d] == BC_FIXED) G.has_fixed = 1;
    }
  G.terms = p->terms;
  G.hyper = p->hyperdifmom;
  G.driver = p->driver;
  for (int i = 0; i < SMAUG_NDRV; i++) G.drv[i] = p->drv[i];
  G.mixed = p->precision == SMAUG_PREC_MIXED;
  // src/divb.cu:165-338 acts in 2D only (its launch covers the k = 0 plane,
  // which its 3D region test excludes)
  G.divb = p->divbon == 1 && p->divbfix != 0 && p->ndim == 2;
  for (int d = 0; d < 3; d++) {
    G.pdx[d] = d < p->ndim ? p->dx[d] : 1.0;
    G.pxmin[d] = d < p->ndim ? p->xmin[d] : 0.0;
  }
}

// Whether a (nd arrays of N cells: spacings or positions) depends, along every
// d, on the d coordinate only: then its values per coordinate (n0 of dim 0,
// then n1 of dim 1, ...) in a1.  Only interior cells count, the ones whose
// spacings and positions the kernels read: the ghost layers hold values
// extrapolated along the other directions as well, a rounding away from
// those of the interior rows wherever the spacing is no short binary
// fraction (every size but 128, 256, ... of the stratified domain; with them
// in the test those grids would read nd*N arrays and evaluate the driver's
// exponentials per cell: 0.352 against 0.322 ms per launch of the stage
// kernel at 96^3, 1.09 against 1.06 ms per RK4 step at 101x75x61).
static bool separable_interior(int nd, const int* n, const std::vector<double>& a, std::vector<double>& a1) {
  const long long n0 = n[0], n1 = n[1], n2 = nd == 3 ? n[2] : 1, N = n0 * n1 * n2;
  const long long lo2 = nd == 3 ? 2 : 0, hi2 = nd == 3 ? n2 - 2 : 1;
  const long long st[3] = {1, n0, n0 * n1}, first[3] = {2, 2, lo2};
  a1.clear();
  for (int d = 0; d < nd; d++) {
    const double* v = a.data() + (size_t)d * N;
    const size_t off = a1.size();
    long long row = 0;  // the line along d through the first interior cell
    for (int q = 0; q < nd; q++)
      if (q != d) row += first[q] * st[q];
    for (int x = 0; x < n[d]; x++) a1.push_back(v[row + x * st[d]]);
    const double* t = a1.data() + off;
    for (long long k = lo2; k < hi2; k++)
      for (long long j = 2; j < n1 - 2; j++) {
        const double* r = v + (k * n1 + j) * n0;
        bool same = true;
        if (d == 0) {
          for (long long i = 2; i < n0 - 2; i++) same &= r[i] == t[i];
        } else {
          const double w = t[d == 1 ? j : k];
          for (long long i = 2; i < n0 - 2; i++) same &= r[i] == w;
        }
        if (!same) return false;
      }
  }
  return true;
}

static void free_ctx(smaug_t* s) {
  if (!s) return;
  for (auto& u : s->U)
    if (u) hipFree(u);
  hipFree(s->bg);
  hipFree(s->prim);
  hipFree(s->shadow);
  hipFree(s->delx);
  hipFree(s->rdelx);
  hipFree(s->dx1);
  hipFree(s->rdx1);
  hipFree(s->pos);
  hipFree(s->dshape);
  hipFree(s->cmax);
  hipFree(s->dts);
  hipFree(s->flag);
  hipFree(s->amap);
  hipFree(s->adj);
  hipFree(s->aprim);
  free_tl(s);
  if (s->own) hipStreamDestroy(s->own);
  delete s;
}

extern "C" int smaug_create(const smaug_params* p, const double* w0, const double* pos, smaug_t** out) {
  if (!p || !w0 || !pos || !out) return fail(SMAUG_E_ARG, "null argument");
  int rc = check_params(p);
  if (rc) return rc;
  smaug_t* s = new smaug_t();
  s->p = *p;
  make_geo(p, s->G);
  s->nd = p->ndim;
  s->np = 2 + 2 * s->nd;
  s->nb = 2 + s->nd;
  s->npr = s->nd + 1;  // v_0..v_{nd-1}, q_e
  s->nvar = 4 + 3 * s->nd;
  s->N = s->G.N;
  const size_t bytes = sizeof(double) * (size_t)s->N;
  hipError_t e = hipStreamCreateWithFlags(&s->own, hipStreamNonBlocking);
  if (e != hipSuccess) {
    delete s;
    return fail(SMAUG_E_HIP, "hipStreamCreate: %s", hipGetErrorString(e));
  }
  s->stream = s->own;
  const int nbuf = p->rkon == 1 ? 4 : 2;
  bool ok = true;
  for (int b = 0; b < nbuf; b++) ok &= hipMalloc(&s->U[b], bytes * s->np) == hipSuccess;
  ok &= hipMalloc(&s->bg, bytes * s->nb) == hipSuccess;
  const size_t pbytes = (s->G.mixed ? sizeof(float) : sizeof(double)) * (size_t)s->N;
  ok &= hipMalloc(&s->prim, pbytes * s->npr) == hipSuccess;
  if (s->G.mixed) ok &= hipMalloc(&s->shadow, sizeof(float) * (size_t)s->N * s->np) == hipSuccess;
  ok &= hipMalloc(&s->delx, bytes * s->nd) == hipSuccess;
  ok &= hipMalloc(&s->rdelx, bytes * s->nd) == hipSuccess;
  ok &= hipMalloc(&s->pos, bytes * s->nd) == hipSuccess;
  ok &= hipMalloc(&s->cmax, sizeof(unsigned long long) * 16) == hipSuccess;
  ok &= hipMalloc(&s->dts, sizeof(double) * 2) == hipSuccess;
  ok &= hipMalloc(&s->flag, sizeof(int)) == hipSuccess;
  if (!ok) {
    free_ctx(s);
    return fail(SMAUG_E_NOMEM, "device allocation failed");
  }
  initgrid_host(s->nd, p->n, pos, s->h_pos, s->h_delx);
  std::vector<double> h_rdelx(s->h_delx.size());
  for (size_t q = 0; q < h_rdelx.size(); q++) h_rdelx[q] = 1.0 / s->h_delx[q];
  // tensor-product grid (delx along d depends on the d coordinate only, the
  // case of every grid built from per-axis positions): the kernels read
  // one spacing per coordinate instead of the nd*N arrays
  std::vector<double> h_dx1, h_rdx1;
  if (separable_interior(s->nd, p->n, s->h_delx, h_dx1)) {
    h_rdx1.resize(h_dx1.size());
    for (size_t q = 0; q < h_dx1.size(); q++) h_rdx1[q] = 1.0 / h_dx1[q];
    ok &= hipMalloc(&s->dx1, sizeof(double) * h_dx1.size()) == hipSuccess;
    ok &= hipMalloc(&s->rdx1, sizeof(double) * h_dx1.size()) == hipSuccess;
    ok = ok && hipMemcpy(s->dx1, h_dx1.data(), sizeof(double) * h_dx1.size(), hipMemcpyHostToDevice) == hipSuccess &&
         hipMemcpy(s->rdx1, h_rdx1.data(), sizeof(double) * h_dx1.size(), hipMemcpyHostToDevice) == hipSuccess;
    if (!ok) {
      free_ctx(s);
      return fail(SMAUG_E_NOMEM, "device allocation failed");
    }
  }
  // vertical driver on a grid whose positions along d depend on the d
  // coordinate only: its shape is a product of per-axis factors, formed
  // once here instead of three exponentials per cell and stage
  std::vector<double> h_pos1;
  double* d_pos1 = nullptr;
  if (p->driver == SMAUG_DRIVER_VERTICAL && separable_interior(s->nd, p->n, s->h_pos, h_pos1)) {
    ok &= hipMalloc(&s->dshape, sizeof(double) * h_pos1.size()) == hipSuccess;
    ok &= hipMalloc(&d_pos1, sizeof(double) * h_pos1.size()) == hipSuccess;
    if (!ok) {
      hipFree(d_pos1);
      free_ctx(s);
      return fail(SMAUG_E_NOMEM, "device allocation failed");
    }
    hipError_t te = hipMemcpy(d_pos1, h_pos1.data(), sizeof(double) * h_pos1.size(), hipMemcpyHostToDevice);
    if (te == hipSuccess) {
      launch_drvtab(s->G, s->stream, d_pos1, s->dshape);
      te = hipGetLastError();
      if (te == hipSuccess) te = hipStreamSynchronize(s->stream);
    }
    hipFree(d_pos1);
    if (te != hipSuccess) {
      free_ctx(s);
      return fail(SMAUG_E_HIP, "driver shape tables: %s", hipGetErrorString(te));
    }
  }
  const double dts0[2] = {p->moddton == 1 ? 1.0e-8 : p->dt, 0.0};  // src/iosmaug.c:105,333-336
  const unsigned long long z12[16] = {0};
  const int z = 0;
  if (hipMemcpy(s->U[0], w0, bytes * s->np, hipMemcpyHostToDevice) != hipSuccess ||
      hipMemcpy(s->bg, w0 + (size_t)s->np * s->N, bytes * s->nb, hipMemcpyHostToDevice) != hipSuccess ||
      hipMemcpy(s->delx, s->h_delx.data(), bytes * s->nd, hipMemcpyHostToDevice) != hipSuccess ||
      hipMemcpy(s->rdelx, h_rdelx.data(), bytes * s->nd, hipMemcpyHostToDevice) != hipSuccess ||
      hipMemcpy(s->pos, s->h_pos.data(), bytes * s->nd, hipMemcpyHostToDevice) != hipSuccess ||
      hipMemcpy(s->cmax, z12, sizeof z12, hipMemcpyHostToDevice) != hipSuccess ||
      hipMemcpy(s->dts, dts0, sizeof dts0, hipMemcpyHostToDevice) != hipSuccess ||
      hipMemcpy(s->flag, &z, sizeof z, hipMemcpyHostToDevice) != hipSuccess) {
    free_ctx(s);
    return fail(SMAUG_E_HIP, "initial upload failed");
  }
  s->qt = p->qt0;
  s->it = p->it0;
  s->cur = 0;
  launch_fill(s->G, s->stream, s->U[0]);  // src/iosmaug.c:480-488
  // every buffer a stage writes starts as the initial state, so ghost cells
  // no stage writes (fixed boundaries) hold their initial values in each
  for (int b = 1; b < nbuf; b++)
    if (hipMemcpyAsync(s->U[b], s->U[0], bytes * s->np, hipMemcpyDeviceToDevice, s->stream) != hipSuccess) {
      free_ctx(s);
      return fail(SMAUG_E_HIP, "initial copy of the stage buffers failed");
    }
  e = hipStreamSynchronize(s->stream);
  if (e != hipSuccess) {
    free_ctx(s);
    return fail(SMAUG_E_HIP, "initial boundary fill: %s", hipGetErrorString(e));
  }
  *out = s;
  return SMAUG_OK;
}

static RhsArgs rhs_args(smaug_t* s, const double* win, const double* base, double* wout, double hfrac,
                        double tdep, int slot) {
  RhsArgs A;
  A.win = win;
  A.wsh = s->G.mixed ? (const void*)s->shadow : (const void*)win;
  A.bg = s->bg;
  A.prim = s->prim;
  A.delx = s->delx;
  A.rdelx = s->rdelx;
  A.dx1 = s->dx1;
  A.rdx1 = s->rdx1;
  A.pos = s->pos;
  A.base = base;
  A.r1 = A.r2 = A.r3 = nullptr;
  A.wout = wout;
  A.cmax_bits = s->cmax + 4 * slot;
  A.zero_next = s->cmax + 4 * (slot ^ 1);
  A.dts = s->dts;
  A.dt_rule = 0;
  A.courant = s->p.courant;
  A.dtcap = s->p.dt;
  A.hfrac = hfrac;
  A.tdep = tdep;
  A.damp = 0.0;
  A.amap = s->amap;
  A.dshape = s->dshape;
  return A;
}

// rule by which the first stage of a step sets dt and the clock (RhsArgs)
static int dt_rule(const smaug_t* s) { return s->p.moddton == 1 ? 2 : 1; }

// one stage: prim of win into the current maxima slot, then the rhs
static void run_stage(smaug_t* s, const double* win, const double* base, double* wout, double hfrac, double tdep,
                      bool first, const double* r1, const double* r2, const double* r3) {
  const int slot = s->cslot;
  launch_prim(s->G, s->stream, win, s->bg, s->prim, s->shadow, s->cmax + 4 * slot, s->flag);
  RhsArgs A = rhs_args(s, win, base, wout, hfrac, tdep, slot);
  if (first) A.dt_rule = dt_rule(s);
  A.r1 = r1;
  A.r2 = r2;
  A.r3 = r3;
  launch_rhs(s->G, s->stream, A);
  s->cslot ^= 1;
}

// time factor of the driver in the coming step: sin(2 pi qt / P) for the
// vertical driver; the constant tdep of fluxtube1; spicule1's tdep in the
// step whose counter p->it is 1 (models/usersource.cu.spicule1:67), else 0
static double driver_tdep_at(const smaug_t* s, int it, double qt) {
  switch (s->p.driver) {
    case SMAUG_DRIVER_VERTICAL:
      return sin(2.0 * M_PI * qt / s->p.drv[1]);
    case SMAUG_DRIVER_TORSIONAL:
      return s->p.drv[1];
    case SMAUG_DRIVER_SPICULE1:
      return it == 1 ? s->p.drv[1] : 0.0;
    default:
      return 0.0;
  }
}
static double driver_tdep(const smaug_t* s) { return driver_tdep_at(s, s->it, s->qt); }

// One time step.  With a tape (device buffer of smaug_tape_doubles values)
// the stage inputs are written into it (w^n, then the three intermediate
// RK states, which the stages use in place of the context's buffers) and
// the step's dt, qt and driver time factor follow them.
static int step_once(smaug_t* s, double* tape = nullptr) {
  s->qt = s->qt + s->p.dt;  // p->qt += DT (src/iosmaug.c:636, quirk Q5)
  const double tdep = driver_tdep(s);
  const long long F = (long long)s->np * s->N;
  const size_t fbytes = sizeof(double) * (size_t)F;
  if (s->p.rkon == 0) {
    double* win = s->U[s->cur];
    double* wout = s->U[s->cur ^ 1];
    if (tape) HIPCHK(hipMemcpyAsync(tape, win, fbytes, hipMemcpyDeviceToDevice, s->stream));
    run_stage(s, win, win, wout, 1.0, tdep, true, nullptr, nullptr, nullptr);
    s->cur ^= 1;
    if (tape) launch_meta(s->stream, tape + F, s->dts, s->qt, tdep);
  } else {
    double* w0 = s->U[0];
    double* w1 = tape ? tape + F : s->U[1];
    double* w2 = tape ? tape + 2 * F : s->U[2];
    double* w3 = tape ? tape + 3 * F : s->U[3];
    if (tape) HIPCHK(hipMemcpyAsync(tape, w0, fbytes, hipMemcpyDeviceToDevice, s->stream));
    if (tape && s->G.has_fixed)  // fixed ghosts of the tape's stage buffers
      for (int k = 1; k <= 3; k++)
        HIPCHK(hipMemcpyAsync(tape + k * F, w0, fbytes, hipMemcpyDeviceToDevice, s->stream));
    run_stage(s, w0, w0, w1, 0.5, tdep, true, nullptr, nullptr, nullptr);
    run_stage(s, w1, w0, w2, 0.5, tdep, false, nullptr, nullptr, nullptr);
    run_stage(s, w2, w0, w3, 1.0, tdep, false, nullptr, nullptr, nullptr);
    run_stage(s, w3, w0, w0, 1.0 / 6.0, tdep, false, w1, w2, w3);
    if (tape) launch_meta(s->stream, tape + 4 * F, s->dts, s->qt, tdep);
  }
  s->it = s->it + 1;
  HIPCHK(hipGetLastError());
  return SMAUG_OK;
}

extern "C" int smaug_step(smaug_t* s, int nsteps) {
  if (!s || nsteps < 0) return fail(SMAUG_E_ARG, "bad arguments to smaug_step");
  for (int n = 0; n < nsteps; n++) {
    int rc = step_once(s);
    if (rc) return rc;
  }
  return SMAUG_OK;
}

static int check_flag(smaug_t* s) {
  int f = 0;
  HIPCHK(hipMemcpyAsync(&f, s->flag, sizeof f, hipMemcpyDeviceToHost, s->stream));
  HIPCHK(hipStreamSynchronize(s->stream));
  if (f) return fail(SMAUG_E_NUMERIC, "non-finite wave speed in the state (blow-up)");
  return SMAUG_OK;
}

extern "C" int smaug_sync(smaug_t* s) {
  if (!s) return fail(SMAUG_E_ARG, "null context");
  HIPCHK(hipStreamSynchronize(s->stream));
  return check_flag(s);
}

extern "C" int smaug_cfl(smaug_t* s, double* cmax_per_dim, double* dt) {
  if (!s) return fail(SMAUG_E_ARG, "null context");
  unsigned long long* slot = s->cmax + 8;
  launch_zero3(s->stream, slot);
  launch_prim(s->G, s->stream, s->U[s->cur], s->bg, s->prim, s->shadow, slot, s->flag);
  unsigned long long bits[3];
  double dts[2];
  HIPCHK(hipMemcpyAsync(bits, slot, sizeof bits, hipMemcpyDeviceToHost, s->stream));
  HIPCHK(hipMemcpyAsync(dts, s->dts, sizeof dts, hipMemcpyDeviceToHost, s->stream));
  HIPCHK(hipStreamSynchronize(s->stream));
  double cm[3];
  for (int d = 0; d < 3; d++) memcpy(&cm[d], &bits[d], sizeof(double));
  if (cmax_per_dim)
    for (int d = 0; d < s->nd; d++) cmax_per_dim[d] = cm[d];
  if (dt) {
    const double* dx = s->p.dx;
    *dt = s->p.moddton == 1 ? cfl_dt(cm[s->nd - 1], s->nd, dx[0], dx[1], dx[2], s->p.courant, s->p.dt) : dts[0];
  }
  return check_flag(s);
}

// ---- smaug_cfl_noalloc: the CFL reduction with no context and no allocation.
// Its scratch (maxima, flag, dt and t; slots kNa* of smaug_dev.h) is this
// file-scope device array: one copy per GPU, held until the process ends.
// Host code never passes the array's name to a kernel (on the host it is a
// stand-in, not a device address): it uses the address hipGetSymbolAddress
// returns for the current device, looked up once per device.
static __device__ __align__(256) unsigned long long scratch[SMAUG_NOALLOC_SCRATCH_BYTES / 8];
static_assert(kNoallocSlots * 8 <= SMAUG_NOALLOC_SCRATCH_BYTES, "scratch slots fit the stated size");

static std::mutex g_scratch_mu;
static constexpr int kMaxDevices = 64;
static unsigned long long* g_scratch_ptr[kMaxDevices];

static int scratch_ptr(unsigned long long** out) {
  int dev = -1;
  HIPCHK(hipGetDevice(&dev));
  if (dev < 0 || dev >= kMaxDevices) return fail(SMAUG_E_UNSUPPORTED, "device index %d out of range", dev);
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (!g_scratch_ptr[dev]) {
    void* ptr = nullptr;
    const hipError_t e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !ptr)
      return fail(SMAUG_E_HIP, "hipGetSymbolAddress(scratch): %s (code %d)", hipGetErrorString(e), (int)e);
    g_scratch_ptr[dev] = (unsigned long long*)ptr;
  }
  *out = g_scratch_ptr[dev];
  return SMAUG_OK;
}

extern "C" int smaug_cfl_noalloc(const smaug_params* p, const double* w_device, double* out_device,
                                 void* hip_stream) {
  if (!p || !w_device || !out_device) return fail(SMAUG_E_ARG, "null argument");
  int rc = check_params(p);
  if (rc) return rc;
  Geo G;
  make_geo(p, G);
  G.mixed = 0;  // wave speeds from the FP64 state; no shadow, no derived fields
  unsigned long long* sc = nullptr;
  rc = scratch_ptr(&sc);
  if (rc) return rc;
  rc = check_range(w_device, sizeof(double) * (size_t)(G.np + 2 + G.nd) * G.N, "w_device");
  if (!rc) rc = check_range(out_device, sizeof(double) * (G.nd + 2), "out_device");
  if (rc) return rc;
  hipStream_t st = (hipStream_t)hip_stream;
  const double* bg = w_device + (size_t)G.np * G.N;
  launch_noalloc_init(st, sc, p->dt);  // src/iosmaug.c:549-550: every step starts from DT
  launch_prim(G, st, w_device, bg, nullptr, nullptr, sc + kNaCmax, reinterpret_cast<int*>(sc + kNaFlag));
  launch_dt(st, sc + kNaCmax, G.nd, p->dx, p->courant, p->dt, p->moddton, reinterpret_cast<double*>(sc + kNaDts));
  launch_noalloc_out(st, sc, G.nd, out_device);
  HIPCHK(hipGetLastError());
  return SMAUG_OK;
}

extern "C" int smaug_fill_ghosts(smaug_t* s) {
  if (!s) return fail(SMAUG_E_ARG, "null context");
  launch_fill(s->G, s->stream, s->U[s->cur]);
  HIPCHK(hipGetLastError());
  return SMAUG_OK;
}

extern "C" int smaug_get_state(const smaug_t* cs, double* w) {
  smaug_t* s = const_cast<smaug_t*>(cs);
  if (!s || !w) return fail(SMAUG_E_ARG, "null argument");
  const size_t bytes = sizeof(double) * (size_t)s->N;
  HIPCHK(hipMemcpyAsync(w, s->U[s->cur], bytes * s->np, hipMemcpyDeviceToHost, s->stream));
  HIPCHK(hipMemcpyAsync(w + (size_t)s->np * s->N, s->bg, bytes * s->nb, hipMemcpyDeviceToHost, s->stream));
  HIPCHK(hipStreamSynchronize(s->stream));
  return check_flag(s);
}

// fixed boundaries: a new current state brings new ghost values, which every
// stage buffer must hold (no stage writes them)
static int copy_fixed_ghosts(smaug_t* s) {
  if (!s->G.has_fixed) return SMAUG_OK;
  const int nbuf = s->p.rkon == 1 ? 4 : 2;
  for (int b = 0; b < nbuf; b++)
    if (b != s->cur)
      HIPCHK(hipMemcpyAsync(s->U[b], s->U[s->cur], sizeof(double) * (size_t)s->N * s->np, hipMemcpyDeviceToDevice,
                            s->stream));
  return SMAUG_OK;
}

extern "C" int smaug_set_state(smaug_t* s, const double* w) {
  if (!s || !w) return fail(SMAUG_E_ARG, "null argument");
  const size_t bytes = sizeof(double) * (size_t)s->N;
  HIPCHK(hipMemcpyAsync(s->U[s->cur], w, bytes * s->np, hipMemcpyHostToDevice, s->stream));
  HIPCHK(hipMemcpyAsync(s->bg, w + (size_t)s->np * s->N, bytes * s->nb, hipMemcpyHostToDevice, s->stream));
  launch_clear_flag(s->stream, s->flag);  // a blow-up of the old state no longer applies
  HIPCHK(hipGetLastError());
  int rc = copy_fixed_ghosts(s);
  if (rc) return rc;
  HIPCHK(hipStreamSynchronize(s->stream));
  return SMAUG_OK;
}

extern "C" int smaug_get_grid(const smaug_t* s, double* pos, double* delx) {
  if (!s) return fail(SMAUG_E_ARG, "null context");
  if (pos) memcpy(pos, s->h_pos.data(), sizeof(double) * s->h_pos.size());
  if (delx) memcpy(delx, s->h_delx.data(), sizeof(double) * s->h_delx.size());
  return SMAUG_OK;
}

extern "C" int smaug_write_out(smaug_t* s, const char* prefix, const char* name) {
  if (!s || !prefix) return fail(SMAUG_E_ARG, "null argument");
  std::vector<double> w((size_t)(s->np + s->nb) * s->N);
  int rc = smaug_get_state(s, w.data());
  if (rc != SMAUG_OK) return rc;
  int it = 0;
  double t = 0;
  rc = smaug_get_clock(s, &it, &t, nullptr, nullptr);
  if (rc != SMAUG_OK) return rc;
  // src/readwrite.c:222: <name>_<it>.out
  std::string path = std::string(prefix) + "_" + std::to_string(it) + ".out";
  return smaug_out_write(path.c_str(), name ? name : "", s->nd, s->p.n, w.data(), s->h_pos.data(), it, t,
                         s->p.gamma, s->p.eta, s->p.g);
}

extern "C" int smaug_get_clock(const smaug_t* cs, int* it, double* t, double* qt, double* dt_last) {
  smaug_t* s = const_cast<smaug_t*>(cs);
  if (!s) return fail(SMAUG_E_ARG, "null context");
  double dts[2];
  HIPCHK(hipMemcpyAsync(dts, s->dts, sizeof dts, hipMemcpyDeviceToHost, s->stream));
  HIPCHK(hipStreamSynchronize(s->stream));
  if (it) *it = s->it;
  if (t) *t = dts[1];
  if (qt) *qt = s->qt;
  if (dt_last) *dt_last = dts[0];
  return SMAUG_OK;
}

extern "C" int smaug_state_device_ptr(const smaug_t* s, void** dptr) {
  if (!s || !dptr) return fail(SMAUG_E_ARG, "null argument");
  *dptr = s->U[s->cur];
  return SMAUG_OK;
}

extern "C" int smaug_set_stream(smaug_t* s, void* stream) {
  if (!s) return fail(SMAUG_E_ARG, "null context");
  HIPCHK(hipStreamSynchronize(s->stream));
  s->stream = stream ? (hipStream_t)stream : s->own;
  return SMAUG_OK;
}

extern "C" int smaug_set_clock(smaug_t* s, int it, double qt) {
  if (!s) return fail(SMAUG_E_ARG, "null context");
  s->it = it;
  s->qt = qt;
  return SMAUG_OK;
}

extern "C" int smaug_save_pert(const smaug_t* cs, double* dst) {
  smaug_t* s = const_cast<smaug_t*>(cs);
  if (!s || !dst) return fail(SMAUG_E_ARG, "null argument");
  int rc = check_range(dst, sizeof(double) * (size_t)s->np * s->N, "smaug_save_pert destination");
  if (rc) return rc;
  HIPCHK(hipMemcpyAsync(dst, s->U[s->cur], sizeof(double) * (size_t)s->np * s->N, hipMemcpyDeviceToDevice,
                        s->stream));
  return SMAUG_OK;
}

extern "C" int smaug_load_pert(smaug_t* s, const double* src) {
  if (!s || !src) return fail(SMAUG_E_ARG, "null argument");
  int rc = check_range(src, sizeof(double) * (size_t)s->np * s->N, "smaug_load_pert source");
  if (rc) return rc;
  HIPCHK(hipMemcpyAsync(s->U[s->cur], src, sizeof(double) * (size_t)s->np * s->N, hipMemcpyDeviceToDevice,
                        s->stream));
  launch_fill(s->G, s->stream, s->U[s->cur]);
  launch_clear_flag(s->stream, s->flag);  // a blow-up of the old state no longer applies
  HIPCHK(hipGetLastError());
  return copy_fixed_ghosts(s);
}

// The differentiable path (driver amplitude map, taped steps, adjoint
// steps) runs only when SMAUG_ADJOINT=1 is set in the environment: its
// kernels are checked against the oracle in a host build but not yet on
// MI355X, where its first run ended in a GPU fault whose cause is not
// identified.
static int adjoint_gate(const char* what) {
  const char* e = getenv("SMAUG_ADJOINT");
  if (e && !strcmp(e, "1")) return SMAUG_OK;
  return fail(SMAUG_E_UNSUPPORTED, "%s is disabled unless SMAUG_ADJOINT=1 (not yet validated on MI355X)", what);
}

extern "C" int smaug_set_driver_map(smaug_t* s, const double* amap, int on_device) {
  if (!s) return fail(SMAUG_E_ARG, "null context");
  if (amap && adjoint_gate("smaug_set_driver_map")) return SMAUG_E_UNSUPPORTED;
  const size_t bytes = sizeof(double) * (size_t)(s->N / s->G.n[0]);
  if (!amap) {
    HIPCHK(hipStreamSynchronize(s->stream));
    hipFree(s->amap);
    s->amap = nullptr;
    return SMAUG_OK;
  }
  if (s->p.driver != SMAUG_DRIVER_VERTICAL)
    return fail(SMAUG_E_ARG, "a driver amplitude map needs driver = SMAUG_DRIVER_VERTICAL");
  if (on_device) {
    const int rc = check_range(amap, bytes, "driver amplitude map");
    if (rc) return rc;
  }
  if (!s->amap) HIPCHK(hipMalloc(&s->amap, bytes));
  HIPCHK(hipMemcpyAsync(s->amap, amap, bytes, on_device ? hipMemcpyDeviceToDevice : hipMemcpyHostToDevice,
                        s->stream));
  if (!on_device) HIPCHK(hipStreamSynchronize(s->stream));
  return SMAUG_OK;
}

extern "C" long long smaug_tape_doubles(const smaug_t* s) {
  if (!s) return fail(SMAUG_E_ARG, "null context");
  return (long long)(s->p.rkon == 1 ? 4 : 1) * s->np * s->N + 8;
}

extern "C" int smaug_step_taped(smaug_t* s, double* tape) {
  if (!s || !tape) return fail(SMAUG_E_ARG, "null argument");
  if (adjoint_gate("smaug_step_taped")) return SMAUG_E_UNSUPPORTED;
  if (s->G.divb) return fail(SMAUG_E_UNSUPPORTED, "the adjoint does not include the divB source terms");
  const int rc = check_range(tape, sizeof(double) * (size_t)smaug_tape_doubles(s), "tape");
  if (rc) return rc;
  return step_once(s, tape);
}

// Adjoint of one step (see include/smaug_hip.h).  Stage k of the forward
// step maps its input s_{k-1} (s_0 = w^n) to s_k; the adjoint runs the
// stages backwards, each as k_adj_mu -> k_prim(FP64) -> k_adj_rhs -> fold.
extern "C" int smaug_adjoint_step(smaug_t* s, const double* tape, const double* wnext, double* lam,
                                  double* gmap) {
  if (!s || !tape || !wnext || !lam) return fail(SMAUG_E_ARG, "null argument");
  if (adjoint_gate("smaug_adjoint_step")) return SMAUG_E_UNSUPPORTED;
  if (s->G.divb) return fail(SMAUG_E_UNSUPPORTED, "the adjoint does not include the divB source terms");
  const long long N = s->N, F = (long long)s->np * N;
  {
    const size_t fb = sizeof(double) * (size_t)F;
    int rc = check_range(tape, sizeof(double) * (size_t)smaug_tape_doubles(s), "tape");
    if (!rc) rc = check_range(wnext, fb, "wnext");
    if (!rc) rc = check_range(lam, fb, "lam");
    if (!rc && gmap) rc = check_range(gmap, sizeof(double) * (size_t)(N / s->G.n[0]), "gmap");
    if (rc) return rc;
  }
  if (!s->adj) {
    HIPCHK(hipMalloc(&s->adj, sizeof(double) * (size_t)(5 * F + N)));
    HIPCHK(hipMalloc(&s->aprim, sizeof(double) * (size_t)(s->npr * N)));
  }
  double* L1 = s->adj;
  double* L2 = L1 + F;
  double* L3 = L2 + F;
  double* MU = L3 + F;
  double* T = MU + F;
  double* gcell = T + F;
  Geo Gd = s->G;
  Gd.mixed = 0;  // the adjoint reads FP64 derived fields
  hipStream_t st = s->stream;
  unsigned long long* cmx = s->cmax + 12;
  const int nst = s->p.rkon == 1 ? 4 : 1;
  const double* meta = tape + nst * F;
  // every launch is checked as it is queued, so a failure names its kernel
  auto launched = [&](const char* what) -> int {
    const hipError_t e = hipGetLastError();
    return e == hipSuccess ? SMAUG_OK : fail(SMAUG_E_HIP, "%s launch: %s (code %d)", what, hipGetErrorString(e), (int)e);
  };
  auto stage = [&](const double* win, const double* lam_out, const double* outr, bool comb, double hfrac,
                   double cb, int base_set, double* target, bool first) -> int {
    AdjMuArgs M;
    memset(&M, 0, sizeof M);
    M.lam_out = lam_out;
    M.outr = outr;
    if (comb) {
      M.c0 = tape;
      M.c1 = tape + F;
      M.c2 = tape + 2 * F;
      M.c3 = tape + 3 * F;
      M.lam_r1 = L1;
      M.lam_r2 = L2;
      M.lam_r3 = L3;
    }
    M.bg = s->bg;
    M.pos = s->pos;
    M.amap = s->amap;
    M.meta = meta;
    M.hfrac = hfrac;
    M.cb = cb;
    M.base_set = base_set;
    M.mu = MU;
    M.lam_base = lam;
    M.gcell = gcell;
    M.gcell_set = first ? 1 : 0;
    launch_adj_mu(s->G, st, M);
    int rc = launched("k_adj_mu");
    if (rc) return rc;
    launch_zero3(st, cmx);
    if ((rc = launched("k_zero3"))) return rc;
    launch_prim(Gd, st, win, s->bg, s->aprim, nullptr, cmx, s->flag);
    if ((rc = launched("k_prim (adjoint stage input)"))) return rc;
    AdjArgs R;
    R.win = win;
    R.bg = s->bg;
    R.prim = s->aprim;
    R.delx = s->delx;
    R.rdelx = s->rdelx;
    R.dx1 = s->dx1;
    R.rdx1 = s->rdx1;
    R.mu = MU;
    R.cmax_bits = cmx;
    R.out = T;
    launch_adj_rhs(s->G, st, R);
    if ((rc = launched("k_adj_rhs"))) return rc;
    launch_adj_fold(s->G, st, T, target);
    return launched("k_adj_fold");
  };
  int rc = SMAUG_OK;
  if (s->p.rkon == 0) {
    rc = stage(tape, lam, wnext, false, 1.0, 0.0, 1, lam, true);
  } else {
    const double *w0 = tape, *s1 = tape + F, *s2 = tape + 2 * F, *s3 = tape + 3 * F;
    // final stage: out = w0 + h/6 acc(s3) + src, w^{n+1} = out + (s1 + 2 s2 + s3 - 4 w0)/3
    rc = stage(s3, lam, wnext, true, 1.0 / 6.0, -4.0 / 3.0, 1, L3, true);
    if (!rc) rc = stage(s2, L3, s3, false, 1.0, 0.0, 0, L2, false);
    if (!rc) rc = stage(s1, L2, s2, false, 0.5, 0.0, 0, L1, false);
    if (!rc) rc = stage(w0, L1, s1, false, 0.5, 0.0, 0, lam, false);
  }
  if (rc) return rc;
  if (gmap) {
    launch_colsum(s->G, st, gcell, gmap);
    return launched("k_colsum");
  }
  return SMAUG_OK;
}

// ---- tangent-linear run --------------------------------------------------
// The stage kernel and k_prim instantiated on Dual (value, tangent) arrays:
// the values follow the forward step from the context's current state, the
// tangents its derivative in the direction given at the start, with the
// hyperdiffusion coefficients, the wave-speed maxima and dt frozen at their
// values (the derivative the adjoint takes).  Own buffers, own maxima slots
// and clock: the context's state and clock are left as they are.

extern "C" int smaug_tl_begin(smaug_t* s, const double* dw0, const double* dbg, const double* damap) {
  if (!s || !dw0) return fail(SMAUG_E_ARG, "null argument");
  if (s->G.divb) return fail(SMAUG_E_UNSUPPORTED, "the tangent-linear step does not include the divB source terms");
  if (damap && !s->amap) return fail(SMAUG_E_ARG, "a driver-map direction needs a driver amplitude map (smaug_set_driver_map)");
  if ((unsigned long long)s->N * sizeof(Dual) >= (1ull << 32))
    return fail(SMAUG_E_ARG, "the tangent-linear step holds fewer than 2^28 cells");
  HIPCHK(hipStreamSynchronize(s->stream));
  free_tl(s);
  const long long F = (long long)s->np * s->N;
  const long long ncol = s->N / s->G.n[0];
  const int nbuf = s->p.rkon == 1 ? 4 : 2;
  bool ok = true;
  for (int b = 0; b < nbuf; b++) ok = ok && hipMalloc(&s->tlU[b], sizeof(Dual) * (size_t)F) == hipSuccess;
  const size_t pt = s->G.mixed ? sizeof(DualF) : sizeof(Dual);
  ok = ok && hipMalloc(&s->tlprim, pt * (size_t)(s->npr * s->N)) == hipSuccess;
  if (s->G.mixed) ok = ok && hipMalloc(&s->tlshadow, sizeof(DualF) * (size_t)F) == hipSuccess;
  ok = ok && hipMalloc(&s->tlbg, sizeof(Dual) * (size_t)(s->nb * s->N)) == hipSuccess;
  if (s->amap) ok = ok && hipMalloc(&s->tlamap, sizeof(Dual) * (size_t)ncol) == hipSuccess;
  ok = ok && hipMalloc(&s->tlcmax, sizeof(unsigned long long) * 8) == hipSuccess;
  ok = ok && hipMalloc(&s->tldts, sizeof(double) * 2) == hipSuccess;
  const long long B = (long long)s->nb * s->N;
  ok = ok && hipMalloc(&s->tltmp, sizeof(double) * (size_t)(2 * F > B ? 2 * F : B)) == hipSuccess;
  if (!ok) {
    free_tl(s);
    return fail(SMAUG_E_HIP, "tangent-linear buffers: allocation failed");
  }
  hipStream_t st = s->stream;
  // the direction with its ghost images (the maps are linear; a fixed
  // ghost keeps the value given), then value and tangent interleaved
  HIPCHK(hipMemcpyAsync(s->tltmp, dw0, sizeof(double) * (size_t)F, hipMemcpyHostToDevice, st));
  Geo Gt = s->G;
  Gt.mixed = 0;
  launch_fill(Gt, st, s->tltmp);
  launch_dual_pack(st, F, s->U[s->cur], s->tltmp, s->tlU[0]);
  for (int b = 1; b < nbuf; b++)  // fixed ghosts of every stage buffer hold the initial values
    HIPCHK(hipMemcpyAsync(s->tlU[b], s->tlU[0], sizeof(Dual) * (size_t)F, hipMemcpyDeviceToDevice, st));
  // the background and its direction (every cell, ghosts included, as given)
  if (dbg) HIPCHK(hipMemcpyAsync(s->tltmp, dbg, sizeof(double) * (size_t)B, hipMemcpyHostToDevice, st));
  launch_dual_pack(st, B, s->bg, dbg ? s->tltmp : nullptr, s->tlbg);
  if (s->tlamap) {
    double* dm = s->tltmp + F;
    if (damap)
      HIPCHK(hipMemcpyAsync(dm, damap, sizeof(double) * (size_t)ncol, hipMemcpyHostToDevice, st));
    launch_dual_pack(st, ncol, s->amap, damap ? dm : nullptr, s->tlamap);
  }
  launch_zero3(st, s->tlcmax);
  launch_zero3(st, s->tlcmax + 4);
  HIPCHK(hipMemcpyAsync(s->tldts, s->dts, sizeof(double) * 2, hipMemcpyDeviceToDevice, st));
  HIPCHK(hipGetLastError());
  HIPCHK(hipStreamSynchronize(st));  // the host arrays may go once this returns
  s->tlcur = 0;
  s->tlslot = 0;
  s->tlit = s->it;
  s->tlqt = s->qt;
  s->tldamp = 0.0;
  s->tl = true;
  return SMAUG_OK;
}

extern "C" int smaug_tl_driver_amplitude(smaug_t* s, double d_amplitude) {
  if (!s) return fail(SMAUG_E_ARG, "null context");
  if (!s->tl) return fail(SMAUG_E_ARG, "no tangent-linear run (smaug_tl_begin)");
  if (s->p.driver == SMAUG_DRIVER_NONE && d_amplitude != 0.0)
    return fail(SMAUG_E_ARG, "no driver: its amplitude has no direction");
  if (s->amap && d_amplitude != 0.0)
    return fail(SMAUG_E_ARG, "with a driver amplitude map the amplitude is the map: give its direction to smaug_tl_begin");
  if (!isfinite(d_amplitude)) return fail(SMAUG_E_ARG, "the amplitude direction is not finite");
  s->tldamp = d_amplitude;
  return SMAUG_OK;
}

static void tl_stage(smaug_t* s, const Geo& Gt, Dual* win, const Dual* base, Dual* wout, double hfrac, double tdep,
                     bool first, const Dual* r1, const Dual* r2, const Dual* r3) {
  hipStream_t st = s->stream;
  const int slot = s->tlslot;
  launch_prim_tl(Gt, st, win, s->tlbg, s->tlprim, s->tlshadow, s->tlcmax + 4 * slot, s->flag);
  RhsArgs A;
  A.win = (const double*)win;
  A.wsh = Gt.mixed ? (const void*)s->tlshadow : (const void*)win;
  A.bg = (const double*)s->tlbg;
  A.prim = s->tlprim;
  A.delx = s->delx;
  A.rdelx = s->rdelx;
  A.dx1 = s->dx1;
  A.rdx1 = s->rdx1;
  A.pos = s->pos;
  A.base = (const double*)base;
  A.r1 = (const double*)r1;
  A.r2 = (const double*)r2;
  A.r3 = (const double*)r3;
  A.wout = (double*)wout;
  A.cmax_bits = s->tlcmax + 4 * slot;
  A.zero_next = s->tlcmax + 4 * (slot ^ 1);
  A.dts = s->tldts;
  A.dt_rule = first ? dt_rule(s) : 0;
  A.courant = s->p.courant;
  A.dtcap = s->p.dt;
  A.hfrac = hfrac;
  A.tdep = tdep;
  A.damp = s->tldamp;
  A.amap = (const double*)s->tlamap;
  A.dshape = s->dshape;
  launch_rhs_tl(Gt, st, A);
  s->tlslot ^= 1;
}

extern "C" int smaug_tl_step(smaug_t* s, int nsteps) {
  if (!s || nsteps < 0) return fail(SMAUG_E_ARG, "bad arguments to smaug_tl_step");
  if (!s->tl) return fail(SMAUG_E_ARG, "no tangent-linear run (smaug_tl_begin)");
  const Geo& Gt = s->G;  // mixed: FP32 dual stencils over FP64 dual states
  for (int n = 0; n < nsteps; n++) {
    s->tlqt = s->tlqt + s->p.dt;  // as the forward step (quirk Q5)
    const double tdep = driver_tdep_at(s, s->tlit, s->tlqt);
    if (s->p.rkon == 0) {
      tl_stage(s, Gt, s->tlU[s->tlcur], s->tlU[s->tlcur], s->tlU[s->tlcur ^ 1], 1.0, tdep, true, nullptr, nullptr,
               nullptr);
      s->tlcur ^= 1;
    } else {
      Dual *w0 = s->tlU[0], *w1 = s->tlU[1], *w2 = s->tlU[2], *w3 = s->tlU[3];
      tl_stage(s, Gt, w0, w0, w1, 0.5, tdep, true, nullptr, nullptr, nullptr);
      tl_stage(s, Gt, w1, w0, w2, 0.5, tdep, false, nullptr, nullptr, nullptr);
      tl_stage(s, Gt, w2, w0, w3, 1.0, tdep, false, nullptr, nullptr, nullptr);
      tl_stage(s, Gt, w3, w0, w0, 1.0 / 6.0, tdep, false, w1, w2, w3);
    }
    s->tlit = s->tlit + 1;
    HIPCHK(hipGetLastError());
  }
  return SMAUG_OK;
}

extern "C" int smaug_tl_get(smaug_t* s, double* w, double* dw) {
  if (!s) return fail(SMAUG_E_ARG, "null context");
  if (!s->tl) return fail(SMAUG_E_ARG, "no tangent-linear run (smaug_tl_begin)");
  const long long F = (long long)s->np * s->N;
  hipStream_t st = s->stream;
  launch_dual_unpack(st, F, s->tlU[s->tlcur], s->tltmp, s->tltmp + F);
  HIPCHK(hipGetLastError());
  if (w) HIPCHK(hipMemcpyAsync(w, s->tltmp, sizeof(double) * (size_t)F, hipMemcpyDeviceToHost, st));
  if (dw) HIPCHK(hipMemcpyAsync(dw, s->tltmp + F, sizeof(double) * (size_t)F, hipMemcpyDeviceToHost, st));
  HIPCHK(hipStreamSynchronize(st));
  return check_flag(s);
}

extern "C" int smaug_tl_end(smaug_t* s) {
  if (!s) return fail(SMAUG_E_ARG, "null context");
  HIPCHK(hipStreamSynchronize(s->stream));
  free_tl(s);
  return SMAUG_OK;
}

extern "C" int smaug_destroy(smaug_t* s) {
  if (!s) return SMAUG_OK;
  hipStreamSynchronize(s->stream);
  free_ctx(s);
  return SMAUG_OK;
}

extern "C" const char* smaug_last_error(void) { return g_err.c_str(); }
extern "C" const char* smaug_version(void) { return "smaug-hip 0.1 (gfx950)"; }

// Times nsteps steps with HIP events on the context stream; reports the mean
// device time of one k_prim, one k_rhs and one full step.
extern "C" int smaug_time_kernels(smaug_t* s, int nsteps, double* ms_prim, double* ms_rhs, double* ms_step) {
  if (!s || nsteps < 1) return fail(SMAUG_E_ARG, "bad arguments");
  const int nst = s->p.rkon == 1 ? 4 : 1;
  hipEvent_t ev[2 * 4 * 2 + 2];
  for (auto& e : ev) HIPCHK(hipEventCreate(&e));
  double tp = 0, tr = 0, ts = 0;
  for (int n = 0; n < nsteps; n++) {
    s->qt = s->qt + s->p.dt;
    const double tdep = driver_tdep(s);
    HIPCHK(hipEventRecord(ev[16], s->stream));
    for (int st = 0; st < nst; st++) {
      double *win, *base, *wout;
      const double *r1 = nullptr, *r2 = nullptr, *r3 = nullptr;
      double hf;
      if (s->p.rkon == 0) {
        win = base = s->U[s->cur];
        wout = s->U[s->cur ^ 1];
        hf = 1.0;
      } else {
        win = s->U[st];
        base = s->U[0];
        wout = st == 3 ? s->U[0] : s->U[st + 1];
        hf = st == 2 ? 1.0 : (st == 3 ? 1.0 / 6.0 : 0.5);
        if (st == 3) {
          r1 = s->U[1];
          r2 = s->U[2];
          r3 = s->U[3];
        }
      }
      const int slot = s->cslot;
      HIPCHK(hipEventRecord(ev[4 * st + 0], s->stream));
      launch_prim(s->G, s->stream, win, s->bg, s->prim, s->shadow, s->cmax + 4 * slot, s->flag);
      HIPCHK(hipEventRecord(ev[4 * st + 1], s->stream));
      RhsArgs A = rhs_args(s, win, base, wout, hf, tdep, slot);
      if (st == 0) A.dt_rule = dt_rule(s);
      A.r1 = r1;
      A.r2 = r2;
      A.r3 = r3;
      HIPCHK(hipEventRecord(ev[4 * st + 2], s->stream));
      launch_rhs(s->G, s->stream, A);
      HIPCHK(hipEventRecord(ev[4 * st + 3], s->stream));
      s->cslot ^= 1;
    }
    HIPCHK(hipEventRecord(ev[17], s->stream));
    HIPCHK(hipEventSynchronize(ev[17]));
    for (int st = 0; st < nst; st++) {
      float a = 0, b = 0;
      HIPCHK(hipEventElapsedTime(&a, ev[4 * st + 0], ev[4 * st + 1]));
      HIPCHK(hipEventElapsedTime(&b, ev[4 * st + 2], ev[4 * st + 3]));
      tp += a;
      tr += b;
    }
    float c = 0;
    HIPCHK(hipEventElapsedTime(&c, ev[16], ev[17]));
    ts += c;
    if (s->p.rkon == 0) s->cur ^= 1;
    s->it++;
  }
  for (auto& e : ev) hipEventDestroy(e);
  if (ms_prim) *ms_prim = tp / (nsteps * nst);
  if (ms_rhs) *ms_rhs = tr / (nsteps * nst);
  if (ms_step) *ms_step = ts / nsteps;
  return check_flag(s);
}
