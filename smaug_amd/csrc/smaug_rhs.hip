// smaug_rhs.hip -- tiled right-hand side of one SMAUG stage (k_rhs).
//
// One workgroup owns a tile of interior cells (TileT: 8x4x8 or 8x8x8 in 3D,
// 16x16 in 2D; one cell or a pair along dim 0 per thread) and builds every
// term of the reference step for it from LDS-staged data, so each
// intermediate is computed once:
//   1. flux phase, per direction d: the fluxes F_f^d of the tile extended by
//      two cells along d go to LDS, then each thread takes the 4th-order
//      divergence (centdiff1/centdiff2).
//   2. hyperdiffusion phase, per variable q (rho, e_int, v_f, b_f): q is
//      staged as the tile plus a 3-cell halo (with the reference's halo
//      substitutions of quirks Q7/Q8); every direction's window of a cell
//      gives nu_{i+-1/2}, the diagonal sources and the cross-term products of
//      the off-diagonal momentum and magnetic sources, which are also formed
//      on the layer outside the tile along the cross direction; after a
//      barrier each thread takes the products' differences.  The v_f phase
//      also applies the background energy terms, which need gradients of v_f
//      only.
//   3. gravity, the stage update, the user source, the RK combination and
//      the ghost-cell images (boundaries fused).
// The stencils work in the stencil precision SH: FP64 (the state itself),
// or, in mixed precision, FP32 -- the shadows k_prim writes, FP32 LDS boxes
// and FP32 arithmetic, which halves the LDS and most of the registers of a
// workgroup and so raises the number resident per CU.  A cell's own values in
// the stencils come from the shadows too (rho_t: the FP32 rho plus the FP64
// rho_b, rounded; m_f at the faces: rho_t v_f): with the FP64 rho instead a
// step's errors against 64 bits agree to five digits (64^3 to 256^3).  The
// background terms, gravity, the stage update (base + h*acc), the driver and
// the RK combination are formed from FP64 values in both.
//
// What bounds it and how that shaped the code (MI355X):
//  * a tile's phases are a chain of memory round trips and barriers, so time
//    falls with every workgroup more that a CU holds: sums are pinned phase
//    by phase (pin) and loads of the own cell repeated rather than kept, which
//    took the FP64 kernel from 150 to 109 VGPRs, and its LDS from 52 to 34 KB:
//    four workgroups per CU instead of three (FP64, k_rhs at 128^3: 0.676 ->
//    0.510 ms; FP32 0.470 -> 0.411);
//  * the code of a tile at the grid's edge (masks, halo substitutions, ghost
//    images) streamed 211 KB of instructions through caches of 64 KB per two
//    CUs; loops in place of unrolled bodies made it 50 KB (one tile by itself:
//    73 -> 48 us);
//  * on grids of few tiles nothing hides a round trip: those keep every box
//    in LDS at once (ALL: 6 barriers for 20, 48 -> 33 us per tile);
//  * on large FP64 grids the boxes' traffic beyond L2 bounds it: 256^3 moves
//    15.0 GB in and 1.7 GB out per launch, 4.7 TB/s of the 4.74 that a plain
//    copy reaches.  Two cells per thread share addresses and the interface
//    between them (22 % fewer VALU, 26 % fewer LDS and 55 % fewer vector memory
//    instructions than the small tile, whose boxes are 25 % larger per cell
//    but mostly found in L2: 15.3 GB): k_rhs at 256^3 4.61 ms before, 3.75
//    with the small tile, 3.54 with the wide one.
#include <math.h>

#include <type_traits>

#include "../../include/smaug_hip.h"
#include "smaug_dev.h"
#include "smaug_ops.h"

namespace smaug {

// Tile of interior cells a workgroup owns: X x Y x Z, XC cells per thread
// (neighbours along dim 0).
template <int ND_, int X_, int Y_, int Z_, int XC_>
struct TileT {
  static constexpr int ND = ND_, X = X_, Y = Y_, Z = Z_, XC = XC_, NT = X_ * Y_ * Z_ / XC_;
};

__host__ __device__ constexpr int imax(int a, int b) { return a > b ? a : b; }
__host__ __device__ constexpr int imin(int a, int b) { return a < b ? a : b; }

template <class TL>
struct Lay {
  static constexpr int ND = TL::ND, XC = TL::XC, NT = TL::NT;
  static constexpr int TX = TL::X, TY = TL::Y, TZ = TL::Z;
  static constexpr int NP = 2 + 2 * ND;
  // halo widths along dim 0: with two cells per thread each box starts an
  // even number of cells before the tile, so a thread's pair is aligned
  static constexpr int HX = XC == 2 ? 4 : 3, RX = XC == 2 ? 2 : 1;
  // q box: tile + 3-cell halo
  static constexpr int QX = TX + 2 * HX, QY = TY + 6, QZ = ND == 3 ? TZ + 6 : 1;
  static constexpr int QN = QX * QY * QZ;
  // region: tile extended by one cell along one axis
  static constexpr int RN = ND == 3 ? imax(imax((TX + 2 * RX) * TY * TZ, TX * (TY + 2) * TZ), TX * TY * (TZ + 2))
                                    : imax((TX + 2 * RX) * TY, TX * (TY + 2));
  // flux region: tile extended by two cells along one axis
  static constexpr int FN = ND == 3 ? imax(imax((TX + 4) * TY * TZ, TX * (TY + 4) * TZ), TX * TY * (TZ + 4))
                                    : imax((TX + 4) * TY, TX * (TY + 4));
  // q box and the ND region arrays of a phase: one product per cross
  // direction and the sum of their energy products
  static constexpr int HYP = QN + ND * RN;
  static constexpr int FLX = (NP - 1) * FN;  // the flux of b_d along d is zero and not kept
  // rho_t on the tile + 1-cell halo, ahead of the area the phases share
  static constexpr int PX = TX + 2 * RX, PY = TY + 2, PZ = ND == 3 ? TZ + 2 : 1;
  static constexpr int PN = PX * PY * PZ;
  static constexpr int SHR = imax(HYP, FLX);  // area the phases share
  // spacing table of a tensor-product grid: delx and 1/delx at the tile's
  // coordinates along each axis
  static constexpr int DXT = TX + TY + TZ;
  static constexpr int DXO = imax(PN + SHR, 2 * QN);  // (the rho and q_e boxes are staged together)
  static constexpr int SMEM = DXO + 2 * DXT;
  // the same with every box, every direction's fluxes and the products of a
  // group of phases at once
  static constexpr int DXO_ALL = imax(PN + NP * QN + ND * ND * RN, ND * FLX);
  static constexpr int SMEM_ALL = DXO_ALL + 2 * DXT;
  static_assert(XC == 1 || (QN % 2 == 0 && RN % 2 == 0 && FN % 2 == 0 && PN % 2 == 0), "pairs stay aligned");
};

// Source cell of the q box's entry at grid coordinates x: the cell itself;
// 5 for coordinate -1 (left-chain halo, quirk Q8); for coordinate n the
// right-chain stray halo (quirk Q7, halo_r_src, here in 32 bits), -1 where
// that one is 0.  Entries further out, and those outside along two
// directions, are in no window of an interior cell: they get some cell.
template <int ND>
__device__ __forceinline__ int q_source(const Geo& G, int x0, int x1, int x2) {
  const int n0 = G.n[0], n1 = G.n[1], n2 = ND == 3 ? G.n[2] : 1;
  const int y0 = x0 == -1 ? 5 : imin(imax(x0, 0), n0 - 1);
  const int y1 = x1 == -1 ? 5 : imin(imax(x1, 0), n1 - 1);
  const int y2 = ND == 3 ? (x2 == -1 ? 5 : imin(imax(x2, 0), n2 - 1)) : 0;
  int c = (y2 * n1 + y1) * n0 + y0;
  if (x0 == n0 || x1 == n1 || (ND == 3 && x2 == n2)) {
    const int pz = ND == 3 ? x2 + 1 : 0;
    const int h = (pz * (n1 + 2) + x1 + 1) * (n0 + 2) + x0 + 1 - (ND == 3 ? n0 * n1 : 0) - n0 - 1;
    const int t = ((ND == 3 ? imin(pz, n2 - 1) : 0) * n1 + imin(x1 + 1, n1 - 1)) * n0 + imin(x0 + 1, n0 - 1);
    c = h >= imax(t, 0) && h < n0 * n1 * n2 ? h : -1;
  }
  return c;
}

// q box of a tile whose box crosses the grid edge: in batches of NB cells
// per thread, every source first, then the NB loads in flight together, then
// the stores.  (A loop, to keep the code small: the edge tiles' code streams
// through the instruction cache of every CU.)
template <class TL, typename SH>
__device__ __forceinline__ void stage_q_edge(const Geo& G, const SH* __restrict__ qa, SH* __restrict__ qb, const int* o) {
  using L = Lay<TL>;
  constexpr int ND = L::ND, NB = ND == 3 ? 4 : 1;
#pragma unroll 1
  for (int l0 = threadIdx.x; l0 < L::QN; l0 += L::NT * NB) {
    int src[NB];
#pragma unroll
    for (int k = 0; k < NB; k++) {
      const int l = imin(l0 + L::NT * k, L::QN - 1);
      const int a = l % L::QX, b = (l / L::QX) % L::QY, c = l / (L::QX * L::QY);
      src[k] = q_source<ND>(G, o[0] - L::HX + a, o[1] - 3 + b, ND == 3 ? o[2] - 3 + c : 0);
    }
    SH v[NB];
#pragma unroll
    for (int k = 0; k < NB; k++) v[k] = src[k] >= 0 ? at(qa, (unsigned)src[k]) : SH(0);
#pragma unroll
    for (int k = 0; k < NB; k++)
      if (l0 + L::NT * k < L::QN) qb[l0 + L::NT * k] = v[k];
  }
}

// q box (tile + 3-cell halo) of one field on its way to LDS: load() issues
// this thread's global loads, store() writes them (of an edge tile store()
// does both).  Each thread owns columns
// along dim 2 of XC neighbouring cells, and, where the workgroup has threads
// enough, a part of the planes.
template <class TL, typename SH, bool EDGE>
struct QBox {
  using L = Lay<TL>;
  static constexpr int ND = L::ND, XC = L::XC;
  static constexpr int NPC = L::QX / XC * L::QY;                 // columns
  static constexpr int NKF = (NPC + L::NT - 1) / L::NT;          // columns per thread
  static constexpr int NG = imax(1, L::NT / NPC);                // parts of the planes
  static constexpr int PG = L::QZ / NG;                          // planes per part
  static_assert(PG * NG == L::QZ, "the parts are equal");
  SH v[NKF][PG][XC];

  __device__ static __forceinline__ bool inside(const Geo& G, const int* o) {
    if (!EDGE) return true;
    bool in = o[0] >= L::HX && o[1] >= 3 && o[0] + L::TX + L::HX <= G.n[0] && o[1] + L::TY + 3 <= G.n[1];
    if (ND == 3) in = in && o[2] >= 3 && o[2] + L::TZ + 3 <= G.n[2];
    return in;
  }
  // (threads without a column load one again, so the loads are
  // unconditional and their registers have no other definition to merge)
  __device__ __forceinline__ void get(const Geo& G, const SH* __restrict__ qa, const int* o) {
    const unsigned zs = (unsigned)G.n[0] * (unsigned)G.n[1];
#pragma unroll
    for (int k = 0; k < NKF; k++) {
      const int t = threadIdx.x + L::NT * k;
      const int gt = NG > 1 ? t / NPC : 0, g = gt < NG ? gt : 0, lt = t - gt * NPC, l = lt < NPC ? lt : 0;
      const int a = XC * (l % (L::QX / XC)), b = l / (L::QX / XC);
      // the box's far edges and corners are in no window: their columns load
      // values that others load anyway
      const bool yin = b >= 2 && b < L::TY + 4;
      const int xa = yin ? a : imin(imax(a, L::HX - XC), L::HX + L::TX);
      const bool out = ND == 3 && !(yin && a >= L::HX - XC && a <= L::HX + L::TX);
      const bool lo = out && g == 0, hi = out && g == NG - 1;
      const unsigned g0 = cix(G, o[0] - L::HX + xa, o[1] - 3 + b, ND == 3 ? o[2] - 3 + g * PG : 0);
#pragma unroll
      for (int c = 0; c < PG; c++) {
        unsigned z = c * zs;
        if (ND == 3 && c < 2) z = lo ? 2 * zs : z;
        if (ND == 3 && c >= PG - 2) z = hi ? (PG - 3) * zs : z;
        ldg<XC>(qa, g0 + z, v[k][c]);
      }
    }
  }
  __device__ __forceinline__ void put(SH* __restrict__ qb) {
#pragma unroll
    for (int k = 0; k < NKF; k++) {
      const int t = threadIdx.x + L::NT * k;
      const int g = NG > 1 ? t / NPC : 0, l = t - g * NPC;
      if (g < NG && l < NPC) {
        const int a = XC * (l % (L::QX / XC)), b = l / (L::QX / XC);
#pragma unroll
        for (int c = 0; c < PG; c++) stl<XC>(qb + a + L::QX * (b + L::QY * (g * PG + c)), v[k][c]);
      }
    }
  }
  __device__ __forceinline__ void load(const Geo& G, const SH* __restrict__ qa, const int* o) {
    if constexpr (!EDGE) get(G, qa, o);
  }
  __device__ __forceinline__ void store(const Geo& G, const SH* __restrict__ qa, SH* __restrict__ qb, const int* o) {
    if constexpr (!EDGE) {
      put(qb);
    } else if (inside(G, o)) {
      get(G, qa, o);
      put(qb);
    } else {
      stage_q_edge<TL, SH>(G, qa, qb, o);
    }
  }
};

// rho_t = rho + rho_b on the tile + 1-cell halo (the sum in the background's
// precision, rounded to the stencils'); cells outside the grid hold 0
template <class TL, typename SH, bool EDGE>
__device__ __forceinline__ void stage_rho_t(const Geo& G, const SH* __restrict__ ws, const typename OwnT<SH>::T* __restrict__ bg,
                                   SH* __restrict__ cb, const int* o) {
  using L = Lay<TL>;
  using OT = typename OwnT<SH>::T;
  constexpr int ND = L::ND, XC = L::XC, NC = L::PN / XC, NK = (NC + L::NT - 1) / L::NT;
  const OT* __restrict__ rb = bg + (long long)bRHOB() * G.N;
  SH r[NK][XC];
  OT b[NK][XC];
#pragma unroll
  for (int k = 0; k < NK; k++) {
    const int l = threadIdx.x + L::NT * k;
    const int a = XC * (l % (L::PX / XC)), q = l / (L::PX / XC);
    const int x[3] = {o[0] - L::RX + a, o[1] - 1 + q % L::PY, ND == 3 ? o[2] - 1 + q / L::PY : 0};
    if (l < NC) {
      if (!EDGE) {
        const unsigned c = cix(G, x[0], x[1], x[2]);
        ldg<XC>(ws, c, r[k]);
        ldg<XC>(rb, c, b[k]);
      } else {
#pragma unroll
        for (int u = 0; u < XC; u++) {
          const int y[3] = {x[0] + u, x[1], x[2]};
          const bool in = in_grid<ND>(G, y);
          const unsigned c = in ? cix(G, y[0], y[1], y[2]) : 0u;
          r[k][u] = in ? at(ws, c) : SH(0);
          b[k][u] = in ? at(rb, c) : OT(0.0);
        }
      }
    }
  }
#pragma unroll
  for (int k = 0; k < NK; k++) {
    const int l = threadIdx.x + L::NT * k;
    if (l < NC) {
      SH s[XC];
#pragma unroll
      for (int u = 0; u < XC; u++) s[u] = (SH)(widen(r[k][u]) + b[k][u]);
      stl<XC>(cb + XC * l, s);
    }
  }
}

// The window of a thread's cells along direction D (0, 1, 2) of a q box:
// the values at offsets -2..2 of each cell and nu_{i+1/2}, nu_{i-1/2} (sc =
// delx * cmax * chyp).  The coefficient of an interface is a ratio of its own
// (see nu_ratios), so two neighbours along dim 0 share the one between them.
template <class TL, typename SH>
struct Win {
  using V = typename ValT<SH>::T;
  static constexpr int XC = TL::XC;
  SH q[XC][5];
  V nr[XC], nl[XC];
  template <int D>
  __device__ __forceinline__ void load(const SH* __restrict__ qb, int qc, int s, const V* sc) {
    if constexpr (D == 0 && XC == 2) {
      SH w[10];
#pragma unroll
      for (int k = 0; k < 10; k += 2) ldl<2>(qb + qc - 4 + k, w + k);
      V y[8];
#pragma unroll
      for (int k = 0; k < 8; k++) y[k] = valof(w[k + 1]);
      V R[3];
      nu_ratios<3>(y, R);
#pragma unroll
      for (int u = 0; u < 2; u++) {
#pragma unroll
        for (int k = 0; k < 5; k++) q[u][k] = w[2 + u + k];
        nl[u] = sc[u] * R[u];
        nr[u] = sc[u] * R[u + 1];
      }
    } else {
      SH w[7][XC];
#pragma unroll
      for (int k = 0; k < 7; k++) ldl<XC>(qb + qc + (k - 3) * s, w[k]);
#pragma unroll
      for (int u = 0; u < XC; u++) {
        V y[7];
#pragma unroll
        for (int k = 0; k < 7; k++) y[k] = valof(w[k][u]);
        V R[2];
        nu_ratios<2>(y, R);
        nl[u] = sc[u] * R[0];
        nr[u] = sc[u] * R[1];
#pragma unroll
        for (int k = 0; k < 5; k++) q[u][k] = w[1 + k][u];
      }
    }
  }
};

// The stage's dt.  The CFL rule is evaluated by every workgroup of the step's
// first stage, from the maxima that stage uses, rather than by a kernel of its
// own before it: 8 launches per RK4 step for 9, 2 per single-stage step for 3.
__device__ __forceinline__ double stage_dt(const Geo& G, const RhsArgs& A) {
  if (A.dt_rule != 2) return A.dts[0];
  return cfl_dt(__longlong_as_double((long long)A.cmax_bits[G.nd - 1]), G.nd, G.pdx[0], G.pdx[1], G.pdx[2], A.courant,
                A.dtcap);
}

// once per launch: the next stage's maxima back to zero, and in the step's
// first stage the clock (dts[0] is written under rule 2 only, where no
// workgroup reads it)
__device__ __forceinline__ void stage_head(const Geo& G, const RhsArgs& A) {
  if (blockIdx.x != 0) return;
  if (A.zero_next && threadIdx.x < 3) A.zero_next[threadIdx.x] = 0ull;
  if (A.dt_rule != 0 && threadIdx.x == 0) {
    const double dt = stage_dt(G, A);
    if (A.dt_rule == 2) A.dts[0] = dt;
    A.dts[1] = A.dts[1] + dt;
  }
}

// The user source and the divB terms of one interior cell (x0, x1, x2) with
// index c, on its updated values out.
template <int ND, typename OT>
__device__ __forceinline__ void add_source(const Geo& G, const RhsArgs& A, unsigned T, int x0, int x1, int x2, unsigned c,
                                           OT rho_c, OT rhob_c, double h, OT* out) {
  const long long N = G.N;
  const int x[3] = {x0, x1, x2};
  const OT* __restrict__ w = (const OT*)A.win;
  const OT* __restrict__ bg = (const OT*)A.bg;
  // divB source terms (divb_parallel, src/divb.cu:165-338, 2D), in FP64 on
  // cells 2 < i,j < n-2: divb from the 4th-order differences over 2 p->dx of
  // b + b_b, zeroed on the layers 3, n-4, n-3 (grad3d's mask with interior
  // transverse indices); m_d += h divb b_d, b_d += h divb m_d/rho_t (a NaN
  // source counts 0); the energy source multiplies wd[bdotv], which the
  // reference never fills, so it is 0
  if constexpr (sizeof(OT) == 8) {  // FP64 state only (the tangent-linear step excludes divB)
  if (ND == 2 && G.divb && x[0] > 2 && x[1] > 2 && x[0] < G.n[0] - 2 && x[1] < G.n[1] - 2) {
    auto g3 = [&](const double* a, int d) -> double {
      const int xd = x[d], nn = G.n[d];
      if (xd == 3 || xd == nn - 4 || xd == nn - 3) return 0.0;
      const unsigned s = d == 0 ? 1u : (unsigned)G.n[0];
      return ((8 * at(a, c + s) - 8 * at(a, c - s) + at(a, c - 2 * s) - at(a, c + 2 * s)) / 6.0) / (2.0 * G.pdx[d]);
    };
    const double divb = (g3(w + (long long)fB(ND, 0) * N, 0) + g3(w + (long long)fB(ND, 1) * N, 1)) +
                        (g3(bg + (long long)bBB(0) * N, 0) + g3(bg + (long long)bBB(1) * N, 1));
    const double rt = rho_c + rhob_c;
#pragma unroll
    for (int d = 0; d < ND; d++) {
      const double sm = -divb * at(w + (long long)fB(ND, d) * N, c);
      const double sb = -divb * at(w + (long long)fMOM(d) * N, c) / rt;
      out[fMOM(d)] -= h * (isnan(sm) ? 0.0 : sm);
      out[fB(ND, d)] -= h * (isnan(sb) ? 0.0 : sb);
    }
  }
  }
  // the drivers; spicule1's acts in the step whose counter is 1 only (tdep is
  // 0 outside it)
  if (!(T & SMAUG_T_SOURCE) || G.driver == SMAUG_DRIVER_NONE || (G.driver == SMAUG_DRIVER_SPICULE1 && A.tdep == 0.0)) return;
  const double* dv = G.drv;
  double ez, exyz;  // the shape: its factor along dim 0, the product of all
  double xp = 0.0, yp = 0.0;
  if (G.driver == SMAUG_DRIVER_VERTICAL && A.dshape) {  // separable grid: per-axis factors formed at set-up
    ez = A.dshape[x[0]];
    const double exx = A.dshape[G.n[0] + x[1]];
    exyz = exx * ez;
    if (ND == 3) exyz = exx * A.dshape[G.n[0] + G.n[1] + x[2]] * ez;
  } else {
    double t0, t1, t2 = 0.0;  // exponents along dims 0, 1, 2
    if (G.driver == SMAUG_DRIVER_SPICULE1) {  // at the grid positions xmin + i dx
      const double z1 = G.pxmin[0] + (double)x[0] * G.pdx[0] - dv[2];
      const double x1 = G.pxmin[1] + (double)x[1] * G.pdx[1] - dv[3];
      t0 = -(z1 * z1) / (dv[5] * dv[5]);
      t1 = -(x1 * x1) / (dv[6] * dv[6]);
    } else {
      const double zp = at(A.pos, c) - dv[2];
      xp = at(A.pos + N, c) - dv[3];
      t0 = -zp * zp / (dv[5] * dv[5]);
      t1 = -xp * xp / (dv[6] * dv[6]);
      if (ND == 3) {
        const double wy = G.driver == SMAUG_DRIVER_TORSIONAL ? dv[7] : dv[6];
        yp = at(A.pos + 2 * N, c) - dv[4];
        t2 = -yp * yp / (wy * wy);
      }
    }
    // one exponential in the code, evaluated along dims 1, 2, 0 (exp(0) = 1
    // for an axis without a factor)
    exyz = 1.0;
#pragma unroll 1
    for (int q = 0; q < 3; q++) {
      ez = exp(q == 0 ? t1 : (q == 1 ? t2 : t0));
      exyz = exyz * ez;
    }
  }
  const OT rto = out[fRHO()] + rhob_c;
  if (G.driver == SMAUG_DRIVER_VERTICAL) {
    // amplitude map: one amplitude per (j,k) column in place of
    // A exp(-dx^2/sxy^2 [- dy^2/sxy^2])
    const OT vz = A.amap ? ((const OT*)A.amap)[x[1] + (ND == 3 ? (long long)G.n[1] * x[2] : 0)] * ez * A.tdep
                         : with_tangent<OT>(dv[0] * exyz * A.tdep, A.damp * exyz * A.tdep);
    out[fMOM(0)] += h * vz * rto;
    out[fE(ND)] += h * (vz * vz) * rto / 2.0;
  } else if (G.driver == SMAUG_DRIVER_TORSIONAL) {  // fluxtube1's (models/usersource.cu.fluxtube1:3-90), 3D
    if constexpr (ND == 3) {
      const OT vx = with_tangent<OT>((dv[0] * yp / dv[9]) * exyz * A.tdep, (A.damp * yp / dv[9]) * exyz * A.tdep);
      const OT vy = with_tangent<OT>(-(dv[0] * xp / dv[8]) * exyz * A.tdep, -(A.damp * xp / dv[8]) * exyz * A.tdep);
      out[fMOM(1)] += h * vx * rto;
      out[fMOM(2)] += h * vy * rto;
      out[fE(ND)] += h * (vx * vx + vy * vy) * rto / 2.0;
    }
  } else {  // spicule1's (models/usersource.cu.spicule1:4-136)
    const OT vvz = with_tangent<OT>(dv[0] * exyz * A.tdep, A.damp * exyz * A.tdep);
    out[fMOM(0)] = out[fMOM(0)] + h * vvz * rto;
  }
}

// Ghost images of the interior cell x with values out: every combination of
// its images across the directions (a fixed direction has none; with n >= 8
// an interior coordinate feeds at most two ghosts per direction), with the
// asymm signs.  Loops over the combinations (indexed by a number in base 3,
// a digit per direction: 0 the cell's own coordinate, 1 and 2 its ghosts)
// and, where the fields' boundary types differ, over the fields, with no
// register array indexed at run time: the code stays small, as every edge
// tile streams it.
template <int ND, typename F>
__device__ __forceinline__ void each_image(const Geo& G, const int* bct, const int* x, F store) {
  const int t0 = bct[0], t1 = bct[1], t2 = bct[2];
  const Img2 I0 = bc_images2(t0, x[0], G.n[0], ND), I1 = bc_images2(t1, x[1], G.n[1], ND);
  const Img2 I2 = ND == 3 ? bc_images2(t2, x[2], G.n[2], ND) : Img2{0, 0, 0};
  if (I0.m + I1.m + I2.m == 0) return;
  const int x0 = x[0], x1 = x[1], x2 = x[2];
  const int a1 = I0.g0, a2 = I0.g1, b1 = I1.g0, b2 = I1.g1, c1 = I2.g0, c2 = I2.g1;
#pragma unroll 1
  for (int q = 1; q < (ND == 3 ? 27 : 9); q++) {
    const int a = q % 3, b = q / 3 % 3, c = q / 9;
    if (a > I0.m || b > I1.m || c > I2.m) continue;
    const unsigned cc = cix(G, a == 0 ? x0 : (a == 1 ? a1 : a2), b == 0 ? x1 : (b == 1 ? b1 : b2),
                            c == 0 ? x2 : (c == 1 ? c1 : c2));
    store(cc, ((a && t0 == BC_ASYMM) ^ (b && t1 == BC_ASYMM)) ^ (ND == 3 && c && t2 == BC_ASYMM));
  }
}
template <int ND, typename OT>
__device__ __forceinline__ void put_images(const Geo& G, OT* __restrict__ wo, const int* x, const OT* out) {
  constexpr int NP = 2 + 2 * ND;
  if (G.bc_uniform) {
    each_image<ND>(G, G.bct[0], x, [&](unsigned cc, bool minus) __attribute__((always_inline)) {
      // (a pointer per lane, stepped field by field: the bases of all fields
      // at once would take the scalar registers of the phases' pointers)
      OT* p = wo + cc;
#pragma unroll
      for (int f = 0; f < NP; f++, p += G.N) *p = pick(minus, -out[f], out[f]);
    });
  } else {
#pragma unroll 1
    for (int f = 0; f < NP; f++) {
      OT v = out[0];
#pragma unroll
      for (int q = 1; q < NP; q++) v = pick(f == q, out[q], v);
      OT* p = wo + (long long)f * G.N;
      each_image<ND>(G, G.bct[f], x, [&](unsigned cc, bool minus) __attribute__((always_inline)) { put(p, cc, pick(minus, -v, v)); });
    }
  }
}

// The terms of one tile whose origin (first interior cell) is o.  EDGE
// false: every cell of the tile lies in [5, n-6] along every direction, so
// no cell of it or of its halos is a ghost or on a zeroed layer, every
// staged box lies inside the grid and no cell has a ghost image; the
// boundary checks are then compiled out (the arithmetic is the same).
// SEP: the grid is a tensor product (A.dx1 set).
// ALL: every direction's fluxes, every q box and the products of a group of
// phases have their own place in LDS, so the phases need 6 barriers and 3
// trips to memory where the others take 20 and 11 (see k_rhs_small).
template <class TL, typename SH, bool EDGE, bool SEP, bool ALL>
__device__ __forceinline__ void rhs_tile(const Geo& G, const RhsArgs& A, SH* __restrict__ sm, const int* o) {
  using L = Lay<TL>;
  using AT = SH;                        // arithmetic type of the stencils
  using V = typename ValT<SH>::T;       // its values (coefficients carry no tangent)
  // own-cell type: FP64 (the own-cell update and the RK combination are
  // FP64 with FP32 stencils too), Dual in the tangent-linear step
  using OT = typename OwnT<SH>::T;
  constexpr int ND = L::ND, XC = L::XC, NP = L::NP;
  constexpr int TX = L::TX, TY = L::TY, TZ = L::TZ;
  const int tid = threadIdx.x;
  const int lc[3] = {tid % (TX / XC) * XC, (tid / (TX / XC)) % TY, ND == 3 ? tid / (TX / XC * TY) : 0};
  const int x[3] = {o[0] + lc[0], o[1] + lc[1], o[2] + lc[2]};  // first cell of the thread
  bool valid[XC], any = false;
#pragma unroll
  for (int u = 0; u < XC; u++) {
    const int y[3] = {x[0] + u, x[1], x[2]};
    valid[u] = !EDGE || interior_c<ND>(G, y);
    any = any || valid[u];
  }
  const long long N = G.N;
  const unsigned c = cix(G, x[0], x[1], x[2]);  // own cell (used by valid threads only)
  const OT* __restrict__ w = (const OT*)A.win;    // own-cell values
  const SH* __restrict__ ws = (const SH*)A.wsh;    // neighbour values (stencil precision)
  const OT* __restrict__ bg = (const OT*)A.bg;  // background (Dual in the tangent-linear step)
  const SH* __restrict__ pr = (const SH*)A.prim;
  const unsigned T = G.terms;
  AT acc[NP][XC];
#pragma unroll
  for (int f = 0; f < NP; f++)
#pragma unroll
    for (int u = 0; u < XC; u++) acc[f][u] = AT(0);

  auto pin_acc = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int f = 0; f < NP; f++)
#pragma unroll
      for (int u = 0; u < XC; u++) pin(acc[f][u]);
  };

  V* const SDX = reinterpret_cast<V*>(sm + (ALL ? L::DXO_ALL : L::DXO));  // spacing table (tensor-product grids)
  if (SEP && tid < L::DXT) {  // visible after the first barrier
    const int n0 = G.n[0], n1 = G.n[1], n2 = ND == 3 ? G.n[2] : 0, o0 = o[0], o1 = o[1], o2 = o[2];
    const bool d0 = tid < TX, d1 = tid < TX + TY;
    const int xx = d0 ? o0 + tid : (d1 ? o1 + tid - TX : o2 + tid - TX - TY);
    const int od = d0 ? 0 : (d1 ? n0 : n0 + n1);
    const bool ing = xx < (d0 ? n0 : (d1 ? n1 : n2));
    SDX[tid] = ing ? (V)A.dx1[od + xx] : V(1);
    SDX[L::DXT + tid] = ing ? (V)A.rdx1[od + xx] : V(1);
  }
  // delx and 1/delx along d at the thread's cells
  auto dxs = [&](int d, V* dx) __attribute__((always_inline)) {
    const int t = d == 0 ? lc[0] : (d == 1 ? TX + lc[1] : TX + TY + lc[2]);
#pragma unroll
    for (int u = 0; u < XC; u++)
      dx[u] = SEP ? SDX[t + (d == 0 ? u : 0)] : (valid[u] ? (V)at(A.delx + (long long)d * N, c + u) : V(1));
  };
  auto rdxs = [&](int d, V* rdx) __attribute__((always_inline)) {
    const int t = L::DXT + (d == 0 ? lc[0] : (d == 1 ? TX + lc[1] : TX + TY + lc[2]));
#pragma unroll
    for (int u = 0; u < XC; u++)
      rdx[u] = SEP ? SDX[t + (d == 0 ? u : 0)] : (valid[u] ? (V)at(A.rdelx + (long long)d * N, c + u) : V(1));
  };
  // XC values of an own-cell array (0 where the cell is not interior); the
  // index is pinned, so values that several phases read come from the cache
  // again and do not occupy registers between them
  auto own = [&](const auto* __restrict__ p, auto* v) __attribute__((always_inline)) {
    using E = std::remove_reference_t<decltype(v[0])>;
    unsigned cc = c;
    pin(cc);
    if (!EDGE || valid[XC - 1]) {  // the tile starts on an interior cell: the last one valid means all are
      ldg<XC>(p, cc, v);
    } else {
#pragma unroll
      for (int u = 0; u < XC; u++) v[u] = valid[u] ? at(p, cc + u) : E(0);
    }
  };

  const bool want_mom = G.hyper && (T & SMAUG_T_HMOM);
  const bool want_eterm = (T & SMAUG_T_ETERM) != 0;
  const bool want_b = G.hyper && (T & SMAUG_T_HB);

  // ------------------------------------------------------------ fluxes
  if (T & SMAUG_T_FLUX) {
    // the thread's own cells: their state is loaded once for every
    // direction; a second slot per direction covers the 2 + 2 halo layers
    // along it, its state loaded while the direction before it is summed
    CellState<ND, AT> S0[XC], S1;
    bool in0[XC];
    auto FB = [&](int d) __attribute__((always_inline)) { return sm + (ALL ? d * L::FLX : 0); };
#pragma unroll
    for (int u = 0; u < XC; u++) {
      const int y[3] = {x[0] + u, x[1], x[2]};
      in0[u] = !EDGE || in_grid<ND>(G, y);
    }
    if (in0[XC - 1]) {
      load_cells<ND, XC, SH, AT>(G, ws, bg, c, S0);
    } else {
#pragma unroll
      for (int u = 0; u < XC; u++)
        if (in0[u]) load_cell<ND, SH, AT>(G, ws, bg, c + u, S0[u]);
    }
    bool in1 = false;
    int l1 = 0;
    // halo slot of direction d: its state (or out of the grid) and its place
    auto halo = [&](int d) __attribute__((always_inline)) {
      const int ex[3] = {d == 0 ? 2 : 0, d == 1 ? 2 : 0, d == 2 ? 2 : 0};
      const int rx = TX + 2 * ex[0], ry = TY + 2 * ex[1];
      const int Td = d == 0 ? TX : (d == 1 ? TY : TZ);
      const int pa = d == 0 ? 1 : 0, qa = d == 2 ? 1 : 2;  // the other two axes
      const int Tp = pa == 0 ? TX : TY;
      const int Fd = Tp * (ND == 3 ? (qa == 1 ? TY : TZ) : 1);  // face of the tile across d
      in1 = false;
      l1 = -1;
      if (tid < 4 * Fd) {
        // along dim 0 the two layers of a side follow each other, so the
        // lanes of a wavefront read neighbouring cells
        const int layer = d == 0 ? tid % 2 + 2 * (tid / (2 * Fd)) : tid / Fd;
        const int r = d == 0 ? tid % (2 * Fd) / 2 : tid - layer * Fd;
        int rc[3] = {0, 0, 0};
        rc[d] = layer < 2 ? layer : Td + layer;  // region coordinates 0, 1 and Td+2, Td+3
        rc[pa] = r % Tp;
        if (ND == 3) rc[qa] = r / Tp;
        const int xr[3] = {o[0] - ex[0] + rc[0], o[1] - ex[1] + rc[1], ND == 3 ? o[2] - ex[2] + rc[2] : 0};
        in1 = !EDGE || in_grid<ND>(G, xr);
        l1 = rc[0] + rx * (rc[1] + ry * rc[2]);
        if (in1) load_cell<ND, SH, AT>(G, ws, bg, cix(G, xr[0], xr[1], xr[2]), S1);
      }
    };
    static_assert(ND == 3 ? 4 * TY * TZ <= L::NT && 4 * TX * TZ <= L::NT && 4 * TX * TY <= L::NT
                          : 4 * TX <= L::NT && 4 * TY <= L::NT,
                  "the halo layers of a direction fit one slot per thread");
    // the fluxes along d of the own cells and the halo slot to LDS
    auto form = [&](int d) __attribute__((always_inline)) {
      const int ex[3] = {d == 0 ? 2 : 0, d == 1 ? 2 : 0, d == 2 ? 2 : 0};
      const int rx = TX + 2 * ex[0], ry = TY + 2 * ex[1];
      // slot of field f (the flux of b_d along d is zero: not kept)
      auto slot = [&](int f) __attribute__((always_inline)) { return (f < fB(ND, d) ? f : f - 1) * L::FN; };
      const int l0 = (lc[0] + ex[0]) + rx * ((lc[1] + ex[1]) + ry * (lc[2] + ex[2]));
      {
        AT F[XC][NP];
#pragma unroll
        for (int u = 0; u < XC; u++) {
          if (in0[u]) {
            pin(S0[u]);
            fluxes_of<ND, AT>(G, S0[u], d, F[u]);
          } else {
#pragma unroll
            for (int f = 0; f < NP; f++) F[u][f] = AT(0);
          }
        }
#pragma unroll
        for (int f = 0; f < NP; f++) {
          if (f == fB(ND, d)) continue;
          AT p[XC];
#pragma unroll
          for (int u = 0; u < XC; u++) p[u] = F[u][f];
          stl<XC>(FB(d) + slot(f) + l0, p);
        }
      }
      if (l1 >= 0) {
        AT F[NP];
        if (in1) {
          fluxes_of<ND, AT>(G, S1, d, F);
        } else {
#pragma unroll
          for (int f = 0; f < NP; f++) F[f] = AT(0);
        }
#pragma unroll
        for (int f = 0; f < NP; f++)
          if (f != fB(ND, d)) FB(d)[slot(f) + l1] = F[f];
      }
    };
    // their divergence
    auto diverge = [&](int d) __attribute__((always_inline)) {
      const int ex[3] = {d == 0 ? 2 : 0, d == 1 ? 2 : 0, d == 2 ? 2 : 0};
      const int rx = TX + 2 * ex[0], ry = TY + 2 * ex[1];
      // slot of field f (the flux of b_d along d is zero: not kept)
      auto slot = [&](int f) __attribute__((always_inline)) { return (f < fB(ND, d) ? f : f - 1) * L::FN; };
      const int l0 = (lc[0] + ex[0]) + rx * ((lc[1] + ex[1]) + ry * (lc[2] + ex[2]));
      V inv[XC];
      rdxs(d, inv);
      bool z[XC];
#pragma unroll
      for (int u = 0; u < XC; u++) {
        inv[u] *= V(1.0 / 12.0);
        z[u] = !valid[u] || z4e<EDGE>(G, zFLUX(ND), d, x[d] + (d == 0 ? u : 0));
      }
      const int s = d == 0 ? 1 : (d == 1 ? rx : rx * ry);
#pragma unroll
      for (int f = 0; f < NP; f++) {
        if (f == fB(ND, d)) continue;
        const AT* Fp = FB(d) + slot(f) + l0;
        AT a[XC], b[XC], e[XC], g[XC];  // F at i-2, i-1, i+1, i+2
        if (d == 0 && XC == 2) {
          AT m[XC], p[XC], q[XC];
          ldl<XC>(Fp - 2, m);
          ldl<XC>(Fp, p);
          ldl<XC>(Fp + 2, q);
          a[0] = m[0];
          b[0] = a[XC - 1] = m[XC - 1];
          b[XC - 1] = p[0];
          e[0] = p[XC - 1];
          g[0] = e[XC - 1] = q[0];
          g[XC - 1] = q[XC - 1];
        } else {
          ldl<XC>(Fp - 2 * s, a);
          ldl<XC>(Fp - s, b);
          ldl<XC>(Fp + s, e);
          ldl<XC>(Fp + 2 * s, g);
        }
#pragma unroll
        for (int u = 0; u < XC; u++)
          acc[f][u] -= z[u] ? AT(0) : ((V(8) * e[u] - V(8) * b[u]) + (a[u] - g[u])) * inv[u];
      }
      pin_acc();
    };
    halo(0);
#pragma unroll
    for (int d = 0; d < ND; d++) {
      form(d);
      if (d + 1 < ND) halo(d + 1);
      if (!ALL) {
        __syncthreads();
        diverge(d);
        __syncthreads();
      }
    }
    if (ALL) {
      __syncthreads();
#pragma unroll
      for (int d = 0; d < ND; d++) diverge(d);
      __syncthreads();
    }
  } else if (SEP) {
    __syncthreads();  // the spacing table
  }

  // ------------------------------------------------------------ hyperdiffusion + energy terms
  SH* const CBX = sm;                                  // rho_t (tile + 1)
  // q box i (ALL: rho, q_e, v_f, b_f; else the one of the phase), region
  // arrays of phase f: products of the cross directions, energy
  auto QB = [&](int i) __attribute__((always_inline)) { return sm + L::PN + (ALL ? i * L::QN : 0); };
  auto NRF = [&](int f) __attribute__((always_inline)) { return sm + L::PN + (ALL ? NP * L::QN + f * ND * L::RN : L::QN); };
  constexpr int QV = 2, QM = 2 + ND;  // boxes of v_0 and b_0
  // tile-cell index in the q box and its strides
  const int qc = (lc[0] + L::HX) + L::QX * ((lc[1] + 3) + L::QY * (ND == 3 ? lc[2] + 3 : 0));
  const int qs[3] = {1, L::QX, L::QX * L::QY};
  const int pc = (lc[0] + L::RX) + L::PX * ((lc[1] + 1) + L::PY * (ND == 3 ? lc[2] + 1 : 0));
  const int ps[3] = {1, L::PX, L::PX * L::PY};

  V cm[ND];
#pragma unroll
  for (int d = 0; d < ND; d++) cm[d] = (V)__longlong_as_double((long long)A.cmax_bits[d]);
  auto scales = [&](int d, V k, V* sc) __attribute__((always_inline)) {
    dxs(d, sc);
#pragma unroll
    for (int u = 0; u < XC; u++) sc[u] *= cm[d] * k;
  };

  const bool mom_phases = want_mom || want_eterm;
  QBox<TL, SH, EDGE> Q;  // the next q box on its way

  // rho (src/hyperdifrhosource1.cu) and e_int (src/hyperdifesource1.cu):
  // both boxes are staged in one round trip (ahead of the rho_t box's use)
  const bool h_rho = G.hyper && (T & SMAUG_T_HRHO), h_e = G.hyper && (T & SMAUG_T_HE);
  const SH* qe = pr + (long long)pQE(ND) * N;
  SH* const box_rho = ALL ? QB(0) : sm;
  SH* const box_e = ALL ? QB(1) : sm + L::QN;
  if (ALL) {  // every box that a phase will read
    auto src = [&](int i) __attribute__((always_inline)) {
      return i == 0 ? ws : (i == 1 ? qe : (i < QM ? pr + (long long)pV(i - QV) * N : ws + (long long)fB(ND, i - QM) * N));
    };
    if constexpr (EDGE) {
      constexpr int NE = (L::QN + L::NT - 1) / L::NT;
      int from[NE];
#pragma unroll
      for (int k = 0; k < NE; k++) {
        const int l = imin(tid + L::NT * k, L::QN - 1);
        const int a = l % L::QX, b = (l / L::QX) % L::QY, e = l / (L::QX * L::QY);
        from[k] = q_source<ND>(G, o[0] - L::HX + a, o[1] - 3 + b, ND == 3 ? o[2] - 3 + e : 0);
      }
      SH v[NP][NE];
#pragma unroll
      for (int i = 0; i < NP; i++)
#pragma unroll
        for (int k = 0; k < NE; k++) v[i][k] = from[k] >= 0 ? at(src(i), (unsigned)from[k]) : SH(0);
      if (want_mom) stage_rho_t<TL, SH, EDGE>(G, ws, bg, CBX, o);
#pragma unroll
      for (int i = 0; i < NP; i++)
#pragma unroll
        for (int k = 0; k < NE; k++)
          if (tid + L::NT * k < L::QN) QB(i)[tid + L::NT * k] = v[i][k];
    } else {
      QBox<TL, SH, EDGE> B[NP];
#pragma unroll
      for (int i = 0; i < NP; i++) B[i].load(G, src(i), o);
      if (want_mom) stage_rho_t<TL, SH, EDGE>(G, ws, bg, CBX, o);
#pragma unroll
      for (int i = 0; i < NP; i++) B[i].store(G, src(i), QB(i), o);
    }
    __syncthreads();
  }
  if (h_rho || h_e) {
    if (!ALL) {
    __builtin_amdgcn_s_setprio(3);
    if (h_rho && h_e) {
      QBox<TL, SH, EDGE> Q2;
      Q.load(G, ws, o);
      Q2.load(G, qe, o);
      __builtin_amdgcn_s_setprio(0);
      Q.store(G, ws, box_rho, o);
      Q2.store(G, qe, box_e, o);
    } else {
      const SH* qa = h_rho ? ws : qe;
      Q.load(G, qa, o);
      __builtin_amdgcn_s_setprio(0);
      Q.store(G, qa, h_rho ? box_rho : box_e, o);
    }
    __syncthreads();
    }
    auto diffuse = [&](const SH* box, int f, int zidx) __attribute__((always_inline)) {
#pragma unroll
      for (int d = 0; d < ND; d++) {
        V sc[XC], rdx[XC];
        scales(d, (V)G.chyp[f], sc);
        rdxs(d, rdx);
        Win<TL, SH> W;
        if (d == 0) W.template load<0>(box, qc, 1, sc);
        else W.template load<1>(box, qc, qs[d], sc);
#pragma unroll
        for (int u = 0; u < XC; u++) {
          const bool z = !valid[u] || z1e<EDGE>(G, zidx, d, x[d] + (d == 0 ? u : 0));
          const AT gr = z ? AT(0) : (W.q[u][3] - W.q[u][2]) * rdx[u];
          const AT gl = z ? AT(0) : (W.q[u][2] - W.q[u][1]) * rdx[u];
          acc[f][u] += (gr * W.nr[u] - gl * W.nl[u]) * rdx[u];
          pin(acc[f][u]);
        }
      }
    };
    if (h_rho) diffuse(box_rho, fRHO(), zRHO);
    if (h_e) diffuse(box_e, fE(ND), zTMP1);
    if (!ALL) __syncthreads();
  }

  // momentum phases (q = v_f): energy terms, diagonal and off-diagonal
  // sources; then magnetic phases (q = b_f).  A phase has two parts with a
  // barrier between them: the windows of the q box (coefficients, diagonal
  // terms, and the cross products of the tile extended by one layer along
  // f), then the differences of the products along f, during which the next
  // phase's q box travels.
  // Products of phase f at the tile's region: cross direction k in NR + k RN,
  // their energy terms summed in NR + (ND-1) RN.
  auto region = [&](int f, int& rx, int& ry, int* ex) __attribute__((always_inline)) {
    ex[0] = f == 0 ? L::RX : 0;
    ex[1] = f == 1 ? 1 : 0;
    ex[2] = f == 2 ? 1 : 0;
    rx = TX + 2 * ex[0];
    ry = TY + 2 * ex[1];
  };
  // the two layers just outside the tile along f: one (cell, cross
  // direction) per thread; the directions of a cell sit in lanes l and l^32
  // of a wavefront, which add up their energy products
  auto border = [&](int f, const SH* qb, AT* NR, V Kc, int zidx, int m0, bool weigh, V fac) __attribute__((always_inline)) {
    int rx, ry, ex[3];
    region(f, rx, ry, ex);
    const int pd = f == 0 ? 1 : 0, qd = f == 2 ? 1 : 2;
    const int Tp = pd == 0 ? TX : TY, Tq = ND == 3 ? (qd == 1 ? TY : TZ) : 1;
    const int Fc = Tp * Tq;
    const int ntask = 2 * Fc * (ND - 1);
    const int k = ND == 3 ? (tid >> 5) & 1 : 0;                      // cross direction
    const int r2 = ND == 3 ? (tid & 31) + 32 * (tid >> 6) : tid;     // border cell
    AT gp = AT(0), ge = AT(0);
    int l = 0;
    if (tid < ntask) {
      const int side = r2 >= Fc ? 1 : 0, r = r2 - side * Fc;
      int bc[3] = {0, 0, 0};
      bc[f] = side ? (f == 0 ? TX : (f == 1 ? TY : TZ)) : -1;
      bc[pd] = r % Tp;
      if (ND == 3) bc[qd] = r / Tp;
      l = (bc[0] + ex[0]) + rx * ((bc[1] + ex[1]) + ry * (bc[2] + ex[2]));
      const int xr[3] = {o[0] + bc[0], o[1] + bc[1], ND == 3 ? o[2] + bc[2] : 0};
      if (!EDGE || interior_c<ND>(G, xr)) {
        const unsigned gq = cix(G, xr[0], xr[1], xr[2]);
        // d != f: the border cell's coordinate along d is a tile coordinate
        const bool kk = ND == 3 && k;
        const int bp = bc[pd], bq = bc[qd], xp = xr[pd], xq = xr[qd], sp = qs[pd], sq = qs[qd];
        const SH* mp = ws + (long long)(m0 + pd) * N;
        const SH* mq = ws + (long long)(m0 + qd) * N;
        const AT mb = at(kk ? mq : mp, gq);
        const int qi = (bc[0] + L::HX) + L::QX * ((bc[1] + 3) + L::QY * (ND == 3 ? bc[2] + 3 : 0));
        const int s = kk ? sq : sp;
        const int tp = (pd == 0 ? 0 : TX) + bp, tq = (qd == 1 ? TX : TX + TY) + bq;
        const int ti = kk ? tq : tp;
        const V cp = cm[pd], cq = cm[ND == 3 ? qd : 0];
        const V cmd = kk ? cq : cp;
        // (edge tiles of FP32 dual numbers read the spacing arrays here: with
        // the table the compiler reserves 68 bytes of scratch that no
        // instruction touches)
        constexpr bool table = SEP && !(EDGE && ND == 3 && std::is_same<SH, DualF>::value);
        const V dxr = table ? SDX[ti] : (V)at(A.delx + (long long)(kk ? qd : pd) * N, gq);
        const V rdxr = table ? SDX[L::DXT + ti] : (V)at(A.rdelx + (long long)(kk ? qd : pd) * N, gq);
        const bool z = kk ? z1e<EDGE>(G, zidx, qd, xq) : z1e<EDGE>(G, zidx, pd, xp);
        SH w7[7];
        V y[7], R[2];
#pragma unroll
        for (int q = 0; q < 7; q++) {
          w7[q] = qb[qi + (q - 3) * s];
          y[q] = valof(w7[q]);
        }
        nu_ratios<2>(y, R);
        const AT t5 = z ? AT(0) : (w7[4] - w7[2]) * rdxr * V(0.5);
        const AT t6 = t5 * (dxr * cmd * Kc * (R[1] + R[0])) * fac;
        ge = t6 * mb;
        gp = weigh ? CBX[(bc[0] + L::RX) + L::PX * ((bc[1] + 1) + L::PY * (ND == 3 ? bc[2] + 1 : 0))] * t6 : t6;
      }
    }
    if (ND == 3) ge = ge + lane_xor32(ge);
    if (tid < ntask) {
      NR[(ND == 3 ? k : 0) * L::RN + l] = gp;
      if (k == 0) NR[(ND - 1) * L::RN + l] = ge;
    }
  };

  if (mom_phases) {
    if (!ALL) {
      Q.load(G, pr + (long long)pV(0) * N, o);
      if (want_mom) stage_rho_t<TL, SH, EDGE>(G, ws, bg, CBX, o);
      Q.store(G, pr + (long long)pV(0) * N, QB(QV), o);
    }
    AT ptb[XC], bb[ND][XC];  // background terms of the energy source, formed in FP64
    if (want_eterm) {
      OT eb[XC], bb2[XC];
      own(bg + (long long)bEB() * N, eb);
#pragma unroll
      for (int d = 0; d < ND; d++) {
        OT b1[XC];
        own(bg + (long long)bBB(d) * N, b1);
#pragma unroll
        for (int u = 0; u < XC; u++) {
          bb2[u] = d == 0 ? b1[u] * b1[u] : bb2[u] + b1[u] * b1[u];
          bb[d][u] = (AT)b1[u];
        }
      }
#pragma unroll
      for (int u = 0; u < XC; u++) ptb[u] = (AT)((G.gamma - 1) * eb[u] - 0.5 * (G.gamma - 2) * bb2[u]);
    }
    AT mo[ND][XC];  // own momenta
    if (want_mom)
#pragma unroll
      for (int d = 0; d < ND; d++) own(ws + (long long)fMOM(d) * N, mo[d]);
    if (!ALL) __syncthreads();
    auto part1 = [&](int f) __attribute__((always_inline)) {
      const SH* qb = QB(QV + f);
      AT* NR = NRF(f);
      int rx, ry, ex[3];
      region(f, rx, ry, ex);
      const int ri = (lc[0] + ex[0]) + rx * ((lc[1] + ex[1]) + ry * (lc[2] + ex[2]));
      const V Kc = (V)G.chyp[fMOM(f)];
      AT ge[XC], rt[XC];
#pragma unroll
      for (int u = 0; u < XC; u++) ge[u] = AT(0);
      if (want_mom) ldl<XC>(CBX + pc, rt);
#pragma unroll
      for (int d = 0; d < ND; d++) {
        V sc[XC], rdx[XC];
        scales(d, Kc, sc);
        rdxs(d, rdx);
        Win<TL, SH> W;
        if (d == 0) W.template load<0>(qb, qc, 1, sc);
        else W.template load<1>(qb, qc, qs[d], sc);
        if (want_eterm) {  // addenergyterms_cd2 for dir f
#pragma unroll
          for (int u = 0; u < XC; u++) {
            const AT g4 = !valid[u] || z4e<EDGE>(G, zVEL(f), d, x[d] + (d == 0 ? u : 0))
                              ? AT(0)
                              : ((V(8) * W.q[u][3] - V(8) * W.q[u][1]) + (W.q[u][0] - W.q[u][4])) * (rdx[u] * V(1.0 / 12.0));
            acc[fE(ND)][u] += d == f ? (bb[f][u] * bb[f][u] - ptb[u]) * g4 : bb[d][u] * bb[f][u] * g4;
          }
        }
        if (want_mom) {
          // diagonal source along d, and the products rho_t*t6, t6*m_d of
          // the cross direction d (src/hyperdifmomsource1.cu,
          // src/hyperdifmomsourcene1.cu); m_f at the faces from rho_t v_f
          AT rp[XC], rm[XC];
          if (d == 0 && XC == 2) {
            AT a[XC], b[XC];
            ldl<XC>(CBX + pc - 2, a);
            ldl<XC>(CBX + pc + 2, b);
            rm[0] = a[XC - 1];
            rm[XC - 1] = rt[0];
            rp[0] = rt[XC - 1];
            rp[XC - 1] = b[0];
          } else {
            ldl<XC>(CBX + pc + ps[d], rp);
            ldl<XC>(CBX + pc - ps[d], rm);
          }
          AT gp[XC];
#pragma unroll
          for (int u = 0; u < XC; u++) {
            const bool z = !valid[u] || z1e<EDGE>(G, zTMP4, d, x[d] + (d == 0 ? u : 0));
            const AT q0 = W.q[u][2], qp = W.q[u][3], qm = W.q[u][1];
            const V hr = rdx[u] * V(0.5);
            const V wd = d == f ? hr : hr * V(0.5);  // (the face averages' 1/2; d == f counts twice)
            const AT gr = z ? AT(0) : (qp - q0) * (W.nr[u] * rdx[u]);
            const AT gl = z ? AT(0) : (q0 - qm) * (W.nl[u] * rdx[u]);
            const AT m0 = rt[u] * q0;
            acc[fMOM(f)][u] += ((rt[u] + rp[u]) * gr - (rt[u] + rm[u]) * gl) * wd;
            acc[fE(ND)][u] += ((m0 + rp[u] * qp) * gr - (m0 + rm[u] * qm) * gl) * wd;
            if (d != f) {
              const AT t6 = z ? AT(0) : (qp - qm) * ((W.nr[u] + W.nl[u]) * (hr * V(0.25)));
              gp[u] = rt[u] * t6;
              ge[u] += t6 * mo[d][u];
            }
          }
          if (d != f) stl<XC>(NR + (d < f ? d : d - 1) * L::RN + ri, gp);
        }
        pin_acc();
      }
      if (want_mom) {
        stl<XC>(NR + (ND - 1) * L::RN + ri, ge);
        border(f, qb, NR, Kc, zTMP4, fMOM(0), true, V(0.25));
      }
    };
    auto part2 = [&](int f) __attribute__((always_inline)) {
      if (want_mom) {
        const AT* NR = NRF(f);
        int rx, ry, ex[3];
        region(f, rx, ry, ex);
        const int sf = f == 0 ? 1 : (f == 1 ? rx : rx * ry);
        const int ri = (lc[0] + ex[0]) + rx * ((lc[1] + ex[1]) + ry * (lc[2] + ex[2]));
        V rdx[XC];
        rdxs(f, rdx);
        AT dif[ND][XC];
#pragma unroll
        for (int k = 0; k < ND; k++) {
          AT p[XC], m[XC];
          const AT* R = NR + k * L::RN + ri;
          if (f == 0 && XC == 2) {
            AT a[XC], b[XC], e[XC];
            ldl<XC>(R - 2, a);
            ldl<XC>(R, b);
            ldl<XC>(R + 2, e);
            m[0] = a[XC - 1];
            p[0] = b[XC - 1];
            m[XC - 1] = b[0];
            p[XC - 1] = e[0];
          } else {
            ldl<XC>(R + sf, p);
            ldl<XC>(R - sf, m);
          }
#pragma unroll
          for (int u = 0; u < XC; u++) {
            const bool z = !valid[u] || z1e<EDGE>(G, k == ND - 1 ? zTMP8 : zTMP7, f, x[f] + (f == 0 ? u : 0));
            dif[k][u] = z ? AT(0) : (p[u] - m[u]) * (rdx[u] * V(0.5));
          }
        }
#pragma unroll
        for (int u = 0; u < XC; u++) {
#pragma unroll
          for (int d = 0; d < ND; d++)
            if (d != f) acc[fMOM(d)][u] += dif[d < f ? d : d - 1][u];
          acc[fE(ND)][u] += dif[ND - 1][u];
        }
        pin_acc();
      }
    };
#pragma unroll
    for (int f = 0; f < ND; f++) {
      part1(f);
      if (!ALL) {
        __syncthreads();
        const bool more = f + 1 < ND;
        const SH* nq = pr + (long long)pV(more ? f + 1 : 0) * N;
        if (more) Q.load(G, nq, o);
        part2(f);
        if (more) {
          Q.store(G, nq, QB(QV), o);
          __syncthreads();
        }
      }
    }
    if (ALL) {
      __syncthreads();
#pragma unroll
      for (int f = 0; f < ND; f++) part2(f);
      __syncthreads();
    }
  }

  // magnetic phases (q = b_f): curl-form cross terms (sb = -1,
  // src/hyperdifbsourcene1.cu) and diagonal terms (sb = +1,
  // src/hyperdifbsource1.cu)
  if (want_b) {
    if (!ALL) {
      Q.load(G, ws + (long long)fB(ND, 0) * N, o);
      Q.store(G, ws + (long long)fB(ND, 0) * N, QB(QM), o);
    }
    AT bo[ND][XC];  // own field
#pragma unroll
    for (int d = 0; d < ND; d++) own(ws + (long long)fB(ND, d) * N, bo[d]);
    if (!ALL) __syncthreads();
    auto part1 = [&](int f) __attribute__((always_inline)) {
      const SH* qb = QB(QM + f);
      AT* NR = NRF(f);
      int rx, ry, ex[3];
      region(f, rx, ry, ex);
      const int ri = (lc[0] + ex[0]) + rx * ((lc[1] + ex[1]) + ry * (lc[2] + ex[2]));
      const V Kc = (V)G.chyp[fB(ND, f)];
      AT ge[XC];
#pragma unroll
      for (int u = 0; u < XC; u++) ge[u] = AT(0);
#pragma unroll
      for (int d = 0; d < ND; d++) {
        if (d == f) continue;
        V sc[XC], rdx[XC];
        scales(d, Kc, sc);
        rdxs(d, rdx);
        Win<TL, SH> W;
        if (d == 0) W.template load<0>(qb, qc, 1, sc);
        else W.template load<1>(qb, qc, qs[d], sc);
        AT gp[XC];
#pragma unroll
        for (int u = 0; u < XC; u++) {
          const bool z = !valid[u] || z1e<EDGE>(G, zTMP1, d, x[d] + (d == 0 ? u : 0));
          const AT q0 = W.q[u][2], qp = W.q[u][3], qm = W.q[u][1];
          const AT gr = z ? AT(0) : (qp - q0) * (W.nr[u] * rdx[u]);
          const AT gl = z ? AT(0) : (q0 - qm) * (W.nl[u] * rdx[u]);
          acc[fB(ND, f)][u] += (gr - gl) * rdx[u];
          acc[fE(ND)][u] += ((q0 + qp) * gr - (q0 + qm) * gl) * (rdx[u] * V(0.5));
          gp[u] = z ? AT(0) : (qp - qm) * ((W.nr[u] + W.nl[u]) * (rdx[u] * V(0.25)));
          ge[u] += gp[u] * bo[d][u];
        }
        stl<XC>(NR + (d < f ? d : d - 1) * L::RN + ri, gp);
        pin_acc();
      }
      stl<XC>(NR + (ND - 1) * L::RN + ri, ge);
      border(f, qb, NR, Kc, zTMP1, fB(ND, 0), false, V(0.5));
    };
    auto part2 = [&](int f) __attribute__((always_inline)) {
      const AT* NR = NRF(f);
      int rx, ry, ex[3];
      region(f, rx, ry, ex);
      const int sf = f == 0 ? 1 : (f == 1 ? rx : rx * ry);
      const int ri = (lc[0] + ex[0]) + rx * ((lc[1] + ex[1]) + ry * (lc[2] + ex[2]));
      V rdx[XC];
      rdxs(f, rdx);
#pragma unroll
      for (int k = 0; k < ND; k++) {
        AT p[XC], m[XC];
        const AT* R = NR + k * L::RN + ri;
        if (f == 0 && XC == 2) {
          AT a[XC], b[XC], e[XC];
          ldl<XC>(R - 2, a);
          ldl<XC>(R, b);
          ldl<XC>(R + 2, e);
          m[0] = a[XC - 1];
          p[0] = b[XC - 1];
          m[XC - 1] = b[0];
          p[XC - 1] = e[0];
        } else {
          ldl<XC>(R + sf, p);
          ldl<XC>(R - sf, m);
        }
#pragma unroll
        for (int u = 0; u < XC; u++) {
          const bool z = !valid[u] || z1e<EDGE>(G, k == ND - 1 ? zTMP5 : zTMP3, f, x[f] + (f == 0 ? u : 0));
          const AT df = z ? AT(0) : (p[u] - m[u]) * (rdx[u] * V(0.5));
          if (k == ND - 1) acc[fE(ND)][u] -= df;
          else acc[fB(ND, k < f ? k : k + 1)][u] -= df;
        }
      }
      pin_acc();
    };
#pragma unroll
    for (int f = 0; f < ND; f++) {
      part1(f);
      if (!ALL) {
        __syncthreads();
        const bool more = f + 1 < ND;
        const SH* nq = ws + (long long)fB(ND, more ? f + 1 : 0) * N;
        if (more) Q.load(G, nq, o);
        part2(f);
        if (more) {
          Q.store(G, nq, QB(QM), o);
          __syncthreads();
        }
      }
    }
    if (ALL) {
      __syncthreads();
#pragma unroll
      for (int f = 0; f < ND; f++) part2(f);
    }
  }

  if (!any) return;
  // ------------------------------------------------------------ gravity
  OT rho_c[XC], rhob_c[XC];
  own(w, rho_c);
  own(bg + (long long)bRHOB() * N, rhob_c);
  if (T & SMAUG_T_GRAV) {
#pragma unroll
    for (int d = 0; d < ND; d++) {
      if (G.g[d] == 0.0) continue;  // no gravity along d: both terms are zero
      OT m1[XC];
      own(w + (long long)fMOM(d) * N, m1);
#pragma unroll
      for (int u = 0; u < XC; u++) {
        acc[fMOM(d)][u] += (AT)(G.g[d] * rho_c[u]);
        acc[fE(ND)][u] += (AT)(rho_c[u] * (G.g[d] * m1[u]) / (rho_c[u] + rhob_c[u]));
      }
    }
  }
  // ------------------------------------------------------------ update, source, RK, ghosts
  const double h = A.hfrac * stage_dt(G, A);
  const OT* __restrict__ base = (const OT*)A.base;
  OT* __restrict__ wo = (OT*)A.wout;
  OT outs[NP][XC];
#pragma unroll
  for (int f = 0; f < NP; f++) {
    OT b1[XC];
    own(base + (long long)f * N, b1);
#pragma unroll
    for (int u = 0; u < XC; u++) outs[f][u] = b1[u] + h * (OT)acc[f][u];
  }
#pragma unroll
  for (int u = 0; u < XC; u++) {
    if (!valid[u]) continue;
    OT out[NP];
#pragma unroll
    for (int f = 0; f < NP; f++) out[f] = outs[f][u];
    add_source<ND, OT>(G, A, T, x[0] + u, x[1], x[2], c + u, rho_c[u], rhob_c[u], h, out);
#pragma unroll
    for (int f = 0; f < NP; f++) outs[f][u] = out[f];
  }
  if (A.r1) {
    if constexpr (XC == 2) {
#pragma unroll
      for (int f = 0; f < NP; f++) {
        const long long o_f = (long long)f * N;
        OT b0[XC], b1[XC], b2[XC], b3[XC];
        own(base + o_f, b0);
        own((const OT*)A.r1 + o_f, b1);
        own((const OT*)A.r2 + o_f, b2);
        own((const OT*)A.r3 + o_f, b3);
#pragma unroll
        for (int u = 0; u < XC; u++) outs[f][u] = outs[f][u] + (b1[u] + 2.0 * b2[u] + b3[u] - 4.0 * b0[u]) / 3;
        // in two halves: with the loads of every field in flight at once the
        // registers of three workgroups per CU do not hold them (16 went to
        // scratch memory, which the runtime has to set up for a first launch)
        if (f == NP / 2 - 1) {
#pragma unroll
          for (int g = 0; g <= f; g++)
#pragma unroll
            for (int u = 0; u < XC; u++) pin(outs[g][u]);
        }
      }
    } else {  // pointers per lane, stepped field by field, as in put_images
      const OT *p0 = base + c, *p1 = (const OT*)A.r1 + c, *p2 = (const OT*)A.r2 + c, *p3 = (const OT*)A.r3 + c;
#pragma unroll
      for (int f = 0; f < NP; f++, p0 += N, p1 += N, p2 += N, p3 += N)
        outs[f][0] = outs[f][0] + (*p1 + 2.0 * *p2 + *p3 - 4.0 * *p0) / 3;
    }
  }
  // the cells themselves, then their ghost images
  if (valid[XC - 1]) {
#pragma unroll
    for (int q = 0; q < NP; q++) stg<XC>(wo + (long long)q * N, c, outs[q]);
  } else {
#pragma unroll
    for (int q = 0; q < NP; q++) put(wo + (long long)q * N, c, outs[q][0]);
  }
  if (!EDGE) return;  // no cell of an inner tile has a ghost image
#pragma unroll
  for (int u = 0; u < XC; u++) {
    if (!valid[u]) continue;
    OT out[NP];
#pragma unroll
    for (int f = 0; f < NP; f++) out[f] = outs[f][u];
    const int y[3] = {x[0] + u, x[1], x[2]};
    put_images<ND, OT>(G, wo, y, out);
  }
}

// Tiles of k_rhs_tiled.  FP64 and FP32: 8 x 4 x 8 in 3D (dim 0 contiguous and
// 8 wide for coalesced rows; deep in z, the direction whose neighbour tiles
// are least likely to still be in L2) and 16 x 16 in 2D.  Dual numbers are
// twice as large in LDS, where one tile per CU fits: 8 x 8 x 8 cells give it
// eight wavefronts to the four of the smaller tile (a tangent-linear step at
// 96^3 4.29 -> 2.45 ms; FP32 pairs the same either way).
template <int ND, typename SH>
struct TileOf {
  using T = TileT<3, 8, 4, 8, 1>;
};
template <typename SH>
struct TileOf<2, SH> {
  using T = TileT<2, 16, 16, 1, 1>;
};
template <>
struct TileOf<3, Dual> {
  using T = TileT<3, 8, 8, 8, 1>;
};
template <>
struct TileOf<3, DualF> {
  using T = TileT<3, 8, 8, 8, 1>;
};
// the tile of k_rhs_small
using SmallTile = TileT<3, 8, 4, 8, 1>;
// the tile of k_rhs_wide: two cells per thread
using WideTile = TileT<3, 8, 8, 8, 2>;

// origin of workgroup b's tile.  XCD-aware tile order: the hardware deals
// consecutive workgroups to the 8 XCDs in turn, so workgroup b runs on XCD
// b%8.  In 3D XCD x takes the slab of tile layers [x*gz/8, (x+1)*gz/8) and
// walks it x fastest, then z, then y, so the z neighbour of a tile runs gx
// tiles after it (its halo planes still in that XCD's L2) and the y
// neighbour gx*gz/8 tiles after it (measured 1.7 % faster at 256^3 than x,
// y, z order, whose z neighbour comes gx*gy tiles later); otherwise XCD x
// takes the tiles [x*nb/8, (x+1)*nb/8) in x, y, z order.
template <class TL>
__device__ __forceinline__ void tile_origin(const Geo& G, int b, int* o) {
  constexpr int ND = TL::ND, TX = TL::X, TY = TL::Y, TZ = TL::Z;
  const int gx = (G.n[0] - 4 + TX - 1) / TX, gy = (G.n[1] - 4 + TY - 1) / TY;
  const int gz = ND == 3 ? (G.n[2] - 4 + TZ - 1) / TZ : 1;
  const int nb = gx * gy * gz;
  int t = b;
  if ((nb & 7) == 0) {
    const int xcd = b & 7, tl = b >> 3;
    if (ND == 3 && (gz & 7) == 0) {
      const int zc = gz >> 3;  // tile layers per XCD
      const int ux = tl % gx, r = tl / gx;
      const int uz = xcd * zc + r % zc, uy = r / zc;
      t = (uz * gy + uy) * gx + ux;
    } else {
      t = xcd * (nb >> 3) + tl;
    }
  }
  o[0] = 2 + t % gx * TX;
  o[1] = 2 + (t / gx) % gy * TY;
  o[2] = ND == 3 ? 2 + t / (gx * gy) * TZ : 0;
}

// inner tile: every cell in [5, n-6] along every direction (the test is
// uniform per workgroup; the first and last tile layer along an axis are
// edge tiles)
template <class TL>
__device__ __forceinline__ bool edge_tile(const Geo& G, const int* o) {
  bool edge = o[0] < 5 || o[0] + TL::X - 1 > G.n[0] - 6 || o[1] < 5 || o[1] + TL::Y - 1 > G.n[1] - 6;
  if (TL::ND == 3) edge = edge || o[2] < 5 || o[2] + TL::Z - 1 > G.n[2] - 6;
  return edge;
}

template <class TL>
static int tiles_of(const Geo& G) {
  int nb = ((G.n[0] - 4 + TL::X - 1) / TL::X) * ((G.n[1] - 4 + TL::Y - 1) / TL::Y);
  if (TL::ND == 3) nb *= (G.n[2] - 4 + TL::Z - 1) / TL::Z;
  return nb;
}

// wavefronts per SIMD the registers must allow
template <int ND, typename SH>
constexpr int min_waves() {
  return ND == 2 ? 2 : (sizeof(SH) == 4 ? 5 : (std::is_same<SH, double>::value ? 4 : 2));
}

// One cell per thread, on a tensor-product grid.  2D tiles keep every box in
// LDS (36 KB in FP64), 3D ones the boxes of a phase.
template <int ND, typename SH>
__global__ __launch_bounds__((TileOf<ND, SH>::T::NT), (min_waves<ND, SH>())) void k_rhs_tiled(Geo G, RhsArgs A) {
  using TL = typename TileOf<ND, SH>::T;
  constexpr bool ALL = ND == 2;
  __shared__ __align__(16) SH sm[ALL ? Lay<TL>::SMEM_ALL : Lay<TL>::SMEM];
  stage_head(G, A);
  int o[3];
  tile_origin<TL>(G, blockIdx.x, o);
  if (edge_tile<TL>(G, o))
    rhs_tile<TL, SH, true, true, ALL>(G, A, sm, o);
  else
    rhs_tile<TL, SH, false, true, ALL>(G, A, sm, o);
}

// the same on any other grid (a kernel of its own: with both in one the
// tensor-product grids ran 2 to 6 % slower)
template <int ND, typename SH>
__global__ __launch_bounds__((TileOf<ND, SH>::T::NT), (min_waves<ND, SH>())) void k_rhs_general(Geo G, RhsArgs A) {
  using TL = typename TileOf<ND, SH>::T;
  __shared__ __align__(16) SH sm[Lay<TL>::SMEM];
  stage_head(G, A);
  int o[3];
  tile_origin<TL>(G, blockIdx.x, o);
  if (edge_tile<TL>(G, o))
    rhs_tile<TL, SH, true, false, false>(G, A, sm, o);
  else
    rhs_tile<TL, SH, false, false, false>(G, A, sm, o);
}

// 3D tensor-product grids of few tiles: every box of a tile in LDS at once
// (158 KB in FP64).  A tile that has a CU to itself waits for memory and
// barriers most of its time: 48 us for the phases one after the other, 33 us
// this way (FP64, 16x12x12; 0.205 -> 0.144 ms per step).
template <typename SH>
__global__ __launch_bounds__(SmallTile::NT, 1) void k_rhs_small(Geo G, RhsArgs A) {
  using TL = SmallTile;
  __shared__ __align__(16) SH sm[Lay<TL>::SMEM_ALL];
  stage_head(G, A);
  int o[3];
  tile_origin<TL>(G, blockIdx.x, o);
  if (edge_tile<TL>(G, o))
    rhs_tile<TL, SH, true, true, true>(G, A, sm, o);
  else
    rhs_tile<TL, SH, false, true, true>(G, A, sm, o);
}

// FP64 on large 3D tensor-product grids: two cells per thread, 8 x 8 x 8
// tiles, three workgroups per CU (167 VGPRs, no scratch, 53.5 KB of LDS).
__global__ __launch_bounds__(WideTile::NT, 3) void k_rhs_wide(Geo G, RhsArgs A) {
  using TL = WideTile;
  __shared__ __align__(16) double sm[Lay<TL>::SMEM];
  stage_head(G, A);
  int o[3];
  tile_origin<TL>(G, blockIdx.x, o);
  if (edge_tile<TL>(G, o))
    rhs_tile<TL, double, true, true, false>(G, A, sm, o);
  else
    rhs_tile<TL, double, false, true, false>(G, A, sm, o);
}

// (the tests compile the dispatch with other limits, to send every grid
// through each kernel)
#ifndef SMAUG_CUS
#define SMAUG_CUS 256
#endif
#ifndef SMAUG_WIDE_TILES
#define SMAUG_WIDE_TILES 12000
#endif
constexpr int kLds = 160 * 1024;  // LDS of a CU

template <int ND, typename SH>
static void launch_tiled_t(const Geo& G, hipStream_t st, const RhsArgs& A) {
  using TL = typename TileOf<ND, SH>::T;
  constexpr int fit = kLds / (int)(sizeof(SH) * Lay<SmallTile>::SMEM_ALL);  // k_rhs_small tiles per CU
  const int nb = tiles_of<TL>(G);
  if (!A.dx1) {
    hipLaunchKernelGGL((k_rhs_general<ND, SH>), dim3(nb), dim3(TL::NT), 0, st, G, A);
    return;
  }
  if constexpr (ND == 3 && fit > 0) {
    // as long as the whole grid is resident at once: FP64 40^3 (250 tiles)
    // 0.041 against 0.054 ms, 48^3 (432) 0.064 against 0.059; FP32, two per
    // CU, 48^3 0.038 against 0.053, 56^3 (686) 0.073 against 0.070.  It stages
    // every box whatever the term mask says, in one round trip: that pays for
    // the phases of v_f and b_f, which make a trip for each box otherwise
    // (32^3 with hyperdiffusion off, RK4 step: 0.119 against 0.126 ms), and
    // not for the fluxes, rho and e_int (16x12x12, single-stage step: fluxes
    // only 0.0211 against 0.0168, with the rho terms 0.0220 against 0.0199)
    const unsigned phases = SMAUG_T_ETERM | (G.hyper ? SMAUG_T_HMOM | SMAUG_T_HB : 0u);
    if (tiles_of<SmallTile>(G) <= SMAUG_CUS * fit && (G.terms & phases)) {
      hipLaunchKernelGGL((k_rhs_small<SH>), dim3(tiles_of<SmallTile>(G)), dim3(SmallTile::NT), 0, st, G, A);
      return;
    }
  }
  if constexpr (std::is_same<SH, double>::value && ND == 3) {
    // two cells per thread pay once the grid is many rounds of tiles: 128^3
    // (4096 wide tiles) 0.513 ms either way, 160^3 (8000) 0.996 against 0.995,
    // 192^3 (13824) 1.541 against 1.596, 256^3 3.51 against 3.73; at 96^3
    // 0.246 against 0.231
    if (tiles_of<WideTile>(G) >= SMAUG_WIDE_TILES) {
      hipLaunchKernelGGL(k_rhs_wide, dim3(tiles_of<WideTile>(G)), dim3(WideTile::NT), 0, st, G, A);
      return;
    }
  }
  hipLaunchKernelGGL((k_rhs_tiled<ND, SH>), dim3(nb), dim3(TL::NT), 0, st, G, A);
}

// the tangent-linear stage: every state array of A (win, base, r1..r3,
// wout, bg and the driver map) holds Dual values, and wsh and prim hold Dual
// values too, or FP32 DualF values when G.mixed
void launch_rhs_tl(const Geo& G, hipStream_t st, const RhsArgs& A) {
  if (G.mixed) {  // FP32 dual stencils (wsh, prim), FP64 dual own cells
    if (G.nd == 3)
      launch_tiled_t<3, DualF>(G, st, A);
    else
      launch_tiled_t<2, DualF>(G, st, A);
  } else if (G.nd == 3) {
    launch_tiled_t<3, Dual>(G, st, A);
  } else {
    launch_tiled_t<2, Dual>(G, st, A);
  }
}

void launch_rhs_tiled(const Geo& G, hipStream_t st, const RhsArgs& A) {
  if (G.nd == 3) {
    if (G.mixed) launch_tiled_t<3, float>(G, st, A);
    else launch_tiled_t<3, double>(G, st, A);
  } else {
    if (G.mixed) launch_tiled_t<2, float>(G, st, A);
    else launch_tiled_t<2, double>(G, st, A);
  }
}

}  // namespace smaug
