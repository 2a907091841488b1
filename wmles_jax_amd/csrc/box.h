// Fused stage kernel body for tensor-product ("box") blocks (box_tile): every face vector has
// one non-zero component, every centroid coordinate depends on one index, so the metrics of a
// block are three one-dimensional tables (BoxEnt: width, its reciprocal and cube root, the
// reciprocal centroid distance across the lower face).  The reference composition is that of
// flux3_tile (viscous.py:6-51, sgs.py, schemes.py, solver.py:78-121); what the
// metrics' zeros remove from it:
//  * no geometry is read per cell (28 face-vector, centroid and volume words per cell and
//    stage in the general form): the tables of a tile sit in LDS, those of the marching
//    direction in registers;
//  * a gradient component is one central difference, an SGS filter width a product of three
//    tabulated cube roots;
//  * the corrected face gradient's normal component is (phi_R - phi_L) / dist exactly, so a
//    face reads four tangential velocity derivatives of each cell instead of twelve
//    gradients, and no temperature gradient is formed at all;
//  * u . S, the pressure flux, HLLC's normal and tau . S are one product each.
//
// One body for both arithmetic forms (R = float: FP32-bulk records in gauge form with the
// FP64 epilogue of flux2.h; R = double: the plain form's eight record planes).  Contraction
// is off in the functions below and the fused multiply-adds are written out, so every
// instance (kernel, mode, scheme, persistent stage) rounds the same way.  FP64 divides, scales and
// sums so that it rounds no more than a form with a division per quotient and each face's flux
// summed by itself; FP32, whose fluxes are 1e-7, takes the cheaper forms.
//
// The state is read, not a primitive record: each thread forms the records of its column and
// of a halo cell one plane ahead (rec_of), so no primitive launch writes 32 / 64 B per cell for
// this one to read back with a halo.  Channel of 256 x 128 x 128 cells, Hybrid + Vreman, mean of the
// three stages by events: FP32 274 us against 253 us on records and 78 us that wrote them; FP64
// 427 us against 461 us + 137 us (a kernel trace reads 282 and 444).  It is bound by vector issue
// (86% of the FP32 launch's cycles, 67% of the lanes active: the Hybrid's upwind branch).
//
// March.  At plane I the tile evaluates the gradient records of plane I, the own i face I-1/2,
// which completes cell I-1, and then the j / k faces of plane I.  The records of planes I-1 and
// I are in LDS (FP64: I, with I-1 in registers), that of I+1 in registers, I-2 of the own column
// too.  46 threads evaluate a ring cell's gradient besides their own; thread row tj = 15 owns
// the column above the tile (the upper ring row), so the halo ring is 124 cells.  Two barriers
// per plane (FP64: three): the gradient records, and the face exchange together with the next
// plane's staging.  sched_barriers keep the scheduler from hoisting a phase's LDS loads into
// the one before: without them the kernels spill 18 to 60 registers and run 1.3 times as long.
#pragma once
#include <type_traits>

#include "flux2.h"

namespace wmx {

namespace {

template <class R>
__device__ __forceinline__ R fm(R a, R b, R c) {
  if constexpr (sizeof(R) == 4) return __builtin_fmaf(a, b, c);
  else return __builtin_fma(a, b, c);
}

// Record of a cell as the box kernels hold it: E = e + |u|^2 / 2 (the KEP fluxes read only
// that sum), or e itself where the central flux is KEEP.
template <class R>
struct BCell {
  R r, u[3], p, T, E;
};
constexpr int NPB = 7;                         // staged record planes
constexpr int BJ = C2J + 1;                    // columns a thread row owns (tile + upper ring row)
constexpr int NHB = H2J * H2K - BJ * TK;       // halo slots (124)
constexpr int NGRB = TK + 2 * C2J;             // ring cells with a gradient record (46)
// gradient planes: d phi_a / dx_b at 3 a + b (phi = u, v, w; FP32 also T), then mu_eff, k_eff,
// theta.  FP32: pitch 18, so that three workgroups' LDS fits a CU
template <class R>
struct GB {
  static constexpr int NV = sizeof(R) == 4 ? 4 : 3;
  static constexpr int MU = 3 * NV, K = MU + 1, TH = MU + 2, N = MU + 3;
  static constexpr int P = sizeof(R) == 4 ? G2K : G2P, S = (G2J - 1) * P + G2K;
};

// Kennedy-Gruber flux of order 2 / 4 as pair sums (kep_pairs_f32) across a face of normal D:
// the mass flux is k[0] F[0], the others k[1] F[1..4].  FP64 of order 4 takes the factors into the
// combination (1/6 of the inner pair, 1/48 of the outer ones): a factor after it would round the
// pressure-sized sum once more.
template <int D, int ORDER, class R>
__device__ __forceinline__ void kep_axis(const BCell<R>& L2, const BCell<R>& L, const BCell<R>& Rc,
                                         const BCell<R>& R2, R S, R* F, R* un4, R* k) {
#pragma clang fp contract(off)
  auto pair = [&](const BCell<R>& a, const BCell<R>& b, R* A, R* sr, R* ww) {
#pragma clang fp contract(off)
    *sr = a.r + b.r;
    R su[3];
#pragma unroll
    for (int c = 0; c < 3; ++c) su[c] = a.u[c] + b.u[c];
    const R sp = a.p + b.p, sE = a.E + b.E;
    const R w = su[D] * S, M = *sr * w;
    A[0] = M;
#pragma unroll
    for (int c = 0; c < 3; ++c) A[1 + c] = c == D ? fm(R(4) * sp, S, M * su[c]) : M * su[c];
    A[4] = fm(sp + sp, w, M * sE);
    *ww = w;
  };
  R sr, w;
  if (ORDER == 2) {
    pair(L, Rc, F, &sr, &w);
    *un4 = R(0.5) * w;
    k[0] = R(0.25);
    k[1] = R(0.125);
    return;
  }
  R A[5], Aa[5], wa, Ab[5], wb, sra, srb;
  pair(L, Rc, A, &sr, &w);
  pair(L, R2, Aa, &sra, &wa);
  pair(L2, Rc, Ab, &srb, &wb);
  *un4 = fm(R(8), w, -(wa + wb)) * R(1.0 / 12.0);
  if constexpr (sizeof(R) == 8) {
    F[0] = fm(R(1.0 / 3.0), A[0], -((Aa[0] + Ab[0]) * R(1.0 / 24.0)));
#pragma unroll
    for (int c = 1; c < 5; ++c) F[c] = fm(R(1.0 / 6.0), A[c], -((Aa[c] + Ab[c]) * R(1.0 / 48.0)));
    k[0] = k[1] = R(1);
    return;
  }
  F[0] = fm(R(8), A[0], -fm(sra, wa, Ab[0]));
#pragma unroll
  for (int c = 1; c < 5; ++c) F[c] = fm(R(8), A[c], -(Aa[c] + Ab[c]));
  k[0] = R(1.0 / 24.0);
  k[1] = R(1.0 / 48.0);
}

// KEEP flux (schemes.py:25-55) of order 2 / 4 across a face of normal D; E holds e.
template <int D, class R>
__device__ __forceinline__ void keep_axis(int order, const BCell<R>& L2, const BCell<R>& L, const BCell<R>& Rc,
                                          const BCell<R>& R2, R S, R* F, R* un4) {
#pragma clang fp contract(off)
  const R h = R(0.5);
  // (sw: the order in which the compiler forms the pressure work of the (L, R2) pair)
  auto two = [&](const BCell<R>& a, const BCell<R>& b, bool sw, R* G, R* ro, R* w) {
#pragma clang fp contract(off)
    const R rho = h * (a.r + b.r), p = h * (a.p + b.p);
    R u[3];
#pragma unroll
    for (int c = 0; c < 3; ++c) u[c] = h * (a.u[c] + b.u[c]);
    const R un = u[D] * S, m = rho * un;
    const R K = h * fm(a.u[2], b.u[2], fm(a.u[1], b.u[1], a.u[0] * b.u[0]));
    const R ua = a.u[D] * S, ub = b.u[D] * S;
    const R P = sw ? fm(b.p, ua, a.p * ub) : fm(a.p, ub, b.p * ua);
    G[0] = m;
#pragma unroll
    for (int c = 0; c < 3; ++c) G[1 + c] = c == D ? fm(p, S, m * u[c]) : m * u[c];
    G[4] = fm(h, P, fm(K, m, (m * h) * (a.E + b.E)));
    *ro = rho;
    *w = un;
  };
  R F0[5], u0, r0;
  two(L, Rc, false, F0, &r0, &u0);
  if (order == 2) {
#pragma unroll
    for (int c = 0; c < 5; ++c) F[c] = F0[c];
    *un4 = u0;
    return;
  }
  R Fa[5], Fb[5], ua, ub, ra, rb;
  two(L, R2, true, Fa, &ra, &ua);
  two(L2, Rc, false, Fb, &rb, &ub);
  const R c23 = R(2.0 / 3.0), c112 = R(1.0 / 12.0);
  Fa[0] = fm(ra, ua, Fb[0]);                     // the sum of the two mass fluxes
#pragma unroll
  for (int c = 0; c < 5; ++c) F[c] = R(2) * fm(c23, F0[c], -(c112 * (c == 0 ? Fa[0] : Fa[c] + Fb[c])));
  *un4 = R(2) * fm(c23, u0, -(c112 * (ua + ub)));
}

// MUSCL reconstruction, positivity fallback and HLLC (schemes.py:100-152) across a face of
// normal D, times the area S; pr is added back to the reconstructed pressures.  The fused
// multiply-adds are those the compiler forms for muscl_hllc_flux<float> in the general
// kernels (the right limiter's a^2 + b^2 depends on whether the limiter is fixed at compile
// time), so the FP32 flux is theirs bit for bit: its rounding is the largest error of an
// FP32-bulk step, and box and general plans then differ far less than either from FP64.
template <int D, int SC, class R>
__device__ __forceinline__ void upwind_axis(R gamma, int limiter, const BCell<R>& L2, const BCell<R>& L,
                                            const BCell<R>& Rc, const BCell<R>& R2, R S, R pr, R er, R* F) {
#pragma clang fp contract(off)
  const R h = R(0.5);
  R wl[5], wr[5];
  const R q0[5] = {L2.r, L2.u[0], L2.u[1], L2.u[2], L2.p}, q1[5] = {L.r, L.u[0], L.u[1], L.u[2], L.p};
  const R q2[5] = {Rc.r, Rc.u[0], Rc.u[1], Rc.u[2], Rc.p}, q3[5] = {R2.r, R2.u[0], R2.u[1], R2.u[2], R2.p};
  // van Albada slope (a (b^2 + eps) + b (a^2 + eps)) / (a^2 + b^2 + 2 eps); sq: a^2 + b^2
  auto lim = [&](R a, R b, R sq) {
#pragma clang fp contract(off)
    if (limiter != 0) return minmod(a, b);
    const R eps = R(1e-12);
    return fdiv<R>(fm(b, fm(a, a, eps), a * fm(b, b, eps)), sq + R(2.0) * eps);
  };
#pragma unroll
  for (int c = 0; c < 5; ++c) {
    const R a = q1[c] - q0[c], b = q2[c] - q1[c], d = q3[c] - q2[c];
    wl[c] = fm(h, lim(a, b, fm(a, a, b * b)), q1[c]);
    wr[c] = fm(-h, lim(b, d, SC == SC_ANY ? fm(b, b, d * d) : fm(d, d, b * b)), q2[c]);
  }
  wl[4] = wl[4] + pr;
  wr[4] = wr[4] + pr;
  if (wl[0] <= R(0) || wl[4] <= R(0) || wr[0] <= R(0) || wr[4] <= R(0)) {
#pragma unroll
    for (int c = 0; c < 5; ++c) { wl[c] = q1[c]; wr[c] = q2[c]; }
    wl[4] = wl[4] + pr;
    wr[4] = wr[4] + pr;
  }
  const R rl = wl[0], pl = wl[4], rr = wr[0], pq = wr[4];
  const R Sm = fsqrt<R>(S * S), n = fdiv<R>(S, Sm);
  const R unl = wl[1 + D] * n, unr = wr[1 + D] * n;
  const R cl = fsqrt<R>(fdiv<R>(gamma * pl, rl)), cr = fsqrt<R>(fdiv<R>(gamma * pq, rr));
  const R sL = fmin(unl - cl, unr - cr), sR = fmax(unl + cl, unr + cr);
  const R dL = sL - unl, dR = sR - unr;
  const R ss = fdiv<R>(fm(-(rr * unr), dR, fm(rl * unl, dL, pq - pl)), fm(rl, dL, -(rr * dR)));
  const bool left = sL >= R(0) || ss >= R(0);
  const R r = left ? rl : rr, p = left ? pl : pq, un = left ? unl : unr, s = left ? sL : sR;
  R u[3];
#pragma unroll
  for (int c = 0; c < 3; ++c) u[c] = left ? wl[1 + c] : wr[1 + c];
  // (a / b + c: FP32 as the multiply-add of the reciprocal that the compiler forms, FP64 the quotient)
  auto div_add = [](R a, R b, R c) {
#pragma clang fp contract(off)
    return sizeof(R) == 4 ? fm(a, fdiv<R>(R(1), b), c) : fdiv<R>(a, b) + c;
  };
  const R kin = fm(u[2], u[2], fm(u[0], u[0], u[1] * u[1]));
  const R E = sizeof(R) == 4 ? div_add(p, gamma - R(1.0), (h * r) * kin) : fm(h * r, kin, fdiv<R>(p, gamma - R(1.0)));
  R G[5];
  G[0] = r * un;
#pragma unroll
  for (int c = 0; c < 3; ++c) G[1 + c] = c == D ? fm(p, n, G[0] * u[c]) : G[0] * u[c];
  G[4] = (E + p) * un;
  if (left ? sL < R(0) : sR > R(0)) {           // a star state lies on the face
    const R a = r * (s - un), d = ss - un, is = fdiv<R>(R(1), s - ss);
    const R f = sizeof(R) == 4 ? a * is : fdiv<R>(a, s - ss);
    const R ed = div_add(p, a, ss), e = sizeof(R) == 4 ? div_add(E, r, d * ed) : fm(d, ed, fdiv<R>(E, r));
    G[0] = fm(s, sizeof(R) == 4 ? fm(a, is, -r) : f - r, G[0]);
#pragma unroll
    for (int c = 0; c < 3; ++c) G[1 + c] = fm(s, fm(f, c == D ? fm(d, n, u[c]) : u[c], -(r * u[c])), G[1 + c]);
    G[4] = fm(s, fm(f, e, -E), G[4]);
  }
  // times the area, in gauge form (flux2.h): less pr S, er x the mass flux (FP64: both 0)
  F[0] = G[0] * Sm;
#pragma unroll
  for (int c = 0; c < 3; ++c) F[1 + c] = c == D ? fm(G[1 + c], Sm, -(pr * S)) : G[1 + c] * Sm;
  F[4] = fm(G[4], Sm, -(er * F[0]));
}

// What a face of normal D reads of a cell's gradient record: with t, s the other two axes
// (increasing), du_D/dt, du_D/ds, du_t/dt, du_s/ds, and (FP32) the derivatives of u, v, w, T
// along D; then mu_eff, k_eff.
template <class R>
struct BGrad {
  static constexpr int N = sizeof(R) == 4 ? 8 : 4;
  R g[N], mu, k;
};
template <int D>
constexpr int bgrad_plane(int i) {
  constexpr int t = D == 0 ? 1 : 0, s = D == 2 ? 1 : 2;
  return i == 0 ? 3 * D + t : i == 1 ? 3 * D + s : i == 2 ? 4 * t : i == 3 ? 4 * s : 3 * (i - 4) + D;
}

// (FP64) the gradient planes that faces of normal 0 do not read: du/dx, dv/dx, dv/dz, dw/dx, dw/dy
constexpr int djk_plane(int v) { return v == 0 ? 0 : v == 1 ? 3 : v + 3; }

// Viscous flux (viscous.py:28-51) through a face of normal D and area S, id = 1 / distance of
// the two centroids: V[0..2] the viscous stress times the area, V[3] the energy flux.  The
// face gradient's normal component g_n + ((phi_R - phi_L) id - g_n) is (phi_R - phi_L) id;
// FP32 keeps the general form's evaluation of it (same rounding, see upwind_axis).
template <int D, class R>
__device__ __forceinline__ void viscous_axis(const BCell<R>& L, const BCell<R>& Rc, const BGrad<R>& a,
                                             const BGrad<R>& b, R id, R d, R S, R* V) {
#pragma clang fp contract(off)
  constexpr int t = D == 0 ? 1 : 0, s = D == 2 ? 1 : 2;
  const R h = R(0.5);
  R g[4], dn[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) g[i] = h * (a.g[i] + b.g[i]);
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    const R df = c < 3 ? Rc.u[c] - L.u[c] : Rc.T - L.T;
    if constexpr (sizeof(R) == 4) {
      const R e = d * id, gn = h * (a.g[4 + c] + b.g[4 + c]);
      dn[c] = fm(e, fm(id, df, -(gn * e)), gn);
    } else {
      dn[c] = df * id;
    }
  }
  const R muf = h * (a.mu + b.mu), kf = h * (a.k + b.k);
  // (u_x + v_y) + w_z in this order
  const R gx = D == 0 ? dn[0] : g[2], gy = D == 1 ? dn[1] : (D == 0 ? g[2] : g[3]), gz = D == 2 ? dn[2] : g[3];
  const R div = (gx + gy) + gz;
  V[D] = (muf * fm(R(-2.0 / 3.0), div, dn[D] + dn[D])) * S;
  V[t] = (muf * (dn[t] + g[0])) * S;
  V[s] = (muf * (dn[s] + g[1])) * S;
  const R uts = fm(h * (L.u[2] + Rc.u[2]), V[2], fm(h * (L.u[0] + Rc.u[0]), V[0], (h * (L.u[1] + Rc.u[1])) * V[1]));
  V[3] = fm(-kf, dn[3] * S, -uts);
}

// Numerical flux through a face of normal D: F[0..4], and (FP32-bulk) w in F[5].  grad(0 / 1)
// reads the left / right cell's BGrad: after the inviscid part, so that the two records are
// not held through it (registers bound the occupancy).
template <int D, int SC, class R, class GF>
__device__ __forceinline__ void face_axis(const NumDev& nd, const BCell<R>& L2, const BCell<R>& L,
                                          const BCell<R>& Rc, const BCell<R>& R2, R thL, R thR, const GF& grad,
                                          R id, R d, R S, R pr, R er, R* F) {
#pragma clang fp contract(off)
  constexpr bool F32 = sizeof(R) == 4;
  auto viscous = [&](R* V) {
    __builtin_amdgcn_sched_barrier(0);
    const BGrad<R> gL = grad(0), gR = grad(1);
    viscous_axis<D, R>(L, Rc, gL, gR, id, d, S, V);
  };
  R V[4], k[2], un4 = R(0);
  if constexpr (SC == SC_KEP2 || SC == SC_KEP4) {
    R A[5];
    kep_axis<D, SC == SC_KEP2 ? 2 : 4, R>(L2, L, Rc, R2, S, A, &un4, k);
    viscous(V);
    F[0] = A[0] * k[0];
#pragma unroll
    for (int c = 0; c < 3; ++c) F[1 + c] = fm(A[1 + c], k[1], -V[c]);
    F[4] = fm(A[4], k[1], V[3]);
    if (F32) F[5] = un4;
    return;
  }
  const int sch = SC == SC_HYB_KEP4_ALBADA ? WMX_SCHEME_HYBRID : nd.scheme;
  const int order = SC == SC_HYB_KEP4_ALBADA ? 4 : nd.order;
  const int limiter = SC == SC_HYB_KEP4_ALBADA ? 0 : nd.limiter;
  R s = sch == WMX_SCHEME_MUSCLHLLC ? R(1) : R(0);
  if (sch == WMX_SCHEME_HYBRID)
    s = fmin(fmax(fdiv<R>(fmax(thL, thR) - R(nd.th0), R(nd.th1 - nd.th0)), R(0)), R(1));
  R Fc[5] = {R(0), R(0), R(0), R(0), R(0)};
  if (s < R(1)) {
    const bool keep = SC == SC_ANY && (sch == WMX_SCHEME_KEEP ||
                                       (sch == WMX_SCHEME_HYBRID && nd.central == WMX_SCHEME_KEEP));
    if (keep) {
      keep_axis<D, R>(order, L2, L, Rc, R2, S, Fc, &un4);
    } else {
      if (order == 2) kep_axis<D, 2, R>(L2, L, Rc, R2, S, Fc, &un4, k);
      else kep_axis<D, 4, R>(L2, L, Rc, R2, S, Fc, &un4, k);
      Fc[0] = Fc[0] * k[0];
#pragma unroll
      for (int c = 1; c < 5; ++c) Fc[c] = Fc[c] * k[1];
    }
  }
  const R wc = R(1) - s;
#pragma unroll
  for (int v = 0; v < 5; ++v) F[v] = wc * Fc[v];
  if (s > R(0)) {
    R Fu[5];
    upwind_axis<D, SC, R>(R(nd.gas.gamma), limiter, L2, L, Rc, R2, S, pr, er, Fu);
#pragma unroll
    for (int v = 0; v < 5; ++v) F[v] = fm(s, Fu[v], F[v]);
  }
  if (F32) F[5] = wc * un4;
  viscous(V);
#pragma unroll
  for (int c = 0; c < 3; ++c) F[1 + c] = F[1 + c] - V[c];
  F[4] = F[4] + V[3];
}

// Gradient record of a cell from its own (u, v, w, T) c, its six neighbours m / p per axis,
// S[d] half the face area of axis d, the volume and the filter width: GB planes.  FP32: the
// Green-Gauss face sums of the general kernels in their rounding (the 1/2 of the face averages
// taken with the area is exact); FP64: the central difference itself (S[d] = 1 / (2 width)).
template <class R>
__device__ __forceinline__ void grad_axis(const NumDev& nd, const R* c, const R (*m)[4], const R (*p)[4],
                                          const R* S, R vol, R delta, R rho, R mu, R* G) {
  R g[9];
  {
#pragma clang fp contract(off)
#pragma unroll
    for (int d = 0; d < 3; ++d)
#pragma unroll
      for (int v = 0; v < GB<R>::NV; ++v) {
        R x;
        if constexpr (sizeof(R) == 4) x = fdiv<R>(fm(c[v] + p[d][v], S[d], -((m[d][v] + c[v]) * S[d])), vol);
        else x = (p[d][v] - m[d][v]) * S[d];
        G[3 * v + d] = x;
        if (v < 3) g[3 * v + d] = x;
      }
  }
  R mut = R(0) * rho;
  if (nd.sgs != WMX_SGS_NONE) {
    const R cs = R(nd.sgs_c);
    R nut;
    if (nd.sgs == WMX_SGS_SMAGORINSKY) nut = nut_smagorinsky<R>(g, delta, cs);
    else if (nd.sgs == WMX_SGS_WALE) nut = nut_wale<R>(g, delta, cs);
    else nut = nut_vreman<R>(g, delta, cs);
    mut = rho * nut;
  }
  G[GB<R>::MU] = mu + mut;
  G[GB<R>::K] = R(nd.gas.cp) * (fdiv<R>(mu, R(nd.gas.Pr)) + fdiv<R>(mut, R(nd.gas.Pr_t)));
  {                                              // Ducros sensor (viscous.py:22-25)
#pragma clang fp contract(off)
    const R div = (g[0] + g[4]) + g[8];
    const R a = g[7] - g[5], b = g[2] - g[6], e = g[3] - g[1];
    G[GB<R>::TH] = fdiv<R>(div * div, fm(div, div, fm(e, e, fm(a, a, b * b))) + R(1e-30));
  }
}

// halo job ht: 0..45 a ring cell whose gradient record the thread also evaluates (halo 2: row -1,
// columns -1 and 16), 46..123 a cell that is only staged (halo 1)
__device__ __forceinline__ void box_halo_job(int ht, int* hj, int* hk, int* halo) {
  if (ht < NGRB) {
    *halo = 2;
    if (ht < TK) { *hj = -1; *hk = ht; }
    else if (ht < TK + C2J) { *hj = ht - TK; *hk = -1; }
    else { *hj = ht - TK - C2J; *hk = TK; }
  } else if (ht < NHB) {
    *halo = 1;
    const int x = ht - NGRB;                     // rows -2 and 16 (20 each), corners of row -1 (4),
    if (x < H2K) { *hj = -2; *hk = x - 2; }        // columns -2 and 17 of rows 0..15, -1 and 16 of row 15
    else if (x < 2 * H2K) { *hj = BJ; *hk = x - H2K - 2; }
    else if (x < 2 * H2K + 4) { const int y = x - 2 * H2K; *hj = -1; *hk = y < 2 ? y - 2 : TK + y - 2; }
    else if (x < 2 * H2K + 4 + 2 * BJ) { const int y = x - 2 * H2K - 4; *hj = y >> 1; *hk = y & 1 ? TK + 1 : -2; }
    else { *hj = C2J; *hk = x - (2 * H2K + 4 + 2 * BJ) ? TK : -1; }
  }
}

}  // namespace

// One marching tile (tiles[tile]) of a box plan's flux launch; called by every thread of a
// 256-thread workgroup.  MODE 0: r = RHS; 1: q + dt r; 2: 3/4 q0 + 1/4 (q + dt r); 3: 1/3 q0 +
// 2/3 (q + dt r)
template <class R, int MODE, int SC>
__device__ __forceinline__ void box_tile(const BlockDev* __restrict__ blks, const int4* __restrict__ tiles,
                                         int ci_len, const NumDev& nd, const Ptrs& qin, const Ptrs& q0,
                                         const Ptrs& out, const double* __restrict__ d_dt, double dt_host,
                                         int zfuse, int tile) {
#pragma clang fp contract(off)
  constexpr bool F32 = sizeof(R) == 4;
  constexpr int NF = F32 ? 6 : 5;                // exchanged values per face
  constexpr int NB = F32 ? 2 : 1;                // staged record planes kept (LDS: FP64 fits one)
  __shared__ R sP[NB][NPB][NP2];
  __shared__ R sG[GB<R>::N][GB<R>::S];
  __shared__ R sFj[NF][NT];                      // slot tile_tid(r, c)
  __shared__ R sFk[NF][NT + C2J + 1];            // slot kface_slot(r, c)
  __shared__ double sW[2][G2K];                  // widths of rows j0-1 .. and columns k0-1 ..
  __shared__ double sIw[F32 ? 1 : 2][F32 ? 1 : G2K];       // (FP64) their reciprocals
  __shared__ double sCb[F32 ? 1 : 2][F32 ? 1 : G2K];       // (FP64) their cube roots
  __shared__ R sH0[F32 ? 1 : 3][F32 ? 1 : NGRB];           // (FP64) the ring cells' u, v, w at I-1
  __shared__ R sId[2][G2K];                      // 1 / centroid distance across the lower face
  __shared__ R sDx[F32 ? 2 : 1][F32 ? G2K : 1];  // (FP32) that distance, signed
  const int4 t = tiles[tile];
  const BlockDev& B = blks[t.x];
  const int j0 = t.y, k0 = t.z, i0 = t.w;
  const int i1 = min(i0 + ci_len, B.n[0]);
  int tid = threadIdx.x;
  int tj = (tid >> 6) + 4 * ((tid >> 4) & 3), tk = tid & 15;         // tile_tid(tj, tk) == tid
  const int ng = B.ng;
  const int* N = B.N;
  const int n0 = B.n[0], n1 = B.n[1], n2 = B.n[2];
  const bool own = tj < C2J;
  const bool act = own && j0 + tj < n1 && k0 + tk < n2;
  const int jl = min(j0 + C2J, n1) - j0, kl = min(k0 + TK, n2) - k0;
  int J = ng + j0 + tj, K = ng + k0 + tk;
  const unsigned cells = (unsigned)B.cells, sI = (unsigned)N[1] * N[2];
  const double dt = d_dt ? d_dt[B.case_id] : dt_host;
  const bool keep = SC == SC_ANY && (nd.scheme == WMX_SCHEME_KEEP ||
                                     (nd.scheme == WMX_SCHEME_HYBRID && nd.central == WMX_SCHEME_KEEP));
  auto p_ok = [&](int jj, int kk) { return jj >= 0 && jj < N[1] && kk >= 0 && kk < N[2]; };
  auto g_ok = [&](int jj, int kk) {
    return jj >= ng - 1 && jj <= ng + n1 && kk >= ng - 1 && kk <= ng + n2;
  };
  const int I0 = ng + i0, Iend = ng + i1;
  auto energy = [&](const R* a, R e) {           // E (KEEP: e)
#pragma clang fp contract(off)
    return keep ? e : fm(R(0.5), fm(a[2], a[2], fm(a[1], a[1], a[0] * a[0])), e);
  };
  auto cell_of = [&](const R* a, const R* b) {
    BCell<R> c;
    c.r = b[0]; c.p = b[1]; c.T = a[3]; c.E = energy(a, b[3]);
#pragma unroll
    for (int x = 0; x < 3; ++x) c.u[x] = a[x];
    return c;
  };
  auto stage = [&](R (*P)[NP2], int s, const BCell<R>& c) {
    P[0][s] = c.r; P[1][s] = c.u[0]; P[2][s] = c.u[1]; P[3][s] = c.u[2];
    P[4][s] = c.p; P[5][s] = c.T; P[6][s] = c.E;
  };
  // a k ghost of a fused side is read at its periodic image
  const int zf = zfuse ? B.zfuse : 0;
  auto kcol = [&](int kk) {
    if ((zf & 1) && kk < ng) return kk + n2;
    if ((zf & 2) && kk >= ng + n2) return kk - n2;
    return kk;
  };
  const double* qi = qin.p[t.x];
  auto load_q = [&](unsigned c, double* q) {
#pragma unroll
    for (int v = 0; v < 5; ++v) q[v] = ldu(qi + v * (size_t)cells, c);
  };
  // own column and its slots; halo job by ht, the thread index turned by a multiple of 64 that
  // changes from one of an XCD's workgroups to the next (the jobs of two wavefronts would
  // otherwise fall on the same two SIMDs of every CU), its cell in one word
  const bool own_p = p_ok(J, K), own_g = g_ok(J, K);
  int sp_own = (tj + 2) * H2K + (tk + 2), sg_own = (tj + 1) * GB<R>::P + (tk + 1);
  int hj = 0, hk = 0, halo = 0;
  box_halo_job((tid + 64 * ((tile >> 3) & 3)) & (NT - 1), &hj, &hk, &halo);
  if (halo && !p_ok(ng + j0 + hj, ng + k0 + hk)) halo = 0;
  const bool halo1 = halo != 0, halo2 = halo == 2, ring_g = halo2 && g_ok(ng + j0 + hj, ng + k0 + hk);
  const int hjob = (hj + 2) | (hk + 2) << 8;
  // The thread's indices, in FP32 formed again from its number in each phase: kept through the
  // march (or hoisted out of it) they took up to 20 registers of the face phases, which spilled,
  // and a reload waits for every load issued before it (256 x 128 x 128 cells: 308 -> 271 us;
  // FP64, which has the registers: 423 us as they are, 431 us formed again)
  auto place = [&]() {
    tid = threadIdx.x;
    if constexpr (F32) asm volatile("" : "+v"(tid));
    tj = (tid >> 6) + 4 * ((tid >> 4) & 3);
    tk = tid & 15;
    J = ng + j0 + tj;
    K = ng + k0 + tk;
    sp_own = (tj + 2) * H2K + (tk + 2);
    sg_own = (tj + 1) * GB<R>::P + (tk + 1);
  };
  int ht, hs;
  auto hplace = [&]() {
    int w = hjob;
    if constexpr (F32) asm volatile("" : "+v"(w));
    hj = (w & 255) - 2;
    hk = (w >> 8) - 2;
    ht = ((int)threadIdx.x + 64 * ((tile >> 3) & 3)) & (NT - 1);
    hs = (hj + 2) * H2K + (hk + 2);
  };
  // metric tables of the tile's rows and columns (index 0: row j0 - 1 / column k0 - 1)
  if (tid < 2 * G2K) {
    const int a = tid < G2K ? 0 : 1, x = tid - a * G2K;
    const int at = (a == 0 ? ng + j0 : ng + k0) - 1 + x;
    if ((a == 0 ? x < BJ + 1 : true) && at < N[1 + a]) {
      const BoxEnt& e = B.box[1 + a][at];
      sW[a][x] = e.w; sId[a][x] = F32 ? R(e.idf) : R(e.id);
      if constexpr (F32) {
        sDx[a][x] = e.df;
      } else {
        sIw[a][x] = e.iw;
        sCb[a][x] = e.cb;
      }
    }
  }
  // ---- prologue: plane I0-1 staged, the records of I0-2 kept, those of I0 in flight
  const BoxEnt* __restrict__ bx = B.box[0];
  double wi = bx[I0 - 1].w, iwi = bx[I0 - 1].iw, cbi = bx[I0 - 1].cb;
  R idi = F32 ? R(bx[I0 - 1].idf) : R(bx[I0 - 1].id), dxi = R(bx[I0 - 1].df);
  double iwi_p = iwi;                            // 1 / width of plane I-1
  BCell<R> W0, W1;                               // own records of I-2 and (FP64; FP32: staged) I-1
  R mu0, Hr = R(0), Hm = R(0);                   // mu of the own cell I, rho and mu of the ring cell
  double qn[5], hq[5];                           // states in flight: own column, halo cell
  R mu1, Hx[4], Hn[4];                           // own mu of the next plane, the halo cell's record there
#pragma unroll
  for (int x = 0; x < 4; ++x) Hx[x] = Hn[x] = R(0);
  auto request = [&](int p) {                    // the states of plane p
    // (the own column clamped into the array)
    load_q((unsigned)p * sI + (unsigned)min(J, N[1] - 1) * N[2] + kcol(min(K, N[2] - 1)), qn);
    hplace();
    if (halo1) load_q((unsigned)p * sI + (unsigned)(ng + j0 + hj) * N[2] + (unsigned)kcol(ng + k0 + hk), hq);
  };
  auto arrive = [&]() {                          // their records
    R a[4], b[4];
    rec_of(nd, qn, B.p_ref, B.T_gauge, B.e_ref, a, b);
    mu1 = b[2];
    if (halo1) rec_of(nd, hq, B.p_ref, B.T_gauge, B.e_ref, Hx, Hn);
    return cell_of(a, b);
  };
  auto stage_plane = [&](R (*P)[NP2], const BCell<R>& c) {
    if (own_p) stage(P, sp_own, c);
    hplace();
    if (halo1) stage(P, hs, cell_of(Hx, Hn));
    mu0 = mu1;
    Hr = Hn[0];
    Hm = Hn[2];
  };
  request(I0 - 2);
  W0 = W1 = arrive();
  if constexpr (F32) {
    stage_plane(sP[NB - 1], W1);
  } else if (halo2) {
#pragma unroll
    for (int x = 0; x < 3; ++x) sH0[x][ht] = Hx[x];
  }
  request(I0 - 1);
  stage_plane(sP[0], arrive());
  request(I0);
  // Outward sum of the own cell I-1 so far, in FP64.  FP32: its lower i face minus its j / k face
  // sums; FP64: the lower i face alone, so that the difference of the two i faces is formed before
  // the smaller sums go in (their sum would round at the size of the flux); those wait in the
  // planes of the own gradient slot that no i face reads, free after the exchange barrier.
  double Cp[NF];
#pragma unroll
  for (int v = 0; v < NF; ++v) Cp[v] = 0.0;
  __syncthreads();
  const double iyz = act ? 1.0 / (sW[0][tj + 1] * sW[1][tk + 1]) : 0.0;
  const R pr = R(F32 ? B.p_ref : 0.0), er = R(F32 ? B.e_ref : 0.0);
  auto wall_of = [&](int d, int cf) {            // the wall-modelled side of face cf, or -1
    const int side = cf == ng ? 0 : (cf == ng + B.n[d] ? 1 : -1);
    return side >= 0 && B.faces[2 * d + side].kind == WMX_BC_WALLMODEL ? side : -1;
  };
  auto wall_flux = [&](int d, int side, int fI, int fJ, int fK, R* F) {
    int t1, t2;
    tangents(d, &t1, &t2);
    const int cc[3] = {fI, fJ, fK};
    const unsigned nw = (unsigned)B.n[t1] * B.n[t2];
    const unsigned w = (unsigned)(cc[t1] - ng) * B.n[t2] + (cc[t2] - ng);
    const double* W = B.wall[2 * d + side];
#pragma unroll
    for (int v = 0; v < 5; ++v) F[v] = (R)ldu(W + v * (size_t)nw, w);
    F[5] = R(0);
  };
  int buf = 0;
  for (int I = I0 - 1; I <= Iend; ++I) {
    const bool inner = I >= I0 && I < Iend;      // plane owned by the tile: j / k faces
    const bool fin = act && I >= I0 + 1;         // cell I-1 is finished at this plane
    R (*P)[NP2] = sP[buf];
    place();
    const BCell<R> Pn = arrive();                // own record of I+1
    auto cell = [&](const R (*Q)[NP2], int s) {
      BCell<R> w;
      w.r = Q[0][s]; w.u[0] = Q[1][s]; w.u[1] = Q[2][s]; w.u[2] = Q[3][s];
      w.p = Q[4][s]; w.T = Q[5][s]; w.E = Q[6][s];
      return w;
    };
    auto grad_of = [&](auto D, int g) {          // a cell's record as faces of normal D read it
      BGrad<R> o;
#pragma unroll
      for (int x = 0; x < BGrad<R>::N; ++x) o.g[x] = sG[bgrad_plane<decltype(D)::value>(x)][g];
      o.mu = sG[GB<R>::MU][g]; o.k = sG[GB<R>::K][g];
      return o;
    };
    __builtin_amdgcn_sched_barrier(0);
    // ---- cell I-1: its state loads go out first, covered by the gradients and the i face
    const unsigned c = (unsigned)(I - 1) * sI + (unsigned)J * N[2] + K;
    // the stage is a0 q0 + a1 (q + dt r).  FP32 keeps one value per component, base = a0 q0 + a1 q,
    // and adds a1 dt r; FP64, where the state's roundings are its largest, keeps q and parks q0
    const double a0 = MODE == 2 ? 0.75 : 1.0 / 3.0, a1 = MODE == 1 ? 1.0 : (MODE == 2 ? 0.25 : 2.0 / 3.0);
    double base[5], vz[5];
    if (MODE >= 1 && fin) {
#pragma unroll
      for (int v = 0; v < 5; ++v) base[v] = ldu(qi + v * (size_t)cells, c);
      if (MODE >= 2) {
        const double* qz = q0.p[t.x];
#pragma unroll
        for (int v = 0; v < 5; ++v) vz[v] = ldu(qz + v * (size_t)cells, c);
      }
    }
    // ---- gradient records of plane I: own column, then the 46 ring cells
    __builtin_amdgcn_s_setprio(2);
    auto grads = [&](const R* mi, const R* pi, int s, int wj_, int wk_, R rho, R mu, R* G) {
#pragma clang fp contract(off)
      R u[4], m[3][4], p[3][4];                  // (u, v, w, T); T only where NV is 4
#pragma unroll
      for (int v = 0; v < GB<R>::NV; ++v) {
        const R* q = P[v < 3 ? 1 + v : 5];
        u[v] = q[s];
        m[0][v] = mi[v]; m[1][v] = q[s - H2K]; m[2][v] = q[s - 1];
        p[0][v] = pi[v]; p[1][v] = q[s + H2K]; p[2][v] = q[s + 1];
      }
      if constexpr (F32) {
        const double a = sW[0][wj_], b = sW[1][wk_];
        const R h = R(0.5), S[3] = {h * R(a * b), h * R(wi * b), h * R(wi * a)}, vol = R((wi * a) * b);
        grad_axis<R>(nd, u, m, p, S, vol, cbrtf(vol), rho, mu, G);
      } else {
        const R delta = R((cbi * sCb[0][wj_]) * sCb[1][wk_]);
        const R S[3] = {R(0.5 * iwi), R(0.5 * sIw[0][wj_]), R(0.5 * sIw[1][wk_])};
        grad_axis<R>(nd, u, m, p, S, R(0), delta, rho, mu, G);
      }
    };
    if (F32 && own_p) W1 = cell(sP[NB - 1 - buf], sp_own);
    R G[GB<R>::N];
#pragma unroll
    for (int v = 0; v < GB<R>::N; ++v) G[v] = R(0);
    if (own_g) {
      const R mi[4] = {W1.u[0], W1.u[1], W1.u[2], W1.T}, pi[4] = {Pn.u[0], Pn.u[1], Pn.u[2], Pn.T};
      grads(mi, pi, sp_own, tj + 1, tk + 1, P[0][sp_own], mu0, G);
    }
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_setprio(1);
    // ---- own i face I-1/2, which completes cell I-1
    if (MODE >= 2 && fin) {
#pragma unroll
      for (int v = 0; v < 5; ++v) {
        if (F32) base[v] = fm(a0, vz[v], a1 * base[v]);
        else sFj[v][tid] = (R)vz[v];             // (own slot: free until the plane's j faces)
      }
    }
    R Fin[6];
#pragma unroll
    for (int v = 0; v < 6; ++v) Fin[v] = R(0);
    if (act && I >= I0) {
      // (the own slot still holds the record of plane I-1)
      auto grad_i = [&](int h) {
        if (h == 0) return grad_of(std::integral_constant<int, 0>(), sg_own);
        BGrad<R> o;
#pragma unroll
        for (int x = 0; x < BGrad<R>::N; ++x) o.g[x] = G[bgrad_plane<0>(x)];
        o.mu = G[GB<R>::MU]; o.k = G[GB<R>::K];
        return o;
      };
      const int side = wall_of(0, I);
      if (side >= 0) wall_flux(0, side, I, J, K, Fin);
      else face_axis<0, SC, R>(nd, W0, W1, cell(P, sp_own), Pn, sG[GB<R>::TH][sg_own], G[GB<R>::TH], grad_i, idi, dxi, R(sW[0][tj + 1] * sW[1][tk + 1]), pr, er, Fin);
    }
    if (!F32 && fin) {
#pragma unroll
      for (int v = 0; v < NF; ++v) Cp[v] = (Cp[v] - (double)Fin[v]) - (double)sG[djk_plane(v)][sg_own];
    }
    if (own_g) {
#pragma unroll
      for (int v = 0; v < GB<R>::N; ++v) sG[v][sg_own] = G[v];
    }
    if (F32) W0 = W1;
    if (fin) {
      // outward sums in FP64; the FP32-bulk energy gets the gauge terms
      const double ivol = iwi_p * iyz;
      double a[NF], r[5];
#pragma unroll
      for (int v = 0; v < NF; ++v) a[v] = F32 ? Cp[v] - (double)Fin[v] : Cp[v];
      if (F32) a[4] = fm(B.p_ref, a[NF - 1], fm(B.e_ref, a[0], a[4]));
#pragma unroll
      for (int v = 0; v < 5; ++v) r[v] = a[v] * ivol;
      if (nd.n_sponge > 0) {
        const double xcv = ldu(B.xc, c);
        const long long mrow = (long long)(I - 1 - ng) * n1 + (J - ng);
        const long long mplane = (long long)n0 * n1;
        for (int sp = 0; sp < nd.n_sponge; ++sp) {
          const double sigma = sponge_sigma(nd.sponge[sp], xcv);
          if (sigma != 0.0) {                    // (rows outside every sponge have no mean)
#pragma unroll
            for (int v = 0; v < 5; ++v)
              r[v] = fm(-sigma, ldu(qi + v * (size_t)cells, c) - ldu(B.sponge_mean + v * mplane, (unsigned)mrow), r[v]);
          }
        }
      }
      double* o = out.p[t.x];
#pragma unroll
      for (int v = 0; v < 5; ++v) {
        double w = MODE == 0 ? r[v] : fm(F32 ? a1 * dt : dt, r[v], base[v]);
        if (!F32 && MODE == 2) w = fm(a0, (double)sFj[v][tid], a1 * w);      // (a1 w is exact)
        if (!F32 && MODE == 3) w = fm(a1, w, a0 * (double)sFj[v][tid]);
        stu(o + v * (size_t)cells, c, w);
      }
    }
    if (I == Iend) break;
    __builtin_amdgcn_sched_barrier(0);
    place();
    if (inner && ring_g) {
      hplace();
      R Gr[GB<R>::N], m[4];
#pragma unroll
      for (int x = 0; x < GB<R>::NV; ++x) {
        if constexpr (F32) m[x] = sP[NB - 1 - buf][x < 3 ? 1 + x : 5][hs];
        else m[x] = sH0[x][ht];
      }
      grads(m, Hx, hs, hj + 1, hk + 1, Hr, Hm, Gr);
      const int sg = (hj + 1) * GB<R>::P + (hk + 1);
#pragma unroll
      for (int v = 0; v < GB<R>::N; ++v) sG[v][sg] = Gr[v];
    }
    if (inner) {
      __builtin_amdgcn_s_setprio(1);
      __syncthreads();                           // the plane's gradient records
      if (tj <= jl && tk < kl) {                 // j face below row tj
        R F[6];
        const int side = wall_of(1, J);
        if (side >= 0) {
          wall_flux(1, side, I, J, K, F);
        } else {
          auto grad = [&](int h) { return grad_of(std::integral_constant<int, 1>(), sg_own - (1 - h) * GB<R>::P); };
          face_axis<1, SC, R>(nd, cell(P, sp_own - 2 * H2K), cell(P, sp_own - H2K), cell(P, sp_own),
                              cell(P, sp_own + H2K), sG[GB<R>::TH][sg_own - GB<R>::P], sG[GB<R>::TH][sg_own], grad, sId[0][tj + 1], F32 ? sDx[0][F32 ? tj + 1 : 0] : R(0), R(wi * sW[1][tk + 1]), pr, er, F);
        }
#pragma unroll
        for (int v = 0; v < NF; ++v) sFj[v][tid] = F[v];
      }
      __builtin_amdgcn_sched_barrier(0);
      place();
      const int rj = own ? tj : tk, rk = own ? tk : kl;   // k face left of (tj, tk) / upper edge of row tk
      if (rj < jl && (own ? rk < kl : true)) {
        R F[6];
        const int side = wall_of(2, ng + k0 + rk);
        if (side >= 0) {
          wall_flux(2, side, I, ng + j0 + rj, ng + k0 + rk, F);
        } else {
          const int sp = (rj + 2) * H2K + (rk + 2), sg = (rj + 1) * GB<R>::P + (rk + 1);
          auto grad = [&](int h) { return grad_of(std::integral_constant<int, 2>(), sg - 1 + h); };
          face_axis<2, SC, R>(nd, cell(P, sp - 2), cell(P, sp - 1), cell(P, sp), cell(P, sp + 1),
                              sG[GB<R>::TH][sg - 1], sG[GB<R>::TH][sg], grad, sId[1][rk + 1], F32 ? sDx[F32 ? 1 : 0][F32 ? rk + 1 : 0] : R(0), R(wi * sW[0][rj + 1]), pr, er, F);
        }
        const int slot = kface_slot(rj, rk);
#pragma unroll
        for (int v = 0; v < NF; ++v) sFk[v][slot] = F[v];
      }
    }
    __builtin_amdgcn_sched_barrier(0);
    place();
    // ---- FP32: plane I+1 staged in the other buffer and the records of I+2 requested before
    //      the exchange barrier, which then covers both
    if (F32) {
      stage_plane(sP[NB - 1 - buf], Pn);
      request(I + 2);
    }
    iwi_p = iwi;
    wi = bx[I + 1].w; iwi = bx[I + 1].iw; cbi = bx[I + 1].cb;
    idi = F32 ? R(bx[I + 1].idf) : R(bx[I + 1].id);
    if (F32) dxi = R(bx[I + 1].df);
    __syncthreads();                             // j / k face exchange
    __builtin_amdgcn_s_setprio(0);
    if (!F32) {                                  // FP64: one buffer, free after the exchange barrier
      W0 = W1;
      if (own_p) W1 = cell(P, sp_own);
      hplace();
      if (ring_g) {
#pragma unroll
        for (int x = 0; x < 3; ++x) sH0[F32 ? 0 : x][F32 ? 0 : ht] = P[1 + x][hs];
      }
      stage_plane(sP[0], Pn);
      request(I + 2);
    }
    // ---- carry: the outward sum of the own cell I so far
    if (act && inner) {
      const int jup = tile_tid(tj + 1, tk), kup = kface_slot(tj, tk + 1);
#pragma unroll
      for (int v = 0; v < NF; ++v) {
        const double d = ((double)sFj[v][jup] - (double)sFj[v][tid]) + ((double)sFk[v][kup] - (double)sFk[v][tid]);
        Cp[v] = F32 ? (double)Fin[v] - d : (double)Fin[v];
        if (!F32) sG[djk_plane(v)][sg_own] = (R)d;
      }
    }
    if (F32) buf ^= 1;
    else __syncthreads();                        // plane I+1 staged
  }
}

}  // namespace wmx
