// Fused stage kernel body for general curvilinear blocks in FP64 (curv_tile): the march of
// box_tile (box.h) with the face vectors, centroids and volumes read per cell.  The tile forms
// the records of its columns and halo from the state one plane ahead, evaluates the Green-Gauss
// gradient records (viscous.py:6-20, sgs.py) in LDS, and the face fluxes from them
// (schemes.py, viscous.py:28-51, solver.py:78-121), so neither records nor gradients go
// through memory and a stage is one launch after the ghost sweep.
//
// LDS: seven record planes of the plane at hand, fifteen gradient planes, the j / k face
// exchange and the 46 ring cells' previous (u, v, w, T): 79 KB, two workgroups per CU; the
// plane before is kept in registers.  Per plane and column 19 geometry words are read for the
// gradients, requested before the records of the next plane are formed; the lower face vectors
// among them serve the i face.  Bound by the latency of the state and geometry loads and by FP64
// issue at two waves per SIMD.  190 x 63 x 33 ramp, Hybrid + Vreman: 134 us per stage (125 in
// stage 1) where primitive, gradient and flux launches on stored records took 12 + 28 + 131;
// 128 x 72 x 56 skewed box, MUSCL + Smagorinsky: 113 us, was 13 + 37 + 132.  Every spilled
// register costs twice, since its reload waits for all loads issued before it: with 127 of them
// the ramp's stage took 182 us.
#pragma once
#include "box.h"

namespace wmx {

namespace {

constexpr int NGC = 15;                        // g[12], mu_eff, k_eff, theta
constexpr int GCS = (G2J - 1) * G2K + G2K;     // gradient slots (17 x 18)

// Kennedy-Gruber flux of order 2 / 4 as pair sums (kep_pairs_f32 in FP64; E = e + |u|^2 / 2)
template <int ORDER>
__device__ __forceinline__ void kep_curv(const BCell<double>& L2, const BCell<double>& L, const BCell<double>& Rc,
                                         const BCell<double>& R2, const double* S, double* F) {
  auto pair = [&](const BCell<double>& a, const BCell<double>& b, double* A) {
    const double sr = a.r + b.r, sp = a.p + b.p, sE = a.E + b.E;
    double su[3];
#pragma unroll
    for (int c = 0; c < 3; ++c) su[c] = a.u[c] + b.u[c];
    const double w = (su[0] * S[0] + su[1] * S[1]) + su[2] * S[2], M = sr * w;
    A[0] = M;
#pragma unroll
    for (int c = 0; c < 3; ++c) A[1 + c] = M * su[c] + (4.0 * sp) * S[c];
    A[4] = M * sE + (sp + sp) * w;
  };
  double A[5];
  pair(L, Rc, A);
  if (ORDER == 2) {
    F[0] = 0.25 * A[0];
#pragma unroll
    for (int v = 1; v < 5; ++v) F[v] = 0.125 * A[v];
    return;
  }
  double Aa[5], Ab[5];
  pair(L, R2, Aa);
  pair(L2, Rc, Ab);
  F[0] = (1.0 / 3.0) * A[0] - (Aa[0] + Ab[0]) * (1.0 / 24.0);
#pragma unroll
  for (int v = 1; v < 5; ++v) F[v] = (1.0 / 6.0) * A[v] - (Aa[v] + Ab[v]) * (1.0 / 48.0);
}

__device__ __forceinline__ CellWT<double> cell_wt(const BCell<double>& c) {
  CellWT<double> w;
  w.r = c.r; w.u = c.u[0]; w.v = c.u[1]; w.w = c.u[2]; w.p = c.p; w.e = c.E;
  return w;
}

// Inviscid part of the numerical flux (times area) of a face with vector S; th the larger of its
// cells' sensors.
template <int SC>
__device__ __forceinline__ void inviscid_curv(const NumDev& nd, const BCell<double>& L2, const BCell<double>& L,
                                              const BCell<double>& Rc, const BCell<double>& R2, double th,
                                              const double* S, double* F) {
  const int scheme = SC == SC_ANY ? nd.scheme : (SC == SC_HYB_KEP4_ALBADA ? WMX_SCHEME_HYBRID : WMX_SCHEME_KEP);
  double s = scheme == WMX_SCHEME_MUSCLHLLC ? 1.0 : 0.0;
  if (scheme == WMX_SCHEME_HYBRID) s = fmin(fmax(fdiv<double>(th - nd.th0, nd.th1 - nd.th0), 0.0), 1.0);
  // (a part whose weight is exactly 0 is not evaluated)
#pragma unroll
  for (int v = 0; v < 5; ++v) F[v] = 0.0;
  if (s < 1.0) {
    if (SC == SC_KEP2) kep_curv<2>(L2, L, Rc, R2, S, F);
    else if (SC == SC_KEP4 || SC == SC_HYB_KEP4_ALBADA) kep_curv<4>(L2, L, Rc, R2, S, F);
    else if (scheme == WMX_SCHEME_KEEP || (scheme == WMX_SCHEME_HYBRID && nd.central == WMX_SCHEME_KEEP))
      central_flux<true>(nd.order, cell_wt(L2), cell_wt(L), cell_wt(Rc), cell_wt(R2), S[0], S[1], S[2], F);
    else if (nd.order == 2) kep_curv<2>(L2, L, Rc, R2, S, F);
    else kep_curv<4>(L2, L, Rc, R2, S, F);
#pragma unroll
    for (int v = 0; v < 5; ++v) F[v] = (1.0 - s) * F[v];
  }
  if ((SC == SC_ANY || SC == SC_HYB_KEP4_ALBADA) && s > 0.0) {
    double Fu[5];
    const int lim = SC == SC_HYB_KEP4_ALBADA ? WMX_LIMITER_ALBADA : nd.limiter;
    muscl_hllc_flux(nd.gas.gamma, lim, cell_wt(L2), cell_wt(L), cell_wt(Rc), cell_wt(R2), S[0], S[1], S[2], Fu);
#pragma unroll
    for (int v = 0; v < 5; ++v) F[v] = F[v] + s * Fu[v];
  }
}

// Viscous part (viscous.py:28-51): gradients at the face with the component along the centroid line
// corrected.  V[0..2] the stress times the area, V[3] heat flux and work; dx the centroid
// difference, gsum(i) the sum of component i of the two cells' gradient records.
template <class GS>
__device__ __forceinline__ void viscous_curv(const BCell<double>& L, const BCell<double>& Rc, GS gsum,
                                             const double* dx, const double* S, double* V) {
  const double id = fdiv<double>(1.0, fsqrt<double>((dx[0] * dx[0] + dx[1] * dx[1]) + dx[2] * dx[2]));
  const double e[3] = {dx[0] * id, dx[1] * id, dx[2] * id};
  double gf[9];
#pragma unroll
  for (int v = 0; v < 3; ++v) {
    double g[3];
#pragma unroll
    for (int x = 0; x < 3; ++x) g[x] = 0.5 * gsum(3 * v + x);
    const double corr = (Rc.u[v] - L.u[v]) * id - ((g[0] * e[0] + g[1] * e[1]) + g[2] * e[2]);
#pragma unroll
    for (int x = 0; x < 3; ++x) gf[3 * v + x] = g[x] + corr * e[x];
  }
  double dTdn;
  {
    double g[3];
#pragma unroll
    for (int x = 0; x < 3; ++x) g[x] = 0.5 * gsum(9 + x);
    const double corr = (Rc.T - L.T) * id - ((g[0] * e[0] + g[1] * e[1]) + g[2] * e[2]);
    dTdn = ((g[0] + corr * e[0]) * S[0] + (g[1] + corr * e[1]) * S[1]) + (g[2] + corr * e[2]) * S[2];
  }
  const double muf = 0.5 * gsum(12), kf = 0.5 * gsum(13);
  const double td = (2.0 / 3.0) * ((gf[0] + gf[4]) + gf[8]);
  const double t00 = muf * ((gf[0] + gf[0]) - td), t11 = muf * ((gf[4] + gf[4]) - td), t22 = muf * ((gf[8] + gf[8]) - td);
  const double t01 = muf * (gf[1] + gf[3]), t02 = muf * (gf[2] + gf[6]), t12 = muf * (gf[5] + gf[7]);
  V[0] = (t00 * S[0] + t01 * S[1]) + t02 * S[2];
  V[1] = (t01 * S[0] + t11 * S[1]) + t12 * S[2];
  V[2] = (t02 * S[0] + t12 * S[1]) + t22 * S[2];
  double w = kf * dTdn;
#pragma unroll
  for (int c = 0; c < 3; ++c) w = w + (0.5 * (L.u[c] + Rc.u[c])) * V[c];
  V[3] = w;
}

// Numerical flux of a face: the viscous part after the inviscid one, so that the records it reads
// are not held through that
template <int SC, class GS>
__device__ __forceinline__ void face_curv(const NumDev& nd, const BCell<double>& L2, const BCell<double>& L,
                                          const BCell<double>& Rc, const BCell<double>& R2, double th, GS gsum,
                                          const double* dx, const double* S, double* F) {
  inviscid_curv<SC>(nd, L2, L, Rc, R2, th, S, F);
  __builtin_amdgcn_sched_barrier(0);
  double V[4];
  viscous_curv(L, Rc, gsum, dx, S, V);
#pragma unroll
  for (int c = 0; c < 4; ++c) F[1 + c] = F[1 + c] - V[c];
}

// A cell's metrics as the gradient reads them: lower and upper face vectors (S[2 d], S[2 d + 1]),
// half the reciprocal volume and the filter width
struct CurvGeo {
  double S[6][3], hiv, cb;
};

__device__ __forceinline__ void geo_load(const BlockDev& B, int I, int J, int K, CurvGeo& o) {
  const unsigned N1 = (unsigned)B.N[1], N2 = (unsigned)B.N[2];
  const unsigned c = ((unsigned)I * N1 + (unsigned)J) * N2 + (unsigned)K;
  const unsigned f[3] = {c, ((unsigned)I * (N1 + 1) + (unsigned)J) * N2 + (unsigned)K,
                         ((unsigned)I * N1 + (unsigned)J) * (N2 + 1) + (unsigned)K};
  const unsigned up[3] = {N1 * N2, N2, 1u};
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    const double* S = B.S[d];
    const size_t fc = (size_t)fcount(B.N, d);
#pragma unroll
    for (int x = 0; x < 3; ++x) {
      o.S[2 * d][x] = ldu(S + x * fc, f[d]);
      o.S[2 * d + 1][x] = ldu(S + x * fc, f[d] + up[d]);
    }
  }
  o.hiv = ldu((const double*)B.P, c);
  o.cb = ldu((const double*)B.P + (size_t)B.cells, c);
}

// Gradient record of a cell from its own (u, v, w, T) c and its neighbours m / p per axis
// (grad_cell's faces and sums), handed to put(component, value): T's first, which nothing else
// of the record reads
template <class PUT>
__device__ __forceinline__ void grad_curv(const NumDev& nd, const CurvGeo& o, const double* c, const double (*m)[4],
                                          const double (*p)[4], double rho, double mu, PUT put) {
  double g[9];
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    const int v = u == 0 ? 3 : u - 1;
    double a[3] = {0.0, 0.0, 0.0};
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      const double lo = m[d][v] + c[v], hi = c[v] + p[d][v];
#pragma unroll
      for (int x = 0; x < 3; ++x) a[x] = a[x] + (hi * o.S[2 * d + 1][x] - lo * o.S[2 * d][x]);
    }
#pragma unroll
    for (int x = 0; x < 3; ++x) {
      const double q = a[x] * o.hiv;
      if (v < 3) g[3 * v + x] = q;
      put(3 * v + x, q);
    }
  }
  double mut = 0.0 * rho;
  if (nd.sgs != WMX_SGS_NONE) {
    double nut;
    if (nd.sgs == WMX_SGS_SMAGORINSKY) nut = nut_smagorinsky<double>(g, o.cb, nd.sgs_c);
    else if (nd.sgs == WMX_SGS_WALE) nut = nut_wale<double>(g, o.cb, nd.sgs_c);
    else nut = nut_vreman<double>(g, o.cb, nd.sgs_c);
    mut = rho * nut;
  }
  put(12, mu + mut);
  put(13, nd.gas.cp * (fdiv<double>(mu, nd.gas.Pr) + fdiv<double>(mut, nd.gas.Pr_t)));
  put(14, ducros<double>(g));
}

}  // namespace

// One marching tile (tiles[tile]) of a curvilinear FP64 plan's flux launch; called by every
// thread of a 256-thread workgroup.  MODE 0: r = RHS; 1: q + dt r; 2: 3/4 q0 + 1/4 (q + dt r);
// 3: 1/3 q0 + 2/3 (q + dt r)
template <int MODE, int SC>
__device__ __forceinline__ void curv_tile(const BlockDev* __restrict__ blks, const int4* __restrict__ tiles,
                                          int ci_len, const NumDev& nd, const Ptrs& qin, const Ptrs& q0,
                                          const Ptrs& out, const double* __restrict__ d_dt, double dt_host,
                                          int zfuse, int tile) {
  __shared__ double sP[NPB][NP2];                // records (BCell) of the plane at hand
  __shared__ double sG[NGC][GCS];                // gradient records of the plane at hand, I-1's until then
  __shared__ double sFj[5][NT];                  // slot tile_tid(r, c)
  __shared__ double sFk[5][NT + C2J + 1];        // slot kface_slot(r, c)
  __shared__ double sH0[4][NGRB];                // the ring cells' u, v, w, T at I-1
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
  auto cell_of = [&](const double* a, const double* b) {
    BCell<double> c;
    c.r = b[0]; c.p = b[1]; c.T = a[3];
    c.E = keep ? b[3] : b[3] + 0.5 * ((a[0] * a[0] + a[1] * a[1]) + a[2] * a[2]);
#pragma unroll
    for (int x = 0; x < 3; ++x) c.u[x] = a[x];
    return c;
  };
  auto stage = [&](int s, const BCell<double>& c) {
    sP[0][s] = c.r; sP[1][s] = c.u[0]; sP[2][s] = c.u[1]; sP[3][s] = c.u[2];
    sP[4][s] = c.p; sP[5][s] = c.T; sP[6][s] = c.E;
  };
  auto cell = [&](int s) {
    BCell<double> w;
    w.r = sP[0][s]; w.u[0] = sP[1][s]; w.u[1] = sP[2][s]; w.u[2] = sP[3][s];
    w.p = sP[4][s]; w.T = sP[5][s]; w.E = sP[6][s];
    return w;
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
  auto load_x = [&](int II, int JJ, int KK, double* x) {       // a cell's centroid
    const unsigned c = (unsigned)II * sI + (unsigned)JJ * N[2] + KK;
#pragma unroll
    for (int d = 0; d < 3; ++d) x[d] = ldu(B.xc + d * (size_t)cells, c);
  };
  auto load_S = [&](int d, unsigned f, double* S) {            // a face vector of direction d
    const size_t fc = (size_t)fcount(N, d);
#pragma unroll
    for (int x = 0; x < 3; ++x) S[x] = ldu(B.S[d] + x * fc, f);
  };
  // own column and its slots; halo job by ht (box_tile's), its cell, slot and kind in one word
  const bool own_p = p_ok(J, K), own_g = g_ok(J, K);
  int sp_own = (tj + 2) * H2K + (tk + 2), sg_own = (tj + 1) * G2K + (tk + 1);
  int hjob, hj = 0, hk = 0, halo = 0;
  box_halo_job((tid + 64 * ((tile >> 3) & 3)) & (NT - 1), &hj, &hk, &halo);
  if (halo && !p_ok(ng + j0 + hj, ng + k0 + hk)) halo = 0;
  const bool halo1 = halo != 0, halo2 = halo == 2, ring_g = halo2 && g_ok(ng + j0 + hj, ng + k0 + hk);
  hjob = (hj + 2) | (hk + 2) << 8;
  // The thread's indices, formed again from its number: kept through the march (or hoisted out
  // of it) they would take thirty registers of the face phases, which spill
  auto place = [&]() {
    tid = threadIdx.x;
    asm volatile("" : "+v"(tid));
    tj = (tid >> 6) + 4 * ((tid >> 4) & 3);
    tk = tid & 15;
    J = ng + j0 + tj;
    K = ng + k0 + tk;
    sp_own = (tj + 2) * H2K + (tk + 2);
    sg_own = (tj + 1) * G2K + (tk + 1);
  };
  int ht, hs;
  auto hplace = [&]() {
    int w = hjob;
    asm volatile("" : "+v"(w));
    hj = (w & 255) - 2;
    hk = (w >> 8) - 2;
    ht = ((int)threadIdx.x + 64 * ((tile >> 3) & 3)) & (NT - 1);
    hs = (hj + 2) * H2K + (hk + 2);
  };
  // ---- prologue: plane I0-1 staged, the records of I0-2 kept, those of I0 in flight
  BCell<double> W0, W1;                          // own records of I-2 and I-1
  double mu0, mu1, Hm = 0.0;                     // mu of the own cell I, of I+1; of the ring cell I
  double qn[5], hq[5];                           // states in flight: own column, halo cell
#pragma unroll
  for (int x = 0; x < 5; ++x) hq[x] = 0.0;
  auto request = [&](int p) {                    // the states of plane p
    // (the own column clamped into the array)
    load_q((unsigned)p * sI + (unsigned)min(J, N[1] - 1) * N[2] + kcol(min(K, N[2] - 1)), qn);
    hplace();
    if (halo1) load_q((unsigned)p * sI + (unsigned)(ng + j0 + hj) * N[2] + (unsigned)kcol(ng + k0 + hk), hq);
  };
  auto arrive = [&]() {                          // the own record
    double a[4], b[4];
    rec_of(nd, qn, 0.0, 0.0, 0.0, a, b);
    mu1 = b[2];
    return cell_of(a, b);
  };
  auto stage_plane = [&](const BCell<double>& c) {
    if (own_p) stage(sp_own, c);
    hplace();
    if (halo1) {                                  // (its record is formed here: five registers in place of eight)
      double a[4], b[4];
      rec_of(nd, hq, 0.0, 0.0, 0.0, a, b);
      stage(hs, cell_of(a, b));
      Hm = b[2];
    }
    mu0 = mu1;
  };
  request(I0 - 2);
  W0 = W1 = arrive();
  if (halo2) {
    double a[4], b[4];
    rec_of(nd, hq, 0.0, 0.0, 0.0, a, b);
#pragma unroll
    for (int x = 0; x < 4; ++x) sH0[x][ht] = a[x];
  }
  request(I0 - 1);
  stage_plane(arrive());
  request(I0);
  // Lower i face of the own cell I-1, and its centroid.  The sum of its j / k faces waits in LDS: the
  // difference of the two i faces is formed first, since a sum through either would round at the
  // size of the flux (where the flow does not change along i, the j and k faces alone are the sum;
  // in a laminar shear they are 1e-9 of the pressure).  In registers it would be spilled.
  double Cp[5], Xp[3];
#pragma unroll
  for (int v = 0; v < 5; ++v) Cp[v] = 0.0;
#pragma unroll
  for (int x = 0; x < 3; ++x) Xp[x] = 0.0;
  double hiv_p = 0.0;                            // half its reciprocal volume
  __syncthreads();
  auto wall_of = [&](int d, int cf) {            // the wall-modelled side of face cf, or -1
    const int side = cf == ng ? 0 : (cf == ng + B.n[d] ? 1 : -1);
    return side >= 0 && B.faces[2 * d + side].kind == WMX_BC_WALLMODEL ? side : -1;
  };
  auto wall_flux = [&](int d, int side, int fI, int fJ, int fK, double* F) {
    int t1, t2;
    tangents(d, &t1, &t2);
    const int cc[3] = {fI, fJ, fK};
    const unsigned nw = (unsigned)B.n[t1] * B.n[t2];
    const unsigned w = (unsigned)(cc[t1] - ng) * B.n[t2] + (cc[t2] - ng);
    const double* W = B.wall[2 * d + side];
#pragma unroll
    for (int v = 0; v < 5; ++v) F[v] = ldu(W + v * (size_t)nw, w);
  };
  for (int I = I0 - 1; I <= Iend; ++I) {
    const bool inner = I >= I0 && I < Iend;      // plane owned by the tile: j / k faces
    const bool fin = act && I >= I0 + 1;         // cell I-1 is finished at this plane
    place();
    // the own cell's metrics go out before the records of I+1 are formed
    CurvGeo geo;
    double Xc[3] = {0.0, 0.0, 0.0};
    if (own_g) {
      geo_load(B, I, J, K, geo);
      load_x(I, J, K, Xc);
    }
    const BCell<double> Pn = arrive();           // own record of I+1
    __builtin_amdgcn_sched_barrier(0);
    // ---- gradient records of plane I: own column, then the 46 ring cells
    __builtin_amdgcn_s_setprio(2);
    auto grads = [&](const CurvGeo& o, const double* mi, const double* pi, int s, double rho, double mu, auto put) {
      double u[4], m[3][4], p[3][4];             // (u, v, w, T)
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const double* q = sP[v < 3 ? 1 + v : 5];
        u[v] = q[s];
        m[0][v] = mi[v]; m[1][v] = q[s - H2K]; m[2][v] = q[s - 1];
        p[0][v] = pi[v]; p[1][v] = q[s + H2K]; p[2][v] = q[s + 1];
      }
      grad_curv(nd, o, u, m, p, rho, mu, put);
    };
    // The own record, and with it the viscous part of the own i face I-1/2 while its velocity
    // gradients are in registers (the own slot still holds the record of plane I-1).  The
    // temperature's gradient waits in the thread's own slots of the j exchange, the viscous part in
    // the same slots until the inviscid part is there.
    const bool iface = act && I >= I0;
    const int iwall = iface ? wall_of(0, I) : -1;
    if (own_g) {
      const double mi[4] = {W1.u[0], W1.u[1], W1.u[2], W1.T}, pi[4] = {Pn.u[0], Pn.u[1], Pn.u[2], Pn.T};
      double g[9], m[3];
      grads(geo, mi, pi, sp_own, sP[0][sp_own], mu0, [&](int x, double q) {
        if (x < 9) g[x] = q;
        else if (x < 12) sFj[x - 9][tid] = q;
        else m[x - 12] = q;
      });
      __builtin_amdgcn_sched_barrier(0);
      double V[4] = {0.0, 0.0, 0.0, 0.0}, th = 0.0;
      if (iface && iwall < 0) {
        const double dx[3] = {Xc[0] - Xp[0], Xc[1] - Xp[1], Xc[2] - Xp[2]};
        viscous_curv(W1, cell(sp_own), [&](int x) {
          return sG[x][sg_own] + (x < 9 ? g[x] : x < 12 ? sFj[x - 9][tid] : m[x - 12]);
        }, dx, geo.S[0], V);
        th = fmax(sG[14][sg_own], m[2]);
      }
#pragma unroll
      for (int v = 0; v < NGC; ++v) sG[v][sg_own] = v < 9 ? g[v] : v < 12 ? sFj[v - 9][tid] : m[v - 12];
#pragma unroll
      for (int v = 0; v < 4; ++v) sFj[v][tid] = V[v];
      sFj[4][tid] = th;
    }
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_setprio(1);
    // ---- own i face I-1/2, which completes cell I-1
    double Fin[5];
#pragma unroll
    for (int v = 0; v < 5; ++v) Fin[v] = 0.0;
    if (iface) {
      if (iwall >= 0) {
        wall_flux(0, iwall, I, J, K, Fin);
      } else {
        inviscid_curv<SC>(nd, W0, W1, cell(sp_own), Pn, sFj[4][tid], geo.S[0], Fin);
#pragma unroll
        for (int v = 0; v < 4; ++v) Fin[1 + v] = Fin[1 + v] - sFj[v][tid];
      }
    }
    __builtin_amdgcn_sched_barrier(0);
    // ---- cell I-1: its state loads covered by the i face
    const unsigned c = (unsigned)(I - 1) * sI + (unsigned)J * N[2] + K;
    // the stage is a0 q0 + a1 (q + dt r)
    const double a0 = MODE == 2 ? 0.75 : 1.0 / 3.0, a1 = MODE == 2 ? 0.25 : 2.0 / 3.0;
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
    __builtin_amdgcn_sched_barrier(0);
    if (fin) {
      const double ivol = hiv_p + hiv_p;
      double r[5];
#pragma unroll
      for (int v = 0; v < 5; ++v) r[v] = ((Cp[v] - Fin[v]) - sFk[v][kface_slot(tj, tk)]) * ivol;
      if (nd.n_sponge > 0) {                     // SmoothRampSponge, smooth_ramp.py:212-221
        const double xcv = ldu(B.xc, c);
        const long long mrow = (long long)(I - 1 - ng) * n1 + (J - ng);
        const long long mplane = (long long)n0 * n1;
        for (int sp = 0; sp < nd.n_sponge; ++sp) {
          const double sigma = sponge_sigma(nd.sponge[sp], xcv);
          if (sigma != 0.0) {                    // (rows outside every sponge have no mean)
#pragma unroll
            for (int v = 0; v < 5; ++v)
              r[v] = r[v] - sigma * (ldu(qi + v * (size_t)cells, c) - ldu(B.sponge_mean + v * mplane, (unsigned)mrow));
          }
        }
      }
      double* o = out.p[t.x];
#pragma unroll
      for (int v = 0; v < 5; ++v) {
        double w = MODE == 0 ? r[v] : __builtin_fma(dt, r[v], base[v]);
        if (MODE == 2) w = __builtin_fma(a0, vz[v], a1 * w);                 // (a1 w is exact)
        if (MODE == 3) w = __builtin_fma(a1, w, a0 * vz[v]);
        stu(o + v * (size_t)cells, c, w);
      }
    }
    if (I == Iend) break;
    __builtin_amdgcn_sched_barrier(0);
    hiv_p = own_g ? geo.hiv : 0.0;
#pragma unroll
    for (int x = 0; x < 3; ++x) Xp[x] = Xc[x];
    place();
    // the j / k faces' centroids across them (and the upper edge k face's metrics)
    int rj = own ? tj : tk, rk = own ? tk : kl;         // k face left of (tj, tk) / upper edge of row tk
    const bool jface = inner && tj <= jl && tk < kl, kface = inner && rj < jl && (own ? rk < kl : true);
    double xj[3] = {0.0, 0.0, 0.0}, xk[3] = {0.0, 0.0, 0.0}, Sj[3] = {0.0, 0.0, 0.0}, Sk[3] = {0.0, 0.0, 0.0};
    if (jface) {
      load_x(I, J - 1, K, xj);
      load_S(1, ((unsigned)I * (N[1] + 1) + (unsigned)J) * N[2] + (unsigned)K, Sj);
    }
    // (the k face's go out before the j face, which covers them)
    double xr[3] = {Xp[0], Xp[1], Xp[2]};
    auto kgeo = [&]() {
      if (!kface) return;
      const int JJ = ng + j0 + rj, KK = ng + k0 + rk;
      load_x(I, JJ, KK - 1, xk);
      load_S(2, ((unsigned)I * N[1] + (unsigned)JJ) * (unsigned)(N[2] + 1) + (unsigned)KK, Sk);
      if (!own) load_x(I, JJ, KK, xr);
    };
    if (inner && ring_g) {
      CurvGeo rg;
      hplace();
      geo_load(B, I, ng + j0 + hj, ng + k0 + hk, rg);
      double m[4], a[4], b[4];
#pragma unroll
      for (int x = 0; x < 4; ++x) m[x] = sH0[x][ht];
      rec_of(nd, hq, 0.0, 0.0, 0.0, a, b);
      const int sg = (hj + 1) * G2K + (hk + 1);
      grads(rg, m, a, hs, sP[0][hs], Hm, [&](int x, double g) { sG[x][sg] = g; });
    }
    if (inner) {
      __builtin_amdgcn_s_setprio(1);
      __syncthreads();                           // the plane's gradient records
      if (jface) {                               // j face below row tj
        double F[5];
        const int side = wall_of(1, J);
        if (side >= 0) {
          wall_flux(1, side, I, J, K, F);
        } else {
          const double dx[3] = {Xp[0] - xj[0], Xp[1] - xj[1], Xp[2] - xj[2]};
          auto gsum = [&](int x) { return sG[x][sg_own - G2K] + sG[x][sg_own]; };
          face_curv<SC>(nd, cell(sp_own - 2 * H2K), cell(sp_own - H2K), cell(sp_own), cell(sp_own + H2K),
                        fmax(sG[14][sg_own - G2K], sG[14][sg_own]), gsum, dx, Sj, F);
        }
#pragma unroll
        for (int v = 0; v < 5; ++v) sFj[v][tid] = F[v];
      }
      __builtin_amdgcn_sched_barrier(0);
      place();
      rj = own ? tj : tk;
      rk = own ? tk : kl;
      kgeo();
      if (kface) {
        double F[5];
        const int KK = ng + k0 + rk, JJ = ng + j0 + rj;
        const int side = wall_of(2, KK);
        if (side >= 0) {
          wall_flux(2, side, I, JJ, KK, F);
        } else {
          const int sp = (rj + 2) * H2K + (rk + 2), sg = (rj + 1) * G2K + (rk + 1);
          const double dx[3] = {xr[0] - xk[0], xr[1] - xk[1], xr[2] - xk[2]};
          auto gsum = [&](int x) { return sG[x][sg - 1] + sG[x][sg]; };
          face_curv<SC>(nd, cell(sp - 2), cell(sp - 1), cell(sp), cell(sp + 1), fmax(sG[14][sg - 1], sG[14][sg]), gsum, dx, Sk, F);
        }
        const int slot = kface_slot(rj, rk);
#pragma unroll
        for (int v = 0; v < 5; ++v) sFk[v][slot] = F[v];
      }
    }
    __builtin_amdgcn_sched_barrier(0);
    __syncthreads();                             // j / k face exchange
    __builtin_amdgcn_s_setprio(0);
    place();
    hplace();
    if (ring_g) {
#pragma unroll
      for (int x = 0; x < 4; ++x) sH0[x][ht] = sP[x < 3 ? 1 + x : 5][hs];
    }
    W0 = W1;
    if (own_p) W1 = cell(sp_own);
    stage_plane(Pn);
    request(I + 2);
    // ---- carry: the lower i face of the own cell I; the sum of its j / k faces takes the own k
    //      face's slot, whose other reader is the row's lane before: in this wavefront, and the sum
    //      that is stored needs the load that reads it
    if (act && inner) {
      const int jup = tile_tid(tj + 1, tk), kown = kface_slot(tj, tk), kup = kface_slot(tj, tk + 1);
#pragma unroll
      for (int v = 0; v < 5; ++v) {
        const double d = (sFj[v][jup] - sFj[v][tid]) + (sFk[v][kup] - sFk[v][kown]);
        Cp[v] = Fin[v];
        sFk[v][kown] = d;
      }
    }
    __syncthreads();                             // plane I+1 staged
  }
}

}  // namespace wmx
