// The TRiSK layered core, FCT transport, SWE solver and air-sea coupling as gfx950 HIP kernels, with the host-side
// sequencing of each C-ABI entry point (the reference's Python drivers: layers.py, transport.py, swe.py, ocean.py).
//
// This file is compiled twice: with ISW_FORM_MIXED=0 and -ffp-contract=off into namespace isw_f64 (the plain FP64 form:
// every operation rounds on its own, as the reference's --fmad=false build), and with ISW_FORM_MIXED=1 and
// -ffp-contract=fast into namespace isw_mix (the reference's mixed form). capi.hip dispatches on the `prec` field.
//
// Design (MI355X): one thread per cell, edge or vertex, 256-thread blocks (four 64-wide waves), layer-major arrays so
// consecutive threads touch consecutive words. The reference's one-kernel-per-loop structure is fused wherever a
// value can be recomputed bit for bit instead of stored and re-read: the Bernoulli (cell) and PV (vertex) passes run
// in one launch; the fast sub-steps run several to a launch on patches with rings of neighbours (k_af_rings, k_bt_rings),
// read the stage's start state directly (no copies) and keep it in registers and LDS between them; the stage flux
// F = h_e * mean(u) is recomputed inside the limiter and the divergence instead of being stored, the limited
// flux's volume Fm is written by each edge's eI cell, and the wall mask is applied inside the kernels that write.
// Sums keep the reference's order (a cell's edges in cellEdge or cellEdgeAsc order, a vertex's three in table order, an
// edge's eoe neighbours ascending) but for two on the ring patches: a fast sub-step adds the wind's forcing Tp + G before
// the gradient (the reference adds them to it one by one), and the limiter sums a cell's outflow in cellEdge order and
// scales the sum by the step (the reference in cellEdgeAsc order, each term scaled). So the FP64 form matches the
// reference's double path to rounding: within 1e-12 of the largest value after a step.
#include <hip/hip_runtime.h>

#include <cmath>
#include <cstdint>
#include <cstdlib>
#include <type_traits>

#include "insilica_hip.h"
#include "diag.hpp"

#if ISW_FORM_MIXED
#define NS isw_mix
#define DIVBY(x, r) ((x) * (r))
typedef float fast;
#else
#define NS isw_f64
#define DIVBY(x, r) ((x) / (r))
typedef double fast;
#endif

namespace NS {

constexpr int BS = 256;
#define TID ((int)(blockIdx.x * blockDim.x + threadIdx.x))

static inline dim3 g1(long n) { return dim3((unsigned)((n + BS - 1) / BS)); }
static inline dim3 g2(long n, int y) { return dim3((unsigned)((n + BS - 1) / BS), (unsigned)y); }

// Passes over cells or vertices (40,962 / 81,920 at level 6) launch 64-thread blocks (one wave each) so that they
// still spread over all 256 CUs; column passes launch (64, L) blocks: 64 cells or edges, one thread row per layer.
constexpr int BS1 = 64;
static inline dim3 c1(long n) { return dim3((unsigned)((n + BS1 - 1) / BS1)); }
static inline dim3 c2(long n, int y) { return dim3((unsigned)((n + BS1 - 1) / BS1), (unsigned)y); }
// (64, 4) blocks over cells (or edges) x rows: four rows of the same 64 elements per block, their index tables
// and stencil weights shared in L1
static inline dim3 c4(long n, int y) { return dim3((unsigned)((n + BS1 - 1) / BS1), (unsigned)((y + 3) / 4)); }

// XCD-aware block order: the dispatcher deals consecutive blocks to the 8 XCDs in turn; renumbered so that each XCD
// takes one contiguous range of blocks, neighbouring cells (Hilbert-ordered) then gather through the same L2.
__device__ __forceinline__ int xblock() {
  const int nb = (int)gridDim.x, b = (int)blockIdx.x;
  const int q = nb >> 3, r = nb & 7, x = b & 7, k = b >> 3;
  return (x < r ? x * (q + 1) : r * (q + 1) + (x - r) * q) + k;
}
#define XTID ((int)(xblock() * blockDim.x + threadIdx.x))

// A cell's six table entries (edges or neighbours; pads -1 last) in three 8-byte loads, so that every gather that
// depends on them can be issued at once; sums then skip the pads in table order, as the reference's loops do.
__device__ __forceinline__ void ring6(const int* __restrict__ tab, int i, int (&e)[6]) {
  const int2* p = reinterpret_cast<const int2*>(tab + (size_t)i * 6);
  const int2 a = p[0], b = p[1], c = p[2];
  e[0] = a.x; e[1] = a.y; e[2] = b.x; e[3] = b.y; e[4] = c.x; e[5] = c.y;
}
__device__ __forceinline__ int ok0(int e) { return e < 0 ? 0 : e; }

// Settings of a layer stack passed by value (reference: Layers.__init__, src/insilica/layers.py:161-218).
struct LP {
  int L, air;
  double grav, cp, kappa, p0, floor_, div_damp, thin, shelf, nu4;
  double gp[ISW_LMAX], drag[ISW_LMAX], stress[ISW_LMAX];
  // a batch of worlds (all NULL for one world): the world of each cell and edge, per-world gravity, del^4 coefficient,
  // fast sub-steps, their length and 1/n per stage (isw_batch)
  const int32_t *wc, *we, *wn;
  const double *wgrav, *wnu4, *wtau, *winv;
  // tides (Boussinesq layers; NULL / 0 without): the potential per cell, the internal tide's drag per edge, the
  // bottom's quadratic drag coefficient
  const double *tide, *cbot;
  double cd_bot;
};

static LP make_lp(const isw_layers* s) {
  LP p;
  p.L = s->L; p.air = s->air;
  p.grav = s->grav; p.cp = s->cp; p.kappa = s->kappa; p.p0 = s->p0; p.floor_ = s->floor_; p.div_damp = s->div_damp;
  p.thin = s->thin; p.shelf = s->shelf; p.nu4 = s->nu4;
  for (int k = 0; k < ISW_LMAX; k++) { p.gp[k] = s->gp[k]; p.drag[k] = s->drag[k]; p.stress[k] = s->stress[k]; }
  const isw_batch* b = s->batch;
  p.wc = b ? b->wc : nullptr; p.we = b ? b->we : nullptr; p.wn = b ? b->nsub : nullptr;
  p.wgrav = b ? b->grav : nullptr; p.wnu4 = b ? b->nu4 : nullptr; p.wtau = b ? b->tau : nullptr;
  p.winv = b ? b->inv_n : nullptr;
  p.tide = s->air ? nullptr : s->tide;
  p.cbot = s->air ? nullptr : s->cbot;
  p.cd_bot = s->air ? 0.0 : s->cd_bot;
  return p;
}

// Gravity at a cell and the del^4 coefficient at an edge: the world's in a batch, else the stack's.
__device__ __forceinline__ double grav_at(const LP& p, int i) { return p.wc ? p.wgrav[p.wc[i]] : p.grav; }
__device__ __forceinline__ double nu4_at(const LP& p, int e) { return p.we ? p.wnu4[p.we[e]] : p.nu4; }

// A fast sub-step's element: in a batch its world's sub-step count and length for this stage (a world whose
// sub-steps are done skips), else the stack's.
struct Sub {
  bool active, last;
  double tau;
};
__device__ __forceinline__ Sub sub_at(const LP& p, const int32_t* wid, int x, int stage, int it, int n, double tau) {
  if (wid) {
    const int w = wid[x];
    n = p.wn[w * 3 + stage];
    tau = p.wtau[w * 3 + stage];
  }
  return Sub{it < n, it == n - 1, tau};
}

// What the DIVBY divisions take: the quantity (plain form) or its stored reciprocal (mixed form).
struct Div {
  const double *A, *de, *AV;
};
static Div divs(const isw_grid* g) {
#if ISW_FORM_MIXED
  return Div{g->rA, g->rde, g->rAV};
#else
  return Div{g->areaCell, g->de, g->areaV};
#endif
}

__global__ void k_copy(long n, const double* __restrict__ a, double* __restrict__ b) {
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) b[i] = a[i];
}

__global__ void k_fill(long n, double v, double* __restrict__ x) {
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) x[i] = v;
}

// A layer's thickness at an edge (layers.cu:42-45), ob NULL.
__device__ __forceinline__ double edge_h(double a, double b, double shelf) {
  const double m = a < b ? a : b;
  return shelf > 0 && m < shelf ? m : 0.5 * (a + b);
}

// A cell's kinetic energy times its area, sum over its edges of l d u^2 / 4, in table order.
__device__ __forceinline__ double cell_ke(const isw_grid& g, const double* __restrict__ ul, const int (&e)[6]) {
  double t[6];
#pragma unroll
  for (int m = 0; m < 6; m++) {
    const int ek = ok0(e[m]);
    t[m] = g.le[ek] * g.de[ek] * 0.25 * ul[ek] * ul[ek];
  }
  double ke = 0;
#pragma unroll
  for (int m = 0; m < 6; m++)
    if (e[m] >= 0) ke += t[m];
  return ke;
}

// ---------------------------------------------------------------------------------------------------------------
// Mesh operators: the vector Laplacian (trisk.cu:14-45). Cells and vertices in one launch.
// ---------------------------------------------------------------------------------------------------------------
__global__ __launch_bounds__(BS) void k_div_curl(isw_grid g, int L, int nbc, const double* __restrict__ u,
                                                 double* __restrict__ D, double* __restrict__ Z) {
  if ((int)blockIdx.x < nbc) {
    const int t = TID;
    if (t >= g.N * L) return;
    const int l = t / g.N, i = t - l * g.N;
    const double* ul = u + (size_t)l * g.E;
    int e[6];
    ring6(g.cellEdge, i, e);
    double tm[6];
#pragma unroll
    for (int k = 0; k < 6; k++) tm[k] = (double)g.cellSign[i * 6 + k] * g.le[ok0(e[k])] * ul[ok0(e[k])];
    double s = 0;
#pragma unroll
    for (int k = 0; k < 6; k++)
      if (e[k] >= 0) s += tm[k];
    D[t] = s / g.areaCell[i];
  } else {
    const int t = (int)((blockIdx.x - nbc) * blockDim.x + threadIdx.x);
    if (t >= g.NV * L) return;
    const int l = t / g.NV, v = t - l * g.NV;
    const double* ul = u + (size_t)l * g.E;
    double z = 0;
#pragma unroll
    for (int k = 0; k < 3; k++) {
      const int e = g.vEdge[v * 3 + k];
      z += (double)g.vEdgeSign[v * 3 + k] * g.de[e] * ul[e];
    }
    Z[t] = z / g.areaV[v];
  }
}

__global__ __launch_bounds__(BS) void k_edge_lap(isw_grid g, int L, const double* __restrict__ D,
                                                 const double* __restrict__ Z, double* __restrict__ out) {
  const int t = XTID;
  if (t >= g.E * L) return;
  const int l = t / g.E, e = t - l * g.E;
  const double* Dl = D + (size_t)l * g.N;
  const double* Zl = Z + (size_t)l * g.NV;
  out[t] = (Dl[g.eJ[e]] - Dl[g.eI[e]]) / g.de[e] - (Zl[g.ev2[e]] - Zl[g.ev1[e]]) / g.le[e];
}


// ---------------------------------------------------------------------------------------------------------------
// Column kernels at the step's start (layers.cu:33-74,165-175,234-250).
// ---------------------------------------------------------------------------------------------------------------
__global__ __launch_bounds__(BS) void k_air_stiff(int N, LP p, const double* __restrict__ h,
                                                  const double* __restrict__ th, double* __restrict__ S) {
  const int i = XTID;
  if (i >= N) return;
  const double gr = grav_at(p, i);
  double pr = 0;
  for (int k = 0; k < p.L; k++) {
    pr += gr * h[(size_t)k * N + i];
    const double dth = th[(size_t)k * N + i] - (k + 1 < p.L ? th[(size_t)(k + 1) * N + i] : 0.0);
    const double dpi = p.kappa * p.cp * pow(pr / p.p0, p.kappa) / pr;
    S[(size_t)k * N + i] = dth > 0 ? dth * gr * dpi : 0.0;
  }
}

__global__ __launch_bounds__(BS) void k_air_gfast(int N, LP p, double rgas, const double* __restrict__ h,
                                                  const double* __restrict__ th, double* __restrict__ Gc) {
  const int i = XTID;
  if (i >= N) return;
  const int L = p.L;
  double mu = 0;
  for (int k = 0; k < L; k++) mu += h[(size_t)k * N + i];
  int kb = L - 1;
  while (kb > 0 && h[(size_t)kb * N + i] < 2 * p.floor_) kb--;
  const double gr = grav_at(p, i);
  const double Ts = th[(size_t)kb * N + i] * pow(gr * mu / p.p0, p.kappa);
  double gc = rgas * Ts / mu;
  double above = 0;
  for (int j = 0; j < L - 1; j++) {
    above += h[(size_t)j * N + i];
    const double dth = th[(size_t)j * N + i] - th[(size_t)(j + 1) * N + i];
    if (dth > 0) gc += dth * rgas * pow(gr * above / p.p0, p.kappa) * above / (mu * mu);
  }
  Gc[i] = gc;
}

__global__ __launch_bounds__(BS) void k_lay_eta(int N, int L, const double* __restrict__ h,
                                                const double* __restrict__ b, double* __restrict__ eta) {
  const int i = XTID;
  if (i >= N) return;
  double z = b[i];
  for (int k = L - 1; k >= 0; k--) z += h[(size_t)k * N + i];
  eta[i] = z;
}

__global__ __launch_bounds__(BS) void k_lay_ubar(isw_grid g, int L, double shelf, const double* __restrict__ h,
                                                 const double* __restrict__ u, const double* __restrict__ wall,
                                                 double* __restrict__ ubar) {
  const int e = XTID;
  if (e >= g.E) return;
  const int N = g.N, eI = g.eI[e], eJ = g.eJ[e];
  double H = 0, U = 0;
  for (int k = 0; k < L; k++) {
    const double he = edge_h(h[(size_t)k * N + eI], h[(size_t)k * N + eJ], shelf);
    H += he;
    U += he * u[(size_t)k * g.E + e];
  }
  ubar[e] = wall && wall[e] == 0 ? 0.0 : U / H;
}

// ---------------------------------------------------------------------------------------------------------------
// Per stage, pass 1: the Bernoulli/Montgomery potential per cell (air_bern / lay_bern, layers.cu:83-158) and the PV
// at vertices (swe_vertex, fused.cu:82-98), in one launch of (64, L) blocks: blocks [0, nbc) take 64 cells, the rest
// 64 vertices; thread row y is layer y. For air each thread takes one interface's Exner power (the expensive `pow`),
// shared with the column through LDS; every thread then replays the column's sums in the reference's order.
// ---------------------------------------------------------------------------------------------------------------
__global__ __launch_bounds__(512) void k_bern_pv(isw_grid g, LP p, Div dv, int nbc, const double* __restrict__ h,
                                                 const double* __restrict__ u, const double* __restrict__ th,
                                                 const double* __restrict__ b, const double* __restrict__ S,
                                                 const double* __restrict__ fV, double* __restrict__ B,
                                                 double* __restrict__ pibar, double* __restrict__ q) {
  const int N = g.N, E = g.E, L = p.L;
  const int j = threadIdx.x, k = threadIdx.y;
  if ((int)blockIdx.x < nbc) {
    __shared__ double sx[ISW_LMAX][BS1];
    const int i = blockIdx.x * BS1 + j;
    const bool live = i < N;
    const int ic = live ? i : 0;
    int e[6];
    ring6(g.cellEdge, ic, e);
    const double ke = cell_ke(g, u + (size_t)k * E, e);
    if (p.air) {
      const double gr = grav_at(p, ic);
      double pr = 0, pt = 0;
      for (int m = 0; m <= k; m++) {
        pt = pr;
        pr = pr + gr * h[(size_t)m * N + ic];
      }
      const double x = pow(pr / p.p0, p.kappa);
      sx[k][j] = x;
      __syncthreads();
      if (!live) return;
      const double xt = k ? sx[k - 1][j] : 0.0;
      pibar[(size_t)k * N + i] = p.cp * (pr * x - pt * xt) / ((p.kappa + 1) * (pr - pt));
      double M = gr * b[i] + th[(size_t)(L - 1) * N + i] * p.cp * sx[L - 1][j];
      for (int m = L - 2; m >= k; m--) M = M + (th[(size_t)m * N + i] - th[(size_t)(m + 1) * N + i]) * p.cp * sx[m][j];
      double P[ISW_LMAX];
      double a = 0;
      for (int m = 0; m < L; m++) { a += h[(size_t)m * N + i]; P[m] = a; }
      double ph = 0;
      for (int m = L - 1; m >= k; m--) ph += S[(size_t)m * N + i] * P[m];
      B[(size_t)k * N + i] = M - ph + DIVBY(ke, dv.A[i]);
    } else {
      if (!live) return;
      double z[ISW_LMAX];
      double s = b[i];
      for (int m = L - 1; m >= 0; m--) { s += h[(size_t)m * N + i]; z[m] = s; }
      double Mp = 0;
      for (int m = 1; m <= k; m++) Mp += p.gp[m - 1] * z[m];
      double Bk = Mp + ke / g.areaCell[i];
      if (p.tide) Bk -= p.tide[i];                 // (the tide's force grad V on every layer, layers.cu:106)
      B[(size_t)k * N + i] = Bk;
    }
  } else {
    const int v = ((int)blockIdx.x - nbc) * BS1 + j;
    if (v >= g.NV) return;
    const int l = k;
    const double* hl = h + (size_t)l * N;
    const double* ul = u + (size_t)l * E;
    double hv = 0, z = 0;
#pragma unroll
    for (int m = 0; m < 3; m++) {
      const int c = g.vCell[v * 3 + m];
      hv += g.kite[c * 6 + g.vSlot[v * 3 + m]] * hl[c] * 1.0;
    }
#pragma unroll
    for (int m = 0; m < 3; m++) {
      const int ee = g.vEdge[v * 3 + m];
      z += (double)g.vEdgeSign[v * 3 + m] * g.de[ee] * ul[ee];
    }
    q[(size_t)l * g.NV + v] = (DIVBY(z, dv.AV[v]) + fV[v]) / DIVBY(hv, dv.AV[v]);
  }
}

// Per stage, pass 2 (lay_edge_hq, layers.cu:254-263): each edge's h_e and q_e; [edge][layer][h_e, u, q_e] packed for
// the PV flux's neighbour gathers.
__global__ __launch_bounds__(BS) void k_edge_hq(isw_grid g, int L, double shelf, const double* __restrict__ h,
                                                const double* __restrict__ q, const double* __restrict__ u,
                                                double* __restrict__ he, fast* __restrict__ pk,
                                                fast* __restrict__ cf) {
  const int t = XTID;
  if (t >= g.E * L) return;
  const int l = t / g.E, e = t - l * g.E;
  const int N = g.N, NV = g.NV;
  const double hv = edge_h(h[(size_t)l * N + g.eI[e]], h[(size_t)l * N + g.eJ[e]], shelf);
  const double qv = 0.5 * (q[(size_t)l * NV + g.ev1[e]] + q[(size_t)l * NV + g.ev2[e]]);
  he[t] = hv;
  if (cf) cf[t] = (fast)(g.le[e] * hv);          // (the air's fast sub-steps' flux coefficient)
  fast* pp = pk + ((size_t)e * L + l) * 3;
  pp[0] = (fast)hv; pp[1] = (fast)u[t]; pp[2] = (fast)qv;
}

// Per stage, pass 3 (lay_slow, layers.cu:269-359): the slow momentum tendency of every layer of an edge (W-weight PV
// flux with the thin-layer cap, -grad B, drag, exact-exponential stress, pibar grad theta for air, del^4), its
// thickness-weighted column mean G, T' = T - G, H_e and the column wind. Bound by the latency of the chain edge -> ~10
// neighbours -> their packed records: the indices and weights load first, then all of a layer's records whether or not
// the edge has that many neighbours (a missing one repeats the first and is left out of the sum), so that no branch
// stands between the loads (three layers at level 6, mixed: 16.0 -> 12.8 us; two at level 7 33.9 -> 27.1).
// One thread per edge with the layers in registers (L a compile-time count): the edge's neighbour list and weights
// load once for every layer and each neighbour's L packed records are one contiguous run. ROWS: a (64, L) block with a
// thread per layer, for meshes too small to fill the card otherwise; the column's blend and mean then go through LDS.
// The column sums run in the reference's layer order in both.
template <int L, bool ROWS>
__global__ __launch_bounds__(ROWS ? 64 * L : BS) void k_slow_e(isw_grid g, LP p, Div dv, double dts,
                                                               const fast* __restrict__ pk, const fast* __restrict__ wf,
                                                               const double* __restrict__ hedge,
                                                               const double* __restrict__ u, const double* __restrict__ B,
                                                               const double* __restrict__ lap4,
                                                               const double* __restrict__ th,
                                                               const double* __restrict__ pibar, double* __restrict__ Tp,
                                                               double* __restrict__ G, double* __restrict__ He,
                                                               double* __restrict__ ubs) {
  const int N = g.N, E = g.E;
  const int at = ROWS ? xblock() * 64 + (int)threadIdx.x : XTID;
  const bool live = at < E;
  if (!ROWS && !live) return;
  const int e = live ? at : 0;
  const int eI = g.eI[e], eJ = g.eJ[e];
  const int m0 = g.eoeStart[e], m1 = g.eoeStart[e + 1];
  constexpr int NB = 10;
  int nb[NB];
  fast w[NB];
#pragma unroll
  for (int m = 0; m < NB; m++) {
    const int mm = m0 + m < m1 ? m0 + m : (m1 > m0 ? m0 : 0);
    nb[m] = g.eoe[mm];
    w[m] = wf[mm];
  }
  const double rde = dv.de[e];
  const double nu4 = lap4 ? nu4_at(p, e) : 0.0;
  auto layer = [&](int k, double& dk, double& hk, double& uk, double& sqk) {
    const size_t o = (size_t)k * E + e;
    const double he = hedge[o];
    const double ue = u[o];
    const fast cap = (fast)(p.thin * he), qf = pk[((size_t)e * L + k) * 3 + 2];
    fast hn[NB], un[NB], qn[NB];
#pragma unroll
    for (int m = 0; m < NB; m++) {
      const fast* pp = pk + ((size_t)nb[m] * L + k) * 3;
      hn[m] = pp[0]; un[m] = pp[1]; qn[m] = pp[2];
    }
    fast Q = 0;
#pragma unroll
    for (int m = 0; m < NB; m++) {
      const fast F2 = (hn[m] > cap ? cap : hn[m]) * un[m];
      const fast Qm = Q + w[m] * F2 * (fast)0.5 * (qf + qn[m]);
      Q = m0 + m < m1 ? Qm : Q;
    }
    for (int m = m0 + NB; m < m1; m++) {           // (meshes with more neighbours per edge than 10)
      const fast* pp = pk + ((size_t)g.eoe[m] * L + k) * 3;
      fast h2 = pp[0];
      if (h2 > cap) h2 = cap;
      const fast F2 = h2 * pp[1];
      Q += wf[m] * F2 * (fast)0.5 * (qf + pp[2]);
    }
    const double shk = p.shelf;
    const double sq0 =
        shk > 0 && he < shk ? (he - 2 * p.floor_ > 0 ? (he - 2 * p.floor_) / (shk - 2 * p.floor_) : 0.0) : 1.0;
    const double sqv = th ? 1.0 : sq0;
    const double* Bl = B + (size_t)k * N;
    double d = Q - DIVBY(sqv * (Bl[eJ] - Bl[eI]), rde) - (p.drag[k] + (1 - sqv) / 21600.0) * ue;
    double ck = p.stress[k];
    if (k == L - 1 && (p.cd_bot > 0 || p.cbot)) {
      // (tides, layers.cu:305-315) the bottom layer's quadratic stress cd |u|, |u| from the normal wind and the TRiSK
      // tangential wind of the packed neighbours' u; the internal tide's drag
      if (p.cd_bot > 0) {
        fast vt = 0;
#pragma unroll
        for (int m = 0; m < NB; m++) vt = m0 + m < m1 ? vt + w[m] * un[m] : vt;
        for (int m = m0 + NB; m < m1; m++) vt += wf[m] * pk[((size_t)g.eoe[m] * L + k) * 3 + 1];
        ck += p.cd_bot * sqrt(ue * ue + (double)vt * (double)vt);
      }
      if (p.cbot) ck += p.cbot[e];
    }
    if (ck != 0) {
      const double r = ck / (he > p.floor_ ? he : p.floor_);
      d = d - ((r * dts > 1e-8) ? (1 - exp(-r * dts)) / dts : r) * ue;
    }
    if (th) {
      const double* tl = th + (size_t)k * N;
      const double* pl = pibar + (size_t)k * N;
      d = d + DIVBY(0.5 * (pl[eI] + pl[eJ]) * (tl[eJ] - tl[eI]), rde);
    }
    if (lap4) d = d - nu4 * lap4[o];
    dk = d;
    hk = he;
    uk = ue;
    sqk = sq0;
  };
  double dk[L], hk[L], uk[L], sqk[L];
  if (ROWS) {
    __shared__ double sc[4][L][64];
    const int j = (int)threadIdx.x, y = (int)threadIdx.y;
    double a, b, c, d;
    layer(y, a, b, c, d);
    sc[0][y][j] = a; sc[1][y][j] = b; sc[2][y][j] = c; sc[3][y][j] = d;
    __syncthreads();
    if (!live) return;
#pragma unroll
    for (int m = 0; m < L; m++) { dk[m] = sc[0][m][j]; hk[m] = sc[1][m][j]; uk[m] = sc[2][m][j]; sqk[m] = sc[3][m][j]; }
  } else {
#pragma unroll
    for (int k = 0; k < L; k++) layer(k, dk[k], hk[k], uk[k], sqk[k]);
  }
  // the blend of a thin layer's tendency with its nearest thick neighbours' (shelf), then the column mean
  const bool blend = th && p.shelf > 0;
  auto blended = [&](int m) {
    double Tm = dk[m];
    if (blend && sqk[m] < 1) {
      double wgt = 0, s = 0;
      bool up = true, down = true;
#pragma unroll
      for (int q = L - 1; q >= 0; q--)
        if (q < m && up && sqk[q] >= 1) { wgt += hk[q]; s += hk[q] * dk[q]; up = false; }
#pragma unroll
      for (int q = 0; q < L; q++)
        if (q > m && down && sqk[q] >= 1) { wgt += hk[q]; s += hk[q] * dk[q]; down = false; }
      if (wgt > 0) Tm = sqk[m] * dk[m] + (1 - sqk[m]) * s / wgt;
    }
    return Tm;
  };
  double H = 0, U = 0, GT = 0;
#pragma unroll
  for (int m = 0; m < L; m++) {
    H += hk[m];
    U += hk[m] * uk[m];
  }
  double Tb[L];
#pragma unroll
  for (int m = 0; m < L; m++) {
    Tb[m] = blended(m);
    GT += hk[m] * Tb[m];
  }
  const double gg = GT / H;
#pragma unroll
  for (int k = 0; k < L; k++) if (!ROWS || k == (int)threadIdx.y) Tp[(size_t)k * E + e] = Tb[k] - gg;
  if (ROWS && threadIdx.y) return;
  G[e] = gg;
  He[e] = H;
  ubs[e] = U / H;
}

// ---------------------------------------------------------------------------------------------------------------
// Air fast sub-steps (layers.cu:182-224): mass then wind, forward-backward, from the stage's start.
// The first sub-step reads the step's start (mu from h0, u from u0) and starts acc; the last writes the stage's wind.
// ---------------------------------------------------------------------------------------------------------------
// The mass sub-step: (64, L) blocks, thread (x, y) updates layer y's mass of one of 64 cells (its six edges gathered
// at once); the column's forward-weighted masses and the linear potential Phi* are then summed through LDS in the
// reference's order (P from the top, Phi from the bottom) by every thread for its own layer.
__global__ __launch_bounds__(512) void k_af_muphi(isw_grid g, LP p, Div dv, int stage, int it, int n, double tau,
                                                  const double* __restrict__ hedge,
                                                  const double* __restrict__ uf, const double* mu_src, double* mu,
                                                  const double* __restrict__ S, double* __restrict__ phi) {
  __shared__ double sa[ISW_LMAX][BS1], sS[ISW_LMAX][BS1];
  const int N = g.N, E = g.E, L = p.L;
  const int j = threadIdx.x, k = threadIdx.y;
  const int i = xblock() * BS1 + j;
  const bool live = i < N;
  const int ic = live ? i : 0;
  const Sub sb = sub_at(p, p.wc, ic, stage, it, n, tau);
  int e[6];
  ring6(g.cellEdge, ic, e);
  const double* hl = hedge + (size_t)k * E;
  const double* ul = uf + (size_t)k * E;
  double t[6];
#pragma unroll
  for (int m = 0; m < 6; m++) {
    const int ek = ok0(e[m]);
    t[m] = (double)g.cellSign[ic * 6 + m] * g.le[ek] * hl[ek] * ul[ek];
  }
  double div = 0;
#pragma unroll
  for (int m = 0; m < 6; m++)
    if (e[m] >= 0) div += t[m];
  const size_t o = (size_t)k * N + ic;
  const double m0 = mu_src[o];
  const double m1 = m0 - DIVBY(sb.tau * div, dv.A[ic]);
  sa[k][j] = m1 + p.div_damp * (m1 - m0);
  sS[k][j] = S[o];
  __syncthreads();
  if (!live || !sb.active) return;
  mu[o] = m1;
  double P[ISW_LMAX];
  double a = 0;
  for (int m = 0; m < L; m++) { a += sa[m][j]; P[m] = a; }
  double ph = 0;
  for (int m = L - 1; m >= k; m--) ph += sS[m][j] * P[m];
  phi[o] = ph;
}

__global__ __launch_bounds__(BS) void k_af_u(isw_grid g, int L, Div dv, LP p, int stage, int it, int n, double tau,
                                             const double* __restrict__ phi, const double* __restrict__ Tp,
                                             const double* __restrict__ G, const double* uin, double* acc, double* uf,
                                             double* un) {
  const int t = XTID;
  if (t >= g.E * L) return;
  const int l = t / g.E, e = t - l * g.E;
  const Sub sb = sub_at(p, p.we, e, stage, it, n, tau);
  if (!sb.active) return;
  const double v = uin[t];
  acc[t] = it == 0 ? 0.0 + v : acc[t] + v;
  const double* pl = phi + (size_t)l * g.N;
  (sb.last ? un : uf)[t] = v + sb.tau * (DIVBY(-(pl[g.eJ[e]] - pl[g.eI[e]]), dv.de[e]) + Tp[t] + G[e]);
}

// ---------------------------------------------------------------------------------------------------------------
// Several fast sub-steps in one launch, on the grid's patches (tables rg_*): a block holds its patch's cells and the
// rings of neighbours within m cells of it, takes the state of all of them in registers once, and steps m times. The
// first step's masses are those of every ring, and each further step's reach one ring less, so the m-th step's are the
// patch's own; what neighbours recompute they compute from the same inputs in the same order, so every copy is the same to
// the bit. Between the steps only LDS is touched: the edges' threads leave each flux coef * u there, the cells' threads
// leave each potential. So a launch pays its chain of dependent loads (arguments, the patch's record, the index lists,
// the values) once for m steps, about 6 us of it before the first step at level 6 (three layers, mixed: 7.7 us for one
// step, 9.4 for two, 11.2 for three); what bounds each further step is LDS: six fluxes per cell, two potentials per edge.
// Two buffers alternate for masses and winds, as a neighbour block may still read a launch's inputs. A patch's cells are of
// one world, so a batch's counts and lengths are the block's.
// ---------------------------------------------------------------------------------------------------------------
constexpr int RBS = 256;
// The sub-steps a launch takes. Air: 3 (level 6, three layers, nfast 15, the 28 sub-steps of a step: 216 us at one per
// launch, 140 at two, 112 at three; at four a patch needs two cells and four edges to a thread, 190 registers and two
// blocks per CU: 125 us. 384 threads with one cell each at five: 113 us). Ocean (one value per cell): 4 (level 7, 70
// sub-steps: 815 us at one, 535 at two, 528 at three, 498 at four; five need five edges to a thread and gain nothing).
constexpr int AIR_STEPS = 3, SEA_STEPS = 4;

struct Ring {
  int c0, e0, own;                                 // the patch's first entries in the lists, its owned edges
  const int* head;
  int k;
  __device__ __forceinline__ int cells(int r) const { return head[3 + r]; }
  __device__ __forceinline__ int edges(int r) const { return head[4 + k + r]; }
};
__device__ __forceinline__ Ring ring_of(const isw_grid& g) {
  const int* h = g.rg_head + 16 * (size_t)xblock();
  return Ring{h[0], h[1], h[2], h, g.rg_k};
}
// A batch's sub-steps left to this launch (at most m) and their length, for the block's world.
__device__ __forceinline__ bool ring_sub(const LP& p, int cell, int stage, int it0, int n, int& m, double& tau,
                                         bool& last) {
  if (p.wc) {
    const int w = p.wc[cell];
    n = p.wn[w * 3 + stage];
    tau = p.wtau[w * 3 + stage];
  }
  m = min(m, n - it0);
  last = it0 + m == n;
  return m > 0;
}
// A cell's six edges in the fluxes left in LDS: their places (in cellEdge order; a missing edge's is `none`, which holds
// 0) and the signs of the cell on them, as the sign bit to flip.
struct RingCell {
  int at[6];
  unsigned flip[6];
  __device__ __forceinline__ void set(const int* __restrict__ s, int none) {
#pragma unroll
    for (int k = 0; k < 3; k++) {
      const unsigned w = (unsigned)s[k];
      const int q0 = (int)(w & 0x7fffu), q1 = (int)(w >> 16 & 0x7fffu);
      at[2 * k] = q0 == 0x7fff ? none : q0;
      at[2 * k + 1] = q1 == 0x7fff ? none : q1;
      flip[2 * k] = (w & 0x8000u) << 16;
      flip[2 * k + 1] = w & 0x80000000u;
    }
  }
  __device__ __forceinline__ double div(const double* F) const {
    double t[6];
#pragma unroll
    for (int k = 0; k < 6; k++) {
      const double f = F[at[k]];
      t[k] = __hiloint2double((int)((unsigned)__double2hiint(f) ^ flip[k]), __double2loint(f));
    }
    return ((((t[0] + t[1]) + t[2]) + t[3]) + t[4]) + t[5];
  }
  // What flows out of the cell (as the reference counts it: a flux that is not a number is its second cell's).
  __device__ __forceinline__ double out(const double* F) const {
    double s = 0;
#pragma unroll
    for (int k = 0; k < 6; k++) {
      const double f = F[at[k]];
      const double x = __hiloint2double((int)((unsigned)__double2hiint(f) ^ flip[k]), __double2loint(f));
      if ((f > 0) != (flip[k] != 0)) s += x;
    }
    return s;
  }
};
// x / d with r = 1 / d at hand: the plain form's rounds as the division does (a quotient corrected by its exact
// remainder; the fix-up keeps an infinite quotient infinite, whose remainder is not a number), the mixed form's is the
// product (its Div holds reciprocals).
__device__ __forceinline__ double over(double x, double d, double r) {
#if ISW_FORM_MIXED
  return x * d;
#else
  const double q = x * r;
  return __builtin_amdgcn_div_fixup(__builtin_fma(__builtin_fma(-q, d, x), r, q), d, x);
#endif
}
__device__ __forceinline__ double recip(double d) {
#if ISW_FORM_MIXED
  return d;
#else
  return 1.0 / d;
#endif
}

// The air's: EPT edges and CPT cells to a thread.
template <int L, int EPT, int CPT>
__global__ __launch_bounds__(RBS) void k_af_rings(isw_grid g, LP p, Div dv, int stage, int it0, int m, int n, double tau,
                                                  const fast* __restrict__ coef, const double* __restrict__ uin,
                                                  const double* __restrict__ mu_src, double* __restrict__ mu_out,
                                                  const double* __restrict__ S, const double* __restrict__ Tp,
                                                  const double* __restrict__ G, double* __restrict__ acc,
                                                  double* __restrict__ uout, double* __restrict__ un) {
  extern __shared__ double sm[];
  constexpr int PE = EPT * RBS + 2, PC = CPT * RBS;
  const int N = g.N, E = g.E, t = (int)threadIdx.x;
  double* F = sm;                                  // [L][PE] coef * u, the last but one 0
  double* phi = sm + L * PE;                       // [L][PC] Phi*
  const Ring r = ring_of(g);
  bool last;
  if (!ring_sub(p, g.rg_cell[r.c0], stage, it0, n, m, tau, last)) return;
  const int ncm = r.cells(m), nem = r.edges(m), nem1 = r.edges(m - 1);
  // the edges' state: the wind, its forcing Tp + G, the flux's coefficient l_e h_e, 1 / d_e (or d_e), both cells' places
  double v[EPT][L], f[EPT][L], de[EPT], rde[EPT], a0[L];
  fast cf[EPT][L];
  int e_[EPT], ec[EPT];
#pragma unroll
  for (int j = 0; j < EPT; j++) {
    const int q = t + j * RBS;
    if (q < nem) e_[j] = g.rg_edge[r.e0 + q];
    if (q < nem1) ec[j] = g.rg_ecell[r.e0 + q];
  }
  int c_[CPT];
  RingCell rc[CPT];
#pragma unroll
  for (int j = 0; j < CPT; j++) {
    const int q = t + j * RBS;
    if (q < ncm) {
      c_[j] = g.rg_cell[r.c0 + q];
      rc[j].set(g.rg_slot + 3 * (size_t)(r.c0 + q), PE - 2);
    }
  }
#pragma unroll
  for (int j = 0; j < EPT; j++) {
    const int q = t + j * RBS;
    if (q < nem) {
      const int e = e_[j];
#pragma unroll
      for (int l = 0; l < L; l++) {
        v[j][l] = uin[(size_t)l * E + e];
        cf[j][l] = coef[(size_t)l * E + e];
      }
      if (q < nem1) {
        de[j] = dv.de[e];
        rde[j] = recip(de[j]);
        const double Ge = G[e];
#pragma unroll
        for (int l = 0; l < L; l++) f[j][l] = Tp[(size_t)l * E + e] + Ge;
      }
    }
  }
  if (t < r.own && it0 > 0) {
#pragma unroll
    for (int l = 0; l < L; l++) a0[l] = acc[(size_t)l * E + e_[0]];
  } else {
#pragma unroll
    for (int l = 0; l < L; l++) a0[l] = 0.0;
  }
  double mu[CPT][L], Sk[CPT][L], A[CPT], rA[CPT];
#pragma unroll
  for (int j = 0; j < CPT; j++)
    if (t + j * RBS < ncm) {
      A[j] = dv.A[c_[j]];
      rA[j] = recip(A[j]);
#pragma unroll
      for (int l = 0; l < L; l++) {
        mu[j][l] = mu_src[(size_t)l * N + c_[j]];
        Sk[j][l] = S[(size_t)l * N + c_[j]];
      }
    }
#pragma unroll
  for (int j = 0; j < EPT; j++) {
    const int q = t + j * RBS;
    if (q < nem)
#pragma unroll
      for (int l = 0; l < L; l++) F[l * PE + q] = (double)cf[j][l] * v[j][l];
  }
  if (t < L) F[t * PE + PE - 2] = 0.0;
  for (int it = 0; it < m; it++) {
    const int nc = r.cells(m - it), ne = it + 1 < m ? r.edges(m - it - 1) : r.own;
    __syncthreads();
    // the masses of the rings this step still reaches, and Phi* from their forward-weighted sum
#pragma unroll
    for (int j = 0; j < CPT; j++) {
      const int q = t + j * RBS;
      if (q >= nc) continue;
      double P[L], a = 0;
#pragma unroll
      for (int l = 0; l < L; l++) {
        const double m0 = mu[j][l];
        const double m1 = m0 - over(tau * rc[j].div(F + l * PE), A[j], rA[j]);
        mu[j][l] = m1;
        a += m1 + p.div_damp * (m1 - m0);
        P[l] = a;
      }
      double ph = 0;
#pragma unroll
      for (int l = L - 1; l >= 0; l--) {
        ph += Sk[j][l] * P[l];
        phi[l * PC + q] = ph;
      }
    }
    __syncthreads();
    // the winds of the edges inside those rings
#pragma unroll
    for (int j = 0; j < EPT; j++) {
      const int q = t + j * RBS;
      if (q >= ne) continue;
      const int cI = ec[j] & 0xffff, cJ = ec[j] >> 16;
#pragma unroll
      for (int l = 0; l < L; l++) {
        if (j == 0) a0[l] += v[j][l];
        v[j][l] = v[j][l] + tau * (over(-(phi[l * PC + cJ] - phi[l * PC + cI]), de[j], rde[j]) + f[j][l]);
        F[l * PE + q] = (double)cf[j][l] * v[j][l];
      }
    }
  }
  if (t < r.own) {
    double* out = last ? un : uout;
#pragma unroll
    for (int l = 0; l < L; l++) {
      acc[(size_t)l * E + e_[0]] = a0[l];
      out[(size_t)l * E + e_[0]] = v[0][l];
    }
  }
  if (t < r.cells(0))
#pragma unroll
    for (int l = 0; l < L; l++) mu_out[(size_t)l * N + c_[0]] = mu[0][l];
}

// The ocean's barotropic sub-steps (layers.cu:366-388), the wall mask of the reference's lay_mask calls fused in: the
// surface height of the rings' cells, its potential Gc (eta + gamma (eta - eta_prev)), the barotropic wind of their
// edges. The last sub-step writes ub_fin (what the stage's update reads).
template <int EPT, int CPT>
__global__ __launch_bounds__(RBS) void k_bt_rings(isw_grid g, Div dv, LP p, int stage, int it0, int m, int n, double tau,
                                                  double gamma, const double* __restrict__ He,
                                                  const double* __restrict__ ub_src, const double* __restrict__ eta_src,
                                                  double* __restrict__ eta_out, const double* __restrict__ G,
                                                  const double* __restrict__ Gc, const double* __restrict__ wall,
                                                  double* __restrict__ acc, double* __restrict__ ub_out,
                                                  double* __restrict__ ub_fin) {
  constexpr int PE = EPT * RBS + 2;
  extern __shared__ double sm[];
  const int t = (int)threadIdx.x;
  double* F = sm;                                  // [PE] l_e H_e u, the last but one 0
  double* x = sm + PE;                             // the potential
  const Ring r = ring_of(g);
  bool last;
  if (!ring_sub(p, g.rg_cell[r.c0], stage, it0, n, m, tau, last)) return;
  const int ncm = r.cells(m), nem = r.edges(m), nem1 = r.edges(m - 1);
  double v[EPT], cf[EPT], f[EPT], de[EPT], rde[EPT], wl[EPT], a0 = 0;
  int e_[EPT], ec[EPT], c_[CPT];
  RingCell rc[CPT];
#pragma unroll
  for (int j = 0; j < EPT; j++) {
    const int q = t + j * RBS;
    if (q < nem) e_[j] = g.rg_edge[r.e0 + q];
    if (q < nem1) ec[j] = g.rg_ecell[r.e0 + q];
  }
#pragma unroll
  for (int j = 0; j < CPT; j++) {
    const int q = t + j * RBS;
    if (q < ncm) {
      c_[j] = g.rg_cell[r.c0 + q];
      rc[j].set(g.rg_slot + 3 * (size_t)(r.c0 + q), PE - 2);
    }
  }
#pragma unroll
  for (int j = 0; j < EPT; j++) {
    const int q = t + j * RBS;
    if (q < nem) {
      const int e = e_[j];
      v[j] = ub_src[e];
      cf[j] = g.le[e] * He[e];
      if (q < nem1) {
        de[j] = dv.de[e];
        rde[j] = recip(de[j]);
        f[j] = G[e];
        wl[j] = wall ? wall[e] : 1.0;
      }
    }
  }
  if (t < r.own && it0 > 0) a0 = acc[e_[0]];
  double et[CPT], A[CPT], rA[CPT], gc[CPT];
#pragma unroll
  for (int j = 0; j < CPT; j++)
    if (t + j * RBS < ncm) {
      et[j] = eta_src[c_[j]];
      A[j] = dv.A[c_[j]];
      rA[j] = recip(A[j]);
      gc[j] = Gc[c_[j]];
    }
#pragma unroll
  for (int j = 0; j < EPT; j++)
    if (t + j * RBS < nem) F[t + j * RBS] = cf[j] * v[j];
  if (t == 0) F[PE - 2] = 0.0;
  for (int it = 0; it < m; it++) {
    const int nc = r.cells(m - it), ne = it + 1 < m ? r.edges(m - it - 1) : r.own;
    __syncthreads();
#pragma unroll
    for (int j = 0; j < CPT; j++) {
      const int q = t + j * RBS;
      if (q >= nc) continue;
      const double e0 = et[j], e1 = e0 - over(tau * rc[j].div(F), A[j], rA[j]);
      x[q] = gc[j] * (e1 + gamma * (e1 - e0));
      et[j] = e1;
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < EPT; j++) {
      const int q = t + j * RBS;
      if (q >= ne) continue;
      if (j == 0) a0 += v[j];
      v[j] = v[j] + tau * (over(-(x[ec[j] >> 16] - x[ec[j] & 0xffff]), de[j], rde[j]) + f[j]);
      if (wl[j] == 0) {
        v[j] = 0;
        if (j == 0) a0 = 0;
      }
      F[q] = cf[j] * v[j];
    }
  }
  if (t < r.own) {
    (last ? ub_fin : ub_out)[e_[0]] = v[0];
    acc[e_[0]] = a0;
  }
  if (t < r.cells(0)) eta_out[c_[0]] = et[0];
}

__global__ __launch_bounds__(BS) void k_bt_eta(isw_grid g, Div dv, LP p, int stage, int it, int n, double tau,
                                               const double* __restrict__ He, const double* __restrict__ ub,
                                               const double* eta_src, double* eta, double* __restrict__ eta_prev) {
  const int i = XTID;
  if (i >= g.N) return;
  const Sub sb = sub_at(p, p.wc, i, stage, it, n, tau);
  if (!sb.active) return;
  const double e0 = eta_src[i];
  eta_prev[i] = e0;
  int e[6];
  ring6(g.cellEdge, i, e);
  double t[6];
#pragma unroll
  for (int m = 0; m < 6; m++) {
    const int ek = ok0(e[m]);
    t[m] = (double)g.cellSign[i * 6 + m] * g.le[ek] * He[ek] * ub[ek];
  }
  double div = 0;
#pragma unroll
  for (int m = 0; m < 6; m++)
    if (e[m] >= 0) div += t[m];
  eta[i] = e0 - DIVBY(sb.tau * div, dv.A[i]);
}

__global__ __launch_bounds__(BS) void k_bt_u(isw_grid g, Div dv, LP p, int stage, int it, int n, double tau,
                                             double gamma, const double* __restrict__ eta,
                                             const double* __restrict__ eta_prev, const double* __restrict__ G,
                                             const double* __restrict__ Gc, const double* __restrict__ wall,
                                             const double* ub_src, double* ub, double* acc) {
  const int e = XTID;
  if (e >= g.E) return;
  const Sub sb = sub_at(p, p.we, e, stage, it, n, tau);
  if (!sb.active) return;
  const double v = ub_src[e];
  double a = it == 0 ? 0.0 + v : acc[e] + v;
  const int i = g.eI[e], j = g.eJ[e];
  const double ej = Gc[j] * (eta[j] + gamma * (eta[j] - eta_prev[j]));
  const double ei = Gc[i] * (eta[i] + gamma * (eta[i] - eta_prev[i]));
  double un = v + sb.tau * (DIVBY(-(ej - ei), dv.de[e]) + G[e]);
  if (wall && wall[e] == 0) { un = 0; a = 0; }
  ub[e] = un;
  acc[e] = a;
}

// ---------------------------------------------------------------------------------------------------------------
// The stage's layer fluxes, limiter and update (layers.cu:220-224,392-447). F is recomputed where it is read:
// air F = h_e acc / n (af_flux); ocean F = h_e (u - ubar*) + h_e ubar_avg (lay_flux), 0 on walls.
// ---------------------------------------------------------------------------------------------------------------
struct FluxSrc {
  int air, stage;
  double inv_n, shelf;
  const int32_t* we;    // a batch's world per edge and per-world 1/n (else NULL: inv_n)
  const double* winv;
  const double *hedge, *acc;                  // air
  const double *hs, *us, *ubs, *bacc, *wall;  // ocean
};

__device__ __forceinline__ double stage_flux(const FluxSrc& f, const isw_grid& g, int l, int e) {
  const size_t o = (size_t)l * g.E + e;
  const double inv_n = f.we ? f.winv[f.we[e] * 3 + f.stage] : f.inv_n;
  if (f.air) return f.hedge[o] * f.acc[o] * inv_n;
  if (f.wall && f.wall[e] == 0) return 0.0;
  const double he = edge_h(f.hs[(size_t)l * g.N + g.eI[e]], f.hs[(size_t)l * g.N + g.eJ[e]], f.shelf);
  return he * (f.us[o] - f.ubs[e]) + he * (f.bacc[e] * inv_n);
}

__global__ __launch_bounds__(BS) void k_scale(isw_grid g, FluxSrc fs, double dts, double floor_,
                                              const double* __restrict__ h0, double* __restrict__ scale, int L) {
  const int t = XTID;
  if (t >= g.N * L) return;
  const int l = t / g.N, i = t - l * g.N;
  int e[6];
  ring6(g.cellEdgeAsc, i, e);
  double f[6];
  bool own[6];
#pragma unroll
  for (int m = 0; m < 6; m++) {
    const int ek = ok0(e[m]);
    f[m] = stage_flux(fs, g, l, ek) * g.le[ek] * dts;
    own[m] = g.eI[ek] == i;
  }
  double out = 0;
#pragma unroll
  for (int m = 0; m < 6; m++) {
    if (e[m] < 0) break;
    if (own[m]) { if (f[m] > 0) out += f[m]; }
    else if (!(f[m] > 0)) out -= f[m];
  }
  const double avail = h0[t] - floor_;
  const double cap = (avail > 0 ? avail : 0.0) * g.areaCell[i];
  scale[t] = out > cap ? cap / out : 1.0;
}

// lay_limit + lay_h: the limited fluxes summed into the new thickness; each edge's eI cell writes its Fm.
__global__ __launch_bounds__(BS) void k_limit_h(isw_grid g, Div dv, FluxSrc fs, double cdt, double dt,
                                                const double* __restrict__ scale, const double* h0, double* hn,
                                                double* __restrict__ Fm, int L) {
  const int t = XTID;
  if (t >= g.N * L) return;
  const int l = t / g.N, i = t - l * g.N;
  const double* sl = scale + (size_t)l * g.N;
  int e[6];
  ring6(g.cellEdge, i, e);
  double f[6], sc[6], le[6];
  int own[6];
#pragma unroll
  for (int m = 0; m < 6; m++) {
    const int ek = ok0(e[m]);
    f[m] = stage_flux(fs, g, l, ek);
    const int eI = g.eI[ek];
    own[m] = eI == i;
    sc[m] = f[m] > 0 ? sl[eI] : sl[g.eJ[ek]];
    le[m] = g.le[ek];
  }
  double div = 0;
#pragma unroll
  for (int m = 0; m < 6; m++) {
    if (e[m] < 0) break;
    const double fl = f[m] * sc[m];
    div += (double)g.cellSign[i * 6 + m] * le[m] * fl;
    if (Fm && own[m]) Fm[(size_t)l * g.E + e[m]] = fl * le[m] * dt;
  }
  const double v0 = h0[t];
  hn[t] = v0 - DIVBY(cdt * div, dv.A[i]);
}

// The limiter and the update in one launch on the grid's ring patches (k_scale, k_limit_h and the ocean's k_lay_u): a
// block leaves the stage's fluxes of its patch's and first ring's edges in LDS, each formed once (a pass over cells forms
// every edge's twice, in each of two passes: at level 7, two layers, 31 + 41 us and 7 us for the winds), then the scales
// of patch and ring, then limits its patch's edges and steps its cells. ring_h0: the step's starting thickness, read for
// the ring's cells too (where the stage writes over it the copy `keep` that the first stage left). Bound by its chain of
// loads at the smaller levels; the sums are in cellEdge order.
template <int L>
__global__ __launch_bounds__(RBS) void k_limit_rings(isw_grid g, Div dv, FluxSrc fs, double cdt, double dt, double floor_,
                                                     const double* __restrict__ ring_h0, double* __restrict__ keep,
                                                     double* __restrict__ hn, double* __restrict__ Fm,
                                                     const double* u0, const double* __restrict__ Tp,
                                                     const double* __restrict__ ub_end, const double* __restrict__ ub0,
                                                     double* un) {
  constexpr int EPT = 2, PE = EPT * RBS + 2, PC = RBS / 2;
  extern __shared__ double sm[];
  double* F = sm;                                  // [L][PE] l_e F, the last but one 0
  double* sc = sm + L * PE;                        // [L][PC] the cells' scales
  const int N = g.N, E = g.E, t = (int)threadIdx.x;
  const Ring r = ring_of(g);
  const int nc0 = r.cells(0), nc1 = r.cells(1), ne0 = r.edges(0), ne1 = r.edges(1);
  int e_[EPT], ec[EPT];
  double f[EPT][L], le[EPT];
#pragma unroll
  for (int j = 0; j < EPT; j++) {
    const int q = t + j * RBS;
    if (q < ne1) e_[j] = g.rg_edge[r.e0 + q];
    if (q < ne0) ec[j] = g.rg_ecell[r.e0 + q];
  }
  // two threads to a cell, each taking every other layer
  const int cq = t >> 1, l0 = t & 1;
  int ci = 0;
  RingCell rc;
  double A = 0, h0[(L + 1) / 2];
  if (cq < nc1) {
    ci = g.rg_cell[r.c0 + cq];
    rc.set(g.rg_slot + 3 * (size_t)(r.c0 + cq), PE - 2);
  }
#pragma unroll
  for (int j = 0; j < EPT; j++) {
    const int q = t + j * RBS;
    if (q < ne1) {
      const int e = e_[j];
      le[j] = g.le[e];
      const double inv_n = fs.we ? fs.winv[fs.we[e] * 3 + fs.stage] : fs.inv_n;
      const double ub = fs.air ? 0.0 : fs.ubs[e], ba = fs.air ? 0.0 : fs.bacc[e] * inv_n;
      const bool wall = !fs.air && fs.wall && fs.wall[e] == 0;
#pragma unroll
      for (int l = 0; l < L; l++) {
        const size_t o = (size_t)l * E + e;
        const double he = fs.hedge[o];
        f[j][l] = fs.air ? he * fs.acc[o] * inv_n : wall ? 0.0 : he * (fs.us[o] - ub) + he * ba;
      }
    }
  }
  if (cq < nc1) {
    A = g.areaCell[ci];
#pragma unroll
    for (int k = 0; k < (L + 1) / 2; k++)
      if (l0 + 2 * k < L) h0[k] = ring_h0[(size_t)(l0 + 2 * k) * N + ci];
  }
  // the ocean's winds, of the owned edges
  if (un && t < r.own) {
    const int e = e_[0];
    const double db = ub_end[e] - ub0[e];
    const bool wall = fs.wall && fs.wall[e] == 0;
#pragma unroll
    for (int l = 0; l < L; l++) {
      const size_t o = (size_t)l * E + e;
      un[o] = wall ? 0.0 : u0[o] + cdt * Tp[o] + db;
    }
  }
#pragma unroll
  for (int j = 0; j < EPT; j++) {
    const int q = t + j * RBS;
    if (q < ne1)
#pragma unroll
      for (int l = 0; l < L; l++) F[l * PE + q] = f[j][l] * le[j];
  }
  if (t < L) F[t * PE + PE - 2] = 0.0;
  __syncthreads();
  if (cq < nc1) {
#pragma unroll
    for (int k = 0; k < (L + 1) / 2; k++) {
      const int l = l0 + 2 * k;
      if (l >= L) continue;
      const double out = rc.out(F + l * PE) * cdt;
      const double avail = h0[k] - floor_;
      const double cap = (avail > 0 ? avail : 0.0) * A;
      sc[l * PC + cq] = out > cap ? cap / out : 1.0;
    }
  }
  __syncthreads();
#pragma unroll
  for (int j = 0; j < EPT; j++) {
    const int q = t + j * RBS;
    if (q < ne0) {
      const int cI = ec[j] & 0xffff, cJ = ec[j] >> 16;
#pragma unroll
      for (int l = 0; l < L; l++) {
        const double fl = f[j][l] * sc[l * PC + (f[j][l] > 0 ? cI : cJ)], lf = le[j] * fl;
        F[l * PE + q] = lf;
        if (Fm && q < r.own) Fm[(size_t)l * E + e_[j]] = lf * dt;
      }
    }
  }
  __syncthreads();
  if (cq < nc0) {
    const double Ad = dv.A[ci], rA = recip(Ad);
#pragma unroll
    for (int k = 0; k < (L + 1) / 2; k++) {
      const int l = l0 + 2 * k;
      if (l >= L) continue;
      const size_t o = (size_t)l * N + ci;
      hn[o] = h0[k] - over(cdt * rc.div(F + l * PE), Ad, rA);
      if (keep) keep[o] = h0[k];
    }
  }
}

__global__ __launch_bounds__(BS) void k_lay_u(int E, int L, double cdt, const double* u0, const double* __restrict__ Tp,
                                              const double* __restrict__ ub_end, const double* __restrict__ ub0,
                                              const double* __restrict__ wall, double* un) {
  const int t = XTID;
  if (t >= E * L) return;
  const int e = t % E;
  const double v = u0[t] + cdt * Tp[t] + (ub_end[e] - ub0[e]);
  un[t] = wall && wall[e] == 0 ? 0.0 : v;
}

// ---------------------------------------------------------------------------------------------------------------
// Interfacial stress, its heat, and the exchange between layers (layers.cu:454-621).
// ---------------------------------------------------------------------------------------------------------------
__global__ __launch_bounds__(BS) void k_lay_vmix(isw_grid g, int L, double c, double dt, double cd,
                                                 const double* __restrict__ h, const double* __restrict__ wall,
                                                 double* __restrict__ u, double* __restrict__ diss) {
  const int e = XTID;
  if (e >= g.E) return;
  const int N = g.N, E = g.E, eI = g.eI[e], eJ = g.eJ[e];
  double d = 0;
  for (int k = 0; k + 1 < L; k++) {
    const double ha = 0.5 * (h[(size_t)k * N + eI] + h[(size_t)k * N + eJ]);
    const double hb = 0.5 * (h[(size_t)(k + 1) * N + eI] + h[(size_t)(k + 1) * N + eJ]);
    double* ua = u + (size_t)k * E + e;
    double* ub = u + (size_t)(k + 1) * E + e;
    const double mean = (ha * *ua + hb * *ub) / (ha + hb);
    const double du0 = *ua - *ub;
    double du1 = du0 * exp(-c * (1 / ha + 1 / hb) * dt);
    if (cd > 0) du1 = du1 / (1 + cd * fabs(du0) * (1 / ha + 1 / hb) * dt);
    *ua = mean + hb / (ha + hb) * du1;
    *ub = mean - ha / (ha + hb) * du1;
    d += 0.5 * ha * hb / (ha + hb) * (du0 * du0 - du1 * du1);
  }
  diss[e] = d;
  if (wall && wall[e] == 0)
    for (int k = 0; k < L; k++) u[(size_t)k * E + e] = 0;
}

__global__ __launch_bounds__(BS) void k_vmix_heat(isw_grid g, LP p, const double* __restrict__ h,
                                                  const double* __restrict__ diss, double* __restrict__ th) {
  const int i = XTID;
  if (i >= g.N) return;
  const int N = g.N, L = p.L;
  int e[6];
  ring6(g.cellEdge, i, e);
  double t[6];
#pragma unroll
  for (int m = 0; m < 6; m++) t[m] = 0.5 * g.le[ok0(e[m])] * g.de[ok0(e[m])] * diss[ok0(e[m])];
  double q = 0;
#pragma unroll
  for (int m = 0; m < 6; m++)
    if (e[m] >= 0) q += t[m];
  if (q == 0) return;
  q /= g.areaCell[i];
  double mu = 0;
  for (int k = 0; k < L; k++) mu += h[(size_t)k * N + i];
  const double gr = grav_at(p, i);
  double pr = 0, xt = 0;
  for (int k = 0; k < L; k++) {
    const double pt = pr;
    pr = pr + gr * h[(size_t)k * N + i];
    const double x = pow(pr / p.p0, p.kappa);
    const double pib = p.cp * (pr * x - pt * xt) / ((p.kappa + 1) * (pr - pt));
    th[(size_t)k * N + i] += q / (mu * pib);
    xt = x;
  }
}

__global__ __launch_bounds__(BS) void k_xch_cell(int N, int L, int seq, const double* __restrict__ wx,
                                                 const double* __restrict__ areaCell, double* __restrict__ h,
                                                 double* __restrict__ M, double* __restrict__ psi) {
  const int i = XTID;
  if (i >= N) return;
  double tr[ISW_LMAX], dm[ISW_LMAX];
  for (int k = 0; k < L; k++) { tr[k] = 0; dm[k] = 0; }
  if (seq) {
    double m[ISW_LMAX], t[ISW_LMAX];
    for (int k = 0; k < L; k++) { const size_t o = (size_t)k * N + i; m[k] = M[o]; t[k] = M[o] * psi[o]; }
    for (int pass = 0; pass < 2; pass++)
      for (int n = 0; n + 1 < L; n++) {
        const int k = pass == 0 ? L - 2 - n : n;
        const double v = wx[(size_t)k * N + i];
        if (pass == 0 ? !(v > 0) : !(v < 0)) continue;
        const int d = v > 0 ? k + 1 : k;
        const double vol = v * areaCell[i], pp = t[d] / m[d];
        m[k] += vol; m[k + 1] -= vol; t[k] += vol * pp; t[k + 1] -= vol * pp;
      }
    for (int k = 0; k < L; k++) {
      const size_t o = (size_t)k * N + i;
      h[o] = h[o] + (m[k] - M[o]) / areaCell[i];
      M[o] = m[k];
      psi[o] = t[k] / m[k];
    }
    return;
  }
  for (int k = 0; k + 1 < L; k++) {
    const double v = wx[(size_t)k * N + i];
    const double pp = v > 0 ? psi[(size_t)(k + 1) * N + i] : psi[(size_t)k * N + i];
    const double vol = v * areaCell[i];
    dm[k] += vol; dm[k + 1] -= vol;
    tr[k] += vol * pp; tr[k + 1] -= vol * pp;
  }
  for (int k = 0; k < L; k++) {
    const size_t o = (size_t)k * N + i;
    const double m1 = M[o] + dm[k];
    psi[o] = (M[o] * psi[o] + tr[k]) / m1;
    M[o] = m1;
    h[o] = h[o] + dm[k] / areaCell[i];
  }
}

__global__ __launch_bounds__(BS) void k_xch_edge(isw_grid g, int L, const double* __restrict__ wx,
                                                 const double* __restrict__ hold, double* __restrict__ u,
                                                 double* __restrict__ diss, const double* __restrict__ lap4,
                                                 double nu4dt, double hthin, double floor_,
                                                 const double* __restrict__ wall) {
  const int e = XTID;
  if (e >= g.E) return;
  const int N = g.N, E = g.E, eI = g.eI[e], eJ = g.eJ[e];
  double mom[ISW_LMAX], hn[ISW_LMAX];
  double k0 = 0, v4 = 0;
  for (int k = 0; k < L; k++) {
    const double he = 0.5 * (hold[(size_t)k * N + eI] + hold[(size_t)k * N + eJ]);
    const double uk = u[(size_t)k * E + e];
    mom[k] = he * uk;
    hn[k] = he;
    k0 += he * uk * uk;
    if (lap4) v4 += he * uk * lap4[(size_t)k * E + e];
  }
  for (int pass = 0; pass < 2; pass++)
    for (int n = 0; n + 1 < L; n++) {
      const int k = pass == 0 ? L - 2 - n : n;
      const double v = 0.5 * (wx[(size_t)k * N + eI] + wx[(size_t)k * N + eJ]);
      if (pass == 0 ? !(v > 0) : !(v < 0)) continue;
      const int d = v > 0 ? k + 1 : k;
      const double ud = hn[d] > floor_ ? mom[d] / hn[d] : u[(size_t)d * E + e];
      mom[k] += v * ud; mom[k + 1] -= v * ud;
      hn[k] += v; hn[k + 1] -= v;
    }
  double un[ISW_LMAX];
  for (int k = 0; k < L; k++) un[k] = mom[k] / hn[k];
  if (hthin > 0)
    for (int k = 0; k < L; k++) {
      const double hm = fmin(hold[(size_t)k * N + eI], hold[(size_t)k * N + eJ]);
      if (hm >= hthin) continue;
      double w = (hthin - hm) / (hthin - floor_);
      if (w > 1) w = 1;
      double hs = 0, ms = 0;
      if (k > 0) { hs += hn[k - 1]; ms += hn[k - 1] * un[k - 1]; }
      if (k + 1 < L) { hs += hn[k + 1]; ms += hn[k + 1] * un[k + 1]; }
      if (hs <= 0) continue;
      w = fmin(w, hs / (hn[k] + hs));
      const double du = w * (ms / hs - un[k]);
      un[k] += du;
      const double dn = hn[k] * du / hs;
      if (k > 0) un[k - 1] -= dn;
      if (k + 1 < L) un[k + 1] -= dn;
    }
  double k1 = 0;
  const bool walled = wall && wall[e] == 0;
  for (int k = 0; k < L; k++) {
    u[(size_t)k * E + e] = walled ? 0.0 : un[k];
    k1 += hn[k] * un[k] * un[k];
  }
  if (diss) diss[e] = 0.5 * (k0 - k1) + nu4dt * v4;
}

// ---------------------------------------------------------------------------------------------------------------
// Transport (fused.cu:124-241; trisk.cu:48-59). Rows y = tracer * Lm + layer; a row's masses and fluxes are layer
// y % Lm's. blockIdx.y is the row.
// ---------------------------------------------------------------------------------------------------------------
__global__ __launch_bounds__(BS) void k_mass_update(isw_grid g, const double* __restrict__ M0,
                                                    const double* __restrict__ Fm, double* __restrict__ M1) {
  const int i = XTID;
  if (i >= g.N) return;
  const int l = blockIdx.y;
  const size_t o = (size_t)l * g.N + i;
  const double* f = Fm + (size_t)l * g.E;
  int e[6];
  ring6(g.cellEdgeAsc, i, e);
  double fv[6];
  bool own[6];
#pragma unroll
  for (int k = 0; k < 6; k++) { fv[k] = f[ok0(e[k])]; own[k] = g.eI[ok0(e[k])] == i; }
  double m = M0[o];
#pragma unroll
  for (int k = 0; k < 6; k++) {
    if (e[k] < 0) break;
    if (own[k]) m -= fv[k]; else m += fv[k];
  }
  M1[o] = m;
}

__device__ __forceinline__ double upwind(const double* Fml, const double* p, const isw_grid& g, int e) {
  const double f = Fml[e];
  return f * (f >= 0 ? p[g.eI[e]] : p[g.eJ[e]]);
}

// 3rd-order flux with upwind weight beta (fused.cu:131-138): f (mean - a - b) + |f| (b - a) beta; the curvature
// stencil on `psf` (the field itself in the plain form, its FP32 copy in the mixed form) with weights wt.
// The high-order flux of one edge from its stencil (eight cells ix with weights w, its two cells I, J), for the
// tracer row ps (psf its stencil copy) and the edge's mass flux f.
__device__ __forceinline__ double hoflux_of(double f, double pI, double pJ, const fast (&v)[8], const fast (&w)[8],
                                            double beta) {
  const fast a = w[0] * v[0] + w[1] * v[1] + w[2] * v[2] + w[3] * v[3];
  const fast b = w[4] * v[4] + w[5] * v[5] + w[6] * v[6] + w[7] * v[7];
  return f * (0.5 * (pI + pJ) - (double)(a + b)) + fabs(f) * ((double)(b - a) * beta);
}
__device__ __forceinline__ double hoflux_at(double f, const double* ps, const fast* psf, const int (&ix)[8],
                                            const fast (&w)[8], int I, int J, double beta) {
  fast v[8];
#pragma unroll
  for (int k = 0; k < 8; k++) v[k] = psf[ix[k]];
  return hoflux_of(f, ps[I], ps[J], v, w, beta);
}
__device__ __forceinline__ void stencil_at(const isw_grid& g, const fast* wt, int e, int (&ix)[8], fast (&w)[8]) {
  const int o = e * 8;
#pragma unroll
  for (int k = 0; k < 8; k++) {
    ix[k] = g.d2idx[o + k];
    w[k] = wt[o + k];
  }
}
__device__ __forceinline__ double hoflux(const double* Fml, const double* ps, const fast* psf, const fast* wt,
                                         const isw_grid& g, int e, double beta) {
  int ix[8];
  fast w[8];
  stencil_at(g, wt, e, ix, w);
  return hoflux_at(Fml[e], ps, psf, ix, w, g.eI[e], g.eJ[e], beta);
}

__global__ __launch_bounds__(BS) void k_tr_td(isw_grid g, int Lm, int rows, const double* __restrict__ M0,
                                              const double* __restrict__ psi, const double* __restrict__ Fm,
                                              const double* __restrict__ M1, double* __restrict__ td,
                                              float* __restrict__ pf) {
  const int i = XTID;
  const int y = blockIdx.y * blockDim.y + threadIdx.y, l = y % Lm;
  if (i >= g.N || y >= rows) return;
  const size_t o = (size_t)y * g.N + i, om = (size_t)l * g.N + i;
  const double* p = psi + (size_t)y * g.N;
  const double* Fml = Fm + (size_t)l * g.E;
  int e[6];
  ring6(g.cellEdgeAsc, i, e);
  double fv[6];
  bool own[6];
#pragma unroll
  for (int k = 0; k < 6; k++) { fv[k] = upwind(Fml, p, g, ok0(e[k])); own[k] = g.eI[ok0(e[k])] == i; }
  double t = M0[om] * psi[o];
#pragma unroll
  for (int k = 0; k < 6; k++) {
    if (e[k] < 0) break;
    if (own[k]) t -= fv[k]; else t += fv[k];
  }
  td[o] = t / M1[om];
  if (pf) pf[o] = (float)psi[o];
}

__global__ __launch_bounds__(BS) void k_tr_hflux(isw_grid g, int Lm, int rows, double frac, double beta,
                                                 const double* __restrict__ src, const fast* __restrict__ srcf,
                                                 const fast* __restrict__ wt, const double* __restrict__ Fm,
                                                 double* __restrict__ Hf) {
  const int e = XTID;
  const int y = blockIdx.y * blockDim.y + threadIdx.y, l = y % Lm;
  if (e >= g.E || y >= rows) return;
  Hf[(size_t)y * g.E + e] =
      frac * hoflux(Fm + (size_t)l * g.E, src + (size_t)y * g.N, srcf + (size_t)y * g.N, wt, g, e, beta);
}

__global__ __launch_bounds__(BS) void k_tr_stage(isw_grid g, int Lm, int rows, double frac, const double* __restrict__ M0,
                                                 const double* __restrict__ psi, const double* __restrict__ Hf,
                                                 const double* __restrict__ Fm, double* __restrict__ out,
                                                 float* __restrict__ pf) {
  const int i = XTID;
  const int y = blockIdx.y * blockDim.y + threadIdx.y, l = y % Lm;
  if (i >= g.N || y >= rows) return;
  const size_t o = (size_t)y * g.N + i, om = (size_t)l * g.N + i;
  const double* Hl = Hf + (size_t)y * g.E;
  const double* Fml = Fm + (size_t)l * g.E;
  int e[6];
  ring6(g.cellEdgeAsc, i, e);
  double fv[6], mv[6];
  bool own[6];
#pragma unroll
  for (int k = 0; k < 6; k++) {
    const int ek = ok0(e[k]);
    fv[k] = Hl[ek];
    mv[k] = frac * Fml[ek];
    own[k] = g.eI[ek] == i;
  }
  double t = M0[om] * psi[o];
  double mx = M0[om];
#pragma unroll
  for (int k = 0; k < 6; k++) {
    if (e[k] < 0) break;
    if (own[k]) { t -= fv[k]; mx -= mv[k]; } else { t += fv[k]; mx += mv[k]; }
  }
  const double r = t / mx;
  out[o] = r;
  if (pf) pf[o] = (float)r;
}

// One RK stage of the transport in one launch on the grid's 64-cell patches (k_tr_hflux then k_tr_stage): block
// (patch, four rows) first computes the third-order flux of every edge of its cells -- its own edges and those
// whose second cell only is in the patch, the latter also computed by the neighbour that owns them, from the same
// inputs, so every copy is the same to the bit -- into LDS, then steps its 64 cells x 4 rows from there. The flux
// array's write and re-read (rows x E doubles each way) and one kernel boundary go away; the arithmetic and every
// sum's order are k_tr_hflux's and k_tr_stage's. pfo: the output's FP32 copy (mixed form; the stencil reads srcf,
// a different buffer, so no block overwrites what another still reads).
__global__ __launch_bounds__(BS) void k_tr_hstage(isw_grid g, int Lm, int rows, double frac, double beta,
                                                  const double* __restrict__ src, const fast* __restrict__ srcf,
                                                  const fast* __restrict__ wt, const double* __restrict__ Fm,
                                                  const double* __restrict__ M0, const double* __restrict__ psi,
                                                  double* __restrict__ out, float* __restrict__ pfo) {
  extern __shared__ double hs[];                   // [4][ptedges] the stage flux of the patch's edges, per row
  const int PT = g.ptedges, N = g.N, E = g.E;
  const int b = xblock();
  const int tx = threadIdx.x, ty = threadIdx.y;
  const int y = blockIdx.y * 4 + ty;
  const bool rowok = y < rows;
  const int l = y % Lm;
  const int e0 = g.pe_off[b], ne = g.pe_off[b + 1] - e0;
  const int i0 = g.pi_off[b], ni = g.pi_off[b + 1] - i0;
  // the stage flux of the patch's edges for the block's four rows: thread t takes edges t, t + BS, ..., each edge's
  // stencil (its eight cells and weights, its two cells) loaded once for the four rows
  const int y0 = blockIdx.y * 4, nq = ne + ni;
  for (int q = ty * BS1 + tx; q < nq; q += BS) {
    const int e = q < ne ? g.pe_edge[e0 + q] : g.pi_edge[i0 + q - ne];
    int ix[8];
    fast w[8];
    stencil_at(g, wt, e, ix, w);
    const int I = g.eI[e], J = g.eJ[e];
#pragma unroll
    for (int r = 0; r < 4; r++) {
      const int yr = y0 + r;
      if (yr < rows) {
        const double f = Fm[(size_t)(yr % Lm) * E + e];
        hs[r * PT + q] = frac * hoflux_at(f, src + (size_t)yr * N, srcf + (size_t)yr * N, ix, w, I, J, beta);
      }
    }
  }
  __syncthreads();
  const int i = b * BS1 + tx;
  if (!rowok || i >= N) return;
  const size_t o = (size_t)y * N + i, om = (size_t)l * N + i;
  const double* Fml = Fm + (size_t)l * E;
  int e[6], sl[6];
  ring6(g.cellEdgeAsc, i, e);
  ring6(g.tc_slot, i, sl);
  double fv[6], mv[6];
#pragma unroll
  for (int k = 0; k < 6; k++) {
    fv[k] = hs[ty * PT + (sl[k] < 0 ? 0 : sl[k] >> 1)];
    mv[k] = frac * Fml[ok0(e[k])];
  }
  double t = M0[om] * psi[o];
  double mx = M0[om];
#pragma unroll
  for (int k = 0; k < 6; k++) {
    if (e[k] < 0) break;
    if (sl[k] & 1) { t -= fv[k]; mx -= mv[k]; } else { t += fv[k]; mx += mv[k]; }
  }
  const double r = t / mx;
  out[o] = r;
  if (pfo) pfo[o] = (float)r;
}

// ---------------------------------------------------------------------------------------------------------------
// The transport on the grid's 64-cell patches. Its scratch holds the rows cell-major, padded to RS, a multiple of four
// (cell i's rows at i * RS ..), so that a stencil's gather of one cell brings four rows in one load: with the rows apart
// (as psi is) each load of a wave touched seventeen lines for 64 values, and every pass was bound by that (15 rows at
// level 6: tr_td 16.5, each stage 23, tr_aflux 14.4, tr_ratios 15.1, tr_apply 17.1 us). A block takes a patch and RC (4 or
// 8) rows; a lane takes four rows of an edge, then two rows of a cell. Each pass forms the fluxes of every edge of its
// cells -- the patch's own edges and those whose second cell only is in it, the latter also formed by the neighbour that
// owns them, from the same inputs, so every copy is the same to the bit -- in LDS, then steps its cells from there (15 rows
// at level 6, mixed: the stages 48.5 us for both, tr_limit 27.3, tr_correct 14.4, tr_turn 5.8: 1.6 to 2.7 TB/s of the bytes
// each cannot do without; one row to a load was 105.4 for all, 120.6 with the rows apart). What is left is the latency of
// the chain edge -> stencil -> eight gathers and the edges formed twice (a patch's rim, a sixth of its edges). The
// arithmetic and every sum's order are k_tr_td's, k_tr_hflux's, k_tr_stage's, k_tr_aflux's, k_tr_ratios's and
// k_tr_apply's; the padding rows hold zeros.
// ---------------------------------------------------------------------------------------------------------------
// A block's patch and rows: blocks run over a patch's row chunks first, so that one XCD's L2 serves them all.
struct TrBlock {
  int b, y0, e0, ne, i0, nq;
  __device__ __forceinline__ int edge(const isw_grid& g, int q) const {
    return q < ne ? g.pe_edge[e0 + q] : g.pi_edge[i0 + q - ne];
  }
};
__device__ __forceinline__ TrBlock tr_block(const isw_grid& g, int chunks, int rc) {
  TrBlock t;
  const int x = xblock();
  t.b = x / chunks;
  t.y0 = (x - t.b * chunks) * rc;
  t.e0 = g.pe_off[t.b];
  t.ne = g.pe_off[t.b + 1] - t.e0;
  t.i0 = g.pi_off[t.b];
  t.nq = t.ne + g.pi_off[t.b + 1] - t.i0;
  return t;
}
// Four (or two) rows of a cell or an edge, in 16-byte loads where the width allows.
__device__ __forceinline__ void rows4(const double* p, double (&v)[4]) {
  const double2 a = reinterpret_cast<const double2*>(p)[0], b = reinterpret_cast<const double2*>(p)[1];
  v[0] = a.x; v[1] = a.y; v[2] = b.x; v[3] = b.y;
}
__device__ __forceinline__ void rows4(const float* p, float (&v)[4]) {
  const float4 a = *reinterpret_cast<const float4*>(p);
  v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w;
}
__device__ __forceinline__ void put4(double* p, const double (&v)[4]) {
  reinterpret_cast<double2*>(p)[0] = make_double2(v[0], v[1]);
  reinterpret_cast<double2*>(p)[1] = make_double2(v[2], v[3]);
}
__device__ __forceinline__ double2 rows2(const double* p) { return *reinterpret_cast<const double2*>(p); }
// The third-order fluxes of four rows of an edge with mass fluxes f, of the field whose rows at the edge's cells are pI,
// pJ, its stencil copy psf.
__device__ __forceinline__ void hoflux4(const fast* __restrict__ psf, const fast* __restrict__ wt, const isw_grid& g,
                                        int RS, int e, int yr, const double (&f)[4], const double (&pI)[4],
                                        const double (&pJ)[4], double beta, double (&h)[4]) {
  int ix[8];
  fast w[8], v[8][4];
  stencil_at(g, wt, e, ix, w);
#pragma unroll
  for (int k = 0; k < 8; k++) rows4(psf + (size_t)ix[k] * RS + yr, v[k]);
#pragma unroll
  for (int r = 0; r < 4; r++) {
    const fast x[8] = {v[0][r], v[1][r], v[2][r], v[3][r], v[4][r], v[5][r], v[6][r], v[7][r]};
    h[r] = hoflux_of(f[r], pI[r], pJ[r], x, w, beta);
  }
}
// The mass fluxes of the rows' layers on an edge.
__device__ __forceinline__ void tr_mass(const double* __restrict__ Fm, int E, int Lm, int e, int yr, double (&f)[4]) {
#pragma unroll
  for (int r = 0; r < 4; r++) f[r] = Fm[(size_t)((yr + r) % Lm) * E + e];
}
// Two rows of a cell moved by the fluxes in LDS (four rows to a place, from hs), in cellEdgeAsc order.
template <int RC>
__device__ __forceinline__ double2 tr_moved(double2 t, const double* hs, const int (&sl)[6]) {
  double2 fv[6];
#pragma unroll
  for (int k = 0; k < 6; k++) fv[k] = rows2(hs + (sl[k] < 0 ? 0 : sl[k] >> 1) * RC);
#pragma unroll
  for (int k = 0; k < 6; k++) {
    if (sl[k] < 0) break;
    if (sl[k] & 1) { t.x -= fv[k].x; t.y -= fv[k].y; } else { t.x += fv[k].x; t.y += fv[k].y; }
  }
  return t;
}

// psi (rows, N) cell-major, and its FP32 copy (mixed form): 64 cells x 16 rows through LDS.
__global__ __launch_bounds__(BS) void k_tr_turn(int N, int rows, int RS, const double* __restrict__ psi,
                                                double* __restrict__ out, float* __restrict__ pf) {
  __shared__ double s[16][BS1 + 1];
  const int i0 = xblock() * BS1, y0 = blockIdx.y * 16, t = (int)threadIdx.x;
  for (int x = t; x < 16 * BS1; x += BS) {
    const int y = x >> 6, c = x & 63;
    s[y][c] = y0 + y < rows && i0 + c < N ? psi[(size_t)(y0 + y) * N + i0 + c] : 0.0;
  }
  __syncthreads();
  const int nr = min(16, RS - y0);
  for (int x = t; x < nr * BS1; x += BS) {
    const int c = x / nr, y = x - c * nr;
    if (i0 + c >= N) break;
    const size_t o = (size_t)(i0 + c) * RS + y0 + y;
    out[o] = s[y][c];
    if (pf) pf[o] = (float)s[y][c];
  }
}

// One RK stage: the third-order fluxes of src (cell-major, stencil copy srcf) and the step of psi by frac of them. The
// first also steps psi upwind (td). pfo: the output's FP32 copy (the stencil reads srcf, a different buffer, so no block
// overwrites what another still reads).
template <int RC, bool TD>
__global__ __launch_bounds__(BS) void k_tr_move(isw_grid g, int Lm, int RS, int chunks, double frac, double beta,
                                                const double* __restrict__ src, const fast* __restrict__ srcf,
                                                const fast* __restrict__ wt, const double* __restrict__ Fm,
                                                const double* __restrict__ M0, const double* __restrict__ M1,
                                                const double* __restrict__ psi, double* __restrict__ out,
                                                float* __restrict__ pfo, double* __restrict__ td) {
  extern __shared__ double sm[];
  const int PT = g.ptedges, N = g.N;
  double* hs = sm;                                 // [edge][RC] the stage's fluxes
  double* us = hs + PT * RC;                       // [edge][RC] (TD) the upwind fluxes
  const TrBlock t = tr_block(g, chunks, RC);
  constexpr int Q = RC / 4, P = RC / 2;
  for (int x = (int)threadIdx.x; x < t.nq * Q; x += BS) {
    const int q = x / Q, y = (x - q * Q) * 4, yr = t.y0 + y;
    if (yr >= RS) continue;
    const int e = t.edge(g, q), I = g.eI[e], J = g.eJ[e];
    double f[4], pI[4], pJ[4], h[4];
    tr_mass(Fm, g.E, Lm, e, yr, f);
    rows4(src + (size_t)I * RS + yr, pI);
    rows4(src + (size_t)J * RS + yr, pJ);
    hoflux4(srcf, wt, g, RS, e, yr, f, pI, pJ, beta, h);
#pragma unroll
    for (int r = 0; r < 4; r++) h[r] = frac * h[r];
    put4(hs + q * RC + y, h);
    if (TD) {
#pragma unroll
      for (int r = 0; r < 4; r++) h[r] = f[r] * (f[r] >= 0 ? pI[r] : pJ[r]);
      put4(us + q * RC + y, h);
    }
  }
  __syncthreads();
  for (int x = (int)threadIdx.x; x < BS1 * P; x += BS) {
    const int c = x / P, y = (x - c * P) * 2, yr = t.y0 + y, i = t.b * BS1 + c;
    if (yr >= RS || i >= N) continue;
    const size_t o = (size_t)i * RS + yr;
    const int la = yr % Lm, lb = (yr + 1) % Lm;
    int sl[6], e[6];
    ring6(g.tc_slot, i, sl);
    ring6(g.cellEdgeAsc, i, e);
    double ma[6], mb[6];
#pragma unroll
    for (int k = 0; k < 6; k++) {
      ma[k] = frac * Fm[(size_t)la * g.E + ok0(e[k])];
      mb[k] = frac * Fm[(size_t)lb * g.E + ok0(e[k])];
    }
    const double2 ps = rows2(psi + o), m0 = make_double2(M0[(size_t)la * N + i], M0[(size_t)lb * N + i]);
    const double2 mp = make_double2(m0.x * ps.x, m0.y * ps.y);
    double2 mx = m0;
#pragma unroll
    for (int k = 0; k < 6; k++) {
      if (sl[k] < 0) break;
      if (sl[k] & 1) { mx.x -= ma[k]; mx.y -= mb[k]; } else { mx.x += ma[k]; mx.y += mb[k]; }
    }
    double2 r = tr_moved<RC>(mp, hs + y, sl);
    r.x /= mx.x;
    r.y /= mx.y;
    *reinterpret_cast<double2*>(out + o) = r;
    if (pfo) *reinterpret_cast<float2*>(pfo + o) = make_float2((float)r.x, (float)r.y);
    if (TD) {
      r = tr_moved<RC>(mp, us + y, sl);
      r.x /= M1[(size_t)la * N + i];
      r.y /= M1[(size_t)lb * N + i];
      *reinterpret_cast<double2*>(td + o) = r;
    }
  }
}

// The antidiffusive fluxes (the third-order ones of p2 less the upwind ones of psi; A, edge-major by rows, written by each
// edge's first cell's patch) and the limiter's ratios.
template <int RC>
__global__ __launch_bounds__(BS) void k_tr_limit(isw_grid g, int Lm, int RS, int chunks, double beta,
                                                 const double* __restrict__ psi, const double* __restrict__ p2,
                                                 const fast* __restrict__ p2f, const fast* __restrict__ wt,
                                                 const double* __restrict__ Fm, const double* __restrict__ td,
                                                 const double* __restrict__ M1, double* __restrict__ A,
                                                 double* __restrict__ Rp, double* __restrict__ Rm) {
  extern __shared__ double sm[];
  const int N = g.N;
  double* as = sm;                                 // [edge][RC]
  const TrBlock t = tr_block(g, chunks, RC);
  constexpr int Q = RC / 4, P = RC / 2;
  for (int x = (int)threadIdx.x; x < t.nq * Q; x += BS) {
    const int q = x / Q, y = (x - q * Q) * 4, yr = t.y0 + y;
    if (yr >= RS) continue;
    const int e = t.edge(g, q), I = g.eI[e], J = g.eJ[e];
    double f[4], pI[4], pJ[4], uI[4], uJ[4], h[4];
    tr_mass(Fm, g.E, Lm, e, yr, f);
    rows4(p2 + (size_t)I * RS + yr, pI);
    rows4(p2 + (size_t)J * RS + yr, pJ);
    rows4(psi + (size_t)I * RS + yr, uI);
    rows4(psi + (size_t)J * RS + yr, uJ);
    hoflux4(p2f, wt, g, RS, e, yr, f, pI, pJ, beta, h);
#pragma unroll
    for (int r = 0; r < 4; r++) h[r] -= f[r] * (f[r] >= 0 ? uI[r] : uJ[r]);
    put4(as + q * RC + y, h);
    if (q < t.ne) put4(A + (size_t)e * RS + yr, h);
  }
  __syncthreads();
  for (int x = (int)threadIdx.x; x < BS1 * P; x += BS) {
    const int c = x / P, y = (x - c * P) * 2, yr = t.y0 + y, i = t.b * BS1 + c;
    if (yr >= RS || i >= N) continue;
    const size_t o = (size_t)i * RS + yr;
    int nb[6], sl[6];
    ring6(g.nbr, i, nb);
    ring6(g.tc_slot, i, sl);
    double2 pv[6], tv[6];
#pragma unroll
    for (int k = 0; k < 6; k++) {
      pv[k] = rows2(psi + (size_t)ok0(nb[k]) * RS + yr);
      tv[k] = rows2(td + (size_t)ok0(nb[k]) * RS + yr);
    }
    const double2 pi = rows2(psi + o), ti = rows2(td + o);
    double2 hi = make_double2(fmax(pi.x, ti.x), fmax(pi.y, ti.y)), lo = make_double2(fmin(pi.x, ti.x), fmin(pi.y, ti.y));
#pragma unroll
    for (int k = 0; k < 6; k++) {
      if (nb[k] < 0) break;
      hi.x = fmax(hi.x, fmax(pv[k].x, tv[k].x));
      hi.y = fmax(hi.y, fmax(pv[k].y, tv[k].y));
      lo.x = fmin(lo.x, fmin(pv[k].x, tv[k].x));
      lo.y = fmin(lo.y, fmin(pv[k].y, tv[k].y));
    }
    const double m1a = M1[(size_t)(yr % Lm) * N + i], m1b = M1[(size_t)((yr + 1) % Lm) * N + i];
    double2 Pp = make_double2(0, 0), Pm = Pp;
#pragma unroll
    for (int k = 0; k < 6; k++) {
      if (sl[k] < 0) break;
      const double2 a = rows2(as + (sl[k] >> 1) * RC + y);
      if (sl[k] & 1) {
        if (a.x > 0) Pm.x += a.x; else Pp.x -= a.x;
        if (a.y > 0) Pm.y += a.y; else Pp.y -= a.y;
      } else {
        if (a.x > 0) Pp.x += a.x; else Pm.x -= a.x;
        if (a.y > 0) Pp.y += a.y; else Pm.y -= a.y;
      }
    }
    auto share = [](double room, double need) { return need > 0 ? fmin(1.0, room / need) : 0.0; };
    *reinterpret_cast<double2*>(Rp + o) =
        make_double2(share((hi.x - ti.x) * m1a, Pp.x), share((hi.y - ti.y) * m1b, Pp.y));
    *reinterpret_cast<double2*>(Rm + o) =
        make_double2(share((ti.x - lo.x) * m1a, Pm.x), share((ti.y - lo.y) * m1b, Pm.y));
  }
}

// The upwind step corrected by the limited antidiffusive fluxes, back into psi's rows through LDS.
template <int RC>
__global__ __launch_bounds__(BS) void k_tr_correct(isw_grid g, int Lm, int rows, int RS, int chunks,
                                                   const double* __restrict__ td, const double* __restrict__ M1,
                                                   const double* __restrict__ A, const double* __restrict__ Rp,
                                                   const double* __restrict__ Rm, double* __restrict__ out) {
  extern __shared__ double sm[];
  __shared__ double turn[RC][BS1 + 1];
  double* as = sm;                                 // [edge][RC] the limited fluxes
  const int N = g.N;
  const TrBlock t = tr_block(g, chunks, RC);
  constexpr int Q = RC / 4, P = RC / 2;
  for (int x = (int)threadIdx.x; x < t.nq * Q; x += BS) {
    const int q = x / Q, y = (x - q * Q) * 4, yr = t.y0 + y;
    if (yr >= RS) continue;
    const int e = t.edge(g, q);
    const size_t oi = (size_t)g.eI[e] * RS + yr, oj = (size_t)g.eJ[e] * RS + yr;
    double a[4], pi[4], pj[4], mi[4], mj[4];
    rows4(A + (size_t)e * RS + yr, a);
    rows4(Rp + oi, pi);
    rows4(Rp + oj, pj);
    rows4(Rm + oi, mi);
    rows4(Rm + oj, mj);
#pragma unroll
    for (int r = 0; r < 4; r++) a[r] *= a[r] > 0 ? fmin(pj[r], mi[r]) : fmin(pi[r], mj[r]);
    put4(as + q * RC + y, a);
  }
  __syncthreads();
  for (int x = (int)threadIdx.x; x < BS1 * P; x += BS) {
    const int c = x / P, y = (x - c * P) * 2, yr = t.y0 + y, i = t.b * BS1 + c;
    if (yr >= RS || i >= N) continue;
    int sl[6];
    ring6(g.tc_slot, i, sl);
    const double m1a = M1[(size_t)(yr % Lm) * N + i], m1b = M1[(size_t)((yr + 1) % Lm) * N + i];
    const double2 ti = rows2(td + (size_t)i * RS + yr);
    const double2 r = tr_moved<RC>(make_double2(ti.x * m1a, ti.y * m1b), as + y, sl);
    turn[y][c] = r.x / m1a;
    turn[y + 1][c] = r.y / m1b;
  }
  __syncthreads();
  for (int x = (int)threadIdx.x; x < BS1 * RC; x += BS) {
    const int y = x >> 6, c = x & 63;
    if (t.y0 + y < rows && t.b * BS1 + c < N) out[(size_t)(t.y0 + y) * N + t.b * BS1 + c] = turn[y][c];
  }
}

__global__ __launch_bounds__(BS) void k_tr_aflux(isw_grid g, int Lm, int rows, double beta, const double* __restrict__ psi,
                                                 const double* __restrict__ p2, const fast* __restrict__ p2f,
                                                 const fast* __restrict__ wt, const double* __restrict__ Fm,
                                                 double* __restrict__ A) {
  // one edge per thread (256 per block), its stencil loaded once for the block's four rows
  const int e = xblock() * BS + threadIdx.y * BS1 + threadIdx.x;
  if (e >= g.E) return;
  int ix[8];
  fast w[8];
  stencil_at(g, wt, e, ix, w);
  const int I = g.eI[e], J = g.eJ[e];
  const int y0 = blockIdx.y * 4;
#pragma unroll
  for (int r = 0; r < 4; r++) {
    const int y = y0 + r;
    if (y < rows) {
      const double f = Fm[(size_t)(y % Lm) * g.E + e];
      const double* p = psi + (size_t)y * g.N;
      A[(size_t)y * g.E + e] = hoflux_at(f, p2 + (size_t)y * g.N, p2f + (size_t)y * g.N, ix, w, I, J, beta) -
                               f * (f >= 0 ? p[I] : p[J]);
    }
  }
}

__global__ __launch_bounds__(BS) void k_tr_ratios(isw_grid g, int Lm, int rows, const double* __restrict__ psi,
                                                  const double* __restrict__ td, const double* __restrict__ M1,
                                                  const double* __restrict__ A, double* __restrict__ Rp,
                                                  double* __restrict__ Rm) {
  const int i = XTID;
  const int y = blockIdx.y * blockDim.y + threadIdx.y, l = y % Lm;
  if (i >= g.N || y >= rows) return;
  const double* p = psi + (size_t)y * g.N;
  const double* t = td + (size_t)y * g.N;
  const double* Al = A + (size_t)y * g.E;
  int nb[6], e[6];
  ring6(g.nbr, i, nb);
  ring6(g.cellEdgeAsc, i, e);
  double pv[6], tv[6], av[6];
  bool own[6];
#pragma unroll
  for (int k = 0; k < 6; k++) {
    pv[k] = p[ok0(nb[k])];
    tv[k] = t[ok0(nb[k])];
    av[k] = Al[ok0(e[k])];
    own[k] = g.eI[ok0(e[k])] == i;
  }
  double hi = fmax(p[i], t[i]), lo = fmin(p[i], t[i]);
#pragma unroll
  for (int k = 0; k < 6; k++) {
    if (nb[k] < 0) break;
    hi = fmax(hi, fmax(pv[k], tv[k]));
    lo = fmin(lo, fmin(pv[k], tv[k]));
  }
  const double m1 = M1[(size_t)l * g.N + i];
  const double qmax = (hi - t[i]) * m1, qmin = (t[i] - lo) * m1;
  double Pp = 0, Pm = 0;
#pragma unroll
  for (int k = 0; k < 6; k++) {
    if (e[k] < 0) break;
    const double a = av[k];
    if (own[k]) { if (a > 0) Pm += a; else Pp -= a; }
    else { if (a > 0) Pp += a; else Pm -= a; }
  }
  Rp[(size_t)y * g.N + i] = Pp > 0 ? fmin(1.0, qmax / Pp) : 0.0;
  Rm[(size_t)y * g.N + i] = Pm > 0 ? fmin(1.0, qmin / Pm) : 0.0;
}

__global__ __launch_bounds__(BS) void k_tr_apply(isw_grid g, int Lm, int rows, const double* __restrict__ td,
                                                 const double* __restrict__ M1, const double* __restrict__ A,
                                                 const double* __restrict__ Rp, const double* __restrict__ Rm,
                                                 double* __restrict__ out) {
  const int i = XTID;
  const int y = blockIdx.y * blockDim.y + threadIdx.y, l = y % Lm;
  if (i >= g.N || y >= rows) return;
  const size_t o = (size_t)y * g.N + i, om = (size_t)l * g.N + i;
  const double* Al = A + (size_t)y * g.E;
  const double* rp = Rp + (size_t)y * g.N;
  const double* rm = Rm + (size_t)y * g.N;
  int e[6];
  ring6(g.cellEdgeAsc, i, e);
  double av[6], cv[6];
  bool own[6];
#pragma unroll
  for (int k = 0; k < 6; k++) {
    const int ek = ok0(e[k]);
    const int eI = g.eI[ek], eJ = g.eJ[ek];
    av[k] = Al[ek];
    cv[k] = av[k] > 0 ? fmin(rp[eJ], rm[eI]) : fmin(rp[eI], rm[eJ]);
    own[k] = eI == i;
  }
  double t = td[o] * M1[om];
#pragma unroll
  for (int k = 0; k < 6; k++) {
    if (e[k] < 0) break;
    if (own[k]) t -= cv[k] * av[k]; else t += cv[k] * av[k];
  }
  out[o] = t / M1[om];
}

// ---------------------------------------------------------------------------------------------------------------
// SWE (fused.cu:27-120): five passes per stage.
// ---------------------------------------------------------------------------------------------------------------
__global__ __launch_bounds__(BS) void k_swe_scale(isw_grid g, double dts, const double* __restrict__ h,
                                                  const double* __restrict__ u, double* __restrict__ scale) {
  const int i = XTID;
  if (i >= g.N) return;
  const int l = blockIdx.y;
  const double* hl = h + (size_t)l * g.N;
  const double* ul = u + (size_t)l * g.E;
  double out = 0;
#pragma unroll
  for (int k = 0; k < 6; k++) {
    const int e = g.cellEdgeAsc[i * 6 + k];
    if (e < 0) break;
    const double f = 0.5 * (hl[g.eI[e]] + hl[g.eJ[e]]) * ul[e] * g.le[e] * dts;
    if (g.eI[e] == i) { if (f > 0) out += f; }
    else if (!(f > 0)) out -= f;
  }
  const double hv = hl[i];
  const double cap = 0.5 * (hv > 0 ? hv : 0.0) * g.areaCell[i];
  scale[(size_t)l * g.N + i] = out > cap ? cap / out : 1.0;
}

__global__ __launch_bounds__(BS) void k_swe_flux(isw_grid g, double dt, const double* __restrict__ h,
                                                 const double* __restrict__ u, const double* __restrict__ scale,
                                                 double* __restrict__ F, double* __restrict__ Fm) {
  const int e = XTID;
  if (e >= g.E) return;
  const int l = blockIdx.y;
  const size_t o = (size_t)l * g.E + e;
  const double* hl = h + (size_t)l * g.N;
  double f = 0.5 * (hl[g.eI[e]] + hl[g.eJ[e]]) * u[o];
  f *= f > 0 ? scale[(size_t)l * g.N + g.eI[e]] : scale[(size_t)l * g.N + g.eJ[e]];
  F[o] = f;
  if (Fm) Fm[o] = f * g.le[e] * dt;
}

__global__ __launch_bounds__(BS) void k_swe_cell(isw_grid g, double grav, double c, const double* __restrict__ h,
                                                 const double* __restrict__ b, const double* __restrict__ F,
                                                 const double* __restrict__ u, const double* h0, double* hn,
                                                 double* __restrict__ B) {
  const int i = XTID;
  if (i >= g.N) return;
  const int l = blockIdx.y;
  const double* Fl = F + (size_t)l * g.E;
  const double* ul = u + (size_t)l * g.E;
  double div = 0, ke = 0;
#pragma unroll
  for (int k = 0; k < 6; k++) {
    const int e = g.cellEdge[i * 6 + k];
    if (e < 0) break;
    div += (double)g.cellSign[i * 6 + k] * g.le[e] * Fl[e];
    ke += g.le[e] * g.de[e] * 0.25 * ul[e] * ul[e];
  }
  const size_t o = (size_t)l * g.N + i;
  const double dh = 0.0 - div / g.areaCell[i];
  B[o] = grav * (h[o] + b[i]) + 0.0 + ke / g.areaCell[i];
  hn[o] = h0[o] + c * dh;
}

__global__ __launch_bounds__(BS) void k_swe_vertex(isw_grid g, Div dv, const double* __restrict__ h,
                                                   const double* __restrict__ u, const double* __restrict__ fV,
                                                   double* __restrict__ q) {
  const int v = XTID;
  if (v >= g.NV) return;
  const int l = blockIdx.y;
  const double* hl = h + (size_t)l * g.N;
  const double* ul = u + (size_t)l * g.E;
  double hv = 0, z = 0;
#pragma unroll
  for (int k = 0; k < 3; k++) {
    const int c = g.vCell[v * 3 + k];
    hv += g.kite[c * 6 + g.vSlot[v * 3 + k]] * hl[c] * 1.0;
  }
#pragma unroll
  for (int k = 0; k < 3; k++) {
    const int e = g.vEdge[v * 3 + k];
    z += (double)g.vEdgeSign[v * 3 + k] * g.de[e] * ul[e];
  }
  q[(size_t)l * g.NV + v] = (DIVBY(z, dv.AV[v]) + fV[v]) / DIVBY(hv, dv.AV[v]);
}

// ---------------------------------------------------------------------------------------------------------------
// Air-sea stress, the land column, the mixed layer's capacity (ocean.cu:17-42,434-471).
// ---------------------------------------------------------------------------------------------------------------
__global__ __launch_bounds__(BS) void k_couple_stress(isw_grid g, int La, double c0, double rho_w, double dt,
                                                      double land_drag0, const double* __restrict__ ha,
                                                      double* __restrict__ ua, const double* __restrict__ ho,
                                                      double* __restrict__ uo, double* __restrict__ diss,
                                                      double* __restrict__ tau_acc, const double* __restrict__ wall,
                                                      const double* __restrict__ cd) {
  const int e = XTID;
  if (e >= g.E) return;
  const int N = g.N, E = g.E, b = La - 1, eI = g.eI[e], eJ = g.eJ[e];
  double c = c0, land_drag = land_drag0;
  if (cd) { c = 0.5 * (cd[eI] + cd[eJ]); land_drag = 1; }
  const double ma = 0.5 * (ha[(size_t)b * N + eI] + ha[(size_t)b * N + eJ]);
  const size_t oa = (size_t)b * E + e;
  const double a0 = ua[oa];
  double a1;
  if (wall && wall[e] == 0) {
    const double du1 = a0 * exp(-land_drag * c / ma * dt);
    a1 = du1;
    diss[e] = 0.5 * ma * (a0 * a0 - du1 * du1);
  } else {
    const double o0 = uo[e];
    const double mo = rho_w * 0.5 * (ho[eI] + ho[eJ]);
    const double mean = (ma * a0 + mo * o0) / (ma + mo);
    const double du0 = a0 - o0;
    const double du1 = du0 * exp(-c * (1 / ma + 1 / mo) * dt);
    a1 = mean + mo / (ma + mo) * du1;
    uo[e] = mean - ma / (ma + mo) * du1;
    diss[e] = 0.5 * ma * mo / (ma + mo) * (du0 * du0 - du1 * du1);
  }
  ua[oa] = a1;
  const double tau = ma * (a0 - a1) / dt;
  tau_acc[e] += tau * tau * dt;
}

__global__ __launch_bounds__(BS) void k_land_column(int N, int K, double c_soil, double k_soil, double dt,
                                                    const double* __restrict__ land, double* __restrict__ T,
                                                    const double* __restrict__ cap, double* __restrict__ Tg,
                                                    const double* __restrict__ dz) {
  const int i = XTID;
  if (i >= N) return;
  if (!(land[i] > 0.5)) return;
  const int n = K + 1;
  double C[ISW_KSOIL + 1], G[ISW_KSOIL + 1], x[ISW_KSOIL + 1], cp_[ISW_KSOIL + 1], dp[ISW_KSOIL + 1];
  C[0] = cap[i];
  x[0] = T[i];
  double half = cap[i] / c_soil / 2;
  for (int k = 1; k < n; k++) {
    const double d = dz[k - 1];
    C[k] = c_soil * d;
    x[k] = Tg[(size_t)(k - 1) * N + i];
    G[k - 1] = dt * k_soil / (half + d / 2);
    half = d / 2;
  }
  G[n - 1] = 0;
  for (int k = 0; k < n; k++) {
    const double a = k ? G[k - 1] : 0.0, c = G[k];
    const double den = C[k] + a + c - (k ? a * cp_[k - 1] : 0.0);
    cp_[k] = c / den;
    dp[k] = (C[k] * x[k] + (k ? a * dp[k - 1] : 0.0)) / den;
  }
  x[n - 1] = dp[n - 1];
  for (int k = n - 2; k >= 0; k--) x[k] = dp[k] + cp_[k] * x[k + 1];
  T[i] = x[0];
  for (int k = 1; k < n; k++) Tg[(size_t)(k - 1) * N + i] = x[k];
}

__global__ __launch_bounds__(BS) void k_ocn_cap(int N, double rho_cw, double c_land, const double* __restrict__ h,
                                                double* __restrict__ cap, const double* __restrict__ land) {
  const int i = XTID;
  if (i >= N) return;
  cap[i] = land && land[i] > 0.5 ? (cap[i] > 0 ? cap[i] : c_land) : rho_cw * h[i];
}

// SWE's edge pass (swe_edge, fused.cu:101-120) with each layer's drag from the layer settings passed by value.
__global__ __launch_bounds__(BS) void k_swe_edge_lp(isw_grid g, LP p, double c, const double* __restrict__ F,
                                                    const double* __restrict__ q, const double* __restrict__ B,
                                                    const double* __restrict__ u, const double* __restrict__ lap4,
                                                    const double* u0, double* un) {
  const int e = XTID;
  if (e >= g.E) return;
  const int l = blockIdx.y;
  const double* Fl = F + (size_t)l * g.E;
  const double* ql = q + (size_t)l * g.NV;
  const double* Bl = B + (size_t)l * g.N;
  const double qa = 0.5 * (ql[g.ev1[e]] + ql[g.ev2[e]]);
  double Q = 0;
  for (int k = g.eoeStart[e]; k < g.eoeStart[e + 1]; k++) {
    const int e2 = g.eoe[k];
    const double qb = 0.5 * (ql[g.ev1[e2]] + ql[g.ev2[e2]]);
    Q += g.w[k] * Fl[e2] * 0.5 * (qa + qb);
  }
  const size_t o = (size_t)l * g.E + e;
  double d = Q - (Bl[g.eJ[e]] - Bl[g.eI[e]]) / g.de[e] - p.drag[l] * u[o];
  if (p.nu4 != 0) d = d - p.nu4 * lap4[o];
  un[o] = u0[o] + c * d;
}

// ===============================================================================================================
// Host sequencing (the reference's Python drivers), all on one stream. Every launch goes through ISW_LAUNCH with the
// kernel's algorithmic bytes for the measurement mode (diag.hpp).
// ===============================================================================================================

// Byte counts: D doubles, I int32, C int8, R fast (the PV-flux and stencil operands' width).
constexpr double D = 8, I = 4, C = 1, R = sizeof(fast);

static double flux_bytes(const FluxSrc& f, double N, double E, double L) {
  return f.air ? 2 * L * E * D : L * N * D + L * E * D + 2 * E * D + (f.wall ? E * D : 0);
}

static void lap(const isw_grid* g, int L, const double* u, double* D1, double* Z1, double* out, hipStream_t st) {
  const double N = g->N, E = g->E, NV = g->NV, l = L;
  const int nbc = (g->N * L + BS - 1) / BS, nbv = (g->NV * L + BS - 1) / BS;
  ISW_LAUNCH("div_curl", l * E * D + 6 * N * (I + C) + E * D + N * D + l * N * D + 3 * NV * (I + C) + E * D + NV * D +
                             l * NV * D,
             k_div_curl, dim3(nbc + nbv), BS, *g, L, nbc, u, D1, Z1);
  ISW_LAUNCH("edge_lap", l * N * D + l * NV * D + 4 * E * I + 2 * E * D + l * E * D,
             k_edge_lap, g1((long)g->E * L), BS, *g, L, D1, Z1, out);
}

// The fast sub-steps that one launch takes on the grid's ring tables, for `rows` values per cell: as many as asked for
// whose rings fit a block's threads (four edges and two cells each) and 64 KB of LDS; 0 without the tables.
// (The kernels come with 2 or 3 edges and one cell to a thread, or 4 edges and two cells; the mesh's largest patch decides
// for all: at level 7 one of 2,561 touches 771 edges within three rings, three more than 3 to a thread.)
static int ring_cpt(const isw_grid* g, int m) { return g->rg_cells[m] > RBS || g->rg_edges[m] > 3 * RBS ? 2 : 1; }
static int ring_ept(const isw_grid* g, int m) {
  const int k = (g->rg_edges[m] + RBS - 1) / RBS, least = ring_cpt(g, m) == 2 ? 4 : 2;
  return k < least ? least : k;
}
static size_t ring_lds(const isw_grid* g, int rows, int m) {
  return (size_t)rows * (ring_ept(g, m) * RBS + 2 + ring_cpt(g, m) * RBS) * sizeof(double);
}
static int ring_most(const isw_grid* g, int rows, int want) {
  if (!g->rg_head || g->rg_owned > RBS || g->rg_cells[0] > RBS) return 0;   // (each on a thread of its own)
  int m = want < g->rg_k ? want : g->rg_k;
  while (m > 0 && (ring_ept(g, m) > 4 || g->rg_cells[m] > 2 * RBS || ring_lds(g, rows, m) > 65536)) m--;
  return m;
}
// f(edges, cells per thread) as compile-time counts, for m sub-steps.
template <class F>
static void ring_launch(const isw_grid* g, int m, F&& f) {
  using std::integral_constant;
  const int e = ring_ept(g, m), c = ring_cpt(g, m);      // (e <= 4: ring_most)
  if (c == 1 && e == 2) f(integral_constant<int, 2>{}, integral_constant<int, 1>{});
  else if (c == 1) f(integral_constant<int, 3>{}, integral_constant<int, 1>{});
  else f(integral_constant<int, 4>{}, integral_constant<int, 2>{});
}
// The next launch's share of `left` sub-steps: as few launches as there can be, as even as they can be.
static int ring_steps(int left, int most) {
  const int launches = (left + most - 1) / most;
  return (left + launches - 1) / launches;
}

// Layers._stage (layers.py:255-309).
static void stage(const isw_grid* g, const isw_layers* s, const LP& p, const Div& dv, int si, const double* hs,
                  const double* us, const double* h0, const double* u0, double c, double dt, int nfast, double* hn,
                  double* un, double* Fm, const double* theta, hipStream_t st) {
  const int N = g->N, E = g->E, L = s->L;
  const double n_ = N, e_ = E, v_ = g->NV, l_ = L, air = s->air ? 1 : 0;
  const int nbc = (N + BS1 - 1) / BS1, nbv = (g->NV + BS1 - 1) / BS1;
  ISW_LAUNCH("bern_pv", l_ * n_ * D * (1 + 3 * air) + l_ * e_ * D + n_ * D + 6 * n_ * I + 2 * e_ * D + n_ * D +
                            l_ * n_ * D + 3 * v_ * (2 * I + 2 * C) + 6 * n_ * D + 2 * v_ * D + l_ * v_ * D,
             k_bern_pv, dim3(nbc + nbv), dim3(BS1, L), *g, p, dv, nbc, hs, us, theta, s->b, s->S, s->fV, s->B,
                                                      s->pibar, s->q);
#if ISW_FORM_MIXED
  fast* pk = s->pkf;
  const fast* wf = g->wf;
  // the air's fast sub-steps' flux coefficients per edge (FP32 in the mixed form)
  fast* cf = s->air && g->rg_head ? s->cfcf : nullptr;
#else
  fast* pk = s->pk;
  const fast* wf = g->w;
  fast* cf = s->air && g->rg_head ? s->cfc : nullptr;
#endif
  ISW_LAUNCH("edge_hq", l_ * n_ * D + l_ * v_ * D + l_ * e_ * D + 4 * e_ * I + l_ * e_ * D + 3 * l_ * e_ * R +
                            (cf ? l_ * e_ * sizeof(fast) + e_ * D : 0),
             k_edge_hq, g1((long)E * L), BS, *g, L, s->shelf, hs, s->q, us, s->hedge, pk, cf);
  const double neoe = g->n_eoe;
  const double slow_bytes = 3 * l_ * e_ * R + neoe * (R + I) + (e_ + 1) * I + 2 * l_ * e_ * D + l_ * n_ * D +
                            2 * e_ * I + e_ * D + (s->nu4 != 0 ? l_ * e_ * D : 0) + air * 2 * l_ * n_ * D + l_ * e_ * D +
                            3 * e_ * D;
  // A thread per layer while the edges alone give a SIMD at most one wave (256 CUs of four): three layers at level 5
  // 10.4 -> 7.9 us, seven of FP64 at level 4 21.7 -> 8.4, at level 5 23.3 -> 14.6; beyond, a thread per edge: three
  // layers at level 6 12.8 us against 15.9, seven of FP64 37.9 against 43.7
#define SLOW_AS(LL, RW, GRID, BLOCK)                                                                               \
  ISW_LAUNCH("slow", slow_bytes, (k_slow_e<LL, RW>), GRID, BLOCK, *g, p, dv, c * dt, pk, wf, s->hedge, us, s->B,     \
             s->nu4 != 0 ? s->L2 : nullptr, s->air ? theta : nullptr, s->air ? s->pibar : nullptr, s->Tp, s->G, s->He, \
             s->ubs)
#define SLOW(LL)                                                                                                   \
  if (LL > 1 && E <= 64 * 1024) {                                                                                    \
    SLOW_AS(LL, true, dim3((unsigned)((E + 63) / 64)), dim3(64, LL));                                               \
  } else {                                                                                                          \
    SLOW_AS(LL, false, g1(E), BS);                                                                                  \
  }
  switch (L) {
    case 1: SLOW(1); break;
    case 2: SLOW(2); break;
    case 3: SLOW(3); break;
    case 4: SLOW(4); break;
    case 5: SLOW(5); break;
    case 6: SLOW(6); break;
    case 7: SLOW(7); break;
    default: SLOW(8); break;
  }
#undef SLOW
  int n = (int)std::ceil(c * nfast);
  if (n < 1) n = 1;
  const double tau = c * dt / n;
  FluxSrc fs{};
  fs.inv_n = 1.0 / n;
  fs.shelf = s->shelf;
  fs.stage = si;
  if (s->batch) {                                  // every world's own sub-steps: the loop runs the largest count
    n = s->batch->nmax[si];
    fs.we = s->batch->we;
    fs.winv = s->batch->inv_n;
  }
  const int KR = s->air ? ring_most(g, L, AIR_STEPS) : ring_most(g, 1, SEA_STEPS);
  if (s->air && KR) {
    // several sub-steps per launch; masses and winds alternate between (muf, mup) and (uf, ufb)
    // the last stage steps the wind in place (un is u0): where a launch might both read u0 (its first sub-step's
    // rings) and write un (a last sub-step), the sub-steps read a copy of u0 instead (s->F is free here)
    const double* uin = u0;
    if (un == u0 && (s->batch || n <= KR)) {
      ISW_LAUNCH("copy", 2 * l_ * e_ * D, k_copy, g1((long)E * L), BS, (long)E * L, u0, s->F);
      uin = s->F;
    }
    const double* mus = h0;
    int flip = 0;
    for (int it = 0; it < n; flip ^= 1) {
      const int m = ring_steps(n - it, KR);
      double* uo = flip ? s->ufb : s->uf;
      double* mo = flip ? s->mup : s->muf;
      // (algorithmic bytes: uin, the coefficients, mu in and out, S, Tp, G, acc, the wind out, 1/A, de, the patches'
      // cell and edge lists once each; the rings' re-reads and Phi* in LDS are free)
      const double bytes = l_ * e_ * D + l_ * e_ * sizeof(fast) + 3 * l_ * n_ * D + l_ * e_ * D + e_ * D +
                           (it == 0 ? 1 : 2) * l_ * e_ * D + l_ * e_ * D + n_ * D + e_ * D + 4 * n_ * I + 2 * e_ * I;
#define RINGS(LL) ring_launch(g, m, [&](auto ept, auto cpt) {                              \
    ISW_LAUNCH_SHM("af_rings", bytes, (k_af_rings<LL, decltype(ept)::value, decltype(cpt)::value>),                    \
                   dim3((unsigned)g->rg_npatch), dim3(RBS), ring_lds(g, L, m), *g, p, dv, si, it, m, n, tau, cf, uin,  \
                   mus, mo, s->S, s->Tp, s->G, s->accL, uo, un);                                                     \
  })
      switch (L) {
        case 1: RINGS(1); break;
        case 2: RINGS(2); break;
        case 3: RINGS(3); break;
        case 4: RINGS(4); break;
        case 5: RINGS(5); break;
        case 6: RINGS(6); break;
        case 7: RINGS(7); break;
        default: RINGS(8); break;
      }
#undef RINGS
      uin = uo;
      mus = mo;
      it += m;
    }
    fs.air = 1;
    fs.hedge = s->hedge;
    fs.acc = s->accL;
  } else if (s->air) {
    for (int it = 0; it < n; it++) {
      const bool first = it == 0;
      ISW_LAUNCH("af_muphi", 2 * l_ * e_ * D + 6 * n_ * (I + C) + e_ * D + n_ * D + 4 * l_ * n_ * D,
                 k_af_muphi, c1(N), dim3(BS1, L), *g, p, dv, si, it, n, tau, s->hedge, first ? u0 : s->uf,
                                                             first ? h0 : s->muf, s->muf, s->S, s->phi);
      ISW_LAUNCH("af_u", l_ * n_ * D + l_ * e_ * D + e_ * D + 2 * e_ * I + e_ * D + 2 * l_ * e_ * D +
                             (first ? 1 : 2) * l_ * e_ * D,
                 k_af_u, g1((long)E * L), BS, *g, L, dv, p, si, it, n, tau, s->phi, s->Tp, s->G,
                 first ? u0 : s->uf, s->accL, s->uf, un);
    }
    fs.air = 1;
    fs.hedge = s->hedge;
    fs.acc = s->accL;
  } else {
    if (KR && s->ubc) {
      // several sub-steps per launch: heights alternate between eta and eta_prev, winds between ubb and ubc, each
      // edge's last sub-step writes ub
      const double* ubs_ = s->ub0;
      const double* ets = s->eta0;
      int flip = 0;
      for (int it = 0; it < n; flip ^= 1) {
        const int m = ring_steps(n - it, KR);
        double* uo = flip ? s->ubc : s->ubb;
        double* eo = flip ? s->eta_prev : s->eta;
        const double bytes = 3 * e_ * D + n_ * D + 3 * n_ * D + e_ * D + e_ * D + (s->wall ? e_ * D : 0) + e_ * D +
                             (it == 0 ? 1 : 2) * e_ * D + 4 * n_ * I + 2 * e_ * I;
        ring_launch(g, m, [&](auto ept, auto cpt) {
          ISW_LAUNCH_SHM("bt_rings", bytes, (k_bt_rings<decltype(ept)::value, decltype(cpt)::value>),
                         dim3((unsigned)g->rg_npatch), dim3(RBS), ring_lds(g, 1, m), *g, dv, p, si, it, m, n, tau,
                         s->div_damp, s->He, ubs_, ets, eo, s->G, s->Gc, s->wall, s->acc, uo, s->ub);
        });
        ubs_ = uo;
        ets = eo;
        it += m;
      }
    } else
    for (int it = 0; it < n; it++) {
      const bool first = it == 0;
      ISW_LAUNCH("bt_eta", 2 * e_ * D + 6 * n_ * (I + C) + e_ * D + n_ * D + 3 * n_ * D,
                 k_bt_eta, c1(N), BS1, *g, dv, p, si, it, n, tau, s->He, first ? s->ub0 : s->ub,
                                                 first ? s->eta0 : s->eta, s->eta, s->eta_prev);
      ISW_LAUNCH("bt_u", 3 * n_ * D + e_ * D + 2 * e_ * I + e_ * D + (s->wall ? e_ * D : 0) + 2 * e_ * D +
                             (first ? 1 : 2) * e_ * D,
                 k_bt_u, g1(E), BS, *g, dv, p, si, it, n, tau, s->div_damp, s->eta, s->eta_prev, s->G,
                                              s->Gc, s->wall, first ? s->ub0 : s->ub, s->ub, s->acc);
    }
    fs.air = 0;
    fs.hs = hs;
    fs.us = us;
    fs.ubs = s->ubs;
    fs.bacc = s->acc;
    fs.wall = s->wall;
  }
  const double fb = flux_bytes(fs, n_, e_, l_);
  if (g->rg_head && g->rg_cells[1] <= RBS / 2 && g->rg_edges[1] <= 2 * RBS && g->rg_owned <= RBS) {
    // one launch on the ring patches; the first stage keeps the starting thickness for the last, which writes over it
    fs.hedge = s->hedge;
    const bool over_h0 = hn == h0;
#define LIMIT(LL)                                                                                                  \
  ISW_LAUNCH_SHM("limit_rings", fb + 3 * l_ * n_ * D + n_ * D + e_ * D + 4 * n_ * I + 2 * e_ * I +                     \
                                    (Fm ? l_ * e_ * D : 0) + (s->air ? 0 : 3 * l_ * e_ * D + 2 * e_ * D),            \
                 k_limit_rings<LL>, dim3((unsigned)g->rg_npatch), dim3(RBS),                                        \
                 (size_t)LL * (2 * RBS + 2 + RBS / 2) * sizeof(double), *g, dv, fs, c * dt, dt, s->floor_,            \
                 over_h0 ? s->hold : h0, si == 0 ? s->hold : nullptr, hn, Fm, u0, s->Tp, s->ub, s->ub0,               \
                 s->air ? nullptr : un)
    switch (L) {
      case 1: LIMIT(1); break;
      case 2: LIMIT(2); break;
      case 3: LIMIT(3); break;
      case 4: LIMIT(4); break;
      case 5: LIMIT(5); break;
      case 6: LIMIT(6); break;
      case 7: LIMIT(7); break;
      default: LIMIT(8); break;
    }
#undef LIMIT
    return;
  }
  ISW_LAUNCH("scale", fb + 6 * n_ * I + 2 * e_ * I + e_ * D + l_ * n_ * D + n_ * D + l_ * n_ * D,
             k_scale, g1((long)N * L), BS, *g, fs, c * dt, s->floor_, h0, s->scale, L);
  ISW_LAUNCH("limit_h", fb + 6 * n_ * (I + C) + 2 * e_ * I + e_ * D + 3 * l_ * n_ * D + n_ * D +
                            (Fm ? l_ * e_ * D : 0),
             k_limit_h, g1((long)N * L), BS, *g, dv, fs, c * dt, dt, s->scale, h0, hn, Fm, L);
  if (!s->air)
    ISW_LAUNCH("lay_u", 3 * l_ * e_ * D + 2 * e_ * D + (s->wall ? e_ * D : 0),
               k_lay_u, g1((long)E * L), BS, E, L, c * dt, u0, s->Tp, s->ub, s->ub0, s->wall, un);
}

int layers_step(const isw_grid* g, const isw_layers* s, double* h, double* u, double* theta, double* Fm, double dt,
                int nfast, hipStream_t st) {
  const LP p = make_lp(s);
  const Div dv = divs(g);
  const int N = g->N, L = s->L;
  const double n_ = N, e_ = g->E, l_ = L;
  // (the last stage's copy of u, where one launch takes all of its sub-steps)
  const int KR = s->air ? ring_most(g, L, AIR_STEPS) : 0;
  if (KR && !s->F && (s->batch || nfast <= KR)) return ISW_EBADARG;
  if (s->air) {
    ISW_LAUNCH("air_stiff", 3 * l_ * n_ * D, k_air_stiff, c1(N), BS1, N, p, h, theta, s->S);
  } else {
    ISW_LAUNCH("lay_eta", (l_ + 2) * n_ * D, k_lay_eta, c1(N), BS1, N, L, h, s->b, s->eta0);
    ISW_LAUNCH("lay_ubar", l_ * n_ * D + l_ * e_ * D + 2 * e_ * I + (s->wall ? e_ * D : 0) + e_ * D,
               k_lay_ubar, g1(g->E), BS, *g, L, s->shelf, h, u, s->wall, s->ub0);
  }
  if (s->nu4 != 0) {
    lap(g, L, u, s->D1, s->Z1, s->L1, st);
    lap(g, L, s->L1, s->D1, s->Z1, s->L2, st);
  }
  stage(g, s, p, dv, 0, h, u, h, u, 1.0 / 3.0, dt, nfast, s->h1, s->u1, nullptr, theta, st);
  stage(g, s, p, dv, 1, s->h1, s->u1, h, u, 1.0 / 2.0, dt, nfast, s->h2, s->u2, nullptr, theta, st);
  stage(g, s, p, dv, 2, s->h2, s->u2, h, u, 1.0, dt, nfast, h, u, Fm, theta, st);
  if ((s->vmix != 0 || s->vmix_cd != 0) && L > 1) {
    ISW_LAUNCH("lay_vmix", l_ * n_ * D + 2 * e_ * I + 2 * l_ * e_ * D + e_ * D + (s->wall ? e_ * D : 0),
               k_lay_vmix, g1(g->E), BS, *g, L, s->vmix, dt, s->vmix_cd, h, s->wall, u, s->diss);
    if (s->air)
      ISW_LAUNCH("vmix_heat", 6 * n_ * I + 3 * e_ * D + n_ * D + 3 * l_ * n_ * D,
                 k_vmix_heat, c1(N), BS1, *g, p, h, s->diss, theta);
  }
  return (int)hipGetLastError();
}

int layers_lap(const isw_grid* g, const isw_layers* s, const double* u, double* out, hipStream_t st) {
  lap(g, s->L, u, s->D1, s->Z1, out, st);
  return (int)hipGetLastError();
}

int layers_gfast(const isw_grid* g, const isw_layers* s, const double* h, const double* theta, hipStream_t st) {
  if (s->air)
    ISW_LAUNCH("air_gfast", 3.0 * s->L * g->N * D,
               k_air_gfast, c1(g->N), BS1, g->N, make_lp(s), s->rd, h, theta, s->Gc);
  return (int)hipGetLastError();
}

int layers_exchange(const isw_grid* g, const isw_layers* s, const double* wx, double* h, double* u, double* M,
                    double* psi, double* theta, int seq, double nu4dt, hipStream_t st) {
  const int N = g->N, L = s->L;
  const double n_ = N, e_ = g->E, l_ = L;
  ISW_LAUNCH("copy", 2 * l_ * n_ * D, k_copy, g1((long)N * L), BS, (long)N * L, h, s->hold);
  const bool heat = s->air && theta;
  ISW_LAUNCH("xch_cell", (l_ - 1) * n_ * D + n_ * D + 6 * l_ * n_ * D,
             k_xch_cell, c1(N), BS1, N, L, seq, wx, g->areaCell, h, M, psi);
  const bool v4 = heat && s->nu4 != 0;
  ISW_LAUNCH("xch_edge", (l_ - 1) * n_ * D + l_ * n_ * D + 2 * e_ * I + 2 * l_ * e_ * D + (heat ? e_ * D : 0) +
                             (v4 ? l_ * e_ * D : 0) + (s->wall ? e_ * D : 0),
             k_xch_edge, g1(g->E), BS, *g, L, wx, s->hold, u, heat ? s->diss : nullptr,
                                                 v4 ? s->L2 : nullptr, v4 ? nu4dt : 0.0, heat ? s->thin_wind : 0.0,
                                                 s->floor_, s->wall);
  if (heat)
    ISW_LAUNCH("vmix_heat", 6 * n_ * I + 3 * e_ * D + n_ * D + 3 * l_ * n_ * D,
               k_vmix_heat, c1(N), BS1, *g, make_lp(s), h, s->diss, theta);
  return (int)hipGetLastError();
}

int vmix_heat(const isw_grid* g, const isw_layers* s, const double* h, const double* diss, double* theta,
              hipStream_t st) {
  const double n_ = g->N, e_ = g->E, l_ = s->L;
  ISW_LAUNCH("vmix_heat", 6 * n_ * I + 3 * e_ * D + n_ * D + 3 * l_ * n_ * D,
             k_vmix_heat, c1(g->N), BS1, *g, make_lp(s), h, diss, theta);
  return (int)hipGetLastError();
}

int mass_update(const isw_grid* g, int L, const double* M0, const double* Fm, double* M1, hipStream_t st) {
  const double n_ = g->N, e_ = g->E, l_ = L;
  ISW_LAUNCH("mass_update", 2 * l_ * n_ * D + l_ * e_ * D + 6 * n_ * I + e_ * I,
             k_mass_update, c2(g->N, L), BS1, *g, M0, Fm, M1);
  return (int)hipGetLastError();
}

// The rows to a block of the passes that keep the rows cell-major on the patches (4 or 8), 0 for those that keep them apart.
// They need the patches, the scratch's rows padded to a multiple of four (rows_pad at least rows_max: a smaller one is
// taken as not given) and every array of it where 16 bytes are loaded at once.
int transport_shape(const isw_grid* g, const isw_transport* tr, int rows) {
  constexpr int CUS = 256;
  const int RS = (rows + 3) / 4 * 4, c4 = RS / 4, c8 = (RS + 7) / 8;
  if (!g->pi_off || g->pcells != BS1 || g->E < g->N || RS > tr->rows_pad || tr->rows_max > tr->rows_pad) return 0;
  if (ISW_FORM_MIXED && !tr->pf2) return 0;
  const void* at[] = {tr->td, tr->p1, tr->p2, tr->Rp, tr->Rm, tr->Hf, tr->A, tr->pf, tr->pf2};
  for (const void* p : at)
    if (reinterpret_cast<uintptr_t>(p) & 15) return 0;
  const long b4 = (long)g->npatch * c4, b8 = (long)g->npatch * c8;
  auto fits = [&](int rc) { return (size_t)g->ptedges * rc * 2 * sizeof(double) <= 65536 ? rc : 0; };
  if (rows < 3) return 0;                          // (2 rows at level 6, FP64: 38 us apart, 43 with two of padding)
  // Four rows to a block: where no more are there, and on meshes so small that every block has a CU of its own (the mixed
  // form: a third of one), for then a pass takes as long as its blocks do, which is less for smaller ones, and padding is
  // free (level 4, 15 rows, FP64: 35.1 us apart, 37.3 eight to a block, 34.0 four; 5 rows 34.1, 35.3, 30.5; level 5, mixed,
  // 15 rows 47.7, 45.0, 43.4; FP64, at two blocks to a CU, 50.1, 49.1, 53.0); and for ten to twelve, which eight to a
  // block would pad to sixteen (12 rows: level 5, FP64, 44.5 us, 47.0, 38.5; level 6, mixed, 100.5, 87.8, 76.5)
  if (c4 == 1 || (c4 == 3 && rows > 9) || b4 <= (ISW_FORM_MIXED ? 3 : 1) * CUS) return fits(4);
  // Eight: they share the edges' tables twice as often (15 rows at level 6: 96.1 us of kernels against 110.4), but cost as
  // much for a padded row as for a real one: with three in four of their rows real or more (9 of 16 at level 6 81 us apart,
  // 88 so; 5 of 8, FP64, 63 and 65, but at level 5, a CU to a block, 37.7 and 36.4; 20 of 24 at level 6 151 and 123), and,
  // of more than one chunk, with five in nine of what the chip could hold in the rounds that its CUs take blocks in (FP64,
  // level 5: 14 rows of seven layers, 0.55 of two rounds, 48.8 us apart and 50.4 so; 15 rows, 0.59, 50.1 and 49.2; level 4:
  // 25 rows, 0.50, 37.4 and 37.8; 28, 0.56, 40.7 and 37.7)
  const long rounds = (b8 + CUS - 1) / CUS;
  const bool real = rows * 4 >= 3 * 8 * c8 || (c8 == 1 && b8 <= CUS);
  const bool held = c8 == 1 || 9l * rows * g->npatch >= 5 * 8 * CUS * rounds;
  return real && held ? fits(8) : 0;
}

// Transport.step_many (transport.py:40-71) on rows stacked in psi; the result is written back into psi.
int transport_step(const isw_grid* g, const isw_transport* tr, const double* M0, const double* M1, const double* Fm,
                   double* psi, int rows, int order, hipStream_t st) {
  const int N = g->N, E = g->E, Lm = tr->L;
  const double n_ = N, e_ = E, l_ = Lm, r_ = rows, mixed = ISW_FORM_MIXED ? 1 : 0;
#if ISW_FORM_MIXED
  float* pf = tr->pf;
  const fast* wt = g->d2wtf;
#else
  float* pf = nullptr;
  const fast* wt = g->d2wt;
#endif
  // On the patches with the rows cell-major: psi's cell-major copy is in Hf, the FP32 copies alternate between pf and pf2
  // (stage 1 writes p1's to pf2; stage 2 reads it and writes p2's to pf).
  const int RC = order == 3 ? transport_shape(g, tr, rows) : 0;
  if (RC) {
    const int RS = (rows + 3) / 4 * 4, chunks = (RS + RC - 1) / RC;
    const size_t lds = (size_t)g->ptedges * RC * sizeof(double);
    const double tabs = 2 * e_ * I + 6 * n_ * I, edge1 = 8 * e_ * (R + I) + l_ * e_ * D + 2 * e_ * I;
    double* pc = tr->Hf;
#if ISW_FORM_MIXED
    float *pfa = tr->pf, *pfb = tr->pf2;
    const fast *f0 = pfa, *f1 = pfb, *f2 = pfa;
#else
    float *pfa = nullptr, *pfb = nullptr;
    const fast *f0 = pc, *f1 = tr->p1, *f2 = tr->p2;
#endif
    const dim3 gp((unsigned)(g->npatch * chunks));
    ISW_LAUNCH("tr_turn", 2 * r_ * n_ * D + mixed * r_ * n_ * 4, k_tr_turn,
               dim3((unsigned)((N + BS1 - 1) / BS1), (unsigned)((RS + 15) / 16)), BS, N, rows, RS, psi, pc, pfa);
    const double mv = 3 * r_ * n_ * D + 2 * mixed * r_ * n_ * 4 + edge1 + l_ * n_ * D + tabs + 6 * n_ * I;
#define TRANSPORT(C)                                                                                              \
  ISW_LAUNCH_SHM("tr_move", mv + r_ * n_ * D + l_ * n_ * D, (k_tr_move<C, true>), gp, BS, 2 * lds, *g, Lm, RS, chunks, \
                 1.0 / 3.0, tr->beta, pc, f0, wt, Fm, M0, M1, pc, tr->p1, pfb, tr->td);                              \
  ISW_LAUNCH_SHM("tr_move", mv, (k_tr_move<C, false>), gp, BS, lds, *g, Lm, RS, chunks, 1.0 / 2.0, tr->beta, tr->p1,   \
                 f1, wt, Fm, M0, M1, pc, tr->p2, pfa, nullptr);                                                     \
  ISW_LAUNCH_SHM("tr_limit", 5 * r_ * n_ * D + mixed * r_ * n_ * 4 + edge1 + l_ * n_ * D + tabs + 6 * n_ * I +         \
                                 r_ * e_ * D,                                                                     \
                 k_tr_limit<C>, gp, BS, lds, *g, Lm, RS, chunks, tr->beta, pc, tr->p2, f2, wt, Fm, tr->td, M1,        \
                 tr->A, tr->Rp, tr->Rm);                                                                          \
  ISW_LAUNCH_SHM("tr_correct", 4 * r_ * n_ * D + r_ * e_ * D + l_ * n_ * D + 2 * e_ * I + tabs, k_tr_correct<C>, gp, BS, \
                 lds, *g, Lm, rows, RS, chunks, tr->td, M1, tr->A, tr->Rp, tr->Rm, psi)
    if (RC == 8) {
      TRANSPORT(8);
    } else {
      TRANSPORT(4);
    }
#undef TRANSPORT
    return (int)hipGetLastError();
  }
  const double cellE = 6 * n_ * I + 2 * e_ * I;  // cellEdgeAsc, eI/eJ
  const double sten = 8 * e_ * (R + I) + l_ * e_ * D + 2 * e_ * I;
  ISW_LAUNCH("tr_td", 2 * l_ * n_ * D + r_ * n_ * D + l_ * e_ * D + cellE + r_ * n_ * D + mixed * r_ * n_ * 4,
             k_tr_td, c4(N, rows), dim3(BS1, 4), *g, Lm, rows, M0, psi, Fm, M1, tr->td, pf);
  if (order == 1) {
    ISW_LAUNCH("copy", 2 * r_ * n_ * D, k_copy, g1((long)N * rows), BS, (long)N * rows, tr->td, psi);
    return (int)hipGetLastError();
  }
#if ISW_FORM_MIXED
  const fast* psf = pf;
  const fast* p1f = pf;
  const fast* p2f = pf;
#else
  const fast* psf = psi;
  const fast* p1f = tr->p1;
  const fast* p2f = tr->p2;
#endif
  const bool fused = g->pi_off && g->pcells == BS1 && (!ISW_FORM_MIXED || tr->pf2) &&
                     (size_t)4 * g->ptedges * sizeof(double) <= 65536;
  if (fused) {
    // (algorithmic bytes: the stencil's field and its FP32 copy, the stencil and its weights, Fm, M0, psi, the
    // output and its copy, the cell rings and the patch tables; the flux stays in LDS)
    const double tabs = 6 * n_ * I + 2 * (n_ / BS1 + 1) * I + 2 * e_ * I + 6 * n_ * I;
    const size_t shm = (size_t)4 * g->ptedges * sizeof(double);
#if ISW_FORM_MIXED
    float* pfb = tr->pf2;
    const fast* p1s = tr->pf2;                     // (stage 1 writes p1's copy to pf2; stage 2 reads it, writes pf)
#else
    float* pfb = nullptr;
    const fast* p1s = tr->p1;
#endif
    const dim3 gp((unsigned)g->npatch, (unsigned)((rows + 3) / 4));
    ISW_LAUNCH_SHM("tr_hstage", r_ * n_ * D + mixed * r_ * n_ * 4 + sten + l_ * n_ * D + r_ * n_ * D + tabs +
                                    r_ * n_ * D + mixed * r_ * n_ * 4,
                   k_tr_hstage, gp, dim3(BS1, 4), shm, *g, Lm, rows, 1.0 / 3.0, tr->beta, psi, psf, wt, Fm, M0, psi,
                   tr->p1, pfb);
    ISW_LAUNCH_SHM("tr_hstage", r_ * n_ * D + mixed * r_ * n_ * 4 + sten + l_ * n_ * D + r_ * n_ * D + tabs +
                                    r_ * n_ * D + mixed * r_ * n_ * 4,
                   k_tr_hstage, gp, dim3(BS1, 4), shm, *g, Lm, rows, 1.0 / 2.0, tr->beta, tr->p1, p1s, wt, Fm, M0,
                   psi, tr->p2, pf);
  } else {
    ISW_LAUNCH("tr_hflux", r_ * n_ * D + mixed * r_ * n_ * 4 + sten + r_ * e_ * D,
               k_tr_hflux, c4(E, rows), dim3(BS1, 4), *g, Lm, rows, 1.0 / 3.0, tr->beta, psi, psf, wt, Fm, tr->Hf);
    ISW_LAUNCH("tr_stage", l_ * n_ * D + r_ * n_ * D + r_ * e_ * D + l_ * e_ * D + cellE + r_ * n_ * D +
                               mixed * r_ * n_ * 4,
               k_tr_stage, c4(N, rows), dim3(BS1, 4), *g, Lm, rows, 1.0 / 3.0, M0, psi, tr->Hf, Fm, tr->p1, pf);
    ISW_LAUNCH("tr_hflux", r_ * n_ * D + mixed * r_ * n_ * 4 + sten + r_ * e_ * D,
               k_tr_hflux, c4(E, rows), dim3(BS1, 4), *g, Lm, rows, 1.0 / 2.0, tr->beta, tr->p1, p1f, wt, Fm,
               tr->Hf);
    ISW_LAUNCH("tr_stage", l_ * n_ * D + r_ * n_ * D + r_ * e_ * D + l_ * e_ * D + cellE + r_ * n_ * D +
                               mixed * r_ * n_ * 4,
               k_tr_stage, c4(N, rows), dim3(BS1, 4), *g, Lm, rows, 1.0 / 2.0, M0, psi, tr->Hf, Fm, tr->p2, pf);
  }
  ISW_LAUNCH("tr_aflux", 2 * r_ * n_ * D + mixed * r_ * n_ * 4 + sten + r_ * e_ * D,
             k_tr_aflux, dim3((unsigned)((E + BS - 1) / BS), (unsigned)((rows + 3) / 4)), dim3(BS1, 4), *g, Lm, rows,
             tr->beta, psi, tr->p2, p2f, wt, Fm, tr->A);
  ISW_LAUNCH("tr_ratios", 2 * r_ * n_ * D + l_ * n_ * D + r_ * e_ * D + 6 * n_ * I + cellE + 2 * r_ * n_ * D,
             k_tr_ratios, c4(N, rows), dim3(BS1, 4), *g, Lm, rows, psi, tr->td, M1, tr->A, tr->Rp, tr->Rm);
  ISW_LAUNCH("tr_apply", r_ * n_ * D + l_ * n_ * D + r_ * e_ * D + 2 * r_ * n_ * D + cellE + r_ * n_ * D,
             k_tr_apply, c4(N, rows), dim3(BS1, 4), *g, Lm, rows, tr->td, M1, tr->A, tr->Rp, tr->Rm, psi);
  return (int)hipGetLastError();
}

int swe_step(const isw_grid* g, const isw_layers* s, double* h, double* u, double* Fm, double dt, hipStream_t st) {
  const LP p = make_lp(s);
  const Div dv = divs(g);
  const int N = g->N, E = g->E, NV = g->NV, L = s->L;
  const double n_ = N, e_ = E, v_ = NV, l_ = L;
  if (s->nu4 != 0) {
    lap(g, L, u, s->D1, s->Z1, s->L1, st);
    lap(g, L, s->L1, s->D1, s->Z1, s->L2, st);
  }
  const double cs[3] = {dt / 3, dt / 2, dt};
  const double* hsv[3] = {h, s->h1, s->h2};
  const double* usv[3] = {u, s->u1, s->u2};
  double* hnv[3] = {s->h1, s->h2, h};
  double* unv[3] = {s->u1, s->u2, u};
  for (int k = 0; k < 3; k++) {
    const double c = cs[k];
    ISW_LAUNCH("swe_scale", l_ * n_ * D + l_ * e_ * D + 6 * n_ * I + 2 * e_ * I + e_ * D + n_ * D + l_ * n_ * D,
               k_swe_scale, c2(N, L), BS1, *g, c, hsv[k], usv[k], s->scale);
    ISW_LAUNCH("swe_flux", l_ * n_ * D + l_ * e_ * D + 2 * e_ * I + l_ * n_ * D + l_ * e_ * D +
                               (k == 2 && Fm ? l_ * e_ * D + e_ * D : 0),
               k_swe_flux, g2(E, L), BS, *g, k == 2 ? dt : 0.0, hsv[k], usv[k], s->scale, s->F,
                                                   k == 2 ? Fm : nullptr);
    ISW_LAUNCH("swe_cell", 2 * l_ * n_ * D + n_ * D + 2 * l_ * e_ * D + 6 * n_ * (I + C) + 2 * e_ * D + n_ * D +
                               2 * l_ * n_ * D,
               k_swe_cell, c2(N, L), BS1, *g, s->grav, c, hsv[k], s->b, s->F, usv[k], h, hnv[k], s->B);
    ISW_LAUNCH("swe_vertex", l_ * n_ * D + l_ * e_ * D + 3 * v_ * (2 * I + 2 * C) + 6 * n_ * D + e_ * D +
                                 2 * v_ * D + l_ * v_ * D,
               k_swe_vertex, c2(NV, L), BS1, *g, dv, hsv[k], usv[k], s->fV, s->q);
    ISW_LAUNCH("swe_edge", l_ * e_ * D + l_ * v_ * D + l_ * n_ * D + l_ * e_ * D + g->n_eoe * (D + I) +
                               (e_ + 1) * I + 4 * e_ * I + e_ * D + (s->nu4 != 0 ? l_ * e_ * D : 0) + 2 * l_ * e_ * D,
               k_swe_edge_lp, g2(E, L), BS, *g, p, c, s->F, s->q, s->B, usv[k], s->L2, u, unv[k]);
  }
  return (int)hipGetLastError();
}

int couple_stress(const isw_grid* g, int La, const double* ha, double* ua, const double* ho, double* uo, double c,
                  double rho_w, double dt, double* diss, double* tau_acc, const double* wall, double land_drag,
                  const double* cd, hipStream_t st) {
  const double n_ = g->N, e_ = g->E;
  ISW_LAUNCH("couple_stress", 2 * n_ * D + 4 * e_ * D + 2 * e_ * I + e_ * D + 2 * e_ * D + (wall ? e_ * D : 0) +
                                  (cd ? n_ * D : 0),
             k_couple_stress, g1(g->E), BS, *g, La, c, rho_w, dt, land_drag, ha, ua, ho, uo, diss, tau_acc,
                                                      wall, cd);
  return (int)hipGetLastError();
}

int land_column(const isw_grid* g, int K, const double* land, double* T, const double* cap, double* Tg,
                const double* dz, double c_soil, double k_soil, double dt, hipStream_t st) {
  const double n_ = g->N;
  ISW_LAUNCH("land_column", n_ * D + 2 * n_ * D + n_ * D + 2.0 * K * n_ * D + K * D,
             k_land_column, c1(g->N), BS1, g->N, K, c_soil, k_soil, dt, land, T, cap, Tg, dz);
  return (int)hipGetLastError();
}

int ocn_cap(const isw_grid* g, const double* h, double rho_cw, double* cap, const double* land, double c_land,
            hipStream_t st) {
  const double n_ = g->N;
  ISW_LAUNCH("ocn_cap", n_ * D + 2 * n_ * D + (land ? n_ * D : 0),
             k_ocn_cap, c1(g->N), BS1, g->N, rho_cw, c_land, h, cap, land);
  return (int)hipGetLastError();
}

int fill(double* x, long n, double v, hipStream_t st) {
  if (n > 0) ISW_LAUNCH("fill", 8.0 * n, k_fill, g1(n), BS, n, v, x);
  return (int)hipGetLastError();
}

}  // namespace NS
