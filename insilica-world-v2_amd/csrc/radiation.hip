// The k-table radiation as gfx950 HIP kernels: the longwave's sub-level set-up and column pass, the shortwave's
// column pass (reference: src/insilica/radiation.py; kernels/air.cu:2111-2511).
//
// Compiled twice, as core.hip: ISW_FORM_MIXED=0 with -ffp-contract=off into isw_f64 (the plain form, `fast` = double,
// the reference's double build with its float32 storage points kept: tables, sub-levels, clamped table positions and
// per-g-point results), ISW_FORM_MIXED=1 with -ffp-contract=fast into isw_mix (`fast` = float and the transcendentals
// in float, as the reference's MIXED build; every g-point sum stays FP64).
//
// Design (MI355X): a 64-aligned block takes columns in turn, one thread per g-point, the column's sub-level properties
// staged once in LDS as what the walk needs (table offsets and shares, amounts). Kernels are instantiated per
// layer count so that every per-g-point array has a compile-time size and stays in VGPRs, and each walks the sub-levels
// once: what the walk back needs is kept as small linear maps per layer instead of being computed again. A column's table
// rows are the same for all its g-points, so their bases are scalar and the lanes differ by g alone. Per-g results go to
// LDS as float32 (the reference's red[][] width) and are summed in FP64 in a fixed order, so results repeat bit for bit.
// Blocks are renumbered so that each XCD takes a contiguous range of columns (the sub-level reads of neighbouring columns
// share cache lines). Measured at 40,962 columns x 7 layers, mixed: lw_column (256 g-points) 3.72 -> 1.44 ms, sw_column
// (224) 6.86 -> 2.18 ms; FP64 at 2,562 x 3 (144 / 112): 192 -> 109 us and 273 -> 113 us.
#include <hip/hip_runtime.h>

#include <cmath>
#include <type_traits>

#include "diag.hpp"
#include "insilica_hip.h"

#if ISW_FORM_MIXED
#define NS isw_mix
typedef float fast;
#else
#define NS isw_f64
typedef double fast;
#endif

namespace NS {

constexpr int NSUB = 4, NVP = 15, NGMAX = 256;
constexpr double PI_ = 3.14159265358979323846;

// The reference's transcendental macros (air.cu:26-38): FP64 in the plain form; in the mixed form FEXP and FPOW run
// in float and return double.
__device__ __forceinline__ double FEXPd(double x) {
#if ISW_FORM_MIXED
  return (double)expf((float)x);
#else
  return exp(x);
#endif
}
__device__ __forceinline__ double FPOWd(double x, double y) {
#if ISW_FORM_MIXED
  return (double)powf((float)x, (float)y);
#else
  return pow(x, y);
#endif
}
// The column passes' exp and quotient: FP64 in the plain form (the reference's operations); in the mixed form the
// hardware's: exp as 2^(x log2 e) (v_exp_f32) and a / b as a times the hardware reciprocal, each within a few float
// steps (the mixed form's bar against FP64 is 1e-4 of the fluxes). fquot stands in the longwave's emission and in the two
// denominators of the shortwave's adding, where an IEEE quotient was no closer to 64 bits.
__device__ __forceinline__ fast fexp(fast x) {
#if ISW_FORM_MIXED
  return __expf(x);
#else
  return exp(x);
#endif
}
__device__ __forceinline__ fast fquot(fast a, fast b) {
#if ISW_FORM_MIXED
  return a * __builtin_amdgcn_rcpf(b);
#else
  return a / b;
#endif
}
// The shortwave's layer optics divide by 1 - (k mu0)^2, which passes through zero where the beam and the diffuse light
// decay alike: what they lose to rounding there is a thousand times larger, so their quotients and square root take one
// Newton step on the hardware's reciprocal and one on the residual (the root one on the residual alone), and the quotients
// the fix-up for zeros and infinities: within a float step of IEEE's for normal operands, mostly equal to them, though
// not shown to be in every case. Six instructions besides the reciprocal where the compiler's division takes ten, for
// it does not scale: where b is denormal its reciprocal is infinite and the Newton step not a number, so what may vanish
// is divided by only above TINY.
constexpr fast TINY = ISW_FORM_MIXED ? (fast)1.17549435e-38f : (fast)0;
__device__ __forceinline__ fast fdiv(fast a, fast b) {
#if ISW_FORM_MIXED
  float y = __builtin_amdgcn_rcpf(b);
  y = __builtin_fmaf(__builtin_fmaf(-b, y, 1.f), y, y);
  const float q = a * y;
  return __builtin_amdgcn_div_fixupf(__builtin_fmaf(__builtin_fmaf(-b, q, a), y, q), b, a);
#else
  return a / b;
#endif
}
__device__ __forceinline__ fast fsqrt(fast x) {         // (x >= 1e-12)
#if ISW_FORM_MIXED
  const float y = __builtin_amdgcn_rsqf(x), s = x * y;
  return __builtin_fmaf(__builtin_fmaf(-s, s, x), 0.5f * y, s);
#else
  return sqrt(x);
#endif
}

// XCD-aware block order (as the stencils'): XCD x takes one contiguous range of blocks.
__device__ __forceinline__ int xblock() {
  const int nb = (int)gridDim.x, b = (int)blockIdx.x;
  const int q = nb >> 3, r = nb & 7, x = b & 7, k = b >> 3;
  return (x < r ? x * (q + 1) : r * (q + 1) + (x - r) * q) + k;
}

// The parameters the radiation reads from the reference's PAR_ORDER array (air.cu:118-127), by value.
struct RadP {
  double eps_s, grav, cp, kappa, p0, tilt, year_s, day_s, cloud_g, bl_q, ice_air, lw_refl, ecc, lam_peri;
  int edge_k;
};

static RadP make_radp(const double* a) {
  RadP p;
  p.eps_s = a[4]; p.grav = a[13]; p.cp = a[14]; p.kappa = a[15]; p.p0 = a[16]; p.tilt = a[17]; p.year_s = a[18];
  p.day_s = a[19]; p.cloud_g = a[59]; p.bl_q = a[89]; p.edge_k = (int)a[101]; p.ice_air = a[102];
  p.lw_refl = a[124]; p.ecc = a[126]; p.lam_peri = a[127];
  return p;
}

// A table position clamped as the reference writes it, fminf(fmaxf(x, 0.f), (n - 1) - 1e-4f): float arguments,
// so the position is rounded to float in either form.
__device__ __forceinline__ float clampf_pos(fast x, int n) {
  return fminf(fmaxf((float)x, 0.f), (float)((fast)(n - 1) - (fast)1e-4f));
}

// Tetens over water (air.cu:160-162), and blended with ice below freezing (air.cu:165-171).
__device__ __forceinline__ fast qsat_w(fast T, fast p, double eps) {
  return (fast)eps * (fast)611.0 * (fast)FEXPd((fast)17.27 * (T - (fast)273.15) / (T - (fast)35.85)) / p;
}
__device__ __forceinline__ fast qsat_a(fast T, fast p, double ice, double eps) {
  const fast w = qsat_w(T, p, eps);
  if (!(ice > 0) || T >= (fast)273.15) return w;
  const fast l = fmin((fast)1, fmax((fast)0, (T - (fast)253.15) / (fast)20));
  const fast si = (fast)eps * (fast)611.0 * (fast)FEXPd((fast)21.875 * (T - (fast)273.16) / (T - (fast)7.66)) / p;
  return l * w + (1 - l) * si;
}

// ---------------------------------------------------------------------------------------------------------------
// lw_setup (air.cu:2145-2229): one thread per (column, layer); 64 columns per block, blockIdx.y the layer.
// Per sub-level: edge temperatures (the layer isothermal above the 380 K edge, else T ~ p^n keeping the layer's mean
// temperature), table positions, gas amounts (vapor at the layer's mean relative humidity), cloud cover and optical
// depth (in the sub-level holding the median of the layer's vapor), air molecules, the haze's share, CIA weight.
// ---------------------------------------------------------------------------------------------------------------
template <int L>
__global__ void __launch_bounds__(64) k_lw_setup(int N, RadP P, isw_lw_tables t, isw_air air, double co2,
                                                  double n2o, double ch4, const double* __restrict__ gx,
                                                  const double* __restrict__ mu_in, const double* __restrict__ theta,
                                                  const double* __restrict__ qv, const double* __restrict__ cloudo,
                                                  double hs, int tmode, float* __restrict__ sub) {
  // No contraction here in either form: the layer edges, the sub-levels' pressures and the vapor's running share are
  // then the same bits in both, and so is every discrete choice made from them (the cloud's sub-level: an even vapor
  // profile puts the median exactly on a sub-level boundary, decided by the last bit). The kernel is a small share of
  // the radiation's time.
#pragma clang fp contract(off)
  const int i = xblock() * 64 + (int)threadIdx.x, k = (int)blockIdx.y;
  if (i >= N) return;
  double pb[L], pib[L], th_k = 0, q_k = 0;
  {
    double p = 0, xt = 0;
#pragma unroll
    for (int j = 0; j < L; j++) {
      const double pt = p;
      p = p + P.grav * mu_in[(size_t)j * N + i];
      pb[j] = p;
      const double x = pow(p / P.p0, P.kappa);
      pib[j] = P.cp * (p * x - pt * xt) / ((P.kappa + 1) * (p - pt));
      xt = x;
    }
  }
  th_k = theta[(size_t)k * N + i];
  q_k = qv ? fmax(qv[(size_t)k * N + i], 0.0) : 0.0;
  double pt = 0, pbk = 0, pibk = 0, pbL = pb[L - 1];
#pragma unroll
  for (int j = 0; j < L; j++)
    if (j == k) { pbk = pb[j]; pibk = pib[j]; }
#pragma unroll
  for (int j = 0; j < L; j++)
    if (j == k - 1) pt = pb[j];
  const bool strat = k < P.edge_k && L >= 3;
  const double Tiso = pibk * th_k / P.cp;
  const double nT = tmode == 1 ? P.kappa : 0.190;
  const double Cn = Tiso * (nT + 1) * (pbk - pt) / (pow(pbk, nT + 1) - pow(pt, nT + 1));
  auto Tof = [&](double p) -> double { return tmode == 0 || strat ? Tiso : Cn * FPOWd(p, nT); };
  const fast fcl = cloudo ? (fast)cloudo[(size_t)k * N + i] : (fast)0;
  const fast tcl = cloudo ? (fast)cloudo[(size_t)(L + 3 + k) * N + i] : (fast)0;
  const double FT[5] = {0, 0.05, 0.2, 0.5, 1}, FE[5] = {0, 0.25, 0.5, 0.75, 1};
  // the layer's vapor sum and the cloud's median test stay FP64 in both forms: with the vapor even (above the edge) the
  // median falls exactly on a sub-level boundary, where float rounding would move the cloud to the next sub-level
  fast qs[NSUB], uas[NSUB];
  double qm = 0;
  double pe[NSUB + 1];
#pragma unroll
  for (int j = 0; j <= NSUB; j++) pe[j] = pt + (k == 0 ? FT[j] : FE[j]) * (pbk - pt);
  const bool blq = P.bl_q > 0 && k == L - 1 && k > 0;
#define W(s, v) sub[((size_t)(s) * NVP + (v)) * N + i]
#pragma unroll
  for (int j = 0; j < NSUB; j++) {
    const int s = k * NSUB + j;
    const double a = pe[j], b = pe[j + 1], pm = a > 0 ? (b - a) / log(b / a) : 0.5 * b;
    const double Tm = Tof(0.5 * (a + b));
    W(s, 0) = (float)Tof(a);
    W(s, 1) = (float)Tof(b);
    // (FP64 pow in both forms: the 160 K cut-off below decides whether a sub-level holds vapor, which moves the cloud)
    const double Tq = th_k * pow(0.5 * (a + b) / P.p0, P.kappa);
    qs[j] = strat || blq ? (fast)1 : (Tq < 160 ? (fast)0 : qsat_a((fast)Tq, (fast)pm, P.ice_air, air.eps));
    qm += (double)qs[j] * ((b - a) / (pbk - pt));
    const fast x = (fast)((t.lp0 - log(pm * air.broad)) / t.dlp), y = (fast)((Tm - t.t0) / t.dtt);
    W(s, 2) = clampf_pos(x, t.NP);
    W(s, 3) = clampf_pos(y, t.NT);
    const fast ua = (fast)((b - a) / (P.grav * air.m_air_kg) * 6.02214076e23 / 1e4);
    const fast yo = clampf_pos((fast)((t.o3lp0 - log(pm)) / t.o3dlp), t.NO3);
    const int io = (int)yo;
    const fast xo3 = (fast)((t.o3[io] + (t.o3[io + 1] - t.o3[io]) * (yo - (fast)io)) * (fast)air.o3);
    const double xc = gx ? gx[(size_t)k * N + i] : co2, xn = gx ? gx[(size_t)(L + k) * N + i] : n2o;
    const double xm = gx ? gx[(size_t)(2 * L + k) * N + i] : ch4;
    W(s, 5) = (float)((fast)xc * ua);
    W(s, 6) = (float)(xo3 * ua);
    W(s, 7) = (float)((fast)xn * ua);
    W(s, 8) = (float)((fast)xm * ua);
    W(s, 11) = (float)fcl;
    W(s, 12) = (float)ua;
    W(s, 13) = (float)(FPOWd(b / pbL, 8000.0 / hs) - FPOWd(a / pbL, 8000.0 / hs));
    W(s, 14) = air.cia ? (float)((double)ua * 1e-20 * (pm / (1.380649e-23 * Tm) * 1e-6) * 1e-20) : 0.f;
    uas[j] = ua;
  }
  // the cloud's sub-level: the one holding the median of the layer's vapor
  int jc = NSUB - 1;
  {
    double cum = 0;
    bool found = false;
#pragma unroll
    for (int j = 0; j < NSUB; j++) {
      cum += qm > 0 ? (double)qs[j] * ((pe[j + 1] - pe[j]) / (pbk - pt)) / qm : 0.25;
      if (!found && cum >= 0.5) { jc = j; found = true; }
    }
  }
  if (blq) jc = 0;
#pragma unroll
  for (int j = 0; j < NSUB; j++) {
    const int s = k * NSUB + j;
    W(s, 10) = j == jc ? (float)tcl : 0.f;
    const fast qj = qm > 0 ? (fast)(q_k * (double)qs[j] / qm) : (fast)q_k;
    const fast x = qj / (1 - qj) * (fast)(air.m_air / 18.01528);
    W(s, 4) = (float)(x * uas[j]);
    W(s, 9) = (float)(x / (fast)0.04);
  }
#undef W
}

// A value that every lane holds alike, in a scalar register: the table rows a column reads are the same for all its
// g-points, so their base addresses cost scalar arithmetic only and each load's lane offset is g.
__device__ __forceinline__ int uni(int x) { return __builtin_amdgcn_readfirstlane(x); }
__device__ __forceinline__ float uni(float x) { return __int_as_float(uni(__float_as_int(x))); }
__device__ __forceinline__ double uni(double x) {
  return __hiloint2double(uni(__double2hiint(x)), uni(__double2loint(x)));
}

// A table row's base address, kept in scalar registers as it is: without this the compiler folds the tables' fixed
// offsets into per-lane addresses that it holds in registers over the whole kernel (two per table row and corner).
typedef const __attribute__((address_space(1))) float* tabp;
__device__ __forceinline__ tabp row_at(const float* tab, size_t off) {
  tabp p = (tabp)tab + off;
  asm("" : "+s"(p));
  return p;
}

// Pins a value computed here to this place: without it the compiler sinks the arithmetic to the value's use at the end
// of the column and keeps its operands, two to three times as many, in registers instead.
__device__ __forceinline__ void pin(fast& x) { asm volatile("" : "+v"(x)); }

// One float at a 32-bit byte offset beside a scalar base: no 64-bit lane address.
__device__ __forceinline__ float at(tabp p, unsigned o) {
  asm("" : "+v"(o));
  return *(tabp)((const __attribute__((address_space(1))) char*)p + o);
}
// The optical depth of one g-point (air.cu:2266-2271,2425-2437): per component k = exp of ln k bilinear in (log p, T),
// times its amount a[c]. load() asks for every corner of a sub-level's cell at once (o: the lane's byte offsets of the four
// corners in a component's table row), depth() uses them. (Loading a sub-level ahead instead was slower wherever its
// registers cost a wave per SIMD: the other waves hide the tables' latency better.)
template <int NCOMP>
struct Corners {
  float v[NCOMP][4];
  __device__ __forceinline__ void load(const float* logk, size_t cell, size_t cs, const unsigned (&o)[4]) {
#pragma unroll
    for (int c = 0; c < NCOMP; c++) {
      const tabp K = row_at(logk, cell + c * cs);
#pragma unroll
      for (int m = 0; m < 4; m++) v[c][m] = at(K, o[m]);
    }
  }
  // ln k is interpolated by its differences on the cell, which are small where ln k is not: by the corners' weights (with
  // log2 e in them, four operations for seven) each weight's rounding took its share of the whole of ln k, and the
  // longwave's error against 64 bits was 1.6% larger on average, 4.5% at most, over 24 sets of columns and tables; so it is
  // 1.0% smaller on average than with one depth at a time, never larger (lw_column at 40,962 x 7 x 256: 1.38 -> 1.44 ms).
  __device__ __forceinline__ fast depth(fast fp, fast ft, const fast* a) const {
    const fast fpt = fp * ft;
    fast tau = 0;
#pragma unroll
    for (int c = 0; c < NCOMP; c++) {
      const fast v00 = v[c][0], v10 = v[c][1], v01 = v[c][2], v11 = v[c][3];
      tau += a[c] * fexp(v00 + (v10 - v00) * fp + (v01 - v00) * ft + (v00 - v01 - v10 + v11) * fpt);
    }
    return fmax((fast)0, tau);
  }
  // The same with water's two tables blended by fh: each operation's rounding then as the layer optics' comment asks.
  __device__ __forceinline__ fast blend(fast fp, fast ft, const fast* u, fast fh) const {
    fast lk[NCOMP];
#pragma unroll
    for (int c = 0; c < NCOMP; c++) {
      const fast v00 = v[c][0], v10 = v[c][1], v01 = v[c][2], v11 = v[c][3];
      lk[c] = fexp(v00 + (v10 - v00) * fp + (v01 - v00) * ft + (v00 - v01 - v10 + v11) * fp * ft);
    }
    static_assert(NCOMP == 7, "the shortwave's components");
    return fmax((fast)0, u[0] * (lk[0] + (lk[1] - lk[0]) * fh) + u[1] * lk[2] + u[2] * lk[3] + u[3] * lk[4] +
                             u[4] * lk[5] + u[5] * lk[6]);
  }
};

// Per-g float values in LDS summed over the g-points: g-point m's values at red[m * S ..], S odd, so that a wave's writes
// fall on different banks and every value's address is the lane's own plus a constant (with rows g-points long, their
// run-time length cost a register per row for the addresses). Eight lanes per row, each adding every eighth g-point in
// FP64, then three exchanges: a fixed order, so results repeat bit for bit. Lane 0 of the eight gets the row's sum. slot(r):
// where row r's values are.
template <int ROWS, int S, class At, class F>
__device__ __forceinline__ void g_sums(const float* red, int NG, At&& slot, F&& put) {
  static_assert(S % 2 == 1 && ROWS <= S, "odd stride");
  const int part = (int)threadIdx.x & 7, nr = (int)blockDim.x >> 3;
  for (int r = (int)threadIdx.x >> 3; r < ROWS; r += nr) {
    const int at = slot(r);
    double v = 0;
    for (int m = part; m < NG; m += 8) v += (double)red[m * S + at];
#pragma unroll
    for (int o = 4; o >= 1; o >>= 1) v += __shfl_xor(v, o);
    if (part == 0) put(r, v);
  }
}

__device__ __forceinline__ int same(int r) { return r; }

// f(S), f(S - 1), .., f(0), each with its own constant.
template <int S, class F>
__device__ __forceinline__ void down_from(F&& f) {
  f(S);
  if constexpr (S > 0) down_from<S - 1>(f);
}

// The columns a block takes in turn: enough of them to share the block's set-up, few enough to leave several blocks per
// slot of the chip (256 CUs, about three blocks each) so that the last ones do not run alone.
static inline int cols_per_block(int N) {
  const int c = N / (256 * 3 * 4);
  return c < 1 ? 1 : c > 8 ? 8 : c;
}

// ---------------------------------------------------------------------------------------------------------------
// lw_column (air.cu:2231-2348): a block takes its columns in turn, one thread per g-point (block = NG rounded up to 64).
// One walk down the sub-levels does everything that costs: each sub-level's transmission t and its emission both ways,
// I' = I t + E down the walk at once, and the way up as the layer's affine maps (T, E) from its bottom to the three
// edges that results need, composed inside the layer (clear and cloudy chains blended by the cover, as the fluxes are).
// The way up is then two multiply-adds per edge. (Recomputing the emission on the way up, with the tables' rows
// addressed per lane, the pass took 3.74 ms at 40,962 x 7 x 256 in the mixed form.)
// ---------------------------------------------------------------------------------------------------------------
template <int L>
struct LwRows {
  static constexpr int NUP = 4 + 6 * L, NDN = 3 * L;
  // the sums of the way down before the way up, in the same LDS, where all of them at once would keep a CU from holding
  // three blocks (at 7 layers: 1.41 ms against 1.89 ms with two blocks)
  static constexpr bool SPLIT = (NUP + NDN) * NGMAX * 4 + 2600 > 160 * 1024 / 3;
  static constexpr int DN0 = SPLIT ? 0 : NUP, S = (SPLIT ? NUP : NUP + NDN) | 1;
};

template <int L>
__global__ void __launch_bounds__(NGMAX) k_lw_column(int N, int cpb, RadP P, isw_lw_tables t,
                                                      const float* __restrict__ sub, const double* __restrict__ Ts,
                                                      double* __restrict__ radf) {
  constexpr int NSS = NSUB * L, RW = L + 1, E0 = 3 * RW + 3;
  using R = LwRows<L>;
  extern __shared__ float red[];                       // R::S per g-point
  __shared__ fast sa[NSS][6], scl[NSS], sfp[NSS], sft[NSS], scia[NSS], sfc[L];   // (amounts; cloud; T share; CIA; cover)
  __shared__ fast spt[NSS + 1], spb[NSS];              // Planck table shares (the last: the surface's)
  __shared__ int so[NSS], sit[NSS], sjt[NSS + 1], sjb[NSS];
  const unsigned g = threadIdx.x, NG = t.NG, row = (unsigned)(t.NT * t.NG);
  const unsigned o4[4] = {4 * g, 4 * (g + row), 4 * (g + NG), 4 * (g + row + NG)};
  const size_t cs = (size_t)t.NP * t.NT * t.NG;
  const int i0 = xblock() * cpb, i1 = min(i0 + cpb, N);
  auto planck_at = [&](fast T, int& j) -> fast {
    const float y = fminf(fmaxf((float)(T - (fast)t.tp0), 0.f), (float)((fast)(t.NTP - 1) - (fast)1e-4f));
    j = (int)y;
    return (fast)y - (fast)j;
  };
  auto stage = [&](int i) {
    if (g < NSS) {
      const int s = g;
#define R_(v) sub[((size_t)s * NVP + (v)) * N + i]
      // lw_setup writes the positions inside the tables; clamped again here so that no input reads outside them
      const fast x = clampf_pos(R_(2), t.NP), y = clampf_pos(R_(3), t.NT);
      const int ip = (int)x, it = (int)y;
      so[s] = (ip * t.NT + it) * t.NG;
      sit[s] = it * t.NG;
      sft[s] = y - (fast)it;
      sfp[s] = x - (fast)ip;
      const fast u0 = R_(4), fh = R_(9), df = (fast)1.66;
      sa[s][0] = df * (u0 * (1 - fh));                 // (water's two tables blended by its share; diffusivity 1.66)
      sa[s][1] = df * (u0 * fh);
#pragma unroll
      for (int c = 1; c < 5; c++) sa[s][c + 1] = df * (fast)R_(4 + c);
      scl[s] = R_(10);
      if (s % NSUB == 0) sfc[s / NSUB] = R_(11);
      scia[s] = df * (fast)R_(14);
      int j;
      spt[s] = planck_at(R_(0), j);
      sjt[s] = j * t.NG;
      spb[s] = planck_at(R_(1), j);
      sjb[s] = j * t.NG;
#undef R_
    }
    if (g == NSS) {                                    // (a block has 64 threads or more, NSS at most 32)
      int j;
      spt[NSS] = planck_at((fast)Ts[i], j);
      sjt[NSS] = j * t.NG;
    }
  };
  if (i0 >= i1) return;
  stage(i0);
  __syncthreads();
#define UP(r, v) red[g * R::S + (r)] = (float)(v)
#define DOWN(r, v) red[g * R::S + R::DN0 + (r)] = (float)(v)
  for (int i = i0; i < i1; i++) {
    const fast refl = P.lw_refl > 0 ? (fast)(1 - P.eps_s) : (fast)0, PIf = (fast)PI_;
    fast I = 0, Icl = 0;
    fast mT[L][3], mE[L][3], cT[L], cE[L];
    // what a sub-level reads from the tables: its gases' corners, the Planck rows of its two edges
    struct {
      Corners<6> k;
      float t0, t1, b0, b1;
    } row_s;
    auto load = [&](int s) {
      const tabp pt = row_at(t.planck, uni(sjt[s])), pb = row_at(t.planck, uni(sjb[s]));
      row_s.t0 = at(pt, o4[0]); row_s.t1 = at(pt, o4[2]);
      row_s.b0 = at(pb, o4[0]); row_s.b1 = at(pb, o4[2]);
      row_s.k.load(t.logk, (size_t)uni(so[s]), cs, o4);
    };
    if (g < NG) {
#pragma unroll
      for (int k = 0; k < L; k++) {
        const fast f = uni(sfc[k]);
        fast Ic = I, Id = I;
        fast tr[NSUB], eu[NSUB], tr2[NSUB], eu2[NSUB];
#pragma unroll
        for (int j = 0; j < NSUB; j++) {
          const int s = k * NSUB + j;
          __builtin_amdgcn_sched_barrier(0);           // (sub-level by sub-level, or the registers run out)
          load(s);
          fast x = row_s.k.depth(sfp[s], sft[s], sa[s]);          // (1.66 times the optical depth)
          if (t.cia) {
            const tabp C = row_at(t.cia, uni(sit[s]));
            x += scia[s] * ((fast)at(C, o4[0]) + ((fast)at(C, o4[2]) - (fast)at(C, o4[0])) * sft[s]);
          }
          // two-stream through the sub-level, the Planck radiance linear in optical depth, diffusivity 1.66
          // (air.cu:2123-2127): t = e^-x, E = B_far (1 - t) + (B_near - B_far) lin
          const fast Bt = row_s.t0 + (fast)(row_s.t1 - row_s.t0) * spt[s];
          const fast Bb = row_s.b0 + (fast)(row_s.b1 - row_s.b0) * spb[s];
          auto through = [&](fast y, fast& tt, fast& ed, fast& eup) {
            tt = fexp(-y);
            const fast om = 1 - tt, thin = y * ((fast)0.5 - y * (fast)(1.0 / 6.0)), thick = 1 - fquot(om, y);
            const fast lin = y > (fast)1e-3 ? thick : thin;
            ed = Bt * om + (Bb - Bt) * lin;
            eup = Bb * om + (Bt - Bb) * lin;
          };
          fast ed;
          through(x, tr[j], ed, eu[j]);
          Ic = Ic * tr[j] + ed;
          if (refl > 0) Icl = Icl * tr[j] + ed;
          if (f > 0) {
            tr2[j] = tr[j];
            eu2[j] = eu[j];
            fast ed2 = ed;
            const fast cl = uni(scl[s]);
            if (cl > 0) through(x + cl, tr2[j], ed2, eu2[j]);
            Id = Id * tr2[j] + ed2;
          }
          const fast mix = f > 0 ? (1 - f) * Ic + f * Id : Ic;
          if (j == 0) DOWN(3 * k + 1, PIf * mix);
          if (j == NSUB - 2) DOWN(3 * k + 2, PIf * mix);
          if (j == NSUB - 1) I = mix;
        }
        DOWN(3 * k, PIf * I);
        fast T1 = 1, E1 = 0, T2 = 1, E2 = 0;
#pragma unroll
        for (int j = NSUB - 1; j >= 0; j--) {
          E1 = E1 * tr[j] + eu[j];
          T1 *= tr[j];
          if (f > 0) {
            E2 = E2 * tr2[j] + eu2[j];
            T2 *= tr2[j];
          }
          const int e = j == NSUB - 1 ? 0 : j == 1 ? 1 : j == 0 ? 2 : -1;
          if (e >= 0) {
            mT[k][e] = f > 0 ? (1 - f) * T1 + f * T2 : T1;
            mE[k][e] = f > 0 ? (1 - f) * E1 + f * E2 : E1;
          }
        }
        cT[k] = T1;
        cE[k] = E1;
#pragma unroll
        for (int e = 0; e < 3; e++) { pin(mT[k][e]); pin(mE[k][e]); }
        pin(cT[k]); pin(cE[k]); pin(I); pin(Icl);
      }
    }
    // the sums of the way down: radf's rows RW + k + 1 and the layers' inner edges
    auto sums_down = [&]() {
      g_sums<R::NDN, R::S>(red + R::DN0, (int)NG, same, [&](int q, double w) {
        const int k = q / 3, m = q - 3 * k;
        radf[(size_t)(m == 0 ? RW + k + 1 : E0 + 6 * k + (m == 1 ? 1 : 4)) * N + i] = w;
      });
    };
    if constexpr (R::SPLIT) {
      __syncthreads();
      sums_down();
      __syncthreads();
    }
    if (g < NG) {
      const tabp ps = row_at(t.planck, uni(sjt[NSS]));
      const float b0 = at(ps, o4[0]), b1 = at(ps, o4[2]);
      const fast Bs = b0 + (fast)(b1 - b0) * spt[NSS];
      fast Iu = refl * I, trs = Bs, Iuc = refl * Icl, trc = Bs;       // (the transmissions weighted by Bs)
      UP(0, PIf * Iu);
#pragma unroll
      for (int k = L - 1; k >= 0; k--) {
        UP(4 + 6 * k, PIf * (Iu * mT[k][0] + mE[k][0]));
        UP(4 + 6 * k + 1, trs * mT[k][0]);
        UP(4 + 6 * k + 2, PIf * (Iu * mT[k][1] + mE[k][1]));
        UP(4 + 6 * k + 3, trs * mT[k][1]);
        Iu = Iu * mT[k][2] + mE[k][2];
        trs *= mT[k][2];
        Iuc = Iuc * cT[k] + cE[k];
        trc *= cT[k];
        UP(4 + 6 * k + 4, PIf * Iu);
        UP(4 + 6 * k + 5, trs);
      }
      UP(1, PIf * Iuc);
      UP(2, trc);
      UP(3, Bs);
    }
    __syncthreads();
    if constexpr (!R::SPLIT) sums_down();
    {
      // the surface's Planck sum (each wave by itself), then the rows, the transmissions over it
      double bsum = 0;
      for (int m = (int)threadIdx.x & 63; m < (int)NG; m += 64) bsum += (double)red[m * R::S + 3];
#pragma unroll
      for (int o = 32; o >= 1; o >>= 1) bsum += __shfl_xor(bsum, o);
      g_sums<R::NUP, R::S>(red, (int)NG, same, [&](int q, double w) {
        int r;
        bool over = false;
        if (q < 4) {
          r = q == 0 ? L : 3 * RW + q - 1;
          over = q == 2;
        } else {
          const int k = (q - 4) / 6, m = q - 4 - 6 * k;
          r = m == 0 ? E0 + 6 * k + 3 : m == 1 ? E0 + 6 * k + 5 : m == 2 ? E0 + 6 * k : m == 3 ? E0 + 6 * k + 2
              : m == 4 ? k : 2 * RW + k;
          over = m & 1;
        }
        radf[(size_t)r * N + i] = over ? w / bsum : w;
        if (q == 3) {
          radf[(size_t)RW * N + i] = 0.0;              // (no light from above)
          radf[(size_t)(2 * RW + L) * N + i] = bsum / bsum;
        }
      });
    }
    if (i + 1 < i1) stage(i + 1);
    __syncthreads();
  }
#undef UP
#undef DOWN
}

// ---------------------------------------------------------------------------------------------------------------
// sw_layer (air.cu:2358-2382): Delta-Eddington reflectance and transmittance of one homogeneous sub-level, for diffuse
// light (Rd, Td) and for the sun's beam at cosine mu0 (Rs, Ts; Tdd the beam's direct transmission).
// ---------------------------------------------------------------------------------------------------------------
__device__ __forceinline__ void sw_layer(fast tau, fast ssa, fast g, fast mu0, fast& Rd, fast& Td, fast& Rs, fast& Ts,
                                         fast& Tdd) {
  const fast f = g * g;
  tau = (1 - ssa * f) * tau;
  ssa = fdiv((1 - f) * ssa, 1 - ssa * f);
  g = fdiv(g - f, 1 - f);
  const fast g1 = (7 - ssa * (4 + 3 * g)) / 4, g2 = -(1 - ssa * (4 - 3 * g)) / 4, g3 = (2 - 3 * g * mu0) / 4;
  const fast g4 = 1 - g3;
  const fast a1 = g1 * g4 + g2 * g3, a2 = g1 * g3 + g2 * g4;
  const fast k = fsqrt(fmax((g1 - g2) * (g1 + g2), (fast)1e-12));
  const fast e = fexp(-k * tau), e2 = e * e, k2e = 2 * k * e;
  fast rf = fdiv(1, k + g1 + (k - g1) * e2);
  Rd = g2 * (1 - e2) * rf;
  Td = k2e * rf;
  Tdd = fexp(fdiv(-tau, mu0));
  const fast km = k * mu0;
  fast om = 1 - km * km;
  if (fabs(om) < (fast)1e-3) om = om < 0 ? (fast)-1e-3 : (fast)1e-3;
  rf = fdiv(ssa * rf, om);
  Rs = rf * ((1 - km) * (a2 + k * g3) - (1 + km) * (a2 - k * g3) * e2 - k2e * (g3 - a2 * mu0) * Tdd);
  Ts = rf * (k2e * (g4 + a1 * mu0) - Tdd * ((1 + km) * (a1 + k * g4) - (1 - km) * (a1 - k * g4) * e2));
  Rs = fmin(fmax(Rs, (fast)0), 1 - Tdd);
  Ts = fmin(fmax(Ts, (fast)0), 1 - Tdd - Rs);
}

// The sun's longitude at time t (air.cu:174-185): Kepler's equation by five Newton steps (circular orbit: uniform).
__device__ double sun_lon(double t, const RadP& P) {
  if (!(P.ecc > 0)) return 2 * PI_ * t / P.year_s;
  const double e = P.ecc, nu0 = -P.lam_peri;
  const double E0 = 2 * atan(sqrt((1 - e) / (1 + e)) * tan(nu0 / 2));
  const double M = E0 - e * sin(E0) + 2 * PI_ * t / P.year_s;
  double E = M;
  for (int it = 0; it < 5; it++) E -= (E - e * sin(E) - M) / (1 - e * cos(E));
  return 2 * atan2(sqrt(1 + e) * sin(E / 2), sqrt(1 - e) * cos(E / 2)) + P.lam_peri;
}

// ---------------------------------------------------------------------------------------------------------------
// sw_column (air.cu:2384-2511): a block takes its columns in turn, one thread per g-point. One walk up the sub-levels
// does everything that costs (table look-ups and optics once each): the clear and all-sky albedos below every edge, and
// each sub-level's map of the light going down through it, Fdir' = d Fdir, Fdif' = a Fdif + c Fdir, with what lies
// below already known. Only the nets at three edges per layer are wanted, so a layer keeps three maps (the second and
// third sub-level's composed) with the albedos below each, 15 values per layer, and the way down is five multiply-adds
// per edge. What bounds it then is the vector ALU: about 240 instructions and 17 transcendentals per sub-level. (Evaluating
// look-ups and optics again on the way down, with the tables' rows addressed per lane and the sun's position found anew by
// one lane per column, the pass took 6.89 ms at 40,962 x 7 x 224 in the mixed form.) The sun's direction at the four times of the interval is found once per block, one lane each.
// ---------------------------------------------------------------------------------------------------------------
template <int L>
__global__ void __launch_bounds__(NGMAX, ISW_FORM_MIXED ? 3 : 1) k_sw_column(int N, int cpb, RadP P, isw_sw_tables t, isw_air air,
                                                      const float* __restrict__ sub, int mode,
                                                      const double* __restrict__ tnow, double interval,
                                                      const double* __restrict__ pos, const double* __restrict__ alb,
                                                      const double* __restrict__ cloudo, double* __restrict__ swf) {
  constexpr int NSS = NSUB * L, S = 6 * L + 1;
  // The mixed form keeps the edges' albedos in the LDS slots that the sums use once they are spent, from four layers on:
  // three waves per SIMD instead of two (15% at 7 layers; three layers fit anyway and lost 5% to it).
  constexpr bool IN_LDS = ISW_FORM_MIXED && L >= 4;
  extern __shared__ float red[];                       // S per g-point
  __shared__ fast su[NSS][6], sfh[NSS], sfp[NSS], sr[NSS], sh[NSS], stc[NSS], sfc[NSS], sli[NSS], sft[NSS], scia[NSS];
  __shared__ int so[NSS], sit[NSS];
  __shared__ fast smu, salb;
  __shared__ double sdir[4][3];                        // the sun's direction over the interval
  const unsigned g = threadIdx.x, NG = t.NG, row = (unsigned)(t.NT * t.NG);
  const unsigned o4[4] = {4 * g, 4 * (g + row), 4 * (g + NG), 4 * (g + row + NG)};
  const size_t cs = (size_t)t.NP * t.NT * t.NG;
  const int i0 = xblock() * cpb, i1 = min(i0 + cpb, N);
  if (mode == 0 && g < 4) {
    const double tt = tnow[0] + (g + 0.5) * interval / 4;
    const double ang = sun_lon(tt, P), dec = asin(sin(P.tilt) * sin(ang));
    const double rot = 2 * PI_ * fmod(tt, P.day_s) / P.day_s;
    sdir[g][0] = cos(dec) * cos(-rot);
    sdir[g][1] = cos(dec) * sin(-rot);
    sdir[g][2] = sin(dec);
  }
  auto stage = [&](int i) {
    if (g < NSS) {
      const int s = g, k = s / NSUB;
#define R_(v) sub[((size_t)s * NVP + (v)) * N + i]
      // (positions clamped to this table's axes: the same values for lw_setup's sub-levels when the tables share their
      // pressure axis, and no read outside the table for any input)
      const fast x = clampf_pos(R_(2), t.NP);
      const fast y = fmaxf(fminf((fast)R_(3) * (fast)t.yscale, (fast)(t.NT - 1) - 1e-4f), 0.f);
      const int ip = (int)x, it = (int)y;
      so[s] = (ip * t.NT + it) * t.NG;
      sit[s] = it * t.NG;
      sft[s] = y - (fast)it;
      sfp[s] = x - (fast)ip;
#pragma unroll
      for (int c = 0; c < 5; c++) su[s][c] = R_(4 + c);
      su[s][5] = (fast)air.o2 * R_(12);
      sfh[s] = R_(9);
      sr[s] = R_(12);
      sh[s] = R_(13);
      scia[s] = R_(14);
      const bool cl = R_(10) > 0 && cloudo;
      sfc[s] = cl ? (fast)cloudo[(size_t)k * N + i] : (fast)0;
      stc[s] = cl ? (fast)(t.inhom * cloudo[(size_t)(2 * L + 3 + k) * N + i]) : (fast)0;
      sli[s] = cl && t.cssa_i ? (fast)cloudo[(size_t)(3 * L + 3 + k) * N + i] : (fast)1;
#undef R_
    }
    if (g == blockDim.x - 1) {                         // the sun: the mean of its cosine over the interval's daylight
      fast m = 0.5;
      if (mode == 0) {
        fast sum = 0;
        int lit = 0;
        for (int j = 0; j < 4; j++) {
          const double cz = pos[3 * (size_t)i] * sdir[j][0] + pos[3 * (size_t)i + 1] * sdir[j][1] +
                            pos[3 * (size_t)i + 2] * sdir[j][2];
          if (cz > 0) {
            sum += (fast)cz;
            lit++;
          }
        }
        m = lit ? sum / lit : (fast)0.05;
      }
      smu = fmax(m, (fast)0.02);
      salb = (fast)alb[i];
    }
  };
  if (i0 >= i1) return;
  __syncthreads();                                     // (the sun's directions)
  stage(i0);
  __syncthreads();
  // (volatile: else the kept albedos stay in registers too)
  volatile __attribute__((address_space(3))) float* slot = (volatile __attribute__((address_space(3))) float*)(red + g * S);
  const unsigned gc = g < NG ? g : 0;
  const fast cssa = t.cssa[gc], ray = t.ray[gc], hzf = t.hzf[gc], wg = t.sun[gc];
  const fast cssa_i = t.cssa_i ? (fast)t.cssa_i[gc] : (fast)0, g_i = t.g_i ? (fast)t.g_i[gc] : (fast)0;
  for (int i = i0; i < i1; i++) {
    if (g < NG) {
      const fast mu0 = smu;
      fast Ad = salb, As = Ad, cAd = Ad, cAs = Ad;
      // per layer and wanted edge (below the first, the third and the last sub-level): the map down to it, 1 - Ad and
      // 1 - As there
      fast md[L][3], ma[L][3], mc[L][3], nd[L][3], ns[L][3];
      auto walk = [&](int s) __attribute__((always_inline)) {
        __builtin_amdgcn_sched_barrier(0);             // (sub-level by sub-level, or the registers run out)
        Corners<7> row_s;
        row_s.load(t.logk, (size_t)uni(so[s]), cs, o4);
        fast tg = row_s.blend(sfp[s], sft[s], su[s], sfh[s]);
        if (t.cia) {
          const tabp C = row_at(t.cia, uni(sit[s]));
          tg += scia[s] * ((fast)at(C, o4[0]) + ((fast)at(C, o4[2]) - (fast)at(C, o4[0])) * sft[s]);
        }
        // the sub-level's optics: molecules, haze and gas (air.cu:2440-2458), with the cloud's share mixed in
        const fast trs = ray * sr[s] * (fast)air.ray, ths = (fast)t.tau550 * hzf * sh[s];
        const fast tt = tg + trs + ths, sc = trs + (fast)t.hssa * ths;
        const fast ssa = tt > TINY ? fmin(fdiv(sc, tt), (fast)(1 - 1e-6)) : (fast)0;
        const fast ga = sc > TINY ? fdiv((fast)t.hg * (fast)t.hssa * ths, sc) : (fast)0;
        fast cRd, cTd, cRs, cTs, cTdd;
        sw_layer(tt, ssa, ga, mu0, cRd, cTd, cRs, cTs, cTdd);
        fast rd = cRd, td = cTd, rs = cRs, ts = cTs, tdd = cTdd;
        const fast f = uni(sfc[s]), tc = uni(stc[s]);
        if (f > 0 && tc > 0) {
          const fast t2 = tt + tc;
          fast cw = cssa, cg = (fast)P.cloud_g;
          if (t.cssa_i) {
            const fast sl = sli[s], wl = sl * cssa, wi = (1 - sl) * cssa_i;
            cw = wl + wi;
            cg = cw > TINY ? fdiv(wl * (fast)P.cloud_g + wi * g_i, cw) : cg;
          }
          const fast sc2 = sc + cw * tc;
          const fast g2 = sc2 > TINY ? fdiv(ga * sc + cg * cw * tc, sc2) : (fast)0;
          fast r1, t1, r2, t3, d1;
          sw_layer(t2, t2 > TINY ? fmin(fdiv(sc2, t2), (fast)(1 - 1e-6)) : (fast)0, g2, mu0, r1, t1, r2, t3, d1);
          rd = (1 - f) * cRd + f * r1;
          td = (1 - f) * cTd + f * t1;
          rs = (1 - f) * cRs + f * r2;
          ts = (1 - f) * cTs + f * t3;
          tdd = (1 - f) * cTdd + f * d1;
        }
        {
          const fast cden = fquot(1, 1 - cAd * cRd);
          const fast n = cRd + cTd * cTd * cAd * cden;
          cAs = cRs + (cTdd * cAs + cTs * cAd) * cTd * cden;
          cAd = n;
        }
        const fast den = fquot(1, 1 - Ad * rd), ta = td * den;
        const fast cm = (rd * As * tdd + ts) * den;
        const int k = s / NSUB, j = s % NSUB;
        const int e = j == 0 ? 0 : j == NSUB - 1 ? 2 : 1;
        if (e == 1 && j == 1) {                        // composed with the sub-level below it
          mc[k][1] = ma[k][1] * cm + mc[k][1] * tdd;
          ma[k][1] *= ta;
          md[k][1] *= tdd;
          pin(mc[k][1]); pin(ma[k][1]); pin(md[k][1]);
        } else {
          md[k][e] = tdd;
          ma[k][e] = ta;
          mc[k][e] = cm;
          pin(mc[k][e]); pin(ma[k][e]); pin(md[k][e]);
          if constexpr (IN_LDS) {
            slot[2 * (3 * k + e)] = 1 - Ad;
            slot[2 * (3 * k + e) + 1] = 1 - As;
          } else {
            nd[k][e] = 1 - Ad;
            ns[k][e] = 1 - As;
            pin(nd[k][e]); pin(ns[k][e]);
          }
        }
        const fast nAd = rd + td * Ad * ta;
        As = rs + (tdd * As + ts * Ad) * ta;
        Ad = nAd;
        pin(As); pin(Ad); pin(cAs); pin(cAd);
      };
      // (the mixed form's walk is unrolled by recursion at any length, the loop's own limit on size is below it; the FP64
      // form's as far as the compiler goes, the rest of the maps then in scratch: 1.45 ms at 9,000 x 7 against 1.6 ms)
      if constexpr (ISW_FORM_MIXED) {
        down_from<NSS - 1>(walk);
      } else {
#pragma unroll
        for (int s = NSS - 1; s >= 0; s--) walk(s);
      }
      // top down: the nets at the edges, each layer's absorption, its top and bottom sub-level's, the surface's
      fast Fdir = 1, Fdif = 0, net = 1 - As;
#pragma unroll
      for (int k = 0; k < L; k++) {
        const fast top = net;
#pragma unroll
        for (int e = 0; e < 3; e++) {
          Fdif = ma[k][e] * Fdif + mc[k][e] * Fdir;
          Fdir *= md[k][e];
          const int q = 2 * (3 * k + e);
          if constexpr (IN_LDS) {
            nd[k][e] = slot[q];
            ns[k][e] = slot[q + 1];
          }
          const fast n2 = Fdir * ns[k][e] + Fdif * nd[k][e];
          if (e != 1) slot[q] = (float)(wg * (net - n2));
          net = n2;
        }
        slot[2 * (3 * k + 2) + 1] = (float)(wg * (top - net));
      }
      slot[2] = (float)(wg * net);
      slot[3] = (float)(wg * cAs);
    }
    __syncthreads();
    // the rows' slots: the layers' absorption, top and bottom sub-level's, then the surface's two
    g_sums<3 * L + 2, S>(red, (int)NG, [](int r) {
      if (r >= 3 * L) return r - 3 * L + 2;
      const int k = r / 3, m = r - 3 * k;
      return 6 * k + (m == 0 ? 5 : m == 1 ? 0 : 4);
    }, [&](int r, double v) {
      const int k = r / 3, m = r - 3 * k;
      const int row = r >= 3 * L ? L + r - 3 * L : m == 0 ? k : L + 1 + 2 * k + m;
      swf[(size_t)row * N + i] = v;
    });
    if (i + 1 < i1) stage(i + 1);
    __syncthreads();
  }
}

// ---------------------------------------------------------------------------------------------------------------
// Host side: one stream, the layer count picks the instantiation.
// ---------------------------------------------------------------------------------------------------------------
static inline int ngpad(int NG) { return (NG + 63) / 64 * 64; }

#define ISW_BY_L(CALL)                                                                                   \
  switch (L) {                                                                                           \
    case 1: { CALL(1); } break;                                                                              \
    case 2: { CALL(2); } break;                                                                          \
    case 3: { CALL(3); } break;                                                                          \
    case 4: { CALL(4); } break;                                                                          \
    case 5: { CALL(5); } break;                                                                          \
    case 6: { CALL(6); } break;                                                                          \
    case 7: { CALL(7); } break;                                                                          \
    case 8: { CALL(8); } break;                                                                          \
    default: return ISW_EBADARG;                                                                         \
  }

int lw_setup(int N, int L, const double* par, const isw_lw_tables* t, const isw_air* air, double co2, double n2o,
             double ch4, const double* gx, const double* mu, const double* theta, const double* qv,
             const double* cloudo, double hs, int tmode, float* sub, hipStream_t st) {
  const RadP P = make_radp(par);
  const dim3 grid((unsigned)((N + 63) / 64), (unsigned)L), block(64);
  const double bytes = (double)L * N * 8 * (2 + (qv ? 1 : 0) + (gx ? 3 : 0)) + (cloudo ? 2.0 * L * N * 8 : 0) +
                       (double)NSUB * L * NVP * N * 4;
#define CALL(LL)                                                                                              \
  ISW_LAUNCH("lw_setup", bytes, k_lw_setup<LL>, grid, block, N, P, *t, *air, co2, n2o, ch4, gx, mu, theta, qv, \
             cloudo, hs, tmode, sub)
  ISW_BY_L(CALL)
#undef CALL
  return (int)hipGetLastError();
}

int lw_column(int N, int L, const double* par, const isw_lw_tables* t, const float* sub, const double* Ts,
              double* radf, hipStream_t st) {
  const RadP P = make_radp(par);
  const int ngp = ngpad(t->NG), rows = 3 * (L + 1) + 3 + 6 * L;
  const int cpb = cols_per_block(N);
  const unsigned nb = (unsigned)((N + cpb - 1) / cpb);
  const double bytes = (double)NSUB * L * NVP * N * 4 + (double)N * 8 + (double)rows * N * 8 +
                       (double)t->NC * t->NP * t->NT * t->NG * 4 + (double)t->NTP * t->NG * 4;
  // (at most 54 KB of LDS, at eight layers)
#define CALL(LL)                                                                                              \
  const size_t shm = (size_t)LwRows<LL>::S * ngp * sizeof(float);                                                    \
  ISW_LAUNCH_SHM("lw_column", bytes, k_lw_column<LL>, dim3(nb), dim3((unsigned)ngp), shm, N, cpb, P, *t, sub, Ts, \
                 radf)
  ISW_BY_L(CALL)
#undef CALL
  return (int)hipGetLastError();
}

int sw_column(int N, int L, const double* par, const isw_sw_tables* t, const isw_air* air, const float* sub, int mode,
              const double* tnow, double interval, const double* pos, const double* alb, const double* cloudo,
              double* swf, hipStream_t st) {
  const RadP P = make_radp(par);
  const int ngp = ngpad(t->NG), rows = 3 * L + 2;
  const size_t shm = (size_t)(6 * L + 1) * ngp * sizeof(float);
  const int cpb = cols_per_block(N);
  const unsigned nb = (unsigned)((N + cpb - 1) / cpb);
  const double bytes = (double)NSUB * L * NVP * N * 4 + (double)N * 8 * (1 + (mode == 0 ? 3 : 0)) +
                       (cloudo ? 3.0 * L * N * 8 : 0) + (double)rows * N * 8 + (double)t->NC * t->NP * t->NT * t->NG * 4;
#define CALL(LL)                                                                                              \
  ISW_LAUNCH_SHM("sw_column", bytes, k_sw_column<LL>, dim3(nb), dim3((unsigned)ngp), shm, N, cpb, P, *t, *air, sub, \
                 mode, tnow, interval, pos, alb, cloudo, swf)
  ISW_BY_L(CALL)
#undef CALL
  return (int)hipGetLastError();
}

}  // namespace NS
