// ts_quad.hpp - the frequency integrals of the spin temperature's shell tables
// on the device (ComputeTs.c:505-625; XRayHeatingFunctions.c:238-375, :673-1220).
//
// A snapshot needs, per shell, the frequency at which the X-ray optical depth
// tau_X reaches 1 (Brent's root over QAG integrals) and 3 x 14 adaptive QAG
// integrals over frequency.  On 16 host threads that is 2.5-3 ms, more than
// the device needs for the whole step up to 192^3, and the adjoint builds the
// tables five times.  A 61-point Gauss-Kronrod rule fits a wave of 64 lanes:
// here one workgroup of two waves is one integral (or one root), a wave's lanes
// the nodes of a rule, its sums butterflies; the waves take the two halves of a
// bisected interval, and the bookkeeping is uniform.  All integrals of all
// shells (and of several builds) run at once: about 9000 rules of some 4000
// vector instructions, 60 us of the whole chip.  The time is the longest chain,
// 60 rules, two at a time: 302 us (434 with one wave), after 121 us of roots,
// beside the shells' passes.  The 128^3 step went from 3.47 to 1.14 ms with one
// wave per integral (0.94 to 0.79 with the second, the shells grouped), a 192^3
// training step from 27.9 to 19.5.
//
// The algorithms, tolerances and interval order are ts_tables.c's (the host
// build, which mrx_ts_snapshot_tables still serves); sums run over the wave in
// another order and exp, log, pow and atan are the device's, so the tables
// agree to rounding (1e-11 is asserted of the step's averages, which are
// linear in them).
#pragma once
#include <hip/hip_runtime.h>

#include <cfloat>

#include "gk61_rule.h"
#include "ts_tables.h"

namespace mrx {

// The x_int tables, the quadrature rule by lane, and the cosmology; uploaded
// once per table set.
struct TsQuadDev {
  double node[64], wk[64], wg[64];  // lane's abscissa on [-1, 1], Kronrod and Gauss weights (0 past lane 60)
  double f_H, f_He, N_b0, hubble_h, omega_m, omega_l, ion_eff;
  float XH[MRX_X_INT_NXHII];
  float E[MRX_X_INT_NENERGY];
  float fheat[MRX_X_INT_NXHII][MRX_X_INT_NENERGY], nLya[MRX_X_INT_NXHII][MRX_X_INT_NENERGY],
    nHI[MRX_X_INT_NXHII][MRX_X_INT_NENERGY], nHeI[MRX_X_INT_NXHII][MRX_X_INT_NENERGY],
    nHeII[MRX_X_INT_NXHII][MRX_X_INT_NENERGY];
};

constexpr int kQuadBuilds = 4;  // table builds of one launch (the adjoint's central differences)

// One snapshot's builds: they differ in the two grid means.
struct TsQuadArgs {
  int nsteps, nbuild;
  int first_snapshot;      // no earlier collapse fraction to interpolate from
  double zp, Z0, Z1, F0;   // redshifts of the previous and this snapshot, the previous collapse fraction
  double F1[kQuadBuilds];  // collapse fraction
  double x_e[kQuadBuilds];
  double nu_min, nu_max, spec_index;  // NuXrayGalThreshold, NuXrayMax [Hz]
  double zpp[MRX_TS_MAX_STEPS];
};

// Output of build b: nu_lower[shell], then the raw integrals [heat, ion, lya][x][shell].
constexpr int kQuadOut = MRX_TS_MAX_STEPS * (1 + 3 * MRX_X_INT_NXHII);
__host__ __device__ constexpr int quad_index(int flag, int x, int ct)
{
  return MRX_TS_MAX_STEPS * (1 + flag * MRX_X_INT_NXHII + x) + ct;
}

namespace quad {

// the plain functions, not the dual numbers' overloads of this namespace's parent
using ::atan;
using ::exp;
using ::fabs;
using ::log;
using ::pow;
using ::sqrt;

#pragma clang fp contract(off)

constexpr double kSpeedOfLight = 2.9979e10;
constexpr double kPlanckCgs = 6.6262e-27;
constexpr double kHubbleCgs = 3.2407789e-18;
constexpr double kNuOverEv = 1.60217646e-12 / kPlanckCgs;
constexpr double kNuHI = 13.60 * kNuOverEv;
constexpr double kNuHeI = 24.59 * kNuOverEv;
constexpr double kNuHeII = kNuHI * 4;
constexpr double kPi = 3.14159265358979323846;
constexpr int kMaxIntervals = 1000;

__device__ __forceinline__ double wave_add(double v)
{
#pragma unroll
  for (int m = 32; m > 0; m >>= 1) v += __shfl_xor(v, m, 64);
  return v;
}

// hydrogen-like cross section of threshold nu0 and charge Z
__device__ __forceinline__ double xsec_H(double nu, double nu0, double Z)
{
  if (nu < nu0) return 0;
  const double eps = sqrt(nu / nu0 - 1), r = nu0 / nu, r2 = r * r;
  return 6.3e-18 / Z / Z * (r2 * r2) * exp(4 - (4 * atan(eps) / eps)) / (1 - exp(-2 * kPi / eps));
}

__device__ __forceinline__ double xsec_HeI(double nu)
{
  if (nu < kNuHeI) return 0;
  const double x = nu / kNuOverEv / 13.61 - 0.4434;
  const double y = sqrt(x * x + 2.136 * 2.136);
  return 9.492e-16 * ((x - 1) * (x - 1) + 2.039 * 2.039) * pow(y, (0.5 * 3.188 - 5.5)) *
         pow(1.0 + sqrt(y / 1.469), -3.188);
}

// The interval lists of one integral (a workgroup of two waves), and the two
// halves' rules on their way from wave to wave.
struct Lists {
  double a[kMaxIntervals], b[kMaxIntervals], r[kMaxIntervals], e[kMaxIntervals];
  double half_r[2], half_e[2], half_asc[2];
};

struct Rule {
  double x, wk, wg;  // this lane's
};

// 61-point Gauss-Kronrod rule on [a, b], a node per lane
template <class F>
__device__ __forceinline__ double gk61(const F& f, const Rule& q, double a, double b, double& err, double& res_abs,
                                       double& res_asc)
{
  const double center = 0.5 * (a + b), half = 0.5 * (b - a), abs_half = fabs(half);
  const bool on = (threadIdx.x & 63) < 61;
  const double v = on ? f(center + half * q.x) : 0.0;
  double res_k = q.wk * v, res_g = q.wg * v;
  res_abs = q.wk * fabs(v);
#pragma unroll
  for (int m = 32; m > 0; m >>= 1) {
    res_k += __shfl_xor(res_k, m, 64);
    res_g += __shfl_xor(res_g, m, 64);
    res_abs += __shfl_xor(res_abs, m, 64);
  }
  const double mean = res_k * 0.5;
  res_asc = wave_add(on ? q.wk * fabs(v - mean) : 0.0);
  err = fabs((res_k - res_g) * half);
  res_abs *= abs_half;
  res_asc *= abs_half;
  if (res_asc != 0 && err != 0) {
    const double s = 200 * err / res_asc, scale = s * sqrt(s);
    err = (scale < 1) ? res_asc * scale : res_asc;
  }
  if (res_abs > DBL_MIN / (50 * DBL_EPSILON)) {
    const double min_err = 50 * DBL_EPSILON * res_abs;
    if (min_err > err) err = min_err;
  }
  return res_k * half;
}

// QAG: bisects the interval with the largest error until the summed error is
// below epsrel |result|; each of the workgroup's two waves takes the rule of one
// half.  Uniform over the workgroup; at most kMaxIntervals intervals.
template <class F>
__device__ double qag61(const F& f, const Rule& q, Lists& l, double a, double b, double epsrel)
{
  const int lane = threadIdx.x & 63;
  double resabs, resasc, e0;
  const double r0 = gk61(f, q, a, b, e0, resabs, resasc);
  double tolerance = epsrel * fabs(r0);
  const double round_off = 50 * DBL_EPSILON * resabs;
  if ((e0 <= round_off && e0 > tolerance) || (e0 <= tolerance && e0 != resasc) || e0 == 0.0) return r0;
  int n = 1;
  __syncthreads();  // the last integral's reads of the lists
  if (threadIdx.x == 0) {
    l.a[0] = a;
    l.b[0] = b;
    l.r[0] = r0;
    l.e[0] = e0;
  }
  __syncthreads();
  double area = r0, errsum = e0;
  int roundoff1 = 0, roundoff2 = 0;
  for (int iteration = 1; iteration < kMaxIntervals; iteration++) {
    // the first interval of largest error
    int k = 0;
    double best = -1.0;
    for (int i = lane; i < n; i += 64)
      if (l.e[i] > best) {
        best = l.e[i];
        k = i;
      }
#pragma unroll
    for (int m = 32; m > 0; m >>= 1) {
      const double eo = __shfl_xor(best, m, 64);
      const int ko = __shfl_xor(k, m, 64);
      if (eo > best || (eo == best && ko < k)) {
        best = eo;
        k = ko;
      }
    }
    k = __builtin_amdgcn_readfirstlane(k);
    const double a1 = l.a[k], b2 = l.b[k], b1 = 0.5 * (a1 + b2), a2 = b1, rk = l.r[k], ek = l.e[k];
    const int w = threadIdx.x >> 6;
    {
      double e, ra, rs;
      const double r = gk61(f, q, w ? a2 : a1, w ? b2 : b1, e, ra, rs);
      if (lane == 0) {
        l.half_r[w] = r;
        l.half_e[w] = e;
        l.half_asc[w] = rs;
      }
    }
    __syncthreads();
    const double r1 = l.half_r[0], r2 = l.half_r[1], e1 = l.half_e[0], e2 = l.half_e[1], rs1 = l.half_asc[0],
                 rs2 = l.half_asc[1];
    const double area12 = r1 + r2, error12 = e1 + e2;
    errsum += (error12 - ek);
    area += area12 - rk;
    if (rs1 != e1 && rs2 != e2) {
      const double delta = rk - area12;
      if (fabs(delta) <= 1.0e-5 * fabs(area12) && error12 >= 0.99 * ek) roundoff1++;
      if (iteration >= 10 && error12 > ek) roundoff2++;
    }
    tolerance = epsrel * fabs(area);
    if (threadIdx.x == 0) {  // every read of entry k and of the halves' slots' last values is past
      l.b[k] = b1;
      l.r[k] = r1;
      l.e[k] = e1;
      l.a[n] = a2;
      l.b[n] = b2;
      l.r[n] = r2;
      l.e[n] = e2;
    }
    __syncthreads();
    n++;
    if (errsum <= tolerance) break;
    if (roundoff1 >= 6 || roundoff2 >= 20) break;
    if (fmax(fabs(a1), fabs(b2)) <= (1 + 100 * DBL_EPSILON) * (fabs(a2) + 1000 * DBL_MIN)) break;
  }
  double result = 0;
  for (int i = 0; i < n; i++) result += l.r[i];
  return result;
}

__device__ __forceinline__ Rule lane_rule(const TsQuadDev& t)
{
  const int lane = threadIdx.x & 63;
  return {t.node[lane], t.wk[lane], t.wg[lane]};
}

// tau_X integrand (XRayHeatingFunctions.c:301-340)
struct TauX {
  const TsQuadDev& t;
  const TsQuadArgs& a;
  double nu_0, x_e, F1;
  __device__ double operator()(double zhat) const
  {
    const double om = sqrt(t.omega_l / t.omega_m), u = (double)(1 + (float)zhat), su = sqrt(u);
    const double x = om / (u * su), dxdz = om / (u * u * su) * (-3.0 / 2.0), s = sqrt(x * x + 1);
    const double const1 = 2 * sqrt(1 + t.omega_m / t.omega_l) / (3.0 * kHubbleCgs * t.hubble_h);
    const double dtdz = const1 * (dxdz * (1 + x / s)) / (x + s);
    const double zz = 1 + zhat, n = t.N_b0 * (zz * zz * zz), nuhat = nu_0 * zz;
    double fcoll = a.first_snapshot ? F1 : a.F0 + (zhat - a.Z0) * (F1 - a.F0) / (a.Z1 - a.Z0);
    if (fcoll < 0.0) fcoll = 0.0;
    double ff = (fcoll < 1e-20) ? 1 : 1 - (t.ion_eff * fcoll) / (1.0 - x_e);
    if (ff < 1e-4) ff = 1e-4;
    const double xs = t.f_H * (1 - x_e) * xsec_H(nuhat, kNuHI, 1) + t.f_He * (1 - x_e) * xsec_HeI(nuhat) +
                      t.f_He * x_e * xsec_H(nuhat, kNuHeII, 2);
    return kSpeedOfLight * dtdz * n * ff * xs;
  }
};

// Brent's root of f on [lo, hi] to relerr of the smaller end (ts_tables.c, mrx_ts_brent)
template <class F>
__device__ double brent(const F& f, double lo, double hi, double relerr, int max_iter)
{
  double a = lo, b = hi, fa = f(a), fb = f(b);
  double c = b, fc = fb, dd = b - a, e = dd;
  for (int it = 0; it < max_iter; it++) {
    if ((fb < 0 && fc < 0) || (fb > 0 && fc > 0)) {
      c = a;
      fc = fa;
      e = dd = b - a;
    }
    if (fabs(fc) < fabs(fb)) {
      a = b;
      b = c;
      c = a;
      fa = fb;
      fb = fc;
      fc = fa;
    }
    const double tol = 0.5 * DBL_EPSILON * fabs(b);
    const double m = 0.5 * (c - b);
    if (fb == 0 || fabs(m) <= tol) return b;
    if (fabs(e) < tol || fabs(fa) <= fabs(fb)) {
      dd = m;
      e = m;
    } else {
      double pp, q;
      const double s = fb / fa;
      if (a == c) {
        pp = 2 * m * s;
        q = 1 - s;
      } else {
        const double r = fb / fc;
        q = fa / fc;
        pp = s * (2 * m * q * (q - r) - (b - a) * (r - 1));
        q = (q - 1) * (r - 1) * (s - 1);
      }
      if (pp > 0)
        q = -q;
      else
        pp = -pp;
      if (2 * pp < fmin(3 * m * q - fabs(tol * q), fabs(e * q))) {
        e = dd;
        dd = pp / q;
      } else {
        dd = m;
        e = m;
      }
    }
    a = b;
    fa = fb;
    b += (fabs(dd) > tol) ? dd : (m > 0 ? +tol : -tol);
    fb = f(b);
    const double cb = ((fb < 0 && fc < 0) || (fb > 0 && fc > 0)) ? a : c;
    const double xl = fmin(b, cb), xu = fmax(b, cb);
    const double min_abs = (xl > 0 && xu > 0) || (xl < 0 && xu < 0) ? fmin(fabs(xl), fabs(xu)) : 0;
    if (fabs(xu - xl) < relerr * min_abs) return b;
  }
  return b;
}

// One x_int table at a node's clamped energy En in bin n_low, bilinear in float
__device__ __forceinline__ float xint_at(const TsQuadDev& t, const float (*tab)[MRX_X_INT_NENERGY], float En, int n,
                                         int m, float dx, float wx)
{
  const float dE = t.E[n + 1] - t.E[n], e = En - t.E[n];
  float lo = (tab[m][n + 1] - tab[m][n]) / dE;
  lo *= e;
  lo += tab[m][n];
  float hi = (tab[m + 1][n + 1] - tab[m + 1][n]) / dE;
  hi *= e;
  hi += tab[m + 1][n];
  float r = (hi - lo) / dx;
  r *= wx;
  r += lo;
  return r;
}

// The heating, ionisation and Ly-alpha integrands (XRayHeatingFunctions.c:673-760)
// at the table's x_e value of index xi
struct NuIntegrand {
  const TsQuadDev& t;
  double x_e, nu_min, pw;
  int flag, m;      // integrand; lower x_e row
  float dx, wx;     // row spacing; offset from the lower row
  __device__ NuIntegrand(const TsQuadDev& t_, const TsQuadArgs& a, int flag_, int xi)
      : t(t_), x_e(t_.XH[xi]), nu_min(a.nu_min), pw(-a.spec_index - 1), flag(flag_)
  {
    float x = t.XH[xi];
    if (x > t.XH[MRX_X_INT_NXHII - 1] * 0.999)
      x = (float)(t.XH[MRX_X_INT_NXHII - 1] * 0.999);
    else if (x < t.XH[0])
      x = (float)(1.001 * t.XH[0]);
    m = MRX_X_INT_NXHII - 1;
    while (x < t.XH[m]) m--;
    dx = t.XH[m + 1] - t.XH[m];
    wx = x - t.XH[m];
  }
  __device__ float tab(const float (*tb)[MRX_X_INT_NENERGY], float En, int n, float below) const
  {
    return (n < 0) ? below : xint_at(t, tb, En, n, m, dx, wx);
  }
  __device__ double operator()(double nu) const
  {
    const double th[3] = {kNuHI, kNuHeI, kNuHeII};
    const double w[3] = {t.f_H * (1 - x_e), t.f_He * (1 - x_e), t.f_He * x_e};
    const double xs[3] = {xsec_H(nu, kNuHI, 1), xsec_HeI(nu), xsec_H(nu, kNuHeII, 2)};
    double s = 0;
#pragma unroll
    for (int i = 0; i < 3; ++i) {
      float En = (float)((nu - th[i]) / kNuOverEv);
      int n;  // the energy's bin, -1 under the lowest
      const float Emax = t.E[MRX_X_INT_NENERGY - 1];
      if (En > 0.999 * Emax)
        En = (float)(Emax * 0.999);
      if (En < t.E[0])
        n = -1;
      else
        n = (En < 1008.88) ? (int)(log(En / 10.0) / 1.98026273e-2) : 232 + (int)(log(En / 1008.88) / 9.53101798e-2);
      if (flag == 0)
        s += tab(t.fheat, En, n, 1.0f) * kPlanckCgs * (nu - th[i]) * w[i] * xs[i];
      else if (flag == 1)
        s += (double)(tab(t.nHI, En, n, 0.0f) + tab(t.nHeI, En, n, 0.0f) + tab(t.nHeII, En, n, 0.0f) + 1) * w[i] *
             xs[i];
      else
        s += tab(t.nLya, En, n, 0.0f) * w[i] * xs[i];
    }
    return s * pow(nu / nu_min, pw);
  }
};

}  // namespace quad

// The shells' lower frequency limits (ComputeTs.c:560-580): one workgroup per shell
// (blockIdx.x) and build (blockIdx.y).
__global__ __launch_bounds__(128) void k_ts_nu_lower(const TsQuadDev* __restrict__ tg, TsQuadArgs a,
                                                   double* __restrict__ out)
{
  __shared__ quad::Lists lists;
  const TsQuadDev& t = *tg;
  const quad::Rule q = quad::lane_rule(t);
  const int ct = blockIdx.x, bd = blockIdx.y;
  const double x_e = a.x_e[bd], F1 = a.F1[bd];
  auto tau = [&](double nu) {
    const quad::TauX f{t, a, nu / (1 + a.zp), x_e, F1};
    return quad::qag61(f, q, lists, a.zpp[ct], a.zp, 0.005);
  };
  double nu;
  if (x_e > 0.9999)
    nu = -1;
  else if (tau(quad::kNuHeI) < 1)
    nu = quad::kNuHeI;
  else
    nu = quad::brent([&](double v) { return tau(v) - 1; }, quad::kNuHeI, 1e6 * quad::kNuOverEv, 0.02, 100);
  if (threadIdx.x == 0) out[(long)bd * kQuadOut + ct] = fmax(nu, a.nu_min);
}

// The frequency integrals: one workgroup per shell (blockIdx.x), integrand and x_e
// entry (blockIdx.y) and build (blockIdx.z), from the shell's lower limit.
__global__ __launch_bounds__(128) void k_ts_freq_integrals(const TsQuadDev* __restrict__ tg, TsQuadArgs a,
                                                         double* __restrict__ out)
{
  __shared__ quad::Lists lists;
  const TsQuadDev& t = *tg;
  const quad::Rule q = quad::lane_rule(t);
  const int ct = blockIdx.x, flag = blockIdx.y / MRX_X_INT_NXHII, x = blockIdx.y % MRX_X_INT_NXHII;
  out += (long)blockIdx.z * kQuadOut;
  const quad::NuIntegrand f(t, a, flag, x);
  const double r = quad::qag61(f, q, lists, out[ct], a.nu_max, 0.01);
  if (threadIdx.x == 0) out[quad_index(flag, x, ct)] = r;
}

#pragma clang fp contract(on)

}  // namespace mrx
