// Point-source sky component: per pixel
//   p_e = I(xi) * exp(alpha * dnu_e),  I = invgamma_prior(a, q)(xi),
//   alpha = alpha_mean + alpha_std * xi_alpha
// (jubik/sky_models.py:376-441, the SkyModel point sources added to the
// diffuse sky at 202; spectral_product_mf_point_sources.py:99-287,
// MultiFrequencyInvGammaSky, without spectral deviations).
//
// The inverse-gamma prior maps a standard normal xi to the inverse-gamma
// variable of shape a and scale q with the same quantile: I = q / y with
// Q(a, y) = Phi(xi), Q the regularised upper incomplete gamma function (if
// Y ~ Gamma(a, 1) then P(q / Y <= x) = Q(a, q / x)).  y is found by Halley
// steps in log y on log P(a, y) = log Phi(-xi) (small y) or log Q(a, y) =
// log Phi(xi) (large y), started for a >= 1 from the Wilson-Hilferty
// approximation of the Gamma quantile (whose standard normal quantile is
// exactly -xi) or, for small y, from the leading term y^a / Gamma(a + 1) of P,
// and for a < 1 from the two-branch approximation of Numerical Recipes (Press
// et al., 3rd edition 2007, section 6.2.1, which also takes Halley steps).  P and
// Q come from their power series (y < a + 1) or the continued fraction of Q
// (modified Lentz); the last steps are in double precision.  The derivative is
// closed-form:
//   d log I / d xi = phi(xi) Gamma(a) / (y^a e^-y).
#include <cmath>

#include "points.hpp"

namespace jubik {

namespace {

constexpr int PSNT = 256;

// Reciprocals 1 / (a + n) of the power series of P, and the constants of the
// shape a, formed once per launch on the host (they were two lgamma and one
// division per term of every Newton step of every pixel).
constexpr int kRecip = 96;
struct GammaShape {
  double a, lga, lga1, loga, sqrta;  // a, log Gamma(a), log Gamma(a + 1), log a, sqrt a
  double recip[kRecip];
};

GammaShape gamma_shape(double a) {
  GammaShape g;
  g.a = a;
  g.lga = std::lgamma(a);
  g.lga1 = std::lgamma(a + 1.0);
  g.loga = std::log(a);
  g.sqrta = std::sqrt(a);
  for (int n = 0; n < kRecip; ++n) g.recip[n] = 1.0 / (a + n);
  return g;
}

// log P(a, y) (want_p) or log Q(a, y), the regularised lower or upper
// incomplete gamma function, y = e^t > 0, in F = double, or in float for the
// first steps of the search below.
template <typename F>
__device__ __forceinline__ F log_pq(const GammaShape& g, F t, F y, bool want_p) {
  constexpr bool kDouble = sizeof(F) == 8;
  const F a = (F)g.a;
  const F lpre = a * t - y - (F)g.lga;  // log(y^a e^-y / Gamma(a))
  if (y < a + F(1)) {
    // P = pre * sum_n y^n / (a (a + 1) ... (a + n))
    constexpr F eps = kDouble ? F(1e-17) : F(1e-8);
    F term = (F)g.recip[0], sum = term;
    int n = 1;
    for (; n < kRecip; ++n) {
      term *= y * (F)g.recip[n];
      sum += term;
      if (term < sum * eps) break;
    }
    if (kDouble && n == kRecip)
      for (; n < 1000; ++n) {
        term *= y / (a + n);
        sum += term;
        if (term < sum * eps) break;
      }
    const F lp = lpre + log(sum);
    return want_p ? lp : log1p(-exp(lp));
  }
  // Q = pre / (y + 1 - a - 1 (1 - a) / (y + 3 - a - 2 (2 - a) / ...))
  constexpr F tiny = kDouble ? F(1e-300) : F(1e-30);
  constexpr F eps = kDouble ? F(1e-16) : F(1e-7);
  F b = y + F(1) - a, c = F(1) / tiny, d = F(1) / b, h = d;
  for (int i = 1; i < (kDouble ? 1000 : 96); ++i) {
    const F an = -(F)i * ((F)i - a);
    b += F(2);
    d = an * d + b;
    if (fabs(d) < tiny) d = tiny;
    c = b + an / c;
    if (fabs(c) < tiny) c = tiny;
    d = F(1) / d;
    const F del = d * c;
    h *= del;
    if (fabs(del - F(1)) < eps) break;
  }
  const F lq = lpre + log(h);
  return want_p ? log1p(-exp(lq)) : lq;
}

// One Halley step in t = log y towards log P (use_p) or log Q = target: with F
// the difference, F' = +-e^(lf - log P), lf = log(y f(y)) and f the Gamma
// density, and F'' / F' = a - y - F', so the second order costs no further
// function.
template <typename F>
__device__ __forceinline__ F halley_step(const GammaShape& g, F t, F target, bool use_p) {
  const F a = (F)g.a;
  const F y = exp(t);
  const F l = log_pq<F>(g, t, y, use_p);
  const F lf = a * t - y - (F)g.lga;
  const F dF = use_p ? exp(lf - l) : -exp(lf - l);
  const F u = (l - target) / dF;
  // as long as its correction is moderate (near the root it is)
  const F corr = F(1) - F(0.5) * u * (a - y - dF);
  const F step = corr > F(0.5) && corr < F(2) ? u / corr : u;
  return fmin(fmax(step, F(-2)), F(2));
}

// log Phi(x) for the standard normal distribution function.
__device__ double log_ndtr(double x) { return log(0.5 * erfc(-x * 0.70710678118654752440)); }

// t = log y with Q(a, y) = Phi(xi); xi is clamped to [-37, 37] (Phi stays
// normal).  Up to four steps in float bring t to a few times 1e-6, where one
// step in double is left to do: the error of a step is of the third order in
// its length, so after one below 1e-5 the rounding of t dominates.  (Measured
// at 512^2 pixels, a = 1.995: Newton steps in double 100 us, Halley steps in
// double with the constants of a hoisted 44 us, with the float start 34 us;
// the FP64 units' work in the series and the fraction bounds it.)
__device__ double invgamma_t(const GammaShape& g, double xi) {
  const double a = g.a;
  xi = fmin(fmax(xi, -37.0), 37.0);
  const bool use_p = xi > 0.0;  // the smaller of the two is the accurate one
  const double target = log_ndtr(-fabs(xi));
  // starting point
  double t;
  const double z = -xi;  // standard normal quantile of P's target
  if (a >= 1.0) {
    const double c = 1.0 - 1.0 / (9.0 * a) + z / (3.0 * g.sqrta);
    // small y: P ~ y^a / Gamma(a + 1)
    t = c > 0.05 ? g.loga + 3.0 * log(c) : ((use_p ? target : log_ndtr(z)) + g.lga1) / a;
  } else {
    // P(a, y) ~ tt (y)^a below y = 1 and ~ 1 - (1 - tt) e^(1 - y) above,
    // tt = 1 - a (0.253 + 0.12 a) (the upper branch from Q, in logs)
    const double tt = 1.0 - a * (0.253 + 0.12 * a);
    const double lp_t = use_p ? target : log_ndtr(z);
    const double lq_t = use_p ? log_ndtr(xi) : target;
    t = lp_t < log(tt) ? (lp_t - log(tt)) / a : log(1.0 - lq_t + log(1.0 - tt));
  }
  if (fabs(xi) < 6.0 && a < 64.0) {
    float tf = (float)t;
    for (int it = 0; it < 4; ++it) {
      const float step = halley_step<float>(g, tf, (float)target, use_p);
      tf -= step;
      if (!(fabsf(step) > 1e-3f)) break;
    }
    // a start that float cannot improve stays as it was
    if (fabs((double)tf - t) < 2.0) t = (double)tf;
  }
  for (int it = 0; it < 100; ++it) {
    const double step = halley_step<double>(g, t, target, use_p);
    t -= step;
    if (fabs(step) < 1e-5) break;
  }
  return t;
}

// log I = log q - t and d log I / d xi = phi(xi) Gamma(a) / (y^a e^-y).
__device__ void invgamma_log(const GammaShape& g, double logq, double xi, double& logi,
                             double& dlog) {
  const double t = invgamma_t(g, xi);
  const double xc = fmin(fmax(xi, -37.0), 37.0);
  logi = logq - t;
  dlog = exp(-0.5 * xc * xc - 0.91893853320467274178 + g.lga - g.a * t + exp(t));
}

// log I, d log I / d xi and alpha per pixel.
template <typename T>
__global__ __launch_bounds__(PSNT) void k_ps_prepare(int64_t n, GammaShape g, double logq,
                                                    const T* __restrict__ xi,
                                                    const T* __restrict__ xa, double amean,
                                                    double astd, T* __restrict__ w) {
  const int64_t i = blockIdx.x * (int64_t)PSNT + threadIdx.x;
  if (i >= n) return;
  const int64_t smp = blockIdx.y;
  T* ws = w + smp * 3 * n;
  double li, dl;
  invgamma_log(g, logq, (double)xi[smp * n + i], li, dl);
  ws[i] = (T)li;
  ws[n + i] = (T)dl;
  ws[2 * n + i] = xa ? (T)(amean + astd * (double)xa[smp * n + i]) : T(0);
}

// skyt[s, e] = sky[s, e] + exp(log I[s] + alpha[s] * dnu[e]).
template <typename T>
__global__ __launch_bounds__(PSNT) void k_ps_add(int S, int E, int64_t n, const T* __restrict__ sky,
                                                const T* __restrict__ w,
                                                const T* __restrict__ dnu,
                                                T* __restrict__ skyt) {
  const int64_t i = blockIdx.x * (int64_t)PSNT + threadIdx.x;
  if (i >= n) return;
  const int s = blockIdx.y;
  const T* ws = w + (int64_t)s * 3 * n;
  const T li = ws[i], al = ws[2 * n + i];
  for (int e = 0; e < E; ++e) {
    const int64_t o = ((int64_t)s * E + e) * n + i;
    skyt[o] = sky[o] + exp(li + (dnu ? al * dnu[e] : T(0)));
  }
}

// g_xi = d log I / d xi * sum_e p_e ct_e, g_xa = astd * sum_e p_e ct_e dnu_e,
// ct the cotangent of the total sky.
template <typename T>
__global__ __launch_bounds__(PSNT) void k_ps_grad(int S, int E, int64_t n, const T* __restrict__ ct,
                                                 const T* __restrict__ w,
                                                 const T* __restrict__ dnu, double astd,
                                                 T* __restrict__ g_xi, T* __restrict__ g_xa) {
  const int64_t i = blockIdx.x * (int64_t)PSNT + threadIdx.x;
  if (i >= n) return;
  const int s = blockIdx.y;
  const T* ws = w + (int64_t)s * 3 * n;
  const T li = ws[i], dl = ws[n + i], al = ws[2 * n + i];
  T a0 = T(0), a1 = T(0);
  for (int e = 0; e < E; ++e) {
    const T de = dnu ? dnu[e] : T(0);
    const T pc = exp(li + al * de) * ct[((int64_t)s * E + e) * n + i];
    a0 += pc;
    a1 += pc * de;
  }
  g_xi[(int64_t)s * n + i] = dl * a0;
  if (g_xa) g_xa[(int64_t)s * n + i] = T(astd) * a1;
}

template <typename T>
__global__ __launch_bounds__(PSNT) void k_invgamma(int64_t n, GammaShape g, double logq,
                                                  const T* __restrict__ xi,
                                                  T* __restrict__ logi,
                                                  T* __restrict__ dlogi) {
  const int64_t i = blockIdx.x * (int64_t)PSNT + threadIdx.x;
  if (i >= n) return;
  double li, dl;
  invgamma_log(g, logq, (double)xi[i], li, dl);
  logi[i] = (T)li;
  if (dlogi) dlogi[i] = (T)dl;
}

unsigned blocks(int64_t n) { return (unsigned)((n + PSNT - 1) / PSNT); }

}  // namespace

int invgamma_prior(int dtype, const void* xi, int64_t n, double a, double q, void* logi,
                   void* dlogi, hipStream_t s) {
  if (n <= 0) return kOk;
  const GammaShape g = gamma_shape(a);
  if (dtype == 0)
    k_invgamma<float><<<blocks(n), PSNT, 0, s>>>(n, g, std::log(q), (const float*)xi,
                                                 (float*)logi, (float*)dlogi);
  else
    k_invgamma<double><<<blocks(n), PSNT, 0, s>>>(n, g, std::log(q), (const double*)xi,
                                                  (double*)logi, (double*)dlogi);
  return check_hip(hipGetLastError(), "invgamma_prior");
}

int ps_prepare(int dtype, const PointSources& ps, int S, int64_t n, const void* xi,
               const void* xa, void* w, hipStream_t s) {
  const GammaShape g = gamma_shape(ps.a);
  const dim3 grid(blocks(n), S);
  if (dtype == 0)
    k_ps_prepare<float><<<grid, PSNT, 0, s>>>(n, g, std::log(ps.q), (const float*)xi,
                                              (const float*)xa, ps.mean, ps.std, (float*)w);
  else
    k_ps_prepare<double><<<grid, PSNT, 0, s>>>(n, g, std::log(ps.q), (const double*)xi,
                                               (const double*)xa, ps.mean, ps.std, (double*)w);
  return check_hip(hipGetLastError(), "point_sources_prepare");
}

int ps_add(int dtype, int S, int E, int64_t n, const void* sky, const void* w, const void* dnu,
           void* skyt, hipStream_t s) {
  const dim3 grid(blocks(n), S);
  if (dtype == 0)
    k_ps_add<float><<<grid, PSNT, 0, s>>>(S, E, n, (const float*)sky, (const float*)w,
                                          (const float*)dnu, (float*)skyt);
  else
    k_ps_add<double><<<grid, PSNT, 0, s>>>(S, E, n, (const double*)sky, (const double*)w,
                                           (const double*)dnu, (double*)skyt);
  return check_hip(hipGetLastError(), "point_sources_add");
}

int ps_grad(int dtype, const PointSources& ps, int S, int E, int64_t n, const void* ct,
            const void* w, const void* dnu, void* g_xi, void* g_xa, hipStream_t s) {
  const dim3 grid(blocks(n), S);
  if (dtype == 0)
    k_ps_grad<float><<<grid, PSNT, 0, s>>>(S, E, n, (const float*)ct, (const float*)w,
                                           (const float*)dnu, ps.std, (float*)g_xi,
                                           (float*)g_xa);
  else
    k_ps_grad<double><<<grid, PSNT, 0, s>>>(S, E, n, (const double*)ct, (const double*)w,
                                            (const double*)dnu, ps.std, (double*)g_xi,
                                            (double*)g_xa);
  return check_hip(hipGetLastError(), "point_sources_grad");
}

}  // namespace jubik
