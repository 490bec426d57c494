// Errors of the double-precision functions of the evaluation kernels (stormm_amd/csrc/mm_device.h)
// on the device, in units of the last place against 80-bit arithmetic on the host, over the
// arguments that the kernels give them; Born radii, bonds and angles against the same formulas in
// the IEEE operations.  Arguments: the names of the functions to check.
#include <cmath>
#include <cstdio>
#include <cstring>
#include <functional>
#include <random>
#include <vector>

#include <hip/hip_runtime.h>

#include "../../stormm_amd/csrc/mm_eval.h"

using namespace stormm_amd;
using D = Prec<double>;

struct Exp {
  static __device__ double eval(double x, double) { return D::exp(x); }
};
struct Log {
  static __device__ double eval(double x, double) { return D::log(x); }
};
struct Tanh {
  static __device__ double eval(double x, double) { return D::tanh(x); }
};
struct Rsqrt {
  static __device__ double eval(double x, double) { return D::rsqrt(x); }
};

template <typename F> __global__ void k_eval(const double *x, const double *y, double *out, int n) {
  const int i = static_cast<int>(blockIdx.x * blockDim.x + threadIdx.x);
  if (i < n) {
    out[i] = F::eval(x[i], y[i]);
  }
}

#define TRY(call)                                                     \
  do {                                                                \
    const hipError_t e_ = (call);                                     \
    if (e_ != hipSuccess) {                                           \
      std::printf("%s: %s\n", #call, hipGetErrorString(e_));          \
      return false;                                                   \
    }                                                                 \
  } while (0)

template <typename F>
static bool evaluate(const std::vector<double> &x, const std::vector<double> &y,
                     std::vector<double> &out) {
  const int n = static_cast<int>(x.size());
  const size_t bytes = x.size() * sizeof(double);
  double *d = nullptr;
  TRY(hipMalloc(&d, 3 * bytes));
  TRY(hipMemcpy(d, x.data(), bytes, hipMemcpyHostToDevice));
  TRY(hipMemcpy(d + n, y.data(), bytes, hipMemcpyHostToDevice));
  hipLaunchKernelGGL((k_eval<F>), dim3((n + 255) / 256), dim3(256), 0, 0, d, d + n, d + 2 * n, n);
  TRY(hipGetLastError());
  out.resize(x.size());
  TRY(hipMemcpy(out.data(), d + 2 * n, bytes, hipMemcpyDeviceToHost));
  TRY(hipFree(d));
  return true;
}

struct Range {
  double lo, hi;
};

// The largest error over 2^18 arguments of each range; `real` is the exact function.
template <typename F>
static bool check(const char *name, double most, const std::vector<Range> &ranges,
                  const std::function<long double(long double, long double)> &real) {
  bool ok = true;
  for (size_t r = 0; r < ranges.size(); r++) {
    std::mt19937_64 rng(7000 + r);
    std::uniform_real_distribution<double> u(0.0, 1.0);
    std::vector<double> x(1 << 18), y(1 << 18), out;
    for (size_t i = 0; i < x.size(); i++) {
      // Every other argument spread over the logarithm where the range does not cross zero.
      const double lo = ranges[r].lo, hi = ranges[r].hi;
      x[i] = (lo > 0.0 && (i & 1)) ? lo * std::pow(hi / lo, u(rng)) : lo + ((hi - lo) * u(rng));
      y[i] = 0.1 + (3.0 * u(rng));
    }
    if (!evaluate<F>(x, y, out)) {
      return false;
    }
    long double worst = 0.0L;
    double at = 0.0;
    for (size_t i = 0; i < x.size(); i++) {
      const long double want = real(x[i], y[i]);
      int e = 0;
      (void)std::frexp(want, &e);
      const long double err = std::fabs((out[i] - want) / std::ldexp(1.0L, e - 53));
      if (!(err <= worst)) {
        worst = err;
        at = x[i];
      }
    }
    std::printf("%s [%g, %g]: %.4Lf ulp at %.17g (at most %g)\n", name, ranges[r].lo, ranges[r].hi,
                worst, at, most);
    ok = ok && worst <= most;
  }
  return ok;
}

// A value that is not a number stays one.
template <typename F> static bool keeps_nan(const char *name) {
  std::vector<double> out;
  const bool ok = evaluate<F>({std::nan(""), -std::nan("")}, {1.0, 1.0}, out) &&
                  std::isnan(out[0]) && std::isnan(out[1]);
  std::printf("%s of a NaN: %s\n", name, ok ? "NaN" : "a number");
  return ok;
}

// Born radii against the same formulas in the IEEE operations, bit for bit.  x: the share of
// 1 / rho that the integral takes away; y: the intrinsic radius; out: 0 for equal.
template <int MODEL> struct Radii {
  static __device__ double eval(double x, double pbr) {
    const int igb = (MODEL == 0) ? 1 : 5;
    // Variables, so that the products below are contracted as the ones of born_radius.
    double al = (MODEL == 1) ? 0.8 : 1.0, be = (MODEL == 1) ? 0.0 : 0.8,
           ga = (MODEL == 1) ? 2.909125 : 4.85;
    const double rho = pbr - 0.09, psi = -x / rho;
    const BornRadius got = born_radius(igb, al, be, ga, rho, pbr, psi);
    double R, dr_dpsi = 0.0;
    if (igb == 1) {
      R = 1.0 / ((1.0 / rho) + psi);
      R = (R < 0.0) ? 30.0 : R;
    }
    else {
      const double fipsi = psi * (-rho);
      const double thi = D::tanh((al - (be * fipsi) + (ga * fipsi * fipsi)) * fipsi);
      R = 1.0 / ((1.0 / rho) - thi / pbr);
      dr_dpsi = (al - ((2.0 * be) - (3.0 * ga * fipsi)) * fipsi) * (1.0 - thi * thi) * rho / pbr;
    }
    return (got.R == R && got.inv_R == 1.0 / R && got.dr_dpsi == dr_dpsi) ? 0.0 : 1.0;
  }
};

// Atoms of a valence term and the forces it adds, for the terms of the evaluation kernels.
struct Atoms {
  Vec3 p[3];
  long long *f;
  __device__ Vec3 disp(int from, int to) const {
    return {p[to].x - p[from].x, p[to].y - p[from].y, p[to].z - p[from].z};
  }
  __device__ void add(int a, long long x, long long y, long long z) const {
    f[3 * a] += x;
    f[3 * a + 1] += y;
    f[3 * a + 2] += z;
  }
};
constexpr double kForceScale = 1099511627776.0;  // 2^40

// A bond of 0.1 to 3 A along x and y, and an angle between bonds of 1 to 2 A that is y, against
// the same terms in the IEEE operations, bit for bit.
struct Bond {
  static __device__ double eval(double x, double y) {
    long long got[6] = {0, 0, 0, 0, 0, 0};
    const Atoms v = {{{0.0, 0.0, 0.0}, {x, 0.3 * y, 0.1}, {}}, got};
    const double kb = 310.0, r0 = 1.09;
    const double e = eval_bond<true>(v, 0, 1, kb, r0, kForceScale);
    const Vec3 d = v.disp(0, 1);
    const double dr = sqrt(dot(d, d));
    const double dl = dr - r0;
    const double fmag = 2.0 * kb * dl / dr;
    return (e == kb * dl * dl && got[0] == fix64(fmag * d.x * kForceScale) &&
            got[1] == fix64(fmag * d.y * kForceScale) &&
            got[2] == fix64(fmag * d.z * kForceScale)) ? 0.0 : 1.0;
  }
};
struct Angle {
  static __device__ double eval(double x, double y) {
    long long got[9] = {0, 0, 0, 0, 0, 0, 0, 0, 0};
    const double l = 1.0 + (0.5 * fabs(x));
    const Atoms v = {{{1.2, 0.0, 0.1 * x}, {0.0, 0.0, 0.0}, {l * cos(y), l * sin(y), 0.0}}, got};
    const double ka = 63.0, th0 = 1.91;
    const double e = eval_angle<true>(v, 0, 1, 2, ka, th0, kForceScale);
    const Vec3 ba = v.disp(1, 0);
    const Vec3 bc = v.disp(1, 2);
    const double mgba = dot(ba, ba);
    const double mgbc = dot(bc, bc);
    const double invbabc = 1.0 / sqrt(mgba * mgbc);
    double costheta = dot(ba, bc) * invbabc;
    costheta = (costheta < -1.0) ? -1.0 : ((costheta > 1.0) ? 1.0 : costheta);
    const double dtheta = acos(costheta) - th0;
    const double dA = -2.0 * ka * dtheta / sqrt(1.0 - (costheta * costheta));
    const double sqba = dA / mgba;
    const double sqbc = dA / mgbc;
    const double mbabc = dA * invbabc;
    return (e == ka * dtheta * dtheta &&
            got[0] == -fix64(((bc.x * mbabc) - (costheta * ba.x * sqba)) * kForceScale) &&
            got[1] == -fix64(((bc.y * mbabc) - (costheta * ba.y * sqba)) * kForceScale) &&
            got[2] == -fix64(((bc.z * mbabc) - (costheta * ba.z * sqba)) * kForceScale) &&
            got[6] == -fix64(((ba.x * mbabc) - (costheta * bc.x * sqbc)) * kForceScale) &&
            got[7] == -fix64(((ba.y * mbabc) - (costheta * bc.y * sqbc)) * kForceScale) &&
            got[8] == -fix64(((ba.z * mbabc) - (costheta * bc.z * sqbc)) * kForceScale)) ? 0.0
                                                                                         : 1.0;
  }
};
template <typename F> static bool check_term(const char *name) {
  std::mt19937_64 rng(9000);
  std::uniform_real_distribution<double> u(0.0, 1.0);
  std::vector<double> x(1 << 18), y(1 << 18), out;
  for (size_t i = 0; i < x.size(); i++) {
    x[i] = 4.0 * (u(rng) - 0.5);
    y[i] = 0.05 + (3.05 * u(rng));
  }
  const bool ran = evaluate<F>(x, y, out);
  size_t differ = 0;
  for (double o : out) {
    differ += (o != 0.0) ? 1 : 0;
  }
  std::printf("%s: %zu of %zu differ\n", name, differ, x.size());
  return ran && differ == 0;
}

static bool check_radii(int model) {
  std::mt19937_64 rng(8000 + model);
  std::uniform_real_distribution<double> u(0.0, 1.0);
  std::vector<double> x(1 << 18), pbr(1 << 18), out;
  for (size_t i = 0; i < x.size(); i++) {
    x[i] = (i == 0) ? 0.0 : 1.5 * u(rng);
    pbr[i] = 1.0 + (2.0 * u(rng));
  }
  const bool ran = (model == 0) ? evaluate<Radii<0>>(x, pbr, out) :
                   (model == 1) ? evaluate<Radii<1>>(x, pbr, out) :
                                  evaluate<Radii<2>>(x, pbr, out);
  size_t differ = 0;
  for (double o : out) {
    differ += (o != 0.0) ? 1 : 0;
  }
  std::printf("born_radius, model %d: %zu of %zu differ\n", model, differ, x.size());
  return ran && differ == 0;
}

static bool check_named(const char *name) {
  const std::string f(name);
  if (f == "exp") {
    // The device library's bound is one unit.
    return check<Exp>(name, 1.0, {{-1.0, 0.0}, {-5.0, -1.0}, {-20.0, -5.0}, {-40.0, -20.0},
                                  {-700.0, -40.0}},
                      [](long double x, long double) { return std::exp(x); }) &&
           keeps_nan<Exp>(name);
  }
  if (f == "log") {
    // Half a unit from the last sum and less than a tenth from the terms below it.
    return check<Log>(name, 0.6, {{0.02, 0.5}, {0.5, 0.9}, {0.9, 1.0}, {1.0, 1.1}, {1.1, 50.0}},
                      [](long double x, long double) { return std::log(x); }) &&
           keeps_nan<Log>(name);
  }
  if (f == "rsqrt") {
    // Half a unit from the last sum; the residual is exact and e^3 a thousandth of a unit.
    return check<Rsqrt>(name, 0.51, {{0.25, 1.0}, {1.0, 4.0}, {1.0, 1.0e5}, {1.0e-6, 1.0}},
                        [](long double x, long double) { return 1.0L / std::sqrt(x); });
  }
  if (f == "tanh") {
    // The device library's error over the same arguments.
    return check<Tanh>(name, 0.859, {{1.0e-8, 1.0e-4}, {1.0e-4, 0.01}, {0.01, 0.5}, {0.5, 3.0},
                                     {3.0, 40.0}, {-1.0, 0.0}},
                       [](long double x, long double) { return std::tanh(x); }) &&
           keeps_nan<Tanh>(name);
  }
  if (f == "born_radius") {
    // Integrals from none to a buried atom's, radii of 1 to 3 A, the three models' constants.
    bool ok = true;
    for (int model = 0; model < 3; model++) {
      ok = check_radii(model) && ok;
    }
    return ok;
  }
  if (f == "bond") {
    return check_term<Bond>(name);
  }
  if (f == "angle") {
    return check_term<Angle>(name);
  }
  std::printf("no function %s\n", name);
  return false;
}

int main(int argc, char **argv) {
  bool ok = argc > 1;
  for (int i = 1; i < argc; i++) {
    ok = check_named(argv[i]) && ok;
  }
  std::printf(ok ? "math ok\n" : "math FAILED\n");
  return ok ? 0 : 1;
}
