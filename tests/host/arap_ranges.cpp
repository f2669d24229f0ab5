// Host harness for the ARAP kernels' SVD (svd_rv_fast of tetmath.h), which
// takes closed-form eigenvectors or Jacobi sweeps by the element's shape.
//
// Line "sqrt E A": square roots in sigma_from, correctly rounded (E) and
// approximate (A), counted by a number type of its own.
// One line per range of singular values: its name, then the worst and the
// root-mean-square relative error of mu (F - R) and of the projected part
// sum_k lambda_k (Q_k : dF) Q_k, first with the FP32 Jacobi basis and FP32
// finish for every element, then by svd_rv_fast; against the FP64 SVD.
#include "../../apple_amd/csrc/tetmath.h"

#include <cmath>
#include <cstdio>
#include <functional>
#include <random>

using namespace apl;

namespace counted {
static int exact = 0, approximate = 0;
struct Num {
  float v;
  Num() = default;
  Num(double x) : v((float)x) {}
};
Num operator+(Num a, Num b) { return a.v + b.v; }
Num operator-(Num a, Num b) { return a.v - b.v; }
Num operator*(Num a, Num b) { return a.v * b.v; }
bool operator<(Num a, Num b) { return a.v < b.v; }
bool operator>(Num a, Num b) { return a.v > b.v; }
Num fabs(Num a) { return std::fabs(a.v); }
Num recip(Num a) { return 1.0f / a.v; }
Num sqrt(Num a) {
  ++exact;
  return std::sqrt(a.v);
}
Num sqrt_r(Num a) {
  ++approximate;
  return std::sqrt(a.v);
}
Num fast_sqrt(Num a) { return sqrt_r(a); }
}  // namespace counted

static Svd<float> svd_sweeps(const M3<float>& G) {
  float a[3][3], e[3];
  ftf_minus_i_f64(G, a);
  M3<float> V;
  jacobi_fast_sweeps(a, V);
  sort_eig(a, V, e);
  return qr_sigma(G, V, e);
}

using Rng = std::mt19937;

static void rotation(Rng& rng, double (&R)[3][3]) {
  std::normal_distribution<double> N(0, 1);
  double q[4], n = 0;
  for (double& c : q) {
    c = N(rng);
    n += c * c;
  }
  for (double& c : q) c /= std::sqrt(n);
  const double w = q[0], x = q[1], y = q[2], z = q[3];
  const double M[3][3] = {{1 - 2 * (y * y + z * z), 2 * (x * y - w * z), 2 * (x * z + w * y)},
                          {2 * (x * y + w * z), 1 - 2 * (x * x + z * z), 2 * (y * z - w * x)},
                          {2 * (x * z - w * y), 2 * (y * z + w * x), 1 - 2 * (x * x + y * y)}};
  for (int i = 0; i < 3; ++i)
    for (int j = 0; j < 3; ++j) R[i][j] = M[i][j];
}

template <class A, class B>
static double rel(const M3<A>& a, const M3<B>& b, double scale) {
  double e = 0;
  for (int i = 0; i < 3; ++i)
    for (int j = 0; j < 3; ++j) e = std::fmax(e, std::fabs((double)a.m[i][j] - (double)b.m[i][j]));
  return e / scale;
}
template <class A>
static double largest(const M3<A>& a) {
  double n = 1e-300;
  for (int i = 0; i < 3; ++i)
    for (int j = 0; j < 3; ++j) n = std::fmax(n, std::fabs((double)a.m[i][j]));
  return n;
}

template <class R>
static M3<R> projected(const Svd<R>& S, const M3<R>& dF) {
  R lam[3], q[3], m[3], c[3];
  arap_lambdas(S.s, lam);
  twist_coords(S, dF, q, m);
  for (int k = 0; k < 3; ++k) c[k] = lam[k] * q[k];
  return twist_combine(S, c);
}

struct Err {
  double worst = 0, sq = 0;
  void add(double e) {
    worst = std::fmax(worst, e);
    sq += e * e;
  }
};

static void run(const char* name, const std::function<void(Rng&, double*)>& sigma) {
  constexpr int N = 20000;
  Rng rng(11);
  std::normal_distribution<double> normal(0, 1);
  Err p[2], q[2];
  for (int it = 0; it < N; ++it) {
    double s[3], A[3][3], B[3][3];
    sigma(rng, s);
    rotation(rng, A);
    rotation(rng, B);
    M3<float> Gf, dFf;
    M3<double> Gd, dFd;
    for (int i = 0; i < 3; ++i)
      for (int j = 0; j < 3; ++j) {
        double f = i == j ? -1 : 0;
        for (int l = 0; l < 3; ++l) f += A[i][l] * s[l] * B[j][l];
        Gd.m[i][j] = Gf.m[i][j] = (float)f;
        dFd.m[i][j] = dFf.m[i][j] = (float)normal(rng);
      }
    const Svd<double> Sd = svd_rv<double>(Gd);
    const M3<double> Pd = udv(Sd, Sd.sm1), Md = projected(Sd, dFd);
    const Svd<float> S[2] = {svd_sweeps(Gf), svd_rv_fast(Gf)};
    for (int k = 0; k < 2; ++k) {
      p[k].add(rel(Pd, udv(S[k], S[k].sm1), largest(Pd)));
      q[k].add(rel(Md, projected(S[k], dFf), largest(dFd)));
    }
  }
  std::printf("%s", name);
  for (int k = 0; k < 2; ++k)
    std::printf(" %.4e %.4e %.4e %.4e", p[k].worst, std::sqrt(p[k].sq / N), q[k].worst, std::sqrt(q[k].sq / N));
  std::printf("\n");
}

int main() {
  for (float e : {-0.2f, -1e-3f, 0.0f, 1e-6f, 0.1f}) {
    counted::Num s, sm1;
    sigma_from(counted::Num(e), counted::Num(1.0), s, sm1);
  }
  std::printf("sqrt %d %d\n", counted::exact, counted::approximate);

  auto near = [](Rng& r, double c) { return c * std::uniform_real_distribution<double>(0.95, 1.05)(r); };
  char name[64];
  for (double c : {0.26, 0.27, 0.3, 0.35, 0.45, 0.6, 0.8, 1.0, 1.3, 2.0, 4.0, 8.0}) {
    std::snprintf(name, sizeof name, "all_%g", c);
    run(name, [&](Rng& r, double* s) { s[0] = near(r, c), s[1] = near(r, c), s[2] = near(r, c); });
  }
  for (double c : {1.5, 2.0, 2.5, 3.0, 3.5, 4.0, 6.0, 8.0, 9.0, 15.0, 25.0}) {
    std::snprintf(name, sizeof name, "long_%g", c);
    run(name, [&](Rng& r, double* s) { s[0] = near(r, c), s[1] = near(r, 1), s[2] = near(r, 1); });
  }
  for (double c : {2.0, 4.0, 5.0, 8.0}) {
    std::snprintf(name, sizeof name, "flat_%g", c);
    run(name, [&](Rng& r, double* s) { s[0] = near(r, c), s[1] = near(r, c), s[2] = near(r, 1); });
  }
  for (double c : {1.25, 2.0, 4.0, 10.0}) {
    std::snprintf(name, sizeof name, "any_%g", c);
    run(name, [&](Rng& r, double* s) {
      for (int i = 0; i < 3; ++i) s[i] = std::exp(std::log(c) * std::uniform_real_distribution<double>(-1, 1)(r));
    });
  }
  for (double c : {1e-4, 1e-3, 1e-2}) {
    std::snprintf(name, sizeof name, "strain_%g", c);
    run(name, [&](Rng& r, double* s) {
      std::normal_distribution<double> N(0, 1);
      for (int i = 0; i < 3; ++i) s[i] = 1 + c * N(r);
    });
  }
  return 0;
}
