// Rounding of the raytracer's hit test against exact arithmetic (__float128): for
// random triangles, origins and poses of any scale, the float64 det and barycentric
// numerators of mt_hit's expressions must lie within hit_rounding of the exact ones,
// and no ray may be longer than max_ray_length.
//
// usage: hit_rounding_check <seed> <cases> <scale of the pose> <shear>
// prints the largest error over its bound and the largest ray over its bound; exits 1
// when one exceeds 1.

#include <algorithm>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <random>

#include "../ugu_amd/csrc/rt_math.h"

namespace {

typedef __float128 Q;

template <class T>
struct Parts {
  T det, u, v;
};

// det and the numerators, in mt_hit's order of operations
template <class T>
Parts<T> parts(const float* o, const float* d, const float (*p)[3]) {
  T e1[3], e2[3], r[3], dd[3];
  for (int k = 0; k < 3; k++) {
    e1[k] = T(p[1][k]) - T(p[0][k]);
    e2[k] = T(p[2][k]) - T(p[0][k]);
    r[k] = T(o[k]) - T(p[0][k]);
    dd[k] = d[k];
  }
  auto cross = [](const T* a, const T* b, T* c) {
    c[0] = a[1] * b[2] - a[2] * b[1];
    c[1] = a[2] * b[0] - a[0] * b[2];
    c[2] = a[0] * b[1] - a[1] * b[0];
  };
  auto dot = [](const T* a, const T* b) { return (a[0] * b[0] + a[1] * b[1]) + a[2] * b[2]; };
  T alpha[3], beta[3];
  cross(dd, e2, alpha);
  cross(r, e1, beta);
  return Parts<T>{dot(e1, alpha), dot(alpha, r), dot(dd, beta)};
}

double l1(const float* a, const float* b) {
  double s = 0.0;
  for (int k = 0; k < 3; k++) s += std::fabs(double(a[k]) - (b ? double(b[k]) : 0.0));
  return s;
}

}  // namespace

int main(int argc, char** argv) {
  if (argc != 5) return 2;
  std::mt19937_64 rng(std::strtoull(argv[1], nullptr, 10));
  const int cases = std::atoi(argv[2]);
  const double scale = std::atof(argv[3]), shear = std::atof(argv[4]);
  std::normal_distribution<double> normal;
  std::uniform_real_distribution<double> exponent(-8.0, 8.0);
  double worst = 0.0, worst_ray = 0.0;
  for (int c = 0; c < cases; c++) {
    // a rotation (Gram-Schmidt), scaled and sheared
    double m[3][3];
    for (int i = 0; i < 3; i++) {
      for (int k = 0; k < 3; k++) m[i][k] = normal(rng);
      for (int j = 0; j < i; j++) {
        double s = 0.0;
        for (int k = 0; k < 3; k++) s += m[i][k] * m[j][k];
        for (int k = 0; k < 3; k++) m[i][k] -= s * m[j][k];
      }
      const double n = std::sqrt(m[i][0] * m[i][0] + m[i][1] * m[i][1] + m[i][2] * m[i][2]);
      for (int k = 0; k < 3; k++) m[i][k] /= n;
    }
    float R[9], d[3], dir[3], o[3], p[3][3];
    for (int i = 0; i < 3; i++)
      for (int k = 0; k < 3; k++) R[3 * i + k] = float(scale * (m[i][k] + shear * m[(i + 1) % 3][k]));
    double n = 0.0, x[3];
    for (double& v : x) n += (v = normal(rng)) * v;
    for (int k = 0; k < 3; k++) dir[k] = float(x[k] / std::sqrt(n));
    double len = 0.0;
    for (int i = 0; i < 3; i++) {
      d[i] = (R[3 * i] * dir[0] + R[3 * i + 1] * dir[1]) + R[3 * i + 2] * dir[2];
      len += double(d[i]) * d[i];
    }
    const double size = std::exp2(exponent(rng)), far = size * std::exp2(exponent(rng));
    for (int k = 0; k < 3; k++) o[k] = float(far * normal(rng));
    double mid[3];
    for (double& v : mid) v = far * normal(rng);
    double edge = 0.0, reach = 0.0;
    for (int i = 0; i < 3; i++)
      for (int k = 0; k < 3; k++) p[i][k] = float(mid[k] + size * normal(rng));
    for (int i = 0; i < 3; i++) {
      edge = std::max(edge, l1(p[i], p[(i + 1) % 3]));
      reach = std::max(reach, l1(p[i], nullptr));
    }
    reach += l1(o, nullptr);
    const double ray = ugu_hip::max_ray_length(R);
    worst_ray = std::max(worst_ray, std::sqrt(len) / (ray * (1.0 + 1e-6)));  // d is rounded
    const Parts<double> got = parts<double>(o, d, p);
    const Parts<Q> want = parts<Q>(o, d, p);
    const double err = std::max({double(fabs(double(Q(got.det) - want.det))),
                                 double(fabs(double(Q(got.u) - want.u))),
                                 double(fabs(double(Q(got.v) - want.v)))});
    worst = std::max(worst, err / ugu_hip::hit_rounding(ray, edge, reach));
  }
  std::printf("error %.4f ray %.4f\n", worst, worst_ray);
  return worst <= 1.0 && worst_ray <= 1.0 ? 0 : 1;
}
