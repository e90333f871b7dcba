// The FP32 node tests in b's frame (spheres_apart_rel, boxes_apart_faces_rel)
// never call a pair of nodes apart that the FP64 forms do not: random boxes
// and spheres, poses up to 1 km from the origin and bodies up to 200 m apart,
// half of the cases moved to within 1e-6 relative of the FP64 threshold.
// Built and run by tests/test_rel_bounds_cpu.py; prints "<cases> <sphere
// violations> <box violations> <apart, spheres: FP64, FP32> <boxes: FP64, FP32>".
#include <algorithm>
#include <cmath>
#include <cstdio>
#include <random>

#define D2_HD inline
using std::cos;
using std::fabs;
using std::sin;
using std::sqrt;
#include "../delta2_amd/csrc/d2_geom.hpp"

static std::mt19937_64 rng(24680);
static double U(double a, double b) { return std::uniform_real_distribution<double>(a, b)(rng); }

static void rand_pose(double* T, double far) {
  d2::quat q{U(-1, 1), U(-1, 1), U(-1, 1), U(-1, 1)};
  const double n = sqrt(q.w * q.w + q.x * q.x + q.y * q.y + q.z * q.z);
  q.w /= n, q.x /= n, q.y /= n, q.z /= n;
  d2::pose(q, d2::v3<double>{U(-far, far), U(-far, far), U(-far, far)}, T);
}
static void rand_node(double sz, double off, float* b) {
  for (int k = 0; k < 3; ++k) {
    const double c = U(-off, off), h = U(0.0, sz);
    b[k] = (float)(c - h), b[3 + k] = (float)(c + h), b[8 + k] = (float)(c + U(-0.1, 0.1) * sz);
  }
  b[6] = (float)U(0.0, 0.01), b[7] = (float)U(0.0, 2.0 * sz), b[11] = 0.f;
}

int main() {
  long long cases = 0, bad[2] = {0, 0}, apart64[2] = {0, 0}, apart32[2] = {0, 0};
  for (int k = 0; k < 200000; ++k) {
    const double sz = std::exp(U(std::log(0.001), std::log(5.0))), far = k % 4 == 0 ? 1000.0 : 5.0;
    const float search = (float)U(0.001, 0.05);
    float ba[12], bb[12];
    rand_node(sz, k % 3 == 0 ? 100.0 : sz, ba), rand_node(sz, k % 3 == 0 ? 100.0 : sz, bb);
    double Ta[16], Tb[16];
    rand_pose(Ta, far), rand_pose(Tb, far);
    // b at a distance around contact from a
    double dir[3] = {U(-1, 1), U(-1, 1), U(-1, 1)};
    const double n = sqrt(dir[0] * dir[0] + dir[1] * dir[1] + dir[2] * dir[2]);
    double dist = U(0.0, k % 3 == 0 ? 300.0 : 6.0 * sz);
    const int form = k & 1;
    auto apart = [&](double x) {
      for (int r = 0; r < 3; ++r) Tb[4 * r + 3] = Ta[4 * r + 3] + x * dir[r] / n;
      return form ? d2::boxes_apart_faces(Ta, Tb, ba, bb, (double)search) : d2::spheres_apart(Ta, Tb, ba, bb, (double)search);
    };
    if (k % 4 < 2 && apart(2000.0)) {  // to the threshold of the FP64 form, then within 1e-6 of it
      double lo = 0.0, hi = 2000.0;
      if (apart(0.0)) continue;
      for (int i = 0; i < 80; ++i) {
        const double mid = 0.5 * (lo + hi);
        (apart(mid) ? hi : lo) = mid;
      }
      dist = lo * (1.0 + U(-1e-6, 1e-6));
    }
    (void)apart(dist);
    float f[d2::PF_FLOATS];
    d2::pair_pose_f32(Ta, Tb, search, f);
    const bool a64[2] = {d2::spheres_apart(Ta, Tb, ba, bb, (double)search), d2::boxes_apart_faces(Ta, Tb, ba, bb, (double)search)};
    const bool a32[2] = {d2::spheres_apart_rel(f, ba, bb), d2::boxes_apart_faces_rel(f, ba, bb)};
    ++cases;
    for (int v = 0; v < 2; ++v) bad[v] += a32[v] && !a64[v], apart64[v] += a64[v], apart32[v] += a32[v];
  }
  printf("%lld %lld %lld %lld %lld %lld %lld\n", cases, bad[0], bad[1], apart64[0], apart32[0], apart64[1], apart32[1]);
  return 0;
}
