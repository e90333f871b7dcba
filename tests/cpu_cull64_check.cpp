// CPU check of the FP64 discrete classification (cull_pair64, d2_cull.hpp):
// a certain miss never hits by the reference's distance, a certain hit always
// does.  Half of the pairs sit at the hit threshold within 1e-6 relative
// (moved along their closest-point direction); triangles of many sizes, thin
// ones, shared vertices and world offsets up to 1 km.  Built and run by
// tests/test_cull64_cpu.py; prints "<cases> <violations> <misses> <certain
// hits> <hits>".
#include <cmath>
#include <cstdio>
#include <random>

#define D2_HD inline
#include <algorithm>
using std::cos;
using std::fabs;
using std::sin;
using std::sqrt;
#include "../delta2_amd/csrc/d2_geom.hpp"
#include "../delta2_amd/csrc/d2_cull.hpp"

static std::mt19937_64 rng(97531);
static double U(double a, double b) { return std::uniform_real_distribution<double>(a, b)(rng); }
static d2::v3<double> V(double s, const d2::v3<double>& o) { return {o.x + U(-s, s), o.y + U(-s, s), o.z + U(-s, s)}; }

int main() {
  long long cases = 0, viol = 0, miss = 0, two = 0, hits = 0;
  for (int k = 0; k < 120000; ++k) {
    const double s = std::exp(U(std::log(0.002), std::log(2.0))), far = k % 6 == 0 ? 1000.0 : 3.0;
    const d2::v3<double> o{U(-far, far), U(-far, far), U(-far, far)};
    d2::tri<double> a{V(s, o), V(s, o), V(s, o)};
    const d2::v3<double> ob = V(k % 3 ? 2.0 * s : 6.0 * s, o);
    const double sb = k % 4 == 0 ? 10.0 * s : s;
    d2::tri<double> b{V(sb, ob), V(sb, ob), V(sb, ob)};
    if (k % 7 == 0) a.c = d2::add(d2::lerp(a.a, a.b, U(0.0, 1.0)), V(1e-3 * s, {0, 0, 0}));  // thin
    if (k % 11 == 0) b.a = a.b;                                                             // a shared vertex
    const double thr = (U(0.001, 0.03) + U(0.0, 0.02)) + U(0.0, k % 5 ? 0.02 : 0.5);
    d2::v3<double> P, Q;
    double d = d2::tri_tri_dist(a, b, P, Q);
    if (k % 2 == 0 && d > 1e-9) {
      const double mv = thr * (1.0 + U(-1e-6, 1e-6)) - d;
      const d2::v3<double> m = d2::scl(d2::dvs(d2::sub(Q, P), d), mv);
      b = {d2::add(b.a, m), d2::add(b.b, m), d2::add(b.c, m)};
      d = d2::tri_tri_dist(a, b, P, Q);
    }
    const bool hit = d < thr;
    const int cls = d2::cull_pair64(a, b, thr, true), quick = d2::cull_pair64(a, b, thr, false);
    ++cases, hits += hit, miss += cls == 0, two += cls == 2;
    viol += (cls == 0 && hit) || (cls == 2 && !hit) || (quick == 0) != (cls == 0) || quick == 2;
  }
  std::printf("%lld %lld %lld %lld %lld\n", cases, viol, miss, two, hits);
  return 0;
}
