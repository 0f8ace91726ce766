// Agreement of primfhllc_sel (one code path) with primfhllc (a branch per
// outcome) on random x-aligned states, bit for bit in double and float (two
// NaNs count as equal), with how often each outcome was reached; and of
// limit_all with limit1 for every limiter.
#include <cstdio>
#include <cstring>
#include <limits>
#include <random>

#include "wx_physics.h"

using namespace wx;

template <typename R> bool same(const R *a, const R *b, int n) {
  for (int q = 0; q < n; q++)
    if (memcmp(&a[q], &b[q], sizeof(R)) != 0 && !(a[q] != a[q] && b[q] != b[q])) return false;
  return true;
}

// outcome of primfhllc: 0 left, 1 right, 2 left star, 3 right star, 4 none
template <typename R> int outcome(const Phys<R> &c, const R *l, const R *r) {
  const R cl = sound(c, l), cr = sound(c, r);
  const R sl = rfmin(l[1] - cl, r[1] - cr), sr = rfmax(l[1] + cl, r[1] + cr);
  if (sl > R(0)) return 0;
  if (sr < R(0)) return 1;
  const R s = (r[4] - l[4] + l[0] * l[1] * (sl - l[1]) - r[0] * r[1] * (sr - r[1])) /
              (l[0] * (sl - l[1]) - r[0] * (sr - r[1]));
  return s >= R(0) ? 2 : (s <= R(0) ? 3 : 4);
}

template <typename R> int run(const char *tag, int n, unsigned seed) {
  Phys<R> c{5, 0, SOLVER_HLLC, 1, R(5.0 / 3.0), R(1.5)};
  std::mt19937_64 g(seed);
  std::uniform_real_distribution<double> U(-1, 1);
  const R odd[] = {R(0), R(-0.0), std::numeric_limits<R>::quiet_NaN(), std::numeric_limits<R>::infinity(),
                   -std::numeric_limits<R>::infinity(), std::numeric_limits<R>::max(), std::numeric_limits<R>::min()};
  int bad = 0, reg[5] = {0};
  for (int t = 0; t < n; t++) {
    R l[5], r[5], a[MAXV], b[MAXV];
    const double vs = t % 3 == 0 ? 6.0 : 1.0;      // supersonic to either side
    for (R *p : {l, r}) {
      p[0] = R(0.1 + std::abs(U(g)));
      p[4] = R(0.01 + std::abs(U(g)));
    }
    const double common = vs * U(g);
    for (int q = 1; q < 4; q++) {
      l[q] = R(common + 0.3 * U(g));
      r[q] = R(common + 0.3 * U(g));
    }
    if (t % 11 == 0) for (int q = 0; q < 5; q++) r[q] = l[q];          // no jump
    if (t % 13 == 0) l[1] = r[1] = R(0);                               // contact at rest
    if (t % 17 == 0) (t & 1 ? l : r)[t / 17 % 5] = odd[t / 85 % 7];    // values a solver meets in a bad cell
    reg[outcome(c, l, r)]++;
    primfhllc(c, l, r, a);
    primfhllc_sel(c, l, r, b);
    if (!same(a, b, 5)) {
      if (++bad < 5) printf("%s case %d: outcome %d\n", tag, t, outcome(c, l, r));
    }
    R x[4][5];
    for (auto &v : x) for (R &q : v) q = t % 19 == 0 ? odd[(t + (&q - &v[0])) % 7] : R(U(g));
    for (int lim = -1; lim <= 6; lim++) {
      R p1[5], p2[5], q1[5], q2[5];
      for (int v = 0; v < 5; v++) {
        p1[v] = p2[v] = x[1][v];
        q1[v] = q2[v] = x[2][v];
        limit1(x[0][v], p1[v], q1[v], x[3][v], lim);
      }
      limit_all<5>(x[0], p2, q2, x[3], lim);
      if (!same(p1, p2, 5) || !same(q1, q2, 5)) bad++;
    }
  }
  printf("%s left %d right %d L* %d R* %d none %d .\n", tag, reg[0], reg[1], reg[2], reg[3], reg[4]);
  return bad;
}

int main() {
  const int d = run<double>("double", 400000, 11), f = run<float>("float", 400000, 12);
  printf("double mismatches %d, float mismatches %d\n", d, f);
  return d || f;
}
