// libm_pow_const against libm_pow, bit for bit, for the exponents that the
// controllers and the initial step use.  Reads doubles x from stdin; prints the
// number of comparisons and of differences, with the first few of them.
#include <cstdio>
#include <cstring>
#include <vector>

#include "../../differential-equations_amd/csrc/de_pow_libm.h"

int main() {
  std::vector<double> xs;
  double buf[4096];
  for (size_t n; (n = fread(buf, sizeof(double), 4096, stdin)) > 0;)
    xs.insert(xs.end(), buf, buf + n);
  const double ys[] = {-0.2, -(1.0 / 4.0), -(1.0 / 5.0), -(1.0 / 6.0), -(1.0 / 7.0),
                       -0.125, -(1.0 / 9.0), 1.0 / 4.0, 1.0 / 5.0, 1.0 / 6.0, 1.0 / 7.0,
                       1.0 / 8.0, 1.0 / 9.0, 0.499, -0.499, 0x1p-10, -0x1p-10};
  long long bad = 0, all = 0;
  for (double y : ys) {
    for (double x : xs) {
      const double a = de::libm_pow_const(x, y), b = de::libm_pow(x, y);
      const bool same = (a != a && b != b) || de::as_u64(a) == de::as_u64(b);
      ++all;
      if (!same && ++bad <= 5) printf("x %a y %a: %a, libm_pow %a\n", x, y, a, b);
    }
  }
  printf("%lld compared, %lld differ\n", all, bad);
  return bad == 0 ? 0 : 1;
}
