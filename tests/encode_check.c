/* cube_encode_v3 against cube_encode_v, the codec's formula, on the CPU */
#include <math.h>
#include "../cafproject_amd/csrc/cube_math.h"

static int64_t bad3(int bytes, double c, const double v[3]) {
  int32_t k[3];
  cube_encode_v3(bytes, c, v, k);
  int64_t n = 0;
  for (int i = 0; i < 3; ++i) n += k[i] != cube_encode_v(bytes, c, v[i]);
  return n;
}
/* n values of u = c*v spread evenly in log from lo to hi, both signs */
int64_t bad_span(int bytes, double c, double lo, double hi, int64_t n) {
  int64_t b = 0;
  const double s = pow(hi / lo, 1.0 / (double)n);
  double u = lo;
  for (int64_t i = 0; i < n; ++i, u *= s) {
    const double v[3] = {u / c, -u / c, 0.7 * u / c};
    b += bad3(bytes, c, v);
  }
  return b;
}
/* around each boundary between two codes: it and 2^-52 .. 2^-8 of it off */
int64_t bad_boundaries(int bytes, double c) {
  const int kmax = bytes == 1 ? 127 : 32767;
  int64_t b = 0;
  for (int k = 0; k < kmax; ++k) {
    const double t = tan((k + 0.5) * (double)CUBE_PI_F / (bytes == 1 ? 255.0 : 65535.0)) / c;
    for (int e = 52; e >= 8; --e) {
      const double v[3] = {t * (1.0 + ldexp(1.0, -e)), -t * (1.0 - ldexp(1.0, -e)), t};
      b += bad3(bytes, c, v);
    }
  }
  return b;
}
int64_t bad_special(int bytes, double c) {
  const double w[6] = {0.0, 1e-320, 1e300, 1.0 / c, INFINITY, 1e-30};
  int64_t b = 0;
  for (int i = 0; i < 6; ++i) {
    const double v[3] = {w[i], -w[i], w[(i + 1) % 6]};
    b += bad3(bytes, c, v);
  }
  return b;
}
/* the most that the margin's 2.9e-6 is off: largest |y| difference, n points */
double worst_y(int64_t n) {
  double m = 0;
  for (int64_t i = 1; i <= n; ++i) {
    const double x = (double)i / (double)n, z = x * x;
    const double q[11] = {0.000937563612006803, -0.006394792927109298, 0.0204678832131648, -0.042088155301232,
                          0.06541381456030451, -0.08713861532823457, 0.11028651356204722, -0.1427443216339156,
                          0.19999129800465953, -0.3333330208965988, 0.9999999966724514};
    double p = q[0];
    for (int j = 1; j < 11; ++j) p = fma(p, z, q[j]);
    const double d = fabs(x * p - atan(x)) * 65535.0 / (double)CUBE_PI_F;
    m = d > m ? d : m;
  }
  return m;
}
