/* the short atan that cube_encode_v3 uses, as the library has it */
#include <math.h>
#include "../cafproject_amd/csrc/cube_math.h"

/* largest error of x*P(x^2) on (0, 1] in units of a 2-byte code, n points */
double worst_fit(int64_t n) {
  double m = 0;
  for (int64_t i = 1; i <= n; ++i) {
    const double x = (double)i / (double)n, d = fabs(x * cube_atan_poly(x * x) - atan(x)) * 65535.0 / (double)CUBE_PI_F;
    m = d > m ? d : m;
  }
  return m;
}
