// line_1d.hip -- line solve, one component, FP64.
#include "line_launch.h"

namespace asam {

void line_1d(hipStream_t s, const Geom& g, const Coef<double>& c, const LineReq& r) {
  if (r.tr) line_t<1, 1, double, double>(s, g, c, r);
  else line_t<1, 0, double, double>(s, g, c, r);
}

}  // namespace asam
