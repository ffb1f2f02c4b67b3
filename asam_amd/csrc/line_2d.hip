// line_2d.hip -- line solve, 2x2 blocks, FP64.
#include "line_launch.h"

namespace asam {

void line_2d(hipStream_t s, const Geom& g, const Coef<double>& c, const LineReq& r) {
  if (r.tr) line_t<2, 1, double, double>(s, g, c, r);
  else line_t<2, 0, double, double>(s, g, c, r);
}

}  // namespace asam
