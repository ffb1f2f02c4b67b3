// line_1f.hip -- line solve, one component, FP32.
#include "line_launch.h"

namespace asam {

void line_1f(hipStream_t s, const Geom& g, const Coef<float>& c, const LineReq& r) {
  if (r.tr) line_t<1, 1, float, float>(s, g, c, r);
  else line_t<1, 0, float, float>(s, g, c, r);
}

}  // namespace asam
