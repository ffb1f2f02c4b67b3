// line_2f.hip -- line solve, 2x2 blocks, FP32.
#include "line_launch.h"

namespace asam {

void line_2f(hipStream_t s, const Geom& g, const Coef<float>& c, const LineReq& r) {
  if (r.tr) line_t<2, 1, float, float>(s, g, c, r);
  else line_t<2, 0, float, float>(s, g, c, r);
}

}  // namespace asam
