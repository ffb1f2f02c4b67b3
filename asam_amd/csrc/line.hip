// line.hip -- vertical-line preconditioner solve (gfx950): one thread per column, or per half
// of a column, 64 columns per wavefront (coalesced along x at every level), loads issued a
// window of levels ahead of the recurrence, the elimination's results staged in LDS.
#include "internal.h"

namespace asam {

// ===================================================================== line solve
int line_blocks(const Geom& g) { return ((g.nx + 63) / 64) * g.ny; }

// Dynamic LDS a line-solve workgroup may take: the device's per-workgroup limit minus
// 4 KiB kept for the static reduction scratch.
size_t lds_device_limit() {
  static int cached = -1;
  if (cached < 0) {
    int dev = 0, v = 0;
    if (hipGetDevice(&dev) != hipSuccess ||
        hipDeviceGetAttribute(&v, hipDeviceAttributeMaxSharedMemoryPerBlock, dev) != hipSuccess)
      v = 0;
    cached = v > 4096 ? v - 4096 : 0;
  }
  return (size_t)cached;
}

// Default staging budget per workgroup: at most 60 KiB, so that two or more workgroups share
// a CU.
size_t lds_budget() {
  const size_t d = lds_device_limit();
  return d < 60 * 1024 ? d : 60 * 1024;
}

// Staging budget the line_lds tuning knob names: 0 none, 1 the default, n >= 2 n KiB
// (never more than the device allows).
size_t lds_budget_for(int line_lds) {
  if (line_lds <= 0) return 0;
  if (line_lds == 1) return lds_budget();
  const size_t want = (size_t)line_lds * 1024, d = lds_device_limit();
  return want < d ? want : d;
}

// Levels of each half of a column of nz levels (of the column, for one wavefront per tile)
// staged in LDS within `budget` bytes.
int lds_levels(int nz, int np, size_t word, size_t budget, int halves) {
  const size_t k = budget / ((size_t)halves * 64 * np * word);
  return k >= (size_t)(nz / halves) ? nz / halves : (int)k;
}

// Compiled in line_<block size><precision>.hip.
void line_1d(hipStream_t s, const Geom& g, const Coef<double>& c, const LineReq& r);
void line_1f(hipStream_t s, const Geom& g, const Coef<float>& c, const LineReq& r);
void line_2d(hipStream_t s, const Geom& g, const Coef<double>& c, const LineReq& r);
void line_2f(hipStream_t s, const Geom& g, const Coef<float>& c, const LineReq& r);

void launch_line(hipStream_t s, const Geom& g, const Coef<double>& c64, const Coef<float>& c32,
                 const LineReq& r) {
  if (g.np1 == 1) {
    if (r.prec == 0) line_1d(s, g, c64, r); else line_1f(s, g, c32, r);
  } else {
    if (r.prec == 0) line_2d(s, g, c64, r); else line_2f(s, g, c32, r);
  }
}

}  // namespace asam
