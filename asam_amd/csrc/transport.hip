// transport.hip -- gfx950 transport stage solve: BiCGStab over the SpDiag transport
// Jacobian with the forward Gauss-Seidel preconditioner (reference
// SRC/MODULE/SpMatrix4CellPar_Mod.f90:56-348, SRC/CG/MatSpDiag_Mod.f90:95-296,
// SRC/MODULE/Vector4Cell_Mod.f90:605-776, 1120-1340).
//
// Data layout in HBM (one block, haloed extents X = nx+2, Y = ny+2, Z = nz+2, m = X*Y*Z):
//   natural: the reference's arrays, x fastest: Val(m, 7) column-major for JacTMom and
//     JacTPot, Val(m, 2) for JacFall; vectors ncomp x m; LU factors ncomp*ncomp x ncell.
//   skewed (Gauss-Seidel only): level k, y-tile jt of TW columns j, row h = i + jj of
//     the tile (jj the column within it), RW entries per row, one per column: the cells of one
//     step of a wavefront whose lanes are the columns (lane l at cell i = step - l) are one
//     contiguous run.  A matrix holds kCoefWords such runs per row, one after the other.  The
//     skew costs 1 + (TW-1)/X of padding, the rows RW/TW (see Dims).
//
// The Gauss-Seidel sweep is the reference's lexicographic forward sweep.  Cell (i, j, k)
// needs the new values of (i-1), (j-1), (k-1) and the old ones of (i+1), (j+1), (k+1), so
// every cell of the hyperplane i+j+k = h can be updated at once, and the next sweep can
// follow two hyperplanes behind: see k_gs_tiles.
//
// Products and sums are not contracted (no FMA) in the operator, the sweep and the
// vector updates, so they round as the reference's separate multiplies and adds.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <string>
#include <vector>

#include "asam_transport.h"
#include "kcommon.h"

namespace asam {
namespace tr {

constexpr int kMaxComp = ASAM_TR_MAX_COMP;
constexpr int kSpinLimit = 1 << 22;

struct Ops {
  int nc;
  int op[kMaxComp];
  double alpha[kMaxComp];
};

struct Dims {
  int nx, ny, nz, X, Y, Z;
  int TW, NJ, HL;         // skewed layout: columns per y-tile, y-tiles, rows per tile and level
  int RW;                 // entries per row: kRow, or for few columns as many, see create
  int ZW;                 // columns of a boundary record's top level
  long m, ncell, slots;   // slots = Z*NJ*HL*RW
};

// Components that go through the sweeps together, one or two per group: two share a matrix
// (the same operator); a component left over fills both places of its group.
struct Groups {
  int n;
  int c[kMaxComp][2];
};

__device__ __forceinline__ bool is_interior(const Dims& d, long r, int& i, int& j, int& k) {
  if (d.m <= 0xffffffffl) {  // uniform; 32-bit divisions take a quarter of the instructions
    const unsigned u = (unsigned)r, w = u / (unsigned)d.X, z = w / (unsigned)d.Y;
    i = (int)(u - w * (unsigned)d.X);
    j = (int)(w - z * (unsigned)d.Y);
    k = (int)z;
  } else {
    i = (int)(r % d.X);
    const long w = r / d.X;
    j = (int)(w % d.Y);
    k = (int)(w / d.Y);
  }
  return i >= 1 && i <= d.nx && j >= 1 && j <= d.ny && k >= 1 && k <= d.nz;
}

// ------------------------------------------------------------------ operator (MatVec)
// y = x + LU^-1 (T x - x) on interior cells, T x on the halo, for all components at once
// (MatVecChem/Met_Vec4CellSp: SpAVec, Axpy(-1), PSolveMatrix, Xpy).  The 7 (14 with
// JacTMom) coefficients of a cell are read once for every component.  Over the interior cells
// also the sums of y u (nd >= 1) and y y (nd = 2), one partial sum per block: for 4 reacting
// components of 256x256x64 that adds 20 us to the 262 us of the launch, where the dots by
// themselves took 69 us and 82 us.
template <int NC>
__global__ __launch_bounds__(256) void k_matvec(Dims d, const double* __restrict__ tmom,
                                                const double* __restrict__ tpot,
                                                const double* __restrict__ fall,
                                                const double* __restrict__ lu,
                                                const double* __restrict__ x,
                                                double* __restrict__ y, Ops ops, int init,
                                                int use_mom, int use_pot, int nd,
                                                const double* __restrict__ u,
                                                double* __restrict__ partial) {
#pragma clang fp contract(off)
  const long r0 = (long)blockIdx.x * blockDim.x + threadIdx.x;
  const bool live = r0 < d.m;
  if (!live && nd == 0) return;
  const long r = live ? r0 : d.m - 1;
  const long XY = (long)d.X * d.Y;
  const long off[7] = {-XY, -(long)d.X, -1, 0, 1, (long)d.X, XY};
  double vp[7], vm[7];
#pragma unroll
  for (int q = 0; q < 7; ++q) {
    const long src = r + off[q];
    const bool ok = src >= 0 && src < d.m;
    vp[q] = (use_pot && ok) ? tpot[q * d.m + src] : 0.0;
    vm[q] = (use_mom && ok) ? tmom[q * d.m + src] : 0.0;
  }
  double s[NC];
#pragma unroll
  for (int c = 0; c < NC; ++c) {
    const double* xc = x + c * d.m;
    const int op = init ? ASAM_TR_POT : ops.op[c];
    const double* v = (op == ASAM_TR_MOM) ? vm : vp;
    double acc = 0.0;
#pragma unroll
    for (int q = 0; q < 7; ++q) {
      const long src = r + off[q];
      if (src >= 0 && src < d.m) acc += v[q] * xc[src];
    }
    if (op == ASAM_TR_FALL) {  // SpABVec: JacFall (offsets 0, XY) scaled by ScaleMat2
      acc += (fall[r] * ops.alpha[c]) * xc[r];
      if (r + XY < d.m) acc += (fall[d.m + r + XY] * ops.alpha[c]) * xc[r + XY];
    }
    s[c] = -1.0 * xc[r] + acc;
  }
  int i = 0, j = 0, k = 0;
  const bool in = (lu || nd > 0) && is_interior(d, r, i, j, k);
  if (lu && in) {
    const long q = (i - 1) + (long)d.nx * ((j - 1) + (long)d.ny * (k - 1));
#pragma unroll
    for (int kc = 0; kc < NC; ++kc)
#pragma unroll
      for (int ic = kc + 1; ic < NC; ++ic)
        s[ic] = s[ic] - lu[((long)ic * NC + kc) * d.ncell + q] * s[kc];
#pragma unroll
    for (int kc = NC - 1; kc >= 0; --kc) {
      s[kc] = s[kc] / lu[((long)kc * NC + kc) * d.ncell + q];
#pragma unroll
      for (int ic = 0; ic < kc; ++ic)
        s[ic] = s[ic] - lu[((long)ic * NC + kc) * d.ncell + q] * s[kc];
    }
  }
  double acc[2] = {0.0, 0.0};
#pragma unroll
  for (int c = 0; c < NC; ++c) {
    const double yc = x[c * d.m + r] + s[c];
    if (live) y[c * d.m + r] = yc;
    if (nd > 0 && live && in) {
      acc[0] = __builtin_fma(yc, u[c * d.m + r], acc[0]);
      acc[1] = __builtin_fma(yc, yc, acc[1]);
    }
  }
  if (nd > 0) block_reduce_store<2>(acc, partial, blockIdx.x, threadIdx.x, 256, gridDim.x);
}

// ------------------------------------------------------------------ division
// t / dg from y = 1/dg (correctly rounded): two residual corrections of t*y.  The first leaves
// a quotient within an ulp and the second rounds correctly (Markstein, IBM J. Res. Dev. 34,
// 1990), as long as no residual underflows, which |t| of 2^-960 and more ensures: |dg| of 2^-60
// and more (to 2^500; the set-up notes a matrix with another diagonal, and the sweeps then
// divide) and quotients of 2^-900 and more.  Five dependent operations in the sweep's serial
// chain instead of the division's dozen.  The sign is that of t*y, also for a zero.
__device__ __forceinline__ double gs_divide(double t, double dg, double y) {
  const double q0 = t * y;
  const double q1 = __builtin_fma(__builtin_fma(-q0, dg, t), y, q0);
  const double q2 = __builtin_fma(__builtin_fma(-q1, dg, t), y, q1);
  return __builtin_copysign(q2, q0);
}
// The caller divides where the quotient of a t other than zero is below 2^-900, infinite or NaN:
// where this is at least kOddKey (the high word without its sign, from 2^-900 on; smaller ones
// wrap).  A maximum of such keys takes vector instructions only: as comparisons joined in scalar
// registers the test cost 2% of the launch at 256x256x64, this way 0.5%.
constexpr unsigned kOddLow = 2 * (1023u - 900u) << 20, kOddKey = (2 * 2047u << 20) - kOddLow;
__device__ __forceinline__ unsigned gs_key(double t, double q) {
  const unsigned u = ((unsigned)__double2hiint(q) << 1) - kOddLow;
  return t != 0.0 ? u : 0u;
}
__device__ __forceinline__ bool gs_plain_diag(double dg) {
  const double m = fabs(dg);
  return m >= 0x1p-60 && m <= 0x1p500;
}

// ------------------------------------------------------------------ skewed layout
// Slot of cell (i, j, k) within an array of one word per cell: y-tile jt = j / TW, column
// jj = j - jt*TW, row h = i + jj of the tile's HL rows (X + TW - 1; X + Y - 1 for one tile).
constexpr int kCoefWords = 8;  // words per cell of a skewed matrix: see k_skew_coef
constexpr int kMaxCols = 53;   // columns of a y-tile at most, see kMaxSweeps below
// Entries of a row of the skewed layout for tiles of 27 columns and more.  Rows of 56 (the most
// that a tile needs, in whole 128-byte lines) would take less memory and more time: an
// application at 256x256x64, four components, 1346 us against 1330, a sweep of 101x77x50 with
// JacFall 42.4 against 41.3.
constexpr int kRow = 64;

// Place of word q of a cell within a matrix row: the words lie in pairs, so that a lane takes
// two with one 16-byte load (a wavefront's load costs the address unit the same 16 cycles
// whatever its width).
__device__ __forceinline__ int coef_word(int RW, int q) { return (q >> 1) * (2 * RW) + (q & 1); }

__device__ __forceinline__ long slot_row(const Dims& d, int jt, int h, int k) {
  return ((long)k * d.NJ + jt) * d.HL + h;
}

// Natural rows j of one (level, y-tile) to skewed rows h, 64 rows h at a time: the loads run
// along x, the stores along y, transposed through LDS (a thread per cell would scatter one
// of the two).  get(jj, i) gives the value of cell (i, j0 + jj); put(h, jj, v) stores it.
// Slots outside the block (i out of range) are not written and never used.
constexpr int kTileH = 64;
__host__ __device__ inline int h_blocks(const Dims& d) { return (d.HL + kTileH - 1) / kTileH; }
template <typename Get, typename Put>
__device__ __forceinline__ void skew_tile(const Dims& d, int jt, int h0, double (*t)[kTileH + 1],
                                          Get&& get, Put&& put) {
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int rows = min(d.TW, d.Y - jt * d.TW);
  for (int jj = wv; jj < rows; jj += 4) {
    const int i = h0 + lane - jj;
    if (i >= 0 && i < d.X) t[jj][lane] = get(jj, i);
  }
  __syncthreads();
  for (int hh = wv; hh < kTileH; hh += 4) {
    const int h = h0 + hh, i = h - lane;
    if (lane < rows && h < d.HL && i >= 0 && i < d.X) put(h, lane, t[lane][hh]);
  }
  __syncthreads();
}

// Row coefficients A(r, r + DiagPtr(q)) = Val(r + DiagPtr(q), q) of every cell, in the order
// the sweep uses them: +1, +X, +XY, -XY, -X, -1, diagonal, and the diagonal's reciprocal.  A coupling that leaves the block is +0 (the set-up has checked that it is
// zero; its sign must not reach the sweep's sums).  Grid (y-tiles x runs of 64 h, 1, levels).
// *odd is set where a diagonal is too large or too small for gs_divide.
__global__ __launch_bounds__(256) void k_skew_coef(Dims d, const double* __restrict__ val,
                                                   double* __restrict__ w, int* odd) {
  __shared__ double t[64][kTileH + 1];
  const int nh = h_blocks(d), jt = blockIdx.x / nh, h0 = (blockIdx.x - jt * nh) * kTileH;
  const int k = blockIdx.z;
  const int di[7] = {1, 0, 0, 0, 0, -1, 0}, dj[7] = {0, 1, 0, 0, -1, 0, 0},
            dk[7] = {0, 0, 1, -1, 0, 0, 0}, dq[7] = {4, 5, 6, 0, 1, 2, 3};
#pragma unroll
  for (int q = 0; q < 7; ++q) {
    skew_tile(
        d, jt, h0, t,
        [&](int jj, int i) {
          const int i2 = i + di[q], j2 = jt * d.TW + jj + dj[q], k2 = k + dk[q];
          const bool in = i2 >= 0 && i2 < d.X && j2 >= 0 && j2 < d.Y && k2 >= 0 && k2 < d.Z;
          return in ? val[(long)dq[q] * d.m + i2 + (long)d.X * (j2 + (long)d.Y * k2)] : 0.0;
        },
        [&](int h, int jj, double v) {
          double* row = w + slot_row(d, jt, h, k) * (kCoefWords * d.RW) + 2 * jj;
          row[coef_word(d.RW, q)] = v;
          if (q == 6) {
            row[coef_word(d.RW, 7)] = 1.0 / v;
            if (!gs_plain_diag(v)) *odd = 1;
          }
        });
  }
}
// JacFall rows: word 0 its diagonal, word 1 its coupling of row r to r + XY.
__global__ __launch_bounds__(256) void k_skew_fall(Dims d, const double* __restrict__ fall,
                                                   double* __restrict__ wf) {
  __shared__ double t[64][kTileH + 1];
  const int nh = h_blocks(d), jt = blockIdx.x / nh, h0 = (blockIdx.x - jt * nh) * kTileH;
  const int k = blockIdx.z;
#pragma unroll
  for (int q = 0; q < 2; ++q)
    skew_tile(
        d, jt, h0, t,
        [&](int jj, int i) {
          const int k2 = k + q;
          return k2 < d.Z ? fall[q * d.m + i + (long)d.X * (jt * d.TW + jj + (long)d.Y * k2)] : 0.0;
        },
        [&](int h, int jj, double v) {
          wf[slot_row(d, jt, h, k) * (2 * d.RW) + 2 * jj + q] = v;
        });
}
// A vector to the skewed layout, the NC components of a group together (they lie side by side
// there), kVecH rows h per block: half a wavefront loads a run of kVecH cells along x of one
// column, the loads of all columns in flight together, and a wavefront stores a row.  Bound by
// memory.  With one component per block the loads and stores of the skewed side move half of
// each 16 bytes: 4 components of 256x256x64 took 120 us (k_skew_vec) and 189 us (k_unskew),
// now 54 us and 56 us (4.9 TB/s).
// Grid (y-tiles x runs of kVecH rows, 1, levels x groups).
constexpr int kVecH = 32;
template <int NC>
__global__ __launch_bounds__(256) void k_skew_vec(Dims d, Groups gr, const double* __restrict__ v,
                                                  double* __restrict__ vs) {
  __shared__ double t[NC][kMaxCols][kVecH + 1];
  const int nh = (d.HL + kVecH - 1) / kVecH, jt = blockIdx.x / nh, h0 = (blockIdx.x - jt * nh) * kVecH;
  const int g = blockIdx.z / d.Z, k = blockIdx.z - g * d.Z;
  const int rows = min(d.TW, d.Y - jt * d.TW);
  {
    const int l = threadIdx.x & (kVecH - 1), r0 = threadIdx.x / kVecH;
    constexpr int RP = 256 / kVecH, NR = (kMaxCols + RP - 1) / RP;
    double x[NR][NC];
#pragma unroll
    for (int q = 0; q < NR; ++q) {
      const int jj = r0 + q * RP, i = h0 + l - jj;
      const bool in = jj < rows && i >= 0 && i < d.X;
      const long cell = i + (long)d.X * (jt * d.TW + jj + (long)d.Y * k);
#pragma unroll
      for (int n = 0; n < NC; ++n) x[q][n] = in ? v[(long)gr.c[g][n] * d.m + cell] : 0.0;
    }
#pragma unroll
    for (int q = 0; q < NR; ++q) {
      const int jj = r0 + q * RP;
      if (jj < rows) {
#pragma unroll
        for (int n = 0; n < NC; ++n) t[n][jj][l] = x[q][n];
      }
    }
  }
  __syncthreads();
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  double* const dst = vs + g * d.slots * NC;
  for (int hh = wv; hh < kVecH; hh += 4) {
    const int h = h0 + hh, i = h - lane;
    if (lane < rows && h < d.HL && i >= 0 && i < d.X) {
      double* const p = dst + (slot_row(d, jt, h, k) * d.RW + lane) * NC;
      if constexpr (NC == 2)
        *reinterpret_cast<double2*>(p) = make_double2(t[0][lane][hh], t[1][lane][hh]);
      else
        *p = t[0][lane][hh];
    }
  }
}
// Back to the natural layout with the six halo faces zero (PSolveSp :734-739), kVecH cells
// along x of every column per block.  Grid (y-tiles x runs of kVecH cells along x, 1, levels x
// groups).
template <int NC>
__global__ __launch_bounds__(256) void k_unskew(Dims d, Groups gr, const double* __restrict__ vs,
                                                double* __restrict__ v) {
  // cell i0 + l of column jj at 34 jj + l: a wavefront writes 33 jj + const, its own bank each
  __shared__ double t[NC][kMaxCols][kVecH + 2];
  const int nx = (d.X + kVecH - 1) / kVecH, jt = blockIdx.x / nx;
  const int i0 = (blockIdx.x - jt * nx) * kVecH;
  const int g = blockIdx.z / d.Z, k = blockIdx.z - g * d.Z;
  const int rows = min(d.TW, d.Y - jt * d.TW);
  const bool inner_k = k >= 1 && k <= d.nz;
  if (inner_k) {
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const double* src = vs + g * d.slots * NC;
    constexpr int NH = (kVecH + kMaxCols - 1 + 3) / 4;  // rows h of a wavefront
    double x[NH][NC];
#pragma unroll
    for (int q = 0; q < NH; ++q) {
      const int l = wv + 4 * q - lane, h = i0 + wv + 4 * q;
      const bool in = lane < rows && l >= 0 && l < kVecH && i0 + l < d.X;
      const double* const p = src + (slot_row(d, jt, h, k) * d.RW + lane) * NC;
#pragma unroll
      for (int n = 0; n < NC; ++n) x[q][n] = 0.0;
      if (in) {
        if constexpr (NC == 2) {
          const double2 w = *reinterpret_cast<const double2*>(p);
          x[q][0] = w.x;
          x[q][1] = w.y;
        } else {
          x[q][0] = *p;
        }
      }
    }
#pragma unroll
    for (int q = 0; q < NH; ++q) {
      const int l = wv + 4 * q - lane;
      if (lane < rows && l >= 0 && l < kVecH) {
#pragma unroll
        for (int n = 0; n < NC; ++n) t[n][lane][l] = x[q][n];
      }
    }
  }
  __syncthreads();
  const int l = threadIdx.x & (kVecH - 1), i = i0 + l;
  if (i >= d.X) return;
  for (int jj = threadIdx.x / kVecH; jj < rows; jj += 256 / kVecH) {
    const int j = jt * d.TW + jj;
    const bool in = inner_k && i >= 1 && i <= d.nx && j >= 1 && j <= d.ny;
#pragma unroll
    for (int n = 0; n < NC; ++n)
      v[(long)gr.c[g][n] * d.m + i + (long)d.X * (j + (long)d.Y * k)] = in ? t[n][jj][l] : 0.0;
  }
}

__global__ void k_zero_int(int* p, int n) {
  const int e = blockIdx.x * blockDim.x + threadIdx.x;
  if (e < n) p[e] = 0;
}

// ------------------------------------------------------------------ Gauss-Seidel sweeps
// Sweeps one launch runs at most: six wavefronts, the polling and the storing one; two such
// blocks fit a CU.
constexpr int kMaxSweeps = 6;
// Columns of a y-tile at most (kMaxCols): a step's values of the top level of a block are five
// runs of 64 (64 columns would take six, and the spare lanes cost less than the extra polls).
constexpr unsigned long long kSentinel = 0xFFF7DEADBEEF0001ull;  // NaN payload: not yet

struct GsArgs {
  Dims d;
  const double* wmom;   // skewed matrices (k_skew_coef)
  const double* wpot;
  const double* wf;     // JacFall rows
  const double* bs;     // groups x slots x NC: right-hand side
  const double* ts;     // groups x slots x NC: right-hand side of the first sweep's substitution
  double* xs;           // groups x slots x NC: result of the last sweep
  double* bnd;          // groups x [block][step]: boundary records
  const int* order;     // blocks (jt + NJ*kb) in the order they are taken
  int* counter;         // ticket
  int* err;             // set when a wait gives up
  int NK, M;
  Groups groups;
  int nsteps;           // X + TW + KR - 2
  int spin_limit;       // polls of a boundary value before a block gives up
  int hold;             // test hook: no block publishes its boundary
};

// t = b - U x_old on every cell (the first sweep of a launch that continues earlier ones).
template <int NC>
__global__ __launch_bounds__(256) void k_gs_upart(GsArgs a, Ops ops, double* __restrict__ tw) {
#pragma clang fp contract(off)
  const Dims& d = a.d;
  const int lane = threadIdx.x & 63;
  const int nh = (d.HL + 3) / 4, jt = blockIdx.x / nh;
  const int h = (blockIdx.x - jt * nh) * 4 + (threadIdx.x >> 6);
  const int q = blockIdx.z / d.Z, k = blockIdx.z - q * d.Z, g = q / NC, n = q - g * NC;
  const int c = a.groups.c[g][n];
  const int j = jt * d.TW + lane, i = h - lane;
  if (h >= d.HL || lane >= d.TW || j >= d.Y || i < 0 || i >= d.X) return;
  const long base = g * d.slots * NC + n;
  const double* const x = a.xs + base;
  const long row = slot_row(d, jt, h, k), e = row * d.RW + lane;
  const double* const w =
      (ops.op[c] == ASAM_TR_MOM ? a.wmom : a.wpot) + row * (kCoefWords * d.RW) + 2 * lane;
  double t = a.bs[base + e * NC];
  if (i + 1 < d.X) t = t - w[coef_word(d.RW, 0)] * x[(e + d.RW) * NC];
  if (j + 1 < d.Y) {
    // the next column: in this tile one row on, or the first of the next tile, row i
    const long e2 = lane + 1 < d.TW ? e + d.RW + 1 : slot_row(d, jt + 1, i, k) * d.RW;
    t = t - w[coef_word(d.RW, 1)] * x[e2 * NC];
  }
  if (k + 1 < d.Z) {
    const double xz = x[(e + (long)d.NJ * d.HL * d.RW) * NC];
    t = t - w[coef_word(d.RW, 2)] * xz;
    if (ops.op[c] == ASAM_TR_FALL)
      t = t - (a.wf[row * (2 * d.RW) + 2 * lane + 1] * ops.alpha[c]) * xz;
  }
  tw[base + e * NC] = t;
}

__global__ __launch_bounds__(256) void k_gs_reset(unsigned long long* p, long n,
                                                  unsigned long long v, int* ticket) {
  if (blockIdx.x == 0 && threadIdx.x == 0) *ticket = 0;
  const long e = 2 * ((long)blockIdx.x * blockDim.x + threadIdx.x);
  if (e + 1 < n) *reinterpret_cast<ulonglong2*>(p + e) = make_ulonglong2(v, v);
  else if (e < n) p[e] = v;
}

__device__ __forceinline__ bool is_sentinel(double v) {
  // no arithmetic gives this payload: the high word is enough
  return __double2hiint(v) == (int)(kSentinel >> 32);
}

// All sweeps of a preconditioner application in one launch.
//
// In the hyperplane order cell (i, j, k) of sweep s can be updated at time T = i + j + k + 2s:
// its new -x, -y, -z neighbours are done at T - 1, and so are the old +x, +y, +z ones, sweep
// s - 1 at T - 1.  So the sweeps follow each other two steps apart and the whole application
// takes X + Y + Z + 2M steps instead of M times X + Y + Z.
//  - A block owns TW columns j by KR levels k of every sweep and marches along x.  Sweep s of
//    block (jt, kb) covers columns jt*TW - s + l (lane l) and levels kb*KR - s + r: shifted by
//    one in both per sweep, so a block needs values of the blocks before it in j and k only.
//    At the block's step T every sweep is at cell i = T - l - r.
//  - One wavefront per sweep; a lane computes the KR levels of its column, for NC components
//    that share their matrix (their coefficients are loaded once).  A step's values pass to
//    the next step through LDS (double buffered, one barrier per step): the wavefront's own
//    for the -y neighbour, sweep s - 1's for the old neighbours.  x_old is never read from
//    memory, and only the last sweep is stored.
//  - Sweep s reads a cell's coefficients two steps after sweep s - 1, from the caches.  A lane
//    refills a level's registers for D steps ahead as soon as it has used them.
//  - A block's top level and last column go to its successors through a record per step,
//    pre-filled with a NaN-payload sentinel and written and read past the caches that are not
//    coherent between XCDs: a value that is not the sentinel is final, so no fence or flag
//    orders them.  One wavefront per block requests the predecessors' values PF steps ahead
//    and puts them in LDS beside the block's own; one stores the block's.  (A store's
//    acknowledgement counts like a load's, so a computing wavefront that stored would wait
//    for it before it could use the loads it issues afterwards.)
//  - Blocks are taken from an atomic ticket in an order in which a block's predecessors come
//    first, so a block waits only for blocks that started before it; every wait is bounded.
//
// What bounds it: the chain of X + Y + Z + 2M steps.  256x256x64, four components, 6 sweeps:
// 1.16 ms for 594 steps, 1.96 us each with the hand-overs between blocks counted in; the
// coefficient loads (28 cycles of the L1 per 16-byte load of a wavefront) take as much of a step
// as the arithmetic, and a block waits for the slowest step of those before it.  One launch per
// sweep with a pass for b - U x_old before it, rows handed over along y, took 4.3 ms.
// 101x77x50, three components: 0.24 ms against 2.1 ms.
//
// Term order of a row as in the reference (GaussSeidel_SpDiag :216-234): b, -U (+1, +X, +XY,
// then JacFall's +XY), -L (-XY, -X, -1), / diag; products and sums are not contracted.  A
// coupling that leaves the block is +0 and so is the value there, so it changes no sum.
constexpr int kLdsRow = 66;     // column -1, 64 columns, pad
constexpr int kZWords = (kMaxSweeps * kMaxCols + 63) / 64;  // runs of 64 in a record's top level
constexpr int PF = 2;           // steps ahead that a block's boundary values are requested
constexpr int kSc1 = 16;        // buffer access: to the coherence point of the device

typedef unsigned u32x2 __attribute__((ext_vector_type(2)));
typedef unsigned u32x4 __attribute__((ext_vector_type(4)));

// The values of NC components at one place.
template <int NC>
struct alignas(8 * NC) Val {
  double c[NC];
};
template <int NC>
__device__ __forceinline__ Val<NC> buf_load(__amdgpu_buffer_rsrc_t r, int off) {
  if constexpr (NC == 1)
    return __builtin_bit_cast(Val<NC>, __builtin_amdgcn_raw_buffer_load_b64(r, off, 0, kSc1));
  else
    return __builtin_bit_cast(Val<NC>, __builtin_amdgcn_raw_buffer_load_b128(r, off, 0, kSc1));
}
template <int NC>
__device__ __forceinline__ void buf_store(__amdgpu_buffer_rsrc_t r, int off, Val<NC> v) {
  if constexpr (NC == 1)
    __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u32x2, v), r, off, 0, kSc1);
  else
    __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, v), r, off, 0, kSc1);
}
template <int NC>
__device__ __forceinline__ bool any_sentinel(const Val<NC>& v) {
  bool m = false;
#pragma unroll
  for (int q = 0; q < NC; ++q) m |= is_sentinel(v.c[q]);
  return m;
}

// DIV: divide by the diagonal (a matrix with an unusual one, or JacFall in it) instead of
// multiplying by its reciprocal.  ROW: entries of a row, 0: as in Dims (the places of a row's
// pairs then take scalar registers and instructions that constants do not: 1.7% of the launch
// at 256x256x64, 4.5% at 101x77x50 with JacFall).
template <int NC, int KR, int D, bool FALL, bool DIV, int ROW, typename OFF>
__global__ __launch_bounds__(512, 2) void k_gs_tiles(GsArgs a, Ops ops) {
#pragma clang fp contract(off)
  using V = Val<NC>;
  extern __shared__ __attribute__((aligned(16))) double lds_raw[];
  V* const lds = reinterpret_cast<V*>(lds_raw);  // [2][M][KR + 1][kLdsRow], level -1, column -1 first
  __shared__ int s_ticket;
  const Dims& d = a.d;
  const int RW = ROW ? ROW : d.RW;
  const int lane = threadIdx.x & 63, M = a.M, TW = d.TW, X = d.X;
  const int s = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  constexpr int kWave = (KR + 1) * kLdsRow;
  const int half = M * kWave;
  for (int e = threadIdx.x; e < 2 * half * NC; e += blockDim.x) lds_raw[e] = 0.0;
  if (threadIdx.x == 0) s_ticket = atomicAdd(a.counter, 1);
  __syncthreads();
  const int ticket = __builtin_amdgcn_readfirstlane(s_ticket);
  const int g = ticket % a.groups.n, blk = a.order[ticket / a.groups.n];
  const int jt = blk % d.NJ, kb = blk / d.NJ;
  const int nsteps = a.nsteps, steps = (nsteps + PF - 1) / PF * PF;
  // a record: top level [sweep][column], last column [sweep][level], NC values each; a single
  // tile has no successor in y, and sweep s has its Y columns at lanes s and up
  const int ZW = d.ZW, zshift = d.NJ == 1 ? 1 : 0;
  const int zrec = M * ZW * NC, yrec = M * KR * NC;
  const long rec = zrec + (d.NJ == 1 ? 0 : yrec), brec = nsteps * rec;
  const long nblk = (long)d.NJ * a.NK;
  double* const bnd = a.bnd + g * nblk * brec;

  if (s == M) {  // the polling wavefront
    const int zlast = kb > 0 ? nsteps - 1 - KR : -2;  // values exist up to this time
    const double* const zrow = bnd + (kb > 0 ? blk - d.NJ : blk) * brec + KR * rec;
    int zdst[kZWords];
#pragma unroll
    for (int q = 0; q < kZWords; ++q) {
      const int e = lane + 64 * q, w = e / ZW;
      // or a pad entry
      zdst[q] = e < M * ZW ? w * kWave + e - w * (ZW - zshift) + 1 : kLdsRow - 1;
    }
    // the column values, and those of level -1 beside them
    int f = lane, ylast = -2, ydst = (kLdsRow - 1) * NC;
    const double* yptr = bnd + blk * brec;
    if (f < yrec) {
      const int c = f % NC, e = f / NC, w = e / KR, r = e - w * KR;
      ydst = (w * kWave + (r + 1) * kLdsRow) * NC + c;
      if (jt > 0) {
        yptr = bnd + (blk - 1) * brec + TW * rec + zrec + f;
        ylast = nsteps - 1 - TW;
      }
    } else if ((f -= yrec) < M * NC) {
      const int c = f % NC, w = f / NC;
      ydst = w * kWave * NC + c;
      if (jt > 0 && kb > 0) {
        yptr = bnd + (blk - d.NJ - 1) * brec + (TW + KR) * rec + (w * TW + TW - 1) * NC + c;
        ylast = nsteps - 1 - TW - KR;
      }
    }
    struct Poll {
      V z[kZWords];
      double y;
    };
    bool broken = false;
    // the values of time th, requested / checked and put in LDS
    auto issue = [&](int th, Poll& p) {
      const __amdgpu_buffer_rsrc_t r = __builtin_amdgcn_make_buffer_rsrc(
          const_cast<double*>(zrow + (th <= zlast ? th : 0) * rec), 0, zrec * 8, 0x00020000);
#pragma unroll
      for (int q = 0; q < kZWords; ++q) p.z[q] = buf_load<NC>(r, (lane + 64 * q) * (8 * NC));
      p.y = __hip_atomic_load(yptr + (th <= ylast ? th * rec : 0), __ATOMIC_RELAXED,
                              __HIP_MEMORY_SCOPE_AGENT);
    };
    auto missing = [&](int th, const Poll& p) {
      bool m = (th <= ylast) & is_sentinel(p.y);
      if (th <= zlast) {
#pragma unroll
        for (int q = 0; q < kZWords; ++q) m |= any_sentinel(p.z[q]);
      }
      return __ballot(m) != 0;
    };
    auto settle = [&](int th, Poll& p) {
      if (missing(th, p) && !broken) {
#pragma clang loop unroll(disable)
        for (int n = 0;; ++n) {
          if (n >= a.spin_limit) {
            __hip_atomic_store(a.err, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            broken = true;
            break;
          }
          __builtin_amdgcn_s_sleep(1);
          issue(th, p);
          if (!missing(th, p)) break;
        }
        // nothing is outstanding here, which the compiler cannot see: without this it would
        // drain the requests ahead on the common path too
        __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0)
      }
      V* const L = lds + (th & 1) * half;
#pragma unroll
      for (int q = 0; q < kZWords; ++q) {
        V v = p.z[q];
        if (th > zlast) v = V{};
        L[zdst[q]] = v;
      }
      reinterpret_cast<double*>(L)[ydst] = th <= ylast ? p.y : 0.0;
    };
    Poll buf[PF];
    issue(-1, buf[0]);
    settle(-1, buf[0]);
#pragma unroll
    for (int u = 0; u < PF; ++u) issue(u, buf[u]);
    __syncthreads();
    for (int T0 = 0; T0 < steps; T0 += PF) {
#pragma unroll
      for (int u = 0; u < PF; ++u) {
        settle(T0 + u, buf[u]);
        issue(T0 + u + PF, buf[u]);
        __syncthreads();
      }
    }
    return;
  }

  if (s == M + 1) {  // the storing wavefront: the block's records and the last sweep's result
    const bool pub_z = kb + 1 < a.NK && !a.hold;
    const bool pub_y = jt + 1 < d.NJ && !a.hold && lane < yrec;
    int zsrc[kZWords];
#pragma unroll
    for (int q = 0; q < kZWords; ++q) {
      const int e = lane + 64 * q, w = e / ZW;
      zsrc[q] = e < M * ZW ? w * kWave + KR * kLdsRow + e - w * (ZW - zshift) + 1 : 0;
    }
    const int ye = lane / NC, yw = ye / KR, yr = ye - yw * KR;
    const int ysrc = pub_y ? (yw * kWave + (yr + 1) * kLdsRow + TW) * NC + lane % NC : 0;
    double* out = bnd + blk * brec;
    const int z = M - 1, j = jt * TW - z + lane;
    const OFF off = ((lane < z ? (OFF)TW : (OFF)d.HL) * RW + (lane < z ? lane - z + TW : lane - z)) *
                    (8 * NC);
    double* const xs = a.xs + g * d.slots * NC;
    bool cell[KR];
#pragma unroll
    for (int r = 0; r < KR; ++r) {
      const int k = kb * KR - z + r;
      cell[r] = (lane < TW) & (j >= 0) & (j < d.Y) & (k >= 0) & (k < d.Z);
    }
    __syncthreads();
    for (int T = 0; T < steps; ++T) {
      __syncthreads();  // step T is in LDS
      const V* const L = lds + (T & 1) * half;
      if (T < nsteps) {
        if (pub_z) {
          const __amdgpu_buffer_rsrc_t r =
              __builtin_amdgcn_make_buffer_rsrc(out, 0, zrec * 8, 0x00020000);
#pragma unroll
          for (int q = 0; q < kZWords; ++q)
            buf_store<NC>(r, (lane + 64 * q) * (8 * NC), L[zsrc[q]]);  // past zrec: dropped
        }
        if (pub_y)
          __hip_atomic_store(out + zrec + lane, reinterpret_cast<const double*>(L)[ysrc],
                             __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        out += rec;
      }
#pragma unroll
      for (int r = 0; r < KR; ++r) {
        const int k = min(max(kb * KR - z + r, 0), d.Z - 1);
        char* const row =
            reinterpret_cast<char*>(xs + slot_row(d, jt - 1, T - r - z, k) * (RW * NC));
        if (cell[r] & ((unsigned)(T - lane - r) < (unsigned)X))
          *reinterpret_cast<V*>(row + off) = L[z * kWave + (r + 1) * kLdsRow + lane + 1];
      }
    }
    return;
  }

  const int j = jt * TW - s + lane;
  const int k0 = kb * KR - s;
  bool col_ok[KR];
#pragma unroll
  for (int r = 0; r < KR; ++r)
    col_ok[r] = (lane < TW) & (j >= 0) & (j < d.Y) & (k0 + r >= 0) & (k0 + r < d.Z);
  const int op = ops.op[a.groups.c[g][0]];
  const bool fall = FALL && op == ASAM_TR_FALL;
  double alpha[NC];
#pragma unroll
  for (int c = 0; c < NC; ++c) alpha[c] = FALL ? ops.alpha[a.groups.c[g][c]] : 0.0;
  const double* const W = op == ASAM_TR_MOM ? a.wmom : a.wpot;
  const double* const B = (s == 0 ? a.ts : a.bs) + g * d.slots * NC;
  // Byte offset of the lane's column from row (jt - 1, h) of a level: the columns before the
  // tile's first lie in tile jt - 1, TW rows on.
  const OFF rowl = lane < s ? TW : d.HL;
  const int col = lane < s ? lane - s + TW : lane - s;
  const OFF offw = (rowl * (kCoefWords * RW) + 2 * col) * 8, offb = (rowl * RW + col) * (8 * NC);
  const OFF offf = (rowl * (2 * RW) + 2 * col) * 8;
  // lanes without a cell load the first column of the lane-independent row instead (in the
  // arrays or their guard rows)
  const OFF sfw = (OFF)d.HL * (kCoefWords * RW * 8), sfb = (OFF)d.HL * (RW * 8 * NC),
            sff = (OFF)d.HL * (2 * RW * 8);
  struct Level {
    double w[kCoefWords], f0, f1;
    V b;
    bool ok;
  };
  auto at = [](const double* p, OFF off) { return reinterpret_cast<const char*>(p) + off; };
  auto load = [&](int T, int r, Level& v) {
    const bool ok = col_ok[r] & ((unsigned)(T - lane - r) < (unsigned)X);
    const long row = slot_row(d, jt - 1, T - r - s, min(max(k0 + r, 0), d.Z - 1));
    const double* const pw = W + row * (kCoefWords * RW);
    const OFF ow = ok ? offw : sfw;
#pragma unroll
    for (int q = 0; q < kCoefWords; q += 2) {
      const double2 x = *reinterpret_cast<const double2*>(at(pw + coef_word(RW, q), ow));
      v.w[q] = x.x;
      v.w[q + 1] = x.y;
    }
    if constexpr (FALL) {
      const double2 x =
          *reinterpret_cast<const double2*>(at(a.wf + row * (2 * RW), ok ? offf : sff));
      v.f0 = x.x;
      v.f1 = x.y;
    }
    v.b = *reinterpret_cast<const V*>(at(B + row * (RW * NC), ok ? offb : sfb));
    v.ok = ok;
  };
  Level lv[D][KR];
  V cur[KR];
#pragma unroll
  for (int r = 0; r < KR; ++r) {
    cur[r] = V{};
#pragma unroll
    for (int u = 0; u < D; ++u) load(u, r, lv[u][r]);
  }
  __syncthreads();
  // the steps of a sweep with or without old values (the first one starts from x = 0)
  auto march = [&](auto old_values) {
    constexpr bool OLD = decltype(old_values)::value;
    for (int T0 = 0; T0 < steps; T0 += 2) {
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        const V* const P = lds + ((u + 1) & 1) * half + s * kWave + lane;  // column l - 1
        const V* const O = P - kWave;                                      // sweep s - 1
        V* const L = lds + (u & 1) * half + s * kWave + lane + 1;
        Level(&v)[KR] = lv[u % D];
        // the chains of all levels and components side by side, without a branch
        double t[KR][NC], x[KR][NC];
        unsigned most = 0;
#pragma unroll
        for (int r = 0; r < KR; ++r) {
          V o0, o1, o2;
          if constexpr (OLD) {
            o0 = O[r * kLdsRow];
            o1 = O[r * kLdsRow + 1];
            o2 = O[(r + 1) * kLdsRow];
          }
          const V below = r == 0 ? P[1] : cur[r > 0 ? r - 1 : 0], west = P[(r + 1) * kLdsRow];
#pragma unroll
          for (int c = 0; c < NC; ++c) {
            double tt = v[r].b.c[c];
            if constexpr (OLD) {
              tt = tt - v[r].w[0] * o0.c[c];
              tt = tt - v[r].w[1] * o1.c[c];
              tt = tt - v[r].w[2] * o2.c[c];
              if (FALL && fall) tt = tt - (v[r].f1 * alpha[c]) * o2.c[c];
            }
            tt = tt - v[r].w[3] * below.c[c];
            tt = tt - v[r].w[4] * west.c[c];
            tt = tt - v[r].w[5] * cur[r].c[c];
            t[r][c] = tt;
          }
        }
#pragma unroll
        for (int r = 0; r < KR; ++r) {
          unsigned key = 0;
#pragma unroll
          for (int c = 0; c < NC; ++c) {
            if constexpr (DIV) {
              double dg = v[r].w[6];
              if (FALL && fall) dg = dg + v[r].f0 * alpha[c];
              x[r][c] = t[r][c] / dg;
            } else {
              x[r][c] = gs_divide(t[r][c], v[r].w[6], v[r].w[7]);
              key = max(key, gs_key(t[r][c], x[r][c]));
            }
          }
          most = max(most, v[r].ok ? key : 0u);
        }
        if (!DIV && __builtin_expect(__ballot(most >= kOddKey) != 0, 0)) {
#pragma unroll
          for (int r = 0; r < KR; ++r)
#pragma unroll
            for (int c = 0; c < NC; ++c) x[r][c] = t[r][c] / v[r].w[6];
        }
#pragma unroll
        for (int r = 0; r < KR; ++r) {
#pragma unroll
          for (int c = 0; c < NC; ++c) cur[r].c[c] = v[r].ok ? x[r][c] : 0.0;
          L[(r + 1) * kLdsRow] = cur[r];
          load(T0 + u + D, r, v[r]);
        }
        __syncthreads();
      }
    }
  };
  if (s > 0) march(std::true_type{});
  else march(std::false_type{});
}

// ------------------------------------------------------------------ dots and updates
// The vector steps of the solve, each one pass over its vectors with the sums that follow it
// (over the interior cells, one partial sum per block).  Bound by memory; 4 components of
// 256x256x64 (138 MB a vector): the last step of an iteration moves 8 vectors in 198 us,
// where three updates and two dots took 330 us for 12.
constexpr int kStepElems = 4;  // elements of a thread
template <typename F>
__device__ __forceinline__ void step_elems(const Dims& d, int nc, F&& f) {
  const long n = (long)nc * d.m;
  const long e0 = (long)blockIdx.x * (256 * kStepElems) + threadIdx.x;
#pragma unroll
  for (int q = 0; q < kStepElems; ++q) {
    const long e = e0 + q * 256;
    if (e >= n) break;
    long r = e;
    if (nc > 1) r -= d.m * (n <= 0xffffffffl ? (long)((unsigned)e / (unsigned)d.m) : e / d.m);
    int i, j, k;
    f(e, is_interior(d, r, i, j, k));
  }
}
// r = b - r (r = A x on entry); rt = p = r; r.r.
__global__ __launch_bounds__(256) void k_step_init(Dims d, int nc, const double* __restrict__ b,
                                                   double* __restrict__ r,
                                                   double* __restrict__ rt,
                                                   double* __restrict__ p,
                                                   double* __restrict__ partial) {
#pragma clang fp contract(off)
  double acc[2] = {0.0, 0.0};
  step_elems(d, nc, [&](long e, bool in) {
    const double v = -1.0 * r[e] + b[e];
    r[e] = v;
    rt[e] = v;
    p[e] = v;
    if (in) acc[0] = __builtin_fma(v, v, acc[0]);
  });
  block_reduce_store<2>(acc, partial, blockIdx.x, threadIdx.x, 256, gridDim.x);
}
// p = r + beta (p - omega v); an update by zero is left out (Axpy_VectorCell :1243).
__global__ __launch_bounds__(256) void k_step_dir(long n, double omega, double beta,
                                                  const double* __restrict__ v,
                                                  const double* __restrict__ r,
                                                  double* __restrict__ p) {
#pragma clang fp contract(off)
  const long e = (long)blockIdx.x * 256 + threadIdx.x;
  if (e >= n) return;
  double q = p[e];
  if (omega != 0.0) q = -omega * v[e] + q;
  p[e] = beta * q + r[e];
}
// s = r - alpha v (into r); s.s.
__global__ __launch_bounds__(256) void k_step_half(Dims d, int nc, double alpha,
                                                   const double* __restrict__ v,
                                                   double* __restrict__ r,
                                                   double* __restrict__ partial) {
#pragma clang fp contract(off)
  double acc[2] = {0.0, 0.0};
  step_elems(d, nc, [&](long e, bool in) {
    double s = r[e];
    if (alpha != 0.0) {
      s = -alpha * v[e] + s;
      r[e] = s;
    }
    if (in) acc[0] = __builtin_fma(s, s, acc[0]);
  });
  block_reduce_store<2>(acc, partial, blockIdx.x, threadIdx.x, 256, gridDim.x);
}
// x += alpha ph + omega rh; r = s - omega t; r.r and rt.r (the next iteration's rho).
__global__ __launch_bounds__(256) void k_step_full(Dims d, int nc, double alpha, double omega,
                                                   const double* __restrict__ ph,
                                                   const double* __restrict__ rh,
                                                   const double* __restrict__ t,
                                                   const double* __restrict__ rt,
                                                   double* __restrict__ x,
                                                   double* __restrict__ r,
                                                   double* __restrict__ partial) {
#pragma clang fp contract(off)
  double acc[2] = {0.0, 0.0};
  step_elems(d, nc, [&](long e, bool in) {
    double xe = x[e], re = r[e];
    if (alpha != 0.0) xe = alpha * ph[e] + xe;
    if (omega != 0.0) {
      xe = omega * rh[e] + xe;
      re = -omega * t[e] + re;
    }
    x[e] = xe;
    r[e] = re;
    if (in) {
      acc[0] = __builtin_fma(re, re, acc[0]);
      acc[1] = __builtin_fma(rt[e], re, acc[1]);
    }
  });
  block_reduce_store<2>(acc, partial, blockIdx.x, threadIdx.x, 256, gridDim.x);
}
// Fixed-order sums of the two partial sums of nblk blocks: thread t adds partials t, t + 1024,
// ..., then the block tree; every run gives the same bits.  out[2]: the sweeps' error word.
__global__ __launch_bounds__(1024) void k_dot_fin(const double* __restrict__ partial, int nblk,
                                                  const int* __restrict__ err,
                                                  double* __restrict__ out) {
  if (threadIdx.x == 0) out[2] = *err;
  double v[2] = {0.0, 0.0};
#pragma unroll 4
  for (int b = threadIdx.x; b < nblk; b += 1024) {
    v[0] += partial[b];
    v[1] += partial[nblk + b];
  }
  block_reduce_store<2>(v, out, 0, threadIdx.x, 1024, 1);
}

__global__ void k_axpy(long n, double a, const double* __restrict__ x, double* __restrict__ y) {
#pragma clang fp contract(off)
  const long e = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (e < n) y[e] = a * x[e] + y[e];
}
}  // namespace tr
}  // namespace asam

using namespace asam;
using namespace asam::tr;

struct asam_tr_ctx {
  int device = 0;
  hipStream_t stream = nullptr;
  Dims d{};
  int nc = 0, iterg = 5;
  Ops ops_mv{}, ops_ps{};  // per-component operator of MatVec and of PSolve
  asam_tr_tuning tune{8, 2, 0, 0};  // gs_rows 4 and more: by size, see sweep_shape
  int hold_boundary = 0;  // test hook (asam_tr_test_hold_boundary)
  bool odd_diag[2] = {false, false};  // JacTMom, JacTPot: a diagonal gs_divide cannot take
  bool have_mom = false, have_pot = false, have_fall = false, have_lu = false;
  std::string err;
  std::vector<void*> allocs;
  double *tmom = nullptr, *tpot = nullptr, *fall = nullptr, *lu = nullptr;
  double *wmom = nullptr, *wpot = nullptr, *wf = nullptr;
  double *bs = nullptr, *xs = nullptr, *ts = nullptr;
  double* bnd = nullptr;  // boundary records, grown on demand
  long bnd_n = 0;
  int* order = nullptr;   // blocks of the sweeps in the order they are taken, for order_kr
  int order_kr = 0;
  std::vector<int> groups;  // sweeps per launch of a preconditioner application
  double *vx = nullptr, *vb = nullptr, *vr = nullptr, *vrt = nullptr, *vrh = nullptr;
  double *vp = nullptr, *vph = nullptr, *vt = nullptr, *vv = nullptr;
  double *partial = nullptr, *dots = nullptr;
  int *sync = nullptr;  // ticket, error word, set-up flag
  int sync_n = 0;
  double* host_dots = nullptr;  // pinned
};

#define TRCHK(ctx, expr)                                                   \
  do {                                                                     \
    hipError_t e_ = (expr);                                                \
    if (e_ != hipSuccess) {                                                \
      (ctx)->err = std::string(#expr) + ": " + hipGetErrorString(e_);      \
      return ASAM_E_HIP;                                                   \
    }                                                                      \
  } while (0)

static int trfail(asam_tr_ctx* c, int code, const char* msg) {
  if (c) c->err = msg;
  return code;
}

template <typename T>
static int tralloc(asam_tr_ctx* c, T** p, size_t count) {
  void* q = nullptr;
  hipError_t e = hipMalloc(&q, (count ? count : 1) * sizeof(T));
  if (e != hipSuccess) {
    c->err = std::string("hipMalloc: ") + hipGetErrorString(e);
    return ASAM_E_NOMEM;
  }
  c->allocs.push_back(q);
  *p = (T*)q;
  return 0;
}

static inline unsigned blocks_for(long n, int bs) { return (unsigned)((n + bs - 1) / bs); }
static inline long step_blocks(const asam_tr_ctx* c) {
  return blocks_for((long)c->nc * c->d.m, 256 * kStepElems);
}

// Rows of a skewed array in front and behind that lanes without a cell may read.
constexpr int kGuardRows = 16;

static void trfree(asam_tr_ctx* c, void* p) {
  for (size_t q = 0; q < c->allocs.size(); ++q)
    if (c->allocs[q] == p) {
      c->allocs.erase(c->allocs.begin() + q);
      break;
    }
  (void)hipFree(p);
}

// A skewed array of `words` words per slot of n slots, with its guard rows (of up to two
// components a slot).
static int skew_alloc(asam_tr_ctx* c, double** p, long n, int words) {
  const size_t guard = (size_t)kGuardRows * c->d.RW * words * 2;
  int rc = tralloc(c, p, (size_t)n * words + 2 * guard);
  if (!rc) *p += guard;
  return rc;
}

extern "C" const char* asam_tr_last_error(const asam_tr_ctx* c) {
  return c ? c->err.c_str() : "null context";
}

extern "C" int asam_tr_destroy(asam_tr_ctx* c) {
  if (!c) return 0;
  (void)hipSetDevice(c->device);
  if (c->stream) (void)hipStreamSynchronize(c->stream);
  for (void* p : c->allocs) (void)hipFree(p);
  if (c->host_dots) (void)hipHostFree(c->host_dots);
  if (c->stream) (void)hipStreamDestroy(c->stream);
  delete c;
  return 0;
}

static int prepare_sweeps(asam_tr_ctx* c, long places);

extern "C" int asam_tr_create(asam_tr_ctx** out, const asam_tr_grid* g) {
  if (!out || !g) return ASAM_E_INVALID;
  *out = nullptr;
  if (g->nx < 1 || g->ny < 1 || g->nz < 1 || g->nz > 126 || g->ncomp < 1 ||
      g->ncomp > kMaxComp || g->iterg < 0 || g->iterg > 32)
    return ASAM_E_INVALID;
  const long X = g->nx + 2L, Y = g->ny + 2L, Z = g->nz + 2L;
  if (X * Y * Z * g->ncomp > (1L << 31)) return ASAM_E_INVALID;
  asam_tr_ctx* c = new asam_tr_ctx();
  auto bail = [&](int rc) {
    asam_tr_destroy(c);
    return rc;
  };
  if (hipGetDevice(&c->device) != hipSuccess) return bail(ASAM_E_HIP);
  if (hipStreamCreateWithFlags(&c->stream, hipStreamNonBlocking) != hipSuccess)
    return bail(ASAM_E_HIP);
  Dims& d = c->d;
  d.nx = g->nx, d.ny = g->ny, d.nz = g->nz;
  d.X = (int)X, d.Y = (int)Y, d.Z = (int)Z;
  d.m = X * Y * Z;
  d.ncell = (long)g->nx * g->ny * g->nz;
  c->nc = g->ncomp;
  c->iterg = g->iterg;
  // the sweeps of an application in launches of nearly equal size
  const int total = g->iterg + 1, nl = (total + kMaxSweeps - 1) / kMaxSweeps;
  for (int q = 0; q < nl; ++q) c->groups.push_back(total / nl + (q < total % nl ? 1 : 0));
  // Components that the sweeps hold at most: groups of two repeat the first one where none is
  // left of its operator kind, and are taken only if that makes fewer groups than components.
  const long places = c->nc <= 2 ? c->nc : c->nc == 3 ? 4 : c->nc + 2 + c->nc % 2;
  // y-tiles of at most `cols` columns that cover Y columns at every sweep's shift.  Rows of
  // kRow entries, of the columns in use where these are few; `compact`: of the columns, rounded
  // up to whole 128-byte lines where that adds at most a quarter.
  auto set_tiles = [&](int cols, bool compact) {
    const int span = d.Y + c->groups[0] - 1;
    d.NJ = (span + cols - 1) / cols;
    d.TW = (span + d.NJ - 1) / d.NJ;
    d.ZW = d.NJ == 1 ? d.Y : d.TW;
    d.HL = d.X + d.ZW - 1;
    const int lines = (d.ZW + 7) / 8 * 8;
    d.RW = d.ZW < 27 ? d.ZW : !compact ? kRow : 4 * lines <= 5 * d.ZW ? lines : d.ZW;
    d.slots = (long)d.Z * d.NJ * d.HL * d.RW;
  };
  // Bytes of the skewed arrays, which must not keep a block off the card.  With few cells in x,
  // wide tiles hold little but skew: above 4 GiB, tiles of X + Z columns (1x100000x20, four
  // components: 14 GB instead of 35).  Above 32 GiB, compact rows (40000x48x100, one
  // component: 42 GB instead of 84).
  const long per = 8 * (2 * kCoefWords + 2 + 2 * places);
  set_tiles(kMaxCols, false);
  if (per * d.slots > (4L << 30) && d.X + d.Z < d.TW) set_tiles(d.X + d.Z, true);
  else if (per * d.slots > (32L << 30)) set_tiles(kMaxCols, true);
  c->ops_mv.nc = c->ops_ps.nc = c->nc;
  for (int q = 0; q < kMaxComp; ++q) {
    c->ops_mv.op[q] = c->ops_ps.op[q] = ASAM_TR_POT;
    c->ops_mv.alpha[q] = c->ops_ps.alpha[q] = 0.0;
  }
  const size_t V = (size_t)c->nc * d.m;
  int rc = 0;
  rc |= tralloc(c, &c->tmom, 7 * (size_t)d.m);
  rc |= tralloc(c, &c->tpot, 7 * (size_t)d.m);
  rc |= tralloc(c, &c->fall, 2 * (size_t)d.m);
  rc |= tralloc(c, &c->lu, (size_t)c->nc * c->nc * d.ncell);
  rc |= skew_alloc(c, &c->wmom, d.slots, kCoefWords);
  rc |= skew_alloc(c, &c->wpot, d.slots, kCoefWords);
  rc |= skew_alloc(c, &c->wf, d.slots, 2);
  rc |= skew_alloc(c, &c->bs, places * d.slots, 1);
  rc |= skew_alloc(c, &c->xs, places * d.slots, 1);
  if (c->groups.size() > 1) rc |= skew_alloc(c, &c->ts, places * d.slots, 1);
  double** vecs[] = {&c->vx, &c->vb, &c->vr, &c->vrt, &c->vrh, &c->vp, &c->vph, &c->vt, &c->vv};
  for (double** v : vecs) rc |= tralloc(c, v, V);
  rc |= tralloc(c, &c->partial, 2 * (size_t)std::max((long)blocks_for(d.m, 256), step_blocks(c)));
  rc |= tralloc(c, &c->dots, 3);
  c->sync_n = 3;  // ticket, error word, set-up flag
  rc |= tralloc(c, &c->sync, (size_t)c->sync_n);
  if (rc) return bail(ASAM_E_NOMEM);
  if (hipHostMalloc((void**)&c->host_dots, 3 * sizeof(double), hipHostMallocDefault) != hipSuccess)
    return bail(ASAM_E_NOMEM);
  if (hipMemsetAsync(c->sync, 0, sizeof(int) * c->sync_n, c->stream) != hipSuccess ||
      hipStreamSynchronize(c->stream) != hipSuccess)
    return bail(ASAM_E_HIP);
  if (int e = prepare_sweeps(c, places)) return bail(e);
  *out = c;
  return 0;
}

// Grid of the kernels that transpose to the skewed layout.
static dim3 skew_grid(const Dims& d, int levels) { return dim3(d.NJ * h_blocks(d), 1, levels); }

extern "C" int asam_tr_set_matrix(asam_tr_ctx* c, int which, int numdiag, int diag,
                                  const int* ptr, const double* val) {
  if (!c || !ptr || !val) return trfail(c, ASAM_E_INVALID, "null argument");
  const Dims& d = c->d;
  const long X = d.X, XY = (long)d.X * d.Y, m = d.m;
  if (which == ASAM_TR_JACTMOM || which == ASAM_TR_JACTPOT) {
    const long want[7] = {-XY, -X, -1, 0, 1, X, XY};
    if (numdiag != 7 || diag != 4) return trfail(c, ASAM_E_INVALID, "NumDiag must be 7, Diag 4");
    for (int q = 0; q < 7; ++q)
      if (ptr[q] != want[q]) return trfail(c, ASAM_E_INVALID, "DiagPtr is not the 7-point layout");
    // couplings across the wrap of the linear index are not neighbour couplings
    for (long r = 0; r < m; ++r) {
      const long i = r % X, jy = (r / X) % d.Y;
      if ((i == X - 1 && val[2 * m + r] != 0.0) || (i == 0 && r > 0 && val[4 * m + r] != 0.0) ||
          (jy == d.Y - 1 && val[1 * m + r] != 0.0) || (jy == 0 && r >= X && val[5 * m + r] != 0.0))
        return trfail(c, ASAM_E_INVALID,
                      "coupling between the ends of consecutive x-rows or y-planes");
      for (int q = 0; q < 7; ++q)
        if (!std::isfinite(val[q * m + r])) return trfail(c, ASAM_E_NAN, "non-finite Val");
    }
    double* dst = which == ASAM_TR_JACTMOM ? c->tmom : c->tpot;
    double* w = which == ASAM_TR_JACTMOM ? c->wmom : c->wpot;
    TRCHK(c, hipSetDevice(c->device));
    TRCHK(c, hipMemcpyAsync(dst, val, 7 * sizeof(double) * m, hipMemcpyHostToDevice, c->stream));
    k_zero_int<<<1, 64, 0, c->stream>>>(c->sync + 2, 1);
    k_skew_coef<<<skew_grid(d, d.Z), 256, 0, c->stream>>>(d, dst, w, c->sync + 2);
    TRCHK(c, hipGetLastError());
    int odd = 0;
    TRCHK(c, hipMemcpyAsync(&odd, c->sync + 2, sizeof(int), hipMemcpyDeviceToHost, c->stream));
    TRCHK(c, hipStreamSynchronize(c->stream));
    c->odd_diag[which] = odd != 0;
    (which == ASAM_TR_JACTMOM ? c->have_mom : c->have_pot) = true;
    return 0;
  }
  if (which == ASAM_TR_JACFALL) {
    if (numdiag != 2 || diag != 1 || ptr[0] != 0 || ptr[1] != XY)
      return trfail(c, ASAM_E_INVALID, "JacFall must have DiagPtr 0, (nx+2)(ny+2), Diag 1");
    for (long e = 0; e < 2 * m; ++e)
      if (!std::isfinite(val[e])) return trfail(c, ASAM_E_NAN, "non-finite Val");
    TRCHK(c, hipSetDevice(c->device));
    TRCHK(c, hipMemcpyAsync(c->fall, val, 2 * sizeof(double) * m, hipMemcpyHostToDevice, c->stream));
    k_skew_fall<<<skew_grid(d, d.Z), 256, 0, c->stream>>>(d, c->fall, c->wf);
    TRCHK(c, hipGetLastError());
    TRCHK(c, hipStreamSynchronize(c->stream));
    c->have_fall = true;
    return 0;
  }
  return trfail(c, ASAM_E_INVALID, "which");
}

extern "C" int asam_tr_set_lu(asam_tr_ctx* c, const double* lu) {
  if (!c) return ASAM_E_INVALID;
  if (!lu) {
    c->have_lu = false;
    return 0;
  }
  const size_t n = (size_t)c->nc * c->nc * c->d.ncell;
  for (size_t e = 0; e < n; ++e)
    if (!std::isfinite(lu[e])) return trfail(c, ASAM_E_NAN, "non-finite LU");
  TRCHK(c, hipSetDevice(c->device));
  TRCHK(c, hipMemcpyAsync(c->lu, lu, n * sizeof(double), hipMemcpyHostToDevice, c->stream));
  TRCHK(c, hipStreamSynchronize(c->stream));
  c->have_lu = true;
  return 0;
}

extern "C" int asam_tr_set_components(asam_tr_ctx* c, const int* op_mv, const int* op_ps,
                                      const double* alpha) {
  if (!c) return ASAM_E_INVALID;
  for (int q = 0; q < c->nc; ++q) {
    const int a = op_mv ? op_mv[q] : ASAM_TR_POT, b = op_ps ? op_ps[q] : ASAM_TR_POT;
    if (a < 0 || a > 2 || b < 0 || b > 2) return trfail(c, ASAM_E_INVALID, "operator code");
    if (alpha && !std::isfinite(alpha[q])) return trfail(c, ASAM_E_NAN, "alpha");
  }
  for (int q = 0; q < c->nc; ++q) {
    c->ops_mv.op[q] = op_mv ? op_mv[q] : ASAM_TR_POT;
    c->ops_ps.op[q] = op_ps ? op_ps[q] : ASAM_TR_POT;
    c->ops_mv.alpha[q] = c->ops_ps.alpha[q] = alpha ? alpha[q] : 0.0;
  }
  return 0;
}

// ------------------------------------------------------------------ launchers
static bool uses(const Ops& o, int nc, int op) {
  for (int q = 0; q < nc; ++q)
    if (o.op[q] == op) return true;
  return false;
}

// The matrices a component table needs have been set (JacTPot always: the first
// residual of BiCGStab takes it for every component).
static int check_ready(asam_tr_ctx* c, const Ops& o) {
  if (!c->have_pot) return trfail(c, ASAM_E_STATE, "JacTPot not set");
  if (uses(o, c->nc, ASAM_TR_MOM) && !c->have_mom)
    return trfail(c, ASAM_E_STATE, "JacTMom not set");
  if (uses(o, c->nc, ASAM_TR_FALL) && !c->have_fall)
    return trfail(c, ASAM_E_STATE, "JacFall not set");
  return 0;
}

template <int NC>
static void matvec_nc(asam_tr_ctx* c, const double* x, double* y, int init, int mom, int nd,
                      const double* u) {
  const Dims& d = c->d;
  k_matvec<NC><<<blocks_for(d.m, 256), 256, 0, c->stream>>>(
      d, c->tmom, c->tpot, c->fall, c->have_lu ? c->lu : nullptr, x, y, c->ops_mv, init, mom,
      1, nd, u, c->partial);
}

// nd sums over the interior cells with it: y.u (1), y.y (2), see sums().
static int launch_matvec(asam_tr_ctx* c, const double* x, double* y, int init, int nd = 0,
                         const double* u = nullptr) {
  const int mom = (!init && uses(c->ops_mv, c->nc, ASAM_TR_MOM)) ? 1 : 0;
  switch (c->nc) {
#define NCCASE(n) \
  case n:         \
    matvec_nc<n>(c, x, y, init, mom, nd, u); \
    break;
    NCCASE(1) NCCASE(2) NCCASE(3) NCCASE(4) NCCASE(5) NCCASE(6) NCCASE(7) NCCASE(8)
    NCCASE(9) NCCASE(10) NCCASE(11) NCCASE(12) NCCASE(13) NCCASE(14) NCCASE(15) NCCASE(16)
#undef NCCASE
    default:
      return trfail(c, ASAM_E_INVALID, "ncomp");
  }
  TRCHK(c, hipGetLastError());
  return 0;
}

template <int NC, int KR, int D, bool FALL, bool DIV>
static void tiles_launch(asam_tr_ctx* c, const GsArgs& a, unsigned blocks) {
  const size_t lds = 2 * (size_t)a.M * (KR + 1) * kLdsRow * sizeof(double) * NC;
  const dim3 threads(64 * (a.M + 2));
  // 32-bit byte offsets within a tile's rows, except for blocks of about a million cells in x
  if ((long)(a.d.HL + 1) * (kCoefWords * a.d.RW * 8) >= (1L << 32))
    k_gs_tiles<NC, KR, D, FALL, DIV, 0, unsigned long>
        <<<blocks, threads, lds, c->stream>>>(a, c->ops_ps);
  else if (a.d.RW == kRow)
    k_gs_tiles<NC, KR, D, FALL, DIV, kRow, unsigned>
        <<<blocks, threads, lds, c->stream>>>(a, c->ops_ps);
  else
    k_gs_tiles<NC, KR, D, FALL, DIV, 0, unsigned>
        <<<blocks, threads, lds, c->stream>>>(a, c->ops_ps);
}

template <int NC, int KR, int D>
static void tiles_kind(asam_tr_ctx* c, const GsArgs& a, unsigned blocks) {
  const bool fall = uses(c->ops_ps, c->nc, ASAM_TR_FALL);
  const bool odd = (uses(c->ops_ps, c->nc, ASAM_TR_MOM) && c->odd_diag[ASAM_TR_JACTMOM]) ||
                   c->odd_diag[ASAM_TR_JACTPOT];
  if (fall) tiles_launch<NC, KR, D, true, true>(c, a, blocks);
  else if (odd) tiles_launch<NC, KR, D, false, true>(c, a, blocks);
  else tiles_launch<NC, KR, D, false, false>(c, a, blocks);
}

// The components in groups of nc_per of the same operator; a group's second place repeats
// its first when no component is left for it.
static Groups make_groups(const asam_tr_ctx* c, int nc_per) {
  Groups g;
  g.n = 0;
  int open[3] = {-1, -1, -1};
  for (int q = 0; q < c->nc; ++q) {
    int& o = open[c->ops_ps.op[q]];
    if (nc_per == 2 && o >= 0) {
      g.c[o][1] = q;
      o = -1;
    } else {
      g.c[g.n][0] = g.c[g.n][1] = q;
      o = g.n++;
    }
  }
  return g;
}

// Levels per block and components per group of the sweeps: those that the tuning names (1-3
// levels), or by size.  A block of two levels of one component takes the shortest steps; with
// up to a block per CU nothing else counts (101x77x50, three components, 174 blocks: 6 sweeps
// in 249 us, against 325 us with three levels and 331 us with two components).  Beyond that,
// blocks of three levels and, where components share a matrix, two of them pass the fewest
// coefficients through the caches per cell (256x256x64, four components: 1238 us, against 1385
// us and 1311 us for one component with two and three levels, 1672 us for two with two).
struct Shape {
  int KR, NC;
};
static Shape sweep_shape(const asam_tr_ctx* c) {
  constexpr int kCus = 256;
  const int named = c->tune.gs_rows;
  auto blocks = [&](int KR, int groups) {
    return (long)groups * c->d.NJ * ((c->d.Z + c->groups[0] - 1 + KR - 1) / KR);
  };
  const int KR = named <= 3 ? named : (blocks(2, c->nc) <= kCus ? 2 : 3);
  const bool pairs = make_groups(c, 2).n < c->nc;
  return {KR, pairs && blocks(KR, c->nc) > kCus ? 2 : 1};
}

// The block order for KR levels per block: by the step of the application at which a block
// starts, which puts its predecessors in j and k before it.
static int ensure_order(asam_tr_ctx* c, int KR) {
  if (c->order_kr == KR) return 0;
  const Dims& d = c->d;
  const int NK = (d.Z + c->groups[0] - 1 + KR - 1) / KR;
  std::vector<int> o((size_t)d.NJ * NK);
  for (size_t q = 0; q < o.size(); ++q) o[q] = (int)q;
  auto start = [&](int b) { return (long)(b % d.NJ) * d.TW + (long)(b / d.NJ) * KR; };
  std::stable_sort(o.begin(), o.end(), [&](int x, int y) { return start(x) < start(y); });
  if (c->order) {
    TRCHK(c, hipStreamSynchronize(c->stream));
    trfree(c, c->order);
    c->order = nullptr;
    c->order_kr = 0;
  }
  if (int rc = tralloc(c, &c->order, o.size())) return rc;
  TRCHK(c, hipMemcpyAsync(c->order, o.data(), o.size() * sizeof(int), hipMemcpyHostToDevice,
                          c->stream));
  TRCHK(c, hipStreamSynchronize(c->stream));
  c->order_kr = KR;
  return 0;
}

// The boundary records hold at least n doubles.
static int ensure_records(asam_tr_ctx* c, long n) {
  if (n <= c->bnd_n) return 0;
  TRCHK(c, hipStreamSynchronize(c->stream));
  if (c->bnd) trfree(c, c->bnd);
  c->bnd = nullptr;
  c->bnd_n = 0;
  if (int rc = tralloc(c, &c->bnd, (size_t)n)) return rc;
  c->bnd_n = n;
  return 0;
}

// Blocks, and doubles of their boundary records per component, of M sweeps in blocks of KR
// levels.
static long sweep_blocks(const asam_tr_ctx* c, int KR) {
  return (long)c->d.NJ * ((c->d.Z + c->groups[0] - 1 + KR - 1) / KR);
}
static long sweep_records(const asam_tr_ctx* c, int KR, int M) {
  return sweep_blocks(c, KR) * (c->d.X + c->d.TW + KR - 2) * M *
         (c->d.ZW + (c->d.NJ == 1 ? 0 : KR));
}

// Block order and boundary records of the default shape, for `places` components.
static int prepare_sweeps(asam_tr_ctx* c, long places) {
  const int KR = sweep_shape(c).KR;
  if (int rc = ensure_order(c, KR)) return rc;
  return ensure_records(c, places * sweep_records(c, KR, c->groups[0]));
}

// One launch of M sweeps over every component; first: from x = 0, else from xs.  The ticket
// is cleared and the boundary records reset to the sentinel first.
template <int NC>
static int launch_sweeps(asam_tr_ctx* c, const Groups& gr, int M, bool first) {
  const Dims& d = c->d;
  const int KR = sweep_shape(c).KR;
  if (int rc = ensure_order(c, KR)) return rc;
  GsArgs a;
  a.d = d;
  a.wmom = c->wmom, a.wpot = c->wpot, a.wf = c->wf;
  a.bs = c->bs, a.xs = c->xs;
  a.ts = first ? c->bs : c->ts;
  a.order = c->order;
  a.counter = c->sync;
  a.err = c->sync + 1;
  a.NK = (d.Z + c->groups[0] - 1 + KR - 1) / KR;
  a.M = M;
  a.groups = gr;
  a.nsteps = d.X + d.TW + KR - 2;
  a.spin_limit = c->tune.gs_spin_limit > 0 ? c->tune.gs_spin_limit : kSpinLimit;
  a.hold = c->hold_boundary;
  const long nblk = sweep_blocks(c, KR), nb = gr.n * NC * sweep_records(c, KR, M);
  if (int rc = ensure_records(c, nb)) return rc;
  a.bnd = c->bnd;
  if (!first)
    k_gs_upart<NC><<<dim3(d.NJ * ((d.HL + 3) / 4), 1, d.Z * gr.n * NC), 256, 0, c->stream>>>(
        a, c->ops_ps, c->ts);
  k_gs_reset<<<blocks_for((nb + 1) / 2, 256), 256, 0, c->stream>>>((unsigned long long*)c->bnd, nb,
                                                                    kSentinel, c->sync);
  const unsigned blocks = (unsigned)(gr.n * nblk);
  if (KR == 1) tiles_kind<NC, 1, 2>(c, a, blocks);
  else if (KR == 2) tiles_kind<NC, 2, NC == 1 ? 2 : 1>(c, a, blocks);
  else tiles_kind<NC, 3, 1>(c, a, blocks);
  TRCHK(c, hipGetLastError());
  return 0;
}

template <int NC>
static int psolve_nc(asam_tr_ctx* c, const double* x, double* y) {
  const Dims& d = c->d;
  const Groups gr = make_groups(c, NC);
  const int levels = d.Z * gr.n;
  k_skew_vec<NC><<<dim3(d.NJ * ((d.HL + kVecH - 1) / kVecH), 1, levels), 256, 0, c->stream>>>(
      d, gr, x, c->bs);
  TRCHK(c, hipGetLastError());
  for (size_t q = 0; q < c->groups.size(); ++q)
    if (int rc = launch_sweeps<NC>(c, gr, c->groups[q], q == 0)) return rc;
  k_unskew<NC><<<dim3(d.NJ * ((d.X + kVecH - 1) / kVecH), 1, levels), 256, 0, c->stream>>>(
      d, gr, c->xs, y);
  TRCHK(c, hipGetLastError());
  return 0;
}

// PSolve_Vec4CellSp: y = GS^(1+IterG)(x) per component, halo zero.  x may equal y.
static int launch_psolve(asam_tr_ctx* c, const double* x, double* y) {
  return sweep_shape(c).NC == 2 ? psolve_nc<2>(c, x, y) : psolve_nc<1>(c, x, y);
}

// The error word of the sweeps' waits: cleared when a call begins, read before it returns.
static const char kWaited[] = "Gauss-Seidel sweep: a workgroup waited past its limit";
static int clear_gs_error(asam_tr_ctx* c) {
  k_zero_int<<<1, 64, 0, c->stream>>>(c->sync + 1, 1);
  TRCHK(c, hipGetLastError());
  return 0;
}
static int check_gs_error(asam_tr_ctx* c) {
  int e = 0;
  TRCHK(c, hipMemcpyAsync(&e, c->sync + 1, sizeof(int), hipMemcpyDeviceToHost,
                          c->stream));
  TRCHK(c, hipStreamSynchronize(c->stream));
  if (e) return trfail(c, ASAM_E_HIP, kWaited);
  return 0;
}

// The two sums of the nblk blocks launched last; results on the host.  Fails where a sweep
// before them gave up waiting.
static int sums(asam_tr_ctx* c, long nblk, double* out) {
  k_dot_fin<<<1, 1024, 0, c->stream>>>(c->partial, (int)nblk, c->sync + 1, c->dots);
  TRCHK(c, hipGetLastError());
  TRCHK(c, hipMemcpyAsync(c->host_dots, c->dots, 3 * sizeof(double), hipMemcpyDeviceToHost,
                          c->stream));
  TRCHK(c, hipStreamSynchronize(c->stream));
  if (c->host_dots[2] != 0.0) return trfail(c, ASAM_E_HIP, kWaited);
  out[0] = c->host_dots[0];
  out[1] = c->host_dots[1];
  return 0;
}

static int axpy(asam_tr_ctx* c, double a, const double* x, double* y) {
  if (a == 0.0) return 0;  // Axpy_VectorCell skips alpha == 0 (:1243)
  const long V = (long)c->nc * c->d.m;
  k_axpy<<<blocks_for(V, 256), 256, 0, c->stream>>>(V, a, x, y);
  TRCHK(c, hipGetLastError());
  return 0;
}
#define TRY(expr)              \
  do {                         \
    if (int rc_ = (expr)) return rc_; \
  } while (0)

// BiCGStabChem/Met_Vec4CellSp (SpMatrix4CellPar_Mod.f90:140-348) on device vectors.
static int solve_dev(asam_tr_ctx* c, double* x, const double* b, int* maxiter, double* tol,
                     asam_tr_info* info) {
  asam_tr_info inf{};
  double *r = c->vr, *rt = c->vrt, *rh = c->vrh, *p = c->vp, *ph = c->vph, *t = c->vt,
         *v = c->vv;
  const int MaxIter = *maxiter;
  const double Tol = *tol;
  TRY(clear_gs_error(c));
  TRY(launch_matvec(c, x, r, 1));  // MatVecChem(r, A, x)
  inf.matvecs = 1;
  const Dims& d = c->d;
  const long V = (long)c->nc * d.m, sb = step_blocks(c), mb = blocks_for(d.m, 256);
  double q2[2];
  k_step_init<<<(unsigned)sb, 256, 0, c->stream>>>(d, c->nc, b, r, rt, p, c->partial);
  TRY(sums(c, sb, q2));
  const double rnorm0 = std::sqrt(q2[0]);
  inf.rnorm0 = rnorm0;
  inf.rnorm = rnorm0;
  inf.status = ASAM_NOT_CONVERGED;
  double rho = 0.0, rho_old, rho_next = q2[0], alpha = 0.0, omega = 0.0, beta, rnorm = rnorm0;
  for (int it = 1; it <= MaxIter; ++it) {
    inf.iterations = it;
    rho_old = rho;
    rho = rho_next;  // rt.r, with the step that wrote r (rt = r at first)
    if (rho == 0.0) {
      *maxiter = it;
      *tol = 0.0;
      inf.status = ASAM_BREAKDOWN;
      break;
    }
    if (it > 1) {  // p = r at first
      beta = (rho / rho_old) * (alpha / omega);
      k_step_dir<<<blocks_for(V, 256), 256, 0, c->stream>>>(V, omega, beta, v, r, p);
    }
    TRY(launch_psolve(c, p, ph));
    TRY(launch_matvec(c, ph, v, 0, 1, rt));
    inf.psolves++, inf.matvecs++;
    TRY(sums(c, mb, q2));
    alpha = rho / q2[0];
    k_step_half<<<(unsigned)sb, 256, 0, c->stream>>>(d, c->nc, alpha, v, r, c->partial);
    TRY(sums(c, sb, q2));
    rnorm = std::sqrt(q2[0]);
    if (rnorm <= Tol * rnorm0) {
      TRY(axpy(c, alpha, ph, x));
      *maxiter = -it;
      *tol = rnorm;
      inf.status = ASAM_CONVERGED;
      break;
    }
    TRY(launch_psolve(c, r, rh));
    TRY(launch_matvec(c, rh, t, 0, 2, r));
    inf.psolves++, inf.matvecs++;
    TRY(sums(c, mb, q2));
    omega = q2[0] / q2[1];
    k_step_full<<<(unsigned)sb, 256, 0, c->stream>>>(d, c->nc, alpha, omega, ph, rh, t, rt, x, r,
                                                     c->partial);
    TRY(sums(c, sb, q2));
    rnorm = std::sqrt(q2[0]);
    rho_next = q2[1];
    if (rnorm <= Tol * rnorm0) {
      *maxiter = it;
      *tol = rnorm;
      inf.status = ASAM_CONVERGED;
      break;
    }
    if (it == MaxIter) {
      *maxiter = 2 * it;
      *tol = rnorm;
      break;
    }
  }
  inf.rnorm = (inf.status == ASAM_BREAKDOWN) ? rnorm : *tol;
  if (!std::isfinite(rnorm)) return trfail(c, ASAM_E_NAN, "non-finite residual");
  TRCHK(c, hipStreamSynchronize(c->stream));  // the last update of x
  if (info) *info = inf;
  return 0;
}

extern "C" int asam_tr_matvec_device(asam_tr_ctx* c, const double* x, double* y, int init) {
  if (!c || !x || !y || x == y) return trfail(c, ASAM_E_INVALID, "x, y must be distinct buffers");
  TRY(check_ready(c, c->ops_mv));
  TRCHK(c, hipSetDevice(c->device));
  TRY(launch_matvec(c, x, y, init));
  TRCHK(c, hipStreamSynchronize(c->stream));
  return 0;
}

extern "C" int asam_tr_psolve_device(asam_tr_ctx* c, const double* x, double* y) {
  if (!c || !x || !y) return trfail(c, ASAM_E_INVALID, "null argument");
  TRY(check_ready(c, c->ops_ps));
  TRCHK(c, hipSetDevice(c->device));
  TRY(clear_gs_error(c));
  TRY(launch_psolve(c, x, y));
  return check_gs_error(c);
}

extern "C" int asam_tr_solve_device(asam_tr_ctx* c, double* x, const double* b, int* maxiter,
                                    double* tol, asam_tr_info* info) {
  if (!c || !x || !b || !maxiter || !tol) return trfail(c, ASAM_E_INVALID, "null argument");
  if (x == b) return trfail(c, ASAM_E_INVALID, "x and b must be distinct buffers");
  if (!(*tol >= 0.0)) return trfail(c, ASAM_E_INVALID, "tol");
  TRY(check_ready(c, c->ops_ps));
  TRY(check_ready(c, c->ops_mv));
  TRCHK(c, hipSetDevice(c->device));
  return solve_dev(c, x, b, maxiter, tol, info);
}

static size_t vbytes(const asam_tr_ctx* c) { return sizeof(double) * c->nc * c->d.m; }

extern "C" int asam_tr_matvec(asam_tr_ctx* c, const double* x, double* y, int init) {
  if (!c || !x || !y) return trfail(c, ASAM_E_INVALID, "null argument");
  TRY(check_ready(c, c->ops_mv));
  TRCHK(c, hipSetDevice(c->device));
  TRCHK(c, hipMemcpyAsync(c->vx, x, vbytes(c), hipMemcpyHostToDevice, c->stream));
  TRY(launch_matvec(c, c->vx, c->vt, init));
  TRCHK(c, hipMemcpyAsync(y, c->vt, vbytes(c), hipMemcpyDeviceToHost, c->stream));
  TRCHK(c, hipStreamSynchronize(c->stream));
  return 0;
}

extern "C" int asam_tr_psolve(asam_tr_ctx* c, const double* x, double* y) {
  if (!c || !x || !y) return trfail(c, ASAM_E_INVALID, "null argument");
  TRY(check_ready(c, c->ops_ps));
  TRCHK(c, hipSetDevice(c->device));
  TRCHK(c, hipMemcpyAsync(c->vx, x, vbytes(c), hipMemcpyHostToDevice, c->stream));
  TRY(clear_gs_error(c));
  TRY(launch_psolve(c, c->vx, c->vt));
  TRCHK(c, hipMemcpyAsync(y, c->vt, vbytes(c), hipMemcpyDeviceToHost, c->stream));
  TRCHK(c, hipStreamSynchronize(c->stream));
  return check_gs_error(c);
}

extern "C" int asam_tr_solve(asam_tr_ctx* c, double* x, const double* b, int* maxiter,
                             double* tol, asam_tr_info* info) {
  if (!c || !x || !b || !maxiter || !tol) return trfail(c, ASAM_E_INVALID, "null argument");
  if (!(*tol >= 0.0)) return trfail(c, ASAM_E_INVALID, "tol");
  TRY(check_ready(c, c->ops_ps));
  TRY(check_ready(c, c->ops_mv));
  TRCHK(c, hipSetDevice(c->device));
  TRCHK(c, hipMemcpyAsync(c->vx, x, vbytes(c), hipMemcpyHostToDevice, c->stream));
  TRCHK(c, hipMemcpyAsync(c->vb, b, vbytes(c), hipMemcpyHostToDevice, c->stream));
  TRY(solve_dev(c, c->vx, c->vb, maxiter, tol, info));
  TRCHK(c, hipMemcpyAsync(x, c->vx, vbytes(c), hipMemcpyDeviceToHost, c->stream));
  TRCHK(c, hipStreamSynchronize(c->stream));
  return 0;
}

extern "C" int asam_tr_get_tuning(const asam_tr_ctx* c, asam_tr_tuning* t) {
  if (!c || !t) return ASAM_E_INVALID;
  *t = c->tune;
  return 0;
}

extern "C" int asam_tr_set_tuning(asam_tr_ctx* c, const asam_tr_tuning* t) {
  if (!c || !t) return ASAM_E_INVALID;
  if (t->gs_rows < 1 || t->gs_rows > 8) return trfail(c, ASAM_E_INVALID, "gs_rows");
  if (t->gs_chunk != 2 && t->gs_chunk != 4) return trfail(c, ASAM_E_INVALID, "gs_chunk");
  if (t->gs_spin_limit < 0) return trfail(c, ASAM_E_INVALID, "gs_spin_limit");
  c->tune = *t;
  return 0;
}

extern "C" int asam_tr_test_hold_boundary(asam_tr_ctx* c, int hold) {
  if (!c) return ASAM_E_INVALID;
  c->hold_boundary = hold != 0;
  return 0;
}

extern "C" int asam_tr_time_kernel(asam_tr_ctx* c, int which, int reps, double* ms) {
  if (!c || !ms || reps < 1 || which < 0 || which > 2) return trfail(c, ASAM_E_INVALID, "argument");
  TRY(check_ready(c, which == 1 ? c->ops_mv : c->ops_ps));
  TRCHK(c, hipSetDevice(c->device));
  TRY(clear_gs_error(c));
  hipEvent_t e0, e1;
  TRCHK(c, hipEventCreate(&e0));
  TRCHK(c, hipEventCreate(&e1));
  int rc = 0;
  auto once = [&]() -> int {
    if (which == 0) {
      if (sweep_shape(c).NC == 2) TRY(launch_sweeps<2>(c, make_groups(c, 2), c->groups[0], true));
      else TRY(launch_sweeps<1>(c, make_groups(c, 1), c->groups[0], true));
    } else if (which == 1) {
      TRY(launch_matvec(c, c->vp, c->vv, 0));
    } else {
      TRY(launch_psolve(c, c->vp, c->vph));
    }
    return 0;
  };
  if (which == 0) rc = launch_psolve(c, c->vp, c->vph);  // the skewed right-hand side
  if (!rc)
    rc = once();
  if (!rc) {
    (void)hipEventRecord(e0, c->stream);
    for (int q = 0; q < reps && !rc; ++q) rc = once();
    (void)hipEventRecord(e1, c->stream);
    (void)hipEventSynchronize(e1);
    float t = 0.0f;
    (void)hipEventElapsedTime(&t, e0, e1);
    *ms = t / reps / (which == 0 ? c->groups[0] : 1);  // 0: per sweep of a launch
  }
  (void)hipEventDestroy(e0);
  (void)hipEventDestroy(e1);
  if (rc) return rc;
  return check_gs_error(c);
}

extern "C" int asam_tr_dev_alloc(asam_tr_ctx* c, void** ptr, size_t bytes) {
  if (!c || !ptr) return ASAM_E_INVALID;
  TRCHK(c, hipSetDevice(c->device));
  TRCHK(c, hipMalloc(ptr, bytes ? bytes : 1));
  return 0;
}
extern "C" int asam_tr_dev_free(asam_tr_ctx* c, void* ptr) {
  if (!c) return ASAM_E_INVALID;
  if (ptr) TRCHK(c, hipFree(ptr));
  return 0;
}
extern "C" int asam_tr_dev_upload(asam_tr_ctx* c, void* dst, const void* src, size_t bytes) {
  if (!c || !dst || !src) return ASAM_E_INVALID;
  TRCHK(c, hipMemcpyAsync(dst, src, bytes, hipMemcpyHostToDevice, c->stream));
  TRCHK(c, hipStreamSynchronize(c->stream));
  return 0;
}
extern "C" int asam_tr_dev_download(asam_tr_ctx* c, void* dst, const void* src, size_t bytes) {
  if (!c || !dst || !src) return ASAM_E_INVALID;
  TRCHK(c, hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, c->stream));
  TRCHK(c, hipStreamSynchronize(c->stream));
  return 0;
}
