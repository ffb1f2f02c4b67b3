// line_launch.h -- vertical-line preconditioner solve kernel and its dispatch; each of the
// line_*.hip files compiles one block size and precision.
#pragma once
#include "line_tile.h"

namespace asam {

size_t lds_budget_for(int line_lds);
int lds_levels(int nz, int np, size_t word, size_t budget, int halves);

// Backward-sweep window: 16 levels with the 8-level forward window (the backward sweep
// holds 6-10 words per level against the forward's 12-14; measured 1-5% faster line
// solves), else the forward window.
template <int P>
constexpr int kBackWindow = P == 8 ? 16 : 0;

// One 64-column tile per workgroup: grid (gxl, ny).
template <int NP, int TR, int MODE, int LDS, int P, int HV, int NT, typename CT, typename VT>
__global__ __launch_bounds__(64 * HV) void k_line(KLine<CT, VT> a) {
  if (a.done && *a.done) return;  // the state before this launch: the same in every workgroup
  extern __shared__ unsigned char lds_raw[];
  CT* stage = reinterpret_cast<CT*>(lds_raw);
  const int blk = blockIdx.x + gridDim.x * blockIdx.y;
  double acc[1] = {0.0};
  if constexpr (MODE == LINE_PLAIN) {
    line_tile<NP, TR, MODE, LDS, P, HV, CT, VT, NT, kBackWindow<P>>(a, blockIdx.x, blockIdx.y,
                                                                    gridDim.x, stage, acc);
  } else {
    // a folded tail (the previous iteration's exit test and beta before the p-step, alpha
    // before the s-step): the scalars come from this workgroup's copy of the state
    __shared__ unsigned long long sk[kTailWords];
    const bool fold = a.fold.kind >= 0;
    bool run = true;
    KLine<CT, VT> b = a;
    if (fold) {
      fold_state<HV>(a.fold, sk, threadIdx.x);
      fold_write(a.fold, sk, threadIdx.x, 64 * HV);
      const KState* s = reinterpret_cast<const KState*>(sk);
      b.st = s;
      run = s->done == 0;
    }
    if (run)
      line_tile<NP, TR, MODE, LDS, P, HV, CT, VT, NT, kBackWindow<P>>(
          b, blockIdx.x, blockIdx.y, gridDim.x, stage, acc);
    if constexpr (MODE == LINE_BICG_S) {
      block_reduce_store<1>(acc, a.partial + (long)a.qslot * kRedBlocks, blk, threadIdx.x,
                            64 * HV);
    }
  }
}

template <int NP, int TR, int LDS, int P, int HV, int NT, typename CT, typename VT>
static void line_mode(hipStream_t s, const Geom& g, const KLine<CT, VT>& a, int mode,
                      size_t lds) {
  const dim3 grid((g.nx + 63) / 64, g.ny), wg(64 * HV);
  switch (mode) {
    case LINE_PLAIN:
      hipLaunchKernelGGL((k_line<NP, TR, LINE_PLAIN, LDS, P, HV, NT, CT, VT>), grid, wg, lds, s,
                         a);
      break;
    case LINE_BICG_P:
      hipLaunchKernelGGL((k_line<NP, TR, LINE_BICG_P, LDS, P, HV, NT, CT, VT>), grid, wg, lds, s,
                         a);
      break;
    default:
      hipLaunchKernelGGL((k_line<NP, TR, LINE_BICG_S, LDS, P, HV, NT, CT, VT>), grid, wg, lds, s,
                         a);
      break;
  }
}

// Cache policy of the factor loads: the tuning's, or by the factors' footprint.
template <int NP, typename CT>
static bool line_nontemporal(const Geom& g) {
  if (g.tune.line_nt != 2) return g.tune.line_nt == 1;
  return (2l * NP * NP + lower_words(NP)) * g.N * (long)sizeof(CT) >
         line_nt_bytes(NP, sizeof(CT));
}

template <int NP, int TR, int LDS, int P, typename CT, typename VT>
static void line_launch(hipStream_t s, const Geom& g, const KLine<CT, VT>& a, int mode,
                        size_t lds) {
  const bool nt = line_nontemporal<NP, CT>(g);
  if constexpr (sizeof(CT) == 8) {
    if (g.halves == 2) {
      if (nt) line_mode<NP, TR, LDS, P, 2, 1, CT, VT>(s, g, a, mode, lds);
      else line_mode<NP, TR, LDS, P, 2, 0, CT, VT>(s, g, a, mode, lds);
      return;
    }
  }
  if (nt) line_mode<NP, TR, LDS, P, 1, 1, CT, VT>(s, g, a, mode, lds);
  else line_mode<NP, TR, LDS, P, 1, 0, CT, VT>(s, g, a, mode, lds);
}

template <int NP, int TR, typename CT, typename VT>
static void line_t(hipStream_t s, const Geom& g, const Coef<CT>& c, const LineReq& r) {
  const int halves = sizeof(CT) == 8 ? g.halves : 1;
  KLine<CT, VT> a;
  a.c = c; a.nx = g.nx; a.ny = g.ny; a.nz = g.nz; a.tiled = g.tune.line_tiled;
  a.src = (const VT*)r.src; a.p = (VT*)r.p; a.v = (const VT*)r.v; a.out = (VT*)r.out;
  a.scale = r.scale; a.st = r.st; a.partial = r.partial; a.done = r.done;
  a.qslot = r.qslot;
  a.fold = r.fold;
  a.kl = r.use_lds ? lds_levels(g.nz, NP, sizeof(CT), lds_budget_for(g.tune.line_lds),
                                halves)
                   : 0;
  const size_t lds = (size_t)a.kl * halves * 64 * NP * sizeof(CT);
  const bool use_lds = a.kl > 0;
  // Default window: 8 levels, but 4 for 2x2 blocks with two wavefronts per tile once a
  // compute unit has a tile: another tile's loads then hide a window's latency.  BiCGStab
  // solves, us with 4 / 8 levels: two wavefronts, 2x2 FP64 128x128x32 585/613, 130x97x40
  // 690/701, 64x64x40 427/428, one component FP64 64x64x40 299/293, 192x128x50 1041/1044; one
  // wavefront, 2x2 FP64 201x150x50 2702/2696, 256x192x56 4144/4114, mixed 256x256x64
  // 2802/2750, one component FP64 256x256x64 2724/2603.
  const int P = g.tune.line_window > 0
                    ? g.tune.line_window
                    : (NP == 2 && halves == 2 && line_blocks(g) >= 256 ? 4 : 8);
  if (use_lds) {
    if (P >= 8) line_launch<NP, TR, 1, 8, CT, VT>(s, g, a, r.mode, lds);
    else if (P >= 4) line_launch<NP, TR, 1, 4, CT, VT>(s, g, a, r.mode, lds);
    else line_launch<NP, TR, 1, 1, CT, VT>(s, g, a, r.mode, lds);
  } else {
    if (P >= 8) line_launch<NP, TR, 0, 8, CT, VT>(s, g, a, r.mode, 0);
    else if (P >= 4) line_launch<NP, TR, 0, 4, CT, VT>(s, g, a, r.mode, 0);
    else line_launch<NP, TR, 0, 1, CT, VT>(s, g, a, r.mode, 0);
  }
}

}  // namespace asam
