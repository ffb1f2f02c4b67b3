// line_tile.h -- vertical-line preconditioner solve of one 64-column tile (shared by
// the single-domain and the ensemble kernels).
#pragma once
#include <type_traits>

#include "kcommon.h"

namespace asam {

template <typename CT, typename VT>
struct KLine {
  Coef<CT> c;
  int nx, ny, nz, tiled;
  const VT* src;
  VT* p;
  const VT* v;
  VT* out;
  const double* scale;
  const KState* st;
  double* partial;
  const int* done;
  int qslot;
  int kl;  // LDS staging: the first kl levels of each half are staged in LDS, the rest in the
           // output vector
  KTail fold;  // scalar tail folded into the launch (k_line only; kind < 0: none)
};

template <typename T> struct M4 { T m[4]; };

// Factor entries are read once per sweep and by no other kernel.  NT = 1 loads them
// nontemporal, so that factors larger than the Infinity Cache do not push out the vectors
// and operator arrays the neighbouring kernels reuse; NT = 0 lets factors that fit stay
// resident across solves.
template <int NT, typename T>
__device__ __forceinline__ M4<T> ld4(const T* __restrict__ p, long c) {
  M4<T> r;
  if constexpr (sizeof(T) == 4) {
    typedef float f4v __attribute__((ext_vector_type(4)));
    const f4v* q = reinterpret_cast<const f4v*>(p + 4 * c);
    f4v v;
    if constexpr (NT) v = __builtin_nontemporal_load(q); else v = *q;
    r.m[0] = v.x; r.m[1] = v.y; r.m[2] = v.z; r.m[3] = v.w;
  } else {
    typedef double d2v __attribute__((ext_vector_type(2)));
    const d2v* q = reinterpret_cast<const d2v*>(p + 4 * c);
    d2v v0, v1;
    if constexpr (NT) {
      v0 = __builtin_nontemporal_load(q);
      v1 = __builtin_nontemporal_load(q + 1);
    } else {
      v0 = q[0];
      v1 = q[1];
    }
    r.m[0] = v0.x; r.m[1] = v0.y; r.m[2] = v1.x; r.m[3] = v1.y;
  }
  return r;
}
template <typename T>
__device__ __forceinline__ V2<T> mv(const M4<T>& q, V2<T> v) {  // q * v, column-major 2x2
  return {q.m[0] * v.a + q.m[2] * v.b, q.m[1] * v.a + q.m[3] * v.b};
}
template <typename T>
__device__ __forceinline__ V2<T> mtv(const M4<T>& q, V2<T> v) {  // q^T * v
  return {q.m[0] * v.a + q.m[1] * v.b, q.m[2] * v.a + q.m[3] * v.b};
}

// One tile of the line solve: 64 columns (i = 64 bxl + lane) of row j, gxl tiles per row.
// Each sweep works through windows of P levels whose loads are all issued before the
// recurrence consumes them (the recurrence itself is sequential, so memory-level parallelism
// has to come from the window and the wavefronts).
//
// HV = 1, one wavefront: elimination from the bottom to the top, back-substitution down.
// HV = 2, two wavefronts: elimination from both ends towards level m (k_factor); the first
// wavefront takes levels 0..m-1 upwards, the second nz-1..m+1 downwards and then m, where the
// halves meet; the back-substitution runs outwards from there.  That halves the serial chain
// of a column and doubles the loads in flight, which counts where the grid has too few tiles
// to hide either (see line_halves for both sides measured).  Kernel times, one / two:
// FP64 64x64x40 one component 12.4 / 9.1 us, 2x2 17.8 / 12.9 us; transposed 2x2 130x97x40
// 31 / 28 us.
//
// NT: cache policy of the factor loads, of the two vectors only this kernel reads (p in
// the p-step, v in the s-step) and of the p-step's store of p (read again only by the next
// iteration's p-step), see ld4.  PBW: levels per window of the back-substitution (0: P); it
// runs after the whole elimination, its partial window first.
//
// All 64 HV threads of the workgroup call it (two barriers with HV = 2).
template <int NP, int TR, int MODE, int LDS, int P, int HV, typename CT, typename VT, int NT = 1,
          int PBW = 0>
__device__ __forceinline__ void line_tile(const KLine<CT, VT>& a, int bxl, int j, int gxl,
                                          CT* stage, double (&acc)[1]) {
  const int nx = a.nx, nz = a.nz;
  const long sz = (long)nx * a.ny;
  const int tid = threadIdx.x & 63;
  const int half = HV == 1 ? 0 : __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int i = bxl * 64 + tid;
  const bool on = i < nx;
  const int mid = nz / 2;
  // levels of this half (ahead of the meeting one)
  const int nf = HV == 1 ? nz : half ? nz - 1 - mid : mid;
  const CT* __restrict__ PL = a.c.pl;
  const CT* __restrict__ PT = a.c.pt;
  const CT* __restrict__ PW = a.c.pw;
  const VT* __restrict__ SRC = a.src;
  const VT* __restrict__ VV = a.v;
  VT* __restrict__ OUT = a.out;
  VT* __restrict__ PP = a.p;
  using V = V2<CT>;
  using M = M4<CT>;
  const long c00 = i + (long)nx * j;
  // factor entries: tiled (64-column tiles, levels contiguous) or x-fastest
  const long f00 = a.tiled ? (((long)j * gxl + bxl) * nz) * 64 + tid : c00;
  const long fs0 = a.tiled ? 64 : sz;
  // the q-th level of this half lies at c0 + q*cs (cells) and f0 + q*fs (factor entries)
  const long c0 = half ? c00 + sz * (nz - 1) : c00, cs = half ? -sz : sz;
  const long f0 = half ? f00 + fs0 * (nz - 1) : f00, fs = half ? -fs0 : fs0;
  CT alpha = 0, beta = 0, omega = 0, sc = 1;
  bool first = false;
  if constexpr (MODE == LINE_BICG_P) {
    first = a.st->iter == 1;
    beta = (CT)a.st->beta; omega = (CT)a.st->omega;
  }
  if constexpr (MODE == LINE_BICG_S) alpha = (CT)a.st->alpha;
  if constexpr (MODE == LINE_PLAIN) { if (a.scale) sc = (CT)(*a.scale); }
  // --- per-level helpers (NP = 1 uses the .a lane of V / m[0] of M only)
  auto ldv = [&](const VT* p, long c) -> V {
    if constexpr (NP == 1) return V{(CT)p[c], (CT)0};
    else { V2<VT> t = ld2(p, c); return V{(CT)t.a, (CT)t.b}; }
  };
  auto ldvo = [&](const VT* p, long c) -> V {  // a vector this kernel alone reads
    if constexpr (NT == 0) return ldv(p, c);
    else if constexpr (NP == 1) return V{(CT)__builtin_nontemporal_load(p + c), (CT)0};
    else {
      typedef VT v2v __attribute__((ext_vector_type(2)));
      const v2v t = __builtin_nontemporal_load(reinterpret_cast<const v2v*>(p + 2 * c));
      return V{(CT)t.x, (CT)t.y};
    }
  };
  auto stvn = [&](VT* p, long c, V v) {
    if constexpr (NP == 1) __builtin_nontemporal_store((VT)v.a, p + c);
    else {
      typedef VT v2v __attribute__((ext_vector_type(2)));
      v2v t; t.x = (VT)v.a; t.y = (VT)v.b;
      __builtin_nontemporal_store(t, reinterpret_cast<v2v*>(p + 2 * c));
    }
  };
  auto stv = [&](VT* p, long c, V v) {
    if constexpr (NP == 1) p[c] = (VT)v.a; else st2(p, c, v.a, v.b);
  };
  auto ldm = [&](const CT* p, long c) -> M {
    if constexpr (NP == 1) {
      if constexpr (NT) return M{{__builtin_nontemporal_load(p + c), (CT)0, (CT)0, (CT)0}};
      else return M{{p[c], (CT)0, (CT)0, (CT)0}};
    } else {
      return ld4<NT>(p, c);
    }
  };
  // a lower block L: for 2x2 blocks the three words (tz, v0, v1) of
  // L = (tz, 1)^T (v0, v1), in m[0..2]
  auto ldl = [&](const CT* p, long c) -> M {
    if constexpr (NP == 1) {
      return ldm(p, c);
    } else {
      const CT* q = p + 3 * c;
      if constexpr (NT)
        return M{{__builtin_nontemporal_load(q), __builtin_nontemporal_load(q + 1),
                  __builtin_nontemporal_load(q + 2), (CT)0}};
      else
        return M{{q[0], q[1], q[2], (CT)0}};
    }
  };
  auto mull = [&](const M& l, V y) -> V {  // L y = (tz s, s), s = v0 y.a + v1 y.b
    if constexpr (NP == 1) {
      return V{l.m[0] * y.a, (CT)0};
    } else {
      const CT s = l.m[1] * y.a + l.m[2] * y.b;
      return V{l.m[0] * s, s};
    }
  };
  auto mullT = [&](const M& l, V z) -> V {  // L^T z = (v0 t, v1 t), t = tz z.a + z.b
    if constexpr (NP == 1) {
      return V{l.m[0] * z.a, (CT)0};
    } else {
      const CT t = l.m[0] * z.a + z.b;
      return V{l.m[1] * t, l.m[2] * t};
    }
  };
  auto mul = [&](const M& m, V v) -> V {  // m * v
    if constexpr (NP == 1) return V{m.m[0] * v.a, (CT)0};
    else return mv(m, v);
  };
  auto mulT = [&](const M& m, V v) -> V {  // m^T * v
    if constexpr (NP == 1) return V{m.m[0] * v.a, (CT)0};
    else return mtv(m, v);
  };
  // Results of the elimination: the first kl levels of the half in LDS (written first, read
  // last, so the ones a round trip through memory would most likely miss in the caches),
  // the others in the output vector (their reads follow the writes closely).  q is the same
  // in every lane, so the test is a uniform branch.
  CT* const st = stage + (long)half * a.kl * NP * 64 + tid;
  auto stage_put = [&](int q, long c, V y) {
    if constexpr (LDS) {
      if (q < a.kl) {
        st[(NP * q) * 64] = y.a;
        if constexpr (NP == 2) st[(2 * q + 1) * 64] = y.b;
        return;
      }
    }
    stv(OUT, c, y);
  };
  auto stage_get = [&](int q, long c) -> V {
    if constexpr (LDS) {
      if (q < a.kl) {
        if constexpr (NP == 1) return V{st[q * 64], (CT)0};
        else return V{st[(2 * q) * 64], st[(2 * q + 1) * 64]};
      }
    }
    return ldv((const VT*)OUT, c);
  };
  struct In {
    V r, p, v;
  };
  auto ld_in = [&](long c) {
    In x{};
    if constexpr (MODE == LINE_PLAIN) x.r = ldv(SRC, c);
    if constexpr (MODE == LINE_BICG_P) {
      x.r = ldv(SRC, c);
      if (!first) { x.p = ldvo((const VT*)PP, c); x.v = ldv(VV, c); }
    }
    if constexpr (MODE == LINE_BICG_S) { x.r = ldv((const VT*)PP, c); x.v = ldvo(VV, c); }
    return x;
  };
  auto form_in = [&](const In& x, long c) {
    V in;
    if constexpr (MODE == LINE_PLAIN) in = V{x.r.a * sc, x.r.b * sc};
    else if constexpr (MODE == LINE_BICG_P) {
      in = first ? x.r
                 : V{x.r.a + beta * (x.p.a - omega * x.v.a),
                     x.r.b + beta * (x.p.b - omega * x.v.b)};
      if constexpr (NT) stvn(PP, c, in); else stv(PP, c, in);
    } else {
      in = V{x.r.a - alpha * x.v.a, x.r.b - alpha * x.v.b};
      stv(PP, c, in);
      acc[0] += (double)in.a * (double)in.a + (double)in.b * (double)in.b;
    }
    return in;
  };
  // --- elimination: y_k = t_k^-1 (in_k - l_k y_prev)   (transposed: in_k - w_prev^T y_prev)
  V yprev{0, 0};
  auto fwd = [&](int q0, auto chk) {
    constexpr bool CHK = decltype(chk)::value;
    In x_[P];
    M l_[P], t_[P];
#pragma unroll
    for (int e = 0; e < P; ++e) {
      const int q = q0 + e;
      if (!CHK || q < nf) {
        x_[e] = ld_in(c0 + cs * q);
        const long f = f0 + fs * q;
        if constexpr (TR == 0) { l_[e] = ldl(PL, f); t_[e] = ldm(PT, f); }
        else l_[e] = (q > 0) ? ldm(PW, f - fs) : M{{0, 0, 0, 0}};
      }
    }
#pragma unroll
    for (int e = 0; e < P; ++e) {
      const int q = q0 + e;
      if (!CHK || q < nf) {
        const long c = c0 + cs * q;
        const V in = form_in(x_[e], c);
        V y;
        if constexpr (TR == 0) {
          const V ly = mull(l_[e], yprev);
          y = mul(t_[e], V{in.a - ly.a, in.b - ly.b});
        } else {
          const V wy = mulT(l_[e], yprev);
          y = V{in.a - wy.a, in.b - wy.b};
        }
        stage_put(q, c, y);
        yprev = y;
      }
    }
  };
  auto eliminate = [&]() {
    const int nfull = nf / P;
    for (int w = 0; w < nfull; ++w) fwd(w * P, std::false_type{});
    if (nfull * P < nf) fwd(nfull * P, std::true_type{});
  };
  V znext{0, 0};
  if constexpr (HV == 1) {
    if (on) eliminate();
  } else {
    __shared__ CT meet[2][NP][64];  // the first half's term of level m, and the solution there
    // the meeting level (second half), and the first half's coupling to it
    const long cm = c0 + cs * nf, fm = f0 + fs * nf;
    In xm{};
    M lm{}, tm{};
    if (on && half) {
      xm = ld_in(cm);
      tm = ldm(PT, fm);
      if constexpr (TR == 0) lm = ldl(PL, fm);
      else if (nf > 0) lm = ldm(PW, fm - fs);
    } else if (on && nf > 0) {
      if constexpr (TR == 0) lm = ldl(PL, f0);  // L_m, kept in the bottom level's unused place
      else lm = ldm(PW, fm - fs);
    }
    if (on) eliminate();
    if (half == 0) {
      V y;
      if constexpr (TR == 0) y = mull(lm, yprev); else y = mulT(lm, yprev);
      meet[0][0][tid] = y.a;
      if constexpr (NP == 2) meet[0][1][tid] = y.b;
    }
    __syncthreads();
    if (half) {
      if (on) {
        V in = form_in(xm, cm), y;
        if constexpr (TR == 0) y = mull(lm, yprev); else y = mulT(lm, yprev);
        in = V{in.a - y.a - meet[0][0][tid], in.b - y.b};
        if constexpr (NP == 2) in.b -= meet[0][1][tid];
        if constexpr (TR == 0) znext = mul(tm, in); else znext = mulT(tm, in);
        stv(OUT, cm, V{-znext.a, -znext.b});
      }
      meet[1][0][tid] = znext.a;
      if constexpr (NP == 2) meet[1][1][tid] = znext.b;
    }
    __syncthreads();
    if (half == 0) {
      znext.a = meet[1][0][tid];
      if constexpr (NP == 2) znext.b = meet[1][1][tid];
    }
  }
  // --- back-substitution: z_k = y_k - w_k z_next   (transposed: t_k^-T (y_k - l_next^T z_next))
  constexpr int PB = PBW > 0 ? PBW : P;
  auto bwd = [&](int q0, auto chk) {
    constexpr bool CHK = decltype(chk)::value;
    V y_[PB];
    M w_[PB], t_[PB];
#pragma unroll
    for (int e = 0; e < PB; ++e) {
      const int q = q0 + e;
      if (!CHK || q < nf) {
        y_[e] = stage_get(q, c0 + cs * q);
        const long f = f0 + fs * q;
        if constexpr (TR == 0) w_[e] = ldm(PW, f);
        else {
          if constexpr (HV == 1) w_[e] = q + 1 < nf ? ldl(PL, f + fs) : M{{0, 0, 0, 0}};
          else w_[e] = ldl(PL, half == 0 && q == nf - 1 ? f0 : f + fs);
          t_[e] = ldm(PT, f);
        }
      }
    }
#pragma unroll
    for (int e = PB - 1; e >= 0; --e) {
      const int q = q0 + e;
      if (!CHK || q < nf) {
        V z;
        if constexpr (TR == 0) {
          const V wz = mul(w_[e], znext);
          z = V{y_[e].a - wz.a, y_[e].b - wz.b};
        } else {
          const V lz = mullT(w_[e], znext);
          z = mulT(t_[e], V{y_[e].a - lz.a, y_[e].b - lz.b});
        }
        stv(OUT, c0 + cs * q, V{-z.a, -z.b});
        znext = z;
      }
    }
  };
  if (on) {
    const int nfb = nf / PB;
    if (nfb * PB < nf) bwd(nfb * PB, std::true_type{});
    for (int w = nfb - 1; w >= 0; --w) bwd(w * PB, std::false_type{});
  }
}

}  // namespace asam
