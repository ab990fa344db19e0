// vkx_long.h -- transforms longer than one workgroup holds, in two launches.
//
// A transform of length L = n1 n2 (x[j1 n2 + j2], X[k1 + n1 k2]) runs as n2 transforms
// of length n1 down the columns, times W_L^(k1 j2), then n1 transforms of length n2
// along the rows.  A workgroup holds a tile of B neighbouring transforms in registers
// and exchanges through LDS between the passes, so each launch reads and writes the data
// once.  Between the launches the data lies in tiles of the second launch,
//   y[k1 / B2][j2][k1 mod B2],
// so that a row workgroup reads one contiguous block; its writes, and the column
// workgroups' reads, are runs of B elements.  The column kernel turns the tile in the
// last LDS exchange it makes anyway: up to there a thread's neighbours hold the
// neighbouring columns (for the reads), from there on the neighbouring frequencies (for
// runs of B2 in y).
#pragma once
#include "vkx_fft.h"

namespace vkx {

// LDS element (b, pos) of a tile at pos PITCH + b, plus B for every R0 positions (R0: the
// first radix): in the first exchange neighbouring threads write R0 positions apart and
// would meet the same banks.  Every later stride is a multiple of R0, so a butterfly's
// legs are constant offsets from one address.
template <class C> struct tile_first { static constexpr int value = pl_first<typename C::fwd>::type::R; };
template <class C> __device__ __forceinline__ int tile_addr(int b, int pos) {
  return pos * C::PITCH + b + (pos / tile_first<C>::value) * C::B;
}
template <class C> constexpr int tile_step(int pos) {  // of a multiple of R0
  return pos * C::PITCH + (pos / tile_first<C>::value) * C::B;
}

template <class C, int R, int NS>
__device__ __forceinline__ void tile_put(cpx<typename C::real>* lds, const cpx<typename C::real>* v, int t, int b) {
  constexpr int W = C::N / R, Q = (W + C::TT - 1) / C::TT;
  sfor<0, Q>([&](auto qc) {
    constexpr int q = decltype(qc)::value;
    const int j = t + q * C::TT;
    if ((q + 1) * C::TT <= W || j < W) {
      const int base = NS == 1 ? j * R : (j / NS) * NS * R + j % NS;
      cpx<typename C::real>* p = lds + tile_addr<C>(b, base);
      sfor<0, R>([&](auto rc) {
        constexpr int r = decltype(rc)::value;
        if constexpr (NS % tile_first<C>::value == 0) p[tile_step<C>(r * NS)] = v[q * R + r];
        else if constexpr (NS == 1 && R == tile_first<C>::value) p[r * C::PITCH] = v[q * R + r];
        else lds[tile_addr<C>(b, base + r * NS)] = v[q * R + r];
      });
    }
  });
}

template <class C, int R>
__device__ __forceinline__ void tile_get(const cpx<typename C::real>* lds, cpx<typename C::real>* v, int t, int b) {
  constexpr int W = C::N / R, Q = (W + C::TT - 1) / C::TT;
  sfor<0, Q>([&](auto qc) {
    constexpr int q = decltype(qc)::value;
    const int j = t + q * C::TT;
    if ((q + 1) * C::TT <= W || j < W) {
      const cpx<typename C::real>* p = lds + tile_addr<C>(b, j);
      sfor<0, R>([&](auto rc) {
        constexpr int r = decltype(rc)::value;
        if constexpr (W % tile_first<C>::value == 0) v[q * R + r] = p[tile_step<C>(r * W)];
        else v[q * R + r] = lds[tile_addr<C>(b, j + r * W)];
      });
    }
  });
}

// The pass list on a tile.  (t, b): position of the thread while neighbours hold
// neighbouring transforms; (tl, bl): its position in the last pass.  A thread that is not
// `on` only meets the barriers.
template <class C, int DIR, class Cur, class... Rest>
__device__ __forceinline__ void tile_passes_(cpx<typename C::real>* v, cpx<typename C::real>* lds, int t, int b,
                                             int tl, int bl, const cpx<typename C::real>* tw, bool on) {
  if (on) pass_compute<C, Cur::R, Cur::NS, DIR>(v, t, tw);
  if constexpr (sizeof...(Rest) > 0) {
    using Nx = typename pl_first<PL<Rest...>>::type;
    constexpr bool last = sizeof...(Rest) == 1;
    if (on) tile_put<C, Cur::R, Cur::NS>(lds, v, t, b);
    __syncthreads();
    const int tn = last ? tl : t, bn = last ? bl : b;
    if (on) tile_get<C, Nx::R>(lds, v, tn, bn);
    if constexpr (!last) __syncthreads();
    tile_passes_<C, DIR, Rest...>(v, lds, tn, bn, tl, bl, tw, on);
  }
}
template <class C, int DIR, class... Ps>
__device__ __forceinline__ void tile_passes(PL<Ps...>, cpx<typename C::real>* v, cpx<typename C::real>* lds, int t,
                                            int b, int tl, int bl, const cpx<typename C::real>* tw, bool on = true) {
  tile_passes_<C, DIR, Ps...>(v, lds, t, b, tl, bl, tw, on);
}

// Columns.  C: N = n1, N2, B (columns of a tile), B2 (rows of a tile of the second
// launch), TILES = ceil(N2 / B), YS (elements of y per transform), INV.
// Slots: 0 y, 1 x, 2 W_L^(j j2) as [j2][j] for j < N / R, 3 W_(R n2)^(r j2) as [j2][r]
// (R: the last radix; k1 = j + r N / R, so the product of the two is W_L^(k1 j2)).  Both
// are held and multiplied in double, so that the twiddle is rounded once: with rounded
// factors 2^20 points came 8 % further from the exact transform.
template <class C, class In>
__device__ __forceinline__ void long_cols_body(const KParams& prm) {
  using real = float;
  using L = typename C::fwd;
  using F0 = typename pl_first<L>::type;
  using FL = typename pl_last<L>::type;
  constexpr int R = FL::R, W = C::N / R;
  __shared__ cpx<real> lds[C::LDS_ELEMS];
  __shared__ cpx<double> rot[C::B * R];
  const int tid = (int)threadIdx.x;
  const int b = tid % C::B, t = tid / C::B, tl = tid % C::TT, bl = tid / C::TT;
  const u32 wg = logical_wg<C>();
  const u32 batch = wg / (u32)C::TILES;
  const int j20 = (int)(wg % (u32)C::TILES) * C::B;
  cpx<real> v[C::VMAX];
  if (C::N2 % C::B == 0 || j20 + b < C::N2) {
    const In in(prm, batch);
    for_layout<C, F0::R>(t, [&](auto slot, u32 n) {
      v[decltype(slot)::value] = in(n * (u32)C::N2 + (u32)(j20 + b));
    });
  } else {
    sfor<0, C::VMAX>([&](auto s) { v[decltype(s)::value] = cpx<real>{0.f, 0.f}; });
  }
  {
    const cpx<double>* rt = bufp<const cpx<double>>(prm, 3) + (u32)j20 * (u32)R;
    const int have = (C::N2 - j20 < C::B ? C::N2 - j20 : C::B) * R;
    for (int i = tid; i < have; i += C::BLOCK) rot[i] = rt[i];
  }
  tile_passes<C, (C::INV ? 1 : -1)>(L{}, v, lds, t, b, tl, bl, bufp<const cpx<real>>(prm, SLOT_TW_FWD));
  const int j2 = j20 + bl;
  if (C::N2 % C::B == 0 || j2 < C::N2) {
    const cpx<double>* col = bufp<const cpx<double>>(prm, 2) + (u32)j2 * (u32)W;
    cpx<real>* y = bufp<cpx<real>>(prm, 0) + (u64)batch * (u64)C::YS;
    constexpr int Q = (W + C::TT - 1) / C::TT;
    sfor<0, Q>([&](auto qc) {
      constexpr int q = decltype(qc)::value;
      constexpr bool full = (q + 1) * C::TT <= W;
      const int j = tl + q * C::TT;
      if (full || j < W) {
        const cpx<double> a = col[j];
        sfor<0, R>([&](auto rc) {
          constexpr int r = decltype(rc)::value;
          cpx<real> w = ccvt<real>(r == 0 ? a : cmul(a, rot[bl * R + r]));
          if constexpr (C::INV) w.y = -w.y;
          const u32 k1 = (u32)(j + r * W);
          y[((k1 / (u32)C::B2) * (u32)C::N2 + (u32)j2) * (u32)C::B2 + k1 % (u32)C::B2] = cmul(v[q * R + r], w);
        });
      }
    });
  }
}

// Rows.  C: N = n2, N1, B (rows of a tile), TILES = ceil(N1 / B), YS, INV, NORMALIZE,
// SCALE.  Slots: 0 X, 1 y.
template <class C, class Out>
__device__ __forceinline__ void long_rows_body(const KParams& prm) {
  using real = float;
  using L = typename C::fwd;
  using F0 = typename pl_first<L>::type;
  using FL = typename pl_last<L>::type;
  __shared__ cpx<real> lds[C::LDS_ELEMS];
  const int tid = (int)threadIdx.x;
  const int b = tid % C::B, t = tid / C::B;
  const u32 wg = logical_wg<C>();
  const u32 batch = wg / (u32)C::TILES, tile = wg % (u32)C::TILES;
  const u32 k1 = tile * (u32)C::B + (u32)b;
  cpx<real> v[C::VMAX];
  if (C::N1 % C::B == 0 || k1 < (u32)C::N1) {
    const cpx<real>* y = bufp<const cpx<real>>(prm, 1) + (u64)batch * (u64)C::YS + (u64)tile * (u64)(C::N * C::B);
    for_layout<C, F0::R>(t, [&](auto slot, u32 n) { v[decltype(slot)::value] = y[n * (u32)C::B + (u32)b]; });
  } else {
    sfor<0, C::VMAX>([&](auto s) { v[decltype(s)::value] = cpx<real>{0.f, 0.f}; });
  }
  tile_passes<C, (C::INV ? 1 : -1)>(L{}, v, lds, t, b, t, b, bufp<const cpx<real>>(prm, SLOT_TW_FWD));
  if (C::N1 % C::B == 0 || k1 < (u32)C::N1) {
    const Out out(prm, batch);
    for_layout<C, FL::R>(t, [&](auto slot, u32 n) {
      cpx<real> z = v[decltype(slot)::value];
      if constexpr (C::NORMALIZE) z = z * (real)C::SCALE;
      out(n * (u32)C::N1 + k1, z);
    });
  }
}

// Where a transform lies: one after another (transform b at b L), in slot SLOT.
template <int SLOT, u64 L> struct PackedIn {
  const cpx<float>* x;
  __device__ __forceinline__ PackedIn(const KParams& prm, u32 b) : x(bufp<const cpx<float>>(prm, SLOT) + (u64)b * L) {}
  __device__ __forceinline__ cpx<float> operator()(u32 i) const { return x[i]; }
};
template <int SLOT, u64 L> struct PackedOut {
  cpx<float>* x;
  __device__ __forceinline__ PackedOut(const KParams& prm, u32 b) : x(bufp<cpx<float>>(prm, SLOT) + (u64)b * L) {}
  __device__ __forceinline__ void operator()(u32 i, cpx<float> z) const { x[i] = z; }
};

}  // namespace vkx
