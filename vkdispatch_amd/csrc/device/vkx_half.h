// vkx_half.h -- column kernels of 2-D real transforms, on packed half spectra.
//
// The row transform of a real image of even width W = 2M leaves M + 1 values per row, of
// which the first and the last are real.  Packed, they share slot 0 (X_0 + i X_M), and a
// row is M values: whole tiles of columns, without an odd one.  Down the columns slot 0
// is then the transform of two real columns at once, Z = A + i B with Hermitian A and B,
//   A[k] = (Z[k] + conj Z[-k]) / 2,  B[k] = (Z[k] - conj Z[-k]) / 2i,
// so a product with another spectrum is taken of A and of B and packed again.  Only the
// workgroups of the first tile do that, through LDS.
#pragma once
#include "vkx_long.h"

namespace vkx {

template <class T> __device__ __forceinline__ void unpack_pair(cpx<T> z, cpx<T> zm, cpx<T>& a, cpx<T>& b) {
  const T h = (T)0.5;
  a = cpx<T>{h * (z.x + zm.x), h * (z.y - zm.y)};
  b = cpx<T>{h * (z.y + zm.y), h * (zm.x - z.x)};
}
template <class T> __device__ __forceinline__ cpx<T> pack_pair(cpx<T> a, cpx<T> b) { return cpx<T>{a.x - b.y, a.y + b.x}; }

// The tile of a workgroup.  Tasks are (tile, group of images), groups fastest, and the
// workgroups of one XCD take consecutive tasks, so a tile's slice of the kernel spectrum
// is read from memory by one XCD.
template <class C, int FIRST = 0> struct HalfTask {
  int b, t, tile, group;
  u32 col;
  bool valid;  // not so: a column beyond the last, which does the last one's work unseen
  __device__ __forceinline__ HalfTask() {
    const int tid = (int)threadIdx.x;
    const u32 wg = logical_wg<C>();
    b = tid % C::B;
    t = tid / C::B;
    tile = (int)(wg / (u32)C::GROUPS) - FIRST;
    group = (int)(wg % (u32)C::GROUPS);
    col = (u32)(tile * C::B + b);
    valid = C::M % C::B == 0 || col < (u32)C::M;
    if (!valid) col = (u32)C::M - 1u;
  }
  // Between the transforms of a loop: addresses are computed again instead of being held
  // in registers through it (64 to 100 of them, which the spectra need).
  __device__ __forceinline__ void forget() { asm volatile("" : "+v"(t), "+v"(b), "+v"(col)); }
};

// Spectra lie as [image][H][SP] (SP >= M values per row).
template <class C> __device__ __forceinline__ u64 half_at(int image) { return (u64)image * (u64)(C::N * C::SP); }

// The rows of a thread's values are apart by constants, so one offset per thread serves
// all of them (the image's address is uniform).
template <class C, int R, class W_, class F> __device__ __forceinline__ void half_rows(const W_& w, F&& f) {
  constexpr int W = C::N / R, Q = (W + C::TT - 1) / C::TT;
  const u32 at = (u32)w.t * (u32)C::SP + w.col;
  sfor<0, Q>([&](auto qc) {
    constexpr int q = decltype(qc)::value;
    if ((q + 1) * C::TT <= W || w.t + q * C::TT < W) {
      sfor<0, R>([&](auto rc) {
        constexpr int r = decltype(rc)::value;
        f(ic<q * R + r>{}, (u32)(q * C::TT + r * W) * (u32)C::SP, at);
      });
    }
  });
}
template <class C, int R, class W_, class T>
__device__ __forceinline__ void half_load(const W_& w, const cpx<T>* s, cpx<T>* v) {
  half_rows<C, R>(w, [&](auto slot, u32 row, u32 at) { v[decltype(slot)::value] = (s + row)[at]; });
}
template <class C, int R, class W_, class T>
__device__ __forceinline__ void half_store(const W_& w, cpx<T>* s, const cpx<T>* v, T scale) {
  if (w.valid) half_rows<C, R>(w, [&](auto slot, u32 row, u32 at) { (s + row)[at] = v[decltype(slot)::value] * scale; });
}

// First tile only (uniform over the workgroup): column 0 between its registers and LDS.
template <class C, int R, class T>
__device__ __forceinline__ void pair_put(const HalfTask<C>& w, const cpx<T>* v, cpx<T>* p) {
  if (w.b == 0) for_layout<C, R>(w.t, [&](auto slot, u32 n) { p[n] = v[decltype(slot)::value]; });
}
template <class C, int R, class T>
__device__ __forceinline__ void pair_get(const HalfTask<C>& w, const cpx<T>* p, cpx<T>* v) {
  if (w.b == 0) for_layout<C, R>(w.t, [&](auto slot, u32 n) { v[decltype(slot)::value] = p[n]; });
}

// Kernel spectrum factor of element (n, col).  KHALF: a half spectrum [H][M + 1] as
// rfft2 gives it, of which the real image only meets the Hermitian part in columns 0 and
// M; otherwise packed [H][M].
template <class C, class T> struct HalfKernel {
  const cpx<T>* k;
  static constexpr u32 KP = C::KHALF ? (u32)(C::M + 1) : (u32)C::M;
  __device__ __forceinline__ cpx<T> plain(u32 n, u32 col) const {
    const cpx<T> z = k[n * KP + col];
    return C::CONJ ? conj(z) : z;
  }
  __device__ __forceinline__ void both(u32 n, cpx<T>& a, cpx<T>& b) const {
    const u32 m = n == 0u ? 0u : (u32)C::N - n;
    if constexpr (C::KHALF) {
      const T h = (T)0.5;
      const cpx<T> a0 = k[n * KP], a1 = k[m * KP], b0 = k[n * KP + (u32)C::M], b1 = k[m * KP + (u32)C::M];
      a = cpx<T>{h * (a0.x + a1.x), h * (a0.y - a1.y)};
      b = cpx<T>{h * (b0.x + b1.x), h * (b0.y - b1.y)};
    } else {
      unpack_pair(k[n * KP], k[m * KP], a, b);
    }
    if constexpr (C::CONJ) { a = conj(a); b = conj(b); }
  }
};

// z <- z . K for column 0 in LDS, each thread taking k and -k (all products are Hermitian).
template <class C, class T> __device__ __forceinline__ void pair_times_kernel(cpx<T>* z, const HalfKernel<C, T>& k) {
#pragma nounroll
  for (u32 n = threadIdx.x; n <= (u32)C::N / 2u; n += (u32)C::BLOCK) {
    const u32 m = n == 0u ? 0u : (u32)C::N - n;
    cpx<T> a, b, ka, kb;
    unpack_pair(z[n], z[m], a, b);
    k.both(n, ka, kb);
    a = cmul(a, ka);
    b = cmul(b, kb);
    z[m] = pack_pair(conj(a), conj(b));
    z[n] = pack_pair(a, b);
  }
}
// sum <- sum + x . conj g for column 0 in LDS.
template <class C, class T>
__device__ __forceinline__ void pair_add_product(cpx<T>* sum, const cpx<T>* x, const cpx<T>* g) {
#pragma nounroll
  for (u32 n = threadIdx.x; n <= (u32)C::N / 2u; n += (u32)C::BLOCK) {
    const u32 m = n == 0u ? 0u : (u32)C::N - n;
    cpx<T> xa, xb, ga, gb;
    unpack_pair(x[n], x[m], xa, xb);
    unpack_pair(g[n], g[m], ga, gb);
    xa = cmul(xa, conj(ga));
    xb = cmul(xb, conj(gb));
    if (m != n) sum[m] = sum[m] + pack_pair(conj(xa), conj(xb));
    sum[n] = sum[n] + pack_pair(xa, xb);
  }
}

// Convolution down the columns: FFT . K . IFFT, in place.  C: N = H, M, SP, B, TILES,
// IMAGES, PER (images per workgroup, one after another with K in registers), GROUPS =
// ceil(IMAGES / PER), KHALF, CONJ, KSTEP (elements from one image's K to the next; 0:
// one for all), SCALE, KEEP (the transforms are also stored).  Slots: 0 spectra, 1 K, 2 the
// transforms.
template <class C, class T>
__device__ __forceinline__ void half_conv_body(const KParams& prm) {
  using L = typename C::fwd;
  using LI = typename C::inv;
  using F0 = typename pl_first<L>::type;
  using FL = typename pl_last<L>::type;
  using IL = typename pl_last<LI>::type;
  __shared__ cpx<T> lds[C::LDS_ELEMS];
  __shared__ cpx<T> mir[C::N];
  HalfTask<C> w;
  const cpx<T>* twf = bufp<const cpx<T>>(prm, SLOT_TW_FWD);
  const cpx<T>* twi = bufp<const cpx<T>>(prm, SLOT_TW_INV);
  cpx<T> kv[C::VMAX];
  auto load_k = [&](const HalfKernel<C, T>& k) {
    for_layout<C, FL::R>(w.t, [&](auto slot, u32 n) { kv[decltype(slot)::value] = k.plain(n, w.col); });
  };
  HalfKernel<C, T> k{bufp<const cpx<T>>(prm, 1)};
  if constexpr (C::KSTEP == 0 && C::PER > 1) load_k(k);
#pragma nounroll
  for (int i = 0; i < C::PER; ++i) {
    const int image = w.group * C::PER + i;
    if (image >= C::IMAGES) break;  // uniform over the workgroup
    w.forget();
    cpx<T>* s = bufp<cpx<T>>(prm, 0) + half_at<C>(image);
    cpx<T> v[C::VMAX];
    half_load<C, F0::R>(w, s, v);
    if constexpr (C::KSTEP != 0) k.k = bufp<const cpx<T>>(prm, 1) + (u64)image * (u64)C::KSTEP;
    if constexpr (C::KSTEP != 0 || C::PER == 1) load_k(k);
    tile_passes<C, -1>(L{}, v, lds, w.t, w.b, w.t, w.b, twf);
    if constexpr (C::KEEP) half_store<C, FL::R>(w, bufp<cpx<T>>(prm, 2) + half_at<C>(image), v, (T)1);
    if (w.tile == 0) {
      pair_put<C, FL::R>(w, v, mir);
      __syncthreads();
      pair_times_kernel<C, T>(mir, k);
      __syncthreads();
    }
    for_layout<C, FL::R>(w.t, [&](auto slot, u32) {
      v[decltype(slot)::value] = cmul(v[decltype(slot)::value], kv[decltype(slot)::value]);
    });
    if (w.tile == 0) pair_get<C, FL::R>(w, mir, v);
    __syncthreads();
    w.forget();
    tile_passes<C, 1>(LI{}, v, lds, w.t, w.b, w.t, w.b, twi);
    half_store<C, IL::R>(w, s, v, (T)C::SCALE);
    if constexpr (C::PER > 1) __syncthreads();
  }
}

// The adjoint of the convolution y = x (*) k down the columns, for the rows' spectra of g,
// the transforms X that half_conv_body kept and the packed spectrum K of k:
//   dx = IFFT(G . K) over g (in place),  partial[group] = IFFT(sum over images X . conj G).
// One read of g and X and one write of dx, where separate transforms of g and x, their
// products and the batch sum crossed memory eight times.  The sum stays in registers over
// the workgroup's PER images.  Column 0 is left to workgroups of its own, the first GROUPS
// (each is one long chain), which hold its spectra in the LDS that the others exchange
// through.
// Slots: 0 g / dx, 1 X, 2 K, 3 partial [GROUPS][H][M].
template <class C> struct HalfColumn : C {  // one column per workgroup
  static constexpr int B = 1, PITCH = 1;
};
template <class C, class T>
__device__ __forceinline__ void half_grad_pair(const KParams& prm, cpx<T>* lds, int group) {
  using L = typename C::fwd;
  using LI = typename C::inv;
  using F0 = typename pl_first<L>::type;
  using FL = typename pl_last<L>::type;
  using IL = typename pl_last<LI>::type;
  using D = HalfColumn<C>;
  constexpr int EX = C::N + C::N / tile_first<C>::value + 1;
  static_assert(EX + 3 * C::N <= C::LDS_ELEMS, "column 0 in LDS");
  cpx<T>*mg = lds + EX, *mx = mg + C::N, *msum = mx + C::N;
  const cpx<T>* twf = bufp<const cpx<T>>(prm, SLOT_TW_FWD);
  const cpx<T>* twi = bufp<const cpx<T>>(prm, SLOT_TW_INV);
  const HalfKernel<C, T> k{bufp<const cpx<T>>(prm, 2)};
  int t = (int)threadIdx.x;
  const bool on = t < C::TT;
  auto forget = [&] { asm volatile("" : "+v"(t)); };
  cpx<T> v[C::VMAX];
  auto load = [&](const cpx<T>* s) {
    if (on) for_layout<D, F0::R>(t, [&](auto slot, u32 n) { v[decltype(slot)::value] = s[n * (u32)C::SP]; });
  };
  auto put = [&](cpx<T>* p) {
    if (on) for_layout<D, FL::R>(t, [&](auto slot, u32 n) { p[n] = v[decltype(slot)::value]; });
  };
  auto get = [&](const cpx<T>* p) {
    if (on) for_layout<D, FL::R>(t, [&](auto slot, u32 n) { v[decltype(slot)::value] = p[n]; });
  };
  for (int n = t; n < C::N; n += C::BLOCK) msum[n] = cpx<T>{(T)0, (T)0};
#pragma nounroll
  for (int i = 0; i < C::PER; ++i) {
    const int image = group * C::PER + i;
    if (image >= C::IMAGES) break;  // uniform over the workgroup
    cpx<T>* s = bufp<cpx<T>>(prm, 0) + half_at<C>(image);
    forget();
    load(s);
    tile_passes<D, -1>(L{}, v, lds, t, 0, t, 0, twf, on);
    put(mg);
    const cpx<T>* xs = bufp<const cpx<T>>(prm, 1) + half_at<C>(image);
    for (int n = (int)threadIdx.x; n < C::N; n += C::BLOCK) mx[n] = xs[(u32)n * (u32)C::SP];
    __syncthreads();
    pair_add_product<C, T>(msum, mx, mg);
    pair_times_kernel<C, T>(mg, k);  // k and -k are one thread's in both
    __syncthreads();
    forget();
    get(mg);
    tile_passes<D, 1>(LI{}, v, lds, t, 0, t, 0, twi, on);
    if (on)
      for_layout<D, IL::R>(t, [&](auto slot, u32 n) { s[n * (u32)C::SP] = v[decltype(slot)::value] * (T)C::SCALE; });
    __syncthreads();
  }
  get(msum);
  tile_passes<D, 1>(LI{}, v, lds, t, 0, t, 0, twi, on);
  if (on) {
    cpx<T>* p = bufp<cpx<T>>(prm, 3) + (u64)group * (u64)(C::N * C::M);
    for_layout<D, IL::R>(t, [&](auto slot, u32 n) { p[n * (u32)C::M] = v[decltype(slot)::value] * (T)C::SCALE; });
  }
}

template <class C, class T>
__device__ __forceinline__ void half_grad_body(const KParams& prm) {
  using L = typename C::fwd;
  using LI = typename C::inv;
  using F0 = typename pl_first<L>::type;
  using FL = typename pl_last<L>::type;
  using IL = typename pl_last<LI>::type;
  __shared__ cpx<T> lds[C::LDS_ELEMS];
  HalfTask<C, 1> w;
  if (w.tile < 0) {  // uniform over the workgroup
    half_grad_pair<C, T>(prm, lds, w.group);
    return;
  }
  if (w.tile == 0 && w.b == 0) w.valid = false;
  const cpx<T>* twf = bufp<const cpx<T>>(prm, SLOT_TW_FWD);
  const cpx<T>* twi = bufp<const cpx<T>>(prm, SLOT_TW_INV);
  const HalfKernel<C, T> k{bufp<const cpx<T>>(prm, 2)};
  cpx<T> sum[C::VMAX];
  sfor<0, C::VMAX>([&](auto i) { sum[decltype(i)::value] = cpx<T>{(T)0, (T)0}; });
#pragma nounroll
  for (int i = 0; i < C::PER; ++i) {
    const int image = w.group * C::PER + i;
    if (image >= C::IMAGES) break;  // uniform over the workgroup
    w.forget();
    cpx<T>* s = bufp<cpx<T>>(prm, 0) + half_at<C>(image);
    cpx<T> g[C::VMAX], x[C::VMAX];
    half_load<C, F0::R>(w, s, g);
    tile_passes<C, -1>(L{}, g, lds, w.t, w.b, w.t, w.b, twf);
    w.forget();
    half_load<C, FL::R>(w, bufp<const cpx<T>>(prm, 1) + half_at<C>(image), x);
    for_layout<C, FL::R>(w.t, [&](auto slot, u32) {
      constexpr int q = decltype(slot)::value;
      sum[q] = sum[q] + cmul(x[q], conj(g[q]));
      asm volatile("" : "+v"(sum[q].x), "+v"(sum[q].y));  // added here, so that X ends here
    });
    w.forget();
    for_layout<C, FL::R>(w.t, [&](auto slot, u32 n) {
      g[decltype(slot)::value] = cmul(g[decltype(slot)::value], k.plain(n, w.col));
    });
    __syncthreads();
    w.forget();
    tile_passes<C, 1>(LI{}, g, lds, w.t, w.b, w.t, w.b, twi);
    half_store<C, IL::R>(w, s, g, (T)C::SCALE);
    __syncthreads();
  }
  tile_passes<C, 1>(LI{}, sum, lds, w.t, w.b, w.t, w.b, twi);
  if (w.valid) {
    cpx<T>* p = bufp<cpx<T>>(prm, 3) + (u64)w.group * (u64)(C::N * C::M);
    for_layout<C, IL::R>(w.t, [&](auto slot, u32 n) {
      p[n * (u32)C::M + w.col] = sum[decltype(slot)::value] * (T)C::SCALE;
    });
  }
}

}  // namespace vkx
