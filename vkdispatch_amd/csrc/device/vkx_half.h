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
// ceil(IMAGES / PER), KHALF, CONJ, SCALE, KEEP (the transforms are also stored).  Slots: 0 spectra, 1 K, 2 the
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
  const HalfKernel<C, T> k{bufp<const cpx<T>>(prm, 1)};
  for_layout<C, FL::R>(w.t, [&](auto slot, u32 n) { kv[decltype(slot)::value] = k.plain(n, w.col); });
#pragma nounroll
  for (int i = 0; i < C::PER; ++i) {
    const int image = w.group * C::PER + i;
    if (image >= C::IMAGES) break;  // uniform over the workgroup
    w.forget();
    cpx<T>* s = bufp<cpx<T>>(prm, 0) + half_at<C>(image);
    cpx<T> v[C::VMAX];
    half_load<C, F0::R>(w, s, v);
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

// ---------------------------------------------------------------------------
// The whole convolution of one image in one workgroup: rows, columns . K, columns and
// rows back, with the image in LDS in between, where three launches crossed memory three
// times.  A line (row or column) belongs to one wave: its TT threads exchange through its
// own LDS without a barrier, and the workgroup meets only twice, between rows and columns.
// C: N = H, M, BLOCK, RP (pitch; chosen so that neither direction meets the same banks),
// IMG (reals per image), RowCfg / ColCfg (N, TT, VMAX, fwd, inv), KHALF / CONJ / KSTEP
// (elements from one image's K to the next; 0: one for all), SCALE (of the whole), ROOTS (a
// multiple of 2M and H).  Slots: 0 images (rows of 2M + 2 reals, in place), 1 K.
//
// Bound by the vector unit: at 256 images of 128^2, one per CU, 19 us, of which the
// transforms' adds and products are 8 (no packed FP32) and memory 4; three launches took 37.
// ---------------------------------------------------------------------------
__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}
template <class C, int STRIDE, int R, int NS, class T>
__device__ __forceinline__ void line_put(cpx<T>* line, const cpx<T>* v, int t) {
  constexpr int W = C::N / R, Q = (W + C::TT - 1) / C::TT;
  sfor<0, Q>([&](auto qc) {
    constexpr int q = decltype(qc)::value;
    const int j = t + q * C::TT;
    if ((q + 1) * C::TT <= W || j < W) {
      cpx<T>* p = line + (NS == 1 ? j * R : (j / NS) * NS * R + j % NS) * STRIDE;
      sfor<0, R>([&](auto rc) { p[decltype(rc)::value * NS * STRIDE] = v[q * R + decltype(rc)::value]; });
    }
  });
}
template <class C, int STRIDE, int R, class T>
__device__ __forceinline__ void line_get(const cpx<T>* line, cpx<T>* v, int t) {
  constexpr int W = C::N / R, Q = (W + C::TT - 1) / C::TT;
  sfor<0, Q>([&](auto qc) {
    constexpr int q = decltype(qc)::value;
    const int j = t + q * C::TT;
    if ((q + 1) * C::TT <= W || j < W) {
      const cpx<T>* p = line + j * STRIDE;
      sfor<0, R>([&](auto rc) { v[q * R + decltype(rc)::value] = p[decltype(rc)::value * W * STRIDE]; });
    }
  });
}
// f(slot, row, column) over `have` rows of M values, lane by lane: one division per call,
// then steps.
template <int M, int IT, class F> __device__ __forceinline__ void row_points(int lane, int have, F&& f) {
  int y = lane / M, n = lane % M;
  sfor<0, IT>([&](auto ic_) {
    if (y < have) f(ic_, y, n);
    n += 64 % M;
    y += 64 / M;
    if (64 % M != 0 && n >= M) { n -= M; y += 1; }
  });
}

// The twiddle table of a pass list (see pass_compute) from the roots of order C::ROOTS.
template <class L> struct list_twiddles;
template <class... Ps> struct list_twiddles<PL<Ps...>> { static constexpr int value = (0 + ... + ((Ps::R - 1) * Ps::NS)); };
template <class C, class T, class... Ps>
__device__ __forceinline__ void fill_twiddles(PL<Ps...>, cpx<T>* tab, const cpx<T>* roots) {
  auto one = [&](auto rc, auto ns) {
    constexpr int R = decltype(rc)::value, NS = decltype(ns)::value, STEP = C::ROOTS / (R * NS);
    if constexpr (NS > 1)
      for (int i = (int)threadIdx.x; i < (R - 1) * NS; i += C::BLOCK)
        tab[NS - 1 + i] = roots[(i / NS + 1) * (i % NS) % (R * NS) * STEP];
  };
  (one(ic<Ps::R>{}, ic<Ps::NS>{}), ...);
}

// The pass list on a line, from registers (first pass's order) to registers (last pass's).
template <class C, int STRIDE, int DIR, class T, class Cur, class... Rest>
__device__ __forceinline__ void line_passes(PL<Cur, Rest...>, cpx<T>* v, cpx<T>* line, int t, const cpx<T>* tw, bool on) {
  if (on) pass_compute<C, Cur::R, Cur::NS, DIR>(v, t, tw);
  if constexpr (sizeof...(Rest) > 0) {
    wave_sync();
    if (on) line_put<C, STRIDE, Cur::R, Cur::NS>(line, v, t);
    wave_sync();
    if (on) line_get<C, STRIDE, pl_first<PL<Rest...>>::type::R>(line, v, t);
    line_passes<C, STRIDE, DIR>(PL<Rest...>{}, v, line, t, tw, on);
  }
}

template <class C, class T>
__device__ __forceinline__ void half_whole_body(const KParams& prm) {
  using RC = typename C::RowCfg;
  using CC = typename C::ColCfg;
  using RF = typename RC::fwd;
  using CF = typename CC::fwd;
  using CI = typename CC::inv;
  __shared__ cpx<T> lds[C::N * C::RP];
  // Twiddles and roots in LDS: a pass then waits for LDS and not for L2, and each of the
  // passes is a link of one chain.  All come from one table of roots of order ROOTS.
  constexpr int NR = list_twiddles<typename RC::fwd>::value, NC = list_twiddles<typename CC::fwd>::value;
  constexpr int PAIRS = C::M / 2 + 1;
  __shared__ cpx<T> tab[NR + 2 * NC + PAIRS];
  const cpx<T>*row_tw = tab, *col_fwd = tab + NR, *col_inv = col_fwd + NC, *roots = col_inv + NC;
  {
    const cpx<T>* w = bufp<const cpx<T>>(prm, SLOT_ROOTS);
    fill_twiddles<C>(RF{}, tab, w);
    fill_twiddles<C>(CF{}, tab + NR, w);
    fill_twiddles<C>(CI{}, tab + NR + NC, w);
    for (int i = (int)threadIdx.x; i < PAIRS; i += C::BLOCK) tab[NR + 2 * NC + i] = w[i * (C::ROOTS / (2 * C::M))];
  }
  const int lane = (int)threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  constexpr int WAVES = C::BLOCK / 64;
  constexpr int RL = 64 / RC::TT, CL = 64 / CC::TT;  // lines of a wave
  const u32 image = blockIdx.x;
  cpx<T>* x = reinterpret_cast<cpx<T>*>(bufp<T>(prm, 0) + (u64)image * (u64)C::IMG);
  const HalfKernel<C, T> k{bufp<const cpx<T>>(prm, 1) + (u64)image * (u64)C::KSTEP};
  constexpr int IT = (RL * C::M + 63) / 64;
  int rt = lane % RC::TT, ct = lane % CC::TT;
  __syncthreads();  // the tables
  // addresses are computed again in each round of a loop, not held through it
  auto forget = [&] { asm volatile("" : "+v"(rt), "+v"(ct)); };

#pragma nounroll
  for (int y0 = wave * RL; y0 < C::N; y0 += WAVES * RL) {
    forget();
    cpx<T>* rows = lds + y0 * C::RP;
    const int have = (C::N - y0 < RL ? C::N - y0 : RL);
    {
      cpx<T> v[IT];  // the wave's rows, every load in flight before the first is waited for
      cpx<T>* xr = x + y0 * (C::M + 1);
      row_points<C::M, IT>(lane, have, [&](auto ic_, int y, int n) { v[decltype(ic_)::value] = xr[y * (C::M + 1) + n]; });
      row_points<C::M, IT>(lane, have, [&](auto ic_, int y, int n) { rows[y * C::RP + n] = v[decltype(ic_)::value]; });
    }
    const bool on = lane < have * RC::TT;
    cpx<T>* row = rows + lane / RC::TT * C::RP;
    cpx<T> v[RC::VMAX];
    wave_sync();
    if (on) line_get<RC, 1, pl_first<RF>::type::R>(row, v, rt);
    line_passes<RC, 1, -1, T>(RF{}, v, row, rt, row_tw, on);
    wave_sync();
    if (on) for_layout<RC, pl_last<RF>::type::R>(rt, [&](auto slot, u32 n) { row[n] = v[decltype(slot)::value]; });
    wave_sync();
    // half-length transform -> packed spectrum, q and M - q by one thread of the row
    if (on) {
      for (int q = rt; q < PAIRS; q += RC::TT) {
        const cpx<T> zk = row[q], zm = row[q == 0 ? 0 : C::M - q];
        if (q == 0) {
          row[0] = cpx<T>{zk.x + zk.y, zk.x - zk.y};
        } else {
          const T h = (T)0.5;
          const cpx<T> e{h * (zk.x + zm.x), h * (zk.y - zm.y)}, o{h * (zk.y + zm.y), h * (zm.x - zk.x)};
          const cpx<T> w = cmul(roots[q], o);
          row[q] = e + w;
          if (2 * q != C::M) row[C::M - q] = conj(e - w);
        }
      }
    }
  }
  __syncthreads();

#pragma nounroll
  for (int c0 = wave * CL; c0 < C::M; c0 += WAVES * CL) {
    forget();
    const int have = (C::M - c0 < CL ? C::M - c0 : CL);
    const bool on = lane < have * CC::TT;
    const int c = on ? c0 + lane / CC::TT : c0;
    cpx<T>* col = lds + c;
    cpx<T> v[CC::VMAX], kv[CC::VMAX];
    const cpx<T>* kc = k.k + (u32)ct * HalfKernel<C, T>::KP + (u32)c;  // the legs are constants apart
    for_layout<CC, pl_last<CF>::type::R>(0, [&](auto slot, u32 n) {
      if (CC::N / pl_last<CF>::type::R % CC::TT == 0 || n + (u32)ct < (u32)CC::N) {
        const cpx<T> z = kc[n * HalfKernel<C, T>::KP];
        kv[decltype(slot)::value] = C::CONJ ? conj(z) : z;
      }
    });
    if (on) line_get<CC, C::RP, pl_first<CF>::type::R>(col, v, ct);
    line_passes<CC, C::RP, -1, T>(CF{}, v, col, ct, col_fwd, on);
    if (c0 == 0) {  // column 0: both of its spectra, with the mirrored values from LDS
      wave_sync();
      if (on && c == 0)
        for_layout<CC, pl_last<CF>::type::R>(ct, [&](auto slot, u32 n) { col[n * C::RP] = v[decltype(slot)::value]; });
      wave_sync();
#pragma nounroll
      for (int n = lane; n <= C::N / 2; n += 64) {
        const int m = n == 0 ? 0 : C::N - n;
        cpx<T> a, b, ka, kb;
        unpack_pair(lds[n * C::RP], lds[m * C::RP], a, b);
        k.both((u32)n, ka, kb);
        a = cmul(a, ka);
        b = cmul(b, kb);
        lds[m * C::RP] = pack_pair(conj(a), conj(b));
        lds[n * C::RP] = pack_pair(a, b);
      }
      wave_sync();
    }
    for_layout<CC, pl_last<CF>::type::R>(ct, [&](auto slot, u32) {
      v[decltype(slot)::value] = cmul(v[decltype(slot)::value], kv[decltype(slot)::value]);
    });
    if (c0 == 0 && on && c == 0)
      for_layout<CC, pl_last<CF>::type::R>(ct, [&](auto slot, u32 n) { v[decltype(slot)::value] = col[n * C::RP]; });
    forget();
    line_passes<CC, C::RP, 1, T>(CI{}, v, col, ct, col_inv, on);
    wave_sync();
    if (on) for_layout<CC, pl_last<CI>::type::R>(ct, [&](auto slot, u32 n) { col[n * C::RP] = v[decltype(slot)::value]; });
  }
  __syncthreads();

#pragma nounroll
  for (int y0 = wave * RL; y0 < C::N; y0 += WAVES * RL) {
    forget();
    cpx<T>* rows = lds + y0 * C::RP;
    const int have = (C::N - y0 < RL ? C::N - y0 : RL);
    const bool on = lane < have * RC::TT;
    cpx<T>* row = rows + lane / RC::TT * C::RP;
    cpx<T> v[RC::VMAX];
    if (on) {
      for (int q = rt; q < PAIRS; q += RC::TT) {
        const cpx<T> a = row[q], am = row[q == 0 ? 0 : C::M - q];
        if (q == 0) {
          row[0] = cpx<T>{a.x + a.y, a.x - a.y};
        } else {
          const cpx<T> e{a.x + am.x, a.y - am.y}, d{a.x - am.x, a.y + am.y};
          const cpx<T> o = cmul(d, conj(roots[q]));
          row[q] = e + mul_i(o);
          if (2 * q != C::M) row[C::M - q] = conj(e + mul_negi(o));
        }
      }
    }
    wave_sync();
    if (on) line_get<RC, 1, pl_first<RF>::type::R>(row, v, rt);
    line_passes<RC, 1, 1, T>(RF{}, v, row, rt, row_tw, on);
    wave_sync();
    if (on)
      for_layout<RC, pl_last<RF>::type::R>(rt, [&](auto slot, u32 n) { row[n] = v[decltype(slot)::value] * (T)C::SCALE; });
    wave_sync();
    cpx<T>* xr = x + y0 * (C::M + 1);
    row_points<C::M, IT>(lane, have, [&](auto, int y, int n) { xr[y * (C::M + 1) + n] = rows[y * C::RP + n]; });
  }
}

}  // namespace vkx
