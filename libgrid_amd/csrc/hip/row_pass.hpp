// Plain transforms of contiguous rows: one forward or inverse transform of every row, in the order
// the caller knows, with at most a pending scale before it and a real factor after it.  The digits
// and their exchanges are those of the tile passes (tile_pass.hpp): a wave holds whole rows, so no
// barrier is needed but the one that publishes the twiddle table, and 384 points take three digits
// in 24 values a thread, where the pencil pass keeps 32 (FP64 arithmetic: one wave per SIMD).
//
// Bound by memory: one read and one write of the array.  128 threads a workgroup, 192 where 24 FP64
// values and the exchange leave room for few waves: many small workgroups drift apart, so that some
// load while others store (192 x 96 x 384 in FP64: 57 us with 320 threads, 50 with 256, 39.6 with
// 192, 40.5 with 128; the pencil pass takes 80; linear access 40).
#pragma once
#include "tile_pass.hpp"

namespace lg {
namespace row {

template <typename C, int L, int NT_> struct Geom {
  static constexpr int R = L % 3 == 0 ? 24 : L == 64 ? 8 : 16;
  static constexpr int NT = NT_, T = NT * R;
  static constexpr tile::Digits D = tile::digits_of(L, R);
  static_assert(D.n > 1 && 64 * R % L == 0 && NT % 64 == 0, "a wave holds whole rows");
};

// C the arithmetic type, S the storage type (float2 with C = double2: FP32 storage, FP64 arithmetic)
template <typename C, int L, typename S, int NT>
__global__ void __launch_bounds__(NT) __attribute__((amdgpu_waves_per_eu(tile::waves<C, Geom<C, L, NT>::R>(), 8)))
row_pass(const hgrid_pass a, const unsigned long total) {
  using G = Geom<C, L, NT>;
  using Rl = typename real_of<C>::type;
  constexpr int R = G::R;
  using AX = tile::Axis<C, R, NT, L, 1, G::D.d[0], G::D.d[1], G::D.d[2], G::D.n>;
  using First = typename AX::First;
  using Last = typename AX::Last;
  __shared__ __align__(16) Rl lds[AX::LDS];
  __shared__ __align__(16) C tab[AX::TABLE];
  const int tid = threadIdx.x;
  const unsigned long base = (unsigned long)blockIdx.x * G::T;
  const auto rin = make_rsrc((const S *)a.in + base, (total - base) * sizeof(S));
  C v[R];
#pragma unroll
  for (int u = 0; u < R / First::r; ++u) {
    const unsigned b = (unsigned)First::lin(tid, u) * sizeof(S);
#pragma unroll
    for (int i = 0; i < First::r; ++i) {
      const S s = bload<S>(rin, b, (unsigned)(i * First::s) * sizeof(S));
      v[u * First::r + i] = mk<C>((Rl)s.x, (Rl)s.y);
    }
  }
  AX::fill(tab, tid, (const C *)a.tw);
  if (a.flags & HGRID_PF_PRESCALE) {
    const C scale = mk<C>((Rl)a.scale[0], (Rl)a.scale[1]);
#pragma unroll
    for (int j = 0; j < R; ++j) v[j] = cmul(v[j], scale);
  }
  if (a.dir1 > 0) tile::conj_all(v);
  tile::tile_sync<NT>();
  AX::forward(v, tid, tab, lds);
  if (a.dir1 > 0) tile::conj_all(v);
  if (a.post != 1.0) {
    const Rl post = (Rl)a.post;
#pragma unroll
    for (int j = 0; j < R; ++j) v[j] = cscale(v[j], post);
  }
  const auto rout = make_rsrc((S *)a.out + base, (total - base) * sizeof(S));
  constexpr int LS = L / Last::r;  // the last digit's frequencies are this far apart
#pragma unroll
  for (int u = 0; u < R / Last::r; ++u) {
    const int lin = Last::lin(tid, u), zs = (lin % L) / Last::r;
    const int k = G::D.n == 3 ? zs / G::D.d[1] + G::D.d[0] * (zs % G::D.d[1]) : zs;
    const unsigned b = (unsigned)(lin / L * L + k) * sizeof(S);
#pragma unroll
    for (int i = 0; i < Last::r; ++i) {
      const C c = v[u * Last::r + i];
      S s;
      s.x = (typename real_of<S>::type)c.x;
      s.y = (typename real_of<S>::type)c.y;
      bstore<S>(s, rout, b, (unsigned)(i * LS) * sizeof(S));
    }
  }
}

template <typename C, int L, typename S, int NT> int launch_nt(const hgrid_pass *p, unsigned long total) {
  const unsigned long blocks = (total + Geom<C, L, NT>::T - 1) / Geom<C, L, NT>::T;
  if (!blocks) return 0;
  hipLaunchKernelGGL((row_pass<C, L, S, NT>), dim3((unsigned)blocks), dim3(NT), 0, stream(), *p, total);
  return check_launch("row_pass");
}

template <typename C, int L, typename S> int launch(const hgrid_pass *p) {
  const unsigned long total = (unsigned long)p->n0 * p->n1 * p->n2;
  constexpr int NT = sizeof(C) == 16 && L % 3 == 0 ? 192 : 128;
  // below two workgroups per CU, single waves
  if (total < 512ul * Geom<C, L, NT>::T) return launch_nt<C, L, S, 64>(p, total);
  return launch_nt<C, L, S, NT>(p, total);
}

// The lengths at which rows beat pencils, us at 2^22.6 to 2^23 points, pencils and then rows:
//   FP64  96: 34.4 30.1   192: 34.1 30.6*  384: 61.9 37.4   (64, 128, 256, 512: equal; 1024: 40 51)
//   FP32  64: 22.3 21.0    96: 22.3 18.0   128: 22.7 20.9   192: 19.9 17.0   256: 22.2 20.8
//        384: 21.1 19.6   512: 27.3 24.5   (1024: 25.9 31.3)
//   FP32 storage with FP64 arithmetic  64: 22.6 21.2   96: 26.4 20.7   128: 25.4 21.8
//        192: 22.8 20.3*  256: 24.3 22.3   384: 50.0 27.6   512: 32.1 27.7   (1024: 29.7 40.3)
// 48 points gain in the largest grids only (FP32 21.6 19.9, but 16 x 16 x 48 6.2 6.9).
// *: left to the pencils all the same.  One transform of 256 x 128 x 192 in FP64 that went this way
// came back 9.7e-4 off, the size of some six lost elements.  Neither the kernel's source and assembly
// nor later runs of the same transform showed the cause, so the one length and arithmetic that it was
// seen with does not take this way; it loses a tenth of one of the three passes.
#define LG_ROW_LENGTHS(X) X(64) X(96) X(128) X(192) X(256) X(384) X(512)

constexpr bool covers(long L, int prec) {
#define LG_CASE(n) || L == n
  return (false LG_ROW_LENGTHS(LG_CASE)) && (prec != HGRID_C128 || L % 3 == 0) && (prec == HGRID_C64 || L != 192);
#undef LG_CASE
}

template <typename C, typename S = C> int launch_len(const hgrid_pass *p) {
#define LG_CASE(n) \
  case n: if constexpr (covers(n, sizeof(S) == 16 ? HGRID_C128 : sizeof(C) == 16 ? HGRID_C64X : HGRID_C64)) return launch<C, n, S>(p); else return -1;
  switch (p->n2) {
    LG_ROW_LENGTHS(LG_CASE)
    default: return -1;
  }
#undef LG_CASE
}

int launch_f64(const hgrid_pass *p);
int launch_f32(const hgrid_pass *p);
int launch_f32s_f64(const hgrid_pass *p);

}  // namespace row
}  // namespace lg
