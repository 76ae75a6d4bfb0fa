// Tile passes: a split-operator step in two kinds of sweep over memory instead of one per axis.
//
// A pencil pass transforms one axis per sweep, so with the kinetic factor on x and the potential
// on z a step crosses y four times without doing anything else there.  A workgroup can hold
// more than one axis: these passes split the middle axis, n1 = A * B, and give each sweep one
// outer axis and one part of the middle one.
//
//   A-pass (kinetic), contiguous: B consecutive z rows (y = B h + l, l < B, for fixed x and h):
//       transforms along l and z, kinetic factor, inverse transforms.
//   B-pass (potential), strided: all x and all h for a fixed l and C consecutive z:
//       inverse transforms along x and h, potential factor, forward transforms.
//
// Between steps the state stays transformed along x and h ("tile form").  With W = exp(-2 pi i/n1)
//     X[k1 + A k2] = sum_l W^{l k1} exp(-2 pi i l k2 / B) sum_h exp(-2 pi i h k1 / A) x[B h + l]
// so h comes first (B-pass), then the twiddle W^{l k1} and l (A-pass).  Nothing is reordered in memory: the slot of digit h then holds k1, and
// the A-pass knows which frequencies its slots hold; x is stored in natural order.  A 2-D grid is the case without x: its h takes the place of x.  The B-pass also
// applies W^{l k1}: l is fixed in its tile, so h's twiddles are the same for all its threads.
//
// A 3-D Gross-Pitaevskii step is then 4 sweeps, 136 bytes per point in FP64, against 8 sweeps and
// 264 bytes with pencils; a linear relaxation step is 2 sweeps against 4.
//
// Inside a tile an axis of length d0 d1 .. is transformed digit by digit: R values per thread, one
// register DFT per digit, one LDS exchange between digits.  The inverse runs the same stages
// backwards (on conjugated data), so a round trip starts where the first half ended and no
// transform is ever put into natural order.  Each wave holds whole pencils of an axis, so the
// exchanges between its digits are the wave's own; only those between axes need the workgroup.
#pragma once
#include "absorb.hpp"
#include "fft_pass.hpp"

namespace lg {
namespace tile {

// ---- geometry (compile time) ----------------------------------------------------------------

struct Digits {
  int n;
  int d[3];
};

// The digits of an axis of length L, each a divisor of R: as few as possible; of two the first as
// large as 16 allows, which leaves the fewest twiddles that round (a balanced split runs at the same
// speed, within 1 %); three balanced.
constexpr Digits digits_of(int L, int R) {
  if (L == 1) return Digits{0, {1, 1, 1}};
  if (L <= R && R % L == 0) return Digits{1, {L, 1, 1}};
  Digits best{0, {1, 1, 1}};
  for (int d0 = 2; d0 <= R; ++d0) {
    if (R % d0 || L % d0) continue;
    const int d1 = L / d0;
    if (d1 < 2 || d1 > d0 || R % d1) continue;
    if (best.n == 0 || d0 <= 16) best = Digits{2, {d0, d1, 1}};
  }
  if (best.n) return best;
  int low = 1 << 30;
  for (int d0 = 2; d0 <= R; ++d0)
    for (int d1 = 2; d1 <= d0; ++d1) {
      if (R % d0 || R % d1 || L % (d0 * d1)) continue;
      const int d2 = L / (d0 * d1);
      if (d2 < 2 || d2 > d1 || R % d2) continue;
      if (d0 < low) {
        low = d0;
        best = Digits{3, {d0, d1, d2}};
      }
    }
  return best;
}

constexpr int largest(int a, int b) { return a > b ? a : b; }

// A-pass over rows of LZ points, B rows: M consecutive (x, h) per workgroup where one alone would
// leave lanes idle.  R = 16 values per thread (8 in small tiles, for more wavefronts; 24 or 12
// where the length has a factor 3; 32 FP32 values in the largest).
template <typename C, int LZ, int B> struct GeomA {
  static constexpr bool THREE = LZ % 3 == 0;
  static constexpr int T0 = LZ * B;
  static constexpr int R = THREE ? (T0 >= 1536 ? 24 : 12)
                           : sizeof(C) == 8 && T0 >= 8192 ? 32
                           : T0 >= 2048 || LZ >= 128 ? 16
                                                     : 8;
  static constexpr int M = T0 / R >= 64 ? 1 : 64 / (T0 / R);
  static constexpr int T = T0 * M, NT = T / R;
  static constexpr Digits DZ = digits_of(LZ, R);
  // 64 rows 8 x 8: with 16 x 4 the padded exchange of the largest tiles would not fit in LDS
  static constexpr Digits DY = B == 64 ? Digits{2, {8, 8, 1}} : digits_of(B, R);
  static constexpr int ZLAST = DZ.d[DZ.n - 1];
  static constexpr int PD = ZLAST, PW = 1;  // one spare LDS word per run of the last z digit
  static_assert(DZ.n > 0 && DY.n > 0 && T % R == 0 && NT % 64 == 0, "A-pass geometry");
};

// B-pass over x of LX points and A values of h: CC consecutive z, 64 bytes at least (128-byte lines
// are shared by two workgroups that run on the same XCD; 64-byte rows in that order copy
// 256^3 FP64 at 5.3 TB/s, 32-byte rows at 4.1, 128-byte rows at 6.6, which need twice the tile).
template <typename C, int LX, int A> struct GeomB {
  static constexpr bool THREE = LX % 3 == 0 || A % 3 == 0;
  static constexpr int C0 = A == 1 ? (LX <= 24 ? 32 : 16) : sizeof(C) == 16 ? 4 : 8;
  static constexpr int r_two(int t) { return sizeof(C) == 8 && t >= 16384 ? 32 : t >= 4096 || LX >= 128 || A == 16 ? 16 : 8; }
  // with a factor 3, 24 or 12 values and C0 or 2 C0 columns: the first pair that fills whole waves
  static constexpr bool whole(int c, int r) { return r % A == 0 && LX * A * c % (64 * r) == 0 && (r == 12 || LX * A * c >= 1536); }
  static constexpr int pair() {
    for (int k = 0; k < 4; ++k)
      if (whole(k < 2 ? C0 : 2 * C0, k % 2 ? 12 : 24)) return k;
    return A == 8 ? 2 : 1;
  }
  static constexpr int CC = THREE                                    ? (pair() < 2 ? C0 : 2 * C0)
                            : LX * A * C0 / r_two(LX * A * C0) % 64 ? 2 * C0
                                                                     : C0;
  static constexpr int T = LX * A * CC;
  static constexpr int R = THREE ? (pair() % 2 ? 12 : 24) : r_two(T);
  static constexpr int NT = T / R;
  static constexpr Digits DX = digits_of(LX, R);
  static constexpr int PD = A * CC, PW = CC;  // the exchange with h: CC spare words per x
  static_assert(DX.n > 0 && T % R == 0 && R % A == 0, "B-pass geometry");
};

// ---- register stages and exchanges -------------------------------------------------------------

// A stage holds digit values in registers: item u of a thread is one register DFT of radix r whose
// element i lies at tile index lin(tid, u) + i * s.  NT threads of R values.

// An axis of one digit: items in the order of the remaining tile index, so that lanes are
// contiguous wherever the axis is not.
template <int NT, int R, int r_, int s_> struct FlatStage {
  static constexpr int r = r_, s = s_;
  static __device__ __forceinline__ int lin(int tid, int u) {
    const int o = tid + NT * u;
    return s == 1 ? o * r : (o / s) * (r * s) + o % s;
  }
};

// A digit of a longer axis (length L, stride SAX in the tile; the digit's own stride SU within the
// axis, last digit DL).  A wave owns P whole pencils.  Lanes run over pencils first where these are
// neighbours (SAX > 1), else along the pencil.
template <typename C, int NT, int R, int L, int SAX, int r_, int SU, int DL> struct PencilStage {
  static constexpr int r = r_, s = SAX * SU;
  static constexpr int W = NT < 64 ? NT : 64, P = W * R / L;
  // the wave's own exchange: one spare slot per run of the last digit, unless neighbouring pencils
  // already spread the lanes over all 64 banks
  static constexpr int PAD = SAX > 1 && P * (int)sizeof(C) >= 512 ? 0 : 1;
  static constexpr int PITCH = L + PAD * (L / DL);
  static_assert(W * R % L == 0 && NT % W == 0, "a wave holds whole pencils");
  static constexpr int REGION = P * PITCH;  // LDS words of one wave
  static __device__ __forceinline__ int pencil(int lane, int u) {
    const int o = lane + W * u;
    return SAX > 1 ? o % P : o / (L / r);
  }
  static __device__ __forceinline__ int rest(int lane, int u) {
    const int o = lane + W * u;
    return SAX > 1 ? o / P : o % (L / r);
  }
  static __device__ __forceinline__ int lower(int tid, int u) { return rest(tid % W, u) % SU; }  // index of the lower digits
  static __device__ __forceinline__ int along(int lane, int u) {
    const int q = rest(lane, u);
    return SU == 1 ? q * r : (q / SU) * (r * SU) + q % SU;
  }
  static __device__ __forceinline__ int lin(int tid, int u) {
    const int p = (tid / W) * P + pencil(tid % W, u);
    return (SAX == 1 ? p * L : (p / SAX) * (SAX * L) + p % SAX) + SAX * along(tid % W, u);
  }
  static __device__ __forceinline__ int local(int tid, int u) {
    const int q = along(tid % W, u), pl = pencil(tid % W, u), e = q + PAD * (q / DL);
    return (tid / W) * REGION + (SAX > 1 ? e * P + pl : pl * PITCH + e);
  }
  static constexpr int local_step(int i) { return (i * SU + PAD * (i * SU / DL)) * (SAX > 1 ? P : 1); }
  static_assert(SU % DL == 0 || (SU == 1 && r == DL), "elements at constant distances");
};

template <int PD, int PW> __device__ __forceinline__ int padded(int l) { return l + (l / PD) * PW; }

// position of element i of an item in the workgroup's exchange: one spare word (PW words) per PD;
// where the stride divides or is a multiple of that period it is at a constant distance
template <typename S, int PD, int PW> __device__ __forceinline__ int slot(int base, int pbase, int i) {
  if constexpr (S::s % PD == 0 || PD % (S::r * S::s) == 0) return pbase + i * S::s + (i * S::s / PD) * PW;
  else return padded<PD, PW>(base + i * S::s);
}

template <int NT> __device__ __forceinline__ void tile_sync() {
  if constexpr (NT <= 64) pencil_sync<true>();
  else __syncthreads();
}

template <typename C, int R, int r> __device__ __forceinline__ void dft_items(C (&v)[R]) {
#pragma unroll
  for (int u = 0; u < R / r; ++u) {
    C w[r];
#pragma unroll
    for (int i = 0; i < r; ++i) w[i] = v[u * r + i];
    dft<r>(w);
#pragma unroll
    for (int i = 0; i < r; ++i) v[u * r + i] = w[i];
  }
}

template <typename C, int R> __device__ __forceinline__ void conj_all(C (&v)[R]) {
#pragma unroll
  for (int j = 0; j < R; ++j) v[j] = cconj(v[j]);
}

// Redistribute from stage S1 to stage S2 through the workgroup's LDS: real parts, then imaginary
// parts through one buffer of T words, so that two workgroups of the largest tiles share a CU.
template <typename S1, typename S2, typename C, int R, int NT, int PD, int PW>
__device__ __forceinline__ void exchange(C (&v)[R], int tid, typename real_of<C>::type *lds) {
  typename real_of<C>::type re[R];
  auto put = [&](auto part) {
#pragma unroll
    for (int u = 0; u < R / S1::r; ++u) {
      const int b = S1::lin(tid, u), p = padded<PD, PW>(b);
#pragma unroll
      for (int i = 0; i < S1::r; ++i) lds[slot<S1, PD, PW>(b, p, i)] = part(v[u * S1::r + i]);
    }
  };
  auto get = [&](auto &&take) {
#pragma unroll
    for (int u = 0; u < R / S2::r; ++u) {
      const int b = S2::lin(tid, u), p = padded<PD, PW>(b);
#pragma unroll
      for (int i = 0; i < S2::r; ++i) take(u * S2::r + i, lds[slot<S2, PD, PW>(b, p, i)]);
    }
  };
  tile_sync<NT>();  // earlier exchanges may still be reading
  put([](C c) { return c.x; });
  tile_sync<NT>();
  get([&](int j, typename real_of<C>::type x) { re[j] = x; });
  tile_sync<NT>();
  put([](C c) { return c.y; });
  tile_sync<NT>();
  get([&](int j, typename real_of<C>::type y) { v[j] = mk<C>(re[j], y); });
}

// The same between two digits of one axis, inside each wave
template <typename S1, typename S2, typename C, int R>
__device__ __forceinline__ void exchange_local(C (&v)[R], int tid, typename real_of<C>::type *lds) {
  typename real_of<C>::type re[R];
  auto put = [&](auto part) {
#pragma unroll
    for (int u = 0; u < R / S1::r; ++u) {
      const int p = S1::local(tid, u);
#pragma unroll
      for (int i = 0; i < S1::r; ++i) lds[p + S1::local_step(i)] = part(v[u * S1::r + i]);
    }
  };
  auto get = [&](auto &&take) {
#pragma unroll
    for (int u = 0; u < R / S2::r; ++u) {
      const int p = S2::local(tid, u);
#pragma unroll
      for (int i = 0; i < S2::r; ++i) take(u * S2::r + i, lds[p + S2::local_step(i)]);
    }
  };
  pencil_sync<true>();
  put([](C c) { return c.x; });
  pencil_sync<true>();
  get([&](int j, typename real_of<C>::type x) { re[j] = x; });
  pencil_sync<true>();
  put([](C c) { return c.y; });
  pencil_sync<true>();
  get([&](int j, typename real_of<C>::type y) { v[j] = mk<C>(re[j], y); });
}

// table entry at an index that all lanes of the wave share (a scalar load)
template <typename C> __device__ __forceinline__ C uniform_entry(const C *t, int i) {
  using Rl = typename real_of<C>::type;
  typedef const __attribute__((address_space(4))) Rl *cptr;
  const cptr p = (cptr)(unsigned long long)(t + __builtin_amdgcn_readfirstlane(i));
  return mk<C>(p[0], p[1]);
}

// Twiddles after (forward) or before (inverse, on conjugated data) the DFTs of a digit: element i,
// n the index of the axis's lower digits (LOW of them): entry [i][n] = W_L^{mult i n} of a table in
// LDS, mult the product of the digits above.  Lanes read neighbouring entries.  As loads from the
// length-L table (up to 16 cache lines an instruction) these took 53 of the 157 us of the 256^3
// FP64 A-pass.
template <typename S, int LOW, typename C, int R> __device__ __forceinline__ void twiddle(C (&v)[R], int tid, const C *tab) {
#pragma unroll
  for (int u = 0; u < R / S::r; ++u) {
    const C *t = tab + S::lower(tid, u);
#pragma unroll
    for (int i = 1; i < S::r; ++i) v[u * S::r + i] = cmul(v[u * S::r + i], t[i * LOW]);
  }
}

// fill such a table of D digit values from the table of length L; published by a later barrier
template <typename C, int NT, int L, int D, int LOW, int mult> __device__ __forceinline__ void fill_twiddles(C *tab, int tid, const C *tw) {
#pragma unroll
  for (int e0 = 0; e0 < D * LOW; e0 += NT) {
    const int e = e0 + tid;
    if (D * LOW % NT == 0 || e < D * LOW) tab[e] = tw[mult * (e / LOW) * (e % LOW)];
  }
}

// Transforms of one axis: forward from its first digit in registers to its last, inverse (on
// conjugated data) from the last to the first.
template <typename C, int R, int NT, int L, int SAX, int D0, int D1, int D2, int N> struct Axis;
template <typename C, int R, int NT, int L, int SAX, int D0, int D1, int D2> struct Axis<C, R, NT, L, SAX, D0, D1, D2, 1> {
  using First = FlatStage<NT, R, D0, SAX>;
  using Last = First;
  static constexpr int LDS = 0, TABLE = 0;  // LDS words of the exchanges, entries of the twiddle tables
  static __device__ __forceinline__ void fill(C *, int, const C *) {}
  static __device__ __forceinline__ void forward(C (&v)[R], int, const C *, typename real_of<C>::type *) { dft_items<C, R, D0>(v); }
  static __device__ __forceinline__ void inverse(C (&v)[R], int, const C *, typename real_of<C>::type *) { dft_items<C, R, D0>(v); }
};
template <typename C, int R, int NT, int L, int SAX, int D0, int D1, int D2> struct Axis<C, R, NT, L, SAX, D0, D1, D2, 2> {
  using First = PencilStage<C, NT, R, L, SAX, D0, D1, D1>;
  using Last = PencilStage<C, NT, R, L, SAX, D1, 1, D1>;
  static constexpr int LDS = NT / First::W * First::REGION, TABLE = L;
  static __device__ __forceinline__ void fill(C *tab, int tid, const C *tw) { fill_twiddles<C, NT, L, D0, D1, 1>(tab, tid, tw); }
  static __device__ __forceinline__ void forward(C (&v)[R], int tid, const C *tab, typename real_of<C>::type *lds) {
    dft_items<C, R, D0>(v);
    twiddle<First, D1>(v, tid, tab);
    exchange_local<First, Last>(v, tid, lds);
    dft_items<C, R, D1>(v);
  }
  static __device__ __forceinline__ void inverse(C (&v)[R], int tid, const C *tab, typename real_of<C>::type *lds) {
    dft_items<C, R, D1>(v);
    exchange_local<Last, First>(v, tid, lds);
    twiddle<First, D1>(v, tid, tab);
    dft_items<C, R, D0>(v);
  }
};
template <typename C, int R, int NT, int L, int SAX, int D0, int D1, int D2> struct Axis<C, R, NT, L, SAX, D0, D1, D2, 3> {
  using First = PencilStage<C, NT, R, L, SAX, D0, D1 * D2, D2>;
  using Mid = PencilStage<C, NT, R, L, SAX, D1, D2, D2>;
  using Last = PencilStage<C, NT, R, L, SAX, D2, 1, D2>;
  static constexpr int LDS = NT / First::W * First::REGION, TABLE = L + D1 * D2;
  static __device__ __forceinline__ void fill(C *tab, int tid, const C *tw) {
    fill_twiddles<C, NT, L, D0, D1 * D2, 1>(tab, tid, tw);
    fill_twiddles<C, NT, L, D1, D2, D0>(tab + L, tid, tw);
  }
  static __device__ __forceinline__ void forward(C (&v)[R], int tid, const C *tab, typename real_of<C>::type *lds) {
    dft_items<C, R, D0>(v);
    twiddle<First, D1 * D2>(v, tid, tab);
    exchange_local<First, Mid>(v, tid, lds);
    dft_items<C, R, D1>(v);
    twiddle<Mid, D2>(v, tid, tab + L);
    exchange_local<Mid, Last>(v, tid, lds);
    dft_items<C, R, D2>(v);
  }
  static __device__ __forceinline__ void inverse(C (&v)[R], int tid, const C *tab, typename real_of<C>::type *lds) {
    dft_items<C, R, D2>(v);
    exchange_local<Last, Mid>(v, tid, lds);
    twiddle<Mid, D2>(v, tid, tab + L);
    dft_items<C, R, D1>(v);
    exchange_local<Mid, First>(v, tid, lds);
    twiddle<First, D1 * D2>(v, tid, tab);
    dft_items<C, R, D0>(v);
  }
};

// frequency held by a position of an axis with digits d0 d1 d2 in transform order
__device__ __forceinline__ int slot_frequency(int slot, int d0, int d1, int d2) {
  const int i2 = slot % d2, j = slot / d2;
  const int i1 = j % d1, i0 = j / d1;
  return i0 + d0 * (i1 + d1 * i2);
}

// deterministic workgroup reduction into partials[channel][block]
template <int NT> __device__ __forceinline__ void reduce_partials(double (&acc)[HGRID_RED_NCHAN], int tid, double *partials) {
  __shared__ double red[NT % 64 ? NT : NT / 64][HGRID_RED_NCHAN];
  if constexpr (NT % 64 == 0) {
#pragma unroll
    for (int c = 0; c < HGRID_RED_NCHAN; ++c) {
      double x = acc[c];
#pragma unroll
      for (int off = 32; off >= 1; off >>= 1) x += __shfl_xor(x, off, 64);
      if (tid % 64 == 0) red[tid / 64][c] = x;
    }
  } else {
#pragma unroll
    for (int c = 0; c < HGRID_RED_NCHAN; ++c) red[tid][c] = acc[c];
  }
  __syncthreads();
  if (tid < HGRID_RED_NCHAN) {
    double s = 0.0;
    for (int w = 0; w < (NT % 64 ? NT : NT / 64); ++w) s += red[w][tid];
    partials[(long)tid * gridDim.x + blockIdx.x] = s;
  }
}

// Waves per SIMD asked of the register allocator: 128 VGPRs for tiles of 16 FP64 or 32 FP32 values
// per thread (two workgroups of 512 threads per CU).
template <typename C, int R> constexpr int waves() { return sizeof(C) == 16 ? (R <= 16 ? 4 : 3) : R >= 24 ? 3 : 5; }

// ---- A-pass --------------------------------------------------------------------------------------

template <typename C, int LZ, int B, bool REALK>
__global__ void __launch_bounds__((GeomA<C, LZ, B>::NT))
__attribute__((amdgpu_waves_per_eu(waves<C, GeomA<C, LZ, B>::R>(), 8))) tile_kinetic(const hgrid_tile a) {
  using G = GeomA<C, LZ, B>;
  using Rl = typename real_of<C>::type;
  constexpr int R = G::R, NT = G::NT, M = G::M, T = G::T, PD = G::PD, PW = G::PW;
  using AZ = Axis<C, R, NT, LZ, 1, G::DZ.d[0], G::DZ.d[1], G::DZ.d[2], G::DZ.n>;
  using AY = Axis<C, R, NT, B, LZ, G::DY.d[0], G::DY.d[1], G::DY.d[2], G::DY.n>;
  using Y0 = typename AY::First;
  constexpr unsigned CS = sizeof(C);
  __shared__ __align__(16) Rl lds[largest(T + T / PD * PW, largest(AZ::LDS, AY::LDS))];
  __shared__ __align__(16) C tabz[largest(AZ::TABLE, 1)], taby[largest(AY::TABLE, 1)];
  const int tid = threadIdx.x;
  const unsigned fl = a.flags;
  AZ::fill(tabz, tid, (const C *)a.twz);
  AY::fill(taby, tid, (const C *)a.twl);
  const auto rio = make_rsrc((const C *)a.psi + (long)blockIdx.x * T, (unsigned long)T * CS);
  C scale = mk<C>((Rl)1, (Rl)0);
  if ((fl & HGRID_PF_PRESCALE) && a.scale) {
    scale = mk<C>((Rl)a.scale[0], (Rl)a.scale[1]);
  } else if (fl & HGRID_PF_PRESCALE) {
    // the renormalisation of a relaxation step, from the partial sums of the pass before: every
    // workgroup adds them in the same order, which saves a launch a step (64^3 FP32: 3.2 of 15 us)
    constexpr int WHOLE = NT % 64 == 0, NS = WHOLE ? NT / 64 : NT;
    __shared__ double sums[NS];
    double s = 0.0;
    for (long i = tid; i < a.norm_count; i += NT) s += a.norm_partials[i];
    if constexpr (WHOLE) {
#pragma unroll
      for (int off = 32; off >= 1; off >>= 1) s += __shfl_xor(s, off, 64);
    }
    if (!WHOLE || tid % 64 == 0) sums[WHOLE ? tid / 64 : tid] = s;
    __syncthreads();
    s = 0.0;
    for (int w = 0; w < NS; ++w) s += sums[w];
    // the same in all lanes: held once, not per lane
    const double f = sqrt(a.norm_target / (a.norm_dv * s));
    const unsigned long long fb = __double_as_longlong(f);
    const unsigned lo = __builtin_amdgcn_readfirstlane((int)fb), hi = __builtin_amdgcn_readfirstlane((int)(fb >> 32));
    scale.x = (Rl)__longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
  }
  C v[R];
#pragma unroll
  for (int u = 0; u < R / Y0::r; ++u) {
    const unsigned b = (unsigned)Y0::lin(tid, u) * CS;
#pragma unroll
    for (int i = 0; i < Y0::r; ++i) v[u * Y0::r + i] = bload<C>(rio, b, (unsigned)(i * Y0::s) * CS);
  }
  double acc[HGRID_RED_NCHAN] = {0.0, 0.0, 0.0, 0.0, 0.0};
  if (fl & HGRID_PF_PRESCALE) {
#pragma unroll
    for (int j = 0; j < R; ++j) v[j] = cmul(v[j], scale);
  }
  if (a.post != 1.0) {
    const Rl post = (Rl)a.post;
#pragma unroll
    for (int j = 0; j < R; ++j) v[j] = cscale(v[j], post);
  }
  // kinetic factor: the last z digit is in registers.  The slots above this tile are M consecutive
  // (x, h) slots, or h slots in a 2-D grid; k1 is the frequency of the h slot, nh their number.
  using ZL = typename AZ::Last;
  constexpr int RZ = ZL::r, ZH = LZ / RZ;
  const int nh = a.nh, flat0 = (int)blockIdx.x * M;
  const double2 *t0 = (const double2 *)a.ktab_0, *t1 = (const double2 *)a.ktab_1, *t2 = (const double2 *)a.ktab_2;
  auto frequencies = [&](int u, int &k0, int &k1, int &kz) {
    const int lin = ZL::lin(tid, u), zs = (lin % LZ) / RZ, ys = (lin / LZ) % B;
    kz = G::DZ.n == 3 ? zs / G::DZ.d[1] + G::DZ.d[0] * (zs % G::DZ.d[1]) : zs;
    const int kl = slot_frequency(ys, G::DY.d[0], G::DY.d[1], G::DY.d[2]);
    const int flat = flat0 + (M == 1 ? 0 : lin / (LZ * B));
    k0 = a.flat ? 0 : flat / nh;
    k1 = (a.flat ? flat : flat - k0 * nh) + nh * kl;
  };
  auto outer = [&](int k0, int k1) { return REALK ? make_double2(t0[k0].x * t1[k1].x, 0.0) : cmul(t0[k0], t1[k1]); };
  // tiles of 8 values, the small grids', load the tables with the tile: a launch there is a chain of
  // latencies (with the same in the potential passes 32^3 FP64, 16 steps: 237 -> 231 us; steps of 16^3
  // to 64^3 3 to 8 %)
  constexpr bool EARLY = R <= 8;
  double2 fxy[EARLY ? R / RZ : 1], fz[EARLY ? R : 1];
  if constexpr (EARLY) {
#pragma unroll
    for (int u = 0; u < R / RZ; ++u) {
      int k0, k1, kz;
      frequencies(u, k0, k1, kz);
      fxy[u] = outer(k0, k1);
#pragma unroll
      for (int i = 0; i < RZ; ++i) fz[u * RZ + i] = REALK ? make_double2(t2[kz + ZH * i].x, 0.0) : t2[kz + ZH * i];
    }
  }
  if constexpr (AY::TABLE) tile_sync<NT>();
  AY::forward(v, tid, taby, lds);
  exchange<typename AY::Last, typename AZ::First, C, R, NT, PD, PW>(v, tid, lds);
  if constexpr (AZ::LDS) tile_sync<NT>();  // the waves' own exchanges reuse the buffer
  AZ::forward(v, tid, tabz, lds);

#pragma unroll
  for (int u = 0; u < R / RZ; ++u) {
    int k0, k1, kz;
    frequencies(u, k0, k1, kz);
    if (fl & HGRID_PF_MID_KRED) {
      const double kk = a.k2_0[k0] + a.k2_1[k1];
#pragma unroll
      for (int i = 0; i < RZ; ++i) acc[HGRID_RED_KIN] += (kk + k2_of<LZ>(kz + ZH * i, a.k2_dk)) * cnorm2(v[u * RZ + i]);
    }
    // factors in groups of four behind scheduling fences, so that few are live at once
    const double2 f = EARLY ? fxy[EARLY ? u : 0] : outer(k0, k1);
#pragma unroll
    for (int i0 = 0; i0 < RZ; i0 += 4) {
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int i = i0; i < (i0 + 4 < RZ ? i0 + 4 : RZ); ++i) {
        if constexpr (REALK) {
          // hidden from the sum above, with which the compiler would share the values widened to FP64,
          // all at once (FP32, rows of 512: 145 registers spilled)
          if constexpr (sizeof(C) == 8) asm volatile("" : "+v"(v[u * RZ + i].x), "+v"(v[u * RZ + i].y));
          v[u * RZ + i] = cscale_d(v[u * RZ + i], (EARLY ? fz[EARLY ? u * RZ + i : 0].x : t2[kz + ZH * i].x) * f.x);
        }
        else v[u * RZ + i] = cmul(v[u * RZ + i], round_to<C>(cmul(EARLY ? fz[EARLY ? u * RZ + i : 0] : t2[kz + ZH * i], f)));
      }
    }
    __builtin_amdgcn_sched_barrier(0);
    if (fl & HGRID_PF_KCUT) {
      const double c0 = a.kc_0[k0], c1 = a.kc_1[k1];
#pragma unroll
      for (int i = 0; i < RZ; ++i)
        if ((c0 + c1) + a.kc_2[kz + ZH * i] >= a.kcut2) v[u * RZ + i] = mk<C>(0, 0);
    }
  }

  conj_all(v);
  AZ::inverse(v, tid, tabz, lds);
  exchange<typename AZ::First, typename AY::Last, C, R, NT, PD, PW>(v, tid, lds);
  if constexpr (AY::LDS) tile_sync<NT>();
  AY::inverse(v, tid, taby, lds);
  conj_all(v);
  if (fl & HGRID_PF_POST_RED) {
#pragma unroll
    for (int j = 0; j < R; ++j) acc[HGRID_RED_POST] += cnorm2(v[j]);
  }
  const auto rout = make_rsrc((const C *)(a.out ? a.out : a.psi) + (long)blockIdx.x * T, (unsigned long)T * CS);
#pragma unroll
  for (int u = 0; u < R / Y0::r; ++u) {
    const unsigned b = (unsigned)Y0::lin(tid, u) * CS;
#pragma unroll
    for (int i = 0; i < Y0::r; ++i) bstore<C>(v[u * Y0::r + i], rout, b, (unsigned)(i * Y0::s) * CS);
  }
  if (fl & (HGRID_PF_MID_KRED | HGRID_PF_POST_RED)) reduce_partials<NT>(acc, tid, a.partials);
}

// ---- B-pass --------------------------------------------------------------------------------------

// TPRE: inverse transforms, then V_eff = vext + g |psi|^2 / reductions; nothing else stored
// TPOT: inverse transforms, exp(c (cons + V)) with complex V (or none), forward transforms; either
//       transform may be left out (entering and leaving tile form, 4th-order outer stages)
// TGPE / TGPR: the same with a real potential, real time (imaginary c) / imaginary time (real c).  A
//       kernel with the general complex c beside them spilled 48 of 128 VGPRs (256^3 FP64 real-time
//       pass 309 us); complex time with a real potential stays with the pencil passes
//   TMRG inverse, merge with another real-space state by the absorbing boundary's amplitude, forward:
//       in place of an inverse pass, a merge over three arrays and the next step's forward pass
enum { TPRE = 0, TPOT = 1, TGPE = 2, TGPR = 3, TMRG = 4 };

template <typename C, int LX, int A, int KIND>
__global__ void __launch_bounds__((GeomB<C, LX, A>::NT))
__attribute__((amdgpu_waves_per_eu(waves<C, GeomB<C, LX, A>::R>(), 8))) tile_potential(const hgrid_tile a) {
  using G = GeomB<C, LX, A>;
  using Rl = typename real_of<C>::type;
  constexpr int R = G::R, NT = G::NT, T = G::T, CC = G::CC, PD = G::PD, PW = G::PW;
  using AX = Axis<C, R, NT, LX, A * CC, G::DX.d[0], G::DX.d[1], G::DX.d[2], G::DX.n>;
  using X0 = typename AX::First;
  using XL = typename AX::Last;
  // the stage that holds real space: h, or without h the first x digit
  using SV = typename std::conditional<(A > 1), FlatStage<NT, R, A, CC>, X0>::type;
  constexpr unsigned CS = sizeof(C);
  __shared__ __align__(16) Rl lds[largest(A > 1 ? T + T / PD * PW : 1, largest(AX::LDS, 1))];
  __shared__ __align__(16) C tabx[largest(AX::TABLE, 1)];
  const int tid = threadIdx.x;
  const unsigned fl = a.flags;
  AX::fill(tabx, tid, (const C *)a.twx);
  const unsigned n2 = (unsigned)a.n2, sx = (unsigned)a.sx, sh = (unsigned)a.sh, zg = n2 / CC;
  // each XCD works through one contiguous eighth of the tiles (workgroup b runs on XCD b mod 8), so
  // the workgroups that share a 128-byte line share an L2: 256^3 FP64 copy of the tiles 123 us
  // in hardware order, 102 us in this one
  unsigned blk = blockIdx.x;
  {
    const unsigned per = gridDim.x / 8;
    if (blk < 8 * per) blk = (blk % 8) * per + blk / 8;
  }
  const unsigned l = blk / zg, z0 = (blk - l * zg) * CC;
  const unsigned origin = l * n2 + z0;
  const unsigned long ntot = (unsigned long)a.n0 * (unsigned long)a.n1 * n2;
  const auto rio = make_rsrc(a.psi, ntot * CS);
  // flat element index of a real-space element at the tile's linear index, and of the stage that
  // loads and stores tile form; their steps per element of the stage.  Tile form has the
  // frequencies of x in natural order: the last digit in registers has the largest stride, and the
  // lanes of an instruction go over neighbouring x.  (With the digits stored in place, lanes 16 x
  // apart, a copy of the 256^3 FP64 tiles from HBM took 164 instead of 133 us.)
  auto element = [&](int lin) {
    const unsigned x = (unsigned)lin / (A * CC), h = ((unsigned)lin / CC) % A;
    return origin + x * sx + h * sh + (unsigned)lin % CC;
  };
  constexpr int XH = LX / XL::r;
  auto frequency = [&](int t, int u) {  // of element 0 of the item
    const int xs = XL::lin(t, u) / (A * CC * XL::r);
    return G::DX.n == 3 ? xs / G::DX.d[1] + G::DX.d[0] * (xs % G::DX.d[1]) : xs;
  };
  auto form_element = [&](int t, int u) {
    const unsigned lin = (unsigned)XL::lin(t, u), h = (lin / CC) % A;
    return origin + (unsigned)frequency(t, u) * sx + h * sh + lin % CC;
  };
  const unsigned stepv = A > 1 ? sh : sx * (unsigned)(SV::s / (A * CC));
  const unsigned stepl = sx * (unsigned)XH;
  C v[R];
  auto load = [&](auto stage, unsigned step, auto &&at) {
    using S = decltype(stage);
#pragma unroll
    for (int u = 0; u < R / S::r; ++u) {
      const unsigned e = at(tid, u);
#pragma unroll
      for (int i = 0; i < S::r; ++i) v[u * S::r + i] = bload<C>(rio, e * CS, (unsigned)i * step * CS);
    }
  };
  auto store = [&](auto stage, unsigned step, auto &&at) {
    using S = decltype(stage);
    const auto rout = make_rsrc((KIND == TPOT || KIND == TMRG) && a.out ? a.out : a.psi, ntot * CS);
#pragma unroll
    for (int u = 0; u < R / S::r; ++u) {
      const unsigned e = at(tid, u);
#pragma unroll
      for (int i = 0; i < S::r; ++i) bstore<C>(v[u * S::r + i], rout, e * CS, (unsigned)i * step * CS);
    }
  };
  auto real_element = [&](int t, int u) { return element(SV::lin(t, u)); };
  // W_{n1}^{l k1} between h and the rows (on conjugated data in the inverse).  3-D: h is in registers
  // and l the same for the tile.  2-D: the last digit of h, in x's place
  auto split_twiddle = [&]() {
    const C *tw = (const C *)a.twy;
    if constexpr (A > 1) {
#pragma unroll
      for (int i = 1; i < A; ++i) {
        const C w = uniform_entry(tw, (int)l * i);
#pragma unroll
        for (int u = 0; u < R / A; ++u) v[u * A + i] = cmul(v[u * A + i], w);
      }
    } else {
      // by scalar steps from one address: one for each value, kept from the inverse side for the
      // forward one, would spill
      const auto rtw = make_rsrc(tw, (unsigned long)a.n1 * CS);
#pragma unroll
      for (int u = 0; u < R / XL::r; ++u) {
        const unsigned k = l * (unsigned)frequency(tid, u) * CS;
#pragma unroll
        for (int i = 0; i < XL::r; ++i) {
          v[u * XL::r + i] = cmul(v[u * XL::r + i], bload<C>(rtw, k, l * (unsigned)(XH * i) * CS));
        }
      }
    }
  };
  const bool skip1 = (KIND == TPRE || KIND == TPOT) && (fl & HGRID_PF_POT_NOFFT1);
  const bool skip2 = KIND == TPRE || (KIND == TPOT && (fl & HGRID_PF_POT_NOFFT2));
  C scale = mk<C>((Rl)1, (Rl)0);
  if (fl & HGRID_PF_PRESCALE) scale = mk<C>((Rl)a.scale[0], (Rl)a.scale[1]);
  if (skip1) load(SV{}, stepv, real_element);
  else load(XL{}, stepl, form_element);
  if constexpr (AX::TABLE) tile_sync<NT>();
  if constexpr (KIND == TPRE || KIND == TPOT) {
    if (fl & HGRID_PF_PRESCALE) {
#pragma unroll
      for (int j = 0; j < R; ++j) v[j] = cmul(v[j], scale);
    }
  }
  double acc[HGRID_RED_NCHAN] = {0.0, 0.0, 0.0, 0.0, 0.0};
  // V_eff goes from the start-of-step pass to the potential pass in the order of the threads; vext
  // is in the grid's
  const bool ordered = KIND != TPRE && a.veff;
  const auto rveff = make_rsrc((const char *)a.veff + (a.veff ? (unsigned long)blk * T * 8 : 0), a.veff ? (unsigned long)T * 8 : 0);
  const auto rpv = ordered ? rveff : make_rsrc(a.vext, a.vext ? ntot * 8 : 0);
  const unsigned steppv = ordered ? NT * 8 : stepv * 8;
  auto potential_offset = [&](int t, int u) { return ordered ? (unsigned)(u * SV::r * NT + t) * 8u : real_element(t, u) * 8u; };
  // the start-of-step pass loads vext ahead of the exchange, which hides the latency (256^3 FP64
  // 160 -> 147 us); the potential passes have no registers for it
  // 1024 threads of 32 values have no registers for the potential of all of them; tiles of 8 values,
  // the small grids', load it with the tile in every kind
  constexpr bool FULL = NT == 1024 && R == 32, EARLY = R <= 8;
  constexpr bool EARLYV = EARLY && (KIND == TGPE || KIND == TGPR);
  double pv[(KIND == TPRE && !FULL) || EARLYV ? R : 1];
  auto load_potential = [&]() {
    if constexpr ((KIND == TPRE && !FULL) || EARLYV) {
#pragma unroll
      for (int u = 0; u < R / SV::r; ++u) {
        const unsigned e = potential_offset(tid, u);
#pragma unroll
        for (int i = 0; i < SV::r; ++i) pv[u * SV::r + i] = bload_f64(rpv, e, (unsigned)i * steppv);
      }
    }
  };
  // another array's value at the thread's real-space element j
  auto value_of = [&](__amdgpu_buffer_rsrc_t array, int j) {
    return bload<C>(array, real_element(tid, j / SV::r) * CS, (unsigned)(j % SV::r) * stepv * CS);
  };
  C early[EARLY && (KIND == TPOT || KIND == TMRG) ? R : 1];
  if constexpr (EARLY && (KIND == TPOT || KIND == TMRG)) {
    const void *array = KIND == TPOT ? a.pot : a.merge;
    const auto ro = make_rsrc(array, array ? ntot * CS : 0);
#pragma unroll
    for (int j = 0; j < R; ++j) early[j] = value_of(ro, j);
  }
  if constexpr (EARLYV) load_potential();
  if (!skip1) {
    conj_all(v);
    if constexpr (A == 1) split_twiddle();
    AX::inverse(v, tid, tabx, lds);
    if constexpr (KIND == TPRE) load_potential();
    if constexpr (A > 1) {
      exchange<X0, SV, C, R, NT, PD, PW>(v, tid, lds);
      split_twiddle();
      dft_items<C, R, A>(v);
    }
    conj_all(v);
    // without h no barrier follows, and the compiler would move the last digit's arithmetic behind the
    // loads of the potential, its twiddles waiting in scratch (96 x 1 in FP64: 81 registers)
    if constexpr (A == 1) {
#pragma unroll
      for (int j = 0; j < R; ++j) asm volatile("" : "+v"(v[j].x), "+v"(v[j].y));
    }
  } else if constexpr (KIND == TPRE) {
    load_potential();
  }

  // factors in small groups behind scheduling fences, so that few evaluations are live at once
  constexpr int GROUP = sizeof(C) == 16 && KIND != TGPR ? 2 : 4;
  if constexpr (KIND == TPRE) {
#pragma unroll
    for (int u = 0; u < R / SV::r; ++u) {
      const unsigned e = FULL ? potential_offset(tid, u) : 0;
      if constexpr (FULL) __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int i = 0; i < SV::r; ++i) {
        const double d = cnorm2(v[u * SV::r + i]), pe = FULL ? bload_f64(rpv, e, (unsigned)i * steppv) : pv[FULL ? 0 : u * SV::r + i];
        if (fl & HGRID_PF_PRE_VEFF) bstore_f64(pe + a.g * d, rveff, (unsigned)tid * 8u, (unsigned)((u * SV::r + i) * NT) * 8u);
        if (fl & HGRID_PF_PRE_RED) {
          acc[HGRID_RED_NORM] += d;
          acc[HGRID_RED_QUART] += d * d;
          acc[HGRID_RED_VEXT] += pe * d;
        }
      }
    }
    if (fl & HGRID_PF_PRE_RED) reduce_partials<NT>(acc, tid, a.partials);
    return;
  } else if constexpr (KIND == TPOT || KIND == TMRG) {
    // values of another array at the tile's real-space elements, four ahead of their use
    auto with_values = [&](const void *array, auto &&apply) {
      if constexpr (EARLY) {
#pragma unroll
        for (int j = 0; j < R; ++j) v[j] = apply(v[j], early[j], j / SV::r, j % SV::r);
        return;
      }
      const auto ro = make_rsrc(array, ntot * CS);
      constexpr int AHEAD = R % 4 == 0 ? 4 : R;
      C p[2][AHEAD];
      auto fetch = [&](int j0, C(&q)[AHEAD]) {
#pragma unroll
        for (int j = 0; j < AHEAD; ++j) q[j] = value_of(ro, j0 + j);
      };
      fetch(0, p[0]);
#pragma unroll
      for (int j0 = 0; j0 < R; j0 += AHEAD) {
        __builtin_amdgcn_sched_barrier(0);
        if (j0 + AHEAD < R) fetch(j0 + AHEAD, p[(j0 / AHEAD + 1) % 2]);
#pragma unroll
        for (int j = 0; j < AHEAD; ++j) {
          if (j % GROUP == 0) __builtin_amdgcn_sched_barrier(0);
          v[j0 + j] = apply(v[j0 + j], p[(j0 / AHEAD) % 2][j], (j0 + j) / SV::r, (j0 + j) % SV::r);
        }
      }
      __builtin_amdgcn_sched_barrier(0);
    };
    if constexpr (KIND == TPOT) {
      if (a.pot) {
        with_values(a.pot, [&](C c, C q, int, int) {
          return cmul(c, phase_factor<C>(a.c_re, a.c_im, a.cons + (double)q.x, (double)q.y));
        });
      }
    } else {
      // the amplitude's shares of x, h and z, from LDS: formed in every thread their divisions spilled
      // up to 265 registers.  The other state's values arrive before the exchange's barrier, behind
      // which the tile's own elements of it, where out is that array, are overwritten.
      static_assert(sizeof(lds) >= (LX + A + CC) * sizeof(double) || A == 1, "room for the shares");
      volatile double *share = (volatile double *)lds;
      tile_sync<NT>();
      for (int e = tid; e < LX + A + CC; e += NT)
        share[e] = e < LX       ? absorb_part(e, a.bounds[0], a.bounds[1])
                   : e < LX + A ? absorb_part((long)l + (long)(e - LX) * a.rows, a.bounds[2], a.bounds[3])
                                : absorb_part((long)z0 + (e - LX - A), a.bounds[4], a.bounds[5]);
      tile_sync<NT>();
      with_values(a.merge, [&](C m, C r, int u, int i) {
#pragma clang fp contract(off)
        const int lin = SV::lin(tid, u);
        const double al = absorb_sum(share[lin / (A * CC)], share[LX + i], share[LX + A + lin % CC]), bl = 1.0 - al;
        return mk<C>((Rl)((bl * (double)r.x + al * (double)m.x) * a.post), (Rl)((bl * (double)r.y + al * (double)m.y) * a.post));
      });
    }
  } else {
    auto factors = [&](auto &&apply) {
#pragma unroll
      for (int u = 0; u < R / SV::r; ++u) {
        const unsigned e = potential_offset(tid, u);
        double p[SV::r];
        auto fetch = [&](int i0, int n) {
#pragma unroll
          for (int i = i0; i < i0 + n; ++i) p[i] = a.cons + (EARLY ? pv[EARLY ? u * SV::r + i : 0] : bload_f64(rpv, e, (unsigned)i * steppv));
        };
        if constexpr (!FULL) fetch(0, SV::r);
#pragma unroll
        for (int i0 = 0; i0 < SV::r; i0 += GROUP) {
          __builtin_amdgcn_sched_barrier(0);
          if constexpr (FULL) fetch(i0, GROUP);
#pragma unroll
          for (int i = i0; i < (i0 + GROUP < SV::r ? i0 + GROUP : SV::r); ++i) apply(v[u * SV::r + i], p[i]);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    };
    if constexpr (KIND == TGPR) {
      factors([&](C &c, double p) { c = cscale_d(c, real_decay(a.c_re * p)); });
    } else {
      factors([&](C &c, double p) { c = cmul(c, unit_phase<C>(a.c_im * p)); });
    }
  }

  if constexpr (KIND != TPRE) {
    if (!skip2) {
      if constexpr (A > 1) {
        dft_items<C, R, A>(v);
        split_twiddle();
        exchange<SV, X0, C, R, NT, PD, PW>(v, tid, lds);
        if constexpr (AX::LDS) tile_sync<NT>();  // the waves' own exchanges reuse the buffer
      }
      AX::forward(v, tid, tabx, lds);
      if constexpr (A == 1) split_twiddle();
    }
    if constexpr (KIND == TGPE || KIND == TGPR) {
      if (fl & HGRID_PF_POST_RED) {
#pragma unroll
        for (int j = 0; j < R; ++j) acc[HGRID_RED_POST] += cnorm2(v[j]);
      }
    }
    if (skip2) store(SV{}, stepv, real_element);
    else store(XL{}, stepl, form_element);
    if constexpr (KIND == TGPE || KIND == TGPR) {
      if (fl & HGRID_PF_POST_RED) reduce_partials<NT>(acc, tid, a.partials);
    }
  }
}

// ---- dispatch ----------------------------------------------------------------------------------

// Rows per A-pass tile of a middle axis (0: not split); the rest, n1 / rows, is A of the B-pass.  In
// FP64 16 rows, so that the A-pass runs in 128- and 256-thread workgroups, several per CU, which
// overlap each other's loads, exchanges and stores: 256^3 A-pass 107 us, against 147 with 32 rows
// (512 threads); the B-pass then has 16 h and 1024 threads, 211 against 190 us, and the whole
// Gross-Pitaevskii step 580 against 611.  In FP32 32 rows from 192 on (256^3 step 378 against 400).
// The longer axes take what fits: a tile of at most 2^15 FP32 or 2^14 FP64 values (768 threads of 24),
// with 64-byte rows in the B-pass.
constexpr int rows_of(bool f64, long n0, long n1) {
  return n1 == 16                                        ? 4
         : n1 == 24 || n1 == 32                          ? 8
         : n1 == 48 || n1 == 64 || n1 == 96 || n1 == 128 ? 16
         : n1 == 192                                     ? (f64 && n0 <= 256 ? 16 : 32)
         : n1 == 256                                     ? (f64 && n0 <= 256 && n0 % 3 != 0 ? 16 : 32)
         : n1 == 384                                     ? (f64 && n0 <= 256 ? 32 : 64)
         : n1 == 512                                     ? (f64 && n0 <= 256 && n0 % 3 != 0 ? 32 : 64)
                                                         : 0;
}
// the tiles that passes are built for
template <typename G, typename C> constexpr bool fits() {
  return G::NT <= (sizeof(C) == 16 && G::R == 24 ? 768 : 1024);
}
template <typename C, int LX, int A> constexpr bool shape_b() {
  if constexpr (A == 16 ? sizeof(C) == 8 || LX % 3 == 0 || LX > 256 : A == 12 ? sizeof(C) == 8 || LX > 256 : A == 1 ? LX > 256 : false)
    return false;
  else
    return fits<GeomB<C, LX, A>, C>();
}
template <typename C, int LZ, int B> constexpr bool shape_a() { return fits<GeomA<C, LZ, B>, C>(); }

#define LG_TILE_LENGTHS(X) X(16) X(24) X(32) X(48) X(64) X(96) X(128) X(192) X(256) X(384) X(512)

int launch_kinetic_f64(const hgrid_tile *p);
int launch_kinetic_f32(const hgrid_tile *p);
int launch_pre_f64(const hgrid_tile *p);
int launch_pre_f32(const hgrid_tile *p);
int launch_pot_f64(const hgrid_tile *p);
int launch_pot_f32(const hgrid_tile *p);
int launch_mrg_f64(const hgrid_tile *p);
int launch_mrg_f32(const hgrid_tile *p);
int launch_gpe_f64(const hgrid_tile *p);
int launch_gpe_f32(const hgrid_tile *p);
int launch_gpr_f64(const hgrid_tile *p);
int launch_gpr_f32(const hgrid_tile *p);

template <typename C, int LZ, int B> int launch_a(const hgrid_tile *p) {
  if constexpr (shape_a<C, LZ, B>()) {
    using G = GeomA<C, LZ, B>;
    const long nb = p->n0 * p->n1 * p->n2 / G::T;
    if (p->flags & HGRID_PF_KIN_REAL)
      hipLaunchKernelGGL((tile_kinetic<C, LZ, B, true>), dim3((unsigned)nb), dim3(G::NT), 0, stream(), *p);
    else
      hipLaunchKernelGGL((tile_kinetic<C, LZ, B, false>), dim3((unsigned)nb), dim3(G::NT), 0, stream(), *p);
    return check_launch("tile_kinetic");
  } else {
    return -1;
  }
}

template <typename C, int B> int launch_a_rows(const hgrid_tile *p) {
#define LG_CASE(n) \
  case n: return launch_a<C, n, B>(p);
  switch (p->n2) {
    LG_TILE_LENGTHS(LG_CASE)
    default: return -1;
  }
#undef LG_CASE
}

template <typename C> int launch_kinetic(const hgrid_tile *p) {
  switch (p->rows) {
    case 4: return launch_a_rows<C, 4>(p);
    case 8: return launch_a_rows<C, 8>(p);
    case 16: return launch_a_rows<C, 16>(p);
    case 32: return launch_a_rows<C, 32>(p);
    case 64: return launch_a_rows<C, 64>(p);
    default: return -1;
  }
}

template <typename C, int LX, int A, int KIND> int launch_b(const hgrid_tile *p) {
  if constexpr (shape_b<C, LX, A>() && (KIND != TMRG || A > 1)) {
    using G = GeomB<C, LX, A>;
    const long nb = p->n0 * p->n1 * p->n2 / G::T;
    hipLaunchKernelGGL((tile_potential<C, LX, A, KIND>), dim3((unsigned)nb), dim3(G::NT), 0, stream(), *p);
    return check_launch("tile_potential");
  } else {
    return -1;
  }
}

template <typename C, int KIND> int launch_potential(const hgrid_tile *p) {
#define LG_CASE(n) \
  case n: \
    switch (p->flat ? 1 : p->nh) { \
      case 1: return launch_b<C, n, 1, KIND>(p); \
      case 3: return launch_b<C, n, 3, KIND>(p); \
      case 4: return launch_b<C, n, 4, KIND>(p); \
      case 6: return launch_b<C, n, 6, KIND>(p); \
      case 8: return launch_b<C, n, 8, KIND>(p); \
      case 12: return launch_b<C, n, 12, KIND>(p); \
      case 16: return launch_b<C, n, 16, KIND>(p); \
      default: return -1; \
    }
  switch (p->flat ? p->nh : p->n0) {
    LG_TILE_LENGTHS(LG_CASE)
    default: return -1;
  }
#undef LG_CASE
}

}  // namespace tile
}  // namespace lg
