// C-ABI of the tile passes (see tile_pass.hpp for the kernels).
#include "tile_pass.hpp"

namespace lg {
namespace tile {

// geometry of the B-pass over x of LX points and A values of h
template <typename C, int LX, int A> static bool plan_b(long points, hgrid_tile *t) {
  if constexpr (shape_b<C, LX, A>()) {
    using G = GeomB<C, LX, A>;
    if (t->n2 % G::CC) return false;
    t->blocks_b = points / G::T;
    t->threads_b = G::NT;
    return true;
  } else {
    return false;
  }
}

template <typename C> static bool plan_x(long lx, int a, long points, hgrid_tile *t) {
#define LG_CASE(n) \
  case n: \
    switch (a) { \
      case 1: return plan_b<C, n, 1>(points, t); \
      case 3: return plan_b<C, n, 3>(points, t); \
      case 4: return plan_b<C, n, 4>(points, t); \
      case 6: return plan_b<C, n, 6>(points, t); \
      case 8: return plan_b<C, n, 8>(points, t); \
      case 12: return plan_b<C, n, 12>(points, t); \
      case 16: return plan_b<C, n, 16>(points, t); \
      default: return false; \
    }
  switch (lx) {
    LG_TILE_LENGTHS(LG_CASE)
    default: return false;
  }
#undef LG_CASE
}

// the A-pass tile of rows z rows of lz points: blocks, if its (x, h) groups divide the grid
template <typename C, int LZ, int B> static bool plan_a(long points, long groups, hgrid_tile *t) {
  if constexpr (shape_a<C, LZ, B>()) {
    using G = GeomA<C, LZ, B>;
    if (groups % G::M) return false;
    t->blocks_a = points / G::T;
    t->threads_a = G::NT;
    return true;
  } else {
    return false;
  }
}

template <typename C, int B> static bool plan_z(long points, long groups, hgrid_tile *t) {
#define LG_CASE(n) \
  case n: return plan_a<C, n, B>(points, groups, t);
  switch (t->n2) {
    LG_TILE_LENGTHS(LG_CASE)
    default: return false;
  }
#undef LG_CASE
}

template <typename C> static bool plan(hgrid_tile *t) {
  const long points = t->n0 * t->n1 * t->n2;
  if (points > 0xffffffffL / (long)sizeof(C)) return false;
  t->flat = t->n0 == 1;
  // 2-D: 4 rows, so that even a 64-point axis leaves 16 for the B-pass
  t->rows = t->flat ? 4 : rows_of(sizeof(C) == 16, t->n0, t->n1);
  if (!t->rows || t->n1 % t->rows) return false;
  t->nh = (int)(t->n1 / t->rows);
  t->sh = t->rows * t->n2;
  t->sx = t->flat ? t->sh : t->n1 * t->n2;
  t->back = (double)(t->n0 * t->nh);
  if (!plan_x<C>(t->flat ? t->nh : t->n0, t->flat ? 1 : t->nh, points, t)) return false;
  const long groups = t->n0 * t->nh;
  bool taken = false;
  switch (t->rows) {
    case 4: taken = plan_z<C, 4>(points, groups, t); break;
    case 8: taken = plan_z<C, 8>(points, groups, t); break;
    case 16: taken = plan_z<C, 16>(points, groups, t); break;
    case 32: taken = plan_z<C, 32>(points, groups, t); break;
    case 64: taken = plan_z<C, 64>(points, groups, t); break;
    default: break;
  }
  if (!taken) return false;
  // Workgroups that fill a CU alone wait for their own loads and stores, which the smaller ones of
  // the pencil passes overlap; their fewer sweeps gain less then.  ms of 6 steps (relaxation: 32),
  // pencils and then tiles; GPE in real time, complex potential, the same 4th order, merged
  // relaxation:
  //   FP64  256 256 512 (A 1024, B  512 threads) 10.3  9.7   9.3  8.5   12.4 16.3   29.7 30.0
  //         256 512 256 (   512,   1024)         10.4  8.5   9.5  7.3   12.7 14.9   29.5 25.8
  //         256 256 256 (   256,   1024)          4.6  3.6   4.1  2.8    5.7  5.5   13.2 10.9
  //         384 256 384 (   512,    512)         17.2 11.4  14.9  9.7   19.5 15.7   44.8 35.2
  //   FP32  512 512 512 (  1024,   1024)         26.1 26.5  22.6 18.9   28.6 33.9   77.9 79.9
  //         512 384 192 (   512,   1024)          7.4  6.9   6.2  4.8    8.0  8.3   21.0 23.4
  //         256 512 256 (   512,    512)          5.3  5.8   4.3  4.1    5.9  6.9   15.2 15.0
  //         256 256 512 (   512,    512)          5.5  5.5   4.4  3.8    6.1  6.6   16.5 14.9
  //         512 256 256 (   256,   1024)          5.5  5.3   4.4  3.3    6.1  6.0   16.0 16.2
  //         256 256 256 (   256,    512)          2.7  2.1   2.1  1.4    2.8  2.3    7.5  5.9
  //         384 384 384 (  1024,    768)         11.9 10.4   9.5  8.1   12.1 12.8   36.2 32.5
  //   FP64  256 192 512 (   512,    512)          7.7  7.4   6.9  6.2    9.2 10.6   22.2 23.2
  //         512 384 128 (   512,    512)          9.8  7.7   9.0  6.3   11.5 11.1   27.8 24.7
  //         192 512 256 (  1024,    256)          7.8  6.4   7.2  5.6    9.6 10.4   22.1 21.7
  // `pencils` tells steps that end in real space and merged relaxations apart, not GPE steps from those with
  // a complex potential.  The first line therefore leaves whole FP32 shapes to the pencils where the GPE step gains
  // nothing or little (its 512 384 192 gains 7 %), although complex potentials would gain there.  384 points
  // along z run better in tiles than the other long axes do, and an h with a factor 3 worse: these
  // exceptions rest on the rows above alone.
  const bool f64 = sizeof(C) == 16;
  const int threads = t->threads_a + t->threads_b;
  if (!f64 && t->n2 != 384 && t->n1 >= 384 && t->threads_a >= 512 && t->threads_b >= 512) return false;
  if (threads >= 1024 && (!f64 || t->n0 == 512 || t->n1 == 512 || t->n2 == 512)) t->pencils |= 1;
  if (f64 && threads >= 1024 && (t->n0 == 512 || t->n2 == 512) && (t->threads_a >= 1024 || (t->nh % 3 == 0 && t->n1 < 384)))
    t->pencils |= 2;
  if (!f64 && threads >= 1280 && t->n2 >= 256 && t->n2 != 384) t->pencils |= 2;
  return true;
}

}  // namespace tile
}  // namespace lg

extern "C" int hgrid_tile_plan(int prec, long n0, long n1, long n2, hgrid_tile *t) {
  *t = hgrid_tile{};
  t->prec = prec;
  t->n0 = n0;
  t->n1 = n1;
  t->n2 = n2;
  t->post = 1.0;
  if (prec == HGRID_C128) return lg::tile::plan<double2>(t);
  if (prec == HGRID_C64) return lg::tile::plan<float2>(t);
  return 0;
}

extern "C" int hgrid_tile_pass(const hgrid_tile *t, int pass) {
  hgrid_tile shape;
  if (!t || !hgrid_tile_plan(t->prec, t->n0, t->n1, t->n2, &shape) || shape.rows != t->rows || shape.nh != t->nh ||
      shape.flat != t->flat || shape.sx != t->sx || shape.sh != t->sh)
    return -1;
  if ((t->flags & HGRID_PF_PRESCALE) && !t->scale && (pass != HGRID_TILE_KINETIC || !t->norm_partials || t->norm_count < 1)) return -1;
  const bool f64 = t->prec == HGRID_C128;
  switch (pass) {
    case HGRID_TILE_KINETIC: return f64 ? lg::tile::launch_kinetic_f64(t) : lg::tile::launch_kinetic_f32(t);
    case HGRID_TILE_START: return f64 ? lg::tile::launch_pre_f64(t) : lg::tile::launch_pre_f32(t);
    case HGRID_TILE_POT: return f64 ? lg::tile::launch_pot_f64(t) : lg::tile::launch_pot_f32(t);
    case HGRID_TILE_MERGE:
      if (!t->merge || t->flat) return -1;
      return f64 ? lg::tile::launch_mrg_f64(t) : lg::tile::launch_mrg_f32(t);
    case HGRID_TILE_GPE:
      if ((!t->veff && !t->vext) || (t->c_re != 0.0 && t->c_im != 0.0)) return -1;
      if (t->c_im == 0.0) return f64 ? lg::tile::launch_gpr_f64(t) : lg::tile::launch_gpr_f32(t);
      return f64 ? lg::tile::launch_gpe_f64(t) : lg::tile::launch_gpe_f32(t);
    default: return -1;
  }
}
