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
  using G = GeomA<C, LZ, B>;
  if (groups % G::M) return false;
  t->blocks_a = points / G::T;
  return true;
}

template <typename C, int B> static bool plan_z(long points, long groups, hgrid_tile *t) {
#define LG_CASE(n) \
  case n: return plan_a<C, n, B>(points, groups, t);
  switch (t->n2) {
    LG_TILE_LENGTHS(LG_CASE)
    case 384: if constexpr (B == 4) return t->flat && plan_a<C, 384, 4>(points, groups, t); else return false;
    case 512: if constexpr (B == 4) return t->flat && plan_a<C, 512, 4>(points, groups, t); else return false;
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
  switch (t->rows) {
    case 4: return plan_z<C, 4>(points, groups, t);
    case 8: return plan_z<C, 8>(points, groups, t);
    case 16: return plan_z<C, 16>(points, groups, t);
    case 32: return plan_z<C, 32>(points, groups, t);
    default: return false;
  }
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
    case HGRID_TILE_GPE:
      if ((!t->veff && !t->vext) || (t->c_re != 0.0 && t->c_im != 0.0)) return -1;
      if (t->c_im == 0.0) return f64 ? lg::tile::launch_gpr_f64(t) : lg::tile::launch_gpr_f32(t);
      return f64 ? lg::tile::launch_gpe_f64(t) : lg::tile::launch_gpe_f32(t);
    default: return -1;
  }
}
