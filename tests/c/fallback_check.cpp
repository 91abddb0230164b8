// Plans whose vectors are wider than an element keep a variant for pointers
// that are not aligned to them: where the planner picked the tile itself, the
// variant keeps it if it fits one tile per work-group at scalar vectors too, or
// its launch is the one a plan of scalar vectors takes; where the caller named
// the tile, it keeps it.  Prints one summary line; exit status 1 on a
// violation.
#include <cstdio>
#include <cstring>
#include <random>
#include <vector>

#include "ttc_plan.h"

using namespace ttc;

int main() {
  std::mt19937 rng(5);
  auto below = [&](int n) { return (int)(rng() % (unsigned)n); };
  long long own = 0, given = 0, moved = 0;
  const int types[][2] = {{TTC_S, TTC_S}, {TTC_D, TTC_D}, {TTC_C, TTC_C}, {TTC_BF16, TTC_BF16}, {TTC_F16, TTC_F16},
                          {TTC_S, TTC_BF16}, {TTC_BF16, TTC_S}, {TTC_S, TTC_D}, {TTC_S, TTC_E4M3}, {TTC_BF16, TTC_E4M3}};
  for (int i = 0; i < 4000; ++i) {
    const int* t = types[below(10)];
    const int dim = 2 + below(5);
    std::vector<int> perm(dim), size(dim);
    for (int k = 0; k < dim; ++k) {
      perm[k] = k;
      size[k] = (1 + below(below(2) ? 8 : 40)) * (below(2) ? 8 : 2);
    }
    long long n = 1;
    for (int k = 0; k < dim; ++k) n *= size[k];
    if (n > (1ll << 30)) continue;
    for (int k = dim - 1; k > 0; --k) std::swap(perm[k], perm[below(k + 1)]);
    const int bz = dtype_bytes(t[1]) == 1 ? 1 : below(2);
    ttc_config_t cfg, one;
    std::memset(&cfg, 0, sizeof(cfg));
    one = cfg;
    one.vec_a = one.vec_b = 1;
    ttc_plan_t a = nullptr, b = nullptr, c = nullptr;
    if (ttc_plan_create(&a, (ttc_dtype_t)t[0], (ttc_dtype_t)t[1], dim, perm.data(), size.data(), nullptr, nullptr, bz, &cfg))
      continue;
    if (a->family == kFamilyRC && a->fallback) {
      const ttc_plan_s* f = a->fallback;
      if (ttc_plan_create(&b, (ttc_dtype_t)t[0], (ttc_dtype_t)t[1], dim, perm.data(), size.data(), nullptr, nullptr, bz, &one))
        return std::printf("FAIL scalar plan %d\n", i), 1;
      const bool same = f->family == b->family && !std::memcmp(f->tile, b->tile, sizeof(f->tile)) &&
                        f->lane_div == b->lane_div && f->small == b->small;
      const bool kept = f->family == a->family && !std::memcmp(f->tile, a->tile, sizeof(f->tile)) &&
                        (f->lane_div != 0 || a->lane_div == 0);
      if (f->va != 1 || f->vb != 1 || !(same || kept))
        return std::printf("FAIL variant of plan %d: tile %d %d %d, a scalar plan's %d %d %d\n", i, f->tile[0],
                           f->tile[1], f->tile[2], b->tile[0], b->tile[1], b->tile[2]), 1;
      ++own;
      moved += std::memcmp(f->tile, a->tile, sizeof(f->tile)) != 0;
      cfg.family = kFamilyRC;
      std::memcpy(cfg.tile, a->tile, sizeof(int) * a->g.rank);
      // (the fused problem, so that the tile's dimensions are its own)
      if (ttc_plan_create(&c, (ttc_dtype_t)t[0], (ttc_dtype_t)t[1], a->g.rank, a->g.perm, a->g.size, nullptr, nullptr, bz,
                          &cfg) == TTC_SUCCESS && c->fallback) {
        if (std::memcmp(c->fallback->tile, c->tile, sizeof(c->tile))) return std::printf("FAIL tile of plan %d\n", i), 1;
        ++given;
      }
    }
    for (ttc_plan_t q : {a, b, c})
      if (q) ttc_plan_destroy(q);
  }
  std::printf("%lld variants of the planner's tiles, %lld of them with a tile of their own, %lld of given tiles\n", own,
              moved, given);
  return 0;
}
