// Tile counts of dimensions within a tile of 2^31 elements: every plan that is
// made for them (all families, type pairs, vector widths) has as many tiles as
// 64-bit arithmetic gives, in every form of its parameters.  Prints one summary
// line; exit status 1 on a violation.
#include <climits>
#include <cstdio>
#include <cstring>

#include "ttc_plan.h"

using namespace ttc;

static long long ceil_div(long long n, long long t) { return (n + t - 1) / t; }

static bool check_plan(const ttc_plan_s* pl, const char* what) {
  const Geometry& g = pl->g;
  long long want = 1;
  for (int k = 0; k < g.rank; ++k) want *= ceil_div(g.size[k], pl->tile[k]);
  bool ok = want < (1ll << 31);
  if (pl->family == kFamilyRC) {
    ok = ok && pl->rc.ntiles >= want && pl->rc.ntiles < (1u << 31);
    if (pl->tile_order <= 2) ok = ok && pl->rc.ntiles == want;
    if (pl->lane_div) {
      ok = ok && pl->lane.walk.ntiles == want;
      long long grid = 1;
      for (int i = 0; i < pl->lane.grank; ++i) grid *= pl->lane.grid[i].d;
      ok = ok && grid == want;
    }
  } else if (pl->family == kFamilyBox) {
    ok = ok && pl->p.ntiles == want;
    for (int k = 0; k < g.rank; ++k) ok = ok && pl->p.gdiv[k].d == ceil_div(g.size[k], pl->tile[k]);
  }
  for (int k = 0; k < g.rank; ++k) ok = ok && pl->tile[k] >= 1 && pl->tile[k] <= g.size[k];
  if (!ok)
    std::fprintf(stderr, "FAIL %s: types %d %d size %d %d family %d tile %d %d v %d %d: want %lld rc %u lane %u box %u\n",
                 what, pl->type_a, pl->type_b, g.size[0], g.size[1], pl->family, pl->tile[0], pl->tile[1], pl->va,
                 pl->vb, want, pl->rc.ntiles, pl->lane_div ? pl->lane.walk.ntiles : 0, pl->p.ntiles);
  return ok;
}

int main() {
  long long plans = 0, lanes = 0, boxes = 0, refused = 0;
  for (int ta = 0; ta < 8; ++ta)
    for (int tb = 0; tb < 8; ++tb) {
      if (!pair_supported(ta, tb)) continue;
      for (int below : {0, 1, 2, 3, 7, 8, 15, 63, 64, 127, 255, 300})
        for (int other : {2, 3, 8, 33})
          for (int swap = 0; swap < 2; ++swap)
            for (int family = 0; family < 3; ++family)
              for (int variant = 0; variant < 4; ++variant) {
                const int n = INT_MAX - below, perm[] = {1, 0};
                const int size[] = {swap ? other : n, swap ? n : other};
                ttc_config_t c;
                std::memset(&c, 0, sizeof(c));
                c.family = family;
                if (variant == 1) c.wg_per_cu = 2;
                if (variant == 2) c.vec_a = c.vec_b = 1, c.tile_order = 3;
                if (variant == 3) c.run_a = 64, c.run_b = 16, c.tile_order = 1;
                for (PlanUse use : {kPlanSingle, kPlanGroupTile, kPlanGroupWalk}) {
                  ttc_plan_t pl = nullptr;
                  if (plan_create(&pl, (ttc_dtype_t)ta, (ttc_dtype_t)tb, 2, perm, size, nullptr, nullptr, 1, &c, use) !=
                      TTC_SUCCESS) {
                    ++refused;
                    continue;
                  }
                  for (const ttc_plan_s* q : {(const ttc_plan_s*)pl, (const ttc_plan_s*)pl->fallback})
                    if (q) {
                      if (!check_plan(q, q == pl ? "plan" : "fallback")) return 1;
                      ++plans;
                      lanes += q->family == kFamilyRC && q->lane_div;
                      boxes += q->family == kFamilyBox;
                    }
                  ttc_plan_destroy(pl);
                }
              }
    }
  std::printf("%lld plans, %lld lane, %lld box, %lld refused\n", plans, lanes, boxes, refused);
  return 0;
}
