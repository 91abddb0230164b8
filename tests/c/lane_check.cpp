// CPU replay of the one-tile-per-work-group row x column launch
// (ttc_lane.hpp) against the planner's parameters, for many geometries, type
// pairs, vector widths and tiles:
//   - rc_tile_of maps the work-groups one to one onto the tile ids, and the
//     grid records decode every id to its own origin and partial flags;
//   - the offset tables, lane by lane and slot by slot, for full and partial
//     tiles: every table and LDS index in bounds, each element of the tile
//     read and written exactly once with its true A and B offset at the same
//     LDS position, every other slot out of the buffer range (>= 2^31), and
//     nothing a padding slot stages lands where the tile's elements are.
// Prints one summary line; exit status 1 on the first violation.
#include <algorithm>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <random>
#include <set>
#include <utility>
#include <vector>

#include "ttc_plan.h"

using namespace ttc;

#define CHECK(cond, ...)                         \
  do {                                           \
    if (!(cond)) {                               \
      std::fprintf(stderr, "FAIL %s: ", #cond);  \
      std::fprintf(stderr, __VA_ARGS__);         \
      std::fprintf(stderr, "\n");                \
      return false;                              \
    }                                            \
  } while (0)

static bool check_walk(const Geometry& g, const int* tile, const RCLaneParams& p) {
  std::vector<char> seen(p.walk.ntiles, 0);
  std::set<std::pair<long long, long long>> origins;
  for (uint32_t w = 0; w < p.walk.ntiles; ++w) {
    const uint32_t t = rc_tile_of(p.walk, w);
    CHECK(t < p.walk.ntiles && !seen[t], "work-group %u: tile %u of %u", w, t, p.walk.ntiles);
    seen[t] = 1;
    uint32_t rem = t;
    long long a = 0, b = 0;
    for (int i = 0; i < p.grank; ++i) {
      const uint32_t q = fdiv(rem, p.grid[i].m, p.grid[i].s), x = rem - q * p.grid[i].d;
      CHECK(q == rem / p.grid[i].d, "division");
      rem = q;
      a += (long long)x * p.grid[i].tsa;
      b += (long long)x * p.grid[i].tsb;
    }
    CHECK(rem == 0, "id %u past the grid", t);
    if (p.walk.ntiles < 20000) origins.insert({a, b});
  }
  if (p.walk.ntiles < 20000) CHECK(origins.size() == p.walk.ntiles, "origins %zu", origins.size());
  (void)g;
  (void)tile;
  return true;
}

static void offsets(const RCLaneParams& p, int first, int n, long long l, long long& oa, long long& ob) {
  oa = ob = 0;
  for (int m = first; m < first + n; ++m) {
    const long long x = l % p.dim[m].d;
    l /= p.dim[m].d;
    oa += x * p.dim[m].sa;
    ob += x * p.dim[m].sb;
  }
}

static bool check_tile(const RCLaneParams& p, int szA, int szB, int va, int vb, int div, int rows, int cols,
                       int lds_bytes, int le) {
  const int NIA = rc_elems(szA) / va / div, NIB = rc_elems(szB) / vb / div;
  const long long nA = (long long)p.kA * NIA, nB = (long long)p.kB * NIB, ntab = nA + nB + p.R + p.C;
  CHECK(p.tab + 4 * ntab <= lds_bytes && p.tab % 16 == 0, "tables end at %lld of %d", p.tab + 4 * ntab, lds_bytes);
  CHECK((long long)(p.spare + va) * le <= p.tab, "data region %d + %d", p.spare, va);
  CHECK(p.kA * (long long)p.la <= kRcThreads && p.kB * (long long)p.lb <= kRcThreads, "lanes");
  std::vector<long long> rA(p.R), rB(nB), cB(p.C), cA(nA);  // true offsets, -1: out of range
  std::vector<uint32_t> colS(nA), rowS(nB), rowA(p.R, 0x55555555u), colB(p.C, 0x55555555u);
  for (long long e = 0; e < std::max(nA, nB); ++e) {
    if (e < nA) CHECK(fdiv((uint32_t)e, p.kAm, p.kAs) == e / p.kA, "column step division");
    if (e < nB) CHECK(fdiv((uint32_t)e, p.kBm, p.kBs) == e / p.kB, "row step division");
  }
  for (long long e = 0; e < nA; ++e) {
    const long long j = e / NIA + (e % NIA) * p.kA;
    long long oa, ob;
    offsets(p, p.na, p.nb, j, oa, ob);
    colS[e] = j < cols ? (uint32_t)oa : kRcTabOOB;
    if (j < p.C) {
      colB[j] = j < cols ? (uint32_t)ob : kRcTabOOB;
      cA[j] = oa, cB[j] = ob;
    }
  }
  for (long long e = 0; e < nB; ++e) {
    const long long i = e / NIB + (e % NIB) * p.kB;
    long long oa, ob;
    offsets(p, 0, p.na, i, oa, ob);
    rowS[e] = i < rows ? (uint32_t)ob : kRcTabOOB;
    if (i < p.R) {
      rowA[i] = i < rows ? (uint32_t)oa : kRcTabOOB;
      rA[i] = oa, rB[i] = ob;
    }
  }
  const long long n = (long long)rows * cols;
  std::vector<int> seen_r(n, 0), seen_w(n, 0);
  std::set<long long> junk;
  for (uint32_t tid = 0; tid < (uint32_t)kRcThreads; ++tid) {
    const uint32_t jl = fdiv(tid, p.lam, p.las), ai = (tid - jl * p.la) * va;
    CHECK(jl == tid / p.la, "lane division");
    const bool on = jl < (uint32_t)p.kA;
    const uint32_t lds0 = on ? ai + jl * p.RP : (uint32_t)p.spare, step = on ? (uint32_t)(p.kA * p.RP) : 0u;
    if (on) CHECK(ai < (uint32_t)p.R && (long long)jl * NIA + NIA <= nA, "read tables");
    const uint32_t rowoff = on ? rowA[ai] : kRcTabOOB;
    for (int it = 0; it < NIA; ++it) {
      const uint32_t off = rowoff + colS[(on ? (size_t)jl * NIA : 0) + it];
      const long long j = (long long)jl + (long long)it * p.kA;
      for (int v = 0; v < va; ++v) {
        const long long at = (long long)lds0 + (long long)it * step + v, i = (long long)ai + v;
        CHECK(at < p.spare + va, "stage index %lld of %d", at, p.spare + va);
        if (on && i < rows && j < cols) {
          CHECK((long long)off + (long long)v * szA == rA[i] + cA[j] && off < 0x80000000u, "A offset of (%lld, %lld)", i, j);
          CHECK(at == i + j * p.RP, "stage position of (%lld, %lld)", i, j);
          CHECK(seen_r[i + j * rows]++ == 0, "read twice (%lld, %lld)", i, j);
        } else {
          CHECK(off >= 0x80000000u && (uint64_t)off + 64 <= 0x100000000ull, "padding read offset %u", off);
          junk.insert(at);
        }
      }
    }
  }
  for (uint32_t tid = 0; tid < (uint32_t)kRcThreads; ++tid) {
    const uint32_t il = fdiv(tid, p.lbm, p.lbs), bj = (tid - il * p.lb) * vb;
    CHECK(il == tid / p.lb, "lane division");
    const bool on = il < (uint32_t)p.kB;
    if (on) CHECK(bj < (uint32_t)p.C && (long long)il * NIB + NIB <= nB, "write tables");
    const uint32_t coloff = on ? colB[bj] : kRcTabOOB;
    const uint32_t lds0 = on ? il + bj * p.RP : 0u, step = on ? (uint32_t)p.kB : 0u;
    for (int it = 0; it < NIB; ++it) {
      const uint32_t off = rowS[(on ? (size_t)il * NIB : 0) + it] + coloff;
      const long long i = (long long)il + (long long)it * p.kB;
      for (int v = 0; v < vb; ++v) {
        const long long at = (long long)lds0 + (long long)it * step + (long long)v * p.RP, j = (long long)bj + v;
        CHECK(at < p.spare + va, "write-walk index %lld of %d", at, p.spare + va);
        if (on && i < rows && j < cols) {
          CHECK((long long)off + (long long)v * szB == rB[i] + cB[j] && off < 0x80000000u, "B offset of (%lld, %lld)", i, j);
          CHECK(at == i + j * p.RP, "write position of (%lld, %lld)", i, j);
          CHECK(seen_w[i + j * rows]++ == 0, "written twice (%lld, %lld)", i, j);
          CHECK(junk.count(at) == 0, "padding staged over (%lld, %lld)", i, j);
        } else {
          CHECK(off >= 0x80000000u && (uint64_t)off + 64 <= 0x100000000ull, "padding write offset %u", off);
        }
      }
    }
  }
  for (long long e = 0; e < n; ++e) CHECK(seen_r[e] == 1 && seen_w[e] == 1, "element %lld missed", e);
  return true;
}

// The few-byte form of a launch against the full one: origins, partial groups
// and the groups' offsets (sdiv itself is checked in main).
static bool check_small(const RCLaneParams& p, const RCLaneSmall& s, int szA, int szB) {
  CHECK(s.ntiles == p.walk.ntiles && s.R == p.R && s.C == p.C && s.Rl == p.Rl && s.Cl == p.Cl && s.kA == p.kA &&
            s.kB == p.kB && s.tab16 * 16 == p.tab && s.spare == p.spare && (s.groups & 15) == p.na &&
            s.groups >> 4 == p.nb && (s.R | 1) == p.RP,
        "small fields");
  const uint32_t step = p.walk.ntiles / 5000 + 1;
  for (uint32_t w = 0; w < p.walk.ntiles; w += w < 64 || w + 64 > p.walk.ntiles ? 1 : step) {
    uint32_t rem = rc_tile_of(p.walk, w), last = 0;
    long long oa = 0, ob = 0;
    for (int g = 0; g < p.grank; ++g) {
      const uint32_t x = rem % p.grid[g].d;
      rem /= p.grid[g].d;
      oa += (long long)x * p.grid[g].tsa * szA;
      ob += (long long)x * p.grid[g].tsb * szB;
      if (x == p.grid[g].d - 1) last |= p.grid[g].part;
    }
    int64_t sa, sb;
    const uint32_t sl = rc_small_origin(&s, w, sa, sb);
    CHECK(sa == oa && sb == ob && sl == last, "small origin");
  }
  for (int side = 0; side < 2; ++side)
    for (int l = 0; l < (side ? p.C : p.R); ++l) {
      const int first = side ? p.na : 0, n = side ? p.nb : p.na;
      int32_t oa = 0, ob = 0, sa, sb;
      uint32_t r = (uint32_t)l;
      for (int m = first; m < first + n; ++m) {
        oa += (int32_t)(r % p.dim[m].d) * p.dim[m].sa;
        ob += (int32_t)(r % p.dim[m].d) * p.dim[m].sb;
        r /= p.dim[m].d;
      }
      rc_small_offsets(&s, first, n, (uint32_t)l, sa, sb);
      CHECK(sa == oa && sb == ob, "small offsets");
    }
  return true;
}

// sdiv_by for every divisor and numerators at its quotients' edges, with
// reciprocals 1 ulp off.
static bool check_sdiv() {
  std::mt19937_64 rng(7);
  for (uint32_t d = 1; d < kSmallCount; d += d < 5000 ? 1 : 1 + (uint32_t)(rng() % 400)) {
    const float inv = 1.0f / (float)d, nudged[3] = {inv, std::nextafterf(inv, 0.0f), std::nextafterf(inv, 2.0f)};
    const uint32_t qmax = (kSmallCount - 1) / d;
    for (int t = 0; t < 40; ++t) {
      const uint32_t q = t == 0 ? 0 : t == 1 ? qmax : (uint32_t)(rng() % (qmax + 1));
      for (const long long n : {(long long)q * d - 1, (long long)q * d, (long long)q * d + d - 1}) {
        if (n < 0 || n >= kSmallCount) continue;
        for (const float f : nudged) CHECK(sdiv_by((uint32_t)n, f) == (uint32_t)n / d, "sdiv");
      }
    }
  }
  return true;
}

int main(int argc, char** argv) {
  const int ncases = argc > 1 ? std::atoi(argv[1]) : 200;
  std::mt19937_64 rng(4242);
  if (!check_sdiv()) return 1;
  const int pairs[][2] = {{TTC_S, TTC_S},       {TTC_D, TTC_D},    {TTC_C, TTC_C}, {TTC_Z, TTC_Z}, {TTC_BF16, TTC_BF16},
                          {TTC_S, TTC_BF16},    {TTC_F16, TTC_S},  {TTC_D, TTC_S}, {TTC_S, TTC_D}, {TTC_C, TTC_Z},
                          {TTC_BF16, TTC_E4M3}, {TTC_S, TTC_E5M2}};
  long long walks = 0, tiles = 0, banded = 0, partial = 0, full_size = 0, far = 0, small = 0;
  for (int c = 0; c < ncases; ++c) {
    const int r = 2 + (int)(rng() % 5);
    int perm[8], size[8], lda[8], ldb[8];
    for (int k = 0; k < r; ++k) perm[k] = k;
    std::shuffle(perm, perm + r, rng);
    long long vol = 1;
    for (int k = 0; k < r; ++k) vol *= size[k] = 1 + (int)(rng() % (k < 2 ? 400 : 24));
    while (vol > (1ll << (c % 8 == 0 ? 25 : 20))) {
      const int k = (int)(std::max_element(size, size + r) - size);
      vol = vol / size[k] * ((size[k] + 1) / 2);
      size[k] = (size[k] + 1) / 2;
    }
    const bool pad = rng() % 4 == 0;
    for (int k = 0; k < r; ++k) {
      lda[k] = size[k] + (pad ? (int)(rng() % 3) : 0);
      ldb[k] = size[perm[k]] + (pad ? (int)(rng() % 3) : 0);
    }
    Geometry g;
    if (make_geometry(r, perm, size, lda, ldb, g) != TTC_SUCCESS || g.elements == 0 || g.rank < 2 || g.perm[0] == 0)
      continue;
    for (const auto& pr : pairs) {
      const int ta = pr[0], tb = pr[1], szA = dtype_bytes(ta), szB = dtype_bytes(tb), le = lds_elem_bytes(ta, tb);
      const int vas[] = {1, widest_vec_a(g, ta)}, vbs[] = {1, widest_vec_b(g, tb)};
      for (int va : vas)
        for (int vb : vbs)
          for (int run : {0, 4, 32, 256})
            for (int div = 1; div <= 2; ++div) {
              int t[kMaxDim], lds = 0;
              const int order = 1 + (int)(rng() % 4), grid = 1 + (int)(rng() % 4);
              RCLaneParams p;
              if (run ? !choose_rc_tile(g, ta, tb, va, vb, run, run, t, nullptr)
                      : !choose_lane_tile(g, ta, tb, va, vb, c % 2 != 0, t))
                continue;
              if (!build_lane_params(g, t, ta, tb, va, vb, grid, order, div, p, lds)) continue;
              bool ok = check_walk(g, t, p);
              RCLaneSmall sp;
              if (div == 2 && build_lane_small(g, t, ta, tb, order, p, sp)) {
                ok = ok && check_small(p, sp, szA, szB);
                ++small;
              }
              ++walks;
              banded += p.walk.bandw != 0;
              full_size += div == 1;
              for (int rows : {p.R, p.Rl})
                for (int cols : {p.C, p.Cl}) {
                  ok = ok && check_tile(p, szA, szB, va, vb, div, rows, cols, lds, le);
                  ++tiles;
                  partial += rows < p.R || cols < p.C;
                }
              if (!ok) {
                std::fprintf(stderr, "case %d types %d->%d va %d vb %d div %d R %d C %d Rl %d Cl %d\n", c, ta, tb, va, vb,
                             div, p.R, p.C, p.Rl, p.Cl);
                return 1;
              }
            }
    }
  }
  // tiles whose A offsets pass 2^30 (dimension 3 has a 25 MB stride in A):
  // taken where no table entry that large can meet kRcTabOOB
  for (const int rows : {128, 64, 100}) {
    const int perm[4] = {3, 1, 0, 2}, size[4] = {256, 192, 128, 96}, tile[kMaxDim] = {rows, 1, 1, 64, 1, 1, 1, 1};
    Geometry g;
    if (make_geometry(4, perm, size, nullptr, nullptr, g) != TTC_SUCCESS) return 1;
    RCLaneParams p;
    int lds = 0;
    const bool fits = build_lane_params(g, tile, TTC_S, TTC_BF16, 4, 8, 0, 2, 1, p, lds);
    if (fits != (rows != 100)) {
      std::fprintf(stderr, "rows %d with A offsets past 2^30: %d\n", rows, fits);
      return 1;
    }
    far += fits;
    for (int cols : {64, 32})
      if (fits && !check_tile(p, 4, 2, 4, 8, 1, rows, cols, lds, 4)) return 1;
  }
  // the units of an fp8 cast: every one taken once, in order
  for (const bool amax : {false, true})
    for (const uint32_t n : {1u, 2u, 63u, 64u, 65u, 66u, 127u, 255u, 256u, 257u, 258u, 259u, 4096u, 100001u, 0x7fffffffu}) {
      const AmaxUnits u = amax_units(n, amax);
      const uint32_t wgs = u.work_groups(), from = wgs > 200000 ? wgs - 1000 : 0;
      bool ok = u.first(0) == 0 && u.first(wgs) == n;
      for (uint32_t w = from; w < wgs; ++w) {
        const uint32_t k = u.first(w + 1) - u.first(w);
        ok = ok && k >= 1 && k <= (!amax || w < kAmaxHead ? 1u : 2u);
      }
      if (!ok) {
        std::fprintf(stderr, "fp8 units: %u, amax %d\n", n, (int)amax);
        return 1;
      }
    }
  std::printf("lane check: %lld walks, %lld banded, %lld full-size instances, %lld tiles, %lld partial, "
              "%lld with A spans past 2^30, %lld in few bytes: ok\n", walks, banded, full_size, tiles, partial, far, small);
  return 0;
}
