// The row copy's launch parameters (one chunk per work-group) against the rows
// they stand for, for every type pair, beta read or not, dimension 0 of 1 to 70
// elements and of the last extents below 2^31: the vectors of a row, shifted as
// the kernel shifts the last one, start inside the row, follow each other
// without a gap and end with the row; the chunks cover all vectors, whose count
// stays below 2^31; and the launch in few bytes of arguments, where there is
// one, takes every vector to the same row.  Prints one summary line; exit status 1 on a violation.
#include <climits>
#include <cstdio>

#include "ttc_plan.h"

using namespace ttc;

#define CHECK(cond)                                                                                              \
  do {                                                                                                           \
    if (!(cond)) {                                                                                               \
      std::fprintf(stderr, "FAIL %s: types %d %d beta %d n0 %d rows %lld v %d unaligned %d nv %u total %u\n",    \
                   #cond, ta, tb, beta, n0, rows, pl->row1_v, pl->row1_unaligned, pl->row1.nv, pl->row1.total); \
      return false;                                                                                              \
    }                                                                                                            \
  } while (0)

static bool check_row(const ttc_plan_s* pl, int ta, int tb, int beta, int n0, long long rows, long long& unaligned,
                      long long& small) {
  const RowParams& p = pl->row1;
  const long long V = pl->row1_v, nv = p.nv;
  CHECK(pl->family == kFamilyRow && p.n0 == n0);
  CHECK(nv * V >= n0 && nv * V - n0 < V);
  CHECK((long long)p.total == rows * nv && rows * nv < (1ll << 31));
  if (pl->row1_unaligned) {
    CHECK(V >= 2 && V <= n0);
    ++unaligned;
  } else {
    CHECK(n0 % V == 0);
  }
  auto start = [&](long long i) {  // as row_chunk
    const int32_t e = (int32_t)(uint32_t)i * (int32_t)V;
    return (long long)(pl->row1_unaligned ? e - row_shift(e, (int32_t)V, p.n0) : e);
  };
  for (long long i = 0; i < nv; i = i + 1 == 200 && nv > 400 ? nv - 200 : i + 1) {
    CHECK(start(i) >= 0 && start(i) + V <= n0);
    CHECK(i == 0 ? start(i) == 0 : start(i) == i * V || i == nv - 1);
    if (i > 0) CHECK(start(i) > start(i - 1) && start(i) <= start(i - 1) + V);
  }
  CHECK(start(nv - 1) + V == n0);
  // the few-byte form of the launch stands for the same rows
  if (pl->small) {
    const RowSmall& q = pl->row_small;
    CHECK(p.total < kSmallCount && q.total == p.total && q.nv == p.nv && q.n0 == p.n0 && q.rank == p.rank);
    CHECK((q.xcd_share != 0) == (p.xcd_share != 0) && q.grid == pl->row1_grid);
    for (uint32_t i = 0; i < p.total; ++i) {
      const uint32_t row = fdiv(i, p.nvm, p.nvs);
      CHECK(row == i / p.nv && sdiv(i, q.nv) == row);
      uint32_t rem = row, rem2 = row;
      for (int k = 0; k < p.rank; ++k) {
        const uint32_t x = rem % p.dn[k].d, d2 = sdiv(rem2, q.dim[k].d), x2 = rem2 - d2 * q.dim[k].d;
        CHECK(fdiv(rem, p.dn[k].m, p.dn[k].s) == rem / p.dn[k].d && x == x2);
        CHECK(p.sa[k] == q.dim[k].sa && p.sb[k] == q.dim[k].sb);
        rem /= p.dn[k].d;
        rem2 = d2;
      }
      CHECK(rem == 0 && rem2 == 0);
    }
    ++small;
  }
  const int szA = dtype_bytes(ta), szB = dtype_bytes(tb);
  const bool once = pl->row1_grid != 0;  // else work-groups walk the chunks
  const long long chunk = 256ll * (once ? row_once_unroll(szA, szB, (int)V, szB == 1, pl->row1_unaligned != 0) : kRowUnroll);
  const long long chunks = once ? pl->row1_grid : pl->p.ntiles;
  CHECK(chunks * chunk >= (long long)p.total && (chunks - 1) * chunk < (long long)p.total);
  return true;
}

int main() {
  long long plans = 0, unaligned = 0, last = 0, small = 0;
  for (int ta = 0; ta < 8; ++ta)
    for (int tb = 0; tb < 8; ++tb) {
      if (!pair_supported(ta, tb)) continue;
      for (int beta = 0; beta < 2; ++beta) {
        if (beta && dtype_bytes(tb) == 1) continue;
        for (int i = 0; i < 80; ++i) {
          const bool huge = i >= 70;
          const int n0 = huge ? INT_MAX - (79 - i) : i + 1;
          // one row; a row of two fused dimensions; rows of their own
          const int perm1[] = {0}, size1[] = {n0}, perm2[] = {0, 1}, size2[] = {n0 / 2, 2};
          const int perm3[] = {0, 2, 1}, size3[] = {n0, 3, 5};
          struct { int dim; const int *perm, *size; int n0; long long rows; } cases[] = {
              {1, perm1, size1, n0, 1}, {2, perm2, size2, n0 / 2 * 2, 1}, {3, perm3, size3, n0, 15}};
          for (auto& c : cases) {
            if (c.n0 < (c.dim == 3 ? 2 : 1) || (huge && c.dim == 3)) continue;
            ttc_plan_t pl = nullptr;
            if (ttc_plan_create(&pl, (ttc_dtype_t)ta, (ttc_dtype_t)tb, c.dim, c.perm, c.size, nullptr, nullptr, !beta,
                                nullptr) != TTC_SUCCESS)
              return std::fprintf(stderr, "FAIL plan %d %d %d\n", ta, tb, n0), 1;
            for (const ttc_plan_s* q : {(const ttc_plan_s*)pl, (const ttc_plan_s*)pl->fallback})
              if (q) {
                if (!check_row(q, ta, tb, beta, c.n0, c.rows, unaligned, small)) return 1;
                ++plans;
                last += huge && q->row1_unaligned;
              }
            ttc_plan_destroy(pl);
          }
        }
      }
    }
  std::printf("%lld plans, %lld unaligned, %lld of them near 2^31, %lld in few bytes\n", plans, unaligned, last, small);
  return 0;
}
