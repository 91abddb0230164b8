// Launch parameters shared by the host planner (ttc_plan.cpp) and the device
// kernels (ttc_kernels.hpp).  Plain C++ so the planner builds without HIP.
//
// Geometry is that of the FUSED problem: rank r <= TTC_MAX_DIM, A-dimension k
// has extent n[k], element stride sa in A and sb in B.  A tile is the box
// t[0] x ... x t[r-1] (t[k] == 1 for dimensions the grid walks over, t[k] ==
// n[k] for dimensions a tile covers fully, 1 < t[k] < n[k] for "split"
// dimensions).  Tiles are numbered in A order (dimension 0 fastest) over the
// tile grid g[k] = ceil(n[k] / t[k]).
#pragma once
#include <stdint.h>

#ifdef __HIPCC__
#define TTC_HD __host__ __device__
#else
#define TTC_HD
#endif

namespace ttc {

constexpr int kMaxDim = 8;     // fused rank limit
constexpr int kThreads = 256;  // work-group size (4 wave64)
constexpr int kRcThreads = 256;  // work-group size of the row x column kernels

// Vectors a thread owns per tile side for vectors of `vec` elements of
// `bytes` bytes: as many as fit 64 bytes of data (16 VGPRs), between 4 and
// 16.  A tile holds at most kThreads * slots_for(vec, bytes) * vec elements
// on each side; planner and kernels use this one rule.
constexpr int slots_for(int vec, int bytes) {
  return 64 / (vec * bytes) > 16 ? 16 : (64 / (vec * bytes) < 4 ? 4 : 64 / (vec * bytes));
}

// n / d for n < 2^31 via one multiply-high (round-up method): with
// s = ceil(log2 d) and m = floor(2^32 (2^s - d) / d) + 1,
// n / d = (mulhi(n, m) + n) >> s.
struct FastDiv {
  uint32_t d, m, s, pad_;
};

inline FastDiv make_fastdiv(uint32_t d) {
  FastDiv f{};
  f.d = d;
  uint32_t s = 0;
  while ((1ull << s) < d) ++s;
  f.s = s;
  f.m = (uint32_t)(((1ull << 32) * ((1ull << s) - d)) / d + 1);
  return f;
}

TTC_HD inline uint32_t fdiv(uint32_t n, uint32_t m, uint32_t s) {
  return ((uint32_t)(((uint64_t)n * m) >> 32) + n) >> s;
}
TTC_HD inline uint32_t fdiv(uint32_t n, const FastDiv& f) { return fdiv(n, f.m, f.s); }

// FastDiv without its padding.
struct DivBy {
  uint32_t d, m, s;
};
inline DivBy make_divby(uint32_t d) {
  const FastDiv f = make_fastdiv(d);
  return DivBy{f.d, f.m, f.s};
}

// Work-groups are dispatched round-robin over the 8 XCDs (work-group w runs
// on XCD w % 8), each XCD with its own L2.
constexpr uint32_t kXcds = 8;

struct TileParams {
  int32_t rank;
  int32_t V;            // elements in a full tile (prod t)
  int32_t t[kMaxDim];   // tile extents
  int32_t n[kMaxDim];   // tensor extents
  int32_t perm[kMaxDim];       // B position q holds A dimension perm[q]
  int32_t sa[kMaxDim];         // A element stride of dim k, used within a tile (int32 checked on host)
  int32_t sb[kMaxDim];         // B element stride of dim k, used within a tile
  int32_t ls[kMaxDim];         // LDS element stride of dim k
  int64_t tsa[kMaxDim];        // t[k] * A stride: tile-to-tile step
  int64_t tsb[kMaxDim];        // t[k] * B stride
  FastDiv tdiv[kMaxDim];       // division by t[k]
  FastDiv gdiv[kMaxDim];       // division by g[k] (tiles along dim k)
  // The same quantities in B order (position q describes A dimension
  // perm[q]), so that device code never indexes this struct with a value
  // known only at run time (that would force a copy into scratch memory).
  FastDiv tdivB[kMaxDim];
  int32_t tB[kMaxDim];
  int32_t sbB[kMaxDim];
  int32_t lsB[kMaxDim];
  int32_t splitB0, splitB1;    // B positions of split0 / split1 (-1 = none)
  // Digit of a split dimension in a tile-linear index l (A or B order):
  // (l / P) mod t, P = product of the tile extents before it in that order.
  FastDiv pA0, pA1, pB0, pB1;  // division by P
  FastDiv ts0, ts1;            // division by t[split]
  uint32_t ntiles;
  int32_t split0, split1;      // dims with partial tiles (-1 = none)
  int32_t tsplit0, tsplit1;    // t[split] (0 when none)
  int32_t lds_stride_b;        // ls[perm[0]]: LDS distance of consecutive B-order elements
  int32_t lds_elems;           // LDS elements used by one tile (with padding)
  int32_t grid_order;          // tile_range order: 0 strided, 1 contiguous, 2 XCD-grouped, 3 XCD shares
};

// Row x column tile (ttc_rc.hpp): the tile's dimensions split into an A
// group (A's leading dimensions, the rows) and a disjoint B group (B's
// leading dimensions, the columns); only the outermost dimension of each
// group may have a partial last tile.
struct RCParams {
  int32_t R, C;          // rows (A-group volume) and columns (B-group volume) of a full tile
  int32_t Rl, Cl;        // rows / columns of the last tile along the split dims (== R / C if none)
  FastDiv dR, dRl, dC, dCl;
  int32_t RP;            // LDS pitch of a column (R | 1)
  int32_t rowA_dense;    // rowA[i] == i * sizeof(TA): the rows are one contiguous run of A
  int32_t colB_dense;    // colB[j] == j * sizeof(TB): the columns are one contiguous run of B
  int32_t na, nb;        // dimensions in the A group / B group
  int32_t ta[kMaxDim];   // tile extents of the A group, A order
  FastDiv dta[kMaxDim];
  int32_t saA[kMaxDim], sbA[kMaxDim];  // A and B byte strides of the A-group dims
  int32_t tb[kMaxDim];   // tile extents of the B group, B order
  FastDiv dtb[kMaxDim];
  int32_t saB[kMaxDim], sbB[kMaxDim];  // A and B byte strides of the B-group dims
  // Tile grid: only the dimensions with more than one tile, in walk order
  // (A order or B order); position g describes one such dimension.
  int32_t grank;
  int32_t n[kMaxDim], t[kMaxDim];
  FastDiv gdiv[kMaxDim];   // division by the number of tiles along the dimension
  int64_t tsa[kMaxDim], tsb[kMaxDim];  // element offset of the next tile along it, in A and B
  int32_t splitA, splitB;  // grid positions of the row group's / column group's partial dimension (-1 none)
  // Grouped walk: one dimension is split into an inner position 0 of
  // `group` tiles and an outer position `gouter` (-1: no split); `gcount`
  // is its number of real tiles, ids past it are empty padding.
  int32_t gouter;
  uint32_t group, gcount;
  int32_t nbuf;            // LDS tile buffers: 2 lets a tile's staging overlap the previous tile's reads
  uint32_t ntiles;         // grid size (with the padding of a grouped walk)
  int32_t grid_order;
  int32_t lds_data_elems;  // tile data region in LDS elements (both walks' reach, a spare vector slot, 16-byte rounding)
  int32_t lds_spare;       // RP * C: where lanes past a partial tile stage their (unused) values
  // Lane-fixed walk of full tiles (fast != 0).  The read walk runs over Rw
  // rows (R rounded up to a power of two that divides the walk step 256 *
  // VA), so a lane keeps one row i for the whole tile and its slot `it`
  // takes column j0 + it * kA; the write walk mirrors it over Cw columns
  // with row step kB.  Positions past R or C read offset tables holding
  // kRcTabOOB, which sends the access out of the buffer range, and stage
  // into the spare slot (lds_spare), so no per-slot bounds test remains.
  // Partial and empty tiles take the general walk.
  int32_t fast;
  int32_t Rw, Cw;          // walk extents (powers of two >= R, C); R, C when fast == 0
  int32_t Rw_shift, Cw_shift;
  int32_t kA, kB;          // column step of the read walk, row step of the write walk
  int32_t nia, nib;        // slots per lane of the read and write walks (rc_elems / vector width)
  int32_t ntab;            // offset-table entries in LDS (layout below)
  int32_t pad_;
};

// LDS offset tables of a row x column launch, int32 byte offsets after the
// tile data: rowA[Rw] rowB[R] colA[C] colB[Cw], then (fast walk only)
// colS[kA * NIA] and rowS[kB * NIB], the read walk's column offsets and the
// write walk's row offsets in slot order (colS[jl * NIA + it] = colA[jl + it
// * kA]); entries past R or C hold kRcTabOOB.  On a side whose walk has such
// slots a table entry is below 2^30 - 64, so the sum of two entries is
// either a real offset (< 2^31) or, if either is kRcTabOOB, in [2^31, 2^32):
// past the buffer range 2^31.  A side without them holds real offsets only,
// whose sums stay below 2^31 (the tile's span).
constexpr uint32_t kRcTabOOB = 0xC0000000u;
constexpr long long kRcFastSpan = (1ll << 30) - 64;

// Order in which a single-op launch hands out its row x column tiles.
struct RCWalk {
  uint32_t ntiles;     // tiles of the launch (no padding ids)
  int32_t grid_order;  // as RCParams::grid_order
  // Bands: the walk's dimension of `bandn` tiles with `bandin` tiles before
  // it runs in bands of `bandw` tiles (the last one narrower), each band's
  // tiles innermost.  bandw 0: no bands.
  uint32_t bandw, bandn, bandin;
  FastDiv dper, dband, dw, dwl;  // divisions by bandn * bandin, bandw * bandin, bandw, the last band's width
};

// Tile of work-group w: a permutation of [0, ntiles).
// grid_order 3: XCD x (work-groups w % 8 == x) takes a contiguous share of
// the tile numbering, so that the tiles in flight on one L2 are neighbours;
// 2: the same within rounds of 512 tiles; otherwise tile w.  Then the bands:
// tiles of a band neighbour each other on A's side and, one band's pass after
// the other, on B's, so both sides' shared cache lines meet in the L2.
TTC_HD inline uint32_t rc_tile_of(const RCWalk& p, uint32_t w) {
  uint32_t id = w;
  if (p.grid_order == 3) {
    const uint32_t x = w % kXcds, q = p.ntiles / kXcds, rem = p.ntiles % kXcds;
    id = x * q + (x < rem ? x : rem) + w / kXcds;
  } else if (p.grid_order == 2) {
    constexpr uint32_t kRound = 512, kPer = kRound / kXcds;
    const uint32_t base = w / kRound * kRound, l = w - base;
    if (base + kRound <= p.ntiles) id = base + l % kXcds * kPer + l / kXcds;
  }
  if (p.bandw) {
    const uint32_t hi = fdiv(id, p.dper);
    uint32_t r = id - hi * p.dper.d;
    const uint32_t b = fdiv(r, p.dband);
    r -= b * p.dband.d;
    const bool last = (b + 1) * p.bandw > p.bandn;
    const uint32_t low = last ? fdiv(r, p.dwl) : fdiv(r, p.dw);
    const uint32_t x = b * p.bandw + (r - low * (last ? p.dwl.d : p.dw.d));
    id = low + p.bandin * (x + p.bandn * hi);
  }
  return id;
}

// One dimension of a tile's row or column group, and one tiled dimension of
// the tile grid, in the single-op launches.
struct RCDim {
  uint32_t d, m, s;  // division by the tile extent (FastDiv)
  int32_t sa, sb;    // A and B byte strides
};
struct RCGridDim {
  uint32_t d, m, s;  // division by the tiles along the dimension
  uint32_t part;     // 1 / 2: its last tile is partial in the row / column group
  int64_t tsa, tsb;  // element offset of the next tile along it, in A and B
};

// Single-op row x column launch (ttc_rc.hpp, RCLane): each lane keeps one
// vector of rows of the read walk (lane tid: column jl + it * kA of slot it,
// jl = tid / la, rows (tid % la) * VA ...) and one vector of columns of the
// write walk (row il + it * kB, il = tid / lb, columns (tid % lb) * VB ...).
// Everything a tile needs besides is two slot-ordered offset tables.  The
// records in use lie together at the front of dim and grid: the kernel reads
// them from the kernel arguments with scalar loads.
struct RCLaneParams {
  int32_t R, C;        // rows and columns of a full tile
  int32_t Rl, Cl;      // of the last tile along the split dimensions
  int32_t RP;          // LDS pitch of a column (R | 1)
  int32_t kA, kB;      // column step of the read walk, row step of the write walk
  uint32_t kAm, kAs, kBm, kBs;  // divisions by them
  uint32_t la, lam, las;  // division by R / VA (lanes per column)
  uint32_t lb, lbm, lbs;  // division by C / VB (lanes per row)
  int32_t spare;       // LDS element where lanes past the walk stage (VA elements)
  int32_t tab;         // byte offset of the tables in LDS: colS[kA * NIA] rowS[kB * NIB] rowA[R] colB[C]
  int32_t na, nb;      // dimensions of the row group, the column group
  int32_t grank;       // tiled grid dimensions, in walk order
  RCWalk walk;
  RCDim dim[kMaxDim];  // row group, then column group
  RCGridDim grid[kMaxDim];
};

// Elements per thread per tile side of the row x column kernels: as many as
// fit 128 bytes, at most 32.
constexpr int rc_elems(int bytes) { return 128 / bytes > 32 ? 32 : 128 / bytes; }

// Row copy for perm[0] == 0, where A and B share the stride-1 dimension:
// a row is one position of the other dimensions, the rows are walked in B
// order, and each lane moves one vector of V elements of dimension 0.
constexpr int kRowUnroll = 4;  // vectors in flight per lane in the row-copy kernel

// Rows of n0 >= v elements in unaligned vectors of v: vectors per row, and how
// far the one that would start at element e is shifted back to end with its
// row.  n0 may lie within v of 2^31: neither n0 + v nor e + v fits an int32.
TTC_HD inline uint32_t row_vectors(int32_t n0, int32_t v) { return ((uint32_t)n0 + (uint32_t)v - 1u) / (uint32_t)v; }
TTC_HD inline int32_t row_shift(int32_t e, int32_t v, int32_t n0) { return e > n0 - v ? e - (n0 - v) : 0; }

// A row copy: kernel argument, and record of a grouped launch's work table.
struct RowParams {
  uint32_t total;         // rows * nv (< 2^31)
  uint32_t nv;            // vectors per row: extent of dimension 0 / V (rounded up on unaligned vectors)
  int32_t n0;             // extent of dimension 0
  int16_t rank;           // row dimensions, in B order
  int16_t xcd_share;      // one chunk per work-group: XCDs take contiguous shares of the chunks (grouped launches:
                          // not read)
  uint32_t nvm, nvs;      // division by nv
  DivBy dn[kMaxDim];      // their extents
  int64_t sa[kMaxDim];    // A byte strides
  int64_t sb[kMaxDim];    // B byte strides
};
inline void row_set_vectors(RowParams& p, uint32_t rows, uint32_t nv) {
  const FastDiv f = make_fastdiv(nv);
  p.total = rows * nv, p.nv = nv, p.nvm = f.m, p.nvs = f.s;
}

// One row x column tile of a grouped launch: element offsets of its origin
// in A and B; flags bit 0: last (partial) tile along the row group, bit 1:
// along the column group.
struct RCTile {
  int64_t a, b;
  uint32_t flags, pad_;
};

// Launches of few dimensions in few bytes of arguments: with at most 112
// (kSmallArgs and A, B, alpha, beta) the host's part of a launch takes 3.0 us,
// with 160 to 992 3.1-3.4 (an empty kernel), and the kernel reads two lines of
// arguments instead of up to ten.  Tiles, and vectors of rows, are counted
// below 2^20, so that divisions go through floats (sdiv).  A tile's chain of
// divisions is longer than with FastDiv's constants: tiles take this form up
// to kSmallBytes read and written, where the host is what a sequence of calls
// waits for (fp32 1024 x 1024, 8 MiB: 4.5 -> 4.3 us per call, fp64 37 x 21 x 19
// x 5 4.5 -> 4.3; complex64 96 x 80 x 110, 13 MB, 4.88 -> 4.98, fp32 2048 x 1024
// 5.03 -> 5.10).  Rows take it wherever it fits (fp32 rows of 64, 31 MB: 5.1 ->
// 4.8).
constexpr uint32_t kSmallCount = 1u << 20;
constexpr long long kSmallBytes = 8ll << 20;
constexpr int kSmallArgs = 80, kSmallDims = 4, kSmallRowDims = 5;

// n / d for n < 2^20: (n + 1/2) / d is at least 1 / 2d off every integer, the
// error of the product below 2^-21 * n / d (a reciprocal within 1 ulp).
TTC_HD inline uint32_t sdiv_by(uint32_t n, float inv) { return (uint32_t)(((float)n + 0.5f) * inv); }
TTC_HD inline uint32_t sdiv(uint32_t n, uint32_t d) {
#ifdef __HIP_DEVICE_COMPILE__
  return sdiv_by(n, __builtin_amdgcn_rcpf((float)d));
#else
  return sdiv_by(n, 1.0f / (float)d);
#endif
}

struct RCSmallDim {
  int32_t sa, sb;  // A and B byte strides
  uint16_t d, n;   // tile extent, tiles along the dimension
};
// RCLaneParams (which see) of up to kSmallDims dimensions.
struct RCLaneSmall {
  uint32_t ntiles;
  uint16_t R, C, Rl, Cl, kA, kB;
  uint16_t tab16, spare;   // byte offset of the tables / 16
  uint32_t bandin_w;       // RCWalk::bandin, bandw << 24
  uint16_t bandn;
  uint8_t grid_order, groups;  // na, nb << 4
  uint16_t grid;           // walk order: a nibble per tiled dimension, index in dim | RCGridDim::part << 2
  uint8_t grank, pad_;
  RCSmallDim dim[kSmallDims];  // row group, column group, other dimensions
};
static_assert(sizeof(RCLaneSmall) == kSmallArgs, "kernel arguments");

// rc_tile_of, and the tile's origin: byte offsets and partial groups (bits of
// RCGridDim::part).  P: a pointer to the parameters, in any address space.
template <class P> TTC_HD inline uint32_t rc_small_tile_of(P p, uint32_t w) {
  uint32_t id = w;
  const uint32_t nt = p->ntiles, order = p->grid_order;
  if (order == 3) {
    const uint32_t x = w % kXcds, q = nt / kXcds, rem = nt % kXcds;
    id = x * q + (x < rem ? x : rem) + w / kXcds;
  } else if (order == 2) {
    constexpr uint32_t kRound = 512, kPer = kRound / kXcds;
    const uint32_t base = w / kRound * kRound, l = w - base;
    if (base + kRound <= nt) id = base + l % kXcds * kPer + l / kXcds;
  }
  const uint32_t bandin = p->bandin_w & 0xffffffu, bandw = p->bandin_w >> 24, bandn = p->bandn;
  if (bandw) {
    const uint32_t per = bandn * bandin, band = bandw * bandin;
    const uint32_t hi = sdiv(id, per);
    uint32_t r = id - hi * per;
    const uint32_t b = sdiv(r, band);
    r -= b * band;
    const uint32_t wide = bandn - b * bandw < bandw ? bandn - b * bandw : bandw;
    const uint32_t low = sdiv(r, wide);
    id = low + bandin * (b * bandw + (r - low * wide) + bandn * hi);
  }
  return id;
}
template <class P> TTC_HD inline uint32_t rc_small_origin(P p, uint32_t w, int64_t& oa, int64_t& ob) {
  uint32_t rem = rc_small_tile_of(p, w), last = 0, map = p->grid;
  oa = ob = 0;
  const int gr = p->grank;
#pragma unroll 1
  for (int g = 0; g < gr; ++g, map >>= 4) {
    const uint32_t k = map & 3u, n = p->dim[k].n, q = sdiv(rem, n), x = rem - q * n;
    rem = q;
    oa += (int64_t)(x * p->dim[k].d) * p->dim[k].sa;
    ob += (int64_t)(x * p->dim[k].d) * p->dim[k].sb;
    if (x == n - 1) last |= map >> 2 & 3u;
  }
  return last;
}
// Byte offsets of position l of a group (of n dimensions from `first` on).
template <class P>
TTC_HD inline void rc_small_offsets(P p, int first, int n, uint32_t l, int32_t& oa, int32_t& ob) {
  oa = ob = 0;
#pragma unroll 1
  for (int m = first; m < first + n; ++m) {
    const uint32_t d = p->dim[m].d, q = sdiv(l, d);
    const int32_t x = (int32_t)(l - q * d);
    l = q;
    oa += x * p->dim[m].sa;
    ob += x * p->dim[m].sb;
  }
}

// RowParams of up to kSmallRowDims row dimensions.
struct RowSmallDim {
  int32_t sa, sb;  // byte strides
  uint32_t d;
};
struct RowSmall {
  uint32_t total, nv;
  int32_t n0;
  uint16_t rank, xcd_share;
  RowSmallDim dim[kSmallRowDims];
  uint32_t grid;
};
static_assert(sizeof(RowSmall) == kSmallArgs, "kernel arguments");

// One-chunk-per-work-group row copy (row_once_kernel): vectors in flight per
// lane.  16-byte vectors: one, so that a launch has the most work-groups (200
// MiB fp32: 6.0 TB/s with one, 5.7 with two, 5.6 with four); unaligned ones
// and those of 8 bytes: two (fp64 rows of 447 with beta, 1.3 GB: 250 us with
// one, 240, 253 with four); of 4 bytes and less: four (fp32 rows of 127 with
// beta, 422 MB: 106, 116, 92; of 9: 73, 70, 62); fp8 casts: four (fp32 128 x
// 4096 x 32 x 8: 159 us with one, 143, 135).
constexpr int row_once_unroll(int bytes_a, int bytes_b, int v, bool fp8, bool unaligned) {
  const int bytes = v * (bytes_a > bytes_b ? bytes_a : bytes_b);
  return fp8 ? 4 : unaligned ? 2 : bytes >= 16 ? 1 : bytes >= 8 ? 2 : 4;
}

// Which units (tiles, chunks) a work-group of an fp8 cast takes.  Without
// amax one each.  With it the first kAmaxHead work-groups take one unit and
// the others two consecutive ones: the head's maxima, committed while the
// others still work, leave few of those with anything to commit (bf16 1024 x
// 4096, 1024 tiles: 17.9 us with one tile each, 10.1 so; 6.3 without amax).
// Three and more cost locality (bf16 8192 x 14336: one 84, two 75, four 79 us;
// fp32: 121, 120, 138). Up to 256 units each commits its own.  (Work-group w
// runs on XCD w % 8: with two units each the XCDs' shares of the walk
// interleave, which these times include.)
constexpr uint32_t kAmaxHead = 64;
struct AmaxUnits {
  uint32_t n, per;
  TTC_HD uint32_t first(uint32_t wg) const {
    if (wg <= kAmaxHead) return wg < n ? wg : n;
    const uint64_t u = kAmaxHead + (uint64_t)(wg - kAmaxHead) * per;
    return u < n ? (uint32_t)u : n;
  }
  uint32_t work_groups() const { return n <= kAmaxHead ? n : kAmaxHead + (n - kAmaxHead + per - 1) / per; }
};
inline AmaxUnits amax_units(uint32_t n, bool amax) {
  return AmaxUnits{n, !amax || n <= 256 ? 1u : 2u};
}

}  // namespace ttc
