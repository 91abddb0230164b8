// Grouped launch of one work-group per tile: every op whose tile the
// lane-fixed walk takes (ttc_lane.hpp) and every row copy, whatever their
// types, in ONE kernel.  A work-group looks up its op, then runs that op's
// instance (type, vector widths, beta read or not) on one tile or one chunk.
//
// Bound by HBM on large ops, by the one launch's latency on small ones.
// Against one persistent kernel per (family, type), one after the other on
// the stream: 26 ops of up to 0.3 MiB 54 -> 8 us, 30 ops of up to 2.2 MiB (17
// MB) 59 -> 17 us, 64 ops of up to 64 MiB (1.03 GB) 327 -> 212 us.
#pragma once
#include <hip/hip_runtime.h>

#include <type_traits>

#include "ttc_batch_kernels.hpp"
#include "ttc_lane.hpp"
#include "ttc_row.hpp"

namespace ttc {

// variant of a type's instances:
//   0 .. 17   row x column: (index_a * 3 + index_b) * 2 + beta_is_zero
//   18 .. 23  row copy, aligned vectors: 18 + index * 2 + beta_is_zero
//   24 .. 31  row copy, unaligned vectors of 2^k elements: 24 + k * 2 + beta_is_zero
// (index: of the vector width in {1, 2, widest}); kind = type pair * 32 + variant.
constexpr int kOneVariants = 32, kOneRow = 18, kOneRowUnaligned = 24;

// Op records, read with scalar loads: what both kinds of op have, then the
// row x column or the row copy's parameters.
struct OneHead {
  const void* A;
  void* B;
  double alpha, beta;
  int32_t kind;
  int32_t pad_[3];
};
// (1 KiB each, so that no record shares a line with another.)
struct alignas(64) OneLane {
  OneHead h;
  RCLaneParams p;
  unsigned char pad_[1024 - sizeof(OneHead) - sizeof(RCLaneParams)];
};
struct OneRow {
  OneHead h;
  RowParams p;
};
// Per op, in launch order: its first tile, and its record among those of its
// kind, with kOneIsRow for row copies.
struct OneIndex {
  uint32_t first, rec;
};
constexpr uint32_t kOneIsRow = 1u << 31;

static_assert(sizeof(OneLane) == 1024 && sizeof(OneRow) == 296, "bytes per op of the work table");
static_assert(alignof(OneLane) <= kTableAlign && alignof(OneRow) <= kTableAlign && alignof(OneIndex) <= kTableAlign,
              "the sections of a work table start at multiples of kTableAlign");
// Parameter records enter the table whole and are read in place: no field can
// be left behind.
static_assert(std::is_trivially_copyable<OneLane>::value && std::is_trivially_copyable<OneRow>::value,
              "records are copied as bytes");

// Tiles per entry of the table that gives the op a block of tiles starts in.
constexpr uint32_t kOneBlock = 64;

using KHead = const __attribute__((address_space(4))) OneHead;
using KOneLane = const __attribute__((address_space(4))) OneLane;
using KOneRow = const __attribute__((address_space(4))) OneRow;

// The launch's tile of work-group w: rounds of 2048 tiles, in which each XCD
// takes 256 consecutive ones, so that neighbours meet in one L2 and every XCD
// gets its share of each op.
TTC_HD inline uint32_t one_tile_of(uint32_t w, uint32_t ntiles) {
  constexpr uint32_t kRound = 2048, kPer = kRound / kXcds;
  const uint32_t base = w / kRound * kRound, l = w - base;
  return base + kRound <= ntiles ? base + l % kXcds * kPer + l / kXcds : w;
}

template <class OP, int W, int I>
__device__ __forceinline__ void one_variant(KHead* o, uint32_t tile, unsigned char* lds) {
  using TA = typename OP::TA;
  using TB = typename OP::TB;
  constexpr bool BETA = (I & 1) == 0;
  if constexpr (I < kOneRow) {
    constexpr int ia = I / 6, ib = (I / 2) % 3;
    if constexpr (index_used(ia, W) && index_used(ib, W))
      RCLane<OP, width_of_index(ia, W), width_of_index(ib, W), BETA, false, 2>::run(
          (KLane*)&((KOneLane*)o)->p, tile, static_cast<const TA*>(o->A), static_cast<TB*>(o->B), lds,
          (typename OP::AL)o->alpha, (typename OP::BE)o->beta, [](float) {});
  } else {
    constexpr bool UNAL = I >= kOneRowUnaligned;
    constexpr int V = UNAL ? 1 << (I - kOneRowUnaligned) / 2 : width_of_index((I - kOneRow) / 2, W);
    constexpr bool used = UNAL ? V >= 2 && V * (int)sizeof(TA) <= 16 && (!BETA || sizeof(TA) <= 2)
                               : index_used((I - kOneRow) / 2, W);
    if constexpr (used)
      (void)row_chunk<OP, V, BETA ? kModeBeta : kModeBz, UNAL>(
          ((KOneRow*)o)->p, tile, static_cast<const TA*>(o->A), static_cast<TB*>(o->B), (typename OP::AL)o->alpha,
          (typename OP::BE)o->beta, 1.0f);
  }
}

template <class OP, int W>
__device__ __forceinline__ void one_type(int variant, KHead* o, uint32_t tile, unsigned char* lds) {
  switch (variant) {
#define TTC_ONE(I) \
  case I: one_variant<OP, W, I>(o, tile, lds); break;
#define TTC_ONE4(I) TTC_ONE(I) TTC_ONE(I + 1) TTC_ONE(I + 2) TTC_ONE(I + 3)
    TTC_ONE4(0) TTC_ONE4(4) TTC_ONE4(8) TTC_ONE4(12) TTC_ONE4(16) TTC_ONE4(20) TTC_ONE4(24) TTC_ONE4(28)
#undef TTC_ONE4
#undef TTC_ONE
    default: break;
  }
}

// lanes, rows: the records; index: the ops, by kind; block: the op that holds
// tile kOneBlock * i, per i.
__global__ void __launch_bounds__(kThreads)
    batch_one_kernel(const OneLane* __restrict__ lanes, const OneRow* __restrict__ rows,
                     const OneIndex* __restrict__ index, const uint32_t* __restrict__ block, uint32_t nops,
                     uint32_t ntiles);

// Defined in ttc_batch_k_one.hip.
const void* batch_one_func();

}  // namespace ttc
