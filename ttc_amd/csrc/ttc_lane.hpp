// Row x column tiles, one tile per work-group: the single-op launch of the
// row x column family (tile, row and column groups as in ttc_rc.hpp).
//
// Bound by HBM.  The dispatcher starts the next tile on whichever CU frees a
// slot first, so the tiles in flight stay neighbours in the walk order
// (rc_tile_of) and the cache lines they share at their edges are fetched and
// written back once; work-groups that stride over many tiles each (the
// pipelined kernel of ttc_rc.hpp) drift apart and lose that.  Time per
// launch, pipelined -> one tile per work-group (copy of 200 MiB: 5.9 TB/s):
//   fp32 6507 x 8057, padded              110 -> 94 us  (4.5 TB/s)
//   fp32 rank 6, odd extents, 200 MiB     131 -> 102    (4.1)
//   fp64 rank 5, beta = 1, 200 MiB        133 -> 118    (5.3)
//   fp32 -> bf16 rank 4 with beta, 2.4 GB 1129 -> 950   (5.1)
//   complex64 96 x 80 x 110               6.3 -> 4.9
//   fp64 37 x 21 x 19 x 5, beta = 1       7.5 -> 4.4 (in few bytes of arguments)
//
// Each lane keeps one vector of rows for the whole read walk and one vector
// of columns for the whole write walk (RCLaneParams), for any row and column
// count: a slot costs one table entry and one add on each side, and partial
// tiles, lanes past the walk and slots past the tile are entries of
// kRcTabOOB, which send the access out of the buffer range.  The code is a
// few KB: a small launch waits for its instructions, so straight-line code
// for every case would cost more than it saves.
#pragma once
#include <type_traits>

#include "ttc_rc.hpp"

namespace ttc {

using KLane = const __attribute__((address_space(4))) RCLaneParams;
using KLaneSmall = const __attribute__((address_space(4))) RCLaneSmall;

// Where a tile's parameters come from: the same members over both forms.
struct LaneFull {
  KLane* kp;
  __device__ __forceinline__ void touch() const { touch_lines<sizeof(RCLaneParams)>(kp); }
  // offsets of tile `wg`'s origin (elements here; what `at` adds), and which
  // groups are partial
  __device__ __forceinline__ uint32_t origin(uint32_t wg, int64_t& bA, int64_t& bB) const {
    RCWalk w;  // copied whole, as 32-bit words: no field can be left behind
    static_assert(sizeof(RCWalk) % 4 == 0 && std::is_trivially_copyable<RCWalk>::value, "RCWalk is copied as words");
    KWord* const s = (KWord*)&kp->walk;
    uint32_t* const d = reinterpret_cast<uint32_t*>(&w);
#pragma unroll
    for (int i = 0; i < (int)(sizeof(RCWalk) / 4); ++i) d[i] = s[i];
    uint32_t rem = uniform(rc_tile_of(w, wg)), last = 0;
    bA = bB = 0;
    const int gr = kp->grank;
#pragma unroll 1
    for (int g = 0; g < gr; ++g) {
      const uint32_t d = kp->grid[g].d, q = fdiv(rem, kp->grid[g].m, kp->grid[g].s), x = rem - q * d;
      rem = q;
      bA += (int64_t)x * kp->grid[g].tsa;
      bB += (int64_t)x * kp->grid[g].tsb;
      if (x == d - 1) last |= kp->grid[g].part;
    }
    return last;
  }
  template <class T> __device__ __forceinline__ static T* at(T* p, int64_t b) { return p + uniform64(b); }
  // Offsets of position l of a group: mixed-radix digits over its tile
  // extents times their byte strides.
  __device__ __forceinline__ void offsets(int first, int n, uint32_t l, int32_t& oa, int32_t& ob) const {
    oa = ob = 0;
#pragma unroll 1
    for (int m = first; m < first + n; ++m) {
      const uint32_t d = kp->dim[m].d, q = fdiv(l, kp->dim[m].m, kp->dim[m].s);
      const int32_t x = (int32_t)(l - q * d);
      l = q;
      oa += x * kp->dim[m].sa;
      ob += x * kp->dim[m].sb;
    }
  }
  __device__ __forceinline__ uint32_t RP() const { return (uint32_t)kp->RP; }
  __device__ __forceinline__ int na() const { return kp->na; }
  __device__ __forceinline__ int nb() const { return kp->nb; }
  __device__ __forceinline__ uint32_t tab() const { return (uint32_t)kp->tab; }
  __device__ __forceinline__ uint32_t by_kA(uint32_t j) const { return fdiv(j, kp->kAm, kp->kAs); }
  __device__ __forceinline__ uint32_t by_kB(uint32_t i) const { return fdiv(i, kp->kBm, kp->kBs); }
  template <int VA> __device__ __forceinline__ uint32_t la() const { return kp->la; }
  template <int VB> __device__ __forceinline__ uint32_t lb() const { return kp->lb; }
  __device__ __forceinline__ uint32_t by_la(uint32_t t, uint32_t) const { return fdiv(t, kp->lam, kp->las); }
  __device__ __forceinline__ uint32_t by_lb(uint32_t t, uint32_t) const { return fdiv(t, kp->lbm, kp->lbs); }
};

struct LaneSmall {
  KLaneSmall* kp;
  __device__ __forceinline__ void touch() const { touch_lines<sizeof(RCLaneSmall)>(kp); }
  __device__ __forceinline__ uint32_t origin(uint32_t wg, int64_t& bA, int64_t& bB) const {
    return rc_small_origin(kp, wg, bA, bB);
  }
  template <class T> __device__ __forceinline__ static T* at(T* p, int64_t b) {
    return reinterpret_cast<T*>(const_cast<char*>(reinterpret_cast<const char*>(p)) + uniform64(b));
  }
  __device__ __forceinline__ void offsets(int first, int n, uint32_t l, int32_t& oa, int32_t& ob) const {
    rc_small_offsets(kp, first, n, l, oa, ob);
  }
  __device__ __forceinline__ uint32_t RP() const { return (uint32_t)kp->R | 1u; }
  __device__ __forceinline__ int na() const { return kp->groups & 15; }
  __device__ __forceinline__ int nb() const { return kp->groups >> 4; }
  __device__ __forceinline__ uint32_t tab() const { return (uint32_t)kp->tab16 * 16u; }
  __device__ __forceinline__ uint32_t by_kA(uint32_t j) const { return sdiv(j, kp->kA); }
  __device__ __forceinline__ uint32_t by_kB(uint32_t i) const { return sdiv(i, kp->kB); }
  template <int VA> __device__ __forceinline__ uint32_t la() const { return (uint32_t)kp->R / VA; }
  template <int VB> __device__ __forceinline__ uint32_t lb() const { return (uint32_t)kp->C / VB; }
  __device__ __forceinline__ uint32_t by_la(uint32_t t, uint32_t la) const { return sdiv(t, la); }
  __device__ __forceinline__ uint32_t by_lb(uint32_t t, uint32_t lb) const { return sdiv(t, lb); }
};

template <class OP, int VA, int VB, bool BETA, bool NT, int DIV>
struct RCLane {
  using TA = typename OP::TA;
  using TB = typename OP::TB;
  using L = typename OP::L;
  static constexpr int NIA = rc_elems((int)sizeof(TA)) / VA / DIV;  // read slots per lane
  static constexpr int NIB = rc_elems((int)sizeof(TB)) / VB / DIV;  // write slots per lane
  static constexpr bool FP8 = is_fp8<OP>::value;

  // The tile of work-group `wg` of the launch (of the op, in a grouped one).
  // after(amax): called between staging and the barrier with max |alpha * a|
  // of this lane's elements (fp8 casts).
  template <class F>
  __device__ __forceinline__ static void run(KLane* kp, uint32_t wg, const TA* __restrict__ A, TB* __restrict__ B,
                                             unsigned char* lds_raw, typename OP::AL alpha, typename OP::BE beta,
                                             F&& after) {
    run(LaneFull{kp}, wg, A, B, lds_raw, alpha, beta, after);
  }
  template <class SRC, class F>
  __device__ __forceinline__ static void run(const SRC src, uint32_t wg, const TA* __restrict__ A,
                                             TB* __restrict__ B, unsigned char* lds_raw, typename OP::AL alpha,
                                             typename OP::BE beta, F&& after) {
    const uint32_t tid = threadIdx.x;
    const auto kp = src.kp;
    src.touch();
    int64_t bA, bB;
    const uint32_t last = src.origin(wg, bA, bB);
    const int R = kp->R, C = kp->C, kA = kp->kA, kB = kp->kB, na = src.na();
    const int rows = (last & 1u) ? kp->Rl : R, cols = (last & 2u) ? kp->Cl : C;
    // tables: colS[jl * NIA + it] = A offset of column jl + it * kA, rowS its
    // mirror image for B; rowA and colB by row and column
    L* const data = reinterpret_cast<L*>(lds_raw);
    int32_t* const colS = reinterpret_cast<int32_t*>(lds_raw + src.tab());
    int32_t* const rowS = colS + kA * NIA;
    int32_t* const rowA = rowS + kB * NIB;
    int32_t* const colB = rowA + R;
    // (columns from the first wave on, rows from the last: each wave computes
    // one kind, or none)
    for (int j = (int)tid; j < kA * NIA; j += kRcThreads) {
      const uint32_t it = src.by_kA((uint32_t)j);
      int32_t* const slot = colS + (j - (int)it * kA) * NIA + it;
      if (j < C) {
        int32_t oa, ob;
        src.offsets(na, src.nb(), (uint32_t)j, oa, ob);
        *slot = j < cols ? oa : (int32_t)kRcTabOOB;
        colB[j] = j < cols ? ob : (int32_t)kRcTabOOB;
      } else {
        *slot = (int32_t)kRcTabOOB;
      }
    }
    for (int i = (int)(kRcThreads - 1 - tid); i < kB * NIB; i += kRcThreads) {
      const uint32_t it = src.by_kB((uint32_t)i);
      int32_t* const slot = rowS + (i - (int)it * kB) * NIB + it;
      if (i < R) {
        int32_t oa, ob;
        src.offsets(0, na, (uint32_t)i, oa, ob);
        *slot = i < rows ? ob : (int32_t)kRcTabOOB;
        rowA[i] = i < rows ? oa : (int32_t)kRcTabOOB;
      } else {
        *slot = (int32_t)kRcTabOOB;
      }
    }
    const uint32_t RP = src.RP();
    // this lane's place in the two walks
    const uint32_t la = src.template la<VA>(), lb = src.template lb<VB>();
    const uint32_t jl = src.by_la(tid, la), ai = (tid - jl * la) * VA;
    const uint32_t il = src.by_lb(tid, lb), bj = (tid - il * lb) * VB;
    const bool onA = jl < (uint32_t)kA, onB = il < (uint32_t)kB;
    const uint32_t sA = onA ? ai + jl * RP : (uint32_t)kp->spare, stepA = onA ? (uint32_t)kA * RP : 0u;
    const uint32_t sB = onB ? il + bj * RP : 0u, stepB = onB ? (uint32_t)kB : 0u;
    __syncthreads();
    const uint32_t rowoff = onA ? (uint32_t)rowA[ai] : kRcTabOOB, coloff = onB ? (uint32_t)colB[bj] : kRcTabOOB;
    const int32_t* const cs = colS + (onA ? jl * NIA : 0u);
    const int32_t* const rs = rowS + (onB ? il * NIB : 0u);
    const BufRes ra = make_res(SRC::at(A, bA)), rb = make_res(SRC::at(B, bB));
    TA va[NIA][VA];
    TB old[NIB][VB];
    uint32_t ob[NIB];
#pragma unroll
    for (int it = 0; it < NIA; ++it) bload<TA, VA>(va[it], ra, rowoff + (uint32_t)cs[it]);
#pragma unroll
    for (int it = 0; it < NIB; ++it) {
      ob[it] = (uint32_t)rs[it] + coloff;
      if constexpr (BETA) bload<TB, VB>(old[it], rb, ob[it]);
    }
    float amax = 0.0f;
#pragma unroll
    for (int it = 0; it < NIA; ++it) {
      L* const q = data + sA + (uint32_t)it * stepA;
#pragma unroll
      for (int v = 0; v < VA; ++v) {
        const L x = OP::prod(alpha, va[it][v]);
        if constexpr (FP8) amax = fmaxf(amax, fabsf(x));  // slots past the tile loaded zeros
        q[v] = x;
      }
    }
    after(amax);
    __syncthreads();
#pragma unroll
    for (int it = 0; it < NIB; ++it) {
      const L* const q = data + sB + (uint32_t)it * stepB;
      TB o[VB];
#pragma unroll
      for (int v = 0; v < VB; ++v) {
        if constexpr (FP8) {
          if constexpr (VB == 1) {
            o[0] = OP::outs(q[0], beta);
          } else if (v % 2 == 0) {
            OP::outs2(q[v * RP], q[(v + 1) * RP], beta, o[v], o[v + 1]);
          }
        } else if constexpr (BETA) {
          o[v] = OP::outb(q[v * RP], beta, old[it][v]);
        } else {
          o[v] = OP::out(q[v * RP]);
        }
      }
      bstore<TB, VB, NT>(rb, ob[it], o);
    }
  }
};

// The parameters are the kernel's first argument, so they sit at the start
// of the kernel-argument segment.
template <class OP, int VA, int VB, bool BETA, bool NT, int DIV>
__global__ void __launch_bounds__(kRcThreads)
    transpose_lane_kernel(const RCLaneParams p, const typename OP::TA* __restrict__ A,
                          typename OP::TB* __restrict__ B, double alpha, double beta) {
  extern __shared__ __align__(16) unsigned char lds_raw[];
  KLane* kp = (KLane*)__builtin_amdgcn_kernarg_segment_ptr();
  RCLane<OP, VA, VB, BETA, NT, DIV>::run(kp, blockIdx.x, A, B, lds_raw, (typename OP::AL)alpha, (typename OP::BE)beta,
                                         [](float) {});
}

template <class OP, int VA, int VB, bool BETA, bool NT, int DIV>
__global__ void __launch_bounds__(kRcThreads)
    transpose_small_kernel(const RCLaneSmall p, const typename OP::TA* __restrict__ A,
                           typename OP::TB* __restrict__ B, double alpha, double beta) {
  extern __shared__ __align__(16) unsigned char lds_raw[];
  const LaneSmall src{(KLaneSmall*)__builtin_amdgcn_kernarg_segment_ptr()};
  RCLane<OP, VA, VB, BETA, NT, DIV>::run(src, blockIdx.x, A, B, lds_raw, (typename OP::AL)alpha,
                                         (typename OP::BE)beta, [](float) {});
}

// fp8 cast-transpose (semantics: cast_fp8_rc_kernel).  Where amax is asked
// for, a work-group takes the tiles AmaxUnits gives it and commits their max
// once (amax_commit_one).  With amax_in, a pass over A has just run: the tiles
// are walked backwards, so that the part of A it read last is still in the
// last-level cache (amax and cast of bf16 8192 x 14336: 113 -> 108 us, fp32:
// 191 -> 184).
template <class OP, int VA, int VB, int DIV>
__global__ void __launch_bounds__(kRcThreads)
    cast_fp8_lane_kernel(const RCLaneParams p, const typename OP::TA* __restrict__ A,
                         typename OP::TB* __restrict__ B, float alpha, const float* __restrict__ scale_in,
                         const float* __restrict__ amax_in, float fp8_max, float scale_host,
                         float* __restrict__ amax_out, float* __restrict__ scale_inv_out, AmaxUnits units) {
  extern __shared__ __align__(16) unsigned char lds_raw[];
  __shared__ float red[kRcThreads / 64];
  KLane* kp = (KLane*)__builtin_amdgcn_kernarg_segment_ptr();
  float scale = scale_host;
  if (scale_in) {
    scale = *scale_in;
  } else if (amax_in) {
    const float m = *amax_in;
    scale = (m > 0.0f && m <= 3.402823466e38f) ? fp8_max / m : 1.0f;
  }
  if (scale_inv_out && blockIdx.x == 0 && threadIdx.x == 0) *scale_inv_out = 1.0f / scale;
  float amax = 0.0f;
  const uint32_t first = units.first(blockIdx.x), end = units.first(blockIdx.x + 1);
  for (uint32_t t = first; t < end; ++t) {
    if (t != first) __syncthreads();  // the previous tile's LDS reads
    RCLane<OP, VA, VB, false, false, DIV>::run(kp, amax_in ? units.n - 1 - t : t, A, B, lds_raw, alpha, scale, [&](float m) {
      amax = fmaxf(amax, m);
      if (amax_out && t + 1 == end) wg_max_publish(amax, red);
    });
  }
  if (amax_out && threadIdx.x == 0) amax_commit_one(wg_max_collect(red), amax_out);
}

}  // namespace ttc
