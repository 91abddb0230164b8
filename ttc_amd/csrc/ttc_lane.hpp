// Row x column tiles, one tile per work-group: the single-op launch of the
// row x column family (tile, row and column groups as in ttc_rc.hpp).
//
// Bound by HBM.  The dispatcher starts the next tile on whichever CU frees a
// slot first, so the tiles in flight stay neighbours in the walk order
// (rc_tile_of) and the cache lines they share at their edges are fetched and
// written back once; work-groups that stride over many tiles each (the
// pipelined kernel of ttc_rc.hpp) drift apart and lose that.  Time per
// launch, pipelined -> one tile per work-group (copy of 200 MiB: 5.5 TB/s):
//   fp32 6507 x 8057, padded              110 -> 95 us  (4.4 TB/s)
//   fp32 rank 6, odd extents, 200 MiB     131 -> 103    (4.1)
//   fp64 rank 5, beta = 1, 200 MiB        133 -> 117    (5.4)
//   fp32 -> bf16 rank 4 with beta, 2.4 GB 1129 -> 980   (4.9)
//   complex64 96 x 80 x 110               6.3 -> 5.3
//   fp64 37 x 21 x 19 x 5, beta = 1       7.5 -> 5.0
//
// Each lane keeps one vector of rows for the whole read walk and one vector
// of columns for the whole write walk (RCLaneParams), for any row and column
// count: a slot costs one table entry and one add on each side, and partial
// tiles, lanes past the walk and slots past the tile are entries of
// kRcTabOOB, which send the access out of the buffer range.  The code is a
// few KB: a small launch waits for its instructions, so straight-line code
// for every case would cost more than it saves.
#pragma once
#include "ttc_rc.hpp"

namespace ttc {

using KLane = const __attribute__((address_space(4))) RCLaneParams;

template <class OP, int VA, int VB, bool BETA, bool NT, int DIV>
struct RCLane {
  using TA = typename OP::TA;
  using TB = typename OP::TB;
  using L = typename OP::L;
  static constexpr int NIA = rc_elems((int)sizeof(TA)) / VA / DIV;  // read slots per lane
  static constexpr int NIB = rc_elems((int)sizeof(TB)) / VB / DIV;  // write slots per lane
  static constexpr bool FP8 = is_fp8<OP>::value;

  // Offsets of position l of a group: mixed-radix digits over its tile
  // extents times their byte strides.
  __device__ __forceinline__ static void offsets(KLane* kp, int first, int n, uint32_t l, int32_t& oa, int32_t& ob) {
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

  // The tile of work-group `wg` of the launch (of the op, in a grouped one).
  // after(amax): called between staging and the barrier with max |alpha * a|
  // of this lane's elements (fp8 casts).
  template <class F>
  __device__ __forceinline__ static void run(KLane* kp, uint32_t wg, const TA* __restrict__ A, TB* __restrict__ B,
                                             unsigned char* lds_raw, typename OP::AL alpha, typename OP::BE beta,
                                             F&& after) {
    const uint32_t tid = threadIdx.x;
    // tile origin
    uint32_t rem;
    {
      RCWalk w;
      w.ntiles = kp->walk.ntiles;
      w.grid_order = kp->walk.grid_order;
      w.bandw = kp->walk.bandw;
      w.bandn = kp->walk.bandn;
      w.bandin = kp->walk.bandin;
      w.dper = FastDiv{kp->walk.dper.d, kp->walk.dper.m, kp->walk.dper.s, 0};
      w.dband = FastDiv{kp->walk.dband.d, kp->walk.dband.m, kp->walk.dband.s, 0};
      w.dw = FastDiv{kp->walk.dw.d, kp->walk.dw.m, kp->walk.dw.s, 0};
      w.dwl = FastDiv{kp->walk.dwl.d, kp->walk.dwl.m, kp->walk.dwl.s, 0};
      rem = uniform(rc_tile_of(w, wg));
    }
    int64_t bA = 0, bB = 0;
    uint32_t last = 0;
    const int gr = kp->grank;
#pragma unroll 1
    for (int g = 0; g < gr; ++g) {
      const uint32_t d = kp->grid[g].d, q = fdiv(rem, kp->grid[g].m, kp->grid[g].s), x = rem - q * d;
      rem = q;
      bA += (int64_t)x * kp->grid[g].tsa;
      bB += (int64_t)x * kp->grid[g].tsb;
      if (x == d - 1) last |= kp->grid[g].part;
    }
    const int R = kp->R, C = kp->C, kA = kp->kA, kB = kp->kB, na = kp->na;
    const int rows = (last & 1u) ? kp->Rl : R, cols = (last & 2u) ? kp->Cl : C;
    // tables: colS[jl * NIA + it] = A offset of column jl + it * kA, rowS its
    // mirror image for B; rowA and colB by row and column
    L* const data = reinterpret_cast<L*>(lds_raw);
    int32_t* const colS = reinterpret_cast<int32_t*>(lds_raw + kp->tab);
    int32_t* const rowS = colS + kA * NIA;
    int32_t* const rowA = rowS + kB * NIB;
    int32_t* const colB = rowA + R;
    for (int e = (int)tid; e < kA * NIA; e += kRcThreads) {
      const int j = e / NIA + (e % NIA) * kA;
      int32_t oa, ob;
      offsets(kp, na, kp->nb, (uint32_t)j, oa, ob);
      colS[e] = j < cols ? oa : (int32_t)kRcTabOOB;
      if (j < C) colB[j] = j < cols ? ob : (int32_t)kRcTabOOB;
    }
    for (int e = (int)(kRcThreads - 1 - tid); e < kB * NIB; e += kRcThreads) {
      const int i = e / NIB + (e % NIB) * kB;
      int32_t oa, ob;
      offsets(kp, 0, na, (uint32_t)i, oa, ob);
      rowS[e] = i < rows ? ob : (int32_t)kRcTabOOB;
      if (i < R) rowA[i] = i < rows ? oa : (int32_t)kRcTabOOB;
    }
    const uint32_t RP = (uint32_t)kp->RP;
    // this lane's place in the two walks
    const uint32_t jl = fdiv(tid, kp->lam, kp->las), ai = (tid - jl * kp->la) * VA;
    const uint32_t il = fdiv(tid, kp->lbm, kp->lbs), bj = (tid - il * kp->lb) * VB;
    const bool onA = jl < (uint32_t)kA, onB = il < (uint32_t)kB;
    const uint32_t sA = onA ? ai + jl * RP : (uint32_t)kp->spare, stepA = onA ? (uint32_t)kA * RP : 0u;
    const uint32_t sB = onB ? il + bj * RP : 0u, stepB = onB ? (uint32_t)kB : 0u;
    __syncthreads();
    const uint32_t rowoff = onA ? (uint32_t)rowA[ai] : kRcTabOOB, coloff = onB ? (uint32_t)colB[bj] : kRcTabOOB;
    const int32_t* const cs = colS + (onA ? jl * NIA : 0u);
    const int32_t* const rs = rowS + (onB ? il * NIB : 0u);
    const BufRes ra = make_res(A + uniform64(bA)), rb = make_res(B + uniform64(bB));
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

// fp8 cast-transpose (semantics: cast_fp8_rc_kernel).  amax only grows during
// a launch: each work-group reads it as it starts, and one whose tile's max
// is not above that value is done; the others look again and then commit one
// atomic.
template <class OP, int VA, int VB, int DIV>
__global__ void __launch_bounds__(kRcThreads)
    cast_fp8_lane_kernel(const RCLaneParams p, const typename OP::TA* __restrict__ A,
                         typename OP::TB* __restrict__ B, float alpha, const float* __restrict__ scale_in,
                         const float* __restrict__ amax_in, float fp8_max, float scale_host,
                         float* __restrict__ amax_out, float* __restrict__ scale_inv_out) {
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
  unsigned int* const am = reinterpret_cast<unsigned int*>(amax_out);
  unsigned int seen = 0;
  if (am && threadIdx.x == 0) seen = __hip_atomic_load(am, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  RCLane<OP, VA, VB, false, false, DIV>::run(kp, blockIdx.x, A, B, lds_raw, alpha, scale, [&](float m) {
    if (!am) return;
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) m = fmaxf(m, __shfl_xor(m, off, 64));
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = m;
  });
  if (am && threadIdx.x == 0) {
    float m = red[0];
#pragma unroll
    for (int w = 1; w < kRcThreads / 64; ++w) m = fmaxf(m, red[w]);
    const unsigned int bits = __float_as_uint(m);
    if (bits > seen && bits > __hip_atomic_load(am, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) atomicMax(am, bits);
  }
}

}  // namespace ttc
