// Row-copy kernel for permutations that keep dimension 0 in place
// (perm[0] == 0 after index fusion): A and B share the stride-1 dimension,
// so every row of dimension 0 is contiguous on both sides and moves without
// an LDS round trip.  The reference handles this case with its own loop
// (ttc/CUDAtranspose.py:179-243, threads along i0, rows in a cyclic block
// distribution); here each lane moves a V-element vector, the rows are
// walked in B order so that consecutive lanes write consecutive bytes of B,
// and every lane keeps U vectors in flight.
#pragma once
#include "ttc_kernels.hpp"

namespace ttc {

// touch_lines over a row kernel's arguments: RowParams, and behind it pointers,
// scalars and scales.  One statement waits for all lines, so that none is left
// for a second wait.
__device__ __forceinline__ void touch_row_args() {
  static_assert(sizeof(RowParams) > 192 && sizeof(RowParams) <= 256, "lines of the arguments");
  KWord* const w = (KWord*)__builtin_amdgcn_kernarg_segment_ptr();
  asm volatile("" ::"s"(w[0]), "s"(w[16]), "s"(w[32]), "s"(w[48]), "s"(w[64]));
}

template <class OP, int V, int MODE>
__global__ void __launch_bounds__(kThreads)
    row_kernel(const RowParams p, const typename OP::TA* __restrict__ A, typename OP::TB* __restrict__ B,
               double alpha, double beta, const float* __restrict__ scale_in, const float* __restrict__ amax_in,
               float fp8_max, float scale_host, float* __restrict__ amax_out, float* __restrict__ scale_inv_out) {
  using TA = typename OP::TA;
  using TB = typename OP::TB;
  using L = typename OP::L;
  constexpr bool FP8 = MODE == kModeFp8;
  constexpr bool BETA = MODE == kModeBeta;
  constexpr bool NT = MODE == kModeBzNt;
  constexpr int U = kRowUnroll;  // vectors in flight per lane
  // (casts to fp8 of 8 to 32 MB 9-11% faster so, of 64 to 128 3-6%)
  touch_row_args();
  float scale = 1.0f;
  if constexpr (FP8) {
    scale = scale_host;
    if (scale_in) {
      scale = *scale_in;
    } else if (amax_in) {
      const float m = *amax_in;
      scale = (m > 0.0f && m <= 3.402823466e38f) ? fp8_max / m : 1.0f;
    }
    if (scale_inv_out && blockIdx.x == 0 && threadIdx.x == 0) *scale_inv_out = 1.0f / scale;
  }
  const typename OP::AL al = (typename OP::AL)alpha;
  const typename OP::BE be = (typename OP::BE)beta;
  const char* a = reinterpret_cast<const char*>(A);
  char* b = reinterpret_cast<char*>(B);
  const uint32_t stride = gridDim.x * (uint32_t)kThreads;  // the host keeps total + U * stride < 2^32
  float amax = 0.0f;
  for (uint32_t g0 = blockIdx.x * (uint32_t)kThreads + threadIdx.x; g0 < p.total; g0 += U * stride) {
    int64_t ob[U];
    bool ok[U];
    TA va[U][V];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const uint32_t g = g0 + (uint32_t)u * stride;
      ok[u] = g < p.total;
      const uint32_t gg = ok[u] ? g : 0u;
      const uint32_t row = fdiv(gg, p.nvm, p.nvs);
      const uint32_t v = gg - row * p.nv;
      int64_t xa = (int64_t)v * (int64_t)(V * sizeof(TA));
      int64_t xb = (int64_t)v * (int64_t)(V * sizeof(TB));
      uint32_t rem = row;
#pragma unroll
      for (int k = 0; k < kMaxDim; ++k) {
        if (k < p.rank) {
          const uint32_t q = fdiv(rem, p.dn[k].m, p.dn[k].s);
          const uint32_t x = rem - q * p.dn[k].d;
          rem = q;
          xa += (int64_t)x * p.sa[k];
          xb += (int64_t)x * p.sb[k];
        }
      }
      ob[u] = xb;
      if (ok[u]) vload<TA, V>(va[u], reinterpret_cast<const TA*>(a + xa));
    }
    TB old[U][V];
    if constexpr (BETA) {
#pragma unroll
      for (int u = 0; u < U; ++u)
        if (ok[u]) vload<TB, V>(old[u], reinterpret_cast<const TB*>(b + ob[u]));
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      if (!ok[u]) continue;
      TB o[V];
      if constexpr (FP8) {
        L x[V];
#pragma unroll
        for (int v = 0; v < V; ++v) {
          x[v] = OP::prod(al, va[u][v]);
          amax = fmaxf(amax, fabsf(x[v]));
        }
        if constexpr (V == 1) {
          o[0] = OP::outs(x[0], scale);
        } else {
#pragma unroll
          for (int v = 0; v < V; v += 2) OP::outs2(x[v], x[v + 1], scale, o[v], o[v + 1]);
        }
      } else if constexpr (BETA) {
#pragma unroll
        for (int v = 0; v < V; ++v) o[v] = OP::outb(OP::prod(al, va[u][v]), be, old[u][v]);
      } else {
#pragma unroll
        for (int v = 0; v < V; ++v) o[v] = OP::out(OP::prod(al, va[u][v]));
      }
      vstore<TB, V, NT>(reinterpret_cast<TB*>(b + ob[u]), o);
    }
  }
  if constexpr (FP8) {
    if (amax_out) block_amax_commit(amax, amax_out);
  }
}

// V elements with the alignment of one element: gfx950 takes vector accesses
// at any such address.
template <class T, int V> struct __attribute__((packed, aligned(sizeof(T)))) RowVec {
  T x[V];
};

// One chunk of kThreads * U vectors per work-group.  The dispatcher keeps
// every CU full to the end of the launch, where a work-group striding over
// the whole tensor (row_kernel) leaves the chip in step with the slowest.
//   UNAL: dimension 0 (extent n0 >= V) is not a whole number of aligned
// vectors.  A row takes ceil(n0 / V) vectors at element alignment, the last
// one shifted back to end at the row's end; its first elements are its
// neighbour's too.  With beta == 0 both write the same values; with beta the
// shifted lane stores only its own elements, since its neighbour's may
// already hold their results.
// Bound by HBM (16-byte vectors) or by the address arithmetic per vector
// (narrow ones).  Striding work-groups -> this kernel, GB/s: fp32 200 MiB
// copy 4740 -> 6010; bf16 128 x 4096 x 32 x 8 perm (0,2,1,3) 4760 -> 5340;
// fp32 rows of 127 3890 -> 4730, of 5 2210 -> 3040; bf16 rows of 127
// 2180 -> 4070, of 5 1270 -> 2240.
// P: RowParams as a kernel argument or in a grouped launch's work table, or
// RowSmall.
// Returns max |alpha * a| of this lane's elements (fp8 casts).
template <class OP, int V, int MODE, bool UNAL, class P>
__device__ __forceinline__ float row_chunk(const P& p, uint32_t w, const typename OP::TA* __restrict__ A,
                                           typename OP::TB* __restrict__ B, typename OP::AL al, typename OP::BE be,
                                           float scale) {
  using TA = typename OP::TA;
  using TB = typename OP::TB;
  using L = typename OP::L;
  constexpr bool kSmall = std::is_same<P, RowSmall>::value;
  constexpr bool FP8 = MODE == kModeFp8;
  constexpr bool BETA = MODE == kModeBeta;
  constexpr bool NT = MODE == kModeBzNt;
  constexpr int U = row_once_unroll((int)sizeof(TA), (int)sizeof(TB), V, FP8, UNAL);
  const uint32_t g0 = w * (uint32_t)(kThreads * U) + threadIdx.x;
  const char* a = reinterpret_cast<const char*>(A);
  char* b = reinterpret_cast<char*>(B);
  int64_t ob[U];
  bool ok[U];
  int skip[U];  // UNAL: leading elements of a shifted vector that are its neighbour's
  TA va[U][V];
  TB old[U][V];
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const uint32_t g = g0 + (uint32_t)(u * kThreads);
    ok[u] = g < p.total;
    const uint32_t gg = ok[u] ? g : 0u;
    uint32_t row;
    if constexpr (kSmall) row = sdiv(gg, p.nv);
    else row = fdiv(gg, p.nvm, p.nvs);
    int32_t e = (int32_t)(gg - row * p.nv) * V;
    skip[u] = 0;
    if constexpr (UNAL) {
      skip[u] = row_shift(e, V, p.n0);
      e -= skip[u];
    }
    int64_t xa = (int64_t)e * (int64_t)sizeof(TA), xb = (int64_t)e * (int64_t)sizeof(TB);
    uint32_t rem = row;
#pragma unroll
    for (int k = 0; k < (kSmall ? kSmallRowDims : kMaxDim); ++k) {
      if (k < p.rank) {
        if constexpr (kSmall) {
          const uint32_t q = sdiv(rem, p.dim[k].d), x = rem - q * p.dim[k].d;
          rem = q;
          xa += (int64_t)x * p.dim[k].sa;
          xb += (int64_t)x * p.dim[k].sb;
        } else {
          const uint32_t q = fdiv(rem, p.dn[k].m, p.dn[k].s);
          const uint32_t x = rem - q * p.dn[k].d;
          rem = q;
          xa += (int64_t)x * p.sa[k];
          xb += (int64_t)x * p.sb[k];
        }
      }
    }
    ob[u] = xb;
    if (!ok[u]) continue;
    if constexpr (UNAL) {
      const RowVec<TA, V> t = *reinterpret_cast<const RowVec<TA, V>*>(a + xa);
      __builtin_memcpy(&va[u][0], &t, sizeof(t));
      if constexpr (BETA) {
        const RowVec<TB, V> o = *reinterpret_cast<const RowVec<TB, V>*>(b + xb);
        __builtin_memcpy(&old[u][0], &o, sizeof(o));
      }
    } else {
      vload<TA, V>(va[u], reinterpret_cast<const TA*>(a + xa));
      if constexpr (BETA) vload<TB, V>(old[u], reinterpret_cast<const TB*>(b + xb));
    }
  }
  float amax = 0.0f;
#pragma unroll
  for (int u = 0; u < U; ++u) {
    if (!ok[u]) continue;
    TB o[V];
    if constexpr (FP8) {
      L x[V];
#pragma unroll
      for (int v = 0; v < V; ++v) {
        x[v] = OP::prod(al, va[u][v]);
        amax = fmaxf(amax, fabsf(x[v]));
      }
      if constexpr (V == 1) {
        o[0] = OP::outs(x[0], scale);
      } else {
#pragma unroll
        for (int v = 0; v < V; v += 2) OP::outs2(x[v], x[v + 1], scale, o[v], o[v + 1]);
      }
    } else if constexpr (BETA) {
#pragma unroll
      for (int v = 0; v < V; ++v) o[v] = OP::outb(OP::prod(al, va[u][v]), be, old[u][v]);
    } else {
#pragma unroll
      for (int v = 0; v < V; ++v) o[v] = OP::out(OP::prod(al, va[u][v]));
    }
    TB* const dst = reinterpret_cast<TB*>(b + ob[u]);
    if constexpr (UNAL) {
      if (!BETA || skip[u] == 0) {
        RowVec<TB, V> t;
        __builtin_memcpy(&t, &o[0], sizeof(t));
        *reinterpret_cast<RowVec<TB, V>*>(dst) = t;
      } else {
#pragma unroll
        for (int v = 0; v < V; ++v)
          if (v >= skip[u]) dst[v] = o[v];
      }
    } else {
      vstore<TB, V, NT>(dst, o);
    }
  }
  return amax;
}

template <class OP, int V, int MODE, bool UNAL>
__global__ void __launch_bounds__(kThreads)
    row_once_kernel(const RowParams p, const typename OP::TA* __restrict__ A, typename OP::TB* __restrict__ B,
                    double alpha, double beta, const float* __restrict__ scale_in, const float* __restrict__ amax_in,
                    float fp8_max, float scale_host, float* __restrict__ amax_out,
                    float* __restrict__ scale_inv_out, AmaxUnits units) {
  constexpr bool FP8 = MODE == kModeFp8;
  touch_row_args();
  float scale = 1.0f;
  if constexpr (FP8) {
    scale = scale_host;
    if (scale_in) {
      scale = *scale_in;
    } else if (amax_in) {
      const float m = *amax_in;
      scale = (m > 0.0f && m <= 3.402823466e38f) ? fp8_max / m : 1.0f;
    }
    if (scale_inv_out && blockIdx.x == 0 && threadIdx.x == 0) *scale_inv_out = 1.0f / scale;
  }
  uint32_t w = blockIdx.x;
  if (p.xcd_share) {
    const uint32_t x = w % kXcds, q = gridDim.x / kXcds, r = gridDim.x % kXcds;
    w = x * q + (x < r ? x : r) + w / kXcds;
  }
  if constexpr (FP8) {
    // the chunks AmaxUnits gives this work-group, one commit; backwards after
    // an amax pass, which leaves the end of A in the last-level cache (bf16 128
    // x 4096 x 32 x 8, both passes: 143 -> 130 us)
    float amax = 0.0f;
    const uint32_t end = units.first(w + 1);
    for (uint32_t c = units.first(w); c < end; ++c)
      amax = fmaxf(amax, row_chunk<OP, V, MODE, UNAL>(p, amax_in ? units.n - 1 - c : c, A, B,
                                                      (typename OP::AL)alpha, (typename OP::BE)beta, scale));
    if (amax_out) {
      __shared__ float red[kThreads / 64];
      wg_max_publish(amax, red);
      __syncthreads();
      if (threadIdx.x == 0) amax_commit_one(wg_max_collect(red), amax_out);
    }
  } else {
    (void)row_chunk<OP, V, MODE, UNAL>(p, w, A, B, (typename OP::AL)alpha, (typename OP::BE)beta, scale);
  }
}

// The same with few bytes of arguments (RowSmall), without casts to fp8.
template <class OP, int V, int MODE, bool UNAL>
__global__ void __launch_bounds__(kThreads)
    row_small_kernel(const RowSmall p, const typename OP::TA* __restrict__ A, typename OP::TB* __restrict__ B,
                     double alpha, double beta) {
  touch_lines<sizeof(RowSmall)>(__builtin_amdgcn_kernarg_segment_ptr());
  uint32_t w = blockIdx.x;
  if (p.xcd_share) {
    const uint32_t x = w % kXcds, q = p.grid / kXcds, r = p.grid % kXcds;
    w = x * q + (x < r ? x : r) + w / kXcds;
  }
  (void)row_chunk<OP, V, MODE, UNAL>(p, w, A, B, (typename OP::AL)alpha, (typename OP::BE)beta, 1.0f);
}

}  // namespace ttc
