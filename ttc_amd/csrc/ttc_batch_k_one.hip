// Grouped launch of one work-group per tile: the kernel over all types.
#include "ttc_batch_one.hpp"

namespace ttc {

using KIdx = const __attribute__((address_space(4))) uint32_t;
using KIndex = const __attribute__((address_space(4))) OneIndex;

__global__ void __launch_bounds__(kThreads)
    batch_one_kernel(const OneLane* __restrict__ lanes, const OneRow* __restrict__ rows,
                     const OneIndex* __restrict__ index, const uint32_t* __restrict__ block, uint32_t nops,
                     uint32_t ntiles) {
  extern __shared__ __align__(16) unsigned char lds_raw[];
  KIndex* kindex = (KIndex*)index;
  KIdx* kblock = (KIdx*)block;
  for (uint32_t w = blockIdx.x; w < ntiles; w += gridDim.x) {
    if (w != blockIdx.x) __syncthreads();  // the previous tile's LDS reads
    const uint32_t id = uniform(one_tile_of(w, ntiles));
    uint32_t op = uniform(kblock[id / kOneBlock]);
    while (op + 1 < nops && kindex[op + 1].first <= id) ++op;
    op = uniform(op);
    const uint32_t tile = id - kindex[op].first, rec = kindex[op].rec;
    // the whole record, before its kind: one wait for both (60 ops, 143 MB: 45.1
    // -> 43.4 us; 40 ops, 7.3 MB: 9.85 -> 9.65)
    KHead* o;
    if (!(rec & kOneIsRow)) {
      o = (KHead*)((KOneLane*)lanes + rec);
      touch_lines<sizeof(OneHead) + sizeof(RCLaneParams)>(o);
    } else {
      o = (KHead*)((KOneRow*)rows + (rec & ~kOneIsRow));
      touch_lines<sizeof(OneRow)>(o);
    }
    const int kind = o->kind, variant = kind % kOneVariants;
    switch (kind / kOneVariants) {
      case kBS: one_type<OpF32<float, float>, 4>(variant, o, tile, lds_raw); break;
      case kBD: one_type<OpDD, 2>(variant, o, tile, lds_raw); break;
      case kBBF16: one_type<OpF32<bf16s, bf16s>, 8>(variant, o, tile, lds_raw); break;
      case kBF16: one_type<OpF32<f16s, f16s>, 8>(variant, o, tile, lds_raw); break;
      case kBC: one_type<OpCC, 2>(variant, o, tile, lds_raw); break;
      case kBZ: one_type<OpZZ, 1>(variant, o, tile, lds_raw); break;
      default: break;
    }
  }
}

const void* batch_one_func() { return reinterpret_cast<const void*>(&batch_one_kernel); }

}  // namespace ttc
