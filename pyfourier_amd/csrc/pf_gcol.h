// Window geometry of the LDS-staged gathers (forward gather in pf_ops.hip,
// coordinate-derivative gather in pf_grad.hip) and their global -> LDS copy.
// HIP device code: include from .hip sources only.
#pragma once

#include "pf_internal.h"

namespace {

// threads per block: the forward gather takes an item's lanes at once (a window
// of more samples than lanes is staged once per item, so more lanes restage
// less: 512 against 256, 3-D 256^3 grid x 32 coils, W = 6 2476 -> 2300 us, and 2190 us
// with the items dealt to the XCDs in chunks; x 8 coils, W = 4 400 -> 320 us); the
// derivative gather's registers allow 256: it runs over the items' halves
constexpr int GCOL_TB = PF_GCOL_MAXS;
constexpr int GCOL_GTB = PF_GCOL_MAXS / 2;
constexpr int GCOL_OUT = 4;  // coil pairs per output store of the forward gather

template <int W, int TB = GCOL_TB>
struct GColShape {
    static constexpr int DZ = pf_gather_dz(W);
    static constexpr int NPL = DZ + W - 1;                          // staged z planes
    static constexpr int PX = PF_GCOL + W - 1;                       // staged points per y and x
    static constexpr int PP = PX * PX;
    static constexpr int NPTS = NPL * PP;
    static constexpr int NK = (NPTS + TB - 1) / TB;       // staged points per thread
};

// 16 bytes global -> LDS for each active lane (the destination is the wave's
// LDS base plus 16 bytes per lane)
__device__ __forceinline__ void gcol_copy16(const float4* src, float4* lds_wave_base) {
    __builtin_amdgcn_global_load_lds(src, (__attribute__((address_space(3))) void*)lds_wave_base, 16, 0, 0);
}

}  // namespace
