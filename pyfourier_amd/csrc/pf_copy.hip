// Copies of a list of arrays into strided buffers (the items of an uneven
// batch into their group's static images / samples) in a few launches.
//
// An item is rows x len complex values, contiguous at the source and with a
// row stride at the destination.  A block copies up to CP_LEN values of one
// row, 16 bytes per lane where both sides are aligned to it.  The item table
// travels in the kernel arguments, so nothing is uploaded per call.  A copy of
// this kind is bound by HBM; one launch per item (as a multi-tensor copy falls
// back to for strided destinations) left 4.4 us per 2.3 MB item: 32 slices x 8
// coils (75 MB) 140 us, here 34 us.
#include <algorithm>

#include "pf_internal.h"

namespace {

constexpr int CP_N = 64;       // items per launch
constexpr int CP_TB = 256;
constexpr int CP_LEN = 4096;   // values per block

struct CopyItems {
    const float2* src[CP_N];
    float2* dst[CP_N];
    int64_t stride[CP_N];  // destination row stride (values)
    int64_t len[CP_N];     // values per row
    unsigned first[CP_N + 1];  // first block of each item
};
static_assert(sizeof(CopyItems) <= 4096 - 64, "item table fits the kernel arguments");

__global__ void __launch_bounds__(CP_TB) k_copy_items(CopyItems t, int n) {
    int i = 0;
    while (i + 1 < n && blockIdx.x >= t.first[i + 1]) ++i;
    const int64_t len = t.len[i];
    const unsigned per_row = (unsigned)((len + CP_LEN - 1) / CP_LEN), b = blockIdx.x - t.first[i];
    const int64_t row = b / per_row, c0 = (int64_t)(b % per_row) * CP_LEN;
    const float2* src = t.src[i] + row * len + c0;
    float2* dst = t.dst[i] + row * t.stride[i] + c0;
    const int m = (int)std::min<int64_t>(CP_LEN, len - c0);
    if (((reinterpret_cast<uintptr_t>(src) | reinterpret_cast<uintptr_t>(dst)) & 15) == 0) {
        const float4* s4 = reinterpret_cast<const float4*>(src);
        float4* d4 = reinterpret_cast<float4*>(dst);
        for (int k = threadIdx.x; k < m / 2; k += CP_TB) d4[k] = s4[k];
        if ((m & 1) && threadIdx.x == 0) dst[m - 1] = src[m - 1];
    } else {
        for (int k = threadIdx.x; k < m; k += CP_TB) dst[k] = src[k];
    }
}

}  // namespace

extern "C" int pf_copy_items(int n, const void* const* src, void* const* dst, const long long* rows, const long long* len,
                             const long long* dst_stride, void* stream) {
    if (n < 0) return pf_fail(PF_ERR_ARG, "negative item count");
    if (n > 0 && (!src || !dst || !rows || !len || !dst_stride)) return pf_fail(PF_ERR_ARG, "null argument");
    for (int i = 0; i < n; ++i) {
        if (rows[i] < 0 || len[i] < 0) return pf_fail(PF_ERR_ARG, "negative item size");
        if (rows[i] > 1 && dst_stride[i] < len[i]) return pf_fail(PF_ERR_ARG, "destination rows overlap");
        if (rows[i] > 0 && len[i] > 0 && (!src[i] || !dst[i])) return pf_fail(PF_ERR_ARG, "null item");
        if ((len[i] + CP_LEN - 1) / CP_LEN * (double)rows[i] > 1e9) return pf_fail(PF_ERR_UNSUPPORTED, "item too large");
    }
    for (int i = 0; i < n;) {
        CopyItems t{};
        int k = 0;
        int64_t blocks = 0;
        for (; i < n && k < CP_N; ++i) {
            const int64_t nb = (len[i] + CP_LEN - 1) / CP_LEN * rows[i];
            if (nb == 0) continue;
            if (blocks + nb > 0x7fffffff) break;
            t.src[k] = static_cast<const float2*>(src[i]);
            t.dst[k] = static_cast<float2*>(dst[i]);
            t.len[k] = len[i];
            t.stride[k] = dst_stride[i];
            t.first[k++] = (unsigned)blocks;
            blocks += nb;
        }
        if (k == 0) continue;
        t.first[k] = (unsigned)blocks;
        hipLaunchKernelGGL(k_copy_items, dim3((unsigned)blocks), dim3(CP_TB), 0, static_cast<hipStream_t>(stream), t, k);
        PF_HIP(hipGetLastError());
    }
    return PF_OK;
}
