// The certificate of a row's donor pool (k4_stats.h), on the device.
#pragma once

#include "iq_common.h"
#include "k4_stats.h"

// One wavefront: whether the donor pool of a row (the channels with src_of >=
// 0: as many donors are picked as the pool holds) is certain under the
// enclosures lo / hi.
__device__ __forceinline__ bool iq_pool_certain(const float *lo, const float *hi, int D, const uint8_t *is_src,
                                                const int16_t *src_of)
{
    const int lane = threadIdx.x & 63;
    uint64_t in = 0, out = ~0ull;        // largest pool key, least key outside
    for (int c = lane; c < D; c += 64) {
        if (is_src[c]) continue;
        if (src_of[c] >= 0) {
            const uint64_t k = iq_err_key(hi[c], c);
            in = k > in ? k : in;
        } else {
            const uint64_t k = iq_err_key(lo[c], c);
            out = k < out ? k : out;
        }
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        const uint64_t a = (uint64_t)__shfl_xor((unsigned long long)in, o, 64);
        const uint64_t b = (uint64_t)__shfl_xor((unsigned long long)out, o, 64);
        in = a > in ? a : in;
        out = b < out ? b : out;
    }
    return in < out;
}
