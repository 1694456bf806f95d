// Index arithmetic of the kernels that is also built for the host (plain C++,
// no HIP headers), where tests check it against the buffers' bounds over all
// the values a launch can take.
#pragma once

#ifdef __HIPCC__
#define PKV_INDEX __host__ __device__ __forceinline__ constexpr
#else
#define PKV_INDEX inline constexpr
#endif

namespace pkv {

// First key of range b (>= 0) of R (> 0) keys, W when it lies past the last of
// the W keys: b R can pass the 32-bit range (16,384 workgroups of at least 2^20
// keys are a setting that pkv_attn_decode_config takes).
PKV_INDEX int range_start(int b, int R, int W) {
    const unsigned long s = (unsigned long)(unsigned)b * (unsigned)R;
    return s < (unsigned long)(unsigned)W ? (int)s : W;
}
// One past the last key of the range that starts at start (<= W).
PKV_INDEX int range_end(int start, int R, int W) { return W - start < R ? W : start + R; }

}  // namespace pkv
