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

// prep_kernel: a row's heads in pairs of one kind, q, then k, then v; a wave's
// half-wave hv (0, 1) takes head 2 i + hv of its kind's pair i. Hq is even, an
// odd Hkv's last pair has one head.
struct PrepPairs {
    int Hq, Hkv, nq, nk;  // heads, pairs
    PKV_INDEX PrepPairs(int hq, int hkv) : Hq(hq), Hkv(hkv), nq(hq / 2), nk((hkv + 1) / 2) {}
    PKV_INDEX int units() const { return nq + 2 * nk; }
    PKV_INDEX bool is_q(int u) const { return u < nq; }
    PKV_INDEX bool is_v(int u) const { return u >= nq + nk; }
    // The head of its kind that half hv of pair u takes, and whether there is one.
    PKV_INDEX int head(int u, int hv) const { return 2 * (u - (is_q(u) ? 0 : is_v(u) ? nq + nk : nq)) + hv; }
    PKV_INDEX bool has(int u, int hv) const { return is_q(u) || head(u, hv) < Hkv; }
    // Where it lies in the token's row [Hq x (q | gate) | k | v], in 256
    // values (absent: its kind's head 0).
    PKV_INDEX int source(int u, int hv) const {
        if (is_q(u)) return 2 * head(u, hv);
        return 2 * Hq + (is_v(u) ? Hkv : 0) + (has(u, hv) ? head(u, hv) : 0);
    }
    // Waves of P pairs per token.
    PKV_INDEX int groups(int P) const { return (units() + P - 1) / P; }
};
// Workgroups of 4 waves for T tokens of `groups` waves; wave i takes token
// i / groups, pairs from P (i % groups) on.
PKV_INDEX unsigned prep_grid(int T, int groups) { return (unsigned)(((long)T * groups + 3) / 4); }

}  // namespace pkv
