// Attention input preparation on gfx950: the reference's attn_prep
// (qwen35.cu:1067-1128), which is where the reference appends K/V to the
// paged cache. For token t and head hh of the qkv row
// [Hq x (q 256 | gate 256) | k Hkv x 256 | v Hkv x 256]:
//   q / k heads: y = bf16(x * scale * w), scale = 1 / sqrt(sum x^2 / 256 + eps)
//     (RMSNorm with f32 weights), then dims 0..63 rotate as pairs (d, d + 32)
//     with bf16 cos / sin of pos * inv_freq[d]:
//       lo' = bf16(bf16(lo c) - bf16(hi s)),  hi' = bf16(bf16(hi c) + bf16(lo s)),
//     pos = rope[axis * rope_stride + t], axis 1 (height) for d % 3 == 1 below
//     3 sec_h, 2 (width) for d % 3 == 2 below 3 sec_w, else 0 (time);
//     q goes to qout[t][hh], k to kcache[slot][hh - Hq];
//   v heads: copied bit for bit to vcache[slot];
//   k and v are skipped for slot_map[t] < 0 (padding rows); q is always written;
//   with an E4M3 cache (kscale / vscale given) k and v are stored as E4M3
//   bytes with an f32 scale per (slot, kv head) (store_e4m3_wave).
//
// Layout (this build's own), prep_kernel: a half-wave takes a head, 8
// consecutive dims per lane (one 16-byte load and store), so a wave takes two
// heads of one kind at a time and P such units in turn, all of their rows
// requested up front. The token's 32 cos / sin pairs are evaluated once per
// wave, one per lane, while the rows are in flight, and shared through 256
// bytes of LDS; the squared sum and the E4M3 amax stay inside the half-wave
// (DPP, one permlane swap), a rotary pair's partner (d + 32) sits 4 lanes
// away inside the same 16-lane row and moves as packed bf16.
// What bounds it: for prompts HBM (8,192 rows at 16 / 4 heads, 201 MB:
// 43.9 us, 4.6 TB/s, where a 2 GiB device copy reaches 4.9; 142.3 us with a
// wave per head, 4 dims per lane and 8 cos / sin evaluations per lane and
// wave, which was bound by VALU issue); for decode steps the launch and one
// dependent round trip (64 rows 5.0 -> 3.0 us).
// prep_head_kernel: one wave per (token, head), 4 dims per lane; the code
// object's attn_prep and odd head counts (pkv_attn_prep says which and why).
#pragma once
#include "pkv_common.h"

namespace pkv {

constexpr int ROPE_DIM = 64;  // rotated leading dims of each head (reference qwen35.cu:23)

struct PrepArgs {
    const uint16_t* qkv;
    int qstride, Hq, Hkv;
    const float* q_norm;
    const float* k_norm;
    const int* rope;
    int rope_stride, sec_h, sec_w;
    const int* slot_map;
    const float* inv_freq;
    uint16_t* qout;
    uint16_t* kcache;
    uint16_t* vcache;
    float* kscale;  // non-null: an E4M3 cache (bytes in kcache / vcache, f32 scale per slot and kv head)
    float* vscale;
    float eps;
    long num_slots;
};

// One head's 256 values (4 per lane) as E4M3 with scale amax / 448 (1 if
// all zero): bytes = e4m3(v * (1 / scale)) (reference store_e4m3,
// qwen35.cu:1055-1065).
__device__ __forceinline__ void store_e4m3_wave(const float (&v)[4], uint8_t* dst, float* scale) {
    const int lane = threadIdx.x & 63;
    float amax = fmaxf(fmaxf(fabsf(v[0]), fabsf(v[1])), fmaxf(fabsf(v[2]), fabsf(v[3])));
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) amax = fmaxf(amax, __shfl_xor(amax, o, 64));
    const float sc = amax > 0.f ? amax / 448.f : 1.f;
    const float inv = 1.f / sc;
    *reinterpret_cast<uint32_t*>(dst + 4 * lane) = f32x4_to_e4m3x4(v[0] * inv, v[1] * inv, v[2] * inv, v[3] * inv);
    if (lane == 0) *scale = sc;
}

// One wave: token t, head hh (q heads, then k heads, then v heads).
__device__ __forceinline__ void prep_head(const PrepArgs& a, int t, int hh) {
    const int lane = threadIdx.x & 63;
    const uint16_t* row = a.qkv + (size_t)t * a.qstride;
    const long slot = a.slot_map[t];
    const bool has_slot = slot >= 0 && slot < a.num_slots;
    if (hh >= a.Hq + a.Hkv) {
        if (!has_slot) return;
        const int vh = hh - a.Hq - a.Hkv;
        const uint16_t* src = row + (size_t)a.Hq * 2 * HEAD_DIM + (size_t)(a.Hkv + vh) * HEAD_DIM;
        const size_t at = (size_t)slot * a.Hkv + vh;
        const uint2 raw = *reinterpret_cast<const uint2*>(src + 4 * lane);
        if (a.vscale) {
            const float x[4] = {bf_lo(raw.x), bf_hi(raw.x), bf_lo(raw.y), bf_hi(raw.y)};
            store_e4m3_wave(x, reinterpret_cast<uint8_t*>(a.vcache) + at * HEAD_DIM, a.vscale + at);
        } else {
            *reinterpret_cast<uint2*>(a.vcache + at * HEAD_DIM + 4 * lane) = raw;
        }
        return;
    }
    const bool is_q = hh < a.Hq;
    if (!is_q && !has_slot) return;
    const uint16_t* src = is_q ? row + (size_t)hh * 2 * HEAD_DIM : row + (size_t)a.Hq * 2 * HEAD_DIM +
                                                                     (size_t)(hh - a.Hq) * HEAD_DIM;
    // The row, the norm weights, then the rotary positions and frequencies
    // of the lane's 4 dims, all requested before anything waits (loads
    // return in order: the squared sum waits for the row alone), so the 4
    // cos / sin evaluations below wait on one round trip, not one each.
    const uint2 raw = *reinterpret_cast<const uint2*>(src + 4 * lane);
    const float4 w = *reinterpret_cast<const float4*>((is_q ? a.q_norm : a.k_norm) + 4 * lane);
    // (Every lane loads them, from valid indices: under a lane condition the
    // compiler could not count the loads, and the squared sum would wait
    // for all of them.)
    int rpos[4];
    float rinv[4];
#pragma unroll
    for (int e = 0; e < 4; e++) {
        const int d = (4 * lane + e) & (ROPE_DIM / 2 - 1);
        const int axis = (d % 3 == 1 && d < 3 * a.sec_h) ? 1 : (d % 3 == 2 && d < 3 * a.sec_w) ? 2 : 0;
        rpos[e] = a.rope[(size_t)axis * a.rope_stride + t];
        rinv[e] = a.inv_freq[d];
    }
    const float x[4] = {bf_lo(raw.x), bf_hi(raw.x), bf_lo(raw.y), bf_hi(raw.y)};
    float ss = x[0] * x[0] + x[1] * x[1] + x[2] * x[2] + x[3] * x[3];
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) ss += __shfl_xor(ss, o, 64);
    const float scale = 1.f / sqrtf(ss / HEAD_DIM + a.eps);
    float y[4] = {rbf(x[0] * scale * w.x), rbf(x[1] * scale * w.y), rbf(x[2] * scale * w.z), rbf(x[3] * scale * w.w)};
    // Rotary: lanes 0..7 hold dims d = 0..31 ("lo"), lanes 8..15 dims d + 32.
    float yp[4];
#pragma unroll
    for (int e = 0; e < 4; e++) yp[e] = dpp<DPP_ROW_ROR8>(y[e]);  // lane i <- lane i ^ 8 of its row
    if (lane < ROPE_DIM / 4) {
        const bool lo_half = lane < ROPE_DIM / 8;
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const float f = (float)rpos[e] * rinv[e];
            const float c = rbf(cosf(f)), s = rbf(sinf(f));
            const float lo = lo_half ? y[e] : yp[e], hi = lo_half ? yp[e] : y[e];
            y[e] = lo_half ? rbf(rbf(lo * c) - rbf(hi * s)) : rbf(rbf(hi * c) + rbf(lo * s));
        }
    }
    if (!is_q && a.kscale) {
        const size_t at = (size_t)slot * a.Hkv + (hh - a.Hq);
        store_e4m3_wave(y, reinterpret_cast<uint8_t*>(a.kcache) + at * HEAD_DIM, a.kscale + at);
        return;
    }
    uint16_t* dst = is_q ? a.qout + ((size_t)t * a.Hq + hh) * HEAD_DIM
                         : a.kcache + ((size_t)slot * a.Hkv + (hh - a.Hq)) * HEAD_DIM;
    *reinterpret_cast<uint2*>(dst + 4 * lane) = make_uint2(pack2(y[0], y[1]), pack2(y[2], y[3]));
}

// Grid (T, ceil((Hq + 2 Hkv) / 4)), 256 threads: wave w takes head 4 y + w.
__global__ void __launch_bounds__(256) prep_head_kernel(PrepArgs a) {
    const int hh = blockIdx.y * 4 + (threadIdx.x >> 6);
    if (hh < a.Hq + 2 * a.Hkv) prep_head(a, blockIdx.x, hh);
}

// Partner lane i ^ 4 inside each 8-lane group: banks (4-lane groups) 0 and 2
// of a row read 4 lanes up, banks 1 and 3 4 lanes down.
__device__ __forceinline__ uint32_t dpp_xor4(uint32_t v) {
    const int up = __builtin_amdgcn_update_dpp(0, (int)v, 0x104 /* row_shl:4 */, 0xf, 0x5, false);
    return (uint32_t)__builtin_amdgcn_update_dpp(up, (int)v, 0x114 /* row_shr:4 */, 0xf, 0xa, false);
}

// Sum over the lane's half-wave of two partials per lane (every lane gets
// it): the partials of dims 0 .. 3 and 4 .. 7 are folded over lane distances
// 16, 8, .. 1 apart, then added, the tree of a 64-lane fold of 4 dims each.
__device__ __forceinline__ float half_sum2(float a, float b) {
    a = add_xor16(a);
    b = add_xor16(b);
    a += dpp<DPP_ROW_ROR8>(a);
    b += dpp<DPP_ROW_ROR8>(b);
    a += __uint_as_float(dpp_xor4(__float_as_uint(a)));
    b += __uint_as_float(dpp_xor4(__float_as_uint(b)));
    a += dpp<DPP_QUAD_XOR2>(a);
    b += dpp<DPP_QUAD_XOR2>(b);
    a += dpp<DPP_QUAD_XOR1>(a);
    b += dpp<DPP_QUAD_XOR1>(b);
    return a + b;
}
// Maximum over the lane's half-wave.
__device__ __forceinline__ float half_max(float v) {
    v = fmaxf(v, dpp<DPP_QUAD_XOR1>(v));
    v = fmaxf(v, dpp<DPP_QUAD_XOR2>(v));
    v = fmaxf(v, dpp<DPP_ROW_HALF_MIRROR>(v));
    v = fmaxf(v, dpp<DPP_ROW_ROR8>(v));
    return max_xor16(v);
}

// 16-byte accesses of rows that the boundary only requires to be 8-byte
// aligned (dword alignment is all that the hardware asks for).
typedef unsigned u32x4_a8 __attribute__((ext_vector_type(4), aligned(8)));

// One head's 256 values (8 per lane of a half-wave) as E4M3 with scale
// amax / 448 (1 if all zero): bytes = e4m3(v * (1 / scale)) (reference
// store_e4m3, qwen35.cu:1055-1065); !ok: nothing stored.
__device__ __forceinline__ void store_e4m3_half(const float (&v)[8], uint8_t* dst, float* scale, bool ok) {
    const int sub = threadIdx.x & 31;
    float amax = 0.f;
#pragma unroll
    for (int e = 0; e < 8; e++) amax = fmaxf(amax, fabsf(v[e]));
    amax = half_max(amax);
    const float sc = amax > 0.f ? amax / 448.f : 1.f;
    const float inv = 1.f / sc;
    if (!ok) return;
    uint32_t* d = reinterpret_cast<uint32_t*>(dst + 8 * sub);
    d[0] = f32x4_to_e4m3x4(v[0] * inv, v[1] * inv, v[2] * inv, v[3] * inv);
    d[1] = f32x4_to_e4m3x4(v[4] * inv, v[5] * inv, v[6] * inv, v[7] * inv);
    if (sub == 0) *scale = sc;
}

// The rotary factors a wave shares: bf16-rounded cos and sin of d = 0 .. 31.
struct PrepLds {
    float c[ROPE_DIM / 2], s[ROPE_DIM / 2];
};

// One wave, token t: units u0 .. u0 + P - 1 of the row's pairs of heads
// (PrepPairs). A pair is of one kind, so whether it is stored (q always, k and
// v with a slot) is one answer for the wave.
template <int P>
__device__ __forceinline__ void prep_units(const PrepArgs& a, PrepLds& lds, int t, int u0) {
    const int lane = threadIdx.x & 63, hv = lane >> 5, sub = lane & 31;
    const PrepPairs pairs(a.Hq, a.Hkv);
    const int nu = pairs.units();
    const uint16_t* row = a.qkv + (size_t)t * a.qstride;
    uint4 raw[P];
#pragma unroll
    for (int i = 0; i < P; i++) {
        // (past the last unit: the last one again, not stored)
        const int src = pairs.source(min(u0 + i, nu - 1), hv);  // in heads of 256
        const u32x4_a8 x = *reinterpret_cast<const u32x4_a8*>(row + (size_t)src * HEAD_DIM + 8 * sub);
        raw[i] = make_uint4(x.x, x.y, x.z, x.w);
    }
    const long slot = a.slot_map[t];
    const bool has_slot = slot >= 0 && slot < a.num_slots;
    // the norm weights of the lane's 8 dims: the unit's kind's (P = 1), else
    // q's and k's
    auto norm8 = [&](const float* n, float (&w)[8]) {
        const float4 w0 = *reinterpret_cast<const float4*>(n + 8 * sub);
        const float4 w1 = *reinterpret_cast<const float4*>(n + 8 * sub + 4);
        w[0] = w0.x, w[1] = w0.y, w[2] = w0.z, w[3] = w0.w;
        w[4] = w1.x, w[5] = w1.y, w[6] = w1.z, w[7] = w1.w;
    };
    float wq[8], wk[8];
    norm8(P == 1 && !pairs.is_q(u0) ? a.k_norm : a.q_norm, wq);
    if (P > 1) norm8(a.Hkv > 0 ? a.k_norm : a.q_norm, wk);
    {
        // cos / sin of d = sub
        const int d = sub;
        const int axis = (d % 3 == 1 && d < 3 * a.sec_h) ? 1 : (d % 3 == 2 && d < 3 * a.sec_w) ? 2 : 0;
        const float f = (float)a.rope[(size_t)axis * a.rope_stride + t] * a.inv_freq[d];
        float s, c;
        sincosf(f, &s, &c);
        if (lane < ROPE_DIM / 2) {
            lds.c[d] = rbf(c);
            lds.s[d] = rbf(s);
        }
    }
    wave_sync();
    // The factors of this lane's 8 dims (lanes 0 .. 7 of the half-wave
    // rotate): y' = bf16(bf16(own c) + bf16(partner s)), the sine negated on
    // the lanes of dims 0 .. 31.
    const bool rot = sub < ROPE_DIM / 8;
    float c8[8], s8[8];
#pragma unroll
    for (int e = 0; e < 8; e++) {
        c8[e] = lds.c[8 * (sub & 3) + e];
        s8[e] = lds.s[8 * (sub & 3) + e];
        if (sub < ROPE_DIM / 16) s8[e] = -s8[e];
    }
#pragma unroll
    for (int i = 0; i < P; i++) {
        const int u = u0 + i;
        if (u >= nu) break;
        const bool is_q = pairs.is_q(u), is_v = pairs.is_v(u);
        if (!is_q && !has_slot) break;  // (k and v units follow q's)
        const int h = pairs.head(u, hv);
        const bool ok = pairs.has(u, hv);
        uint32_t y[4] = {raw[i].x, raw[i].y, raw[i].z, raw[i].w};
        float x[8];
#pragma unroll
        for (int e = 0; e < 4; e++) {
            x[2 * e] = bf_lo(y[e]);
            x[2 * e + 1] = bf_hi(y[e]);
        }
        if (!is_v) {
            const float ss = half_sum2(x[0] * x[0] + x[1] * x[1] + x[2] * x[2] + x[3] * x[3],
                                       x[4] * x[4] + x[5] * x[5] + x[6] * x[6] + x[7] * x[7]);
            const float scale = 1.f / sqrtf(ss / HEAD_DIM + a.eps);
            float w[8];
#pragma unroll
            for (int e = 0; e < 8; e++) w[e] = P > 1 && !is_q ? wk[e] : wq[e];
#pragma unroll
            for (int e = 0; e < 4; e++)
                y[e] = pack2_hw(x[2 * e] * scale * w[2 * e], x[2 * e + 1] * scale * w[2 * e + 1]);
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const uint32_t yp = dpp_xor4(y[e]);
                const uint32_t yc = pack2_hw(bf_lo(y[e]) * c8[2 * e], bf_hi(y[e]) * c8[2 * e + 1]);
                const uint32_t ys = pack2_hw(bf_lo(yp) * s8[2 * e], bf_hi(yp) * s8[2 * e + 1]);
                const uint32_t r = pack2_hw(bf_lo(yc) + bf_lo(ys), bf_hi(yc) + bf_hi(ys));
                y[e] = rot ? r : y[e];
            }
        }
        if (is_q) {
            *reinterpret_cast<u32x4_a8*>(a.qout + ((size_t)t * a.Hq + h) * HEAD_DIM + 8 * sub) =
                u32x4_a8{y[0], y[1], y[2], y[3]};
            continue;
        }
        uint16_t* cache = is_v ? a.vcache : a.kcache;
        const size_t at = (size_t)slot * a.Hkv + h;
        if (a.kscale) {
#pragma unroll
            for (int e = 0; e < 4; e++) {
                x[2 * e] = bf_lo(y[e]);
                x[2 * e + 1] = bf_hi(y[e]);
            }
            store_e4m3_half(x, reinterpret_cast<uint8_t*>(cache) + at * HEAD_DIM, (is_v ? a.vscale : a.kscale) + at,
                            ok);
        } else if (ok) {
            *reinterpret_cast<u32x4_a8*>(cache + at * HEAD_DIM + 8 * sub) = u32x4_a8{y[0], y[1], y[2], y[3]};
        }
    }
}

// P units per wave, groups = ceil(units / P) waves per token, wave i of the
// launch taking group i % groups of token i / groups. 256 threads.
template <int P>
__global__ void __launch_bounds__(256) prep_kernel(PrepArgs a, int T, int groups) {
    __shared__ PrepLds lds[4];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const long i = (long)blockIdx.x * 4 + wave;
    const int t = (int)(i / groups), u0 = (int)(i % groups) * P;
    if (t < T) prep_units<P>(a, lds[wave], t, u0);
}

}  // namespace pkv
