// What the kernels of the stochastic-rounding merge share: the rounding itself, the packed saturating add, and the numbers that
// torch.rand draws.
#pragma once

#include "i8f_common.hpp"
#include "../../include/i8f_drawn.h"

namespace i8f {
namespace {

__device__ __forceinline__ float sr_round(float xs, float noise) {
    const float f = floorf(xs);
    const float frac = xs - f;
    const float v = noise < frac ? f + 1.0f : f;
    return fminf(fmaxf(v, -128.0f), 127.0f);  // NaN becomes -128
}

__device__ __forceinline__ int sat8(int v) { return min(max(v, -128), 127); }

// sat8(w + r) for four int8 weights packed in wp and four integer-valued r in [-128, 127], packed again.  With both
// moved up by 128 the sum is a float in [0, 510] minus 128 and the saturating float-to-byte conversion does the clamp.
__device__ __forceinline__ uint32_t add_sat8_pack(uint32_t wp, const float (&r)[4]) {
    const uint32_t u = wp ^ 0x80808080u;
    uint32_t o = 0;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const float t = (float)((u >> (8 * e)) & 0xffu) + r[e];
        o = __builtin_amdgcn_cvt_pk_u8_f32(t, e, o);  // v_cvt_pk_u8_f32 clamps to 0..255
    }
    return o ^ 0x80808080u;
}

// What torch.rand writes on this GPU from a freshly seeded generator: element e, with i = e / lanes (lanes: the threads of its
// launch), is made of word i % 4 of Philox 4x32-10 (Salmon, Moraes, Dror and Shaw, "Parallel random numbers: as easy as 1, 2, 3",
// 2011) with the seed as key and the counter (i / 4, 0, e % lanes, 0).
__device__ __forceinline__ uint32_t xor3(uint32_t a, uint32_t b, uint32_t c) { return __builtin_amdgcn_bitop3_b32(a, b, c, 0x96); }

__device__ __forceinline__ void philox(uint32_t position, uint32_t lane, uint32_t k0, uint32_t k1, uint32_t (&out)[4]) {
    constexpr uint32_t M0 = 0xD2511F53u, M1 = 0xCD9E8D57u, W0 = 0x9E3779B9u, W1 = 0xBB67AE85u;
    uint32_t c0 = position, c1 = 0, c2 = lane, c3 = 0;
#pragma unroll
    for (int i = 0; i < 10; ++i) {
        const uint64_t p0 = (uint64_t)M0 * c0, p1 = (uint64_t)M1 * c2;
        c0 = xor3((uint32_t)(p1 >> 32), c1, k0 + W0 * i), c1 = (uint32_t)p1;
        c2 = xor3((uint32_t)(p0 >> 32), c3, k1 + W1 * i), c3 = (uint32_t)p0;
    }
    out[0] = c0, out[1] = c1, out[2] = c2, out[3] = c3;
}

// the uniform number of a word: in (0, 1], and 1 is handed out as 0
constexpr uint32_t ONE_WORDS = 0xffffff80u;  // words from here on round to 1
__device__ __forceinline__ float uniform_of(uint32_t x) {
    return x >= ONE_WORDS ? 0.0f : __builtin_fmaf((float)x, 0x1p-32f, 0x1p-32f);
}

constexpr int MAX_FACTORS = 8;
int64_t up256(int64_t bytes) { return (bytes + 255) / 256 * 256; }

}  // namespace

// A checked call of i8f_lora_merge_sr_drawn, and its form for few elements (lora_merge.hip), of ranks up to FEW_MAX_RANK.
struct DrawnCall {
    const int8_t *w;
    const float *ws;
    float ws_host;
    bool row_scale;
    const i8f_lora_factors *factors;
    int count, rank;   // rank: the sum
    float lora_scale;
    uint64_t seed;
    int64_t lanes, N, K;
    int8_t *out;
    void *workspace;
};
constexpr int64_t FEW_MAX_RANK = 224;
int64_t merge_few_workspace_bytes(int64_t N, int64_t K, int64_t rank, int count);
int merge_few(const DrawnCall &c, hipStream_t st);

}  // namespace i8f
