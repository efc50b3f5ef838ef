// The int8 GEMM for operands that the tiled kernel's 16-byte direct global -> LDS loads and 16-byte stores do not fit:
// K % 16 != 0, N % 8 != 0, pointers that are not 16-byte aligned, matrices of 2^31 bytes and more.
#pragma once

#include "i8f_common.hpp"

namespace i8f {
namespace gemm {

// One output from its accumulator: the epilogue of the tiled kernel for one element.
template <int OUT>
__device__ __forceinline__ void finish_one(const GemmArgs &g, int acc, int m, int n, float xs, float ws, float b) {
    const int64_t idx = (int64_t)m * g.N + n;
    if constexpr (OUT == OUT_I32) {
        ((int *)g.out)[idx] = acc;
    } else {
        constexpr int DT = OUT == OUT_BF16 ? I8F_BF16 : (OUT == OUT_F16 ? I8F_F16 : I8F_F32);
        const float a = (float)acc;
        float t;
        if (g.order == I8F_EPI_TORCH) {
            if (g.row_scale) {
                t = a * xs;
                t = t * ws;
            } else {
                const float sc = ws * xs;
                t = a * sc;
            }
            t = round_to_dtype<DT>(t);
            if (g.bias) t = t + round_to_dtype<DT>(b);
        } else {
            const float sc = xs * ws;
            t = a * sc;
            if (g.bias) t = t + b;
        }
        if (g.gate) t = round_to_dtype<DT>(t) * load_as_f32<DT>(g.gate, (int64_t)(m / g.gate_rows) * g.N + n);
        if (g.addend) t = round_to_dtype<DT>(t) + load_as_f32<DT>(g.addend, idx);
        store_from_f32<DT>(g.out, idx, t);
    }
}

// Four waves compute a BM x BN tile (a quarter each) with v_mfma_i32_32x32x32_i8 over K-tiles of 128 bytes.  A thread
// fetches 16-byte chunks of operand rows from whatever byte address they have (the hardware splits a load that straddles a
// line) into registers, two K-tiles ahead, and writes them to LDS in the swizzled layout of the tiled kernel; a row's
// last chunk, where K is no multiple of 16, is cut from the 16 bytes that end the row, so nothing outside the matrices is read.
// LDS is double-buffered: one barrier per K-tile.  The accumulators go through LDS once more so that a wave stores whole
// runs of a row, element by element: rows of N outputs start at any address.
// TINY: K < 16, where a row has no 16 bytes to end it.
// GROUPS of four waves take every GROUPS-th K-tile each, with stages of their own, and their sums meet in LDS in the epilogue:
// integers, so that the order changes nothing.
// What bounds it: 333 x 1001 x 1160 (96 workgroups) 7.5 us, 3 of them the launch, the first loads and the epilogue, then 0.9 us
// a pair of K-tiles: the chain from LDS write to product, and half as much again for chunks that straddle lines.  One group, and
// so ten links instead of five, takes 9.1 us, four groups 8.3 (17 x 1500 x 1500 7.9, 6.4 and 6.9; 500 x 1400 x 1400 9.8, 8.1 and 9.0); 4096 x 3071 x 3083
// 90 us, the loads of the two workgroups of a CU.  Two things made it that: the loads of a K-tile are issued without a branch
// or a use near them (the compiler put a wait for all loads in flight at each join: 11.8 and 110 us before), and the
// epilogue's operands come first instead of last.  Two waves to a SIMD is what the registers have to leave room for: with one
// the larger shape takes 119 us.
// PAST: past the last K-tile (loads ahead, groups without one) every lane fetches the same 16 bytes; else the last K-tile again.
// K-tiles that nobody needs are as many as needed ones where K is short, and with K odd their chunks cost as much as any: us, one group,
// two without and with PAST, 30 x 301 x 17 5.0, 5.5 and 4.4, 35 x 967 x 257 5.8, 6.4 and 5.7, 512 x 2041 x 121 6.2, 6.5 and 5.5.  With K a
// multiple of 4 they cost little and the selection of addresses as much: a layer of 333 x 1160 into 1001 in a row 10.20 without, 10.46 with it.
template <int OUT, int BM, int BN, bool TINY, int GROUPS, bool PAST>
__global__ __launch_bounds__((256 * GROUPS), (GROUPS < 2 ? 2 : GROUPS)) void gemm_i8_ragged_kernel(const GemmArgs g) {
    constexpr int AHEAD = 2;  // K-tiles in flight (4, 6 and 8 measured the same or slower)
    constexpr int BK = 128, MI = BM / 64, NJ = BN / 64;
    constexpr int XC = BM * 8 / 256, WC = BN * 8 / 256;  // 16-byte chunks per thread and K-tile
    constexpr int STAGE = (BM + BN) * BK;
    constexpr int PITCH = BN + 4;                         // ints per row of the output tile in LDS
    constexpr int SMEM_GROUP = 2 * STAGE > BM * PITCH * 4 ? 2 * STAGE : BM * PITCH * 4, SMEM = GROUPS * SMEM_GROUP;
    static_assert(SMEM + BM * 4 <= 160 * 1024 && 256 % BN == 0, "LDS; a thread keeps one column in the epilogue");
    __shared__ __attribute__((aligned(16))) char smem[SMEM];
    __shared__ float s_xs[BM];

    const int group = GROUPS == 1 ? 0 : __builtin_amdgcn_readfirstlane(threadIdx.x >> 8);
    const int tid = threadIdx.x & 255, lane = tid & 63;   // within the group of four waves
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave >> 1, wn = wave & 1, l32 = lane & 31, lhalf = lane >> 5;
    const int tiles_m = (g.M + BM - 1) / BM;
    const int m0 = (int)(blockIdx.x % (unsigned)tiles_m) * BM, n0 = (int)(blockIdx.x / (unsigned)tiles_m) * BN;
    const int K = g.K, KT = (int)(((int64_t)K + BK - 1) / BK);

    // the epilogue's operands, requested in front of everything else: the thread's column, and (for all) the tile's rows
    const int n = n0 + tid % BN;
    float ws = 0.0f, b = 0.0f, xs = 0.0f;
    if constexpr (OUT != OUT_I32) {
        const int nc = min(n, g.N - 1);
        ws = g.ws ? g.ws[g.row_scale ? nc : 0] : g.ws_host;
        if (g.bias) {
            if (g.bias_dtype == I8F_F32) b = ((const float *)g.bias)[nc];
            else if (g.bias_dtype == I8F_BF16) b = bf16_bits_to_f32(((const uint16_t *)g.bias)[nc]);
            else b = f16_bits_to_f32(((const uint16_t *)g.bias)[nc]);
        }
        if ((int)threadIdx.x < BM) xs = g.xs[min(m0 + tid, g.M - 1)];
    }

    const int8_t *src[XC + WC];   // the rows of this thread's chunks; rows past the end repeat the last one (never stored)
    int dst[XC + WC];
    const int c = tid & 7;
#pragma unroll
    for (int t = 0; t < XC + WC; ++t) {
        const bool is_x = t < XC;
        const int row = (is_x ? t : t - XC) * 32 + (tid >> 3);
        src[t] = is_x ? g.x + (int64_t)min(m0 + row, g.M - 1) * K : g.w + (int64_t)min(n0 + row, g.N - 1) * K;
        dst[t] = (is_x ? 0 : BM * BK) + row * BK + (c ^ swz<8>(row)) * 16;
    }
    v4i reg[AHEAD][XC + WC];
    // A K-tile's loads and nothing else: no branch and no use of what they bring, or the compiler would wait for all of them here.
    auto fetch = [&](int kt, v4i (&r)[XC + WC]) __attribute__((always_inline)) {
        if constexpr (TINY) {  // K < 16: the only chunk with bytes in it is the first
#pragma unroll
            for (int t = 0; t < XC + WC; ++t) {
                uint32_t b[4] = {0, 0, 0, 0};
#pragma unroll
                for (int e = 0; e < 15; ++e)
                    if (c == 0 && e < K) b[e / 4] |= (uint32_t)(uint8_t)src[t][e] << (8 * (e % 4));
                r[t] = v4i{(int)b[0], (int)b[1], (int)b[2], (int)b[3]};
            }
        } else {
            const bool there = !PAST || kt < KT;
            const uint32_t pos = min((uint32_t)(PAST ? kt : min(kt, KT - 1)) * BK + c * 16, (uint32_t)K - 16);
#pragma unroll
            for (int t = 0; t < XC + WC; ++t) __builtin_memcpy(&r[t], there ? src[t] + pos : g.w, 16);
        }
    };
    // of the last K-tile's chunks, which end with the row: what precedes the chunk in them is shifted out
    const int left = K - (KT - 1) * BK - c * 16;
    const int sh = TINY || left >= 16 ? 0 : (left > 0 ? (16 - left) * 8 : 128);
    auto cut_tail = [&](v4i (&r)[XC + WC]) __attribute__((always_inline)) {
#pragma unroll
        for (int t = 0; t < XC + WC; ++t) {
            uint64_t lo = (uint32_t)r[t].x | (uint64_t)(uint32_t)r[t].y << 32, hi = (uint32_t)r[t].z | (uint64_t)(uint32_t)r[t].w << 32;
            if (sh >= 128) lo = hi = 0;
            else if (sh >= 64) lo = hi >> (sh - 64), hi = 0;
            else if (sh > 0) lo = lo >> sh | hi << (64 - sh), hi >>= sh;
            r[t] = v4i{(int)(uint32_t)lo, (int)(uint32_t)(lo >> 32), (int)(uint32_t)hi, (int)(uint32_t)(hi >> 32)};
        }
    };

    v16i acc[MI][NJ];
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int j = 0; j < NJ; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[i][j][r] = 0;

    const int sw = swz<8>(l32);
    auto step = [&](int kt, v4i (&r)[XC + WC], char *st) __attribute__((always_inline)) {
        if (kt == KT - 1) cut_tail(r);
#pragma unroll
        for (int t = 0; t < XC + WC; ++t) *(v4i *)(st + dst[t]) = r[t];
        if constexpr (!TINY) fetch(kt + AHEAD * GROUPS, r);
        // (a bare barrier: __syncthreads() would also wait for the loads of the next K-tiles)
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
        if (GROUPS > 1 && kt >= KT) return;   // (the other groups' last K-tiles)
        // (the small tile has one product per wave and k-step: all of its fragments first, one LDS latency instead of four)
        constexpr int AT_ONCE = MI * NJ == 1 ? 4 : 1;
#pragma unroll
        for (int k0 = 0; k0 < 4; k0 += AT_ONCE) {
            v4i xf[AT_ONCE][MI], wf[AT_ONCE][NJ];
#pragma unroll
            for (int u = 0; u < AT_ONCE; ++u) {
                const int ko = (((k0 + u) * 2 + lhalf) ^ sw) * 16;
#pragma unroll
                for (int i = 0; i < MI; ++i) xf[u][i] = *(const v4i *)(st + (wm * (BM / 2) + i * 32 + l32) * BK + ko);
#pragma unroll
                for (int j = 0; j < NJ; ++j) wf[u][j] = *(const v4i *)(st + BM * BK + (wn * (BN / 2) + j * 32 + l32) * BK + ko);
            }
            if constexpr (AT_ONCE > 1) __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int u = 0; u < AT_ONCE; ++u)
#pragma unroll
                for (int i = 0; i < MI; ++i)
#pragma unroll
                    for (int j = 0; j < NJ; ++j) acc[i][j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(wf[u][j], xf[u][i], acc[i][j], 0, 0, 0);
        }
    };
    if (KT > 0) {
#pragma unroll
        for (int u = 0; u < (TINY ? 1 : AHEAD); ++u) {
            fetch(u * GROUPS + group, reg[u]);
            __builtin_amdgcn_sched_barrier(0);  // (in the order in which they are waited for)
        }
    }
    for (int kt = 0; kt < KT; kt += AHEAD * GROUPS) {
#pragma unroll
        for (int u = 0; u < AHEAD; ++u) {
            if (kt + u * GROUPS >= KT) break;
            step(kt + u * GROUPS + group, reg[u], smem + group * SMEM_GROUP + (u & 1) * STAGE);
        }
    }

    __syncthreads();
    int *const tile = (int *)(smem + group * SMEM_GROUP);
    if ((int)threadIdx.x < BM) s_xs[tid] = xs;
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int j = 0; j < NJ; ++j)
#pragma unroll
            for (int qd = 0; qd < 4; ++qd)
                *(v4i *)(tile + (wm * (BM / 2) + i * 32 + l32) * PITCH + wn * (BN / 2) + j * 32 + qd * 8 + lhalf * 4) =
                    v4i{acc[i][j][4 * qd], acc[i][j][4 * qd + 1], acc[i][j][4 * qd + 2], acc[i][j][4 * qd + 3]};
    __syncthreads();
    if (n >= g.N) return;
#pragma unroll 8
    for (int row = (int)threadIdx.x / BN; row < BM; row += 256 * GROUPS / BN) {
        if (m0 + row < g.M) {
            int sum = 0;
#pragma unroll
            for (int o = 0; o < GROUPS; ++o) sum += ((const int *)(smem + o * SMEM_GROUP))[row * PITCH + tid % BN];
            finish_one<OUT>(g, sum, m0 + row, n, OUT == OUT_I32 ? 0.0f : s_xs[row], ws, b);
        }
    }
}

template <int OUT>
int launch_ragged(const GemmArgs &g, hipStream_t st) {
    const int64_t t128 = (((int64_t)g.M + 127) / 128) * (((int64_t)g.N + 127) / 128);
    const int64_t t64 = (((int64_t)g.M + 63) / 64) * (((int64_t)g.N + 63) / 64);
    // 128 x 128 tiles once there is one for every CU: half the bytes per product (1024 x 3001 x 3083, 192 tiles: 40.0 us
    // against 41.4 with 64 x 64 tiles; 2500 x 2501 x 1160, 400 tiles: 26.7 both; 2100 x 3001 x 3083, 408 tiles: 62 against
    // 83); below that they leave CUs idle (1500 x 1500 x 1500, 144 tiles: 21.9 against 16.2).
    auto launch = [&](auto PAST) {
        constexpr bool P = decltype(PAST)::value;
        if (t128 >= 256) hipLaunchKernelGGL((gemm_i8_ragged_kernel<OUT, 128, 128, false, 1, P>), dim3((unsigned)t128), dim3(256), 0, st, g);
        else if (t64 <= 256) hipLaunchKernelGGL((gemm_i8_ragged_kernel<OUT, 64, 64, false, 2, P>), dim3((unsigned)t64), dim3(512), 0, st, g);
        else hipLaunchKernelGGL((gemm_i8_ragged_kernel<OUT, 64, 64, false, 1, P>), dim3((unsigned)t64), dim3(256), 0, st, g);
    };
    if (g.K < 16) hipLaunchKernelGGL((gemm_i8_ragged_kernel<OUT, 64, 64, true, 1, false>), dim3((unsigned)t64), dim3(256), 0, st, g);
    else if (g.K % 4) launch(std::true_type{});
    else launch(std::false_type{});
    return check_launch();
}

}  // namespace gemm
}  // namespace i8f
