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
// What bounds it: the latency of the loads, a K-tile taking about as long as a round trip to L2 (333 x 1001 x 1160, 96
// workgroups: 10.1 us for 0.8 GOP; 1536 us with one thread per output, the form this kernel replaces).
template <int OUT, int BM, int BN>
__global__ __launch_bounds__(256) void gemm_i8_ragged_kernel(const GemmArgs g) {
    constexpr int BK = 128, MI = BM / 64, NJ = BN / 64;
    constexpr int XC = BM * 8 / 256, WC = BN * 8 / 256;  // 16-byte chunks per thread and K-tile
    constexpr int STAGE = (BM + BN) * BK;
    constexpr int PITCH = BN + 4;                         // ints per row of the output tile in LDS
    constexpr int SMEM = 2 * STAGE > BM * PITCH * 4 ? 2 * STAGE : BM * PITCH * 4;
    static_assert(SMEM <= 160 * 1024 && 256 % BN == 0, "LDS; a thread keeps one column in the epilogue");
    __shared__ __attribute__((aligned(16))) char smem[SMEM];

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave >> 1, wn = wave & 1, l32 = lane & 31, lhalf = lane >> 5;
    const int tiles_m = (g.M + BM - 1) / BM;
    const int m0 = (int)(blockIdx.x % (unsigned)tiles_m) * BM, n0 = (int)(blockIdx.x / (unsigned)tiles_m) * BN;
    const int K = g.K, KT = (K + BK - 1) / BK;

    const int8_t *src[XC + WC];   // this thread's chunks at K-tile 0; rows past the end repeat the last one (never stored)
    int dst[XC + WC];
    const int c = tid & 7;
#pragma unroll
    for (int t = 0; t < XC + WC; ++t) {
        const bool is_x = t < XC;
        const int row = (is_x ? t : t - XC) * 32 + (tid >> 3);
        src[t] = (is_x ? g.x + (int64_t)min(m0 + row, g.M - 1) * K : g.w + (int64_t)min(n0 + row, g.N - 1) * K) + c * 16;
        dst[t] = (is_x ? 0 : BM * BK) + row * BK + (c ^ swz<8>(row)) * 16;
    }
    v4i reg[2][XC + WC];
    auto fetch = [&](int kt, v4i (&r)[XC + WC]) __attribute__((always_inline)) {
        const int kb = kt * BK;
        if (kb + BK <= K) {
#pragma unroll
            for (int t = 0; t < XC + WC; ++t) __builtin_memcpy(&r[t], src[t] + kb, 16);
        } else {
#pragma unroll
            for (int t = 0; t < XC + WC; ++t) {
                const int left = K - kb - c * 16;  // bytes of the row from this chunk on
                uint64_t lo = 0, hi = 0;
                if (K >= 16) {  // the row's last 16 bytes, moved down by what precedes the chunk in them
                    v4i v;
                    __builtin_memcpy(&v, src[t] + kb + (left < 16 ? left - 16 : 0), 16);
                    lo = (uint32_t)v.x | (uint64_t)(uint32_t)v.y << 32, hi = (uint32_t)v.z | (uint64_t)(uint32_t)v.w << 32;
                    const int sh = left >= 16 ? 0 : (left > 0 ? (16 - left) * 8 : 128);
                    if (sh >= 128) lo = hi = 0;
                    else if (sh >= 64) lo = hi >> (sh - 64), hi = 0;
                    else if (sh > 0) lo = lo >> sh | hi << (64 - sh), hi >>= sh;
                } else {
                    for (int e = 0; e < left; ++e) {
                        const uint64_t b = (uint8_t)src[t][e];
                        if (e < 8) lo |= b << (8 * e);
                        else hi |= b << (8 * (e - 8));
                    }
                }
                r[t] = v4i{(int)(uint32_t)lo, (int)(uint32_t)(lo >> 32), (int)(uint32_t)hi, (int)(uint32_t)(hi >> 32)};
            }
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
#pragma unroll
        for (int t = 0; t < XC + WC; ++t) *(v4i *)(st + dst[t]) = r[t];
        if (kt + 2 < KT) fetch(kt + 2, r);
        // (a bare barrier: __syncthreads() would also wait for the loads of the next K-tiles)
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) {
            const int ko = ((ks * 2 + lhalf) ^ sw) * 16;
            v4i xf[MI], wf[NJ];
#pragma unroll
            for (int i = 0; i < MI; ++i) xf[i] = *(const v4i *)(st + (wm * (BM / 2) + i * 32 + l32) * BK + ko);
#pragma unroll
            for (int j = 0; j < NJ; ++j) wf[j] = *(const v4i *)(st + BM * BK + (wn * (BN / 2) + j * 32 + l32) * BK + ko);
#pragma unroll
            for (int i = 0; i < MI; ++i)
#pragma unroll
                for (int j = 0; j < NJ; ++j) acc[i][j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(wf[j], xf[i], acc[i][j], 0, 0, 0);
        }
    };
    if (KT > 0) fetch(0, reg[0]);
    if (KT > 1) fetch(1, reg[1]);
    for (int kt = 0; kt < KT; kt += 2) {
        step(kt, reg[0], smem);
        if (kt + 1 < KT) step(kt + 1, reg[1], smem + STAGE);
    }

    __syncthreads();
    int *const tile = (int *)smem;
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int j = 0; j < NJ; ++j)
#pragma unroll
            for (int qd = 0; qd < 4; ++qd)
                *(v4i *)(tile + (wm * (BM / 2) + i * 32 + l32) * PITCH + wn * (BN / 2) + j * 32 + qd * 8 + lhalf * 4) =
                    v4i{acc[i][j][4 * qd], acc[i][j][4 * qd + 1], acc[i][j][4 * qd + 2], acc[i][j][4 * qd + 3]};
    __syncthreads();
    const int n = n0 + tid % BN;
    if (n >= g.N) return;
    float ws = 0.0f, b = 0.0f;
    if constexpr (OUT != OUT_I32) {
        ws = g.ws ? g.ws[g.row_scale ? n : 0] : g.ws_host;
        if (g.bias) {
            if (g.bias_dtype == I8F_F32) b = ((const float *)g.bias)[n];
            else if (g.bias_dtype == I8F_BF16) b = bf16_bits_to_f32(((const uint16_t *)g.bias)[n]);
            else b = f16_bits_to_f32(((const uint16_t *)g.bias)[n]);
        }
    }
#pragma unroll 4
    for (int row = tid / BN; row < BM; row += 256 / BN) {
        if (m0 + row < g.M) finish_one<OUT>(g, tile[row * PITCH + tid % BN], m0 + row, n, OUT == OUT_I32 ? 0.0f : g.xs[m0 + row], ws, b);
    }
}

template <int OUT>
int launch_ragged(const GemmArgs &g, hipStream_t st) {
    const int64_t t128 = (((int64_t)g.M + 127) / 128) * (((int64_t)g.N + 127) / 128);
    const int64_t t64 = (((int64_t)g.M + 63) / 64) * (((int64_t)g.N + 63) / 64);
    // 128 x 128 tiles once they fill two workgroups on every CU: they fetch half the bytes per product, but a CU with one or two
    // of them has too few loads in flight (2500 x 2501 x 1160, 400 tiles: 33.1 us against 29.0 with 64 x 64 tiles, four or
    // five workgroups to a CU; 4096 x 3071 x 3083, 768 tiles: 102 us against 123)
    if (t128 >= 512) hipLaunchKernelGGL((gemm_i8_ragged_kernel<OUT, 128, 128>), dim3((unsigned)t128), dim3(256), 0, st, g);
    else hipLaunchKernelGGL((gemm_i8_ragged_kernel<OUT, 64, 64>), dim3((unsigned)t64), dim3(256), 0, st, g);
    return check_launch();
}

}  // namespace gemm
}  // namespace i8f
