// The row-wise quantiser with the first product of a dynamic LoRA beside it (included by quant_rowwise.hip).
#include "quant_lora_entry.hpp"

namespace i8f {
namespace {

typedef float v4f __attribute__((ext_vector_type(4)));
typedef uint32_t v4u __attribute__((ext_vector_type(4)));
typedef __bf16 v8bf __attribute__((ext_vector_type(8)));
typedef _Float16 v8h __attribute__((ext_vector_type(8)));

template <int DT>
__device__ __forceinline__ v4f lora_mfma(v4u a, v4u b, v4f c) {
    if constexpr (DT == I8F_BF16) return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(v8bf, a), __builtin_bit_cast(v8bf, b), c, 0, 0, 0);
    else return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(v8h, a), __builtin_bit_cast(v8h, b), c, 0, 0, 0);
}

// q and scale of 16 rows of x as quant16_kernel leaves them, and t = x A^T [M, 16 RT] of the rows' dtype (binary32 sums, one
// rounding); x is read once for both.  Eight waves share the rows: wave w takes blocks w, w + 8, ... of 64 columns of all
// sixteen.  Eight neighbouring lanes load the 128 bytes of a row, of x and of A alike, and the tiles change to the matrix
// unit's layout in LDS of the wave's own.  Loading that layout directly, with neighbouring lanes in different rows, moves 16
// bytes a cycle and CU, and took 11.4 us at 1357 x 3072, rank 32.  us of a launch in a replayed graph, against the quantiser's
// and that of the BLAS library's product, on one x and on twelve in turn (from HBM): 1357 x 3072, rank 32 7.3 against 2.9 +
// 6.5 and 7.8 against 3.7 + 7.7 (a profiler shows 8.5); 4608 rows 13.9, 4.7 + 8.2 and 18.1, 8.9 + 11.9; 9729 rows 24.0, 13.9 + 13.0
// and 27.6, 16.7 + 16.6; 16384 rows, rank 64 44.4, 22.0 + 18.7 and 48.5, 26.6 + 23.3.  Bound by a CU's loads: 16 rows of x and the whole of A, 290 KB of them, for each workgroup; with more rows to share A
// the chip would stand idle at the sizes where it matters, and registers for two workgroups a CU (128) spill: 15.2 -> 17.9.
// BLOCKS: 64-column blocks to a wave at most; FEWEST: that every wave has.
template <int DT, int RT, int BLOCKS, int FEWEST>
__global__ __launch_bounds__(512) void quant_lora_kernel(const char *__restrict__ x, int M, int K, int64_t ldx_bytes, const char *__restrict__ la,
                                                         int8_t *__restrict__ q, float *__restrict__ scale, char *__restrict__ t) {
    __shared__ float s_max[8][16];
    __shared__ union {
        v4u tile[8][1 + RT][128];  // [wave][x, A...][row * 8 + (16-byte chunk ^ row & 7)]
        v4f sum[8][RT][64];
    } sh;
    constexpr int AHEAD = RT == 1 ? 4 : RT == 2 ? 3 : 1;  // blocks of A under way beyond the one in use
    const int tid = threadIdx.x, lane = tid & 63, r = lane >> 3, c = lane & 7;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int row = blockIdx.x * 16 + r, blocks = K / 64;  // (the lane's rows: row and row + 8)
    const char *x0 = x + (int64_t)min(row, M - 1) * ldx_bytes + c * 16, *x1 = x + (int64_t)min(row + 8, M - 1) * ldx_bytes + c * 16;
    const char *ar = la + (int64_t)r * K * 2 + c * 16;
    const int64_t eight = (int64_t)16 * K;  // bytes of eight rows of A
    v4u xv[BLOCKS][2], a[BLOCKS][RT][2];
    auto fetch = [&](int b) {
        const int off = (b < FEWEST || wave + 8 * b < blocks ? wave + 8 * b : 0) * 128;
#pragma unroll
        for (int i = 0; i < RT; ++i) a[b][i][0] = *(const v4u *)(ar + 2 * i * eight + off), a[b][i][1] = *(const v4u *)(ar + (2 * i + 1) * eight + off);
    };
#pragma unroll
    for (int b = 0; b < BLOCKS; ++b) {
        const int off = (b < FEWEST || wave + 8 * b < blocks ? wave + 8 * b : 0) * 128;
        xv[b][0] = *(const v4u *)(x0 + off), xv[b][1] = *(const v4u *)(x1 + off);
        if (b < AHEAD) fetch(b);
    }
    __builtin_amdgcn_sched_barrier(0);
    v4f acc[RT];
#pragma unroll
    for (int i = 0; i < RT; ++i) acc[i] = (v4f)0.0f;
    float m0 = 0.0f, m1 = 0.0f;
    v4u(*tile)[128] = sh.tile[wave];
    const int put = r * 8 + (c ^ r), fr = lane & 15, fg = lane >> 4;
#pragma unroll
    for (int b = 0; b < BLOCKS; ++b) {
        if (b + AHEAD < BLOCKS) fetch(b + AHEAD);
        __builtin_amdgcn_sched_barrier(0);
        if (b < FEWEST || wave + 8 * b < blocks) {
            tile[0][put] = xv[b][0], tile[0][put + 64] = xv[b][1];
#pragma unroll
            for (int i = 0; i < RT; ++i) tile[1 + i][put] = a[b][i][0], tile[1 + i][put + 64] = a[b][i][1];
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            __builtin_amdgcn_wave_barrier();
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const int get = fr * 8 + ((4 * h + fg) ^ (fr & 7));
                const v4u xf = tile[0][get];
#pragma unroll
                for (int i = 0; i < RT; ++i) acc[i] = lora_mfma<DT>(tile[1 + i][get], xf, acc[i]);
            }
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            __builtin_amdgcn_wave_barrier();
            float v[16];
            expand16<DT>(__builtin_bit_cast(uint4, xv[b][0]), __builtin_bit_cast(uint4, xv[b][1]), v);
#pragma unroll
            for (int j = 0; j < 8; j += 2) m0 = max3_abs(m0, v[j], v[j + 1]), m1 = max3_abs(m1, v[8 + j], v[9 + j]);
        }
    }
#pragma unroll
    for (int d = 1; d < 8; d *= 2) m0 = fmaxf(m0, __shfl_xor(m0, d)), m1 = fmaxf(m1, __shfl_xor(m1, d));
    if (c == 0) s_max[wave][r] = m0, s_max[wave][r + 8] = m1;
    __syncthreads();  // (the tiles are done with)
#pragma unroll
    for (int i = 0; i < RT; ++i) sh.sum[wave][i][lane] = acc[i];
#pragma unroll
    for (int w = 0; w < 8; ++w) m0 = fmaxf(m0, s_max[w][r]), m1 = fmaxf(m1, s_max[w][r + 8]);
    float s0, s1, i0, i1;
    scale_and_inverse16<true>(m0, s0, i0);
    scale_and_inverse16<true>(m1, s1, i1);
    int8_t *q0 = q + (int64_t)row * K + c * 8, *q1 = q0 + (int64_t)8 * K;
#pragma unroll
    for (int b = 0; b < BLOCKS; ++b) {
        float v[16];
        expand16<DT>(__builtin_bit_cast(uint4, xv[b][0]), __builtin_bit_cast(uint4, xv[b][1]), v);
        const uint4 o = quant16_magic(v, i0, i1);
        if (b < FEWEST || wave + 8 * b < blocks) {
            const int off = (wave + 8 * b) * 64;
            if (row < M) stream_store8(q0 + off, make_uint2(o.x, o.y));
            if (row + 8 < M) stream_store8(q1 + off, make_uint2(o.z, o.w));
        }
    }
    if (wave == 0 && c == 0) {
        if (row < M) scale[row] = s0;
        if (row + 8 < M) scale[row + 8] = s1;
    }
    __syncthreads();
    const int m = blockIdx.x * 16 + fr;
    if (wave < RT && m < M) {   // the waves' sums, in wave order: ranks 16 wave + 4 fg ... of row m
        v4f sum = sh.sum[0][wave][lane];
#pragma unroll
        for (int w = 1; w < 8; ++w) sum += sh.sum[w][wave][lane];
        uint2 o;
        if constexpr (DT == I8F_BF16) o = make_uint2(f32x2_to_bf16x2_bits(sum.x, sum.y), f32x2_to_bf16x2_bits(sum.z, sum.w));
        else o = make_uint2(f32x2_to_f16x2_bits(sum.x, sum.y), f32x2_to_f16x2_bits(sum.z, sum.w));
        *(uint2 *)(t + ((int64_t)m * (16 * RT) + 16 * wave + 4 * fg) * 2) = o;
    }
}

template <int DT, int RT>
int launch_quant_lora(const char *x, int M, int K, int64_t ldx_bytes, const char *la, int8_t *q, float *scale, char *t, hipStream_t st) {
    const dim3 grid((unsigned)((M + 15) / 16));
    const int per = (K / 64 + 7) / 8;  // blocks of a wave
    auto go = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, grid, dim3(512), 0, st, x, M, K, ldx_bytes, la, q, scale, t);
        return check_launch();
    };
    if (per <= 2) return go(quant_lora_kernel<DT, RT, 2, 0>);
    if (per <= 4) return go(quant_lora_kernel<DT, RT, 4, 2>);
    if (per <= 6) return go(quant_lora_kernel<DT, RT, 6, 4>);
    if (per <= 8) return go(quant_lora_kernel<DT, RT, 8, 6>);
    if constexpr (RT <= 2)  // (with more the loads' registers would spill)
        if (per <= 12) return go(quant_lora_kernel<DT, RT, 12, 8>);
    return I8F_ERR_UNSUPPORTED;
}

template <int DT>
int launch_quant_lora_rank(int rank, const char *x, int M, int K, int64_t ldx_bytes, const char *la, int8_t *q, float *scale, char *t, hipStream_t st) {
    switch (rank) {
    case 16: return launch_quant_lora<DT, 1>(x, M, K, ldx_bytes, la, q, scale, t, st);
    case 32: return launch_quant_lora<DT, 2>(x, M, K, ldx_bytes, la, q, scale, t, st);
    case 48: return launch_quant_lora<DT, 3>(x, M, K, ldx_bytes, la, q, scale, t, st);
    default: return launch_quant_lora<DT, 4>(x, M, K, ldx_bytes, la, q, scale, t, st);
    }
}

}  // namespace
}  // namespace i8f

extern "C" int i8f_internal_quant_lora(const void *x, int dtype, int64_t M, int64_t K, int64_t ldx, const void *lora_a, int64_t rank, int8_t *q,
                                       float *scale, void *t, void *stream) {
    using namespace i8f;
    if ((dtype != I8F_BF16 && dtype != I8F_F16) || !x || !lora_a || !q || !scale || !t || M < 1 || M > 0x7fffffff || K < 64 || K > 6144 || K % 64 ||
        ldx < K || ldx % 8 || rank < 16 || rank > 64 || rank % 16)
        return I8F_ERR_UNSUPPORTED;
    if (((uintptr_t)x | (uintptr_t)lora_a | (uintptr_t)q | (uintptr_t)t) % 16) return I8F_ERR_UNSUPPORTED;
    if (int rc = check_device()) return rc;
    auto go = dtype == I8F_BF16 ? launch_quant_lora_rank<I8F_BF16> : launch_quant_lora_rank<I8F_F16>;
    return go((int)rank, (const char *)x, (int)M, (int)K, ldx * 2, (const char *)lora_a, q, scale, (char *)t, (hipStream_t)stream);
}
