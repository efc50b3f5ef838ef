// The low-rank merge that draws its noise: two launches whose result is, bit for bit, that of the merge on torch's own noise
// (lora_merge.hip, where the form for few elements is, too).
//
//   draw_bytes_kernel    the upper byte of every element's random word, and the factors in the form the merge multiplies
//   merge_drawn_kernel   an approximate quotient from 16-bit matrix products, rounded against those bytes; the few
//                        elements that an error bound or a byte's missing bits leave open are done again, in the end by definition
//
// Both approximations only ever say "certain" or "open", so neither can change a result.
//
// us, 12288 x 3072 rank 32, 9216 x 3072 ranks 16 + 32 + 64, 3072 x 12288 rank 128, 12288 x 12288 rank 8: both launches
// 53, 57, 87, 173 (the first 17, 15, 18, 57).  With 16-bit halves of the words and binary32 products, whose 64 cycles a pair of
// ranks share the SIMD with the vector instructions (the form for few elements), 66, 97, 140, 174; with torch.rand and the merge on
// its tensor 86, 121 for the first two.
#include "merge_round.hpp"

namespace i8f {
namespace {

typedef float v16f __attribute__((ext_vector_type(16)));
typedef _Float16 v8h __attribute__((ext_vector_type(8)));

constexpr int PIECE = 8;   // ranks in a 16-byte piece of binary16

// The factors of the LoRAs that are merged together, and what the first launch makes of them: of several, `up` side by side
// [N,R]; `down`, of several side by side and each times its multiplier (rounded), with the ranks of a column together [K,R]; and both times powers of two as sums of two binary16 values, in the
// order in which the merge reads them: split_up[n][rank / 8][part], a power to a row, and split_down[column / 32][rank / 16][part]
// [64 lanes], a power to 32 columns.  rows and columns: the reciprocal of that power, and the row's norm or the largest column's.
struct Factors {
    const float *up[MAX_FACTORS], *down[MAX_FACTORS];
    float mult[MAX_FACTORS];
    int first[MAX_FACTORS + 1];   // first rank of each; [n] = the sum R
    int n, pieces;                // pieces: of a padded row
    uint32_t N, K;
    float *up_out, *down_out;
    uint4 *split_up, *split_down;
    float2 *rows, *columns;
};

// The power of two that brings `largest` into [2^14, 2^15), and its reciprocal.  False where the products of two such powers
// would not be ordinary numbers (NaN included); 1 for an all-zero factor.
__device__ __forceinline__ bool scaling(float largest, float &there, float &back) {
    const bool ok = largest >= 0x1p-40f && largest <= 0x1p+40f;
    const uint32_t e = (__float_as_uint(largest) >> 23) & 0xffu;
    there = ok ? __uint_as_float((268u - e) << 23) : 1.0f;
    back = ok ? __uint_as_float((e - 14u) << 23) : 1.0f;
    return ok || largest == 0.0f;
}

// x = hi + lo up to 2^-22 |x| and, where a part is below binary16's normal range, 2^-14
__device__ __forceinline__ void split8(const float (&v)[8], float scale, v8h &hi, v8h &lo) {
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        const float x = v[i] * scale;   // (exact: a power of two)
        const _Float16 h = (_Float16)x;
        hi[i] = h, lo[i] = (_Float16)(x - (float)h);
    }
}

constexpr float NORM_SLACK = 1.0f + 0x1p-10f;   // over the roundings of a norm and of the products it goes into

// eight neighbouring lanes to a row of `up`
__device__ __forceinline__ void prepare_rows(const Factors &f, uint32_t block, uint32_t blocks) {
    const int part = threadIdx.x & 7, R = f.first[f.n];
    for (uint32_t n = block * 32 + threadIdx.x / 8; n < f.N; n += blocks * 32) {
        float v[4][8] = {};
        for (int l = 0; l < f.n; ++l) {
            const int r = f.first[l + 1] - f.first[l];
            const float *src = f.up[l] + (uint64_t)n * r;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int own = (part + 8 * i) * PIECE - f.first[l];   // of the piece's first rank
                if (own > -PIECE && own < r) {
#pragma unroll
                    for (int t = 0; t < 8; ++t) {   // (loads without branches between them)
                        const float x = src[min(max(own + t, 0), r - 1)];
                        v[i][t] = own + t >= 0 && own + t < r ? x : v[i][t];
                    }
                }
            }
        }
        float largest = 0.0f, sum = 0.0f;
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int t = 0; t < 8; ++t) largest = fmaxf(largest, fabsf(v[i][t])), sum = __builtin_fmaf(v[i][t], v[i][t], sum);
#pragma unroll
        for (int s = 1; s < 8; s *= 2) largest = fmaxf(largest, __shfl_xor(largest, s)), sum += __shfl_xor(sum, s);
        float there, back;
        const bool ok = scaling(largest, there, back);
        if (part == 0) f.rows[n] = make_float2(back, ok ? __builtin_sqrtf(sum) * NORM_SLACK : __builtin_inff());   // (a NaN is in the sum)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int piece = part + 8 * i;
            if (piece < f.pieces) {
                v8h hi, lo;
                split8(v[i], there, hi, lo);
                uint4 *dst = f.split_up + ((uint64_t)n * f.pieces + piece) * 2;
                dst[0] = __builtin_bit_cast(uint4, hi), dst[1] = __builtin_bit_cast(uint4, lo);
                if (f.n > 1) {
#pragma unroll
                    for (int t = 0; t < 8; ++t)
                        if (piece * PIECE + t < R) f.up_out[(uint64_t)n * R + piece * PIECE + t] = v[i][t];
                }
            }
        }
    }
}

// a workgroup of 256 threads to 32 columns of `down`
__device__ __forceinline__ void prepare_columns(const Factors &f, uint32_t block) {
    __shared__ float sums[256], tops[4];
    const int R = f.first[f.n], col = threadIdx.x % 32, part = threadIdx.x / 32;
    const uint32_t k = block * 32 + col;
    const bool in = k < f.K;
    float v[4][8] = {};   // of pieces part, part + 8, ...
    for (int l = 0; l < f.n; ++l) {
        const int r = f.first[l + 1] - f.first[l];
        const float *src = f.down[l] + (in ? k : 0);
        const float mult = f.n > 1 ? f.mult[l] : 1.0f;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int own = (part + 8 * i) * PIECE - f.first[l];
            if (own > -PIECE && own < r) {
#pragma unroll
                for (int t = 0; t < 8; ++t) {
                    const float x = src[(uint64_t)min(max(own + t, 0), r - 1) * f.K] * mult;
                    v[i][t] = own + t >= 0 && own + t < r ? x : v[i][t];
                }
            }
        }
    }
    float largest = 0.0f, sum = 0.0f;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
#pragma unroll
        for (int t = 0; t < 8; ++t) {
            if (!in) v[i][t] = 0.0f;
            largest = fmaxf(largest, fabsf(v[i][t])), sum = __builtin_fmaf(v[i][t], v[i][t], sum);
        }
    }
    sums[threadIdx.x] = sum;
    largest = wave_max(largest);
    if (threadIdx.x % 64 == 0) tops[threadIdx.x / 64] = largest;
    __syncthreads();
    float there, back;
    const bool ok = scaling(fmaxf(fmaxf(tops[0], tops[1]), fmaxf(tops[2], tops[3])), there, back);
    if (threadIdx.x < 64) {
        sum = 0.0f;
#pragma unroll
        for (int p = 0; p < 8; ++p) sum += sums[p * 32 + col];
        const bool bad = __builtin_amdgcn_ballot_w64(sum != sum) != 0;
        sum = wave_max(sum);   // of a column's squares
        if (threadIdx.x == 0) f.columns[block] = make_float2(back, ok && !bad ? __builtin_sqrtf(sum) * NORM_SLACK : __builtin_inff());
    }
    // Row 8 q + 4 h + e of a block's product is its column 16 h + 4 q + e, so that a lane ends up with 16 neighbouring columns.
    const int row = 8 * ((col >> 2) & 3) + 4 * (col >> 4) + (col & 3);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int piece = part + 8 * i;
        if (piece < f.pieces) {
            v8h hi, lo;
            split8(v[i], there, hi, lo);
            uint4 *dst = f.split_down + ((uint64_t)block * (f.pieces / 2) + piece / 2) * 128 + row + 32 * (piece & 1);
            dst[0] = __builtin_bit_cast(uint4, hi), dst[64] = __builtin_bit_cast(uint4, lo);
#pragma unroll
            for (int t = 0; t < 8; t += 4)
                if (in && piece * PIECE + t < R)   // (R % 4 == 0)
                    *(float4 *)(f.down_out + (uint64_t)k * R + piece * PIECE + t) = make_float4(v[i][t], v[i][t + 1], v[i][t + 2], v[i][t + 3]);
        }
    }
}

// The upper byte of every element's word (0 for those that give 0) as noise[k / 16][n][16], the order in which the merge reads:
// neighbouring rows side by side.  A thread calls the generator for sixteen neighbouring lanes, which are of one row; a call's four
// words belong to elements `lanes` apart.  The threads of a wave take neighbouring rows.  The first blocks prepare the factors.
// Bound by the generator: 18 64-bit products and 19 three-way exclusive ors a call, 37 of its 45 vector instructions, 8 and 4 cycles each.
// (A thread of eight lanes pays its 40 instructions of addresses twice as often: 19.5 us for 17.6 at 12288 x 3072.)
__global__ __launch_bounds__(256, 6) void draw_bytes_kernel(uint32_t seed_lo, uint32_t seed_hi, uint32_t lanes, uint32_t rows, uint32_t first_chunk,
                                                         uint32_t column_blocks, uint32_t row_blocks, uint32_t rows_on, uint32_t columns_on, uint32_t rows_inverse, uint32_t K_inverse,
                                                         uint4 *noise, const Factors f) {
    if (blockIdx.y < first_chunk) {
        const uint32_t block = blockIdx.y * gridDim.x + blockIdx.x;
        if (block < column_blocks) prepare_columns(f, block);
        else if (block < column_blocks + row_blocks) prepare_rows(f, block - column_blocks, row_blocks);
        return;
    }
    const uint32_t chunk = blockIdx.y - first_chunk, at = blockIdx.x * 256 + threadIdx.x, K = f.K, N = f.N;
    // (quotients by products with 2^32 / divisor, which are exact or one too small)
    uint32_t run = __umulhi(at, rows_inverse);
    run += at - run * rows >= rows;
    const uint32_t row = at - run * rows, s0 = row * K + run * 16;
    const uint32_t first = 4 * chunk * lanes;   // element of the chunk's lane 0: row n0, column k0
    uint32_t n0 = __umulhi(first, K_inverse);
    n0 += first - n0 * K >= K;
    uint32_t n = n0 + row, k = first - n0 * K + run * 16;
    if (k >= K) k -= K, ++n;
    if (run >= K / 16 || s0 >= lanes || n >= N) return;
    uint32_t o[4][4];   // of word q, elements 4 g ... 4 g + 3
#pragma unroll
    for (int g = 0; g < 4; ++g) {
        uint32_t x[4][4], top = 0;
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            philox(chunk, s0 + 4 * g + t, seed_lo, seed_hi, x[t]);
            top = max(max(top, x[t][0]), x[t][1]), top = max(max(top, x[t][2]), x[t][3]);
        }
        if (top >= ONE_WORDS) {
#pragma unroll
            for (int t = 0; t < 4; ++t)
#pragma unroll
                for (int q = 0; q < 4; ++q) x[t][q] = x[t][q] >= ONE_WORDS ? 0u : x[t][q];
        }
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const uint32_t a = __builtin_amdgcn_perm(x[1][q], x[0][q], 0x0c0c0703u), b = __builtin_amdgcn_perm(x[3][q], x[2][q], 0x0c0c0703u);
            o[q][g] = __builtin_amdgcn_perm(b, a, 0x05040100u);
        }
    }
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        if (n < N) noise[(k / 16) * N + n] = make_uint4(o[q][0], o[q][1], o[q][2], o[q][3]);
        n += rows_on, k += columns_on;
        if (k >= K) k -= K, ++n;
    }
}

struct DrawnArgs {
    const int8_t *w;
    const float *ws;
    float ws_host;
    int row_scale;
    const float *up, *down;   // (side by side; down [K,R])
    int rank;
    float lora_scale;
    uint32_t N, K, lanes, seed_lo, seed_hi;
    const uint4 *noise, *split_up, *split_down;
    const float2 *rows, *columns;
    int8_t *out;
};

// One element by the definition, from the whole word.
__device__ __forceinline__ float word_noise(const DrawnArgs &a, uint32_t e) {
    const uint32_t i = e / a.lanes;
    uint32_t x[4];
    philox(i / 4, e - i * a.lanes, a.seed_lo, a.seed_hi, x);
    const uint32_t lo = i & 1 ? x[1] : x[0], hi = i & 1 ? x[3] : x[2];
    return uniform_of(i & 2 ? hi : lo);
}

__device__ __forceinline__ float from_lane(int lane, float v) { return __int_as_float(__builtin_amdgcn_ds_bpermute(lane * 4, __float_as_int(v))); }
__device__ __forceinline__ uint32_t from_lane(int lane, uint32_t v) { return (uint32_t)__builtin_amdgcn_ds_bpermute(lane * 4, (int)v); }

// The rounding of element (n, k), with all its operands, of every lane that needs it, by the definition.  Called by whole waves.  The chain of
// a sum cannot be shared out but its operands can: sixteen elements at a time, an element's ranks over four lanes, whose
// loads are one trip to memory together; the sum then goes from each of the four to the next.  `down` is read with its columns'
// ranks together: an element then takes a line for 32 ranks (of [R,K] one for every rank: 3072 x 12288, rank 128, 77 for 72 us).
template <int STEPS>
__device__ __forceinline__ float defined_rounding(const DrawnArgs &a, int lane, bool need, uint32_t n, uint32_t k, float sc, float noise) {
    constexpr int AT_ONCE = STEPS <= 8 ? STEPS : STEPS / 2, QUARTER = 4 * AT_ONCE;   // 16-rank steps in registers, ranks of a lane
    static_assert(STEPS % AT_ONCE == 0, "whole rounds");
    const int group = lane >> 4, entry = lane & 15;
    float result = 0.0f;
    for (uint64_t left = __builtin_amdgcn_ballot_w64(need); left != 0;) {
        const uint32_t place = __builtin_amdgcn_mbcnt_hi((uint32_t)(left >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)left, 0));
        const bool taken = __builtin_amdgcn_inverse_ballot_w64(left) && place < 16;
        const int to = taken ? (int)place : 32;   // (32: looked at by nobody)
        uint32_t en = (uint32_t)__builtin_amdgcn_ds_permute(to * 4, (int)n), ek = (uint32_t)__builtin_amdgcn_ds_permute(to * 4, (int)k);
        en = from_lane(entry, en), ek = from_lane(entry, ek);
        if (entry >= __builtin_popcountll(left)) en = 0, ek = 0;
        float s = 0.0f;
#pragma unroll 1
        for (int j0 = 0; j0 < a.rank; j0 += 4 * QUARTER) {
            const int first = j0 + group * QUARTER;
            const float *u = a.up + (uint64_t)en * a.rank + first, *d = a.down + (uint64_t)ek * a.rank + first;
            float4 uv[QUARTER / 4], dv[QUARTER / 4];
#pragma unroll
            for (int i = 0; i < QUARTER / 4; ++i) {
                uv[i] = dv[i] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
                if (first + 4 * i < a.rank) uv[i] = *(const float4 *)(u + 4 * i), dv[i] = *(const float4 *)(d + 4 * i);   // (a.rank % 4 == 0)
            }
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                float t = s;
#pragma unroll
                for (int i = 0; i < QUARTER / 4; ++i) {   // (beyond the rank 0 * 0)
                    t = __builtin_fmaf(uv[i].x, dv[i].x, t), t = __builtin_fmaf(uv[i].y, dv[i].y, t);
                    t = __builtin_fmaf(uv[i].z, dv[i].z, t), t = __builtin_fmaf(uv[i].w, dv[i].w, t);
                }
                s = from_lane(((g + 1) % 4) * 16 + entry == lane ? g * 16 + entry : lane, group == g ? t : s);
            }
        }
        const float sum = from_lane((int)place & 15, s);   // (behind the last quarter it is the first one's)
        if (taken) result = sr_round(sum * a.lora_scale / sc, noise);
        left &= ~__builtin_amdgcn_ballot_w64(taken);
    }
    return result;
}
__device__ __forceinline__ int8_t add_sat8(uint32_t w, float r) { return (int8_t)sat8((int)(int8_t)w + (int)r); }

// The merge.  A wave takes tiles of 32 rows and COLS columns by itself: the weights go through an LDS tile of its own and leave it as
// results, the noise and the tile's rows of `up` go straight to registers, `down` lies in LDS for the workgroup, and there is no
// barrier after it has been put there.  The product D[k][n] is three binary16 products of the factors' high and low parts; its
// columns are laid out so that a lane holds 16 neighbouring columns of one row.  An element takes 8 vector instructions, four of
// them for its rounding.  One in 256 is open and goes to a list, which 64 lanes answer together from whole words; what that leaves
// open (one in ten thousand at rank 32) waits until some have come together.
//
// A wave has about two tiles, so that start (6 us with the launch) and end show.  12288 x 3072, rank 32: 33 us for 113 MB, half of
// its cycles with a vector instruction in issue; without the list and what follows 30.5, without the products 28.  Sixteen waves to a
// CU where they fit the registers (twelve: 35 us, eight: 38.5); beyond rank 64 a tile's rows of `up` leave room for eight (rank 112 42 us,
// twelve with spills 66).  All products of a tile first, for four chains instead of one, or those of the next block beside the
// rounding of this one: no faster.  Answers for the whole of a wave at its end, by byte stores over what is stored: 37 for 35 us.
// STEPS: 16-rank steps of the padded product.  PER_CU: workgroups that share the waves of a CU.
template <int STEPS, int PER_CU>
struct DrawnShape {
    static constexpr int BLOCKS = STEPS <= 12 ? 4 : 2, COLS = 32 * BLOCKS;         // 32-column blocks of a workgroup
    static constexpr int PER_SIMD = STEPS <= 2 ? 4 : STEPS <= 4 ? 3 : 2, WAVES = 4 * PER_SIMD / PER_CU;
    static constexpr int PANEL = BLOCKS * STEPS * 2048;                           // `down`, two parts of 1 KB to a block and step
    static constexpr int PITCH = COLS + 16, TILE = 32 * PITCH;                    // a wave's weights
    static constexpr int MOST_OPEN = 48, LIST = BLOCKS * MOST_OPEN;               // open elements of a block, of a tile
    static constexpr int LATER = 32;                                              // elements left to the definition after which it is turned to
    static constexpr int WAVE = TILE + LIST * 8 + (LATER + LIST) * 5;
    static constexpr int BYTES = PANEL + WAVES * ((WAVE + 15) / 16 * 16);
    static_assert((BYTES + 64) * PER_CU <= 160 * 1024, "LDS");
};

template <int STEPS, int PER_CU>
__global__ __launch_bounds__((DrawnShape<STEPS, PER_CU>::WAVES * 64), (DrawnShape<STEPS, PER_CU>::PER_SIMD)) void merge_drawn_kernel(const DrawnArgs a) {
    using T = DrawnShape<STEPS, PER_CU>;
    constexpr int NT = T::WAVES * 64, BLOCKS = T::BLOCKS, COLS = T::COLS;
    __shared__ __attribute__((aligned(16))) char lds[T::BYTES];
    __shared__ float back[BLOCKS];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int l32 = lane & 31, half = lane >> 5;
    const uint32_t N = a.N, K = a.K, k0 = blockIdx.x * COLS;

    char *const tile = lds + T::PANEL + wave * ((T::WAVE + 15) / 16 * 16);
    float *const list_x = (float *)(tile + T::TILE);            // open elements of a tile: quotient; place in the tile, weight
    uint32_t *const list_at = (uint32_t *)(list_x + T::LIST);
    uint32_t *const later_at = list_at + T::LIST;               // elements left to the definition: row and column, weight
    uint8_t *const later_w = (uint8_t *)(later_at + T::LATER + T::LIST);
    const uint32_t nblocks = (N + 31) / 32, step = gridDim.y * T::WAVES;
    uint32_t block = wave * gridDim.y + blockIdx.y;   // (so that the waves with a block more are spread over the workgroups)

    constexpr int PPR = COLS / 16, RPI = 64 / PPR;   // 16-byte pieces to a row of the tile, rows to a wave's load
    const int w_row = lane / PPR, w_piece = lane % PPR;
    const bool w_in = k0 + w_piece * 16 < K;
    auto row_in = [&](uint32_t n) { return n < N ? n : N - 1; };   // rows past the end repeat the last one, unstored
    v4u_t w_r[BLOCKS];
    auto fetch_weights = [&](uint32_t blk) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < BLOCKS; ++i)
            if (w_in) w_r[i] = *(const v4u_t *)(a.w + (row_in(blk * 32 + i * RPI + w_row) * K + k0 + w_piece * 16));
    };
    uint4 nz_r;
    auto fetch_noise = [&](uint32_t blk, int b) __attribute__((always_inline)) {
        nz_r = a.noise[min(k0 / 16 + 2 * b + half, K / 16 - 1) * N + row_in(blk * 32 + l32)];
    };
    v8h u_r[STEPS][2];   // a tile's rows of `up`, for all of its columns
    auto up_piece = [&](uint32_t blk, int ks, int part) __attribute__((always_inline)) {
        return __builtin_bit_cast(v8h, a.split_up[((uint64_t)row_in(blk * 32 + l32) * (2 * STEPS) + 2 * ks + half) * 2 + part]);
    };
    float sc_r;
    float2 row_r;
    auto fetch_rows = [&](uint32_t blk) __attribute__((always_inline)) {
        const uint32_t n = row_in(blk * 32 + l32);
        sc_r = a.ws ? a.ws[a.row_scale ? n : 0] : a.ws_host;
        row_r = a.rows[n];
#pragma unroll
        for (int ks = 0; ks < STEPS; ++ks) u_r[ks][0] = up_piece(blk, ks, 0), u_r[ks][1] = up_piece(blk, ks, 1);
    };
    {   // the workgroup's columns of `down` to LDS, with the first block's operands
        constexpr int PIECES = T::PANEL / 16, PER = (PIECES + NT - 1) / NT;
        const uint4 *src = a.split_down + (uint64_t)blockIdx.x * PIECES;
        uint4 v[PER];
#pragma unroll
        for (int i = 0; i < PER; ++i) v[i] = src[min(tid + i * NT, PIECES - 1)];
        const uint32_t mine = min(block, nblocks - 1);
        fetch_weights(mine);
        fetch_noise(mine, 0);
        fetch_rows(mine);
#pragma unroll
        for (int i = 0; i < PER; ++i) *(uint4 *)(lds + min(tid + i * NT, PIECES - 1) * 16) = v[i];
    }
    float columns_norm = 0.0f;   // the largest (a NaN does not occur)
#pragma unroll
    for (int b = 0; b < BLOCKS; ++b) columns_norm = fmaxf(columns_norm, a.columns[blockIdx.x * BLOCKS + b].y);
    columns_norm = __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(columns_norm)));
    if (tid < BLOCKS) back[tid] = a.columns[blockIdx.x * BLOCKS + tid].x;
    __syncthreads();
    if (block >= nblocks) return;

    // ---- a wave's own work: blocks of 32 rows, no barrier from here on ------------------------------------------------
    // How far the approximate quotient may be from the definition's, as a multiple of |f| times the norms of the two factors' row
    // and column (which bound the sum of the products' magnitudes): 2^-24 for each of the definition's additions, twice that for
    // each of the matrix unit's (whatever its inner order is; the cross products go first, and what their additions lose is below
    // 2^-9 of that), 3 * 2^-22 for the two splits and the product of the low parts, 2^-22 for parts below binary16's normal
    // range, 7 * 2^-24 for the reciprocal, the products with lora_scale and f, and the definition's own product and quotient, 2^-24 for
    // the difference of quotient and noise, whose rounding grows with the quotient (2^-16 at 300, beyond which it is not asked for).
    // That is 3 rank + 24 times 2^-24; 32 leaves something for the norms' and this bound's own roundings.
    const float coefficient = (float)(3 * a.rank + 32) * 0x1p-24f;
    constexpr float ROUNDINGS = 0x1p-22f;   // of the same difference where the quotient is below 1, and of the distances, which are
    // the products of 32 columns with the block's rows
    auto product = [&](int b, v16f &acc) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < 16; ++i) acc[i] = 0.0f;
        const char *p = lds + b * STEPS * 2048 + lane * 16;
#pragma unroll
        for (int ks = 0; ks < STEPS; ++ks) {
            const v8h dh = *(const v8h *)(p + ks * 2048), dl = *(const v8h *)(p + ks * 2048 + 1024);
            acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(dl, u_r[ks][0], acc, 0, 0, 0);
            acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(dh, u_r[ks][1], acc, 0, 0, 0);
        }
#pragma unroll
        for (int ks = 0; ks < STEPS; ++ks) acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(*(const v8h *)(p + ks * 2048), u_r[ks][0], acc, 0, 0, 0);
    };

    uint32_t later = 0;
    while (true) {
        const uint32_t next = min(block + step, nblocks - 1);   // (past the end the last block again, unused)
        const bool last_tile = block + step >= nblocks;
#pragma unroll
        for (int i = 0; i < BLOCKS; ++i) *(v4u_t *)(tile + (i * RPI + w_row) * T::PITCH + w_piece * 16) = w_r[i];
        fetch_weights(next);
        const float sc = sc_r, f0 = __builtin_amdgcn_rcpf(sc) * a.lora_scale, f1 = f0 * row_r.x;
        const float most = row_r.y * columns_norm * fabsf(f0), error = coefficient * most;   // of a quotient, of its error
        const bool usual = sc >= 0x1p-110f && sc <= 0x1p+110f && error <= 0x1p-4f;   // (a NaN is not)
        // open: further than `sure` from the middle between two whole numbers; always so in an unusual row
        const float sure = usual ? 0.5f - 0x1p-9f - 0x1p-14f - error : -1.0f;   // (2^-14: y is rounded twice, up to 2^9)
        const bool clamps = __builtin_amdgcn_ballot_w64(!(most <= 100.0f)) != 0;   // a quotient may have to be clamped
        const bool row_ok = block * 32 + l32 < N;
        uint32_t count = 0, skipped = 0;   // open elements of the tile, blocks with too many
#pragma unroll 1
        for (int b = 0; b < BLOCKS; ++b) {
            const uint32_t nz[4] = {nz_r.x, nz_r.y, nz_r.z, nz_r.w};
            if (b + 1 < BLOCKS) fetch_noise(block, b + 1);
            else fetch_noise(next, 0);
            v16f acc;
            product(b, acc);
            if (b + 1 == BLOCKS) fetch_rows(next);
            const float f = f1 * back[b];

            // With u = 255 - (weight + 128) the result, in the same terms, is u + floor(noise - quotient), saturated.  A 16-bit value of u
            // and the noise's byte is both operands in one conversion; y is that sum less 1/2, a byte's noise taken at the middle
            // of its range, so that the result is the whole number next to it.
            char *const mine = tile + l32 * T::PITCH + b * 32 + half * 16;
            const v4u_t wp = *(const v4u_t *)mine;
            const uint64_t in = __builtin_amdgcn_ballot_w64(row_ok && k0 + b * 32 + half * 16 < K);
            uint64_t open[16];
            float r[16];
            uint32_t total = 0;
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const uint32_t u = wp[q] ^ 0x7f7f7f7fu;
                const uint32_t pair[2] = {__builtin_amdgcn_perm(u, nz[q], 0x05010400u), __builtin_amdgcn_perm(u, nz[q], 0x07030602u)};
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const int i = 4 * q + e;
                    const float both = (float)(e % 2 ? pair[e / 2] >> 16 : pair[e / 2] & 0xffffu);
                    const float y = __builtin_fmaf(both, 0x1p-8f, __builtin_fmaf(acc[i], -f, 0x1p-9f - 0.5f));
                    r[i] = __builtin_rintf(y);
                    open[i] = __builtin_amdgcn_fcmpf(fabsf(y - r[i]), sure, 10);   // greater, or not comparable
                }
            }
            if (clamps) {   // what is added is saturated by itself first
#pragma unroll
                for (int i = 0; i < 16; ++i) {
                    const float u = (float)(((wp[i / 4] ^ 0x7f7f7f7fu) >> (8 * (i % 4))) & 0xffu);
                    r[i] = u + __builtin_amdgcn_fmed3f(r[i] - u, -127.0f, 128.0f);
                }
            }
#pragma unroll
            for (int i = 0; i < 16; ++i) open[i] &= in, total += __builtin_popcountll(open[i]);   // (what is not stored is not looked at)
            if (__builtin_expect(total <= T::MOST_OPEN, 1)) {
                uint32_t o[4];
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    o[q] = 0;
#pragma unroll
                    for (int e = 0; e < 4; ++e) o[q] = __builtin_amdgcn_cvt_pk_u8_f32(r[4 * q + e], e, o[q]);   // (clamps to 0 ... 255)
                    o[q] ^= 0x7f7f7f7fu;
                }
                *(v4u_t *)mine = v4u_t{o[0], o[1], o[2], o[3]};
#pragma unroll
                for (int i = 0; i < 16; ++i) {
                    if (open[i] != 0) {
                        const uint32_t to = __builtin_amdgcn_mbcnt_hi((uint32_t)(open[i] >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)open[i], count));
                        if (__builtin_amdgcn_inverse_ballot_w64(open[i])) {
                            list_x[to] = acc[i] * f;
                            list_at[to] = (uint32_t)(mine - tile + i) | ((wp[i / 4] >> (8 * (i % 4))) & 0xffu) << 16;
                        }
                        count += __builtin_popcountll(open[i]);
                    }
                }
            } else {
                skipped |= 1u << b;   // (the weights stay in the tile)
            }
        }

        // The open elements side by side, from their whole words.  What an error of the quotient could decide, and is not
        // beyond int8 for certain, is left for later.
        while (count != 0) {
            const uint32_t base = count > 64 ? count - 64 : 0;
            const bool there = base + lane < count;
            const uint32_t at = list_at[there ? base + lane : base], row = (at & 0xffffu) / T::PITCH, col = (at & 0xffffu) % T::PITCH;
            const float x = list_x[there ? base + lane : base], row_error = from_lane(row, error);
            const uint32_t n = block * 32 + row;
            const float z = x - word_noise(a, n * K + k0 + col), r = ceilf(z), d = r - z, slack = ROUNDINGS + row_error;
            const bool open = there && !(d >= slack && d <= 1.0f - slack) && !(fabsf(x) - row_error > 300.0f);
            if (there) tile[at & 0xffffu] = add_sat8(at >> 16, fminf(fmaxf(r, -128.0f), 127.0f));
            const uint64_t left = __builtin_amdgcn_ballot_w64(open);
            if (open) {
                const uint32_t to = __builtin_amdgcn_mbcnt_hi((uint32_t)(left >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)left, later));
                later_at[to] = n << 7 | col, later_w[to] = (uint8_t)(at >> 16);
            }
            later += __builtin_popcountll(left);
            count = base;
        }
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int t = 0; t < BLOCKS; ++t) {
            const v4u_t v = *(const v4u_t *)(tile + (t * RPI + w_row) * T::PITCH + w_piece * 16);
            const uint32_t n = block * 32 + t * RPI + w_row;
            if (n < N && w_in) stream_store16(a.out + (n * K + k0 + w_piece * 16), make_uint4(v.x, v.y, v.z, v.w));
        }

        // By the definition, over what has been stored: the elements left for later (a wave has one or two of a tile at rank 32; many
        // together cost as much as one), and the blocks of rows that the bound says little of, a column of every lane at a time.
        if (__builtin_expect(skipped != 0 || later >= T::LATER || (last_tile && later != 0), 0)) {
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // the tiles are stored
            const uint32_t down_to = last_tile ? 0 : T::LATER - 1;
            int i = 0;
            while (skipped != 0 || later > down_to) {
                bool need;
                uint32_t n, k, w;
                if (skipped != 0) {
                    const int b = __builtin_ctz(skipped);
                    n = block * 32 + l32, k = k0 + b * 32 + half * 16 + i, need = row_ok && k < K;
                    w = (uint8_t)tile[l32 * T::PITCH + (k - k0)];
                    if (++i == 16) i = 0, skipped &= skipped - 1;
                } else {
                    const uint32_t base = later > 64 ? later - 64 : 0;
                    need = base + lane < later;
                    const uint32_t at = later_at[need ? base + lane : base];
                    n = at >> 7, k = k0 + (at & 127u), w = later_w[need ? base + lane : base];
                    later = base;
                }
                if (!need) n = 0, k = 0;
                const float r = defined_rounding<STEPS>(a, lane, need, n, k, a.ws ? a.ws[a.row_scale ? n : 0] : a.ws_host, word_noise(a, n * K + k));
                if (need) a.out[n * K + k] = add_sat8(w, r);
            }
        }
        __builtin_amdgcn_wave_barrier();
        if (last_tile) break;
        block += step;
    }
}

// Workgroups of a column panel, as many as the CUs hold, and the tiles that the busiest CU gets.
struct Bands {
    int64_t columns, bands, busiest;
    Bands(int64_t N, int64_t K, int cols, int64_t per_cu) {
        const int64_t nblocks = (N + 31) / 32, slots = 256 * per_cu;
        columns = (K + cols - 1) / cols;
        bands = slots / columns;
        bands = bands < 1 ? 1 : bands > nblocks ? nblocks : bands;
        busiest = (columns * bands + slots - 1) / slots * per_cu * ((nblocks + bands - 1) / bands);
    }
};

template <int STEPS, int PER_CU>
int launch_shape(const DrawnArgs &a, const Bands &b, hipStream_t st) {
    hipLaunchKernelGGL((merge_drawn_kernel<STEPS, PER_CU>), dim3((unsigned)b.columns, (unsigned)b.bands), dim3(DrawnShape<STEPS, PER_CU>::WAVES * 64), 0, st, a);
    return check_launch();
}

// Whole panels to a workgroup and whole workgroups to a CU leave CUs idle where the panels divide 256 badly (18432 columns are 144 panels).
// Two workgroups of eight waves to a CU are dealt out more evenly but put every panel into LDS twice as often.  us, one and two, with
// the busiest CU's tiles: 2048 x 18432 rank 16 59.2 and 53.9 (64 and 44), 12288 x 12288 rank 8 172 and 159 (192 and 154), 3072 x 12288
// rank 16 53.9 and 51.4, rank 32 56.3 and 53.8 (48 and 40), 4096 x 11008 rank 16 61.0 and 57.5 (64 and 52), 2048 x 11008 rank 16 36.9 and 35.7
// (32 and 26); 4096 x 8320 rank 32 48.3 and 49.3 (43 and 38), 12288 x 3072 rank 32 46.7 and 48.3 (39 and 38).  Six waves, of ranks above 32, do
// not fill the four SIMDs evenly: 4096 x 11008 rank 48 68 and 82.
constexpr int MAX_SHARED_STEPS = 2;
inline bool two_to_a_cu(const Bands &one, const Bands &two) { return two.busiest * 20 <= one.busiest * 17; }

template <int STEPS>
int launch_steps(const DrawnArgs &a, hipStream_t st) {
    const Bands one(a.N, a.K, DrawnShape<STEPS, 1>::COLS, 1);
    if constexpr (STEPS <= MAX_SHARED_STEPS) {
        const Bands two(a.N, a.K, DrawnShape<STEPS, 2>::COLS, 2);
        if (two_to_a_cu(one, two)) return launch_shape<STEPS, 2>(a, two, st);
    }
    return launch_shape<STEPS, 1>(a, one, st);
}

// the steps that are built: every one up to 8, then 10, 12 and 16 (14 have a tile's rows of `up` in registers that spill: 9216 x 3072, rank
// 224, 178 us, in 16 steps 145)
int steps_of(int64_t rank) {
    const int s = (int)((rank + 15) / 16);
    return s <= 1 ? 1 : s <= 8 ? s : s <= 12 ? (s + 1) / 2 * 2 : 16;
}

// blocks of 32 columns, of whole workgroups of the merge
int64_t column_blocks_of(int64_t K) { return (K + 127) / 128 * 4; }

int launch_merge(const DrawnArgs &a, hipStream_t st) {
    switch (steps_of(a.rank)) {
    case 1: return launch_steps<1>(a, st);
    case 2: return launch_steps<2>(a, st);
    case 3: return launch_steps<3>(a, st);
    case 4: return launch_steps<4>(a, st);
    case 5: return launch_steps<5>(a, st);
    case 6: return launch_steps<6>(a, st);
    case 7: return launch_steps<7>(a, st);
    case 8: return launch_steps<8>(a, st);
    case 10: return launch_steps<10>(a, st);
    case 12: return launch_steps<12>(a, st);
    default: return launch_steps<16>(a, st);
    }
}

// Which form is the faster one, by an estimate of both in us (a sum of what they do, fitted to 1279 shapes of 64 to 18432 rows, 128 to 14000
// columns and ranks 4 to 192, alone and in stacks, operands from HBM).  It is off by 6 and 5 % (standard deviation), and what it picks is
// 0.5 % slower than the better one on average, over 10 % in 11 of them; a line at N K rank = 2^28 is 0.9 % slower where K % 128 == 0, 3 % elsewhere.
// Few elements are the case for the form of lora_merge.hip: 1024 x 1024 rank 16 8.9 and 12.6 us, 3072 x 3072 rank 16 18.5 and 19.7, 2048 x 1024
// rank 32 10.5 and 14.4, rank 64 14.0 and 16.6, and of ranks up to 8, whose products are nothing, more: 12288 x 3072 rank 8 46.4 and 49.9, 18432 x 3072
// rank 4 63.9 and 68.1.  Against it: 2048 x 2048 rank 64 18.7 and 17.7, 5120 x 4096 rank 16 31.4 and 29.7, 8192 x 8192 rank 4 75.4 and 69.5; columns
// that are no whole lines (1168 x 1632 ranks 4 + 64 + 4 24.6 and 18.7, 392 x 10016 ranks 4 + 64 30.2 and 21.6).
bool takes_few_form(int64_t N, int64_t K, int64_t rank, int count) {
    if (rank > FEW_MAX_RANK || N < 1 || K < 1 || N * K >= (1ll << 26)) return false;   // (8192 x 8192 is the first beyond what was fitted)
    const double elements = (double)N * K * 0x1p-20, factors = (double)(N + K) * rank * 0x1p-20, stack = count > 1;
    // the form for few elements: wave steps of a SIMD (launch_mfma, roughly), of which each is products of the padded rank
    const int64_t padded = rank <= 8 ? (rank + 3) / 4 * 4 : rank <= 32 ? (rank <= 16 ? 16 : 32) : rank <= 128 ? (rank + 15) / 16 * 16 : (rank + 31) / 32 * 32;
    const int64_t waves = padded == 48 || padded == 64 ? 4 : 8, slots = padded <= 32 ? 512 : padded <= 64 ? 768 : 256;
    const int64_t columns = (K + 32 * waves - 1) / (32 * waves), nblocks = (N + 31) / 32;
    const int64_t fit = slots / columns, bands = fit < 1 ? 1 : fit < nblocks ? fit : nblocks;
    const double few_steps = (double)((columns * bands + 255) / 256 * ((nblocks + bands - 1) / bands) * waves / 4);
    // the other: tiles of the busiest CU and of a wave
    const int64_t steps = steps_of(rank), waves_of_cu = steps <= 2 ? 16 : steps <= 4 ? 12 : 8;
    const int cols = steps <= 12 ? 128 : 64;
    const Bands one(N, K, cols, 1), two(N, K, cols, 2);
    const double busiest = (double)(steps <= MAX_SHARED_STEPS && two_to_a_cu(one, two) ? two : one).busiest;
    const double tiles = (double)(int64_t)((busiest + waves_of_cu - 1) / waves_of_cu);
    double few, many;
    if (K % 128 == 0) {
        few = 7.37 + 0.688 * elements + 0.0451 * padded + few_steps * (0.225 + 0.0168 * padded) + stack * (0.43 + 5.17 * factors);
        many = 9.35 + 0.368 * elements + 0.577 * steps + 0.527 * busiest + tiles * (1.007 + 0.416 * steps) + 3.14 * factors + 0.77 * stack;
    } else {
        few = 9.10 + 0.575 * elements + 0.0528 * padded + few_steps * (0.402 + 0.0159 * padded) + stack * (0.88 + 4.42 * factors);
        many = 10.57 + 0.769 * elements + 0.467 * steps + busiest * (0.275 + 0.0044 * steps) + tiles * (0.156 + 0.464 * steps) + 3.27 * factors + 0.89 * stack;
    }
    return few < many;
}

int64_t many_workspace_bytes(int64_t N, int64_t K, int64_t rank, int count) {
    const int64_t steps = steps_of(rank), column_blocks = column_blocks_of(K);
    const int64_t split = up256(N * steps * 64) + up256(N * 8) + up256(column_blocks * steps * 2048) + up256(column_blocks * 8);
    return up256(N * K) + split + up256(4 * K * rank) + (count > 1 ? 4 * N * rank : 0);
}

int merge_many(const DrawnCall &c, hipStream_t st) {
    const int64_t N = c.N, K = c.K, lanes = c.lanes, chunks = (N * K + 4 * lanes - 1) / (4 * lanes);
    Factors f{};
    f.n = c.count;
    for (int i = 0; i < c.count; ++i) {
        f.up[i] = c.factors[i].up, f.down[i] = c.factors[i].down, f.mult[i] = c.factors[i].mult;
        f.first[i + 1] = f.first[i] + (int)c.factors[i].rank;
    }
    char *at = (char *)c.workspace;
    DrawnArgs a{};
    a.w = c.w, a.ws = c.ws, a.ws_host = c.ws_host, a.row_scale = c.row_scale;
    a.up = c.factors[0].up, a.rank = c.rank, a.lora_scale = c.lora_scale;
    a.N = (uint32_t)N, a.K = (uint32_t)K, a.out = c.out;
    a.seed_lo = (uint32_t)c.seed, a.seed_hi = (uint32_t)(c.seed >> 32), a.lanes = (uint32_t)lanes;
    f.N = a.N, f.K = a.K, f.pieces = 2 * steps_of(c.rank);
    const int64_t column_blocks = column_blocks_of(K);
    uint4 *const noise = (uint4 *)at;
    a.noise = noise, at += up256(N * K);
    a.split_up = f.split_up = (uint4 *)at, at += up256(N * f.pieces * 32);
    a.rows = f.rows = (float2 *)at, at += up256(N * 8);
    a.split_down = f.split_down = (uint4 *)at, at += up256(column_blocks * f.pieces * 1024);
    a.columns = f.columns = (float2 *)at, at += up256(column_blocks * 8);
    a.down = f.down_out = (float *)at, at += up256(4 * K * c.rank);
    if (c.count > 1) a.up = f.up_out = (float *)at;
    // rows of K that the generator's threads cover, of which a thread takes 16 elements; blocks of `up`: 32 rows, half a round of the
    // chip at most
    const int64_t rows = (lanes + K - 1) / K, columns = (rows * (K / 16) + 255) / 256, row_blocks = (N + 31) / 32 < 1024 ? (N + 31) / 32 : 1024;
    const int64_t first_chunk = (column_blocks + row_blocks + columns - 1) / columns;
    auto inverse = [](int64_t d) { return d > 1 ? (uint32_t)((1ll << 32) / d) : 0xffffffffu; };
    auto draw = [&](int64_t first, int64_t last) {   // rows of blocks
        hipLaunchKernelGGL(draw_bytes_kernel, dim3((unsigned)columns, (unsigned)(last - first)), dim3(256), 0, st, a.seed_lo, a.seed_hi, a.lanes,
                           (uint32_t)rows, (uint32_t)(first_chunk - first), (uint32_t)column_blocks, (uint32_t)row_blocks,
                           (uint32_t)(lanes / K), (uint32_t)(lanes % K), inverse(rows), inverse(K), noise, f);
        return check_launch();
    };
    const bool once = first_chunk + chunks <= 65535;
    if (int rc = draw(0, once ? first_chunk + chunks : first_chunk)) return rc;
    if (!once)
        if (int rc = draw(first_chunk, first_chunk + chunks)) return rc;
    return launch_merge(a, st);
}

}  // namespace
}  // namespace i8f

// form: 0 the one for few elements, 1 the other, -1 the faster one
extern "C" int64_t i8f_internal_merge_drawn_workspace_bytes(int form, int64_t N, int64_t K, int64_t rank, int count) {
    using namespace i8f;
    if (N < 0 || K < 0 || rank < 0 || N > (1 << 29) || K > (1 << 29) || rank > 256) return 0;
    return (form < 0 ? takes_few_form(N, K, rank, count) : form == 0) ? merge_few_workspace_bytes(N, K, rank, count) : many_workspace_bytes(N, K, rank, count);
}

extern "C" int i8f_internal_merge_drawn(int form, const int8_t *w, const float *w_scale, float w_scale_host, int scale_mode,
                                        const i8f_lora_factors *factors, int count, float lora_scale,
                                        uint64_t seed, int64_t lanes, int64_t N, int64_t K, int8_t *w_out,
                                        void *workspace, int64_t workspace_bytes, void *stream) {
    using namespace i8f;
    if (N < 0 || K < 0) return I8F_ERR_INVALID;
    if (scale_mode != I8F_SCALE_TENSOR && scale_mode != I8F_SCALE_ROW) return I8F_ERR_INVALID;
    if (N == 0 || K == 0) return I8F_OK;
    if (!w || !w_out || !factors || count < 1 || !workspace || lanes <= 0) return I8F_ERR_INVALID;
    if (scale_mode == I8F_SCALE_ROW && !w_scale) return I8F_ERR_INVALID;
    if (count > MAX_FACTORS) return I8F_ERR_UNSUPPORTED;
    int rank = 0;
    for (int i = 0; i < count; ++i) {
        if (!factors[i].up || !factors[i].down || factors[i].rank <= 0) return I8F_ERR_INVALID;
        if (factors[i].rank > 256 - rank) return I8F_ERR_UNSUPPORTED;
        rank += (int)factors[i].rank;
    }
    if (K % 16 || K >= (1 << 24) || N > (1 << 29) / K || rank % 4 || lanes % 256 || lanes > (1 << 24)) return I8F_ERR_UNSUPPORTED;
    if ((uintptr_t)w % 16 || (uintptr_t)w_out % 16 || (uintptr_t)workspace % 16 || (count == 1 && (uintptr_t)factors[0].up % 16)) return I8F_ERR_UNSUPPORTED;
    if (count > 1 && (N + K) * rank >= (1ll << 31)) return I8F_ERR_UNSUPPORTED;   // (elements are counted in 32 bits)
    if ((N * K + 4 * lanes - 1) / (4 * lanes) > 65535) return I8F_ERR_UNSUPPORTED;
    const bool few = form < 0 ? takes_few_form(N, K, rank, count) : form == 0;
    if (few && rank > FEW_MAX_RANK) return I8F_ERR_UNSUPPORTED;
    if (workspace_bytes < i8f_internal_merge_drawn_workspace_bytes(form, N, K, rank, count)) return I8F_ERR_INVALID;
    if (int rc = check_device()) return rc;
    const DrawnCall call{w, w_scale, w_scale_host, scale_mode == I8F_SCALE_ROW, factors, count, rank, lora_scale, seed, lanes, N, K, w_out, workspace};
    return few ? merge_few(call, (hipStream_t)stream) : merge_many(call, (hipStream_t)stream);
}

extern "C" int64_t i8f_lora_merge_sr_drawn_workspace_bytes(int64_t N, int64_t K, int64_t rank, int count) {
    return i8f_internal_merge_drawn_workspace_bytes(-1, N, K, rank, count);
}

extern "C" int i8f_lora_merge_sr_drawn(const int8_t *w, const float *w_scale, float w_scale_host, int scale_mode,
                                       const i8f_lora_factors *factors, int count, float lora_scale,
                                       uint64_t seed, int64_t lanes, int64_t N, int64_t K, int8_t *w_out,
                                       void *workspace, int64_t workspace_bytes, void *stream) {
    return i8f_internal_merge_drawn(-1, w, w_scale, w_scale_host, scale_mode, factors, count, lora_scale, seed, lanes, N, K, w_out, workspace,
                                    workspace_bytes, stream);
}
