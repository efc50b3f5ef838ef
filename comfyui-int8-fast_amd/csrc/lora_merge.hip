// Stochastic-rounding LoRA merge into int8 weights, one pass over HBM.
//
//   xs  = delta_f / w_scale                 correctly rounded division (sr_row: how it is obtained)
//   f   = floor(xs);  frac = xs - f
//   dq  = sat8(noise < frac ? f + 1 : f)    strict compare, noise supplied
//   w'  = sat8(w + dq)
//
// (stochastic_round_int8_delta, int8_quant.py:36-62, and the int8 add of
// calculate_weight, :313-316.)  The reference runs this as about a dozen
// elementwise torch launches over [N,K] float/int32 temporaries.
//
// delta_f is either read (10 bytes per element in total) or rebuilt from the
// rank-r factors in registers (6 bytes per element):
//   acc = 0; for j < r: acc = fmaf(up[n,j], down[j,k], acc); delta_f = acc * lora_scale
// The factors are small (r*(N+K) floats) and stay in cache.
#include "merge_round.hpp"

namespace i8f {
namespace {

struct MergeArgs {
    const int8_t *w;  // nullptr: write dq itself (stochastic_round_int8_delta alone)
    const float *ws;
    float ws_host;
    int row_scale;
    const float *delta;
    const float *up;
    const float *down;
    int rank;
    float lora_scale;
    const float *noise;
    int64_t N, K;
    int8_t *out;
    // instead of noise: the upper halves of the generator's words (draw_words_kernel), and what gives the words themselves
    const uint16_t *drawn;
    uint32_t seed_lo, seed_hi, lanes;
};

// A weight row's scale with what the fast quotient below needs.
struct RowScale {
    float sc, rcp;
    bool fast;
};

__device__ __forceinline__ RowScale row_scale(float sc) {
    RowScale r;
    r.sc = sc;
    r.rcp = 1.0f / sc;                              // correctly rounded
    r.fast = sc >= 0x1p-20f && sc <= 0x1p+20f;      // false for NaN
    return r;
}

// Stochastic rounding of NE elements of one weight row: r[e] = sat8(noise < frac ? floor + 1 : floor) as a float.
//
// The quotient delta / sc is the correctly rounded one.  With y = RN(1/sc) computed once per row, q = delta * y followed by
// two corrections q += RN(delta - sc q) * y (each an fma pair) gives it in five instructions instead of the division's
// eleven: after the first correction q is within one ulp of the quotient, the remainder delta - sc q is then exact, and a
// correction of such a q with a correctly rounded reciprocal rounds correctly (Markstein's theorem) as long as nothing
// overflows or underflows: 2^-20 <= sc <= 2^20 and 2^-102 <= |delta| <= 2^80 make every intermediate a normal number.
// A zero delta gives a zero quotient on either route.  A smaller non-zero delta has |quotient| < 2^-82; whatever the
// corrections make of it (same sign or a zero of either sign, still tiny), floor and compare give the same result as
// for the true quotient when 2^-82 <= noise < 1, which is tested on the noise's bit pattern (so NaN and negative noise
// fail).  A NaN delta gives NaN on either route.  Lanes that fail a test redo their elements with the division.
struct SrGuard {
    float dmax = 0.0f;
    uint32_t nmin = 0xffffffffu, nmax = 0u;
    template <int NE>
    __device__ __forceinline__ void add(const float (&delta)[NE], const float (&noise)[NE]) {
#pragma unroll
        for (int e = 0; e < NE; ++e) {
            dmax = fmaxf(dmax, fabsf(delta[e]));
            const uint32_t nb = __float_as_uint(noise[e]);
            nmin = min(nmin, nb), nmax = max(nmax, nb);
        }
    }
    __device__ __forceinline__ bool fast(const RowScale &rs) const {
        return rs.fast && dmax <= 0x1p+80f && nmin >= 0x16800000u /* 2^-82 */ && nmax < 0x3f800000u /* 1 */;
    }
};

__device__ __forceinline__ float fast_quotient(float delta, const RowScale &rs) {
    float q = delta * rs.rcp;
    float t = __builtin_fmaf(-rs.sc, q, delta);
    q = __builtin_fmaf(t, rs.rcp, q);
    t = __builtin_fmaf(-rs.sc, q, delta);
    return __builtin_fmaf(t, rs.rcp, q);
}

template <int NE>
__device__ __forceinline__ void sr_row(const float (&delta)[NE], const float (&noise)[NE], const RowScale &rs, float (&r)[NE]) {
    float xs[NE];
    SrGuard g;
    g.add(delta, noise);
#pragma unroll
    for (int e = 0; e < NE; ++e) xs[e] = fast_quotient(delta[e], rs);
    if (__builtin_expect(!g.fast(rs), 0)) {
#pragma unroll
        for (int e = 0; e < NE; ++e) xs[e] = delta[e] / rs.sc;
    }
#pragma unroll
    for (int e = 0; e < NE; ++e) r[e] = sr_round(xs[e], noise[e]);
}

// ---- noise drawn here, for few elements --------------------------------------------------------------------------
// The upper 16 bits of every element's word (0 for those that give 0), and the merge below reading them instead of the numbers; only
// the elements whose rounding the other 16 bits decide draw their word again.  A thread calls the generator for eight
// neighbouring lanes, 32 elements.  These two launches wait for less than those of lora_merge_drawn.hip, which splits the factors first
// and lists what is open: where there are few elements or products that is what counts (takes_few_form, with both sides measured).
//
// Several LoRAs: the first `extra` rows of workgroups write the factors side by side, up [N,R] and each `down` times its
// multiplier (rounded) [R,K], while the others draw.
struct Stack {
    const float *up[MAX_FACTORS], *down[MAX_FACTORS];
    float mult[MAX_FACTORS];
    int first[MAX_FACTORS + 1];   // first rank of each; [n] = the sum R
    int n;
    uint32_t N, K;
    float *up_out, *down_out;
};

__device__ __forceinline__ void stack_factors(const Stack &f, uint32_t at, uint32_t step) {
    const uint32_t R = f.first[f.n], ups = f.N * R, all = ups + R * f.K;
#pragma unroll 4
    for (uint32_t i = at; i < all; i += step) {
        const bool is_up = i < ups;
        const uint32_t j = is_up ? i % R : (i - ups) / f.K;   // rank
        int l = 0;
#pragma unroll
        for (int t = 1; t < MAX_FACTORS; ++t) l = t < f.n && (int)j >= f.first[t] ? t : l;
        const uint32_t r = f.first[l + 1] - f.first[l], own = j - f.first[l];
        if (is_up) f.up_out[i] = f.up[l][i / R * r + own];
        else f.down_out[i - ups] = f.down[l][own * f.K + (i - ups) % f.K] * f.mult[l];
    }
}

__global__ __launch_bounds__(256) void draw_words_kernel(uint32_t seed_lo, uint32_t seed_hi, uint32_t lanes, uint32_t numel, uint16_t *out, uint32_t extra,
                                                         const Stack stack) {
    if (blockIdx.y < extra) return stack_factors(stack, (blockIdx.y * gridDim.x + blockIdx.x) * 256 + threadIdx.x, extra * gridDim.x * 256);
    const uint32_t chunk = blockIdx.y - extra;
    const uint32_t s0 = (blockIdx.x * 256 + threadIdx.x) * 8, at = 4 * chunk * lanes + s0;
    if (s0 >= lanes || at >= numel) return;
    uint32_t x[8][4], top = 0;
#pragma unroll
    for (int t = 0; t < 8; ++t) {
        philox(chunk, s0 + t, seed_lo, seed_hi, x[t]);
        top = max(max(top, max(x[t][0], x[t][1])), max(x[t][2], x[t][3]));
    }
    if (top >= ONE_WORDS) {
#pragma unroll
        for (int t = 0; t < 8; ++t)
#pragma unroll
            for (int q = 0; q < 4; ++q) x[t][q] = x[t][q] >= ONE_WORDS ? 0u : x[t][q];
    }
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        uint32_t o[4];
#pragma unroll
        for (int t = 0; t < 4; ++t) o[t] = __builtin_amdgcn_perm(x[2 * t + 1][q], x[2 * t][q], 0x07060302u);  // two upper halves
        if (at + q * lanes < numel) stream_store16(out + at + q * lanes, make_uint4(o[0], o[1], o[2], o[3]));
    }
}

// VEC: 4 elements per thread with 16-byte loads when K % 4 == 0 and pointers are aligned, else 1
template <int VEC, bool FUSED>
__global__ __launch_bounds__(256) void lora_merge_kernel(const MergeArgs a) {
    const int64_t n = blockIdx.y;
    const int64_t k0 = ((int64_t)blockIdx.x * 256 + threadIdx.x) * VEC;
    if (k0 >= a.K) return;
    const float sc = a.ws ? a.ws[a.row_scale ? n : 0] : a.ws_host;
    const int64_t base = n * a.K + k0;

    float d[VEC], nz[VEC];
    if constexpr (FUSED) {
        float acc[VEC];
#pragma unroll
        for (int e = 0; e < VEC; ++e) acc[e] = 0.0f;
        const float *upr = a.up + n * a.rank;
        for (int j = 0; j < a.rank; ++j) {
            const float u = upr[j];
            if constexpr (VEC == 4) {
                const float4 dn = *(const float4 *)(a.down + (int64_t)j * a.K + k0);
                acc[0] = fmaf(u, dn.x, acc[0]);
                acc[1] = fmaf(u, dn.y, acc[1]);
                acc[2] = fmaf(u, dn.z, acc[2]);
                acc[3] = fmaf(u, dn.w, acc[3]);
            } else {
                acc[0] = fmaf(u, a.down[(int64_t)j * a.K + k0], acc[0]);
            }
        }
#pragma unroll
        for (int e = 0; e < VEC; ++e) d[e] = acc[e] * a.lora_scale;
    } else {
        if constexpr (VEC == 4) {
            const float4 t = *(const float4 *)(a.delta + base);
            d[0] = t.x, d[1] = t.y, d[2] = t.z, d[3] = t.w;
        } else {
            d[0] = a.delta[base];
        }
    }
    if constexpr (VEC == 4) {
        const float4 t = *(const float4 *)(a.noise + base);
        nz[0] = t.x, nz[1] = t.y, nz[2] = t.z, nz[3] = t.w;
    } else {
        nz[0] = a.noise[base];
    }

    float r[VEC];
    sr_row<VEC>(d, nz, row_scale(sc), r);

    if constexpr (VEC == 4) {
        stream_store4(a.out + base, add_sat8_pack(a.w ? *(const uint32_t *)(a.w + base) : 0u, r));
    } else {
        a.out[base] = (int8_t)sat8((a.w ? (int)a.w[base] : 0) + (int)r[0]);
    }
}

// Fused low-rank form on the vector ALUs (K not a multiple of 16).  A thread owns 4 consecutive columns and keeps the RANK x 4
// slice of `down` it needs in registers for the whole kernel; the block then walks a band of rows.
// Per row and thread that leaves 16 bytes of noise and 4 bytes of weight to read, 4 bytes to write,
// and the row of `up`, which is the same for every lane and comes through scalar loads.  (Indexing
// the other way round, every element re-reads its column of `down` from L2: 32 bytes of cache
// traffic per byte of weight.)  The sum over the rank is the same fma chain in increasing j.
// One row is fetched ahead; fetching further ahead costs registers, hence resident waves, and is
// slower: the kernel is bound by the fma chain, not by memory.
template <int RANK>
__global__ __launch_bounds__(256) void lora_merge_band_kernel(const MergeArgs a, int rows_per_block) {
    const int64_t k0 = ((int64_t)blockIdx.x * 256 + threadIdx.x) * 4;
    const bool col_ok = k0 < a.K;  // K % 4 == 0 here
    float4 dn[RANK];
#pragma unroll
    for (int j = 0; j < RANK; ++j)
        dn[j] = col_ok ? *(const float4 *)(a.down + (int64_t)j * a.K + k0) : make_float4(0.f, 0.f, 0.f, 0.f);

    const int64_t n_begin = (int64_t)blockIdx.y * rows_per_block;
    const int64_t n_end = n_begin + rows_per_block < a.N ? n_begin + rows_per_block : a.N;
    if (n_begin >= n_end || !col_ok) return;

    float4 nz = *(const float4 *)(a.noise + n_begin * a.K + k0);
    uint32_t wp = *(const uint32_t *)(a.w + n_begin * a.K + k0);
    for (int64_t n = n_begin; n < n_end; ++n) {
        const float4 nz_cur = nz;
        const uint32_t wp_cur = wp;
        if (n + 1 < n_end) {  // next row's operands are in flight while this row is computed
            nz = *(const float4 *)(a.noise + (n + 1) * a.K + k0);
            wp = *(const uint32_t *)(a.w + (n + 1) * a.K + k0);
        }
        const float sc = a.ws ? a.ws[a.row_scale ? n : 0] : a.ws_host;
        const float *upr = a.up + n * RANK;
        float acc[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int j = 0; j < RANK; ++j) {
            const float u = upr[j];
            acc[0] = fmaf(u, dn[j].x, acc[0]);
            acc[1] = fmaf(u, dn[j].y, acc[1]);
            acc[2] = fmaf(u, dn[j].z, acc[2]);
            acc[3] = fmaf(u, dn[j].w, acc[3]);
        }
        const float nzv[4] = {nz_cur.x, nz_cur.y, nz_cur.z, nz_cur.w};
        float d[4], r[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) d[e] = acc[e] * a.lora_scale;
        sr_row<4>(d, nzv, row_scale(sc), r);
        stream_store4(a.out + n * a.K + k0, add_sat8_pack(wp_cur, r));
    }
}

// The same fused form on the matrix cores.  v_mfma_f32_32x32x2_f32 adds two products per output to
// its accumulator, the k = 0 product first and each with a single rounding, so a sequence of them
// over j = (0,1), (2,3), ... is the fma chain in increasing j of the definition above, bit for bit
// (the parity tests check this against a CPU fmaf chain).  The output block is computed transposed,
// D[k][n] = sum_j down[j][k] * up[n][j]: a lane then holds, for ONE weight row n, four groups of
// four consecutive k, so the rounding step works on 16-byte noise and 4-byte weight pieces.
//
// A workgroup of 8 waves owns 256 columns (ranks 48 and 64: 4 waves, 128 columns) and walks blocks of 32 rows (every bands-th one).  The noise of a
// block goes from global memory straight into one of two LDS tiles (buffer_load ... lds: a wave
// instruction moves 1 KB of one noise row, no registers involved) while the block before it is
// worked on; weights and `up` travel through registers.  Every wave takes the 32 x 32 piece of its
// own 32 columns from the tiles in the layout above; results go back through the weight tile so that
// they leave in 256-byte runs.  Each wave keeps its slice of `down` in RANK/2 registers.
//
// The product of block i+1 is computed while block i is rounded: the matrix instructions (64 cycles
// each, one dependent chain) are dealt out between the vector instructions of the rounding, so a
// wave keeps both units busy instead of using them in turn.
//
// Ranks beyond 32 (large LoRAs, stacks of LoRAs with their factors side by side): the product is what bounds the kernel,
// RANK / 2 matrix instructions of 64 cycles per 32 x 32 piece and wave, two to four times the time of the rounding's vector
// instructions, with which they share the SIMD.  9216 x 3072: rank 64 57 us, rank 128 91 us (240 and 451 us on the vector
// ALUs, every element fetching its column of `down` from L2).  Rank 64 in workgroups of four waves, three to a CU: 57 us
// against 62 us in one workgroup of eight; from 96 on a wave's slice of `down` leaves room for two waves on a SIMD
// either way, and the workgroup of eight is the faster one (79 us against 87 us at rank 96).
typedef float v16f __attribute__((ext_vector_type(16)));
typedef float v4f __attribute__((ext_vector_type(4)));
typedef int v4i_t __attribute__((ext_vector_type(4)));

template <int RANK, bool DRAWN>
struct MfmaMergeLds {
    static constexpr int WAVES = RANK == 48 || RANK == 64 ? 4 : 8, COLS = WAVES * 32;
    // One wave load moves 1 KB of noise: NZ_ROWS rows of the tile.  Pitch 260 words: the column reads of 16 rows hit 16
    // different bank groups; of two rows in one piece the second has its 16-byte chunks swapped in groups of four.
    static constexpr int NZ_SIZE = DRAWN ? 2 : 4;   // bytes of noise to an element
    static constexpr int NZ_ROWS = 1024 / (COLS * NZ_SIZE), NZ_PITCH = 1024 + 16;
    static constexpr int UPV = RANK <= 32 ? 1 : 4;   // products whose `up` operands one LDS read brings
    static constexpr int UP_PITCH = RANK * 4 + 4 * UPV;
    static constexpr int WB_PITCH = COLS + 16;
    static constexpr int NZ_BYTES = 32 / NZ_ROWS * NZ_PITCH;
    static constexpr int NZ = 0, UP = 2 * NZ_BYTES, WB = UP + ((32 * UP_PITCH + 15) / 16) * 16;
    static constexpr int BYTES = WB + 32 * WB_PITCH;
};

// Workgroup barrier for data exchanged through LDS only: waits for this wave's LDS operations and leaves its global
// loads and stores in flight (__syncthreads() would wait for those as well).
__device__ __forceinline__ void lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// One wave-wide load of 16 bytes per lane from a buffer straight into LDS: lane l lands at lds_base + 16 l.  Bytes
// beyond the buffer's size arrive as zeros.  The compiler does not see this load: what waits for it is an explicit
// s_waitcnt vmcnt in the caller.
__device__ __forceinline__ void buffer_to_lds16(v4i_t rsrc, uint32_t lds_base, uint32_t voffset, uint32_t soffset) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds"
                 :
                 : "s"(lds_base), "v"(voffset), "s"(rsrc), "s"(soffset)
                 : "memory", "m0");
}

// p and bytes are the same in every lane; readfirstlane tells the compiler so (64-bit address arithmetic runs on the
// vector ALUs and would otherwise leave the descriptor in vector registers, where a buffer instruction cannot take it).
__device__ __forceinline__ v4i_t buffer_resource(const void *p, uint32_t bytes) {
    const uint64_t a = (uint64_t)p;
    v4i_t r = {__builtin_amdgcn_readfirstlane((int)(uint32_t)a), __builtin_amdgcn_readfirstlane((int)((uint32_t)(a >> 32) & 0xffffu)),
               __builtin_amdgcn_readfirstlane((int)bytes), 0x00020000};
    return r;
}

// PAD: a.rank is a multiple of 4 below RANK, and the products beyond it are 0 * 0, which leave the sum as it is.
template <int RANK, bool PAD, bool DRAWN>
__global__ __launch_bounds__((MfmaMergeLds<RANK, DRAWN>::WAVES * 64), RANK <= 32 ? 4 : RANK <= 64 ? 3 : 2) void lora_merge_mfma_kernel(const MergeArgs a, int bands) {
    using T = MfmaMergeLds<RANK, DRAWN>;
    constexpr int NT = T::WAVES * 64, P = RANK / 2;
    static_assert(P % T::UPV == 0, "the products of a piece, UPV at a time");
    __shared__ __attribute__((aligned(16))) char lds[T::BYTES];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int l32 = lane & 31, half = lane >> 5;
    // Workgroup (band, column block) takes the row blocks band, band + bands, band + 2 bands, ... of its 256 columns,
    // so that the workgroups running at the same time read neighbouring rows.
    const int64_t nblocks = (a.N + 31) / 32;
    const int band = blockIdx.y;
    const int count = (int)((nblocks - band + bands - 1) / bands);
    if (count <= 0) return;
    auto block_of = [&](int it) { return band + (int64_t)it * bands; };

    const int64_t k0 = (int64_t)blockIdx.x * T::COLS;      // first column of the workgroup (K % 16 == 0 here)
    const int64_t kcol = k0 + wave * 32 + l32;             // this lane's column
    const int rank = PAD ? a.rank : RANK;
    float da[P];
#pragma unroll
    for (int p = 0; p < P; ++p) {
        const bool in = kcol < a.K && 2 * p + half < rank;
        const float v = a.down[in ? (int64_t)(2 * p + half) * a.K + kcol : 0];
        da[p] = in ? v : 0.0f;
    }

    // Noise: wave w moves 1 KB pieces w, w + WAVES, ... of a block (NZ_ROWS rows each), a lane 16 bytes.  The buffer
    // starts at the block's first row and the workgroup's first column and ends with the array, so rows past N
    // read as zeros (their results are not stored).
    const uint32_t row_bytes = (uint32_t)a.K * T::NZ_SIZE;
    const uint32_t lds_base = (uint32_t)(uintptr_t)lds;
    constexpr int NZ_LANES = 64 / T::NZ_ROWS;   // of a wave load, to a row
    const uint32_t nz_lane = DRAWN ? (uint32_t)(lane / NZ_LANES) * row_bytes + (uint32_t)(lane % NZ_LANES) * 16u
                             : T::NZ_ROWS == 1 ? (uint32_t)lane * 16u : (uint32_t)half * row_bytes + (uint32_t)(l32 ^ (4 * half)) * 16u;
    auto fetch_noise = [&](int64_t nb, int buf) __attribute__((always_inline)) {
        const int64_t first = nb * 32 * a.K + k0;
        const int64_t left = (a.N * a.K - first) * T::NZ_SIZE;
        const v4i_t rsrc = buffer_resource(DRAWN ? (const char *)(a.drawn + first) : (const char *)(a.noise + first), left < 0xffffffffll ? (uint32_t)left : 0xffffffffu);
#pragma unroll
        for (int i = 0; i < 32 / (T::NZ_ROWS * T::WAVES); ++i)
            buffer_to_lds16(rsrc, lds_base + T::NZ + buf * T::NZ_BYTES + (wave + T::WAVES * i) * T::NZ_PITCH, nz_lane,
                            (uint32_t)((wave + T::WAVES * i) * T::NZ_ROWS) * row_bytes);
    };
    // Weights (one 16-byte piece per thread: of one row), the row scale and the 16-byte pieces of
    // the 32 rows of `up` (a.rank % 4 == 0: a piece is either in its row or beyond it), through registers.
    constexpr int UPV = T::UPV;
    typedef float upv_t __attribute__((ext_vector_type(UPV)));
    constexpr int UP_PIECES = 32 * RANK / 4;             // 16-byte pieces of the padded block of `up`
    constexpr int UPT = (UP_PIECES + NT - 1) / NT;       // pieces per thread
    const int wb_row = tid / (T::COLS / 16), wb_col = tid % (T::COLS / 16);
    const bool wb_col_ok = k0 + wb_col * 16 < a.K;
    auto clampn = [&](int64_t n) { return n < a.N ? n : a.N - 1; };  // rows past the end repeat the last one, unstored
    auto fetch_weights = [&](int64_t nb, v4u_t &wb, float &sc) __attribute__((always_inline)) {
        if (wb_col_ok) wb = *(const v4u_t *)(a.w + clampn(nb * 32 + wb_row) * a.K + k0 + wb_col * 16);
        sc = a.ws ? a.ws[a.row_scale ? clampn(nb * 32 + l32) : 0] : a.ws_host;
    };
    auto fetch_up = [&](int64_t nb, v4f (&up)[UPT]) __attribute__((always_inline)) {
#pragma unroll
        for (int u = 0; u < UPT; ++u) {
            const int piece = tid + u * NT, row = piece * 4 / RANK, j = piece * 4 % RANK;
            if (piece < UP_PIECES && j < rank) up[u] = *(const v4f *)(a.up + clampn(nb * 32 + row) * rank + j);
        }
    };
    auto park_up = [&](const v4f (&up)[UPT]) __attribute__((always_inline)) {
#pragma unroll
        for (int u = 0; u < UPT; ++u) {
            const int piece = tid + u * NT;
            if (piece < UP_PIECES) {
                float *row = (float *)(lds + T::UP + (piece * 4 / RANK) * T::UP_PITCH), *dst = row + piece * 4 % RANK;
                if constexpr (UPV == 1) {
                    dst[0] = up[u].x, dst[1] = up[u].y, dst[2] = up[u].z, dst[3] = up[u].w;
                } else {  // a lane's operands of consecutive products, ranks half, 2 + half, 4 + half, ..., side by side
                    dst = row + piece * 4 % RANK / 2;
                    *(float2 *)dst = make_float2(up[u].x, up[u].z);
                    *(float2 *)(dst + P) = make_float2(up[u].y, up[u].w);
                }
            }
        }
    };
    auto up_operands = [&](int p) __attribute__((always_inline)) {  // of products p ... p + UPV - 1
        upv_t v;
        __builtin_memcpy(&v, __builtin_assume_aligned(lds + T::UP + l32 * T::UP_PITCH + (UPV == 1 ? 2 * p + half : half * P + p) * 4, UPV * 4), UPV * 4);
        return v;
    };
    auto product = [&](int p0, int p1, v16f &acc) __attribute__((always_inline)) {
#pragma unroll
        for (int p = p0; p < p1; p += UPV) {
            const upv_t u = up_operands(p);
#pragma unroll
            for (int e = 0; e < UPV; ++e) acc = __builtin_amdgcn_mfma_f32_32x32x2f32(da[p + e], u[e], acc, 0, 0, 0);
        }
    };

    v4f up_r[UPT] = {};
    v4u_t wb_r = {};
    float sc_r = 1.0f;
    v16f acc_cur, acc_next;
#pragma unroll
    for (int i = 0; i < 16; ++i) acc_cur[i] = 0.0f;
    // the first block's product; every later one is computed beside the rounding of its predecessor
    fetch_up(block_of(0), up_r);
    fetch_noise(block_of(0), 0);
    fetch_weights(block_of(0), wb_r, sc_r);
    park_up(up_r);
    fetch_up(block_of(1), up_r);
    lds_barrier();
    product(0, P, acc_cur);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the first block's noise is in its tile
    lds_barrier();

    for (int it = 0; it < count; ++it) {
        const int64_t nb = block_of(it);
        const int buf = it & 1;
        const char *nz_tile = lds + T::NZ + buf * T::NZ_BYTES;
        park_up(up_r);  // of the next block
        *(v4u_t *)(lds + T::WB + wb_row * T::WB_PITCH + wb_col * 16) = wb_r;
        const float sc = sc_r;
        lds_barrier();  // this block's noise landed before the last barrier of the block before (or of the prologue)
        if (it + 1 < count) {
            fetch_noise(block_of(it + 1), buf ^ 1);
            fetch_weights(block_of(it + 1), wb_r, sc_r);
        }
        if (it + 2 < count) fetch_up(block_of(it + 2), up_r);

        uint32_t o[4];
        auto weight_quad = [&](int q) __attribute__((always_inline)) {
            return *(const uint32_t *)(lds + T::WB + l32 * T::WB_PITCH + wave * 32 + 8 * q + 4 * half);
        };
#pragma unroll
        for (int i = 0; i < 16; ++i) acc_next[i] = 0.0f;
        if constexpr (DRAWN) {
            // floor(xs) + (noise < frac) is the whole number above z = xs - noise, unless z is so close to one that the other
            // halves of the words, or the roundings on the way, leave it open.  How far z may be from the definition's: 2^-17, a
            // word's upper half taken at the middle of its range; 2^-24 * 2.1, the roundings of noise and fraction; and 7 * 2^-24
            // * |xs|, |xs| <= |z| + 1: two units for the reciprocal and one each for its product with lora_scale, the two fma
            // steps, and the definition's own product and quotient.  Together at most 1.08 * 2^-17 + 7 * 2^-24 * |z|; 1.125 * 2^-17
            // is asked for.  Of 256 elements with |z| of a few units one group in 200 is left open and redone.
            const float f = __builtin_amdgcn_rcpf(sc) * a.lora_scale;
            // (lora_scale 0, a LoRA switched off by its strength: xs is 0, or NaN with a sum that is not finite, and so is z plus the
            // noise.  Left to the definition every element drew its word again: 12288 x 3072, rank 32, 133 us with the noise for 66.)
            const bool usual = sc >= 0x1p-20f && sc <= 0x1p+20f && (fabsf(f) >= 0x1p-100f || a.lora_scale == 0.0f) && fabsf(f) <= 0x1p+100f;
            float zmax[4] = {};
            uint32_t dmin[4], dmax[4];   // (bits, so that a NaN is the largest)
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                product(q * P / (4 * UPV) * UPV, (q + 1) * P / (4 * UPV) * UPV, acc_next);
                const uint2 n4 = *(const uint2 *)(nz_tile + (l32 / T::NZ_ROWS) * T::NZ_PITCH + (l32 % T::NZ_ROWS) * (T::COLS * 2) + (wave * 32 + 8 * q + 4 * half) * 2);
                const uint32_t n[4] = {n4.x & 0xffffu, n4.x >> 16, n4.y & 0xffffu, n4.y >> 16};
                float r[4];
                dmin[q] = 0xffffffffu, dmax[q] = 0u;
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const float z = __builtin_fmaf((float)n[e], -0x1p-16f, __builtin_fmaf(acc_cur[4 * q + e], f, -0x1p-17f));
                    r[e] = ceilf(z);
                    const uint32_t d = __float_as_uint(r[e] - z);
                    zmax[q] = fmaxf(zmax[q], fabsf(z)), dmin[q] = min(dmin[q], d), dmax[q] = max(dmax[q], d);
                }
                o[q] = add_sat8_pack(weight_quad(q), r);
            }
#pragma unroll
            for (int i = 0; i < P; ++i) {
                __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);        // one matrix instruction
                __builtin_amdgcn_sched_group_barrier(0x002, P <= 96 ? 192 / P : 2, 0);  // its share of the vector work
            }
            __builtin_amdgcn_sched_barrier(0);
            uint32_t open = 0;   // groups of four that have a lane without an answer
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const float eps = __builtin_fmaf(zmax[q], 7.0f * 0x1p-24f, 0x1.2p-17f);
                const bool sure = usual && zmax[q] <= 64.0f && dmin[q] >= __float_as_uint(eps) && dmax[q] <= __float_as_uint(1.0f - eps);
                open |= __builtin_amdgcn_ballot_w64(!sure) != 0 ? 1u << q : 0u;
            }
            const uint32_t e0 = (uint32_t)(clampn(nb * 32 + l32) * a.K + k0) + wave * 32 + 4 * half;
            while (__builtin_expect(open != 0, 0)) {  // by the definition, from the whole words
                const int q = __builtin_ctz(open);
                open &= open - 1;
                const uint32_t e = e0 + 8 * q, i = e / a.lanes, lane_of = e - i * a.lanes;
                float r[4];
#pragma unroll
                for (int t = 0; t < 4; ++t) {
                    uint32_t x[4];
                    philox(i / 4, lane_of + t, a.seed_lo, a.seed_hi, x);
                    const uint32_t lo = i & 1 ? x[1] : x[0], hi = i & 1 ? x[3] : x[2];
                    const float acc = q == 0 ? acc_cur[t] : q == 1 ? acc_cur[4 + t] : q == 2 ? acc_cur[8 + t] : acc_cur[12 + t];
                    r[t] = sr_round(acc * a.lora_scale / sc, uniform_of(i & 2 ? hi : lo));
                }
                const uint32_t v = add_sat8_pack(weight_quad(q), r);
                o[0] = q == 0 ? v : o[0], o[1] = q == 1 ? v : o[1], o[2] = q == 2 ? v : o[2], o[3] = q == 3 ? v : o[3];
            }
        } else {
            const RowScale rs = row_scale(sc);
            float d[16];
            SrGuard guard;
            auto noise_quad = [&](int q, float (&nzv)[4]) __attribute__((always_inline)) {
                const int chunk = wave * 8 + 2 * q + half;
                const v4f nz = *(const v4f *)(T::NZ_ROWS == 1 ? nz_tile + l32 * T::NZ_PITCH + chunk * 16
                                                              : nz_tile + (l32 >> 1) * T::NZ_PITCH + (l32 & 1) * 512 + (chunk ^ (4 * (l32 & 1))) * 16);
                nzv[0] = nz.x, nzv[1] = nz.y, nzv[2] = nz.z, nzv[3] = nz.w;
            };
#pragma unroll
            for (int q = 0; q < 4; ++q) {  // the noise is read again where it is used: sixteen registers fewer across the block
                float nzv[4], dq[4];
                noise_quad(q, nzv);
#pragma unroll
                for (int e = 0; e < 4; ++e) dq[e] = d[4 * q + e] = acc_cur[4 * q + e] * a.lora_scale;
                guard.add(dq, nzv);
            }
            if (__builtin_amdgcn_ballot_w64(!guard.fast(rs)) == 0) {
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    product(q * P / (4 * UPV) * UPV, (q + 1) * P / (4 * UPV) * UPV, acc_next);
                    float r[4], nzv[4];
                    noise_quad(q, nzv);
#pragma unroll
                    for (int e = 0; e < 4; ++e) r[e] = sr_round(fast_quotient(d[4 * q + e], rs), nzv[e]);
                    o[q] = add_sat8_pack(weight_quad(q), r);
                }
#pragma unroll
                for (int i = 0; i < P; ++i) {
                    __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);        // one matrix instruction
                    __builtin_amdgcn_sched_group_barrier(0x002, P <= 112 ? 224 / P : 2, 0);  // its share of the vector work
                }
            } else {  // some lane needs the division: every lane takes it
                product(0, P, acc_next);
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    float r[4], nzv[4];
                    noise_quad(q, nzv);
#pragma unroll
                    for (int e = 0; e < 4; ++e) r[e] = sr_round(d[4 * q + e] / rs.sc, nzv[e]);
                    o[q] = add_sat8_pack(weight_quad(q), r);
                }
            }
        }
        acc_cur = acc_next;
        // results: back through the weight tile (each lane overwrites exactly the bytes it read),
        // then one 16-byte store per thread
#pragma unroll
        for (int q = 0; q < 4; ++q) *(uint32_t *)(lds + T::WB + l32 * T::WB_PITCH + wave * 32 + 8 * q + 4 * half) = o[q];
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the next block's noise is in its tile (and this wave's last store is out)
        lds_barrier();
        const v4u_t obv = *(const v4u_t *)(lds + T::WB + wb_row * T::WB_PITCH + wb_col * 16);
        const int64_t nrow = nb * 32 + wb_row;
        if (nrow < a.N && wb_col_ok) stream_store16(a.out + nrow * a.K + k0 + wb_col * 16, make_uint4(obv.x, obv.y, obv.z, obv.w));
        lds_barrier();  // the weight and `up` tiles are free for the next block
    }
}

template <int RANK, bool DRAWN>
int launch_mfma(const MergeArgs &a, hipStream_t st) {
    using T = MfmaMergeLds<RANK, DRAWN>;
    const int64_t col_blocks = (a.K + T::COLS - 1) / T::COLS, nblocks = (a.N + 31) / 32;
    if (col_blocks > 0x7fffffffll) return I8F_ERR_UNSUPPORTED;
    // Two workgroups fit a CU (LDS), so 512 run at a time.  Bands are chosen for the fewest block steps on the busiest
    // CU: rounds of 512 workgroups times the blocks of a band, plus half a step for a workgroup's start (its first
    // product is not overlapped with anything); a tie goes to fewer rounds, then to more bands (more of the chip reading).
    // (Ranks 48 and 64 in workgroups of four waves, three to a CU; above it the slice of `down` leaves room for one of eight.)
    constexpr int64_t SLOTS = RANK <= 32 ? 512 : RANK <= 64 ? 768 : 256;
    int64_t max_bands = 4 * SLOTS / col_blocks + 1;
    if (max_bands > nblocks) max_bands = nblocks;
    if (max_bands > 65535) max_bands = 65535;
    int64_t bands = 1, best = -1, best_rounds = 0;
    for (int64_t b = 1; b <= max_bands; ++b) {
        const int64_t rounds = (col_blocks * b + SLOTS - 1) / SLOTS, steps2 = 2 * ((nblocks + b - 1) / b) + 1;
        if (best < 0 || rounds * steps2 < best || (rounds * steps2 == best && rounds <= best_rounds))
            best = rounds * steps2, best_rounds = rounds, bands = b;
    }
    const dim3 grid((unsigned)col_blocks, (unsigned)bands);
    if constexpr (!DRAWN) {
        if (a.rank == RANK) {
            hipLaunchKernelGGL((lora_merge_mfma_kernel<RANK, false, false>), grid, dim3(T::WAVES * 64), 0, st, a, (int)bands);
            return check_launch();
        }
    }
    hipLaunchKernelGGL((lora_merge_mfma_kernel<RANK, true, DRAWN>), grid, dim3(T::WAVES * 64), 0, st, a, (int)bands);
    return check_launch();
}

template <bool DRAWN>
int launch_rank(const MergeArgs &a, hipStream_t st) {
    // the next larger rank that is built, the rest zeros: a padded product costs no more than its share of RANK
    // (3072 x 1552, an odd multiple of 16 columns, rank 32: 13.5 us against 22.3 us for the band form below).  Up to 32
    // the noise stream hides the products and powers of two are enough; beyond, the products are the time, so every 16
    // up to 128 and every 32 up to 256 is built: 9216 x 3072, us, padded to the next of 64, 96, 128, 192, 256 and as it
    // is: rank 48 54.6 and 47.1, 80 78.2 and 70.2, 112 92.3 and 84.1, 160 144.5 and 126.9, 224 186.1 and 154.6.
    if (a.rank <= 4) return launch_mfma<4, DRAWN>(a, st);
    if (a.rank <= 8) return launch_mfma<8, DRAWN>(a, st);
    if (a.rank <= 16) return launch_mfma<16, DRAWN>(a, st);
    if (a.rank <= 32) return launch_mfma<32, DRAWN>(a, st);
    if (a.rank <= 48) return launch_mfma<48, DRAWN>(a, st);
    if (a.rank <= 64) return launch_mfma<64, DRAWN>(a, st);
    if (a.rank <= 80) return launch_mfma<80, DRAWN>(a, st);
    if (a.rank <= 96) return launch_mfma<96, DRAWN>(a, st);
    if (a.rank <= 112) return launch_mfma<112, DRAWN>(a, st);
    if (a.rank <= 128) return launch_mfma<128, DRAWN>(a, st);
    if (a.rank <= 160) return launch_mfma<160, DRAWN>(a, st);
    if (a.rank <= 192) return launch_mfma<192, DRAWN>(a, st);
    if (a.rank <= 224) return launch_mfma<224, DRAWN>(a, st);
    if constexpr (DRAWN) return I8F_ERR_UNSUPPORTED;   // (FEW_MAX_RANK)
    else return launch_mfma<256, DRAWN>(a, st);
}

template <int RANK>
int launch_band(const MergeArgs &a, hipStream_t st) {
    const unsigned col_blocks = (unsigned)((a.K + 1023) / 1024);
    // enough row bands to fill the chip several times over, each long enough to amortise its slice of `down`
    int64_t bands = (256 * 12 + col_blocks - 1) / col_blocks;
    int64_t rows = (a.N + bands - 1) / bands;
    if (rows < 16) rows = 16;
    bands = (a.N + rows - 1) / rows;
    if (bands > 65535) return I8F_ERR_UNSUPPORTED;
    hipLaunchKernelGGL((lora_merge_band_kernel<RANK>), dim3(col_blocks, (unsigned)bands), dim3(256), 0, st, a, (int)rows);
    return check_launch();
}

int run(MergeArgs &a, hipStream_t st) {
    if (a.N == 0 || a.K == 0) return I8F_OK;
    if (a.N > 65535 * 1024ll) return I8F_ERR_UNSUPPORTED;
    const bool fused = a.delta == nullptr;
    auto al = [](const void *p, int n) { return p == nullptr || (uintptr_t)p % n == 0; };
    const bool vec = a.K % 4 == 0 && al(a.w, 4) && al(a.out, 4) && al(a.noise, 16) && al(a.delta, 16) &&
                     (!fused || al(a.down, 16));
    // (K < 2^24: the 32 rows of a block are addressed with 32-bit byte offsets from the block's first element)
    if (fused && vec && a.w && a.N < (1ll << 31) && a.K % 16 == 0 && a.K < (1 << 24) && al(a.up, 16) && al(a.w, 16) && al(a.out, 16) &&
        a.rank % 4 == 0 && a.rank > 0 && a.rank <= 256)
        return launch_rank<false>(a, st);
    if (fused && vec && a.w && a.N < (1ll << 31)) {
        switch (a.rank) {
        case 4: return launch_band<4>(a, st);
        case 8: return launch_band<8>(a, st);
        case 16: return launch_band<16>(a, st);
        case 32: return launch_band<32>(a, st);
        default: break;  // other ranks take the per-element kernel below
        }
    }
    // grid.y is limited to 65535: fold larger N into several launches
    for (int64_t n0 = 0; n0 < a.N; n0 += 65535) {
        MergeArgs b = a;
        const int64_t rows = a.N - n0 < 65535 ? a.N - n0 : 65535;
        b.N = rows;
        if (b.w) b.w += n0 * a.K;
        b.out += n0 * a.K;
        b.noise += n0 * a.K;
        if (b.delta) b.delta += n0 * a.K;
        if (b.up) b.up += n0 * a.rank;
        if (b.ws && b.row_scale) b.ws += n0;
        const int per_block = 256 * (vec ? 4 : 1);
        dim3 grid((unsigned)((a.K + per_block - 1) / per_block), (unsigned)rows);
        if (vec) {
            if (fused) hipLaunchKernelGGL((lora_merge_kernel<4, true>), grid, dim3(256), 0, st, b);
            else hipLaunchKernelGGL((lora_merge_kernel<4, false>), grid, dim3(256), 0, st, b);
        } else {
            if (fused) hipLaunchKernelGGL((lora_merge_kernel<1, true>), grid, dim3(256), 0, st, b);
            else hipLaunchKernelGGL((lora_merge_kernel<1, false>), grid, dim3(256), 0, st, b);
        }
        if (int rc = check_launch()) return rc;
    }
    return I8F_OK;
}

}  // namespace
}  // namespace i8f

extern "C" int i8f_sr_quant_delta(const float *x, const float *scale, float scale_host, int scale_mode,
                                  const float *noise, int64_t N, int64_t K, int8_t *dq, void *stream) {
    using namespace i8f;
    if (N < 0 || K < 0) return I8F_ERR_INVALID;
    if (scale_mode != I8F_SCALE_TENSOR && scale_mode != I8F_SCALE_ROW) return I8F_ERR_INVALID;
    if (N == 0 || K == 0) return I8F_OK;
    if (!x || !noise || !dq) return I8F_ERR_INVALID;
    if (scale_mode == I8F_SCALE_ROW && !scale) return I8F_ERR_INVALID;
    if (int rc = check_device()) return rc;
    MergeArgs a{};
    a.ws = scale, a.ws_host = scale_host, a.row_scale = scale_mode == I8F_SCALE_ROW;
    a.delta = x, a.noise = noise, a.N = N, a.K = K, a.out = dq;
    return run(a, (hipStream_t)stream);
}

extern "C" int i8f_lora_merge_sr(const int8_t *w, const float *w_scale, float w_scale_host, int scale_mode,
                                 const float *delta, const float *up, const float *down, int64_t rank,
                                 float lora_scale, const float *noise, int64_t N, int64_t K, int8_t *w_out,
                                 void *stream) {
    using namespace i8f;
    if (N < 0 || K < 0) return I8F_ERR_INVALID;
    if (scale_mode != I8F_SCALE_TENSOR && scale_mode != I8F_SCALE_ROW) return I8F_ERR_INVALID;
    if (N == 0 || K == 0) return I8F_OK;
    if (!w || !noise || !w_out) return I8F_ERR_INVALID;
    if (scale_mode == I8F_SCALE_ROW && !w_scale) return I8F_ERR_INVALID;
    if (!delta) {
        if (!up || !down || rank < 0) return I8F_ERR_INVALID;
        if (rank > 256) return I8F_ERR_UNSUPPORTED;
    }
    if (int rc = check_device()) return rc;
    MergeArgs a{};
    a.w = w, a.ws = w_scale, a.ws_host = w_scale_host, a.row_scale = scale_mode == I8F_SCALE_ROW;
    a.delta = delta, a.up = up, a.down = down, a.rank = (int)rank, a.lora_scale = lora_scale;
    a.noise = noise, a.N = N, a.K = K, a.out = w_out;
    return run(a, (hipStream_t)stream);
}

namespace i8f {

int64_t merge_few_workspace_bytes(int64_t N, int64_t K, int64_t rank, int count) {
    return up256(2 * N * K) + (count > 1 ? up256(4 * N * rank) + 4 * K * rank : 0);
}

int merge_few(const DrawnCall &c, hipStream_t st) {
    const int64_t N = c.N, K = c.K, columns = (c.lanes + 2047) / 2048, chunks = (N * K + 4 * c.lanes - 1) / (4 * c.lanes);
    // workgroups for the factors: 4 elements a thread, one round of the chip at most
    int64_t extra = c.count > 1 ? ((N + K) * c.rank + 1023) / 1024 : 0;
    extra = ((extra < 2048 ? extra : 2048) + columns - 1) / columns;
    MergeArgs a{};
    a.w = c.w, a.ws = c.ws, a.ws_host = c.ws_host, a.row_scale = c.row_scale;
    a.up = c.factors[0].up, a.down = c.factors[0].down, a.rank = c.rank, a.lora_scale = c.lora_scale;
    a.N = N, a.K = K, a.out = c.out;
    a.drawn = (const uint16_t *)c.workspace, a.seed_lo = (uint32_t)c.seed, a.seed_hi = (uint32_t)(c.seed >> 32), a.lanes = (uint32_t)c.lanes;
    Stack stack{};
    stack.n = c.count;
    for (int i = 0; i < c.count; ++i) {
        stack.up[i] = c.factors[i].up, stack.down[i] = c.factors[i].down, stack.mult[i] = c.factors[i].mult;
        stack.first[i + 1] = stack.first[i] + (int)c.factors[i].rank;
    }
    if (c.count > 1) {
        stack.N = (uint32_t)N, stack.K = (uint32_t)K;
        stack.up_out = (float *)((char *)c.workspace + up256(2 * N * K));
        stack.down_out = (float *)((char *)stack.up_out + up256(4 * N * c.rank));
        a.up = stack.up_out, a.down = stack.down_out;
    }
    auto draw = [&](int64_t blocks, int64_t factor_blocks) {   // rows of blocks
        hipLaunchKernelGGL(draw_words_kernel, dim3((unsigned)columns, (unsigned)blocks), dim3(256), 0, st, a.seed_lo, a.seed_hi, a.lanes,
                           (uint32_t)(N * K), (uint16_t *)c.workspace, (uint32_t)factor_blocks, stack);
        return check_launch();
    };
    const bool once = chunks + extra <= 65535;
    if (int rc = draw(once ? chunks + extra : extra, extra)) return rc;
    if (!once)
        if (int rc = draw(chunks, 0)) return rc;
    return launch_rank<true>(a, st);
}

}  // namespace i8f
