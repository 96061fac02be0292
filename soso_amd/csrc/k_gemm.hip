// k_gemm.hip -- products of several tokens per weight row (GpuDispatch::matmul,
// crates/soso-llm-core/src/gpu.rs:443-455): Q4_K, Q6_K and Q8_0 rows against x
// split into two f16 parts, on the f16 matrix cores.
//
// Arithmetic.  x is scaled by a power of two 2^s per token and 256-column
// super-block (its largest element into [2^14, 2^15); s <= 126) and written as hi + lo,
// two f16 numbers whose sum is within 2^-23 of every element above 2^-16 of
// the block's largest, and within 2^-39 of the largest below that (the integer
// kernels' digits: within 2^-22 of the largest of 128 or 256 columns).  What
// would push the rest below that floor is taken out (gm_take_out) and marked by
// a negative 2^-s: single elements, whose products are added at the end with the
// weights dequantized exactly, and where the two 128-column halves are too far
// apart for one scale the larger half, which goes through the matrix cores by
// itself at the end.  Weights times the block scales are whole
// numbers: Q4_K's sc q (up to 945) exact in f16, Q6_K's sc (q - 32) (up to
// 4096) exact as two f16, Q8_0's codes exact (its f32 scales are applied to the
// block's sums).  Every product is exact in the f32 accumulators; a
// super-block's sum S is one chain, and per super-block out += 2^-s d S in f32,
// for Q4_K 2^-s (d S - dmin M) with M = sum m_j xsum_j over the eight
// sub-blocks' f32 sums of x, split in two as x is (a sum of 32, scaled by 2^-5
// more: within 2^-23 of sums above 2^-11 of the block's largest element, 2^-34 of
// that element below).  Against 64 bits (normal x,
// 4096 x 4096): 4.0e-7 (Q4_K), 1.8e-7 (Q6_K), 1.4e-7 (Q8_0) where the integer
// digits gave 1.3e-6, 9.0e-7 and 5.4e-7; with x's mean at 3 or 100 times its spread,
// all positive, heavy-tailed or of blocks far apart in size 0.1 to 0.9 of their error
// (Q4_K with a mean, against the batched vector kernel: 7.7e-8 after 4.2e-8).  A block that holds an Inf or a NaN
// gets 2^-s = NaN: NaN products, as the CPU's dot gives Inf or NaN.
//
// v_mfma_f32_32x32x16_f16 operands (lane l: n = l % 32, f = l / 32):
//   A (32 x 16): token n, k = 8 f .. 8 f + 7      <- LDS, x as staged below
//   B (16 x 32): weight row n, the same k          <- registers, dequantized
//   D (32 x 32): column n = weight row, register i = token 8 (i / 4) + 4 f + i % 4
// A and B only have to agree on which element a (f, byte) slot of a step
// holds, so the order is the weights'.  Q4_K and Q8_0: step t = 0..3 of a
// 64-element unit takes its 32-element block t / 2, elements 16 f + 8 (t % 2) +
// {0, 2, 1, 3, 4, 6, 5, 7} (the order in which masking a dword with 0x000F000F
// yields byte pairs); Q6_K: quarter t of the unit's half, elements 16 k + 8 f +
// the same eight (k: the unit's parity).
#include "mv_core.hpp"

#include <algorithm>

typedef _Float16 gm_h2 __attribute__((ext_vector_type(2)));
typedef _Float16 gm_h8 __attribute__((ext_vector_type(8)));
typedef float gm_f4 __attribute__((ext_vector_type(4)));
typedef float gm_f16v __attribute__((ext_vector_type(16)));
typedef uint32_t gm_u4 __attribute__((ext_vector_type(4))); // (a HIP uint4 array here ends up in scratch memory)

// Staged x, for tiles of 32 tokens (rows past n are zeros):
//   F [tile][unit][step 4][hi, lo][half f][32 x 16 B]   8 KiB per unit
//   M [tile][super-block][lane 64][16 B]            eight sub-block sums, hi (f = 0) and lo (f = 1)
//   P [tile][super-block][32] f32                   2^-s per token
struct GmX {
    const uint8_t *f, *m;
    const float *p;
};
constexpr int GM_UNIT = 8192, GM_SUMS = 1024;

// Where x is written to LDS token by token, token m's 16 bytes of a piece sit at
// place m ^ gm_swz(unit, step, lo): a token's pieces would else all meet in the
// same banks (two thirds of the LDS cycles of a MoE layer of 512 tokens, gate /
// up 123 -> 98 us).  The 16 places that span the banks are distinct over the
// units and steps of one token (gm_stage_rows), and, with bit 0 of the token,
// over the steps and parts of one unit (the MoE kernel's gather).
__device__ __forceinline__ constexpr int gm_swz(int unit, int step, int lo)
{
    return 4 * step + 2 * (lo ^ ((unit >> 1) & 1)) + (unit & 1);
}
// Lane (n, f)'s fragment of a unit written so (x: its 8 KiB in LDS).
__device__ __forceinline__ gm_h8 gm_frag_at(const uint8_t *x, int lane, int unit, int step, int lo)
{
    return *(const gm_h8 *)(x + step * 2048 + lo * 1024 + ((16 * lane) ^ (16 * gm_swz(unit, step, lo))));
}

__device__ __forceinline__ uint32_t gm_pack(float a, float b)
{
    return __builtin_bit_cast(uint32_t, gm_h2{(_Float16)a, (_Float16)b});
}

// Maximum over the 32 lanes of this lane's half wavefront.
__device__ __forceinline__ float gm_half_max(float v)
{
    auto st = [](float a, uint32_t b) { return fmaxf(a, __uint_as_float(b)); };
    v = st(v, dpp_keep<0xB1>(__float_as_uint(v)));
    v = st(v, dpp_keep<0x4E>(__float_as_uint(v)));
    v = st(v, dpp_keep<0x141>(__float_as_uint(v)));
    v = st(v, dpp_keep<0x140>(__float_as_uint(v)));
    v = st(v, dpp_keep<0x142, 0xA>(__float_as_uint(v)));
    const int lo = __builtin_amdgcn_readlane(__float_as_int(v), 31), hi = __builtin_amdgcn_readlane(__float_as_int(v), 63);
    return __int_as_float((threadIdx.x & 32) ? hi : lo);
}
__device__ __forceinline__ float gm_abs_max(gm_f4 v)
{
    return fmaxf(fmaxf(fabsf(v[0]), fabsf(v[1])), fmaxf(fabsf(v[2]), fabsf(v[3])));
}
// Above this an element of a 128-column half (32 lanes, four finite columns
// each) is taken out: 2^14 times ref, the third largest of its 16 maxima of 8
// columns, so that what stays loses less to the parts' floor than to digits of
// its own (22 bits of up to 16 times its third largest).  A half with no more than
// two such maxima (at most 16 elements) has no third: ref is its smallest
// element, and where the largest is beyond 2^14 times that all are taken out.
__device__ __forceinline__ float gm_outlier_thr(gm_f4 v, float &ref)
{
    const int lane = threadIdx.x & 63;
    float cm = gm_abs_max(v), least = INFINITY;
#pragma unroll
    for (int i = 0; i < 4; i++)
        if (v[i] != 0.0f) least = fminf(least, fabsf(v[i]));
    least = -gm_half_max(-least);
    cm = fmaxf(cm, dpp_f<0xB1>(cm));
    const float largest = gm_half_max(cm);
    for (int r = 0; r < 2; r++) {
        const uint64_t top = __ballot(cm == gm_half_max(cm));
        const uint32_t mine = lane < 32 ? (uint32_t)top : (uint32_t)(top >> 32);
        if (__builtin_ctz(mine) >> 1 == (lane & 31) >> 1) cm = -1.0f;
    }
    const float third = gm_half_max(cm);
    ref = third > 0.0f ? third : least;
    return third > 0.0f || largest <= 16384.0f * least ? 16384.0f * ref : 0.0f;
}

// Takes a super-block's outliers out of v (finite) and returns whether there were
// any (uniform); larger: the lanes of the larger half, where it is beyond 2^14
// times the other's ref.
__device__ __forceinline__ bool gm_take_out(gm_f4 &v, bool &larger)
{
    float ref;
    const float thr = gm_outlier_thr(v, ref);
    bool mine = false;
#pragma unroll
    for (int i = 0; i < 4; i++)
        if (fabsf(v[i]) > thr) {
            v[i] = 0.0f;
            mine = true;
        }
    const float m = gm_half_max(gm_abs_max(v)), all = wave_max_dpp(m);
    const float least = -wave_max_dpp(m > 0.0f ? -ref : -INFINITY); // (every lane takes part)
    larger = m == all && all > 16384.0f * least;
    return __ballot(mine) != 0;
}

// Where the pieces of a token's 256 columns go: as a row of a 32-token tile
// (above), or for TOK token by token -- unit u at 256 u, then step, hi / lo,
// half f of 16 bytes each; sums hi, then lo.
template <bool TOK> struct GmPlace {
    static constexpr int UNIT = TOK ? 256 : GM_UNIT, STEP = TOK ? 64 : 2048, LO = TOK ? 32 : 1024, HALF = TOK ? 16 : 512;
    static constexpr int SUM_LO = TOK ? 16 : 512;
};
constexpr int GM_TOK = 1024, GM_TOK_SUMS = 32; // bytes per token and super-block, TOK

// 256 columns of R tokens (four per lane and token, v[k]) in f16 parts: the
// fragments at xf(k), the sub-blocks' sums at xm(k) (Q4_K) and 2^-s at xp(k), for
// the tokens k < count.  The tokens' steps interleave: one token after another
// left each with the latency of a dozen dependent lane moves.
// row(k): the token's row of its tile (not TOK).  halves: only the larger halves
// that were left out without it (2^-s negative where there is one).  valid: how many
// of the columns are the row's (Q8_0; zeros past them).
template <int FMT, int R, bool TOK, class Row, class XF, class XM, class XP>
__device__ __forceinline__ void gm_stage_rows(gm_f4 (&v)[R], int lane, int count, Row row, XF xf, XM xm, XP xp,
                                              bool halves = false, int valid = 256)
{
    // this lane's group of eight columns: unit u, step st, half f
    const int c8 = lane >> 1;
    int u, st, f;
    if constexpr (FMT == FMT_Q6K) {
        u = 2 * (c8 >> 4) + ((c8 >> 1) & 1);
        st = (c8 >> 2) & 3;
        f = c8 & 1;
    } else {
        u = c8 >> 3;
        st = 2 * ((c8 >> 2) & 1) + (c8 & 1);
        f = (c8 >> 1) & 1;
    }
    using P = GmPlace<TOK>;
    const int at = u * P::UNIT + st * P::STEP + f * P::HALF + 8 * (lane & 1);
    auto st_max = [](float a, uint32_t b) { return fmaxf(a, __uint_as_float(b)); };
    auto st_min = [](float a, uint32_t b) { return fminf(a, __uint_as_float(b)); };
    float mx[R], mn[R], sm[R];
#pragma unroll
    for (int k = 0; k < R; k++) {
        mx[k] = gm_abs_max(v[k]);
        sm[k] = (v[k][0] + v[k][1]) + (v[k][2] + v[k][3]);
        if (sm[k] != sm[k]) mx[k] = INFINITY; // a NaN element (or Inf - Inf): the block is non-finite
    }
    // the maximum over the wavefront and the smallest maximum of its 32-column
    // groups: within 2^14 of each other, nothing is taken out (the two largest
    // 8-column maxima sit in at most two groups of each 128, so both halves'
    // third is at least the smallest group's maximum).  Q8_0, whose last super-block
    // may hold fewer columns: groups of 16, of 8 in a half of 32 columns, without
    // those past the end (at zero they would send every token through the rare code:
    // 333 x 4448 at 64 tokens 20.6 -> 22.6 us)
#define GM_STEP(C, ROWS)                                                                                               \
    _Pragma("unroll") for (int k = 0; k < R; k++) mx[k] = st_max(mx[k], dpp_keep<C, ROWS>(__float_as_uint(mx[k])));
    GM_STEP(0xB1, 0xf)
    if constexpr (FMT == FMT_Q80) {
        const bool in = 4 * lane < valid, short_half = 128 * (lane >> 5) + 64 > valid;
#pragma unroll
        for (int k = 0; k < R; k++) {
            mn[k] = mx[k];
            mx[k] = st_max(mx[k], dpp_keep<0x4E>(__float_as_uint(mx[k])));
            mn[k] = !in ? INFINITY : short_half ? mn[k] : mx[k];
            mn[k] = st_min(mn[k], dpp_keep<0x4E>(__float_as_uint(mn[k])));
        }
    } else {
        GM_STEP(0x4E, 0xf)
        GM_STEP(0x141, 0xf)
#pragma unroll
        for (int k = 0; k < R; k++) mn[k] = mx[k];
    }
#define GM_STEP2(C, ROWS)                                                                                              \
    GM_STEP(C, ROWS)                                                                                                   \
    _Pragma("unroll") for (int k = 0; k < R; k++) mn[k] = st_min(mn[k], dpp_keep<C, ROWS>(__float_as_uint(mn[k])));
    if constexpr (FMT == FMT_Q80) {
        GM_STEP2(0x141, 0xf)
    }
    GM_STEP2(0x140, 0xf)
    GM_STEP2(0x142, 0xA)
    GM_STEP2(0x143, 0xC)
#undef GM_STEP2
#undef GM_STEP
    bool odd = false;
    float sign[R];
#pragma unroll
    for (int k = 0; k < R; k++) {
        mx[k] = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(mx[k]), 63));
        mn[k] = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(mn[k]), 63));
        sign[k] = 1.0f;
        odd = odd || !(mx[k] <= 16384.0f * mn[k]) || !(mx[k] < INFINITY);
    }
    if (__builtin_expect(odd, 0) && !halves) {
        // Zero groups alone call for nothing: where a half has three 8-column maxima
        // above zero its third is at least the smallest of them.  (14336 x 4096 in Q4_K
        // with a zero 32-column group per super-block, 8 / 32 tokens: 28.8 / 54.8 us
        // through the code below, 22.2 / 31.3 with this.)
        odd = false;
#pragma unroll
        for (int k = 0; k < R; k++) {
            float c = gm_abs_max(v[k]);
            c = fmaxf(c, dpp_f<0xB1>(c));
            const uint64_t some = __ballot(c > 0.0f); // two lanes per maximum
            const int n0 = __popc((uint32_t)some), n1 = __popc((uint32_t)(some >> 32));
            const float least = -wave_max_dpp(c > 0.0f ? -c : -INFINITY);
            const bool fine = mx[k] <= 16384.0f * least && mx[k] < INFINITY && (n0 == 0 || n0 >= 6) && (n1 == 0 || n1 >= 6);
            mn[k] = fine ? mx[k] : 0.0f;
            odd = odd || !fine;
        }
    }
    if (__builtin_expect(odd || halves, 0)) { // uniform; rare, so one copy of the code for all tokens
#pragma unroll 1
        for (int k = 0; k < R; k++) {
            gm_f4 w = v[0];
            float m = mx[0], least = mn[0], sum = sm[0], sg = 1.0f;
#pragma unroll
            for (int i = 1; i < R; i++) {
#pragma unroll
                for (int q = 0; q < 4; q++) w[q] = k == i ? v[i][q] : w[q];
                m = k == i ? mx[i] : m;
                least = k == i ? mn[i] : least;
                sum = k == i ? sm[i] : sum;
            }
            if (!(m < INFINITY)) {
                w = gm_f4{0.f, 0.f, 0.f, 0.f};
                m = sum = 0.0f;
                sg = __builtin_nanf("");
            } else if (halves || m > 16384.0f * least) {
                bool larger;
                const bool outliers = gm_take_out(w, larger);
                if ((outliers && !halves) || __ballot(larger) != 0) sg = -1.0f;
                if (larger != halves) w = gm_f4{0.f, 0.f, 0.f, 0.f};
                m = wave_max_dpp(gm_abs_max(w));
                sum = (w[0] + w[1]) + (w[2] + w[3]);
            }
#pragma unroll
            for (int i = 0; i < R; i++) {
#pragma unroll
                for (int q = 0; q < 4; q++) v[i][q] = k == i ? w[q] : v[i][q];
                mx[i] = k == i ? m : mx[i];
                sm[i] = k == i ? sum : sm[i];
                sign[i] = k == i ? sg : sign[i];
            }
        }
    }
    int s[R];
#pragma unroll
    for (int k = 0; k < R; k++) {
        // at most 126: 2^-s is a normal number, so that its sign can mark
        // outliers above a block of subnormals (whose bits all fit at 2^126)
        s[k] = min(126, 15 - __builtin_amdgcn_frexp_expf(mx[k]));
        float e[4], lo[4];
#pragma unroll
        for (int i = 0; i < 4; i++) {
            e[i] = ldexpf(v[k][i], s[k]);
            lo[i] = e[i] - (float)(_Float16)e[i];
        }
        if (k < count) { // uniform
            uint8_t *hd = xf(k) + at, *ld = hd + P::LO;
            if constexpr (!TOK) {
                hd += 16 * (row(k) ^ gm_swz(u, st, 0));
                ld += 16 * (row(k) ^ gm_swz(u, st, 1));
            }
            *(uint2 *)hd = make_uint2(gm_pack(e[0], e[2]), gm_pack(e[1], e[3]));
            *(uint2 *)ld = make_uint2(gm_pack(lo[0], lo[2]), gm_pack(lo[1], lo[3]));
        }
    }
    if constexpr (FMT == FMT_Q4K) {
        // the sub-blocks' sums (8 lanes), scaled by 2^(s - 5): at most 2^15
#pragma unroll
        for (int k = 0; k < R; k++) sm[k] = seg_sum_dpp<8>(sm[k]);
        if ((lane & 7) == 0) {
#pragma unroll
            for (int k = 0; k < R; k++)
                if (k < count) {
                    const float q = ldexpf(sm[k], s[k] - 5);
                    const _Float16 hi = (_Float16)q;
                    uint8_t *d = xm(k) + 2 * (lane >> 3);
                    *(_Float16 *)d = hi;
                    *(_Float16 *)(d + P::SUM_LO) = (_Float16)(q - (float)hi);
                }
        }
    }
    if (lane == 0) {
#pragma unroll
        for (int k = 0; k < R; k++)
            if (k < count) *xp(k) = sign[k] * ldexpf(1.0f, -s[k]);
    }
}

// One workgroup per (32-token tile, super-block): eight wavefronts of four
// tokens each; the fragments meet in LDS and leave as one contiguous 32 KiB.  row_cols:
// the row's own columns (cols: padded with zeros to a multiple of 64).
template <int FMT>
__global__ void __launch_bounds__(512) k_gm_stage(const float *__restrict__ x, int n, int cols, int row_cols,
                                                  uint8_t *__restrict__ xf, uint8_t *__restrict__ xm,
                                                  float *__restrict__ xp)
{
    __shared__ uint4 frag[4 * GM_UNIT / 16];
    __shared__ uint4 sums[GM_SUMS / 16];
    const int nb = (cols + 255) >> 8, tile = (int)blockIdx.x / nb, sb = (int)blockIdx.x % nb;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const bool in = 256 * sb + 4 * lane < cols; // (a last super-block may be partial: zeros)
    gm_f4 v[4];
#pragma unroll
    for (int k = 0; k < 4; k++) {
        const int t = 32 * tile + 4 * wave + k;
        v[k] = gm_f4{0.f, 0.f, 0.f, 0.f};
        if (in && t < n) v[k] = *(const gm_f4 *)(x + (size_t)t * cols + 256 * sb + 4 * lane);
    }
    gm_stage_rows<FMT, 4, false>(
        v, lane, 4, [&](int k) { return 4 * wave + k; }, [&](int) { return (uint8_t *)frag; },
        [&](int k) { return (uint8_t *)sums + 16 * (4 * wave + k); },
        [&](int k) { return xp + (size_t)blockIdx.x * 32 + 4 * wave + k; }, false, row_cols - 256 * sb);
    __syncthreads();
    uint4 *of = (uint4 *)(xf + (size_t)blockIdx.x * (4 * GM_UNIT));
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const int w = i * 512 + threadIdx.x, pc = (w >> 5) & 15; // unit i, piece pc (step, part, half), token w % 32
        of[w] = frag[w ^ gm_swz(i, pc >> 2, (pc >> 1) & 1)];
    }
    if (FMT == FMT_Q4K && threadIdx.x < 64)
        ((uint4 *)(xm + (size_t)blockIdx.x * GM_SUMS))[threadIdx.x] = sums[threadIdx.x];
}

// The same token by token (rows whose tiles are not known yet): four rows of
// one super-block per wavefront.  F [row][super-block][GM_TOK], M [row][super-
// block][GM_TOK_SUMS], P [row][super-block].
__global__ void __launch_bounds__(256) k_gm_stage_tok(const float *__restrict__ x, int n, int cols,
                                                      uint8_t *__restrict__ xf, uint8_t *__restrict__ xm,
                                                      float *__restrict__ xp)
{
    const int nb = cols >> 8, lane = threadIdx.x & 63;
    const long w = (long)blockIdx.x * 4 + (threadIdx.x >> 6);
    const int sb = (int)(w % nb);
    const long t0 = w / nb * 4;
    if (t0 >= n) return; // no barriers here
    gm_f4 v[4];
#pragma unroll
    for (int k = 0; k < 4; k++) {
        v[k] = gm_f4{0.f, 0.f, 0.f, 0.f};
        if (t0 + k < n) v[k] = *(const gm_f4 *)(x + (size_t)(t0 + k) * cols + 256 * sb + 4 * lane);
    }
    auto at = [&](int k) { return (size_t)(t0 + k) * nb + sb; };
    gm_stage_rows<FMT_Q4K, 4, true>(
        v, lane, (int)min(4l, n - t0), [&](int) { return 0; }, [&](int k) { return xf + at(k) * GM_TOK; },
        [&](int k) { return xm + at(k) * GM_TOK_SUMS; }, [&](int k) { return xp + at(k); });
}

// (typedefs of the compiler's own vectors: a HIP uint4 array that a lambda
// fills ends up in scratch memory)
__device__ __forceinline__ gm_u4 gm_ld(rsrc_t r, uint32_t off)
{
    return __builtin_bit_cast(gm_u4, __builtin_amdgcn_raw_buffer_load_b128(r, (int)off, 0, 0));
}
__device__ __forceinline__ gm_h2 gm_h2_of(uint32_t v) { return __builtin_bit_cast(gm_h2, v); }
__device__ __forceinline__ gm_h2 gm_dup(float v) { return gm_h2{(_Float16)v, (_Float16)v}; }

// Bytes a and b of w as the f16 pair 1024 + byte (0x6400 | byte).
template <int a, int b>
__device__ __forceinline__ gm_h2 gm_bytes(uint32_t w)
{
    return gm_h2_of(__builtin_amdgcn_perm(0x64646464u, w, 0x04000400u | (uint32_t)a | ((uint32_t)b << 16)));
}
// The same byte b (0 .. 3, a constant after unrolling) twice.
__device__ __forceinline__ gm_h2 gm_byte_dup(uint32_t w, int b)
{
    return gm_h2_of(__builtin_amdgcn_perm(0x64646464u, w, 0x04000400u | (uint32_t)b | ((uint32_t)b << 16)));
}

__device__ __forceinline__ gm_h8 gm_join(gm_h2 a, gm_h2 b, gm_h2 c, gm_h2 d)
{
    return gm_h8{a[0], a[1], b[0], b[1], c[0], c[1], d[0], d[1]};
}

// gfx950's swap of a in lanes 32 .. 63 with b in lanes 0 .. 31.
__device__ __forceinline__ void gm_swap32(uint32_t &a, uint32_t &b)
{
    const auto r = __builtin_amdgcn_permlane32_swap(a, b, false, false);
    a = r[0];
    b = r[1];
}
__device__ __forceinline__ void gm_swap32(gm_u4 &a, gm_u4 &b)
{
#pragma unroll
    for (int i = 0; i < 4; i++) {
        uint32_t x = a[i], y = b[i];
        gm_swap32(x, y);
        a[i] = x;
        b[i] = y;
    }
}

// The weights of a wavefront's 64 rows for half a super-block (units 2 i and 2
// i + 1), format by format.  load: lane (n, k = lane / 32) requests, of rows n
// and 32 + n, the 16 bytes of unit k in every plane, so that a row's bytes are
// read 32 at a time; split: lane swaps (a plane or half index against the
// lane's k) hand lane (n, f) what its operand takes of each unit; frag<>: the
// operand of step t of unit v (0 or 1).  head_*: what a row holds once per
// super-block, lane l requesting row l's.  SETS: halves in flight.
template <int FMT, int SETS>
struct GmW;

// A half super-block of Q4_K as the operands take it.
struct GmQ4K {
    static constexpr int PARTS = 1; // operands per step (hi, and lo where a weight needs two f16)
    gm_u4 q[2][2];                  // [rows 32 j][unit]: the 16 code bytes of plane f
    uint32_t sc4[2][2], m4[2][2], dd[2];
    // the scales of a super-block's eight sub-blocks (get_scale_min_k4,
    // dequant.rs:150-159), four per dword
    __device__ __forceinline__ void scales(gm_u4 h, int j)
    {
        dd[j] = h[0];
        sc4[j][0] = h[1] & 0x3F3F3F3Fu;
        m4[j][0] = h[2] & 0x3F3F3F3Fu;
        sc4[j][1] = (h[3] & 0x0F0F0F0Fu) | ((h[1] >> 2) & 0x30303030u);
        m4[j][1] = ((h[3] >> 4) & 0x0F0F0F0Fu) | ((h[2] >> 2) & 0x30303030u);
    }
    // Step t of unit v of half i.  A masked nibble q is the subnormal f16 q
    // 2^-24 (16 q 2^-24 where the high nibbles stay in place) and its product
    // with sc 2^10 (sc 2^6) is q sc 2^-14, exact: a dword costs one shift, four
    // ands and four packed multiplies.
    __device__ __forceinline__ void frag(int i, int v, int t, int j, gm_h8 (&b)[PARTS]) const
    {
        const int sub = 4 * i + 2 * v + (t >> 1);
        const gm_h2 sc = (gm_byte_dup(sc4[j][sub >> 2], sub & 3) - gm_dup(1024.0f)) * gm_dup(t < 2 ? 1024.0f : 64.0f);
        const uint32_t mask = t < 2 ? 0x000F000Fu : 0x00F000F0u;
        const uint32_t w0 = q[j][v][2 * (t & 1)], w1 = q[j][v][2 * (t & 1) + 1];
        b[0] = gm_join(gm_h2_of(w0 & mask) * sc, gm_h2_of((w0 >> 8) & mask) * sc, gm_h2_of(w1 & mask) * sc,
                       gm_h2_of((w1 >> 8) & mask) * sc);
    }
    __device__ __forceinline__ float scale(int j) const { return 16384.0f * half_bits_to_f32(dd[j] & 0xffffu); }
    __device__ __forceinline__ float min_scale(int j) const { return -32.0f * half_bits_to_f32(dd[j] >> 16); }
    __device__ __forceinline__ gm_h8 mins(int j) const
    {
        const gm_h2 k = gm_dup(1024.0f);
        return gm_join(gm_bytes<0, 1>(m4[j][0]) - k, gm_bytes<2, 3>(m4[j][0]) - k, gm_bytes<0, 1>(m4[j][1]) - k,
                       gm_bytes<2, 3>(m4[j][1]) - k);
    }
};

template <int SETS>
struct GmW<FMT_Q4K, SETS> : GmQ4K {
    gm_u4 L[SETS][2][2], hn;
    uint32_t off_h, off_q, row32, plane;
    __device__ __forceinline__ void init(int row, int lane, size_t stride, int U)
    {
        const int nb = U >> 2;
        off_h = (uint32_t)((row + lane) * stride);
        off_q = (uint32_t)((row + (lane & 31)) * stride) + 16u * (uint32_t)(nb + (lane >> 5));
        row32 = (uint32_t)(32 * stride);
        plane = 64u * (uint32_t)nb;
    }
    __device__ __forceinline__ void head_load(rsrc_t rs, int sb) { hn = gm_ld(rs, off_h + 16u * (uint32_t)sb); }
    __device__ __forceinline__ void load(rsrc_t rs, int half, int set)
    {
#pragma unroll
        for (int j = 0; j < 2; j++)
#pragma unroll
            for (int k = 0; k < 2; k++)
                L[set][j][k] = gm_ld(rs, off_q + (uint32_t)j * row32 + (uint32_t)k * plane + 32u * (uint32_t)half);
    }
    __device__ __forceinline__ void head()
    {
        gm_u4 h[2] = {hn, hn};
        gm_swap32(h[0], h[1]);
        scales(h[0], 0);
        scales(h[1], 1);
    }
    __device__ __forceinline__ void split(int, int set)
    {
#pragma unroll
        for (int j = 0; j < 2; j++) {
            q[j][0] = L[set][j][0];
            q[j][1] = L[set][j][1];
            gm_swap32(q[j][0], q[j][1]);
        }
    }
};

template <int SETS>
struct GmW<FMT_Q6K, SETS> {
    static constexpr int PARTS = 2;
    gm_u4 L[SETS][2][3], hn;
    uint32_t dn;
    uint32_t q[2][3][2][2]; // [rows][QH, QLa, QLb][unit][dword]: bytes 8 f .. 8 f + 7
    uint32_t sc4[2][4], dd[2]; // scales + 128
    uint32_t off_h, off_d, off_q, row32, plane;
    __device__ __forceinline__ void init(int row, int lane, size_t stride, int U)
    {
        const int nb = U >> 2;
        off_h = (uint32_t)((row + lane) * stride);
        off_d = off_h + 208u * (uint32_t)nb;
        off_q = (uint32_t)((row + (lane & 31)) * stride) + 16u * (uint32_t)(nb + (lane >> 5));
        row32 = (uint32_t)(32 * stride);
        plane = 64u * (uint32_t)nb;
    }
    __device__ __forceinline__ void head_load(rsrc_t rs, int sb)
    {
        hn = gm_ld(rs, off_h + 16u * (uint32_t)sb);
        dn = bld2(rs, off_d + 2u * (uint32_t)sb);
    }
    __device__ __forceinline__ void load(rsrc_t rs, int half, int set)
    {
#pragma unroll
        for (int j = 0; j < 2; j++)
#pragma unroll
            for (int k = 0; k < 3; k++)
                L[set][j][k] = gm_ld(rs, off_q + (uint32_t)j * row32 + (uint32_t)k * plane + 32u * (uint32_t)half);
    }
    __device__ __forceinline__ void head()
    {
        gm_u4 h[2] = {hn, hn};
        gm_swap32(h[0], h[1]);
        dd[0] = dd[1] = dn;
        gm_swap32(dd[0], dd[1]);
#pragma unroll
        for (int j = 0; j < 2; j++)
#pragma unroll
            for (int k = 0; k < 4; k++) sc4[j][k] = h[j][k] ^ 0x80808080u;
    }
    __device__ __forceinline__ void split(int, int set)
    {
#pragma unroll
        for (int j = 0; j < 2; j++)
#pragma unroll
            for (int k = 0; k < 3; k++)
#pragma unroll
                for (int w = 0; w < 2; w++) {
                    q[j][k][0][w] = L[set][j][k][w];
                    q[j][k][1][w] = L[set][j][k][2 + w];
                    gm_swap32(q[j][k][0][w], q[j][k][1][w]);
                }
    }
    // Step t: quarter t of the half.  sc (q - 32) is a whole number up to
    // 4096: its f16 rounding and the remainder (at most 1) are both exact.
    __device__ __forceinline__ void frag(int i, int v, int t, int j, gm_h8 (&b)[PARTS]) const
    {
        const int s = 8 * i + v + 2 * t;
        const gm_h2 sc = gm_byte_dup(sc4[j][s >> 2], s & 3) - gm_dup(1152.0f);
        gm_h2 hi[4], lo[4];
#pragma unroll
        for (int w = 0; w < 2; w++) {
            const uint32_t l = q[j][1 + (t & 1)][v][w], hq = q[j][0][v][w];
            const uint32_t c = ((t < 2 ? l : l >> 4) & 0x0F0F0F0Fu) |
                               (t == 0 ? (hq << 4) & 0x30303030u
                                : t == 1 ? (hq << 2) & 0x30303030u
                                : t == 2 ? hq & 0x30303030u
                                         : (hq >> 2) & 0x30303030u);
            const gm_h2 a = gm_bytes<0, 2>(c) - gm_dup(1056.0f), d = gm_bytes<1, 3>(c) - gm_dup(1056.0f);
            hi[2 * w] = a * sc;
            hi[2 * w + 1] = d * sc;
            lo[2 * w] = __builtin_elementwise_fma(a, sc, -hi[2 * w]);
            lo[2 * w + 1] = __builtin_elementwise_fma(d, sc, -hi[2 * w + 1]);
        }
        b[0] = gm_join(hi[0], hi[1], hi[2], hi[3]);
        b[1] = gm_join(lo[0], lo[1], lo[2], lo[3]);
    }
    __device__ __forceinline__ float scale(int j) const { return half_bits_to_f32(dd[j] & 0xffffu); }
};

template <int SETS>
struct GmW<FMT_Q80, SETS> {
    static constexpr int PARTS = 1;
    gm_u4 L[SETS][2][4], hs[SETS];
    gm_u4 q[2][2][2]; // [rows][block][unit]: the block's code bytes 16 f .. 16 f + 15
    gm_u4 sc[2];      // the half's four block scales (f32 bits)
    uint32_t off_h, off_q, row32, plane;
    int U;
    __device__ __forceinline__ void init(int row, int lane, size_t stride, int U_)
    {
        U = U_;
        off_h = (uint32_t)((row + lane) * stride);
        off_q = (uint32_t)((row + (lane & 31)) * stride) + ((8u * (uint32_t)U + 15u) & ~15u) + 16u * (uint32_t)(lane >> 5);
        row32 = (uint32_t)(32 * stride);
        plane = 16u * (uint32_t)U;
    }
    __device__ __forceinline__ void head_load(rsrc_t, int) {}
    __device__ __forceinline__ void head() {}
    __device__ __forceinline__ void load(rsrc_t rs, int half, int set)
    {
        hs[set] = gm_ld(rs, off_h + 16u * (uint32_t)half);
#pragma unroll
        for (int j = 0; j < 2; j++)
#pragma unroll
            for (int k = 0; k < 4; k++)
                L[set][j][k] = gm_ld(rs, off_q + (uint32_t)j * row32 + (uint32_t)k * plane + 32u * (uint32_t)half);
    }
    __device__ __forceinline__ void split(int half, int set)
    {
        // Units past the row's end (a partial last super-block) hold whatever
        // follows in memory: zero scales, and x is staged as zeros there.
        gm_u4 h = hs[set];
        if (2 * half + 1 >= U) { // uniform
            h[2] = h[3] = 0u;
            if (2 * half >= U) h[0] = h[1] = 0u;
        }
        sc[0] = sc[1] = h;
        gm_swap32(sc[0], sc[1]);
#pragma unroll
        for (int j = 0; j < 2; j++)
#pragma unroll
            for (int b = 0; b < 2; b++) {
                q[j][b][0] = L[set][j][2 * b];
                q[j][b][1] = L[set][j][2 * b + 1];
                gm_swap32(q[j][b][0], q[j][b][1]);
            }
    }
    __device__ __forceinline__ void frag(int, int v, int t, int j, gm_h8 (&b)[PARTS]) const
    {
        const gm_h2 k = gm_dup(1152.0f);
        const uint32_t w0 = q[j][t >> 1][v][2 * (t & 1)] ^ 0x80808080u;
        const uint32_t w1 = q[j][t >> 1][v][2 * (t & 1) + 1] ^ 0x80808080u;
        b[0] = gm_join(gm_bytes<0, 2>(w0) - k, gm_bytes<1, 3>(w0) - k, gm_bytes<0, 2>(w1) - k, gm_bytes<1, 3>(w1) - k);
    }
    __device__ __forceinline__ float block_scale(int v, int b, int j) const
    {
        return __builtin_bit_cast(float, (uint32_t)sc[j][2 * v + b]);
    }
};

// Weight (row, column c) as the reference dequantizes it (dq_* in
// k_matvec.hip); U units per packed row.
template <int FMT>
__device__ float gm_weight(const uint8_t *__restrict__ row, int c, int U)
{
    const int nb = U >> 2, sb = c >> 8, e = c & 255;
    if constexpr (FMT == FMT_Q4K) {
        const uint8_t *H = row + 16 * sb, *s = H + 4;
        const float d = f16_to_f32_ref(H[0] | (H[1] << 8)), dmin = f16_to_f32_ref(H[2] | (H[3] << 8));
        const int u = 4 * sb + (e >> 6), j = e >> 5, b = e & 31;
        const int q = row[16 * nb + (b < 16 ? 0 : 16 * U) + 16 * u + (b & 15)];
        const int sc = j < 4 ? s[j] & 63 : (s[j + 4] & 15) | ((s[j - 4] >> 6) << 4);
        const int m = j < 4 ? s[j + 4] & 63 : (s[j + 4] >> 4) | ((s[j] >> 6) << 4);
        return __fsub_rn(__fmul_rn(__fmul_rn(d, (float)sc), (float)((e & 32) ? q >> 4 : q & 15)),
                         __fmul_rn(dmin, (float)m));
    } else if constexpr (FMT == FMT_Q80) {
        const int u = c >> 6, b = c & 63;
        const int8_t q = (int8_t)row[((8 * U + 15) & ~15) + 16 * U * (b >> 4) + 16 * u + (b & 15)];
        return __fmul_rn((float)q, ((const float *)row)[c >> 5]);
    } else {
        const int h = e >> 7, t = (e >> 5) & 3, k = (e >> 4) & 1, i = e & 15, u = 4 * sb + 2 * h + k;
        const int l = row[16 * nb + 16 * U * (1 + (t & 1)) + 16 * u + i], hi = row[16 * nb + 16 * u + i];
        const int q = (int)((t < 2 ? l & 15 : l >> 4) | (((hi >> (2 * t)) & 3) << 4)) - 32;
        const uint8_t *D = row + 16 * nb + 48 * U + 2 * sb;
        const int sc = (int8_t)row[16 * sb + 8 * h + k + 2 * t];
        return __fmul_rn(__fmul_rn(f16_to_f32_ref(D[0] | (D[1] << 8)), (float)sc), (float)q);
    }
}

// Of a workgroup's super-blocks and tokens, those whose 2^-s is negative: 64 of
// each in turn, so a set bit may stand for others too.  (Every super-block and token
// of a tile looked at where one had a mark: MoE layers with heavy-tailed activations,
// 16 experts of 1024 x 512 at 72 tokens 122 us against 71, 128 of 2048 x 768 at 512
// tokens 338 against 256.)
struct GmTaken {
    uint64_t blocks = 0, tokens = 0;
    __device__ __forceinline__ void mark(int sb, float p)
    {
        const uint64_t t = __ballot(p < 0.0f);
        tokens |= t;
        blocks |= (uint64_t)(t != 0) << (sb & 63);
    }
    __device__ __forceinline__ bool any() const { return blocks != 0; }
    __device__ __forceinline__ bool block(int sb) const { return (blocks >> (sb & 63)) & 1; }
    __device__ __forceinline__ bool has(int sb, int t) const { return block(sb) && ((tokens >> t) & 1); }
};

// The products of the elements that the staging took out of a tile's tokens 0
// .. nt - 1 (x rows xrow(t)) in super-blocks sb0 .. sb1 - 1, found again by the
// same rule, into the sums of this lane's two weight rows w0 and w1 (null: past
// the matrix).  Token t of the tile is register 4 (t / 8) + t % 4 of half t / 4
// % 2.  taken: which tokens and super-blocks to look at.  Rare: kept out of the
// streaming loop.
template <int FMT, class XRow>
__device__ __forceinline__ void gm_add_outliers(gm_f16v (&acc)[2], const uint8_t *w0, const uint8_t *w1, int cols,
                                                XRow xrow, int nt, int sb0, int sb1, const GmTaken &taken, int m)
{
    const int lane = threadIdx.x & 63;
    for (int sb = sb0; sb < sb1; sb++)
        for (int t = 0; t < nt; t++) {
            if (!taken.has(sb - sb0, 32 * m + t)) continue; // uniform
            gm_f4 v = {0.f, 0.f, 0.f, 0.f};
            if (256 * sb + 4 * lane < cols) v = *(const gm_f4 *)(xrow(t) + 256 * sb + 4 * lane);
            const float sm = (v[0] + v[1]) + (v[2] + v[3]);
            if (__ballot(!(gm_abs_max(v) < INFINITY) || sm != sm)) continue; // non-finite: every output is NaN already
            float ref;
            const float thr = gm_outlier_thr(v, ref);
            const bool mine = ((t >> 2) & 1) == lane >> 5;
#pragma unroll
            for (int i = 0; i < 4; i++) {
                uint64_t todo = __ballot(fabsf(v[i]) > thr);
                while (todo) { // uniform
                    const int src = __builtin_ctzll(todo), c = 256 * sb + 4 * src + i;
                    todo &= todo - 1;
                    const float xv = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v[i]), src));
#pragma unroll
                    for (int j = 0; j < 2; j++) {
                        const uint8_t *w = j ? w1 : w0;
                        const float p = mine && w ? gm_weight<FMT>(w, c, cols >> 6) * xv : 0.0f;
#pragma unroll
                        for (int k = 0; k < 16; k++)
                            if (k == 4 * (t >> 3) + (t & 3)) acc[j][k] += p;
                    }
                }
            }
        }
}

// acc += 2^-s (d S - 32 dmin M), Q6_K and Q8_0 without M (and Q8_0's scales, d,
// are in S already): a super-block's sums S of the 32 tokens whose 2^-s is at p;
// am: their sub-blocks' sums (Q4_K), wt: the weights after head().
template <int FMT, class W>
__device__ __forceinline__ void gm_fold(gm_f16v (&acc)[2], const gm_f16v (&S)[2], const W &wt, const float *p, int f,
                                        gm_h8 am)
{
    float pt[16]; // 2^-s of this lane's tokens
#pragma unroll
    for (int k = 0; k < 4; k++) {
        const gm_f4 v = *(const gm_f4 *)(p + 8 * k + 4 * f);
#pragma unroll
        for (int i = 0; i < 4; i++) pt[4 * k + i] = v[i];
    }
    const gm_f16v zero = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int j = 0; j < 2; j++) {
        if constexpr (FMT == FMT_Q4K) {
            const float d = wt.scale(j), dm = wt.min_scale(j);
            const gm_f16v M = __builtin_amdgcn_mfma_f32_32x32x16_f16(am, wt.mins(j), zero, 0, 0, 0);
#pragma unroll
            for (int i = 0; i < 16; i++) acc[j][i] = fmaf(fabsf(pt[i]), fmaf(d, S[j][i], dm * M[i]), acc[j][i]);
        } else if constexpr (FMT == FMT_Q6K) {
            const float d = wt.scale(j);
#pragma unroll
            for (int i = 0; i < 16; i++) acc[j][i] = fmaf(fabsf(pt[i]), d * S[j][i], acc[j][i]);
        } else {
#pragma unroll
            for (int i = 0; i < 16; i++) acc[j][i] = fmaf(fabsf(pt[i]), S[j][i], acc[j][i]);
        }
    }
}

// The larger halves that the staging left out of a tile's super-blocks sb0 .. sb1
// - 1, found again by the same rule: staged by themselves and multiplied as the
// rest were.  Rare, so without prefetching; the workgroup's four wavefronts call it
// together.  head(sb), half(sb, i): load a super-block's, a half's weights into wt;
// xf (four units), xm, xp: LDS of a staged tile.  With every other half of x 1e6
// times its neighbour, 14336 x 4096 in Q4_K takes 111 us per call at 8 tokens and
// 370 at 128, ordinary x 31 and 64 (by gm_add_outliers 2849 and 30415).  A scale
// per half, folded in mid-block, took 44 and 72, but its registers cost k_gemm_few
// 5 to 47 % on ordinary x, a second pass of k_gemm_few 10 to 20 %.
template <int FMT, class W, class XRow, class Head, class Half>
__device__ __forceinline__ void gm_add_halves(gm_f16v (&acc)[2], W &wt, int cols, XRow xrow, int nt, int sb0, int sb1,
                                              const GmTaken &taken, Head head, Half half, uint8_t *xf, uint8_t *xm,
                                              float *xp)
{
    const int lane = threadIdx.x & 63, f = lane >> 5, wave = threadIdx.x >> 6;
    constexpr int PARTS = W::PARTS;
    const gm_f16v zero = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll 1
    for (int sb = sb0; sb < sb1; sb++) {
        if (!taken.block(sb - sb0)) continue; // uniform over the workgroup
        __syncthreads(); // the last tile's readers are done
#pragma unroll 1
        for (int t0 = wave; t0 < 32; t0 += 16) { // tokens t0 + 4 k; past nt zeros
            gm_f4 v[4];
#pragma unroll
            for (int k = 0; k < 4; k++) {
                v[k] = gm_f4{0.f, 0.f, 0.f, 0.f};
                if (t0 + 4 * k < nt && 256 * sb + 4 * lane < cols)
                    v[k] = *(const gm_f4 *)(xrow(t0 + 4 * k) + 256 * sb + 4 * lane);
            }
            gm_stage_rows<FMT, 4, false>(
                v, lane, 4, [&](int k) { return t0 + 4 * k; }, [&](int) { return xf; },
                [&](int k) { return xm + 16 * (t0 + 4 * k); }, [&](int k) { return xp + t0 + 4 * k; }, true);
        }
        __syncthreads();
        if (__ballot(xp[lane & 31] < 0.0f) == 0) continue; // uniform over the workgroup
        head(sb);
        gm_f16v S[2] = {zero, zero}, T[2] = {zero, zero}; // T: Q8_0, its scales applied
#pragma unroll
        for (int p = 0; p < 4; p++) {
            if (!(p & 1)) half(sb, p >> 1);
#pragma unroll
            for (int t = 0; t < 4; t++) {
                __builtin_amdgcn_sched_barrier(0); // (no loads ahead: the registers are the kernels')
                const gm_h8 hi = gm_frag_at(xf + p * GM_UNIT, lane, p, t, 0), lo = gm_frag_at(xf + p * GM_UNIT, lane, p, t, 1);
#pragma unroll
                for (int j = 0; j < 2; j++) {
                    gm_h8 b[PARTS];
                    wt.frag(p >> 1, p & 1, t, j, b);
                    S[j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(lo, b[0], S[j], 0, 0, 0);
                    if constexpr (PARTS == 2) S[j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(hi, b[1], S[j], 0, 0, 0);
                    S[j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(hi, b[0], S[j], 0, 0, 0);
                    if constexpr (FMT == FMT_Q80) {
                        if (t & 1) {
                            T[j] += wt.block_scale(p & 1, t >> 1, j) * S[j];
                            S[j] = zero;
                        }
                    }
                }
            }
        }
        gm_fold<FMT>(acc, FMT == FMT_Q80 ? T : S, wt, xp, f, *(const gm_h8 *)(xm + (FMT == FMT_Q4K ? 16 * lane : 0)));
    }
    __syncthreads();
}

// A workgroup of four wavefronts owns 256 rows (64 per wavefront, two 32-row
// tiles) and MT tiles of 32 tokens, over the super-blocks of its split.  A
// wavefront dequantizes its own rows' operands in registers, once for all its
// tokens; x comes through LDS, a unit ahead, and each 1 KiB fragment read there
// feeds two products.  Bound by the matrix cores (two products per weight and
// token, three for Q6_K) and the dequantization beside them.  Measured on
// MI355X (us, before -> here; TFLOP/s of the product): Q4_K 14336 x 4096 at 512
// tokens 319 -> 138 (436), 4096 x 14336 at 199 228 -> 80 (292); Q6_K 4096 x
// 14336 at 256 3271 -> 106 (284, vector by vector before); Q8_0 4096 x 4096 at
// 512 187 -> 78 (220).  With the weight loads' 32-byte pieces read from one
// place instead 124 us at 14336 x 4096 x 512; codes loaded by one lane each (16
// bytes per row and load) took 213, x's next unit requested where the scheduler
// put it 204.  A whole super-block's codes in flight measured the same.
template <int FMT, int MT>
__global__ void __launch_bounds__(256, 2) k_gemm(const uint8_t *__restrict__ W, size_t stride, int rows, int cols,
                                                 GmX x, const float *__restrict__ xs32, int n, int ntt, int nsplit,
                                                 int items, float *__restrict__ out)
{
    // consecutive items share their rows (the token tiles of a row block) and
    // stay on one XCD (workgroups go round the eight in turn), so a row
    // block's weights come out of HBM once per XCD that holds it
    const int per = (items + 7) / 8, w = ((int)blockIdx.x & 7) * per + ((int)blockIdx.x >> 3);
    if (w >= items || ((int)blockIdx.x >> 3) >= per) return;
    const int tt = w % ntt, sp = w / ntt % nsplit, rb = w / (ntt * nsplit);
    const int lane = threadIdx.x & 63, f = lane >> 5, nl = lane & 31;
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int nb = (cols + 255) >> 8, U = 4 * nb; // staged super-blocks and units
    const int sb0 = (int)((long)nb * sp / nsplit), sb1 = (int)((long)nb * (sp + 1) / nsplit);
    const int r0 = 256 * rb, rend = min(rows, r0 + 256);
    const rsrc_t rs = make_rsrc(W + (size_t)r0 * stride, (uint32_t)((size_t)(rend - r0) * stride));
    constexpr int XW = 2 * MT; // 16-byte words of a unit's x per thread
    __shared__ gm_u4 xs[2][(MT > 2 ? MT : 2) * GM_UNIT / 16]; // (four units for gm_add_halves)
    __shared__ float ps[2][MT * 32];
    __shared__ gm_u4 ms[FMT == FMT_Q4K ? GM_SUMS / 16 : 1]; // (gm_add_halves)
    // this workgroup's token tiles, MT * U units
    const rsrc_t rx = make_rsrc(x.f + (size_t)tt * MT * U * GM_UNIT, (uint32_t)((size_t)MT * U * GM_UNIT));
    const float *xp = x.p + ((size_t)(tt * MT + (int)(threadIdx.x >> 5)) * nb) * 32 + (threadIdx.x & 31);
    GmW<FMT, 1> wt;
    wt.init(64 * wave, lane, stride, cols >> 6);
    constexpr int PARTS = GmW<FMT, 1>::PARTS;

    gm_f16v acc[MT][2], S[MT][2];
    const gm_f16v zero = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int m = 0; m < MT; m++)
#pragma unroll
        for (int j = 0; j < 2; j++) acc[m][j] = zero;
    gm_u4 xr[XW];
    auto load_x = [&](int u) {
#pragma unroll
        for (int k = 0; k < XW; k++)
            xr[k] = __builtin_bit_cast(gm_u4, __builtin_amdgcn_raw_buffer_load_b128(
                                                  rx, 16 * (int)threadIdx.x,
                                                  ((k >> 1) * U + u) * GM_UNIT + 4096 * (k & 1), 0));
    };
    auto store_x = [&](int b) {
#pragma unroll
        for (int k = 0; k < XW; k++) xs[b][(k >> 1) * (GM_UNIT / 16) + 256 * (k & 1) + threadIdx.x] = xr[k];
    };
    // Q8_0: the super-block's sums, each block's scale applied
    gm_f16v T[FMT == FMT_Q80 ? MT : 1][2];
    GmTaken taken;
    load_x(4 * sb0);
    wt.head_load(rs, sb0);
    wt.load(rs, 2 * sb0, 0);
    store_x(0);
    __syncthreads();
    for (int sb = sb0; sb < sb1; sb++) {
        wt.head();
        gm_h8 am[MT] = {};
        float pv = 0.0f;
#pragma unroll
        for (int p = 0; p < 4; p++) {
            const int u = 4 * sb + p;
            if (!(p & 1)) wt.split(2 * sb + (p >> 1), 0);
            // in flight during this unit's products: the next unit's x (the
            // last unit's once more at the end) and, every other unit, the next
            // half super-block's weights
            load_x(min(u + 1, 4 * sb1 - 1));
            if (p == 1) wt.load(rs, 2 * sb + 1, 0);
            if (p == 3) {
                const int sn = min(sb + 1, sb1 - 1);
                wt.load(rs, 2 * sn, 0);
                wt.head_load(rs, sn);
                if (FMT == FMT_Q4K) {
#pragma unroll
                    for (int m = 0; m < MT; m++)
                        am[m] = *(const gm_h8 *)(x.m + ((size_t)(tt * MT + m) * nb + sb) * GM_SUMS + 16 * lane);
                }
                if ((int)threadIdx.x < MT * 32) pv = xp[(size_t)sb * 32];
            }
            __builtin_amdgcn_sched_barrier(0); // (the scheduler would sink the loads to their use)
            const uint8_t *xb = (const uint8_t *)xs[p & 1] + 16 * lane;
            // step i = t * MT + m: the next step's x (and codes) are fetched
            // while this one's products run
            gm_h8 ah[2], al[2], b[2][2][PARTS];
            ah[0] = *(const gm_h8 *)xb;
            al[0] = *(const gm_h8 *)(xb + 1024);
#pragma unroll
            for (int j = 0; j < 2; j++) wt.frag(p >> 1, p & 1, 0, j, b[0][j]);
#pragma unroll
            for (int i = 0; i < 4 * MT; i++) {
                const int t = i / MT, m = i % MT, t1 = (i + 1) / MT, m1 = (i + 1) % MT;
                if (i + 1 < 4 * MT) {
                    ah[(i + 1) & 1] = *(const gm_h8 *)(xb + m1 * GM_UNIT + t1 * 2048);
                    al[(i + 1) & 1] = *(const gm_h8 *)(xb + m1 * GM_UNIT + t1 * 2048 + 1024);
                    if (m == MT - 1) {
#pragma unroll
                        for (int j = 0; j < 2; j++) wt.frag(p >> 1, p & 1, t1, j, b[t1 & 1][j]);
                    }
                }
                const gm_h8 hi = ah[i & 1], lo = al[i & 1];
                // the sums start at the super-block's (Q8_0: the block's) first step
                const bool first = FMT == FMT_Q80 ? !(t & 1) : p == 0 && t == 0;
#pragma unroll
                for (int j = 0; j < 2; j++)
                    S[m][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(lo, b[t & 1][j][0], first ? zero : S[m][j], 0, 0, 0);
                if constexpr (PARTS == 2) {
#pragma unroll
                    for (int j = 0; j < 2; j++)
                        S[m][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(hi, b[t & 1][j][PARTS - 1], S[m][j], 0, 0, 0);
                }
#pragma unroll
                for (int j = 0; j < 2; j++)
                    S[m][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(hi, b[t & 1][j][0], S[m][j], 0, 0, 0);
                if constexpr (FMT == FMT_Q80) {
                    if (t & 1) {
#pragma unroll
                        for (int j = 0; j < 2; j++) {
                            const float s = wt.block_scale(p & 1, t >> 1, j);
#pragma unroll
                            for (int e = 0; e < 16; e++)
                                T[m][j][e] = p == 0 && t == 1 ? s * S[m][j][e] : fmaf(s, S[m][j][e], T[m][j][e]);
                            // (keeps the scaling here: sunk to the super-block's
                            // end, it would hold every block's sums until then)
                            asm volatile("" : "+v"(T[m][j]));
                        }
                    }
                }
            }
            store_x((p + 1) & 1);
            if (p == 3 && (int)threadIdx.x < MT * 32) ps[sb & 1][threadIdx.x] = pv;
            __syncthreads();
        }
        taken.mark(sb - sb0, ps[sb & 1][lane & (32 * MT - 1)]);
#pragma unroll
        for (int m = 0; m < MT; m++)
            gm_fold<FMT>(acc[m], *(FMT == FMT_Q80 ? &T[FMT == FMT_Q80 ? m : 0] : &S[m]), wt, ps[sb & 1] + 32 * m, f, am[m]);
    }
    if (__builtin_expect(taken.any(), 0)) {
#pragma unroll
        for (int m = 0; m < MT; m++) {
            const int t0 = 32 * (tt * MT + m), r = r0 + 64 * wave + nl;
            gm_add_outliers<FMT>(
                acc[m], r < rows ? W + (size_t)r * stride : nullptr, r + 32 < rows ? W + (size_t)(r + 32) * stride : nullptr,
                cols, [&](int t) { return xs32 + (size_t)(t0 + t) * cols; }, min(32, n - t0), sb0, sb1, taken, m);
            gm_add_halves<FMT>(
                acc[m], wt, cols, [&](int t) { return xs32 + (size_t)(t0 + t) * cols; }, min(32, n - t0), sb0, sb1, taken,
                [&](int sb) { wt.head_load(rs, sb), wt.head(); },
                [&](int sb, int i) { wt.load(rs, 2 * sb + i, 0), wt.split(2 * sb + i, 0); }, (uint8_t *)xs, (uint8_t *)ms,
                ps[0]);
        }
    }
    float *o = out + (size_t)sp * n * rows;
#pragma unroll
    for (int m = 0; m < MT; m++)
#pragma unroll
        for (int j = 0; j < 2; j++) {
            const int row = r0 + 64 * wave + 32 * j + nl;
#pragma unroll
            for (int i = 0; i < 16; i++) {
                const int t = 32 * (tt * MT + m) + 8 * (i >> 2) + 4 * f + (i & 3);
                if (t < n && row < rows) o[(size_t)t * rows + row] = acc[m][j][i];
            }
        }
}

// The same for few tokens: one tile of 32, x converted by every workgroup
// itself (a conversion launch took longer than it saved: 14336 x 4096 at 2 / 8 /
// 16 tokens 24.8 / 24.9 / 25.5 us with one, 18.6 / 20.7 / 22.9 without) a
// super-block ahead of its products, one barrier per super-block and a whole
// super-block of weights in flight.
template <int FMT>
__global__ void __launch_bounds__(256, 2) k_gemm_few(const uint8_t *__restrict__ W, size_t stride, int rows, int cols,
                                                     const float *__restrict__ x, int n_all, int ntt, int nsplit, int items,
                                                     float *__restrict__ out)
{
    const int per = (items + 7) / 8, w = ((int)blockIdx.x & 7) * per + ((int)blockIdx.x >> 3);
    if (w >= items) return;
    const int tt = w % ntt, sp = w / ntt % nsplit, rb = w / (ntt * nsplit);
    const int n = min(32, n_all - 32 * tt); // this tile's tokens
    x += (size_t)32 * tt * cols;
    const int lane = threadIdx.x & 63, f = lane >> 5, nl = lane & 31;
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int nb = (cols + 255) >> 8;
    const int sb0 = (int)((long)nb * sp / nsplit), sb1 = (int)((long)nb * (sp + 1) / nsplit);
    const int r0 = 256 * rb, rend = min(rows, r0 + 256);
    const rsrc_t rs = make_rsrc(W + (size_t)r0 * stride, (uint32_t)((size_t)(rend - r0) * stride));
    GmW<FMT, 2> wt;
    wt.init(64 * wave, lane, stride, cols >> 6);
    constexpr int PARTS = GmW<FMT, 2>::PARTS;
    wt.head_load(rs, sb0);
    wt.load(rs, 2 * sb0, 0);
    wt.load(rs, 2 * sb0 + 1, 1);
    // the staged tile's four units, sums and 2^-s, double-buffered
    constexpr int SUMS = FMT == FMT_Q4K ? GM_SUMS : 16;
    __shared__ gm_u4 xs[2][4 * GM_UNIT / 16];
    __shared__ gm_u4 ms[2][SUMS / 16];
    __shared__ float ps[2][32];
    // tokens wave + 4 k, k = 4 g + i: a lane's four columns of each
    gm_f4 xv[2][4];
    const int tmax = (n - wave + 3) >> 2; // this wavefront's tokens
    auto load_x = [&](int sb) {
        const bool in = 256 * sb + 4 * lane < cols;
#pragma unroll
        for (int k = 0; k < 8; k++) {
            xv[k >> 2][k & 3] = gm_f4{0.f, 0.f, 0.f, 0.f};
            if (k < tmax && in)
                xv[k >> 2][k & 3] = *(const gm_f4 *)(x + (size_t)(wave + 4 * k) * cols + 256 * sb + 4 * lane);
        }
    };
    auto store_x = [&](int b) {
#pragma unroll
        for (int g = 0; g < 2; g++)
            if (4 * g < tmax) // uniform
                gm_stage_rows<FMT, 4, false>(
                    xv[g], lane, tmax - 4 * g, [&](int k) { return wave + 16 * g + 4 * k; },
                    [&](int) { return (uint8_t *)xs[b]; },
                    [&](int k) { return (uint8_t *)ms[b] + 16 * (wave + 16 * g + 4 * k); },
                    [&](int k) { return &ps[b][wave + 16 * g + 4 * k]; });
    };
    load_x(sb0);
    __builtin_amdgcn_sched_barrier(0);
    // (the products' rows of tokens past n are never stored, whatever their x; their
    // 2^-s must not be a mark)
    if (threadIdx.x < 64 && ((int)threadIdx.x & 31) >= n) (&ps[0][0])[threadIdx.x] = 0.0f;
    store_x(0);
    load_x(min(sb0 + 1, sb1 - 1));
    __syncthreads();
    gm_f16v acc[2], S[2];
    const gm_f16v zero = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    acc[0] = acc[1] = zero;
    GmTaken taken;
    for (int sb = sb0; sb < sb1; sb++) {
        const int cur = (sb - sb0) & 1, sn = min(sb + 1, sb1 - 1);
        wt.head();
        wt.head_load(rs, sn);
        // a step's x is read from LDS a step ahead, where the registers hold it
        constexpr bool AHEAD = FMT == FMT_Q4K;
        const uint8_t *xb = (const uint8_t *)xs[cur];
        gm_h8 ah[2], al[2];
        ah[0] = gm_frag_at(xb, lane, 0, 0, 0);
        al[0] = gm_frag_at(xb, lane, 0, 0, 1);
#pragma unroll
        for (int p = 0; p < 4; p++) {
            if (!(p & 1)) {
                wt.split(2 * sb + (p >> 1), p >> 1);
                wt.load(rs, 2 * sn + (p >> 1), p >> 1);
                __builtin_amdgcn_sched_barrier(0);
            }
#pragma unroll
            for (int t = 0; t < 4; t++) {
                // (Q6_K: the 16 addresses anew, not kept in registers that would spill)
                int ln = lane;
                if (FMT == FMT_Q6K) asm volatile("" : "+v"(ln));
                const int i1 = 4 * p + t + (AHEAD ? 1 : 0);
                if (i1 < 16) {
                    ah[i1 & 1] = gm_frag_at(xb + (i1 >> 2) * GM_UNIT, ln, i1 >> 2, i1 & 3, 0);
                    al[i1 & 1] = gm_frag_at(xb + (i1 >> 2) * GM_UNIT, ln, i1 >> 2, i1 & 3, 1);
                }
                gm_h8 b[2][PARTS];
#pragma unroll
                for (int j = 0; j < 2; j++) wt.frag(p >> 1, p & 1, t, j, b[j]);
                const gm_h8 hi = ah[t & 1], lo = al[t & 1];
                const bool first = p == 0 && t == 0;
#pragma unroll
                for (int j = 0; j < 2; j++)
                    S[j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(lo, b[j][0], first ? zero : S[j], 0, 0, 0);
                if constexpr (PARTS == 2) {
#pragma unroll
                    for (int j = 0; j < 2; j++)
                        S[j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(hi, b[j][PARTS - 1], S[j], 0, 0, 0);
                }
#pragma unroll
                for (int j = 0; j < 2; j++)
                    S[j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(hi, b[j][0], S[j], 0, 0, 0);
            }
        }
        taken.mark(sb - sb0, ps[cur][lane & 31]);
        gm_fold<FMT>(acc, S, wt, ps[cur], f, *(const gm_h8 *)((const uint8_t *)ms[cur] + (FMT == FMT_Q4K ? 16 * lane : 0)));
        if (sb + 1 < sb1) { // uniform
            store_x(cur ^ 1);
            load_x(min(sb + 2, sb1 - 1));
            __syncthreads();
        }
    }
    if (__builtin_expect(taken.any(), 0)) {
        gm_add_halves<FMT>(
            acc, wt, cols, [&](int t) { return x + (size_t)t * cols; }, n, sb0, sb1, taken,
            [&](int sb) { wt.head_load(rs, sb), wt.head(); },
            [&](int sb, int i) { wt.load(rs, 2 * sb + i, i), wt.split(2 * sb + i, i); }, (uint8_t *)xs[0],
            (uint8_t *)ms[0], ps[0]);
        const int r = r0 + 64 * wave + nl;
        gm_add_outliers<FMT>(
            acc, r < rows ? W + (size_t)r * stride : nullptr, r + 32 < rows ? W + (size_t)(r + 32) * stride : nullptr,
            cols, [&](int t) { return x + (size_t)t * cols; }, n, sb0, sb1, taken, 0);
    }
    float *o = out + ((size_t)sp * n_all + 32 * tt) * rows;
#pragma unroll
    for (int j = 0; j < 2; j++) {
        const int row = r0 + 64 * wave + 32 * j + nl;
#pragma unroll
        for (int i = 0; i < 16; i++) {
            const int t = 8 * (i >> 2) + 4 * f + (i & 3);
            if (t < n && row < rows) o[(size_t)t * rows + row] = acc[j][i];
        }
    }
}

// Tile-major Q4_K (the registered MoE experts' copies, tile_q4k in k_mfma.hip:
// per 16-row tile and super-block the rows' headers, then lane 16 g + n's 8 code
// bytes 8 g of row n of units 0 and 1, then of 2 and 3).  Lane (n, f) of a
// 32-row tile takes k-groups 2 f and 2 f + 1 of its row: contiguous loads, no
// swaps.  base: the wavefront's first row of both 32-row tiles.
template <int SETS>
struct GmTiled : GmQ4K {
    gm_u4 L[SETS][2][2], hn[2];
    uint32_t off[2], sbs;
    __device__ __forceinline__ void init(int row0, int row1, int lane, int nb)
    {
        const uint32_t nl = (uint32_t)(lane & 31);
        sbs = 2304u;
        off[0] = ((uint32_t)(row0 >> 4) + (nl >> 4)) * (uint32_t)nb * sbs + 16u * (nl & 15);
        off[1] = ((uint32_t)(row1 >> 4) + (nl >> 4)) * (uint32_t)nb * sbs + 16u * (nl & 15);
        g = 512u * (uint32_t)(lane >> 5) + 256u;
    }
    uint32_t g;
    __device__ __forceinline__ void head_load(const rsrc_t (&rs)[2], int sb)
    {
#pragma unroll
        for (int j = 0; j < 2; j++) hn[j] = gm_ld(rs[j], off[j] + sbs * (uint32_t)sb);
    }
    __device__ __forceinline__ void load(const rsrc_t (&rs)[2], int half, int set)
    {
#pragma unroll
        for (int j = 0; j < 2; j++)
#pragma unroll
            for (int k = 0; k < 2; k++)
                L[set][j][k] = gm_ld(rs[j], off[j] + g + sbs * (uint32_t)(half >> 1) + 1024u * (uint32_t)(half & 1) +
                                                256u * (uint32_t)k);
    }
    __device__ __forceinline__ void head()
    {
        scales(hn[0], 0);
        scales(hn[1], 1);
    }
    __device__ __forceinline__ void split(int set)
    {
#pragma unroll
        for (int j = 0; j < 2; j++) {
            const gm_u4 a = L[set][j][0], b = L[set][j][1];
            q[j][0] = gm_u4{a[0], a[1], b[0], b[1]};
            q[j][1] = gm_u4{a[2], a[3], b[2], b[3]};
        }
    }
};

// The MoE experts of a prompt's tokens (gate / up 303 -> 98 us, down 118 -> 63
// for 512 tokens of 128 experts of 2048 x 768 at top-8, 0.22 and 0.17 PFLOP/s;
// the integer kernel's workgroups converted eight tokens at a time and decoded
// each weight once per eight): k_gemm_few over (tile of 32 slots of an
// active expert, row block), x gathered by the slot list (x row = slot / xdiv,
// output row = slot).  NMAT 2: 128 rows of gate and of up side by side, the
// output silu(gate) * up (gemm.rs:210-226); NMAT 1: 256 rows of down.
// recs[4 a ..] = {expert, slots, first slot in list, 0}, at most 256 of them;
// tab*: tile-major experts, row*: the same row-major (for the outliers).
// STAGED: x's rows come in f16 parts (k_gm_stage_tok); else every workgroup
// converts its tokens, to the same bits.
template <int NMAT, bool STAGED>
__global__ void __launch_bounds__(256, 2)
    k_gemm_moe(const uint8_t *const *__restrict__ tabA, const uint8_t *const *__restrict__ tabB,
               const uint8_t *const *__restrict__ rowA, const uint8_t *const *__restrict__ rowB, size_t stride, int rows,
               int cols, const float *__restrict__ xs, GmX xg, int xdiv, const int *__restrict__ list,
               const int *__restrict__ recs, const int *__restrict__ n_recs, int nblk, float *__restrict__ out)
{
    __shared__ int it_s[4];
    __shared__ int slot_s[32];
    const int lane = threadIdx.x & 63, f = lane >> 5, nl = lane & 31;
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int item = (int)blockIdx.x / nblk, rb = (int)blockIdx.x % nblk;
    if (wave == 0) {
        // the record whose tiles hold this item: a scan over the records'
        // tile counts, four per lane
        const int nr = *n_recs;
        int c[4], tot = 0;
#pragma unroll
        for (int k = 0; k < 4; k++) {
            c[k] = 4 * lane + k < nr ? recs[4 * (4 * lane + k) + 1] : 0;
            tot += (c[k] + 31) >> 5;
        }
        int incl = tot;
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
            const int y = __shfl_up(incl, o, 64);
            if (lane >= o) incl += y;
        }
        if (lane == 63 && item >= incl) it_s[0] = -1;
        int run = incl - tot;
#pragma unroll
        for (int k = 0; k < 4; k++) {
            const int t = (c[k] + 31) >> 5;
            if (item >= run && item < run + t) {
                it_s[0] = recs[4 * (4 * lane + k)];
                it_s[1] = c[k] - 32 * (item - run);
                it_s[2] = recs[4 * (4 * lane + k) + 2] + 32 * (item - run);
            }
            run += t;
        }
    }
    __syncthreads();
    const int e = __builtin_amdgcn_readfirstlane(it_s[0]);
    if (e < 0) return; // uniform: fewer tiles than the grid allows
    const int n = min(32, __builtin_amdgcn_readfirstlane(it_s[1])), first = __builtin_amdgcn_readfirstlane(it_s[2]);
    constexpr int ROWS = NMAT == 2 ? 128 : 256, WROWS = ROWS / 4;
    const int nb = cols >> 8, r0 = ROWS * rb, rend = min(rows, r0 + ROWS);
    const uint32_t strip = (uint32_t)((size_t)(rend - r0) * stride);
    const rsrc_t rs[2] = {make_rsrc(tabA[e] + (size_t)r0 * stride, strip),
                          make_rsrc((NMAT == 2 ? tabB : tabA)[e] + (size_t)r0 * stride, strip)};
    GmTiled<2> wt;
    wt.init(WROWS * wave, WROWS * wave + (NMAT == 2 ? 0 : 32), lane, nb);
    wt.head_load(rs, 0);
    wt.load(rs, 0, 0);
    wt.load(rs, 1, 1);
    __shared__ gm_u4 xb_s[2][4 * GM_UNIT / 16];
    __shared__ gm_u4 ms[2][GM_SUMS / 16];
    __shared__ float ps[2][32];
    if ((int)threadIdx.x < n) slot_s[threadIdx.x] = list[first + threadIdx.x];
    if constexpr (!STAGED) { // (as in k_gemm_few)
        if (threadIdx.x < 64 && ((int)threadIdx.x & 31) >= n) (&ps[0][0])[threadIdx.x] = 0.0f;
    }
    __syncthreads();
    // STAGED: thread (token m, i): pieces 2 i and 2 i + 1 (of 16) of every unit;
    // a token's 256 bytes of a unit are read by eight lanes
    const int xm = (int)threadIdx.x >> 3, xi = (int)threadIdx.x & 7;
    const size_t xtok = STAGED ? (size_t)(slot_s[min(xm, n - 1)] / xdiv) * nb : 0;
    const size_t mtok = STAGED ? (size_t)(slot_s[min(nl, n - 1)] / xdiv) * nb : 0; // threads 0 .. 63: sums and 2^-s
    gm_u4 xr[8], mr;
    float pr = 0.0f;
    // else: tokens wave + 4 k, k = 4 g + i
    gm_f4 xv[2][4];
    const int tmax = (n - wave + 3) >> 2; // this wavefront's tokens
    const float *xrow[8];
    if constexpr (!STAGED) {
#pragma unroll
        for (int k = 0; k < 8; k++)
            xrow[k] = xs + (size_t)(__builtin_amdgcn_readfirstlane(slot_s[min(wave + 4 * k, n - 1)]) / xdiv) * cols;
    }
    auto load_x = [&](int sb) {
        if constexpr (STAGED) {
#pragma unroll
            for (int k = 0; k < 8; k++) {
                xr[k] = gm_u4{0u, 0u, 0u, 0u};
                if (xm < n) xr[k] = *(const gm_u4 *)(xg.f + (xtok + sb) * GM_TOK + 256 * (k >> 1) + 32 * xi + 16 * (k & 1));
            }
            mr = gm_u4{0u, 0u, 0u, 0u};
            pr = 0.0f;
            if (wave == 0 && nl < n) {
                mr = *(const gm_u4 *)(xg.m + (mtok + sb) * GM_TOK_SUMS + 16 * f);
                pr = xg.p[mtok + sb];
            }
        } else {
#pragma unroll
            for (int k = 0; k < 8; k++) {
                xv[k >> 2][k & 3] = gm_f4{0.f, 0.f, 0.f, 0.f};
                if (k < tmax) xv[k >> 2][k & 3] = *(const gm_f4 *)(xrow[k] + 256 * sb + 4 * lane);
            }
        }
    };
    auto store_x = [&](int b) {
        if constexpr (STAGED) {
#pragma unroll
            for (int k = 0; k < 8; k++) // unit k / 2's piece 2 xi + k % 2: step xi / 2, part xi % 2, half k % 2
                xb_s[b][(k >> 1) * (GM_UNIT / 16) + 32 * (2 * xi + (k & 1)) + (xm ^ gm_swz(k >> 1, xi >> 1, xi & 1))] =
                    xr[k];
            if (wave == 0) {
                ms[b][lane] = mr;
                if (f == 0) ps[b][nl] = pr;
            }
        } else {
#pragma unroll
            for (int g = 0; g < 2; g++)
                if (4 * g < tmax) // uniform
                    gm_stage_rows<FMT_Q4K, 4, false>(
                        xv[g], lane, tmax - 4 * g, [&](int k) { return wave + 16 * g + 4 * k; },
                        [&](int) { return (uint8_t *)xb_s[b]; },
                        [&](int k) { return (uint8_t *)ms[b] + 16 * (wave + 16 * g + 4 * k); },
                        [&](int k) { return &ps[b][wave + 16 * g + 4 * k]; });
        }
    };
    load_x(0);
    store_x(0);
    load_x(min(1, nb - 1));
    __syncthreads();
    gm_f16v acc[2], S[2];
    const gm_f16v zero = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    acc[0] = acc[1] = zero;
    GmTaken taken;
    for (int sb = 0; sb < nb; sb++) {
        const int cur = sb & 1, sn = min(sb + 1, nb - 1);
        wt.head();
        wt.head_load(rs, sn);
        // a step's x is read from LDS a step ahead, where the registers hold it
        constexpr bool AHEAD = STAGED;
        const uint8_t *xb = (const uint8_t *)xb_s[cur];
        gm_h8 ah[2], al[2];
        ah[0] = gm_frag_at(xb, lane, 0, 0, 0);
        al[0] = gm_frag_at(xb, lane, 0, 0, 1);
#pragma unroll
        for (int p = 0; p < 4; p++) {
            if (!(p & 1)) {
                wt.split(p >> 1);
                wt.load(rs, 2 * sn + (p >> 1), p >> 1);
                __builtin_amdgcn_sched_barrier(0);
            }
#pragma unroll
            for (int t = 0; t < 4; t++) {
                const int i1 = 4 * p + t + (AHEAD ? 1 : 0);
                if (i1 < 16) {
                    ah[i1 & 1] = gm_frag_at(xb + (i1 >> 2) * GM_UNIT, lane, i1 >> 2, i1 & 3, 0);
                    al[i1 & 1] = gm_frag_at(xb + (i1 >> 2) * GM_UNIT, lane, i1 >> 2, i1 & 3, 1);
                }
                gm_h8 b[2][1];
#pragma unroll
                for (int j = 0; j < 2; j++) wt.frag(p >> 1, p & 1, t, j, b[j]);
                const gm_h8 hi = ah[t & 1], lo = al[t & 1];
#pragma unroll
                for (int j = 0; j < 2; j++)
                    S[j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(lo, b[j][0], p == 0 && t == 0 ? zero : S[j], 0, 0, 0);
#pragma unroll
                for (int j = 0; j < 2; j++)
                    S[j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(hi, b[j][0], S[j], 0, 0, 0);
            }
        }
        taken.mark(sb, ps[cur][lane & 31]);
        gm_fold<FMT_Q4K>(acc, S, wt, ps[cur], f, *(const gm_h8 *)((const uint8_t *)ms[cur] + 16 * lane));
        if (sb + 1 < nb) { // uniform
            store_x(cur ^ 1);
            load_x(min(sb + 2, nb - 1));
            __syncthreads();
        }
    }
    const int row = r0 + WROWS * wave + nl; // NMAT 2: of gate and up; NMAT 1: and row + 32
    if (__builtin_expect(taken.any(), 0)) {
        gm_add_halves<FMT_Q4K>(
            acc, wt, cols, [&](int t) { return xs + (size_t)(slot_s[t] / xdiv) * cols; }, n, 0, nb, taken,
            [&](int sb) { wt.head_load(rs, sb), wt.head(); },
            [&](int sb, int i) { wt.load(rs, 2 * sb + i, i), wt.split(i); }, (uint8_t *)xb_s[0], (uint8_t *)ms[0], ps[0]);
        const int row1 = NMAT == 2 ? row : row + 32;
        gm_add_outliers<FMT_Q4K>(
            acc, row < rows ? rowA[e] + (size_t)row * stride : nullptr,
            row1 < rows ? (NMAT == 2 ? rowB : rowA)[e] + (size_t)row1 * stride : nullptr, cols,
            [&](int t) { return xs + (size_t)(slot_s[t] / xdiv) * cols; }, n, 0, nb, taken, 0);
    }
#pragma unroll
    for (int i = 0; i < 16; i++) {
        const int t = 8 * (i >> 2) + 4 * f + (i & 3);
        if (t >= n) continue;
        float *o = out + (size_t)slot_s[t] * rows;
        if constexpr (NMAT == 2) {
            const float g = acc[0][i];
            if (row < rows) o[row] = g / (1.0f + expf(-g)) * acc[1][i];
        } else {
            if (row < rows) o[row] = acc[0][i];
            if (row + 32 < rows) o[row + 32] = acc[1][i];
        }
    }
}

// y = the splits' partial sums, added in split order; eight splits' values are
// requested at a time (one after another, a thread's chain of round trips was
// longer than the products: 1117 x 6912 at 49 tokens, 27 splits).
template <typename T> // float, or four (where the splits' starts are 16-byte aligned)
__global__ void __launch_bounds__(256) k_gm_reduce(const float *__restrict__ part, long count, int nsplit,
                                                   float *__restrict__ y)
{
    const long i = ((long)blockIdx.x * 256 + threadIdx.x) * (long)(sizeof(T) / 4);
    if (i >= count) return;
    T s = *(const T *)(part + i);
    for (int k0 = 1; k0 < nsplit; k0 += 8) {
        T v[8];
#pragma unroll
        for (int k = 0; k < 8; k++) v[k] = *(const T *)(part + min(k0 + k, nsplit - 1) * count + i);
#pragma unroll
        for (int k = 0; k < 8; k++)
            if (k0 + k < nsplit) s += v[k]; // uniform
    }
    *(T *)(y + i) = s;
}

static bool gemm_shape_ok(uint8_t dtype, size_t rows, size_t cols)
{
    return (dtype == SOSO_HIP_DTYPE_Q4_K || dtype == SOSO_HIP_DTYPE_Q8_0 || dtype == SOSO_HIP_DTYPE_Q6_K) &&
           cols % (dtype == SOSO_HIP_DTYPE_Q8_0 ? 64 : 256) == 0 && cols >= 256 && cols <= (1u << 20) && rows > 0 &&
           rows < ((size_t)1 << 31) - 256 && (size_t)256 * packed_row_stride(dtype, cols) < ((size_t)1 << 31);
}

// Where these kernels are the faster ones, from both sides measured on
// MI355X over rows x cols from 300 x 512 to 14336 x 14336 (us, before -> here):
//  * Rows of more than 4096 columns ran vector by vector below 16 tokens (and
//    always for Q6_K): 4096 x 14336 at 4 tokens 40 -> 22 (Q4_K), 50 -> 32
//    (Q6_K); at 3 small matrices lose (300 x 8192: 17 -> 20).  Q8_0 wins from
//    6 (79 -> 58; at 4: 53 -> 59).
//  * Q4_K up to 4096 columns: against the batched vector kernel (below 16
//    tokens) from 8 tokens and 2^22 weights (14336 x 4096 36.5 -> 20.9, 2048 x
//    2048 10.1 -> 9.8; 768 x 2048 8.8 -> 9.4), from 9 for smaller ones of 3584
//    and more (300 x 3584 11.7 -> 10.4; at 8: 10.2 -> 10.2).  Against the integer
//    matrix-core kernels, whose time is one chain along the columns, everywhere
//    from 3584 columns (300 / 1024 / 4096 / 14336 rows at 16 tokens 13.9 / 14.0 /
//    14.3 / 24.4 -> 10.8 / 11.2 / 13.0 / 20.9, at 64 14.4 / 14.6 / 24.9 / 58.4 ->
//    12.4 / 13.7 / 20.3 / 36.6; at 3072 columns 14336 rows at 48 tokens 30.3 ->
//    34.3, 300 at 33 11.5 -> 12.3); with fewer columns past 2^24 weights at 17
//    to 32 tokens (14336 x 2048 at 16 / 20 / 32 / 48: 15.1 / 25.3 / 24.2 / 23.2
//    -> 16.5 / 18.4 / 20.7 / 27.2), and past 64 tokens from 2.1e8 products at
//    2048 columns (1024 x 2048 at 100: 14.1 -> 12.7; 100 x 2048 at 1000: 11.6 ->
//    12.4), 8e8 below (14336 x 768 at 70 20.8 -> 17.5, 1000 x 1280 at 600 23.8 ->
//    20.0; 1000 x 1024 at 700 18.2 -> 19.2, 8192 x 512 at 128 11.5 -> 13.4).
//    Near these lines a call can be up to a tenth slower than it was: 14336 rows
//    one or two tokens past 64, which the integer kernels take by themselves (x
//    1536 at 65 / 66 29.4 / 27.6 -> 30.4 / 29.8), 1000 x 2304 at 70 11.8 -> 13.0.
//    Whole rounds of 16 tokens go through the integer kernels in one pass while
//    all their workgroups fit the GPU: four per CU up to 1024 columns (4096 x 768
//    at 256 16.7 -> 22.3, 8192 x 768 at 128 16.5 -> 18.8, 2048 x 1024 at 400 19.0
//    -> 21.1; past it 14336 x 768 at 80 28.5 -> 18.8), two below 2048 (4096 x 1536
//    at 128 17.2 -> 20.8; at 144 28.2 -> 21.4), one up to 2816 and 256 tokens (2048 x 2304
//    at 128 17.3 -> 21.2, 1000 x 2560 at 256 18.8 -> 20.8; 300 x 2304 at 512 20.8
//    -> 18.3).  Their form with x staged once (whole 1024-column chunks, a full
//    grid) holds out longer: 2048 x 2048 at 128 / 256 tokens 14.8 / 24.8 -> 16.1 /
//    21.3, 4096 x 1024 at 400 / 512 28.3 / 29.9 -> 22.1 / 23.9, 14336 x 1024 at 144
//    27.9 -> 30.7.
//  * Q6_K up to 4096 columns: past 2^24 weights from 8 tokens (14336 x 4096
//    41.7 -> 27.6); smaller ones, 2^24 itself among them, from 48 tokens (1000 x
//    1024 38.9 -> 15.4): not for the times, but because below that they keep the
//    batched vector kernel and with it the bits of single matvecs.
//  * Q8_0, whose four code planes cost its lines four visits: past 2^24 weights
//    from 33 tokens (14336 x 4096 at 64: 97 -> 51; at 32: 51 -> 53), smaller ones
//    from 16: always from 3072 columns (512 x 4096 24.1 -> 14.4, 1000 x 3072 18.9
//    -> 14.4; at 12: 17 -> 14, at 8: 10 -> 14), from 1.9e8 products at 2048 (1500
//    x 2048 at 64 21.8 -> 15.3, 4096 x 2048 at 32 21.8 -> 16.9; 512 x 2048 at 128
//    13.2 -> 14.9), 5e8 at 1024 (4096 x 1536 at 80 25.3 -> 22.6; at 64 16.1 ->
//    18.0, 300 x 1536 at 1000 25.9 -> 27.5) and 1e9 below (300 x 768 at 4500 54.8
//    -> 39.0; 8192 x 512 at 128 14.8 -> 16.4).  Against the form with x staged
//    once, from 1e9 products (2048 x 2048 at 128 / 256: 17.0 / 30.8 -> 20.5 / 27.4,
//    4096 x 4096 at 64 27.4 -> 25.2), 1.5e9 at 1024 columns (4096 x 1024 at 64 /
//    256 / 512: 10.5 / 23.3 / 41.6 -> 15.7 / 28.8 / 33.8).  Widths that are no
//    multiple of 256 ran on the batched vector kernel: from 16 tokens (5000 x
//    1440 26.3 -> 17.2), if 2^22 weights or 1024 columns (2014 x 768 at 149:
//    15.6 -> 16.3).
bool gemm_wins(const soso_hip *h, uint8_t dtype, size_t rows, size_t cols, size_t n)
{
    if (n < 4 || n > (1u << 20) || !gemm_shape_ok(dtype, rows, cols)) return false;
    const size_t weights = rows * cols, work = weights * n, cu = (size_t)h->num_cu;
    const bool large = weights > (1u << 24), small = weights < (1u << 22);
    // the integer kernels' workgroups (64 rows x 16 tokens) where every one has 16 tokens
    const size_t wgs = (rows + 63) / 64 * (n / 16);
    if (dtype == SOSO_HIP_DTYPE_Q8_0) {
        if (cols > 4096) return n >= 6;
        if (cols % 256) return n >= 16 && (!small || cols >= 1024);
        if (n < (large ? 33 : 16)) return false;
        if (n % 16 == 0 && cols % 1024 == 0 && wgs * 5 >= cu * 4) return work >= (cols >= 2048 ? 1000000000u : 1500000000u);
        return cols >= 3072 || work >= (cols >= 2048 ? 190000000u : cols >= 1024 ? 500000000u : 1000000000u);
    }
    if (cols > 4096) return true;
    if (dtype == SOSO_HIP_DTYPE_Q6_K) return n >= (large ? 8 : 48);
    if (cols >= 3584) return n >= (small ? 9 : 8);
    if (!small && n < 16) return n >= 8;
    if (n <= 64) return large && n > 16 && n <= 32;
    if (n % 16 == 0) {
        if (wgs <= cu * (cols <= 1024 ? 4 : cols < 2048 ? 2 : cols > 2048 && cols < 3072 && n <= 256 ? 1 : 0)) return false;
        if (cols % 1024 == 0) {
            if (n <= (cols < 2048 ? 240 : 128)) return work >= 3000000000u;
            if (cols < 2048 && (rows + 255) / 256 * (n / 16) * 5 >= cu * 4) return work >= 1500000000u;
        }
    }
    return work >= (cols >= 2048 ? 210000000u : 800000000u);
}

static int gm_reduce(soso_hip *h, const float *part, size_t count, size_t nsplit, float *y)
{
    if (count % 4 == 0 && ((uintptr_t)y & 15) == 0)
        k_gm_reduce<gm_f4><<<(unsigned)((count + 1023) / 1024), 256, 0, h->stream>>>(part, (long)count, (int)nsplit, y);
    else
        k_gm_reduce<float><<<(unsigned)((count + 255) / 256), 256, 0, h->stream>>>(part, (long)count, (int)nsplit, y);
    return hip_check(h, hipGetLastError(), "gemm reduce launch");
}

template <int FMT>
static int launch_gemm_fmt(soso_hip *h, const Weight &w, const float *x, size_t n, float *y)
{
    const size_t cols = weight_kcols(w), rows = w.rows, nb = (cols + 255) / 256, rb = (rows + 255) / 256;
    const size_t stride = packed_row_stride(w.dtype, cols);
    // Few tokens, or a small product: a chain of super-blocks per workgroup that
    // is short on round trips beats more products per weight (4096 x 4096 at 64
    // tokens 20.6 us against 25.4, 6905 x 1280 at 200 26.6 against 33.3; at 200
    // tokens 4096 x 4096 42.3 against 35.2, 14336 x 4096 at 64 43.4 against
    // 37.5).
    const bool few = FMT != FMT_Q80 && (n <= 32 || rows * cols * n <= ((size_t)1 << 31));
    // (Q8_0's per-block scales need a second set of sums: one token tile)
    const size_t MT = FMT != FMT_Q80 && !few ? 2 : 1;
    const size_t ntt = (n + 32 * MT - 1) / (32 * MT), tiles = ntt * MT;
    // as many column splits as fill the GPU's workgroup slots: two per CU, one
    // for few tokens (fewer partial sums; 14336 x 4096 at 2 / 8 / 32 tokens
    // 18.6 / 20.2 / 27.9 us against 19.3 / 20.9 / 28.9 with two)
    const size_t slots = (few ? 1 : 2) * (size_t)h->num_cu;
    const size_t nsplit = std::max<size_t>(1, std::min(nb, slots / (ntt * rb)));
    const size_t items = rb * nsplit * ntt;
    const unsigned grid = (unsigned)((items + 7) / 8 * 8);
    float *part = y;
    if (nsplit > 1) {
        part = (float *)scratch_get(h, 17, nsplit * n * rows * 4);
        if (!part) return SOSO_HIP_DECLINED;
    }
    if (few) {
        if constexpr (FMT != FMT_Q80)
            k_gemm_few<FMT><<<grid, 256, 0, h->stream>>>((const uint8_t *)w.dev, stride, (int)rows, (int)cols, x,
                                                         (int)n, (int)ntt, (int)nsplit, (int)items, part);
    } else {
        const size_t f_b = tiles * nb * (4 * GM_UNIT), m_b = tiles * nb * GM_SUMS, p_b = tiles * nb * 128;
        uint8_t *xg = (uint8_t *)scratch_get(h, 16, f_b + m_b + p_b);
        if (!xg) return SOSO_HIP_DECLINED;
        float *xp = (float *)(xg + f_b + m_b);
        const GmX gx{xg, xg + f_b, xp};
        k_gm_stage<FMT><<<(unsigned)(tiles * nb), 512, 0, h->stream>>>(x, (int)n, (int)cols, (int)w.cols, xg, xg + f_b, xp);
        k_gemm<FMT, FMT == FMT_Q80 ? 1 : 2><<<grid, 256, 0, h->stream>>>(
            (const uint8_t *)w.dev, stride, (int)rows, (int)cols, gx, x, (int)n, (int)ntt, (int)nsplit, (int)items, part);
    }
    const int rc = hip_check(h, hipGetLastError(), "gemm launch");
    return rc == SOSO_HIP_OK && nsplit > 1 ? gm_reduce(h, part, n * rows, nsplit, y) : rc;
}

// DECLINED when the scratch it needs cannot be had (memory, or a slot that
// would have to grow inside a graph capture): the other kernels, which need
// none, take the call.
int launch_gemm(soso_hip *h, const Weight &w, const float *x, size_t n, float *y)
{
    switch (w.dtype) {
    case SOSO_HIP_DTYPE_Q4_K: return launch_gemm_fmt<FMT_Q4K>(h, w, x, n, y);
    case SOSO_HIP_DTYPE_Q8_0: return launch_gemm_fmt<FMT_Q80>(h, w, x, n, y);
    default: return launch_gemm_fmt<FMT_Q6K>(h, w, x, n, y);
    }
}

// One grouped product of a registered MoE layer's Q4_K experts with tile-major
// copies (nmat 2: gate / up, 1: down) over the active-expert records; slots: the
// call's (token, rank) pairs, each in at most one record's list; n: x's rows.
// x is converted once per call where scratch may be had (not fixed, and memory),
// else by every workgroup: the same bits.
int launch_gemm_moe(soso_hip *h, int nmat, const uint8_t *const *tiled, const uint8_t *const *row_major, size_t n_groups,
                    size_t rows, size_t cols, size_t slots, size_t max_recs, const float *xs, size_t n, int xdiv,
                    const int *list, const int *recs, const int *n_recs, bool fixed, float *out)
{
    if (max_recs > 256 || !tiled_q4k_ok(SOSO_HIP_DTYPE_Q4_K, rows, cols) ||
        !gemm_shape_ok(SOSO_HIP_DTYPE_Q4_K, rows, cols))
        return SOSO_HIP_DECLINED;
    const size_t nblk = (rows + (nmat == 2 ? 127 : 255)) / (nmat == 2 ? 128 : 256), tiles = slots / 32 + max_recs;
    const size_t stride = packed_row_stride(SOSO_HIP_DTYPE_Q4_K, cols), nb = cols / 256;
    const unsigned grid = (unsigned)(tiles * nblk);
    const size_t f_b = n * nb * GM_TOK, m_b = n * nb * GM_TOK_SUMS, p_b = n * nb * 4;
    uint8_t *xg = fixed ? nullptr : (uint8_t *)scratch_get(h, 16, f_b + m_b + p_b);
    GmX gx{xg, xg + f_b, (const float *)(xg + f_b + m_b)};
    if (xg)
        k_gm_stage_tok<<<(unsigned)(((n + 3) / 4 * nb + 3) / 4), 256, 0, h->stream>>>(xs, (int)n, (int)cols, xg,
                                                                                     xg + f_b, (float *)(xg + f_b + m_b));
#define GM_MOE(NM, ST)                                                                                                 \
    k_gemm_moe<NM, ST><<<grid, 256, 0, h->stream>>>(tiled, NM == 2 ? tiled + n_groups : nullptr, row_major,           \
                                                    NM == 2 ? row_major + n_groups : nullptr, stride, (int)rows,      \
                                                    (int)cols, xs, gx, xdiv, list, recs, n_recs, (int)nblk, out)
    if (nmat == 2 && xg) GM_MOE(2, true);
    else if (nmat == 2) GM_MOE(2, false);
    else if (xg) GM_MOE(1, true);
    else GM_MOE(1, false);
#undef GM_MOE
    return hip_check(h, hipGetLastError(), "gemm moe launch");
}
