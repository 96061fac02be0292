// k_gdn.hip -- Gated DeltaNet (Qwen3.5) on the device: the recurrence of
// GpuDispatch::gdn_bloque (crates/soso-llm-core/src/gpu.rs:577-599), as
// soso's CPU path computes it (bloque35.rs:372-465; one token of the decode
// layer, arch.rs:586-768, is the same with n = 1).
//
// With S the head's d x d state (d = 128), per token
//     delta_j = (v_j - g sum_i S_ij k_i) beta
//     S_ij   <- g S_ij + k_i delta_j
//     o_j     = sum_i S_ij q_i = g (sum_i S_ij q_i before) + delta_j (k . q)
// then rmsnorm(o) with the ssm_norm weights and o *= silu(z).  Nothing joins
// two columns j before the norm, so the columns of a head run apart:
//   k_gdn_conv  a wavefront per token and q/k head pair or value head: the
//               causal conv over the history window, SiLU, and for q / k the
//               l2 normalisation (q also scaled by 1 / sqrt(d)) -> u [n][C],
//               C = 2 n_k d + n_v d, and k . q [n][n_k]
//   k_gdn_rec   the recurrence in eight workgroups per value head, the state
//               in registers for the whole block, read once and written once;
//               both sums of a token in one pass over the rows, then DPP adds
//               across a column's lanes: no barrier per token; o takes v's place
//               in u, so that out may be z's buffer
//   k_gdn_norm  the norm and the gate, a wavefront per token and head
//   k_gdn_rec_few  up to GDN_FEW tokens: a workgroup per head, norm and gate
//               included (one launch less)
// Both recurrences add in the same order, so a block's bits do not depend on how
// its tokens were split into calls.  One workgroup of 1024 threads per head,
// four workgroup barriers per token, took 370 us for 256 tokens of 32 heads;
// the state traffic per block is 2 * n_v d^2 * 4 bytes (2 MiB each way for 32
// heads), independent of n.
#include "internal.hpp"

constexpr int GDN_D = 128;    // head dim handled (gdn_bloque: d == 128 only)
// Tokens up to which one workgroup takes a whole head (us per call, 32 value
// heads, one workgroup per head / eight and the norm's launch: 4 tokens 8.98,
// 5 9.93 / 9.8, 8 12.6 / 9.8).
constexpr int GDN_FEW = 4;
constexpr int GDN_CHUNK = 32; // tokens staged in LDS at a time beyond

__device__ __forceinline__ float gdn_silu(float x) { return x / (1.0f + expf(-x)); }

// sum over the wavefront, returned to all lanes
__device__ __forceinline__ float gdn_sum64(float v)
{
    v = seg_sum_dpp<64>(v);
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 63));
}

// silu(conv) of two channels (2 lane, 2 lane + 1 of head hh) for token t
__device__ __forceinline__ float2 gdn_conv2(const float *__restrict__ hist, const float *__restrict__ conv, int C,
                                            int kernel, int ch, int t)
{
    float a = 0.0f, b = 0.0f;
    for (int k = 0; k < kernel; k++) {
        const float2 h = *(const float2 *)(hist + (size_t)(t + k) * C + ch);
        a = __fadd_rn(a, __fmul_rn(conv[(size_t)ch * kernel + k], h.x));
        b = __fadd_rn(b, __fmul_rn(conv[(size_t)(ch + 1) * kernel + k], h.y));
    }
    return make_float2(gdn_silu(a), gdn_silu(b));
}

// Wavefront: unit (a q/k head pair, then the value heads) of one token; kernel
// widths 1..4 unrolled (KW), others by the loop (KW = 0).  (2 / 4 / 8 tokens
// per wavefront, sharing their window: 256 tokens 55.5 / 58.1 / 66.1 us per call
// against 54.8.)
template <int KW>
__global__ void __launch_bounds__(256) k_gdn_conv(const float *__restrict__ hist, const float *__restrict__ conv, int n,
                                                  int n_k, int n_v, int kernel_, float eps, float *__restrict__ u,
                                                  float *__restrict__ kq)
{
    const int kernel = KW ? KW : kernel_;
    const int lane = threadIdx.x & 63, units = n_k + n_v;
    const long gw = (long)blockIdx.x * 4 + (threadIdx.x >> 6);
    const int unit = (int)(gw % units);
    const long t = gw / units;
    if (t >= n) return; // no barriers here
    const int C = (2 * n_k + n_v) * GDN_D;
    const bool qk = unit < n_k;
    const int ch = (qk ? unit : n_k + unit) * GDN_D + 2 * lane; // q head, or value head
    float *ut = u + (size_t)t * C;
    float2 q = gdn_conv2(hist, conv, C, kernel, ch, (int)t);
    if (qk) {
        const int ck = ch + n_k * GDN_D;
        float2 k = gdn_conv2(hist, conv, C, kernel, ck, (int)t);
        const float qn = 1.0f / sqrtf(gdn_sum64(q.x * q.x + q.y * q.y) + eps);
        const float kn = 1.0f / sqrtf(gdn_sum64(k.x * k.x + k.y * k.y) + eps);
        const float sc = 1.0f / sqrtf((float)GDN_D);
        q = make_float2(q.x * qn * sc, q.y * qn * sc);
        k = make_float2(k.x * kn, k.y * kn);
        *(float2 *)(ut + ck) = k;
        const float d = gdn_sum64(fmaf(k.x, q.x, k.y * q.y));
        if (lane == 0) kq[(size_t)t * n_k + unit] = d;
    }
    *(float2 *)(ut + ch) = q;
}

// rmsnorm(o) over the head (gemm.rs:93-100) with its weights, then the SiLU
// gate, of columns 2 lane and 2 lane + 1
__device__ __forceinline__ float2 gdn_norm2(float2 o, float2 z, const float *__restrict__ norm, int lane, float eps)
{
    const float scale = 1.0f / sqrtf(gdn_sum64(o.x * o.x + o.y * o.y) / (float)GDN_D + eps);
    const float2 w = *(const float2 *)(norm + 2 * lane);
    return make_float2(__fmul_rn(__fmul_rn(__fmul_rn(o.x, scale), w.x), gdn_silu(z.x)),
                       __fmul_rn(__fmul_rn(__fmul_rn(o.y, scale), w.y), gdn_silu(z.y)));
}

// The sums over a row group's eight rows (rows 4 r .. 4 r + 3 and 64 + 4 r ..
// 64 + 4 r + 3 of group r = 0 .. 15, so that LDS reads are contiguous), and a
// token's step once both sums over the 16 groups are there: the pieces that
// both recurrence kernels share, so that their bits agree.
__device__ __forceinline__ void gdn_group(const float (&S)[8], const float4 (&k)[2], const float4 (&q)[2], float &p,
                                          float &r)
{
    const float kk[8] = {k[0].x, k[0].y, k[0].z, k[0].w, k[1].x, k[1].y, k[1].z, k[1].w};
    const float qq[8] = {q[0].x, q[0].y, q[0].z, q[0].w, q[1].x, q[1].y, q[1].z, q[1].w};
    float p1 = S[4] * kk[4], r1 = S[4] * qq[4];
    p = S[0] * kk[0];
    r = S[0] * qq[0];
#pragma unroll
    for (int i = 1; i < 4; i++) {
        p = fmaf(S[i], kk[i], p);
        p1 = fmaf(S[4 + i], kk[4 + i], p1);
        r = fmaf(S[i], qq[i], r);
        r1 = fmaf(S[4 + i], qq[4 + i], r1);
    }
    p += p1;
    r += r1;
}
__device__ __forceinline__ float gdn_delta(float v, float g, float beta, float p) { return fmaf(-g, p, v) * beta; }
__device__ __forceinline__ float gdn_out(float delta, float kq, float g, float r) { return fmaf(delta, kq, g * r); }
__device__ __forceinline__ void gdn_update(float (&S)[8], const float4 (&k)[2], float g, float delta)
{
    const float kk[8] = {k[0].x, k[0].y, k[0].z, k[0].w, k[1].x, k[1].y, k[1].z, k[1].w};
#pragma unroll
    for (int i = 0; i < 8; i++) S[i] = fmaf(kk[i], delta, g * S[i]);
}

// Up to GDN_FEW tokens: a workgroup per head, thread (r, j): column j, row
// groups 2 r and 2 r + 1 (whole rows of the state per load).  The groups' sums
// meet in LDS, one barrier per token; every thread of a column adds them.
__global__ void __launch_bounds__(1024) k_gdn_rec_few(const float *__restrict__ u, const float *__restrict__ kq,
                                                      const float *z, const float *__restrict__ decay,
                                                      const float *__restrict__ beta, const float *__restrict__ norm,
                                                      float *__restrict__ state, float *out, int n, int n_k, int n_v,
                                                      float eps)
{
    constexpr int D = GDN_D;
    __shared__ float qk[GDN_FEW][2 * D];
    __shared__ float vs[GDN_FEW][D];
    __shared__ float2 part[2][8][D];
    __shared__ float os[GDN_FEW][D];
    const int vh = blockIdx.x, kh = vh % n_k, tid = threadIdx.x, j = tid & (D - 1), r = tid >> 7;
    const int qd = n_k * D, C = 2 * qd + n_v * D, vd = n_v * D;
    float *st = state + (size_t)vh * D * D + j;
    for (int w = tid; w < n * 3 * D; w += 1024) { // n q, k, v rows of the head
        const int t = w / (3 * D), c = w % (3 * D);
        const float x = u[(size_t)t * C + (c < D ? kh * D + c : c < 2 * D ? qd + kh * D + c - D : 2 * qd + vh * D + c - 2 * D)];
        if (c < 2 * D) qk[t][c] = x;
        else vs[t][c - 2 * D] = x;
    }
    float S[2][8];
#pragma unroll
    for (int a = 0; a < 2; a++)
#pragma unroll
        for (int i = 0; i < 8; i++) S[a][i] = st[(size_t)(64 * (i >> 2) + 4 * (2 * r + a) + (i & 3)) * D];
    __syncthreads();
    for (int t = 0; t < n; t++) {
        const float g = decay[(size_t)t * n_v + vh], b = beta[(size_t)t * n_v + vh], d = kq[(size_t)t * n_k + kh];
        float4 k4[2][2], q4[2][2];
#pragma unroll
        for (int a = 0; a < 2; a++)
#pragma unroll
            for (int h = 0; h < 2; h++) {
                q4[a][h] = *(const float4 *)&qk[t][64 * h + 4 * (2 * r + a)];
                k4[a][h] = *(const float4 *)&qk[t][D + 64 * h + 4 * (2 * r + a)];
            }
        float p0, r0, p1, r1;
        gdn_group(S[0], k4[0], q4[0], p0, r0);
        gdn_group(S[1], k4[1], q4[1], p1, r1);
        part[t & 1][r][j] = make_float2(p0 + p1, r0 + r1);
        __syncthreads();
        float2 s[8];
#pragma unroll
        for (int a = 0; a < 8; a++) s[a] = part[t & 1][a][j];
        const float p = ((s[0].x + s[1].x) + (s[2].x + s[3].x)) + ((s[4].x + s[5].x) + (s[6].x + s[7].x));
        const float ro = ((s[0].y + s[1].y) + (s[2].y + s[3].y)) + ((s[4].y + s[5].y) + (s[6].y + s[7].y));
        const float dj = gdn_delta(vs[t][j], g, b, p);
        gdn_update(S[0], k4[0], g, dj);
        gdn_update(S[1], k4[1], g, dj);
        if (r == 0) os[t][j] = gdn_out(dj, d, g, ro);
    }
#pragma unroll
    for (int a = 0; a < 2; a++)
#pragma unroll
        for (int i = 0; i < 8; i++) st[(size_t)(64 * (i >> 2) + 4 * (2 * r + a) + (i & 3)) * D] = S[a][i];
    __syncthreads();
    const int lane = tid & 63, wave = tid >> 6;
    if (wave < n) {
        const size_t o = (size_t)wave * vd + vh * D + 2 * lane;
        *(float2 *)(out + o) =
            gdn_norm2(*(const float2 *)&os[wave][2 * lane], *(const float2 *)(z + o), norm, lane, eps);
    }
}

// Longer blocks: 16 columns per workgroup, four per wavefront, a column's 16
// row groups in 16 lanes: 256 workgroups, a wavefront per SIMD, for 32 heads.
// Bound by the chain of one token's instructions (about 70, 0.15 us): 256 tokens
// of 16 q/k and 32 value heads took 385 us per call on MI355X with a workgroup
// and four barriers per token and head, 55 us now; 64 tokens 86.8 -> 19.8.
__global__ void __launch_bounds__(256) k_gdn_rec(float *__restrict__ u, const float *__restrict__ kq,
                                                 const float *__restrict__ decay, const float *__restrict__ beta,
                                                 float *__restrict__ state, int n, int n_k, int n_v)
{
    constexpr int D = GDN_D, COLS = 16, NT = 256, TC = GDN_CHUNK, KQ = TC * 2 * D / 4 / NT, VW = TC * COLS / NT;
    __shared__ float qk[2][TC][2 * D];
    __shared__ float vs[2][TC][COLS];
    __shared__ float4 gs[2][TC]; // g, beta, k . q
    __shared__ float os[TC][COLS];
    const int vh = (int)blockIdx.x % n_v, c0 = (int)blockIdx.x / n_v * COLS, kh = vh % n_k;
    const int tid = threadIdx.x, cl = tid >> 4, rg = tid & 15; // column of the workgroup, row group
    const int qd = n_k * D, C = 2 * qd + n_v * D;
    float *st = state + (size_t)vh * D * D + c0 + cl;
    float S[8];
#pragma unroll
    for (int i = 0; i < 8; i++) S[i] = st[(size_t)(64 * (i >> 2) + 4 * rg + (i & 3)) * D];
    // a chunk on its way: tokens t .. t + m - 1
    float4 nqk[KQ], ng;
    float nv[VW];
    auto fetch = [&](int t, int m) {
#pragma unroll
        for (int k = 0; k < KQ; k++) {
            const int w = k * NT + tid, tt = w / (2 * D / 4), c = w % (2 * D / 4) * 4; // q, then k
            nqk[k] = make_float4(0.f, 0.f, 0.f, 0.f);
            if (tt < m) nqk[k] = *(const float4 *)(u + (size_t)(t + tt) * C + (c < D ? kh * D + c : qd + kh * D + c - D));
        }
#pragma unroll
        for (int k = 0; k < VW; k++) {
            const int w = k * NT + tid, tt = w / COLS;
            nv[k] = tt < m ? u[(size_t)(t + tt) * C + 2 * qd + vh * D + c0 + w % COLS] : 0.0f;
        }
        ng = make_float4(0.f, 0.f, 0.f, 0.f);
        if (tid < m) {
            const size_t g = (size_t)(t + tid) * n_v + vh;
            ng = make_float4(decay[g], beta[g], kq[(size_t)(t + tid) * n_k + kh], 0.0f);
        }
    };
    auto store = [&](int b) {
#pragma unroll
        for (int k = 0; k < KQ; k++) *(float4 *)(&qk[b][0][0] + 4 * (k * NT + tid)) = nqk[k];
#pragma unroll
        for (int k = 0; k < VW; k++) (&vs[b][0][0])[k * NT + tid] = nv[k];
        if (tid < TC) gs[b][tid] = ng;
    };
    struct Ops { // a token's operands
        float4 q[2], k[2], g;
        float v;
    };
    fetch(0, min(TC, n));
    store(0);
    __syncthreads();
    int b = 0;
    for (int t0 = 0; t0 < n; t0 += TC) {
        const int m = min(TC, n - t0);
        if (t0 + TC < n) {
            fetch(t0 + TC, min(TC, n - t0 - TC)); // in flight during this chunk's recurrence
            __builtin_amdgcn_sched_barrier(0);
        }
        auto operands = [&](int t, Ops &o) {
            t = min(t, m - 1);
#pragma unroll
            for (int h = 0; h < 2; h++) {
                o.q[h] = *(const float4 *)&qk[b][t][64 * h + 4 * rg];
                o.k[h] = *(const float4 *)&qk[b][t][D + 64 * h + 4 * rg];
            }
            o.g = gs[b][t];
            o.v = vs[b][t][cl];
        };
        auto step = [&](const Ops &o, int t) {
            float p, r;
            gdn_group(S, o.k, o.q, p, r);
            p = seg_sum_dpp<16>(p);
            r = seg_sum_dpp<16>(r);
            const float dj = gdn_delta(o.v, o.g.x, o.g.y, p);
            gdn_update(S, o.k, o.g.x, dj);
            os[t][cl] = gdn_out(dj, o.g.z, o.g.x, r); // (the column's 16 lanes write the same value)
        };
        // two sets of operands in turn, each read from LDS a token ahead
        Ops oa, ob;
        operands(0, oa);
        int t = 0;
        for (; t + 2 <= m; t += 2) {
            operands(t + 1, ob);
            step(oa, t);
            operands(t + 2, oa);
            step(ob, t + 1);
        }
        if (t < m) step(oa, t);
        if (t0 + TC < n) store(b ^ 1);
        __syncthreads(); // the chunk's outputs, and the next chunk, are in LDS
        for (int w = tid; w < m * (COLS / 4); w += NT) {
            const int tt = w / (COLS / 4), c = w % (COLS / 4) * 4;
            // in v's place: this workgroup alone reads it, and has
            *(float4 *)(u + (size_t)(t0 + tt) * C + 2 * qd + vh * D + c0 + c) = *(const float4 *)&os[tt][c];
        }
        __syncthreads(); // os is rewritten by the next chunk
        b ^= 1;
    }
#pragma unroll
    for (int i = 0; i < 8; i++) st[(size_t)(64 * (i >> 2) + 4 * rg + (i & 3)) * D] = S[i];
}

// Wavefront per (token, value head): o from u to out (which may be z).
__global__ void __launch_bounds__(256) k_gdn_norm(const float *__restrict__ u, const float *z,
                                                  const float *__restrict__ norm, float *out, unsigned heads, unsigned n_k,
                                                  unsigned n_v, float eps)
{
    const int lane = threadIdx.x & 63;
    const unsigned w = blockIdx.x * 4 + (threadIdx.x >> 6), t = w / n_v; // below 65536^2 (gdn_unsupported)
    if (w >= heads) return;
    const size_t o = (size_t)w * GDN_D + 2 * lane, C = (size_t)(2 * n_k + n_v) * GDN_D;
    const float2 x = *(const float2 *)(u + t * C + (2 * n_k + (w - t * n_v)) * GDN_D + 2 * lane);
    *(float2 *)(out + o) = gdn_norm2(x, *(const float2 *)(z + o), norm, lane, eps);
}

const char *gdn_unsupported(size_t n, size_t n_k, size_t n_v, size_t d, size_t kernel)
{
    if (d != GDN_D) return "gdn: head dim must be 128";
    if (n == 0 || n_k == 0 || n_v == 0 || kernel == 0 || kernel > 16) return "gdn: empty block or kernel outside 1..16";
    if (n_v > 65535 || n_k > 65535 || n > 65535) return "gdn: too many heads or tokens (grid limits)";
    return nullptr;
}

size_t gdn_scratch_floats(size_t n, size_t n_k, size_t n_v) { return n * ((2 * n_k + n_v) * GDN_D + n_k); }

int launch_gdn_block(soso_hip *h, const float *hist, const float *conv, const float *z, const float *decay,
                     const float *beta, const float *norm, float *state, float *out, float *u, int n, int n_k,
                     int n_v, int kernel, float eps)
{
    float *kq = u + (size_t)n * (2 * n_k + n_v) * GDN_D;
    const unsigned cg = (unsigned)(((long)(n_k + n_v) * n + 3) / 4);
#define GDN_CONV(KW) k_gdn_conv<KW><<<cg, 256, 0, h->stream>>>(hist, conv, n, n_k, n_v, kernel, eps, u, kq)
    switch (kernel) {
    case 1: GDN_CONV(1); break;
    case 2: GDN_CONV(2); break;
    case 3: GDN_CONV(3); break;
    case 4: GDN_CONV(4); break;
    default: GDN_CONV(0); break;
    }
#undef GDN_CONV
    int rc = hip_check(h, hipGetLastError(), "gdn conv launch");
    if (rc != SOSO_HIP_OK) return rc;
    if (n <= GDN_FEW) {
        k_gdn_rec_few<<<(unsigned)n_v, 1024, 0, h->stream>>>(u, kq, z, decay, beta, norm, state, out, n, n_k, n_v, eps);
        return hip_check(h, hipGetLastError(), "gdn recurrence launch");
    }
    k_gdn_rec<<<(unsigned)n_v * (GDN_D / 16), 256, 0, h->stream>>>(u, kq, decay, beta, state, n, n_k, n_v);
    rc = hip_check(h, hipGetLastError(), "gdn recurrence launch");
    if (rc != SOSO_HIP_OK) return rc;
    const long heads = (long)n * n_v;
    k_gdn_norm<<<(unsigned)((heads + 3) / 4), 256, 0, h->stream>>>(u, z, norm, out, (unsigned)heads, (unsigned)n_k,
                                                                  (unsigned)n_v, eps);
    return hip_check(h, hipGetLastError(), "gdn norm launch");
}
