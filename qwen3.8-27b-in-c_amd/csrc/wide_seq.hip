// Prompt path (gfx950): the two token-mixing layers over many tokens at once, causal gated
// attention and the Gated-DeltaNet recurrence (wide.hip holds the matrix products).
#include "qgpu_internal.h"

typedef _Float16 v8h __attribute__((ext_vector_type(8)));
typedef __bf16 v8b __attribute__((ext_vector_type(8)));
typedef float v4f __attribute__((ext_vector_type(4)));
typedef const __attribute__((address_space(1))) void *gptr_t;
typedef __attribute__((address_space(3))) void *lptr_t;

#define FA_HD   256
#define FA_TP   32            // positions per K/V tile
#define FA_TB   64            // tokens per block: 16 per wave
#define FA_KB   32768         // bytes of a tile's K planes; its V planes follow

// ---------------------------------------------------------------- attention
// K and V of 32 positions as matrix-core operands, once per layer and chunk (every query block
// reads them in this form): K as fp16 hi + lo, V as bf16 hi + lo (the split-precision
// products of attn.hip, same parts).  K: per (16 positions, 32 dims) the A operand of
// v_mfma_f32_16x16x32_f16, V: per 16 dims the A operand of the 32-position product, whose K-slot
// 8g + j is position 4g + j (j < 4) or 16 + 4g + j - 4: the order in which a lane holds the
// probabilities.  Positions past the live end are zero.
__global__ __launch_bounds__(256) void k_wide_kv(const float *__restrict__ kc, const float *__restrict__ vc,
                                                 uint8_t *__restrict__ P, uint32_t n_tile, uint32_t live, int n_kv)
{
    const uint32_t t = blockIdx.x, kvh = blockIdx.y, p0 = t * FA_TP;
    uint8_t *o = P + ((uint64_t)kvh * n_tile + t) * (2 * FA_KB);
    const uint64_t row = (uint64_t)n_kv * FA_HD;
    const float *K = kc + kvh * FA_HD, *V = vc + kvh * FA_HD;
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const uint32_t e = threadIdx.x + 256 * i, ln = e & 63, c = (e >> 6) & 7, sub = e >> 9;
        const uint32_t pos = p0 + sub * 16 + (ln & 15);
        float x[8] = { 0, 0, 0, 0, 0, 0, 0, 0 };
        if (pos < live) {
            const float *s = K + pos * row + 32 * c + 8 * (ln >> 4);
            const float4 a = *(const float4 *)s, b = *(const float4 *)(s + 4);
            x[0] = a.x; x[1] = a.y; x[2] = a.z; x[3] = a.w; x[4] = b.x; x[5] = b.y; x[6] = b.z; x[7] = b.w;
        }
        v8h hi, lo;
#pragma unroll
        for (int j = 0; j < 8; j++) { hi[j] = (_Float16)x[j]; lo[j] = (_Float16)(x[j] - (float)hi[j]); }
        *(v8h *)(o + ((sub * 8 + c) * 2) * 1024 + ln * 16) = hi;
        *(v8h *)(o + ((sub * 8 + c) * 2 + 1) * 1024 + ln * 16) = lo;
    }
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const uint32_t e = threadIdx.x + 256 * i, ln = e & 63, dt = e >> 6, g = ln >> 4;
        v8b hi, lo;
#pragma unroll
        for (int j = 0; j < 8; j++) {
            const uint32_t pos = p0 + (j < 4 ? 4 * g + j : 16 + 4 * g + j - 4);
            const float x = pos < live ? V[pos * row + 16 * dt + (ln & 15)] : 0.0f;
            hi[j] = (__bf16)x;
            lo[j] = (__bf16)(x - (float)hi[j]);
        }
        *(v8b *)(o + FA_KB + (dt * 2) * 1024 + ln * 16) = hi;
        *(v8b *)(o + FA_KB + (dt * 2 + 1) * 1024 + ln * 16) = lo;
    }
}

struct WideAttn {
    const float *q;                     // normalised and rotated; the gates follow each head's q
    uint64_t ldq;
    const uint8_t *P;
    float *out;
    uint64_t ldo;
    uint32_t n_tile, pos0, M, n_head, n_kv, nq;
};

// Causal flash attention: a block is one query head and 64 tokens (16 per wave); the K/V tiles of 32
// positions pass through LDS, K of the next tile loading behind the P.V product and V behind the
// scores.  Scores as S^T = K Q^T (a lane: one token, its positions 4g + i of two 16-row tiles), so
// the probabilities are already the B operand of O^T = V^T P^T and a token's running maximum and
// rescale factor stay in its own lanes.
__global__ __launch_bounds__(256, 2) void k_wide_attn(const WideAttn a)
{
    __shared__ __attribute__((aligned(16))) uint8_t Ks[FA_KB], Vs[FA_KB];
    const int lane = threadIdx.x & 63, n = lane & 15, g = lane >> 4;
    const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    // (kv head, query head of its group, token tile): the last tiles, which see the most
    // positions, first; where the kv heads divide the 8 XCDs each XCD keeps to one of them (its L2)
    const uint32_t per = a.n_head / a.n_kv;
    uint32_t kvh, it;
    if (8 % a.n_kv == 0) {
        const uint32_t x = blockIdx.x & 7, share = 8 / a.n_kv;
        kvh = x / share;
        it = (blockIdx.x >> 3) * share + x % share;
    } else {
        kvh = blockIdx.x % a.n_kv;
        it = blockIdx.x / a.n_kv;
    }
    if (it >= per * a.nq) return;
    const uint32_t h = kvh * per + it % per, qt = a.nq - 1 - it / per;
    const uint32_t t0 = qt * FA_TB + wv * 16, tok = t0 + n, row = min(tok, a.M - 1);
    const uint32_t qpos = a.pos0 + tok;                               // this lane's position
    const uint32_t nt = (a.pos0 + min(qt * FA_TB + FA_TB, a.M) - 1) / FA_TP + 1;
    const float *qr = a.q + (uint64_t)row * a.ldq + (uint64_t)h * 2 * FA_HD;
    v8h qh[8], ql[8];
    const float qs = 0.0625f * 1.44269504088896340736f;               // 1/sqrt(256), scores in log2 units
#pragma unroll
    for (int c = 0; c < 8; c++) {
        const float4 x0 = *(const float4 *)(qr + 32 * c + 8 * g), x1 = *(const float4 *)(qr + 32 * c + 8 * g + 4);
        const float x[8] = { x0.x, x0.y, x0.z, x0.w, x1.x, x1.y, x1.z, x1.w };
#pragma unroll
        for (int j = 0; j < 8; j++) {
            qh[c][j] = (_Float16)x[j];
            ql[c][j] = (_Float16)(x[j] - (float)qh[c][j]);
        }
    }
    const v4f z4 = { 0.0f, 0.0f, 0.0f, 0.0f };
    v4f O[16];
#pragma unroll
    for (int d = 0; d < 16; d++) O[d] = z4;
    float m = -INFINITY, l = 0.0f;
    const uint8_t *base = a.P + (uint64_t)kvh * a.n_tile * (2 * FA_KB);
    const uint32_t l16 = (uint32_t)lane * 16;
    auto load = [&](const uint8_t *src, uint8_t *dst) {
#pragma unroll
        for (int i = 0; i < 8; i++) {
            const int c = wv * 8 + i;
            __builtin_amdgcn_global_load_lds((gptr_t)(src + c * 1024 + l16), (lptr_t)(dst + c * 1024), 16, 0, 0);
        }
    };
    load(base, Ks);
    __builtin_amdgcn_s_waitcnt(0x0F70);
    __syncthreads();
    for (uint32_t t = 0; t < nt; t++) {
        load(base + (uint64_t)t * (2 * FA_KB) + FA_KB, Vs);
        v4f s[2], x[2];
        s[0] = s[1] = x[0] = x[1] = z4;
#pragma unroll
        for (int c = 0; c < 8; c++)
#pragma unroll
            for (int u = 0; u < 2; u++) {
                const v8h kh = *(const v8h *)(Ks + ((u * 8 + c) * 2) * 1024 + l16);
                const v8h kl = *(const v8h *)(Ks + ((u * 8 + c) * 2 + 1) * 1024 + l16);
                x[u] = __builtin_amdgcn_mfma_f32_16x16x32_f16(kl, qh[c], x[u], 0, 0, 0);
                s[u] = __builtin_amdgcn_mfma_f32_16x16x32_f16(kh, qh[c], s[u], 0, 0, 0);
                x[u] = __builtin_amdgcn_mfma_f32_16x16x32_f16(kh, ql[c], x[u], 0, 0, 0);
            }
        __builtin_amdgcn_s_waitcnt(0x0F70);
        __syncthreads();                              // V is in, every wave is done with K
        if (t + 1 < nt) load(base + (uint64_t)(t + 1) * (2 * FA_KB), Ks);
        float p[8], mx = m;
#pragma unroll
        for (int u = 0; u < 2; u++)
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const uint32_t pos = t * FA_TP + 16 * u + 4 * g + i;
                p[4 * u + i] = pos <= qpos ? (s[u][i] + x[u][i]) * qs : -INFINITY;
                mx = fmaxf(mx, p[4 * u + i]);
            }
        mx = fmaxf(mx, __shfl_xor(mx, 16));
        mx = fmaxf(mx, __shfl_xor(mx, 32));           // finite: position 0 is live for every token
        const float al = __builtin_amdgcn_exp2f(m - mx);
        if (__any(mx > m)) {
            l *= al;
#pragma unroll
            for (int d = 0; d < 16; d++)
#pragma unroll
                for (int i = 0; i < 4; i++) O[d][i] *= al;
        }
        m = mx;
        v8b ph, pl;
#pragma unroll
        for (int j = 0; j < 8; j++) {
            const float e = __builtin_amdgcn_exp2f(p[j] - mx);
            l += e;
            ph[j] = (__bf16)e;
            pl[j] = (__bf16)(e - (float)ph[j]);
        }
#pragma unroll
        for (int d = 0; d < 16; d++) {
            const v8b vh = *(const v8b *)(Vs + (d * 2) * 1024 + l16), vl = *(const v8b *)(Vs + (d * 2 + 1) * 1024 + l16);
            O[d] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vl, ph, O[d], 0, 0, 0);
            O[d] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vh, pl, O[d], 0, 0, 0);
            O[d] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vh, ph, O[d], 0, 0, 0);
        }
        __builtin_amdgcn_s_waitcnt(0x0F70);
        __syncthreads();                              // the next K is in, every wave is done with V
    }
    l += __shfl_xor(l, 16);
    l += __shfl_xor(l, 32);
    if (tok >= a.M) return;
    const float *gate = qr + FA_HD;
    float *o = a.out + (uint64_t)tok * a.ldo + (uint64_t)h * FA_HD;
#pragma unroll
    for (int d = 0; d < 16; d++) {
        const float4 gv = *(const float4 *)(gate + 16 * d + 4 * g);
        *(float4 *)(o + 16 * d + 4 * g) = make_float4((O[d][0] / l) * (1.0f / (1.0f + expf(-gv.x))),
                                                      (O[d][1] / l) * (1.0f / (1.0f + expf(-gv.y))),
                                                      (O[d][2] / l) * (1.0f / (1.0f + expf(-gv.z))),
                                                      (O[d][3] / l) * (1.0f / (1.0f + expf(-gv.w))));
    }
}

static bool al16(const void *p) { return ((uintptr_t)p & 15) == 0; }

extern "C" int qgpu_wide_attn(qgpu_wide *w, const float *q, uint64_t ldq, const float *kcache, const float *vcache,
                              int pos, int n, int n_head, int n_kv, int head_dim, float *out, uint64_t ldo)
{
    int rc = qg::ensure_init();
    if (rc) return rc;
    if (head_dim != FA_HD) return QGPU_E_RANGE;
    if (!w || !q || !kcache || !vcache || !out || n < 1 || pos < 0 || n_kv < 1 || n_head < 1 || n_head % n_kv ||
        n_kv != w->n_kv || pos > w->n_ctx - n || ldq % 4 || ldo % 4 || !al16(q) || !al16(kcache) || !al16(vcache) || !al16(out))
        return QGPU_E_ARG;
    WideAttn a = {};
    a.q = q; a.ldq = ldq; a.P = w->kv; a.out = out; a.ldo = ldo;
    a.n_tile = (uint32_t)(w->n_ctx + FA_TP - 1) / FA_TP;
    a.pos0 = (uint32_t)pos; a.M = (uint32_t)n; a.n_head = (uint32_t)n_head; a.n_kv = (uint32_t)n_kv;
    a.nq = (a.M + FA_TB - 1) / FA_TB;
    const uint32_t live = a.pos0 + a.M;
    hipLaunchKernelGGL(k_wide_kv, dim3((live + FA_TP - 1) / FA_TP, n_kv), dim3(256), 0, qg::stream, kcache, vcache,
                       w->kv, a.n_tile, live, n_kv);
    QG_LAUNCH_CHECK();
    const uint32_t items = (uint32_t)(n_head / n_kv) * a.nq;           // per kv head
    const uint32_t blocks = 8 % n_kv == 0 ? 8 * ((items * n_kv + 7) / 8 + 1) : items * n_kv;
    hipLaunchKernelGGL(k_wide_attn, dim3(blocks), dim3(256), 0, qg::stream, a);
    QG_LAUNCH_CHECK();
    return QGPU_OK;
}

// ---------------------------------------------------------------- Gated DeltaNet
#define GW_HK  128            // head_k_dim = head_v_dim
#define GW_TT  8              // tokens per wave of the conv pass

static __device__ __forceinline__ float silu_g(float v) { return v / (1.0f + expf(-v)); }

struct WideGdn {
    const float *x;           // conv inputs [M][ldx]
    uint64_t ldx;
    const float *cw, *cin;    // taps and window before the first token, [channel][4]
    float *cout;              // window after the last token
    const float *beta, *alpha;
    uint64_t ldba;
    const float *dtb, *sa, *sin;
    float *sout;              // states before the first and after the last token
    float *y;                 // [M][channels]: q (normalised, / sqrt(128)), k (normalised), v
    float *gb, *gd, *gr, *gk; // [head][ldg]: beta, decay and its reciprocal per v-head, k.q per k-head
    float *out;
    uint64_t ldo;
    uint32_t M, ldg;
    int n_k, n_v;
    float eps;
};

// Conv + SiLU of all tokens, the L2 norms of q and k, k.q, and the gates: everything the
// recurrence needs that does not depend on the state.  Wave (8 tokens, head): a k-head's q and k
// channels, or a v-head's channels; the last row of blocks computes the gates.
__global__ __launch_bounds__(256) void k_wide_conv(const WideGdn p)
{
    const int lane = threadIdx.x & 63;
    const uint32_t tt = blockIdx.x * 4 + (threadIdx.x >> 6), t0 = tt * GW_TT;
    const int grp = blockIdx.y;
    const uint32_t chan = (uint32_t)(2 * p.n_k + p.n_v) * GW_HK;
    if (grp == p.n_k + p.n_v) {
        // the gates of a v-head for a group of 8 tokens (tokens past the end, up to the recurrence's step of
        // 32: a step that changes nothing): the decay since the group's start and its reciprocal, or, where
        // that product gets too small to divide by, the token's own decay and 0 for the whole group
        for (uint32_t e = threadIdx.x; e < 4u * p.n_v; e += 256) {
            const uint32_t tg = blockIdx.x * 4 * GW_TT + (e / p.n_v) * GW_TT, h = e % p.n_v;
            float dec[GW_TT], all = 1.0f, D = 1.0f;
#pragma unroll
            for (int u = 0; u < GW_TT; u++) {
                const uint32_t t = tg + u;
                float b = 0.0f;
                dec[u] = 1.0f;
                if (t < p.M) {
                    const float av = p.alpha[t * p.ldba + h] + p.dtb[h];
                    const float sp = av > 30.0f ? av : log1pf(expf(av));
                    dec[u] = expf(p.sa[h] * sp);
                    b = 1.0f / (1.0f + expf(-p.beta[t * p.ldba + h]));
                } else if (h < (uint32_t)p.n_k) {
                    p.gk[(uint64_t)h * p.ldg + t] = 0.0f;
                }
                p.gb[(uint64_t)h * p.ldg + t] = b;
                all *= dec[u];
            }
            const bool one = all > 0x1p-40f && all < 0x1p40f;
#pragma unroll
            for (int u = 0; u < GW_TT; u++) {
                D *= dec[u];
                p.gd[(uint64_t)h * p.ldg + tg + u] = one ? D : dec[u];
                p.gr[(uint64_t)h * p.ldg + tg + u] = one ? 1.0f / D : 0.0f;
            }
        }
        return;
    }
    if (t0 >= p.M) return;
    const uint32_t te = min(t0 + GW_TT, p.M);
    const bool qk = grp < p.n_k;
    const uint32_t c0 = qk ? grp * GW_HK + 2 * lane : (p.n_k + grp) * GW_HK + 2 * lane;   // v-head grp - n_k starts at 2 n_k
    const uint32_t c1 = p.n_k * GW_HK + c0;                                               // its k channels
    float2 w0[4], w1[4];      // window of the three inputs before the token, then the token's
    float4 f0[2], f1[2];
    f0[0] = *(const float4 *)(p.cw + 4 * (uint64_t)c0); f0[1] = *(const float4 *)(p.cw + 4 * (uint64_t)c0 + 4);
    if (qk) { f1[0] = *(const float4 *)(p.cw + 4 * (uint64_t)c1); f1[1] = *(const float4 *)(p.cw + 4 * (uint64_t)c1 + 4); }
    auto hist = [&](int back, uint32_t c) {                  // input `back` tokens before t0
        if (t0 >= (uint32_t)back) return *(const float2 *)(p.x + (uint64_t)(t0 - back) * p.ldx + c);
        const float *s = p.cin + 4 * (uint64_t)c + (4 - back + t0);
        return make_float2(s[0], s[4]);
    };
#pragma unroll
    for (int i = 0; i < 3; i++) {
        w0[i] = hist(3 - i, c0);
        if (qk) w1[i] = hist(3 - i, c1);
    }
    float2 x0[GW_TT], x1[GW_TT];
#pragma unroll
    for (int b = 0; b < GW_TT; b++) {
        const uint32_t t = min(t0 + b, p.M - 1);
        x0[b] = *(const float2 *)(p.x + (uint64_t)t * p.ldx + c0);
        if (qk) x1[b] = *(const float2 *)(p.x + (uint64_t)t * p.ldx + c1);
    }
    const float qscale = 1.0f / sqrtf((float)GW_HK);
#pragma unroll
    for (int b = 0; b < GW_TT; b++) {
        const uint32_t t = t0 + b;
        if (t >= te) break;
        w0[3] = x0[b];
        const float a0 = silu_g(((w0[0].x * f0[0].x + w0[1].x * f0[0].y) + w0[2].x * f0[0].z) + w0[3].x * f0[0].w);
        const float a1 = silu_g(((w0[0].y * f0[1].x + w0[1].y * f0[1].y) + w0[2].y * f0[1].z) + w0[3].y * f0[1].w);
        float *y = p.y + (uint64_t)t * chan;
        if (qk) {
            w1[3] = x1[b];
            const float k0 = silu_g(((w1[0].x * f1[0].x + w1[1].x * f1[0].y) + w1[2].x * f1[0].z) + w1[3].x * f1[0].w);
            const float k1 = silu_g(((w1[0].y * f1[1].x + w1[1].y * f1[1].y) + w1[2].y * f1[1].z) + w1[3].y * f1[1].w);
            const float qn = sqrtf(wave_sum64(fmaf(a1, a1, a0 * a0))), kn = sqrtf(wave_sum64(fmaf(k1, k1, k0 * k0)));
            const float qs = 1.0f / (qn > p.eps ? qn : p.eps) * qscale, ks = 1.0f / (kn > p.eps ? kn : p.eps);
            const float2 qv = make_float2(a0 * qs, a1 * qs), kv = make_float2(k0 * ks, k1 * ks);
            const float kq = wave_sum64(fmaf(qv.y, kv.y, qv.x * kv.x));
            *(float2 *)(y + c0) = qv;
            *(float2 *)(y + c1) = kv;
            if (lane == 0) p.gk[(uint64_t)grp * p.ldg + t] = kq;
        } else {
            *(float2 *)(y + c0) = make_float2(a0, a1);
        }
        if (t + 1 == p.M) {                                  // the window after the last token
            *(float4 *)(p.cout + 4 * (uint64_t)c0) = make_float4(w0[0].x, w0[1].x, w0[2].x, w0[3].x);
            *(float4 *)(p.cout + 4 * (uint64_t)c0 + 4) = make_float4(w0[0].y, w0[1].y, w0[2].y, w0[3].y);
            if (qk) {
                *(float4 *)(p.cout + 4 * (uint64_t)c1) = make_float4(w1[0].x, w1[1].x, w1[2].x, w1[3].x);
                *(float4 *)(p.cout + 4 * (uint64_t)c1 + 4) = make_float4(w1[0].y, w1[1].y, w1[2].y, w1[3].y);
            }
        }
        w0[0] = w0[1]; w0[1] = w0[2]; w0[2] = w0[3];
        if (qk) { w1[0] = w1[1]; w1[1] = w1[2]; w1[2] = w1[3]; }
    }
}

// The delta rule over all tokens, one launch: state rows are independent, so a wave keeps eight of
// them in registers (8 lanes x 16 columns each) from the first token to the last.  Bound by the
// instructions of the chain of M steps at one wave per SIMD (about 95 a step), once the loads are far
// enough ahead: y is larger than an L2, so its latency is over a microsecond, eight steps or more.  q, k,
// v and the gates go to LDS by direct loads, one instruction per token for q and k, four groups of eight
// tokens deep.  The decay is applied once per group: within one the registers hold S / D, D the decay
// since the group's start, so a step is one multiply-add per element.
// Measured at 48 heads, 1992 tokens: 691 us with loads to registers four tokens ahead and the decay in
// every step, 478 us with the LDS ring, 427 us so (464 us with 16 lanes x 8 columns for a pair of rows:
// half the LDS reads, more reduction steps).
// A wave per block spreads the n_v * 16 waves over all compute units; the waves of a head share an
// XCD's L2 where the heads divide the XCDs.
#define GW_U 8                            // tokens per group
#define GW_V    (GW_U * 1024)             // a group in LDS: q and k of each token, then v (8 rows),
#define GW_G    (GW_V + GW_U * 32)        // then the gates (beta, decay, 1 / decay, k.q)
#define GW_RING (GW_G + 256)
__global__ __launch_bounds__(64, 1) void k_wide_recur(const WideGdn p)
{
    __shared__ __attribute__((aligned(16))) uint8_t R0[GW_RING], R1[GW_RING], R2[GW_RING], R3[GW_RING];
    const int lane = threadIdx.x & 63, cc = lane & 7;
    int h = blockIdx.x >> 4, part = blockIdx.x & 15;
    if (p.n_v % 8 == 0) {
        const int i = blockIdx.x >> 3;
        h = (i >> 4) * 8 + (blockIdx.x & 7);
        part = i & 15;
    }
    const int kh = h % p.n_k, j = part * 8 + (lane >> 3);
    const uint32_t chan4 = (uint32_t)(2 * p.n_k + p.n_v) * GW_HK * 4, last = p.M - 1;
    const uint64_t so = ((uint64_t)h * GW_HK + j) * GW_HK + cc * 4;
    float S[16];
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const float4 v = *(const float4 *)(p.sin + so + i * 32);
        S[4 * i] = v.x; S[4 * i + 1] = v.y; S[4 * i + 2] = v.z; S[4 * i + 3] = v.w;
    }
    const __amdgpu_buffer_rsrc_t rsK = __builtin_amdgcn_make_buffer_rsrc((void *)(p.y + kh * GW_HK), 0, 0x7FFFFFFF, 0x00020000);
    const __amdgpu_buffer_rsrc_t rsV = __builtin_amdgcn_make_buffer_rsrc((void *)(p.y + (2 * p.n_k + h) * GW_HK + part * 8), 0, 0x7FFFFFFF, 0x00020000);
    const uint32_t oqk = lane < 32 ? (uint32_t)lane * 16 : (uint32_t)(p.n_k * GW_HK * 4 + (lane - 32) * 16);
    const __amdgpu_buffer_rsrc_t rsG = __builtin_amdgcn_make_buffer_rsrc((void *)p.gb, 0, 0x7FFFFFFF, 0x00020000);
    const uint32_t grow = (lane & 3) * p.n_v + ((lane & 3) == 3 ? kh : h);     // beta, decay, reciprocal, k.q rows
    // tokens past the end load the last one's rows (and gates that leave the state as it is)
    auto load = [&](uint8_t *R, uint32_t t) {
#pragma unroll
        for (int u = 0; u < GW_U; u++)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rsK, (lptr_t)(R + u * 1024), 16, oqk, min(t + u, last) * chan4, 0, 0);
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rsV, (lptr_t)(R + GW_V), 4,
                                                 min(t + (lane >> 3), last) * chan4 + (lane & 7) * 4, 0, 0, 0);
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rsG, (lptr_t)(R + GW_G), 4,
                                                 lane < 4 * GW_U ? (grow * p.ldg + min(t + (lane >> 2), p.ldg - 1)) * 4 : 0x80000000u,
                                                 0, 0, 0);
    };
    // lane cc of a row keeps the group's token cc: one store per group (tokens past the end have an offset
    // past the buffer)
    const __amdgpu_buffer_rsrc_t rsO = __builtin_amdgcn_make_buffer_rsrc((void *)(p.out + (uint64_t)h * GW_HK), 0, 0x7FFFFFFF, 0x00020000);
    const uint32_t ldo4 = (uint32_t)p.ldo * 4, oo = (uint32_t)cc * ldo4 + (uint32_t)j * 4;
    struct Tok { float4 q[4], k[4], gt; float v; };
    auto read = [&](const uint8_t *R, int u) {
        Tok T;
        const uint8_t *r = R + u * 1024 + cc * 16;
#pragma unroll
        for (int i = 0; i < 4; i++) {
            T.k[i] = *(const float4 *)(r + 512 + i * 128);
            T.q[i] = *(const float4 *)(r + i * 128);
        }
        T.v = *(const float *)(R + GW_V + u * 32 + (lane >> 3) * 4);
        T.gt = *(const float4 *)(R + GW_G + u * 16);
        return T;
    };
    // one token: the registers hold S / D before and after (rD = 1 / D); its output
    auto token = [&](const Tok &T, float D, float rD) {
        float q[16], k[16], sk[4], sq[4];
#pragma unroll
        for (int i = 0; i < 4; i++) {
            q[4 * i] = T.q[i].x; q[4 * i + 1] = T.q[i].y; q[4 * i + 2] = T.q[i].z; q[4 * i + 3] = T.q[i].w;
            k[4 * i] = T.k[i].x; k[4 * i + 1] = T.k[i].y; k[4 * i + 2] = T.k[i].z; k[4 * i + 3] = T.k[i].w;
        }
#pragma unroll
        for (int i = 0; i < 4; i++) { sk[i] = S[i] * k[i]; sq[i] = S[i] * q[i]; }
#pragma unroll
        for (int i = 4; i < 16; i++) {
            sk[i & 3] = fmaf(S[i], k[i], sk[i & 3]);
            sq[i & 3] = fmaf(S[i], q[i], sq[i & 3]);
        }
        float a = (sk[0] + sk[1]) + (sk[2] + sk[3]), b = (sq[0] + sq[1]) + (sq[2] + sq[3]);
        a += dpp_mov<0xB1>(a);  b += dpp_mov<0xB1>(b);           // the row's eight lanes
        a += dpp_mov<0x4E>(a);  b += dpp_mov<0x4E>(b);
        a += dpp_mov<0x141>(a); b += dpp_mov<0x141>(b);
        const float d = fmaf(-D, a, T.v) * T.gt.x, c = d * rD;
#pragma unroll
        for (int i = 0; i < 16; i++) S[i] = fmaf(c, k[i], S[i]);
        return fmaf(d, T.gt.w, D * b);
    };
    auto apply = [&](const uint8_t *R, uint32_t t) {
        float out = 0.0f;
        if (__builtin_amdgcn_readfirstlane(__builtin_bit_cast(int, *(const float *)(R + GW_G + 8)))) {
            Tok T[2];
            T[0] = read(R, 0);
#pragma unroll
            for (int u = 0; u < GW_U; u++) {
                if (u + 1 < GW_U) T[(u + 1) & 1] = read(R, u + 1);
                const Tok &x = T[u & 1];
                const float o = token(x, x.gt.y, x.gt.z);
                out = cc == u ? o : out;
                if (u + 1 == GW_U)
#pragma unroll
                    for (int i = 0; i < 16; i++) S[i] *= x.gt.y;
            }
        } else {                                             // the decay token by token
#pragma unroll 1
            for (int u = 0; u < GW_U; u++) {
                const Tok x = read(R, u);
#pragma unroll
                for (int i = 0; i < 16; i++) S[i] *= x.gt.y;
                const float o = token(x, 1.0f, 1.0f);
                out = cc == u ? o : out;
            }
        }
        __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, out), rsO, t + cc < p.M ? oo : 0x80000000u, t * ldo4, 0);
    };
    // a group is in LDS when at most the three groups issued after it (ten loads each) are in flight
#define GW_STEP(RL, RA, T) do { load(RL, (T) + 3 * GW_U); asm volatile("s_waitcnt vmcnt(30)" ::: "memory"); apply(RA, T); } while (0)
    load(R0, 0);
    load(R1, GW_U);
    load(R2, 2 * GW_U);
    for (uint32_t t = 0; t < p.M; t += 4 * GW_U) {
        GW_STEP(R3, R0, t);
        GW_STEP(R0, R1, t + GW_U);
        GW_STEP(R1, R2, t + 2 * GW_U);
        GW_STEP(R2, R3, t + 3 * GW_U);
    }
#undef GW_STEP
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");      // no direct load may land after the block's LDS is given back
#pragma unroll
    for (int i = 0; i < 4; i++)
        *(float4 *)(p.sout + so + i * 32) = make_float4(S[4 * i], S[4 * i + 1], S[4 * i + 2], S[4 * i + 3]);
}

extern "C" int qgpu_wide_gdn(qgpu_wide *w, const float *x, uint64_t ldx, int n, const float *conv_w,
                             const float *conv_in, float *conv_out, const float *beta_raw, const float *alpha_raw,
                             uint64_t ldba, const float *dt_bias, const float *ssm_a, const float *ssm_in,
                             float *ssm_out, int n_k, int n_v, int head_dim, float eps, float *out, uint64_t ldo)
{
    int rc = qg::ensure_init();
    if (rc) return rc;
    if (head_dim != GW_HK) return QGPU_E_RANGE;
    if (!w || !x || !conv_w || !conv_in || !conv_out || !beta_raw || !alpha_raw || !dt_bias || !ssm_a || !ssm_in ||
        !ssm_out || !out || n < 1 || n > w->rows || n_k < 1 || n_v < 1 || n_v % n_k || n_k + 3 * n_v > w->gdn_heads ||
        (2 * n_k + n_v) > w->gdn_chan || ldx % 2 || ldo % 2 || (uint64_t)n * ldo >= (1u << 29) || (uint64_t)n * w->gdn_chan >= (1u << 22) || !al16(x) || !al16(conv_w) || !al16(conv_in) ||
        !al16(conv_out) || !al16(ssm_in) || !al16(ssm_out) || !al16(out))
        return QGPU_E_ARG;
    WideGdn p = {};
    p.x = x; p.ldx = ldx; p.cw = conv_w; p.cin = conv_in; p.cout = conv_out; p.beta = beta_raw; p.alpha = alpha_raw;
    p.ldba = ldba; p.dtb = dt_bias; p.sa = ssm_a; p.sin = ssm_in; p.sout = ssm_out; p.y = w->y;
    p.ldg = (uint32_t)w->rows;
    p.gb = w->gate; p.gd = p.gb + (uint64_t)n_v * p.ldg; p.gr = p.gd + (uint64_t)n_v * p.ldg;
    p.gk = p.gr + (uint64_t)n_v * p.ldg;
    p.out = out; p.ldo = ldo; p.M = (uint32_t)n; p.n_k = n_k; p.n_v = n_v; p.eps = eps;
    hipLaunchKernelGGL(k_wide_conv, dim3((n + 4 * GW_TT - 1) / (4 * GW_TT), n_k + n_v + 1), dim3(256), 0, qg::stream, p);
    QG_LAUNCH_CHECK();
    hipLaunchKernelGGL(k_wide_recur, dim3(n_v * 16), dim3(64), 0, qg::stream, p);
    QG_LAUNCH_CHECK();
    return QGPU_OK;
}
