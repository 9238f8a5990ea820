// Prompt path (gfx950): matrix products over many tokens at once.
//
// The GEMV path reads every weight once per 8 tokens; a prompt of n tokens reads them n/8
// times.  Here a chunk of up to WIDE_ROWS tokens goes through each matrix in one product on
// the half-precision matrix cores, so the weights are read once per 128 tokens (and from the
// caches) and the product, not the weight stream, is the bound.
//
// Precision.  The activations stay 22-bit values: a row times a power of two (its largest
// magnitude in [2^14, 2^15)) is held as hi + lo, two fp16 numbers (x - hi - lo <= 2^-22 |x|, or
// 2^-39 of the row's largest value where lo is subnormal; the GEMV path's digits keep 2^-23 of the
// super-block's largest).  The weights' integer codes (int8 codebook values, 4..6-bit and int8
// quants) are exact in fp16, every product is exact in fp32, and a sub-block's sum meets its scale
// (d x the sub-block's integer scale, fp32) in one fp32 multiply-add per output.
//
// Layout.  Activations: per (16-row tile, 32-column sub-block) 2 KB, one 128-byte line per row: its
// hi parts, then its lo parts, each in four 16-byte groups g of the elements 4g..4g+3 and
// 16+4g..16+4g+3.  Group g of row m is lane g*16 + m's A operand of v_mfma_f32_16x16x32_f16, and its
// order the one in which the packed weight records hold their lanes' dwords (gemv.hip), so a lane's
// nibble dword decodes straight into its B operand.  The direct loads to LDS put the groups in lane order.
//
// Schedule.  A block of 4 waves owns 16*MTL tokens x 256 weight rows (64 per wave: the
// wave decodes its own weights in registers, and the activation tile is shared through LDS).  The
// (tile, super-block) units of a launch are cut into equal contiguous runs, one per resident
// block; a tile that more than one block computes leaves partial sums that k_wide_fix adds in
// block order, so results do not depend on timing.  (Adding them in the block that counts in last
// instead was no faster with two blocks per tile and 1.9x slower with seven: 17408 -> 5120 at 512
// tokens 199 -> 376 us, one block reading what the fix kernel spreads over all units.)
#include "qgpu_internal.h"
#include <new>

typedef _Float16 v8h __attribute__((ext_vector_type(8)));
typedef _Float16 v4h __attribute__((ext_vector_type(4)));
typedef _Float16 v2h __attribute__((ext_vector_type(2)));
typedef float v4f __attribute__((ext_vector_type(4)));
typedef uint32_t u4v __attribute__((ext_vector_type(4)));

#define WIDE_NT    4                    // 16-row weight tiles per wave
#define WIDE_N     (4 * WIDE_NT * 16)   // weight rows per block
#define WIDE_SUB   2048                 // bytes of one (16-row tile, sub-block): hi and lo planes
#define WIDE_MAXG  512                  // blocks of a launch: two per compute unit

struct WideMat {
    const uint8_t *W;
    float *out;
    uint64_t ldo;
    uint32_t rows, nt16, tile0;         // weight rows, their 16-row tiles, first 256-row tile in the launch
};
struct WideArgs {
    WideMat m[QGPU_MAX_MULTI];
    int n_mat, accum, pair;             // pair: m[0] and m[1] are a gate and its up projection (WIDE_PAIR)
    uint32_t nsb, M, mblk, G, U;        // super-blocks, tokens, token blocks, blocks, units
    const uint8_t *A, *S;
    const float *xs;
    float *piece;
};

// block that computes unit u
static __host__ __device__ __forceinline__ uint32_t unit_block(uint32_t u, uint32_t G, uint32_t U)
{
    return (uint32_t)((((uint64_t)u + 1) * G - 1) / U);
}

static __device__ __forceinline__ float h2f(uint32_t h16) { return (float)__builtin_bit_cast(_Float16, (unsigned short)h16); }
static __device__ __forceinline__ float silu_w(float v) { return v / (1.0f + expf(-v)); }
static __device__ __forceinline__ uint32_t u4_get(uint4 v, int i) { return i == 0 ? v.x : i == 1 ? v.y : i == 2 ? v.z : v.w; }

// four unsigned bytes u -> four fp16 values u - 128 (0x6400 | u is 1024 + u; the sum is exact), two per dword
static __device__ __forceinline__ void bytes_h4(uint32_t u, float bias, uint32_t &d0, uint32_t &d1)
{
    const v2h b = { (_Float16)bias, (_Float16)bias };
    d0 = __builtin_bit_cast(uint32_t, __builtin_bit_cast(v2h, __builtin_amdgcn_perm(0x64646464u, u, 0x04010400u)) + b);
    d1 = __builtin_bit_cast(uint32_t, __builtin_bit_cast(v2h, __builtin_amdgcn_perm(0x64646464u, u, 0x04030402u)) + b);
}
static __device__ __forceinline__ v8h pack_h8(uint32_t lo, uint32_t hi, float bias)
{
    uint4 r;
    bytes_h4(lo, bias, r.x, r.y);
    bytes_h4(hi, bias, r.z, r.w);
    return __builtin_bit_cast(v8h, r);
}
// bit c (c < 4) of x to bit 0 of byte c
static __device__ __forceinline__ uint32_t spread4(uint32_t x) { return (x * 0x00204081u) & 0x01010101u; }

// ---------------------------------------------------------------- weight records
// One lane's slice of a 16-row record, by halves of four sub-blocks: hdr() loads what the whole
// super-block shares, half() the quants of one half; code(ib) decodes a sub-block's eight elements
// to fp16 integers and scale(ib) gives its fp32 factor.  Loads go through a buffer resource at the
// wave's first tile: a scalar offset per record, one vector offset for all of them.
typedef __amdgpu_buffer_rsrc_t rsrc_t;
static __device__ __forceinline__ uint4 ld128(rsrc_t rs, uint32_t vo, uint32_t so)
{
    return __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(rs, vo, so, 0));
}
static __device__ __forceinline__ uint2 ld64(rsrc_t rs, uint32_t vo, uint32_t so)
{
    return __builtin_bit_cast(uint2, __builtin_amdgcn_raw_buffer_load_b64(rs, vo, so, 0));
}
template <int FMT> struct WideW;

template <> struct WideW<T_IQ4_XS> {
    uint2 h;
    uint4 q;
    __device__ __forceinline__ void hdr(rsrc_t rs, uint32_t so, uint32_t l16) { h = ld64(rs, (l16 & 240) >> 1, so); }
    __device__ __forceinline__ void half(rsrc_t rs, uint32_t so, uint32_t l16, int hf)
    {
        q = ld128(rs, l16 + IQ4_HDR_BYTES + hf * 1024, so);
    }
    // codebook + 128 as one byte: two 8-entry v_perm_b32 tables indexed by the whole nibble, whose
    // out-of-range selectors give 0x00 or 0xFF and are undone in the other table (xor)
    __device__ __forceinline__ v8h code(int ib) const
    {
        const uint32_t d = u4_get(q, ib & 3), lo = d & 0x0F0F0F0Fu, hi = (d >> 4) & 0x0F0F0F0Fu;
        const uint32_t ul = __builtin_amdgcn_perm(0x8995A24Fu, 0x3F2D18FEu, lo) ^
                            __builtin_amdgcn_perm(0x0E263AB5u, 0x59668D81u, lo ^ 0x08080808u);
        const uint32_t uh = __builtin_amdgcn_perm(0x8995A24Fu, 0x3F2D18FEu, hi) ^
                            __builtin_amdgcn_perm(0x0E263AB5u, 0x59668D81u, hi ^ 0x08080808u);
        return pack_h8(ul, uh, -1152.0f);
    }
    __device__ __forceinline__ float scale(int ib) const
    {
        uint32_t s;
        if (ib < 5) s = h.y >> (6 * ib);
        else if (ib < 7) s = h.x >> (16 + 6 * (ib - 5));
        else s = (h.x >> 28) | ((h.y >> 30) << 4);
        return h2f(h.x & 0xFFFFu) * (float)(((int)(s << 26)) >> 26);
    }
};

static __device__ __forceinline__ uint32_t kq_sc(uint4 h, int ib)
{
    return ib < 5 ? (h.y >> (6 * ib)) & 63u : (h.w >> (6 * (ib - 5))) & 63u;
}
static __device__ __forceinline__ uint32_t kq_m(uint4 h, int ib)
{
    if (ib < 5) return (h.z >> (6 * ib)) & 63u;
    if (ib < 7) return (h.w >> (18 + 6 * (ib - 5))) & 63u;
    return (h.y >> 30) | ((h.z >> 30) << 2) | ((h.w >> 30) << 4);
}
template <> struct WideW<T_Q4_K> {
    uint4 h, q;
    __device__ __forceinline__ void hdr(rsrc_t rs, uint32_t so, uint32_t l16) { h = ld128(rs, l16 & 240, so); }
    __device__ __forceinline__ void half(rsrc_t rs, uint32_t so, uint32_t l16, int hf)
    {
        q = ld128(rs, l16 + 256 + hf * 1024, so);
    }
    __device__ __forceinline__ v8h code(int ib) const
    {
        const uint32_t d = u4_get(q, ib & 3);
        return pack_h8(d & 0x0F0F0F0Fu, (d >> 4) & 0x0F0F0F0Fu, -1024.0f);
    }
    __device__ __forceinline__ float scale(int ib) const { return h2f(h.x & 0xFFFFu) * (float)kq_sc(h, ib); }
};
template <> struct WideW<T_Q5_K> {
    uint4 h, q;
    uint32_t hb;
    __device__ __forceinline__ void hdr(rsrc_t rs, uint32_t so, uint32_t l16) { h = ld128(rs, l16 & 240, so); }
    __device__ __forceinline__ void half(rsrc_t rs, uint32_t so, uint32_t l16, int hf)
    {
        q = ld128(rs, l16 + 256 + hf * 1024, so);
        hb = (uint32_t)__builtin_amdgcn_raw_buffer_load_b32(rs, (l16 >> 1) + 2304 + hf * 4, so, 0);
    }
    __device__ __forceinline__ v8h code(int ib) const
    {
        const uint32_t d = u4_get(q, ib & 3), b = (hb >> (8 * (ib & 3))) & 0xFFu;
        return pack_h8((d & 0x0F0F0F0Fu) | (spread4(b & 15u) << 4), ((d >> 4) & 0x0F0F0F0Fu) | (spread4(b >> 4) << 4),
                       -1024.0f);
    }
    __device__ __forceinline__ float scale(int ib) const { return h2f(h.x & 0xFFFFu) * (float)kq_sc(h, ib); }
};
template <> struct WideW<T_Q6_K> {
    uint4 h, q;
    uint2 hb;
    float d;
    __device__ __forceinline__ void hdr(rsrc_t rs, uint32_t so, uint32_t l16)
    {
        h = ld128(rs, l16 & 240, so);
        d = h2f((uint16_t)__builtin_amdgcn_raw_buffer_load_b16(rs, 256 + ((l16 & 240) >> 3), so, 0));
    }
    __device__ __forceinline__ void half(rsrc_t rs, uint32_t so, uint32_t l16, int hf)
    {
        q = ld128(rs, l16 + 288 + hf * 1024, so);
        hb = ld64(rs, l16 + 2336 + hf * 8, so);
    }
    __device__ __forceinline__ v8h code(int ib) const
    {
        const uint32_t v = u4_get(q, ib & 3), t = ((ib & 2) ? hb.y : hb.x) >> (4 * (ib & 1));
        return pack_h8((v & 0x0F0F0F0Fu) | ((t << 4) & 0x30303030u), ((v >> 4) & 0x0F0F0F0Fu) | ((t << 2) & 0x30303030u),
                       -1056.0f);
    }
    // elements 0..15 (u = 0) and 16..31 (u = 1) of the sub-block
    __device__ __forceinline__ float scale16(int ib, int u) const
    {
        return d * (float)(int)(int8_t)(u4_get(h, ib >> 1) >> (16 * (ib & 1) + 8 * u));
    }
};
template <> struct WideW<T_Q8_0> {
    uint4 h, q[2];
    __device__ __forceinline__ void hdr(rsrc_t rs, uint32_t so, uint32_t l16) { h = ld128(rs, l16 & 240, so); }
    __device__ __forceinline__ void half(rsrc_t rs, uint32_t so, uint32_t l16, int hf)
    {
        q[0] = ld128(rs, l16 + 256 + hf * 2048, so);
        q[1] = ld128(rs, l16 + 256 + hf * 2048 + 1024, so);
    }
    __device__ __forceinline__ v8h code(int ib) const
    {
        const uint4 v = q[(ib >> 1) & 1];
        const uint32_t lo = (ib & 1) ? v.z : v.x, hi = (ib & 1) ? v.w : v.y;
        return pack_h8(lo ^ 0x80808080u, hi ^ 0x80808080u, -1152.0f);
    }
    __device__ __forceinline__ float scale(int ib) const { return h2f((u4_get(h, ib >> 1) >> (16 * (ib & 1))) & 0xFFFFu); }
};

// ---------------------------------------------------------------- the product
typedef const __attribute__((address_space(1))) void *gptr_t;
typedef __attribute__((address_space(3))) void *lptr_t;

// Stage: two sub-blocks of the block's activation tile (MTL * 4 KB), brought into one of two LDS
// buffers by direct loads while the other is used; one barrier per stage.  Bound by the matrix cores
// (55% of their cycles at 1992 tokens) beside the multiply-adds and decoding on the vector units (49%).
// Loads take scalar offsets from buffer resources, the next quants the registers of the ones just
// decoded, and a row tile's multiply-adds run beside the next tile's products: 256 registers hold it, two
// waves per SIMD.  Power bounds it too: with zero activations the same cycles take 1.10 ms instead of 1.40.
// (v_mfma_f32_32x32x16_f16 halves the header and scale work: 6% less time for a 33-token prompt, 3% more for
// 1999 tokens.)  5120 -> 34816 at 1992 / 256 tokens 1537 / 231 -> 1440 / 208 us, 17408 -> 5120 765 /
// 140 -> 708 / 133 us, against per-lane addresses, copies of the next quants and no such overlap.
template <int FMT, int MTL>
__global__ __launch_bounds__(256, 2) void k_wide_gemm(const WideArgs a)
{
    constexpr bool MIN = FMT == T_Q4_K || FMT == T_Q5_K;
    constexpr uint32_t REC = packed_rec_bytes(FMT);
    __shared__ __attribute__((aligned(16))) uint8_t As0[MTL * 2 * WIDE_SUB], As1[MTL * 2 * WIDE_SUB];
    __shared__ __attribute__((aligned(16))) uint8_t Ss[MIN ? MTL * 1024 : 16];
    const int lane = threadIdx.x & 63, n = lane & 15;
    const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    // neighbouring runs of units share activations and weights: give each XCD (block index mod 8) a
    // contiguous range of them
    const uint32_t g = a.G % 8 == 0 ? (blockIdx.x & 7) * (a.G / 8) + (blockIdx.x >> 3) : blockIdx.x;
    uint32_t u = (uint32_t)((uint64_t)g * a.U / a.G);
    const uint32_t ue = (uint32_t)((uint64_t)(g + 1) * a.U / a.G);
    const uint64_t nsub = (uint64_t)a.nsb * 8;
    const uint32_t l16 = (uint32_t)lane * 16;
    // lane g*16 + m fetches part g of row m: rows lie in memory one after the other, operands lane by lane in LDS
    const uint32_t va = (uint32_t)n * 128 + (uint32_t)(lane >> 4) * 16, vs = (uint32_t)n * 64 + (uint32_t)(lane >> 4) * 16;
    const v4f z4 = { 0.0f, 0.0f, 0.0f, 0.0f };
    while (u < ue) {
        const uint32_t tile = u / a.nsb, sb0 = u - tile * a.nsb, sb1 = min(a.nsb, sb0 + (ue - u));
        const uint32_t nt = tile / a.mblk, mb = tile - nt * a.mblk;
        int j = 0;
        while (!a.pair && j + 1 < a.n_mat && nt >= a.m[j + 1].tile0) j++;
        // this wave's first weight row; a pair's block holds 128 rows of each matrix, tiles 0, 1 of a wave the gate's
        const uint32_t row0 = (nt - a.m[j].tile0) * (a.pair ? WIDE_N / 2 : WIDE_N) + wv * (a.pair ? WIDE_NT * 8 : WIDE_NT * 16);
        // its records: past the matrix's end any loadable one (the results are dropped)
        const uint32_t tstr = a.nsb * REC, t0 = min(row0 / 16, a.m[j].nt16 - 1);
        const rsrc_t rsW = __builtin_amdgcn_make_buffer_rsrc((void *)(a.m[j].W + (uint64_t)t0 * tstr), 0, 0x7FFFFFFF, 0x00020000);
        const rsrc_t rsU = __builtin_amdgcn_make_buffer_rsrc((void *)((a.pair ? a.m[1].W : a.m[j].W) + (uint64_t)t0 * tstr), 0, 0x7FFFFFFF, 0x00020000);
        uint32_t rec[WIDE_NT];
#pragma unroll
        for (int t = 0; t < WIDE_NT; t++)
            rec[t] = min((uint32_t)(a.pair ? t % (WIDE_NT / 2) : t), a.m[j].nt16 - 1 - t0) * tstr + sb0 * REC;
#define RSW(t) ((t) < WIDE_NT / 2 ? rsW : rsU)
        v4f acc[MTL][WIDE_NT];
#pragma unroll
        for (int mt = 0; mt < MTL; mt++)
#pragma unroll
            for (int t = 0; t < WIDE_NT; t++) acc[mt][t] = z4;
        // this wave's MTL 1 KB chunks of a stage: chunk c = (row tile c / 4, sub-block c % 4 / 2, plane c % 2)
        const rsrc_t rsA = __builtin_amdgcn_make_buffer_rsrc(
            (void *)(a.A + ((uint64_t)mb * MTL * nsub + (uint64_t)sb0 * 8) * WIDE_SUB), 0, 0x7FFFFFFF, 0x00020000);
        auto stage = [&](uint32_t s, uint8_t *buf) {
#pragma unroll
            for (int i = 0; i < MTL; i++) {
                const int c = wv * MTL + i;
                __builtin_amdgcn_raw_ptr_buffer_load_lds(
                    rsA, (lptr_t)(buf + c * 1024), 16, va,
                    ((c >> 2) * (uint32_t)nsub + 2 * s) * WIDE_SUB + ((c >> 1) & 1) * WIDE_SUB + (c & 1) * 64, 0, 0);
            }
        };
        WideW<FMT> w[WIDE_NT];
        stage(0, As0);
#pragma unroll
        for (int t = 0; t < WIDE_NT; t++) { w[t].hdr(RSW(t), rec[t], l16); w[t].half(RSW(t), rec[t], l16, 0); }
        __builtin_amdgcn_s_waitcnt(0x0F70);          // vmcnt(0): the direct loads are in LDS
        __syncthreads();
        const uint32_t ns = (sb1 - sb0) * 4;
        for (uint32_t sb = sb0; sb < sb1; sb++) {
            const uint32_t step = sb + 1 < sb1 ? REC : 0;
#pragma unroll
            for (int q = 0; q < 4; q++) {
                const uint32_t s = (sb - sb0) * 4 + q;
                uint8_t *cur = (q & 1) ? As1 : As0, *nxt = (q & 1) ? As0 : As1;
                stage(min(s + 1, ns - 1), nxt);              // (the last stage again at the end: no branch)
                if (MIN && q == 2) {
#pragma unroll
                    for (int i = 0; i < (MTL + 3) / 4; i++) {
                        const int c = wv + 4 * i;
                        if (c < MTL)
                            __builtin_amdgcn_global_load_lds(
                                (gptr_t)(a.S + (((uint64_t)mb * MTL + c) * a.nsb + sb) * 1024 + vs),
                                (lptr_t)(Ss + c * 1024), 16, 0, 0);
                    }
                }
                if constexpr (MIN) {
                    if (q == 3) {
                        // minus dmin * sum_ib m_ib (sum of sub-block ib): the sums, split in three fp16
                        // parts (K-slots 8p + ib), times the integer mins
#pragma unroll
                        for (int t = 0; t < WIDE_NT; t++) {
                            v8h mb8;
#pragma unroll
                            for (int ib = 0; ib < 8; ib++) mb8[ib] = (_Float16)(float)kq_m(w[t].h, ib);
                            const float dm = -32.0f * h2f(w[t].h.x >> 16);
#pragma unroll
                            for (int mt = 0; mt < MTL; mt++) {
                                const v8h sf = *(const v8h *)(Ss + mt * 1024 + l16);
                                const v4f d = __builtin_amdgcn_mfma_f32_16x16x32_f16(sf, mb8, z4, 0, 0, 0);
#pragma unroll
                                for (int i = 0; i < 4; i++) acc[mt][t][i] = fmaf(d[i], dm, acc[mt][t][i]);
                                asm volatile("" : "+v"(acc[mt][t]));
                            }
                        }
                    }
                }
#pragma unroll
                for (int sub = 0; sub < 2; sub++) {
                    const int ib = 2 * q + sub;
                    v8h B[WIDE_NT];
                    float dl[WIDE_NT], dl2[WIDE_NT];
#pragma unroll
                    for (int t = 0; t < WIDE_NT; t++) {
                        B[t] = w[t].code(ib);
                        if constexpr (FMT == T_Q6_K) { dl[t] = w[t].scale16(ib, 0); dl2[t] = w[t].scale16(ib, 1); }
                        else dl[t] = w[t].scale(ib);
                    }
                    // the last decode of a half: its registers take the next half's quants (and header), in
                    // flight during this sub-block's products
                    if (sub == 1 && q == 1) {
#pragma unroll
                        for (int t = 0; t < WIDE_NT; t++) w[t].half(RSW(t), rec[t], l16, 1);
                    }
                    if (sub == 1 && q == 3) {
#pragma unroll
                        for (int t = 0; t < WIDE_NT; t++) {
                            rec[t] += step;
                            w[t].hdr(RSW(t), rec[t], l16);
                            w[t].half(RSW(t), rec[t], l16, 0);
                        }
                    }
                    // products of row tile mt beside the multiply-adds of tile mt - 1 and the operand reads of mt + 1
                    v8h ah[2], al[2];
                    v4f d[2][WIDE_NT], e[2][WIDE_NT];
                    const uint8_t *ap = cur + sub * WIDE_SUB + l16;
                    al[0] = *(const v8h *)(ap + 1024);
                    ah[0] = *(const v8h *)ap;
#pragma unroll
                    for (int mt = 0; mt <= MTL; mt++) {
                        const int x = mt & 1, y = x ^ 1;
                        if (mt + 1 < MTL) {
                            al[y] = *(const v8h *)(ap + (mt + 1) * 2 * WIDE_SUB + 1024);
                            ah[y] = *(const v8h *)(ap + (mt + 1) * 2 * WIDE_SUB);
                        }
                        if (mt < MTL) {
                            if constexpr (FMT == T_Q6_K) {
                                const v4h al0 = { al[x][0], al[x][1], al[x][2], al[x][3] }, al1 = { al[x][4], al[x][5], al[x][6], al[x][7] };
                                const v4h ah0 = { ah[x][0], ah[x][1], ah[x][2], ah[x][3] }, ah1 = { ah[x][4], ah[x][5], ah[x][6], ah[x][7] };
#pragma unroll
                                for (int t = 0; t < WIDE_NT; t++) {
                                    const v4h b0 = { B[t][0], B[t][1], B[t][2], B[t][3] }, b1 = { B[t][4], B[t][5], B[t][6], B[t][7] };
                                    d[x][t] = __builtin_amdgcn_mfma_f32_16x16x16f16(al0, b0, z4, 0, 0, 0);
                                    e[x][t] = __builtin_amdgcn_mfma_f32_16x16x16f16(al1, b1, z4, 0, 0, 0);
                                    d[x][t] = __builtin_amdgcn_mfma_f32_16x16x16f16(ah0, b0, d[x][t], 0, 0, 0);
                                    e[x][t] = __builtin_amdgcn_mfma_f32_16x16x16f16(ah1, b1, e[x][t], 0, 0, 0);
                                }
                            } else {
#pragma unroll
                                for (int t = 0; t < WIDE_NT; t++) d[x][t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(al[x], B[t], z4, 0, 0, 0);
#pragma unroll
                                for (int t = 0; t < WIDE_NT; t++) d[x][t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(ah[x], B[t], d[x][t], 0, 0, 0);
                            }
                        }
                        if (mt > 0) {
#pragma unroll
                            for (int t = 0; t < WIDE_NT; t++)
#pragma unroll
                                for (int i = 0; i < 4; i++)
                                    acc[mt - 1][t][i] = FMT == T_Q6_K
                                        ? fmaf(d[y][t][i], dl[t], fmaf(e[y][t][i], dl2[t], acc[mt - 1][t][i]))
                                        : fmaf(d[y][t][i], dl[t], acc[mt - 1][t][i]);
                            // (they are otherwise moved to the end of the loop body, and the products spilled until then)
#pragma unroll
                            for (int t = 0; t < WIDE_NT; t++) asm volatile("" : "+v"(acc[mt - 1][t]));
                        }
                    }
                }
                __builtin_amdgcn_s_waitcnt(0x0F70);
                __syncthreads();
            }
        }
        // ---- a tile shared between blocks: partial sums, in register order, for k_wide_fix
        if (sb1 - sb0 != a.nsb) {
            constexpr uint32_t PB = MTL * 16 * WIDE_N * 4;                       // bytes of a piece
            const uint32_t pv = threadIdx.x * 16;
            {
                const rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc((char *)a.piece + (uint64_t)(2 * g + (sb0 == 0)) * PB, 0, PB, 0x00020000);
#pragma unroll
                for (int mt = 0; mt < MTL; mt++)
#pragma unroll
                    for (int t = 0; t < WIDE_NT; t++)
                        __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u4v, acc[mt][t]), rs, pv, (mt * WIDE_NT + t) * 4096, 0);
            }
            u += sb1 - sb0;
            continue;
        }
        // ---- results: lane (g, n), register i: token 16 mt + 4 g + i, weight row 16 t + n
        const uint32_t g4 = 4 * (uint32_t)(lane >> 4);
#pragma unroll
        for (int mt = 0; mt < MTL; mt++) {
            const uint32_t r0 = (mb * MTL + mt) * 16 + g4;
            const float4 x4 = *(const float4 *)(a.xs + r0);
            const float xr[4] = { x4.x, x4.y, x4.z, x4.w };
            if (a.pair) {                                    // silu(gate) * up: tiles t and t + 2
#pragma unroll
                for (int t = 0; t < WIDE_NT / 2; t++) {
                    const uint32_t c = row0 + 16 * t + n;
#pragma unroll
                    for (int i = 0; i < 4; i++)
                        if (r0 + i < a.M && c < a.m[0].rows)
                            a.m[0].out[(uint64_t)(r0 + i) * a.m[0].ldo + c] =
                                silu_w(acc[mt][t][i] * xr[i]) * (acc[mt][t + WIDE_NT / 2][i] * xr[i]);
                }
                continue;
            }
#pragma unroll
            for (int t = 0; t < WIDE_NT; t++) {
                const uint32_t c = row0 + 16 * t + n;
#pragma unroll
                for (int i = 0; i < 4; i++)
                    if (r0 + i < a.M && c < a.m[j].rows) {
                        float *o = a.m[j].out + (uint64_t)(r0 + i) * a.m[j].ldo + c;
                        const float v = acc[mt][t][i] * xr[i];
                        *o = a.accum ? *o + v : v;
                    }
            }
        }
        u += sb1 - sb0;
    }
}

// Adds the pieces of the tiles that several blocks computed, in block order: block (tile, row tile mt, weight
// tile t; with a pair, both its halves), the product kernel's lanes and registers, so pieces are written and
// read in whole lines, eight at a time: a narrow output of few tokens has up to 26 pieces a tile and few
// tiles, and is bound by the latency of reading them (all four weight tiles in a block, four pieces at a time:
// a 33-token prompt 2.51 ms, so 2.37; 129 tokens 3.96 -> 3.86).  A block's last piece starts at its tile's first
// unit (slot 1), its first one does not (slot 0).
template <int MTL>
__global__ __launch_bounds__(256) void k_wide_fix(const WideArgs a)
{
    const uint32_t tile = blockIdx.x, mt = blockIdx.y, tz = blockIdx.z, u0 = tile * a.nsb;
    const uint32_t ga = unit_block(u0, a.G, a.U), gb = unit_block(u0 + a.nsb - 1, a.G, a.U);
    if (ga == gb) return;
    const uint32_t nt = tile / a.mblk, mb = tile - nt * a.mblk, wv = threadIdx.x >> 6, n = threadIdx.x & 15;
    const uint32_t r0 = (mb * MTL + mt) * 16 + 4 * ((threadIdx.x >> 4) & 3);
    if ((mb * MTL + mt) * 16 >= a.M) return;
    constexpr uint64_t PS = MTL * 16 * WIDE_N;
    auto sum = [&](uint32_t t) {
        const float *P = a.piece + (mt * WIDE_NT + t) * 1024 + threadIdx.x * 4;
        v4f s = *(const v4f *)(P + (uint64_t)(2 * ga + 1) * PS);
        for (uint32_t q = ga + 1; q <= gb; q += 8) {
            v4f v[8];
#pragma unroll
            for (int k = 0; k < 8; k++) v[k] = *(const v4f *)(P + (uint64_t)(2 * min(q + k, gb)) * PS);
#pragma unroll
            for (int k = 0; k < 8; k++)
                if (q + k <= gb) s += v[k];
        }
        return s;
    };
    const float4 x4 = *(const float4 *)(a.xs + r0);
    const float xr[4] = { x4.x, x4.y, x4.z, x4.w };
    const v4f s = sum(tz);
    if (a.pair) {
        const v4f up = sum(tz + WIDE_NT / 2);
        const uint32_t c = nt * (WIDE_N / 2) + wv * (WIDE_NT * 8) + 16 * tz + n;
#pragma unroll
        for (int i = 0; i < 4; i++)
            if (r0 + i < a.M && c < a.m[0].rows)
                a.m[0].out[(uint64_t)(r0 + i) * a.m[0].ldo + c] = silu_w(s[i] * xr[i]) * (up[i] * xr[i]);
        return;
    }
    int j = 0;
    while (j + 1 < a.n_mat && nt >= a.m[j + 1].tile0) j++;
    const uint32_t c = (nt - a.m[j].tile0) * WIDE_N + wv * (WIDE_NT * 16) + 16 * tz + n;
#pragma unroll
    for (int i = 0; i < 4; i++)
        if (r0 + i < a.M && c < a.m[j].rows) {
            float *o = a.m[j].out + (uint64_t)(r0 + i) * a.m[j].ldo + c;
            const float v = s[i] * xr[i];
            *o = a.accum ? *o + v : v;
        }
}

// ---------------------------------------------------------------- activation preparation
struct WidePrep {
    const float *x, *y, *w, *w2;
    uint64_t ldx, ldy;
    uint32_t M, ne0, seg;               // tokens, columns, segment length (two-segment RMSNorm)
    float eps;
    uint8_t *A, *S;                     // S: NULL when no matrix needs the sums
    float *xs;
};
#define WP_CAT 4                        // internal kind: the two-segment RMSNorm

// One token per block of NTH threads; a thread holds GPT groups of eight elements, each one lane's
// share of a sub-block (4g..4g+3 and 16+4g..16+4g+3), so the row is read once and the planes
// are written from registers: a sub-block's hi and lo parts are one 128-byte line.  Bound by memory
// traffic in two phases, read then write: 3.4 TB/s at 1992 tokens x 17408 (81 us; 111 us with 256 threads
// a row and 16-byte parts 256 bytes apart).
template <int KIND, int GPT, int NTH>
__global__ __launch_bounds__(NTH) void k_wide_prep(const WidePrep p)
{
    __shared__ float red[3][NTH / 64];
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
    const uint32_t r = blockIdx.x;
    const uint32_t ng = p.ne0 / 8;
    float v[GPT][8];
    float s0 = 0.0f, s1 = 0.0f, mx = 0.0f;
    const float *x = p.x + (uint64_t)r * p.ldx;
    const float *y = KIND == QGPU_ACT_SILU_MUL || KIND == QGPU_ACT_GATED_NORM || KIND == WP_CAT ? p.y + (uint64_t)r * p.ldy : nullptr;
#pragma unroll
    for (int i = 0; i < GPT; i++) {
        const uint32_t q = tid + i * NTH, k0 = (q >> 2) * 32 + 4 * (q & 3);
        const bool live = q < ng;
        const bool s2 = KIND == WP_CAT && k0 >= p.seg;
        const float *src = s2 ? y + (k0 - p.seg) : x + k0;
        const float4 z = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        const float4 a0 = live ? *(const float4 *)src : z, a1 = live ? *(const float4 *)(src + 16) : z;
        float e[8] = { a0.x, a0.y, a0.z, a0.w, a1.x, a1.y, a1.z, a1.w };
        float f[8] = { 0, 0, 0, 0, 0, 0, 0, 0 };
        if (KIND != QGPU_ACT_COPY) {
            const float *fp = KIND == QGPU_ACT_SILU_MUL ? y + k0 : KIND == QGPU_ACT_GATED_NORM ? p.w + (k0 & 127) :
                              s2 ? p.w2 + (k0 - p.seg) : p.w + k0;
            const float4 f0 = live ? *(const float4 *)fp : z, f1 = live ? *(const float4 *)(fp + 16) : z;
            f[0] = f0.x; f[1] = f0.y; f[2] = f0.z; f[3] = f0.w; f[4] = f1.x; f[5] = f1.y; f[6] = f1.z; f[7] = f1.w;
        }
        if (KIND == QGPU_ACT_RMSNORM || KIND == WP_CAT) {
            float ss = 0.0f;
#pragma unroll
            for (int c = 0; c < 8; c++) { ss = fmaf(e[c], e[c], ss); v[i][c] = e[c]; }
            if (s2) s1 += ss; else s0 += ss;
        } else if (KIND == QGPU_ACT_SILU_MUL) {
#pragma unroll
            for (int c = 0; c < 8; c++) v[i][c] = silu_w(e[c]) * f[c];
        } else if (KIND == QGPU_ACT_GATED_NORM) {
            // a head of 128 elements is 16 neighbouring lanes
            float ss = 0.0f;
#pragma unroll
            for (int c = 0; c < 8; c++) ss = fmaf(e[c], e[c], ss);
            const float sc = 1.0f / sqrtf(rowsum16(ss) / 128.0f + p.eps);
            const float4 g0 = live ? *(const float4 *)(y + k0) : z, g1 = live ? *(const float4 *)(y + k0 + 16) : z;
            const float gy[8] = { g0.x, g0.y, g0.z, g0.w, g1.x, g1.y, g1.z, g1.w };
#pragma unroll
            for (int c = 0; c < 8; c++) v[i][c] = ((e[c] * sc) * f[c]) * silu_w(gy[c]);
        } else {
#pragma unroll
            for (int c = 0; c < 8; c++) v[i][c] = e[c];
        }
    }
    float sc0 = 1.0f, sc1 = 1.0f;
    if (KIND == QGPU_ACT_RMSNORM || KIND == WP_CAT) {
        s0 = wave_sum64(s0);
        if (KIND == WP_CAT) s1 = wave_sum64(s1);
        if (lane == 0) { red[0][wv] = s0; red[1][wv] = s1; }
        __syncthreads();
        float t0 = 0.0f, t1 = 0.0f;
#pragma unroll
        for (int i = 0; i < NTH / 64; i++) { t0 += red[0][i]; t1 += red[1][i]; }
        const float nrm = (float)p.seg;
        sc0 = 1.0f / sqrtf(t0 / nrm + p.eps);
        if (KIND == WP_CAT) sc1 = 1.0f / sqrtf(t1 / nrm + p.eps);
#pragma unroll
        for (int i = 0; i < GPT; i++) {
            const uint32_t q = tid + i * NTH, k0 = (q >> 2) * 32 + 4 * (q & 3);
            const bool s2 = KIND == WP_CAT && k0 >= p.seg;
            const float *fp = s2 ? p.w2 + (k0 - p.seg) : p.w + k0;
            if (q < ng) {
                const float4 f0 = *(const float4 *)fp, f1 = *(const float4 *)(fp + 16);
                const float f[8] = { f0.x, f0.y, f0.z, f0.w, f1.x, f1.y, f1.z, f1.w };
                const float sc = s2 ? sc1 : sc0;
#pragma unroll
                for (int c = 0; c < 8; c++) v[i][c] = (v[i][c] * sc) * f[c];
            }
        }
    }
#pragma unroll
    for (int i = 0; i < GPT; i++)
#pragma unroll
        for (int c = 0; c < 8; c++) mx = fmaxf(mx, fabsf(v[i][c]));
    mx = wave_max64(mx);
    if (lane == 0) red[2][wv] = mx;
    __syncthreads();
#pragma unroll
    for (int i = 0; i < NTH / 64; i++) mx = fmaxf(mx, red[2][i]);
    // the row's power of two: its largest magnitude to [2^14, 2^15)
    int sh = 0;
    if (mx > 0.0f && isfinite(mx)) {
        int E;
        frexpf(mx, &E);
        sh = 15 - E;
    }
    if (tid == 0) p.xs[r] = ldexpf(1.0f, -sh);
    const uint64_t nsub = p.ne0 / 32, nsb = p.ne0 / 256;
    uint8_t *At = p.A + (uint64_t)(r >> 4) * nsub * WIDE_SUB + (r & 15) * 128;
    uint8_t *St = p.S + (uint64_t)(r >> 4) * nsb * 1024 + (r & 15) * 64;
#pragma unroll
    for (int i = 0; i < GPT; i++) {
        const uint32_t q = tid + i * NTH, s = q >> 2, g = q & 3;
        v8h hi, lo;
        float sum = 0.0f;
#pragma unroll
        for (int c = 0; c < 8; c++) {
            const float t = ldexpf(v[i][c], sh);
            hi[c] = (_Float16)t;
            lo[c] = (_Float16)(t - (float)hi[c]);
            sum += t;
        }
        // the sub-block's sum (its four lanes) x 2^-5, in three fp16 parts: the K-quants' min term
        sum += dpp_mov<0xB1>(sum);
        sum += dpp_mov<0x4E>(sum);
        sum *= 0.03125f;
        const _Float16 p0 = (_Float16)sum, p1 = (_Float16)(sum - (float)p0);
        const _Float16 p2 = (_Float16)((sum - (float)p0) - (float)p1);
        if (q < ng) {
            *(v8h *)(At + (uint64_t)s * WIDE_SUB + g * 16) = hi;
            *(v8h *)(At + (uint64_t)s * WIDE_SUB + 64 + g * 16) = lo;
            if (p.S && g < 3) *(_Float16 *)(St + (uint64_t)(s >> 3) * 1024 + g * 16 + (s & 7) * 2) = g == 0 ? p0 : g == 1 ? p1 : p2;
        }
    }
}

// ---------------------------------------------------------------- entry points
extern "C" int qgpu_wide_free(qgpu_wide *w)
{
    if (!w) return QGPU_OK;
    if (qg::stream) (void)hipStreamSynchronize(qg::stream);
    (void)hipFree(w->A);
    (void)hipFree(w->S);
    (void)hipFree(w->xs);
    if (w->y != w->piece) (void)hipFree(w->y);
    (void)hipFree(w->piece);
    (void)hipFree(w->kv);
    (void)hipFree(w->gate);
    delete w;
    return QGPU_OK;
}

extern "C" int qgpu_wide_create(int max_rows, uint64_t max_k, int n_ctx, int n_kv, int n_k, int n_v, qgpu_wide **out)
{
    int rc = qg::ensure_init();
    if (rc) return rc;
    if (!out || max_rows < 1 || max_rows > (1 << 20) || !max_k || max_k % 256 || max_k > MAX_K || n_ctx < 0 ||
        n_kv < 0 || n_k < 0 || n_v < 0 || n_k > 256 || n_v > 256)
        return QGPU_E_ARG;
    *out = nullptr;
    qgpu_wide *w = new (std::nothrow) qgpu_wide();
    if (!w) return QGPU_E_ARG;
    w->rows = (max_rows + 127) / 128 * 128;
    w->max_k = max_k;
    const size_t sb = (size_t)w->rows / 16 * (max_k / 256) * 1024, xb = (size_t)w->rows * sizeof(float);
    const size_t pb = (size_t)2 * WIDE_MAXG * 128 * WIDE_N * sizeof(float);
    hipError_t e = hipMalloc((void **)&w->A, (size_t)w->rows * max_k * 4);
    if (e == hipSuccess) e = hipMalloc((void **)&w->S, sb);
    if (e == hipSuccess) e = hipMalloc((void **)&w->xs, xb);
    if (e == hipSuccess) e = hipMalloc((void **)&w->piece, pb);
    w->n_ctx = n_ctx;
    w->n_kv = n_kv;
    if (e == hipSuccess && n_ctx && n_kv) e = hipMalloc((void **)&w->kv, ((size_t)n_ctx + 31) / 32 * n_kv * 65536);
    w->gdn_heads = n_k + 3 * n_v;
    w->gdn_chan = 2 * n_k + n_v;
    // the recurrence's inputs live between two products: in the pieces' memory where they fit
    const size_t yb = (size_t)w->rows * w->gdn_chan * 128 * sizeof(float);
    if (e == hipSuccess && n_k && n_v) {
        if (yb <= pb) w->y = w->piece;
        else e = hipMalloc((void **)&w->y, yb);
    }
    if (e == hipSuccess && n_k && n_v) e = hipMalloc((void **)&w->gate, (size_t)w->rows * w->gdn_heads * sizeof(float));
    // rows past a call's tokens are multiplied too and their results dropped; the fourth part of the sums is 0
    if (e == hipSuccess) e = hipMemsetAsync(w->A, 0, (size_t)w->rows * max_k * 4, qg::stream);
    if (e == hipSuccess) e = hipMemsetAsync(w->S, 0, sb, qg::stream);
    if (e == hipSuccess) e = hipMemsetAsync(w->xs, 0, xb, qg::stream);
    if (e != hipSuccess) {
        (void)hipGetLastError();
        qgpu_wide_free(w);
        return (int)e;
    }
    *out = w;
    return QGPU_OK;
}

extern "C" int qgpu_wide_supports(const qgpu_tensor *W)
{
    return W && W->packed && W->ne0 <= MAX_K;
}

static bool al16(const void *p) { return ((uintptr_t)p & 15) == 0; }

extern "C" int qgpu_wide_prepare(qgpu_wide *w, const qgpu_act *act, int n, uint64_t ne0, int sums)
{
    int rc = qg::ensure_init();
    if (rc) return rc;
    if (!w || !act || !act->x || n < 1 || n > w->rows || !ne0 || ne0 % 256 || ne0 > w->max_k) return QGPU_E_ARG;
    if (act->n_part || act->embd || act->tok || act->xout) return QGPU_E_ARG;
    WidePrep p = {};
    p.x = act->x; p.ldx = act->ldx; p.y = act->y; p.ldy = act->ldy; p.w = act->w; p.w2 = act->w2;
    p.M = (uint32_t)n; p.ne0 = (uint32_t)ne0; p.seg = (uint32_t)ne0; p.eps = act->eps;
    p.A = w->A; p.S = sums ? w->S : nullptr; p.xs = w->xs;
    int kind = act->kind;
    switch (kind) {
    case QGPU_ACT_COPY: break;
    case QGPU_ACT_RMSNORM:
        if (!p.w) return QGPU_E_ARG;
        if (act->seg && act->seg != ne0) {
            if (act->seg * 2 != ne0 || act->seg % 32 || !p.y || !p.w2) return QGPU_E_ARG;
            p.seg = (uint32_t)act->seg;
            kind = WP_CAT;
        }
        break;
    case QGPU_ACT_SILU_MUL: if (!p.y) return QGPU_E_ARG; break;
    case QGPU_ACT_GATED_NORM: if (!p.y || !p.w || act->seg != 128) return QGPU_E_ARG; break;
    default: return QGPU_E_ARG;
    }
    if (!al16(p.x) || p.ldx % 4 || (p.y && (!al16(p.y) || p.ldy % 4)) || !al16(p.w) || !al16(p.w2)) return QGPU_E_ARG;
    const dim3 grid((unsigned)n);
#define WP(KD, G, N) hipLaunchKernelGGL((k_wide_prep<KD, G, N>), grid, dim3(N), 0, qg::stream, p)
#define WPK(KD) do { if (ne0 <= 3 * 2048) WP(KD, 3, 256); else if (ne0 <= 5 * 2048) WP(KD, 5, 256); \
                     else if (ne0 <= 3 * 8192) WP(KD, 3, 1024); else WP(KD, 8, 1024); } while (0)
    switch (kind) {
    case QGPU_ACT_COPY: WPK(QGPU_ACT_COPY); break;
    case QGPU_ACT_RMSNORM: WPK(QGPU_ACT_RMSNORM); break;
    case WP_CAT: WPK(WP_CAT); break;
    case QGPU_ACT_SILU_MUL: WPK(QGPU_ACT_SILU_MUL); break;
    default: WPK(QGPU_ACT_GATED_NORM); break;
    }
#undef WPK
#undef WP
    QG_LAUNCH_CHECK();
    return QGPU_OK;
}

template <int MTL>
static int wide_launch(int type, WideArgs &a)
{
    a.mblk = (a.M + MTL * 16 - 1) / (MTL * 16);
    uint64_t tiles = 0;
    for (int j = 0; j < a.n_mat; j++) {
        a.m[j].tile0 = (uint32_t)tiles;
        if (!a.pair || !j) tiles += (a.m[j].rows + (a.pair ? WIDE_N / 2 : WIDE_N) - 1) / (a.pair ? WIDE_N / 2 : WIDE_N);
    }
    tiles *= a.mblk;
    if (tiles * a.nsb >= 0xFFFFFFFFull) return QGPU_E_RANGE;
    a.U = (uint32_t)tiles * a.nsb;
    a.G = a.U < WIDE_MAXG ? a.U : WIDE_MAXG;
#define WG(F) hipLaunchKernelGGL((k_wide_gemm<F, MTL>), dim3(a.G), dim3(256), 0, qg::stream, a)
    switch (type) {
    case T_IQ4_XS: WG(T_IQ4_XS); break;
    case T_Q4_K: WG(T_Q4_K); break;
    case T_Q5_K: WG(T_Q5_K); break;
    case T_Q6_K: if constexpr (MTL <= 4) WG(T_Q6_K); break;
    case T_Q8_0: if constexpr (MTL <= 4) WG(T_Q8_0); break;
    default: return QGPU_E_TYPE;
    }
#undef WG
    QG_LAUNCH_CHECK();
    hipLaunchKernelGGL((k_wide_fix<MTL>), dim3((unsigned)tiles, MTL, a.pair ? WIDE_NT / 2 : WIDE_NT), dim3(256), 0, qg::stream, a);
    QG_LAUNCH_CHECK();
    return QGPU_OK;
}

static void wide_mat(WideMat &m, const qgpu_tensor *W, float *out, uint64_t ldo)
{
    m.W = (const uint8_t *)W->data;
    m.out = out;
    m.ldo = ldo;
    m.rows = (uint32_t)W->ne1;
    m.nt16 = (uint32_t)((W->ne1 + 15) / 16);
}

static int wide_go(qgpu_wide *w, int type, uint64_t ne0, int n, WideArgs &a)
{
    a.nsb = (uint32_t)(ne0 / 256);
    a.M = (uint32_t)n;
    a.A = w->A; a.S = w->S; a.xs = w->xs; a.piece = w->piece;
    // tokens per block by the tokens of the call: a block's decode work does not shrink with its tokens, so the
    // smallest tile that holds them all, at most 128 (Q6_K, Q8_0: 64, their records take more registers)
    const bool narrow = type == T_Q6_K || type == T_Q8_0;
    const int mtl = n <= 32 ? 2 : (n <= 64 || narrow) ? 4 : 8;
    return mtl == 2 ? wide_launch<2>(type, a) : mtl == 4 ? wide_launch<4>(type, a) : wide_launch<8>(type, a);
}

extern "C" int qgpu_wide_gemm(qgpu_wide *w, const qgpu_tensor *const *Ws, int n_mat, int n, float *const *outs,
                              const uint64_t *ldos, int flags)
{
    int rc = qg::ensure_init();
    if (rc) return rc;
    if (!w || !Ws || !outs || !ldos || n_mat < 1 || n_mat > QGPU_MAX_MULTI || n < 1 || n > w->rows) return QGPU_E_ARG;
    for (int j = 0; j < n_mat; j++) {
        if (!Ws[j] || !outs[j] || Ws[j]->ne0 != Ws[0]->ne0 || Ws[j]->ne0 > w->max_k || ldos[j] < Ws[j]->ne1) return QGPU_E_ARG;
        if (!Ws[j]->packed) return QGPU_E_TYPE;
    }
    // one launch per format
    unsigned done = 0;
    for (int j0 = 0; j0 < n_mat; j0++) {
        if (done >> j0 & 1) continue;
        WideArgs a = {};
        a.accum = (flags & QGPU_GEMV_ACCUM) != 0;
        const int type = Ws[j0]->type;
        for (int j = j0; j < n_mat; j++) {
            if (Ws[j]->type != type) continue;
            done |= 1u << j;
            wide_mat(a.m[a.n_mat++], Ws[j], outs[j], ldos[j]);
        }
        rc = wide_go(w, type, Ws[0]->ne0, n, a);
        if (rc) return rc;
    }
    return QGPU_OK;
}

// silu(gate) * up in the product's epilogue: a block holds the same rows of both matrices, so one fp32 value
// per pair is written and read back instead of two.
extern "C" int qgpu_wide_gemm_silu(qgpu_wide *w, const qgpu_tensor *gate, const qgpu_tensor *up, int n, float *out,
                                   uint64_t ldo)
{
    int rc = qg::ensure_init();
    if (rc) return rc;
    if (!w || !gate || !up || !out || n < 1 || n > w->rows || gate->ne0 != up->ne0 || gate->ne1 != up->ne1 ||
        gate->ne0 > w->max_k || ldo < gate->ne1)
        return QGPU_E_ARG;
    if (!gate->packed || !up->packed || gate->type != up->type) return QGPU_E_TYPE;
    WideArgs a = {};
    a.n_mat = 2;
    a.pair = 1;
    wide_mat(a.m[0], gate, out, ldo);
    wide_mat(a.m[1], up, out, ldo);
    return wide_go(w, gate->type, gate->ne0, n, a);
}
