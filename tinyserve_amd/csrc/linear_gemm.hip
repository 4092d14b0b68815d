// y[t, n] = sum_k W[n, k] x[t, k] (+ bias[n]) for many bf16 tokens on the bf16 matrix cores,
// straight from the stored weights: GGUF Q8_0 / Q4_K / Q5_K / Q6_K blocks, checkpoint-order
// MXFP4 blocks, or a bf16 matrix (the router).
//
// Workgroup = 8 waves = RW row groups of 32 weight rows x KW K groups (RW KW = 8), against
// 32 MT tokens. K advances in steps of 128 KW values: wave (rg, kw) takes the 4 units (32
// values each) 4 kw .. 4 kw + 3 of the step for its 32 rows. Lane (g, rr) = (lane / 32,
// lane % 32) loads the codes of values 16 g .. 16 g + 15 of every unit of row rr straight into
// registers one step ahead (each code byte is read by one lane of the workgroup, so LDS would
// only add a pass), decodes them into the A operands of the unit's two K steps of
// v_mfma_f32_32x32x16_bf16 and multiplies the MT token tiles with each operand. K is permuted
// alike in A and B: K step s of a unit covers values 8 s .. 8 s + 7 (g = 0) and 16 + 8 s ..
// (g = 1). The tokens' step (the B operands, shared by the row groups) comes in one step ahead by
// buffer-to-LDS copies into one of two XOR-swizzled tiles. The KW partial sums meet in LDS.
//
// Precision. bf16 x MXFP4 and bf16 x bf16 products are exact in the bf16 MFMA. A GGUF weight is
// the fp32 value the block format defines (decode_unit's), carried whole as three bf16 terms of 8
// significant bits each (lg_split), so its products are exact too and the sums are fp32, as in the
// row kernels. (Two terms, the second rounded, keep 2^-16 of the weight, and sums that cancel come
// out of the wrong bits. The third costs Q6_K 2048 x 4096, 24 tokens, 15.2 -> 18.0 us, Q4_K 4096 x
// 2048, 512 tokens, 24.7 -> 30.2 us.) Results with other output types stay on the row kernels. A
// sum that is not finite is formed again value by value in fp32 (lg_exact): an infinite activation
// meets a zero term as NaN, where the plain product may be infinite.
#include "fused_common.h"
#include "mfma_tile.h"

namespace tsa {
namespace {

constexpr int LG_THREADS = 512;
constexpr int LG_MXFP4 = 0, LG_BF16 = 1;  // formats beside the ggml type ids

typedef int lg_v4i __attribute__((ext_vector_type(4)));
typedef float lg_v16f __attribute__((ext_vector_type(16)));

struct LgParams {
    const uint8_t* w;       // the 16-byte boundary at or below the weights
    const uint8_t* scales;  // MXFP4: the e8m0 bytes' dword at or below
    uint32_t w_records, s_records, w_mis, s_mis;
    const uint16_t* x;
    uint32_t x_records;
    const void* bias;
    int bias_dtype;
    uint16_t* y;
    int T, N, K, KU;        // KU = K / 32 units per row
    int y_vec;              // y rows are whole 16-byte chunks
};

__device__ __forceinline__ lg_v4i lg_desc(const void* p, uint32_t bytes) {
    const uint64_t a = reinterpret_cast<uint64_t>(p);
    return lg_v4i{__builtin_amdgcn_readfirstlane((int)(uint32_t)a), __builtin_amdgcn_readfirstlane((int)(uint32_t)(a >> 32)),
                  __builtin_amdgcn_readfirstlane((int)bytes), 0x00020000};
}

// Lane l's 16 bytes at buffer offset voff land at LDS byte lds + 16 l (inline assembly: the
// compiler would otherwise wait for every copy before any later LDS read).
__device__ __forceinline__ void lg_dma(const lg_v4i& r, uint32_t voff, uint32_t lds) {
    asm volatile("s_mov_b32 m0, %2\n\t" TSA_COPY_WAIT "buffer_load_dwordx4 %0, %1, 0 offen lds" ::"v"(voff), "s"(r),
                 "s"(__builtin_amdgcn_readfirstlane((int)lds))
                 : "memory", "m0");
}

// Raw dwords a lane holds of a step's 4 units. SD: a K-quant row may start inside a
// super-block (K % 256 != 0), so every unit is fetched by itself.
template <int F, bool SD> constexpr int lg_nraw() {
    return F == 8 ? 24 : F == 12 ? (SD ? 32 : 12) : F == 13 ? (SD ? 48 : 16) : F == 14 ? (SD ? 48 : 19)
                   : F == LG_MXFP4 ? 10 : 32;
}

struct LgBufs {
    __amdgpu_buffer_rsrc_t w, s;
};
__device__ __forceinline__ uint32_t lg_ld(const __amdgpu_buffer_rsrc_t& r, uint32_t o) {
    return __builtin_amdgcn_raw_buffer_load_b32(r, (int)o, 0, 0);
}
__device__ __forceinline__ void lg_ld4(const __amdgpu_buffer_rsrc_t& r, uint32_t o, uint32_t* d) {
    const u32x4 v = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(r, (int)o, 0, 0));
    d[0] = v[0], d[1] = v[1], d[2] = v[2], d[3] = v[3];
}
// 20 bytes from the dword at or below o: the 16 bytes at o are lg_16(d, o & 3)
__device__ __forceinline__ void lg_ld5(const __amdgpu_buffer_rsrc_t& r, uint32_t o, uint32_t* d) {
    lg_ld4(r, o & ~3u, d);
    d[4] = lg_ld(r, (o & ~3u) + 16);
}
__device__ __forceinline__ void lg_16(const uint32_t* d, uint32_t ob, uint32_t (&q)[4]) {
#pragma unroll
    for (int i = 0; i < 4; ++i) q[i] = __builtin_amdgcn_alignbyte(d[i + 1], d[i], ob);
}

// Units j .. j + 3 of weight row `row`, lane half g (half super-block H of an aligned K-quant
// row: j % 8 = 4 H). Rows past the matrix read zeros or (the last one) its final dwords.
template <int F, bool SD>
__device__ __forceinline__ void lg_load(const LgParams& p, const LgBufs& b, uint32_t row, int j, int g,
                                        uint32_t (&R)[lg_nraw<F, SD>()]) {
    const uint32_t U = row * (uint32_t)p.KU + (uint32_t)j;
    if constexpr (F == 8) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const uint32_t o = p.w_mis + 34u * (U + i);
            R[6 * i] = lg_ld(b.w, o & ~3u);
            lg_ld5(b.w, o + 2 + 16 * g, R + 6 * i + 1);
        }
    } else if constexpr (F == 12 || F == 13) {
        constexpr uint32_t TS = F == 12 ? 144 : 176, QS = F == 12 ? 16 : 48;
        if constexpr (SD) {
            constexpr int NU = F == 12 ? 8 : 12;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const uint32_t u = (U + i) & 7u, o = TS * ((U + i) >> 3);
                lg_ld4(b.w, o, R + NU * i);
                lg_ld4(b.w, o + QS + 32 * (u >> 1) + 16 * g, R + NU * i + 4);
                if constexpr (F == 13) lg_ld4(b.w, o + 16 + 16 * g, R + NU * i + 8);
            }
        } else {
            const uint32_t o = TS * (U >> 3), h = (uint32_t)(j >> 2) & 1u;
            lg_ld4(b.w, o, R);
            lg_ld4(b.w, o + QS + 64 * h + 16 * g, R + 4);
            lg_ld4(b.w, o + QS + 64 * h + 32 + 16 * g, R + 8);
            if constexpr (F == 13) lg_ld4(b.w, o + 16 + 16 * g, R + 12);
        }
    } else if constexpr (F == 14) {
        if constexpr (SD) {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const uint32_t u = (U + i) & 7u, o = p.w_mis + 210u * ((U + i) >> 3);
                lg_ld5(b.w, o + 64 * (u >> 2) + 32 * (u & 1) + 16 * g, R + 12 * i);
                lg_ld5(b.w, o + 128 + 32 * (u >> 2) + 16 * g, R + 12 * i + 5);
                R[12 * i + 10] = lg_ld(b.w, (o + 192 + 2 * u) & ~3u);
                R[12 * i + 11] = lg_ld(b.w, (o + 208) & ~3u);
            }
        } else {
            const uint32_t o = p.w_mis + 210u * (U >> 3), h = (uint32_t)(j >> 2) & 1u;
            lg_ld5(b.w, o + 64 * h + 16 * g, R);
            lg_ld5(b.w, o + 64 * h + 32 + 16 * g, R + 5);
            lg_ld5(b.w, o + 128 + 32 * h + 16 * g, R + 10);
#pragma unroll
            for (int i = 0; i < 3; ++i) R[15 + i] = lg_ld(b.w, ((o + 192 + 8 * h) & ~3u) + 4 * i);
            R[18] = lg_ld(b.w, (o + 208) & ~3u);
        }
    } else if constexpr (F == LG_MXFP4) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            typedef uint32_t u2 __attribute__((ext_vector_type(2)));
            const u2 v = __builtin_bit_cast(u2, __builtin_amdgcn_raw_buffer_load_b64(b.w, (int)(16u * (U + i) + 8 * g), 0, 0));
            R[2 * i] = v[0], R[2 * i + 1] = v[1];
        }
        const uint32_t o = p.s_mis + U;
        R[8] = lg_ld(b.s, o & ~3u);
        R[9] = lg_ld(b.s, (o & ~3u) + 4);
    } else {
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int s = 0; s < 2; ++s) lg_ld4(b.w, 64u * (U + i) + 32 * g + 16 * s, R + 8 * i + 4 * s);
    }
}

// Two bf16 words in one: the upper halves of a and b.
__device__ __forceinline__ uint32_t lg_upper(uint32_t a, uint32_t b) { return __builtin_amdgcn_perm(b, a, 0x07060302u); }

// 16 values as three terms of packed bf16 words, upper half by upper half: each takes the 8 leading
// significant bits of what the one before leaves, 24 in all, so v = t[0] + t[1] + t[2] exactly
// (down to bf16's smallest number).
__device__ __forceinline__ void lg_split(const float (&v)[16], uint32_t (&t)[3][8]) {
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        float a = v[2 * i], b = v[2 * i + 1];
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            const uint32_t ua = __float_as_uint(a), ub = __float_as_uint(b);
            t[k][i] = lg_upper(ua, ub);
            a -= __uint_as_float(ua & 0xFFFF0000u), b -= __uint_as_float(ub & 0xFFFF0000u);
        }
    }
}

// Unit i (0 .. 3) of the step as A operands: the terms' words 4 s .. 4 s + 3 for K step s (one term
// unless the weights are GGUF). H: the half super-block of an aligned K-quant row.
template <int F> constexpr int lg_terms() { return F == LG_MXFP4 || F == LG_BF16 ? 1 : 3; }
template <int F, bool SD, int H>
__device__ __forceinline__ void lg_decode(const LgParams& p, const uint32_t (&R)[lg_nraw<F, SD>()], uint32_t row, int j,
                                          int i, int g, uint32_t (&t)[lg_terms<F>()][8]) {
    if constexpr (F == LG_MXFP4) {
        const uint32_t ob = (p.s_mis + row * (uint32_t)p.KU + (uint32_t)j) & 3u;
        const float s = e8m0_to_f32((__builtin_amdgcn_alignbyte(R[9], R[8], ob) >> (8 * i)) & 0xFFu);
#pragma unroll
        for (int k = 0; k < 2; ++k) {
            const u32x4 v = __builtin_bit_cast(u32x4, expand(R[2 * i + k], s));
#pragma unroll
            for (int d = 0; d < 4; ++d) t[0][4 * k + d] = v[d];
        }
    } else if constexpr (F == LG_BF16) {
#pragma unroll
        for (int d = 0; d < 8; ++d) t[0][d] = R[8 * i + d];
    } else {
        float v[16];
        const uint32_t U = row * (uint32_t)p.KU + (uint32_t)(j + i);
        if constexpr (F == 8) {
            const uint32_t o = p.w_mis + 34u * U;
            uint32_t q[4];
            lg_16(R + 6 * i + 1, (o + 2) & 3u, q);
            const float d = f16_bits_to_f32(R[6 * i] >> (8 * (o & 3u)));
#pragma unroll
            for (int w = 0; w < 4; ++w)
#pragma unroll
                for (int e = 0; e < 4; ++e) v[4 * w + e] = d * (float)(int8_t)((q[w] >> (8 * e)) & 0xFFu);
        } else if constexpr (F == 12 || F == 13) {
            const uint32_t u = SD ? U & 7u : (uint32_t)(4 * H + i);
            const uint32_t* hd = SD ? R + (F == 12 ? 8 : 12) * i : R;
            const uint32_t* qs = SD ? hd + 4 : R + 4 + 4 * (i >> 1);
            const uint32_t* qh = SD ? hd + 8 : R + 12;
            uint32_t sc, m;
            if constexpr (SD) {
                k_scale_min_at(hd, u, sc, m);
            } else {
                const uint32_t s3[3] = {hd[1], hd[2], hd[3]};
                k_scale_min(s3, 4 * H + i, sc, m);
            }
            const float a = f16_bits_to_f32(hd[0] & 0xFFFFu) * (float)sc, c = f16_bits_to_f32(hd[0] >> 16) * (float)m;
            const uint32_t sh = 4 * (u & 1);
#pragma unroll
            for (int w = 0; w < 4; ++w) {
                uint32_t q = (qs[w] >> sh) & 0x0F0F0F0Fu;
                if constexpr (F == 13) q |= ((qh[w] >> u) & 0x01010101u) << 4;
                // masked once for its four bytes (the compiler extracts each by itself otherwise:
                // Q4_K 4096 x 2048, 512 tokens, 27.3 -> 24.4 us per call, with two terms per weight)
                asm("" : "+v"(q));
#pragma unroll
                for (int e = 0; e < 4; ++e) v[4 * w + e] = a * (float)((q >> (8 * e)) & 0xFFu) - c;
            }
        } else {
            const uint32_t u = SD ? U & 7u : (uint32_t)(4 * H + i), um = u & 3u;
            const uint32_t o = p.w_mis + 210u * (U >> 3), ob = o & 3u;  // 0 or 2
            uint32_t ql[4], qh[4];
            float d, dd;
            if constexpr (SD) {
                lg_16(R + 12 * i, ob, ql);
                lg_16(R + 12 * i + 5, ob, qh);
                const uint32_t sw = R[12 * i + 10] >> (8 * ((o + 192 + 2 * u) & 3u) + 8 * g);
                d = f16_bits_to_f32(R[12 * i + 11] >> (8 * ((o + 208) & 3u)));
                dd = 0.25f * (d * (float)(int8_t)(sw & 0xFFu));
            } else {
                lg_16(R + 5 * (i & 1), ob, ql);
                lg_16(R + 10, ob, qh);
                const uint32_t sw = __builtin_amdgcn_alignbyte(R[16 + (i >> 1)], R[15 + (i >> 1)], ob) >> (16 * (i & 1) + 8 * g);
                d = f16_bits_to_f32(R[18] >> (8 * ob));
                dd = 0.25f * (d * (float)(int8_t)(sw & 0xFFu));
            }
            const uint32_t shl = 4 * (um >> 1), shh = 2 * um;
#pragma unroll
            for (int w = 0; w < 4; ++w) {
                // four signed bytes 4 (q - 32): q ^ 32 is q - 32 in 6-bit two's complement
                uint32_t q = ((((ql[w] >> shl) & 0x0F0F0F0Fu) | (((qh[w] >> shh) & 0x03030303u) << 4)) ^ 0x20202020u) << 2;
                asm("" : "+v"(q));
#pragma unroll
                for (int e = 0; e < 4; ++e) v[4 * w + e] = dd * (float)(int8_t)((q >> (8 * e)) & 0xFFu);
            }
        }
        lg_split(v, t);
    }
}

// Unit j's part of the dot product of weight row n and token t in fp32, value by value (MXFP4: the
// codes' dot product, then the block's scale).
template <int F>
__device__ __forceinline__ float lg_exact(const LgParams& p, int t, int n, int j) {
    const int64_t U = (int64_t)n * p.KU + j;
    const u32x4* xr = reinterpret_cast<const u32x4*>(p.x + (int64_t)t * p.K + 32 * j);
    float v[32], d = 0.0f;
    if constexpr (F == LG_MXFP4) {
        const u32x4 c = reinterpret_cast<const u32x4*>(p.w)[U];
#pragma unroll
        for (int k = 0; k < 32; ++k) v[k] = e2m1_to_f32((c[k >> 3] >> (4 * (k & 7))) & 15u);
    } else if constexpr (F == LG_BF16) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const u32x4 c = reinterpret_cast<const u32x4*>(p.w)[4 * U + i];
#pragma unroll
            for (int k = 0; k < 8; ++k) v[8 * i + k] = __uint_as_float(k & 1 ? c[k >> 1] & 0xFFFF0000u : c[k >> 1] << 16);
        }
    } else {
        using Tr = GgufTraits<F>;
        decode_unit<F, Tr::FAST_A>(p.w + p.w_mis + U / Tr::UPB * Tr::TS, (int)(U % Tr::UPB), v);
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const u32x4 x = xr[i];
#pragma unroll
        for (int k = 0; k < 8; ++k) d = fmaf(v[8 * i + k], __uint_as_float(k & 1 ? x[k >> 1] & 0xFFFF0000u : x[k >> 1] << 16), d);
    }
    if constexpr (F == LG_MXFP4) d *= e8m0_to_f32(p.scales[p.s_mis + U]);
    return d;
}

__device__ __forceinline__ bool lg_finite(float v) { return (__float_as_uint(v) & 0x7F800000u) != 0x7F800000u; }

// The results of a wave (lane: rows n .. n + 7 of token t, `live` of them) that are not finite, again
// in fp32: NaN for all of a token that holds one, else the whole wave forms one after the other, its
// lanes over the units. us per call, finite / one token with a NaN / one with an infinity / all
// tokens with a NaN / with an infinity: Q6_K 2048 x 4096, 24 tokens 18 / 20 / 76 / 47 / 945, Q4_K 4096 x
// 2048, 512 tokens 32 / 35 / 143 / 47 / 1160, MXFP4 5760 x 2880, 77 tokens 13 / 15 / 256 / 27 / 2230 (a
// thread for 8 results, one after the other: 950, 365, 2200 for the one NaN; the row kernels take
// 59, 1210, 247 for any values).
template <int F>
__device__ __forceinline__ void lg_redo(const LgParams& p, int t, int n, int live, float (&v)[8]) {
    const int lane = threadIdx.x & 63;
    uint32_t bad = 0;
#pragma unroll
    for (int e = 0; e < 8; ++e) bad |= e < live && !lg_finite(v[e]) ? 1u << e : 0u;
    for (uint64_t m = __ballot(bad != 0), fine = 0; m;) {  // fine: lanes whose token is known to hold no NaN
        const int l = __ffsll((unsigned long long)m) - 1, tl = __builtin_amdgcn_readlane(t, l);
        if (!(fine >> l & 1)) {
            bool nan = false;
            for (int c = lane; c < p.K / 8; c += 64) {
                const u32x4 x = *reinterpret_cast<const u32x4*>(p.x + (int64_t)tl * p.K + 8 * c);
#pragma unroll
                for (int i = 0; i < 4; ++i) nan |= (x[i] & 0x7FFFu) > 0x7F80u || (x[i] & 0x7FFF0000u) > 0x7F800000u;
            }
            const uint64_t same = __ballot(t == tl);
            if (__ballot(nan)) {
#pragma unroll
                for (int d = 0; d < 8; ++d) v[d] = t == tl && (bad >> d & 1) ? __uint_as_float(0x7FC00000u) : v[d];
                m &= ~same;
                continue;
            }
            fine = same;
        }
        const int nl = __builtin_amdgcn_readlane(n, l);
        for (uint32_t w = __builtin_amdgcn_readlane(bad, l); w; w &= w - 1) {
            const int e = __builtin_ctz(w);
            float s = 0.0f;
            for (int j = lane; j < p.KU; j += 64) s += lg_exact<F>(p, tl, nl + e, j);
            s = wave_sum(s);
#pragma unroll
            for (int d = 0; d < 8; ++d) v[d] = lane == l && d == e ? s : v[d];
        }
        m &= m - 1;
    }
}

__host__ __device__ constexpr int lg_xbytes(int MT, int KW) { return 32 * MT * 256 * KW; }  // one token tile of a step
__host__ __device__ constexpr int lg_lds(int MT, int KW) {
    const int rows = 32 * (8 / KW), stage = KW * 32 * MT * (rows + 4) * 4, x = 2 * lg_xbytes(MT, KW);
    return x > stage ? x : stage;
}

template <int F, int MT, int KW, bool SD>
__global__ void __launch_bounds__(LG_THREADS) lin_gemm_kernel(LgParams p) {
    extern __shared__ __align__(16) uint8_t smem[];
    constexpr int RW = 8 / KW, ROWS = 32 * RW, TOK = 32 * MT, STEP = 128 * KW, CH = STEP / 8, XB = lg_xbytes(MT, KW);
    constexpr int NX = MT * KW, NR = lg_nraw<F, SD>(), TERMS = lg_terms<F>();
    // Workgroups are dealt round the 8 XCDs by linear id: renumbered so that each XCD takes a
    // run of row tiles with all their token tiles (the weights of a row tile share one L2).
    const int tt = (p.T + TOK - 1) / TOK, total = (int)gridDim.x, lin = (int)blockIdx.x;
    const int xcd = lin & 7, q8 = total >> 3, rem = total & 7;
    const int wid = xcd * q8 + (xcd < rem ? xcd : rem) + (lin >> 3);  // a bijection of [0, total)
    const int n0 = wid / tt * ROWS, t0 = wid % tt * TOK;
    const int tid = threadIdx.x, lane = tid & 63, wave = uniform(tid >> 6);
    const int kw = wave % KW, rg = wave / KW, g = lane >> 5, rr = lane & 31;
    const int steps = (p.KU + 4 * KW - 1) / (4 * KW);
    const uint32_t row = (uint32_t)(n0 + 32 * rg + rr < p.N ? n0 + 32 * rg + rr : p.N - 1);  // past N: any row, not stored

    // Token tile: token r's step as CH chunks of 16 bytes, chunk c in slot c ^ (r % 32) (the 32
    // tokens of an operand read fall on distinct banks). Copy i of wave w fills chunks
    // 64 (NX w + i) + lane; tokens past T and columns past K read zeros (offsets past the end).
    const lg_v4i rx = lg_desc(p.x, p.x_records);
    const uint32_t lds0 = (uint32_t)reinterpret_cast<uintptr_t>(smem);
    uint32_t xo[NX];
    int xc[NX];
#pragma unroll
    for (int i = 0; i < NX; ++i) {
        const int q = 64 * (NX * wave + i) + lane, r = q / CH, c = (q % CH) ^ (r & 31);
        xc[i] = 8 * c;
        xo[i] = t0 + r < p.T ? (uint32_t)(t0 + r) * (uint32_t)p.K * 2u + 16u * (uint32_t)c : 0x80000000u;
    }
    auto issue_x = [&](int s) {
        const uint32_t dst = lds0 + (uint32_t)(s & 1) * XB + 1024u * (uint32_t)(NX * wave);
#pragma unroll
        for (int i = 0; i < NX; ++i)
            lg_dma(rx, STEP * s + xc[i] < p.K ? xo[i] + (uint32_t)s * (2 * STEP) : 0x80000000u, dst + 1024u * i);
    };

    LgBufs b;
    b.w = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(p.w), (short)0, (int)p.w_records, 0x00020000);
    b.s = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(F == LG_MXFP4 ? p.scales : p.w), (short)0,
                                            (int)(F == LG_MXFP4 ? p.s_records : p.w_records), 0x00020000);

    lg_v16f acc[MT];
#pragma unroll
    for (int t = 0; t < MT; ++t)
#pragma unroll
        for (int i = 0; i < 16; ++i) acc[t][i] = 0.0f;

    auto units = [&](const uint32_t (&R)[NR], int j, const uint8_t* xt, auto hc) {
        constexpr int H = decltype(hc)::value;
        const uint8_t* xr = xt + rr * (16 * CH);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            if (j + i >= p.KU) break;  // wave-uniform: past the row's end
            uint32_t w[TERMS][8];
            lg_decode<F, SD, H>(p, R, row, j, i, g, w);
#pragma unroll
            for (int s = 0; s < 2; ++s) {
                const int c = (4 * (4 * kw + i) + 2 * g + s) ^ rr;
                bf16x8 B[MT];
#pragma unroll
                for (int t = 0; t < MT; ++t) B[t] = *reinterpret_cast<const bf16x8*>(xr + t * (512 * CH) + 16 * c);
#pragma unroll
                for (int m = 0; m < TERMS; ++m) {
                    const bf16x8 A =
                        __builtin_bit_cast(bf16x8, u32x4{w[m][4 * s], w[m][4 * s + 1], w[m][4 * s + 2], w[m][4 * s + 3]});
#pragma unroll
                    for (int t = 0; t < MT; ++t) acc[t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(A, B[t], acc[t], 0, 0, 0);
                }
            }
        }
    };

    uint32_t R[NR], Rn[NR];
    lg_load<F, SD>(p, b, row, 4 * kw, g, R);
    issue_x(0);
    for (int s = 0; s < steps; ++s) {
        // This wave's copies and loads of step s have landed (nothing newer flies), then the
        // barrier: every wave's copies have, and tile (s + 1) % 2, last read in step s - 1, is free.
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
#pragma unroll
        for (int i = 0; i < NR; ++i) asm volatile("" : "+v"(R[i]));  // loaded: no later wait for them
        __syncthreads();
        const int j = 4 * KW * s + 4 * kw;
        if (s + 1 < steps) {
            lg_load<F, SD>(p, b, row, j + 4 * KW < p.KU ? j + 4 * KW : j, g, Rn);
            issue_x(s + 1);
        }
        const uint8_t* xt = smem + (s & 1) * XB;
        if (F == 8 || F == LG_MXFP4 || F == LG_BF16 || SD || (kw & 1) == 0) units(R, j, xt, std::integral_constant<int, 0>{});
        else units(R, j, xt, std::integral_constant<int, 1>{});
        if (s + 1 < steps) {
#pragma unroll
            for (int i = 0; i < NR; ++i) R[i] = Rn[i];
        }
    }

    // The partial sums: acc[t][4u + r] is row 32 rg + 8u + 4g + r, token 32 t + rr, over the
    // wave's K. Into stage[kw][token][row], then 8 rows of a token per thread: summed over kw,
    // the bias added, rounded once.
    __syncthreads();
    constexpr int SS = ROWS + 4;
    float* stage = reinterpret_cast<float*>(smem);
#pragma unroll
    for (int t = 0; t < MT; ++t)
#pragma unroll
        for (int u = 0; u < 4; ++u)
            *reinterpret_cast<float4*>(stage + (kw * TOK + 32 * t + rr) * SS + 32 * rg + 8 * u + 4 * g) =
                make_float4(acc[t][4 * u], acc[t][4 * u + 1], acc[t][4 * u + 2], acc[t][4 * u + 3]);
    __syncthreads();
    static_assert(TOK * (ROWS / 8) % 64 == 0, "whole waves below");
    for (int i = tid; i < TOK * (ROWS / 8); i += LG_THREADS) {
        const int tk = i / (ROWS / 8), c = 8 * (i % (ROWS / 8)), t = t0 + tk, n = n0 + c;
        float v[8] = {0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int k = 0; k < KW; ++k) {
            const float4 a = *reinterpret_cast<const float4*>(stage + (k * TOK + tk) * SS + c);
            const float4 d = *reinterpret_cast<const float4*>(stage + (k * TOK + tk) * SS + c + 4);
            v[0] += a.x, v[1] += a.y, v[2] += a.z, v[3] += a.w;
            v[4] += d.x, v[5] += d.y, v[6] += d.z, v[7] += d.w;
        }
        const int live = t < p.T ? (p.N - n < 8 ? p.N - n : 8) : 0;  // 0 or less: none
        float b[8];  // without a bias -0, which leaves every sum as it is
#pragma unroll
        for (int e = 0; e < 8; ++e) b[e] = -0.0f;
        if (p.bias) {
#pragma unroll
            for (int e = 0; e < 8; ++e)
                if (e < live) b[e] = load_act(p.bias, p.bias_dtype, n + e);
        }
        uint32_t top = 0;
#pragma unroll
        for (int e = 0; e < 8; ++e) top = max(top, __float_as_uint(v[e]) << 1);
        if (__builtin_expect(__ballot(live > 0 && top >= 0xFF000000u) != 0, 0)) lg_redo<F>(p, t, n, live, v);
        uint32_t o[4];
#pragma unroll
        for (int d = 0; d < 4; ++d) o[d] = pack_bf16x2(v[2 * d] + b[2 * d], v[2 * d + 1] + b[2 * d + 1]);
        uint16_t* dst = p.y + (int64_t)t * p.N + n;
        if (p.y_vec) {
            if (live > 0) *reinterpret_cast<uint4*>(dst) = make_uint4(o[0], o[1], o[2], o[3]);
        } else {
#pragma unroll
            for (int e = 0; e < 8; ++e)
                if (e < live) dst[e] = (uint16_t)(o[e >> 1] >> (16 * (e & 1)));
        }
    }
}

template <int F, int MT, int KW, bool SD>
hipError_t lg_launch(const LgParams& p, hipStream_t st) {
    const void* fn = reinterpret_cast<const void*>(&lin_gemm_kernel<F, MT, KW, SD>);
    constexpr int lds = lg_lds(MT, KW), rows = 32 * (8 / KW), tok = 32 * MT;
    const hipError_t e = ensure_dynamic_lds(fn, lds);
    if (e != hipSuccess) return e;
    const int64_t grid = (int64_t)((p.N + rows - 1) / rows) * ((p.T + tok - 1) / tok);
    LgParams q = p;
    void* args[] = {&q};
    return hipLaunchKernel(fn, dim3((unsigned)grid), dim3(LG_THREADS), args, lds, st);
}

// The tile (32 MT tokens x 256 / KW rows): the one with the least rounds x round time, a round
// being one workgroup on every CU. More K groups per workgroup shorten a round and re-read the
// tokens more often, more tokens per workgroup share a decoded weight. A round of each, us, at K
// 2048 / 8192: Q4_K 9.1 13.9 18.4 32.3 48.2 / 30.1 48.5 62.6 113.8 178.8, Q8_0 12.6 20.5 25.3 39.6
// 55.2 / 40.3 65.2 79.5 144.7 208.7, Q6_K 11.1 17.9 22.0 38.2 53.6 / 36.2 62.4 74.8 140.6 196.8, bf16 9.0
// 15.3 17.9 29.3 37.5 / 28.0 47.9 55.3 131.2 150.5, MXFP4 7.2 9.3 11.6 20.2 29.6 / 19.8 31.4 37.4 61.4
// 87.5. With the costs here the pick is the fastest of the five in all of 230 calls measured with
// each tile (GGUF N 512 .. 5760, K 2048 .. 8192, 20 .. 1500 tokens; bf16 128 and 512 rows). MXFP4 has
// its own: two of its 2x2 workgroups share a CU (registers and LDS), so 4x2 costs more against
// them (5760 x 2880, 1024 tokens: 49 and 63 us); within 3% of the fastest in all of 70 calls.
template <int F, bool SD>
hipError_t lg_pick(const LgParams& p, hipStream_t st) {
    struct Tile { int mt, kw, cost; };
    constexpr bool MX = F == LG_MXFP4;
    constexpr Tile tiles[5] = {{1, 8, 81}, {1, 4, MX ? 105 : 123}, {2, 4, MX ? 130 : 150}, {2, 2, MX ? 211 : 250}, {4, 2, MX ? 356 : 350}};
    const int64_t cus = num_cus() > 0 ? num_cus() : 256;
    int best = 0;
    int64_t least = INT64_MAX;
    for (int i = 0; i < 5; ++i) {
        const int rows = 256 / tiles[i].kw, tok = 32 * tiles[i].mt;
        const int64_t wgs = (int64_t)((p.N + rows - 1) / rows) * ((p.T + tok - 1) / tok);
        const int64_t cost = (wgs + cus - 1) / cus * tiles[i].cost;
        if (cost < least) least = cost, best = i;
    }
    switch (best) {
        case 0: return lg_launch<F, 1, 8, SD>(p, st);
        case 1: return lg_launch<F, 1, 4, SD>(p, st);
        case 2: return lg_launch<F, 2, 4, SD>(p, st);
        case 3: return lg_launch<F, 2, 2, SD>(p, st);
        default: return lg_launch<F, 4, 2, SD>(p, st);
    }
}

int lg_run(int fmt, LgParams& p, hipStream_t st) {
    p.KU = p.K / 32;
    p.y_vec = p.N % 8 == 0 && (reinterpret_cast<uintptr_t>(p.y) & 15u) == 0;
    p.x_records = (uint32_t)((int64_t)p.T * p.K * 2);
    const bool sd = p.K % 256 != 0;
    hipError_t e = hipErrorInvalidValue;
    switch (fmt) {
        case 8: e = lg_pick<8, false>(p, st); break;
        case 12: e = sd ? lg_pick<12, true>(p, st) : lg_pick<12, false>(p, st); break;
        case 13: e = sd ? lg_pick<13, true>(p, st) : lg_pick<13, false>(p, st); break;
        case 14: e = sd ? lg_pick<14, true>(p, st) : lg_pick<14, false>(p, st); break;
        case LG_MXFP4: e = lg_pick<LG_MXFP4, false>(p, st); break;
        default: e = lg_pick<LG_BF16, false>(p, st); break;
    }
    TSA_HIP_CHECK(e);
    return TSA_OK;
}

// Sizes the kernel's 32-bit offsets hold, and x rows it can copy in 16-byte chunks.
bool lg_shape_ok(const void* x, int64_t T, int64_t N, int64_t K) {
    return K % 32 == 0 && K >= 32 && N * K < ((int64_t)1 << 31) && T * K * 2 < ((int64_t)1 << 31) && T * N < ((int64_t)1 << 40) &&
           T < ((int64_t)1 << 30) && (reinterpret_cast<uintptr_t>(x) & 15u) == 0 &&
           ((N + 31) / 32) * ((T + 31) / 32) < ((int64_t)1 << 31);
}

}  // namespace

// Whether the GGUF matrix-core linear takes a call: bf16 tokens and results, blocks on the
// boundary their decoder reads them at.
bool lg_gguf_supported(int type, const void* w, const void* x, int x_dtype, int y_dtype, int64_t T, int64_t N, int64_t K) {
    const uintptr_t al = type == 12 || type == 13 ? 15u : 1u;
    return x_dtype == TSA_BF16 && y_dtype == TSA_BF16 && (reinterpret_cast<uintptr_t>(w) & al) == 0 && lg_shape_ok(x, T, N, K);
}

int lg_gguf(int type, const uint8_t* w, int64_t w_bytes, const void* x, int64_t T, int64_t K, void* y, int64_t N,
            hipStream_t st) {
    LgParams p{};
    p.w_mis = (uint32_t)(reinterpret_cast<uintptr_t>(w) & 15u);
    p.w = w - p.w_mis;
    const int64_t rec = (w_bytes + p.w_mis + 15) & ~(int64_t)15;
    p.w_records = rec < 0xFFFFFFF0ll ? (uint32_t)rec : 0xFFFFFFF0u;
    p.x = static_cast<const uint16_t*>(x);
    p.y = static_cast<uint16_t*>(y);
    p.T = (int)T, p.N = (int)N, p.K = (int)K;
    return lg_run(type, p, st);
}

// MXFP4 blocks in the checkpoint order: bf16 tokens and results, 16-byte-aligned blocks.
bool lg_mxfp4_supported(const void* blocks, const void* x, int x_dtype, int y_dtype, int64_t T, int64_t N, int64_t K) {
    return x_dtype == TSA_BF16 && y_dtype == TSA_BF16 && (reinterpret_cast<uintptr_t>(blocks) & 15u) == 0 &&
           lg_shape_ok(x, T, N, K);
}

int lg_mxfp4(const uint8_t* blocks, const uint8_t* scales, const void* bias, int bias_dtype, const void* x, int64_t T,
             void* y, int64_t N, int64_t K, hipStream_t st) {
    LgParams p{};
    p.w = blocks;
    p.w_records = (uint32_t)(N * K / 2);
    p.s_mis = (uint32_t)(reinterpret_cast<uintptr_t>(scales) & 3u);
    p.scales = scales - p.s_mis;
    p.s_records = (uint32_t)((N * K / 32 + p.s_mis + 3) & ~(int64_t)3);
    p.bias = bias;
    p.bias_dtype = bias_dtype;
    p.x = static_cast<const uint16_t*>(x);
    p.y = static_cast<uint16_t*>(y);
    p.T = (int)T, p.N = (int)N, p.K = (int)K;
    return lg_run(LG_MXFP4, p, st);
}

// A bf16 matrix [N, K] (the router): bf16 tokens and results, 16-byte-aligned rows.
bool lg_bf16_supported(const void* w, int w_dtype, const void* x, int x_dtype, int y_dtype, int64_t T, int64_t N, int64_t K) {
    return w_dtype == TSA_BF16 && x_dtype == TSA_BF16 && y_dtype == TSA_BF16 &&
           (reinterpret_cast<uintptr_t>(w) & 15u) == 0 && lg_shape_ok(x, T, N, K);
}

int lg_bf16(const void* w, const void* bias, int bias_dtype, const void* x, int64_t T, void* y, int64_t N, int64_t K,
            hipStream_t st) {
    LgParams p{};
    p.w = static_cast<const uint8_t*>(w);
    p.w_records = (uint32_t)(2 * N * K);
    p.bias = bias;
    p.bias_dtype = bias_dtype;
    p.x = static_cast<const uint16_t*>(x);
    p.y = static_cast<uint16_t*>(y);
    p.T = (int)T, p.N = (int)N, p.K = (int)K;
    return lg_run(LG_BF16, p, st);
}

}  // namespace tsa
