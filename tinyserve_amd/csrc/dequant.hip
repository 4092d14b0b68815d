// Bit-exact dequantisation kernels: GGUF (Q8_0/Q4_K/Q5_K/Q6_K, F32/F16) and MXFP4.
//
// One thread decodes 8 consecutive values of a 32-value unit and writes them with 16-byte
// stores, so a wave's stores are whole lines: what bounds the kernels is HBM (a unit per
// thread, 64 bytes from its neighbour's, in dword stores took 78 us for 8192 x 4096 Q5_K to
// bf16, 90 MB; this form 16.4 us, 5.5 TB/s). The four threads of a unit read its header again, from L1. The
// arithmetic per value is formats.h's, to the bit.
#include "formats.h"

namespace tsa {
namespace {

// 8 bytes at p (A: the caller's alignment of the block p lies in).
template <int A>
__device__ __forceinline__ void ld_8bytes(const uint8_t* p, uint32_t (&w)[2]) {
    __builtin_memcpy(w, __builtin_assume_aligned(p, A >= 8 ? 8 : A), 8);
}

// Values 8 h .. 8 h + 7 of unit u of the block at b.
template <int TYPE, int A>
__device__ __forceinline__ void decode8(const uint8_t* b, int u, int h, float (&v)[8]) {
    uint32_t q[2];
    if constexpr (TYPE == 8) {
        const float d = f16_bits_to_f32(ld_u16<A>(b));
        ld_8bytes<A>(b + 2 + 8 * h, q);
#pragma unroll
        for (int i = 0; i < 8; ++i) v[i] = d * (float)(int8_t)byte_of(q, i);
    } else if constexpr (TYPE == 12 || TYPE == 13) {
        uint32_t hd[4], sc, m;
        __builtin_memcpy(hd, __builtin_assume_aligned(b, A), 16);
        ld_8bytes<A>(b + (TYPE == 12 ? 16 : 48) + 32 * (u >> 1) + 8 * h, q);
        uint32_t hb[2] = {0u, 0u};
        if constexpr (TYPE == 13) ld_8bytes<A>(b + 16 + 8 * h, hb);
        k_scale_min_at(hd, (uint32_t)u, sc, m);
        const float a = f16_bits_to_f32(hd[0] & 0xFFFFu) * (float)sc, c = f16_bits_to_f32(hd[0] >> 16) * (float)m;
#pragma unroll
        for (int w = 0; w < 2; ++w) {
            uint32_t qq = (q[w] >> (4 * (u & 1))) & 0x0F0F0F0Fu;
            if constexpr (TYPE == 13) qq |= ((hb[w] >> u) & 0x01010101u) << 4;
#pragma unroll
            for (int i = 0; i < 4; ++i) v[4 * w + i] = a * (float)((qq >> (8 * i)) & 0xFFu) - c;
        }
    } else {
        const int hh = u >> 2, t = u & 3;
        uint32_t qh[2];
        ld_8bytes<A>(b + 64 * hh + 32 * (t & 1) + 8 * h, q);
        ld_8bytes<A>(b + 128 + 32 * hh + 8 * h, qh);
        const float d = f16_bits_to_f32(ld_u16<A>(b + 208)) * (float)(int8_t)b[192 + 2 * u + (h >> 1)];
#pragma unroll
        for (int w = 0; w < 2; ++w) {
            const uint32_t qq = ((q[w] >> (4 * (t >> 1))) & 0x0F0F0F0Fu) | (((qh[w] >> (2 * t)) & 0x03030303u) << 4);
#pragma unroll
            for (int i = 0; i < 4; ++i) v[4 * w + i] = d * (float)((int)((qq >> (8 * i)) & 0xFFu) - 32);
        }
    }
}

// 8 values to out[base ..]: vec, whole 16-byte stores (base a multiple of 8, out 16-byte
// aligned); otherwise element by element.
__device__ __forceinline__ void store8(void* out, int dtype, int64_t base, const float (&v)[8], bool vec) {
    if (!vec) {
#pragma unroll
        for (int i = 0; i < 8; ++i) store_out(out, dtype, base + i, v[i]);
        return;
    }
    if (dtype == TSA_F32) {
        float4* o = reinterpret_cast<float4*>(static_cast<float*>(out) + base);
        o[0] = make_float4(v[0], v[1], v[2], v[3]);
        o[1] = make_float4(v[4], v[5], v[6], v[7]);
        return;
    }
    uint32_t w[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const uint32_t lo = dtype == TSA_BF16 ? f32_to_bf16_bits(v[2 * i]) : f32_to_f16_bits(v[2 * i]);
        const uint32_t hi = dtype == TSA_BF16 ? f32_to_bf16_bits(v[2 * i + 1]) : f32_to_f16_bits(v[2 * i + 1]);
        w[i] = lo | (hi << 16);
    }
    *reinterpret_cast<uint4*>(static_cast<uint16_t*>(out) + base) = make_uint4(w[0], w[1], w[2], w[3]);
}

template <int TYPE, int A>
__global__ void __launch_bounds__(256) gguf_dequant_kernel(const uint8_t* __restrict__ data, int64_t n_units,
                                                           void* __restrict__ out, int out_dtype, int vec) {
    using Tr = GgufTraits<TYPE>;
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x, unit = i >> 2;
    if (unit >= n_units) return;
    float v[8];
    decode8<TYPE, A>(data + unit / Tr::UPB * Tr::TS, (int)(unit % Tr::UPB), (int)(i & 3), v);
    store8(out, out_dtype, 8 * i, v, vec);
}

// F32 / F16 "dequantisation" (tinyserve/gguf_dequant_torch.py:54-59): reinterpret and convert.
__global__ void __launch_bounds__(256) plain_dequant_kernel(const uint8_t* __restrict__ data, int src_f16,
                                                            int64_t n, void* __restrict__ out, int out_dtype) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    float v;
    if (src_f16) {
        uint16_t h;
        __builtin_memcpy(&h, data + 2 * i, 2);
        v = f16_bits_to_f32(h);
    } else {
        __builtin_memcpy(&v, data + 4 * i, 4);
    }
    store_out(out, out_dtype, i, v);
}

// MXFP4 [N, K]: thread i holds 4 of a block's 16 bytes, values 8 i .. 8 i + 7 of the output.
__global__ void __launch_bounds__(256) mxfp4_dequant_kernel(const uint8_t* __restrict__ blocks,
                                                            const uint8_t* __restrict__ scales, int64_t n_blocks,
                                                            void* __restrict__ out, int out_dtype, int vec) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x, c = i >> 2;
    if (c >= n_blocks) return;
    uint32_t w;
    __builtin_memcpy(&w, blocks + 4 * i, 4);
    const float s = e8m0_to_f32(scales[c]);
    float v[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) v[j] = e2m1_to_f32((w >> (4 * j)) & 15u) * s;
    store8(out, out_dtype, 8 * i, v, vec);
}

// MXFP4 to the transposed [K, N]: one thread per 16-byte block (32 values) of row n, group g.
__global__ void __launch_bounds__(256) mxfp4_dequant_t_kernel(const uint8_t* __restrict__ blocks,
                                                              const uint8_t* __restrict__ scales, int64_t N, int64_t G,
                                                              void* __restrict__ out, int out_dtype) {
    const int64_t c = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (c >= N * G) return;
    const int64_t n = c / G, g = c % G;
    uint32_t w[4];
    __builtin_memcpy(w, blocks + c * 16, 16);
    const float s = e8m0_to_f32(scales[c]);
#pragma unroll
    for (int j = 0; j < 16; ++j) {
        const uint32_t byte = (w[j >> 2] >> (8 * (j & 3))) & 0xFFu;
        const int64_t k0 = 32 * g + 2 * j;
        store_out(out, out_dtype, k0 * N + n, e2m1_to_f32(byte & 15u) * s);
        store_out(out, out_dtype, (k0 + 1) * N + n, e2m1_to_f32(byte >> 4) * s);
    }
}

// 32-value units per launch: a launch takes fewer than 2^32 threads, four per unit. A multiple of a
// super-block's 8, and of 16 bytes in every type's blocks and output.
constexpr int64_t LAUNCH_UNITS = (int64_t)1 << 28;

inline unsigned grid_for(int64_t n, int threads) { return (unsigned)((n + threads - 1) / threads); }

}  // namespace
}  // namespace tsa

using namespace tsa;

extern "C" int tsa_gguf_dequant(int ggml_type, const void* data, int64_t data_bytes, int64_t n_elems, void* out,
                                int out_dtype, void* stream) {
    clear_error();
    TSA_REQUIRE(valid_dtype(out_dtype), TSA_ERR_INVALID_ARG, "out_dtype %d is not F32(0)/F16(1)/BF16(2)", out_dtype);
    TSA_REQUIRE(n_elems >= 0 && data_bytes >= 0, TSA_ERR_INVALID_ARG, "negative size");
    if (n_elems == 0) return TSA_OK;
    TSA_REQUIRE(data != nullptr && out != nullptr, TSA_ERR_INVALID_ARG, "null pointer");
    hipStream_t st = as_stream(stream);
    if (ggml_type == 0 || ggml_type == 1) {
        const int64_t need = n_elems * (ggml_type == 0 ? 4 : 2);
        TSA_REQUIRE(data_bytes >= need, TSA_ERR_WEIGHT_TOO_SMALL, "data too small: got %lld bytes, expected %lld",
                    (long long)data_bytes, (long long)need);
        hipLaunchKernelGGL(plain_dequant_kernel, dim3(grid_for(n_elems, 256)), dim3(256), 0, st,
                           static_cast<const uint8_t*>(data), ggml_type == 1, n_elems, out, out_dtype);
        TSA_LAUNCH_CHECK();
        return TSA_OK;
    }
    int be, ts;
    TSA_REQUIRE(gguf_geometry(ggml_type, &be, &ts), TSA_ERR_UNSUPPORTED_TYPE,
                "Unsupported GGML quantization type %d. Supported: [0, 1, 8, 12, 13, 14]", ggml_type);
    TSA_REQUIRE(n_elems % be == 0, TSA_ERR_SHAPE, "n_elems (%lld) must be a multiple of the block size (%d)",
                (long long)n_elems, be);
    const int64_t need = n_elems / be * ts;
    TSA_REQUIRE(data_bytes >= need, TSA_ERR_WEIGHT_TOO_SMALL, "data too small: got %lld bytes, expected %lld",
                (long long)data_bytes, (long long)need);
    const int64_t n_units = n_elems / 32;
    const uint8_t* d = static_cast<const uint8_t*>(data);
    const bool a16 = (reinterpret_cast<uintptr_t>(data) & 15) == 0;
    const bool a2 = (reinterpret_cast<uintptr_t>(data) & 1) == 0;
    const bool out_ok = (reinterpret_cast<uintptr_t>(out) & (out_dtype == TSA_F32 ? 15 : 3)) == 0;
    TSA_REQUIRE(out_ok, TSA_ERR_INVALID_ARG, "out must be %d-byte aligned", out_dtype == TSA_F32 ? 16 : 4);
    const int vec = (reinterpret_cast<uintptr_t>(out) & 15) == 0;
    const dim3 block(256);
    for (int64_t u0 = 0; u0 < n_units; u0 += LAUNCH_UNITS, d += LAUNCH_UNITS * 32 / be * ts) {
        const int64_t nu = n_units - u0 < LAUNCH_UNITS ? n_units - u0 : LAUNCH_UNITS;
        const dim3 grid(grid_for(4 * nu, 256));
        void* o = static_cast<uint8_t*>(out) + u0 * 32 * dtype_size(out_dtype);
        switch (ggml_type) {
            case 8:
                if (a2) hipLaunchKernelGGL((gguf_dequant_kernel<8, 2>), grid, block, 0, st, d, nu, o, out_dtype, vec);
                else hipLaunchKernelGGL((gguf_dequant_kernel<8, 1>), grid, block, 0, st, d, nu, o, out_dtype, vec);
                break;
            case 12:
                if (a16) hipLaunchKernelGGL((gguf_dequant_kernel<12, 16>), grid, block, 0, st, d, nu, o, out_dtype, vec);
                else hipLaunchKernelGGL((gguf_dequant_kernel<12, 1>), grid, block, 0, st, d, nu, o, out_dtype, vec);
                break;
            case 13:
                if (a16) hipLaunchKernelGGL((gguf_dequant_kernel<13, 16>), grid, block, 0, st, d, nu, o, out_dtype, vec);
                else hipLaunchKernelGGL((gguf_dequant_kernel<13, 1>), grid, block, 0, st, d, nu, o, out_dtype, vec);
                break;
            default:
                if (a2) hipLaunchKernelGGL((gguf_dequant_kernel<14, 2>), grid, block, 0, st, d, nu, o, out_dtype, vec);
                else hipLaunchKernelGGL((gguf_dequant_kernel<14, 1>), grid, block, 0, st, d, nu, o, out_dtype, vec);
                break;
        }
        TSA_LAUNCH_CHECK();
    }
    return TSA_OK;
}

extern "C" int tsa_mxfp4_dequant(const void* blocks, const void* scales, int64_t N, int64_t K, void* out,
                                 int out_dtype, int transpose, void* stream) {
    clear_error();
    TSA_REQUIRE(valid_dtype(out_dtype), TSA_ERR_INVALID_ARG, "out_dtype %d is not F32(0)/F16(1)/BF16(2)", out_dtype);
    TSA_REQUIRE(N >= 0 && K >= 0, TSA_ERR_INVALID_ARG, "negative size");
    TSA_REQUIRE(K % 32 == 0, TSA_ERR_SHAPE, "in_features (%lld) must be a multiple of 32", (long long)K);
    if (N == 0 || K == 0) return TSA_OK;
    TSA_REQUIRE(blocks && scales && out, TSA_ERR_INVALID_ARG, "null pointer");
    const int64_t G = K / 32;
    const uint8_t *bl = static_cast<const uint8_t*>(blocks), *sc = static_cast<const uint8_t*>(scales);
    if (transpose)
        hipLaunchKernelGGL(mxfp4_dequant_t_kernel, dim3(grid_for(N * G, 256)), dim3(256), 0, as_stream(stream), bl, sc, N, G,
                           out, out_dtype);
    else
        for (int64_t c0 = 0; c0 < N * G; c0 += LAUNCH_UNITS) {
            const int64_t nc = N * G - c0 < LAUNCH_UNITS ? N * G - c0 : LAUNCH_UNITS;
            hipLaunchKernelGGL(mxfp4_dequant_kernel, dim3(grid_for(4 * nc, 256)), dim3(256), 0, as_stream(stream), bl + 16 * c0,
                               sc + c0, nc, static_cast<uint8_t*>(out) + c0 * 32 * dtype_size(out_dtype), out_dtype,
                               (int)((reinterpret_cast<uintptr_t>(out) & 15) == 0));
            TSA_LAUNCH_CHECK();
        }
    TSA_LAUNCH_CHECK();
    return TSA_OK;
}
