// Prefill side of the MoE path: expert-major grouping of (token, j) assignments and the
// batched expert FFN over many tokens.
#include "fused_common.h"
#include "moe_group.h"

namespace tsa {
int validate_layout(const tsa_expert_layout* L);
bool pf_mxt_supported(const tsa_expert_layout& L, int x_dtype, int64_t T, int k);
int64_t pf_mxt_workspace_bytes(const tsa_expert_layout& L, int64_t T, int k, int64_t E);
int pf_mxt_prefill(const tsa_expert_layout& L, const uint8_t* pool, int64_t n_slots, const int32_t* expert_slot,
                   int64_t E, const int32_t* idx, const float* weights, int64_t T, int k, const uint16_t* x, void* y,
                   int y_dtype, uint8_t* ws, hipStream_t stream);
bool gf_supported(const tsa_expert_layout& L, int x_dtype, int64_t T, int k);
int64_t gf_workspace_bytes(const tsa_expert_layout& L, int64_t T, int k, int64_t E);
int gf_prefill(const tsa_expert_layout& L, const uint8_t* pool, int64_t n_slots, const int32_t* expert_slot, int64_t E,
               const int32_t* idx, const float* weights, int64_t T, int k, const uint16_t* x, void* y, int y_dtype,
               uint8_t* ws, hipStream_t stream);

namespace {

__global__ void __launch_bounds__(GROUP_THREADS) group_kernel(const int32_t* __restrict__ idx, int64_t n, int E,
                                                              int32_t* __restrict__ counts,
                                                              int32_t* __restrict__ offsets,
                                                              int32_t* __restrict__ perm, GroupTiles tiles) {
    extern __shared__ __align__(16) unsigned char gsm[];
    if (tiles.table) group_assignments<true>(idx, n, E, counts, offsets, perm, tiles, GROUP_WAVES, gsm);
    else group_assignments<false>(idx, n, E, counts, offsets, perm, tiles, GROUP_WAVES, gsm);
}

__global__ void __launch_bounds__(256) map_slots_kernel(const int32_t* __restrict__ idx, int64_t n,
                                                        const int32_t* __restrict__ expert_slot, int64_t E,
                                                        int32_t* __restrict__ slots) {
    const int64_t a = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (a >= n) return;
    const int e = idx[a];
    slots[a] = (e >= 0 && e < E) ? expert_slot[e] : -1;
}

}  // namespace

// tile_rows > 0: also the tile table of the resident experts (table: int4 entries).
int launch_group_kernel(const int32_t* idx, int64_t n, int E, int32_t* counts, int32_t* offsets, int32_t* perm,
                        hipStream_t stream, const int32_t* expert_slot, int64_t n_slots, int tile_rows,
                        int* n_entries, void* table) {
    const int lds = group_lds_bytes(E);
    const hipError_t e = ensure_dynamic_lds(reinterpret_cast<const void*>(&group_kernel), lds);
    TSA_REQUIRE(e == hipSuccess, TSA_ERR_HIP, "hipFuncSetAttribute(LDS %d): %s", lds, hipGetErrorString(e));
    const GroupTiles tiles{expert_slot, n_slots, tile_rows, n_entries, tile_rows > 0 ? static_cast<int4*>(table) : nullptr};
    hipLaunchKernelGGL(group_kernel, dim3(1), dim3(GROUP_THREADS), lds, stream, idx, n, E, counts, offsets, perm,
                       tiles);
    TSA_LAUNCH_CHECK();
    return TSA_OK;
}

}  // namespace tsa

using namespace tsa;

extern "C" int tsa_group_by_expert(const int32_t* idx, int64_t T, int k, int64_t E, int32_t* counts, int32_t* offsets,
                                   int32_t* perm, void* stream) {
    clear_error();
    TSA_REQUIRE(T >= 0 && k >= 1 && E >= 1 && E <= MAX_GROUP_E, TSA_ERR_SHAPE,
                "bad grouping shape (T %lld, k %d, E %lld; E must be <= %d)", (long long)T, k, (long long)E,
                MAX_GROUP_E);
    TSA_REQUIRE(T * k < (int64_t)1 << 31, TSA_ERR_SHAPE, "too many assignments");
    TSA_REQUIRE(idx && counts && offsets && (perm || T == 0), TSA_ERR_INVALID_ARG, "null pointer");
    return launch_group_kernel(idx, T * k, (int)E, counts, offsets, perm, as_stream(stream), nullptr, 0, 0, nullptr,
                               nullptr);
}

// Workspace of the token-chunked decode path: the assignments' slots, then a decode workspace.
static int64_t chunked_ws(const tsa_expert_layout& L, int64_t T, int k) {
    int64_t dec = 0;
    tsa_moe_decode_workspace_size(&L, T, k, &dec);
    return ((T * k * 4 + 255) / 256) * 256 + dec;
}

// MXFP4 tiled pools with bf16 activations take the grouped MFMA GEMMs, and so do GGUF pools
// (gf_supported: bf16 activations, dimensions multiples of 32, enough assignments); every
// other call runs the decode kernels over chunks of tokens. The workspace covers the
// largest form the layout can take (the x dtype is not known here).
static int64_t prefill_ws(const tsa_expert_layout& L, int64_t T, int k, int64_t E) {
    const int64_t c = chunked_ws(L, T, k);
    int64_t g = 0;
    if (L.format == TSA_EXPERT_MXFP4 && L.mx_tiled) g = pf_mxt_workspace_bytes(L, T, k, E);
    if (gf_supported(L, TSA_BF16, T, k)) g = gf_workspace_bytes(L, T, k, E);
    return g > c ? g : c;
}

extern "C" int tsa_moe_prefill_workspace_size(const tsa_expert_layout* layout, int64_t T, int k, int64_t E,
                                              int64_t* bytes) {
    clear_error();
    int rc = validate_layout(layout);
    if (rc) return rc;
    TSA_REQUIRE(T >= 0 && k >= 1 && E >= 1 && bytes, TSA_ERR_INVALID_ARG, "bad T/k/E/bytes");
    *bytes = prefill_ws(*layout, T, k, E);
    return TSA_OK;
}

extern "C" int tsa_moe_prefill(const tsa_expert_layout* layout, const void* pool, int64_t n_slots,
                               const int32_t* expert_slot, int64_t E, const int32_t* idx, const float* weights,
                               int64_t T, int k, const void* x, int x_dtype, void* y, int y_dtype, void* workspace,
                               int64_t workspace_bytes, void* stream) {
    clear_error();
    int rc = validate_layout(layout);
    if (rc) return rc;
    TSA_REQUIRE(T >= 0 && k >= 1 && E >= 1, TSA_ERR_INVALID_ARG, "bad T/k/E");
    if (T == 0) return TSA_OK;
    TSA_REQUIRE(expert_slot && idx && weights, TSA_ERR_INVALID_ARG, "null pointer");
    TSA_REQUIRE(E <= 1024, TSA_ERR_SHAPE, "E %lld exceeds 1024", (long long)E);
    const int64_t need = prefill_ws(*layout, T, k, E);
    TSA_REQUIRE(workspace && workspace_bytes >= need, TSA_ERR_WORKSPACE, "workspace too small: got %lld bytes, need %lld",
                (long long)workspace_bytes, (long long)need);
    if (pf_mxt_supported(*layout, x_dtype, T, k)) {
        TSA_REQUIRE(x && y, TSA_ERR_INVALID_ARG, "null pointer");
        return pf_mxt_prefill(*layout, static_cast<const uint8_t*>(pool), n_slots, expert_slot, E, idx, weights, T, k,
                              static_cast<const uint16_t*>(x), y, y_dtype, static_cast<uint8_t*>(workspace),
                              as_stream(stream));
    }
    if (gf_supported(*layout, x_dtype, T, k) && (reinterpret_cast<uintptr_t>(pool) & 15u) == 0 &&
        (reinterpret_cast<uintptr_t>(x) & 15u) == 0) {
        TSA_REQUIRE(x && y, TSA_ERR_INVALID_ARG, "null pointer");
        return gf_prefill(*layout, static_cast<const uint8_t*>(pool), n_slots, expert_slot, E, idx, weights, T, k,
                          static_cast<const uint16_t*>(x), y, y_dtype, static_cast<uint8_t*>(workspace),
                          as_stream(stream));
    }
    int32_t* slots = static_cast<int32_t*>(workspace);
    const int64_t off = ((T * k * 4 + 255) / 256) * 256;
    hipLaunchKernelGGL(map_slots_kernel, dim3((unsigned)((T * k + 255) / 256)), dim3(256), 0, as_stream(stream), idx,
                       T * k, expert_slot, E, slots);
    TSA_LAUNCH_CHECK();
    return tsa_moe_decode(layout, pool, n_slots, slots, weights, T, k, x, x_dtype, y, y_dtype,
                          static_cast<uint8_t*>(workspace) + off, workspace_bytes - off, stream);
}
