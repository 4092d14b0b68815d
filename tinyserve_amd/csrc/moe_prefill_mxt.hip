// Batched (prefill) MoE over MXFP4 experts in the 16-row MFMA tile order: the grouped
// expert GEMMs on the matrix cores.
//
// After the (token, expert) assignments are sorted expert-major (group_assignments), each
// expert's rows form one contiguous run of the sorted order, cut into tiles of up to 128
// rows (pf_table). Two persistent GEMM launches then cover every (row tile, weight
// tile) pair:
//   gate_up: h[i, :] = SwiGLU(x[token(i)] W_gu^T + b_gu), bf16, in sorted order;
//   down:    yk[a, :] = h[i] W_dn^T + b_dn, bf16, by assignment id a = perm[i]
// (bf16 like the reference's per-expert outputs), and a combine pass forms
// y[t] = sum_j w[t, j] yk[t k + j] over j in order, so every output has one writer and the
// result does not depend on scheduling.
//
// GEMM workgroup: 8 waves, a 256-weight-row x 128-token tile; wave (wn, wt) owns 64 rows
// x 64 tokens = 2 x 2 blocks of v_mfma_f32_32x32x16_bf16 (that form issues at the bf16
// peak with 4 independent chains per wave; 16x16x32 needs about 16). K advances in 128-wide
// pieces. Weights are the A operand: the MXFP4 16-row tile order delivers a 16-row piece
// as one contiguous 1 KB, which v_cvt_scalef32_pk_bf16_fp4 expands exactly (scale folded
// in). Activations are the B operand. Both reach LDS by direct buffer-to-LDS loads issued
// ahead of use (weights, which mostly come from HBM or the MALL, 4 pieces ahead in a 5-deep
// ring; activations, which mostly hit L2, 1 piece ahead), with one wait + barrier per piece.
// Workgroups are persistent, one per CU. XCD x (workgroup b runs on XCD b % 8) owns a
// group of row tiles, with all their weight tiles, in row-tile-major order, so the
// workgroups running together on an XCD share a row tile's activations in its L2. The
// table kernel forms the 8 groups to balance an estimated cost (a tile costs 96 + rows, in
// rows: partial row tiles are cheaper, not free), and each group ends on its cheapest row
// tiles. An XCD's workgroups take its tiles one at a time from a per-XCD counter (the next
// one is requested when a tile starts), so they finish together whatever the tiles cost.
//
// Semantics: tinyserve/expert_pipeline.py:166-239 (group by expert, batched forward,
// weighted scatter), tinyserve/_model_hooks.py:380-394 (MXFP4 expert with biases,
// clamped SwiGLU).

#include "fused_common.h"
#include "mfma_tile.h"
#include "moe_group.h"
#include "fp6_terms.h"

namespace tsa {

int64_t mx_tile_scale_bytes(int64_t K);

namespace {

constexpr int PF_THREADS = 512;
constexpr int PF_BM = 128;                        // sorted rows (tokens) per workgroup tile
constexpr int PF_BN = 256;                        // weight rows per workgroup tile
constexpr int PF_XST = 2;                         // activation stages (mostly L2 hits)
constexpr int PF_WST = 5;                         // weight stages (from HBM / MALL: issued further ahead)
constexpr int PF_XAHEAD = PF_XST - 1;
constexpr int PF_WAHEAD = PF_WST - 1;
static_assert(PF_WAHEAD > PF_XAHEAD && PF_WAHEAD < 5, "weights of piece i must be issued before its activations");
constexpr int PF_XBYTES = PF_BM * 128 * 2;        // a piece of bf16 activations: 32 KB
constexpr int PF_WBYTES = (PF_BN / 16) * 1024;    // a piece of MXFP4 weights: 16 KB
constexpr int PF_SBYTES = (PF_BN / 16) * 256;     // one scale word per lane of every row tile: 4 KB
constexpr int PF_WOFF = PF_XST * PF_XBYTES;
constexpr int PF_SOFF = PF_WOFF + PF_WST * PF_WBYTES;
constexpr int PF_BIAS_OFF = PF_SOFF + 2 * PF_SBYTES;  // the tile's 256 bias values (up to 1 KB)
constexpr int PF_LDS = PF_BIAS_OFF + 1024;            // 153 KB
constexpr int PF_CTR_STRIDE = 32;                 // ints between per-XCD tile counters (one 128-byte line each)
constexpr int PF_CTR_INTS = 2 * 8 * PF_CTR_STRIDE;  // gate_up's 8 counters, then down's
constexpr int PF_HS_GU = 272;   // LDS row stride (bytes) of the staged gate_up outputs: 128 h + 16 B
constexpr int PF_HS_DN = 528;   // ... of the staged down outputs: 256 values + 16 B
static_assert(PF_BM * PF_HS_DN <= PF_LDS, "the staged outputs fit in the stages");
constexpr int PF_COST0 = 96;  // a tile's estimated cost is PF_COST0 + rows (measured: 16 rows ~0.5 x 128 rows)
// fp6 form of the activations (TSA_PREFILL_FP6): a row is a run of records, one per 128-wide
// piece of K: 4 blocks of 32 values, each 24 bytes of hi codes then 24 of lo codes
// (fp6_terms.h), then the 4 hi scale bytes, then 12 bytes of padding (208 = 13 x 16 bytes:
// whole DMA chunks, and a record stride of 52 dwords keeps the operand reads of 8
// consecutive tokens on distinct LDS banks).
constexpr int PF_QREC = 208;
constexpr int PF_QSCALE = 192;
constexpr int PF_QCHUNKS = PF_QREC / 16;

struct PfEntry {
    int slot, row0, rows, expert;
};

struct PfGemm {
    tsa_expert_layout L;
    const uint8_t* pool;
    const int* n_entries;     // device: [0] all table entries, [1 + x] .. [2 + x] XCD x's group
    const PfEntry* table;
    const void* src;          // gate_up: x rows gathered through perm; down: h rows in sorted order
    int64_t src_rows;         // rows of src (bounds of its buffer resource)
    int64_t src_stride;       // bytes per src row (bf16: 2 K; fp6 records: 208 MP)
    const int32_t* perm;      // sorted position -> assignment id (token * k + j)
    int* ctr;                 // 8 per-XCD tile counters (stride PF_CTR_STRIDE), zero at launch
    int k;
    uint16_t* out;            // gate_up: h [n, N / 2] (bf16 form); down: yk [T k, N]
    uint8_t* qout;            // gate_up in the fp6 form: h as fp6 records, rows of out_stride bytes
    int64_t out_stride;
    int N, K, NT, MP;         // weight rows, reduction length, tiles along N, pieces along K
    int64_t w_off, s_off, b_off;        // slot offsets of the tiled blocks, tiled scales, bias (< 0: none)
    int64_t tile_bytes, stile_bytes;    // per 16-row tile
};

typedef int v4i __attribute__((ext_vector_type(4)));
typedef float v16f __attribute__((ext_vector_type(16)));

// Raw buffer descriptor (base, num_records bytes; loads past the end return zero), its
// words from the first lane: the copies' "s" operand must sit in scalar registers, which
// the compiler only guarantees for values it can prove wave-uniform.
__device__ __forceinline__ v4i buf_desc(const void* p, uint32_t bytes) {
    const uint64_t a = reinterpret_cast<uint64_t>(p);
    return v4i{__builtin_amdgcn_readfirstlane((int)(uint32_t)a), __builtin_amdgcn_readfirstlane((int)(uint32_t)(a >> 32)),
               __builtin_amdgcn_readfirstlane((int)bytes), 0x00020000};
}

// 16 (or 4) bytes per lane from buffer offset voff straight into LDS at lds + 16 lane (or
// 4 lane): one contiguous 1 KB (256 B) per wave. Issued as inline assembly so that the
// compiler does not place its conservative vmcnt(0) before every later LDS read: the K loop
// waits for exactly what it needs (pf_wait). Loads return in order, so the compiler's own
// waits for its loads can only get stricter, never too weak.
__device__ __forceinline__ void pf_dma(const v4i& r, uint32_t voff, uint32_t lds) {
    asm volatile("s_mov_b32 m0, %2\n\t" TSA_COPY_WAIT "buffer_load_dwordx4 %0, %1, 0 offen lds" ::"v"(voff), "s"(r), "s"(lds)
                 : "memory", "m0");
}
__device__ __forceinline__ void pf_dma4(const v4i& r, uint32_t voff, uint32_t lds) {
    asm volatile("s_mov_b32 m0, %2\n\t" TSA_COPY_WAIT "buffer_load_dword %0, %1, 0 offen lds" ::"v"(voff), "s"(r), "s"(lds)
                 : "memory", "m0");
}

// This wave's loads except the newest n are complete (and its LDS work), then the
// workgroup barrier: every wave's part of the piece is in LDS, and every wave is done
// reading the stages that are refilled next.
#define PF_WAIT_CASE(n) \
    case n: asm volatile("s_waitcnt vmcnt(" #n ") lgkmcnt(0)\n\ts_barrier" ::: "memory"); break;
__device__ __forceinline__ void pf_wait(int n) {
    switch (n) {  // n above 16 waits for 16 (stricter)
        PF_WAIT_CASE(0) PF_WAIT_CASE(1) PF_WAIT_CASE(2) PF_WAIT_CASE(3) PF_WAIT_CASE(4) PF_WAIT_CASE(5)
        PF_WAIT_CASE(6) PF_WAIT_CASE(7) PF_WAIT_CASE(8) PF_WAIT_CASE(9) PF_WAIT_CASE(10) PF_WAIT_CASE(11)
        PF_WAIT_CASE(12) PF_WAIT_CASE(13) PF_WAIT_CASE(14) PF_WAIT_CASE(15)
        default: asm volatile("s_waitcnt vmcnt(16) lgkmcnt(0)\n\ts_barrier" ::: "memory"); break;
    }
}
#undef PF_WAIT_CASE

// One 128-wide piece of a wave's 64-row x 64-token block on v_mfma_f32_32x32x16_bf16
// (2 x 2 blocks of 32 x 32). K order within the piece: step j (0..7) covers, for lanes
// 32g..32g+31, dword 2g + j%2 of MXFP4 block j/2, so a weight lane (row r, group g) reads
// the 8 contiguous bytes at 16 (16 (j/2) + r%16) + 8g of its 16-row tile, and the
// activation fragment (subtile, j) is one contiguous 1 KB, laid out so by the DMA. NB of
// the 2 token subtiles are live. Lanes whose block starts at or past K get a zero weight
// operand (past the end of a row the bytes belong to the next tile, and the activations
// there are stand-ins).
template <int NB>
__device__ __forceinline__ void pf_piece(v16f (&acc)[2][2], const uint8_t* xs, const uint8_t* ws, const uint8_t* ss,
                                         int mp, int K, int wn, int wt, int lane) {
    const int g = lane >> 5, rr = lane & 31;
    uint2 A[2][4];
    float s[2][4];
#pragma unroll
    for (int rb = 0; rb < 2; ++rb) {
        const int rt = 4 * wn + 2 * rb + (rr >> 4);  // row tile in the workgroup tile
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int lt = 16 * q + (rr & 15);      // the 16-row tile's lane holding this row's block q
            A[rb][q] = *reinterpret_cast<const uint2*>(ws + rt * 1024 + 16 * lt + 8 * g);
            s[rb][q] = e8m0_to_f32(ss[rt * 256 + 4 * lt + (mp & 3)]);
        }
    }
    if (128 * (mp + 1) > K) {  // the row's last, partial piece
#pragma unroll
        for (int rb = 0; rb < 2; ++rb)
#pragma unroll
            for (int q = 0; q < 4; ++q)
                if (128 * mp + 32 * q >= K) A[rb][q] = make_uint2(0u, 0u);
    }
    // activations: token row (64 wt + 32 b + lane % 32) of the piece, chunk 4 (j / 2) + 2g + j % 2
    // stored at slot chunk ^ (token % 16)
    const uint8_t* xrow = xs + (64 * wt + rr) * 256;
    auto bfrag = [&](int b, int j) {
        const int ch = 4 * (j >> 1) + 2 * g + (j & 1);
        return *reinterpret_cast<const bf16x8*>(xrow + b * 32 * 256 + 16 * (ch ^ (rr & 15)));
    };
    bf16x8 B[2][NB];
#pragma unroll
    for (int b = 0; b < NB; ++b) B[0][b] = bfrag(b, 0);
#pragma unroll
    for (int j = 0; j < 8; ++j) {
        if (j < 7) {
#pragma unroll
            for (int b = 0; b < NB; ++b) B[(j + 1) & 1][b] = bfrag(b, j + 1);
        }
        __builtin_amdgcn_sched_barrier(0);  // the next step's reads go out before this step's MFMAs
#pragma unroll
        for (int rb = 0; rb < 2; ++rb) {
            const uint32_t w = (j & 1) ? A[rb][j >> 1].y : A[rb][j >> 1].x;
            const bf16x8 Af = expand(w, s[rb][j >> 1]);
#pragma unroll
            for (int b = 0; b < NB; ++b)
                acc[rb][b] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(Af, B[j & 1][b], acc[rb][b], 0, 0, 0);
        }
        __builtin_amdgcn_sched_barrier(0);
    }
}

typedef int v8i __attribute__((ext_vector_type(8)));

// acc += A (fp4 weights, e8m0 scale sa) x B (fp6 e2m3 activations, scale byte OPB of sb).
template <int OPB>
__device__ __forceinline__ v16f mfma_f4f6(const v8i& a, const v8i& b, const v16f& c, int sa, int sb) {
    return __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(a, b, c, 4, 2, 0, sa, OPB, sb);
}

// The K loop of one tile, as a stream of steps s = -PF_WAHEAD .. MP - 1: step s waits for
// and multiplies piece s (s >= 0), then issues the activations of piece s + PF_XAHEAD and
// the weights of piece s + PF_WAHEAD, in that order. The weights of piece i therefore go
// out in an earlier step than its activations, so once this wave's loads up to X(s) are
// complete, W(s) and its scale word are too; the loads newer than X(s) are counted
// exactly (never fewer than issued: a wait for fewer outstanding is only stricter). NB = 0:
// the wave has no live block in this tile and only takes part in the loads and barriers.
template <int NB, class IX, class IW, class WL>
__device__ __forceinline__ void pf_kloop(v16f (&acc)[2][2], IX& issue_x, IW& issue_w, WL& w_loads, int MP, int K,
                                         int wn, int wt, int lane) {
    extern __shared__ __align__(16) uint8_t smem[];
    auto x_loads = [&](int i) { return i >= 0 && i < MP ? 4 : 0; };
    for (int st = -PF_WAHEAD; st < MP; ++st) {
        if (st >= 0) {
            int newer = w_loads(st - PF_XAHEAD + PF_WAHEAD);
#pragma unroll
            for (int u = st - PF_XAHEAD + 1; u < st; ++u) newer += x_loads(u + PF_XAHEAD) + w_loads(u + PF_WAHEAD);
            pf_wait(newer);
        }
        if (st + PF_XAHEAD >= 0 && st + PF_XAHEAD < MP) issue_x(st + PF_XAHEAD);
        if (st + PF_WAHEAD < MP) issue_w(st + PF_WAHEAD);
        if (NB > 0 && st >= 0) {
            const uint8_t* xs = smem + (st % PF_XST) * PF_XBYTES;
            const uint8_t* ws = smem + PF_WOFF + (st % PF_WST) * PF_WBYTES;
            const uint8_t* ss = smem + PF_SOFF + ((st >> 2) & 1) * PF_SBYTES;
            pf_piece<NB ? NB : 1>(acc, xs, ws, ss, st, K, wn, wt, lane);
        }
    }
}

template <bool GATE_UP>
__global__ void __launch_bounds__(PF_THREADS, 1) pf_gemm_kernel(PfGemm p) {
    extern __shared__ __align__(16) uint8_t smem[];
    const int tid = threadIdx.x, lane = tid & 63, wave = uniform(tid >> 6);
    const int wn = wave & 3, wt = wave >> 2;
    const int g = lane >> 5, rr = lane & 31;
    const int N = p.N, K = p.K, MP = p.MP;
    const int xcd = blockIdx.x & 7, R = gridDim.x >> 3;
    const int m0 = uniform(p.n_entries[1 + xcd]);
    const int total = (uniform(p.n_entries[2 + xcd]) - m0) * p.NT;  // this XCD's tiles
    int* const ctr = p.ctr + PF_CTR_STRIDE * xcd;
    __shared__ int s_next;
    const int W = (int)(p.stile_bytes >> 8);  // scale words per lane
    const uint32_t lds0 = (uint32_t)reinterpret_cast<uintptr_t>(smem);
    const v4i xr = buf_desc(p.src, (uint32_t)(p.src_rows * p.src_stride));

    // The first tile of workgroup b is b / 8; later ones come from the counter (offset by R,
    // so the first R are never handed out twice).
    for (int tl = (int)(blockIdx.x >> 3); tl < total;) {
        const int m = m0 + tl / p.NT, nt = tl % p.NT;
        int grabbed = 0;
        if (tid == 0) grabbed = R + __hip_atomic_fetch_add(ctr, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        const PfEntry e = p.table[m];
        const int slot = uniform(e.slot), row0 = uniform(e.row0), rows = uniform(e.rows);
        const uint8_t* base = p.pool + (int64_t)slot * p.L.slot_bytes;

        // Activation DMA: each instruction copies 4 whole token rows of the piece (4 x 256 B,
        // coalesced): lanes 16 i .. 16 i + 15 carry token 4 (4 w + c) + i (c = 0..3), lane slot
        // s = lane % 16 the row's 16-byte chunk s ^ (token % 16). The swizzle keeps the B
        // fragment reads (one chunk of 32 tokens per lane group) free of bank conflicts.
        // Tokens past the tile's rows re-read token 0's row (their columns are dropped).
        uint32_t xoff[4];
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            int tok = 16 * wave + 4 * c + (lane >> 4);
            if (tok >= rows) tok = 0;
            const int64_t srow = GATE_UP ? p.perm[row0 + tok] / p.k : row0 + tok;
            xoff[c] = (uint32_t)(srow * p.src_stride);
        }
        // Weight DMA: wave w fills row tiles 2w, 2w+1 of the workgroup's 16; one resource
        // spans the workgroup's live tiles (tiles past N read zero).
        const int rtw = nt * (PF_BN / 16);
        int nrw = N / 16 - rtw;
        nrw = nrw > PF_BN / 16 ? PF_BN / 16 : nrw;
        const v4i wr = buf_desc(base + p.w_off + (int64_t)rtw * p.tile_bytes, (uint32_t)(nrw * p.tile_bytes));
        const uint32_t tb = (uint32_t)p.tile_bytes;
        // Scale DMA: with the weights of the first piece of every group of 4, word mp / 4 of
        // the same row tiles (chunked lane-major: word w of a lane at 1024 (w / 4) + 4 width
        // lane + 4 (w % 4), width = min(4, W - 4 (w / 4))) into ring slot (mp / 4) % 2.
        const v4i sr = buf_desc(base + p.s_off + (int64_t)rtw * p.stile_bytes, (uint32_t)(nrw * p.stile_bytes));
        const uint32_t sb = (uint32_t)p.stile_bytes;
        auto issue_x = [&](int mp) {
            const uint32_t st = lds0 + (uint32_t)((mp % PF_XST) * PF_XBYTES) + 16 * wave * 256;
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                const int tok = 16 * wave + 4 * c + (lane >> 4);
                int kk = 128 * mp + 8 * ((lane & 15) ^ (tok & 15));
                if (kk >= K) kk = 0;  // stand-in inside the row; its weight operand is zeroed
                pf_dma(xr, xoff[c] + 2 * kk, st + c * 1024);
            }
        };
        auto issue_w = [&](int mp) {  // 2 loads, + 2 scale loads when mp % 4 == 0
            const uint32_t st = lds0 + PF_WOFF + (uint32_t)((mp % PF_WST) * PF_WBYTES);
#pragma unroll
            for (int jj = 0; jj < 2; ++jj)
                pf_dma(wr, (2 * wave + jj) * tb + 1024 * mp + 16 * lane, st + (2 * wave + jj) * 1024);
            if ((mp & 3) == 0) {
                const int w = mp >> 2;
                const int wc = W - 4 * (w >> 2) < 4 ? W - 4 * (w >> 2) : 4;
#pragma unroll
                for (int jj = 0; jj < 2; ++jj)
                    pf_dma4(sr, (2 * wave + jj) * sb + 1024 * (w >> 2) + 4 * wc * lane + 4 * (w & 3),
                            lds0 + PF_SOFF + (w & 1) * PF_SBYTES + (2 * wave + jj) * 256);
            }
        };
        auto w_loads = [&](int mp) { return mp >= 0 && mp < MP ? 2 + ((mp & 3) == 0 ? 2 : 0) : 0; };

        // This wave's block: row tiles rtw + 4wn .. +3 (two 32-row blocks), tokens 64 wt .. +63.
        const int rt0 = rtw + 4 * wn;
        const bool rows_live = rt0 < N / 16;
        int nsub = (rows - 64 * wt + 31) >> 5;
        nsub = nsub < 0 ? 0 : (nsub > 2 ? 2 : nsub);
        const bool active = rows_live && nsub > 0;

        // The tile's bias, copied into LDS now (wave 0, before the K loop's loads, so that every
        // later wait covers it) and read by the epilogue; rows past N read zero (the buffer
        // range check).
        const int bes = p.L.bias_dtype == TSA_F32 ? 4 : 2;
        if (wave == 0 && p.b_off >= 0) {
            const int64_t brows = N - 16 * rtw;
            const v4i br = buf_desc(base + p.b_off + (int64_t)16 * rtw * bes, (uint32_t)(brows > 0 ? brows * bes : 0));
            for (int i = 0; i < bes; ++i) pf_dma4(br, 256 * i + 4 * lane, lds0 + PF_BIAS_OFF + 256 * i);
        }

        v16f acc[2][2];
#pragma unroll
        for (int a = 0; a < 2; ++a)
#pragma unroll
            for (int b = 0; b < 2; ++b)
#pragma unroll
                for (int v = 0; v < 16; ++v) acc[a][b][v] = 0.0f;
        // One K loop per live-subtile count, so the accumulators keep one register home
        // (a per-piece branch made the compiler copy them after every piece).
        if (!active) pf_kloop<0>(acc, issue_x, issue_w, w_loads, MP, K, wn, wt, lane);
        else if (nsub == 2) pf_kloop<2>(acc, issue_x, issue_w, w_loads, MP, K, wn, wt, lane);
        else pf_kloop<1>(acc, issue_x, issue_w, w_loads, MP, K, wn, wt, lane);
        if (tid == 0) s_next = grabbed;
        __syncthreads();  // every wave is done with the last stages before the next tile refills them
        tl = uniform(s_next);  // rewritten only after the next tile's K loop, which has a barrier per piece

        // Epilogue, 1: the outputs (bias added; SwiGLU for gate_up) as bf16 into LDS, one row
        // per token (the stages are free: every wave is past the K loop's last LDS read).
        // acc[rb][b][4u + r] is row 32 rb + 8u + 4g + r of the wave's 64 (r = 0..3), token
        // column 64 wt + 32 b + (lane % 32).
        constexpr int HS = GATE_UP ? PF_HS_GU : PF_HS_DN;
        if (active) {
#pragma unroll
            for (int rb = 0; rb < 2; ++rb) {
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    const int c = 64 * wn + 32 * rb + 8 * u + 4 * g;  // weight row within the workgroup tile
                    if (16 * rtw + c >= N) continue;  // N % 32 == 16: the block's second row tile is past N
                    const v4f bias = p.b_off >= 0 ? bias_value(*reinterpret_cast<const u32x4*>(smem + PF_BIAS_OFF + c * bes),
                                                               p.L.bias_dtype)
                                                  : v4f{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
                    for (int b = 0; b < 2; ++b) {
                        const int tk = 64 * wt + 32 * b + rr;
                        if (b >= nsub || tk >= rows) continue;
                        const v4f v = v4f{acc[rb][b][4 * u], acc[rb][b][4 * u + 1], acc[rb][b][4 * u + 2], acc[rb][b][4 * u + 3]} + bias;
                        if (GATE_UP)
                            *reinterpret_cast<uint32_t*>(smem + tk * HS + c) =
                                pack_bf16x2(swiglu_oai_fast(p.L, v[0], v[1]), swiglu_oai_fast(p.L, v[2], v[3]));
                        else
                            *reinterpret_cast<uint2*>(smem + tk * HS + 2 * c) = make_uint2(pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3]));
                    }
                }
            }
        }
        __syncthreads();
        // 2: whole rows out, 16 bytes (8 values) per lane, consecutive lanes along a row:
        // gate_up h[row0 + tk, 128 nt ..] (256 B a row), down yk[perm[row0 + tk], 256 nt ..] (512 B).
        constexpr int CPR = GATE_UP ? 16 : 32;  // 16-byte chunks per row
        const int ncol = GATE_UP ? N / 2 - 128 * nt : N - 256 * nt;  // live values in the row (multiple of 8)
#pragma unroll
        for (int j = 0; j < PF_BM * CPR / PF_THREADS; ++j) {
            const int i = tid + PF_THREADS * j, tk = i / CPR, ch = i % CPR;
            if (tk >= rows || 8 * ch >= ncol) continue;
            const uint4 v = *reinterpret_cast<const uint4*>(smem + tk * HS + 16 * ch);
            if (GATE_UP) {
                *reinterpret_cast<uint4*>(p.out + (int64_t)(row0 + tk) * (N / 2) + 128 * nt + 8 * ch) = v;
            } else {
                const int64_t asg = p.perm[row0 + tk];
                *reinterpret_cast<uint4*>(p.out + asg * N + 256 * nt + 8 * ch) = v;
            }
        }
        __syncthreads();  // the staged rows are read before the next tile's loads refill the stages
    }
}

// ---- the fp6 form's GEMM (pf6_gemm_kernel)
//
// The same tile (256 weight rows x 128 sorted rows, wave (wn, wt) 64 x 64), schedule and sorted
// rows as pf_gemm_kernel, on v_mfma_scale_f32_32x32x64_f8f6f4 with the weights as stored (fp4,
// e8m0 scales) against the activations' fp6 hi and lo terms. What bounds it: the LDS (a piece
// moves about 43 KB in and 132 KB out of it, as long as its 128 MFMAs take) and the copies,
// with the matrix cores busy a third of the time; so the K loop is kept free of everything
// else:
//  - one stream of pieces over all of a workgroup's tiles: the next tile is asked for as a tile
//    starts, and its first pieces are copied while the last ones multiply and the epilogue,
//    which works in registers, runs (rows of fewer than P6_STREAM pieces restart per tile);
//  - activations are copied by waves 0 .. 3 and weights by waves 4 .. 7, so each wave waits
//    only for its own kind: loads return in order, and a wave waiting for the activations 2
//    pieces ahead would also wait for the weights 3 ahead;
//  - a K step's operands are read while the step before multiplies, across the barrier;
//  - the starts, ends and hand-overs of tiles keep about 155 scalar registers in lanes; a copy that
//    reads one of them back has its wait states (TSA_COPY_WAIT);
//  - stage positions are running byte offsets, LDS destinations immediates of the copies; the
//    steady part of the loop has no tail checks, the tile's last 4 pieces are written out.
// 2880 x 2880, top-4 of 32 experts, whole call (us; one loop with all reads and waits at its top
// before, now): 2048 tokens 453 -> 425, 700 260 -> 238, 128 162 -> 148, 24 125 -> 115, 5 83 -> 77.
// (Reads and copies placed between the MFMAs instead of ahead of them: 436 us at 2048 tokens.)

// LDS of pf6_gemm_kernel: three activation stages, four weight stages, a ring of three scale
// groups (one word per lane of the 16 row tiles: 4 pieces), two tiles' biases and permutations.
constexpr int P6_XB = PF_BM * PF_QREC;  // 26 KB
constexpr int P6_XST = 3, P6_WST = 4;
constexpr int P6_WOFF = P6_XST * P6_XB;
constexpr int P6_SOFF = P6_WOFF + P6_WST * PF_WBYTES;
constexpr int P6_BOFF = P6_SOFF + 3 * PF_SBYTES;
constexpr int P6_POFF = P6_BOFF + 2 * 1024;
constexpr int P6_LDS = P6_POFF + 2 * PF_BM * 4;
static_assert(P6_LDS <= 160 * 1024, "LDS per workgroup");
constexpr int P6_STREAM = 8;  // rows of at least this many pieces run on into the next tile (fewer cannot:
                              // the next tile is known after 3 pieces, its copies start 4 before the end)

// pf_dma / pf_dma4 to lds + IMM, with a scalar byte offset soff added to voff.
template <int IMM>
__device__ __forceinline__ void p6_dma(const v4i& r, uint32_t voff, uint32_t soff, uint32_t lds) {
    asm volatile("s_add_u32 m0, %3, %4\n\t" TSA_COPY_WAIT "buffer_load_dwordx4 %0, %1, %2 offen lds" ::"v"(voff), "s"(r), "s"(soff),
                 "s"(__builtin_amdgcn_readfirstlane((int)lds)), "n"(IMM)
                 : "memory", "m0", "scc");
}
template <int IMM>
__device__ __forceinline__ void p6_dma4(const v4i& r, uint32_t voff, uint32_t soff, uint32_t lds) {
    asm volatile("s_add_u32 m0, %3, %4\n\t" TSA_COPY_WAIT "buffer_load_dword %0, %1, %2 offen lds" ::"v"(voff), "s"(r), "s"(soff),
                 "s"(__builtin_amdgcn_readfirstlane((int)lds)), "n"(IMM)
                 : "memory", "m0", "scc");
}

// One table entry by a scalar load (after an inline-assembly copy the compiler would use a
// vector load, whose wait would also wait for the copies).
__device__ __forceinline__ PfEntry p6_entry(const PfEntry* t) {
    v4i e;
    asm volatile("s_load_dwordx4 %0, %1, 0x0\n\ts_waitcnt lgkmcnt(0)" : "=&s"(e) : "s"(t) : "memory");
    return PfEntry{e[0], e[1], e[2], e[3]};
}

// One K step's operands (64 values: blocks 2 ks + q of a piece) of a wave's 64 rows x 64 tokens
// on v_mfma_scale_f32_32x32x64_f8f6f4, 2 x 2 blocks of 32 x 32: lane (q, r) = (lane / 32,
// lane % 32) holds the 16 bytes of block 2 ks + q of weight row 32 rb + r and its scale byte,
// and that block's 24 bytes of hi and 24 of lo codes of token column 32 b + r.
typedef uint32_t u32x12 __attribute__((ext_vector_type(12)));
struct P6Ops {
    u32x4 A[2];
    u32x12 B[2];  // hi in dwords 0 .. 5, lo in 6 .. 11
    int sa[2];
};

template <bool GATE_UP>
__global__ void __launch_bounds__(PF_THREADS) pf6_gemm_kernel(PfGemm p) {
    extern __shared__ __align__(16) uint8_t smem[];
    __shared__ int s_next;
    const int tid = threadIdx.x, lane = tid & 63, wave = uniform(tid >> 6);
    const int wn = wave & 3, wt = wave >> 2, q = lane >> 5, rr = lane & 31;
    const int N = p.N, K = p.K, MP = p.MP, NT = p.NT;
    const int xcd = blockIdx.x & 7, R = gridDim.x >> 3;
    const int m0 = uniform(p.n_entries[1 + xcd]);
    const int total = (uniform(p.n_entries[2 + xcd]) - m0) * NT;  // this XCD's tiles
    int* const ctr = p.ctr + PF_CTR_STRIDE * xcd;
    const int W = (int)(p.stile_bytes >> 8);  // scale words per lane
    const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t*)smem;
    const v4i xr = buf_desc(p.src, (uint32_t)(p.src_rows * p.src_stride));
    const uint32_t tb = (uint32_t)p.tile_bytes, sb = (uint32_t)p.stile_bytes;
    const int bes = p.L.bias_dtype == TSA_F32 ? 4 : 2;
    const bool xw = wave < 4;                 // waves 0 .. 3 copy activations, 4 .. 7 weights and scales
    const bool stream = MP >= P6_STREAM;

    // The first tile of workgroup b is b / 8; later ones come from the counter (offset by R,
    // so the first R are never handed out twice).
    int tl = (int)(blockIdx.x >> 3);
    if (tl >= total) return;

    struct Tile { int row0, rows, nt; const uint8_t* base; };
    auto tile = [&](int t) {
        const int m = t / NT;
        const PfEntry e = p6_entry(p.table + m0 + m);
        return Tile{e.row0, e.rows, t - m * NT, p.pool + (int64_t)e.slot * p.L.slot_bytes};
    };

    int xg = 0, wg = 0, sg = 0;  // byte offsets of the stage / slot the next piece is copied into
    int xc = 0, wc = 0, sc = 0;  // ... and of the current piece's
    auto next3 = [](int v, int step) { return v == 2 * step ? 0 : v + step; };
    auto next4 = [](int v, int step) { return v == 3 * step ? 0 : v + step; };

    // What the copying waves hold of the tile they copy. Activations: instruction i of a piece's
    // 26 carries 16-byte chunks 64 i + lane of its 128 records (wave w: i = w + 4 c); rows past
    // the tile re-read token 0's, and whole instructions past the last 32 rows are left out
    // (their columns are dropped). Weights: wave 4 + w fills row tiles 4 w .. 4 w + 3.
    uint32_t xoff[7];
    int xin = 0;
    v4i wr = xr, sr = xr;
    auto copy_perm = [&](const Tile& t, int ps) {  // wave 1: the tile's 128 permutation entries
        if (wave == 1) {
            const v4i pr = buf_desc(p.perm + t.row0, 4u * (uint32_t)t.rows);
#pragma unroll
            for (int i = 0; i < 2; ++i) pf_dma4(pr, 256 * i + 4 * lane, lds0 + P6_POFF + 512 * ps + 256 * i);
        }
    };
    auto set_x = [&](const Tile& t, int ps) {
        xin = (((t.rows + 31) & ~31) * PF_QCHUNKS + 63) / 64;
        if (!xw) return;
        int ln = lane;
        asm volatile("" : "+v"(ln));  // per tile, not kept in registers over the K loop
        const uint32_t stride = (uint32_t)p.src_stride;
#pragma unroll
        for (int c = 0; c < 7; ++c) {
            const uint32_t ci = 64 * (wave + 4 * c) + ln;
            uint32_t tok = ci / PF_QCHUNKS;
            const uint32_t ch = ci - PF_QCHUNKS * tok;
            if ((int)tok >= t.rows) tok = 0;
            const uint32_t srow =
                GATE_UP ? *reinterpret_cast<const uint32_t*>(smem + P6_POFF + 512 * ps + 4 * tok) / (uint32_t)p.k : t.row0 + tok;
            xoff[c] = srow * stride + 16 * ch;
        }
    };
    auto set_w = [&](const Tile& t) {
        const int rtw = t.nt * (PF_BN / 16);
        int nrw = N / 16 - rtw;
        nrw = nrw > PF_BN / 16 ? PF_BN / 16 : nrw;  // tiles past N read zero
        wr = buf_desc(t.base + p.w_off + (int64_t)rtw * p.tile_bytes, (uint32_t)nrw * tb);
        sr = buf_desc(t.base + p.s_off + (int64_t)rtw * p.stile_bytes, (uint32_t)nrw * sb);
    };
    // Piece mp of the tile set last, into its stage (the bias with the first activations).
    auto issue_x = [&](const Tile& t, int mp, int bs) {
        if (mp == 0 && wave == 0 && p.b_off >= 0) {
            const int64_t brows = N - PF_BN * t.nt;
            const v4i br = buf_desc(t.base + p.b_off + (int64_t)PF_BN * t.nt * bes, (uint32_t)(brows > 0 ? brows * bes : 0));
            for (int i = 0; i < bes; ++i) pf_dma4(br, 256 * i + 4 * lane, lds0 + P6_BOFF + 1024 * bs + 256 * i);
        }
        const uint32_t dst = lds0 + (uint32_t)xg + 1024u * (uint32_t)wave, so = (uint32_t)mp * PF_QREC;
        if (xin == 26) {  // more than 96 rows: every instruction (6 or 7 of each wave)
            p6_dma<0>(xr, xoff[0], so, dst);
            p6_dma<4096>(xr, xoff[1], so, dst);
            p6_dma<2 * 4096>(xr, xoff[2], so, dst);
            p6_dma<3 * 4096>(xr, xoff[3], so, dst);
            p6_dma<4 * 4096>(xr, xoff[4], so, dst);
            p6_dma<5 * 4096>(xr, xoff[5], so, dst);
            if (wave < 2) p6_dma<6 * 4096>(xr, xoff[6], so, dst);
        } else {
            p6_dma<0>(xr, xoff[0], so, dst);
            if (wave + 4 < xin) p6_dma<4096>(xr, xoff[1], so, dst);
            if (wave + 8 < xin) p6_dma<2 * 4096>(xr, xoff[2], so, dst);
            if (wave + 12 < xin) p6_dma<3 * 4096>(xr, xoff[3], so, dst);
            if (wave + 16 < xin) p6_dma<4 * 4096>(xr, xoff[4], so, dst);
        }
    };
    const uint32_t t4 = 4 * (uint32_t)(wave & 3);
    uint32_t wo[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) wo[i] = (t4 + i) * tb + 16 * lane;
    auto issue_w = [&](int mp) {  // 4 loads, and 4 of the group's scale words when mp % 4 == 0
        const uint32_t dst = lds0 + P6_WOFF + (uint32_t)wg + 1024u * t4, so = 1024u * (uint32_t)mp;
        p6_dma<0>(wr, wo[0], so, dst);
        p6_dma<1024>(wr, wo[1], so, dst);
        p6_dma<2048>(wr, wo[2], so, dst);
        p6_dma<3072>(wr, wo[3], so, dst);
        if ((mp & 3) == 0) {
            const int w = mp >> 2, nw = W - 4 * (w >> 2) < 4 ? W - 4 * (w >> 2) : 4;
            const uint32_t sd = lds0 + P6_SOFF + (uint32_t)sg + 256u * t4, v = t4 * sb + 4 * nw * lane;
            const uint32_t ss = 1024 * (w >> 2) + 4 * (w & 3);
            p6_dma4<0>(sr, v, ss, sd);
            p6_dma4<256>(sr, v + sb, ss, sd);
            p6_dma4<512>(sr, v + 2 * sb, ss, sd);
            p6_dma4<768>(sr, v + 3 * sb, ss, sd);
        }
    };
    // every wave keeps every position (a store behind a branch on the wave's role would put them
    // in memory): after activations, and after weights of piece mp (end: the tile's last)
    auto next_x = [&]() { xg = next3(xg, P6_XB); };
    auto next_w = [&](int mp, bool end) {
        wg = next4(wg, PF_WBYTES);
        sg = (mp & 3) == 3 || end ? next3(sg, PF_SBYTES) : sg;
    };

    P6Ops o0, o1;
    int sh[2];
    uint32_t shn[2] = {0u, 0u};

    // Operand reads: lane-dependent bases, everything else scalar or an immediate. Blocks at or
    // past K get a zero weight operand with a unit scale (their activation records are zero, but
    // the weight bytes and scales there belong to the next tile).
    const uint8_t* const xb = smem + (64 * wt + rr) * PF_QREC + 48 * q;
    const uint8_t* const xsb = smem + (64 * wt + rr) * PF_QREC + PF_QSCALE;
    const uint8_t* const wb = smem + P6_WOFF + (4 * wn + (rr >> 4)) * 1024 + 16 * (16 * q + (rr & 15));
    const uint8_t* const sbp = smem + P6_SOFF + (4 * wn + (rr >> 4)) * 256 + 4 * (16 * q + (rr & 15));
    auto read_a = [&](P6Ops& o, int ks, int mp) {
        const uint8_t* w = wb + wc + 512 * ks;
        const uint8_t* s = sbp + sc + (mp & 3) + 128 * ks;
#pragma unroll
        for (int rb = 0; rb < 2; ++rb) {
            o.A[rb] = *reinterpret_cast<const u32x4*>(w + 2048 * rb);
            o.sa[rb] = s[512 * rb];
        }
    };
    auto read_b = [&](P6Ops& o, int ks, int b) {
        const u32x4* xp = reinterpret_cast<const u32x4*>(xb + xc + 96 * ks + 32 * b * PF_QREC);
        const u32x4 d0 = xp[0], d1 = xp[1], d2 = xp[2];
        const auto d01 = __builtin_shufflevector(d0, d1, 0, 1, 2, 3, 4, 5, 6, 7);
        const auto d2x = __builtin_shufflevector(d2, d2, 0, 1, 2, 3, -1, -1, -1, -1);
        o.B[b] = __builtin_shufflevector(d01, d2x, 0, 1, 2, 3, 4, 5, 6, 7, 8, 9, 10, 11);
    };
    auto past_k = [&](P6Ops& o, int ks, int mp, bool tail) {
        if (tail && 128 * mp + 64 * ks + 64 > K && 128 * mp + 32 * (2 * ks + q) >= K) {
#pragma unroll
            for (int rb = 0; rb < 2; ++rb) {
                o.A[rb] = u32x4{0u, 0u, 0u, 0u};
                o.sa[rb] = 127;
            }
        }
    };
    // the two columns' hi scales of a piece: block q in byte 0, block 2 + q in byte 2
    auto read_scales = [&]() {
#pragma unroll
        for (int b = 0; b < 2; ++b)
            shn[b] = *reinterpret_cast<const uint32_t*>(xsb + xc + 32 * b * PF_QREC);
    };
    auto use_scales = [&]() {
#pragma unroll
        for (int b = 0; b < 2; ++b) sh[b] = (int)(shn[b] >> (8 * q));
    };

    v16f acc[2][2];
    int nsub = 0;  // the wave's live 32-token columns
    // One column's hi or lo products of a K step, both row blocks.
    auto mul = [&](const P6Ops& o, auto ksc, int b, bool low) {
        constexpr int KS = decltype(ksc)::value;
        if (nsub <= b) return;
        const v8i t = low ? __builtin_bit_cast(v8i, __builtin_shufflevector(o.B[b], o.B[b], 6, 7, 8, 9, 10, 11, -1, -1))
                          : __builtin_bit_cast(v8i, __builtin_shufflevector(o.B[b], o.B[b], 0, 1, 2, 3, 4, 5, -1, -1));
        const int sb = low ? sh[b] - 0x05050505 : sh[b];  // lo scale = hi scale - 5 (every scale byte is >= 5)
#pragma unroll
        for (int rb = 0; rb < 2; ++rb)
            acc[rb][b] = mfma_f4f6<2 * KS>(
                __builtin_bit_cast(v8i, __builtin_shufflevector(o.A[rb], o.A[rb], 0, 1, 2, 3, -1, -1, -1, -1)), t, acc[rb][b],
                o.sa[rb], sb);
    };
    // the MFMAs stay on this side of the next barrier (the compiler would sink them past it)
    auto pin = [&]() {
#pragma unroll
        for (int rb = 0; rb < 2; ++rb)
#pragma unroll
            for (int b = 0; b < 2; ++b) asm volatile("" : "+v"(acc[rb][b]));
    };
    // Step 1's operands are read while step 0 multiplies ..
    using K0 = std::integral_constant<int, 0>;
    using K1 = std::integral_constant<int, 1>;
    auto front = [&](int mp, bool tail) {
        read_a(o1, 1, mp);
        read_b(o1, 1, 0);
        read_b(o1, 1, 1);
        __builtin_amdgcn_sched_barrier(0);
        mul(o0, K0{}, 0, false);
        mul(o0, K0{}, 0, true);
        mul(o0, K0{}, 1, false);
        mul(o0, K0{}, 1, true);
        __builtin_amdgcn_sched_barrier(0);
        past_k(o1, 1, mp, tail);
        pin();
    };
    // .. and, after the copies, step 0's of the next piece (nmp) while step 1 multiplies.
    auto back = [&](int nmp, bool next, bool tail, auto copy) {
        copy();
        if (next) {
            xc = next3(xc, P6_XB);
            wc = next4(wc, PF_WBYTES);
            sc = (nmp & 3) == 0 ? next3(sc, PF_SBYTES) : sc;
            read_a(o0, 0, nmp);
            read_b(o0, 0, 0);
            read_b(o0, 0, 1);
            read_scales();
        }
        __builtin_amdgcn_sched_barrier(0);
        mul(o1, K1{}, 0, false);
        mul(o1, K1{}, 0, true);
        mul(o1, K1{}, 1, false);
        mul(o1, K1{}, 1, true);
        __builtin_amdgcn_sched_barrier(0);
        if (next) past_k(o0, 0, nmp, tail);
        use_scales();
        pin();
    };
    // This wave's copies but the newest have landed (activations: all but the n of one piece;
    // weights: all but two pieces', 8 copies and 4 more if one of them begins a scale group),
    // then the barrier: piece st + 1 is in LDS and every wave holds piece st in registers.
    auto wait_x = [&](int n) {  // n <= the wave's copies of a piece: 1, 3, 5 or 6 by the tile's 32-row groups
        if (n >= 5) {
            if (n == 6) asm volatile("s_waitcnt vmcnt(6) lgkmcnt(0)\n\ts_barrier" ::: "memory");
            else asm volatile("s_waitcnt vmcnt(5) lgkmcnt(0)\n\ts_barrier" ::: "memory");
        } else {
            if (n == 3) asm volatile("s_waitcnt vmcnt(3) lgkmcnt(0)\n\ts_barrier" ::: "memory");
            else asm volatile("s_waitcnt vmcnt(1) lgkmcnt(0)\n\ts_barrier" ::: "memory");
        }
    };
    auto wait_w = [&](bool group) {
        if (group) asm volatile("s_waitcnt vmcnt(12) lgkmcnt(0)\n\ts_barrier" ::: "memory");
        else asm volatile("s_waitcnt vmcnt(8) lgkmcnt(0)\n\ts_barrier" ::: "memory");
    };
    auto x_class = [&](int rows) { return rows > 96 ? 6 : rows > 64 ? 5 : rows > 32 ? 3 : 1; };

    Tile cur = tile(tl), nxt = cur;
    int ps = 0;         // the current tile's bias and permutation slot
    bool fresh = true;  // nothing of the current tile is in flight yet
    for (;;) {
        if (fresh) {  // start the stream: the first tile, or a tile after rows too short to run on
            copy_perm(cur, ps);
            pf_wait(0);
            set_x(cur, ps);
            set_w(cur);
            for (int i = 0; i < 4 && i < MP; ++i) {
                if (xw) {
                    if (i < 3) issue_x(cur, i, ps);
                } else {
                    issue_w(i);
                }
                if (i < 3) next_x();
                next_w(i, i == MP - 1);
            }
            pf_wait(0);
            read_a(o0, 0, 0);
            read_b(o0, 0, 0);
            read_b(o0, 0, 1);
            past_k(o0, 0, 0, true);
            read_scales();
            use_scales();
            fresh = false;
        }
        nsub = (cur.rows - 64 * wt + 31) >> 5;
        nsub = cur.nt * (PF_BN / 16) + 4 * wn >= N / 16 || nsub < 0 ? 0 : (nsub > 2 ? 2 : nsub);
#pragma unroll
        for (int a = 0; a < 2; ++a)
#pragma unroll
            for (int b = 0; b < 2; ++b)
#pragma unroll
                for (int v = 0; v < 16; ++v) acc[a][b][v] = 0.0f;

        // Piece st multiplies while the copies run ahead, activations by 3 pieces, weights by 4,
        // past the tile's end those of the next tile. The epilogue needs no stage, so the stream
        // runs on under it.
        bool more = false;  // the next tile is known and runs on in the stream
        if (stream) {
            int grabbed = 0;
            const int xn = x_class(cur.rows);
            for (int st = 0; st < MP - 4; ++st) {
                front(st, false);
                if (xw) wait_x(xn);
                else wait_w(((st + 2) & 3) == 0 || ((st + 3) & 3) == 0);
                if (st < 3) {  // the next tile: asked for, announced, read
                    if (st == 0) {
                        if (tid == 0) grabbed = R + __hip_atomic_fetch_add(ctr, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    } else if (st == 1) {
                        if (tid == 0) s_next = grabbed;
                    } else {
                        tl = uniform(s_next);
                        more = tl < total;
                        if (more) {
                            nxt = tile(tl);
                            copy_perm(nxt, ps ^ 1);
                        }
                    }
                }
                back(st + 1, true, false, [&]() {
                    if (xw) issue_x(cur, st + 3, ps);
                    else issue_w(st + 4);
                    next_x();
                    next_w(st + 4, st + 4 == MP - 1);
                });
            }
#pragma unroll
            for (int e = 4; e >= 1; --e) {  // the last four pieces, st = MP - e
                const int st = MP - e;
                front(st, e == 1);
                if (e > 1 || more) {
                    // (waits for all of a piece that may be absent or of another size: a few stricter ones a tile)
                    if (xw) {
                        if (e > 2) wait_x(xn);
                        else pf_wait(0);
                    } else if (more || e == 4) {
                        wait_w(e == 2);  // then the next tile's pieces 0 (a group's first) and 1 are newer
                    } else {
                        pf_wait(0);
                    }
                }
                back(e == 1 ? 0 : st + 1, e > 1 || more, e == 2, [&]() {
                    if (xw) {
                        if (e == 4) {
                            issue_x(cur, MP - 1, ps);
                        } else if (more) {
                            if (e == 3) set_x(nxt, ps ^ 1);
                            issue_x(nxt, 3 - e, ps ^ 1);
                        }
                    } else if (more) {
                        if (e == 4) set_w(nxt);
                        issue_w(4 - e);
                    }
                    next_x();
                    next_w(4 - e, false);
                });
            }
        } else {
            for (int st = 0; st < MP; ++st) {
                front(st, true);
                if (st + 1 < MP) {
                    pf_wait(0);
                }
                back(st + 1, st + 1 < MP, true, [&]() {
                    if (xw && st + 3 < MP) issue_x(cur, st + 3, ps);
                    if (!xw && st + 4 < MP) issue_w(st + 4);
                    next_x();
                    next_w(st + 4, st + 4 == MP - 1);
                });
            }
        }

        // Epilogue, in registers. acc[rb][b][4u + i] is row 32 rb + 8u + 4q + i of the wave's 64,
        // token 64 wt + 32 b + rr: lane halves hold the halves of a token's run of rows, and a
        // swap of column 1 of the lower lanes with column 0 of the upper ones
        // (v_permlane32_swap) gives lane l all of token 64 wt + l's.
        const int tk = 64 * wt + lane;
        const uint8_t* bias = smem + P6_BOFF + 1024 * ps;
        auto rows4 = [&](int rb, int u, int b) {  // the lane's 4 rows with their bias
            const int c = 64 * wn + 32 * rb + 8 * u + 4 * q;
            v4f v = v4f{acc[rb][b][4 * u], acc[rb][b][4 * u + 1], acc[rb][b][4 * u + 2], acc[rb][b][4 * u + 3]};
            if (p.b_off >= 0) v += bias_value(*reinterpret_cast<const u32x4*>(bias + c * bes), p.L.bias_dtype);
            return v;
        };
        if (nsub > 0) {
            if constexpr (GATE_UP) {  // the wave's 64 rows are one 32-value block of h: its fp6 terms to the row's record
                float v[32];
#pragma unroll
                for (int rb = 0; rb < 2; ++rb)
#pragma unroll
                    for (int u = 0; u < 4; ++u) {
                        const v4f a = rows4(rb, u, 0), b = rows4(rb, u, 1);
#pragma unroll
                        for (int i = 0; i < 2; ++i) {
                            const float h0 = swiglu_oai_fast(p.L, a[2 * i], a[2 * i + 1]);
                            const float h1 = swiglu_oai_fast(p.L, b[2 * i], b[2 * i + 1]);
                            const auto s = __builtin_amdgcn_permlane32_swap(__float_as_uint(h0), __float_as_uint(h1), false, false);
                            v[16 * rb + 4 * u + i] = __uint_as_float(s[0]);
                            v[16 * rb + 4 * u + 2 + i] = __uint_as_float(s[1]);
                        }
                    }
                if (tk < cur.rows) {
                    uint32_t hi[6], lo[6];
                    const uint32_t scl = fp6_terms(v, hi, lo);
                    uint8_t* rec = p.qout + (int64_t)(cur.row0 + tk) * p.out_stride + (int64_t)cur.nt * PF_QREC;
                    *reinterpret_cast<uint4*>(rec + 48 * wn) = make_uint4(hi[0], hi[1], hi[2], hi[3]);
                    *reinterpret_cast<uint4*>(rec + 48 * wn + 16) = make_uint4(hi[4], hi[5], lo[0], lo[1]);
                    *reinterpret_cast<uint4*>(rec + 48 * wn + 32) = make_uint4(lo[2], lo[3], lo[4], lo[5]);
                    rec[PF_QSCALE + wn] = (uint8_t)scl;
                }
            } else {
                const int64_t asg = *reinterpret_cast<const int*>(smem + P6_POFF + 512 * ps + 4 * tk);
                uint16_t* dst = p.out + asg * N + PF_BN * cur.nt + 64 * wn;
#pragma unroll
                for (int rb = 0; rb < 2; ++rb)
#pragma unroll
                    for (int u = 0; u < 4; ++u) {
                        const v4f a = rows4(rb, u, 0), b = rows4(rb, u, 1);
                        const auto s0 = __builtin_amdgcn_permlane32_swap(pack_bf16x2(a[0], a[1]), pack_bf16x2(b[0], b[1]), false, false);
                        const auto s1 = __builtin_amdgcn_permlane32_swap(pack_bf16x2(a[2], a[3]), pack_bf16x2(b[2], b[3]), false, false);
                        if (tk < cur.rows && PF_BN * cur.nt + 64 * wn + 32 * rb + 8 * u < N)
                            *reinterpret_cast<uint4*>(dst + 32 * rb + 8 * u) = make_uint4(s0[0], s1[0], s0[1], s1[1]);
                    }
            }
        } else if constexpr (GATE_UP) {  // blocks past the row's end: zero codes with a unit scale
            const int cb = 4 * cur.nt + wn;
            if (32 * cb >= N / 2 && tk < cur.rows) {
                uint8_t* rec = p.qout + (int64_t)(cur.row0 + tk) * p.out_stride + (int64_t)cur.nt * PF_QREC;
#pragma unroll
                for (int i = 0; i < 3; ++i) *reinterpret_cast<uint4*>(rec + 48 * wn + 16 * i) = make_uint4(0u, 0u, 0u, 0u);
                rec[PF_QSCALE + wn] = 127;
            }
        }
        if (more) {
            cur = nxt;
            ps ^= 1;
            continue;
        }
        if (stream) return;  // no tile left
        if (tid == 0) s_next = R + __hip_atomic_fetch_add(ctr, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __syncthreads();
        tl = uniform(s_next);
        if (tl >= total) return;
        cur = tile(tl);
        xg = wg = sg = xc = wc = sc = 0;
        fresh = true;
        __syncthreads();  // s_next is read and every wave is done with the tile before it is refilled
    }
}

// Tile table: expert e with a resident slot and c_e sorted rows gets ceil(c_e / 128)
// entries (slot, first sorted row, rows, e), in 8 contiguous groups, one per XCD of the
// GEMM launches: n_entries[1 + x] .. n_entries[2 + x] for XCD x, n_entries[0] = all. The
// full 128-row entries (experts in order) are cut into 8 contiguous runs, so an expert's
// row tiles stay on few XCDs and share its weights in L2; then the partial ones, largest
// first, each go to the group with the least estimated cost so far (PF_COST0 + rows per
// entry). Within a group the full entries come first, then the partial ones largest first. Equal-row partial entries are ranked in any order: the results do not
// depend on the order. Also zeroes the GEMMs' tile counters. 1024 threads, E <= 1024; cnt: E
// ints of LDS.
__device__ __forceinline__ void pf_table(const int32_t* __restrict__ idx, int64_t n,
                                         const int32_t* __restrict__ expert_slot, int E, int64_t n_slots,
                                         int* __restrict__ n_entries, PfEntry* __restrict__ table,
                                         int* __restrict__ ctr, int* cnt) {
    __shared__ int wsum[16];
    __shared__ int hist[PF_BM];    // partial entries with r rows
    __shared__ int pos[PF_BM];     // rank (offset by the full entries) of the next partial entry with r rows
    __shared__ int prow[1024];     // partial entries by rank: rows
    __shared__ int pgrp[1024], pidx[1024];  // ... group and place among the group's partial entries
    __shared__ int gstart[8], gfull[8];
    const int e = threadIdx.x;
    if (e < PF_CTR_INTS) ctr[e] = 0;
    if (e < PF_BM) hist[e] = 0;
    int slot = -1, c = 0, nt = 0, r = 0;
    if (e < E) {
        cnt[e] = 0;
        slot = expert_slot[e];
    }
    __syncthreads();
    for (int64_t a0 = e; a0 < n; a0 += 1024 * GROUP_AHEAD) {  // the experts' counts
        int ev[GROUP_AHEAD];
#pragma unroll
        for (int j = 0; j < GROUP_AHEAD; ++j) ev[j] = a0 + 1024 * j < n ? idx[a0 + 1024 * j] : -1;
#pragma unroll
        for (int j = 0; j < GROUP_AHEAD; ++j)
            if (ev[j] >= 0 && ev[j] < E) atomicAdd(&cnt[ev[j]], 1);
    }
    __syncthreads();
    if (e < E) c = cnt[e];
    if (slot >= 0 && slot < n_slots) {
        nt = c / PF_BM;
        r = c % PF_BM;
    }
    int all_rows;
    const int o = block_incl_sum(c, wsum, all_rows) - c;  // the expert's first sorted row
    __syncthreads();  // hist cleared
    if (r > 0) atomicAdd(&hist[r], 1);
    int F;
    const int pre = block_incl_sum(nt, wsum, F);  // inclusive scan of the full entries (its barriers order hist)
    // pos[b] = F + partial entries with more than b rows: F + all of hist - its inclusive
    // prefix sum to b, by wave 0 (lane l: b = 2l, 2l + 1)
    static_assert(PF_BM == 128, "two hist entries per lane of one wave");
    if (e < 64) {
        const int h0 = hist[2 * e], h1 = hist[2 * e + 1];
        int s = h0 + h1;
        for (int d = 1; d < 64; d <<= 1) {
            const int t = __shfl_up(s, d, 64);
            if (e >= d) s += t;
        }
        const int all = __shfl(s, 63, 64);
        pos[2 * e] = F + all - (s - h1);
        pos[2 * e + 1] = F + all - s;
    }
    __syncthreads();
    const int P = pos[0] - F;
    __syncthreads();  // pos[0] is read before the partial entries take ranks (r > 0 never touches it)
    int q = -1;
    if (r > 0) {
        q = atomicAdd(&pos[r], 1) - F;
        prow[q] = r;
    }
    __syncthreads();
    if (e < 64) {  // the groups, by wave 0: lane x < 8 holds group x; P <= E steps of an argmin
        const int x = e;
        const int nf = x < 8 ? F * (x + 1) / 8 - F * x / 8 : 0;
        int cost = x < 8 ? nf * (PF_COST0 + PF_BM) : 0x7FFFFFFF, np = 0;
        int rn = P > 0 ? prow[0] : 0;
        for (int i = 0; i < P; ++i) {
            const int r_i = rn;
            if (i + 1 < P) rn = prow[i + 1];  // read ahead, off the cost dependency
            int key = x < 8 ? (cost << 3) | x : 0x7FFFFFFF;  // the least cost, ties to the lower group
            key = min(key, dpp_i<0xB1, 0xF, 0xF>(key, key));   // quad_perm [1,0,3,2]
            key = min(key, dpp_i<0x4E, 0xF, 0xF>(key, key));   // quad_perm [2,3,0,1]
            key = min(key, dpp_i<0x141, 0xF, 0xF>(key, key));  // row_half_mirror: the other quad of the 8
            if (x == (key & 7)) {
                pgrp[i] = x;
                pidx[i] = np++;
                cost += PF_COST0 + r_i;
            }
        }
        int s = x < 8 ? nf + np : 0;  // exclusive scan over the 8 groups
        for (int d = 1; d < 8; d <<= 1) {
            const int v = __shfl_up(s, d);
            if (x >= d) s += v;
        }
        if (x < 8) {
            gfull[x] = nf;
            gstart[x] = s - nf - np;
            n_entries[1 + x] = s - nf - np;
            if (x == 7) {
                n_entries[9] = s;
                n_entries[0] = s;
            }
        }
    }
    __syncthreads();
    for (int j = 0; j < nt; ++j) {
        const int f = pre - nt + j;  // full entry f: run x with F x / 8 <= f < F (x + 1) / 8
        int x = 0;
#pragma unroll
        for (int y = 1; y < 8; ++y) x += F * y / 8 <= f ? 1 : 0;
        table[gstart[x] + f - F * x / 8] = PfEntry{slot, o + PF_BM * j, PF_BM, e};
    }
    if (q >= 0) {
        const int x = pgrp[q];
        table[gstart[x] + gfull[x] + pidx[q]] = PfEntry{slot, o + PF_BM * nt, r, e};
    }
}

// x [rows, K] bf16 -> fp6 records (rows of MP records; blocks at or past K as zero codes with a
// unit scale). One thread per (row, 32-value block).
__device__ __forceinline__ void pf_quant(const uint16_t* __restrict__ x, int64_t rows, int K, int MP,
                                         uint8_t* __restrict__ out, int64_t g) {
    const int nb = 4 * MP;
    if (g >= rows * nb) return;
    const int64_t r = g / nb;
    const int b = (int)(g - r * nb);
    uint32_t hi[6], lo[6], sc = 127u;
    if (32 * b < K) {
        // a bounded buffer resource over x: no alignment assumption beyond the element's
        const __amdgpu_buffer_rsrc_t xr = __builtin_amdgcn_make_buffer_rsrc(
            const_cast<uint16_t*>(x), (short)0, (int)(rows * K * 2), 0x00020000);
        float v[32];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const u32x4 w = __builtin_bit_cast(
                u32x4, __builtin_amdgcn_raw_buffer_load_b128(xr, (int)((r * K + 32 * b + 8 * i) * 2), 0, 0));
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                v[8 * i + 2 * j] = bf16_bits_to_f32(w[j] & 0xFFFFu);
                v[8 * i + 2 * j + 1] = bf16_bits_to_f32(w[j] >> 16);
            }
        }
        sc = fp6_terms(v, hi, lo);
    } else {
#pragma unroll
        for (int d = 0; d < 6; ++d) hi[d] = lo[d] = 0u;
    }
    uint8_t* rec = out + r * (int64_t)MP * PF_QREC + (int64_t)(b >> 2) * PF_QREC;
    const int bq = b & 3;
    *reinterpret_cast<uint4*>(rec + 48 * bq) = make_uint4(hi[0], hi[1], hi[2], hi[3]);
    *reinterpret_cast<uint4*>(rec + 48 * bq + 16) = make_uint4(hi[4], hi[5], lo[0], lo[1]);
    *reinterpret_cast<uint4*>(rec + 48 * bq + 32) = make_uint4(lo[2], lo[3], lo[4], lo[5]);
    rec[PF_QSCALE + bq] = (uint8_t)sc;
}

// All that the GEMMs need before them, in one launch: workgroup 0 groups the assignments
// (perm), workgroup 1 counts them by itself and forms the tile table, the rest form x's fp6
// records. Each was a launch of its own, small ones mostly launch: 32 experts, hidden 2880, top
// 4, us: 24 tokens 4.2 + 5.5 + 4.2 -> 6.5 (and two launch gaps), 2047 tokens 8.1 + 9.0 + 7.7 -> 13.
struct PfPrep {
    const int32_t* idx;
    int64_t n;
    int E, nw;                // nw: waves that group
    int32_t *counts, *offsets, *perm;
    const int32_t* expert_slot;
    int64_t n_slots;
    int* n_entries;
    PfEntry* table;
    int* ctr;
    const uint16_t* x;
    int64_t T;
    int K, MP;
    uint8_t* xq;
};
__global__ void __launch_bounds__(1024) pf_prepare_kernel(PfPrep p) {
    extern __shared__ __align__(16) unsigned char gsm[];
    if (blockIdx.x == 0)
        group_assignments<false>(p.idx, p.n, p.E, p.counts, p.offsets, p.perm, GroupTiles{}, p.nw, gsm);
    else if (blockIdx.x == 1)
        pf_table(p.idx, p.n, p.expert_slot, p.E, p.n_slots, p.n_entries, p.table, p.ctr, reinterpret_cast<int*>(gsm));
    else
        pf_quant(p.x, p.T, p.K, p.MP, p.xq, (int64_t)(blockIdx.x - 2) * 1024 + threadIdx.x);
}

// y[t] = sum_j w[t, j] yk[t k + j] over the live assignments, j in order; 8 columns per thread.
__global__ void __launch_bounds__(256) pf_combine_kernel(const uint16_t* __restrict__ yk,
                                                         const int32_t* __restrict__ idx,
                                                         const float* __restrict__ w,
                                                         const int32_t* __restrict__ expert_slot, int64_t E,
                                                         int64_t n_slots, int64_t T, int k, int H, void* y,
                                                         int y_dtype) {
    const int64_t g = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int cpr = H / 8;
    if (g >= T * cpr) return;
    const int64_t t = g / cpr;
    const int c = (int)(g % cpr);
    float acc[8] = {0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
    // Four assignments at a time: their ids, weights and output rows are loaded together
    // (a dropped assignment's row is read but not used), then the slots, then the sums in
    // j order.
    constexpr int JB = 4;
    for (int j0 = 0; j0 < k; j0 += JB) {
        int e[JB];
        float wj[JB];
        u32x4 v[JB];
#pragma unroll
        for (int jj = 0; jj < JB; ++jj) {
            const int j = j0 + jj;
            e[jj] = j < k ? idx[t * k + j] : -1;
            wj[jj] = j < k ? w[t * k + j] : 0.0f;
            v[jj] = j < k ? *reinterpret_cast<const u32x4*>(yk + (t * k + j) * H + 8 * c) : u32x4{0u, 0u, 0u, 0u};
        }
        bool live[JB];
#pragma unroll
        for (int jj = 0; jj < JB; ++jj) {
            live[jj] = e[jj] >= 0 && e[jj] < E;
            if (live[jj]) {
                const int s = expert_slot[e[jj]];
                live[jj] = s >= 0 && s < n_slots;
            }
        }
#pragma unroll
        for (int jj = 0; jj < JB; ++jj) {
            if (!live[jj]) continue;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                acc[2 * i] += wj[jj] * bf16_bits_to_f32(v[jj][i] & 0xFFFFu);
                acc[2 * i + 1] += wj[jj] * bf16_bits_to_f32(v[jj][i] >> 16);
            }
        }
    }
    if (y_dtype == TSA_BF16) {  // one 16-byte store (H % 8 == 0 keeps it aligned)
        *reinterpret_cast<uint4*>(static_cast<uint16_t*>(y) + t * H + 8 * c) =
            make_uint4(pack_bf16x2(acc[0], acc[1]), pack_bf16x2(acc[2], acc[3]), pack_bf16x2(acc[4], acc[5]),
                       pack_bf16x2(acc[6], acc[7]));
        return;
    }
#pragma unroll
    for (int i = 0; i < 8; ++i) store_out(y, y_dtype, t * H + 8 * c + i, acc[i]);
}

}  // namespace

// ---------------------------------------------------------------- host side

// Whether the tiled MXFP4 grouped-GEMM path covers this call (else the caller uses the
// fused decode kernel token chunk by token chunk).
static int64_t q6_row_bytes(int64_t K) { return (K + 127) / 128 * PF_QREC; }

bool pf_mxt_supported(const tsa_expert_layout& L, int x_dtype, int64_t T, int k) {
    const int64_t n = T * k, lim = (int64_t)1 << 32;
    const bool bf16_ok = T * L.hidden * 2 < lim && n * L.inter * 2 < lim;
    const bool q6_ok = L.prefill_mfma != TSA_PREFILL_FP6 || (T * q6_row_bytes(L.hidden) < lim &&
                                                            n * q6_row_bytes(L.inter) < lim);
    return L.format == TSA_EXPERT_MXFP4 && L.mx_tiled && x_dtype == TSA_BF16 && L.hidden % 16 == 0 &&
           L.inter % 16 == 0 && bf16_ok && q6_ok;
}

static int64_t al256(int64_t v) { return (v + 255) / 256 * 256; }

struct PfWs {
    int64_t counts, offsets, perm, nent, ctr, table, h, xq, yk, total;
};

static PfWs pf_ws_layout(const tsa_expert_layout& L, int64_t T, int k, int64_t E) {
    const int64_t n = T * k;
    PfWs w;
    int64_t o = 0;
    w.counts = o; o += al256(4 * E);
    w.offsets = o; o += al256(4 * (E + 1));
    w.perm = o; o += al256(4 * n);
    w.nent = o; o += 256;
    w.ctr = o; o += al256(4 * PF_CTR_INTS);
    w.table = o; o += al256((int64_t)sizeof(PfEntry) * (n / PF_BM + E + 1));
    const bool q6 = L.prefill_mfma == TSA_PREFILL_FP6;
    w.h = o; o += al256(q6 ? n * q6_row_bytes(L.inter) : 2 * n * L.inter);  // h: fp6 records or bf16
    w.xq = o; o += q6 ? al256(T * q6_row_bytes(L.hidden)) : 0;              // x as fp6 records
    w.yk = o; o += al256(2 * n * L.hidden);
    w.total = o;
    return w;
}

int64_t pf_mxt_workspace_bytes(const tsa_expert_layout& L, int64_t T, int k, int64_t E) {
    return pf_ws_layout(L, T, k, E).total;
}

// y[t] = sum_j w[t, j] yk[t k + j] over the live assignments, j in order (H % 8 == 0).
int pf_combine(const uint16_t* yk, const int32_t* idx, const float* w, const int32_t* expert_slot, int64_t E,
               int64_t n_slots, int64_t T, int k, int H, void* y, int y_dtype, hipStream_t stream) {
    const int64_t threads = T * (H / 8);
    hipLaunchKernelGGL(pf_combine_kernel, dim3((unsigned)((threads + 255) / 256)), dim3(256), 0, stream, yk, idx, w,
                       expert_slot, E, n_slots, T, k, H, y, y_dtype);
    TSA_LAUNCH_CHECK();
    return TSA_OK;
}

int pf_mxt_prefill(const tsa_expert_layout& L, const uint8_t* pool, int64_t n_slots, const int32_t* expert_slot,
                   int64_t E, const int32_t* idx, const float* weights, int64_t T, int k, const uint16_t* x, void* y,
                   int y_dtype, uint8_t* ws, hipStream_t stream) {
    const PfWs w = pf_ws_layout(L, T, k, E);
    int32_t* counts = reinterpret_cast<int32_t*>(ws + w.counts);
    int32_t* offsets = reinterpret_cast<int32_t*>(ws + w.offsets);
    int32_t* perm = reinterpret_cast<int32_t*>(ws + w.perm);
    int* nent = reinterpret_cast<int*>(ws + w.nent);
    int* ctr = reinterpret_cast<int*>(ws + w.ctr);
    PfEntry* table = reinterpret_cast<PfEntry*>(ws + w.table);
    uint16_t* h = reinterpret_cast<uint16_t*>(ws + w.h);
    uint16_t* yk = reinterpret_cast<uint16_t*>(ws + w.yk);
    const int H = (int)L.hidden, I = (int)L.inter;

    const bool q6 = L.prefill_mfma == TSA_PREFILL_FP6;
    uint8_t* xq = ws + w.xq;
    const int MPH = (H + 127) / 128;
    // 16 waves group where their LDS leaves the records' workgroups two per CU, else 8
    const int nw = group_lds_bytes((int)E, 16) <= 64 * 1024 ? 16 : 8, glds = group_lds_bytes((int)E, nw);
    const hipError_t le = ensure_dynamic_lds(reinterpret_cast<const void*>(pf_prepare_kernel), glds);
    TSA_REQUIRE(le == hipSuccess, TSA_ERR_HIP, "hipFuncSetAttribute(LDS %d): %s", glds, hipGetErrorString(le));
    const PfPrep pp{idx, T * k, (int)E, nw, counts, offsets, perm, expert_slot, n_slots, nent, table, ctr, x, T, H, MPH, xq};
    const int64_t recs = q6 ? T * 4 * MPH : 0;
    hipLaunchKernelGGL(pf_prepare_kernel, dim3((unsigned)(2 + (recs + 1023) / 1024)), dim3(1024), glds, stream, pp);
    TSA_LAUNCH_CHECK();

    const void* f_gu = q6 ? reinterpret_cast<const void*>(pf6_gemm_kernel<true>) : reinterpret_cast<const void*>(pf_gemm_kernel<true>);
    const void* f_dn = q6 ? reinterpret_cast<const void*>(pf6_gemm_kernel<false>) : reinterpret_cast<const void*>(pf_gemm_kernel<false>);
    const int lds = q6 ? P6_LDS : PF_LDS;
    for (const void* f : {f_gu, f_dn}) {
        const hipError_t e = ensure_dynamic_lds(f, lds);
        TSA_REQUIRE(e == hipSuccess, TSA_ERR_HIP, "hipFuncSetAttribute(LDS %d): %s", lds, hipGetErrorString(e));
    }
    const int grid = (num_cus() / 8) * 8;
    PfGemm g{};
    g.L = L;
    g.pool = pool;
    g.n_entries = nent;
    g.table = table;
    g.perm = perm;
    g.ctr = ctr;
    g.k = k;
    void* args[] = {&g};
    // gate_up: [2I, H] -> h
    g.src = q6 ? static_cast<const void*>(xq) : static_cast<const void*>(x);
    g.src_rows = T;
    g.src_stride = q6 ? q6_row_bytes(H) : 2 * (int64_t)H;
    g.out = h;
    g.qout = ws + w.h;
    g.out_stride = q6_row_bytes(I);
    g.N = 2 * I;
    g.K = H;
    g.NT = (2 * I + PF_BN - 1) / PF_BN;
    g.MP = (H + 127) / 128;
    g.w_off = L.gate_off;
    g.s_off = L.gate_scales_off;
    g.b_off = L.gate_bias_off;
    g.tile_bytes = 16 * (int64_t)H / 2;
    g.stile_bytes = mx_tile_scale_bytes(H);
    TSA_HIP_CHECK(hipLaunchKernel(f_gu, dim3(grid), dim3(PF_THREADS), args, lds, stream));
    // down: [H, I] -> yk
    g.src = ws + w.h;
    g.src_rows = T * k;
    g.src_stride = q6 ? q6_row_bytes(I) : 2 * (int64_t)I;
    g.ctr = ctr + 8 * PF_CTR_STRIDE;
    g.out = yk;
    g.N = H;
    g.K = I;
    g.NT = (H + PF_BN - 1) / PF_BN;
    g.MP = (I + 127) / 128;
    g.w_off = L.down_off;
    g.s_off = L.down_scales_off;
    g.b_off = L.down_bias_off;
    g.tile_bytes = 16 * (int64_t)I / 2;
    g.stile_bytes = mx_tile_scale_bytes(I);
    TSA_HIP_CHECK(hipLaunchKernel(f_dn, dim3(grid), dim3(PF_THREADS), args, lds, stream));

    return pf_combine(yk, idx, weights, expert_slot, E, n_slots, T, k, H, y, y_dtype, stream);
}

}  // namespace tsa
