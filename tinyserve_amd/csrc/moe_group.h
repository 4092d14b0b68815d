// The expert-major grouping of (token, j) assignments, for one workgroup of a kernel.
#pragma once

#include "fused_common.h"

namespace tsa {
namespace {

constexpr int GROUP_THREADS = 512;
constexpr int GROUP_WAVES = GROUP_THREADS / 64;
constexpr int MAX_GROUP_E = 1024;
constexpr int GROUP_AHEAD = 8;  // id batches loaded ahead per wave

// Optional tile table (the grouped GGUF GEMMs' work list): per resident expert in id order,
// entries of up to `rows` sorted rows {slot, first sorted row, rows, 0}; n_entries[0] = their
// count.
struct GroupTiles {
    const int32_t* expert_slot;
    int64_t n_slots;
    int rows;
    int* n_entries;
    int4* table;
};

// LDS of the grouping by nw waves for E experts: per (wave, expert) counters, the experts'
// offsets, and per (wave, expert) 64-bit lane masks (8-byte aligned).
__host__ __device__ constexpr int group_lds_bytes(int E, int nw = GROUP_WAVES) {
    return ((nw + 1) * E * 4 + 7) / 8 * 8 + nw * E * 8;
}

// Stable counting sort of assignment ids by expert, by the first nw waves of one workgroup
// (every wave of it calls this and takes the barriers). Wave w owns one contiguous chunk of
// the assignments (a multiple of 64 long) and walks it in batches of 64. Pass 1 counts per (wave, expert) with LDS atomic adds (a wave owns its row of
// counters; the order of the adds does not matter). An exclusive scan over the waves, per
// expert, then gives each wave its first rank inside the expert, and a scan over the
// experts the offsets. Pass 2 walks the same batches in the same order and places each
// assignment at offset + the wave's running rank + its rank among the batch's lanes of the
// same expert: every lane ORs its bit into its wave's mask of the expert and reads the mask
// back (LDS runs one wave's instructions in order), the lowest lane of each group then
// clears the mask and advances the running rank. Every expert's run keeps assignment order
// (token-major), as the reference's grouping does. TILES: it also writes the tile table
// between the passes (512 threads, each two experts; the slots are loaded first).
template <bool TILES>
__device__ __forceinline__ void group_assignments(const int32_t* __restrict__ idx, int64_t n, int E,
                                                  int32_t* __restrict__ counts, int32_t* __restrict__ offsets,
                                                  int32_t* __restrict__ perm, const GroupTiles& tiles, int nw,
                                                  unsigned char* gsm) {
    int* wcnt = reinterpret_cast<int*>(gsm);  // [wave][expert]
    int* eoff = wcnt + nw * E;
    unsigned long long* wmask = reinterpret_cast<unsigned long long*>(gsm + ((nw + 1) * E * 4 + 7) / 8 * 8);
    __shared__ int n_all;
    const int nthreads = (int)blockDim.x, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const unsigned long long below = (1ull << lane) - 1ull;
    static_assert(2 * GROUP_THREADS >= MAX_GROUP_E, "two experts per thread for the tile table");
    int es[2] = {-1, -1};  // the tile table's experts 2 tid, 2 tid + 1: their slots, loaded early
    if constexpr (TILES) {
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const int e = 2 * tid + i;
            if (e < E) {
                es[i] = tiles.expert_slot[e];
                if (es[i] >= tiles.n_slots) es[i] = -1;
            }
        }
    }
    for (int i = tid; i < nw * E; i += nthreads) {
        wcnt[i] = 0;
        wmask[i] = 0ull;
    }
    __syncthreads();
    int* cnt = wcnt + wave * E;
    unsigned long long* msk = wmask + wave * E;
    const int64_t chunk = ((n + nw - 1) / nw + 63) / 64 * 64;
    const int64_t a0 = wave * chunk, a1 = wave >= nw ? 0 : a0 + chunk < n ? a0 + chunk : n;
    // Batches of 64 assignments in order; the ids of GROUP_AHEAD batches are loaded together
    // so the wave waits for one memory round trip per GROUP_AHEAD batches, not per batch.
    for (int64_t b0 = a0; b0 < a1; b0 += 64 * GROUP_AHEAD) {
        int ev[GROUP_AHEAD];
#pragma unroll
        for (int j = 0; j < GROUP_AHEAD; ++j) {
            const int64_t a = b0 + 64 * j + lane;
            ev[j] = a < a1 ? idx[a] : -1;
        }
#pragma unroll
        for (int j = 0; j < GROUP_AHEAD; ++j)
            if (ev[j] >= 0 && ev[j] < E) atomicAdd(&cnt[ev[j]], 1);
    }
    __syncthreads();
    for (int e = tid; e < E; e += nthreads) {
        int run = 0;
        for (int w = 0; w < nw; ++w) {
            const int c = wcnt[w * E + e];
            wcnt[w * E + e] = run;
            run += c;
        }
        eoff[e] = run;
    }
    __syncthreads();
    if (wave == 0) {  // offsets: exclusive scan of the totals, 16 experts per lane at most
        const int per = (E + 63) / 64;
        int loc = 0;
        for (int j = 0; j < per; ++j)
            if (lane * per + j < E) loc += eoff[lane * per + j];
        int inc = loc;
        for (int d = 1; d < 64; d <<= 1) {
            const int v = __shfl_up(inc, d, 64);
            if (lane >= d) inc += v;
        }
        int run = inc - loc;
        for (int j = 0; j < per; ++j) {
            const int e = lane * per + j;
            if (e < E) {
                const int c = eoff[e];
                counts[e] = c;
                offsets[e] = run;
                eoff[e] = run;
                run += c;
            }
        }
        if (lane == 63) {
            offsets[E] = inc;
            n_all = inc;
        }
    }
    __syncthreads();
    if constexpr (TILES) {  // eoff holds the offsets; a count is the next offset minus its own
        int c[2], nt[2];
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const int e = 2 * tid + i;
            c[i] = e < E && es[i] >= 0 ? (e + 1 < E ? eoff[e + 1] : n_all) - eoff[e] : 0;
            nt[i] = (c[i] + tiles.rows - 1) / tiles.rows;
        }
        __shared__ int wsum[16];
        int total;
        int first = block_incl_sum(nt[0] + nt[1], wsum, total) - nt[0] - nt[1];
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const int e = 2 * tid + i;
            for (int j = 0; j < nt[i]; ++j) {
                const int r = c[i] - tiles.rows * j;
                tiles.table[first++] = make_int4(es[i], eoff[e] + tiles.rows * j, r < tiles.rows ? r : tiles.rows, 0);
            }
        }
        if (tid == 0) tiles.n_entries[0] = total;
    }
    for (int64_t b0 = a0; b0 < a1; b0 += 64 * GROUP_AHEAD) {
        int ev[GROUP_AHEAD];
#pragma unroll
        for (int j = 0; j < GROUP_AHEAD; ++j) {
            const int64_t a = b0 + 64 * j + lane;
            ev[j] = a < a1 ? idx[a] : -1;
        }
#pragma unroll
        for (int j = 0; j < GROUP_AHEAD; ++j) {
            const int e = ev[j];
            if (e >= 0 && e < E) {
                atomicOr(&msk[e], 1ull << lane);
                const unsigned long long m = msk[e];  // after every lane's OR: this batch's lanes of e
                const int at = eoff[e] + cnt[e] + __popcll(m & below);
                perm[at] = (int32_t)(b0 + 64 * j + lane);
                if (!(m & below)) {  // after every lane of the group read the mask and the count
                    msk[e] = 0ull;
                    cnt[e] += __popcll(m);
                }
            }
        }
    }
}

}  // namespace
}  // namespace tsa
