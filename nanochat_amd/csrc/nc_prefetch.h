// Weights on their way while the memory is idle.  A forward pass reads each weight once, and the weights of a model of more than 256 MB have left the
// last-level cache by the next pass: the linears of a prompt, whose tiles wait for one K-step of their operands after the other, then run at the
// latency of HBM (us, weights in HBM / in that cache: 1792 x 1664 x 6656 33.7 / 24.3, 1792 x 4992 x 1664 27.2 / 22.7, 1792 x 6656 x 1664 29.5 / 25.2).
// (Smaller models too have their weights pushed out by what runs between two passes: us without / with, other models' passes in between, and in brackets with the card to
// itself: GPT of depth 12 (110 MB) 500 tokens 822 / 790 (794 / 783), depth 10, 200 tokens 573 / 566 (562 / 573), dense Palilix of width 1024 (172 MB) 500 tokens 380 / 369 (352 /
// 354.5), Zodirax of width 1024, 200 tokens 484 / 478 (458 / 465).  So no rule looks at the size of the model.)
// A launch that computes while the memory has nothing to do (attention of a prompt) carries some workgroups more that read the weights of the
// linears behind it, 32 KB at a time, one run of addresses after the other, and throw away what they read.
#pragma once
#include "nc_common.h"

#define NC_AHEAD_RANGES 4
#define NC_AHEAD_WGS 128                      // workgroups of 256 threads: 33 MB in some 8 us
struct NcAhead {
    const void* p[NC_AHEAD_RANGES];
    uint32_t bytes[NC_AHEAD_RANGES];
    int n;
    void add(const void* ptr, size_t size) {
        if (n == NC_AHEAD_RANGES || !ptr || ((uintptr_t)ptr & 15) || size >= 1u << 31) return;
        p[n] = ptr, bytes[n] = (uint32_t)size, n++;
    }
};
// Launches that read nothing ahead take a form of their kernel without the argument and the check, which stood in front of everything else (us with them /
// without: window attention of 40 tokens 7.4 / 6.7, selective scan 22.1 / 21.8).
struct NcNoAhead {};
// Launches whose grid counts rows in z carry the workgroups that read ahead in the slices behind them.  launch(grid, NcAhead or NcNoAhead); MAY: whether the first of the two occurs
template <bool MAY = true, typename Launch>
static inline void nc_launch_ahead(dim3 grid, const NcAhead* a, Launch&& launch) {
    const unsigned per = grid.x * grid.y, slices = (NC_AHEAD_WGS + per - 1) / per;
    if constexpr (MAY) {
        if (a && a->n > 0 && grid.z + slices <= 65535) {
            grid.z += slices;
            launch(grid, *a);
            return;
        }
    }
    launch(grid, NcNoAhead{});
}

// What a mixer's launch is told beside its own work: what to read ahead, or (the last mixers of a prompt) the rows whose results are wanted, flat indices row * T + token.
struct NcBehind : NcAhead {
    const int32_t* chosen;
    int n_chosen;                 // 0: all rows
};
// Launches of tiles of tokens take a form that leaves out the tiles without a chosen one; it reads nothing ahead.
struct NcChosen {
    const int32_t* rows;
    int n;
};
template <typename Launch>
static inline void nc_launch_behind(dim3 grid, const NcBehind* a, Launch&& launch) {
    if (a && a->n_chosen > 0) launch(grid, NcChosen{a->chosen, a->n_chosen});
    else nc_launch_ahead(grid, a, launch);
}

// for the `wg`th of `wgs` workgroups of THREADS threads; a load past the end of a range returns zeros.  (Not with the non-temporal hint: such loads leave
// nothing in the last-level cache.)
template <int THREADS>
__device__ __forceinline__ void read_ahead(const NcAhead& a, int wg, int wgs) {
    constexpr uint32_t CHUNK = 32768, UNROLL = CHUNK / (16 * THREADS);
#pragma unroll
    for (int r = 0; r < NC_AHEAD_RANGES; r++) {
        if (r >= a.n) return;
        const uint32_t n = a.bytes[r];
        const __amdgpu_buffer_rsrc_t desc = __builtin_amdgcn_make_buffer_rsrc((void*)a.p[r], 0, n, 0x00020000);
        for (uint32_t c = (uint32_t)wg * CHUNK; c < n; c += (uint32_t)wgs * CHUNK) {
            v4i v[UNROLL];
#pragma unroll
            for (uint32_t i = 0; i < UNROLL; i++) v[i] = __builtin_amdgcn_raw_buffer_load_b128(desc, c + (i * THREADS + threadIdx.x) * 16, 0, 0);
            v4i x = v[0];
#pragma unroll
            for (uint32_t i = 1; i < UNROLL; i++) x ^= v[i];
            asm volatile("" ::"v"(x));            // (the loads are not dead code)
        }
    }
}
// whether this workgroup is one of those (it has read its share then and has nothing else to do)
template <int THREADS>
__device__ __forceinline__ bool reads_ahead(const NcAhead& a, int rows) {
    if ((int)blockIdx.z < rows) return false;
    const int wg = blockIdx.x + gridDim.x * (blockIdx.y + gridDim.y * ((int)blockIdx.z - rows));
    if (wg < NC_AHEAD_WGS) read_ahead<THREADS>(a, wg, NC_AHEAD_WGS);
    return true;
}
template <int THREADS>
__device__ __forceinline__ bool reads_ahead(NcNoAhead, int) { return false; }
template <int THREADS>
__device__ __forceinline__ bool reads_ahead(const NcChosen&, int) { return false; }
// whether none of the rows first .. end - 1 is chosen; the same in every wave
template <typename A>
__device__ __forceinline__ bool none_chosen(const A&, int64_t, int64_t) { return false; }
__device__ __forceinline__ bool none_chosen(const NcChosen& c, int64_t first, int64_t end) {
    bool hit = false;
    for (int i = threadIdx.x & 63; i < c.n; i += 64) hit |= c.rows[i] >= first && c.rows[i] < end;
    return __builtin_amdgcn_ballot_w64(hit) == 0;
}
