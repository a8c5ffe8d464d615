// The layers of a decode step of few rows in one launch: 1 .. NC_STEP_ROWS rows of one token each, from the embedded rows to the normalised rows that
// the lm_head reads (nanochat/gpt.py:495-508).
//
// What bounds such a step is not bytes: a layer is five products and an attention that each need all of the one before, and as launches of their own they cost 4 to 7 us
// each, of which two are the boundary, one to two the first trip to memory, and the rest mostly the weights' trip behind it.  Here 128 or 256 workgroups stay on the chip
// and hand each other the rows through memory:
//
//   qkv     every workgroup keeps all residual rows and repeats the row pass for itself, a wave to a row: x += mlp, lambda mix, norm, amax, e4m3 in LDS; then
//           16-column tiles of the product                                                                                        -> q|k|v, bf16
//   heads   a workgroup per (row, kv head), several where there are few of them: rotary, QK-norm, gate, append, attention         -> y
//   proj    all rows of y, amax, e4m3; tiles                                                                                      -> o
//   fc      the row pass again (x += o, norm), relu^2 in the epilogue                                                             -> h
//   mlp     all rows of h, amax, e4m3; tiles                                                                                      -> o
//
// The hand-off is the data itself: each layer has memory of its own for what its workgroups send (`exchange`), every word of it is written once, and whoever needs it
// loads until no word has the value that the embedding launch left there (all ones, a NaN that is never sent).  Stores and loads go to the point of coherence
// (sc1); there is no counter, no fence and no barrier between workgroups: a row is heard 0.5 to 1 us after it was sent.  (Before that: counters, the best of the barriers
// tried, one per XCD and a wave that polls all eight, 2.5 us with the stores' acknowledgement and the loads behind it; a word per workgroup 4.7 us; release and acquire
// fences, which write back and invalidate whole L2s, 19 to 35.)
//
// Eight waves make rows and four multiply, so that what a wave waits for never stands behind another kind of loads (they return in order).  The weights are asked for once
// the rows are here: a unit accepts a kilobyte of loads in some 40 clocks, and rows that were polled behind 60 to 100 KB of weights came 1 to 2 us later (depth 20, 8 rows 655 us a
// step with the weights first, 620 with the rows first; bringing them into the L2 by workgroups that do nothing else gained nothing more).
//
// Who takes part.  Nothing promises that the chip holds all workgroups at once: another stream's kernels may have their places.  So the workgroups
// register, and whoever has waited long enough for the others closes the list: those on it share the work out among themselves (`team`), the others leave when they start.
// A team of any size gives the same bits, and everything that is waited for behind the registration comes from workgroups that are running.
// Only a workspace that somebody else writes to could keep one waiting: a wait ends after seconds (NC_STEP_WAIT_POLLS; the longest of a running team, a share of a million keys
// beside an idle one, is some 50 ms).  Whoever gives up says so in the amax of the last rows, with a NaN that no later one takes away: the logits are NaN.
// How long: a team of n takes wgs / n rounds of tiles for every product, so what is missed by beginning with few grows as 1 / n, while other streams' kernels end
// in some 20 to 800 us and leave their places (list_polls).  us a step, 30 us whatever the team / so, beside prompts of 1792 tokens on another stream: depth 20, 8 rows
// 800 .. 1360 / 605 .. 650 (a quarter of the teams had 32 to 60 workgroups, now none less than 96), depth 26, 8 rows 930 .. 1670 / 930 .. 1060; beside steps of 64 rows
// 673 .. 735 / 618 .. 644 and 1006 .. 1176 / 965 .. 987; two such steps beside each other 1108 / 1084.  (Teams of so many, us a step of depth 20, 8 rows: 1 44900,
// 8 6310, 32 1955, 64 1085, 128 730, 256 575.)
//
// us a step, separate launches / this, one card: depth 4, one row of 63 keys 119 / 64; depth 10, 3 rows of 500 345 / 205; depth 16, 4 rows of 1000 563 / 344; depth 18, 5 rows of 400 670 / 462;
// depth 20, 640 keys, one row 702 / 446, 8 rows 798 / 551; depth 24 with 6 key heads, 8 rows of 1500 1017 / 686; depth 26, 2000 keys, one row 969 / 644, 8 rows 1176 / 881.
#include <atomic>
#include <stddef.h>
#include <type_traits>
#include <hip/hip_runtime.h>
#include "nc_common.h"
#include "nc_kernels.h"
#include "nc_rope.h"

#define MFMA_F8(acc, b, a) __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4((b), (a), (acc), 0, 0, 0, 0, 0, 0)

namespace {
#define INLINE __attribute__((always_inline))
constexpr int WAVES = 12, THREADS = 64 * WAVES;
constexpr int ROW_WAVES = NC_STEP_ROWS, GW = WAVES - ROW_WAVES;      // waves that make rows, and waves that multiply
constexpr int KV_WAVES = WAVES - 3;         // waves that read keys and values, at most (the others finish the row's own heads, G + 2 of them)
constexpr int MERGE_STRIDE = 132;           // floats of a wave's part of a head: maximum, sum, pad, pad, 128 sums
constexpr uint32_t OOB = 0x80000000u;
constexpr int SC1 = 16;                     // buffer loads at device scope: from the point of coherence, where the other workgroups' stores went
constexpr uint32_t UNWRITTEN = 0xffffffffu;

// words (NC_STEP_WORDS, zero before the launch), each on a line of its own
constexpr int LINE = 32;
enum { W_LIST = 0, W_TEAM = LINE };
constexpr uint32_t LIST_CLOSED = 1u << 30;
// Polls of half a microsecond or more before a list of `registered` workgroups of `wgs` is closed: some 30 us, and for every round of tiles behind the second as long as such a round takes
// (`round_polls`), at most some 8 ms (a bound for kernels that wait for each other's places).
constexpr uint32_t LIST_POLLS = 64, LIST_POLLS_MOST = 1u << 14;
__host__ __device__ inline uint32_t list_polls(uint32_t registered, uint32_t wgs, uint32_t round_polls) {
    const uint32_t n = registered < 1 ? 1 : registered, more = 2 * n >= wgs ? 0 : (wgs - 2 * n + n - 1) / n;      // rounds behind the second
    return LIST_POLLS + (more * round_polls < LIST_POLLS_MOST ? more * round_polls : LIST_POLLS_MOST);
}

// Registers that a condition may leave alone are "written" here without an instruction: the compiler would otherwise carry what an earlier layer left in them
// through the whole loop.
__device__ __forceinline__ void fresh_value(v4i& v) { asm volatile("" : "=v"(v)); }
typedef float v2f __attribute__((ext_vector_type(2)));
template <int T, int R>
struct Weights {
    v4i v[T][R][2];
    __device__ __forceinline__ Weights() {
#pragma unroll
        for (int t = 0; t < T; t++)
#pragma unroll
            for (int r = 0; r < R; r++) fresh_value(v[t][r][0]), fresh_value(v[t][r][1]);
    }
};
template <int N>
struct Pieces {                             // 16-byte pieces of rows
    v4i v[N];
    __device__ __forceinline__ Pieces() {
#pragma unroll
        for (int i = 0; i < N; i++) fresh_value(v[i]);
    }
    __device__ __forceinline__ v4i& operator[](int i) { return v[i]; }
    __device__ __forceinline__ const v4i& operator[](int i) const { return v[i]; }
};

// A workgroup's tiles of a weight [N, K]: wave kw takes K-steps kw, kw + GW, ...; a lane's 32 K-bytes of a step are pieces kb and 4 + kb of its 128.
template <int T, int R>
__device__ __forceinline__ void fetch_weights(Weights<T, R>& w, const uint8_t* B, int N, int K, int tile0, int tiles, int kw, int lane) {
    const __amdgpu_buffer_rsrc_t desc = __builtin_amdgcn_make_buffer_rsrc((void*)B, 0, N * K, 0x00020000);
    const int frow = lane & 15, kb = lane >> 4;
#pragma unroll
    for (int t = 0; t < T; t++)
#pragma unroll
        for (int r = 0; r < R; r++) {
            const int ks = kw + GW * r;
            const uint32_t vo = (t < tiles && ks < (K >> 7)) ? (uint32_t)((tile0 + t) * 16 + frow) * (uint32_t)K + (uint32_t)(ks * 128 + kb * 16) : OOB;
#pragma unroll
            for (int h = 0; h < 2; h++) w.v[t][r][h] = __builtin_amdgcn_raw_buffer_load_b128(desc, vo, h * 64, 0);
        }
}

// e4m3 rows in LDS: [K-step][8 rows][128 bytes], 16-byte pieces swizzled by the row
__device__ __forceinline__ void panel_store(uint8_t* panel, int row, int c, const v4i& w, float scale) {
    uint32_t o[2];
#pragma unroll
    for (int j = 0; j < 2; j++)
        // no clamp needed: |x| <= amax gives |x*scale| <= 448*(1+2^-23), which rounds to 448 like the clamped value
        o[j] = e4m3_pack4_hw(bf16_lo(w[2 * j]) * scale, bf16_hi(w[2 * j]) * scale, bf16_lo(w[2 * j + 1]) * scale, bf16_hi(w[2 * j + 1]) * scale);
    *(uint2*)(panel + (c >> 7) * 1024 + row * 128 + ((((c & 127) >> 4) ^ row) << 4) + (c & 8)) = make_uint2(o[0], o[1]);
}

// This wave's K-steps of the tiles; the sums of its 8 rows go to part[kw][t].
template <int T, int R>
__device__ __forceinline__ void multiply(const Weights<T, R>& w, const uint8_t* panel, int nks, int tiles, int kw, v4f* part, int lane) {
    const int frow = lane & 15, kb = lane >> 4, row = frow & 7;       // (rows 8 .. 15 repeat the first eight and are not looked at)
    v4f acc[T];
#pragma unroll
    for (int t = 0; t < T; t++) acc[t] = v4f{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int r = 0; r < R; r++) {
        const int ks = kw + GW * r;
        if (ks < nks) {
            const uint8_t* p = panel + ks * 1024 + row * 128;
            const v4i alo = *(const v4i*)(p + ((kb ^ row) << 4)), ahi = *(const v4i*)(p + (((4 + kb) ^ row) << 4));
            v8i a;
            a[0] = alo[0], a[1] = alo[1], a[2] = alo[2], a[3] = alo[3], a[4] = ahi[0], a[5] = ahi[1], a[6] = ahi[2], a[7] = ahi[3];
#pragma unroll
            for (int t = 0; t < T; t++) {
                if (t < tiles) {
                    const v4i lo = w.v[t][r][0], hi = w.v[t][r][1];
                    v8i b;
                    b[0] = lo[0], b[1] = lo[1], b[2] = lo[2], b[3] = lo[3], b[4] = hi[0], b[5] = hi[1], b[6] = hi[2], b[7] = hi[3];
                    acc[t] = MFMA_F8(acc[t], b, a);
                }
            }
        }
    }
    if (frow < 8) {
#pragma unroll
        for (int t = 0; t < T; t++)
            if (t < tiles) part[(kw * T + t) * 32 + kb * 8 + frow] = acc[t];
    }
}
// the sums of (tile j / 32, columns 4 (j % 32 / 8) .. + 3, row j % 8) over the waves
template <int T>
__device__ __forceinline__ v4f join_waves(const v4f* part, int j) {
    v4f s = part[(j >> 5) * 32 + (j & 31)];
#pragma unroll
    for (int w = 1; w < GW; w++) s += part[(w * T + (j >> 5)) * 32 + (j & 31)];
    return s;
}

// Values on their way to other workgroups: no NaN has the bits of an unwritten word.
__device__ __forceinline__ float sendable(float v) { return v == v ? v : __uint_as_float(0x7fc00000u); }
__device__ __forceinline__ void store8_sc1(void* p, uint32_t lo, uint32_t hi) {
    __hip_atomic_store((unsigned long long*)p, ((unsigned long long)hi << 32) | lo, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ v4i load16_sc1(__amdgpu_buffer_rsrc_t desc, uint32_t off) { return __builtin_amdgcn_raw_buffer_load_b128(desc, off, 0, SC1); }
__device__ __forceinline__ void send4(bf16_t* p, float a, float b, float c, float d) {
    store8_sc1(p, pack_bf16(sendable(a), sendable(b)), pack_bf16(sendable(c), sendable(d)));
}
__device__ __forceinline__ bool unwritten(const v4i& v) {
    const uint32_t a = (uint32_t)v[0] > (uint32_t)v[1] ? (uint32_t)v[0] : (uint32_t)v[1], b = (uint32_t)v[2] > (uint32_t)v[3] ? (uint32_t)v[2] : (uint32_t)v[3];
    return (a > b ? a : b) == UNWRITTEN;
}
__device__ __forceinline__ v4i pack8(const float (&v)[8]) {
    return v4i{(int)pack_bf16(v[0], v[1]), (int)pack_bf16(v[2], v[3]), (int)pack_bf16(v[4], v[5]), (int)pack_bf16(v[6], v[7])};
}
__device__ __forceinline__ __amdgpu_buffer_rsrc_t rows_desc(const void* p, int bytes) { return __builtin_amdgcn_make_buffer_rsrc((void*)p, 0, bytes, 0x00020000); }
// Running maxima of bf16 magnitudes, two to a word, as integers: they order like the values, and a NaN lies above infinity.
typedef uint16_t v2u16 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ uint32_t amax_pairs(uint32_t am, const v4i& v) {
#pragma unroll
    for (int j = 0; j < 4; j++)
        am = __builtin_bit_cast(uint32_t, __builtin_elementwise_max(__builtin_bit_cast(v2u16, am), __builtin_bit_cast(v2u16, (uint32_t)v[j] & 0x7fff7fffu)));
    return am;
}
__device__ __forceinline__ float amax_of_pairs(uint32_t am) { return amax_join(bf16_lo(am), bf16_hi(am)); }

// maximum and sum over the wave without a trip through LDS (the sum in wave_sum's order)
__device__ __forceinline__ float row16_max_bits(float v) {
    auto step = [](uint32_t a, uint32_t b) { return a > b ? a : b; };
    uint32_t m = __float_as_uint(v);
    m = step(m, __float_as_uint(dpp_f32<0x128>(__uint_as_float(m))));
    m = step(m, __float_as_uint(dpp_f32<0x124>(__uint_as_float(m))));
    m = step(m, __float_as_uint(dpp_f32<0x122>(__uint_as_float(m))));
    m = step(m, __float_as_uint(dpp_f32<0x121>(__uint_as_float(m))));
    return __uint_as_float(m);
}
__device__ __forceinline__ v2i swap16(float v) {
    const auto r = __builtin_amdgcn_permlane16_swap(__float_as_int(v), __float_as_int(v), false, false);
    return v2i{(int)r[0], (int)r[1]};
}
__device__ __forceinline__ v2i swap32(float v) {
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_int(v), __float_as_int(v), false, false);
    return v2i{(int)r[0], (int)r[1]};
}
__device__ __forceinline__ float fast_wave_amax(float v) {
    v = row16_max_bits(v);
    v2i r = swap16(v);
    v = amax_join(__int_as_float(r[0]), __int_as_float(r[1]));
    r = swap32(v);
    return amax_join(__int_as_float(r[0]), __int_as_float(r[1]));
}
__device__ __forceinline__ float fast_wave_sum(float v) {
    v = row16_sum(v);
    v2i r = swap16(v);
    v = __int_as_float(r[0]) + __int_as_float(r[1]);
    r = swap32(v);
    return __int_as_float(r[0]) + __int_as_float(r[1]);
}

// LDS: 8 rows of up to 4 E bytes, and in attention the fresh heads and the waves' parts; then the residual rows, and the waves' sums of a product
template <int G>
__host__ __device__ constexpr int panel_bytes(int E) {
    const int heads = ((G + 2) * 128 + KV_WAVES * G * MERGE_STRIDE) * 4;
    return 8 * 4 * E > heads ? 8 * 4 * E : heads;
}

// a / b of whole numbers that the whole wave has, 0 <= a < 2^24 (NC_STEP_MAX_KEYS), 0 < b: the reciprocal is at most one off
__device__ __forceinline__ int small_quotient(int a, int b) {
    int q = __builtin_amdgcn_readfirstlane((int)((float)a * __builtin_amdgcn_rcpf((float)b)));
    q = q * b > a ? q - 1 : q;
    return (q + 1) * b <= a ? q + 1 : q;
}

// A pointer to device memory out of its bits.  (From a bare integer the compiler makes flat accesses, which count on both counters: every wait for LDS would
// then wait for the loads in flight as well.)
template <typename P>
__device__ __forceinline__ P* device_pointer(uint64_t bits) { return (P*)(__attribute__((address_space(1))) P*)bits; }

// How many workgroups share the keys of a row's kv head when there are `most` of them: 128 keys or more for each of up to 12, 1024 for each of up to 24 (their parts are joined 12 at a time).
// us a step of one row, up to 12 / so, and the separate launches' 16: 60000 keys, depth 4 288 / 189, 264, depth 12 927 / 648, 937, depth 26 2514 / 2122, 2547; 120000 keys, depth 4 350 / 227, 307.
__host__ __device__ inline int step_splits(int most, int wgs, int pairs) {
    const int few = (most + NC_STEP_SPLIT_KEYS - 1) / NC_STEP_SPLIT_KEYS, many = most / NC_STEP_LONG_SPLIT_KEYS;
    const int wanted = few < NC_STEP_FEW_SPLITS ? few : many < NC_STEP_FEW_SPLITS ? NC_STEP_FEW_SPLITS : many < NC_STEP_MAX_SPLITS ? many : NC_STEP_MAX_SPLITS;
    const int room = wgs / pairs, splits = wanted < room ? wanted : room;
    return splits < 1 ? 1 : splits;
}

// a uniform value out of LDS
template <typename T>
__device__ __forceinline__ T argument(const uint32_t* at) {
    if constexpr (sizeof(T) == 8) {
        const uint64_t v = (uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)at[1]) << 32 | (uint32_t)__builtin_amdgcn_readfirstlane((int)at[0]);
        if constexpr (std::is_pointer_v<T>) return device_pointer<std::remove_pointer_t<T>>(v);
        else return __builtin_bit_cast(T, v);
    } else {
        return __builtin_bit_cast(T, __builtin_amdgcn_readfirstlane((int)*at));
    }
}

// NV: 512-column pieces of a residual row, so E <= 512 NV (and <= NC_STEP_MAX_E).  G: query heads per kv head.
// The first ROW_WAVES waves hear the other workgroups and make the rows, a wave to a row; then they sum what the last GW waves have multiplied, and send it.  In attention the first G + 2
// finish the row's own heads, and the first G of them join what the others have read.
template <int NV, int G>
__global__ __launch_bounds__(THREADS) __attribute__((amdgpu_waves_per_eu(3, 3))) void step_kernel(NcStepArgs, NcStepLayers) {
    constexpr int TMAX = NV == 1 ? 1 : 2;                          // tiles of a workgroup: c_fc has E / 4 of them (step_wgs)
    constexpr int E_MAX = NV < 4 ? 512 * NV : NC_STEP_MAX_E;
    constexpr int RA = (E_MAX / 128 + GW - 1) / GW;                // K-steps of a wave: E / 128 over GW waves
    constexpr int RF = (4 * E_MAX / 128 + GW - 1) / GW;            //            and 4 E / 128
    constexpr int HF = E_MAX / 128;                                // 512-column pieces of an activation row of 4 E columns

    extern __shared__ __align__(16) uint8_t lds[];
    uint8_t* const panel = lds;                                    // (panel_bytes)
    __shared__ uint32_t table[(sizeof(NcStepArgs) + sizeof(NcStepLayers)) / 4];
    __shared__ float scales[NC_STEP_MAX_LAYERS][8];                // per layer: inverse scales of q, k, v, proj, fc, mlp; lambdas of x and x0
    __shared__ uint64_t red[ROW_WAVES];                            // (round of the meeting, amax)
    __shared__ __align__(16) bf16_t gate_in[NC_STEP_ROWS][16];
    __shared__ float last_amax[ROW_WAVES];
    __shared__ int pos_of[NC_STEP_ROWS], splits_of[NC_STEP_MAX_LAYERS];
    __shared__ uint32_t said[2];

    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), kw = wave - ROW_WAVES;
    int tid = threadIdx.x, lane = tid & 63, idx = blockIdx.x;
    // Every phase starts with this: what it computes from them would otherwise be hoisted out of the loop over the layers, and five phases' worth of it
    // does not fit the registers.
    auto phase = [&]() INLINE { asm volatile("" : "+v"(tid), "+v"(lane)); };
    {
        // The arguments and what the layers' pointers of single values point at go to LDS, once: a phase that asked memory for its own, in the argument segment (host
        // memory) and behind it, started 1.2 us later.
        const uint32_t* src = device_pointer<const uint32_t>((uint64_t)__builtin_amdgcn_kernarg_segment_ptr());
        const int words = (int)(sizeof(NcStepArgs) / 4) + (int)(sizeof(NcStepLayer) / 4) * ((const NcStepArgs*)(const void*)src)->L;
        for (int i = tid; i < words; i += THREADS) table[i] = src[i];
        if (tid < ROW_WAVES) red[tid] = 0;
    }
    __syncthreads();
#define ARG(name) (argument<decltype(NcStepArgs::name)>(table + offsetof(NcStepArgs, name) / 4))
#define LAYER(name, layer) (argument<decltype(NcStepLayer::name)>(table + (sizeof(NcStepArgs) + offsetof(NcStepLayer, name)) / 4 + (layer) * (int)(sizeof(NcStepLayer) / 4)))
    const int layers = ARG(L), wgs = ARG(wgs);
    int team = wgs;
    bf16_t* const x_rows = (bf16_t*)(lds + panel_bytes<G>(ARG(E)));
    v4f* const part = (v4f*)(x_rows + NC_STEP_ROWS * ARG(E));
    if (tid < ARG(B)) pos_of[tid] = ARG(cache_seqlens)[tid];
    for (int i = tid; i < layers * 8; i += THREADS) {
        const int layer = i >> 3, what = i & 7;
        const uint32_t* t = table + sizeof(NcStepArgs) / 4 + layer * (int)(sizeof(NcStepLayer) / 4);
        const size_t from = what < 3 ? offsetof(NcStepLayer, inv_qkv) : what == 3 ? offsetof(NcStepLayer, inv_attn_proj) : what == 4 ? offsetof(NcStepLayer, inv_fc) : offsetof(NcStepLayer, inv_mlp_proj);
        const float* p = what == 6 ? ARG(resid_lambdas) + layer : what == 7 ? ARG(x0_lambdas) + layer : device_pointer<const float>((uint64_t)t[from / 4 + 1] << 32 | t[from / 4]) + (what < 3 ? what : 0);
        scales[layer][what] = what < 6 ? *p : rbf(*p);
    }
    __syncthreads();
    if (tid < layers) {
        // how many workgroups share a row's keys
        const int Tmax = ARG(Tmax), B = ARG(B), window = (int)table[sizeof(NcStepArgs) / 4 + tid * (int)(sizeof(NcStepLayer) / 4) + offsetof(NcStepLayer, window_left) / 4];
        int most = 0;
        for (int b = 0; b < B; b++) {
            const int hi = pos_of[b] > Tmax - 1 ? Tmax - 1 : pos_of[b], n = window < 0 || hi < window ? hi : window;
            most = n > most ? n : most;
        }
        splits_of[tid] = step_splits(most, wgs, B * ARG(Hkv));
    }
    // (registered once the positions have been read: the workgroup that advances them finishes after everybody on the list has)
    if (tid == 0) said[0] = __hip_atomic_fetch_add(ARG(words) + W_LIST, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __syncthreads();
    if (said[0] >= LIST_CLOSED) return;                            // the others have shared the work out already

    // ---- the others: loads until all of a wave's pieces have been written, or the wait is given up, and every later one of this workgroup with it
    auto give_up = [&]() INLINE { table[offsetof(NcStepArgs, wait_polls) / 4] = 0; };
    auto hear = [&](auto&& load_all) INLINE {
        for (uint32_t spin = 0;; spin++) {
            asm volatile("" ::: "memory");                         // (a load of the next round is another load)
            if (__builtin_amdgcn_ballot_w64(load_all()) == 0) break;
            if (spin >= ARG(wait_polls)) {
                give_up();
                break;
            }
        }
    };
    auto from_others = [&](int layer, int offset) INLINE { return ARG(exchange) + (size_t)layer * ARG(layer_bytes) + offset; };

    // ---- the residual rows, in LDS: row w belongs to wave w, a lane's columns are (64 it + lane) 8 .. + 7
    auto at = [&](int it) INLINE { return (it * 64 + lane) * 8; };
    auto row_off = [&](int row, int c, int cols) INLINE { return c < cols ? (uint32_t)(row * cols + c) * 2u : OOB; };
    auto load_x0 = [&](Pieces<NV>& to) INLINE {
        const __amdgpu_buffer_rsrc_t desc = rows_desc(ARG(x0), ARG(B) * ARG(E) * 2);
#pragma unroll
        for (int it = 0; it < NV; it++) to[it] = __builtin_amdgcn_raw_buffer_load_b128(desc, row_off(wave, at(it), ARG(E)), 0, 0);
    };
    if (wave < ARG(B)) {
        Pieces<NV> x;
        load_x0(x);
#pragma unroll
        for (int it = 0; it < NV; it++)
            if (at(it) < ARG(E)) *(v4i*)(x_rows + wave * ARG(E) + at(it)) = x[it];
    }

    // x (+= o) (l0 x + l1 z | x - l0 z); the normalised rows go to xn, their amax of this wave is returned.  gpt.py:500, 151-152, 503-508
    enum { PLAIN, MIX, BACKOUT };
    auto hear_rows = [&](const void* from, Pieces<NV>& av) INLINE {
        const __amdgpu_buffer_rsrc_t desc = rows_desc(from, ARG(B) * ARG(E) * 2);
        hear([&]() INLINE {
            bool wait = false;
#pragma unroll
            for (int it = 0; it < NV; it++) av[it] = load16_sc1(desc, row_off(wave, at(it), ARG(E)));
#pragma unroll
            for (int it = 0; it < NV; it++) wait |= unwritten(av[it]);
            return wait;
        });
    };
    auto row_pass = [&](auto kind_of, bool add, bool save, float l0, float l1, const Pieces<NV>& av, const Pieces<NV>& zv, Pieces<NV>& xn) INLINE {
        constexpr int KIND = decltype(kind_of)::value;
        const int E = ARG(E);
        Pieces<NV> x;
#pragma unroll
        for (int it = 0; it < NV; it++) x[it] = at(it) < E ? *(const v4i*)(x_rows + wave * E + at(it)) : v4i{0, 0, 0, 0};
        float ss = 0.f, v[NV][8];
#pragma unroll
        for (int it = 0; it < NV; it++) {
            v4i xw = x[it];
            const v4i zw = zv[it], aw = av[it];
            // every step in pairs of columns: `xw` is the rounded pair, v its two values
            auto round = [&](int j) INLINE {
                xw[j] = (int)pack_bf16(v[it][2 * j], v[it][2 * j + 1]);
                v[it][2 * j] = bf16_lo(xw[j]), v[it][2 * j + 1] = bf16_hi(xw[j]);
            };
#pragma unroll
            for (int j = 0; j < 4; j++) {
                v[it][2 * j] = bf16_lo(xw[j]), v[it][2 * j + 1] = bf16_hi(xw[j]);
                if (add) {
                    v[it][2 * j] += bf16_lo(aw[j]), v[it][2 * j + 1] += bf16_hi(aw[j]);
                    round(j);
                }
            }
            if (save && at(it) < E) *(v4i*)(ARG(xb) + (size_t)wave * E + at(it)) = xw;
            if (KIND != PLAIN) {
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    float z0 = bf16_lo(zw[j]), z1 = bf16_hi(zw[j]);
                    if (KIND == MIX) {
                        z0 *= l1, z1 *= l1, v[it][2 * j] *= l0, v[it][2 * j + 1] *= l0;
                        rbf2(z0, z1), rbf2(v[it][2 * j], v[it][2 * j + 1]);
                        v[it][2 * j] += z0, v[it][2 * j + 1] += z1;
                    } else {
                        z0 *= l0, z1 *= l0;
                        rbf2(z0, z1);
                        v[it][2 * j] -= z0, v[it][2 * j + 1] -= z1;
                    }
                    round(j);
                }
            }
            if (at(it) < E) *(v4i*)(x_rows + wave * E + at(it)) = xw;
            // (columns past E hold zeros: the loads gave zeros there)
#pragma unroll
            for (int j = 0; j < 8; j++) ss += v[it][j] * v[it][j];
        }
        ss = fast_wave_sum(ss);
        const float rstd = 1.0f / sqrtf(ss / (float)E + RMS_EPS);
        uint32_t am = 0u;
#pragma unroll
        for (int it = 0; it < NV; it++) {
#pragma unroll
            for (int j = 0; j < 8; j++) v[it][j] *= rstd;
            xn[it] = pack8(v[it]);
            am = amax_pairs(am, xn[it]);
        }
        return amax_of_pairs(am);
    };
    // The scale of the rows whose amax the row waves hold.  They meet in LDS by themselves: the waves that multiply are busy asking for their weights, one to two microseconds.
    uint32_t round = 0;
    auto tensor_scale = [&](float am) INLINE {
        am = fast_wave_amax(am);
        round++;
        if (lane == 0) __hip_atomic_store(&red[wave], (uint64_t)round << 32 | __float_as_uint(am), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        uint64_t v;
        do v = __hip_atomic_load(&red[lane & (ROW_WAVES - 1)], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        while (__builtin_amdgcn_ballot_w64((uint32_t)(v >> 32) != round) != 0);
        return scale_from_amax(fast_wave_amax(__uint_as_float((uint32_t)v)));
    };
    auto rows_to_panel = [&](const Pieces<NV>& xn, float scale) INLINE {
        if (wave < ARG(B)) {
#pragma unroll
            for (int it = 0; it < NV; it++)
                if (at(it) < ARG(E)) panel_store(panel, wave, at(it), xn[it], scale);
        }
    };

    // One product of the rows that rows() brings to the panel (it returns their scale): store(sum, row, column) takes four columns at a time.
    // The multiplying waves fetch their weights behind the stores of the product before: a unit accepts a kilobyte of loads in some 40 clocks, and behind a phase's weights
    // (60 to 100 KB) those stores would leave a microsecond later.
    auto product = [&](auto t_of, auto r_of, const uint8_t* weight, int N, int K, auto&& rows, auto&& store) INLINE {
        constexpr int T = decltype(t_of)::value, R = decltype(r_of)::value;
        const int each = ((N >> 4) + wgs - 1) / wgs, B = ARG(B);
        if (kw >= 0) {
            for (int vw = idx; vw < wgs; vw += team) {
                const int left = (N >> 4) - vw * each, tiles = left < each ? left : each;
                if (vw != idx && tiles <= 0) break;
                Weights<T, R> w;
                if (vw == idx) __syncthreads();                    // the rows are here
                fetch_weights(w, weight, N, K, vw * each, tiles, kw, lane);
                if (vw == idx) __syncthreads();                    // the panel is complete
                multiply(w, panel, K >> 7, tiles, kw, part, lane);
                __syncthreads();
                __syncthreads();
            }
        } else {
            const float inv_a = 1.0f / rows();
            __syncthreads();
            for (int vw = idx; vw < wgs; vw += team) {
                const int left = (N >> 4) - vw * each, tiles = left < each ? left : each;
                if (vw != idx && tiles <= 0) break;
                __syncthreads();
                if (tid < tiles * 32) {
                    const v4f s = join_waves<T>(part, tid);
                    const int row = tid & 7, col = (vw * each + (tid >> 5)) * 16 + ((tid & 31) >> 3) * 4;
                    if (row < B) store(s * inv_a, row, col);
                }
                __syncthreads();
            }
        }
    };

    for (int layer = 0; layer < layers; layer++) {
        // ---------------------------------------------------------------- q|k|v of rows made here
        {
            phase();
            const int E = ARG(E), HE = ARG(H) * 128, KE = ARG(Hkv) * 128, qkv_w = HE + 2 * KE;
            const float rl = scales[layer][6], xl = scales[layer][7], i0 = scales[layer][0], i1 = scales[layer][1], i2 = scales[layer][2];
            if (layer == 0) {
                // who is here
                int asks = wave;                                   // (its own copy: the comparison would be kept, in memory, through the loop)
                asm volatile("" : "+s"(asks));
                if (asks == 0) {
                    uint32_t v = 0, spin = 0;
                    for (;; spin++) {
                        v = __hip_atomic_load(ARG(words) + W_LIST, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                        if (v >= LIST_CLOSED || v == (uint32_t)wgs) break;
                        if (spin >= LIST_POLLS && spin >= list_polls((uint32_t)__builtin_amdgcn_readfirstlane((int)v), (uint32_t)wgs, ARG(round_polls))) {
                            if (lane == 0) v = __hip_atomic_fetch_or(ARG(words) + W_LIST, LIST_CLOSED, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                            v = (uint32_t)__builtin_amdgcn_readfirstlane((int)v);
                            if (v < LIST_CLOSED && lane == 0) __hip_atomic_store(ARG(words) + W_TEAM, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                            break;
                        }
                    }
                    if (v >= LIST_CLOSED)                          // whoever closed the list is about to say how long it was
                        for (spin = 0; spin < ARG(wait_polls); spin++)
                            if ((v = __hip_atomic_load(ARG(words) + W_TEAM, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) != 0) break;
                    if (v - 1u >= (uint32_t)wgs) v = (uint32_t)wgs, give_up();       // (not one of a team: somebody else writes here.  Every wait below still ends)
                    if (lane == 0) said[1] = v;
                }
                __syncthreads();
                team = __builtin_amdgcn_readfirstlane((int)said[1]);
                if (team != wgs) idx = __builtin_amdgcn_readfirstlane((int)said[0]);
            }
            product(std::integral_constant<int, TMAX>{}, std::integral_constant<int, RA>{}, LAYER(w_qkv, layer), qkv_w, E,
                    [&]() INLINE {
                        Pieces<NV> zv, xn, av;
                        float am = 0.f;
                        if (wave < ARG(B)) {
                            load_x0(zv);
                            if (layer > 0) hear_rows(from_others(layer - 1, ARG(off_mlp)), av);
                        }
                        __syncthreads();
                        if (wave < ARG(B)) {
                            am = row_pass(std::integral_constant<int, MIX>{}, layer > 0, layer > 0 && layer - 1 == layers / 2 && idx == 0, rl, xl, av, zv, xn);
                            if (lane < 2) *(v4i*)&gate_in[wave][lane * 8] = xn[0];
                        }
                        const float scale = tensor_scale(am);
                        rows_to_panel(xn, scale);
                        return scale;
                    },
                    [&](v4f s, int row, int col) INLINE {
                        float ib = i0, ik = i1, iv = i2;           // (copies first: a choice among the variables would keep them all in memory)
                        ib = col >= HE ? ik : ib, ib = col >= HE + KE ? iv : ib;
                        send4((bf16_t*)from_others(layer, 0) + (size_t)row * qkv_w + col, s[0] * ib, s[1] * ib, s[2] * ib, s[3] * ib);
                    });
        }

        // ---------------------------------------------------------------- heads
        const int splits = __builtin_amdgcn_readfirstlane(splits_of[layer]);
        {
            phase();
            const int B = ARG(B), H = ARG(H), Hkv = ARG(Hkv), Tmax = ARG(Tmax), window = LAYER(window_left, layer);
            const int units = B * Hkv * splits;
            bf16_t* const k_cache = ARG(k_cache) + (size_t)layer * ARG(layer_elems);
            bf16_t* const v_cache = ARG(v_cache) + (size_t)layer * ARG(layer_elems);
            // (several to a workgroup only in a team that is not complete; from the last one down, because the first workgroup of a pair waits for those behind it)
            int u = idx;
            while (u + team < units) u += team;
            for (; u >= idx && u < units; u -= team) {
                constexpr int UNROLL = G == 1 ? 8 : 6, KPI = 4, TASKS = G + 2, KVW = WAVES - TASKS;
                float* const fresh = (float*)panel;                                    // [TASKS][128]
                float* const merge = fresh + TASKS * 128;                              // [KVW][G][MERGE_STRIDE]
                const int pair = small_quotient(u, splits), split = u - pair * splits, b = small_quotient(pair, Hkv), hk = pair - b * Hkv;
                const int sub = lane & 15, ksel = lane >> 4;
                int hi = __builtin_amdgcn_readfirstlane(pos_of[b]);
                if (hi > Tmax - 1) hi = Tmax - 1;
                const int lo = window < 0 || hi < window ? 0 : hi - window, nw = splits * KVW;
                // a wave's run of keys: a batch of loads at least, waves behind the last key have nothing to do
                int chunk = (small_quotient(hi - lo + nw - 1, nw) + 3) & ~3;
                chunk = chunk < KPI * UNROLL ? KPI * UNROLL : chunk;
                const int first = lo + split * KVW * chunk, keys_here = hi - first;
                const int active = keys_here <= 0 ? 1 : keys_here >= KVW * chunk ? KVW : small_quotient(keys_here + chunk - 1, chunk);
                if (wave < TASKS) {
                    // the row's own heads: 0 .. G-1 the query heads, G the key head, G+1 the value head.  What does not come from the others is asked for first.
                    const int hh = wave < G ? hk * G + wave : wave == G ? H + hk : H + Hkv + hk;
                    NcRopeSrc r{};
                    r.ve_table = LAYER(ve_table, layer), r.ve_gate_w = LAYER(ve_gate_w, layer);
                    RopeRaw<1> raw;
                    raw.e1 = raw.e2 = raw.xg = 0u, raw.inv_b = 0.f;
                    if (wave <= G) {
                        const int rp = hi < 0 ? 0 : hi < ARG(rope_len) ? hi : ARG(rope_len) - 1;
                        raw.e1 = ARG(cos_t)[(size_t)rp * 64 + lane], raw.e2 = ARG(sin_t)[(size_t)rp * 64 + lane];
                    } else if (r.ve_table) {
                        int64_t tok = ARG(idx)[b];
                        if (tok < 0 || tok >= ARG(vocab_rows)) tok = 0;
                        const bf16_t* ve = r.ve_table + ((size_t)tok * Hkv + hk) * 128;
                        raw.e1 = ve[lane], raw.e2 = ve[lane + 64];
                        int at_lane = lane;                                            // (its own copy: the address would be kept, in memory, through the loop)
                        asm volatile("" : "+v"(at_lane));
                        raw.xg = gate_in[b][at_lane < 12 ? at_lane : 0];
                    }
                    const int qkv_w = (H + 2 * Hkv) * 128;
                    const __amdgpu_buffer_rsrc_t desc_qkv = rows_desc(from_others(layer, 0), B * qkv_w * 2);
                    const uint32_t off = (uint32_t)(b * qkv_w + hh * 128 + lane) * 2u;
                    uint32_t got[2];
                    hear([&]() INLINE {
                        got[0] = (uint16_t)__builtin_amdgcn_raw_buffer_load_b16(desc_qkv, off, 0, SC1);
                        got[1] = (uint16_t)__builtin_amdgcn_raw_buffer_load_b16(desc_qkv, off, 128, SC1);
                        return got[0] == (UNWRITTEN & 0xffffu) || got[1] == (UNWRITTEN & 0xffffu);
                    });
                    raw.t1[0] = __uint_as_float(got[0]), raw.t2[0] = __uint_as_float(got[1]);
                    float y1, y2;
                    rope_head_finish(r, b, hh, H, Hkv, lane, raw, 0.f, y1, y2);
                    fresh[wave * 128 + lane] = y1, fresh[wave * 128 + lane + 64] = y2;
                    if (wave >= G && split == 0 && hi >= 0 && hi < Tmax) {
                        bf16_t* dst = (wave == G ? k_cache : v_cache) + (((size_t)b * Tmax + hi) * Hkv + hk) * 128;
                        dst[lane] = f32_to_bf16(y1);
                        dst[lane + 64] = f32_to_bf16(y2);
                    }
                    __syncthreads();
                } else if (wave - TASKS >= active) {
                    __syncthreads();
                } else {
                    const int kv = wave - TASKS, k_begin = first + kv * chunk;
                    int k_end = k_begin + chunk;
                    if (k_end > hi) k_end = hi;
                    const size_t key_stride = (size_t)Hkv * 128;
                    const bf16_t* const kbase = k_cache + ((size_t)b * Tmax * Hkv + hk) * 128 + sub * 8;
                    const bf16_t* const vbase = v_cache + ((size_t)b * Tmax * Hkv + hk) * 128 + sub * 8;
                    // (unconditional loads of a clamped key, which then gets weight zero: as in attn_partial_kernel)
                    uint4 kr[UNROLL], vr[UNROLL];
                    const int k_last = k_end - 1 > 0 ? k_end - 1 : 0;
                    auto fetch_k = [&](int kb0) INLINE {
#pragma unroll
                        for (int i = 0; i < UNROLL; i++) {
                            const int j = kb0 + KPI * i + ksel;
                            kr[i] = nt_load16(kbase + (size_t)(j < k_end ? j : k_last) * key_stride);
                        }
                    };
                    auto fetch_v = [&](int kb0) INLINE {
#pragma unroll
                        for (int i = 0; i < UNROLL; i++) {
                            const int j = kb0 + KPI * i + ksel;
                            vr[i] = nt_load16(vbase + (size_t)(j < k_end ? j : k_last) * key_stride);
                        }
                    };
                    fetch_k(k_begin < k_end ? k_begin : 0);
                    fetch_v(k_begin < k_end ? k_begin : 0);
                    __syncthreads();
                    const float qscale = 1.4426950408889634f * 0.08838834764831845f;
                    float qf[G][8], m[G], l[G], acc[G][8];
#pragma unroll
                    for (int h = 0; h < G; h++) {
                        m[h] = -1.0e30f, l[h] = 0.f;
                        float d = 0.f;
#pragma unroll
                        for (int e = 0; e < 8; e++) {
                            qf[h][e] = fresh[h * 128 + sub * 8 + e] * qscale, acc[h][e] = 0.f;
                            d = fmaf(qf[h][e], fresh[G * 128 + sub * 8 + e], d);
                        }
                        d = row16_sum(d);
                        if (split == 0 && kv == 0 && ksel == 0) {  // the row's own key
                            m[h] = d, l[h] = 1.f;
#pragma unroll
                            for (int e = 0; e < 8; e++) acc[h][e] = fresh[(G + 1) * 128 + sub * 8 + e];
                        }
                    }
                    auto batch = [&](int kb0, auto prefetch) INLINE {
                        bool ok[UNROLL];
                        float sc[G][UNROLL];
#pragma unroll
                        for (int i = 0; i < UNROLL; i++) {
                            ok[i] = kb0 + KPI * i + ksel < k_end;
                            const uint32_t w[4] = {kr[i].x, kr[i].y, kr[i].z, kr[i].w};
                            float kf[8];
#pragma unroll
                            for (int j = 0; j < 4; j++) kf[2 * j] = bf16_lo(w[j]), kf[2 * j + 1] = bf16_hi(w[j]);
#pragma unroll
                            for (int h = 0; h < G; h++) {
                                float d = 0.f;
#pragma unroll
                                for (int e = 0; e < 8; e++) d = fmaf(qf[h][e], kf[e], d);
                                d = row16_sum(d);
                                sc[h][i] = ok[i] ? d : -1.0e30f;
                            }
                        }
                        if (decltype(prefetch)::value) fetch_k(kb0 + KPI * UNROLL);
#pragma unroll
                        for (int h = 0; h < G; h++) {
                            float mn = m[h];
#pragma unroll
                            for (int i = 0; i < UNROLL; i++) mn = fmaxf(mn, sc[h][i]);
                            const float corr = exp2f(m[h] - mn);
                            m[h] = mn;
                            l[h] *= corr;
#pragma unroll
                            for (int d = 0; d < 8; d++) acc[h][d] *= corr;
#pragma unroll
                            for (int i = 0; i < UNROLL; i++) sc[h][i] = ok[i] ? exp2f(sc[h][i] - mn) : 0.f;
                        }
#pragma unroll
                        for (int i = 0; i < UNROLL; i++) {
                            const uint32_t w[4] = {vr[i].x, vr[i].y, vr[i].z, vr[i].w};
                            float vf[8];
#pragma unroll
                            for (int j = 0; j < 4; j++) vf[2 * j] = bf16_lo(w[j]), vf[2 * j + 1] = bf16_hi(w[j]);
#pragma unroll
                            for (int h = 0; h < G; h++) {
                                l[h] += sc[h][i];
#pragma unroll
                                for (int d = 0; d < 8; d++) acc[h][d] = fmaf(sc[h][i], vf[d], acc[h][d]);
                            }
                        }
                        if (decltype(prefetch)::value) fetch_v(kb0 + KPI * UNROLL);
                    };
                    if (k_begin < k_end) {
                        int kb0 = k_begin;
                        for (; kb0 + KPI * UNROLL < k_end; kb0 += KPI * UNROLL) batch(kb0, std::true_type{});
                        batch(kb0, std::false_type{});
                    }
                    // the four 16-lane groups of the wave
#pragma unroll
                    for (int h = 0; h < G; h++) {
                        v2i r = swap16(m[h]);
                        float mm = fmaxf(__int_as_float(r[0]), __int_as_float(r[1]));
                        r = swap32(mm);
                        mm = fmaxf(__int_as_float(r[0]), __int_as_float(r[1]));
                        const float w = exp2f(m[h] - mm);
                        auto over_groups = [&](float v) INLINE {
                            v2i r = swap16(v);
                            v = __int_as_float(r[0]) + __int_as_float(r[1]);
                            r = swap32(v);
                            return __int_as_float(r[0]) + __int_as_float(r[1]);
                        };
                        const float lw = over_groups(l[h] * w);
                        float* const out = merge + (kv * G + h) * MERGE_STRIDE;
                        v4f lo4, hi4;
#pragma unroll
                        for (int d = 0; d < 4; d++) lo4[d] = over_groups(acc[h][d] * w), hi4[d] = over_groups(acc[h][4 + d] * w);
                        if (ksel == 0) {
                            if (sub == 0) out[0] = mm, out[1] = lw;
                            *(v4f*)(out + 4 + sub * 8) = lo4, *(v4f*)(out + 8 + sub * 8) = hi4;
                        }
                    }
                }
                __syncthreads();
                if (wave < G) {
                    // the waves' parts of head `wave`: half of the lanes take the even ones, half the odd ones
                    const int h = wave, d = (lane & 31) * 4, half = lane >> 5, head = hk * G + h;
                    constexpr int PARTS = (KVW + 1) / 2;
                    v2f ml[PARTS];
                    v4f part4[PARTS];
#pragma unroll
                    for (int i = 0; i < PARTS; i++) {
                        const int w = 2 * i + half;
                        const float* p = merge + ((w < active ? w : 0) * G + h) * MERGE_STRIDE;
                        ml[i] = *(const v2f*)p, part4[i] = *(const v4f*)(p + 4 + d);
                    }
                    float mm = ml[0][0];
#pragma unroll
                    for (int i = 0; i < PARTS; i++) mm = fmaxf(mm, ml[i][0]);            // (some more than once)
                    v2i r = swap32(mm);
                    mm = fmaxf(__int_as_float(r[0]), __int_as_float(r[1]));
                    float ls = 0.f;
                    v4f s = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
                    for (int i = 0; i < PARTS; i++) {
                        const float sc = 2 * i + half < active ? exp2f(ml[i][0] - mm) : 0.f;
                        ls += ml[i][1] * sc;
                        s += part4[i] * sc;
                    }
                    r = swap32(ls);
                    ls = __int_as_float(r[0]) + __int_as_float(r[1]);
#pragma unroll
                    for (int e = 0; e < 4; e++) {
                        r = swap32(s[e]);
                        s[e] = __int_as_float(r[0]) + __int_as_float(r[1]);
                    }
                    // keys in several workgroups: the first one's waits for the parts of the others ([pair][split - 1][G][MERGE_STRIDE], maximum and sum first)
                    float* const parts = (float*)(ARG(parts) + (size_t)layer * ARG(parts_bytes)) + ((size_t)pair * (splits - 1) * G + h) * MERGE_STRIDE;
                    if (split > 0) {
                        float* const mine = parts + (size_t)(split - 1) * G * MERGE_STRIDE;
                        if (half == 0) coherent_store_f4(mine + 4 + d, sendable(s[0]), sendable(s[1]), sendable(s[2]), sendable(s[3]));
                        if (lane == 0) store8_sc1(mine, __float_as_uint(sendable(mm)), __float_as_uint(sendable(ls)));
                    } else {
                        const __amdgpu_buffer_rsrc_t desc = rows_desc(parts, ((splits - 1) * G - h) * MERGE_STRIDE * 4);
                        for (int from_split = 0; from_split < splits - 1; from_split += NC_STEP_FEW_SPLITS) {
                            constexpr int OTHERS = NC_STEP_FEW_SPLITS / 2;
                            const int others = splits - 1 - from_split;
                            Pieces<OTHERS> o;
                            v2i oml[OTHERS];
#pragma unroll
                            for (int i = 0; i < OTHERS; i++) asm volatile("" : "=v"(oml[i]));
                            // (a part that does not exist reads as zeros: the lanes of an odd count ask behind the end)
                            hear([&]() INLINE {
                                bool wait = false;
#pragma unroll
                                for (int i = 0; i < OTHERS; i++)
                                    if (2 * i < others) {
                                        const uint32_t from = 2 * i + half < others ? (uint32_t)((from_split + 2 * i + half) * G * MERGE_STRIDE) * 4u : OOB;
                                        oml[i] = __builtin_amdgcn_raw_buffer_load_b64(desc, from, 0, SC1);
                                        o[i] = load16_sc1(desc, from == OOB ? OOB : from + 16 + d * 4);
                                    }
#pragma unroll
                                for (int i = 0; i < OTHERS; i++)
                                    if (2 * i < others) wait |= unwritten(o[i]) || (uint32_t)oml[i][0] == UNWRITTEN || (uint32_t)oml[i][1] == UNWRITTEN;
                                return wait;
                            });
                            float all = mm;
#pragma unroll
                            for (int i = 0; i < OTHERS; i++)
                                if (2 * i < others) all = fmaxf(all, 2 * i + half < others ? __int_as_float(oml[i][0]) : mm);
                            r = swap32(all);
                            all = fmaxf(__int_as_float(r[0]), __int_as_float(r[1]));
                            const float own = half == 0 ? exp2f(mm - all) : 0.f;
                            ls *= own, s *= own, mm = all;
#pragma unroll
                            for (int i = 0; i < OTHERS; i++)
                                if (2 * i < others) {
                                    const float sc = 2 * i + half < others ? exp2f(__int_as_float(oml[i][0]) - all) : 0.f;
                                    ls += __int_as_float(oml[i][1]) * sc;
#pragma unroll
                                    for (int e = 0; e < 4; e++) s[e] += __int_as_float(o[i][e]) * sc;
                                }
                            r = swap32(ls);
                            ls = __int_as_float(r[0]) + __int_as_float(r[1]);
#pragma unroll
                            for (int e = 0; e < 4; e++) {
                                r = swap32(s[e]);
                                s[e] = __int_as_float(r[0]) + __int_as_float(r[1]);
                            }
                        }
                        if (half == 0) send4((bf16_t*)from_others(layer, ARG(off_y)) + ((size_t)b * H + head) * 128 + d, s[0] / ls, s[1] / ls, s[2] / ls, s[3] / ls);
                    }
                }
                __syncthreads();
            }
        }

        // ---------------------------------------------------------------- attention projection of y
        {
            phase();
            const float inv = scales[layer][3];
            product(std::integral_constant<int, 1>{}, std::integral_constant<int, RA>{}, LAYER(w_attn_proj, layer), ARG(E), ARG(E),
                    [&]() INLINE {
                        // piece p = (row, 512 columns), dealt to the waves
                        const int B = ARG(B), E = ARG(E), per_row = (E + 511) >> 9, pieces = B * per_row;
                        Pieces<NV> y;
                        uint32_t am = 0u;
                        const __amdgpu_buffer_rsrc_t desc_y = rows_desc(from_others(layer, ARG(off_y)), B * E * 2);
                        hear([&]() INLINE {
                            bool wait = false;
#pragma unroll
                            for (int j = 0; j < NV; j++) {
                                const int p = wave + ROW_WAVES * j;
                                if (p < pieces) y[j] = load16_sc1(desc_y, row_off(p / per_row, at(p % per_row), E));
                            }
#pragma unroll
                            for (int j = 0; j < NV; j++) wait |= wave + ROW_WAVES * j < pieces && unwritten(y[j]);
                            return wait;
                        });
                        __syncthreads();
#pragma unroll
                        for (int j = 0; j < NV; j++)
                            if (wave + ROW_WAVES * j < pieces) am = amax_pairs(am, y[j]);
                        const float scale = tensor_scale(amax_of_pairs(am));
#pragma unroll
                        for (int j = 0; j < NV; j++) {
                            const int p = wave + ROW_WAVES * j;
                            if (p < pieces && at(p % per_row) < E) panel_store(panel, p / per_row, at(p % per_row), y[j], scale);
                        }
                        return scale;
                    },
                    [&](v4f s, int row, int col) INLINE {
                        send4((bf16_t*)from_others(layer, ARG(off_proj)) + (size_t)row * ARG(E) + col, s[0] * inv, s[1] * inv, s[2] * inv, s[3] * inv);
                    });
        }

        // ---------------------------------------------------------------- c_fc of rows made here, relu^2
        {
            phase();
            const float inv = scales[layer][4];
            product(std::integral_constant<int, TMAX>{}, std::integral_constant<int, RA>{}, LAYER(w_fc, layer), 4 * ARG(E), ARG(E),
                    [&]() INLINE {
                        Pieces<NV> xn, av;
                        float am = 0.f;
                        if (wave < ARG(B)) hear_rows(from_others(layer, ARG(off_proj)), av);
                        __syncthreads();
                        if (wave < ARG(B)) am = row_pass(std::integral_constant<int, PLAIN>{}, true, false, 0.f, 0.f, av, av, xn);
                        const float scale = tensor_scale(am);
                        rows_to_panel(xn, scale);
                        return scale;
                    },
                    [&](v4f s, int row, int col) INLINE {
                        float h[4];
#pragma unroll
                        for (int j = 0; j < 4; j++) {
                            const float t = relu_keep_nan(rbf(s[j] * inv));
                            h[j] = t * t;
                        }
                        send4((bf16_t*)from_others(layer, ARG(off_h)) + (size_t)row * 4 * ARG(E) + col, h[0], h[1], h[2], h[3]);
                    });
        }

        // ---------------------------------------------------------------- MLP projection
        {
            phase();
            const float inv = scales[layer][5];
            product(std::integral_constant<int, 1>{}, std::integral_constant<int, RF>{}, LAYER(w_mlp_proj, layer), ARG(E), 4 * ARG(E),
                    [&]() INLINE {
                        // pieces of 512 columns, 4 E of them a row, dealt to the waves four at a time (what lies past the last row reads as zeros)
                        const int per_row = ARG(E) >> 7, pieces = ARG(B) * per_row, inv_row = 65536 / per_row + 1;
                        const __amdgpu_buffer_rsrc_t desc_h = rows_desc(from_others(layer, ARG(off_h)), ARG(B) * ARG(E) * 8);
                        Pieces<HF> h;
                        uint32_t am = 0u;
                        {
                            hear([&]() INLINE {
                                bool wait = false;
#pragma unroll
                                for (int q = 0; q < HF; q += 4)
                                    if (q * ROW_WAVES < pieces) {
#pragma unroll
                                        for (int j = q; j < (q + 4 < HF ? q + 4 : HF); j++) h[j] = load16_sc1(desc_h, (uint32_t)((wave + ROW_WAVES * j) * 512 + lane * 8) * 2u);
                                    }
#pragma unroll
                                for (int q = 0; q < HF; q += 4)
                                    if (q * ROW_WAVES < pieces) {
#pragma unroll
                                        for (int j = q; j < (q + 4 < HF ? q + 4 : HF); j++) wait |= unwritten(h[j]);
                                    }
                                return wait;
                            });
                            __syncthreads();
#pragma unroll
                            for (int q = 0; q < HF; q += 4)
                                if (q * ROW_WAVES < pieces) {
#pragma unroll
                                    for (int j = q; j < (q + 4 < HF ? q + 4 : HF); j++) am = amax_pairs(am, h[j]);
                                }
                        }
                        const float scale = tensor_scale(amax_of_pairs(am));
#pragma unroll
                        for (int j = 0; j < HF; j++) {
                            const int p = wave + ROW_WAVES * j, row = (p * inv_row) >> 16;
                            if (p < pieces) panel_store(panel, row, (p - row * per_row) * 512 + lane * 8, h[j], scale);
                        }
                        return scale;
                    },
                    [&](v4f s, int row, int col) INLINE {
                        send4((bf16_t*)from_others(layer, ARG(off_mlp)) + (size_t)row * ARG(E) + col, s[0] * inv, s[1] * inv, s[2] * inv, s[3] * inv);
                    });
        }
    }
    // ---------------------------------------------------------------- the last rows: x += mlp, less the saved rows, norm
    const float GAVE_UP = __uint_as_float(0x7fc00000u);
    if (idx != 0) {
        if (tid == 0 && ARG(wait_polls) == 0) amax_publish(ARG(head_site), GAVE_UP);
        return;
    }
    phase();
    const int B = ARG(B), E = ARG(E);
    const float bl = rbf(*ARG(backout_lambda));
    float am = 0.f;
    Pieces<NV> xn;
    if (wave < B) {
        Pieces<NV> zv, av;
        hear_rows(from_others(layers - 1, ARG(off_mlp)), av);
        const __amdgpu_buffer_rsrc_t desc = rows_desc(ARG(xb), B * E * 2);
#pragma unroll
        for (int it = 0; it < NV; it++) zv[it] = __builtin_amdgcn_raw_buffer_load_b128(desc, row_off(wave, at(it), E), 0, 0);
        am = row_pass(std::integral_constant<int, BACKOUT>{}, true, false, bl, 0.f, av, zv, xn);
#pragma unroll
        for (int it = 0; it < NV; it++)
            if (at(it) < E) *(v4i*)(ARG(xn) + (size_t)wave * E + at(it)) = xn[it];
    }
    if (wave < ROW_WAVES) {
        am = fast_wave_amax(am);
        if (lane == 0) last_amax[wave] = am;
    }
    __syncthreads();
    if (tid == 0) {
        float all = last_amax[0];
#pragma unroll
        for (int w = 1; w < ROW_WAVES; w++) all = amax_join(all, last_amax[w]);
        amax_publish(ARG(head_site), ARG(wait_polls) == 0 ? GAVE_UP : all);
    }
    if (ARG(advance) && tid < B) ARG(cache_seqlens)[tid] = pos_of[tid] + ARG(advance);
}
}  // namespace

// ------------------------------------------------------------------------------------------------
// Workgroups, one to a compute unit.  Half of the units where a product has no more than two tiles for each of them then (us a step, 128 / 256: depth 4, one row 63.5 / 65.7,
// depth 8 with 2 key heads, 8 rows 154 / 165, depth 10, 3 rows 205 / 210, depth 16 with 4 key heads, 5 rows 352 / 360), all of them for wider models (depth 20, 8 rows 730 with 128 of
// 256 started / 551, depth 26, 8 rows of 2000 keys 1178 / 881), and where there are many keys: those are read as fast as there are units (128 / 256 / the separate launches, depth 10, 8 rows of 2000
// keys in every layer 305 / 289 / 388, 8000 570 / 460 / 576, depth 12, 8 rows of 8000 882 / 620 / 743, of 60000 5043 / 3020 / 3104, depth 16, 6 rows of 8000 1220 / 855 / 1066; from some 40 to 100 thousand keys
// of all heads on, which models of 2048 positions do not have: 82 thousand, depth 16, 8 rows 419 / 420).  By the room in the cache: where the rows are is not known here.
static int step_wgs(int E, int64_t keys) { return E <= 1024 && (keys < NC_STEP_MANY_KEYS || nc_cu_count() < 256) ? 128 : 256; }

bool nc_step_fits(int B, int L, int E, int H, int Hkv) {
    if (B < 1 || B > NC_STEP_ROWS || L < 3 || L > NC_STEP_MAX_LAYERS || E > NC_STEP_MAX_E || E != H * 128 || Hkv < 1 || (H != Hkv && H != 2 * Hkv)) return false;
    return nc_cu_count() >= step_wgs(E, 0);
}

// A round of tiles of all of a step's products, in polls: a workgroup takes in some 4 KB of weights between two of them (us for one more round, measured with so many workgroups started:
// depth 4, one row 4, depth 10, 3 rows 47, depth 20, 8 rows 170, depth 26, 8 rows 270).
static uint32_t round_polls(const NcStepArgs& a) {
    return (uint32_t)((int64_t)a.L * a.E * (a.E * 10 + a.Hkv * 256) / a.wgs / 4096);
}

uint32_t nc_step_list_polls(const NcStepArgs& a, int registered) { return list_polls((uint32_t)registered, (uint32_t)a.wgs, a.round_polls); }

size_t nc_step_exchange(NcStepArgs& a, int most_keys, int mean_keys) {
    int at = 0;
    auto take = [&](int bytes) {
        const int here = at;
        at += (bytes + 255) & ~255;
        return here;
    };
    a.wgs = step_wgs(a.E, (int64_t)a.B * a.Hkv * mean_keys), a.round_polls = round_polls(a);
    take(a.B * (a.H + 2 * a.Hkv) * 256);
    a.off_y = take(a.B * a.E * 2);
    a.off_proj = take(a.B * a.E * 2);
    a.off_h = take(a.B * a.E * 8);
    a.off_mlp = take(a.B * a.E * 2);
    a.layer_bytes = at;
    a.parts = a.exchange + (size_t)a.layer_bytes * a.L;
    const int pairs = a.B * a.Hkv;
    a.parts_bytes = (pairs * (step_splits(most_keys, a.wgs, pairs) - 1) * (a.H / a.Hkv) * MERGE_STRIDE * 4 + 255) & ~255;
    return (size_t)(a.layer_bytes + a.parts_bytes) * a.L;
}

template <int NV, int G>
static int launch(const NcStepArgs& a, const NcStepLayers& layers, int present, hipStream_t s) {
    const int lds_bytes = panel_bytes<G>(a.E) + NC_STEP_ROWS * a.E * 2 + GW * NV * 512;
    static std::atomic<uint64_t> has_lds{0};          // a bit per device
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0) dev = 0;
    if (dev >= 64 || !(has_lds.load(std::memory_order_relaxed) >> dev & 1)) {
        const hipError_t e = hipFuncSetAttribute((const void*)step_kernel<NV, G>, hipFuncAttributeMaxDynamicSharedMemorySize, 120 * 1024);
        if (e != hipSuccess) NC_FAIL(-2, "step: %s", hipGetErrorString(e));
        if (dev < 64) has_lds.fetch_or(1ull << dev, std::memory_order_relaxed);
    }
    hipLaunchKernelGGL((step_kernel<NV, G>), dim3(present), dim3(THREADS), lds_bytes, s, a, layers);
    NC_CHECK_LAUNCH("step");
    return 0;
}

int nc_launch_step(const NcStepArgs& a, const NcStepLayers& layers, int present, hipStream_t s) {
    NC_CHECK_ARG(nc_step_fits(a.B, a.L, a.E, a.H, a.Hkv) && (a.wgs == 256 || (a.wgs == 128 && a.E <= 1024)) && present >= 0 && present <= a.wgs, "step: not a shape of this kernel");
    if (present == 0) present = a.wgs;
#define STEP(NVV) (a.H == a.Hkv ? launch<NVV, 1>(a, layers, present, s) : launch<NVV, 2>(a, layers, present, s))
    return a.E <= 512 ? STEP(1) : a.E <= 1024 ? STEP(2) : a.E <= 1536 ? STEP(3) : STEP(4);
#undef STEP
}
