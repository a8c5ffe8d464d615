// A meeting of all workgroups of a launch on the maximum of what each of them holds in its registers: the producers of an FP8 linear's input learn
// the tensorwise amax while the tensor is still in registers and write it as e4m3 at once, where a conversion launch would read it back.
//
// Memory (NC_MEETING_WORDS words, all zero before the launch): one word per workgroup, its maximum with the top bit set once it has arrived, and
// behind them one bit per workgroup that left (below).  One trip to memory out, one back: every workgroup stores its word and polls everybody's, so
// there is no counter for hundreds of atomics to queue up at.  What the polls cost grows with the square of the workgroups, all of them reading the same
// lines (row passes of 1792 rows: 112 workgroups 12.1 us, 224 10.7, 448 13.7), so few large workgroups meet best; a launch that meets has at most
// NC_MEETING_WGS (nc_meeting_wgs).  Words and bits are read and written with device-scope atomics, at the device's point of coherence; no fence is needed on the way everybody takes.
//
// The launch is sized so that the chip holds all of it, but a workgroup may still not have started because another stream's kernel has its place.
// The wait is therefore bounded: a workgroup whose polls run out LEAVES.  It stores its values as bf16 in memory, makes them visible, sets its bit and
// looks once more; then it ends, which makes room for who has not started.  Whoever completes the meeting finds the bits and converts
// what was left behind (meeting_take: each bit is taken by one workgroup).  No bit is overlooked: the workgroup Z whose word came last finds the
// meeting complete at its first poll and reads the bits after its word was acknowledged; a leaver either finds Z's word at its last look (and
// goes on like everybody), or its bit was set before Z's word was and Z sees it.
#pragma once
#include "nc_common.h"
#include "nc_kernels.h"

#define NC_MEETING_WGS 256               // a word and a bit each, and every poll looks at all of them
#define NC_MEETING_WORDS (NC_MEETING_WGS + NC_MEETING_WGS / 32)
#define NC_MEETING_SPINS 400u             // polls of about half a microsecond before a workgroup leaves

static_assert(NC_MEETING_WGS % 64 == 0 && NC_MEETING_WGS / 32 <= 64, "a wave looks at 64 words at a time and at all bits at once");

// how many workgroups of one to a compute unit can meet
static inline int nc_meeting_wgs() { return nc_cu_count() < NC_MEETING_WGS ? nc_cu_count() : NC_MEETING_WGS; }

struct NcMeeting {
    uint32_t* words;          // nullptr: none
    uint32_t spins;
};

// rows that a kernel writes as e4m3 after a meeting
struct NcQuantRows {
    uint8_t* out;             // [rows][cols]
    float* inv_out;
    NcMeeting meeting;
    int rows;
};

struct MeetingView {
    bool complete;            // everybody's word is there:
    uint32_t amax;            //   the maximum of all
    bool left;                //   somebody has left values behind
};

// For one whole wave of the workgroup (a maximum is a non-negative float's bits, NaN included).
__device__ __forceinline__ MeetingView meeting_look(const NcMeeting& m, int wgs) {
    const int lane = threadIdx.x & 63;
    constexpr int POLLS = NC_MEETING_WGS / 64;
    uint32_t v[POLLS];
#pragma unroll
    for (int i = 0; i < POLLS; i++) {
        const int w = i * 64 + lane;
        v[i] = w < wgs ? __hip_atomic_load(m.words + w, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) : 0x80000000u;
    }
    const uint32_t bits = lane < NC_MEETING_WGS / 32 ? __hip_atomic_load(m.words + NC_MEETING_WGS + lane, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) : 0u;
    uint32_t all = 0x80000000u, mx = 0u;
#pragma unroll
    for (int i = 0; i < POLLS; i++) {
        const uint32_t a = v[i] & 0x7fffffffu;
        all &= v[i], mx = a > mx ? a : mx;
    }
    return MeetingView{__builtin_amdgcn_ballot_w64(all == 0u) == 0, mx, __builtin_amdgcn_ballot_w64(bits != 0u) != 0};
}
__device__ __forceinline__ MeetingView meeting_wait(const NcMeeting& m, int wgs) {
    for (uint32_t spin = 0;; spin++) {
        MeetingView view = meeting_look(m, wgs);
        if (view.complete || spin >= m.spins) {
            view.amax = wave_max_u32(view.amax);
            return view;
        }
        __builtin_amdgcn_s_sleep(4);
    }
}

// The whole meeting, for every thread of a workgroup of WAVES waves; am: each thread's maximum.  meanwhile(): what can be stored while the words travel;
// leave() stores the workgroup's values as bf16.
// Returns false when the workgroup left (its values are in memory and somebody else's business), else true with the tensor's amax and whether
// meeting_take has to be called once the workgroup's own values are converted.
template <int WAVES, typename Meanwhile, typename Leave>
__device__ __forceinline__ bool meeting(const NcMeeting& m, int wgs, int self, float am, float& amax, bool& left, Meanwhile&& meanwhile, Leave&& leave) {
    __shared__ uint32_t red[WAVES], out[3];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    am = wave_amax(am);
    if (lane == 0) red[wave] = __float_as_uint(am);
    __syncthreads();
    uint32_t before = 0u;
    if (threadIdx.x == 0) {
        uint32_t t = red[0];
#pragma unroll
        for (int w = 1; w < WAVES; w++) t = red[w] > t ? red[w] : t;
        before = __hip_atomic_exchange(m.words + self, t | 0x80000000u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    meanwhile();
    if (wave == 0) {
        asm volatile("" ::"v"(before) : "memory");       // the word is there (the exchange has returned) before anything is looked at
        const MeetingView view = meeting_wait(m, wgs);
        if (lane == 0) out[0] = view.complete, out[1] = view.amax, out[2] = view.left;
    }
    __syncthreads();
    if (!out[0]) {
        leave();
        __threadfence();                      // everything this thread stored is visible to the device ...
        __syncthreads();
        if (wave == 0) {
            if (lane == 0) {                  // ... before the bit is
                const uint32_t before = __hip_atomic_fetch_or(m.words + NC_MEETING_WGS + self / 32, 1u << (self % 32), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                asm volatile("" ::"v"(before) : "memory");
            }
            asm volatile("" ::: "memory");
            __builtin_amdgcn_s_waitcnt(0);
            asm volatile("" ::: "memory");
            MeetingView view = meeting_look(m, wgs);
            view.amax = wave_max_u32(view.amax);
            if (lane == 0) out[0] = view.complete, out[1] = view.amax, out[2] = view.left;
        }
        __syncthreads();
        if (!out[0]) return false;
    }
    amax = __uint_as_float(out[1]), left = out[2] != 0;
    return true;
}

// Converts what workgroups have left behind; convert(w) is called by all threads together for each workgroup w that this one takes over.
template <typename Convert>
__device__ __forceinline__ void meeting_take(const NcMeeting& m, int wgs, Convert&& convert) {
    __shared__ uint32_t got;
    for (int w = 0; w < wgs; w++) {
        __syncthreads();
        if (threadIdx.x == 0) {
            uint32_t* const p = m.words + NC_MEETING_WGS + w / 32;
            const uint32_t bit = 1u << (w % 32);
            got = (__hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) & bit) != 0 &&
                  (__hip_atomic_fetch_and(p, ~bit, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) & bit) != 0;
        }
        __syncthreads();
        if (!got) continue;
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
        convert(w);
    }
}

// four bf16 values, and sixteen (two 16-byte vectors), as e4m3
__device__ __forceinline__ uint32_t e4m3_of_bf16x4(uint32_t lo, uint32_t hi, float scale) {
    return fp8_pack4<0, true>(clamp448(bf16_lo(lo) * scale), clamp448(bf16_hi(lo) * scale), clamp448(bf16_lo(hi) * scale), clamp448(bf16_hi(hi) * scale));
}
__device__ __forceinline__ uint4 e4m3_of_bf16x16(const uint4& a, const uint4& b, float scale) {
    return make_uint4(e4m3_of_bf16x4(a.x, a.y, scale), e4m3_of_bf16x4(a.z, a.w, scale), e4m3_of_bf16x4(b.x, b.y, scale), e4m3_of_bf16x4(b.z, b.w, scale));
}
// what the launch leaves beside the values: once, by whoever converts workgroup 0's
__device__ __forceinline__ void meeting_result(float amax, float scale, float* inv_out, uint32_t* out_amax) {
    *inv_out = 1.0f / scale;
    if (out_amax) amax_publish(out_amax, amax);
}
