// One head of the q|k|v post-processing of CausalSelfAttention.forward (nanochat/gpt.py:89-104), done by one wave:
// lane L holds elements L and L+64 of the 128-wide head, which is exactly one rotary pair.
//   q and k heads: rotary by the position's angle -> rms_norm over the head -> * 1.2
//   v heads:       v + 3*sigmoid(W_g . xn[:12])[head] * ve[token id, head, :]   (layers with a value embedding)
// Every value is rounded to bf16 wherever the eager bf16 graph of the reference materialises a tensor.
// Shared by the stand-alone rotary/append kernel and by the decode attention kernel that does this work itself.
#pragma once
#include "nc_common.h"
#include "nc_kernels.h"

#define RMS_EPS 1.1920928955078125e-07f   // fp32 machine epsilon: F.rms_norm's default eps

__device__ __forceinline__ float sigmoidf_(float x) { return 1.0f / (1.0f + expf(-x)); }

struct NcRopeSrc {
    const bf16_t* qkv;        // bf16 [tokens, ld_qkv] output of the q|k|v linear, or nullptr when it is still in partials
    int ld_qkv;
    NcPartialSrc pq;
    const bf16_t* xn;         // normalised layer input (the value-embedding gate reads its first 12 channels)
    int ld_xn;
    const int64_t* idx;       // token ids
    const bf16_t* ve_table;   // nullptr: layer without value embedding
    const float* ve_gate_w;
    const bf16_t* cos_t;
    const bf16_t* sin_t;
    int rope_len;
    int vocab_rows;
    const bf16_t* k_new;      // only for the attention kernel's plain-append form: finished new keys / values [tokens, Hkv, 128]
    const bf16_t* v_new;
};

// The loads of one head, issued in one go so that their latency is paid once and a caller can put other loads behind them:
// the first PRE split partials (or the bf16 value), the rotary pair or the value-embedding pair, and for a value head the
// twelve gate inputs (lane c < 12 holds channel c).
template <int PRE>
struct RopeRaw {
    // exactly what the loads returned: a conversion at load time would make the loading code wait for the value
    float t1[PRE], t2[PRE];   // partial sums; without partials t1[0], t2[0] hold the two bf16 values as loaded (bits in the low half)
    uint32_t e1, e2;          // q, k heads: cos, sin;  v heads with a value embedding: ve[lane], ve[lane + 64]   (bf16 bits)
    uint32_t xg;              // v heads: xn[lane] for lane < 12   (bf16 bits)
    float inv_b;              // partials: inverse weight scale of the head's segment
};

// hh in [0, H): query head; [H, H+Hkv): key head; [H+Hkv, H+2Hkv): value head.
template <int PRE>
__device__ __forceinline__ void rope_head_load(const NcRopeSrc& r, int token, int pos, int hh, int H, int Hkv, int lane, RopeRaw<PRE>& w) {
    // every field gets a value before the first load is issued (a store to a register that may hold a pending load makes the
    // compiler wait for the load; an unset field sends the whole struct to scratch memory)
    w.e1 = w.e2 = w.xg = 0u;
    w.inv_b = 0.f;
#pragma unroll
    for (int u = 0; u < PRE; u++) w.t1[u] = w.t2[u] = 0.f;
    if (r.pq.parts) {
        const float* pp = r.pq.parts + (size_t)token * r.pq.ld + hh * 128 + lane;
#pragma unroll
        for (int u = 0; u < PRE; u++) {
            const size_t o = (size_t)(u < r.pq.nsplit ? u : 0) * r.pq.split_stride;
            w.t1[u] = pp[o], w.t2[u] = pp[o + 64];
        }
        // q | k | v segments end on head boundaries, so the head decides the segment
        w.inv_b = r.pq.inv_b[hh * 128 >= r.pq.seg_end1 ? 2 : (hh * 128 >= r.pq.seg_end0 ? 1 : 0)];
    } else {
        const bf16_t* src = r.qkv + (size_t)token * r.ld_qkv + (size_t)hh * 128;
        w.t1[0] = __uint_as_float((uint32_t)src[lane]), w.t2[0] = __uint_as_float((uint32_t)src[lane + 64]);
    }
    if (hh < H + Hkv) {
        const int rp = pos < r.rope_len ? (pos < 0 ? 0 : pos) : r.rope_len - 1;
        w.e1 = r.cos_t[(size_t)rp * 64 + lane], w.e2 = r.sin_t[(size_t)rp * 64 + lane];
        w.xg = r.cos_t[lane];      // never read for a q or k head; loaded so that xg is the result of a load on every path (see above)
    } else if (r.ve_table) {
        const int hv = hh - H - Hkv;
        int64_t tok = r.idx[token];
        if (tok < 0 || tok >= r.vocab_rows) tok = 0;
        const bf16_t* ve = r.ve_table + ((size_t)tok * Hkv + hv) * 128;
        w.e1 = ve[lane], w.e2 = ve[lane + 64];
        w.xg = r.xn[(size_t)token * r.ld_xn + (lane < 12 ? lane : 0)];
    }
}

// Returns the finished pair.
template <int PRE>
__device__ __forceinline__ void rope_head_finish(const NcRopeSrc& r, int token, int hh, int H, int Hkv, int lane, const RopeRaw<PRE>& w,
                                                 float a_amax /* amax of the linear's input (the word(s) r.pq.a_amax names), read by the caller; used with partials only */, float& o1,
                                                 float& o2) {
    // The conversions below must stay here: moved up to the loads (the compiler does that when it merges the branches of the load
    // step) they would make the loading code wait.  An empty asm that "rewrites" the raw values pins their first use to this point.
    uint32_t e1 = w.e1, e2 = w.e2, xg = w.xg;
    float t10 = w.t1[0], t20 = w.t2[0];
    asm volatile("" : "+v"(e1), "+v"(e2), "+v"(xg), "+v"(t10), "+v"(t20)::"memory");
    float x1, x2;
    if (r.pq.parts) {
        // the linear's output still sits in split partials: add them up in split order, scale, round to bf16
        const int col = hh * 128 + lane;
        float a1 = 0.f, a2 = 0.f;
#pragma unroll
        for (int u = 0; u < PRE; u++)
            if (u < r.pq.nsplit) a1 += u ? w.t1[u] : t10, a2 += u ? w.t2[u] : t20;
        // splits beyond the first PRE, eight at a time, loads first, sums after (see mix_norm_vec_kernel)
        const float* pp = r.pq.parts + (size_t)token * r.pq.ld + col;
        for (int sp0 = PRE; sp0 < r.pq.nsplit; sp0 += 8) {
            float t1[8], t2[8];
#pragma unroll
            for (int u = 0; u < 8; u++) {
                const size_t o = (size_t)(sp0 + u < r.pq.nsplit ? sp0 + u : sp0) * r.pq.split_stride;
                t1[u] = pp[o], t2[u] = pp[o + 64];
            }
#pragma unroll
            for (int u = 0; u < 8; u++)
                if (sp0 + u < r.pq.nsplit) a1 += t1[u], a2 += t2[u];
        }
        const float inv_a = 1.0f / scale_from_amax(a_amax);
        x1 = rbf((a1 * inv_a) * w.inv_b);
        x2 = rbf((a2 * inv_a) * w.inv_b);
    } else {
        x1 = bf16_to_f32((bf16_t)__float_as_uint(t10)), x2 = bf16_to_f32((bf16_t)__float_as_uint(t20));
    }
    if (hh < H + Hkv) {
        const float c = bf16_to_f32((bf16_t)e1), s = bf16_to_f32((bf16_t)e2);
        float y1 = rbf(rbf(x1 * c) + rbf(x2 * s));
        float y2 = rbf(rbf(x1 * (-s)) + rbf(x2 * c));
        const float ss = wave_sum(y1 * y1 + y2 * y2);
        const float rstd = 1.0f / sqrtf(ss / 128.0f + RMS_EPS);
        o1 = rbf(rbf(y1 * rstd) * 1.2f);
        o2 = rbf(rbf(y2 * rstd) * 1.2f);
    } else {
        const int hv = hh - H - Hkv;
        if (r.ve_table) {
            float dot = 0.f;
#pragma unroll
            for (int cidx = 0; cidx < 12; cidx++)
                dot += bf16_to_f32((bf16_t)__builtin_amdgcn_readlane((int)xg, cidx)) * rbf(r.ve_gate_w[hv * 12 + cidx]);
            const float gate = rbf(3.0f * rbf(sigmoidf_(rbf(dot))));
            x1 = rbf(x1 + rbf(gate * bf16_to_f32((bf16_t)e1)));
            x2 = rbf(x2 + rbf(gate * bf16_to_f32((bf16_t)e2)));
        }
        o1 = x1, o2 = x2;
    }
}

__device__ __forceinline__ void rope_head(const NcRopeSrc& r, int token, int pos, int hh, int H, int Hkv, int lane, float& o1, float& o2) {
    RopeRaw<8> w;
    const uint32_t amax_lane = r.pq.parts ? amax_load_lane(r.pq.a_amax) : 0u;
    rope_head_load(r, token, pos, hh, H, Hkv, lane, w);
    rope_head_finish(r, token, hh, H, Hkv, lane, w, amax_from_lanes(amax_lane), o1, o2);
}

// ------------------------------------------------------------------------------------------------
// The same for many tokens whose q|k|v rows are finished bf16 values: eight lanes share a head, each holding eight consecutive elements of its first half
// and the eight they pair with in the second half (element j rotates with j + 64), all accesses 16 bytes wide; the mean of squares of the QK-norm is a
// sum over the 8 lanes.  Same rounding points as rope_head_finish.  Used by the stand-alone kernel and by the epilogue of the q|k|v linear.
struct NcRopeDst {
    const int32_t* cache_seqlens;
    bf16_t *k_cache, *v_cache, *q_out;
    int T, H, Hkv, Tmax;
};
struct RopeVecRaw {           // what one head of one token needs beside its values, as loaded
    uint4 e1, e2;             // q, k heads: cos, sin;  v heads with a value embedding: its two halves
    uint4 xg0;
    uint2 xg1;                // v heads: xn[0 .. 11]
    int b, pos;
};
__device__ __forceinline__ void rope_vec_load(const NcRopeSrc& r, const NcRopeDst& d, int token, int hh, int part, RopeVecRaw& w) {
    w.b = token / d.T;
    w.pos = d.cache_seqlens[w.b] + token % d.T;
    w.e1 = w.e2 = w.xg0 = make_uint4(0, 0, 0, 0);
    w.xg1 = make_uint2(0, 0);
    if (hh < d.H + d.Hkv) {
        const int rp = w.pos < r.rope_len ? (w.pos < 0 ? 0 : w.pos) : r.rope_len - 1;
        w.e1 = *(const uint4*)(r.cos_t + (size_t)rp * 64 + part * 8), w.e2 = *(const uint4*)(r.sin_t + (size_t)rp * 64 + part * 8);
    } else if (r.ve_table) {
        int64_t tok = r.idx[token];
        if (tok < 0 || tok >= r.vocab_rows) tok = 0;
        const bf16_t* ve = r.ve_table + ((size_t)tok * d.Hkv + (hh - d.H - d.Hkv)) * 128 + part * 8;
        w.e1 = *(const uint4*)ve, w.e2 = *(const uint4*)(ve + 64);
        const bf16_t* xg = r.xn + (size_t)token * r.ld_xn;
        w.xg0 = *(const uint4*)xg, w.xg1 = *(const uint2*)(xg + 8);
    }
}
// The arithmetic is what bounds it (1792 tokens of 39 heads: 6 us of instructions over the whole chip): two roundings to a conversion.
__device__ __forceinline__ void rbf2(float& a, float& b) {
    const uint32_t u = pack_bf16(a, b);
    a = bf16_lo(u), b = bf16_hi(u);
}
// xa, xb: the lane's elements of the head; every lane of the eight takes part, `live` ones store
__device__ __forceinline__ void rope_vec_finish(const NcRopeSrc& r, const NcRopeDst& d, const RopeVecRaw& w, uint4 xa, uint4 xb, int token, int hh, int part, bool live) {
    const uint32_t wa[4] = {xa.x, xa.y, xa.z, xa.w}, wb[4] = {xb.x, xb.y, xb.z, xb.w};
    const uint32_t ea[4] = {w.e1.x, w.e1.y, w.e1.z, w.e1.w}, eb[4] = {w.e2.x, w.e2.y, w.e2.z, w.e2.w};
    float x1[8], x2[8], o1[8], o2[8];
#pragma unroll
    for (int j = 0; j < 4; j++) {
        x1[2 * j] = bf16_lo(wa[j]), x1[2 * j + 1] = bf16_hi(wa[j]);
        x2[2 * j] = bf16_lo(wb[j]), x2[2 * j + 1] = bf16_hi(wb[j]);
    }
    if (hh < d.H + d.Hkv) {
        float ss = 0.f;
#pragma unroll
        for (int e = 0; e < 8; e++) {
            const float c = (e & 1) ? bf16_hi(ea[e >> 1]) : bf16_lo(ea[e >> 1]);
            const float sn = (e & 1) ? bf16_hi(eb[e >> 1]) : bf16_lo(eb[e >> 1]);
            float a = x1[e] * c, b = x2[e] * sn, f = x1[e] * (-sn), g = x2[e] * c;
            rbf2(a, b), rbf2(f, g);
            a += b, f += g;
            rbf2(a, f);
            o1[e] = a, o2[e] = f;
            ss += o1[e] * o1[e] + o2[e] * o2[e];
        }
        ss += __shfl_xor(ss, 1);
        ss += __shfl_xor(ss, 2);
        ss += __shfl_xor(ss, 4);
        const float rstd = 1.0f / sqrtf(ss / 128.0f + RMS_EPS);
#pragma unroll
        for (int e = 0; e < 8; e++) {
            float a = o1[e] * rstd, b = o2[e] * rstd;
            rbf2(a, b);
            o1[e] = a * 1.2f, o2[e] = b * 1.2f;               // (rounded where they are packed)
        }
    } else {
#pragma unroll
        for (int e = 0; e < 8; e++) o1[e] = x1[e], o2[e] = x2[e];
        if (r.ve_table) {
            const int hv = hh - d.H - d.Hkv;
            const uint32_t xg[6] = {w.xg0.x, w.xg0.y, w.xg0.z, w.xg0.w, w.xg1.x, w.xg1.y};
            float dot = 0.f;
#pragma unroll
            for (int c = 0; c < 12; c++) dot += ((c & 1) ? bf16_hi(xg[c >> 1]) : bf16_lo(xg[c >> 1])) * rbf(r.ve_gate_w[hv * 12 + c]);
            const float gate = rbf(3.0f * rbf(sigmoidf_(rbf(dot))));
#pragma unroll
            for (int e = 0; e < 8; e++) {
                const float v1 = (e & 1) ? bf16_hi(ea[e >> 1]) : bf16_lo(ea[e >> 1]);
                const float v2 = (e & 1) ? bf16_hi(eb[e >> 1]) : bf16_lo(eb[e >> 1]);
                float a = gate * v1, b = gate * v2;
                rbf2(a, b);
                o1[e] += a, o2[e] += b;                       // (rounded where they are packed)
            }
        }
    }
    if (!live) return;
    bf16_t* dst;
    if (hh < d.H) dst = d.q_out + ((size_t)token * d.H + hh) * 128;
    else {
        if (w.pos < 0 || w.pos >= d.Tmax) return;
        const bool is_k = hh < d.H + d.Hkv;
        dst = (is_k ? d.k_cache : d.v_cache) + (((size_t)w.b * d.Tmax + w.pos) * d.Hkv + (is_k ? hh - d.H : hh - d.H - d.Hkv)) * 128;
    }
    dst += part * 8;
    *(uint4*)dst = make_uint4(pack_bf16(o1[0], o1[1]), pack_bf16(o1[2], o1[3]), pack_bf16(o1[4], o1[5]), pack_bf16(o1[6], o1[7]));
    *(uint4*)(dst + 64) = make_uint4(pack_bf16(o2[0], o2[1]), pack_bf16(o2[2], o2[3]), pack_bf16(o2[4], o2[5]), pack_bf16(o2[6], o2[7]));
}
// what the eight lanes ask of their pointers
static inline bool rope_vec_aligned(const NcRopeSrc& r, const NcRopeDst& d) {
    return r.ld_xn % 8 == 0 && (((uintptr_t)d.k_cache | (uintptr_t)d.v_cache | (uintptr_t)d.q_out | (uintptr_t)r.cos_t | (uintptr_t)r.sin_t | (uintptr_t)r.ve_table | (uintptr_t)r.xn) & 15) == 0;
}
