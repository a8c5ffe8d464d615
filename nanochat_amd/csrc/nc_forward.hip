// Host-side sequencing of one GPT.forward(idx, kv_cache=...) on a stream: the native replacement of the
// Python loop at nanochat/gpt.py:459-524 (and of the module calls it makes into gpt.py:84-153 and
// fp8.py:202-213).  One call enqueues every kernel of the step; no host synchronisation, no allocation.
//
// A decode step of up to 8 rows (where nc_step_fits): three launches, embedding, all layers, lm_head.
// Per layer, decode otherwise (M = B*T <= 128 rows), 7 or 8 launches, each making a single dependent trip to memory:
//   mix_norm            x += mlp_out(prev) [read from split partials]; x = rl*x + xl*x0; xn = norm(x); amax(xn)
//   linear q|k|v        quantize xn inside the GEMM; K split over workgroups           -> fp32 partials
//   attention           each (row, kv head) workgroup first sums its heads' partials (three weight scales), applies
//                       rotary, QK-norm, gain and the VE gate, appends key and value to the cache, then attends over
//                       the cache; amax(y)                                             -> y
//                       (small batches, where attention is split over several workgroups per head, and T > 1 keep the
//                       stand-alone qkv_rope_append kernel in front)
//   linear c_proj       quantize y inside                                              -> partials
//   mix_norm            x += o [from partials]; xn = norm(x); amax(xn)
//   linear c_fc         quantize xn inside; up to 64 rows of up to 2048 columns relu^2 and amax as well -> h2, otherwise -> partials and
//   finish_partials     sum, scale, relu^2, amax                                       -> h2
//   linear mlp c_proj   quantize h2 inside                                             -> partials (added by the next mix_norm)
// Prefill (M > 128) uses the tiled GEMM instead of the fused small-M linear.  Where its workgroups are all resident at once (and the call has more than one
// token per row for the third), a producer writes what the next launch reads, 8 launches a layer instead of 12:
//   mix_norm            the workgroups meet on the amax of the rows and write them as e4m3
//   linear c_fc         relu^2, the meeting, e4m3
//   linear q|k|v        rotary, QK-norm, gain, VE gate and append in its epilogue
// otherwise the convert kernel and the rotary kernel follow as launches of their own.  Attention's launch also reads the weights of the next linears ahead
// where that pays (reads_ahead, nc_prefetch.h); its output goes through the convert kernel.  The two narrow projections of a few hundred rows leave partial sums to mix_norm as well.
//
// Workspace (carved from the caller's buffer, 256-byte aligned pieces), M = B*T rows:
//   x, x0, xn, xb, o      bf16 [M,E]        residual stream, its initial value, normed rows, backout, GEMM out
//   qkv                   bf16 [M,(H+2Hkv)*128]
//   qh, y                 bf16 [M,H*128]    rotated queries, attention output
//   h, h2                 bf16 [M,4E]       c_fc output (prefill only; or relu^2 of it as e4m3), relu^2
//   a8                    u8   [M,4E]       quantized activations (prefill only)
//   xl                    bf16 [B,E]        last-position rows (last_only lm_head at T > 1)
//   inv                   fp32 [4L+1]       activation inverse scales (prefill only)
//   zeroed                u32               amax sites [4L+1] x 8 slots on separate lines | attention split counters,
//                                           | meetings (prefill only), cleared by the embedding kernel at the start of the call
//   gemm_parts, attn_parts                  split partials of the small-M linears and of attention
//   step_words, step_exchange               the one launch of a step of few rows (nc_step.hip): registration, and what its workgroups hand each other
#include <stdio.h>
#include "../../include/nanochat_amd.h"
#include "nc_common.h"
#include "nc_kernels.h"
#include "nc_meeting.h"
#include "nc_prefetch.h"
#include "nc_rope.h"

#define TRY(call)              \
    do {                       \
        int rc__ = (call);     \
        if (rc__) return rc__; \
    } while (0)

// Reading a shared prompt once for all rows costs two more launches per layer (the stand-alone rotary kernel and the shared-keys kernel,
// ~12-14 us together with the merge) and saves the per-row streaming of the shared keys the layer sees: rows x kv heads x keys x 512
// bytes at ~6 TB/s.  It is taken when that is at least ~14 us: 164 000 (row, kv head, key) units -- 197 shared keys at 64 rows of 13
// heads (a full-context layer always; a 512-key window until it has moved most of the way out of the prompt), 394 at 32 rows.
// (measured through the harness at d26, 1792-token prompt: 8 / 16 / 32 rows 1.38 / 1.58 / 2.14 -> 1.30 / 1.43 / 1.79 ms per step)
#define NC_SHARED_MIN_ROW_HEADS 64
#define NC_SHARED_MIN_KEYS 128
#define NC_SHARED_MIN_UNITS 164000L

namespace {
struct Carver {
    uint8_t* base;
    size_t off = 0;
    explicit Carver(void* p) : base((uint8_t*)p) {}
    template <typename T>
    T* take(size_t count) {
        off = (off + 255) & ~(size_t)255;
        T* r = base ? (T*)(base + off) : nullptr;
        off += count * sizeof(T);
        return r;
    }
};

struct Workspace {
    bf16_t *x, *x0, *xn, *xb, *o, *qkv, *qh, *y, *h, *h2, *xl;
    bf16_t* x2;                // second residual-stream buffer of the one- and two-row decode step (see fused_rows())
    uint8_t* a8;
    float* inv;
    uint32_t *amax, *attn_counters;
    // handle of amax site i (tagged: NC_AMAX_SLOTS words on separate lines, see amax_read / amax_publish)
    uint32_t* site(int i) const { return nc_amax_slotted(amax + (size_t)i * NC_AMAX_SLOTS * NC_AMAX_STRIDE); }
    uint32_t* meetings;        // prompts: one per amax site, for the launches that write their site's e4m3 rows themselves
    NcMeeting meeting(int i) const { return NcMeeting{meetings + (size_t)i * NC_MEETING_WORDS, NC_MEETING_SPINS}; }
    int zero_words;
    uint8_t *gemm_parts, *gemm_parts2, *attn_parts, *shared_parts;
    uint32_t* step_words;      // steps of few rows (nc_step.hip): NC_STEP_WORDS, and the amax site of the rows they leave
    uint8_t* step_exchange;
    size_t step_exchange_bytes;
    uint32_t* step_site() const { return nc_amax_slotted(step_words + NC_STEP_WORDS); }
    size_t gemm_part_bytes, attn_part_bytes, shared_part_bytes;
    size_t total;
};

// One or two rows (a chat session's decode step): the residual/norm passes and the relu^2 pass are folded into the linears that consume
// them (NcRowRecipe), five launches per layer instead of eight.  Each such linear reads its input recipe's partial sums from one
// buffer and writes its own into the other, and the residual stream alternates between two buffers in the same way, because the
// workgroups of one launch must not overwrite what their neighbours still read.
bool fused_rows(const nc_model_desc* m, int M) {
    const int E = m->n_embd, qkv_w = (m->n_head + 2 * m->n_kv_head) * 128;
    if (M > NC_RECIPE_MAX_ROWS || E > 2048 || 4 * E > NC_RECIPE_MAX_K || E % 8 != 0) return false;
    // every linear of a layer must leave split partial sums (the recipe of the next one reads them)
    return nc_gemm_decode_splits(qkv_w, E) > 1 && nc_gemm_decode_splits(E, m->n_head * 128) > 1 && nc_gemm_decode_splits(4 * E, E) > 1 &&
           nc_gemm_decode_splits(E, 4 * E) > 1;
}

constexpr int STEP_CLEARED = NC_STEP_WORDS + NC_AMAX_SLOTS * NC_AMAX_STRIDE;

Workspace carve(const nc_model_desc* m, int B, int T, void* base) {
    const size_t M = (size_t)B * T, E = m->n_embd;
    const size_t qkv_w = (size_t)(m->n_head + 2 * m->n_kv_head) * 128;
    const bool small = M <= 128;
    Carver c(base);
    Workspace w;
    w.x = c.take<bf16_t>(M * E);
    w.x2 = c.take<bf16_t>(fused_rows(m, (int)M) ? M * E : 0);
    w.x0 = c.take<bf16_t>(M * E);
    w.xn = c.take<bf16_t>(M * E);
    w.xb = c.take<bf16_t>(M * E);
    w.o = c.take<bf16_t>(M * E);
    w.qkv = c.take<bf16_t>(M * qkv_w);
    w.qh = c.take<bf16_t>(M * m->n_head * 128);
    w.y = c.take<bf16_t>(M * m->n_head * 128);
    w.h = c.take<bf16_t>(small ? 0 : M * 4 * E);
    w.h2 = c.take<bf16_t>(M * 4 * E);
    w.a8 = c.take<uint8_t>(small ? 0 : M * 4 * E);
    w.xl = c.take<bf16_t>((size_t)B * E);
    w.inv = c.take<float>(4 * (size_t)m->n_layer + 1);
    const size_t amax_words = (4 * (size_t)m->n_layer + 1) * NC_AMAX_SLOTS * NC_AMAX_STRIDE;     // one slotted site per FP8 linear input
    // attention split counters and partials only when some layer's launch really splits its keys over workgroups (never with 16 or
    // more queries per row, which take the matrix-core kernel, and never once rows x kv heads fill the chip); the cache length is not
    // known here, so each layer is sized for its whole window
    int max_splits = 1;
    if (T < 16)
        for (int i = 0; i < m->n_layer; i++) {
            const int sp = nc_attn_splits(B, T, m->n_kv_head, m->layers ? m->layers[i].window_left : -1, 1 << 30);
            max_splits = sp > max_splits ? sp : max_splits;
        }
    const size_t attn_words = max_splits > 1 ? nc_attn_counter_bytes(B, T, m->n_head) / 4 : 0;
    const size_t meeting_words = small ? 0 : (4 * (size_t)m->n_layer + 1) * NC_MEETING_WORDS;
    uint32_t* zero = c.take<uint32_t>(amax_words + attn_words + meeting_words);
    w.amax = zero;
    w.attn_counters = zero ? zero + amax_words : nullptr;
    w.meetings = zero ? zero + amax_words + attn_words : nullptr;
    w.zero_words = (int)(amax_words + attn_words + meeting_words);
    size_t gneed = 0;
    if (small) {
        const int shapes[5][2] = {{(int)qkv_w, (int)E}, {(int)E, m->n_head * 128}, {(int)(4 * E), (int)E}, {(int)E, (int)(4 * E)},
                                  {m->vocab_size, (int)E}};
        for (auto& sh : shapes) {
            const size_t n = nc_gemm_decode_partial_bytes_auto((int)M, sh[0], sh[1]);
            gneed = n > gneed ? n : gneed;
        }
    } else {
        const int shapes[2][2] = {{(int)E, m->n_head * 128}, {(int)E, (int)(4 * E)}};
        for (auto& sh : shapes) {
            const int ks = nc_gemm_prompt_splits((int)M, sh[0], sh[1]);
            const size_t n = ks > 1 ? ks * M * sh[0] * sizeof(float) : 0;
            gneed = n > gneed ? n : gneed;
        }
    }
    w.gemm_part_bytes = gneed;
    w.gemm_parts = c.take<uint8_t>(gneed);
    w.gemm_parts2 = c.take<uint8_t>(fused_rows(m, (int)M) ? gneed : 0);
    w.attn_part_bytes = max_splits > 1 ? nc_attn_partial_bytes(B, T, m->n_head) / 16 * max_splits : 0;
    w.attn_parts = c.take<uint8_t>(w.attn_part_bytes);
    // partial results of the shared first part of the cache (rows that begin with one replicated prompt): whatever the shared length
    // turns out to be, the launch cuts it into at most as many chunks as a whole cache row would get
    w.shared_part_bytes = (T == 1 && (long)B * m->n_kv_head >= NC_SHARED_MIN_ROW_HEADS) ? nc_attn_shared_partial_bytes(B, m->n_head, m->n_kv_head, 1 << 20) : 0;
    w.shared_parts = c.take<uint8_t>(w.shared_part_bytes);
    const bool step = T == 1 && nc_step_fits(B, m->n_layer, m->n_embd, m->n_head, m->n_kv_head);
    w.step_words = c.take<uint32_t>(step ? STEP_CLEARED : 0);
    NcStepArgs sizes{};
    sizes.B = B, sizes.L = m->n_layer, sizes.E = m->n_embd, sizes.H = m->n_head, sizes.Hkv = m->n_kv_head;
    w.step_exchange_bytes = step ? nc_step_exchange(sizes, NC_STEP_MAX_KEYS, NC_STEP_MAX_KEYS) : 0;      // (the most it takes: the cache's length is not known here)
    w.step_exchange = c.take<uint8_t>(w.step_exchange_bytes);
    w.total = (c.off + 255) & ~(size_t)255;
    return w;
}

// Whether the attention launches of a prompt read the weights of the linears behind them ahead (nc_prefetch.h), E (qkv_w + H 128 + 8 E) bytes a layer.
// The tiles of more than 128 rows wait for their weights.  Up to 64 rows the linears are streams of the weight themselves and gain nothing, while attention
// (6.6 us for 40 tokens of 13 heads) ends with the reading (9.8 us for 33 MB): us without / with, depth 26, 16 tokens 1229 / 1281, 32 1377 / 1415, 64 1565 / 1604.  Between
// the two it depends on whether the reading ends with attention: 20 MB (depth 20) 65 tokens 1274 / 1246, 128 1446 / 1390, 4 x 17 1255 / 1265, 24 MB (depth 22) 65
// tokens 1476 / 1463, 128 1663 / 1633, but 28 MB (depth 24) 65 tokens 1592 / 1607, 4 x 24 1698 / 1711, 33 MB (depth 26) 65 tokens 1851 / 1867, 128 2113 / 2098, 4 x 20
// 1906 / 1922.  Beyond 128 rows, depth 26: 8 x 32 1854 / 1761, 64 x 16 3001 / 2733.
constexpr size_t AHEAD_LAYER_BYTES_FEW = 24u << 20;
bool reads_ahead(const nc_model_desc* m, int M) {
    const size_t E = m->n_embd, layer = E * ((size_t)(2 * m->n_head + 2 * m->n_kv_head) * 128 + 8 * E);
    return M > 128 || (M > 64 && layer <= AHEAD_LAYER_BYTES_FEW);
}

// cached keys that a row sees in a layer when its cache is full: at most, and in the mean of the layers
struct VisibleKeys {
    int most, mean;
};
VisibleKeys visible_keys(const nc_model_desc* m, int Tmax) {
    int most = 0;
    int64_t sum = 0;
    for (int i = 0; i < m->n_layer; i++) {
        const int w = m->layers[i].window_left, n = w >= 0 && w < Tmax ? w : Tmax;
        most = n > most ? n : most, sum += n;
    }
    return VisibleKeys{most, (int)(sum / m->n_layer)};
}

// Whether a step goes through nc_step.hip.  Launches of their own have what one has not: times of each kernel (the profiler), rows of any alignment, a
// prompt that is read once for all rows, and a model without the subtraction at its end.
bool takes_step(const nc_model_desc* m, const nc_cache_desc* kv, int B) {
    const uintptr_t pointers = (uintptr_t)m->wte | (uintptr_t)kv->prev_in | (uintptr_t)kv->prev_out | (uintptr_t)kv->k_cache | (uintptr_t)kv->v_cache;
    return nc_step_fits(B, m->n_layer, m->n_embd, m->n_head, m->n_kv_head) && !nc_prof_on() && (pointers & 15) == 0 && m->backout_lambda &&
           kv->max_seq_len < NC_STEP_MAX_KEYS && !(kv->shared_prefix > 0 && B * m->n_kv_head >= NC_SHARED_MIN_ROW_HEADS);
}

// One launch reads what all layers point at: what the separate launches refuse, each where it comes to it, is refused in front of it.
int check_step(const nc_model_desc* m, const nc_cache_desc* kv) {
    NC_CHECK_ARG(m->layers && m->resid_lambdas && m->x0_lambdas, "gpt_forward: layers or their lambdas missing");
    NC_CHECK_ARG(m->cos && m->sin && m->rope_len > 0, "gpt_forward: rotary source missing");
    NC_CHECK_ARG(kv->max_seq_len > 0, "gpt_forward: a cache of %d tokens", kv->max_seq_len);
    for (int i = 0; i < m->n_layer; i++) {
        const nc_layer_desc& ly = m->layers[i];
        NC_CHECK_ARG(ly.w_qkv && ly.inv_qkv && ly.w_attn_proj && ly.w_fc && ly.w_mlp_proj, "gpt_forward: layer %d has no FP8 weights", i);
        NC_CHECK_ARG(ly.inv_attn_proj && ly.inv_fc && ly.inv_mlp_proj, "gpt_forward: layer %d has no weight scales", i);
        NC_CHECK_ARG((((uintptr_t)ly.w_qkv | (uintptr_t)ly.w_attn_proj | (uintptr_t)ly.w_fc | (uintptr_t)ly.w_mlp_proj) & 15) == 0,
                     "gpt_forward: layer %d: weights must be 16-byte aligned", i);
        NC_CHECK_ARG(!ly.ve_table || ly.ve_gate_w, "gpt_forward: layer %d: value embedding needs gate weights", i);
    }
    return 0;
}

NcGemmSegs one_seg(int n) { return NcGemmSegs{1, {n, 0, 0, 0}}; }

__global__ void gather_last_rows_kernel(const bf16_t* __restrict__ x, bf16_t* __restrict__ out, int T, int E) {
    const int b = blockIdx.x;
    const bf16_t* src = x + ((size_t)b * T + (T - 1)) * E;
    for (int c = threadIdx.x; c < E; c += blockDim.x) out[(size_t)b * E + c] = src[c];
}

const NcPartialSrc NO_PARTIALS{nullptr, 0, 0, 0, nullptr, nullptr, 0, 0};

int tap_copy(bf16_t* dst, const bf16_t* src, size_t elems, hipStream_t s) {
    const hipError_t e = hipMemcpyAsync(dst, src, elems * sizeof(bf16_t), hipMemcpyDeviceToDevice, s);
    if (e != hipSuccess) NC_FAIL(-2, "gpt_forward: tap copy failed: %s", hipGetErrorString(e));
    return 0;
}

// One FP8 linear on `rows` rows of bf16 input whose amax sits in slot `site`.  Small M: the result is either
// in `out` (single split: epilogue done in the GEMM) or described by *src (split partials for the consumer).
struct LinearRunner {
    const Workspace& w;
    hipStream_t s;
    // The same linear with its input rows made inside the kernel (one or two rows); the partial sums go to `parts_buf`.
    int run_recipe(const NcRowRecipe& recipe, int rows, int site, const uint8_t* w8, const float* inv_w, NcGemmSegs segs, int N, int K,
                   uint8_t* parts_buf, NcPartialSrc* src) const {
        int used = 1;
        const int want = nc_gemm_decode_splits(N, K);
        // (a single split would need the epilogue in the GEMM; every linear of a layer splits K, and the recipe path relies on it)
        NC_CHECK_ARG(want > 1, "gpt_forward: the fused small-batch step needs split linears (N=%d K=%d)", N, K);
        TRY(nc_launch_gemm_decode(nullptr, 1, nullptr, nullptr, w8, inv_w, segs, nullptr, 0, 0.f, nullptr, rows, N, K, N, (float*)parts_buf,
                                  w.gemm_part_bytes, want, &used, s, &recipe));
        *src = NcPartialSrc{(const float*)parts_buf, used, N, (size_t)rows * N, w.site(site), inv_w,
                            segs.nseg > 1 ? segs.end[0] : 0x7fffffff, segs.nseg > 2 ? segs.end[1] : 0x7fffffff};
        return 0;
    }
    // relu^2 of a linear of many rows as e4m3 at w.h, its inverse scale in w.inv + out_site; false: not a shape of that launch
    bool run_relu2_e4m3(const bf16_t* in, const uint8_t* in8, int rows, int site, const uint8_t* w8, const float* inv_w, int N, int K, int out_site, const uint8_t** out8, int* rc) const {
        *out8 = nullptr;
        if (rows <= 128 || !nc_gemm_relu2_e4m3_kernel(rows, N, K)) return false;
        *rc = in8 ? 0 : nc_launch_convert_only(in, (int64_t)rows * K, w.a8, w.inv + site, w.site(site), s);
        if (!*rc) *rc = nc_launch_gemm_relu2_e4m3(in8 ? in8 : w.a8, w8, w.inv + site, inv_w, (uint8_t*)w.h, w.inv + out_site, w.site(out_site), w.h2,
                                                   w.meeting(out_site), rows, N, K, s);
        *out8 = (const uint8_t*)w.h;
        return true;
    }
    int run(const bf16_t* in, int rows, int site, const uint8_t* w8, const float* inv_w, NcGemmSegs segs, void* out, int out_kind,
            float softcap, uint32_t* out_amax, int N, int K, int ldc, NcPartialSrc* src, uint8_t* parts_buf = nullptr, const uint8_t* in8 = nullptr) const {
        if (src) *src = NO_PARTIALS;
        uint8_t* const pbuf = parts_buf ? parts_buf : w.gemm_parts;
        if (rows <= 128) {
            int used = 1;
            TRY(nc_launch_gemm_decode(in, 1, w.site(site), nullptr, w8, inv_w, segs, out, out_kind, softcap, out_amax, rows, N, K, ldc,
                                      (float*)pbuf, w.gemm_part_bytes, src || out_kind == 2 ? 0 : 1, &used, s));
            if (used == 1) return 0;
            if (src) {
                *src = NcPartialSrc{(const float*)pbuf, used, N, (size_t)rows * N, w.site(site), inv_w,
                                    segs.nseg > 1 ? segs.end[0] : 0x7fffffff, segs.nseg > 2 ? segs.end[1] : 0x7fffffff};
                return 0;
            }
            return nc_launch_finish_partials((const float*)pbuf, used, w.site(site), nullptr, inv_w, segs, out, out_kind, softcap,
                                             out_amax, rows, N, ldc, s);
        }
        // large M: explicit convert pass (unless the rows are e4m3 already: in8, their inverse scale in w.inv + site), tiled GEMM
        if (!in8) {
            TRY(nc_launch_convert_only(in, (int64_t)rows * K, w.a8, w.inv + site, w.site(site), s));
            in8 = w.a8;
        }
        const int splits = src && out_kind == 0 && segs.nseg == 1 ? nc_gemm_prompt_splits(rows, N, K) : 1;
        if (splits > 1) {
            TRY(nc_launch_gemm_partials(in8, w8, (float*)pbuf, w.gemm_part_bytes, splits, rows, N, K, s));
            *src = NcPartialSrc{(const float*)pbuf, splits, N, (size_t)rows * N, w.site(site), inv_w, 0x7fffffff, 0x7fffffff};
            return 0;
        }
        if (out_kind == 2) {
            // relu^2 and its amax in the GEMM's epilogue; past the 32-bit buffer offsets, the plain-load kernel and a separate pass
            if ((long)rows * K < (1L << 31) && (long)N * K < (1L << 31))
                return nc_launch_gemm(in8, w8, w.inv + site, inv_w, segs, out, 2, 0.f, rows, N, K, ldc, 0, nullptr, 0, s, 0, out_amax);
            TRY(nc_launch_gemm(in8, w8, w.inv + site, inv_w, segs, w.h, 0, 0.f, rows, N, K, N, 0, nullptr, 0, s));
            return nc_launch_relu2(w.h, (bf16_t*)out, (int64_t)rows * N, out_amax, s);
        }
        return nc_launch_gemm(in8, w8, w.inv + site, inv_w, segs, out, out_kind, softcap, rows, N, K, ldc, 0, nullptr, 0, s);
    }
};
}  // namespace

extern "C" size_t nc_gpt_workspace_bytes(const nc_model_desc* model, int B, int T) {
    if (!model || B <= 0 || T <= 0) return 0;
    return carve(model, B, T, nullptr).total;
}

extern "C" int nc_gpt_reads_ahead(const nc_model_desc* model, int B, int T) { return model && B > 0 && T >= 16 && reads_ahead(model, B * T); }

// tap_x (or nullptr): bf16 [L+1, M, E], slot i = the residual stream as layer i reads it (after the lambda mix, gpt.py:500), slot L = the
// final normalised rows (gpt.py:508).  tap_y (or nullptr): bf16 [L, M, H*128], the attention outputs before c_proj (gpt.py:113-124).
static int gpt_forward_impl(const nc_model_desc* m, const nc_cache_desc* kv, const int64_t* idx, int B, int T, float* logits_out,
                            int last_only, void* workspace, size_t workspace_bytes, bf16_t* tap_x, bf16_t* tap_y, hipStream_t s, int present = 0,
                            uint32_t wait_polls = NC_STEP_WAIT_POLLS) {
    NC_CHECK_ARG(m && kv && idx && logits_out && workspace, "gpt_forward: null pointer");
    NC_CHECK_ARG(B > 0 && T > 0, "gpt_forward: bad batch/time B=%d T=%d", B, T);
    NC_CHECK_ARG(m->n_embd == m->n_head * 128, "gpt_forward: head_dim must be 128 (n_embd=%d n_head=%d)", m->n_embd, m->n_head);
    NC_CHECK_ARG(m->n_embd % 16 == 0 && m->n_embd >= 128, "gpt_forward: n_embd=%d must pass the FP8 filter", m->n_embd);
    NC_CHECK_ARG(kv->batch == B, "gpt_forward: cache batch %d != B %d", kv->batch, B);
    NC_CHECK_ARG(kv->k_cache && kv->v_cache && kv->cache_seqlens && kv->prev_out, "gpt_forward: cache pointers missing");
    NC_CHECK_ARG(((uintptr_t)workspace & 255) == 0, "gpt_forward: workspace must be 256-byte aligned");
    Workspace w = carve(m, B, T, workspace);
    NC_CHECK_ARG(workspace_bytes >= w.total, "gpt_forward: workspace of %zu bytes needed, %zu given", w.total, workspace_bytes);

    const int L = m->n_layer, E = m->n_embd, H = m->n_head, Hkv = m->n_kv_head, M = B * T;
    const int qkv_w = (H + 2 * Hkv) * 128;
    const size_t layer_elems = (size_t)B * kv->max_seq_len * Hkv * 128;
    const LinearRunner lin{w, s};
    int site = 0;   // amax / inv slot of the next FP8 linear input

    // a step of few rows: embedding, one launch for all layers, lm_head
    if (T == 1 && !tap_x && !tap_y && takes_step(m, kv, B)) {
        TRY(check_step(m, kv));
        NcStepArgs a{};
        a.x0 = w.x0, a.xb = w.xb, a.xn = w.xn, a.exchange = w.step_exchange, a.words = w.step_words, a.head_site = w.step_site();
        a.k_cache = kv->k_cache, a.v_cache = kv->v_cache, a.cache_seqlens = (int32_t*)kv->cache_seqlens, a.idx = idx, a.cos_t = m->cos, a.sin_t = m->sin;
        a.resid_lambdas = m->resid_lambdas, a.x0_lambdas = m->x0_lambdas, a.backout_lambda = m->backout_lambda;
        a.layer_elems = layer_elems;
        a.B = B, a.L = L, a.E = E, a.H = H, a.Hkv = Hkv, a.Tmax = kv->max_seq_len, a.rope_len = m->rope_len, a.vocab_rows = m->padded_vocab, a.advance = kv->advance;
        a.wait_polls = wait_polls;
        NcStepLayers layers{};
        for (int i = 0; i < L; i++) {
            const nc_layer_desc& ly = m->layers[i];
            layers.layer[i] = NcStepLayer{ly.w_qkv, ly.inv_qkv, ly.w_attn_proj, ly.inv_attn_proj, ly.w_fc, ly.inv_fc, ly.w_mlp_proj, ly.inv_mlp_proj,
                                          ly.ve_table, ly.ve_gate_w, ly.window_left, 0};
        }
        const VisibleKeys keys = visible_keys(m, kv->max_seq_len);
        const size_t fill = nc_step_exchange(a, keys.most, keys.mean);
        NC_CHECK_ARG(fill <= w.step_exchange_bytes, "gpt_forward: exchange of %zu bytes, %zu in the workspace", fill, w.step_exchange_bytes);
        TRY(nc_launch_embed_norm_smear(idx, m->wte, m->smear_w, m->smear_lambda, kv->prev_in, kv->prev_out, w.x, w.x0, B, T, E, m->padded_vocab, w.step_words,
                                       STEP_CLEARED, s, w.step_exchange, fill));
        TRY(nc_launch_step(a, layers, present, s));
        return nc_launch_gemm_decode(w.xn, 1, w.step_site(), nullptr, m->w_lm_head, m->inv_lm_head, one_seg(m->vocab_size), logits_out, 1, m->softcap, nullptr, M,
                                     m->vocab_size, E, m->vocab_size, (float*)w.gemm_parts, w.gemm_part_bytes, 1, nullptr, s);
    }
    NC_CHECK_ARG(present == 0, "gpt_forward: not a step that one launch takes");

    // x0 is the post-smear embedding; layer 0 reads it through both x and x0 (gpt.py:495,500)
    TRY(nc_launch_embed_norm_smear(idx, m->wte, m->smear_w, m->smear_lambda, kv->prev_in, kv->prev_out, w.x, w.x0, B, T, E,
                                   m->padded_vocab, w.amax, w.zero_words, s));

    // output of the previous MLP projection, still to be added into the residual stream: bf16 rows or split partials
    const bf16_t* pending_add = nullptr;
    NcPartialSrc pending_parts = NO_PARTIALS;
    // rows8: whether the pass left its rows as e4m3 in w.a8, their inverse scale in w.inv (a prompt's layers; the last rows are gathered first)
    const uint8_t* rows8 = nullptr;
    auto mix = [&](const float* rl, const float* xl, const float* bl, const bf16_t* bsrc, bf16_t* save, uint32_t* amax,
                   int32_t* bump = nullptr, int bump_by = 0, bool to_e4m3 = false) -> int {
        const NcQuantRows q8{w.a8, w.inv + site, to_e4m3 ? w.meeting(site) : NcMeeting{}, M};
        const NcQuantRows* const q = to_e4m3 && M > 128 && nc_mix_norm_e4m3_fits(M, E, pending_parts.parts != nullptr) ? &q8 : nullptr;
        rows8 = q ? w.a8 : nullptr;
        if (pending_parts.parts)
            return nc_launch_mix_norm_p(w.x, pending_parts, w.x0, rl, xl, bl, bsrc, save, w.xn, M, E, amax, s, bump, bump_by, q);
        return nc_launch_mix_norm(w.x, pending_add, w.x0, rl, xl, bl, bsrc, save, w.xn, M, E, amax, s, bump, bump_by, q);
    };
    // (measured at d26, steps without a synchronisation in between: one row 1.30 -> 1.13 ms, two rows 1.37 -> 1.27 ms)
    const bool fused = T == 1 && fused_rows(m, M);
    bf16_t *xcur = w.x, *xalt = w.x2;            // fused step: the residual stream alternates between the two
    uint8_t *pin = w.gemm_parts, *pout = w.gemm_parts2;      // ... and so do the partial sums: pending_parts always sits in `pin`
    for (int i = 0; i < L && fused; i++) {
        const nc_layer_desc& ly = m->layers[i];
        NC_CHECK_ARG(ly.w_qkv && ly.inv_qkv && ly.w_attn_proj && ly.w_fc && ly.w_mlp_proj, "gpt_forward: layer %d has no FP8 weights", i);
        // q|k|v linear on rows it makes itself: x += mlp_out(prev layer); [save backout]; x = rl*x + xl*x0; xn = norm(x)
        NcRowRecipe mix1{};
        mix1.kind = 1, mix1.x_in = xcur, mix1.x_out = xalt, mix1.add = nullptr, mix1.padd = pending_parts, mix1.x0 = w.x0;
        mix1.resid_lambda = m->resid_lambdas + i, mix1.x0_lambda = m->x0_lambdas + i;
        mix1.save = (i > 0 && (i - 1) == L / 2) ? w.xb : nullptr, mix1.xn_out = w.xn, mix1.amax_out = w.site(site);
        NcGemmSegs qkv_segs{3, {H * 128, (H + Hkv) * 128, qkv_w, 0}};
        NcPartialSrc qsrc;
        TRY(lin.run_recipe(mix1, M, site, ly.w_qkv, ly.inv_qkv, qkv_segs, qkv_w, E, pout, &qsrc));
        { bf16_t* t = xcur; xcur = xalt; xalt = t; }
        { uint8_t* t = pin; pin = pout; pout = t; }          // the q|k|v partial sums are in `pin` now
        site++;
        if (tap_x) TRY(tap_copy(tap_x + (size_t)i * M * E, xcur, (size_t)M * E, s));
        bf16_t* kc = kv->k_cache + (size_t)i * layer_elems;
        bf16_t* vc = kv->v_cache + (size_t)i * layer_elems;
        const NcRopeSrc rope{nullptr, qkv_w, qsrc, w.xn, E, idx, ly.ve_table, ly.ve_gate_w, m->cos, m->sin, m->rope_len, m->padded_vocab,
                             nullptr, nullptr};
        TRY(nc_launch_attention_fused(rope, kc, vc, kv->cache_seqlens, ly.window_left, w.y, B, H, Hkv, kv->max_seq_len, w.attn_counters,
                                      w.attn_parts, w.attn_part_bytes, w.site(site), 0, 1, s));
        if (tap_y) TRY(tap_copy(tap_y + (size_t)i * M * H * 128, w.y, (size_t)M * H * 128, s));
        // attention c_proj reads y as before; its partial sums go to the other buffer (the q|k|v ones are consumed by now)
        TRY(lin.run(w.y, M, site, ly.w_attn_proj, ly.inv_attn_proj, one_seg(E), w.o, 0, 0.f, nullptr, E, H * 128, E, &pending_parts, pout));
        NC_CHECK_ARG(pending_parts.parts, "gpt_forward: the fused small-batch step needs a split attention projection");
        { uint8_t* t = pin; pin = pout; pout = t; }
        site++;
        // c_fc on rows it makes itself: x += attn_out; xn = norm(x)
        NcRowRecipe mix2{};
        mix2.kind = 1, mix2.x_in = xcur, mix2.x_out = xalt, mix2.padd = pending_parts, mix2.xn_out = w.xn, mix2.amax_out = w.site(site);
        NcPartialSrc fsrc;
        TRY(lin.run_recipe(mix2, M, site, ly.w_fc, ly.inv_fc, one_seg(4 * E), 4 * E, E, pout, &fsrc));
        { bf16_t* t = xcur; xcur = xalt; xalt = t; }
        { uint8_t* t = pin; pin = pout; pout = t; }
        site++;
        // MLP projection on rows it makes itself: h2 = relu(c_fc(xn))^2
        NcRowRecipe act{};
        act.kind = 2, act.padd = fsrc, act.amax_out = w.site(site);
        TRY(lin.run_recipe(act, M, site, ly.w_mlp_proj, ly.inv_mlp_proj, one_seg(E), E, 4 * E, pout, &pending_parts));
        { uint8_t* t = pin; pin = pout; pout = t; }
        site++;
    }
    if (fused && xcur != w.x) {
        // the last pass below works on w.x
        const hipError_t e = hipMemcpyAsync(w.x, xcur, (size_t)M * E * sizeof(bf16_t), hipMemcpyDeviceToDevice, s);
        if (e != hipSuccess) NC_FAIL(-2, "gpt_forward: copy of the residual rows failed: %s", hipGetErrorString(e));
    }
    for (int i = 0; i < L && !fused; i++) {
        const nc_layer_desc& ly = m->layers[i];
        NC_CHECK_ARG(ly.w_qkv && ly.inv_qkv && ly.w_attn_proj && ly.w_fc && ly.w_mlp_proj, "gpt_forward: layer %d has no FP8 weights", i);
        // x += mlp_out(prev layer); [save backout]; x = rl*x + xl*x0; xn = norm(x)
        bf16_t* save = (i > 0 && (i - 1) == L / 2) ? w.xb : nullptr;
        TRY(mix(m->resid_lambdas + i, m->x0_lambdas + i, nullptr, nullptr, save, w.site(site), nullptr, 0, true));
        if (tap_x) TRY(tap_copy(tap_x + (size_t)i * M * E, w.x, (size_t)M * E, s));
        // q|k|v = FP8 linear(xn): one activation quantization, three weight scales
        NcGemmSegs qkv_segs{3, {H * 128, (H + Hkv) * 128, qkv_w, 0}};
        bf16_t* kc = kv->k_cache + (size_t)i * layer_elems;
        bf16_t* vc = kv->v_cache + (size_t)i * layer_elems;
        NcPartialSrc qsrc = NO_PARTIALS;
        bool heads_done = false;
        if (T > 1 && M > 128) {
            // a prompt: the linear finishes its heads itself
            if (!rows8) {
                TRY(nc_launch_convert_only(w.xn, (int64_t)M * E, w.a8, w.inv + site, w.site(site), s));
                rows8 = w.a8;
            }
            const NcRopeSrc rope{nullptr, qkv_w, NO_PARTIALS, w.xn, E, idx, ly.ve_table, ly.ve_gate_w, m->cos, m->sin, m->rope_len, m->padded_vocab, nullptr, nullptr};
            const int rc = nc_launch_gemm_qkv_rope(rows8, ly.w_qkv, w.inv + site, ly.inv_qkv, qkv_segs, rope,
                                                   NcRopeDst{kv->cache_seqlens, kc, vc, w.qh, T, H, Hkv, kv->max_seq_len}, M, E, s);
            if (rc < 0) return rc;
            heads_done = rc == 0;
        }
        if (!heads_done) TRY(lin.run(w.xn, M, site, ly.w_qkv, ly.inv_qkv, qkv_segs, w.qkv, 0, 0.f, nullptr, qkv_w, E, qkv_w, &qsrc, nullptr, rows8));
        site++;
        // rows that begin with one replicated prompt: a layer that sees a long stretch of it reads that stretch once for all rows
        bool shared_done = false;
        if (T == 1 && (long)B * Hkv >= NC_SHARED_MIN_ROW_HEADS && kv->shared_prefix > 0 && kv->uniform_pos >= kv->shared_prefix && w.shared_parts) {
            const int first_visible = ly.window_left < 0 ? 0 : (kv->uniform_pos - ly.window_left > 0 ? kv->uniform_pos - ly.window_left : 0);
            const int shared_visible = kv->shared_prefix - first_visible;
            if (shared_visible >= NC_SHARED_MIN_KEYS && (long)shared_visible * B * Hkv >= NC_SHARED_MIN_UNITS && kv->shared_prefix < kv->max_seq_len) {
                if (qsrc.parts)
                    TRY(nc_launch_qkv_rope_append_p(qsrc, w.xn, E, idx, ly.ve_table, ly.ve_gate_w, m->cos, m->sin, m->rope_len,
                                                    kv->cache_seqlens, kc, vc, w.qh, B, T, H, Hkv, kv->max_seq_len, m->padded_vocab, s));
                else
                    TRY(nc_launch_qkv_rope_append(w.qkv, qkv_w, w.xn, E, idx, ly.ve_table, ly.ve_gate_w, m->cos, m->sin, m->rope_len,
                                                  kv->cache_seqlens, kc, vc, w.qh, B, T, H, Hkv, kv->max_seq_len, m->padded_vocab, s));
                TRY(nc_launch_attention_shared(w.qh, kc, vc, kv->cache_seqlens, kv->shared_prefix, ly.window_left, w.y, B, H, Hkv,
                                               kv->max_seq_len, 0, w.shared_parts, w.shared_part_bytes, w.site(site), s));
                shared_done = true;
            }
        }
        if (shared_done) {
            // (q, the new cache rows and the attention output are already written)
        } else if (T == 1) {
            // decode: the attention workgroups finish their own q|k|v heads and append to the cache themselves
            const NcRopeSrc rope{qsrc.parts ? nullptr : w.qkv, qkv_w, qsrc, w.xn, E, idx, ly.ve_table, ly.ve_gate_w, m->cos, m->sin,
                                 m->rope_len, m->padded_vocab, nullptr, nullptr};
            TRY(nc_launch_attention_fused(rope, kc, vc, kv->cache_seqlens, ly.window_left, w.y, B, H, Hkv, kv->max_seq_len,
                                          w.attn_counters, w.attn_parts, w.attn_part_bytes, w.site(site), 0, 1, s));
        } else {
            if (heads_done) {
            } else if (qsrc.parts)
                TRY(nc_launch_qkv_rope_append_p(qsrc, w.xn, E, idx, ly.ve_table, ly.ve_gate_w, m->cos, m->sin, m->rope_len,
                                                kv->cache_seqlens, kc, vc, w.qh, B, T, H, Hkv, kv->max_seq_len, m->padded_vocab, s));
            else
                TRY(nc_launch_qkv_rope_append(w.qkv, qkv_w, w.xn, E, idx, ly.ve_table, ly.ve_gate_w, m->cos, m->sin, m->rope_len,
                                              kv->cache_seqlens, kc, vc, w.qh, B, T, H, Hkv, kv->max_seq_len, m->padded_vocab, s));
            // meanwhile the weights of the linears up to the next attention come out of HBM
            NcAhead ahead{};
            if (reads_ahead(m, M)) {
                ahead.add(ly.w_attn_proj, (size_t)E * H * 128);
                ahead.add(ly.w_fc, (size_t)4 * E * E);
                ahead.add(ly.w_mlp_proj, (size_t)4 * E * E);
                if (i + 1 < L) ahead.add(m->layers[i + 1].w_qkv, (size_t)qkv_w * E);
                else ahead.add(m->w_lm_head, (size_t)m->vocab_size * E);
            }
            TRY(nc_launch_attention(w.qh, kc, vc, kv->cache_seqlens, ly.window_left, w.y, B, T, H, Hkv, kv->max_seq_len, 0,
                                    w.attn_counters, w.attn_parts, w.attn_part_bytes, w.site(site), 0, 1, s, &ahead));
        }
        if (tap_y) TRY(tap_copy(tap_y + (size_t)i * M * H * 128, w.y, (size_t)M * H * 128, s));
        TRY(lin.run(w.y, M, site, ly.w_attn_proj, ly.inv_attn_proj, one_seg(E), w.o, 0, 0.f, nullptr, E, H * 128, E, &pending_parts));
        pending_add = pending_parts.parts ? nullptr : w.o;
        site++;
        // x += attn_out; xn = norm(x)
        TRY(mix(nullptr, nullptr, nullptr, nullptr, nullptr, w.site(site), nullptr, 0, true));
        // h2 = relu(c_fc(xn))^2 with its amax in the next slot, or as e4m3
        const uint8_t* h8;
        int rc = 0;
        if (!lin.run_relu2_e4m3(w.xn, rows8, M, site, ly.w_fc, ly.inv_fc, 4 * E, E, site + 1, &h8, &rc))
            rc = lin.run(w.xn, M, site, ly.w_fc, ly.inv_fc, one_seg(4 * E), w.h2, 2, 0.f, w.site(site + 1), 4 * E, E, 4 * E, nullptr, nullptr, rows8);
        if (rc) return rc;
        site++;
        TRY(lin.run(w.h2, M, site, ly.w_mlp_proj, ly.inv_mlp_proj, one_seg(E), w.o, 0, 0.f, nullptr, E, 4 * E, E, &pending_parts, nullptr, h8));
        pending_add = pending_parts.parts ? nullptr : w.o;
        site++;
    }
    // x += mlp_out(last layer); x -= backout_lambda * x_backout; xn = norm(x)      (gpt.py:506-508)
    {
        const bool last_is_backout = (L - 1) == L / 2;     // L == 1 or 2
        if (last_is_backout) {
            // the saved rows and the subtraction need the same x1: do the add first, then the backout pass
            TRY(mix(nullptr, nullptr, nullptr, nullptr, w.xb, nullptr));
            pending_add = nullptr;
            pending_parts = NO_PARTIALS;
        }
        // every layer has read the positions by now: a one-token step may have them advanced here instead of by a launch of the caller's
        const bool bump = kv->advance != 0 && T == 1 && E % 8 == 0 && E <= 8192;
        NC_CHECK_ARG(kv->advance == 0 || bump, "gpt_forward: cache_desc.advance needs T == 1 (and n_embd %% 8 == 0, <= 8192)");
        TRY(mix(nullptr, nullptr, m->backout_lambda, w.xb, nullptr, w.site(site), bump ? (int32_t*)kv->cache_seqlens : nullptr, kv->advance));
        if (tap_x) TRY(tap_copy(tap_x + (size_t)L * M * E, w.xn, (size_t)M * E, s));
    }
    // lm_head.  Its activation scale is tensorwise over all M rows (that is what the reference quantizes),
    // even when only the last position of every row is projected.
    const bf16_t* head_in = w.xn;
    int head_rows = M;
    if (last_only && T > 1) {
        hipLaunchKernelGGL(gather_last_rows_kernel, dim3(B), dim3(256), 0, s, w.xn, w.xl, T, E);
        NC_CHECK_LAUNCH("gather_last_rows");
        head_in = w.xl;
        head_rows = B;
    }
    TRY(lin.run(head_in, head_rows, site, m->w_lm_head, m->inv_lm_head, one_seg(m->vocab_size), logits_out, 1, m->softcap, nullptr,
                m->vocab_size, E, m->vocab_size, nullptr));
    return 0;
}

extern "C" int nc_gpt_forward(const nc_model_desc* m, const nc_cache_desc* kv, const int64_t* idx, int B, int T, float* logits_out,
                              int last_only, void* workspace, size_t workspace_bytes, nc_stream_t stream) {
    return gpt_forward_impl(m, kv, idx, B, T, logits_out, last_only, workspace, workspace_bytes, nullptr, nullptr, (hipStream_t)stream);
}

extern "C" int nc_gpt_step_list_polls(const nc_model_desc* m, int B, int max_seq_len, int registered) {
    if (!m || !m->layers || !nc_step_fits(B, m->n_layer, m->n_embd, m->n_head, m->n_kv_head)) return 0;
    NcStepArgs a{};
    a.B = B, a.L = m->n_layer, a.E = m->n_embd, a.H = m->n_head, a.Hkv = m->n_kv_head;
    const VisibleKeys keys = visible_keys(m, max_seq_len);
    (void)nc_step_exchange(a, keys.most, keys.mean);
    return (int)nc_step_list_polls(a, registered);
}

extern "C" int nc_gpt_forward_present(const nc_model_desc* m, const nc_cache_desc* kv, const int64_t* idx, int B, float* logits_out, void* workspace,
                                      size_t workspace_bytes, int present, nc_stream_t stream) {
    NC_CHECK_ARG(present > 0, "gpt_forward_present: no workgroups");
    return gpt_forward_impl(m, kv, idx, B, 1, logits_out, 1, workspace, workspace_bytes, nullptr, nullptr, (hipStream_t)stream, present);
}

extern "C" int nc_gpt_forward_giving_up(const nc_model_desc* m, const nc_cache_desc* kv, const int64_t* idx, int B, float* logits_out, void* workspace,
                                        size_t workspace_bytes, int present, int wait_polls, nc_stream_t stream) {
    NC_CHECK_ARG(present > 0 && wait_polls > 0, "gpt_forward_giving_up: %d workgroups, %d polls", present, wait_polls);
    return gpt_forward_impl(m, kv, idx, B, 1, logits_out, 1, workspace, workspace_bytes, nullptr, nullptr, (hipStream_t)stream, present, (uint32_t)wait_polls);
}

extern "C" int nc_gpt_forward_tapped(const nc_model_desc* m, const nc_cache_desc* kv, const int64_t* idx, int B, int T, float* logits_out,
                                     int last_only, void* workspace, size_t workspace_bytes, uint16_t* tap_x, uint16_t* tap_y,
                                     nc_stream_t stream) {
    return gpt_forward_impl(m, kv, idx, B, T, logits_out, last_only, workspace, workspace_bytes, tap_x, tap_y, (hipStream_t)stream);
}
