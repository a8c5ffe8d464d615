// Linears of the layer stack:  out[M,N] = A[M,K] . W[N,K]^T  on the matrix cores, bfloat16 (v_mfma_f32_16x16x32_bf16) or true 32-bit
// (v_mfma_f32_16x16x4_f32) operands, 32-bit sums.  Both formats share one data path counted in bytes: a lane supplies 16 bytes of row
// (lane & 15) from K-piece (lane >> 4), which is one bf16 instruction or four fp32 ones -- which k a lane's bytes stand for does not
// matter as long as both operands agree.  Operands are issued as (W, A), so a lane ends up with four consecutive output columns of
// one output row.
//
//   linear_tiled_kernel  tiles of 32 x 64 to 128 x 256 outputs, operands straight into a ring of LDS stages; the summed index may be dealt to
//                        several workgroups, whose consumer adds their sums.
//   linear_big_kernel    bf16 tiles of 256 x 256 (and halves of 256 x 128 behind whole rounds of them), unsplit, for many rows.
//   linear_few_kernel    few rows of a small weight, or a summed index that is no multiple of 64: operands straight into registers, no LDS in
//                        the loop.
//
// A stacked weight is several matrices that read the same input; the epilogue sends each run of output columns its own way (store,
// gelu, silu, GLUs, softplus, router logits, residual add, soft-capped logits).  Rows can be grouped by weight (experts).
#include <atomic>
#include "nc_stack.h"

typedef __bf16 v8bf __attribute__((ext_vector_type(8)));
typedef __attribute__((address_space(3))) void* lds_ptr_t;

namespace {
template <typename T> struct Mma;
template <> struct Mma<bf16_t> {
    static __device__ __forceinline__ v4f run(const v4i& w, const v4i& a, const v4f& c) {
        return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(v8bf, w), __builtin_bit_cast(v8bf, a), c, 0, 0, 0);
    }
};
template <> struct Mma<float> {
    static __device__ __forceinline__ v4f run(const v4i& w, const v4i& a, const v4f& c) {
        const v4f wf = __builtin_bit_cast(v4f, w), af = __builtin_bit_cast(v4f, a);
        v4f r = c;
#pragma unroll
        for (int j = 0; j < 4; j++) r = __builtin_amdgcn_mfma_f32_16x16x4f32(wf[j], af[j], r, 0, 0, 0);
        return r;
    }
};

// One instruction of the same.  PARTS instructions make up 16 bytes; the caller puts other accumulators between them.  The memory operations on
// both sides stay on their sides, so that the loads and LDS reads of a step lie between its products as they are written.  (The builtin, not an asm
// statement: the compiler has to see a matrix instruction to keep its distance from the copies and zeros that it puts around it.)
template <typename T> constexpr int MMA_PARTS = sizeof(T) == 2 ? 1 : 4;
template <typename T>
__device__ __forceinline__ void mma_part(v4f& acc, const v4i& w, const v4i& a, int part) {
    if constexpr (sizeof(T) == 2) acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(v8bf, w), __builtin_bit_cast(v8bf, a), acc, 0, 0, 0);
    else acc = __builtin_amdgcn_mfma_f32_16x16x4f32(__builtin_bit_cast(v4f, w)[part], __builtin_bit_cast(v4f, a)[part], acc, 0, 0, 0);
    asm volatile("" ::: "memory");
}

// four consecutive columns n .. n+3 (n a multiple of 4, all in one segment) of output row `row`
template <typename T>
__device__ __forceinline__ void store_cols(const NcLinear& g, int64_t out_off, int row, int n, v4f v) {
    int s = 0, base = 0;
#pragma unroll
    for (int i = 0; i < 3; i++)
        if (i + 1 < g.nseg && n >= g.seg[i].end) s = i + 1, base = g.seg[i].end;
    const NcSeg sg = g.seg[s];
    const int c = n - base;
    switch (sg.kind) {
        case NC_SEG_PLAIN: st4_f32((T*)sg.out + out_off + (int64_t)row * sg.ld + c, v); break;
        case NC_SEG_GELU:
            st4_f32((T*)sg.out + out_off + (int64_t)row * sg.ld + c,
                    v4f{gelu_tanh_f32(v[0]), gelu_tanh_f32(v[1]), gelu_tanh_f32(v[2]), gelu_tanh_f32(v[3])});
            break;
        case NC_SEG_GLU: {
            T* o = (T*)sg.out + out_off + (int64_t)row * sg.ld + (c >> 1);
            const float y0 = clamped_glu_f32(v[0], v[1], sg.p0), y1 = clamped_glu_f32(v[2], v[3], sg.p0);
            if constexpr (sizeof(T) == 2) *(uint32_t*)o = pack_bf16(y0, y1);
            else o[0] = y0, o[1] = y1;
            break;
        }
        case NC_SEG_SILU: st4_f32((T*)sg.out + out_off + (int64_t)row * sg.ld + c, v4f{silu_f32(v[0]), silu_f32(v[1]), silu_f32(v[2]), silu_f32(v[3])}); break;
        case NC_SEG_SWIGLU: {
            T* o = (T*)sg.out + out_off + (int64_t)row * sg.ld + (c >> 1);
            const float y0 = silu_f32(v[0]) * v[1], y1 = silu_f32(v[2]) * v[3];
            if constexpr (sizeof(T) == 2) *(uint32_t*)o = pack_bf16(y0, y1);
            else o[0] = y0, o[1] = y1;
            break;
        }
        case NC_SEG_SOFTPLUS: {
            const v4f z = v + *(const v4f*)(sg.bias + c);
            *(v4f*)((float*)sg.out + out_off + (int64_t)row * sg.ld + c) = v4f{softplus_f32(z[0]), softplus_f32(z[1]), softplus_f32(z[2]), softplus_f32(z[3])};
            break;
        }
        case NC_SEG_F32: *(v4f*)((float*)sg.out + out_off + (int64_t)row * sg.ld + c) = v; break;
        case NC_SEG_RESIDUAL: {
            v4f* o = (v4f*)((float*)sg.out + out_off + (int64_t)row * sg.ld + c);
            *o = *o + v;
            break;
        }
        default: {
            float* o = (float*)sg.out + out_off + (int64_t)row * sg.ld + c;
#pragma unroll
            for (int r = 0; r < 4; r++)
                if (n + r < g.N) {
                    const float z = v[r] * sg.p0;
                    o[r] = sg.p1 > 0.f ? sg.p1 * tanhf(z / sg.p1) : z;
                }
        }
    }
}

// eight consecutive columns n .. n+7 (column c of segment sg, a multiple of 8) of output row `row`
typedef uint32_t v4u_a8 __attribute__((ext_vector_type(4), aligned(8)));       // (rows of an output are 8-byte aligned, no more)
template <typename T>
__device__ __forceinline__ void st8_f32(T* p, v4f a, v4f b) {
    if constexpr (sizeof(T) == 2) *(v4u_a8*)p = v4u_a8{pack_bf16(a[0], a[1]), pack_bf16(a[2], a[3]), pack_bf16(b[0], b[1]), pack_bf16(b[2], b[3])};
    else *(v4f*)p = a, *(v4f*)(p + 4) = b;
}
template <typename T>
__device__ __forceinline__ void store_cols8(const NcSeg& sg, int N, int64_t out_off, int row, int n, int c, v4f a, v4f b) {
    const int64_t at = out_off + (int64_t)row * sg.ld;
    auto each = [](v4f v, auto f) { return v4f{f(v[0]), f(v[1]), f(v[2]), f(v[3])}; };
    switch (sg.kind) {
        case NC_SEG_PLAIN: st8_f32((T*)sg.out + at + c, a, b); break;
        case NC_SEG_GELU: st8_f32((T*)sg.out + at + c, each(a, gelu_tanh_f32), each(b, gelu_tanh_f32)); break;
        case NC_SEG_SILU: st8_f32((T*)sg.out + at + c, each(a, silu_f32), each(b, silu_f32)); break;
        case NC_SEG_GLU:
            st4_f32((T*)sg.out + at + (c >> 1), v4f{clamped_glu_f32(a[0], a[1], sg.p0), clamped_glu_f32(a[2], a[3], sg.p0), clamped_glu_f32(b[0], b[1], sg.p0),
                                                    clamped_glu_f32(b[2], b[3], sg.p0)});
            break;
        case NC_SEG_SWIGLU:
            st4_f32((T*)sg.out + at + (c >> 1), v4f{silu_f32(a[0]) * a[1], silu_f32(a[2]) * a[3], silu_f32(b[0]) * b[1], silu_f32(b[2]) * b[3]});
            break;
        case NC_SEG_SOFTPLUS:
            st8_f32((float*)sg.out + at + c, each(a + *(const v4f*)(sg.bias + c), softplus_f32), each(b + *(const v4f*)(sg.bias + c + 4), softplus_f32));
            break;
        case NC_SEG_F32: st8_f32((float*)sg.out + at + c, a, b); break;
        case NC_SEG_RESIDUAL: {
            float* o = (float*)sg.out + at + c;
            st8_f32(o, *(const v4f*)o + a, *(const v4f*)(o + 4) + b);
            break;
        }
        default: {
            float* o = (float*)sg.out + at + c;
#pragma unroll
            for (int r = 0; r < 8; r++)
                if (n + r < N) {
                    const float z = (r < 4 ? a[r & 3] : b[r & 3]) * sg.p0;
                    o[r] = sg.p1 > 0.f ? sg.p1 * tanhf(z / sg.p1) : z;
                }
        }
    }
}

// What a workgroup works on: which rows of A, which weight, where the output starts.
struct Span {
    int row0, rows;          // output rows [row0, row0 + rows)
    int64_t a_off, w_off, out_off;
};
__device__ __forceinline__ bool find_span(const NcLinear& g, int y, int batch, int tile_rows, Span& sp) {
    if (g.tiles) {
        if (y >= *g.n_tiles) return false;
        const int32_t* t = g.tiles + NC_TILE_WORDS * y;
        sp = Span{t[1], t[2], 0, (int64_t)t[0] * g.w_stride, 0};
        return true;
    }
    sp = Span{y * tile_rows, min(g.M - y * tile_rows, tile_rows), batch * g.a_stride, batch * g.w_stride, batch * g.out_stride};
    return sp.rows > 0;
}
__device__ __forceinline__ int64_t a_row(const NcLinear& g, int row) { return g.a_rows ? g.a_rows[row] / g.a_div : row; }

// ------------------------------------------------------------------------------------------------
// MT tiles of 16 rows x NB tiles of 16 weight rows per workgroup; wave w takes K-steps [its share] of 64 bytes.
// U K-steps are asked for at a time.  STREAM: the weight is loaded with the hint that nobody reads it again (see the tiled kernel).
template <typename T, int MT, int NB, int U, bool STREAM>
__global__ __launch_bounds__(256) void linear_few_kernel(NcLinear g, int split_bits) {
    __shared__ v4f red[4][MT * NB][64];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int split = (int)blockIdx.z & (g.splits - 1);
    Span sp;
    if (!find_span(g, blockIdx.y, (int)blockIdx.z >> split_bits, 16 * MT, sp)) return;
    const int n0 = blockIdx.x * 16 * NB, frow = lane & 15, piece = lane >> 4;
    const uint8_t* wp[NB];
    const uint8_t* ap[MT];
#pragma unroll
    for (int j = 0; j < NB; j++) {
        const int n = min(n0 + 16 * j + frow, g.N - 1);
        wp[j] = (const uint8_t*)((const T*)g.w + sp.w_off + (int64_t)n * g.ldw) + piece * 16;
    }
#pragma unroll
    for (int i = 0; i < MT; i++) {
        const int64_t m = a_row(g, sp.row0 + min(16 * i + frow, sp.rows - 1));
        ap[i] = (const uint8_t*)((const T*)g.a + sp.a_off + m * g.lda) + piece * 16;
    }
    v4f acc[MT][NB];
#pragma unroll
    for (int i = 0; i < MT; i++)
#pragma unroll
        for (int j = 0; j < NB; j++) acc[i][j] = v4f{0.f, 0.f, 0.f, 0.f};

    const int steps = g.K * (int)sizeof(T) / 64, share = 4 * split + wave, s0 = steps * share >> (split_bits + 2), s1 = steps * (share + 1) >> (split_bits + 2);
    auto step = [&](int s, auto unroll) {
        constexpr int N_ = decltype(unroll)::value;
        v4i wf[N_][NB], af[N_][MT];
#pragma unroll
        for (int u = 0; u < N_; u++) {
#pragma unroll
            for (int j = 0; j < NB; j++) {
                const v4i* const p = (const v4i*)(wp[j] + (int64_t)(s + u) * 64);
                wf[u][j] = STREAM ? __builtin_nontemporal_load(p) : *p;
            }
#pragma unroll
            for (int i = 0; i < MT; i++) af[u][i] = *(const v4i*)(ap[i] + (int64_t)(s + u) * 64);
        }
#pragma unroll
        for (int u = 0; u < N_; u++)
#pragma unroll
            for (int j = 0; j < NB; j++)
#pragma unroll
                for (int i = 0; i < MT; i++) acc[i][j] = Mma<T>::run(wf[u][j], af[u][i], acc[i][j]);
    };
    int s = s0;
    for (; s + U <= s1; s += U) step(s, std::integral_constant<int, U>{});
    if constexpr (U == 8)
        if (s + 4 <= s1) step(s, std::integral_constant<int, 4>{}), s += 4;
    for (; s < s1; s++) step(s, std::integral_constant<int, 1>{});

#pragma unroll
    for (int i = 0; i < MT; i++)
#pragma unroll
        for (int j = 0; j < NB; j++) red[wave][i * NB + j][lane] = acc[i][j];
    __syncthreads();
    for (int t = wave; t < MT * NB; t += 4) {
        const int i = t / NB, j = t % NB;
        const int m = 16 * i + frow, n = n0 + 16 * j + 4 * piece;
        if (m >= sp.rows || n >= g.N) continue;
        const v4f v = (red[0][t][lane] + red[1][t][lane]) + (red[2][t][lane] + red[3][t][lane]);
        if (g.partials) *(v4f*)(g.partials + ((int64_t)split * g.M + sp.row0 + m) * g.N + n) = v;
        else store_cols<T>(g, sp.out_off, sp.row0 + m, n, v);
    }
}

// ------------------------------------------------------------------------------------------------
// BM x BN outputs, WM x WN waves of 16-row, 16-column tiles, K-steps of 128 bytes.  Operand tiles go from global memory straight into LDS,
// 1 KB (8 rows x 128 bytes) per load instruction; chunk c (16 bytes) of row r is kept at slot c ^ SWZ(r), the permutation being applied
// on the global side, so that the fragment reads of 16 rows are free of bank conflicts.  A ring of STAGES: the loads of STAGES - 1 steps
// are in flight while one is multiplied.  Past the end of K the loads are issued all the same (into stages nobody reads any more), so
// that the barrier counts the same number of loads in every step.
//
// Up to 64 rows it is a stream of the weight; the few-rows kernel, with both operands in registers, read every activation from the L2 once per 32
// columns and waited for each batch of its loads (64 x 12352 x 2048: 32.5 us, 17 of them without the activations).  Its weights (FEW), as the
// few-rows kernel's, are loaded with the hint that nobody reads them again, so that they do not push out of the L2 what a step's other launches find
// there (us a step, without / with: Palilix, width 2048, 8 layers, 64 rows 1622 / 1498, Zodirax 16 rows 638 / 613, 1 row 560 / 499, its window append 7.8 /
// 6.1 and head 29.2 / 26.7; fp32, width 384, 2 rows 267 / 262, width 896, 8 rows 367 / 332, and 262 / 293 where one small model runs alone and its
// weights would stay in the 256 MB behind the L2).
//
// What bounds it on many rows: the loads.  A compute unit takes some 35 bytes per clock straight into LDS (4096^3, 128 x 256: 88 us of loads alone, 62 of
// products, 105 of both), which is why the widest tile that fills the chip is the one to take.  4096^3 140 -> 117 us, 1792 x 12352 x 2048
// 120 -> 95 (954 TFLOP/s; the library's own product 90-95), 1792 x 2048 x 4096 41 -> 33: most of it by the epilogue, which cost 15 us per
// round of tiles where its stores take 3.
#define TILE_SWZ(row) (((row) & 7) ^ (((row) >> 3) & 1))
#define TILE_OOB 0x80000000u       // a buffer offset past every descriptor: the load returns zeros
#define TILE_GROUP_M 8

// Tile order: workgroups are dealt to the 8 XCDs (each with an L2 of its own) in turn, so every XCD gets a contiguous run of the
// sequence, and the sequence walks bands of TILE_GROUP_M tile rows column by column.
__device__ __forceinline__ void tile_order(int id, int tiles_m, int tiles_n, int& tm, int& tn) {
    const int total = tiles_m * tiles_n, xcd = id & 7, slot = id >> 3;
    const int lin = xcd * (total >> 3) + min(xcd, total & 7) + slot;
    const int band = TILE_GROUP_M * tiles_n, first = (lin / band) * TILE_GROUP_M, rows = min(TILE_GROUP_M, tiles_m - first);
    tm = first + (lin % band) % rows, tn = (lin % band) / rows;
}

// Grouped rows: every XCD gets a contiguous run of (group, column tile, row tile of the group), the row tiles innermost, so that a weight
// tile is read by neighbours.  The launch covers the most tiles there can be; those past the actual count leave.
__device__ __forceinline__ bool group_tile_order(const NcLinear& g, int id, int tiles_n, int& tm, int& tn) {
    const int total = *g.n_tiles * tiles_n;
    if (id >= total) return false;
    const int xcd = id & 7, lin = xcd * (total >> 3) + min(xcd, total & 7) + (id >> 3);
    const int32_t* t = g.tiles + NC_TILE_WORDS * (lin / tiles_n);
    const int first = t[3], count = t[4], o = lin - first * tiles_n;
    tm = first + o % count, tn = o / count;
    return true;
}

template <bool STREAM>
__device__ __forceinline__ void tile_load(const void* base, uint32_t bytes, uint8_t* st, uint32_t lane_off, int k_off) {
    __builtin_amdgcn_raw_ptr_buffer_load_lds(__builtin_amdgcn_make_buffer_rsrc((void*)base, 0, bytes, 0x00020000), (lds_ptr_t)st, 16, lane_off, k_off, 0,
                                             STREAM ? 2 : 0);      // (bit 1: non-temporal)
}

template <typename T, int BM, int BN, int WM, int WN, int STAGES, bool FEW>
__global__ __launch_bounds__(64 * WM * WN) void linear_tiled_kernel(NcLinear g, int tiles_m, int tiles_n, int split_bits, uint32_t a_bytes) {
    constexpr int NW = WM * WN, WTM = BM / WM / 16, WTN = BN / WN / 16, STAGE = (BM + BN) * 128, A_P = BM / 8 / NW, W_P = BN / 8 / NW;
    // s_waitcnt vmcnt(loads of the STAGES - 2 youngest steps) lgkmcnt(0)
    constexpr int FLIGHT = (STAGES - 2) * (A_P + W_P), FIRST = FLIGHT + (A_P + W_P) / 2, WAIT = 0x0070 | (FLIGHT & 15) | ((FLIGHT >> 4) << 14);
    static_assert(A_P >= 1 && W_P >= 1 && NW % 2 == 0 && STAGES >= 3, "waves");
    extern __shared__ __align__(16) uint8_t lds[];
    int tm, tn;
    if (g.tiles) {
        if (!group_tile_order(g, blockIdx.x, tiles_n, tm, tn)) return;
    } else {
        tile_order(blockIdx.x, tiles_m, tiles_n, tm, tn);
    }
    Span sp;
    const int split = (int)blockIdx.y & (g.splits - 1);
    if (!find_span(g, tm, (int)blockIdx.y >> split_bits, BM, sp)) return;
    const int n0 = tn * BN;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wm = wave / WN, wn = wave % WN, frow = lane & 15, piece = lane >> 4;
    // staging: piece i of this wave is the 1 KB block (wave + NW i) of its operand's part of the stage; this lane's row inside an 8-row
    // block, and the global chunk that belongs in its LDS slot
    const int sub = lane >> 3, gch = (lane & 7) ^ sub ^ (wave & 1);
    // (the chunks of a lane's row that the halves of a step take; the same for both operands)
    const int rd_lo = frow * 128 + (((FEW ? piece : 2 * piece) ^ TILE_SWZ(frow)) << 4), rd_hi = frow * 128 + (((FEW ? 4 + piece : 2 * piece + 1) ^ TILE_SWZ(frow)) << 4);
    const uint32_t row_a = (uint32_t)(g.lda * sizeof(T)), row_w = (uint32_t)(g.ldw * sizeof(T));
    // this workgroup's share of the summed index, in half steps of 64 bytes, and the steps that hold it
    const int halves = g.K * (int)sizeof(T) / 64, h0 = halves * split >> split_bits, h1 = halves * (split + 1) >> split_bits;
    const int steps = halves / 2, k0 = h0 / 2, ksteps = (h1 + 1) / 2 - k0;
    const uint8_t* const A = (const uint8_t*)((const T*)g.a + sp.a_off) + k0 * 128;
    const uint8_t* const W = (const uint8_t*)((const T*)g.w + sp.w_off + (int64_t)n0 * g.ldw) + k0 * 128;
    a_bytes -= k0 * 128;
    const uint32_t w_bytes = (uint32_t)(min(g.N - n0, BN) - 1) * row_w + (uint32_t)(steps - k0) * 128;
    uint32_t vo_a[A_P], vo_w[W_P];
#pragma unroll
    for (int i = 0; i < A_P; i++) {
        const int r = 8 * (wave + NW * i) + sub;
        vo_a[i] = r < sp.rows ? (uint32_t)a_row(g, sp.row0 + r) * row_a + gch * 16 : TILE_OOB;
    }
#pragma unroll
    for (int i = 0; i < W_P; i++) {
        const int r = 8 * (wave + NW * i) + sub;
        vo_w[i] = n0 + r < g.N ? (uint32_t)r * row_w + gch * 16 : TILE_OOB;
    }
    // FEW: the sum in four chains, a quarter of the share each: the same additions in the same order as in linear_few_kernel, so that a row's
    // result does not depend on which of the kernels a batch of up to 64 rows took.  (The number of shares is the caller's.)
    constexpr int CHAINS = FEW ? 4 : 1;
    v4f acc[CHAINS][WTM][WTN];
#pragma unroll
    for (int c = 0; c < CHAINS; c++)
#pragma unroll
        for (int i = 0; i < WTM; i++)
#pragma unroll
            for (int j = 0; j < WTN; j++) acc[c][i][j] = v4f{0.f, 0.f, 0.f, 0.f};
    // A step has two halves (the low and the high 64 bytes of K of a lane's 128-byte row).  While the low half multiplies, the fragments of the
    // high half are read; then every wave has read all of its stage, the waves meet, and while the high half multiplies, the low fragments of
    // the next step are read: neither the barrier nor an LDS read is ever waited for with the matrix cores idle.  The stage that was read is
    // free from the meeting on: the loads of step kt + STAGES go there, spread over the products.
    auto meet = [&]() {
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_waitcnt(WAIT);    // the operands of the next step have landed, this step's fragments are read (this wave's share; the barrier says everybody's)
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
    };
    constexpr int LOADS = A_P + W_P, EARLY = LOADS / 2, PRODUCTS = WTM * WTN, READS = WTM + WTN;
    auto load = [&](int i, int k_off, uint8_t* st) {
        if (i < A_P) tile_load<false>(A, a_bytes, st + i * NW * 1024, vo_a[i], k_off);
        else tile_load<FEW>(W, w_bytes, st + BM * 128 + (i - A_P) * NW * 1024, vo_w[i - A_P], k_off);
    };
    // 16-row tiles of this wave that hold rows at all: the last tile of a group of rows is seldom full
    const int valid = __builtin_amdgcn_readfirstlane((sp.rows - wm * (BM / WM) + 15) >> 4);
    enum { ALL, NONE, SOME, READ };           // which products a half step has; READ: none, but the fragments of the next half are read
    v4i al[WTM], ah[WTM], wl[WTN], wh[WTN];
    // half a step: products of (w, a), between them the reads of the other half's fragments and the loads [L0, L1) of a later step
    auto half = [&](const v4i (&a)[WTM], const v4i (&w)[WTN], v4i (&na)[WTM], v4i (&nw)[WTN], const uint8_t* pa, const uint8_t* pw, int rd, auto l0, auto l1, int k_off,
                    uint8_t* st, auto rows, auto chain) __attribute__((always_inline)) {
        constexpr int ROWS = decltype(rows)::value, CHAIN = decltype(chain)::value, L0 = decltype(l0)::value, NL = decltype(l1)::value - L0;
#pragma unroll
        for (int j = 0; j < WTN; j++)
#pragma unroll
            for (int p = 0; p < MMA_PARTS<T>; p++)
#pragma unroll
                for (int i = 0; i < WTM; i++) {
                    const int n = j * WTM + i;
                    if (p == 0) {
#pragma unroll
                        for (int r = 0; r < READS; r++)
                            if (ROWS != NONE && r * PRODUCTS / READS / 2 == n) {
                                if (r == 0) nw[0] = *(const v4i*)(pw + rd);
                                else if (r <= WTM) na[r - 1] = *(const v4i*)(pa + (r - 1) * 2048 + rd);
                                else nw[r - WTM] = *(const v4i*)(pw + (r - WTM) * 2048 + rd);
                            }
#pragma unroll
                        for (int r = 0; r < NL; r++)
                            if ((2 * r + 1) * PRODUCTS / (2 * NL) == n) load(L0 + r, k_off, st);
                    }
                    if (ROWS == ALL || (ROWS == SOME && i < valid)) mma_part<T>(acc[CHAIN][i][j], w[j], a[i], p);
                }
    };
    const int wa = wm * (BM / WM) * 128, ww = BM * 128 + wn * (BN / WN) * 128;
#pragma unroll
    for (int i = 0; i < STAGES; i++)
#pragma unroll
        for (int r = 0; r < (i < STAGES - 1 ? LOADS : EARLY); r++) load(r, i < ksteps ? i * 128 : 0, lds + i * STAGE + wave * 1024);
    __builtin_amdgcn_s_waitcnt(0x0F70 | (FIRST & 15) | ((FIRST >> 4) << 14));
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    wl[0] = *(const v4i*)(lds + ww + rd_lo);
#pragma unroll
    for (int i = 0; i < WTM; i++) al[i] = *(const v4i*)(lds + wa + i * 2048 + rd_lo);
#pragma unroll
    for (int j = 1; j < WTN; j++) wl[j] = *(const v4i*)(lds + ww + j * 2048 + rd_lo);
    int kt = 0, cur = 0, prev = (STAGES - 1) * STAGE;     // the step; byte offsets of the stage being read and of the one before it
    auto low = [&](auto rows, auto chain) __attribute__((always_inline)) {
        const int k1 = kt + STAGES - 1 < ksteps ? (kt + STAGES - 1) * 128 : 0;
        half(al, wl, ah, wh, lds + cur + wa, lds + cur + ww, rd_hi, std::integral_constant<int, EARLY>{}, std::integral_constant<int, LOADS>{}, k1,
             lds + prev + wave * 1024, rows, chain);
        meet();
    };
    auto high = [&](auto rows, auto chain) __attribute__((always_inline)) {
        const int next = cur + STAGE == STAGES * STAGE ? 0 : cur + STAGE, k2 = kt + STAGES < ksteps ? (kt + STAGES) * 128 : 0;
        half(ah, wh, al, wl, lds + next + wa, lds + next + ww, rd_lo, std::integral_constant<int, 0>{}, std::integral_constant<int, EARLY>{}, k2,
             lds + cur + wave * 1024, rows, chain);
        prev = cur, cur = next, kt++;
    };
    // half steps [from, to) into one chain; a half outside the share is read and not multiplied
    auto run = [&](int from, int to, auto rows, auto chain) __attribute__((always_inline)) {
        if (from >= to) return;
        if (from & 1) high(rows, chain);
        while (2 * (k0 + kt) + 1 < to) low(rows, chain), high(rows, chain);
        if (to & 1) low(rows, chain);
    };
    using std::integral_constant;
    if constexpr (FEW) {
        const integral_constant<int, SOME> rows;
        const int e1 = halves * (4 * split + 1) >> (split_bits + 2), e2 = halves * (4 * split + 2) >> (split_bits + 2), e3 = halves * (4 * split + 3) >> (split_bits + 2);
        if (h0 & 1) low(integral_constant<int, READ>{}, integral_constant<int, 0>{});
        run(h0, e1, rows, integral_constant<int, 0>{});
        run(e1, e2, rows, integral_constant<int, 1>{});
        run(e2, e3, rows, integral_constant<int, 2>{});
        run(e3, h1, rows, integral_constant<int, 3>{});
#pragma unroll
        for (int i = 0; i < WTM; i++)
#pragma unroll
            for (int j = 0; j < WTN; j++) acc[0][i][j] = (acc[0][i][j] + acc[1][i][j]) + (acc[2][i][j] + acc[3][i][j]);
    } else {
        if (h0 & 1) low(integral_constant<int, READ>{}, integral_constant<int, 0>{});
        if (valid >= WTM) run(h0, h1, integral_constant<int, ALL>{}, integral_constant<int, 0>{});
        else if (valid <= 0) run(h0, h1, integral_constant<int, NONE>{}, integral_constant<int, 0>{});
        else run(h0, h1, integral_constant<int, SOME>{}, integral_constant<int, 0>{});
    }
    // the loads past the end of K are still landing: they must be done before the workgroup gives its LDS back
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(0x0F70);
    __builtin_amdgcn_s_barrier();
    // out through LDS, each wave its own part: a lane then has eight neighbouring columns of a row, so a store is whole lines, and the code of
    // the epilogues is there once (inlined per accumulator it was 16 times as long, and took longer than its stores)
    constexpr int ROW = BN / WN + 4;                          // floats: rows shifted by four banks
    constexpr int FIT = STAGES * STAGE / (NW * 64 * ROW), SUBS = FIT >= WTM ? WTM : FIT >= 4 ? 4 : FIT >= 2 ? 2 : 1;      // 16-row tiles at a time
    static_assert(FIT >= 1 && WTM % SUBS == 0, "output staging");
    float* const own = (float*)lds + wave * 16 * SUBS * ROW;
    constexpr int CHUNKS = BN / WN / 8, ROWS_AT_ONCE = 64 / CHUNKS;
    const int c = 8 * (lane % CHUNKS), n = n0 + wn * (BN / WN) + c;
    NcSeg sg = g.seg[0];
    int base = 0;
#pragma unroll
    for (int i = 1; i < 4; i++)
        if (i < g.nseg && n >= g.seg[i - 1].end) sg = g.seg[i], base = g.seg[i - 1].end;
    if (g.partials) sg = NcSeg{g.N, NC_SEG_F32, g.partials + (int64_t)split * g.M * g.N, g.N, 0.f, 0.f, nullptr}, base = 0;
#pragma unroll
    for (int i0 = 0; i0 < WTM; i0 += SUBS) {
#pragma unroll
        for (int i = 0; i < SUBS; i++)
#pragma unroll
            for (int j = 0; j < WTN; j++) *(v4f*)(own + (16 * i + frow) * ROW + 16 * j + 4 * piece) = acc[0][i0 + i][j];
#pragma unroll 1
        for (int r = lane / CHUNKS; r < 16 * SUBS; r += ROWS_AT_ONCE) {
            const int m = wm * (BM / WM) + 16 * i0 + r;
            if (m >= sp.rows || n >= g.N) break;
            const float* v = own + r * ROW + c;
            store_cols8<T>(sg, g.N, sp.out_off, sp.row0 + m, n, n - base, *(const v4f*)v, *(const v4f*)(v + 4));
        }
    }
}

// ------------------------------------------------------------------------------------------------
// 256 x 256 outputs of many bf16 rows, eight waves of 64 x 128 (4 x 2): a K-step of 128 bytes asks the LDS for 196 KB of fragments and 64 KB of operands beside
// 2048 clocks of products, where the 128 x 256 tiles ask for 131 + 48 KB beside 1024: those run at the rate of the LDS, these at that of the products.
// The rows go through a ring of three stages and are read a step ahead into registers of their own, the weight through two stages, read one group of
// products ahead (160 KB in all; three stages of both do not fit).  What is left of the tiles behind whole rounds over the compute units is cut into halves
// of 256 x 128 where those fit one round: 1792 rows are 7 tiles of 256, and rounds of whole tiles alone would lose what they gain.  Same products in the same
// order as in linear_tiled_kernel.  us, 128 x 256 tiles / these: 1792 x 21760 x 4096 291 / 258, x 22528 290 / 260, x 8192 106 / 92, 1792 x 12544 x 2048 91 / 81, x
// 7936 58 / 51, 4096^3 112 / 99.5 (1.38 PFLOP/s; a large product of the library's 1.23).
struct BigFrag {
    v4i lo, hi;
};
template <int NS>
__device__ __forceinline__ void big_tile(const NcLinear& g, int m0, int n0, uint32_t a_bytes, uint8_t* lds) {
    constexpr int A_ST = 256 * 128, W_ST = 32 * NS * 128, W_P = NS / 2, HP = 4, WCOLS = 16 * NS;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), wm = wave >> 1, wn = wave & 1, frow = lane & 15, piece = lane >> 4;
    const int sub = lane >> 3, gch = (lane & 7) ^ sub ^ (wave & 1);
    const int rd_lo = frow * 128 + ((2 * piece ^ TILE_SWZ(frow)) << 4), rd_hi = frow * 128 + (((2 * piece + 1) ^ TILE_SWZ(frow)) << 4);
    const uint32_t row_a = (uint32_t)g.lda * 2, row_w = (uint32_t)g.ldw * 2;
    const int ksteps = g.K / 64;
    const uint8_t* const A = (const uint8_t*)g.a;
    const uint8_t* const W = (const uint8_t*)((const bf16_t*)g.w + (int64_t)n0 * g.ldw);
    const uint32_t w_bytes = (uint32_t)(min(g.N - n0, 32 * NS) - 1) * row_w + (uint32_t)g.K * 2;
    // piece i of this wave is the 1 KB block (wave + 8 i) of its operand's stage
    uint32_t vo_a[HP], vo_w[W_P];
#pragma unroll
    for (int i = 0; i < HP; i++) {
        const int r = m0 + 8 * wave + 64 * i + sub;
        vo_a[i] = r < g.M ? (uint32_t)r * row_a + gch * 16 : TILE_OOB;
    }
#pragma unroll
    for (int i = 0; i < W_P; i++) {
        const int r = 8 * wave + 64 * i + sub;
        vo_w[i] = n0 + r < g.N ? (uint32_t)r * row_w + gch * 16 : TILE_OOB;
    }
    v4f acc[4][NS];
#pragma unroll
    for (int i = 0; i < 4; i++)
#pragma unroll
        for (int j = 0; j < NS; j++) acc[i][j] = v4f{0.f, 0.f, 0.f, 0.f};
    uint8_t* const ring_w = lds + 3 * A_ST;
    auto load_a = [&](int r, int t, int at) {
        if (t < ksteps) tile_load<false>(A, a_bytes, lds + at + wave * 1024 + r * 8192, vo_a[r], t * 128);
    };
    auto load_w = [&](int r, int t, int buf) {
        if (t < ksteps) tile_load<false>(W, w_bytes, ring_w + buf * W_ST + wave * 1024 + r * 8192, vo_w[r], t * 128);
    };
    auto frag = [&](const uint8_t* p) { return BigFrag{*(const v4i*)(p + rd_lo), *(const v4i*)(p + rd_hi)}; };
    auto meet = [&](bool in_flight) {
        asm volatile("" ::: "memory");
        if (in_flight) __builtin_amdgcn_s_waitcnt(0x0070 | HP);      // (the rows of the step three ahead may still be on their way)
        else __builtin_amdgcn_s_waitcnt(0x0070);
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
    };
    BigFrag held[2][4];
    int at0 = 0, at1 = A_ST, at2 = 2 * A_ST;        // stages of the rows of this step, the next and the one after
    auto step = [&](int t, auto parity) __attribute__((always_inline)) {
        constexpr int P = decltype(parity)::value, Q = 1 - P, LOADS = W_P + HP, PRODUCTS = 8 * NS;
        const uint8_t* const ws = ring_w + P * W_ST + wn * WCOLS * 128;
        const uint8_t* const as = lds + at1 + wm * 64 * 128;
        BigFrag wf[2];
        wf[0] = frag(ws);
#pragma unroll
        for (int j = 0; j < NS; j++) {
            if (j + 1 < NS) wf[(j + 1) & 1] = frag(ws + (j + 1) * 2048);
#pragma unroll
            for (int i = 0; i < 4; i++)
                if (i * NS / 4 == j) held[Q][i] = frag(as + i * 2048);
#pragma unroll
            for (int n = 0; n < 8; n++) {
                const int i = n & 3;
#pragma unroll
                for (int r = 0; r < LOADS; r++)
                    if (r * PRODUCTS / LOADS == 8 * j + n) {
                        if (r < W_P) load_w(r, t + 1, Q);
                        else load_a(r - W_P, t + 3, at0);
                    }
                mma_part<bf16_t>(acc[i][j], n < 4 ? wf[j & 1].lo : wf[j & 1].hi, n < 4 ? held[P][i].lo : held[P][i].hi, 0);
            }
        }
        meet(t + 3 < ksteps);
        const int first = at0;
        at0 = at1, at1 = at2, at2 = first;
    };
#pragma unroll
    for (int r = 0; r < W_P; r++) load_w(r, 0, 0);
#pragma unroll
    for (int r = 0; r < 3 * HP; r++) load_a(r % HP, r / HP, r / HP * A_ST);
    asm volatile("" ::: "memory");
    if (ksteps > 2) __builtin_amdgcn_s_waitcnt(0x0070 | (2 * HP));   // the first step's operands
    else __builtin_amdgcn_s_waitcnt(0x0070);
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
#pragma unroll
    for (int i = 0; i < 4; i++) held[0][i] = frag(lds + wm * 64 * 128 + i * 2048);
    meet(ksteps > 2);
    int kt = 0;
    for (; kt + 1 < ksteps; kt += 2) {
        step(kt, std::integral_constant<int, 0>{});
        step(kt + 1, std::integral_constant<int, 1>{});
    }
    if (kt < ksteps) step(kt, std::integral_constant<int, 0>{});
    // out through LDS, each wave its own part (see linear_tiled_kernel)
    constexpr int ROW = WCOLS + 4, SUBS = 2, CHUNKS = WCOLS / 8, ROWS_AT_ONCE = 64 / CHUNKS;
    static_assert(8 * 16 * SUBS * ROW * 4 <= 3 * A_ST + 2 * W_ST, "output staging");
    float* const own = (float*)lds + wave * 16 * SUBS * ROW;
    const int c = 8 * (lane % CHUNKS), n = n0 + wn * WCOLS + c;
    NcSeg sg = g.seg[0];
    int base = 0;
#pragma unroll
    for (int i = 1; i < 4; i++)
        if (i < g.nseg && n >= g.seg[i - 1].end) sg = g.seg[i], base = g.seg[i - 1].end;
    if (g.partials) sg = NcSeg{g.N, NC_SEG_F32, g.partials, g.N, 0.f, 0.f, nullptr}, base = 0;
#pragma unroll
    for (int i0 = 0; i0 < 4; i0 += SUBS) {
#pragma unroll
        for (int i = 0; i < SUBS; i++)
#pragma unroll
            for (int j = 0; j < NS; j++) *(v4f*)(own + (16 * i + frow) * ROW + 16 * j + 4 * piece) = acc[i0 + i][j];
#pragma unroll 1
        for (int r = lane / CHUNKS; r < 16 * SUBS; r += ROWS_AT_ONCE) {
            const int m = m0 + wm * 64 + 16 * i0 + r;
            if (m >= g.M || n >= g.N) break;
            const float* v = own + r * ROW + c;
            store_cols8<bf16_t>(sg, g.N, 0, m, n, n - base, *(const v4f*)v, *(const v4f*)(v + 4));
        }
    }
}
// `full` workgroups with a whole tile, the rest with half a one
__global__ __launch_bounds__(512) void linear_big_kernel(NcLinear g, int tiles_m, int full, uint32_t a_bytes) {
    extern __shared__ __align__(16) uint8_t lds[];
    // every XCD gets a contiguous run of the tiles, and of the halves behind them; a band of TILE_GROUP_M tile rows column by column
    const bool half = (int)blockIdx.x >= full;
    const int id = half ? (int)blockIdx.x - full : (int)blockIdx.x, total = half ? (int)gridDim.x - full : full;
    const int lin = (id & 7) * (total >> 3) + min(id & 7, total & 7) + (id >> 3), tile = half ? full + lin / 2 : lin;
    const int tiles_n = (g.N + 255) / 256, band = TILE_GROUP_M * tiles_n, first = tile / band * TILE_GROUP_M, rows = min(TILE_GROUP_M, tiles_m - first);
    const int m0 = (first + tile % band % rows) * 256, n0 = tile % band / rows * 256 + (half ? lin % 2 * 128 : 0);
    if (n0 >= g.N) return;
    if (half) big_tile<4>(g, m0, n0, a_bytes, lds);
    else big_tile<8>(g, m0, n0, a_bytes, lds);
}

int reserve_dynamic_lds(const void* fn, int bytes, std::atomic<uint64_t>& done) {
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev > 63) dev = 0;
    if (done.load(std::memory_order_relaxed) >> dev & 1) return 0;
    if (hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, bytes) != hipSuccess) NC_FAIL(-2, "linear: %d bytes of LDS refused", bytes);
    done.fetch_or(1ull << dev, std::memory_order_relaxed);
    return 0;
}

int check_linear(const NcLinear& l, int dtype) {
    NC_CHECK_ARG(l.a && l.w && l.nseg <= 4, "linear: null operand");
    NC_CHECK_ARG(l.M > 0 && l.N > 0 && l.K > 0 && l.K % 32 == 0 && l.batch >= 1, "linear: bad shape M=%d N=%d K=%d batch=%d", l.M, l.N, l.K, l.batch);
    NC_CHECK_ARG(dtype == 0 || dtype == 1, "linear: dtype must be 0 (bfloat16) or 1 (float)");
    NC_CHECK_ARG(l.lda % (dtype ? 4 : 8) == 0 && l.ldw % (dtype ? 4 : 8) == 0 && l.ldw >= l.K && ((uintptr_t)l.a & 15) == 0 && ((uintptr_t)l.w & 15) == 0, "linear: operands must be 16-byte aligned");
    NC_CHECK_ARG(l.splits >= 1 && (l.splits & (l.splits - 1)) == 0 && l.splits <= 64 && (int64_t)l.K * l.splits < 1 << 29 && (l.splits == 1 || l.partials), "linear: %d shares of %d", l.splits, l.K);
    NC_CHECK_ARG(!l.partials || (l.batch == 1 && !l.tiles && l.N % 16 == 0), "linear: partial sums of %d columns", l.N);
    for (int i = 0; i < l.nseg; i++)
        NC_CHECK_ARG(l.seg[i].kind == NC_SEG_LOGITS || (l.seg[i].end % 16 == 0 && l.seg[i].ld % 4 == 0), "linear: segments must end at multiples of 16 columns");
    return 0;
}

// what the tiles' 32-bit offsets reach: the rows of A of a launch (a gathered row index is below M / a_div), the weight rows of a tile
constexpr int64_t TILE_BYTES = 1ll << 31;
int64_t linear_a_bytes(const NcLinear& l, int es) { return (((l.a_rows ? (l.M + l.a_div - 1) / l.a_div : l.M) - 1) * l.lda + l.K) * es; }

template <typename T, int MT, int NB, int U = 4, bool STREAM = true>
int launch_few(const NcLinear& l, int ytiles, hipStream_t s) {
    hipLaunchKernelGGL((linear_few_kernel<T, MT, NB, U, STREAM>), dim3((l.N + 16 * NB - 1) / (16 * NB), ytiles, l.batch * l.splits), dim3(256), 0, s, l, __builtin_ctz(l.splits));
    NC_CHECK_LAUNCH("linear_few");
    return 0;
}
template <typename T>
int launch_few_t(const NcLinear& l, hipStream_t s) {
    // One workgroup per compute unit or two wait for their loads, which eight steps at a time halve (bf16, 4 rows, K = 2048, N = 2048 6.6 -> 6.0 us,
    // K = 4096 10.3 -> 9.2, six experts of 2048 x 2048 and back a step of 255 -> 244; from 16384 columns on 9.5 -> 10.3, and no fp32 launch gains).
    const int64_t cols = (int64_t)l.N * (l.tiles ? l.max_tiles : l.batch * l.splits);
    const bool ahead = sizeof(T) == 2 && cols <= 12288;
    // (experts' weights without the hint: bf16, experts of 1024, width 2048, 16 rows a step of 609 us with it, 581 without; width 1024, 8 rows 303 / 294)
    if (l.tiles) return ahead ? launch_few<T, 1, 1, 8, false>(l, l.max_tiles, s) : launch_few<T, 1, 1, 4, false>(l, l.max_tiles, s);
    if (l.M <= 16) return ahead ? launch_few<T, 1, 1, 8>(l, 1, s) : launch_few<T, 1, 1>(l, 1, s);
    return l.M <= 32 ? launch_few<T, 2, 2>(l, 1, s) : launch_few<T, 4, 2>(l, (l.M + 63) / 64, s);
}
template <typename T, int BM, int BN, int WM, int WN, int STAGES, bool FEW>
int launch_tiled(const NcLinear& l, hipStream_t s) {
    static std::atomic<uint64_t> done{0};
    constexpr int LDS = (BM + BN) * 128 * STAGES;
    const void* fn = (const void*)linear_tiled_kernel<T, BM, BN, WM, WN, STAGES, FEW>;
    if (int rc = reserve_dynamic_lds(fn, LDS, done)) return rc;
    const int tm = l.tiles ? l.max_tiles : (l.M + BM - 1) / BM, tn = (l.N + BN - 1) / BN;
    const int64_t a_bytes = linear_a_bytes(l, sizeof(T));
    NC_CHECK_ARG(a_bytes < TILE_BYTES && BN * l.ldw * (int64_t)sizeof(T) < TILE_BYTES, "linear: operand past 2 GiB");
    hipLaunchKernelGGL((linear_tiled_kernel<T, BM, BN, WM, WN, STAGES, FEW>), dim3(tm * tn, l.batch * l.splits), dim3(64 * WM * WN), LDS, s, l, tm, tn,
                       __builtin_ctz(l.splits), (uint32_t)a_bytes);
    NC_CHECK_LAUNCH("linear_tiled");
    return 0;
}
// whole tiles of 256 x 256 of a launch; the others are cut in two where the halves fit half a round
int big_full_tiles(int64_t tiles) {
    const int cus = nc_cu_count(), rest = (int)(tiles % cus);
    return (int)(2 * rest <= cus ? tiles - rest : tiles);
}
int launch_big(const NcLinear& l, hipStream_t s) {
    static std::atomic<uint64_t> done{0};
    constexpr int LDS = 5 * 256 * 128;
    if (int rc = reserve_dynamic_lds((const void*)linear_big_kernel, LDS, done)) return rc;
    const int64_t a_bytes = linear_a_bytes(l, 2);
    NC_CHECK_ARG(!l.tiles && !l.a_rows && l.batch == 1 && l.splits == 1 && l.K % 64 == 0, "linear: not a product of the 256 x 256 tiles");
    NC_CHECK_ARG(a_bytes < TILE_BYTES && 256 * l.ldw * 2 < TILE_BYTES, "linear: operand past 2 GiB");
    const int tm = (l.M + 255) / 256, tn = (l.N + 255) / 256, tiles = tm * tn, full = big_full_tiles(tiles);
    hipLaunchKernelGGL(linear_big_kernel, dim3(full + 2 * (tiles - full)), dim3(512), LDS, s, l, tm, full, (uint32_t)a_bytes);
    NC_CHECK_LAUNCH("linear_big");
    return 0;
}
// tile shapes: 1 = 64 x 128 (two workgroups per compute unit), 2 = 128 x 256, 3 = 128 x 128, 4 = 64 x 64 (two), 5 = 32 x 64 (two),
// 6 = 32 x 32 (two)
constexpr int BIG_SHAPE = 7;                  // bf16: 256 x 256 and halves of it
constexpr int SHAPES = 6, SHAPE_ROWS[SHAPES + 1] = {0, 64, 128, 128, 64, 32, 32}, SHAPE_COLS[SHAPES + 1] = {0, 128, 256, 128, 64, 64, 32};
template <typename T>
int launch_tiled_shape(const NcLinear& l, int shape, hipStream_t s) {
    if (l.few) {
        if (shape == 4) return launch_tiled<T, 64, 64, 2, 2, 4, true>(l, s);
        if (shape == 5) return launch_tiled<T, 32, 64, 1, 4, 6, true>(l, s);
        if (shape == 6) return launch_tiled<T, 32, 32, 2, 2, 8, true>(l, s);
    }
    switch (shape) {
        case 1: return launch_tiled<T, 64, 128, 2, 2, 3, false>(l, s);
        case 2: return launch_tiled<T, 128, 256, 2, 4, 3, false>(l, s);
        case 3: return launch_tiled<T, 128, 128, 2, 4, 3, false>(l, s);
        case 4: return launch_tiled<T, 64, 64, 2, 2, 4, false>(l, s);
        case 5: return launch_tiled<T, 32, 64, 1, 4, 6, false>(l, s);
        default: return launch_tiled<T, 32, 32, 2, 2, 8, false>(l, s);
    }
}

// us at K = 2048 (bf16) or 1024 (fp32), tenths: what a launch takes per round of tiles over the compute units, and beside the rounds.  A tile of
// bf16 costs its loads, one of fp32 its products, where narrow tiles lose less.
constexpr int ROUND_COST[2][SHAPES + 1] = {{0, 125, 270, 185, 90, 60, 50}, {0, 320, 1200, 620, 175, 100, 70}}, BASE_COST[2][SHAPES + 1] = {{0, 10, 0, 0, 10, 25, 25}, {0, 30, 0, 0, 30, 40, 40}};
constexpr int BIG_COST = 500, BIG_HALF_COST = 295;       // ... of a round of 256 x 256 tiles, and of one of halves of them
int64_t shape_tiles(const NcLinear& l, int shape) {
    return (int64_t)((l.M + SHAPE_ROWS[shape] - 1) / SHAPE_ROWS[shape]) * ((l.N + SHAPE_COLS[shape] - 1) / SHAPE_COLS[shape]) * l.batch * l.splits;
}
// The shape with the least rounds times cost.  Few rows are a stream of the weight, which the narrow tiles with the most loads in flight read
// best.  Measured, us, 64x128 / 128x256 / 128x128 / 64x64 / 32x64 / 32x32: bf16, K = 2048: 1792 x 2048 21 / 25 / 17.6, 1792 x 12352
// 118 / 94 / 116, 700 x 4096 22 / 27 / 17.5 / 23 / 30, 333 x 2048 13 / 25 / 16 / 9.9 / 12, 80 x 2048 13 / 24 / 16 / 8.9 / 7.8 / 7.3; up to 64
// rows, the last three and linear_few_kernel: 64 x 4096 13.7 / 10.9 / 8.7, 17.4, 64 x 12288 15.7 / 18.9 / 20.2, 32, 16 x 12288 14.5 / 12.3 / 13.3,
// 16.5, 16 x 32768 29 / 26 / 30, 41.  fp32, K = 1024: 1792 x 4096 127 / 124 / 128 / 122 / 136, 333 x 4096 37 / 120 / 64 / 38 / 35, 80 x 4096
// 35 / 92 / 50 / 22 / 15, 64 x 4096 22.4 / 15.0 / 11.1, 21.5.  Over sums of 128 to 8192 and 80 to 1792 rows the choice is 0.6 % (bf16) and 1.1 % (fp32)
// above the best tile on average, with costs that leave the length of the sum out.
int choose_shape(const NcLinear& l, int dtype) {
    const int cus = nc_cu_count();
    int shape = 0;
    int64_t best = 0;
    for (int i = SHAPES; i >= (l.M <= NC_FEW_ROWS ? 4 : 1); i--) {
        const int64_t cost = (shape_tiles(l, i) + cus - 1) / cus * ROUND_COST[dtype][i] + BASE_COST[dtype][i];
        if (!shape || cost < best) best = cost, shape = i;
    }
    if (!dtype && !l.tiles && !l.a_rows && l.batch == 1 && l.splits == 1 && l.M > NC_FEW_ROWS) {
        const int64_t tiles = (int64_t)((l.M + 255) / 256) * ((l.N + 255) / 256), full = big_full_tiles(tiles);
        if ((full + cus - 1) / cus * BIG_COST + (full < tiles ? BIG_HALF_COST : 0) < best) shape = BIG_SHAPE;
    }
    return shape;
}

double linear_units(const NcLinear& l, int dtype, bool few) {
    // the few-rows kernel is a stream of the weight (bytes), the tiled one a product (flops)
    return few ? (double)l.batch * l.N * l.K * (dtype ? 4 : 2) : 2.0 * l.batch * l.M * l.N * l.K;
}
int64_t linear_tag(const NcLinear& l) { return ((int64_t)l.N << 32) | (uint32_t)l.K; }
}  // namespace

int nc_linear_splits(int dtype, int M, int N, int K) {
    int splits = 1;
    if (M <= NC_FEW_ROWS) {
        const int nb = M <= 16 ? 16 : 32, wgs = (N + nb - 1) / nb;
        while (splits < 8 && wgs * splits < 384 && K / (splits * 2) >= 256) splits *= 2;
    } else if (dtype && K % 64 == 0 && K >= 512) {
        // fp32: four shares, whatever the number of rows above NC_FEW_ROWS, so that a row's sums do not depend on how many of them came with it.  (The chosen rows of a prompt
        // go through the last output matrix by themselves: their number counts there, not the prompt's length.)  Few tiles fill the chip with
        // them (333 x 1024 x 5120: 152 us in one piece, 45 in four), many lose nothing (a prompt of 1792 tokens, in one piece / two / four: width
        // 2048 6675 / 6637 / 6414 us, 1024 3307 / 3319 / 3349, 640 1425 / 1376 / 1363).  bf16 sums of many rows stay one chain.
        splits = 4;
    }
    return splits;
}

int nc_launch_linear_few(int dtype, const NcLinear& l, hipStream_t s, int cls) {
    if (int rc = check_linear(l, dtype)) return rc;
    NC_CHECK_ARG(!l.tiles || l.tile_rows <= NC_GROUP_TILE_FEW, "linear: group tiles of %d rows", l.tile_rows);
    NcProfScope prof(cls, linear_units(l, dtype, true), s, linear_tag(l));
    return dtype ? launch_few_t<float>(l, s) : launch_few_t<bf16_t>(l, s);
}

int nc_launch_linear_tiled(int dtype, const NcLinear& l, hipStream_t s, int cls, int shape) {
    if (int rc = check_linear(l, dtype)) return rc;
    NC_CHECK_ARG(l.K % 64 == 0 && l.splits <= l.K / 64 && shape >= 0 && (shape <= SHAPES || (shape == BIG_SHAPE && !dtype)), "linear: the tiled kernel takes whole K-steps");
    NcProfScope prof(cls, linear_units(l, dtype, !l.tiles ? l.M <= NC_FEW_ROWS : l.tile_rows <= 32), s, linear_tag(l));
    if (!shape) shape = !l.tiles ? choose_shape(l, dtype) : l.tile_rows <= 32 ? 5 : l.tile_rows <= 64 ? (l.few ? 4 : 1) : 2;
    if (shape == BIG_SHAPE) return launch_big(l, s);
    // (the wider shapes have one chain: they are no place for a group whose sums are those of few rows)
    if (l.tiles) NC_CHECK_ARG(l.tile_rows <= SHAPE_ROWS[shape] && (!l.few || shape >= 4), "linear: group tiles of %d rows", l.tile_rows);
    return dtype ? launch_tiled_shape<float>(l, shape, s) : launch_tiled_shape<bf16_t>(l, shape, s);
}

// The few-rows kernel or a tile: same sums, so only time decides.  In the few-rows kernel four waves share the summed index, which pays where its
// workgroups of 16 columns are few per compute unit or the whole weight is short; its price is that every workgroup reads every row from the L2.
// us, few-rows kernel / best tile, by columns (times batch and shares):
//   bf16, 4 rows     K = 512: 8192 4.7 / 5.2, 32768 9.6 / 9.2      1024: 6144 6.1 / 6.0, 32768 16.0 / 14.8     2048: 4096 7.0 / 8.1, 8192 9.6 / 9.1
//   bf16, 16 rows    K = 512: 4096 4.1 / 5.0, 16384 7.8 / 6.1      1024: 4096 5.2 / 5.9, 6144 7.2 / 6.1       4096: 2048 12.1 / 11.8, 8192 21 / 13.5
//   bf16, 32 rows    K = 128: 8192 3.4 / 4.0                       512: 8192 5.9 / 5.2, 16384 8.7 / 6.2       1024: 2048 8.0 / 6.1
//   fp32, 4 rows     K = 512: 8192 7.9 / 7.3, 16384 12.1 / 9.4     1024: 4096 10.0 / 10.1, 8128 11.2 / 12.5 between a step's other launches
//   fp32, 16 rows    K = 512: 4096 7.0 / 7.1, 16384 14 / 9.6       2048: 4096 17.9 / 16.5, 8192 24 / 17       32 rows, 256: 8192 6.5 / 6.8
bool few_is_faster(const NcLinear& l, int dtype) {
    const int64_t cols = (int64_t)l.N * l.batch * l.splits, k = l.K / l.splits, weight = cols * k;
    if (l.M <= 16 && (cols <= 4096 || weight <= (l.M > 8 && (dtype ? cols > 8192 : k > 512) ? 4 << 20 : 8 << 20))) return true;
    return l.M <= 32 && k <= 512 && weight <= 4 << 20;
}
int nc_launch_linear(int dtype, const NcLinear& l, hipStream_t s) {
    // (the few-rows kernel has no limit on the size of its operands)
    const int es = dtype ? 4 : 2;
    if (l.M <= NC_FEW_ROWS && (linear_a_bytes(l, es) >= TILE_BYTES || 64 * l.ldw * es >= TILE_BYTES)) return nc_launch_linear_few(dtype, l, s);
    return l.K % 64 || few_is_faster(l, dtype) ? nc_launch_linear_few(dtype, l, s) : nc_launch_linear_tiled(dtype, l, s);
}
