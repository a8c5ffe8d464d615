// FP8 (e4m3 x e4m3) scaled GEMM for gfx950:  out[M,N] = bf16((A[M,K] . B[N,K]^T in fp32) * inv_a * inv_b)
// Replaces torch._scaled_mm as called at nanochat/fp8.py:143-153 (row-major A, K-contiguous B, fp32
// accumulation, bf16 output).  B may be several weight matrices stacked along N, each with its own
// tensorwise inv-scale (the reference's c_q/c_k/c_v are three Float8Linear modules).
//
// The kernels use v_mfma_f32_16x16x128_f8f6f4 (the full-rate fp8 MFMA of CDNA4): a lane supplies 32
// consecutive K bytes of row (lane & 15) from K-block (lane >> 4).  Operands are issued as (B, A) so a
// lane ends up holding four consecutive output columns of one output row, which packs into one 8-byte
// bf16 store.
//
//   gemm_bl_kernel      M large (prefill, isolated Float8Linear): BMxBNx128 tiles, double-buffered swizzled LDS fed
//                       through two register stages of buffer loads (for the 128x128 tile the fills and loads are
//                       placed between the MFMA groups by hand), bf16 epilogue staged through LDS.
//   gemm_dl_kernel      256x256x128 tiles whose operands go from global memory straight into LDS (no staging registers,
//   gemm_dlp_kernel     no LDS fill instructions); the second is the persistent form for shapes of several rounds of tiles.
//   gemm_tile_kernel    the same tiling with plain global loads (64-bit addressing) for operands past 2 GiB.
//   M <= 128 (decode) is weight-bandwidth bound and handled by gemm_decode_kernel in nc_gemm_decode.hip.
#include <type_traits>
#include "nc_common.h"
#include "nc_kernels.h"
#include "nc_meeting.h"
#include "nc_rope.h"

// 16-byte chunk c of LDS row r (128-byte rows) is kept at chunk slot c ^ NC_SWZ(r) by the buffer-load kernels.  Measured on
// gfx950: with this mapping a fragment read (16 rows per 16 lanes, ds_read_b128) runs at the rate of a lane-linear read
// (~215 B/clk/CU); XOR with (r & 7) alone, or with (r >> 1) & 7, runs at 60% of that.
#define NC_SWZ(row) (((row) & 7) ^ (((row) >> 3) & 1))
#define MFMA_F8(acc, b, a) __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4((b), (a), (acc), 0, 0, 0, 0, 0, 0)

struct EpilogueArgs {
    const float* inv_a;
    const float* inv_b;
    NcGemmSegs segs;
    void* out;
    int out_kind;            // 0 bf16, 1 fp32 softcap, 2 bf16 relu(v)^2 with the amax of the result published to out_amax, 4 its e4m3 (q8_epilogue)
    float softcap;
    int ldc;
    uint32_t* out_amax;
    // out_kind 4
    NcMeeting meeting;
    bf16_t* left;            // [M, N]: where a workgroup that leaves the meeting puts its tile
    float* inv_out;
};
// out_kind 5: the q|k|v linear of a prompt, whose rows go on to rotary, norm and cache (rope_epilogue)
struct RopeArgs {
    NcRopeSrc src;
    NcRopeDst dst;
};
struct NoRope {};

// relu(bf16(v))^2, to be rounded to bf16 by the caller's pack: the two eager ops of nanochat/gpt.py:139 on a bf16 tensor
__device__ __forceinline__ float relu2_of(float v) {
    const float h = relu_keep_nan(rbf(v));
    return h * h;
}
// largest of eight non-negative bf16 values in a 16-byte vector, the first `count` of them
__device__ __forceinline__ float max_bf16x8(const uint4& v, int count) {
    const uint32_t w[4] = {v.x, v.y, v.z, v.w};
    uint32_t m = 0;
#pragma unroll
    for (int r = 0; r < 8; r++) {
        const uint32_t b = (w[r >> 1] >> ((r & 1) * 16)) & 0xffffu;
        if (r < count) m = b > m ? b : m;             // non-negative bf16: integer order is value order
    }
    return __uint_as_float(m << 16);
}

__device__ __forceinline__ float seg_scale(const EpilogueArgs& e, int col) {
    int s = 0;
#pragma unroll
    for (int i = 0; i < 3; i++)
        if (i + 1 < e.segs.nseg && col >= e.segs.end[i]) s = i + 1;
    return e.inv_b[s];
}

// four consecutive columns n..n+3 of output row m
__device__ __forceinline__ void store4(const EpilogueArgs& e, float inv_a, v4f acc, int m, int n, int M, int N) {
    if (m >= M || n >= N) return;
    const float inv_b = seg_scale(e, n);
    float v[4];
#pragma unroll
    for (int r = 0; r < 4; r++) v[r] = (acc[r] * inv_a) * inv_b;
    if (e.out_kind == 0) {
        bf16_t* o = (bf16_t*)e.out + (size_t)m * e.ldc + n;
        if (n + 3 < N) {
            uint2 p = make_uint2(pack_bf16(v[0], v[1]), pack_bf16(v[2], v[3]));
            *(uint2*)o = p;
        } else {
            for (int r = 0; r < 4 && n + r < N; r++) o[r] = f32_to_bf16(v[r]);
        }
    } else {
        float* o = (float*)e.out + (size_t)m * e.ldc + n;
        for (int r = 0; r < 4 && n + r < N; r++) o[r] = e.softcap * tanhf(rbf(v[r]) / e.softcap);
    }
}

// Tile order.  Workgroups are dealt to the 8 XCDs round robin (workgroup id % 8) and each XCD has its own 4 MB L2,
// so (1) every XCD gets a contiguous run of the tile sequence, and (2) the sequence walks the tile grid in bands of
// GROUP_M tile rows, column by column inside a band: the ~64 tiles an XCD works on at one time then cover about
// GROUP_M rows x 8 columns and share GROUP_M A panels and 8 B panels (a few MB) instead of streaming all of B
// past one A panel.
#define NC_GROUP_M 8
__device__ __forceinline__ void tile_coords(int wg, int tiles_m, int tiles_n, int& tm, int& tn) {
    const int ntiles = tiles_m * tiles_n;
    const int per = ntiles / 8, rem = ntiles % 8;
    const int xcd = wg % 8, local = wg / 8;
    const int seq = xcd * per + (xcd < rem ? xcd : rem) + local;
    const int band_tiles = NC_GROUP_M * tiles_n;
    const int band = seq / band_tiles, in_band = seq % band_tiles;
    const int rows_here = min(NC_GROUP_M, tiles_m - band * NC_GROUP_M);
    tm = band * NC_GROUP_M + in_band % rows_here;
    tn = in_band / rows_here;
}

// ------------------------------------------------------------------------------------------------
// Tile kernel.  LDS rows are 128 bytes (one K step); 16-byte chunk c of row r lives at chunk slot
// c ^ (r & 7), which makes both the row-major fills and the per-lane fragment reads conflict free.
template <int BM, int BN>
__global__ __launch_bounds__(256) void gemm_tile_kernel(const uint8_t* __restrict__ A, const uint8_t* __restrict__ B,
                                                        EpilogueArgs ep, int M, int N, int K, int tiles_m, int tiles_n) {
    constexpr int WTM = BM / 32, WTN = BN / 32;          // 16x16 tiles per wave along M and N
    constexpr int A_CH = BM * 8 / 256, B_CH = BN * 8 / 256;
    extern __shared__ __align__(16) uint8_t lds[];
    auto tile_a = [&](int buf) -> uint8_t* { return lds + buf * (BM + BN) * 128; };
    auto tile_b = [&](int buf) -> uint8_t* { return lds + buf * (BM + BN) * 128 + BM * 128; };

    int tm, tn;
    tile_coords(blockIdx.x, tiles_m, tiles_n, tm, tn);
    const int m0 = tm * BM, n0 = tn * BN;

    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int wm = wave >> 1, wn = wave & 1;
    const int frow = lane & 15, kb = lane >> 4;

    v4f acc[WTM][WTN];
#pragma unroll
    for (int i = 0; i < WTM; i++)
#pragma unroll
        for (int j = 0; j < WTN; j++) acc[i][j] = v4f{0.f, 0.f, 0.f, 0.f};

    uint4 ra[A_CH], rb[B_CH];
    auto load_regs = [&](int kt) {
#pragma unroll
        for (int c = 0; c < A_CH; c++) {
            const int id = tid + c * 256, row = id >> 3, ch = id & 7;
            const int gr = m0 + row, gk = kt * 128 + ch * 16;
            ra[c] = (gr < M && gk < K) ? *(const uint4*)(A + (size_t)gr * K + gk) : make_uint4(0, 0, 0, 0);
        }
#pragma unroll
        for (int c = 0; c < B_CH; c++) {
            const int id = tid + c * 256, row = id >> 3, ch = id & 7;
            const int gr = n0 + row, gk = kt * 128 + ch * 16;
            rb[c] = (gr < N && gk < K) ? *(const uint4*)(B + (size_t)gr * K + gk) : make_uint4(0, 0, 0, 0);
        }
    };
    auto store_lds = [&](int buf) {
#pragma unroll
        for (int c = 0; c < A_CH; c++) {
            const int id = tid + c * 256, row = id >> 3, ch = id & 7;
            *(uint4*)(tile_a(buf) + row * 128 + ((ch ^ (row & 7)) << 4)) = ra[c];
        }
#pragma unroll
        for (int c = 0; c < B_CH; c++) {
            const int id = tid + c * 256, row = id >> 3, ch = id & 7;
            *(uint4*)(tile_b(buf) + row * 128 + ((ch ^ (row & 7)) << 4)) = rb[c];
        }
    };
    auto read_frag = [&](const uint8_t* base, int row) -> v8i {
        const int sw = row & 7;
        const uint4 lo = *(const uint4*)(base + row * 128 + (((2 * kb) ^ sw) << 4));
        const uint4 hi = *(const uint4*)(base + row * 128 + (((2 * kb + 1) ^ sw) << 4));
        v8i f;
        f[0] = lo.x, f[1] = lo.y, f[2] = lo.z, f[3] = lo.w, f[4] = hi.x, f[5] = hi.y, f[6] = hi.z, f[7] = hi.w;
        return f;
    };

    const int ksteps = (K + 127) / 128;
    load_regs(0);
    store_lds(0);
    __syncthreads();
    for (int kt = 0; kt < ksteps; kt++) {
        const int buf = kt & 1;
        if (kt + 1 < ksteps) load_regs(kt + 1);
        v8i af[WTM];
#pragma unroll
        for (int i = 0; i < WTM; i++) af[i] = read_frag(tile_a(buf), wm * (BM / 2) + i * 16 + frow);
#pragma unroll
        for (int j = 0; j < WTN; j++) {
            const v8i bf = read_frag(tile_b(buf), wn * (BN / 2) + j * 16 + frow);
#pragma unroll
            for (int i = 0; i < WTM; i++) acc[i][j] = MFMA_F8(acc[i][j], bf, af[i]);
        }
        if (kt + 1 < ksteps) store_lds(buf ^ 1);
        __syncthreads();
    }

    const float inv_a = *ep.inv_a;
#pragma unroll
    for (int i = 0; i < WTM; i++)
#pragma unroll
        for (int j = 0; j < WTN; j++) {
            const int m = m0 + wm * (BM / 2) + i * 16 + frow;
            const int n = n0 + wn * (BN / 2) + j * 16 + 4 * kb;
            store4(ep, inv_a, acc[i][j], m, n, M, N);
        }
}

// Epilogue of the buffer-load kernels: scale, convert and store one workgroup tile.
template <int BM, int BN, int WGM, int WGN, int OUT_KIND>
__device__ __forceinline__ void bl_epilogue(v4f (&acc)[BM / WGM / 16][BN / WGN / 16], uint8_t* lds, const EpilogueArgs& ep, float inv_a,
                                            const float (&sc)[4], int m0, int n0, int M, int N) {
    constexpr int WTM = BM / WGM / 16, WTN = BN / WGN / 16;
    constexpr int STAGE = (BM + BN) * 128;
    const int lane = threadIdx.x & 63, wave = threadIdx.x / 64;
    const int wm = wave / WGN, wn = wave % WGN;
    const int frow = lane & 15, kb = lane >> 4;
    if (OUT_KIND != 1) {
        // bf16 output goes through LDS so that every store instruction writes whole 128-byte lines: each wave parks its
        // (BM/WGM) x (BN/WGN) block in its own LDS region (16-byte chunk c of row r at chunk c ^ (r & 7)), then reads it
        // back with one row segment per group of LPR lanes and stores 16 bytes per lane.
        constexpr int WROWS = BM / WGM, WCOLS = BN / WGN, ROWB = WCOLS * 2, LPR = ROWB / 16, RPI = 64 / LPR;
        static_assert(LPR % 8 == 0 && LPR <= 64 && WGM * WGN * WROWS * ROWB <= 2 * STAGE, "epilogue staging");
        constexpr bool relu2 = OUT_KIND == 2;
        float am = 0.f;
        __syncthreads();                                       // every wave is done with the operand tiles
        uint8_t* reg = lds + wave * WROWS * ROWB;
#pragma unroll
        for (int j = 0; j < WTN; j++) {
            const int n = n0 + wn * WCOLS + j * 16 + 4 * kb;
            float inv_b = sc[0];
#pragma unroll
            for (int i = 0; i < 3; i++)
                if (i + 1 < ep.segs.nseg && n >= ep.segs.end[i]) inv_b = sc[i + 1];
            const int chunk = 2 * j + (kb >> 1);
#pragma unroll
            for (int i = 0; i < WTM; i++) {
                const int row = i * 16 + frow;
                const v4f a4 = acc[i][j];
                float o4[4];
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    o4[r] = (a4[r] * inv_a) * inv_b;
                    if (relu2) o4[r] = relu2_of(o4[r]);
                }
                const uint2 pk = make_uint2(pack_bf16_hw(o4[0], o4[1]), pack_bf16_hw(o4[2], o4[3]));
                *(uint2*)(reg + row * ROWB + ((chunk ^ (row & 7)) << 4) + (kb & 1) * 8) = pk;
            }
        }
        // the region is private to the wave: its own LDS writes only have to land before its reads
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_s_waitcnt(0xc07f);                    // lgkmcnt(0)
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        const bool vec16 = (ep.ldc % 8 == 0) && (((uintptr_t)ep.out & 15) == 0);
        const int lrow_e = lane / LPR, c = lane % LPR;
        const int n = n0 + wn * WCOLS + c * 8;
#pragma unroll
        for (int it = 0; it < WROWS / RPI; it++) {
            const int row = it * RPI + lrow_e;
            const int m = m0 + wm * WROWS + row;
            const uint4 v = *(const uint4*)(reg + row * ROWB + ((c ^ (row & 7)) << 4));
            if (m >= M || n >= N) continue;
            if (relu2) am = amax_join(am, max_bf16x8(v, N - n));
            bf16_t* o = (bf16_t*)ep.out + (size_t)m * ep.ldc + n;
            if (n + 8 <= N) {
                if (vec16) __builtin_nontemporal_store(v4i{(int)v.x, (int)v.y, (int)v.z, (int)v.w}, (v4i*)o);
                else {
                    *(uint2*)o = make_uint2(v.x, v.y);
                    *(uint2*)(o + 4) = make_uint2(v.z, v.w);
                }
            } else {
                const uint32_t w[4] = {v.x, v.y, v.z, v.w};
                for (int r = 0; r < 8 && n + r < N; r++) o[r] = (bf16_t)(w[r >> 1] >> ((r & 1) * 16));
            }
        }
        if (relu2) {
            // one publication per workgroup: the waves meet once more and the first thread joins their maxima
            __shared__ float wave_am[WGM * WGN];
            am = wave_amax(am);
            if (lane == 0) wave_am[wave] = am;
            __syncthreads();
            if (threadIdx.x == 0) {
                float t = wave_am[0];
#pragma unroll
                for (int w = 1; w < WGM * WGN; w++) t = amax_join(t, wave_am[w]);
                amax_publish(ep.out_amax, t);
            }
        }
    } else {
#pragma unroll
        for (int j = 0; j < WTN; j++) {
            const int n = n0 + wn * (BN / WGN) + j * 16 + 4 * kb;
            float inv_b = sc[0];
#pragma unroll
            for (int i = 0; i < 3; i++)
                if (i + 1 < ep.segs.nseg && n >= ep.segs.end[i]) inv_b = sc[i + 1];
#pragma unroll
            for (int i = 0; i < WTM; i++) {
                const int m = m0 + wm * (BM / WGM) + i * 16 + frow;
                if (m >= M || n >= N) continue;
                float* o = (float*)ep.out + (size_t)m * ep.ldc + n;
                for (int r = 0; r < 4 && n + r < N; r++)
                    o[r] = ep.softcap * tanhf(rbf((acc[i][j][r] * inv_a) * inv_b) / ep.softcap);
            }
        }
    }
    // no barrier and no wait here: the kernel ends, and a wave may retire with its stores still on their way, which frees the
    // CU for the next workgroup while the output drains
}

// ------------------------------------------------------------------------------------------------
// relu^2 as the next linear reads it: every workgroup holds its tile until the launch knows the amax of the whole result (nc_meeting.h), and the tile
// leaves as e4m3.  The launch of one round that writes bf16 ends in 24 MB of stores (1792 x 6656) that a conversion launch reads back: 26.7 + 8.4 us;
// this way 29.3 us.  Same roundings (bf16, then e4m3 of that) and the same bits.  One tile per workgroup, all workgroups on the chip at once
// (nc_gemm_relu2_e4m3_kernel).  N is a multiple of 16.
template <int BM, int BN>
__device__ __forceinline__ void q8_convert_left(const EpilogueArgs& ep, int wg, float amax, float scale, int M, int N, int tiles_m, int tiles_n) {
    int tm, tn;
    tile_coords(wg, tiles_m, tiles_n, tm, tn);
    for (int id = threadIdx.x; id < BM * (BN / 16); id += blockDim.x) {
        const int m = tm * BM + id / (BN / 16), n = tn * BN + id % (BN / 16) * 16;
        if (m >= M || n >= N) continue;
        const uint4* src = (const uint4*)(ep.left + (size_t)m * N + n);
        *(uint4*)((uint8_t*)ep.out + (size_t)m * ep.ldc + n) = e4m3_of_bf16x16(src[0], src[1], scale);
    }
    if (wg == 0 && threadIdx.x == 0) meeting_result(amax, scale, ep.inv_out, ep.out_amax);
}
template <int BM, int BN, int WGM, int WGN>
__device__ __forceinline__ void q8_epilogue(v4f (&acc)[BM / WGM / 16][BN / WGN / 16], uint8_t* lds, const EpilogueArgs& ep, float inv_a, const float (&sc)[4],
                                            int m0, int n0, int M, int N, int tiles_m, int tiles_n) {
    constexpr int WTM = BM / WGM / 16, WTN = BN / WGN / 16, WROWS = BM / WGM, WCOLS = BN / WGN, PITCH = WCOLS + 16, PIECES = WROWS * (WCOLS / 16);
    static_assert(PIECES % 64 == 0 && WGM * WGN * WROWS * PITCH <= 2 * (BM + BN) * 128, "epilogue staging");
    const int lane = threadIdx.x & 63, wave = threadIdx.x / 64, wm = wave / WGN, wn = wave % WGN, frow = lane & 15, kb = lane >> 4;
    uint2 held[WTM][WTN];                                      // the bf16 values, four neighbouring columns each
    float am = 0.f;
#pragma unroll
    for (int j = 0; j < WTN; j++) {
        const int n = n0 + wn * WCOLS + j * 16 + 4 * kb;
        float inv_b = sc[0];
#pragma unroll
        for (int i = 0; i < 3; i++)
            if (i + 1 < ep.segs.nseg && n >= ep.segs.end[i]) inv_b = sc[i + 1];
#pragma unroll
        for (int i = 0; i < WTM; i++) {
            const v4f a4 = acc[i][j];
            float o4[4];
#pragma unroll
            for (int r = 0; r < 4; r++) o4[r] = relu2_of((a4[r] * inv_a) * inv_b);
            const uint2 pk = make_uint2(pack_bf16_hw(o4[0], o4[1]), pack_bf16_hw(o4[2], o4[3]));
            held[i][j] = pk;
            if (m0 + wm * WROWS + i * 16 + frow < M && n < N)
                am = amax_fold(amax_fold(amax_fold(amax_fold(am, bf16_lo(pk.x)), bf16_hi(pk.x)), bf16_lo(pk.y)), bf16_hi(pk.y));
        }
    }
    float amax;
    bool left;
    const bool here = meeting<WGM * WGN>(ep.meeting, gridDim.x, blockIdx.x, am, amax, left, [] {}, [&] {
#pragma unroll
        for (int j = 0; j < WTN; j++)
#pragma unroll
            for (int i = 0; i < WTM; i++) {
                const int m = m0 + wm * WROWS + i * 16 + frow, n = n0 + wn * WCOLS + j * 16 + 4 * kb;
                if (m < M && n < N) *(uint2*)(ep.left + (size_t)m * N + n) = held[i][j];
            }
    });
    if (!here) return;
    const float scale = scale_from_amax(amax);
    if (blockIdx.x == 0 && threadIdx.x == 0) meeting_result(amax, scale, ep.inv_out, ep.out_amax);
    // (every wave is done with the operand tiles: the meeting has barriers)
    uint8_t* reg = lds + wave * WROWS * PITCH;
#pragma unroll
    for (int j = 0; j < WTN; j++)
#pragma unroll
        for (int i = 0; i < WTM; i++) *(uint32_t*)(reg + (i * 16 + frow) * PITCH + j * 16 + 4 * kb) = e4m3_of_bf16x4(held[i][j].x, held[i][j].y, scale);
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_s_waitcnt(0xc07f);                        // lgkmcnt(0): the region is private to the wave
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
    for (int it = 0; it < PIECES / 64; it++) {
        const int id = it * 64 + lane, row = id / (WCOLS / 16), c = id % (WCOLS / 16);
        const int m = m0 + wm * WROWS + row, n = n0 + wn * WCOLS + c * 16;
        if (m < M && n < N) *(uint4*)((uint8_t*)ep.out + (size_t)m * ep.ldc + n) = *(const uint4*)(reg + row * PITCH + c * 16);
    }
    if (left) meeting_take(ep.meeting, gridDim.x, [&](int w) { q8_convert_left<BM, BN>(ep, w, amax, scale, M, N, tiles_m, tiles_n); });
}

// ------------------------------------------------------------------------------------------------
// The q|k|v linear of a prompt with what comes behind it: a tile is 128 columns wide, which is one head, so rotary, QK-norm, gain, value embedding and the
// append to the cache are done on the tile as it leaves through LDS, and the 18 MB of bf16 rows (1792 x 4992) that a launch of its own read back are
// never written.  Same roundings as the two launches, same bits.  1792 x 4992 x 1664 in a d26 prompt: 26.6 us against 20.0 and 14.2.
template <int BM, int WGM, int WGN>
__device__ __forceinline__ void rope_epilogue(v4f (&acc)[BM / WGM / 16][128 / WGN / 16], uint8_t* lds, const EpilogueArgs& ep, const RopeArgs& rope, float inv_a,
                                              const float (&sc)[4], int m0, int n0, int M) {
    constexpr int WTM = BM / WGM / 16, WTN = 128 / WGN / 16, WROWS = BM / WGM, WCOLS = 128 / WGN, PITCH = 272, NT = 64 * WGM * WGN, ROUNDS = BM / (NT / 8);
    static_assert(BM % (NT / 8) == 0 && BM * PITCH <= 2 * (BM + 128) * 128, "epilogue staging");
    const int lane = threadIdx.x & 63, wave = threadIdx.x / 64, wm = wave / WGN, wn = wave % WGN, frow = lane & 15, kb = lane >> 4;
    const int hh = n0 / 128, part = threadIdx.x & 7;
    // (every segment is whole heads: one scale for the tile)
    float inv_b = sc[0];
#pragma unroll
    for (int i = 0; i < 3; i++)
        if (i + 1 < ep.segs.nseg && n0 >= ep.segs.end[i]) inv_b = sc[i + 1];
    __syncthreads();                                       // every wave is done with the operand tiles
#pragma unroll
    for (int j = 0; j < WTN; j++)
#pragma unroll
        for (int i = 0; i < WTM; i++) {
            const v4f a4 = acc[i][j];
            *(uint2*)(lds + (wm * WROWS + i * 16 + frow) * PITCH + (wn * WCOLS + j * 16 + 4 * kb) * 2) =
                make_uint2(pack_bf16_hw((a4[0] * inv_a) * inv_b, (a4[1] * inv_a) * inv_b), pack_bf16_hw((a4[2] * inv_a) * inv_b, (a4[3] * inv_a) * inv_b));
        }
    // (asked for here, where the accumulators' registers are free)
    RopeVecRaw raw[ROUNDS];
#pragma unroll
    for (int it = 0; it < ROUNDS; it++) rope_vec_load(rope.src, rope.dst, min(m0 + it * (NT / 8) + (int)(threadIdx.x >> 3), M - 1), hh, part, raw[it]);
    __syncthreads();
#pragma unroll
    for (int it = 0; it < ROUNDS; it++) {
        const int row = it * (NT / 8) + (threadIdx.x >> 3), token = m0 + row;
        const uint8_t* src = lds + row * PITCH + part * 16;
        rope_vec_finish(rope.src, rope.dst, raw[it], *(const uint4*)src, *(const uint4*)(src + 128), min(token, M - 1), hh, part, token < M);
    }
}

// ------------------------------------------------------------------------------------------------
// Buffer-load tile kernel: the same tiling, LDS layout and MFMA mapping as gemm_tile_kernel, with a main
// loop free of branches.  Global reads go through buffer descriptors, whose hardware range check returns
// zeros for rows past M / N and for the K tail, so no load sits under a lane mask and the loads of K-steps
// k+2 and k+3 stay in flight (two register stages) while step k is computed; the waits the compiler places
// then count outstanding loads instead of draining them.  Waves form a WGM x WGN grid over the BM x BN tile.
#define NC_BUF_OOB 0x80000000u
// Accumulate in place: tying the result to the accumulator operand keeps every 16x16 tile in the same four
// accumulation registers for the whole K loop (the builtin lets the register allocator pick a different result
// tuple, which it repairs with dozens of register copies per K-step once the loop is unrolled).
// A_FMT is the format of the activation-side operand (the instruction's second source, `blgp`): 0 = e4m3, 1 = e5m2, the
// gradient format of the backward GEMMs (nanochat/fp8.py:165).  The weight-side operand is always e4m3.
template <int A_FMT = 0>
__device__ __forceinline__ void mfma_f8_acc(v4f& acc, const v8i& b, const v8i& a) {
    if (A_FMT == 0) asm("v_mfma_f32_16x16x128_f8f6f4 %0, %1, %2, %0" : "+a"(acc) : "v"(b), "v"(a));
    else asm("v_mfma_f32_16x16x128_f8f6f4 %0, %1, %2, %0 blgp:1" : "+a"(acc) : "v"(b), "v"(a));
}
// Same, pinned in program order against every memory operation: used where the LDS fills and global loads of the
// next steps are placed between groups of MFMAs by hand, so that the LDS, load and matrix pipes work at the same time.
template <int A_FMT = 0>
__device__ __forceinline__ void mfma_f8_acc_ordered(v4f& acc, const v8i& b, const v8i& a) {
    if (A_FMT == 0) asm volatile("v_mfma_f32_16x16x128_f8f6f4 %0, %1, %2, %0" : "+a"(acc) : "v"(b), "v"(a) : "memory");
    else asm volatile("v_mfma_f32_16x16x128_f8f6f4 %0, %1, %2, %0 blgp:1" : "+a"(acc) : "v"(b), "v"(a) : "memory");
}
template <int BM, int BN, int WGM, int WGN, int OUT_KIND, bool INTERLEAVE = false, int A_FMT = 0>
__global__ __launch_bounds__(64 * WGM * WGN) void gemm_bl_kernel(const uint8_t* __restrict__ A, const uint8_t* __restrict__ B,
                                                                 EpilogueArgs ep, int M, int N, int K, int tiles_m, int tiles_n) {
    constexpr int NT = 64 * WGM * WGN;
    constexpr int WTM = BM / WGM / 16, WTN = BN / WGN / 16;     // 16x16 tiles per wave along M and N
    constexpr int A_CH = BM * 8 / NT, B_CH = BN * 8 / NT;       // 16-byte pieces per thread and K-step
    constexpr int PASS_ROWS = NT / 8;                           // tile rows covered by one piece of every thread
    constexpr int STAGE = (BM + BN) * 128;
    static_assert(PASS_ROWS % 16 == 0 && BM % (16 * WGM) == 0 && BN % (16 * WGN) == 0, "tile shape");
    extern __shared__ __align__(16) uint8_t lds[];

    int tm, tn;
    tile_coords(blockIdx.x, tiles_m, tiles_n, tm, tn);
    const int m0 = tm * BM, n0 = tn * BN;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid / 64;
    const int wm = wave / WGN, wn = wave % WGN;
    const int frow = lane & 15, kb = lane >> 4;

    const __amdgpu_buffer_rsrc_t desc_a = __builtin_amdgcn_make_buffer_rsrc((void*)A, 0, M * K, 0x00020000);
    const __amdgpu_buffer_rsrc_t desc_b = __builtin_amdgcn_make_buffer_rsrc((void*)B, 0, N * K, 0x00020000);

    // this thread's pieces: chunk `ch` of rows lrow, lrow + PASS_ROWS, ...
    const int lrow = tid >> 3, ch = tid & 7;
    uint32_t avo[A_CH], bvo[B_CH];
#pragma unroll
    for (int c = 0; c < A_CH; c++) {
        const int r = m0 + lrow + c * PASS_ROWS;
        avo[c] = r < M ? (uint32_t)r * (uint32_t)K + ch * 16 : NC_BUF_OOB;
    }
#pragma unroll
    for (int c = 0; c < B_CH; c++) {
        const int r = n0 + lrow + c * PASS_ROWS;
        bvo[c] = r < N ? (uint32_t)r * (uint32_t)K + ch * 16 : NC_BUF_OOB;
    }
    const int lw = lrow * 128 + ((ch ^ NC_SWZ(lrow)) << 4);                 // LDS fill offset of piece 0 (PASS_ROWS keeps the swizzle)
    const int sw = NC_SWZ(frow);
    const int rd_lo = frow * 128 + (((2 * kb) ^ sw) << 4), rd_hi = frow * 128 + (((2 * kb + 1) ^ sw) << 4);
    const int a_rd = wm * (BM / WGM) * 128, b_rd = BM * 128 + wn * (BN / WGN) * 128;

    const int ksteps = (K + 127) / 128, kfull = K / 128;
    const bool ch_in_tail = ch * 16 >= K % 128;                            // only looked at for the partial last step

    v4f acc[WTM][WTN];
#pragma unroll
    for (int i = 0; i < WTM; i++)
#pragma unroll
        for (int j = 0; j < WTN; j++) acc[i][j] = v4f{0.f, 0.f, 0.f, 0.f};

    v4i ra[2][A_CH], rb[2][B_CH];
#define BL_LOAD(SLOT, T)                                                                                  \
    do {                                                                                                  \
        const int t__ = (T);                                                                              \
        const bool cut__ = t__ >= ksteps || (t__ == kfull && ch_in_tail);                                 \
        _Pragma("unroll") for (int c = 0; c < A_CH; c++)                                                  \
            ra[SLOT][c] = __builtin_amdgcn_raw_buffer_load_b128(desc_a, cut__ ? NC_BUF_OOB : avo[c], t__ * 128, 0); \
        _Pragma("unroll") for (int c = 0; c < B_CH; c++)                                                  \
            rb[SLOT][c] = __builtin_amdgcn_raw_buffer_load_b128(desc_b, cut__ ? NC_BUF_OOB : bvo[c], t__ * 128, 0); \
    } while (0)
#define BL_FILL(SLOT, BUF)                                                                                \
    do {                                                                                                  \
        uint8_t* st__ = lds + (BUF) * STAGE + lw;                                                         \
        _Pragma("unroll") for (int c = 0; c < A_CH; c++) *(v4i*)(st__ + c * PASS_ROWS * 128) = ra[SLOT][c]; \
        _Pragma("unroll") for (int c = 0; c < B_CH; c++) *(v4i*)(st__ + BM * 128 + c * PASS_ROWS * 128) = rb[SLOT][c]; \
    } while (0)
    auto frag = [&](const uint8_t* base) -> v8i {
        const v4i lo = *(const v4i*)(base + rd_lo);
        const v4i hi = *(const v4i*)(base + rd_hi);
        return v8i{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
    };
    auto compute = [&](int buf) {
        const uint8_t* st = lds + buf * STAGE;
        v8i af[WTM];
#pragma unroll
        for (int i = 0; i < WTM; i++) af[i] = frag(st + a_rd + i * 2048);
#pragma unroll
        for (int j = 0; j < WTN; j++) {
            const v8i bf = frag(st + b_rd + j * 2048);
#pragma unroll
            for (int i = 0; i < WTM; i++) mfma_f8_acc<A_FMT>(acc[i][j], bf, af[i]);
        }
    };
    // Step kt computes from LDS buffer kt & 1, then moves tile kt+1 (register slot (kt+1) & 1, loaded two
    // steps ago) into the other buffer and refills that slot with tile kt+3.
#define BL_STEP(KT, BUF)                 \
    do {                                 \
        compute(BUF);                    \
        BL_FILL((BUF) ^ 1, (BUF) ^ 1);   \
        BL_LOAD((BUF) ^ 1, (KT) + 3);    \
        __syncthreads();                 \
        __builtin_amdgcn_sched_barrier(0); \
    } while (0)
    // Interleaved step: the fill of the other LDS buffer and the reload of that register slot are cut into WTN
    // portions, one after each group of WTM MFMAs; B fragments are fetched one group ahead.
    constexpr int PIECES = A_CH + B_CH, PPG = (PIECES + WTN - 1) / WTN;
#define BL_STEP_I(KT, BUF)                                                                                     \
    do {                                                                                                       \
        const uint8_t* st__ = lds + (BUF) * STAGE;                                                             \
        uint8_t* fl__ = lds + ((BUF) ^ 1) * STAGE + lw;                                                        \
        const int t__ = (KT) + 3;                                                                              \
        const bool cut__ = t__ >= ksteps || (t__ == kfull && ch_in_tail);                                      \
        v8i af__[WTM], bf__[2];                                                                                \
        _Pragma("unroll") for (int i = 0; i < WTM; i++) af__[i] = frag(st__ + a_rd + i * 2048);                \
        bf__[0] = frag(st__ + b_rd);                                                                           \
        _Pragma("unroll") for (int j = 0; j < WTN; j++) {                                                      \
            if (j + 1 < WTN) bf__[(j + 1) & 1] = frag(st__ + b_rd + (j + 1) * 2048);                           \
            _Pragma("unroll") for (int q = 0; q < PPG; q++) {                                                  \
                const int p = j * PPG + q;                                                                     \
                const int pa = p < A_CH ? p : 0, pb = (p >= A_CH && p < PIECES) ? p - A_CH : 0;   /* in-range when not taken */ \
                if (p < A_CH) {                                                                                \
                    *(v4i*)(fl__ + pa * PASS_ROWS * 128) = ra[(BUF) ^ 1][pa];                                  \
                    ra[(BUF) ^ 1][pa] = __builtin_amdgcn_raw_buffer_load_b128(desc_a, cut__ ? NC_BUF_OOB : avo[pa], t__ * 128, 0); \
                } else if (p < PIECES) {                                                                       \
                    *(v4i*)(fl__ + BM * 128 + pb * PASS_ROWS * 128) = rb[(BUF) ^ 1][pb];                       \
                    rb[(BUF) ^ 1][pb] = __builtin_amdgcn_raw_buffer_load_b128(desc_b, cut__ ? NC_BUF_OOB : bvo[pb], t__ * 128, 0); \
                }                                                                                              \
            }                                                                                                  \
            _Pragma("unroll") for (int i = 0; i < WTM; i++) mfma_f8_acc_ordered<A_FMT>(acc[i][j], bf__[j & 1], af__[i]); \
        }                                                                                                      \
        __syncthreads();                                                                                       \
    } while (0)

    int kt = 0;
    {
        BL_LOAD(0, 0);
        BL_LOAD(1, 1);
        BL_FILL(0, 0);
        BL_LOAD(0, 2);
        __syncthreads();
        if (INTERLEAVE) {
            for (; kt + 1 < ksteps; kt += 2) {
                BL_STEP_I(kt, 0);
                BL_STEP_I(kt + 1, 1);
            }
        } else {
            for (; kt + 1 < ksteps; kt += 2) {
                BL_STEP(kt, 0);
                BL_STEP(kt + 1, 1);
            }
        }
        if (kt < ksteps) compute(0);
    }
#undef BL_STEP_I
#undef BL_LOAD
#undef BL_FILL
#undef BL_STEP

    // the last MFMAs must have left the pipeline before the accumulators are read (16 passes at most)
    asm volatile("s_nop 15\n\ts_nop 15" ::: "memory");
#pragma unroll
    for (int i = 0; i < WTM; i++)
#pragma unroll
        for (int j = 0; j < WTN; j++) asm volatile("" : "+a"(acc[i][j]));

    // epilogue: the (at most four) per-segment weight scales are fetched once
    const float inv_a = *ep.inv_a;
    float sc[4];
#pragma unroll
    for (int i = 0; i < 4; i++) sc[i] = ep.inv_b[i < ep.segs.nseg ? i : 0];
    bl_epilogue<BM, BN, WGM, WGN, OUT_KIND>(acc, lds, ep, inv_a, sc, m0, n0, M, N);
}


#include <atomic>
namespace {
int cu_count() { return nc_cu_count(); }
// Raises a kernel's limit of dynamic LDS (always to the same value), once per device.  The flags belong to the kernel: over
// fifty of them ask here, and a table that they shared had room for 32, behind which every launch searched it and set the limit again (0.1 us of 5.7).
template <auto KERNEL>
int reserve_lds(size_t bytes) {
    static std::atomic<uint64_t> done{0};
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev > 63) dev = 0;
    if (done.load(std::memory_order_acquire) >> dev & 1) return 0;
    const hipError_t e = hipFuncSetAttribute((const void*)KERNEL, hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes);
    if (e != hipSuccess) NC_FAIL(-2, "fp8_gemm: cannot reserve %zu bytes of LDS: %s", bytes, hipGetErrorString(e));
    done.fetch_or(1ull << dev, std::memory_order_release);
    return 0;
}
}  // namespace

template <int BM, int BN, int WGM, int WGN, bool INTERLEAVE, int A_FMT, int OUT_KIND>
static int launch_bl_as(const uint8_t* a, const uint8_t* b, const EpilogueArgs& ep, int M, int N, int K, hipStream_t s) {
    const int tiles_m = (M + BM - 1) / BM, tiles_n = (N + BN - 1) / BN;
    const size_t lds_bytes = 2 * (size_t)(BM + BN) * 128;
    if (int rc = reserve_lds<gemm_bl_kernel<BM, BN, WGM, WGN, OUT_KIND, INTERLEAVE, A_FMT>>(lds_bytes)) return rc;
    hipLaunchKernelGGL((gemm_bl_kernel<BM, BN, WGM, WGN, OUT_KIND, INTERLEAVE, A_FMT>), dim3(tiles_m * tiles_n), dim3(64 * WGM * WGN), lds_bytes, s, a, b,
                       ep, M, N, K, tiles_m, tiles_n);
    return 0;
}
template <int BM, int BN, int WGM, int WGN, bool INTERLEAVE = false, int A_FMT = 0>
static int launch_bl(const uint8_t* a, const uint8_t* b, const EpilogueArgs& ep, int M, int N, int K, hipStream_t s) {
    NC_CHECK_ARG((long)M * K < (1L << 31) && (long)N * K < (1L << 31), "fp8_gemm: buffer-load kernels need M*K and N*K below 2^31");
    if (ep.out_kind == 0) return launch_bl_as<BM, BN, WGM, WGN, INTERLEAVE, A_FMT, 0>(a, b, ep, M, N, K, s);
    NC_CHECK_ARG(A_FMT == 0, "fp8_gemm: an e5m2 operand goes with plain bf16 output");
    if (ep.out_kind == 1) return launch_bl_as<BM, BN, WGM, WGN, INTERLEAVE, 0, 1>(a, b, ep, M, N, K, s);
    return launch_bl_as<BM, BN, WGM, WGN, INTERLEAVE, 0, 2>(a, b, ep, M, N, K, s);
}


// ------------------------------------------------------------------------------------------------
// Direct-to-LDS kernels: 256x256x128 tiles, 8 waves (4 x 2, 64x128 outputs each), one workgroup per CU.  The operand
// tiles never pass through registers: every wave issues eight 1 KB `buffer_load_dwordx4 ... lds` per K-step, each of
// which lands 8 rows x 128 bytes in consecutive LDS; the swizzle of the LDS layout (chunk c of row r at slot
// c ^ NC_SWZ(r)) is applied on the global side, lane (sub, slot) fetching chunk slot ^ NC_SWZ(row) of its row, so each
// group of 8 lanes still reads one whole 128-byte line.  That removes the ds_write phase (a 64 KB stage costs ~860
// cycles at the 76 B/clk LDS write rate, next to 2048 cycles of MFMA) and the staging registers.  K must be a multiple
// of 128 (a K tail would need zero fill inside rows, which the range check of the descriptor cannot give); bf16 output.
typedef __attribute__((address_space(3))) void* lds_ptr_t;

struct DlGeom {
    int lane, wave, wm, wn, frow, kb;
    int sub, gch;          // this lane's row inside an 8-row block and the global chunk that belongs in its LDS slot
    int rd_lo, rd_hi;      // fragment read offsets inside a 16-row block
};
__device__ __forceinline__ DlGeom dl_geom() {
    DlGeom g;
    g.lane = threadIdx.x & 63, g.wave = threadIdx.x / 64;
    g.wm = g.wave / 2, g.wn = g.wave % 2;
    g.frow = g.lane & 15, g.kb = g.lane >> 4;
    g.sub = g.lane >> 3, g.gch = (g.lane & 7) ^ g.sub ^ (g.wave & 1);
    const int sw = NC_SWZ(g.frow);
    g.rd_lo = g.frow * 128 + (((2 * g.kb) ^ sw) << 4), g.rd_hi = g.frow * 128 + (((2 * g.kb + 1) ^ sw) << 4);
    return g;
}
__device__ __forceinline__ v8i dl_frag(const uint8_t* base, const DlGeom& g) {
    const v4i lo = *(const v4i*)(base + g.rd_lo);
    const v4i hi = *(const v4i*)(base + g.rd_hi);
    return v8i{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
}
// FIRST starts the accumulation from zero (C operand 0) instead of reading the accumulators.
template <int A_FMT = 0>
__device__ __forceinline__ void mfma_f8_first_ordered(v4f& acc, const v8i& b, const v8i& a) {
    if (A_FMT == 0) asm volatile("v_mfma_f32_16x16x128_f8f6f4 %0, %1, %2, 0" : "=a"(acc) : "v"(b), "v"(a) : "memory");
    else asm volatile("v_mfma_f32_16x16x128_f8f6f4 %0, %1, %2, 0 blgp:1" : "=a"(acc) : "v"(b), "v"(a) : "memory");
}
// One K-step of a wave: 64 rows x (128 or, for a half-width tile, 64) columns from the stage at `st`.
// `behind_first_reads` runs once the step's first fragment reads are on their way: the place to issue the operand loads of a later
// step, so that they do not stand between the barrier and the reads the first MFMA waits for.
struct DlNothing {
    __device__ void operator()() const {}
};
template <bool HALF, bool FIRST = false, int A_FMT = 0, typename F = DlNothing>
__device__ __forceinline__ void dl_compute(v4f (&acc)[4][8], const uint8_t* st, const DlGeom& g, F&& behind_first_reads = F()) {
    constexpr int WTN = HALF ? 4 : 8;
    const uint8_t* a = st + g.wm * 64 * 128;
    const uint8_t* b = st + 256 * 128 + g.wn * (HALF ? 64 : 128) * 128;
    v8i af[4], bf[2];
    bf[0] = dl_frag(b, g);
#pragma unroll
    for (int i = 0; i < 4; i++) af[i] = dl_frag(a + i * 2048, g);
    behind_first_reads();
#pragma unroll
    for (int j = 0; j < WTN; j++) {
        if (j + 1 < WTN) bf[(j + 1) & 1] = dl_frag(b + (j + 1) * 2048, g);    // one group ahead of its use
#pragma unroll
        for (int i = 0; i < 4; i++) {
            if (FIRST) mfma_f8_first_ordered<A_FMT>(acc[i][j], bf[j & 1], af[i]);
            else mfma_f8_acc_ordered<A_FMT>(acc[i][j], bf[j & 1], af[i]);
        }
    }
}

// The barrier that ends a K-step of the direct-to-LDS kernels.  The operand loads write LDS behind the compiler's back,
// so the wait for them is explicit: every vector memory operation of this wave has completed (the loads of the next step, and
// the stores of the previous tile's epilogue that were issued behind them), then the workgroup meets.  (Left to the compiler, the
// barrier after the first K-step of a tile came out as vmcnt(6), which on the first tile does not cover all of the step's loads.
// Letting the 16 stores of the previous tile stay in flight across this barrier, vmcnt(16), was measured 1 % slower.)
__device__ __forceinline__ void dl_step_barrier() {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(0x0F70);     // vmcnt(0), other counters untouched
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}

// The K loop of the tiles that are launched one by one: eight waves in a 4 x 2 grid.  One operand is HELD, four blocks of 16 rows per wave whose fragments are
// read a step ahead into registers of their own, through a ring of three stages; the other is STREAMED, NS blocks per wave, each read one group of
// products ahead of its use, through two stages.  With both operands read behind the barrier a step began with ten LDS reads per wave (80 KB a workgroup,
// 640 clocks) that nothing overlapped; now with two, the held operand's loads have two steps to arrive, and the loads go out between the products.  us, before /
// after: 8192 x 1664 x 6656 112.7 / 107.5 in 256 x 192 tiles, 85.5 / 82 in 256 x 256 ones; of thirteen steps 1792 x 4992 x 1664 19.9 / 20.0, 1792 x 6656 x 1664
// 22.0 / 21.9: what is left there is the launch, the first loads and the write.  Same products in the same order.
//   A_HELD: rows of A in the grid's first direction (acc[held][streamed]), else rows of B in the second (acc[streamed][held]).
//   HP: held pieces of 1 KB per wave and step: what may still be in flight when a step ends, while there is a step three ahead to load.
__device__ __forceinline__ void dl_piece(const uint8_t* p, int bytes, uint8_t* st, uint32_t vo, int k_off) {
    __builtin_amdgcn_raw_ptr_buffer_load_lds(__builtin_amdgcn_make_buffer_rsrc((void*)p, 0, bytes, 0x00020000), (lds_ptr_t)st, 16, vo, k_off, 0, 0);
}
template <bool A_HELD, int NS> constexpr int dl_stream_stage() { return (A_HELD ? 32 : 64) * NS * 128; }
template <bool A_HELD, int NS, int HP> constexpr int dl_ring_lds() { return 3 * HP * 8192 + 2 * dl_stream_stage<A_HELD, NS>(); }
template <bool A_HELD, int NS, int HP, int A_FMT, typename Acc>
__device__ __forceinline__ void dl_ring(Acc& acc, const uint8_t* A, int a_bytes, const uint8_t* B, int b_bytes, uint8_t* lds, const DlGeom& g, int wave_s,
                                        const uint32_t* vo_h, const uint32_t* vo_s, int ksteps) {
    constexpr int H_ST = HP * 8192, S_ST = dl_stream_stage<A_HELD, NS>(), S_PIECES = S_ST / 1024, S_ROUNDS = (S_PIECES + 7) / 8, WAIT = 0x0070 | HP;
    uint8_t* const ring_s = lds + 3 * H_ST;
    const int rd_h = (A_HELD ? g.wm : g.wn) * 64 * 128, rd_s = (A_HELD ? g.wn : g.wm) * 16 * NS * 128;
    // piece r of a step's loads: S_ROUNDS of the streamed operand first, then HP of the held one
    auto load_h = [&](int r, int t, int at) {
        if (t < ksteps) dl_piece(A_HELD ? A : B, A_HELD ? a_bytes : b_bytes, lds + at + wave_s * 1024 + r * 8192, vo_h[r], t * 128);
    };
    auto load_s = [&](int r, int t, int buf) {
        if (t < ksteps && (S_PIECES % 8 == 0 || wave_s + 8 * r < S_PIECES))       // uniform per wave
            dl_piece(A_HELD ? B : A, A_HELD ? b_bytes : a_bytes, ring_s + buf * S_ST + wave_s * 1024 + r * 8192, vo_s[r], t * 128);
    };
    auto meet = [&](bool in_flight) {
        asm volatile("" ::: "memory");
        if (in_flight) __builtin_amdgcn_s_waitcnt(WAIT);
        else __builtin_amdgcn_s_waitcnt(0x0070); // the next step's streamed operand and the held one behind it have landed, every fragment is read (this wave's share)
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
    };
    v8i held[2][4];
    int at0 = 0, at1 = H_ST, at2 = 2 * H_ST;     // stages of the held operand of this step, the next and the one after
    auto step = [&](int t, auto parity) __attribute__((always_inline)) {
        constexpr int P = decltype(parity)::value, Q = 1 - P;
        const uint8_t* const ss = ring_s + P * S_ST + rd_s;
        const uint8_t* const hs = lds + at1 + rd_h;
        v8i sf[2];
        sf[0] = dl_frag(ss, g);
#pragma unroll
        for (int j = 0; j < NS; j++) {
            if (j + 1 < NS) sf[(j + 1) & 1] = dl_frag(ss + (j + 1) * 2048, g);    // one group ahead of its use
#pragma unroll
            for (int i = 0; i < 4; i++)
                if (i * NS / 4 == j) held[Q][i] = dl_frag(hs + i * 2048, g);
#pragma unroll
            for (int i = 0; i < 4; i++) {
#pragma unroll
                for (int r = 0; r < S_ROUNDS + HP; r++)
                    if (r * 4 * NS / (S_ROUNDS + HP) == 4 * j + i) {
                        if (r < S_ROUNDS) load_s(r, t + 1, Q);
                        else load_h(r - S_ROUNDS, t + 3, at0);
                    }
                if constexpr (A_HELD) mfma_f8_acc_ordered<A_FMT>(acc[i][j], sf[j & 1], held[P][i]);
                else mfma_f8_acc_ordered<A_FMT>(acc[j][i], held[P][i], sf[j & 1]);
            }
        }
        meet(t + 3 < ksteps);
        const int first = at0;
        at0 = at1, at1 = at2, at2 = first;
    };
#pragma unroll
    for (int r = 0; r < S_ROUNDS; r++) load_s(r, 0, 0);
#pragma unroll
    for (int r = 0; r < 3 * HP; r++) load_h(r % HP, r / HP, r / HP * H_ST);
    asm volatile("" ::: "memory");
    if (ksteps > 2) __builtin_amdgcn_s_waitcnt(0x0070 | (2 * HP));       // the first step's operands
    else __builtin_amdgcn_s_waitcnt(0x0070);
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
#pragma unroll
    for (int i = 0; i < 4; i++) held[0][i] = dl_frag(lds + at0 + rd_h + i * 2048, g);
    meet(ksteps > 2);
    int kt = 0;
    for (; kt + 1 < ksteps; kt += 2) {
        step(kt, std::integral_constant<int, 0>{});
        step(kt + 1, std::integral_constant<int, 1>{});
    }
    if (kt < ksteps) step(kt, std::integral_constant<int, 0>{});
}

// Short sums take a K loop of two stages: the ring asks for two steps of its held operand before the first products, and what it saves a step is little beside few
// columns.  us, two stages / ring: 256 x 128 tiles, 2048 x 4096 x 256 8.1 / 8.4, x 1024 12.7 / 12.8, x 1536 16.3 / 16.2, x 4096 34.6 / 32.0; 256 x 160 tiles, 1792 x 4992 x
// 256 9.5 / 9.7, x 1024 14.7 / 14.9, x 1536 18.4 / 18.3, x 4096 37.0 / 36.4; 256 x 192 tiles, 1792 x 6656 x 128 8.3 / 8.5, x 256 10.0 / 10.1, x 512 12.2 / 12.1; 256 x 256
// tiles, 8192 x 2048 x 128 10.1 / 10.4, x 256 11.95 / 12.0, x 768 17.2 / 17.3, x 1536 25.5 / 25.3.  NJ: columns of a tile / 32.  (The relu^2 linear of a
// prompt that leaves e4m3 keeps the ring: its weight comes from HBM; depth 14, 1300 tokens 1200 / 1176, depth 12, 4 x 400 958 / 942.)
constexpr bool dl_two_stages(int NJ, int K) { return K <= (NJ <= 5 ? 1024 : 128); }

// One tile per workgroup, launched tile by tile (any M, N).
template <int A_FMT, int OUT_KIND, bool RING = OUT_KIND == 0>
__global__ __launch_bounds__(512) void gemm_dl_kernel(const uint8_t* __restrict__ A, const uint8_t* __restrict__ B, EpilogueArgs ep, int M,
                                                      int N, int K, int tiles_m, int tiles_n) {
    constexpr int STAGE = 512 * 128;
    extern __shared__ __align__(16) uint8_t lds[];
    int tm, tn;
    tile_coords(blockIdx.x, tiles_m, tiles_n, tm, tn);
    const int m0 = tm * 256, n0 = tn * 256;
    const DlGeom g = dl_geom();
    const int wave_s = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const __amdgpu_buffer_rsrc_t desc_a = __builtin_amdgcn_make_buffer_rsrc((void*)A, 0, M * K, 0x00020000);
    const __amdgpu_buffer_rsrc_t desc_b = __builtin_amdgcn_make_buffer_rsrc((void*)B, 0, N * K, 0x00020000);

    // piece i of this wave is the 1 KB block (wave + 8 i) of the stage: tile rows 8 wave + 64 i + sub, A for i < 4, B after
    uint32_t vo[8];
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const int ra = m0 + 8 * g.wave + 64 * i + g.sub, rb = n0 + 8 * g.wave + 64 * i + g.sub;
        vo[i] = ra < M ? (uint32_t)ra * (uint32_t)K + g.gch * 16 : NC_BUF_OOB;
        vo[4 + i] = rb < N ? (uint32_t)rb * (uint32_t)K + g.gch * 16 : NC_BUF_OOB;
    }
    const int ksteps = K / 128;

    v4f acc[4][8];
#pragma unroll
    for (int i = 0; i < 4; i++)
#pragma unroll
        for (int j = 0; j < 8; j++) acc[i][j] = v4f{0.f, 0.f, 0.f, 0.f};

    auto fetch = [&](int t, int buf) {
        if (t < ksteps) {
            uint8_t* st = lds + buf * STAGE + wave_s * 1024;      // uniform: the LDS address of a load goes through M0
#pragma unroll
            for (int i = 0; i < 8; i++)
                __builtin_amdgcn_raw_ptr_buffer_load_lds(i < 4 ? desc_a : desc_b, (lds_ptr_t)(st + i * 8192), 16, vo[i], t * 128, 0, 0);
        }
    };
    if constexpr (RING) {
        dl_ring<true, 8, 4, A_FMT>(acc, A, M * K, B, N * K, lds, g, wave_s, vo, vo + 4, ksteps);
    } else {
        // (and where there is no room for the third stage beside the words of the other epilogues)
        // step kt computes from buffer kt & 1 while the loads of step kt + 1 land in the other one; the barrier at its end
        // says both that those loads are complete for every wave and that nobody reads buffer kt & 1 any more
        fetch(0, 0);
        dl_step_barrier();
        int kt = 0;
        for (; kt + 1 < ksteps; kt += 2) {
            dl_compute<false, false, A_FMT>(acc, lds, g, [&] { fetch(kt + 1, 1); });
            dl_step_barrier();
            dl_compute<false, false, A_FMT>(acc, lds + STAGE, g, [&] { fetch(kt + 2, 0); });
            dl_step_barrier();
        }
        if (kt < ksteps) dl_compute<false, false, A_FMT>(acc, lds, g);
    }

    asm volatile("s_nop 15\n\ts_nop 15" ::: "memory");
#pragma unroll
    for (int i = 0; i < 4; i++)
#pragma unroll
        for (int j = 0; j < 8; j++) asm volatile("" : "+a"(acc[i][j]));
    const float inv_a = *ep.inv_a;
    float sc[4];
#pragma unroll
    for (int i = 0; i < 4; i++) sc[i] = ep.inv_b[i < ep.segs.nseg ? i : 0];
    if constexpr (OUT_KIND == 4) q8_epilogue<256, 256, 4, 2>(acc, lds, ep, inv_a, sc, m0, n0, M, N, tiles_m, tiles_n);
    else bl_epilogue<256, 256, 4, 2, OUT_KIND>(acc, lds, ep, inv_a, sc, m0, n0, M, N);
}

// ------------------------------------------------------------------------------------------------
// The same tile-by-tile kernel with a narrower tile: 256 rows x 32 NJ columns (NJ = 4 .. 7 blocks of 16 columns per wave).  A launch of
// one round -- a prompt of one to two thousand rows -- lasts as long as one tile, whatever the number of CUs that got one: 1792 x 4992
// is 140 tiles of 256 x 256 on 256 CUs, but 224 tiles of 256 x 160, each 5/8 of the matrix work.  The launch picks NJ (dl_pick_nj).
// Epilogue for a wave block of 64 x 16 NJ outputs, bf16 (RELU2: relu(v)^2 and its maximum): the block is parked in the wave's own
// LDS region (rows of 32 NJ + 16 bytes) and leaves as a linear sequence of 16-byte pieces, so a store instruction writes runs of
// 32 NJ contiguous bytes per row.
template <int NJ, bool RELU2>
__device__ __forceinline__ void dln_epilogue(v4f (&acc)[4][NJ], uint8_t* lds, const EpilogueArgs& ep, float inv_a, const float (&sc)[4],
                                             const DlGeom& g, int m0, int n0, int M, int N) {
    constexpr int WCOLS = 16 * NJ, ROWB = WCOLS * 2, PITCH = ROWB + 16, LPR = ROWB / 16, PIECES = 64 * LPR;
    static_assert(8 * 64 * PITCH <= 2 * (256 + 32 * NJ) * 128, "epilogue staging");
    float am = 0.f;
    __syncthreads();                                       // every wave is done with the operand tiles
    uint8_t* reg = lds + g.wave * 64 * PITCH;
#pragma unroll
    for (int j = 0; j < NJ; j++) {
        const int n = n0 + g.wn * WCOLS + j * 16 + 4 * g.kb;
        float inv_b = sc[0];
#pragma unroll
        for (int i = 0; i < 3; i++)
            if (i + 1 < ep.segs.nseg && n >= ep.segs.end[i]) inv_b = sc[i + 1];
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const int row = i * 16 + g.frow;
            const v4f a4 = acc[i][j];
            float o4[4];
#pragma unroll
            for (int r = 0; r < 4; r++) {
                o4[r] = (a4[r] * inv_a) * inv_b;
                if (RELU2) o4[r] = relu2_of(o4[r]);
            }
            *(uint2*)(reg + row * PITCH + j * 32 + g.kb * 8) = make_uint2(pack_bf16_hw(o4[0], o4[1]), pack_bf16_hw(o4[2], o4[3]));
        }
    }
    // the region is private to the wave: its own LDS writes only have to land before its reads
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_s_waitcnt(0xc07f);                    // lgkmcnt(0)
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    const bool vec16 = (ep.ldc % 8 == 0) && (((uintptr_t)ep.out & 15) == 0);
#pragma unroll
    for (int it = 0; it < PIECES / 64; it++) {
        const int id = it * 64 + g.lane, row = id / LPR, c = id % LPR;
        const int m = m0 + g.wm * 64 + row, n = n0 + g.wn * WCOLS + c * 8;
        const uint4 v = *(const uint4*)(reg + row * PITCH + c * 16);
        if (m >= M || n >= N) continue;
        if (RELU2) am = amax_join(am, max_bf16x8(v, N - n));
        bf16_t* o = (bf16_t*)ep.out + (size_t)m * ep.ldc + n;
        if (n + 8 <= N) {
            if (vec16) __builtin_nontemporal_store(v4i{(int)v.x, (int)v.y, (int)v.z, (int)v.w}, (v4i*)o);
            else {
                *(uint2*)o = make_uint2(v.x, v.y);
                *(uint2*)(o + 4) = make_uint2(v.z, v.w);
            }
        } else {
            const uint32_t w[4] = {v.x, v.y, v.z, v.w};
            for (int r = 0; r < 8 && n + r < N; r++) o[r] = (bf16_t)(w[r >> 1] >> ((r & 1) * 16));
        }
    }
    if (RELU2) {
        __shared__ float wave_am[8];
        am = wave_amax(am);
        if (g.lane == 0) wave_am[g.wave] = am;
        __syncthreads();
        if (threadIdx.x == 0) {
            float t = wave_am[0];
#pragma unroll
            for (int w = 1; w < 8; w++) t = amax_join(t, wave_am[w]);
            amax_publish(ep.out_amax, t);
        }
    }
}

template <int NJ, int A_FMT = 0, typename F = DlNothing>
__device__ __forceinline__ void dln_compute(v4f (&acc)[4][NJ], const uint8_t* st, const DlGeom& g, F&& behind_first_reads = F()) {
    const uint8_t* a = st + g.wm * 64 * 128;
    const uint8_t* b = st + 256 * 128 + g.wn * (16 * NJ) * 128;
    v8i af[4], bf[2];
    bf[0] = dl_frag(b, g);
#pragma unroll
    for (int i = 0; i < 4; i++) af[i] = dl_frag(a + i * 2048, g);
    behind_first_reads();
#pragma unroll
    for (int j = 0; j < NJ; j++) {
        if (j + 1 < NJ) bf[(j + 1) & 1] = dl_frag(b + (j + 1) * 2048, g);    // one group ahead of its use
#pragma unroll
        for (int i = 0; i < 4; i++) mfma_f8_acc_ordered<A_FMT>(acc[i][j], bf[j & 1], af[i]);
    }
}

// the operand loads of one K-step: `st` is the wave's first 1 KB piece of the stage (uniform: the LDS address of a load goes through M0)
template <int NJ>
__device__ __forceinline__ void dln_fetch(const uint8_t* A, int a_bytes, const uint8_t* B, int b_bytes, uint8_t* st, const uint32_t* vo_a,
                                          const uint32_t* vo_b, int wave_s, int k_off) {
    const __amdgpu_buffer_rsrc_t desc_a = __builtin_amdgcn_make_buffer_rsrc((void*)A, 0, a_bytes, 0x00020000);
    const __amdgpu_buffer_rsrc_t desc_b = __builtin_amdgcn_make_buffer_rsrc((void*)B, 0, b_bytes, 0x00020000);
#pragma unroll
    for (int i = 0; i < 4; i++) __builtin_amdgcn_raw_ptr_buffer_load_lds(desc_a, (lds_ptr_t)(st + i * 8192), 16, vo_a[i], k_off, 0, 0);
#pragma unroll
    for (int i = 0; i < (4 * NJ + 7) / 8; i++)
        if (wave_s + 8 * i < 4 * NJ)                      // uniform per wave
            __builtin_amdgcn_raw_ptr_buffer_load_lds(desc_b, (lds_ptr_t)(st + 256 * 128 + i * 8192), 16, vo_b[i], k_off, 0, 0);
}

template <int NJ, int OUT_KIND, int A_FMT = 0, bool RING = true>
__global__ __launch_bounds__(512) void gemm_dln_kernel(const uint8_t* __restrict__ A, const uint8_t* __restrict__ B, EpilogueArgs ep, int M,
                                                       int N, int K, int tiles_m, int tiles_n) {
    constexpr int BN = 32 * NJ, STAGE = (256 + BN) * 128, B_ROUNDS = (BN / 8 + 7) / 8;
    extern __shared__ __align__(16) uint8_t lds[];
    int tm, tn;
    tile_coords(blockIdx.x, tiles_m, tiles_n, tm, tn);
    const int m0 = tm * 256, n0 = tn * BN;
    const DlGeom g = dl_geom();
    const int wave_s = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);

    // piece i of this wave is the 1 KB block (wave + 8 i) of its operand's part of the stage: tile rows 8 wave + 64 i + sub
    uint32_t vo_a[4], vo_b[B_ROUNDS];
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const int ra = m0 + 8 * g.wave + 64 * i + g.sub;
        vo_a[i] = ra < M ? (uint32_t)ra * (uint32_t)K + g.gch * 16 : NC_BUF_OOB;
    }
#pragma unroll
    for (int i = 0; i < B_ROUNDS; i++) {
        const int rb = n0 + 8 * g.wave + 64 * i + g.sub;
        vo_b[i] = rb < N ? (uint32_t)rb * (uint32_t)K + g.gch * 16 : NC_BUF_OOB;
    }
    const int ksteps = K / 128;

    v4f acc[4][NJ];
#pragma unroll
    for (int i = 0; i < 4; i++)
#pragma unroll
        for (int j = 0; j < NJ; j++) acc[i][j] = v4f{0.f, 0.f, 0.f, 0.f};

    if constexpr (RING) {
        dl_ring<true, NJ, 4, A_FMT>(acc, A, M * K, B, N * K, lds, g, wave_s, vo_a, vo_b, ksteps);
    } else {
        auto fetch = [&](int t, int buf) {
            if (t < ksteps) dln_fetch<NJ>(A, M * K, B, N * K, lds + buf * STAGE + wave_s * 1024, vo_a, vo_b, wave_s, t * 128);
        };
        fetch(0, 0);
        dl_step_barrier();
        int kt = 0;
        for (; kt + 1 < ksteps; kt += 2) {
            dln_compute<NJ, A_FMT>(acc, lds, g, [&] { fetch(kt + 1, 1); });
            dl_step_barrier();
            dln_compute<NJ, A_FMT>(acc, lds + STAGE, g, [&] { fetch(kt + 2, 0); });
            dl_step_barrier();
        }
        if (kt < ksteps) dln_compute<NJ, A_FMT>(acc, lds, g);
    }

    asm volatile("s_nop 15\n\ts_nop 15" ::: "memory");
#pragma unroll
    for (int i = 0; i < 4; i++)
#pragma unroll
        for (int j = 0; j < NJ; j++) asm volatile("" : "+a"(acc[i][j]));
    const float inv_a = *ep.inv_a;
    float sc[4];
#pragma unroll
    for (int i = 0; i < 4; i++) sc[i] = ep.inv_b[i < ep.segs.nseg ? i : 0];
    if constexpr (OUT_KIND == 4) q8_epilogue<256, BN, 4, 2>(acc, lds, ep, inv_a, sc, m0, n0, M, N, tiles_m, tiles_n);
    else dln_epilogue<NJ, OUT_KIND == 2>(acc, lds, ep, inv_a, sc, g, m0, n0, M, N);
}

// The same once more with tiles of 64 WTM rows x 128 columns (WTM = 2 .. 6 blocks of 16 rows per wave): whole heads of the q|k|v linear, for rope_epilogue.  The
// 320-row tile has the area of the 256 x 160 one.
template <int WTM>
__global__ __launch_bounds__(512) void gemm_rope_kernel(const uint8_t* __restrict__ A, const uint8_t* __restrict__ B, EpilogueArgs ep, RopeArgs rope, int M, int N,
                                                        int K, int tiles_m, int tiles_n) {
    constexpr int BM = 64 * WTM;
    extern __shared__ __align__(16) uint8_t lds[];
    int tm, tn;
    tile_coords(blockIdx.x, tiles_m, tiles_n, tm, tn);
    const int m0 = tm * BM, n0 = tn * 128;
    const DlGeom g = dl_geom();
    const int wave_s = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    // piece i of this wave is the 1 KB block (wave + 8 i) of its operand's part of the stage: tile rows 8 wave + 64 i + sub
    uint32_t vo_a[WTM], vo_b[2];
#pragma unroll
    for (int i = 0; i < WTM; i++) {
        const int ra = m0 + 8 * g.wave + 64 * i + g.sub;
        vo_a[i] = ra < M ? (uint32_t)ra * (uint32_t)K + g.gch * 16 : NC_BUF_OOB;
    }
#pragma unroll
    for (int i = 0; i < 2; i++) {
        const int rb = n0 + 8 * g.wave + 64 * i + g.sub;
        vo_b[i] = rb < N ? (uint32_t)rb * (uint32_t)K + g.gch * 16 : NC_BUF_OOB;
    }
    const int ksteps = K / 128;
    v4f acc[WTM][4];
#pragma unroll
    for (int i = 0; i < WTM; i++)
#pragma unroll
        for (int j = 0; j < 4; j++) acc[i][j] = v4f{0.f, 0.f, 0.f, 0.f};
    dl_ring<false, WTM, 2, 0>(acc, A, M * K, B, N * K, lds, g, wave_s, vo_b, vo_a, ksteps);

    asm volatile("s_nop 15\n\ts_nop 15" ::: "memory");
#pragma unroll
    for (int i = 0; i < WTM; i++)
#pragma unroll
        for (int j = 0; j < 4; j++) asm volatile("" : "+a"(acc[i][j]));
    const float inv_a = *ep.inv_a;
    float sc[4];
#pragma unroll
    for (int i = 0; i < 4; i++) sc[i] = ep.inv_b[i < ep.segs.nseg ? i : 0];
    rope_epilogue<BM, 4, 2>(acc, lds, ep, rope, inv_a, sc, m0, n0, M);
}

// load r of the A_P + 4 operand loads of one K-step of gemm_dr_kernel: `st` is the wave's first 1 KB piece of the stage, its pieces lie 4 KB apart
template <int A_P>
__device__ __forceinline__ void dr_load(const uint8_t* A, int a_bytes, const uint8_t* B, int b_bytes, uint8_t* st, int b_part, const uint32_t* vo_a,
                                        const uint32_t* vo_b, int r, int k_off) {
    const __amdgpu_buffer_rsrc_t desc_a = __builtin_amdgcn_make_buffer_rsrc((void*)A, 0, a_bytes, 0x00020000);
    const __amdgpu_buffer_rsrc_t desc_b = __builtin_amdgcn_make_buffer_rsrc((void*)B, 0, b_bytes, 0x00020000);
    if (r < A_P) __builtin_amdgcn_raw_ptr_buffer_load_lds(desc_a, (lds_ptr_t)(st + r * 4096), 16, vo_a[r], k_off, 0, 0);
    else __builtin_amdgcn_raw_ptr_buffer_load_lds(desc_b, (lds_ptr_t)(st + b_part + (r - A_P) * 4096), 16, vo_b[r - A_P], k_off, 0, 0);
}

// ------------------------------------------------------------------------------------------------
// Direct-to-LDS tiles for a narrow weight under a prompt: BM x 128 outputs (BM = 64, 96, 128), four waves (2 x 2, BM/2 x 64 each), and a
// ring of FOUR operand stages.  Where the 256-row tiles would leave most CUs without one (1792 x 1664: 49 or 91 tiles), the launch is
// one round of small tiles, one workgroup of one wave per SIMD on each CU: nothing hides the latency of a K-step's operands then but
// the depth of the prefetch.  The register-staged tiles have two K-steps in flight and pay a ds_write phase per step; here the operands
// of four steps ahead are on their way into LDS while one is multiplied from registers that were filled during the step before, and a step costs its
// loads (28 KB at some 35 bytes a clock for 96 x 128) or its products, whichever is longer: 0.40 -> 0.33 us a step by the second set of registers.  Past
// the end of K the loads are issued all the same (the first step's operands again, into stages nobody reads), so that
// the count the barrier waits for is the same in every step.
//
// OUT_KIND 3: the K-steps are dealt to gridDim.y workgroups per tile, which leave raw fp32 sums ([share][M][N] at ep.out) for the row pass
// that adds the linear's output to the residual stream anyway (nc_gemm_prompt_splits).
template <int BM, int OUT_KIND, typename Rope = NoRope>
__global__ __launch_bounds__(256) void gemm_dr_kernel(const uint8_t* __restrict__ A, const uint8_t* __restrict__ B, EpilogueArgs ep, int M,
                                                      int N, int K, int tiles_m, int tiles_n, Rope rope) {
    constexpr int WTM = BM / 32, STAGE = (BM + 128) * 128, A_P = BM / 32, LOADS = A_P + 4;
    // s_waitcnt vmcnt(n * LOADS) lgkmcnt(0): the loads of the n youngest steps may still be in flight, no LDS read
    constexpr int WAIT2 = 0x0070 | ((2 * LOADS) & 15) | (((2 * LOADS) >> 4) << 14), WAIT3 = 0x0070 | ((3 * LOADS) & 15) | (((3 * LOADS) >> 4) << 14);
    extern __shared__ __align__(16) uint8_t lds[];
    int tm, tn;
    tile_coords(blockIdx.x, tiles_m, tiles_n, tm, tn);
    const int m0 = tm * BM, n0 = tn * 128;
    DlGeom g = dl_geom();
    g.wm = g.wave >> 1, g.wn = g.wave & 1;
    const int wave_s = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    // piece i of this wave is the 1 KB block (wave + 4 i) of its operand's part of the stage: tile rows 8 wave + 32 i + sub
    uint32_t vo_a[A_P], vo_b[4];
#pragma unroll
    for (int i = 0; i < A_P; i++) {
        const int ra = m0 + 8 * g.wave + 32 * i + g.sub;
        vo_a[i] = ra < M ? (uint32_t)ra * (uint32_t)K + g.gch * 16 : NC_BUF_OOB;
    }
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const int rb = n0 + 8 * g.wave + 32 * i + g.sub;
        vo_b[i] = rb < N ? (uint32_t)rb * (uint32_t)K + g.gch * 16 : NC_BUF_OOB;
    }
    const int k_first = OUT_KIND == 3 ? (int)((long)(K / 128) * blockIdx.y / gridDim.y) : 0;
    const int ksteps = OUT_KIND == 3 ? (int)((long)(K / 128) * (blockIdx.y + 1) / gridDim.y) - k_first : K / 128;
    A += k_first * 128, B += k_first * 128;

    v4f acc[WTM][4];
#pragma unroll
    for (int i = 0; i < WTM; i++)
#pragma unroll
        for (int j = 0; j < 4; j++) acc[i][j] = v4f{0.f, 0.f, 0.f, 0.f};

    auto fetch = [&](int t) {
#pragma unroll
        for (int r = 0; r < LOADS; r++)
            dr_load<A_P>(A, M * K - k_first * 128, B, N * K - k_first * 128, lds + (t & 3) * STAGE + wave_s * 1024, BM * 128, vo_a, vo_b, r, t < ksteps ? t * 128 : 0);
    };
    // One step: its products, between them the reads of the next step's fragments (into other registers) and the loads of the step four ahead.  Neither
    // the barrier nor an LDS read is waited for with the matrix cores idle: when the waves meet, every wave has read all of the stage of the step to be
    // multiplied, so that stage is free for loads, and the next one has landed.
    const int a_rd = g.wm * (BM / 2) * 128, b_rd = BM * 128 + g.wn * 64 * 128;
    v8i fa[2][WTM], fb[2][4];
    auto step = [&](int t, auto parity) __attribute__((always_inline)) {
        constexpr int P = decltype(parity)::value, Q = 1 - P, READS = WTM + 4, PRODUCTS = 4 * WTM;
        const uint8_t* const st = lds + ((t + 1) & 3) * STAGE;
        const int k_off = t + 4 < ksteps ? (t + 4) * 128 : 0;
        uint8_t* const to = lds + (t & 3) * STAGE + wave_s * 1024;
#pragma unroll
        for (int j = 0; j < 4; j++)
#pragma unroll
            for (int i = 0; i < WTM; i++) {
                const int n = j * WTM + i;
#pragma unroll
                for (int r = 0; r < READS; r++)
                    if (r * PRODUCTS / READS == n) {
                        if (r == 0) fb[Q][0] = dl_frag(st + b_rd, g);
                        else if (r <= WTM) fa[Q][r - 1] = dl_frag(st + a_rd + (r - 1) * 2048, g);
                        else fb[Q][r - WTM] = dl_frag(st + b_rd + (r - WTM) * 2048, g);
                    }
#pragma unroll
                for (int r = 0; r < LOADS; r++)
                    if (r * PRODUCTS / LOADS == n) dr_load<A_P>(A, M * K - k_first * 128, B, N * K - k_first * 128, to, BM * 128, vo_a, vo_b, r, k_off);
                mfma_f8_acc_ordered<0>(acc[i][j], fb[P][j], fa[P][i]);
            }
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_waitcnt(WAIT2);   // the operands of step t + 2 have landed, the fragments of step t + 1 are read (this wave's share; the barrier says everybody's)
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
    };
    fetch(0);
    fetch(1);
    fetch(2);
    fetch(3);
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(WAIT3);
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    fb[0][0] = dl_frag(lds + b_rd, g);
#pragma unroll
    for (int i = 0; i < WTM; i++) fa[0][i] = dl_frag(lds + a_rd + i * 2048, g);
#pragma unroll
    for (int j = 1; j < 4; j++) fb[0][j] = dl_frag(lds + b_rd + j * 2048, g);
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(WAIT2);
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    int kt = 0;
    for (; kt + 1 < ksteps; kt += 2) {
        step(kt, std::integral_constant<int, 0>{});
        step(kt + 1, std::integral_constant<int, 1>{});
    }
    if (kt < ksteps) step(kt, std::integral_constant<int, 0>{});
    // the loads past the end of K are still landing in the stages: they must be done before the epilogue reuses the memory
    dl_step_barrier();

    asm volatile("s_nop 15\n\ts_nop 15" ::: "memory");
#pragma unroll
    for (int i = 0; i < WTM; i++)
#pragma unroll
        for (int j = 0; j < 4; j++) asm volatile("" : "+a"(acc[i][j]));
    if constexpr (OUT_KIND == 3) {
        float* const out = (float*)ep.out + (size_t)blockIdx.y * M * N;
#pragma unroll
        for (int i = 0; i < WTM; i++)
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const int m = m0 + g.wm * (BM / 2) + 16 * i + g.frow, n = n0 + g.wn * 64 + 16 * j + 4 * g.kb;
                if (m < M && n < N) *(v4f*)(out + (size_t)m * N + n) = acc[i][j];
            }
        return;
    } else {
        const float inv_a = *ep.inv_a;
        float sc[4];
#pragma unroll
        for (int i = 0; i < 4; i++) sc[i] = ep.inv_b[i < ep.segs.nseg ? i : 0];
        if constexpr (OUT_KIND == 4) q8_epilogue<BM, 128, 2, 2>(acc, lds, ep, inv_a, sc, m0, n0, M, N, tiles_m, tiles_n);
        else if constexpr (OUT_KIND == 5) rope_epilogue<BM, 2, 2>(acc, lds, ep, rope, inv_a, sc, m0, n0, M);
        else bl_epilogue<BM, 128, 2, 2, OUT_KIND>(acc, lds, ep, inv_a, sc, m0, n0, M, N);
    }
}

// Epilogue of the persistent kernel: the wave's 64 x (128 | 64) block leaves 16 rows at a time through a 4 KB LDS region of
// its own (past the two operand stages, so the loads of the next tile keep landing meanwhile), every store instruction
// writing whole 128-byte lines.
template <bool HALF, bool RELU2>
__device__ __forceinline__ void dlp_epilogue(v4f (&acc)[4][8], uint8_t* reg, const EpilogueArgs& ep, float inv_a, const float (&sc)[4],
                                             const DlGeom& g, int m0, int n0, int M, int N) {
    constexpr int WTN = HALF ? 4 : 8, WCOLS = WTN * 16, ROWB = WCOLS * 2, LPR = ROWB / 16, RPI = 64 / LPR;
    const bool vec16 = (ep.ldc % 8 == 0) && (((uintptr_t)ep.out & 15) == 0);
    const uint32_t reg_off = (uint32_t)(uintptr_t)(lds_ptr_t)reg;       // the region's byte offset in LDS
    constexpr bool relu2 = RELU2;
    float am = 0.f;
    const int lrow_e = g.lane / LPR, c = g.lane % LPR;
    const int n_st = n0 + g.wn * WCOLS + c * 8;
    float inv_b[WTN];
#pragma unroll
    for (int j = 0; j < WTN; j++) {
        const int n = n0 + g.wn * WCOLS + j * 16 + 4 * g.kb;
        inv_b[j] = sc[0];
#pragma unroll
        for (int i = 0; i < 3; i++)
            if (i + 1 < ep.segs.nseg && n >= ep.segs.end[i]) inv_b[j] = sc[i + 1];
    }
#pragma unroll
    for (int i = 0; i < 4; i++) {
#pragma unroll
        for (int j = 0; j < WTN; j++) {
            const int chunk = 2 * j + (g.kb >> 1);
            const v4f a4 = acc[i][j];
            float o4[4];
#pragma unroll
            for (int r = 0; r < 4; r++) {
                o4[r] = (a4[r] * inv_a) * inv_b[j];
                if (relu2) o4[r] = relu2_of(o4[r]);
            }
            const v2i pk = {(int)pack_bf16_hw(o4[0], o4[1]), (int)pack_bf16_hw(o4[2], o4[3])};
            // written and read back with explicit instructions: an LDS access the compiler generates here waits for the next
            // tile's operand loads (vmcnt(0)), because it cannot tell this region from the stages they are landing in
            asm volatile("ds_write_b64 %0, %1" ::"v"(reg_off + g.frow * ROWB + ((chunk ^ (g.frow & 7)) << 4) + (g.kb & 1) * 8), "v"(pk) : "memory");
        }
        // the region is private to the wave: its own LDS writes only have to land before its reads
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_s_waitcnt(0xc07f);                    // lgkmcnt(0)
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        v4i rd[16 / RPI];
#pragma unroll
        for (int it = 0; it < 16 / RPI; it++) {
            const int row = it * RPI + lrow_e;
            asm volatile("ds_read_b128 %0, %1" : "=v"(rd[it]) : "v"(reg_off + row * ROWB + ((c ^ (row & 7)) << 4)) : "memory");
        }
        if (16 / RPI == 4) asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(rd[0]), "+v"(rd[1]), "+v"(rd[2 % (16 / RPI)]), "+v"(rd[3 % (16 / RPI)])::"memory");
        else asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(rd[0]), "+v"(rd[1])::"memory");
#pragma unroll
        for (int it = 0; it < 16 / RPI; it++) {
            const int row = it * RPI + lrow_e;
            const int m = m0 + g.wm * 64 + i * 16 + row;
            const uint4 v = make_uint4((uint32_t)rd[it][0], (uint32_t)rd[it][1], (uint32_t)rd[it][2], (uint32_t)rd[it][3]);
            if (m >= M || n_st >= N) continue;
            if (relu2) am = amax_join(am, max_bf16x8(v, N - n_st));
            bf16_t* o = (bf16_t*)ep.out + (size_t)m * ep.ldc + n_st;
            if (n_st + 8 <= N) {
                if (vec16) __builtin_nontemporal_store(v4i{(int)v.x, (int)v.y, (int)v.z, (int)v.w}, (v4i*)o);
                else {
                    *(uint2*)o = make_uint2(v.x, v.y);
                    *(uint2*)(o + 4) = make_uint2(v.z, v.w);
                }
            } else {
                const uint32_t w[4] = {v.x, v.y, v.z, v.w};
                for (int r = 0; r < 8 && n_st + r < N; r++) o[r] = (bf16_t)(w[r >> 1] >> ((r & 1) * 16));
            }
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");   // the reads are done before the next 16 rows overwrite the region
    }
    if (relu2) {
        am = wave_amax(am);
        if (g.lane == 0) amax_publish(ep.out_amax, am);
    }
}

// Persistent form: 8 x 32 workgroups, each walking its own list of tiles as one uninterrupted stream of K-steps (the
// first loads of the next tile are in flight while the current one is finished and stored).  XCD x (workgroup id % 8)
// owns `rows_per_xcd` consecutive tile rows; its 32 workgroups form rows_per_xcd x (32 / rows_per_xcd) slots, slot
// (r, c) owning tile row r and the c-th share of the N range counted in 128-column units.  A share is cut into full
// 256-column tiles plus, when its unit count is odd, one half-width tile at its end, so no workgroup rounds its work up
// to whole 256x256 tiles.
template <int A_FMT, bool RELU2>
__global__ __launch_bounds__(512) void gemm_dlp_kernel(const uint8_t* __restrict__ A, const uint8_t* __restrict__ B, EpilogueArgs ep,
                                                       int M, int N, int K, int rows_per_xcd, int nu) {
    constexpr int STAGE = 512 * 128;
    extern __shared__ __align__(16) uint8_t lds[];
    const DlGeom g = dl_geom();
    const int wave_s = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int xcd = blockIdx.x % 8, slot = blockIdx.x / 8;
    const int cols = 32 / rows_per_xcd;
    const int sc_c = slot % cols, sc_r = slot / cols;
    const int m0 = (xcd * rows_per_xcd + sc_r) * 256;
    const int ub = nu * sc_c / cols, ue = nu * (sc_c + 1) / cols;
    const int count = ue - ub, nitems = (count + 1) / 2;
    const bool has_half = count & 1;
    if (nitems == 0) return;
    // A share with an odd unit count has one half-width tile: at its end in the even slots, at its start in the odd ones, so that the
    // workgroups do not all reach their epilogues -- 128 KB of stores each -- at the same moments (M = 8192, N = 4992: 63 -> 61 us,
    // N = 6656: 82.5 -> 80 us, alternating in one process)
    const bool half_first = has_half && (slot & 1);
    auto item = [&](int q, int& n0, bool& half) {
        half = has_half && q == (half_first ? 0 : nitems - 1);
        n0 = (ub + 2 * q - ((half_first && q > 0) ? 1 : 0)) * 128;
    };

    const __amdgpu_buffer_rsrc_t desc_a = __builtin_amdgcn_make_buffer_rsrc((void*)A, 0, M * K, 0x00020000);
    const __amdgpu_buffer_rsrc_t desc_b = __builtin_amdgcn_make_buffer_rsrc((void*)B, 0, N * K, 0x00020000);
    const int ksteps = K / 128;
    uint32_t vo_a[4], vo_b[4];
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const int ra = m0 + 8 * g.wave + 64 * i + g.sub;
        vo_a[i] = ra < M ? (uint32_t)ra * (uint32_t)K + g.gch * 16 : NC_BUF_OOB;
    }
    // the fetch cursor runs ahead of the compute cursor, across tile boundaries
    int fq = 0, fkt = 0, fbuf = 0;
    bool f_half = false;
    auto set_fetch_item = [&](int q) {
        int n0;
        item(q, n0, f_half);
        // The lane's row and chunk are worked out again here from the lane id rather than kept in registers across the K loop:
        // the kernel has none to spare (kept live, the row offset was spilled, and its reload put a vmcnt(0) into the stream
        // of operand loads once per tile).  The asm keeps the compiler from hoisting the computation back out.
        int lane_id;
        asm volatile("v_mbcnt_lo_u32_b32 %0, -1, 0\n\tv_mbcnt_hi_u32_b32 %0, -1, %0" : "=v"(lane_id));
        const int sub = lane_id >> 3, gch = (lane_id & 7) ^ sub ^ (wave_s & 1);
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const int rb = n0 + 8 * wave_s + 64 * i + sub;
            vo_b[i] = rb < N ? (uint32_t)rb * (uint32_t)K + gch * 16 : NC_BUF_OOB;
        }
    };
    auto fetch_next = [&]() {
        if (fq >= nitems) return;
        uint8_t* st = lds + fbuf * STAGE + wave_s * 1024;      // uniform: the LDS address of a load goes through M0
#pragma unroll
        for (int i = 0; i < 4; i++) __builtin_amdgcn_raw_ptr_buffer_load_lds(desc_a, (lds_ptr_t)(st + i * 8192), 16, vo_a[i], fkt * 128, 0, 0);
#pragma unroll
        for (int i = 0; i < 2; i++) __builtin_amdgcn_raw_ptr_buffer_load_lds(desc_b, (lds_ptr_t)(st + (4 + i) * 8192), 16, vo_b[i], fkt * 128, 0, 0);
        if (!f_half) {
#pragma unroll
            for (int i = 2; i < 4; i++) __builtin_amdgcn_raw_ptr_buffer_load_lds(desc_b, (lds_ptr_t)(st + (4 + i) * 8192), 16, vo_b[i], fkt * 128, 0, 0);
        }
        fbuf ^= 1;
        if (++fkt == ksteps) {
            fkt = 0;
            if (++fq < nitems) set_fetch_item(fq);
        }
    };

    // the scales live in scalar registers across the K loops (as vector registers they were spilled, and the reloads in the
    // epilogue waited for the operand loads issued just before it)
    auto uniform = [](float v) { return __uint_as_float(__builtin_amdgcn_readfirstlane(__float_as_uint(v))); };
    const float inv_a = uniform(*ep.inv_a);
    float sc[4];
#pragma unroll
    for (int i = 0; i < 4; i++) sc[i] = uniform(ep.inv_b[i < ep.segs.nseg ? i : 0]);
    uint8_t* epi = lds + 2 * STAGE + wave_s * 4096;

    // Invariant at the top of every K-step: its own operands have landed (the barrier before it) and the loads of the step
    // after it are already in flight.  After the barrier that ends a step, its buffer is free and takes the loads of
    // the step after next; at the end of a tile those are the next tile's, and they travel while the tile is stored.
    set_fetch_item(0);
    fetch_next();
    dl_step_barrier();
    fetch_next();
    int buf = 0;
    auto tile = [&](int n0, auto half_tag) {
        constexpr bool HALF = decltype(half_tag)::value;
        v4f acc[4][8];
        dl_compute<HALF, true, A_FMT>(acc, lds + buf * STAGE, g);
        dl_step_barrier();
        buf ^= 1;
        for (int kt = 1; kt < ksteps; kt++) {
            // the loads into the buffer that the barrier has just freed go out behind this step's first fragment reads
            dl_compute<HALF, false, A_FMT>(acc, lds + buf * STAGE, g, fetch_next);
            dl_step_barrier();
            buf ^= 1;
        }
        fetch_next();
        // the last MFMAs must have left the pipeline before the accumulators are read
        asm volatile("s_nop 15\n\ts_nop 15" ::: "memory");
#pragma unroll
        for (int i = 0; i < 4; i++)
#pragma unroll
            for (int j = 0; j < (HALF ? 4 : 8); j++) asm volatile("" : "+a"(acc[i][j]));
        int m0_here = m0;
        asm volatile("" : "+s"(m0_here));          // keeps the store addresses of all tiles from being precomputed (and spilled)
        // the epilogue's lane geometry is worked out afresh (see set_fetch_item): values kept for it across the K loop were
        // spilled, and their reloads at this point waited for the next tile's operand loads that had just been issued
        int lane_e;
        asm volatile("v_mbcnt_lo_u32_b32 %0, -1, 0\n\tv_mbcnt_hi_u32_b32 %0, -1, %0" : "=v"(lane_e));
        DlGeom ge;
        ge.lane = lane_e, ge.wave = wave_s, ge.wm = wave_s / 2, ge.wn = wave_s % 2, ge.frow = lane_e & 15, ge.kb = lane_e >> 4;
        ge.sub = ge.gch = ge.rd_lo = ge.rd_hi = 0;
        dlp_epilogue<HALF, RELU2>(acc, epi, ep, inv_a, sc, ge, m0_here, n0, M, N);
    };
    for (int q = 0; q < nitems; q++) {
        int n0;
        bool half;
        item(q, n0, half);
        if (half) tile(n0, std::true_type{});
        else tile(n0, std::false_type{});
    }
}

static bool dlp_eligible(int M, int /*N*/, int K) {
    const int tiles_m = (M + 255) / 256;
    if (K % 128 != 0 || tiles_m % 8 != 0) return false;
    const int rx = tiles_m / 8;
    return rx >= 1 && rx <= 32 && (rx & (rx - 1)) == 0;
}

template <int A_FMT, int OUT_KIND>
static int launch_dl_as(const uint8_t* a, const uint8_t* b, const EpilogueArgs& ep, int M, int N, int K, bool persistent, hipStream_t s) {
    const int tiles_m = (M + 255) / 256, tiles_n = (N + 255) / 256;
    constexpr size_t STAGES = 2 * 512 * 128;
    if (persistent) {
        if (int rc = reserve_lds<gemm_dlp_kernel<A_FMT, OUT_KIND == 2>>(STAGES + 8 * 4096)) return rc;
        hipLaunchKernelGGL((gemm_dlp_kernel<A_FMT, OUT_KIND == 2>), dim3(256), dim3(512), STAGES + 8 * 4096, s, a, b, ep, M, N, K, tiles_m / 8, (N + 127) / 128);
        return 0;
    }
    auto launch = [&](auto ring, size_t lds_bytes) -> int {
        if (int rc = reserve_lds<gemm_dl_kernel<A_FMT, OUT_KIND, ring>>(lds_bytes)) return rc;
        hipLaunchKernelGGL((gemm_dl_kernel<A_FMT, OUT_KIND, ring>), dim3(tiles_m * tiles_n), dim3(512), lds_bytes, s, a, b, ep, M, N, K, tiles_m, tiles_n);
        return 0;
    };
    if constexpr (OUT_KIND == 0)
        if (!dl_two_stages(8, K)) return launch(std::true_type{}, dl_ring_lds<true, 8, 4>());
    return launch(std::false_type{}, STAGES);
}

// Blocks of 16 columns per wave (tile width 32 NJ, NJ = 4 .. 8) for a launch of 256-row tiles that is not persistent.  Measured at
// K = 1664 a round of tiles lasts about 6 + NJ units (the A side of a K-step, the launch and the epilogue cost the same at any width:
// 16.6 / 18.5 / 19.7 / 22.0 / 23.4 us for NJ = 4 .. 8 with 80 tiles) and up to a fifth longer when every CU has a tile (28.1 us with 240
// tiles of 256 x 256).  The full width is kept unless a narrower tile is at least 8 % cheaper by that count:
// 1792 x 4992: 140 tiles of 256 x 256, 24.1 us -> 224 of 256 x 160, 20.6 us; 1792 x 6656: 182 tiles, 25.4 -> 245 of 256 x 192, 22.2 us.
static double dl_cost(int nj, int M, int N, int cus, long* tiles_out) {
    const long tiles = (long)((M + 255) / 256) * ((N + 32 * nj - 1) / (32 * nj));
    if (tiles_out) *tiles_out = tiles;
    double cost = 0.0;
    for (long left = tiles; left > 0; left -= cus) cost += (6.0 + nj) * (1.0 + 0.2 * (double)(left < cus ? left : cus) / cus);
    return cost;
}
static int dl_pick_nj(int M, int N) {
    const int cus = cu_count();
    int best = 8;
    const double full = dl_cost(8, M, N, cus, nullptr);
    double best_cost = 0.92 * full;
    for (int nj = 7; nj >= 4; nj--) {
        const double c = dl_cost(nj, M, N, cus, nullptr);
        if (c < best_cost) best = nj, best_cost = c;
    }
    return best;
}
// whether some narrower tile gives the launch one round with at least 150 of 256 CUs busy (then the 256-row tiles beat the 128 x 128
// ones although the 256 x 256 tiles would leave most CUs idle: 1024 x 4992 x 1664 16.6 us against 18.4)
static bool dl_narrow_fills(int M, int N) {
    const int cus = cu_count();
    for (int nj = 4; nj <= 7; nj++) {
        long tiles;
        (void)dl_cost(nj, M, N, cus, &tiles);
        if (tiles <= cus && 256 * tiles >= 150L * cus) return true;
    }
    return false;
}
template <int NJ, int OUT_KIND, int A_FMT>
static int launch_dln_as(const uint8_t* a, const uint8_t* b, const EpilogueArgs& ep, int M, int N, int K, hipStream_t s) {
    const int tiles_m = (M + 255) / 256, tiles_n = (N + 32 * NJ - 1) / (32 * NJ);
    auto launch = [&](auto ring, size_t lds_bytes) -> int {
        if (int rc = reserve_lds<gemm_dln_kernel<NJ, OUT_KIND, A_FMT, ring>>(lds_bytes)) return rc;
        hipLaunchKernelGGL((gemm_dln_kernel<NJ, OUT_KIND, A_FMT, ring>), dim3(tiles_m * tiles_n), dim3(512), lds_bytes, s, a, b, ep, M, N, K, tiles_m, tiles_n);
        return 0;
    };
    if constexpr (OUT_KIND != 4)
        if (dl_two_stages(NJ, K)) return launch(std::false_type{}, 2 * (256 + 32 * NJ) * 128);
    return launch(std::true_type{}, dl_ring_lds<true, NJ, 4>());
}
template <int NJ>
static int launch_dln_nj(int a_fmt, const uint8_t* a, const uint8_t* b, const EpilogueArgs& ep, int M, int N, int K, hipStream_t s) {
    if (a_fmt == 1) return launch_dln_as<NJ, 0, 1>(a, b, ep, M, N, K, s);
    if (ep.out_kind == 4) return launch_dln_as<NJ, 4, 0>(a, b, ep, M, N, K, s);
    return ep.out_kind == 2 ? launch_dln_as<NJ, 2, 0>(a, b, ep, M, N, K, s) : launch_dln_as<NJ, 0, 0>(a, b, ep, M, N, K, s);
}
// bf16 or (e4m3 first operand only) relu^2 output, K a multiple of 128
static int launch_dln(int nj, int a_fmt, const uint8_t* a, const uint8_t* b, const EpilogueArgs& ep, int M, int N, int K, hipStream_t s) {
    NC_CHECK_ARG((long)M * K < (1L << 31) && (long)N * K < (1L << 31), "fp8_gemm: buffer-load kernels need M*K and N*K below 2^31");
    NC_CHECK_ARG(K % 128 == 0, "fp8_gemm: the direct-to-LDS kernels need K %% 128 == 0, got %d", K);
    NC_CHECK_ARG(ep.out_kind != 1, "fp8_gemm: the direct-to-LDS kernels write bf16 only");
    NC_CHECK_ARG(a_fmt == 0 || ep.out_kind == 0, "fp8_gemm: the relu^2 epilogue goes with an e4m3 first operand");
    switch (nj) {
        case 4: return launch_dln_nj<4>(a_fmt, a, b, ep, M, N, K, s);
        case 5: return launch_dln_nj<5>(a_fmt, a, b, ep, M, N, K, s);
        case 6: return launch_dln_nj<6>(a_fmt, a, b, ep, M, N, K, s);
        case 7: return launch_dln_nj<7>(a_fmt, a, b, ep, M, N, K, s);
    }
    NC_FAIL(-1, "fp8_gemm: tile widths of 128, 160, 192 and 224 columns only, not %d", 32 * nj);
}

template <int BM, int OUT_KIND, typename Rope = NoRope>
static int launch_dr_as(const uint8_t* a, const uint8_t* b, const EpilogueArgs& ep, int M, int N, int K, hipStream_t s, int splits = 1, Rope rope = Rope{}) {
    const int tiles_m = (M + BM - 1) / BM, tiles_n = (N + 127) / 128;
    const size_t lds_bytes = 4 * (size_t)(BM + 128) * 128;
    if (int rc = reserve_lds<gemm_dr_kernel<BM, OUT_KIND, Rope>>(lds_bytes)) return rc;
    hipLaunchKernelGGL((gemm_dr_kernel<BM, OUT_KIND, Rope>), dim3(tiles_m * tiles_n, splits), dim3(256), lds_bytes, s, a, b, ep, M, N, K, tiles_m, tiles_n, rope);
    return 0;
}
// e4m3 operands, bf16 or relu^2 output, K a multiple of 128
template <int BM>
static int launch_dr(const uint8_t* a, const uint8_t* b, const EpilogueArgs& ep, int M, int N, int K, hipStream_t s) {
    NC_CHECK_ARG((long)M * K < (1L << 31) && (long)N * K < (1L << 31), "fp8_gemm: buffer-load kernels need M*K and N*K below 2^31");
    NC_CHECK_ARG(K % 128 == 0, "fp8_gemm: the direct-to-LDS kernels need K %% 128 == 0, got %d", K);
    NC_CHECK_ARG(ep.out_kind != 1, "fp8_gemm: the direct-to-LDS kernels write bf16 only");
    if constexpr (BM < 128)
        if (ep.out_kind == 4) return launch_dr_as<BM, 4>(a, b, ep, M, N, K, s);      // (what pick_kernel takes)
    return ep.out_kind == 2 ? launch_dr_as<BM, 2>(a, b, ep, M, N, K, s) : launch_dr_as<BM, 0>(a, b, ep, M, N, K, s);
}

// the relu^2 epilogue is a variant of its own so that the plain kernels keep their register budget
template <int A_FMT>
static int launch_dl(const uint8_t* a, const uint8_t* b, const EpilogueArgs& ep, int M, int N, int K, bool persistent, hipStream_t s) {
    NC_CHECK_ARG((long)M * K < (1L << 31) && (long)N * K < (1L << 31), "fp8_gemm: buffer-load kernels need M*K and N*K below 2^31");
    NC_CHECK_ARG(K % 128 == 0, "fp8_gemm: the direct-to-LDS kernels need K %% 128 == 0, got %d", K);
    NC_CHECK_ARG(ep.out_kind != 1, "fp8_gemm: the direct-to-LDS kernels write bf16 only");
    if (persistent)
        NC_CHECK_ARG(dlp_eligible(M, N, K), "fp8_gemm: the persistent kernel needs M/256 (rounded up) to be 8, 16, ... 256 tile rows, got M=%d", M);
    if (A_FMT == 0 && ep.out_kind == 2) return launch_dl_as<0, 2>(a, b, ep, M, N, K, persistent, s);
    if (A_FMT == 0 && ep.out_kind == 4 && !persistent) return launch_dl_as<0, 4>(a, b, ep, M, N, K, false, s);
    NC_CHECK_ARG(ep.out_kind == 0, "fp8_gemm: the relu^2 epilogue goes with an e4m3 first operand");
    return launch_dl_as<A_FMT, 0>(a, b, ep, M, N, K, persistent, s);
}

// ------------------------------------------------------------------------------------------------
template <int BM, int BN>
static int launch_tile(const uint8_t* a, const uint8_t* b, const EpilogueArgs& ep, int M, int N, int K, hipStream_t s) {
    const int tiles_m = (M + BM - 1) / BM, tiles_n = (N + BN - 1) / BN;
    const size_t lds_bytes = 2 * (size_t)(BM + BN) * 128;
    if (int rc = reserve_lds<gemm_tile_kernel<BM, BN>>(lds_bytes)) return rc;
    hipLaunchKernelGGL((gemm_tile_kernel<BM, BN>), dim3(tiles_m * tiles_n), dim3(256), lds_bytes, s, a, b, ep, M, N, K, tiles_m, tiles_n);
    return 0;
}

// The kernel of a bf16, relu^2 or softcapped linear of e4m3 operands (the selectors of nc_launch_gemm).
static int pick_kernel(int M, int N, int K, int out_kind) {
    int which;
    if (M <= 128) which = 1;
    else if ((long)M * K >= (1L << 31) || (long)N * K >= (1L << 31)) which = 4;   // past the 32-bit buffer offsets
    else {
        const int cus = cu_count();
        const long t256 = (long)((M + 255) / 256) * ((N + 255) / 256);
        const long rounds = (t256 + cus - 1) / cus;
        const long t128 = (long)((M + 127) / 128) * ((N + 127) / 128);
        if (out_kind != 1 && K % 128 == 0 && (8 * t256 >= 5 * cus || t128 > 2 * cus || dl_narrow_fills(M, N))) {
            // 256x256 tiles fed straight into LDS whenever they occupy at least 5/8 of the CUs, or the 128x128 tiles, four times
            // as many, would not fit the chip in one round of two workgroups per CU (below that the small tiles fill the chip
            // better: 18 us against 22 for 1280 x 4992 x 1664, but 25 against 22.4 for 1792 rows); from two rounds of tiles on,
            // the persistent form, which neither rounds the last round up nor pays a prologue per tile
            which = (t256 >= 2 * cus && dlp_eligible(M, N, K)) ? 9 : 8;
            if (which == 8) {
                const int nj = dl_pick_nj(M, N);
                if (nj < 8) which = 8 + nj;           // 12 .. 15
            }
        } else {
            // 256x256 tiles move half the bytes per flop through L2 and LDS but run one workgroup per CU: take them
            // when their count fills whole rounds of the CUs well, else the 128x128 tiles (two workgroups per CU)
            which = (M >= 1024 && N >= 512 && 10 * t256 >= 8 * rounds * cus && rounds <= 2) ? 7 : 5;
            // a prompt of a few hundred to two thousand rows against a narrow weight leaves CUs without a 128x128 tile, and each
            // tile's K loop is one dependent step after the other: lower tiles put a workgroup on more CUs with less MFMA work per
            // step, as long as they still fit one round of one workgroup per CU (512..1024 rows x 1664 columns with 64-row tiles:
            // 8 us against 10.7 at K = 1664, 21 against 31 at K = 6656; 1792 rows with 96-row tiles: 10.0 / 11.5 and 27.9 / 30.5; the same for
            // the relu^2 linear where it has that few, us of 128-row / 64-row tiles with the clearing of its amax word: 170 x 4096 x 1024 11.6 / 9.3,
            // 200 x 6656 x 1664 14.4 / 12.0, 1000 x 2048 x 512 10.9 / 10.2, 1000 x 1100 x 144 10.7 / 8.1; of 128-row / 96-row tiles: 500 x 5120 x 1280
            // 13.9 / 13.0, 700 x 4096 x 1024 13.7 / 12.6, x 1008 13.9 / 12.8)
            if (which == 5) {
                const long tn = (N + 127) / 128;
                if ((long)((M + 63) / 64) * tn <= cus) which = 10;
                else if ((long)((M + 95) / 96) * tn <= cus) which = 11;
                // the same tiles fed straight into a ring of four LDS stages where K allows it: three K-steps of operands on their
                // way instead of two and no ds_write phase (1792 x 1664 x 6656: 27.5 -> 21.3 us, 1000 rows: 21.9 -> 17.1 us)
                if (which >= 10 && K % 128 == 0 && out_kind != 1) which += 6;
            }
        }
    }
    return which;
}

int nc_launch_gemm(const uint8_t* a, const uint8_t* b, const float* inv_a, const float* inv_b, NcGemmSegs segs,
                   void* out, int out_kind, float softcap, int M, int N, int K, int ldc, int force_kernel, void* workspace,
                   size_t workspace_bytes, hipStream_t s, int a_fmt, uint32_t* out_amax) {
    NC_CHECK_ARG(a && b && inv_a && inv_b && out, "fp8_gemm: null pointer");
    NC_CHECK_ARG(M >= 0 && N > 0 && K > 0, "fp8_gemm: bad shape M=%d N=%d K=%d", M, N, K);
    NC_CHECK_ARG(K % 16 == 0, "fp8_gemm: K=%d must be a multiple of 16", K);
    NC_CHECK_ARG(ldc >= N, "fp8_gemm: ldc=%d < N=%d", ldc, N);
    NC_CHECK_ARG(((uintptr_t)a & 15) == 0 && ((uintptr_t)b & 15) == 0, "fp8_gemm: operands must be 16-byte aligned");
    NC_CHECK_ARG(out_kind >= 0 && out_kind <= 2, "fp8_gemm: out_kind must be 0 (bf16), 1 (softcapped fp32) or 2 (bf16 relu^2 + amax)");
    NC_CHECK_ARG(out_kind != 2 || (out_amax && M > 128 && (long)M * K < (1L << 31) && (long)N * K < (1L << 31) && (force_kernel == 0 || force_kernel >= 5)),
                 "fp8_gemm: the relu^2 epilogue needs an amax word, M > 128, operands below 2 GiB and a buffer-load kernel");
    NC_CHECK_ARG(segs.nseg >= 1 && segs.nseg <= 4, "fp8_gemm: 1..4 column segments supported, got %d", segs.nseg);
    for (int i = 0; i < segs.nseg; i++) {
        NC_CHECK_ARG(segs.end[i] % 4 == 0 || segs.end[i] == N, "fp8_gemm: segment end %d must be a multiple of 4", segs.end[i]);
        NC_CHECK_ARG(i == 0 || segs.end[i] > segs.end[i - 1], "fp8_gemm: segment ends must increase");
    }
    NC_CHECK_ARG(segs.end[segs.nseg - 1] == N, "fp8_gemm: last segment must end at N");
    if (out_kind != 1)
        NC_CHECK_ARG(((uintptr_t)out & 7) == 0 && ldc % 4 == 0, "fp8_gemm: bf16 output needs 8-byte alignment and ldc %% 4 == 0");
    NC_CHECK_ARG(a_fmt == 0 || a_fmt == 1, "fp8_gemm: the format of a must be 0 (e4m3fn) or 1 (e5m2)");
    if (M == 0) return 0;
    EpilogueArgs ep{inv_a, inv_b, segs, out, out_kind, softcap, ldc, out_amax, NcMeeting{}, nullptr, nullptr};
    if (a_fmt == 1) {
        // gradient operand (the backward GEMMs): bf16 output through the 128x128 buffer-load tile or the 256x256 direct-to-LDS tiles
        NC_CHECK_ARG(out_kind == 0, "fp8_gemm: an e5m2 operand goes with bf16 output");
        NC_CHECK_ARG((long)M * K < (1L << 31) && (long)N * K < (1L << 31), "fp8_gemm: e5m2 operands need M*K and N*K below 2^31");
        int which = force_kernel;
        if (which == 0) {
            const int cus = cu_count();
            const long t256 = (long)((M + 255) / 256) * ((N + 255) / 256);
            which = (K % 128 == 0 && (8 * t256 >= 5 * cus || dl_narrow_fills(M, N))) ? ((t256 >= 2 * cus && dlp_eligible(M, N, K)) ? 9 : 8) : 5;
            if (which == 8) {
                const int nj = dl_pick_nj(M, N);
                if (nj < 8) which = 8 + nj;               // 12 .. 15: the narrower 256-row tiles
            }
        }
        NC_CHECK_ARG(which == 5 || which == 8 || which == 9 || (which >= 12 && which <= 15),
                     "fp8_gemm: kernels 5, 8, 9 and 12..15 take an e5m2 operand, not %d", force_kernel);
        NcProfScope prof(1, 2.0 * M * N * K, s, ((int64_t)N << 32) | (uint32_t)K);
        int rc = which == 5 ? launch_bl<128, 128, 2, 2, true, 1>(a, b, ep, M, N, K, s)
                            : (which >= 12 ? launch_dln(which - 8, 1, a, b, ep, M, N, K, s) : launch_dl<1>(a, b, ep, M, N, K, which == 9, s));
        if (rc) return rc;
        NC_CHECK_LAUNCH("fp8_gemm");
        return 0;
    }

    // force_kernel: 0 auto, 1 small-M, 4 plain-load tile 128x128, 5/6/7 buffer-load tiles 128x128 / 256x128 / 256x256,
    // 8 direct-to-LDS 256x256 tile by tile, 9 the same persistent, 10 / 11 buffer-load tiles 64x128 / 96x128,
    // 12 .. 15 direct-to-LDS tiles of 256 x 128 / 160 / 192 / 224 tile by tile, 16 / 17 / 18 direct-to-LDS tiles of 64 / 96 / 128 x 128
    // with four stages
    const int which = force_kernel ? force_kernel : pick_kernel(M, N, K, out_kind);
    int rc = 0;
    if (which != 1) NC_CHECK_ARG(which >= 4 && which <= 18, "fp8_gemm: unknown kernel selector %d", force_kernel);
    NcProfScope prof(which == 1 ? -1 : 1, 2.0 * M * N * K, s, ((int64_t)N << 32) | (uint32_t)K);
    if (which == 1) {
        NC_CHECK_ARG(M <= 128, "fp8_gemm: the small-M kernel needs M <= 128, got %d", M);
        // split-K when the caller brought room for the partial sums, finished by a second small kernel
        int ks = nc_gemm_decode_splits(N, K);
        if (ks > 1 && (!workspace || workspace_bytes < (size_t)ks * M * N * sizeof(float))) ks = 1;
        int used = 1;
        rc = nc_launch_gemm_decode(a, 0, nullptr, inv_a, b, inv_b, segs, out, out_kind, softcap, nullptr, M, N, K, ldc, (float*)workspace,
                                   workspace_bytes, ks, &used, s);
        if (rc) return rc;
        if (used > 1)
            return nc_launch_finish_partials((const float*)workspace, used, nullptr, inv_a, inv_b, segs, out, out_kind, softcap, nullptr, M,
                                             N, ldc, s);
        return 0;
    } else if (which == 4) rc = launch_tile<128, 128>(a, b, ep, M, N, K, s);
    else if (which == 5) rc = launch_bl<128, 128, 2, 2, true>(a, b, ep, M, N, K, s);
    else if (which == 6) rc = launch_bl<256, 128, 4, 2, false>(a, b, ep, M, N, K, s);
    else if (which == 7) rc = launch_bl<256, 256, 4, 2, false>(a, b, ep, M, N, K, s);
    else if (which == 8) rc = launch_dl<0>(a, b, ep, M, N, K, false, s);
    else if (which == 9) rc = launch_dl<0>(a, b, ep, M, N, K, true, s);
    else if (which == 10) rc = launch_bl<64, 128, 2, 2, true>(a, b, ep, M, N, K, s);
    else if (which == 11) rc = launch_bl<96, 128, 2, 2, true>(a, b, ep, M, N, K, s);
    else if (which == 16) rc = launch_dr<64>(a, b, ep, M, N, K, s);
    else if (which == 17) rc = launch_dr<96>(a, b, ep, M, N, K, s);
    else if (which == 18) rc = launch_dr<128>(a, b, ep, M, N, K, s);
    else if (which >= 12) rc = launch_dln(which - 8, 0, a, b, ep, M, N, K, s);
    else NC_FAIL(-1, "fp8_gemm: unknown kernel selector %d", force_kernel);
    if (rc) return rc;
    NC_CHECK_LAUNCH("fp8_gemm");
    return 0;
}

// The tiles of the q|k|v linear that finish its heads: those of 64 or 96 x 128 where pick_kernel takes them (16, 17), otherwise 64 w x 128 (returned as
// 100 + w); 0: none.  Two workgroups of the 128-row tile fit a CU (80 KB of LDS each), one of the higher ones, whose epilogue nothing overlaps.  So the low tile
// is taken in one round of one or two to a CU and wherever the others need a second round; a single round of higher tiles beats it (i) at 192 rows, (ii) where the
// low ones would go into a second round.  us, 128-row tiles / the best of the others (w) / a linear and a rotary launch: 1300 x 4992 x 1664 19.5 / 21.4 (4) / 25.8,
// 1792 x 29.4 / 25.3 (5) / 31.8, 2048 x 29.5 / 28.8 (6) / 33.9, 3072 x 35.6 / 41.3 (4) / 44.3, 4096 x 46.9 / 50.1 (5) / 61.4, 6144 x 67.0 / 80.6 (4) / 81.6; few key heads,
// 1300 x 3072 x 1536 17.0 / 16.8 (3) / 24.7, 2048 x 18.1 / 20.5 (4) / 23.7, 3072 x 28.6 / 25.2 (5) / 32.0, 4096 x 29.6 / 38.5 (4) / 37.6, 8192 x 1536 x 768 22.1 / 28.8 (4) / 33.4.
static int rope_tiles(int M, int N, int K) {
    if (M <= 128 || N % 128 != 0 || K % 128 != 0 || (long)M * K >= (1L << 31) || (long)N * K >= (1L << 31)) return 0;
    const int which = pick_kernel(M, N, K, 0);
    if (which == 16 || which == 17) return which;
    const long cus = cu_count(), columns = N / 128, low = (M + 127) / 128 * columns;
    if (low <= cus) return 102;
    for (int w = 3; w <= 6; w++)
        if ((M + 64 * w - 1) / (64 * w) * columns <= cus) return w == 3 || low > 2 * cus ? 100 + w : 102;
    return 102;
}
template <int WTM>
static int launch_gemm_rope(const uint8_t* a, const uint8_t* b, const EpilogueArgs& ep, const RopeArgs& rope, int M, int N, int K, hipStream_t s) {
    const int tiles_m = (M + 64 * WTM - 1) / (64 * WTM), tiles_n = N / 128;
    const size_t lds_bytes = dl_ring_lds<false, WTM, 2>();
    if (int rc = reserve_lds<gemm_rope_kernel<WTM>>(lds_bytes)) return rc;
    hipLaunchKernelGGL(gemm_rope_kernel<WTM>, dim3(tiles_m * tiles_n), dim3(512), lds_bytes, s, a, b, ep, rope, M, N, K, tiles_m, tiles_n);
    return 0;
}
// 1: not a shape or an alignment of this launch
int nc_launch_gemm_qkv_rope(const uint8_t* a, const uint8_t* b, const float* inv_a, const float* inv_b, NcGemmSegs segs, const NcRopeSrc& src, const NcRopeDst& dst,
                            int M, int K, hipStream_t s, int force_kernel) {
    NC_CHECK_ARG(a && b && inv_a && inv_b, "qkv_rope: null pointer");
    NC_CHECK_ARG(dst.T > 0 && dst.H > 0 && dst.Hkv > 0 && dst.H % dst.Hkv == 0 && dst.Tmax > 0, "qkv_rope: bad shape");
    const int N = (dst.H + 2 * dst.Hkv) * 128, fits = rope_tiles(M, N, K), which = fits && force_kernel ? force_kernel : fits;
    NC_CHECK_ARG(!which || which == 16 || which == 17 || (which >= 102 && which <= 106), "qkv_rope: unknown kernel selector %d", force_kernel);
    if (!which || M % dst.T != 0 || !rope_vec_aligned(src, dst)) return 1;
    NC_CHECK_ARG((((uintptr_t)a | (uintptr_t)b) & 15) == 0, "qkv_rope: operands must be 16-byte aligned");
    NC_CHECK_ARG(src.cos_t && src.sin_t && src.rope_len > 0 && dst.cache_seqlens && dst.k_cache && dst.v_cache && dst.q_out && (!src.ve_table || (src.ve_gate_w && src.xn && src.idx && src.ld_xn >= 12)),
                 "qkv_rope: null pointer");
    NC_CHECK_ARG(segs.nseg >= 1 && segs.nseg <= 4 && segs.end[segs.nseg - 1] == N, "qkv_rope: segments must end at %d columns", N);
    for (int i = 0; i < segs.nseg; i++) NC_CHECK_ARG(segs.end[i] % 128 == 0, "qkv_rope: segments must be whole heads");
    EpilogueArgs ep{};
    ep.inv_a = inv_a, ep.inv_b = inv_b, ep.segs = segs;
    const RopeArgs rope{src, dst};
    NcProfScope prof(1, 2.0 * M * N * K, s, ((int64_t)N << 32) | (uint32_t)K);
    const int rc = which == 16 ? launch_dr_as<64, 5, RopeArgs>(a, b, ep, M, N, K, s, 1, rope)
                   : which == 17 ? launch_dr_as<96, 5, RopeArgs>(a, b, ep, M, N, K, s, 1, rope)
                   : which == 102 ? launch_gemm_rope<2>(a, b, ep, rope, M, N, K, s)
                   : which == 103 ? launch_gemm_rope<3>(a, b, ep, rope, M, N, K, s)
                   : which == 104 ? launch_gemm_rope<4>(a, b, ep, rope, M, N, K, s)
                   : which == 105 ? launch_gemm_rope<5>(a, b, ep, rope, M, N, K, s) : launch_gemm_rope<6>(a, b, ep, rope, M, N, K, s);
    if (rc) return rc;
    NC_CHECK_LAUNCH("qkv_rope");
    return 0;
}

// The kernel that leaves relu^2 of a linear as e4m3 (out_kind 4), or 0: the tiles of pick_kernel where they are one round of one workgroup per CU (each
// takes more than half of a CU's LDS), so that all of them can hold their tile until everybody's amax is known.
int nc_gemm_relu2_e4m3_kernel(int M, int N, int K) {
    if (M <= 128 || N % 16 != 0 || K % 128 != 0 || (long)M * K >= (1L << 31) || (long)N * K >= (1L << 31)) return 0;
    const int which = pick_kernel(M, N, K, 2);
    const int bm = which == 16 ? 64 : which == 17 ? 96 : 256, bn = which >= 16 ? 128 : which >= 12 ? 32 * (which - 8) : 256;
    if (which != 8 && (which < 12 || which > 17)) return 0;
    const long wgs = (long)((M + bm - 1) / bm) * ((N + bn - 1) / bn);
    return wgs <= nc_meeting_wgs() ? which : 0;
}

int nc_launch_gemm_relu2_e4m3(const uint8_t* a, const uint8_t* b, const float* inv_a, const float* inv_b, uint8_t* out, float* inv_out, uint32_t* out_amax,
                              bf16_t* left, NcMeeting meeting, int M, int N, int K, hipStream_t s) {
    NC_CHECK_ARG(a && b && inv_a && inv_b && out && inv_out && left && meeting.words, "fp8_gemm_relu2_e4m3: null pointer");
    NC_CHECK_ARG((((uintptr_t)a | (uintptr_t)b | (uintptr_t)out | (uintptr_t)left) & 15) == 0, "fp8_gemm_relu2_e4m3: operands must be 16-byte aligned");
    const int which = nc_gemm_relu2_e4m3_kernel(M, N, K);
    NC_CHECK_ARG(which != 0, "fp8_gemm_relu2_e4m3: M=%d N=%d K=%d is not one round of tiles", M, N, K);
    EpilogueArgs ep{inv_a, inv_b, NcGemmSegs{1, {N, 0, 0, 0}}, out, 4, 0.f, N, out_amax, meeting, left, inv_out};
    NcProfScope prof(1, 2.0 * M * N * K, s, ((int64_t)N << 32) | (uint32_t)K);
    const int rc = which == 8 ? launch_dl<0>(a, b, ep, M, N, K, false, s)
                   : which == 16 ? launch_dr<64>(a, b, ep, M, N, K, s)
                   : which == 17 ? launch_dr<96>(a, b, ep, M, N, K, s) : launch_dln(which - 8, 0, a, b, ep, M, N, K, s);
    if (rc) return rc;
    NC_CHECK_LAUNCH("fp8_gemm_relu2_e4m3");
    return 0;
}

// Shares of K that a linear of more than 128 rows is cut into when its consumer adds partial sums: as many as give every CU a workgroup of 64 x 128
// outputs, of four steps at least (what the ring of stages holds; of eight 0 to 2 % slower or faster, of two the same).  A prompt of a few hundred
// tokens leaves most CUs without a tile of a narrow weight otherwise, and K = 4 E is one chain of 32 to 52 steps of half a microsecond (170 rows,
// 1024 x 4096: 24 tiles, 17 us).  us a prompt, in one piece / in shares: depth 16, 170 tokens 1208 / 1045, depth 20, 250 1776 / 1492, 500 1965 / 1756,
// depth 26, 200 2257 / 1968, 400 2624 / 2418, depth 12, 1000 1096 / 1054.  From more than cus / 2 tiles on there is nothing to fill.  (The q|k|v linear
// has three times the tiles and a consumer that reads fp32 sums more slowly than bf16: 1045 / 1087.)  Nor do shares pay for up to 768 columns once the
// row pass would take a wave to a row, which it does for bf16 rows only: the chain saved is 4 to 12 steps there (one piece / shares: depth 4, 800 rows
// 296 / 320, 1792 334 / 357, depth 6, 1792 524 / 541, depth 8, 1100 648 / 676, depth 12, 1300 1122 / 1138; depth 14, 1100 1317 / 1317, depth 16, 1024
// 1551 / 1533).
int nc_gemm_prompt_splits(int M, int N, int K) {
    if (M <= 128 || K % 128 != 0 || N % 8 != 0 || N > 8192 || (long)M * K >= (1L << 31) || (long)N * K >= (1L << 31)) return 1;
    if (N <= 768 && nc_mix_norm_wave_rows(M, N)) return 1;
    const long tiles = (long)((M + 63) / 64) * ((N + 127) / 128);
    long s = cu_count() / tiles;
    if (s > 8) s = 8;
    if (s > K / 512) s = K / 512;
    return s < 1 ? 1 : (int)s;
}

int nc_launch_gemm_partials(const uint8_t* a, const uint8_t* b, float* parts, size_t part_bytes, int splits, int M, int N, int K, hipStream_t s) {
    NC_CHECK_ARG(a && b && parts && splits > 1 && splits <= K / 128 && splits <= nc_gemm_prompt_splits(M, N, K), "fp8_gemm: %d shares of K=%d", splits, K);
    NC_CHECK_ARG((((uintptr_t)a | (uintptr_t)b | (uintptr_t)parts) & 15) == 0 && part_bytes >= (size_t)splits * M * N * sizeof(float),
                 "fp8_gemm: %d shares need %zu bytes of 16-byte aligned room", splits, (size_t)splits * M * N * sizeof(float));
    EpilogueArgs ep{};
    ep.out = parts;
    NcProfScope prof(1, 2.0 * M * N * K, s, ((int64_t)N << 32) | (uint32_t)K);
    if (const int rc = launch_dr_as<64, 3>(a, b, ep, M, N, K, s, splits)) return rc;
    NC_CHECK_LAUNCH("fp8_gemm");
    return 0;
}
