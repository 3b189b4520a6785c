// Few-row GEMM (2 to 64 rows): y[M, N] = x[M, K] . deq(W[N, K])^T in one launch, x read as it is.
// For the calls of batched decoding that the tiled kernels serve badly (the reference's
// matmul_t_q*_tiled range, src/lib/webgpu/shaders.ts:120-168, 425-527): few rows per weight, so the weight
// stream and the latency of its loads bound them, not the matrix cores.
//
// A block owns 32 CW columns; its waves are CW column waves x KW k waves. K is cut into pieces of 256; k
// wave `kw` takes every KW-th piece of the block's range. For a piece a wave holds the codes of its 32
// columns in registers (128 bytes of each q4 row: whole lines) and their scales, loaded one piece ahead,
// and the x rows of the piece in LDS as f16, each row scaled by a power of two of its own largest
// magnitude in that piece (xprep_up: no launch before this one has to see the whole row). The piece's
// product, eight slices of 16 k per 128 as in the tiled GEMM, is multiplied by that scale and added up in
// f32. The k waves' sums meet in LDS in a fixed order. With gridDim.y > 1 every block covers a slice of
// the pieces and writes its partial tile to `part` for brik_splitk_reduce.
//
// What bounds it: the instructions of one or two waves per SIMD. A piece of 32 columns is 208 to dequantize and
// about 50 per row pair to stage (8 rows: 520 in all, 2 us a piece), beside one round trip for the weights;
// loading W two or three pieces ahead, or holding the kernel to 128 registers for more waves, measured
// slower. So x is converted once per block of columns, the 8- and 16-row tiles split K over four waves of a
// block before splitting it over blocks (no partial tiles to sum), and 32 and 64 rows share the staged x
// over 128 columns. It took the place of a staging launch, a split-K launch (2-byte scale loads, 32 rows at
// a time) and the sum: q4 8 x 2560 x 9728 16.1 -> 10.8 us, q8 33 x 9728 x 2560 34.8 -> 18.6 us,
// q4 16 x 9728 x 2560 27.4 -> 12.6 us, q4 16 x 896 x 4864 9.8 -> 6.1 us.
// f16 weights (FMT_F16, K % 8 == 0) run the same pieces with no scales, both operands in natural k order.
#include "common.h"

namespace {

constexpr int FEW_K = 256;           // k of one piece: two steps of 128
constexpr int FEW_G = FEW_K / BRIK_GROUP;

// One wave's weights of a piece: codes of two steps (WCodes mapping), and 16 bytes of scales (lanes 0-31)
// or mins (lanes 32-63): the 8 groups of column lane & 31.
template <int FMT>
struct FewW {
    WCodes<FMT> c[2];
    u32x4_t s;
};

template <int FMT>
struct FewPlanes {
    brsrc_t r0, r1, rs;              // rs: scales on lanes 0-31, mins on lanes 32-63 is one resource each
    brsrc_t rm;
    uint32_t colg;                   // flat group index of this lane's column, group 0
    uint32_t glast;                  // last flat group at which 8 groups end inside the plane
    int G, h;
    uint32_t col;                    // f16: byte offset of this lane's column (and k half) in W
    int K;
};

template <int FMT>
__device__ __forceinline__ void few_load(FewW<FMT>& f, const FewPlanes<FMT>& p, int q)
{
    if constexpr (FMT == FMT_F16) {
        // slice s of step t: halves k = 256 q + 128 t + 16 s + 8 h ..; past K an offset past the buffer's end
        // (zeros, so an infinite weight of the next row cannot meet x's zero padding)
        const bool whole = FEW_K * (q + 1) <= p.K;   // uniform
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
            for (int s = 0; s < 8; ++s) {
                const int k = 128 * t + 16 * s;
                const uint32_t off = whole || FEW_K * q + k + 8 * p.h < p.K ? p.col + (uint32_t)(FEW_K * q + k) * 2u : 0xFFFFFF00u;
                const u32x4_t v = __builtin_amdgcn_raw_buffer_load_b128(p.r0, off, 0, 0);
#pragma unroll
                for (int j = 0; j < 4; ++j) f.c[t].w[4 * s + j] = v[j];
            }
        return;
    }
    const uint32_t start = min(p.colg + (uint32_t)(FEW_G * q), p.glast) * 2u;
    f.s = p.h && FMT != FMT_Q8 ? __builtin_bit_cast(u32x4_t, __builtin_amdgcn_raw_buffer_load_b128(p.rm, start, 0, 0))
                               : __builtin_bit_cast(u32x4_t, __builtin_amdgcn_raw_buffer_load_b128(p.rs, start, 0, 0));
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int e = 0; e < 2; ++e) {
            // past the row's end: codes of the next row, or zeros past the plane; their scales are masked
            const uint32_t g = p.colg + (uint32_t)(FEW_G * q + 2 * p.h) + (uint32_t)(4 * t + e);
            WCodes<FMT>& w = f.c[t];
            if constexpr (FMT == FMT_Q4) {
                const u32x4_t v = __builtin_amdgcn_raw_buffer_load_b128(p.r0, g * 16, 0, 0);
#pragma unroll
                for (int j = 0; j < 4; ++j) w.w[4 * e + j] = v[j];
            } else if constexpr (FMT == FMT_Q8) {
#pragma unroll
                for (int k = 0; k < 2; ++k) {
                    const u32x4_t v = __builtin_amdgcn_raw_buffer_load_b128(p.r0, g * 32 + 16 * k, 0, 0);
#pragma unroll
                    for (int j = 0; j < 4; ++j) w.w[8 * e + 4 * k + j] = v[j];
                }
            } else {
                const u32x2_t v = __builtin_amdgcn_raw_buffer_load_b64(p.r0, g * 8, 0, 0);
                w.w[2 * e] = v.x;
                w.w[2 * e + 1] = v.y;
                w.w[4 + e] = __builtin_amdgcn_raw_buffer_load_b32(p.r1, g * 4, 0, 0);
            }
        }
}

// Largest magnitude of 8 values. v_max3 of magnitudes without the quieting that fmaxf asks for: a row with
// a NaN has no finite output, so which scale it takes does not matter.
__device__ __forceinline__ float few_absmax8(f32x4_t a, f32x4_t b)
{
    float m, n;
    asm("v_max3_f32 %0, |%1|, |%2|, |%3|" : "=v"(m) : "v"(a.x), "v"(a.y), "v"(a.z));
    asm("v_max3_f32 %0, |%1|, |%2|, |%3|" : "=v"(n) : "v"(a.w), "v"(b.x), "v"(b.y));
    asm("v_max3_f32 %0, |%1|, |%2|, %0" : "+v"(m) : "v"(b.z), "v"(b.w));
    asm("v_max_f32 %0, %0, %1" : "+v"(m) : "v"(n));
    return m;
}

// max(v, v of the lane a DPP control names)
template <int CTRL>
__device__ __forceinline__ float dpp_max(float v)
{
    const int o = __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, v), CTRL, 0xF, 0xF, false);
    float r;
    asm("v_max_f32 %0, %1, %2" : "=v"(r) : "v"(v), "v"(o));
    return r;
}

// Maximum over the 32 lanes of a half wave.
__device__ __forceinline__ float half_max(float v)
{
    v = dpp_max<DPP_QUAD_1032>(v);
    v = dpp_max<DPP_QUAD_2301>(v);
    v = dpp_max<DPP_ROW_ROR4>(v);
    v = dpp_max<DPP_ROW_ROR8>(v);
    const float o = __shfl_xor(v, 16);
    asm("v_max_f32 %0, %0, %1" : "+v"(v) : "v"(o));
    return v;
}

// Orders a wave's LDS writes before its own later reads of what other lanes wrote (a wave's LDS operations
// complete in issue order, so this only binds the compiler).
__device__ __forceinline__ void wave_lds_fence()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront", "local");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront", "local");
}

// XR: rows of x held in LDS (M <= XR); CW x KW waves. MB row blocks of 32 (the last may be half used).
template <int FMT, int XR, int CW, int KW, int D>
__device__ __forceinline__ void few_body(const float* __restrict__ x, const uint8_t* __restrict__ p0,
                                         const uint8_t* __restrict__ p1, const uint16_t* __restrict__ sc,
                                         const uint16_t* __restrict__ mn, float* __restrict__ y,
                                         float* __restrict__ part, int M, int K, int N, int qps)
{
    constexpr int MB = (XR + 31) / 32, NB = CW > 1 ? 2 : 1, NT = 64 * CW * KW;
    // one piece of x: [step][row][256 bytes + 16]; the pad puts the 16 rows of a read phase on 16 different
    // bank groups, so every fragment read is one address and an immediate offset
    constexpr int XROWP = 272, XB = 2 * XR * XROWP;
    constexpr int RP = XR / (2 * CW);                // row pairs a wave stages
    constexpr int XBYTES = KW * NB * XB, RED = KW > 1 ? KW * CW * MB * 4096 : 0;
    constexpr int MAIN = XBYTES > RED ? XBYTES : RED;
    __shared__ __attribute__((aligned(16))) unsigned char smem[MAIN + KW * NB * XR * 4 + CW * KW * 1024];

    const int tid = (int)threadIdx.x, lane = tid & 63, h = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), cw = wave % CW, kw = wave / CW;
    const int G = K / BRIK_GROUP, nq = (K + FEW_K - 1) / FEW_K;
    const int KS = (int)gridDim.y, slice = (int)blockIdx.y;
    const int q0 = slice * qps, q1 = min(q0 + qps, nq);        // q0 < nq: the host sizes gridDim.y so
    const int iters = (q1 - q0 + KW - 1) / KW;
    const int n0 = ((int)blockIdx.x * CW + cw) * 32, ncol = n0 + (lane & 31);

    const size_t wel = (size_t)N * K;
    FewPlanes<FMT> pl;
    if constexpr (FMT == FMT_F16) {
        pl.r0 = make_rsrc(p0, (uint32_t)(wel * 2));
    } else if constexpr (FMT == FMT_Q8) {
        pl.r0 = make_rsrc(p0, (uint32_t)wel);
    } else if constexpr (FMT == FMT_Q4) {
        pl.r0 = make_rsrc(p0, (uint32_t)(wel / 2));
    } else {
        pl.r0 = make_rsrc(p0, (uint32_t)(wel / 4));
        pl.r1 = make_rsrc(p1, (uint32_t)(wel / 8));
    }
    const uint32_t groups = (uint32_t)((size_t)N * G);
    if constexpr (FMT != FMT_F16) pl.rs = make_rsrc(sc, groups * 2);
    if constexpr (FMT == FMT_Q4 || FMT == FMT_Q3) pl.rm = make_rsrc(mn, groups * 2);
    pl.colg = (uint32_t)min(ncol, N - 1) * (uint32_t)G;
    pl.glast = groups - FEW_G;
    pl.G = G;
    pl.h = h;
    pl.col = (uint32_t)min(ncol, N - 1) * (uint32_t)K * 2u + 16u * (uint32_t)h;
    pl.K = K;

    unsigned char* const xb0 = smem + kw * NB * XB;
    float* const rs0 = reinterpret_cast<float*>(smem + MAIN) + kw * NB * XR;
    unsigned char* const sb = smem + MAIN + KW * NB * XR * 4 + wave * 1024;

    // x of a piece: this wave's row pairs (row 2 (RP cw + i) + (lane >> 5), 8 floats per lane); rows past M
    // lie past the buffer's end, and so does the offset given to lanes past K: both read zeros
    const brsrc_t rx = make_rsrc(x, (uint32_t)((size_t)M * K * 4));
    const uint32_t xoff = (uint32_t)((2 * RP * cw + h) * K + 8 * (lane & 31)) * 4u;
    f32x4_t xa[RP], xc[RP];
    auto load_x = [&](int q) {
        const uint32_t off = FEW_K * q + 8 * (lane & 31) < K ? xoff + (uint32_t)(FEW_K * 4 * q) : 0xFFFFFF00u;
#pragma unroll
        for (int i = 0; i < RP; ++i) {
            xa[i] = __builtin_bit_cast(f32x4_t, __builtin_amdgcn_raw_buffer_load_b128(rx, off, 8 * i * K, 0));
            xc[i] = __builtin_bit_cast(f32x4_t, __builtin_amdgcn_raw_buffer_load_b128(rx, off + 16, 8 * i * K, 0));
        }
    };
    auto store_x = [&](int buf) {
        unsigned char* const xb = xb0 + buf * XB + ((lane & 31) >> 4) * (XR * XROWP) + (lane & 15) * 16;
#pragma unroll
        for (int i = 0; i < RP; ++i) {
            const int m = 2 * (RP * cw + i) + h;
            if (2 * (RP * cw + i) >= M) break;       // uniform
            float down;
            const float up = xprep_up(half_max(few_absmax8(xa[i], xc[i])), down);
            if ((lane & 31) == 0) rs0[buf * XR + m] = down;
            *(half8_t*)(xb + m * XROWP) = to_h8_order<FMT == FMT_F16>(xa[i], xc[i], up);
        }
    };

    floatx16_t tot[MB];
#pragma unroll
    for (int b = 0; b < MB; ++b)
#pragma unroll
        for (int r = 0; r < 16; ++r) tot[b][r] = 0.f;
    int arow[MB];                                    // LDS byte offset of this lane's A row and k half
#pragma unroll
    for (int b = 0; b < MB; ++b) arow[b] = min(32 * b + (lane & 31), M - 1) * XROWP + (FMT == FMT_F16 ? 16 : 128) * h;
    const DeqConst dk = DeqConst::make();

    // x before W: loads complete in order, so the rows are converted while the weights are on their way
    // a k wave without a piece left multiplies zeros: its scales are masked below, f16 weights read as zeros
    auto piece = [&](int q) { return FMT == FMT_F16 ? (q < q1 ? q : nq) : min(q, nq - 1); };
    FewW<FMT> wq[D];
    load_x(q0 + kw < q1 ? q0 + kw : nq);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int d = 0; d < D; ++d) few_load(wq[d], pl, piece(q0 + d * KW + kw));
    __builtin_amdgcn_sched_barrier(0);
    store_x(0);
    for (int it0 = 0; it0 < iters; it0 += D)
#pragma unroll
    for (int d = 0; d < D; ++d) {
        const int it = it0 + d;
        if (it >= iters) break;                      // uniform over the block
        FewW<FMT>& w = wq[d];
        const int q = q0 + it * KW + kw, qn = q + KW, buf = NB == 2 ? it & 1 : 0;
        if constexpr (CW > 1) __syncthreads();       // x of this piece staged; the other buffer free
        WCodes<FMT> cur[2];
        cur[0] = w.c[0];
        cur[1] = w.c[1];
        if constexpr (FMT != FMT_F16) {
            // this piece's scales and mins through the wave's own LDS (lane = plane x column -> any group)
            *(u32x4_t*)(sb + lane * 16) = w.s;
            wave_lds_fence();
            const uint32_t first = pl.colg + (uint32_t)(FEW_G * q);
            const int shift = (int)(first - min(first, pl.glast));
#pragma unroll
            for (int t = 0; t < 2; ++t)
#pragma unroll
                for (int e = 0; e < 2; ++e) {
                    const int g = 4 * t + 2 * h + e, at = min(g + shift, FEW_G - 1);
                    const bool live = q < q1 && FEW_G * q + g < G;
                    const uint32_t s = *(const uint16_t*)(sb + (lane & 31) * 16 + at * 2);
                    const uint32_t m = FMT == FMT_Q8 ? 0u : *(const uint16_t*)(sb + 512 + (lane & 31) * 16 + at * 2);
                    cur[t].s[e] = live ? s : 0u;
                    cur[t].m[e] = live ? m : 0u;
                }
        }
        if (it + 1 < iters) load_x(qn < q1 ? qn : nq);
        __builtin_amdgcn_sched_barrier(0);
        if (it + D < iters) few_load(w, pl, piece(q + D * KW));
        __builtin_amdgcn_sched_barrier(0);
        floatx16_t acc[MB];
#pragma unroll
        for (int b = 0; b < MB; ++b)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[b][r] = 0.f;
        const unsigned char* const xb = xb0 + buf * XB;
        const GroupOps go0 = group_ops<FMT>(cur[0], dk), go1 = group_ops<FMT>(cur[1], dk);
        // slice i = 8 t + s: its A fragments are read one slice ahead, and no further (the scheduling
        // barrier: left alone the compiler reads all 16 first, which takes 64 registers per row block)
        auto read_a16 = [&](half8_t (&a)[MB], int i) {
#pragma unroll
            for (int b = 0; b < MB; ++b)
                a[b] = *(const half8_t*)(xb + arow[b] + (i >> 3) * (XR * XROWP) + (i & 7) * (FMT == FMT_F16 ? 32 : 16));
        };
        half8_t a[2][MB];
        read_a16(a[0], 0);
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            if (i < 15) read_a16(a[(i + 1) & 1], i + 1);
            half8_t bf;
            if constexpr (FMT == FMT_F16) {
                const uint32_t* d = cur[i >> 3].w + 4 * (i & 7);
                bf = __builtin_bit_cast(half8_t, u32x4_t{d[0], d[1], d[2], d[3]});
            } else {
                bf = b_frag<FMT>(cur[i >> 3], i < 8 ? go0 : go1, i & 7);
            }
#pragma unroll
            for (int b = 0; b < MB; ++b)
                acc[b] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a[i & 1][b], bf, acc[b], 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
        }
        // times the piece's row scales (register r of a tile: row 8 (r >> 2) + 4 h + (r & 3))
#pragma unroll
        for (int b = 0; b < MB; ++b)
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                const int r0 = 32 * b + 8 * g + 4 * h;
                if (XR < 32 && 8 * g >= XR) break;
                const f32x4_t s4 = *(const f32x4_t*)(rs0 + buf * XR + r0);
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    tot[b][4 * g + e] = fmaf(acc[b][4 * g + e], s4[e], tot[b][4 * g + e]);
            }
        wave_lds_fence();
        if (it + 1 < iters) store_x(NB == 2 ? buf ^ 1 : 0);
    }

    float* const out = KS > 1 ? part + (size_t)slice * M * N : y;
    if constexpr (KW == 1) {
        if (ncol < N)
#pragma unroll
            for (int b = 0; b < MB; ++b)
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    const int m = 32 * b + 8 * (r >> 2) + 4 * h + (r & 3);
                    if (m < M) out[(size_t)m * N + ncol] = tot[b][r];
                }
    } else {
        __syncthreads();                             // every wave is done with its x pieces
        float* const red = reinterpret_cast<float*>(smem);
#pragma unroll
        for (int b = 0; b < MB; ++b)
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const int row = 8 * (r >> 2) + 4 * h + (r & 3);
                red[((wave * MB + b) * 32 + row) * 32 + (lane & 31)] = tot[b][r];
            }
        __syncthreads();
        for (int i = tid; i < MB * 32 * 32 * CW; i += NT) {
            const int c = i & 31, row = (i >> 5) % (MB * 32), cc = (i >> 5) / (MB * 32);
            if (row >= M) continue;
            const int n = ((int)blockIdx.x * CW + cc) * 32 + c;
            float v = red[((cc * MB) * 32 + row) * 32 + c];
#pragma unroll
            for (int k = 1; k < KW; ++k) v += red[(((k * CW + cc) * MB) * 32 + row) * 32 + c];
            if (n < N) out[(size_t)row * N + n] = v;
        }
    }
}

}  // namespace

// Kernels: brik_gemm_few_<fmt>_r<XR>_<CW>x<KW>, in the order of the runtime's table (kFewTiles); grid (column
// blocks of 32 CW, K slices of qps pieces), 64 CW KW threads.
#define BRIK_GEMM_FEW(FMTN, FMT, XR, CW, KW, D)                                                           \
    extern "C" __global__ __launch_bounds__(64 * CW * KW) void brik_gemm_few_##FMTN##_r##XR##_##CW##x##KW( \
        const float* __restrict__ x, const uint8_t* __restrict__ p0, const uint8_t* __restrict__ p1,      \
        const uint16_t* __restrict__ sc, const uint16_t* __restrict__ mn, float* __restrict__ y,          \
        float* __restrict__ part, int M, int K, int N, int qps)                                           \
    {                                                                                                     \
        few_body<FMT, XR, CW, KW, D>(x, p0, p1, sc, mn, y, part, M, K, N, qps);                           \
    }
#ifndef BRIK_FEW_TILES
#define BRIK_FEW_TILES(X, FMTN, FMT)                                                                      \
    X(FMTN, FMT, 8, 1, 4, 1) X(FMTN, FMT, 16, 1, 4, 1) X(FMTN, FMT, 16, 2, 4, 1)                          \
    X(FMTN, FMT, 32, 4, 1, 1) X(FMTN, FMT, 64, 4, 1, 1)
#endif
BRIK_FEW_TILES(BRIK_GEMM_FEW, q4, FMT_Q4)
BRIK_FEW_TILES(BRIK_GEMM_FEW, q8, FMT_Q8)
BRIK_FEW_TILES(BRIK_GEMM_FEW, q3, FMT_Q3)
BRIK_FEW_TILES(BRIK_GEMM_FEW, f16, FMT_F16)
