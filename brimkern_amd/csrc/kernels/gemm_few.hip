// Few-row GEMM (2 to 64 rows): y[M, N] = x[M, K] . deq(W[N, K])^T in one launch, x read as it is.
// For the calls of batched decoding that the tiled kernels serve badly (the reference's
// matmul_t_q*_tiled range, src/lib/webgpu/shaders.ts:120-168, 425-527): few rows per weight, so the weight
// stream and the latency of its loads bound them, not the matrix cores.
//
// A block owns 32 CW columns; its waves are CW column waves x KW k waves. K is cut into pieces of 256; k
// wave `kw` takes every KW-th piece of the block's range. For a piece a wave holds the codes of its 32
// columns and their scales in registers, loaded one piece ahead in whole lines and then turned through LDS
// (FewCfg), and the x rows of the piece in LDS as f16, each row scaled by a power of two of its own largest
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
// a time) and the sum: q4 8 x 2560 x 9728 16.3 -> 10.4 us, q8 33 x 9728 x 2560 34.8 -> 17.7 us,
// q4 16 x 9728 x 2560 27.4 -> 12.6 us, q4 16 x 896 x 4864 9.8 -> 6.1 us.
// f16 weights (FMT_F16, K % 8 == 0) run the same pieces with no scales, both operands in natural k order.
#include "common.h"

namespace {

constexpr int FEW_K = 256;           // k of one piece: two steps of 128
constexpr int FEW_G = FEW_K / BRIK_GROUP;

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

// How a wave brings in the codes of a piece (32 columns x 256 k; f16: twice 128 k): a load instruction covers
// runs of PB bytes of RPI rows, 16 bytes per lane, and the rows then pass through the wave's own LDS (16 bytes
// further apart, so the reads below meet no bank twice) to the lane that owns their column. Loaded by column,
// every lane of an instruction is in another row and the texture addresser takes them one after the other.
// Measured against that: 8 x 2560 x 9728 q3 14.6 -> 12.7 us, f16 17.1 -> 15.1, q4 11.5 -> 11.3; 33 x 9728 x 2560
// q8 19.8 -> 19.1, q3 21.2 -> 20.0; f16 16 x 2560 x 9728 19.4 -> 15.6.
template <int FMT>
struct FewCfg {
    static constexpr int PB = FMT == FMT_Q4 ? 128 : FMT == FMT_Q3 ? 64 : 256;
    static constexpr int LPR = PB / 16, RPI = 64 / LPR, NI = 32 / RPI;
    static constexpr int PARTS = FMT == FMT_F16 ? 2 : 1;          // loads of the codes region per piece
    static constexpr int STRIDE = PB + 16, HI = 32 * STRIDE;      // q3's high bits: 32 bytes a row, 48 apart
    static constexpr int S = HI + (FMT == FMT_Q3 ? 32 * 48 : 0);  // scales, mins: 16 bytes per column each
    static constexpr int BYTES = S + (FMT == FMT_F16 ? 0 : 1024);
};

template <int FMT>
struct FewW {
    u32x4_t c[FewCfg<FMT>::PARTS][FewCfg<FMT>::NI];
    u32x4_t hi;                      // q3
    u32x4_t s;                       // 8 scales (lanes 0-31) or mins (lanes 32-63) of column lane & 31
};

template <int FMT>
struct FewPlanes {
    brsrc_t r0, r1;
    uint32_t off, off1;              // byte offset of this lane's first chunk in r0 (and r1), piece 0
    uint32_t step;                   // bytes from one load instruction's rows to the next's
    const uint16_t* sp;              // this lane half's plane: scales or mins
    uint32_t sgrp;                   // flat group index in it of column lane & 31, group 0
    uint32_t glast;                  // last flat group at which 8 groups end inside the plane
    int G, K;

    // n0: the wave's first column. Rows past N read the next matrix or zeros past the plane: their columns
    // are not stored.
    __device__ __forceinline__ void begin(const uint8_t* p0, const uint8_t* p1, const uint16_t* sc, const uint16_t* mn,
                                          int N, int K_, int n0, size_t e, size_t E)
    {
        using C = FewCfg<FMT>;
        const int lane = (int)threadIdx.x & 63;
        const size_t wel = (size_t)N * K_;
        const size_t row = FMT == FMT_F16 ? (size_t)K_ * 2 : FMT == FMT_Q8 ? K_ : FMT == FMT_Q4 ? K_ / 2 : K_ / 4;
        G = K_ / BRIK_GROUP;
        K = K_;
        r0 = make_rsrc(p0 + e * row * N, (uint32_t)(row * N));
        off = (uint32_t)(n0 + lane / C::LPR) * (uint32_t)row + 16u * (uint32_t)(lane % C::LPR);
        step = (uint32_t)C::RPI * (uint32_t)row;
        if constexpr (FMT == FMT_Q3) {
            r1 = make_rsrc(p1 + e * wel / 8, (uint32_t)(wel / 8));
            off1 = (uint32_t)(n0 + lane / 2) * (uint32_t)(K_ / 8) + 16u * (uint32_t)(lane % 2);
        }
        sp = lane < 32 || FMT == FMT_Q8 ? sc : mn;
        sgrp = (uint32_t)(e * N * G) + (uint32_t)min(n0 + (lane & 31), N - 1) * (uint32_t)G;
        glast = (uint32_t)(E * N * G) - FEW_G;
    }
};

typedef u32x4_t u32x4_2_t __attribute__((aligned(2)));

template <int FMT>
__device__ __forceinline__ void few_load(FewW<FMT>& f, const FewPlanes<FMT>& p, int q)
{
    using C = FewCfg<FMT>;
    if constexpr (FMT != FMT_F16)
        f.s = *(const u32x4_2_t*)(p.sp + min(p.sgrp + (uint32_t)(FEW_G * q), p.glast));
#pragma unroll
    for (int t = 0; t < C::PARTS; ++t) {
        const uint32_t at = p.off + (uint32_t)((C::PARTS * q + t) * C::PB);
        // f16: chunks past K get an offset past the buffer's end (N K < 2^31 halves; zeros, so an infinite weight of the next row
        // cannot meet x's zero padding); the other formats' dead groups have their scales masked
        const uint32_t dead = FMT == FMT_F16 && FEW_K * q + 128 * t + 8 * ((int)(threadIdx.x & 63) % C::LPR) >= p.K ? 0xFFFFFFF0u : 0u;
#pragma unroll
        for (int i = 0; i < C::NI; ++i)
            f.c[t][i] = __builtin_amdgcn_raw_buffer_load_b128(p.r0, (at + (uint32_t)i * p.step) | dead, 0, 0);
    }
    if constexpr (FMT == FMT_Q3) f.hi = __builtin_amdgcn_raw_buffer_load_b128(p.r1, p.off1 + 32u * (uint32_t)q, 0, 0);
}

// Writes what few_load brought of part t (and, with part 0, the scales) into the wave's LDS region.
template <int FMT>
__device__ __forceinline__ void few_spread(const FewW<FMT>& f, unsigned char* wb, int t)
{
    using C = FewCfg<FMT>;
    const int lane = (int)threadIdx.x & 63;
#pragma unroll
    for (int i = 0; i < C::NI; ++i)
        *(u32x4_t*)(wb + (C::RPI * i + lane / C::LPR) * C::STRIDE + 16 * (lane % C::LPR)) = f.c[t][i];
    if constexpr (FMT == FMT_Q3) *(u32x4_t*)(wb + C::HI + (lane / 2) * 48 + 16 * (lane % 2)) = f.hi;
    if constexpr (FMT != FMT_F16) *(u32x4_t*)(wb + C::S + lane * 16) = f.s;
}

// This lane's two steps of codes, scales and mins of piece q (lane half h: groups 4 t + 2 h + e of its
// column). live: whether the piece is one of this wave's.
template <int FMT>
__device__ __forceinline__ void few_codes(WCodes<FMT> (&cur)[2], const FewPlanes<FMT>& p, const unsigned char* wb, int q,
                                          bool live)
{
    using C = FewCfg<FMT>;
    const int lane = (int)threadIdx.x & 63, h = lane >> 5;
    const unsigned char* const row = wb + (lane & 31) * C::STRIDE;
    const uint32_t first = p.sgrp + (uint32_t)(FEW_G * q);
    const int shift = (int)(first - min(first, p.glast));          // a 16-byte load moved back from the plane's end
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int e = 0; e < 2; ++e) {
            const int g = 4 * t + 2 * h + e;
            if constexpr (FMT == FMT_Q4) {
                const u32x4_t v = *(const u32x4_t*)(row + g * 16);
#pragma unroll
                for (int j = 0; j < 4; ++j) cur[t].w[4 * e + j] = v[j];
            } else if constexpr (FMT == FMT_Q8) {
#pragma unroll
                for (int k = 0; k < 2; ++k) {
                    const u32x4_t v = *(const u32x4_t*)(row + g * 32 + 16 * k);
#pragma unroll
                    for (int j = 0; j < 4; ++j) cur[t].w[8 * e + 4 * k + j] = v[j];
                }
            } else {
                const u32x2_t v = *(const u32x2_t*)(row + g * 8);
                cur[t].w[2 * e] = v.x;
                cur[t].w[2 * e + 1] = v.y;
                cur[t].w[4 + e] = *(const uint32_t*)(wb + C::HI + (lane & 31) * 48 + g * 4);
            }
            const int at = min(g + shift, FEW_G - 1);
            const uint32_t s = *(const uint16_t*)(wb + C::S + (lane & 31) * 16 + at * 2);
            const uint32_t m = FMT == FMT_Q8 ? 0u : *(const uint16_t*)(wb + C::S + 512 + (lane & 31) * 16 + at * 2);
            const bool ok = live && FEW_G * q + g < p.G;
            cur[t].s[e] = ok ? s : 0u;
            cur[t].m[e] = ok ? m : 0u;
        }
}

// acc += the piece's product: x rows at xa (this lane's row and k half of the first row block; the steps STEP
// bytes apart, row blocks 32 * XROWP), codes cur, or f16 rows in wb (part 1 spread when part 0 is done).
// The fragments of a slice are read one slice ahead and no further (the scheduling barrier: left alone the
// compiler reads all 16 first, which takes 64 registers per row block).
template <int FMT, int MB, int XROWP, int STEP>
__device__ __forceinline__ void few_mma(floatx16_t (&acc)[MB], const unsigned char* const (&xa)[MB], const WCodes<FMT> (&cur)[2],
                                        const DeqConst& dk, unsigned char* wb, const FewW<FMT>& w)
{
    using C = FewCfg<FMT>;
    const int lane = (int)threadIdx.x & 63, h = lane >> 5;
    GroupOps go[2];
    if constexpr (FMT != FMT_F16) {
        go[0] = group_ops<FMT>(cur[0], dk);
        go[1] = group_ops<FMT>(cur[1], dk);
    }
    auto read_a = [&](half8_t (&a)[MB], int i) {
#pragma unroll
        for (int b = 0; b < MB; ++b)
            a[b] = *(const half8_t*)(xa[b] + (i >> 3) * STEP + (i & 7) * (FMT == FMT_F16 ? 32 : 16));
    };
    half8_t a[2][MB];
    read_a(a[0], 0);
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        if (i < 15) read_a(a[(i + 1) & 1], i + 1);
        half8_t bf;
        if constexpr (FMT == FMT_F16) {
            if (i == 8) {
                wave_lds_fence();
                few_spread(w, wb, 1);
                wave_lds_fence();
            }
            bf = *(const half8_t*)(wb + (lane & 31) * C::STRIDE + (i & 7) * 32 + 16 * h);
        } else {
            bf = b_frag<FMT>(cur[i >> 3], go[i >> 3], i & 7);
        }
#pragma unroll
        for (int b = 0; b < MB; ++b) acc[b] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a[i & 1][b], bf, acc[b], 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
    }
}

// XR: rows of x held in LDS (M <= XR); CW x KW waves. MB row blocks of 32 (the last may be half used).
template <int FMT, int XR, int CW, int KW>
__device__ __forceinline__ void few_body(const float* __restrict__ x, const uint8_t* __restrict__ p0,
                                         const uint8_t* __restrict__ p1, const uint16_t* __restrict__ sc,
                                         const uint16_t* __restrict__ mn, float* __restrict__ y,
                                         float* __restrict__ part, int M, int K, int N, int qps)
{
    constexpr int MB = (XR + 31) / 32, NT = 64 * CW * KW, WB = FewCfg<FMT>::BYTES;
    // one piece of x: [step][row][256 bytes + 16]; the pad puts the 16 rows of a read phase on 16 different
    // bank groups, so every fragment read is one address and an immediate offset
    constexpr int XROWP = 272, STEP = XR * XROWP, XB = 2 * STEP;
    constexpr int RP = XR / (2 * CW);                // row pairs a wave stages
    constexpr int LIVE = KW * XB + CW * KW * WB, RED = KW > 1 ? KW * CW * MB * 4096 : 0;
    __shared__ __attribute__((aligned(16))) unsigned char smem[(LIVE > RED ? LIVE : RED) + KW * XR * 4];

    const int tid = (int)threadIdx.x, lane = tid & 63, h = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), cw = wave % CW, kw = wave / CW;
    const int nq = (K + FEW_K - 1) / FEW_K;
    const int KS = (int)gridDim.y, slice = (int)blockIdx.y;
    const int q0 = slice * qps, q1 = min(q0 + qps, nq);        // q0 < nq: the host sizes gridDim.y so
    const int iters = (q1 - q0 + KW - 1) / KW;
    const int n0 = ((int)blockIdx.x * CW + cw) * 32, ncol = n0 + (lane & 31);

    FewPlanes<FMT> pl;
    pl.begin(p0, p1, sc, mn, N, K, n0, 0, 1);
    unsigned char* const xb = smem + kw * XB;
    unsigned char* const wb = smem + KW * XB + wave * WB;
    float* const rs = reinterpret_cast<float*>(smem + (LIVE > RED ? LIVE : RED)) + kw * XR;

    // x of a piece: this wave's row pairs (row 2 (RP cw + i) + h, 8 floats per lane); rows past M lie past the
    // buffer's end, and so does the offset given to lanes past K: both read zeros
    const brsrc_t rx = make_rsrc(x, (uint32_t)((size_t)M * K * 4));
    const uint32_t xoff = (uint32_t)((2 * RP * cw + h) * K + 8 * (lane & 31)) * 4u;
    f32x4_t xa[RP], xc[RP];
    auto load_x = [&](int q) {
        const uint32_t at = xoff + (uint32_t)(FEW_K * 4 * q), dead = FEW_K * q + 8 * (lane & 31) < K ? 0u : 0xFFFFFF00u;
#pragma unroll
        for (int i = 0; i < RP; ++i) {
            const uint32_t o = (at + (uint32_t)(8 * i * K)) | dead;
            xa[i] = __builtin_bit_cast(f32x4_t, __builtin_amdgcn_raw_buffer_load_b128(rx, o, 0, 0));
            xc[i] = __builtin_bit_cast(f32x4_t, __builtin_amdgcn_raw_buffer_load_b128(rx, o | 16u, 0, 0));
        }
    };
    auto store_x = [&]() {
        unsigned char* const xw = xb + ((lane & 31) >> 4) * STEP + (lane & 15) * 16;
#pragma unroll
        for (int i = 0; i < RP; ++i) {
            const int m = 2 * (RP * cw + i) + h;
            if (2 * (RP * cw + i) >= M) break;       // uniform
            float down;
            const float up = xprep_up(half_max(few_absmax8(xa[i], xc[i])), down);
            if ((lane & 31) == 0) rs[m] = down;
            *(half8_t*)(xw + m * XROWP) = to_h8_order<FMT == FMT_F16>(xa[i], xc[i], up);
        }
    };

    floatx16_t tot[MB];
#pragma unroll
    for (int b = 0; b < MB; ++b)
#pragma unroll
        for (int r = 0; r < 16; ++r) tot[b][r] = 0.f;
    const unsigned char* xrow[MB];                   // this lane's A row and k half
#pragma unroll
    for (int b = 0; b < MB; ++b)
        xrow[b] = xb + min(32 * b + (lane & 31), M - 1) * XROWP + (FMT == FMT_F16 ? 16 : 128) * h;
    const DeqConst dk = DeqConst::make();

    // x before W: loads complete in order, so the rows are converted while the weights are on their way.
    // A k wave without a piece left multiplies zeros: its x reads as zeros and its scales are masked, f16
    // weights read as zeros
    auto piece = [&](int q) { return FMT == FMT_F16 ? (q < q1 ? q : nq) : min(q, nq - 1); };
    FewW<FMT> w;
    load_x(q0 + kw < q1 ? q0 + kw : nq);
    __builtin_amdgcn_sched_barrier(0);
    few_load(w, pl, piece(q0 + kw));
    __builtin_amdgcn_sched_barrier(0);
    for (int it = 0; it < iters; ++it) {
        const int q = q0 + it * KW + kw, qn = q + KW;
        const bool more = it + 1 < iters;            // uniform over the block
        if (CW > 1 && it) __syncthreads();           // the previous piece's rows are read
        store_x();
        if (more) load_x(qn < q1 ? qn : nq);
        __builtin_amdgcn_sched_barrier(0);
        few_spread(w, wb, 0);
        if constexpr (CW > 1) __syncthreads();       // x of this piece staged
        else wave_lds_fence();
        WCodes<FMT> cur[2];
        FewW<FMT> rest;                              // f16: the second half of the piece, spread by few_mma
        if constexpr (FMT == FMT_F16) rest = w;
        else few_codes(cur, pl, wb, q, q < q1);
        if (more) few_load(w, pl, piece(qn));
        __builtin_amdgcn_sched_barrier(0);
        floatx16_t acc[MB];
#pragma unroll
        for (int b = 0; b < MB; ++b)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[b][r] = 0.f;
        few_mma<FMT, MB, XROWP, STEP>(acc, xrow, cur, dk, wb, rest);
        // times the piece's row scales (register r of a tile: row 8 (r >> 2) + 4 h + (r & 3))
#pragma unroll
        for (int b = 0; b < MB; ++b)
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                const int r0 = 32 * b + 8 * g + 4 * h;
                if (XR < 32 && 8 * g >= XR) break;
                const f32x4_t s4 = *(const f32x4_t*)(rs + r0);
#pragma unroll
                for (int e = 0; e < 4; ++e) tot[b][4 * g + e] = fmaf(acc[b][4 * g + e], s4[e], tot[b][4 * g + e]);
            }
        wave_lds_fence();                            // this piece's rows and codes are read
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
#define BRIK_GEMM_FEW(FMTN, FMT, XR, CW, KW)                                                              \
    extern "C" __global__ __launch_bounds__(64 * CW * KW) void brik_gemm_few_##FMTN##_r##XR##_##CW##x##KW( \
        const float* __restrict__ x, const uint8_t* __restrict__ p0, const uint8_t* __restrict__ p1,      \
        const uint16_t* __restrict__ sc, const uint16_t* __restrict__ mn, float* __restrict__ y,          \
        float* __restrict__ part, int M, int K, int N, int qps)                                           \
    {                                                                                                     \
        few_body<FMT, XR, CW, KW>(x, p0, p1, sc, mn, y, part, M, K, N, qps);                           \
    }
#ifndef BRIK_FEW_TILES
#define BRIK_FEW_TILES(X, FMTN, FMT)                                                                      \
    X(FMTN, FMT, 8, 1, 4) X(FMTN, FMT, 16, 1, 4) X(FMTN, FMT, 16, 2, 4)                          \
    X(FMTN, FMT, 32, 4, 1) X(FMTN, FMT, 64, 4, 1)
#endif
BRIK_FEW_TILES(BRIK_GEMM_FEW, q4, FMT_Q4)
BRIK_FEW_TILES(BRIK_GEMM_FEW, q8, FMT_Q8)
BRIK_FEW_TILES(BRIK_GEMM_FEW, q3, FMT_Q3)
BRIK_FEW_TILES(BRIK_GEMM_FEW, f16, FMT_F16)
