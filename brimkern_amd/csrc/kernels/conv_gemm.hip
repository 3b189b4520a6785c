// Convolution as an MFMA GEMM over the taps, without im2col rows: out[co, p] = bias[co] + sum over taps of
// W[co, :, tap] . x[:, pixel of p at that tap], for channel counts that are multiples of 32 (the reference's
// conv2d_direct_q8 / q4, src/lib/webgpu/shaders.ts:1026-1123). Two launches:
//   1. brik_conv_prep_<fmt>: the input as f16 pixel rows [H W][Cin] in channel order, each row times a power
//      of two of its own largest magnitude (xprep_up), and W dequantized to f16 in MFMA fragment order
//      (gemm_frag.hip: panels of 32 output channels, lane 32 h + r of a fragment holding 8 channels of row r),
//      k running over (tap, channel) instead of the flat (channel, tap).
//   2. brik_gemm_conv_<tile>: W fragments and pixel rows through LDS, 32 channels of one tap a step. A block's
//      pixel rows of a tap are the input's rows at that tap's offset: a lane whose tap lies outside the image
//      loads from past the end of the buffer, zeros. The sums of a tap are multiplied by the scales of its
//      pixel rows (one value per lane: a lane of the result tile holds one pixel) and added up in f32.
// With gridDim.y > 1 a block covers a slice of the steps and writes a partial tile to `part` for
// brik_splitk_reduce, the bias in slice 0's.
//
// What bounds it: a step takes 0.2 us of one or two waves per SIMD issuing its instructions one after the other
// (64 x 64 tile; MFMA 0.03), the same with 8 or 16 buffers, with a barrier per step or every second, and with
// fragments read one slice or one step ahead; 128 x 128, four times the products, 0.24 alone and 0.4 on a full
// chip. So long sums are sliced until the blocks fill the chip. It took the place of three launches that wrote
// and read the input kh kw times (channel maxima 4.8 us, im2col 10 us, and a GEMM of dependent steps that
// dequantized W in every row tile, 25 us, for 320 x 64 x 64, 320 channels, 3 x 3): 36.7 -> 30.2 us a call
// there (staging 8, product 21, sum 5), 320 x 14 x 15, 28 channels 25.9 -> 14.2, 608 x 61 x 80, 206 channels,
// 5 x 5, stride 2 124.6 -> 37.1.
#include "common.h"
#include "stage_abi.h"

namespace {

constexpr int CP_PIX = 16, CP_CH = 512;              // staging: pixels of a block, channels of a round
constexpr int CP_XROW = CP_CH * 2 + 16;              // LDS bytes between pixels

// Pixels [16 b, 16 b + 16) of the input, all channels, as scaled f16 rows. Thread (g, q) holds channels
// g + 64 u of pixel q; up to 512 channels are read once.
__device__ __forceinline__ void conv_stage_pixels(unsigned char* smem, const float* __restrict__ inp,
                                                  uint16_t* __restrict__ xt, float* __restrict__ xs, int Cin, int HW, int b)
{
    const int tid = (int)threadIdx.x, q = tid & 15, g = tid >> 4;
    const int p = b * CP_PIX + q, pc = min(p, HW - 1);
    float* const part = reinterpret_cast<float*>(smem + CP_PIX * CP_XROW);      // [64][17]
    float v[8];
    auto load = [&](int c0) {
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            const int ci = c0 + g + 64 * u;
            v[u] = ci < Cin ? inp[(size_t)ci * HW + pc] : 0.f;
        }
    };
    float mx = 0.f;
    for (int c0 = 0; c0 < Cin; c0 += CP_CH) {
        load(c0);
#pragma unroll
        for (int u = 0; u < 8; ++u) mx = fmaxf(mx, fabsf(v[u]));
    }
    part[g * 17 + q] = mx;
    __syncthreads();
    mx = 0.f;
#pragma unroll
    for (int k = 0; k < 64; ++k) mx = fmaxf(mx, part[k * 17 + q]);
    float down;
    const float up = xprep_up(mx, down);
    if (g == 0 && p < HW) xs[p] = down;
    for (int c0 = 0; c0 < Cin; c0 += CP_CH) {
        if (Cin > CP_CH) load(c0);
        if (c0) __syncthreads();                     // the previous round is written out
#pragma unroll
        for (int u = 0; u < 8; ++u)
            *(_Float16*)(smem + q * CP_XROW + (g + 64 * u) * 2) = (_Float16)(v[u] * up);
        __syncthreads();
        const int nch = min(Cin - c0, CP_CH) / 8;    // 16-byte chunks of a pixel
        for (int i = tid; i < CP_PIX * nch; i += 1024) {
            const int r = i / nch, c = i - r * nch;
            if (b * CP_PIX + r < HW)
                *(u32x4_t*)(xt + (size_t)(b * CP_PIX + r) * Cin + c0 + 8 * c) = *(const u32x4_t*)(smem + r * CP_XROW + 16 * c);
        }
    }
}

// 32 output channels x 32 input channels, every tap: flat weights [co][32 cb taps, 32 (cb + 1) taps), whole
// groups of each row, to two fragments per tap. smem: taps x 2 KiB.
template <int FMT>
__device__ __forceinline__ void conv_stage_weights(unsigned char* smem, const void* __restrict__ p0,
                                                   const uint16_t* __restrict__ sc, const uint16_t* __restrict__ mn,
                                                   uint16_t* __restrict__ wf, int Cin, int Cout, int taps, int panel, int cb)
{
    const int tid = (int)threadIdx.x, K = Cin * taps, units = 4 * taps;      // units of 8 weights per row
    for (int i = tid; i < 32 * units; i += 1024) {
        const int r = i / units, u = i - r * units;
        const int co = min(32 * panel + r, Cout - 1);                        // rows past Cout are not stored
        const uint32_t at = (uint32_t)co * (uint32_t)K + (uint32_t)(32 * cb * taps + 8 * u);
        const float s = f16_bits_to_f32(sc[at >> 5]);
        float w[8];
        if constexpr (FMT == FMT_Q8) {
            const u32x2_t c = *(const u32x2_t*)(static_cast<const uint8_t*>(p0) + at);
#pragma unroll
            for (int e = 0; e < 8; ++e) w[e] = (float)(int8_t)(c[e >> 2] >> (8 * (e & 3))) * s;
        } else {
            const uint32_t c = *(const uint32_t*)(static_cast<const uint8_t*>(p0) + at / 2);
            const float m = f16_bits_to_f32(mn[at >> 5]);
#pragma unroll
            for (int e = 0; e < 8; ++e) w[e] = fmaf((float)(c >> (4 * e) & 15u), s, m);
        }
        int ci = 8 * u / taps, tap = 8 * u - ci * taps;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            *(_Float16*)(smem + tap * 2048 + (ci >> 4) * 1024 + ((ci >> 3 & 1) * 32 + r) * 16 + (ci & 7) * 2) = (_Float16)w[e];
            if (++tap == taps) {
                tap = 0;
                ++ci;
            }
        }
    }
    __syncthreads();
    const int S = K / 16;                            // fragments of a panel
    for (int i = tid; i < taps * 128; i += 1024) {
        const int tap = i >> 7, o = i & 127;
        *(u32x4_t*)(wf + ((size_t)panel * S + (size_t)tap * (Cin / 16) + 2 * cb) * 512 + o * 8) = *(const u32x4_t*)(smem + i * 16);
    }
}

template <int FMT>
__device__ __forceinline__ void conv_prep(unsigned char* smem, const float* __restrict__ inp, uint16_t* __restrict__ xt,
                                          float* __restrict__ xs, const void* __restrict__ p0,
                                          const uint16_t* __restrict__ sc, const uint16_t* __restrict__ mn,
                                          uint16_t* __restrict__ wf, int Cin, int HW, int Cout, int taps, int xblocks)
{
    const int b = (int)blockIdx.x;                   // uniform
    if (b < xblocks) {
        conv_stage_pixels(smem, inp, xt, xs, Cin, HW, b);
        return;
    }
    const int ncb = Cin / 32, i = b - xblocks;
    conv_stage_weights<FMT>(smem, p0, sc, mn, wf, Cin, Cout, taps, i / ncb, i % ncb);
}

// Block tile: WR x WC waves of WA x WB blocks of 32 output channels x 32 pixels; XQ LDS buffers of a step.
template <int WR_, int WC_, int WA_, int WB_, int XQ_>
struct CTile {
    static constexpr int WR = WR_, WC = WC_, WA = WA_, WB = WB_, XQ = XQ_;
    static constexpr int NW = WR * WC, NT = 64 * NW;
    static constexpr int BMB = WR * WA, BNB = WC * WB;
    static constexpr int BM = 32 * BMB, BN = 32 * BNB;
    static constexpr int XBUF = BMB * 2048, BUF = (BMB + BNB) * 2048;      // bytes of a step: W, then pixel rows
    static constexpr int AL = (BMB * 2 + NW - 1) / NW, BL = (BNB * 2 + NW - 1) / NW, LD = AL + BL;
    static constexpr int SCALES = XQ * BUF;                                 // then [taps][BN] row scales
    static constexpr int BIAS = SCALES + BRIK_CONV_GEMM_MAX_TAPS * BN * 4;  // then the bias of the BM rows
    static constexpr int SMEM = BIAS + BM * 4;
    static_assert(XQ >= 3 && SMEM <= 160 * 1024 && WA - 1 + WB <= 15 && (XQ - 2) * LD < 64, "tile");
};

__device__ __forceinline__ float ds_read_b32_at(uint32_t addr)
{
    float v;
    asm volatile("ds_read_b32 %0, %1" : "=v"(v) : "v"(addr));
    return v;
}

struct ConvShape {
    int Cin, H, W, Cout, kw, taps, stride, pad, OW, P;
};

template <class T>
__device__ __forceinline__ void conv_tile_run(unsigned char* smem, const uint16_t* __restrict__ wf,
                                              const uint16_t* __restrict__ xt, const float* __restrict__ xs,
                                              const float* __restrict__ bias, float* __restrict__ dst, const ConvShape& c,
                                              int t0, int t1, int mt, int nt)
{
    constexpr int WA = T::WA, WB = T::WB, XQ = T::XQ, LD = T::LD;
    const int tid = threadIdx.x, lane = tid & 63, h = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wr = wave / T::WC, wc = wave % T::WC;
    const int RB = (c.Cout + 31) / 32, csteps = c.Cin / 32, S = c.taps * csteps * 2;
    const brsrc_t rw = make_rsrc(wf, (uint32_t)((size_t)RB * S * 1024));
    const brsrc_t rx = make_rsrc(xt, (uint32_t)((size_t)c.H * c.W * c.Cin * 2));
    const uint32_t voff = (uint32_t)lane * 16;

    uint32_t abase0[T::AL], adst[T::AL], bdst[T::BL], chunk[T::BL], boffs[T::BL], nboffs[T::BL];
    int y0[T::BL], x0[T::BL];
#pragma unroll
    for (int i = 0; i < T::AL; ++i) {
        const int q = min(T::NW * i + wave, T::BMB * 2 - 1);
        abase0[i] = (uint32_t)(min(mt * T::BMB + (q >> 1), RB - 1) * S + (q & 1)) * 1024u;
        adst[i] = (uint32_t)q * 1024u;
    }
#pragma unroll
    for (int i = 0; i < T::BL; ++i) {
        const int q = min(T::NW * i + wave, T::BNB * 2 - 1), r = 16 * q + (lane >> 2);
        const int p = min(nt * T::BN + r, c.P - 1), oy = p / c.OW;
        y0[i] = oy * c.stride - c.pad;
        x0[i] = (p - oy * c.OW) * c.stride - c.pad;
        chunk[i] = (uint32_t)(((lane & 3) ^ ((r >> 2) & 3)) * 16);
        bdst[i] = (uint32_t)(T::XBUF + q * 1024);
    }
    // the loads run ahead of the products: their step and its tap and channel block. The row offsets of the
    // tap after it are kept ready (nboffs, renewed at each end of a tap of the products, and one end of a tap
    // of the loads lies between two of those), so that moving on is a select and no branch
    const int tap0 = t0 / csteps;
    int fstep = t0, fc = t0 - tap0 * csteps, ky = tap0 / c.kw, kx = tap0 - ky * c.kw;
    auto seek = [&](uint32_t (&o)[T::BL], int ty, int tx) {
#pragma unroll
        for (int i = 0; i < T::BL; ++i) {
            const int iy = y0[i] + ty, ix = x0[i] + tx;
            const bool in = (uint32_t)iy < (uint32_t)c.H && (uint32_t)ix < (uint32_t)c.W;
            const uint32_t at = (uint32_t)(iy * c.W + ix) * (uint32_t)(2 * c.Cin) + chunk[i];
            o[i] = in ? at : 0x80000000u;
        }
    };
    auto seek_next = [&]() {
        const bool wrap = kx + 1 == c.kw;
        seek(nboffs, wrap ? ky + 1 : ky, wrap ? 0 : kx + 1);
    };
    auto load = [&](int u, uint32_t buf) {
        if (u < T::AL)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rw, (lds_void_t*)(smem + buf + adst[u]), 16, voff,
                                                     (int)(abase0[u] + (uint32_t)fstep * 2048u), 0, 0);
        else
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rx, (lds_void_t*)(smem + buf + bdst[u - T::AL]), 16,
                                                     boffs[u - T::AL], fc * 64, 0, 0);
    };
    // past the last step: its weights again, and pixel rows in range
    auto advance = [&]() {
        fstep = min(fstep + 1, t1 - 1);
        const bool turn = fc + 1 == csteps, wrap = turn && kx + 1 == c.kw;
        fc = turn ? 0 : fc + 1;
        kx = wrap ? 0 : kx + (turn ? 1 : 0);
        ky += wrap ? 1 : 0;
#pragma unroll
        for (int i = 0; i < T::BL; ++i) boffs[i] = turn ? nboffs[i] : boffs[i];
        return turn;
    };

    half8_t a[2][WA], b[2][WB];
    floatx16_t acc[WA][WB], tot[WA][WB];
#pragma unroll
    for (int i = 0; i < WA; ++i)
#pragma unroll
        for (int j = 0; j < WB; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[i][j][r] = tot[i][j][r] = 0.f;
    // the scales of the pixel rows of this slice's taps: loaded ahead of the first steps (loads return in
    // order), written to LDS by asm (the compiler would hold an ordinary LDS write until the direct loads
    // to LDS are done)
    const int nscale = ((t1 - 1) / csteps + 1 - tap0) * T::BN;
    auto scale = [&](int e) {
        const int tap = tap0 + e / T::BN, p = min(nt * T::BN + e % T::BN, c.P - 1), oy = p / c.OW, ky = tap / c.kw;
        const int iy = oy * c.stride - c.pad + ky, ix = (p - oy * c.OW) * c.stride - c.pad + tap - ky * c.kw;
        const bool in = (uint32_t)iy < (uint32_t)c.H && (uint32_t)ix < (uint32_t)c.W;
        return xs[in ? iy * c.W + ix : 0];           // outside: times a sum of zeros
    };
    const uint32_t scl = lds_addr(smem + T::SCALES);
    const float bias_row = bias && tid < T::BM ? bias[min(mt * T::BM + tid, c.Cout - 1)] : 0.f;
    float sc0[3];
#pragma unroll
    for (int i = 0; i < 3; ++i) sc0[i] = scale(min(tid + T::NT * i, nscale - 1));
    seek(boffs, ky, kx);
    seek_next();
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int q = 0; q < XQ - 1; ++q) {
#pragma unroll
        for (int u = 0; u < LD; ++u) load(u, (uint32_t)(q * T::BUF));
        if (advance()) seek_next();
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < 3; ++i)
        if (tid + T::NT * i < nscale) store_rscale(scl + 4 * (uint32_t)(tid + T::NT * i), sc0[i]);
    if (tid < T::BM) store_rscale(lds_addr(smem + T::BIAS) + 4 * (uint32_t)tid, bias_row);
    for (int e = tid + 3 * T::NT; e < nscale; e += T::NT) store_rscale(scl + 4 * (uint32_t)e, scale(e));
    wait_vm<(XQ - 2) * LD>();                        // step 0
    step_barrier();
    const uint32_t abase = lds_addr(smem) + (uint32_t)(wr * WA * 2048) + voff;
    uint32_t boff[2];                                // pixel fragment of slice s: row lane & 31, chunk 2 s + h
#pragma unroll
    for (int s = 0; s < 2; ++s)
        boff[s] = lds_addr(smem) + T::XBUF + (uint32_t)(wc * WB * 2048 + (lane & 31) * 64) +
                  (uint32_t)(((2 * s + h) ^ ((lane >> 2) & 3)) * 16);
    uint32_t srow = scl + (uint32_t)(wc * WB * 32 + (lane & 31)) * 4u;
    float sv[WB];
#pragma unroll
    for (int j = 0; j < WB; ++j) sv[j] = ds_read_b32_at(srow + 128u * (uint32_t)j);
    lds_wait();
#pragma unroll
    for (int j = 0; j < WB; ++j) tie(sv[j]);
    auto read = [&](int s, uint32_t nb) {
#pragma unroll
        for (int j = 0; j < WB; ++j) b[s][j] = ds_read_b128_by<2048>(boff[s] + nb, j);
#pragma unroll
        for (int i = 0; i < WA; ++i)
            a[s][i] = s == 0 ? ds_read_b128_by<2048>(abase + nb, i) : ds_read_b128_by<2048, 1024>(abase + nb, i);
        __builtin_amdgcn_sched_barrier(0);
    };
    auto arrived = [&](int s) {
#pragma unroll
        for (int i = 0; i < WA; ++i) tie(a[s][i]);
#pragma unroll
        for (int j = 0; j < WB; ++j) tie(b[s][j]);
        __builtin_amdgcn_sched_barrier(0);
    };
    read(0, 0);
    read(1, 0);

    // Step t multiplies buffer xq, whose fragments were read during step t - 1. It begins where the wave waits
    // for its loads of step t + 1 and meets the others, then loads step t + XQ - 1 into the buffer of step
    // t - 1; a slice's fragments of step t + 1 are read as soon as its products are issued.
    uint32_t xq = 0;
    int t = t0, left = min((tap0 + 1) * csteps, t1) - t0;   // steps left of the current tap
    while (true) {
        for (int n = 0; n < left; ++n) {
            const uint32_t x1 = xq + 1 == (uint32_t)XQ ? 0u : xq + 1, xfill = xq == 0 ? (uint32_t)XQ - 1 : xq - 1;
            wait_vm<(XQ - 3) * LD>();
            asm volatile("s_barrier" ::: "memory");
#pragma unroll
            for (int s = 0; s < 2; ++s) {
                lds_wait_n<WA + WB>();
                arrived(s);
#pragma unroll
                for (int i = 0; i < WA; ++i)
#pragma unroll
                    for (int j = 0; j < WB; ++j)
                        acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a[s][i], b[s][j], acc[i][j], 0, 0, 0);
                __builtin_amdgcn_sched_barrier(0);
                read(s, x1 * T::BUF);
                if (s == 0)
#pragma unroll
                    for (int u = 0; u < LD; ++u) load(u, xfill * T::BUF);
                __builtin_amdgcn_sched_barrier(0);
            }
            advance();
            xq = x1;
        }
        // the end of a tap; the fragments in flight first: moves may not touch their registers before
        lds_wait();
        arrived(0);
        arrived(1);
        t += left;
        left = min(csteps, t1 - t);
        srow += 4 * T::BN;
        seek_next();
#pragma unroll
        for (int j = 0; j < WB; ++j) {
#pragma unroll
            for (int i = 0; i < WA; ++i)
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    tot[i][j][r] = fmaf(acc[i][j][r], sv[j], tot[i][j][r]);
                    acc[i][j][r] = 0.f;
                }
        }
        if (left <= 0) break;                        // uniform
#pragma unroll
        for (int j = 0; j < WB; ++j) sv[j] = ds_read_b32_at(srow + 128u * (uint32_t)j);
        lds_wait();
#pragma unroll
        for (int j = 0; j < WB; ++j) tie(sv[j]);
    }
    wait_vm<0>();                                    // no load of this block lands in LDS after it
#pragma unroll
    for (int i = 0; i < WA; ++i) {
        const int row0 = (wr * WA + i) * 32 + 4 * h, co0 = mt * T::BM + row0;
        f32x4_t bv[4];
#pragma unroll
        for (int g = 0; g < 4; ++g) bv[g] = *(const f32x4_t*)(smem + T::BIAS + (row0 + 8 * g) * 4);
#pragma unroll
        for (int j = 0; j < WB; ++j) {
            const int p = nt * T::BN + (wc * WB + j) * 32 + (lane & 31);
            if (p >= c.P) continue;
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const int co = co0 + 8 * (r >> 2) + (r & 3);
                if (co < c.Cout) dst[(size_t)co * c.P + p] = tot[i][j][r] + bv[r >> 2][r & 3];
            }
        }
    }
}

}  // namespace

// brik_conv_prep_<fmt>: blocks [0, xblocks) stage 16 pixels each, the others 32 x 32 weights of every tap.
#define BRIK_CONV_PREP(FMTN, FMT)                                                                         \
    extern "C" __global__ __launch_bounds__(1024, 8) void brik_conv_prep_##FMTN(                          \
        const float* __restrict__ inp, uint16_t* __restrict__ xt, float* __restrict__ xs,                 \
        const void* __restrict__ p0, const uint16_t* __restrict__ sc, const uint16_t* __restrict__ mn,    \
        uint16_t* __restrict__ wf, int Cin, int HW, int Cout, int taps, int xblocks)                      \
    {                                                                                                     \
        __shared__ __attribute__((aligned(16))) unsigned char smem[BRIK_CONV_GEMM_MAX_TAPS * 2048];            \
        static_assert(BRIK_CONV_GEMM_MAX_TAPS * 2048 >= CP_PIX * CP_XROW + 64 * 17 * 4, "staging");            \
        conv_prep<FMT>(smem, inp, xt, xs, p0, sc, mn, wf, Cin, HW, Cout, taps, xblocks);                  \
    }
BRIK_CONV_PREP(q8, FMT_Q8)
BRIK_CONV_PREP(q4, FMT_Q4)

// brik_gemm_conv_<WR><WC>_<WA>x<WB>, in the order of the runtime's table (kConvTiles); grid (tiles, slices of
// sps steps).
#define BRIK_GEMM_CONV(WR, WC, WA, WB, XQ)                                                                \
    extern "C" __global__ __launch_bounds__(64 * WR * WC) void brik_gemm_conv_##WR##WC##_##WA##x##WB(     \
        const uint16_t* __restrict__ wf, const uint16_t* __restrict__ xt, const float* __restrict__ xs,   \
        const float* __restrict__ bias, float* __restrict__ out, float* __restrict__ part, int Cin, int H, \
        int W, int Cout, int kw, int taps, int stride, int pad, int OW, int P, int sps)                   \
    {                                                                                                     \
        using T = CTile<WR, WC, WA, WB, XQ>;                                                              \
        __shared__ __attribute__((aligned(1024))) unsigned char smem[T::SMEM];                            \
        int mt, nt;                                                                                       \
        frag_tile_of((int)blockIdx.x, (Cout + T::BM - 1) / T::BM, (P + T::BN - 1) / T::BN, mt, nt);       \
        const int t0 = (int)blockIdx.y * sps, t1 = min(t0 + sps, taps * (Cin / 32));                      \
        float* dst = gridDim.y > 1 ? part + (size_t)blockIdx.y * Cout * P : out;                          \
        const ConvShape c{Cin, H, W, Cout, kw, taps, stride, pad, OW, P};                                 \
        conv_tile_run<T>(smem, wf, xt, xs, blockIdx.y == 0 ? bias : nullptr, dst, c, t0, t1, mt, nt);     \
    }
BRIK_GEMM_CONV(2, 2, 1, 1, 8)
BRIK_GEMM_CONV(4, 2, 1, 2, 8)
