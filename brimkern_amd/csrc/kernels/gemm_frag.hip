// Large GEMM: y[M, N] = x[M, K] . W[N, K]^T on operands staged in MFMA fragment order.
// The same products as the tiled GEMM of gemm.hip (the reference's matmul_t_q*_tiled / _shared,
// src/lib/webgpu/shaders.ts:120-168, 425-527, 531-577), for launches of enough rows that dequantizing W
// once, instead of once per row tile, pays for the extra pass.
//
// A fragment is what one v_mfma_f32_32x32x16_f16 operand holds: 32 rows (or columns) x 16 k, 1024 bytes,
// lane l = 32 h + r holding the 8 halves of row r and k half h at byte 16 l. A panel is 32 rows of x or
// of W: its fragments in k order, S of them. Two launches:
//   1. brik_frag_prep_<fmt>: x rows scaled by a power of two and rounded to f16 exactly as brik_xprep_f16
//      does, and W dequantized to f16 exactly as the tiled GEMM's registers hold it, both written as
//      fragments (zeros past K).
//   2. brik_gemm_frag_<tile>: x fragments go through LDS (direct global->LDS loads, XQ buffers of 64 k),
//      W fragments straight into the registers of the waves that use them, 7 slices ahead.
// The order of every sum is that of the tiled GEMM (the same k in the same MFMA slot, slices in the
// same order), so the results are the same bits.
//
// What bounds it: the 64 bytes per clock of a CU's vector-memory path and the 128 of its LDS against the
// MFMAs. In fragment order every load instruction is one contiguous KiB and every LDS read lane-linear (no
// conflicts, immediate offsets), and with x through LDS and W through the registers neither path takes more
// than about 0.9 of the MFMA time (192 x 256 tile, per slice of 384 MFMA clocks: 22 KiB loaded, 24 KiB read
// from LDS). Rows of MFMAs are separated by one counted LDS wait, and one barrier serves 64 k. Measured
// alone (random operands): K = 9728, N = 2560, M = 4096 174 us, 1.17 PFLOP/s, where this card's library
// runs plain f16 in 163 us; K = 2560, N = 9728, M = 1024 53 us (library 53). The tiled GEMM took 249-273 us
// and 80 us there, its x staging apart. Staging: 38 us for 4096 x 9728 (6.3 TB/s), 12.5 us for the weights
// (5.2 TB/s; 21 us with 112 registers, one block of 1024 threads per CU).
#include "common.h"
#include "stage_abi.h"

namespace {

// Block tile of the fragment GEMM: WR x WC waves, each WA x WB tiles of 32 x 32. XQ LDS buffers of x, one
// step (4 slices, 64 k) each; W is loaded RS - 1 slices ahead into a ring of RS slices (4 or 8).
template <int WR_, int WC_, int WA_, int WB_, int XQ_, int RS_ = 8>
struct FTile {
    static constexpr int WR = WR_, WC = WC_, WA = WA_, WB = WB_, XQ = XQ_, RS = RS_;
    static constexpr int NW = WR * WC, NT = 64 * NW;
    static constexpr int BMB = WR * WA, BNB = WC * WB;          // 32-row / 32-column blocks
    static constexpr int BM = 32 * BMB, BN = 32 * BNB;
    static constexpr int XBUF = BMB * 4096;
    static constexpr int AL = BMB * 4 / NW;                     // direct loads per wave and step
    static constexpr int AL0 = (AL + 1) / 2;                    // of them in slice 2, the rest in slice 3
    static constexpr int SMEM = XQ * XBUF + BM * 4;
    // vector-memory operations a wave has issued after the x loads of step t + 1 when it reaches the
    // barrier of step t (slice 2): those of the steps between, and the W loads of slices 0 and 1
    static constexpr int VM_X = (XQ - 3) * (4 * WB + AL) + 2 * WB;
    // and after those of step 0 at the end of the prologue
    static constexpr int VM_X0 = (RS - 1) * WB + (XQ - 2) * AL;
    static_assert(XQ >= 4 && (RS == 8 || RS == 4) && BMB * 4 % NW == 0 && SMEM <= 160 * 1024 && VM_X < 64 &&
                  VM_X0 < 64 && WA <= 15, "tile");
};

// The fragment of block i at OFF past `base`, blocks STRIDE bytes apart.
template <int STRIDE, int OFF = 0>
__device__ __forceinline__ half8_t ds_read_b128_by(uint32_t base, int i)
{
    half8_t v;
    asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(v) : "v"(base), "i"(OFF + STRIDE * i));
    return v;
}

// Wait until at most N LDS operations of this wave are outstanding (they complete in issue order; the
// loop issues no scalar loads).
template <int N>
__device__ __forceinline__ void lds_wait_n()
{
    asm volatile("s_waitcnt lgkmcnt(%0)" ::"i"(N));
}

// The accumulators times the row scales `rs` (of the tile's rows, in LDS) into y. D layout of a 32 x 32
// tile: lane holds column lane & 31, register r row 8 (r >> 2) + 4 (lane >> 5) + (r & 3).
template <class T>
__device__ __forceinline__ void frag_store(const floatx16_t (&acc)[T::WA][T::WB], const float* rs, float* __restrict__ y,
                                           int M, int N, int ldy, int mt, int nt, int wr, int wc)
{
    const int lane = (int)threadIdx.x & 63, h = lane >> 5;
    const int m0 = mt * T::BM, n0 = nt * T::BN + wc * T::WB * 32 + (lane & 31);
#pragma unroll
    for (int i = 0; i < T::WA; ++i)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int r0 = 32 * (wr * T::WA + i) + 8 * q + 4 * h;
            const f32x4_t s4 = *reinterpret_cast<const f32x4_t*>(rs + r0);
#pragma unroll
            for (int j = 0; j < T::WB; ++j) {
                const int n = n0 + 32 * j;
                if (n >= N) continue;
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const int m = m0 + r0 + e;
                    if (m < M) y[(size_t)m * ldy + n] = acc[i][j][4 * q + e] * s4[e];
                }
            }
        }
}

// One block tile. xf, wf: panels of S fragments (S a multiple of 8); RB, CB: panels of x and of W; y row
// stride ldy; rows past M and columns past N are not stored (panels past the last repeat it).
template <class T>
__device__ __forceinline__ void frag_tile_run(unsigned char* smem, const uint16_t* __restrict__ xf,
                                              const float* __restrict__ rscale, const uint16_t* __restrict__ wf,
                                              float* __restrict__ y, int M, int N, int ldy, int S, int RB, int CB,
                                              int mt, int nt)
{
    constexpr int WA = T::WA, WB = T::WB, XQ = T::XQ, AL = T::AL;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wr = wave / T::WC, wc = wave % T::WC;
    const brsrc_t rx = make_rsrc(xf, (uint32_t)((size_t)RB * S * 1024));
    const brsrc_t rw = make_rsrc(wf, (uint32_t)((size_t)CB * S * 1024));
    const uint32_t voff = (uint32_t)lane * 16;
    const int steps = S / 4;                         // even

    // panel bases (bytes) of this wave's direct loads (load i of a step: 1 KiB piece 4 of panel
    // (NW i + wave) / 4) and of its W columns
    uint32_t xbase[AL], wbase[WB];
#pragma unroll
    for (int i = 0; i < AL; ++i) {
        const int q = T::NW * i + wave;
        xbase[i] = (uint32_t)(min(mt * T::BMB + (q >> 2), RB - 1) * S + (q & 3)) * 1024u;
    }
#pragma unroll
    for (int j = 0; j < WB; ++j) wbase[j] = (uint32_t)(min(nt * T::BNB + wc * WB + j, CB - 1) * S) * 1024u;

    auto load_x = [&](int i, int step, uint32_t buf) {
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rx, (lds_void_t*)(smem + buf + (T::NW * i + wave) * 1024), 16, voff,
                                                 (int)(xbase[i] + (uint32_t)step * 4096u), 0, 0);
    };
    auto load_w = [&](int j, int slice) {
        return __builtin_bit_cast(half8_t, __builtin_amdgcn_raw_buffer_load_b128(
                                               rw, voff, (int)(wbase[j] + (uint32_t)slice * 1024u), 0));
    };

    const float rs_row = tid < T::BM ? rscale[min(mt * T::BM + tid, M - 1)] : 0.f;
    half8_t a[WA], b[T::RS][WB];
    floatx16_t acc[WA][WB];
#pragma unroll
    for (int i = 0; i < WA; ++i)
#pragma unroll
        for (int j = 0; j < WB; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;

    // Prologue, in the order the steps keep (so the waits the compiler derives at the loop's head are those
    // of every step): x steps 0 .. XQ - 4, then W slices 0 .. RS - 2 with x steps XQ - 3 and XQ - 2 among them.
    auto load_x_half = [&](int part, int step, uint32_t buf) {
#pragma unroll
        for (int i = part ? T::AL0 : 0; i < (part ? AL : T::AL0); ++i) load_x(i, min(step, steps - 1), buf);
        __builtin_amdgcn_sched_barrier(0);
    };
#pragma unroll
    for (int q = 0; q < XQ - 3; ++q) {
        load_x_half(0, q, (uint32_t)(q * T::XBUF));
        load_x_half(1, q, (uint32_t)(q * T::XBUF));
    }
#pragma unroll
    for (int s = 1; s < 8; ++s) {                    // slice s of the two steps before step 0
        const int w = s + T::RS - 9;
        if (w >= 0) {
#pragma unroll
            for (int j = 0; j < WB; ++j) b[w][j] = load_w(j, w);
            __builtin_amdgcn_sched_barrier(0);
        }
        if (s == 2 || s == 3) load_x_half(s - 2, XQ - 3, (uint32_t)((XQ - 3) * T::XBUF));
        if (s == 6 || s == 7) load_x_half(s - 6, XQ - 2, (uint32_t)((XQ - 2) * T::XBUF));
    }
    wait_vm<T::VM_X0>();                             // x step 0
    step_barrier();
    if (tid < T::BM) store_rscale(lds_addr(smem + XQ * T::XBUF) + 4 * (uint32_t)tid, rs_row);
    const uint32_t abase = lds_addr(smem) + (uint32_t)(wr * WA * 4096) + voff;
#pragma unroll
    for (int i = 0; i < WA; ++i) a[i] = ds_read_b128_by<4096>(abase, i);

    // Step t multiplies x buffer xq. At slice 2 the wave waits for its own x loads of step t + 1 and meets
    // the others: after that step t + 1 may be read and the buffer of step t - 1 refilled (step
    // t + XQ - 1). Slice g loads W slice g + RS - 1 into the registers of slice g - 1. Loads past the end
    // are clamped and never used. The x fragment of a row block is read for the next slice into the same
    // registers right after the row's MFMAs, so WA - 1 younger reads are outstanding when it is needed.
    uint32_t xq = 0;
    int t = 0;
    do {
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            const uint32_t x1 = xq + 1 == (uint32_t)XQ ? 0u : xq + 1;
            const uint32_t xfill = xq == 0 ? (uint32_t)XQ - 1 : xq - 1;
            const int xstep = min(t + XQ - 1, steps - 1);
#pragma unroll
            for (int s = 0; s < 4; ++s) {
                constexpr int RS = T::RS;
                const int slot = (4 * u + s) % RS;
                if (s == 2) {
                    wait_vm<T::VM_X>();
                    asm volatile("s_barrier" ::: "memory");
                }
                const int wslice = min(4 * t + s + RS - 1, S - 1);
                const int nx = s == 2 ? T::AL0 : s == 3 ? AL - T::AL0 : 0, ops = WB + nx;
                const uint32_t anext = abase + (s == 3 ? x1 : xq) * T::XBUF;
#pragma unroll
                for (int i = 0; i < WA; ++i) {
                    lds_wait_n<WA - 1>();
                    tie(a[i]);
#pragma unroll
                    for (int j = 0; j < WB; ++j) {
                        acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a[i], b[slot][j], acc[i][j], 0, 0, 0);
                        __builtin_amdgcn_sched_barrier(0);
                        if (j == 0) {
#pragma unroll
                            for (int k = i * ops / WA; k < (i + 1) * ops / WA; ++k) {
                                if (k < WB) b[(slot + RS - 1) % RS][k] = load_w(k, wslice);
                                else load_x((s == 3 ? T::AL0 : 0) + k - WB, xstep, xfill * T::XBUF);
                            }
                            __builtin_amdgcn_sched_barrier(0);
                        }
                    }
                    a[i] = s == 0 ? ds_read_b128_by<4096, 1024>(anext, i) : s == 1 ? ds_read_b128_by<4096, 2048>(anext, i)
                         : s == 2 ? ds_read_b128_by<4096, 3072>(anext, i) : ds_read_b128_by<4096>(anext, i);
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
            xq = x1;
            ++t;
        }
    } while (t < steps);
    // the x fragments read for a step that does not run: landed before their registers are reused
    lds_wait();
#pragma unroll
    for (int i = 0; i < WA; ++i) tie(a[i]);
    wait_vm<0>();

    frag_store<T>(acc, reinterpret_cast<const float*>(smem + XQ * T::XBUF), y, M, N, ldy, mt, nt, wr, wc);
}

// Tile (row, column) of block b: blocks are dealt to the 8 XCDs round-robin, so each XCD takes a run of
// consecutive tiles, ordered in groups of 4 row tiles x all column tiles, which share panels in its L2.
__device__ __forceinline__ void frag_tile_of(int b, int nMT, int nNT, int& mt, int& nt)
{
    const int total = nMT * nNT, per = total / 8, extra = total % 8;
    const int xcd = b & 7, idx = b >> 3;
    const int k = xcd * per + min(xcd, extra) + idx;
    const int gsz = 4 * nNT, g = k / gsz, w = k - g * gsz;
    const int rows = min(4, nMT - 4 * g);
    mt = 4 * g + w % rows;
    nt = w / rows;
}

template <class T>
__device__ __forceinline__ void frag_gemm(const uint16_t* __restrict__ xf, const float* __restrict__ rscale,
                                          const uint16_t* __restrict__ wf, float* __restrict__ y, int M, int N,
                                          int ldy, int S)
{
    __shared__ __attribute__((aligned(1024))) unsigned char smem[T::SMEM];
    int mt, nt;
    frag_tile_of((int)blockIdx.x, (M + T::BM - 1) / T::BM, (N + T::BN - 1) / T::BN, mt, nt);
    frag_tile_run<T>(smem, xf, rscale, wf, y, M, N, ldy, S, (M + 31) / 32, (N + 31) / 32, mt, nt);
}

// ---- staging ------------------------------------------------------------------------------------

// Rows R g .. R g + R - 1 of x into fragments: 1024 threads, thread = (row tid % R, 8-float chunk tid / R of
// every 1024 / R), so a store of a wave writes runs of 16 R bytes. FRAG_CH chunks per thread are held in
// registers between the maximum and the store; longer rows are read twice. R = 8 for rows of up to
// FRAG_CH * 1024 elements, else 4: the kernel then stays within 64 VGPRs, two blocks per CU.
constexpr int FRAG_CH = 5;
static_assert(FRAG_CH * 1024 == BRIK_FRAG_ROWS8_MAX_K, "rows per staging block");

// Halves offset of 8-element chunk c (k = 8 c ..) of row r of panel rb: step c >> 4 of 128 k, lane half
// (c >> 3) & 1, slice c & 7 (gemm.hip's k mapping).
// NAT: slice c >> 1, half c & 1 (k = 16 s + 8 h + i), the f16-weight mapping.
template <bool NAT>
__device__ __forceinline__ size_t frag_chunk_at(int rb, int r, int c, int S)
{
    if constexpr (NAT) return ((size_t)rb * S + (c >> 1)) * 512 + (c & 1) * 256 + r * 8;
    return ((size_t)rb * S + 8 * (c >> 4) + (c & 7)) * 512 + ((c >> 3) & 1) * 256 + r * 8;
}

template <int R, bool NAT = false>
__device__ __forceinline__ void frag_rows(const float* __restrict__ x, uint16_t* __restrict__ xf,
                                          float* __restrict__ rscale, int g, int M, int K, int S, float (*wmax)[8])
{
    constexpr int CH = FRAG_CH, C = 1024 / R;          // chunks held, chunks per pass
    const int tid = threadIdx.x, r = tid % R, c0 = tid / R;
    const int m = R * g + r, nch = K / 8, nchp = S * 2;
    const float* xr = x + (size_t)min(m, M - 1) * K;
    f32x4_t v[CH][2];
    float mx = 0.f;
#pragma unroll
    for (int i = 0; i < CH; ++i) {
        const int c = c0 + C * i;
        v[i][0] = v[i][1] = f32x4_t{0.f, 0.f, 0.f, 0.f};
        if (c < nch) {
            v[i][0] = *(const f32x4_t*)(xr + c * 8);
            v[i][1] = *(const f32x4_t*)(xr + c * 8 + 4);
        }
    }
#pragma unroll
    for (int i = 0; i < CH; ++i) mx = fmaxf(mx, absmax8(v[i][0], v[i][1]));
    for (int c = c0 + C * CH; c < nch; c += C)
        mx = fmaxf(mx, absmax8(*(const f32x4_t*)(xr + c * 8), *(const f32x4_t*)(xr + c * 8 + 4)));
#pragma unroll
    for (int o = R; o < 64; o <<= 1) mx = fmaxf(mx, __shfl_xor(mx, o));
    if ((tid & 63) < R) wmax[tid >> 6][r] = mx;
    __syncthreads();
#pragma unroll
    for (int w = 0; w < 16; ++w) mx = fmaxf(mx, wmax[w][r]);
    if (m >= M) return;
    float down;
    const float up = xprep_up(mx, down);
    if (c0 == 0) rscale[m] = down;
    const int rb = m >> 5, rr = m & 31;
#pragma unroll
    for (int i = 0; i < CH; ++i) {
        const int c = c0 + C * i;
        if (c < nchp) *(half8_t*)(xf + frag_chunk_at<NAT>(rb, rr, c, S)) = to_h8_order<NAT>(v[i][0], v[i][1], up);
    }
    for (int c = c0 + C * CH; c < nchp; c += C) {
        f32x4_t p = {0.f, 0.f, 0.f, 0.f}, q = p;
        if (c < nch) {
            p = *(const f32x4_t*)(xr + c * 8);
            q = *(const f32x4_t*)(xr + c * 8 + 4);
        }
        *(half8_t*)(xf + frag_chunk_at<NAT>(rb, rr, c, S)) = to_h8_order<NAT>(p, q, up);
    }
}

// 32 columns x 128 k of W: lane 32 h + c dequantizes groups 4 t + 2 h and 4 t + 2 h + 1 of column c, the
// fragments of slices 8 t .. 8 t + 7. Groups past K and columns past N give zeros.
template <int FMT>
__device__ __forceinline__ void frag_dequant(const uint8_t* __restrict__ p0, const uint8_t* __restrict__ p1,
                                             const uint16_t* __restrict__ sc, const uint16_t* __restrict__ mn,
                                             uint16_t* __restrict__ wf, int n0, int N, int K, int cb, int t, int S)
{
    const int lane = threadIdx.x & 63, h = lane >> 5;
    const int G = K / BRIK_GROUP, n = n0 + 32 * cb + (lane & 31), g0 = 4 * t + 2 * h;
    const size_t gb = (size_t)min(n, N - 1) * G;
    WCodes<FMT> f;
#pragma unroll
    for (int e = 0; e < 2; ++e) {
        const size_t g = gb + min(g0 + e, G - 1);
        if constexpr (FMT == FMT_Q4) {
            const u32x4_t v = *(const u32x4_t*)(p0 + g * 16);
#pragma unroll
            for (int j = 0; j < 4; ++j) f.w[4 * e + j] = v[j];
        } else if constexpr (FMT == FMT_Q8) {
#pragma unroll
            for (int k = 0; k < 2; ++k) {
                const u32x4_t v = *(const u32x4_t*)(p0 + g * 32 + 16 * k);
#pragma unroll
                for (int j = 0; j < 4; ++j) f.w[8 * e + 4 * k + j] = v[j];
            }
        } else {
            const u32x2_t v = *(const u32x2_t*)(p0 + g * 8);
            f.w[2 * e] = v.x;
            f.w[2 * e + 1] = v.y;
            f.w[4 + e] = *(const uint32_t*)(p1 + g * 4);
        }
        f.s[e] = sc[g];
        f.m[e] = FMT == FMT_Q8 ? 0u : mn[g];
    }
#pragma unroll
    for (int e = 0; e < 2; ++e)
        if (g0 + e >= G || n >= N) f.s[e] = f.m[e] = 0u;
    const GroupOps go = group_ops<FMT>(f, DeqConst::make());
    uint16_t* dst = wf + ((size_t)cb * S + 8 * t) * 512 + lane * 8;
#pragma unroll
    for (int sl = 0; sl < 8; ++sl) *(half8_t*)(dst + sl * 512) = b_frag<FMT>(f, go, sl);
}

// Blocks [0, xblocks) stage 8 (4 past BRIK_FRAG_ROWS8_MAX_K) rows of x each; the others dequantize W, 16 waves of one 32 x 128 piece
// each (piece = column panel x step). xblocks == 0 when the rows were staged before.
template <int FMT>
__device__ __forceinline__ void frag_prep(const float* __restrict__ x, uint16_t* __restrict__ xf,
                                          float* __restrict__ rscale, const uint8_t* __restrict__ p0,
                                          const uint8_t* __restrict__ p1, const uint16_t* __restrict__ sc,
                                          const uint16_t* __restrict__ mn, uint16_t* __restrict__ wf, int M, int K,
                                          int n0, int N, int CB, int S, int xblocks)
{
    __shared__ float wmax[16][8];
    if ((int)blockIdx.x < xblocks) {
        if (K <= BRIK_FRAG_ROWS8_MAX_K) frag_rows<8>(x, xf, rscale, (int)blockIdx.x, M, K, S, wmax);
        else frag_rows<4>(x, xf, rscale, (int)blockIdx.x, M, K, S, wmax);
        return;
    }
    const int T = S / 8, item = ((int)blockIdx.x - xblocks) * 16 + (int)(threadIdx.x >> 6);
    const int cb = item / T;
    if (cb >= CB) return;
    frag_dequant<FMT>(p0, p1, sc, mn, wf, n0, N, K, cb, item % T, S);
}


// ---- f16 weights ----------------------------------------------------------------------------------
// The same product with W as given, [N, K] f16 rows (the reference's MATMUL_T_F16W, shaders.ts:2240-2259):
// re-laying W out would read and write it once more, so its rows go through LDS beside x, 32 k (64 bytes) of
// each row and step, by direct loads of 16 rows each, XQ - 2 steps ahead. The 16-byte chunk c of row r sits
// at chunk c ^ ((r >> 2) & 3) of its 64 bytes, so the 16 rows of a read phase touch all 64 banks. Both
// operands are in natural order: slice s, half h, element i is k = 16 s + 8 h + i.
// The tiled GEMM's f16 form loaded each W row 16 bytes per lane straight into registers, so a load touched 32
// lines, and its steps waited for them: 0.6 us and more per 128 k whatever the rows. What bounds this one
// is LDS (192 x 256 tile, per slice of 384 MFMA clocks: 40 KiB read, 14 KiB written) and, for small tiles,
// the load latency, hence 32-k steps and as many in flight as fit: 64-k steps in three buffers ran
// 256 x 128 at 42 us where six 32-k buffers run 34.9 (512 x 2560 x 9728). Per call, before -> after:
// M = 512, K = 2560, N = 9728 56 -> 40 us; M = 4096, K = 9728, N = 2560 421 -> 246 us (product 188 us,
// 1.08 PFLOP/s); M = 128, K = 2560, N = 1024 48 -> 16 us. Few rows (gemm_few.hip): M = 8, K = 9728, N = 2560
// 150 -> 15.6 us.
template <int WR_, int WC_, int WA_, int WB_, int XQ_>
struct HTile {
    static constexpr int WR = WR_, WC = WC_, WA = WA_, WB = WB_, XQ = XQ_;
    static constexpr int NW = WR * WC, NT = 64 * NW;
    static constexpr int BMB = WR * WA, BNB = WC * WB;
    static constexpr int BM = 32 * BMB, BN = 32 * BNB;
    static constexpr int XBUF = BMB * 2048, BUF = (BMB + BNB) * 2048;      // bytes of a step: x, then W rows
    // direct loads per wave and step (1 KiB pieces dealt round-robin; a wave without a last piece repeats it)
    static constexpr int AL = (BMB * 2 + NW - 1) / NW, BL = (BNB * 2 + NW - 1) / NW, LD = AL + BL;
    static constexpr int SMEM = XQ * BUF + BM * 4;
    static_assert(XQ >= 3 && SMEM <= 160 * 1024 && WA - 1 + WB <= 15 && (XQ - 2) * LD < 64, "tile");
};

template <class T>
__device__ __forceinline__ void f16_tile_run(unsigned char* smem, const uint16_t* __restrict__ xf,
                                             const float* __restrict__ rscale, const uint16_t* __restrict__ w,
                                             float* __restrict__ y, int M, int N, int K, int S, int RB, int mt, int nt)
{
    constexpr int WA = T::WA, WB = T::WB, XQ = T::XQ, LD = T::LD;
    const int tid = threadIdx.x, lane = tid & 63, h = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wr = wave / T::WC, wc = wave % T::WC;
    const brsrc_t rx = make_rsrc(xf, (uint32_t)((size_t)RB * S * 1024));
    const brsrc_t rw = make_rsrc(w, (uint32_t)((size_t)N * K * 2));
    const uint32_t voff = (uint32_t)lane * 16;
    const int steps = S / 2, full = K / 32;          // full: steps of 32 live k

    uint32_t xbase[T::AL], woff[T::BL], xdst[T::AL], wdst[T::BL];
#pragma unroll
    for (int i = 0; i < T::AL; ++i) {
        const int q = min(T::NW * i + wave, T::BMB * 2 - 1);
        xbase[i] = (uint32_t)(min(mt * T::BMB + (q >> 1), RB - 1) * S + (q & 1)) * 1024u;
        xdst[i] = (uint32_t)q * 1024u;
    }
#pragma unroll
    for (int i = 0; i < T::BL; ++i) {
        const int q = min(T::NW * i + wave, T::BNB * 2 - 1), r = 16 * q + (lane >> 2);
        woff[i] = (uint32_t)min(nt * T::BN + r, N - 1) * (uint32_t)K * 2u + (uint32_t)(((lane & 3) ^ ((r >> 2) & 3)) * 16);
        wdst[i] = (uint32_t)(T::XBUF + q * 1024);
    }
    // W's step is in its vector offset, moved on by each load: the range check of a buffer load leaves the scalar
    // offset out, and the last step of the last row may run up to 48 bytes past the end of W. Steps past the last
    // read a next row's values or nothing.
    auto load = [&](int u, int step, uint32_t buf) {
        if (u < T::AL)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rx, (lds_void_t*)(smem + buf + xdst[u]), 16, voff,
                                                     (int)(xbase[u] + (uint32_t)step * 2048u), 0, 0);
        else {
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rw, (lds_void_t*)(smem + buf + wdst[u - T::AL]), 16,
                                                     woff[u - T::AL], 0, 0, 0);
            woff[u - T::AL] += 64;
        }
    };

    const float rs_row = tid < T::BM ? rscale[min(mt * T::BM + tid, M - 1)] : 0.f;
    half8_t a[WA], b[2][WB];
    floatx16_t acc[WA][WB];
#pragma unroll
    for (int i = 0; i < WA; ++i)
#pragma unroll
        for (int j = 0; j < WB; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;
#pragma unroll
    for (int q = 0; q < XQ - 1; ++q)
#pragma unroll
        for (int u = 0; u < LD; ++u) load(u, min(q, steps - 1), (uint32_t)(q * T::BUF));
    wait_vm<(XQ - 2) * LD>();                        // step 0
    step_barrier();
    if (tid < T::BM) store_rscale(lds_addr(smem + XQ * T::BUF) + 4 * (uint32_t)tid, rs_row);
    const uint32_t abase = lds_addr(smem) + (uint32_t)(wr * WA * 2048) + voff;
    uint32_t boff[2];                                // W fragment of slice s: row lane & 31, chunk 2 s + h
#pragma unroll
    for (int s = 0; s < 2; ++s)
        boff[s] = lds_addr(smem) + T::XBUF + (uint32_t)(wc * WB * 2048 + (lane & 31) * 64) +
                  (uint32_t)(((2 * s + h) ^ ((lane >> 2) & 3)) * 16);
#pragma unroll
    for (int j = 0; j < WB; ++j) b[0][j] = ds_read_b128_by<2048>(boff[0], j);
#pragma unroll
    for (int i = 0; i < WA; ++i) a[i] = ds_read_b128_by<2048>(abase, i);
    // every LDS and scalar operation so far: the loop's counted waits then count LDS reads alone
    lds_wait();

    // Step t multiplies buffer xq; at slice 1 the wave waits for its loads of step t + 1 and meets the others,
    // then loads step t + XQ - 1 into the buffer of step t - 1. W fragments are read a slice ahead, x
    // fragments into the registers of the row just multiplied.
    uint32_t xq = 0;
    for (int t = 0; t < full; ++t) {
        const uint32_t x1 = xq + 1 == (uint32_t)XQ ? 0u : xq + 1, xfill = xq == 0 ? (uint32_t)XQ - 1 : xq - 1;
        const int fill = min(t + XQ - 1, steps - 1);
#pragma unroll
        for (int s = 0; s < 2; ++s) {
            const int cur = s, nxt = s ^ 1;
            const uint32_t nb = (s == 1 ? x1 : xq) * T::BUF;
            if (s == 1) {
                wait_vm<(XQ - 3) * LD>();
                asm volatile("s_barrier" ::: "memory");
            }
#pragma unroll
            for (int i = 0; i < WA; ++i) {
                if (i == 0) {
                    lds_wait_n<WA - 1>();
#pragma unroll
                    for (int j = 0; j < WB; ++j) tie(b[cur][j]);
                } else {
                    lds_wait_n<WA - 1 + WB>();
                }
                tie(a[i]);
                if (i == 0) {
#pragma unroll
                    for (int j = 0; j < WB; ++j) b[nxt][j] = ds_read_b128_by<2048>(boff[nxt] + nb, j);
                }
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int j = 0; j < WB; ++j) {
                    acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a[i], b[cur][j], acc[i][j], 0, 0, 0);
                    __builtin_amdgcn_sched_barrier(0);
                    if (s == 1) {
                        const int o = i * WB + j;
#pragma unroll
                        for (int u = o * LD / (WA * WB); u < (o + 1) * LD / (WA * WB); ++u) load(u, fill, xfill * T::BUF);
                        __builtin_amdgcn_sched_barrier(0);
                    }
                }
                a[i] = s == 0 ? ds_read_b128_by<2048, 1024>(abase + nb, i) : ds_read_b128_by<2048>(abase + nb, i);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        xq = x1;
    }
    lds_wait();
#pragma unroll
    for (int i = 0; i < WA; ++i) tie(a[i]);
#pragma unroll
    for (int j = 0; j < WB; ++j) tie(b[0][j]);
    wait_vm<0>();
    if (steps > full) {
        // the last step's K - 32 full live k: chunks past K hold a next row's values or none, taken as zeros
        lds_barrier();                               // every wave's loads of the step have landed
        const uint32_t nb = xq * T::BUF;
#pragma unroll
        for (int s = 0; s < 2; ++s) {
            if (32 * full + 16 * s >= K) break;
            const bool live = 32 * full + 16 * s + 8 * h < K;
            half8_t bt[WB];
#pragma unroll
            for (int j = 0; j < WB; ++j) {
                u32x4_t v = *(const u32x4_t*)(smem + nb + (boff[s] - lds_addr(smem)) + 2048 * j);
#pragma unroll
                for (int e = 0; e < 4; ++e) v[e] = live ? v[e] : 0u;
                bt[j] = __builtin_bit_cast(half8_t, v);
            }
#pragma unroll
            for (int i = 0; i < WA; ++i) {
                const half8_t at = *(const half8_t*)(smem + nb + wr * WA * 2048 + lane * 16 + 1024 * s + 2048 * i);
#pragma unroll
                for (int j = 0; j < WB; ++j)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(at, bt[j], acc[i][j], 0, 0, 0);
            }
        }
    }
    frag_store<T>(acc, reinterpret_cast<const float*>(smem + XQ * T::BUF), y, M, N, N, mt, nt, wr, wc);
}

template <class T>
__device__ __forceinline__ void f16_gemm(const uint16_t* __restrict__ xf, const float* __restrict__ rscale,
                                         const uint16_t* __restrict__ w, float* __restrict__ y, int M, int N, int K,
                                         int S)
{
    __shared__ __attribute__((aligned(1024))) unsigned char smem[T::SMEM];
    int mt, nt;
    frag_tile_of((int)blockIdx.x, (M + T::BM - 1) / T::BM, (N + T::BN - 1) / T::BN, mt, nt);
    f16_tile_run<T>(smem, xf, rscale, w, y, M, N, K, S, (M + 31) / 32, mt, nt);
}

}  // namespace

#define BRIK_FRAG_PREP(FMTN, FMT)                                                                         \
    extern "C" __global__ __launch_bounds__(1024, 8) void brik_frag_prep_##FMTN(                             \
        const float* __restrict__ x, uint16_t* __restrict__ xf, float* __restrict__ rscale,               \
        const uint8_t* __restrict__ p0, const uint8_t* __restrict__ p1, const uint16_t* __restrict__ sc,  \
        const uint16_t* __restrict__ mn, uint16_t* __restrict__ wf, int M, int K, int n0, int N, int CB,  \
        int S, int xblocks)                                                                               \
    {                                                                                                     \
        frag_prep<FMT>(x, xf, rscale, p0, p1, sc, mn, wf, M, K, n0, N, CB, S, xblocks);                   \
    }
BRIK_FRAG_PREP(q4, FMT_Q4) BRIK_FRAG_PREP(q8, FMT_Q8) BRIK_FRAG_PREP(q3, FMT_Q3)

// Fragment GEMM kernels: brik_gemm_frag_<WR><WC>_<WA>x<WB> (block tile 32 WR WA x 32 WC WB), in the order
// of the runtime's table (kFragTiles).
#define BRIK_GEMM_FRAG(WR, WC, WA, WB, XQ, RS)                                                            \
    extern "C" __global__ __launch_bounds__(64 * WR * WC) void brik_gemm_frag_##WR##WC##_##WA##x##WB(     \
        const uint16_t* __restrict__ xf, const float* __restrict__ rscale, const uint16_t* __restrict__ wf, \
        float* __restrict__ y, int M, int N, int ldy, int S)                                              \
    {                                                                                                     \
        frag_gemm<FTile<WR, WC, WA, WB, XQ, RS>>(xf, rscale, wf, y, M, N, ldy, S);                        \
    }
#ifndef BRIK_FRAG_TILES
#define BRIK_FRAG_TILES(X) X(2, 4, 3, 2, 4, 4) X(1, 8, 4, 1, 4, 8) X(1, 4, 4, 1, 4, 8) X(1, 4, 2, 1, 4, 8)
#endif
BRIK_FRAG_TILES(BRIK_GEMM_FRAG)

// Rows of x in natural order for the f16-weight GEMM (S slices of 16 k per panel, zeros past K).
extern "C" __global__ __launch_bounds__(1024, 8) void brik_frag_rows_f16(const float* __restrict__ x,
                                                                         uint16_t* __restrict__ xf,
                                                                         float* __restrict__ rscale, int M, int K,
                                                                         int S)
{
    __shared__ float wmax[16][8];
    if (K <= BRIK_FRAG_ROWS8_MAX_K) frag_rows<8, true>(x, xf, rscale, (int)blockIdx.x, M, K, S, wmax);
    else frag_rows<4, true>(x, xf, rscale, (int)blockIdx.x, M, K, S, wmax);
}

// f16-weight GEMM kernels: brik_gemm_h_<WR><WC>_<WA>x<WB>, in the order of the runtime's table (kHalfTiles).
#define BRIK_GEMM_H(WR, WC, WA, WB, XQ)                                                                   \
    extern "C" __global__ __launch_bounds__(64 * WR * WC) void brik_gemm_h_##WR##WC##_##WA##x##WB(        \
        const uint16_t* __restrict__ xf, const float* __restrict__ rscale, const uint16_t* __restrict__ w, \
        float* __restrict__ y, int M, int N, int K, int S)                                                \
    {                                                                                                     \
        f16_gemm<HTile<WR, WC, WA, WB, XQ>>(xf, rscale, w, y, M, N, K, S);                                \
    }
#ifndef BRIK_HALF_TILES
#define BRIK_HALF_TILES(X) X(2, 4, 3, 2, 5) X(4, 2, 2, 2, 6) X(4, 2, 1, 2, 5) X(2, 2, 1, 1, 9)
#endif
BRIK_HALF_TILES(BRIK_GEMM_H)
