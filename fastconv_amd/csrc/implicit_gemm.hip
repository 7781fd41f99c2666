// Implicit-GEMM convolution on gfx950 fp32 MFMA:
//   y[n][k][oh][ow] = sum_{c,r,s} w[k][c][r][s] * x[n][c][oh*sh + r - pt][ow*sw + s - pl]
// seen as D[K][N*OH*OW] = Wp^T[K][Kred] * col[Kred][N*OH*OW], where the column
// matrix is never written to memory: each workgroup gathers its BK x BN slice of
// it straight into LDS.  The filter is re-laid once to Wp[Kred_pad][K_pad]
// (output channel fastest) so that its tiles are straight 16-byte copies, as in
// the Winograd GEMM.
#include <algorithm>
#include <cmath>
#include <cstdio>
#include <mutex>
#include <type_traits>
#include <utility>

#include "fc_internal.h"
#include "split_mfma.h"

namespace {

typedef float floatx16 __attribute__((ext_vector_type(16)));
typedef float floatx4 __attribute__((ext_vector_type(4)));   // native vector: arrays of it stay in registers

// Order of the reduction index.  Channel-major (the column-matrix rows of
// convLayer/im2colConv.cpp:285-309): kred = (c*kh + r)*kw + s.  Tap-major, used whenever the channel
// count is a whole number of LDS stages (C % BK == 0): kred = (r*kw + s)*C + c, so that the BK rows of a
// stage share one filter tap -- one in-image test and one window offset per stage instead of one per
// gathered element, and consecutive rows are consecutive channels (no table lookups in the loop).
// The packed filter and the row table follow whichever order the layer uses.
// The split kernel (igemm_split_kernel) has orders of its own, padded so that a lane's 8 rows can be read without a look at
// each: blocks of 16 channels, tap by tap within a block, so that the taps of a block find its pixels in the cache (tap-major
// reads the whole input once per tap: 400 -> 32 channels 3x3/2 at 153x153, batch 12, 370 us against 221); or channel-major with every window row in runs of 8 or 4 columns.
// Row table entry for reduction row kred (tap (r, s) of channel c):
//   [2*kred]   = c*H*W + r*W + s      (offset from the window origin)
//   [2*kred+1] = r << 16 | s          (31 << 16 | 31 for padding rows: a mask bit that is never set)
enum { IG_ORDER_CHANNEL, IG_ORDER_TAP, IG_ORDER_BLOCK, IG_ORDER_ROW8, IG_ORDER_ROW4 };

__global__ __launch_bounds__(256) void igemm_pack_filter_kernel(const float *__restrict__ w,
                                                                float *__restrict__ Wp,
                                                                int32_t *__restrict__ table, int K, int C,
                                                                int kh, int kw, int H, int W, int rows,
                                                                int Kred_pad, int K_pad, int order) {
    const int k = blockIdx.x * 64 + (threadIdx.x & 63);
    for (int kred = blockIdx.y * 4 + (threadIdx.x >> 6); kred < Kred_pad; kred += 4 * gridDim.y) {
        int c = 0, r = 31, s = 31;
        bool real = kred < rows;
        if (real) {
            if (order == IG_ORDER_TAP) {
                const int t = kred / C;
                c = kred - t * C;
                r = t / kw;
                s = t - r * kw;
            } else if (order == IG_ORDER_BLOCK) {
                const int stage = kred / 16, block = stage / (kh * kw), t = stage - block * (kh * kw);
                c = block * 16 + kred % 16;
                r = t / kw;
                s = t - r * kw;
                real = c < C;
            } else {
                const int run = order == IG_ORDER_ROW8 ? 8 : order == IG_ORDER_ROW4 ? 4 : 1;
                const int width = (kw + run - 1) / run * run;      // rows of the reduction per window row
                c = kred / (kh * width);
                const int rs = kred - c * kh * width;
                r = rs / width;
                s = rs - r * width;
                real = s < kw;
            }
        }
        if (k < K_pad)
            Wp[(size_t)kred * K_pad + k] = (k < K && real) ? w[((size_t)k * C + c) * (kh * kw) + r * kw + s] : 0.f;
        if (blockIdx.x == 0 && (threadIdx.x & 63) == 0) {
            table[2 * kred] = real ? c * H * W + r * W + s : 0;
            table[2 * kred + 1] = real ? (r << 16) | s : (31 << 16) | 31;
        }
    }
}

// 16-byte words of 32 output channels and one stage of the split filter: three parts x two halves of 8 rows x 32 channels.
constexpr int kSplitBlockWords = 3 * 64;

struct IgemmParams {
    const float *x;
    const float *Wp;
    const fc_uintx4 *Ws;           // the filter split into its parts, where products are split
    const int32_t *table;
    const float *bias;
    float *y;
    int N, C, H, W, K, OH, OW, kh, kw, sh, sw, pt, pl, relu;
    int Kred_pad, K_pad;
    long Npix;
    int nKB, nPB;
    int splitK, stagesPerSplit;   // reduction split over blockIdx.y; partial sums go to ws
    int sumStages;                // split products in two levels of sums: stages added up in the first
    float *ws;                    // [splitK][K][Npix] when splitK > 1
    long xBytes;                  // size of the input tensor
    int fastStore;                // K is a whole number of tiles, every output byte offset fits 32 bits, bias 16-byte aligned
    fc_fastdiv divOHW, divOW;
    // row orders: pixels and stages past which no run of window columns starts before x (ig_before)
    long pixBefore;
    int stagesBefore;
};

template <int BM, int BN, int BK, int WGM, int WGN>
struct IgTile {
    static constexpr int BM_ = BM, BN_ = BN, BK_ = BK, WGM_ = WGM, WGN_ = WGN;
    static constexpr int THREADS = 64 * WGM * WGN;
    static constexpr int WM = BM / WGM, WN = BN / WGN;
    static constexpr int MI = WM / 32, NI = WN / 32;
    static constexpr int A_VEC = BK * BM / 4;
    static constexpr int A_LD = A_VEC / THREADS;
    static constexpr int A_ROWS = THREADS * 4 / BM;     // filter-tile rows per copy pass
    static constexpr int ROW_STEP = THREADS / BN;       // gather: one column, every ROW_STEP-th row
    static constexpr int B_LD = BK / ROW_STEP;
    static constexpr int LDS_BYTES = 2 * BK * (BM + BN) * 4;
    // wavefronts per SIMD the register allocation must leave room for (the second argument of
    // __launch_bounds__ in HIP): four for the four-wavefront tiles up to 128x128 and 64x256
    static constexpr int MIN_WAVES = (BM * BN <= 128 * 128 && WGM * WGN == 4) ? 4 : 1;
    static_assert(THREADS % BN == 0 && BK % ROW_STEP == 0, "gather mapping");
    static_assert(BN % 64 == 0, "a wavefront gathers one row of the column matrix");
    static_assert(A_VEC % THREADS == 0 && A_LD >= 1, "every thread copies the same number of float4");
    static_assert(WM % 32 == 0 && WN % 32 == 0, "wave tile must be whole 32x32 MFMA blocks");
};

// Copy passes as pack expansions (literal register-array indices, see wino_gemm.hip).
template <int... I>
__device__ __forceinline__ void ig_load_rows(floatx4 (&r)[sizeof...(I)], const float *p, size_t rowStride,
                                             std::integer_sequence<int, I...>) {
    ((r[I] = *reinterpret_cast<const floatx4 *>(p + (size_t)I * rowStride)), ...);
}
// The same from a base all lanes share (scalar registers) and one 32-bit byte offset per lane: no vector
// instruction goes into the addresses (see load_rows in wino_gemm.hip).
template <int... I>
__device__ __forceinline__ void ig_load_rows_at(floatx4 (&r)[sizeof...(I)], const float *base, uint32_t laneOff, size_t rowStride,
                                                std::integer_sequence<int, I...>) {
    asm volatile("" : "+v"(laneOff));
    const float *b = uniform_ptr(base);
    ((r[I] = *reinterpret_cast<const floatx4 *>(reinterpret_cast<const char *>(b) + laneOff), b = uniform_ptr(b + rowStride)), ...);
}
template <int... I>
__device__ __forceinline__ void ig_store_rows(float *lds, const floatx4 (&r)[sizeof...(I)], int rowStride,
                                              std::integer_sequence<int, I...>) {
    ((*reinterpret_cast<floatx4 *>(lds + I * rowStride) = r[I]), ...);
}

// One gathered element of the column matrix.  The row (reduction index) is the same
// for the whole wavefront, so its table entry lives in scalar registers; the
// per-pixel part of the bounds test is two bit masks computed once per thread.
// The load is unconditional (an element outside the image reads the start of the image
// instead) and its value is not touched here: whether it counts is recorded as bit `slot`
// of `okBits` and applied when the element is written to LDS, so that the loads of a
// stage stay in flight under the MFMAs of the stage before.
// MASKED = false: no test at all (kept for completeness; the buffer modes below serve such layers).
template <bool MASKED>
__device__ __forceinline__ float ig_gather(const float *ximg, int pixOff, uint32_t maskR, uint32_t maskS,
                                           const int32_t *table, int kred, int slot, uint32_t &okBits) {
    const int off = table[2 * kred];
    if (!MASKED) return ximg[pixOff + off];
    const int rs = table[2 * kred + 1];
    const bool ok = ((maskR >> (rs >> 16)) & (maskS >> (rs & 0xffff)) & 1u) != 0;
    okBits |= ok ? (1u << slot) : 0u;
    return ximg[ok ? pixOff + off : 0];
}
template <bool MASKED, int... I>
__device__ __forceinline__ uint32_t ig_gather_rows(float (&r)[sizeof...(I)], const float *ximg, int pixOff,
                                                   uint32_t maskR, uint32_t maskS, const int32_t *table, int kred0,
                                                   int rowStep, std::integer_sequence<int, I...>) {
    uint32_t okBits = 0;
    ((r[I] = ig_gather<MASKED>(ximg, pixOff, maskR, maskS, table, kred0 + I * rowStep, I, okBits)), ...);
    return okBits;
}
template <bool MASKED, int... I>
__device__ __forceinline__ void ig_scatter_rows(float *lds, const float (&r)[sizeof...(I)], uint32_t okBits, int rowStride,
                                                std::integer_sequence<int, I...>) {
    ((lds[I * rowStride] = (!MASKED || ((okBits >> I) & 1u)) ? r[I] : 0.f), ...);
}

// The same element through a buffer resource over the whole input tensor (tensors below 2 GiB): the
// address is one 32-bit byte offset from a scalar base, and a tap outside the image gets bit 31 of
// its offset set, which puts it past the end of the buffer: the hardware's range check returns 0
// for it without touching memory.  No 64-bit address arithmetic, no select at the LDS write.
// invLo / invHi: bit t = r*kw + s is set when tap (r, s) of this thread's pixel lies outside the
// image (taps 64 and up, which only padding rows of the reduction name, count as outside).
template <bool MASKED>
__device__ __forceinline__ float ig_gather_buf(__amdgpu_buffer_rsrc_t xres, uint32_t pixByte, uint32_t invLo, uint32_t invHi,
                                               const int32_t *table, int kred, int kw) {
    uint32_t voff = pixByte + 4u * (uint32_t)table[2 * kred];
    if (MASKED) {
        const int rs = table[2 * kred + 1];
        const uint32_t t = (uint32_t)(rs >> 16) * (uint32_t)kw + (uint32_t)(rs & 0xffff);     // wave-uniform
        const uint32_t word = t < 32u ? invLo : invHi;
        const uint32_t bad = t < 64u ? (word >> (t & 31u)) & 1u : 1u;
        voff |= bad << 31;
    }
    return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(xres, voff, 0, 0));
}
template <bool MASKED, int... I>
__device__ __forceinline__ void ig_gather_rows_buf(float (&r)[sizeof...(I)], __amdgpu_buffer_rsrc_t xres, uint32_t pixByte,
                                                   uint32_t invLo, uint32_t invHi, const int32_t *table, int kred0, int rowStep,
                                                   int kw, std::integer_sequence<int, I...>) {
    ((r[I] = ig_gather_buf<MASKED>(xres, pixByte, invLo, invHi, table, kred0 + I * rowStep, kw)), ...);
}

// How the B tile (a slice of the column matrix) reaches LDS.  IG_GATHER is the fallback of the two
// buffer modes for input tensors of 2 GiB and more.
// IG_TAP_*: the buffer gather for tap-major layers (see igemm_pack_filter_kernel).
enum { IG_GATHER = 0, IG_POINTWISE = 1, IG_BUF_MASKED = 2, IG_TAP_MASKED = 3, IG_TAP_INSIDE = 4 };

// Workgroups are dealt to the 8 XCDs round-robin by linear id, and every XCD has an L2 of its own.
// Tiles are numbered pixel block major, output-channel block minor, and every XCD owns a contiguous
// eighth of that sequence: the output-channel blocks that share one block of gathered pixels run
// side by side on ONE XCD and find the pixels in its L2 (dealt round-robin, every XCD would fetch
// every pixel block: measured 4-6x the algorithmic traffic on the ResNet-50 projections).
// Returns false for a workgroup past the last tile.
__device__ __forceinline__ bool ig_decode_tile(const IgemmParams &p, int *kb, int *pb) {
    const int nTiles = p.nKB * p.nPB, perXcd = (nTiles + 7) >> 3;
    const int tileId = (blockIdx.x & 7) * perXcd + (blockIdx.x >> 3);
    if ((int)(blockIdx.x >> 3) >= perXcd || tileId >= nTiles) return false;
    *pb = tileId / p.nKB;
    *kb = tileId - *pb * p.nKB;
    return true;
}

// The accumulators of a workgroup tile to y, with this bias and ReLU, or to this split's partial sums.
// REPLACE: the sums are there already, without bias and ReLU; those that are not finite give way to the accumulators.
template <class TL, bool REPLACE = false>
__device__ __forceinline__ void ig_store_tile(const floatx16 (&acc)[TL::MI][TL::NI], const IgemmParams &p, const float *bias, int relu,
                                              int kb, int pb, int wm0, int wn0, int lrow, int lcol) {
    auto sum = [](const float *there, float v) __attribute__((always_inline)) { return REPLACE && __builtin_isfinite(*there) ? *there : v; };
    constexpr int BM = TL::BM_, BN = TL::BN_, MI = TL::MI, NI = TL::NI;
    // epilogue: column = pixel (lane%32), rows = output channels.  Register i of an accumulator
    // block is row 8*(i/4) + 4*(lane/32) + i%4: element (row r, column c) of the tile goes to
    // dst[colOff(c) + (rowBase + r) * rowStride], with dst = y (colOff = n*K*OHW + pixel in image,
    // rowStride = OHW) or the partial-sum slab of this split (colOff = pixel, rowStride = Npix).
    const int OHW = p.OH * p.OW;
    const bool partial = p.splitK > 1;
    const int rowBase = kb * BM + wm0 + 4 * lrow;
    if (p.fastStore) {
        // every row of the tile is a real output channel and every byte offset fits 32 bits: a
        // scalar base, one 32-bit offset per store, no predicates
        char *dst = reinterpret_cast<char *>(partial ? p.ws : p.y);
        const uint32_t rowStride = 4u * (partial ? (uint32_t)p.Npix : (uint32_t)OHW);      // bytes
        const uint32_t slab = partial ? (uint32_t)blockIdx.y * (uint32_t)p.K * (uint32_t)p.Npix : 0u;
        const bool plain = partial || (bias == nullptr && !relu);
#pragma unroll
        for (int ni = 0; ni < NI; ni++) {
            const long opix = (long)pb * BN + wn0 + ni * 32 + lcol;
            if (opix >= p.Npix) continue;
            uint32_t off;
            if (partial) {
                off = slab + (uint32_t)opix;
            } else {
                const uint32_t n = fc_div((uint32_t)opix, p.divOHW);
                off = n * (uint32_t)p.K * (uint32_t)OHW + ((uint32_t)opix - n * (uint32_t)OHW);
            }
            off = 4u * off + (uint32_t)rowBase * rowStride;
            if (plain) {
#pragma unroll
                for (int mi = 0; mi < MI; mi++)
#pragma unroll
                    for (int i = 0; i < 16; i++) {
                        float *d = reinterpret_cast<float *>(dst + (off + (uint32_t)(mi * 32 + 8 * (i / 4) + (i % 4)) * rowStride));
                        *d = sum(d, acc[mi][ni][i]);
                    }
            } else {
#pragma unroll
                for (int mi = 0; mi < MI; mi++)
#pragma unroll
                    for (int q = 0; q < 4; q++) {
                        floatx4 bq = {0.f, 0.f, 0.f, 0.f};
                        if (bias) bq = *reinterpret_cast<const floatx4 *>(bias + rowBase + mi * 32 + 8 * q);
#pragma unroll
                        for (int j = 0; j < 4; j++) {
                            float *d = reinterpret_cast<float *>(dst + (off + (uint32_t)(mi * 32 + 8 * q + j) * rowStride));
                            float v = sum(d, acc[mi][ni][q * 4 + j]) + bq[j];
                            if (relu) v = __builtin_elementwise_maximum(v, 0.f);      // keeps a NaN
                            *d = v;
                        }
                    }
            }
        }
        return;
    }
    if (partial) {
        // partial sums, [split][k][pixel]; igemm_reduce_kernel adds them up in split order
        float *wz = p.ws + (size_t)blockIdx.y * p.K * p.Npix;
#pragma unroll
        for (int ni = 0; ni < NI; ni++) {
            const long opix = (long)pb * BN + wn0 + ni * 32 + lcol;
            if (opix >= p.Npix) continue;
#pragma unroll
            for (int mi = 0; mi < MI; mi++)
#pragma unroll
                for (int i = 0; i < 16; i++) {
                    const int k = rowBase + mi * 32 + 8 * (i / 4) + (i % 4);
                    if (k < p.K) {
                        float *d = wz + (size_t)k * p.Npix + opix;
                        *d = sum(d, acc[mi][ni][i]);
                    }
                }
        }
        return;
    }
#pragma unroll
    for (int ni = 0; ni < NI; ni++) {
        const long opix = (long)pb * BN + wn0 + ni * 32 + lcol;
        if (opix >= p.Npix) continue;
        const uint32_t n = fc_div((uint32_t)opix, p.divOHW);
        const uint32_t pp = (uint32_t)opix - n * (uint32_t)OHW;
        float *yn = p.y + (size_t)n * p.K * OHW + pp;
#pragma unroll
        for (int mi = 0; mi < MI; mi++)
#pragma unroll
            for (int i = 0; i < 16; i++) {
                const int k = rowBase + mi * 32 + 8 * (i / 4) + (i % 4);
                if (k < p.K) {
                    float *d = yn + (size_t)k * OHW;
                    float v = sum(d, acc[mi][ni][i]);
                    if (bias) v += bias[k];
                    if (relu) v = __builtin_elementwise_maximum(v, 0.f);      // keeps a NaN
                    *d = v;
                }
            }
    }
}

// PW: pointwise layers (1x1, stride 1, no padding: the column matrix IS the input, row c of it
// is channel c of x, contiguous over the pixels) whose pixels-per-image count is a multiple of 4
// and whose channel count is a multiple of BK copy the B tile as 16-byte vectors, unconditionally:
// a pixel group past the end re-reads the last group (its columns are never stored).
template <class TL, int MODE, bool REPLACE = false>
__device__ __forceinline__ void ig_tile(const IgemmParams &p, const int kb, const int pb, float (*As)[TL::BK_ * TL::BM_],
                                        float (*Bs)[TL::BK_ * TL::BN_]) {
    constexpr bool PW = MODE == IG_POINTWISE, TAP = MODE == IG_TAP_MASKED || MODE == IG_TAP_INSIDE;
    constexpr bool BUF = MODE == IG_BUF_MASKED || TAP;
    constexpr int BM = TL::BM_, BN = TL::BN_, BK = TL::BK_;
    constexpr int MI = TL::MI, NI = TL::NI, A_LD = TL::A_LD, B_LD = TL::B_LD;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int wm0 = (wave / TL::WGN_) * TL::WM, wn0 = (wave % TL::WGN_) * TL::WN;
    // filter tile: straight 16-byte copies
    const int arow = tid / (BM / 4), acol = (tid % (BM / 4)) * 4;
    const float *ag = p.Wp + (size_t)kb * BM;                     // uniform; the lane adds aOff bytes
    const uint32_t aOff = 4u * ((uint32_t)arow * (uint32_t)p.K_pad + acol);
    const size_t aStage = (size_t)BK * p.K_pad, aPass = (size_t)TL::A_ROWS * p.K_pad;
    const int aLds = arow * BM + acol;

    // the pixel column this thread gathers; its wavefront shares the row
    const int gcol = tid % BN;
    const int grow0 = __builtin_amdgcn_readfirstlane(tid / BN);
    const long pix = (long)pb * BN + gcol;
    const float *ximg = p.x;
    int pixOff = 0;
    uint32_t maskR = 0, maskS = 0;
    if (pix < p.Npix) {
        const uint32_t n = fc_div((uint32_t)pix, p.divOHW);
        const uint32_t pp = (uint32_t)pix - n * (uint32_t)(p.OH * p.OW);
        const uint32_t oh = fc_div(pp, p.divOW), ow = pp - oh * p.OW;
        const int ih0 = (int)oh * p.sh - p.pt, iw0 = (int)ow * p.sw - p.pl;
        ximg = p.x + (size_t)n * p.C * p.H * p.W;
        pixOff = ih0 * p.W + iw0;
        // bit r of maskR: row ih0 + r is inside the image (likewise maskS for columns)
        for (int r = 0; r < p.kh; r++) maskR |= ((unsigned)(ih0 + r) < (unsigned)p.H) ? (1u << r) : 0u;
        for (int q = 0; q < p.kw; q++) maskS |= ((unsigned)(iw0 + q) < (unsigned)p.W) ? (1u << q) : 0u;
    }
    // buffer modes: byte offset of the window origin in the whole tensor, and the taps outside the image
    uint32_t pixByte = 0, invLo = ~0u, invHi = ~0u;
    __amdgpu_buffer_rsrc_t xres = __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(p.x), 0, BUF ? (int)p.xBytes : 0, 0x00020000);
    if (BUF && pix < p.Npix) {
        pixByte = 4u * (uint32_t)((long)(ximg - p.x) + pixOff);
        if (MODE == IG_BUF_MASKED || MODE == IG_TAP_MASKED) {
            const uint32_t rowBits = ~maskS & ((1u << p.kw) - 1u);      // taps of one window row outside the image
            uint64_t inv = 0;
            for (int r = 0; r < p.kh; r++) {
                const uint32_t bits = ((maskR >> r) & 1u) ? rowBits : ((1u << p.kw) - 1u);
                if (r * p.kw < 64) inv |= (uint64_t)bits << (r * p.kw);
            }
            if (p.kh * p.kw < 64) inv |= ~0ull << (p.kh * p.kw);
            invLo = (uint32_t)inv;
            invHi = (uint32_t)(inv >> 32);
        }
    }
    const int bLds = grow0 * BN + gcol;

    // pointwise: this thread's 4-pixel column group and first row of each copy pass
    constexpr int BV_LD = BK * BN / 4 / TL::THREADS, BV_ROWS = TL::THREADS * 4 / BN;
    static_assert((BK * BN / 4) % TL::THREADS == 0, "every thread copies the same number of float4");
    using SeqBV = std::make_integer_sequence<int, BV_LD>;
    const int vrow = tid / (BN / 4), vcol = (tid % (BN / 4)) * 4;
    const int HW = p.H * p.W;
    const float *vg = p.x;      // uniform; the lane adds vOff bytes (the pointwise path is taken for inputs below 4 GiB)
    uint32_t vOff = 0;
    if (PW) {
        const long pix4 = min((long)pb * BN + vcol, p.Npix - 4);
        const uint32_t n = fc_div((uint32_t)pix4, p.divOHW);
        vOff = 4u * ((n * (uint32_t)p.C + vrow) * (uint32_t)HW + ((uint32_t)pix4 - n * (uint32_t)HW));
    }
    const size_t vPass = (size_t)BV_ROWS * HW, vStage = (size_t)BK * HW;
    const int vLds = vrow * BN + vcol;
    floatx4 rv[BV_LD];

    using SeqA = std::make_integer_sequence<int, A_LD>;
    using SeqB = std::make_integer_sequence<int, B_LD>;
    floatx4 ra[A_LD];
    float rb[B_LD];
    uint32_t rbOk = 0;      // bit i: rb[i] lies inside the image
    // this block's share of the reduction
    const int nStagesAll = p.Kred_pad / BK;
    const int sBegin = blockIdx.y * p.stagesPerSplit, sEnd = min(sBegin + p.stagesPerSplit, nStagesAll);
    // Tap-major gather: the BK rows of a stage are channels tapC .. tapC+BK-1 of one tap (tapR, tapS).
    // Stages are gathered in order, so the tap and the channel are running counters, wave-uniform
    // (scalar registers); only the last addition of an element's offset is per lane.
    const uint32_t chanStep = 4u * (uint32_t)(p.H * p.W);
    int tapT = 0, tapR = 0, tapS = 0, tapC = 0;
    if (TAP) {
        const int stagesPerTap = p.C / BK;          // tap-major layers only: C % BK == 0
        tapT = sBegin / stagesPerTap;
        tapC = (sBegin - tapT * stagesPerTap) * BK;
        tapR = tapT / p.kw;
        tapS = tapT - tapR * p.kw;
    }
    auto tap_gather = [&]() __attribute__((always_inline)) {
        const uint32_t voff = pixByte + 4u * (uint32_t)(tapR * p.W + tapS);
        // the poison bit goes on last: the window origin of a border pixel is a negative (wrapped) offset,
        // and adding a channel to an already poisoned offset could carry out of bit 31 again
        uint32_t poison = 0;
        if (MODE == IG_TAP_MASKED) {
            const uint32_t word = tapT < 32 ? invLo : invHi;
            poison = ((word >> (tapT & 31)) & 1u) << 31;
        }
        const uint32_t chan0 = (uint32_t)(tapC + grow0) * chanStep;
#pragma unroll
        for (int i = 0; i < B_LD; i++)
            rb[i] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(
                        xres, (voff + (chan0 + (uint32_t)(i * TL::ROW_STEP) * chanStep)) | poison, 0, 0));
        tapC += BK;
        if (tapC == p.C) {
            tapC = 0;
            tapT++;
            if (++tapS == p.kw) { tapS = 0; tapR++; }
        }
    };
    ag += (size_t)sBegin * aStage;
    ig_load_rows_at(ra, ag, aOff, aPass, SeqA());
    if (PW) {
        vg += (size_t)sBegin * vStage;
        ig_load_rows_at(rv, vg, vOff, vPass, SeqBV());
    } else if (TAP) {
        tap_gather();
    } else if (BUF) {
        ig_gather_rows_buf<true>(rb, xres, pixByte, invLo, invHi, p.table, sBegin * BK + grow0, TL::ROW_STEP, p.kw, SeqB());
    } else {
        rbOk = ig_gather_rows<true>(rb, ximg, pixOff, maskR, maskS, p.table, sBegin * BK + grow0, TL::ROW_STEP, SeqB());
    }

    floatx16 acc[MI][NI];
#pragma unroll
    for (int mi = 0; mi < MI; mi++)
#pragma unroll
        for (int ni = 0; ni < NI; ni++)
#pragma unroll
            for (int i = 0; i < 16; i++) acc[mi][ni][i] = 0.f;

    ig_store_rows(&As[0][aLds], ra, TL::A_ROWS * BM, SeqA());
    if (PW) ig_store_rows(&Bs[0][vLds], rv, BV_ROWS * BN, SeqBV());
    else ig_scatter_rows<!BUF>(&Bs[0][bLds], rb, rbOk, TL::ROW_STEP * BN, SeqB());
    // stage s of the reduction into the staging registers (stages are requested in order: the operands' bases are
    // running pointers in scalar registers, one stage further per call)
    const float *agNext = uniform_ptr(ag + aStage), *vgNext = uniform_ptr(vg + vStage);
    auto load_stage = [&](const int s) __attribute__((always_inline)) {
        ig_load_rows_at(ra, agNext, aOff, aPass, SeqA());
        agNext = uniform_ptr(agNext + aStage);
        if (PW) {
            ig_load_rows_at(rv, vgNext, vOff, vPass, SeqBV());
            vgNext = uniform_ptr(vgNext + vStage);
        }
        else if (TAP) tap_gather();
        else if (BUF) ig_gather_rows_buf<true>(rb, xres, pixByte, invLo, invHi, p.table, s * BK + grow0, TL::ROW_STEP, p.kw, SeqB());
        else rbOk = ig_gather_rows<true>(rb, ximg, pixOff, maskR, maskS, p.table, s * BK + grow0, TL::ROW_STEP, SeqB());
    };
    if (sBegin + 1 < sEnd) load_stage(sBegin + 1);
    __syncthreads();

    const int lrow = lane >> 5, lcol = lane & 31;
    const int aFrag = lrow * BM + wm0 + lcol, bFrag = lrow * BN + wn0 + lcol;
    for (int s = sBegin; s < sEnd; s++) {
        const int buf = (s - sBegin) & 1;
        const float *as = As[buf], *bs = Bs[buf];
        const bool more = s + 1 < sEnd;
        // fragments two reduction steps (kk, kk+2) at a time, a pair ahead of their MFMAs: one ds_read2st64 per
        // 32-wide block and pair, both offsets immediates off an opaque base register (see wino_gemm.hip)
        typedef const __attribute__((address_space(3))) float *LdsPtr;
        LdsPtr asb[MI], bsb[NI];
#pragma unroll
        for (int mi = 0; mi < MI; mi++) {
            asb[mi] = (LdsPtr)(as + aFrag + mi * 32);
            asm volatile("" : "+v"(asb[mi]));
        }
#pragma unroll
        for (int ni = 0; ni < NI; ni++) {
            bsb[ni] = (LdsPtr)(bs + bFrag + ni * 32);
            asm volatile("" : "+v"(bsb[ni]));
        }
        float a[2][2][MI], bb[2][2][NI];
#pragma unroll
        for (int mi = 0; mi < MI; mi++) {
            a[0][0][mi] = asb[mi][0];
            a[0][1][mi] = asb[mi][2 * BM];
        }
#pragma unroll
        for (int ni = 0; ni < NI; ni++) {
            bb[0][0][ni] = bsb[ni][0];
            bb[0][1][ni] = bsb[ni][2 * BN];
        }
#pragma unroll
        for (int kq = 0; kq < BK / 4; kq++) {
            const int cur = kq & 1, nxt = cur ^ 1;
            if (kq + 1 < BK / 4) {
#pragma unroll
                for (int mi = 0; mi < MI; mi++) {
                    a[nxt][0][mi] = asb[mi][(4 * kq + 4) * BM];
                    a[nxt][1][mi] = asb[mi][(4 * kq + 6) * BM];
                }
#pragma unroll
                for (int ni = 0; ni < NI; ni++) {
                    bb[nxt][0][ni] = bsb[ni][(4 * kq + 4) * BN];
                    bb[nxt][1][ni] = bsb[ni][(4 * kq + 6) * BN];
                }
            }
            // the reads of the next pair are issued before the MFMAs of this one
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int st = 0; st < 2; st++)
#pragma unroll
                for (int mi = 0; mi < MI; mi++)
#pragma unroll
                    for (int ni = 0; ni < NI; ni++)
                        acc[mi][ni] = __builtin_amdgcn_mfma_f32_32x32x2f32(a[cur][st][mi], bb[cur][st][ni], acc[mi][ni], 0, 0, 0);
            if (4 * kq == BK / 2 && more) {
                // the next stage goes to the other LDS buffer half way through this one's MFMAs,
                // and the one after it is requested at once: a whole stage in flight
                ig_store_rows(&As[buf ^ 1][aLds], ra, TL::A_ROWS * BM, SeqA());
                if (PW) ig_store_rows(&Bs[buf ^ 1][vLds], rv, BV_ROWS * BN, SeqBV());
                else ig_scatter_rows<!BUF>(&Bs[buf ^ 1][bLds], rb, rbOk, TL::ROW_STEP * BN, SeqB());
                if (s + 2 < sEnd) load_stage(s + 2);
            }
        }
        __syncthreads();
    }

    ig_store_tile<TL, REPLACE>(acc, p, p.bias, p.relu, kb, pb, wm0, wn0, lrow, lcol);
}

template <class TL, int MODE>
__global__ __launch_bounds__(TL::THREADS, TL::MIN_WAVES) void igemm_conv_kernel(const IgemmParams p) {
    __shared__ __attribute__((aligned(16))) float As[2][TL::BK_ * TL::BM_];
    __shared__ __attribute__((aligned(16))) float Bs[2][TL::BK_ * TL::BN_];
    int kb, pb;
    if (ig_decode_tile(p, &kb, &pb)) ig_tile<TL, MODE>(p, kb, pb, As, Bs);
}

// The same layer on the bf16 matrix cores at fp32 accuracy (see split_mfma.h), for inputs below 2 GiB.
//
// A wavefront owns all rows of 32 pixel columns, so that a column is gathered and split by the
// wavefront that multiplies it and goes from memory to the matrix core without leaving its registers: a lane holds 8
// consecutive reduction rows of one pixel, which is its share of a 32x32x16 product.  The filter has been split when it was
// packed and goes to LDS by direct loads, one stage ahead, for all wavefronts of the workgroup.
// Four bytes a lane, a load costs the CU's address unit 18 to 21 cycles.  A stage of a 128x128 tile takes 32 loads of columns
// and 12 of the filter, some 880 cycles, beside 768 of products; both operands through registers took 64 loads.  Counted on
// 128 -> 128 3x3/2 at 56x56, batch 32: the address units are busy 81 % of the cycles and the matrix pipes 33 % with 64x64
// tiles, 62 % and 39 % with 128x64, where a wavefront waits a third of its life for data or at a barrier.  Window rows in
// runs are 16 bytes a lane, 8 loads a stage: on the 7x7/2 stem vector instructions take 59 % of the SIMD's cycles and the
// matrix pipes 47 %, the address units 60 %.
// Measured as calls in turn on one box, batch 32, fp32 instructions -> both operands split in the kernel -> this: 256 -> 256 3x3/2
// at 28x28 94 -> 80 -> 70 us, 7x7/2 stem 106 -> 87 -> 62 (72 amid the layers of ResNet-50), 64 -> 64 3x3 at 56x56 83 -> 66 -> 52,
// 256 -> 256 1x1 at 56x56 123 -> 93 -> 79, 512 -> 2048 1x1 at 7x7 42 -> 34 -> 29; 32 -> 16 3x3 at 97x97, batch 55, (32 rows a
// tile) 124 -> 122 -> 73.  Prefetch of the operands across a whole stage with three LDS buffers in place of two: -3 to +8 %, two
// wavefronts a SIMD in place of four.
template <int BM, int BN, int WAVES>
struct IgSplit {
    static constexpr int BM_ = BM, BN_ = BN, THREADS = 64 * WAVES;
    static constexpr int WN = BN / WAVES, MI = BM / 32, NI = WN / 32;
    static constexpr int STAGE_WORDS = kSplitBlockWords * (BM / 32);      // of the filter
    // the tile that forms values again that are not finite: same threads
    typedef IgTile<64, 64, 16, 2, THREADS / 128> Again;
    static constexpr int LDS_WORDS = 2 * STAGE_WORDS > Again::LDS_BYTES / 16 ? 2 * STAGE_WORDS : Again::LDS_BYTES / 16;
    // wavefronts per SIMD the two sums leave registers for
    static constexpr int MIN_WAVES = MI * NI > 2 ? 2 : 4;
    static_assert(Again::THREADS == THREADS && BM % Again::BM_ == 0 && BN % Again::BN_ == 0, "same workgroup");
};
// Tile shape of a public configuration on the bf16 matrix cores (void: none).
template <class TL> struct IgSplitOf { typedef void type; };

// How the reduction rows of a stage lie in the input (orders of the reduction: ig_order).
//   SP_INSIDE      16 channels of one window tap, no tap outside the image
//   SP_MASKED      the same with taps outside the image
//   SP_PAD         the same with channels past the last one
//   SP_ROW8        two runs of 8 columns of a window row of one channel: 16-byte loads
//   SP_ROW4        four runs of 4 columns
//   SP_POINT       pointwise layers under tiles of 64 rows: 16 channels, read four pixels a lane and turned through LDS
//   SP_POINT32     the same with the packed filter in fp32, split on its way to LDS
//   SP_TRI         as SP_PAD, for windows of 3 columns and at most one column of left padding: the three stages of a window row and
//                  16 channels from one 12-byte load a channel
enum { SP_INSIDE, SP_MASKED, SP_PAD, SP_ROW8, SP_ROW4, SP_POINT, SP_POINT32, SP_TRI };

template <int MI_, class S>
struct IgSplitPart {
    static constexpr int BM_ = S::BM_, BN_ = S::BN_, MI = MI_, NI = S::NI;
};

// One workgroup tile, of which the first MI blocks of 32 rows of each wavefront hold output channels.
// LEVELS (tiles of 128 rows): every p.sumStages stages the sum of the hi * hi products is added to a second one, and begun again.  A
// product of 16 rows is rounded at the size of the sum it is added to, so that the error of one sum grows with its length; this way a reduction
// in fewer parts has no larger one (ig_expected_parts).  Three of the second sum's four blocks of rows fit the registers two wavefronts a
// SIMD leave, the last one lies in LDS (both in LDS: three 128x64 workgroups a CU in place of four, 256 -> 256 3x3/2 at 28x28 batch 32
// 72 us / 57).  Columns of window rows of three taps (SP_TRI) leave no registers for it: 57 us would be 55.
template <class S, int MODE, int MI, bool LEVELS>
__device__ __forceinline__ void ig_split_tile(const IgemmParams &p, const int kb, const int pb, fc_uintx4 *smem) {
    constexpr bool ROW = MODE == SP_ROW8 || MODE == SP_ROW4, POINT = MODE == SP_POINT || MODE == SP_POINT32;
    constexpr int NI = S::NI, WAVES = S::THREADS / 64;
    constexpr uint32_t OUTSIDE = 0x80000000u;      // past the end of x whatever scalar offset is added: reads 0
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wn0 = wave * S::WN;
    const int lrow = lane >> 5, lcol = lane & 31;
    const int nStagesAll = p.Kred_pad / 16;
    const int sBegin = blockIdx.y * p.stagesPerSplit, sEnd = min(sBegin + p.stagesPerSplit, nStagesAll);

    // pixels of this lane: byte offset of the window in the tensor, window rows and columns outside the image
    uint32_t pixByte[NI], rowBad[NI], colBad[NI];
#pragma unroll
    for (int ni = 0; ni < NI; ni++) {
        const long pix = (long)pb * S::BN_ + wn0 + ni * 32 + lcol;
        pixByte[ni] = OUTSIDE;
        rowBad[ni] = colBad[ni] = ~0u;
        if (POINT) {      // pixels 4 * (lane % 8) .. + 3, channels lane / 8 and 8 on
            const long first = (long)pb * S::BN_ + wn0 + ni * 32 + 4 * (lane & 7);
            if (first < p.Npix) {
                const uint32_t n = fc_div((uint32_t)first, p.divOHW), image = (uint32_t)(p.H * p.W);
                pixByte[ni] = 4u * ((n * (uint32_t)p.C + (uint32_t)(lane >> 3)) * image + ((uint32_t)first - n * image));
            }
        } else if (pix < p.Npix) {
            const uint32_t n = fc_div((uint32_t)pix, p.divOHW);
            const uint32_t pp = (uint32_t)pix - n * (uint32_t)(p.OH * p.OW);
            const uint32_t oh = fc_div(pp, p.divOW), ow = pp - oh * p.OW;
            const int ih0 = (int)oh * p.sh - p.pt, iw0 = (int)ow * p.sw - p.pl;
            pixByte[ni] = 4u * (n * (uint32_t)(p.C * p.H * p.W) + (uint32_t)(ih0 * p.W + iw0));
            if (MODE == SP_TRI && iw0 < 0) pixByte[ni] += 4u;      // from its first column inside the image
            if (!ROW) pixByte[ni] += 8u * lrow * 4u * (uint32_t)(p.H * p.W);      // the lane's first channel of a stage
            if (MODE != SP_INSIDE) {
                for (int r = 0; r < p.kh; r++) rowBad[ni] &= (unsigned)(ih0 + r) < (unsigned)p.H ? ~(1u << r) : ~0u;
                for (int q = 0; q < p.kw; q++) colBad[ni] &= (unsigned)(iw0 + q) < (unsigned)p.W ? ~(1u << q) : ~0u;
            }
        }
    }
    const __amdgpu_buffer_rsrc_t xres = __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(p.x), 0, (int)p.xBytes, 0x00020000);
    auto load1 = [&](const uint32_t voff, const uint32_t soff) __attribute__((always_inline)) {
        return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(xres, voff, soff, 0));
    };

    typedef float floatx3 __attribute__((ext_vector_type(3)));
    float raw[NI][8];
    floatx3 raw3[NI][8];      // SP_TRI: a window row of each channel
    // -- blocks of channels: the tap and the first channel of the stage, counted in scalar registers
    const uint32_t chanStep = 4u * (uint32_t)(p.H * p.W);
    int tapR = 0, tapS = 0, tapC = 0;
    uint32_t voff[NI];
    auto tap = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int ni = 0; ni < NI; ni++) {
            voff[ni] = pixByte[ni] + 4u * (uint32_t)(tapR * p.W + tapS);
            if (MODE != SP_INSIDE) voff[ni] = ((rowBad[ni] >> tapR) | (colBad[ni] >> tapS)) & 1u ? OUTSIDE : voff[ni];
        }
    };
    // -- row orders: table entries of the runs of the stage to fetch, fetched themselves a stage before
    constexpr int RUNS = MODE == SP_ROW8 ? 2 : 4, RUN = 16 / RUNS;
    int runOff[RUNS], runTap[RUNS];
    uint32_t cols[NI][2], rowVoff[NI][2];      // of the stage in `raw`: columns of the runs inside the image, offsets
    auto table = [&](const int s) __attribute__((always_inline)) {
#pragma unroll
        for (int u = 0; u < RUNS; u++) {
            runOff[u] = p.table[2 * (16 * s + RUN * u)];
            runTap[u] = p.table[2 * (16 * s + RUN * u) + 1];
        }
    };
    if (ROW) {
        table(sBegin);
    } else {
        const int block = sBegin / (p.kh * p.kw), t = sBegin - block * (p.kh * p.kw);
        tapC = block * 16;
        tapR = t / p.kw;
        tapS = t - tapR * p.kw;
        if (MODE != SP_TRI) tap();
    }
    // fetches stage s; stages are fetched in order
    auto fetch = [&](const int s) __attribute__((always_inline)) {
        if (ROW) {
#pragma unroll
            for (int v = 0; v < RUNS / 2; v++) {
                const int off = lrow ? runOff[RUNS / 2 + v] : runOff[v], rs = lrow ? runTap[RUNS / 2 + v] : runTap[v];
#pragma unroll
                for (int ni = 0; ni < NI; ni++) {
                    const uint32_t vo = (rowBad[ni] >> (rs >> 16)) & 1u ? OUTSIDE : pixByte[ni] + 4u * (uint32_t)off;
                    cols[ni][v] = ~colBad[ni] >> (rs & 0xffff);
                    rowVoff[ni][v] = vo;
#pragma unroll
                    for (int h = 0; h < RUN / 4; h++) {
                        const floatx4 d = __builtin_bit_cast(floatx4, __builtin_amdgcn_raw_buffer_load_b128(xres, vo, 16 * h, 0));
#pragma unroll
                        for (int j = 0; j < 4; j++) raw[ni][v * RUN + 4 * h + j] = d[j];
                    }
                }
            }
            table(min(s + 1, nStagesAll - 1));
            return;
        }
        if constexpr (MODE == SP_TRI) {      // the window row that stage s begins or, at the first stage, lies in
            const int left = p.C - tapC - 8 * lrow;      // channels of the lane's 8 that exist
#pragma unroll
            for (int ni = 0; ni < NI; ni++) {
                const uint32_t vo = (rowBad[ni] >> tapR) & 1u ? OUTSIDE : pixByte[ni] + 4u * (uint32_t)(tapR * p.W);
#pragma unroll
                for (int i = 0; i < 8; i++)
                    raw3[ni][i] = __builtin_bit_cast(floatx3, __builtin_amdgcn_raw_buffer_load_b96(
                                                                  xres, i < left ? vo : OUTSIDE, (uint32_t)min(tapC + i, p.C - 1) * chanStep, 0));
            }
            tapR++;
            const bool all = tapR == p.kh;
            tapR = all ? 0 : tapR;
            tapC += all ? 16 : 0;
            return;
        }
        if (POINT) {
            const int left = p.C - 16 * s - (lane >> 3);      // channels from the lane's first on that exist
#pragma unroll
            for (int ni = 0; ni < NI; ni++)
#pragma unroll
                for (int h = 0; h < 2; h++) {
                    const floatx4 d = __builtin_bit_cast(floatx4, __builtin_amdgcn_raw_buffer_load_b128(
                                                                      xres, 8 * h < left ? pixByte[ni] : OUTSIDE, (uint32_t)min(16 * s + 8 * h, p.C - 1) * chanStep, 0));
#pragma unroll
                    for (int j = 0; j < 4; j++) raw[ni][4 * h + j] = d[j];
                }
            return;
        }
        const int left = p.C - tapC - 8 * lrow;      // channels of the lane's 8 that exist
#pragma unroll
        for (int i = 0; i < 8; i++) {
            const int c = MODE == SP_PAD ? min(tapC + i, p.C - 1) : tapC + i;
#pragma unroll
            for (int ni = 0; ni < NI; ni++)
                raw[ni][i] = load1(MODE == SP_PAD && i >= left ? OUTSIDE : voff[ni], (uint32_t)c * chanStep);
        }
        tapS++;
        const bool row = tapS == p.kw;
        tapS = row ? 0 : tapS;
        tapR += row ? 1 : 0;
        const bool all = tapR == p.kh;
        tapR = all ? 0 : tapR;
        tapC += all ? 16 : 0;
        tap();
    };
    // the stage in `raw` as operand words of the three parts
    fc_uintx4 b[NI][3];
    // readAgain: runs that start before x are read again, element by element (whether a 16-byte load there gives the elements
    // inside x is left open)
    auto split = [&](auto readAgain) __attribute__((always_inline)) {
        if constexpr (POINT) {
            // four pixels of one channel -> eight channels of one pixel, through this wavefront's own [16 channels][32 pixels]
            float *const turn = reinterpret_cast<float *>(smem + S::LDS_WORDS) + wave * 512;
#pragma unroll
            for (int ni = 0; ni < NI; ni++) {
#pragma unroll
                for (int h = 0; h < 2; h++)
                    *reinterpret_cast<floatx4 *>(turn + 256 * h + 4 * lane) = floatx4{raw[ni][4 * h], raw[ni][4 * h + 1], raw[ni][4 * h + 2], raw[ni][4 * h + 3]};
                fc_wave_sync();      // lanes read what other lanes wrote
#pragma unroll
                for (int i = 0; i < 8; i++) raw[ni][i] = turn[(8 * lrow + i) * 32 + lcol];
                fc_wave_sync();      // before the next block or stage is written
            }
        }
        if (ROW) {
            if constexpr (decltype(readAgain)::value) {
#pragma unroll
                for (int ni = 0; ni < NI; ni++)
#pragma unroll
                    for (int i = 0; i < 8; i++) {
                        const uint32_t vo = rowVoff[ni][i / RUN], at = vo + 4u * (uint32_t)(i % RUN);
                        const float d = load1((int)at < 0 ? OUTSIDE : at, 0);      // (an immediate offset would not wrap)
                        raw[ni][i] = vo != OUTSIDE && (int)vo < 0 ? d : raw[ni][i];
                    }
            }
#pragma unroll
            for (int ni = 0; ni < NI; ni++)
#pragma unroll
                for (int i = 0; i < 8; i++) {
                    const int keep = (int)(cols[ni][i / RUN] << (31 - i % RUN)) >> 31;
                    raw[ni][i] = __builtin_bit_cast(float, __builtin_bit_cast(int, raw[ni][i]) & keep);
                }
        }
#pragma unroll
        for (int ni = 0; ni < NI; ni++) fc_split8(raw[ni], b[ni], 1);
    };
    // filter words of the next stage to LDS: whole wavefronts, 16 bytes a lane
    constexpr int PIECES = MI * kSplitBlockWords / 64;
    const fc_uintx4 *fbase = p.Ws + ((size_t)sBegin * (p.K_pad / 32) + (size_t)kb * (S::BM_ / 32)) * kSplitBlockWords;
    const size_t fstep = (size_t)(p.K_pad / 32) * kSplitBlockWords;
    auto filter = [&](const int buf) __attribute__((always_inline)) {
        const fc_uintx4 *src = uniform_ptr(fbase);
#pragma unroll
        for (int i = 0; i < (PIECES + WAVES - 1) / WAVES; i++) {
            const int piece = wave + i * WAVES;
            if (PIECES % WAVES == 0 || piece < PIECES)
                __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void *)(src + piece * 64 + lane),
                                                 (__attribute__((address_space(3))) void *)(smem + buf * S::STAGE_WORDS + piece * 64), 16, 0, 0);
        }
        fbase = uniform_ptr(fbase + fstep);
    };

    // SP_POINT32: four rows of one channel to registers, and as halves of operand words to LDS a stage later
    float rows[4];
    auto filterRows = [&](const int s) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < 4; i++) rows[i] = p.Wp[(size_t)(16 * s + 4 * wave + i) * p.K_pad + lane];
    };
    auto filterSplit = [&](const int buf) __attribute__((always_inline)) {
        typedef uint32_t uintx2 __attribute__((ext_vector_type(2)));
        uintx2 part[3];
#pragma unroll
        for (int i = 0; i < 2; i++) {
            uint32_t h, m, l;
            fc_split2(rows[2 * i], rows[2 * i + 1], h, m, l);
            part[0][i] = h; part[1][i] = m; part[2][i] = l;
        }
        uintx2 *const to = reinterpret_cast<uintx2 *>(smem + buf * S::STAGE_WORDS + lrow * kSplitBlockWords + (wave >> 1) * 32 + lcol) + (wave & 1);
#pragma unroll
        for (int i = 0; i < 3; i++) to[2 * i * 64] = part[i];
    };

    floatx16 acc[MI][NI], small[MI][NI];
    fc_zero<MI, NI>(acc);
    fc_zero<MI, NI>(small);
    // more: a stage follows; column: of its window row, where three stages share their loads
    auto stage = [&](const int s, const bool more, auto readAgain, auto column) __attribute__((always_inline)) {
        const int buf = (s - sBegin) & 1;
        if constexpr (MODE == SP_TRI) {
            constexpr int q = decltype(column)::value;
#pragma unroll
            for (int ni = 0; ni < NI; ni++) {
                const int keep = (int)(~colBad[ni] << (31 - q)) >> 31;
                const bool shifted = colBad[ni] & 1u;
#pragma unroll
                for (int i = 0; i < 8; i++) {
                    const float v = q == 0 || shifted ? raw3[ni][i][q == 2 ? 1 : 0] : raw3[ni][i][q];
                    raw[ni][i] = __builtin_bit_cast(float, __builtin_bit_cast(int, v) & keep);
                }
            }
        }
        split(readAgain);
        if constexpr (MODE == SP_POINT32) filterSplit(buf);
        if constexpr (MODE != SP_POINT32) __builtin_amdgcn_s_waitcnt(0x0f70);      // vmcnt(0): this wavefront's filter words of the stage are in LDS
        __syncthreads();                         // and those of the others, which have read the stage before
        const fc_uintx4 *as = smem + buf * S::STAGE_WORDS + lane;
        fc_bf16x8 a[3][MI];
#pragma unroll
        for (int q = 2; q >= 0; q--)
#pragma unroll
            for (int mi = 0; mi < MI; mi++) a[q][mi] = __builtin_bit_cast(fc_bf16x8, as[mi * kSplitBlockWords + q * 64]);
        if (more) {      // (behind the reads: the compiler has reads of LDS wait for direct loads before them)
            if constexpr (MODE == SP_POINT32) filterRows(s + 1);
            else filter(buf ^ 1);
            if (MODE != SP_TRI || decltype(column)::value == 2) fetch(s + 1);
        }
        constexpr int pa[5] = {2, 1, 0, 1, 0}, pb[5] = {0, 1, 2, 0, 1};
#pragma unroll
        for (int q = 0; q < 5; q++)
#pragma unroll
            for (int mi = 0; mi < MI; mi++)
#pragma unroll
                for (int ni = 0; ni < NI; ni++)
                    small[mi][ni] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[pa[q]][mi], __builtin_bit_cast(fc_bf16x8, b[ni][pb[q]]), small[mi][ni], 0, 0, 0);
#pragma unroll
        for (int mi = 0; mi < MI; mi++)
#pragma unroll
            for (int ni = 0; ni < NI; ni++)
                acc[mi][ni] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[0][mi], __builtin_bit_cast(fc_bf16x8, b[ni][0]), acc[mi][ni], 0, 0, 0);
    };
    constexpr int HELD = 3;      // blocks of the second sum in registers
    static_assert(!LEVELS || (MI == HELD + 1 && NI == 1), "one block in LDS, four words a lane");
    floatx16 second[HELD];
    floatx4 *const secondLds = reinterpret_cast<floatx4 *>(smem + S::LDS_WORDS) + wave * 256 + lane;
    if constexpr (LEVELS) {
#pragma unroll
        for (int mi = 0; mi < HELD; mi++)
#pragma unroll
            for (int i = 0; i < 16; i++) second[mi][i] = 0.f;
#pragma unroll
        for (int q = 0; q < 4; q++) secondLds[64 * q] = floatx4{0.f, 0.f, 0.f, 0.f};
    }
    // the first sum to the second; at the end the whole to the first
    auto carry = [&](const bool end) __attribute__((always_inline)) {
        if constexpr (LEVELS) {
#pragma unroll
            for (int mi = 0; mi < HELD; mi++)
#pragma unroll
                for (int i = 0; i < 16; i++) {
                    second[mi][i] += acc[mi][0][i];
                    acc[mi][0][i] = end ? second[mi][i] : 0.f;
                }
#pragma unroll
            for (int q = 0; q < 4; q++) {
                floatx4 d = secondLds[64 * q];
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    d[i] += acc[HELD][0][4 * q + i];
                    acc[HELD][0][4 * q + i] = end ? d[i] : 0.f;
                }
                if (!end) secondLds[64 * q] = d;
            }
        }
    };
    if constexpr (MODE == SP_POINT32) filterRows(sBegin);
    else filter(0);
    fetch(sBegin);
    int s = sBegin;
    if constexpr (ROW) {
        // one number for the workgroup: all its wavefronts meet at the same barriers
        const int stagesBefore = (long)pb * S::BN_ < p.pixBefore ? p.stagesBefore : 0;
#pragma unroll 1
        for (; s < sEnd && s < stagesBefore; s++) stage(s, s + 1 < sEnd, std::true_type(), std::integral_constant<int, 0>());
#pragma unroll 1
        for (; s < sEnd; s++) stage(s, s + 1 < sEnd, std::false_type(), std::integral_constant<int, 0>());
    } else if constexpr (MODE == SP_TRI) {
        // three stages a round; a part of a split reduction may begin and end within a window row
        const int skip = tapS;
#pragma unroll 1
        for (s -= skip; s < sEnd; s += 3) {
            if (s >= sBegin) stage(s, s + 1 < sEnd, std::false_type(), std::integral_constant<int, 0>());
            if (s + 1 >= sBegin && s + 1 < sEnd) stage(s + 1, s + 2 < sEnd, std::false_type(), std::integral_constant<int, 1>());
            if (s + 2 < sEnd) stage(s + 2, s + 3 < sEnd, std::false_type(), std::integral_constant<int, 2>());
        }
    } else {
#pragma unroll 1
        for (int left = p.sumStages; s + 1 < sEnd; s++) {
            stage(s, true, std::false_type(), std::integral_constant<int, 0>());
            if constexpr (LEVELS)
                if (--left == 0) {
                    carry(false);
                    left = p.sumStages;
                }
        }
        stage(s, false, std::false_type(), std::integral_constant<int, 0>());
    }
    if constexpr (LEVELS) carry(true);
    fc_join<MI, NI>(acc, small);
    const bool again = __syncthreads_or(fc_not_finite<MI, NI>(acc));
    ig_store_tile<IgSplitPart<MI, S>>(acc, p, again ? nullptr : p.bias, again ? 0 : p.relu, kb, pb, 0, wn0, lrow, lcol);
    if (again) {
        // a smaller tile at a time, which leaves the registers to the loop above; the table knows any order
        typedef typename S::Again Sub;
        float *const f = reinterpret_cast<float *>(smem);
        constexpr int QM = S::BM_ / Sub::BM_, QN = S::BN_ / Sub::BN_;
        __syncthreads();      // the whole tile is in y, or in the partial sums
        for (int q = 0; q < QM * QN; q++)
            ig_tile<Sub, IG_GATHER, true>(p, kb * QM + q / QN, pb * QN + q % QN, reinterpret_cast<float (*)[16 * Sub::BM_]>(f),
                                     reinterpret_cast<float (*)[16 * Sub::BN_]>(f + 2 * 16 * Sub::BM_));
    }
}

template <class S, int MODE, bool LEVELS = false>
__global__ __launch_bounds__(S::THREADS, (MODE == SP_ROW4 || MODE == SP_INSIDE) && S::MIN_WAVES > 3 ? 3 : S::MIN_WAVES) void igemm_split_kernel(const IgemmParams p) {
    __shared__ fc_uintx4 smem[S::LDS_WORDS + (LEVELS ? S::THREADS / 64 * 256 : 0) + (MODE == SP_POINT || MODE == SP_POINT32 ? S::THREADS / 64 * 128 : 0)];
    int kb, pb;
    if (!ig_decode_tile(p, &kb, &pb)) return;
    // 32 rows of a 64-row tile past the last output channel are not multiplied
    if (S::BM_ == 64 && p.K - kb * 64 <= 32) ig_split_tile<S, MODE, 1, false>(p, kb, pb, smem);
    else ig_split_tile<S, MODE, S::MI, LEVELS>(p, kb, pb, smem);
}

// The packed filter as operand words: [stage][block of 32 output channels][part][half of the stage][channel], 16 bytes each,
// after the fp32 filter (which forms values again that are not finite).
__global__ __launch_bounds__(256) void igemm_split_filter_kernel(const float *__restrict__ Wp, fc_uintx4 *__restrict__ Ws, int K_pad, long total) {
    const long id = (long)blockIdx.x * 256 + threadIdx.x;
    if (id >= total) return;
    const int lane = (int)(id & 63), row = lane & 31, half = lane >> 5;
    const long block = id >> 6;      // stage * (K_pad / 32) + block of channels
    const long stage = block / (K_pad / 32), kb = block - stage * (K_pad / 32);
    const float *src = Wp + (size_t)(16 * stage + 8 * half) * K_pad + kb * 32 + row;
    float v[8];
#pragma unroll
    for (int i = 0; i < 8; i++) v[i] = src[(size_t)i * K_pad];
    fc_split8(v, Ws + (size_t)block * kSplitBlockWords + lane, 64);
}

#include "implicit_gemm_short.h"

// Sums the partial results of a split reduction in split order (so the result does
// not depend on which workgroup finished first), adds bias, applies ReLU, writes NCHW.
__global__ __launch_bounds__(256) void igemm_reduce_kernel(const float *__restrict__ ws, const float *__restrict__ bias,
                                                           float *__restrict__ y, int K, long Npix, int OHW,
                                                           int splitK, int relu, fc_fastdiv divOHW) {
    const long pix = (long)blockIdx.x * 256 + threadIdx.x;
    const int k = blockIdx.y;
    if (pix >= Npix) return;
    const size_t slab = (size_t)K * Npix;
    const float *src = ws + (size_t)k * Npix + pix;
    float v = src[0];
    for (int z = 1; z < splitK; z++) v += src[(size_t)z * slab];
    if (bias) v += bias[k];
    if (relu) v = __builtin_elementwise_maximum(v, 0.f);      // keeps a NaN
    const uint32_t n = fc_div((uint32_t)pix, divOHW);
    y[((size_t)n * K + k) * OHW + (pix - (long)n * OHW)] = v;
}

typedef IgTile<128, 128, 16, 2, 2> Ig0;
typedef IgTile<64, 128, 16, 1, 2> Ig1;
typedef IgTile<128, 64, 16, 2, 1> Ig2;
typedef IgTile<64, 64, 16, 2, 2> Ig3;
typedef IgTile<32, 64, 16, 1, 1> Ig4;
typedef IgTile<256, 128, 16, 2, 2> Ig5;
typedef IgTile<128, 256, 16, 2, 2> Ig6;
typedef IgTile<64, 256, 16, 1, 4> Ig7;
template <> struct IgSplitOf<Ig0> { typedef IgSplit<128, 128, 4> type; };
template <> struct IgSplitOf<Ig1> { typedef IgSplit<64, 128, 4> type; };
template <> struct IgSplitOf<Ig2> { typedef IgSplit<128, 64, 2> type; };
template <> struct IgSplitOf<Ig3> { typedef IgSplit<64, 64, 2> type; };
// (a wavefront's registers hold the two sums of 128x32 at most)
template <> struct IgSplitOf<Ig5> { typedef IgSplit<128, 128, 4> type; };
template <> struct IgSplitOf<Ig6> { typedef IgSplit<128, 128, 4> type; };
template <> struct IgSplitOf<Ig7> { typedef IgSplit<64, 128, 4> type; };

const fc_gemm_config kIgConfigs[] = {
#define FC_CFG(id, T) {id, T::BM_, T::BN_, T::BK_, T::WGM_, T::WGN_, T::LDS_BYTES, 1}
    FC_CFG(0, Ig0), FC_CFG(1, Ig1), FC_CFG(2, Ig2), FC_CFG(3, Ig3),
    FC_CFG(4, Ig4), FC_CFG(5, Ig5), FC_CFG(6, Ig6), FC_CFG(7, Ig7),
#undef FC_CFG
};
constexpr int kNumIgConfigs = sizeof(kIgConfigs) / sizeof(kIgConfigs[0]);

// Tiles that run in their place where products are split (0: none).
struct IgTileSize {
    int bm, bn;
};
template <class TL>
constexpr IgTileSize ig_split_tile_size() {
    typedef typename IgSplitOf<TL>::type S;
    if constexpr (std::is_void<S>::value) return {0, 0};
    else return {S::BM_, S::BN_};
}
const IgTileSize kIgSplitTiles[] = {ig_split_tile_size<Ig0>(), ig_split_tile_size<Ig1>(), ig_split_tile_size<Ig2>(), ig_split_tile_size<Ig3>(),
                                    ig_split_tile_size<Ig4>(), ig_split_tile_size<Ig5>(), ig_split_tile_size<Ig6>(), ig_split_tile_size<Ig7>()};
static_assert(sizeof(kIgSplitTiles) / sizeof(kIgSplitTiles[0]) == kNumIgConfigs, "one per configuration");

// The column matrix of a pointwise layer is its input, read 16 bytes a lane where that is possible.
bool ig_point(const fc_conv_shape &s) {
    return s.kh == 1 && s.kw == 1 && s.sh == 1 && s.sw == 1 && s.pt == 0 && s.pb == 0 && s.pl == 0 && s.pr == 0;
}
bool ig_pointwise(const fc_conv_shape &s, int bk, bool x16) {
    return ig_point(s) && (s.H * s.W) % 4 == 0 && s.C % bk == 0 && x16 && 4l * s.N * s.C * s.H * s.W < (1l << 32);
}

// Split products: four consecutive pixels of a pointwise layer lie in one image, so that they are one 16-byte load of a channel
// (any alignment; beyond the last pixel of a single image it reads on into the next channel, or 0, for pixels that are not stored).
bool ig_four_pixels(const fc_conv_shape &s) { return ig_point(s) && ((s.H * s.W) % 4 == 0 || s.N == 1); }

// No tap of any window leaves the image, and the reduction has no padding rows.
bool ig_inside(const fc_conv_shape &s, int bk) {
    const int OH = fc_out_dim(s.H, s.pt, s.pb, s.kh, s.sh), OW = fc_out_dim(s.W, s.pl, s.pr, s.kw, s.sw);
    return s.pt == 0 && s.pl == 0 && (OH - 1) * s.sh + s.kh <= s.H && (OW - 1) * s.sw + s.kw <= s.W && (s.C * s.kh * s.kw) % bk == 0;
}

// Whether a tile of this configuration runs on the bf16 matrix cores with its filter packed in parts (a pointwise layer is a block whose only
// tap is inside): for inputs below 2 GiB, but not for pointwise layers of up to 64 output channels, whose x the fp32 kernel reads 16 bytes a
// lane, nor for reductions of two or three stages; their filter is packed in fp32, and those of many pixels are split from it in the kernel
// (ig_point_few, ig_short).  For the others of them, best tile on fp32 / on a filter in parts, batch 32, us: 1x1 128 -> 32 at 56x56 13.4 / 14.2,
// 512 -> 64 at 28x28 23.4 / 23.4, 64 -> 64 at 56x56 12.4 / 11.5.
bool ig_splits(const fc_conv_shape &s, const fc_gemm_config &c) {
    if (c.waves_k > 1 || c.bm % 64 != 0 || 4l * s.N * s.C * s.H * s.W >= (1l << 31) || (long)s.C * s.kh * s.kw <= 48) return false;
    if (ig_pointwise(s, c.bk, true) && s.K <= 64) return false;
    return s.kh * s.kw <= 64 || (s.C % c.bk == 0 && ig_inside(s, c.bk));
}

// The tile that runs a layer under a configuration.
IgTileSize ig_tile_size(const fc_conv_shape &s, const fc_gemm_config &c) {
    if (c.id < kNumIgConfigs && ig_splits(s, c)) return kIgSplitTiles[c.id];
    return {c.bm, c.bn};
}

// Order of the reduction rows where products are split, and their number (before rounding up to a stage).  A row in runs is
// taken at 0.85 (8 columns) and 0.9 (4) of the time of one in blocks.  80 drawn layers without whole blocks (3x3, 5x5, 7x7),
// every order at its best tile: 0.97 and 0.99 in the median, half-filled runs and blocks spread it from 0.76 to 1.58; the order
// so chosen is 0.5 % behind the best of the three on average and 9 % at most.
int ig_split_order(const fc_conv_shape &s, long *rows) {
    const long taps = (long)s.kh * s.kw;
    *rows = s.C * taps;
    if (s.C % 16 == 0) return IG_ORDER_BLOCK;
    const long block = fc_round_up(s.C, 16) * taps;
    const long row8 = 8l * s.C * s.kh * ((s.kw + 7) / 8), row4 = 4l * s.C * s.kh * ((s.kw + 3) / 4);
    const double costBlock = 1.0 * block, costRow8 = 0.85 * fc_round_up(row8, 16), costRow4 = 0.9 * fc_round_up(row4, 16);
    if (costBlock <= costRow8 && costBlock <= costRow4) { *rows = block; return IG_ORDER_BLOCK; }
    if (costRow8 <= costRow4) { *rows = row8; return IG_ORDER_ROW8; }
    *rows = row4;
    return IG_ORDER_ROW4;
}

// Order of the reduction rows of a configuration and their number.
int ig_order(const fc_conv_shape &s, const fc_gemm_config &c, long *rows) {
    if (ig_splits(s, c)) return ig_split_order(s, rows);
    *rows = (long)s.C * s.kh * s.kw;
    return s.C % c.bk == 0 ? IG_ORDER_TAP : IG_ORDER_CHANNEL;
}

// Whether a layer runs in igemm_short_kernel: up to four stages of rows and at least 25 blocks of 32 channels and 32 pixels a CU
// (below, a tile is as soon done as the filter is split, us: 1x1 26 -> 233 at 99x99, one image, 7.0 / 7.7, 31 -> 128 at 112x112 batch
// 4 10.7 / 11.0, 3x3 3 -> 22 at 93x84 batch 23 11.9 / 13.0).  Window rows in runs, but for 49 to 64 output channels on few pixels,
// which fill a tile and leave a walking wavefront one or two blocks (best tile / walking: 5 -> 64 3x3/2 at 112x112 batch 16 9.5 / 9.9,
// 1 -> 58 7x7/2 at 93x147 batch 31 11.5 / 13.4).  Pointwise layers of more than 64 channels and at most three stages that the fp32
// kernel does not read 16 bytes a lane, and those where two or three stages write 64 MB and more (32 -> 272 at 52x53 batch 36 55 / 36,
// 48 -> 240 at 154x34 batch 18 47 / 32; below: 48 -> 256 at 56x56 batch 16 16.1 / 16.5, 32 -> 128 at 90x90 batch 8 10.3 / 11.1;
// one stage: 16 -> 512 at 38x38 batch 62 49 / 57; four: 64 -> 304 at 111x111 batch 39 268 / 299).  With up to two stages and more
// than 512 channels the pixels are read by many groups of workgroups: 2 -> 1005 at 165x91 batch 8 150 / 183.  A single product is as exact on fp32
// instructions as a float can be (2.52e-8 against 64 bits, this 2.58e-8; two products 3.12e-8 / 2.61e-8, 48 of them 1.24e-7 / 4.3e-8).
bool ig_short(const fc_conv_shape &s) {
    long rows;
    const int order = ig_split_order(s, &rows);
    const long npix = (long)s.N * fc_out_dim(s.H, s.pt, s.pb, s.kh, s.sh) * fc_out_dim(s.W, s.pl, s.pr, s.kw, s.sw);
    const double yBytes = 4.0 * s.K * (double)npix;
    if ((long)s.C * s.kh * s.kw < 2 || rows > 64 || s.kh * s.kw > 64 || 4l * s.N * s.C * s.H * s.W >= (1l << 31) || yBytes > kShortNoStore) return false;
    if ((rows <= 32 && s.K > 512) || (npix + 31) / 32 * ((s.K + 31) / 32) < 25 * 256) return false;
    if (order != IG_ORDER_BLOCK) return s.K <= 48 || s.K > 64 || npix >= 32 * 8192;
    return ig_point(s) && s.K > 64 && rows <= 48 && (!ig_pointwise(s, 16, true) || (rows > 16 && yBytes >= 64e6));
}

// Pointwise layers of 33 to 64 output channels whose filter is packed in fp32, on three workgroups of 128 pixels a CU and more: split from
// that filter.  Us, fp32 instructions / this: 256 -> 64 at 56x56 batch 32 38.7 / 36.3, 64 -> 64 12.5 / 12.2, 96 -> 64 at 102x102 batch 28 49.1 /
// 48.3.  Eight layers of 88 000 to 97 000 pixels are 2 to 10 % faster too, sixteen of 50 000 to 82 000 between 4 % slower and 10 % faster
// (256 -> 64 at 56x56 batch 16 20.2 / 18.4, batch 24 26.9 / 27.9), of 40 000 slower (64 -> 64 at 200x200 7.1 / 7.9, 512 -> 64 29.6 / 37.9).
// A filter packed in parts is the faster one (this / packed in parts: 100 -> 64 at 102x102 batch 28 50.3 / 49.4, 900 -> 64 at 104x104 batch
// 10 109 / 100, 200 -> 40 at 100x100 batch 12 31.4 / 29.4).
bool ig_point_few(const fc_conv_shape &s) {
    return ig_four_pixels(s) && s.K > 32 && s.K <= 64 && s.C > 48 && (long)s.N * s.H * s.W >= 768 * 128 && 4l * s.N * s.C * s.H * s.W < (1l << 31);
}

// Stages of the first of two levels of sums.  Errors of sums in one level are smallest in parts of about the root of the number of stages
// each; more than 15 give no time, fewer cost some: 256 -> 256 3x3/2 at 28x28 batch 32, 144 stages, in five parts 9 57.6 us and 8.9e-8 against
// 64 bits, 15 56.6 and 9.6e-8 (one level, eight parts: 1.05e-7); 144 -> 832 3x3/2 at 44x22 batch 4, 81 stages, 9 8.3e-8, 15 9.2e-8 (eight
// parts: 9.1e-8).
int ig_sum_stages(int stages) { return std::max(4, std::min(15, (int)sqrt((double)stages))); }

// Row orders, runs of `run` columns: which of them may start before x.  The row of such a run is inside the image, so that it
// starts (n * C + c) * H * W + row * W - pl floats from the start of x or later: images, channels, rows below these bounds.
void ig_before(const fc_conv_shape &s, int run, IgemmParams &p) {
    p.pixBefore = 0;
    p.stagesBefore = 0;
    if (s.pl == 0) return;
    const long last = s.pl - 1, image = (long)s.H * s.W;
    const long n = last / (s.C * image), oh = (s.pt + last / s.W) / s.sh, channels = std::min<long>(s.C, 1 + last / image);
    p.pixBefore = (n * p.OH + std::min<long>(p.OH, oh + 1)) * p.OW;
    p.stagesBefore = (int)((channels * s.kh * ((s.kw + run - 1) / run) * run + 15) / 16);
}

bool ig_sums_in_levels(const fc_conv_shape &s, IgTileSize tile, long blocks, int stages, int parts);

// The kernels behind the plans of the LDS-tiled configurations.  A layer that is left to the library goes to the kernels for short reductions
// and for few output channels by the lines above; a caller's own configuration is the tile that it names, so that configurations can be
// compared.
enum { IG_RUN_CONV, IG_RUN_SPLIT, IG_RUN_POINT_FEW, IG_RUN_SHORT };
int ig_route(const fc_conv_shape &s, const fc_gemm_config &cfg, int K_pad, int splitK) {
    const bool few = ig_point_few(s) && K_pad == 64 && !ig_splits(s, cfg);
    if (splitK == 1 && (few || ig_short(s)) && cfg.id == fc_igemm_default_config(&s)) return few ? IG_RUN_POINT_FEW : IG_RUN_SHORT;
    return ig_splits(s, cfg) ? IG_RUN_SPLIT : IG_RUN_CONV;
}

template <class TL>
void launch(fc_context *ctx, const fc_conv_shape &s, const fc_gemm_config &cfg, IgemmParams &p) {
    const int route = ig_route(s, cfg, p.K_pad, p.splitK);
    if (route == IG_RUN_POINT_FEW) {
        typedef IgSplit<64, 128, 4> S;
        p.nKB = 1;
        p.nPB = (int)((p.Npix + S::BN_ - 1) / S::BN_);
        igemm_split_kernel<S, SP_POINT32><<<dim3((unsigned)((p.nPB + 7l) / 8 * 8)), dim3(S::THREADS), 0, ctx->stream>>>(p);
        return;
    }
    if (route == IG_RUN_SHORT) {
        long rows;
        const int order = ig_split_order(s, &rows);
        ig_before(s, order == IG_ORDER_ROW8 ? 8 : 4, p);
        ig_short_launch(ctx, order == IG_ORDER_ROW8 ? SP_ROW8 : order == IG_ORDER_ROW4 ? SP_ROW4 : ig_four_pixels(s) ? SP_POINT : SP_PAD,
                        rows, ig_splits(s, cfg), p);
        return;
    }
    if constexpr (!std::is_void<typename IgSplitOf<TL>::type>::value) {
        if (route == IG_RUN_SPLIT) {
            typedef typename IgSplitOf<TL>::type S;
            const dim3 grid((unsigned)(((long)p.nKB * p.nPB + 7) / 8 * 8), (unsigned)p.splitK), block(S::THREADS);
            long rows;
            const int order = ig_order(s, cfg, &rows);
            ig_before(s, order == IG_ORDER_ROW8 ? 8 : 4, p);
            auto run = [&](auto mode, auto levels) { igemm_split_kernel<S, decltype(mode)::value, decltype(levels)::value><<<grid, block, 0, ctx->stream>>>(p); };
            constexpr std::false_type one{};
            if (order == IG_ORDER_ROW8) return run(std::integral_constant<int, SP_ROW8>(), one);
            if (order == IG_ORDER_ROW4) return run(std::integral_constant<int, SP_ROW4>(), one);
            if constexpr (S::BM_ == 64) {
                // two 16-byte loads a stage and wavefront in place of eight of 4 bytes, whole layers of batch 32, us: 256 -> 64 at
                // 56x56 28.2 / 26.0, 1024 -> 256 at 14x14 34.7 / 32.9, 112 -> 208 at 68x68 batch 4 13.4 / 12.3.  Tiles of 128 rows
                // load half as often for their products: 64 -> 256 at 56x56 30.6 / 32.3, 144 -> 112 at 130x130 batch 35 173 / 178.  Nor where
                // few wavefronts a CU walk a long reduction, whose every stage waits for the turn: 976 -> 96 at 40x77 batch 8, 61 stages, 770
                // workgroups, 58.9 / 61.2, 720 -> 96 at 116x116 batch 2 39.2 / 42.8; 944 -> 80 at 164x164 batch 2, 1682, 88.5 / 82.7.
                const long pairs = (long)p.nKB * p.nPB * p.splitK * (S::THREADS / 128);
                if (ig_four_pixels(s) && (p.stagesPerSplit <= 40 || pairs >= 1024)) return run(std::integral_constant<int, SP_POINT>(), one);
            } else {
                const int stages = p.Kred_pad / 16;
                if (ig_sums_in_levels(s, {S::BM_, S::BN_}, (long)p.nKB * p.nPB, stages, p.splitK)) {
                    constexpr std::true_type two{};
                    p.sumStages = ig_sum_stages(stages);
                    if (ig_inside(s, 16)) return run(std::integral_constant<int, SP_INSIDE>(), two);
                    return run(std::integral_constant<int, SP_MASKED>(), two);
                }
                // strided layers under tiles of 128 rows, batch 32, us: 128 -> 128 at 56x56 76.0 / 71.9, 256 -> 256 at 28x28 69.6 / 67.0,
                // 32 -> 448 at 100x100 batch 22 107.8 / 103.6.  (Stride 1 loads find their lines in the cache: 256 -> 256 at 56x56 batch 8
                // 192 / 197; tiles of 64 rows lose a wavefront a SIMD to the registers: 64 -> 64 at 56x56 50.8 / 57.2)
                if (s.kw == 3 && s.sw > 1 && s.pl <= 1) return run(std::integral_constant<int, SP_TRI>(), one);
            }
            if (s.C % 16 != 0) return run(std::integral_constant<int, SP_PAD>(), one);
            if (ig_inside(s, 16)) return run(std::integral_constant<int, SP_INSIDE>(), one);
            return run(std::integral_constant<int, SP_MASKED>(), one);
        }
    }
    const bool x16 = ((uintptr_t)p.x & 15) == 0;
    const bool pointwise = ig_pointwise(s, TL::BK_, x16), inside = ig_inside(s, TL::BK_);
    // one 32-bit byte offset with bit 31 to spare reaches every element of the tensor
    const bool buffer = p.xBytes < (1l << 31);
    const bool tapMajor = p.C % TL::BK_ == 0;      // the order fc_igemm_pack_filter laid the filter out in
    const dim3 grid((unsigned)(((p.nKB * p.nPB + 7) / 8) * 8), (unsigned)p.splitK), block(TL::THREADS);
    if (pointwise) igemm_conv_kernel<TL, IG_POINTWISE><<<grid, block, 0, ctx->stream>>>(p);
    else if (buffer && tapMajor && inside) igemm_conv_kernel<TL, IG_TAP_INSIDE><<<grid, block, 0, ctx->stream>>>(p);
    else if (buffer && tapMajor && p.kh * p.kw <= 64) igemm_conv_kernel<TL, IG_TAP_MASKED><<<grid, block, 0, ctx->stream>>>(p);
    else if (buffer && p.kh * p.kw <= 64) igemm_conv_kernel<TL, IG_BUF_MASKED><<<grid, block, 0, ctx->stream>>>(p);      // the taps of a window are one 64-bit mask
    else igemm_conv_kernel<TL, IG_GATHER><<<grid, block, 0, ctx->stream>>>(p);
}

// Layers on split products whose reduction is cut into parts by their expected time: windows over whole blocks of channels, several
// images, strided or 100 stages and more.  The others keep as many parts as fill the chip (ig_parts_to_fill): 1x1 layers as the
// expected times do not tell their tiles apart so well (512 -> 2048 at 7x7 batch 32 28 / 33 us), window rows in runs and blocks with
// channels missing as they are ahead and behind about as often (28 -> 38 at 9x45 batch 52 14.9 / 18.6, 548 -> 175 at 21x113 batch 10 235 /
// 245, 168 -> 631 at 8x8 batch 18 36.9 / 31.9).  Neither several images nor 100 stages is where it ceases to pay: 24 layers of one image take 0.93 of the
// time by it, 24 of several at stride 1 with fewer stages 0.96 (0.80 to 1.08 each; 192 -> 360 5x5/2 at 100x115 85 / 69, 128 -> 672 3x3 at 10x8 batch
// 51 67 / 55, 16 -> 384 at 33x33 batch 16 17.9 / 19.4), so that the line could be drawn lower.
bool ig_parts_by_time(const fc_conv_shape &s) {
    const long taps = (long)s.kh * s.kw;
    return taps > 1 && s.N > 1 && s.C % 16 == 0 && (s.sh > 1 || s.sw > 1 || s.C / 16 * taps >= 100);
}

// Expected time of a layer on the bf16 matrix cores, in us, under one of the tile shapes 128x128, 64x128, 128x64 and 64x64
// (configurations 0 to 3).  A CU takes a stage of a workgroup every `cycles` (block or row order), however many it holds, and
// one workgroup takes at least `latency` for it; beside that the start of a round, memory, and for a split reduction the pass
// over the partial sums.  The constants are a least squares fit.  On 217 drawn layers that it was not made on (1x1, 3x3, 5x5 and 7x7,
// one to 64 images, 1 to 1024 channels, 0.1 to 60 GFLOP; profiles/igemm_untuned_choice.txt): standard deviation 12 %, the choice
// among the four 1.7 % behind the best of them on average, 5.6 % or more on a tenth of the layers, 26 % at most.  On 1495 layers under up to ten
// numbers of parts each: 14 %, the choice among all of them 3.3 % behind the best on average (2.3 % in row orders, with 1.2 of `latency`), 11 % or more on a tenth; constants
// fitted to those, for 1x1 layers apart, choose no better (3.1 %).
struct IgSplitCost {
    int bm, bn, perCu;
    double cyclesBlock, cyclesRow, latency, start;
};
const IgSplitCost kIgSplitCost[] = {{128, 128, 2, 1121, 1032, 1602, 928}, {64, 128, 4, 756, 713, 1041, 535},
                                    {128, 64, 4, 621, 563, 1821, 711}, {64, 64, 8, 420, 398, 1031, 313}};

// `refined`: with the grid as it is launched, in whole eights of tiles, where the number of parts is chosen by what fits the chip at once, and
// with 1.2 of `latency` in row orders; the untuned tile is chosen without first (ig_split_default_config).
double ig_split_us(const fc_conv_shape &s, int config, const fc_igemm_plan &plan, bool refined) {
    const IgSplitCost &c = kIgSplitCost[config];
    long rows;
    const int order = ig_order(s, kIgConfigs[config], &rows);
    const double stages = ceil(ceil(rows / 16.0) / plan.split_k), kBlocks = ceil((double)s.K / c.bm);
    double cycles = order == IG_ORDER_BLOCK ? c.cyclesBlock : c.cyclesRow;
    if (c.bm == 64 && s.K % 64 != 0 && s.K % 64 <= 32) cycles *= (kBlocks - 1 + 0.59) / kBlocks;      // half of the last rows
    const double tiles = kBlocks * ceil((double)plan.Npix / c.bn), latency = refined && order != IG_ORDER_BLOCK ? 1.2 * c.latency : c.latency;
    const double blocks = (refined && ig_parts_by_time(s) ? ceil(tiles / 8) * 8 : tiles) * plan.split_k, slots = 256.0 * c.perCu;
    auto round = [&](double perCu) { return stages * fmax(latency, perCu * cycles) + c.start * (1 + 2.3 * perCu); };
    const double full = floor(blocks / slots), rest = blocks - full * slots;
    const double compute = (full * round(c.perCu) + (rest > 0 ? round(ceil(rest / 256)) : 0)) / 2000;
    const double bytes = 4.0 * ((double)s.N * s.C * s.H * s.W / (s.kh * s.kw == 1 ? s.sh * s.sw : 1) + (double)s.K * plan.Npix);
    const double memory = bytes / 4.99e6;
    const double us = 4.5 + sqrt(sqrt(compute * compute * compute * compute + memory * memory * memory * memory));
    return plan.split_k > 1 ? us + 3.4 + 2.0 * plan.ws_bytes / 6.65e6 : us;
}

// The same for a kernel that splits the reduction over the wavefronts of a workgroup (same layers: 19 %).
double ig_ws_us(const fc_conv_shape &s, const fc_gemm_config &c, long npix) {
    const double mt = c.bm / 16, nt = c.bn / 16, units = ceil((double)s.C * s.kh * s.kw / 16);
    const double perCu = ceil(ceil((double)s.K / c.bm) * ceil((double)npix / c.bn) / 256);
    const bool table = s.C % 16 != 0, row3 = !table && s.kw == 3;
    const double loads = (mt + 4 * nt / (row3 ? 3 : 1)) * 7.06;
    const double cycles = fmax(loads, 17.1 * mt * nt) + 18.8 * (mt + nt) + (table ? 36.7 * nt : 0);
    return 3.5 + (perCu * units * cycles + 52.8 * perCu * mt * nt * c.waves_k) / 2000;
}

// Small layers do not fill 256 CUs with their tiles: the reduction in as many parts as make about three workgroups per CU,
// keeping >= 4 LDS stages per part.
int ig_parts_to_fill(long blocks, int stages) {
    int splitK = 1;
    // A grid of two to four workgroups per CU is placed unevenly by the dispatcher (some CUs get
    // one more than their share and set the time of the launch): with a long reduction, splitting
    // it to about six per CU is worth the second pass (measured: 3x3 stride-2 layers of ResNet-50
    // at batch 32 -9 %, 2048 -> 512 at 7x7 -6 %; with a short reduction the second pass costs more).
    const bool longReduction = stages >= 64;
    const long below = longReduction ? 1024 : 512, target = longReduction ? 1536 : 768;
    if (blocks < below) {
        splitK = (int)((target + blocks - 1) / blocks);
        if (splitK > stages / 4) splitK = stages / 4;
        if (splitK > 32) splitK = 32;
        if (splitK < 1) splitK = 1;
    }
    return splitK;
}

// A reduction of `stages` in at most `parts` of equal length, none of them empty.
int ig_whole_parts(int stages, int parts) {
    const int per = (stages + parts - 1) / parts;
    return (stages + per - 1) / per;
}

// Whether a tile adds up in two levels: cut by time into fewer parts than fill the chip.
bool ig_sums_in_levels(const fc_conv_shape &s, IgTileSize tile, long blocks, int stages, int parts) {
    return tile.bm == 128 && ig_parts_by_time(s) && parts < ig_whole_parts(stages, ig_parts_to_fill(blocks, stages));
}

// The kernel that adds up partial sums has one workgroup row per output channel.
constexpr int kMaxReduceChannels = 65535;

// Plans that cannot run because of their partial sums (kMaxReduceChannels) are behind all others.
// A layer that the best tile would fill the chip with only in several parts (ig_parts_to_fill, whether it is then split or not) goes to
// the kernels that split it inside the workgroup where those are expected ahead, from 9 parts on also where they are 15 % behind and
// from 21 on 50 %: the model then favours the tiles.  Of 1495 drawn layers 321 go, at 0.71 of the tile's time on average; where they
// take 20 us and more the two are level.
int ig_plan_to_fill(const fc_conv_shape *s, int config, fc_igemm_plan *plan);
int ig_split_default_config(const fc_conv_shape *s) {
    int best = 3;
    double bestUs = 1e300;
    bool bestRuns = false;
    fc_igemm_plan plan, bestPlan = {};
    for (int id = 0; id < 4; id++) {
        if (ig_plan_to_fill(s, id, &plan) != FC_OK) continue;
        const double us = ig_split_us(*s, id, plan, false);
        const bool runs = plan.split_k == 1 || s->K <= kMaxReduceChannels;
        if (runs != bestRuns ? runs : us < bestUs) { bestUs = us; best = id; bestPlan = plan; bestRuns = runs; }
    }
    const int parts = bestPlan.split_k;      // 0: a layer that fc_igemm_make_plan refuses
    const int ws = parts > 1 ? fc_igemm_ws_choose(s, plan.Npix) : -1;
    if (ws >= 0) {
        fc_gemm_config c;
        fc_igemm_ws_get_config(ws, kNumIgConfigs + ws, &c);
        const double behind = parts > 20 ? 1.5 : parts > 8 ? 1.15 : 1.0;
        if (!bestRuns || ig_ws_us(*s, c, plan.Npix) < bestUs * behind) return kNumIgConfigs + ws;
    }
    // A second look where parts are chosen by time, and among layers in row orders that fill the chip unsplit: a tile that is expected ahead
    // and asks for no more memory, so that callers who had room for the first one have it for this, and whose sums are no longer.  (The static workspace takes plans
    // past its size of the untuned tile alone: the first one stays where its plan is such a one.)
    const bool byTime = ig_parts_by_time(*s);
    long rows;
    if (parts == 0 || (!byTime && (parts > 1 || ig_split_order(*s, &rows) == IG_ORDER_BLOCK))) return best;
    const size_t room = bestPlan.Wp_bytes + bestPlan.table_bytes + bestPlan.ws_bytes;
    double least = (byTime ? 0.94 : 1.0) * ig_split_us(*s, best, bestPlan, true);
    fc_igemm_make_plan(s, best, &plan);
    if (plan.ws_bytes > (size_t)FC_IGEMM_STATIC_WS_BYTES) return best;
    if (plan.split_k < parts) least = ig_split_us(*s, best, plan, true);
    const int first = best;
    for (int id = 0; id < 4; id++) {
        if (id == first || fc_igemm_make_plan(s, id, &plan) != FC_OK || plan.Wp_bytes + plan.table_bytes + plan.ws_bytes > room) continue;
        const IgSplitCost &c = kIgSplitCost[id];
        const long blocks = (long)(plan.K_pad / c.bm) * ((plan.Npix + c.bn - 1) / c.bn);
        if (plan.split_k < parts && !ig_sums_in_levels(*s, {c.bm, c.bn}, blocks, plan.Kred_pad / 16, plan.split_k)) continue;
        const double us = ig_split_us(*s, id, plan, true);
        if (us < least) { least = us; best = id; }
    }
    return best;
}

}  // namespace

// Configuration ids: the LDS-tiled shapes of this file first, then the shapes of implicit_gemm_wavesplit.hip.
extern "C" int fc_igemm_num_configs(void) { return kNumIgConfigs + fc_igemm_ws_num_shapes(); }

extern "C" int fc_igemm_get_config(int id, fc_gemm_config *cfg) {
    if (!cfg || id < 0 || id >= fc_igemm_num_configs()) return FC_ERR_INVALID;
    if (id < kNumIgConfigs) *cfg = kIgConfigs[id];
    else fc_igemm_ws_get_config(id - kNumIgConfigs, id, cfg);
    return FC_OK;
}

// Untuned choice on fp32 instructions: padded multiply-adds divided by the rate each tile shape sustains relative to
// 64x64x16 (measured on MI355X over pointwise, strided and 3x3 layers at batch 32; the shapes with
// 128 accumulators per wavefront run one or two workgroups per CU and fall far behind) and by how
// evenly the grid fills the chip.
extern "C" int fc_igemm_default_config(const fc_conv_shape *s) {
    if (!fc_shape_ok(s)) return FC_ERR_INVALID;
    // (1x1 layers of at most 32 output channels have the choice below, with 32 rows a tile or the reduction split inside the
    // workgroup.  Batch 32, us, that choice / best of the split tiles: stride 2 256 -> 32 at 56x56 15.4 / 18.7, 1024 -> 24
    // at 27x27 20.9 / 24.6, 128 -> 32 at 56x56 13.4 / 14.2; 256 -> 32 at 55x55 23.0 / 20.2.)
    if (ig_splits(*s, kIgConfigs[3]) && !(s->kh * s->kw == 1 && s->K <= 32 && s->C % 16 == 0)) return ig_split_default_config(s);
    static const double kRate[] = {0.93, 0.81, 0.82, 1.00, 0.75, 0.60, 0.62, 0.84};
    static_assert(sizeof(kRate) / sizeof(kRate[0]) == sizeof(kIgConfigs) / sizeof(kIgConfigs[0]), "one rate per configuration");
    const double M = s->K, Kr = (double)s->C * s->kh * s->kw;
    const double Np = (double)s->N * fc_out_dim(s->H, s->pt, s->pb, s->kh, s->sh) * fc_out_dim(s->W, s->pl, s->pr, s->kw, s->sw);
    int best = 0;
    double bestCost = 1e300;
    for (int id = 0; id < kNumIgConfigs; id++) {
        const fc_gemm_config &c = kIgConfigs[id];
        const double mp = ceil(M / c.bm) * c.bm, np = ceil(Np / c.bn) * c.bn, kp = ceil(Kr / c.bk) * c.bk;
        const double blocks = (mp / c.bm) * (np / c.bn);
        const double slots = 256.0 * (c.bm * c.bn > 128 * 128 ? 1 : 4);
        // small layers split their reduction until about 768 workgroups exist (fc_igemm_make_plan)
        const double eff_blocks = blocks < 512 ? 768.0 : blocks;
        const double fill = eff_blocks / (ceil(eff_blocks / slots) * slots);
        const double cost = mp * np * kp / (kRate[id] * (0.8 + 0.2 * fill));
        if (cost < bestCost) { bestCost = cost; best = id; }
    }
    // A layer that this tile shape can only fill the chip with by splitting the reduction over workgroups
    // (a pass of partial sums through memory and a second launch) goes to the kernels that split it inside
    // the workgroup instead, while it is small enough for them.
    fc_igemm_plan plan;
    if (fc_igemm_make_plan(s, best, &plan) == FC_OK && plan.split_k > 1) {
        const int ws = fc_igemm_ws_choose(s, plan.Npix);
        if (ws >= 0) return kNumIgConfigs + ws;
    }
    return best;
}

// The reduction of a plan in such parts.
static void ig_set_parts(fc_igemm_plan &plan, int stages, int parts) {
    plan.split_k = ig_whole_parts(stages, parts);
    plan.ws_bytes = plan.split_k > 1 ? sizeof(float) * (size_t)plan.split_k * plan.shape.K * plan.Npix : 0;
}

// In no more parts than have room for their sums: the packed filter does not depend on the number of parts.
static void ig_split_to_fit(fc_igemm_plan &plan, size_t ws_bytes) {
    fc_gemm_config cfg;
    fc_igemm_get_config(plan.config, &cfg);
    const size_t parts = ws_bytes / (sizeof(float) * (size_t)plan.shape.K * plan.Npix);
    ig_set_parts(plan, plan.Kred_pad / cfg.bk, (int)std::max<size_t>(1, std::min<size_t>(plan.split_k, parts)));
}

namespace {

// A plan in the parts that fill the chip (ig_parts_to_fill).
int ig_plan_to_fill(const fc_conv_shape *s, int config, fc_igemm_plan *plan) {
    if (!plan || !fc_shape_ok(s)) return FC_ERR_INVALID;
    fc_gemm_config cfg;
    const int rc = fc_igemm_get_config(config, &cfg);
    if (rc) return rc;
    if (s->kh > 31 || s->kw > 31) return FC_ERR_UNSUPPORTED;      // the in-image test is a 32-bit mask per axis
    plan->shape = *s;
    plan->OH = fc_out_dim(s->H, s->pt, s->pb, s->kh, s->sh);
    plan->OW = fc_out_dim(s->W, s->pl, s->pr, s->kw, s->sw);
    const long kred = (long)s->C * s->kh * s->kw;
    const long npix = (long)s->N * plan->OH * plan->OW;
    if (kred >= (1l << 28) || npix >= (1l << 31) || (long)s->C * s->H * s->W >= (1l << 31)) return FC_ERR_UNSUPPORTED;
    plan->Kred = (int)kred;
    long rows = kred;
    bool split = false;
    if (config < kNumIgConfigs) {
        split = ig_splits(*s, cfg);
        ig_order(*s, cfg, &rows);
        if (rows >= (1l << 28)) return FC_ERR_UNSUPPORTED;
    }
    plan->Kred_pad = (int)fc_round_up(rows, cfg.bk);
    const IgTileSize tile = ig_tile_size(*s, cfg);
    plan->K_pad = (int)fc_round_up(s->K, tile.bm);
    plan->Npix = npix;
    plan->config = config;
    // in fp32 and, where products are split, in three bf16 parts
    plan->Wp_bytes = (sizeof(float) + (split ? 6 : 0)) * (size_t)plan->Kred_pad * plan->K_pad;
    plan->table_bytes = sizeof(int32_t) * 2 * (size_t)plan->Kred_pad;
    if (config >= kNumIgConfigs) {
        // the reduction is split inside the workgroups: one launch, no workspace
        if (!fc_igemm_ws_supports(s)) return FC_ERR_UNSUPPORTED;
        plan->split_k = 1;
        plan->ws_bytes = 0;
        return FC_OK;
    }
    const long blocks = (long)(plan->K_pad / tile.bm) * ((npix + tile.bn - 1) / tile.bn);
    const int stages = plan->Kred_pad / cfg.bk;
    ig_set_parts(*plan, stages, ig_parts_to_fill(blocks, stages));
    return FC_OK;
}

// In the number of parts, at least four stages each and no more than fill the chip, that is expected to take the least time where that is 6 %
// less (ig_parts_by_time), under tiles of 128 rows, which then add up in two levels.  Before / with this and the untuned tile after it, us, and
// error against 64 bits: batch 32 256 -> 256 3x3/2 at 28x28, 128x64 tiles in 8 / 5 parts, 67.5 / 56.8, 1.05e-7 / 9.1e-8; 128 -> 128 3x3/2 at 56x56,
// 128x64 in 4 / 128x128 in 2, 75.5 / 59.5, 9.8e-8 / 8.1e-8; 512 -> 512 3x3/2 at 14x14, 128x64 / 128x128 in 9, 69.9 / 58.3, 1.16e-7 / 1.05e-7.  The error
// of none of 103 drawn layers that it changes is larger, and they take 0.90 of the time on average, 0.75 to 1.12 (496 -> 176 3x3 at 30x30 batch 4).
void ig_expected_parts(fc_igemm_plan &plan) {
    const IgTileSize tile = kIgSplitTiles[plan.config];
    int config = 0;      // the one of the four costed tiles that runs
    while (kIgSplitCost[config].bm != tile.bm || kIgSplitCost[config].bn != tile.bn) config++;
    if (tile.bm != 128) return;
    const int stages = plan.Kred_pad / 16, fill = plan.split_k;
    int best = fill;
    double bestUs = plan.shape.K > kMaxReduceChannels ? 1e300 : 0.94 * ig_split_us(plan.shape, config, plan, true);
    for (int parts = 1; parts < fill; parts++) {
        ig_set_parts(plan, stages, parts);
        if (plan.split_k != parts || (parts > 1 && plan.shape.K > kMaxReduceChannels)) continue;
        const double us = ig_split_us(plan.shape, config, plan, true);
        if (us < bestUs) { bestUs = us; best = parts; }
    }
    ig_set_parts(plan, stages, best);
}

}  // namespace

extern "C" int fc_igemm_make_plan(const fc_conv_shape *s, int config, fc_igemm_plan *plan) {
    const int rc = ig_plan_to_fill(s, config, plan);
    if (rc == FC_OK && plan->split_k > 1 && fc_igemm_splits_products(plan) && ig_parts_by_time(*s)) ig_expected_parts(*plan);
    return rc;
}

extern "C" int fc_igemm_splits_products(const fc_igemm_plan *plan) {
    return plan && plan->config >= 0 && plan->config < kNumIgConfigs && ig_splits(plan->shape, kIgConfigs[plan->config]) ? 1 : 0;
}

extern "C" const char *fc_igemm_kernel_name(const fc_igemm_plan *plan) {
    if (!plan || plan->config < 0 || plan->config >= fc_igemm_num_configs()) return "";
    if (plan->config >= kNumIgConfigs) return "igemm_wavesplit_kernel";
    const int route = ig_route(plan->shape, kIgConfigs[plan->config], plan->K_pad, plan->split_k);
    return route == IG_RUN_CONV ? "igemm_conv_kernel" : route == IG_RUN_SHORT ? "igemm_short_kernel" : "igemm_split_kernel";
}

extern "C" int fc_igemm_on_bf16(const fc_igemm_plan *plan) {
    return plan && plan->config >= 0 && plan->config < kNumIgConfigs &&
           ig_route(plan->shape, kIgConfigs[plan->config], plan->K_pad, plan->split_k) != IG_RUN_CONV ? 1 : 0;
}

static int ig_plan_check(fc_context *ctx, const fc_igemm_plan *plan) {
    if (!fc_ctx_ok(ctx)) return FC_ERR_STATE;
    if (!plan) return fc_set_error(ctx, FC_ERR_INVALID, "null plan", hipSuccess);
    fc_igemm_plan chk;
    const int rc = ig_plan_to_fill(&plan->shape, plan->config, &chk);
    if (rc) return fc_set_error(ctx, rc, "plan does not describe a supported layer", hipSuccess);
    // Parts chosen by time are not chosen again on every call (0.2 us in place of 3.7 to 5.2): any number of them that leaves each four
    // stages is run, as the packed filter does not depend on it.
    const int stages = chk.Kred_pad / 16;
    if (plan->split_k > 0 && plan->split_k <= std::max(1, std::min(32, stages / 4)) && fc_igemm_splits_products(&chk) && ig_parts_by_time(chk.shape))
        ig_set_parts(chk, stages, plan->split_k);
    if (!fc_same_igemm_plan(chk, *plan))
        return fc_set_error(ctx, FC_ERR_INVALID, "plan fields were modified after fc_igemm_make_plan", hipSuccess);
    return FC_OK;
}

extern "C" int fc_igemm_pack_filter(fc_context *ctx, const fc_igemm_plan *plan, const float *w_dev, float *Wp_dev,
                                    int32_t *table_dev) {
    const int rc = ig_plan_check(ctx, plan);
    if (rc) return rc;
    if (!w_dev || !Wp_dev || !table_dev) return fc_set_error(ctx, FC_ERR_INVALID, "fc_igemm_pack_filter: null buffer", hipSuccess);
    const fc_conv_shape &s = plan->shape;
    // (padded window rows or channels may take the rows of the packed filter past this)
    if (fc_round_up(plan->Kred, 16) / 4 > 65535) return fc_set_error(ctx, FC_ERR_UNSUPPORTED, "fc_igemm_pack_filter: reduction too long", hipSuccess);
    const dim3 grid((plan->K_pad + 63) / 64, std::min((plan->Kred_pad + 3) / 4, 65535));
    if (plan->config >= kNumIgConfigs) return fc_igemm_ws_pack(ctx, plan, w_dev, Wp_dev, table_dev);
    fc_gemm_config cfg;
    fc_igemm_get_config(plan->config, &cfg);
    long rows;
    const int order = ig_order(s, cfg, &rows);
    fc_stage_scope scope(ctx, FC_STAGE_FILTER_PACK);
    igemm_pack_filter_kernel<<<grid, dim3(256), 0, ctx->stream>>>(w_dev, Wp_dev, table_dev, s.K, s.C, s.kh, s.kw, s.H,
                                                                 s.W, (int)rows, plan->Kred_pad, plan->K_pad, order);
    FC_LAUNCH_CHECK(ctx, "igemm_pack_filter_kernel");
    if (ig_splits(s, cfg)) {
        const long total = (long)(plan->Kred_pad / 16) * (plan->K_pad / 32) * 64;
        if ((total + 255) / 256 >= (1l << 31)) return fc_set_error(ctx, FC_ERR_UNSUPPORTED, "fc_igemm_pack_filter: filter too large", hipSuccess);
        igemm_split_filter_kernel<<<dim3((unsigned)((total + 255) / 256)), dim3(256), 0, ctx->stream>>>(
            Wp_dev, reinterpret_cast<fc_uintx4 *>(Wp_dev + (size_t)plan->Kred_pad * plan->K_pad), plan->K_pad, total);
        FC_LAUNCH_CHECK(ctx, "igemm_split_filter_kernel");
    }
    return FC_OK;
}

// Launches of one layer; `timed` brackets the GEMM kernel with events when stage timing is on.
static int igemm_run(fc_context *ctx, const fc_igemm_plan *plan, const float *x_dev, const float *Wp_dev,
                     const int32_t *table_dev, const float *bias_dev, int relu, float *ws_dev, float *y_dev, bool timed,
                     const char *entry);

extern "C" int fc_conv_implicit_gemm(fc_context *ctx, const fc_igemm_plan *plan, const float *x_dev,
                                     const float *Wp_dev, const int32_t *table_dev, const float *bias_dev, int relu,
                                     float *ws_dev, float *y_dev) {
    const int rc = ig_plan_check(ctx, plan);
    if (rc) return rc;
    return igemm_run(ctx, plan, x_dev, Wp_dev, table_dev, bias_dev, relu, ws_dev, y_dev, true, "fc_conv_implicit_gemm");
}

// ---- the same layer with the split-reduction workspace in a static device array ----

// Partial sums of a split reduction, [split][K][N*OH*OW] floats, for callers that cannot allocate.
// Every GPU the library runs on holds its own copy of this array until the process ends.
static __device__ __align__(256) float scratch[FC_IGEMM_STATIC_WS_BYTES / sizeof(float)];

// Device address of `scratch` per device, looked up once per device with that device current.
static const int kMaxDevices = 64;
static float *g_scratch_ptr[kMaxDevices];
static bool g_scratch_known[kMaxDevices];
// The context that uses the array of a device: the first one to call fc_conv_implicit_gemm_static there, until it is
// destroyed.  Calls of one context are ordered on its stream; another context's would race with them, so they are refused.
static fc_context *g_scratch_owner[kMaxDevices];
static std::mutex g_scratch_mutex;

// Called by fc_destroy.
void fc_igemm_static_release(fc_context *ctx) {
    if (ctx->device < 0 || ctx->device >= kMaxDevices) return;
    std::lock_guard<std::mutex> lock(g_scratch_mutex);
    if (g_scratch_owner[ctx->device] == ctx) g_scratch_owner[ctx->device] = nullptr;
}

// Called by fc_init with ctx->device current.
int fc_igemm_static_init(fc_context *ctx) {
    if (ctx->device < 0 || ctx->device >= kMaxDevices)
        return fc_set_error(ctx, FC_ERR_UNSUPPORTED, "fc_igemm_static_init: device index above 63", hipSuccess);
    std::lock_guard<std::mutex> lock(g_scratch_mutex);
    if (!g_scratch_known[ctx->device]) {
        float *ptr = nullptr;
        FC_HIP_CHECK(ctx, hipGetSymbolAddress((void **)&ptr, HIP_SYMBOL(scratch)));
        if (!ptr) return fc_set_error(ctx, FC_ERR_HIP, "fc_igemm_static_init: null address of the static workspace", hipSuccess);
        g_scratch_ptr[ctx->device] = ptr;
        g_scratch_known[ctx->device] = true;
    }
    ctx->igemm_static_ws = g_scratch_ptr[ctx->device];
    return FC_OK;
}

extern "C" int fc_conv_implicit_gemm_static(fc_context *ctx, const fc_igemm_plan *plan, const float *x_dev,
                                            const float *Wp_dev, const int32_t *table_dev, const float *bias_dev,
                                            int relu, float *y_dev) {
    const int rc = ig_plan_check(ctx, plan);
    if (rc) return rc;
    fc_igemm_plan fits = *plan;
    if (plan->ws_bytes > (size_t)FC_IGEMM_STATIC_WS_BYTES) {
        if (plan->config != fc_igemm_default_config(&plan->shape)) {
            char msg[200];
            snprintf(msg, sizeof msg, "fc_conv_implicit_gemm_static: this layer needs %zu bytes of split-reduction workspace, "
                     "the static one holds %d: use fc_conv_implicit_gemm with a workspace of the caller's", plan->ws_bytes,
                     FC_IGEMM_STATIC_WS_BYTES);
            return fc_set_error(ctx, FC_ERR_UNSUPPORTED, msg, hipSuccess);
        }
        ig_split_to_fit(fits, FC_IGEMM_STATIC_WS_BYTES);
    }
    if (!ctx->igemm_static_ws) return fc_set_error(ctx, FC_ERR_STATE, "fc_conv_implicit_gemm_static: static workspace not set up", hipSuccess);
    {
        std::lock_guard<std::mutex> lock(g_scratch_mutex);
        fc_context *&owner = g_scratch_owner[ctx->device];
        if (owner == nullptr) owner = ctx;
        if (owner != ctx)
            return fc_set_error(ctx, FC_ERR_STATE, "fc_conv_implicit_gemm_static: the static workspace of this GPU is in use by another "
                                "context (one context per GPU may use it at a time; it is free again once that context is destroyed)", hipSuccess);
    }
    // Nothing has to start at zero: every partial sum the reduction reads ([split][k < K][pixel < Npix]) is
    // written by this call's GEMM kernel first.  No event brackets (creating an event may allocate).
    return igemm_run(ctx, &fits, x_dev, Wp_dev, table_dev, bias_dev, relu, ctx->igemm_static_ws, y_dev, false,
                     "fc_conv_implicit_gemm_static");
}

static int igemm_run(fc_context *ctx, const fc_igemm_plan *plan, const float *x_dev, const float *Wp_dev,
                     const int32_t *table_dev, const float *bias_dev, int relu, float *ws_dev, float *y_dev, bool timed,
                     const char *entry) {
    char msg[160];
    auto fail = [&](int status, const char *what) {
        snprintf(msg, sizeof msg, "%s: %s", entry, what);
        return fc_set_error(ctx, status, msg, hipSuccess);
    };
    if (!x_dev || !Wp_dev || !table_dev || !y_dev) return fail(FC_ERR_INVALID, "null buffer");
    if ((uintptr_t)Wp_dev & 15) return fail(FC_ERR_INVALID, "Wp must be 16-byte aligned");
    if (plan->split_k > 1 && !ws_dev) return fail(FC_ERR_INVALID, "this plan splits the reduction and needs ws_bytes of workspace");
    if (plan->config >= kNumIgConfigs)
        return fc_igemm_ws_run(ctx, plan, plan->config - kNumIgConfigs, x_dev, Wp_dev, table_dev, bias_dev, relu, y_dev, timed);
    fc_gemm_config cfg;
    fc_igemm_get_config(plan->config, &cfg);
    const fc_conv_shape &s = plan->shape;
    IgemmParams p;
    p.x = x_dev; p.Wp = Wp_dev; p.table = table_dev; p.bias = bias_dev; p.y = y_dev;
    p.Ws = reinterpret_cast<const fc_uintx4 *>(Wp_dev + (size_t)plan->Kred_pad * plan->K_pad);
    p.N = s.N; p.C = s.C; p.H = s.H; p.W = s.W; p.K = s.K; p.OH = plan->OH; p.OW = plan->OW;
    p.kh = s.kh; p.kw = s.kw; p.sh = s.sh; p.sw = s.sw; p.pt = s.pt; p.pl = s.pl; p.relu = relu;
    p.Kred_pad = plan->Kred_pad; p.K_pad = plan->K_pad; p.Npix = plan->Npix;
    p.xBytes = 4l * s.N * s.C * s.H * s.W;
    const IgTileSize tile = ig_tile_size(s, cfg);
    p.nKB = plan->K_pad / tile.bm;
    p.nPB = (int)((plan->Npix + tile.bn - 1) / tile.bn);
    p.divOHW = fc_make_fastdiv((uint32_t)(plan->OH * plan->OW));
    p.divOW = fc_make_fastdiv((uint32_t)plan->OW);
    p.splitK = plan->split_k;
    p.stagesPerSplit = ((plan->Kred_pad / cfg.bk) + plan->split_k - 1) / plan->split_k;
    p.sumStages = 0;
    p.ws = ws_dev;
    p.fastStore = s.K % tile.bm == 0 && 4.0 * s.N * s.K * plan->OH * plan->OW < 4294967296.0 &&
                  4.0 * plan->split_k * s.K * (double)plan->Npix < 4294967296.0 && ((uintptr_t)bias_dev & 15) == 0;
    if ((long)p.nKB * p.nPB >= (1l << 31)) return fail(FC_ERR_UNSUPPORTED, "grid too large");
    fc_stage_scope scope(ctx, timed ? FC_STAGE_IMPLICIT_GEMM : -1);
    switch (plan->config) {
        case 0: launch<Ig0>(ctx, s, cfg, p); break;
        case 1: launch<Ig1>(ctx, s, cfg, p); break;
        case 2: launch<Ig2>(ctx, s, cfg, p); break;
        case 3: launch<Ig3>(ctx, s, cfg, p); break;
        case 4: launch<Ig4>(ctx, s, cfg, p); break;
        case 5: launch<Ig5>(ctx, s, cfg, p); break;
        case 6: launch<Ig6>(ctx, s, cfg, p); break;
        case 7: launch<Ig7>(ctx, s, cfg, p); break;
        default: return fail(FC_ERR_INVALID, "unknown tile configuration");
    }
    FC_LAUNCH_CHECK(ctx, "igemm_conv_kernel");
    if (plan->split_k > 1) {
        const dim3 rgrid((unsigned)((plan->Npix + 255) / 256), (unsigned)s.K);
        if (rgrid.y > kMaxReduceChannels) return fail(FC_ERR_UNSUPPORTED, "more than 65535 channels");
        igemm_reduce_kernel<<<rgrid, dim3(256), 0, ctx->stream>>>(ws_dev, bias_dev, y_dev, s.K, plan->Npix,
                                                                  plan->OH * plan->OW, plan->split_k, relu, p.divOHW);
        FC_LAUNCH_CHECK(ctx, "igemm_reduce_kernel");
    }
    return FC_OK;
}
