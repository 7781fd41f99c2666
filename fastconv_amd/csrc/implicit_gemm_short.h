// Implicit GEMM of short reductions on the bf16 matrix cores (see split_mfma.h): a few stages of 16 rows, as in the first
// layer of a network or a 1x1 layer of few channels.  Such a layer mostly writes y, and a workgroup that takes one tile
// spends its life on the way in and out of it.  Here a workgroup stays: it lays its output channels' filter into LDS once, and
// each of its wavefronts then walks over blocks of 32 pixels by itself, without a barrier.  It gathers and splits the whole
// column of each pixel once for all output channels of the workgroup, asks for the columns of its next block before it
// multiplies, and so has loads, products and stores of different blocks in flight beside those of the other wavefronts.
// The filter is split as it goes to LDS, so that the packed one stays as it is.
// What bounds it are the stores of y, 4 bytes a lane: 522 of a wavefront's 670 vector-memory instructions on 3x3 3 -> 64 at 224x224 batch 32,
// whose address units are busy 82 % of the cycles (vector instructions 61 %, matrix pipes 27 %); memory could take them in 0.57 of the time.
// Measured, us, one tile a workgroup on fp32 instructions / this: 3x3 3 -> 64 at 224x224 batch 32 128 / 105 (3.9 TB/s of y; a plain
// fill reaches 6.9), 4 -> 128 at 112x112 batch 16 41 / 30, 4 -> 80 at 102x189 batch 30 119 / 67, 3 -> 808 at 104x104 batch 8 93 / 72;
// 1x1 18 -> 85 at 106x106 batch 18 45 / 19, 48 -> 240 at 154x34 batch 18 47 / 32, 48 -> 213 at 159x159 batch 18 209 / 182.  Tried and
// no faster: columns asked for two blocks ahead, or the first ones before the filter; stores of 16 bytes a lane through LDS (3 -> 808
// 66 / 77 with a filter split beforehand: the LDS they take leaves room for fewer channels).
#pragma once

struct IgShortParams {
    int blocksPerWg, groups;      // 32-channel blocks a workgroup holds, groups of them
    int walkers;                  // workgroups that walk over the pixels of an XCD, per group
    long pixBlocks, perXcd;       // blocks of 32 pixels, all and of an XCD
    uint32_t yBytes;
    int row[64];                  // of the packed filter for each row of this kernel's order, -1: padding
    int runOff[16], runTap[16];   // row orders: offset of a run from the window origin, window row << 16 | column
};
constexpr uint32_t kShortNoStore = 0xfffffff0u;      // past the end of y: the host checks that y ends before it

// MODE: SP_POINT, SP_PAD (pointwise layers; channels of one pixel), SP_ROW8, SP_ROW4.
template <int STAGES, int MODE>
__global__ __launch_bounds__(256, STAGES <= 2 ? 4 : STAGES == 3 ? 3 : 2) void igemm_short_kernel(const IgemmParams p, const IgShortParams q) {
    constexpr bool ROW = MODE == SP_ROW8 || MODE == SP_ROW4;
    constexpr int RUNS = MODE == SP_ROW8 ? 2 : 4, RUN = 16 / RUNS;
    constexpr uint32_t OUTSIDE = 0x80000000u;
    extern __shared__ fc_uintx4 shortLds[];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int lrow = lane >> 5, lcol = lane & 31;
    // every XCD walks over a contiguous range of the pixels, its workgroups side by side, so that the lines of y and of x that
    // neighbouring blocks share meet in one L2; the groups of channels that read the same pixels are neighbours on one XCD
    const int xcd = (int)blockIdx.x & 7, j = (int)blockIdx.x >> 3;
    const int group = j % q.groups;
    const long rangeEnd = min(q.pixBlocks, (xcd + 1) * q.perXcd);
    const int firstBlock = group * q.blocksPerWg, nBlocks = min(q.blocksPerWg, (p.K + 31) / 32 - firstBlock);

    // LDS: filter words [block][stage][part][half][channel], the channels' bias, a slot per wavefront to turn columns in
    fc_uintx4 *const filter = shortLds;
    float *const bias = reinterpret_cast<float *>(shortLds + q.blocksPerWg * STAGES * kSplitBlockWords);
    float *const turn = bias + q.blocksPerWg * 32 + wave * 512;
    // eight rows of 64 channels at a time, four such pieces asked for before the first is split
    const int pieces = (nBlocks + 1) / 2 * STAGES * 2;
    for (int i0 = wave; i0 < pieces; i0 += 16) {
        float v[4][8];
#pragma unroll
        for (int u = 0; u < 4; u++) {
            const int i = min(i0 + 4 * u, pieces - 1), s2 = i % (STAGES * 2), block = i / (STAGES * 2) * 2 + lrow;
            const float *const column = p.Wp + (firstBlock + min(block, nBlocks - 1)) * 32 + lcol;
#pragma unroll
            for (int e = 0; e < 8; e++) {
                const int row = q.row[8 * s2 + e];
                v[u][e] = column[(size_t)max(row, 0) * p.K_pad];
                v[u][e] = row >= 0 ? v[u][e] : 0.f;
            }
        }
#pragma unroll
        for (int u = 0; u < 4; u++) {
            const int i = i0 + 4 * u, s2 = i % (STAGES * 2), block = i / (STAGES * 2) * 2 + lrow;
            if (i < pieces && block < nBlocks) fc_split8(v[u], filter + (block * STAGES + s2 / 2) * kSplitBlockWords + s2 % 2 * 32 + lcol, 64);
        }
    }
    for (int e = tid; e < nBlocks * 32; e += 256) bias[e] = p.bias && firstBlock * 32 + e < p.K ? p.bias[firstBlock * 32 + e] : 0.f;
    __syncthreads();

    const uint32_t image = (uint32_t)(p.H * p.W), chanStep = 4u * image, OHW = (uint32_t)(p.OH * p.OW);
    const __amdgpu_buffer_rsrc_t xres = __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(p.x), 0, (int)p.xBytes, 0x00020000);
    auto load1 = [&](const uint32_t voff, const uint32_t soff) __attribute__((always_inline)) {
        return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(xres, voff, soff, 0));
    };
    // the window of a pixel: byte offset of its origin, window rows and columns outside the image
    auto window = [&](const long pix, uint32_t &origin, uint32_t &rowBad, uint32_t &colBad) __attribute__((always_inline)) {
        origin = OUTSIDE;
        rowBad = colBad = ~0u;
        if (pix < p.Npix) {
            const uint32_t n = fc_div((uint32_t)pix, p.divOHW), pp = (uint32_t)pix - n * OHW;
            const uint32_t oh = fc_div(pp, p.divOW), ow = pp - oh * p.OW;
            const int ih0 = (int)oh * p.sh - p.pt, iw0 = (int)ow * p.sw - p.pl;
            origin = 4u * (n * (uint32_t)p.C * image + (uint32_t)(ih0 * p.W + iw0));
            for (int r = 0; r < p.kh; r++) rowBad &= (unsigned)(ih0 + r) < (unsigned)p.H ? ~(1u << r) : ~0u;
            for (int c = 0; c < p.kw; c++) colBad &= (unsigned)(iw0 + c) < (unsigned)p.W ? ~(1u << c) : ~0u;
        }
    };

    float raw[STAGES][8];
    uint32_t cols[STAGES][2];      // row orders: columns of the runs inside the image
    // beforeX: some run may start before x, and is read element by element (whether a 16-byte load there gives the elements
    // inside x is left open)
    auto fetch = [&](const long block, auto beforeX) __attribute__((always_inline)) {
        if constexpr (MODE == SP_POINT) {      // pixels 4 * (lane % 8) .. + 3, channels lane / 8 and 8 on
            const long first = block * 32 + 4 * (lane & 7);
            uint32_t origin = OUTSIDE;
            if (first < p.Npix) {
                const uint32_t n = fc_div((uint32_t)first, p.divOHW);
                origin = 4u * ((n * (uint32_t)p.C + (uint32_t)(lane >> 3)) * image + ((uint32_t)first - n * image));
            }
#pragma unroll
            for (int s = 0; s < STAGES; s++)
#pragma unroll
                for (int h = 0; h < 2; h++) {
                    const int c = 16 * s + 8 * h;
                    const floatx4 d = __builtin_bit_cast(floatx4, __builtin_amdgcn_raw_buffer_load_b128(
                                                                      xres, c + (lane >> 3) < p.C ? origin : OUTSIDE, (uint32_t)min(c, p.C - 1) * chanStep, 0));
#pragma unroll
                    for (int i = 0; i < 4; i++) raw[s][4 * h + i] = d[i];
                }
        } else if constexpr (MODE == SP_PAD) {
            uint32_t origin, rowBad, colBad;
            window(block * 32 + lcol, origin, rowBad, colBad);
            const uint32_t vo = origin == OUTSIDE ? OUTSIDE : origin + 8u * lrow * chanStep;
#pragma unroll
            for (int s = 0; s < STAGES; s++)
#pragma unroll
                for (int i = 0; i < 8; i++)
                    raw[s][i] = load1(16 * s + 8 * lrow + i < p.C ? vo : OUTSIDE, (uint32_t)min(16 * s + i, p.C - 1) * chanStep);
        } else {
            uint32_t origin, rowBad, colBad;
            window(block * 32 + lcol, origin, rowBad, colBad);
#pragma unroll
            for (int s = 0; s < STAGES; s++)
#pragma unroll
                for (int v = 0; v < RUNS / 2; v++) {
                    const int u0 = RUNS * s + v, u1 = u0 + RUNS / 2;
                    const int off = lrow ? q.runOff[u1] : q.runOff[u0], rs = lrow ? q.runTap[u1] : q.runTap[u0];
                    const uint32_t vo = (rowBad >> (rs >> 16)) & 1u ? OUTSIDE : origin + 4u * (uint32_t)off;
                    cols[s][v] = ~colBad >> (rs & 0xffff);
                    if constexpr (decltype(beforeX)::value) {
#pragma unroll
                        for (int i = 0; i < RUN; i++) {
                            const uint32_t at = vo + 4u * (uint32_t)i;
                            raw[s][v * RUN + i] = load1((int)at < 0 ? OUTSIDE : at, 0);
                        }
                    } else {
#pragma unroll
                        for (int h = 0; h < RUN / 4; h++) {
                            const floatx4 d = __builtin_bit_cast(floatx4, __builtin_amdgcn_raw_buffer_load_b128(xres, vo, 16 * h, 0));
#pragma unroll
                            for (int i = 0; i < 4; i++) raw[s][v * RUN + 4 * h + i] = d[i];
                        }
                    }
                }
        }
    };
    fc_uintx4 b[STAGES][3];
    auto split = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int s = 0; s < STAGES; s++) {
            if constexpr (MODE == SP_POINT) {      // four pixels of one channel -> eight channels of one pixel
#pragma unroll
                for (int h = 0; h < 2; h++)
                    *reinterpret_cast<floatx4 *>(turn + 256 * h + 4 * lane) = floatx4{raw[s][4 * h], raw[s][4 * h + 1], raw[s][4 * h + 2], raw[s][4 * h + 3]};
                fc_wave_sync();      // lanes read what other lanes wrote
#pragma unroll
                for (int i = 0; i < 8; i++) raw[s][i] = turn[(8 * lrow + i) * 32 + lcol];
                fc_wave_sync();      // before the next stage is written
            }
            if constexpr (ROW) {
#pragma unroll
                for (int i = 0; i < 8; i++) {
                    const int keep = (int)(cols[s][i / RUN] << (31 - i % RUN)) >> 31;
                    raw[s][i] = __builtin_bit_cast(float, __builtin_bit_cast(int, raw[s][i]) & keep);
                }
            }
            fc_split8(raw[s], b[s], 1);
        }
    };

    // stores go through a buffer resource over y: a lane past the last pixel or channel stores outside it, without a branch,
    // so that the loads of the next block are waited for with the stores after them left in flight
    const float floorv = p.relu ? 0.f : -__builtin_inff();
    const __amdgpu_buffer_rsrc_t yres = __builtin_amdgcn_make_buffer_rsrc(p.y, 0, (int)q.yBytes, 0x00020000);
    auto process = [&](const long block) __attribute__((always_inline)) {
        const long pix = block * 32 + lcol;
        const uint32_t n = fc_div((uint32_t)pix, p.divOHW);
        // bytes from y: this lane's pixel, 4 channels down for the upper half of the wavefront
        const uint32_t yOff = pix < p.Npix ? 4u * (n * (uint32_t)p.K * OHW + ((uint32_t)pix - n * OHW) + 4u * lrow * OHW) : kShortNoStore;
        int kb = 0;
        do {
            floatx16 acc[1][1], small[1][1];
            fc_zero<1, 1>(acc);
            fc_zero<1, 1>(small);
            const fc_uintx4 *as = filter + kb * (STAGES * kSplitBlockWords) + lane;
#pragma unroll
            for (int s = 0; s < STAGES; s++) {
                fc_bf16x8 a[3];
#pragma unroll
                for (int part = 0; part < 3; part++) a[part] = __builtin_bit_cast(fc_bf16x8, as[s * kSplitBlockWords + part * 64]);
                constexpr int pa[5] = {2, 1, 0, 1, 0}, pb[5] = {0, 1, 2, 0, 1};
#pragma unroll
                for (int i = 0; i < 5; i++)
                    small[0][0] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[pa[i]], __builtin_bit_cast(fc_bf16x8, b[s][pb[i]]), small[0][0], 0, 0, 0);
                acc[0][0] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[0], __builtin_bit_cast(fc_bf16x8, b[s][0]), acc[0][0], 0, 0, 0);
            }
            fc_join<1, 1>(acc, small);
            const int k0 = (firstBlock + kb) * 32;
            if (__builtin_amdgcn_ballot_w64(fc_not_finite<1, 1>(acc))) {      // those values again with fp32 instructions
                uint32_t origin, rowBad, colBad;
                window(pix, origin, rowBad, colBad);
                floatx16 again;
#pragma unroll
                for (int i = 0; i < 16; i++) again[i] = 0.f;
                for (int kr = lrow; kr < p.Kred_pad; kr += 2) {
                    const int rs = p.table[2 * kr + 1];
                    const bool out = ((rowBad >> (rs >> 16)) | (colBad >> (rs & 0xffff))) & 1u;
                    const float v = load1(out ? OUTSIDE : origin + 4u * (uint32_t)p.table[2 * kr], 0);
                    again = __builtin_amdgcn_mfma_f32_32x32x2f32(p.Wp[(size_t)kr * p.K_pad + k0 + lcol], v, again, 0, 0, 0);
                }
#pragma unroll
                for (int i = 0; i < 16; i++) acc[0][0][i] = __builtin_isfinite(acc[0][0][i]) ? acc[0][0][i] : again[i];
            }
            const uint32_t row = 4u * (uint32_t)k0 * OHW;
            const int left = p.K - k0 - 4 * lrow;      // channels from the lane's first on that exist
#pragma unroll
            for (int g = 0; g < 4; g++) {      // register 4g + i: channel k0 + 8g + 4 * lrow + i
                const floatx4 add = *reinterpret_cast<const floatx4 *>(bias + kb * 32 + 8 * g + 4 * lrow);
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    const float v = __builtin_elementwise_maximum(acc[0][0][4 * g + i] + add[i], floorv);
                    __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, v), yres, 8 * g + i < left ? yOff : kShortNoStore,
                                                          row + 4u * (uint32_t)min(8 * g + i, p.K - 1 - k0) * OHW, 0);
                }
            }
        } while (++kb < nBlocks);
    };
    const long step = 4l * q.walkers;
    long block = xcd * q.perXcd + 4l * (j / q.groups) + wave;
    if constexpr (ROW)
        for (; block * 32 < p.pixBefore && block < rangeEnd; block += step) {
            fetch(block, std::true_type());
            split();
            process(block);
        }
    if (block >= rangeEnd) return;
    const long last = block + (rangeEnd - 1 - block) / step * step;
    fetch(block, std::false_type());
    for (; block <= last; block += step) {
        split();
        fetch(min(block + step, last), std::false_type());
        process(block);
    }
}

// Dynamic LDS of a workgroup.
static inline size_t ig_short_lds(int stages, int blocks, int mode) { return (size_t)blocks * (stages * kSplitBlockWords * 16 + 128) + (mode == SP_POINT ? 4 * 2048 : 0); }

template <int STAGES>
static void ig_short_launch_mode(fc_context *ctx, int mode, dim3 grid, size_t lds, const IgemmParams &p, const IgShortParams &q) {
    if constexpr (STAGES <= 3) {      // (pointwise layers have no more: ig_short)
        if (mode == SP_POINT) return igemm_short_kernel<STAGES, SP_POINT><<<grid, dim3(256), lds, ctx->stream>>>(p, q);
        if (mode == SP_PAD) return igemm_short_kernel<STAGES, SP_PAD><<<grid, dim3(256), lds, ctx->stream>>>(p, q);
    }
    if (mode == SP_ROW8) igemm_short_kernel<STAGES, SP_ROW8><<<grid, dim3(256), lds, ctx->stream>>>(p, q);
    else igemm_short_kernel<STAGES, SP_ROW4><<<grid, dim3(256), lds, ctx->stream>>>(p, q);
}

// rows: of the reduction in this kernel's order; packed: the packed filter has them in that order (plans of split products).
static void ig_short_launch(fc_context *ctx, int mode, long rows, bool packed, const IgemmParams &p) {
    const int stages = (int)((rows + 15) / 16), blocks = (p.K + 31) / 32;
    const int perCu = stages <= 2 ? 4 : 3;      // workgroups the registers leave a CU
    const long slots = (long)ctx->props.multiProcessorCount * perCu;
    IgShortParams q = {};
    for (int u = 0; u < 64; u++) {
        q.row[u] = u < p.Kred_pad ? u : -1;
        if (!packed && (mode == SP_ROW8 || mode == SP_ROW4)) {
            const int run = mode == SP_ROW8 ? 8 : 4, width = (p.kw + run - 1) / run * run, cr = u / width, col = u - cr * width;
            q.row[u] = u < rows && col < p.kw ? cr * p.kw + col : -1;
        }
    }
    if (mode == SP_ROW8 || mode == SP_ROW4) {
        const int run = mode == SP_ROW8 ? 8 : 4, width = (p.kw + run - 1) / run * run;
        for (int i = 0; i < 16; i++) {
            const int u = i * run, cr = u / width, c = cr / p.kh, r = cr - c * p.kh, col = u - cr * width;
            q.runOff[i] = u < rows ? (c * p.H + r) * p.W + col : 0;
            q.runTap[i] = u < rows ? r << 16 | col : 31 << 16 | 31;
        }
    }
    q.pixBlocks = (p.Npix + 31) / 32;
    // as many channels as LDS holds, fewer where there are not enough pixels for all workgroups
    const long wgs = (q.pixBlocks + 3) / 4;
    q.blocksPerWg = (int)std::min<long>(blocks, std::max<long>(1, blocks * wgs / slots));
    while (q.blocksPerWg > 1 && ig_short_lds(stages, q.blocksPerWg, mode) > std::min<size_t>(65536, 163840 / perCu)) q.blocksPerWg--;
    q.groups = (blocks + q.blocksPerWg - 1) / q.blocksPerWg;
    q.blocksPerWg = (blocks + q.groups - 1) / q.groups;
    q.yBytes = (uint32_t)(4l * p.N * p.K * p.OH * p.OW);
    q.perXcd = (wgs + 7) / 8 * 4;
    q.walkers = (int)std::min<long>(std::max<long>(1, slots / 8 / q.groups), q.perXcd / 4);
    const dim3 grid((unsigned)(8 * q.walkers * q.groups));
    const size_t lds = ig_short_lds(stages, q.blocksPerWg, mode);
    switch (stages) {
        case 1: ig_short_launch_mode<1>(ctx, mode, grid, lds, p, q); break;
        case 2: ig_short_launch_mode<2>(ctx, mode, grid, lds, p, q); break;
        case 3: ig_short_launch_mode<3>(ctx, mode, grid, lds, p, q); break;
        default: ig_short_launch_mode<4>(ctx, mode, grid, lds, p, q); break;
    }
}
