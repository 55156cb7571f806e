/*
 * codec_enc.hpp - the encoder's launches (prism_encode and the end-to-end
 * frame; the stage calls keep the stages apart: codec.hpp).
 */
#pragma once
#include "codec.hpp"

/* enc0 + enc1 in one launch, 8 waves. A block is 4 x 32 enc1 outputs at r1
 * (y1, x1). Their stride-2 taps need e0 rows 2 y1 - 1 .. 2 y1 + 7 and columns
 * 2 x1 - 1 .. 2 x1 + 63, a 9 x 65 region, whose own taps need the 11 x 67
 * frame window around it. The window goes into LDS as in enc0, enc0 of the
 * region into a second LDS array (the same fragments, k order, rounding and
 * ReLU as the stage kernel prism_codec_enc0; zeros where it leaves the map; the halo row and
 * column, 12 % of the region, are the neighbours' too), the block's own 8 x 64
 * e0 pixels from there to the e0 map (the decoder's skip) as whole rows, and
 * enc1 reads its taps from that array (k = tap * 32 + ic, as
 * prism_codec_enc1). Outputs equal the two separate launches bit for bit.
 *
 * Persistent: a workgroup takes its blocks from one XCD's band of the map,
 * keeps both stages' weight fragments in registers and requests the next
 * block's window before this block's math, two pixels of a plane per load.
 * 66 KB of LDS, two workgroups or 16 waves per CU. The LDS port bounds it
 * next to memory (236 MB at 1920x1080), so enc0 takes 3 k-steps, and an enc1
 * wave takes one row tile (w / 2) of the 4 rows of one 16-column tile (w % 2)
 * region row by region row: rows 2, 4 and 6 are read once for the two output
 * rows that share them (27 operand reads for 36 MFMAs). 960x540 23.9 -> 18.8
 * us, 1920x1080 97 -> 67 (against one block a workgroup, 4 waves); without its
 * stores it takes 45, without memory at all 42. */
struct Enc01 {
    static constexpr int BR = CODEC_ENC01_ROWS, BC = CODEC_ENC01_COLS; /* 4 x 32 */
    static constexpr int CH = 9, CP = ENC0_CP, KS0 = ENC0_KS, KS1 = 9;
    static constexpr int ER = 2 * BR + 1, EC = 2 * BC + 1, LDE = 40; /* the e0 region, 32 channels a pixel */
    static constexpr int FR = ER + 2, FC = EC + 3, FP = FC / 2;      /* the frame window, columns in pairs */
    static constexpr int NREG = ER * EC, NPX = BR * BC;
    static constexpr int LDO = 64 + 8;                               /* e1 staging row (halfs) */
    static_assert(FR * FP <= 512, "one pixel pair a thread");
    static_assert(BR == 4 && BC == 32, "8 waves: 4 row tiles x 2 column tiles");
};
struct Enc01Lds {
    union {
        __attribute__((aligned(16))) f16 s_in[Enc01::FR * Enc01::FC * Enc01::CP + 8]; /* frame window */
        __attribute__((aligned(16))) f16 e1[Enc01::NPX * Enc01::LDO];                 /* then the e1 tile */
    };
    __attribute__((aligned(16))) f16 e0s[Enc01::NREG * Enc01::LDE];
    __attribute__((aligned(16))) float b0[32], b1[64];
};

/* EVEN: the frame's width is even, so pixel pairs start at whole dwords. */
template <bool EVEN>
__device__ __forceinline__ void codec_enc01(const CodecArgs& a0, const CodecArgs& a1, Enc01Lds& L, int per_frame,
                                            int nblk) {
    using E = Enc01;
    f16* const s_in = L.s_in;
    f16* const e0s = L.e0s;
    const int lane = lane_id();
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int l16 = lane & 15, g = lane >> 4;
    const int W0 = a0.out_w, H0 = a0.out_h, W1 = a1.out_w, H1 = a1.out_h;
    const int bxn = (W1 + E::BC - 1) / E::BC;

    /* this thread's pixel pair of a window, every plane: one dword load each
     * (frames of odd width: two halves), zeros outside the frame */
    const int pr = (int)threadIdx.x / E::FP, pc = 2 * ((int)threadIdx.x - pr * E::FP);
    const bool pair = pr < E::FR;
    unsigned v[E::CH], vh[EVEN ? 1 : E::CH];
    auto load_window = [&](int f, int y1, int x1) {
        const __amdgpu_buffer_rsrc_t m =
            __builtin_amdgcn_make_buffer_rsrc((void*)(a0.in + (int64_t)f * a0.in_frame), (short)0, (int)(a0.in_frame * 2),
                                              0x00020000);
        const int gy = 2 * y1 - 2 + pr, gx = 2 * x1 - 2 + pc;
        const bool row = pair && gy >= 0 && gy < H0;
        const uint32_t at = (uint32_t)((gy * W0 + gx) * 2), plane = (uint32_t)(W0 * H0 * 2);
        const bool in0 = row && gx >= 0 && gx < W0, in1 = row && gx + 1 >= 0 && gx + 1 < W0;
        if constexpr (EVEN) { /* both pixels are in or out */
#pragma unroll
            for (int c = 0; c < E::CH; ++c)
                v[c] = __builtin_amdgcn_raw_buffer_load_b32(m, in0 ? at + c * plane : CODEC_OOB, 0, 0);
        } else {
#pragma unroll
            for (int c = 0; c < E::CH; ++c) {
                v[c] = __builtin_amdgcn_raw_buffer_load_b16(m, in0 ? at + c * plane : CODEC_OOB, 0, 0);
                vh[c] = __builtin_amdgcn_raw_buffer_load_b16(m, in1 ? at + c * plane + 2 : CODEC_OOB, 0, 0);
            }
        }
    };
    auto store_window = [&]() {
        if (!pair) return;
        if constexpr (!EVEN) {
#pragma unroll
            for (int c = 0; c < E::CH; ++c) v[c] = (v[c] & 0xffffu) | (vh[c] << 16);
        }
        unsigned p[10]; /* two pixels of ENC0_CP halfs */
#pragma unroll
        for (int c = 0; c + 1 < E::CH; c += 2) {
            p[c / 2] = (v[c] & 0xffffu) | (v[c + 1] << 16);
            p[5 + c / 2] = (v[c] >> 16) | (v[c + 1] & 0xffff0000u);
        }
        p[4] = v[8] & 0xffffu;
        p[9] = v[8] >> 16;
        u2* d = reinterpret_cast<u2*>(s_in + (pr * E::FC + pc) * E::CP);
#pragma unroll
        for (int k = 0; k < 5; ++k) d[k] = u2{p[2 * k], p[2 * k + 1]};
    };
    auto origin = [&](int i, int& f, int& y1, int& x1) {
        const int blk = codec_band(i, nblk);
        f = blk / per_frame;
        const int b = blk - f * per_frame, by = b / bxn;
        y1 = by * E::BR;
        x1 = (b - by * bxn) * E::BC;
    };

    int i = blockIdx.x, f, y1, x1;
    if (i >= nblk) return; /* the grid is rounded up to whole XCD turns */
    origin(i, f, y1, x1);
    load_window(f, y1, x1);
    const int rt = wave >> 1, ct = wave & 1; /* enc1: row tile, column tile */
    h8 wf0[2][E::KS0], wf1[E::KS1];
    {
        const FragSrc s0(a0.w, 2u * E::KS0 * 1024u), s1(a1.w, 4u * E::KS1 * 1024u);
#pragma unroll
        for (int ks = 0; ks < E::KS0; ++ks)
#pragma unroll
            for (int r = 0; r < 2; ++r) wf0[r][ks] = s0.load(r * E::KS0 + ks, lane * 16);
#pragma unroll
        for (int ks = 0; ks < E::KS1; ++ks) wf1[ks] = s1.load(rt * E::KS1 + ks, lane * 16);
        if (threadIdx.x < 32) L.b0[threadIdx.x] = a0.b[threadIdx.x];
        if (threadIdx.x < 64) L.b1[threadIdx.x] = a1.b[threadIdx.x];
    }
    /* e0 of 16 region pixels: window pixel at src, region pixel at dst, zeros
     * (enc1's padding) where it is not in the map */
    auto enc0_tile = [&](const f16* src, f16* dst, bool inmap, bool store) {
        f4 acc[2] = {*reinterpret_cast<const f4*>(L.b0 + 4 * g), *reinterpret_cast<const f4*>(L.b0 + 16 + 4 * g)};
#pragma unroll
        for (int ks = 0; ks < E::KS0; ++ks) {
            const h8 b = enc0_operand(src + ks * E::FC * E::CP, g);
            acc[0] = mfma_16x16x32(wf0[0][ks], b, acc[0]);
            acc[1] = mfma_16x16x32(wf0[1][ks], b, acc[1]);
        }
#pragma unroll
        for (int r = 0; r < 2; ++r) {
            const h4 hv = relu_h4(acc[r]);
            if (store) *reinterpret_cast<h4*>(dst + 16 * r) = inmap ? hv : h4{};
        }
    };
    /* enc0: 4 tiles of 16 columns a region row from column 1 on, this wave's
     * column tile w % 4 of rows w / 4, w / 4 + 2, ... */
    const int ec = 1 + 16 * (wave & 3) + l16, er0 = wave >> 2;
    const f16* const src0 = s_in + (er0 * E::FC + ec) * E::CP;
    f16* const dst0 = e0s + (er0 * E::EC + ec) * E::LDE + 4 * g;
    /* enc1: this lane's region pixel for tap (0, 0) of the first output row */
    const f16* const b1 = e0s + 2 * (16 * ct + l16) * E::LDE + 8 * g;

    while (true) { /* uniform over the workgroup */
        store_window();
        __syncthreads(); /* the window is in */
        const int cf = f, cy = y1, cx = x1;
        i += gridDim.x;
        const bool more = i < nblk;
        if (more) {
            origin(i, f, y1, x1);
            load_window(f, y1, x1);
        }
        /* ---- enc0 for the region */
        {
            const int ey0 = 2 * cy - 1; /* region row 0 */
            const bool xin = 2 * cx - 1 + ec < W0;
#pragma unroll
            for (int it = 0; it < 5; ++it) {
                if (it == 4 && er0) break; /* rows 1, 3, 5, 7 (uniform) */
                const int gy = ey0 + er0 + 2 * it;
                enc0_tile(src0 + 2 * it * E::FC * E::CP, dst0 + 2 * it * E::EC * E::LDE, xin && gy >= 0 && gy < H0, true);
            }
            if (wave == 4) { /* column 0, the halo: its 9 rows are one more tile */
                const int er = min(l16, E::ER - 1), gy = ey0 + er;
                enc0_tile(s_in + er * E::FC * E::CP, e0s + er * E::EC * E::LDE + 4 * g, cx > 0 && gy >= 0 && gy < H0,
                          l16 < E::ER);
            }
        }
        __syncthreads(); /* the region is complete; the window is dead */
        /* ---- the block's own e0 pixels (region rows and columns from 1 on) */
        uint16_t* e0map = a0.out + (int64_t)cf * a0.out_frame;
        codec_store_block<4 * E::NPX, 4, 512>(
            [&](int pl) { return e0s + ((1 + pl / (2 * E::BC)) * E::EC + 1 + pl % (2 * E::BC)) * E::LDE; }, [&](int pl) {
                const int Y = 2 * cy + pl / (2 * E::BC), X = 2 * cx + pl % (2 * E::BC);
                return Y < H0 && X < W0 ? e0map + ((int64_t)Y * W0 + X) * 32 : nullptr;
            });
        /* ---- enc1: region row rr is tap row ky = rr - 2y of output row y */
        {
            const f4 bias = *reinterpret_cast<const f4*>(L.b1 + 16 * rt + 4 * g);
            f4 acc[E::BR];
#pragma unroll
            for (int y = 0; y < E::BR; ++y) acc[y] = bias;
#pragma unroll
            for (int rr = 0; rr < E::ER; ++rr) {
#pragma unroll
                for (int kx = 0; kx < 3; ++kx) {
                    const h8 b = *reinterpret_cast<const h8*>(b1 + (rr * E::EC + kx) * E::LDE);
#pragma unroll
                    for (int y = 0; y < E::BR; ++y) {
                        const int ky = rr - 2 * y;
                        if (ky >= 0 && ky < 3) acc[y] = mfma_16x16x32(wf1[3 * ky + kx], b, acc[y]);
                    }
                }
            }
#pragma unroll
            for (int y = 0; y < E::BR; ++y)
                *reinterpret_cast<h4*>(L.e1 + (E::BC * y + 16 * ct + l16) * E::LDO + 16 * rt + 4 * g) = relu_h4(acc[y]);
        }
        __syncthreads();
        uint16_t* e1map = a1.out + (int64_t)cf * a1.out_frame;
        codec_store_block<E::NPX, 8, 512>([&](int pl) { return L.e1 + pl * E::LDO; }, [&](int pl) {
            const int Y = cy + pl / E::BC, X = cx + pl % E::BC;
            return Y < H1 && X < W1 ? e1map + ((int64_t)Y * W1 + X) * 64 : nullptr;
        });
        if (!more) break;
        __syncthreads(); /* the e1 tile is out */
    }
}

extern "C" __global__ void __launch_bounds__(512, 4) prism_codec_enc01(CodecArgs a0, CodecArgs a1, int per_frame,
                                                                       int nblk) {
    __shared__ Enc01Lds lds;
    if (a0.out_w & 1) /* uniform */
        codec_enc01<false>(a0, a1, lds, per_frame, nblk);
    else
        codec_enc01<true>(a0, a1, lds, per_frame, nblk);
}
/* enc2 and enc3: a stride-2 conv3x3 to 128 channels over an LDS window, 8
 * waves, wave w output row tile w. A block is BR x BC output pixels, TT tiles
 * of 16 (BC = 16: one row each, BC = 8: two rows); the input window under it,
 * (2 BR + 1) x (2 BC + 1) pixels of CIN channels (zeros past the map), is
 * copied into LDS and every wave reads its operands from there, one k-step (a
 * tap's 32 channels, k = tap * CIN + ic) ahead of the MFMAs, and its weight
 * fragments DW k-steps ahead: no input pixel or weight fragment is fetched by
 * more than one wave of the workgroup. The output tile leaves as whole pixels.
 * Persistent over one XCD's band of blocks; the next block's window is
 * requested before this block's end. 128 VGPRs, two workgroups fit a CU (enc2
 * launches one up to four blocks per CU: codec_enc2_slots). enc2 + enc3 at
 * 960x540 9.0 + 6.8 us, at 1920x1080 29 + 22 (one fused launch of 8
 * waves per CU, enc2 recomputing its halo: 19.6 and 80). Without the operand
 * reads enc3 would be 20 % faster, without its weights 7 %. Blocks of 8 x 8
 * for enc3 (half the weight bytes): 22 against 23.7 us at 1920x1080, 5 %
 * slower over four 960x540 frames; not kept.
 *
 * Window loads: thread t takes chunk t % TPR of the first 2 BC columns of
 * rows t / TPR, t / TPR + RPI, ..., so a row's bound check is uniform over
 * the wave and the addresses are one base and a stride; the last column is one
 * load more. */
template <int CIN, int BR, int BC>
struct ConvLds {
    static constexpr int WR = 2 * BR + 1, WC = 2 * BC + 1, LDW = CIN + 8, LDO = 128 + 8;
    __attribute__((aligned(16))) f16 win[WR * WC * LDW];
    __attribute__((aligned(16))) f16 tile[BR * BC * LDO];
    __attribute__((aligned(16))) float b[128];
};
template <int CIN, int BR, int BC, int DW>
__device__ __forceinline__ void codec_conv(const CodecArgs& a, ConvLds<CIN, BR, BC>& L, int per_frame, int nblk) {
    using C = ConvLds<CIN, BR, BC>;
    constexpr int CPT = CIN / 32, KS = 9 * CPT, COUT = 128, TT = BR * BC / 16, CPP = CIN / 8;
    constexpr int TPR = 2 * BC * CPP, RPI = 512 / TPR, IT = (C::WR + RPI - 1) / RPI;
    static_assert((BC == 16 || BC == 8) && BR * BC % 16 == 0, "whole token tiles");
    static_assert(512 % TPR == 0 && TPR % 64 == 0 && C::WR * CPP <= 512, "window loads");
    const int lane = lane_id();
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int l16 = lane & 15, g = lane >> 4;
    const int iw = a.in_w, ih = a.in_h, ow = a.out_w, oh = a.out_h;
    const int bxn = (ow + BC - 1) / BC;
    /* this thread's window chunk: row wr0 (uniform over the wave) + k RPI,
     * column wc; and its chunk of the last column (row lr) */
    const int wr0 = wave / (TPR / 64), tt = (int)threadIdx.x % TPR, wc = tt / CPP, c8 = (tt % CPP) * 8;
    const int lr = (int)threadIdx.x / CPP, l8 = ((int)threadIdx.x % CPP) * 8;
    h8 v[IT + 1];
    auto load_window = [&](int f, int y, int x) {
        const MapSrc m(a.in + (int64_t)f * a.in_frame, (uint32_t)(a.in_frame * 2));
        const int gy = 2 * y - 1 + wr0, gx = 2 * x - 1 + wc;
        const bool xin = gx >= 0 && gx < iw;
        const uint32_t at = (uint32_t)(((gy * iw + gx) * CIN + c8) * 2), step = (uint32_t)(RPI * iw * CIN * 2);
#pragma unroll
        for (int k = 0; k < IT; ++k) {
            const int yy = gy + k * RPI;
            const bool row = wr0 + k * RPI < C::WR && yy >= 0 && yy < ih; /* uniform */
            v[k] = m.load(row && xin ? at + k * step : CODEC_OOB);
        }
        const int ly = 2 * y - 1 + lr, lx = 2 * x - 1 + 2 * BC;
        const bool ok = lr < C::WR && ly >= 0 && ly < ih && lx < iw;
        v[IT] = m.load(ok ? (uint32_t)(((ly * iw + lx) * CIN + l8) * 2) : CODEC_OOB);
    };
    auto origin = [&](int i, int& f, int& y, int& x) {
        const int blk = codec_band(i, nblk);
        f = blk / per_frame;
        const int b = blk - f * per_frame, by = b / bxn;
        y = by * BR;
        x = (b - by * bxn) * BC;
    };
    int i = blockIdx.x, f, y, x;
    if (i >= nblk) return; /* the grid is rounded up to whole XCD turns */
    origin(i, f, y, x);
    load_window(f, y, x);
    const FragSrc wsrc(a.w, (unsigned)(COUT / 16 * KS * 1024));
    if (threadIdx.x < COUT) L.b[threadIdx.x] = a.b[threadIdx.x];
    /* this lane's window pixel for tap (0, 0) of tile 0 */
    const f16* const src =
        L.win + (BC == 16 ? 2 * l16 : 2 * (l16 >> 3) * C::WC + 2 * (l16 & 7)) * C::LDW + 8 * g;
    auto operand = [&](int ks, int t) {
        const int tap = ks / CPT, c = ks % CPT;
        return *reinterpret_cast<const h8*>(src + (((32 / BC) * t + tap / 3) * C::WC + tap % 3) * C::LDW + 32 * c);
    };
    while (true) { /* uniform over the workgroup */
        h8 w[DW];
#pragma unroll
        for (int ks = 0; ks < DW; ++ks) w[ks] = wsrc.load(wave * KS + ks, lane * 16);
#pragma unroll
        for (int k = 0; k < IT; ++k)
            if (wr0 + k * RPI < C::WR) /* uniform */
                *reinterpret_cast<h8*>(L.win + ((wr0 + k * RPI) * C::WC + wc) * C::LDW + c8) = v[k];
        if (lr < C::WR) *reinterpret_cast<h8*>(L.win + (lr * C::WC + 2 * BC) * C::LDW + l8) = v[IT];
        __syncthreads(); /* the window is in; the previous output tile is out */
        const int cf = f, cy = y, cx = x;
        i += gridDim.x;
        const bool more = i < nblk;
        const f4 bias = *reinterpret_cast<const f4*>(L.b + 16 * wave + 4 * g);
        f4 acc[TT];
        h8 bc[TT], bn[TT];
#pragma unroll
        for (int t = 0; t < TT; ++t) {
            acc[t] = bias;
            bc[t] = operand(0, t);
        }
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
            if (ks + 1 < KS) {
#pragma unroll
                for (int t = 0; t < TT; ++t) bn[t] = operand(ks + 1, t);
            }
#pragma unroll
            for (int t = 0; t < TT; ++t) acc[t] = mfma_16x16x32(w[ks % DW], bc[t], acc[t]);
            if (ks + DW < KS) w[ks % DW] = wsrc.load(wave * KS + ks + DW, lane * 16);
            if (ks + 1 < KS) {
#pragma unroll
                for (int t = 0; t < TT; ++t) bc[t] = bn[t];
            }
            /* the next window goes out behind the last fragments: loads
             * retire in order, so any fragment after it would wait for it */
            if (ks + DW == KS - 1 && more) {
                origin(i, f, y, x);
                load_window(f, y, x);
            }
            sched_fence();
        }
#pragma unroll
        for (int t = 0; t < TT; ++t)
            *reinterpret_cast<h4*>(L.tile + (16 * t + l16) * C::LDO + 16 * wave + 4 * g) = relu_h4(acc[t]);
        __syncthreads(); /* the output tile is complete; the window is dead */
        uint16_t* out = a.out + (int64_t)cf * a.out_frame;
        codec_store_block<BR * BC, COUT / 8, 512>([&](int p) { return L.tile + p * C::LDO; }, [&](int p) {
            const int Y = cy + p / BC, X = cx + p % BC;
            return Y < oh && X < ow ? out + ((int64_t)Y * ow + X) * COUT : nullptr;
        });
        if (!more) break;
    }
}

extern "C" __global__ void __launch_bounds__(512, 4) prism_codec_enc2(CodecArgs a, int per_frame, int nblk) {
    __shared__ ConvLds<64, CODEC_ENC2_ROWS, CODEC_ENC2_COLS> lds;
    codec_conv<64, CODEC_ENC2_ROWS, CODEC_ENC2_COLS, 4>(a, lds, per_frame, nblk);
}
extern "C" __global__ void __launch_bounds__(512, 4) prism_codec_enc3(CodecArgs a, int per_frame, int nblk) {
    __shared__ ConvLds<128, CODEC_ENC3_ROWS, CODEC_ENC3_COLS> lds;
    codec_conv<128, CODEC_ENC3_ROWS, CODEC_ENC3_COLS, 8>(a, lds, per_frame, nblk);
}
