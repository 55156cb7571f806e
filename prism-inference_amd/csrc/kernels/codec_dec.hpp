/*
 * codec_dec.hpp - the decoder's launches: dec3, and dec2 + dec1 + output conv
 * + PixelShuffle + sigmoid in one (stages and reference lines: codec.hpp).
 *
 * Every decoder stage is a pointwise conv over [NN-upsampled coarse map | skip
 * map], so the coarse channels' share of the sum is the same for the four
 * fine pixels (2y + dy, 2x + dx) over a coarse pixel: it is accumulated once
 * per coarse pixel (the bias first, then k ascending), and each fine pixel
 * continues from those accumulators with its skip channels. A token tile's
 * 16 columns are therefore 16 coarse pixels, or the same 16 pixels' (dy, dx)
 * children (a phase), so a lane's accumulators carry over without moving
 * between lanes. Same values in the same order as one pass over all k.
 *
 * What bounds them is memory (dec21_out at 1920x1080 moves 282 MB, dec3 75
 * MB), so the kernels are persistent: a wave holds its weight fragments in
 * registers for all of its workgroup's blocks (in the one-block form each
 * block streamed 124 KB of weights, more than its 35 KB of pixels, through
 * the CU's vector memory pipe), and the next block's pixels are requested
 * before this block's math. Input tiles pass through LDS in 16-byte chunks,
 * whole cache lines of the map per wave load. Against one block a workgroup:
 * dec21_out 86 -> 53 us (5.3 TB/s) and dec3 23.9 -> 16.5 at 1920x1080, both
 * together 26.9 -> 22.7 at 960x540.
 */
#pragma once
#include "codec.hpp"

/* Slot of a fine pixel (row dy, column 2c + dx of a 2 x 32 block) in an LDS
 * tile kept in phase order: a phase's 16 pixels are consecutive. */
__device__ __forceinline__ int dec_slot(int dy, int col) { return (2 * dy + (col & 1)) * 16 + (col >> 1); }

/* The 2 x 32 fine blocks of a map of w x h pixels, frame after frame. */
struct DecBlock {
    int f, y, x; /* frame, first fine row and column */
    __device__ __forceinline__ DecBlock(int blk, int w, int per_frame) {
        const int bxn = (w + 31) / 32;
        f = blk / per_frame;
        const int b = blk - f * per_frame;
        y = 2 * (b / bxn);
        x = 32 * (b - (b / bxn) * bxn);
    }
};

/* A thread's chunks of a block's input: CC 16-byte chunks of the 16 coarse
 * pixels (CUP channels), CS of the 64 skip pixels (CSKIP channels). */
template <int CUP, int CSKIP>
struct DecTile {
    static constexpr int NC = 16 * CUP / 8 / 256, NS = 64 * CSKIP / 8 / 256;
    static constexpr int LC = CUP + 8, LS = CSKIP + 8; /* LDS pixel strides (halfs) */
    static_assert(NC * 256 * 8 == 16 * CUP && NS * 256 * 8 == 64 * CSKIP, "whole chunks per thread");
    h8 c[NC], s[NS];
    /* requests the block's pixels; those past the map read zero */
    __device__ __forceinline__ void load(const CodecArgs& a, const DecBlock& b) {
        const MapSrc mc(a.in + (int64_t)b.f * a.in_frame, (uint32_t)(a.in_frame * 2));
        const MapSrc ms(a.skip + (int64_t)b.f * a.skip_frame, (uint32_t)(a.skip_frame * 2));
        const int cy = min(b.y >> 1, a.in_h - 1);
#pragma unroll
        for (int k = 0; k < NC; ++k) {
            const int q = threadIdx.x + 256 * k, p = q / (CUP / 8), c8 = (q % (CUP / 8)) * 8;
            const int cx = min((b.x >> 1) + p, a.in_w - 1);
            c[k] = mc.load((uint32_t)(((cy * a.in_w + cx) * CUP + c8) * 2));
        }
#pragma unroll
        for (int k = 0; k < NS; ++k) {
            const int q = threadIdx.x + 256 * k, p = q / (CSKIP / 8), c8 = (q % (CSKIP / 8)) * 8;
            const int y = b.y + (p >> 5), x = b.x + (p & 31);
            s[k] = ms.load(y < a.out_h && x < a.out_w ? (uint32_t)(((y * a.out_w + x) * CSKIP + c8) * 2) : CODEC_OOB);
        }
    }
    __device__ __forceinline__ void store(f16* lc, f16* ls) const {
#pragma unroll
        for (int k = 0; k < NC; ++k) {
            const int q = threadIdx.x + 256 * k;
            *reinterpret_cast<h8*>(lc + (q / (CUP / 8)) * LC + (q % (CUP / 8)) * 8) = c[k];
        }
#pragma unroll
        for (int k = 0; k < NS; ++k) {
            const int q = threadIdx.x + 256 * k, p = q / (CSKIP / 8);
            *reinterpret_cast<h8*>(ls + dec_slot(p >> 5, p & 31) * LS + (q % (CSKIP / 8)) * 8) = s[k];
        }
    }
};

/* RT row tiles of one stage over a block in LDS: out(phase, r, acc) receives
 * each phase's accumulators. w: the wave's fragments, k-step-major. */
template <int CUP, int CSKIP, int RT, class Out>
__device__ __forceinline__ void dec_gemm(const h8 (&w)[RT][(CUP + CSKIP) / 32], const f4 (&bias)[RT], const f16* lc,
                                         const f16* ls, int l16, int g, Out&& out) {
    using T = DecTile<CUP, CSKIP>;
    constexpr int KC = CUP / 32, KF = CSKIP / 32;
    f4 cacc[RT];
#pragma unroll
    for (int r = 0; r < RT; ++r) cacc[r] = bias[r];
#pragma unroll
    for (int ks = 0; ks < KC; ++ks) {
        const h8 b = *reinterpret_cast<const h8*>(lc + l16 * T::LC + 32 * ks + 8 * g);
#pragma unroll
        for (int r = 0; r < RT; ++r) cacc[r] = mfma_16x16x32(w[r][ks], b, cacc[r]);
    }
#pragma unroll
    for (int p = 0; p < 4; ++p) {
        f4 acc[RT];
#pragma unroll
        for (int r = 0; r < RT; ++r) acc[r] = cacc[r];
#pragma unroll
        for (int ks = 0; ks < KF; ++ks) {
            const h8 b = *reinterpret_cast<const h8*>(ls + (16 * p + l16) * T::LS + 32 * ks + 8 * g);
#pragma unroll
            for (int r = 0; r < RT; ++r) acc[r] = mfma_16x16x32(w[r][KC + ks], b, acc[r]);
        }
        out(p, acc);
    }
}

template <int RT, int KS>
__device__ __forceinline__ void dec_weights(const uint16_t* w, const float* b, int rt0, int rows, int lane, int g,
                                            h8 (&wf)[RT][KS], f4 (&bias)[RT]) {
    const FragSrc src(w, (unsigned)(rows / 16 * KS * 1024));
#pragma unroll
    for (int r = 0; r < RT; ++r) {
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) wf[r][ks] = src.load((rt0 + r) * KS + ks, lane * 16);
        const int ch = 16 * (rt0 + r) + 4 * g;
        bias[r] = f4{b[ch], b[ch + 1], b[ch + 2], b[ch + 3]};
    }
}

/* dec3 (128 + 128 -> 128), 2 x 32 blocks of the r2 map: wave w computes row
 * tiles 2w and 2w + 1 of every pixel; the output tile leaves as whole pixels,
 * 16 bytes per lane. Workgroup b takes blocks b, b + gridDim.x, ... of nblk. */
__device__ __forceinline__ void codec_dec3(const CodecArgs& a, int per_frame, int nblk) {
    using T = DecTile<128, 128>;
    constexpr int C = 128, LO = C + 8;
    __shared__ __attribute__((aligned(16))) f16 lc[16 * T::LC], ls[64 * T::LS], lo[64 * LO];
    const int lane = lane_id();
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int l16 = lane & 15, g = lane >> 4;
    int blk = blockIdx.x;
    T t;
    DecBlock b(blk, a.out_w, per_frame);
    t.load(a, b);
    h8 w[2][8];
    f4 bias[2];
    dec_weights<2, 8>(a.w, a.b, 2 * wave, C, lane, g, w, bias);
    for (; blk < nblk; blk += gridDim.x) { /* uniform over the workgroup */
        t.store(lc, ls);
        __syncthreads(); /* the block is in; the previous one's output is out of lo */
        const DecBlock cur = b;
        if (blk + (int)gridDim.x < nblk) {
            b = DecBlock(blk + gridDim.x, a.out_w, per_frame);
            t.load(a, b);
        }
        dec_gemm<128, 128, 2>(w, bias, lc, ls, l16, g, [&](int p, const f4(&acc)[2]) {
#pragma unroll
            for (int r = 0; r < 2; ++r)
                *reinterpret_cast<h4*>(lo + (16 * p + l16) * LO + 16 * (2 * wave + r) + 4 * g) = relu_h4(acc[r]);
        });
        __syncthreads();
        uint16_t* out = a.out + (int64_t)cur.f * a.out_frame;
        codec_store_block<64, C / 8, 256>([&](int p) { return lo + dec_slot(p >> 5, p & 31) * LO; }, [&](int p) {
            const int y = cur.y + (p >> 5), x = cur.x + (p & 31);
            return y < a.out_h && x < a.out_w ? out + ((int64_t)y * a.out_w + x) * C : nullptr;
        });
    }
}

/* dec2 + dec1 + output conv + PixelShuffle(2) + sigmoid, 2 x 32 blocks of the
 * r1 map with the 4 x 64 r0 pixels over each: dec2's wave w computes row tile
 * w for the block's 64 pixels into LDS, then dec1's wave w takes 16 of those
 * pixels (row w / 2, columns 16 (w % 2)..+15) and their 64 r0 children, the
 * e0 skip channels straight from memory to the lane (its B fragment). The
 * dec2 map never reaches memory. The two children side by side are four
 * display pixels of a row, one 8-byte store. a2: dec2's arguments (out
 * unused), a1: dec1's (in unused). */
__device__ __forceinline__ void codec_dec21(const CodecArgs& a2, const CodecArgs& a1, int per_frame, int nblk) {
    using T = DecTile<128, 64>;
    constexpr int LD = 64 + 8;
    constexpr float LOG2E = 1.4426950408889634f;
    __shared__ __attribute__((aligned(16))) f16 lc[16 * T::LC], ls[64 * T::LS], d2s[64 * LD];
    const int lane = lane_id();
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int l16 = lane & 15, g = lane >> 4;
    const int w0 = a1.out_w, h0 = a1.out_h;
    /* this lane's r1 pixel within a block, and its dec2 output in LDS */
    const int dy = wave >> 1, col = 16 * (wave & 1) + l16;
    const f16* up = d2s + dec_slot(dy, col) * LD + 8 * g;
    /* the skip channels of its four r0 children (2 ey + ex) */
    auto load_e0 = [&](const DecBlock& b, h8(&e)[4]) {
        const MapSrc m(a1.skip + (int64_t)b.f * a1.skip_frame, (uint32_t)(a1.skip_frame * 2));
        const int y = 2 * (b.y + dy), x = 2 * (b.x + col);
#pragma unroll
        for (int p = 0; p < 4; ++p) {
            const int yy = y + (p >> 1), xx = x + (p & 1);
            e[p] = m.load(yy < h0 && xx < w0 ? (uint32_t)(((yy * w0 + xx) * 32 + 8 * g) * 2) : CODEC_OOB);
        }
    };
    int blk = blockIdx.x;
    T t;
    h8 e0[4];
    DecBlock b(blk, a2.out_w, per_frame);
    t.load(a2, b);
    load_e0(b, e0);
    h8 wa[1][6], wb[2][3];
    f4 ba[1], bb[2];
    dec_weights<1, 6>(a2.w, a2.b, wave, 64, lane, g, wa, ba);
    dec_weights<2, 3>(a1.w, a1.b, 0, 32, lane, g, wb, bb);
    /* the 32 -> 12 weights: one fragment (rows 12..15 zero), columns permuted */
    const h8 wo = FragSrc(a1.w2, 1024u).load(0, lane * 16);
    const f4 bo = {a1.b2[4 * g], a1.b2[4 * g + 1], a1.b2[4 * g + 2], a1.b2[4 * g + 3]};
    const int dw = 2 * w0, dh = 2 * h0;
    for (; blk < nblk; blk += gridDim.x) { /* uniform over the workgroup */
        t.store(lc, ls);
        __syncthreads(); /* the block is in; every wave is done with the previous dec2 tile */
        const DecBlock cur = b;
        h8 e[4];
#pragma unroll
        for (int p = 0; p < 4; ++p) e[p] = e0[p];
        if (blk + (int)gridDim.x < nblk) {
            b = DecBlock(blk + gridDim.x, a2.out_w, per_frame);
            t.load(a2, b);
            load_e0(b, e0);
        }
        dec_gemm<128, 64, 1>(wa, ba, lc, ls, l16, g, [&](int p, const f4(&acc)[1]) {
            *reinterpret_cast<h4*>(d2s + (16 * p + l16) * LD + 16 * wave + 4 * g) = relu_h4(acc[0]);
        });
        __syncthreads();
        f4 cacc[2] = {bb[0], bb[1]};
#pragma unroll
        for (int ks = 0; ks < 2; ++ks) {
            const h8 u = *reinterpret_cast<const h8*>(up + 32 * ks);
#pragma unroll
            for (int r = 0; r < 2; ++r) cacc[r] = mfma_16x16x32(wb[r][ks], u, cacc[r]);
        }
        const int y0 = 2 * (cur.y + dy), x0 = 2 * (cur.x + col);
        uint16_t* disp = a1.out + (int64_t)cur.f * a1.out_frame;
#pragma unroll
        for (int ey = 0; ey < 2; ++ey) {
            h4 s[2]; /* the sigmoids of the two children's channels 4g..4g+3 */
#pragma unroll
            for (int ex = 0; ex < 2; ++ex) {
                h4 y[2];
#pragma unroll
                for (int r = 0; r < 2; ++r) y[r] = relu_h4(mfma_16x16x32(wb[r][2], e[2 * ey + ex], cacc[r]));
                const h8 yb = {y[0][0], y[0][1], y[0][2], y[0][3], y[1][0], y[1][1], y[1][2], y[1][3]};
                const h4 o12 = cvt_h4(mfma_16x16x32(wo, yb, bo));
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    s[ex][i] = (_Float16)fast_rcp(1.0f + fast_exp2(-(float)o12[i] * LOG2E));
            }
            if (g == 3 || y0 + ey >= h0 || x0 >= w0) continue; /* rows 12..15 are padding */
            /* channel 4g + 2sy + sx -> RGB plane g, display pixel (2y + sy, 2x + sx) */
#pragma unroll
            for (int sy = 0; sy < 2; ++sy) {
                uint16_t* row = disp + ((int64_t)g * dh + 2 * (y0 + ey) + sy) * dw + 2 * x0;
                const h4 px = {s[0][2 * sy], s[0][2 * sy + 1], s[1][2 * sy], s[1][2 * sy + 1]};
                if (x0 + 1 < w0) {
                    /* 8 bytes at a 4-byte boundary (a frame of odd width) */
                    typedef h4 h4_a4 __attribute__((aligned(4)));
                    *reinterpret_cast<h4_a4*>(row) = px;
                } else {
                    *reinterpret_cast<h2*>(row) = h2{px[0], px[1]};
                }
            }
        }
    }
}

extern "C" __global__ void __launch_bounds__(256, 3) prism_codec_dec3(CodecArgs a, int per_frame, int nblk) {
    codec_dec3(a, per_frame, nblk);
}
extern "C" __global__ void __launch_bounds__(256, 3) prism_codec_dec21_out(CodecArgs a2, CodecArgs a1, int per_frame,
                                                                           int nblk) {
    codec_dec21(a2, a1, per_frame, nblk);
}
