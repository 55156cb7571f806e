/*
 * codec.hpp - the conv encoder and fused decoder around the transformer
 * (the end-to-end frame of vulkan_engine/prism_moe_bench.cpp:387-471).
 *
 * Every stage is one implicit GEMM on fp16 MFMA, C^T = W * P^T: the packed
 * weights are the A operand (16 output channels x 32 k per fragment) and the
 * B operand is gathered per lane straight from the input maps, 16 output
 * pixels per token tile. Accumulators start at the bias; the result is
 * rounded to fp16 once (the reference rounds each 288-wide split partial
 * sum, strided_conv_split_*ch.comp.glsl:84-93, which its comments call the
 * same output), then ReLU. Maps between stages are NHWC fp16 (a pixel's
 * channels contiguous, so a lane's 8 channels are one 16-byte load); the
 * frame coming in and the display image going out are CHW, as in the
 * reference.
 *
 *   enc0  conv3x3 s1  9 -> 32  + ReLU  conv3x3_coopvec_9ch.comp.glsl:27-72
 *         (reads the CHW frame through an LDS window per 4 x 64 pixel block)
 *   enc1  conv3x3 s2 32 -> 64  + ReLU  strided_conv_coopvec_32ch.comp.glsl:30-77
 *   enc2  conv3x3 s2 64 -> 128 + ReLU  strided_conv_split_64ch.comp.glsl:30-93
 *   enc3  conv3x3 s2 128-> 128 + ReLU  strided_conv_split_128ch.comp.glsl:32-94
 *         (NHWC taps: k = tap*Cin + ic; the host permutes the weight columns)
 *   dec3  NN-up(128) ++ skip e2(128) -> PW 256 -> 128 + ReLU   dec3_fused.comp.glsl:27-63
 *   dec2  NN-up(128) ++ skip e1(64)  -> PW 192 -> 64  + ReLU   dec2_fused.comp.glsl:27-55
 *   dec1  NN-up(64)  ++ skip e0(32)  -> PW 96  -> 32  + ReLU   dec1_fused.comp.glsl:27-55
 *         then PW 32 -> 12 (pw_conv_coopvec_32to12.comp.glsl:28-55) and
 *         PixelShuffle(2) + sigmoid (pixelshuffle_sigmoid.comp.glsl:28-56)
 *         in the same kernel: dec1's accumulator lanes hold channels
 *         4g..4g+3 and 16+4g..16+4g+3 of their pixel, which is a B fragment
 *         of the 32 -> 12 GEMM under the permuted k numbering
 *         k(g, j) = 16*(j/4) + 4g + j%4 (the host packs that weight with its
 *         columns permuted to match). The 12 channels round to fp16 (the
 *         reference's out12 map), then sigmoid in fp32, fp16 again, written
 *         as 2x2 display pixels of the lane's RGB plane.
 *
 * enc1, dec2 and dec1_out as stages: workgroup = 4 waves; a wave takes TT
 * consecutive 16-pixel tiles (pixels in row-major order of the output map,
 * blockIdx.y = frame) and all COUT output channels. Each k-step's weight
 * fragments and B fragments are loaded one k-step ahead of its MFMAs. Loads
 * at padded or out-of-map positions return zeros through the input buffer's
 * range check (MapSrc). enc2, enc3 and the fused enc0 + enc1: codec_enc.hpp;
 * dec3 and the fused dec2 + dec1 + output: codec_dec.hpp.
 */
#pragma once
#include "common.hpp"

/* Output pixel of one lane in one token tile. */
struct CodecPix {
    int y, x;
    bool valid;
};

/* The B gathers read a frame's map through a buffer resource whose range is
 * the map: a lane whose operand is zero (a tap in the conv padding) or
 * unused (a pixel past the map's end, whose output column is never stored)
 * gets the offset CODEC_OOB, and the range check returns zeros for it. Each
 * lane's byte offsets are 32-bit (the host keeps a frame's largest map under
 * 2 GiB) and computed once per token tile, so a load is one instruction with
 * its k-step's channel offset in the immediate field. */
static constexpr uint32_t CODEC_OOB = 0x80000000u;
struct MapSrc {
    __amdgpu_buffer_rsrc_t r;
    __device__ __forceinline__ MapSrc(const uint16_t* base, uint32_t bytes)
        : r(__builtin_amdgcn_make_buffer_rsrc((void*)base, (short)0, (int)bytes, 0x00020000)) {}
    __device__ __forceinline__ h8 load(uint32_t off) const {
        return __builtin_bit_cast(h8, __builtin_amdgcn_raw_buffer_load_b128(r, off, 0, 0));
    }
};

/* conv3x3 (pad 1) over an NHWC map with CIN channels; k = tap*CIN + ic. A
 * tile's per-lane state: the byte offset of each of the 9 taps' input pixel
 * (channel 8g), CODEC_OOB where the tap falls in the padding. */
template <int CIN, int STRIDE>
struct SrcConvNHWC {
    static constexpr int KS = 9 * CIN / 32;
    MapSrc m;
    int iw, ih;
    struct Pix {
        uint32_t off[9];
    };
    __device__ __forceinline__ Pix prep(const CodecPix& p, int g) const {
        Pix q;
        const int iy0 = p.y * STRIDE - 1, ix0 = p.x * STRIDE - 1;
        const int base = ((iy0 * iw + ix0) * CIN + 8 * g) * 2; /* may be negative: only in-map taps use it */
#pragma unroll
        for (int tap = 0; tap < 9; ++tap) {
            const int iy = iy0 + tap / 3, ix = ix0 + tap % 3;
            const bool ok = p.valid && iy >= 0 && iy < ih && ix >= 0 && ix < iw;
            q.off[tap] = ok ? (uint32_t)(base + ((tap / 3) * iw + tap % 3) * CIN * 2) : CODEC_OOB;
        }
        return q;
    }
    __device__ __forceinline__ h8 load(int ks, const Pix& q) const { /* ks compile-time */
        constexpr int CPT = CIN / 32; /* k-steps per tap */
        return m.load(q.off[ks / CPT] + (uint32_t)(ks % CPT * 64));
    }
};

/* Decoder input: channels [0, CUP) from the NN-upsampled coarse map (pixel
 * (min(y/2, uh-1), min(x/2, uw-1))), then [CUP, CUP+CSKIP) from the skip map
 * at the same pixel. */
template <int CUP, int CSKIP>
struct SrcDec {
    static constexpr int KS = (CUP + CSKIP) / 32;
    MapSrc mu, ms;
    int uw, uh, ow;
    struct Pix {
        uint32_t up, skip;
    };
    __device__ __forceinline__ Pix prep(const CodecPix& p, int g) const {
        const int uy = min(p.y >> 1, uh - 1), ux = min(p.x >> 1, uw - 1);
        return Pix{p.valid ? (uint32_t)(((uy * uw + ux) * CUP + 8 * g) * 2) : CODEC_OOB,
                   p.valid ? (uint32_t)(((p.y * ow + p.x) * CSKIP + 8 * g) * 2) : CODEC_OOB};
    }
    __device__ __forceinline__ h8 load(int ks, const Pix& q) const { /* ks compile-time */
        if (32 * ks < CUP) return mu.load(q.up + (uint32_t)(64 * ks));
        return ms.load(q.skip + (uint32_t)(64 * ks - 2 * CUP));
    }
};

/* The GEMM: acc[r][t] = bias + W[16 r.., :] * P[:, tile t] for the matrix's RT
 * row tiles. */
template <class Src, int RT, int TT>
__device__ __forceinline__ void codec_gemm(const Src& src, const uint16_t* w, const float* bias, const CodecPix (&px)[TT],
                                           int g, int lane, f4 (&acc)[RT][TT]) {
    constexpr int KS = Src::KS;
    const FragSrc wsrc(w, (unsigned)(RT * KS * 1024));
#pragma unroll
    for (int r = 0; r < RT; ++r) {
        const int ch = 16 * r + 4 * g;
        const f4 bb = {bias[ch], bias[ch + 1], bias[ch + 2], bias[ch + 3]};
#pragma unroll
        for (int t = 0; t < TT; ++t) acc[r][t] = bb;
    }
    typename Src::Pix q[TT];
#pragma unroll
    for (int t = 0; t < TT; ++t) q[t] = src.prep(px[t], g);
    h8 bc[TT], bn[TT], wc[RT], wn[RT];
#pragma unroll
    for (int t = 0; t < TT; ++t) bc[t] = src.load(0, q[t]);
#pragma unroll
    for (int r = 0; r < RT; ++r) wc[r] = wsrc.load(r * KS, lane * 16);
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
        if (ks + 1 < KS) {
#pragma unroll
            for (int t = 0; t < TT; ++t) bn[t] = src.load(ks + 1, q[t]);
#pragma unroll
            for (int r = 0; r < RT; ++r) wn[r] = wsrc.load(r * KS + ks + 1, lane * 16);
        }
#pragma unroll
        for (int r = 0; r < RT; ++r)
#pragma unroll
            for (int t = 0; t < TT; ++t) acc[r][t] = mfma_16x16x32(wc[r], bc[t], acc[r][t]);
        if (ks + 1 < KS) {
#pragma unroll
            for (int t = 0; t < TT; ++t) bc[t] = bn[t];
#pragma unroll
            for (int r = 0; r < RT; ++r) wc[r] = wn[r];
        }
        sched_fence();
    }
}

/* The pixel block a workgroup takes: workgroups are dealt to the 8 XCDs in
 * turn (workgroup b to XCD b % 8), each with its own L2, so consecutive
 * blocks (which share input rows: the conv taps' halo, the stride-2 rows
 * between two output rows, the decoder's upsampled rows) go to the same XCD
 * in a contiguous band of about 1/8 of the n blocks: the first n % 8 XCDs take
 * n/8 + 1 blocks, the others n/8 (a permutation of [0, n), whatever the
 * hardware's actual placement). BAND = false keeps the launch order (dec1_out
 * runs 0.4 us faster with every XCD sweeping the map top to bottom together;
 * enc0, enc1, dec2 1.7, 1.6, 0.2 us faster banded at 960x540). */
__device__ __forceinline__ int codec_band(int i, int n) {
    const int q = n >> 3, r = n & 7, x = i & 7, j = i >> 3;
    return x < r ? x * (q + 1) + j : r * (q + 1) + (x - r) * q + j;
}
template <bool BAND>
__device__ __forceinline__ int codec_block() {
    if constexpr (!BAND) return (int)blockIdx.x;
    return codec_band((int)blockIdx.x, (int)gridDim.x);
}

/* A workgroup's output block from LDS to memory in 16-byte chunks (NPX
 * pixels of CPP chunks, NT threads). Every LDS read is issued before the
 * first store: a read under a store's condition costs one LDS round trip per
 * pass. src(pl): the LDS address of block pixel pl's first channel; dst(pl):
 * the memory address of its first channel, or nullptr past the map. */
template <int NPX, int CPP, int NT, class Src, class Dst>
__device__ __forceinline__ void codec_store_block(Src&& src, Dst&& dst) {
    constexpr int N = NPX * CPP, IT = (N + NT - 1) / NT;
    h8 v[IT];
#pragma unroll
    for (int it = 0; it < IT; ++it) {
        const int q = min((int)threadIdx.x + NT * it, N - 1);
        v[it] = *reinterpret_cast<const h8*>(src(q / CPP) + (q % CPP) * 8);
    }
#pragma unroll
    for (int it = 0; it < IT; ++it) {
        const int q = (int)threadIdx.x + NT * it;
        if (q < N) {
            uint16_t* d = dst(q / CPP);
            if (d) *reinterpret_cast<h8*>(d + (q % CPP) * 8) = v[it];
        }
    }
}

/* A workgroup's 4 waves take TT consecutive 16-pixel tiles each. */
template <int TT, bool BAND>
__device__ __forceinline__ void codec_pixels(const CodecArgs& a, int wave, int l16, CodecPix (&px)[TT]) {
    const int npix = a.out_w * a.out_h;
    const int p0 = (codec_block<BAND>() * 4 + wave) * TT * 16;
#pragma unroll
    for (int t = 0; t < TT; ++t) {
        const int p = p0 + 16 * t + l16;
        px[t].valid = p < npix;
        const int q = px[t].valid ? p : 0;
        px[t].y = q / a.out_w;
        px[t].x = q - px[t].y * a.out_w;
    }
}

/* One stage: GEMM, ReLU, fp16, NHWC store. The workgroup's pixels are
 * consecutive, so its output is one contiguous block: the tile is assembled
 * in LDS and leaves as whole pixel rows, 16 bytes per lane (a store straight
 * from the accumulators writes 16 pixels x 32 bytes per instruction). */
template <class Src, int COUT, int TT, bool BAND>
__device__ __forceinline__ void codec_stage(const CodecArgs& a, const Src& src) {
    constexpr int RT = COUT / 16;
    static_assert(COUT % 16 == 0, "whole row tiles");
    constexpr int NPX = 4 * TT * 16, LDO = COUT + 8; /* pixels per workgroup, padded LDS row */
    __shared__ __attribute__((aligned(16))) f16 otile[NPX * LDO];
    const int lane = lane_id();
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int l16 = lane & 15, g = lane >> 4;
    CodecPix px[TT];
    codec_pixels<TT, BAND>(a, wave, l16, px);
    f4 acc[RT][TT];
    codec_gemm<Src, RT, TT>(src, a.w, a.b, px, g, lane, acc);
    const int pl0 = wave * TT * 16; /* this wave's first pixel in the workgroup's block */
#pragma unroll
    for (int t = 0; t < TT; ++t)
#pragma unroll
        for (int r = 0; r < RT; ++r)
            *reinterpret_cast<h4*>(otile + (pl0 + 16 * t + l16) * LDO + 16 * r + 4 * g) = relu_h4(acc[r][t]);
    __syncthreads();
    const int64_t p0 = (int64_t)codec_block<BAND>() * NPX, npix = (int64_t)a.out_w * a.out_h;
    uint16_t* out = a.out + (int64_t)blockIdx.y * a.out_frame;
    codec_store_block<NPX, COUT / 8, 256>([&](int pl) { return otile + pl * LDO; },
                                          [&](int pl) { return p0 + pl < npix ? out + (p0 + pl) * COUT : nullptr; });
}

/* dec1's output tiles (acc: its 32 channels, bias in) -> ReLU, fp16, the
 * 32 -> 12 conv, fp16, sigmoid, fp16, PixelShuffle(2) into the CHW display. */
template <int TT>
__device__ __forceinline__ void codec_out_shuffle(const CodecArgs& a, const CodecPix (&px)[TT], const f4 (&acc)[2][TT],
                                                  int g, int lane) {
    const int f = blockIdx.y;
    /* the 32 -> 12 weights: one fragment (rows 12..15 zero), columns permuted */
    const h8 wo = FragSrc(a.w2, 1024u).load(0, lane * 16);
    const f4 bo = {a.b2[4 * g], a.b2[4 * g + 1], a.b2[4 * g + 2], a.b2[4 * g + 3]};
    constexpr float LOG2E = 1.4426950408889634f;
    const int dw = 2 * a.out_w, dh = 2 * a.out_h;
    uint16_t* disp = a.out + (int64_t)f * a.out_frame;
#pragma unroll
    for (int t = 0; t < TT; ++t) {
        h4 y[2];
#pragma unroll
        for (int r = 0; r < 2; ++r) y[r] = relu_h4(acc[r][t]); /* dec1 output, r16 + ReLU */
        const h8 yb = {y[0][0], y[0][1], y[0][2], y[0][3], y[1][0], y[1][1], y[1][2], y[1][3]};
        const h4 o12 = cvt_h4(mfma_16x16x32(wo, yb, bo)); /* out12 channels 4g..4g+3 */
        if (!px[t].valid || g == 3) continue;             /* rows 12..15 are padding */
        h4 s;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const float v = (float)o12[i];
            s[i] = (_Float16)fast_rcp(1.0f + fast_exp2(-v * LOG2E));
        }
        /* channel 4g + 2sy + sx -> RGB plane g, display pixel (2y + sy, 2x + sx) */
        uint16_t* base = disp + ((int64_t)g * dh + 2 * px[t].y) * dw + 2 * px[t].x;
        const uint32_t top = __builtin_bit_cast(uint32_t, __builtin_shufflevector(s, s, 0, 1));
        const uint32_t bot = __builtin_bit_cast(uint32_t, __builtin_shufflevector(s, s, 2, 3));
        *reinterpret_cast<uint32_t*>(base) = top;
        *reinterpret_cast<uint32_t*>(base + dw) = bot;
    }
}

/* dec1 + output conv + PixelShuffle(2) + sigmoid. */
template <int TT>
__device__ __forceinline__ void codec_dec_out(const CodecArgs& a) {
    const int lane = lane_id();
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int l16 = lane & 15, g = lane >> 4;
    CodecPix px[TT];
    codec_pixels<TT, false>(a, wave, l16, px);
    const int f = blockIdx.y;
    const SrcDec<64, 32> src{MapSrc(a.in + (int64_t)f * a.in_frame, (uint32_t)(a.in_frame * 2)),
                             MapSrc(a.skip + (int64_t)f * a.skip_frame, (uint32_t)(a.skip_frame * 2)), a.in_w, a.in_h,
                             a.out_w};
    f4 acc[2][TT];
    codec_gemm<SrcDec<64, 32>, 2, TT>(src, a.w, a.b, px, g, lane, acc);
    codec_out_shuffle<TT>(a, px, acc, g, lane);
}

/* enc0's operands. A frame window sits in LDS pixel-interleaved, ENC0_CP = 10
 * halfs a pixel (the 9 channels and a zero), so the 3 taps of a kernel row are
 * 30 consecutive halfs of a window row: one k-step. The reduction index is
 * k = 32 ky + 10 kx + ic, 3 k-steps (the host packs W's stored column ic * 9 +
 * tap there, zeros elsewhere). The odd dword stride (5) keeps the reads of 16
 * consecutive pixels free of bank conflicts. (9 taps x 16 halfs a pixel, 5
 * k-steps, read 1.7 times the LDS bytes, which bound the fused launch; the
 * sums of the two differ in their last bits, their error against 64 bits does
 * not: 3.9e-4 over the encoder.) */
static constexpr int ENC0_CP = 10, ENC0_KS = 3;
typedef unsigned u4 __attribute__((ext_vector_type(4)));
typedef unsigned u2 __attribute__((ext_vector_type(2)));

/* B fragment of kernel row ky for the pixel whose tap (0, 0) is at `src`: 8
 * halfs from 8 g of the row's 30; the last two of lane group 3 belong to the
 * next pixel and are made zero (their weights are, but the pixel may hold a
 * NaN). */
__device__ __forceinline__ h8 enc0_operand(const f16* src, int g) {
    const unsigned* p = reinterpret_cast<const unsigned*>(src + 8 * g);
    u4 v = {p[0], p[1], p[2], p[3]};
    v[3] = g == 3 ? 0u : v[3];
    return __builtin_bit_cast(h8, v);
}

/* The frame window under a block: FR x FC pixels of the 9-channel CHW frame
 * from pixel (gy0, gx0), into LDS as ENC0_CP halfs a pixel (zeros where the
 * window leaves the frame), by 256 threads. Every load of a
 * thread is issued before its first LDS store, so the window costs one memory
 * round trip; a load for a pixel outside the frame reads pixel 0, and its
 * value is replaced by zero. */
template <int FR, int FC>
__device__ __forceinline__ void codec_frame_window(const f16* frame, int W0, int H0, int gy0, int gx0, f16* s_in) {
    constexpr int NPX = FR * FC, IT = (NPX + 255) / 256, CH = 9;
    const int64_t plane = (int64_t)W0 * H0;
    f16 v[IT][CH];
    bool ok[IT];
#pragma unroll
    for (int it = 0; it < IT; ++it) {
        const int px = min((int)threadIdx.x + 256 * it, NPX - 1);
        const int r = px / FC, x = px - r * FC;
        const int gy = gy0 + r, gx = gx0 + x;
        ok[it] = gy >= 0 && gy < H0 && gx >= 0 && gx < W0;
        const f16* src = frame + (ok[it] ? (int64_t)gy * W0 + gx : 0);
#pragma unroll
        for (int c = 0; c < CH; ++c) v[it][c] = src[c * plane];
    }
#pragma unroll
    for (int it = 0; it < IT; ++it) {
        const int px = threadIdx.x + 256 * it;
        if (px < NPX) {
            h2* d = reinterpret_cast<h2*>(s_in + px * ENC0_CP);
#pragma unroll
            for (int c = 0; c < CH; c += 2)
                d[c / 2] = ok[it] ? h2{v[it][c], c + 1 < CH ? v[it][c + 1 < CH ? c + 1 : c] : (f16)0.f} : h2{};
        }
    }
}

/* enc0: conv3x3 9 -> 32 + ReLU straight from the CHW frame. A workgroup
 * takes a block of CODEC_ENC0_ROWS x 64 output pixels (wave w: row w, 4 tiles
 * of 16 columns). The block's input window with its 1-pixel halo is first
 * copied into LDS (codec_frame_window, one thread per pixel). Grid: x =
 * ceil(W/CODEC_ENC0_COLS) * ceil(H/CODEC_ENC0_ROWS), y = frames. */
__device__ __forceinline__ void codec_enc0_body(const CodecArgs& a) {
    constexpr int IR = CODEC_ENC0_ROWS + 2, IC = CODEC_ENC0_COLS + 2, CP = ENC0_CP, KS = ENC0_KS,
                  TT = CODEC_ENC0_COLS / 16;
    __shared__ __attribute__((aligned(16))) f16 s_in[IR * IC * CP + 8]; /* + the last operand's two spare halfs */
    const int lane = lane_id();
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int l16 = lane & 15, g = lane >> 4;
    const int W = a.out_w, H = a.out_h;
    const int bxn = (W + CODEC_ENC0_COLS - 1) / CODEC_ENC0_COLS;
    const int blk = codec_block<true>();
    const int by0 = (blk / bxn) * CODEC_ENC0_ROWS, bx0 = (blk % bxn) * CODEC_ENC0_COLS;
    codec_frame_window<IR, IC>(reinterpret_cast<const f16*>(a.in) + (int64_t)blockIdx.y * a.in_frame, W, H, by0 - 1,
                               bx0 - 1, s_in);
    __syncthreads();
    const FragSrc wsrc(a.w, 2u * KS * 1024u);
    f4 acc[2][TT];
#pragma unroll
    for (int r = 0; r < 2; ++r) {
        const int ch = 16 * r + 4 * g;
        const f4 bb = {a.b[ch], a.b[ch + 1], a.b[ch + 2], a.b[ch + 3]};
#pragma unroll
        for (int t = 0; t < TT; ++t) acc[r][t] = bb;
    }
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
        const h8 w0 = wsrc.load(0 * KS + ks, lane * 16), w1 = wsrc.load(1 * KS + ks, lane * 16);
#pragma unroll
        for (int t = 0; t < TT; ++t) {
            const h8 b = enc0_operand(s_in + ((wave + ks) * IC + 16 * t + l16) * CP, g);
            acc[0][t] = mfma_16x16x32(w0, b, acc[0][t]);
            acc[1][t] = mfma_16x16x32(w1, b, acc[1][t]);
        }
    }
    const int oy = by0 + wave;
    uint16_t* out = a.out + (int64_t)blockIdx.y * a.out_frame;
#pragma unroll
    for (int t = 0; t < TT; ++t) {
        const int ox = bx0 + 16 * t + l16;
        if (oy >= H || ox >= W) continue;
        uint16_t* row = out + ((int64_t)oy * W + ox) * 32 + 4 * g;
#pragma unroll
        for (int r = 0; r < 2; ++r) {
            *reinterpret_cast<h4*>(row + 16 * r) = relu_h4(acc[r][t]);
        }
    }
}

#define CODEC_FRAME(p, n) ((p) + (int64_t)blockIdx.y * (n))
#define CODEC_IN_MAP MapSrc(CODEC_FRAME(a.in, a.in_frame), (uint32_t)(a.in_frame * 2))
#define CODEC_SKIP_MAP MapSrc(CODEC_FRAME(a.skip, a.skip_frame), (uint32_t)(a.skip_frame * 2))

extern "C" __global__ void __launch_bounds__(256) prism_codec_enc0(CodecArgs a) { codec_enc0_body(a); }
extern "C" __global__ void __launch_bounds__(256) prism_codec_enc1(CodecArgs a) {
    codec_stage<SrcConvNHWC<32, 2>, 64, CODEC_TT_ENC1, true>(a, SrcConvNHWC<32, 2>{CODEC_IN_MAP, a.in_w, a.in_h});
}
extern "C" __global__ void __launch_bounds__(256) prism_codec_dec2(CodecArgs a) {
    codec_stage<SrcDec<128, 64>, 64, CODEC_TT_DEC2, true>(
        a, SrcDec<128, 64>{CODEC_IN_MAP, CODEC_SKIP_MAP, a.in_w, a.in_h, a.out_w});
}
extern "C" __global__ void __launch_bounds__(256) prism_codec_dec1_out(CodecArgs a) { codec_dec_out<CODEC_TT_DEC1>(a); }
#undef CODEC_FRAME
#undef CODEC_IN_MAP
#undef CODEC_SKIP_MAP
