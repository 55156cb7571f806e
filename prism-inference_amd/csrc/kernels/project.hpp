/*
 * project.hpp - projection adapters either side of the block chain.
 *
 * Restates shaders/pw_project_128to256.comp.glsl:25-37 (y = r16(W x + b), then
 * ReLU) and shaders/pw_project_256to128.comp.glsl:25-32 (y = r16(W x + b)),
 * which the reference runs one thread per token, as a GEMM over 64-token
 * tiles: C^T = W * X^T with the packed weights as the A operand. A tile's 64
 * token rows are one contiguous block in and one out (HWC): they pass through
 * an LDS tile as whole rows, 16 bytes per lane, and the B fragments (token
 * 16t + l16, channels 32ks + 8g .. +7) are read from there. Workgroup =
 * NW waves; wave w computes output rows [w*OUT/NW, +OUT/NW) of a tile's 64
 * tokens, accumulators starting at the bias. Persistent: workgroup b takes
 * tiles b, b + G, b + 2G, ... (G = the grid), holds its waves' weight
 * fragments in registers across them, and requests the next tile's rows
 * before the current tile's MFMAs. On 8 waves a wave holds half the weights
 * (112 VGPRs, 16 waves per CU instead of 8: both d256 launches of 4 and 6
 * frames of 68x120 15.2 -> 13.9 and 19.9 -> 18.3 us); which launches take
 * them: project_w8 (engine/rules.h).
 */
#pragma once
#include "common.hpp"

template <int IN, int OUT, bool RELU, int NW>
__device__ __forceinline__ void project_body(const ProjArgs& a) {
    constexpr int KS = IN / 32;  /* k-steps                     */
    constexpr int NT = 64 * NW;  /* threads                     */
    constexpr int RT = OUT / 16 / NW; /* 16-row output tiles per wave */
    constexpr int TT = 4;        /* 16-token tiles per token tile */
    constexpr int LI = IN + 8, LO = OUT + 8;  /* padded LDS rows (halfs) */
    constexpr int EI = 64 * IN / 8 / NT;      /* 16-byte input chunks per thread  */
    constexpr int EO = 64 * OUT / 8 / NT;     /* 16-byte output chunks per thread */
    static_assert(IN % 32 == 0 && RT >= 1 && EI >= 1 && EO >= 1, "shape");
    __shared__ __attribute__((aligned(16))) f16 tin[64 * LI];
    __shared__ __attribute__((aligned(16))) f16 tout[64 * LO];

    const int lane = lane_id();
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int l16 = lane & 15;
    const int g = lane >> 4;
    const int64_t ntiles = (a.n_tokens + 63) / 64;

    /* the rows of token tile `tile` (one contiguous block): 16 bytes per
     * lane, whole cache lines per wave load; rows past the end read the
     * tile's last row (no branch around the loads, so they go out together)
     * and are kept as zero */
    auto load_rows = [&](int64_t tile, h8 (&x)[EI]) {
        const int64_t tok0 = tile * 64;
        const int rows = (int)min<int64_t>(64, a.n_tokens - tok0);
#pragma unroll
        for (int k = 0; k < EI; ++k) {
            const int q = threadIdx.x + NT * k, r = q / (IN / 8), c8 = (q % (IN / 8)) * 8;
            const h8 v = *reinterpret_cast<const h8*>(a.in + (tok0 + min(r, rows - 1)) * IN + c8);
            x[k] = r < rows ? v : h8{};
        }
    };
    int64_t tile = blockIdx.x;
    h8 xin[EI];
    if (tile < ntiles) load_rows(tile, xin);
    /* this wave's weight fragments and its bias, held for every tile */
    const FragSrc src(a.w, (unsigned)(OUT * IN * 2));
    h8 wf[RT][KS];
#pragma unroll
    for (int ks = 0; ks < KS; ++ks)
#pragma unroll
        for (int r = 0; r < RT; ++r) wf[r][ks] = src.load((wave * RT + r) * KS + ks, lane * 16);
    f4 bias[RT];
#pragma unroll
    for (int r = 0; r < RT; ++r) {
        const int ch = (wave * RT + r) * 16 + 4 * g;
        bias[r] = f4{a.b[ch], a.b[ch + 1], a.b[ch + 2], a.b[ch + 3]};
    }

    for (; tile < ntiles; tile += gridDim.x) { /* uniform over the workgroup */
        const int64_t tok0 = tile * 64;
        const int rows = (int)min<int64_t>(64, a.n_tokens - tok0);
#pragma unroll
        for (int k = 0; k < EI; ++k) {
            const int q = threadIdx.x + NT * k, r = q / (IN / 8), c8 = (q % (IN / 8)) * 8;
            *reinterpret_cast<h8*>(tin + r * LI + c8) = xin[k];
        }
        __syncthreads(); /* the input tile is in; the previous tile's output rows are out of tout */
        /* the next tile's rows go out now and arrive under this tile's MFMAs */
        if (tile + gridDim.x < ntiles) load_rows(tile + gridDim.x, xin);

        f4 acc[RT][TT]; /* starts at the bias */
#pragma unroll
        for (int r = 0; r < RT; ++r)
#pragma unroll
            for (int t = 0; t < TT; ++t) acc[r][t] = bias[r];
#pragma unroll
        for (int ks = 0; ks < KS; ++ks)
#pragma unroll
            for (int t = 0; t < TT; ++t) {
                const h8 xf = *reinterpret_cast<const h8*>(tin + (16 * t + l16) * LI + 32 * ks + 8 * g);
#pragma unroll
                for (int r = 0; r < RT; ++r) acc[r][t] = mfma_16x16x32(wf[r][ks], xf, acc[r][t]);
            }
#pragma unroll
        for (int t = 0; t < TT; ++t)
#pragma unroll
            for (int r = 0; r < RT; ++r) {
                *reinterpret_cast<h4*>(tout + (16 * t + l16) * LO + (wave * RT + r) * 16 + 4 * g) =
                    RELU ? relu_h4(acc[r][t]) : cvt_h4(acc[r][t]);
            }
        __syncthreads(); /* the output tile is complete; every wave is done reading tin */
        /* every LDS read first, then the stores (a read under a store's
           condition costs one LDS round trip per pass) */
        h8 yo[EO];
#pragma unroll
        for (int k = 0; k < EO; ++k) {
            const int q = threadIdx.x + NT * k, r = q / (OUT / 8), c8 = (q % (OUT / 8)) * 8;
            yo[k] = *reinterpret_cast<const h8*>(tout + r * LO + c8);
        }
#pragma unroll
        for (int k = 0; k < EO; ++k) {
            const int q = threadIdx.x + NT * k, r = q / (OUT / 8), c8 = (q % (OUT / 8)) * 8;
            if (r < rows) *reinterpret_cast<h8*>(a.out + (tok0 + r) * OUT + c8) = yo[k];
        }
    }
}

/* up: encoder channels (128) -> model dim, ReLU; down: model dim -> 128 */
extern "C" __global__ void __launch_bounds__(512, 4) prism_project_up_d256_w8(ProjArgs a) {
    project_body<128, 256, true, 8>(a);
}
extern "C" __global__ void __launch_bounds__(512, 4) prism_project_down_d256_w8(ProjArgs a) {
    project_body<256, 128, false, 8>(a);
}
extern "C" __global__ void __launch_bounds__(256, 2) prism_project_down_d256(ProjArgs a) {
    project_body<256, 128, false, 4>(a);
}
extern "C" __global__ void __launch_bounds__(256, 2) prism_project_up_d128(ProjArgs a) {
    project_body<128, 128, true, 4>(a);
}
extern "C" __global__ void __launch_bounds__(256, 2) prism_project_down_d128(ProjArgs a) {
    project_body<128, 128, false, 4>(a);
}
