/*
 * prism_kernels.hip - the gfx950 code object (prism_kernels.hsaco) loaded by
 * the host engine with hipModuleLoad and launched with hipModuleLaunchKernel.
 *
 * Kernels (extern "C" names, one per stage and supported shape):
 *   prism_attn_d{256,128}[_w8]                     attention stage (4 or 8 waves)
 *   prism_attn_d{256,128}[_w8]_r{1..4}             attention + fused routing
 *   prism_attn_d{256,128}[_w8]_ffn                 a dense block in one launch
 *   prism_chain_d{256,128}[_w8]                    every block of a dense chain in one launch
 *   prism_router_d{256,128}_n{1..4}                router + counting sort
 *   prism_expert_d{256,128}_bm64[_w8], _d256_bm{128,96}  grouped expert FFN
 *   prism_project_{up,down}_d{256,128}[_w8]        projection adapters (128 <-> dim)
 *   prism_codec_enc{0,1}, prism_codec_dec2         conv encoder / fused decoder stages
 *   prism_codec_enc01, prism_codec_dec21_out       the same, fused in the frame (persistent)
 *   prism_codec_enc{2,3}, prism_codec_dec3         stages and frame alike (persistent)
 *   prism_codec_dec1_out                           dec1 + output conv + PixelShuffle + sigmoid
 *   prism_zero_i32                                 clears routing counters
 */
#include "attn.hpp"
#include "router.hpp"
#include "expert.hpp"
#include "project.hpp"
#include "codec.hpp"
#include "codec_enc.hpp"
#include "codec_dec.hpp"

/* Routing counters must start at zero; a kernel (not a memset node) keeps
 * the launch safe under stream capture. */
extern "C" __global__ void __launch_bounds__(256) prism_zero_i32(int32_t* p, int32_t n) {
    for (int i = blockIdx.x * 256 + threadIdx.x; i < n; i += gridDim.x * 256) p[i] = 0;
}
