/* The engine's dispatch rules (csrc/engine/rules.h) for ctypes. */
#include "../prism-inference_amd/csrc/engine/rules.h"

using namespace prism;

static prism_model_desc desc(int dim, int experts, int h, int w) {
    prism_model_desc d{};
    d.dim = dim;
    d.n_experts = experts;
    d.spatial_h = h;
    d.spatial_w = w;
    return d;
}

extern "C" {
/* sub-chains, negative where every block runs in one launch */
int chain(int dim, int experts, int h, int w, int batch) {
    const ChainPlan p = chain_plan(desc(dim, experts, h, w), batch);
    return p.one_launch ? -p.split : p.split;
}
/* of the last sub-chain's launches, the largest */
static int last_frames(const ChainPlan& p, int batch) { return batch - batch * (p.split - 1) / p.split; }
int chain_attention_waves(int dim, int experts, int h, int w, int batch) {
    const ChainPlan p = chain_plan(desc(dim, experts, h, w), batch);
    return chain_attn_w8(desc(dim, experts, h, w), p, (long long)((w + 7) / 8) * ((h + 7) / 8) * last_frames(p, batch)) ? 8 : 4;
}
int chain_expert_waves(int dim, int experts, int h, int w, int batch) {
    const ChainPlan p = chain_plan(desc(dim, experts, h, w), batch);
    const int partial = experts > 1 ? experts : 0;
    const long long n = (long long)h * w * last_frames(p, batch), tiles = ((n + 63) / 64 + partial + 7) / 8 * 8;
    return expert_w8(dim, tiles, n, partial, &p) ? 8 : 4;
}
/* the leading blocks' expert weights past the memory-side cache? */
int chain_expert_streams(int dim, int experts, int h, int w, int batch) {
    return expert_wnt(true, chain_expert_waves(dim, experts, h, w, batch) == 8,
                      chain_plan(desc(dim, experts, h, w), batch));
}
int attention_waves(int dim, long long windows) { return attn_w8(dim, windows) ? 8 : 4; }
int projection_waves(int dim, int up, long long tiles) { return project_w8(dim, up, tiles) ? 8 : 4; }
long long projection_grid(int dim, long long tiles) { return project_grid(dim, tiles); }
int enc2_slots(long long blocks) { return codec_enc2_slots(blocks); }
unsigned grid_of(long long blocks, int slots) { return even_grid(blocks, slots); }
}
