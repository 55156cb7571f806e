"""Which kernels and grids the engine chooses, by size (csrc/engine/rules.h):
the edges of each rule."""
import pytest

ONE = -1  # every block in one launch


@pytest.mark.parametrize("dim,experts,h,w,batch,plan", [
    (256, 64, 64, 64, 3, 1), (256, 64, 64, 64, 4, 2),      # 192 | 256 windows
    (256, 16, 135, 240, 1, 1),                             # one frame never splits
    # more than 32 experts: not while windows and filled tiles are one round
    (256, 64, 56, 75, 3, 1), (256, 32, 56, 75, 3, 2),      # 210 windows, 229 tiles
    (256, 64, 56, 128, 2, 1), (256, 64, 57, 128, 2, 2),    # 256 tiles | 260
    (256, 64, 17, 25, 21, 1), (256, 64, 17, 25, 22, 2),    # 252 | 264 windows
    (128, 1, 68, 120, 1, ONE), (128, 1, 68, 120, 16, ONE),  # d128: always together
    (256, 1, 64, 64, 4, ONE),                              # 256 windows
    (256, 1, 64, 64, 8, ONE), (256, 1, 64, 64, 9, 2),      # 512 | 576
    # 257 to 341 windows' worth of work, a half-padded one counting 2/3: sub-chains
    (256, 1, 24, 32, 22, 2), (256, 1, 24, 32, 28, 2), (256, 1, 24, 32, 29, ONE),  # 264, 336 | 348
    (256, 1, 17, 25, 22, 2), (256, 1, 17, 25, 31, 2), (256, 1, 17, 25, 33, ONE),  # 372 (124 half) | 396 (132)
    (256, 1, 25, 33, 16, 2), (256, 1, 80, 80, 3, 2), (256, 1, 96, 88, 2, 2),      # 320 (80), 300, 264
    (256, 1, 21, 28, 28, 2), (256, 1, 20, 28, 33, ONE),    # 5 rows: no half ones, 336 | 4 rows: 396 (132)
    (256, 1, 68, 120, 2, ONE), (256, 1, 9, 24, 43, ONE),   # only half windows past the 256th
    (256, 1, 136, 128, 1, ONE),                            # 272 windows of one frame
    (256, 1, 135, 240, 2, 2),
])
def test_chain_plan(rules, dim, experts, h, w, batch, plan):
    assert rules.chain(dim, experts, h, w, batch) == plan


def test_attention_waves(rules):
    assert [rules.attention_waves(256, n) for n in (1, 256, 257)] == [8, 8, 4]
    assert [rules.chain_attention_waves(256, 1, 24, 32, b) for b in (21, 22, 28, 29, 43)] == [8, 8, 8, 4, 4]
    assert [rules.attention_waves(128, n) for n in (511, 512)] == [8, 4]


@pytest.mark.parametrize("experts,h,w,batch,attention,expert", [
    (64, 64, 64, 8, 8, 8),        # 512 windows: 256 a sub-chain, 320 tiles
    (64, 68, 120, 4, 8, 8),       # 540: both on 8 waves
    (64, 72, 120, 4, 8, 8),       # ... also at 334 tiles
    (64, 66, 118, 4, 8, 8),       # 307 tiles
    (64, 33, 51, 16, 4, 8),       # 275 tiles
    (64, 115, 77, 4, 4, 8), (64, 75, 75, 6, 4, 8), (64, 45, 80, 10, 4, 4),  # 344, 328 | 352
    (32, 84, 100, 4, 4, 8), (32, 92, 104, 4, 4, 4),                         # 296 | 336
    (64, 24, 64, 24, 4, 4),       # 576 windows
    (32, 68, 120, 4, 4, 8), (16, 68, 120, 4, 4, 8), (16, 72, 120, 5, 4, 4),
    (64, 24, 64, 23, 8, 8), (64, 96, 120, 3, 4, 4),  # 264 and 288 | 180 and 360: unequal halves
    (64, 68, 120, 16, 4, 4),
    # no sub-chains: filled tiles, n / 64 and half a tile per expert
    (64, 112, 128, 1, 8, 8), (64, 114, 126, 1, 8, 4),  # 256 | 257
    (16, 124, 128, 1, 8, 8), (16, 126, 126, 1, 8, 4),
    (1, 128, 128, 1, 8, 8), (1, 130, 130, 1, 4, 4),    # a dense chain's last FFN
])
def test_waves_of_routed_sub_chains(rules, experts, h, w, batch, attention, expert):
    assert rules.chain_attention_waves(256, experts, h, w, batch) == attention
    assert rules.chain_expert_waves(256, experts, h, w, batch) == expert


@pytest.mark.parametrize("h,w,batch,streams", [
    (68, 120, 1, True), (68, 120, 2, True), (135, 240, 1, True),  # 8 waves | 4 waves, one chain
    (68, 120, 8, False), (68, 120, 10, False),                    # 4 waves beside another sub-chain
])
def test_leading_blocks_weights_past_the_cache(rules, h, w, batch, streams):
    assert bool(rules.chain_expert_streams(256, 64, h, w, batch)) == streams


@pytest.mark.parametrize("dim,tiles,grid,up,down", [
    (256, 1, 1, 8, 8), (256, 513, 513, 8, 8), (256, 900, 900, 8, 8), (256, 1024, 1024, 8, 8),
    (256, 1025, 512, 8, 4), (256, 2040, 512, 8, 4),
    (128, 512, 512, 4, 4), (128, 513, 512, 4, 4),
])
def test_projection_launches(rules, dim, tiles, grid, up, down):
    assert rules.projection_grid(dim, tiles) == grid
    assert (rules.projection_waves(dim, 1, tiles), rules.projection_waves(dim, 0, tiles)) == (up, down)


@pytest.mark.parametrize("blocks,grid", [(256, 256), (257, 129), (510, 255), (1024, 256), (1025, 342), (2040, 510)])
def test_enc2_keeps_to_one_workgroup_per_cu(rules, blocks, grid):
    """Two per CU pull the clock down for the chain that follows."""
    assert rules.grid_of(blocks, rules.enc2_slots(blocks)) == grid


@pytest.mark.parametrize("blocks,slots", [(1, 512), (511, 512), (512, 512), (513, 512), (1021, 256), (10**6, 768)])
def test_every_workgroup_of_a_persistent_launch_has_a_block(rules, blocks, slots):
    g = rules.grid_of(blocks, slots)
    each = -(-blocks // g)
    assert 0 < g <= slots and (each - 1) * g < blocks <= each * g
    assert each == -(-blocks // slots)
