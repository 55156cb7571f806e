"""The chain's choice of kernels and sub-chains by the number of windows: 8-wave
workgroups up to one per CU (256 windows at d256, 511 at d128),
4-wave ones above; two sub-chains above 192 windows (MoE) or 512 (dense). Frames never interact, so a frame's
output is the same bits whichever side of an edge its batch lies on."""
import numpy as np
import pytest

import prism_amd as P


@pytest.mark.gpu
@pytest.mark.parametrize("name,batches", [
    ("moe64", (1, 3, 4, 5, 9)),     # 64, 192 | 256 windows; a sub-chain of 256, of 320
    ("moe32", (1, 3, 4, 9)),
    ("std256", (1, 4, 5, 8, 9)),
    ("dense128", (1, 7, 8, 9)),     # 448 | 512 | 576
])
def test_frame_is_the_same_in_every_batch(hip, engine, device_arena, name, batches):
    H, W = 61, 59  # 8 x 8 windows, ragged on both edges
    cfg = P.CONFIGS[name]
    desc = cfg.desc(n_blocks=2, H=H, W=W)
    blob, offs = P.synth_weights(desc, seed=5, routing=cfg.routing)
    engine.load_weights(desc, blob, offs)
    d, n = cfg.dim, H * W
    x = P.synth_features(cfg, batch=max(batches), H=H, W=W, seed=6).reshape(max(batches), n * d)
    dx, dy = device_arena(x.nbytes), device_arena(x.nbytes)
    hip.upload(dx.ptr, x)
    ref = None
    for b in batches:
        for graph in (False, True):
            print(f"[dispatch] {name} batch {b} graph {graph}", flush=True)
            hip.memset(dy.ptr, 0xFF, x.nbytes)
            engine.forward(dx.ptr, dy.ptr, b, graph=graph)
            hip.sync()
            y = hip.download(np.empty((b, n * d), np.uint16), dy.ptr)
            if ref is None:
                ref = y
            assert (y[0] == ref[0]).all(), f"batch {b}: frame 0 differs"
            if b == max(batches):  # the last frame (of the second sub-chain) on its own
                engine.forward(dx.ptr + (b - 1) * n * d * 2, dy.ptr, 1, graph=graph)
                hip.sync()
                assert (hip.download(np.empty(n * d, np.uint16), dy.ptr) == y[b - 1]).all()
