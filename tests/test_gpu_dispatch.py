"""The chain's choice of kernels and sub-chains by the number of windows (the
rules' edges: test_dispatch_rules.py). Frames never interact, so a frame's output is
the same bits whichever side of an edge its batch lies on."""
import numpy as np
import pytest

import prism_amd as P


@pytest.mark.gpu
@pytest.mark.parametrize("name,batches", [
    ("moe64", (1, 3, 4, 5, 9)),     # 64, 192 | 256 windows; a sub-chain of 256, of 320
    ("moe32", (1, 3, 4, 9)),
    ("std256", (1, 4, 5, 6, 8, 9)),  # 256 | 320 in 8-wave sub-chains | 384, 512 | 576 in 4-wave ones
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
    ref = []  # every frame on its own
    for f in range(max(batches)):
        engine.forward(dx.ptr + f * n * d * 2, dy.ptr, 1)
        hip.sync()
        ref.append(hip.download(np.empty(n * d, np.uint16), dy.ptr))
    assert all((ref[0] != r).any() for r in ref[1:])
    for b in batches:
        for graph in (False, True):
            print(f"[dispatch] {name} batch {b} graph {graph}", flush=True)
            hip.memset(dy.ptr, 0xFF, x.nbytes)
            engine.forward(dx.ptr, dy.ptr, b, graph=graph)
            hip.sync()
            y = hip.download(np.empty((b, n * d), np.uint16), dy.ptr)
            for f in range(b):
                assert (y[f] == ref[f]).all(), f"batch {b}: frame {f} differs"


@pytest.mark.gpu
@pytest.mark.parametrize("name,H,W,batch", [
    ("moe64", 24, 64, 22),   # 528 windows, more than 32 experts: both sub-chains on 8 waves
    ("moe64", 24, 64, 23),   # ... of 264 and 288
    ("moe64", 17, 25, 48),   # 576 windows, few tokens: by their own windows
    ("std256", 17, 25, 23),  # 276 windows, a third of them half padded: sub-chains
    ("std256", 9, 24, 43),   # 258, the last two half padded: one launch
])
def test_small_frames_in_a_large_batch(hip, engine, device_arena, name, H, W, batch):
    """First, middle (the sub-chains' seam) and last frames as on their own."""
    cfg = P.CONFIGS[name]
    desc = cfg.desc(n_blocks=2, H=H, W=W)
    blob, offs = P.synth_weights(desc, seed=5, routing=cfg.routing)
    engine.load_weights(desc, blob, offs)
    d, n = cfg.dim, H * W
    x = P.synth_features(cfg, batch=batch, H=H, W=W, seed=6).reshape(batch, n * d)
    dx, dy, dz = device_arena(x.nbytes), device_arena(x.nbytes), device_arena(n * d * 2)
    hip.upload(dx.ptr, x)
    print(f"[dispatch] {name} {H}x{W} batch {batch}", flush=True)
    hip.memset(dy.ptr, 0xFF, x.nbytes)
    engine.forward(dx.ptr, dy.ptr, batch)
    hip.sync()
    y = hip.download(np.empty((batch, n * d), np.uint16), dy.ptr)
    for f in sorted({0, 1, batch // 2 - 1, batch // 2, batch // 2 + 1, batch - 2, batch - 1}):
        engine.forward(dx.ptr + f * n * d * 2, dz.ptr, 1)
        hip.sync()
        assert (y[f] == hip.download(np.empty(n * d, np.uint16), dz.ptr)).all(), f"frame {f} differs"


@pytest.mark.gpu
@pytest.mark.parametrize("name,batch", [("std256", 1), ("std256", 5), ("dense128", 1), ("dense128", 8)])
@pytest.mark.parametrize("beta_blocks", [(), (0,), (2,), (0, 1, 2)])
def test_dense_chain_in_one_launch(hip, engine, device_arena, name, batch, beta_blocks):
    """Blocks with and without an LN1 beta (whose padded window slots need the
    blob's own bias) in one launch: the stage calls' output bit for bit."""
    H, W, nb = 61, 59, 3
    cfg = P.CONFIGS[name]
    desc = cfg.desc(n_blocks=nb, H=H, W=W)
    blob, offs = P.synth_weights(desc, seed=7, routing=cfg.routing)
    d, n = cfg.dim, batch * H * W
    for b in beta_blocks:
        beta = np.random.default_rng(b).normal(0, 0.2, d).astype(np.float16)
        blob[offs[b].ln1_b:offs[b].ln1_b + d] = beta.view(np.uint16)
    engine.load_weights(desc, blob, offs)
    x = P.synth_features(cfg, batch=batch, H=H, W=W, seed=8).reshape(-1)
    dx, dy, feats = device_arena(x.nbytes), device_arena(x.nbytes), device_arena(3 * x.nbytes)
    hip.upload(dx.ptr, x)
    hip.upload(feats.ptr, x)
    print(f"[dispatch] {name} batch {batch} beta in blocks {beta_blocks}", flush=True)
    engine.forward(dx.ptr, dy.ptr, batch)
    cur, nxt = 0, 2 * n * d
    for b in range(nb):
        assert engine.attn(engine.attn_push(b, cur, n * d), feats.ptr, batch) == 0, engine.error()
        assert engine.experts(engine.expert_push(b, H * W, n * d, nxt), feats.ptr, None, batch) == 0, engine.error()
        cur, nxt = nxt, cur
    hip.sync()
    got = hip.download(np.empty(n * d, np.uint16), dy.ptr)
    ref = hip.download(np.empty(n * d, np.uint16), feats.ptr + cur * 2)
    assert (got == ref).all(), f"{int((got != ref).sum())} values differ"


@pytest.mark.gpu
@pytest.mark.parametrize("name", ["moe16", "moe64"])
@pytest.mark.parametrize("H,W,batch", [
    (8, 8, 1),      # one workgroup: one ticket group
    (8, 56, 1),     # 7 and 9 workgroups: fewer groups than 8, one of them with two tickets
    (8, 72, 1),
    (17, 61, 3),    # 72 windows: 8 groups of 9
    (61, 59, 5),    # 320: 4-wave attention
])
def test_stage_counts_by_the_last_workgroup(hip, engine, device_arena, name, H, W, batch):
    """The routing stage calls' totals, moved by the launch's last workgroup:
    exact on every call, each of which finds the row and tickets cleared."""
    cfg = P.CONFIGS[name]
    desc = cfg.desc(n_blocks=1, H=H, W=W)
    blob, offs = P.synth_weights(desc, seed=9, routing=cfg.routing)
    engine.load_weights(desc, blob, offs)
    T, d, N = H * W, cfg.dim, cfg.n_experts
    n = batch * T
    x = P.synth_features(cfg, batch=batch, H=H, W=W, seed=10).reshape(-1)
    feats, aux = device_arena(2 * x.nbytes), device_arena(P.aux_elems(N, n) * 4)
    hip.upload(feats.ptr, x)
    pa = engine.attn_push(0, 0, n * d, H, W)
    for call in ("attn_route", "router", "attn_route", "router"):
        print(f"[dispatch] {name} {H}x{W} batch {batch} {call}", flush=True)
        hip.memset(aux.ptr, 0xFF, P.aux_elems(N, n) * 4)
        pr = engine.router_push(0, T, n * d, 0, n, n + N)
        rc = engine.attn_route(pa, pr, feats.ptr, aux.ptr, batch) if call == "attn_route" else \
            engine.router(pr, feats.ptr, aux.ptr, batch)
        assert rc == 0, engine.error()
        hip.sync()
        host = hip.download(np.empty(n + N, np.int32), aux.ptr)
        assert (host[n:] == np.bincount(host[:n], minlength=N)).all()


@pytest.mark.gpu
@pytest.mark.parametrize("name,W", [("moe16", 248), ("moe16", 249), ("moe64", 224), ("moe64", 225)])
def test_expert_stage_at_the_edge_of_one_round(hip, engine, device_arena, name, W):
    """n / 64 + n_experts / 2 = 256 tiles (8 waves) and 257 (4 waves): a frame's
    rows are the same bits alone, in a batch of two (4 waves), and its first quarter's
    alone (8 waves)."""
    H, d = 64, P.CONFIGS[name].dim
    cfg = P.CONFIGS[name]
    desc = cfg.desc(n_blocks=1, H=H, W=W)
    blob, offs = P.synth_weights(desc, seed=11, routing=cfg.routing)
    engine.load_weights(desc, blob, offs)
    T, N = H * W, cfg.n_experts
    x = P.synth_features(cfg, batch=2, H=H, W=W, seed=12).reshape(-1)
    feats, aux = device_arena(2 * x.nbytes), device_arena(P.aux_elems(N, 2 * T) * 4)
    ys = []
    for batch, T in ((1, H * W), (2, H * W), (1, H * W // 4)):
        n = batch * T
        hip.upload(feats.ptr, x)
        hip.memset(feats.ptr + x.nbytes, 0xFF, x.nbytes)  # NaN: every row must be written
        print(f"[dispatch] experts {name} {H}x{W} batch {batch}", flush=True)
        assert engine.router(engine.router_push(0, T, 0, 0, n, n + N), feats.ptr, aux.ptr, batch) == 0, engine.error()
        push = engine.expert_push(0, T, 0, x.size, 0, n, n + N)
        assert engine.experts(push, feats.ptr, aux.ptr, batch) == 0, engine.error()
        hip.sync()
        ys.append(hip.download(np.empty(n * d, np.uint16), feats.ptr + x.nbytes))
    frame = H * W * d
    assert (ys[0] == ys[1][:frame]).all() and (ys[2] == ys[0][:frame // 4]).all()
    assert np.isfinite(ys[1].view(np.float16)).all()


@pytest.mark.gpu
def test_no_lds_beside_an_8_wave_expert_tile_for_an_attention_window(hip):
    """160 KB a CU; sub-chains run slower where there is."""
    import ctypes as C
    import os

    rt, mod, fn = C.CDLL("libamdhip64.so"), C.c_void_p(), C.c_void_p()
    path = os.path.join(os.path.dirname(os.path.abspath(P.__file__)), "prism_kernels.hsaco")
    assert rt.hipModuleLoad(C.byref(mod), path.encode()) == 0

    def lds(kernel):
        v = C.c_int()
        assert rt.hipModuleGetFunction(C.byref(fn), mod, kernel.encode()) == 0
        assert rt.hipFuncGetAttribute(C.byref(v), 1, fn) == 0  # HIP_FUNC_ATTRIBUTE_SHARED_SIZE_BYTES
        return v.value

    try:
        least = min(lds(f"prism_attn_d256{w}_r{r}") for w in ("", "_w8") for r in (1, 2, 3, 4))
        assert 64 * 1024 < least < 80 * 1024
        assert lds("prism_expert_d256_bm64_w8") + least > 160 * 1024
    finally:
        assert rt.hipModuleUnload(mod) == 0
