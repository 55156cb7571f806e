"""prism_encode and prism_decode against the stage calls they replace, bit for
bit, at the edges of their blocks: map sizes one below, at and one above a
block's, odd sizes at every resolution, several frames, and more blocks than
the persistent launches have workgroups. enc2, enc3 and dec3 are the same kernels
in both, so their loops over several blocks are compared with launches in which
a workgroup has one block (those meet the oracle in test_gpu_codec.py)."""
import numpy as np
import pytest

import oracle as O
import prism_amd as P


@pytest.mark.gpu
@pytest.mark.parametrize("render,batch", [
    ((8, 8), 1),       # one token
    ((61, 5), 2),      # r1 31 x 3, every map odd or one row
    ((64, 32), 1),     # r1 32 x 16: whole blocks
    ((65, 33), 3),     # one pixel into the next block, both ways
    ((130, 9), 1),
    ((259, 131), 2),   # odd at every resolution
    ((960, 540), 3),   # several blocks per workgroup
])
def test_encode_decode_equal_the_stage_calls(hip, engine, device_arena, render, batch):
    r = P.codec_resolutions(*render)
    (w0, h0), (w1, h1), (w2, h2), (w3, h3) = r
    desc = P.CONFIGS["moe16"].desc(n_blocks=1, H=h3, W=w3)
    blob, offs = P.synth_weights(desc, seed=2)
    engine.load_weights(desc, blob, offs)
    cblob, coffs, _ = P.synth_codec(desc, seed=4, render_w=w0, render_h=h0)
    engine.load_codec(cblob, coffs)
    rng = np.random.default_rng(w0 + h0)
    frame = O.f32_to_f16bits(rng.standard_normal(batch * 9 * h0 * w0).astype(np.float32))
    sizes = {"e0": w0 * h0 * 32, "e1": w1 * h1 * 64, "e2": w2 * h2 * 128, "e3": w3 * h3 * 128, "d3": w2 * h2 * 128,
             "d2": w1 * h1 * 64, "disp": w0 * h0 * 12}
    m = {k: device_arena(batch * n * 2 + 256) for k, n in sizes.items()}
    df, db, dd = device_arena(frame.nbytes), device_arena(batch * sizes["e3"] * 2 + 256), \
        device_arena(batch * sizes["disp"] * 2 + 256)
    hip.upload(df.ptr, frame)
    print(f"[codec blocks] {render} batch {batch}: maps {r}", flush=True)
    for st, (src, skip, dst) in enumerate([(df, None, "e0"), (m["e0"], None, "e1"), (m["e1"], None, "e2"),
                                           (m["e2"], None, "e3"), (m["e3"], "e2", "d3"), (m["d3"], "e1", "d2"),
                                           (m["d2"], "e0", "disp")]):
        engine.codec_stage(st, src.ptr, m[skip].ptr if skip else None, m[dst].ptr, batch)
    for a in (db, dd):
        hip.memset(a.ptr, 0xAB, a.nbytes)
    engine.encode(df.ptr, db.ptr, batch)
    engine.decode(db.ptr, dd.ptr, batch)
    hip.sync()

    def words(a, n):
        return hip.download(np.empty(n, np.uint16), a.ptr)

    n = batch * sizes["e3"]
    got, ref = words(db, n + 128), words(m["e3"], n)
    assert (got[:n] == ref).all(), f"bottleneck: {int((got[:n] != ref).sum())} values differ"
    assert (got[n:] == 0xABAB).all(), "written past the bottleneck"
    n = batch * sizes["disp"]
    got, ref = words(dd, n + 128), words(m["disp"], n)
    assert (got[:n] == ref).all(), f"display: {int((got[:n] != ref).sum())} values differ"
    assert (got[n:] == 0xABAB).all(), "written past the display"


@pytest.mark.gpu
@pytest.mark.parametrize("render,batch", [
    ((960, 540), 3),   # 1,530 / 765 / 1,632 blocks: 3, 2 and 3 a workgroup
    ((957, 531), 3),   # ragged blocks on both edges, a workgroup's blocks of several frames
    ((331, 251), 11),  # small frames: every workgroup crosses from one to another
])
def test_stages_over_several_blocks_equal_single_ones(hip, engine, rules, device_arena, render, batch):
    r = P.codec_resolutions(*render)
    (w0, h0), (w1, h1), (w2, h2), (w3, h3) = r
    desc = P.CONFIGS["moe16"].desc(n_blocks=1, H=h3, W=w3)
    blob, offs = P.synth_weights(desc, seed=2)
    engine.load_weights(desc, blob, offs)
    cblob, coffs, _ = P.synth_codec(desc, seed=4, render_w=w0, render_h=h0)
    engine.load_codec(cblob, coffs)

    def blocks(w, h, rows, cols):
        return -(-w // cols) * -(-h // rows)

    # stage, input, skip, output elements of a frame; a frame's blocks; workgroups held at once
    e1, e2, e3 = w1 * h1 * 64, w2 * h2 * 128, w3 * h3 * 128
    b2, b3, bd = blocks(w2, h2, 4, 16), blocks(w3, h3, 4, 8), blocks(w2, h2, 2, 32)
    for st, nin, nskip, nout, blk, slots in ((2, e1, 0, e2, b2, rules.enc2_slots), (3, e2, 0, e3, b3, lambda n: 512),
                                             (4, e3, e2, e2, bd, lambda n: 768)):
        assert batch * blk > slots(batch * blk), "one block a workgroup: nothing to compare"
        rng = np.random.default_rng(st)
        src, skip = (O.f32_to_f16bits(np.maximum(rng.standard_normal((batch, n)), 0).astype(np.float32))
                     for n in (nin, max(nskip, 8)))
        dsrc, dskip = device_arena(src.nbytes), device_arena(skip.nbytes)
        hip.upload(dsrc.ptr, src)
        hip.upload(dskip.ptr, skip)
        out = device_arena(batch * nout * 2 + 256)

        def run(first, n):
            hip.memset(out.ptr, 0xAB, out.nbytes)
            engine.codec_stage(st, dsrc.ptr + first * nin * 2, dskip.ptr + first * nskip * 2 if nskip else None, out.ptr, n)
            hip.sync()
            got = hip.download(np.empty(n * nout + 128, np.uint16), out.ptr)
            assert (got[n * nout:] == 0xABAB).all(), "written past the map"
            return got[:n * nout].reshape(n, nout)

        print(f"[codec blocks] stage {st} {render} batch {batch}: {batch * blk} blocks", flush=True)
        whole = run(0, batch)
        # frames at once with a block a workgroup (enc2 of a 960x540 frame: two, as against the oracle)
        per = max(1, 256 // blk)
        assert per * blk <= slots(per * blk) or st == 2
        for f in range(0, batch, per):
            one = run(f, min(per, batch - f))
            assert (one == whole[f:f + per]).all(), f"stage {st}, frames from {f}"
