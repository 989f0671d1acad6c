"""Whole dense blocks split into row bands across workgroups (`d8s_dense_block_parts`, block kind
"parts") on the GPU: every band count of the 32 x 32 and 16 x 16 blocks of the configuration-4 encoder
gives the bytes of the default encoder (two launches per layer / one workgroup per image), exact
against the C oracle on sampled pixels of its own inputs, under graph replay too (the kernel clears its
own synchronisation words for the next launch), with no bounded wait running out.  Two such runners on
two streams at once stay exact.  The 64- and 128-wide blocks split into bands give the same bytes too,
and an error word planted from the host makes the pass's features NaN and the next call raise."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from oracle import checks
from rsna_knee_efficiency_amd import dense8s, densenet, synthetic

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def c4(dev):
    model = densenet.seeded_densenet169(0).to(dev)
    cal = dense8s.calibrate(model, [synthetic.normalise(torch.from_numpy(c).to(dev))
                                    for c in np.split(synthetic.study_u8(64, 512, seed=7), 8)])
    plan = dense8s.make_plan(model.cpu(), cal, 512)
    pack = dense8s.make_pack(plan, 24, input_kind="u8")
    x = torch.from_numpy(synthetic.c5_study(0)[:24]).to(dev)
    base = dense8s.Dense8SEncoder(pack, dev.index or 0, 24, fused={0: "tile"})
    return {"plan": plan, "pack": pack, "x": x, "want": base(x).clone()}


def test_parts_options():
    meta = dense8s.pack_meta(dense8s.make_plan(densenet.seeded_densenet169(0), _fake_cal(), 512), 24)
    b = meta["blocks"]
    assert dense8s.parts_options(b[3]) == [1, 2, 4, 8]
    assert dense8s.parts_options(b[2]) == [4, 8, 16, 32]
    assert dense8s.parts_for(b[3], 24) == 8 and dense8s.parts_for(b[3], 96) == 2
    assert dense8s.parts_for(b[2], 24) == 8 and dense8s.parts_for(b[2], 96) is None


def _fake_cal():
    import sys
    from pathlib import Path
    sys.path.insert(0, str(Path(__file__).resolve().parent / "golden"))
    import make_tables
    return make_tables.fake_cal()


@pytest.mark.parametrize("kinds", [{2: "parts:8", 3: "parts:8"}, {2: "parts:4", 3: "parts:4"},
                                   {2: "parts:16", 3: "parts:2"}, {2: "parts:32", 3: "parts:1"}])
def test_parts_same_bytes(dev, c4, kinds):
    print(f"parts {kinds}", flush=True)
    enc = dense8s.Dense8SEncoder(c4["pack"], dev.index or 0, 24, fused={0: "tile", **kinds})
    got = enc(c4["x"]).clone()
    assert enc.sync_errors() == 0
    assert torch.equal(got, c4["want"])
    enc.capture(24)
    for _ in range(3):
        g = enc(c4["x"]).clone()
        _ = (c4["x"].float() * 2).sum()
        torch.cuda.synchronize(dev)
        assert torch.equal(g, c4["want"])
    assert enc.sync_errors() == 0


def test_parts_layers_exact(dev, c4):
    """The default band counts at 24 images traced: every layer of the banded blocks exact."""
    enc = dense8s.Dense8SEncoder(c4["pack"], dev.index or 0, 24, fused={0: "tile", 2: "parts", 3: "parts"})
    assert enc.fused[2] == "parts:8" and enc.fused[3] == "parts:8"
    trace, f = enc.trace(c4["x"])
    assert enc.sync_errors() == 0
    par = dense8s.kernel_params(c4["plan"])
    res = checks.summarize(checks.check_trace(enc, trace, f.cpu().numpy(), par, max_rows=1024))
    print(res)
    assert res["block"]["launches"] == 64 and res["block"]["mismatch"] == 0, res["block"]
    assert res["conv1"]["mismatch"] == 0 and res["trans"]["mismatch"] == 0
    assert res["final"]["equal"]


def test_parts_two_runners_at_once(dev, c4):
    encs = [dense8s.Dense8SEncoder(c4["pack"], dev.index or 0, 24, fused={0: "tile", 2: "parts", 3: "parts"})
            for _ in range(2)]
    xs = [c4["x"], torch.flip(c4["x"], dims=[0]).contiguous()]
    want = [c4["want"], None]
    base = dense8s.Dense8SEncoder(c4["pack"], dev.index or 0, 24, fused={0: "tile"})
    want[1] = base(xs[1]).clone()
    for e in encs:
        e.capture(24)
    for k in range(3):
        outs = dense8s.encode_concurrent([(encs[0], xs[0], False), (encs[1], xs[1], False)])
        got = [o.clone() for o in outs]
        torch.cuda.synchronize(dev)
        assert torch.equal(got[0], want[0]) and torch.equal(got[1], want[1]), k
    assert sum(e.sync_errors() for e in encs) == 0


@pytest.fixture(scope="module")
def small_first(dev):
    """A seeded DenseNet with 4 layers in its first block at 128 px: that block is 32 x 32 with 2
    groups in (below every prologue chunk of the banded kernel)."""
    model = densenet.seeded_densenet169(5, blocks=(4, 1, 2, 2)).to(dev)
    x_u8 = synthetic.study_u8(8, 128, seed=3)
    cal = dense8s.calibrate(model, [synthetic.normalise(torch.from_numpy(x_u8).to(dev))])
    pack = dense8s.make_pack(dense8s.make_plan(model.cpu(), cal, 128), 8, input_kind="u8")
    assert pack["meta"]["blocks"][0]["c0"] // 32 == 2 and pack["meta"]["blocks"][0]["L"] == 4
    x = torch.from_numpy(x_u8).to(dev)
    kinds = dense8s.fused_blocks(pack["meta"], None)
    kinds[0] = "conv"
    want = dense8s.Dense8SEncoder(pack, dev.index or 0, 8, fused=kinds)(x).clone()
    return {"pack": pack, "x": x, "kinds": kinds, "want": want}


@pytest.mark.parametrize("parts", [4, 8, 16, 32])
def test_parts_groups_below_first_chunk(dev, small_first, parts):
    """Layers whose second-newest group falls in the first prologue chunk (it is stored by the conv2
    that runs after the chunk was requested, and comes from conv2's copy in LDS): every band size
    (256, 128, 64 and 32 pixels) gives the bytes of two launches per layer."""
    print(f"small first block, parts:{parts}", flush=True)
    kinds = dict(small_first["kinds"])
    kinds[0] = f"parts:{parts}"
    enc = dense8s.Dense8SEncoder(small_first["pack"], dev.index or 0, 8, fused=kinds)
    got = enc(small_first["x"]).clone()
    assert enc.sync_errors() == 0
    assert torch.equal(got, small_first["want"])


@pytest.mark.parametrize("kinds", [{1: "parts:16"}, {1: "parts:32"}, {1: "parts:64"}, {0: "parts:128"}])
def test_parts_wide_maps(dev, c4, kinds):
    """The 64 x 64 block (12 layers) in 256-, 128- and 64-pixel bands and the 128 x 128 block (6 layers)
    in one-row bands: more bands than compute units (384 to 3072 workgroups), so images start as
    earlier ones finish; the bytes of the default encoder."""
    print(f"wide parts {kinds}", flush=True)
    enc = dense8s.Dense8SEncoder(c4["pack"], dev.index or 0, 24, fused={0: "tile", **kinds})
    got = enc(c4["x"]).clone()
    assert enc.sync_errors() == 0
    assert torch.equal(got, c4["want"])


@pytest.fixture(scope="module")
def odd_maps(dev):
    """Seeded DenseNets with short blocks at 288 px (maps 72, 36, 18, 9) and 416 px (104, 52, 26, 13): the
    features with every layer as two launches."""
    out = {}
    for img, n in ((288, 3), (416, 2)):
        model = densenet.seeded_densenet169(6, blocks=(2, 2, 4, 3)).to(dev)
        x_u8 = synthetic.study_u8(n, img, seed=4)
        cal = dense8s.calibrate(model, [synthetic.normalise(torch.from_numpy(x_u8).to(dev))])
        plan = dense8s.make_plan(model.cpu(), cal, img)
        pack = dense8s.make_pack(plan, n, input_kind="u8")
        x = torch.from_numpy(x_u8).to(dev)
        out[img] = {"plan": plan, "pack": pack, "x": x, "n": n,
                    "want": dense8s.Dense8SEncoder(pack, dev.index or 0, n, fused={})(x).clone()}
    return out


@pytest.mark.parametrize("img,block,bands", [
    (288, 2, 18), (416, 3, 13),                    # one pixel tile, partly filled (18 and 13 pixels)
    (288, 1, 36), (288, 3, 2),                     # two (36 pixels; bands of 5 and 4 rows)
    (288, 0, 72), (288, 2, 5), (288, 3, 1),        # up to four (72 pixels; uneven bands; one band, 81 pixels)
    (416, 3, 3),                                   # 65 pixels: a tile of one pixel, bands of 5, 4 and 4 rows
    (288, 0, 36), (416, 2, 4),                     # six (144 pixels; 182 in uneven bands)
    (288, 0, 24), (416, 1, 13), (416, 0, 104)])    # eight (216, 208 pixels); 104-wide rows
def test_bands_same_bytes(dev, odd_maps, img, block, bands):
    """Bands of any row count and width (`d8s_dense_block_bands`): the bytes of two launches per layer,
    eager and under graph replay, with no bounded wait running out."""
    print(f"bands img={img} block={block} bands={bands}", flush=True)
    m = odd_maps[img]
    enc = dense8s.Dense8SEncoder(m["pack"], dev.index or 0, m["n"], fused={block: f"bands:{bands}"})
    assert torch.equal(enc(m["x"]).clone(), m["want"])
    enc.capture(m["n"])
    for _ in range(2):
        g = enc(m["x"]).clone()
        _ = (m["x"].float() * 2).sum()
        torch.cuda.synchronize(dev)
        assert torch.equal(g, m["want"])
    assert enc.sync_errors() == 0


@pytest.mark.parametrize("img,n,kinds", [
    (288, 64, {1: "bands:8", 2: "bands:3", 3: "bands:3"}),       # 512 and 192 workgroups; 36, 18 and 9 wide
    (416, 65, {2: "bands:5", 3: "bands:4"}),                      # 325 and 260: bands of 6 and 5, 4 and 3 rows
])
def test_bands_several_rounds_and_two_runners(dev, odd_maps, img, n, kinds):
    """Ragged bands of more workgroups than CUs (an image's bands start as others end), alone and with a second
    runner's ragged bands beside them (`encode_concurrent`), eager and replayed."""
    m = odd_maps[img]
    print(f"bands in rounds img={img} n={n} {kinds}", flush=True)
    pack = dense8s.make_pack(m["plan"], n, input_kind="u8")
    encs = [dense8s.Dense8SEncoder(pack, dev.index or 0, n, fused=kinds) for _ in range(2)]
    pick = torch.arange(n, device=dev) % m["n"]
    x, want = m["x"][pick].contiguous(), m["want"][pick]
    xs, wants = [x, x.flip(0).contiguous()], [want, want.flip(0)]
    for rep in range(3):
        if rep == 1:
            for e in encs:
                e.capture(n)
        assert torch.equal(encs[0](x), want), rep
        outs = [o.clone() for o in dense8s.encode_concurrent([(e, v, False) for e, v in zip(encs, xs)])]
        torch.cuda.synchronize(dev)
        assert all(torch.equal(o, w) for o, w in zip(outs, wants)), rep
    assert sum(e.sync_errors() for e in encs) == 0


def test_pair_with_kinds_of_its_own(dev, odd_maps):
    """A pair whose blocks run as other kinds than each encoder's own: each encoder's features, eager and
    replayed; kinds the caller gave stay."""
    m = odd_maps[416]
    n = 65
    pack = dense8s.make_pack(m["plan"], n, input_kind="u8")
    encs = [dense8s.Dense8SEncoder(pack, dev.index or 0, n) for _ in range(2)]
    x = m["x"][torch.arange(n, device=dev) % m["n"]].contiguous()
    want = m["want"][torch.arange(n, device=dev) % m["n"]]
    pair = dense8s.EncoderPair(*encs)
    ran = [s.entry for s in pair.programs()[0]]
    print(f"pair of {encs[0].fused}: {sorted(set(ran))}", flush=True)
    assert ran != [s.entry for s in encs[0].program] and encs[0].max_bands > 0
    for rep in range(3):
        if rep == 1:
            pair.capture(n)
        fa, fb = pair(x)
        assert torch.equal(fa, want) and torch.equal(fb, want), rep
        assert torch.equal(encs[0](x), want)          # its own program beside the pair's
    # block 1 (52 wide) runs fused alone and as two launches in the pair, unless a variant is recorded for it
    entries = lambda prog, bi: {st.entry for st in prog if st.block == bi and st.family != "trans"}  # noqa: E731
    assert entries(encs[0].program, 1) == {"d8s_dense"} and entries(pair.programs()[0], 1) == {"d8s_conv1", "d8s_conv2"}
    varied = dict(pack, meta=dense8s.pack_meta(m["plan"], n, input_kind="u8", c2={52: "32x4"}))
    kept = dense8s.EncoderPair(*(dense8s.Dense8SEncoder(varied, dev.index or 0, n) for _ in range(2)))
    assert entries(kept.programs()[0], 1) == {"d8s_dense"}
    given = [dense8s.Dense8SEncoder(pack, dev.index or 0, n, fused=encs[0].fused) for _ in range(2)]
    own = dense8s.EncoderPair(*given)
    assert own.programs()[0] is given[0].program and own.max_bands == given[0].max_bands
    fa, fb = own(x)
    assert torch.equal(fa, want) and torch.equal(fb, want)
    assert sum(e.sync_errors() for e in encs + given) == 0


def test_bands_unordered_runners(dev, odd_maps):
    """Four one-image runners with default kinds, each called from a stream of its own with nothing between
    them: every pass's features, and no wait runs out."""
    img = 288
    plan = odd_maps[img]["plan"]
    pack = dense8s.make_pack(plan, 1, input_kind="u8")
    encs = [dense8s.Dense8SEncoder(pack, dev.index or 0, 1) for _ in range(4)]
    assert encs[0].max_bands > 1
    print(f"unordered runners, kinds {encs[0].fused}", flush=True)
    xs = [odd_maps[img]["x"][k % 3:k % 3 + 1].contiguous() for k in range(4)]
    want = [odd_maps[img]["want"][k % 3:k % 3 + 1] for k in range(4)]
    for e in encs:
        e.capture(1)
    streams = [torch.cuda.Stream(dev) for _ in encs]
    torch.cuda.synchronize(dev)
    for rep in range(20):
        for e, x, st in zip(encs, xs, streams):
            with torch.cuda.stream(st):
                e(x)
    torch.cuda.synchronize(dev)
    for e, w in zip(encs, want):
        assert torch.equal(e.out[:1], w)
    assert sum(e.sync_errors() for e in encs) == 0


def test_parts_wait_error_surfaces(dev, c4):
    """A non-zero error word (planted by the host, as an expired wait would leave it) makes the pass's
    features NaN, reaches the host-mapped report, and makes the next call raise PartsWaitError, which
    clears it: the call after that is exact again.  The same under graph replay."""
    enc = dense8s.Dense8SEncoder(c4["pack"], dev.index or 0, 24, fused={0: "tile", 2: "parts", 3: "parts"})
    assert enc._checked and enc._report is not None
    for graphs in (False, True):
        if graphs:
            enc.capture(24)
        assert torch.equal(enc(c4["x"]).clone(), c4["want"])
        torch.cuda.synchronize(dev)
        enc._sync[2].fill_(3)
        bad = enc(c4["x"]).clone()
        torch.cuda.synchronize(dev)
        assert torch.isnan(bad).all(), graphs
        assert int(enc._report[0]) == 3, graphs
        with pytest.raises(dense8s.PartsWaitError):
            enc(c4["x"])
        assert int(enc._report[0]) == 0 and enc.sync_errors(clear=False) == 0
        assert torch.equal(enc(c4["x"]).clone(), c4["want"]), graphs
    assert enc.calls["graph"] >= 2
