"""The timed cases of this framework: what a user's program calls, at the sizes it calls it with.

A submission prepares each study's raw crops (`prep`), gathers and zooms its windows (`tta`), encodes
them with one or two weight seeds (`dense8s`), and turns the window features into logits (`head`); a
caller of the C ABI runs single dense layers.  `listed()` names one case per way these are used,
`draw(rng)` gives further ones of the same ranges, `prepare` / `run` are the program around one call,
`work` what the call cannot do without, `exact` its result in 64 bits and `tolerance` how far a correct
implementation may be from another.

The encoders are DenseNet169 with seeded weights, calibrated once on the host (the weights are a
user's fixed model, so they do not depend on a case's seed; its images do).
"""
from __future__ import annotations

import ctypes
from functools import lru_cache

import numpy as np
import torch
import torch.nn.functional as F

import __graft_entry__

__graft_entry__.load_package()
from rsna_knee_efficiency_amd import dense8s, densenet, head, hip, prep, tta  # noqa: E402

DEV = "cuda:0"
MEAN, STD = 0.5, 0.25
FEATURES, SLOTS, PER_SLOT, CONTEXT, FINDINGS = 1664, 8, 11, 256, 12
BLOCK_LAYERS = (6, 12, 32, 32)
CROPS_MM = (110.0, 150.0)


# --- the cases ----------------------------------------------------------------------------------
def listed() -> list[dict]:
    return [
        # one 24-slice study, uint8 slices, to its 8 logits: the latency of a single request
        dict(name="study512", path="encode", n=24, img=512, input="u8", flip="none", seeds=1, logits=8),
        # the two weight seeds of the final model over two crops of 24 slices with flip-TTA: throughput
        dict(name="ensemble512_tta", path="encode", n=96, img=512, input="u8", flip="tta", seeds=2, logits=0),
        # a study of 88 windows at 288 px, already normalised to fp16 by the caller
        dict(name="study288", path="encode", n=88, img=288, input="f16", flip="none", seeds=1, logits=0),
        # the 11 windows of one slot: the smallest call a serving loop makes
        dict(name="slot288", path="encode", n=11, img=288, input="f16", flip="none", seeds=1, logits=0),
        # a side whose maps (104, 52, 26, 13) fit no power of two, an odd batch, mirrored images
        dict(name="odd416", path="encode", n=37, img=416, input="u8", flip="mirror", seeds=1, logits=0),
        # one dense layer (1x1 then 3x3) through the C ABI, batch 24
        dict(name="layer64", path="layer", n=24, h=64, w=64, c0=128, c=320),
        # the head over 8 studies of 88 windows, and over a single study of 44
        dict(name="head8x88", path="head", b=8, windows=88),
        dict(name="head1x44", path="head", b=1, windows=44),
        # a study's four series at two crops each, 24 slices (0..22 read): raw uint16 to uint8 volume
        dict(name="prep512", path="prep", img=512, slices=24, read=23,
             series="0.3125:1 0.2:1 0.45:1 0.35:0.9"),
        # stacks a caller has already resized to float32
        dict(name="float288", path="stacks", r=8, k=24, img=288),
        # the zoom view of a study's windows, gathered from its uint8 volume
        dict(name="zoom512", path="windows", b=1, k=24, windows=88, h=512, w=512,
             scale=1.1, tx=0.0, ty=0.0),
        # the same view of fp16 windows the caller already holds
        dict(name="view288", path="view", b=1, windows=88, h=288, w=288, scale=1.1, tx=0.0, ty=0.0),
    ]


def _log_int(rng, lo: int, hi: int) -> int:
    return int(round(lo * (hi / lo) ** rng.random()))


def draw(rng) -> dict:
    path = rng.choice(("encode", "encode", "encode", "layer", "head", "prep", "stacks", "windows", "view"))
    if path == "encode":
        flip = rng.choice(("none", "none", "mirror", "tta"))
        n = _log_int(rng, 1, 96)
        return dict(path=path, n=n + n % 2 if flip == "tta" else n, img=32 * rng.randint(3, 16),
                    input=rng.choice(("u8", "u8", "f16")), flip=flip, seeds=1,
                    logits=rng.choice((0, 0, 8)))
    if path == "layer":
        h = _log_int(rng, 7, 128)
        g0 = rng.choice((2, 4, 8, 20))
        return dict(path=path, n=_log_int(rng, 1, 96), h=h, w=rng.choice((h, h, h, rng.randint(7, 128))),
                    c0=32 * g0, c=32 * (g0 + rng.randint(0, 31)))
    if path == "head":
        return dict(path=path, b=_log_int(rng, 1, 16), windows=rng.randint(8, 128))
    if path == "prep":
        m = rng.randint(1, 4)
        return dict(path=path, img=32 * rng.randint(4, 16), slices=24, read=rng.choice((23, 24)),
                    series=" ".join(f"{rng.uniform(0.2, 0.6):.4f}:{rng.choice((1, 1, 0.9, 0.75))}"
                                    for _ in range(m)))
    if path == "stacks":
        return dict(path=path, r=rng.randint(1, 16), k=rng.randint(3, 32), img=8 * rng.randint(8, 64))
    h = _log_int(rng, 64, 512)
    w = h if rng.random() < 0.7 else _log_int(rng, 64, 512)
    scale, tx, ty = rng.choice(((1.1, 0.0, 0.0), (1.2, 0.03, -0.02), (0.9, 0.0, 0.05), (1.0, 0.02, 0.0)))
    if path == "windows" and rng.random() < 0.25:
        scale, tx, ty = 1.0, 0.0, 0.0            # the gather alone
    case = dict(path=path, b=1, windows=_log_int(rng, 4, 88), h=h, w=w, scale=scale, tx=tx, ty=ty)
    return dict(case, k=24) if path == "windows" else case


# --- inputs -------------------------------------------------------------------------------------
def _gen(seed: int) -> torch.Generator:
    return torch.Generator(device=DEV).manual_seed(int(seed))


def _field(k: int, h: int, w: int, g: torch.Generator) -> torch.Tensor:
    """(k, h, w) float32 in about -1 .. 1: blobs drifting from slice to slice, as anatomy does."""
    def u(lo, hi, *shape):
        return lo + (hi - lo) * torch.rand(shape, generator=g, device=DEV)
    z = torch.arange(k, device=DEV).view(-1, 1)
    cy, cx, sig, amp = u(0, 1, 12), u(0, 1, 12), u(0.05, 0.25, 12), u(-1, 1, 12)
    dy, dx = u(-0.01, 0.01, 12), u(-0.01, 0.01, 12)
    ys, xs = torch.arange(h, device=DEV) / h, torch.arange(w, device=DEV) / w
    gy = amp * torch.exp(-((ys.view(1, -1, 1) - (cy + z * dy).unsqueeze(1)) / sig) ** 2 / 2)
    gx = torch.exp(-((xs.view(1, -1, 1) - (cx + z * dx).unsqueeze(1)) / sig) ** 2 / 2)
    f = torch.bmm(gy, gx.transpose(1, 2).contiguous())
    return f / f.abs().amax().clamp_min(1e-6)


def _slices_u8(k: int, h: int, w: int, g: torch.Generator) -> torch.Tensor:
    noise = torch.rand((k, h, w), generator=g, device=DEV) * 80 - 40
    return (128 + 90 * _field(k, h, w, g) + noise).round_().clamp_(0, 255).to(torch.uint8)


def _images(n: int, img: int, kind: str, g: torch.Generator) -> torch.Tensor:
    """n windows of 3 neighbouring slices each, as uint8 or as normalised fp16."""
    vol = _slices_u8(n + 2, img, img, g)
    x = torch.stack([vol[:n], vol[1:n + 1], vol[2:]], 1).contiguous()
    return x if kind == "u8" else ((x.float() / 255 - MEAN) / STD).half()


@lru_cache(maxsize=None)
def _model(weights: int):
    """A DenseNet169 and its calibration, both made on the host from the weight seed."""
    model = densenet.seeded_densenet169(weights)
    g = torch.Generator().manual_seed(77)
    smooth = F.interpolate(torch.randn((4, 3, 8, 8), generator=g), size=(256, 256), mode="bicubic")
    x = (smooth / 2 + torch.rand(smooth.shape, generator=g) - 0.5).clamp(-2, 2)
    with torch.no_grad():
        return model, dense8s.calibrate(model, [x])


@lru_cache(maxsize=None)
def _tables(weights: int, img: int) -> tuple:
    model, cal = _model(weights)
    plan = dense8s.make_plan(model, cal, img)
    return plan, dense8s.pack_params(plan)


def _pack(weights: int, case: dict) -> dict:
    plan, par = _tables(weights, case["img"])
    mean, std = ((MEAN,) * 3, (STD,) * 3) if case["input"] == "u8" else ((0.0,) * 3, (1.0,) * 3)
    meta = dense8s.pack_meta(plan, case["n"], input_kind=case["input"], mean=mean, std=std)
    return {"meta": meta, "engines": {}, "par": par, "cubin": None}


def _logit_weights(k: int) -> tuple:
    rng = np.random.default_rng(5)
    return rng.normal(0, FEATURES ** -0.5, (k, FEATURES)), rng.normal(0, 0.1, k)


@lru_cache(maxsize=None)
def _head_weights() -> dict:
    g = torch.Generator().manual_seed(9)

    def lin(*shape):
        return torch.randn(shape, generator=g) / shape[-1] ** 0.5

    def vec(n, mean=0.0, s=0.02):
        return mean + s * torch.randn((n,), generator=g)

    d, c, t = FEATURES, CONTEXT, FINDINGS
    L = "ctx.layers.0."
    return {"slot_emb": 0.02 * torch.randn((SLOTS, d), generator=g), "ctx_in.weight": lin(c, d),
            "ctx_in.bias": vec(c), "ctx_pos": 0.02 * torch.randn((PER_SLOT, c), generator=g),
            L + "self_attn.in_proj_weight": lin(3 * c, c), L + "self_attn.in_proj_bias": vec(3 * c),
            L + "self_attn.out_proj.weight": lin(c, c), L + "self_attn.out_proj.bias": vec(c),
            L + "linear1.weight": lin(2 * c, c), L + "linear1.bias": vec(2 * c),
            L + "linear2.weight": lin(c, 2 * c), L + "linear2.bias": vec(c),
            L + "norm1.weight": vec(c, 1.0, 0.1), L + "norm1.bias": vec(c),
            L + "norm2.weight": vec(c, 1.0, 0.1), L + "norm2.bias": vec(c),
            "ctx_out.weight": lin(d, c), "ctx_out.bias": vec(d), "attn.weight": lin(t, d),
            "attn.bias": vec(t), "cls_w": lin(t, d), "cls_b": vec(t)}


def _head_inputs(case: dict, seed: int) -> tuple:
    g = _gen(seed)
    b, w = case["b"], case["windows"]
    z = 0.7 * torch.randn((b, w, FEATURES), generator=g, device=DEV).abs()   # pooled ReLU features
    slot_of = (torch.arange(w) // PER_SLOT) % SLOTS
    mask = torch.rand((b, SLOTS), generator=g, device=DEV) < 0.9             # most studies lack a series
    mask[:, 0] = True
    return z, slot_of, mask


def _layer_inputs(case: dict, seed: int) -> dict:
    """A dense layer as the encoder's plan makes it: the store's channels at full int8 range, BatchNorm
    prologue in fp16, weights quantised per output channel, epilogues calibrated to the data."""
    g = _gen(seed)
    n, hw, c, c0 = case["n"], case["h"] * case["w"], case["c"], case["c0"]
    G, G0 = c // 32, c0 // 32

    def q8(*shape):
        x = torch.randn(shape, generator=g, device=DEV)
        return (x * (127 / 4.5)).round_().clamp_(-127, 127).to(torch.int8)

    def wq(*shape):
        return (torch.randn(shape, generator=g, device=DEV) * 36).round_().clamp_(-127, 127).to(torch.int8)

    a = (0.8 + 0.4 * torch.rand((c,), generator=g, device=DEV)) * (4.5 / 127) / 4.5
    b = 0.05 * torch.randn((c,), generator=g, device=DEV)
    abh = torch.stack([a.view(-1, 2), b.view(-1, 2)], 1).half().reshape(-1, 4).contiguous()
    w1 = wq(G, 128, 32)
    w2 = wq(4, 9, 32, 32)
    gd = torch.stack([(0.8 + 0.4 * torch.rand((128,), generator=g, device=DEV)) / (255 * 36 * c ** 0.5),
                      0.2 + 0.05 * torch.randn((128,), generator=g, device=DEV)], 1).contiguous()
    sc = (0.8 + 0.4 * torch.rand((32,), generator=g, device=DEV)) * (127 / (4 * 110 * 36 * 1152 ** 0.5))
    return dict(in0=q8(n, G0, hw, 32), seg=q8(max(G - G0, 1), n, hw, 32), w1=w1, abh=abh, gd=gd,
                w1sum=w1.int().sum((0, 2)).int(), w2=w2, sc=sc.float().contiguous(),
                w2sum=w2.int().sum((0, 1, 3)).int(),
                bott=torch.empty((4, n * hw, 32), dtype=torch.uint8, device=DEV),
                out=torch.empty((n, hw, 32), dtype=torch.int8, device=DEV))


def _series(case: dict) -> list:
    """(pixel spacing in mm, columns per row) of each of the study's series."""
    return [tuple(float(v) for v in s.split(":")) for s in case["series"].split()]


def _payload(case: dict, seed: int) -> dict:
    """One study's raw crops: MRI-like fields on a zero background, cropped to the larger box."""
    g = _gen(seed)
    k = case["slices"]
    raws, rescs, meta, off = [], [], [], 0
    for j, (ps, aspect) in enumerate(_series(case)):
        rows = int(round(max(CROPS_MM) / ps))
        cols = int(round(rows * aspect))
        ys = torch.linspace(-1, 1, rows, device=DEV).view(-1, 1)
        xs = torch.linspace(-1, 1, cols, device=DEV).view(1, -1)
        body = ys ** 2 + (xs / 0.85) ** 2 < 0.8
        v = 600 + 400 * _field(k, rows, cols, g) + 60 * torch.randn((k, rows, cols), generator=g, device=DEV)
        raws.append(torch.where(body, v.round_().clamp_(0, 4095), torch.zeros_like(v)).to(torch.int16).view(-1))
        row = np.zeros(prep.N_META, np.int64)
        row[prep.M_SLOT], row[prep.M_MODE], row[prep.M_K] = j, prep.MODE_GPU, k
        row[prep.M_HR], row[prep.M_WR], row[prep.M_RAW_OFF], row[prep.M_FLIP] = rows, cols, off, j % 3
        row[prep.M_RESC] = -1
        if j % 2:
            row[prep.M_RESC] = k * len(rescs)
            rescs.append(torch.tensor([[1.2265625 - 0.25 * j, 13.25 * j - 18]], dtype=torch.float64).repeat(k, 1))
        for s, mm in enumerate(CROPS_MM):
            h, w = min(int(round(mm / ps)), rows), min(int(round(mm / ps)), cols)
            y0, x0 = (rows - h) // 2, (cols - w) // 2
            row[prep.M_BOX + 4 * s: prep.M_BOX + 4 * s + 4] = (y0, y0 + h, x0, x0 + w)
        meta.append(row)
        off += k * rows * cols
    return {"raw": torch.cat(raws), "u8": torch.empty(0, dtype=torch.uint8, device=DEV),
            "resc": (torch.cat(rescs) if rescs else torch.empty((0, 2), dtype=torch.float64)).to(DEV),
            "meta": np.stack(meta)}


def _float_stacks(case: dict, seed: int) -> torch.Tensor:
    g = _gen(seed)
    r, k, img = case["r"], case["k"], case["img"]
    x = torch.stack([_field(k, img, img, g) for _ in range(r)])
    x = 500 + 400 * x + 50 * torch.randn(x.shape, generator=g, device=DEV)
    return x.clamp_(min=0).contiguous()          # the air around the knee reads as zero


def _window_inputs(case: dict, seed: int) -> tuple:
    g = _gen(seed)
    s, k, m = SLOTS, case["k"], case["windows"]
    vol = _slices_u8(case["b"] * s * k, case["h"], case["w"], g).view(case["b"], s, k, case["h"], case["w"])
    first = (torch.arange(m) // PER_SLOT % s) * k + torch.arange(m) % PER_SLOT * 2
    return vol, torch.stack([first, first + 1, first + 2], 1).reshape(-1).to(DEV)


def _view_inputs(case: dict, seed: int) -> torch.Tensor:
    n = case["b"] * case["windows"]
    vol = _slices_u8(n + 2, case["h"], case["w"], _gen(seed)).half() / 255
    return torch.stack([vol[:n], vol[1:n + 1], vol[2:]], 1).view(case["b"], case["windows"], 3, case["h"], case["w"])


# --- the program around a call ------------------------------------------------------------------
FLIPS = {"none": False, "mirror": True, "tta": "tta"}


def prepare(case: dict, seed: int) -> dict:
    st = {"case": case}
    path = case["path"]
    if path == "encode":
        flip = FLIPS[case["flip"]]
        n_in = case["n"] // 2 if flip == "tta" else case["n"]
        st["encs"] = [dense8s.Dense8SEncoder(_pack(w, case), 0, case["n"]) for w in range(case["seeds"])]
        for e in st["encs"]:
            e.capture(n_in, flip)
        st["x"], st["flip"] = _images(n_in, case["img"], case["input"], _gen(seed)), flip
        if case["logits"]:
            st["head"] = head.LinearHead(*_logit_weights(case["logits"]), DEV)
    elif path == "layer":
        st |= _layer_inputs(case, seed)
        p = {k: v.data_ptr() for k, v in st.items() if isinstance(v, torch.Tensor)}
        n, h, w = case["n"], case["h"], case["w"]
        st["c1"] = hip.GemmArgs(p["in0"], p["seg"], p["w1"], p["abh"], p["gd"], p["w1sum"], p["bott"],
                                case["c0"] // 32, case["c"] // 32, n, h * w, w, n * h * w, 128, 0)
        st["c2"] = hip.Conv2Args(p["bott"], p["w2"], p["sc"], p["w2sum"], p["out"], n, h, w, 0)
    elif path == "head":
        st["head"] = head.KneeHead(_head_weights(), DEV)
        st["z"], st["slot_of"], st["mask"] = _head_inputs(case, seed)
    elif path == "prep":
        st["payload"] = _payload(case, seed)
        st["spec"] = prep.PrepSpec(img=case["img"], slices=case["slices"], n_seq=len(_series(case)),
                                   n_scales=len(CROPS_MM))
    elif path == "stacks":
        st["x"] = _float_stacks(case, seed)
    elif path == "windows":
        st["vol"], st["idx"] = _window_inputs(case, seed)
        st["buf"] = torch.empty((case["b"] * case["windows"], 3, case["h"], case["w"]), dtype=torch.float16,
                                device=DEV)
    else:
        st["x"] = _view_inputs(case, seed)
    return st


def run(st: dict):
    case = st["case"]
    path = case["path"]
    if path == "encode":
        if case["seeds"] > 1:
            return dense8s.encode_concurrent([(e, st["x"], st["flip"]) for e in st["encs"]])
        f = st["encs"][0](st["x"], flip=st["flip"])
        return (f, st["head"](f)) if case["logits"] else f
    if path == "layer":
        stream = torch.cuda.current_stream().cuda_stream
        hip.call("d8s_conv1", ctypes.byref(st["c1"]), ctypes.c_void_p(stream))
        hip.call("d8s_conv2", ctypes.byref(st["c2"]), ctypes.c_void_p(stream))
        return st["bott"], st["out"]
    if path == "head":
        return st["head"](st["z"], st["slot_of"], st["mask"])
    if path == "prep":
        return prep.payloads_to_uint8([st["payload"]], st["spec"], DEV, read_slices=(0, case["read"]))
    if path == "stacks":
        return prep.to_uint8_hist_batch(st["x"])
    if path == "windows":
        tta.windows_u8(st["vol"], st["idx"], st["buf"], case["scale"], case["tx"], case["ty"])
        return st["buf"]
    return tta.affine_windows(st["x"], case["scale"], case["tx"], case["ty"])


# --- what a pass cannot do without --------------------------------------------------------------
def work(case: dict) -> dict:
    path = case["path"]
    if path == "encode":
        n, img, side, c = case["n"], case["img"], case["img"] // 4, 64
        macs, wts = n * 64 * 147 * (img // 2) ** 2, 64 * 147 * 2
        for b, layers in enumerate(BLOCK_LAYERS):
            for _ in range(layers):
                macs += n * side * side * (128 * c + 1152 * 32)
                wts += 128 * c + 1152 * 32
                c += 32
            if b < 3:
                side, c = side // 2, c // 2
                macs += n * side * side * c * 2 * c              # pooled first
                wts += 2 * c * c
        n_in = n // 2 if case["flip"] == "tta" else n
        moved = n_in * 3 * img * img * (1 if case["input"] == "u8" else 2)
        return {"bytes": moved + case["seeds"] * (wts + n * FEATURES * 4), "flops": 2 * macs * case["seeds"]}
    if path == "layer":
        m, c = case["n"] * case["h"] * case["w"], case["c"]
        return {"bytes": m * (c + 128 + 32) + 128 * c + 36864, "flops": 2 * m * (128 * c + 36864)}
    if path == "head":
        b, w, d, c, t = case["b"], case["windows"], FEATURES, CONTEXT, FINDINGS
        wts = 2 * d * c + 4 * c * c + 4 * c * c + 2 * t * d + SLOTS * d
        macs = b * w * (2 * d * c + 8 * c * c + 2 * w * c + 2 * t * d)
        return {"bytes": 4 * (b * w * d + wts + b * t), "flops": 2 * macs}
    if path == "prep":
        n_in = n_out = 0
        for ps, aspect in _series(case):
            rows = int(round(max(CROPS_MM) / ps))
            n_in += case["read"] * rows * int(round(rows * aspect))
            n_out += len(CROPS_MM) * case["slices"] * case["img"] ** 2
        return {"bytes": 2 * n_in + n_out, "flops": 9 * n_out}
    if path == "stacks":
        n = case["r"] * case["k"] * case["img"] ** 2
        return {"bytes": 5 * n, "flops": 2 * n}
    n = case["b"] * case["windows"] * 3 * case["h"] * case["w"]
    if path == "windows":
        src = case["b"] * len(set(_slice_set(case))) * case["h"] * case["w"]
        return {"bytes": src + 2 * n, "flops": 8 * n}
    return {"bytes": 4 * n, "flops": 8 * n}


def _slice_set(case: dict) -> list:
    firsts = [(m // PER_SLOT % SLOTS) * case["k"] + m % PER_SLOT * 2 for m in range(case["windows"])]
    return [f + i for f in firsts for i in range(3)]


# --- tolerances ---------------------------------------------------------------------------------
def tolerance(case: dict):
    """Integer and byte paths are the same in any order of summation.  The encoder's int32 sums are
    exact too; its stem's fp32 sums are not, and a byte that flips there travels through the layers:
    about four times the distance of the present features from `exact` (1e-3 to 2e-3).  The head is
    float32 throughout (1e-7 from `exact`)."""
    path = case["path"]
    if path in ("layer", "prep", "stacks"):
        return "exact"
    if path == "encode":
        return {"rel": 8e-3}
    if path == "head":
        return {"rel": 1e-6}
    return {"rel": 1e-3, "max": 2e-3}            # one rounding to fp16, bilinear weights in fp32


# --- the results in 64 bits ---------------------------------------------------------------------
def _f64(a) -> torch.Tensor:
    t = torch.from_numpy(np.ascontiguousarray(a)) if isinstance(a, np.ndarray) else a
    return t.to(DEV).double()


def _round_fp16(t: torch.Tensor) -> torch.Tensor:
    """The nearest fp16 value in one rounding (a conversion through float32 could round twice)."""
    _, e = torch.frexp(t)
    ulp = torch.ldexp(torch.ones_like(t), (e - 11).clamp_min(-24))
    return torch.round(t / ulp) * ulp


def _prologue(x: torch.Tensor, abh) -> torch.Tensor:
    h = torch.as_tensor(abh).cpu().contiguous().view(torch.float16).double().to(DEV).view(-1, 2, 2)
    a, b = h[:, 0].reshape(-1, 1), h[:, 1].reshape(-1, 1)
    return torch.round(_round_fp16(a * x + b).clamp(0, 1) * 255)


def _conv1(u: torch.Tensor, w1, gd) -> torch.Tensor:
    w = _f64(w1).permute(1, 0, 2).reshape(128, -1)               # [G][128][32] -> [128][C]
    g = _f64(gd)
    return torch.round((g[:, :1] * (w @ u) + g[:, 1:]).clamp(0, 1) * 255)


def _conv2(v: torch.Tensor, w2, sc, h: int, w: int) -> torch.Tensor:
    """v [n][128][h * w] -> [n][32][h * w]; the weights are [block][tap][output][input]."""
    wt = _f64(w2).permute(1, 2, 0, 3).reshape(9, 32, 128)
    p = F.pad(v.view(-1, 128, h, w), (1, 1, 1, 1))
    acc = 0
    for t in range(9):
        acc = acc + wt[t] @ p[:, :, t // 3:t // 3 + h, t % 3:t % 3 + w].reshape(-1, 128, h * w)
    return torch.round((acc * _f64(sc).view(-1, 1)).clamp(-127, 127))


def _exact_encoder(weights: int, case: dict, x: torch.Tensor) -> torch.Tensor:
    """Features (n, 1664): the int8 network with every sum and product in 64 bits (the roundings to
    fp16, u8 and int8 are the network's own)."""
    _, par = _tables(weights, case["img"])
    s = case["img"] // 4
    if case["input"] == "u8":
        lut = ((torch.arange(256, dtype=torch.float64) / 255 - MEAN) / STD).numpy().astype(np.float16)
        x = _f64(lut)[x.long()]
    x = x.double()
    w16 = _f64(np.ascontiguousarray(par["S_w16"]).view(np.float16)).view(64, 3, 7, 8)[..., 1:].reshape(64, 147)
    cols = F.unfold(x.float(), 7, padding=3, stride=2).double()  # copies only: fp16 values, exact
    y = ((w16 @ cols + _f64(par["S_bias"]).view(-1, 1)).clamp_min(0) * _f64(par["S_inv"]).view(-1, 1))
    y = torch.round(y.clamp(max=127)).view(-1, 64, 2 * s, 2 * s)
    store = F.max_pool2d(y.float(), 3, 2, 1).double().view(-1, 64, s * s)
    for b, layers in enumerate(BLOCK_LAYERS):
        for li in range(layers):
            t = f"L{b}_{li}_"
            v = _conv1(_prologue(store, par[t + "abh"]), par[t + "w1"], par[t + "gdu"])
            store = torch.cat([store, _conv2(v, par[t + "w2k"], par[t + "c2u"], s, s)], 1)
        if b < 3:
            u = _prologue(store, par[f"T{b}_abh"]).view(-1, store.shape[1], s // 2, 2, s // 2, 2).sum((3, 5))
            w = _f64(par[f"T{b}_w"]).permute(1, 0, 2).reshape(store.shape[1] // 2, -1)
            s //= 2
            acc = w @ u.view(-1, store.shape[1], s * s) / 4
            store = torch.round((acc * _f64(par[f"T{b}_gdf"])[:, :1]).clamp(-127, 127))
    ab = _f64(par["F_ab"])
    return (ab[:, :1] * store + ab[:, 1:]).clamp_min(0).mean(2)


def _exact_encode(case: dict, seed: int):
    flip = case["flip"]
    x = _images(case["n"] // 2 if flip == "tta" else case["n"], case["img"], case["input"], _gen(seed))
    if flip != "none":
        x = torch.cat([x, x.flip(3)]) if flip == "tta" else x.flip(3)
    step = max(1, 8 * 512 * 512 // case["img"] ** 2)
    outs = [torch.cat([_exact_encoder(w, case, c) for c in x.split(step)]) for w in range(case["seeds"])]
    if case["seeds"] > 1:
        return outs
    if not case["logits"]:
        return outs[0]
    w, b = (_f64(v.astype(np.float32)) for v in _logit_weights(case["logits"]))
    return outs[0], outs[0] @ w.t() + b


def _exact_layer(case: dict, seed: int):
    t = _layer_inputs(case, seed)
    n, h, w, c = case["n"], case["h"], case["w"], case["c"]
    bott = torch.empty((4, n, h * w, 32), dtype=torch.float64, device=DEV)
    out = torch.empty((n, h * w, 32), dtype=torch.float64, device=DEV)
    for i in range(n):
        groups = [t["in0"][i]] + ([t["seg"][:, i]] if c > case["c0"] else [])
        x = torch.cat(groups).double().permute(0, 2, 1).reshape(c, h * w)
        v = _conv1(_prologue(x, t["abh"]), t["w1"], t["gd"])
        bott[:, i] = v.view(4, 32, -1).transpose(1, 2)
        out[i] = _conv2(v.unsqueeze(0), t["w2"], t["sc"], h, w)[0].t()
    return bott.view(4, n * h * w, 32), out


def _exact_head(case: dict, seed: int) -> torch.Tensor:
    p = {k: v.to(DEV).double() for k, v in _head_weights().items()}
    z, slot_of, mask = _head_inputs(case, seed)
    slot_of = slot_of.to(DEV)
    b, w, heads = case["b"], case["windows"], CONTEXT // 64
    f = z.double() + p["slot_emb"][slot_of]
    valid = mask[:, slot_of]
    L = "ctx.layers.0."

    def linear(x, name):
        return x @ p[name + ".weight"].t() + p[name + ".bias"]

    def norm(x, name):
        return F.layer_norm(x, (CONTEXT,), p[name + ".weight"], p[name + ".bias"])

    h = linear(f, "ctx_in") + p["ctx_pos"][torch.arange(w, device=DEV) % PER_SLOT]
    qkv = norm(h, L + "norm1") @ p[L + "self_attn.in_proj_weight"].t() + p[L + "self_attn.in_proj_bias"]
    q, k, v = qkv.view(b, w, 3, heads, 64).permute(2, 0, 3, 1, 4)
    s = (q / 8) @ k.transpose(-1, -2)
    keep = valid | ~valid.any(1, keepdim=True)
    s = s.masked_fill(~keep[:, None, None, :], float("-inf")).softmax(-1)
    h = h + linear((s @ v).transpose(1, 2).reshape(b, w, CONTEXT), L + "self_attn.out_proj")
    h = h + linear(linear(norm(h, L + "norm2"), L + "linear1").clamp_min(0), L + "linear2")
    f = f + linear(h, "ctx_out")
    a = linear(f, "attn").masked_fill(~keep[:, :, None], float("-inf")).softmax(1)
    return ((a.transpose(1, 2) @ f) * p["cls_w"]).sum(-1) + p["cls_b"]


def _area_matrix(n_in: int, n_out: int) -> torch.Tensor:
    """Each output's share of the source cells it covers (INTER_AREA)."""
    r = n_in / n_out
    lo = torch.arange(n_out, dtype=torch.float64, device=DEV).view(-1, 1) * r
    cell = torch.arange(n_in, dtype=torch.float64, device=DEV)
    cover = (torch.minimum(lo + r, cell + 1) - torch.maximum(lo, cell)).clamp_min(0)
    return cover / cover.sum(1, keepdim=True)


def _resize(x: torch.Tensor, img: int) -> torch.Tensor:
    h, w = x.shape[1:]
    if (h, w) == (img, img):
        return x
    if h > img:
        return _area_matrix(h, img) @ x @ _area_matrix(w, img).t()
    return F.interpolate(x.unsqueeze(0), size=(img, img), mode="bilinear", align_corners=False)[0]


def _to_u8(x: torch.Tensor) -> torch.Tensor:
    s, _ = x.reshape(-1).sort()
    ends = []
    for p in (0.01, 0.99):
        v = (s.numel() - 1) * p
        ends.append(s[int(v)] + (s[int(v) + 1] - s[int(v)]) * (v - int(v)))
    lo, hi = ends
    return ((x - lo) * (255 / (hi - lo))).clamp(0, 255).floor() if hi > lo else torch.zeros_like(x)


def _exact_prep(case: dict, seed: int) -> torch.Tensor:
    pay = _payload(case, seed)
    k, img, m = case["slices"], case["img"], len(_series(case))
    vol = torch.zeros((1, len(CROPS_MM) * m, k, img, img), dtype=torch.float64, device=DEV)
    for j, row in enumerate(pay["meta"]):
        hr, wr, off = (int(row[i]) for i in (prep.M_HR, prep.M_WR, prep.M_RAW_OFF))
        x = pay["raw"][off:off + k * hr * wr].view(k, hr, wr).double()
        if row[prep.M_RESC] >= 0:
            r = pay["resc"][int(row[prep.M_RESC])].float().double()
            x = x * r[0] + r[1]
        flip = int(row[prep.M_FLIP])
        a, z = (k - case["read"], k) if flip == prep.FLIP_SLICES else (0, case["read"])
        for s in range(len(CROPS_MM)):
            y0, y1, x0, x1 = (int(v) for v in row[prep.M_BOX + 4 * s: prep.M_BOX + 4 * s + 4])
            u = torch.zeros((k, img, img), dtype=torch.float64, device=DEV)
            u[a:z] = _to_u8(_resize(x[a:z, y0:y1, x0:x1], img))
            vol[0, j + s * m] = u.flip(2) if flip == prep.FLIP_X else u.flip(0) if flip == prep.FLIP_SLICES else u
    return vol


def _exact_view(x: torch.Tensor, case: dict) -> torch.Tensor:
    """x (N, 1, h, w) float64; the grid is the view's own, in fp16."""
    if (case["scale"], case["tx"], case["ty"]) == (1.0, 0.0, 0.0):
        return x
    theta = torch.tensor([[[1 / case["scale"], 0, -2 * case["tx"]], [0, 1 / case["scale"], -2 * case["ty"]]]],
                         device=DEV, dtype=torch.float16)
    grid = F.affine_grid(theta, (1, 1, case["h"], case["w"]), align_corners=False).double()
    return F.grid_sample(x.view(1, -1, case["h"], case["w"]), grid, align_corners=False)


def exact(case: dict, seed: int):
    path = case["path"]
    if path == "encode":
        return _exact_encode(case, seed)
    if path == "layer":
        return _exact_layer(case, seed)
    if path == "head":
        return _exact_head(case, seed)
    if path == "prep":
        return _exact_prep(case, seed)
    if path == "stacks":
        return torch.stack([_to_u8(s) for s in _float_stacks(case, seed).double()])
    if path == "windows":
        vol, idx = _window_inputs(case, seed)
        lut = (torch.arange(256, device=DEV).half() * (1 / 255)).double()
        x = lut[vol.view(case["b"], -1, case["h"], case["w"])[:, idx].long()]
        return _exact_view(x, case).view(-1, 3, case["h"], case["w"])
    x = _view_inputs(case, seed)
    return _exact_view(x.double(), case).view(x.shape)
