"""The geometric TTA view (`d8s_grid_sample`): bit for bit against the reference's own operations on
the same GPU (`F.affine_grid` + `F.grid_sample` in fp16, src/knee/tta.py:131-148, and the uint8
gather through the u / 255 table, src/knee/infer.py:986-1012), and within fp16 rounding of a float64
bilinear restatement on the CPU."""
from __future__ import annotations

import numpy as np
import pytest
import torch
import torch.nn.functional as F

from rsna_knee_efficiency_amd import tta

pytestmark = pytest.mark.gpu

VIEWS = [(1.10, 0.0, 0.0), (0.95, 0.0, 0.0), (1.05, 0.0, 0.0), (1.0, 0.03, 0.0), (1.0, 0.0, -0.03),
         (1.10, 0.03, -0.03)]


def _reference(w: torch.Tensor, scale: float, tx: float, ty: float) -> torch.Tensor:
    """src/knee/tta.py:131-148 as torch operations."""
    b, k, d, h, wd = w.shape
    x = w.reshape(b * k, d, h, wd)
    theta = torch.tensor([[1.0 / scale, 0.0, -2.0 * tx], [0.0, 1.0 / scale, -2.0 * ty]],
                         device=x.device, dtype=x.dtype).unsqueeze(0)
    grid = F.affine_grid(theta, (1, d, h, wd), align_corners=False).expand(b * k, h, wd, 2)
    x = F.grid_sample(x, grid, mode="bilinear", padding_mode="zeros", align_corners=False)
    return x.reshape(b, k, d, h, wd)


def _bilinear_f64(img: np.ndarray, grid: np.ndarray) -> np.ndarray:
    """Bilinear sampling with zero padding, align_corners=False, in float64 (grid given)."""
    h, w = img.shape
    ix = ((grid[..., 0].astype(np.float64) + 1) * w - 1) / 2
    iy = ((grid[..., 1].astype(np.float64) + 1) * h - 1) / 2
    x0, y0 = np.floor(ix).astype(int), np.floor(iy).astype(int)
    out = np.zeros(ix.shape)
    for dy in (0, 1):
        for dx in (0, 1):
            xx, yy = x0 + dx, y0 + dy
            wgt = (1 - np.abs(ix - xx)) * (1 - np.abs(iy - yy))
            ok = (xx >= 0) & (xx < w) & (yy >= 0) & (yy < h)
            out += np.where(ok, img[np.clip(yy, 0, h - 1), np.clip(xx, 0, w - 1)], 0.0) * wgt
    return out


@pytest.mark.parametrize("view", VIEWS, ids=[f"s{v[0]}_tx{v[1]}_ty{v[2]}" for v in VIEWS])
def test_affine_windows_is_the_reference_on_the_gpu(dev, view):
    print(f"view {view}", flush=True)
    g = torch.Generator().manual_seed(3)
    w = torch.rand((2, 3, 3, 96, 80), generator=g).half().to(dev)
    got = tta.affine_windows(w, *view)
    ref = _reference(w, *view)
    diff = int((got != ref).sum())
    assert diff == 0, f"{diff} values differ, max {float((got.float() - ref.float()).abs().max())}"
    # and within fp16 rounding of the float64 restatement on the same (fp16) grid
    grid = tta.view_grid(96, 80, 3, *view, torch.float16, dev).float().cpu().numpy()
    want = _bilinear_f64(w[1, 2, 1].float().cpu().numpy(), grid)
    assert np.abs(got[1, 2, 1].float().cpu().numpy() - want).max() <= 2.0 ** -11 + 1e-6


def test_affine_windows_identity_and_full_size(dev):
    w = torch.rand((1, 11, 3, 512, 512), device=dev).half()
    assert tta.affine_windows(w) is w
    got = tta.affine_windows(w, 1.10)
    assert torch.equal(got, _reference(w, 1.10, 0.0, 0.0))


U8_SHAPES = [(64, 48), (40, 46), (512, 512)]


@pytest.mark.parametrize("view", [(1.0, 0.0, 0.0)] + VIEWS, ids=["identity"] + [f"s{v[0]}_tx{v[1]}_ty{v[2]}" for v in VIEWS])
@pytest.mark.parametrize("hw", U8_SHAPES, ids=[f"{h}x{w}" for h, w in U8_SHAPES])
def test_windows_u8_is_the_reference_chain(dev, view, hw):
    """gather_u8_f16 + affine_windows of the submission path (infer.py:986-1012) in one kernel: every
    view, on widths that take the four-pixel kernel (a multiple of 4, both its window path and its
    per-pixel path at the borders) and one that does not."""
    h, w = hw
    b, s, k = (2, 2, 7) if h < 512 else (1, 1, 9)
    print(f"windows_u8 view {view} {h}x{w}", flush=True)
    g = torch.Generator().manual_seed(5)
    v = torch.randint(0, 256, (b, s, k, h, w), generator=g, dtype=torch.uint8).to(dev)
    idx = torch.tensor([0, 1, 2, 2, 3, 4, 8, 9, 13] if s * k > 13 else [0, 1, 2, 2, 3, 4, 6, 7, 8],
                       dtype=torch.int64, device=dev)
    depth = 3
    out = torch.empty((b * idx.numel() // depth, depth, h, w), dtype=torch.float16, device=dev)
    tta.windows_u8(v, idx, out, *view)
    lut = torch.arange(256, dtype=torch.uint8, device=dev).half().mul_(1.0 / 255.0)
    x = lut[v.view(b, s * k, h, w).index_select(1, idx).long()].view(b * idx.numel() // depth, depth, h, w)
    if view != (1.0, 0.0, 0.0):
        x = _reference(x.view(-1, 1, depth, h, w), *view).view(-1, depth, h, w)
    assert torch.equal(out, x)


def test_lut_is_u_over_255():
    lut = tta.lut_u8_f16("cpu").float().numpy()
    u = np.arange(256) / 255.0
    assert np.abs(lut - u).max() <= 2.0 ** -12 and lut[0] == 0 and lut[255] == 1


@pytest.mark.parametrize("view", [(1.0, 0.0, 0.0), (1.10, 0.0, 0.0)])
def test_windows_u8_slice_checks(dev, view):
    """The slice indices are checked once per tensor and in-place version: a valid in-place change is
    seen, an index outside the volume raises; through the C ABI (no host check) such an index is
    clamped into the volume."""
    import ctypes
    from rsna_knee_efficiency_amd import hip
    b, s, k, h, w = 1, 2, 5, 32, 40
    g = torch.Generator().manual_seed(6)
    v = torch.randint(0, 256, (b, s, k, h, w), generator=g, dtype=torch.uint8).to(dev)
    idx = torch.tensor([0, 1, 2, 7, 8, 9], dtype=torch.int64, device=dev)
    out = torch.empty((2, 3, h, w), dtype=torch.float16, device=dev)
    a = tta.windows_u8(v, idx, out, *view).clone()
    idx[0] = 4                                     # in place, still inside the volume
    bb = tta.windows_u8(v, idx, out, *view).clone()
    assert torch.equal(a[1], bb[1]) and not torch.equal(a[0, 0], bb[0, 0])
    idx[0] = 10
    with pytest.raises(ValueError):
        tta.windows_u8(v, idx, out, *view)
    bad = torch.tensor([0, -1, 2, 10, 8, 9], dtype=torch.int64, device=dev)
    gp = 0 if view == (1.0, 0.0, 0.0) else tta.view_grid(h, w, 1, *view, torch.float16, dev).data_ptr()
    out2 = torch.full((2, 3, h, w), 7.0, dtype=torch.float16, device=dev)
    args = hip.GridArgs(src=v.data_ptr(), slice_idx=bad.data_ptr(), lut=tta.lut_u8_f16(dev).data_ptr(),
                        grid=gp, out=out2.data_ptr(), kind=1, N=6, H=h, W=w, B=1, SK=s * k, M=6)
    hip.call("d8s_grid_sample", ctypes.byref(args), ctypes.c_void_p(torch.cuda.current_stream(dev).cuda_stream))
    torch.cuda.synchronize(dev)
    clamped = torch.tensor([0, 0, 2, 9, 8, 9], dtype=torch.int64, device=dev)
    ref = torch.empty_like(out2)
    tta.windows_u8(v, clamped, ref, *view)
    assert torch.equal(out2, ref)


SHIFTED_VIEWS = [(1.5, 0.0, 0.0), (1.25, 0.11, -0.2), (0.8, 0.0, 0.05), (0.6, 0.0, 0.0), (1.0, 0.02, 0.0)]


@pytest.mark.parametrize("kind,view", [(1, (1.0, 0.0, 0.0))] + [(k, v) for k in (0, 1) for v in SHIFTED_VIEWS])
@pytest.mark.parametrize("h,w,off", [(5, 4, 0), (7, 8, 0), (9, 12, 0), (33, 64, 0), (33, 64, 1), (20, 61, 0), (3, 3, 1)])
def test_grid_sample_kernels_agree(dev, kind, h, w, off, view):
    """The four-pixel form's three paths (zoom in, zoom out, borders), narrow and odd images, images that
    start at an odd element (`off`: the one-pixel form, the gather's unaligned loads) and group remainders,
    through the C ABI: bit for bit torch's grid_sample (the table alone for the identity) on the same
    values, and nothing written around the output."""
    import ctypes
    from rsna_knee_efficiency_amd import hip
    n, sk = 19, 5
    print(f"grid kind={kind} {h}x{w} off={off} view={view}", flush=True)
    g = torch.Generator().manual_seed(h * w + off)
    lut = tta.lut_u8_f16(dev)
    idx = torch.randint(0, sk, (n,), generator=g).to(dev)
    if kind == 1:
        buf = torch.randint(0, 256, (off + sk * h * w,), generator=g, dtype=torch.uint8).to(dev)
        imgs = lut[buf[off:].view(sk, h, w)[idx].long()]
    else:
        buf = torch.rand((off + n * h * w,), generator=g).half().to(dev)
        imgs = buf[off:].view(n, h, w)
    out = torch.full((8 + n * h * w + 8,), 9.0, dtype=torch.float16, device=dev)
    grid = None if view == (1.0, 0.0, 0.0) else tta.view_grid(h, w, 1, *view, torch.float16, dev)
    a = hip.GridArgs(src=buf.data_ptr() + off * buf.element_size(), slice_idx=idx.data_ptr(), lut=lut.data_ptr(),
                     grid=0 if grid is None else grid.data_ptr(), out=out.data_ptr() + 16, kind=kind, N=n, H=h, W=w,
                     B=1, SK=sk, M=n)
    hip.call("d8s_grid_sample", ctypes.byref(a), ctypes.c_void_p(torch.cuda.current_stream(dev).cuda_stream))
    want = imgs if grid is None else F.grid_sample(imgs.contiguous()[:, None], grid.expand(n, h, w, 2), mode="bilinear",
                                                   padding_mode="zeros", align_corners=False)[:, 0]
    assert torch.equal(out[8:-8].view(n, h, w), want)
    assert bool((out[:8] == 9).all()) and bool((out[-8:] == 9).all())


@pytest.mark.parametrize("kind,w,scale", [(0, 4, 1.1), (1, 4, 1.1), (0, 3, 1.1), (1, 3, 1.1), (1, 4, 1.0)])
def test_grid_sample_many_images(dev, kind, w, scale):
    """As many images as the entry point takes (524287), past what one launch's y blocks of the four-pixel
    form hold, as the one-pixel form (3 wide) and as the gather: every image as torch's grid_sample gives it."""
    import ctypes
    from rsna_knee_efficiency_amd import hip
    n, h, sk = 65536 * 8 - 1, 2, 7
    g = torch.Generator().manual_seed(3)
    lut = tta.lut_u8_f16(dev)
    idx = torch.randint(0, sk, (n,), generator=g).to(dev)
    if kind == 1:
        src = torch.randint(0, 256, (sk, h, w), generator=g, dtype=torch.uint8).to(dev)
        imgs = lut[src.long()]
    else:
        src = torch.rand((n, h, w), generator=g).half().to(dev)
        imgs = src
    out = torch.full((n, h, w), 9.0, dtype=torch.float16, device=dev)
    grid = tta.view_grid(h, w, 1, 1.1, 0.0, 0.0, torch.float16, dev)
    a = hip.GridArgs(src=src.data_ptr(), slice_idx=idx.data_ptr(), lut=lut.data_ptr(),
                     grid=grid.data_ptr() if scale != 1.0 else 0, out=out.data_ptr(), kind=kind, N=n, H=h, W=w,
                     B=1, SK=sk, M=n)
    hip.call("d8s_grid_sample", ctypes.byref(a), ctypes.c_void_p(torch.cuda.current_stream(dev).cuda_stream))
    if scale == 1.0:
        assert torch.equal(out, imgs[idx])
        return
    # (torch's own launch over a batch of images; the volume's 7 slices once)
    want = torch.cat([F.grid_sample(c[:, None], grid.expand(len(c), h, w, 2), mode="bilinear", padding_mode="zeros",
                                    align_corners=False)[:, 0] for c in imgs.split(65536)])
    assert torch.equal(out, want[idx] if kind == 1 else want)


@pytest.mark.parametrize("kind", [0, 1])
@pytest.mark.parametrize("h,w", [(9, 12), (40, 256), (21, 61)])
def test_grid_sample_infinite_coordinates(dev, kind, h, w):
    """Infinite coordinates beside ordinary ones (a scale past fp16's range): those pixels have no tap inside
    the image and are zero, the others are torch's grid_sample."""
    import ctypes
    from rsna_knee_efficiency_amd import hip
    n, sk = 11, 5
    print(f"infinite coordinates kind={kind} {h}x{w}", flush=True)
    g = torch.Generator().manual_seed(h * w)
    grid = tta.view_grid(h, w, 1, 1.1, 0.0, 0.0, torch.float16, dev).clone()
    bad = (torch.rand((h, w, 2), generator=g) < 0.05).to(dev)
    ordinary = grid.clone()
    grid[bad] = float("inf")
    grid[1::2][bad[1::2]] = float("-inf")
    lut = tta.lut_u8_f16(dev)
    idx = torch.randint(0, sk, (n,), generator=g).to(dev)
    if kind == 1:
        src = torch.randint(0, 256, (sk, h, w), generator=g, dtype=torch.uint8).to(dev)
        imgs = lut[src[idx].long()]
    else:
        src = torch.rand((n, h, w), generator=g).half().to(dev)
        imgs = src
    want = F.grid_sample(imgs[:, None], ordinary.expand(n, h, w, 2), mode="bilinear", padding_mode="zeros",
                         align_corners=False)[:, 0]
    want[:, bad.any(2)] = 0
    out = torch.full((n, h, w), 9.0, dtype=torch.float16, device=dev)
    a = hip.GridArgs(src=src.data_ptr(), slice_idx=idx.data_ptr(), lut=lut.data_ptr(), grid=grid.data_ptr(),
                     out=out.data_ptr(), kind=kind, N=n, H=h, W=w, B=1, SK=sk, M=n)
    hip.call("d8s_grid_sample", ctypes.byref(a), ctypes.c_void_p(torch.cuda.current_stream(dev).cuda_stream))
    assert torch.equal(out, want)


@pytest.mark.parametrize("kind", [0, 1])
@pytest.mark.parametrize("h,w", [(9, 12), (40, 256), (37, 60)])
@pytest.mark.parametrize("view", [1.8, 2.5, 4.0, 0.75, 0.55, 0.5, 0.4, 0.25, -1.0, -1.3, -0.6, "turn", "noise", "nan"])
def test_grid_sample_forms(dev, kind, h, w, view):
    """Every form of the four-pixel kernel: zooms in and out of any scale, mirrored images, a rotation, a grid of
    noise (no taps together) and one with NaN and infinite coordinates beside ordinary ones, where a wave's
    lanes differ; a group remainder of images.  Bit for bit the one-pixel form, and torch's grid_sample where the
    coordinates are finite."""
    import ctypes
    import math
    from rsna_knee_efficiency_amd import hip
    n, sk = 11, 5
    print(f"grid forms kind={kind} {h}x{w} view={view}", flush=True)
    g = torch.Generator().manual_seed(h * w)
    if view == "noise":
        grid = (torch.rand((h, w, 2), generator=g) * 2.4 - 1.2).half().to(dev)
    else:
        a = math.radians(20) if view == "turn" else 0.0
        s = view if isinstance(view, float) else 1.1
        theta = torch.tensor([[[math.cos(a) / s, -math.sin(a) / s, 0.03], [math.sin(a) / s, math.cos(a) / s, -0.02]]])
        grid = F.affine_grid(theta, (1, 1, h, w), align_corners=False)[0].half().to(dev).contiguous()
        if view == "nan":
            pick = torch.rand((h, w), generator=g).to(dev)
            grid[pick < 0.02] = float("nan")
            grid[pick > 0.98] = float("inf")
    lut = tta.lut_u8_f16(dev)
    idx = torch.randint(0, sk, (n,), generator=g).to(dev)
    if kind == 1:
        src = torch.randint(0, 256, (sk, h, w), generator=g, dtype=torch.uint8).to(dev)
        imgs = lut[src[idx].long()]
    else:
        src = torch.rand((n, h, w), generator=g).half().to(dev)
        imgs = src
    outs = []
    for shift in (0, 1):                           # an output at an odd element takes the one-pixel form
        buf = torch.full((8 + n * h * w + 8,), 9.0, dtype=torch.float16, device=dev)
        a = hip.GridArgs(src=src.data_ptr(), slice_idx=idx.data_ptr(), lut=lut.data_ptr(), grid=grid.data_ptr(),
                         out=buf.data_ptr() + 16 - 2 * shift, kind=kind, N=n, H=h, W=w, B=1, SK=sk, M=n)
        hip.call("d8s_grid_sample", ctypes.byref(a), ctypes.c_void_p(torch.cuda.current_stream(dev).cuda_stream))
        assert bool((buf[:8 - shift] == 9).all()) and bool((buf[n * h * w + 8 - shift:] == 9).all())
        outs.append(buf[8 - shift:8 - shift + n * h * w].view(n, h, w).clone())
    assert torch.equal(outs[0].view(torch.int16), outs[1].view(torch.int16))
    if view != "nan":
        want = F.grid_sample(imgs[:, None], grid.expand(n, h, w, 2), mode="bilinear", padding_mode="zeros",
                             align_corners=False)[:, 0]
        assert torch.equal(outs[0], want)


def test_view_grid_made_on_a_busy_stream(dev):
    """A view's grid is made on the stream that first asks for it; a second stream that asks while the first is
    still busy gets the finished grid."""
    h, w = 48, 64
    g = torch.Generator().manual_seed(8)
    v = torch.randint(0, 256, (1, 2, 4, h, w), generator=g, dtype=torch.uint8).to(dev)
    idx = torch.tensor([0, 1, 2, 5, 6, 7], dtype=torch.int64, device=dev)
    tta.windows_u8(v, idx, torch.empty((2, 3, h, w), dtype=torch.float16, device=dev))    # (idx checked)
    lut = tta.lut_u8_f16(dev)
    x = lut[v.view(1, 8, h, w).index_select(1, idx).long()].view(1, 2, 3, h, w)
    torch.cuda.synchronize(dev)
    for scale in (1.1375, 0.8625):
        outs = [torch.zeros((2, 3, h, w), dtype=torch.float16, device=dev) for _ in range(2)]
        torch.cuda.synchronize(dev)
        streams = [torch.cuda.Stream(dev) for _ in range(2)]
        with torch.cuda.stream(streams[0]):
            torch.cuda._sleep(50_000_000)
            tta.windows_u8(v, idx, outs[0], scale)
        with torch.cuda.stream(streams[1]):
            tta.windows_u8(v, idx, outs[1], scale)
        torch.cuda.synchronize(dev)
        want = _reference(x, scale, 0.0, 0.0).view(2, 3, h, w)
        assert torch.equal(outs[0], want) and torch.equal(outs[1], want)
