"""The strip kernels of every family on views: sources and outputs with a row pitch and an offset of their
own, so that output pairs are not aligned for one store, against the packed result; and float images
with a NaN or an infinity, whose effect ends at the network's receptive field."""
import numpy as np
import pytest
import torch

import oracle_lib as OL
from anime4kcpp_amd import _native, hip, synth

pytestmark = pytest.mark.gpu
NETS = {"net8": lambda: hip.Net8("b4_hdn"), "net8 b18": lambda: hip.Net8("b18_hdn"), "art f16": lambda: hip.NetArt("f16"),
        "art f32": lambda: hip.NetArt("f32"), "fsr f8": lambda: hip.NetFsr("f8"), "fsr f16": lambda: hip.NetFsr("f16")}
RUNS = [(n, p) for n in NETS for p in (("fp32", "fp16", "bf16") if n.startswith("net8") else ("fp32",))]


def _upscale(net, name, prec, src, dst=None, **kw):
    return net.upscale(src, dst, precision=prec, **kw) if name.startswith("net8") else net.upscale(src, dst, **kw)


def _convert(host, dtype):
    top = {np.uint8: 255, np.uint16: 65535}.get(dtype)
    return (host * top + 0.5).astype(dtype) if top else host.astype(dtype)


@pytest.mark.parametrize("dtype", [np.uint8, np.uint16, np.float16, np.float32])
@pytest.mark.parametrize("name,prec", RUNS)
def test_views_equal_packed(cuda, name, prec, dtype):
    w, h = 131, 77
    net = NETS[name]()
    s = torch.from_numpy(_convert(synth.flat_shaded(5, w, h, dtype=np.float32), dtype)).to(cuda)
    want = _upscale(net, name, prec, s)
    big = torch.zeros((h, w + 5), dtype=s.dtype, device=cuda)
    big[:, 3:3 + w] = s
    out = torch.zeros((2 * h, 2 * w + 7), dtype=s.dtype, device=cuda)
    _upscale(net, name, prec, big[:, 3:3 + w], out[:, 1:1 + 2 * w])
    torch.cuda.synchronize()
    net.close()
    assert torch.equal(out[:, 1:1 + 2 * w], want)
    around = out.cpu().numpy()
    assert not around[:, 0].any() and not around[:, 1 + 2 * w:].any()


@pytest.mark.parametrize("dtype", [np.uint8, np.uint16, np.float16, np.float32])
def test_layer_split_views_equal_packed(cuda, dtype):
    w, h = 131, 77
    net = hip.Net("hdn1")
    s = torch.from_numpy(_convert(synth.flat_shaded(6, w, h, dtype=np.float32), dtype)).to(cuda)
    ws = torch.empty(_native.lib().achip_pass8_workspace_bytes(w, h), dtype=torch.uint8, device=cuda)
    want = net.upscale(s, workspace=ws)
    big = torch.zeros((h, w + 5), dtype=s.dtype, device=cuda)
    big[:, 3:3 + w] = s
    out = torch.zeros((2 * h, 2 * w + 7), dtype=s.dtype, device=cuda)
    net.upscale(big[:, 3:3 + w], out[:, 1:1 + 2 * w], workspace=ws)
    torch.cuda.synchronize()
    net.close()
    assert torch.equal(out[:, 1:1 + 2 * w], want)
    around = out.cpu().numpy()
    assert not around[:, 0].any() and not around[:, 1 + 2 * w:].any()


# conv3x3 layers (and a conv5x5 as two): how far a source pixel reaches, in source pixels
REACH = {"legacy": 9, "net8": 6, "net8 b18": 20, "art f16": 7, "art f32": 7, "fsr f8": 7, "fsr f16": 7}


@pytest.mark.parametrize("bad", [float("nan"), float("inf"), float("-inf")])
@pytest.mark.parametrize("name,prec", [("legacy", "fp32"), ("legacy", "fp16"), ("legacy", "bf16")] + RUNS)
def test_non_finite_pixels_stay_local(cuda, name, prec, bad):
    """One NaN or infinite source pixel changes no output outside the receptive field; the 16-bit kernels'
    patches of four rows (a zero weight times it is a NaN) reach one row further per layer."""
    w, h = 150, 131
    net = hip.Net("hdn1") if name == "legacy" else NETS[name]()
    x = synth.flat_shaded(7, w, h, dtype=np.float32)
    kw = {}
    if name == "legacy":
        kw = {"precision": prec}
        if prec == "fp32":
            kw["workspace"] = torch.empty(_native.lib().achip_pass8_workspace_bytes(w, h), dtype=torch.uint8, device=cuda)
    run = (lambda s: net.upscale(s, **kw)) if name == "legacy" else (lambda s: _upscale(net, name, prec, s))
    clean = run(torch.from_numpy(x).to(cuda)).cpu().numpy()
    r = REACH[name]
    rows = r if prec == "fp32" else 2 * r
    for px, py in ((63, 64), (0, 0), (w - 1, h - 1), (61, 17)):
        y = x.copy()
        y[py, px] = bad
        got = run(torch.from_numpy(y).to(cuda)).cpu().numpy()
        inside = np.zeros_like(clean, dtype=bool)
        inside[2 * max(py - rows, 0):2 * (py + rows + 1), 2 * max(px - r, 0):2 * (px + r + 1)] = True
        assert np.array_equal(got[~inside], clean[~inside]), (px, py)
    net.close()


@pytest.mark.parametrize("bad", [float("nan"), float("inf"), float("-inf")])
@pytest.mark.parametrize("name", ["legacy", "net8", "art f16", "art f32", "fsr f8", "fsr f16"])
def test_non_finite_pixels_as_the_oracle(cuda, name, bad):
    """FP32 layers without zero weights: a NaN or an infinity gives the oracle's outputs (max and min take
    the other operand of a NaN there too)."""
    w, h = 150, 131
    x = synth.flat_shaded(7, w, h, dtype=np.float32)
    x[64, 63] = x[0, 149] = bad
    s = torch.from_numpy(x).to(cuda)
    if name == "legacy":
        net = hip.Net("hdn1")
        ws = torch.empty(_native.lib().achip_pass8_workspace_bytes(w, h), dtype=torch.uint8, device=cuda)
        got, want = net.upscale(s, workspace=ws), OL.oracle_pass(x, *hip.load_weights("hdn1"))
    else:
        net = NETS[name]()
        got = net.upscale(s)
        want = (OL.oracle_pass8(x, *hip.load_weights8("b4_hdn")) if name == "net8" else
                OL.oracle_artcnn(x, *hip.load_weights_artcnn(name[4:])) if name[:3] == "art" else
                OL.oracle_fsrcnnx(x, *hip.load_weights_fsrcnnx(name[4:])))
    assert np.abs(got.cpu().numpy() - want).max() <= 1e-5
    net.close()
