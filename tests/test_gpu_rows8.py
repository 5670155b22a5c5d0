"""The streamed FP32 layers of the 8-channel networks (conv8_rows.hpp): strips of 64 computed
columns that keep 56 to 64 of them, any even number of rows, two or four layers per launch by the
image's size.  Sizes at the edges of the strips, odd heights, both sides of the size rule (a tall
narrow image has its strip-rows cheaply), every remainder of the layer count; ACNetLegacy against
the fused kernel, bit for bit, the others against the FP32 oracle with the bars of their own tests."""
import ctypes

import numpy as np
import pytest
import torch

import oracle_lib as OL
from anime4kcpp_amd import _native, hip, synth

pytestmark = pytest.mark.gpu
EDGES = [(2, 9), (55, 4), (57, 7), (58, 1), (59, 30), (60, 33), (61, 2), (64, 5), (113, 19), (117, 12), (121, 6), (128, 3)]
TALL = [(61, 12290), (63, 6161)]   # more strip-rows than four strips of 12 on 256 compute units


@pytest.mark.parametrize("w,h", EDGES + TALL)
def test_legacy_layers_and_batch(cuda, w, h):
    net = hip.Net("hdn1", 0)
    L = _native.lib()
    s = torch.from_numpy(synth.flat_shaded(900 + w + h, w, h)).to(cuda)
    fused = net.upscale(s, config=0)
    got = torch.empty_like(fused)
    need = L.achip_pass8_workspace_bytes(w, h)
    ws = torch.empty(need, dtype=torch.uint8, device=cuda)
    assert L.achip_pass_layers(net.handle, ctypes.c_void_p(s.data_ptr()), 4 * w, hip.elem_type(s.dtype), w, h,
                               ctypes.c_void_p(got.data_ptr()), 8 * w, hip.elem_type(got.dtype), ctypes.c_void_p(ws.data_ptr()),
                               need, None) == 0, _native.last_error()
    small = s[: min(h, 7), : min(w, 61)]
    batch = net.upscale_batch_layers([s, small])
    torch.cuda.synchronize()
    assert torch.equal(got, fused) and torch.equal(batch[0], fused)
    assert torch.equal(batch[1], net.upscale(small, config=0))
    net.close()


def _acnet8(blocks):
    k, b, a, _ = hip.load_weights8("b18_hdn")
    return (np.concatenate([k[:72 + 576 * blocks], k[-288:]]), np.concatenate([b[:8 + 8 * blocks], b[-4:]]), a[:8 * (blocks + 1)], blocks)


@pytest.mark.parametrize("blocks,w,h", [(b, *EDGES[b]) for b in range(1, 10)] + [(1, *TALL[0])] + [(b, *TALL[1]) for b in (2, 3, 4, 7)])
def test_acnet8_depths(cuda, blocks, w, h):
    wts = _acnet8(blocks)
    x = synth.flat_shaded(950 + w + h, w, h)
    net = hip.Net8("b4", 0, weights=wts)
    got = net.upscale(torch.from_numpy(x).to(cuda)).cpu().numpy()
    assert np.abs(got - OL.oracle_pass8(x, *wts)).max() <= 1e-5
    net.close()


@pytest.mark.parametrize("w,h", EDGES)
def test_fsrcnnx8_edges(cuda, w, h):
    k, b, a, f, blocks = hip.load_weights_fsrcnnx("f8")
    x = synth.flat_shaded(970 + w + h, w, h)
    net = hip.NetFsr("f8", 0)
    got = net.upscale(torch.from_numpy(x).to(cuda)).cpu().numpy()
    assert np.abs(got - OL.oracle_fsrcnnx(x, k, b, a, f, blocks)).max() <= 1e-5
    net.close()


@pytest.mark.parametrize("dims", [[(56, 5), (57, 1), (113, 20), (3, 40)], [(512, 300)] * 3, [(61, 2100), (240, 256), (7, 9)], [(700, 512)] * 4])
def test_batch_splits(cuda, dims):
    """Small batches take four layers per launch, larger ones two: each image is its own fused pass."""
    net = hip.Net("hdn3", 0)
    srcs = [torch.from_numpy(synth.flat_shaded(990 + i + w, w, h, dtype=np.uint8)).to(cuda) for i, (w, h) in enumerate(dims)]
    out = net.upscale_batch_layers(srcs)
    for s, d in zip(srcs, out):
        assert torch.equal(d, net.upscale(s, config=0))
    net.close()
