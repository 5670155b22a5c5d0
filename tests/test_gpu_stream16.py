"""The streamed 16-bit passes: ACNetLegacy (stream16.hpp): strips of 64 output columns, any even
number of rows per strip.  Sizes at the edges of strips (one column more and less than 64 and
128, images narrower than a strip's margin, odd heights, one row more and less than the
128-row strips of configuration 1) against the FP64 restatement with test_gpu_mfma's bounds;
the two configurations cut the image differently and must agree bit for bit, as must a batch
and the same images alone."""
import numpy as np
import pytest
import torch

from anime4kcpp_amd import hip, synth
from oracle_lib import oracle_pass8_f64, oracle_pass_f64, to_float
from test_gpu_mfma import BOUNDS, err_report

pytestmark = pytest.mark.gpu

SIZES = [(1, 1), (2, 1), (1, 5), (7, 9), (8, 16), (9, 2), (63, 127), (64, 128), (65, 129), (71, 31), (72, 33), (73, 3),
         (127, 130), (129, 257), (136, 40), (200, 1), (1, 140)]


@pytest.fixture(scope="module")
def net(cuda):
    n = hip.Net("hdn2", 0)
    yield n
    n.close()


@pytest.mark.parametrize("prec", ["fp16", "bf16"])
@pytest.mark.parametrize("w,h", SIZES)
def test_strip_edges(net, weights, cuda, prec, w, h):
    src = synth.flat_shaded(800 + w + 3 * h, w, h)
    s = torch.from_numpy(src).to(cuda)
    got = net.upscale(s, precision=prec, config=0)
    other = net.upscale(s, precision=prec, config=1)
    torch.cuda.synchronize()
    assert torch.equal(got, other)
    k, b = weights["hdn2"]
    mx, mean, _ = err_report(got.cpu().numpy(), oracle_pass_f64(to_float(src), k, b))
    assert mx <= BOUNDS[prec][0] and mean <= BOUNDS[prec][1]


@pytest.mark.parametrize("dtype", [np.uint8, np.uint16, np.float16, np.float32])
def test_types_and_strides(net, cuda, dtype):
    """Every element type, from views with a pitch of their own (odd element offsets, so output
    pairs that no single store can take), equals the packed image's result."""
    w, h = 131, 77
    host = synth.flat_shaded(5, w, h, dtype=np.float32)
    top = {np.uint8: 255, np.uint16: 65535}.get(dtype)
    arr = (host * top + 0.5).astype(dtype) if top else host.astype(dtype)
    s = torch.from_numpy(arr).to(cuda)
    want = net.upscale(s, precision="fp16")
    big = torch.zeros((h, w + 5), dtype=s.dtype, device=cuda)
    big[:, 3:3 + w] = s
    out = torch.zeros((2 * h, 2 * w + 7), dtype=s.dtype, device=cuda)
    net.upscale(big[:, 3:3 + w], out[:, 1:1 + 2 * w], precision="fp16")
    torch.cuda.synchronize()
    assert torch.equal(out[:, 1:1 + 2 * w], want)
    around = out.cpu().numpy()
    assert not around[:, 0].any() and not around[:, 1 + 2 * w:].any()


@pytest.mark.parametrize("prec", ["fp16", "bf16"])
@pytest.mark.parametrize("config", [0, 1])
def test_batch_of_edges(net, cuda, prec, config):
    srcs = [torch.from_numpy(synth.flat_shaded(900 + i, w, h, dtype=np.uint8)).to(cuda) for i, (w, h) in enumerate(SIZES)]
    out = net.upscale_batch(srcs, precision=prec, config=config)
    for i, s in enumerate(srcs):
        alone = net.upscale(s, precision=prec)
        torch.cuda.synchronize()
        assert torch.equal(out[i], alone), SIZES[i]


SIZES8 = [(1, 1), (2, 9), (59, 5), (60, 16), (61, 17), (62, 70), (63, 71), (64, 30), (69, 2), (70, 12), (71, 13), (125, 68)]


@pytest.mark.parametrize("prec", ["fp16", "bf16"])
@pytest.mark.parametrize("variant", ["b4_hdn", "b8_hdn", "b18_box_hdn"])
def test_acnet8_strip_edges(cuda, prec, variant):
    """ACNet<8>: 70, 62 and (two launches) 62 and 60 output columns per strip."""
    k, b, a, blocks = hip.load_weights8(variant)
    net = hip.Net8(variant)
    for w, h in SIZES8:
        src = synth.flat_shaded(300 + w + 3 * h, w, h)
        got = net.upscale(torch.from_numpy(src).to(cuda), precision=prec)
        torch.cuda.synchronize()
        mx, mean, _ = err_report(got.cpu().numpy(), oracle_pass8_f64(to_float(src), k, b, a, blocks))
        assert mx <= BOUNDS[prec][0] and mean <= BOUNDS[prec][1], (w, h)
    net.close()


@pytest.mark.parametrize("blocks", [1, 2, 3, 8, 9, 10, 17, 18, 19, 27])
def test_acnet8_crop(cuda, blocks):
    """Every cut of the blocks into launches: a crop's outputs further than the receptive field
    from its border are the whole image's, bit for bit, in strips that start elsewhere."""
    k, b, a, _ = hip.load_weights8("b18_hdn")
    pick = [i % 18 for i in range(blocks)]
    kk = np.concatenate([k[:72]] + [k[72 + 576 * i:72 + 576 * (i + 1)] for i in pick] + [k[-288:]])
    bb = np.concatenate([b[:8]] + [b[8 + 8 * i:16 + 8 * i] for i in pick] + [b[-4:]])
    aa = np.concatenate([a[:8]] + [a[8 + 8 * i:16 + 8 * i] for i in pick])
    net = hip.Net8("b4", weights=(kk, bb, aa, blocks))
    src = torch.from_numpy(synth.flat_shaded(41, 230, 180, dtype=np.uint8)).to(cuda)
    whole = net.upscale(src, precision="fp16", out_dtype=torch.float32)
    x, y, w, h, m = 37, 23, 150, 121, blocks + 2
    part = net.upscale(src[y:y + h, x:x + w], precision="fp16", out_dtype=torch.float32)
    torch.cuda.synchronize()
    assert torch.equal(part[2 * m:2 * (h - m), 2 * m:2 * (w - m)], whole[2 * (y + m):2 * (y + h - m), 2 * (x + m):2 * (x + w - m)])
    net.close()


def test_more_columns_than_one_grid_dimension(net, cuda):
    """360 million columns, a row high: the strips go along the grid's y.  Around the image's ends and at
    spots between (a strip's first and last columns), the outputs are those of a part of the image."""
    w = 360_000_001
    src = torch.from_numpy(synth.flat_shaded(43, 1 << 16, 1, dtype=np.uint8)).to(cuda).repeat(1, w // (1 << 16) + 1)[:, :w].contiguous()
    got = net.upscale(src, precision="fp16")
    for x in (0, 64 * 1234567 - 200, w // 2, w - 400):
        a, b = max(x - 20, 0), min(x + 420, w)
        part = net.upscale(src[:, a:b].contiguous(), precision="fp16")
        lo, hi = (0 if a == 0 else x), (w if b == w else x + 400)
        assert torch.equal(got[:, 2 * lo:2 * hi], part[:, 2 * (lo - a):2 * (hi - a)]), x


def test_batch_strips_start_together(net, cuda):
    """200 strips of 128 rows on 256 compute units take about as long as 16 of them: every workgroup of
    the queue has one strip before any takes a second (which makes it twice as long)."""
    def us(w):
        src = [torch.zeros((128, w), dtype=torch.uint8, device=cuda)]
        dst = [torch.empty((256, 2 * w), dtype=torch.uint8, device=cuda)]
        best = float("inf")
        for _ in range(8):
            e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            e0.record()
            for _ in range(10):
                net.upscale_batch(src, dst, precision="fp16", config=1)
            e1.record()
            torch.cuda.synchronize()
            best = min(best, e0.elapsed_time(e1) * 100)
        return best
    few, many = us(16 * 64), us(200 * 64)
    assert many < 1.5 * few, (few, many)
