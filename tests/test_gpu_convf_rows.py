"""The 16- and 32-channel layers and tails as strips of 32 (64) columns, one per wave
(convf_rows.hpp): widths at the edges of strips, and tall narrow images whose strips have 1 to 9 rows
(each way into and out of the loop over rows), against the FP32 oracle with the networks' own bar."""
import numpy as np
import pytest
import torch

import oracle_lib as OL
from anime4kcpp_amd import hip, synth

pytestmark = pytest.mark.gpu
SIZES = [(1, 2), (31, 3), (33, 1), (63, 2), (64, 7), (65, 5), (96, 4)] + [(33, h) for h in (700, 1100, 1600, 2100, 2600, 3100, 3700, 4200)]


@pytest.mark.parametrize("family,variant", [("art", "f16"), ("art", "f32"), ("fsr", "f16")])
@pytest.mark.parametrize("w,h", SIZES)
def test_strip_edges(cuda, family, variant, w, h):
    x = synth.flat_shaded(1100 + w + h, w, h)
    if family == "art":
        wts, net, oracle = hip.load_weights_artcnn(variant), hip.NetArt(variant, 0), OL.oracle_artcnn
    else:
        wts, net, oracle = hip.load_weights_fsrcnnx(variant), hip.NetFsr(variant, 0), OL.oracle_fsrcnnx
    got = net.upscale(torch.from_numpy(x).to(cuda)).cpu().numpy()
    net.close()
    assert np.abs(got - oracle(x, *wts)).max() <= 1e-5
