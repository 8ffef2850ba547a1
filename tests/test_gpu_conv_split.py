"""Parity of the split-reduction convolution kernel and of the LDS-tiled kernel's walk over 16-byte units with the CPU oracle:
every tile of both, forced, on reductions that end inside a slice, a step and a wave's share, channel counts that are no
multiple of 64, windows that leave the image, both zero-point terms, ragged last tiles in both directions, the 64-bit
integer epilogue, permuted outputs and the fused residual add."""
import numpy as np
import pytest

import npu_plugin_amd as nce
from tests import cases as K
from tests.test_gpu_parity import check, _permuted_run

pytestmark = pytest.mark.gpu

KERNELS = [f"SPLIT={i}" for i in range(1, 6)] + [f"TILED={i}" for i in range(1, 8)]
LRELU = dict(mode=nce.PPE_LPRELU, clamp_low=0, clamp_high=250, lrelu_mult=1638, lrelu_shift=14)

SHAPES = [
    # n, h, w, ic, oc, k, s, pads, kwargs
    (1, 5, 5, 16, 16, (1, 1), (1, 1), (0, 0, 0, 0), dict()),                                    # one unit of the reduction
    (2, 9, 11, 48, 80, (3, 3), (2, 2), (1, 1, 1, 1), dict(in_zp=5, ppe=LRELU)),                 # 27 units, weight sums
    (1, 14, 14, 256, 48, (3, 3), (1, 1), (1, 1, 1, 1), dict(in_zp=200)),                        # several slices per wave
    (1, 13, 7, 112, 208, (5, 3), (1, 2), (1, 1, 2, 2), dict(in_zp=117, w_signed=False, w_zp=121)),   # both zero-point terms
    (2, 7, 7, 528, 32, (1, 1), (1, 1), (0, 0, 0, 0), dict(in_signed=True, in_zp=-7, out_signed=True, out_zp=-128)),
    (1, 12, 12, 16, 272, (7, 7), (2, 2), (3, 3, 3, 3), dict(in_zp=0, w_signed=False, w_zp=128)),
    (1, 11, 11, 32, 64, (11, 11), (4, 4), (5, 5, 5, 5), dict(in_zp=99)),
    (1, 10, 10, 64, 96, (3, 3), (1, 1), (1, 1, 1, 1), dict(in_zp=3, ppe=dict(mode=nce.PPE_NOOP, clamp_low=0, clamp_high=255, round_mode=nce.ROUND_HALF_EVEN))),
    (1, 10, 10, 64, 96, (3, 3), (1, 1), (1, 1, 1, 1), dict(in_zp=3, scale_lo=20.0, scale_hi=255.0)),   # may saturate int32
    (1, 10, 10, 80, 64, (3, 3), (1, 1), (1, 1, 1, 1), dict(scale_lo=2e-13, scale_hi=9e-13)),            # shifts above 52
]


@pytest.mark.parametrize("kernel", KERNELS)
@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: f"{s[0]}x{s[1]}x{s[2]}x{s[3]}_{s[4]}_k{s[5][0]}x{s[5][1]}s{s[6][0]}")
def test_shapes(tuned, kernel, shape):
    n, h, w, ic, oc, k, s, pads, kw = shape
    name, value = kernel.split("=")
    executor = tuned(**{"NCE_HIP_CONV_" + name: value})
    check(K.conv_case(5100 + ic + oc + h, n, h, w, ic, oc, k=k, s=s, pads=pads, **kw), executor)


@pytest.mark.parametrize("kernel", KERNELS)
def test_permuted_output_and_variants(tuned, kernel):
    name, value = kernel.split("=")
    executor = tuned(**{"NCE_HIP_CONV_" + name: value})
    case = K.conv_case(5200, 2, 9, 10, 48, 64, in_zp=77)
    got, want = _permuted_run(case, "nchw", executor)
    assert np.array_equal(got, want)
    boxes = [([0, 0, 0], [5, 8, 63]), ([4, 0, 0], [9, 8, 31]), ([4, 0, 16], [9, 8, 63])]  # (overlapping: one launch each)
    check(K.conv_case(5201, 1, 9, 10, 48, 64, in_zp=77, variants=boxes), executor)


@pytest.mark.parametrize("shape", range(1, 6))
def test_fused_add(tuned, shape):
    """The graph's residual adds inside split-reduction launches: every tensor of a small ResNet-50 pass."""
    import torch
    executor = tuned(NCE_HIP_CONV_SPLIT=shape)
    graph = K.ResNet50Graph(batch=1, size=32)
    x = graph.make_input()
    want = K.run_graph_oracle(graph, x)
    dg = K.DeviceGraph(graph, executor, x)
    stream = torch.cuda.current_stream().cuda_stream
    dg.run(stream)
    executor.synchronize(stream)
    for i, (b, w) in enumerate(zip(dg.buffers, want)):
        assert np.array_equal(b.cpu().numpy(), w), f"tensor {i} {w.shape}"
