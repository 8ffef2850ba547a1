"""Parity of the band convolution kernel with the CPU oracle: every run length, forced, on runs that cross rows and images, rings
that wrap, strides with several column planes, boxes and permuted outputs, both zero-point terms and the 64-bit integer epilogue."""
import numpy as np
import pytest

import npu_plugin_amd as nce
from tests import cases as K
from tests.test_gpu_parity import check, _permuted_run

pytestmark = pytest.mark.gpu

LRELU = dict(mode=nce.PPE_LPRELU, clamp_low=0, clamp_high=250, lrelu_mult=1638, lrelu_shift=14)

SHAPES = [
    # n, h, w, ic, oc, k, s, pads, kwargs
    (1, 5, 5, 16, 16, (2, 1), (1, 1), (0, 0, 0, 0), dict()),                                             # fewer pixels than a fragment row
    (40, 7, 7, 16, 48, (3, 3), (1, 1), (1, 1, 1, 1), dict(in_zp=5, ppe=LRELU)),                          # a run spans many images
    (3, 61, 67, 16, 2064, (7, 7), (2, 2), (3, 3, 3, 3), dict(in_zp=99)),                                 # several runs of a workgroup: the ring wraps
    (9, 33, 30, 32, 4112, (3, 3), (1, 1), (1, 1, 1, 1), dict(in_zp=0, w_signed=False, w_zp=128)),        # ... and crosses images
    (5, 20, 23, 48, 4112, (5, 3), (1, 2), (1, 1, 2, 2), dict(in_zp=117, w_signed=False, w_zp=121)),      # both zero-point terms
    (2, 30, 31, 80, 96, (3, 5), (3, 3), (2, 2, 1, 1), dict(in_signed=True, in_zp=-7, out_signed=True, out_zp=-128)),
    (2, 10, 10, 16, 32, (3, 3), (1, 1), (1, 1, 1, 1), dict(in_zp=3, scale_lo=20.0, scale_hi=255.0)),     # may saturate int32
    (2, 10, 10, 48, 64, (3, 3), (1, 1), (1, 1, 1, 1), dict(scale_lo=2e-13, scale_hi=9e-13)),             # shifts above 52
]


@pytest.mark.parametrize("run", range(1, 5))
@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: f"{s[0]}x{s[1]}x{s[2]}x{s[3]}_{s[4]}_k{s[5][0]}x{s[5][1]}s{s[6][0]}")
def test_shapes(tuned, run, shape):
    n, h, w, ic, oc, k, s, pads, kw = shape
    check(K.conv_case(5300 + ic + oc + h, n, h, w, ic, oc, k=k, s=s, pads=pads, **kw), tuned(NCE_HIP_CONV_BAND=run))


@pytest.mark.parametrize("run", range(1, 5))
def test_permuted_output_and_variants(tuned, run):
    executor = tuned(NCE_HIP_CONV_BAND=run)
    got, want = _permuted_run(K.conv_case(5400, 2, 9, 10, 48, 64, in_zp=77), "nchw", executor)
    assert np.array_equal(got, want)
    boxes = [([0, 0, 0], [5, 8, 63]), ([4, 0, 0], [9, 8, 31]), ([4, 0, 16], [9, 8, 63])]  # (overlapping: one launch each)
    check(K.conv_case(5401, 1, 9, 10, 48, 64, in_zp=77, variants=boxes), executor)
