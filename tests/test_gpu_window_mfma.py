"""Parity of depthwise convolutions and average pools on the matrix cores with the CPU oracle: windows that end inside a reduction
step, strips and runs that are cut short, runs across images, one to five channel groups, strides with several column planes, both
zero-point terms (the byte that does not fit among them), permuted outputs and the 64-bit integer epilogue; and channel slabs of
unequal and equal sizes in the vector kernel."""
import numpy as np
import pytest

import npu_plugin_amd as nce
from tests import cases as K
from tests.test_gpu_parity import check, _permuted_run

pytestmark = pytest.mark.gpu

LRELU = dict(mode=nce.PPE_LPRELU, clamp_low=0, clamp_high=250, lrelu_mult=1638, lrelu_shift=14)
DW = [
    # n, h, w, c, k, s, pads, kwargs
    (1, 5, 5, 16, (2, 1), (1, 1), (0, 0, 0, 0), dict()),
    (20, 7, 7, 32, (3, 3), (1, 1), (1, 1, 1, 1), dict(in_zp=5, ppe=LRELU)),                      # a run spans images
    (1, 9, 131, 80, (5, 5), (1, 1), (2, 2, 2, 2), dict(in_zp=99)),                               # strips, a slab of one group
    (2, 30, 23, 64, (7, 7), (2, 2), (3, 3, 3, 3), dict(in_zp=0, w_signed=False, w_zp=0)),        # 128 as two steps
    (2, 19, 40, 48, (5, 3), (1, 3), (1, 1, 2, 2), dict(in_zp=117, w_signed=False, w_zp=121)),    # both zero-point terms
    (1, 16, 16, 96, (7, 7), (1, 1), (3, 3, 3, 3), dict(in_signed=True, in_zp=-7, out_signed=True, out_zp=-128)),
    (1, 12, 12, 16, (3, 3), (1, 1), (1, 1, 1, 1), dict(scale_lo=2e-13, scale_hi=9e-13)),         # shifts above 52
]


@pytest.mark.parametrize("shape", DW, ids=lambda s: "x".join(map(str, s[:4])) + f"_k{s[4][0]}x{s[4][1]}s{s[5][0]}")
def test_depthwise(tuned, shape):
    n, h, w, c, k, s, pads, kw = shape
    check(K.dw_case(6100 + c + h, n, h, w, c, k=k, s=s, pads=pads, **kw), tuned(NCE_HIP_WINDOW_MFMA=1))


@pytest.mark.parametrize("shape", [(3, 15, 17, 48, 3, 2), (2, 40, 70, 80, 7, 1), (1, 6, 6, 16, 2, 2)], ids=str)
def test_average_pool(tuned, shape):
    n, h, w, c, k, s = shape
    check(K.pool_case(6200 + c, False, n, h, w, c, k=(k, k), s=(s, s), pads=(1, 1, 1, 1), in_zp=77), tuned(NCE_HIP_WINDOW_MFMA=1))


def test_permuted_output(tuned):
    got, want = _permuted_run(K.dw_case(6300, 2, 9, 10, 48, in_zp=77), "nchw", tuned(NCE_HIP_WINDOW_MFMA=1))
    assert np.array_equal(got, want)


@pytest.mark.parametrize("channels", [144, 208, 192, 448])  # 5 + 4, 7 + 6, 6 + 6, 8 + 8 + 8 + 4 groups
def test_slabs(tuned, channels):
    check(K.dw_case(6400 + channels, 2, 9, 11, channels, in_zp=33), tuned(NCE_HIP_WINDOW_MFMA=0))
