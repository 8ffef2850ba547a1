"""Parity of the average pool that spreads a window's taps over lanes (windows above nine taps without a compile-time form)
with the CPU oracle: channel groups from one to more than a wavefront's eight, ragged last slabs, windows larger than what
one round of requests covers, padding, tables, signed storage and the other requantisation modes."""
import pytest

import npu_plugin_amd as nce
from tests import cases as K
from tests.test_gpu_parity import check

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,h,w,c,k,s,pads,kw", [
    (3, 7, 7, 1280, (7, 7), (1, 1), (0, 0, 0, 0), {}),
    (5, 7, 7, 16, (7, 7), (1, 1), (0, 0, 0, 0), dict(in_zp=0, out_zp=0)),
    (2, 9, 8, 144, (4, 3), (2, 1), (1, 1, 2, 1), dict(in_signed=True, in_zp=-7, out_zp=3)),
    (2, 23, 21, 48, (11, 11), (2, 3), (5, 5, 5, 5), dict(in_zp=255)),
    (1, 12, 12, 80, (6, 7), (1, 2), (3, 2, 3, 1), dict(with_table=True, in_zp=19)),
    (2, 10, 10, 32, (10, 1), (1, 1), (0, 0, 0, 0), dict(ppe=dict(mode=nce.PPE_NOOP, clamp_low=0, clamp_high=255, quant_mult=26214, quant_shift=18,
                                                                 round_mode=nce.ROUND_HALF_EVEN))),
    (2, 8, 8, 272, (8, 8), (1, 1), (0, 0, 0, 0), dict(ppe=dict(mode=nce.PPE_LPRELU, clamp_low=0, clamp_high=255, quant_mult=32768, quant_shift=21,
                                                               lrelu_mult=300, lrelu_shift=10), in_zp=131)),
])
def test_avgpool_split(executor, n, h, w, c, k, s, pads, kw):
    check(K.pool_case(4100 + c + h, False, n, h, w, c, k=k, s=s, pads=pads, **kw), executor)
