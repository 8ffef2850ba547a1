"""Single-task enqueues keep the launches of a descriptor for its next call; a descriptor that changed must not see them."""
import pytest

from tests import cases as K

pytestmark = pytest.mark.gpu


def test_changed_descriptor_is_planned_anew(executor):
    """A descriptor enqueued before, then changed in place, runs as it stands now (its earlier launches are not reused)."""
    import torch
    case = K.pool_case(4200, False, 2, 7, 7, 64, k=(7, 7), s=(1, 1), pads=(0, 0, 0, 0))
    dc = K.DeviceCase(case)
    stream = torch.cuda.current_stream().cuda_stream
    for zp, hi in ((128, 255), (100, 255), (100, 140)):
        case.out_zp, case.ppe["clamp_high"] = zp, hi
        dc.task.desc.output.zero_point = zp
        dc.task._ppe.clamp_high = hi
        for _ in range(2):
            dc.output.fill_(0)
            executor.enqueue(dc.task, stream)
            executor.synchronize(stream)
            assert (dc.output.cpu().numpy() == K.run_oracle(case)).all()
