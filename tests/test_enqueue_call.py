"""Executor.enqueue's native method: arguments, the error of an executor without a device, and every state of a task that has to go
through finalize() (not wired yet, another variant list, another PPE task, several variants)."""
import ctypes as C

import numpy as np
import pytest

import npu_plugin_amd as nce


def make_task():
    x, y = np.zeros((1, 4, 4, 16), np.uint8), np.zeros((1, 4, 4, 16), np.uint8)
    task = nce.NCEClusterTask(nce.TASK_ELTWISE, nce.activation(x), weights=nce.activation(x), output=nce.activation(y))
    task.addWholeOutputDPUTask()
    task.addPPETask(nce.PPE_ADD, 0, 255, quant_mult=1, quant_shift=0, in1_quant_mult=1, in2_quant_mult=1)
    return task


@pytest.mark.parametrize("args,kwargs", [(0, {}), (3, {}), (1, {"task": 1}), (1, {"queue": 0})])
def test_arguments(args, kwargs):
    executor, task = nce.Executor(-1), make_task()
    with pytest.raises(TypeError):
        executor.enqueue(*[task, 0, 0][:args], **kwargs)


@pytest.mark.parametrize("stream", [None, 0, C.c_void_p(0)])
@pytest.mark.parametrize("change", ["fresh", "wired", "ppe", "variant", "two", "cleared"])
def test_reaches_the_library(stream, change):
    executor, task = nce.Executor(-1), make_task()
    if change != "fresh":
        task.finalize()
    if change == "ppe":
        task.addPPETask(nce.PPE_ADD, 0, 200, quant_mult=1, quant_shift=0, in1_quant_mult=1, in2_quant_mult=1)
    if change in ("variant", "two"):
        if change == "variant":
            task._variants.clear()
        task.addWholeOutputDPUTask()
    if change == "cleared":
        task.desc.num_variants = 0
    with pytest.raises(nce.NCEError):  # (no device: it validates, it does not launch)
        executor.enqueue(task, stream=stream)
    if change != "two":
        assert task.desc.num_variants == 1 and C.addressof(task.desc.variants.contents) == C.addressof(task._variants[0])
    assert C.addressof(task.desc.ppe.contents) == C.addressof(task._ppe)
