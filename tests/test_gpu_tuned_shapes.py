"""The flash workgroup size the autotuner reports names a launch that runs.

A pure fluid's mixed flash and FP64 steps of one wave per cell (up to 65,536
cells) launch workgroups of their own size: nothing to choose, 64 reported.  A
binary mixed step's refinement takes the tuned size, and the step that
follows is the untuned one's, bit for bit."""
import ctypes as C

import numpy as np
import pytest

from helpers import binary_case, config, cube_case
from reactive_amd import abi, lib as rlib
from reactive_amd.abi import FP64, MIXED

pytestmark = pytest.mark.gpu
AUTOTUNE = 0x200


def steps(case, flags):
    lib = rlib.load()
    err = C.create_string_buffer(1024)
    hem = lib.reactive_gpu_hem_create_v1(case["model"], len(case["model"]), len(case["q"]), err, 1024)
    cfg = config(len(case["q"]), len(case["faces"]), ns=case["ns"])
    tr = lib.reactive_transport_create(1, C.byref(cfg), rlib.ptr(case["volume"]), rlib.ptr(case["faces"]), None, None, None,
                                       None, err, 1024)
    step = lib.reactive_amd_step_create(tr, hem, err, 1024)
    assert step, err.value
    assert lib.reactive_amd_step_load(step, rlib.ptr(case["q"]), rlib.ptr(case["states"])) == 0
    rep = abi.StepReport.fresh()
    for _ in range(2):
        assert lib.reactive_amd_step_run(step, 0.4, 1.0, 1, flags, C.byref(rep)) == 0, lib.reactive_amd_step_error(step)
    q = np.zeros_like(case["q"])
    assert lib.reactive_amd_step_read(step, rlib.ptr(q), None) == 0
    lib.reactive_amd_step_destroy(step)
    lib.reactive_transport_destroy(tr)
    lib.reactive_gpu_hem_destroy_v1(hem)
    return q, rep.flashBlock


@pytest.mark.parametrize("kind,mode,choice", [("pure", MIXED, (64,)), ("pure", FP64, (64,)), ("binary", MIXED, (64, 128, 256))])
def test_reported_workgroup_size_is_one_that_runs(kind, mode, choice):
    for seed in (3, 4, 5):
        case = cube_case(9, seed=seed) if kind == "pure" else binary_case(7, seed=seed)
        tuned, block = steps(case, mode | AUTOTUNE)
        plain, _ = steps(case, mode)
        assert block in choice
        assert np.array_equal(tuned.view(np.uint64), plain.view(np.uint64))
