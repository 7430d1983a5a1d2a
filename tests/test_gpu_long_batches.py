"""Batches longer than one cell per wave takes, and long queues.

FP64 batches and steps of more than 65,536 cells run one cell per lane
(stepFlashKernel, hemFlashKernel: lanes.hip, and step.hip and hem.hip for a
pure fluid's plain flash); every other test of those modes is shorter.  Small
sets tiled to that length, bit for bit the oracle's twin: plain, analytic
Jacobian, no liquid, boundary search, capillary recovery; a resident step's
flash against the batch flash of its parts; the allocation-free batch's
per-lane partial sums, which it takes above 16,384 cells.

The mixed flash's deferred cells run on three waves each up to 4,096 of them
and on one beyond: a binary cell that defers, alone and 5,000 times.  Its
solves leave their loops in different iterations on the lanes of a wave; a
build that lost the early ones' results failed it."""
import ctypes as C

import numpy as np
import pytest

from helpers import Device, binary_case, config, cube_case, oracle_flash
from reactive_amd import abi, cases, lib as rlib, model
from reactive_amd.abi import FP64, MIXED
from test_gpu_capillary import cap_records, host_batch, load, twin
from test_gpu_dispatch import flash, inputs
from test_zz_no_alloc import COUNTERS, run

pytestmark = pytest.mark.gpu
LONG = 65537


@pytest.mark.parametrize("species,liquid,analytic", [(1, "N2O", 1), (1, None, 0), (2, "N2O", 0), (2, "N2O", 1), (2, None, 0)])
def test_fp64_lane_batches_are_the_oracles(species, liquid, analytic):
    _, q, e, seeds = inputs(species)
    pick = np.linspace(0, len(e) - 1, 65).astype(int)
    mb = model.model_bytes(model.build_model(gas_species=("N2O", "N2")[:species], liquid=liquid, analytic_jacobian=analytic))
    expected, eok, counts = oracle_flash(mb, q[pick], e[pick], seeds[pick], twin=True)
    tile = np.arange(LONG) % 65
    got, ok, prof = flash(mb, q[pick][tile], e[pick][tile], seeds[pick][tile], FP64)
    assert np.array_equal(ok, eok[tile])
    assert np.array_equal(got, expected.view(np.uint8).reshape(65, -1)[tile])
    assert prof.phaseEvaluations == int(counts[tile, 0].sum())
    assert prof.residualEvaluations == int(counts[tile, 1].sum())


@pytest.mark.parametrize("name", ["n2o", "trace_capillary", "trace", "trace_analytic", "binary"])
def test_capillary_and_boundary_lane_batches_are_the_oracles(name):
    d = load(name)
    n = len(d["energy"])
    expected, eok, counts = twin(d)
    tile = np.arange(LONG) % n
    long = {k: (v if k == "model" else np.ascontiguousarray(v[tile])) for k, v in d.items() if k == "model" or len(v) == n}
    states, ok, prof = host_batch(long, "color" in d)
    assert np.array_equal(ok, eok[tile])
    raw = states.view(np.uint8).reshape(LONG, -1)
    assert np.array_equal(raw, expected.view(np.uint8).reshape(n, -1)[tile])
    assert prof.phaseEvaluations == int(counts[tile, 0].sum())


@pytest.mark.parametrize("species,analytic", [(2, 0), (1, 1)])
def test_fp64_lane_step_is_the_batch_flash_of_its_parts(species, analytic):
    n = 41
    cube = cases.pure_n2o_cube if species == 1 else cases.binary_cube
    faces, volume, q, seeds, _ = cube(n, seed=5)
    mb = model.model_bytes(model.build_model(gas_species=("N2O", "N2")[:species], analytic_jacobian=analytic))
    lib = rlib.load()
    err = C.create_string_buffer(1024)

    def batch(q, seeds):
        raw, ok, _ = flash(mb, q[:, :species], cases.internal_energy(q, species), seeds, FP64)
        return raw, ok

    half = len(q) // 2
    start = seeds.copy()
    for a, b in ((0, half), (half, len(q))):
        raw, ok = batch(q[a:b], seeds[a:b])
        start[a:b] = np.where(ok == 1, raw.view(start.dtype).ravel(), start[a:b])
        bad = np.where(ok == 0)[0] + a
        good = np.where(ok == 1)[0][0] + a
        q[bad], start[bad] = q[good], start[good]
    hem = lib.reactive_gpu_hem_create_v1(mb, len(mb), len(q), err, 1024)
    cfg = config(len(q), len(faces), ns=species)
    tr = lib.reactive_transport_create(1, C.byref(cfg), rlib.ptr(volume), rlib.ptr(faces), None, None, None, None, err, 1024)
    step = lib.reactive_amd_step_create(tr, hem, err, 1024)
    assert step, err.value
    assert lib.reactive_amd_step_load(step, rlib.ptr(q), rlib.ptr(start)) == 0
    rep = abi.StepReport.fresh()
    assert lib.reactive_amd_step_run(step, 0.4, 1.0, 1, FP64, C.byref(rep)) == 0, lib.reactive_amd_step_error(step)
    end, states = np.zeros_like(q), np.zeros_like(start)
    assert lib.reactive_amd_step_read(step, rlib.ptr(end), rlib.ptr(states)) == 0
    for a, b in ((0, half), (half, len(q))):
        raw, ok = batch(end[a:b], start[a:b])
        expected = np.where(ok == 1, raw.view(start.dtype).ravel(), start[a:b])
        assert expected.tobytes() == states[a:b].tobytes()
    lib.reactive_amd_step_destroy(step)
    lib.reactive_transport_destroy(tr)
    lib.reactive_gpu_hem_destroy_v1(hem)


def test_noalloc_batch_of_one_cell_per_lane():
    lib = rlib.load()
    case = cube_case(8, seed=4)
    n = 16385
    tile = np.arange(n) % len(case["energy"])
    q, e = np.ascontiguousarray(case["q"][tile, :1]), np.ascontiguousarray(case["energy"][tile])
    err = C.create_string_buffer(1024)
    h = lib.reactive_gpu_hem_create_resident_v1(case["model"], len(case["model"]), n, err, 1024)
    assert h, err.value
    dev = Device()
    bufs = (dev.put(q), dev.put(e), dev.put(case["states"][tile]), dev.put(np.zeros(n, abi.CAPILLARY_DTYPE)))
    order = np.random.default_rng(1).permutation(n).astype(np.uint32)
    ref, rprof = run(lib, "reactive_gpu_hem_run_resident_v1", h, dev, bufs, order, n)
    out, prof = run(lib, "reactive_gpu_hem_run_resident_noalloc_v1", h, dev, bufs, order, n)
    assert out.tobytes() == ref.tobytes()
    for f in COUNTERS:
        assert getattr(prof, f) == getattr(rprof, f), f
    dev.close()
    lib.reactive_gpu_hem_destroy_v1(h)


@pytest.fixture(scope="module")
def deferring():
    """A cell of the 96^3 binary box: its FP32 search leaves a gas candidate
    alone, and the FP64 restarts find the liquid of a few 1e-6 of the mass."""
    _, _, q, seeds, _ = cases.binary_cube(96, seed=2026)
    c = slice(754816, 754817)
    mb = model.model_bytes(model.build_model(gas_species=("N2O", "N2")))
    return mb, np.ascontiguousarray(q[c, :2]), cases.internal_energy(q[c], 2), seeds[c].copy()


@pytest.mark.parametrize("count", [1, 4096, 5000])
def test_deferred_cells_do_not_depend_on_the_queue(deferring, count):
    mb, q, e, seeds = deferring
    f64, fok, _ = flash(mb, q, e, seeds, FP64)
    lib = rlib.load()
    err = C.create_string_buffer(1024)
    hem = lib.reactive_gpu_hem_create_v1(mb, len(mb), count, err, 1024)
    assert hem and lib.reactive_amd_hem_set_arithmetic(hem, MIXED) == 0
    tile = np.zeros(count, int)
    states, ok, prof = seeds[tile], np.zeros(count, np.int32), abi.HemProfile.fresh()
    assert lib.reactive_gpu_hem_run_v1(hem, rlib.ptr(np.ascontiguousarray(q[tile])), rlib.ptr(np.ascontiguousarray(e[tile])),
                                       count, rlib.ptr(states), rlib.ptr(ok), C.byref(prof), err, 1024) == 0, err.value
    single, queued = C.c_uint64(), C.c_uint64()
    assert lib.reactive_amd_hem_mixed_report(hem, C.byref(single), C.byref(queued)) == 0
    lib.reactive_gpu_hem_destroy_v1(hem)
    assert queued.value == count
    assert fok[0] == 1 and (ok == 1).all()
    root = f64.view(states.dtype).ravel()[0]
    # both stop inside the model's tolerances, 1e-9 in volume and energy
    assert abs(states["T"][0] / root["T"] - 1) < 1e-7 and abs(states["p"][0] / root["p"] - 1) < 1e-7
    raw = states.view(np.uint8).reshape(count, -1)
    assert (raw == raw[0]).all()
    assert prof.phaseEvaluations % count == 0 and prof.phaseEvaluations // count == 1953
