"""The kernels a flash is sent to, at the sizes where the choice changes.

FP64 batches of at most 65,536 cells run one cell per wave, larger ones one
cell per lane; both are the reference arithmetic, so every cell of a batch
has the bits the oracle's twin has for it, whatever the batch's size: tiles
of one small set, on both sides of the line and around the edges of a wave.

The mixed flash sends a pure fluid's cells through its saturation table, a
binary's through the searches of independent starts, with crawling starts and
restarts on groups of lanes and deferred cells on a workgroup.  A cell's
result must not depend on which other cells its lists hold, so a batch's
cells have the same bits in any order and in batches of any size.

A step's load and read change the layout of q on the device, in tiles of 256
cells and eight variables: what is read back is what was loaded, bit for bit."""
import ctypes as C

import numpy as np
import pytest

from helpers import binary_case, config, cube_case, jet_case, oracle_flash
from reactive_amd import abi, cases, lib as rlib
from reactive_amd.abi import FP64, MIXED

pytestmark = pytest.mark.gpu


def inputs(species):
    case = cube_case(8, seed=4) if species == 1 else binary_case(6, seed=9)
    q = np.ascontiguousarray(case["q"][:, :species])
    return case["model"], q, cases.internal_energy(case["q"], species), case["seeds"]


def flash(mb, q, e, seeds, mode, capacity=None):
    lib = rlib.load()
    err = C.create_string_buffer(1024)
    hem = lib.reactive_gpu_hem_create_v1(mb, len(mb), capacity or len(e), err, 1024)
    assert hem, err.value
    assert lib.reactive_amd_hem_set_arithmetic(hem, mode) == 0
    states, ok, prof = seeds.copy(), np.zeros(len(e), np.int32), abi.HemProfile.fresh()
    rc = lib.reactive_gpu_hem_run_v1(hem, rlib.ptr(np.ascontiguousarray(q)), rlib.ptr(np.ascontiguousarray(e)), len(e),
                                     rlib.ptr(states), rlib.ptr(ok), C.byref(prof), err, 1024)
    assert rc == 0, err.value
    lib.reactive_gpu_hem_destroy_v1(hem)
    return states.view(np.uint8).reshape(len(e), -1), ok, prof


@pytest.mark.parametrize("species,count", [(1, 1), (1, 63), (1, 65), (1, 65536), (1, 65537), (2, 1), (2, 65), (2, 65537)])
def test_fp64_batches_of_any_size_are_the_oracles(species, count):
    mb, q, e, seeds = inputs(species)
    base = min(count, len(e) if species == 1 else 65)
    pick = np.linspace(0, len(e) - 1, base).astype(int)
    expected, eok, counts = oracle_flash(mb, q[pick], e[pick], seeds[pick], twin=True)
    expected = expected.view(np.uint8).reshape(base, -1)
    tile = np.arange(count) % base
    got, ok, prof = flash(mb, q[pick][tile], e[pick][tile], seeds[pick][tile], FP64)
    assert np.array_equal(ok, eok[tile])
    assert np.array_equal(got, expected[tile])
    assert prof.phaseEvaluations == int(counts[tile, 0].sum())
    assert prof.residualEvaluations == int(counts[tile, 1].sum())


@pytest.mark.parametrize("species,count", [(1, 1), (1, 511), (1, 6000), (2, 1), (2, 215), (2, 1500)])
def test_mixed_results_do_not_depend_on_the_batch(species, count):
    mb, q, e, seeds = inputs(species)
    whole, wok, _ = flash(mb, q, e, seeds, MIXED)
    pick = np.random.default_rng(count).permutation(np.arange(max(count, len(e))) % len(e))[:count]
    got, ok, _ = flash(mb, q[pick], e[pick], seeds[pick], MIXED, capacity=max(count, 7))
    assert np.array_equal(ok, wok[pick])
    assert np.array_equal(got, whole[pick])


@pytest.mark.parametrize("n,kind", [(2, "pure"), (5, "pure"), (7, "binary"), (16, "pure"), (12, "jets")])
def test_load_and_read_keep_every_bit(n, kind):
    lib = rlib.load()
    case = binary_case(n, seed=2) if kind == "binary" else jet_case(n, seed=3) if kind == "jets" else cube_case(n, seed=2)
    err = C.create_string_buffer(1024)
    hem = lib.reactive_gpu_hem_create_v1(case["model"], len(case["model"]), len(case["q"]), err, 1024)
    fq = case.get("fixed_q")
    cfg = config(len(case["q"]), len(case["faces"]), ns=case["ns"], fixed=0 if fq is None else len(fq))
    tr = lib.reactive_transport_create(1, C.byref(cfg), rlib.ptr(case["volume"]), rlib.ptr(case["faces"]), rlib.ptr(fq),
                                       rlib.ptr(case.get("fixed_tstates")), None, None, err, 1024)
    step = lib.reactive_amd_step_create(tr, hem, err, 1024)
    assert step, err.value
    for seed in (1, 2):  # a second load replaces the first
        rng = np.random.default_rng(seed)
        q = np.ascontiguousarray(rng.standard_normal(case["q"].shape))
        states = case["states"].copy()
        states["p"] = rng.uniform(1e5, 1e7, len(q))
        assert lib.reactive_amd_step_load(step, rlib.ptr(q), rlib.ptr(states)) == 0
        back, sback = np.zeros_like(q), np.zeros_like(states)
        assert lib.reactive_amd_step_read(step, rlib.ptr(back), rlib.ptr(sback)) == 0
        assert np.array_equal(back.view(np.uint64), q.view(np.uint64))
        assert sback.tobytes() == states.tobytes()
        only = np.zeros_like(q)
        assert lib.reactive_amd_step_read(step, rlib.ptr(only), None) == 0
        assert np.array_equal(only.view(np.uint64), q.view(np.uint64))
    lib.reactive_amd_step_destroy(step)
    lib.reactive_transport_destroy(tr)
    lib.reactive_gpu_hem_destroy_v1(hem)
