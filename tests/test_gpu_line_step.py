"""The fused line step of the preconditioner (csrc/line_step.hpp) at the edges
of its tiles (FP32: 32 x 2 columns, FP64: 16 x 1), of its segments (4, 8 or 16
levels per thread) and of its launch rules, against the FP64 oracle's preconditioner."""
import numpy as np
import pytest

import hipmem
import mg_reference as mg

pytestmark = pytest.mark.gpu

ROWS = [n for n in mg.NAMES if n not in ("AC", "AD", "AU")]


def preconditioned(pcf, abi, oracle_mod, shape, precision, storage="fp32", iterations=2):
    nx, ny, nz = shape
    nl = pcf.examples.gaussian_hills_3d(x_size=nx, y_size=ny, z_size=nz, n_hills=3, precision=precision)
    nl.poisson.preconditioner_iterations = iterations
    nl.poisson.preconditioner_storage = storage
    gpu = pcf.State(nl)
    orc = oracle_mod.Oracle(pcf.to_config(nl), abi)
    for s in (gpu, orc):
        s.compute_sponges(0.5, 3.0)
        s.compute_operator(0.8, 1.0)
    if storage == "bf16":  # the coefficients the horizontal part reads
        for n in ROWS:
            orc.set_vector(n, mg.bf16(orc.get_vector(n)))
    x = np.random.default_rng(21).standard_normal(shape)
    dx = hipmem.DeviceArray(x.shape).upload(x)
    dy = hipmem.DeviceArray(x.shape)
    gpu.apply_preconditioner_device(dx.ptr, dy.ptr)
    got, want = dy.download(), orc.apply_preconditioner(x)
    return float(np.max(np.abs(got - want)) / np.max(np.abs(want)))


@pytest.mark.parametrize("shape,storage,iterations", [
    ((33, 3, 9), "fp32", 2), ((31, 1, 5), "fp32", 2), ((64, 5, 128), "bf16", 2), ((34, 7, 129), "fp32", 3),
    ((40, 3, 256), "bf16", 2), ((8, 3, 257), "fp32", 2), ((7, 4, 300), "bf16", 3), ((512, 130, 65), "fp32", 2),
    ((512, 130, 65), "bf16", 3), ((30, 4, 8), "fp32", 1)])
def test_fp32_line_step_matches_the_oracle(pcf, abi, oracle_mod, shape, storage, iterations):
    """FP32 rounding of a step: a 23-term sum and two recurrences that damp
    within some 30 levels, about 90 rounding errors of 6e-8 in terms a few
    times the result, up to three steps: 1e-4 of the max norm holds; a wrong
    index or segment gives 1e-2 and more."""
    err = preconditioned(pcf, abi, oracle_mod, shape, "mixed", storage, iterations)
    print(shape, storage, iterations, err)
    assert err <= 1e-4, err


@pytest.mark.parametrize("shape,storage,iterations", [
    ((31, 3, 4), "fp32", 3), ((40, 5, 17), "fp32", 2), ((33, 4, 41), "fp32", 3), ((64, 3, 60), "fp32", 2),
    ((33, 3, 61), "fp32", 2), ((260, 254, 64), "fp32", 2), ((516, 480, 17), "fp32", 2), ((516, 480, 17), "bf16", 3),
    ((40, 5, 17), "bf16", 2)])
def test_fp32_line_step_of_flat_grids_matches_the_oracle(pcf, abi, oracle_mod, shape, storage, iterations):
    """Four levels per thread (up to 64 levels where eight leave half a
    segment beyond the top, with bf16 storage on wide grids) and the sizes
    beside them, one and four columns per thread: the bound above."""
    err = preconditioned(pcf, abi, oracle_mod, shape, "mixed", storage, iterations)
    print(shape, storage, iterations, err)
    assert err <= 1e-4, err


@pytest.mark.parametrize("shape,storage,iterations", [
    ((33, 3, 257), "fp32", 3), ((8, 3, 272), "bf16", 2), ((31, 5, 512), "fp32", 2), ((66, 1, 513), "bf16", 3),
    ((34, 3, 600), "fp32", 1), ((34, 3, 601), "fp32", 4), ((33, 3, 1030), "bf16", 2),
    ((256, 33, 257), "fp32", 3), ((250, 34, 300), "bf16", 2), ((260, 30, 520), "fp32", 2)])
def test_fp32_line_step_of_tall_columns_matches_the_oracle(pcf, abi, oracle_mod, shape, storage, iterations):
    """Columns of one to three chunks, the last one shorter or full, in half
    tiles (grids of up to 128 tiles) and whole ones, with partial tiles: the
    bound above."""
    err = preconditioned(pcf, abi, oracle_mod, shape, "mixed", storage, iterations)
    print(shape, storage, iterations, err)
    assert err <= 1e-4, err


@pytest.mark.parametrize("shape,iterations", [
    ((16, 4, 4), 2), ((17, 1, 5), 2), ((15, 3, 129), 2), ((33, 5, 128), 3), ((20, 3, 256), 2), ((20, 3, 257), 2),
    ((120, 50, 100), 2), ((120, 51, 100), 2), ((31, 7, 9), 1)])
def test_fp64_line_step_matches_the_oracle(pcf, abi, oracle_mod, shape, iterations):
    """FP64, both sides of the launch rule (256 levels, 600000 cells), the
    same operations in the same order as the oracle: 1e-13."""
    err = preconditioned(pcf, abi, oracle_mod, shape, "fp64", iterations=iterations)
    assert err <= 1e-13, err
