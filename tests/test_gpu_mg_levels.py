"""The multigrid V-cycle of the mixed solve on the grids whose levels take
other kernels than the smaller ones of test_gpu_mixed.py, against the FP64
restatement (mg_reference.py).  FP32 rounding through the levels stays below
1e-3 of the result's max norm (see test_multigrid_vcycle_matches_fp64_restatement
for its size); a wrong index, sign, level or coefficient gives errors of order
one."""
import numpy as np
import pytest

import hipmem
import mg_reference as mg

pytestmark = pytest.mark.gpu


def vcycle_error(pcf, shape, storage, nu=2, coarse=4):
    nx, ny, nz = shape
    nl = pcf.examples.mountain_wave_3d(x_size=nx, y_size=ny, z_size=nz, iterations=3)
    p = nl.poisson
    p.precision, p.preconditioner_type, p.preconditioner_storage = "mixed", "multigrid", storage
    p.mg_smoothing_steps, p.mg_coarse_steps = nu, coarse
    gpu = pcf.State(nl)
    gpu.compute_sponges(0.8, 3.0)
    gpu.compute_operator(0.8, 1.0)
    c = pcf.output.constants(nl)
    lv = mg.levels({n: gpu.get_vector(n) for n in mg.NAMES}, nl.domain.lx / c["lref"] / nx,
                   nl.domain.ly / c["lref"] / ny, p.dtau, round_apply=mg.bf16 if storage == "bf16" else None)
    x = np.random.default_rng(5).standard_normal(shape)
    want = mg.vcycle(lv, x, nu=nu, coarse_steps=coarse)
    dx, dy = hipmem.DeviceArray(shape).upload(x), hipmem.DeviceArray(shape)
    gpu.apply_preconditioner_device(dx.ptr, dy.ptr)
    err = float(np.max(np.abs(dy.download() - want)) / np.max(np.abs(want)))
    print(shape, storage, nu, coarse, "levels", len(lv), "rel err", err)
    gpu.close()
    return err


@pytest.mark.parametrize("shape,storage", [((68, 40, 264), "fp32"), ((48, 64, 520), "fp32"), ((68, 40, 264), "bf16")])
def test_tall_levels_match_the_restatement(pcf, shape, storage):
    """More than 256 levels on the levels smoothed by line steps (2720
    columns; beyond 512 levels all)."""
    assert vcycle_error(pcf, shape, storage) <= 1e-3


@pytest.mark.parametrize("storage", ["fp32", "bf16"])
@pytest.mark.parametrize("shape", [(64, 45, 24), (45, 64, 24), (32, 30, 70), (33, 24, 264)])
def test_unpaired_levels_match_the_restatement(pcf, shape, storage):
    """An odd size: 2 x 1 and 1 x 2 aggregation of finest levels smoothed by
    line steps (2880 columns), whose first coarse levels of 1440 columns are
    z fastest and rounded with bf16 storage; finest levels of at most 1024
    columns, paired and not, up to 264 levels."""
    assert vcycle_error(pcf, shape, storage) <= 1e-3


@pytest.mark.parametrize("shape,storage", [
    ((16, 16, 160), "fp32"), ((28, 24, 238), "fp32"), ((28, 24, 239), "bf16"), ((32, 32, 200), "bf16"),
    ((16, 12, 257), "bf16"), ((32, 30, 200), "fp32"), ((44, 48, 200), "bf16")])
def test_small_levels_of_many_levels_match_the_restatement(pcf, shape, storage):
    """129 to 512 levels, four and eight per lane, of levels smoothed column
    by column and of the coarsest one; both sides of the finest level's rule
    (1024 columns, 256 levels, 160000 cells), whose line steps read unrounded
    coefficients up to 1024 columns with either storage.  Four steps on the
    coarsest level as above: the twenty of the default leave 2e-3 at
    16 x 16 x 160, the rounding of the scan over a wavefront's lanes on the
    nearly singular level."""
    assert vcycle_error(pcf, shape, storage) <= 1e-3


@pytest.mark.parametrize("storage", ["fp32", "bf16"])
@pytest.mark.parametrize("shape", [(260, 128, 128), (132, 66, 136)])
def test_production_levels_match_the_restatement(pcf, shape, storage):
    """Four columns per thread (4.26 million cells, a partial tile in x), whose
    step with the correction reads two coarse cells at once and whose residual
    sums x pairs in the thread; 136 levels on more than 128 tiles, sixteen
    levels per thread."""
    assert vcycle_error(pcf, shape, storage) <= 1e-3
