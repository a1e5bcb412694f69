"""FluidKernelFFT (L, L^-1) on the GPU against the FP64 oracle.

Bar: relative L2 <= 1e-5 against the FP64 restatement of
DiffOper::Apply(Inverse)OperatorOnTheFly (DiffOper.cxx:747-905)."""
import numpy as np
import pytest

import oracle
from atlaswerks_amd import synth

pytestmark = pytest.mark.gpu

TOL = 1e-5

SIZES = [(8, 8, 8), (6, 10, 12), (24, 40, 36), (32, 31, 36), (64, 64, 64), (17, 9, 5),
         (96, 48, 40), (1, 16, 16), (128, 128, 128), (32, 64, 256), (256, 256, 16),
         (128, 32, 64)]
# axes with a prime factor above 13 (dense products): 67, 71, 127, 181 on each axis, 217 =
# 7 * 31 and 61
PRIME_SIZES = [(12, 20, 67), (16, 127, 10), (181, 12, 14), (61, 67, 71), (36, 217, 181),
               (1, 1, 181)]
# axes whose pass blocks stage more than 64 KiB of LDS (up to 159 KiB): 2500 along x,
# the primes 1021 along x, 3001 along y and 1499 along z (chirp-z transforms)
LONG_SIZES = [(3, 4, 2500), (4, 5, 1021), (2, 3001, 3), (1499, 3, 2)]


def _field(shape, seed):
    return synth.smooth_noise_field(shape, sigma=1.5, seed=seed)


@pytest.mark.parametrize("shape", SIZES + PRIME_SIZES + LONG_SIZES)
@pytest.mark.parametrize("inverse", [True, False])
def test_operator_matches_oracle(shape, inverse):
    import torch
    from atlaswerks_amd.fluid import DiffOperGPU, DiffOperParam
    from gpu_util import aos, host, rel_l2, soa, to_dev
    nz, ny, nx = shape
    print("fluid", shape, "inverse", inverse, flush=True)
    f = _field(shape, seed=nx * 7 + ny)
    sp = (1.0, 1.25, 0.8)
    p = DiffOperParam(alpha=0.01, beta=0.01, gamma=0.001)
    op = DiffOperGPU((nx, ny, nz), sp, p)
    d = to_dev(f)
    if inverse:
        op.ApplyInverseOperator(d)
    else:
        op.ApplyOperator(d)
    got = host(d)
    ref = oracle.diffoper(aos(f), sp=sp, alpha=0.01, beta=0.01, gamma=0.001, inverse=inverse)
    err = rel_l2(got, soa(ref))
    assert err <= TOL, err


@pytest.mark.parametrize("shape", [(16, 16, 16), (24, 40, 36)])
@pytest.mark.parametrize("lpow,divfree", [(1.0, False), (0.5, False), (1.0, True), (2.0, True)])
def test_eigen_and_divfree(shape, lpow, divfree):
    from atlaswerks_amd.fluid import DiffOperGPU, DiffOperParam
    from gpu_util import aos, host, rel_l2, soa, to_dev
    nz, ny, nx = shape
    print("fluid eigen", shape, lpow, divfree, flush=True)
    f = _field(shape, seed=3)
    sp = (1.0, 1.0, 1.5)
    p = DiffOperParam(alpha=0.02, beta=0.01, gamma=0.01, lpow=lpow, use_eigen_lut=True,
                      divergence_free=divfree)
    op = DiffOperGPU((nx, ny, nz), sp, p)
    for inverse in (True, False):
        d = to_dev(f)
        (op.ApplyInverseOperator if inverse else op.ApplyOperator)(d)
        ref = oracle.diffoper(aos(f), sp=sp, alpha=0.02, beta=0.01, gamma=0.01, inverse=inverse,
                              lpow=lpow, eigen=True, divfree=divfree)
        err = rel_l2(host(d), soa(ref))
        assert err <= TOL, (inverse, err)


def test_round_trip_identity():
    """L(L^-1 f) = f on the GPU (DiffOperRoutineTests.cxx:120-158)."""
    from atlaswerks_amd.fluid import DiffOperGPU
    from gpu_util import host, rel_l2, to_dev
    shape = (32, 32, 32)
    f = _field(shape, seed=11)
    op = DiffOperGPU((32, 32, 32), (1.0, 1.25, 1.0))
    d = to_dev(f)
    op.ApplyInverseOperator(d)
    op.ApplyOperator(d)
    assert rel_l2(host(d), f) <= 1e-5


@pytest.mark.parametrize("knobs", [{"fft_order": 1}, {"x_rt": 2}, {"x_rt": 4, "y_tx": 2, "z_tx": 1},
                                   {"fft_order": 1, "x_rt": 6, "y_tx": 4, "z_tx": 2}])
@pytest.mark.parametrize("shape", [(24, 40, 36), (36, 48, 60), (12, 20, 67), (128, 128, 128)])
def test_tuned_fft_plans_match_oracle(shape, knobs):
    """Axes with two radices, a dense product or a kernel of their own under plan knobs
    (which only other lengths read, see the staged axes below): L^-1 within the same 1e-5
    of the FP64 oracle."""
    from atlaswerks_amd import autotune
    from atlaswerks_amd.fluid import DiffOperGPU, DiffOperParam
    from gpu_util import aos, host, rel_l2, soa, to_dev
    nz, ny, nx = shape
    print("fluid plan", shape, knobs, flush=True)
    f = _field(shape, seed=11)
    sp = (1.0, 1.25, 0.8)
    try:
        for k, v in knobs.items():
            autotune.set_knob(k, v)
        op = DiffOperGPU((nx, ny, nz), sp, DiffOperParam(alpha=0.01, beta=0.01, gamma=0.001))
    finally:
        for k in autotune.PLAN_KNOBS:
            autotune.set_knob(k, 0)
    d = to_dev(f)
    op.ApplyInverseOperator(d)
    ref = oracle.diffoper(aos(f), sp=sp, alpha=0.01, beta=0.01, gamma=0.001, inverse=True)
    assert rel_l2(host(d), soa(ref)) <= TOL


# A length with a prime factor above 13 is transformed as a matrix product in tiles of
# 32 outputs k <= n / 2: the first such length, one short of / exactly / one past one,
# two, four and eight tiles, and the two sides of the longest (511)
DENSE_LENGTHS = [17, 19, 61, 62, 67, 127, 134, 251, 254, 257, 262, 502, 509, 511, 514]


@pytest.mark.parametrize("axis", [0, 1, 2])
@pytest.mark.parametrize("n", DENSE_LENGTHS)
def test_dense_axis_matches_oracle(n, axis):
    """L^-1 with one dense axis.  Bar: the two transforms of that axis, each a sum of
    n / 2 terms in runs of 16 (n = 511: 16 runs, so at most about 2 sqrt(16) roundings
    of 2^-24 in the mean square and the folds before and after: 6e-7), four short ones
    and the solve (5e-7): 1.7e-6."""
    from atlaswerks_amd.fluid import DiffOperGPU, DiffOperParam
    from gpu_util import aos, host, rel_l2, soa, to_dev
    shape = [5, 12, 9]
    shape[axis] = n
    nz, ny, nx = shape
    print("fluid dense", shape, flush=True)
    f = _field(tuple(shape), seed=n + axis)
    sp = (1.0, 1.25, 0.8)
    op = DiffOperGPU((nx, ny, nz), sp, DiffOperParam(alpha=0.01, beta=0.01, gamma=0.001))
    d = to_dev(f)
    op.ApplyInverseOperator(d)
    ref = oracle.diffoper(aos(f), sp=sp, alpha=0.01, beta=0.01, gamma=0.001, inverse=True)
    assert rel_l2(host(d), soa(ref)) <= 1.7e-6


@pytest.mark.parametrize("shape", [(23, 19, 37), (34, 20, 62), (17, 29, 67)])
def test_dense_axes_greedy_matches_oracle(shape):
    """The force, energy and composition of the greedy step around dense axes, row
    groups that end inside a plane among them: energies and field as the greedy parity
    tests' bars (1e-3, relative L2 1e-5), single and back-to-back iterations alike."""
    import torch
    from atlaswerks_amd.greedy import GreedyWarp
    from gpu_util import host, rel_l2, soa
    print("greedy dense", shape, flush=True)
    t, h, _ = synth.pair(shape, seed=2, max_disp=1.5)
    target = oracle.apply(t, np.moveaxis(h, 0, -1), dtype=np.float32)
    hd, _, _, ed, _ = oracle.greedy_run(t, target, 6)
    I0, I1 = torch.from_numpy(t).cuda(), torch.from_numpy(target).cuda()
    w = GreedyWarp(I0, I1, 6)
    data = w.RunWarp()
    assert np.max(np.abs(data.energies() - ed) / ed) < 1e-3
    assert rel_l2(host(data.Def1To0), soa(hd)) <= 1e-5


# A length with two radices up to 32 (prime factors up to 13) is transformed in
# registers: every radix as the larger and most as the smaller of the two, one radix
# alone, and the longest
RADIX_LENGTHS = [2, 3, 7, 11, 13, 14, 26, 39, 44, 60, 72, 80, 110, 143, 165, 168, 182, 195, 208, 240, 270, 286,
                 315, 320, 325, 384, 405, 416, 420, 448, 450, 810, 960, 1024]


@pytest.mark.parametrize("axis", [0, 1, 2])
@pytest.mark.parametrize("n", RADIX_LENGTHS)
def test_radix_axis_matches_oracle(n, axis):
    """L^-1 with one long two-radix axis.  Bar: six transforms of at most 10 levels of
    butterflies (2^-24 each in the mean square, sqrt(60) in all: 4.6e-7) and the solve
    (5e-7): 1e-6."""
    from atlaswerks_amd.fluid import DiffOperGPU, DiffOperParam
    from gpu_util import aos, host, rel_l2, soa, to_dev
    shape = [5, 12, 9]
    shape[axis] = n
    nz, ny, nx = shape
    print("fluid radix", shape, flush=True)
    f = _field(tuple(shape), seed=n + axis)
    sp = (1.0, 1.25, 0.8)
    op = DiffOperGPU((nx, ny, nz), sp, DiffOperParam(alpha=0.01, beta=0.01, gamma=0.001))
    d = to_dev(f)
    op.ApplyInverseOperator(d)
    ref = oracle.diffoper(aos(f), sp=sp, alpha=0.01, beta=0.01, gamma=0.001, inverse=True)
    assert rel_l2(host(d), soa(ref)) <= 1e-6


@pytest.mark.parametrize("shape", [(6, 20, 40), (5, 16, 64), (5, 11, 100), (4, 9, 150), (3, 10, 300), (3, 21, 134),
                                   (1, 16, 40), (16, 1, 48), (2, 24, 17)])
def test_force_columns_match_oracle(shape):
    """The force formed by columns (quarters, halves or all of a block's rows per
    thread) and voxel by voxel (row groups over a plane's end, rows longer than the
    block) in one grid: the greedy parity tests' bars."""
    import torch
    from atlaswerks_amd.greedy import GreedyWarp
    from gpu_util import host, rel_l2, soa
    print("greedy columns", shape, flush=True)
    t, h, _ = synth.pair(shape, seed=4, max_disp=1.0)
    target = oracle.apply(t, np.moveaxis(h, 0, -1), dtype=np.float32)
    sp = (1.2, 0.9, 1.0)
    hd, _, _, ed, _ = oracle.greedy_run(t, target, 4, sp=sp)
    data = GreedyWarp(torch.from_numpy(t).cuda(), torch.from_numpy(target).cuda(), 4, spacing=sp).RunWarp()
    assert np.max(np.abs(data.energies() - ed) / ed) < 1e-3
    assert rel_l2(host(data.Def1To0), soa(hd)) <= 1e-5


# Axes that run the LDS stages: small primes without two radices up to 32 (343 = 7^3, 245,
# 429), chirp-z past the dense lengths (514 = 2 * 257), and a single voxel; rows past the
# two-radix lengths (1100); row groups over a plane's end and past the volume's
STAGED_SHAPES = [(3, 7, 343), (2, 5, 514), (3, 11, 1), (2, 3, 1100), (3, 343, 6), (2, 514, 5), (245, 4, 6),
                 (514, 3, 5), (7, 5, 429)]


def _axis_staged(shape):
    from atlaswerks_amd import _lib
    return [bool(_lib.load().awk_fft_axis_staged(a, n)) for a, n in enumerate(shape[::-1])]


@pytest.mark.parametrize("knobs", [{}, {"fft_order": 1}, {"x_rt": 2}, {"x_rt": 4, "y_tx": 2, "z_tx": 1},
                                   {"fft_order": 1, "x_rt": 6, "y_tx": 4, "z_tx": 2}])
@pytest.mark.parametrize("shape", STAGED_SHAPES)
def test_staged_axis_plans_match_oracle(shape, knobs):
    """L^-1 with an axis that reads the plan knobs, under each of the plans the autotuner
    chooses between.  Bar: the operator tests' 1e-5."""
    from atlaswerks_amd import autotune
    from atlaswerks_amd.fluid import DiffOperGPU, DiffOperParam
    from gpu_util import aos, host, rel_l2, soa, to_dev
    nz, ny, nx = shape
    print("fluid staged", shape, knobs, flush=True)
    assert any(_axis_staged(shape))
    f = _field(shape, seed=13)
    sp = (1.0, 1.25, 0.8)
    try:
        for k, v in knobs.items():
            autotune.set_knob(k, v)
        op = DiffOperGPU((nx, ny, nz), sp, DiffOperParam(alpha=0.01, beta=0.01, gamma=0.001))
    finally:
        for k in autotune.PLAN_KNOBS:
            autotune.set_knob(k, 0)
    d = to_dev(f)
    op.ApplyInverseOperator(d)
    ref = oracle.diffoper(aos(f), sp=sp, alpha=0.01, beta=0.01, gamma=0.001, inverse=True)
    assert rel_l2(host(d), soa(ref)) <= TOL


@pytest.mark.parametrize("shape", STAGED_SHAPES)
def test_staged_axes_greedy_matches_oracle(shape):
    """The force, energy, composition and next deformed image around the LDS stages: the
    greedy parity tests' bars."""
    import torch
    from atlaswerks_amd.greedy import GreedyWarp
    from gpu_util import host, rel_l2, soa
    print("greedy staged", shape, flush=True)
    t, h, _ = synth.pair(shape, seed=4, max_disp=1.0)
    target = oracle.apply(t, np.moveaxis(h, 0, -1), dtype=np.float32)
    sp = (1.2, 0.9, 1.0)
    hd, _, _, ed, _ = oracle.greedy_run(t, target, 4, sp=sp)
    data = GreedyWarp(torch.from_numpy(t).cuda(), torch.from_numpy(target).cuda(), 4, spacing=sp).RunWarp()
    assert np.max(np.abs(data.energies() - ed) / ed) < 1e-3
    assert rel_l2(host(data.Def1To0), soa(hd)) <= 1e-5


# Mean relative error against 64 bits of L^-1 through the mixed-radix LDS stages that the
# plans of these lengths took the place of (the seeds and spacing below)
STAGES_ERROR = [((36, 36, 36), 4, 1.894e-7), ((42, 42, 42), 4, 1.941e-7), ((84, 84, 84), 4, 2.116e-7),
                ((100, 100, 100), 2, 2.161e-7), ((30, 30, 30), 4, 1.566e-7), ((5, 200, 12), 2, 1.347e-7),
                ((34, 34, 34), 4, 2.087e-7), ((51, 51, 51), 4, 2.126e-7), ((68, 68, 68), 4, 2.094e-7),
                ((85, 85, 85), 4, 2.146e-7)]


@pytest.mark.parametrize("shape,seeds,stages", STAGES_ERROR)
def test_operator_error_is_no_larger_than_the_stages(shape, seeds, stages):
    """A plan is no less precise than what it replaced: the mean error over the seeds within
    2 % of the stages' (the spread of the ratio between such sets of seeds)."""
    from atlaswerks_amd.fluid import DiffOperGPU, DiffOperParam
    from gpu_util import aos, host, rel_l2, soa, to_dev
    nz, ny, nx = shape
    print("fluid error", shape, flush=True)
    sp = (1.0, 1.25, 0.8)
    op = DiffOperGPU((nx, ny, nz), sp, DiffOperParam(alpha=0.01, beta=0.01, gamma=0.001))
    err = []
    for seed in range(1, seeds + 1):
        f = _field(shape, seed)
        d = to_dev(f)
        op.ApplyInverseOperator(d)
        ref = oracle.diffoper(aos(f), sp=sp, alpha=0.01, beta=0.01, gamma=0.001, inverse=True)
        err.append(rel_l2(host(d), soa(ref)))
    assert np.mean(err) <= 1.02 * stages, np.mean(err) / stages
