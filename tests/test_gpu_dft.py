"""Dense-product grid transforms (FP64 matrix cores) and mixed-radix ones against the library transforms.

The same PME electrostatics of the 256-water box through the context's own
choice of passes and through hipFFT (MBPOL_HIP_PME_FFT=hipfft, which the parity
tests pin to the FP64 oracle).  Grids cover the edges of the dense form: folded
lengths N/2 + 1 around the 16-output tiles and the 4-input steps, every front
radix (1-4), prime lengths, axes of different forms in one grid, and lengths
whose columns take more than 64 KB of LDS.

Tolerance: both transform in FP64 with a relative rounding error below 1e-14
(under 2^10 terms of a sum); the charges cancel in the energy and forces by at
most 1e3 and the solver applies the operator 60 times, so 1e-10 relative bounds
the difference.
"""
import os

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

GRIDS = [(6, 7, 9), (17, 19, 23), (30, 31, 32), (33, 62, 61), (63, 64, 65), (48, 51, 50), (76, 84, 91), (121, 137, 143),
         (144, 127, 182), (128, 84, 252), (18, 22, 307), (20, 512, 18), (509, 16, 20)]


@pytest.fixture(scope='module')
def mb():
    import mbpol_openmm_plugin_amd as m
    if m.device_count() < 1:
        pytest.fail('no GPU visible to libmbpol_hip.so')
    return m


def evaluate(mb, grid, mode):
    waters, L = mb.systems.config1()
    sysm = mb.forcefield.create_system(256, nonbonded_method='PME', box=L, ewald_alpha=3.4, pme_grid=grid,
                                       dipole_epsilon=1e-8, components=16)
    old = os.environ.pop('MBPOL_HIP_PME_FFT', None)
    if mode:
        os.environ['MBPOL_HIP_PME_FFT'] = mode
    try:
        ctx = mb.Context(sysm, precision='mixed')
    finally:
        os.environ.pop('MBPOL_HIP_PME_FFT', None)
        if old is not None:
            os.environ['MBPOL_HIP_PME_FFT'] = old
    ctx.setPositions(mb.forcefield.water_positions_with_m(waters))
    st = ctx.getState(components=16)
    return st.getPotentialEnergy(), st.getForces(), st.stats['iterations']


@pytest.mark.parametrize('grid', GRIDS, ids=lambda g: 'x'.join(map(str, g)))
def test_dense_passes_match_library_transforms(mb, grid):
    e0, f0, n0 = evaluate(mb, grid, 'hipfft')
    e1, f1, n1 = evaluate(mb, grid, None)
    rel_f = np.sqrt(np.mean((f1 - f0) ** 2) / np.mean(f0 ** 2))
    print(grid, 'energy %.10f vs %.10f' % (e1, e0), 'forces %.2g' % rel_f, 'iterations', n1, n0, flush=True)
    assert n1 == n0
    assert abs(e1 - e0) <= 1e-10 * abs(e0)
    assert rel_f <= 1e-10


# smooth lengths: two to six stages, radices 2 to 13, the longest; z above 320 has mixed-radix z passes by default
RADIX = [(12, 15, 16), (30, 32, 33), (63, 64, 65), (48, 50, 52), (84, 77, 99), (121, 143, 144), (125, 128, 126),
         (18, 20, 324), (16, 18, 512), (16, 512, 18), (512, 18, 16), (16, 18, 1000)]


@pytest.mark.parametrize('mode', ['radix', None])
@pytest.mark.parametrize('grid', RADIX, ids=lambda g: 'x'.join(map(str, g)))
def test_mixed_radix_passes_match_library_transforms(mb, grid, mode):
    e0, f0, n0 = evaluate(mb, grid, 'hipfft')
    e1, f1, n1 = evaluate(mb, grid, mode)
    rel_f = np.sqrt(np.mean((f1 - f0) ** 2) / np.mean(f0 ** 2))
    print(grid, mode, 'energy %.10f vs %.10f' % (e1, e0), 'forces %.2g' % rel_f, 'iterations', n1, n0, flush=True)
    assert n1 == n0
    assert abs(e1 - e0) <= 1e-10 * abs(e0)
    assert rel_f <= 1e-10
