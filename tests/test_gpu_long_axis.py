"""PME electrostatics of a box that is long in z against the same box with x and z exchanged.

Spreading goes by grid lines along z, which are cut into segments of 64 to 127 points: one short
segment and lengths around two, several, segments of unequal length, and lines of more points than
one block's LDS would hold (over 1204).  Lengths for the dense products, the mixed radix and the
library transforms, with the spreading in the z pass and before it.

Tolerance: energies and forces of mirrored systems are equal up to FP64 rounding, which the transforms
(relative 1e-14), the cancelling charges (1e3) and 60 applications in the solver bound by 1e-10, as
for the transforms' own tests.
"""
import os

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope='module')
def mb():
    import mbpol_openmm_plugin_amd as m
    if m.device_count() < 1:
        pytest.fail('no GPU visible to libmbpol_hip.so')
    return m


def waters_in(box, lattice):
    rng = np.random.default_rng(11)
    site = np.stack(np.meshgrid(*(np.arange(c) for c in lattice), indexing='ij'), axis=-1).reshape(-1, 3)
    oxygen = (site + 0.5) * np.array(box) / np.array(lattice) + rng.uniform(-0.015, 0.015, (len(site), 3))
    h = np.array([[0.0, 0.0, 0.0], [0.0757, 0.0586, 0.0], [-0.0757, 0.0586, 0.0]])
    turn = np.linalg.qr(rng.normal(size=(len(site), 3, 3)))[0]
    return oxygen[:, None] + h @ turn + rng.integers(-1, 2, (len(site), 1, 3)) * np.array(box)


def evaluate(mb, waters, box, grid):
    sysm = mb.forcefield.create_system(len(waters), nonbonded_method='PME', box=box, ewald_alpha=3.4, pme_grid=grid,
                                       dipole_epsilon=1e-8, components=16)
    ctx = mb.Context(sysm, precision='mixed')
    ctx.setPositions(mb.forcefield.water_positions_with_m(waters))
    st = ctx.getState(components=16)
    return st.getPotentialEnergy(), st.getForces(), st.stats['iterations']


@pytest.mark.parametrize('nz, env', [
    (127, {'MBPOL_HIP_SPREAD_FUSED': '0'}),  # one segment
    (128, {'MBPOL_HIP_SPREAD_FUSED': '0'}),  # two
    (191, {'MBPOL_HIP_SPREAD_FUSED': '0'}),  # two of unequal length
    (192, {'MBPOL_HIP_PME_FFT': 'radix'}),   # three, before the mixed-radix z pass
    (324, {}),                               # smooth and above the dense z pass
    (499, {}),                               # dense, 16 whole lines
    (512, {}),
    (521, {}),                               # no form of its own: library transforms
    (1000, {}),
    (1204, {}),
    (1205, {}),
    (1536, {}),
])
def test_long_z_as_long_x(mb, monkeypatch, nz, env):
    for k in ('MBPOL_HIP_SPREAD_FUSED', 'MBPOL_HIP_PME_FFT'):
        monkeypatch.delenv(k, raising=False)
    box, lattice = np.array([1.9, 2.1, 6.2]), (6, 6, 18)
    waters = waters_in(box, lattice)
    e1, f1, n1 = evaluate(mb, waters[:, :, ::-1], box[::-1], (nz, 20, 18))
    for k, v in env.items():
        monkeypatch.setenv(k, v)
    e0, f0, n0 = evaluate(mb, waters, box, (18, 20, nz))
    rel = np.sqrt(np.mean((f1[:, ::-1] - f0) ** 2) / np.mean(f0 ** 2))
    print(nz, env, 'energy %.10f vs %.10f' % (e0, e1), 'forces %.2g' % rel, 'iterations', n0, n1, flush=True)
    assert n0 == n1
    assert abs(e0 - e1) <= 1e-10 * abs(e1)
    assert rel <= 1e-10
