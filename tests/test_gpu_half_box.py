"""3-body energies where two oxygens of a trimer are half the box apart.

Waters on a lattice of four cells an axis: every second neighbour is at L/2 up to rounding, where the
minimum image is a matter of the last bit of (a - c) / L.  The pair itself is beyond the cutoff, but
which image of c is taken decides its distance from b, and so a whole trimer.  The kernels form the
quotient as the oracle (and the list's own filter) does; edges for which the product with 1/L rounds
to another index on some lattice separation.

Tolerance: the parity tests' (1e-9 of the energy, 1e-8 of the RMS force): FP64 sums in another order.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope='module')
def mb():
    import mbpol_openmm_plugin_amd as m
    if m.device_count() < 1:
        pytest.fail('no GPU visible to libmbpol_hip.so')
    return m


def lattice(L):
    x = (np.arange(4) + 0.5) * L / 4
    oxygen = np.stack(np.meshgrid(x, x, x, indexing='ij'), axis=-1).reshape(-1, 3)
    rng = np.random.default_rng(7)
    h = np.array([[0.0, 0.0, 0.0], [0.0757, 0.0586, 0.0], [-0.0757, 0.0586, 0.0]])
    turn = np.linalg.qr(rng.normal(size=(len(oxygen), 3, 3)))[0]
    return oxygen[:, None] + h @ turn, x


@pytest.mark.parametrize('kernel', ['orbit', 'terms'])
@pytest.mark.parametrize('L', [1.143, 1.281, 1.396, 1.46, 1.47])
def test_threebody_at_half_the_box(mb, oracle, monkeypatch, L, kernel):
    waters, x = lattice(L)
    d = x[:, None] - x[None]
    assert (np.floor(d / L + 0.5) != np.floor(d * (1.0 / L) + 0.5)).any()
    monkeypatch.setenv('MBPOL_HIP_3B_KERNEL', kernel)
    sysm = mb.forcefield.create_system(len(waters), nonbonded_method='PME', box=L, components=4)
    pos = mb.forcefield.water_positions_with_m(waters)
    ctx = mb.Context(sysm, precision='double')
    ctx.setPositions(pos)
    st = ctx.getState(components=4)
    E, F = oracle.evaluate_system(sysm, pos, components=4)
    err = np.sqrt(np.mean((st.getForces() - F) ** 2) / np.mean(F ** 2))
    print(L, kernel, st.getPotentialEnergy(), E['threebody'], 'force rel rms %.2g' % err, flush=True)
    assert abs(st.getPotentialEnergy() - E['threebody']) <= 1e-9 * abs(E['threebody'])
    assert err <= 1e-8
