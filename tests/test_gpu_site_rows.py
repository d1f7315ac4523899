"""Electrostatics neighbour rows (a wave for four sites of the cell order, over their cells' ranges) against brute force.

The number of site pairs within the cutoff and of (polarisable, polarisable) pairs, exactly, in boxes
whose columns cross the boundary on either side, with the fewest cells, with edges of their own per
axis, with ranges of more than 64 members (a dense slab) and empty ones, and without cells.
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


def waters_in(rng, lattice, low, high):
    """One rigid water per lattice cell of the slab low..high (nm)."""
    site = np.stack(np.meshgrid(*(np.arange(c) for c in lattice), indexing='ij'), axis=-1).reshape(-1, 3)
    step = (np.asarray(high) - low) / np.asarray(lattice)
    oxygen = low + (site + 0.5) * step + rng.uniform(-0.01, 0.01, (len(site), 3))
    h = np.array([[0.0, 0.0, 0.0], [0.0757, 0.0586, 0.0], [-0.0757, 0.0586, 0.0]])
    return oxygen[:, None, :] + h


@pytest.mark.parametrize('box, lattice, slab', [
    ((1.9, 1.9, 1.9), (6, 6, 6), None),            # too small for cells
    ((2.25, 2.25, 2.25), (7, 7, 7), None),         # five cells an axis
    ((2.3, 2.75, 3.2), (7, 8, 10), None),
    ((2.71, 2.26, 4.6), (8, 7, 9), None),
    ((2.3, 2.3, 3.0), (9, 9, 10), None),           # cells of about 20 waters: ranges above 64 sites
    ((2.3, 2.3, 6.0), (7, 7, 7), (0.3, 2.4)),      # empty cells
])
def test_row_counts(mb, box, lattice, slab):
    box = np.array(box)
    rng = np.random.default_rng(3)
    low, high = np.zeros(3), box.copy()
    if slab:
        low[2], high[2] = slab
    waters = waters_in(rng, lattice, low, high)
    waters += rng.integers(-1, 2, (len(waters), 1, 3)) * box  # images outside the box
    n = len(waters)
    sysm = mb.forcefield.create_system(n, nonbonded_method='PME', box=box, ewald_alpha=3.4, pme_grid=(32, 32, 36),
                                       dipole_epsilon=1e-2, components=16)
    ctx = mb.Context(sysm, precision='mixed')
    pos = mb.forcefield.water_positions_with_m(waters)
    ctx.setPositions(pos)
    st = ctx.getState(components=16).stats
    polarisable = np.arange(4 * n) % 4 != 3
    pairs = pol = 0
    for b in range(0, 4 * n, 256):
        d = pos[b:b + 256, None] - pos[None]
        d -= np.floor(d / box + 0.5) * box
        near = (d * d).sum(-1) <= 0.81
        near[np.arange(len(near)), np.arange(b, b + len(near))] = False
        pairs += int(near.sum())
        pol += int(near[polarisable[b:b + 256]][:, polarisable].sum())
    print(n, 'waters', st['num_elec_pairs'], pairs // 2, st['num_pol_pairs'], pol, 'lanes', ctx.getTuning('site_lanes'),
          flush=True)
    assert st['num_elec_pairs'] == pairs // 2
    assert st['num_pol_pairs'] == pol
