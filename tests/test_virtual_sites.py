"""Placing virtual sites as arrays (System.computeVirtualSites) against the plain loop over sites."""
import numpy as np
import pytest

import mbpol_openmm_plugin_amd as mb


def loop(system, positions):
    pos = np.array(positions, dtype=np.float64).reshape(-1, 3)
    for s, v in system._vsites.items():
        pos[s] = sum(w * pos[p] for p, w in zip(v.particles, v.weights))
    return pos


def water_system(n, dependent=False):
    system = mb.System()
    rng = np.random.default_rng(n)
    for w in range(n):
        for m in (16.0, 1.0, 1.0, 0.0):
            system.addParticle(m)
        a, b = rng.uniform(0.1, 0.4, 2)
        first = 4 * (w - 1) + 3 if dependent and w else 4 * w
        system.setVirtualSite(4 * w + 3, mb.ThreeParticleAverageSite(first, 4 * w + 1, 4 * w + 2, 1 - a - b, a, b))
    return system, rng.normal(size=(4 * n, 3))


# exactly equal: the same products, summed in the same order
@pytest.mark.parametrize('n,dependent', [(0, False), (1, False), (7, False), (300, False), (1, True), (7, True)])
def test_same_positions_as_the_loop(n, dependent):
    system, pos = water_system(n, dependent)
    for _ in range(2):
        assert np.array_equal(system.computeVirtualSites(pos), loop(system, pos))
        pos = pos[::-1].copy()


def test_changed_sites_are_seen():
    system, pos = water_system(5)
    system.computeVirtualSites(pos)
    site = system._vsites[7]
    site.weights = (0.2, 0.3, 0.5)
    assert np.array_equal(system.computeVirtualSites(pos), loop(system, pos))
    site.weights = [0.6, 0.3, 0.1]
    system.computeVirtualSites(pos)
    site.weights[0] = 0.5
    assert np.array_equal(system.computeVirtualSites(pos), loop(system, pos))
    site.particles = (3, 5, 6)  # from another virtual site: one by one
    assert np.array_equal(system.computeVirtualSites(pos), loop(system, pos))
    system.setVirtualSite(11, mb.ThreeParticleAverageSite(-12, 9, 10, 0.5, 0.25, 0.25))
    assert np.array_equal(system.computeVirtualSites(pos), loop(system, pos))
