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


@pytest.mark.parametrize('field, dtype', [('weights', None), ('weights', np.float32), ('weights', np.longdouble),
                                          ('particles', None)])
def test_numpy_sites_called_again(field, dtype):
    """Sites whose weights or particles are arrays, changed in place between calls."""
    system, pos = water_system(5)
    for s in (3, 11):
        site = system._vsites[s]
        setattr(site, field, np.array(getattr(site, field), dtype=dtype))
    for _ in range(3):
        assert np.array_equal(system.computeVirtualSites(pos), loop(system, pos))
    site = system._vsites[11]
    if field == 'weights':
        site.weights[1] = 0.375
    else:
        site.particles[2] = 9
    for _ in range(2):
        assert np.array_equal(system.computeVirtualSites(pos), loop(system, pos))


@pytest.mark.parametrize('particles, weights', [
    ((4.0, 5, 6), (0.5, 0.25, 0.25)),     # not an index
    ((4.5, 5, 6), (0.5, 0.25, 0.25)),
    ((4, 5, 600), (0.5, 0.25, 0.25)),     # no such particle
    ((4, 5, 6), ('0.5', 0.25, 0.25)),     # not numbers
    ((4, 5, 6), (0.5, None, 0.25)),
])
def test_what_the_loop_refuses(particles, weights):
    system, pos = water_system(3)
    site = system._vsites[7]
    site.particles, site.weights = particles, weights
    with pytest.raises(Exception) as plain:
        loop(system, pos)
    for _ in range(2):
        with pytest.raises(plain.type):
            system.computeVirtualSites(pos)


@pytest.mark.parametrize('particles, weights', [
    ((4, 5), (0.5, 0.5)),                       # two parents
    ((-8, 5, 6), (0.5, 0.25, 0.25)),            # from the end
    ((-5, 5, 6), (0.5, 0.25, 0.25)),            # from the end, another site
    ((4, 5, 6), ((0.5, 0.6, 0.7), 0.25, 0.25)),  # a weight per coordinate
    ((4, 5, 6), (1, 0, 0)),
])
def test_what_the_loop_takes(particles, weights):
    system, pos = water_system(3)
    site = system._vsites[7]
    site.particles = particles
    site.weights = tuple(np.array(w) if isinstance(w, tuple) else w for w in weights)
    for _ in range(2):
        assert np.array_equal(system.computeVirtualSites(pos), loop(system, pos))


def test_more_positions_than_particles():
    """Negative indices count from the end of the positions given."""
    system, pos = water_system(3)
    system._vsites[7].particles = (-4, 5, 6)
    longer = np.concatenate([pos, pos + 1.0])
    assert np.array_equal(system.computeVirtualSites(longer), loop(system, longer))


def test_system_without_the_kept_arrays():
    """A System restored from attributes saved before the arrays were kept."""
    system, pos = water_system(4)
    old = mb.System.__new__(mb.System)
    old.__dict__.update({k: v for k, v in system.__dict__.items() if k != '_vsite_arrays'})
    assert np.array_equal(old.computeVirtualSites(pos), loop(old, pos))
