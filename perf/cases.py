"""The work whose speed this repository is measured on.

A case is one call (or a few MD steps) that a program using the package makes
again and again: an energy+force evaluation of a whole system through the
Force/Context API, one Force of it on positions resident on the GPU, Langevin
steps, a batch of independent clusters, or the electrostatic potential on a
grid of points.  Sizes run from a 14-water cluster, where launches and
latency count, to a 13,824-water periodic box, and most are not powers of two.

``prepare`` builds synthetic water from the seed: oxygens on a lattice of
liquid density (or of a loose cluster), each moved at random inside the space
that keeps O-O distances above 2.6 Angstrom, with randomly oriented monomers of
thermal bond lengths and angles.  A program keeps one Context for its system
and hands it new positions; so the ``state`` and ``map`` cases share one
Context among the states of a case.  Where positions stay on the GPU, each
state owns its Context.
"""
import math

import numpy as np
import torch

from mbpol_openmm_plugin_amd import api, forcefield

SPACING = 0.31037  # nm per lattice cell at the density of a 4096-water, 4.966 nm box
TERMS = {'all': api.MBPOL_ALL, 'twobody': api.MBPOL_TWOBODY, 'threebody': api.MBPOL_THREEBODY,
         'dispersion': api.MBPOL_DISPERSION, 'electrostatics': api.MBPOL_ELECTROSTATICS}


def _box(waters, nx, ny, nz, lx=None, ly=None, lz=None):
    """A periodic box holding `waters` waters on an nx x ny x nz lattice (edges in nm)."""
    return {'waters': waters, 'nx': nx, 'ny': ny, 'nz': nz, 'lx': lx or round(nx * SPACING, 4),
            'ly': ly or round(ny * SPACING, 4), 'lz': lz or round(nz * SPACING, 4)}


def listed():
    return [
        # the smallest whole evaluation: a gas-phase cluster without cutoffs, one call per step of an outer program
        dict(name='cluster 14', kind='state', precision='mixed', terms='all', waters=14),
        # the smallest periodic box of the tests (256 waters, 19.71 Angstrom), all terms
        dict(name='box 256', kind='state', precision='mixed', terms='all',
             **_box(256, 7, 7, 6, 1.971, 1.971, 1.971)),
        # a box that does not fill its lattice, in the reference's own arithmetic and dipole iteration
        dict(name='box 500 double', kind='state', precision='double', terms='all', **_box(500, 8, 8, 8)),
        # the benchmark's box, positions and forces on the host side as an MD engine hands them over
        dict(name='box 4096', kind='state', precision='mixed', terms='all', **_box(4096, 16, 16, 16)),
        # the largest box, positions resident on the GPU
        dict(name='box 13824', kind='resident', precision='mixed', terms='all', **_box(13824, 24, 24, 24)),
        # dynamics: Langevin steps on resident positions, each solve started from the last step's dipoles
        dict(name='md 1000', kind='md', precision='mixed', terms='all', steps=4, **_box(1000, 10, 10, 10)),
        # many independent clusters of 3 to 64 waters in one evaluation (energy of every cluster)
        dict(name='clusters 512', kind='batch', precision='mixed', terms='all', clusters=512, smallest=3, most=64),
        # one Force each, as a program that sums force groups itself or times them calls it
        dict(name='two-body 2700', kind='resident', precision='mixed', terms='twobody', **_box(2700, 14, 14, 14)),
        dict(name='three-body 3000', kind='resident', precision='mixed', terms='threebody', **_box(3000, 14, 15, 15)),
        dict(name='electrostatics 2197', kind='resident', precision='mixed', terms='electrostatics',
             **_box(2197, 13, 13, 13)),
        dict(name='dispersion 5000', kind='resident', precision='mixed', terms='dispersion', **_box(5000, 17, 17, 18)),
        # the electrostatic potential on a grid of points around the molecules of a box
        dict(name='map 256', kind='map', precision='mixed', terms='electrostatics', points=8000,
             **_box(256, 7, 7, 6, 1.971, 1.971, 1.971)),
    ]


def _log_uniform(rng, a, b):
    return int(round(math.exp(rng.uniform(math.log(a), math.log(b)))))


def _draw_box(rng, fewest, most):
    """A box of about log-uniform size, not cubic in general, with up to an eighth of its lattice empty."""
    n = _log_uniform(rng, fewest, most)
    while True:
        side = n ** (1.0 / 3.0)
        nx, ny = (max(6, int(round(side * rng.uniform(0.85, 1.15)))) for _ in range(2))
        nz = max(6, -(-n // (nx * ny)))
        if 0.85 * nx * ny * nz <= n <= nx * ny * nz:
            return _box(n, nx, ny, nz)
        n += rng.randint(1, 40)


def draw(rng):
    """One more case of the same ranges: every kind, its sizes spread over the logarithm of their range."""
    kind = rng.choice(['cluster', 'box', 'box', 'box', 'double', 'resident', 'md', 'batch', 'force', 'force', 'map'])
    if kind == 'cluster':
        return dict(kind='state', precision='mixed', terms='all', waters=_log_uniform(rng, 3, 64))
    if kind == 'box':
        return dict(kind='state', precision='mixed', terms='all', **_draw_box(rng, 216, 6000))
    if kind == 'double':
        return dict(kind='state', precision='double', terms='all', **_draw_box(rng, 216, 2000))
    if kind == 'resident':
        return dict(kind='resident', precision='mixed', terms='all', **_draw_box(rng, 1000, 12000))
    if kind == 'md':
        return dict(kind='md', precision='mixed', terms='all', steps=4, **_draw_box(rng, 216, 3000))
    if kind == 'batch':
        return dict(kind='batch', precision='mixed', terms='all', clusters=_log_uniform(rng, 16, 700), smallest=3,
                    most=rng.randint(12, 64))
    if kind == 'map':
        return dict(kind='map', precision='mixed', terms='electrostatics', points=_log_uniform(rng, 50, 20000),
                    **_draw_box(rng, 216, 1500))
    terms = rng.choice(['twobody', 'threebody', 'electrostatics', 'dispersion'])
    return dict(kind='resident', precision='double' if terms == 'dispersion' and rng.random() < 0.3 else 'mixed',
                terms=terms, **_draw_box(rng, 216, 6000))


# ---------------------------------------------------------------------------
# water
# ---------------------------------------------------------------------------
def _rng(seed, *more):
    return np.random.Generator(np.random.PCG64([int(seed), *more]))


def _monomers(rng, oxygen):
    """Waters (n, 3, 3) in nm around the oxygens (n, 3): thermal geometry, random orientation."""
    n = len(oxygen)
    r = 0.09572 + rng.normal(0.0, 0.002, (n, 2))
    half = 0.5 * np.deg2rad(104.52 + rng.normal(0.0, 3.0, n))
    q = rng.normal(size=(n, 4))
    a, b, c, d = (q / np.linalg.norm(q, axis=1, keepdims=True)).T
    rot = np.array([[a * a + b * b - c * c - d * d, 2 * (b * c - a * d), 2 * (b * d + a * c)],
                    [2 * (b * c + a * d), a * a - b * b + c * c - d * d, 2 * (c * d - a * b)],
                    [2 * (b * d - a * c), 2 * (c * d + a * b), a * a - b * b - c * c + d * d]]).transpose(2, 0, 1)
    local = np.zeros((n, 3, 3))
    local[:, 1, 0], local[:, 1, 1] = r[:, 0] * np.sin(half), r[:, 0] * np.cos(half)
    local[:, 2, 0], local[:, 2, 1] = -r[:, 1] * np.sin(half), r[:, 1] * np.cos(half)
    return oxygen[:, None, :] + local @ rot.transpose(0, 2, 1)


def _jitter(rng, n, radius):
    """Displacements inside a ball."""
    v = rng.normal(size=(n, 3))
    v /= np.linalg.norm(v, axis=1, keepdims=True)
    return v * (radius * rng.uniform(size=(n, 1)) ** (1.0 / 3.0))


def _box_waters(case, seed):
    rng = _rng(seed, case['waters'])
    cells = [case['nx'], case['ny'], case['nz']]
    step = np.array([case['lx'], case['ly'], case['lz']]) / cells
    site = np.stack(np.meshgrid(*(np.arange(c) for c in cells), indexing='ij'), axis=-1).reshape(-1, 3)
    site = site[np.sort(rng.choice(len(site), size=case['waters'], replace=False))]
    oxygen = (site + 0.5) * step + _jitter(rng, len(site), max(0.0, 0.5 * (step.min() - 0.26)))
    return _monomers(rng, oxygen)


def _cluster_waters(rng, n):
    """n waters of a loose cluster: the lattice points nearest to a random centre."""
    m = 2 + int(math.ceil(n ** (1.0 / 3.0)))
    site = np.stack(np.meshgrid(*(np.arange(m + 1),) * 3, indexing='ij'), axis=-1).reshape(-1, 3)
    centre = 0.5 * m + rng.uniform(-0.5, 0.5, 3)
    near = site[np.argsort(((site - centre) ** 2).sum(axis=1), kind='stable')[:n]]
    return _monomers(rng, (near - centre) * 0.33 + _jitter(rng, n, 0.035))


# ---------------------------------------------------------------------------
# systems and contexts
# ---------------------------------------------------------------------------
def _system(case):
    if 'nx' in case:
        return forcefield.create_system(case['waters'], nonbonded_method='PME',
                                        box=[case['lx'], case['ly'], case['lz']], ewald_error_tolerance=1e-5,
                                        dipole_epsilon=1e-8, components=TERMS[case['terms']])
    return forcefield.create_system(case['waters'], nonbonded_method='CutoffNonPeriodic', twobody_cutoff=1e10,
                                    threebody_cutoff=1e10, nonbonded_cutoff=1e3, dipole_epsilon=1e-8,
                                    components=TERMS[case['terms']])


_kept = {}  # the Context that a program keeps for its system: one, that of the last case asked for


def _kept_context(case):
    key = tuple(sorted((k, v) for k, v in case.items() if k not in ('name', 'points')))
    if key not in _kept:
        _kept.clear()
        _kept[key] = api.Context(_system(case), precision=case['precision'])
    return _kept[key]


def _batch_sizes(case):
    return _rng(case['clusters'], case['most']).integers(case['smallest'], case['most'] + 1, size=case['clusters'])


def prepare(case, seed):
    kind = case['kind']
    if kind not in ('state', 'map'):
        _kept.clear()
    if kind == 'batch':
        sizes, rng = _batch_sizes(case), _rng(seed, case['clusters'])
        system, positions, _ = forcefield.create_cluster_batch([_cluster_waters(rng, int(n)) for n in sizes])
        ctx = api.Context(system, precision=case['precision'])
        ctx.uploadPositions(positions)
        return {'kind': kind, 'ctx': ctx}
    if 'nx' in case:
        waters = _box_waters(case, seed)
    else:
        waters = _cluster_waters(_rng(seed, case['waters']), case['waters'])
    positions = forcefield.water_positions_with_m(waters)
    if kind in ('state', 'map'):
        state = {'kind': kind, 'ctx': _kept_context(case), 'positions': positions}
        if kind == 'map':
            edges = np.array([case['lx'], case['ly'], case['lz']])
            state['points'] = _rng(seed, case['points'], 1).uniform(size=(case['points'], 3)) * edges
        return state
    ctx = api.Context(_system(case), precision=case['precision'])
    if kind == 'resident':
        ctx.uploadPositions(positions)
        return {'kind': kind, 'ctx': ctx, 'dipoles': case['terms'] == 'electrostatics'}
    ctx.setPositions(positions)
    ctx.setDipoleGuess('previous')
    md = api.LangevinIntegrator(ctx, 300.0, 5.0, 0.0005, seed=int(seed) % (1 << 31) + 1)
    return {'kind': kind, 'ctx': ctx, 'md': md, 'steps': case['steps']}


def run(state):
    kind, ctx = state['kind'], state['ctx']
    if kind == 'state':
        ctx.setPositions(state['positions'])
        s = ctx.getState()
        return {'energy': s.getPotentialEnergy(), 'components': s.getComponentEnergies(), 'forces': s.getForces()}
    if kind == 'map':
        ctx.setPositions(state['positions'])
        return {'potential': ctx.getElectrostaticPotential(state['points'])}
    if kind == 'md':
        energies, kinetic = state['md'].step(state['steps'])
        return {'energies': energies, 'kinetic': kinetic, 'positions': state['md'].getPositions()}
    out = {'energies': ctx.evaluateResident(), 'forces': ctx.downloadForces()}
    if kind == 'batch':
        out['clusters'] = ctx.getGroupEnergies()
    elif state['dipoles']:
        out['dipoles'] = ctx.getInducedDipoles()
    return out


# ---------------------------------------------------------------------------
# the work a case cannot do without
# ---------------------------------------------------------------------------
def _sphere(case, radius):
    """Waters within `radius` nm of a point of the box."""
    return case['waters'] / (case['lx'] * case['ly'] * case['lz']) * 4.0 / 3.0 * math.pi * radius ** 3


def work(case):
    """Positions read and forces written once; the polynomials' operations (31.0e3 a dimer, 112.5e3 a
    contributing trimer), about 30 a dispersion pair, and for the electrostatics 300 a site pair, 20 a pair of
    polarisable sites and field evaluation (10 of them) and the grid transforms."""
    if case['kind'] == 'batch':
        sizes = _batch_sizes(case).astype(float)
    else:
        sizes = np.array([float(case['waters'])])
    n = sizes.sum()
    if 'nx' in case:
        dimers = 0.5 * n * _sphere(case, 0.65)
        trimers = 0.25 * n * _sphere(case, 0.45) ** 2
        pairs = 0.5 * n * _sphere(case, 0.9)
        k = math.prod(math.ceil(2 * 3.654826 * case[e] / (3 * 0.1)) for e in ('lx', 'ly', 'lz'))
        grid = 2 * 5.0 * k * math.log2(k) / 2
    else:
        dimers = pairs = float((sizes * (sizes - 1) / 2).sum())
        trimers = float(np.minimum(sizes * (sizes - 1) * (sizes - 2) / 6, 10.0 * sizes).sum())
        grid = 0.0
    term = case['terms']
    flops = 0.0
    if term in ('all', 'twobody'):
        flops += 31.0e3 * dimers
    if term in ('all', 'threebody'):
        flops += 112.5e3 * trimers
    if term in ('all', 'dispersion'):
        flops += 30.0 * 9 * pairs
    if term in ('all', 'electrostatics'):
        flops += 300.0 * 16 * pairs + 10 * (20.0 * 9 * pairs + grid)
    bytes_ = 2 * 96.0 * n
    if case['kind'] == 'map':
        flops += 20.0 * 4 * n * case['points']
        bytes_ = 96.0 * n + 32.0 * case['points']
    times = case.get('steps', 1)
    return {'bytes': times * bytes_, 'flops': times * flops}


def exact(case, seed):
    """The dispersion in 64 bits; the other terms' surfaces have no plain form to compute them by."""
    if case['terms'] != 'dispersion':
        return None
    t = forcefield.tables()['forcefield']
    device = 'cuda' if torch.cuda.is_available() else 'cpu'
    where = dict(dtype=torch.float64, device=device)
    # C6/d6 tables: [first type + 4 * second type], types O, H
    c6 = torch.tensor(t['dispersion_C6'], **where).reshape(4, 4).T
    d6 = torch.tensor(t['dispersion_d6'], **where).reshape(4, 4).T
    n = case['waters']
    x = torch.tensor(_box_waters(case, seed).reshape(-1, 3), **where)
    edges = torch.tensor([case['lx'], case['ly'], case['lz']], **where)
    kind = torch.tensor([0, 1, 1], device=device).repeat(n)
    mol = torch.arange(3 * n, device=device) // 3
    force, energy = torch.zeros_like(x), torch.zeros((), **where)
    for b in range(0, 3 * n, 512):
        d = x[b:b + 512, None, :] - x[None, :, :]
        d -= torch.floor(d / edges + 0.5) * edges
        r2 = (d * d).sum(-1)
        near = (r2 < 0.81) & (mol[b:b + 512, None] != mol[None, :])
        r2 = torch.where(near, r2, torch.ones_like(r2))
        c, k = c6[kind[b:b + 512]][:, kind], d6[kind[b:b + 512]][:, kind]
        r = r2.sqrt()
        y = k * r
        s, term = torch.ones_like(y), torch.ones_like(y)
        for m in range(1, 7):
            term = term * y / m
            s = s + term
        damp = torch.exp(-y)
        tt = 1.0 - s * damp
        slope = 6.0 * c * tt / (r2 ** 3 * r) - c * k * term * damp / r2 ** 3
        near = near.to(torch.float64)
        energy -= 0.5 * (near * c * tt / r2 ** 3).sum()
        force[b:b + 512] = -((near * slope / r)[:, :, None] * d).sum(1)
    full = torch.zeros((n, 4, 3), **where)
    full[:, :3] = force.reshape(n, 3, 3)
    energies = np.zeros(6)
    energies[3] = energies[5] = float(energy)
    return {'energies': energies, 'forces': full.reshape(-1, 3).cpu().numpy()}
