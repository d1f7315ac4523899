"""Results do not depend on what a Context has evaluated before.

The 2- and 3-body lists grow when a configuration needs more room and keep it.  How a unit's passes are
spread over blocks, which shows in the last bits, has to follow from the list's length, not from that room:
the same sparse configuration, in a fresh Context and after a dense one, gives the same bits.  List lengths
for every spread: 1, 2, 3 and 6 blocks a trimer unit, 1 and 2 a dimer unit.
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


def context(mb, n, components, kernel, monkeypatch):
    monkeypatch.setenv('MBPOL_HIP_2B_KERNEL', kernel)
    monkeypatch.setenv('MBPOL_HIP_3B_KERNEL', kernel)
    sysm = mb.forcefield.create_system(n, nonbonded_method='CutoffNonPeriodic', components=components)
    return mb.Context(sysm, precision='double')


def evaluate(mb, ctx, waters, components):
    ctx.setPositions(mb.forcefield.water_positions_with_m(waters))
    st = ctx.getState(components=components)
    return st.getPotentialEnergy(), st.getForces(), st.stats


KEEP = [3, 12, 60, 120, 150, 180, 240]


def dense_box(mb):
    """256 waters with their oxygens drawn together (2.34 Angstrom at least), so that lists are long."""
    box = mb.systems.config1()[0]
    return box - 0.1 * box[:, :1]


def sparse_box(box, keep):
    """The first `keep` waters as they are, the others far from them and from each other."""
    sparse = box.copy()
    sparse[keep:] += np.arange(1, len(box) - keep + 1)[:, None, None] * np.array([5.0, 0.0, 0.0])
    return sparse


@pytest.mark.parametrize('components', [2, 4, 6])
@pytest.mark.parametrize('keep', KEEP)
def test_bits_do_not_depend_on_earlier_configurations(mb, monkeypatch, components, keep):
    box = dense_box(mb)
    sparse = sparse_box(box, keep)
    fresh = context(mb, len(box), components, 'orbit', monkeypatch)
    e0, f0, st = evaluate(mb, fresh, sparse, components)
    caps = [fresh.getTuning(k) for k in ('dimer_capacity', 'trimer_capacity')]
    grown = context(mb, len(box), components, 'orbit', monkeypatch)
    evaluate(mb, grown, box, components)
    e1, f1, _ = evaluate(mb, grown, sparse, components)
    print(keep, components, st['num_dimers'], st['num_trimers'], caps,
          [grown.getTuning(k) for k in ('dimer_capacity', 'trimer_capacity')], flush=True)
    assert e1 == e0
    assert np.array_equal(f1, f0)


def test_lengths_cover_every_split(mb, monkeypatch):
    """The configurations above reach every number of blocks a unit is spread over (256 CUs)."""
    box = dense_box(mb)
    ctx = context(mb, len(box), 6, 'orbit', monkeypatch)
    two, three = set(), set()
    for keep in KEEP:
        st = evaluate(mb, ctx, sparse_box(box, keep), 6)[2]
        units2, units3 = (st['num_dimers'] + 63) // 64, (st['num_trimers'] + 63) // 64
        two.add(2 if 2 * units2 <= 256 else 1)
        three.add(next(q for q in (6, 3, 2, 1) if q * units3 <= 256 or q == 1))
        print(keep, units2, units3, flush=True)
    assert three == {1, 2, 3, 6}
    assert 2 in two


@pytest.mark.parametrize('graph', [False, True])
def test_short_list_after_long_ones(mb, monkeypatch, graph):
    """The kernel that joins units of several blocks is left out of long lists' launches: a list that turns
    short at once, eagerly or in a replayed graph, still gives a fresh Context's bits, and so do long ones."""
    box = mb.systems.config2()[0][:1500]
    few, some = sparse_box(box, 40), sparse_box(box, 400)
    want = {}
    for k, w in (('few', few), ('some', some), ('all', box)):
        want[k] = evaluate(mb, context(mb, len(box), 6, 'orbit', monkeypatch), w, 6)
    assert 64 * 128 < want['all'][2]['num_dimers'] and want['few'][2]['num_dimers'] <= 64 * 128
    ctx = context(mb, len(box), 6, 'orbit', monkeypatch)
    ctx.setGraph(graph)
    waters = {'few': few, 'some': some, 'all': box}
    for k in ('all', 'all', 'all', 'few', 'few', 'all', 'all', 'some', 'few', 'some', 'all', 'all', 'all', 'few'):
        e, f, st = evaluate(mb, ctx, waters[k], 6)
        print(k, st['num_dimers'], st['num_trimers'], e, flush=True)
        assert e == want[k][0]
        assert np.array_equal(f, want[k][1])
    if graph:
        assert ctx.getTuning('graph_replays') > 0
