"""A kernel that cannot be launched makes the call fail, on either stream and thread.

The process loads tests/host/refuse_launch.cpp before the package, which has the HIP runtime refuse
the launches of one kernel by name (on the host: nothing of it reaches the GPU).  Kernels whose absence
leaves every index in bounds are chosen: they only add into, or convert, what others have written.  The
next evaluation, with the launch back, gives the same energies as before.
"""
import os
import subprocess
import sys

import pytest

pytestmark = pytest.mark.gpu

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.abspath(os.path.join(HERE, '..'))

CHILD = r'''
import ctypes, sys
refuse = ctypes.CDLL(sys.argv[2], mode=ctypes.RTLD_GLOBAL)
sys.path.insert(0, sys.argv[1])
import numpy as np
import mbpol_openmm_plugin_amd as mb
waters, L = mb.systems.config1()
sysm = mb.forcefield.create_system(256, nonbonded_method='PME', box=L, ewald_error_tolerance=1e-5, dipole_epsilon=1e-6)
ctx = mb.Context(sysm, precision='mixed')
ctx.setPositions(mb.forcefield.water_positions_with_m(waters))
for _ in range(2):
    want = ctx.getState().getComponentEnergies()
pts = np.random.default_rng(1).uniform(0, L, (10, 3))
def refused(name, call):
    refuse.refuse_name(name.encode())
    refuse.refused()
    try:
        call()
        error = None
    except mb.MBPolError as e:
        error = str(e)
    n = refuse.refused()
    refuse.refuse_name(b'')
    print(name, 'refused', n, 'error', error, flush=True)
    assert n > 0, name
    assert error and 'launch' in error, name
    again = ctx.getState().getComponentEnergies()
    assert again == want, (name, again, want)
for name in ('k_forces_to_double', 'k_pip_split', 'k_disp_finish', 'k_add_forces_fix'):
    refused(name, ctx.getState)
refused('k_potential_at_points', lambda: ctx.getElectrostaticPotential(pts))
refused('k_system_moments', ctx.getSystemElectrostaticsMoments)
md = mb.LangevinIntegrator(ctx, 300.0, 5.0, 0.0005)
refused('k_md_thermostat', lambda: md.step(1))
print('__DONE__', flush=True)
'''


@pytest.mark.parametrize('fork', ['thread', 'early', 'late'])
def test_refused_launch_is_an_error(tmp_path, fork):
    lib = str(tmp_path / 'librefuse.so')
    subprocess.check_call(['g++', '-O1', '-std=c++17', '-fPIC', '-shared', os.path.join(HERE, 'host', 'refuse_launch.cpp'),
                           '-o', lib, '-ldl'])
    env = dict(os.environ, MBPOL_HIP_FORK=fork, MBPOL_HIP_TUNE='0')
    p = subprocess.run([sys.executable, '-u', '-c', CHILD, ROOT, lib], env=env, timeout=100, stdout=subprocess.PIPE,
                       stderr=subprocess.STDOUT, text=True)
    print(p.stdout, flush=True)
    assert p.returncode == 0 and '__DONE__' in p.stdout
