"""Host side of the library without a GPU: device memory that a solver takes and the kernels that it launches,
against a stand-in HIP runtime that records launches (tests/isa/hostsim.py). Each test runs in a process of its
own, since the stand-in has to be loaded before the library."""
import os
import subprocess
import sys

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
PRE = f"""
import sys
sys.path[:0] = [{os.path.join(HERE, 'isa')!r}]
import hostsim
sim = hostsim.HostSim()
from cgfdm_amd import model as M, solver as S
"""


def run(code):
    r = subprocess.run([sys.executable, "-c", PRE + code], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stdout[-2000:] + r.stderr[-3000:]


@pytest.mark.parametrize("precision", [4, 8])
@pytest.mark.parametrize("free_surface", [True, False])
def test_absorbing_frame_takes_three_states(precision, free_surface):
    """The auxiliary state of a slab cell is kept three times (9 components): the state at the step's start and two
    stage buffers. With a buffer for each stage state a grid that filled the memory no longer fitted."""
    run(f"""
used = []
for npml in (0, 7):
    m = M.small_config(nx=31, ny=26, nz=22, npml=npml, free_surface={free_surface}, nt=4)
    g = S.Solver(m, precision={precision})
    used.append(g.device_bytes())
    assert used[-1] == sim.used
    g.close()
cells = 7 * (2 * 26 * 22 + 2 * 31 * 22 + {1 if free_surface else 2} * 31 * 26)
assert used[1] - used[0] == 27 * cells * {precision}, (used, cells)
""")
