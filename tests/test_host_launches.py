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


@pytest.mark.parametrize("scheme,precision", [("CGFDM", 4), ("CGFDM", 8), ("AWENO", 4), ("AWENO", 8)])
def test_staging_buffer_gives_way_to_the_solver(scheme, precision):
    """The buffer that fields and slices are packed into takes only memory that is left: a grid that fits without it
    is made, station records that fit without it too, and fields and slices are still copied, row by row if need
    be."""
    run(f"""
import numpy as np
def make():
    m = M.small_config(nx=40, ny=33, nz=30, npml=4, nt=4)
    m.stations, m.src_cells, m.src_rate = None, None, None
    return m, S.Solver(m, precision={precision}, scheme=S.SCHEME_{scheme})
def copies(g):
    for c in range(9):
        g.set_field(c, np.zeros(g.shape))
        assert g.field(c).shape == g.shape
        assert g.slice(c, 0, 5).size == 33 * 30 and g.slice(c, 1, 5).size == 40 * 30 and g.slice(c, 2, 5).size == 40 * 33
    g.step(1)
    g.synchronize()
def pieces(g):
    sim.names()
    g.field(3)
    return sim.names().count('k_gather')
m, g = make()
full, stage = g.device_bytes(), 8 * g.N
assert pieces(g) == 1
g.close()
assert sim.used == 0
sim.limit = full - stage + 8 * 46  # the grid and one row of 46
m, g = make()
assert pieces(g) == 39 * 36
copies(g)
g.close()
sim.limit = full + 4096
m, g = make()
assert pieces(g) == 1
n = (4096 + stage // 2) // (4 * 9 * 4)
S._check(g.L.cgfdm_set_stations(g.h, n, S._ptr(np.full((n, 3), 5, np.int32))))
assert 1 < pieces(g) < 40 and g.device_bytes() == sim.used <= sim.limit
copies(g)
g.close()
""")


@pytest.mark.parametrize("scheme,precision,coef,size", [
    ("CGFDM", 4, 0, (24, 20, 16)), ("CGFDM", 4, 1, (24, 20, 16)), ("CGFDM", 8, 0, (24, 20, 16)),
    ("CGFDM", 4, 0, (130, 100, 26)), ("AWENO", 4, 0, (24, 20, 16)), ("AWENO", 8, 0, (24, 20, 16)),
    ("AWENO", 4, 0, (70, 90, 40))])
@pytest.mark.parametrize("free_surface", [True, False])
def test_timing_and_names_describe_the_launches_of_a_step(scheme, precision, coef, size, free_surface):
    """Kernel timing times the launches that a step makes without it, and the kernel names are names of them."""
    run(f"""
m = M.small_config(nx={size[0]}, ny={size[1]}, nz={size[2]}, npml=4, nt=8, free_surface={free_surface})
g = S.Solver(m, precision={precision}, coef_storage={coef}, scheme=S.SCHEME_{scheme})
sim.launches.clear()
g.step(2)
plain = list(sim.launches)
sim.launches.clear()
g.timing(True)
g.step(2)
t = g.timing(False)
assert sim.launches == plain, (plain, sim.launches)
names = [n for n, _ in plain]
stages = 4 if '{scheme}' == 'CGFDM' else 3
assert names.count(g.kernel_name(0)) == 2 * stages == t['interior_n'], (g.kernel_name(0), names)
if '{scheme}' == 'AWENO' or {free_surface}:
    assert names.count(g.kernel_name(1)) == 2 * stages, (g.kernel_name(1), names)
    assert t['surface_n'] == (0 if g.kernel_name(1) == 'cg_stage' else 2 * stages)
""")


def test_no_fp64_kernel_of_both_updates():
    """The one launch of both ME-AWENO updates is for FP32 only: an FP64 instance would be compiled for nothing."""
    lib = os.path.join(os.path.dirname(HERE), "cgfdm3d-eqr-sc_amd", "cgfdm_amd", "libcgfdm_amd.so")
    with open(lib, "rb") as f:
        names = f.read()
    assert b"aw14aw_update_bothIf" in names and b"aw14aw_update_bothId" not in names


@pytest.mark.parametrize("size,march", [((59, 90, 78), False), ((400, 400, 6), False), ((64, 60, 40), False),
                                        ((250, 240, 4), False), ((100, 150, 130), True), ((160, 150, 90), True)])
def test_marching_kernels_where_they_are_faster(size, march):
    """ME-AWENO in FP32: grids that are thin, or narrow with half-empty waves, take the kernels with the flux array,
    which are the faster ones there by a fifth (measured); deep ones of a million cells and more march."""
    run(f"""
m = M.small_config(nx={size[0]}, ny={size[1]}, nz={size[2]}, npml=0, nt=4, hills=0, layered=False)
g = S.Solver(m, precision=4, scheme=S.SCHEME_AWENO)
assert g.kernel_name(0) == ('aw_yflux' if {march} else 'aw_faces'), g.kernel_name(0)
""")
