"""Interior-kernel variants and the tight device layout against the oracle.

The library picks its interior kernel and device layout from environment
knobs read at cgfdm_create (register z-marching with chunks of 5 planes and
of the whole column, x-paired, plane-tile and LDS z-marching interior
kernels; CGFDM_ROW_ALIGN=0 for the tight layout). Each variant steps the
curvilinear PML + free-surface case and must match the FP32 oracle as the
default does (3e-5 relative L2 per field).
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

VARIANTS = [
    ("cgfdm", "CGFDM_INTERIOR_ZREG", "5"),
    ("cgfdm", "CGFDM_INTERIOR_ZREG", "64"),
    ("cgfdm", "CGFDM_INTERIOR_KC", "-1"),
    ("cgfdm", "CGFDM_INTERIOR_KC", "1"),
    ("cgfdm", "CGFDM_INTERIOR_KC", "16"),
    ("cgfdm", "CGFDM_ROW_ALIGN", "0"),
    ("aweno", "CGFDM_ROW_ALIGN", "0"),
]


def rel_l2(a, b):
    n = np.linalg.norm(b)
    return float(np.linalg.norm(np.asarray(a, np.float64) - b) / (n if n > 0 else 1.0))


@pytest.mark.parametrize("scheme,var,val", VARIANTS)
def test_variant_matches_oracle(scheme, var, val, monkeypatch, oracle_mod):
    from cgfdm_amd import solver
    import test_gpu_parity as P
    monkeypatch.setenv(var, val)
    m = P.make("curvilinear_pml_fs")
    print(f"variant {scheme} {var}={val}: {m.nx}x{m.ny}x{m.nz}, FP32, 12 steps", flush=True)
    if scheme == "cgfdm":
        g = solver.Solver(m, precision=4)
        o = oracle_mod.Oracle(m, prec=4, threads=8)
    else:
        g = solver.Solver(m, precision=4, scheme=solver.SCHEME_AWENO)
        o = oracle_mod.AwenoOracle(m, prec=4, threads=8)
    g.step(12)
    g.synchronize()
    o.step(12)
    for v in range(9):
        err = rel_l2(g.field(v), o.field(v))
        assert err < 3e-5, (scheme, var, val, v, err)
    sg, so = g.stations(), o.stations()
    assert rel_l2(sg, so) < 3e-5


# One launch per stage for grids of at most 1024 blocks, two for larger ones, the
# interior's last eight regions cut into eighths: grids on both sides of the line,
# with whole and partial tiles and region counts of 2, 5, 8 and 13.
@pytest.mark.parametrize("nx,ny,nz", [(24, 16, 12), (70, 40, 20), (66, 60, 40), (130, 100, 26)])
@pytest.mark.parametrize("coef", [0, 1])
def test_stage_launches_match_oracle(nx, ny, nz, coef, oracle_mod):
    from cgfdm_amd import model as M
    from cgfdm_amd import solver
    m = M.small_config(nx=nx, ny=ny, nz=nz, npml=4, hills=2, layered=True, free_surface=True, nt=8)
    print(f"{nx}x{ny}x{nz} coef {coef}, FP32, 8 steps", flush=True)
    g = solver.Solver(m, precision=4, coef_storage=coef)
    o = oracle_mod.Oracle(m, prec=4, threads=8)
    g.step(8)
    g.synchronize()
    o.step(8)
    # FP32: as above; fp16 storage: the rounding of the coefficients, 2^-11 of a layer's range, over 8 steps
    tol = 3e-5 if coef == 0 else 5e-3
    for v in range(9):
        err = rel_l2(g.field(v), o.field(v))
        assert err < tol, (nx, ny, nz, coef, v, err)


# The block order from a state that fills the grid, so that a cell left out, done twice or misplaced shows: last
# tile columns of 1, 32 (in blocks of 32 by 8), 33 and 63 cells, 5 to 33 tile rows in regions of 1, 2 (the default)
# and 3, region counts that eight divides and does not, regions of one tile column; one launch per stage (up to
# 1024 blocks) and two. Tolerances as above.
@pytest.mark.parametrize("nx,ny,nz,fs,prec,coef,env", [
    (65, 18, 12, True, 4, 0, {}),
    (96, 22, 13, False, 4, 0, {}),
    (97, 33, 12, True, 8, 0, {"CGFDM_INTERIOR_RTY": "3"}),
    (127, 64, 11, False, 8, 0, {"CGFDM_INTERIOR_RTY": "1"}),
    (31, 130, 14, True, 4, 1, {}),
    (130, 100, 26, True, 4, 0, {}),
    (150, 66, 24, True, 4, 2, {"CGFDM_INTERIOR_RTY": "3"}),
    (140, 40, 30, True, 4, 0, {"CGFDM_INTERIOR_RTX": "1"}),
])
def test_block_order_reaches_every_cell(nx, ny, nz, fs, prec, coef, env, oracle_mod, monkeypatch):
    from cgfdm_amd import model as M
    from cgfdm_amd import solver
    H = M.HALO
    for k, v in env.items():
        monkeypatch.setenv(k, v)
    m = M.small_config(nx=nx, ny=ny, nz=nz, npml=4, hills=2, layered=True, free_surface=fs, nt=8)
    print(f"{nx}x{ny}x{nz} fs {fs} precision {prec} coef {coef} {env}, 3 steps", flush=True)
    g = solver.Solver(m, precision=prec, coef_storage=coef)
    o = oracle_mod.Oracle(m, prec=prec if coef == 0 else 8, threads=8)
    rng = np.random.default_rng(nx)
    for v in range(9):
        w = np.zeros(g.shape)
        w[H:-H, H:-H, H:-H] = rng.standard_normal((nz, ny, nx)) * (1.0 if v < 3 else 1e7)
        g.set_field(v, w)
        o.set_field(v, w)
    g.step(3)
    o.step(3)
    tol = 1e-10 if prec == 8 else 3e-5 if coef == 0 else 5e-3 if coef == 1 else 4e-2
    for v in range(9):
        a, b = g.field(v), o.field(v)
        assert rel_l2(a, b) < tol, (v, rel_l2(a, b))
        # the last 32 columns by themselves
        assert rel_l2(a[..., -H - 32:], b[..., -H - 32:]) < tol, v
