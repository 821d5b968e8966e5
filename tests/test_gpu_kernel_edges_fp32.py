"""The precision form at the grids of test_gpu_kernel_edges.py: kernel variants
against each other bit for bit (the same operations in the same order), and the
oracle at the form's bar (relative L2 velocity error <= 1e-5)."""
import numpy as np
import pytest

from elmm_amd import capi, cases
from helpers import velocity_rel_l2
from oracle_py import Oracle
from test_gpu_kernel_edges import _periodic_images

pytestmark = pytest.mark.gpu

BAR = 1e-5


def _solver(cfg, refine=0, steps=2, cuboids=(), sources=(), seed=7, oracle=False):
    case = capi.Case(cfg, cuboids=cuboids, sources=sources)
    f = cases.initial_fields(cfg, u0=1.5, amp=0.2, seed=seed)
    c32 = capi.with_precision(cfg, capi.FP32_REFINED, refine)
    out = [capi.Solver(c32, case)] + ([Oracle(cfg, case)] if oracle else [])
    for x, c in zip(out, (c32, cfg)):
        cases.upload_initial(x, c, f)
        x.init()
        x.step(steps)
    return out if oracle else out[0]


def _same_fields(a, b, cfg):
    for field in [0, 1, 2, capi.F_PR, capi.F_VISC] + [capi.F_SCALAR + s for s in range(cfg.nscalars)]:
        np.testing.assert_array_equal(a.download(field), b.download(field))


def _within_bar(s, o, cfg):
    err = velocity_rel_l2(s, o, cfg)
    print(f"{cfg.nx}x{cfg.ny}x{cfg.nz}: rel L2 velocity {err:.2e}", flush=True)
    assert err <= BAR


@pytest.mark.parametrize("refine", [0, 1])
@pytest.mark.parametrize("nx,ny,nz", [(6, 9, 5), (12, 27, 4), (18, 24, 7), (81, 54, 5), (162, 36, 4), (486, 6, 4),
                                      (8, 243, 5), (768, 12, 4), (972, 4, 4), (4, 972, 4), (64, 576, 4)])
def test_mixed_radix_groups(require_gpu, nx, ny, nz, refine):
    cfg = cases.uniform_config(nx, ny, nz, dx=1.0, dt=0.02)
    s, o = _solver(cfg, refine, steps=1, oracle=True)
    _within_bar(s, o, cfg)


# the pivot table against the kernel that divides (refine 1: 32-bit spectra)
@pytest.mark.parametrize("refine", [0, 1])
@pytest.mark.parametrize("nx,ny,nz", [(8, 6, 4), (6, 9, 5), (16, 4, 7), (8, 12, 8), (16, 9, 9), (4, 4, 33),
                                      (8, 6, 350)])
def test_z_solve_lengths(require_gpu, monkeypatch, nx, ny, nz, refine):
    cfg = cases.uniform_config(nx, ny, nz, dx=1.0, dt=0.02)
    table = _solver(cfg, refine)
    monkeypatch.setenv("ELMM_ZPIPE", "0")
    _same_fields(table, _solver(cfg, refine), cfg)


# the default tile and walks against other tiles and chunks
@pytest.mark.parametrize("nx,ny,nz", [(64, 8, 5), (66, 10, 17), (128, 12, 31), (36, 64, 65)])
def test_walk_remainders(require_gpu, monkeypatch, nx, ny, nz):
    kw = {} if nx % 11 else dict(poisson_solver=capi.POISSON_MG)
    cfg = cases.uniform_config(nx, ny, nz, dx=1.0, dt=0.02, nscalars=2, **kw)
    src = [(2.5, 2.5, 0.5, 1.0, 0), (nx - 1.5, 3.5, 1.5, 2.0, 1)]
    s, o = _solver(cfg, sources=src, oracle=True)
    _within_bar(s, o, cfg)
    for k, v in (("ELMM_MOM_TILE", "32x8"), ("ELMM_ZCHUNK", "7"), ("ELMM_SGS_ZCHUNK", "5")):
        monkeypatch.setenv(k, v)
    _same_fields(s, _solver(cfg, sources=src), cfg)


@pytest.mark.parametrize("nx,ny,nz", [(4, 8, 6), (8, 4, 6), (24, 18, 8), (64, 32, 12)])
def test_ghosts_are_images(require_gpu, monkeypatch, nx, ny, nz):
    cfg = cases.uniform_config(nx, ny, nz, dx=1.0, dt=0.02, nscalars=1)
    cub = [(-1.2, 1.2, -1.2, 1.2, 0.0, 2.2), (nx - 1.4, nx + 1.4, ny / 2 - 1.1, ny / 2 + 1.1, 0.0, 3.1)]
    s, o = _solver(cfg, cuboids=cub, oracle=True)
    _within_bar(s, o, cfg)
    for c in range(3):
        a = s.download(c)
        np.testing.assert_array_equal(a[:, :, 3:3 + nz], _periodic_images(a, nx, ny)[:, :, 3:3 + nz])
    monkeypatch.setenv("ELMM_GHOST_DELTA", "0")
    _same_fields(s, _solver(cfg, cuboids=cub), cfg)


@pytest.mark.parametrize("lb", [-2, 1])
@pytest.mark.parametrize("nx,ny,nz,mg,refine", [(16, 8, 6, False, 0), (16, 8, 6, False, 1), (12, 18, 7, False, 0),
                                                (12, 18, 7, False, 1), (20, 12, 6, True, 0)])
def test_w_uploaded_between_steps(require_gpu, nx, ny, nz, mg, refine, lb):
    kw = dict(poisson_solver=capi.POISSON_MG) if mg else {}
    cfg = cases.uniform_config(nx, ny, nz, dx=1.0, dt=0.02, **kw)
    s, o = _solver(cfg, refine, oracle=True)
    n = np.array(capi.ghosted_shape(cfg)) - (0 if lb == -2 else 6)
    w = np.random.default_rng(11).uniform(-0.3, 0.3, n).astype(np.float32).astype(np.float64)
    for x in (s, o):
        x.upload(capi.F_W, w, lb=lb)
        x.step(2)
    _within_bar(s, o, cfg)
