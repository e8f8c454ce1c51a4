"""The x passes and the row kernel with one component per wave group (few rows): every row length
that takes them, at rows fewer than, equal to and one more than a workgroup's, against the FP64
oracle.  Bars: the field's parity bar of 1e-6 relative L2, one step's 1e-6 of M (FP32 rounding of a
few operations on values of one size, a step changes M by less than a tenth)."""
import numpy as np
import pytest
import torch

from boris2_amd import api
import oracle_lib as O

pytestmark = pytest.mark.gpu
H = (4e-9, 4e-9, 4e-9)
ALL = api.BM_MOD_DEMAG | api.BM_MOD_EXCHANGE | api.BM_MOD_ANIS_UNI | api.BM_MOD_ZEEMAN


def nz_open(nz):
    N = 1
    while nz > 1 and N < 2 * nz:
        N *= 2
    return N


def rel(a, b):
    return np.linalg.norm(a - b) / np.linalg.norm(b)


@pytest.mark.parametrize("n", [(2, 65, 1), (4, 33, 2), (6, 64, 1), (8, 31, 2), (12, 65, 1), (16, 33, 2), (24, 31, 1), (32, 17, 2),
                               (48, 15, 1), (64, 9, 3), (96, 8, 1), (128, 5, 2), (192, 3, 2), (256, 3, 3), (384, 1, 2), (512, 5, 1),
                               (768, 3, 1), (1024, 2, 2), (33, 10, 2), (100, 7, 1)])
def test_field_set_added_planar_and_energy(gpu, n):
    nc = n[0] * n[1] * n[2]
    M0 = api.random_magnetisation(nc, 8e5, 11).astype(np.float32)
    M = torch.from_numpy(M0).cuda()
    d = api.Demag(n, H)
    ref = O.OracleDemag(n, H, Nz_override=nz_open(n[2]))(M0.astype(np.float64))
    e = torch.zeros(1, device="cuda")
    Hs = d.convolute(M, energy=e)
    base = torch.full_like(M, 1e4)
    Ha = d.convolute(M, base.clone(), clear_out=False)
    assert rel(Hs.cpu().numpy().astype(np.float64), ref) <= 1e-6
    assert rel(Ha.cpu().numpy().astype(np.float64) - 1e4, ref) <= 1e-6
    assert rel(d.convolute_planar(M).cpu().numpy().T.astype(np.float64), ref) <= 1e-6
    want = -api.MU0 / 2 * (M0.astype(np.float64) * ref).sum() / nc
    assert abs(e.item() - want) <= 1e-6 * api.MU0 / 2 * 8e5 * np.linalg.norm(ref) / np.sqrt(nc)
    d.close()


@pytest.mark.parametrize("n", [(64, 9, 1), (128, 5, 2), (192, 3, 1), (256, 3, 2), (384, 2, 2), (512, 5, 1), (768, 3, 1), (1024, 3, 1), (8, 65, 2)])
@pytest.mark.parametrize("method", [api.BM_EVAL_RK4, api.BM_EVAL_RKDP54, api.BM_EVAL_TEULER, api.BM_EVAL_AHEUN])
def test_steps(gpu, n, method):
    nc = n[0] * n[1] * n[2]
    p = api.FMParams(Ms=1e6, A=1.5e-11, alpha=0.1, K1=5e5, ea=(0.0, 0.0, 1.0), Ha=(0.0, 0.0, 4e4), modules=ALL)
    M0 = api.random_magnetisation(nc, p.Ms, 5).astype(np.float32)
    s = api.FMSolver(method, n, H, p, M0)
    dt = 2e-15 if method == api.BM_EVAL_AHEUN else 1e-14       # no rejected step; the largest step, so no other one
    s.set_dt(dt)
    s.set_astep(dT_max=dt)
    s.run_to_iteration(2)
    o = O.OracleSim(method, n, H, p)
    o.set_M(M0.astype(np.float64))
    o.set_dt(dt)
    o.set_astep(dtmax=dt)
    o.run_to_iteration(2)
    assert rel(s.M.cpu().numpy().astype(np.float64), o.get_M()) <= 1e-6
    s.close()


@pytest.mark.parametrize("n,pbc", [((64, 9, 2), (3, 0, 0)), ((256, 6, 1), (2, 2, 0)), ((512, 4, 2), (2, 0, 0)), ((48, 16, 1), (2, 1, 0))])
def test_periodic_rows(gpu, n, pbc):
    nc = n[0] * n[1] * n[2]
    M0 = api.random_magnetisation(nc, 8e5, 3).astype(np.float32)
    d = api.Demag(n, H, pbc)
    ref = O.OracleDemag(n, H, pbc=pbc)(M0.astype(np.float64))
    assert rel(d.convolute(torch.from_numpy(M0).cuda()).cpu().numpy().astype(np.float64), ref) <= 1e-6
    d.close()


@pytest.mark.parametrize("nx,ny,groups", [(64, 8, None), (128, 6, [0, 0, 1, 2, 2]), (192, 3, [0, 1, 1]), (512, 3, [0, 0])])
@pytest.mark.parametrize("method", [api.BM_EVAL_RK4, api.BM_EVAL_RKDP54])
def test_layer_stack_rows_match_the_separate_passes(gpu, monkeypatch, nx, ny, groups, method):
    """Per-layer values, meshes of several planes, per-layer fields: the row kernel against the
    separate x passes and stage kernel, the same arithmetic (FP32 rounding, 5 steps)."""
    L = 3 if groups is None else len(groups)
    rng = np.random.default_rng(nx)
    p = api.FMParams(Ms=8e5, A=1.3e-11, alpha=0.1, K1=1e5, ea=(0.0, 0.0, 1.0), Ha=(1e4, 0.0, 2e4), modules=ALL)
    M0 = (api.random_magnetisation(L * nx * ny, 1.0, 3) * 8e5).astype(np.float32)
    out = []
    for row in ("1", "0"):
        monkeypatch.setenv("BM_ROW_KERNEL", row)
        rng = np.random.default_rng(nx)
        lay = dict(A=rng.uniform(1e-11, 2e-11, L), alpha=rng.uniform(0.02, 0.2, L), K1=rng.uniform(0, 2e5, L))
        s = api.LayerStackSolver(method, nx, ny, 4e-9, 4e-9, [4e-9] * L, [4e-9 * l for l in range(L)], p, M0=M0, **lay)
        s.set_layer_meshes(groups, rng.uniform(-2e4, 2e4, (L, 3)) if groups else None)
        s.set_ms_map(np.repeat(rng.uniform(7e5, 9e5, L), nx * ny))
        s.set_dt(2e-14)
        s.set_astep(dT_max=2e-14)
        s.run_to_iteration(5)
        out.append(s.M.cpu().numpy().astype(np.float64))
        s.close()
    assert rel(out[0], out[1]) <= 5e-7


def test_stack_field_function_may_use_the_stacks_handle(gpu):
    """A field function that convolves with the stack's own multilayer handle (for an energy, say)
    must not disturb the run: the same bits as with one that leaves the handle alone."""
    L, nx, ny = 3, 64, 8
    p = api.FMParams(Ms=8e5, A=1.3e-11, alpha=0.1, modules=api.BM_MOD_DEMAG | api.BM_MOD_EXCHANGE)
    M0 = api.random_magnetisation(L * nx * ny, 8e5, 4).astype(np.float32)
    other = torch.from_numpy(M0[::-1].copy()).cuda()
    out = []
    for use in (False, True):
        s = api.LayerStackSolver(api.BM_EVAL_RK4, nx, ny, 4e-9, 4e-9, [4e-9] * L, [4e-9 * l for l in range(L)], p, M0=M0)

        def field(M):
            if use:
                s.mlayer.convolute(other)
            return torch.full_like(M, 1e4)
        s.set_extra_field(field)
        s.set_dt(2e-14)
        s.run_to_iteration(3)
        out.append(s.M.clone())
        s.close()
    assert torch.equal(out[0], out[1])


# 256 cells per row: workgroups (two rows each) up to three per compute unit, from there to four (no
# fourth wave), and more
@pytest.mark.parametrize("ny,nz", [(127, 12), (220, 7), (128, 16), (129, 16)])
@pytest.mark.parametrize("method", [api.BM_EVAL_RK4, api.BM_EVAL_RKDP54])
def test_steps_around_the_fourth_wave(gpu, ny, nz, method):
    test_steps(gpu, (256, ny, nz), method)


def test_layer_stack_without_the_fourth_wave(gpu, monkeypatch):
    test_layer_stack_rows_match_the_separate_passes(gpu, monkeypatch, 256, 192, [0, 0, 1, 1, 2, 3, 4, 4, 5], api.BM_EVAL_RK4)
