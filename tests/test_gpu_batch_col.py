"""The column kernel in a batch: launch shapes of the middle passes, pinned or tuned, change no bit
(256 and 512 cells per row among them, N.x / 2 a multiple of the compute units), a mesh does not
depend on its neighbours, radix tuning chooses the form per column group, and a report gives
every pass's own time and carries the choices to another batch."""
import numpy as np
import pytest
import torch

from boris2_amd import api

pytestmark = pytest.mark.gpu
H = (4e-9, 4e-9, 4e-9)
# 2D, N.z 4 to 32, radix-3 lines, one column more than the compute units; the last two have lines too
# long for a workgroup (N.z 64) and a z length without a column form
SIZES = [(64, 96, 1), (256, 64, 1), (64, 48, 2), (128, 32, 4), (256, 32, 8), (256, 64, 5), (512, 16, 12), (48, 32, 16), (32, 32, 24), (16, 16, 48)]
STACKS = [(64, 48, 3), (96, 32, 7), (32, 64, 12)]


def batch(autotune=False, sizes=SIZES, stacks=STACKS, use_graph=True):
    rng = np.random.default_rng(31)
    meshes, M0, layers = [], [], []
    for q, n in enumerate(list(sizes) + list(stacks)):
        p = api.FMParams(Ms=float(rng.uniform(5e5, 1.1e6)), A=1.3e-11, alpha=0.1, modules=api.BM_MOD_DEMAG | api.BM_MOD_EXCHANGE)
        meshes.append((n, H, p))
        M0.append(api.random_magnetisation(n[0] * n[1] * n[2], p.Ms, 80 + q).astype(np.float32))
        hz = [4e-9 if l % 2 else 8e-9 for l in range(n[2])]
        layers.append(dict(hz=hz, z0=[12e-9 * l for l in range(n[2])]) if q >= len(sizes) else None)
    return api.BatchSolver(api.BM_EVAL_RK4, meshes, M0, layers=layers, autotune=autotune, use_graph=use_graph)


def run(b, steps=3):
    b.set_dt(40e-15)
    b.run(steps)
    torch.cuda.synchronize()
    return b.M.clone()


def nz_open(nz):
    N = 1
    while nz > 1 and N < 2 * nz:
        N *= 2
    return N


def separate_passes(b, sizes=SIZES, stacks=STACKS):
    """Pin a launch shape of every y, z, 2D and product pass of the batch."""
    for n in sizes:
        for p, s in ([("y2d", 2 * n[1])] if n[2] == 1 else [("y_fwd", 2 * n[1]), ("y_inv", 2 * n[1]), ("z", nz_open(n[2]))]):
            b.set_schedule(p, s, per_cu=2 if p == "z" else 4)
    for n in stacks:
        b.set_schedule("y_fwd", 2 * n[1], per_cu=4); b.set_schedule("y_inv", 2 * n[1], per_cu=4); b.set_schedule("ml_mult", n[2], per_cu=4)


@pytest.mark.parametrize("sizes,stacks", [([n], []) for n in SIZES] + [([], [n]) for n in STACKS], ids=str)
def test_pinned_launch_shape_changes_no_bit(gpu, sizes, stacks):
    a, b = batch(sizes=sizes, stacks=stacks), batch(sizes=sizes, stacks=stacks)
    separate_passes(b, sizes, stacks)
    assert torch.equal(run(a), run(b))
    a.close(); b.close()


@pytest.mark.parametrize("sizes,stacks", [([n], []) for n in SIZES[1:8]] + [([], [(16, 32, L)]) for L in range(2, 17)], ids=str)
def test_column_and_separate_passes(gpu, sizes, stacks):
    """The two forms of a column group agree to FP32 rounding (5e-7 of a field, over 3 steps that
    change M by a tenth), and the default is the column kernel."""
    n = (sizes + stacks)[0]
    name = "col_ml" if stacks else "col_2d" if n[2] == 1 else f"col_z{nz_open(n[2])}"
    out = []
    for f in (0, 1, 2):
        b = batch(sizes=sizes, stacks=stacks)
        b.set_schedule(name, 2 * n[1], f=f)
        out.append(run(b))
        b.close()
    assert torch.equal(out[0], out[1])
    assert (out[0] - out[2]).double().norm() <= 5e-7 * out[0].double().norm()


def test_a_mesh_does_not_depend_on_its_neighbours(gpu):
    """Lines of several columns per workgroup alone, of one beside a mesh with more planes."""
    a, b = batch(sizes=[(256, 8, 5)], stacks=[]), batch(sizes=[(256, 8, 5), (256, 8, 8), (512, 8, 6)], stacks=[])
    run(a), run(b)
    assert torch.equal(a.mesh(0), b.mesh(0))
    a.close(); b.close()


def test_plain_tuning_changes_no_bit_and_its_report_applies(gpu):
    a, t = batch(), batch(autotune=True)
    want, got = run(a), run(t)
    assert torch.equal(want, got)
    rep = t.autotune_report()
    lines = {(l.split()[0], int(l.split()[1])): l.split() for l in rep}
    cols = {k: v for k, v in lines.items() if k[0].startswith("col_")}
    assert set(cols) == {("col_2d", 192), ("col_2d", 128), ("col_z4", 96), ("col_z8", 64), ("col_z16", 64), ("col_z16", 128),
                         ("col_z32", 32), ("col_z32", 64), ("col_ml", 96), ("col_ml", 64), ("col_ml", 128)}, rep
    assert all(v[2] == "f=0" for v in cols.values()), rep
    # the meshes without a column form have tuned passes, and every line has a time of its own
    for k in (("z", 64), ("z", 128), ("y_fwd", 32), ("y_inv", 64)):
        assert lines[k][3] != "per_cu=0", rep
    us = [float(l.split()[-2]) for l in rep]
    assert min(us) > 0 and len(set(us)) > len(us) // 2, rep
    b = batch()
    b.apply_report(rep)
    assert [l.rsplit(" ", 2)[0] for l in b.autotune_report()] == [l.rsplit(" ", 2)[0] for l in rep]
    assert torch.equal(want, run(b))
    for s in (a, t, b):
        s.close()


@pytest.mark.parametrize("use_graph", [True, False])
def test_radix_tuning_chooses_per_group(gpu, use_graph):
    """Radix tuning may take either form of any group; its report, applied to another batch, runs the
    same forms."""
    a, t = batch(), batch(autotune="radix", use_graph=use_graph)
    want, got = run(a), run(t)
    assert (want - got).double().norm() <= 1e-6 * want.double().norm()
    rep = t.autotune_report()
    assert all(l.split()[2] in ("f=1", "f=2") for l in rep if l.startswith("col_")), rep
    b = batch()
    b.apply_report(rep)
    assert torch.equal(got, run(b))
    for s in (a, t, b):
        s.close()


def test_a_radix_schedule_takes_the_separate_pass(gpu):
    a, b, c = (batch(sizes=[(64, 64, 1)], stacks=[]) for _ in range(3))
    b.set_schedule("y2d", 128, radix=1)
    c.set_schedule("col_2d", 128, f=1)
    c.set_schedule("y2d", 128, radix=1)
    want, got = run(a), run(b)
    assert not torch.equal(want, got) and torch.equal(got, run(c))
    for s in (a, b, c):
        s.close()


def test_column_schedules_refused(gpu):
    b = batch(sizes=[(64, 64, 1)], stacks=[])
    for name, size, kw in (("col_2d", 128, dict(f=3)), ("col_2d", 128, dict(f=-1)), ("col_2d", 128, dict(f=1, per_cu=4)),
                           ("col_2d", 128, dict(f=1, radix=1)), ("col_2d", 64, dict(f=1)), ("col_z4", 128, dict(f=1)), ("col", 128, dict(f=1))):
        with pytest.raises(RuntimeError, match="error 1"):
            b.set_schedule(name, size, **kw)
    b.close()


def test_one_group_of_unlike_meshes_follows_the_single_runs(gpu):
    """One (N.y, N.z) group of 257, 129 and 513 columns and 8, 6 and 5 planes against each mesh alone
    (2e-6 relative L2, the bar of batched against single runs)."""
    sizes = [(256, 32, 8), (128, 32, 6), (512, 30, 5)]
    b = batch(sizes=sizes, stacks=[])
    M0 = b.M.clone()
    run(b)
    for q, (n, h, p) in enumerate(b.meshes):
        s = api.FMSolver(api.BM_EVAL_RK4, n, h, p, M0[int(b.offsets[q]):int(b.offsets[q + 1])].cpu().numpy())
        s.set_dt(40e-15)
        s.run_to_iteration(3)
        assert (s.M - b.mesh(q)).double().norm() <= 2e-6 * s.M.double().norm()
        s.close()
    b.close()
