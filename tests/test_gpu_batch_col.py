"""The column kernel in a batch: a mesh does not depend on its neighbours."""
import numpy as np
import pytest
import torch

from boris2_amd import api

pytestmark = pytest.mark.gpu
H = (4e-9, 4e-9, 4e-9)


def batch(sizes, stacks, autotune=False, pbc=None):
    rng = np.random.default_rng(31)
    meshes, M0, layers = [], [], []
    for q, n in enumerate(list(sizes) + list(stacks)):
        p = api.FMParams(Ms=float(rng.uniform(5e5, 1.1e6)), A=1.3e-11, alpha=0.1, modules=api.BM_MOD_DEMAG | api.BM_MOD_EXCHANGE)
        meshes.append((n, H, p))
        M0.append(api.random_magnetisation(n[0] * n[1] * n[2], p.Ms, 80 + q).astype(np.float32))
        hz = [4e-9 if l % 2 else 8e-9 for l in range(n[2])]
        layers.append(dict(hz=hz, z0=[12e-9 * l for l in range(n[2])]) if q >= len(sizes) else None)
    return api.BatchSolver(api.BM_EVAL_RK4, meshes, M0, layers=layers, autotune=autotune, pbc=pbc)


def run(b, steps=3):
    b.set_dt(40e-15)
    b.run(steps)
    torch.cuda.synchronize()
    return b.M.clone()


def test_a_mesh_does_not_depend_on_its_neighbours(gpu):
    """Lines of several columns per workgroup alone, of one beside a mesh with more planes."""
    a, b = batch(sizes=[(256, 8, 5)], stacks=[]), batch(sizes=[(256, 8, 5), (256, 8, 8), (512, 8, 6)], stacks=[])
    run(a), run(b)
    assert torch.equal(a.mesh(0), b.mesh(0))
    a.close(); b.close()
