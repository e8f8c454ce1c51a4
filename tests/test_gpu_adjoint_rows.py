"""The adjoint's row kernels (one kernel between two convolutions' middle passes) at the edges of
their row groups: the shortest rows, rows of part of a wave and of a whole one, the fourth wave of
the per-cell work, radix-3 rows, and row counts that leave the last group ragged."""
import numpy as np
import pytest
import torch

import oracle_lib as O
from boris2_amd import api
from test_gpu_adjoint import oracle_grads, problem

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [(8, 6, 2), (32, 24, 1), (96, 6, 2), (128, 12, 1), (128, 6, 2), (256, 6, 2), (512, 6, 1)])
def test_adjoint_rows_match_oracle(gpu, n):
    n, p, Ms, m0, mt = problem(n, seed=sum(n))
    dt, steps = 250e-15, 8
    L0, g0, ga0 = oracle_grads(n, p, Ms, m0, mt, dt, steps)
    r = api.RK4Adjoint(n, (4e-9,) * 3, p, torch.tensor(Ms, dtype=torch.float32), dt, steps, 3)
    L, _ = r.forward(torch.tensor(m0, dtype=torch.float32), torch.tensor(mt, dtype=torch.float32))
    g, ga = r.backward()
    g = g.cpu().numpy().astype(np.float64)
    eg, ea = np.linalg.norm(g - g0) / np.linalg.norm(g0), abs(ga - ga0) / abs(ga0)
    print(f"{n}: loss {abs(L - L0):.2e}, dL/dMs rel L2 {eg:.2e}, dL/damp rel {ea:.2e}")
    # the bounds of the 40-step comparison of the same problem (FP32 forward's departure, linear in the steps)
    assert abs(L - L0) <= 1e-6
    assert eg <= 5e-5
    assert ea <= 5e-5
    r.close()


@pytest.mark.parametrize("n,pbc", [((32, 16, 1), (0, 2, 0)), ((64, 12, 4), (0, 2, 2)), ((16, 6, 4), (0, 0, 1))], ids=str)
def test_adjoint_rows_with_periodic_y_and_z(gpu, n, pbc):
    """Open x keeps the row kernels, whose exchange then wraps around along the other axes."""
    n, p, Ms, m0, mt = problem(n, seed=sum(n))
    dt, steps = 250e-15, 8
    a = O.OracleAdjoint(n, (4e-9,) * 3, p, Ms, dt, steps, pbc=pbc)
    L0, _ = a.forward(m0, mt)
    g0, ga0 = a.backward(m0, mt)
    r = api.RK4Adjoint(n, (4e-9,) * 3, p, torch.tensor(Ms, dtype=torch.float32), dt, steps, 3, pbc=pbc)
    L, _ = r.forward(torch.tensor(m0, dtype=torch.float32), torch.tensor(mt, dtype=torch.float32))
    g, ga = r.backward()
    g = g.cpu().numpy().astype(np.float64)
    eg, ea = np.linalg.norm(g - g0) / np.linalg.norm(g0), abs(ga - ga0) / abs(ga0)
    print(f"{n} {pbc}: loss {abs(L - L0):.2e}, dL/dMs rel L2 {eg:.2e}, dL/damp rel {ea:.2e}")
    assert abs(L - L0) <= 1e-6
    assert eg <= 5e-5
    assert ea <= 5e-5
    r.close()


def test_adjoint_holds_no_array_beyond_its_own(gpu):
    """Device memory of an instance of 1 M cells: checkpoints (3), the tape of one step (9), the two
    working states, acc, the field, three stage inputs and the eight arrays of the backward pass, 12
    bytes a cell each, and 8 bytes a cell of dL/dMs, within a third of one array."""
    n, cells = (1024, 1024, 1), 1 << 20
    Ms = torch.full((cells,), 8e5, device="cuda")
    p = api.FMParams(Ms=8e5, A=1.3e-11, alpha=0.1, modules=api.BM_MOD_EXCHANGE)
    one = api.RK4Adjoint((8, 8, 1), (4e-9,) * 3, p, Ms[:64], 1e-14, 2, 1)     # the library's code is on the device
    m = torch.ones(64, 3, device="cuda")
    one.forward(m, m)
    torch.cuda.synchronize()
    free = torch.cuda.mem_get_info()[0]
    r = api.RK4Adjoint(n, (4e-9,) * 3, p, Ms, 1e-14, 2, 1)
    used = free - torch.cuda.mem_get_info()[0]
    r.close(); one.close()
    print(f"{used / cells:.2f} bytes a cell")
    assert used <= (12 * (3 + 9 + 2 + 1 + 1 + 3 + 8) + 8 + 4) * cells
