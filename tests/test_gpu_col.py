"""The middle passes as one kernel per kx column (bm_col): every line length and z length it serves,
at the fewest and most planes or layers of each, open and periodic y, against the FP64 oracle (the
field's parity bar, 1e-6 relative L2), and against the separate passes, whose arithmetic it repeats
(FP32 rounding: 5e-7; a field evaluation's own error is below 2e-7)."""
import ctypes as C

import numpy as np
import pytest
import torch

from boris2_amd import _lib, api
import oracle_lib as O

pytestmark = pytest.mark.gpu
H = (4e-9, 4e-9, 4e-9)


def rel(a, b):
    return np.linalg.norm(a - b) / np.linalg.norm(b)


def nz_open(nz):
    N = 1
    while nz > 1 and N < 2 * nz:
        N *= 2
    return N


# N.y = 4 ... 1024 (2D); N.z = 4 (nz 2), 8 (3, 4), 16 (5, 8), 32 (9, 16); column counts around the
# lanes of a wave and beyond the compute units
OPEN = [(6, 2, 1), (4, 3, 1), (8, 4, 1), (12, 6, 1), (16, 8, 1), (2, 12, 1), (24, 16, 1), (32, 24, 1), (64, 32, 1), (48, 48, 1), (8, 64, 1),
        (16, 96, 1), (12, 128, 1), (6, 192, 1), (4, 256, 1), (6, 384, 1), (4, 512, 1), (8, 100, 1),
        (8, 8, 2), (16, 2, 3), (12, 24, 4), (6, 96, 4), (4, 256, 4), (8, 48, 5), (6, 64, 8), (4, 250, 8), (2, 384, 5), (8, 16, 9), (12, 64, 16),
        (6, 128, 16), (2, 48, 12), (260, 12, 8)]


@pytest.mark.parametrize("n", OPEN)
def test_open(gpu, monkeypatch, n):
    M0 = api.random_magnetisation(n[0] * n[1] * n[2], 8e5, 2).astype(np.float32)
    M = torch.from_numpy(M0).cuda()
    d = api.Demag(n, H)
    got = d.convolute(M).cpu().numpy().astype(np.float64)
    ref = O.OracleDemag(n, H, Nz_override=nz_open(n[2]))(M0.astype(np.float64))
    assert rel(got, ref) <= 1e-6
    monkeypatch.setenv("BM_YZY", "0")
    s = api.Demag(n, H)
    assert rel(got, s.convolute(M).cpu().numpy().astype(np.float64)) <= 5e-7
    d.close(); s.close()


@pytest.mark.parametrize("n,pbc", [((8, 12, 1), (0, 3, 0)), ((16, 64, 4), (2, 2, 0)), ((8, 96, 8), (0, 2, 0)), ((4, 256, 2), (0, 2, 0)), ((6, 32, 16), (0, 2, 0))])
def test_periodic_y(gpu, n, pbc):
    M0 = api.random_magnetisation(n[0] * n[1] * n[2], 8e5, 4).astype(np.float32)
    d = api.Demag(n, H, pbc)
    ref = O.OracleDemag(n, H, Nz_override=nz_open(n[2]), pbc=pbc)(M0.astype(np.float64))
    assert rel(d.convolute(torch.from_numpy(M0).cuda()).cpu().numpy().astype(np.float64), ref) <= 1e-6
    d.close()


# layers of one thickness and of two; as many as 512 threads hold, then 1024
@pytest.mark.parametrize("nx,ny,L,pbc", [(8, 8, 1, (0, 0)), (16, 24, 2, (0, 0)), (12, 64, 3, (0, 0)), (6, 256, 4, (0, 0)), (8, 64, 16, (0, 0)), (4, 128, 9, (0, 0)),
                                         (4, 128, 16, (0, 0)), (4, 512, 2, (0, 0)), (4, 512, 3, (0, 0)), (6, 384, 3, (0, 0)), (8, 32, 5, (0, 2)), (16, 64, 12, (2, 2))])
def test_layers(gpu, nx, ny, L, pbc):
    hz = [4e-9 if l % 3 else 8e-9 for l in range(L)]
    z0 = [12e-9 * l for l in range(L)]
    M0 = api.random_magnetisation(nx * ny * L, 8e5, 6).astype(np.float32)
    d = api.MultiLayerDemag(nx, ny, 4e-9, 4e-9, hz, z0, pbc)
    ref = O.OracleMLayer(nx, ny, 4e-9, 4e-9, np.array(hz), np.array(z0), pbc)(M0.astype(np.float64))
    assert rel(d.convolute(torch.from_numpy(M0).cuda()).cpu().numpy().astype(np.float64), np.asarray(ref).reshape(-1, 3)) <= 1e-6
    d.close()


# of these only (512, 128, 12) packs the two columns (N.z 16 or 32, 2^a N.y); test_packed_columns has the form
@pytest.mark.parametrize("n", [(256, 64, 1), (256, 33, 8), (256, 24, 3), (512, 32, 2), (512, 128, 12), (256, 96, 6), (512, 100, 1)])
def test_first_and_last_column_as_one(gpu, n):
    """N.x / 2 a multiple of the compute units: columns 0 and N.x / 2 share a workgroup."""
    M0 = api.random_magnetisation(n[0] * n[1] * n[2], 8e5, 2).astype(np.float32)
    d = api.Demag(n, H)
    ref = O.OracleDemag(n, H, Nz_override=nz_open(n[2]))(M0.astype(np.float64))
    assert rel(d.convolute(torch.from_numpy(M0).cuda()).cpu().numpy().astype(np.float64), ref) <= 1e-6
    d.close()


# layers never pack: one column more than the compute units
@pytest.mark.parametrize("nx,ny,L", [(256, 32, 3), (256, 64, 6), (512, 24, 4)])
def test_layers_first_and_last_column_as_one(gpu, nx, ny, L):
    z0 = [8e-9 * l for l in range(L)]
    M0 = api.random_magnetisation(nx * ny * L, 8e5, 6).astype(np.float32)
    d = api.MultiLayerDemag(nx, ny, 4e-9, 4e-9, [4e-9] * L, z0)
    ref = O.OracleMLayer(nx, ny, 4e-9, 4e-9, np.full(L, 4e-9), np.array(z0))(M0.astype(np.float64))
    assert rel(d.convolute(torch.from_numpy(M0).cuda()).cpu().numpy().astype(np.float64), np.asarray(ref).reshape(-1, 3)) <= 1e-6
    d.close()


@pytest.mark.parametrize("n", [(64, 64, 1), (64, 32, 4), (32, 32, -3)])
def test_column_pass_is_timed_as_itself(gpu, n):
    """Launch timing counts the column kernel (kind 11) and no y, z, 2D or product pass; n[2] < 0: layers."""
    L = _lib.load()
    if n[2] < 0:
        d = api.MultiLayerDemag(n[0], n[1], 4e-9, 4e-9, [4e-9] * 3, [8e-9 * l for l in range(3)])
    else:
        d = api.Demag(n, H)
    M = torch.ones((n[0] * n[1] * abs(n[2]), 3), device="cuda")
    _lib.check(L.bm_prof_begin(16))
    d.convolute(M)
    torch.cuda.synchronize()
    _lib.check(L.bm_prof_end())
    count = {}
    for k, name in enumerate(_lib.PROF_KINDS):
        c = C.c_longlong()
        _lib.check(L.bm_prof_query(k, C.byref(c), None, None, None))
        if c.value:
            count[name] = c.value
    assert count == {"fwd_x_r2c": 1, "column_pass": 1, "inv_x_c2r": 1}
    d.close()


@pytest.mark.parametrize("n,pbc,col", [((384, 512, 1), (0, 0, 0), 1), ((400, 400, 1), (0, 0, 0), 0), ((768, 385, 1), (0, 0, 0), 0), ((1024, 400, 1), (0, 0, 0), 1),
                                       ((1024, 1024, 1), (2, 2, 0), 0)])
def test_2d_lines_of_1024(gpu, n, pbc, col):
    """Between two and four columns per compute unit these take the 2D y pass, else the column kernel;
    either way the field is the oracle's."""
    L = _lib.load()
    ncu = torch.cuda.get_device_properties(0).multi_processor_count
    if ncu != 256:
        pytest.skip("the column counts are chosen around 256 compute units")
    M0 = api.random_magnetisation(n[0] * n[1], 8e5, 2).astype(np.float32)
    M = torch.from_numpy(M0).cuda()
    d = api.Demag(n, H, pbc)
    _lib.check(L.bm_prof_begin(16))
    got = d.convolute(M).cpu().numpy().astype(np.float64)
    _lib.check(L.bm_prof_end())
    c = C.c_longlong()
    _lib.check(L.bm_prof_query(_lib.PROF_KINDS.index("column_pass"), C.byref(c), None, None, None))
    N = d.info()[0]
    assert N[1] == 1024 and c.value == col
    ref = O.OracleDemag(n, H, pbc=pbc)(M0.astype(np.float64))
    assert rel(got, ref) <= 1e-6
    d.close()


# the packed form (columns 0 and N.x / 2 as one line): N.z 16 and 32, nx a multiple of 256, one column per
# workgroup; the shortest and longest lines, ragged ny, the fewest and most planes; periodic y and x
PACKED = [((256, 8, 6), None), ((256, 16, 5), None), ((256, 30, 8), None), ((256, 60, 7), None), ((512, 128, 5), None), ((256, 250, 8), None),
          ((256, 512, 5), None), ((1024, 32, 6), None), ((256, 8, 9), None), ((256, 30, 16), None), ((512, 60, 12), None), ((256, 128, 16), None),
          ((256, 250, 9), None), ((256, 64, 8), (0, 2, 0)), ((512, 128, 16), (0, 2, 0)), ((512, 64, 6), (2, 2, 0)), ((512, 30, 10), (2, 0, 0))]


@pytest.mark.parametrize("n,pbc", PACKED, ids=str)
def test_packed_columns(gpu, n, pbc):
    if (n[0] // (2 if pbc and pbc[0] else 1)) % torch.cuda.get_device_properties(0).multi_processor_count:
        pytest.skip("N.x / 2 is not a multiple of the compute units")
    M0 = api.random_magnetisation(n[0] * n[1] * n[2], 8e5, 7).astype(np.float32)
    d = api.Demag(n, H, pbc or (0, 0, 0))
    ref = O.OracleDemag(n, H, Nz_override=nz_open(n[2]), pbc=pbc)(M0.astype(np.float64))
    assert rel(d.convolute(torch.from_numpy(M0).cuda()).cpu().numpy().astype(np.float64), ref) <= 1e-6
    d.close()
