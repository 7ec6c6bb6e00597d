"""The filter, interpolation and diagnostics kernels over their ranges of sizes: both
polynomial orders, every number of points, element lists in any order, fewer elements than
one turn of a workgroup and more than one turn of all of them."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
EPS = 2.3e-16


def _state(E, N, seed):
    rng = np.random.default_rng(seed)
    Q = rng.uniform(-1.0, 1.0, (E, 5, (N + 1) ** 3))
    Q[:, 0] = rng.uniform(0.5, 1.5, Q[:, 0].shape)
    return Q


@pytest.mark.parametrize("N", [3, 4])
@pytest.mark.parametrize("p", range(1, 9))
@pytest.mark.parametrize("order", ["stacked", "shuffled", "part"])
def test_interpolation(N, p, order):
    import torch
    from cmdg import abi, closure
    nx, ny, nz, q = 3, 2, 5, N + 1
    iy, ix, iz = np.meshgrid(np.arange(ny), np.arange(nx), np.arange(nz), indexing="ij")
    eijk = np.stack([ix.ravel(), iy.ravel(), iz.ravel()], 1).astype(np.int32)
    if order != "stacked":
        eijk = eijk[np.random.default_rng(p).permutation(len(eijk))]
    if order == "part":
        eijk = np.ascontiguousarray(eijk[:7])
    E = len(eijk)
    Q = _state(E, N, 10 * N + p)
    L = closure.interpolation_matrix(N, p)
    out = torch.full((3, nz * p, ny * p, nx * p), np.nan, dtype=torch.float64, device="cuda")
    Qd, ed = torch.from_numpy(Q).cuda(), torch.from_numpy(eijk).cuda()
    rc = abi.load_library().cmdg_interpolate_equispaced(
        C.c_void_p(Qd.data_ptr()), C.c_void_p(ed.data_ptr()), E, N, p, C.c_void_p(np.ascontiguousarray(L).ctypes.data),
        nx * p, ny * p, nz * p, C.c_void_p(out.data_ptr()), C.c_void_p(torch.cuda.current_stream().cuda_stream))
    assert rc == abi.CMDG_OK
    got = out.cpu().numpy()
    u = (Q[:, 1:4] / Q[:, :1]).reshape(E, 3, q, q, q)
    v = np.einsum("zk,yj,xi,eckji->eczyx", L, L, L, u)
    ref = np.full(got.shape, np.nan)
    for e, (a, b, c) in enumerate(eijk):
        ref[:, c * p:c * p + p, b * p:b * p + p, a * p:a * p + p] = v[e]
    # three sums of q terms and a division, each product at most |u| max sum |L|^3
    tol = (3 * q + 2) * EPS * np.abs(u).max() * np.abs(L).sum(1).max() ** 3
    assert np.array_equal(np.isnan(got), np.isnan(ref))
    assert np.nanmax(np.abs(got - ref)) <= tol


@pytest.mark.parametrize("N", [3, 4])
@pytest.mark.parametrize("n", [1, 2, 5])
def test_box_filter(N, n):
    import torch
    from cmdg import abi, closure
    q, E = N + 1, n
    Q = _state(8 * E, N, N + n)
    ch = np.random.default_rng(n).permutation(8 * E).astype(np.int32)
    P = closure.filter_projection(N)
    Qd, cd = torch.from_numpy(Q).cuda(), torch.from_numpy(ch).cuda()
    out = torch.empty((E, 11, q ** 3), dtype=torch.float64, device="cuda")
    rc = abi.load_library().cmdg_box_filter(
        C.c_void_p(Qd.data_ptr()), C.c_void_p(cd.data_ptr()), E, N, C.c_void_p(np.ascontiguousarray(P).ctypes.data),
        C.c_void_p(out.data_ptr()), C.c_void_p(torch.cuda.current_stream().cuda_stream))
    assert rc == abi.CMDG_OK
    m = np.concatenate([Q] + [(Q[:, 1 + a] * Q[:, 1 + b] / Q[:, 0])[:, None] for a in range(3) for b in range(a, 3)], 1)
    m = m[ch].reshape(E, 2, 2, 2, 11, q, q, q)
    ref = np.einsum("zkc,yjb,xia,ezyxfcba->efkji", P, P, P, m).reshape(E, 11, q ** 3)
    tol = (3 * 2 * q + 4) * EPS * np.abs(m).max() * np.abs(P).sum((0, 2)).max() ** 3
    assert np.abs(out.cpu().numpy() - ref).max() <= tol


@pytest.mark.parametrize("N", [3, 4])
@pytest.mark.parametrize("ne", [(1, 1, 1), (3, 1, 2), (17, 13, 12), (29, 27, 26)])
def test_diagnostics(N, ne):
    import torch
    from cmdg import abi, atmos
    from cmdg.dg import DGModel
    from cmdg.grid import uniform_brick
    prm = atmos.ideal_gas_parameters()
    grid = uniform_brick(ne, (0, 0, 0), (1.0 * ne[0], 0.9 * ne[1], 1.1 * ne[2]), N=N, lean=True)
    cfg = atmos.AtmosConfig(prm, turbulence=abi.SMAGORINSKY_LILLY)
    dg = DGModel(cfg, grid)
    Q = _state(grid.nelem, N, ne[0])
    Q[:, 4] = 5.0 + np.abs(Q[:, 4])
    Qd = torch.from_numpy(Q).cuda()
    M = np.ascontiguousarray(grid.mass.T)
    for s in range(5):
        # double-double on the device: the product's and the result's rounding remain
        import math
        ref = math.fsum((M * Q[:, s]).ravel())
        assert abs(dg.weightedsum(Qd, s) - ref) <= 2 * EPS * np.abs(M * Q[:, s]).sum()
    x = [c.T.reshape(grid.nelem, N + 1, N + 1, N + 1) for c in grid.coords]
    md = np.full(x[0].shape, np.inf)
    for a, ax in ((0, 3), (1, 2), (2, 1)):
        d = np.abs(np.diff(x[a], axis=ax))
        lo = [slice(None)] * 4
        hi = [slice(None)] * 4
        lo[ax], hi[ax] = slice(0, N), slice(1, N + 1)
        md[tuple(lo)] = np.minimum(md[tuple(lo)], d)
        md[tuple(hi)] = np.minimum(md[tuple(hi)], d)
    u = np.sqrt((Q[:, 1:4] ** 2).sum(1)) / Q[:, 0]
    adv = (0.1 * u / md.reshape(u.shape)).max()
    assert abs(dg.courant(Qd, 0.1, "advective") - adv) <= 1e-14 * adv
    T = prm.T_0 + (Q[:, 4] / Q[:, 0] - u ** 2 / 2) / prm.cv_d
    c = np.sqrt(prm.cp_d / prm.cv_d * prm.R_d * T)
    ref = (0.1 * (u + c) / md.reshape(u.shape)).max()
    assert abs(dg.courant(Qd, 0.1, "nondiffusive") - ref) <= 1e-14 * ref
    assert dg.not_finite_fields(Qd) == []
    for s, e in ((0, 0), (2, grid.nelem - 1), (4, grid.nelem // 2)):
        Qb = Qd.clone()
        Qb[e, s, (N + 1) ** 3 - 1] = float("nan") if s else float("inf")
        assert len(dg.not_finite_fields(Qb)) == 1
    dg.close()
