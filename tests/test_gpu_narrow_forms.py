"""The narrow kernels, which large meshes run, on small ones (CMDG_WIDE_BLOCKS=0), where the
defaults take wide blocks and the storage order: the neighbours' static trace, per-element
static fields, element orders, and the brick constructor's order."""
import os

import numpy as np
import pytest

from cmdg import abi, atmos
from oracle import oracle as O
from test_gpu_block_forms import _run, _same
from test_gpu_brick import _cases as brick_cases
from test_gpu_fullsize import rel_l2
from test_gpu_parity import MIXED_RHS_RTOL, RTOL, _case

pytestmark = pytest.mark.gpu
PRECISIONS = [abi.FP64, abi.MIXED]


def _model(cfg, grid, aux, precision, **env):
    from cmdg.dg import DGModel
    os.environ.update(env)
    try:
        return DGModel(cfg, grid, aux=aux, precision=precision)
    finally:
        for k in env:
            os.environ.pop(k)


@pytest.mark.parametrize("steps", [0, 3])
@pytest.mark.parametrize("N", [3, 4])
@pytest.mark.parametrize("precision", PRECISIONS)
@pytest.mark.parametrize("form", [{"CMDG_NEIGHBOUR_STATIC_TRACE": "1"}, {"CMDG_STATIC_AUX_CLASSES": "0"},
                                  {"CMDG_NEIGHBOUR_STATIC_TRACE": "1", "CMDG_STATIC_AUX_CLASSES": "0"},
                                  {"CMDG_ELEMENT_TILE": "2", "CMDG_TILED_PASSES": "both"},
                                  {"CMDG_ELEMENT_TILE": "2,0,2", "CMDG_TILED_PASSES": "both"}],
                         ids=["trace", "no classes", "trace, no classes", "tiles", "columns"])
def test_narrow_forms_agree(form, precision, N, steps):
    case = _case("les_walls", N)
    dg = _model(*case[:3], precision, CMDG_WIDE_BLOCKS="0", **form)
    assert dg.static_aux_continuous == ("CMDG_NEIGHBOUR_STATIC_TRACE" not in form)
    assert dg.static_aux_classes == ("CMDG_STATIC_AUX_CLASSES" not in form)
    assert dg.tiled_traversal == ("CMDG_ELEMENT_TILE" in form)
    dg.close()
    _same(_run(*case, precision, steps, CMDG_WIDE_BLOCKS="0"), _run(*case, precision, steps, CMDG_WIDE_BLOCKS="0", **form))


@pytest.mark.parametrize("wide", ["0", "1"])
@pytest.mark.parametrize("N", [3, 4])
@pytest.mark.parametrize("precision", PRECISIONS)
@pytest.mark.parametrize("field", ["ref_rho", "ref_p", "Phi"])
def test_per_element_static_fields(field, precision, N, wide):
    """A static field that differs from node to node, so on the two sides of every face:
    ref_p and Phi take the neighbour's static trace.  Against the oracle."""
    import torch
    from cmdg.dg import to_device, to_host
    cfg, grid, aux, Q0 = _case("les_walls", N)
    aux = np.array(aux, order="F", copy=True)
    k = cfg.layout[field]
    aux[:, k, :] *= 1 + 1e-3 * np.random.default_rng(17).uniform(-1, 1, aux[:, k, :].shape)
    ref = O.Oracle(cfg, grid, aux).tendency(Q0)
    dg = _model(cfg, grid, aux, precision, CMDG_WIDE_BLOCKS=wide)
    assert dg.geometry_kind == "affine" and not dg.static_aux_classes
    assert dg.static_aux_continuous == (field == "ref_rho")
    Q = to_device(Q0)
    dQ = torch.full_like(Q, float("nan"))
    dg(dQ, Q, None, 0.0)
    got = to_host(dQ)
    for s in range(5):
        r = rel_l2(got[:, s], ref[:, s])
        assert r < (RTOL if precision == abi.FP64 else MIXED_RHS_RTOL), (s, r)
    dg.close()


@pytest.mark.parametrize("case", [c[0] for c in brick_cases()])
def test_brick_order_is_the_array_order(case):
    """2 x 2 columns in both passes of a brick given by its break points against those of the same
    brick given by arrays, with the narrow blocks that large meshes run."""
    from cmdg.dg import to_device
    from cmdg import closure
    from cmdg.grid import uniform_brick
    import torch
    name, prm, g, cfg, precision = next(c for c in brick_cases() if c[0] == case)
    kw = dict(N=4, periodicity=g["periodicity"], boundary=g["boundary"])
    full = uniform_brick(g["n"], g["lo"], g["hi"], **kw)
    aux = atmos.init_aux(cfg, full)
    Q0 = (atmos.taylor_green(prm, full, mach=0.1) if name.startswith("tgv") else
          atmos.rising_bubble(prm, full, radius=100.0, centre=(200.0, 150.0, 150.0), seed=5))
    out = []
    for grid in (full, uniform_brick(g["n"], g["lo"], g["hi"], lean=True, **kw)):
        dg = _model(cfg, grid, aux, precision, CMDG_WIDE_BLOCKS="0", CMDG_ELEMENT_TILE="2,0,2", CMDG_TILED_PASSES="both")
        assert dg.tiled_traversal
        if cfg.turbulence == abi.LEARNED_CLOSURE:
            dg.set_closure(closure.MLPParams.constant(0.21 ** 2))
        Q = to_device(Q0)
        T = torch.full_like(Q, float("nan"))
        dg(T, Q, None, 0.0)
        out.append(T.cpu())
        dg.close()
    assert torch.isfinite(out[0]).all() and torch.equal(out[0], out[1])


@pytest.mark.parametrize("shape", [(13, 2, 13), (11, 3, 23), (30, 3, 4), (2, 5, 37), (16, 2, 16)])
@pytest.mark.parametrize("precision", PRECISIONS)
def test_default_columns_narrow(precision, shape):
    """The default columns in both passes against the storage order, narrow blocks in both."""
    from cmdg.grid import uniform_brick
    prm = atmos.ideal_gas_parameters()
    grid = uniform_brick(shape, (0.0, 0.0, 0.0), (6.0, 5.0, 4.0), N=4)
    cfg = atmos.AtmosConfig(prm, turbulence=abi.SMAGORINSKY_LILLY, C_smag=0.21)
    Q0 = atmos.taylor_green(prm, grid, mach=0.1)
    Q0[:, 1:4, :] *= 1 + 0.05 * np.random.default_rng(7).uniform(-1, 1, Q0[:, 1:4, :].shape)
    case = (cfg, grid, atmos.init_aux(cfg, grid), Q0)
    walk = dict(CMDG_WIDE_BLOCKS="0", CMDG_TILED_PASSES="both")
    dg = _model(*case[:3], precision, **walk)
    assert dg.tiled_traversal
    dg.close()
    _same(_run(*case, precision, 0, **walk), _run(*case, precision, 0, CMDG_WIDE_BLOCKS="0", CMDG_ELEMENT_TILE="0"))
