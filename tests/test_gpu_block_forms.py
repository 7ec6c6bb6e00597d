"""Forms of the brick passes that only choose who computes what, or through which buffer the
state goes: wide blocks (the face tasks in waves of their own), and an odd number of steps
through the third state buffer, by the copy kernel and by the gradient pass's copy.  Every
form gives the same bits."""
import os

import numpy as np
import pytest

from cmdg import abi, atmos
from test_gpu_parity import CASES, _case

pytestmark = pytest.mark.gpu


def _run(cfg, grid, aux, Q0, precision, steps, mlp=None, **env):
    from cmdg.dg import DGModel, LSRK54CarpenterKennedy, solve, to_device, to_host
    import torch
    os.environ.update(env)
    try:
        dg = DGModel(cfg, grid, aux=aux, precision=precision)
    finally:
        for k in env:
            os.environ.pop(k)
    if mlp is not None:
        dg.set_closure(mlp)
    Q = to_device(Q0)
    if steps == 0:
        T = torch.full_like(Q, 0.5)
        dg(T, Q, None, 0.0, 2.0, 0.25)
        out = [to_host(T)]
    else:
        solver = LSRK54CarpenterKennedy(dg, Q, dt=1e-4, t0=0.0)
        solve(Q, solver, numberofsteps=steps)
        out = [to_host(Q), to_host(solver.dQ)]
    out.append(to_host(dg.state_auxiliary))
    dg.close()
    return out


def _same(a, b):
    for x, y in zip(a, b):
        assert np.isfinite(x).all() and np.array_equal(x, y)


@pytest.mark.parametrize("steps", [0, 1, 2])
@pytest.mark.parametrize("N", [3, 4])
@pytest.mark.parametrize("precision", [abi.FP64, abi.MIXED])
@pytest.mark.parametrize("name", CASES)
def test_wide_blocks(name, precision, N, steps):
    case = _case(name, N)
    _same(_run(*case, precision, steps, CMDG_WIDE_BLOCKS="0"), _run(*case, precision, steps, CMDG_WIDE_BLOCKS="1"))


@pytest.mark.parametrize("N", [3, 4])
@pytest.mark.parametrize("name", ["les_walls", "tgv_smagorinsky"])
def test_wide_blocks_learned(name, N):
    from cmdg import closure
    cfg, grid, aux, Q0 = _case(name, N)
    kw = dict(orientation=cfg.orientation, ref_profile=cfg.ref_profile, gravity_source=cfg.gravity_source)
    cfg = atmos.AtmosConfig(cfg.params, turbulence=abi.LEARNED_CLOSURE, C_smag=0.21, **kw)
    mlp = closure.MLPParams.random(seed=5, y0=0.04, scale=np.r_[np.full(9, 0.05), 0.01])
    for steps in (0, 1):
        _same(_run(cfg, grid, aux, Q0, abi.MIXED, steps, mlp, CMDG_WIDE_BLOCKS="0"),
              _run(cfg, grid, aux, Q0, abi.MIXED, steps, mlp, CMDG_WIDE_BLOCKS="1"))


@pytest.mark.parametrize("steps", [1, 3, 4])
@pytest.mark.parametrize("variant", ["euler_periodic", "les_walls", "les_walls general", "tgv_smagorinsky mixed"])
def test_state_buffers(variant, steps):
    name, _, form = variant.partition(" ")
    case = _case(name)
    env = {"CMDG_GENERAL_GEOMETRY": "1"} if form == "general" else {}
    prec = abi.MIXED if form == "mixed" else abi.FP64
    _same(_run(*case, prec, steps, **env), _run(*case, prec, steps, CMDG_THIRD_STATE_BUFFER="0", **env))


@pytest.mark.parametrize("steps", [0, 2])
@pytest.mark.parametrize("N", [3, 4])
@pytest.mark.parametrize("name", CASES)
def test_wide_blocks_general(name, N, steps):
    case = _case(name, N)
    env = {"CMDG_GENERAL_GEOMETRY": "1"}
    _same(_run(*case, abi.FP64, steps, CMDG_WIDE_BLOCKS="0", **env),
          _run(*case, abi.FP64, steps, CMDG_WIDE_BLOCKS="1", **env))


@pytest.mark.parametrize("shape", [(11, 3, 23), (2, 5, 37), (21, 2, 20)])
@pytest.mark.parametrize("precision", [abi.FP64, abi.MIXED])
def test_columns_walk_every_element(precision, shape):
    """The default columns on cross-sections that no column count divides."""
    from cmdg.grid import uniform_brick
    prm = atmos.ideal_gas_parameters()
    grid = uniform_brick(shape, (0.0, 0.0, 0.0), (6.0, 5.0, 4.0), N=3)
    cfg = atmos.AtmosConfig(prm, turbulence=abi.SMAGORINSKY_LILLY, C_smag=0.21)
    Q0 = atmos.taylor_green(prm, grid, mach=0.1)
    Q0[:, 1:4, :] *= 1 + 0.05 * np.random.default_rng(7).uniform(-1, 1, Q0[:, 1:4, :].shape)
    case = (cfg, grid, atmos.init_aux(cfg, grid), Q0)
    _same(_run(*case, precision, 0, CMDG_TILED_PASSES="both"), _run(*case, precision, 0, CMDG_ELEMENT_TILE="0"))
