"""The z-marching kernels at the sizes of the oracle tests, where the dispatch takes bricks or a thread per node: the
kernels that larger grids run, over half-widths, stage forms, dissipation, Hall term, flux forms and both precisions."""

import numpy as np
import pytest

from inductioneq_amd.schedules import INTEGRATORS

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("brick", ["0", "1"])
@pytest.mark.parametrize("real", ["double", "float"])
@pytest.mark.parametrize("ops", ["2ndOrder", "4thOrder", "6thOrder"])
@pytest.mark.parametrize("integrator", INTEGRATORS)
@pytest.mark.parametrize("hall,diss,u", [(True, "HIGH_ORDER", (0.0, 0.0, 0.0)), (True, "HIGH_ORDER", (0.3, -0.2, 0.1)),
                                         (True, None, (0.0, 0.0, 0.0)), (True, None, (0.3, -0.2, 0.1)),
                                         (False, "HIGH_ORDER", (0.5, 0.2, -0.4)), (False, None, (0.5, 0.2, -0.4))])
def test_fused_step_in_either_kernel_family(ops, integrator, hall, diss, u, real, brick, monkeypatch):
    """As test_fused_step_matches_reference_schedule, with the z-marches (IEQ_BRICK = 0: one kernel per Hall stage, the
    stage march without the Hall term) and with the bricks."""
    from test_gpu_parity import test_fused_step_matches_reference_schedule as check

    monkeypatch.setenv("IEQ_BRICK", brick)
    check(ops, integrator, hall, diss, u, real)


@pytest.mark.parametrize("ops,n,integrator,source,real", [
    ("6thOrder", (31, 11, 13), "SSPRK33", "ZERO", "double"),
    ("6thOrder", (33, 16, 10), "CarpenterKennedy2N54", "CENTRAL", "float"),
    ("4thOrder", (65, 8, 9), "SSPRK104", "ZERO", "double"),
    ("2ndOrder", (37, 17, 5), "KennedyCarpenterLewis2R54C", "ZERO", "float"),
])
def test_split_hall_march_equals_oracle(ops, n, integrator, source, real):
    """The march pair (EMF, then the stage) that FP32 stages with convection take beyond the bricks, at ragged sizes:
    1e-12 and 2e-5 of the largest value as for the other fused kernels."""
    import torch
    from test_gpu_fused import TOL, _device_args, _Env, _oracle_steps, _periodic_cfg, _relerr

    from inductioneq_amd.problems import hall_dt, random_modes_field
    from inductioneq_amd.program import Program

    u = (0.3, -0.2, 0.1)
    cfg = _periodic_cfg(n, real, ops, True, "HIGH_ORDER", u, ho_factor=0.5, form_source=source)
    B0 = random_modes_field(n, seed=4, kmax=2, amp=0.3)
    cfg.dt = hall_dt(B0, (cfg.dx, cfg.dy, cfg.dz), 6, c_hall=0.8, cfl=0.3)
    prog = Program(cfg)
    args = _device_args(prog, B0, 2 if "2N" in integrator else 3, u, 1.25)
    with _Env(IEQ_BRICK=0, IEQ_FUSED_SPLIT=1):
        prog.step(integrator, 2, args)
        torch.cuda.synchronize()
    assert prog.last_step_fused
    hb, _ = _oracle_steps(cfg, B0, integrator, 2, u, 1.25)
    e = _relerr(args[0][:, : cfg.num_nodes].double().cpu().numpy().T, hb[0][: cfg.num_nodes, :3].astype(np.float64))
    assert e <= TOL[real], e


@pytest.mark.parametrize("zc", ["3", "32"])
@pytest.mark.parametrize("ops", ["2ndOrder", "4thOrder", "6thOrder", "2ndOrderExtended", "4thOrderExtended", "6thOrderExtended"])
@pytest.mark.parametrize("diss", [None, "HIGH_ORDER", "FIRST_ORDER"])
@pytest.mark.parametrize("per,real", [(False, "double"), (False, "float"), (True, "double"), (True, "float")])
def test_tiled_stage_kernel(ops, diss, per, real, zc):
    """The z-marching stage kernel of the reference schedule (a stated z-chunk keeps it on small grids): every operator
    set and dissipation, every flux form over the cases, bounded with SAT data and periodic with a velocity of time."""
    from test_gpu_tiled import FORMS, OPSETS, _cfg, _check, _run_both

    k = OPSETS.index(ops) + 3 * [None, "HIGH_ORDER", "FIRST_ORDER"].index(diss) + 2 * per + (real == "float")
    cfg = _cfg(ops, (37, 21, 19), per, diss, FORMS[k % len(FORMS)], "alfven_periodic_2D" if per else "rotation_2D", real)
    prog, db, hb, path = _run_both(cfg, "SSPRK33", variable_u=per, env={"IEQ_TILED_ZC": zc})
    assert path == "tiled"
    _check(cfg, prog, db, hb, "SSPRK33", "%s %s %s %s" % (ops, diss, per, real))


@pytest.mark.parametrize("integrator", INTEGRATORS)
@pytest.mark.parametrize("per", [False, True])
def test_tiled_stage_kernel_in_every_integrator(integrator, per):
    from test_gpu_tiled import FORMS, _cfg, _check, _run_both

    cfg = _cfg("4thOrder", (40, 26, 22), per, None, FORMS[per], "alfven_periodic_2D" if per else "gaussian_rotation_3D", "double")
    prog, db, hb, path = _run_both(cfg, integrator, variable_u=per, env={"IEQ_TILED_ZC": "5"})
    assert path == "tiled"
    _check(cfg, prog, db, hb, integrator, integrator)


@pytest.mark.parametrize("real,n", [("double", (76, 75, 74)), ("float", (110, 106, 104))])
def test_tiled_stage_kernel_where_the_rule_takes_it(real, n):
    """Periodic grids of a few nodes more than the rule's bound (400 k FP64, 1.2 M FP32) against a thread per node, one
    step: the same sums in another order, 1e-13 and 1e-6 of the largest value."""
    import torch
    from test_gpu_tiled import FORMS, _aos, _cfg, _fields

    from inductioneq_amd.program import Program
    from inductioneq_amd.schedules import rk_schedule

    cfg = _cfg("6thOrder", n, True, "HIGH_ORDER", FORMS[3], "alfven_periodic_2D", real)
    prog = Program(cfg)
    names, nf = rk_schedule("SSPRK33", False, True)
    B, U = _fields(cfg, 9)
    import os

    out = {}
    for mode in ("0", "1"):
        os.environ["IEQ_NO_TILED"] = mode
        try:
            regs = [prog.upload_real4(_aos(cfg, B))] + [prog.vector() for _ in range(nf - 1)]
            prog.run(names, regs + [prog.vector(), prog.upload_real4(_aos(cfg, U)), prog.scalar(1.0), prog.time_buffer(0.1)])
            torch.cuda.synchronize()
        finally:
            os.environ.pop("IEQ_NO_TILED", None)
        out[mode] = regs[0][:, : cfg.num_nodes].double()
    e = float((out["0"] - out["1"]).abs().max() / out["1"].abs().max())
    assert e <= (1e-13 if real == "double" else 1e-6), e
