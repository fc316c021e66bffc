"""curl B, curl B / rho and the velocity with a thread per node and with the directions on waves of their own, against
the oracle: planes of one node less and more than a block's 256, boundary rows in every wave and in some, and both
sides of the rule between the two kernels."""
import math

import numpy as np
import pytest

from inductioneq_amd.settings import ProgramConfig

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ops,n,per,real", [
    ("2ndOrder", (17, 15, 9), False, "float"),            # a block of 255: rows of three directions loaded together
    ("2ndOrder", (256, 3, 5), False, "float"),            # waves without and with an x face
    ("2ndOrderExtended", (257, 5, 12), False, "float"),
    ("2ndOrderExtended", (70, 66, 20), False, "double"),
    ("4thOrder", (16, 16, 9), False, "double"),           # one block a plane
    ("4thOrder", (130, 40, 9), False, "float"),
    ("4thOrder", (130, 40, 30), False, "float"),          # 156 k nodes: a thread per node, beyond it
    ("4thOrder", (90, 85, 60), False, "double"),          # 459 k
    ("2ndOrder", (90, 50, 41), True, "double"),           # 184 k
    ("6thOrder", (200, 20, 14), False, "double"),         # directions on waves of their own
    ("6thOrder", (200, 20, 14), False, "float"),
    ("6thOrderExtended", (20, 130, 17), False, "double"),
    ("6thOrder", (130, 129, 110), False, "double"),       # 1.84 M nodes: a thread per node
    ("2ndOrder", (130, 122, 118), False, "float"),        # columns
    ("2ndOrderExtended", (200, 96, 99), False, "float"),
    ("6thOrder", (257, 9, 10), True, "float"),            # periodic: central rows only
    ("4thOrderExtended", (11, 93, 12), True, "double"),
])
@pytest.mark.parametrize("part", [False, True])
def test_curl_and_velocity_equal_oracle(ops, n, per, real, part):
    """FP64 1e-12 of the largest value (two sums of at most 15 products), FP32 2e-5."""
    import torch
    from pyoracle import Oracle

    from inductioneq_amd.program import Program
    from test_gpu_parity import _aos, _relerr

    lo, hi = (0.0, 2 * math.pi) if per else (-1.0, 1.0)
    cfg = ProgramConfig(real=real, opset=ops, nx=n[0], ny=n[1], nz=n[2], xmin=lo, xmax=hi, ymin=lo, ymax=hi, zmin=lo,
                        zmax=hi, periodic=per, hall=True, testcase="hall_periodic", w_size=64)
    prog, orc = Program(cfg), Oracle(cfg)
    g = tuple(max(1, v - 1 - k) for k, v in enumerate(n)) if part else n
    rng = np.random.default_rng(6)
    tol = 1e-12 if real == "double" else 2e-5
    hb = _aos(cfg, rng.standard_normal((cfg.num_nodes, 3)))
    hc = _aos(cfg, np.full((cfg.num_nodes, 3), 3.0))
    db, dc = prog.upload_real4(hb), prog.upload_real4(hc)
    orc.run("calc_curl", [hb, hc], g=g)
    prog.run("calc_curl", [db, dc], g=g)
    assert _relerr(prog.download_real4(dc)[: cfg.num_nodes, :3], hc[: cfg.num_nodes, :3]) <= tol

    hr = (1.0 + 0.2 * rng.random(cfg.num_nodes_pad)).astype(cfg.dtype)
    host = [hb, hb.copy(), hb.copy(), _aos(cfg, np.full((cfg.num_nodes, 3), 3.0)), _aos(cfg, np.full((cfg.num_nodes, 3), 2.0)),
            hr, orc.time(0.4)]
    dev = [prog.upload_real4(a) for a in host[:5]] + [prog.upload_real(hr), prog.time_buffer(0.4)]
    names = ["calc_curlB_rho_2_3args", "calc_u_3_args"]
    orc.run(names, host, g=g)
    for lst in (names[:1], names[1:], names):
        for k in (3, 4):
            dev[k].fill_(3.0 if k == 3 else 2.0)
        prog.run(lst, dev, g=g)
        torch.cuda.synchronize()
        for k, name in ((3, names[0]), (4, names[1])):
            if name in lst:
                assert _relerr(prog.download_real4(dev[k])[: cfg.num_nodes, :3], host[k][: cfg.num_nodes, :3]) <= tol, (lst, name)
            else:
                assert bool((dev[k] == (3.0 if k == 3 else 2.0)).all())


@pytest.mark.parametrize("ops,n,per,real", [
    ("6thOrder", (130, 120, 118), False, "float"),          # columns, z-chunks of 1; boundary rows in most x waves
    ("2ndOrderExtended", (200, 90, 101), False, "double"),  # columns
    ("4thOrder", (128, 64, 230), True, "double"),           # columns, periodic
    ("6thOrderExtended", (130, 120, 118), False, "double"),  # a thread per node: wide rows in FP64
    ("4thOrder", (300, 230, 31), False, "float"),           # ... and few planes
    ("6thOrder", (257, 13, 14), False, "float"),
    ("2ndOrder", (9, 85, 12), True, "float"),
    ("2ndOrder", (300, 31, 8), False, "float"),             # short rows in FP32: loaded together
    ("2ndOrderExtended", (20, 19, 40), False, "float"),
])
@pytest.mark.parametrize("part", [False, True])
def test_operators_on_both_sides_of_the_column_rule(ops, n, per, real, part):
    from test_gpu_node import test_column_kernels_equal_oracle as check

    check(ops, n, per, real, part)
