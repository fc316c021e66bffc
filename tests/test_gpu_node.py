"""Kernels in which a thread owns its nodes and reads the neighbours through the caches, against the oracle.

Sizes where the split of the grid or the stencil form changes: planes of less than one 256-node run and of
many, z-chunks of several planes with a short last one, grids on which every node has a boundary row (narrower
than two closures), and periodic grids as narrow as the stencil.
"""
import numpy as np
import pytest

from inductioneq_amd.settings import ProgramConfig

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ops,n,per,tc,real", [
    ("2ndOrder", (130, 129, 33), False, "gaussian_rotation_3D", "float"),   # 66 runs, z-chunks of 3, last one full
    ("4thOrder", (200, 160, 19), False, "hall_travelling_wave", "double"),  # 125 runs, z-chunks of 3, last of 1
    ("6thOrder", (8, 9, 10), False, "rotation_3D", "double"),               # every node within a closure
    ("6thOrderExtended", (15, 40, 16), False, "alfven_periodic_2D", "float"),
    ("4thOrder", (5, 6, 7), True, "hall_periodic", "double"),               # as narrow as the stencil, one run
    ("6thOrder", (520, 513, 11), True, "confined_domain", "float"),          # more runs than blocks
])
def test_diagnostics_split(ops, n, per, tc, real):
    """Sums of at most 2.9 M terms of one sign in FP64 in another order: 1e-12 relative."""
    import torch

    from inductioneq_amd.program import Program
    from test_gpu_diagnostics import _cfg, _oracle_diag

    cfg = _cfg(ops, n, per, tc, real)
    prog = Program(cfg)
    B = np.random.default_rng(3).standard_normal((cfg.num_nodes, 3)).astype(cfg.dtype).astype(np.float64)
    b = prog.vector()
    b[:, : cfg.num_nodes] = torch.as_tensor(B.T.copy(), dtype=prog.torch_dtype)
    got = prog.diagnostics(b, 0.2)
    want = _oracle_diag(cfg, B, 0.2)
    for g, w in zip((got["energy"], got["divergence_norm"], got["error_norm"]), want):
        assert abs(g - w) <= 1e-12 * abs(w), (got, want)


def _stage_case(ops, n, per, hall, diss, real, seed=11):
    from test_gpu_tiled import FORMS, _cfg, _fields

    cfg = _cfg(ops, n, per, diss, FORMS[seed % len(FORMS)], "hall_periodic" if hall else "rotation_2D", real)
    cfg.hall = hall
    B, U = _fields(cfg, seed)
    return cfg, B, U


@pytest.mark.parametrize("ops,n,per,hall,diss,real", [
    ("4thOrder", (13, 5, 9), False, True, None, "double"),             # a run of 64 nodes and one of 1; y within two closures
    ("6thOrder", (8, 8, 7), False, True, "HIGH_ORDER", "double"),      # runs of exactly 64, boundary rows in every direction
    ("6thOrderExtended", (70, 16, 15), False, True, "ADAPTIVE", "double"),
    ("2ndOrderExtended", (5, 30, 6), True, True, "FIRST_ORDER", "double"),
    ("4thOrderExtended", (12, 11, 65), False, False, "ADAPTIVE", "float"),
    ("6thOrder", (130, 11, 10), True, False, "HIGH_ORDER", "float"),     # periodic, runs across row ends
    ("2ndOrder", (2, 20, 18), False, True, None, "double"),            # two nodes in x
    ("6thOrderExtended", (64, 8, 17), False, False, "FIRST_ORDER", "float"),  # y as narrow as the reference reads in bounds
])
@pytest.mark.parametrize("part", [False, True])
def test_node_kernels_equal_oracle(ops, n, per, hall, diss, real, part):
    """calc_curlB_rho, calc_u and the two kinds of stage (SSPRK33_3b: two operands; CarpenterKennedy2N54_2a: in
    place) against the oracle, on the whole grid and on a part of it whose other nodes stay as they were.
    FP64 1e-12 of the largest value (sums of at most 3 x 15 x 9 products), FP32 2e-5."""
    import os

    import torch
    from pyoracle import Oracle

    from inductioneq_amd.program import Program
    from test_gpu_tiled import TOL, _aos

    cfg, B, U = _stage_case(ops, n, per, hall, diss, real)
    g = tuple(max(1, v - 1 - k) for k, v in enumerate(n)) if part else n
    prog, orc = Program(cfg), Oracle(cfg)
    rng = np.random.default_rng(4)
    regs = [_aos(cfg, B + 0.1 * rng.standard_normal(B.shape)) for _ in range(3)]
    rho = (1.0 + 0.2 * rng.random(cfg.num_nodes_pad)).astype(cfg.dtype)
    os.environ["IEQ_NO_TILED"] = "1"
    try:
        for names, nf in ((["calc_curlB_rho_3_3args", "calc_u_3_args", "SSPRK33_3b"], 3),
                          (["calc_curlB_rho_1_2args", "CarpenterKennedy2N54_2a"], 2)):
            names = [k for k in names if hall or not k.startswith("calc_curlB")]
            host = [r.copy() for r in regs[:nf]] + [orc.vec(), _aos(cfg, U), rho.copy(), orc.time(0.3)]
            dev = [prog.upload_real4(a) for a in host[: nf + 2]] + [prog.upload_real(host[nf + 2])]
            dev.append(torch.tensor([0.3, 0.3], dtype=prog.torch_dtype, device="cuda"))
            for k in names:
                orc.run(k, host, g=g)
                prog.run(k, dev, g=g)
            for i in range(nf + 2):
                got = prog.download_real4(dev[i])[: cfg.num_nodes, :3].astype(np.float64)
                want = host[i][: cfg.num_nodes, :3].astype(np.float64)
                e = np.abs(got - want).max() / max(np.abs(want).max(), 1e-300)
                assert e <= TOL[real], (names, i, e)
    finally:
        os.environ.pop("IEQ_NO_TILED", None)


@pytest.mark.parametrize("ops", ["2ndOrder", "4thOrder", "6thOrder", "2ndOrderExtended", "4thOrderExtended", "6thOrderExtended"])
@pytest.mark.parametrize("diss,real", [(None, "double"), ("HIGH_ORDER", "float"), ("FIRST_ORDER", "double")])
def test_tiled_stage_on_small_grids(ops, diss, real):
    """The z-marching kernel where a thread per node would be taken (a stated z-chunk keeps the tiles)."""
    from test_gpu_tiled import FORMS, _cfg, _check, _run_both

    cfg = _cfg(ops, (37, 21, 19), False, diss, FORMS[2], "rotation_2D", real)
    prog, db, hb, path = _run_both(cfg, "SSPRK33", env={"IEQ_TILED_ZC": "4"})
    assert path == "tiled"
    _check(cfg, prog, db, hb, "SSPRK33", "%s %s" % (ops, diss))


@pytest.mark.parametrize("integrator", ["SSPRK33", "SSPRK104", "KennedyCarpenterLewis2R54C", "CalvoFrancoRandez2R64",
                                        "CarpenterKennedy2N54", "ToulorgeDesmet2N84F"])
@pytest.mark.parametrize("per,hall,real", [(False, True, "double"), (True, True, "float"), (False, False, "double")])
def test_kernel_list_equals_its_kernels_one_by_one(integrator, per, hall, real):
    """A list shares launches (curl + velocity, time kernels, the halves of a 2N stage with a second copy of b1);
    after it every argument is what the kernels leave one by one.  Whole lists of one and three steps (odd and even
    numbers of 2N stages), and lists that end within a step: after a time kernel, between the halves of a stage.
    The arithmetic per node is the same; 1e-13 (FP32 1e-6) of the largest value allows for other contractions."""
    import torch

    from inductioneq_amd.program import Program
    from inductioneq_amd.schedules import rk_schedule
    from test_gpu_tiled import _aos

    cfg, B, U = _stage_case("4thOrder", (21, 10, 12), per, hall, None, real)
    prog = Program(cfg)
    names, nf = rk_schedule(integrator, hall, True)
    rng = np.random.default_rng(8)
    host = [_aos(cfg, B + 0.1 * rng.standard_normal(B.shape)) for _ in range(nf)]

    def fresh():
        a = [prog.upload_real4(h) for h in host] + [prog.vector(), prog.upload_real4(_aos(cfg, U)), prog.scalar(1.3)]
        return a + [torch.tensor([0.2, 0.25], dtype=prog.torch_dtype, device="cuda")]

    tol = 1e-13 if real == "double" else 1e-6
    for lst in [names, names * 3] + [names[:k] for k in range(len(names) // 2, len(names) // 2 + 5)]:
        one, all_ = fresh(), fresh()
        for k in lst:
            prog.run(k, one)
        prog.run(lst, all_)
        torch.cuda.synchronize()
        for i, (x, y) in enumerate(zip(all_, one)):
            x, y = (v[..., : cfg.num_nodes].double() if v.numel() > 2 else v.double() for v in (x, y))
            assert float((x - y).abs().max()) <= tol * max(float(y.abs().max()), 1e-300), (len(lst), i)


def test_lists_on_two_streams_share_the_second_copy_of_b1():
    """Two solves of one program on two streams in turn, without a wait between the calls, equal the same solves
    one after the other bit for bit."""
    import torch

    from inductioneq_amd.program import Program
    from inductioneq_amd.schedules import rk_schedule
    from test_gpu_tiled import _aos

    cfg, B, U = _stage_case("6thOrder", (48, 40, 44), False, True, None, "double")
    cfg.dt = 1e-5  # within the Hall term's stability limit: the states stay finite
    prog = Program(cfg)
    names, nf = rk_schedule("CarpenterKennedy2N54", True, True)

    def solve(streams, scale):
        regs = [[prog.upload_real4(_aos(cfg, B * c))] + [prog.vector() for _ in range(nf)] +
                [prog.upload_real4(_aos(cfg, U)), prog.scalar(1.0), prog.time_buffer()] for c in scale]
        torch.cuda.synchronize()
        for _ in range(4):
            for s, a in zip(streams, regs):
                with torch.cuda.stream(s):
                    prog.use_current_stream()
                    prog.run(names * 2, a)
        torch.cuda.synchronize()
        return [a[0].clone() for a in regs]

    s1, s2 = torch.cuda.Stream(), torch.cuda.Stream()
    both = solve((s1, s2), (1.0, 0.5))
    assert bool(torch.isfinite(both[0]).all())
    assert torch.equal(both[0], solve((s1,), (1.0,))[0])
    assert torch.equal(both[1], solve((s1,), (0.5,))[0])
