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


@pytest.mark.parametrize("ops,lap,n,zc,real", [
    ("4thOrder", "WIDE_STENCIL_DIRICHLET", (40, 36, 30), "8", "double"),        # half-width 4: ragged tiles, last chunk of 4
    ("2ndOrder", "NARROW_STENCIL_DIRICHLET", (67, 18, 13), "2", "double"),      # half-width 1: three tiles in x, one plane left
    ("2ndOrder", "WIDE_STENCIL_DIRICHLET", (34, 34, 9), "16", "float"),         # half-width 2: one chunk longer than the grid
    ("2ndOrderExtended", "WIDE_STENCIL_LNS", (26, 24, 28), "12", "double"),     # half-width 3, no boundary nodes left out
    ("4thOrder", "WIDE_STENCIL_LNS", (33, 17, 28), "10", "float"),              # half-width 5
    ("4thOrderExtended", "WIDE_STENCIL_DIRICHLET", (70, 30, 32), "8", "double"),  # half-width 6: 64 x 8 tiles
])
def test_cg_march_equals_oracle(ops, lap, n, zc, real, monkeypatch):
    """The Laplacian's z-march on small grids (there a thread per node is the rule) against the oracle after
    8 iterations: FP64 1e-10 of the largest value as for the other form; FP32 1e-4 (rounding of 2^-24 over
    27 terms and 8 iterations, times the condition of the first ones, which is below 60)."""
    import torch

    from inductioneq_amd.harness import clean_div_cg
    from test_gpu_cg import _setup

    monkeypatch.setenv("IEQ_LAP_ZC", zc)
    prog, orc, cfg, aos = _setup(ops, lap, n, real)
    aos = aos.astype(np.float32).astype(np.float64)
    hb = aos.copy()
    want = clean_div_cg(orc.cfg, orc, hb, 1e-9, 8)
    db = prog.upload_real4(aos.astype(cfg.dtype))
    got = prog.clean_div_cg(db, abs_threshold=1e-9, max_iterations=8)
    torch.cuda.synchronize()
    tol = 1e-10 if real == "double" else 1e-4
    assert got["iterations"] == want["iterations"] == 8
    phi_w, phi_g = want["phi"][: cfg.num_nodes], prog.download_real(got["phi"])[: cfg.num_nodes]
    assert np.abs(phi_g - phi_w).max() <= tol * np.abs(phi_w).max()
    b_g = prog.download_real4(db)[: cfg.num_nodes, :3]
    assert np.abs(b_g - hb[: cfg.num_nodes, :3]).max() <= tol * np.abs(hb[:, :3]).max()


@pytest.mark.parametrize("zc", [None, "8"])
def test_cg_calls_leave_nothing_behind(zc, monkeypatch):
    """A solve after one of a field without divergence (no iteration, field unchanged), one of NaN and one that
    was cut short equals the first solve of a program bit for bit."""
    import torch
    from test_gpu_cg import _setup

    if zc:
        monkeypatch.setenv("IEQ_LAP_ZC", zc)
    prog, _, cfg, aos = _setup("4thOrder", "WIDE_STENCIL_DIRICHLET", (35, 33, 34), "double")
    first = prog.upload_real4(aos)
    r1 = prog.clean_div_cg(first, abs_threshold=1e-6, max_iterations=25)
    zero = prog.vector()
    r0 = prog.clean_div_cg(zero, abs_threshold=1e-6, max_iterations=25)
    assert r0["iterations"] == 0 and not zero.any() and not r0["phi"].any()
    bad = torch.full_like(first, float("nan"))
    prog.clean_div_cg(bad, abs_threshold=1e-6, max_iterations=25)
    inf = torch.zeros_like(first)
    inf[0, cfg.num_nodes // 2] = float("inf")
    prog.clean_div_cg(inf, abs_threshold=1e-6, max_iterations=25)
    prog.clean_div_cg(prog.upload_real4(2.0 * aos), abs_threshold=1e-6, max_iterations=3)
    again = prog.upload_real4(aos)
    r2 = prog.clean_div_cg(again, abs_threshold=1e-6, max_iterations=25)
    torch.cuda.synchronize()
    assert r1["iterations"] == r2["iterations"] == 25
    assert torch.equal(first, again) and torch.equal(r1["phi"], r2["phi"])
    assert r1["divergence_norm_final"] == r2["divergence_norm_final"]


@pytest.mark.parametrize("ops,n,per,real", [
    ("4thOrder", (200, 160, 101), False, "float"),         # 125 runs of 256 nodes, z-chunks of 3, the last of 2
    ("6thOrder", (16, 16, 9), False, "double"),            # one run exactly, boundary rows on most planes
    ("2ndOrderExtended", (257, 5, 6), True, "double"),     # the last run of 5 nodes
    ("6thOrderExtended", (19, 27, 33), True, "float"),     # 513 nodes: two runs and one node
    ("2ndOrder", (2, 85, 3), False, "double"),
    ("4thOrderExtended", (300, 130, 61), True, "double"),  # periodic, z-chunks of 2, the last of 1
])
@pytest.mark.parametrize("part", [False, True])
def test_column_kernels_equal_oracle(ops, n, per, real, part):
    """Divergence, curl, gradient and projection on the whole grid and on a part of it whose other nodes stay as
    they were: FP64 1e-12 of the largest value (three sums of at most 11 products), FP32 2e-5."""
    import torch
    from pyoracle import Oracle

    from inductioneq_amd.program import Program
    from test_gpu_parity import _aos, _relerr, _scal

    lo, hi = (0.0, 2 * np.pi) if per else (-1.0, 1.0)
    cfg = ProgramConfig(real=real, opset=ops, nx=n[0], ny=n[1], nz=n[2], xmin=lo, xmax=hi, ymin=lo, ymax=hi, zmin=lo,
                        zmax=hi, periodic=per, testcase="hall_periodic" if per else "rotation_2D", w_size=64,
                        laplace="WIDE_STENCIL_LNS")
    prog, orc = Program(cfg), Oracle(cfg)
    g = tuple(max(1, v - 1 - k) for k, v in enumerate(n)) if part else n
    rng = np.random.default_rng(5)
    hb, hp = _aos(cfg, rng.standard_normal((cfg.num_nodes, 3))), _scal(cfg, rng.standard_normal(cfg.num_nodes))
    db, dp = prog.upload_real4(hb), prog.upload_real(hp)
    tol = 1e-12 if real == "double" else 2e-5
    hs, ds = _scal(cfg, np.full(cfg.num_nodes, 3.0)), prog.scalar(3.0)
    orc.run("calc_div", [hb, hs], g=g)
    prog.run("calc_div", [db, ds], g=g)
    assert _relerr(prog.download_real(ds)[: cfg.num_nodes], hs[: cfg.num_nodes]) <= tol
    for name, ha, da in (("calc_curl", hb, db), ("calc_grad", hp, dp)):
        hv = _aos(cfg, np.full((cfg.num_nodes, 3), 3.0))
        dv = prog.upload_real4(hv)
        orc.run(name, [ha, hv], g=g)
        prog.run(name, [da, dv], g=g)
        assert _relerr(prog.download_real4(dv)[: cfg.num_nodes, :3], hv[: cfg.num_nodes, :3]) <= tol, name
    if not per:
        orc.run("projector_divcleaning", [hb, hp], g=g)
        prog.run("projector_divcleaning", [db, dp], g=g)
        torch.cuda.synchronize()
        assert _relerr(prog.download_real4(db)[: cfg.num_nodes, :3], hb[: cfg.num_nodes, :3]) <= tol
