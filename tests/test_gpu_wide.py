"""Kernels of the reference schedule on a grid whose xy-planes take more than 4 GiB a component (32-bit in-plane byte
offsets wrap) and that has more than 2^30 nodes (a launch with four threads a node is refused).

The fields repeat a 16 x 8 x 2 tile, so that on the periodic grid every tile of a result equals the result on the
periodic grid of one tile: same spacings, and the same operations in the same order per node."""
import pytest

from inductioneq_amd.settings import ProgramConfig

pytestmark = pytest.mark.gpu

TILE = (16, 8, 2)
WIDE = (33008, 33000, 2)  # 1.089e9 nodes a plane: 4.36 GB in FP32


def _cfg(n, diss=None):
    cfg = ProgramConfig(real="float", opset="2ndOrder", nx=n[0], ny=n[1], nz=n[2], xmin=0, xmax=1, ymin=0, ymax=1, zmin=0,
                        zmax=1, dx=0.1, dy=0.2, dz=0.4, dt=1e-2, periodic=True, hall=True, dissipation=diss,
                        testcase="hall_travelling_wave", w_size=64)
    return cfg


def _tile(parts, seed):
    import torch

    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return torch.rand((parts,) + TILE[::-1], generator=g, device="cuda") + 0.5


def _field(prog, n, tile):
    """The tile repeated over the grid of n nodes, in the library's layout."""
    f = prog.vector() if tile.shape[0] == 3 else prog.scalar()
    v = f.view(tile.shape[0], -1)[:, : n[0] * n[1] * n[2]].view(tile.shape[0], n[2], n[1] // 8, 8, n[0] // 16, 16)
    v.copy_(tile[:, :, None, :, None, :].expand_as(v))
    return f


def _same(f, small, n, parts):
    """Every tile of f equals the small grid's result (2e-6 of the largest value: contractions may differ)."""
    v = f.view(parts, -1)[:, : n[0] * n[1] * n[2]].view(parts, n[2], n[1] // 8, 8, n[0] // 16, 16)
    t = small.view(parts, -1)[:, : 16 * 8 * 2].view(parts, 2, 8, 16)
    assert bool((t != 0).any())
    tol = 2e-6 * float(t.abs().max())
    for c in range(parts):
        for z in range(2):
            d = v[c, z].sub(t[c, z][None, :, None, :])
            assert float(d.abs_().max()) <= tol, (c, z)
            del d


@pytest.fixture(autouse=True)
def _room():
    import torch

    if torch.cuda.mem_get_info()[0] < 200 << 30:
        pytest.skip("needs 200 GB of free device memory")
    yield
    torch.cuda.empty_cache()


def test_stage_kernels_on_wide_planes():
    import torch

    from inductioneq_amd.program import Program

    out = {}
    for n in (TILE, WIDE):
        prog = Program(_cfg(n, "HIGH_ORDER"))
        b, u, J = _field(prog, n, _tile(3, 1)), _field(prog, n, _tile(3, 2)), prog.vector()
        rho, res, t = _field(prog, n, _tile(1, 3)), prog.vector(), prog.time_buffer()
        prog.run("calc_curlB_rho_1_3args", [b, b, b, J, u, rho, t])
        prog.run("SSPRK33_2b", [b, b, res, J, u, rho, t])
        torch.cuda.synchronize()
        if n == TILE:
            out = {"J": J, "res": res}
        else:
            del b, u, rho
            _same(J, out["J"], n, 3)
            del J
            _same(res, out["res"], n, 3)


def test_column_kernels_on_wide_planes():
    import torch

    from inductioneq_amd.program import Program

    for name, parts, res in (("calc_div", 3, 1), ("calc_curl", 3, 3), ("calc_grad", 1, 3)):
        small = None
        for n in (TILE, WIDE):
            prog = Program(_cfg(n))
            f = _field(prog, n, _tile(parts, 4))
            out = prog.vector() if res == 3 else prog.scalar()
            prog.run(name, [f, out])
            torch.cuda.synchronize()
            del f
            if n == TILE:
                small = out
            else:
                _same(out, small, n, res)
            del out


@pytest.mark.parametrize("analytic", [0, 1])
def test_diagnostics_on_planes_of_2_to_the_31_nodes(analytic):
    """Sums over the tiles are the tile's times their number (1e-9: up to 4e9 equal terms in another order), the norms
    its square root; the error is against a field of the coordinates, so there the whole is compared with four parts of
    it that do not take the wide kernel: quarters of the y range, each with its coordinates."""
    import math

    import torch

    from inductioneq_amd.program import Program

    n = (46352, 46336, 2)  # 2.148e9 nodes a plane
    tile = _tile(3, 5)

    def diag(n, **kw):
        cfg = _cfg(n)
        for k, v in kw.items():
            setattr(cfg, k, v)
        prog = Program(cfg)
        d = prog.diagnostics(_field(prog, n, tile), 0.0)
        torch.cuda.empty_cache()
        return d

    whole = diag(n)
    if not analytic:
        one, m = diag(TILE), (n[0] // 16) * (n[1] // 8)
        assert abs(whole["energy"] - m * one["energy"]) <= 1e-9 * whole["energy"]
        assert abs(whole["divergence_norm"] - math.sqrt(m) * one["divergence_norm"]) <= 1e-9 * whole["divergence_norm"]
    else:
        half = (n[0], n[1] // 4, n[2])
        parts = [diag(half, ymin=k * half[1] * 0.2)["error_norm"] for k in range(4)]
        want = math.sqrt(sum(p * p for p in parts))
        assert want > 0 and abs(whole["error_norm"] - want) <= 1e-9 * want
