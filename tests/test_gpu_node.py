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
