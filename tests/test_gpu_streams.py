"""One program driven on several streams in turn: the buffers it keeps are handed over between its calls."""
import numpy as np
import pytest

from inductioneq_amd.problems import hall_dt, random_modes_field

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ops,n,real", [("6thOrder", (70, 66, 64), "double"), ("4thOrder", (64, 48, 50), "float")])
def test_fused_2n_steps_on_two_streams(ops, n, real):
    """Two solves of one program in turn on two streams, without a wait between the calls, equal the same solves one
    after the other bit for bit: the 2N schemes' second b1 belongs to the program."""
    import torch
    from test_gpu_fused import _device_args, _periodic_cfg

    from inductioneq_amd.program import Program

    u, rho = (0.3, -0.2, 0.1), 1.25
    cfg = _periodic_cfg(n, real, ops, True, "HIGH_ORDER", u, ho_factor=0.5)
    B0 = random_modes_field(n, seed=4, kmax=2, amp=0.3)
    cfg.dt = hall_dt(B0, (cfg.dx, cfg.dy, cfg.dz), 6, c_hall=0.8, cfl=0.3)
    prog = Program(cfg)

    def solve(streams, scale):
        regs = [_device_args(prog, np.asarray(B0) * c, 2, u, rho) for c in scale]
        torch.cuda.synchronize()
        for _ in range(6):
            for s, a in zip(streams, regs):
                with torch.cuda.stream(s):
                    prog.use_current_stream()
                    prog.step("CarpenterKennedy2N54", 3, a, uniform=(*u, rho))
                    assert prog.last_step_fused
        torch.cuda.synchronize()
        return [a[0].clone() for a in regs]

    s1, s2 = torch.cuda.Stream(), torch.cuda.Stream()
    both = solve((s1, s2), (1.0, 0.5))
    assert bool(torch.isfinite(both[0]).all())
    assert torch.equal(both[0], solve((s1,), (1.0,))[0])
    assert torch.equal(both[1], solve((s1,), (0.5,))[0])


def test_first_2n_list_while_another_stream_is_captured():
    """A program's first 2N list beside a capture on another stream: the capture ends whole, its replays give the
    eager result, and the list's result is that of a list without a capture."""
    import torch

    from inductioneq_amd.program import Program
    from inductioneq_amd.schedules import rk_schedule
    from test_gpu_node import _stage_case
    from test_gpu_tiled import _aos

    cfg, B, U = _stage_case("4thOrder", (40, 30, 20), False, True, None, "double")
    cfg.dt = 1e-5
    names, nf = rk_schedule("CarpenterKennedy2N54", True, True)
    side, work = torch.cuda.Stream(), torch.cuda.Stream()

    def solve(capture):
        prog = Program(cfg)
        a = [prog.upload_real4(_aos(cfg, B))] + [prog.vector() for _ in range(nf)]
        a += [prog.upload_real4(_aos(cfg, U)), prog.scalar(1.0), prog.time_buffer()]
        x, y, g = torch.ones(1000, device="cuda"), torch.zeros(1000, device="cuda"), torch.cuda.CUDAGraph()
        torch.cuda.synchronize()
        with torch.cuda.stream(work):
            prog.use_current_stream()
        if capture:
            with torch.cuda.graph(g, stream=side):
                torch.add(x, 2.0, out=y)
                prog.run(names, a)
        else:
            prog.run(names, a)
        torch.cuda.synchronize()
        for k in range(3 if capture else 0):
            x.fill_(float(k))
            g.replay()
            torch.cuda.synchronize()
            assert bool((y == k + 2.0).all())
        return a[0].clone()

    assert torch.equal(solve(True), solve(False))


def test_2n_steps_captured_between_eager_ones():
    """2N steps on the default stream, then captured on another and replayed with eager steps on the first between the
    replays: every replay gives what the same step gives eagerly."""
    import torch
    from test_gpu_fused import _device_args, _periodic_cfg

    from inductioneq_amd.program import Program

    u, rho = (0.3, -0.2, 0.1), 1.25
    cfg = _periodic_cfg((40, 33, 26), "double", "6thOrder", True, "HIGH_ORDER", u, ho_factor=0.5)
    B0 = np.asarray(random_modes_field((40, 33, 26), seed=4, kmax=2, amp=0.3))
    cfg.dt = hall_dt(B0, (cfg.dx, cfg.dy, cfg.dz), 6, c_hall=0.8, cfl=0.3)
    prog = Program(cfg)
    step = lambda a: prog.step("CarpenterKennedy2N54", 3, a, uniform=(*u, rho))
    inputs = [_device_args(prog, B0 * c, 2, u, rho)[0].clone() for c in (1.0, 0.7, 0.4)]
    want = []
    prog.use_current_stream()
    for b in inputs:
        a = _device_args(prog, B0, 2, u, rho)
        a[0].copy_(b)
        step(a)
        torch.cuda.synchronize()
        want.append(a[0].clone())
    eager, captured, g = _device_args(prog, B0, 2, u, rho), _device_args(prog, B0, 2, u, rho), torch.cuda.CUDAGraph()
    step(eager)
    with torch.cuda.graph(g):
        prog.use_current_stream()
        step(captured)
    prog.use_current_stream()
    for k, b in enumerate(inputs):
        captured[0].copy_(b)
        captured[1].zero_()
        captured[5].zero_()
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(captured[0], want[k]), k
        eager[0].copy_(inputs[1])
        step(eager)
        torch.cuda.synchronize()
        assert torch.equal(eager[0], want[1]), k
