"""Host code of the library around its launches (error paths, launch shapes, ordering), with a recording HIP runtime
in place of the real one: no GPU, no kernel runs."""
import pytest
from hostrun import build_hip, hostrun


@pytest.fixture(scope="module")
def hip(tmp_path_factory):
    return build_hip(tmp_path_factory.mktemp("hip"))


@pytest.mark.parametrize("nth", [4, 5])
@pytest.mark.parametrize("zc", [None, "8"])
def test_refused_cg_launch_fails_the_call(hip, nth, zc):
    """A Laplacian (the call's 4th launch) or an update (5th) that cannot be launched: an error, as for the launches
    before and after the iterations, and no solution reported."""
    hostrun(hip, """
        h = build(opset="4thOrder", nx=20, ny=20, nz=20, laplace="WIDE_STENCIL_DIRICHLET")
        b, phi = ctypes.create_string_buffer(3 * 8064 * 8), ctypes.create_string_buffer(8064 * 8)
        call = lambda: lib.ieq_clean_div_cg(h, ctypes.addressof(b), ctypes.addressof(phi), 1e-9, 0.0, 20, ctypes.byref(_capi.CgResult()))
        assert call() == 0
        names = [l[1] for l in log("launch")]
        assert "k_cg_lap" in names[3] and "k_cg_update" in names[4], names
        for n in (%d, len(names), 1):
            fail("hipLaunchKernel", n)
            assert call() != 0, n
            assert H.host_hip_last() == 0  # and nothing is left for the next call to trip over
        assert call() == 0
    """ % nth, **({"IEQ_LAP_ZC": zc} if zc else {}))


def test_uniformity_word_is_zeroed_after_a_failed_attempt(hip):
    """ieq_step's check compares its number with a device word that starts at 0; a word whose zeroing failed would
    let a field that varies pass as uniform, so the next call makes and zeroes another."""
    hostrun(hip, """
        h = build(opset="4thOrder", nx=12, ny=12, nz=12, periodic=True, testcase="uniform_flow")
        args = far(7)
        step = lambda: lib.ieq_step(h, b"SSPRK33", 1, 0, (P * 7)(*args), 7, None)
        fail("hipMemsetAsync")
        assert step() != 0
        word = log("malloc")[0]
        assert word[2] == "8" and ["free", word[1]] in log("free")
        H.host_hip_clear()
        assert step() == 0, lib.ieq_last_error(h)
        kinds = [(l[0], l[2] if l[0] != "launch" else l[1]) for l in log("malloc", "memset", "launch")]
        assert kinds[0] == ("malloc", "8") and kinds[1] == ("memset", "8") and "k_uniform_check" in kinds[2][1], kinds
    """)


@pytest.mark.parametrize("n", [(1024, 1024, 1024), (1030, 1021, 2100)])
def test_stage_kernels_launch_on_grids_of_2_to_the_30_nodes(hip, n):
    """A list of the stage kernels on more nodes than one launch of four threads a node can take: no launch is
    refused, and the blocks of each kernel, of 64 or 256 nodes, are those of every plane."""
    hostrun(hip, """
        n = %r
        h = build(real="float", opset="4thOrder", nx=n[0], ny=n[1], nz=n[2], hall=True, testcase="hall_periodic")
        names = ["calc_curlB_rho_2_3args", "calc_u_3_args", "SSPRK33_2b"]
        for k in names + [names]:
            H.host_hip_clear()
            assert run(h, k, far(7), n) == 0, lib.ieq_last_error(h)
            assert not log("refused")
            blocks = {}
            for l in log("launch"):
                if "node" in l[1]:
                    assert l[3:5] == ["1", "1"] and l[5] == "256"
                    blocks[l[1]] = blocks.get(l[1], 0) + int(l[2])
            assert blocks
            for name, v in blocks.items():
                run_ = 256 if "flat" in name else 64
                assert v == (n[0] * n[1] + run_ - 1) // run_ * n[2], blocks
    """ % (n,))


@pytest.mark.parametrize("g", [(0, 12, 12), (12, 0, 12), (12, 12, 0)])
def test_empty_ndrange_is_refused(hip, g):
    """Every kernel over nodes refuses an NDRange without work-items, and a stage time that a time kernel of the
    list set before the refused kernel is stored all the same."""
    hostrun(hip, """
        g = %r
        h = build(opset="4thOrder", nx=12, ny=12, nz=12, hall=True, testcase="hall_periodic", laplace="WIDE_STENCIL_LNS")
        two, seven = far(2), far(7)
        for name, args in [("calc_div", two), ("calc_curl", two), ("calc_grad", two), ("calc_div_divcleaning", two),
                           ("calc_laplace_divcleaning", two), ("projector_divcleaning", two),
                           ("calc_curlB_rho_1_3args", seven), ("calc_u_3_args", seven), ("SSPRK33_2b", seven)]:
            H.host_hip_clear()
            assert run(h, name, args, g) == _capi.IEQ_ERR_HIP, name
            assert not log("launch") and H.host_hip_last() == 0, name
        for name in ("calc_u_3_args", "SSPRK33_2b"):
            H.host_hip_clear()
            assert run(h, ["SSPRK33_2a", name], seven, g) == _capi.IEQ_ERR_HIP
            assert ["k_time" in l[1] for l in log("launch")] == [True]
    """ % (g,))


@pytest.mark.parametrize("nth,copied", [(1, False), (2, True), (3, False), (4, True)])
def test_list_that_fails_at_a_fused_stage_leaves_the_last_b1(hip, nth, copied):
    """A 2N list whose nth stage is refused: after an odd number of stages b1 lives in the second copy and is copied
    back, after an even number it is in the caller's field and stays as it is."""
    hostrun(hip, """
        h = build(opset="4thOrder", nx=12, ny=10, nz=9)
        names, nf = rk_schedule("CarpenterKennedy2N54", False, False)
        n = 3 * 1088
        bufs = [ctypes.create_string_buffer(bytes([k + 1]) * (8 * n), 8 * n) for k in range(nf + 4)]
        args = [ctypes.addressof(b) for b in bufs]
        assert run(h, names * 2, args, (12, 10, 9)) == 0
        stages = [k for k, l in enumerate(log("launch")) if "k_node_stage" in l[1]]
        H.host_hip_clear()
        fail("hipLaunchKernel", stages[%d - 1] + 1)
        assert run(h, names * 2, args, (12, 10, 9)) == _capi.IEQ_ERR_HIP
        back = [l for l in log("memcpy") if int(l[1], 16) == args[0]]
        assert len(back) == %d, log()
    """ % (nth, copied))


def test_b1_copied_back_after_an_error_keeps_what_follows_its_nodes(hip):
    hostrun(hip, """
        h = build(opset="4thOrder", nx=12, ny=10, nz=9)  # 1080 nodes, components 1088 apart
        names, nf = rk_schedule("CarpenterKennedy2N54", False, False)
        bufs = [(ctypes.c_double * (3 * 1088))(*([7.0] * (3 * 1088))) for k in range(nf + 4)]
        args = [ctypes.addressof(b) for b in bufs]
        fail("hipLaunchKernel", 2)
        assert run(h, names * 2, args, (12, 10, 9)) == _capi.IEQ_ERR_HIP
        assert any(v != 7.0 for v in bufs[0][:1080])  # the second copy's bytes: the test runtime computes nothing
        for c in range(3):
            assert bufs[0][c * 1088 + 1080 : (c + 1) * 1088] == [7.0] * 8, c
    """)


@pytest.mark.parametrize("call", ["step", "list"])
def test_program_buffers_are_handed_from_stream_to_stream(hip, call):
    """2N stages keep a second b1 with the program (fused steps and lists alike).  Leaving a stream marks the end of
    its use there, the next call that uses it on another stream waits for the mark before it launches, and nothing
    is marked or waited for while the stream stays the same or is being captured."""
    hostrun(hip, """
        fused = %r == "step"
        h = build(opset="4thOrder", nx=16, ny=12, nz=12, periodic=fused, testcase="uniform_flow")
        names, nf = rk_schedule("CarpenterKennedy2N54", False, False)
        u3 = (ctypes.c_double * 3)(0.1, 0.0, 0.2)
        bufs = [ctypes.create_string_buffer(3 * 2304 * 8) for _ in range(6)]

        def go(stream, shared=True):
            H.host_hip_clear()
            assert lib.ieq_set_stream(h, P(stream)) == 0
            a = [ctypes.addressof(b) for b in bufs]
            if not shared:
                assert run(h, "CarpenterKennedy2N54_1a", a, (16, 12, 12)) == 0
            elif fused:
                assert lib.ieq_step_uniform(h, b"CarpenterKennedy2N54", 1, u3, 1.0, (P * 6)(*a), 6, None) == 0
            else:
                assert run(h, names, a, (16, 12, 12)) == 0
            lines = [(l[0], l[1] if l[0] == "wait" else l[2]) for l in log("wait", "record")]
            n = [l[0] for l in log("wait", "record", "launch")].index("launch")
            assert n == len(lines), "marks and waits come before the launches"
            return lines

        A, B, C, D = 0x1000, 0x2000, 0x3000, 0x4000
        assert go(A) == go(A) == []
        assert go(B) == [("record", hex(A)), ("wait", hex(B))]
        assert go(B) == []
        assert go(C, shared=False) == [("record", hex(B))]
        assert go(A) == [("wait", hex(A))]  # B's mark: C has not used the buffer
        H.host_hip_capture(P(D))
        assert go(D) == [("record", hex(A))]
        H.host_hip_capture(P(-1))
        assert go(D) == [("wait", hex(D))]
        assert go(A) == [("record", hex(D)), ("wait", hex(A))]
        assert go(A) == []
    """ % call)


def test_the_lists_second_b1_is_allocated_in_relaxed_capture_mode(hip):
    """A 2N list launches kernels and allocates its second b1 once; the allocation must not end a capture that another
    stream or thread has begun, which the mode of the calling thread decides.  The mode is as before afterwards."""
    hostrun(hip, """
        h = build(opset="4thOrder", nx=12, ny=10, nz=9)
        names, nf = rk_schedule("CarpenterKennedy2N54", False, False)
        assert run(h, names, far(6), (12, 10, 9)) == 0
        assert [l[-1] for l in log("malloc")] == ["relaxed"]
        mode = ctypes.c_int(2)
        H.hipThreadExchangeStreamCaptureMode(ctypes.byref(mode))
        assert mode.value == 0
    """)


@pytest.mark.parametrize("integrator,field,other", [("SSPRK33", 4, 3), ("SSPRK33", 4, 0), ("SSPRK33", 4, 5),
                                                    ("CarpenterKennedy2N54", 0, 3), ("CarpenterKennedy2N54", 1, 2)])
@pytest.mark.parametrize("inside", [0, 4096])
def test_lists_on_arguments_that_share_memory_run_one_by_one(hip, integrator, field, other, inside):
    """With two arguments in one buffer, or one that begins inside another, the kernels' order is part of the result:
    a list launches exactly what its kernels launch one by one."""
    hostrun(hip, """
        h = build(opset="4thOrder", nx=12, ny=10, nz=9, hall=True, testcase="hall_periodic")
        names, nf = rk_schedule(%r, True, True)

        def kernels(args, names):
            H.host_hip_clear()
            for k in names:
                assert run(h, k, args, (12, 10, 9)) == 0
            return [l[1] for l in log("launch")]

        args = far(nf + 4)
        whole = names * 2
        assert len(kernels(args, [whole])) < len(kernels(args, whole))
        args[%d] = args[%d] + %d
        assert kernels(args, [whole]) == kernels(args, whole)
    """ % (integrator, field, other, inside))


def test_unused_arguments_may_share_memory(hip):
    """Without the Hall term nothing uses curlB_rho and rho: what is passed for them does not keep launches apart."""
    hostrun(hip, """
        h = build(opset="4thOrder", nx=12, ny=10, nz=9)
        names, nf = rk_schedule("CarpenterKennedy2N54", False, False)
        args = far(6)
        n = []
        for a in (args, args[:2] + [args[3], args[3], args[3], args[5]]):
            H.host_hip_clear()
            assert run(h, names * 2, a, (12, 10, 9)) == 0
            n.append(len(log("launch")))
        assert n[0] == n[1]
    """)


@pytest.mark.parametrize("real,below,above", [("float", (32767, 32768, 9), (32768, 32768, 9)), ("double", (8191, 65536, 9), (8192, 65536, 9))])
def test_planes_of_4_gib_take_64_bit_offsets(hip, real, below, above):
    """In-plane byte offsets of 32 bits wrap where a component's plane takes 4 GiB: kernels with 64-bit offsets there."""
    hostrun(hip, """
        names = {}
        for n in (%r, %r, (300, 300, 9)):
            h = build(real=%r, opset="4thOrder", nx=n[0], ny=n[1], nz=n[2], hall=True, testcase="hall_periodic",
                      laplace="WIDE_STENCIL_LNS")
            H.host_hip_clear()
            for k in ("calc_curlB_rho_2_3args", "SSPRK33_2b"):
                assert run(h, k, far(7), n) == 0, lib.ieq_last_error(h)
            for k in ("calc_div", "calc_curl", "calc_grad", "projector_divcleaning"):
                assert run(h, k, far(2), n) == 0, lib.ieq_last_error(h)
            names[n] = {l[1] for l in log("launch")}
        below, above, small = names.values()
        assert below == small and not above & small, names
    """ % (below, above, real))


@pytest.mark.parametrize("n", [(65600, 65600, 2), (1024, 1024, 1024), (100, 90, 80)])
def test_column_kernels_launch_shape(hip, n):
    """Runs of 256 nodes of a plane times planes or z-chunks, in rows that HIP takes (4.3e9 nodes a plane: 1.7e7
    runs)."""
    hostrun(hip, """
        n = %r
        h = build(real="float", opset="4thOrder", nx=n[0], ny=n[1], nz=n[2], testcase="rotation_2D", laplace="WIDE_STENCIL_LNS")
        for k in ("calc_div", "calc_grad", "projector_divcleaning"):
            H.host_hip_clear()
            assert run(h, k, far(2), n) == 0, lib.ieq_last_error(h)
            (l,) = log("launch", "refused")
            x, y, z, threads = [int(v) for v in l[2:6]]
            runs = (n[0] * n[1] + 255) // 256
            zc = max(1, min(16, runs * n[2] // 4096)) if "column" in l[1] else 1
            assert ("column" in l[1]) == (n == (1024, 1024, 1024))
            need = runs * -(-n[2] // zc)
            assert z == 1 and threads == 256 and need <= x * y < need + x, (x, y, need)
    """ % (n,))


@pytest.mark.parametrize("w_size,bricks", [(64, True), (1 << 28, True), (1 << 29, False)])
def test_bricks_only_where_their_offsets_fit(hip, w_size, bricks):
    """A brick reaches the second component by a 32-bit byte offset from the first: components of more than 2 GiB (here
    by the padding to W_SIZE) keep the z-march."""
    hostrun(hip, """
        h = build(real="double", opset="6thOrder", nx=40, ny=40, nz=40, periodic=True, testcase="uniform_flow", w_size=%d)
        assert lib.ieq_step_uniform(h, b"SSPRK33", 1, (ctypes.c_double * 3)(0.1, 0.2, 0.3), 1.0, (P * 7)(*far(7)), 7, None) == 0
        stages = [l[1] for l in log("launch") if "stage" in l[1]]
        assert len(stages) == 3 and all(("brick" in k) == bool(%d) for k in stages), stages
        a = P()
        assert lib.ieq_adjoint_create(ctypes.byref(a), h, 2, 1) == 0, lib.ieq_last_error(h)
        H.host_hip_clear()
        c = ctypes.c_double(0.0)
        assert lib.ieq_adjoint_forward(a, P(1 << 42), P(2 << 42), 1.0, (ctypes.c_double * 3)(0.1, 0.2, 0.3), ctypes.byref(c)) == 0, lib.ieq_last_error(h)
        stages = [l[1] for l in log("launch") if "stage" in l[1]]
        assert stages and all(("brick" in k) == bool(%d) for k in stages), stages
    """ % (w_size, bricks, bricks))


def test_fused_2n_register_is_cleared_by_a_kernel(hip):
    """The register is allocated by the first 2N step and cleared before use: by a kernel, as a memset in a captured
    graph is not to be had, and again by the first call that is not captured."""
    hostrun(hip, """
        h = build(opset="4thOrder", nx=16, ny=12, nz=12, periodic=True, testcase="uniform_flow")
        bufs = [ctypes.create_string_buffer(3 * 2304 * 8) for _ in range(6)]
        lib.ieq_set_stream(h, P(0x1000))

        def step():
            H.host_hip_clear()
            assert lib.ieq_step_uniform(h, b"CarpenterKennedy2N54", 1, (ctypes.c_double * 3)(0.1, 0.0, 0.2), 1.0,
                                        (P * 6)(*[ctypes.addressof(b) for b in bufs]), 6, None) == 0
            assert not log("memset")
            return ["k_zero" in l[1] for l in log("launch")]

        H.host_hip_capture(P(0x1000))
        assert step()[0] and step()[0]
        H.host_hip_capture(P(-1))
        assert step()[0] and not any(step())
    """)


def test_adjoint_buffers_are_handed_from_stream_to_stream(hip):
    """A forward solve on one stream and the backward on another: the second waits for the first's snapshots."""
    hostrun(hip, """
        h, a, c = build(opset="4thOrder", nx=16, ny=12, nz=12, periodic=True, hall=True, testcase="uniform_flow"), P(), ctypes.c_double(1.0)
        bufs = [ctypes.create_string_buffer(3 * 2304 * 8) for _ in range(4)]
        b = [ctypes.addressof(x) for x in bufs]
        assert lib.ieq_set_stream(h, P(0x1000)) == 0
        assert lib.ieq_adjoint_create(ctypes.byref(a), h, 3, 3) == 0, lib.ieq_last_error(h)
        assert lib.ieq_adjoint_forward(a, P(b[0]), P(b[1]), 1.0, (ctypes.c_double * 3)(0.1, 0.2, 0.3), None) == 0, lib.ieq_last_error(h)
        H.host_hip_clear()
        assert lib.ieq_set_stream(h, P(0x2000)) == 0
        assert lib.ieq_adjoint_backward(a, P(b[2]), P(b[3]), (ctypes.c_double * 4)(), None) == 0, lib.ieq_last_error(h)
        kinds = [(l[0], l[1] if l[0] == "wait" else l[-1]) for l in log("wait", "record", "launch")]
        assert kinds[:2] == [("record", "0x1000"), ("wait", "0x2000")], kinds[:4]
        assert {k for k in kinds[2:]} <= {("record", "0x2000"), ("launch", "0x2000")}, kinds[:4]
    """)
