"""Which launch a call takes, and what it may ask of the device around it:
requested launch shapes are the ones that run, default ones take no memory
that a caller cannot spare, and sizes past 32-bit launch or index limits give
the results of the smaller ones."""
import ctypes
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

GLOBAL, THREAD_LOCAL, RELAXED = 0, 1, 2  # hipStreamCaptureMode


@pytest.fixture(scope="module")
def lib():
    from numbacs_amd import _lib

    _lib.torch()
    return _lib


@pytest.fixture
def configs(lib):
    from numbacs_amd import autotune

    saved = {(k, p): autotune.get(k, p) for k in range(4) for p in (0, 1)}
    orders = {p: autotune.get_order(p) for p in (0, 1)}
    yield autotune
    for (k, p), cfg in saved.items():
        autotune.set_config(k, p, cfg)
    for p, o in orders.items():
        autotune.set_order(p, o)


class Capture:
    """Capture of one stream of its own by the HIP runtime the library uses."""

    def __init__(self, lib, mode):
        self.hip = ctypes.CDLL(lib.LIB_PATH)
        self.stream = lib.torch().cuda.Stream()
        self.mode = mode

    def __enter__(self):
        lib_stream = ctypes.c_void_p(self.stream.cuda_stream)
        assert self.hip.hipStreamBeginCapture(lib_stream, self.mode) == 0
        return self

    def __exit__(self, *exc):
        graph, count = ctypes.c_void_p(), ctypes.c_size_t()
        self.status = self.hip.hipStreamEndCapture(ctypes.c_void_p(self.stream.cuda_stream),
                                                   ctypes.byref(graph))
        self.nodes = 0
        if self.status == 0 and graph.value:
            assert self.hip.hipGraphGetNodes(graph, None, ctypes.byref(count)) == 0
            self.nodes = count.value
            self.hip.hipGraphDestroy(graph)


def kernels_of(lib, call):
    """Number of kernels that call() enqueues on the current stream, by a
    capture; called once before it, so that its workspaces are there."""
    capture = Capture(lib, RELAXED)
    with lib.torch().cuda.stream(capture.stream):
        call()
        capture.stream.synchronize()
        with capture:
            call()
    assert capture.status == 0
    return capture.nodes


def small_spline(extrap_mode="constant"):
    from numbacs_amd.flows import get_flow_2D

    n = (8, 20, 18)
    C = np.random.default_rng(1).standard_normal((2,) + tuple(m + 2 for m in n))
    return get_flow_2D(tuple((0.0, 1.0, m) for m in n), C[0], C[1], extrap_mode=extrap_mode)


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("cfg", [(4, 64, 4), (2, 64, 4), (4, 128, 2), (1, 256, 8)])
@pytest.mark.parametrize("shape", [(9, 33), (801, 501)])
def test_requested_queue_is_what_runs(lib, configs, precision, cfg, shape):
    """A queue launch is two kernels (the ring's start, the persistent grid),
    also for fewer tiles than the grid has wavefronts and for more than 16
    rounds of them; the map equals the grid launch's at the same lanes."""
    from numbacs_amd.integration import flowmap_grid_2d_device

    f = small_spline("nearest")
    xd, yd = (lib.to_dev(np.linspace(0.0, 1.0, n)) for n in shape)
    out = lib.empty(shape + (2,))
    call = lambda: flowmap_grid_2d_device(f, 0.0, 0.5, xd, yd, [1.0], precision=precision, out=out)
    configs.set_config(2, precision, cfg)
    assert kernels_of(lib, call) == 2
    call()
    got = lib.to_host(out)
    configs.set_config(2, precision, cfg[:2] + (0,))
    call()
    assert np.array_equal(got, lib.to_host(out))


@pytest.mark.parametrize("kind,precision,n", [(0, 0, 90000), (0, 0, 150000), (0, 1, 150000),
                                              (0, 1, 300000), (1, 0, 90000), (1, 1, 90000)])
def test_requested_queue_batch(lib, configs, kind, precision, n):
    """A requested queue holds the states of the lane groups that run: analytic
    flows on both sides of the double gyre's pair limits."""
    from numbacs_amd.batch import FTLEBatch
    from numbacs_amd.flows import get_predefined_flow

    flow, p, dom = get_predefined_flow(("double_gyre", "bickley_jet")[kind])
    x, y = np.linspace(*dom[0], n // 100), np.linspace(*dom[1], 100)
    b = FTLEBatch(flow, [dict(t0=0.0, T=0.5, x=x, y=y)], p, precision=("fp64", "fp32")[precision],
                  ftle=False)
    configs.set_config(kind, precision, (1, 64, 4))
    assert kernels_of(lib, b.run) == 2
    b.run()
    got = b.results()[0]["flowmap"]
    configs.set_config(kind, precision, (1, 64, 0))
    assert kernels_of(lib, b.run) == 1
    b.run()
    assert np.array_equal(got, b.results()[0]["flowmap"])
    b.close()


@pytest.mark.parametrize("precision", [0, 1])
def test_default_bickley_batch_takes_no_memory(lib, precision):
    """A batch keeps no solver states unless its launch shape was set to the
    queue: 1.4 M particles would hold 150 MB and more.  Its maps equal the
    single grids'."""
    from numbacs_amd.batch import FTLEBatch
    from numbacs_amd.flows import get_predefined_flow
    from numbacs_amd.integration import flowmap_grid_2d_device

    torch = lib.torch()
    flow, p, dom = get_predefined_flow("bickley_jet")
    x, y = np.linspace(*dom[0], 1401), np.linspace(*dom[1], 1001)
    b = FTLEBatch(flow, [dict(t0=0.0, T=0.5, x=x, y=y)], p, precision=("fp64", "fp32")[precision],
                  ftle=False)
    torch.cuda.synchronize()
    before = torch.cuda.mem_get_info()[0]
    b.run()
    torch.cuda.synchronize()
    assert before - torch.cuda.mem_get_info()[0] < 64 << 20
    got = b.results()[0]["flowmap"]
    want = flowmap_grid_2d_device(flow, 0.0, 0.5, lib.to_dev(x), lib.to_dev(y), p,
                                  precision=precision)
    assert np.array_equal(got, lib.to_host(want))
    b.close()


@pytest.mark.parametrize("precision", [0, 1])
def test_default_bickley_map_of_long_solves(lib, precision):
    """A wavefront waits in the queue for a bounded time, so a map that allows
    more steps than the entry points' default takes the grid launch, which holds
    no states; the queue's stream holds 112 bytes a slot."""
    from numbacs_amd.flows import get_predefined_flow
    from numbacs_amd.integration import flowmap_grid_2d_device

    torch = lib.torch()
    flow, p, dom = get_predefined_flow("bickley_jet")
    hip, stream = ctypes.CDLL(lib.LIB_PATH), ctypes.c_void_p()
    assert hip.hipStreamCreateWithFlags(ctypes.byref(stream), 1) == 0  # without a workspace yet
    xd, yd = (lib.to_dev(np.linspace(*d, n)) for d, n in zip(dom, (1401, 1001)))
    out = [lib.empty((1401, 1001, 2)) for _ in range(2)]
    held = []
    with torch.cuda.stream(torch.cuda.ExternalStream(stream.value)):
        for dst, steps in zip(out, (100001, 100000)):
            torch.cuda.synchronize()
            before = torch.cuda.mem_get_info()[0]
            flowmap_grid_2d_device(flow, 0.0, 0.5, xd, yd, p, max_steps=steps, precision=precision,
                                   out=dst)
            torch.cuda.synchronize()
            held.append(before - torch.cuda.mem_get_info()[0])
    assert held[0] < 64 << 20 < held[1]
    assert torch.equal(*out)


def test_default_bickley_map_during_another_capture(lib):
    """A default flow map on one stream while another is being captured, in
    the mode that refuses allocations meanwhile and is invalidated by them: the
    map runs and the capture goes on."""
    from numbacs_amd.flows import get_predefined_flow

    torch = lib.torch()
    flow, p, dom = get_predefined_flow("bickley_jet")
    nx, ny = 711, 333
    xd, yd = lib.to_dev(np.linspace(*dom[0], nx)), lib.to_dev(np.linspace(*dom[1], ny))
    out, want = lib.empty((nx, ny, 2)), lib.empty((nx, ny, 2))
    p = np.ascontiguousarray(p, dtype=np.float64)
    hip = ctypes.CDLL(lib.LIB_PATH)

    def run(dst, stream):
        return lib.load().nbx_flowmap_grid_2d(
            flow.handle, 0.0, 2.0, lib.ptr(xd), nx, lib.ptr(yd), ny, p.ctypes.data, p.size, 1e-6,
            1e-8, None, 100000, 0, lib.ptr(dst), None, None, stream)

    torch.cuda.synchronize()
    other = ctypes.c_void_p()  # a stream that has no workspace yet
    assert hip.hipStreamCreateWithFlags(ctypes.byref(other), 1) == 0
    with Capture(lib, GLOBAL) as capture:
        rc = run(out, other.value)
    assert rc == 0, lib.load().nbx_last_error()
    assert capture.status == 0
    assert hip.hipStreamSynchronize(other) == 0
    assert run(want, lib.stream_ptr()) == 0
    assert torch.equal(out, want)


def test_captured_queue_keeps_its_workspace(lib, configs):
    """A requested queue captured on a stream, then a larger map of the default
    configuration on the same stream: the graph's workspace is not grown away
    from under it.  Replayed several times, with eager maps between."""
    from numbacs_amd.flows import get_predefined_flow
    from numbacs_amd.integration import flowmap_grid_2d_device

    torch = lib.torch()
    flow, p, dom = get_predefined_flow("bickley_jet")

    def axes(*n):
        return [lib.to_dev(np.linspace(*d, m)) for d, m in zip(dom, n)]

    small, large = axes(301, 111), axes(801, 401)
    out, eager, big = (lib.empty(s + (2,)) for s in ((301, 111), (301, 111), (801, 401)))
    stream, graph = torch.cuda.Stream(), torch.cuda.CUDAGraph()
    default = configs.get(1, 0)
    with torch.cuda.stream(stream):
        configs.set_config(1, 0, (1, 64, 1))
        flowmap_grid_2d_device(flow, 0.0, 5.0, *small, p, out=eager)
        stream.synchronize()
        with torch.cuda.graph(graph, stream=stream):
            flowmap_grid_2d_device(flow, 0.0, 5.0, *small, p, out=out)
        configs.set_config(1, 0, default)
        for _ in range(3):
            flowmap_grid_2d_device(flow, 0.0, 5.0, *large, p, out=big)
            out.zero_()
            graph.replay()
            stream.synchronize()
            assert torch.equal(out, eager)


def constant_flow(n, value):
    from numbacs_amd.flows import get_flow_2D

    torch = __import__("torch")
    C = torch.full(tuple(m + 2 for m in n), value, dtype=torch.float64, device="cuda")
    return get_flow_2D(tuple((0.0, 1.0, m) for m in n), C, -C)


def test_closed_flows_memory_comes_back(lib):
    """What a closed flow leaves behind while another is open (2 x 71 MB here)
    is given back on request, and by closing the last one; a flow of more than
    256 MiB leaves nothing."""
    from numbacs_amd import flows

    torch = lib.torch()

    def free():
        torch.cuda.synchronize()
        torch.cuda.empty_cache()
        return torch.cuda.mem_get_info()[0]

    n = (64, 256, 256)
    kept = constant_flow((4, 5, 6), 1.0)
    flows.release_memory()
    start = free()
    a = constant_flow(n, 2.0)
    assert start - free() > 128 << 20
    a.close()
    flows.release_memory()
    assert start - free() < 8 << 20
    constant_flow((256, 256, 256), 2.0).close()
    assert start - free() < 8 << 20
    b, c = constant_flow(n, 2.0), constant_flow(n, 3.0)
    b.close()
    c.close()
    kept.close()
    assert start - free() < 8 << 20


def test_closing_waits_for_the_flow_s_work(lib):
    """A flow closed while a map over it runs on a side stream, and a flow of its
    size made at once: the map is the closed flow's."""
    from numbacs_amd.integration import flowmap_grid_2d_device

    torch = lib.torch()
    n, shape = (32, 96, 96), (1200, 900)
    kept = constant_flow((4, 5, 6), 1.0)
    # (0.3 to the right and down: inside the unit box all the way)
    xd, yd = (lib.to_dev(np.linspace(a, a + 0.1, m)) for a, m in zip((0.2, 0.6), shape))
    side, out = torch.cuda.Stream(), lib.empty(shape + (2,))
    want = None
    for turn in range(4):
        a = constant_flow(n, 0.5)
        torch.cuda.synchronize()
        with torch.cuda.stream(side):
            for _ in range(8):  # some milliseconds
                flowmap_grid_2d_device(a, 0.0, 0.6, xd, yd, [1.0], rtol=1e-10, atol=1e-13, out=out)
        a.close()
        b = constant_flow(n, -0.5)
        torch.cuda.synchronize()
        got = lib.to_host(out)
        want = got if want is None else want
        assert np.abs(got[..., 0] - lib.to_host(xd)[:, None] - 0.3).max() < 1e-9
        assert np.array_equal(got, want)
        b.close()
    kept.close()


@pytest.mark.parametrize("mode", [THREAD_LOCAL, RELAXED])
def test_closing_a_flow_during_a_capture(lib, mode):
    """Where frees are allowed -- in another thread than the capture's (batches
    are captured that way), or in the relaxed mode -- a flow may be closed
    while a stream is being captured; the capture goes on."""
    kept, flow = constant_flow((4, 5, 6), 1.0), constant_flow((8, 9, 10), 2.0)
    lib.torch().cuda.synchronize()
    with Capture(lib, mode) as capture:
        if mode == RELAXED:
            flow.close()
        else:
            other = threading.Thread(target=flow.close)
            other.start()
            other.join()
    assert capture.status == 0
    kept.close()


@pytest.mark.parametrize("precision", [0, 1])
def test_spline_arrays_above_2_gib(lib, precision):
    """The 4-lane kernel's 32-bit offsets at the far end of a coefficient array
    of 2.7 GB: a unit-spaced grid's last corner against a flow of that corner's
    coefficients alone.  Cell positions are exact in both, so the bits are
    equal."""
    from numbacs_amd.flows import get_flow_2D
    from numbacs_amd.integration import flowmap_grid_2d_device

    torch = lib.torch()
    n, first = (18, 1022, 8190), (0, 1000, 8160)
    gen = torch.Generator(device="cuda").manual_seed(3)
    C = [torch.zeros(tuple(m + 2 for m in n), dtype=torch.float64, device="cuda")
         for _ in range(2)]
    corner = []
    for c in C:
        part = c[:, first[1]:, first[2]:]
        part.copy_(torch.rand(part.shape, generator=gen, dtype=torch.float64, device="cuda") - 0.5)
        corner.append(part.contiguous())
    big = get_flow_2D(tuple((0.0, m - 1.0, m) for m in n), *C)
    small = get_flow_2D(tuple((float(a), m - 1.0, m - a) for a, m in zip(first, n)), *corner)
    del C, c, part
    xd, yd = (lib.to_dev(np.linspace(a + 6.0, m - 5.0, 37)) for a, m in zip(first[1:], n[1:]))
    got, want = (flowmap_grid_2d_device(f, 13.0, 3.5, xd, yd, [1.0], precision=precision)
                 for f in (big, small))
    assert float((got - torch.stack(torch.meshgrid(xd, yd, indexing="ij"), -1)).abs().max()) > 0.1
    assert torch.equal(got, want)
    big.close()
    small.close()
    torch.cuda.empty_cache()


@pytest.mark.parametrize("shape", [(1, 23170, 23170), (23171, 23171, 1)])
def test_prefilter_of_more_lines_than_one_launch_holds(lib, shape):
    """Axes of one sample with 2^29 lines and more across them (8 threads of the
    line-group kernels each): a coefficient of such an axis equals its sample,
    and along the others the coefficients interpolate it."""
    from numbacs_amd.flows import prefilter3_device

    torch = lib.torch()
    gen = torch.Generator(device="cuda").manual_seed(5)
    U = torch.rand(shape, generator=gen, dtype=torch.float64, device="cuda") - 0.5
    C = prefilter3_device(U)
    one = shape.index(1)
    planes = [C.select(one, k) for k in range(3)]
    assert torch.equal(planes[0], planes[1]) and torch.equal(planes[2], planes[1])
    # (c[i-1] + 4 c[i] + c[i+1]) / 6 along both long axes
    c = planes[1][-4001:, -4001:]
    for axis in (0, 1):
        m = c.shape[axis] - 2
        c = (c.narrow(axis, 0, m) + 4 * c.narrow(axis, 1, m) + c.narrow(axis, 2, m)) / 6
    u = U.select(one, 0)[-c.shape[0]:, -c.shape[1]:]
    # rounding of coefficients up to 9 times the samples, and of the check's sums
    assert float((c - u).abs().max()) < 64 * 2.0 ** -52 * 4.5
    del U, C, planes, c, u
    torch.cuda.empty_cache()


def test_trilinear_map_of_more_threads_than_a_pair_launch_holds(lib):
    """2^31 particles, all but one row masked: one lane each fits a launch, two
    do not."""
    from numbacs_amd.flows import get_flow_linear_2D
    from numbacs_amd.integration import flowmap_grid_2d_device

    torch = lib.torch()
    n = (4, 9, 8)
    U = np.random.default_rng(2).standard_normal((2,) + n)
    f = get_flow_linear_2D(tuple((0.0, 1.0, m) for m in n), U[0], U[1])
    nx, ny, row = 65536, 32768, 40000
    xd, yd = (torch.linspace(0, 1, m, dtype=torch.float64, device="cuda") for m in (nx, ny))
    mask = torch.ones((nx, ny), dtype=torch.uint8, device="cuda")
    mask[row] = 0
    got = flowmap_grid_2d_device(f, 0.1, 0.3, xd, yd, [1.0], maskd=mask)
    want = flowmap_grid_2d_device(f, 0.1, 0.3, xd[row:row + 1].contiguous(), yd, [1.0])
    assert torch.equal(got[row], want[0])
    assert not got[row - 1].any() and not got[row + 1].any() and not got[-1].any()
    del got, mask
    torch.cuda.empty_cache()


def test_output_layer_backward_of_many_narrow_rows(lib):
    """2^26 rows of 8 columns: the deltas of the first and last rows against
    two roundings to bf16 from float64."""
    torch = lib.torch()
    n, width = 1 << 26, 8
    dev = dict(device="cuda")
    gen = torch.Generator(device="cuda").manual_seed(9)
    h = torch.zeros((n, width), dtype=torch.bfloat16, **dev)
    dy = torch.rand((n, 2), generator=gen, **dev)
    pre = torch.rand((n, width), generator=gen, **dev)
    W = torch.rand((width, 2), generator=gen, **dev).to(torch.bfloat16)
    gW, gb = torch.empty((width, 2), **dev), torch.empty(2, **dev)
    da = torch.full((n, width), float("nan"), dtype=torch.bfloat16, **dev)
    lib.check(lib.load().nbx_mlp_out_backward(
        lib.ptr(dy), lib.ptr(h), lib.ptr(pre), n, width, lib.ptr(W), lib.ptr(gW), lib.ptr(gb),
        lib.ptr(da), lib.stream_ptr()))
    assert not da.isnan().any() and not gW.any()
    for part in (slice(0, 999), slice(n - 1001, n)):
        p = pre[part].double()
        t = torch.tanh(0.7978845608028654 * (p + 0.044715 * p ** 3))
        slope = 0.5 * (1 + t) + 0.5 * p * (1 - t ** 2) * 0.7978845608028654 * (
            1 + 3 * 0.044715 * p ** 2)
        dh = dy[part].double() @ W.double().T
        err = (2.0 ** -7 * dh + 2.0 ** -21 * dh) * slope.abs() + 1e-5 * dh
        assert ((da[part].double() - dh * slope).abs() <= err).all()
    del h, dy, pre, da
    torch.cuda.empty_cache()


def test_captured_percentile_keeps_its_workspace(lib):
    """Once any percentile has run on a stream a larger one may be captured there
    without an allocation, and larger ones run after it do not grow the
    workspace away from under the graph.  Replayed several times."""
    torch = lib.torch()
    rng = np.random.default_rng(4)
    few, some, many = (lib.to_dev(rng.standard_normal(n)) for n in (100, 5000, 300001))
    result, eager = lib.empty((2,)), lib.empty((2,))
    hip, handle = ctypes.CDLL(lib.LIB_PATH), ctypes.c_void_p()
    assert hip.hipStreamCreateWithFlags(ctypes.byref(handle), 1) == 0  # without a workspace yet
    torch.cuda.synchronize()
    stream, graph = torch.cuda.ExternalStream(handle.value), torch.cuda.CUDAGraph()

    def percentile(f, out):
        lib.check(lib.load().nbx_percentile(lib.ptr(f), f.numel(), 90.0, lib.ptr(out),
                                            lib.stream_ptr()))

    with torch.cuda.stream(stream):
        percentile(few, eager)
        with torch.cuda.graph(graph, stream=stream):
            percentile(some, result[:1])
            percentile(many, result[1:])
        for _ in range(3):
            percentile(many, eager[1:])
            result.zero_()
            graph.replay()
            percentile(some, eager[:1])
            stream.synchronize()
            assert torch.equal(result, eager)
    for k, f in enumerate((some, many)):
        ref = np.percentile(lib.to_host(f), 90.0)
        assert abs(float(eager[k]) - ref) <= 4 * np.spacing(abs(ref))


def test_percentile_of_more_than_2_to_the_32_values(lib):
    """Counts past 32 bits: whole numbers around zero, of which no digit's bin
    holds as many; those from 2^33 up have more below them."""
    torch = lib.torch()
    n, low = 3 << 31, -(3 << 30)
    f, out = lib.empty((n,)), lib.empty((1,))
    for a in range(0, n, 1 << 30):  # (one call makes fewer than 2^32)
        torch.arange(low + a, low + a + (1 << 30), out=f[a:a + (1 << 30)]).mul_(4)
    for q in (0.0, 25.0, 50.0, 75.0, 99.0, 100.0):
        lib.check(lib.load().nbx_percentile(lib.ptr(f), n, q, lib.ptr(out), lib.stream_ptr()))
        # numpy's virtual index from low; it and the lerp round some 2^33 a few times
        assert abs(float(out[0]) / 4 - (low + (n - 1) * (q / 100.0))) <= 4 * np.spacing(2.0 ** 33)
    del f
    torch.cuda.empty_cache()


def test_releasing_memory_beside_running_maps(lib):
    """A thread that keeps releasing the library's memory while another runs
    default Bickley maps, whose queue's workspace it may take as soon as a launch
    is enqueued: it waits for the work, and the maps stay the same."""
    from numbacs_amd import flows
    from numbacs_amd.integration import flowmap_grid_2d_device

    torch = lib.torch()
    flow, p, dom = flows.get_predefined_flow("bickley_jet")
    xd, yd = (lib.to_dev(np.linspace(*d, n)) for d, n in zip(dom, (801, 401)))
    want = flowmap_grid_2d_device(flow, 0.0, 3.0, xd, yd, p)
    outs = [lib.empty((801, 401, 2)) for _ in range(12)]
    torch.cuda.synchronize()
    done, errors = threading.Event(), []

    def release():
        try:
            while not done.is_set():
                flows.release_memory()
        except Exception as e:  # noqa: BLE001
            errors.append(e)

    thread = threading.Thread(target=release)
    thread.start()
    try:
        with torch.cuda.stream(torch.cuda.Stream()):
            for out in outs:
                flowmap_grid_2d_device(flow, 0.0, 3.0, xd, yd, p, out=out)
        torch.cuda.synchronize()
    finally:
        done.set()
        thread.join()
    assert not errors
    for out in outs:
        assert torch.equal(out, want)
