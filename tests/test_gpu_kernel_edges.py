"""Kernels at the sizes where their tiling changes: remainders, group edges,
the smallest sizes and the hand-over between variants."""
import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu


def relerr(a, b):
    return float(np.abs(a - b).max() / max(np.abs(b).max(), 1e-300))


@pytest.mark.parametrize("shape", [
    (1, 1, 1), (2, 3, 4), (17, 16, 15), (18, 33, 31), (3, 25, 26), (5, 32, 65),
    # 32 lines a block up to 253 samples on the axis, then 16, 8, ... and from
    # 8190 one thread per line in global memory
    (2, 253, 3), (2, 254, 3), (3, 509, 2), (3, 510, 2), (510, 2, 35), (2, 2, 1022),
    (2, 8189, 1), (1, 8190, 2), (2, 1, 8190), (8190, 1, 2)])
def test_prefilter_line_groups(shape):
    """Against the oracle's recursion; the two differ by the contraction of a
    few operations, each within an ulp of coefficients of order one (the
    recursion damps earlier errors by 0.27 a step), so 1e-13 holds with room."""
    from numbacs_amd import _lib
    from numbacs_amd.flows import prefilter3_device

    U = np.random.default_rng(sum(shape)).standard_normal(shape)
    C = _lib.to_host(prefilter3_device(U))
    assert C.shape == tuple(n + 2 for n in shape)
    assert relerr(C, oracle.prefilter3(U)) < 1e-13


def test_flow_arrays_are_reused_safely():
    """A flow made while others of its size come and go evaluates its own
    coefficients: replaced handles, handles of near sizes, two alive at once,
    and a fresh start after the last has closed."""
    from numbacs_amd.flows import flow_velocity, get_flow_2D, get_flow_linear_2D

    rng = np.random.default_rng(7)
    pts, t = rng.uniform(0.1, 0.9, (50, 2)), rng.uniform(0.1, 0.9, 50)
    p = np.array([1.0])

    def make(k):
        n = (9 + k % 2, 12, 11)  # near sizes share blocks
        grid = tuple((0.0, 1.0, m) for m in n)
        if k % 3 == 2:
            return get_flow_linear_2D(grid, np.full(n, k + 1.0), np.full(n, -k - 1.0))
        C = np.full(tuple(m + 2 for m in n), k + 1.0)  # constant coefficients: constant field
        return get_flow_2D(grid, C, -C)

    kept, current = make(100), None
    for k in range(12):
        current = make(k)  # the previous handle closes after this one is made
        for f, v in ((current, k + 1.0), (kept, 101.0)):
            got = flow_velocity(f, t, pts, p)
            assert np.allclose(got[:, 0], v, rtol=1e-12) and np.allclose(got[:, 1], -v, rtol=1e-12)
    kept.close()
    current.close()
    assert np.allclose(flow_velocity(make(3), t, pts, p)[:, 0], 4.0, rtol=1e-12)


@pytest.mark.parametrize("kind", ["double_gyre", "trilinear"])
@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("shape", [(1, 1), (3, 11), (33, 4), (8, 65)])
def test_pair_lanes_equal_one_lane(kind, precision, shape):
    """The two-lane solver runs the one-lane solver's operations: flow maps,
    status and step counts equal bit for bit (the batch of a size above the
    double gyre's pair limit, and a map's point list, as counterparts)."""
    from numbacs_amd import _lib
    from numbacs_amd.flows import get_flow_linear_2D, get_predefined_flow
    from numbacs_amd.integration import flowmap_grid_2d_device

    rng = np.random.default_rng(3)
    if kind == "double_gyre":
        flow, p, _ = get_predefined_flow(kind, int_direction=-1.0)
        p[3], box, t0, T = 0.02, ((0.0, 2.0), (0.0, 1.0)), 1.0, -7.0
    else:
        n = (9, 21, 17)
        U, V = rng.standard_normal((2,) + n)
        flow = get_flow_linear_2D(tuple((0.0, 1.0, m) for m in n), U, V)
        p, box, t0, T = np.array([1.0]), ((-0.05, 1.05), (-0.05, 1.05)), 0.1, 0.8
    nx, ny = shape
    x, y = np.linspace(*box[0], nx), np.linspace(*box[1], ny)

    def run(xs, ys):
        st, ns = (_lib.empty((len(xs), len(ys)), "i32") for _ in range(2))
        fm = flowmap_grid_2d_device(flow, t0, T, _lib.to_dev(xs), _lib.to_dev(ys), p,
                                    precision=precision, status=st, nsteps=ns)
        return [_lib.to_host(a) for a in (fm, st, ns)]

    got = run(x, y)
    assert (got[1] == 1).all()
    # the same rows inside a map of 300,000 particles: one lane per particle
    # for the double gyre
    xs = np.concatenate([x, np.linspace(*box[0], 300000 // ny)])
    for a, b in zip(got, run(xs, y)):
        assert np.array_equal(a, b[:nx])


@pytest.mark.parametrize("precision", [0, 1])
def test_bickley_queue_equals_grid_launch(precision):
    """The default tile queue (more tiles than wavefronts) against the grid
    launch, and a map small enough to take the grid launch by itself."""
    from numbacs_amd import _lib, autotune
    from numbacs_amd.flows import get_predefined_flow
    from numbacs_amd.integration import flowmap_grid_2d_device

    flow, p, dom = get_predefined_flow("bickley_jet")
    saved = autotune.get(1, precision)
    assert saved[2] > 0

    def run(nx, ny):
        return _lib.to_host(flowmap_grid_2d_device(
            flow, 0.0, 9.0, _lib.to_dev(np.linspace(*dom[0], nx)),
            _lib.to_dev(np.linspace(*dom[1], ny)), p, precision=precision))

    try:
        got = [run(*n) for n in ((711, 333), (9, 33))]
        autotune.set_config(1, precision, (1, 64, 0))
        want = [run(*n) for n in ((711, 333), (9, 33))]
    finally:
        autotune.set_config(1, precision, saved)
    for a, b in zip(got, want):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("n", [1, 63, 64, 65, 1000])
@pytest.mark.parametrize("kind", ["plain", "wide", "negative", "nonfinite"])
def test_fused_inference_where_rounding_is_undecided(n, kind):
    """The fused kernel's short forms of GELU, sine and cosine hand over to the
    library functions wherever these could round otherwise, so it equals the
    layer-by-layer kernels bit for bit: ordinary particles, features of
    thousands of revolutions, activations below -4 throughout (every one is
    handed over, so the lists fill), and arguments that are not finite."""
    import torch
    from numbacs_amd.surrogate import MLPSurrogate

    rng = np.random.default_rng(n)
    net = MLPSurrogate([0.0] * 4, [1.0] * 4, out_scale=[10.0, 5.0], seed=n)
    x = rng.uniform(-1, 1, (n, 4)).astype(np.float32)
    if kind == "wide":
        x *= rng.choice(np.float32([1e1, 1e3, 1e4, 1e7]), (n, 1))
    if kind == "negative":
        for b in net.b[:4]:
            b.fill_(-6.0)
    if kind == "nonfinite":
        x[rng.integers(0, n, 3), rng.integers(0, 4, 3)] = [np.inf, -np.inf, np.nan]
    inp = torch.tensor(x, device="cuda")
    a, b = net.predict_device(inp), net.predict_device_unfused(inp)
    assert torch.equal(torch.isnan(a), torch.isnan(b))
    assert torch.equal(torch.nan_to_num(a), torch.nan_to_num(b))


@pytest.mark.parametrize("kind", ["constant", "low bits", "two values", "infinite", "wide"])
@pytest.mark.parametrize("n", [1, 2, 2049, 65536, 65537, 300001])
def test_percentile_key_list(n, kind):
    """The percentile's list of keys that share the leading 22 bits: short,
    exactly full, and overflowing (all keys equal there, decided by the low
    digits over the whole array).  Exact: order statistics and numpy's lerp,
    which the device rounds once per step (fused multiply-add)."""
    from fractions import Fraction

    from numbacs_amd import _lib

    def reference(f, q):
        vi = (n - 1) * (q / 100.0)
        lo = min(int(vi), n - 1)
        part = np.sort(f)
        a, b, g = float(part[lo]), float(part[min(lo + 1, n - 1)]), vi - int(vi)
        if not (np.isfinite(a) and np.isfinite(b)):
            with np.errstate(invalid="ignore"):
                return np.percentile(f, q)
        d = Fraction(b - a)
        return float(Fraction(b) - d * Fraction(1 - g) if g >= 0.5 else Fraction(a) + d * Fraction(g))

    rng = np.random.default_rng(n)
    f = {"constant": lambda: np.full(n, -0.25),
         "low bits": lambda: 1.0 + rng.integers(0, 1 << 30, n) * 2.0 ** -52,
         "two values": lambda: rng.choice([1.0, 1.0 + 2.0 ** -52], n),
         "infinite": lambda: rng.choice([-np.inf, -1.0, 0.0, -0.0, 5e-324], n),
         "wide": lambda: rng.standard_normal(n) * 10.0 ** rng.integers(-300, 300, n)}[kind]()
    fd, out = _lib.to_dev(f), _lib.empty((1,))
    for q in (0.0, 37.3, 50.0, 90.0, 100.0):
        _lib.check(_lib.load().nbx_percentile(_lib.ptr(fd), n, q, _lib.ptr(out),
                                              _lib.stream_ptr()))
        got = _lib.to_host(out)[0]
        ref = reference(f, q)
        assert got == ref or (np.isnan(got) and np.isnan(ref))


@pytest.mark.parametrize("shape", [(5, 5), (16, 64), (17, 65), (16, 200), (300, 64), (33, 129),
                                   (130, 257)])
@pytest.mark.parametrize("gaps", [0.0, 0.3, 0.6])
def test_ridge_components_across_tiles(shape, gaps):
    """Half the grid is ridge points that touch diagonally (every second point
    of a checkerboard), with gaps: one component over all tiles, many that
    cross their borders, thousands of single points.  Equal to the oracle."""
    from numbacs_amd.extraction import ftle_ridges

    nx, ny = shape
    rng = np.random.default_rng(nx * ny)
    x, y = np.arange(nx) / 8.0, np.arange(ny) / 8.0
    i, j = np.indices(shape)
    f = 1.0 + 0.5 * (-1.0) ** (i + j) + 0.01 * rng.random(shape)
    f[rng.random(shape) < gaps] = 0.0
    ev = np.zeros(shape + (2,))
    ev[..., 0] = 1.0
    for least, q in ((1, 0), (3, 0), (1, 60)):
        got = ftle_ridges(f, ev, x, y, percentile=q, min_ridge_pts=least)
        ref = oracle.ridges(f, ev, x, y, percentile_=q, min_ridge_pts=least)
        assert len(got) == len(ref)
        for a, b in zip(got, ref):
            assert np.array_equal(a, b)


@pytest.mark.parametrize("M,N,K", [(64, 64, 32), (128, 64, 96), (64, 192, 128), (192, 128, 160),
                                   (64, 64, 288)])
def test_gemm_turns(M, N, K):
    """All four forms of the GEMM where its turns of 128 k end: one slab of 32,
    remainders of one to three slabs, several turns.  FP32 results: each is a sum
    of K products of bf16 values (exact in float) rounded K times, so within
    K ulps of the sum of magnitudes; the bf16 outputs within one bf16 ulp more."""
    import torch
    from numbacs_amd import _lib

    lib = _lib.load()
    rng = np.random.default_rng(M + N + K)

    def bf16(*shape):
        return torch.tensor(rng.standard_normal(shape), dtype=torch.bfloat16, device="cuda")

    def run(mode, A, B, c32=None, c16=None, bias=None, pre=None):
        ptr = lambda v: None if v is None else _lib.ptr(v)
        _lib.check(lib.nbx_mlp_gemm(mode, ptr(A), ptr(B), M, N, K, ptr(c32), ptr(c16), ptr(bias),
                                    ptr(pre), _lib.stream_ptr()))

    def out(dtype):
        return torch.full((M, N), float("nan"), dtype=dtype, device="cuda")

    d = lambda v: v.double().cpu()
    eps = K * 2.0 ** -23
    A, B, At, Bt = bf16(M, K), bf16(K, N), bf16(K, M), bf16(N, K)
    bias = torch.tensor(rng.standard_normal(N), dtype=torch.float32, device="cuda")
    pre = torch.tensor(rng.standard_normal((M, N)), dtype=torch.float32, device="cuda")

    def inner(a):
        return 0.7978845608028654 * (a + 0.044715 * a ** 3)

    for mode, left, right in ((3, d(A), d(B)), (2, d(At).T, d(B))):
        c = out(torch.float32)
        run(mode, A if mode == 3 else At, B, c32=c)
        assert ((d(c) - left @ right).abs() <= eps * (left.abs() @ right.abs())).all()
    c, h = out(torch.float32), out(torch.bfloat16)
    run(0, A, B, c32=c, c16=h, bias=bias)
    ref = d(A) @ d(B) + d(bias)
    assert ((d(c) - ref).abs() <= eps * (d(A).abs() @ d(B).abs() + d(bias).abs())).all()
    g = 0.5 * d(c) * (1 + torch.tanh(inner(d(c))))
    assert ((d(h) - g).abs() <= 2.0 ** -8 * g.abs() + 1e-6 * (1 + d(c).abs())).all()
    h = out(torch.bfloat16)
    run(1, A, Bt, c16=h, pre=pre)
    dh, t = d(A) @ d(Bt).T, torch.tanh(inner(d(pre)))
    slope = 0.5 * (1 + t) + 0.5 * d(pre) * (1 - t ** 2) * 0.7978845608028654 * (
        1 + 3 * 0.044715 * d(pre) ** 2)
    # two roundings to bf16, and eps of the product's magnitudes
    err = (2.0 ** -7 * dh.abs() + 2 * eps * (d(A).abs() @ d(Bt).abs().T)) * slope.abs() + 1e-5 * dh.abs()
    assert ((d(h) - dh * slope).abs() <= err).all()


@pytest.mark.parametrize("n", [1, 31, 33, 127, 129, 1000])
@pytest.mark.parametrize("width", [64, 256, 320])
def test_column_sums_of_partial_groups(n, width):
    """Column sums where a block's row groups are cut short or empty, and for
    more columns than a group has threads; within n ulps of the magnitudes."""
    import torch
    from numbacs_amd import _lib

    rng = np.random.default_rng(n + width)
    da = torch.tensor(rng.standard_normal((n, width)), dtype=torch.bfloat16, device="cuda")
    gb = torch.full((width,), float("nan"), dtype=torch.float32, device="cuda")
    _lib.check(_lib.load().nbx_mlp_colsum(_lib.ptr(da), n, width, _lib.ptr(gb), _lib.stream_ptr()))
    ref = da.double()
    assert ((gb.double() - ref.sum(0)).abs() <= n * 2.0 ** -23 * ref.abs().sum(0)).all()


@pytest.mark.parametrize("M,N,K", [(64, 64, 32), (64, 128, 224), (128, 64, 512), (64, 192, 1056),
                                   (256, 256, 1024)])
def test_weight_grad_with_column_sums(M, N, K):
    """The fused weight and bias gradients, without and with a split batch and
    with a last part that ends inside a turn; each within K ulps of the
    magnitudes it sums."""
    import torch
    from numbacs_amd import _lib

    rng = np.random.default_rng(M + N + K)
    h, da = (torch.tensor(rng.standard_normal((K, w)), dtype=torch.bfloat16, device="cuda")
             for w in (M, N))
    gW = torch.full((M, N), float("nan"), dtype=torch.float32, device="cuda")
    gb = torch.full((N,), float("nan"), dtype=torch.float32, device="cuda")
    _lib.check(_lib.load().nbx_mlp_weight_grad(_lib.ptr(h), _lib.ptr(da), M, N, K, _lib.ptr(gW),
                                               _lib.ptr(gb), _lib.stream_ptr()))
    hd, dd = h.double().cpu(), da.double().cpu()
    eps = K * 2.0 ** -23
    assert ((gW.double().cpu() - hd.T @ dd).abs() <= eps * (hd.abs().T @ dd.abs())).all()
    assert ((gb.double().cpu() - dd.sum(0)).abs() <= eps * dd.abs().sum(0)).all()


@pytest.mark.parametrize("n", [1, 3, 63, 65, 130])
@pytest.mark.parametrize("width", [8, 64, 256, 264, 512])
def test_output_layer_of_any_width(n, width):
    """The output layer forward and backward where its rows' blocks and its
    chunks of 256 columns are cut short.  Sums within width (or n) ulps of the
    magnitudes; the deltas two roundings to bf16 from float64."""
    import torch
    from numbacs_amd import _lib

    lib, rng = _lib.load(), np.random.default_rng(n + width)

    def dev(a, dtype):
        return torch.tensor(a, dtype=dtype, device="cuda")

    h, W = (dev(rng.standard_normal(s), torch.bfloat16) for s in ((n, width), (width, 2)))
    b, dy, pre = (dev(rng.standard_normal(s), torch.float32) for s in ((2,), (n, 2), (n, width)))
    y = torch.full((n, 2), float("nan"), device="cuda")
    gW, gb = torch.full((width, 2), float("nan"), device="cuda"), torch.zeros(2, device="cuda")
    da = torch.full((n, width), float("nan"), dtype=torch.bfloat16, device="cuda")
    s = _lib.stream_ptr()
    _lib.check(lib.nbx_mlp_out_forward(_lib.ptr(h), n, width, _lib.ptr(W), _lib.ptr(b),
                                       _lib.ptr(y), s))
    _lib.check(lib.nbx_mlp_out_backward(_lib.ptr(dy), _lib.ptr(h), _lib.ptr(pre), n, width,
                                        _lib.ptr(W), _lib.ptr(gW), _lib.ptr(gb), _lib.ptr(da), s))
    y, gW, gb, da, h, W, b, dy, pre = (v.double().cpu()
                                       for v in (y, gW, gb, da, h, W, b, dy, pre))
    ulp = 2.0 ** -23
    assert ((y - (h @ W + b)).abs() <= (width + 1) * ulp * (h.abs() @ W.abs() + b.abs())).all()
    assert ((gW - h.T @ dy).abs() <= (n + 1) * ulp * (h.abs().T @ dy.abs())).all()
    assert ((gb - dy.sum(0)).abs() <= (n + 1) * ulp * dy.abs().sum(0)).all()
    t = torch.tanh(0.7978845608028654 * (pre + 0.044715 * pre ** 3))
    slope = 0.5 * (1 + t) + 0.5 * pre * (1 - t ** 2) * 0.7978845608028654 * (
        1 + 3 * 0.044715 * pre ** 2)
    dh, mag = dy @ W.T, dy.abs() @ W.abs().T
    err = (2.0 ** -7 * dh.abs() + 4 * ulp * mag) * slope.abs() + 1e-5 * dh.abs()
    assert ((da - dh * slope).abs() <= err).all()


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("kind", ["double_gyre", "spline", "trilinear"])
def test_zero_absolute_tolerance_near_zero(kind, precision):
    """Error norms whose scale rtol |y| is subnormal: the lane groups' quotients
    by a shared reciprocal hand over to the division there.  The double gyre's
    pair equals its one-lane form bit for bit; gridded flows of velocities
    as small end every solve."""
    from numbacs_amd import _lib
    from numbacs_amd.flows import get_flow_2D, get_flow_linear_2D, get_predefined_flow
    from numbacs_amd.integration import flowmap_grid_2d_device

    v = np.array([1e-310, -3e-308, 2e-303, 1e-300, -1e-285, 1e-270, 1e-200, 0.3])
    rng = np.random.default_rng(8)
    if kind == "double_gyre":
        flow, p, _ = get_predefined_flow(kind, int_direction=-1.0)
        T = 3.0
    else:
        n = (6, 9, 8)
        U, V = rng.uniform(0.5, 1.5, (2,) + n) * 1e-300
        grid = ((0.0, 5.0, n[0]), (-1.0, 1.0, n[1]), (-1.0, 1.0, n[2]))
        if kind == "spline":
            from numbacs_amd.flows import prefilter3_device

            flow = get_flow_2D(grid, prefilter3_device(U), prefilter3_device(V))
        else:
            flow = get_flow_linear_2D(grid, U, V)
        p, T = np.array([1.0]), 2.0

    def run(xs, ys):
        st, ns = (_lib.empty((len(xs), len(ys)), "i32") for _ in range(2))
        fm = flowmap_grid_2d_device(flow, 0.5, T, _lib.to_dev(xs), _lib.to_dev(ys), p, atol=0.0,
                                    precision=precision, status=st, nsteps=ns)
        return [_lib.to_host(a) for a in (fm, st, ns)]

    fm, status, steps = run(v, v)
    assert (status == 1).all()
    if kind == "double_gyre":
        xs = np.concatenate([v, np.full(100000, 1.0)])  # one lane per particle
        for a, b in zip((fm, status, steps), run(xs, v)):
            assert np.array_equal(a, b[:len(v)])
