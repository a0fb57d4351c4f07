"""The tile kernels' arithmetic: fp32 operands as three bf16 pieces each, six
products of them on the matrix cores.  Error against fp64, operands that have
no such split (infinities, NaN, magnitudes past bf16's largest), and the
sizes where a tile, a stage or a chunk ends."""
import contextlib
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _torch():
    import torch
    return torch


@pytest.fixture(scope="module")
def lib():
    import tlgemm
    _torch().cuda.init()
    L = tlgemm.load()
    L.check(L.tlg_init(0), "tlg_init")
    return L


def run(lib, op, X, W, dY, grouped):
    """The primitive on device copies (accumulating ones from zero), as numpy."""
    torch = _torch()
    M, K, N = X.shape[0], X.shape[1], W.shape[1]
    x, w, dy = (torch.from_numpy(np.ascontiguousarray(a)).cuda() for a in (X, W, dY))
    shape = {"mm": (M, N), "mm_bt": (M, K), "mm_atb": (K, N)}[op]
    out = torch.zeros(shape, device="cuda")
    a, b = {"mm": (x, w), "mm_bt": (dy, w), "mm_atb": (x, dy)}[op]
    st = torch.cuda.current_stream().cuda_stream
    if grouped:
        lib.group([dict(op=op, beta=0 if op == "mm" else 1, C=out.data_ptr(), M=M, K=K, N=N, A=[a.data_ptr()],
                        B=[b.data_ptr()])], st)
    else:
        {"mm": lib.mm, "mm_bt": lib.mm_bt, "mm_atb": lib.mm_atb}[op](out.data_ptr(), a.data_ptr(), b.data_ptr(), M, K,
                                                                    N, st)
    torch.cuda.synchronize()
    return out.cpu().numpy()


def want(op, X, W, dY):
    X, W, dY = (a.astype(np.float64) for a in (X, W, dY))
    with np.errstate(all="ignore"):
        return {"mm": lambda: X @ W, "mm_bt": lambda: dY @ W.T, "mm_atb": lambda: X.T @ dY}[op]()


def reduction(op, M, K, N):
    return {"mm": K, "mm_bt": N, "mm_atb": M}[op]


# (M, K, N): a tile, stage or chunk (of the 32x32 shape; the others' lie among
# multiples of these) ends one short, exactly, or one past
EDGES = [(9, 16, 16), (70, 1, 33), (70, 33, 1), (70, 3, 2), (1030, 2, 5), (9, 130, 3), (67, 261, 254), (32, 32, 32), (33, 20, 68), (64, 15, 64), (65, 17, 63), (127, 48, 129), (128, 128, 128),
         (257, 131, 259), (300, 64, 36), (513, 4, 72), (1024, 512, 192), (2050, 72, 516)]


@pytest.mark.parametrize("op", ["mm", "mm_bt", "mm_atb"])
@pytest.mark.parametrize("shape", EDGES, ids=str)
def test_error_against_fp64(lib, op, shape):
    """check_error by the automatic rules (32x32 tiles at all but the largest of
    these sizes)."""
    for grouped in (False, True):
        check_error(lib, op, grouped, shape)


def check_error(lib, op, grouped, shape):
    """Each product is exact to 2^-25 and each 16-step MFMA adds one rounding
    of the running sum (2^-24): over R steps the error's 2-norm stays under
    2^-24 (1 + sqrt(R / 16)) times the result's for random signs, with room
    for the rounding inside an MFMA (x 4)."""
    M, K, N = shape
    r = np.random.default_rng(M * 7 + K)
    X = r.standard_normal((M, K), dtype=np.float32)
    W = (0.02 * r.standard_normal((K, N))).astype(np.float32)
    dY = (0.01 * r.standard_normal((M, N))).astype(np.float32)
    ref = want(op, X, W, dY)
    R = reduction(op, M, K, N)
    tol = 4 * 2.0 ** -24 * (1 + np.sqrt(R / 16))
    if grouped and (M % 4 and op == "mm_atb" or K % 4 or N % 4):
        return
    got = run(lib, op, X, W, dY, grouped)
    err = np.linalg.norm(got - ref) / np.linalg.norm(ref)
    assert err <= tol, (op, shape, grouped, err, tol)


@pytest.mark.parametrize("op", ["mm", "mm_bt", "mm_atb"])
@pytest.mark.parametrize("grouped", [False, True])
@pytest.mark.parametrize("shape", [(40, 36, 52), (200, 132, 260)], ids=str)
def test_operands_without_a_split(lib, op, grouped, shape):
    """Infinities, NaN and values that round to bf16's infinity give what fp32
    sums give, and leave the outputs they do not enter alone."""
    check_without_a_split(lib, op, grouped, shape)


def check_without_a_split(lib, op, grouped, shape):
    M, K, N = shape
    r = np.random.default_rng(3)
    X = r.standard_normal((M, K), dtype=np.float32)
    W = r.standard_normal((K, N), dtype=np.float32)
    dY = r.standard_normal((M, N), dtype=np.float32)
    a, b = {"mm": (X, W), "mm_bt": (dY, W), "mm_atb": (X, dY)}[op]
    a[3, 5], a[17, 2], a[8, 9] = np.inf, np.nan, np.float32(3.4e38)
    b[1, 7], b[6, 11] = -np.inf, np.float32(-3.4e38)
    if op == "mm_atb":
        a[:, 20] = 0.0                               # 0 x inf
    got, ref = run(lib, op, X, W, dY, grouped), want(op, X, W, dY)
    assert np.array_equal(np.isnan(got), np.isnan(ref))
    inf = np.isinf(ref)
    assert np.array_equal(got[inf], np.sign(ref[inf]) * np.inf)
    # elsewhere each of R roundings is at most 2^-24 of the terms' absolute sum
    # (where that sum is in range: a partial sum past it is infinite in fp32)
    terms = want(op, *(np.abs(np.where(np.isfinite(t), t, 0.0)) for t in (X, W, dY)))
    fine = np.isfinite(ref) & (terms < 3.3e38)
    assert fine.any()
    assert (np.abs(got[fine] - ref[fine]) <= reduction(op, M, K, N) * 2.0 ** -24 * terms[fine]).all()


@pytest.mark.parametrize("scale", [1e-30, 1e-18, 1e18])
def test_magnitudes(lib, scale):
    """The pieces keep fp32's exponent range: tiny and huge operands are as
    exact as ordinary ones while the products are in range."""
    r = np.random.default_rng(5)
    X = (scale * r.standard_normal((96, 80))).astype(np.float32)
    W = (r.standard_normal((80, 112)) / (scale if scale > 1 else 1)).astype(np.float32)
    got, ref = run(lib, "mm", X, W, W[:1], False), want("mm", X, W, W[:1])
    assert np.linalg.norm(got - ref) <= 4 * 2.0 ** -24 * (1 + np.sqrt(5)) * np.linalg.norm(ref)


# every shape of the automatic rules, pinned: single calls whole and split,
# grouped launches (128x128, 128x64, 64x64, 64x32 and 32x32 tiles, wave groups
# along the reduction and none)
PINNED = [(False, c, sp) for c in (9, 8, 3, 15) for sp in (1, 3)] + [(True, c, 0) for c in (33, 47, 34, 35, 41, 21, 15)]


# extents one short of, at and one past 128 and 256, aligned and odd
WIDE = [(127, 129, 255), (129, 255, 127), (255, 127, 129), (257, 193, 131), (128, 128, 256), (132, 260, 124),
        (252, 68, 388), (36, 512, 132), (516, 132, 36)]


@contextlib.contextmanager
def pinned(lib, grouped, cfg, splits):
    lib.check(lib.tlg_tune_group(cfg) if grouped else lib.tlg_tune_force(cfg, splits), "pin")
    try:
        yield
    finally:
        lib.check(lib.tlg_tune_group(-1) if grouped else lib.tlg_tune_force(-1, 0), "unpin")


@pytest.mark.parametrize("op", ["mm", "mm_bt", "mm_atb"])
@pytest.mark.parametrize("pin", PINNED, ids=str)
def test_error_on_every_shape(lib, op, pin):
    """The bound of the automatic choice on each tile shape, where the large
    tiles' rows, columns, stages and chunks end; single calls with rows that are
    no whole float4s too."""
    for shape in EDGES + WIDE:
        with pinned(lib, *pin):
            check_error(lib, op, pin[0], shape)


@pytest.mark.parametrize("op", ["mm", "mm_bt", "mm_atb"])
@pytest.mark.parametrize("pin", PINNED, ids=str)
def test_operands_without_a_split_on_every_shape(lib, op, pin):
    """The same on each tile shape, at ragged sizes past one and two of the
    largest tiles (aligned rows, and odd ones for the single calls)."""
    for shape in ((200, 132, 260), (304, 260, 132)) + (() if pin[0] else ((201, 131, 259),)):
        with pinned(lib, *pin):
            check_without_a_split(lib, op, pin[0], shape)


@pytest.mark.parametrize("op", ["mm", "mm_bt", "mm_atb"])
def test_a_nan_does_not_stall_the_launch(lib, op):
    """One NaN in each operand sends a row and a column of outputs, and NaN
    weights every output, through the fp32 sums.  On the matrix cores that takes 2
    to 5 times the finite call (one lane per output took 25 to 80 times)."""
    torch = _torch()
    M, K, N = 4096, 256, 768
    X, W, dY = (torch.randn(*s, device="cuda") for s in ((M, K), (K, N), (M, N)))
    a, b, out = {"mm": (X, W, torch.zeros(M, N, device="cuda")), "mm_bt": (dY, W, torch.zeros(M, K, device="cuda")),
                 "mm_atb": (X, dY, torch.zeros(K, N, device="cuda"))}[op]
    f = {"mm": lib.mm, "mm_bt": lib.mm_bt, "mm_atb": lib.mm_atb}[op]
    st = torch.cuda.current_stream().cuda_stream

    def us():
        best = 1e9
        for _ in range(5):
            e0, e1 = (torch.cuda.Event(enable_timing=True) for _ in range(2))
            e0.record()
            for _ in range(5):
                f(out.data_ptr(), a.data_ptr(), b.data_ptr(), M, K, N, st)
            e1.record()
            torch.cuda.synchronize()
            best = min(best, 200 * e0.elapsed_time(e1))
        return best

    finite = us()
    a[5, 7] = b[3, 5] = float("nan")
    one = us()
    b[:] = float("nan")
    every = us()
    print(op, "finite", finite, "one NaN", one, "all", every, flush=True)
    assert max(one, every) <= 12 * finite, (finite, one, every)


# operand magnitudes from where an unscaled third piece would end (2^-110) down
# to fp32's subnormals
TINY = [1e-32, 1e-34, 1e-36, 1e-38, 1e-40]


def fp32_of(x):
    """x to the nearest fp32 and that value in fp64, by integers below 2^-126: a
    library loaded earlier may have set the CPU to flush subnormals."""
    sub = np.abs(x) < 2.0 ** -126
    k = np.rint(np.where(sub, np.ldexp(x, 149), 0)).astype(np.int64)
    f = np.where(sub, 1.0, x).astype(np.float32)
    bits = np.where(sub, np.abs(k) | (k < 0).astype(np.int64) << 31, f.view(np.uint32).astype(np.int64))
    return bits.astype(np.uint32).view(np.float32), np.where(sub, np.ldexp(k.astype(np.float64), -149), f.astype(np.float64))


def check_tiny(lib, op, grouped, shape, scale):
    """One operand at `scale`, the other so large that the sums are ordinary
    numbers, below 2^112 and past it (where the tiles take the fp32 blocks):
    the bound of test_error_against_fp64."""
    M, K, N = shape
    r = np.random.default_rng(K + N)
    names = {"mm": ("X", "W"), "mm_bt": ("dY", "W"), "mm_atb": ("X", "dY")}[op]
    dims = {"X": (M, K), "W": (K, N), "dY": (M, N)}
    tol = 4 * 2.0 ** -24 * (1 + np.sqrt(reduction(op, M, K, N) / 16))
    for small, big in (names, names[::-1]):
        for large in {min(1 / scale, 1e30), min(1 / scale, 1e36)}:
            o = {n: np.zeros(d, np.float32) for n, d in dims.items()}
            o64 = {n: np.zeros(d) for n, d in dims.items()}
            o[small], o64[small] = fp32_of(scale * r.standard_normal(dims[small]))
            o[big], o64[big] = fp32_of(large * r.standard_normal(dims[big]))
            ref = want(op, o64["X"], o64["W"], o64["dY"])
            got = run(lib, op, o["X"], o["W"], o["dY"], grouped)
            err = np.linalg.norm(got - ref) / np.linalg.norm(ref)
            assert err <= tol, (op, grouped, shape, scale, large, small, err, tol)


@pytest.mark.parametrize("scale", TINY)
@pytest.mark.parametrize("op", ["mm", "mm_bt", "mm_atb"])
@pytest.mark.parametrize("grouped", [False, True])
def test_tiny_operands(lib, op, grouped, scale):
    for shape in ((40, 36, 52), (200, 132, 260)) + (() if grouped else ((67, 61, 254),)):
        check_tiny(lib, op, grouped, shape, scale)


@pytest.mark.parametrize("op", ["mm", "mm_bt", "mm_atb"])
@pytest.mark.parametrize("pin", PINNED, ids=str)
def test_tiny_operands_on_every_shape(lib, op, pin):
    with pinned(lib, *pin):
        for scale in (1e-36, 1e-40):
            check_tiny(lib, op, pin[0], (200, 132, 260), scale)


@pytest.mark.parametrize("op", ["mm", "mm_bt", "mm_atb"])
@pytest.mark.parametrize("R", [1, 2, 3])
def test_shortest_reductions(lib, op, R):
    """R steps are R roundings of 2^-24 of the terms' absolute sum, as in fp32, on
    every tile shape: the piece products that are left out add nothing to it."""
    M, K, N = {"mm": (300, R, 260), "mm_bt": (300, 260, R), "mm_atb": (R, 300, 260)}[op]
    r = np.random.default_rng(R)
    X, W, dY = (r.standard_normal(s, dtype=np.float32) for s in ((M, K), (K, N), (M, N)))
    bound = R * 2.0 ** -24 * want(op, *(np.abs(t) for t in (X, W, dY)))
    for pin in PINNED + [(False, -1, 0), (True, -1, 0)]:
        if pin[0] and op != "mm_atb":
            continue                       # grouped calls take reductions of whole float4s there
        with pinned(lib, *pin):
            err = np.abs(run(lib, op, X, W, dY, pin[0]) - want(op, X, W, dY))
        assert (err <= bound).all(), (op, R, pin, (err / bound).max())


@pytest.mark.parametrize("call", [("mm", 4096, 2048, 384), ("mm_bt", 4096, 384, 2048), ("mm_atb", 8192, 1024, 1024),
                                  ("mm", 1024, 4096, 960)], ids=str)
def test_large_outputs_run_whole(lib, call):
    """From 240 64x64 tiles on no call splits its reduction: a split's partials
    lie in a workspace that a call on another stream would write too."""
    assert lib.kernel_name(*call)[1] == 1
    torch = _torch()
    op, M, K, N = call
    dims = {"mm": ((M, K), (K, N), (M, N)), "mm_bt": ((M, N), (K, N), (M, K)), "mm_atb": ((M, K), (M, N), (K, N))}[op]
    f = {"mm": lib.mm, "mm_bt": lib.mm_bt, "mm_atb": lib.mm_atb}[op]
    torch.manual_seed(1)
    one, two, both = [], [], [torch.cuda.Stream() for _ in range(2)]
    ops = [tuple(torch.randn(*s, device="cuda") for s in dims[:2]) for _ in both]
    for outs, streams in ((one, both[:1] * 2), (two, both)):
        outs += [torch.zeros(*dims[2], device="cuda") for _ in both]
        torch.cuda.synchronize()
        for _ in range(4):
            for (a, b), c, s in zip(ops, outs, streams):
                f(c.data_ptr(), a.data_ptr(), b.data_ptr(), M, K, N, s.cuda_stream)
        torch.cuda.synchronize()
    assert all(torch.equal(x, y) for x, y in zip(one, two))


def test_tile_policy_hook(lib):
    """A list of candidates takes the automatic one's place and a candidate of -1
    puts it back; min_waves scales whichever is there."""
    torch = _torch()
    M, K, N = 4096, 256, 768
    x, w, y = (torch.randn(*s, device="cuda") for s in ((M, K), (K, N), (M, N)))

    def shape():
        lib.group([dict(op="mm", C=y.data_ptr(), M=M, K=K, N=N, A=[x.data_ptr()], B=[w.data_ptr()])])
        torch.cuda.synchronize()
        return lib.tlg_group_kernel().decode()

    def policy(cands, min_waves=0.0):
        c = (ctypes.c_int * max(1, len(cands)))(*cands)
        return lib.tlg_tune_group_policy(c, len(cands), min_waves, 0)

    start = shape()
    try:
        assert policy([], 30.0) == 0 and "Tile<64, 32, " in shape() and "Tile<64, 32, " not in start
        assert policy([], 3.0) == 0 and shape() == start
        assert policy([33, 15]) == 0 and "Tile<32, 32, " in shape()          # 192 of 768 items
        assert policy([], 0.5) == 0 and "Tile<128, 128, " in shape()
        assert policy([-1], 3.0) == 0 and shape() == start
        for bad in ([2], [99], [-1, 3], [-2]):
            assert policy(bad) != 0 and shape() == start
    finally:
        lib.check(policy([-1], 3.0), "policy")
