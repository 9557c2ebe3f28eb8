"""The scratch buffer in which dh_lra keeps K: its size, its return, and calls that
cannot have it, through the C ABI."""
import pytest

import darray_optimizer_amd as dh

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def nothing_unwiped(dev):
    """Earlier tests leave a large buffer; once it is given back, new ones are refused
    until the driver has wiped it (an eighth of the memory at 25 GB/s)."""
    import time

    import torch
    wait = torch.cuda.get_device_properties(0).total_memory / 8 / 25e9
    solve(dev, *problem(300, 8, 8)[:2])  # a handle's first solve may do without a buffer
    dev.scratch_trim()
    time.sleep(wait)
    yield
    time.sleep(wait)


def problem(n, d, l, seed=0, labels=False):
    import torch
    g = torch.Generator(device="cuda").manual_seed(seed + n + d + l)
    X = 0.3 * torch.randn((n, d), dtype=torch.float64, device="cuda", generator=g)
    Om = torch.randn((l, n), dtype=torch.float64, device="cuda", generator=g)
    y = 0.5 + torch.rand(n, dtype=torch.float64, device="cuda", generator=g) if labels else None
    return X, Om, y


def solve(h, X, Om, q=1, y=None, prec=dh.DH_PREC_F64):
    import torch
    Q, W = torch.empty_like(Om), torch.empty_like(Om)
    assert h.lra(X, Om, 0.5 / X.shape[1], q, Q, W, y=y, prec=prec) == 0
    return Q, W


def test_scratch_is_reported_and_given_back(dev):
    """8 bytes per entry of K (rows in 64s, columns in 16s) after a solve, none after
    a trim, and the same solve again."""
    import torch
    X, Om, _ = problem(3001, 40, 24)
    dev.scratch_trim()
    assert dev.scratch_bytes() == 0
    a = solve(dev, X, Om)
    assert dev.scratch_bytes() == 8 * 3008 * 3008
    held = dev.workspace_bytes()
    dev.scratch_trim()
    assert dev.scratch_bytes() == 0 and dev.workspace_bytes() == held
    b = solve(dev, X, Om)
    assert torch.equal(a[0], b[0]) and torch.equal(a[1], b[1])


@pytest.fixture
def limit(dev):
    """Allocations of `dev` beyond the given bytes, the scratch buffer included, fail."""
    import ctypes as C
    fn = dh._capi.lib().dh_debug_alloc_limit
    fn.argtypes, fn.restype = [C.c_void_p, C.c_size_t], C.c_int
    yield lambda h, b: fn(h.h, int(b))
    fn(dev.h, 0)


def test_allocations_take_the_idle_scratch_back(limit):
    """A workspace, dh_malloc and the batch's plan in memory that the idle scratch
    buffer fills: each gives it back and succeeds; what is larger still fails."""
    import ctypes as C

    import torch
    h = dh.Handle(0)
    X, Om, _ = problem(3000, 40, 24)
    solve(h, X, Om)
    solve(h, X, Om)
    size = h.scratch_bytes()
    assert size >= 8 * 3000 * 3000
    limit(h, size)
    p = C.c_void_p()
    dh._capi.call("dh_malloc", h.h, size // 2, C.byref(p))
    assert p.value and h.scratch_bytes() == 0
    dh._capi.call("dh_free", h.h, p)
    with pytest.raises(dh.DHError):
        dh._capi.call("dh_malloc", h.h, 2 * size, C.byref(p))
    assert not p.value
    limit(h, 0)
    solve(h, X, Om)
    assert h.scratch_bytes() == size
    limit(h, size)
    K = torch.empty((3000, 3000), dtype=torch.float64, device="cuda")
    torch.nn.init.eye_(K)
    assert h.potrf(K) == 0  # new workspaces
    assert h.scratch_bytes() == 0
    limit(h, 0)
    solve(h, X, Om)
    limit(h, size)
    probs = [{"X": X, "y": None, "Omega": Om, "gamma": 0.01, "q": 0, "Q": torch.empty_like(Om),
              "W": torch.empty_like(Om)}]
    info, _ = h.lra_batched(probs, prec=dh.DH_PREC_BF16)
    assert info == 0 and h.scratch_bytes() == 0
    h.close()


@pytest.mark.parametrize("prec,d", [("f64", 40), ("f64", 300), ("f16", 200), ("fp8", 256)])
def test_lra_without_the_memory_for_kept_k(limit, prec, d):
    """Memory for every workspace or for K, not for both: the solve gives K up and
    returns the bits of a solve that kept it."""
    import torch
    which = {"f64": dh.DH_PREC_F64, "f16": dh.DH_PREC_F16, "fp8": dh.DH_PREC_FP8}[prec]
    X, Om, y = problem(13000, d, 140, labels=True)
    dev = dh.Handle(0)
    dev.scratch_trim()
    a = solve(dev, X, Om, 2, y, which)
    kept = dev.scratch_bytes()
    assert kept >= (8 if prec == "f64" else 2) * 13000 * 13000
    h = dh.Handle(0)
    limit(h, kept)
    b = solve(h, X, Om, 2, y, which)
    assert h.scratch_bytes() == 0  # given up
    limit(h, 0)
    assert torch.equal(a[0], b[0]) and torch.equal(a[1], b[1])
    c = solve(h, X, Om, 2, y, which)
    assert h.scratch_bytes() == kept and torch.equal(a[1], c[1])
    h.close()
    dev.close()


def test_lra_error_without_the_memory_for_its_copies(limit):
    """n > 6400 with no room for the point-major copies of X, Q and W: the 64 x 64
    tiles, which need none.  Both sum n^2 squares that agree to the rounding of
    K - Q W^T, whose entries are of the order of one (l = 20 products)."""
    h = dh.Handle(0)
    h.scratch_trim()
    X, Q, y = problem(6500, 24, 20, labels=True)
    W = problem(6500, 24, 20, seed=1)[1]
    a = h.lra_error(X, 0.3, Q, W, y=y)
    h.close()
    h = dh.Handle(0)
    copies = 8 * 16 * 6500 * (2 + 2 * 2)
    limit(h, copies)  # and an eighth of headroom
    b = h.lra_error(X, 0.3, Q, W, y=y)
    assert h.workspace_bytes() < copies
    assert abs(a[0] - b[0]) <= 1e-13 * a[0] and abs(a[1] - b[1]) <= 1e-13 * a[1]
    h.close()


def kept_and_not(h, X, Om, q, y, prec):
    """The solve on kept K (it must have been kept) and with K formed in every pass."""
    import ctypes as C
    fn = dh._capi.lib().dh_debug_no_scratch
    fn.argtypes, fn.restype = [C.c_void_p, C.c_int], C.c_int
    h.scratch_trim()
    a = solve(h, X, Om, q, y, prec)
    size = h.scratch_bytes()
    assert size >= (8 if prec == dh.DH_PREC_F64 or X.shape[1] > 256 else 2) * X.shape[0] ** 2
    h.scratch_trim()
    fn(h.h, 1)
    try:
        b = solve(h, X, Om, q, y, prec)
        assert h.scratch_bytes() == 0
    finally:
        fn(h.h, 0)
    return a, b


@pytest.mark.parametrize("prec", ["f16", "bf16"])
@pytest.mark.parametrize("n,d,l,q", [(8192, 129, 130, 1), (8201, 200, 144, 2), (8300, 256, 280, 1),
                                     (8193, 256, 272, 1), (12037, 140, 260, 2),
                                     (8500, 256, 544, 1)])
def test_16_bit_solves_on_kept_k_return_the_fused_bits(dev, prec, n, d, l, q):
    """9 and 17 column blocks, single and paired, whole and ragged row tiles, chunks
    and columns, with labels that are not +-1."""
    import torch
    X, Om, y = problem(n, d, l, labels=True)
    a, b = kept_and_not(dev, X, Om, q, y, {"f16": dh.DH_PREC_F16, "bf16": dh.DH_PREC_BF16}[prec])
    assert torch.equal(a[0], b[0]) and torch.equal(a[1], b[1])


@pytest.mark.parametrize("prec,n,d,l,q", [("f64", 65, 8, 17, 1), ("f64", 3001, 20, 40, 1),
                                          ("f64", 2050, 64, 272, 0), ("f64", 2999, 130, 300, 1),
                                          ("f64", 301, 250, 290, 2), ("f64", 5001, 257, 33, 1),
                                          ("f64", 1501, 300, 560, 0), ("f64", 11800, 260, 5, 0),
                                          ("f16", 2000, 300, 50, 1), ("fp8", 300, 130, 140, 1),
                                          ("fp8", 2051, 256, 544, 1), ("fp8", 4099, 200, 288, 2)])
def test_solves_on_kept_k_return_the_same_bits(dev, prec, n, d, l, q):
    """Every feature width of the forming kernel, one and two column groups, odd
    sizes, triangle against row blocks above 256 features (FP64 for every
    precision there), FP8; labels that are not +-1."""
    import torch
    X, Om, y = problem(n, d, l, labels=True)
    which = {"f64": dh.DH_PREC_F64, "f16": dh.DH_PREC_F16, "fp8": dh.DH_PREC_FP8}[prec]
    a, b = kept_and_not(dev, X, Om, q, y, which)
    assert torch.equal(a[0], b[0]) and torch.equal(a[1], b[1])


@pytest.mark.parametrize("n,l,kept", [(4096, 138, False), (8192, 138, True), (8192, 272, False),
                                      (8192, 544, False), (8500, 272, True)])
def test_16_bit_solves_keep_k_where_that_pays(dev, n, l, kept):
    X, Om, _ = problem(n, 256, l)
    dev.scratch_trim()
    solve(dev, X, Om, 1, prec=dh.DH_PREC_F16)
    assert (dev.scratch_bytes() > 0) == kept


@pytest.mark.parametrize("n,d,l,q,kept", [(8192, 16, 16, 0, False), (8000, 32, 32, 1, False),
                                          (16384, 8, 20, 0, False), (8192, 16, 16, 2, True),
                                          (8192, 33, 16, 0, True), (8192, 16, 33, 0, True),
                                          (4096, 16, 16, 0, True), (10000, 16, 16, 0, True),
                                          (16384, 8, 20, 1, True), (20000, 16, 16, 0, True),
                                          (8192, 300, 16, 0, True)])
def test_f64_keeps_k_where_that_pays(dev, n, d, l, q, kept):
    """With two column blocks and up to 32 features a kept pass is no faster than a
    fused one where the grid has about one workgroup per CU (256 of them)."""
    X, Om, _ = problem(n, d, l)
    dev.scratch_trim()
    solve(dev, X, Om, q)
    assert (dev.scratch_bytes() > 0) == kept


@pytest.mark.parametrize("n,d,l,q,first", [(3000, 16, 16, 0, False), (4096, 64, 100, 1, False),
                                           (4096, 256, 16, 2, True), (2048, 16, 16, 0, True),
                                           (3000, 300, 16, 0, True), (8192, 64, 138, 1, True)])
def test_a_handles_first_solve_takes_a_buffer_where_it_alone_pays(dev, n, d, l, q, first):
    """Allocation and release of more than 64 MB take as long as a small solve gains,
    so a program with a handle per solve does without; the second solve takes it."""
    import torch
    X, Om, _ = problem(n, d, l)
    dev.scratch_trim()
    h = dh.Handle(0)
    a = solve(h, X, Om, q)
    assert (h.scratch_bytes() > 0) == first
    b = solve(h, X, Om, q)
    assert h.scratch_bytes() > 0
    assert torch.equal(a[0], b[0]) and torch.equal(a[1], b[1])
    h.close()


def test_handles_made_for_every_solve_do_not_wait_for_the_wipe(limit):
    """A handle per solve gives K's buffer back each time, and the driver wipes freed
    memory at a limited rate: buffers are taken no faster than that (25 GB/s, after
    the first eighth of the device's memory), the other solves form K in every
    pass and return the same bits."""
    import time

    import torch
    X, Om, _ = problem(20000, 16, 16)
    total = torch.cuda.get_device_properties(0).total_memory
    size, kept, t0, first = 8 * 20032 * 20000, 0, time.perf_counter(), None
    for _ in range(40):
        h = dh.Handle(0)
        h.scratch_trim()  # as the last handle's end does
        out = solve(h, X, Om, 2)
        kept += h.scratch_bytes() >= size
        h.scratch_trim()
        h.close()
        first = first or out
        assert torch.equal(out[0], first[0]) and torch.equal(out[1], first[1])
    allowed = total / 8 + 25e9 * (time.perf_counter() - t0) + 2 * size
    assert 1 <= kept and kept * size <= allowed
