"""Exact products at the edges of their plans, every output against the oracle: lines run by their bands or joined
into one band each (whichever the planner's cost rule takes), extended rows that are the lines themselves or a
list (zero, status and fallback lines in between), operands whose lines are adjacent in memory or whose entries
are, shapes around the digit kernel's 32 and 256 entries and the product's 128 x 128 tiles, and the widest and
narrowest precisions."""
import ctypes as C
import threading

import numpy as np
import pytest

import lfcases

pytestmark = pytest.mark.gpu


def entries(rng, bits, count, kind):
    x = lfcases.random_records(rng, bits, count, 0)
    w = bits // 32
    if kind == "single":
        e = rng.integers(-20, 21, size=count)
    elif kind == "bands":  # three bands a line: joined where lines are many
        e = 200 * rng.integers(-1, 2, size=count) + rng.integers(-9, 10, size=count)
    elif kind == "rare":   # a second band on a few lines only
        e = np.where(rng.random(count) < 0.003, -150, 0) + rng.integers(-15, 16, size=count)
    else:                  # "edge": spreads at max_spread, all-ones mantissas
        e = rng.choice([-256, 0, 256], size=count)
        x[:, :w] = 0xFFFFFFFF
    x[:, w] = lfcases.i32(e)
    x[rng.random(count) < 0.1] = lfcases.zero(bits)
    return x


@pytest.mark.parametrize("bits", [64, 256, 544, 1024])
@pytest.mark.parametrize("kind", ["single", "bands", "rare", "edge"])
@pytest.mark.parametrize("m,n,k", [(1, 1, 1), (5, 129, 33), (130, 3, 65), (17, 16, 257), (33, 40, 128)])
def test_products(capi, oracle, bits, kind, m, n, k):
    print(f"[gpu] product bits={bits} {kind} {m}x{n}x{k}", flush=True)
    rng = np.random.default_rng(bits + 13 * m + 7 * n + k)
    A, B = entries(rng, bits, m * k, kind), entries(rng, bits, k * n, kind)
    if m > 4:
        A[2 * k:3 * k] = lfcases.zero(bits)     # a zero line
        A[4 * k, bits // 32 + 2] = 2            # a status line
    if n > 10 and kind == "rare":
        B[7, bits // 32] = lfcases.i32(-5000)   # a line past max_spread
    want = oracle.gemm(bits, False, A, B, m, n, k)
    got, _, _, _ = capi.gemm(bits, False, A, B, m, n, k)
    assert (got == want).all()
    At = np.ascontiguousarray(A.reshape(m, k, -1).transpose(1, 0, 2)).reshape(k * m, -1)
    got, _, _, _ = capi.gemm(bits, True, At, B, m, n, k)
    assert (got == want).all()
    C0 = lfcases.random_records(rng, bits, m * n, 100)
    got, _, _, _ = capi.gemm(bits, False, A, B, m, n, k, C_in=C0, subtract=True)
    assert (got == oracle.gemm(bits, False, A, B, m, n, k, C0, True)).all()


@pytest.mark.parametrize("bits", [96, 512])
@pytest.mark.parametrize("kind", ["single", "bands", "rare"])
@pytest.mark.parametrize("rows,cols", [(1, 2), (40, 17), (130, 131)])
def test_symmetric_products(capi, oracle, bits, kind, rows, cols):
    rng = np.random.default_rng(bits + rows)
    A = entries(rng, bits, rows * cols, kind)
    want = oracle.syrk(bits, A, rows, cols, lower_only=False)
    full, _, _, _ = capi.syrk(bits, A, rows, cols, lower_only=False)
    assert (full == want).all()
    lower, _, _, _ = capi.syrk(bits, A, rows, cols, lower_only=True)
    keep = np.tril(np.ones((cols, cols), bool)).reshape(-1)
    assert (lower[keep] == want[keep]).all()


def on_a_thread(call):
    """Runs `call` on a thread of its own, whose planner buffers go back to the device with it."""
    failed = []

    def run():
        try:
            call()
        except Exception as e:  # noqa: BLE001
            failed.append(e)

    t = threading.Thread(target=run)
    t.start()
    t.join()
    assert failed == []


def free_memory(capi):
    free, total = C.c_size_t(), C.c_size_t()
    assert capi.lib().hipMemGetInfo(C.byref(free), C.byref(total)) == 0  # the HIP runtime that the library is linked with
    return free.value


def test_joined_plan_that_does_not_fit_gives_way_to_the_bands(capi, oracle):
    """A product whose few lines of two bands make the joined plan the cheaper one and the larger one, with device memory
    left for the band plan alone: the outputs are those of the joined plan, and the oracle's in a few rows."""
    bits, m, k = 64, 9000, 32
    rng = np.random.default_rng(5)
    A, B = entries(rng, bits, m * k, "rare"), entries(rng, bits, k * m, "rare")

    a, b, c = capi.Buffer(bits, m * k), capi.Buffer(bits, k * m), capi.Buffer(bits, m * m)
    a.upload(A)
    b.upload(B)
    on_a_thread(lambda: capi.gemm_resident(bits, False, a, b, m, m, k, c))
    want = c.download()

    def side(x, lines_first):  # lines in tiles, bands in tiles, widest line (every band is at most 30 wide)
        e = lfcases.get_exp(x, bits).reshape((m, k) if lines_first else (k, m))
        e = np.where((lfcases.get_sign(x, bits) != 0).reshape(e.shape), e, 10**6)
        e = e if lines_first else e.T
        high, low = (abs(e) <= 20).any(axis=1), (e < -100).any(axis=1)
        return -(-m // 128) * 128, -(-int(high.sum() + low.sum()) // 128) * 128, int(max(r[r < 10**5].max() - r.min() for r in e))

    (jr, br, wa), (jc, bc, wb) = side(A, True), side(B, False)
    digits_residues = lambda width, rows, cols: ((135 + 2 * width) // 16 + 1) * (2 * rows * cols + 2 * 64 * (rows + cols))  # noqa: E731
    joined, bands = digits_residues(max(wa, wb), jr, jc), digits_residues(30, br, bc) + 2**30  # (and their CRT stage)
    assert joined > bands + 2**29
    c.upload(np.zeros_like(want))
    fill = capi.DeviceMemory(free_memory(capi) - (joined + bands) // 2)
    print(f"[gpu] joined {joined / 2**30:.2f} GiB, bands {bands / 2**30:.2f} GiB, left {free_memory(capi) / 2**30:.2f} GiB", flush=True)
    try:
        on_a_thread(lambda: capi.gemm_resident(bits, False, a, b, m, m, k, c))
    finally:
        fill.free()
    got = c.download()
    assert np.array_equal(got, want)
    for i in (0, 17, m - 1):
        assert (got[i * m:(i + 1) * m] == oracle.gemm(bits, False, A[i * k:(i + 1) * k], B, 1, m, k)).all(), f"row {i}"


@pytest.mark.parametrize("bits", [64, 512])
@pytest.mark.parametrize("m,n,k", [(30000, 3, 5), (3, 30000, 5), (66001, 1, 3), (257, 256, 2), (640, 75, 4)])
def test_outputs_in_row_order_whatever_the_rows_length(capi, oracle, bits, m, n, k):
    """Workgroups of 64 and of 256 consecutive outputs over rows of 1, 3, 75, 256 and 30,000."""
    rng = np.random.default_rng(bits + m)
    A, B = entries(rng, bits, m * k, "single"), entries(rng, bits, k * n, "single")
    if m > 4:
        A[2 * k:3 * k] = lfcases.zero(bits)
        A[4 * k, bits // 32 + 2] = 2
    got, _, _, _ = capi.gemm(bits, False, A, B, m, n, k)
    assert (got == oracle.gemm(bits, False, A, B, m, n, k)).all()


@pytest.mark.parametrize("cols", [63, 200, 300])
def test_symmetric_outputs_in_row_order(capi, oracle, cols):
    """Workgroups that cross the diagonal, lie above it, or hold the end of one row and the start of the next."""
    bits, rows = 96, 5
    A = entries(np.random.default_rng(cols), bits, rows * cols, "single")
    want = oracle.syrk(bits, A, rows, cols, lower_only=False)
    full, _, _, _ = capi.syrk(bits, A, rows, cols, lower_only=False)
    assert (full == want).all()
    lower, _, _, _ = capi.syrk(bits, A, rows, cols, lower_only=True)
    keep = np.tril(np.ones((cols, cols), bool)).reshape(-1)
    assert (lower[keep] == want[keep]).all()


def test_more_rows_than_a_launch_has_workgroups_of_one(capi):
    """2^24 rows of one output: with a workgroup of 256 a row, more threads than a launch can have.  K = 1, so the
    product is the element-wise one with a broadcast factor."""
    bits, m = 64, 1 << 24
    rng = np.random.default_rng(3)
    A, B = lfcases.random_records(rng, bits, m, 9), lfcases.random_records(rng, bits, 1, 9)
    a, b, c, want = capi.Buffer(bits, m), capi.Buffer(bits, 1), capi.Buffer(bits, m), capi.Buffer(bits, m)
    a.upload(A)
    b.upload(B)
    on_a_thread(lambda: capi.gemm_resident(bits, False, a, b, m, 1, 1, c))  # (60 GB of buffers)
    capi.elementwise(bits, "mul", a, b, None, want, b_index=(1, 1))
    assert np.array_equal(c.download(), want.download())


@pytest.mark.parametrize("bits", [64, 544, 1024])
@pytest.mark.parametrize("width", [534, 539, 541, 542, 600])
def test_bands_around_the_widest_of_the_crt_classes(capi, oracle, bits, width):
    """Lines of one band as wide as the wider CRT class holds (542 bits less those of the terms), below it and past it."""
    rng = np.random.default_rng(bits + width)
    m, n = 5, 7
    for k in (2, 3):
        A, B = lfcases.random_records(rng, bits, m * k, 0), lfcases.random_records(rng, bits, k * n, 0)
        A[:, bits // 32] = lfcases.i32(np.where(np.arange(m * k) % k == 0, 0, -width))
        B[:, bits // 32] = lfcases.i32(np.where(np.arange(k * n) // n == k - 1, 0, -width))
        got, _, _, _ = capi.gemm(bits, False, A, B, m, n, k, options=capi.LinalgOptions.default(band_bits=1024, max_spread=8192))
        assert (got == oracle.gemm(bits, False, A, B, m, n, k)).all(), k
