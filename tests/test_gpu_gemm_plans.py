"""Exact products at the edges of their plans, every output against the oracle: lines run by their bands or joined
into one band each (whichever the planner's cost rule takes), extended rows that are the lines themselves or a
list (zero, status and fallback lines in between), operands whose lines are adjacent in memory or whose entries
are, shapes around the digit kernel's 32 and 256 entries and the product's 128 x 128 tiles, and the widest and
narrowest precisions."""
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
