"""The digit-per-lane block kernels of the factorization and the solves (limbforge_amd/csrc/factor_wave.hpp) at
their edges, bit for bit against the oracle: the smallest and widest precisions they take and the first one
past them, a precision whose mantissa fills whole digits (416 bits), mantissas that are all ones or a power
of two (rounding carries, exact sums), zero entries and right-hand sides, negative diagonals, exponent spreads
inside, across and past the accumulators' columns, statuses, and blocks at and around 32 rows."""
import numpy as np
import pytest

import lfcases
from factor_cases import spd

pytestmark = pytest.mark.gpu

BITS = [64, 96, 256, 416, 512, 640, 672]


def special_mantissas(rng, x, bits):
    """A fifth of the values all ones, a fifth powers of two, a fifth one unit above one."""
    w = bits // 32
    pick = rng.integers(0, 5, size=x.shape[0])
    x[pick == 0, :w] = 0xFFFFFFFF
    x[(pick == 1) | (pick == 2), :w] = 0
    x[(pick == 1) | (pick == 2), w - 1] = 0x80000000
    x[pick == 2, 0] |= 1
    return x


def triangle(rng, bits, n, span):
    L = special_mantissas(rng, lfcases.random_records(rng, bits, n * n, span), bits)
    L[rng.random(n * n) < 0.2] = lfcases.zero(bits)
    d = np.arange(n) * (n + 1)
    L[d] = special_mantissas(rng, lfcases.random_records(rng, bits, n, span // 2), bits)
    return L


@pytest.mark.parametrize("bits", BITS)
@pytest.mark.parametrize("span", [0, 30, 200, 1500])
def test_triangular_solves(capi, oracle, bits, span):
    rng = np.random.default_rng(bits + 7 * span)
    for n, nrhs, block in ((1, 1, 32), (31, 2, 32), (32, 3, 32), (33, 1, 32), (70, 5, 32), (40, 2, 7), (35, 2, 33)):
        print(f"[gpu] solve bits={bits} span={span} n={n} nrhs={nrhs} block={block}", flush=True)
        L = triangle(rng, bits, n, span)
        B = special_mantissas(rng, lfcases.random_records(rng, bits, n * nrhs, span), bits)
        B[rng.random(n * nrhs) < 0.2] = lfcases.zero(bits)
        if n == 33:  # a status in the second block, a zero on the diagonal of the first
            B[32 * nrhs, bits // 32 + 2] = 4
            L[5 * (n + 1)] = lfcases.zero(bits)
        for passes in (1, 2):
            want = oracle.solve(bits, L, n, B, nrhs, block, passes)
            got, _, _ = capi.solve(bits, passes, L, n, B, nrhs, block=block)
            bad = np.nonzero((got != want).any(axis=1))[0]
            assert bad.size == 0, f"n={n} passes={passes}: {bad.size} entries differ, first row {bad[0] // nrhs}"


@pytest.mark.parametrize("bits", BITS)
@pytest.mark.parametrize("kind", ["moderate", "graded", "wide", "banded", "spread"])
def test_factorizations(capi, oracle, bits, kind):
    """Blocks of 32, 31, 1 and 5 columns; zero entries with fill (banded), spreads past the columns (spread)."""
    rng = np.random.default_rng(3 * bits + len(kind))
    for n, block in ((1, 32), (2, 32), (31, 32), (65, 32), (33, 5)):
        print(f"[gpu] cholesky bits={bits} {kind} n={n} block={block}", flush=True)
        A = spd(oracle, rng, bits, n, kind)
        want, piv, psign, pstat = oracle.cholesky(bits, A, n, block)
        got, info = capi.cholesky(bits, A, n, block=block)
        assert (info.pivot, info.pivot_sign, info.pivot_status) == (piv, psign, pstat)
        bad = np.nonzero((got != want).any(axis=1))[0]
        assert bad.size == 0, f"n={n} block={block}: {bad.size} entries differ, first ({bad[0] // n},{bad[0] % n})"


@pytest.mark.parametrize("bits", [64, 256, 640])
def test_squares_of_short_factors(capi, oracle, bits):
    """A = L0 L0^T exactly, L0 of few-bit integers: every sum, root and quotient is exact."""
    rng = np.random.default_rng(bits)
    n, w = 34, bits // 32
    L0 = np.tril(rng.integers(-7, 8, size=(n, n)))
    L0[np.arange(n), np.arange(n)] = rng.integers(1, 9, size=n)
    V = L0 @ L0.T
    A = np.zeros((n * n, w + 3), np.uint32)
    for k, v in enumerate(V.reshape(-1)):
        if v:
            e = int(abs(v)).bit_length() - 1
            A[k, w - 1] = (int(abs(v)) << (31 - e)) & 0xFFFFFFFF
            A[k, w] = e
            A[k, w + 1] = lfcases.i32(1 if v > 0 else -1)
    want, piv, _, _ = oracle.cholesky(bits, A, n, 32)
    got, info = capi.cholesky(bits, A, n, block=32)
    assert info.pivot == piv == n
    assert (got == want).all()


@pytest.mark.parametrize("bits", [64, 256, 640, 672])
def test_sign_zero_is_zero_whatever_the_limbs(capi, oracle, bits):
    """Records of sign 0 whose limbs and exponents are not zero, in the matrix, the factor and the right-hand sides:
    each is a zero, as with zero limbs."""
    rng = np.random.default_rng(11 * bits)
    n, nrhs, block, w = 67, 3, 32, bits // 32
    A = spd(oracle, rng, bits, n, "moderate")
    i, j = np.tril_indices(n, -1)
    pick = rng.random(i.size) < 0.3
    i, j = i[pick], j[pick]
    for x, y in ((i, j), (j, i)):
        A[x * n + y] = lfcases.random_records(rng, bits, i.size, 6)
        A[x * n + y, w + 1] = 0
    d = np.arange(n) * (n + 1)
    A[d, w] = lfcases.i32(lfcases.get_exp(A[d], bits) + 8)  # diagonally dominant: positive definite whatever went to zero
    clean = A.copy()
    clean[clean[:, w + 1] == 0] = lfcases.zero(bits)
    want, piv, _, _ = oracle.cholesky(bits, clean, n, block)
    assert piv == n
    got, info = capi.cholesky(bits, A, n, block=block)
    assert info.pivot == n
    bad = np.nonzero((got != want).any(axis=1))[0]
    assert bad.size == 0, f"{bad.size} entries differ, first ({bad[0] // n},{bad[0] % n})"
    L, B = want.copy(), lfcases.random_records(rng, bits, n * nrhs, 8)
    L[i * n + j] = A[i * n + j]
    B[rng.random(n * nrhs) < 0.3, w + 1] = 0
    cl, cb = L.copy(), B.copy()
    cl[cl[:, w + 1] == 0] = lfcases.zero(bits)
    cb[cb[:, w + 1] == 0] = lfcases.zero(bits)
    for passes in (1, 2):
        want = oracle.solve(bits, cl, n, cb, nrhs, block, passes)
        got, _, _ = capi.solve(bits, passes, L, n, B, nrhs, block=block)
        bad = np.nonzero((got != want).any(axis=1))[0]
        assert bad.size == 0, f"passes={passes}: {bad.size} entries differ, first row {bad[0] // nrhs}"


@pytest.mark.parametrize("bits", [64, 256, 640])
def test_sign_zero_entry_at_every_digit_offset(capi, oracle, bits):
    """One record of sign 0 with limbs in a column whose other terms are zeros, at every offset of its mantissa in the
    26-bit digits: on some of them a block that takes its limbs for a value still decides the entry's rounding."""
    rng = np.random.default_rng(bits)
    n, w = 3, bits // 32
    A = np.stack([lfcases.zero(bits)] * (n * n))
    for i in range(n):
        A[i * n + i] = lfcases.random_records(rng, bits, 1, 0)[0]
        A[i * n + i, w + 1] = 1
    clean = A.copy()
    want, piv, _, _ = oracle.cholesky(bits, clean, n, 32)
    assert piv == n
    for e in range(-13, 13):
        A[n] = lfcases.random_records(rng, bits, 1, 0)[0]
        A[n, w], A[n, w + 1] = lfcases.i32(e), 0
        got, info = capi.cholesky(bits, A, n, block=32)
        assert info.pivot == n
        bad = np.nonzero((got != want).any(axis=1))[0]
        assert bad.size == 0, f"exponent {e}: {bad.size} entries differ, first ({bad[0] // n},{bad[0] % n})"


@pytest.mark.parametrize("bits", [64, 256, 640])
@pytest.mark.parametrize("where", ["rhs", "factor", "diagonal", "zero", "overflow", "underflow"])
def test_statuses_part_way(capi, oracle, bits, where):
    """A right-hand side's status, a factor entry's, a diagonal entry's, a zero divisor, and quotients past the exponent
    range, in the first, a middle and the last row of a block: the rows before them, those after them in the block, and
    the updates of later blocks, in columns with and without them."""
    rng = np.random.default_rng(bits + sum(map(ord, where)))
    n, nrhs, w = 70, 5, bits // 32
    for i in (0, 13, 31, 45):
        L = triangle(rng, bits, n, 30)
        B = lfcases.random_records(rng, bits, n * nrhs, 30)
        if where == "rhs":
            B[i * nrhs + 1, w + 2], B[i * nrhs + 3, w + 2] = 2, 4
        elif where == "factor":
            L[max(i, 1) * n + max(i, 1) // 2, w + 2] = 4
        elif where == "diagonal":
            L[i * (n + 1), w + 2] = 1
        elif where == "zero":
            L[i * (n + 1)] = lfcases.zero(bits)
        else:
            sign = 1 if where == "overflow" else -1
            L[i * (n + 1), w] = lfcases.i32(-sign * 600000000)
            B[i * nrhs + 2, w] = lfcases.i32(sign * 600000000)
        print(f"[gpu] solve {where} bits={bits} row {i}", flush=True)
        for passes in (1, 2):
            want = oracle.solve(bits, L, n, B, nrhs, 32, passes)
            got, _, _ = capi.solve(bits, passes, L, n, B, nrhs, block=32)
            bad = np.nonzero((got != want).any(axis=1))[0]
            assert bad.size == 0, f"row {i} passes={passes}: {bad.size} entries differ, first ({bad[0] // nrhs},{bad[0] % nrhs})"


@pytest.mark.parametrize("bits", [64, 256, 288, 640])
@pytest.mark.parametrize("diagonal", ["ones", "powers", "mixed"])
def test_pivots_that_are_powers_of_two(capi, oracle, bits, diagonal):
    """Roots that are powers of two, whose reciprocals are too: a unit diagonal (the first pivot of every such matrix), a
    diagonal matrix of powers of four and of two (every pivot, every other one), and such blocks beside general ones."""
    rng = np.random.default_rng(bits + len(diagonal))
    n, w = 67, bits // 32
    A = np.stack([lfcases.zero(bits)] * (n * n))
    for i in range(n):
        e = 0 if diagonal == "ones" else int(rng.integers(-9, 10))
        A[i * n + i] = lfcases.one(bits, e)
        for j in range(i):
            if diagonal == "ones" or (diagonal == "mixed" and i >= 32 and rng.random() < 0.3):
                x = lfcases.random_records(rng, bits, 1, 0)[0]
                x[w] = lfcases.i32(-22 - int(rng.integers(0, 9)))
                A[i * n + j] = A[j * n + i] = x
    want, piv, _, _ = oracle.cholesky(bits, A, n, 32)
    got, info = capi.cholesky(bits, A, n, block=32)
    assert info.pivot == piv == n
    bad = np.nonzero((got != want).any(axis=1))[0]
    assert bad.size == 0, f"{bad.size} entries differ, first ({bad[0] // n},{bad[0] % n})"


@pytest.mark.parametrize("bits", [b for b in range(64, 641, 32) if b not in BITS])
def test_every_width(capi, oracle, bits):
    """The widths between those above: the digit counts, the room of the columns and the pivot's iteration differ at each."""
    rng = np.random.default_rng(17 * bits)
    n, nrhs, block = 40, 3, 32
    for kind in ("moderate", "spread"):
        A = spd(oracle, rng, bits, n, kind)
        want, piv, psign, pstat = oracle.cholesky(bits, A, n, block)
        got, info = capi.cholesky(bits, A, n, block=block)
        assert (info.pivot, info.pivot_sign, info.pivot_status) == (piv, psign, pstat)
        assert (got == want).all(), kind
    for span in (30, 600):
        L = triangle(rng, bits, n, span)
        B = special_mantissas(rng, lfcases.random_records(rng, bits, n * nrhs, span), bits)
        for passes in (1, 2):
            got, _, _ = capi.solve(bits, passes, L, n, B, nrhs, block=block)
            assert (got == oracle.solve(bits, L, n, B, nrhs, block, passes)).all(), f"span={span} passes={passes}"


def hard_pivots(rng, bits, count):
    """Positive records whose roots and reciprocals lie at the edges of their roundings: all ones and one unit less, powers
    of two and one unit more, squares of short and of long mantissas, and the values nearest to squares halfway between
    two mantissas."""
    w, out = bits // 32, []
    for i in range(count):
        kind, e, full = i % 7, int(rng.integers(-3, 4)), 1 << (bits - 1)
        long = full | int.from_bytes(rng.bytes(bits // 8), "little") >> 1
        if kind < 4:
            m = (2 * full - 1, 2 * full - 2, full, full + 1)[kind]
        else:
            root = (int(rng.integers(3, 1 << 16)), long >> (bits // 2) << (bits // 2), 2 * long + 1)[kind - 4]
            square = root * root
            shift = square.bit_length() - bits
            m = square << -shift if shift <= 0 else (square + (1 << (shift - 1))) >> shift
            if m >> bits:
                m, shift = m >> 1, shift + 1
            e = 2 * (e // 2) + (square.bit_length() - 1) % 2  # an exponent of the square's parity
        x = lfcases.one(bits, e)
        x[:w] = [(m >> (32 * k)) & 0xFFFFFFFF for k in range(w)]
        out.append(x)
    return np.stack(out)


@pytest.mark.parametrize("bits", range(64, 641, 32))
def test_pivots_at_the_edges_of_their_roundings(capi, oracle, bits):
    """Two blocks of such pivots with nothing between them, and rows below that each pivot's reciprocal divides."""
    rng = np.random.default_rng(bits)
    n, k, w = 70, 64, bits // 32
    A = np.stack([lfcases.zero(bits)] * (n * n))
    A[np.arange(k) * (n + 1)] = hard_pivots(rng, bits, k)
    for i in range(k, n):
        A[i * (n + 1)] = lfcases.one(bits, 24)
        row = special_mantissas(rng, lfcases.random_records(rng, bits, k, 3), bits)
        for j in range(k):
            A[i * n + j] = A[j * n + i] = row[j]
    want, piv, _, _ = oracle.cholesky(bits, A, n, 32)
    got, info = capi.cholesky(bits, A, n, block=32)
    assert info.pivot == piv == n
    bad = np.nonzero((got != want).any(axis=1))[0]
    assert bad.size == 0, f"{bad.size} entries differ, first ({bad[0] // n},{bad[0] % n})"
