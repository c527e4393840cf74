"""The column division (limbforge_amd/csrc/div_core.hpp) bit for bit against the oracle where it can go wrong:
quotients within a unit of 2^-32N of halfway (which Knuth's division decides), exact quotients, mantissas all ones
and powers of two, quotients at a binade's ends, exponent limits, zeros and statuses, outputs on their operands, at
the smallest and largest widths and where 26-bit digits fill a mantissa exactly (416 bits)."""
import numpy as np
import pytest

import lfcases

pytestmark = pytest.mark.gpu

BITS = [64, 96, 256, 416, 544, 992, 1024]


def to_int(r, bits):
    return sum(int(r[i]) << (32 * i) for i in range(bits // 32))


def division_cases(rng, bits, count):
    a, b = lfcases.binary_cases(rng, bits, count)
    for x in (a, b):
        pick = rng.integers(0, 8, size=count)
        w = bits // 32
        x[pick == 0, :w] = 0xFFFFFFFF
        x[(pick == 1) | (pick == 2), :w] = 0
        x[(pick == 1) | (pick == 2), w - 1] = 0x80000000
        x[pick == 2, 0] |= 1
    for k in range(0, count, 5):
        B = to_int(b[k], bits)
        if not B:
            continue
        Q = (1 << (bits - 1)) | int.from_bytes(rng.bytes(bits // 8), "little") >> 1
        if k % 2:   # a / b next to the midpoint above Q
            A = B * (2 * Q + 1)
        else:       # a / b next to Q itself
            A = B * Q
        A = (A >> (A.bit_length() - bits)) + int(rng.integers(-1, 2))
        if A.bit_length() != bits:
            continue
        a[k, :bits // 32] = [(A >> (32 * i)) & 0xFFFFFFFF for i in range(bits // 32)]
        a[k, bits // 32 + 2] = 0
        a[k, bits // 32 + 1] = 1
    return a, b


@pytest.mark.parametrize("bits", BITS)
def test_division(capi, oracle, bits):
    rng = np.random.default_rng(bits)
    a, b = division_cases(rng, bits, 1337)
    want = oracle.elementwise(bits, capi.OPS["div"], a, b, b)
    got, _, _ = capi.run_host(bits, "div", a, b)
    bad = np.nonzero((got != want).any(axis=1))[0]
    assert bad.size == 0, f"{bad.size} quotients differ, first {bad[:8].tolist()}"
    # in place over either operand, resident
    for over in (0, 1):
        A, B = capi.Buffer(bits, len(a)), capi.Buffer(bits, len(a))
        A.upload(a)
        B.upload(b)
        capi.elementwise(bits, "div", A, B, None, (A, B)[over])
        assert ((A, B)[over].download() == want).all()


@pytest.mark.parametrize("bits", [64, 256, 416, 1024])
def test_complex_division(capi, oracle, bits):
    rng = np.random.default_rng(7 * bits)
    n = 700
    re, d = division_cases(rng, bits, n)
    im, e = division_cases(rng, bits, n)
    e[::2] = lfcases.zero(bits)  # half of the divisors real: |y|^2 = d^2, quotients next to halfway stay rare but exact ones do not
    x, y = np.concatenate([re, im], axis=1), np.concatenate([d, e], axis=1)
    want = oracle.elementwise(bits, capi.OPS["complex_div"], x, y, y)
    got, _, _ = capi.run_host(bits, "complex_div", x, y)
    bad = np.nonzero((got != want).any(axis=1))[0]
    assert bad.size == 0, f"{bad.size} quotients differ, first {bad[:8].tolist()}"
