"""CPU check of the append kernels' test for the mean of squares (csrc/append.hpp mean_is_settled).

The reference sums x_i^2 (x bf16, 256 values) in double, left to right, and rounds the mean to float
(src/ref/ops.cpp:79-90). The kernels sum in tree orders and keep the tree's mean when
float(m - m 2^-43) == float(m + m 2^-43). This test sums vectors with wide exponent spans in the two
kernels' orders and requires: where the test admits the tree's sum, its rounded mean is the
left-to-right one's, bit for bit; a mean on a rounding boundary is not admitted; and N(0,1) rows are."""
import numpy as np

from util import bf16_bits_to_f32, f32_to_bf16_bits


def tree_sum(x):
    """One row per wave: 4 values per lane in order, then the cross-lane steps (lane ^ 1, lane ^ 2, the mirrors
    within 8 and 16 lanes, lane ^ 16, lane ^ 32)."""
    part = [sum(float(x[4 * l + e]) ** 2 for e in range(4)) for l in range(64)]
    for p in (lambda l: l ^ 1, lambda l: l ^ 2, lambda l: (l & ~7) | (7 - (l & 7)), lambda l: (l & ~15) | (15 - (l & 15)),
              lambda l: l ^ 16, lambda l: l ^ 32):
        part = [part[l] + part[p(l)] for l in range(64)]
    assert len(set(part)) == 1
    return part[0]


def sum16(x):
    """Four rows per wave: 16 values per lane in order, then the steps within 16 lanes."""
    part = []
    for l in range(16):
        t = 0.0
        for e in range(16):
            t += float(x[16 * l + e]) ** 2
        part.append(t)
    for p in (lambda l: l ^ 1, lambda l: l ^ 2, lambda l: (l & ~7) | (7 - (l & 7)), lambda l: 15 - l):
        part = [part[l] + part[p(l)] for l in range(16)]
    assert len(set(part)) == 1
    return part[0]


def settled(s):
    m = s / 256.0
    return np.float32(m - m * 2.0 ** -43) == np.float32(m + m * 2.0 ** -43)


def boundary_row(rng):
    """Squares that sum to 256 + 2^-16, i.e. a mean half way between two floats, in random order, with
    a few tiny elements whose squares get lost in some orders of summing and not in others."""
    x = np.zeros(256)
    x[:245] = 1.0
    x[245] = 3.0
    x[246] = np.sqrt(2.0 ** -16)
    x[247:249] = 1.0
    x[249:256] = 2.0 ** -23  # squares of 2^-46: seven of them stay below an ulp of 256
    rng.shuffle(x)
    return x


def test_mean_criterion():
    rng = np.random.default_rng(11)
    admitted = 0
    for trial in range(1500):
        if trial % 3 == 0:
            x = boundary_row(rng)
        else:
            x = rng.normal(0, 1, 256) * np.exp2(rng.integers(-40, 6, 256) * (rng.random(256) < 0.1))
        x = bf16_bits_to_f32(f32_to_bf16_bits(x.astype(np.float32))).astype(np.float64)
        seq = 0.0
        for v in x:
            seq = seq + v * v
        for s in (tree_sum(x), sum16(x)):
            if settled(s):
                admitted += 1
                assert np.float32(s / 256.0) == np.float32(seq / 256.0), trial
            if trial % 3 == 0:
                assert not settled(s), "a mean on a rounding boundary"
    assert admitted > 1900  # (the 1,000 random rows, either order)
