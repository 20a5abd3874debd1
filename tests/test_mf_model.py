"""CPU model of the matrix-core Montgomery squaring (csrc/mont_mf.h): numbers of
balanced bytes, 16 x 16 x 64 byte products whose A and B operands are shifted
copies of the factors, q = -x^2 N^-1 mod R from the low tiles, (x^2 + q N) / R
from the high tiles with everything below word LW - 1 dropped and a rounding
there.  At each width and in both fragment layouts the model's tiles give the
integers' own x^2 mod R and (x^2 + q N) / R, for random N and x and for the
largest ones (N just below R / 2^16 and x = +-40 N, bytes of -128), no tile leaves
32 bits, a word's carry stays below the bias of 2^18 and the result below 0.62 N
(for |x| <= N below 0.51 N)."""
import random

import numpy as np
import pytest

PAD = 64


class Layout:
    def __init__(self, KB):
        self.KB = KB
        self.shared = KB in (3, 9)
        self.LW = 16 * KB + 1 if self.shared else 16 * KB - 1
        self.HB = (16 * KB if KB < 4 else KB // 4 * 64) if self.shared else self.LW - 1
        self.HOFF = -15 if self.shared else -1
        self.T = (self.LW + 63) // 64
        self.UMAX = self.LW // 16
        self.UH = (self.HB - self.HOFF - 15) // 16
        self.NB = (self.LW + 14) // 16 + 1
        self.NBH = (self.LW - 1 - self.HOFF) // 16 + 1
        self.R = 1 << (32 * self.LW)

    def balanced(self, x):
        """x mod R as balanced bytes."""
        flip = sum(0x80808080 << (32 * i) for i in range(self.LW))
        u = ((x + flip) % self.R).to_bytes(4 * self.LW, "little")
        return (np.frombuffer(u, dtype=np.uint8) ^ 0x80).astype(np.int8).astype(np.int64)

    def buffer(self, digits):
        a = np.zeros(4 * (PAD + 16 * self.KB + 64), dtype=np.int64)
        a[4 * PAD:4 * PAD + 4 * self.LW] = digits
        return a

    def a_fragment(self, buf, u):
        """A[row][k]: lane 16 h + row holds k = 16 h + 4 e + i."""
        if not -3 <= u <= self.UMAX:
            return None
        row, k = np.meshgrid(np.arange(16), np.arange(64), indexing="ij")
        h, e, i = k // 16, k // 4 % 4, k % 4
        byte = 4 * (15 + 16 * u + 16 * (row // 4) - 4 * h - e) + row % 4 - i
        return buf[4 * PAD + byte]

    def b_fragment(self, buf, first):
        k, col = np.meshgrid(np.arange(64), np.arange(16), indexing="ij")
        return buf[4 * (PAD + first + col + 4 * (k // 16) + k // 4 % 4) + k % 4]

    def tile(self, a, b, blocks, first, u0):
        d = np.zeros((16, 16), dtype=np.int64)
        for c in range(blocks):
            f = self.a_fragment(a, u0 - c)
            if f is not None:
                d += f @ self.b_fragment(b, 16 * c + first)
        assert np.abs(d).max() < 1 << 31
        cols = np.zeros(256, dtype=np.int64)
        for row in range(16):
            cols[64 * (row // 4) + row % 4 + 4 * np.arange(16)] = d[row]
        return cols

    def low(self, a, b):
        return np.concatenate([self.tile(a, b, self.NB, -15, 4 * q) for q in range(self.T)])

    def high(self, a, b):
        return np.concatenate([self.tile(a, b, self.NBH, self.HOFF, self.UH + 4 * q) for q in range(self.T)])


def words(cols):
    """Column sums of each word, as integers."""
    return [sum(int(v) << (8 * i) for i, v in enumerate(w)) for w in cols.reshape(-1, 4)]


def value(ws):
    return sum(w << (32 * i) for i, w in enumerate(ws))


def square(L, x, N):
    ni = pow(N, -1, L.R)
    xb, nb, ib = (L.buffer(L.balanced(v)) for v in (x, N, ni))
    low = L.low(xb, xb)
    if L.shared and L.HB % 64 == 0:  # the first high tile is this low tile
        assert (L.high(xb, xb)[:256] == low[256 * (L.HB // 64):256 * (L.HB // 64) + 256]).all()
    t = value(words(low)[:L.LW]) % L.R
    assert t == x * x % L.R
    qb = L.balanced(-value(words(L.low(ib, L.buffer(L.balanced(t))))[:L.LW]))
    q = value(words(qb))
    assert (x * x + q * N) % L.R == 0
    sums = words(L.high(xb, xb) + L.high(nb, L.buffer(qb)))
    assert max(abs(w) for w in sums) >> 32 < 1 << 18
    y = (value(sums[L.LW - 1 - L.HB:]) + (1 << 31)) >> 32
    assert y == (x * x + q * N) // L.R
    return y


@pytest.mark.parametrize("KB", range(1, 10))
def test_squaring(KB):
    L, rng = Layout(KB), random.Random(KB)
    bits = 32 * L.LW - 16
    for top in (bits, bits - 480 if KB > 1 else bits - 100):
        N = rng.getrandbits(top) | 1 | 1 << (top - 1)
        y = square(L, rng.randrange(-N, N), N)
        assert 100 * abs(y) <= 51 * N
    N = (1 << bits) - 1
    for x in (N, -N, 40 * N, -40 * N, value([-0x80808080] * (L.LW - 1)) % (40 * N)):
        y = square(L, x, N)
        assert 100 * abs(y) <= 62 * N
