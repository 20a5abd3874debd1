"""Calls of more numbers than one dispatch can give a workgroup each (2^32
threads: 2^26 one-wavefront workgroups, 2^25 of two).  Nearly every number is
even, so a test of it ends at once."""
import numpy as np
import pytest

import hipmem
import pgap

pytestmark = pytest.mark.gpu

STRIDE = 1 << 22  # workgroups of a matrix-core launch at most (kernels.h)


# a bound of 2300 bits is too wide for one lane per number, and strong Lucas
# runs on the matrix cores at any width
@pytest.mark.parametrize("kind,bases,rows,bits", [(pgap.FERMAT2, (), (1 << 26) + 3, 2300),
                                                  (pgap.SPRP, (2,), (1 << 26) + 3, 2300),
                                                  (pgap.LUCAS, (), (1 << 25) + 3, 64)])
def test_batch(engine, kind, bases, rows, bits):
    n = np.zeros(rows, dtype=np.uint32)
    n[4::1 << 20] = 1 << 20
    primes = [1, STRIDE - 1, STRIDE, 3 * STRIDE + 7, rows - 2, rows - 1]
    n[primes] = (1 << 31) - 1
    n[STRIDE + 1] = 341 * 7  # composite
    d_n = hipmem.DeviceArray.from_host(n)
    d_o = hipmem.DeviceArray(rows, np.uint8)
    engine.prp_device(d_n.ptr, 1, rows, d_o.ptr, kind, bases, bits)
    engine.sync()
    assert engine.last_launch().matrix_tests == rows
    assert np.nonzero(d_o.to_host())[0].tolist() == primes


def test_mixed(engine):
    rows = (1 << 26) + 3
    even, prime = (1 << 2299) + 2, (1 << 2203) - 1
    words = np.concatenate([pgap.to_limbs([even], 72)[0], pgap.to_limbs([prime], 69)[0]])
    offset = np.zeros(rows, dtype=np.uint64)
    limbs = np.full(rows, 72, dtype=np.uint32)
    primes = [0, STRIDE, STRIDE + 5, rows - 1]
    offset[primes], limbs[primes] = 72, 69
    got = engine.prp_mixed_packed(words, offset, limbs)
    assert engine.last_launch().matrix_tests == rows
    assert np.nonzero(got)[0].tolist() == primes
