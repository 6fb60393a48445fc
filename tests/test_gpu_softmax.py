"""Row softmax over the widths at which its kernel changes form."""

import numpy as np
import pytest

from test_gpu_kernels import dev

pytestmark = pytest.mark.gpu


# one unit, fewer than four, remainders of a lane's four, the widest row that is held in registers, and wider
@pytest.mark.parametrize("stride", [1, 3, 1023, 4098, 27278, 32768, 32769])
def test_softmax(pkg, dsx, rng, stride):
    z = (rng.standard_normal((5, stride)) * 4).astype(np.float32)
    d = dev(pkg, z)
    pkg.check(dsx.dsx_activation(d.ptr, 5, stride, 7, None))
    e = np.exp(z.astype(np.float64) - z.max(axis=1, keepdims=True))
    want = e / e.sum(axis=1, keepdims=True)
    # arguments of exp within 40, rounded once and scaled once (2 x 40 x 2^-24), exp itself 2 ulp, sums of 33 and 16 terms in turn and 10
    # halvings, three more roundings: 150 x 2^-24 = 9e-6, of every unit
    assert (np.abs(d.numpy() - want) <= 9e-6 * want + 1e-38).all()


# the widest row of every form and the next one, in numbers of rows that do and do not fill the last workgroup
@pytest.mark.parametrize("rows", [1, 4, 7])
@pytest.mark.parametrize("stride", [2, 5, 256, 257, 511, 512, 513, 1024, 1025, 2047, 2048, 2049, 4096, 4097, 8192, 8193, 16384, 16385])
def test_forms(pkg, dsx, rng, rows, stride):
    z = (rng.standard_normal((rows + 1, stride)) * 4).astype(np.float32)
    z[0, stride // 2] = -np.inf
    d = dev(pkg, z)
    pkg.check(dsx.dsx_activation(d.ptr, rows, stride, 7, None))
    got = d.numpy()
    assert np.array_equal(got[rows], z[rows])      # (the row behind them)
    e = np.exp(z[:rows].astype(np.float64) - z[:rows].max(axis=1, keepdims=True))
    want = e / e.sum(axis=1, keepdims=True)
    # as above; no lane adds more than 32 units in turn
    assert (np.abs(got[:rows] - want) <= 9e-6 * want + 1e-38).all()


def test_many_narrow_rows(pkg, dsx):
    """A row of 100 units takes a wavefront and not sixteen: 16,384 of them cost less than ten times what another activation does (296 us against 5
    when every row had a workgroup of 1,024 lanes)."""
    import time
    d = pkg.DeviceArray((16384, 100), np.float32)
    took = {}
    for act in (1, 7):
        times = []
        for _ in range(9):
            pkg.check(dsx.dsx_sync())
            t = time.perf_counter()
            for _ in range(20):
                pkg.check(dsx.dsx_activation(d.ptr, 16384, 100, act, None))
            pkg.check(dsx.dsx_sync())
            times.append(time.perf_counter() - t)
        took[act] = sorted(times)[4]
    assert took[7] < 10 * took[1]
