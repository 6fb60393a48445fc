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
