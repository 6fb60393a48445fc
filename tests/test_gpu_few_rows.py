"""Dense layers of few rows or few output tiles (fc_rows_kernel) against float64, at the edges of its tiles and of its dispatch."""
import ctypes as C

import numpy as np
import pytest

from parity import assert_close

pytestmark = pytest.mark.gpu

# (batch, k, n): one row, one block of 32 and one row more, two blocks, the last batch that takes this kernel; k below one chunk of
# eight, no multiple of it, split and not; n a multiple of 4, of 2, odd, one column past a tile, narrow layers on both splits
SHAPES = [(1, 128, 27278), (8, 500, 8191), (32, 37, 4096), (33, 64, 4225), (64, 7, 5002), (65, 600, 4100), (128, 512, 4099),
          (5, 40, 300001), (3, 24, 263000), (40, 256, 262148), (1, 1024, 1024), (70, 300, 130), (256, 77, 1000), (17, 33, 1), (9, 2000, 63)]


@pytest.mark.parametrize("batch,k,n", SHAPES)
@pytest.mark.parametrize("accumulate", [0, 1])
def test_few_rows_layer(pkg, dsx, rng, batch, k, n, accumulate):
    print("[case] few rows batch=%d k=%d n=%d accumulate=%d" % (batch, k, n, accumulate), flush=True)
    pitch = k + 3                                             # rows of X at every alignment
    X = rng.standard_normal((batch, pitch), dtype=np.float32)
    W = rng.standard_normal((k, n), dtype=np.float32) * np.float32(1.0 / np.sqrt(k))
    bias = rng.standard_normal(n, dtype=np.float32)
    Z0 = rng.standard_normal((batch, n + 5), dtype=np.float32)
    dX, dW, db, Z = (pkg.DeviceArray.from_numpy(a) for a in (X, W, bias, Z0))
    params = pkg.ActParams(0.2, 1.5, 1.05)
    act = 1 if accumulate else 0
    pkg.check(dsx.dsx_fc_forward(dX.ptr, pitch, dW.ptr, 0, db.ptr, Z.ptr, n + 5, batch, k, n, accumulate, act, C.byref(params)))
    got = Z.numpy()
    x = X[:, :k].astype(np.float64) @ W.astype(np.float64) + bias + (Z0[:, :n] if accumulate else 0.0)
    want = np.tanh(x) if accumulate else 1.0 / (1.0 + np.exp(-x))
    # k products of unit variance / k summed in fp32: about sqrt(k) roundings of 2^-24 each on sums of size 1, far below 1e-5; the
    # activations' slopes are at most 1
    assert_close(got[:, :n], want, "few rows", rel=1e-5, abs_floor=1.0)
    assert np.array_equal(got[:, n:], Z0[:, n:])              # nothing written past n


@pytest.mark.parametrize("batch,k,n", [(1, 128, 27278), (8, 64, 8192), (33, 96, 8229), (64, 16, 33000), (3, 32, 263001), (100, 512, 8200)])
def test_few_rows_segment_maxima(pkg, dsx, rng, batch, k, n):
    print("[case] few rows maxima batch=%d k=%d n=%d" % (batch, k, n), flush=True)
    X = rng.standard_normal((batch, k), dtype=np.float32)
    W = rng.standard_normal((k, n), dtype=np.float32) * np.float32(1.0 / np.sqrt(k))
    W[:, n // 2] = np.nan                                     # a NaN score is no maximum
    nseg = (n + 63) // 64
    dX, dW, Z = pkg.DeviceArray.from_numpy(X), pkg.DeviceArray.from_numpy(W), pkg.DeviceArray((batch, n), np.float32)
    sm = pkg.DeviceArray.from_numpy(np.full((batch, nseg), 7.0, dtype=np.float32))
    sw = C.c_uint32(0)
    pkg.check(dsx.dsx_fc_forward_segmax(dX.ptr, k, dW.ptr, 0, None, Z.ptr, n, batch, k, n, 3, None, sm.ptr, C.byref(sw)))
    assert sw.value == 64
    z = np.full((batch, nseg * 64), -np.inf, dtype=np.float32)
    z[:, :n] = np.nan_to_num(Z.numpy(), nan=-np.inf)
    assert np.array_equal(sm.numpy(), z.reshape(batch, nseg, 64).max(axis=2))
