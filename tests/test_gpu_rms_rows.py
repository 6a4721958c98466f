"""rmsnorm over many short rows (a wave per row): every width's edge, the last
workgroup partly filled, in place, and a row whose mean sits on an f32
rounding boundary, which takes the sequential replay. Bit for bit."""
import numpy as np
import pytest

import oracle as O
import uq
from uq import ops
from test_gpu_ops import assert_bitwise

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows", [1024, 1031])
@pytest.mark.parametrize("n", [1, 63, 64, 65, 127, 128])
def test_rmsnorm_many_short_rows(n, rows):
    rng = np.random.default_rng(n + rows)
    X = (rng.standard_normal((rows, n)) * rng.choice([1e-3, 1.0, 40.0], (rows, n))).astype(np.float32)
    X[1] = 0.0
    if n == 128:  # mean 2^-5 (1 + 2^-24), the midpoint of two f32 values
        X[rows - 1] = 0.0
        X[rows - 1, 124:] = [1.0, 1.0, 1.0, np.nextafter(np.float32(1.0), np.float32(2.0))]
    w = rng.standard_normal(n).astype(np.float32)
    d, dw = uq.DeviceArray.from_numpy(X), uq.DeviceArray.from_numpy(w)
    ops.rmsnorm_d(d, d, dw, n, rows, 1e-6)
    uq.synchronize()
    got = d.download(np.float32, rows * n).reshape(rows, n)
    for r in [0, 1, 2, 3, 4, 5, rows // 2, rows - 2, rows - 1]:
        assert_bitwise(got[r], O.rmsnorm(X[r], w, 1e-6), f"rmsnorm n={n} row {r}")
