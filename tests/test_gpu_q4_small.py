"""GPU check of the Wo product for up to four sequences (q4_small_kernel) against float64:
one block to four rounds of blocks per wave (full ones and part-filled last ones), block counts
that leave waves idle, row counts off its 16-row tiles, and for each batch the largest inputs its
LDS takes (16352, 9312, 6496, 4992) beside the first that it does not. Bound: 1e-6 of the sum of |w x|, as for the other shapes."""
import numpy as np
import pytest

import pkv
from pkv import hip
from tests.test_gpu_q4 import _dequant

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("c_in,c_out,batch", [
    (32, 16, 1), (96, 50, 3), (480, 1, 2), (512, 17, 4), (4096, 2816, 1), (4096, 100, 4), (8192, 2816, 2),
    (8192, 40, 3), (16384 + 32, 30, 1), (20480, 33, 1), (4128, 2816, 3),
    (16352, 33, 1), (12320, 40, 1), (9312, 50, 2), (6496, 40, 3), (4992, 40, 4),
    (16384, 30, 1), (9344, 20, 2), (6528, 20, 3), (5024, 20, 4),
])
def test_few_sequences_within_dot_bound(gpu, c_in, c_out, batch):
    print(f"[q4 small] c_in={c_in} c_out={c_out} batch={batch}", flush=True)
    rng = np.random.default_rng(c_in + c_out + batch)
    packed = rng.integers(0, 256, (c_out, c_in // 2), dtype=np.uint8)
    scales = (rng.random((c_out, c_in // 32)) * 0.02 - 0.01).astype(np.float32)
    x = rng.standard_normal((batch, c_in)).astype(np.float32)
    dw, ds, dx = (hip.DeviceArray.from_numpy(a) for a in (packed, scales, x))
    out = hip.DeviceArray((batch, c_out), np.float32)
    out.fill_bytes_(255)
    pkv.q4_matmul(dw, ds, dx, out, c_in, c_out, batch)
    w = _dequant(packed, scales).astype(np.float64)
    want = x.astype(np.float64) @ w.T
    bound = 1e-6 * (np.abs(x.astype(np.float64)) @ np.abs(w).T)
    assert np.all(np.abs(out.numpy() - want) <= bound)
