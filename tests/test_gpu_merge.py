"""GPU parity of the merge of many pieces per sequence (stream_merge_many_kernel: few sequences
over the whole chip) against the oracle: a sequence in fewer pieces than one round of requests,
a few rounds, and more pieces than a workgroup has threads, in double and float partials.
Tolerances: tests/parity.py."""
import numpy as np
import pytest

from pkv import BF16, F32
from tests.test_gpu_attend import _batched_case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("geom,ctx,kv_dtype", [
    ((16, 8, 256), [511], F32), ((16, 8, 256), [40], F32), ((16, 2, 512), [8000], F32),
    ((16, 2, 512), [3000, 17, 2500], F32), ((16, 2, 512), [6000], BF16), ((2, 1, 256), [30000], BF16),
    ((2, 1, 256), [20000, 100], F32),
])
def test_many_pieces(gpu, geom, ctx, kv_dtype):
    print(f"[merge] {geom} contexts {ctx} {kv_dtype}", flush=True)
    rng = np.random.default_rng(sum(ctx))
    _batched_case(rng, len(ctx), 1, np.array(ctx), *geom, 16, 0, kv_dtype, 0.0625)
