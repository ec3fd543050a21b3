"""QACT of the common form (groups of 32 or ROW mode) over the sizes where its kernel changes: ranges a
wave or a workgroup holds in registers, 1 to 8 chunks a lane, and past them, against the oracle bit
for bit (`opentpu/fp32.py:321-343`), with zero rows, zero groups, NaN and infinite values."""
import numpy as np
import pytest

from conftest import same_bits
from oracle import fp32 as F

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("row_mode", [False, True])
@pytest.mark.parametrize("M,K,width", [(1, 32, 32), (3, 96, 96), (5, 512, 512), (5, 544, 544), (1100, 544, 544), (2, 1056, 1056),
                                       (1030, 2048, 2048), (1, 2080, 2080), (3, 4128, 4128), (2, 8192, 8192), (2, 8224, 8224),
                                       (7, 1280, 256), (260, 3072, 768), (2, 6144, 3072)])
def test_qact_sizes(M, K, width, row_mode):
    from opentpu_amd import _lib as X
    rng = np.random.default_rng(M + K)
    x = (rng.standard_normal((M, K)) * np.exp(rng.uniform(-3, 3, (M, K // 32, 1))).repeat(32, 2).reshape(M, K)).astype(np.float32)
    x[-1, :32] = 0                                        # a zero group, a zero row, special values
    if M > 2:
        x[1] = 0
        x[0, 5], x[0, 40] = np.nan, 1e-40
    print("qact sizes", M, K, width, row_mode, flush=True)
    R = K // width
    xd = X.dev(x, np.float32)
    q, S, d = X.empty((M, K), np.int8), X.empty((R, M), np.float32), X.empty((M, K // 32), np.uint8)
    X.call("otpu_qact_ranges", X.ptr(xd), None, M, K, K, width, 32, X.Q_ROW if row_mode else 0, None, None, X.ptr(q), K,
           X.ptr(S), X.ptr(d), K // 32, X.stream())
    for r in range(R):
        w = slice(r * width, (r + 1) * width)
        qo, So, do = F.quantize_mx(np.ascontiguousarray(x[:, w]), 32, row_mode=row_mode)
        assert np.array_equal(X.host(q)[:, w], qo)
        assert same_bits(X.host(S)[r], So)
        assert np.array_equal(X.host(d)[:, w.start // 32:w.stop // 32], do)
