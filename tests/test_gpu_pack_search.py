"""The 4-bit weight packers' search where it can go wrong, against the float64 oracle bit for bit
(`opentpu/quant.py:325-400`): equal errors and quotients on a midpoint (values on half-steps of one
scale), multipliers that coincide, magnitudes at both ends of fp32, rows of less than a wave's
sub-blocks, of exactly that many and of more, and rows that are not 16-byte aligned."""
import warnings

import numpy as np
import pytest

from oracle import formats as Q

pytestmark = pytest.mark.gpu


def weights(K):
    rng = np.random.default_rng(K)
    W = np.empty((40, K), np.float32)
    W[0:8] = rng.standard_normal((8, K))
    W[8:12] = rng.standard_normal((4, K)) * np.exp(rng.uniform(-6, 6, (4, K // 32))).repeat(32, 1)
    W[12:18] = rng.integers(-14, 15, (6, K)) * 0.5            # half-steps: ties and exact zeros
    W[18:24] = rng.integers(-24, 25, (6, K)) * 0.25 * np.exp2(rng.integers(-9, 9, (6, K // 16))).repeat(16, 1)
    W[24:28] = rng.standard_normal((4, K)) * 1e-38            # subnormals
    W[28:30] = rng.integers(-3, 4, (2, K)) * np.float32(1e-45)
    W[30:32] = np.clip(rng.standard_normal((2, K)) * 1e38, -3e38, 3e38)
    W[32:36] = (rng.random((4, K)) < 0.04) * rng.standard_normal((4, K))     # most groups nearly empty
    W[36] = 0
    W[37] = 1
    W[38:40] = np.sign(rng.standard_normal((2, K))) * 7 + (rng.random((2, K)) < 0.1) * 0.5
    return W


@pytest.mark.parametrize("fmt", ["int4", "fp4", "nvfp4"])
@pytest.mark.parametrize("K,ldw", [(128, 128), (384, 385), (1024, 1024), (2048, 2048), (2176, 2179), (4224, 4224)])
def test_packer_search(fmt, K, ldw):
    from opentpu_amd import _lib as X
    from opentpu_amd.quant import row_bytes, scale_bytes
    W = weights(K)
    N, rb, sb = len(W), row_bytes(K, fmt), max(8, scale_bytes(K, fmt, False))
    Wp = np.zeros((N, ldw), np.float32)
    Wp[:, :K] = W
    print("packer search", fmt, K, ldw, flush=True)
    Wd, rows, srows = X.dev(Wp, np.float32), X.empty((N, rb), np.uint8), X.empty((N, sb), np.uint8)
    X.call("otpu_pack_x4", X.ptr(Wd), N, K, ldw, X.FMT[fmt], X.ptr(rows), rb, X.ptr(srows), sb, X.stream())
    with warnings.catch_warnings():
        warnings.simplefilter("ignore", RuntimeWarning)       # the subnormal rows' quotients
        r0, s0 = Q.pack_nv(W) if fmt == "nvfp4" else Q.pack_x4(W, fmt)
    r, s = X.host(rows), X.host(srows)
    bad = np.flatnonzero((r != r0).any(1) | (s != s0).any(1))
    assert not len(bad), bad
