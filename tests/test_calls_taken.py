"""Which calls the entry points take, by their host checks alone: a call that passes them fails only
at its launch (there is no device here), one that does not is refused before it."""
import os

import pytest

from opentpu_amd import _lib as X

pytestmark = pytest.mark.skipif(not os.path.exists(X.LIB_PATH) or os.path.exists("/dev/kfd"),
                                reason="a built library and no GPU (the calls' addresses are not memory)")
P = 4096                                                  # an address that passes every alignment check


def refusal(name, *args):
    """The refusal's text (OTPU_EINVAL, EALIGN, EFORMAT), or None where the checks take the call."""
    lib = X.load()
    rc = getattr(lib, name)(*args)
    return lib.otpu_last_error().decode() if rc in (-1, -2, -3) else None


def row_bytes(fmt, K):
    KB = K // 128
    return (K if fmt == "int8" else K // 2), {"int8": 4 + 4 * -(-KB // 4), "nvfp4": 16 + 8 * KB + 8 * (KB & 1)}.get(
        fmt, 8 + 4 * KB + 4 * (KB & 1))


@pytest.mark.parametrize("fmt", ["int4", "fp4", "nvfp4"])
def test_fold_takes_every_row(fmt):
    """otpu_mm_qin_fold: every K of whole 256-column chunks up to 8192, in ranges of 256 and in one."""
    for K in range(256, 8192 + 1, 256):
        rs, srs = row_bytes(fmt, K)
        for width in (256, K):
            assert refusal("otpu_mm_qin_fold", P, None, None, None, K, width, P, rs, P, srs, 8, X.FMT[fmt], 0, 0, P,
                           None) is None, K
    rs, srs = row_bytes(fmt, 8448)
    assert refusal("otpu_mm_qin_fold", P, None, None, None, 8448, 256, P, rs, P, srs, 8, X.FMT[fmt], 0, 0, P, None)
