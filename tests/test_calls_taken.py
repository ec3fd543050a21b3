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


def dot_refusal(fmt, M, K, width, *, ldq=None, ldda=None, rs=None, srs=None, k0=0, flags=0):
    r, sr = row_bytes(fmt, K + 128 * k0)
    return refusal("otpu_mm_dot", P, K if ldq is None else ldq, P, P, K // 32 if ldda is None else ldda, M, K, width, P,
                   r if rs is None else rs, P, sr if srs is None else srs, 8, X.FMT[fmt], flags, k0, 0, None, P, 8, None)


@pytest.mark.parametrize("fmt", ["int8", "int4", "nvfp4"])
def test_mm_dot_checks_a_range(fmt):
    """otpu_mm_dot over more columns than one MM takes: a range's columns are checked, the strides and the
    last range's scale blocks against the whole row."""
    K = 40960
    r, sr = row_bytes(fmt, K)
    for M in (1, 8, 300):
        assert dot_refusal(fmt, M, K, 5120) is None
        assert dot_refusal(fmt, M, K, 5120, k0=2) is None
        assert "at most" in dot_refusal(fmt, M, K, K)
        assert dot_refusal(fmt, M, K, 5120, ldq=K - 16)
        assert dot_refusal(fmt, M, K, 5120, ldda=K // 32 - 4)
        assert dot_refusal(fmt, M, K, 5120, rs=r - 16)
        assert dot_refusal(fmt, M, K, 5120, srs=sr - 16)
        assert dot_refusal(fmt, M, K, 5120, k0=-1)
        assert dot_refusal(fmt, M, K, 5120, srs=8 if fmt != "nvfp4" else 16)
        if fmt != "nvfp4":                                # (plain rows: a scale a row, no blocks)
            assert dot_refusal(fmt, M, K, 5120, srs=8, flags=X.RSC) is None
