"""Which launches `mxu.dot` picks, on the CPU: the library's calls are recorded, not made."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

from opentpu_amd import _lib as X                         # noqa: E402
from opentpu_amd import mxu                               # noqa: E402


@pytest.fixture
def calls(monkeypatch):
    made = []
    monkeypatch.setattr(X, "call", lambda name, *args: made.append((name,) + args))
    monkeypatch.setattr(X, "stream", lambda: None)
    monkeypatch.setattr(X, "torch", lambda: torch)
    monkeypatch.setattr(X, "dev", lambda x, dt: x)
    monkeypatch.setattr(X, "empty", lambda shape, dt: torch.empty(shape, dtype=getattr(torch, np.dtype(dt).name)))
    return made


def weight(N, K, fmt):
    from opentpu_amd.quant import row_bytes, scale_bytes
    u8 = lambda n: torch.zeros((N, n), dtype=torch.uint8)  # noqa: E731
    return mxu.QWeight(u8(row_bytes(K, fmt)), u8(scale_bytes(K, fmt)), fmt, K)


@pytest.mark.parametrize("fmt,ranges", [("int8", None), ("int4", None), ("int4", [256] * 4)])
def test_a_row_written_over_is_quantized_first(calls, fmt, ranges):
    """A launch that quantizes the row in every workgroup must not store over it: out on x, on its end, on
    its start; not out behind it."""
    K = N = 1024
    buf = torch.zeros(4 * K)
    x = buf[K:2 * K].view(1, K)
    w = weight(N, K, fmt)
    for o0, over in ((K, True), (2 * K - 4, True), (4, True), (2 * K, False), (0, False)):
        calls.clear()
        mxu.dot(x, w, out=buf[o0:o0 + N].view(1, N), ranges=ranges)
        names = [c[0] for c in calls]
        assert names[0].startswith("otpu_qact" if over else "otpu_mm_qin"), (o0, names)
