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


def operand(M, K, ranges, sa_rows=None):
    R = len(ranges) if sa_rows is None else sa_rows
    return torch.zeros((M, K), dtype=torch.int8), torch.zeros((R, M)), torch.zeros((M, K // 32), dtype=torch.uint8), ranges


@pytest.mark.parametrize("M", [1, 6])
def test_an_operand_is_read_no_further_than_it_goes(calls, M):
    """Ranges over a part of the operand's columns, and scales that are not a row a range, run a launch a
    range: otpu_mm_dot takes its ranges from K, and a scale a range and row."""
    w = weight(64, 1024, "int4")
    for ranges in ([256], [256, 256], [512]):
        calls.clear()
        mxu.dot(operand(M, 1024, ranges), w)
        assert [c[0] for c in calls] == ["otpu_mm"] * len(ranges), ranges
        assert [c[7] for c in calls] == ranges
    q, Sa, da, rg = operand(M, 1024, [256] * 4)
    for S in (list(Sa), Sa.t().contiguous().t(), Sa.repeat(1, 2)[:, :M]) + ((Sa[:, 0],) if M == 1 else ()):
        calls.clear()
        mxu.dot((q, S, da, rg), w)
        want = ["otpu_mm_dot"] if isinstance(S, torch.Tensor) and S.dim() == 2 and S.is_contiguous() else ["otpu_mm"] * 4
        assert [c[0] for c in calls] == want
    calls.clear()
    with pytest.raises(IndexError):
        mxu.dot(operand(M, 1024, [256] * 4, sa_rows=3), w)
    assert "otpu_mm_dot" not in [c[0] for c in calls]


@pytest.mark.parametrize("shape", [(1024,), (1, 1024, 1024), (2, 1024, 3)])
def test_rows_are_a_matrix(calls, shape):
    with pytest.raises(ValueError):
        mxu.dot(torch.zeros(shape), weight(64, 1024, "int4"))
    assert not calls


@pytest.mark.parametrize("M,fmt,widths", [(1, "int8", [256] * 4), (1, "int4", [512, 256, 256]), (3, "int4", [256] * 4)])
def test_ranges_are_read_once(calls, M, fmt, widths):
    """Any iterable of widths, as a list of them."""
    made = []
    for ranges in (widths, tuple(widths), iter(widths)):
        calls.clear()
        mxu.dot(torch.zeros((M, 1024)), weight(64, 1024, fmt), ranges=ranges)
        made.append([c[0] for c in calls])
    assert made[0] == made[1] == made[2] and made[0]
