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


def names(calls):
    return [c[0][5:] for c in calls]


@pytest.mark.skipif(not __import__("os").path.exists(X.LIB_PATH), reason="libotpu_amd.so not built")
@pytest.mark.parametrize("fmt,N,K,width,want", [
    ("int4", 4096, 1024, None, ["mm_qin"]), ("int4", 16384, 4096, None, ["qact", "mm_dot"]),
    ("int8", 4096, 4096, None, ["mm_qin"]), ("int8", 64, 6400, None, ["qact", "mm_dot"]),
    ("int8", 64, 8448, None, ["mm_qin"]), ("int8", 12288, 12288, None, ["qact", "mm_dot"]),
    ("nvfp4", 64, 16384, None, ["mm_qin"]), ("nvfp4", 64, 16640, None, ["qact", "mm_dot"]),
    ("int4", 64, 384, None, ["qact", "mm_dot"]),          # (an odd block count: half a chunk)
    ("int4", 1024, 3072, 256, ["mm_qin_fold"]), ("int4", 8448, 8192, 256, ["qact_ranges", "mm_dot"]),
    ("int4", 64, 8448, 256, ["qact_ranges", "mm_dot"]), ("int4", 64, 8448, 768, ["qact_ranges", "mm_ranges"]),
    ("int4", 2048, 6144, 768, ["mm_qin_fold"]), ("int4", 4096, 6144, 768, ["qact_ranges", "mm_ranges"]),
    ("int4", 64, 1024, 128, ["qact_ranges"] + ["mm"] * 8), ("int8", 64, 1024, 128, ["qact_ranges", "mm_dot"]),
    ("int4", 4096, 6144, None, ["mm_qin"]), ("int4", 4104, 6144, None, ["qact", "mm_dot"]),
    ("int4", 20000, 2048, None, ["mm_qin"]), ("int4", 32800, 2048, None, ["qact", "mm_dot"]),
    ("int8", 64, 10240, 1280, ["qact_ranges", "mm_ranges"]), ("int8", 64, 8192, 1024, ["qact_ranges", "mm_dot"]),
    ("int8", 20000, 512, 256, ["qact_ranges", "mm_ranges"]), ("int8", 19999, 512, 256, ["qact_ranges", "mm_dot"])])
def test_one_rows_launches(calls, fmt, N, K, width, want):
    mxu.dot(torch.zeros((1, K)), weight(N, K, fmt), ranges=None if width is None else [width] * (K // width))
    assert names(calls) == want


@pytest.mark.parametrize("M,fmt,N,want", [(2, "int4", 12287, "mm_dot"), (2, "int8", 20000, "mm_ranges"), (2, "int8", 19999, "mm_dot"), (3, "int4", 12288, "mm_dot"),
                                          (4, "nvfp4", 24576, "mm_ranges"), (4, "int8", 24576, "mm_dot"), (5, "int4", 24576, "mm_dot")])
def test_few_rows_launches_in_ranges(calls, M, fmt, N, want):
    w = weight(N, 512, fmt)
    for x in (torch.zeros((M, 512)), operand(M, 512, [256, 256])):
        calls.clear()
        mxu.dot(x, w, ranges=[256, 256])
        assert names(calls)[-1] == want
        calls.clear()
        mxu.dot(x, w, ranges=[256, 256], acc=torch.zeros((M, N)))
        assert names(calls)[-1] == want
    u = mxu.QWeight(w.rows, None, fmt, 512)               # (ASCALE: otpu_mm_ranges has none)
    mxu.dot(torch.zeros((M, 512)), u, ranges=[256, 256], acc=torch.zeros((M, N)), acc_scale=torch.zeros(M))
    assert names(calls)[-1] == "mm_dot"


@pytest.mark.parametrize("fmt", ["int8", "int4"])
def test_an_operands_mode_picks_the_kernel(calls, fmt):
    """quantize_ranges' operand says whether its offsets are one; parts put together by hand say nothing."""
    w = weight(64, 512, fmt)
    for row in (True, False):
        op = mxu.quantize_ranges(torch.zeros((6, 512)), None, row)
        assert isinstance(op, tuple) and len(op) == 4 and op[3] == [512]
        for x, act in ((op, X.ACT_ROW if row else X.ACT_ANY if fmt == "int8" else X.ACT_MX), (tuple(op), X.ACT_ANY),
                       (op[:3] + ([512],), X.ACT_ANY)):
            calls.clear()
            mxu.dot(x, w)
            assert names(calls) == ["mm_dot"] and calls[0][17] == act


@pytest.mark.parametrize("K,want", [(1 << 19, "mm_ranges"), (3 << 19, "mm_dot")])
def test_a_workspace_of_ranges_is_bounded(calls, K, want):
    """A row a range of fp32 for one row on 20000 weight rows: 164 MB over 2048 ranges, 492 MB over 6144."""
    w = mxu.QWeight(torch.empty((20000, 1), dtype=torch.uint8), torch.empty((20000, 1), dtype=torch.uint8), "int4", K)
    mxu.dot(torch.empty((1, K)), w, ranges=[256] * (K // 256))
    assert names(calls) == ["qact_ranges", want]
