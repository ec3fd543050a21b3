"""MM of several activation rows on the MFMA kernels -- the batch kernel (csrc/batch_impl.h), the
prefill kernel (csrc/prefill_impl.h) and the GEMMs with the prefill walk inside them -- and
otpu_mm_dot's ranges, against the C oracle bit for bit (`opentpu/isasim.py:749-910`,
`opentpu/compiler.py:2686-2720`).  Sizes at the edges of tiles, of the K splits and of the rules
that pick a kernel; offsets inside and outside the kernels' int32 windows."""
import numpy as np
import pytest

from conftest import same_bits
from oracle import cpu as OC
from oracle import fp32 as F
from oracle import mm as MM
from test_gpu_gemm4 import CASES as GEMM4_CASES
from test_gpu_gemm4 import activations, say, weights

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def X():
    import torch
    assert torch.cuda.is_available(), "GPU tests need a GPU"
    from opentpu_amd import _lib
    _lib.load()
    return _lib


def mm_dot(X, q, Sa, da, rows, srows, fmt, K, width, flags=0, k0=0, act=0, old=None, alpha=None, N=None):
    M, N = q.shape[0], rows.shape[0] if N is None else N
    qd, Sd, dd = X.dev(q, np.int8), X.dev(Sa, np.float32), X.dev(da, np.uint8)
    w, ws = X.dev(rows, np.uint8), X.dev(srows, np.uint8)
    al = X.dev(alpha, np.float32) if alpha is not None else None
    out = X.empty((M, N), np.float32) if old is None else X.dev(old, np.float32).clone()
    X.call("otpu_mm_dot", X.ptr(qd), K, X.ptr(Sd), X.ptr(dd), K // 32, M, K, width, X.ptr(w), w.shape[1], X.ptr(ws),
           ws.shape[1], N, X.FMT[fmt], flags, k0, act, X.ptr(al), X.ptr(out), N, X.stream())
    return X.host(out)


def int8_weights(rng, N, K, wk):
    from oracle import formats as Q
    W = rng.standard_normal((N, K)).astype(np.float32) * 0.02
    if wk == "spread":                                    # block offsets over several octaves
        W *= np.exp2(-rng.integers(0, 7, (N, K // 128))).repeat(128, 1).astype(np.float32)
    if wk == "far":                                       # ... past every window
        W *= np.exp2(-rng.integers(0, 20, (N, K // 128))).repeat(128, 1).astype(np.float32)
    return Q.pack_rsc(W) if wk == "rsc" else Q.pack_int8x(W)


def operands(rng, M, N, K, fmt, wk, ak, k0=0):
    q, Sa, da = activations(rng, M, K, ak)
    if fmt == "int8":
        rows, srows = int8_weights(rng, N, K + 128 * k0, wk)
        rows = np.ascontiguousarray(rows[:, 128 * k0:])
    else:
        rows, srows = weights(rng, N, K, fmt, wk, k0)
    return q, Sa, da, rows, srows, {"rsc": MM.RSC, "unit": MM.UNIT}.get(wk, 0)


WIN = (0, 3, 6, 8)                                        # offsets up to and past the block windows
KINDS = [("int8", "x8", "mx"), ("int8", "spread", "mx"), ("int8", "far", WIN), ("int8", "rsc", (0, 20)),
         ("int4", "x4", "mx"), ("int4", "spread", WIN), ("int4", "rsc", "mx"), ("fp4", "wide", "mx"),
         ("fp4", "x4", (2, 5, 9)), ("nvfp4", "x4", "mx"), ("nvfp4", "tiny", WIN), ("nvfp4", "unit", "mx"),
         ("nvfp4", "wider", "wide")]


@pytest.mark.parametrize("M,N,K", [(5, 1, 128), (16, 100, 1024), (17, 257, 384), (33, 1000, 2048), (50, 2500, 256)])
@pytest.mark.parametrize("fmt,wk,ak", KINDS)
def test_batch(X, M, N, K, fmt, wk, ak):
    from opentpu_amd import mxu
    rng = np.random.default_rng(M + N + K)
    q, Sa, da, rows, srows, fl = operands(rng, M, N, K, fmt, wk, ak)
    say("batch", M, N, K, fmt, wk, ak)
    got = mxu.mm(q, Sa, da, rows, srows, fmt, K, rsc=wk == "rsc", unit=wk == "unit")
    assert same_bits(got, OC.mm(q, Sa, da, rows, srows, fmt, K, flags=fl))


@pytest.mark.parametrize("M,N,K,act", [(100, 8100, 256, 2), (500, 8100, 384, 2), (500, 8100, 384, 0), (129, 26000, 128, 1)])
@pytest.mark.parametrize("fmt,wk,ak", KINDS + [("int8", "rsc", "mx"), ("int8", "rsc", WIN), ("int8", "x8", "row"),
                                               ("fp4", "x4", "row"), ("nvfp4", "x4", "row")])
def test_prefill(X, M, N, K, act, fmt, wk, ak):
    """The prefill kernel (32 and 64 rows a tile), and 4-bit weights on the GEMM where offsets are unknown."""
    rng = np.random.default_rng(M + N + K)
    q, Sa, da, rows, srows, fl = operands(rng, M, N, K, fmt, wk, ak)
    say("prefill", M, N, K, act, fmt, wk, ak)
    got = mm_dot(X, q, Sa, da, rows, srows, fmt, K, K, fl, act=act)
    assert same_bits(got, OC.mm(q, Sa, da, rows, srows, fmt, K, flags=fl))


@pytest.mark.parametrize("M,N,K,act", [(500, 8100, 2048, 0), (300, 8100, 2048, 1), (129, 16200, 2048, 1)])
@pytest.mark.parametrize("fmt,wk,ak", [("int8", "rsc", "row"), ("int8", "rsc", "mx"), ("int8", "unit", (0, 3)), ("int8", "rsc", (0, 20)),
                                       ("int4", "x4", "row"), ("int4", "spread", WIN), ("int4", "rsc", "row"), ("fp4", "x4", "row"),
                                       ("fp4", "wide", "mx"), ("nvfp4", "x4", "row"), ("nvfp4", "tiny", "mx")])
def test_gemm_ragged_tiles(X, M, N, K, act, fmt, wk, ak):
    """Calls the rule sends to the 128 x 128 GEMMs (their offsets unknown, or said to be one), whose last tiles
    end inside; activations of any offsets (the walk in the GEMMs)."""
    rng = np.random.default_rng(M + N)
    q, Sa, da, rows, srows, fl = operands(rng, M, 60, K, fmt, wk, ak)
    say("gemm ragged", M, N, K, act, fmt, wk, ak)
    rep = lambda a: np.resize(a, (N, a.shape[1]))  # noqa: E731
    got = mm_dot(X, q, Sa, da, rep(rows), rep(srows), fmt, K, K, fl, act=act)
    want = OC.mm(q, Sa, da, rows, srows, fmt, K, flags=fl)
    assert same_bits(got, want[:, np.arange(N) % 60])


GEMM_KINDS = [c for c in GEMM4_CASES] + [(0, 0, K, "int8", wk, ak, 0) for K, wk, ak in [
    (1024, "rsc", "row"), (640, "unit", "row"), (128, "rsc", "row"), (4096, "rsc", "mx"), (8192, "rsc", "mx"), (6144, "rsc", "row"),
    (256, "rsc", "row"), (128, "unit", "mx"), (1024, "rsc", (0, 1)), (1024, "rsc", (0, 1, 2)), (1024, "rsc", (1, 3, 4)),
    (1024, "rsc", (0, 20)), (1024, "rsc", (2, 5, 17)), (1024, "unit", (0, 31)), (4096, "rsc", (0, 1)), (4224, "rsc", (0, 2)),
    (8192, "rsc", (1,)), (512, "rsc", (20, 30)), (2048, "unit", "wide")]]


@pytest.mark.parametrize("M0,N0,K,fmt,wk,ak,k0", GEMM_KINDS)
def test_gemm_kinds(X, M0, N0, K, fmt, wk, ak, k0):
    """The kinds of weights, offsets and K of the small GEMM cases (test_gpu_gemm4.py, test_gpu_parity.py: so few
    rows and columns run the batch kernel) at sizes that the rule sends to the GEMMs: a round of 128 x 128 tiles
    where the prefill kernel has three or four, the call saying that its offsets are one, which picks a kernel and
    changes no bit.  One row tile (its rows ending inside it unless K is short), or four."""
    M, N = ((128 if K < 512 else 100), 31990) if K <= 2048 else (500, 8190)
    rng = np.random.default_rng(K + len(wk))
    q, Sa, da = activations(rng, M, K, ak)
    if fmt == "int8":
        rows, srows = int8_weights(rng, 60, K, "rsc")
    else:
        rows, srows = weights(rng, 60, K, fmt, wk, k0)
    fl = {"rsc": MM.RSC, "unit": MM.UNIT}.get(wk, 0)
    rep = lambda a: np.resize(a, (N, a.shape[1]))  # noqa: E731
    idx = np.arange(N) % 60
    say("gemm kinds", M, N, K, fmt, wk, ak, k0)
    got = mm_dot(X, q, Sa, da, rep(rows), rep(srows), fmt, K, K, fl, k0=k0, act=1)
    assert same_bits(got, OC.mm(q, Sa, da, rows, srows, fmt, K, flags=fl, k0=k0)[:, idx])
    if K in (512, 640, 1024):                             # onto old values
        old = rng.standard_normal((M, 60)).astype(np.float32)
        got = mm_dot(X, q, Sa, da, rep(rows), rep(srows), fmt, K, K, fl | MM.ACC, k0=k0, act=1, old=np.ascontiguousarray(old[:, idx]))
        assert same_bits(got, OC.mm(q, Sa, da, rows, srows, fmt, K, flags=fl | MM.ACC, k0=k0, old=old)[:, idx])


@pytest.mark.parametrize("M,N,K", [(5, 18305, 2048), (6, 20480, 4096), (7, 18305, 2048), (5, 18305, 2304), (16, 20000, 256), (17, 18400, 256),
                                   (8, 20481, 4096), (6, 32769, 2048), (8, 32770, 2048), (6, 8193, 4096), (5, 8192, 4096), (5, 18305, 512),
                                   (6, 18305, 1024), (5, 18305, 6144), (16, 30720, 1024), (9, 30721, 1024), (16, 16385, 1536), (10, 49152, 3072),
                                   (6, 45056, 2048), (8, 10240, 2048), (6, 32900, 1024)])
@pytest.mark.parametrize("fmt,wk,ak", [("int8", "rsc", "mx"), ("int8", "spread", "mx"), ("int4", "x4", "mx"), ("nvfp4", "x4", WIN)])
def test_few_rows_on_many_weights(X, M, N, K, fmt, wk, ak):
    """Both sides of the lines between the GEMV, the batch and the prefill kernel, onto old values."""
    rng = np.random.default_rng(M + K)
    q, Sa, da, rows, srows, fl = operands(rng, M, 60, K, fmt, wk, ak)
    old = rng.standard_normal((M, 60)).astype(np.float32)
    idx = np.arange(N) % 60
    rep = lambda a: np.resize(a, (N, a.shape[1]))  # noqa: E731
    say("few rows", M, N, K, fmt, wk, ak)
    got = mm_dot(X, q, Sa, da, rep(rows), rep(srows), fmt, K, K, fl | MM.ACC, act=2, old=np.ascontiguousarray(old[:, idx]))
    assert same_bits(got, OC.mm(q, Sa, da, rows, srows, fmt, K, flags=fl | MM.ACC, old=old)[:, idx])


@pytest.mark.parametrize("fmt,lo,hi", [("int4", 0x88, 0x77), ("nvfp4", 0xFF, 0x77)])
def test_prefill_largest_products(X, fmt, lo, hi):
    """Group products at the ends of their range: activations -128 and 127 (any int8 may come as an
    operand) on the largest weights of either sign, offsets 0 and 2."""
    M, N, K = 100, 8100, 256
    rng = np.random.default_rng(3)
    _, _, _, rows, srows, _ = operands(rng, 1, N, K, fmt, "x4", "mx")
    rows = rows.copy()
    rows[0::2], rows[1::2] = lo, hi
    q = np.where(np.arange(M) % 2, 127, -128).astype(np.int8)[:, None].repeat(K, 1)
    Sa = np.full(M, 0.01, np.float32)
    da = np.zeros((M, K // 32), np.uint8)
    da[::3, ::2] = 2
    say("prefill largest products", fmt)
    got = mm_dot(X, q, Sa, da, rows, srows, fmt, K, K, act=2)
    cut = np.ascontiguousarray
    assert same_bits(got[:, :40], OC.mm(q, Sa, da, cut(rows[:40]), cut(srows[:40]), fmt, K))


@pytest.mark.parametrize("fmt,K,sd,M,N", [("int8", 256, 9, 100, 8100), ("int8", 512, 8, 520, 8200), ("int4", 16768, 1, 100, 8100),
                                          ("fp4", 11136, 1, 100, 8100), ("nvfp4", 23424, 2, 100, 8100)])
def test_prefill_sums_of_lowest_values(X, fmt, K, sd, M, N):
    """Activations of -128 on the largest weights and multipliers, one row at offset 0 beside rows at
    sd: the block sums a count of 127 a value would let past 2^31 (int8 2 * 4 * 32 * 128 * 128 * 2^9)."""
    KB = K // 128
    byte = {"int8": 0x80, "int4": 0x88, "fp4": 0xFF, "nvfp4": 0xFF}[fmt]
    rows = np.full((N, KB * (128 if fmt == "int8" else 64)), byte, np.uint8)
    one = np.ones((N, 1), np.float32).view(np.uint8)
    if fmt == "int8":
        srows = one
    elif fmt == "nvfp4":                                  # E 15, m 15: the largest multiplier, offset 0
        srows = np.concatenate([one, np.zeros((N, 12), np.uint8), np.full((N, 8 * KB + 8 * (KB & 1)), 0x7F, np.uint8)], 1)
    else:
        word = np.full((N, KB + (KB & 1)), sum(63 << (8 + 6 * b) for b in range(4)), np.uint32)
        srows = np.concatenate([one, np.zeros((N, 4), np.uint8), word.view(np.uint8).reshape(N, -1)], 1)
    q = np.full((M, K), -128, np.int8)
    q[3::5] = 127
    da = np.full((M, K // 32), sd, np.uint8)
    da[::7] = 0
    Sa = np.ones(M, np.float32)
    fl = MM.RSC if fmt == "int8" else 0
    say("prefill lowest values", fmt, K)
    got = mm_dot(X, q, Sa, da, rows, srows, fmt, K, K, fl, act=2)
    cut = np.ascontiguousarray
    assert same_bits(got[:, :40], OC.mm(q, Sa, da, cut(rows[:40]), cut(srows[:40]), fmt, K, flags=fl))
    assert same_bits(got[:, N - 8:], OC.mm(q, Sa, da, cut(rows[N - 8:]), cut(srows[N - 8:]), fmt, K, flags=fl))


@pytest.mark.parametrize("K,top", [(2048, 6), (4096, 5), (1024, 7), (2048, 5)])
def test_gemm_sums_of_lowest_values(X, K, top):
    """The int8 GEMM's two planes (offsets 0 and top a tile) of -128s: K 128^2 2^top reaches 2^31 (the last
    case half of it: the planes take it)."""
    M, N = 512, 8192
    rows = np.full((N, K), 0x80, np.uint8)
    rows[1::2] = 0x7F
    srows = np.ones((N, 1), np.float32).view(np.uint8)
    q = np.full((M, K), -128, np.int8)
    da = np.zeros((M, K // 32), np.uint8)
    da[5::64] = top
    Sa = np.ones(M, np.float32)
    say("gemm lowest values", K, top)
    got = mm_dot(X, q, Sa, da, rows, srows, "int8", K, K, MM.RSC, act=0)
    cut = np.ascontiguousarray
    assert same_bits(got[:, 1000:1020], OC.mm(q, Sa, da, cut(rows[1000:1020]), cut(srows[1000:1020]), "int8", K, flags=MM.RSC))


@pytest.mark.parametrize("fmt", ["int8", "int4", "nvfp4"])
def test_prefill_long_sums(X, fmt):
    """Sums that leave int32 inside the walk: every product at its largest over K = 16384."""
    rng = np.random.default_rng(3)
    M, N, K = 512, 8192, 16384
    _, _, _, rows, srows, _ = operands(rng, 1, N, 256, fmt, "x8" if fmt == "int8" else "x4", "mx")
    rep = K // 256
    rows = np.tile(rows, (1, rep))
    rows[:] = {"int8": 0x7F, "int4": 0x77, "nvfp4": 0x77}[fmt]
    KB = K // 128
    if fmt == "int8":
        srows = np.concatenate([srows[:, :4], np.zeros((N, KB), np.uint8)], 1)
    elif fmt == "int4":
        word = np.full((N, KB), sum(63 << (8 + 6 * b) for b in range(4)), np.uint32)
        srows = np.concatenate([srows[:, :4], np.zeros((N, 4), np.uint8), word.view(np.uint8).reshape(N, 4 * KB)], 1)
    else:
        srows = np.concatenate([srows[:, :16], np.full((N, 8 * KB), 0x7F, np.uint8)], 1)
    q = np.full((M, K), 127, np.int8)
    q[1::2] = -127
    da = rng.integers(0, 3, (M, K // 32)).astype(np.uint8)
    Sa = np.ones(M, np.float32)
    say("prefill long", fmt)
    got = mm_dot(X, q, Sa, da, rows, srows, fmt, K, K, act=2)
    rows_s, srows_s = np.ascontiguousarray(rows[:40]), np.ascontiguousarray(srows[:40])
    assert same_bits(got[:, :40], OC.mm(q, Sa, da, rows_s, srows_s, fmt, K))


@pytest.mark.parametrize("M,N", [(1, 300), (4, 70), (5, 1024), (40, 999), (200, 12000), (257, 17000)])
@pytest.mark.parametrize("fmt,K,width", [("int8", 1152, 384), ("int8", 1536, 128), ("int4", 768, 256), ("fp4", 3072, 256),
                                         ("nvfp4", 1536, 768)])
def test_dot_ranges(X, M, N, fmt, K, width):
    """A QACT range per MM, the MMs' outputs added in range order; ACC's old values first."""
    rng = np.random.default_rng(M + N + K)
    if M * N * K > 2e9:
        N = int(2e9 / M / K) // 8 * 8 + 3
    R = K // width
    _, _, _, rows, srows, _ = operands(rng, 1, N, K, fmt, "spread", "mx")
    x = (rng.standard_normal((M, K)) * rng.standard_normal((M, K))).astype(np.float32)
    parts = [F.quantize_mx(x[:, r * width:(r + 1) * width], 32) for r in range(R)]
    q, da = np.concatenate([p[0] for p in parts], 1), np.concatenate([p[2] for p in parts], 1)
    Sa = np.stack([p[1] for p in parts])
    old = rng.standard_normal((M, N)).astype(np.float32)
    say("dot ranges", M, N, fmt, K, width)
    bpb = 128 if fmt == "int8" else 64
    for flags, want in ((0, None), (MM.ACC, old)):
        got = mm_dot(X, q, Sa, da, rows, srows, fmt, K, width, flags, act=2, old=None if want is None else old)
        for r in range(R):
            kb = r * width // 128
            rw = np.ascontiguousarray(rows[:, kb * bpb:(kb + width // 128) * bpb])
            f = 0 if want is None else MM.ACC
            want = OC.mm(np.ascontiguousarray(parts[r][0]), parts[r][1], parts[r][2], rw, srows, fmt, width, flags=f, k0=kb, old=want)
        assert same_bits(got, want)


@pytest.mark.parametrize("M,N", [(20, 200), (200, 12000)])
def test_rows_acc_ascale_k0(X, M, N):
    from opentpu_amd import mxu
    rng = np.random.default_rng(M)
    K = 256
    q, Sa, da, rows, srows, _ = operands(rng, M, N, K, "fp4", "x4", "mx", k0=2)
    old = rng.standard_normal((M, N)).astype(np.float32)
    alpha = rng.standard_normal(M).astype(np.float32)
    say("rows acc / ascale / k0", M, N)
    got = mxu.mm(q, Sa, da, rows, srows, "fp4", K, k0=2, acc=old)
    assert same_bits(got, OC.mm(q, Sa, da, rows, srows, "fp4", K, flags=MM.ACC, k0=2, old=old))
    zs = np.zeros((N, 8), np.uint8)
    got = mm_dot(X, q, Sa, da, rows, zs, "fp4", K, K, MM.UNIT | MM.ACC | MM.ASCALE, act=2, old=old, alpha=alpha)
    assert same_bits(got, OC.mm(q, Sa, da, rows, zs, "fp4", K, flags=MM.UNIT | MM.ACC | MM.ASCALE, old=old, alpha=alpha))


def test_mm_dot_refuses(X):
    rng = np.random.default_rng(1)
    q, Sa, da, rows, srows, _ = operands(rng, 6, 32, 512, "int4", "x4", "mx")
    for kw in ({"width": 128}, {"width": 300}, {"width": 512, "act": 3}, {"width": 512, "flags": MM.RMAX}):
        with pytest.raises(X.OtpuError):
            mm_dot(X, q, Sa, da, rows, srows, "int4", 512, kw["width"], kw.get("flags", 0), act=kw.get("act", 0))


@pytest.mark.parametrize("fmt,ranges", [("int4", [256, 256, 256]), ("int8", [768])])
def test_dot_of_an_operands_rows(X, fmt, ranges):
    """Rows of a longer operand: Sa's strides are those of the whole; offsets from an odd address."""
    import torch
    from opentpu_amd import mxu
    rng = np.random.default_rng(7)
    N, K = 70, 768
    _, _, _, rows, srows, _ = operands(rng, 1, N, K, fmt, "spread", "mx")
    w = mxu.QWeight.from_packed(rows, srows, fmt, K)
    x = torch.from_numpy(rng.standard_normal((20, K)).astype(np.float32)).cuda()
    q, Sa, da, rg = mxu.quantize_ranges(x, ranges)
    say("dot of rows 4..16", fmt, ranges)
    want = X.host(mxu.dot(x[4:17].contiguous(), w, ranges=ranges))
    assert same_bits(X.host(mxu.dot((q[4:17], Sa[:, 4:17], da[4:17], rg), w)), want)
    odd = torch.empty((13 * (K // 32) + 1,), dtype=torch.uint8, device="cuda")[1:].view(13, K // 32)
    odd.copy_(da[4:17])
    assert same_bits(X.host(mxu.dot((q[4:17], Sa[:, 4:17].contiguous(), odd, rg), w)), want)
