"""`mxu.dot` itself at the edges of the rules that pick its launches, against the C oracle's MM a range
(`opentpu/compiler.py:2686-2720`) bit for bit."""
import numpy as np
import pytest

from conftest import same_bits
from oracle import chain as CH
from oracle import cpu as OC
from oracle import formats as Q
from oracle import mm as MM
from test_gpu_gemm4 import say, spread

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def mxu():
    import torch
    assert torch.cuda.is_available(), "GPU tests need a GPU"
    from opentpu_amd import _lib, mxu
    _lib.load()
    return mxu


def packed(rng, N, K, fmt):
    W = (spread(rng, N, K, 1.5, 128) * 0.02).astype(np.float32)
    return Q.pack_rsc(W) if fmt == "rsc" else Q.quantize_mxu(W, fmt)


def qweight(mxu, rows, srows, fmt, K):
    return mxu.QWeight.from_packed(rows, srows, "int8" if fmt == "rsc" else fmt, K, fmt == "rsc")


@pytest.mark.parametrize("fmt", ["int4", "fp4", "nvfp4"])
def test_one_row_in_ranges_of_every_width(mxu, fmt):
    """One row, 4-bit weights: K every multiple of 256 up to 8192, in ranges of 256 and of half of K or
    K's chunk (`opentpu/kernels/mlp.py:8-30`)."""
    from opentpu_amd.chain import down_chunk
    rng = np.random.default_rng(11)
    N = 40
    rows, srows = packed(rng, N, 8192, fmt)
    x = spread(rng, 1, 8192, 2.0, 32)
    for K in range(512, 8192 + 1, 256):
        r = np.ascontiguousarray(rows[:, :K // 2])
        w = qweight(mxu, r, srows, fmt, K)
        for width in sorted({256, down_chunk(K, fmt), K // 2 if K % 512 == 0 else K}):
            say("one row", fmt, K, width)
            got = mxu.dot(np.ascontiguousarray(x[:, :K]), w, ranges=[width] * (K // width))
            assert same_bits(got, CH.ranges_dot(x[:, :K], (r, srows), fmt, width, mm=OC.mm)), (K, width)


@pytest.mark.parametrize("fmt,F_dim", [("int4", 2304), ("nvfp4", 2560), ("fp4", 4864)])
def test_chain_of_widths_the_fold_splits_evenly(mxu, fmt, F_dim):
    """A chain whose down projection has 72, 80 or 152 pieces a row: the persistent step and the launches
    a linear."""
    from opentpu_amd.chain import DecodeChain, Shape
    sh = Shape(hidden=256, q_dim=512, kv_dim=256, F=F_dim, layers=2)
    say("chain", fmt, F_dim)
    ch = DecodeChain.synthetic(sh, fmt, seed0=41, std=0.05)
    host = [{k: (r.cpu().numpy(), s.cpu().numpy()) for k, (r, s) in l.items()} for l in ch.layers]
    x = np.random.default_rng(5).standard_normal((1, 256)).astype(np.float32)
    want = CH.step(x, host, fmt, 512, F_dim, None, mm=OC.mm)
    assert ch.persistent and same_bits(ch.step(x).cpu().numpy(), want)
    assert ch.chain_error() == 0
    ch.persistent = False
    assert same_bits(ch.step(x).cpu().numpy(), want)


@pytest.mark.parametrize("fmt,M,K,width", [("int8", 8, 40960, 5120), ("int4", 1, 40960, 5120), ("nvfp4", 3, 33024, 768),
                                           ("rsc", 40, 32768, 16384), ("int4", 1, 1 << 24, 16384)])
def test_ranges_past_one_mms_columns(mxu, fmt, M, K, width):
    """More columns than one MM takes (32640), each range within; and past 32-bit offsets in a tile."""
    import torch
    rng = np.random.default_rng(K + M)
    N = 9 if K < 1 << 20 else 2
    base, sr = packed(rng, N, width, fmt)
    R = K // width
    rows = np.concatenate([np.roll(base, i % N, 0) for i in range(R)], 1)
    head = {"nvfp4": 16, "int4": 8}.get(fmt, 4)
    per = {"int8": 1, "int4": 4, "nvfp4": 8, "rsc": 0}[fmt] * width // 128
    srows = np.concatenate([sr[:, :head]] + [np.roll(sr[:, head:head + per], i % N, 0) for i in range(R)], 1)
    x = rng.standard_normal((M, K)).astype(np.float32)
    say("ranges past one MM", fmt, M, K, width)
    got = mxu.dot(torch.from_numpy(x).cuda(), qweight(mxu, rows, srows, fmt, K), ranges=[width] * R).cpu().numpy()
    want = None
    for r in range(R):
        q, Sa, da = OC.qact(x[:, r * width:(r + 1) * width])
        b = base.shape[1]
        want = OC.mm(q, Sa, da, np.ascontiguousarray(rows[:, r * b:(r + 1) * b]), srows, "int8" if fmt == "rsc" else fmt,
                     width, flags=(MM.RSC if fmt == "rsc" else 0) | (MM.ACC if r else 0),
                     k0=0 if fmt == "rsc" else r * width // 128, old=want)
    assert same_bits(got, want)


@pytest.mark.parametrize("fmt,K,width", [("int8", 1024, 1024), ("int4", 4096, 4096), ("nvfp4", 2048, 256), ("int8", 1024, 256)])
def test_one_row_written_over(mxu, fmt, K, width):
    """out= on the row that is multiplied, or on a part of it."""
    import torch
    rng = np.random.default_rng(K + width)
    rows, srows = packed(rng, K, K, fmt)
    w = qweight(mxu, rows, srows, fmt, K)
    x = spread(rng, 1, K, 2.0, 32)
    want = CH.ranges_dot(x, (rows, srows), fmt, width, mm=OC.mm)
    say("one row written over", fmt, K, width)
    for off in (0, 4, -8, K // 2):
        buf = torch.zeros((3 * K,), device="cuda")
        xd, out = buf[K:2 * K].view(1, K), buf[K + off:2 * K + off].view(1, K)
        xd.copy_(torch.from_numpy(x))
        assert mxu.dot(xd, w, out=out, ranges=[width] * (K // width)) is out
        assert same_bits(out.cpu().numpy(), want), off


@pytest.mark.parametrize("fmt,M", [("int8", 7), ("int4", 1), ("fp4", 70)])
def test_ranges_over_a_part_of_an_operand(mxu, fmt, M):
    """An operand's ranges may cover its first columns only; a scale a range as a vector (one row)."""
    import torch
    rng = np.random.default_rng(M)
    N, K = 50, 1024
    rows, srows = packed(rng, N, K, fmt)
    w = qweight(mxu, rows, srows, fmt, K)
    x = torch.from_numpy(spread(rng, M, K, 2.0, 32)).cuda()
    q, Sa, da, _ = mxu.quantize_ranges(x, [256] * 4)
    host = x.cpu().numpy()
    for R in (1, 2, 4):
        say("ranges over a part", fmt, M, R)
        want = CH.ranges_dot(host[:, :256 * R], (rows, srows), fmt, 256, mm=OC.mm)
        for S in (Sa[:R],) + ((Sa[:R, 0].contiguous(),) if M == 1 else ()):
            assert same_bits(mxu.dot((q, S, da, [256] * R), w).cpu().numpy(), want)


def oracle_dot(x, rows, srows, fmt, K, widths, old=None, row_mode=False):
    """The oracle's dot: a QACT and an MM a range, the MMs' outputs added in range order."""
    want, c0 = old, 0
    bpb = 128 if fmt in ("int8", "rsc") else 64
    for i, n in enumerate(widths):
        q, Sa, da = OC.qact(np.ascontiguousarray(x[:, c0:c0 + n]), row_mode=row_mode)
        kb = c0 // 128
        want = OC.mm(q, Sa, da, np.ascontiguousarray(rows[:, kb * bpb:(kb + n // 128) * bpb]), srows, "int8" if fmt == "rsc" else fmt,
                     n, flags=(MM.RSC if fmt == "rsc" else 0) | (MM.ACC if want is not None else 0),
                     k0=0 if fmt == "rsc" else kb, old=want)
        c0 += n
    return want


ONE = [(40, 256, None), (40, 384, None), (20000, 2048, None), (32800, 2048, None), (40, 6144, None), (40, 6400, None), (40, 8192, None),
       (40, 8448, None), (70, 16384, None), (70, 16640, None), (4096, 6144, None), (4104, 6144, None),
       (12287, 512, 256), (12288, 512, 256), (20000, 512, 256), (60, 10240, 1280), (30, 8192, 256), (30, 8448, 256), (30, 8448, 768), (4096, 6144, 768), (50, 1024, 128),
       (50, 1024, (512, 256, 256)), (50, 1024, (256, 512, 256))]


@pytest.mark.parametrize("fmt", ["int8", "rsc", "int4", "fp4", "nvfp4"])
def test_one_row_at_the_rules_edges(mxu, fmt):
    """One row on both sides of each line of the rules that pick its launches; unequal ranges; a row whose
    weights are half a chunk."""
    import torch
    rng = np.random.default_rng(3)
    for N, K, width in ONE:
        widths = [K] if width is None else list(width) if isinstance(width, tuple) else [width] * (K // width)
        some = min(N, 64)
        rows, srows = packed(rng, some, K, fmt)
        rows, srows = np.resize(rows, (N, rows.shape[1])), np.resize(srows, (N, srows.shape[1]))
        x = spread(rng, 1, K, 2.0, 32)
        say("one row", fmt, N, K, width)
        got = mxu.dot(torch.from_numpy(x).cuda(), qweight(mxu, rows, srows, fmt, K), ranges=widths).cpu().numpy()
        want = oracle_dot(x, np.ascontiguousarray(rows[:some]), np.ascontiguousarray(srows[:some]), fmt, K, widths)
        assert same_bits(got, np.resize(want[0], (1, N))), (N, K, width)


@pytest.mark.parametrize("M,fmt,N", [(1, "int8", 20000), (2, "int4", 12288), (2, "rsc", 20003), (3, "nvfp4", 24576), (4, "fp4", 24600),
                                     (4, "int4", 24575)])
def test_few_rows_on_many_weights_in_ranges(mxu, M, fmt, N):
    """The GEMV of every range and the sum of their rows: overwriting, onto old values, from an operand."""
    import torch
    rng = np.random.default_rng(M + N)
    K, width, some = 768, 256, 50
    rows, srows = packed(rng, some, K, fmt)
    w = qweight(mxu, np.resize(rows, (N, rows.shape[1])), np.resize(srows, (N, srows.shape[1])), fmt, K)
    x = spread(rng, M, K, 2.0, 32)
    xd = torch.from_numpy(x).cuda()
    old = np.resize(rng.standard_normal((M, some)).astype(np.float32), (M, some))
    idx = np.arange(N) % some
    say("few rows", M, fmt, N)
    want = oracle_dot(x, rows, srows, fmt, K, [width] * 3)[:, idx]
    assert same_bits(mxu.dot(xd, w, ranges=[width] * 3).cpu().numpy(), want)
    assert same_bits(mxu.dot(mxu.quantize_ranges(xd, [width] * 3), w).cpu().numpy(), want)
    acc = torch.from_numpy(np.ascontiguousarray(old[:, idx])).cuda()
    assert same_bits(mxu.dot(xd, w, acc=acc, ranges=[width] * 3).cpu().numpy(), oracle_dot(x, rows, srows, fmt, K, [width] * 3, old)[:, idx])


def test_dots_under_capture(mxu):
    """One dot of each route in a graph: replays on new rows with eager work between, and on another stream."""
    import torch
    rng = np.random.default_rng(9)
    calls = []
    for fmt, M, N, K, width in (("int4", 1, 256, 1024, 1024), ("int4", 1, 256, 3072, 256), ("int8", 1, 20000, 512, 256),
                                ("nvfp4", 2, 12288, 512, 256), ("fp4", 6, 300, 512, 256), ("rsc", 130, 8200, 256, 256)):
        rows, srows = packed(rng, 50, K, fmt)
        w = qweight(mxu, np.resize(rows, (N, rows.shape[1])), np.resize(srows, (N, srows.shape[1])), fmt, K)
        calls.append((torch.zeros((M, K), device="cuda"), w, [width] * (K // width)))
    run = lambda: [mxu.dot(x, w, ranges=r) for x, w, r in calls]  # noqa: E731
    run()
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        outs = run()
    say("dots under capture")
    side = torch.cuda.Stream()
    for i in range(4):
        for x, _, _ in calls:
            x.copy_(torch.from_numpy(spread(rng, *x.shape, 2.0, 32)))
        eager = [t.cpu().numpy() for t in run()]
        torch.cuda.synchronize()
        with torch.cuda.stream(side if i % 2 else torch.cuda.current_stream()):
            g.replay()
            torch.cuda.synchronize()
        for a, b in zip(outs, eager):
            assert same_bits(a.cpu().numpy(), b), i
    with torch.cuda.stream(side):                         # eager on a stream of its own
        again = run()
    side.synchronize()
    assert all(same_bits(a.cpu().numpy(), b) for a, b in zip(again, eager))
