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
