"""The MM operator and its callers on the GPU: `mm` (one MM instruction's work), `dot` (the
operator API: QACT per range, an MM per range accumulated with ACC, as the reference's
`Builder.dot`, `opentpu/compiler.py:2622-2726`), `lm_head_argmax` and `greedy` (the LM head's
greedy sink, `opentpu/llm/generate.py:251-286`), `argmax` (VOP ARGMAX).

Arrays: numpy in -> numpy out (copied through the device); device tensors stay on the device
and every call is queued on the current torch stream."""
from __future__ import annotations

import functools
from dataclasses import dataclass

import numpy as np

from . import _lib as X
from . import fp32 as F
from .quant import D, WINDOW, quantize_mxu, row_bytes, scale_bytes

UNIT, ACC, RMAX, ASCALE, PAIR, RSC = X.UNIT, X.ACC, X.RMAX, X.ASCALE, X.PAIR, X.RSC


def _flags(unit=False, rsc=False, acc=False, ascale=False, rmax=False) -> int:
    return (UNIT if unit else 0) | (RSC if rsc else 0) | (ACC if acc else 0) | \
        (ASCALE if ascale else 0) | (RMAX if rmax else 0)


def mm(q, Sa, da, rows, srows, fmt: str, K: int, *, rsc: bool = False, unit: bool = False,
       k0: int = 0, acc=None, alpha=None, rmax: bool = False):
    """MM of activations (q int8 [M, K], Sa [M], da uint8 [M, K/32]: one QACT range) and weight
    rows (element rows [N, rs], scale rows [N, srs]; `opentpu/isasim.py:749-910`).

    acc: the old output [M, N] (ACC: y = old + mm; with alpha [M] also ASCALE:
    y = old * alpha + mm, needs unit).  rmax: also return the row maxima.  Returns y [M, N]."""
    numpy_in = X.is_numpy(q)
    qd = X.dev(q, np.int8)
    Sad = X.dev(Sa, np.float32)
    dad = X.dev(da, np.uint8)
    wd = X.dev(rows, np.uint8)
    sd = X.dev(srows, np.uint8) if srows is not None else None
    M, N = qd.shape[0], wd.shape[0]
    out = X.empty((M, N), np.float32) if acc is None else X.dev(acc, np.float32).clone()
    al = X.dev(alpha, np.float32) if alpha is not None else None
    rm = X.empty((M,), np.float32) if rmax else None
    fl = _flags(unit, rsc, acc is not None, alpha is not None, rmax)
    X.call("otpu_mm", X.ptr(qd), qd.shape[1], X.ptr(Sad), X.ptr(dad), dad.shape[1], M, K, X.ptr(wd),
           wd.shape[1], X.ptr(sd), sd.shape[1] if sd is not None else 0, N, X.FMT[fmt], fl, k0,
           X.ptr(al), X.ptr(out), N, X.ptr(rm), X.stream())
    if numpy_in:
        return (X.host(out), X.host(rm)) if rmax else X.host(out)
    return (out, rm) if rmax else out


def mm_acc(q, da, rows, srows, fmt: str, K: int, *, rsc: bool = False, unit: bool = False, k0: int = 0):
    """The exact int64 accumulators [M, N] of MM (no epilogue)."""
    numpy_in = X.is_numpy(q)
    qd, dad = X.dev(q, np.int8), X.dev(da, np.uint8)
    wd = X.dev(rows, np.uint8)
    sd = X.dev(srows, np.uint8) if srows is not None else None
    M, N = qd.shape[0], wd.shape[0]
    acc = X.empty((M, N), np.int64)
    X.call("otpu_mm_acc", X.ptr(qd), qd.shape[1], X.ptr(dad), dad.shape[1], M, K, X.ptr(wd), wd.shape[1],
           X.ptr(sd), sd.shape[1] if sd is not None else 0, N, X.FMT[fmt], _flags(unit, rsc), k0,
           X.ptr(acc), X.stream())
    return X.host(acc) if numpy_in else acc


def mm_spl(q, Sa, da, w_hi, w_lo, Sw, nterms: int, *, acc=None):
    """MM SPL (`opentpu/isasim.py:757-770`, `docs/isa.md:414-441`): one MM over a split
    operand's terms, one 128-block of int8 RSC weights a part.  q int8 [M, 128] (2 terms) or
    [M, 256] (3 terms: hi then lo, as `fp32.qact(hl=True)` gives them side by side), Sa [M] and
    da [M, 4] the hi part's, w_hi / w_lo the weights' hi and lo rows [N, 128] (`quantize_mxu(W,
    "int8", rsc=True)` and `(..., lo=True)`), Sw [N] the hi rows' scales.  acc: ACC into it."""
    numpy_in = X.is_numpy(q)
    qd = X.dev(q, np.int8)
    Sad, dad = X.dev(Sa, np.float32), X.dev(da, np.uint8)
    wh, wl = X.dev(w_hi, np.uint8), X.dev(w_lo, np.uint8)
    M, N = qd.shape[0], wh.shape[0]
    T = X.torch()
    w = T.cat([wh[:, :D], wl[:, :D]], 1).contiguous()     # hi rows, each followed by its lo row
    ws = X.dev(np.asarray(Sw, np.float32).reshape(-1) if X.is_numpy(Sw) else Sw, np.float32)
    out = X.empty((M, N), np.float32) if acc is None else X.dev(acc, np.float32).clone()
    X.call("otpu_mm_spl", X.ptr(qd), qd.shape[1], X.ptr(Sad), X.ptr(dad), dad.shape[1], M, nterms, X.ptr(w),
           2 * D, D, X.ptr(ws), 4, N, RSC | (ACC if acc is not None else 0), X.ptr(out), N, X.stream())
    return X.host(out) if numpy_in else out


def lm_head_argmax(q, Sa, da, rows, srows, fmt: str, K: int, *, rsc: bool = False, k0: int = 0,
                   base: int = 0, logits: bool = True):
    """One activation row times the vocabulary rows, with the greedy pick fused: returns
    (token, logits or None, best) where best = max over n of key(y_n) << 32 | ~(base + n)."""
    numpy_in = X.is_numpy(q)
    qd, Sad, dad = X.dev(q, np.int8), X.dev(Sa, np.float32), X.dev(da, np.uint8)
    wd, sd = X.dev(rows, np.uint8), X.dev(srows, np.uint8)
    N = wd.shape[0]
    lg = X.empty((N,), np.float32) if logits else None
    best = X.zeros((X.LM_STATE_BYTES // 8,), np.int64)   # the result word, the running maxima (zero)
    tok = X.empty((1,), np.int32)
    X.call("otpu_lm_head_argmax", X.ptr(qd), X.ptr(Sad), X.ptr(dad), K, X.ptr(wd), wd.shape[1], X.ptr(sd),
           sd.shape[1], N, X.FMT[fmt], _flags(rsc=rsc), k0, base, X.ptr(lg), X.ptr(best), X.ptr(tok),
           X.stream())
    if numpy_in:
        return (int(X.host(tok)[0]), X.host(lg) if logits else None,
                int(X.host(best).view(np.uint64)[0]))
    return tok, lg, best[:1]


def argmax(x, base: int = 0):
    """VOP ARGMAX of each row of x [rows, cols]: (max values [rows], first index + base [rows])
    (`opentpu/isasim.py:1141-1152`; the index comes back as the i2f'd fp32 the VOP writes)."""
    numpy_in = X.is_numpy(x)
    xd = X.dev(np.atleast_2d(x) if numpy_in else x, np.float32)
    if xd.dim() == 1:
        xd = xd.reshape(1, -1)
    rows, cols = xd.shape
    pairs = X.empty((rows, 2), np.float32)
    X.call("otpu_argmax", X.ptr(xd), rows, cols, cols, base, X.ptr(pairs), 2, X.stream())
    if numpy_in:
        p = X.host(pairs)
        return p[:, 0], p[:, 1].astype(np.int64)
    return pairs[:, 0], pairs[:, 1]


@dataclass
class QWeight:
    """A streamed weight resident on the device: element rows, scale rows, format, K (the
    reference's `runtime.Weight` once placed, `opentpu/runtime.py:38-51`; the descriptor
    `compiler.QTensor`).  rsc: the scale rows are Sw alone."""
    rows: object
    srows: object
    fmt: str
    K: int
    rsc: bool = False

    @property
    def N(self) -> int:
        return self.rows.shape[0]

    @staticmethod
    def from_float(W, fmt: str = "int8", rsc: bool = False) -> "QWeight":
        """Pack W [N, K] on the GPU (quantize_mxu) and keep it there."""
        Wd = X.dev(W, np.float32)
        rows, srows = quantize_mxu(Wd, fmt, rsc=rsc)
        return QWeight(rows, srows, fmt, Wd.shape[1], rsc)

    @staticmethod
    def from_packed(rows, srows, fmt: str, K: int, rsc: bool = False) -> "QWeight":
        """Rows packed elsewhere (e.g. by the reference's quantize_mxu): loaded unchanged."""
        if rows.shape[1] < row_bytes(K, fmt) or srows.shape[1] < scale_bytes(K, fmt, rsc):
            raise ValueError("QWeight: rows or scale rows shorter than the format's")
        return QWeight(X.dev(rows, np.uint8), X.dev(srows, np.uint8), fmt, K, rsc)


def _check_ranges(ranges, K: int) -> list:
    ranges = [K] if ranges is None else list(ranges)
    if sum(ranges) != K or any(r % D for r in ranges):
        raise ValueError(f"quantize_ranges: ranges {ranges} over {K} columns")
    return ranges


def _qact_equal(xd, ranges, row_mode: bool, q: int, Sa: int, da: int, stream) -> None:
    """QACT of equal ranges into packed buffers (their addresses), one launch."""
    M, K = xd.shape
    fl = X.Q_ROW if row_mode else 0
    if len(ranges) > 1:
        X.call("otpu_qact_ranges", xd.data_ptr(), None, M, K, K, ranges[0], 32, fl, None, None, q, K, Sa, da, K // 32, stream)
    else:
        X.call("otpu_qact", xd.data_ptr(), M, K, K, 32, fl, None, None, q, K, Sa, da, K // 32, None, 0, stream)


class Operand(tuple):
    """(q, Sa, da, ranges) as quantize_ranges returns it, with its mode: the offsets of a ROW operand are all 0.
    A dot picks a kernel by it (a plain tuple's offsets are unknown); no bit of its result depends on it."""
    row = False


def _operand(q, Sa, da, ranges, row: bool) -> Operand:
    op = Operand((q, Sa, da, ranges))
    op.row = row
    return op


def quantize_ranges(x, ranges=None, row_mode: bool = False):
    """QACT of x [M, K] in column ranges (widths summing to K, each a multiple of 128; default
    one range): the int8 operand [M, K], Sa per range [n_ranges, M], da [M, K/32] and the ranges (an
    Operand)."""
    xd = X.dev(x, np.float32)
    M, K = xd.shape
    ranges = _check_ranges(ranges, K)
    q = X.empty((M, K), np.int8)
    da = X.empty((M, K // 32), np.uint8)
    Sa = X.empty((len(ranges), M), np.float32)
    if min(ranges) == max(ranges):
        _qact_equal(xd, ranges, row_mode, q.data_ptr(), Sa.data_ptr(), da.data_ptr(), X.stream())
        return _operand(q, Sa, da, ranges, bool(row_mode))
    flags = X.Q_ROW if row_mode else 0
    c0 = 0
    for i, w in enumerate(ranges):
        xs = xd[:, c0:c0 + w]
        X.call("otpu_qact", X.ptr(xs), M, w, K, 32, flags, None, None, C_ptr(q, c0), K,
               X.ptr(Sa[i]), C_ptr(da, c0 // 32), K // 32, None, 0, X.stream())
        c0 += w
    return _operand(q, Sa, da, ranges, bool(row_mode))


def C_ptr(t, off: int):
    import ctypes
    return ctypes.c_void_p(t.data_ptr() + off * t.element_size())


# One row's launches: QACT inside the GEMV (otpu_mm_qin, otpu_mm_qin_fold) saves a launch of ~3 us, and every
# workgroup quantizes the whole row again.  So the columns they quantize together (otpu_qin_columns) decide.  Up
# to 3M (2M past 16384 weight rows) the single launch is the faster nearly everywhere (weight rows x columns, us,
# one / two launches: int4 4096 x 1024 4.6 / 6.1, 4096 x 6144 (3M) 8.3 / 9.3, 16384 x 4096 14.3 / 11.4, 12288 x 16384
# 63 / 37; int8 4096 x 4096 7.6 / 8.6, 12288 x 12288 59 / 39).  A fold of 256-column ranges: up to 8M (int4 1024 x
# 3072 5.8 / 10.5, 8192 x 8192 28.8 / 24.8); of wider ones, whose sums a team's first lane adds one after another: up
# to 3M (2048 x 6144 11.4 / 11.5, 4096 x 6144 16.1 / 11.8).
QIN_COLUMNS = 3 << 20
TALL_QIN_COLUMNS = 2 << 20
FOLD_COLUMNS = 8 << 20
WIDE_FOLD_COLUMNS = 3 << 20
OFF_COLS = 1 << 24                                        # otpu_mm_dot's rows: 32-bit offsets over a tile's rows


@functools.lru_cache(maxsize=4096)
def _row_launch(fmt: str, N: int, K: int, width: int) -> bool:
    """Whether one row's QACT and MM over ranges of `width` run as one launch."""
    cols = X.load().otpu_qin_columns(K, width, N, X.FMT[fmt])
    if width < K:
        return 0 < cols <= (FOLD_COLUMNS if width == 256 else WIDE_FOLD_COLUMNS)
    # (int8 rows of eight pieces a lane: the kernel's prologue is compiled for 16384 columns and leaves one wave
    # a SIMD; 4096 x 8192 16.7 us against 11.7.  Past 8192 the other GEMV walks segments: 4096 x 10240 19.9 / 21.1)
    return 0 < cols <= (QIN_COLUMNS if N <= 16384 else TALL_QIN_COLUMNS) and not (fmt == "int8" and 6144 < K <= 8192)


# ... and in ranges: the GEMV of every range and the sum of their rows (otpu_mm_ranges) in place of otpu_mm_dot's
# tiles of 16 and 32 rows, where those are mostly padding and weights enough stream by.  One row (us, GEMV / tiles,
# QACT in): int4 12288 x 8192 18.6 / 29.7, 2048 x 8192 10.6 / 12.7, 4096 x 1024 8.8 / 7.4; int8 2048 x 16384 13.9 /
# 19.4, 16384 x 8192 35.7 / 29.6.  Two (without QACT): int4 12288 x 2048 12.2 / 16.9, 8192 x 2048 10.9 / 7.8; int8 20000 x
# 1024 10.5 / 13.9.  Four: 70000 x 1024 int4 39.9 / 45.3, int8 34.0 / 29.0.  It takes a workspace of a row a range, so
# not where that is large.
PART_BYTES = 1 << 28


def _stream_ranges(M: int, N: int, fmt: str, width: int) -> bool:
    if fmt == "int8":
        return M <= 2 and (N >= 20000 or (M == 1 and width >= 1280))
    if M <= 2:
        return N >= 12288 or (M == 1 and width >= 512)
    return M <= 4 and N >= 24576


def _overlap(a, b) -> bool:
    """Whether the memory two contiguous tensors hold overlaps."""
    pa, pb = a.data_ptr(), b.data_ptr()
    return pa < pb + b.numel() * b.element_size() and pb < pa + a.numel() * a.element_size()


def _dot_row(x, w: QWeight, ranges, out, given: bool) -> bool:
    """One fp32 row x (a contiguous device tensor [1, K]) @ w^T into out in one launch, QACT and the
    ranges' ACC chain inside; False where no such kernel takes the call, or out, where the caller gave
    it, overlaps x (every workgroup reads the row while others store)."""
    K, width = w.K, ranges[0]
    if len(ranges) > 1 and min(ranges) != max(ranges):
        return False
    if x.data_ptr() % 16 or not _row_launch(w.fmt, w.N, K, width) or (given and _overlap(x, out)):
        return False
    ws, srs = (0, 0) if w.srows is None else (w.srows.data_ptr(), w.srows.shape[1])
    fl = _flags(w.srows is None, w.rsc)
    if width == K:
        X.call("otpu_mm_qin", x.data_ptr(), None, None, None, 1, 0, K, K, w.rows.data_ptr(), w.rows.shape[1], ws, srs,
               w.N, X.FMT[w.fmt], fl, 0, out.data_ptr(), w.N, 0, X.stream())
        return True
    if fl:
        return False
    X.call("otpu_mm_qin_fold", x.data_ptr(), None, None, None, K, width, w.rows.data_ptr(), w.rows.shape[1], ws, srs,
           w.N, X.FMT[w.fmt], 0, 0, out.data_ptr(), X.stream())
    return True


def _scratch(*sizes):
    """The addresses of buffers of these sizes (bytes, each aligned to 256) and the allocation that
    holds them, to be kept until the launches that use them are queued."""
    offs, n = [], 0
    for b in sizes:
        offs.append(n)
        n += (b + 255) & ~255
    t = X.empty((n,), np.uint8)
    p = t.data_ptr()
    return *(p + o for o in offs), t


def _operand_act(x, w: QWeight) -> int:
    """What an operand's mode says of its offsets to otpu_mm_dot.  Of MX offsets and plain weights (RSC, UNIT)
    nothing is said: two a tile are the faster on the GEMM (int8 512 x 2048 x 8192 21 us against 32), three not
    (33.5 / 32.3); on 4-bit weights with scale rows either is the slower there (int4 51.9 and 48.1 / 46.1)."""
    if not isinstance(x, Operand):
        return X.ACT_ANY
    if x.row:
        return X.ACT_ROW
    return X.ACT_ANY if w.fmt == "int8" or w.rsc or w.srows is None else X.ACT_MX


def dot(x, w: QWeight, acc=None, out=None, ranges=None, row_mode: bool = False, rowmax: bool = False,
        acc_scale=None):
    """x [M, K] (fp32, quantized here, or a (q, Sa, da, ranges) operand from quantize_ranges)
    @ w^T -> [M, N] fp32, as `ol.dot` lowers it: one QACT per range, one MM per range, the
    first overwriting (or ACC into `acc`, or ASCALE with acc_scale), the rest ACC.  The
    4-bit formats need ranges that start on even blocks (a 128-byte chunk holds two blocks).
    rowmax: also return the row maxima of the final sums (MM RMAX on the last range).

    Equal ranges run as one QACT launch and one MM launch (otpu_mm_dot: the ACC chain inside; few rows
    on many weights otpu_mm_ranges), one fp32 row as a single launch where that is the faster; anything
    else as a launch per range."""
    numpy_in = X.is_numpy(x)
    if acc is not None and out is not None:
        raise ValueError("dot: give either acc= or out=")
    N = w.N
    operand = isinstance(x, tuple)
    xd = None
    if not operand:
        xd = X.dev(x, np.float32)
        M, K = xd.shape
        if K != w.K:
            raise ValueError(f"dot: K mismatch {K} vs {w.K}")
        ranges = _check_ranges(ranges, K)
        if M == 1 and not (row_mode or rowmax) and acc is None and acc_scale is None:
            y = out if out is not None else X.empty((1, N), np.float32)
            if _dot_row(xd, w, ranges, y, out is not None):
                return X.host(y) if numpy_in else y
    else:
        q, Sa, da, ranges = x
        M, K = q.shape
        if K != w.K:
            raise ValueError(f"dot: K mismatch {K} vs {w.K}")
    unit = w.srows is None
    chunk = D if w.fmt == "int8" else 2 * D
    width = ranges[0]
    one = not rowmax and K < OFF_COLS and (len(ranges) == 1 or (min(ranges) == max(ranges) and width % chunk == 0))
    if operand and one:                                   # ranges short of the row, scales of other shapes or
        one = (da.data_ptr() % 4 == 0 and sum(ranges) == K  # strides, offsets of odd addresses: a launch a range
               and (len(ranges) == 1 or (isinstance(Sa, X.torch().Tensor) and Sa.is_contiguous()
                                         and Sa.dim() == 2 and Sa.shape[0] >= len(ranges) and Sa.shape[1] == M)))
    if not operand and not one:
        q, Sa, da, ranges = quantize_ranges(xd, ranges, row_mode)
    y = X.dev(acc, np.float32) if acc is not None else (out if out is not None else X.empty((M, N), np.float32))
    al = X.dev(acc_scale, np.float32) if acc_scale is not None else None
    if one:
        s = X.stream()
        R = len(ranges)
        stream = (R > 1 and al is None and R < 1 << 16 and 4 * R * M * N <= PART_BYTES
                  and _stream_ranges(M, N, w.fmt, width))
        sizes = (4 * R * M * N,) if stream else ()
        if operand:
            qp, Sp, dp, act = q.data_ptr(), Sa[0].data_ptr(), da.data_ptr(), _operand_act(x, w)
            *part, _scr = _scratch(*sizes) if stream else (None,)
        else:                                             # the operand's three parts in one allocation
            qp, Sp, dp, *part, _scr = _scratch(M * K, 4 * M * R, M * (K // 32), *sizes)
            act = X.ACT_ROW if row_mode else X.ACT_MX
            _qact_equal(xd, ranges, row_mode, qp, Sp, dp, s)
        ws, srs = (0, 0) if unit else (w.srows.data_ptr(), w.srows.shape[1])
        fl = _flags(unit, w.rsc, acc is not None, al is not None)
        if stream:
            X.call("otpu_mm_ranges", qp, K, Sp, dp, K // 32, M, K, width, w.rows.data_ptr(), w.rows.shape[1], ws, srs, N,
                   X.FMT[w.fmt], fl, 0, part[0], y.data_ptr(), N, s)
        else:
            X.call("otpu_mm_dot", qp, K, Sp, dp, K // 32, M, K, width, w.rows.data_ptr(), w.rows.shape[1], ws, srs, N,
                   X.FMT[w.fmt], fl, 0, act, X.ptr(al), y.data_ptr(), N, s)
        return X.host(y) if numpy_in else y
    bpb = D if w.fmt == "int8" else D // 2
    rm = X.empty((M,), np.float32) if rowmax else None
    c0 = 0
    for i, width in enumerate(ranges):
        k0 = c0 // D
        first, last = i == 0, i == len(ranges) - 1
        accf = acc is not None or not first
        fl = _flags(unit, w.rsc, accf, al is not None and first, rowmax and last)
        X.call("otpu_mm", C_ptr(q, c0), K, X.ptr(Sa[i]), C_ptr(da, c0 // 32), K // 32, M, width,
               C_ptr(w.rows, k0 * bpb), w.rows.shape[1], X.ptr(w.srows), w.srows.shape[1] if not unit else 0,
               N, X.FMT[w.fmt], fl, 0 if (unit or w.rsc) else k0, X.ptr(al) if first else None, X.ptr(y), N,
               X.ptr(rm) if (rowmax and last) else None, X.stream())
        c0 += width
    if numpy_in:
        return (X.host(y), X.host(rm)) if rowmax else X.host(y)
    return (y, rm) if rowmax else y


class Greedy:
    """The LM head's greedy sink over vocabulary chunks (`opentpu/llm/generate.py:251-286`):
    each chunk's rows run through `lm_head_argmax` with its first row as the index base, and the
    token is the best over the chunks' (key << 32 | ~index) words, ties to the lowest index."""

    def __init__(self):
        self.best = 0

    def feed(self, best_word: int) -> None:
        self.best = max(self.best, best_word)

    def token(self) -> int:
        return int(~self.best & 0xFFFFFFFF)


def greedy(x, w: QWeight, chunk: int | None = None) -> int:
    """The greedy token of x [1, K] @ w^T (w: the LM head), in vocabulary chunks (all rows at
    once by default): the argmax of the fp32 logits, the lowest index on ties."""
    q, Sa, da = F.quantize_mx(X.dev(x, np.float32).reshape(1, -1), 32)
    N = w.N
    chunk = chunk or N
    g = Greedy()
    for c0 in range(0, N, chunk):
        n = min(chunk, N - c0)
        _, _, best = lm_head_argmax(q, Sa, da, w.rows[c0:c0 + n], w.srows[c0:c0 + n], w.fmt, w.K,
                                    rsc=w.rsc, base=c0, logits=False)
        g.feed(int(X.host(best).view(np.uint64)[0]))
    return g.token()


__all__ = ["mm", "mm_acc", "mm_spl", "lm_head_argmax", "argmax", "QWeight", "quantize_ranges", "dot", "Greedy",
           "greedy", "UNIT", "ACC", "RMAX", "ASCALE", "RSC", "WINDOW"]
