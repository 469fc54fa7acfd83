"""Columns of at most 16 rows (one thread per column): the oracle's results, and byte for byte what the tile kernels give, whose
sums they follow. Needs an MI355X."""
import numpy as np
import pytest
import torch

import datagen
import parity
from cntk_amd import Matrix, MatrixQuantizerImpl, QuantizedMatrix, qcol_bytes

pytestmark = pytest.mark.gpu

PATH_TILE = 1
F32, F64 = torch.float32, torch.float64
# (columns: part of a workgroup, one past a whole one, several columns per thread with a remainder)
SHAPES = [(r, c) for r in range(1, 18) for c in (1, 255, 257, 1031)] + [(1, 600001), (2, 300007), (3, 270001), (5, 262145), (8, 262143)]
# columns of several QWords get a thread each from 98304 columns on
MANY = [(2, 98305), (3, 98304), (4, 98303), (5, 100001), (6, 98307), (7, 98400), (9, 98561), (11, 98304), (13, 98310), (16, 98304)]


def _make(rows, cols, dtype, gen, offset):
    scale = lambda s: (torch.randn(rows * cols + 4, generator=gen, device="cuda:0") * s).to(dtype)[offset:offset + rows * cols]
    g, r = scale(0.01), scale(0.002)
    if cols > 8:
        g[:rows] = 0.0  # a column without spread, one of zeros of both signs
        r[:rows] = 0.0
        g[rows:2 * rows] = -0.0
        r[rows:2 * rows] = -0.0
    return g, r


@pytest.mark.parametrize("dtype,nbits,zt", [(F32, b, z) for b, z in ((1, False), (1, True), (2, False), (4, False), (8, False), (16, False), (32, False))] +
                         [(F64, b, z) for b, z in ((1, False), (1, True), (4, False), (8, False), (32, False), (64, False))])
def test_quantize_unquantize(dtype, nbits, zt):
    plain, tile = MatrixQuantizerImpl.Create(0, False), MatrixQuantizerImpl.Create(0, False)
    tile._set_tuning(quantize_path=PATH_TILE)
    gen = torch.Generator(device="cuda:0")
    gen.manual_seed(datagen.case_seed(nbits))
    for n, (rows, cols) in enumerate(SHAPES + MANY):
        g, r = _make(rows, cols, dtype, gen, n % 4)
        kw = dict(dtype=dtype)
        G = Matrix(rows, cols, 0, g, **kw)
        R1, R2, R3 = (Matrix(rows, cols, 0, r.clone(), **kw) for _ in range(3))
        Q1, Q2 = QuantizedMatrix(rows, cols, nbits, 0, **kw), QuantizedMatrix(rows, cols, nbits, 0, **kw)
        plain.QuantizeAsync(G, R1, Q1, R1, zt)
        tile.QuantizeAsync(G, R2, Q2, R3, zt)
        out = Matrix(rows, cols, **kw)
        plain.UnquantizeAsync(Q1, out)
        torch.cuda.synchronize()
        assert np.array_equal(Q1.to_numpy(), Q2.to_numpy()), ("packed", rows, cols)
        assert parity.bits_equal(R1.to_numpy(), R3.to_numpy()), ("residual", rows, cols)
        if cols < 1000:
            parity.check_quantize(G.to_numpy(), r.cpu().numpy().reshape(cols, rows).T, Q1.to_numpy(), R1.to_numpy(), nbits, zt)
        if cols < 1000 or n % 2:
            parity.check_unquantize(Q1.to_numpy(), rows, cols, nbits, out.to_numpy())


@pytest.mark.parametrize("nbits,zt,k", [(1, False, 1), (1, True, 9), (2, False, 3), (4, False, 4), (8, False, 8), (16, False, 5), (32, False, 2)])
def test_stripe_reduction(nbits, zt, k):
    """Alone, in a set, and as the tile kernel does it."""
    qz, tile = MatrixQuantizerImpl.Create(0, False), MatrixQuantizerImpl.Create(0, False)
    tile._set_tuning(quantize_path=PATH_TILE)
    gen = torch.Generator(device="cuda:0")
    gen.manual_seed(datagen.case_seed(70 + nbits))
    owner = k // 2
    shapes = [(r, c) for r in (1, 2, 3, 4, 7, 8, 9, 15, 16, 17) for c in (5, 257, 1031)] + [(2, 98305), (5, 98304), (9, 98303), (12, 98311)]
    runs = [[], [], []]
    for n, (rows, cols) in enumerate(shapes):
        packed = []
        for _ in range(k):
            g, r = _make(rows, cols, F32, gen, 0)
            q = QuantizedMatrix(rows, cols, nbits, 0)
            qz.QuantizeAsync(Matrix(rows, cols, 0, g), Matrix(rows, cols, 0, r), q, Matrix(rows, cols), zt)
            packed.append(q)
        _, res = _make(rows, cols, F32, gen, n % 4)
        for run in runs:
            run.append((packed, Matrix(rows, cols, 0, res.clone()), QuantizedMatrix(rows, cols, nbits, 0), Matrix(rows, cols)))
    for q, s, o, a in runs[0]:
        tile.StripeReduceAsync(q, owner, s, o, zt, agg_out=a)
    for q, s, o, a in runs[1]:
        qz.StripeReduceAsync(q, owner, s, o, zt, agg_out=a)
    qz.StripeReduceBatchAsync(runs[2], owner, zt)
    torch.cuda.synchronize()
    for i, shape in enumerate(shapes):
        for run in runs[1:]:
            assert np.array_equal(runs[0][i][2].to_numpy(), run[i][2].to_numpy()), ("packed", shape)
            assert parity.bits_equal(runs[0][i][1].to_numpy(), run[i][1].to_numpy()), ("stripe residual", shape)
            assert parity.bits_equal(runs[0][i][3].to_numpy(), run[i][3].to_numpy()), ("aggregate", shape)


def _same(a, b):
    """Equal, or both not a number."""
    return torch.equal(torch.where(a.isnan(), torch.zeros_like(a), a), torch.where(b.isnan(), torch.zeros_like(b), b)) and torch.equal(a.isnan(), b.isnan())


@pytest.mark.parametrize("dtype,nbits,zt", [(F32, 1, False), (F32, 1, True), (F32, 2, False), (F32, 4, False), (F32, 8, False), (F32, 32, False),
                                            (F64, 1, False), (F64, 8, False), (F64, 64, False)])
def test_special_values_and_offsets(dtype, nbits, zt):
    """NaN, infinities, zeros of both signs and tiny values, one kind per column; gradient and residuals each at an offset of their
    own within 16 bytes; the packed matrix at the alignment of a value. What the tile kernels give."""
    plain, tile = MatrixQuantizerImpl.Create(0, False), MatrixQuantizerImpl.Create(0, False)
    tile._set_tuning(quantize_path=PATH_TILE)
    gen = torch.Generator(device="cuda:0")
    gen.manual_seed(datagen.case_seed(900 + nbits))
    tiny = torch.finfo(dtype).tiny
    kinds = [float("nan"), float("inf"), -float("inf"), 0.0, -0.0, tiny, tiny / 4, torch.finfo(dtype).max]
    word, size = (torch.int64, 8) if dtype == F64 else (torch.int32, 4)
    for n, (rows, cols) in enumerate([(r, 300) for r in range(1, 17)] + [(3, 98400), (5, 98305), (12, 98304)]):
        def at(offset, fill=None):
            v = torch.empty(rows * cols + 4, dtype=dtype, device="cuda:0")[offset:offset + rows * cols]
            return v.normal_(generator=gen) if fill is None else v.copy_(fill)

        g, r = at(n % 4), at((n + 1) % 4)
        for k, x in enumerate(kinds):
            g[(20 + k) * rows:(21 + k) * rows] = x  # whole columns ...
            r[(20 + k) * rows:(21 + k) * rows] = 0.0
            g[(40 + k) * rows + k % rows] = x       # ... and one value of a column
            r[(60 + k) * rows + k % rows] = x
        runs = []
        for qz in (plain, tile):
            out = at((n + 2) % 4, r)
            buffer = torch.empty(qcol_bytes(nbits, rows, dtype) * cols + 8, dtype=torch.uint8, device="cuda:0")[size % 8:]
            q = QuantizedMatrix(rows, cols, nbits, 0, buffer[:qcol_bytes(nbits, rows, dtype) * cols], dtype=dtype)
            qz.QuantizeAsync(Matrix(rows, cols, 0, g), Matrix(rows, cols, 0, r), q, Matrix(rows, cols, 0, out), zt)
            runs.append((q, out))
        torch.cuda.synchronize()
        (q1, o1), (q2, o2) = runs
        v1, v2 = [q.buffer.clone().view(dtype).view(cols, -1) for q in (q1, q2)]
        assert _same(v1[:, :2], v2[:, :2]), ("bounds", rows, cols)
        if nbits != size * 8:
            assert torch.equal(v1.contiguous().view(word)[:, 2:], v2.contiguous().view(word)[:, 2:]), ("words", rows, cols)
        else:  # the codes are the values themselves
            assert _same(v1[:, 2:], v2[:, 2:]), ("values", rows, cols)
        assert _same(o1, o2), ("residual", rows, cols)
