"""Columns of at most 16 rows (one thread per column): the oracle's results, and byte for byte what the tile kernels give, whose
sums they follow. Needs an MI355X."""
import numpy as np
import pytest
import torch

import datagen
import parity
from cntk_amd import Matrix, MatrixQuantizerImpl, QuantizedMatrix

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
