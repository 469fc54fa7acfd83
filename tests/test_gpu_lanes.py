"""Short columns, a few lanes of a wavefront each: byte for byte what the tile kernels give, whose sums they follow, as calls of their
own and as members of a gradient set. Needs an MI355X."""
import numpy as np
import pytest
import torch

import datagen
import parity
from cntk_amd import Matrix, MatrixQuantizerImpl, QuantizedMatrix

pytestmark = pytest.mark.gpu

PATH_TILE = 1
F32, F64 = torch.float32, torch.float64
# heights: the first of its kernel, a column of fewer QWords than lanes, the edges of every number of lanes (160 / 161, 320 / 321, 640 / 641 floats;
# 64 / 65, 128 / 129, 256 / 257 doubles) and of 4, 8, 16 and 20 elements per lane, the last odd one
ROWS = {F32: [17, 31, 32, 33, 64, 65, 128, 129, 147, 160, 161, 256, 257, 320, 321, 511, 512, 513, 640, 641, 1023, 1025, 1279],
        F64: [17, 32, 33, 63, 64, 65, 127, 128, 129, 255, 256, 257, 511, 512]}
# ... and the last height of all, every lane with 20 elements: only matrices off the 16-byte grid come here with it (an index in the list that is no multiple
# of 4, so an offset that is none; as whole aligned pieces it is a column kernel's)
UNALIGNED_ROWS = {F32: [1280], F64: []}
# columns: a wavefront that is not full, workgroups with wavefronts beyond the last column, whole ones and one column more
COLS = [1, 7, 33, 64, 65]
CASES = [(F32, b, z) for b, z in ((1, False), (1, True), (2, False), (4, False), (8, False), (16, False))] + \
        [(F64, b, z) for b, z in ((1, False), (1, True), (4, False), (32, False))]


def _make(rows, cols, dtype, gen, offset):
    """Gradient and residual at an offset of `offset` elements, with a column without spread, one of zeros of both signs, one with
    an infinity and one with a NaN where there are columns enough."""
    scale = lambda s, o: (torch.randn(rows * cols + 4, generator=gen, device="cuda:0") * s).to(dtype)[o:o + rows * cols]
    g, r = scale(0.01, offset), scale(0.002, (offset + (rows & 1)) % 4)
    if cols > 8:
        g[:2 * rows] = 0.0
        r[:2 * rows] = 0.0
        g[rows:2 * rows:2] = -0.0
        g[2 * rows + rows // 2] = float("inf")
        g[3 * rows + 5] = float("nan")
    return g, r


def _bytes(m):
    return (m.buffer if isinstance(m, QuantizedMatrix) else m.data).cpu().numpy().view(np.uint8)


def _pair(plain, tile, rows, cols, nbits, dtype, zt, gen, offset):
    g, r = _make(rows, cols, dtype, gen, offset)
    kw = dict(dtype=dtype)
    G = Matrix(rows, cols, 0, g, **kw)
    out = []
    for qz in (plain, tile):
        R = Matrix(rows, cols, 0, torch.empty(rows * cols + 4, dtype=dtype, device="cuda:0")[offset:offset + rows * cols].copy_(r), **kw)
        Q = QuantizedMatrix(rows, cols, nbits, 0, **kw)
        qz.QuantizeAsync(G, R, Q, R, zt)
        out.append((Q, R))
    return g, r, out


@pytest.mark.parametrize("dtype,nbits,zt", CASES)
def test_quantize(dtype, nbits, zt):
    plain, tile = MatrixQuantizerImpl.Create(0, False), MatrixQuantizerImpl.Create(0, False)
    tile._set_tuning(quantize_path=PATH_TILE)
    gen = torch.Generator(device="cuda:0")
    gen.manual_seed(datagen.case_seed(nbits))
    for n, rows in enumerate(ROWS[dtype] + UNALIGNED_ROWS[dtype]):
        for cols in COLS:
            g, r, ((Q1, R1), (Q2, R2)) = _pair(plain, tile, rows, cols, nbits, dtype, zt, gen, n % 4)
            torch.cuda.synchronize()
            assert np.array_equal(_bytes(Q1), _bytes(Q2)), ("packed", rows, cols)
            assert np.array_equal(_bytes(R1), _bytes(R2)), ("residual", rows, cols)
            if cols == 7:  # (no infinities there) against the oracle
                host = [x.cpu().numpy().reshape((rows, cols), order="F") for x in (g, r)]
                parity.check_quantize(host[0], host[1], Q1.to_numpy(), R1.to_numpy(), nbits, zt)


@pytest.mark.parametrize("workers", [1, 2, 8, 11])
@pytest.mark.parametrize("dtype,nbits,zt", [(F32, 1, False), (F32, 2, False), (F32, 4, False), (F32, 8, False), (F64, 1, True), (F64, 8, False)])
def test_stripe_reduce(dtype, nbits, zt, workers):
    plain, tile = MatrixQuantizerImpl.Create(0, False), MatrixQuantizerImpl.Create(0, False)
    tile._set_tuning(quantize_path=PATH_TILE)
    gen = torch.Generator(device="cuda:0")
    gen.manual_seed(datagen.case_seed(nbits) + workers)
    for n, rows in enumerate(ROWS[dtype] + UNALIGNED_ROWS[dtype]):
        for cols in (1, 33, 65):
            kw = dict(dtype=dtype)
            stripes = []
            for _ in range(workers):
                g, r = _make(rows, cols, dtype, gen, 0)
                Q = QuantizedMatrix(rows, cols, nbits, 0, **kw)
                R = Matrix(rows, cols, 0, r.clone(), **kw)
                tile.QuantizeAsync(Matrix(rows, cols, 0, g, **kw), R, Q, R, zt)
                stripes.append(Q)
            sr = (torch.randn(rows * cols + 4, generator=gen, device="cuda:0") * 0.003).to(dtype)
            got = []
            for qz in (plain, tile):
                S = Matrix(rows, cols, 0, sr.clone()[n % 4:n % 4 + rows * cols], **kw)
                Q, A = QuantizedMatrix(rows, cols, nbits, 0, **kw), Matrix(rows, cols, 0, **kw)
                qz.StripeReduceAsync(stripes, workers // 2, S, Q, zt, A)
                got.append((Q, S, A))
            torch.cuda.synchronize()
            for what, x, y in zip(("packed", "residual", "aggregate"), got[0], got[1]):
                assert np.array_equal(_bytes(x), _bytes(y)), (what, rows, cols)


@pytest.mark.parametrize("full", [False, True])
@pytest.mark.parametrize("dtype,nbits,zt", [(F32, 1, True), (F32, 4, False), (F32, 16, False), (F64, 2, False), (F64, 16, False)])
def test_members_of_a_set(dtype, nbits, zt, full):
    """Quantized and reduced (one worker) in one call each: the bytes of the tile kernels, also where the owner's result replaces its stripe. A
    set that is resident as a whole has all of these members on lanes, one that fills the device (full) those whose LDS is no more than
    their tiles'."""
    plain, tile = MatrixQuantizerImpl.Create(0, False), MatrixQuantizerImpl.Create(0, False)
    tile._set_tuning(quantize_path=PATH_TILE)
    gen = torch.Generator(device="cuda:0")
    gen.manual_seed(datagen.case_seed(nbits) + 1)
    kw = dict(dtype=dtype)
    items, want, stripes = [], [], []
    for n, rows in enumerate(ROWS[dtype] + [128] * full):
        cols = COLS[n % len(COLS)] if n < len(ROWS[dtype]) else 80000
        g, r = _make(rows, cols, dtype, gen, 0)
        G = Matrix(rows, cols, 0, g, **kw)
        both = []
        for _ in range(2):
            both.append((Matrix(rows, cols, 0, r.clone(), **kw), QuantizedMatrix(rows, cols, nbits, 0, **kw), Matrix(rows, cols, 0, **kw)))
        items.append((G, both[0][0], both[0][1], both[0][0]))
        stripes.append(([both[0][1]], both[0][2], both[0][1], None))
        R, Q, S = both[1]
        tile.QuantizeAsync(G, R, Q, R, zt)
        tile.StripeReduceAsync([Q], 0, S, Q, zt)
        want.append((R, Q, S))
    plain.QuantizeBatchAsync(plain.PrepareQuantizeBatch(items), zt)
    plain.StripeReduceBatchAsync(plain.PrepareStripeReduceBatch(stripes), [0] * len(stripes), zt)
    torch.cuda.synchronize()
    for (G, R, Q, _), (_, S, _, _), (R2, Q2, S2) in zip(items, stripes, want):
        for what, x, y in (("residual", R, R2), ("packed", Q, Q2), ("stripe residual", S, S2)):
            assert np.array_equal(_bytes(x), _bytes(y)), (what, G.rows, G.cols)
