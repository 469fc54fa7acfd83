"""Tall columns in strips: ragged ends at every remainder, every number of copies of the strips' partial sums, and a launch whose scratch
buffer has no room for copies. The strips in passes (nothing waits, one copy) add the same sums in the same order and tell whether the exchange
is right; they load a column as the single launch does, so the loads of the ragged ends are held against the CPU oracle. Needs an MI355X."""
import numpy as np
import pytest
import torch

import cntk_amd
import datagen
import oracle
import parity
from cntk_amd import Matrix, MatrixQuantizerImpl, QuantizedMatrix

pytestmark = pytest.mark.gpu

PATH_STRIP, PATH_STRIP_PASSES = 6, 7
F32, F64 = torch.float32, torch.float64
WORDS = {F32: {1: 512, 2: 1024, 4: 2048, 8: 2048, 16: 2048}, F64: {1: 128, 4: 512, 32: 1024}}  # QWords per strip


def _quantize(qz, g, r, rows, cols, nbits, dtype, zt):
    G, R = Matrix(rows, cols, 0, g, dtype=dtype), Matrix(rows, cols, 0, r.clone(), dtype=dtype)
    Q = QuantizedMatrix(rows, cols, nbits, 0, dtype=dtype)
    Q.buffer.fill_(0xA5)
    qz.QuantizeAsync(G, R, Q, R, zt)
    qz.WaitQuantizeAsyncDone()
    torch.cuda.synchronize()
    return Q.buffer, R.data.view(torch.uint8)


def _column(m, rows, j, dtype):
    """Column j as the oracle takes it."""
    return np.asfortranarray(m.view(dtype)[j * rows:(j + 1) * rows].cpu().numpy().reshape((rows, 1)))


# strips per column: fewer than share a copy, the edges of 1, 2 and 3 copies, the edges of the pause before the first look (8, 27),
# more than a wavefront has lanes, and more than 16 copies of four take (65); ends: whole strips, one QWord more, a piece
# that runs over the column's end by one to three elements, a last bit position that is nearly or almost empty
@pytest.mark.parametrize("dtype,nbits,zt", [(F32, 1, False), (F32, 1, True), (F32, 2, False), (F32, 4, False), (F32, 8, False), (F32, 16, False),
                                            (F64, 1, False), (F64, 4, False), (F64, 32, False)])
def test_strips_against_passes(dtype, nbits, zt):
    qz = MatrixQuantizerImpl.Create(0, False)
    gen = torch.Generator(device="cuda:0")
    gen.manual_seed(datagen.case_seed(97, nbits))
    words, per = WORDS[dtype][nbits], (32 if dtype == F32 else 64) // nbits
    for strips in (2, 4, 5, 8, 9, 27, 28, 64, 65, 70):
        if strips > qz._strip_max_strips(nbits, zt, dtype):
            continue
        for extra in (0, 1, 2, 3, 5, per, words * per - 1, words * per // 2 + 1):
            rows = (strips - 1) * words * per + (extra if extra else words * per)
            cols = 3 if strips < 28 else 1
            print(dtype, nbits, zt, "strips", strips, "rows", rows, "cols", cols, flush=True)
            g = (torch.randn(rows * cols + 3, generator=gen, device="cuda:0") * 0.01).to(dtype)[extra & 1:][:rows * cols]
            r = (torch.randn(rows * cols, generator=gen, device="cuda:0") * 0.002).to(dtype)
            if cols > 1:
                g[rows // 3] = float("inf")
                g[rows + 7] = float("nan")
            outs = []
            for path in (PATH_STRIP, PATH_STRIP_PASSES):
                qz._set_tuning(quantize_path=path)
                outs.append(_quantize(qz, g, r, rows, cols, nbits, dtype, zt))
            assert torch.equal(outs[0][0], outs[1][0]) and torch.equal(outs[0][1], outs[1][1]), (strips, rows)
            if strips <= 5:  # the last column, which is finite
                packed, j = outs[0][0].cpu().numpy(), cols - 1
                qcol = packed.size // cols
                parity.check_quantize(_column(g, rows, j, dtype), _column(r, rows, j, dtype), packed[j * qcol:].copy(), _column(outs[0][1], rows, j, dtype), nbits, zt)


@pytest.mark.parametrize("dtype,nbits,zt", [(F32, 1, False), (F32, 1, True), (F32, 2, False), (F32, 4, False), (F32, 8, False), (F32, 16, False),
                                            (F64, 1, False), (F64, 4, False), (F64, 32, False)])
def test_ragged_stripes_against_the_oracle(dtype, nbits, zt):
    """The fused reduction of two workers' stripes of 11 strips (three copies of the records), at every kind of ragged end."""
    qz = MatrixQuantizerImpl.Create(0, False)
    words, per, cols, workers = WORDS[dtype][nbits], (32 if dtype == F32 else 64) // nbits, 2, 2
    npdt = np.float32 if dtype == F32 else np.float64
    for extra in (0, 1, 2, 3, 5, per, words * per - 1, words * per // 2 + 1):
        rows = 10 * words * per + (extra if extra else words * per)
        print(dtype, nbits, zt, "rows", rows, flush=True)
        assert qz.StripeReduceTakes(rows, cols, nbits, zt, dtype)
        zeros = np.zeros((rows, cols), npdt, order="F")
        stripes, agg = [], None
        for w in range(workers):
            q, _ = oracle.quantize(datagen.normal(70 + w + extra, rows, cols, dtype=npdt), zeros, nbits, zt, threads=8)
            Q = QuantizedMatrix(rows, cols, nbits, 0, dtype=dtype)
            Q.from_numpy(q)
            stripes.append(Q)
            agg = oracle.unquantize(q, rows, cols, nbits, dtype=npdt, threads=8) if w == 0 else \
                oracle.unquantize(q, rows, cols, nbits, out=agg, add=True, threads=8)
        sres = datagen.normal(80 + extra, rows, cols, 0.002, dtype=npdt)
        S, Out = Matrix.from_numpy(sres), QuantizedMatrix(rows, cols, nbits, 0, dtype=dtype)
        Out.buffer.fill_(0xA5)
        qz.StripeReduceAsync(stripes, 0, S, Out, zt)
        qz.WaitStripeReduceDone()
        torch.cuda.synchronize()
        parity.check_quantize(agg, sres, Out.to_numpy(), S.to_numpy(), nbits, zt)


@pytest.mark.parametrize("dtype,rows", [(F32, 102401), (F64, 51201)])
def test_recorded_launch_without_room_for_copies(dtype, rows):
    """7 strips x 4000 (2000) columns: the starting buffer of 1 MB holds one copy of the records and not two, and a stream
    under capture cannot wait for a larger one."""
    cols = 4000 if dtype == F32 else 2000
    gen = torch.Generator(device="cuda:0")
    gen.manual_seed(rows)
    g = torch.randn(rows * cols, generator=gen, device="cuda:0").to(dtype)
    r = torch.zeros(rows * cols, dtype=dtype, device="cuda:0")
    want = _quantize(MatrixQuantizerImpl.Create(0, False), g, r, rows, cols, 1, dtype, False)  # an eager launch takes the room
    qz = MatrixQuantizerImpl.Create(0, False)
    G, R, Q = Matrix(rows, cols, 0, g, dtype=dtype), Matrix(rows, cols, 0, r.clone(), dtype=dtype), QuantizedMatrix(rows, cols, 1, 0, dtype=dtype)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=torch.cuda.Stream()):
        qz.SetMainStream(torch.cuda.current_stream().cuda_stream)
        qz.QuantizeAsync(G, R, Q, R, False)
    for _ in range(3):
        R.data.zero_()
        Q.buffer.zero_()
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(Q.buffer, want[0]) and torch.equal(R.data.view(torch.uint8), want[1])


@pytest.mark.parametrize("recorded", [False, True])
@pytest.mark.parametrize("dtype,rows", [(F32, 102401), (F64, 51201)])
def test_no_memory_for_copies(dtype, rows, recorded):
    """7 strips x 4000 (2000) columns, whose records in one copy fit the starting buffer: where a larger one is refused, the launch takes that one copy in
    the buffer it has, whether a recorded launch uses it or not; what does not fit it is refused and leaves the buffer in use."""
    cols = 4000 if dtype == F32 else 2000
    gen = torch.Generator(device="cuda:0")
    gen.manual_seed(rows + 1)
    g = torch.randn(rows * cols, generator=gen, device="cuda:0").to(dtype)
    r = torch.zeros(rows * cols, dtype=dtype, device="cuda:0")
    small = (rows, 40)
    gs, rs = g[:rows * 40], r[:rows * 40]
    want, want_small = (_quantize(MatrixQuantizerImpl.Create(0, False), *x, 1, dtype, False) for x in ((g, r, rows, cols), (gs, rs) + small))
    qz = MatrixQuantizerImpl.Create(0, False)
    G, R, Q = Matrix(*small, 0, gs, dtype=dtype), Matrix(*small, 0, rs.clone(), dtype=dtype), QuantizedMatrix(*small, 1, 0, dtype=dtype)
    graph = torch.cuda.CUDAGraph()
    if recorded:
        with torch.cuda.graph(graph, stream=torch.cuda.Stream()):
            qz.SetMainStream(torch.cuda.current_stream().cuda_stream)
            qz.QuantizeAsync(G, R, Q, R, False)
        qz.SetMainStream(torch.cuda.current_stream().cuda_stream)
    qz._set_strip_scratch_limit(1 << 20)
    for step in range(3):
        got = _quantize(qz, g, r, rows, cols, 1, dtype, False)
        assert torch.equal(got[0], want[0]) and torch.equal(got[1], want[1]), step
        with pytest.raises(cntk_amd.QuantizerError):  # (twice the columns: more than the buffer holds even in one copy)
            _quantize(qz, *(torch.zeros(rows * cols * 2, dtype=dtype, device="cuda:0") for _ in range(2)), rows, cols * 2, 1, dtype, False)
        if recorded:
            R.data.zero_()
            Q.buffer.zero_()
            torch.cuda.synchronize()
            graph.replay()
            torch.cuda.synchronize()
            assert torch.equal(Q.buffer, want_small[0]) and torch.equal(R.data.view(torch.uint8), want_small[1]), step
    qz._set_strip_scratch_limit(1 << 40)
    got = _quantize(qz, g, r, rows, cols, 1, dtype, False)
    assert torch.equal(got[0], want[0]) and torch.equal(got[1], want[1])
