"""The register grids of the gradient-set calls (columns kept in registers on 256 or 1024 threads, many matrices per launch):
the bytes are those of one call per matrix, whose parity with the oracle the other tests hold. Needs an MI355X."""
import numpy as np
import pytest
import torch

import datagen
import parity
from cntk_amd import Matrix, MatrixQuantizerImpl, QuantizedMatrix

pytestmark = pytest.mark.gpu

# heights on both sides of every line between the kernels: edge elements on 256 threads (2049 .. 7168 rows not a multiple of 4) and
# on 1024 (up to 24576 rows by pieces per thread, 102368 in launches of their own), whole pieces on 256 threads with more
# than six pieces each (6148 .. 14336 rows) and on 1024
EDGE = [(2049, 40), (4071, 5), (4099, 3), (7166, 9), (7169, 3), (9305, 7), (12258, 2), (16359, 2), (16361, 3), (24547, 2), (24555, 1)]
WHOLE = [(6148, 70), (8192, 40), (9304, 33), (14308, 36), (14336, 34), (14340, 3), (16384, 2), (24576, 2), (24580, 1)]
# doubles: from 6145 rows on 1024 threads, up to six pieces each in the shared grid
DOUBLE = [(6145, 3), (6883, 1), (6884, 40), (8187, 2), (8192, 3), (12258, 2), (12288, 2), (12303, 2), (300, 30), (6144, 2)]
SMALL = [(64, 64), (429, 37), (21, 960), (2048, 1), (9280, 1), (13000, 2)]


def _matrices(shapes, nbits, seed, dtype=torch.float32):
    # slices of one allocation at odd offsets: the columns of a matrix start anywhere within 16 bytes, the same in both runs
    gen = torch.Generator(device="cuda:0")
    gen.manual_seed(datagen.case_seed(seed))
    out = []
    for i, (r, c) in enumerate(shapes):
        off = 0 if r % 4 == 0 else i % 4
        g, res = [(torch.randn(r * c + 4, generator=gen, device="cuda:0") * s).to(dtype)[off:off + r * c] for s in (0.01, 0.002)]
        out.append((Matrix(r, c, 0, g, dtype=dtype), Matrix(r, c, 0, res, dtype=dtype), QuantizedMatrix(r, c, nbits, 0, dtype=dtype)))
    return out


@pytest.mark.parametrize("nbits,zt", [(1, False), (1, True), (2, False), (8, False), (16, False)])
@pytest.mark.parametrize("shapes", [EDGE, WHOLE, EDGE[:2] + SMALL, EDGE + WHOLE + SMALL], ids=["edge", "whole", "few", "all"])
def test_quantize(shapes, nbits, zt):
    _check_quantize(shapes, nbits, zt, torch.float32)


@pytest.mark.parametrize("nbits,zt", [(1, False), (1, True), (4, False), (16, False)])
def test_quantize_of_few_columns_of_six_pieces(nbits, zt):
    """At most 32 columns of 5124 to 6144 rows (6140: not on lines, so one piece more per thread) are in registers, the next height is staged in memory."""
    _check_quantize([(5124, 1), (5632, 32), (6112, 7), (6140, 5), (6144, 20), (6176, 32)] + SMALL, nbits, zt, torch.float32)


@pytest.mark.parametrize("nbits", [1, 8])
def test_quantize_of_few_tall_columns_alone(nbits):
    """A large set made of nothing but the few tall columns that would be staged in memory: there is nothing else to hide them, so they
    share a register grid (64 x 14336 x 32 at 1 bit: 108 us staged, 65 us so)."""
    _check_quantize([(14336, 32)] * 55 + [(13312, 31)] * 4, nbits, False, torch.float32)


@pytest.mark.parametrize("nbits,zt", [(1, False), (1, True), (4, False), (32, False)])
def test_quantize_doubles(nbits, zt):
    _check_quantize(DOUBLE, nbits, zt, torch.float64)


def _check_quantize(shapes, nbits, zt, dtype):
    qz = MatrixQuantizerImpl.Create(0, False)
    one, many = _matrices(shapes, nbits, nbits, dtype), _matrices(shapes, nbits, nbits, dtype)
    for _ in range(2):
        for g, r, q in one:
            qz.QuantizeAsync(g, r, q, r, zt)
        qz.QuantizeBatchAsync([(g, r, q, r) for g, r, q in many], zt)
        qz.WaitQuantizeAsyncDone()
        torch.cuda.synchronize()
        for (_, r1, q1), (_, r2, q2), shape in zip(one, many, shapes):
            assert np.array_equal(q1.to_numpy(), q2.to_numpy()), ("packed", shape)
            assert parity.bits_equal(r1.to_numpy(), r2.to_numpy()), ("residual", shape)


def _stripes(qz, shapes, nbits, zt, k, dtype=torch.float32):
    workers = [_matrices(shapes, nbits, 20 * w + nbits, dtype) for w in range(k)]
    for ms in workers:
        for g, r, q in ms:
            qz.QuantizeAsync(g, r, q, r, zt)
    sres = [r for _, r, _ in _matrices(shapes, nbits, 999, dtype)]
    agg = [Matrix(r, c, dtype=dtype) for r, c in shapes]
    return [[ms[i][2] for ms in workers] for i in range(len(shapes))], sres, agg


@pytest.mark.parametrize("nbits,zt,k", [(1, False, 1), (1, True, 8), (1, False, 9), (2, False, 3), (8, False, 1), (8, False, 8), (16, False, 2)])
@pytest.mark.parametrize("shapes", [EDGE, WHOLE, EDGE[:2] + SMALL, EDGE + WHOLE + SMALL], ids=["edge", "whole", "few", "all"])
def test_stripe_reduction(shapes, nbits, zt, k):
    _check_stripe_reduction(shapes, nbits, zt, k, torch.float32)


@pytest.mark.parametrize("nbits,zt,k", [(1, True, 1), (1, False, 8), (8, False, 3), (32, False, 2)])
def test_stripe_reduction_doubles(nbits, zt, k):
    _check_stripe_reduction(DOUBLE, nbits, zt, k, torch.float64)


def _check_stripe_reduction(shapes, nbits, zt, k, dtype):
    qz = MatrixQuantizerImpl.Create(0, False)
    owner = k // 2
    q1, s1, a1 = _stripes(qz, shapes, nbits, zt, k, dtype)
    q2, s2, a2 = _stripes(qz, shapes, nbits, zt, k, dtype)
    for q, s, a in zip(q1, s1, a1):
        qz.StripeReduceAsync(q, owner, s, q[owner], zt, agg_out=a)
    qz.StripeReduceBatchAsync([(q, s, q[owner], a) for q, s, a in zip(q2, s2, a2)], owner, zt)
    qz.WaitStripeReduceDone()
    torch.cuda.synchronize()
    for i, shape in enumerate(shapes):
        assert np.array_equal(q1[i][owner].to_numpy(), q2[i][owner].to_numpy()), ("packed", shape)
        assert parity.bits_equal(s1[i].to_numpy(), s2[i].to_numpy()), ("stripe residual", shape)
        assert parity.bits_equal(a1[i].to_numpy(), a2[i].to_numpy()), ("aggregate", shape)


# a single worker's stripes: tiles and short columns, whole pieces up to 3 / 6 per thread on both sides of each line (with and without a line
# shift), the register grids, slices that start anywhere within 16 bytes
SINGLE = [(16, 300), (300, 31), (512, 65), (1024, 40), (1028, 9), (2048, 33), (2052, 8), (3044, 9), (3068, 5), (3072, 9), (3076, 7), (4608, 11),
          (6116, 4), (6140, 3), (6144, 6), (6148, 70), (2049, 4), (2051, 6), (7166, 3), (9305, 2), (14336, 40), (16384, 2)]


@pytest.mark.parametrize("nbits,zt", [(1, False), (1, True), (2, False), (4, False), (8, False), (16, False), (32, False)])
def test_single_worker_stripes(nbits, zt):
    qz = MatrixQuantizerImpl.Create(0, False)
    shapes = [s for s in SINGLE if nbits < 32 or s[0] <= 14336]  # (32-bit codes: no stripes above)
    one, many = _stripes(qz, shapes, nbits, zt, 1), _stripes(qz, shapes, nbits, zt, 1)
    batch = qz.PrepareStripeReduceBatch([(q, s, q[0], a) for q, s, a in zip(*many)])
    for step in range(3):
        for q, s, a in zip(*one):
            qz.StripeReduceAsync(q, 0, s, q[0], zt, agg_out=a)
        qz.StripeReduceBatchAsync(batch, 0, zt)
        torch.cuda.synchronize()
        for i, shape in enumerate(shapes):
            assert np.array_equal(one[0][i][0].to_numpy(), many[0][i][0].to_numpy()), ("packed", shape, step)
            assert parity.bits_equal(one[1][i].to_numpy(), many[1][i].to_numpy()), ("stripe residual", shape, step)
            assert parity.bits_equal(one[2][i].to_numpy(), many[2][i].to_numpy()), ("aggregate", shape, step)


@pytest.mark.parametrize("nbits,k", [(1, 2), (4, 1), (8, 3)])
def test_stripes_called_again(nbits, k):
    """Called again a list is launched from its table, which also knows the stripes with launches of their own (too tall for the register
    grids; the only member of the general grids), while another list, without a table, comes in between."""
    qz = MatrixQuantizerImpl.Create(0, False)
    shapes = [(24580, 2), (9305, 3), (64, 64), (7169, 2), (24555, 1), (14340, 2)]
    lists = [_stripes(qz, s, nbits, False, k) for s in (shapes, shapes, [(24580, 1), (40, 3)])]
    sets = [qz.PrepareStripeReduceBatch([(q, s, q[0], a) for q, s, a in zip(*l)]) for l in lists]
    for _ in range(3):
        for q, s, a in zip(*lists[0]):
            qz.StripeReduceAsync(q, 0, s, q[0], False, agg_out=a)
        qz.StripeReduceBatchAsync(sets[1], 0, False)
        qz.StripeReduceBatchAsync(sets[2], 0, False)
        torch.cuda.synchronize()
        for i, shape in enumerate(shapes):
            (q1, s1, a1), (q2, s2, a2) = [[part[i] for part in l] for l in lists[:2]]
            assert np.array_equal(q1[0].to_numpy(), q2[0].to_numpy()), ("packed", shape)
            assert parity.bits_equal(s1.to_numpy(), s2.to_numpy()), ("stripe residual", shape)
            assert parity.bits_equal(a1.to_numpy(), a2.to_numpy()), ("aggregate", shape)


def test_stripes_with_a_forced_path():
    """A kernel path forced on a handle is that of the stripes that are no members of the general grids, also where the list was called
    before without it."""
    qz = MatrixQuantizerImpl.Create(0, False)
    shapes = [(4099, 3), (5001, 2), (6147, 4)]  # on the tile path another order of additions: other bounds
    one, many = _stripes(qz, shapes, 4, False, 2), _stripes(qz, shapes, 4, False, 2)
    batch = qz.PrepareStripeReduceBatch([(q, s, q[0], a) for q, s, a in zip(*many)])
    for path in (0, 1, 0):
        qz._set_tuning(quantize_path=path)
        for q, s, a in zip(*one):
            qz.StripeReduceAsync(q, 0, s, q[0], False, agg_out=a)
        qz.StripeReduceBatchAsync(batch, 0, False)
        torch.cuda.synchronize()
        for i, shape in enumerate(shapes):
            assert np.array_equal(one[0][i][0].to_numpy(), many[0][i][0].to_numpy()), ("packed", path, shape)
            assert parity.bits_equal(one[1][i].to_numpy(), many[1][i].to_numpy()), ("stripe residual", path, shape)


def test_recorded_stripes_without_a_table():
    """Stripes that each had a launch of their own could always be recorded without an eager call before; they still can."""
    _check_recorded([(9305, 3), (7169, 2), (4099, 2)], 2, 2, eager_first=False)


@pytest.mark.parametrize("shapes,nbits,k", [([(8192, 40), (40, 1)], 2, 1), ([(14336, 34), (64, 64)], 8, 2), ([(9304, 33), (2048, 3), (9305, 2)], 4, 1),
                                            ([(8192, 40), (9304, 5)], 2, 2), ([(6148, 70), (429, 37), (21, 960)], 2, 1)])
def test_recorded_stripes_after_a_call(shapes, nbits, k):
    """A list that was called once can be recorded, whatever the call made of it: a layer of whole pieces and its bias are a member of
    a register grid and one of the general grids, with nothing to share a grid with in either, so that the call builds no table."""
    _check_recorded(shapes, nbits, k, eager_first=True)


def _check_recorded(shapes, nbits, k, eager_first):
    qz = MatrixQuantizerImpl.Create(0, False)
    q1, s1, a1 = _stripes(qz, shapes, nbits, False, k)
    q2, s2, a2 = _stripes(qz, shapes, nbits, False, k)

    def one_by_one():
        for q, s, a in zip(q1, s1, a1):
            qz.StripeReduceAsync(q, 0, s, q[0], False, agg_out=a)
        qz.WaitStripeReduceDone()

    def as_a_set():
        qz.StripeReduceBatchAsync([(q, s, q[0], a) for q, s, a in zip(q2, s2, a2)], 0, False)

    if eager_first:
        one_by_one()
        as_a_set()
    torch.cuda.synchronize()
    side, graph = torch.cuda.Stream(), torch.cuda.CUDAGraph()
    qz.SetMainStream(side.cuda_stream)
    with torch.cuda.graph(graph, stream=side):
        as_a_set()
    qz.SetMainStream(torch.cuda.current_stream().cuda_stream)
    for _ in range(3):
        one_by_one()
        graph.replay()
        torch.cuda.synchronize()
        for i, shape in enumerate(shapes):
            assert np.array_equal(q1[i][0].to_numpy(), q2[i][0].to_numpy()), ("packed", shape)
            assert parity.bits_equal(s1[i].to_numpy(), s2[i].to_numpy()), ("stripe residual", shape)
            assert parity.bits_equal(a1[i].to_numpy(), a2[i].to_numpy()), ("aggregate", shape)
