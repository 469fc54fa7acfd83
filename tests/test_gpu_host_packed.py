"""Packed matrices in host memory: coherent pinned memory is written and read by the kernels where it lies, any other goes through
the handle's staging buffer. Either way the bytes are those of a packed matrix in device memory (whose parity with the oracle
the other files check), and nothing outside the packed matrix is touched."""
import ctypes

import pytest
import torch

import cntk_amd
from cntk_amd import Matrix, MatrixQuantizerImpl, QuantizedMatrix, qcol_bytes

pytestmark = pytest.mark.gpu

# (rows, columns, bits): what decides the kernels -- 255 / 256 QWords per column, columns in runs of 16 x 8 (127 / 128 / 129 /
# 260), tile decoder against row-major one (1023 / 1024 columns from 1664 rows on), short columns, one column, strips
SHAPES = [(512, 512, 1), (2048, 127, 1), (2048, 128, 1), (2048, 260, 1), (2048, 1025, 1), (2049, 129, 2), (1664, 1023, 1),
          (8160, 40, 1), (8192, 40, 1), (1023, 130, 8), (1024, 130, 8), (1, 1, 1), (7, 5000, 4), (16, 300, 1), (16, 98305, 4), (3, 98304, 16), (147, 999, 1), (20001, 9, 2),
          (110000, 3, 1), (33, 40, 32), (131071, 3, 4), (131072, 2, 1), (200003, 3, 8), (131075, 2, 32), (6000, 70, 1), (1800, 33, 4)]
SHAPES_F64 = [(2048, 130, 1), (511, 1025, 1), (8128, 20, 1), (8192, 20, 1), (3, 700, 4), (9001, 17, 8), (65537, 3, 1), (100003, 2, 8), (65536, 2, 64), (1500, 40, 4), (3000, 50, 2)]


# hipHostMalloc's flags, and whether the memory is coherent
DEFAULT, PORTABLE, MAPPED, WRITE_COMBINED, COHERENT, NON_COHERENT = 0, 1, 2, 4, 0x40000000, 0x80000000
KINDS = {"default": (DEFAULT, True), "mapped": (MAPPED, True), "portable_coherent": (PORTABLE | COHERENT, True), "portable": (PORTABLE, False),
         "write_combined": (WRITE_COMBINED, False), "non_coherent": (NON_COHERENT, False), "non_coherent_mapped": (NON_COHERENT | MAPPED, False)}


class HostMemory:
    """A byte tensor over memory of hipHostMalloc."""

    def __init__(self, size, flags):
        self.hip, self.at = ctypes.CDLL("libamdhip64.so"), ctypes.c_void_p()
        assert self.hip.hipHostMalloc(ctypes.byref(self.at), ctypes.c_size_t(size), ctypes.c_uint(flags)) == 0
        self.bytes = torch.frombuffer((ctypes.c_ubyte * size).from_address(self.at.value), dtype=torch.uint8)

    def free(self):
        torch.cuda.synchronize()
        assert self.hip.hipHostFree(self.at) == 0


def pinned_slice(size, before):
    """A byte tensor in pinned memory inside a larger allocation, and that allocation."""
    whole = torch.full((before + size + 256,), 0x5A, dtype=torch.uint8, pin_memory=True)
    return whole[before:before + size], whole


@pytest.mark.parametrize("dedicated", [False, True], ids=["main_stream", "dedicated_stream"])
@pytest.mark.parametrize("shape", SHAPES, ids=["%dx%d_%dbit" % s for s in SHAPES])
def test_float(shape, dedicated):
    check(*shape, torch.float32, dedicated)


@pytest.mark.parametrize("shape", SHAPES, ids=["%dx%d_%dbit" % s for s in SHAPES])
def test_float_at_four_bytes(shape):
    """The packed matrix at the alignment of a value and no better, as a transport's message may have it."""
    check(*shape, torch.float32, False, before=4 * 27)


@pytest.mark.parametrize("shape", SHAPES_F64, ids=["%dx%d_%dbit" % s for s in SHAPES_F64])
def test_double(shape):
    check(*shape, torch.float64, False)


def check(rows, cols, nbits, dtype, dedicated, before=8 * 13):
    qz = MatrixQuantizerImpl.Create(0, dedicated)
    gen = torch.Generator(device="cuda:0")
    gen.manual_seed(rows * 131 + cols)
    size = qcol_bytes(nbits, rows, dtype) * cols
    n = rows * cols
    g = torch.randn(n, generator=gen, device="cuda:0", dtype=dtype)
    G = Matrix(rows, cols, 0, g)
    pinned, whole = pinned_slice(size, before)
    pageable = torch.zeros(size, dtype=torch.uint8)
    places = {"device": QuantizedMatrix(rows, cols, nbits, 0, dtype=dtype),
              "pinned": QuantizedMatrix(rows, cols, nbits, cntk_amd.CPUDEVICE, pinned, dtype=dtype),
              "pageable": QuantizedMatrix(rows, cols, nbits, cntk_amd.CPUDEVICE, pageable, dtype=dtype)}
    res = {k: Matrix(rows, cols, dtype=dtype) for k in places}
    out = {k: Matrix(rows, cols, dtype=dtype) for k in places}
    torch.cuda.synchronize()
    for step in range(2):  # the residual carried once, the second result added to the first
        for k, q in places.items():
            qz.QuantizeAsync(G, res[k], q, res[k], False)
            qz.WaitQuantizeAsyncDone()
            if k == "pinned":
                # the host may read, move and write back what it was waited for
                copy = q.buffer.clone()
                q.buffer.fill_(0)
                q.buffer.copy_(copy)
            qz.UnquantizeAsync(q, out[k], add=step > 0)
            qz.WaitUnquantizeAsyncDone()
        torch.cuda.synchronize()
        for k in ("pinned", "pageable"):
            assert torch.equal(places[k].buffer, places["device"].buffer.cpu()), k
            assert torch.equal(res[k].data, res["device"].data), k
            assert torch.equal(out[k].data, out["device"].data), k
    assert bool((whole[:before] == 0x5A).all()) and bool((whole[before + size:] == 0x5A).all())


# one shape per decoder that reads host memory: the LDS-free row-major one (256 QWords of 4 bytes, 128 of 8), the tile decoder, the
# decoder of the matrix in device memory
REWRITE = [(torch.float32, (8192, 40, 1)), (torch.float32, (512, 512, 1)), (torch.float32, (2048, 127, 1)), (torch.float32, (300, 64, 8)),
           (torch.float64, (8192, 20, 1)), (torch.float64, (511, 1025, 1)), (torch.float64, (2000, 40, 1))]


@pytest.mark.parametrize("kind", list(KINDS))
@pytest.mark.parametrize("dtype,shape", REWRITE, ids=["%s_%dx%d_%dbit" % (("f32" if t == torch.float32 else "f64",) + s) for t, s in REWRITE])
def test_host_rewrites_between_decodes(dtype, shape, kind):
    """What a transport does: the packed matrix leaves, another worker's arrives in the same buffer and is decoded from there."""
    rows, cols, nbits = shape
    flags, coherent = KINDS[kind]
    size = qcol_bytes(nbits, rows, dtype) * cols
    memory = HostMemory(size, flags)
    qz, other = MatrixQuantizerImpl.Create(0, False), MatrixQuantizerImpl.Create(0, False)
    gen = torch.Generator(device="cuda:0")
    gen.manual_seed(rows + nbits)
    here = QuantizedMatrix(rows, cols, nbits, cntk_amd.CPUDEVICE, memory.bytes, dtype=dtype)
    there = QuantizedMatrix(rows, cols, nbits, 0, dtype=dtype)
    out, expected = Matrix(rows, cols, dtype=dtype), Matrix(rows, cols, dtype=dtype)
    for step in range(3):
        g = [Matrix(rows, cols, 0, torch.randn(rows * cols, generator=gen, device="cuda:0", dtype=dtype)) for _ in range(2)]
        zero = Matrix(rows, cols, dtype=dtype)
        left = Matrix(rows, cols, dtype=dtype)
        qz.QuantizeAsync(g[0], zero, here, left, False)
        qz.WaitQuantizeAsyncDone()
        sent = memory.bytes.clone()
        other.QuantizeAsync(g[0], zero, there, left, False)
        other.WaitQuantizeAsyncDone()
        assert torch.equal(sent, there.buffer.cpu()), ("sent", step)
        for received in (1, 0):  # the other matrix, then the first one again
            other.QuantizeAsync(g[received], zero, there, left, False)
            other.UnquantizeAsync(there, expected)
            other.WaitUnquantizeAsyncDone()
            memory.bytes.copy_(there.buffer.cpu())
            qz.UnquantizeAsync(here, out)
            qz.WaitUnquantizeAsyncDone()
            assert torch.equal(out.data, expected.data), ("decoded", step, received)
    # coherent memory is used in place, what the host and the device may see differently is copied
    staged = cntk_amd.lib().cntkq_debug_staging_bytes(qz._h)
    assert staged == 0 if coherent else staged >= size
    memory.free()


@pytest.mark.parametrize("kind", ["default", "non_coherent"])
def test_order_across_main_streams(kind):
    """A handle's host-resident packed matrix is decoded after it was written, and written twice in the order of the calls, also where
    the caller changes the handle's main stream in between without waiting."""
    rows, cols = 2048, 300
    size = qcol_bytes(1, rows) * cols
    memory = HostMemory(size, KINDS[kind][0])
    qz = MatrixQuantizerImpl.Create(0, False)
    gen = torch.Generator(device="cuda:0")
    gen.manual_seed(3)
    g = [Matrix(rows, cols, 0, torch.randn(rows * cols, generator=gen, device="cuda:0")) for _ in range(2)]
    zero, left = Matrix(rows, cols), Matrix(rows, cols)
    here = QuantizedMatrix(rows, cols, 1, cntk_amd.CPUDEVICE, memory.bytes)
    packed, expected = [], []
    for m in g:
        there, e = QuantizedMatrix(rows, cols, 1, 0), Matrix(rows, cols)
        qz.QuantizeAsync(m, zero, there, left, False)
        qz.UnquantizeAsync(there, e)
        packed.append(there)
        expected.append(e)
    out = [Matrix(rows, cols), Matrix(rows, cols)]
    left2 = Matrix(rows, cols)
    first, second = torch.cuda.Stream(), torch.cuda.Stream()
    torch.cuda.synchronize()
    for step in range(2):
        memory.bytes.zero_()
        with torch.cuda.stream(first):
            torch.cuda._sleep(20000000)  # the write starts some milliseconds after the calls below were made
        qz.SetMainStream(first.cuda_stream)
        qz.QuantizeAsync(g[0], zero, here, left, False)
        qz.SetMainStream(second.cuda_stream)
        qz.UnquantizeAsync(here, out[0])
        qz.WaitUnquantizeAsyncDone()
        assert torch.equal(out[0].data, expected[0].data)
        with torch.cuda.stream(first):
            torch.cuda._sleep(20000000)
        qz.SetMainStream(first.cuda_stream)
        qz.QuantizeAsync(g[0], zero, here, left, False)
        qz.SetMainStream(second.cuda_stream)
        qz.QuantizeAsync(g[1], zero, here, left2, False)
        qz.UnquantizeAsync(here, out[1])
        torch.cuda.synchronize()
        assert torch.equal(memory.bytes, packed[1].buffer.cpu())
        assert torch.equal(out[1].data, expected[1].data)
    memory.free()


@pytest.mark.parametrize("kind", ["default", "non_coherent"])
def test_recorded_calls_are_refused(kind):
    """Calls with a host-resident packed matrix are not recorded into a graph, wherever the memory is written from."""
    rows, cols = 512, 8
    memory = HostMemory(qcol_bytes(1, rows) * cols, KINDS[kind][0])
    qz = MatrixQuantizerImpl.Create(0, False)
    here = QuantizedMatrix(rows, cols, 1, cntk_amd.CPUDEVICE, memory.bytes)
    g, res, out = Matrix(rows, cols), Matrix(rows, cols), Matrix(rows, cols)
    word = torch.zeros(1, device="cuda:0")
    torch.cuda.synchronize()
    side, graph = torch.cuda.Stream(), torch.cuda.CUDAGraph()
    qz.SetMainStream(side.cuda_stream)
    with torch.cuda.graph(graph, stream=side):
        word.add_(1.0)
        with pytest.raises(cntk_amd.QuantizerLogicError, match="host-resident packed matrix cannot be recorded"):
            qz.QuantizeAsync(g, res, here, res, False)
        with pytest.raises(cntk_amd.QuantizerLogicError, match="host-resident packed matrix cannot be recorded"):
            qz.UnquantizeAsync(here, out)
    memory.free()
