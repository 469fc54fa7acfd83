"""Which kernel a call takes, on both sides of the lines that the rules draw. The rules are host code: no device is needed."""
import ctypes

import pytest

import cntk_amd


def short(rows, cols, nbits, workers=0, double=0):
    L = cntk_amd.lib()
    return bool(L.cntkq_debug_short_columns_f64(rows, cols, nbits) if double else L.cntkq_debug_short_columns(rows, cols, nbits, workers))


@pytest.mark.parametrize("nbits", [1, 2, 4, 8, 16, 32])
def test_short_columns_of_one_qword(nbits):
    """One thread per column whatever their number, as far as a column is one QWord."""
    last = min(16, 32 // nbits)
    for rows in range(1, last + 1):
        for cols in (1, 300, 16000, 10 ** 6):
            assert short(rows, cols, nbits)
            for workers in (1, 4):
                assert short(rows, cols, nbits, workers)
    assert not short(17, 10 ** 6, nbits) and not short(17, 10 ** 6, nbits, 1)


@pytest.mark.parametrize("rows,nbits,qwords", [(9, 4, 2), (16, 4, 2), (5, 8, 2), (16, 8, 4), (3, 16, 2), (12, 16, 6), (2, 32, 2), (6, 32, 6)])
def test_short_columns_of_several_qwords(rows, nbits, qwords):
    """... and with more QWords only where the columns fill the device (16 x 16000 at 8 bits: 5.2 us, the tile kernel 3.4)."""
    for cols in (1, 300, 16000, 64000, 98303):
        assert not short(rows, cols, nbits)
        for workers in (1, 2, 4, 8):
            assert not short(rows, cols, nbits, workers)
    assert short(rows, 98304, nbits)
    for workers in (1, 2, 4, 8, 9):
        assert short(rows, 98304, nbits, workers) == (workers <= 8 and qwords <= (5 if workers <= 4 else 3))


@pytest.mark.parametrize("rows,nbits", [(13, 16), (16, 16), (7, 32), (8, 32), (16, 32)])
def test_short_columns_of_many_qwords(rows, nbits):
    """The tile kernels keep them (16 x 300000 at 32 bits and 8 workers: nine times faster)."""
    assert not short(rows, 10 ** 6, nbits) and not short(rows, 10 ** 6, nbits, 1) and not short(rows, 10 ** 6, nbits, 8)


def test_short_columns_at_two_bits_and_many_workers():
    assert short(12, 16000, 2, 16) and not short(12, 16000, 2, 17) and short(16, 16000, 2, 4) and not short(16, 16000, 2, 5)
    assert short(16, 32768, 2, 64) and short(16, 16000, 1, 64) and short(8, 16000, 4, 64)


def test_short_columns_of_doubles():
    assert short(10, 5, 1, double=1) and not short(11, 65535, 1, double=1) and short(11, 65536, 1, double=1) and not short(17, 10 ** 6, 1, double=1)
    assert not short(9, 98303, 8, double=1) and short(9, 98304, 8, double=1) and short(12, 98304, 16, double=1)
    assert not short(13, 10 ** 6, 16, double=1) and not short(4, 10 ** 6, 64, double=1)


# quantizer_kernels_batch.h, UnqKind
VEC4, SCALAR, SEGMENT, ROWS, TILE, DIRECT, FLAT = range(7)


def decoder(rows, cols, nbits, host=0, double=0):
    L = cntk_amd.lib()
    return (L.cntkq_debug_decoder_f64 if double else L.cntkq_debug_decoder)(rows, cols, nbits, host)


@pytest.mark.parametrize("rows,cols,nbits,kind", [
    (1663, 40, 1, TILE), (1664, 1024, 1, TILE), (1664, 1023, 1, ROWS), (6000, 1000, 1, ROWS), (8160, 1023, 1, ROWS), (8160, 1024, 1, TILE),
    (8161, 1023, 1, DIRECT), (3072, 100, 1, ROWS), (2048, 100, 1, DIRECT), (1800, 1023, 4, ROWS), (2304, 1023, 4, DIRECT), (1, 40, 1, TILE),
    (131071, 9, 8, DIRECT), (131072, 9, 8, SCALAR), (600000, 6, 1, SCALAR), (131072, 5000, 1, SCALAR)])
def test_decoder_out_of_host_memory(rows, cols, nbits, kind):
    """Every line crosses the bus once (6000 x 1000 at 1 bit took 72 us with the decoder of device memory, 33 with the column in LDS; 600000 x 6 at 8 bits 291 us
    row-major, 87 with a thread per QWord)."""
    assert decoder(rows, cols, nbits, host=1) == kind


@pytest.mark.parametrize("rows,cols,nbits,kind", [
    (1500, 1023, 4, TILE), (1663, 40, 1, TILE), (1666, 1023, 4, ROWS), (1666, 1024, 4, TILE), (3000, 600, 2, ROWS), (8160, 500, 1, DIRECT),
    (7000, 500, 1, ROWS), (65535, 9, 8, DIRECT), (65536, 9, 8, SCALAR), (600000, 6, 1, SCALAR)])
def test_decoder_of_doubles_out_of_host_memory(rows, cols, nbits, kind):
    assert decoder(rows, cols, nbits, host=1, double=1) == kind


@pytest.mark.parametrize("double,nbits,cols", [(0, 1, 96000), (0, 2, 400000), (0, 4, 1000000), (0, 8, 12000000), (1, 1, 48000), (1, 2, 128000),
                                               (1, 4, 500000), (1, 8, 8000000)])
def test_decoder_of_one_row(double, nbits, cols):
    """The tile decoder from this many columns on (1 x 4000 at 2 bits: 1.9 us without, 3.6 with it), for all of them in host memory."""
    few = decoder(1, cols - 1, nbits, double=double)
    assert few not in (TILE, ROWS, DIRECT, FLAT) and decoder(1, 4, nbits, double=double) not in (TILE, ROWS, DIRECT, FLAT)
    assert decoder(1, cols, nbits, double=double) == TILE and decoder(2, 4, nbits, double=double) == TILE
    assert decoder(1, 4, nbits, host=1, double=double) == TILE


def test_decoder_of_one_row_of_wide_codes():
    for nbits in (16, 32):
        assert decoder(1, 2 * 10 ** 7, nbits) == SCALAR and decoder(1, 2 * 10 ** 7, nbits, double=1) == SCALAR


def test_stripes_in_register_grids():
    """Whole pieces, more than six per thread: a single worker's, and at 1 bit up to eight workers' (9304 x 14 at 8 bits and 8 workers took
    25 us in the general grid, 35 in a register grid); odd heights and 1024 threads whatever the workers."""
    def shares(*a):
        return bool(cntk_amd.lib().cntkq_debug_stripe_shares_register_grid(*a))

    for rows in (6176, 9304, 14336):
        for cols in (1, 64, 1000):
            for nbits in (2, 4, 8, 16):
                assert shares(rows, cols, nbits, 1)
                assert not any(shares(rows, cols, nbits, k) for k in (2, 3, 4, 8))
            assert shares(rows, cols, 1, 1) and shares(rows, cols, 1, 8) and not shares(rows, cols, 1, 9)
    for nbits in (2, 8):
        assert shares(9305, 3, nbits, 4) and shares(20000, 3, nbits, 4) and shares(4099, 3, nbits, 8)
        assert not shares(4096, 3, nbits, 1) and not shares(2048, 3, nbits, 4)


def test_heights_of_few_tall_columns():
    """Staged in memory beside 8 M elements: 8192 rows 22.9 us, 26.1 with a register grid of their own; 14336 rows 33.0 and 27.6."""
    L = cntk_amd.lib()
    assert [L.cntkq_debug_staged_max_rows(b) for b in (1, 2, 4, 8, 16)] == [8192, 8192, 8192, 10240, 10240]


TILES, COLUMNS, STAGED, REGISTERS_6, LANES = 0, 1, 5, 7, 14
SMALL_LDS = 20480  # eight workgroups in a compute unit; a set's members above it may get a launch of their own


def member(rows, nbits, workers=0, double=0, cols=100, resident=0):
    """(kind, bytes of LDS) of a member of a set's general grid, one that fills the device or one that is resident as a whole."""
    L = cntk_amd.lib()
    lds = ctypes.c_size_t()
    kind = (L.cntkq_debug_set_member_f64 if double else L.cntkq_debug_set_member)(rows, cols, nbits, workers, resident, ctypes.byref(lds))
    return kind, lds.value


def tile_lds(rows, nbits, workers, double):
    """A column tile: at most 5120 floats or 2048 doubles, a few lanes' scratch, QWords where several threads share one, the workers' levels."""
    threads, most, word = (256, 2048, 64) if double else (256, 5120, 32)
    lanes = 8
    while lanes < threads and (rows > lanes * 32 or threads // lanes * rows > most):
        lanes *= 2
    columns, qwords = threads // lanes, -(-rows * nbits // word)
    values = (columns * rows + 1) & ~1 if double else (columns * rows + 7) & ~3
    words = columns * qwords if nbits <= (4 if double else 2) else 0
    return ((74 if double else 76) + values + words + 2 * workers * columns) * (8 if double else 4)


@pytest.mark.parametrize("double,workers", [(0, 0), (0, 1), (1, 0), (1, 1)])
def test_short_members_of_a_set_stay_in_their_grid(double, workers):
    """A short column is on lanes only where a compute unit holds as many of its workgroups as of the tiles that the member was before: 147 rows at 4 bits
    need 19.1 KB as tiles and 21.6 on lanes, and everything else of the grid would be given those too."""
    for nbits in (1, 2, 4, 8, 16, 32):
        for rows in range(17, 513 if double else 1024):
            kind, lds = member(rows, nbits, workers, double)
            tiles = tile_lds(rows, nbits, workers, double)
            assert kind in (TILES, LANES)
            assert kind == LANES or lds == tiles, (rows, nbits)
            assert 163840 // lds >= min(8, 163840 // tiles) and (lds <= SMALL_LDS or tiles > SMALL_LDS), (rows, nbits, lds, tiles)


def test_short_members_on_lanes():
    """ResNet-50's heights (64, 128, 147, 256, 512, 576) and an odd one."""
    lanes = {rows: [b for b in (1, 2, 4, 8, 16) if member(rows, b)[0] == LANES] for rows in (33, 64, 128, 147, 256, 512, 576)}
    assert lanes == {33: [1, 2, 4, 8, 16], 64: [1, 2, 4, 8, 16], 128: [1, 2, 4], 147: [1, 2], 256: [1, 2, 4], 512: [1, 2, 4], 576: [1, 2]}
    assert [b for b in (1, 2, 4, 8, 16) if member(147, b, 1)[0] == LANES] == [1, 2] and member(147, 1, 2)[0] == TILES


@pytest.mark.parametrize("workers", [0, 1])
def test_short_members_of_a_resident_grid(workers):
    """Their LDS costs nothing: on lanes whatever it is, also stripes of more than 1 M elements (300 x 3685 at 4 bits)."""
    for nbits in (1, 2, 4, 8, 16):
        for rows, cols in ((17, 1000), (147, 100), (300, 3685), (512, 512), (576, 2000), (1023, 1500)):
            assert member(rows, nbits, workers, cols=cols, resident=1)[0] == LANES
            assert member(min(rows, 512), nbits, workers, double=1, cols=cols, resident=1)[0] == LANES
    assert member(300, 4, 1, cols=3685)[0] == TILES and member(31, 1, 1, cols=10000, resident=1)[0] == TILES
    assert member(300, 4, 2, cols=100, resident=1)[0] == TILES


@pytest.mark.parametrize("nbits", [1, 2, 4, 8, 16])
def test_few_columns_of_a_set_that_registers_hold(nbits):
    """Up to six pieces for each of 256 threads: in registers however few there are; above, at most 32 columns are staged in memory."""
    for cols in (1, 32, 33, 400):
        assert member(5632, nbits, cols=cols)[0] == member(6144, nbits, cols=cols)[0] == REGISTERS_6
        assert member(6144, nbits, cols=cols)[1] <= SMALL_LDS
    assert member(6176, nbits, cols=32)[0] == STAGED


def on_lanes(rows, n, nbits, workers=0, double=0):
    L = cntk_amd.lib()
    return bool((L.cntkq_debug_lanes_f64 if double else L.cntkq_debug_lanes)(rows, max(1, n // rows), nbits, workers))


def test_quantize_on_lanes():
    for nbits in (1, 2, 4, 8, 16):
        for rows in (17, 33, 161, 512, 1023, 1280):
            assert on_lanes(rows, 10 ** 4, nbits) and on_lanes(rows, 4 * 10 ** 7, nbits)
        assert not on_lanes(16, 10 ** 6, nbits) and not on_lanes(1281, 10 ** 6, nbits)
    assert not on_lanes(512, 10 ** 6, 32)
    for nbits in (1, 2, 4, 8, 16, 32):  # doubles: 17 x 294117 at 16 bits 28.0 us with tiles, 30.2 on lanes
        assert on_lanes(17, 10 ** 6, nbits, double=1) and on_lanes(32, 10 ** 7, nbits, double=1) and on_lanes(512, 10 ** 7, nbits, double=1)
        assert on_lanes(31, 2 * 10 ** 6, nbits, double=1) == (nbits < 8) and not on_lanes(513, 10 ** 6, nbits, double=1)


@pytest.mark.parametrize("rows,n,nbits,most", [
    (64, 10 ** 6, 1, 16), (512, 10 ** 5, 1, 16), (576, 10 ** 6, 2, 12), (147, 10 ** 6, 4, 8), (1023, 10 ** 6, 8, 6), (512, 10 ** 5, 16, 6),
    (63, 500000, 4, 8), (32, 500000, 8, 5), (31, 120000, 2, 8), (17, 120000, 16, 5), (512, 1100000, 1, 2), (63, 600000, 1, 2), (31, 140000, 1, 2)])
def test_stripes_on_lanes_by_workers(rows, n, nbits, most):
    """Up to this many workers (512 x 1953 at 4 bits: 1.17 times as fast with 8 workers, 0.95 with 16; 32 x 31250 0.87 and 0.74)."""
    assert [k for k in range(1, 65) if on_lanes(rows, n, nbits, k)] == list(range(1, most + 1))


def test_short_members_beside_a_staged_column():
    """142 x 31690 at 1 bit beside 3 columns of 8000 rows staged in memory (4.5 M elements): 16.8 us with tiles, 19.3 on lanes; 10 M 26.8 and 26.3."""
    L = cntk_amd.lib()
    for rows, least in ((17, 0), (32, 0), (33, 5), (127, 5), (128, 8), (400, 8), (401, 5), (1279, 5)):
        assert L.cntkq_debug_lanes_beside_staged(rows, least << 20) and not (least and L.cntkq_debug_lanes_beside_staged(rows, (least << 20) - 1))


def test_large_stripes_on_lanes():
    """One and two workers above 1 M elements: with no fewer workgroups to a compute unit than tiles have (319 x 25078 at 16 bits: 28.8 us with tiles, 33.8 on
    lanes), two of them at 4 bits and more with most of a lane's elements there (65 x 46153 at 8 bits: 14.3 and 15.1 us)."""
    n = 8 * 10 ** 6
    for nbits in (1, 2):
        assert all(on_lanes(rows, n, nbits, k) for rows in (32, 65, 161, 512, 641) for k in (1, 2))
    for rows, nbits in ((319, 8), (1279, 4), (513, 16), (129, 16)):
        assert not on_lanes(rows, n, nbits, 1) and not on_lanes(rows, n, nbits, 2) and on_lanes(rows, 10 ** 6, nbits, 2)
    for rows in (65, 161, 321, 641):
        assert on_lanes(rows, n, 4, 1) and not on_lanes(rows, n, 4, 2)
    assert on_lanes(256, n, 4, 2) and not on_lanes(31, 300000, 1, 1) and on_lanes(31, 250000, 1, 1)


@pytest.mark.parametrize("rows,n,nbits,most", [
    (32, 500000, 4, 8), (512, 10 ** 5, 8, 6), (512, 10 ** 5, 16, 4), (200, 500000, 32, 4), (24, 500000, 1, 4), (24, 60000, 1, 8), (23, 10 ** 5, 1, 2),
    (512, 600000, 1, 2), (17, 10 ** 7, 32, 2)])
def test_stripes_of_doubles_on_lanes_by_workers(rows, n, nbits, most):
    assert [k for k in range(1, 65) if on_lanes(rows, n, nbits, k, double=1)] == list(range(1, most + 1))
