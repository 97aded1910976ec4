"""The launch shape of the x sweeps, from the host code itself: every tile fits
its threads and its LDS planes, the tiles and chunks cover the interior, and
32-bit byte offsets reach every plane of a chunk on the largest grids."""
import itertools

import pytest

import sweepshape


@pytest.fixture(scope="module")
def shape(tmp_path_factory):
    return sweepshape.build(tmp_path_factory.mktemp("shape"))


def columns(nzi, ntz):
    return [64] * (ntz - 1) + [nzi - 64 * (ntz - 1)]


@pytest.mark.parametrize("m", [1, 2, 3, 4])
def test_tiles(shape, m):
    sizes = sorted(set(range(2, 81)) | {127, 128, 129, 136, 137, 191, 200, 201, 513})
    for nzi, nyi, tile_y in itertools.product(sizes, (2, 3, 7, 8, 9, 15, 16, 17, 33, 100), (0, 4, 8, 16)):
        items = 16 if m == 2 else 0   # coefficients a surface row stages, one per thread
        s = shape((11 + 2 * m, nyi + 2 * m, nzi + 2 * m), m, (0, tile_y, 0), row_items=items)
        rows, threads = s['rows'], s['threads']
        case = (nzi, nyi, tile_y, s)
        cols = columns(nzi, s['ntz'])
        assert 0 < min(cols) and max(cols) <= 72 and (len(cols) == 1 or cols[-1] >= 9), case
        assert 1 <= rows <= (tile_y or 16) and rows * (s['tyn'] - 1) < nyi <= rows * s['tyn'], case
        assert threads % 64 == 0 and threads <= 512, case
        for c in set(cols):
            assert rows * c <= threads, case
            assert (rows + 2 * m) * (c + 2 * m) <= s['plane'], case
            # halo items: one per thread, a second where the kernel takes one
            assert 2 * m * c <= threads * (2 if s['second'] else 1) and 2 * m * rows <= threads, case
        assert items * rows * (2 if len(cols) == 1 else 1) <= threads, case
        assert s['nb'] == s['ntz'] * s['tyn'] * -(-11 // s['xc']), case


@pytest.mark.parametrize("m", [1, 4])
@pytest.mark.parametrize("elem", [2, 4, 8])
def test_chunks_within_32_bit_offsets(shape, m, elem):
    """grids up to 2^31 elements, chunks chosen and asked for: a thread's byte
    offset of 8 bytes per element, plane to plane, stays below 2^32"""
    for dims in ((1280, 1280, 1280), (2, 2, 32768), (60, 6000, 5900), (10, 14000, 15000), (32768, 250, 250),
                 (250, 32768, 200)):
        dims = tuple(max(d, 2 * m + 2) for d in dims)
        for x_chunk in (0, 1, 8, 100, 1 << 20):
            s = shape(dims, m, (0, 0, x_chunk), elem=elem)
            plane = dims[1] * s['pitch']
            assert dims[0] * plane < 1 << 31, dims
            xi = dims[0] - 2 * m
            assert 1 <= s['xc'] <= xi and s['nb'] == s['ntz'] * s['tyn'] * -(-xi // s['xc'])
            assert s['xc'] * plane * 8 < 1 << 32, (dims, x_chunk, s)
