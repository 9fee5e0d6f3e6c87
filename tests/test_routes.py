"""Which launches a product becomes, by the planner alone: host code, no GPU."""
import ctypes

import pytest

from tritonformer_amd import _lib

PLAIN, BITS, MASK = 0, 1, 2
CUS = 256


def route(m, n, k, kind=PLAIN, vec=True):
    """[(columns, configuration, slices)] of the launches on a chip of 256 CUs."""
    rows = (ctypes.c_int64 * 16)()
    count = _lib.load_diag().tf_diag_gemm_route(CUS, m, n, k, int(vec), kind, rows, 4)
    assert count > 0
    return [tuple(rows[4 * i:4 * i + 3]) for i in range(count)]


def tiles(m, n, tm, tn):
    return -(-m // tm) * -(-n // tn)


@pytest.mark.parametrize("m,n,k", [(3968, 4160, 512), (1920, 8512, 2304), (384, 34496, 2048), (896, 36416, 128),
                                   (312, 35136, 704)])
@pytest.mark.parametrize("kind", [PLAIN, BITS])
def test_the_remainder_of_a_cut_is_priced_like_the_whole(m, n, k, kind):
    """Two rounds of 128x128 tiles, the second nearly empty, or one round of 256x256 tiles and a few columns: the cost model
    of whole rounds finds both nearly equal (the cut has to win by 3 us) and keeps the one launch.  Counted at what it costs on
    the idle chip, a second scale, the remainder makes the cut look cheaper, and splits its contraction where the launch did
    not."""
    assert route(m, n, k, kind) == [(n, 3, 1)]


@pytest.mark.parametrize("m,n,k,kind,want", [
    # one round of large tiles at the most: the tile that fills it (64x64: 6, 128x64: 7), slices those of the larger tile
    (16, 256, 256, PLAIN, [(256, 6, 1)]),
    (128, 1024, 1024, PLAIN, [(1024, 6, 1)]),
    (128, 1024, 4096, PLAIN, [(1024, 6, 4)]),
    (128, 1024, 4096, MASK, [(1024, 6, 1)]),
    (128, 768, 8192, PLAIN, [(768, 6, 8)]),
    (960, 768, 768, PLAIN, [(768, 6, 1)]),
    (512, 256, 256, BITS, [(256, 6, 1)]),
    (2048, 1024, 1024, PLAIN, [(1024, 7, 1)]),
    # whole rounds
    (2048, 4096, 1024, PLAIN, [(4096, 4, 1)]),
    (4096, 1536, 6144, PLAIN, [(1536, 4, 1)]),
    (8192, 1024, 4096, PLAIN, [(1024, 4, 1)]),
    (8192, 4096, 1024, BITS, [(4096, 2, 1)]),
    # whole rounds and a remainder
    (8192, 3072, 1024, PLAIN, [(2048, 2, 1), (1024, 4, 1)]),
    (4096, 6144, 1536, BITS, [(4096, 2, 1), (2048, 4, 1)]),
    (1024, 50304, 8192, PLAIN, [(49152, 2, 1), (1152, 4, 7)]),
])
def test_tiles_of_a_product(m, n, k, kind, want):
    assert route(m, n, k, kind) == want


def test_operands_of_any_alignment_take_the_register_staged_tiles():
    assert route(4113, 2051, 1733, vec=False) == [(2051, 0, 1)]
    assert route(100, 333, 129, vec=False) == [(333, 1, 1)]
    assert all(cfg < 2 for _, cfg, _ in route(100, 328, 129))  # contraction not a multiple of 64


def test_small_tiles_serve_no_more_than_one_round_of_larger_ones():
    for m in (16, 64, 200, 520, 1024, 1800, 3072, 4096):
        for n in (64, 328, 768, 1024, 2304, 4096, 6144):
            for k in (64, 512, 1024, 4096):
                for _, cfg, splits in route(m, n, k):
                    if cfg in (6, 7):
                        assert min(tiles(m, n, 256, 128), tiles(m, n, 256, 256)) * splits <= CUS


def test_route_rejects_bad_arguments():
    f, rows = _lib.load_diag().tf_diag_gemm_route, (ctypes.c_int64 * 4)()
    assert f(0, 64, 64, 64, 1, 0, rows, 1) == -1 and f(256, 0, 64, 64, 1, 0, rows, 1) == -1
    assert f(256, 64, 64, 64, 1, 4, rows, 1) == -1 and f(256, 64, 64, 64, 1, 0, None, 1) == -1
    assert f(256, 8192, 3072, 1024, 1, 0, rows, 1) == -1  # two launches, room for one


@pytest.mark.parametrize("m,n,k,vec,want", [
    # operands of any alignment: 256x128 tiles where these fill one round, 256x256 tiles for whole rounds, 128x128 for few
    (4113, 1733, 2051, False, [(1733, 8, 1)]),
    (2051, 1733, 4113, False, [(1733, 8, 2)]),
    (8192, 50257, 1024, False, [(50257, 0, 1)]),
    (100, 5001, 129, False, [(5001, 1, 1)]),
    # a short contraction is mostly start and write-out, which 128x128 tiles overlap; a long one holds 256x128 tiles up
    (7488, 2624, 64, True, [(2624, 3, 1)]),
    (4096, 2048, 8192, True, [(2048, 4, 1)]),
    (8192, 1024, 50304, True, [(1024, 2, 2)]),
])
def test_rates_of_the_tiles(m, n, k, vec, want):
    assert route(m, n, k, vec=vec) == want


@pytest.mark.parametrize("m,n,k,kind,vec,want", [
    # two rounds of 256x128 tiles take longer than one of 256x256, and long contractions longer than short ones by the step
    (8192, 2048, 12288, PLAIN, True, (2, 1)),
    (14976, 1984, 12800, PLAIN, True, (2, 1)),
    (11136, 960, 12224, PLAIN, True, (2, 1)),
    # one or two steps are start and write-out, which more and smaller tiles have less of; 128x64 tiles on just over one workgroup per CU
    (40, 1536, 64, PLAIN, True, (6, 1)),
    (7296, 560, 832, PLAIN, True, (4, 1)),
    (7432, 144, 3968, PLAIN, True, (4, 3)),
    # operands of any alignment, unsplit: 128x128 tiles up to one per CU, 256x128 where they would be more
    (1509, 105, 7035, MASK, False, (1, 1)),
    (2334, 1614, 9044, MASK, False, (1, 1)),
    (1563, 2665, 5116, MASK, False, (8, 1)),
    # split: 256x256 in slices
    (10712, 616, 6012, PLAIN, False, (0, 2)),
    (966, 7598, 9983, PLAIN, False, (0, 2)),
])
def test_tiles_that_were_the_slower_ones(m, n, k, kind, vec, want):
    """Each of these ran 1.05 to 1.5 times as long on the tiles that a fit to warm operands had taken."""
    assert route(m, n, k, kind, vec) == [(n, *want)]
