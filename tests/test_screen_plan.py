"""Where a screened search stores its sums and what it does with the columns behind them: decided on the host, from the workspace that was laid
out (no GPU)."""
import ctypes as C
import itertools

import pytest


def plan(lib, pkg, batch, rows, padding, k, dim=32):
    room, stored, ranges = C.c_uint64(), C.c_uint64(), C.c_int()
    pkg.check(lib.dsx_testing_screen_columns(batch, dim, rows, padding, k, C.byref(room), C.byref(stored), C.byref(ranges)))
    return room.value, stored.value, ranges.value


def around(x):
    return [x - 257, x - 8, x - 1, x, x + 1, x + 8, x + 300]


# the widths and products at which whole rows stop being stored
SHAPES = [(b, r) for b, r in itertools.chain(((b, r) for b in (1, 64, 512, 513, 1000, 4096) for edge in (8192, 131072, 1048576) for r in around(edge)),
                                             ((b, r) for b in (2000, 10000, 65600, 120000, 131073) for sums in (28, 30) for r in around((1 << sums) // b)),
                                             ((b, 49152 + 512 * k + r) for b in (257, 1024, 1700, 4096) for k in (1, 100, 150) for r in (-8, -1, 0, 1, 8)),
                                             ((b, r) for b in (257, 513, 1023) for k in (1, 100, 150, 256) for r in around(((1 << 26) + (k << 22)) // b)))]


@pytest.mark.parametrize("k", [1, 100, 256])
def test_what_is_stored_fits_what_was_laid_out(pkg, k):
    lib = pkg.load_library()
    for batch, rows in SHAPES:
        for padding in (0, 1, 4, 7, 8, 300, rows // 2, rows - 1):
            if padding >= rows:
                continue
            room, stored, ranges = plan(lib, pkg, batch, rows, padding, k)
            assert stored <= (room + 255) // 256 * 256 and stored <= room, (batch, rows, padding, k)


@pytest.mark.parametrize("k", [1, 100, 150, 256])
def test_every_search_ends_with_its_results(pkg, k):
    """Results come from the stored sums, or from the last of the ranges behind them: where the first block is everything there are none."""
    lib = pkg.load_library()
    for batch, rows in SHAPES + [(120000, 10000), (70000, 16384), (66000, 16380), (140000, 8192), (33000, 32768)]:
        for padding in (0, 7, 300, rows // 2, rows - 1):
            if padding < rows:
                room, stored, ranges = plan(lib, pkg, batch, rows, padding, k)
                assert ranges == (stored < rows - padding), (batch, rows, padding, k)


def test_where_sums_are_stored(pkg):
    """Up to 2^28 of them, for more than 256 rows of a wide table and small k up to fewer; beyond, ranges are the faster way."""
    lib = pkg.load_library()
    for batch, n, k, ranges in ((1024, 27278, 10, 0), (4096, 54271, 10, 0), (4096, 54272, 10, 1), (4, 1000000, 10, 0), (256, 1048576, 10, 0), (4096, 65537, 10, 1), (4096, 131072, 10, 1),
                                (512, 1000000, 10, 1), (4096, 1000000, 10, 1), (2049, 131072, 100, 1), (2048, 131072, 100, 0), (2048, 131072, 10, 1),
                                (4096, 49663, 1, 0), (4096, 49664, 1, 1), (1024, 65536, 1, 0), (1024, 98304, 10, 0), (1024, 131072, 10, 1), (512, 400000, 1, 1),
                                (512, 262144, 32, 0), (512, 524288, 32, 1)):
        assert plan(lib, pkg, batch, n, 0, k)[2] == ranges, (batch, n, k)


@pytest.mark.parametrize("dim,n,bytes_kept", [(16, 1000000, 0), (64, 1000000, 0), (65, 1000000, 128), (128, 19999, 0), (128, 20000, 128), (256, 300000, 256), (257, 300000, 0),
                                              (320, 300000, 0), (321, 300000, 512), (1024, 27278, 1024), (128, 1048577, 0)])
def test_tables_hold_bytes_where_searches_may_go_by_them(pkg, dim, n, bytes_kept):
    """Beside both copies and the norms: a column's bytes, and 4.7 for units, errors and what sums start from."""
    lib = pkg.load_library()
    rows = (n + 255) // 256 * 256
    others = rows * ((dim + 63) // 64 * 64) * 2 + n * ((dim + 3) // 4 * 4) * 4 + rows * 4 + rows // 64 * 4
    extra = lib.dsx_screen_table_bytes(n, dim) - others
    assert 0 <= extra - (rows * (bytes_kept + 4) if bytes_kept else 0) <= (rows if bytes_kept else 0) + 4096


@pytest.mark.parametrize("queries", [4096, 16384, 65536])
def test_words_of_many_rows_have_a_bound(pkg, queries):
    """What a search in bytes works in beside what one in halves does: 1 GiB, and what its rows take themselves."""
    lib = pkg.load_library()
    n, dim, k = 1000000, 128, 100
    try:
        for bytes_of in (lambda: lib.dsx_knn_workspace_bytes_prepared(n, dim, queries, k), lambda: lib.dsx_knn_workspace_bytes_f16_prepared(n, dim, queries, k) - n * (dim + 8)):
            pkg.check(lib.dsx_testing_set_screen_bytes(0))
            in_bytes = bytes_of()
            pkg.check(lib.dsx_testing_set_screen_bytes(2))
            assert in_bytes <= bytes_of() + (1 << 30) + queries * (dim + 24) + (40 << 20)
    finally:
        pkg.check(lib.dsx_testing_reset())
