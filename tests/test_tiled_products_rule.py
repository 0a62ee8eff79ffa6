"""Which products of many rows this package's own tiles take (host code of the kernel library: no GPU needed)."""
import pytest

PLAIN, GATED, ACTIVATED, SUMS = range(4)
ROWS = {1: 64, 2: 128, 3: 128, 4: 256}
COLUMNS = {1: 64, 2: 64, 3: 128, 4: 256}
ADDED = 1 << 12


@pytest.fixture(scope="module")
def plan():
    from llmserver_amd.kernels import library
    return library.load("product").lsa_product_plan


def test_sizes_that_no_tile_takes_stay_the_librarys(plan):
    for form in range(4):
        assert not plan(form, 190, 4096, 2048 + 32) and not plan(form, 190, 4100, 2048) and not plan(form, 190, 0, 2048) and not plan(form, 0, 4096, 2048)
        assert not plan(form, 190, 4096, 0)
    assert not plan(-1, 190, 4096, 2048) and not plan(4, 190, 4096, 2048)
    assert not plan(GATED, 4096, 2 ** 18, 4096 + 64)            # offsets into gate and up rows end at 4 GB


def test_small_tiles_go_round_the_compute_units_once(plan):
    """But for those of 64 x 64, two of whose workgroups fit a unit; and only plain and gated products of up to 128 rows have parts that another launch adds up."""
    seen, added = set(), set()
    for form in range(4):
        for rows in (17, 33, 64, 100, 128, 190, 333, 500, 777, 1000, 2048, 5000):
            for columns, inner in ((1024, 2048), (2048, 2048), (2048, 6144), (4096, 1024), (4096, 4096), (6144, 2560), (8192, 4096), (12288, 2048), (12288, 4096)):
                whole = plan(form, rows, columns, inner)
                tile, parts = whole % 16, whole % ADDED // 16
                seen.add((form, tile))
                if whole >= ADDED:
                    added.add(form)
                    assert form in (PLAIN, GATED) and rows <= 128 and parts > 1
                assert parts in ((1,) if form != SUMS and whole < ADDED else (1, 2, 4, 8)) or not tile
                if tile in (1, 2, 3):
                    width = COLUMNS[tile] // (2 if form == GATED else 1)
                    assert -(-rows // ROWS[tile]) * -(-columns // width) * parts <= (512 if tile == 1 and parts == 1 else 256) and inner // 64 >= 4 * parts
                assert tile != 4 or form == GATED
    assert {tile for _, tile in seen} == {0, 1, 2, 3, 4} and {form for form, tile in seen if tile} == {PLAIN, GATED, ACTIVATED, SUMS}
    assert added == {PLAIN, GATED}


def test_products_that_were_measured_to_be_faster(plan):
    for form, rows, columns, inner in ((PLAIN, 190, 4096, 2048), (PLAIN, 2048, 2048, 2048), (PLAIN, 33, 4096, 4096), (PLAIN, 33, 32768, 4096), (PLAIN, 333, 4096, 1024), (GATED, 190, 6144, 2048),
                                       (GATED, 33, 8192, 4096), (GATED, 64, 2816, 4096), (GATED, 2048, 12288, 4096), (SUMS, 33, 2048, 2048), (SUMS, 190, 2048, 6144), (SUMS, 333, 2560, 9728), (ACTIVATED, 333, 8448, 2048)):
        assert plan(form, rows, columns, inner), (form, rows, columns, inner)
    for form, rows, columns, inner in ((PLAIN, 2048, 6144, 4096), (PLAIN, 2048, 4096, 12288), (PLAIN, 640, 16384, 4096), (PLAIN, 60, 2048, 2048),
                                       (GATED, 333, 6144, 2048), (GATED, 2048, 8448, 2048), (ACTIVATED, 2048, 8192, 4096), (SUMS, 20, 4096, 8192), (SUMS, 2048, 4096, 12288)):
        assert not plan(form, rows, columns, inner), (form, rows, columns, inner)


def test_gated_products_of_short_inner_dimensions_stay_where_they_were(plan):
    """Neither small tiles nor large ones: the kernel that shares the activations, or the library, has them."""
    assert not any(plan(GATED, rows, columns, inner) for rows in (17, 33, 70, 206, 777, 2048, 9000) for columns in (32, 64, 96, 768, 3072, 12288) for inner in (64, 128, 512, 960))


def test_sums_of_large_weights_on_few_tiles_stay_with_the_few_row_kernel(plan):
    """Output and down projections whose tiles leave compute units idle, at a batch's 17 to 128 rows; where they do not, or the weight is small, the tiles keep them."""
    for rows in (17, 28, 29, 33, 48, 64):
        for columns, inner in ((5120, 5120), (5120, 8192), (5120, 17408), (5120, 25600)):
            assert plan(SUMS, rows, columns, inner) < 32, (rows, columns, inner)
    assert all(plan(SUMS, rows, 4096, 8192) < 32 for rows in (17, 24, 28, 29, 32))
    assert all(plan(SUMS, rows, 5120, 25600) < 32 for rows in (65, 96, 128))
    assert all(plan(SUMS, rows, columns, inner) >= 32 for rows in (17, 33, 64, 128) for columns, inner in ((2048, 6144), (4096, 4096), (2560, 9728)))
    assert all(plan(SUMS, rows, 4096, 12288) >= 32 for rows in (48, 64, 112, 128))


def test_large_gated_tiles_are_not_taken_for_a_few_slabs(plan):
    """A launch of 256 x 256 tiles costs some 13 us beside its slabs: 16 or 32 of them on a part of the compute units are the library's."""
    assert not any(plan(GATED, rows, 3072, 1024) % 16 == 4 for rows in (17, 256, 641, 820, 1000, 1024, 1100, 1200, 1280, 1400))
    assert all(plan(GATED, rows, 3072, 1024) % 16 == 4 for rows in (2001, 2048, 2300, 2560))
    assert not any(plan(GATED, rows, 6144, 2048) % 16 == 4 for rows in (257, 512, 700, 768, 820)) and plan(GATED, 1200, 6144, 2048) % 16 == 4
    assert not any(plan(GATED, rows, 17408, 5120) for rows in (17, 24, 29, 48, 64))          # (136 compute units pull its weights)


def test_tiles_whose_rows_are_full_are_priced_so(plan):
    """A slab of a tile with all its rows takes longer than one whose last rows repeat: whole multiples of 128 rows do not go to tiles of 128 x 64 for one row more to a launch."""
    assert plan(PLAIN, 512, 2048, 2048) == 16 + 1
    for form, rows, columns, inner in ((PLAIN, 768, 2048, 2048), (PLAIN, 384, 4096, 2048), (SUMS, 384, 2048, 1408), (SUMS, 512, 2048, 1408), (ACTIVATED, 384, 8192, 4096)):
        assert plan(form, rows, columns, inner) < (32 if form == SUMS else 1), (form, rows, columns, inner)
    for rows in (1792, 1900, 2001, 2047, 2048):                  # one round of tiles of 128 x 128, whatever the last one holds
        assert plan(PLAIN, rows, 2048, 2048) == 16 + 3, rows
    for form, rows, columns, inner in ((PLAIN, 820, 2048, 2048), (PLAIN, 320, 4096, 2048), (PLAIN, 333, 4096, 2048), (PLAIN, 448, 4096, 2048), (ACTIVATED, 257, 8448, 2048)):
        assert plan(form, rows, columns, inner), (form, rows, columns, inner)


def test_a_large_weight_in_parts_stays_with_the_library_up_to_32_rows(plan):
    """The library cuts the inner dimension there itself; from 33 rows on it does not, and weights of up to 50 MB are faster in parts before that too."""
    assert not any(plan(PLAIN, rows, 4096, 8192) for rows in range(17, 33))
    assert all(plan(PLAIN, rows, 4096, 8192) for rows in (33, 44, 64, 100))
    assert all(plan(PLAIN, rows, columns, inner) for rows in (17, 28, 32) for columns, inner in ((2048, 8448), (4096, 4096)))


def test_tiles_are_priced_by_their_last_block_of_rows_and_by_who_else_reads_the_weight(plan):
    """Sizes where the tiles were measured to be 1.15 times as fast as the other way and more, and which a price by how full all rows are together had refused."""
    for form, rows, columns, inner in ((GATED, 100, 8448, 2048), (GATED, 128, 8448, 2048), (PLAIN, 38, 10304, 2048), (PLAIN, 45, 10304, 2048), (PLAIN, 128, 3328, 2048), (PLAIN, 126, 4240, 2048),
                                       (PLAIN, 46, 2048, 4096), (PLAIN, 592, 2048, 2112)):
        assert plan(form, rows, columns, inner), (form, rows, columns, inner)


def test_sums_of_more_than_1100_rows_are_the_librarys(plan):
    assert not any(plan(SUMS, rows, 1024, inner) for rows in (1101, 1121, 1338, 1980) for inner in (2048, 3072)) and plan(SUMS, 900, 1024, 3072) >= 32


def test_tiles_of_32_columns_do_not_move_the_plans_lines(plan):
    """They run where the plan takes small tiles; what goes in parts or to the library, which may round otherwise, goes there as it did: gated products of 32 rows in two parts, products of
    33 rows of 6,144 x 4,096 by the library."""
    assert plan(GATED, 32, 2816, 4096) == ADDED + 32 + 1 and plan(GATED, 48, 3072, 4096) >= ADDED and plan(PLAIN, 33, 4096, 4096) >= ADDED
    assert not plan(PLAIN, 33, 6144, 4096) and not plan(PLAIN, 17, 7168, 5120) and not plan(PLAIN, 192, 1024, 3072)
