"""Which 32-bit products of a few rows leave the library (host code of the kernel library: no GPU needed)."""
import pytest


@pytest.fixture(scope="module")
def fits():
    from llmserver_amd.kernels import library
    return lambda rows, outputs, inner: bool(library.load("gemm").lsa_gemm_few_f32_fits(rows, outputs, inner))


def test_products_that_were_measured_to_be_faster_leave_the_library(fits):
    for rows in (1, 2, 4, 8):
        for outputs, inner in ((64, 512), (1024, 1024), (2048, 2048), (4096, 1024), (6144, 1024), (151936, 1024)):
            assert fits(rows, outputs, inner), (rows, outputs, inner)
    assert fits(2, 1024, 3072) and fits(4, 4096, 2048) and fits(4, 4096, 768) and fits(6, 151936, 2048) and fits(16, 151936, 1024)


def test_products_that_the_library_makes_faster_stay_there(fits):
    for rows in (1, 2, 8, 16):
        for outputs, inner in ((2560, 9728), (9728, 2560), (2560, 2048), (1024, 8192), (6144, 1536), (6144, 512), (16384, 512), (65536, 512), (151936, 512),
                               (65536, 2560), (151936, 2560), (1024, 508), (1024, 514), (0, 1024)):
            assert not fits(rows, outputs, inner), (rows, outputs, inner)
    assert not fits(8, 1024, 3072) and not fits(8, 4096, 2048) and not fits(8, 151936, 2048) and not fits(16, 16384, 1024) and not fits(9, 1024, 1024)
    assert not fits(0, 1024, 1024) and not fits(17, 151936, 1024)


def test_rounds_of_workgroups_do_not_refuse_what_is_faster_between_them(fits):
    """Eight rows of the weight a workgroup: 4,096 to 8,192 of them at 2,048 numbers are faster than the library's product for up to four rows, whole rounds or not."""
    for rows in (1, 2, 3, 4):
        assert all(fits(rows, outputs, 2048) for outputs in (4096, 4097, 4104, 5120, 6144, 7168, 7372, 7373, 8192)), rows
    assert not any(fits(5, outputs, 2048) for outputs in (4096, 5120, 8192)) and not any(fits(2, 5120, inner) for inner in (1536, 2044, 2052, 4096))
