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
