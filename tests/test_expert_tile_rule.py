"""Which tiles the sorted products of routed experts take (host code of the kernel library: no GPU needed)."""
import pytest


@pytest.fixture(scope="module")
def tile_rows():
    from llmserver_amd.kernels import library
    lib = library.load("experts")
    return lambda pairs, experts, inter, width, aligned=True: lib.lsa_experts_tile_rows(pairs, experts, inter, width, 1 if aligned else 0)


def test_wide_tiles_want_whole_pieces_of_16_bytes(tile_rows):
    """Their loads straight into LDS take 16 bytes at multiples of 16; tensors that begin elsewhere keep the tiles whose loads go through registers."""
    assert tile_rows(12288, 64, 1408, 2048) == 256
    assert tile_rows(12288, 64, 1408, 2048, aligned=False) == 64


def test_wide_tiles_end_where_their_offsets_do(tile_rows):
    """Offsets of 32 bits into the rows of all pairs and into one expert's matrices."""
    most = (2 ** 32 - 1) // (2 * 4096) - 1                      # pairs of rows of 4,096 bfloat16 numbers
    assert tile_rows(most, 64, 1408, 4096) == 256 and tile_rows(most + 2, 64, 1408, 4096) == 64
    assert tile_rows(most, 64, 4096, 1408) == 256 and tile_rows(most + 2, 64, 4096, 1408) == 64
    assert tile_rows(1000, 8, 32768 - 32, 32768) == 256 and tile_rows(1000, 8, 32768, 32768) == 64
