"""Which tiles the sorted products of routed experts take (host code of the kernel library: no GPU needed)."""
import pytest
import torch

from llmserver_amd.kernels.ops import HipOps


@pytest.fixture(scope="module")
def tile_rows():
    from llmserver_amd.kernels import library
    lib = library.load("experts")
    return lambda pairs, experts, inter, width, plain=False, aligned=True: lib.lsa_experts_tile_rows(pairs, experts, inter, width, int(plain), int(aligned))


def test_wide_tiles_want_whole_pieces_of_16_bytes(tile_rows):
    """Their loads straight into LDS take 16 bytes at multiples of 16; tensors that begin elsewhere keep the tiles whose loads go through registers."""
    assert tile_rows(12288, 64, 1408, 2048) == 256
    assert tile_rows(12288, 64, 1408, 2048, aligned=False) == 64


def test_wide_tiles_end_where_their_offsets_do(tile_rows):
    """Offsets of 32 bits into the rows of all pairs and into one expert's matrices."""
    most = (2 ** 32 - 1) // (2 * 4096) - 1                      # pairs of rows of 4,096 bfloat16 numbers
    assert tile_rows(most, 64, 1408, 4096) == 256 and tile_rows(most + 2, 64, 1408, 4096) == 64
    assert tile_rows(most, 64, 4096, 1408) == 256 and tile_rows(most + 2, 64, 4096, 1408) == 64
    assert tile_rows(1000, 3, 32768 - 32, 32768) == 256 and tile_rows(1000, 3, 32768, 32768) == 64


def test_wide_tiles_where_they_were_measured_to_be_faster(tile_rows):
    """Enough pairs an expert and enough tiles to go round the compute units; few experts or small ones keep the narrow tiles."""
    for experts, each, width, inter in ((64, 40, 2048, 1408), (64, 192, 2048, 1408), (16, 128, 4096, 2048), (8, 128, 4096, 2048), (8, 400, 2048, 1408),
                                        (64, 96, 1024, 512)):
        assert tile_rows(experts * each, experts, inter, width) == 256, (experts, each, width, inter)
    for experts, each, width, inter in ((64, 39, 2048, 1408), (4, 128, 4096, 2048), (4, 192, 4096, 2048), (8, 192, 2048, 1408), (4, 256, 2048, 1408),
                                        (1, 256, 1024, 512), (16, 192, 1024, 512), (1, 400, 4096, 2048)):
        assert tile_rows(experts * each, experts, inter, width) == 64, (experts, each, width, inter)
    assert tile_rows(16 * 100, 16, 1024, 2048) == 256 and tile_rows(16 * 100, 16, 1024, 2048, plain=True) == 64


def test_short_inner_dimensions_want_more_pairs_for_wide_tiles(tile_rows):
    """A wide launch of a few slabs is mostly its start."""
    for each in (40, 64, 100, 128, 199):
        assert tile_rows(64 * each, 64, 256, 1024) == 64 and tile_rows(64 * each, 64, 1024, 256) == 64, each
    assert tile_rows(64 * 200, 64, 256, 1024) == 256 and tile_rows(64 * 40, 64, 512, 1024) == 256


def test_sorted_products_where_they_were_measured_to_be_faster():
    """(Tensors without storage: what is not refused by its sizes is refused for where it lives.)"""
    def taken(pairs, experts, width, inter, plain=False):
        make = lambda *shape, dtype=torch.bfloat16: torch.empty(*shape, dtype=dtype, device="meta")
        try:
            return HipOps.experts_sorted(HipOps.__new__(HipOps), make(pairs, width), make(experts, (1 if plain else 2) * inter, width),
                                         make(experts, width, inter), make(pairs, 1, dtype=torch.int32), make(pairs, 1, dtype=torch.float32),
                                         make(pairs, width, dtype=torch.float32), activation="relu2" if plain else "silu")
        except ValueError as error:
            assert "must live on the GPU" in str(error)
            return True
    assert taken(72, 64, 2048, 1408) and taken(9, 8, 512, 512) and not taken(48, 64, 2048, 1408) and not taken(127, 128, 4096, 2048)
    for experts, width, inter in ((2, 512, 512), (8, 2048, 1408), (16, 1024, 512), (32, 2048, 768), (64, 2048, 768), (72, 2048, 768)):
        assert not taken(experts, experts, width, inter)
    for experts, width, inter in ((32, 4096, 2048), (64, 2048, 1408), (96, 1024, 512), (128, 2048, 1408)):
        assert taken(experts, experts, width, inter)
    assert taken(64, 64, 2048, 1408) and not taken(64, 64, 2048, 1408, plain=True)
