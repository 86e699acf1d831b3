"""The k-chunk kernel where several waves share a chunk (few chunks on 32 and 64
wide tiles) and where a CU holds two workgroups (more than 256 tiles of 32 x 32),
to the bounds of the kernel's own tests."""
import pytest

from tests.test_gpu_chunk import pytestmark, test_three_kernels_at_tile_and_chunk_edges as _three  # noqa: F401


# tiles of 64: 210-225 of 1, 3 and 4 chunks; of 32: 272 of 4 chunks, 306 of 9, exactly 256 of 9
@pytest.mark.parametrize("shift", [0, 1])
@pytest.mark.parametrize("st,op", [("f32", "f32"), ("f32", "bf16"), ("f16", "f16")])
@pytest.mark.parametrize("M,K,B", [(900, 128, 900), (900, 129, 901), (897, 300, 900), (900, 385, 850), (900, 512, 833),
                                   (514, 400, 500), (520, 1100, 550), (512, 1030, 500)])
def test_shared_chunks(M, K, B, st, op, shift):
    _three(M, K, B, st, op, shift)
