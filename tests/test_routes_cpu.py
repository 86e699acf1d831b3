"""Which kernel a standalone call runs (ipc_kernel_route: the host rules alone, no GPU)."""
import pytest

from lich_amd import _native as nat

PRED, INFER, WEIGHT = 0, 1, 2
DMA, TALL, CHUNK = range(3, 7), 7, range(16, 19)


def route(kind, M, K, B, groups=1, st="bf16", act="relu", tile=-1):
    code = {"fp32": nat.DT_F32, "fp16": nat.DT_F16, "bf16": nat.DT_BF16}[st]
    return nat.lib().ipc_kernel_route(kind, M, K, B, groups, code, nat.act_code(act), tile)


@pytest.mark.parametrize("kind,M,K,B,want", [
    # few tiles, an operand of 2^31 bytes or more: the LDS-DMA kernel (the
    # k-chunk kernel's 32-bit offsets cannot reach it, the tile kernel takes 2-5 times as long)
    (WEIGHT, 1024, 1024, 1 << 20, DMA), (PRED, 1024, 1 << 20, 512, DMA), (INFER, 1024, 1 << 20, 1024, DMA),
    (PRED, 256, (1 << 22) + 64, 256, DMA),
    # just below
    (WEIGHT, 1024, 1024, 1 << 19, CHUNK), (PRED, 1024, 1 << 19, 512, CHUNK),
    # 257-512 tiles: inference updates of at most 128 products stay on the tile kernel's 64 x 64 tiles
    (INFER, 2048, 128, 1024, [1]), (INFER, 2048, 64, 1024, [1]), (INFER, 2048, 192, 1024, CHUNK),
    (INFER, 2048, 192, 1088, DMA), (PRED, 2048, 128, 1024, DMA), (WEIGHT, 2048, 1024, 128, DMA),
    (PRED, 1024, 1024, 1024, CHUNK), (INFER, 1024, 128, 1024, CHUNK),
])
def test_automatic_16_bit_calls(kind, M, K, B, want):
    assert route(kind, M, K, B) in want
