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


def test_workspace_bytes_are_those_of_the_call():
    """0 exactly where the call would not use a workspace (0 used to be promised
    that, and more than 0 asked for, by calls of few tiles that ignored it)."""
    lib, tanh = nat.lib(), nat.act_code("tanh")
    wb, wt = lib.ipc_s16_workspace_bytes, lib.ipc_s16_workspace_bytes_tile
    assert wb(PRED, tanh, 1024, 1024, 1024, 1) == 1024 * 1024 * 2  # the k-chunk kernel reads it
    assert wb(PRED, tanh, 1024, 1031, 1025, 1) == 1031 * 1025 * 2
    for tile in range(7):  # explicit tiles: the LDS-DMA kernel's only
        assert wt(PRED, tanh, 1024, 1024, 1024, 1, tile) == (1024 * 1024 * 2 if tile >= 3 else 0)
    assert wt(WEIGHT, tanh, 1024, 1024, 1031, 1, 3) == 0  # a tile the call would be refused for
    # the inference update: only where it runs on the LDS-DMA kernel
    assert wb(INFER, tanh, 1024, 65536, 1024, 1) == 0 and wt(INFER, tanh, 1024, 65536, 1024, 1, 3) == 2 * (1 << 27)
    assert lib.ipc_s16_preactivates(INFER, tanh, 1024, 65536, 1024) == 0
    try:
        assert lib.ipc_set_s16_preactivate(1) == 0
        assert wb(PRED, tanh, 64, 784, 128, 1) == 784 * 128 * 2 and wb(INFER, tanh, 64, 64, 64, 1) == 0
        assert wb(INFER, tanh, 4096, 4096, 1024, 1) == 2 * (4096 * 4096 + 4096 * 1024)
        assert lib.ipc_set_s16_preactivate(0) == 0 and wb(PRED, tanh, 8192, 8192, 8192, 1) == 0
    finally:
        lib.ipc_set_s16_preactivate(-1)


@pytest.mark.parametrize("M,N,want", [(64, 128, [16, 17, 18]), (512, 480, [16, 17, 18]), (512, 512, [17, 17, 18]),
                                      (704, 1088, [17, 17, 18]), (768, 1024, [17, 18, 18]), (1024, 1024, [17, 18, 18])])
def test_generic_tiles_run_as_asked_for(M, N, want):
    """No id runs a larger tile than it names, and each automatic choice has an id."""
    for call in ((PRED, M, 300, N), (INFER, M, 300, N), (WEIGHT, M, N, 300)):
        ids = [route(*call, st="fp32", tile=t) for t in (0, 1, 2)]
        assert ids == want and route(*call, st="fp32") in ids
        assert [route(*call, st="fp16", tile=t) for t in (0, 1, 2)] == [0, 1, 2]  # the tile kernel
    assert route(PRED, 4096, 4096, 2048, st="fp32", tile=0) == 0 and route(INFER, 4096, 4096, 2048, st="fp32", tile=0) == 17


@pytest.mark.parametrize("kind,M,K,B,st,act,chunk", [
    (PRED, 4096, 780, 2048, "fp32", "sigmoid", False), (PRED, 4096, 780, 2048, "fp32", "relu", True),
    (PRED, 4096, 900, 2048, "fp16", "silu", True), (PRED, 4096, 780, 2048, "fp16", "silu", False),
    (PRED, 4096, 780, 2048, "fp16", "tanh", True), (PRED, 4096, 780, 2048, "fp32", "tanh", False),
    (PRED, 1920, 780, 2048, "fp32", "sigmoid", True), (PRED, 4096, 1412, 2048, "fp16", "sigmoid", True),
    (INFER, 4096, 780, 2048, "fp32", "sigmoid", True),
    (WEIGHT, 2048, 4096, 780, "fp32", "gelu", False), (WEIGHT, 2048, 4096, 780, "fp16", "gelu", True),
])
def test_many_tiles_of_a_partly_filled_round(kind, M, K, B, st, act, chunk):
    """Loaders with a costly activation: the tile kernel, which the k-chunk kernel had slowed down."""
    assert (route(kind, M, K, B, st=st, act=act) in CHUNK) == chunk


@pytest.mark.parametrize("dims,B,wmode,op,want", [
    # the rank-B update, a launch a layer on the phased path
    ((10, 65, 65, 65, 65, 256), 32, "outer", "fp32", "narrow"), ((10, 65, 65, 65, 65, 256), 17, "outer", "fp32", "phased"),
    ((10, 65, 65, 550), 32, "outer", "fp32", "phased"), ((10, 128, 128, 256), 24, "outer", "fp16", "narrow"),
    ((10, 128, 128, 128, 128, 256), 24, "outer", "fp16", "phased"), ((10, 65, 65, 256), 32, "gemm", "fp32", "phased"),
    # a few small layers
    ((3, 66, 20), 4, "auto", "fp32", "narrow"), ((10, 65, 64), 64, "gemm", "fp16", "narrow"),
    ((10, 65, 64), 65, "gemm", "fp16", "phased"), ((10, 65, 129), 64, "gemm", "fp16", "phased"),
    ((10, 128, 64), 4, "gemm", "fp32", "phased"), ((10, 65, 65, 64), 4, "gemm", "fp32", "phased"),
    # no upper end in B
    ((10, 64, 64, 64, 784), 65536, "gemm", "fp32", "phased"),
])
def test_automatic_path_of_narrow_nets_past_the_resident_sizes(dims, B, wmode, op, want):
    import ctypes

    lib, h = nat.lib(), ctypes.c_void_p()
    code = {"fp32": nat.DT_F32, "fp16": nat.DT_F16}[op]
    assert lib.ipc_plan_create(ctypes.byref(h), len(dims) - 1, (ctypes.c_int * len(dims))(*dims), B, 0, code, 1,
                               nat.act_code("tanh"), 1e-4, 0.5, 1, nat.WMODE[wmode], nat.FUSED["auto"]) == nat.IPC_OK
    try:
        assert nat.PATH_NAMES[lib.ipc_plan_path(h)] == want
    finally:
        lib.ipc_plan_destroy(h)


def test_launches_stay_below_the_thread_limit():
    """2^23 groups of one tile: 2^32 threads in the k-chunk kernel's workgroups of
    512, which a launch may not have; the tile kernel's 256 fit, as before it."""
    assert route(INFER, 16, 257, 16, groups=(1 << 23) - 1) == 18
    assert route(INFER, 16, 257, 16, groups=1 << 23) == 2
    assert route(INFER, 16, 257, 16, groups=1 << 23, st="fp32") == 2
    assert [route(INFER, 128, 257, 128, groups=g, st="fp32", tile=0) for g in (1 << 18, 1 << 19)] == [17, 18]
