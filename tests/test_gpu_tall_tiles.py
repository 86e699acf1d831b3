"""The 512 x 64 tiles of the 16-bit prediction and forward with an exponential
activation: the bits of the 256 x 128 tiles (the same k order and epilogue) at the
edges of either tile, with groups, over contractions of one to many k-steps, and
those of the call lent a workspace, which leaves them."""
import pytest
import torch

from lich_amd import _native as nat
from lich_amd.kernels import ForwardKernel, KernelConfig, PredictionErrorKernel
from tests.helpers import DEV, gen, randn, report

pytestmark = pytest.mark.gpu


# (more than 256 tiles of 64 x 64, or the k-chunk kernel runs; the third and the last fall back to 256 x 128, as
# their rows would pad further: the automatic choice itself)
@pytest.mark.parametrize("dt", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("act", ["tanh", "sigmoid", "silu", "gelu"])
@pytest.mark.parametrize("M,K,B,groups", [(512, 64, 2112, 1), (1000, 192, 1096, 1), (1537, 128, 776, 1), (300, 64, 1032, 4),
                                          (600, 128, 2048, 1)])
def test_tall_tiles_give_the_same_bits(M, K, B, groups, act, dt):
    report("tall", M=M, K=K, B=B, groups=groups, act=act, dt=str(dt))
    g = gen(M + K + B)

    def make(rows, cols, scale=1.0):
        t = (randn((groups, rows, cols), g) * scale).to(dt).to(DEV)
        return t if groups > 1 else t[0]

    xu, w, xl = make(K, B), make(M, K, K ** -0.5), make(M, B)
    outs = []
    for tile in (None, 3):
        cfg = KernelConfig(tile=tile) if tile else KernelConfig()
        e, o = torch.zeros_like(xl), torch.zeros_like(xl)
        PredictionErrorKernel("p", M, K, B, act, dt, cfg, None, groups)(xu, w, xl, e)
        kf = ForwardKernel("f", M, K, B, act, dt, cfg, None, groups)
        kf(xu, w, o)
        outs.append((e, o))
    torch.cuda.synchronize()
    assert all(torch.equal(a, b) for a, b in zip(*outs))
    assert outs[0][0].abs().sum() > 0


TALL, DEFAULT, LARGE = 7, 3, 6


@pytest.mark.parametrize("dt", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("act,M,K,B,groups,want", [
    ("tanh", 1000, 1024, 1096, 1, TALL),    # 24 rows short of two tiles, 8 columns into the 18th: 16 k-steps
    ("gelu", 2040, 2048, 648, 1, TALL),     # 32 k-steps
    ("silu", 1530, 1088, 1480, 1, TALL),    # 17 k-steps
    ("sigmoid", 500, 1024, 1160, 2, TALL),
    ("tanh", 4096, 128, 4096, 1, LARGE),    # 256 x 256 tiles fill the CUs: tanh stays there
    ("sigmoid", 4096, 128, 4096, 1, TALL),
    ("silu", 1537, 128, 776, 1, DEFAULT),   # a row past three tiles
    ("relu", 1000, 1024, 1096, 1, DEFAULT),
])
def test_long_contractions_and_the_lines_of_the_rule(act, M, K, B, groups, want, dt):
    report("tall-long", M=M, K=K, B=B, groups=groups, act=act, dt=str(dt))
    route = nat.lib().ipc_kernel_route
    assert route(0, M, K, B, groups, nat.dtype_code(dt), nat.act_code(act), -1) == want
    g = gen(M + K + B)

    def make(rows, cols, scale=1.0):
        t = (randn((groups, rows, cols), g) * scale).to(dt).to(DEV)
        return t if groups > 1 else t[0]

    xu, w, xl = make(K, B), make(M, K, K ** -0.5), make(M, B)
    outs = []
    for tile, lend in ((3, False), (-1, False), (-1, True)):
        e, o = torch.zeros_like(xl), torch.zeros_like(xl)
        for k, args in ((PredictionErrorKernel("p", M, K, B, act, dt, KernelConfig(tile=tile), None, groups), (xu, w, xl, e)),
                        (ForwardKernel("f", M, K, B, act, dt, KernelConfig(tile=tile), None, groups), (xu, w, o))):
            ws = k.new_workspace() if lend else None
            assert ws is None or ws.numel() >= 2 * groups * K * B
            k(*args, workspace=ws)
        outs.append((e, o))
    assert nat.lib().ipc_s16_workspace_bytes(0, nat.act_code(act), M, K, B, groups) == \
        (2 * groups * K * B if act != "relu" and M >= 1024 and K * B >= 1 << 20 else 0)
    torch.cuda.synchronize()
    assert all(torch.equal(a, b) for other in outs[1:] for a, b in zip(outs[0], other))
    assert outs[0][0].abs().sum() > 0
