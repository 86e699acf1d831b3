"""The 512 x 64 tiles of the 16-bit prediction and forward with an exponential
activation: the bits of the 256 x 128 tiles (the same k order and epilogue) at the
edges of either tile, with groups, and the workspace call's bits."""
import pytest
import torch

from lich_amd.kernels import ForwardKernel, KernelConfig, PredictionErrorKernel
from tests.helpers import DEV, gen, randn, report

pytestmark = pytest.mark.gpu


# (more than 256 tiles of 64 x 64, or the k-chunk kernel runs; the last falls back: 600 rows pad to 1024)
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
