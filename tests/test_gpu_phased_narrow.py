"""Narrow nets past the sizes of the layer-resident kernel take the phased path's
k-chunk launches: the first hidden errors are exactly 0, and the steps agree with
the column kernel's (the same operand rounding and prediction order; a sum added in
another order may turn an operand by one unit)."""
import pytest
import torch

from lich_amd import HipIPC, IPCConfig
from oracle import ipc_oracle as O
from tests.helpers import DEV, rel_err, report

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims,B,op,act,wmode,save", [
    ((10, 65, 65, 784), 1, torch.float32, "tanh", "auto", False),
    ((10, 64, 64, 300), 129, torch.float16, "relu", "gemm", True),
    ((7, 128, 128, 128, 129), 33, torch.bfloat16, "sigmoid", "gemm", False),
    ((1, 128, 2000), 513, torch.float16, "tanh", "gemm", False),
    ((10, 100, 30, 128), 16, torch.float16, "silu", "auto", True),
    ((10, 16, 784), 1000, torch.float32, "gelu", "gemm", True),
])
def test_automatic_path_agrees_with_the_column_kernel(dims, B, op, act, wmode, save):
    report("phased-narrow", dims=dims, B=B, op=op, act=act, wmode=wmode, save=save)
    w0 = O.init_weights(dims, seed=5, init="xavier_uniform")
    x, _l, y = O.make_batch(dims, B, seed=5)
    ms = []
    for fused in ("auto", "narrow"):
        m = HipIPC(IPCConfig(dims=dims, activation=act, dtype=op, fused=fused, weight_update_mode=wmode,
                             recompute_activation=not save), device=DEV, weights=w0)
        m.initialize_batch(x.to(DEV), y.to(DEV))
        m.run_steps(1)
        torch.cuda.synchronize()
        assert all(torch.count_nonzero(m.e[l]) == 0 for l in range(1, len(dims) - 1))
        m.run_steps(2)
        torch.cuda.synchronize()
        ms.append(m)
    assert [m.path for m in ms] == ["phased", "narrow"]
    # states: a unit of the operand type at most.  fp32: sums of n <= 2000 terms in two orders
    # differ by about sqrt(n) 2^-24 of their magnitude, 2.7e-6, in each of three steps
    tol = {torch.float32: 8e-6, torch.float16: 2.0 ** -11, torch.bfloat16: 2.0 ** -8}[op]
    for a, b in zip(ms[0].x[:-1] + ms[0].w, ms[1].x[:-1] + ms[1].w):
        assert rel_err(a.double().cpu(), b.double().cpu()) <= tol
