"""A workspace lent to an automatic 16-bit call is used whichever kernel runs: it
holds f(X_upper) afterwards, and the result has the bits of the call without one."""
import pytest
import torch

from lich_amd import _native as nat
from lich_amd.kernels import ForwardKernel, InferenceUpdateKernel, PredictionErrorKernel, WeightUpdateKernel
from tests.helpers import DEV, gen, randn, report

pytestmark = pytest.mark.gpu


# mode, sizes, workspace of the prediction and of the weight update
@pytest.mark.parametrize("mode,M,K,B,groups", [
    (-1, 1024, 1024, 1024, 1),      # k-chunk kernel, 256 tiles of 64
    (-1, 1024, 8192, 136, 1),       # k-chunk kernel, 48 tiles
    (-1, 1100, 1031, 1025, 1),      # rows the LDS-DMA kernel refuses, odd lengths
    (-1, 2048, 1024, 1096, 2),      # LDS-DMA kernel
    (1, 33, 70, 17, 3), (1, 64, 784, 128, 1), (1, 5, 1, 3, 1),
])
@pytest.mark.parametrize("act,dt", [("silu", torch.bfloat16), ("tanh", torch.float16), ("relu", torch.bfloat16)])
def test_lent_workspace_is_used_and_changes_no_bit(mode, M, K, B, groups, act, dt):
    report("lent-workspace", mode=mode, M=M, K=K, B=B, groups=groups, act=act, dt=str(dt))
    g = gen(M + K + B)

    def make(rows, cols, scale=1.0):
        t = (randn((groups, rows, cols), g) * scale).to(dt).to(DEV)
        return t if groups > 1 else t[0]

    xu, w, xl, e = make(K, B), make(M, K, K ** -0.5), make(M, B), make(M, B)
    fx = {"silu": torch.nn.functional.silu, "tanh": torch.tanh, "relu": torch.relu}[act](xu.float())
    cfg = (M, K, B, act, dt, None, None, groups)
    try:
        assert nat.lib().ipc_set_s16_preactivate(mode) == 0
        kernels = (PredictionErrorKernel("p", *cfg), ForwardKernel("f", *cfg),
                   WeightUpdateKernel("w", *cfg, alpha=0.01, recompute_activation=True))
        for k in kernels:
            need = 0 if (act == "relu" and mode < 0) else groups * K * B * 2
            assert k.workspace_bytes == need
            out = []
            for lend in (False, True):
                ws = torch.full((max(need, 16) // 2,), float("nan"), device=DEV, dtype=dt) if lend else None
                if k.kind == "w":
                    wd = w.clone()
                    k(wd, e, xu, workspace=ws)
                    out.append(wd)
                else:
                    o = torch.zeros_like(xl)
                    k(*((xu, w, xl, o) if k.kind == "p" else (xu, w, o)), workspace=ws)
                    out.append(o)
            torch.cuda.synchronize()
            assert torch.equal(out[0], out[1]) and out[0].isfinite().all()
            if need:
                # f(X) or its transpose, per group
                got, ref = ws[:need // 2].float().view(groups, -1), fx.view(groups, K, B)
                assert any(torch.allclose(got, r.reshape(groups, -1), rtol=2 ** -7, atol=1e-3)
                           for r in (ref, ref.transpose(1, 2)))
        # the inference update's copies serve the LDS-DMA kernel only
        ki = InferenceUpdateKernel("i", *cfg, gamma=0.5, save_activation=False)
        route = nat.lib().ipc_kernel_route(1, M, K, B, groups, nat.dtype_code(dt), nat.act_code(act), -1)
        assert (ki.workspace_bytes > 0) == (mode == 1 and 3 <= route < 16)
    finally:
        nat.lib().ipc_set_s16_preactivate(-1)


def test_lent_workspace_under_graph_capture():
    """Both launches of a k-chunk call with a workspace are recorded; replays, with
    the workspace overwritten and eager calls in between, give the eager bits."""
    M, K, B, dt = 1024, 1024, 1024, torch.float16
    report("lent-workspace-graph")
    g = gen(7)
    xu, w, xl = (randn(s, g).to(dt).to(DEV) for s in ((K, B), (M, K), (M, B)))
    w.mul_(K ** -0.5)
    k = PredictionErrorKernel("p", M, K, B, "gelu", dt, None, None)
    assert nat.lib().ipc_kernel_route(0, M, K, B, 1, nat.dtype_code(dt), nat.act_code("gelu"), -1) >= 16
    ws, eager, out = k.new_workspace(), torch.zeros_like(xl), torch.zeros_like(xl)
    k(xu, w, xl, eager)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=torch.cuda.Stream()):
        k(xu, w, xl, out, workspace=ws)
    for _ in range(3):
        out.zero_()
        ws.fill_(255)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, eager)
        k(xu, w, xl, out)
        assert torch.equal(out, eager)
