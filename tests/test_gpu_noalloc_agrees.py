"""``ipc_steps_noalloc`` gives an automatic plan's bits at every narrow net it
takes, on whichever path the plan runs, on both sides of every line between
them: several calls in a row, and under graph capture."""
import ctypes

import pytest
import torch

from lich_amd import HipIPC, IPCConfig, _native as nat
from lich_amd.trainer import _ptr_array
from oracle import ipc_oracle as O
from tests.helpers import DEV, report

pytestmark = pytest.mark.gpu


def _noalloc(m, x, e, w, wmode, steps):
    dims, B = m.cfg.dims, int(x[0].shape[1])
    d = (ctypes.c_int * len(dims))(*dims)
    nat.check(nat.lib().ipc_steps_noalloc(len(dims) - 1, d, B, _ptr_array(x), _ptr_array(e), _ptr_array(w),
                                          nat.dtype_code(m.cfg.dtype), m.pred_split, nat.act_code(m.cfg.activation),
                                          float(m.cfg.alpha), float(m.cfg.gamma), nat.WMODE[wmode], steps,
                                          nat.current_stream_handle(DEV)))


@pytest.mark.parametrize("dims,B,op,act,wmode,path", [
    ((10, 64, 64, 784), 128, torch.float16, "tanh", "gemm", "resident"),
    ((10, 64, 64, 784), 129, torch.float16, "tanh", "gemm", "phased"),
    ((10, 65, 65, 784), 128, torch.bfloat16, "relu", "gemm", "phased"),
    ((10, 65, 65, 784), 3, torch.float32, "silu", "auto", "phased"),
    ((10, 128, 128, 100), 32, torch.float16, "tanh", "outer", "narrow"),
    ((10, 128, 128, 128, 100), 32, torch.float32, "tanh", "outer", "phased"),
    ((10, 128, 128, 128, 100), 16, torch.float16, "gelu", "outer", "phased"),
    ((3, 66, 20), 4, torch.float32, "tanh", "auto", "narrow"),
    ((100, 700), 40, torch.float16, "sigmoid", "gemm", "phased"),
    ((7, 128, 128, 128, 129), 513, torch.float32, "gelu", "gemm", "phased"),
    ((20, 64, 784), 1100, torch.float16, "sigmoid", "gemm", "phased"),
])
def test_noalloc_has_the_automatic_plans_bits(dims, B, op, act, wmode, path):
    report("noalloc-agrees", dims=dims, B=B, op=op, act=act, wmode=wmode)
    w0 = O.init_weights(dims, seed=B, init="xavier_uniform")
    x_in, _l, y = O.make_batch(dims, B, seed=B)
    m = HipIPC(IPCConfig(dims=dims, activation=act, dtype=op, weight_update_mode=wmode, alpha=1e-6,
                         hierarchical_policy_auto=False), device=DEV, weights=w0)
    m.initialize_batch(x_in.to(DEV), y.to(DEV))
    assert m.path == path
    x, e, w = [t.clone() for t in m.x], [t.clone() for t in m.e], [t.clone() for t in m.w]
    s, graph = torch.cuda.Stream(), torch.cuda.CUDAGraph()

    def check():
        torch.cuda.synchronize()
        assert all(a.isfinite().all() and torch.equal(a, b) for a, b in zip(m.x + m.e[:-1] + m.w, x + e[:-1] + w))

    m.run_steps(3)
    _noalloc(m, x, e, w, wmode, 1)
    _noalloc(m, x, e, w, wmode, 2)
    check()
    with torch.cuda.graph(graph, stream=s):
        _noalloc(m, x, e, w, wmode, 2)
    for _ in range(2):
        graph.replay()
        m.run_steps(2)
        check()
    m.check_steps()
    assert nat.lib().ipc_noalloc_check(nat.current_stream_handle(DEV)) == nat.IPC_OK
