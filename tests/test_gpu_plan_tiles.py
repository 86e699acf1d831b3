"""Tiles set by id on a phased plan with 16-bit storage run the tile kernel, as
the standalone calls do: one step has the bits of the three calls with that id."""
import pytest
import torch

from lich_amd import HipIPC, IPCConfig, _native as nat
from lich_amd.kernels import KernelConfig, build_inference_update, build_prediction_error, build_weight_update
from oracle import ipc_oracle as O
from tests.helpers import DEV, report

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dt", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("tile", [0, 1, 2])
def test_plan_tiles_are_the_tile_kernels(tile, dt):
    report("plan-tiles", tile=tile, dt=str(dt))
    dims, B = (10, 130, 300, 1100), 290
    w0 = O.init_weights(dims, seed=4, init="xavier_uniform")
    x_in, _l, y = O.make_batch(dims, B, seed=4)
    m = HipIPC(IPCConfig(dims=dims, activation="tanh", dtype=dt, master_dtype=dt, fused="phased", alpha=0.01,
                         kernel=KernelConfig(tile=tile)), device=DEV, weights=w0)
    m.initialize_batch(x_in.to(DEV), y.to(DEV))
    x, w = [t.clone() for t in m.x], [t.clone() for t in m.w]
    m.run_steps(1)
    cfg, L = KernelConfig(tile=tile), len(w)
    e = [torch.empty_like(t) for t in x]
    for l in range(L):
        build_prediction_error(dims[l], dims[l + 1], B, "tanh", dt, cfg)(x[l + 1], w[l], x[l], e[l])
    for l in range(1, L):
        build_inference_update(dims[l], dims[l - 1], B, "tanh", dt, cfg, 0.5, False)(x[l], e[l], w[l - 1], e[l - 1])
    for l in range(L):
        build_weight_update(dims[l], dims[l + 1], B, "tanh", dt, cfg, 0.01, True)(w[l], e[l], x[l + 1])
    torch.cuda.synchronize()
    assert nat.lib().ipc_plan_path(m._plan) == nat.PATH_PHASED
    assert all(torch.equal(a, b) for a, b in zip(m.e[:L] + m.x + m.w, e[:L] + x + w))
