"""The wide path's 64 x 64 tiles, which a plan picks where the default tiles
would leave most CUs idle: every launch's configuration gives the bits of the
default one (configuration 0 asked for explicitly), on nets at the tile's edges,
with and without the copies of W (contractions off the 64-k grid), k-split output
layers and the saved activations, and the first hidden errors stay exactly 0."""
import pytest
import torch

from lich_amd import HipIPC, IPCConfig
from oracle import ipc_oracle as O
from tests.helpers import DEV, report

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims,B,op,split,act,save", [
    ((10, 200, 200, 784), 64, torch.bfloat16, 2, "tanh", False),
    ((10, 193, 65, 129), 33, torch.float16, 2, "silu", True),      # one past the tiles, odd batch
    ((10, 192, 64, 128), 1, torch.float16, 1, "relu", False),
    ((64, 1024, 640, 64), 130, torch.bfloat16, 2, "gelu", True),   # W read directly, k-split layer 0
    ((1, 130, 4096), 63, torch.float16, 2, "sigmoid", False),
])
def test_small_tiles_give_the_default_bits(dims, B, op, split, act, save):
    report("wide-small", dims=dims, B=B, op=op, split=split, act=act)
    w0 = O.init_weights(dims, seed=3, init="xavier_uniform")
    x, _l, y = O.make_batch(dims, B, seed=3)
    outs = []
    for cfg in (None, (0, 0, 0, -1)):
        m = HipIPC(IPCConfig(dims=dims, activation=act, dtype=op, pred_split=split, fused="wide", wide_config=cfg,
                             recompute_activation=not save), device=DEV, weights=w0)
        m.initialize_batch(x.to(DEV), y.to(DEV))
        m.run_steps(1)
        torch.cuda.synchronize()
        assert all(torch.count_nonzero(m.e[l]) == 0 for l in range(1, len(dims) - 1))
        m.run_steps(2)
        torch.cuda.synchronize()
        outs.append([t.clone() for t in m.x + m.e[:-1] + m.w + ([] if m.a is None else m.a[1:])])
    assert all(torch.equal(a, b) for a, b in zip(*outs))
