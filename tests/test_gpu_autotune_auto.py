"""The automatic choice is a candidate of the tuner: kept where nothing beats it
clearly, so that a tuned net is not slower than an untuned one."""
import pytest
import torch

from lich_amd import HipIPC, IPCConfig, autotune as AT
from lich_amd.trainer import init_weights_cpu
from tests.helpers import DEV, report

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("auto_us,want", [(9.0, -1), (10.0, -1), (10.1, -1), (11.0, 1)])
def test_standalone_tuner_keeps_the_automatic_choice_on_a_tie(auto_us, want):
    report("autotune-auto-kernels", auto_us=auto_us)
    timer = lambda kind, M, K, tile, us: auto_us if tile == -1 else 10.0 if tile == 1 else 20.0  # noqa: E731
    table = AT.tune_standalone([(64, 784, 128)], "relu", torch.float16, reps=1, replays=1, timer=timer)
    assert len(table.entries) == 3 and all(e.config.tile_id() == want for e in table.entries)


def test_wide_tuner_keeps_the_automatic_choice_and_the_plan_runs_it():
    report("autotune-auto-wide")
    dims, B = (10, 512, 512, 512, 784), 256
    seen = []

    def timer(phase, cand, us):
        seen.append((phase, *cand))
        return 10.0 if cand[0] == -1 else 10.05 if phase == "infer" else 5.0 if (phase, cand[0]) == ("weight", 1) else 30.0

    chosen = AT.tune_wide(dims, B, "tanh", torch.float16, reps=1, replays=1, timer=timer)
    assert chosen == {"pred": -1, "infer": -1, "weight": 1, "ksplit": -1}
    assert ("pred", -1, 1) in seen  # the k-split varies with it
    w0 = init_weights_cpu(dims, seed=1, init="xavier_uniform")
    x = torch.rand((784, B), generator=torch.Generator().manual_seed(1)).to(DEV)
    y = torch.nn.functional.one_hot(torch.arange(B) % 10, 10).float().T.contiguous().to(DEV)
    outs = []
    for wc in (None, (-1, -1, 1, -1)):
        m = HipIPC(IPCConfig(dims=dims, activation="tanh", dtype=torch.float16, wide_config=wc,
                             hierarchical_policy_auto=False), device=DEV, weights=w0)
        m.initialize_batch(x, y)
        m.run_steps(2)
        outs.append([t.clone() for t in m.x + m.e[:-1] + m.w])
    torch.cuda.synchronize()
    assert m.path == "wide" and all(torch.equal(a, b) for a, b in zip(*outs))
