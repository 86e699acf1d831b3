"""The k-chunk kernel (generic calls with few output tiles) at the sizes where
it can go wrong: edges of its 16 / 32 / 64 tiles, contractions around its
128-k chunks and around one round of its 8 or 16 waves, odd row lengths and
2-byte-aligned bases in 16-bit storage, groups.

Every result is held to the float64 product of the rounded operands within
the bound of an fp32 sum of K products in any order, K * 2^-24 * sum |a||b|,
plus the roundings the epilogue makes (activations identity / relu, so that
the rounded operands are known exactly)."""
import pytest
import torch

from lich_amd import HipIPC, IPCConfig
from lich_amd.kernels import (InferenceUpdateKernel, KernelConfig, PredictionErrorKernel, WeightUpdateKernel,
                              build_forward)
from oracle import ipc_oracle as O
from tests.helpers import DEV, gen, randn, report

pytestmark = pytest.mark.gpu

DT = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}
UNIT = {"f32": 2.0 ** -24, "f16": 2.0 ** -11, "bf16": 2.0 ** -8}  # relative rounding of one value
SHAPES = [(1, 1, 1), (15, 127, 17), (17, 128, 15), (16, 129, 33), (33, 300, 65), (64, 1024, 63), (65, 1025, 31),
          (18, 2049, 20), (130, 31, 257), (800, 140, 1000)]


def _place(t, dt, shift):
    """A device copy whose base is `shift` elements past an aligned address."""
    buf = torch.zeros(t.numel() + 8, device=DEV, dtype=dt)
    v = buf[shift:shift + t.numel()].view(t.shape)
    v.copy_(t)
    return v


def _round(t, op):
    return t.to(DT[op]).double()


def _check(out, ref, slack, K, mag, st):
    """|out - ref| within the fp32 sum's bound and `slack` times one rounding of the storage type."""
    bound = (K + 4) * 2.0 ** -24 * mag + UNIT[st] * slack + 1e-30
    bad = (out.double().cpu() - ref).abs() > bound
    assert not bad.any(), f"{int(bad.sum())} of {bad.numel()} past the bound"


@pytest.mark.parametrize("shift", [0, 1])
@pytest.mark.parametrize("st,op", [("f32", "f32"), ("f32", "f16"), ("f16", "f16"), ("bf16", "bf16")])
@pytest.mark.parametrize("M,K,B", SHAPES)
def test_three_kernels_at_tile_and_chunk_edges(M, K, B, st, op, shift):
    report("chunk", M=M, K=K, B=B, st=st, op=op, shift=shift)
    g = gen(M + 3 * K + 7 * B)
    dt, cfg = DT[st], KernelConfig()
    xu, w, xl = (randn(s, g).to(dt).float() for s in ((K, B), (M, K), (M, B)))
    # prediction + error, relu in the loader
    e = _place(torch.zeros(M, B), dt, shift)
    PredictionErrorKernel("p", M, K, B, "relu", dt, cfg, DT[op])(_place(xu, dt, shift), _place(w, dt, shift),
                                                                 _place(xl, dt, shift), e)
    a, b = _round(w, op), _round(torch.relu(xu), op)
    acc, mag = a @ b, a.abs() @ b.abs()
    _check(e, xl.double() - acc, acc.abs() + 2 * (xl.double() - acc).abs(), K, mag, st)
    # inference update keeping f(X): W_lower [K][M] read transposed
    wl, el, er = (randn(s, g).to(dt).float() for s in ((K, M), (K, B), (M, B)))
    x, ao = _place(xl, dt, shift), _place(torch.zeros(M, B), dt, shift)
    InferenceUpdateKernel("i", M, K, B, "identity", dt, cfg, DT[op], gamma=0.5, save_activation=True)(
        x, _place(er, dt, shift), _place(wl, dt, shift), _place(el, dt, shift), ao)
    a, b = _round(wl, op).T.contiguous(), _round(el, op)
    acc, mag = a @ b, a.abs() @ b.abs()
    ref = xl.double() + 0.5 * (acc - er.double())
    slack = 2 * (ref.abs() + acc.abs() + er.double().abs())
    _check(x, ref, slack, K, mag, st)
    _check(ao, ref, slack, K, mag, st)
    # weight update, contraction over K columns of a batch
    w0 = randn((M, B), g).to(dt).float()
    eb, xb = randn((M, K), g).to(dt).float(), randn((B, K), g).to(dt).float()
    wd = _place(w0, dt, shift)
    WeightUpdateKernel("w", M, B, K, "relu", dt, cfg, DT[op], alpha=0.1, recompute_activation=True)(
        wd, _place(eb, dt, shift), _place(xb, dt, shift))
    a, b = _round(eb, op), _round(torch.relu(xb), op).T.contiguous()
    acc, mag = a @ b, a.abs() @ b.abs()
    ref = w0.double() + 0.1 * acc
    _check(wd, ref, 2 * ref.abs() + 0.2 * acc.abs(), K, 0.1 * mag, st)


@pytest.mark.parametrize("op", ["f32", "bf16"])
@pytest.mark.parametrize("M,K,B", [(15, 127, 17), (65, 1025, 63), (70, 2100, 40)])
def test_tiles_and_groups_give_the_same_bits(M, K, B, op):
    report("chunk-tiles", M=M, K=K, B=B, op=op)
    g = gen(5)
    xu, w, xl = (randn(s, g).to(DEV) for s in ((2, K, B), (2, M, K), (2, M, B)))
    outs = []
    for tile in (-1, 0, 1, 2):
        e = torch.empty((2, M, B), device=DEV)
        PredictionErrorKernel("p", M, K, B, "tanh", torch.float32, KernelConfig(tile=tile), DT[op], groups=2,
                              split=1 if op == "f32" else 3)(xu, w, xl, e)
        outs.append(e)
    one = torch.empty((M, B), device=DEV)
    PredictionErrorKernel("p", M, K, B, "tanh", torch.float32, KernelConfig(), DT[op],
                          split=1 if op == "f32" else 3)(xu[1], w[1], xl[1], one)
    assert all(torch.equal(outs[0], o) for o in outs[1:]) and torch.equal(one, outs[0][1])


def test_values_outside_the_operands_reach_no_result():
    """NaN right behind the operands in memory, and rows of NaN-free results
    next to a NaN row: only that row is NaN."""
    M, K, B = 37, 131, 21
    for st in ("f32", "f16"):
        dt = DT[st]
        def fenced(r, c):
            buf = torch.full((r * c + 64,), float("nan"), device=DEV, dtype=dt)
            v = buf[1:1 + r * c].view(r, c)
            v.copy_(torch.ones(r, c))
            return v
        w, xu, xl, e = fenced(M, K), fenced(K, B), fenced(M, B), fenced(M, B)
        w[3, 5] = float("nan")
        PredictionErrorKernel("p", M, K, B, "identity", dt, KernelConfig(), dt)(xu, w, xl, e)
        good = torch.cat([e[:3], e[4:]])
        assert torch.isnan(e[3]).all() and (good == 1 - K).all()
        x, el, wl = fenced(M, B), fenced(K, B), fenced(K, M)
        InferenceUpdateKernel("i", M, K, B, "identity", dt, KernelConfig(), dt, gamma=1.0, save_activation=False)(
            x, fenced(M, B), wl, el)
        assert (x == K).all()


@pytest.mark.parametrize("dims,B,op,split", [((10, 70, 300, 2100), 40, torch.float32, None),
                                             ((10, 90, 80, 3700), 33, torch.bfloat16, 3)])
def test_phased_plan_keeps_the_exact_wavefront(dims, B, op, split):
    """The forward initialisation and the prediction phase run the same kernel
    (on their own tiles): the hidden errors of the first step are exactly 0."""
    report("chunk-wavefront", dims=dims, B=B)
    w0 = O.init_weights(dims, seed=2, init="xavier_uniform")
    x, _l, y = O.make_batch(dims, B, seed=2)
    m = HipIPC(IPCConfig(dims=dims, activation="tanh", dtype=op, pred_split=split, fused="phased"), device=DEV,
               weights=w0)
    m.initialize_batch(x.to(DEV), y.to(DEV))
    m.run_steps(1)
    torch.cuda.synchronize()
    assert all(torch.count_nonzero(m.e[l]) == 0 for l in range(1, len(dims) - 1))
    assert torch.count_nonzero(m.e[0]) > 0
    out = torch.empty((dims[-2], B), device=DEV)
    build_forward(dims[-2], dims[-1], B, "tanh", torch.float32, operand_dtype=op, split=m.pred_split)(
        x.to(DEV), w0[-1].to(DEV), out)
    assert torch.equal(out, m.x[-2])
