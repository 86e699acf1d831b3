"""The rank-B outer-product weight update at the edges of its tiles (256 columns,
8 or 16 rows), with rows and bases that allow 4-element loads and that do not."""
import pytest
import torch

from lich_amd import build_weight_update_outer
from tests.helpers import DEV, report

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,K,B,groups,dt,shift", [
    (1, 1, 1, 1, torch.float32, 0), (7, 260, 32, 1, torch.float32, 0), (9, 257, 5, 2, torch.bfloat16, 0),
    (130, 1024, 12, 1, torch.float16, 0), (129, 4097, 9, 3, torch.float32, 0), (2047, 1028, 8, 1, torch.bfloat16, 0),
    (33, 512, 16, 1, torch.float16, 1), (520, 4096, 4, 1, torch.float32, 3), (515, 4092, 3, 1, torch.bfloat16, 2),
])
def test_outer_at_tile_edges(M, K, B, groups, dt, shift):
    """`shift`: elements by which W and X start off their allocation."""
    report("outer-edges", M=M, K=K, B=B, groups=groups, dt=str(dt), shift=shift)
    g = torch.Generator().manual_seed(M + K + B)

    def make(rows, cols):
        flat = torch.randn(groups * rows * cols + shift, generator=g).to(dt).to(DEV)
        t = flat[shift:].view(groups, rows, cols)
        return t if groups > 1 else t[0]

    w, x, e = make(M, K), make(K, B), make(M, B).clone()
    w0, alpha = w.double().cpu(), 0.25
    a = torch.relu(x).double().cpu()
    build_weight_update_outer(M, K, B, "relu", dt, alpha, True, groups)(w, e, x)
    torch.cuda.synchronize()
    ref = w0 + alpha * (e.double().cpu() @ a.transpose(-1, -2).contiguous())
    # B products and sums, the scaling and the addition round in fp32 (relative
    # to the sum of magnitudes), the result once more in the storage type
    mag = w0.abs() + alpha * (e.double().cpu().abs() @ a.transpose(-1, -2).contiguous())
    unit = {torch.float32: 0.0, torch.float16: 2.0 ** -11, torch.bfloat16: 2.0 ** -8}[dt]
    bound = (B + 3) * 2.0 ** -24 * mag * (1 + unit) + unit * ref.abs() + 2.0 ** -25
    assert ((w.double().cpu() - ref).abs() <= bound).all()


@pytest.mark.parametrize("K", [1, 63, 64, 65, 128, 129, 192, 257, 320])
@pytest.mark.parametrize("B,dt,shift", [(7, torch.float32, 0), (9, torch.float16, 0), (24, torch.bfloat16, 0),
                                        (32, torch.float32, 0), (31, torch.float32, 1), (12, torch.float16, 1)])
def test_outer_where_threads_share_a_column(K, B, dt, shift):
    """Blocks of at most 64, 128 and 256 columns, whole and partial groups of 8 batch values."""
    test_outer_at_tile_edges(21, K, B, 1, dt, shift)
