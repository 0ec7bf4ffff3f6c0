"""Row lengths on both sides of every step of the fused producers' dispatch, whose last vectors lie beyond the row.  The
gather has no transcendental: codes and scales are the oracle's bits; the gated product is held to the bounds of
tests/test_moe_gpu.py."""
import pytest
import torch

from mslk_amd import moe
from oracle import fp8_rowwise_oracle as O
from tests.helpers import bits32, codes

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
STEPS = [8, 512, 520, 1024, 1032, 2048, 2056, 4096, 4104, 6144, 6152, 8192, 8200, 16384, 16392]


@pytest.mark.parametrize("rows,Ds", [(7, STEPS), (2053, STEPS[:7]), (2053, [1536, 1544])])
def test_gather_and_gated_product_around_every_step(rows, Ds):
    g = torch.Generator().manual_seed(rows)
    for D in Ds:
        x = torch.randn(rows, 2 * D, generator=g).bfloat16()
        x[0, D - 1] = 30.0        # the maximum in the last vector
        x[0, 2 * D - 1] = 2.0
        token, expert = torch.randperm(rows, generator=g).int(), torch.randint(0, 3, (rows,), generator=g).int()
        scores = torch.randn(rows, 3, generator=g)
        xd = x.to(DEV)
        q, s = moe.gather_scale_quant_dense_tokens(xd[:, :D].contiguous(), token.to(DEV), expert.to(DEV), scores.to(DEV))
        rq, rs = O.gather_scale_quant_dense_tokens(x[:, :D].contiguous(), token, expert, scores)
        assert torch.equal(codes(q), codes(rq)) and torch.equal(bits32(s), bits32(rs)), f"gather, D = {D}"
        q, s = moe.silu_mul_quant(xd[:, :D], xd[:, D:])
        rq, rs = O.silu_mul_quant(x[:, :D], x[:, D:])
        assert torch.allclose(s.cpu(), rs, rtol=2e-6, atol=0), f"gated product, D = {D}"
        a, b = codes(q).int(), codes(rq).int()
        steps = (torch.where(a > 127, 128 - a, a) - torch.where(b > 127, 128 - b, b)).abs()
        # (one code of the shortest row already exceeds the share that is allowed)
        assert steps.max() <= 1 and (steps != 0).sum() <= max(1, 2e-4 * steps.numel()), f"gated product, D = {D}"


def test_an_infinite_score_leaves_an_infinite_scale():
    """Lanes beyond the row hold zero, and zero times infinity must not reach the row's maximum."""
    x = torch.ones(3, 2056, dtype=torch.bfloat16, device=DEV)
    index = torch.arange(3, dtype=torch.int32, device=DEV)
    scores = torch.tensor([[1.0], [float("inf")], [float("nan")]], device=DEV)
    _, s = moe.gather_scale_quant_dense_tokens(x, index, torch.zeros_like(index), scores)
    s = s.cpu()
    assert torch.isfinite(s[0]) and torch.isinf(s[1]) and torch.isnan(s[2])
