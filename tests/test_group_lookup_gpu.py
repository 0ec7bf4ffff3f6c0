"""Extents of more than 64 groups in device memory: the lookup keeps the first 128 groups in registers and reads the rest 64 at
a time, so groups around those edges, empty ones and inconsistent extents are checked against a product per group.  Integer
codes and power-of-two scales: the fp32 sums are exact and the outputs compare bit for bit."""
import pytest
import torch

import mslk_amd  # noqa: F401

pytestmark = pytest.mark.gpu
DEV, F8 = "cuda:0", torch.float8_e4m3fn
N, K = 64, 256


def _sizes(G, seed):
    g = torch.Generator().manual_seed(seed)
    sizes = torch.randint(0, 9, (G,), generator=g)
    for i in (0, 63, 64, 127, 128, G - 1):
        if i < G:
            sizes[i] = (i % 3) * 70   # empty, or more than one 64-row half of a tile
    return sizes


def _operands(total, G, seed):
    g = torch.Generator().manual_seed(seed)
    x = torch.randint(-8, 9, (total, K), generator=g).float()
    w = torch.randint(-8, 9, (G, N, K), generator=g).float()
    xs = torch.pow(2.0, torch.randint(-3, 4, (total,), generator=g).float())
    ws = torch.pow(2.0, torch.randint(-3, 4, (G, N), generator=g).float())
    return x, w, xs, ws


def _want(x, w, xs, ws, sizes, total):
    out, r0 = torch.full((total, N), 777.0, dtype=torch.bfloat16), 0
    for gi, m in enumerate(sizes.tolist()):
        out[r0:r0 + m] = ((x[r0:r0 + m] @ w[gi].t()) * ws[gi] * xs[r0:r0 + m, None]).to(torch.bfloat16)
        r0 += m
    return out


@pytest.mark.parametrize("G", [1, 63, 64, 65, 127, 128, 129, 192, 200])
@pytest.mark.parametrize("spare", [0, 5])
def test_rows_of_every_group(G, spare):
    """`spare`: rows behind the last group belong to nobody and stay as they were."""
    sizes = _sizes(G, G)
    total = int(sizes.sum()) + spare
    x, w, xs, ws = _operands(total, G, G + 1)
    want = _want(x, w, xs, ws, sizes, total)
    d = [x.to(F8).to(DEV), w.to(F8).to(DEV), xs.to(DEV), ws.to(DEV)]
    out = torch.full((total, N), 777.0, dtype=torch.bfloat16, device=DEV)
    torch.ops.mslk.f8f8bf16_rowwise_grouped_mm(*d, sizes.cumsum(0).to(torch.int32).to(DEV), out)
    assert torch.equal(out.cpu(), want)
    got = torch.ops.mslk.f8f8bf16_rowwise_grouped_stacked(*d, sizes.to(DEV)).cpu()
    used = total - spare
    assert torch.equal(got[:used], want[:used])


@pytest.mark.parametrize("G", [65, 129, 200])
def test_columns_of_every_group(G):
    sizes = _sizes(G, G)
    total = int(sizes.sum())
    x, w, xs, ws = _operands(total, G, G + 1)   # rows of the offsets side; here WQ carries the offsets
    out = torch.empty((N, total), dtype=torch.bfloat16, device=DEV)
    torch.ops.mslk.f8f8bf16_rowwise_grouped_mm(w.to(F8).to(DEV), x.to(F8).to(DEV), ws.to(DEV), xs.to(DEV),
                                               sizes.cumsum(0).to(torch.int32).to(DEV), out)
    want, r0 = torch.empty((N, total), dtype=torch.bfloat16), 0
    for gi, m in enumerate(sizes.tolist()):
        want[:, r0:r0 + m] = ((w[gi] @ x[r0:r0 + m].t()) * xs[r0:r0 + m] * ws[gi][:, None]).to(torch.bfloat16)
        r0 += m
    assert torch.equal(out.cpu(), want)


@pytest.mark.parametrize("bad", [3, 64, 100, 130])
def test_groups_from_the_first_inconsistent_one_on_write_nothing(bad):
    G = 140
    sizes = _sizes(G, 5)
    total = int(sizes.sum())
    x, w, xs, ws = _operands(total, G, 6)
    d = [x.to(F8).to(DEV), w.to(F8).to(DEV), xs.to(DEV), ws.to(DEV)]
    good = sizes.clone()
    good[bad:] = 0
    want = _want(x, w, xs, ws, good, total)
    ends = sizes.cumsum(0).to(torch.int32)
    ends[bad] = total + 1   # beyond the rows
    out = torch.full((total, N), 777.0, dtype=torch.bfloat16, device=DEV)
    torch.ops.mslk.f8f8bf16_rowwise_grouped_mm(*d, ends.to(DEV), out)
    assert torch.equal(out.cpu(), want)
    wrong = sizes.clone()
    wrong[bad] = 2 ** 40
    got = torch.ops.mslk.f8f8bf16_rowwise_grouped_stacked(*d, wrong.to(DEV)).cpu()
    used = int(good.sum())
    assert torch.equal(got[:used], want[:used])
