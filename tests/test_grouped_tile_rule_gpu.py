"""Groups of rows take 128 x 128 or 256 x 256 tiles by the rows per group and the tile count: sizes on both sides of that line and
at the edges of both tiles, as lists, sizes and offsets.  Integer codes and power-of-two scales: the fp32 sums are exact and the
outputs compare bit for bit."""
import pytest
import torch

import mslk_amd  # noqa: F401

pytestmark = pytest.mark.gpu
DEV, F8 = "cuda:0", torch.float8_e4m3fn


@pytest.mark.parametrize("sizes,N,K", [
    ([1, 127, 128, 129, 0, 255, 256, 257], 520, 528),                # few tiles, K and N remainders
    ([128] * 8, 8192, 512),                                          # 128 rows per group: small tiles, a full pass of them
    ([129] * 8, 8200, 512),                                          # one more: large tiles
    ([1100, 3, 64, 65, 192, 193], 6152, 640),                        # large tiles, every ragged height
    ([16 * (i % 5) + 1 for i in range(70)], 1032, 512),              # a list of more groups than one launch holds
    ([1024], 8192, 512),                                             # 512 small tiles
    ([1025], 8192, 512),                                             # 576
    ([2048] * 4, 1024, 512),                                         # sizes on the device, full tiles of a short K: small ones
    ([2049, 2047, 2000, 2096], 1024, 768),                           # a longer K: large ones
    ([130] + [2] * 7, 8192, 512),                                    # as a list: two passes of small tiles, one of large ones
    ([130] + [2] * 8, 8192, 512),                                    # two passes of either: small ones
    ([37, 410, 200], 1000, 520),                                     # K % 16 != 0: scalar tiles
])
def test_rows_of_every_group(sizes, N, K):
    g = torch.Generator().manual_seed(len(sizes) + N + K)
    G, total = len(sizes), sum(sizes)
    x = torch.randint(-8, 9, (total, K), generator=g).float()
    w = torch.randint(-8, 9, (G, N, K), generator=g).float()
    xs = torch.pow(2.0, torch.randint(-3, 4, (total,), generator=g).float())
    ws = torch.pow(2.0, torch.randint(-3, 4, (G, N), generator=g).float())
    parts = zip(x.split(sizes), w, ws, xs.split(sizes))
    want = torch.cat([((a @ b.t()) * s * r[:, None]).to(torch.bfloat16) for a, b, s, r in parts])
    xq, wq, xs, ws = x.to(F8).to(DEV), w.to(F8).to(DEV), xs.to(DEV), ws.to(DEV)
    m = torch.tensor(sizes)
    assert torch.equal(torch.ops.mslk.f8f8bf16_rowwise_grouped_stacked(xq, wq, xs, ws, m.to(DEV)).cpu(), want)
    out = torch.full((total, N), 777.0, dtype=torch.bfloat16, device=DEV)
    torch.ops.mslk.f8f8bf16_rowwise_grouped_mm(xq, wq, xs, ws, m.cumsum(0).to(torch.int32).to(DEV), out)
    assert torch.equal(out.cpu(), want)
    lists = [list(xq.split(sizes)), list(wq.unbind(0)), list(xs.split(sizes)), list(ws.unbind(0))]
    assert torch.equal(torch.ops.mslk.f8f8bf16_rowwise_grouped_cat(*lists).cpu(), want)
