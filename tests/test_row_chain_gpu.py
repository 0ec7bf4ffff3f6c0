"""256 x 256 tiles of row groups one after the other: every workgroup walks several tiles whose K steps form one chain, a K that is
no multiple of the step ends in a step over the last 128 bytes, and what does not fill a last pass goes to further workgroups.
Integer codes and power-of-two scales: the fp32 sums are exact and the outputs compare bit for bit."""
import pytest
import torch

import mslk_amd  # noqa: F401
from tests.helpers import grouped_kernel

pytestmark = pytest.mark.gpu
DEV, F8 = "cuda:0", torch.float8_e4m3fn


def _operands(sizes, N, K):
    g = torch.Generator().manual_seed(len(sizes) + N + K)
    G, total = len(sizes), sum(sizes)
    x = torch.randint(-8, 9, (total, K), generator=g).float()
    w = torch.randint(-8, 9, (G, N, K), generator=g).float()
    xs = torch.pow(2.0, torch.randint(-3, 4, (total,), generator=g).float())
    ws = torch.pow(2.0, torch.randint(-3, 4, (G, N), generator=g).float())
    parts = zip(x.split(sizes), w, ws, xs.split(sizes))
    want = torch.cat([((a @ b.t()) * s * r[:, None]).to(torch.bfloat16) for a, b, s, r in parts])
    return x.to(F8).to(DEV), w.to(F8).to(DEV), xs.to(DEV), ws.to(DEV), want


@pytest.mark.parametrize("sizes,N,K", [
    ([257, 300, 1, 511, 64, 65, 128, 129, 192, 193, 256], 4096, 272),   # three steps, the last of 16 bytes; every ragged height
    ([2304], 8192, 384),               # 36 tiles for the 32 CUs of an XCD: the last four in quarters
    ([256] * 5 + [200] * 8, 8192, 400),   # 52 tiles: twenty left over, a tail of 16 bytes
    ([700] * 5, 8192, 640),            # 60 tiles: more than three quarters of a pass left over, walked
    ([2000, 300, 5, 40], 8008, 512),   # the last column tile is not full
    ([900, 901], 7944, 1040),          # ... and leaves less than half a tile
    ([1500, 1500], 8192, 256),         # two steps: not for the chain
    ([129 + i % 140 for i in range(130)], 2048, 384),   # more groups than two lookups hold
])
def test_tiles_in_a_chain(sizes, N, K):
    xq, wq, xs, ws, want = _operands(sizes, N, K)
    m = torch.tensor(sizes)
    assert torch.equal(torch.ops.mslk.f8f8bf16_rowwise_grouped_stacked(xq, wq, xs, ws, m.to(DEV)).cpu(), want)
    out = torch.full((sum(sizes), N), 777.0, dtype=torch.bfloat16, device=DEV)
    torch.ops.mslk.f8f8bf16_rowwise_grouped_mm(xq, wq, xs, ws, m.cumsum(0).to(torch.int32).to(DEV), out)
    assert torch.equal(out.cpu(), want)
    if K < 512:
        return   # lists take no shorter rows
    lists = [list(xq.split(sizes)), list(wq.unbind(0)), list(xs.split(sizes)), list(ws.unbind(0))]
    assert torch.equal(torch.ops.mslk.f8f8bf16_rowwise_grouped_cat(*lists).cpu(), want)


@pytest.mark.parametrize("N", [8200, 8232, 8168, 8192 + 56])
@pytest.mark.parametrize("sizes", [[263, 264, 265, 271, 272, 273, 7, 8, 9], [1031, 1032, 1033, 15, 16, 17]])
def test_stores_of_ragged_tiles(sizes, N):
    """Eight rows and 64 columns go out together: rows that end next to a multiple of eight, columns inside a group of 64; and nothing
    beyond them is written."""
    K = 400
    xq, wq, xs, ws, want = _operands(sizes, N, K)
    rows = sum(sizes)
    assert grouped_kernel(0, len(sizes), rows, N, K).startswith("grouped_rows<256,256>")
    buffer = torch.full((rows + 64, N), 777.0, dtype=torch.bfloat16, device=DEV)
    off = torch.tensor(sizes).cumsum(0).to(torch.int32).to(DEV)
    torch.ops.mslk.f8f8bf16_rowwise_grouped_mm(xq, wq, xs, ws, off, buffer[32:32 + rows])
    out = buffer.cpu()
    assert torch.equal(out[32:32 + rows], want)
    assert (out[:32] == 777.0).all() and (out[32 + rows:] == 777.0).all()


def test_codes_beyond_a_row_do_not_count():
    """The last step of K = 400 reads bytes the step before has consumed, and NaN codes among them count once."""
    sizes, N, K = [600, 700], 2048, 400
    xq, wq, xs, ws, _ = _operands(sizes, N, K)
    xq.view(torch.uint8)[5, 300] = 0x7F
    wq.view(torch.uint8)[1, 77, 390] = 0x7F
    out = torch.ops.mslk.f8f8bf16_rowwise_grouped_stacked(xq, wq, xs, ws, torch.tensor(sizes).to(DEV)).float()
    nan = torch.isnan(out)
    want = torch.zeros_like(nan)
    want[5, :] = True
    want[600:, 77] = True
    assert torch.equal(nan, want)


def test_lists_of_different_k():
    """A list may hold groups of different K: the chain changes over from one row pitch to another."""
    parts = [_operands([rows], 4096, K) for rows, K in ((700, 512), (300, 1024), (513, 528), (900, 640), (256, 1536))]
    out = torch.ops.mslk.f8f8bf16_rowwise_grouped([p[0] for p in parts], [p[1][0] for p in parts], [p[2] for p in parts], [p[3][0] for p in parts])
    for y, p in zip(out, parts):
        assert torch.equal(y.cpu(), p[4])
