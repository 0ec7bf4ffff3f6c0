"""256 x 256 tiles of row groups one after the other: every workgroup walks several tiles whose K steps form one chain, a K that is
no multiple of the step ends in a step over the last 128 bytes, and what does not fill a last pass goes to further workgroups.
Integer codes and power-of-two scales: the fp32 sums are exact and the outputs compare bit for bit."""
import pytest
import torch

import mslk_amd  # noqa: F401
from tests.helpers import grouped_kernel, grouped_list_kernel

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
    """The last step of K = 400 reads bytes the step before has consumed: they count once, and codes of the rows around do not."""
    sizes, N, K = [2300, 2400], 8192, 400   # 76 tiles for the 32 CUs of an XCD: two walked each, twelve left over
    assert grouped_kernel(0, len(sizes), sum(sizes), N, K).startswith("grouped_rows<256,256>")
    xq, wq, xs, ws, finite = _operands(sizes, N, K)
    x8, w8 = xq.view(torch.uint8), wq.view(torch.uint8)
    rows = [5, 255, 2299, 2300, 4698]               # among them the last one of a tile and of a group, and the first of a group
    cols = {0: [77, 256, 8191], 1: [0, 300, 8190]}
    places = [272, 383, 384, 399, 0]                # consumed by the step before: from 272 on; by the last one alone: from 384 on
    for row, k in zip(rows, places):
        x8[row, k] = 0x7F
    for g, k in ((0, 300), (1, 390)):
        for col in cols[g]:
            w8[g, col, k] = 0x7F
    want = finite.clone()
    want[rows] = float("nan")
    want[:2300, cols[0]] = float("nan")
    want[2300:, cols[1]] = float("nan")
    out = torch.ops.mslk.f8f8bf16_rowwise_grouped_stacked(xq, wq, xs, ws, torch.tensor(sizes).to(DEV)).cpu()
    assert torch.equal(torch.isnan(out), torch.isnan(want))
    assert torch.equal(out.nan_to_num(0.0), want.nan_to_num(0.0))


def test_lists_of_different_k():
    """A list may hold groups of different K: the chain changes over from one row pitch to another, and between rows that are a whole number
    of steps and rows that are not.  At most 32 tiles per panel and 33 entries from one tile of a workgroup to its next (but where its
    entries go round the end of a pass): the two are of different groups, and no two groups have the same K."""
    rows = [(700, 300, 513, 900, 256, 1000)[i % 6] for i in range(44)]
    ks = [512 + 16 * ((i * 13) % 44) for i in range(44)]
    N = 2040   # the last column tile is not full
    assert len(set(ks)) == len(ks) and any(k % 128 == 0 for k in ks)
    kernel = grouped_list_kernel(rows, N, ks)
    assert kernel.startswith("grouped_listed<256,256>") and _longest(kernel) >= 96, kernel   # three tiles per workgroup
    parts = [_operands([m], N, k) for m, k in zip(rows, ks)]
    out = torch.ops.mslk.f8f8bf16_rowwise_grouped([p[0] for p in parts], [p[1][0] for p in parts], [p[2] for p in parts], [p[3][0] for p in parts])
    for y, p in zip(out, parts):
        assert torch.equal(y.cpu(), p[4])


def _longest(kernel):
    return int(kernel.split("longest=")[1].split()[0])


def test_left_over_tiles_of_lists_in_quarters():
    sizes, N, K = [2304], 8192, 528
    kernel = grouped_list_kernel(sizes, N, K)
    assert kernel.startswith("grouped_listed<256,256>")
    left = _longest(kernel) - 32
    assert 1 <= left <= 8, kernel   # at most a quarter of the 32 CUs of an XCD
    xq, wq, xs, ws, want = _operands(sizes, N, K)
    out = torch.ops.mslk.f8f8bf16_rowwise_grouped([xq], [wq[0]], [xs], [ws[0]])
    assert torch.equal(out[0].cpu(), want)


@pytest.mark.parametrize("form,sizes,N,K", [
    ("sizes", [8000, 300, 8596], 65536, 272),
    ("offsets", [129 + i % 128 for i in range(130)], 32768, 272),   # more groups than two lookups hold
    ("list", [8000, 300, 8596], 65536, 512),
])
def test_more_tiles_than_one_lookup_finds(form, sizes, N, K):
    """A workgroup finds 64 of its tiles at a time: more than 64 * 256 of them."""
    total, G = sum(sizes), len(sizes)
    assert sum((m + 255) // 256 for m in sizes) * (N // 256) > 64 * 256
    kernel = grouped_list_kernel(sizes, N, K) if form == "list" else grouped_kernel(1 if form == "offsets" else 0, G, total, N, K)
    assert kernel.startswith("grouped_listed<256,256>" if form == "list" else "grouped_rows<256,256>"), kernel
    if form == "list":
        assert _longest(kernel) > 64 * 32 + 32
    g = torch.Generator(device=DEV).manual_seed(N + K + G)
    codes = torch.arange(-8, 9, device=DEV).float().to(F8).view(torch.uint8)
    draw = lambda *shape: codes[torch.randint(0, 17, shape, generator=g, device=DEV, dtype=torch.int32)].view(F8)
    xq, wq = draw(total, K), torch.stack([draw(N, K).view(torch.uint8) for _ in sizes]).view(F8)
    xs = torch.pow(2.0, torch.randint(-3, 4, (total,), generator=g, device=DEV).float())
    ws = torch.pow(2.0, torch.randint(-3, 4, (G, N), generator=g, device=DEV).float())
    m = torch.tensor(sizes, device=DEV)
    if form == "sizes":
        out = torch.ops.mslk.f8f8bf16_rowwise_grouped_stacked(xq, wq, xs, ws, m)
    elif form == "offsets":
        out = torch.empty(total, N, dtype=torch.bfloat16, device=DEV)
        torch.ops.mslk.f8f8bf16_rowwise_grouped_mm(xq, wq, xs, ws, m.cumsum(0).to(torch.int32), out)
    else:
        out = torch.cat(torch.ops.mslk.f8f8bf16_rowwise_grouped(list(xq.split(sizes)), list(wq.unbind(0)), list(xs.split(sizes)), list(ws.unbind(0))))
    row = 0
    for i, size in enumerate(sizes):   # sums below 2^24: exact in fp32
        w = wq[i].float()
        for r in range(row, row + size, 4096):
            e = min(r + 4096, row + size)
            want = ((xq[r:e].float() @ w.t()) * ws[i] * xs[r:e, None]).to(torch.bfloat16)
            assert torch.equal(out[r:e], want), (i, r)
        row += size


@pytest.mark.parametrize("K", [2880, 1040, 400])
def test_rows_do_not_depend_on_the_tiles_they_fall_into(K):
    """Random codes of the whole range, whose sums round: the last step of the chain has its codes at the end of the matrix instruction's
    k positions and zeros in front, the other tiles the reverse, and the sums are the same bit for bit."""
    N, rows = 8192, 2304
    g = torch.Generator().manual_seed(K)
    draw = lambda *shape: (torch.randint(0, 127, shape, generator=g) + 128 * torch.randint(0, 2, shape, generator=g)).to(torch.uint8).view(F8).to(DEV)
    xq, wq = draw(2 * rows, K), draw(2, N, K)
    xs, ws = (torch.rand(n, generator=g).add(0.5).to(DEV) for n in ((2 * rows,), (2, N)))
    stacked = lambda x, w, s, t, sizes: torch.ops.mslk.f8f8bf16_rowwise_grouped_stacked(x, w, s, t, torch.tensor(sizes).to(DEV))
    assert grouped_kernel(0, 2, 2 * rows, N, K) == grouped_kernel(0, 1, rows, N, K) == "grouped_rows<256,256> workgroups=512"
    walked = stacked(xq, wq, xs, ws, [rows, rows])[:rows]                    # 72 tiles for the 32 CUs of an XCD: two each, eight left over
    quarters = stacked(xq[:rows], wq[:1], xs[:rows], ws[:1], [rows])         # 36: the last four in quarters
    assert grouped_kernel(0, 1, 128, N, K).startswith("grouped_device<128,128>")
    small = torch.cat([stacked(xq[r:r + 128], wq[:1], xs[r:r + 128], ws[:1], [128]) for r in range(0, rows, 128)])
    assert torch.equal(walked, quarters) and torch.equal(walked, small)
