"""2D-2D grouped products: workgroups take the K slices longest first and in runs dealt to the XCDs, so every tile of every
group has to be written exactly once whatever the tile count per group and the order of the lengths.  Integer codes and
power-of-two scales: the fp32 sums are exact and the outputs compare bit for bit."""
import pytest
import torch

import mslk_amd  # noqa: F401

pytestmark = pytest.mark.gpu
DEV, F8 = "cuda:0", torch.float8_e4m3fn


def _run(ks, M, N):
    g = torch.Generator().manual_seed(sum(ks) + M + N)
    G, total = len(ks), sum(ks)
    xi, wi = (torch.randint(-8, 9, (r, total), generator=g).float() for r in (M, N))
    xs, ws = (torch.pow(2.0, torch.randint(-3, 4, (G * r,), generator=g).float()) for r in (M, N))
    out = torch.full((G, M, N), 777.0, dtype=torch.bfloat16, device=DEV)
    ends = torch.tensor(ks).cumsum(0).to(torch.int32).to(DEV)
    torch.ops.mslk.f8f8bf16_rowwise_grouped_mm(xi.to(F8).to(DEV), wi.to(F8).to(DEV), xs.to(DEV), ws.to(DEV), ends, out)
    torch.cuda.synchronize()
    k0 = 0
    for gi, k in enumerate(ks):
        want = (xi[:, k0:k0 + k] @ wi[:, k0:k0 + k].t()) * ws[gi * N:(gi + 1) * N] * xs[gi * M:(gi + 1) * M, None]
        assert torch.equal(out[gi].cpu(), want.to(torch.bfloat16)), f"group {gi}, slice of {k}"
        k0 += k


@pytest.mark.parametrize("ks,M,N", [
    ([16 * (i * 7 % 11) for i in range(70)], 100, 120),    # one tile per group, more groups than lanes, equal and empty slices
    ([48, 400, 0, 400, 128, 16], 300, 296),                # nine tiles: runs of two, the last run of a group reaches into the next
    ([16 * (i % 5) for i in range(16)], 1000, 704),        # twelve 256-row tiles per group
    ([640], 2000, 1912),                                   # one group
    ([256, 128, 512], 130, 40),                            # two tiles: fewer than XCDs
])
def test_every_tile_of_every_slice(ks, M, N):
    _run(ks, M, N)


@pytest.mark.parametrize("ks,M,N", [
    ([128] * 6, 1000, 1104),                               # 72 tiles per group, more than a tile per CU: groups in order ...
    ([16, 48, 1024, 16, 0, 16], 1000, 1104),               # ... and by falling length, dealt to the XCDs
    ([112, 128, 96, 128, 128, 112, 128], 1000, 1104),      # nearly equal: in order, XCDs begin inside a group
    ([16] * 65 + [4096], 1408, 1400),                      # the longest slice behind the first 64 groups
    ([16 * (i % 3) for i in range(66)], 1408, 1400),
    ([32] * 40, 640, 640),                                 # 25 tiles per group: too few to deal out
])
def test_both_orders_of_the_slices(ks, M, N):
    _run(ks, M, N)
