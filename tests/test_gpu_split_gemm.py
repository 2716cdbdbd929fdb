"""The batched product on split operands (three bf16 parts per fp32 value) against float64, at the edges of its four
tiles (64 x 64, 128 x 128, 256 x 128, 128 x 256), of its steps of 32 values of k and of their fold every 128."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"

# 256 products of these sizes take the named tile on 256 compute units
TILES = {"64x64": (64, 64), "128x128": (128, 128), "256x128": (256, 128), "128x256": (128, 256)}


@pytest.mark.parametrize("akm,bkm", [(0, 0), (0, 1), (1, 0), (1, 1)])
@pytest.mark.parametrize("k", [1, 32, 65, 129, 260])
@pytest.mark.parametrize("tile,less", [("64x64", 0), ("64x64", 1), ("128x128", 0), ("128x128", 3), ("256x128", 0),
                                       ("256x128", 2), ("128x256", 0), ("128x256", 1)])
def test_split_product_at_tile_edges(pbg, tile, less, k, akm, bkm):
    m, n = (x - less for x in TILES[tile])
    print("split gemm", tile, m, n, k, akm, bkm, flush=True)
    batch = 256
    g = torch.Generator(device=DEV).manual_seed(m * n + k)
    # magnitudes over 12 binades: every part of every value counts
    draw = lambda *s: torch.randn(*s, generator=g, device=DEV) * torch.exp2(torch.randint(-6, 7, s, generator=g, device=DEV).float())
    a, b = draw(batch, *((k, m) if akm else (m, k))), draw(batch, *((k, n) if bkm else (n, k)))
    c = torch.full((batch, m, n), float("nan"), device=DEV)
    pbg.native.gemm(a, b, c, batch, m, n, k, a.shape[2], b.shape[2], n, m * k, n * k, m * n, akm, bkm, alpha=0.5)
    a64, b64 = a.double(), b.double()
    a64 = a64.transpose(1, 2).contiguous() if akm else a64
    b64 = b64 if bkm else b64.transpose(1, 2).contiguous()
    want, size = 0.5 * torch.bmm(a64, b64), (0.5 * torch.bmm(a64.abs(), b64.abs())).clamp_min(1e-30)
    # the products left out are below 2^-26 of |a b|; a partial sum takes at most 24 instructions (128 values of k, six part
    # pairs), each rounding its result once (half an ulp of at most the sum of |a b|) and aligning its 32 products to 2^-24 of
    # the largest; then one addition per partial sum
    bound = (2.0 ** -24) * (2 * 24 + k // 128 + 2) * size
    assert torch.isfinite(c).all()
    worst = ((c.double() - want).abs() / bound).max()
    assert float(worst) <= 1.0, float(worst)
    # and on the whole that of independent roundings: an entry takes N = 6 * min(k, 128) / 32 + k / 128 + 2 of them, each with
    # an rms of half an ulp / sqrt(3) <= 2^-24 / sqrt(3) of at most the sum of |a b|
    roundings = 6 * -(-min(k, 128) // 32) + k // 128 + 2
    rms = float((((c.double() - want) / size) ** 2).mean().sqrt())
    assert rms <= 2.0 ** -24 * (roundings / 3) ** 0.5, rms
