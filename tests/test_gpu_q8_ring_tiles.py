"""The bf16 Q8_0 linear's tiles (32 x 128 to 256 x 256) at their edges, against 64 bits. The sizes are picked so that
the dispatch's costs choose the named tile."""
import pytest
import torch

pytestmark = pytest.mark.gpu
TDT = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}

TILES = [(tile, m, n, k) for k in (960, 1024) for tile, m, n in (
         ("32x128", 129, 1500), ("32x128", 160, 1537), ("64x128", 700, 1500), ("64x128", 704, 1601),
         ("128x128", 1400, 1500), ("128x128, two a CU", 7100, 1100), ("160x128", 1400, 3100), ("128x256", 1100, 7000),
         ("256x256", 1500, 6000))] \
    + [("32x128", 16, 32000, 256), ("32x128", 5, 32700, 512), ("32x128", 257, 4096, 64), ("128x128", 2049, 1024, 128)]


@pytest.mark.parametrize("ydt", ["bf16", "f32", "f16"])
@pytest.mark.parametrize("tile,m,n,k", TILES)
def test_q8_linear_ring_tiles(tile, m, n, k, ydt):
    """|error| <= (k / 32 + 40) 2^-23 sum |x w| (an f32 sum's last place per MFMA) plus the result's rounding."""
    from lux3d_fused import ops
    dev = torch.device("cuda:0")
    print(f"\n[case] q8 ring tile {tile} m={m} n={n} k={k} -> {ydt}", flush=True)
    g = torch.Generator(device="cpu").manual_seed(m + n + k)
    qs = torch.randint(-128, 128, (n, k), generator=g, dtype=torch.int32).to(torch.int8).to(dev)
    scales = (torch.rand((n, k // 32), generator=g) * 0.01 + 1e-4).to(torch.float16).float().to(dev)
    x = torch.randn((m, k + 64), generator=g).to(dev).to(torch.bfloat16)[:, :k]   # row-strided x
    bias = torch.randn(n, generator=g).to(dev) if n % 2 == 0 else None
    y = ops.q8_0_linear(x, qs, scales, bias, TDT[ydt])
    w = (qs.double().reshape(n, -1, 32) * scales.double()[:, :, None]).reshape(n, k).to(torch.bfloat16).double()
    want = x.double() @ w.t().contiguous()
    mag = x.double().abs() @ w.abs().t().contiguous()
    if bias is not None:
        want = want + bias.double()
    u = {"bf16": 2.0 ** -8, "f16": 2.0 ** -11, "f32": 2.0 ** -23}[ydt]
    bound = (k / 32 + 40) * 2.0 ** -23 * mag + u * want.abs() + (2.0 ** -24 if ydt == "f16" else 0.0)
    err = (y.double() - want).abs()
    assert bool((err <= bound).all()), float((err / bound).max())
