"""The f32 Q8_0 linear's tiles (128 x 256, 64 x 128 with one and two k groups, 32 x 128 with three) at their edges and
uneven shares of k, against 64 bits. The sizes are picked so that the dispatch's costs choose the named tile."""
import pytest
import torch

pytestmark = pytest.mark.gpu
TDT = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}


# k of 2, 30, 32 and 34 steps of 32; two groups are taken from 4 steps on
TILES = [(tile, m, n, k) for tile, m, n in (("32x128 / 3", 129, 1500), ("32x128 / 3", 160, 1537), ("64x128", 700, 1500),
                                            ("64x128 / 2", 700, 1500), ("64x128", 1100, 2060),
                                            ("64x128, aligned", 1088, 2176), ("128x256", 1100, 4100))
         for k in ((64,) if (tile, m) == ("64x128", 700) else
                   (128 if tile == "64x128 / 2" else 64, 960, 1024, 1088))] \
    + [("32x128 / 3", 16, 32000, 512), ("32x128 / 3", 7, 30001, 576)]


@pytest.mark.parametrize("ydt", ["f32", "bf16", "f16"])
@pytest.mark.parametrize("tile,m,n,k", TILES)
def test_q8_linear_f32_tiles(tile, m, n, k, ydt):
    """|error| <= (k / 32 + 40) 2^-23 sum |x w| (an f32 sum's last place per MFMA, block and group) plus the result's
    rounding."""
    from lux3d_fused import ops
    dev = torch.device("cuda:0")
    print(f"\n[case] q8 f32 tile {tile} m={m} n={n} k={k} -> {ydt}", flush=True)
    g = torch.Generator(device="cpu").manual_seed(m + n + k)
    qs = torch.randint(-128, 128, (n, k), generator=g, dtype=torch.int32).to(torch.int8).to(dev)
    scales = (torch.rand((n, k // 32), generator=g) * 0.01 + 1e-4).to(torch.float16).float().to(dev)
    x = torch.randn((m, k + 64), generator=g).to(dev)[:, :k]   # row-strided x
    bias = torch.randn(n, generator=g).to(dev) if n % 2 == 0 else None
    y = ops.q8_0_linear(x, qs, scales, bias, TDT[ydt])
    w = (qs.double().reshape(n, -1, 32) * scales.double()[:, :, None]).reshape(n, k)
    want = x.double() @ w.t().contiguous()
    mag = x.double().abs() @ w.abs().t().contiguous()
    if bias is not None:
        want = want + bias.double()
    u = {"bf16": 2.0 ** -8, "f16": 2.0 ** -11, "f32": 2.0 ** -23}[ydt]
    bound = (k / 32 + 40) * 2.0 ** -23 * mag + u * want.abs() + (2.0 ** -24 if ydt == "f16" else 0.0)
    err = (y.double() - want).abs()
    assert bool((err <= bound).all()), float((err / bound).max())


def test_q8_linear_f32_infinite_x_stays_in_its_row():
    """A group that has no step left adds nothing: a row of infinities stays the only row that is not finite."""
    from lux3d_fused import ops
    dev = torch.device("cuda:0")
    m, n, k = 129, 1500, 1088
    g = torch.Generator(device="cpu").manual_seed(5)
    qs = torch.randint(1, 128, (n, k), generator=g, dtype=torch.int32).to(torch.int8).to(dev)
    scales = torch.full((n, k // 32), 0.01, device=dev)
    x = torch.rand((m, k), generator=g).to(dev)
    x[7, 5] = float("inf")
    y = ops.q8_0_linear(x, qs, scales, None, torch.float32)
    assert not bool(torch.isfinite(y[7]).any())
    assert bool(torch.isfinite(y[:7]).all()) and bool(torch.isfinite(y[8:]).all())
