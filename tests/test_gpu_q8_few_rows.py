"""The few-rows Q8_0 linear (wavefronts split k) at the edges of its row and
column tiles, chunk pairs and dispatch rule, against 64 bits."""
import pytest
import torch

pytestmark = pytest.mark.gpu
TDT = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}


def _weights(n, k, seed, dev):
    g = torch.Generator(device="cpu").manual_seed(seed)
    qs = torch.randint(-128, 128, (n, k), generator=g, dtype=torch.int32).to(torch.int8).to(dev)
    scales = (torch.rand((n, k // 32), generator=g) * 0.01 + 1e-4).to(torch.float16).float().to(dev)
    return qs, scales


# k: one chunk, one pair, an odd number of chunks, and what 4, 8 and 16 wavefronts cover in one and more turns
KS = [64, 128, 192, 576, 1088, 2112, 4160]
SIZES = [(1, 1), (2, 15), (15, 16), (16, 33), (17, 17), (63, 40), (64, 16), (65, 50), (130, 31)]


@pytest.mark.parametrize("xdt,ydt", [("bf16", "bf16"), ("bf16", "f32"), ("f32", "f32"), ("f32", "f16")])
@pytest.mark.parametrize("k", KS)
@pytest.mark.parametrize("m,n", SIZES)
def test_q8_linear_few_rows(m, n, k, xdt, ydt):
    """|error| <= (k / 32 + 40) 2^-23 sum |x w| (an f32 sum's last place per MFMA, block and wavefront) plus the
    result's rounding."""
    from lux3d_fused import ops
    dev = torch.device("cuda:0")
    print(f"\n[case] q8 few rows m={m} n={n} k={k} {xdt}->{ydt}", flush=True)
    qs, scales = _weights(n, k, m * 1000 + n + k, dev)
    g = torch.Generator(device="cpu").manual_seed(k + m)
    x = torch.randn((m, 2 * k), generator=g).to(dev).to(TDT[xdt])[:, :k]   # row-strided x
    bias = torch.randn(n, generator=g).to(dev) if n % 2 else None
    y = ops.q8_0_linear(x, qs, scales, bias, TDT[ydt])
    w = (qs.double().reshape(n, -1, 32) * scales.double()[:, :, None]).reshape(n, k)
    if xdt == "bf16":
        w = w.to(torch.bfloat16).double()
    want = x.double() @ w.t().contiguous()
    mag = x.double().abs() @ w.abs().t().contiguous()
    if bias is not None:
        want = want + bias.double()
    u = {"bf16": 2.0 ** -8, "f16": 2.0 ** -11, "f32": 2.0 ** -23}[ydt]
    bound = (k / 32 + 40) * 2.0 ** -23 * mag + u * want.abs() + (2.0 ** -24 if ydt == "f16" else 0.0)
    err = (y.double() - want).abs()
    assert bool((err <= bound).all()), float((err / bound).max())


@pytest.mark.parametrize("xdt", ["bf16", "f32"])
def test_q8_linear_paths_agree(xdt):
    """Rows of one call on the tiles' path (many rows) and of calls on the few-rows path: the same product up to the
    order of the f32 sums."""
    from lux3d_fused import ops
    dev = torch.device("cuda:0")
    n, k = 2064, 1024
    qs, scales = _weights(n, k, 9, dev)
    x = torch.randn((1500, k), generator=torch.Generator(device="cpu").manual_seed(1)).to(dev).to(TDT[xdt])
    whole = ops.q8_0_linear(x, qs, scales, None, torch.float32)
    for m in (1, 16, 17, 200):
        part = ops.q8_0_linear(x[:m], qs, scales, None, torch.float32)
        assert float((part - whole[:m]).norm() / whole[:m].norm()) < 1e-6, m


def test_q8_linear_few_rows_infinite_x_stays_in_its_row():
    from lux3d_fused import ops
    dev = torch.device("cuda:0")
    qs, scales = _weights(40, 640, 4, dev)
    x = torch.randn((5, 640), generator=torch.Generator(device="cpu").manual_seed(2)).to(dev).to(torch.bfloat16)
    want = ops.q8_0_linear(x, qs, scales)
    x[2, 100] = float("inf")
    got = ops.q8_0_linear(x, qs, scales)
    assert not torch.isfinite(got[2]).any()
    keep = [0, 1, 3, 4]
    assert torch.equal(got[keep], want[keep])
