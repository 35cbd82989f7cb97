"""The pipelined attention kernel (D 64 / 128, bf16 / f16) at the edges of its
key steps and stages, query tiles and dispatch rules, against the oracle."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu
TDT = {"bf16": torch.bfloat16, "f16": torch.float16}


@pytest.fixture(scope="module")
def dev():
    if not torch.cuda.is_available():
        pytest.skip("no ROCm device")
    return torch.device("cuda:0")


def _check(got, q, k, v, scale, dt):
    """|error| <= 4 u max|v| + u |want| with u the type's unit roundoff: a probability's rounding changes a weight by
    at most u of itself on both sides of the quotient, exponentials and f32 sums stay below another u, and the output
    is rounded once."""
    q, k, v = (t.double() for t in (q, k, v))
    s = q @ k.transpose(-1, -2).contiguous() * scale
    want = torch.softmax(s, -1) @ v
    u = 2.0 ** -8 if dt == "bf16" else 2.0 ** -11
    err = (got.double() - want).abs()
    bound = 4 * u * v.abs().amax() + u * want.abs()
    assert bool((err <= bound).all()), float((err / bound).max())


# (b, h, lq, lk): 1-9 key blocks of 32 and their remainders (D 64 is pipelined from 65 keys on but for 128 and 192), 256
# keys (the shortest D 128 takes), one row, query tiles of 128 / 256 and one more, and grids on both sides of each rule
# of the dispatch
SHAPES = [(1, 3, 130, 1), (2, 80, 130, 31), (2, 80, 130, 33), (2, 80, 129, 64), (2, 80, 128, 95), (2, 80, 127, 96),
          (2, 80, 1, 128), (2, 80, 130, 129), (2, 80, 130, 160), (2, 80, 130, 65), (2, 80, 130, 192), (2, 80, 130, 193), (2, 80, 130, 191), (2, 80, 130, 224), (2, 80, 130, 255),
          (2, 80, 130, 256), (2, 80, 257, 257), (2, 80, 130, 289), (1, 16, 1024, 300), (1, 16, 1029, 300),
          (4, 16, 2048, 70), (1, 48, 300, 64), (1, 100, 300, 130), (1, 64, 420, 130)]


@pytest.mark.parametrize("dt", ["bf16", "f16"])
@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("b,h,lq,lk", SHAPES)
def test_sdpa_pipelined(dev, b, h, lq, lk, d, dt):
    from lux3d_fused import ops
    print(f"\n[case] sdpa pipelined [{b},{h},{lq},{lk},{d}] {dt}", flush=True)
    g = torch.Generator(device="cpu").manual_seed(lq * 7 + lk + d)
    make = lambda n: torch.randn((b, n, h, d), generator=g).to(dev).to(TDT[dt]).transpose(1, 2)  # noqa: E731
    q, k, v = make(lq), make(lk), make(lk)
    k = k * 3    # maxima that move by more than the 2^8 that the running reference allows
    scale = d ** -0.5
    out = torch.full((b, h, lq, d), float("nan"), dtype=TDT[dt], device=dev)
    ops.sdpa(q, k, v, scale, out=out)
    _check(out, q, k, v, scale, dt)


@pytest.mark.parametrize("d", [64, 128])
def test_sdpa_pipelined_rising_scores(dev, d):
    """Scores that rise along the keys, so that every block moves the reference maximum and rescales the sums, and a
    last key that outweighs all others."""
    from lux3d_fused import ops
    print(f"\n[case] sdpa pipelined rising scores d={d}", flush=True)
    b, h, lq, lk = 2, 40, 140, 333
    g = torch.Generator(device="cpu").manual_seed(d)
    q = torch.ones((b, h, lq, d)).to(dev).to(torch.bfloat16)
    k = (torch.arange(lk).float()[None, None, :, None] * 0.25 / d * torch.ones((b, h, lk, d))).to(dev).to(torch.bfloat16)
    k[:, :, -1] = 120.0 / d
    v = torch.randn((b, h, lk, d), generator=g).to(dev).to(torch.bfloat16)
    _check(ops.sdpa(q, k, v, 1.0), q, k, v, 1.0, "bf16")


# one to a few workgroups, which pipeline from 224 keys on, and more than 256, from 400 on
@pytest.mark.parametrize("h,lq,lk", [(3, lk, lk) for lk in (192, 193, 223, 224, 225, 256, 287, 300, 320, 351)]
                         + [(160, 130, lk) for lk in (399, 400, 416, 447)])
@pytest.mark.parametrize("rotate", [False, True])
def test_sdpa_f32_pipelined(dev, h, lq, lk, rotate):
    """The pipelined f32 kernel (D 64) over odd and even numbers of 32-key blocks and their remainders, against 64
    bits: |error| <= (d + lk) 2^-22 max|v|, an f32 sum's last place per product in scores and output, and 1.2e-6 of the
    result's 2-norm: f32 arithmetic stays near 5e-7 over these sizes, while q, k, p or v without their third term, or
    a product without that of the second terms, give 2.0e-6 and more."""
    from lux3d_fused import ops
    print(f"\n[case] sdpa f32 pipelined h={h} lq={lq} lk={lk} rotate={rotate}", flush=True)
    b, d = 1, 64
    g = torch.Generator(device="cpu").manual_seed(lk)
    q, k, v = (torch.randn((b, n, h, d), generator=g).to(dev).transpose(1, 2) for n in (lq, lk, lk))
    out = torch.full((b, h, lq, d), float("nan"), device=dev)
    qd = q.double()
    if rotate:
        ang = torch.randn((lq - 5, d), generator=g).to(dev)
        cos, sin = torch.cos(ang), torch.sin(ang)
        ops.sdpa_dinov3_rope(q, cos, sin, 5, k, v, 0.125, out=out)
        t = qd[:, :, 5:]
        turned = torch.cat([-t[..., d // 2:], t[..., :d // 2]], -1)
        qd = torch.cat([qd[:, :, :5], t * cos.double() + turned * sin.double()], 2)
    else:
        ops.sdpa(q, k, v, 0.125, out=out)
    want = torch.softmax(qd @ k.double().transpose(-1, -2).contiguous() * 0.125, -1) @ v.double()
    err = out.double() - want
    assert float(err.abs().max()) <= (d + lk) * 2.0 ** -22 * float(v.abs().max())
    assert float(err.norm()) <= 1.2e-6 * float(want.norm())


def test_sdpa_f32_pipelined_reversed_keys(dev):
    """A negative token stride addresses the same keys backwards: the same softmax up to the order of the sums."""
    from lux3d_fused import _lib, ops
    print("\n[case] sdpa f32 pipelined reversed keys", flush=True)
    b, h, lk, d = 1, 2, 333, 64
    g = torch.Generator(device="cpu").manual_seed(3)
    q, k, v = (torch.randn((b, h, lk, d), generator=g).to(dev) for _ in range(3))

    def backwards(t):
        return _lib.descriptor(t.data_ptr() + (lk - 1) * d * 4, _lib.F32, list(t.shape), [h * lk * d, lk * d, -d, 1])

    import ctypes
    out = torch.empty_like(q)
    _lib.call("lux3d_sdpa", ops.desc(q), ctypes.pointer(backwards(k)), ctypes.pointer(backwards(v)), 0.125,
              ops.desc(out), torch.cuda.current_stream().cuda_stream)
    want = ops.sdpa(q, k.flip(2).contiguous(), v.flip(2).contiguous(), 0.125)
    assert torch.equal(out, want)


def _backwards(t):
    """Descriptor of [B, H, L, D] `t` with its tokens in reverse order: a negative stride, which the direct loads of
    the pipelined kernel do not address, so that the register-staged kernel takes the call."""
    from lux3d_fused import _lib
    st = list(t.stride())
    code = {torch.bfloat16: _lib.BF16, torch.float16: _lib.F16}[t.dtype]
    return _lib.descriptor(t.data_ptr() + (t.shape[2] - 1) * st[2] * t.element_size(), code, list(t.shape),
                           [st[0], st[1], -st[2], st[3]])


# grids on both sides of the 128- / 256-query rule and beyond the key groups of either kernel; D 128 from the 256 keys
# where the pipelined kernel starts, D 64 from one key (pipelined from 65, but for 128 and 192); 1-6 pairs of 32-key blocks, whole, cut and with an odd block
STAGED = [(400, 128, lk, 64, "") for lk in (1, 32, 33, 64, 65, 96, 97, 127, 130, 160, 192, 193, 224, 256, 320, 333)] \
    + [(512, 256, lk, 64, "") for lk in (1, 33, 64, 95, 129, 192, 256, 300)] \
    + [(2, 130, lk, 128, "") for lk in (256, 257, 288, 289, 320, 383, 20000)] \
    + [(h, lq, lk, d, pro) for h, lq, lk, d in ((400, 128, 130, 64), (512, 256, 95, 64), (2, 130, 289, 128))
       for pro in ("_layernorm_rope2d", "_rms_norm_heads", "_l2norm_rope3d")]


@pytest.mark.parametrize("dt", ["bf16", "f16"])
@pytest.mark.parametrize("h,lq,lk,d,pro", STAGED)
def test_sdpa_pipelined_has_the_bits_of_the_register_staged_kernel(dev, h, lq, lk, d, pro, dt):
    """The pipelined kernel does the arithmetic of the register-staged one in its order (a reference maximum and a row
    sum for each 64 keys), with each of the q prologues: the same keys through either give the same bits. Scores vary
    enough to move the reference maximum."""
    from lux3d_fused import _lib, ops
    print(f"\n[case] pipelined / staged {pro} [{h},{lq},{lk},{d}] {dt}", flush=True)
    g = torch.Generator(device="cpu").manual_seed(lq + lk + d)
    q = (torch.randn((1, h, lq, d), generator=g) * 1.5).to(dev).to(TDT[dt])
    k, v = (torch.randn((1, h, lk, d), generator=g).to(dev).to(TDT[dt]) for _ in range(2))
    k = k * 3
    w, b = (1 + 0.1 * torch.randn(d, generator=g)).to(dev), (0.1 * torch.randn(d, generator=g)).to(dev)
    scale, stream = d ** -0.5, torch.cuda.current_stream().cuda_stream
    if pro == "_l2norm_rope3d":
        ang = torch.randn((lq, d // 2), generator=g).to(dev)
        head = (q, (1 + 0.1 * torch.randn((h, d), generator=g)).to(dev), torch.cos(ang), torch.sin(ang))
    elif pro == "_layernorm_rope2d":
        ang = torch.randn((1, 1, lq, d), generator=g).to(dev)
        head = (q, w, b, 1e-6, torch.cos(ang), torch.sin(ang))
    else:
        head = (q, w, 1e-6) if pro else (q,)

    def run(kd, vd):
        out = torch.full_like(q, float("nan"))
        _lib.call("lux3d_sdpa" + pro, *(ops._d(a) if torch.is_tensor(a) else a for a in head), kd, vd, scale,
                  ops._d(out), stream)
        return out
    kf, vf = k.flip(2).contiguous(), v.flip(2).contiguous()
    pipelined, staged = run(ops._d(kf), ops._d(vf)), run(_backwards(k), _backwards(v))
    assert not bool(torch.isnan(staged).any())
    assert torch.equal(pipelined, staged)


@pytest.mark.parametrize("first", [31, 32, 50, 63])
@pytest.mark.parametrize("h,lq,d", [(400, 128, 64), (512, 256, 64), (2, 130, 128)])
def test_sdpa_pipelined_first_keys_masked_by_infinity(dev, h, lq, d, first):
    """Keys masked by a score of -inf, fewer than the 64 of the first reference maximum, weigh nothing."""
    from lux3d_fused import ops
    print(f"\n[case] sdpa -inf first={first} h={h} lq={lq} d={d}", flush=True)
    g = torch.Generator(device="cpu").manual_seed(first + d)
    lk = 300
    q, k, v = (torch.randn((1, h, n, d), generator=g).to(dev).to(torch.bfloat16) for n in (lq, lk, lk))
    q[..., 0], k[..., 0] = 1, 0
    masked = k.clone()
    masked[:, :, :first, 0] = float("-inf")
    out = ops.sdpa(q, masked, v, d ** -0.5)
    _check(out, q, k[:, :, first:], v[:, :, first:], d ** -0.5, "bf16")


@pytest.mark.parametrize("dt", ["bf16", "f16"])
@pytest.mark.parametrize("h,lq,d", [(400, 128, 64), (512, 256, 64), (2, 130, 128)])
@pytest.mark.parametrize("lk", [257, 289, 300, 320, 350])
def test_sdpa_pipelined_keys_past_lk_are_not_read(dev, h, lq, lk, d, dt):
    """K and V are views into a buffer whose 160 rows past Lk of every head are NaN (the pipeline loads up to 160 rows
    ahead): none reaches the output, with even and odd numbers of blocks and whole and cut last ones."""
    from lux3d_fused import ops
    print(f"\n[case] pipelined nan tail [{h},{lq},{lk},{d}] {dt}", flush=True)
    g = torch.Generator(device="cpu").manual_seed(lk * 3 + d)
    buf = torch.full((2, 1, h, lk + 160, d), float("nan"))
    buf[:, :, :, :lk] = torch.randn((2, 1, h, lk, d), generator=g)
    buf = buf.to(dev).to(TDT[dt])
    k, v = buf[0, :, :, :lk], buf[1, :, :, :lk]
    q = torch.randn((1, h, lq, d), generator=g).to(dev).to(TDT[dt])
    _check(ops.sdpa(q, k, v, d ** -0.5), q, k, v, d ** -0.5, dt)
