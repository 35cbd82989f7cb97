"""The framework's main path as measured cases: the operators of one transformer
or sparse-convolution layer of the VGGT, DINOv3, TripoSG and TRELLIS.2 models,
each through the entry point that a program calls (`lux3d_fused.ops`).

A case is a dict of plain values; "kind" names the operator:
  norm           residual (+ LayerScale) + LayerNorm
  pre_block      that and q/k LayerNorm + 2D RoPE, VGGT's attention pre-block
  gate_modulate  gated residual + AdaLN modulate over ragged segments
  qk_rope3d      q/k L2 norm + 3D RoPE from voxel coordinates
  attention      softmax attention of one model's layer ("model")
  q8_linear      Q8_0 linear, bf16 or f32 activations
  q8_int8        Q8_0 linear with candle's CPU arithmetic
  sparse_conv    submanifold 3x3x3 convolution on f32 voxel features
`draw` gives further cases of the same kinds over the sizes that these models
run at: short and long sequences, odd and ragged sizes, both dtypes.
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "candle-3d_amd"))
from lux3d_fused import ops  # noqa: E402

DTYPES = {"bf16": torch.bfloat16, "f32": torch.float32}
BYTES = {"bf16": 2, "f32": 4}


def listed():
    return [
        # DINOv3 ViT-L/16 at 512 x 512: one residual + LayerNorm of the image
        # encoder in f32, the smallest call a program makes
        {"name": "norm_dinov3", "kind": "norm", "rows": 1029, "width": 1024, "dtype": "f32"},
        # VGGT frame attention on 8 frames: the block's pre-attention part
        {"name": "pre_block_vggt", "kind": "pre_block", "frames": 8, "grid": 37, "dtype": "bf16"},
        # TRELLIS.2 SLAT block on a ragged batch of 24k and 40k voxels: between attention and MLP
        {"name": "gate_modulate_slat", "kind": "gate_modulate", "seg0": 24000, "seg1": 40000, "width": 1536},
        # the same batch's q / k preparation
        {"name": "qk_rope3d_slat", "kind": "qk_rope3d", "tokens": 64000},
        # VGGT frame attention, 8 frames of 1374 tokens, 16 heads x 64
        {"name": "attention_vggt", "kind": "attention", "model": "vggt", "batch": 8, "tokens": 1374, "dtype": "bf16"},
        # TRELLIS.2 SLAT self-attention over the 40k-voxel batch element, 12 heads x 128: the longest sequence
        {"name": "attention_slat", "kind": "attention", "model": "slat", "batch": 1, "tokens": 40000, "dtype": "bf16"},
        # DINOv3 self-attention in f32 (the encoder's precision), 16 heads x 64, rotation of q in the call
        {"name": "attention_dinov3", "kind": "attention", "model": "dinov3", "batch": 1, "tokens": 1029, "dtype": "f32"},
        # TripoSG feed-forward up-projection with quantized weights, both halves of the guidance pair
        {"name": "q8_linear_triposg", "kind": "q8_linear", "m": 4096, "k": 2048, "n": 8192, "dtype": "bf16"},
        # TRELLIS.2 AdaLN linear: one modulation vector per batch element, the shortest product of a step
        {"name": "q8_linear_adaln", "kind": "q8_linear", "m": 2, "k": 1536, "n": 9216, "dtype": "bf16"},
        # DINOv3 MLP up-projection with the reference's CPU arithmetic
        {"name": "q8_int8_dinov3", "kind": "q8_int8", "m": 1029, "k": 1024, "n": 4096},
        # TRELLIS.2 decoder, stage of 256 channels at resolution 256: a convolution that reuses its stage's rulebook
        {"name": "sparse_conv_stage2", "kind": "sparse_conv", "route": "rulebook", "voxels": 150000, "channels": 256,
         "res": 256, "set": "scatter", "order": "shuffled"},
        # its first stage, 1024 channels at the SLAT resolution, straight from the coordinates
        {"name": "sparse_conv_stage0", "kind": "sparse_conv", "route": "coords", "voxels": 24000, "channels": 1024,
         "res": 64, "set": "surface", "order": "scan"},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["norm", "pre_block", "gate_modulate", "qk_rope3d", "attention", "attention", "q8_linear",
                       "q8_linear", "q8_int8", "sparse_conv", "sparse_conv"])
    if kind == "norm":
        return {"kind": kind, "rows": _log(rng, 257, 11000), "width": rng.choice([1024, 1536, 2048]),
                "dtype": rng.choice(["f32", "bf16"])}
    if kind == "pre_block":
        return {"kind": kind, "frames": rng.randint(1, 12), "grid": rng.randint(16, 37),
                "dtype": rng.choice(["bf16", "f32"])}
    if kind == "gate_modulate":
        return {"kind": kind, "seg0": _log(rng, 1500, 24000), "seg1": _log(rng, 1500, 40000),
                "width": rng.choice([1536, 1536, 2048])}
    if kind == "qk_rope3d":
        return {"kind": kind, "tokens": _log(rng, 2000, 64000)}
    if kind == "attention":
        model = rng.choice(["vggt", "vggt_global", "slat", "triposg", "dinov3"])
        if model == "vggt":
            return {"kind": kind, "model": model, "batch": rng.randint(1, 10), "tokens": 5 + rng.randint(16, 37) ** 2,
                    "dtype": rng.choice(["bf16", "f32"])}
        if model == "vggt_global":  # all frames' tokens as one sequence
            return {"kind": kind, "model": model, "batch": 1,
                    "tokens": rng.randint(2, 8) * (5 + rng.randint(16, 37) ** 2), "dtype": "bf16"}
        if model == "slat":
            return {"kind": kind, "model": model, "batch": 1, "tokens": _log(rng, 2000, 32000), "dtype": "bf16"}
        if model == "triposg":
            return {"kind": kind, "model": model, "batch": rng.choice([1, 2, 2]), "tokens": _log(rng, 512, 4096),
                    "dtype": "bf16"}
        return {"kind": kind, "model": model, "batch": rng.choice([1, 1, 2]), "tokens": 5 + rng.randint(14, 36) ** 2,
                "dtype": rng.choice(["f32", "f32", "bf16"])}
    if kind in ("q8_linear", "q8_int8"):
        k, n = rng.choice([(1024, 4096), (4096, 1024), (1024, 3072), (2048, 8192), (8192, 2048), (1536, 9216),
                           (1536, 1536)])
        m = rng.randint(1, 8) if kind == "q8_linear" and rng.random() < 0.25 else _log(rng, 64, 4400)
        case = {"kind": kind, "m": m, "k": k, "n": n}
        if kind == "q8_linear":
            case["dtype"] = rng.choice(["bf16", "bf16", "f32"])
        return case
    channels = rng.choice([1024, 512, 256, 128, 64])
    voxels = _log(rng, 2000, min(150000, 24000 * (1024 // channels)))
    shape = rng.choice(["scatter", "surface"])
    # `scatter` fills 25-75% of a shell of about 8 res^2 cells, `surface` is a closed surface 1-3 voxels thick
    res = int(math.sqrt(voxels / (8 * rng.uniform(0.25, 0.75)))) if shape == "scatter" else \
        int(math.sqrt(voxels / (2 * rng.uniform(1.0, 3.0))))
    return {"kind": kind, "route": rng.choice(["rulebook", "coords"]), "voxels": voxels, "channels": channels,
            "res": max(res, 24) + 6, "set": shape, "order": rng.choice(["scan", "scan", "shuffled"])}


# ---- inputs -------------------------------------------------------------------

class _Inputs:
    """Seeded tensors on the GPU, drawn in a fixed order."""

    def __init__(self, seed):
        self.dev = torch.device("cuda")
        self.g = torch.Generator(device=self.dev).manual_seed(int(seed) * 7919 + 17)
        self.rng = np.random.default_rng(int(seed) + 101)

    def normal(self, shape, dtype=torch.float32, mean=0.0, std=1.0):
        t = torch.randn(shape, generator=self.g, device=self.dev, dtype=torch.float32)
        return t.mul_(std).add_(mean).to(dtype)

    def q8_blocks(self, n, k):
        """GGML Q8_0 blocks of an [n, k] weight of standard deviation about 1/sqrt(k)."""
        nb = n * k // 32
        q = torch.randint(-127, 128, (nb, 32), generator=self.g, device=self.dev, dtype=torch.int32).to(torch.int8)
        d = torch.rand((nb, 1), generator=self.g, device=self.dev) * 0.02 + 0.004
        d = (d / math.sqrt(k)).to(torch.float16)
        return torch.cat([d.view(torch.uint8), q.view(torch.uint8)], dim=1).reshape(-1)


def _positions(frames, grid, dev):
    """VGGT token positions: five special tokens at (0, 0), then (y + 1, x + 1) of the patch grid."""
    pos = torch.zeros((frames, 5 + grid * grid, 2), dtype=torch.int32)
    yy, xx = torch.meshgrid(torch.arange(grid), torch.arange(grid), indexing="ij")
    pos[:, 5:, 0] = (yy.reshape(-1) + 1).to(torch.int32)
    pos[:, 5:, 1] = (xx.reshape(-1) + 1).to(torch.int32)
    return pos.to(dev)


def _voxels(case, rng):
    """int32 [n, 3] distinct voxels around a sphere of a res^3 grid, in scan (x, y, z) or shuffled order."""
    n, res = case["voxels"], case["res"]
    c = res / 2 + rng.uniform(-0.5, 0.5, 3)
    rad = res * 0.4
    if case["set"] == "scatter":  # a random part of a thick shell
        keys = np.zeros(0, np.int64)
        while keys.size < n:
            p = rng.standard_normal((n * 2, 3))
            p = p / np.linalg.norm(p, axis=1, keepdims=True) * (rad + rng.uniform(-2.0, 2.0, (n * 2, 1))) + c
            p = np.clip(np.floor(p), 0, res - 1).astype(np.int64)
            keys = np.unique(np.concatenate([keys, (p[:, 0] * res + p[:, 1]) * res + p[:, 2]]))
        keys = rng.permutation(keys)[:n]
    else:  # the n cells nearest to a slightly bumpy sphere
        a = np.arange(res) + 0.5
        x, y, z = (a[:, None, None] - c[0]), (a[None, :, None] - c[1]), (a[None, None, :] - c[2])
        r = np.sqrt((x * x + y * y + z * z).astype(np.float32))
        bump = 0.04 * np.sin(x * (9.0 / res)) * np.cos(y * (11.0 / res))
        off = np.abs(r * (1.0 + bump.astype(np.float32)) - np.float32(rad)).reshape(-1)
        keys = np.argpartition(off, n)[:n].astype(np.int64)
    keys = np.sort(keys)
    if case["order"] == "shuffled":
        keys = rng.permutation(keys)
    return np.stack([keys // (res * res), keys // res % res, keys % res], axis=1).astype(np.int32)


def _heads_views(qkv):
    """q, k, v as [B, H, L, D] views of a fused [B, L, 3, H, D] projection."""
    v = qkv.permute(2, 0, 3, 1, 4)
    return v[0], v[1], v[2]


HEADS = {"vggt": (16, 64), "vggt_global": (16, 64), "slat": (12, 128), "triposg": (16, 128), "dinov3": (16, 64)}


def prepare(case, seed):
    i = _Inputs(seed)
    kind = case["kind"]
    s = {"case": case}
    dt = DTYPES[case.get("dtype", "bf16")]
    if kind == "norm":
        shape = (1, case["rows"], case["width"])
        c = case["width"]
        s.update(x=i.normal(shape, dt), a=i.normal(shape, dt), gamma=i.normal(c, mean=0.2, std=0.02),
                 w=i.normal(c, mean=1.0, std=0.02), b=i.normal(c, std=0.02))
    elif kind == "pre_block":
        b, n, h, d = case["frames"], 5 + case["grid"] ** 2, 16, 64
        s.update(x=i.normal((b, n, 1024), dt), a=i.normal((b, n, 1024), dt), gamma=i.normal(1024, mean=1.0, std=0.02),
                 w=i.normal(1024, mean=1.0, std=0.02), b=i.normal(1024, std=0.02),
                 qkv=i.normal((b, n, 3, h, d), dt),
                 q_norm=(i.normal(d, mean=1.0, std=0.02), i.normal(d, std=0.02), 1e-5),
                 k_norm=(i.normal(d, mean=1.0, std=0.02), i.normal(d, std=0.02), 1e-5),
                 pos=_positions(b, case["grid"], i.dev))
    elif kind == "gate_modulate":
        rows, c = case["seg0"] + case["seg1"], case["width"]
        s.update(x=i.normal((rows, c), torch.bfloat16), h=i.normal((rows, c), torch.bfloat16),
                 t_emb=i.normal((2, 6 * c), std=0.1), modulation=i.normal((6 * c,), std=0.1),
                 offs=torch.tensor([0, case["seg0"], rows], dtype=torch.int64, device=i.dev))
    elif kind == "qk_rope3d":
        n = case["tokens"]
        s.update(qkv=i.normal((1, n, 3, 12, 128), torch.bfloat16), gq=i.normal((12, 128), mean=1.0, std=0.02),
                 gk=i.normal((12, 128), mean=1.0, std=0.02),
                 coords=torch.randint(0, 64, (n, 3), generator=i.g, device=i.dev, dtype=torch.int32))
    elif kind == "attention":
        b, n = case["batch"], case["tokens"]
        h, d = HEADS[case["model"]]
        if case["model"] == "triposg":  # q, k, v as the per-head thirds of [B, L, H, 3 D]
            s.update(qkv=i.normal((b, n, h, 3 * d), dt), qw=i.normal(d, mean=1.0, std=0.1),
                     kw=i.normal(d, mean=1.0, std=0.1))
        elif case["model"] == "dinov3":
            ang = i.normal((n - 5, d // 2), std=2.0)
            s.update(q=i.normal((b, n, h, d), dt), k=i.normal((b, n, h, d), dt), v=i.normal((b, n, h, d), dt),
                     cos=torch.cos(torch.cat([ang, ang], 1)), sin=torch.sin(torch.cat([ang, ang], 1)))
        else:
            s["qkv"] = i.normal((b, n, 3, h, d), dt)
    elif kind in ("q8_linear", "q8_int8"):
        m, k, n = case["m"], case["k"], case["n"]
        x = i.normal((m, k), dt if kind == "q8_linear" else torch.float32)
        qs, scales = ops.q8_0_repack(i.q8_blocks(n, k), n, k)
        s.update(x=x, qs=qs, scales=scales, bias=i.normal(n, std=0.5))
    else:
        c = case["channels"]
        coords = torch.from_numpy(_voxels(case, i.rng)).to(i.dev)
        n = coords.shape[0]
        s.update(coords=coords, x=i.normal((n, c)),
                 conv=ops.SparseConv3d(i.normal((c, 3, 3, 3, c), std=1.0 / math.sqrt(27 * c)), i.normal(c), c, c))
        if case["route"] == "rulebook":
            s["on"] = ops.SparseRulebook(ops.sparse_neighbors(coords))
        else:
            s["on"] = coords
    return s


def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "norm":
        return ops.residual_layer_norm(s["x"], s["a"], s["gamma"], s["w"], s["b"], 1e-5)
    if kind == "pre_block":
        h, y = ops.residual_layer_norm(s["x"], s["a"], s["gamma"], s["w"], s["b"], 1e-5)
        q, k, _ = _heads_views(s["qkv"])
        q, k = ops.qk_layernorm_rope2d(q, k, s["q_norm"], s["k_norm"], positions=s["pos"], base=100.0)
        return h, y, q, k
    if kind == "gate_modulate":
        p, base = ops.chunk_modulation(s["t_emb"]), s["modulation"].chunk(6)
        return ops.gated_residual_adaln_modulate(s["x"], s["h"], p[2], p[3], p[4], gate_base=base[2],
                                                 shift_base=base[3], scale_base=base[4], seg_offsets=s["offs"])
    if kind == "qk_rope3d":
        return ops.qk_l2norm_rope3d(s["qkv"][:, :, 0], s["qkv"][:, :, 1], s["gq"], s["gk"], coords=s["coords"])
    if kind == "attention":
        h, d = HEADS[case["model"]]
        scale = 1.0 / math.sqrt(d)
        if case["model"] == "triposg":
            q, k, v = (s["qkv"][..., j * d:(j + 1) * d].transpose(1, 2) for j in range(3))
            k = ops.rms_norm_heads(k, s["kw"])
            return ops.sdpa_rms_norm_heads(q, s["qw"], 1e-6, k, v, scale)
        if case["model"] == "dinov3":
            q, k, v = (s[j].transpose(1, 2) for j in "qkv")
            return ops.sdpa_dinov3_rope(q, s["cos"], s["sin"], 5, k, v, scale)
        return ops.sdpa(*_heads_views(s["qkv"]), scale)
    if kind == "q8_linear":
        return ops.q8_0_linear(s["x"], s["qs"], s["scales"], s["bias"], out_dtype=DTYPES[case["dtype"]])
    if kind == "q8_int8":
        return ops.q8_0_linear_int8(s["x"], s["qs"], s["scales"], s["bias"])
    return s["conv"].forward(s["on"], s["x"])


# ---- what a pass cannot do without --------------------------------------------

def _taps(coords):
    """(row, neighbour row, tap) counts of a voxel set: present neighbours over all 27 offsets."""
    c = coords.astype(np.int64) + 1
    side = int(c.max()) + 2
    key = np.sort((c[:, 0] * side + c[:, 1]) * side + c[:, 2])
    pairs = key.size
    for t in range(14, 27):  # the other 13 offsets mirror these
        off = ((t // 9 - 1) * side + (t % 9 // 3 - 1)) * side + (t % 3 - 1)
        at = np.searchsorted(key, key + off)
        pairs += 2 * int(np.count_nonzero(key[np.minimum(at, key.size - 1)] == key + off))
    return pairs


def work(case):
    kind = case["kind"]
    e = BYTES[case.get("dtype", "bf16")]
    if kind == "norm":
        return {"bytes": 4 * case["rows"] * case["width"] * e + 12 * case["width"], "flops": 0}
    if kind == "pre_block":
        rows = case["frames"] * (5 + case["grid"] ** 2)
        return {"bytes": 8 * rows * 1024 * e + rows * 8 + 3 * 4096 + 4 * 256, "flops": 0}
    if kind == "gate_modulate":
        return {"bytes": 4 * (case["seg0"] + case["seg1"]) * case["width"] * 2 + 9 * case["width"] * 4 + 24, "flops": 0}
    if kind == "qk_rope3d":
        return {"bytes": case["tokens"] * (4 * 12 * 128 * 2 + 12) + 2 * 12 * 128 * 4, "flops": 0}
    if kind == "attention":
        h, d = HEADS[case["model"]]
        b, n = case["batch"], case["tokens"]
        tables = 2 * (n - 5) * d * 4 if case["model"] == "dinov3" else 0
        return {"bytes": 4 * b * n * h * d * e + tables, "flops": 4 * b * h * n * n * d}
    if kind in ("q8_linear", "q8_int8"):
        m, k, n = case["m"], case["k"], case["n"]
        e = e if kind == "q8_linear" else 4
        return {"bytes": m * k * e + n * k + n * k // 32 * 4 + n * 4 + m * n * e, "flops": 2 * m * k * n}
    n, c = case["voxels"], case["channels"]
    pairs = _taps(_voxels(case, np.random.default_rng(1)))
    table = 12 * n if case["route"] == "coords" else 8 * pairs
    return {"bytes": 2 * n * c * 4 + 27 * c * c * 4 + c * 4 + table, "flops": 2 * pairs * c * c}


def tolerance(case):
    kind = case["kind"]
    f32 = case.get("dtype", "bf16") == "f32"
    if kind in ("norm", "pre_block"):
        # f32: sums of up to 2048 values in another order, an angle's sine; bf16: one rounding of the result
        return {"rel": 2e-6, "max": 2e-5} if f32 else {"rel": 4e-3, "max": 0.03}
    if kind in ("gate_modulate", "qk_rope3d"):
        return {"rel": 4e-3, "max": 0.03}
    if kind == "attention":
        # bf16: probabilities and result rounded once; f32: sums in another order
        return {"rel": 4e-6, "max": 5e-5} if f32 else {"rel": 0.01, "max": 0.06}
    if kind == "q8_linear":
        return {"rel": 2e-6, "max": 2e-5} if f32 else {"rel": 5e-3, "max": 0.03}
    if kind == "q8_int8":
        # integer block products and an f32 sum over the blocks: 1e-7; an x that a division's last bit puts on the
        # other side of a rounding step: 1e-5
        return {"rel": 5e-5, "max": 2e-3}
    return {"rel": 4e-6, "max": 4e-5}      # f32 products, sums of up to 27 x 1024 in another order


# ---- the same in 64 bits ---------------------------------------------------------

def _ln(x, eps):
    mean = x.mean(-1, keepdim=True)
    x = x - mean
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps)


def _rope2d(x, pos, base):
    """VGGT's 2D rotation of [B, H, N, D] heads: the halves by y and x, rotate_half inside each."""
    half = x.shape[-1] // 2
    out = []
    for axis in range(2):
        v = x[..., axis * half:(axis + 1) * half]
        inv = 1.0 / base ** (torch.arange(0, half, 2, device=x.device, dtype=torch.float64) / half)
        ang = pos[..., axis].double()[:, None, :, None] * inv
        ang = torch.cat([ang, ang], -1)
        turned = torch.cat([-v[..., half // 2:], v[..., :half // 2]], -1)
        out.append(v * torch.cos(ang) + turned * torch.sin(ang))
    return torch.cat(out, -1)


def _softmax_attention(q, k, v, scale):
    """f64 attention of [B, H, L, D], in blocks of queries."""
    out = torch.empty_like(q)
    step = max(1, (1 << 28) // max(1, k.shape[2]) // 8)
    for b in range(q.shape[0]):
        for h in range(q.shape[1]):
            kt, vv = k[b, h].t().contiguous(), v[b, h].contiguous()
            for a in range(0, q.shape[2], step):
                out[b, h, a:a + step] = torch.softmax(q[b, h, a:a + step] @ kt * scale, -1) @ vv
    return out


def _exact_attention(case, s):
    h, d = HEADS[case["model"]]
    scale = 1.0 / math.sqrt(d)
    if case["model"] == "triposg":
        q, k, v = (s["qkv"][..., j * d:(j + 1) * d].transpose(1, 2).double() for j in range(3))

        def rms(t, w):
            return t / torch.sqrt((t * t).mean(-1, keepdim=True) + 1e-6) * w.double()
        # the operators store the normalised q and k in bf16
        q, k = (rms(t, w).to(torch.bfloat16).double() for t, w in ((q, s["qw"]), (k, s["kw"])))
    elif case["model"] == "dinov3":
        q, k, v = (s[j].transpose(1, 2).double() for j in "qkv")
        t = q[:, :, 5:]
        turned = torch.cat([-t[..., d // 2:], t[..., :d // 2]], -1)
        q = torch.cat([q[:, :, :5], t * s["cos"].double() + turned * s["sin"].double()], 2)
        if case["dtype"] == "bf16":  # the rotated q is stored in bf16
            q = q.to(torch.bfloat16).double()
    else:
        q, k, v = (t.double() for t in _heads_views(s["qkv"]))
    return _softmax_attention(q, k, v, scale)


def _exact_conv(s):
    coords, x = s["coords"].long() + 1, s["x"].double()
    w = s["conv"].weight27.double()
    side = int(coords.max().item()) + 2
    key = (coords[:, 0] * side + coords[:, 1]) * side + coords[:, 2]
    order = torch.argsort(key)
    ranked = key[order]
    out = s["conv"].bias.double().expand(x.shape[0], -1).clone()
    for t in range(27):
        off = ((t // 9 - 1) * side + (t % 9 // 3 - 1)) * side + (t % 3 - 1)
        at = torch.searchsorted(ranked, key + off).clamp_(max=key.numel() - 1)
        dst = torch.nonzero(ranked[at] == key + off).reshape(-1)
        out[dst] += x[order[at[dst]]] @ w[t].t().contiguous()
    return out


def exact(case, seed):
    s = prepare(case, seed)
    kind = case["kind"]
    if kind in ("norm", "pre_block"):
        dt = s["x"].dtype
        h = s["x"].double() + s["a"].double() * s["gamma"].double()
        # the residual stream is stored in its dtype and the norm reads what was stored
        y = _ln(h.to(dt).double(), 1e-5) * s["w"].double() + s["b"].double()
        if kind == "norm":
            return h, y
        q, k, _ = _heads_views(s["qkv"])
        q, k = (_rope2d(_ln(t.double(), eps) * w.double() + b.double(), s["pos"], 100.0)
                for t, (w, b, eps) in ((q, s["q_norm"]), (k, s["k_norm"])))
        return h, y, q, k
    if kind == "gate_modulate":
        rows = s["x"].shape[0]
        seg = (torch.arange(rows, device=s["x"].device) >= case["seg0"]).long()
        mod = (s["t_emb"].double() + s["modulation"].double()).chunk(6, -1)
        x = s["x"].double() + s["h"].double() * mod[2][seg]
        y = _ln(x.to(torch.bfloat16).double(), 1e-6) * (1.0 + mod[4][seg]) + mod[3][seg]
        return x, y
    if kind == "qk_rope3d":
        n, fd = case["tokens"], 128 // 2 // 3
        f = 1.0 / 10000.0 ** (torch.arange(fd, device=s["qkv"].device, dtype=torch.float64) / fd)
        ang = torch.zeros((n, 64), device=s["qkv"].device, dtype=torch.float64)
        ang[:, :3 * fd] = (s["coords"].double()[:, :, None] * f).reshape(n, 3 * fd)
        cos, sin = torch.cos(ang)[None, :, None], torch.sin(ang)[None, :, None]
        out = []
        for j, g in ((0, s["gq"]), (1, s["gk"])):
            v = s["qkv"][:, :, j].double()
            v = v / v.norm(dim=-1, keepdim=True).clamp(1e-12, 1e30) * g.double() * math.sqrt(128.0)
            re, im = v[..., 0::2], v[..., 1::2]
            out.append(torch.stack([re * cos - im * sin, re * sin + im * cos], -1).flatten(-2))
        return tuple(out)
    if kind == "attention":
        return _exact_attention(case, s)
    if kind == "q8_linear":
        w = s["qs"].double().reshape(case["n"], -1, 32) * s["scales"].double()[:, :, None]
        w = w.reshape(case["n"], -1)
        if case["dtype"] == "bf16":  # the weight dequantizes to the activations' type
            w = w.to(torch.bfloat16).double()
        return s["x"].double() @ w.t().contiguous() + s["bias"].double()
    if kind == "q8_int8":
        xb = s["x"].reshape(case["m"], -1, 32)
        d = xb.abs().amax(-1, keepdim=True) / 127.0
        v = xb * (1.0 / d)  # f32, as the reference quantizes
        q = torch.where(v < 0, torch.ceil(v - 0.5), torch.floor(v + 0.5)).clamp(-128, 127)
        x = (q.double() * d.to(torch.float16).double()).reshape(case["m"], -1)
        w = (s["qs"].double().reshape(case["n"], -1, 32) * s["scales"].double()[:, :, None]).reshape(case["n"], -1)
        return x @ w.t().contiguous() + s["bias"].double()
    return _exact_conv(s)
