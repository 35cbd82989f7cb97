"""The ordered sparse convolution (lux3d_sparse_order +
lux3d_sparse_conv3d_ordered): the row order is a permutation sorted by tap
masks, and the convolution matches the oracle at the edges of its tiles, for
every tile shape and pass count."""
import numpy as np
import pytest
import torch

from test_gpu_sparse import dev, ops, orc, random_coords  # noqa: F401 (fixtures)

pytestmark = pytest.mark.gpu


def _table(n, seed, full):
    """A neighbour table with missing, out-of-range and (full) all-present rows; the centre is not always there."""
    rng = np.random.default_rng(seed)
    nbr = rng.integers(0, n, (n, 27)).astype(np.int32)
    nbr[rng.random((n, 27)) < (0.0 if full else 0.7)] = -1
    nbr[::7, 13] = -1
    nbr[5::11, 4] = n + 3          # past the rows: missing
    nbr[3::13] = -1                # rows without any neighbour
    return nbr


@pytest.mark.parametrize("passes", [3, 9])
@pytest.mark.parametrize("n", [1, 255, 256, 257, 3000])
def test_sparse_order_table(dev, ops, n, passes):
    print(f"\n[case] sparse_order n={n} passes={passes}", flush=True)
    nbr = _table(n, n, False)
    t = 27 // passes
    got = ops._sparse_order(torch.from_numpy(nbr).to(dev), passes).cpu().numpy()
    want = np.where((nbr >= 0) & (nbr < n), nbr, -1)
    for s in range(passes):
        rows = got[s, :, 0]
        assert np.array_equal(np.sort(rows), np.arange(n))
        assert np.array_equal(got[s, :, 1:], want[rows, s * t:(s + 1) * t])
        mask = ((got[s, :, 1:] >= 0) << np.arange(t)).sum(1)
        key = (t - (got[s, :, 1:] >= 0).sum(1)) * 512 + mask
        assert (np.diff(key) >= 0).all()   # most taps first, then by mask


# Tiles of 64 x 128, 128 x 64 (up to 64 channels, or up to 128 with 512 row
# tiles) and 128 x 128 (from 1024 tiles on), at their edges.
CASES = [(1, 64, 64), (63, 64, 40), (129, 80, 64), (65, 64, 65), (127, 64, 128), (128, 16, 130), (1000, 96, 200),
         (64 * 1024 + 5, 64, 100), (8 * 1024, 128, 2049)]


@pytest.mark.parametrize("passes", [3, 9])
@pytest.mark.parametrize("n,cin,cout", CASES)
def test_sparse_conv3d_ordered(dev, ops, orc, n, cin, cout, passes):
    """|error| <= (6 27 Cin / 16 + 64) 2^-23 sum |x w|: every accumulation of a 16-deep product step, tap sum and
    output loses at most one unit in the last place of a partial sum, and partial sums stay below the sum of
    magnitudes; a product's dropped terms are below 2^-24 of it."""
    print(f"\n[case] ordered conv n={n} cin={cin} cout={cout} passes={passes}", flush=True)
    nbr = _table(n, n + cin, n < 500)
    rng = np.random.default_rng(cin + cout)
    x = rng.standard_normal((n, cin)).astype(np.float32)
    w27 = (rng.standard_normal((27, cout, cin)) / np.sqrt(27 * cin)).astype(np.float32)
    bias = rng.standard_normal(cout).astype(np.float32) if cout % 2 else None
    conv = ops.SparseConv3d(torch.from_numpy(w27).permute(1, 0, 2).contiguous().to(dev),
                            None if bias is None else torch.from_numpy(bias).to(dev), cin, cout)
    feats = torch.from_numpy(x).to(dev)
    out = torch.full((n, cout), float("nan"), device=dev)
    conv._forward_ordered(ops._sparse_order(torch.from_numpy(nbr).to(dev), passes), feats, out)
    out = out.cpu().numpy()
    assert np.isfinite(out).all()
    rows = np.arange(n) if n <= 1000 else np.unique(np.concatenate([np.arange(70), np.arange(n - 70, n),
                                                                    rng.choice(n, 200)]))
    valid = np.where(nbr < n, nbr, -1)[rows]
    want, mag = orc.sparse_conv3d(x, valid, w27, bias, with_abs=True)
    bound = (6 * 27 * cin / 16 + 64) * 2.0 ** -23 * mag.astype(np.float64) + 2.0 ** -23 * np.abs(want) + 1e-30
    err = np.abs(out[rows].astype(np.float64) - want)
    assert (err <= bound).all(), f"worst {np.max(err / bound):.3f} of the bound"
    # the bound of one output allows more than a lost third term costs. Over all outputs: an f32 chain's rounding steps
    # of 2^-25 each (root mean square) on partial sums no larger than the result's scale stay near 2e-7, without the
    # third terms of x and w, or without the product of the second ones, the relative error is 2e-6 and more
    exact = np.zeros((len(rows), cout))
    for k in range(27):
        has = valid[:, k] >= 0
        exact[has] += x[valid[has, k]].astype(np.float64) @ w27[k].astype(np.float64).T
    if bias is not None:
        exact += bias
    assert np.linalg.norm(out[rows] - exact) <= 1e-6 * np.linalg.norm(exact)


@pytest.mark.parametrize("passes", [3, 9])
@pytest.mark.parametrize("n,cin,cout", [(129, 64, 64), (127, 64, 128), (1000, 96, 200), (64 * 1024 + 5, 64, 100),
                                        (8 * 1024, 128, 2049)])
def test_sparse_conv3d_ordered_keeps_all_bits(dev, ops, n, cin, cout, passes):
    """One product per output, of a value with 24 significant bits and a power of two, is exact: every term of x and
    of the weights takes part, in every tile shape."""
    print(f"\n[case] ordered conv, one product n={n} cin={cin} cout={cout} passes={passes}", flush=True)
    rng = np.random.default_rng(n + cout)
    nbr = _table(n, n + cin, n < 500)
    tap, chan = rng.integers(0, 27, cout), rng.integers(0, cin, cout)
    full = lambda s: ((rng.integers(1 << 23, 1 << 24, s) | 1) * 2.0 ** -23 * rng.choice([-1, 1], s))  # noqa: E731
    power = lambda s: 2.0 ** rng.integers(-3, 4, s)  # noqa: E731
    table = ops._sparse_order(torch.from_numpy(nbr).to(dev), passes)
    for x, w in ((full((n, cin)), power(cout)), (power((n, cin)), full(cout))):
        x, w = x.astype(np.float32), w.astype(np.float32)
        w27 = np.zeros((27, cout, cin), dtype=np.float32)
        w27[tap, np.arange(cout), chan] = w
        conv = ops.SparseConv3d(torch.from_numpy(w27).permute(1, 0, 2).contiguous().to(dev), None, cin, cout)
        out = torch.full((n, cout), float("nan"), device=dev)
        conv._forward_ordered(table, torch.from_numpy(x).to(dev), out)
        src = nbr[:, tap]
        has = (src >= 0) & (src < n)
        want = np.where(has, x[np.where(has, src, 0), chan] * w, np.float32(0))
        assert np.array_equal(out.cpu().numpy(), want)


def test_sparse_conv3d_ordered_under_capture(dev, ops):
    """forward() captured from a rulebook and from a neighbour table: every replay has the eager result, with eager
    work between replays and new features in the captured buffer."""
    print("\n[case] ordered conv under capture", flush=True)
    coords = random_coords(9000, 64, 5, True)
    n, cin, cout = len(coords), 128, 256
    g = torch.Generator(device="cpu").manual_seed(n)
    x = torch.randn((n, cin), generator=g).to(dev)
    conv = ops.SparseConv3d((torch.randn((cout, 27, cin), generator=g) / (27 * cin) ** 0.5).to(dev), None, cin, cout)
    assert conv._order_pays(n)
    nbr = ops.sparse_neighbors(torch.from_numpy(coords).to(dev))
    rb = ops.SparseRulebook(nbr)
    conv.forward(rb, x), conv.forward(nbr, x)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        a, b = conv.forward(rb, x), conv.forward(nbr, x)
    for i in range(4):
        x.normal_()
        want = conv.forward(rb, x), conv.forward(nbr, x)
        a.fill_(float("nan")), b.fill_(float("nan"))
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(a, want[0]) and torch.equal(b, want[1]), i


def test_sparse_rulebook_of_no_voxels(dev, ops):
    print("\n[case] rulebook and ordered conv without voxels", flush=True)
    rb = ops.SparseRulebook(torch.empty((0, 27), dtype=torch.int32, device=dev))
    conv = ops.SparseConv3d(torch.zeros((64, 27, 64), device=dev), None, 64, 64)
    assert conv.forward(rb, torch.empty((0, 64), device=dev)).shape == (0, 64)
    assert rb.counts.cpu().tolist() == [0] * 27


@pytest.mark.parametrize("passes", [3, 9])
def test_sparse_conv3d_ordered_exact_sums(dev, ops, orc, passes):
    """Whole-number inputs whose sums are exact in f32: equal to the oracle bit for bit; an infinite weight reaches
    the rows that have its tap and no other row of their tiles."""
    cin, cout = 64, 96
    coords = random_coords(2000, 24, 22, True)
    n = len(coords)
    rng = np.random.default_rng(23)
    x = rng.integers(-4, 5, (n, cin)).astype(np.float32)
    w27 = (rng.integers(-3, 4, (27, cout, cin)) * 0.25).astype(np.float32)
    nbr = orc.sparse_neighbors(coords)
    table = ops._sparse_order(torch.from_numpy(nbr).to(dev), passes)
    out = torch.empty((n, cout), device=dev)

    def run(w):
        conv = ops.SparseConv3d(torch.from_numpy(w).permute(1, 0, 2).contiguous().to(dev), None, cin, cout)
        conv._forward_ordered(table, torch.from_numpy(x).to(dev), out)
        return out.cpu().numpy()

    want = orc.sparse_conv3d(x, nbr, w27, None)
    assert np.array_equal(run(w27), want)
    w27[2] = np.inf
    has = nbr[:, 2] >= 0
    got = run(w27)
    assert 0 < has.sum() < n and not np.isfinite(got[has]).any()
    w27[2] = 0.0
    assert np.array_equal(got[~has], orc.sparse_conv3d(x, nbr, w27, None)[~has])


def test_sparse_conv3d_routes_agree(dev, ops, orc):
    """forward() from coordinates, from a neighbour table, from a rulebook built on it before the table's buffer is
    reused and from one without row orders, on the sizes where the route or the pass count changes."""
    for n0, cin, cout in ((8192, 128, 64), (4100, 768, 64), (4000, 256, 96), (8100, 128, 64), (20000, 128, 256), (60, 512, 96)):
        coords = random_coords(n0, 64, n0, True)
        n = len(coords)
        g = torch.Generator(device="cpu").manual_seed(n)
        x = torch.randn((n, cin), generator=g).to(dev)
        conv = ops.SparseConv3d((torch.randn((cout, 27, cin), generator=g) / (27 * cin) ** 0.5).to(dev), None, cin, cout)
        c = torch.from_numpy(coords).to(dev)
        nbr = ops.sparse_neighbors(c)
        rb = ops.SparseRulebook(nbr)
        want = conv.forward(nbr, x)
        got = [conv.forward(c, x)]
        nbr.fill_(-1)
        got.append(conv.forward(rb, x))
        del rb.tables
        got.append(conv.forward(rb, x))
        for y in got:
            # f32 sums of up to 27 Cin terms in another order
            assert float((y - want).norm() / want.norm()) < 4e-6, (n, cin)
