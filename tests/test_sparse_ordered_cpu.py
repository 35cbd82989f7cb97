"""Argument checks of the ordered sparse convolution's entries and the rule that picks its pass count (no GPU work)."""
from test_abi_cpu import T, status

from lux3d_fused import _lib, ops


def test_sparse_ordered_argument_errors():
    nbr, ws = T([100, 27], _lib.I32), T([1536], _lib.I32)
    ok3, ok9 = T([3, 100, 10], _lib.I32), T([9, 100, 4], _lib.I32)
    for bad in (T([3, 99, 10], _lib.I32), T([3, 100, 4], _lib.I32), T([9, 100, 10], _lib.I32), T([27, 100, 2], _lib.I32)):
        rc, msg = status("lux3d_sparse_order", nbr, bad, ws, None)
        assert rc == _lib.ERR_SHAPE and "table must be" in msg
    assert status("lux3d_sparse_order", nbr, ok3, T([1535], _lib.I32), None)[0] == _lib.ERR_SHAPE
    assert status("lux3d_sparse_order", T([100, 26], _lib.I32), ok3, ws, None)[0] == _lib.ERR_SHAPE
    assert status("lux3d_sparse_order", T([100, 27], _lib.I64), ok3, ws, None)[0] == _lib.ERR_DTYPE
    x, w, out = T([100, 64], _lib.F32), T([27, 40, 64], _lib.F32), T([100, 40], _lib.F32)
    planes = T([27 * 64 * 64 * 3])
    fn = "lux3d_sparse_conv3d_ordered"
    assert status(fn, x, ok9, w, T([27 * 64 * 64 * 3 - 1]), None, out, None)[0] == _lib.ERR_SHAPE
    assert status(fn, x, T([9, 99, 4], _lib.I32), w, planes, None, out, None)[0] == _lib.ERR_SHAPE
    assert status(fn, T([100, 60], _lib.F32), ok3, T([27, 40, 60], _lib.F32), planes, None, out, None)[0] == _lib.ERR_SHAPE
    assert status(fn, x, ok3, T([27, 40, 64]), planes, None, out, None)[0] == _lib.ERR_DTYPE
    assert status(fn, x, ok3, w, planes, T([41], _lib.F32), out, None)[0] == _lib.ERR_SHAPE
    assert status(fn, T([100, 64], _lib.F32, data=0x100004), ok3, w, planes, None, out, None)[0] == _lib.ERR_LAYOUT
    big = 1 << 23   # x of 2^31 bytes
    rc, msg = status(fn, T([big, 64], _lib.F32), T([3, big, 10], _lib.I32), w, planes, None, T([big, 40], _lib.F32), None)
    assert rc == _lib.ERR_SHAPE and "2^31" in msg


def test_pass_counts():
    assert [ops._order_passes(n, 1024) for n in (4095, 4096, 24575, 24576)] == [3, 9, 9, 3]
    assert ops._order_passes(8000, 512) == 3


def test_calls_that_order_their_rows():
    """Both sides of each line of the rule for a call on a neighbour table."""
    def pays(n, cin, cout):
        conv = ops.SparseConv3d.__new__(ops.SparseConv3d)
        conv.in_channels, conv.out_channels = cin, cout
        return conv._order_pays(n)
    for cin, cout, line in ((1024, 1024, 16), (512, 8, 16), (256, 32, 256), (496, 1024, 256), (128, 64, 32768),
                            (128, 128, 16384), (128, 256, 8192), (192, 192, 8192), (240, 16, 69906), (128, 8, 98304),
                            (64, 64, 98304)):
        assert [pays(n, cin, cout) for n in (line - 1, line)] == [False, True], (cin, cout)
