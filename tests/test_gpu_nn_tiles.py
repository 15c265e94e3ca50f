"""The tiled convolution kernels of the warm-start network against the numpy
oracle at the edges of their tiles (256 and 64 pixels, 16 channels, one to
four channel tiles, image borders inside a tile, widths that are no powers of
two), and the fused calls against the single ones they replace."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _dev(tenet, a):
    from idmx.warmstart import _Buf
    b = _Buf(tenet, a.nbytes)
    b.h2d(a)
    return b


def _f32(u16):
    return (u16.astype(np.uint32) << 16).view(np.float32)


CASES = [(1, 1, 1, 64, 64), (3, 5, 7, 8, 16), (1, 9, 28, 16, 33), (2, 16, 16, 32, 64),
         (5, 8, 8, 64, 64), (2, 4, 4, 128, 32), (1, 3, 130, 16, 16), (1, 33, 64, 8, 16),
         (2, 64, 64, 16, 1), (1, 16, 32, 64, 16), (3, 8, 16, 32, 32), (1, 2, 256, 16, 32)]


@pytest.mark.parametrize('N,H,W,Cin,Cout', CASES)
def test_conv_tiles_match_oracle(tenet, N, H, W, Cin, Cout):
    from idmx import _lib
    from idmx.warmstart import _Buf, _bf16
    from oracle import nn_ref
    rng = np.random.default_rng(N * 1000 + H + W + Cin)
    x = nn_ref.bf16_round(rng.standard_normal((N, H, W, Cin)).astype(np.float32))
    w = (rng.standard_normal((Cout, 9 * Cin)) / np.sqrt(9 * Cin)).astype(np.float32)
    wb = nn_ref.bf16_round(w)
    b = rng.standard_normal(Cout).astype(np.float32)
    g = nn_ref.bf16_round(rng.standard_normal((N, H, W, Cout)).astype(np.float32))
    h = tenet.handle
    dx_, dw_, db_, dwf, dg = (_dev(tenet, a) for a in (_bf16(x), _bf16(w), b, w, _bf16(g)))
    out, out32 = _Buf(tenet, N * H * W * Cout * 2), _Buf(tenet, N * H * W * Cout * 4)
    _lib.call('idmx_nn_conv3x3_fwd', h, dx_.ptr, dw_.ptr, db_.ptr, out.ptr, out32.ptr, N, H, W,
              Cin, Cout, 1)
    ref = nn_ref.conv3x3(x, wb, b)
    assert np.abs(out32.d2h(np.float32, ref.shape) - ref).max() <= 1e-5 * max(1.0, np.abs(ref).max())
    got = _f32(out.d2h(np.uint16, ref.shape))
    assert np.abs(got - np.maximum(ref, 0)).max() <= 8e-3 * max(1.0, np.abs(ref).max())
    gw, gb = _dev(tenet, np.ones_like(w)), _dev(tenet, np.ones_like(b))
    _lib.call('idmx_nn_conv3x3_bwd_weight', h, dx_.ptr, dg.ptr, gw.ptr, gb.ptr, N, H, W, Cin,
              Cout)
    rw, rb = nn_ref.conv3x3_bwd_weight(x, g)
    assert np.abs(gw.d2h(np.float32, rw.shape) - 1 - rw).max() <= 1e-4 * max(1.0, np.abs(rw).max())
    assert np.abs(gb.d2h(np.float32, rb.shape) - 1 - rb).max() <= 1e-4 * max(1.0, np.abs(rb).max())
    scratch, dxo = _Buf(tenet, w.size * 2), _Buf(tenet, x.size * 2)
    _lib.call('idmx_nn_conv3x3_bwd_data', h, dg.ptr, dwf.ptr, scratch.ptr, dxo.ptr, N, H, W, Cin,
              Cout)
    rd = nn_ref.conv3x3_bwd_data(g, wb, Cin)
    assert np.abs(_f32(dxo.d2h(np.uint16, x.shape)) - rd).max() <= 8e-3 * max(1.0, np.abs(rd).max())


@pytest.mark.parametrize('N,H,W,Cin,Cout', [(3, 8, 8, 64, 64), (2, 16, 16, 16, 1),
                                            (1, 6, 10, 4, 5), (2, 32, 32, 32, 16)])
def test_fused_layer_backward_equals_single_calls(tenet, N, H, W, Cin, Cout):
    from idmx import _lib
    from idmx.warmstart import _Buf, _bf16
    rng = np.random.default_rng(7)
    h = tenet.handle
    x, y, g = (_bf16(rng.standard_normal((N, H, W, c)).astype(np.float32))
               for c in (Cin, Cout, Cout))
    w = rng.standard_normal((Cout, 9 * Cin)).astype(np.float32)
    dx_, dy_, dwf = _dev(tenet, x), _dev(tenet, y), _dev(tenet, w)
    res = []
    for fused in (True, False):
        dg = _dev(tenet, g)
        gw, gb = _Buf(tenet, w.nbytes), _Buf(tenet, 4 * Cout)
        sc, dxo = _Buf(tenet, w.size * 2), _Buf(tenet, x.nbytes)
        if fused:
            _lib.call('idmx_nn_conv3x3_bwd', h, dx_.ptr, dy_.ptr, dg.ptr, dwf.ptr, sc.ptr,
                      dxo.ptr, gw.ptr, gb.ptr, N, H, W, Cin, Cout)
        else:
            _lib.call('idmx_nn_relu_bwd', h, dy_.ptr, dg.ptr, dg.ptr, N * H * W * Cout)
            _lib.call('idmx_nn_conv3x3_bwd_weight', h, dx_.ptr, dg.ptr, gw.ptr, gb.ptr, N, H, W,
                      Cin, Cout)
            _lib.call('idmx_nn_conv3x3_bwd_data', h, dg.ptr, dwf.ptr, sc.ptr, dxo.ptr, N, H, W,
                      Cin, Cout)
        res.append((dg.d2h(np.uint16, g.shape), dxo.d2h(np.uint16, x.shape),
                    gw.d2h(np.float32, w.shape), gb.d2h(np.float32, (Cout,))))
    assert np.array_equal(res[0][0], res[1][0]) and np.array_equal(res[0][1], res[1][1])
    for a, b in zip(res[0][2:], res[1][2:]):
        # one sum of N H W products, in FP32, in another order at most
        assert np.abs(a - b).max() <= 1e-5 * max(1.0, np.abs(b).max())


@pytest.mark.parametrize('N,H,W,C,Cs', [(2, 4, 6, 16, 16), (3, 5, 3, 64, 8), (1, 2, 2, 3, 5)])
def test_cat_and_skip_gradient(tenet, N, H, W, C, Cs):
    from idmx import _lib
    from idmx.warmstart import _Buf, _bf16
    from oracle import nn_ref
    rng = np.random.default_rng(11)
    h = tenet.handle
    x = nn_ref.bf16_round(rng.standard_normal((N, H, W, C)).astype(np.float32))
    sk = nn_ref.bf16_round(rng.standard_normal((N, 2 * H, 2 * W, Cs)).astype(np.float32))
    dx_, ds_ = _dev(tenet, _bf16(x)), _dev(tenet, _bf16(sk))
    y = _Buf(tenet, N * 4 * H * W * (C + Cs) * 2)
    _lib.call('idmx_nn_cat_up2', h, dx_.ptr, ds_.ptr, y.ptr, N, H, W, C, Cs)
    got = _f32(y.d2h(np.uint16, (N, 2 * H, 2 * W, C + Cs)))
    assert np.array_equal(got[..., :C], x.repeat(2, 1).repeat(2, 2))
    assert np.array_equal(got[..., C:], sk)
    # gradient of a tensor (Cs channels) that feeds the pool and that skip
    dp = nn_ref.bf16_round(rng.standard_normal((N, H, W, Cs)).astype(np.float32))
    ddp = _dev(tenet, _bf16(dp))
    out, tmp = _Buf(tenet, sk.size * 2), _Buf(tenet, sk.size * 2)
    _lib.call('idmx_nn_pool2_bwd_add', h, ddp.ptr, y.ptr, out.ptr, tmp.ptr, N, 2 * H, 2 * W, Cs,
              C + Cs, C)
    ref = nn_ref.bf16_round(0.25 * dp.repeat(2, 1).repeat(2, 2) + sk)
    assert np.array_equal(_f32(out.d2h(np.uint16, sk.shape)), ref)
