"""The network's tiled convolutions at the sizes where their launch rule picks
256-pixel tiles, two or four output-channel tiles per block, nearly all of the
96 KB of staged rows, and, in the weight gradient, several chunks of pixels
per block: against the numpy oracle (on the first, a middle and the last image
where every image is its own), the last tile and chunk partly empty."""
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


# N, H, W, Cin, Cout and (pixels, channel tiles) per block of the pass
FWD = [(67, 31, 16, 16, 32, (64, 2)), (67, 31, 16, 8, 64, (64, 4)), (67, 31, 16, 32, 32, (64, 2)),
       (71, 62, 16, 8, 16, (256, 1)), (129, 65, 16, 16, 32, (256, 2)),
       (131, 63, 16, 16, 64, (256, 4)), (67, 31, 16, 128, 32, (256, 1)),
       (67, 31, 32, 64, 16, (256, 1))]


@pytest.mark.parametrize('N,H,W,Cin,Cout,shape', FWD)
def test_conv_tile_shapes(tenet, N, H, W, Cin, Cout, shape):
    """Forward, and backward-data of the layer with the channels exchanged
    (the same kernel and launch, on flipped weights)."""
    from idmx import _lib
    from idmx.warmstart import _Buf, _bf16
    from oracle import nn_ref
    P, cots = N * H * W, (Cout + 15) // 16
    assert P % shape[0] != 0
    # the launch rule: 256 pixels where that makes 256 blocks, channel tiles
    # that leave 512
    m = 4 if Cin <= 16 else 2 if Cin == 32 else 1
    ct = 4 if cots % 4 == 0 and m >= 4 else 2 if cots % 2 == 0 and m >= 2 else 1
    tp = 256 if -(-P // 256) * (cots // ct) >= 256 else 64
    while ct > 1 and -(-P // tp) * (cots // ct) < 512:
        ct //= 2
    assert (tp, ct) == shape
    rng = np.random.default_rng(P + Cin)
    h, pick = tenet.handle, [0, N // 2, N - 1]
    x = nn_ref.bf16_round(rng.standard_normal((N, H, W, Cin), dtype=np.float32))
    w = (rng.standard_normal((Cout, 9 * Cin)) / np.sqrt(9 * Cin)).astype(np.float32)
    wb = nn_ref.bf16_round(w)
    b = rng.standard_normal(Cout).astype(np.float32)
    bufs = [_dev(tenet, a) for a in (_bf16(x), _bf16(w), b)]
    out, out32 = _Buf(tenet, P * Cout * 2), _Buf(tenet, P * Cout * 4)
    _lib.call('idmx_nn_conv3x3_fwd', h, bufs[0].ptr, bufs[1].ptr, bufs[2].ptr, out.ptr, out32.ptr,
              N, H, W, Cin, Cout, 1)
    ref = nn_ref.conv3x3(x[pick], wb, b)
    got = out32.d2h(np.float32, (N, H, W, Cout))[pick]
    # 9 Cin products in FP32; bf16 outputs carry 2^-8 of their value
    assert np.abs(got - ref).max() <= 1e-5 * max(1.0, np.abs(ref).max())
    got = _f32(out.d2h(np.uint16, (N, H, W, Cout)))[pick]
    assert np.abs(got - np.maximum(ref, 0)).max() <= 8e-3 * max(1.0, np.abs(ref).max())
    # a layer Cout -> Cin whose gradient tensor is x
    wd = (rng.standard_normal((Cin, 9 * Cout)) / np.sqrt(9 * Cout)).astype(np.float32)
    dwd, scratch = _dev(tenet, wd), _Buf(tenet, wd.size * 2)
    dx = _Buf(tenet, P * Cout * 2)
    _lib.call('idmx_nn_conv3x3_bwd_data', h, bufs[0].ptr, dwd.ptr, scratch.ptr, dx.ptr, N, H, W,
              Cout, Cin)
    ref = nn_ref.conv3x3_bwd_data(x[pick], nn_ref.bf16_round(wd), Cout)
    got = _f32(dx.d2h(np.uint16, (N, H, W, Cout)))[pick]
    assert np.abs(got - ref).max() <= 8e-3 * max(1.0, np.abs(ref).max())


# chunks of 64 pixels below 2^15, of 256 above; 256 blocks share the chunks
BWD = [(67, 31, 32, 16, 16), (67, 31, 32, 8, 32), (133, 31, 16, 32, 64), (35, 31, 64, 16, 1),
       (67, 33, 32, 128, 32), (270, 31, 8, 64, 64), (19, 31, 32, 16, 32)]


@pytest.mark.parametrize('N,H,W,Cin,Cout', BWD)
def test_layer_backward_over_several_chunks_per_block(tenet, N, H, W, Cin, Cout):
    """The fused layer backward: ReLU mask, weight gradient, its sums in the
    backward-data launch, and the input gradient."""
    from idmx import _lib
    from idmx.warmstart import _Buf, _bf16
    from oracle import nn_ref
    P = N * H * W
    assert (P % (64 if P < 32768 else 256) != 0) and (P < 32768 or P > 65536)
    rng = np.random.default_rng(P + Cout)
    h, pick = tenet.handle, [0, N // 2, N - 1]
    x, y, g = (nn_ref.bf16_round(rng.standard_normal((N, H, W, c), dtype=np.float32))
               for c in (Cin, Cout, Cout))
    w = (rng.standard_normal((Cout, 9 * Cin)) / np.sqrt(9 * Cin)).astype(np.float32)
    dx_, dy_, dg, dwf = (_dev(tenet, a) for a in (_bf16(x), _bf16(y), _bf16(g), w))
    gw, gb = _dev(tenet, np.ones_like(w)), _dev(tenet, np.ones(Cout, np.float32))
    scratch, dxo = _Buf(tenet, w.size * 2), _Buf(tenet, P * Cin * 2)
    _lib.call('idmx_nn_conv3x3_bwd', h, dx_.ptr, dy_.ptr, dg.ptr, dwf.ptr, scratch.ptr, dxo.ptr,
              gw.ptr, gb.ptr, N, H, W, Cin, Cout)
    g = np.where(y > 0, g, 0).astype(np.float32)
    assert np.array_equal(_f32(dg.d2h(np.uint16, g.shape)), g)
    rw, rb = nn_ref.conv3x3_bwd_weight(x, g)
    # sums of P products in FP32, in chunks
    assert np.abs(gw.d2h(np.float32, rw.shape) - 1 - rw).max() <= 1e-4 * np.abs(rw).max()
    assert np.abs(gb.d2h(np.float32, rb.shape) - 1 - rb).max() <= 1e-4 * np.abs(rb).max()
    rd = nn_ref.conv3x3_bwd_data(g[pick], nn_ref.bf16_round(w), Cin)
    got = _f32(dxo.d2h(np.uint16, x.shape))[pick]
    assert np.abs(got - rd).max() <= 8e-3 * max(1.0, np.abs(rd).max())
