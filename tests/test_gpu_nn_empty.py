"""A weight gradient over no pixels adds nothing and is no error, whatever the
tiled kernels make of the other sizes."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('Cin,Cout', [(16, 32), (8, 1), (4, 5)])
@pytest.mark.parametrize('N,H,W', [(0, 16, 16), (2, 0, 16), (2, 16, 0)])
def test_weight_gradient_of_no_pixels(tenet, N, H, W, Cin, Cout):
    from idmx import _lib
    from idmx.warmstart import _Buf
    w0 = np.arange(Cout * 9 * Cin, dtype=np.float32)
    b0 = np.arange(Cout, dtype=np.float32)
    gw, gb = _Buf(tenet, w0.nbytes), _Buf(tenet, b0.nbytes)
    gw.h2d(w0)
    gb.h2d(b0)
    x, g = _Buf(tenet, 4096), _Buf(tenet, 4096)
    _lib.call('idmx_nn_conv3x3_bwd_weight', tenet.handle, x.ptr, g.ptr, gw.ptr, gb.ptr, N, H, W,
              Cin, Cout)
    assert np.array_equal(gw.d2h(np.float32, w0.shape), w0)
    assert np.array_equal(gb.d2h(np.float32, b0.shape), b0)
