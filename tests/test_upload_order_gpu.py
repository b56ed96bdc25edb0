"""Small host uploads into a batch whose device arrays the caller holds: they are
in place when the call returns, also for a reader on a stream of its own."""
import ctypes

import numpy as np
import pytest

from gpusim2grid_amd import _capi
from gpusim2grid_amd import synthetic as syn

pytestmark = pytest.mark.gpu


def _peek(ptr, n, stream):
    """n complex values of row 0 of a tiled [n][64] array, read on `stream`."""
    import torch

    class Arr:
        __cuda_array_interface__ = dict(shape=(n, 64, 2), typestr="<f8", data=(ptr, False), version=3, strides=None)

    with torch.cuda.stream(stream):
        a = torch.as_tensor(Arr(), device="cuda")[:, 0].clone()
    stream.synchronize()
    return torch.view_as_complex(a).cpu().numpy()


@pytest.mark.parametrize("shared_row", [False, True])
def test_small_uploads_are_in_place_on_return(shared_row):
    import torch
    g = syn.grid_118()
    s = torch.cuda.Stream()
    other = torch.cuda.Stream()
    B = _capi.Batch(_capi.Plan.from_grid(g.Ybus, g.pv, g.pq, g.slack), 1, stream=ctypes.c_void_p(s.cuda_stream))
    S, V = g.Sbus.astype(np.complex128), g.flat_start().astype(np.complex128)
    row = (lambda a: a) if shared_row else (lambda a: a[None])
    B.set_sbus(row(S))
    B.set_v(row(V))
    pv, ps = ctypes.c_void_p(), ctypes.c_void_p()
    assert _capi.lib().g2g_batch_device_arrays(B._h, ctypes.byref(pv), ctypes.byref(ps)) == 0
    np.testing.assert_array_equal(_peek(ps.value, g.n_bus, other), S)  # (the uploads before the call, too)
    np.testing.assert_array_equal(_peek(pv.value, g.n_bus, other), V)
    x = torch.randn(4096, 4096, device="cuda")
    torch.cuda.synchronize()
    for k in range(1, 4):
        with torch.cuda.stream(s):  # milliseconds of work ahead of the upload on the batch's stream
            for _ in range(20):
                x = torch.tanh(x @ x)
        B.set_sbus(row(S * k))
        np.testing.assert_array_equal(_peek(ps.value, g.n_bus, other), S * k)
        with torch.cuda.stream(s):
            for _ in range(20):
                x = torch.tanh(x @ x)
        B.set_v(row(V * k))
        np.testing.assert_array_equal(_peek(pv.value, g.n_bus, other), V * k)
    s.synchronize()
