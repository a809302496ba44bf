"""Copies between the host's field layouts and the device: whole blocks in
place of row-by-row copies.  Grids with one block and with several (a block
holds 4 MB of rows; padded rows leave a ragged last one)."""
import numpy as np
import pytest

from relax_amd import fourier, load
from relax_amd._lib import ptr
from relax_amd.model import Model

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [(32, 32, 32), (64, 256, 256), (1024, 32, 128)])
@pytest.mark.parametrize("align", [0, 1])
def test_state_round_trip(n, align):
    n1, n2, h3 = n[0], n[1], n[2] // 2
    rng = np.random.default_rng(5)
    p = n1 + 2 * align
    u = [rng.standard_normal((h3, n2, p), np.float32) for _ in range(4)]
    tau, sig = (rng.standard_normal((h3, n2, n1, 6), np.float32) for _ in range(2))
    with Model(*n, 1.0, 1.0, 1.0, 3e4, 3e4) as m:
        m.upload(*u[:3], tau, sig, u[3], align_data=align)
        # the caller's padding stays as it is
        out = [np.full((h3, n2, p), 7.0, np.float32) for _ in range(4)]
        t2, s2 = np.zeros_like(tau), np.zeros_like(sig)
        assert load().relax_model_download(m.handle, *[ptr(a) for a in out[:3]], ptr(t2), ptr(s2), ptr(out[3]), None,
                                           align) == 0
        top = [np.full((n2, p), 7.0, np.float32) for _ in range(3)]
        assert load().relax_model_surface(m.handle, *[ptr(a) for a in top], align) == 0
    for a, b in zip(u, out):
        assert np.array_equal(a[..., :n1], b[..., :n1])
        assert np.all(b[..., n1:] == 7.0)
    for a, b in zip(u, top):
        assert np.array_equal(a[0, :, :n1], b[:, :n1])
        assert np.all(b[:, n1:] == 7.0)
    assert np.array_equal(tau, t2) and np.array_equal(sig, s2)


@pytest.mark.parametrize("n", [(16, 16, 16), (64, 64, 512)])
def test_packed_rows_equal_padded(n):
    n1, n2, n3 = n
    rng = np.random.default_rng(6)
    x = rng.standard_normal((n3, n2, n1), np.float32)
    a = np.zeros((n3, n2, n1 + 2), np.float32)
    a[..., :n1] = x
    b = np.zeros((n3, n2, n1 + 2), np.float32)
    b.reshape(-1)[:x.size] = x.reshape(-1)
    for d in (-1, 1):
        fourier.fft3(a, n1, n2, n3, 0.5, 1.0, 2.0, d, align_data=1)
        fourier.fft3(b, n1, n2, n3, 0.5, 1.0, 2.0, d, align_data=0)
        if d < 0:
            assert np.array_equal(a, b)
    assert np.array_equal(a[..., :n1], b.reshape(-1)[:x.size].reshape(x.shape))
