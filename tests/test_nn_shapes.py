"""The network's convolution and weight-gradient entries (hgrid_nn_conv3, hgrid_nn_conv3_wgrad) at the
channel counts and strides that its own layers do not have.

Inputs are multiples of 1/64 that BF16 holds, so products are multiples of 2^-12 and FP32 sums below
2^12 are exact: a convolution rounds once, to BF16 (2^-9 of a value at most; the bar is 2^-8 of the norm), a weight
gradient's sums by at most 1e-5 as in test_gpu_surrogate.py."""
import ctypes as C

import numpy as np
import pytest

TAPS = [(t // 9 - 1, t // 3 % 3 - 1, t % 3 - 1) for t in range(27)]


def upload(lg, a, dtype=np.uint16):
    h = (a.astype(np.float32).view(np.uint32) >> 16).astype(np.uint16) if dtype is np.uint16 else np.ascontiguousarray(a, dtype)
    p = C.c_void_p()
    assert lg.hgrid_malloc(C.byref(p), h.nbytes) == 0
    assert lg.hgrid_memcpy_h2d(p, h.ctypes.data, h.nbytes) == 0
    return p


def download(lg, p, n, dtype):
    out = np.empty(n, dtype)
    assert lg.hgrid_memcpy_d2h(out.ctypes.data, p, out.nbytes) == 0
    return out


@pytest.mark.gpu
@pytest.mark.parametrize("S,cin,cout", [(8, 184, 16), (8, 192, 64), (8, 200, 16), (8, 200, 32), (16, 208, 48), (8, 256, 64), (2, 200, 16)])
def test_convolution(lg, S, cin, cout):
    """Channels around 192, where the kernel changes, with every tile shape of output channels."""
    print(f"[case] convolution S {S} cin {cin} cout {cout}", flush=True)
    rng = np.random.default_rng(S + cin + cout)
    n, lgS = 2 * S**3, S.bit_length() - 1
    xs, xo, ys, yo = cin + 24, 16, cout + 8, 8
    X = rng.integers(-127, 128, (n, xs)) / 64.0
    W = rng.integers(-127, 128, (cout, 27, cin)) / 64.0
    bias = rng.integers(-64, 65, cout) / 64.0
    f = lg.hgrid_nn_conv3
    f.argtypes = [C.c_void_p, C.c_int, C.c_int, C.c_int, C.c_void_p, C.c_void_p, C.c_void_p, C.c_int, C.c_int, C.c_int, C.c_void_p,
                  C.c_int, C.c_int, C.c_int, C.c_long, C.c_int]
    px, pw, pb, py = upload(lg, X), upload(lg, W), upload(lg, bias, np.float32), upload(lg, np.zeros((n, ys)))
    assert f(px, xs, xo, cin, pw, pb, py, ys, yo, cout, None, 0, 0, lgS, n, 0) == 0
    got = (download(lg, py, n * ys, np.uint16).astype(np.uint32) << 16).view(np.float32).reshape(n, ys)
    for p in (px, pw, pb, py):
        lg.hgrid_free(p)
    x5 = X[:, xo:xo + cin].reshape(2, S, S, S, cin)
    want = bias + sum(np.roll(x5, [-k for k in d], (1, 2, 3)).reshape(n, cin) @ W[:, t].T for t, d in enumerate(TAPS))
    assert not got[:, :yo].any()
    assert np.linalg.norm(got[:, yo:] - want) < 2.0**-8 * np.linalg.norm(want)


@pytest.mark.gpu
@pytest.mark.parametrize("S,cin,cout,pad", [(64, 24, 16, 24), (32, 40, 32, 24), (16, 184, 16, 24), (8, 24, 32, 24), (8, 16, 16, 22),
                                            (16, 32, 32, 22), (4, 24, 16, 24)])
def test_weight_gradient(lg, S, cin, cout, pad):
    """Channel counts that are not 8 or a multiple of 16, and strides that are no multiple of 8, on cubes of
    the row kernel; and a smaller side."""
    print(f"[case] weight gradient S {S} cin {cin} cout {cout} pad {pad}", flush=True)
    rng = np.random.default_rng(S + cin + cout)
    n, lgS = 2 * S**3, S.bit_length() - 1
    xs, xo, ys, yo = cin + pad, pad - 8, cout + pad, pad - 16
    X = rng.integers(-127, 128, (n, xs)) / 64.0
    dY = rng.integers(-127, 128, (n, ys)) / 64.0
    f = lg.hgrid_nn_conv3_wgrad
    f.argtypes = [C.c_void_p, C.c_int, C.c_int, C.c_int, C.c_void_p, C.c_int, C.c_int, C.c_int, C.c_int, C.c_long, C.c_void_p,
                  C.c_void_p]
    for name in ("hgrid_nn_wgrad_partials", "hgrid_nn_wgrad_chunks", "hgrid_nn_wgrad_chunk"):
        getattr(lg, name).argtypes = [C.c_long, C.c_int]
        getattr(lg, name).restype = C.c_long
    lg.hgrid_nn_reduce.argtypes = [C.c_void_p, C.c_long, C.c_long, C.c_void_p, C.c_int]
    m = 27 * cin * cout
    nparts, nchunks = lg.hgrid_nn_wgrad_partials(n, lgS), lg.hgrid_nn_wgrad_chunks(n, lgS)
    assert nchunks == -(-n // lg.hgrid_nn_wgrad_chunk(n, lgS))
    px, py, part, bpart, out = upload(lg, X), upload(lg, dY), C.c_void_p(), C.c_void_p(), C.c_void_p()
    for p, count in ((part, nparts * m), (bpart, nchunks * cout), (out, m + cout)):
        assert lg.hgrid_malloc(C.byref(p), 4 * count) == 0
    assert f(py, ys, yo, cout, px, xs, xo, cin, lgS, n, part, bpart) == 0
    assert lg.hgrid_nn_reduce(part, nparts, m, out, 0) == 0
    assert lg.hgrid_nn_reduce(bpart, nchunks, cout, out.value + 4 * m, 0) == 0
    got = download(lg, out, m + cout, np.float32)
    for p in (px, py, part, bpart, out):
        lg.hgrid_free(p)
    x5 = X[:, xo:xo + cin].reshape(-1, S, S, S, cin)
    y2 = dY[:, yo:yo + cout]
    ref = np.empty((cout, 27, cin))
    for t, d in enumerate(TAPS):
        ref[:, t] = y2.T @ np.roll(x5, [-k for k in d], (1, 2, 3)).reshape(n, cin)
    assert np.linalg.norm(got[:m] - ref.ravel()) / np.linalg.norm(ref) < 1e-5
    assert np.linalg.norm(got[m:] - y2.sum(0)) / np.linalg.norm(y2.sum(0)) < 1e-5
