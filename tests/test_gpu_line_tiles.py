"""Stand-alone transforms on the tile kernels (compiled lengths, and the other
even lengths up to 2048) and beyond them, against scipy's transforms (which
share FFTW's unnormalised definitions): every kind, lines along and across
memory, one line per outer step, counts that leave a partial tile, padding
between lines untouched; FP64 and FP32.  Tolerance 40 eps log2(n) of the
largest output: an FFT's rounding grows with its log2(n) passes.
The kept tables: more lengths than are kept, several threads, and after
flutas_fft_cleanup."""
import ctypes as C
import threading

import numpy as np
import pytest
import scipy.fft as sf

pytestmark = pytest.mark.gpu

KINDS = {"R2HC": 0, "HC2R": 1, "REDFT01": 4, "REDFT10": 5, "REDFT11": 6, "RODFT01": 8,
         "RODFT10": 9, "RODFT11": 10}


def _ref(kind, x):
    n = x.shape[0]
    if kind == "R2HC":
        h = np.fft.rfft(x, axis=0)
        return np.concatenate([h.real, h.imag[1:n - n // 2][::-1]])
    if kind == "HC2R":
        h = x[:n // 2 + 1].astype(complex)
        h[1:n - n // 2] += 1j * x[n // 2 + 1:][::-1]
        return np.fft.irfft(h, n, axis=0) * n
    t = {"01": 3, "10": 2, "11": 4}[kind[-2:]]
    return (sf.dct if kind[1] == "E" else sf.dst)(x, type=t, axis=0)


# n, then (stride, howmany1, dist1, howmany2, dist2) of a buffer with gaps
def _geoms(n):
    return [(1, 17, n + 3, 3, 17 * (n + 3) + 5), (19, 17, 1, 2, 19 * n + 1),
            (2, 1, 7, 35, 2 * n + 1), (1, 1, 1, 1, 0)]


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("n", [2, 30, 32, 90, 128, 400, 462, 512, 1024, 1030, 2046, 2048, 2050])
def test_lines_match_scipy(api, n, dtype):
    rng = np.random.default_rng(n)
    fn = api.lib.flutas_fft_guru if dtype is np.float64 else api.lib.flutas_fft_guru_f32
    ct = C.c_double if dtype is np.float64 else C.c_float
    tol = 40 * np.finfo(dtype).eps * max(1.0, np.log2(n))
    for st, h1, d1, h2, d2 in _geoms(n):
        idx = (np.arange(n)[:, None, None] * st + np.arange(h1)[None, :, None] * d1 +
               np.arange(h2)[None, None, :] * d2)
        size = int(idx.max()) + 5
        for kind, code in KINDS.items():
            host = rng.standard_normal(size).astype(dtype)
            dev = api.DeviceArray.from_host(host)
            rc = fn(C.c_int(code), C.c_int(n), C.c_longlong(st), C.c_int(h1), C.c_longlong(d1),
                    C.c_int(h2), C.c_longlong(d2), C.cast(C.c_void_p(dev.ptr), C.POINTER(ct)))
            assert rc == 0, api.lib.flutas_last_error().decode()
            got, ref = dev.to_host(), host.astype(np.float64)
            ref[idx] = _ref(kind, host[idx].astype(np.float64))
            err = np.max(np.abs(got[idx] - ref[idx])) / np.max(np.abs(ref[idx]))
            assert err <= tol, (kind, n, st, err)
            out = np.ones(size, bool)
            out[idx] = False
            np.testing.assert_array_equal(got[out], host[out])


def test_kept_tables(api):
    def run(seed):
        rng = np.random.default_rng(seed)
        for n in rng.permutation(np.arange(10, 58, 2)):  # 24 lengths, 16 kept
            x = rng.standard_normal((n, 5))
            d = api.DeviceArray.from_host(np.asfortranarray(x))
            api.fft_lines("REDFT10", d, int(n), 5)
            err = np.max(np.abs(d.to_host() - _ref("REDFT10", x)))
            bad.append(err) if err > 1e-11 else None

    bad = []
    run(0)
    threads = [threading.Thread(target=run, args=(s,)) for s in (1, 2, 3)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert api.lib.flutas_fft_cleanup() == 0
    run(4)
    assert not bad
