"""Tables of the stand-alone transforms shared by threads: more lengths in use
than are kept, every call's result against scipy's transform (40 eps log2(n) of
the largest output), and any failure of a thread reported."""
import threading

import numpy as np
import pytest
import scipy.fft as sf

pytestmark = pytest.mark.gpu


def test_threads_share_kept_tables(api):
    bad, done = [], []

    def work(seed):
        try:
            rng = np.random.default_rng(seed)
            lengths = [int(n) for n in rng.permutation(np.r_[np.arange(10, 58, 2), 64, 128, 2050])]
            for n in lengths:
                x = rng.standard_normal((n, 5))
                d = api.DeviceArray.from_host(np.asfortranarray(x))
                api.fft_lines("REDFT10", d, n, 5)
                ref = sf.dct(x, type=2, axis=0)
                err = np.max(np.abs(d.to_host() - ref)) / np.max(np.abs(ref))
                if not err <= 40 * np.finfo(np.float64).eps * np.log2(n):
                    bad.append((seed, n, err))
                if seed == 3 and n % 16 == 0:
                    assert api.lib.flutas_fft_cleanup() == 0
                done.append(n)
        except BaseException as e:  # a thread's own end would pass unseen
            bad.append((seed, repr(e)))

    threads = [threading.Thread(target=work, args=(s,)) for s in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad, bad
    assert len(done) == 4 * 27
    assert api.lib.flutas_fft_cleanup() == 0
