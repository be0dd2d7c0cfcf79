"""The stand-alone Thomas at row counts around its row chunks (8 rows forward, 4
in the cyclic form, 16 back; 4 and 8 up to 8 rows; one chunk ahead; loads past
the end left out below 128 rows and clamped above) and system counts around a
wave and around the 2^21 from which workgroups are four waves:
solution and overwritten c bitwise equal to the same operations in numpy (which
rounds every one of them).
"""
import numpy as np
import pytest

from pascal_poisson_fft_amd import api

pytestmark = pytest.mark.gpu


def _plain(a, b, c, d):
    c, d = c.copy(), d.copy()
    d[0], c[0] = d[0] / b[0], c[0] / b[0]
    for k in range(1, len(d)):
        r = 1.0 / (b[k] - a[k] * c[k - 1])
        d[k], c[k] = r * (d[k] - a[k] * d[k - 1]), r * c[k]
    for k in range(len(d) - 2, -1, -1):
        d[k] = d[k] - c[k] * d[k + 1]
    return c, d


def _cyclic(a, b, c, d):
    c, d, e, n = c.copy(), d.copy(), np.zeros_like(d), len(d)
    e[1] = -a[1]
    e[n - 1] = -c[n - 1]
    d[1], e[1], c[1] = d[1] / b[1], e[1] / b[1], c[1] / b[1]
    for k in range(2, n):
        r = 1.0 / (b[k] - a[k] * c[k - 1])
        d[k], e[k], c[k] = r * (d[k] - a[k] * d[k - 1]), r * (e[k] - a[k] * e[k - 1]), r * c[k]
    for k in range(n - 2, 0, -1):
        d[k], e[k] = d[k] - c[k] * d[k + 1], e[k] - c[k] * e[k + 1]
    d[0] = (d[0] - a[0] * d[n - 1] - c[0] * d[1]) / (b[0] + a[0] * e[n - 1] + c[0] * e[1])
    d[1:] = d[1:] + d[0] * e[1:]
    return c, d


@pytest.mark.parametrize("n,nsys", [(n, nsys) for n in (1, 2, 3, 4, 5, 6, 7, 8, 9, 10, 11, 13, 14, 16, 17, 18, 19, 26, 32, 33,
                                                        34, 35, 50, 127, 128, 129, 136, 145) for nsys in (1, 63, 130)] +
                         [(n, nsys) for n in (3, 6) for nsys in (2**21 - 30, 2**21 + 70)])
def test_row_chunks_bitwise(n, nsys):
    rng = np.random.default_rng(n * 1000 + nsys)
    a, c, d = rng.uniform(0.1, 1.0, (n, nsys)), rng.uniform(0.1, 1.0, (n, nsys)), rng.standard_normal((n, nsys))
    b = -(a + c) - rng.uniform(0.5, 2.0, (n, nsys))
    plan = api.TDMAPlanMany(nsys, 1, n)
    for solve, want in ((plan.solve, _plain), (plan.solve_cycle, _cyclic)):
        if n < 2 and want is _cyclic:
            with pytest.raises(api.PPFError):
                solve(*(api.DeviceArray.from_host(x) for x in (a, b, c, d)))
            continue
        dev = [api.DeviceArray.from_host(x) for x in (a, b, c, d)]
        solve(*dev)
        api.sync()
        cw, dw = want(a, b, c, d)
        assert np.array_equal(dev[3].download(), dw)
        assert np.array_equal(dev[2].download(), cw)
        for x in dev:
            x.free()
    plan.destroy()
