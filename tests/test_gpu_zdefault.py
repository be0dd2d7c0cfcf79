"""The z-pass shape of a plan that was not tuned, at the line lengths where the
rule changes shape, on a small grid (few workgroups: 8-column shapes) and on one
with four 16-column workgroups per CU, against the FP64 oracle.

FP64 plans are held to 1e-12 up to 512 rows and to 1e-11 above: the pinned
(0,0) line is ill conditioned, and the oracle's own FP64 Thomas on it is off an
80-bit solve of these inputs by up to 0.5e-12 of the whole solution at 514 rows
and 1.06e-12 at 770 (0.16e-12 at 512), so that two correct FP64 algorithms may
differ by a few times that.  FP32_IR plans
run one FP32 solve without corrections: storage rounding is 6e-8 a pass over
five passes, relative to the largest values of a field whose smallest modes
dominate, so 5e-6 bounds it and a wrong row or mask (order one) does not pass.
"""
import numpy as np
import pytest

from oracle import oracle as O
from pascal_poisson_fft_amd import api
from pascal_poisson_fft_amd.grid import make_axis

pytestmark = pytest.mark.gpu

SMALL = [2, 8, 24, 26, 400, 402, 512, 514, 768, 770, 1024, 1026, 1536, 1538, 2048, 2050, 3072, 3074, 4096]
LARGE = [2, 4, 24, 26, 64, 66, 128, 130, 256, 258, 320, 322, 384, 386, 416, 418, 448, 450, 512, 514, 768, 770, 1022]


def _solve(n1, n2, n3, pbc, precision, zvariant=0, pz=False):
    L = (2.0, 3.0, 1.5)
    ax, ay = make_axis(n1, L[0], pbc[0]), make_axis(n2, L[1], pbc[1])
    az = make_axis(n3, L[2], pz, uniform=pz, gamma=1.6)
    f = np.random.default_rng(n1 + n3).standard_normal((n3, n2, n1))
    f -= float(np.einsum("kji,k->", f, az.dx[1:n3 + 1])) / (az.dx[1:n3 + 1].sum() * n1 * n2)
    ref = O.solve(f, L, (pbc[0], pbc[1], pz), ax.dmx, ay.dmx, az.dmx, az.dx)
    plan = api.FFTPoisson(n1, n2, n3, L, (pbc[0], pbc[1], pz), precision=precision)
    plan.set_zvariant(zvariant)
    dev = api.Problem3D(f, ax, ay, az)
    try:
        args = (dev.rhs, dev.p, dev.dmx1, dev.dmx2, dev.dmx3, dev.dx3)
        plan.solve_sweeps(*args, 0)
        api.sync()
        got = dev.p.download()
    finally:
        dev.free()
        plan.clean()
    return float(np.linalg.norm(got - ref) / np.linalg.norm(ref))


@pytest.mark.parametrize("precision", [api.PPF_PREC_FP64, api.PPF_PREC_FP32_IR], ids=["fp64", "fp32"])
@pytest.mark.parametrize("n1,n2,n3", [(20, 12, n) for n in SMALL] + [(160, 120, n) for n in LARGE])
def test_default_z_shape_matches_oracle(n1, n2, n3, precision):
    # 20 columns, and the 162 of periodic x, leave a ragged last column tile
    pbc = (n3 % 4 == 2, n3 % 8 >= 4)
    err = _solve(n1, n2, n3, pbc, precision)
    bar = (1e-12 if n3 <= 512 else 1e-11) if precision == api.PPF_PREC_FP64 else 5e-6
    assert err <= bar, err


@pytest.mark.parametrize("precision", [api.PPF_PREC_FP64, api.PPF_PREC_FP32_IR], ids=["fp64", "fp32"])
@pytest.mark.parametrize("n3", [2, 4, 30, 32, 34, 62, 64, 66, 96, 130])
def test_one_thread_per_line_matches_oracle(n3, precision):
    """The one-thread-per-line solve around its 32-row chunks: lines within one
    chunk, whole chunks, and one pair of rows past them; ragged columns."""
    err = _solve(20, 12, n3, (n3 % 4 == 2, n3 % 8 >= 4), precision, zvariant=6)
    bar = 1e-12 if precision == api.PPF_PREC_FP64 else 5e-6
    assert err <= bar, err


@pytest.mark.parametrize("precision", [api.PPF_PREC_FP64, api.PPF_PREC_FP32_IR], ids=["fp64", "fp32"])
@pytest.mark.parametrize("n1,n2,n3,v", [(20, 12, 4, 0), (20, 12, 130, 0), (20, 12, 402, 0), (20, 12, 770, 0),
                                        (20, 12, 1026, 0), (20, 12, 2050, 0), (160, 120, 4, 0), (160, 120, 66, 0),
                                        (160, 120, 130, 0), (160, 120, 386, 0), (160, 120, 514, 0), (20, 12, 4, 6),
                                        (20, 12, 34, 6), (20, 12, 96, 6)])
def test_periodic_z_matches_oracle(n1, n2, n3, v, precision):
    """Periodic z through the default shapes and the one-thread-per-line kernel
    (6, the default at 2050 rows), walls and periods in x and y: the z ghost
    planes are the wrapped end planes, also for FP32_IR (no correction runs, so
    nothing rewrites them).  FP64 bars: 1e-11 over 270 rows, where the oracle's
    own FP64 solve of uniform lines is up to 4e-12 (512 rows) off an 80-bit one;
    lines of 2 rows are left out, where the reference's cyclic form drops a
    coupling."""
    err = _solve(n1, n2, n3, (n3 % 4 == 2, n3 % 8 >= 4), precision, zvariant=v, pz=True)
    bar = (1e-12 if n3 <= 270 else 1e-11) if precision == api.PPF_PREC_FP64 else 5e-6
    assert err <= bar, err


@pytest.mark.parametrize("precision", [api.PPF_PREC_FP64, api.PPF_PREC_FP32_IR], ids=["fp64", "fp32"])
@pytest.mark.parametrize("n3", [192, 194, 256, 258, 320, 322, 384, 386, 448, 450, 512, 514, 768, 770, 1024])
def test_default_z_shape_of_middle_grids(n3, precision):
    """Between one and four 16-column workgroups per CU (120 x 96: 768 with
    walls in x and y, on 256 CUs) lines over 192 rows take 16 columns a
    workgroup, the same bits as the shape pinned: 8 columns made them up to a
    third slower there."""
    n1, n2, L = 120, 96, (2.0, 3.0, 1.5)
    ax, ay, az = make_axis(n1, L[0], False), make_axis(n2, L[1], False), make_axis(n3, L[2], False)
    f = np.random.default_rng(n3).standard_normal((n3, n2, n1))
    plan = api.FFTPoisson(n1, n2, n3, L, (False, False, False), precision=precision)
    dev = api.Problem3D(f - f.mean(), ax, ay, az)
    shape = next(v for rows, v in ((192, 5), (256, 1), (320, 7), (384, 12), (448, 17), (512, 3), (768, 12), (1024, 3))
                 if n3 <= rows)
    got = []
    try:
        for v in (0, shape):
            plan.set_zvariant(v)
            plan.solve_sweeps(dev.rhs, dev.p, dev.dmx1, dev.dmx2, dev.dmx3, dev.dx3, 0)
            api.sync()
            got.append(dev.p.download())
    finally:
        dev.free()
        plan.clean()
    ref = O.solve(f - f.mean(), L, (False, False, False), ax.dmx, ay.dmx, az.dmx, az.dx)
    err = float(np.linalg.norm(got[0] - ref) / np.linalg.norm(ref))
    bar = (1e-12 if n3 <= 512 else 1e-11) if precision == api.PPF_PREC_FP64 else 5e-6
    assert np.array_equal(got[0], got[1]) and err <= bar, err
