"""x passes over line lengths with odd factors (a thread's share of a line and
of the column tiles differs with the length), FP64 and FP32, every x form, with
a ragged last tile of lines, against the FP64 oracle.

FP64 at the solve's 1e-12.  FP32 (one uncorrected FP32 solve): storage rounding
of 6e-8 a pass over five passes, bounded by 5e-6 of the field as a gross-error
bar; FP32_IR to its 1e-10 runs the refinement forms of the same kernels.
"""
import numpy as np
import pytest

from oracle import oracle as O
from pascal_poisson_fft_amd import api
from pascal_poisson_fft_amd.grid import make_axis

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("per", [False, True], ids=["N", "P"])
@pytest.mark.parametrize("n1", [10, 12, 24, 28, 48, 56, 96, 112, 120, 192, 240, 320, 384, 448, 480, 640, 768, 896, 960])
def test_x_forms_match_oracle(n1, per):
    n2, n3, L = 10, 14, (2.0, 3.0, 1.5)
    ax, ay = make_axis(n1, L[0], per), make_axis(n2, L[1], False)
    az = make_axis(n3, L[2], False, uniform=False, gamma=1.5)
    f = np.random.default_rng(n1).standard_normal((n3, n2, n1))
    f -= float(np.einsum("kji,k->", f, az.dx[1:n3 + 1])) / (az.dx[1:n3 + 1].sum() * n1 * n2)
    ref = O.solve(f, L, (per, False, False), ax.dmx, ay.dmx, az.dmx, az.dx)
    dev = api.Problem3D(f, ax, ay, az)
    args = (dev.rhs, dev.p, dev.dmx1, dev.dmx2, dev.dmx3, dev.dx3)
    try:
        for precision, bar in ((api.PPF_PREC_FP64, 1e-12), (api.PPF_PREC_FP32_IR, 5e-6)):
            plan = api.FFTPoisson(n1, n2, n3, L, (per, False, False), precision=precision, tol=1e-10)
            for form in (0, 1, 2, 3):
                plan.set_variants(form, 0, 0)
                dev.p.fill_zero()
                plan.solve_sweeps(*args, 0)
                api.sync()
                err = float(np.linalg.norm(dev.p.download() - ref) / np.linalg.norm(ref))
                assert err <= bar, (precision, form, err)
                if precision == api.PPF_PREC_FP32_IR:
                    plan.solve(*args)
                    api.sync()
                    err = float(np.linalg.norm(dev.p.download() - ref) / np.linalg.norm(ref))
                    assert err <= 1e-10, (form, err)
            plan.clean()
    finally:
        dev.free()
