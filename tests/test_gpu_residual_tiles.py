"""Residual tiles (64 cells of a wave, TY rows, kz planes) and the ghost layers
re-derived after refinement, at extents where a wave, a row block or a plane
block is cut short; on 256 CUs the last three take blocks of 4 rows by 8 planes,
2 by 8 and 8 by 16, the smaller ones 2 by 4.

The residual is a sum of squares of FP64 differences: against the oracle's, on a
random iterate, 1e-12 relative (as in the other residual tests).  The ghost
layers are the same few products of the interior cells in another kernel, so
they equal numpy's to a few roundings of the largest value: 1e-14.
"""
import numpy as np
import pytest

from oracle import oracle as O
from pascal_poisson_fft_amd import api
from pascal_poisson_fft_amd.grid import make_axis

pytestmark = pytest.mark.gpu

BCS = [(False, False), (True, True), (True, False), (False, True)]


def _axes(n, pbc):
    return (make_axis(n[0], 2.0, pbc[0]), make_axis(n[1], 3.0, pbc[1]),
            make_axis(n[2], 1.5, pbc[2], uniform=pbc[2], gamma=1.5))


@pytest.mark.parametrize("pbc", BCS, ids=["NN", "PP", "PN", "NP"])
@pytest.mark.parametrize("n", [(8, 8, 2), (10, 10, 6), (64, 10, 34), (80, 24, 18), (128, 12, 66), (320, 14, 10),
                               (192, 192, 40), (480, 240, 98), (480, 30, 300),
                               (480, 240, 290)])
def test_residual_tiles_match_oracle(n, pbc):
    ax, ay, az = _axes(n, pbc + (False,))
    rng = np.random.default_rng(sum(n))
    f, P = rng.standard_normal(n[::-1]), rng.standard_normal((n[2] + 2, n[1] + 2, n[0] + 2))
    plan = api.FFTPoisson(*n, (ax.L, ay.L, az.L), pbc + (False,))
    dev = api.Problem3D(f, ax, ay, az)
    try:
        dev.p.upload(P)
        got = plan.residual(dev.rhs, dev.p, dev.dmx3, dev.dx3)
        ref = O.rel_residual(f, P, (ax.L, ay.L, az.L), pbc, az.dmx, az.dx)
        assert abs(got - ref) <= 1e-12 * ref, (got, ref)
    finally:
        dev.free()
        plan.clean()


@pytest.mark.parametrize("pz", [False, True], ids=["wall_z", "periodic_z"])
@pytest.mark.parametrize("pbc", BCS, ids=["NN", "PP", "PN", "NP"])
@pytest.mark.parametrize("n", [(8, 8, 4), (48, 20, 14), (96, 128, 36)])
def test_refined_ghost_layers(n, pbc, pz):
    axes = _axes(n, pbc + (pz,))
    f = np.random.default_rng(sum(n)).standard_normal(n[::-1])
    w = axes[2].dx[1:n[2] + 1]
    f -= float(np.einsum("kji,k->", f, w)) / (w.sum() * n[0] * n[1])
    plan = api.FFTPoisson(*n, tuple(a.L for a in axes), pbc + (pz,), precision=api.PPF_PREC_FP32_IR, tol=1e-10)
    dev = api.Problem3D(f, *axes)
    try:
        st = plan.solve(dev.rhs, dev.p, dev.dmx1, dev.dmx2, dev.dmx3, dev.dx3)
        api.sync()
        got = dev.p.download()
    finally:
        dev.free()
        plan.clean()
    assert st.sweeps >= 1
    want = got.copy()
    for wrap in (False, True):  # walls along x, y, z, then wraps along x, y, z
        for axis, a in ((2, axes[0]), (1, axes[1]), (0, axes[2])):
            if a.pbc != wrap:
                continue
            v, m, d = np.moveaxis(want, axis, 0), a.nm, a.dmx
            if wrap:
                v[0], v[m + 1] = v[m], v[1]
            else:
                for g, i, j, p, q in ((0, 1, 2, d[1], d[2]), (m + 1, m, m - 1, d[m + 1], d[m])):
                    s = (p + q) ** 2
                    v[g] = s / (s - p * p) * v[i] - p * p / (s - p * p) * v[j]
    assert np.abs(got - want).max() <= 1e-14 * np.abs(want).max()


@pytest.mark.parametrize("n", [(16, 12, 10), (96, 64, 40)])
def test_first_correction_launched_ahead_of_its_test(n):
    """Below a tol of 1e-9 the first correction is launched with its test, gated
    by it: the bits and the sweep count of the solve that waits for the test
    (a tol just above), none for a zero or a NaN right-hand side, and further
    sweeps, or a miss, where one is not enough."""
    axes = _axes(n, (False, True, False))
    f = np.random.default_rng(sum(n)).standard_normal(n[::-1])
    w = axes[2].dx[1:n[2] + 1]
    f -= float(np.einsum("kji,k->", f, w)) / (w.sum() * n[0] * n[1])

    def run(rhs, tol, sweeps=8):
        plan = api.FFTPoisson(*n, tuple(a.L for a in axes), (False, True, False), precision=api.PPF_PREC_FP32_IR,
                              tol=tol, max_sweeps=sweeps)
        dev = api.Problem3D(rhs, *axes)
        try:
            st = plan.solve(dev.rhs, dev.p, dev.dmx1, dev.dmx2, dev.dmx3, dev.dx3, allow_not_converged=True)
            api.sync()
            return dev.p.download(), st.sweeps, st.rel_residual
        finally:
            dev.free()
            plan.clean()

    waits, ahead = run(f, 1.01e-9), run(f, 0.99e-9)
    assert ahead[1] == waits[1] == 1 and ahead[2] == waits[2] <= 0.99e-9
    np.testing.assert_array_equal(ahead[0], waits[0])
    assert run(f, 1e-30, 1)[1:] == waits[1:]  # the cap ends it after one, above tol
    more = run(f, 1e-30, 3)
    assert more[1] == 3 and more[2] <= waits[2]
    zero = run(np.zeros_like(f), 1e-10)
    assert zero[1:] == (0, 0.0) and not zero[0].any()
    g = f.copy()
    g[0, 0, 0] = np.nan
    bad = run(g, 1e-10)
    assert bad[1] == 0 and np.isnan(bad[2])
