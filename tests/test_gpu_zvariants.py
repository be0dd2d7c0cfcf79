"""Every z-pass kernel shape, pinned with ppf_plan_set_zvariant, against the
FP64 oracle.

The autotuner may return these shapes, so each one must be correct on its own,
at z extents that stress its partitions (K rows a thread: 8, 12, 16, 20, 24, 28,
32, 48): 96, 240, 504 and 512 (whole last partitions of one K or another), 136,
144, 168 and 270 (a cut last partition, down to 2 rows), 768 (the projection
stream's extent), 1500 (above 1024, where the default is K = 32 and 8 columns)
-- and 2050, where an FP64 plan runs the one-thread-per-line Thomas.  Both z-row
layouts are covered: Neumann y (rows 1..n2m) and periodic y with Neumann x (R2C
columns, rows 0..n2m+1).

A shape that does not fit an extent (its partitions exceed the workgroup or its
rows the id's) is rejected with PPF_ERR_UNSUPPORTED, never run; the test records
which.

Tolerance: <= 1e-12 relative L2 of the ghosted solution against the oracle
for z lines of up to 1024 rows.  Longer stretched lines are worse conditioned
than that bar: the oracle's own FP64 Thomas on the pinned (0,0) mode of a
1500-row tanh-1.6 line differs from an 80-bit extended-precision solve by
5.5e-12 (7.0e-12 at 2050 rows), so two correct FP64 algorithms may differ by
that much; there the bar is 1e-11.  As a check against gross errors (a wrong
row or sign leaves a residual of order one) every solve must also leave an
FP64 relative residual <= max(1e-11, twice the oracle's own): on long
stretched lines the oracle's residual itself is about 2e-12, because the
operator's coefficients span several orders of magnitude.
"""
import numpy as np
import pytest

from oracle import oracle as O
from pascal_poisson_fft_amd import api
from pascal_poisson_fft_amd.grid import make_axis

pytestmark = pytest.mark.gpu

VARIANTS = list(range(1, 18))
UNSUPPORTED = -5


def _tol(n3):
    return 1e-12 if n3 <= 1024 else 1e-11


def _res_bar(f, ref, L, pbc, az):
    return max(1e-11, 2.0 * O.rel_residual(f, ref, L, pbc, az.dmx, az.dx))


def _case(n1, n2, n3, pbc, seed):
    L = (2.0, 3.0, 1.5)
    ax, ay = make_axis(n1, L[0], pbc[0]), make_axis(n2, L[1], pbc[1])
    az = make_axis(n3, L[2], False, uniform=False, gamma=1.6)
    f = np.random.default_rng(seed).standard_normal((n3, n2, n1))
    w = az.dx[1:n3 + 1]
    f -= float(np.einsum("kji,k->", f, w)) / (w.sum() * n1 * n2)
    ref = O.solve(f, L, (pbc[0], pbc[1], False), ax.dmx, ay.dmx, az.dmx, az.dx)
    return L, ax, ay, az, f, ref


@pytest.mark.parametrize("pbc", [(False, False), (False, True)], ids=["NN", "NP"])
@pytest.mark.parametrize("n3", [96, 136, 144, 168, 240, 270, 504, 512, 768, 1500])
def test_every_zvariant_matches_oracle(pbc, n3):
    n1, n2 = 24, 16
    L, ax, ay, az, f, ref = _case(n1, n2, n3, pbc, seed=n3 + 7 * pbc[1])
    plan = api.FFTPoisson(n1, n2, n3, L, (pbc[0], pbc[1], False))
    dev = api.Problem3D(f, ax, ay, az)
    res_bar = _res_bar(f, ref, L, pbc, az)
    ran, rejected = [], []
    try:
        for v in VARIANTS:
            print(f"n3m={n3} pbc={pbc} zvariant={v}", flush=True)
            plan.set_zvariant(v)
            dev.p.fill_zero()
            try:
                plan.solve(dev.rhs, dev.p, dev.dmx1, dev.dmx2, dev.dmx3, dev.dx3)
            except api.PPFError as e:
                assert e.code == UNSUPPORTED, e
                rejected.append(v)
                continue
            api.sync()
            got = dev.p.download()
            err = float(np.linalg.norm(got - ref) / np.linalg.norm(ref))
            res = plan.residual(dev.rhs, dev.p, dev.dmx3, dev.dx3)
            assert err <= _tol(n3) and res <= res_bar, (v, err, res, res_bar)
            ran.append(v)
    finally:
        dev.free()
        plan.clean()
    print(f"  ran {ran}; unsupported at this extent {rejected}")
    # the default shape of this extent and the one-thread-per-line kernel run
    assert (3 if n3 <= 1024 else 4) in ran and 6 in ran


@pytest.mark.parametrize("pbc", [(False, False), (True, False)], ids=["NN", "PN"])
def test_long_z_lines_use_one_thread_per_line(pbc):
    """n3m = 2050 > 2048: the default is the one-thread-per-line Thomas."""
    n1, n2, n3 = 16, 8, 2050
    print(f"n3m={n3} pbc={pbc} default z kernel", flush=True)
    L, ax, ay, az, f, ref = _case(n1, n2, n3, pbc, seed=3)
    got = api.solve_host(f, ax, ay, az)
    err = float(np.linalg.norm(got - ref) / np.linalg.norm(ref))
    res = O.rel_residual(f, got, L, (pbc[0], pbc[1]), az.dmx, az.dx)
    bar = _res_bar(f, ref, L, pbc, az)
    assert err <= _tol(n3) and res <= bar, (err, res, bar)


@pytest.mark.parametrize("pbc", [(False, False), (True, True), (True, False), (False, True)],
                         ids=["NN", "PP", "PN", "NP"])
@pytest.mark.parametrize("n1,n2,n3", [(512, 64, 8), (64, 512, 8), (160, 96, 12), (24, 1024, 4), (1024, 16, 4)])
def test_xy_variants_match_oracle(pbc, n1, n2, n3):
    """Every x- and y-pass variant the tuner can pick (threads per line: one
    butterfly per stage, or half the threads with two; x also without the
    register prefetch, on a persistent grid or one workgroup per tile) against
    the oracle, at 1e-12, for every boundary branch."""
    L, ax, ay, az, f, ref = _case(n1, n2, n3, pbc, seed=n1 + n2 + n3)
    plan = api.FFTPoisson(n1, n2, n3, L, (pbc[0], pbc[1], False))
    dev = api.Problem3D(f, ax, ay, az)
    try:
        for xv, yv in ((0, 1), (1, 0), (1, 1), (2, 0), (2, 1), (3, 0), (3, 1)):
            print(f"{n1}x{n2}x{n3} pbc={pbc} xv={xv} yv={yv}", flush=True)
            plan.set_variants(xv, yv, 0)
            assert plan.variants() == (xv, yv, 0)
            dev.p.fill_zero()
            plan.solve(dev.rhs, dev.p, dev.dmx1, dev.dmx2, dev.dmx3, dev.dx3)
            api.sync()
            err = float(np.linalg.norm(dev.p.download() - ref) / np.linalg.norm(ref))
            assert err <= 1e-12, (xv, yv, err)
    finally:
        dev.free()
        plan.clean()


@pytest.mark.parametrize("pbc", [(False, False), (True, False)], ids=["NN", "PN"])
def test_split_x_variants_match_oracle(pbc):
    """The x-forward and x-inverse passes on different forms (variants value
    f + 16 i: forward f, inverse i), as the tuner may pick them, against the
    oracle at 1e-12; the value reads back as set, and a pair that is not a
    valid split is rejected."""
    n1, n2, n3 = 512, 32, 8
    L, ax, ay, az, f, ref = _case(n1, n2, n3, pbc, seed=11)
    plan = api.FFTPoisson(n1, n2, n3, L, (pbc[0], pbc[1], False))
    dev = api.Problem3D(f, ax, ay, az)
    try:
        for xf, xi in ((2, 3), (3, 2), (0, 3), (3, 0)):
            code = xf + 16 * xi
            print(f"{n1}x{n2}x{n3} pbc={pbc} x forward {xf} inverse {xi}", flush=True)
            plan.set_variants(code, 0, 0)
            assert plan.variants() == (code, 0, 0)
            dev.p.fill_zero()
            plan.solve(dev.rhs, dev.p, dev.dmx1, dev.dmx2, dev.dmx3, dev.dx3)
            api.sync()
            err = float(np.linalg.norm(dev.p.download() - ref) / np.linalg.norm(ref))
            assert err <= 1e-12, (xf, xi, err)
        for bad in (4, 1 + 16, 5 + 16, 2 + 16 * 4, -1):
            with pytest.raises(api.PPFError):
                plan.set_variants(bad, 0, 0)
    finally:
        dev.free()
        plan.clean()


@pytest.mark.parametrize("xv", [2, 3])
@pytest.mark.parametrize("pbc", [(False, False), (True, False)], ids=["NN", "PN"])
def test_x_variant_without_prefetch_fp32_ir(pbc, xv):
    """The refinement forms of the x passes (residual read in place, correction
    added into P) in the variants without the register prefetch (persistent
    grid, one workgroup per tile): FP32_IR reaches 1e-10 and matches the oracle
    to 1e-10."""
    n1, n2, n3 = 512, 64, 8
    L, ax, ay, az, f, ref = _case(n1, n2, n3, pbc, seed=7)
    plan = api.FFTPoisson(n1, n2, n3, L, (pbc[0], pbc[1], False), precision=api.PPF_PREC_FP32_IR, tol=1e-10)
    dev = api.Problem3D(f, ax, ay, az)
    try:
        plan.set_variants(xv, 0, 0)
        st = plan.solve(dev.rhs, dev.p, dev.dmx1, dev.dmx2, dev.dmx3, dev.dx3)
        api.sync()
        err = float(np.linalg.norm(dev.p.download() - ref) / np.linalg.norm(ref))
        assert st.rel_residual <= 1e-10 and err <= 1e-10, (st.sweeps, st.rel_residual, err)
    finally:
        dev.free()
        plan.clean()


def test_tuner_caches_per_shape_and_keeps_parity():
    """The tuner picks one variant per pass; a second plan of the same shape
    gets the same picks from the cache; the tuned solve matches the oracle."""
    n1, n2, n3, pbc = 96, 64, 40, (True, False)
    L, ax, ay, az, f, ref = _case(n1, n2, n3, pbc, seed=5)
    dev = api.Problem3D(f, ax, ay, az)
    plans = [api.FFTPoisson(n1, n2, n3, L, (pbc[0], pbc[1], False)) for _ in range(2)]
    try:
        args = (dev.rhs, dev.p, dev.dmx1, dev.dmx2, dev.dmx3, dev.dx3)
        z = plans[0].tune(*args)
        v = plans[0].variants()
        print(f"tuned variants {v}", flush=True)
        xf, xi = (v[0], v[0]) if v[0] < 4 else (v[0] % 16, v[0] // 16)
        assert v[2] == z and 0 <= xf < 4 and 0 <= xi < 4 and v[1] in (0, 1) and z > 0
        assert plans[1].tune(*args) == z and plans[1].variants() == v
        for pl in plans:
            dev.p.fill_zero()
            pl.solve(*args)
            api.sync()
            assert float(np.linalg.norm(dev.p.download() - ref) / np.linalg.norm(ref)) <= 1e-12
    finally:
        for pl in plans:
            pl.clean()
        dev.free()


@pytest.mark.parametrize("n3", [1026, 1400, 1536, 2050, 2544])
def test_tuned_long_lines_keep_their_accuracy(n3):
    """FP64 lines over 1024 rows: the tuner does not trade accuracy for time.
    K = 48 is the fastest shape there, and on these (uniform, periodic x and y)
    up to 2e-11 away from an 80-bit z solve at 1536 rows and 4e-11 at 2050,
    where K = 24 and 32 and one thread per line stay within the 1e-11 of lines
    this long.  Over 2048 rows the tuned plan runs what an untuned one does."""
    n1, n2, L = 16, 96, (2.0, 2.0, 2.0)
    ax, ay, az = make_axis(n1, L[0], True), make_axis(n2, L[1], True), make_axis(n3, L[2], False)
    f = np.random.default_rng(0).standard_normal((n3, n2, n1))
    f -= f.mean()
    plan = api.FFTPoisson(n1, n2, n3, L, (True, True, False))
    dev = api.Problem3D(f, ax, ay, az)
    args = (dev.rhs, dev.p, dev.dmx1, dev.dmx2, dev.dmx3, dev.dx3)
    try:
        plan.solve(*args)
        api.sync()
        default = dev.p.download()
        v = plan.tune(*args)
        print(f"n3m={n3} tuned z shape {v}", flush=True)
        dev.p.fill_zero()
        plan.solve(*args)
        api.sync()
        got = dev.p.download()
    finally:
        dev.free()
        plan.clean()
    if n3 > 2048:
        assert v == 6 and np.array_equal(got, default)
        return
    assert v in (4, 13)
    ref = O.solve(f, L, (True, True, False), ax.dmx, ay.dmx, az.dmx, az.dx)
    assert float(np.linalg.norm(got - ref) / np.linalg.norm(ref)) <= 1e-11


def _periodic_z(n1, n2, n3, pbc, precision=api.PPF_PREC_FP64):
    L = (2.0, 3.0, 1.5)
    ax, ay, az = make_axis(n1, L[0], pbc[0]), make_axis(n2, L[1], pbc[1]), make_axis(n3, L[2], True)
    f = np.random.default_rng(n1 + n3).standard_normal((n3, n2, n1))
    f -= f.mean()
    ref = O.solve(f, L, (pbc[0], pbc[1], True), ax.dmx, ay.dmx, az.dmx, az.dx)
    return api.FFTPoisson(n1, n2, n3, L, (pbc[0], pbc[1], True), precision=precision), api.Problem3D(f, ax, ay, az), ref


def _pinned(plan, dev, v):
    plan.set_zvariant(v)
    dev.p.fill_zero()
    plan.solve_sweeps(dev.rhs, dev.p, dev.dmx1, dev.dmx2, dev.dmx3, dev.dx3, 0)
    api.sync()
    return dev.p.download()


def test_periodic_z_runs_the_pinned_shape():
    """With periodic z an id means its own shape up to its rows, as with walls:
    the bits of the default where the default is that shape (20 rows by 16
    columns at 200 rows of a large grid), not those of shape 3.  Past its rows
    it stands for shape 3, or 4 over 1024 rows."""
    plan, dev, ref = _periodic_z(160, 120, 200, (True, False))
    try:
        default, k20, k32 = (_pinned(plan, dev, v) for v in (0, 7, 3))
    finally:
        dev.free()
        plan.clean()
    assert np.linalg.norm(default - ref) <= 1e-12 * np.linalg.norm(ref)
    assert np.array_equal(k20, default) and not np.array_equal(k20, k32)
    for n3, ids, same in ((600, (7, 8, 11), 3), (1030, (7, 9, 10, 17), 4)):
        plan, dev, _ = _periodic_z(16, 12, n3, (False, False))
        try:
            want = _pinned(plan, dev, same)
            for v in ids:
                assert np.array_equal(_pinned(plan, dev, v), want), (n3, v)
        finally:
            dev.free()
            plan.clean()


@pytest.mark.parametrize("n3", [30, 270, 512, 1500, 2544])
def test_every_zvariant_fp32(n3):
    """The same shapes on FP32 workspaces (one solve without corrections), up
    to the last rows K = 48 takes: storage rounding of 6e-8 a pass over five
    passes, bounded by 5e-6 as a gross-error bar."""
    n1, n2, pbc = 24, 16, (True, False)
    L, ax, ay, az, f, ref = _case(n1, n2, n3, pbc, seed=n3)
    plan = api.FFTPoisson(n1, n2, n3, L, (True, False, False), precision=api.PPF_PREC_FP32_IR)
    dev = api.Problem3D(f, ax, ay, az)
    ran = []
    try:
        for v in VARIANTS:
            try:
                got = _pinned(plan, dev, v)
            except api.PPFError as e:
                assert e.code == UNSUPPORTED, e
                continue
            err = float(np.linalg.norm(got - ref) / np.linalg.norm(ref))
            assert err <= 5e-6, (v, err)
            ran.append(v)
    finally:
        dev.free()
        plan.clean()
    assert {6, 14} <= set(ran)


@pytest.mark.parametrize("pbc", [(False, False), (True, True), (True, False), (False, True)],
                         ids=["NN", "PP", "PN", "NP"])
@pytest.mark.parametrize("n3", [8, 30, 96, 200, 256, 270, 512, 768, 1022])
def test_every_zvariant_periodic_z(pbc, n3):
    """Every shape that takes these rows with periodic z: whole last partitions
    and cut ones for each K, the wrapped end planes of z among the compared
    values (an FP64 solve writes them in the z pass).  1e-12 up to 270 rows and
    1e-11 above: on these uniform lines the oracle's FP64 cyclic Thomas is off
    an 80-bit z solve by 1.2e-12 at 256 rows already, 4.3e-12 at 512 and
    1.3e-11 at 768."""
    plan, dev, ref = _periodic_z(24, 16, n3, pbc)
    ran = []
    try:
        for v in VARIANTS:
            try:
                got = _pinned(plan, dev, v)
            except api.PPFError as e:
                assert e.code == UNSUPPORTED, e
                continue
            err = float(np.linalg.norm(got - ref) / np.linalg.norm(ref))
            ends = np.abs(got[[0, -1]] - got[[-2, 1]]).max() / np.abs(ref).max()
            print(f"n3m={n3} pbc={pbc} zvariant={v} {err:.1e} {ends:.1e}", flush=True)
            assert err <= (1e-12 if n3 <= 270 else 1e-11) and ends <= 1e-13, (v, err, ends)
            ran.append(v)
    finally:
        dev.free()
        plan.clean()
    assert {3, 6, 9, 10} <= set(ran)
