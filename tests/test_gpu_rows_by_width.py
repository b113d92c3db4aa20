"""The correlation with each kernel row at the shortest transform its own
width allows (the last correlation group, the default) against the one with
every row of a harmonic at the harmonic's length: the same planes.

Either form's powers lie within 1e-5 of the 64-bit powers (relative, floor 1:
test_gpu_parity.py), so the two lie within 2e-5 of each other.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

TOL = 2e-5


def _spectrum(N, seed):
    rng = np.random.Generator(np.random.PCG64(seed))
    n = N // 2
    f = (rng.standard_normal(n) + 1j * rng.standard_normal(n)).astype(np.complex64)
    f[rng.integers(0, n, 40)] *= 20.0
    return f


def _plan(N, fft, zmax, wmax, numharm, **kw):
    from prestozl_amd import binding as B
    plan = B.Plan(B.make_config(N=N, dt=1e-4, numbins=N // 2, zmax=zmax, wmax=wmax, wmaxP=wmax > 0, numharm=numharm,
                                sigma=4.0, batchsize=3, **kw))
    plan.set_spectrum(fft)
    return plan


def _planes(plan, rstep, form):
    plan.set_corr_group(*form)
    return [plan.plane(rstep, i)[0] for i in range(len(plan.harms))]


def _width_form():
    from prestozl_amd import binding as B
    groups = B.corr_groups()
    assert groups[-1].startswith("rows by width")
    return len(groups) - 1, True


# every held length from 128 to 4096: the shortest windows (32 harmonics at
# zmax 4), kernels of one width (zmax 0), the 2048- and 4096-point fundamentals,
# a fractional first bin (r maps from tables, windows that start on half bins)
@pytest.mark.parametrize("N,zmax,wmax,numharm,kw", [
    (1 << 17, 4, 0, 32, {}), (1 << 17, 0, 0, 2, {}), (1 << 17, 60, 40, 8, {}), (1 << 18, 200, 300, 16, {}),
    (1 << 18, 200, 500, 16, {}), (1 << 17, 100, 100, 16, dict(rlo=1000.25))])
def test_planes_equal_whole_rows(N, zmax, wmax, numharm, kw):
    fft = _spectrum(N, zmax + wmax + numharm)
    plan = _plan(N, fft, zmax, wmax, numharm, **kw)
    assert plan.corr_group() == _width_form()  # the default
    last = plan.geom.nrsteps - 1
    for rstep in sorted({0, last // 2, last}):  # both ends of the band reach past the spectrum
        a = _planes(plan, rstep, _width_form())
        b = _planes(plan, rstep, (-1, False))
        for i, (x, y) in enumerate(zip(a, b)):
            err = np.max(np.abs(x - y) / np.maximum(y, 1.0))
            h = plan.harms[i]
            assert err < TOL, (rstep, h.harmnum, h.numharm, err)
    plan.close()


@pytest.mark.parametrize("bad", [np.nan, np.inf])
def test_not_finite_values_spread_as_far(bad):
    """A value that is not finite makes the powers NaN in the rsteps and
    harmonics whose whole segment holds it, not only in the rows that reach it;
    the others are as without it."""
    N = 1 << 17
    fft = _spectrum(N, 5)
    fft[20000] = bad
    plan = _plan(N, fft, 100, 100, 4)
    mid = int((20000 - plan.geom.rlo) // (plan.geom.corr_uselen // 2))
    seen = set()
    for rstep in range(mid - 2, mid + 3):
        a = _planes(plan, rstep, _width_form())
        b = _planes(plan, rstep, (-1, False))
        for x, y in zip(a, b):
            assert np.array_equal(np.isnan(x), np.isnan(y))
            assert not np.isinf(x).any()
            seen.add(bool(np.isnan(x).any()))
            ok = ~np.isnan(y)
            if ok.any():
                assert np.max(np.abs(x[ok] - y[ok]) / np.maximum(y[ok], 1.0)) < TOL
    assert seen == {True, False}
    plan.close()


@pytest.mark.parametrize("wmax,per_batch", [(300, 1), (500, 2)])
def test_statistics_of_the_launch_form(wmax, per_batch):
    """A search's statistics count the launches of the form in use (rows of more
    than 2048 points have a launch of their own) and the bank it reads."""
    N = 1 << 18
    plan = _plan(N, _spectrum(N, wmax), 200, wmax, 16)
    batches = -(-plan.geom.nrsteps // plan.launch()[0])
    st = plan.search()[1]
    assert (st["corr_launches"], st["group_launches"]) == (per_batch * batches, per_batch * batches)
    bank = plan.geom.bank_bytes  # the rows' by width
    plan.set_corr_group(-1)
    whole = plan.search()[1]
    assert (whole["corr_launches"], whole["group_launches"]) == (len(plan.fftlens()) * batches, 0)
    whole_bank = sum(8 * h.numw * h.numz * h.fftlen for h in plan.harms)
    assert whole_bank > bank
    # beside the banks the two forms differ by the segments, which both figures hold alike
    assert st["bytes_alg"] - st["bytes_alg_corr"] == whole["bytes_alg"] - whole["bytes_alg_corr"]
    segments = plan.geom.nrsteps * sum(4 * h.fftlen for h in plan.harms)
    planes = st["bytes_alg"] - st["bytes_alg_corr"]
    assert whole["bytes_alg_corr"] == pytest.approx(planes + segments + whole_bank, rel=1e-12)
    plan.close()
