"""pzl_get_kernel's rows: the 64-bit row rounded once, at every length, without
building a bank that the plan's searches do not read."""
import numpy as np
import pytest

import pyoracle as O

pytestmark = pytest.mark.gpu


# 32 harmonics at zmax 4 have lengths of 128 .. 2048, (200, 300, 16) adds 192 .. 1280
@pytest.mark.parametrize("zmax,wmax,numharm", [(4, 0, 32), (200, 300, 16)])
def test_rows_are_rounded_once(zmax, wmax, numharm):
    from prestozl_amd import binding as B
    N = 1 << 18
    kw = dict(N=N, dt=1e-4, numbins=N // 2, zmax=zmax, wmax=wmax, numharm=numharm, sigma=4.0, wmaxP=True)
    plan = B.Plan(B.make_config(**kw))
    held = plan.device_bytes()
    obs = O.create_accelobs(O.make_params(**kw))
    seen = set()
    for idx, (nh, hn) in enumerate(O.harmonics(obs)):
        h = plan.harms[idx]
        if h.fftlen in seen:
            continue
        seen.add(h.fftlen)
        wi = h.numw // 2  # w = 0: other rows come from a chirp of 32-bit samples
        for zi in sorted({0, h.numz // 3, h.numz - 1}):
            k64 = O.kernel(obs, nh, hn, zi, wi, O.FP64)
            got = plan.kernel(idx, wi * h.numz + zi).astype(np.complex128)
            # One rounding to 24 bits: half an ulp, 2^-24 of the value.  The two
            # 64-bit rows differ by the rounding of phases of up to 300 radians,
            # 5e-14 in each of up to 1000 response values below 0.1: 1e-13 in a
            # row's value (at most about 1) if they add at random, 5e-12 if in step.
            slack = 1e-11 * np.abs(k64).max()
            for g, k in ((got.real, k64.real), (got.imag, k64.imag)):
                assert np.all(np.abs(g - k) <= 2.0 ** -24 * np.abs(k) + slack), (h.fftlen, zi)
    assert any(n & (n - 1) for n in seen)
    assert plan.device_bytes() == held
    plan.close()
