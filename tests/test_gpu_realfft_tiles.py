"""realfft at the lengths of its compiled four-step tiles and their edges."""
import numpy as np
import pytest

from prestozl_amd import binding as B

pytestmark = pytest.mark.gpu


# n/2 = M1 * M2 as the library splits it
@pytest.mark.parametrize("M1,M2", [
    (256, 128),    # compiled columns, run-time rows
    (256, 243),    # an odd row count: tiles of one column
    (256, 256), (512, 256), (512, 512), (1024, 512), (1024, 1024), (2048, 1024), (2048, 2048), (4096, 2048),
    (288, 256),    # run-time columns, compiled rows
    (1056, 1000),  # run-time passes, tiles of 8, a last partial round of threads
])
def test_against_float64(M1, M2):
    n = 2 * M1 * M2
    x = np.random.default_rng(M1 + M2).standard_normal(n).astype(np.float32)
    ref = np.fft.rfft(x.astype(np.float64))
    packed = ref[:-1].copy()
    packed[0] = ref[0].real + 1j * ref[-1].real
    # Each of the log2 n radix-2 levels rounds a value a few times to 2^-24 of
    # its size; errors add at worst linearly: 4 roundings per level of the rms,
    # and 6 sigma for the largest of up to 2^24 values.
    tol = 2.0 ** -24 * 4 * np.log2(n)
    got = np.asarray(B.realfft(x, -1)).view(np.complex64).astype(np.complex128)
    d = np.abs(got - packed)
    rms = np.sqrt(np.mean(np.abs(packed) ** 2))
    assert np.sqrt(np.mean(d ** 2)) <= tol * rms
    assert d.max() <= 6 * tol * rms
    back = np.asarray(B.realfft(packed.astype(np.complex64).view(np.float32), 1)).astype(np.float64)
    d = np.abs(back - x)
    assert np.sqrt(np.mean(d ** 2)) <= tol
    assert d.max() <= 6 * tol
