"""The axis smoother against an FP64 FFT on the CPU."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def smoothed(f, sigma):
    F = np.fft.rfftn(f)
    for a, m in enumerate(f.shape):
        x = np.arange(m) * 2 * np.pi / m
        g = np.exp(-x ** 2 / (2 * sigma ** 2)) + np.exp(-(x - 2 * np.pi) ** 2 / (2 * sigma ** 2))
        G = (np.fft.rfft if a == 2 else np.fft.fft)(g / g.sum())
        F = F * G.reshape([-1 if d == a else 1 for d in range(3)])
    return np.fft.irfftn(F, s=f.shape, axes=(0, 1, 2))


@pytest.mark.parametrize("width", [0.02, 0.1, 0.5, 0.75, 1.0, 1.3, 2.0])
@pytest.mark.parametrize("n", [(32, 32, 32), (48, 80, 96), (128, 96, 160), (96, 128, 256)])
def test_smoother_radii_and_sizes(n, width):
    """Tap radii 1 to 24 (the compile-time ones and the general loop), two and eight points a thread, z lines
    that leave threads of a block without a point; FP64 sums, so the error is the result's rounding."""
    from glia_amd import rd
    print("case smooth", n, width, flush=True)
    f = np.random.default_rng(5).standard_normal(n).astype(np.float32)
    sigma = width * 2 * np.pi / n[0]
    s = rd.RDSolver(n)
    s.set_field(0, "work", f)
    s.smooth_field(0, "work", sigma)
    ref = smoothed(f.astype(np.float64), sigma)
    # three roundings to FP32 of values no larger than the input's: 3 x 2^-24 of the input norm
    assert np.linalg.norm(s.get_field(0, "work") - ref) < 3 * 2.0 ** -24 * np.linalg.norm(f)
    s.close()
