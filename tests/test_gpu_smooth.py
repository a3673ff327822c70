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


@pytest.mark.parametrize("offset", [0, 1])
@pytest.mark.parametrize("width", [0.1, 0.3, 1.0, 1.3])
@pytest.mark.parametrize("n", [(16, 17, 18), (31, 33, 34), (45, 50, 77), (20, 24, 1028), (91, 109, 122)])
def test_smoother_any_length_and_alignment(n, width, offset):
    """Caller-owned fields of any length: groups of points that end short, lines that are no multiple of four
    points or longer than a block, axes too short for the shared windows, fields off the 16-byte grid; nothing
    is written past the field."""
    import ctypes
    import torch
    from glia_amd import _lib
    print("case smooth any", n, width, offset, flush=True)
    L = _lib.load()
    ng = n[0] * n[1] * n[2]
    f = np.random.default_rng(7).standard_normal(n).astype(np.float32)
    fin, fout = torch.zeros(ng + 8, device="cuda"), torch.full((ng + 8,), 7.0, device="cuda")
    fin[offset:offset + ng] = torch.from_numpy(f.ravel()).cuda()
    torch.cuda.synchronize()
    sigma = width * 2 * np.pi / max(n)
    err = ctypes.create_string_buffer(256)
    rc = L.glia_rd_smooth_noalloc((ctypes.c_int * 3)(*n), ctypes.c_void_p(fin.data_ptr() + 4 * offset),
                                  ctypes.c_void_p(fout.data_ptr() + 4 * offset), float(sigma), None, err, 256)
    assert rc == 0, err.value
    torch.cuda.synchronize()
    out = fout.cpu().numpy()
    assert np.all(out[:offset] == 7.0) and np.all(out[offset + ng:] == 7.0)
    ref = smoothed(f.astype(np.float64), sigma)
    got = out[offset:offset + ng].reshape(n)
    assert np.linalg.norm(got - ref) < 3 * 2.0 ** -24 * np.linalg.norm(f)
