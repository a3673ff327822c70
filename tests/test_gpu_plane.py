"""The plane pass of the diffusion operator against an FP64 FFT on the CPU: every pair of sides (lines that
do not fill a wave, more waves in one layout than in the other, two planes a block) and the pairs next to the
rule's border, with a coefficient that vanishes on whole planes, on whole groups of 32 lines and on
parts of a group, and one that vanishes nowhere; every X length with planes left out."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def apply_d(k, f):
    n = f.shape
    w = [np.fft.fftfreq(n[0], 1.0 / n[0]), np.fft.fftfreq(n[1], 1.0 / n[1]), np.fft.rfftfreq(n[2], 1.0 / n[2])]
    for a, m in zip(w, n):
        a[np.abs(a) == m // 2] = 0.0
    w = [w[0][:, None, None], w[1][None, :, None], w[2][None, None, :]]
    F = np.fft.rfftn(f)
    out = sum(1j * a * np.fft.rfftn(k * np.fft.irfftn(1j * a * F, s=n, axes=(0, 1, 2))) for a in w)
    return np.fft.irfftn(out, s=n, axes=(0, 1, 2))


def fields(n, kind, rng):
    k = rng.uniform(0.1, 1.0, n)
    if kind == "sparse":
        k[: n[0] // 4] = 0.0             # whole planes
        k[:, : n[1] // 2] = 0.0          # whole groups of lines (at n1 >= 64) and a part of one
        k[n[0] // 2, n[1] - 3:] = 0.0
        k[:, :, n[2] // 2:] = 0.0        # half of every line
        k[n[0] // 4 + 1] = 0.0
        k[n[0] // 4 + 1, n[1] // 3, 5] = 0.7  # one nonzero in a plane
    if kind == "stripes":
        k[rng.random(n[0]) < 0.5] = 0.0  # scattered zero planes, in every word of their mask
    return k.astype(np.float32)


# every pair of sides that has a plane pass (within a factor of two)
SIDES = [(a, b) for a in (32, 48, 64, 80, 96, 128, 160, 192, 256) for b in (32, 64, 96, 128, 160, 192, 256)
         if max(a, b) <= 2 * min(a, b)]


@pytest.mark.parametrize("kind", ["dense", "sparse"])
@pytest.mark.parametrize("n", [(32, a, b) for a, b in SIDES] + [(48, 64, 64), (80, 128, 128), (48, 80, 160)])
def test_operator_on_planes(n, kind):
    from glia_amd import rd
    print("case plane", n, kind, flush=True)
    rng = np.random.default_rng([n[0], n[1], kind == "sparse"])
    s = rd.RDSolver(n, nmembers=2)
    f = [rng.standard_normal(n).astype(np.float32) for _ in range(2)]
    k = [fields(n, kind, rng), fields(n, "dense", rng)]  # the members' masks differ
    for m in range(2):
        s.set_field(m, "k", k[m])
        s.set_field(m, "work", f[m])
    s.apply_d("work", "ct")
    for m in range(2):
        ref = apply_d(k[m].astype(np.float64), f[m].astype(np.float64))
        err = np.linalg.norm(s.get_field(m, "ct") - ref) / np.linalg.norm(ref)
        # six transforms of log2(n) <= 24 levels in FP32: 24 eps = 1.4e-6 a transform at the worst
        assert err < 5e-6, err
    s.close()


@pytest.mark.parametrize("kind", ["stripes", "dense", "zero"])
@pytest.mark.parametrize("n", [(48, 160, 160), (64, 160, 160), (64, 128, 128), (80, 128, 128), (96, 128, 96), (128, 96, 96),
                               (160, 96, 96), (192, 64, 96), (256, 64, 64)])
def test_operator_with_planes_left_out(n, kind):
    """From 2^21 points the X passes leave out the rows of planes where k is zero: every X length, two planes
    a block of which one is zero, and rows that hold another field's values from the call before."""
    from glia_amd import rd
    print("case planes left out", n, kind, flush=True)
    assert 2 * n[0] * n[1] * n[2] >= 2 ** 21
    rng = np.random.default_rng([n[0], n[1], n[2], len(kind)])
    s = rd.RDSolver(n, nmembers=2)
    f = [rng.standard_normal(n).astype(np.float32) for _ in range(2)]
    k = [fields(n, kind, rng) if kind != "zero" else np.zeros(n, np.float32), fields(n, "stripes", rng)]
    for m in range(2):  # leaves other values in every row of the work slots
        s.set_field(m, "k", np.ones(n, np.float32))
        s.set_field(m, "work", 1e3 * f[1 - m])
    s.apply_d("work", "ct")
    for m in range(2):
        s.set_field(m, "k", k[m])
        s.set_field(m, "work", f[m])
    s.apply_d("work", "ct")
    for m in range(2):
        ref = apply_d(k[m].astype(np.float64), f[m].astype(np.float64))
        err = np.linalg.norm(s.get_field(m, "ct") - ref)
        # the bound of test_operator_on_planes; an operator that is zero gives exactly zero
        assert err <= 5e-6 * np.linalg.norm(ref), err
    s.close()


@pytest.mark.parametrize("kind", ["dense", "sparse"])
@pytest.mark.parametrize("n,plane", [((32, 32, 64), True), ((32, 32, 96), False), ((32, 64, 32), True), ((32, 80, 32), False),
                                     ((32, 128, 64), True), ((32, 160, 64), False), ((32, 48, 96), True),
                                     ((32, 48, 128), False), ((32, 128, 256), True), ((32, 96, 256), False)])
def test_operator_at_the_rules_border(n, plane, kind):
    """Sides within a factor of two take the plane pass, the next ones the separate passes: the same operator."""
    from glia_amd import rd
    print("case plane border", n, kind, flush=True)
    rng = np.random.default_rng([n[1], n[2], len(kind)])
    s = rd.RDSolver(n)
    s.set_coefficients(0, 0.05, 8.0)
    s.precFactor()
    f = rng.standard_normal(n).astype(np.float32)
    s.set_field(0, "work", f)
    s.profile(True)
    s.diffusion_solve("work", 0.01)
    prof = s.profile_get()
    s.profile(False)
    assert (prof["plane_div"][0] > 0) == plane and (prof["z_diff"][0] > 0) != plane
    k = fields(n, kind, rng)
    s.set_field(0, "k", k)
    s.set_field(0, "work", f)
    s.apply_d("work", "ct")
    ref = apply_d(k.astype(np.float64), f.astype(np.float64))
    err = np.linalg.norm(s.get_field(0, "ct") - ref) / np.linalg.norm(ref)
    assert err < 5e-6, err  # the bound of test_operator_on_planes
    s.close()


def test_zero_coefficient_and_a_field_written_after_creation():
    """All planes skipped gives exactly zero, and the skip follows a coefficient changed in place."""
    from glia_amd import rd
    n = (32, 64, 64)
    print("case plane zero", n, flush=True)
    rng = np.random.default_rng(3)
    s = rd.RDSolver(n)
    f = rng.standard_normal(n).astype(np.float32)
    s.set_field(0, "work", f)
    s.set_field(0, "k", np.zeros(n, np.float32))
    s.apply_d("work", "ct")
    assert not np.any(s.get_field(0, "ct"))
    k = fields(n, "dense", rng)
    s.set_field(0, "k", k)
    s.apply_d("work", "ct")
    ref = apply_d(k.astype(np.float64), f.astype(np.float64))
    assert np.linalg.norm(s.get_field(0, "ct") - ref) < 5e-6 * np.linalg.norm(ref)
    s.close()


def elastic(mu, lam, scr, avg):
    n = mu.shape
    w = [np.fft.fftfreq(n[0], 1.0 / n[0]), np.fft.fftfreq(n[1], 1.0 / n[1]), np.fft.rfftfreq(n[2], 1.0 / n[2])]
    for a, m in zip(w, n):
        a[np.abs(a) == m // 2] = 0.0
    w = [w[0][:, None, None], w[1][None, :, None], w[2][None, None, :]]
    r2c, c2r = np.fft.rfftn, lambda F: np.fft.irfftn(F, s=n, axes=(0, 1, 2))
    w2 = sum(a * a for a in w)

    def A(u):
        U = [r2c(c) for c in u]
        L = r2c(lam * c2r(1j * sum(a * F for a, F in zip(w, U))))
        S = [[r2c(mu * c2r(1j * (w[j] * U[i] + w[i] * U[j]))) for j in range(3)] for i in range(3)]
        return np.stack([c2r(1j * (sum(w[j] * S[i][j] for j in range(3)) + w[i] * L)) - scr * u[i] for i in range(3)])

    def B(f):
        F = [r2c(c) for c in f]
        s1, s2 = -avg[2] - avg[0] * w2, avg[0] + avg[1]
        c = s2 / (1.0 - w2 * s2 / s1) / s1 ** 2
        wf = sum(a * G for a, G in zip(w, F))
        return np.stack([c2r(F[d] / s1 + c * w[d] * wf) for d in range(3)])

    return A, B


@pytest.mark.parametrize("n", [(32, a, b) for a, b in SIDES] + [(64, 160, 96), (96, 160, 96), (96, 96, 192)])
def test_elasticity_on_planes(n):
    """Operator, preconditioner and a solve whose residual is measured with the FP64 operator; every
    pair of sides, and the mixes of fused and separate passes that launches of one and of three lanes take by how
    they fill the chip."""
    from glia_amd import elasticity
    from glia_amd.synth import tissue_and_tumor
    print("case plane elasticity", n, flush=True)
    c, wm, gm, csf, vt, bg = tissue_and_tumor(n)
    s = elasticity.ElasticitySolver(n)
    s.set_material(c, wm, gm, csf, vt, bg)
    mu, lam, scr, avg = s.material()
    A, B = elastic(*[a.astype(np.float64) for a in (mu, lam, scr)], avg)
    rng = np.random.default_rng(sum(n))
    u = rng.standard_normal((3,) + n).astype(np.float32)
    for got, ref in ((s.apply(u), A(u.astype(np.float64))), (s.precondition(u), B(u.astype(np.float64)))):
        err = np.linalg.norm(got - ref) / np.linalg.norm(ref)
        assert err < 5e-6, err  # as the diffusion operator's bound
    f = (-1e2 * np.stack(np.gradient(c, *[2 * np.pi / m for m in n]))).astype(np.float32)
    x, its, reason, _ = s.solve(f)
    f = f.astype(np.float64)
    res = np.linalg.norm(B(f - A(x.astype(np.float64)))) / np.linalg.norm(B(f))
    assert reason == "rtol" and res < 1.01e-3, (its, reason, res)
    s.close()
