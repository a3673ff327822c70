"""div v at the departure points is interpolated by the first launch that needs it: whichever call, field
order and count that is, every field equals the one advected alone, bit for bit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("modes", [(1,), (2, 1), (1, 2, 1), (2,) * 8 + (1,), (1,) * 9, (2,) * 9])
def test_first_use_of_div_v(modes):
    import torch
    from glia_amd import adv
    from glia_amd.synth import reference_velocity
    n, dt = (32, 48, 64), 0.02
    print("case adv div", modes, flush=True)
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a, dtype=np.float32)).cuda()  # noqa: E731
    v = [dev(a) for a in reference_velocity(n)]
    rng = np.random.default_rng(2)
    f = [dev(rng.standard_normal(n)) for _ in modes]
    torch.cuda.synchronize()
    ref = []
    for x, m in zip(f, modes):
        s = adv.SemiLagrangianSolver(n)
        s.set_velocity(*v)
        y = x.clone()
        torch.cuda.synchronize()
        s.solve(y, dt, m)
        s.sync()
        ref.append(y)
        s.close()
    s = adv.SemiLagrangianSolver(n)
    s.set_velocity(*v)
    for _ in range(2):  # the second pass uses the kept interpolation
        out = s.advect(f, modes, dt)
        s.sync()
        for a, b in zip(out, ref):
            assert torch.equal(a, b)
    s.close()
