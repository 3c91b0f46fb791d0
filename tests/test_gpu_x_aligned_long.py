"""The inverse x pass of 1024-point lines from aligned lanes (outputs above 2 GB),
on a grid whose last tile of lines is partial: the residual of the solution stays
within rounding, 20 eps max|diagonal| max|p| / max|f|, and no halo value is
touched."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_large_output(api):
    ng, cbc = (1024, 66, 3800), "PPDDDD"
    dl = tuple(1.0 / n for n in ng)
    one = np.full(ng[2] + 2, 1.0 / dl[2])
    plan = api.PoissonPlan(ng, tuple(1.0 / d for d in dl), one, one, cbc)
    f = np.zeros([n + 2 for n in ng], order="F")
    rng = np.random.default_rng(3)
    for k in range(1, ng[2] + 1):
        f[1:-1, 1:-1, k] = rng.random(ng[:2], dtype=np.float32) - 0.5
    print(f"aligned stores {ng} {cbc}", flush=True)
    fd = api.DeviceArray.from_host(f)
    fmax = max(f.max(), -f.min())
    f[...] = 7.5
    pd = api.DeviceArray.from_host(f)
    plan.solve_into(fd, pd)
    rel = plan.residual(fd, pd)
    p = pd.to_host()
    for face in (p[0], p[-1], p[:, 0], p[:, -1], p[:, :, 0], p[:, :, -1]):
        np.testing.assert_array_equal(face, 7.5)
    q = p[1:-1, 1:-1, 1:-1]
    diag = sum(2.0 / d ** 2 for d in dl)
    bound = 20 * np.finfo(float).eps * diag * max(q.max(), -q.min()) / fmax
    assert rel <= bound, (rel, bound)
    plan.destroy()
