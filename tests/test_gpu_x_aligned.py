"""Large FP64 outputs in lines of 512 and 1024 points (stored from lanes aligned
to memory lines) on grids whose last tile of lines is partial: the residual of
the solution stays within rounding, 20 eps max|diagonal| max|p| / max|f|, and no
halo value is touched."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ng,cbc", [((512, 130, 1024), "NNNNDD"), ((1024, 66, 1000), "PPDDDD")])
def test_large_output(api, ng, cbc):
    dl = (1.0 / ng[0], 1.0 / ng[1], 1.0 / ng[2])
    one = np.full(ng[2] + 2, 1.0 / dl[2])
    plan = api.PoissonPlan(ng, tuple(1.0 / d for d in dl), one, one, cbc)
    f = np.zeros([n + 2 for n in ng], order="F")
    f[1:-1, 1:-1, 1:-1] = np.random.default_rng(3).standard_normal(ng[::-1]).T
    print(f"aligned stores {ng} {cbc}", flush=True)
    fd, pd = api.DeviceArray.from_host(f), api.DeviceArray(f.shape)
    pd.upload(np.full(f.shape, 7.5, order="F"))
    plan.solve_into(fd, pd)
    rel = plan.residual(fd, pd)
    # the residual call reads the field alone: its halo is still 7.5
    p = pd.to_host()
    for face in (p[0], p[-1], p[:, 0], p[:, -1], p[:, :, 0], p[:, :, -1]):
        np.testing.assert_array_equal(face, 7.5)
    diag = sum(2.0 / d ** 2 for d in dl)
    bound = 20 * np.finfo(float).eps * diag * np.max(np.abs(p[1:-1, 1:-1, 1:-1])) / np.max(np.abs(f))
    assert rel <= bound, (rel, bound)
    plan.destroy()
