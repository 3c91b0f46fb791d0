"""The FP32 solve (flutas_psolve_solve_f32) on an FP64 plan in z chunks of
its own: whole slabs (set_zchunks(1)), the plan's default and every count
the grid allows, against the FP64 oracle (1e-4 of max|p|, the bound of FP32
fields) and against the whole-slab walk (2e-5: both round the stored field to
FP32 at the same points).  The FP64 solve of the same plan keeps its own
tables (1e-12 of the oracle)."""
import ctypes as C

import numpy as np
import pytest

from cases import gauge_free, interior, relmax, z_metrics

pytestmark = pytest.mark.gpu

CASES = [
    ((64, 32, 96), "PPPPNN", 1.5),
    ((48, 32, 70), "PPPPDD", 1.2),
    ((32, 64, 50), "NNDDPP", 0.0),   # cyclic z, a partial last group
    ((32, 512, 40), "PPPPNN", 1.5),  # blocked FP64 work field, plane-major FP32
]


def _case(oracle, ng, cbc, alpha):
    dzc, dzf, dzci, dzfi, _, _ = z_metrics(oracle, ng[2], alpha, 1.0)
    dli = (ng[0] / 6.0, ng[1] / 3.0, float(ng[2]))
    g = np.random.default_rng(sum(ng)).standard_normal(ng)
    if "D" not in cbc:
        w = dzf[1:ng[2] + 1][None, None, :]
        g -= np.sum(g * w) / (np.sum(w) * ng[0] * ng[1])
    f = np.zeros(tuple(n + 2 for n in ng), order="F")
    f[1:-1, 1:-1, 1:-1] = g.astype(np.float32)
    ref = f.copy(order="F")
    oracle.Solver(ng, dli, dzci, dzfi, cbc).solve(ref, pin_gauge=True)
    return f, ref, dzci, dzfi, dli


def _solve32(api, plan, d):
    rc = api.lib.flutas_psolve_solve_f32(C.c_void_p(plan._h),
                                         C.cast(C.c_void_p(d.ptr), C.POINTER(C.c_float)))
    assert rc == 0, api.lib.flutas_last_error().decode()


@pytest.mark.parametrize("ng,cbc,alpha", CASES)
def test_f32_chunks_on_fp64_plan(api, oracle, ng, cbc, alpha):
    f, ref, dzci, dzfi, dli = _case(oracle, ng, cbc, alpha)
    f32 = np.asfortranarray(f.astype(np.float32))
    free = gauge_free if "D" not in cbc else (lambda a: a)
    plan = api.PoissonPlan(ng, dli, dzci, dzfi, cbc)
    fd, pd = api.DeviceArray.from_host(f), api.DeviceArray(f.shape)
    whole = None
    for n in (1, 0, 2, 3, 4, 5, 6, 8):
        if whole is not None or n == 1:
            plan.set_zchunks(n)
        print(f"f32 chunks asked {n} {ng} {cbc}", flush=True)
        d = api.DeviceArray.from_host(f32)
        _solve32(api, plan, d)
        got = interior(d.to_host().astype(np.float64))
        if whole is None:
            whole = got
        assert relmax(free(got), free(interior(ref))) <= 1e-4
        assert relmax(free(got), free(whole)) <= 2e-5, n
        plan.solve_into(fd, pd)
        assert relmax(free(interior(pd.to_host())), free(interior(ref))) <= 1e-12, n
    plan.destroy()
