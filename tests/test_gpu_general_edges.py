"""Line lengths without a compiled plan at the edges of what the other tests
cover: non-finite FP32 fields, with the general kernels in x, in y and in
both."""
import ctypes as C

import numpy as np
import pytest

from cases import interior, relmax, z_metrics

pytestmark = pytest.mark.gpu


def _solve32(api, plan, d):
    return api.lib.flutas_psolve_solve_f32(C.c_void_p(plan._h),
                                           C.cast(C.c_void_p(d.ptr), C.POINTER(C.c_float)))


@pytest.mark.parametrize("bad", [np.nan, np.inf])
@pytest.mark.parametrize("ng", [(36, 64, 20), (64, 300, 20), (90, 154, 20), (64, 32, 20)])
def test_f32_nonfinite_is_reported(api, oracle, ng, bad):
    """As flutas_psolve_solve_f32 states for the four-pass pipeline; a field
    without it solves on the same plan before and after."""
    _, _, dzci, dzfi, _, _ = z_metrics(oracle, ng[2], 0.0, 1.0)
    plan = api.PoissonPlan(ng, tuple(float(n) for n in ng), dzci, dzfi, "PPDDNN")
    f = np.zeros(tuple(n + 2 for n in ng), np.float32, order="F")
    f[1:-1, 1:-1, 1:-1] = np.random.default_rng(1).standard_normal(ng)
    g = f.copy(order="F")
    g[5, 7, 4] = bad
    for field, code in ((f, 0), (g, api.FLUTAS_ENONFINITE), (f, 0)):
        d = api.DeviceArray.from_host(field)
        assert _solve32(api, plan, d) == code
        assert np.all(np.isfinite(d.to_host())) == (code == 0)
    plan.destroy()


@pytest.mark.parametrize("bad", [np.nan, -np.inf])
@pytest.mark.parametrize("ng", [(36, 64, 20), (64, 300, 20), (90, 154, 20)])
def test_refined_nonfinite_gives_the_right_hand_side_back(api, oracle, ng, bad):
    """In place the field comes back bit for bit, halo included; out of place
    the right-hand side is not written."""
    _, _, dzci, dzfi, _, _ = z_metrics(oracle, ng[2], 0.0, 1.0)
    plan = api.PoissonPlan(ng, tuple(float(n) for n in ng), dzci, dzfi, "PPDDNN",
                           precision=api.FP32_REFINE, tol=1e-8)
    f = np.asfortranarray(np.random.default_rng(2).standard_normal([n + 2 for n in ng]))
    f[5, 7, 4] = bad
    d, p = api.DeviceArray.from_host(f), api.DeviceArray(f.shape)
    for call in (lambda: plan.solve(d), lambda: plan.solve_async(d), lambda: plan.solve_into(d, p)):
        with pytest.raises(api.FlutasError) as e:
            call()
        assert e.value.code == api.FLUTAS_ENONFINITE
        np.testing.assert_array_equal(d.to_host(), f)
    plan.destroy()


@pytest.mark.parametrize("ng", [(2, 2, 4), (6, 10, 4), (90, 2, 8), (2, 90, 6), (30, 30, 8), (360, 2, 4),
                                (2, 1000, 4), (30, 34, 8), (90, 30, 4), (60, 60, 10)])
@pytest.mark.parametrize("cbc", ["PPDDNN", "NDPPPP"])
def test_few_planes_match_oracle(api, oracle, ng, cbc):
    """Both sides of the rule for few values in few planes, FP64 and FP32
    fields, to the bounds of every length."""
    dzc, dzf, dzci, dzfi, _, _ = z_metrics(oracle, ng[2], 0.0, 1.1)
    dli = (ng[0] / 1.0, ng[1] / 0.8, ng[2] / 1.1)
    f = np.zeros(tuple(n + 2 for n in ng), order="F")
    f[1:-1, 1:-1, 1:-1] = np.random.default_rng(sum(ng)).standard_normal(ng).astype(np.float32)
    ref = f.copy(order="F")
    oracle.Solver(ng, dli, dzci, dzfi, cbc).solve(ref, pin_gauge=True)
    plan = api.PoissonPlan(ng, dli, dzci, dzfi, cbc)
    d, p = api.DeviceArray.from_host(f), api.DeviceArray(f.shape)
    p.zero()
    plan.solve_into(d, p)
    assert relmax(interior(p.to_host()), interior(ref)) <= 1e-12
    s = api.DeviceArray.from_host(np.asfortranarray(f.astype(np.float32)))
    assert _solve32(api, plan, s) == 0
    assert relmax(interior(s.to_host().astype(np.float64)), interior(ref)) <= 1e-4
    plan.destroy()


def _random_case(oracle, ng, cbc, seed):
    dzc, dzf, dzci, dzfi, _, _ = z_metrics(oracle, ng[2], 0.0, 1.1)
    dli = (ng[0] / 1.0, ng[1] / 0.8, ng[2] / 1.1)
    f = np.zeros(tuple(n + 2 for n in ng), order="F")
    f[1:-1, 1:-1, 1:-1] = np.random.default_rng(seed).standard_normal(ng).astype(np.float32)
    ref = f.copy(order="F")
    oracle.Solver(ng, dli, dzci, dzfi, cbc).solve(ref, pin_gauge=True)
    return f, interior(ref), dzci, dzfi, dli


@pytest.mark.parametrize("ng", [(90, 512, 18), (36, 512, 20), (254, 512, 6), (6, 512, 40)])
@pytest.mark.parametrize("cbc", ["NNDDNN", "PPNDPP"])
def test_general_x_with_a_blocked_work_field(api, oracle, ng, cbc):
    """512-point y lines keep the FP64 work field in blocks of up to 8 slabs (2
    for 90 and 254, 4 for 36): the general x passes write and read it."""
    f, ref, dzci, dzfi, dli = _random_case(oracle, ng, cbc, 5)
    plan = api.PoissonPlan(ng, dli, dzci, dzfi, cbc)
    d, p = api.DeviceArray.from_host(f), api.DeviceArray(f.shape)
    for n in (0, 1, 2):
        plan.set_zchunks(n)
        p.zero()
        plan.solve_into(d, p)
        assert relmax(interior(p.to_host()), ref) <= 1e-12
    plan.destroy()


@pytest.mark.parametrize("n", [22, 34, 254, 514, 1020, 1026, 2046])
@pytest.mark.parametrize("axis", [0, 1])
def test_f32_and_refined_long_and_prime_lengths(api, oracle, n, axis):
    """The FP32 chain at lists with a prime, tiles of fewer lines and slab groups
    of two and four columns a thread: FP32 fields to 1e-4, refined solves to
    their residual and 1e-9, as at every length.  20 lines: one full tile of 16
    and a partial one."""
    ng = (n, 20, 38) if axis == 0 else (6, n, 38)
    cbc = "NDPPNN" if axis == 0 else "PPDDPP"
    f, ref, dzci, dzfi, dli = _random_case(oracle, ng, cbc, n)
    plan = api.PoissonPlan(ng, dli, dzci, dzfi, cbc)
    s = api.DeviceArray.from_host(np.asfortranarray(f.astype(np.float32)))
    assert _solve32(api, plan, s) == 0
    assert relmax(interior(s.to_host().astype(np.float64)), ref) <= 1e-4
    plan.destroy()
    plan = api.PoissonPlan(ng, dli, dzci, dzfi, cbc, precision=api.FP32_REFINE, tol=1e-9)
    d, p = api.DeviceArray.from_host(f), api.DeviceArray(f.shape)
    p.zero()
    plan.solve_into(d, p)
    assert plan.stats()[1] <= 1e-9
    assert relmax(interior(p.to_host()), ref) <= 1e-9
    plan.destroy()


@pytest.mark.parametrize("ng", [(36, 60, 70), (22, 300, 40), (90, 520, 22)])
def test_chunk_counts_stay_within_what_is_asked(api, oracle, ng):
    _, _, dzci, dzfi, _, _ = z_metrics(oracle, ng[2], 0.0, 1.0)
    plan = api.PoissonPlan(ng, tuple(float(n) for n in ng), dzci, dzfi, "PPDDNN")
    assert 1 <= plan.set_zchunks(0) <= 8
    for n in range(1, 9):
        assert 1 <= plan.set_zchunks(n) <= n
    plan.destroy()
