"""Line lengths without a compiled plan on the four-pass pipeline (the
kernels of general.hip, src/solver_cpu.f90:20-115 and src/fft.f90:233-291):
against the C FP64 oracle at the edges of their tiles and groups, in x and in
y, for every boundary pair.

Tolerances: the FP64 solve to 1e-12 relative max-norm, as every length (the
longest direct sum here has 257 terms, 257 eps = 6e-14); refined solves to
their 1e-10 residual and 1e-9 of the oracle; FP32 fields to 1e-4."""
import ctypes as C

import numpy as np
import pytest

from cases import gauge_free, interior, relmax, z_metrics

pytestmark = pytest.mark.gpu

LENGTHS = [
    2, 4, 6, 10,            # one to five complex points
    14, 18, 22, 26, 30,     # one odd radix
    34, 62, 254,            # primes beyond the butterflies: 17, 31, 127
    60, 66, 90, 154,        # mixed radices; one and two columns past a wave
    250, 258, 360,          # groups of 16 and 8 planes; 43
    510, 514, 528, 1020,    # one and two columns per thread; 257
    1026, 1200, 2046,       # four columns per thread
]
PAIRS = ["PP", "NN", "DD", "ND", "DN"]


def _case(oracle, ng, cbc, alpha, seed):
    lengths = (1.0, 0.8, 1.1)
    dzc, dzf, dzci, dzfi, _, _ = z_metrics(oracle, ng[2], alpha, lengths[2])
    dli = tuple(n / l for n, l in zip(ng, lengths))
    g = np.random.default_rng(seed).standard_normal(ng)
    singular = all(c in "PN" for c in cbc)
    if singular:
        w = dzf[1:ng[2] + 1][None, None, :]
        g -= np.sum(g * w) / (np.sum(w) * ng[0] * ng[1])
    f = np.zeros(tuple(n + 2 for n in ng), order="F")
    f[1:-1, 1:-1, 1:-1] = g
    s = oracle.Solver(ng, dli, dzci, dzfi, cbc)
    ref = f.copy(order="F")
    s.solve(ref, pin_gauge=True)
    return f, interior(ref), dzci, dzfi, dli, singular


def _solve(api, ng, cbc, f, dzci, dzfi, dli, **kw):
    plan = api.PoissonPlan(ng, dli, dzci, dzfi, cbc, **kw)
    d, p = api.DeviceArray.from_host(f), api.DeviceArray(f.shape)
    p.zero()
    plan.solve_into(d, p)
    return plan, d, p


@pytest.mark.parametrize("n", LENGTHS)
@pytest.mark.parametrize("axis", [0, 1])
def test_general_lengths_match_oracle(api, oracle, n, axis):
    q = LENGTHS.index(n)
    pair = PAIRS[(q + axis) % len(PAIRS)]
    z = ["NN", "PP", "DD"][q % 3]
    # 20 lines are one full tile of 16 and a partial one; 38 planes end in a
    # partial group and (z chunks of short walks) a short last chunk
    ng = (n, 20, 38) if axis == 0 else (6, n, 38)
    cbc = pair + "NN" + z if axis == 0 else "PP" + pair + z
    alpha = 0.0 if z == "PP" else 1.2
    print(f"general {ng} {cbc}", flush=True)
    f, ref, dzci, dzfi, dli, singular = _case(oracle, ng, cbc, alpha, 100 + n)
    plan, d, p = _solve(api, ng, cbc, f, dzci, dzfi, dli)
    got = p.to_host()
    assert relmax(interior(got), ref) <= 1e-12
    np.testing.assert_array_equal(got[0], 0.0)  # the halo is untouched
    # the residual of a solution correct to rounding is eps |L| |p| / |f|,
    # which the grid decides: that of the oracle's own solution
    r = np.zeros_like(f)
    r[1:-1, 1:-1, 1:-1] = ref
    assert plan.residual(d, p) <= 2 * plan.residual(d, api.DeviceArray.from_host(r)) + 1e-13
    stages = [name for name, _ in plan.profile(d, p, 1)]
    assert stages == ["P1_x_fwd", "P2_yz_fwd", "P3_zy_bwd", "P4_x_bwd"]
    plan.destroy()


@pytest.mark.parametrize("ng,cbc", [((36, 60, 70), "PPPPNN"), ((22, 300, 40), "NNDDPP"),
                                    ((90, 520, 22), "DDNNDD")])
def test_general_chunk_counts(api, oracle, ng, cbc):
    f, ref, dzci, dzfi, dli, singular = _case(oracle, ng, cbc, 0.0, 7)
    plan, d, p = _solve(api, ng, cbc, f, dzci, dzfi, dli)
    seen = set()
    for n in range(0, 9):
        got = plan.set_zchunks(n)
        assert 1 <= got <= max(n, 8)
        seen.add(got)
        p.zero()
        plan.solve_into(d, p)
        print(f"general {ng} {cbc} chunks {got}", flush=True)
        assert relmax(interior(p.to_host()), ref) <= 1e-12, got
    assert len(seen) >= 2
    plan.destroy()


@pytest.mark.parametrize("ng,cbc", [((36, 90, 40), "PPPPNN"), ((66, 300, 24), "NNNNPP"),
                                    ((128, 180, 34), "NDPPDD"), ((250, 64, 20), "DDNNNN")])
def test_general_refined_and_f32(api, oracle, ng, cbc):
    f, ref, dzci, dzfi, dli, singular = _case(oracle, ng, cbc, 0.0, 11)
    plan, d, p = _solve(api, ng, cbc, f, dzci, dzfi, dli, precision=api.FP32_REFINE, tol=1e-10)
    it, rr = plan.stats()
    assert rr <= 1e-10 and it >= 1
    free = gauge_free if singular else (lambda a: a)
    assert relmax(free(interior(p.to_host())), free(ref)) <= 1e-9
    plan.destroy()
    # an FP32 field on an FP64 plan
    plan = api.PoissonPlan(ng, dli, dzci, dzfi, cbc)
    s = api.DeviceArray.from_host(np.asfortranarray(f.astype(np.float32)))
    rc = api.lib.flutas_psolve_solve_f32(C.c_void_p(plan._h),
                                         C.cast(C.c_void_p(s.ptr), C.POINTER(C.c_float)))
    assert rc == 0
    got = interior(s.to_host().astype(np.float64))
    assert relmax(gauge_free(got), gauge_free(ref)) <= 1e-4
    plan.destroy()


@pytest.mark.parametrize("bad", [np.nan, np.inf])
def test_general_nonfinite(api, oracle, bad):
    ng, cbc = (36, 300, 10), "PPPPNN"
    f, _, dzci, dzfi, dli, _ = _case(oracle, ng, cbc, 0.0, 3)
    f[5, 7, 4] = bad
    plan = api.PoissonPlan(ng, dli, dzci, dzfi, cbc)
    d = api.DeviceArray.from_host(f)
    with pytest.raises(api.FlutasError) as e:
        plan.solve(d)
    assert e.value.code == api.FLUTAS_ENONFINITE
    plan.destroy()


def test_general_graph_replays(api, oracle):
    """A recorded solve (tiles above 64 KB of LDS) replayed, against the
    eager one, bit for bit."""
    ng, cbc = (1000, 300, 12), "PPNNNN"
    f, _, dzci, dzfi, dli, _ = _case(oracle, ng, cbc, 0.0, 4)
    plan = api.PoissonPlan(ng, dli, dzci, dzfi, cbc)
    d = api.DeviceArray.from_host(f)
    plan.solve_async(d)
    api.synchronize()
    ref = d.to_host()
    with api.Graph() as g:
        plan.solve_async(d)
    for _ in range(3):
        d.upload(f)
        g.launch()
        api.synchronize()
        np.testing.assert_array_equal(d.to_host(), ref)
        plan.residual(d, d)
    g.destroy()
    plan.destroy()
