"""What the host side of the library allocates, launches and waits for, and what
it does when device memory is short, on the CPU: the library over a stand-in
for the HIP runtime that records launches and bounds the memory."""
import pytest

import hipsim


# FP64 and refined plans whose y lines run the general kernels
@pytest.mark.parametrize("ng,kw", [((90, 300, 60), "{}"), ((64, 154, 60), "dict(precision=32)")])
def test_plan_survives_a_chunk_count_that_does_not_fit(tmp_path, ng, kw):
    hipsim.run(f"""
ng = {ng}
p = plan(ng, **{kw})
f, g = field(ng), field(ng)
first = p.set_zchunks(2)
assert first == 2
d32 = field(ng, np.float32)
assert solve32(p, d32) == 0
used = sim.sim_used()

def solves():
    sim.sim_reset()
    rc = api.lib.flutas_psolve_solve_into(C.c_void_p(p._h), f.c, g.c)
    assert sim.sim_count(2) == 0, "a launch was refused"
    return rc, [l[0] for l in launches()]

rc, names = solves()
assert rc in (0, api.FLUTAS_ENOTCONV), rc
# room for what there is and nothing more
sim.sim_limit(used)
for call in (lambda: p.set_zchunks(8), lambda: p.tune(f, g, 1)):
    try:
        call()
        raise SystemExit("tables beyond the memory")
    except api.FlutasError as e:
        assert "memory" in str(e), e
    n = C.c_int()
    api.lib.flutas_psolve_zchunks(C.c_void_p(p._h), C.byref(n))
    assert 1 <= n.value <= 2
    assert solves()[0] == rc
    assert solve32(p, d32) == 0 and sim.sim_count(2) == 0
sim.sim_limit(UNLIMITED)
assert p.set_zchunks(8) > 2
assert solves() == (rc, names)
assert solve32(p, d32) == 0
p.destroy(); f.free(); g.free(); d32.free()
api.lib.flutas_fft_cleanup()
assert sim.sim_used() == 0, "device memory left"
""", tmp_path)


def test_plans_do_not_lower_each_others_lds_limit(tmp_path):
    """The dynamic LDS limit of a kernel is one for the process: plans and
    transforms of other lengths must not lower it between another thread's
    setting and its launch."""
    hipsim.run("""
big = [(1998, 1000, 20), (1400, 706, 20), (1362, 1362, 20), (1026, 2046, 20)]
fields = [(plan(ng, **kw), field(ng), field(ng)) for ng in big
          for kw in ({}, dict(precision=32))]
d = api.DeviceArray((2046, 40))
for _ in range(2):
    for p, f, g in fields:
        api.lib.flutas_psolve_solve_into(C.c_void_p(p._h), f.c, g.c)
    for n in (2046, 1400, 1026):
        api.fft_lines("R2HC", d, n, 20)
lds = {l[3] for l in launches()}
assert len([v for v in lds if v > 64 * 1024]) >= 3, lds
assert sim.sim_count(2) == 0
assert sim.sim_lowered() == 0
""", tmp_path)


@pytest.mark.parametrize("ng", [(40000, 40000, 4), (4, 40000, 40000), (40000, 4, 40000),
                                (33000, 33000, 4)])
def test_boundary_calls_on_large_flat_grids(tmp_path, ng):
    """A launch holds fewer than 2^32 threads; faces beyond that go one by one."""
    hipsim.run(f"""
ng = {ng}
# 60 GB of addresses, no memory: nothing here touches the fields
p = api.DeviceArray([1])
fake = type("F", (api.DeviceArray,), dict(__init__=lambda s: None, free=lambda s: None))
a = fake()
a.shape, a.dtype, a.ptr = tuple(n + 2 for n in ng), np.dtype(np.float64), p.ptr
dz = np.full(ng[2] + 2, 0.5)
for cbc in ("PPPPPP", "DDNNND", "PPPPNN"):
    api.boundp(cbc, ng, (0.0,) * 6, (1.0, 1.0, 1.0), 0.5, 0.5, a)
    api.boundp_halo(cbc, ng, (0.0,) * 6, 1, 1, (1.0, 1.0, 1.0), dz, dz, a)
api.bounduvw("D" * 18, ng, np.zeros(18), 1, 1, [0] * 6, (1.0, 1.0, 1.0), dz, dz, a, a, a)
assert sim.sim_count(2) == 0 and len(launches()) > 0
""", tmp_path)


def test_refused_transforms_keep_no_tables(tmp_path):
    """Lines too long for a workgroup's LDS (64 KB, two buffers) are refused
    without tables; the longest that run keep no more than is stated, and
    flutas_fft_cleanup gives all of it back."""
    hipsim.run("""
def lines(n, f32=False, kind="REDFT10"):
    fn = api.lib.flutas_fft_guru_f32 if f32 else api.lib.flutas_fft_guru
    ct = C.c_float if f32 else C.c_double
    code = dict(REDFT10=5, REDFT00=3, RODFT00=7)[kind]
    return fn(C.c_int(code), C.c_int(n), C.c_longlong(1), C.c_int(1), C.c_longlong(n), C.c_int(1),
              C.c_longlong(0), C.cast(C.c_void_p(d.ptr), C.POINTER(ct)))

d = api.DeviceArray([1 << 14])
before = sim.sim_used()
for n in (4098, 1 << 16, 1 << 20, (1 << 31) - 2):
    assert lines(n) == api.FLUTAS_EUNSUPPORTED
    assert lines(n, kind="REDFT00") == api.FLUTAS_EUNSUPPORTED
    assert lines(n + 1 if n < 1 << 30 else n, kind="RODFT00") == api.FLUTAS_EUNSUPPORTED
assert lines(8194, True) == api.FLUTAS_EUNSUPPORTED
assert lines(2050, kind="REDFT00") == api.FLUTAS_EUNSUPPORTED
assert sim.sim_used() == before and not launches()
assert lines(4096) == 0 and lines(8192, True) == 0 and lines(2049, kind="REDFT00") == 0
assert 0 < sim.sim_used() - before <= 2 * 700000
for n in range(8192, 8192 - 400, -2):
    lines(n, True)
assert sim.sim_used() - before <= 16 * 700000
assert api.lib.flutas_fft_cleanup() == 0
assert sim.sim_used() == before
""", tmp_path)


@pytest.mark.parametrize("ng,gp", [((60, 300, 128), 8), ((6, 1200, 64), 4), ((66, 154, 128), 16)])
@pytest.mark.parametrize("z", ["NN", "PP"])
def test_chunk_tables_hold_what_is_read(tmp_path, ng, gp, z):
    """Per column and plane group d, with two chunks or more m, with periodic z
    q2; beyond that a few values per column and chunk."""
    hipsim.run(f"""
nx, ny, nz = {ng}
per = {z == "PP"}
p = plan({ng}, "PPDD{z}")

def used(n):
    assert p.set_zchunks(n) == n
    return sim.sim_used()

def tables(n):
    slots = n * (7 if per else 5) + per
    return 8 * nx * ny * ((1 + (n > 1) + per) * -(-nz // {gp}) + slots)

assert used(4) - used(1) == tables(4) - tables(1)
total = used(1)
field8 = 8 * nx * ny * nz
assert total - tables(1) < 1.3 * field8 + 4e6, (total, tables(1), field8)
""", tmp_path)


@pytest.mark.parametrize("ng,cbc,kw", [
    ((360, 300, 64), "PPDDNN", "{}"), ((6, 1200, 100), "PPDDPP", "{}"),
    ((128, 154, 90), "NNDDNN", "dict(precision=32)"), ((300, 64, 90), "PPDDPP", "{}"),
    ((100, 100, 100), "PPDDNN", "{}"), ((128, 200, 100), "PPDDPP", "dict(precision=32)")])
def test_plans_fit_where_the_line_path_fits(tmp_path, ng, cbc, kw):
    """A plan needs no more memory than its work field, the elimination's
    checkpoints and the small tables: the padding and the chunk tables are
    left out where they do not fit, and the plan solves all the same."""
    hipsim.run(f"""
import os
ng, cbc = {ng}, "{cbc}"
compiled = all(n in (64, 100, 128, 200) for n in ng[:2])
nx, ny, nz = ng
def make():
    before = sim.sim_used()
    p = plan(ng, cbc, **{kw})
    return p, sim.sim_used() - before
if compiled:
    # no line path to compare with: a dense field, one value per 8 planes and column
    # (two for periodic z), and what is small
    fp64, groups = not {kw}, -(-nz // 8)
    need = 8 * nx * ny * (nz + groups * (2 if cbc[4] == "P" else 1))
    need += 0 if fp64 else 8 * (nx + 2) * (ny + 2) * (nz + 2)
    need += 16 * (nx * ny + nx * nz + ny * nz) + 400000
else:
    os.environ["FLUTAS_UNFUSED"] = "1"
    p, need = make()
    p.destroy()
    del os.environ["FLUTAS_UNFUSED"]
f, g = field(ng), field(ng)
rich, most = make()
rich.destroy()
sim.sim_limit(sim.sim_used() + need)
p, got = make()
assert got <= need < most, (got, need, most)
sim.sim_reset()
assert api.lib.flutas_psolve_solve_into(C.c_void_p(p._h), f.c, g.c) in (0, api.FLUTAS_ENOTCONV)
assert sim.sim_count(2) == 0 and len(launches()) >= 4
p.destroy()
# an FP32 field on an FP64 plan: the work field dense, whole slabs
sim.sim_limit(UNLIMITED)
if not {kw}:
    d32 = field(ng, np.float32)
    p, got = make()
    sim.sim_limit(sim.sim_used() + 4 * nx * ny * nz)
    assert solve32(p, d32) == 0 and sim.sim_count(2) == 0
    p.destroy()
""", tmp_path)


@pytest.mark.parametrize("ng,cbc", [((64, 64, 96), "PPDDNN"), ((90, 128, 200), "PPDDPP"),
                                    ((64, 154, 96), "PPDDNN"), ((512, 512, 8), "PPPPNN")])
def test_first_f32_solve_stays_on_its_stream(tmp_path, ng, cbc):
    """One allocation, no wait for the device (other streams go on), every
    launch on the solve's stream; the second solve is the four passes."""
    hipsim.run(f"""
ng = {ng}
p, d = plan(ng, "{cbc}"), field(ng, np.float32)
api.lib.flutas_set_stream(C.c_void_p(0x1234))
sim.sim_reset()
assert solve32(p, d) == 0
assert sim.sim_count(0) == 1 and sim.sim_count(1) == 0, (sim.sim_count(0), sim.sim_count(1))
first = launches()
assert all(l[4] == 0x1234 for l in first)
assert len(first) == 4 + any("k_zchunk_tables" in l[0] for l in first)
sim.sim_reset()
assert solve32(p, d) == 0
assert launches() == first[-4:]
assert sim.sim_count(0) == sim.sim_count(1) == 0
# another count, then the plan's own again
for n in (3, 0):
    p.set_zchunks(n)
    assert solve32(p, d) == 0 and sim.sim_count(2) == 0
p.destroy()
d.free()
assert sim.sim_used() == 0
""", tmp_path)


@pytest.mark.parametrize("ng,kw,line", [
    ((2, 2, 4), "{}", True), ((60, 6, 8), "{}", True), ((30, 34, 8), "{}", False),
    ((60, 6, 10), "{}", False), ((90, 90, 4), "{}", False), ((64, 6, 4), "{}", False),
    ((6, 64, 4), "{}", False), ((60, 6, 8), "dict(precision=32)", False)])
def test_route_of_small_plans(tmp_path, ng, kw, line):
    """Few values in at most 8 planes, both lengths without a compiled plan and
    without a large prime: the line path; else the four passes."""
    hipsim.run(f"""
ng = {ng}
p, f, g = plan(ng, **{kw}), field(ng), field(ng)
sim.sim_reset()
api.lib.flutas_psolve_solve_into(C.c_void_p(p._h), f.c, g.c)
names = [l[0] for l in launches()]
assert any("k_lines" in n for n in names) == {line}, names
""", tmp_path)
