"""Which form of the inverse x pass a plan launches: lanes aligned to memory lines
for large FP64 outputs, above 512 MB in lines of 512 points and above 2 GB in
lines of 1024 (on the CPU, over the stand-in for the HIP runtime)."""
import pytest

import hipsim


@pytest.mark.parametrize("ng,aligned", [
    ((512, 512, 256), True), ((512, 64, 1900), False), ((512, 64, 1960), True),
    ((1024, 512, 256), False), ((1024, 768, 200), False), ((1024, 1024, 240), True),
    ((640, 640, 400), False)])
def test_aligned_lanes(tmp_path, ng, aligned):
    hipsim.run(f"""
p = plan({ng})
d = api.DeviceArray([1])
sim.sim_reset()
assert api.lib.flutas_psolve_solve_into(C.c_void_p(p._h), d.c, d.c) == 0
(k,) = [l[0] for l in launches() if "k_x_bwd" in l[0]]
# k_x_bwd<T, Tout, NC, TJ, NT, ACC, ALIGN>
assert ("Lb0ELb1EE" in k) == {aligned} and ("Lb0ELb0EE" in k) != {aligned}, k
""", tmp_path)
