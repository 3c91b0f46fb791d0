"""The one-launch boundary calls (boundp, boundp_halo, bounduvw: every n above
2 nh) at their edges against the oracle, bit for bit: the smallest grids of
the launch, faces of 255, 256 and 257 points (workgroups of 256), halos up to 8,
every composition of rules at edges and corners, and n = 2 nh, which stays with
the face launches."""
import numpy as np
import pytest

from cases import z_metrics

pytestmark = pytest.mark.gpu

GRIDS = [(3, 3, 3), (4, 3, 5), (2, 5, 4), (17, 17, 17), (18, 16, 17), (258, 3, 4), (3, 257, 4)]


@pytest.mark.parametrize("ng", GRIDS)
@pytest.mark.parametrize("cbc", ["PPPPPP", "PPNDPP", "DNPPNN", "NNDDND"])
def test_boundp_edges(api, oracle, ng, cbc):
    bc = tuple(b if c != "P" else 0.0 for b, c in zip((0.2, -0.1, 0.3, 0.4, 0.7, -0.3), cbc))
    dzc, dzf, _, _, _, _ = z_metrics(oracle, ng[2], 1.4, 1.0)
    dl = tuple(1.0 / n for n in ng)
    p = np.asfortranarray(np.random.default_rng(sum(ng)).standard_normal([n + 2 for n in ng]))
    ref, dev = p.copy(order="F"), api.DeviceArray.from_host(p)
    for _ in range(2):
        oracle.boundp(cbc, ng, bc, 1, dl, dzc, dzf, ref)
        api.boundp(cbc, ng, bc, dl, dzc[0], dzc[ng[2]], dev)
        np.testing.assert_array_equal(dev.to_host(), ref)


@pytest.mark.parametrize("nh,ng", [(1, (3, 3, 3)), (1, (17, 18, 16)), (2, (5, 6, 5)),
                                   (2, (4, 6, 5)), (8, (17, 18, 19))])
@pytest.mark.parametrize("seed", [0, 1, 2])
def test_velocity_and_halo_edges(api, oracle, nh, ng, seed):
    rng = np.random.default_rng(100 * nh + seed)
    dzc, dzf, _, _, _, _ = z_metrics(oracle, ng[2], 1.2, 1.0, nh)
    dl = (0.21, 0.17, 1.0 / ng[2])
    shape = [n + 2 * nh for n in ng]
    # side fastest, then direction, then field; a direction periodic or two
    # kinds drawn per field and side
    cbc, bc = [], []
    for _ in range(3):
        for _ in range(3):
            pair = ["P", "P"] if rng.integers(0, 3) == 0 else list(rng.choice(["D", "N"], 2))
            cbc += pair
            bc += [0.0 if t == "P" else rng.uniform(-1, 1) for t in pair]
    cbc, bc = "".join(cbc), np.array(bc)
    host = [np.asfortranarray(rng.standard_normal(shape)) for _ in range(3)]
    ref = [a.copy(order="F") for a in host]
    dev = [api.DeviceArray.from_host(a) for a in host]
    print(f"halo {nh} {ng} {cbc}", flush=True)
    for _ in range(2):
        oracle.bounduvw(cbc, ng, bc, nh, nh, [0] * 6, dl, dzc, dzf, *ref)
        api.bounduvw(cbc, ng, bc, nh, nh, [0] * 6, dl, dzc, dzf, *dev)
        for c in range(3):
            np.testing.assert_array_equal(dev[c].to_host(), ref[c], err_msg=f"component {c}")
    q, qd = host[0].copy(order="F"), api.DeviceArray.from_host(host[0])
    oracle.boundp_nh(cbc[:6], ng, bc[:6], nh, nh, dl, dzc, dzf, q)
    api.boundp_halo(cbc[:6], ng, bc[:6], nh, nh, dl, dzc, dzf, qd)
    np.testing.assert_array_equal(qd.to_host(), q)
