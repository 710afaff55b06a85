"""Where the pressure solve keeps its columns in LDS: two blocks to a CU, or one
round of one block a CU of the device at hand, up to 202 levels."""
import numpy as np
import pytest

from conftest import load_ic, load_oracle, load_params, load_pkg
from host_runtime import host_run


@pytest.mark.parametrize("cus", [256, 128, 32])
def test_rule_follows_the_device(cus):
    out = host_run(f"""
rt.cus = {cus}
res = []
for nx, ny, nz in ((512, 512, 95), (512, 512, 96), (128, 128, 128), (64, 128, 128), (64, 64, 202), (64, 64, 203), (32, 32, 202)):
    with pkg.LesGpu(P.LesParams(nx=nx, ny=ny, nz=nz, sgs_model=P.SGS_CST_SMAG)) as g:
        rt.clear()
        g.press_stag_array(1.5)
        res.append([nx, ny, nz, [("lds" if "lds" in l["name"] else "memory", l["lds"]) for l in rt.launches() if "tridiag" in l["name"]]])
print(json.dumps(res))
""")
    for nx, ny, nz, solves in out:
        lds = 8 * ((nz + 1) * 64 + nz * 32 + 1024)  # x and g of 32 modes, two chunks of bet
        blocks = -(-(nx // 2) * (ny - 1) // 32)
        inside = 2 * lds <= 160 * 1024 or (lds <= 160 * 1024 and blocks <= cus)
        assert solves == [["lds", lds] if inside else ["memory", 0]], (nx, ny, nz)


@pytest.mark.gpu
@pytest.mark.parametrize("nz", [202, 203])
def test_pressure_on_both_sides_of_the_bound_equals_oracle(nz):
    """Operations and order are the oracle's: p bit for bit."""
    pkg, O, P, ic = load_pkg(), load_oracle(), load_params(), load_ic()
    prm = P.LesParams(nx=16, ny=24, nz=nz, cs_count=2)
    u, v, w = ic.log_law_ic(prm.nx, prm.ny, nz, prm.lz, prm.z0, 0.1, seed=nz)
    o = O.Oracle(prm)
    o.set_ic(u, v, w)
    o.step(2)
    with pkg.LesGpu(prm) as g:
        g.set_ic(u, v, w)
        g.step(2)
        for name in ("p", "dpdz", "u", "w"):
            got, ref = g.download(name)[1:-1], o.get(name)[1:-1]
            assert np.array_equal(got, ref), (name, np.abs(got - ref).max())
