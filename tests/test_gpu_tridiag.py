"""The pressure solve at heights around the 16-row chunks of its sweeps and
around the tallest column that is kept in LDS (201 levels)."""
import numpy as np
import pytest

from conftest import load_ic, load_oracle, load_params, load_pkg

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nz", [3, 15, 16, 17, 31, 33, 64, 200, 201, 202, 208, 209])
@pytest.mark.parametrize("nx, ny", [(8, 12), (16, 16)])
def test_pressure_of_every_chunk_remainder_equals_oracle(nx, ny, nz):
    """Operations and order are the oracle's: p and grad p bit for bit.  4 x 11
    and 8 x 15 solved modes: the last block of 32 is not whole."""
    pkg, O, P, ic = load_pkg(), load_oracle(), load_params(), load_ic()
    prm = P.LesParams(nx=nx, ny=ny, nz=nz, cs_count=2)
    u, v, w = ic.log_law_ic(nx, ny, nz, prm.lz, prm.z0, 0.1, seed=nz)
    o = O.Oracle(prm)
    o.set_ic(u, v, w)
    o.step(2)
    with pkg.LesGpu(prm) as g:
        g.set_ic(u, v, w)
        g.step(2)
        for name in ("p", "dpdx", "dpdy", "dpdz", "u", "v", "w"):
            got, ref = g.download(name)[1:-1], o.get(name)[1:-1]
            assert np.array_equal(got, ref), (name, np.abs(got - ref).max())
