"""The library's own stream and the default stream give the same state, also
where default-stream work in torch changes the fields between the calls."""
import numpy as np
import pytest

from conftest import load_ic, load_params, load_pkg

pytestmark = pytest.mark.gpu


class _Memory:
    def __init__(self, ptr, shape):
        self.__cuda_array_interface__ = {"shape": shape, "typestr": "<f8", "data": (ptr, False), "version": 2}


@pytest.mark.parametrize("precision", [0, 1])
def test_both_streams_give_the_same_state(precision):
    torch = pytest.importorskip("torch")
    pkg, P, ic = load_pkg(), load_params(), load_ic()
    prm = P.LesParams(nx=64, ny=48, nz=24, precision=precision, cs_count=2)
    u, v, w = ic.log_law_ic(prm.nx, prm.ny, prm.nz, prm.lz, prm.z0, 0.1, seed=3)
    states = []
    for own in (True, False, None):
        with pkg.LesGpu(prm, own_stream=bool(own)) as g:
            g.set_ic(u, v, w)
            field = torch.as_tensor(_Memory(g.field_ptr("u")[0], g.shape), device="cuda")
            for i in range(4):
                if own is None:  # changes between calls
                    g.lib.les_set_default_stream(i & 1)
                g.step(2)
                field.mul_(1.0 + 2.0 ** -i)  # not waited for
            g.step(1)
            states.append({n: g.download(n) for n in ("u", "v", "w", "p", "cs_opt2", "F_LM")})
    for s in states[1:]:
        for n, a in s.items():
            assert np.array_equal(a, states[0][n]), n
    assert np.isfinite(states[0]["u"][1:-1]).all()
