"""The dynamic models' test filters take 21, 7 or 3 fields a launch, by the
size of the spectra, and the surrogate's features 9 or 3: one grid of each,
against the oracle."""
import numpy as np
import pytest

from conftest import load_ic, load_oracle, load_params, load_pkg, rel_l2

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("model", ["SGS_LASD", "SGS_DYN_SMAG"])
@pytest.mark.parametrize("grid", [(32, 32, 16), (96, 96, 64), (128, 128, 96)])  # 21, 7, 3
def test_update_of_every_batch_matches_oracle(grid, model):
    """The coefficient of an FP64 update (the second step's) and what follows
    from it; the bar is the step parity tests' relative L2."""
    pkg, O, P, ic = load_pkg(), load_oracle(), load_params(), load_ic()
    nx, ny, nz = grid
    prm = P.LesParams(nx=nx, ny=ny, nz=nz, sgs_model=getattr(P, model), cs_count=2, dyn_init=2)
    u, v, w = ic.log_law_ic(nx, ny, nz, prm.lz, prm.z0, 0.1, seed=nz)
    o = O.Oracle(prm)
    o.set_ic(u, v, w)
    o.step(2)
    names = ["cs_opt2", "nu_t", "u"] + (["F_LM", "F_MM", "F_QN", "F_NN"] if model == "SGS_LASD" else [])
    with pkg.LesGpu(prm) as g:
        g.set_ic(u, v, w)
        g.step(2)
        for name in names:
            got, ref = g.download(name)[1:-1], o.get(name)[1:-1]
            assert rel_l2(got, ref) <= 1e-11, (name, np.abs(got - ref).max())
        assert not np.all(g.download("cs_opt2")[1:-1] == 0.03)


def test_features_of_the_small_batch():
    """Features on a grid that takes 3 fields a launch (the feature tests' own
    grids take 9), to the bounds of those tests."""
    from test_gpu_features import test_features_match_the_restatement as check
    check((192, 192, 96))
