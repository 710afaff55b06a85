"""Every transform length of the library, along x and along y: the kernels
have an instance per length, each with its own split into register phases."""
import numpy as np
import pytest

from conftest import load_ic, load_oracle, load_params, load_pkg, rel_l2

pytestmark = pytest.mark.gpu

# 2^a 3^b, multiples of 4, 3/2 of it at most 1024
LENGTHS = [8, 12, 16, 24, 32, 36, 48, 64, 72, 96, 108, 128, 144, 192, 216, 256, 288, 324, 384, 432, 512, 576, 648]
FIELDS = {"u": (1, -1), "v": (1, -1), "w": (1, -1), "p": (1, -1), "rhsx": (1, -1), "rhsy": (1, -1), "rhsz": (1, -1),
          "dudx": (1, None), "dudy": (1, None), "dwdx": (1, None), "dwdy": (1, None), "cs_opt2": (1, None),
          "F_LM": (1, None), "F_MM": (1, None), "F_QN": (1, None), "F_NN": (1, None)}


@pytest.mark.parametrize("axis", ["x", "y"])
@pytest.mark.parametrize("n", LENGTHS)
def test_step_of_every_length_matches_oracle(n, axis):
    """Two FP64 steps, the second with a coefficient update (every column and
    row kernel of the step).  The operations are the oracle's, but for some
    lengths with several factors of 3 the two host tables of twiddles differ
    in last bits, so the bar is the parity tests' relative L2."""
    pkg, O, P, ic = load_pkg(), load_oracle(), load_params(), load_ic()
    nx, ny = (n, 16) if axis == "x" else (16, n)
    prm = P.LesParams(nx=nx, ny=ny, nz=5, cs_count=2)
    u, v, w = ic.log_law_ic(nx, ny, prm.nz, prm.lz, prm.z0, 0.1, seed=n)
    o = O.Oracle(prm)
    o.set_ic(u, v, w)
    o.step(2)
    with pkg.LesGpu(prm) as g:
        g.set_ic(u, v, w)
        g.step(2)
        for name, (a, b) in FIELDS.items():
            got, ref = g.download(name)[a:b], o.get(name)[a:b]
            assert rel_l2(got, ref) <= 1e-11, (name, np.abs(got - ref).max())


@pytest.mark.parametrize("axis", ["x", "y"])
@pytest.mark.parametrize("n", LENGTHS)
def test_fp32_kernels_of_every_length(n, axis):
    """The mixed mode's FP32 kernels against the FP64 ones on white-noise
    fields.  A transform of up to 7 stages, each value rounded about 6 times a
    stage (2^-24 relative), forward and inverse and three transforms deep at
    most in the convection: 3 * 2 * 7 * 6 * 6e-8 = 1.5e-5 of the result."""
    pkg, P = load_pkg(), load_params()
    nx, ny = (n, 16) if axis == "x" else (16, n)
    tol = 1.5e-5
    rng = np.random.default_rng(n)
    noise = {f: rng.standard_normal((7, ny, nx)) for f in ("u", "v", "w", "txx", "txy", "txz", "tyy", "tyz", "tzz")}
    out = []
    for prec in (P.PREC_FP64, P.PREC_MIXED):
        with pkg.LesGpu(P.LesParams(nx=nx, ny=ny, nz=5, precision=prec)) as g:
            for f, a in noise.items():
                g.upload(f, a.astype(np.float32).astype(np.float64))
            g.compute_vel_grad()
            got = {f: g.download(f)[1:] for f in ("dudx", "dudy", "dvdx", "dvdy", "dwdx", "dwdy")}
            g.compute_rhs_adv()
            got.update({f: g.download(f)[1:-1] for f in ("rhsx", "rhsy", "rhsz")})
            for alpha in (2, 4):
                g.test_filter("txx", alpha)
                got[f"filter{alpha}"] = g.download("txx")[1:]
        out.append(got)
    worst = {f: rel_l2(out[1][f], out[0][f]) for f in out[0] if np.abs(out[0][f]).max() > 0}
    assert worst and all(e <= tol for e in worst.values()), worst
