"""The kernels of every length that the step and procedure tests of all lengths
do not reach: the column passes of the 2D transforms alone, in both precisions,
and the FP32 test filter with two results."""
import numpy as np
import pytest

from conftest import load_params, load_pkg, rel_l2
from test_gpu_lengths import LENGTHS

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("axis", ["x", "y"])
@pytest.mark.parametrize("n", LENGTHS)
@pytest.mark.parametrize("precision", [0, 1])
def test_2d_transforms_match_numpy(n, axis, precision):
    """White noise, forward against numpy's transform in 64 bits, and back.  Two
    transforms of up to 7 stages (a 16-point one has 2), each value rounded
    about 6 times a stage: 9 * 6 = 54 roundings of 6e-8 or 1.1e-16, at most 3.3e-6
    or 6e-15 of the result, twice that for the way there and back.  FP64 bar
    1e-13: the tables of cosines come from two libraries."""
    torch = pytest.importorskip("torch")
    pkg, P = load_pkg(), load_params()
    nx, ny = (n, 16) if axis == "x" else (16, n)
    nz = 5
    real, cplx = (np.float64, np.complex128) if precision == 0 else (np.float32, np.complex64)
    tol = 1e-13 if precision == 0 else 3.3e-6
    a = np.random.default_rng(n).standard_normal((nz + 2, ny, nx)).astype(real)
    with pkg.LesGpu(P.LesParams(nx=nx, ny=ny, nz=nz, precision=precision)) as g:
        d = torch.from_numpy(a).cuda()
        s = torch.zeros((nz + 2, ny, nx // 2 + 1, 2), dtype=d.dtype, device="cuda")
        b = torch.zeros_like(d)
        torch.cuda.synchronize()
        g.fft2d_r2c(d.data_ptr(), s.data_ptr(), nz + 2, 0.5)
        g.fft2d_c2r(s.data_ptr(), b.data_ptr(), nz + 2)
        spectrum, back = s.cpu().numpy().view(cplx)[..., 0], b.cpu().numpy()
    assert rel_l2(spectrum, 0.5 * np.fft.rfft2(a.astype(np.float64))) <= tol
    assert rel_l2(back, 0.5 * nx * ny * a.astype(np.float64)) <= 2 * tol


@pytest.mark.parametrize("axis", ["x", "y"])
@pytest.mark.parametrize("n", LENGTHS)
def test_fp32_two_result_filter_of_every_length(n, axis):
    """The first coefficient update on white noise, mixed against FP64: F_MM comes
    from the results of the 2 delta filter, F_NN from those of the 4 delta one.
    A filtered field is off by at most 1.5e-5 (the bar of the single filter), a
    product of two by twice that; M is a difference of two such terms, M:M the
    product of two M, and the differences lose at most a factor of 8:
    2 * 2 * 3e-5 * 8 = 1e-3.  A wrong place or twiddle is off by its whole size."""
    pkg, P = load_pkg(), load_params()
    nx, ny = (n, 16) if axis == "x" else (16, n)
    rng = np.random.default_rng(n)
    noise = {f: rng.standard_normal((7, ny, nx)).astype(np.float32).astype(np.float64) for f in ("u", "v", "w")}
    out = []
    for prec in (P.PREC_FP64, P.PREC_MIXED):
        with pkg.LesGpu(P.LesParams(nx=nx, ny=ny, nz=5, precision=prec, cs_count=2)) as g:
            for f, a in noise.items():
                g.upload(f, a)
            g.compute_vel_grad()
            g.sgs_stress(2, 2)
            out.append({f: g.download(f)[1:-1] for f in ("F_MM", "F_NN")})
    for f, ref in out[0].items():
        assert np.isfinite(ref).all() and np.abs(ref).max() > 0, f
        assert rel_l2(out[1][f], ref) <= 1e-3, (f, rel_l2(out[1][f], ref))


@pytest.mark.parametrize("n", LENGTHS)
def test_tke_record_of_every_length(n):
    """The cleaned pressure's forward rows at every length, in either load order:
    the sums against the oracle's, to the bar of the step at all lengths
    (relative to the sums of |value|, as the sums run in another order)."""
    from test_gpu_tke import _compare, _run
    dev, orc, ab = _run((n, 16, 6), load_params().PREC_FP64, steps=2, seed=n)
    _compare(dev, orc, ab, 1e-11)
