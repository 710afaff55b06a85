"""The mixed mode's FP64 Nyquist removal: the row and column sums formed while
the forward row transforms load their input, at every length."""
import numpy as np
import pytest

from conftest import load_params, load_pkg
from test_gpu_lengths import LENGTHS

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ny", [8, 24])
@pytest.mark.parametrize("nx", LENGTHS)
def test_nyquist_modes_are_removed_in_fp64(nx, ny):
    """u, v, w less their modes kx = nx/2 and ky = ny/2, restated with plain
    sums.  White noise of order 1, means over at most 648 values added in
    double precision: errors below 648 * 2^-53 * 6 = 4.4e-13 in each of the
    three terms, 2e-12 together."""
    pkg, P = load_pkg(), load_params()
    rng = np.random.default_rng(nx + ny)
    sx, sy = 1 - 2 * (np.arange(nx) & 1), 1 - 2 * (np.arange(ny) & 1)
    with pkg.LesGpu(P.LesParams(nx=nx, ny=ny, nz=5, precision=P.PREC_MIXED)) as g:
        f = {n: rng.standard_normal((7, ny, nx)) for n in ("u", "v", "w")}
        for n, a in f.items():
            g.upload(n, a)
        g.compute_vel_grad()
        for n, a in f.items():
            A = (a * sx).mean(axis=2, keepdims=True)
            B = (a * sy[:, None]).mean(axis=1, keepdims=True)
            C = (a * sx * sy[:, None]).mean(axis=(1, 2), keepdims=True)
            ref = a - A * sx - B * sy[:, None] + C * sx * sy[:, None]
            if n == "w":
                ref[1] = 0  # the wall
            assert np.abs(g.download(n)[1:6] - ref[1:6]).max() <= 2e-12, n
