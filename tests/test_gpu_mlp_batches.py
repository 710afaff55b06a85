"""The surrogate's gradient at the batch sizes where its sums change shape:
one strip of rows, the split of the weight gradients beyond 1024 rows (128-row
chunks, 256 of them staged at a time), whole and partial rounds of the column
sums (4096 rows)."""
import importlib.util

import numpy as np
import pytest

from conftest import ORACLE_DIR, load_params, load_pkg

pytestmark = pytest.mark.gpu

spec = importlib.util.spec_from_file_location("mlp_oracle", ORACLE_DIR / "mlp_oracle.py")
M = importlib.util.module_from_spec(spec)
spec.loader.exec_module(M)


@pytest.mark.parametrize("n", [16, 1008, 1024, 1040, 4096, 4112, 33296])
def test_gradient_of_a_batch(n):
    torch = pytest.importorskip("torch")
    pkg, P = load_pkg(), load_params()
    rng = np.random.default_rng(n)
    X = rng.standard_normal((n, 12)).astype(np.float32)
    T = rng.standard_normal((n, 2)).astype(np.float32)
    v = M.init_params(5).astype(np.float32)
    norm = np.concatenate([np.zeros(12), np.ones(12), np.zeros(2), np.ones(2), [6.0]]).astype(np.float32)
    with pkg.LesGpu(P.LesParams(nx=16, ny=16, nz=8, precision=P.PREC_MIXED)) as g:
        g.mlp_set_weights(np.concatenate([v, norm]))
        dX, dT = torch.from_numpy(X).cuda(), torch.from_numpy(T).cuda()
        xb = torch.empty((n, 16), dtype=torch.int16, device="cuda")
        yn = torch.empty((n, 16), dtype=torch.float32, device="cuda")
        torch.cuda.synchronize()
        g.mlp_prepare(dX.data_ptr(), dT.data_ptr(), n, xb.data_ptr(), yn.data_ptr())
        grad, loss = g.mlp_grad(xb.data_ptr(), yn.data_ptr(), n)
    # the same bf16 roundings on the CPU, the bars of the 2048-row check
    ref_loss, ref_grad, _ = M.loss_and_grad(v.astype(np.float64), X.astype(np.float64), T.astype(np.float64), "bf16")
    assert abs(loss - ref_loss) <= 1e-4 * ref_loss
    for name, a, b in zip(["W1", "b1", "W2", "b2", "W3", "b3", "W4", "b4"], M.unpack(grad.astype(np.float64)), M.unpack(ref_grad)):
        assert np.linalg.norm(a - b) <= 3e-3 * np.linalg.norm(b), name
