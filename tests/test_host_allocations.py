"""Out of device memory: a call that fails leaves nothing half allocated behind
it, so that the next one allocates again instead of launching on null buffers.
On the stand-in runtime; no GPU."""
from host_runtime import host_run

SURROGATE = """
import numpy as np
def weights(g):
    w = np.ones(g.mlp_size(), dtype=np.float32)
    return g.lib.les_mlp_set_weights(w.ctypes.data_as(ctypes.POINTER(ctypes.c_float)), w.size)
x = np.zeros(4096 * 16, dtype=np.float32)
def train(g, n):
    loss = ctypes.c_double()
    return g.lib.les_mlp_train_step(x.ctypes.data, x.ctypes.data, n, 1e-3, ctypes.byref(loss))
prm = P.LesParams(nx=16, ny=16, nz=8, precision=P.PREC_MIXED)
"""


def test_training_after_a_failed_allocation():
    out = host_run(SURROGATE + """
res = []
g = pkg.LesGpu(prm)
assert weights(g) == 0
base = rt.live
assert train(g, 4096) == 0
buffers = rt.live - base
g.close()
for k in range(1, buffers + 1):
    g = pkg.LesGpu(prm)
    weights(g)
    base = rt.live
    rt.fail_at = k
    rc = train(g, 4096)
    left, launched = rt.live - base, [l["name"] for l in rt.launches() if "gemm" in l["name"]]
    rt.fail_at = 0
    # a retry with a smaller batch, and a call that looks at the runtime's last error
    n0 = rt.mallocs
    retry, got = train(g, 1024), rt.mallocs - n0
    step = g.lib.les_step(1)
    g.close()
    res.append([rc, left, retry, got, step])
print(json.dumps(dict(buffers=buffers, res=res, live=rt.live, bad=rt.bad)))
""")
    assert out["buffers"] > 8 and out["live"] == 0 and out["bad"] == 0
    for rc, left, retry, got, step in out["res"]:
        assert (rc, left, retry, got, step) == (3, 0, 0, out["buffers"], 0)


def test_growing_batches_give_the_smaller_buffers_back():
    out = host_run(SURROGATE + """
g = pkg.LesGpu(prm)
weights(g)
live = []
for n in (1024, 2048, 1024, 4096):
    assert train(g, n) == 0
    live.append(rt.live)
g.close()
print(json.dumps(dict(live=live, left=rt.live, bad=rt.bad)))
""")
    assert len(set(out["live"])) == 1 and out["left"] == 0 and out["bad"] == 0


def test_weights_after_a_failed_allocation():
    out = host_run(SURROGATE + """
res = []
g = pkg.LesGpu(prm)
base = rt.live
assert weights(g) == 0
buffers = rt.live - base
g.close()
for k in range(1, buffers + 1):
    g = pkg.LesGpu(prm)
    base = rt.live
    rt.fail_at = k
    rc, left = weights(g), rt.live - base
    rt.fail_at = 0
    early = train(g, 1024)  # no weights yet: refused
    n0 = rt.mallocs
    again, got = weights(g), rt.mallocs - n0
    g.close()
    res.append([rc, left, early, again, got])
print(json.dumps(dict(buffers=buffers, res=res, live=rt.live, bad=rt.bad)))
""")
    assert out["buffers"] > 20 and out["live"] == 0 and out["bad"] == 0
    for r in out["res"]:
        assert r == [3, 0, 1, 0, out["buffers"]]


def test_statistics_and_tke_budget_after_a_failed_allocation():
    out = host_run("""
prm = P.LesParams(nx=16, ny=16, nz=8)
res = []
for name, use in (("les_stat_init", "les_stat_accumulate"), ("les_tke_init", "les_tke_accumulate")):
    g = pkg.LesGpu(prm)
    init, call = getattr(g.lib, name), getattr(g.lib, use)
    base = rt.live
    assert init() == 0
    buffers = rt.live - base
    assert init() == 0 and rt.live == base + buffers  # a second call only clears
    g.close()
    for k in range(1, buffers + 1):
        g = pkg.LesGpu(prm)
        base = rt.live
        rt.fail_at = k
        rc, left = init(), rt.live - base
        rt.fail_at = 0
        early, again, got = call(), init(), rt.live - base - buffers
        g.close()
        res.append([rc, left, early, again, got])
print(json.dumps(dict(res=res, live=rt.live, bad=rt.bad)))
""")
    assert len(out["res"]) == 4 + 8 and out["live"] == 0 and out["bad"] == 0
    for r in out["res"]:
        assert r == [3, 0, 1, 0, 0]
