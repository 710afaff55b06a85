"""Which stream and device the library's work goes to, on the stand-in runtime
(no GPU): a blocking stream of its own unless the caller asks for the default
stream, and the device of les_init whatever device is current at a call."""
import pytest
from host_runtime import host_run

CALLS = """
def calls(g):
    b = (ctypes.c_double * 64)()
    L = g.lib
    L.les_step(3)
    L.les_compute_vel_grad(); L.les_compute_rhs_adv(); L.les_press_stag_array(1.5); L.les_projection(1.5)
    L.les_sgs_stress(2, 2); L.les_wall_law(); L.les_ab2(1.5, -0.5)
    L.les_test_filter(pkg.FID["txx"], 2); L.les_ddz_uv(pkg.FID["dudz"], pkg.FID["u"])
    L.les_compute_dealias_convec(*(pkg.FID[f] for f in ("rhsx", "rhsy", "rhsz")))
    g.download("txx"); g.download("dpdx"); g.layer("ustar")
    g.stat_init(); g.stat_accumulate(); g.stat_profiles()
    g.tke_init(); g.tke_accumulate(); g.tke_download()
    g.running_diagnostics(); L.les_check_nan(ctypes.byref(ctypes.c_int()))
    if g.prm.precision:
        w = (ctypes.c_float * g.mlp_size())()
        L.les_mlp_set_weights(w, g.mlp_size())
        x = (ctypes.c_float * (2048 * 16))()
        L.les_mlp_train_step(x, x, 2048, 1e-3, b)
        L.les_mlp_forward(x, 2048, x)
        L.les_step(3)
def kinds():
    w = [l.split() for l in rt.log() if l.startswith("stream")]
    return {x[1]: x[2] for x in w}
"""


@pytest.mark.parametrize("precision", [0, 1, 2])
def test_calls_run_on_a_blocking_stream_of_the_library(precision):
    """The main stream of the C interface and, asked for, the default stream;
    what a step puts beside it goes to non-blocking streams."""
    out = host_run(CALLS + f"""
prm = P.LesParams(nx=16, ny=16, nz=8, precision={precision}, cs_count=2)
lib = pkg.library()
g = pkg.LesGpu(prm, own_stream=True)
k = kinds()
calls(g)
own = sorted(set(k.get(l["stream"], l["stream"]) for l in rt.launches()))
n = len(rt.launches())
lib.les_set_default_stream(1)
rt.clear()
calls(g)
default = sorted(set(k.get(l["stream"], l["stream"]) for l in rt.launches()))
lib.les_set_default_stream(0)
rt.clear()
calls(g)
again = sorted(set(k.get(l["stream"], l["stream"]) for l in rt.launches()))
g.close()
made, gone = list(k), [l.split()[1] for l in rt.log() if l.startswith("destroy")]
g = pkg.LesGpu(prm)
rt.clear()
g.step(1)
python = sorted(set(l["stream"] for l in rt.launches()) - set(kinds()))
g.close()
print(json.dumps(dict(n=n, own=own, default=default, again=again, left=sorted(set(made) - set(gone)), bad=rt.bad, python=python)))
""")
    assert out["n"] > 100 and out["bad"] == 0 and out["left"] == []
    assert out["own"] == out["again"] == ["blocking", "nonblocking"]
    assert out["default"] == ["(nil)", "nonblocking"]
    assert "(nil)" in out["python"]


def test_c_interface_starts_on_its_own_stream():
    out = host_run("""
prm = P.LesParams(nx=16, ny=16, nz=8)
lib = pkg.library()
c = pkg._Params()
for name, _ in pkg._Params._fields_:
    setattr(c, name, getattr(prm, name))
assert lib.les_init(ctypes.byref(c)) == 0
lib.les_set_overlap(0)
assert lib.les_step(1) == 0
w = [l.split() for l in rt.log() if l.startswith("stream")]
print(json.dumps([dict((x[1], x[2]) for x in w).get(l["stream"]) for l in rt.launches()]))
""")
    assert out and set(out) == {"blocking"}


@pytest.mark.parametrize("own", [False, True])
@pytest.mark.parametrize("precision", [0, 1, 2])
def test_calls_go_to_the_device_of_les_init(precision, own):
    """A caller with several devices has another one current at the calls: on
    the default stream a launch would go there, with this device's memory."""
    out = host_run(CALLS + f"""
g = pkg.LesGpu(P.LesParams(nx=16, ny=16, nz=8, precision={precision}, cs_count=2), own_stream={own})
rt.clear()
rt.device = 3
calls(g)
now = rt.device
where = sorted(set(l["device"] for l in rt.launches()))
mem = sorted(set(l.split()[-1] for l in rt.log() if l.startswith("malloc")))
n = len(rt.launches())
g.close()
print(json.dumps(dict(n=n, where=where, mem=mem, now=now, end=rt.device)))
""")
    assert out["n"] > 100
    assert out["where"] == [0] and out["mem"] == ["0"]
    assert out["now"] == 3 and out["end"] == 3
