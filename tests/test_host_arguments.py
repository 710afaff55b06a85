"""Field ids outside the enum are refused by every entry point that takes one,
before anything is launched (on the stand-in runtime; no GPU)."""
from host_runtime import host_run


def test_field_ids_outside_the_enum_are_refused():
    out = host_run("""
n = len(pkg.FIELDS)
b = (ctypes.c_double * 4096)()
u, t, r = pkg.FID["u"], pkg.FID["txx"], pkg.FID["rhsx"]
res = []
for prec in (0, 1):
    with pkg.LesGpu(P.LesParams(nx=8, ny=8, nz=4, precision=prec)) as g:
        L = g.lib
        ok = {"les_grad_velocity_filt": (u, t, t), "les_div_stress": (r, t, t, t, 1, 0), "les_ddz_uv": (t, u), "les_ddz_w": (t, u),
              "les_compute_dealias_convec": (r, r, r), "les_test_filter": (t, 2), "les_download_field": (t, b),
              "les_upload_field": (t, b), "les_field_ptr": (t, ctypes.byref(ctypes.c_void_p()), ctypes.byref(ctypes.c_int()))}
        ids = {"les_div_stress": 4, "les_test_filter": 1}
        for name, args in ok.items():
            assert getattr(L, name)(*args) == 0, name
            for i in range(ids.get(name, len([a for a in args if isinstance(a, int)]))):
                for bad in (-1, n, 1 << 20):
                    rt.clear()
                    rc = getattr(L, name)(*args[:i], bad, *args[i + 1:])
                    res.append([name, i, bad, rc, len(rt.launches())])
print(json.dumps(res))
""")
    assert len(out) > 80
    for r in out:
        assert r[3:] == [10, 0], r
