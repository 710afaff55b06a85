"""Fields of the test filters in a launch, by the size of their spectra: 21, 7 or
3 of the plain procedure's, with 21 the surrogate's nine in one launch and else
three (on the stand-in runtime; no GPU)."""
import pytest
from host_runtime import host_run


@pytest.mark.parametrize("grid, plain, surrogate", [((64, 64, 64), 21, 9), ((96, 96, 96), 21, 9), ((128, 128, 96), 7, 3),
                                                    ((144, 144, 128), 7, 3), ((192, 192, 96), 3, 3)])
def test_fields_in_a_launch(grid, plain, surrogate):
    out = host_run(f"""
prm = P.LesParams(nx={grid[0]}, ny={grid[1]}, nz={grid[2]}, cs_count=1, precision=P.PREC_LEARNED, judge_every=1000)
lhx, spectra = prm.nx // 2 + 1, 8 * (prm.nx // 2 + 1) * prm.ny * (prm.nz + 2)
with pkg.LesGpu(prm) as g:
    w = (ctypes.c_float * g.mlp_size())()
    g.lib.les_mlp_set_weights(w, g.mlp_size())
    g.step(2)  # the plain procedure on all levels
    rt.clear()
    g.step(1)  # the surrogate's chain on the third stream, the plain procedure on the band
    fields = [(l["stream"], l["grid"][1]) for l in rt.launches() if "k_cols_reg" in l["name"] and "ELi2ELi2ELb1ELb1" in l["name"]]
print(json.dumps(dict(fields=fields, spectra=spectra)))
""")
    by_stream = {}
    for stream, n in out["fields"]:
        by_stream.setdefault(stream, []).append(n)
    assert sorted(by_stream.values()) == sorted([[plain] * (21 // plain), [surrogate] * (9 // surrogate)])
    assert surrogate == 3 or 27 * out["spectra"] <= 256 << 20


def test_small_grids_need_no_more_buffers():
    """les_init and les_finalize pay for each buffer: grids that filter 21 fields
    at once take one more than those that filter 3, none without a dynamic model."""
    out = host_run("""
res = {}
for name, grid, model in (("21", (64, 64, 64), P.SGS_LASD), ("7", (128, 128, 64), P.SGS_LASD), ("3", (256, 256, 128), P.SGS_LASD),
                          ("static", (64, 64, 64), P.SGS_CST_SMAG)):
    rt.clear()
    with pkg.LesGpu(P.LesParams(nx=grid[0], ny=grid[1], nz=grid[2], sgs_model=model, precision=P.PREC_MIXED)) as g:
        n0 = sum(l.startswith("malloc") for l in rt.log())
        w = (ctypes.c_float * g.mlp_size())()
        g.lib.les_mlp_set_weights(w, g.mlp_size())
        n1 = sum(l.startswith("malloc") for l in rt.log())
    res[name] = [n0, n1 - n0]
print(json.dumps(dict(res=res, live=rt.live, bad=rt.bad)))
""")
    r = out["res"]
    assert r["21"] == [r["3"][0] + 1, r["3"][1] + 1] and r["7"] == [r["3"][0] + 1, r["3"][1]]
    assert r["static"][0] == r["3"][0] and out["live"] == 0 and out["bad"] == 0
