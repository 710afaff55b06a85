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
