"""The timing mode names the kernels that ran: every name of les_kernel_stat is
that of a launched kernel (on the stand-in runtime; no GPU)."""
import re

import pytest
from host_runtime import host_run


@pytest.mark.parametrize("grid, solve", [((16, 16, 8), "k_tridiag_lds"), ((16, 16, 202), "k_tridiag_lds"),
                                         ((16, 16, 203), "k_tridiag"), ((256, 256, 96), "k_tridiag")])
def test_names_are_those_of_the_launched_kernels(grid, solve):
    out = host_run(f"""
res = []
for prec in (0, 1, 2):
    for dealias in (0, 1):
        if prec == 2 and dealias: continue
        with pkg.LesGpu(P.LesParams(nx={grid[0]}, ny={grid[1]}, nz={grid[2]}, cs_count=2, precision=prec, dealias=dealias, judge_every=4)) as g:
            if prec:
                w = (ctypes.c_float * g.mlp_size())()
                g.lib.les_mlp_set_weights(w, g.mlp_size())
            g.tke_init()
            g.set_timing(True)
            rt.clear()
            g.step(6)
            g.tke_accumulate()
            stats = g.kernel_stats()
            res.append([list(stats), [l["name"] for l in rt.launches()], {{k: v["calls"] for k, v in stats.items()}}])
print(json.dumps(res))
""")
    for names, launches, calls in out:
        ran = {}
        for n in launches:  # _Z<length><name>...
            m = re.match(r"_Z(\d+)", n)
            k = n[m.end():m.end() + int(m.group(1))]
            ran[k] = ran.get(k, 0) + 1
        for n in names:
            base = re.split(r"[< ]", n)[0]
            assert base.startswith("hipMem") or base in ran, n
        assert calls[solve] == ran[solve] == 6
        assert {"k_tridiag", "k_tridiag_lds"} - {solve} - set(ran) - set(names)
    assert len(out) == 5


def test_profiler_names_of_the_solve():
    import importlib.util
    from conftest import PKG_DIR
    spec = importlib.util.spec_from_file_location("profile_summary", PKG_DIR / "profile_summary.py")
    ps = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(ps)
    assert ps.rocprof_key("k_tridiag_lds(TriArgs)") == "k_tridiag_lds"
    assert re.search(ps.FAMILY_KERNELS["tridiag"], "k_tridiag_lds(TriArgs)")
