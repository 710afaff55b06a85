"""Every transform launch has its kernel: an operation and precision without one
does not compile, and a step launches the same kernels at every length (on the
stand-in runtime; no GPU)."""
import re
import subprocess

import pytest
from conftest import PKG_DIR
from host_runtime import host_run
from test_gpu_lengths import LENGTHS

HIPCC = "/opt/rocm/bin/hipcc"


def _compiles(body, tmp_path):
    src = tmp_path / "t.hip"
    src.write_text(f'#include "{PKG_DIR}/csrc/fft_launch.h"\nbool f() {{ return {body}; }}\n')
    r = subprocess.run([HIPCC, "--offload-arch=gfx950", "--cuda-host-only", "-std=c++17", "-fsyntax-only", str(src)],
                       capture_output=True, text=True)
    assert r.returncode == 0 or "static" in r.stderr, r.stderr
    return r.returncode == 0


COLS = "cols_reg<{0}, {1}>(false, 16, ColArgs<{0}>(), 1, nullptr, 0)"
ROWS = "rows_r2c_reg<double, {0}, {1}>(false, 16, RowR2CArgs<double, {0}>(), 1, nullptr, 0)"


def test_calls_with_a_kernel_compile(tmp_path):
    ops = ["COP_GRAD, 3, true, true", "COP_DIV, 1, true, true", "COP_DIV, 1, true, false", "COP_FILT1, 1, true, true",
           "COP_FILT2, 2, true, true", "COP_COPY, 1, true, false", "COP_COPY, 1, false, true", "COP_PGRAD, 3, false, true"]
    f32 = ["COP_GRAD, 2, true, true"] + ops[1:2] + ops[3:7]
    modes = ["LOAD_SCALE", "LOAD_SCALE_DIV", "LOAD_AB2_SCALE_DIV", "LOAD_PCLEAN"]
    calls = [COLS.format("double", o) for o in ops] + [COLS.format("float", o) for o in f32]
    calls += [ROWS.format("double", m) for m in modes] + [ROWS.format("float", "LOAD_SCALE")]
    assert _compiles(" && ".join(calls), tmp_path)


@pytest.mark.parametrize("call", [
    COLS.format("float", "COP_GRAD, 3, true, true"), COLS.format("double", "COP_GRAD, 2, true, true"),
    COLS.format("float", "COP_DIV, 1, true, false"), COLS.format("float", "COP_PGRAD, 3, false, true"),
    COLS.format("double", "COP_COPY, 1, true, true"), ROWS.format("float", "LOAD_AB2_SCALE_DIV"),
    ROWS.format("float", "LOAD_PCLEAN")])
def test_calls_without_a_kernel_do_not_compile(call, tmp_path):
    assert not _compiles(call, tmp_path)


def test_a_step_launches_the_same_kernels_at_every_length():
    """8 rows to a band of the mixed mode's Nyquist sums: lengths along y that
    are no multiple of 8 sum in a kernel of their own."""
    out = host_run(f"""
res = []
for n in {LENGTHS}:
    for nx, ny in ((n, 16), (16, n)):
        for prec in (0, 1):
            with pkg.LesGpu(P.LesParams(nx=nx, ny=ny, nz=5, cs_count=2, precision=prec)) as g:
                g.tke_init()
                rt.clear()
                g.step(2)
                g.tke_accumulate()
                g.test_filter("txx", 4)
                x = (ctypes.c_double * (nx + 2) * ny * 8)()
                g.fft2d_r2c(ctypes.addressof(x), ctypes.addressof(x), 2)
                g.fft2d_c2r(ctypes.addressof(x), ctypes.addressof(x), 2)
                res.append([nx, ny, prec, [l["name"] for l in rt.launches()],
                            max(l["lds"] for l in rt.launches()), max(l["block"] for l in rt.launches())])
print(json.dumps(res))
""")
    assert len(out) == 4 * len(LENGTHS)
    seen = {}
    for nx, ny, prec, names, lds, block in out:
        kernels = []
        for n in names:  # _Z<length><name>...
            m = re.match(r"_Z(\d+)", n)
            kernels.append(n[m.end():m.end() + int(m.group(1))])
        assert seen.setdefault((prec, prec and ny % 8 == 0), kernels) == kernels, (nx, ny, prec)
        assert lds <= 160 * 1024 and block <= 1024
    assert len(seen) == 3 and all(len(k) > 50 for k in seen.values())


def test_short_lines_spread_their_nyquist_sums():
    """A wavefront of the forward rows with Nyquist sums adds its bands of 8 rows
    one after the other: at most 4 of them below 128 points, where one wavefront
    could hold the lines of 16."""
    out = host_run(f"""
res = []
for n in {[n for n in LENGTHS if n < 128]}:
    with pkg.LesGpu(P.LesParams(nx=n, ny=64, nz=30, precision=1)) as g:
        rt.clear()
        g.grad_velocity_filt("u", "dudx", "dudy")
        l, = [l for l in rt.launches() if "r2c_nyq" in l["name"]]
        res.append([n, 32 * 8, l["grid"][0] * l["block"] // 64])
print(json.dumps(res))
""")
    for n, bands, wavefronts in out:
        assert bands <= 4 * wavefronts, n


def test_many_field_rows_are_streamed_from_108_points():
    """AB2 predictor (load mode 2) and cleaned pressure (3): which of the two
    load orders a length takes."""
    out = host_run(f"""
res = []
for n in {LENGTHS}:
    with pkg.LesGpu(P.LesParams(nx=n, ny=16, nz=5)) as g:
        g.tke_init()
        rt.clear()
        g.step(1)
        g.tke_accumulate()
        res.append([n] + [l["name"] for l in rt.launches() if "r2c_reg" in l["name"]])
print(json.dumps(res))
""")
    for n, *names in out:
        streamed = "1" if n >= 108 else "0"
        for mode in "23":
            assert [s for s in names if f"ELi{mode}ELb{streamed}E" in s] and \
                not [s for s in names if f"ELi{mode}ELb{'10'[int(streamed)]}E" in s], (n, mode)
