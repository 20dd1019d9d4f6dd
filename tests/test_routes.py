"""The rules that choose a kernel for a call, on the CPU: tests/c_abi/routes.cpp
calls them in the library with the sizes of a call and 256 compute units."""
import ctypes as C
import os
import shutil
import subprocess

import pytest

import minirun_hip as M

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CUS = 256


@pytest.fixture(scope="module")
def routes(tmp_path_factory):
    hipcc = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
    if shutil.which(hipcc) is None:
        pytest.skip("no hipcc")
    M.load()
    out = str(tmp_path_factory.mktemp("routes") / "libroutes.so")
    lib = os.path.dirname(M.LIB_PATH)
    r = subprocess.run([hipcc, "-x", "hip", "--offload-arch=gfx950", "-O1", "-std=c++17", "-fPIC", "-shared",
                        "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
                        "-I", os.path.join(ROOT, "minirun-app_amd", "csrc"), "-I", os.path.join(ROOT, "include"),
                        os.path.join(ROOT, "tests", "c_abi", "routes.cpp"), "-o", out, "-L", lib, "-lminirun_hip",
                        f"-Wl,-rpath,{lib}"], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    return C.CDLL(out)


@pytest.mark.parametrize("tokens,keys,many", [
    (1, 1000, False), (1, 65536, False), (1, 196608, False), (1, 196609, False), (1, 262144, False),
    (2, 65536, False), (2, 100000, True), (4, 49152, False), (4, 65536, True), (8, 65536, True),
    (1200, 300, True), (4001, 1000, True), (16384, 4096, True),
])
def test_index_scores_kernel(routes, tokens, keys, many):
    """The many-token kernel only where a workgroup gets two tokens or more."""
    for heads in (16, 64):
        run = routes.route_index_run(tokens, heads, 128, keys, CUS)
        assert (2 <= run <= tokens) if many else run == 0, run
    assert routes.route_index_run(tokens, 24, 128, keys, CUS) == 0  # heads not in steps of 16


@pytest.mark.parametrize("rows,keys,ratio,start,few", [
    # the largest count that the radix select takes
    (1, 1000, 4, 3999, 128), (1, 256, 4, 1023, 32), (1, 128, 4, 511, 16), (1, 64, 4, 255, 0),
    (256, 256, 1, 0, 16), (512, 512, 1, 0, 16), (768, 768, 1, 0, 32), (512, 128, 4, 0, 4), (256, 64, 4, 0, 0),
    (1024, 1000, 1, 0, 8), (1024, 256, 4, 0, 0), (4001, 1000, 4, 0, 4), (4000, 250, 16, 0, 0),
])
def test_short_rows_sorted_or_selected(routes, rows, keys, ratio, start, few):
    for selected in sorted({1, few, few + 1, 2 * few + 1, min(512, keys), keys} - {0}):
        assert bool(routes.route_topk_sorts(rows, keys, ratio, start, selected, CUS)) == (selected > few), selected


GEMV, FEW, TILES, GROUP_TILES = range(4)  # ProjRoute


def projection(routes, tokens, out_f, in_f, group=0, sdt="bf16", x_pad=0, ydt="bf16"):
    rows = C.c_int()
    r = routes.route_projection(tokens, out_f, in_f, group, ("bf16", "f16", "f32").index(sdt), x_pad, int(ydt == "f32"),
                                CUS, C.byref(rows))
    return r, rows.value


@pytest.mark.parametrize("tokens,out_f,in_f,route", [
    (65536, 131073, 64, FEW),        # 5.6e6 workgroups of 512 threads
    (131072, 262145, 64, GEMV),      # more threads than a grid has
    (2 ** 31 - 1, 7, 64, GEMV),
    (2 ** 31 - 1, 1001, 64, GEMV),
    (131072, 262144, 64, TILES),     # rows that the 128-row tiles take
])
def test_few_token_tiles_fit_a_grid(routes, tokens, out_f, in_f, route):
    assert projection(routes, tokens, out_f, in_f)[0] == route
