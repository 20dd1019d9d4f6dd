"""The rules that choose a kernel for a call, on the CPU: tests/c_abi/routes.cpp
calls them in the library with the sizes of a call and 256 compute units."""
import ctypes as C
import itertools
import os
import shutil
import subprocess

import pytest

import minirun_hip as M
import test_gpu_few_tokens as few_tokens
import test_gpu_prefill_block as prefill_block
import test_gpu_proj_gemm as proj_gemm

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


def parameters(test):
    """The parameter sets of a test function, as dicts."""
    axes = []
    for mark in test.pytestmark:
        if mark.name == "parametrize":
            names = [n.strip() for n in mark.args[0].split(",")]
            axes.append([dict(zip(names, v if len(names) > 1 else (v,))) for v in mark.args[1]])
    return [{k: v for d in combo for k, v in d.items()} for combo in itertools.product(*axes)]


@pytest.mark.parametrize("test,route", [
    (proj_gemm.test_linear_tiles, TILES), (proj_gemm.test_affine_tiles, TILES),
    (proj_gemm.test_linear_mfma_k3_shapes, TILES), (proj_gemm.test_affine_mfma_block_shapes, GROUP_TILES),
    (proj_gemm.test_linear_mfma_edges, FEW),
    (few_tokens.test_linear_few_tokens, FEW), (few_tokens.test_affine_few_tokens, FEW),
    (few_tokens.test_affine_many_tokens, GROUP_TILES),
])
def test_gpu_tests_run_what_they_name(routes, test, route):
    """Each size of a GPU test of one kernel goes to that kernel."""
    for c in parameters(test):
        affine = "affine" in test.__name__
        got = projection(routes, c.get("tokens", proj_gemm.T_FULL), c["out_f"], c["in_f"],
                         c.get("group", 64) if affine else 0, c.get("sdt", "bf16"), c.get("x_pad", 0), c.get("ydt", "f32"))
        if test is few_tokens.test_linear_few_tokens and c["out_f"] > 12000 and c["tokens"] > 64:
            assert got[0] == TILES  # the widest shape leaves the few-token tiles first
            continue
        assert got[0] == route, (c, got)
        assert got[1] == c.get("rows", got[1]), (c, got)


def test_gpu_tests_reach_both_tile_heights(routes):
    heights = {projection(routes, c["tokens"], c["out_f"], c["in_f"], c["group"], c["sdt"], c["x_pad"], c["ydt"])[1]
               for c in parameters(few_tokens.test_affine_many_tokens)}
    assert heights == {64, 128}


def test_gpu_affine_edges_run_both_kinds(routes):
    for c in parameters(proj_gemm.test_affine_mfma_edges):
        r = projection(routes, c["tokens"], c["out_f"], c["in_f"], c["group"], c["sdt"], c["x_pad"], c["ydt"])[0]
        assert r == (FEW if c["group"] % 64 == 0 else TILES), c


@pytest.mark.parametrize("test", [few_tokens.test_affine_non_finite, few_tokens.test_affine_non_finite_rows,
                                  few_tokens.test_rows_do_not_see_what_follows_them])
def test_gpu_tests_of_odd_values_run_both_kinds(routes, test):
    for c in parameters(test):
        if not c.get("experts"):
            out_f = c.get("out_f", 6000 if c["tokens"] > 64 else 40)
            r = projection(routes, c["tokens"], out_f, c["in_f"], 64, c.get("sdt", "bf16"), 64, "f32")[0]
            assert r == (FEW if c["tokens"] < 100 else r) and r in (FEW, GROUP_TILES), c
    assert {projection(routes, c["tokens"], c.get("out_f", 6000), c["in_f"], 64)[0]
            for c in parameters(test) if c["tokens"] > 64 and not c.get("experts")} >= {GROUP_TILES}


def test_gpu_cross_path_test_runs_three_paths(routes):
    for group, large in ((64, GROUP_TILES), (0, TILES)):
        got = [projection(routes, t, 1536, 7168, group, ydt="f32")[0] for t in proj_gemm.CROSS_TOKENS]
        assert got == [GEMV, FEW, large]


def gather(routes, c):
    return routes.route_gather(c["tokens"], c["experts"], c["per_token"], c["out_f"], c["in_f"], c["group"])


def test_gpu_gather_tests_run_what_they_name(routes):
    assert all(gather(routes, c) == -1 for c in parameters(few_tokens.test_gather_few_pairs))
    assert all(gather(routes, c) == FEW for c in parameters(few_tokens.test_gather_tokens_an_expert_together))
    for c in parameters(few_tokens.test_rows_do_not_see_what_follows_them):
        if c["experts"]:
            assert gather(routes, dict(c, per_token=2, out_f=400, group=64)) == FEW, c


@pytest.mark.parametrize("tokens,experts,per_token,out_f,in_f,together", [
    (16, 128, 8, 768, 2048, False), (32, 128, 8, 768, 2048, True),   # two pairs an expert
    (32, 64, 4, 512, 1024, False), (40, 64, 4, 512, 1024, True),     # enough work
    (64, 1, 1, 768, 2048, False), (200, 1, 1, 768, 2048, True),
    (200, 4000, 64, 768, 2048, False),                               # more experts than a workgroup counts
])
def test_gather_rule(routes, tokens, experts, per_token, out_f, in_f, together):
    assert routes.route_gather(tokens, experts, per_token, out_f, in_f, 64) == (FEW if together else -1)


def test_gpu_prefill_block_tests_run_stacked(routes):
    """The 4-bit block test of many tokens takes its q_a, kv_a and g_proj as one
    launch, in tiles of both heights."""
    d, heights = prefill_block.STACK, set()
    rows = d["q_lora_rank"] + d["kv_rank"] + d["rope"] + d["heads"] * d["v"]
    for c in parameters(prefill_block.test_affine_stacked_projections):
        assert routes.route_stack(c["T"], rows, d["hidden"], 1, CUS)
        tiles = sum(-(-n // 256) for n in (d["q_lora_rank"], d["kv_rank"] + d["rope"], d["heads"] * d["v"]))
        heights.add(projection(routes, c["T"], 256 * tiles, d["hidden"], 64)[1])
    assert heights == {64, 128}
