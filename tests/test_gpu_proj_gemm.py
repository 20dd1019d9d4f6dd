"""Token-tiled projections on MFMA: mr_linear (k3Linear, Linear.swift:55-57)
and mr_affine_matmul (affineMM, AffineWeights.swift:239-254) at 64 or more
tokens, against the oracle (fp64 accumulation of the exact fp32 weights).

Which kernel a size runs on is pinned in test_routes.py.  At T = 4096 the oracle
runs on sampled rows (both ends of the first and last
tiles, tile boundaries, a few seeded rows) and every column; the smaller
cases check every output.  Bar: |hip - oracle| <= 1e-2 + 2e-2 |oracle|
elementwise (mla_inputs.within_tolerance), plus the output-scale error.
"""
import numpy as np
import pytest

import mla_inputs as MI
import oracle as O
from test_gpu_block import check, dev, f32, sync

pytestmark = pytest.mark.gpu

T_FULL = 4096


@pytest.fixture(scope="module")
def M():
    import minirun_hip as M

    M.load()
    return M


def sample_rows(t, seed):
    rows = {0, 1, 127, 128, 255, 256, t // 2, t - 2, t - 1}
    rng = np.random.default_rng(seed)
    rows.update(int(r) for r in rng.integers(0, t, 4))
    return np.array(sorted(r for r in rows if r < t))


# K3 (dense bf16, 96 heads) projection shapes: q_a, o_proj, kv_a, q_b
@pytest.mark.parametrize("out_f,in_f", [(1536, 7168), (7168, 12288), (576, 7168), (18432, 1536)])
@pytest.mark.parametrize("ydt", ["f32", "bf16"])
def test_linear_mfma_k3_shapes(M, out_f, in_f, ydt):
    print(f"linear mfma T={T_FULL} [{out_f}, {in_f}] y={ydt}", flush=True)
    import torch

    w = O.normal_bf16(f"pg.lin.{out_f}.{in_f}", (out_f, in_f), std=in_f ** -0.5, threads=16)
    x = O.normal_bf16(f"pg.lin.x.{in_f}", (T_FULL, in_f), threads=16)
    y = M.linear(dev(x), M.DenseWeights(dev(w)), out_dtype=torch.float32 if ydt == "f32" else torch.bfloat16)
    sync()
    rows = sample_rows(T_FULL, out_f)
    ref = O.linear(O.bf16_to_f32(x[rows]), w, acc=1, threads=16)
    check(f32(y)[rows], ref, f"linear-mfma-{out_f}x{in_f}-{ydt}", scale_bar=1e-5 if ydt == "f32" else 1e-2)


# cfg-5 affine 4-bit projection shapes (group 64, bf16 scales): q_a, q_b, kv_a, o_proj
@pytest.mark.parametrize("name,out_f,in_f", [("q_a", 1536, 7168), ("q_b", 24576, 1536), ("kv_a", 576, 7168),
                                             ("o_proj", 7168, 16384)])
@pytest.mark.parametrize("centred", [False, True])
def test_affine_mfma_block_shapes(M, name, out_f, in_f, centred):
    print(f"affine mfma T={T_FULL} {name} [{out_f}, {in_f}] centred={centred}", flush=True)
    import torch

    w = MI.affine_weight(f"pg.{name}", out_f, in_f, centred=centred)
    x = O.normal_bf16(f"pg.{name}.x", (T_FULL, in_f), threads=16)
    wt = M.AffineWeights(dev(w[0]), dev(w[1]), dev(w[2]))
    y = M.affine_mm(dev(x), wt, out_dtype=torch.float32)
    yb = M.affine_mm(dev(x), wt, out_dtype=torch.bfloat16)
    sync()
    rows = sample_rows(T_FULL, in_f)
    ref = O.affine_matmul(O.bf16_to_f32(x[rows]), *w, acc=1, threads=16)
    tag = f"affine-mfma-{name}{'-centred' if centred else ''}"
    check(f32(y)[rows], ref, tag, scale_bar=1e-5)
    check(f32(yb)[rows], ref, tag + "-bf16", scale_bar=1e-2)


def affine_operand(tag, out_f, in_f, group, sdt):
    """4-bit operand with scales / biases in dtype sdt ("bf16", "f16", "f32"),
    as the oracle's arrays and the device tensors."""
    import torch

    packed = O.u32(f"{tag}.p", (out_f, in_f // 8))
    s = O.bf16_to_f32(O.abs_normal_bf16(f"{tag}.s", (out_f, in_f // group), std=0.01))
    b = O.bf16_to_f32(O.normal_bf16(f"{tag}.b", (out_f, in_f // group), std=0.01))
    if sdt == "bf16":
        sa, ba, code = O.f32_to_bf16(s), O.f32_to_bf16(b), O.BF16
        ts, tb = dev(sa), dev(ba)
    elif sdt == "f16":
        sa, ba, code = np.float16(s).view(np.uint16), np.float16(b).view(np.uint16), O.F16
        ts, tb = torch.from_numpy(sa).view(torch.float16).cuda(), torch.from_numpy(ba).view(torch.float16).cuda()
    else:
        sa, ba, code = (s * 1.37).astype(np.float32), (b * 0.71).astype(np.float32), O.F32
        ts, tb = torch.from_numpy(sa).cuda(), torch.from_numpy(ba).cuda()
    return packed, sa, ba, code, ts, tb


# groups that are no multiple of 64 run on the dequantizing tiles, the others on
# the few-token tiles at these sizes
AFFINE_EDGES = [
    (64, 256, 512, 64, "bf16", 0, "f32"),
    (100, 200, 512, 32, "f16", 8, "f32"),      # ragged M and N tiles, padded x rows, group 32
    (65, 1000, 832, 64, "bf16", 0, "bf16"),    # 13 groups
    (300, 264, 4096, 128, "f32", 16, "f32"),
    (513, 8, 96, 32, "bf16", 0, "bf16"),       # one output chunk, three k-tiles
]


@pytest.mark.parametrize("tokens,out_f,in_f,group,sdt,x_pad,ydt", AFFINE_EDGES)
def test_affine_mfma_edges(M, tokens, out_f, in_f, group, sdt, x_pad, ydt):
    print(f"affine mfma edges T={tokens} [{out_f}, {in_f}] g={group} scales={sdt} pad={x_pad} y={ydt}", flush=True)
    import torch

    packed, sa, ba, code, ts, tb = affine_operand(f"pge.{tokens}.{out_f}.{in_f}", out_f, in_f, group, sdt)
    x = O.normal_bf16(f"pge.x.{tokens}.{in_f}", (tokens, in_f + x_pad))
    xt = dev(x)[:, :in_f]
    w = M.AffineWeights(dev(packed), ts, tb, group_size=group)
    y = M.affine_mm(xt, w, out_dtype=torch.float32 if ydt == "f32" else torch.bfloat16)
    sync()
    ref = O.affine_matmul(O.bf16_to_f32(x[:, :in_f]), packed, sa, ba, group=group, scale_dtype=code, acc=1)
    check(f32(y), ref, f"affine-mfma-edge-{tokens}x{out_f}x{in_f}", scale_bar=1e-5 if ydt == "f32" else 1e-2)


# small products: the few-token tiles
LINEAR_EDGES = [
    (64, 256, 512, 0, "f32"), (100, 200, 512, 8, "f32"), (65, 1000, 832, 0, "bf16"), (513, 8, 128, 0, "bf16"),
    (257, 264, 1024, 24, "f32"),
]


@pytest.mark.parametrize("tokens,out_f,in_f,x_pad,ydt", LINEAR_EDGES)
def test_linear_mfma_edges(M, tokens, out_f, in_f, x_pad, ydt):
    print(f"linear mfma edges T={tokens} [{out_f}, {in_f}] pad={x_pad} y={ydt}", flush=True)
    import torch

    w = O.normal_bf16(f"ple.{out_f}.{in_f}", (out_f, in_f), std=in_f ** -0.5)
    x = O.normal_bf16(f"ple.x.{tokens}.{in_f}", (tokens, in_f + x_pad))
    y = M.linear(dev(x)[:, :in_f], M.DenseWeights(dev(w)), out_dtype=torch.float32 if ydt == "f32" else torch.bfloat16)
    sync()
    ref = O.linear(O.bf16_to_f32(x[:, :in_f]), w, acc=1)
    check(f32(y), ref, f"linear-mfma-edge-{tokens}x{out_f}x{in_f}", scale_bar=1e-5 if ydt == "f32" else 1e-2)


# dense tiles of gemm.hip: token rows of a tile, then the size
LINEAR_TILES = [
    (128, 2001, 2056, 32, 0, "f32"),     # one k-tile; ragged M and N tiles
    (128, 2001, 2056, 96, 8, "bf16"),    # fewer k-tiles than stages, padded x rows
    (128, 1999, 2304, 288, 24, "f32"),   # nine k-tiles
    (256, 4001, 4104, 64, 8, "f32"),     # tiles of 256 rows, one with 161
    (256, 3900, 4360, 160, 0, "bf16"),
]
# its dequantizing form: groups of a multiple of 32 that is none of 64
AFFINE_TILES = [
    (128, 300, 264, 4096, 32, "f32", 16, "f32"),
    (128, 130, 520, 480, 96, "f32", 0, "bf16"),    # three k-tiles to a group
    (128, 257, 1032, 672, 224, "f16", 8, "f32"),   # seven
    (256, 4001, 4104, 96, 32, "f16", 0, "f32"),
    (256, 3900, 4360, 192, 96, "f32", 8, "bf16"),
    (256, 4001, 4104, 32, 32, "bf16", 0, "f32"),   # one k-tile
]


def bar(mag, ref, k, ydt, split=0.0):
    """K / 8 + 32 roundings of fp32 partial sums no larger than mag = sum |x| |w|
    (tests/test_gpu_few_tokens.py), a weight's split into two bf16 parts, 2^-18 of
    each product, and the output's rounding to bf16."""
    return ((k / 8 + 32) * 2.0 ** -24 + split) * mag + (2.0 ** -8 * np.abs(ref) if ydt == "bf16" else 0.0) + 1e-30


def compare(y, x, w, k, ydt, split=0.0):
    """Every output against float64, 1000 rows at a time."""
    for i in range(0, len(x), 1000):
        xd = x[i:i + 1000].astype(np.float64)
        ref = xd @ w.T
        d = np.abs(y[i:i + 1000].astype(np.float64) - ref)
        over = d - bar(np.abs(xd) @ np.abs(w).T, ref, k, ydt, split)
        assert not (over > 0).any(), f"rows from {i}: max over the bar {over.max():.3e}, max |d| {d.max():.3e}"


@pytest.mark.parametrize("rows,tokens,out_f,in_f,x_pad,ydt", LINEAR_TILES)
def test_linear_tiles(M, rows, tokens, out_f, in_f, x_pad, ydt):
    print(f"linear tiles of {rows} T={tokens} [{out_f}, {in_f}] pad={x_pad} y={ydt}", flush=True)
    import torch

    w = O.normal_bf16(f"plt.{out_f}.{in_f}", (out_f, in_f), std=in_f ** -0.5, threads=16)
    x = O.normal_bf16(f"plt.x.{tokens}.{in_f}", (tokens, in_f + x_pad), threads=16)
    y = M.linear(dev(x)[:, :in_f], M.DenseWeights(dev(w)), out_dtype=torch.float32 if ydt == "f32" else torch.bfloat16)
    sync()
    compare(f32(y), O.bf16_to_f32(x[:, :in_f]), O.bf16_to_f32(w).astype(np.float64), in_f, ydt)


@pytest.mark.parametrize("rows,tokens,out_f,in_f,group,sdt,x_pad,ydt", AFFINE_TILES)
def test_affine_tiles(M, rows, tokens, out_f, in_f, group, sdt, x_pad, ydt):
    print(f"affine tiles of {rows} T={tokens} [{out_f}, {in_f}] g={group} scales={sdt} pad={x_pad} y={ydt}", flush=True)
    import torch

    packed, sa, ba, code, ts, tb = affine_operand(f"pat.{out_f}.{in_f}", out_f, in_f, group, sdt)
    x = O.normal_bf16(f"pat.x.{tokens}.{in_f}", (tokens, in_f + x_pad), threads=16)
    y = M.affine_mm(dev(x)[:, :in_f], M.AffineWeights(dev(packed), ts, tb, group_size=group),
                    out_dtype=torch.float32 if ydt == "f32" else torch.bfloat16)
    sync()
    conv = {O.BF16: O.bf16_to_f32, O.F16: lambda a: a.view(np.float16).astype(np.float32), O.F32: lambda a: a}[code]
    q = ((packed[..., None] >> np.arange(0, 32, 4, dtype=np.uint32)) & 15).reshape(out_f, in_f).astype(np.float32)
    s, b = np.repeat(conv(sa), group, -1), np.repeat(conv(ba), group, -1)
    w = ((s * q).astype(np.float32) + b).astype(np.float64)
    compare(f32(y), O.bf16_to_f32(x[:, :in_f]), w, in_f, ydt, split=2.0 ** -18)


CROSS_TOKENS = (1, 8, 2000)  # a GEMV, the few-token tiles, the large tiles


@pytest.mark.parametrize("affine", [True, False])
def test_paths_match_each_other(M, affine):
    """The first eight rows of a prompt through the large tiles, alone through the
    few-token tiles, and one by one through the GEMV: each inside the bar of the
    oracle, and within fp32 rounding of the others."""
    import torch

    x = O.normal_bf16("pgm.x", (CROSS_TOKENS[2], 7168), threads=16)
    if affine:
        w = MI.affine_weight("pgm.q_a", 1536, 7168)
        wt = M.AffineWeights(dev(w[0]), dev(w[1]), dev(w[2]))
        ref = O.affine_matmul(O.bf16_to_f32(x[:8]), *w, acc=1, threads=16)
        call = M.affine_mm
    else:
        w = O.normal_bf16("pgm.dense", (1536, 7168), std=7168 ** -0.5, threads=16)
        wt = M.DenseWeights(dev(w))
        ref = O.linear(O.bf16_to_f32(x[:8]), w, acc=1, threads=16)
        call = M.linear
    got = {"tiles": f32(call(dev(x), wt, out_dtype=torch.float32))[:8],
           "few": f32(call(dev(x[:8]), wt, out_dtype=torch.float32)),
           "gemv": np.concatenate([f32(call(dev(x[i:i + 1]), wt, out_dtype=torch.float32)) for i in range(8)])}
    sync()
    for name, y in got.items():
        check(y, ref, f"{name}-rows", scale_bar=1e-5)
        np.testing.assert_allclose(y, got["tiles"], rtol=1e-4, atol=1e-3)
