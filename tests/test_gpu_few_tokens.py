"""Projections of a few tokens (mr_linear, mr_affine_matmul, 2 to about 100
tokens; 4-bit also many) and routed experts (mr_affine_gather_matmul) on MFMA, at the edges of
their tiles: 16 tokens, 16 to 48 weight rows, 32 (dense) or 128 (4-bit) k per
wave and ring entry, 8 waves over K.

Reference: float64 numpy over the exact float32 weights.  Bar, elementwise: a
sum over K in fp32 with at most K roundings of partial sums no larger than
sum |x| |w| (affine: of the scaled and the bias part, sum |x| (|s| q + |b|)),
times 2^-24 each; the chains are shorter than K / 8, so K / 8 + 32 of them are
allowed; bf16 outputs add half a unit in the last place (2^-9 relative, and
again for the sum's own error on a tie)."""
import numpy as np
import pytest

import oracle as O
from test_gpu_block import dev, f32, sync
from test_gpu_proj_gemm import affine_operand

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def M():
    import minirun_hip as M

    M.load()
    return M


def bar(mag, ref, k, ydt):
    return (k / 8 + 32) * 2.0 ** -24 * mag + (2.0 ** -8 * np.abs(ref) if ydt == "bf16" else 0.0) + 1e-30


def compare(got, ref, mag, k, ydt):
    d = np.abs(got.astype(np.float64) - ref)
    over = d - bar(mag, ref, k, ydt)
    assert not (over > 0).any(), f"max over the bar {over.max():.3e}, max |d| {d.max():.3e}"


def tdt(ydt):
    import torch

    return torch.float32 if ydt == "f32" else torch.bfloat16


@pytest.mark.parametrize("tokens", [2, 15, 16, 17, 32, 33, 64, 65, 100])
@pytest.mark.parametrize("out_f,in_f,x_pad,ydt", [
    (8, 32, 0, "f32"),        # one ring entry in all, half a row tile
    (50, 288, 8, "bf16"),     # 9 entries: one wave has two; ragged rows, padded x
    (4104, 544, 0, "f32"),    # two or three row tiles per workgroup, 17 entries
    (12296, 96, 0, "bf16"),
])
def test_linear_few_tokens(M, tokens, out_f, in_f, x_pad, ydt):
    print(f"linear few T={tokens} [{out_f}, {in_f}] pad={x_pad} y={ydt}", flush=True)
    w = O.normal_bf16(f"lf.{out_f}.{in_f}", (out_f, in_f), std=in_f ** -0.5)
    x = O.normal_bf16(f"lf.x.{tokens}.{in_f}", (tokens, in_f + x_pad))
    y = f32(M.linear(dev(x)[:, :in_f], M.DenseWeights(dev(w)), out_dtype=tdt(ydt)))
    sync()
    xd, wd = O.bf16_to_f32(x[:, :in_f]).astype(np.float64), O.bf16_to_f32(w).astype(np.float64)
    compare(y, xd @ wd.T, np.abs(xd) @ np.abs(wd).T, in_f, ydt)


def dequant(packed, sa, ba, code, group):
    """(exact float32 weights, |s| q + |b|) as float64"""
    conv = {O.BF16: O.bf16_to_f32, O.F16: lambda a: a.view(np.float16).astype(np.float32), O.F32: lambda a: a}[code]
    q = ((packed[..., None] >> np.arange(0, 32, 4, dtype=np.uint32)) & 15).reshape(*packed.shape[:-1], -1)
    s, b = np.repeat(conv(sa), group, -1), np.repeat(conv(ba), group, -1)
    w = (s * q.astype(np.float32)).astype(np.float32) + b
    return w.astype(np.float64), (np.abs(s) * q + np.abs(b)).astype(np.float64)


@pytest.mark.parametrize("tokens", [2, 16, 17, 33, 64, 65])
@pytest.mark.parametrize("out_f,in_f,group,sdt,x_pad,ydt", [
    (6, 64, 64, "bf16", 0, "f32"),       # one group: half a ring entry
    (40, 192, 64, "f16", 8, "f32"),      # an odd group count; ragged row tile
    (33, 1152, 128, "f32", 0, "bf16"),   # 9 entries, one scale per entry
    (34, 1088, 64, "bf16", 0, "bf16"),   # 17 groups: scales on both halves of a dword
    (64, 2048, 256, "bf16", 16, "f32"),
])
def test_affine_few_tokens(M, tokens, out_f, in_f, group, sdt, x_pad, ydt):
    print(f"affine few T={tokens} [{out_f}, {in_f}] g={group} scales={sdt} pad={x_pad} y={ydt}", flush=True)
    packed, sa, ba, code, ts, tb = affine_operand(f"af.{out_f}.{in_f}", out_f, in_f, group, sdt)
    x = O.normal_bf16(f"af.x.{tokens}.{in_f}", (tokens, in_f + x_pad))
    w = M.AffineWeights(dev(packed), ts, tb, group_size=group)
    y = f32(M.affine_mm(dev(x)[:, :in_f], w, out_dtype=tdt(ydt)))
    sync()
    wd, mag = dequant(packed, sa, ba, code, group)
    xd = O.bf16_to_f32(x[:, :in_f]).astype(np.float64)
    compare(y, xd @ wd.T, np.abs(xd) @ mag.T, in_f, ydt)


@pytest.mark.parametrize("tokens,out_f,in_f,group,sdt,x_pad,ydt", [
    (1990, 2056, 64, 64, "f32", 0, "f32"),      # one group: 3 of 4 iterations past the end; ragged tiles both ways
    (2000, 2056, 192, 64, "f16", 8, "bf16"),    # an odd group count
    (1985, 2304, 1152, 128, "f32", 0, "f32"),   # one scale for two groups
    (700, 6000, 1088, 64, "bf16", 0, "f32"),    # 17 groups: scales on both halves of a dword
    (330, 6000, 1088, 64, "bf16", 16, "bf16"),  # tiles of 64 tokens
    (321, 6008, 832, 64, "f16", 0, "f32"),      # the same, 13 groups
    (385, 6000, 1536, 192, "f32", 0, "f32"),    # three groups a scale
])
def test_affine_many_tokens(M, tokens, out_f, in_f, group, sdt, x_pad, ydt):
    """Tiles of 128 or 64 tokens x 256 weight rows (affine_gemm.hip)."""
    print(f"affine many T={tokens} [{out_f}, {in_f}] g={group} scales={sdt} pad={x_pad} y={ydt}", flush=True)
    packed, sa, ba, code, ts, tb = affine_operand(f"am.{out_f}.{in_f}", out_f, in_f, group, sdt)
    x = O.normal_bf16(f"am.x.{tokens}.{in_f}", (tokens, in_f + x_pad))
    w = M.AffineWeights(dev(packed), ts, tb, group_size=group)
    y = f32(M.affine_mm(dev(x)[:, :in_f], w, out_dtype=tdt(ydt)))
    sync()
    wd, mag = dequant(packed, sa, ba, code, group)
    xd = O.bf16_to_f32(x[:, :in_f]).astype(np.float64)
    compare(y, xd @ wd.T, np.abs(xd) @ mag.T, in_f, ydt)


@pytest.mark.parametrize("tokens,out_f,in_f", [(3, 40, 256), (40, 40, 256), (2000, 2056, 192), (330, 6000, 1088)])
def test_affine_non_finite(M, tokens, out_f, in_f):
    """An infinite activation and one that overflows the unscaled sums give
    what dequantized weights give; rows without one are untouched."""
    print(f"affine, non-finite T={tokens} [{out_f}, {in_f}]", flush=True)
    packed, sa, ba, code, ts, tb = affine_operand(f"afi.{out_f}", out_f, in_f, 64, "bf16")
    x = O.bf16_to_f32(O.normal_bf16(f"afi.x.{tokens}", (tokens, in_f)))
    x[0, 70] = np.inf
    x[1, 3] = 3e38  # 3e38 * 15 overflows; times a scale of about 0.01 it does not
    xb = O.f32_to_bf16(x)
    w = M.AffineWeights(dev(packed), ts, tb, group_size=64)
    y = f32(M.affine_mm(dev(xb), w, out_dtype=tdt("f32")))
    sync()
    wd, mag = dequant(packed, sa, ba, code, 64)
    xd = O.bf16_to_f32(xb).astype(np.float64)
    with np.errstate(invalid="ignore", over="ignore"):
        ref = xd @ wd.T
        ref[0] = (xd[0] * wd).sum(-1)
    np.testing.assert_array_equal(y[0], ref[0].astype(np.float32))
    ok = np.abs(ref[1:]) < 3e38
    got = np.where(ok, y[1:], 0).astype(np.float64)
    compare(got, np.where(ok, ref[1:], 0), np.abs(xd[1:]) @ mag.T, in_f, "f32")


@pytest.mark.parametrize("tokens,experts,per_token,out_f,in_f,group,sdt,ydt", [
    (8, 4, 2, 40, 192, 64, "bf16", "f32"),     # four tokens an expert, odd groups, ragged rows
    (33, 2, 1, 6, 64, 64, "f16", "bf16"),      # more than 16 tokens an expert
    (40, 8, 4, 64, 1152, 128, "f32", "f32"),
    (700, 16, 6, 34, 128, 64, "bf16", "bf16"),  # 4200 pairs: two scans
])
@pytest.mark.parametrize("bad", [False, True])
def test_gather_few_pairs(M, tokens, experts, per_token, out_f, in_f, group, sdt, ydt, bad):
    """Routed experts, a GEMV per pair; with `bad`, some ids are out of range
    (zeros) and one expert has no token."""
    print(f"gather few T={tokens} E={experts} k={per_token} [{out_f}, {in_f}] g={group} {sdt} {ydt} bad={bad}", flush=True)
    import torch

    packed, sa, ba, code, ts, tb = affine_operand(f"gf.{experts}.{out_f}.{in_f}", experts * out_f, in_f, group, sdt)
    rng = np.random.default_rng(tokens * 7 + experts)
    ids = rng.integers(1 if bad else 0, experts, (tokens, per_token)).astype(np.int32)
    if bad:
        ids[::3, 0] = -1
        ids[1::5, -1] = experts
    x = O.normal_bf16(f"gf.x.{tokens}.{in_f}", (tokens, in_f))
    w = M.AffineWeights(dev(packed).reshape(experts, out_f, -1), ts.reshape(experts, out_f, -1),
                        tb.reshape(experts, out_f, -1), group_size=group)
    y = f32(M.affine_gather_mm(dev(x), w, torch.from_numpy(ids).cuda(), out_dtype=tdt(ydt)))
    sync()
    wd, mag = (a.reshape(experts, out_f, in_f) for a in dequant(packed, sa, ba, code, group))
    xd = O.bf16_to_f32(x).astype(np.float64)
    ref, m = np.zeros((tokens, per_token, out_f)), np.zeros((tokens, per_token, out_f))
    for e in range(experts):
        t, j = np.nonzero(ids == e)
        ref[t, j], m[t, j] = xd[t] @ wd[e].T, np.abs(xd[t]) @ mag[e].T
    compare(y, ref, m, in_f, ydt)


@pytest.mark.parametrize("in_f", [64, 192, 1088])  # odd group counts: the last 128 k end in the next row
@pytest.mark.parametrize("tokens,experts", [(2, 0), (16, 0), (40, 0), (330, 0), (1400, 4)])
def test_rows_do_not_see_what_follows_them(M, tokens, experts, in_f):
    """A row's outputs are the same bits whatever its padding and the other
    tokens hold, NaN and infinities among it."""
    import torch

    out_f = 400 if experts else (6000 if tokens > 64 else 40)
    print(f"affine, a row beside NaN T={tokens} E={experts} [{out_f}, {in_f}]", flush=True)
    packed, _, _, _, ts, tb = affine_operand(f"anb.{experts}.{out_f}.{in_f}", max(1, experts) * out_f, in_f, 64, "bf16")
    x = O.bf16_to_f32(O.normal_bf16(f"anb.x.{tokens}.{in_f}", (tokens, in_f + 64)))
    odd = x.copy()
    odd[:, in_f:] = np.nan
    odd[1::3, :64] = np.nan
    odd[2::3, :8] = np.inf
    ids = torch.from_numpy(np.random.default_rng(5).integers(0, max(1, experts), (tokens, 2)).astype(np.int32)).cuda()

    def call(a):
        v = dev(O.f32_to_bf16(a))[:, :in_f]
        if experts:
            w = M.AffineWeights(dev(packed).reshape(experts, out_f, -1), ts.reshape(experts, out_f, -1),
                                tb.reshape(experts, out_f, -1), group_size=64)
            return M.affine_gather_mm(v, w, ids, out_dtype=tdt("f32"))
        return M.affine_mm(v, M.AffineWeights(dev(packed), ts, tb, group_size=64), out_dtype=tdt("f32"))

    y, z = f32(call(x)), f32(call(odd))
    sync()
    np.testing.assert_array_equal(z[0::3], y[0::3])
    assert np.isnan(z[1::3]).all()


@pytest.mark.parametrize("tokens,out_f,in_f,sdt", [
    (14, 40, 256, "bf16"), (70, 37, 16384, "f32"), (2000, 2056, 192, "f16"), (330, 6000, 1088, "bf16"),
])
def test_affine_non_finite_rows(M, tokens, out_f, in_f, sdt):
    """Rows with NaN, infinities (one, of both signs, everywhere) or sums that
    overflow unscaled, against what dequantized weights give; one weight row is
    positive throughout, one has an infinite group."""
    print(f"affine, non-finite rows T={tokens} [{out_f}, {in_f}] {sdt}", flush=True)
    import torch

    packed, sa, ba, code, ts, tb = affine_operand(f"afr.{out_f}.{in_f}", out_f, in_f, 64, sdt)
    top = {"bf16": 0x7FFF, "f16": 0x7FFF, "f32": None}[sdt]
    ba = ba.copy()
    ba[0] = np.abs(ba[0]) if top is None else ba[0] & top  # weights of row 0: all >= 0
    ba[5, -1] = {"bf16": 0x7F80, "f16": 0x7C00, "f32": np.inf}[sdt]
    tb = torch.from_numpy(ba).view({"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}[sdt]).cuda()
    x = O.bf16_to_f32(O.normal_bf16(f"afr.x.{tokens}.{in_f}", (tokens, in_f))).copy()
    last = in_f - 1
    x[1::7, 0::in_f - 1] = np.nan
    x[2::7, last // 2] = np.inf
    x[3::7, 3], x[3::7, last] = np.inf, -np.inf
    x[4::7] = np.inf
    x[5::7, 1:130] = -np.inf  # more infinities than are taken one by one
    x[6::7, 9] = 3e38
    xb = O.f32_to_bf16(x)
    y = f32(M.affine_mm(dev(xb), M.AffineWeights(dev(packed), ts, tb, group_size=64), out_dtype=tdt("f32")))
    sync()
    wd, mag = dequant(packed, sa, ba, code, 64)
    xd = O.bf16_to_f32(xb).astype(np.float64)
    for kind in range(7):
        rows = np.arange(kind, tokens, 7)[:6]
        with np.errstate(invalid="ignore", over="ignore"):
            ref = np.stack([(xd[r] * wd).sum(-1) for r in rows])
            m = np.stack([(np.abs(xd[r]) * mag).sum(-1) for r in rows])
        fin = np.isfinite(ref)
        np.testing.assert_array_equal(np.where(fin, 0, y[rows]), np.where(fin, 0, ref).astype(np.float32), str(kind))
        compare(np.where(fin, y[rows], 0), np.where(fin, ref, 0), np.where(fin, m, 0), in_f, "f32")
        assert fin.any() == (kind in (0, 6))
    assert (y[4::7, 0] == np.inf).all() and (y[5::7, 0] == -np.inf).all()


@pytest.mark.parametrize("tokens", [13, 300])
def test_non_finite_rows_cost_little(M, tokens):
    """Activations that are NaN, or hold an infinity in every row, take a small
    multiple of the time of finite ones (1.2 to 4.4 measured; an output at a
    time per lane it was 200 to 1000)."""
    import torch

    out_f, in_f = 7168, 16384
    print(f"affine, time of non-finite rows T={tokens} [{out_f}, {in_f}]", flush=True)
    packed = torch.randint(-2 ** 31, 2 ** 31 - 1, (out_f, in_f // 8), device="cuda").to(torch.int32)
    s = (torch.randn(out_f, in_f // 64, device="cuda").abs() * 0.01).to(torch.bfloat16)
    w = M.AffineWeights(packed, s, -7.5 * s, group_size=64)
    x = torch.randn(tokens, in_f, device="cuda").to(torch.bfloat16)
    one = x.clone()
    one[:, 77] = float("inf")

    def us(v):
        M.affine_mm(v, w)
        best = float("inf")
        for _ in range(3):
            a, b = torch.cuda.Event(True), torch.cuda.Event(True)
            a.record()
            M.affine_mm(v, w)
            M.affine_mm(v, w)
            b.record()
            b.synchronize()
            best = min(best, a.elapsed_time(b) * 500)
        return best

    t = us(x)
    for v, name in ((torch.full_like(x, float("nan")), "nan"), (one, "inf")):
        assert us(v) < 12 * t, name


def routing(kind, tokens, experts, per_token):
    """ids [tokens, per_token]: uniform; all on one expert; half of the slots on
    one; counts at the edges of passes of 16 and of windows, the rest on the last
    expert; or half of them out of range."""
    rng = np.random.default_rng(tokens + experts)
    ids = rng.integers(0, experts, (tokens, per_token)).astype(np.int32)
    if kind == "one":
        ids[:] = experts - 1
    elif kind == "half":
        ids[:, :(per_token + 1) // 2] = experts // 2
    elif kind == "edges":
        flat = np.full(tokens * per_token, experts - 1, np.int32)
        counts = [1, 15, 16, 17, 31, 32, 33, 47, 48, 49, 64, 65, 128, 129][:experts - 1]
        at = np.cumsum([0] + counts)
        for e, (i, j) in enumerate(zip(at[:-1], at[1:])):
            flat[i:j] = e
        ids = rng.permutation(flat).reshape(tokens, per_token)
    elif kind == "bad":
        ids[::2] = experts
        ids[::4, 0] = -2 ** 31
    return ids


@pytest.mark.parametrize("kind", ["uniform", "one", "half", "edges", "bad"])
@pytest.mark.parametrize("tokens,experts,per_token,out_f,in_f,group,sdt,ydt", [
    (700, 16, 6, 98, 192, 64, "bf16", "bf16"),   # 4200 pairs: two scans; an odd group count, ragged rows
    (300, 128, 8, 40, 1152, 128, "f32", "f32"),
    (700, 3, 6, 90, 192, 64, "f16", "f32"),
    (6000, 4, 2, 96, 64, 64, "bf16", "f32"),     # more windows of one expert than workgroups for them
])
def test_gather_tokens_an_expert_together(M, tokens, experts, per_token, out_f, in_f, group, sdt, ydt, kind):
    print(f"gather T={tokens} E={experts} k={per_token} [{out_f}, {in_f}] g={group} {sdt} {ydt} {kind}", flush=True)
    import torch

    packed, sa, ba, code, ts, tb = affine_operand(f"gt.{experts}.{out_f}.{in_f}", experts * out_f, in_f, group, sdt)
    ids = routing(kind, tokens, experts, per_token)
    x = O.normal_bf16(f"gt.x.{tokens}.{in_f}", (tokens, in_f))
    w = M.AffineWeights(dev(packed).reshape(experts, out_f, -1), ts.reshape(experts, out_f, -1),
                        tb.reshape(experts, out_f, -1), group_size=group)
    y = f32(M.affine_gather_mm(dev(x), w, torch.from_numpy(ids).cuda(), out_dtype=tdt(ydt)))
    sync()
    wd, mag = (a.reshape(experts, out_f, in_f) for a in dequant(packed, sa, ba, code, group))
    xd = O.bf16_to_f32(x).astype(np.float64)
    ref, m = np.zeros((tokens, per_token, out_f)), np.zeros((tokens, per_token, out_f))
    for e in range(experts):
        t, j = np.nonzero(ids == e)
        ref[t, j], m[t, j] = xd[t] @ wd[e].T, np.abs(xd[t]) @ mag[e].T
    compare(y, ref, m, in_f, ydt)


def test_a_hot_expert_is_no_chain(M):
    """200 tokens, 8 slots each, all on one of 128 experts: a small multiple of the
    time that spread slots take (1.2 measured; 13 with one workgroup per expert
    and row tile)."""
    import torch

    experts, out_f, in_f = 128, 768, 2048
    print(f"gather, time of a hot expert E={experts} [{out_f}, {in_f}]", flush=True)
    packed = torch.randint(-2 ** 31, 2 ** 31 - 1, (experts, out_f, in_f // 8), device="cuda").to(torch.int32)
    s = (torch.randn(experts, out_f, in_f // 64, device="cuda").abs() * 0.01).to(torch.bfloat16)
    w = M.AffineWeights(packed, s, -7.5 * s, group_size=64)
    x = torch.randn(200, in_f, device="cuda").to(torch.bfloat16)
    spread = torch.rand(200, experts, device="cuda").topk(8, dim=1).indices.to(torch.int32).contiguous()

    def us(ids):
        M.affine_gather_mm(x, w, ids)
        best = float("inf")
        for _ in range(5):
            a, b = torch.cuda.Event(True), torch.cuda.Event(True)
            a.record()
            for _ in range(10):
                M.affine_gather_mm(x, w, ids)
            b.record()
            b.synchronize()
            best = min(best, a.elapsed_time(b) * 100)
        return best

    assert us(torch.full_like(spread, 5)) < 4 * us(spread)
