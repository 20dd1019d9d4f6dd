"""Projections of a few tokens (mr_linear, 2 to about 100 tokens) on MFMA, at the
edges of their tiles: 16 tokens, 16 to 48 weight rows, 32 k per wave and ring
entry, 8 waves over K.

Reference: float64 numpy over the exact float32 weights.  Bar, elementwise: a
sum over K in fp32 with at most K roundings of partial sums no larger than
sum |x| |w|, times 2^-24 each; the chains are shorter than K / 8, so K / 8 + 32 of them are
allowed; bf16 outputs add half a unit in the last place (2^-9 relative, and
again for the sum's own error on a tie)."""
import numpy as np
import pytest

import oracle as O
from test_gpu_block import dev, f32, sync

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
