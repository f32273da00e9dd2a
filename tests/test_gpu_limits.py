"""Batches at the far ends of the sizes a launch takes: pairs of more than
6144 strips, rows longer than a 32-bit lane offset reaches, border gaps far
below 2^-2^20.  Against the FP64 oracle, or against the same pair in a smaller
batch, at the tolerances of the parity tests."""

from __future__ import annotations

import numpy as np
import pytest
import torch

import orihime_amd as ohm
from helpers import abs_err, rel_err
from oracle import oracle as O
from orihime_amd import _lib, embed

pytestmark = pytest.mark.gpu


def _kernel_names(call):
    from torch.profiler import ProfilerActivity, profile

    torch.cuda.synchronize()
    with profile(activities=[ProfilerActivity.CPU, ProfilerActivity.CUDA]) as prof:
        call()
        torch.cuda.synchronize()
    return {getattr(e, "name", "") or getattr(e, "key", "") for e in prof.events()}


@pytest.mark.parametrize("grid", ["0", "1"])
@pytest.mark.parametrize("rows", [64 * 6144 + 1, 983040])
def test_tall_linear_pairs_run_the_exponent_tracked_sweeps(rows, grid, monkeypatch):
    print("tall linear pair", rows, "grid", grid, flush=True)
    monkeypatch.setenv("OHM_GRID", grid)
    rng = np.random.default_rng(rows)
    s = rng.normal(size=(1, rows, 3)).astype(np.float32)
    go, T = -0.75, 0.73
    x = torch.from_numpy(s).cuda()
    kw = dict(gap_score=go, temperature=T)
    out = {}

    def run():
        out["value"], out["map"] = ohm.sw_value(x, **kw), ohm.sw(x, **kw)

    names = _kernel_names(run)
    f64 = O.sw_forward(s.astype(np.float64), go, T, prec="f64")
    assert rel_err(out["value"].cpu().numpy(), f64[0], 1e-3) < 1e-5
    assert abs_err(out["map"].cpu().numpy(), f64[1]) < 1e-4
    assert any("scaled" in n for n in names), sorted(n for n in names if "sw" in n)


@pytest.mark.parametrize("rows", [64 * 6144 + 1, 740_000, 983040])
def test_tall_embedding_pairs_fused(rows):
    print("tall fused embedding pair", rows, flush=True)
    g = torch.Generator().manual_seed(rows)
    Q = (torch.randn(1, rows, 32, generator=g) / 32 ** 0.25).to(torch.bfloat16).cuda()
    K = (torch.randn(1, 3, 32, generator=g) / 32 ** 0.25).to(torch.bfloat16).cuda()
    ln = torch.tensor([[rows, 3]], dtype=torch.int32).cuda()
    a, b = (embed.soft_align_embeddings(Q, K, ln, fused=f).cpu().numpy() for f in (True, False))
    assert np.isfinite(a).all() and rel_err(a, b) < 1e-5


# 16 rows of 72 M columns: 60 bytes a column is past 2^32
WIDE = 72_000_000


def test_rows_past_a_32_bit_lane_offset():
    """The C entry point (the operators bound L1 x L2 further below)."""
    print("rows of", WIDE, "columns", flush=True)
    lengths = torch.tensor([[16, 40]], dtype=torch.int32).cuda()
    small = torch.randn(1, 16, 40, generator=torch.Generator().manual_seed(9)).cuda()
    x = torch.zeros(1, 16, WIDE, device="cuda")
    x[:, :, :40] = small
    go, ge, T = -2.0, -0.5, 0.73
    value, only, m = torch.empty(1, device="cuda"), torch.empty(1, device="cuda"), torch.empty_like(x)
    _lib.affine_forward(x, lengths, None, go, ge, T, value=only)
    _lib.affine_forward(x, lengths, None, go, ge, T, value=value, map=m)
    f64 = O.sw_affine_forward(small.cpu().numpy().astype(np.float64), go, ge, T, prec="f64")
    for v in (value, only):
        assert rel_err(v.cpu().numpy(), f64[0]) < 1e-5
    assert abs_err(m[:, :, :40].cpu().numpy(), f64[1]) < 1e-4
    assert not m[:, :, 40:].any()
    del x, m
    torch.cuda.empty_cache()


def test_fused_embeddings_with_long_key_rows():
    print("fused embeddings,", WIDE, "keys", flush=True)
    g = torch.Generator(device="cuda").manual_seed(11)
    lengths = torch.tensor([[16, 40]], dtype=torch.int32).cuda()
    Q = torch.randn(1, 16, 32, generator=g, device="cuda").to(torch.bfloat16)
    K = torch.zeros(1, WIDE, 32, device="cuda", dtype=torch.bfloat16)
    K[:, :40] = torch.randn(1, 40, 32, generator=g, device="cuda").to(torch.bfloat16)
    wide = embed.soft_align_embeddings(Q, K, lengths, fused=True)
    near = embed.soft_align_embeddings(Q, K[:, :40].contiguous(), lengths, fused=True)
    assert rel_err(wide.cpu().numpy(), near.cpu().numpy()) < 1e-5
    del K
    torch.cuda.empty_cache()


@pytest.mark.parametrize("rows", list(range(165_100, 165_301, 20)))
def test_global_border_gaps_past_the_absent_exponent(rows):
    """Steep gaps down 165 000 rows, four strong matches: cells, adjoints and
    the partition near and below 2^-2^20."""
    print("global pair", rows, "x 4", flush=True)
    s = np.full((1, rows, 4), -1.0, np.float32)
    for j in range(4):
        s[0, (rows // 5) * (j + 1), j] = 60.0
    kw = dict(gap_open_score=-4.4, gap_extend_score=-4.4, temperature=1.0)
    x = torch.from_numpy(s).cuda()
    value, m = ohm.nw_affine_value(x, **kw).cpu().numpy(), ohm.nw_affine(x, **kw).cpu().numpy()
    f64 = O.nw_affine_forward(s.astype(np.float64), -4.4, -4.4, 1.0, prec="f64")
    assert rel_err(value, f64[0]) < 1e-5
    # four matches (the gaps' FP32 sums near 7e5 leave a few percent)
    assert np.isfinite(m).all() and abs(float(m.sum()) - 4.0) < 0.4
