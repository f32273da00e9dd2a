"""Excluded cells next to strong matches: a block of steps that the forward
sweep accepts with one exponent per lane may have to be redone by the reverse
sweep (its adjoints climb faster than the cells), starting from cells that are
exactly zero.  Every model and launch shape, value, map and parameter
gradients, against the FP64 oracle at the tolerances of the parity tests."""

from __future__ import annotations

import numpy as np
import pytest
import torch

import orihime_amd as ohm
from helpers import abs_err, rel_err
from oracle import oracle as O
from orihime_amd import _lib

pytestmark = pytest.mark.gpu

ORACLE = {"sw": O.sw_forward, "sw_affine": O.sw_affine_forward, "sv_affine": O.sv_affine_forward,
          "nw_affine": O.nw_affine_forward}
T = 1.0


def _hole(B, L1, L2):
    """Weak background, strong matches one below the diagonal, one cell excluded."""
    s = np.full((B, L1, L2), -3.0, np.float32)
    n = min(L1 - 1, L2)
    s[:, np.arange(n) + 1, np.arange(n)] = 5.0
    mask = np.zeros(s.shape, bool)
    mask[:, 0, 0] = True
    return s, mask


def _strong(B, L1, L2, match, seed):
    rng = np.random.default_rng([seed, B, L1, L2])
    s = (rng.normal(size=(B, L1, L2)) * 1.5 - 1.0).astype(np.float32)
    n = min(L1, L2)
    s[:, np.arange(n), np.arange(n)] += np.float32(match)
    return s, np.zeros(s.shape, bool), rng


def _columns(B, L1, L2, width, match=7.0):
    s, mask, _ = _strong(B, L1, L2, match, width)
    mask[:, :, :width] = True
    return s, mask


def _rows(B, L1, L2, width, match=7.0):
    s, mask, _ = _strong(B, L1, L2, match, width)
    mask[:, :width] = True
    return s, mask


def _scattered(B, L1, L2, match):
    s, mask, rng = _strong(B, L1, L2, match, 3)
    return s, rng.random(s.shape) < 0.2


def _noise(B, L1, L2, scale):
    rng = np.random.default_rng([4, B, L1, L2])
    s = np.clip(rng.normal(size=(B, L1, L2)) * scale, -75, 75).astype(np.float32)
    return s, rng.random(s.shape) < 0.1


def _inside(B, L1, L2, match=7.0):
    """A hole across the matches and the last corner left out (global: paths
    past it are trailing gaps)."""
    s, mask, _ = _strong(B, L1, L2, match, 5)
    mask[:, 10:19, 5:30] = True
    mask[:, (3 * L1) // 4:, (3 * L2) // 4:] = True
    return s, mask


CASES = {
    "hole": lambda: _hole(2, 64, 64),
    "column1": lambda: _columns(2, 70, 90, 1),
    "columns5": lambda: _columns(2, 150, 141, 5),
    "columns8": lambda: _columns(2, 64, 100, 8, 8.0),
    "columns70": lambda: _columns(2, 270, 200, 70),
    "rows1": lambda: _rows(2, 90, 70, 1),
    "rows8": lambda: _rows(2, 150, 141, 8, 8.0),
    "rows70": lambda: _rows(2, 200, 270, 70),
    "scattered": lambda: _scattered(24, 130, 120, 7.0),
    "noise8": lambda: _noise(8, 100, 90, 8.0),
    "noise15": lambda: _noise(8, 100, 90, 15.0),
    "inside": lambda: _inside(2, 150, 160),
}
# the launch shapes: one launch per pair, groups of strips and, of the affine
# model, separate launches and teams
SHAPES = {"fused": {"OHM_GRID": "0"}, "grid": {"OHM_GRID": "1"}, "separate": {"OHM_GRID": "0", "OHM_FUSED": "0"},
          "team": {"OHM_GRID": "0", "OHM_FUSED": "0", "OHM_TEAMS": "1"}}


@pytest.mark.parametrize("kind", list(CASES))
@pytest.mark.parametrize("family,shape", [(f, x) for f in ORACLE for x in SHAPES
                                          if f == "sw_affine" or x in ("fused", "grid")])
def test_excluded_cells_match_the_oracle(family, kind, shape, monkeypatch):
    print("excluded cells", family, kind, shape, flush=True)
    for k, v in SHAPES[shape].items():
        monkeypatch.setenv(k, v)
    s, mask = CASES[kind]()
    go, ge = (-1.0, 0.0) if family == "sw" else (-11.0, -1.0)
    x = torch.from_numpy(s).cuda().requires_grad_()
    p = [torch.tensor(v, device="cuda", requires_grad=True) for v in ((go, T) if family == "sw" else (go, ge, T))]
    kw = dict(zip(("gap_score", "temperature") if family == "sw" else
                  ("gap_open_score", "gap_extend_score", "temperature"), p), mask=torch.from_numpy(mask).cuda())
    value = getattr(ohm, family + "_value")(x, **kw)
    grads = [[g.cpu().numpy() for g in torch.autograd.grad(value[b], (x, *p), retain_graph=True)]
             for b in range(len(s))]
    with torch.no_grad():
        m = getattr(ohm, family)(x, **kw).cpu().numpy()
        only = getattr(ohm, family + "_value")(x, **kw).cpu().numpy()
    value = value.detach().cpu().numpy()

    ref = s.astype(np.float64)
    top = np.where(mask, -np.inf, ref).max(axis=(1, 2), keepdims=True)
    ref = np.where(mask, top - (sum(s.shape[1:]) * 80.0 + 200.0) * T, ref)
    ln = np.tile(np.array(s.shape[1:], np.int32), (len(s), 1))
    f64 = ORACLE[family](ref, *((go, T) if family == "sw" else (go, ge, T)), ln, prec="f64")
    assert all(np.isfinite(a).all() for a in (value, only, m, *(g for row in grads for g in row)))
    assert rel_err(value, f64[0], 1e-3) < 1e-5 and rel_err(only, f64[0], 1e-3) < 1e-5
    assert abs_err(m, f64[1]) < 1e-4
    assert abs_err(np.where(mask, 0.0, np.stack([row[0][b] for b, row in enumerate(grads)])), f64[1]) < 1e-4
    for k in range(len(p) - 1):
        assert rel_err([float(row[1 + k]) for row in grads], f64[2 + k], 1.0) < 1e-4


@pytest.mark.parametrize("grid", ["0", "1"])
@pytest.mark.parametrize("family", ["sw", "sw_affine"])
def test_masked_tails_keep_every_pair(family, grid, monkeypatch):
    """Pairs masked past a last row and column, at every offset from the edges
    of strips and blocks: none leaves the exponent range (workspace word 8
    counts the pairs that the log-domain sweeps redo)."""
    print("masked tails", family, "grid", grid, flush=True)
    monkeypatch.setenv("OHM_GRID", grid)
    B, L1, L2 = 64, 200, 150
    rng = np.random.default_rng(21)
    s = rng.normal(size=(B, L1, L2)).astype(np.float32)
    go, ge, t = (-0.75, 0.0, 0.73) if family == "sw" else (-8.0, -0.5, 0.5)
    ln = np.stack([60 + np.arange(B) * 2, 100 + np.arange(B) % 48], axis=1).astype(np.int32)
    for b in range(B):
        s[b, ln[b, 0]:] = s[b, :, ln[b, 1]:] = -(sum(s.shape[1:]) * 80.0 + 200.0) * t
    x = torch.from_numpy(s).cuda()
    value, m, g0, g1, g2 = (torch.empty(n, device="cuda") for n in (B, s.shape, B, B, B))
    ws = torch.empty(_lib.workspace_bytes(family != "sw", _lib.OP_FORWARD, B, L1, L2, -1), dtype=torch.uint8,
                     device="cuda")
    if family == "sw":
        _lib.linear_forward(x, None, None, go, t, value=value, map=m, grad_gap=g0, grad_temp=g2, workspace=ws)
        f64 = O.sw_forward(s.astype(np.float64), go, t, prec="f64")
    else:
        _lib.affine_forward(x, None, None, go, ge, t, value=value, map=m, grad_open=g0, grad_ext=g1, grad_temp=g2,
                            workspace=ws)
        f64 = O.sw_affine_forward(s.astype(np.float64), go, ge, t, prec="f64")
        assert rel_err(g1.cpu().numpy(), f64[3], 1.0) < 1e-4
    torch.cuda.synchronize()
    assert int(ws[:256].view(torch.int32)[8].item()) == 0
    assert rel_err(value.cpu().numpy(), f64[0], 1e-3) < 1e-5
    assert abs_err(m.cpu().numpy(), f64[1]) < 1e-4
    assert rel_err(g0.cpu().numpy(), f64[2], 1.0) < 1e-4


@pytest.mark.parametrize("shape", list(SHAPES))
@pytest.mark.parametrize("rows", [63, 200])
def test_flagged_pairs_are_redone_in_every_launch_shape(rows, shape, monkeypatch):
    """Pairs whose scores jump from -75 T to 75 T between adjacent columns leave
    the exponent range and are redone by the log-domain sweeps, which run after
    both exponent-tracked ones; the others are not."""
    print("flagged pairs", rows, shape, flush=True)
    for k, v in SHAPES[shape].items():
        monkeypatch.setenv(k, v)
    rng = np.random.default_rng(rows)
    s = rng.normal(size=(5, rows, 90)).astype(np.float32)
    s[1::2] = -75.0
    s[1::2, :, 40] = 75.0
    ln = np.tile(np.array([rows, 90], np.int32), (5, 1))
    ln[2] = [rows - 20, 50]
    out = [x.cpu().numpy() for x in torch.ops.orihime.soft_sw_affine_with_grads(
        torch.from_numpy(s).cuda(), -11.0, -1.0, T, torch.from_numpy(ln).cuda())]
    f64 = O.sw_affine_forward(s.astype(np.float64), -11.0, -1.0, T, ln, prec="f64")
    assert all(np.isfinite(x).all() for x in out)
    assert rel_err(out[0], f64[0], 1e-3) < 1e-5
    assert abs_err(out[1], f64[1]) < 1e-4
    assert rel_err(out[2], f64[2], 1.0) < 1e-4 and rel_err(out[3], f64[3], 1.0) < 1e-4
