"""Exponent-tracked sweeps of the linear, Saigo-Vert and global models, per
pair and in groups of strips: edges of strips, blocks and chunks, inputs whose
blocks renormalise or leave the range, excluded cells, border exponents past
the float range, and gaps past the host's line (the log-domain sweeps).
Against the FP64 oracle at the tolerances of the parity tests."""

from __future__ import annotations

import numpy as np
import pytest
import torch

import orihime_amd as ohm
from helpers import abs_err, rel_err
from oracle import oracle as O

pytestmark = pytest.mark.gpu

ORACLE = {"sw": O.sw_forward, "sv_affine": O.sv_affine_forward, "nw_affine": O.nw_affine_forward}
# (gap_open, gap_ext, T): the benchmark's sharp scoring, shallow gaps, past the line
PARAMS = {"sharp": (-8.0, -0.5, 0.5), "shallow": (-1.25, -0.25, 0.73), "beyond": (-3.0, -0.3, 0.1)}


def _run(family, s, ln, go, ge, T):
    st, lt = torch.from_numpy(s).cuda(), torch.from_numpy(ln).cuda()
    p = [torch.tensor(v, device="cuda", requires_grad=True) for v in ((go, T) if family == "sw" else (go, ge, T))]
    kw = dict(zip(("gap_score", "temperature") if family == "sw" else
                  ("gap_open_score", "gap_extend_score", "temperature"), p))
    value = getattr(ohm, family + "_value")(st, lengths=lt, **kw)
    grads = [torch.autograd.grad(value[b], p, retain_graph=True) for b in range(len(s))]
    with torch.no_grad():
        only = getattr(ohm, family + "_value")(st, lengths=lt, **kw)
        m = getattr(ohm, family)(st, lengths=lt, **kw)
    g = np.array([[x.item() for x in row] for row in grads])
    return value.detach().cpu().numpy(), only.cpu().numpy(), m.cpu().numpy(), g


def _scores(kind, B, L1, L2):
    rng = np.random.default_rng([len(kind), B, L1, L2])
    s = rng.normal(size=(B, L1, L2)).astype(np.float32)
    if kind == "matches":  # a block grows past 2^58
        n = min(L1, L2)
        s[:, np.arange(n), np.arange(n)] = 6.0
    elif kind == "walls":  # and falls below 2^-64
        s[:, 20:29] = -15.0
        s[:, :, 33:50] = -15.0
    elif kind == "masked":  # past the last row and column, and a block inside
        s[:, (3 * L1) // 4:] = -np.inf
        s[:, :, (2 * L2) // 3:] = -np.inf
        s[:, 10:14, 5:9] = -np.inf
    return s


@pytest.mark.parametrize("grid", ["0", "1"])
@pytest.mark.parametrize("params", list(PARAMS))
@pytest.mark.parametrize("kind,shape", [("random", (2, 1, 1)), ("random", (2, 64, 17)), ("random", (2, 5, 300)),
                                        ("random", (2, 321, 65)), ("random", (3, 130, 200)),
                                        ("matches", (2, 150, 140)), ("walls", (2, 70, 90)),
                                        ("masked", (2, 140, 150))],
                         ids=lambda v: v if isinstance(v, str) else "x".join(map(str, v)))
@pytest.mark.parametrize("family", list(ORACLE))
def test_models_match_the_oracle(family, kind, shape, params, grid, monkeypatch):
    go, ge, T = PARAMS[params]
    if family == "sw":
        go = ge
    if kind == "masked" and family == "nw_affine":
        pytest.skip("a masked corner leaves the global model the border gaps alone")
    if kind == "walls" and params == "beyond":
        pytest.skip("outside the domain: |score| / T = 150")
    print("model sweeps", family, kind, shape, params, "grid", grid, flush=True)
    monkeypatch.setenv("OHM_GRID", grid)
    s = _scores(kind, *shape)
    ln = np.tile(np.array(shape[1:], np.int32), (shape[0], 1))
    ln[0] = [max(1, shape[1] - 7), max(1, shape[2] - 3)]
    if kind == "masked":
        ln[0] = shape[1:]
    value, only, m, g = _run(family, s, ln, go, ge, T)
    ref = s.astype(np.float64)
    if kind == "masked":
        ref = np.where(np.isinf(ref), np.nanmax(np.where(np.isinf(ref), np.nan, ref)) -
                       (sum(shape[1:]) * 80.0 + 200.0) * T, ref)
    args = (go, T) if family == "sw" else (go, ge, T)
    f64 = ORACLE[family](ref, *args, ln, prec="f64")
    assert rel_err(value, f64[0], 1e-3) < 1e-5 and rel_err(only, f64[0], 1e-3) < 1e-5
    assert abs_err(m, f64[1]) < 1e-4
    for k in range(len(args) - 1):
        assert rel_err(g[:, k], f64[2 + k], 1.0) < 1e-4


@pytest.mark.parametrize("grid", ["0", "1"])
@pytest.mark.parametrize("family", ["sw_affine", *ORACLE])
def test_blocks_left_out_after_a_failed_attempt(family, grid, monkeypatch):
    """Long runs of strong matches (attempts fail, the pauses between them grow
    to 15 blocks) that begin and end inside noise (they shrink again)."""
    print("attempts", family, "grid", grid, flush=True)
    monkeypatch.setenv("OHM_GRID", grid)
    B, L1, L2 = 2, 330, 900
    rng = np.random.default_rng(12)
    s = (rng.normal(size=(B, L1, L2)) * 1.5 - 1.0).astype(np.float32)
    i = np.arange(300)
    s[0, i, i + 10] += 8.0
    s[1, i, 2 * i + 200] += 9.0
    ln = np.tile(np.array([L1, L2], np.int32), (B, 1))
    go, ge, T = (-1.0, 0.0, 1.0) if family == "sw" else (-11.0, -1.0, 1.0)
    value, only, m, g = _run(family, s, ln, go, ge, T)
    args = (go, T) if family == "sw" else (go, ge, T)
    f64 = {"sw_affine": O.sw_affine_forward, **ORACLE}[family](s.astype(np.float64), *args, ln, prec="f64")
    assert rel_err(value, f64[0], 1e-3) < 1e-5 and rel_err(only, f64[0], 1e-3) < 1e-5
    assert abs_err(m, f64[1]) < 1e-4
    for k in range(len(args) - 1):
        assert rel_err(g[:, k], f64[2 + k], 1.0) < 1e-4
