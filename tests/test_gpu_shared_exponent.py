"""Shared-exponent blocks of the affine sweeps: inputs whose blocks leave the
accepted range are redone with renormalising steps, and parameters past the
host's line run the renormalising steps alone.  Both against the FP64 oracle
at the tolerances of the other parity tests."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from helpers import abs_err, rel_err
from oracle import oracle as O

pytestmark = pytest.mark.gpu

# (gap_open, gap_ext, T); the host's line is |go| + 8 |ge| <= 60 T ln 2
PARAMS = {"inside": (-8.0, -0.5, 0.5), "on_the_line": (-5.0, -0.4, 0.2), "beyond": (-3.0, -0.3, 0.1)}


def _scores(kind, B, L1, L2):
    rng = np.random.default_rng([len(kind), B, L1, L2])
    s = rng.normal(size=(B, L1, L2)).astype(np.float32)
    if kind == "matches":  # runs of strong matches: a block grows past 2^58
        for b in range(B):
            n = min(L1, L2 - 3)
            s[b, np.arange(n), np.arange(n) + 3] = 6.0
    elif kind == "walls":  # rows and columns of strong mismatches: cells fall below 2^-64
        s[:, 20:29] = -15.0
        s[:, :, 33:50] = -15.0
    return s


@pytest.mark.parametrize("params", list(PARAMS))
@pytest.mark.parametrize("kind", ["random", "matches", "walls"])
@pytest.mark.parametrize("shape", [(3, 200, 210), (70, 65, 81), (2, 63, 130)], ids=lambda s: "x".join(map(str, s)))
def test_blocks_outside_the_range_match_the_oracle(shape, kind, params):
    go, ge, T = PARAMS[params]
    s = _scores(kind, *shape)
    rng = np.random.default_rng(5)
    ln = np.stack([rng.integers(n // 2, n + 1, size=shape[0]) for n in shape[1:]], axis=1).astype(np.int32)
    ln[0] = shape[1:]
    print("shared exponent", shape, kind, params, flush=True)
    out = [x.cpu().numpy() for x in torch.ops.orihime.soft_sw_affine_with_grads(
        torch.from_numpy(s).cuda(), go, ge, T, torch.from_numpy(ln).cuda())]
    k = min(shape[0], 4)
    f64 = O.sw_affine_forward(s[:k].astype(np.float64), go, ge, T, ln[:k], prec="f64")
    assert all(np.isfinite(x).all() for x in out)
    assert rel_err(out[0][:k], f64[0], 1e-3) < 1e-5
    assert abs_err(out[1][:k], f64[1]) < 1e-4
    assert rel_err(out[2][:k], f64[2], 1.0) < 1e-4
    assert rel_err(out[3][:k], f64[3], 1.0) < 1e-4
