"""Strip hand-off through LDS (the waves of a workgroup; groups of four strips
of the grid kernels): pairs whose strips end on and next to a round or group
edge, with fewer and more columns than a ring holds.  Against the FP64 oracle
at the tolerances of the parity tests, and against each other: the sweeps do
the same arithmetic, only Z is combined per wave or per strip."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from helpers import abs_err, rel_err
from oracle import oracle as O
import orihime_amd as ohm

pytestmark = pytest.mark.gpu

GO, GE, T = -8.0, -0.5, 0.5


@pytest.mark.parametrize("L2", [1, 16, 63, 65, 150])
@pytest.mark.parametrize("L1", [64, 256, 257, 520, 577])
def test_hand_off_edges(L1, L2, monkeypatch):
    print("hand-off", L1, L2, flush=True)
    rng = np.random.default_rng([L1, L2])
    s = (rng.normal(size=(2, L1, L2)) * 2 - 0.5).astype(np.float32)
    ln = np.array([[L1, L2], [max(1, L1 - 65), max(1, L2 - 1)]], np.int32)
    f64 = O.sw_affine_forward(s.astype(np.float64), GO, GE, T, ln, prec="f64")
    st, lt = torch.from_numpy(s).cuda(), torch.from_numpy(ln).cuda()
    maps = []
    for env in ({"OHM_GRID": "1"}, *({"OHM_GRID": "0", "OHM_FUSED": f, "OHM_WAVES": w}
                                     for f, w in (("1", "1"), ("1", "4"), ("0", "4"), ("1", "8")))):
        for k, v in {"OHM_TEAMS": "0", **env}.items():
            if k == "OHM_TEAMS" and env["OHM_GRID"] == "1":
                monkeypatch.delenv(k, raising=False)
            else:
                monkeypatch.setenv(k, v)
        out = [x.cpu().numpy() for x in torch.ops.orihime.soft_sw_affine_with_grads(st, GO, GE, T, lt)]
        only = ohm.sw_affine_value(st, gap_open_score=GO, gap_extend_score=GE, temperature=T, lengths=lt).cpu().numpy()
        maps.append(out[1])
        assert rel_err(out[0], f64[0], 1e-3) < 1e-5 and rel_err(only, f64[0], 1e-3) < 1e-5
        assert abs_err(out[1], f64[1]) < 1e-4
        assert rel_err(out[2], f64[2], 1.0) < 1e-4 and rel_err(out[3], f64[3], 1.0) < 1e-4
    for m in maps[1:]:
        assert abs_err(m, maps[0]) < 1e-6
