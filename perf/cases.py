"""Timed workloads of the alignment framework: what its users run, through the
public functions, over the range of sizes, families, directions and dtypes
that they run it on.

A case names a kind of call and its sizes:

  map        posteriors for inference: ``<family>(scores, ...)``, no gradient
  score      alignment scores for ranking: ``<family>_value(scores, ...)``, no gradient
  step       a training step on the value: value, d loss / d scores and, with
             ``learn``, d loss / d gap scores and temperature
  map_step   a training step on the posteriors: the map and the pull-back of
             a map gradient to the scores
  ragged     the packed form of many pairs of different lengths: value, map
             and parameter gradients in one call
  embed      scores from embeddings: value, d loss / d queries and keys

``lengths`` says how a padded batch carries its pairs: "full" (every pair has
the padded size), "ragged" (a length tensor, uniform from a fraction of the
padded size up) or "mask" (the same lengths as a boolean mask of excluded
cells).  ``work`` counts each input and output once and the recurrences'
arithmetic per cell.  ``exact`` evaluates the recurrences and their
derivatives in 64 bits by torch autograd, one anti-diagonal at a time.
"""

from __future__ import annotations

import math

import torch

import orihime_amd as ohm
from orihime_amd import embed, ragged

# (gap_open or gap, gap_extend, temperature) that the framework's benchmark
# and its reference grid run: a protein-like scoring at unit temperature, a
# sharper one for long ragged batches, the grid's shallow gaps, and the one
# of embedding scores
SHARP, UNIT, GRID, EMBED = (-8.0, -0.5, 0.5), (-11.0, -1.0, 1.0), (-1.25, -0.25, 0.73), (-4.0, -0.5, 0.25)
LINEAR_GRID = (-0.75, 0.0, 0.73)


# a padded size over the shortest length that pairs of it have (default 8)
_SHORTEST = {"ragged": 16, "embed": 6}


def _case(kind, family, B, L1, L2, params, lengths="full", learn=False, dtype="float32", D=0, name=None):
    c = {"kind": kind, "family": family, "B": B, "L1": L1, "L2": L2, "lengths": lengths, "learn": learn,
         "dtype": dtype, "D": D, "open": params[0], "extend": params[1], "temperature": params[2]}
    return {"name": name, **c} if name else c


def listed():
    return [
        # posteriors of a handful of short sequences: latency is all there is
        _case("map", "sw_affine", 8, 64, 64, GRID, name="map_8x64"),
        # a small training step with learned gap score and temperature
        # (the nn layers with learnable parameters), linear gaps, odd widths
        _case("step", "sw", 32, 128, 117, LINEAR_GRID, "ragged", learn=True, name="learn_32x128"),
        # one long pair, linear gaps: the largest single-pair shape of the grid
        _case("map", "sw", 1, 2048, 2048, LINEAR_GRID, name="pair_2048"),
        # ranking many candidates by score; the scores come from a bfloat16 network
        _case("score", "sw_affine", 1024, 256, 243, UNIT, dtype="bfloat16", name="rank_1024x256"),
        # the fixed-shape training step of the benchmark
        _case("step", "sw_affine", 256, 512, 512, UNIT, name="step_256x512"),
        # the packed ragged batch of the benchmark
        _case("ragged", "sw_affine", 2048, 1024, 1024, SHARP, "ragged", name="ragged_2048x1024"),
        # long sequences, few pairs, forward and backward
        _case("step", "sw_affine", 16, 4096, 4096, UNIT, name="long_16x4096"),
        # a loss on the posteriors (second order), padded batch with lengths
        _case("map_step", "sw_affine", 64, 384, 391, UNIT, "ragged", name="posterior_64x384"),
        # global alignment trained on a padded batch
        _case("step", "nw_affine", 256, 384, 400, UNIT, "ragged", name="global_256x384"),
        # global alignment of a few long pairs (the tests' largest)
        _case("map", "nw_affine", 2, 1100, 1000, UNIT, name="global_pairs_2x1100"),
        # match-anchored local alignment, excluded cells given as a mask
        _case("step", "sv_affine", 256, 320, 333, UNIT, "mask", name="anchored_256x320"),
        # alignment of learned embeddings, from the embeddings to their gradients
        _case("embed", "sw_affine", 512, 768, 768, EMBED, "ragged", D=128, name="embed_512x768"),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """A case between and around the listed ones of its kind."""
    how = rng.choice(["small", "small", "pair", "rank", "batch", "batch", "ragged", "long", "posterior", "global",
                      "global", "global_pairs", "anchored", "embed"])
    dtype = rng.choice(["float32", "float32", "bfloat16"])
    lengths = rng.choice(["full", "ragged"])
    if how == "small":
        family = rng.choice(["sw", "sw_affine"])
        learn = rng.random() < 0.5
        return _case("step" if learn else "map", family, _log(rng, 1, 64), _log(rng, 16, 160), _log(rng, 16, 160),
                     LINEAR_GRID if family == "sw" else GRID, lengths, learn=learn)
    if how == "pair":
        family = rng.choice(["sw", "sw_affine"])
        return _case("map", family, _log(rng, 1, 4), _log(rng, 512, 2048), _log(rng, 512, 2048),
                     LINEAR_GRID if family == "sw" else GRID, lengths)
    if how == "rank":
        return _case("score", "sw_affine", _log(rng, 128, 2048), _log(rng, 64, 512), _log(rng, 64, 512), UNIT, lengths,
                     dtype=dtype)
    if how == "batch":
        family = rng.choice(["sw", "sw_affine"])
        return _case("step", family, _log(rng, 64, 512), _log(rng, 96, 640), _log(rng, 96, 640),
                     LINEAR_GRID if family == "sw" else UNIT, rng.choice(["full", "ragged", "mask"]), dtype=dtype)
    if how == "ragged":
        return _case("ragged", "sw_affine", _log(rng, 128, 2048), _log(rng, 128, 1024), _log(rng, 128, 1024), SHARP,
                     "ragged")
    if how == "long":
        return _case("step", "sw_affine", _log(rng, 2, 16), _log(rng, 1024, 4096), _log(rng, 1024, 4096), UNIT, lengths)
    if how == "posterior":
        return _case("map_step", "sw_affine", _log(rng, 8, 128), _log(rng, 64, 512), _log(rng, 64, 512), UNIT, lengths)
    if how == "global":
        L1 = _log(rng, 64, 512)
        return _case("step", "nw_affine", _log(rng, 32, 512), L1, int(L1 * rng.uniform(0.85, 1.15)), UNIT, lengths,
                     dtype=dtype)
    if how == "global_pairs":
        L1 = _log(rng, 256, 1100)
        return _case("map", "nw_affine", _log(rng, 1, 4), L1, int(L1 * rng.uniform(0.85, 1.0)), UNIT, lengths)
    if how == "anchored":
        return _case("step", "sv_affine", _log(rng, 32, 512), _log(rng, 64, 512), _log(rng, 64, 512), UNIT,
                     rng.choice(["full", "ragged", "mask"]))
    side = _log(rng, 128, 768)
    return _case("embed", "sw_affine", _log(rng, 16, 512), side, max(64, side - rng.randint(0, 63)), EMBED, "ragged",
                 D=rng.choice([32, 64, 128, 256]))


# --------------------------------------------------------------------------
# Inputs
# --------------------------------------------------------------------------


def _lengths(case, seed):
    """The pairs' lengths [B, 2] (host, int32): one draw per shape, in an order
    of the seed's, so that a packed batch has the same number of cells whatever
    the seed."""
    B, L1, L2 = case["B"], case["L1"], case["L2"]
    if case["lengths"] == "full":
        return torch.tensor([[L1, L2]] * B, dtype=torch.int32)
    part = _SHORTEST.get(case["kind"], 8)
    g = torch.Generator().manual_seed(2)
    pairs = torch.stack([torch.randint(max(1, L // part), L + 1, (B,), generator=g) for L in (L1, L2)], dim=1)
    if case["family"] == "nw_affine":  # global: sequences of comparable length
        ratio = 0.8 + 0.45 * torch.rand(B, generator=g)
        pairs[:, 1] = (pairs[:, 0] * ratio * L2 / L1).round().long().clamp(1, L2)
    order = torch.randperm(B, generator=torch.Generator().manual_seed(2 * seed + 1))
    return pairs[order].to(torch.int32)


def _mask(lengths, L1, L2):
    """True outside a pair's lengths [B, L1, L2]."""
    rows = torch.arange(L1, device=lengths.device)[None, :, None] >= lengths[:, 0, None, None]
    cols = torch.arange(L2, device=lengths.device)[None, None, :] >= lengths[:, 1, None, None]
    return rows | cols


def _offsets(lengths):
    cells = lengths[:, 0].long() * lengths[:, 1].long()
    return torch.cumsum(cells, 0) - cells, int(cells.sum())


def prepare(case, seed):
    dev = torch.device("cuda")
    g = torch.Generator(device=dev).manual_seed(2 * seed)
    B, L1, L2 = case["B"], case["L1"], case["L2"]
    host = _lengths(case, seed)
    ln = host.to(dev)
    s = {"case": case, "lengths": ln if case["lengths"] == "ragged" else None, "mask": None}
    if case["kind"] == "embed":
        D = case["D"]
        s["Q"] = (torch.randn(B, L1, D, generator=g, device=dev) / D ** 0.5).to(torch.bfloat16).requires_grad_()
        s["K"] = (torch.randn(B, L2, D, generator=g, device=dev) / D ** 0.5).to(torch.bfloat16).requires_grad_()
        s["weight"] = torch.randn(B, generator=g, device=dev)
        return s
    if case["kind"] == "ragged":
        offsets, total = _offsets(host)
        s["offsets"] = offsets.to(dev)
        s["scores"] = torch.randn(total, generator=g, device=dev)
        return s
    x = torch.randn(B, L1, L2, generator=g, device=dev)
    if case["temperature"] == UNIT[2]:
        x = x * 2 - 0.5
    s["scores"] = x.to(getattr(torch, case["dtype"]))
    if case["lengths"] == "mask":
        s["mask"] = _mask(ln, L1, L2)
    names = ("gap_score",) if case["family"] == "sw" else ("gap_open_score", "gap_extend_score")
    values = (case["open"], case["extend"])[:len(names)] + (case["temperature"],)
    s["names"] = (*names, "temperature")
    s["params"] = [torch.tensor(v, device=dev, requires_grad=True) for v in values] if case["learn"] else list(values)
    if case["kind"] in ("step", "map_step"):
        s["scores"].requires_grad_()
        s["weight"] = torch.randn(x.shape if case["kind"] == "map_step" else (B,), generator=g, device=dev)
    return s


# --------------------------------------------------------------------------
# One pass
# --------------------------------------------------------------------------


def run(s):
    c = s["case"]
    kind = c["kind"]
    if kind == "embed":
        value = embed.soft_align_embeddings(s["Q"], s["K"], s["lengths"], gap_open=c["open"], gap_ext=c["extend"],
                                            temperature=c["temperature"])
        dQ, dK = torch.autograd.grad(value, (s["Q"], s["K"]), s["weight"])
        return {"value": value, "dQ": dQ, "dK": dK}
    if kind == "ragged":
        out = ragged.sw_affine_forward(s["scores"], s["lengths"], s["offsets"], gap_open_score=c["open"],
                                       gap_extend_score=c["extend"], temperature=c["temperature"], L1max=c["L1"],
                                       L2max=c["L2"])
        return dict(zip(("value", "map", "d_open", "d_extend", "d_temperature"), out))
    kw = dict(zip(s["names"], s["params"]), lengths=s["lengths"], mask=s["mask"],
              dtype=None if c["dtype"] == "float32" else torch.float32)
    if kind == "map":
        return {"map": getattr(ohm, c["family"])(s["scores"], **kw)}
    if kind == "score":
        return {"value": getattr(ohm, c["family"] + "_value")(s["scores"], **kw)}
    wrt = [s["scores"], *s["params"]] if c["learn"] else [s["scores"]]
    if kind == "map_step":
        m = getattr(ohm, c["family"])(s["scores"], **kw)
        return {"map": m, "grads": torch.autograd.grad(m, wrt, s["weight"])}
    value = getattr(ohm, c["family"] + "_value")(s["scores"], **kw)
    return {"value": value, "grads": torch.autograd.grad(value, wrt, s["weight"])}


# --------------------------------------------------------------------------
# What a pass cannot do without
# --------------------------------------------------------------------------

# floating-point operations per cell of the recurrences in linear units
# (exponentials counted as one): forward of the linear and affine models, the
# adjoint with its contractions, and the tangent of both
_FORWARD = {"sw": 7, "sw_affine": 13, "nw_affine": 13, "sv_affine": 13}
_ADJOINT = {"sw": 10, "sw_affine": 18, "nw_affine": 18, "sv_affine": 18}


def work(case):
    B, L1, L2 = case["B"], case["L1"], case["L2"]
    # the expected cells of the lengths' distribution
    lo = _SHORTEST.get(case["kind"], 8)
    cells = B * L1 * L2
    useful = cells if case["lengths"] == "full" else int(cells * (0.5 * (1 + 1 / lo)) ** 2)
    if case["family"] == "nw_affine" and case["lengths"] != "full":
        useful = int(cells * (1 + 1 / lo + 1 / lo ** 2) / 3)
    fwd, adj = useful * _FORWARD[case["family"]], useful * _ADJOINT[case["family"]]
    if case["kind"] == "embed":
        D = case["D"]
        rows = int(B * (L1 + L2) * 0.5 * (1 + 1 / lo))
        # the embeddings in, their gradients out (whole, padding included)
        return {"bytes": 2 * D * (rows + B * (L1 + L2)), "flops": 6 * D * useful + fwd + adj}
    if case["kind"] == "ragged":
        return {"bytes": 8 * useful, "flops": fwd + adj}
    width = 4 if case["dtype"] == "float32" else 2
    masked = cells if case["lengths"] == "mask" else 0
    if case["kind"] == "score":
        return {"bytes": width * useful + masked, "flops": fwd}
    if case["kind"] == "map_step":
        # scores and map gradient in; map and score gradient out (whole)
        return {"bytes": 8 * useful + 8 * cells, "flops": 3 * (fwd + adj)}
    out = 4 if case["kind"] == "map" else width
    return {"bytes": width * useful + masked + out * cells, "flops": fwd + adj}


# --------------------------------------------------------------------------
# The same in 64 bits
# --------------------------------------------------------------------------

_FAR = -1e30  # log weight of what no alignment reaches


def _skew(x):
    """[B, L1, L2] -> L1 + L2 + 1 slices [B, L1 + 1]: entry (b, i) of slice d is
    the score of cell (i, d - i), 1-based, or _FAR outside the matrix."""
    B, L1, L2 = x.shape
    W = L1 + L2 + 2
    y = torch.nn.functional.pad(x, (1, W - L2 - 1, 1, 0), value=_FAR)
    # one column back per row; what would be a negative column is the padding
    # of the row before
    return y.as_strided((L1 + L2 + 1, B, L1 + 1), (1, (L1 + 1) * W, W - 1)).unbind(0)


def _log_partition(family, x, lengths, go, ge):
    """log Z [B] of scores x [B, L1, L2] and gap scores in units of the
    temperature."""
    B, L1, L2 = x.shape
    local, ends_anywhere = family != "nw_affine", family in ("sw", "sw_affine")
    far = torch.full_like(go, _FAR)
    d_to_i = go if family in ("sw", "nw_affine") else far
    i_to_d = go if family in ("sw", "nw_affine", "sv_affine") else far
    into_i = torch.stack([go, ge, d_to_i]).reshape(3, -1, 1)
    into_d = torch.stack([go, i_to_d, ge]).reshape(3, -1, 1)
    X = _skew(x)
    n1, n2 = (lengths[:, k, None].to(x.device) for k in (0, 1))
    i = torch.arange(L1 + 1, device=x.device)[None, :]
    edge = torch.full((3, B, 1), _FAR, dtype=x.dtype, device=x.device)
    none = torch.full((3, B, L1 + 1), _FAR, dtype=x.dtype, device=x.device)
    two, one = none, none
    if not local:  # the empty alignment of two empty prefixes
        one = none.clone()
        one[0, :, 0] = 0.0
    totals, finals = [torch.zeros(B, dtype=x.dtype, device=x.device)], None
    for d in range(1, L1 + L2 + 1):
        up = torch.cat([edge, one[:, :, :-1]], dim=2)
        diag = torch.cat([edge, two[:, :, :-1]], dim=2)
        a = torch.logsumexp(diag, dim=0)
        if local:
            a = torch.logaddexp(a, torch.zeros_like(a))
        M = X[d] + a
        now = torch.stack([M, torch.logsumexp(up + into_i, dim=0), torch.logsumexp(one + into_d, dim=0)])
        inside = (i <= d) & (d - i <= n2) & (i <= n1)
        if local:
            inside = inside & (i >= 1) & (d - i >= 1)
            ends = now if ends_anywhere else now[:1]
            totals.append(torch.logsumexp(torch.where(inside, ends, _FAR), dim=(0, 2)))
        else:
            last = torch.where((i == n1) & (d - i == n2), now, _FAR)
            final = torch.logsumexp(last, dim=(0, 2))
            finals = final if finals is None else torch.maximum(finals, final)
        two, one = one, torch.where(inside, now, _FAR)
    return torch.logsumexp(torch.stack(totals), dim=0) if local else finals


def _value64(family, x, lengths, excluded, go, ge, T):
    y = x / T
    if excluded is not None:
        y = torch.where(excluded, _FAR, y)
    return T * _log_partition(family, y, lengths, go / T, ge / T)


def _params64(c, dev):
    go, ge, T = (torch.tensor(v, dtype=torch.float64, device=dev, requires_grad=True)
                 for v in (c["open"], c["extend"], c["temperature"]))
    return go, go if c["family"] == "sw" else ge, T


def exact(case, seed):
    s = prepare(case, seed)
    c, kind, family = case, case["kind"], case["family"]
    dev = torch.device("cuda")
    host = _lengths(case, seed)
    if case["lengths"] == "mask":  # excluded cells, the padded shape
        lengths, excluded = torch.tensor([[c["L1"], c["L2"]]] * c["B"], dtype=torch.int32), s["mask"]
    else:
        lengths, excluded = host, None
    go, ge, T = _params64(c, dev)
    if kind == "ragged":
        return _exact_ragged(s, host, go, ge, T)
    if kind == "embed":
        Q, K = (s[k].detach().double().requires_grad_() for k in ("Q", "K"))
        value = _in_parts(c, lengths, lambda b, l1, l2: _value64(
            family, Q[b, :l1] @ K[b, :l2].transpose(1, 2).contiguous(), lengths[b], None, go, ge, T), (Q, K), s["weight"])
        return {"value": value, "dQ": Q.grad, "dK": K.grad}
    x = s["scores"].detach().double().requires_grad_()
    if kind == "score":
        with torch.no_grad():
            return {"value": _value64(family, x, lengths, excluded, go, ge, T)}
    if kind == "map_step":
        value = _value64(family, x, lengths, excluded, go, ge, T)
        m, = torch.autograd.grad(value.sum(), x, create_graph=True)
        return {"map": m.detach(), "grads": torch.autograd.grad(m, [x], s["weight"].double())}
    weight = s["weight"].double() if kind == "step" else torch.ones(c["B"], dtype=torch.float64, device=dev)
    value = _in_parts(c, lengths, lambda b, l1, l2: _value64(
        family, x[b, :l1, :l2], lengths[b], None if excluded is None else excluded[b, :l1, :l2], go, ge, T),
        (x, go, ge, T), weight)
    if kind == "map":
        return {"map": x.grad}
    params = [go, T] if family == "sw" else [go, ge, T]
    return {"value": value, "grads": [x.grad, *[p.grad for p in params]] if c["learn"] else [x.grad]}


def _in_parts(c, lengths, value_of, inputs, weight):
    """value_of over the batch, a few hundred million cells at a time, with
    the gradients of sum(weight * value) accumulated in ``inputs``."""
    per = max(1, int(2.8e8 // (c["L1"] * c["L2"])))
    values = []
    for b0 in range(0, c["B"], per):
        b = slice(b0, min(c["B"], b0 + per))
        l1, l2 = (int(v) for v in lengths[b].amax(dim=0))
        v = value_of(b, l1, l2)
        torch.autograd.backward((v * weight[b].double()).sum(), inputs=list(inputs))
        values.append(v.detach())
    return torch.cat(values)


def _exact_ragged(s, host, go, ge, T):
    """Pairs of similar size together, padded to their largest."""
    c, dev = s["case"], s["scores"].device
    offsets, _ = _offsets(host)
    order = torch.argsort(host.amax(dim=1).long() * (1 << 16) + host.amin(dim=1).long(), descending=True)
    B = c["B"]
    value = torch.empty(B, dtype=torch.float64, device=dev)
    flat = torch.empty(s["scores"].numel(), dtype=torch.float64, device=dev)
    per_pair = torch.empty(3, B, dtype=torch.float64, device=dev)
    at = 0
    while at < B:
        top = int(host[order[at]].amax())
        part = order[at:at + max(1, int(2.8e8 // (top * top)))]
        at += len(part)
        ln = host[part]
        l1, l2 = (int(v) for v in ln.amax(dim=0))
        lnd = ln.to(dev)
        rows, cols = torch.arange(l1, device=dev)[None, :, None], torch.arange(l2, device=dev)[None, None, :]
        index = offsets[part].to(dev)[:, None, None] + rows * lnd[:, 1, None, None] + cols
        outside = _mask(lnd, l1, l2)
        index = torch.where(outside, 0, index)
        x = s["scores"][index].double().requires_grad_()
        p = [q.detach().expand(len(part)).clone().reshape(-1, 1, 1).requires_grad_() for q in (go, ge, T)]
        v = _value64_pairs(c["family"], x, ln, p)
        grads = torch.autograd.grad(v.sum(), [x, *p])
        value[part.to(dev)] = v.detach()
        flat[index[~outside]] = grads[0][~outside]
        for k in range(3):
            per_pair[k, part.to(dev)] = grads[1 + k].reshape(-1)
    return {"value": value, "map": flat, "d_open": per_pair[0], "d_extend": per_pair[1], "d_temperature": per_pair[2]}


def _value64_pairs(family, x, lengths, params):
    """The value with each pair's own parameters [n, 1, 1]."""
    go, ge, T = params
    return T.reshape(-1) * _log_partition(family, x / T, lengths, (go / T).reshape(-1), (ge / T).reshape(-1))
