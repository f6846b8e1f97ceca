"""The work that is timed: what a program that serves a GRINQH-quantized model has this package do.

A case is a dict of plain values.  ``kind`` says which public entry points it goes through:

* ``linears``: quantized linears, each on an input of its own, through ``torch.ops.grinqh.gemm_or_gemv``
  (``mode`` "reference": one row graded, more rows dense) or ``grinqh_gemv_batch_union`` ("union": every batch
  graded on its column maxima).  ``layers`` repeats the shapes with other weights, as the layers of a model do.
* ``mlp``: a decoder's MLP half with the producers that emit the grading statistic: ``rmsnorm_sigma`` (with the
  residual add) and gate_up, ``silu_mul_sigma`` and down.  The activation starts from a given gate_up result, so that a
  last bit of the first product cannot move a channel across a threshold of the second.
* ``load``: ``prepare_weight``, the repack that every weight goes through when a checkpoint is loaded.

``graph`` true replays the calls as one captured HIP graph, the way a serving loop runs its decode steps; false
calls them eagerly.  Shapes are those of bench.py (Llama-3-8B and 70B linears) and generic ragged ones; weights are
symmetric round-to-nearest codes of 0.02 N(0, 1) per scale group, activations N(0, 1) with 1 % of the channels
20 times larger, thresholds percentiles of the batch's channel maxima.
"""
from __future__ import annotations

import math
import os
import sys

import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "vllm-grinqh-plugin_amd"))

import grinqh.kernel as gk  # noqa: E402  (registers torch.ops.grinqh)
from grinqh.producer import gemv_batch_union_sigma, rmsnorm_sigma, silu_mul_sigma  # noqa: E402
from grinqh.utils import prepare_weight  # noqa: E402

EPS = 1e-5
DTYPES = {"f16": torch.float16, "bf16": torch.bfloat16}

# (K, N) of the linears of one layer
SHAPES = {
    "8b": ((4096, 6144), (4096, 4096), (4096, 28672), (14336, 4096)),   # qkv, o_proj, gate_up, down
    "8b_qkv": ((4096, 6144),),
    "8b_o": ((4096, 4096),),
    "8b_gate_up": ((4096, 28672),),
    "8b_down": ((14336, 4096),),
    "70b_qkv": ((8192, 10240),),
    "70b_gate_up": ((8192, 57344),),
    "70b_down": ((28672, 8192),),
    "ragged": ((2080, 6160),),          # a row count past the scale groups, a partial column block
    "ragged_wide": ((3168, 11216),),
    "small": ((1024, 2560), (1024, 1024), (1024, 5632), (2816, 1024)),
}


def _case(name, kind, shape, rows, **more):
    c = {"kind": kind, "shape": shape, "rows": rows, "dtype": "f16", "bits": 8, "group": 128, "mode": "reference",
         "bias": False, "graph": False, "layers": 1}
    c.update(more)
    if name:
        c["name"] = name
    return c


def listed():
    return [
        # a single call of the op for one token: launches and host time are all there is
        _case("op_1row", "linears", "8b_qkv", 1),
        # the same entry point with the other options: bf16, 4 bits, short scale groups, bias, ragged sizes
        _case("op_3rows_ragged", "linears", "ragged", 3, dtype="bf16", bits=4, group=64, mode="union", bias=True),
        # one decode step of a single sequence: every linear of four layers, graded, weights from HBM
        _case("step_1row", "linears", "8b", 1, graph=True, layers=4),
        # small serving batches under the default dispatch (dense above one row)
        _case("step_16rows", "linears", "8b", 16, graph=True, layers=2),
        # larger batches, graded on the batch
        _case("step_47rows_union", "linears", "8b", 47, mode="union", graph=True, layers=2),
        # the same range in bf16, the dtype most checkpoints run in
        _case("step_64rows_bf16", "linears", "8b", 64, dtype="bf16", graph=True, layers=2),
        # decode through the fused producers: norm, gate_up, activation, down
        _case("mlp_32rows", "mlp", "8b", 32, mode="union", graph=True, layers=2),
        # short prompts and chunked prefill
        _case("prefill_150rows", "linears", "8b", 150),
        _case("prefill_390rows_bf16", "linears", "8b", 390, dtype="bf16", mode="union"),
        # long prompts
        _case("prefill_2048rows_bf16", "linears", "8b", 2048, dtype="bf16"),
        _case("prefill_4096rows_70b", "linears", "70b_gate_up", 4096, mode="union"),
        # loading a layer of a checkpoint
        _case("load_layer", "load", "8b", 0),
    ]


def draw(rng):
    kind = rng.choices(("linears", "mlp", "load"), (16, 2, 1))[0]
    if kind == "load":
        return _case(None, kind, rng.choice(list(SHAPES)), 0, bits=rng.choice((8, 8, 6, 4, 2)), layers=rng.randint(1, 3))
    dtype = rng.choice(("f16", "bf16"))
    if kind == "mlp":
        return _case(None, kind, rng.choice(("8b", "small")), rng.randint(1, 64), dtype=dtype, mode="union",
                     graph=rng.random() < 0.7, layers=rng.randint(1, 3), bits=rng.choice((8, 8, 8, 6, 4)))
    # rows over their logarithm, decode and prefill alike
    rows = int(round(math.exp(rng.uniform(0.0, math.log(4096.0)))))
    shape = rng.choice(("8b", "8b", "8b", "8b_gate_up", "8b_down", "70b_qkv", "70b_down", "ragged", "ragged_wide", "small"))
    return _case(None, kind, shape, rows, dtype=dtype, mode=rng.choice(("reference", "union")),
                 bits=rng.choice((8, 8, 8, 6, 4, 2)), group=rng.choice((128, 128, 128, 64, 32)),
                 bias=rng.random() < 0.2, graph=rows <= 64 and rng.random() < 0.7,
                 layers=rng.randint(1, 3) if rows <= 256 else 1)


# ---------------------------------------------------------------- inputs

def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _weight(g, K, N, case):
    """(codes int8 [K, N], scales [ceil(K / group), N])"""
    gs, lim = case["group"], (1 << (case["bits"] - 1)) - 1
    groups = -(-K // gs)
    w = 0.02 * torch.randn((groups * gs, N), generator=g, device="cuda")
    w[K:] = 0.0
    w = w.view(groups, gs, N)
    s = (w.abs().amax(1) / lim).clamp_min(1e-8) if lim else w.abs().amax(1)
    s = s.to(DTYPES[case["dtype"]])
    q = torch.round(w / s.float().unsqueeze(1)).clamp_(-lim - 1, lim).to(torch.int8)
    return q.view(groups * gs, N)[:K].contiguous(), s


def _activations(g, rows, K, case):
    x = torch.randn((rows, K), generator=g, device="cuda")
    loud = torch.randperm(K, generator=g, device="cuda")[: -(-K // 100)]
    x[:, loud] *= 20
    return x.to(DTYPES[case["dtype"]])


def _thresholds(x, case):
    """Percentiles of the channel maxima, each moved to the widest gap nearby, as a calibration that is to hold
    under rounding would place them."""
    if case["mode"] == "reference" and case["rows"] > 1:
        return [0.0, 0.0, 0.0, 0.0]     # not graded
    v = x.double().abs().amax(0).sort().values
    n, t = v.numel(), [0.0]
    for q in (0.5, 0.8, 0.95) if case["rows"] <= 64 else (0.7, 0.9, 0.98):
        i = min(int(q * n), n - 34)
        near = v[max(i - 32, 0):i + 33]
        j = int((near[1:] - near[:-1]).argmax())
        t.append(float((near[j] + near[j + 1]) / 2))
    return t


def _shapes(case):
    s = SHAPES[case["shape"]]
    return (s[2:] if case["kind"] == "mlp" else s) * case["layers"]


def _inputs(case, seed):
    """What both the calls and exact() start from."""
    g = _generator(seed)
    if case["kind"] == "load":
        return [{"codes": _weight(g, K, N, case)[0]} for K, N in _shapes(case)]
    dtype, items = DTYPES[case["dtype"]], []
    if case["kind"] == "linears":
        for K, N in _shapes(case):
            codes, scale = _weight(g, K, N, case)
            x = _activations(g, case["rows"], K, case)
            bias = torch.randn(N, generator=g, device="cuda").to(dtype) if case["bias"] else None
            items.append({"codes": codes, "scale": scale, "x": x, "bias": bias, "thr": _thresholds(x, case)})
        return items
    shapes = _shapes(case)
    for k in range(0, len(shapes), 2):
        (H, F2), (F, _) = shapes[k], shapes[k + 1]
        up, down = _weight(g, H, F2, case), _weight(g, F, H, case)
        h = 0.1 * _activations(g, case["rows"], H, case)
        res = torch.randn((case["rows"], H), generator=g, device="cuda").to(dtype)
        norm = (1 + 0.1 * torch.randn(H, generator=g, device="cuda")).to(dtype)
        it = {"codes": up[0], "scale": up[1], "codes2": down[0], "scale2": down[1], "h": h, "res": res, "norm": norm}
        y = _norm(it, dtype, torch.float32)[0]
        it["thr"] = _thresholds(y, case)
        it["gu"] = _product(y, *up, it["thr"], None, case, torch.float32).to(dtype)
        it["thr2"] = _thresholds(_activation(it["gu"], dtype, torch.float32), case)
        items.append(it)
    return items


# ---------------------------------------------------------------- the calls

_side_stream = None


def _pack(item, case):
    item = dict(item)
    for c in ("codes", "codes2"):
        if c in item:
            item[c.replace("codes", "planes")] = prepare_weight(item.pop(c), case["bits"])
    return item


def prepare(case, seed):
    items = _inputs(case, seed)
    if case["kind"] == "load":
        return {"case": case, "items": items}
    st = {"case": case, "items": [_pack(i, case) for i in items]}
    if case["graph"]:
        # as a serving loop does: warmed up and captured on a stream of its own, then replayed for every step
        global _side_stream
        if _side_stream is None:
            _side_stream = torch.cuda.Stream()
        _side_stream.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(_side_stream):
            _calls(st)
        torch.cuda.synchronize()
        st["graph"] = torch.cuda.CUDAGraph()
        with torch.cuda.graph(st["graph"], stream=_side_stream):
            st["out"] = _calls(st)
    return st


def _calls(st):
    c, out = st["case"], []
    bits, gs = c["bits"], c["group"]
    if c["kind"] == "load":
        return [prepare_weight(i["codes"], bits).view(torch.int32) for i in st["items"]]
    if c["kind"] == "mlp":
        for i in st["items"]:
            y, sig, res = rmsnorm_sigma(i["h"], i["norm"], EPS, i["res"])
            gu = gemv_batch_union_sigma(y, i["planes"], i["scale"], None, bits, gs, i["scale"].shape[1] // 4, i["thr"], sig)
            a, asig = silu_mul_sigma(i["gu"])
            d = gemv_batch_union_sigma(a, i["planes2"], i["scale2"], None, bits, gs, i["scale2"].shape[1] // 4, i["thr2"], asig)
            out.append([res, y, gu, a, d])
        return out
    for i in st["items"]:
        n4 = i["scale"].shape[1] // 4
        if c["mode"] == "union":
            out.append(gk.grinqh_gemv_batch_union(i["x"], i["planes"], i["scale"], i["bias"], bits, gs, n4, i["thr"]))
        else:
            out.append(torch.ops.grinqh.gemm_or_gemv(i["x"], i["planes"], i["scale"], i["bias"], bits, gs, n4, i["thr"]))
    return out


def run(state):
    if "graph" in state:
        state["graph"].replay()
        return state["out"]
    return _calls(state)


# ---------------------------------------------------------------- work, tolerance, exact results

def work(case):
    rows, bits = case["rows"], case["bits"]
    total = {"bytes": 0.0, "flops": 0.0}
    if case["kind"] == "load":
        for K, N in _shapes(case):
            total["bytes"] += K * N + K * N * bits / 8
        return total
    planes = float(bits // 2)
    if case["mode"] == "union" or rows == 1:     # planes that the grading needs, on average
        more = (0.5, 0.2, 0.05) if rows <= 64 else (0.3, 0.1, 0.02)
        planes = 1.0 + sum(more[: bits // 2 - 1])
    for K, N in _shapes(case):
        total["bytes"] += planes * K * N / 4 + 2 * N * -(-K // case["group"]) + 2 * rows * (K + N) + 2 * N * case["bias"]
        total["flops"] += 2 * rows * K * N
    if case["kind"] == "mlp":   # the norm's and the activation's own inputs and outputs
        for (H, F2), (F, _) in zip(_shapes(case)[0::2], _shapes(case)[1::2]):
            total["bytes"] += 2 * rows * (4 * H + 3 * F) + 2 * H
    return total


def tolerance(case):
    if case["kind"] == "load":
        return "exact"
    # one rounding of the output, and on some paths one of the scaled weight: 2^-11 (f16) or 2^-8 (bf16) at most,
    # about 0.4 of that in the 2-norm; a bias adds a rounding, a product after a norm or an activation two
    unit = 2.0 ** -11 if case["dtype"] == "f16" else 2.0 ** -8
    return {"rel": (4 if case["kind"] == "mlp" else 1.5) * unit, "max": (40 if case["kind"] == "mlp" else 8) * unit}


def _norm(i, dtype, wide):
    h = (i["h"].to(wide) + i["res"].to(wide)).to(dtype)
    v = h.to(wide)
    y = (v * torch.rsqrt(v.square().mean(-1, keepdim=True) + EPS)).to(dtype)
    return (y.to(wide) * i["norm"].to(wide)).to(dtype), h


def _activation(gu, dtype, wide):
    g, u = gu.to(dtype).to(wide).chunk(2, -1)
    return (torch.nn.functional.silu(g).to(dtype).to(wide) * u).to(dtype)


def _product(x, codes, scale, thr, bias, case, wide):
    """x @ (w_eff * scale) (+ bias) unrounded, w_eff from the zones that each channel's maximum reaches."""
    K, N, bits, gs = codes.shape[0], codes.shape[1], case["bits"], case["group"]
    w = codes
    if case["mode"] == "union" or x.shape[0] == 1:
        top = x.float().abs().amax(0)
        keep, beta, last = torch.zeros(K, dtype=torch.int32, device=x.device), torch.zeros(K, dtype=torch.int32, device=x.device), 0
        for z in range(bits // 2):
            on = (top > torch.tensor(thr[z], dtype=torch.float32)).int()
            mid = (1 << (bits - 1)) >> (2 * z + 2)
            keep |= on * (3 << (bits - 2 - 2 * z))
            beta += on * (mid - last)
            last = mid
        sign = -(1 << (bits - 1))
        u = codes.int() & ((1 << bits) - 1) & keep.unsqueeze(1)
        w = torch.where(u >= -sign, u + 2 * sign, u) + beta.unsqueeze(1)
    y = torch.zeros((x.shape[0], N), dtype=wide, device=x.device)
    step = max(1, 4096 // gs) * gs
    for k in range(0, K, step):     # by parts of K: the 64-bit weight need not be held whole
        e = min(K, k + step)
        s = scale[k // gs:-(-e // gs)].to(wide).repeat_interleave(gs, 0)[: e - k]
        y += x[:, k:e].to(wide) @ (w[k:e].to(wide) * s)
    return y if bias is None else y + bias.to(wide)


def exact(case, seed):
    if case["kind"] == "load":
        return None
    dtype, out = DTYPES[case["dtype"]], []
    for i in _inputs(case, seed):
        if case["kind"] == "linears":
            out.append(_product(i["x"], i["codes"], i["scale"], i["thr"], i["bias"], case, torch.float64))
            continue
        # the products in 64 bits from what the norm and the activation hand over in the activation dtype
        y, h = _norm(i, dtype, torch.float64)
        gu = _product(y, i["codes"], i["scale"], i["thr"], None, case, torch.float64)
        a = _activation(i["gu"], dtype, torch.float64)
        d = _product(a, i["codes2"], i["scale2"], i["thr2"], None, case, torch.float64)
        out.append([h.double(), y.double(), gu, a.double(), d])
    return out
