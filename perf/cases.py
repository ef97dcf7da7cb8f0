"""The work that a program using this package has it do, as cases to be timed.

A case is one of three things:

* ``layer``: the four int4 projections of a decoder layer, for ``m`` tokens, in ``layers`` layers one after
  another: RMSNorm + QKV (``rmsnorm_awq_fused_linear``, reference layout), the attention output, gate and
  up together, and down (``AWQWeight`` / ``PackedInt4Weight.matmul``).  Each projection has an input of its
  own, so an output depends on one projection and its tolerance on one rounding.
* ``mlp``: the gated MLP of one decoded token over symmetric group-32 weights: the fused gate / up /
  activation launch, then the down projection (again on an input of its own).
* ``moe``: ``fused_moe`` (routing, gated int4 experts, the weighted sum).

``captured`` cases are decode steps: a serving loop captures its step once, as a HIP graph over buffers that
it keeps, and replays it for every token.  The others are eager calls, as prefill runs them.
"""
import torch

from litevllm_amd import (AWQExperts, AWQWeight, PackedInt4Weight, fused_moe,
                          packed_int4_symmetric_fused_gate_up_m1, rmsnorm_awq_fused_linear)
from litevllm_amd import ops

DEVICE = "cuda"
DTYPES = {"f16": torch.float16, "bf16": torch.bfloat16}
EPS = 1e-6


def _layer(name, m, dtype="f16", hidden=4096, qkv=6144, inter=12288, group=128, zeros=True, bias=False, layers=1, captured=False):
    return {"name": name, "kind": "layer", "m": m, "dtype": dtype, "hidden": hidden, "qkv": qkv, "inter": inter,
            "group": group, "zeros": zeros, "bias": bias, "layers": layers, "captured": captured}


def _mlp(name, dtype, hidden, inter, layers, captured):
    return {"name": name, "kind": "mlp", "m": 1, "dtype": dtype, "hidden": hidden, "inter": inter, "layers": layers,
            "captured": captured}


def _moe(name, m, dtype="f16", experts=64, topk=8, hidden=2048, inter=1024, group=128, captured=False):
    return {"name": name, "kind": "moe", "m": m, "dtype": dtype, "experts": experts, "topk": topk, "hidden": hidden,
            "inter": inter, "group": group, "captured": captured}


def listed():
    return [
        # one user, one token: each launch is a few microseconds
        _layer("decode-1", 1, layers=3, captured=True),
        # a small batch of a bf16 model
        _layer("decode-8-bf16", 8, "bf16", layers=2, captured=True),
        # an ordinary serving batch
        _layer("decode-32", 32, layers=2, captured=True),
        # a large, ragged serving batch, with a bias on the attention output
        _layer("decode-57", 57, bias=True, layers=2, captured=True),
        # a short prompt, or a chunk of one beside a decode batch
        _layer("chunk-200", 200, layers=2),
        # a long prompt
        _layer("prefill-2048", 2048),
        # a prompt of odd length on a bf16 model
        _layer("prefill-1000-bf16", 1000, "bf16"),
        # the layer of a small model called eagerly, one token: host time and launches count
        _layer("eager-small", 1, hidden=2048, qkv=2560, inter=5632),
        # the symmetric group-32 MLP of a dense model, one token
        _mlp("mlp-g32-1", "bf16", 5376, 21504, 1, True),
        # a decode batch through 64 experts
        _moe("moe-16", 16, captured=True),
        # a prompt through 64 experts
        _moe("moe-512", 512),
        # a part of a prompt on a bf16 model
        _moe("moe-130-bf16", 130, "bf16"),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(lo * (hi / lo) ** rng.random()))))


def draw(rng):
    kind = rng.choice(("layer", "layer", "layer", "moe", "moe", "mlp"))
    if kind == "mlp":
        c = _mlp("", rng.choice(("f16", "bf16")), 128 * rng.randint(8, 42), 8 * _log_int(rng, 88, 2688), rng.choice((1, 2)),
                 rng.random() < 0.7)
    elif kind == "moe":
        group = rng.choice((32, 64, 128, 128))
        c = _moe("", _log_int(rng, 1, 512), rng.choice(("f16", "f16", "bf16")), rng.choice((16, 32, 64)), rng.choice((2, 4, 8)),
                 128 * rng.randint(8, 16), 128 * rng.randint(2, 8), group, rng.random() < 0.5)
    else:
        m = _log_int(rng, 1, 2048)
        c = _layer("", m, rng.choice(("f16", "f16", "bf16")), 128 * rng.randint(8, 32), 8 * _log_int(rng, 160, 768),
                   128 * _log_int(rng, 10, 96), rng.choice((32, 64, 128, 128)), rng.random() < 0.7, rng.random() < 0.3,
                   2 if m <= 64 else 1, m <= 64)
    del c["name"]
    return c


# ------------------------------------------------------------------ inputs
class _Made:
    """Seeded inputs: int4 values uniform, scales |N(0, 0.02)| + 1e-4, activations N(0, 1)."""

    def __init__(self, seed):
        self.g = torch.Generator(device=DEVICE)
        self.g.manual_seed(int(seed))

    def words(self, *shape):
        return torch.randint(-2 ** 31, 2 ** 31, shape, generator=self.g, device=DEVICE, dtype=torch.int64).to(torch.int32)

    def normal(self, *shape, dtype=torch.float16, scale=1.0):
        return (torch.randn(shape, generator=self.g, device=DEVICE) * scale).to(dtype)

    def scales(self, *shape):
        return (torch.randn(shape, generator=self.g, device=DEVICE).abs() * 0.02 + 1e-4).to(torch.float16)

    def rows(self, m, k, dtype):
        """Activations with 0.1 % of the channels 20 times as large, as in trained models."""
        x = torch.randn((m, k), generator=self.g, device=DEVICE)
        x[:, torch.randperm(k, generator=self.g, device=DEVICE)[: max(1, k // 1000)]] *= 20.0
        return x.to(dtype)


def _weight(made, k, n, group, zeros):
    """Packed tensors of one projection: AutoAWQ layout with zero points, reference layout without."""
    if zeros:
        return {"layout": "autoawq", "qweight": made.words(k, n // 8), "scales": made.scales(k // group, n),
                "qzeros": made.words(k // group, n // 8)}
    return {"layout": "ref", "qweight": made.words(n, k // 8), "scales": made.scales(n, k // group), "qzeros": None}


def _linear(w, group, prefix):
    if w["qzeros"] is None:
        return PackedInt4Weight(w["qweight"], w["scales"], group_size=group, prefix=prefix, profile_hint="qwen35_9b_awq")
    return AWQWeight(w["qweight"], w["scales"], w["qzeros"], group_size=group, prefix=prefix, profile_hint="qwen35_9b_awq",
                     layout="autoawq")


def _layer_data(case, seed):
    made, dt = _Made(seed), DTYPES[case["dtype"]]
    m, h, i, g = case["m"], case["hidden"], case["inter"], case["group"]
    data = []
    for _ in range(case["layers"]):
        groups = h // g
        qkv = {"layout": "ref", "qweight": made.words(case["qkv"], h // 8), "scales": made.scales(case["qkv"], groups),
               "qzeros": made.words(case["qkv"], (groups + 7) // 8) if case["zeros"] else None}
        data.append({
            "qkv": qkv, "o": _weight(made, h, h, g, case["zeros"]), "gate_up": _weight(made, h, 2 * i, g, case["zeros"]),
            "down": _weight(made, i, h, g, case["zeros"]), "norm": made.normal(h, dtype=dt, scale=0.1) + 1.0,
            "bias": made.normal(h, dtype=dt) if case["bias"] else None,
            "x_qkv": made.rows(m, h, dt), "x_o": made.normal(m, h, dtype=dt), "x_gate_up": made.rows(m, h, dt),
            "x_down": made.normal(m, i, dtype=dt)})
    return data


def _mlp_data(case, seed):
    made, dt = _Made(seed), DTYPES[case["dtype"]]
    h, i = case["hidden"], case["inter"]
    return [{"gate": _weight(made, h, i, 32, False), "up": _weight(made, h, i, 32, False),
             "down": _weight(made, i, h, 32, False) if i % 32 == 0 else None,
             "x": made.normal(1, h, dtype=dt), "x_down": made.normal(1, i, dtype=dt)} for _ in range(case["layers"])]


def _moe_data(case, seed):
    made, dt = _Made(seed), DTYPES[case["dtype"]]
    e, h, i, g = case["experts"], case["hidden"], case["inter"], case["group"]

    def stack(k, n):
        return {"qweight": made.words(e, k, n // 8), "scales": made.scales(e, k // g, n), "qzeros": made.words(e, k // g, n // 8)}

    return {"gate_up": stack(h, 2 * i), "down": stack(i, h), "x": made.normal(case["m"], h, dtype=dt),
            "logits": made.normal(case["m"], e, dtype=dt)}


# ------------------------------------------------------------------ the calls
def _layer_pass(case, data, linears):
    out = []
    for d, lin in zip(data, linears):
        q = d["qkv"]
        out.append(rmsnorm_awq_fused_linear(d["x_qkv"], q["qweight"], q["scales"], q["qzeros"], case["group"], d["norm"], EPS))
        out.append(lin["o"].matmul(d["x_o"], d["bias"]))
        out.append(lin["gate_up"].matmul(d["x_gate_up"]))
        out.append(lin["down"].matmul(d["x_down"]))
    return out


def _mlp_pass(case, data, linears):
    out = []
    for d, lin in zip(data, linears):
        out.append(packed_int4_symmetric_fused_gate_up_m1(d["x"], d["gate"]["qweight"], d["up"]["qweight"], d["gate"]["scales"],
                                                          d["up"]["scales"], 32, activation="gelu_pytorch_tanh"))
        if lin is not None:
            out.append(lin.matmul(d["x_down"]))
    return out


def _moe_pass(case, data, experts):
    return [fused_moe(data["x"], experts[0], experts[1], data["logits"], case["topk"])]


def prepare(case, seed):
    if case["kind"] == "layer":
        data = _layer_data(case, seed)
        linears = [{k: _linear(d[k], case["group"], "layers.0.%s" % k) for k in ("o", "gate_up", "down")} for d in data]
        call = _layer_pass
    elif case["kind"] == "mlp":
        data = _mlp_data(case, seed)
        linears = [_linear(d["down"], 32, "layers.0.mlp.down_proj") if d["down"] is not None else None for d in data]
        call = _mlp_pass
    else:
        data = _moe_data(case, seed)
        linears = [AWQExperts(**data[k], group_size=case["group"], layout="autoawq") for k in ("gate_up", "down")]
        ops.prepare_moe_stream(data["gate_up"]["qweight"], True)
        ops.prepare_moe_stream(data["down"]["qweight"], False)
        call = _moe_pass
    state = {"case": case, "call": call, "data": data, "linears": linears, "graph": None}
    call(case, data, linears)  # a program warms its weights up: the kernels' copies of them are built here
    if case["captured"]:
        torch.cuda.synchronize()
        state["graph"] = torch.cuda.CUDAGraph()
        with torch.cuda.graph(state["graph"]):
            state["out"] = call(case, data, linears)
    return state


def run(state):
    if state["graph"] is not None:
        state["graph"].replay()
        return state["out"]
    return state["call"](state["case"], state["data"], state["linears"])


# ------------------------------------------------------------------ what a pass cannot do without
def _gemm_work(m, k, n, group, zeros, bias=False):
    groups = k // group
    b = k * n // 2 + groups * n * 2 + (groups * n // 2 if zeros else 0) + m * (k + n) * 2 + (2 * n if bias else 0)
    return b, 2 * m * k * n


def work(case):
    m, h, i = case["m"], case["hidden"], case["inter"]
    if case["kind"] == "layer":
        g, z = case["group"], case["zeros"]
        parts = [_gemm_work(m, h, case["qkv"], g, z), _gemm_work(m, h, h, g, z, case["bias"]), _gemm_work(m, h, 2 * i, g, z),
                 _gemm_work(m, i, h, g, z), (2 * h, 4 * m * h)]
        return {"bytes": case["layers"] * sum(p[0] for p in parts), "flops": case["layers"] * sum(p[1] for p in parts)}
    if case["kind"] == "mlp":
        b, f = _gemm_work(1, h, 2 * i, 32, False)
        b -= 2 * i  # the activated product has half as many columns
        if i % 32 == 0:
            bd, fd = _gemm_work(1, i, h, 32, False)
            b, f = b + bd, f + fd
        return {"bytes": case["layers"] * b, "flops": case["layers"] * f}
    # experts that a uniform router reaches at least once
    e, k, g = case["experts"], case["topk"], case["group"]
    reached = e * (1.0 - (1.0 - k / e) ** m)
    per = 3 * h * i // 2 + (h // g * 2 * i + i // g * h) * 2 + (h // g * 2 * i + i // g * h) // 2
    return {"bytes": int(reached * per + m * (2 * h + e) * 2), "flops": 2 * m * k * 3 * h * i}


def tolerance(case):
    # outputs are rounded once to 16 bits from 32-bit sums; weights are rounded to 16 bits or not, by path
    # (measured against exact() on MI355X: f16 2.0e-4 to 4.6e-4, bf16 1.6e-3 to 3.7e-3)
    if case["dtype"] == "f16":
        return {"rel": 1.6e-3, "max": 8e-3}
    return {"rel": 1e-2, "max": 4e-2}


# ------------------------------------------------------------------ 64-bit answers
_AWQ_ORDER = (0, 2, 4, 6, 1, 3, 5, 7)  # nibble i of an AutoAWQ word is this column


def _unpack(words, autoawq):
    """int32 [..., w] -> [..., 8 w] values 0 .. 15."""
    nib = torch.stack([(words >> (4 * i)) & 15 for i in range(8)], dim=-1)
    if autoawq:
        nib = nib[..., [_AWQ_ORDER.index(c) for c in range(8)]]
    return nib.flatten(-2)


def _dense(w, group):
    """The weight as a 64-bit [K, N] matrix."""
    auto = w.get("layout", "autoawq") == "autoawq"
    q = _unpack(w["qweight"], auto)
    s = w["scales"].double()
    if auto:
        z = _unpack(w["qzeros"], True) if w["qzeros"] is not None else 8
        z = z.repeat_interleave(group, 0) if w["qzeros"] is not None else z
        return (q - z).double() * s.repeat_interleave(group, 0)
    if w["qzeros"] is None:
        return ((q - 8).double() * s.repeat_interleave(group, 1)).t()
    z = _unpack(w["qzeros"], False)[:, : s.shape[1]]
    return ((q - z.repeat_interleave(group, 1)).double() * s.repeat_interleave(group, 1)).t()


def _act(g, silu):
    if silu:
        return g * torch.sigmoid(g)
    return g * torch.sigmoid(2 * 0.7978845608028654 * (g + 0.044715 * g ** 3))


def exact(case, seed):
    if case["kind"] == "layer":
        out = []
        for d in _layer_data(case, seed):
            x = d["x_qkv"].double()
            x = x * torch.rsqrt((x * x).mean(1, keepdim=True) + EPS) * d["norm"].double()
            out.append(x @ _dense(d["qkv"], case["group"]))
            y = d["x_o"].double() @ _dense(d["o"], case["group"])
            out.append(y + d["bias"].double() if d["bias"] is not None else y)
            out.append(d["x_gate_up"].double() @ _dense(d["gate_up"], case["group"]))
            out.append(d["x_down"].double() @ _dense(d["down"], case["group"]))
        return out
    if case["kind"] == "mlp":
        out = []
        for d in _mlp_data(case, seed):
            x = d["x"].double()
            out.append(_act(x @ _dense(d["gate"], 32), False) * (x @ _dense(d["up"], 32)))
            if d["down"] is not None:
                out.append(d["x_down"].double() @ _dense(d["down"], 32))
        return out
    # the router rounds its probabilities to the logits' type: ties go to the lower expert
    d = _moe_data(case, seed)
    i, x = case["inter"], d["x"].double()
    p = torch.softmax(d["logits"].double(), -1).to(d["logits"].dtype)
    w, ids = torch.sort(p.float(), dim=-1, descending=True, stable=True)
    w, ids = w[:, : case["topk"]].to(p.dtype), ids[:, : case["topk"]]
    w = (w / w.sum(-1, keepdim=True)).double()
    out = torch.zeros_like(x)
    for e in range(case["experts"]):
        rows, slot = (ids == e).nonzero(as_tuple=True)
        if rows.numel() == 0:
            continue
        part = {k: {n: t[e] for n, t in d[k].items()} for k in ("gate_up", "down")}
        gu = x[rows] @ _dense(part["gate_up"], case["group"])
        y = (_act(gu[:, :i], True) * gu[:, i:]) @ _dense(part["down"], case["group"])
        out.index_add_(0, rows, y * w[rows, slot, None])
    return [out]
