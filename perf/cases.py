"""The work that a user of this package has it do, as cases that can be timed and compared.

Six kinds of case, each through the entry points that a program calls:

* ``layer``    ``ExpertSSDMoE(x)``: one routed-MoE layer, prefill or batched decode, called eagerly
* ``ffn``      ``MoEDecoderFFN(streams)``: the FFN site of a decoder layer (hyper-connection, norm, MoE,
               hyper_residual), called eagerly
* ``verify``   the MoE layers of one few-token step on given hidden states, captured in a HIP graph
* ``step``     one decode step through layers of (RMSNorm + MXFP8 linear + MoE), captured in a HIP graph
* ``linear``   ``DeferredLinear(x)``: a resident linear in bf16, MXFP8 or MXFP4
* ``quantize`` ``DeferredLinear.quantize_to_mxfp``: the start-up conversion of a resident linear

Geometries (d, E, k, I) are the package's own: the small one (1024, 16, 2, 512), the benchmark's
(2048, 128, 8, 768) and the real one (4096, 288, 8, 2048).  Expert codes are uniform E2M1, their scales
have the checkpoint's statistics (two dominant exponents and 1 % others); activations are bf16 N(0, 1),
router weights f32 N(0, 0.02), resident weights bf16 N(0, 0.02).
"""

import math
import os
import sys

import torch

_ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
for _path in (_ROOT, os.path.join(_ROOT, "src")):
    if _path not in sys.path:
        sys.path.insert(0, _path)

from glm53flash.expert_ssd import HBMExpertBank  # noqa: E402
from glm53flash.layers import DeferredLinear  # noqa: E402
from glm53flash.model import MoEDecoderFFN  # noqa: E402
from glm53flash.model_config import GLMTextConfig  # noqa: E402
from glm53flash.moe import ExpertSSDMoE  # noqa: E402
from livglm_amd import native  # noqa: E402

SMALL = {"d": 1024, "E": 16, "k": 2, "I": 512}
BENCH = {"d": 2048, "E": 128, "k": 8, "I": 768}
REAL = {"d": 4096, "E": 288, "k": 8, "I": 2048}
EPS = 1e-6
LIMIT = 10.0
SCALING = 2.5
SINKHORN = 20
HC = 4


def _moe(kind, name, T, geometry, shared="bf16", routing="uniform", **more):
    return {"kind": kind, "name": name, "T": T, **geometry, "shared": shared, "routing": routing, **more}


def listed():
    return [
        # the smallest call there is: one token through a small layer, launched by itself
        _moe("layer", "layer_t1_small", 1, SMALL),
        # single-stream decode: one token through four layers of the stack
        _moe("step", "step_t1", 1, BENCH, layers=4),
        # speculative decode: the two-token verify step
        _moe("verify", "verify_t2", 2, BENCH, layers=4),
        # the same two tokens through the whole FFN site at the real geometry
        _moe("ffn", "ffn_t2_real", 2, REAL),
        # a small decode batch, odd, on a resident MXFP8 shared expert
        _moe("layer", "layer_t23_mxfp8", 23, BENCH, shared="mxfp8"),
        # a decode batch with hot experts
        _moe("layer", "layer_t64_zipf", 64, BENCH, routing="zipf"),
        # a short prompt or a prefill chunk that fills no tile
        _moe("layer", "layer_t333", 333, BENCH),
        # a prompt at the real geometry, resident weights quantised
        _moe("layer", "layer_t1023_real", 1023, REAL, shared="mxfp8"),
        # a long prefill chunk
        _moe("layer", "layer_t4096", 4096, BENCH),
        # a prompt through the FFN site
        _moe("ffn", "ffn_t1500", 1500, BENCH),
        # a prompt through a resident projection of the real width
        {"kind": "linear", "name": "linear_t1500_mxfp8", "T": 1500, "n_in": 4096, "n_out": 4096, "fmt": "mxfp8"},
        # start-up: one resident projection converted
        {"kind": "quantize", "name": "quantize_mxfp8", "n_in": 4096, "n_out": 4096, "bits": 8},
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["layer", "layer", "layer", "layer", "ffn", "ffn", "verify", "step", "linear", "linear",
                       "quantize"])
    if kind == "linear":
        return {"kind": kind, "T": _log_int(rng, 1, 4096), "n_in": 256 * rng.randint(4, 16),
                "n_out": 128 * rng.randint(8, 36), "fmt": rng.choice(["mxfp8", "mxfp8", "mxfp4", "bf16"])}
    if kind == "quantize":
        return {"kind": kind, "n_in": 32 * rng.randint(32, 128), "n_out": _log_int(rng, 500, 4096),
                "bits": rng.choice([8, 8, 4])}
    near = {"d": 512 * rng.randint(2, 6), "E": 8 * rng.randint(8, 20), "k": rng.randint(4, 8),
            "I": 128 * rng.randint(4, 10)}  # a geometry of nobody in particular
    if kind in ("step", "verify"):
        T = 1 if kind == "step" else rng.randint(1, 4)
        return {"kind": kind, "T": T, **rng.choice([BENCH, near, near]), "shared": "bf16", "routing": "uniform",
                "layers": rng.randint(2, 3 if kind == "step" else 8)}
    geometry = rng.choice([BENCH, BENCH, BENCH, REAL, SMALL, near])
    T = _log_int(rng, 1, 1023 if geometry is REAL else 2048 if geometry is near else 4096)
    if kind == "ffn":
        T = min(T, 2048)
    return {"kind": kind, "T": T, **geometry, "shared": rng.choice(["bf16", "bf16", "mxfp8", "mxfp4"]),
            "routing": rng.choice(["uniform", "uniform", "zipf"])}


# ---------------------------------------------------------------- inputs, from the seed alone


class _Draw:
    def __init__(self, seed):
        self.g = torch.Generator(device="cuda")
        self.g.manual_seed(seed)

    def normal(self, *shape, std=1.0, mean=0.0):
        return torch.randn(shape, device="cuda", generator=self.g) * std + mean

    def codes(self, *shape):
        n = math.prod(shape)
        words = torch.randint(-(1 << 63), (1 << 63) - 1, ((n + 7) // 8,), device="cuda", generator=self.g)
        return words.view(torch.uint8)[:n].reshape(shape)

    def scales(self, *shape):
        n = math.prod(shape)
        v = torch.where(torch.rand(n, device="cuda", generator=self.g) < 0.56, 121, 122).to(torch.uint8)
        other = torch.randint(110, 128, (n,), dtype=torch.uint8, device="cuda", generator=self.g)
        odd = torch.rand(n, device="cuda", generator=self.g) < 0.01
        return torch.where(odd, other, v).reshape(shape)

    def order(self, n):
        return torch.randperm(n, device="cuda", generator=self.g)


def _layer_inputs(case, r, forced=False):
    d, E, k, I = case["d"], case["E"], case["k"], case["I"]
    bias = torch.zeros(E, device="cuda")
    if forced:  # the decode trace's routing: a boost that dominates every score
        bias[r.order(E)[:k]] = 10.0
    elif case["routing"] == "zipf":
        bias[r.order(E)] = torch.arange(1, E + 1, device="cuda", dtype=torch.float32) ** -1.1
    out = {"router.weight": r.normal(E, d, std=0.02), "router.bias": bias}
    for part, rows, cols in (("gate_proj", I, d), ("up_proj", I, d), ("down_proj", d, I)):
        out[f"{part}.weight_packed"] = r.codes(E, rows, cols // 2)
        out[f"{part}.weight_scale"] = r.scales(E, rows, cols // 32)
        out[f"shared.{part}"] = r.normal(rows, cols, std=0.02).bfloat16()
    return out


def _hc_inputs(case, r):
    d, M = case["d"], 2 * HC + HC * HC
    return {"streams": r.normal(case["T"], HC, d), "fn": r.normal(M, HC * d, std=0.02),
            "base": r.normal(M, std=0.5), "scale": torch.rand(3, device="cuda", generator=r.g) + 0.5,
            "norm": r.normal(d, std=0.1, mean=1.0).bfloat16().float()}


def _inputs(case, seed):
    r = _Draw(seed)
    if case["kind"] == "linear":
        return {"x": r.normal(case["T"], case["n_in"]).bfloat16(),
                "w": r.normal(case["n_out"], case["n_in"], std=0.02).bfloat16()}
    if case["kind"] == "quantize":
        return {"w": r.normal(case["n_out"], case["n_in"], std=0.02).bfloat16()}
    if case["kind"] == "ffn":
        return {"hc": _hc_inputs(case, r), "layers": [_layer_inputs(case, r)]}
    T, d = case["T"], case["d"]
    got = {"layers": [_layer_inputs(case, r, case["kind"] == "step") for _ in range(case.get("layers", 1))]}
    got["x"] = [r.normal(T, d).bfloat16() for _ in (got["layers"] if case["kind"] == "verify" else range(1))]
    if case["kind"] == "step":
        got["w"] = [r.normal(d, d, std=0.02).bfloat16() for _ in got["layers"]]
        got["norm"] = [r.normal(d, std=0.1, mean=1.0).bfloat16().float() for _ in got["layers"]]
    return got


# ---------------------------------------------------------------- what a program keeps


def _config(case):
    return GLMTextConfig(hidden_size=case["d"], moe_intermediate_size=case["I"], n_routed_experts=case["E"],
                         num_experts_per_tok=case["k"], routed_scaling_factor=SCALING, swiglu_limit=LIMIT,
                         rms_norm_eps=EPS, hc_mult=HC, hc_sinkhorn_iters=SINKHORN, hc_eps=EPS)


def _bank_factory(case, weights):
    def make(layer_idx):
        bank = HBMExpertBank(layer=layer_idx, num_experts=case["E"], hidden_size=case["d"],
                             intermediate_size=case["I"], swiglu_limit=LIMIT, device="cuda")
        bank.load_bank({n: t for n, t in weights.items() if n.endswith(("packed", "scale"))})
        return bank
    return make


def _attach(moe, case, weights):
    moe.gate.weight = weights["router.weight"]
    moe.gate.e_score_correction_bias = weights["router.bias"]
    for part in ("gate_proj", "up_proj", "down_proj"):
        linear = getattr(moe.shared_experts, part)
        linear.weight = weights[f"shared.{part}"]
        if case["shared"] != "bf16":
            linear.quantize_to_mxfp(8 if case["shared"] == "mxfp8" else 4)


def _linear(n_in, n_out, w, bits=None):
    linear = DeferredLinear(n_in, n_out)
    linear.weight = w
    if bits:
        linear.quantize_to_mxfp(bits)
    return linear


def prepare(case, seed):
    got = _inputs(case, seed)
    kind = case["kind"]
    state = {"kind": kind}
    if kind == "linear":
        bits = {"bf16": None, "mxfp8": 8, "mxfp4": 4}[case["fmt"]]
        return {**state, "x": got["x"], "linear": _linear(case["n_in"], case["n_out"], got["w"], bits)}
    if kind == "quantize":
        return {**state, "case": case, "w": got["w"]}
    config = _config(case)
    if kind == "ffn":
        site = MoEDecoderFFN(config, 0, _bank_factory(case, got["layers"][0]))
        _attach(site.mlp, case, got["layers"][0])
        hc = got["hc"]
        site.ffn_hc.fn, site.ffn_hc.base, site.ffn_hc.scale = hc["fn"], hc["base"], hc["scale"]
        site.post_attention_layernorm.weight = hc["norm"]
        return {**state, "streams": hc["streams"], "site": site}
    moes = []
    for i, weights in enumerate(got["layers"]):
        moes.append(ExpertSSDMoE(config, i, _bank_factory(case, weights)))
        _attach(moes[-1], case, weights)
    if kind == "layer":
        return {**state, "x": got["x"][0], "moe": moes[0]}
    # a decode loop's step: run once, then captured
    state.update(moes=moes, x=got["x"], norm=got.get("norm"),
                 linears=[_linear(case["d"], case["d"], w, 8) for w in got.get("w", ())])
    eager = _verify_step if kind == "verify" else _decode_step
    eager(state)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        state["out"] = eager(state)
    state["graph"] = graph
    return state


def _verify_step(state):
    return [(m(x), m.last_weights, m.last_indices) for m, x in zip(state["moes"], state["x"])]


def _decode_step(state):
    x, outs = state["x"][0], []
    for moe, linear, norm in zip(state["moes"], state["linears"], state["norm"]):
        if not outs:
            a = linear(x)
        else:  # the previous layer's f32 output, normed and multiplied in one launch
            T, d = x.shape
            a = torch.empty((T, d), dtype=torch.bfloat16, device="cuda")
            native.call("glm_rms_norm_linear", torch.cuda.current_stream().cuda_stream, x.data_ptr(), T, d,
                        norm.data_ptr(), EPS, linear.weight.data_ptr(), linear.scales.data_ptr(),
                        native.GLM_FMT_MXFP8, d, a.data_ptr())
        x = moe(a)
        outs.append((x, moe.last_weights, moe.last_indices))
    return outs


def run(state):
    kind = state["kind"]
    if kind == "layer":
        moe = state["moe"]
        return moe(state["x"]), moe.last_weights, moe.last_indices
    if kind == "ffn":
        site = state["site"]
        return site(state["streams"]), site.mlp.last_weights, site.mlp.last_indices
    if kind == "linear":
        return state["linear"](state["x"])
    if kind == "quantize":
        case = state["case"]
        linear = _linear(case["n_in"], case["n_out"], state["w"], case["bits"])
        return linear.weight, linear.scales
    state["graph"].replay()
    return state["out"]


# ---------------------------------------------------------------- what a pass cannot do without


def _matrix_bytes(n_out, n_in, fmt):
    return n_out * n_in * {"bf16": 2, "mxfp8": 1 + 1 / 32, "mxfp4": 1 / 2 + 1 / 32}[fmt]


def _moe_work(case, distinct=None):
    T, d, E, k, I = case["T"], case["d"], case["E"], case["k"], case["I"]
    if distinct is None:  # experts that T tokens of uniform routing reach
        distinct = E * (1 - (1 - k / E) ** T)
    b = (3 * _matrix_bytes(I, d, "mxfp4") * distinct + 3 * _matrix_bytes(I, d, case["shared"]) + E * d * 4
         + T * (2 * d + 4 * d + 8 * k))
    return b, 6 * d * I * T * (k + 1) + 2 * E * d * T


def work(case):
    kind = case["kind"]
    if kind == "linear":
        T, m, n = case["T"], case["n_in"], case["n_out"]
        return {"bytes": _matrix_bytes(n, m, case["fmt"]) + 2 * T * (m + n), "flops": 2 * T * m * n}
    if kind == "quantize":
        n = case["n_in"] * case["n_out"]
        return {"bytes": n * (2 + case["bits"] / 8 + 1 / 32), "flops": 0}
    T, d = case["T"], case["d"]
    b, f = _moe_work(case, min(case["E"], T * case["k"]) if kind == "step" else None)
    if kind == "ffn":
        M = 2 * HC + HC * HC
        b += 4 * M * HC * d + 8 * T * HC * d - 2 * T * d - 4 * T * d  # streams in and out, not x and y
        f += 2 * T * M * HC * d + 2 * T * d * (HC + HC * HC)
    if kind == "step":
        b += _matrix_bytes(d, d, "mxfp8")
        f += 2 * T * d * d
    n = case.get("layers", 1)
    return {"bytes": n * b, "flops": n * f}


def tolerance(case):
    if case["kind"] == "quantize":
        return "exact"
    # bf16 roundings of the intermediates that fall the other way when a sum is taken in another order;
    # a step's later layers carry those of the earlier ones on
    rel = {"linear": 1e-3, "layer": 2e-3, "verify": 2e-3, "ffn": 2e-3, "step": 2e-2}[case["kind"]]
    return {"rel": rel, "differ": 1e-3}


# ---------------------------------------------------------------- the same in 64 bits


def _e2m1(codes):
    table = torch.tensor([0, 0.5, 1, 1.5, 2, 3, 4, 6], dtype=torch.float64, device="cuda")
    table = torch.cat([table, -table])
    low, high = (codes & 15).long(), (codes >> 4).long()
    return torch.stack([table[low], table[high]], -1).reshape(*codes.shape[:-1], -1)


def _scaled(values, scales):
    rows, cols = values.shape
    s = torch.exp2(scales.double() - 127)
    return (values.reshape(rows, cols // 32, 32) * s.reshape(rows, -1, 1)).reshape(rows, cols)


def _mx(w, bits):
    """What a bf16 matrix is after its conversion: nearest power-of-two group scales, elements rounded to
    nearest even and saturated."""
    v = w.double().reshape(w.shape[0], -1, 32)
    top = 448.0 if bits == 8 else 6.0
    amax = v.abs().amax(-1, keepdim=True)
    s = torch.exp2(torch.round(torch.log2(amax.clamp_min(1e-300) / top)).clamp(-127, 127))
    q = (v / s).clamp(-top, top)
    if bits == 8:
        q = q.float().to(torch.float8_e4m3fn).double()
    else:
        a = q.abs()
        step = torch.where(a < 2, 0.5, torch.where(a < 4, 1.0, 2.0)).double()
        q = torch.sign(q) * torch.round(a / step) * step
    return (q * s).reshape(w.shape)


def _resident(w, fmt):
    return w.double() if fmt == "bf16" else _mx(w, 8 if fmt == "mxfp8" else 4)


def _swiglu(g, u):
    g = g.clamp(max=LIMIT)
    return g * torch.sigmoid(g) * u.clamp(-LIMIT, LIMIT)


def _exact_moe(case, p, x):
    x = x.double()
    k = case["k"]
    scores = torch.sigmoid(x @ p["router.weight"].double().T)
    top = torch.topk(scores + p["router.bias"].double(), k, dim=-1).indices.flip(-1)
    weights = scores.gather(-1, top)
    weights = weights / (weights.sum(-1, keepdim=True) + 1e-20) * SCALING
    m = {part: _resident(p[f"shared.{part}"], case["shared"]) for part in ("gate_proj", "up_proj", "down_proj")}
    out = _swiglu(x @ m["gate_proj"].T, x @ m["up_proj"].T) @ m["down_proj"].T
    for e in torch.unique(top).tolist():
        t, j = torch.nonzero(top == e, as_tuple=True)
        m = {part: _scaled(_e2m1(p[f"{part}.weight_packed"][e]), p[f"{part}.weight_scale"][e])
             for part in ("gate_proj", "up_proj", "down_proj")}
        y = _swiglu(x[t] @ m["gate_proj"].T, x[t] @ m["up_proj"].T) @ m["down_proj"].T
        out.index_add_(0, t, y * weights[t, j, None])
    return out, weights, None  # equal choices have no order of their own


def _exact_norm(x, w=None):
    y = x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS)
    return y if w is None else y * w.double()


def _exact_ffn(case, got):
    hc, h = got["hc"], got["hc"]["streams"].double()
    T, d = case["T"], case["d"]
    base, scale = hc["base"].double(), hc["scale"].double()
    mixed = _exact_norm(h.reshape(T, HC * d)) @ hc["fn"].double().T
    pre = torch.sigmoid(mixed[:, :HC] * scale[0] + base[:HC]) + EPS
    post = 2 * torch.sigmoid(mixed[:, HC:2 * HC] * scale[1] + base[HC:2 * HC])
    comb = torch.softmax((mixed[:, 2 * HC:] * scale[2] + base[2 * HC:]).reshape(T, HC, HC), -1) + EPS
    comb = comb / (comb.sum(-2, keepdim=True) + EPS)
    for _ in range(SINKHORN - 1):
        comb = comb / (comb.sum(-1, keepdim=True) + EPS)
        comb = comb / (comb.sum(-2, keepdim=True) + EPS)
    # the MoE layer takes bf16
    normed = _exact_norm((pre[:, :, None] * h).sum(1), hc["norm"]).bfloat16()
    y, weights, _ = _exact_moe(case, got["layers"][0], normed)
    return post[:, :, None] * y[:, None] + comb.transpose(1, 2) @ h, weights, None


def exact(case, seed):
    kind = case["kind"]
    if kind == "quantize":
        return None  # codes and scale bytes are whole numbers
    got = _inputs(case, seed)
    if kind == "linear":
        return got["x"].double() @ _resident(got["w"], case["fmt"]).T
    if kind == "ffn":
        return _exact_ffn(case, got)
    if kind == "layer":
        return _exact_moe(case, got["layers"][0], got["x"][0])
    if kind == "verify":
        return [_exact_moe(case, p, x) for p, x in zip(got["layers"], got["x"])]
    x, outs = got["x"][0], []
    for p, w, norm in zip(got["layers"], got["w"], got["norm"]):
        if outs:
            x = _exact_norm(x, norm).bfloat16()  # the linear takes bf16 and gives bf16
        outs.append(_exact_moe(case, p, (x.double() @ _mx(w, 8).T).bfloat16()))
        x = outs[-1][0]
    return outs
