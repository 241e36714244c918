"""The calls that a Boltz-2 program makes of this package, as measurable cases: Pairformer blocks and their triangle
modules, the diffusion token transformer's step, the MSA block and the 64-channel template stack, in the two precisions
of BOLTZ_MLX_PRECISION ("fp32", the default, and "f16", the production mode).

listed() are the fixed cases, draw(rng) gives more of the same ranges, prepare() makes what a program holds before the
call, run() is one pass through the public modules, work() what the pass cannot do without, tolerance() how far another
correct implementation at the same precision may be off, and exact() the same pass in 64 bits in plain torch.
"""

from __future__ import annotations

import math

import torch

from boltz_mlx_amd import kernels as K
from boltz_mlx_amd.layers.msa import MSALayer
from boltz_mlx_amd.layers.pairformer import PairformerLayer, PairformerModule, PairformerNoSeqModule
from boltz_mlx_amd.layers.transformersv2 import DiffusionStepGraph, DiffusionTransformer
from boltz_mlx_amd.layers.triangular_attention.attention import (
    TriangleAttentionEndingNode,
    TriangleAttentionStartingNode,
)
from boltz_mlx_amd.layers.triangular_mult import TriangleMultiplicationIncoming, TriangleMultiplicationOutgoing

# The model's widths: single 384 (16 heads), pair 128 (4 heads of 32), MSA 64, template pair 64, diffusion tokens 768
# (16 heads, 24 layers).
CS, CZ, CM, CT, HEADS = 384, 128, 64, 64, 4
DIFF_DIM, DIFF_HEADS, DIFF_DEPTH = 768, 16, 24


def listed() -> list:
    return [
        # a short peptide through one block in the default precision: launches and host time
        {"name": "layer_fp32_n29", "op": "layer", "mode": "fp32", "n": 29, "blocks": 1},
        # one block on a small protein, the fp32 parity configuration
        {"name": "layer_fp32_n128", "op": "layer", "mode": "fp32", "n": 128, "blocks": 1},
        # a middle-sized complex (an odd token count) in the default precision, as the overflow guard recomputes it
        {"name": "trunk_fp32_n513", "op": "trunk", "mode": "fp32", "n": 513, "blocks": 1},
        # an ordinary protein in production precision: four blocks of the trunk, an odd token count
        {"name": "trunk_f16_n203", "op": "trunk", "mode": "f16", "n": 203, "blocks": 4},
        # the largest complex of the benchmark: two blocks of the trunk
        {"name": "trunk_f16_n1000", "op": "trunk", "mode": "f16", "n": 1000, "blocks": 2},
        # triangle attention as a module, each node and precision
        {"name": "tri_att_fp32_n400", "op": "tri_att", "mode": "fp32", "n": 400, "first": False},
        {"name": "tri_att_f16_n400", "op": "tri_att", "mode": "f16", "n": 400, "first": True},
        # triangle multiplication as a module, each direction and precision
        {"name": "tri_mul_fp32_n333", "op": "tri_mul", "mode": "fp32", "n": 333, "first": False},
        {"name": "tri_mul_f16_n800", "op": "tri_mul", "mode": "f16", "n": 800, "first": True},
        # one sampler step of the diffusion token transformer over five samples
        {"name": "diffusion_f16_n400", "op": "diffusion", "mode": "f16", "n": 400, "samples": 5},
        # one MSA block over a deep alignment
        {"name": "msa_f16_n400_s1024", "op": "msa", "mode": "f16", "n": 400, "rows": 1024},
        # the template embedder's 64-channel pair stack
        {"name": "template_f16_n400", "op": "template", "mode": "f16", "n": 400, "blocks": 2},
    ]


def _size(rng, lo: int, hi: int) -> int:
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng) -> dict:
    op = rng.choice(["layer", "trunk", "trunk", "tri_att", "tri_mul", "diffusion", "msa", "template"])
    mode = rng.choice(["fp32", "f16"])
    if op == "layer":
        return {"op": op, "mode": mode, "n": _size(rng, 16, 256), "blocks": 1}
    if op == "trunk":
        if mode == "fp32":
            return {"op": op, "mode": mode, "n": _size(rng, 128, 513), "blocks": 1}
        return {"op": op, "mode": mode, "n": _size(rng, 128, 1000), "blocks": rng.randint(1, 2)}
    if op in ("tri_att", "tri_mul"):
        return {"op": op, "mode": mode, "n": _size(rng, 48, 640 if mode == "fp32" else 1000),
                "first": rng.random() < 0.5}
    if op == "diffusion":
        return {"op": op, "mode": "f16", "n": _size(rng, 48, 400), "samples": rng.randint(1, 5)}
    if op == "msa":
        return {"op": op, "mode": mode, "n": _size(rng, 64, 400), "rows": _size(rng, 16, 1024)}
    return {"op": op, "mode": mode, "n": _size(rng, 48, 400), "blocks": rng.randint(1, 2)}


# ------------------------------------------------------------------------------------------------ parameters

def _under(prefix: str, d: dict) -> dict:
    return {f"{prefix}.{k}": v for k, v in d.items()}


def _tri_mul_shapes(d: int) -> dict:
    return {"norm_in.weight": (d,), "norm_in.bias": (d,), "p_in.weight": (2 * d, d), "g_in.weight": (2 * d, d),
            "norm_out.weight": (d,), "norm_out.bias": (d,), "p_out.weight": (d, d), "g_out.weight": (d, d)}


def _tri_att_shapes(d: int) -> dict:
    hc = 32 * HEADS
    return {"layer_norm.weight": (d,), "layer_norm.bias": (d,), "linear.weight": (HEADS, d),
            "mha.linear_q.weight": (hc, d), "mha.linear_k.weight": (hc, d), "mha.linear_v.weight": (hc, d),
            "mha.linear_o.weight": (d, hc), "mha.linear_g.weight": (hc, d)}


def _transition_shapes(d: int) -> dict:
    return {"norm.weight": (d,), "norm.bias": (d,), "fc1.weight": (4 * d, d), "fc2.weight": (4 * d, d),
            "fc3.weight": (d, 4 * d)}


def _pair_shapes(d: int) -> dict:
    return {**_under("tri_mul_out", _tri_mul_shapes(d)), **_under("tri_mul_in", _tri_mul_shapes(d)),
            **_under("tri_att_start", _tri_att_shapes(d)), **_under("tri_att_end", _tri_att_shapes(d)),
            **_under("transition_z", _transition_shapes(d))}


def _attention_shapes(d: int) -> dict:
    return {"proj_q.weight": (d, d), "proj_q.bias": (d,), "proj_k.weight": (d, d), "proj_v.weight": (d, d),
            "proj_g.weight": (d, d), "proj_o.weight": (d, d)}


def _layer_shapes() -> dict:
    return {"pre_norm_s.weight": (CS,), "pre_norm_s.bias": (CS,), **_under("attention", _attention_shapes(CS)),
            "attention.proj_z.0.weight": (CZ,), "attention.proj_z.0.bias": (CZ,),
            "attention.proj_z.1.weight": (16, CZ), **_pair_shapes(CZ),
            **_under("transition_s", _transition_shapes(CS))}


def _diffusion_shapes() -> dict:
    d = DIFF_DIM
    ada = {"s_norm.weight": (d,), "s_scale.weight": (d, d), "s_scale.bias": (d,), "s_bias.weight": (d, d)}
    return {**_under("adaln", ada), **_under("pair_bias_attn", _attention_shapes(d)),
            "output_projection_linear.weight": (d, d), "output_projection_linear.bias": (d,),
            **_under("transition.adaln", ada), "transition.swish_gate.0.weight": (4 * d, d),
            "transition.a_to_b.weight": (2 * d, d), "transition.b_to_a.weight": (d, 2 * d),
            "transition.output_projection.0.weight": (d, d), "transition.output_projection.0.bias": (d,)}


def _msa_shapes() -> dict:
    pwa = {"norm_m.weight": (CM,), "norm_m.bias": (CM,), "norm_z.weight": (CZ,), "norm_z.bias": (CZ,),
           "proj_m.weight": (256, CM), "proj_g.weight": (256, CM), "proj_z.weight": (8, CZ), "proj_o.weight": (CM, 256)}
    opm = {"norm.weight": (CM,), "norm.bias": (CM,), "proj_a.weight": (32, CM), "proj_b.weight": (32, CM),
           "proj_o.weight": (CZ, 1024), "proj_o.bias": (CZ,)}
    return {**_under("msa_transition", _transition_shapes(CM)), **_under("pair_weighted_averaging", pwa),
            **_under("outer_product_mean", opm), **_under("pairformer_layer", _pair_shapes(CZ))}


def _shapes(case: dict) -> dict:
    op = case["op"]
    if op == "layer":
        return _layer_shapes()
    if op == "trunk":
        return {k: v for i in range(case["blocks"]) for k, v in _under(f"layers.{i}", _layer_shapes()).items()}
    if op == "template":
        return {k: v for i in range(case["blocks"]) for k, v in _under(f"layers.{i}", _pair_shapes(CT)).items()}
    if op == "diffusion":
        return {k: v for i in range(DIFF_DEPTH) for k, v in _under(f"layers.{i}", _diffusion_shapes()).items()}
    return {"tri_att": _tri_att_shapes, "tri_mul": _tri_mul_shapes}[op](CZ) if op != "msa" else _msa_shapes()


def _params(case: dict, gen: torch.Generator) -> dict:
    """Seeded weights of trained size: matrices N(0, 1 / fan_in) (those that write a residual stream half that wide),
    LayerNorm weights 1 + N(0, 0.1), biases N(0, 0.1)."""
    out = {}
    for name, shape in _shapes(case).items():
        t = torch.randn(shape, generator=gen, device="cuda")
        if len(shape) == 2:
            t *= shape[1] ** -0.5
            if name.endswith(("p_out.weight", "linear_o.weight", "fc3.weight", "proj_o.weight", "b_to_a.weight")):
                t *= 0.5
        else:
            t *= 0.1
            if name.endswith("weight"):
                t += 1.0
        out[name] = t
    return out


def _inputs(case: dict, seed: int) -> tuple[dict, dict]:
    """(parameters, activations and masks), on the GPU, from the seed alone. The last twentieth of the tokens is
    padding (pair_mask = token_i token_j) and a tenth of an alignment's entries are gaps."""
    gen = torch.Generator(device="cuda").manual_seed(seed)
    p = _params(case, gen)
    n, op = case["n"], case["op"]

    def randn(*shape):
        return torch.randn(shape, generator=gen, device="cuda")

    tok = torch.ones((1, n), device="cuda")
    tok[:, n - n // 20:] = 0.0
    x = {"mask": tok, "pair_mask": tok[:, :, None] * tok[:, None, :]}
    if op in ("layer", "trunk"):
        x.update(s=randn(1, n, CS), z=randn(1, n, n, CZ))
    elif op in ("tri_att", "tri_mul"):
        x.update(z=randn(1, n, n, CZ))
    elif op == "template":
        x.update(z=randn(1, n, n, CT))
    elif op == "msa":
        gaps = (torch.rand((1, case["rows"], n), generator=gen, device="cuda") > 0.1).float()
        x.update(z=randn(1, n, n, CZ), m=randn(1, case["rows"], n, CM), msa_mask=gaps * tok[:, None])
    else:
        b = case["samples"]
        x.update(a=randn(b, n, DIFF_DIM), s=randn(1, n, DIFF_DIM), mask=tok.expand(b, n).contiguous(),
                 bias=randn(1, n, n, DIFF_DEPTH * DIFF_HEADS))
    return p, x


# ------------------------------------------------------------------------------------------------ one pass

def _module(case: dict) -> torch.nn.Module:
    op = case["op"]
    with torch.device("cuda"):
        if op == "layer":
            return PairformerLayer(CS, CZ)
        if op == "trunk":
            return PairformerModule(CS, CZ, case["blocks"])
        if op == "template":
            return PairformerNoSeqModule(CT, case["blocks"])
        if op == "msa":
            return MSALayer(CM, CZ)
        if op == "tri_att":
            return (TriangleAttentionStartingNode if case["first"] else TriangleAttentionEndingNode)(CZ, 32, HEADS)
        if op == "tri_mul":
            return (TriangleMultiplicationOutgoing if case["first"] else TriangleMultiplicationIncoming)(CZ)
        return DiffusionTransformer(DIFF_DEPTH, DIFF_HEADS, DIFF_DIM, DIFF_DIM)


def prepare(case: dict, seed: int) -> dict:
    """The module with its weights, the inputs and, for the diffusion step, what the sampler keeps over its steps: the
    conditioning, the layers' pair biases and the captured step."""
    p, x = _inputs(case, seed)
    if case["op"] == "diffusion":  # one Linear under two names
        p.update({k.replace("output_projection_linear.", "output_projection.0."): v for k, v in p.items()
                  if ".output_projection_linear." in k})
    K.set_precision(case["mode"])
    with torch.no_grad():
        module = _module(case).eval()
        module.load_state_dict(p)
        state = {"op": case["op"], "mode": case["mode"], "module": module, "x": x}
        if case["op"] == "diffusion":
            cond, prepared = module.precompute_cond(x["s"]), module.prepare(x.pop("bias"))
            state["step"] = DiffusionStepGraph(module, x["a"], cond, prepared, x["mask"], multiplicity=case["samples"])
    return state


def run(state: dict):
    op, module, x = state["op"], state["module"], state["x"]
    K.set_precision(state["mode"])
    with torch.no_grad():
        if op == "diffusion":
            return state["step"](x["a"])
        if op in ("layer", "trunk"):
            return module(x["s"], x["z"], x["mask"], x["pair_mask"])
        if op == "msa":
            return module(x["z"], x["m"], x["pair_mask"], x["msa_mask"])
        return module(x["z"], x["pair_mask"])


# ------------------------------------------------------------------------------------------------ work and tolerance

def _tri_mul_flops(n: int, d: int) -> float:
    return 2.0 * d * n ** 3 + 2.0 * (4 * d * d + 2 * d * d) * n ** 2


def _tri_att_flops(n: int, d: int) -> float:
    hc = 32 * HEADS
    return 4.0 * hc * n ** 3 + 2.0 * (d * (4 * hc + HEADS) + hc * d) * n ** 2


def _pair_flops(n: int, d: int) -> float:
    return 2 * _tri_mul_flops(n, d) + 2 * _tri_att_flops(n, d) + 24.0 * d * d * n ** 2


def _single_flops(n: int) -> float:
    return 2.0 * 16 * CZ * n ** 2 + 4.0 * CS * n ** 2 + (10.0 + 24.0) * CS * CS * n


def work(case: dict) -> dict:
    """Operations of the definition; bytes of the inputs, weights and outputs, each once."""
    n, op = case["n"], case["op"]
    weights = 4.0 * sum(math.prod(s) for s in _shapes(case).values())
    if op in ("layer", "trunk"):
        return {"bytes": 8.0 * n * (n * CZ + CS) + 4.0 * n * n + weights,
                "flops": case["blocks"] * (_pair_flops(n, CZ) + _single_flops(n))}
    if op == "template":
        return {"bytes": 8.0 * n * n * CT + 4.0 * n * n + weights, "flops": case["blocks"] * _pair_flops(n, CT)}
    if op in ("tri_att", "tri_mul"):
        return {"bytes": 8.0 * n * n * CZ + 4.0 * n * n + weights,
                "flops": (_tri_att_flops if op == "tri_att" else _tri_mul_flops)(n, CZ)}
    if op == "msa":
        s = case["rows"]
        flops = (2.0 * s * n * CM * (512 + 256 + 64) + 2.0 * 8 * CZ * n * n + 2.0 * 256 * s * n * n
                 + 24.0 * CM * CM * s * n + 2.0 * 1024 * s * n * n + 2.0 * 1024 * CZ * n * n)
        return {"bytes": 8.0 * (n * n * CZ + s * n * CM) + 4.0 * n * (n + s) + weights, "flops": flops + _pair_flops(n, CZ)}
    b, d = case["samples"], DIFF_DIM
    stepped = DIFF_DEPTH * (5 + 6 + 2) * d * d  # the weights a step reads, in the storage type
    return {"bytes": 8.0 * b * n * d + 2.0 * stepped + 2.0 * DIFF_DEPTH * DIFF_HEADS * n * n,
            "flops": b * n * (2.0 * stepped + DIFF_DEPTH * 4.0 * n * d)}


# About four times the relative error against 64 bits that these paths measure: fp32 sums (up to 6.6e-7; two orders of
# the same sums differ by more), and fp16 operands and intermediates with fp32 sums (single modules 7e-4; in whole blocks
# the update's error stands beside the residual stream, and the roundings of one layer travel through the next).
TOLERANCE = {("tri_att", "f16"): 3e-3, ("tri_mul", "f16"): 3e-3, ("layer", "f16"): 1.5e-3, ("trunk", "f16"): 2.5e-3,
             ("msa", "f16"): 1.5e-3, ("template", "f16"): 2e-3, ("diffusion", "f16"): 3e-3}


def tolerance(case: dict) -> dict:
    return {"rel": 5e-6 if case["mode"] == "fp32" else TOLERANCE[case["op"], "f16"]}


# ------------------------------------------------------------------------------------------------ 64 bits

def _sub(p: dict, prefix: str) -> dict:
    return {k[len(prefix) + 1:]: v for k, v in p.items() if k.startswith(prefix + ".")}


def _ln(x, w=None, b=None):
    return torch.nn.functional.layer_norm(x, x.shape[-1:], w, b, 1e-5)


def _masked(logits, bias):
    """logits + bias; where the bias masks, summed in 32 bits as the model defines it: a row whose keys are all masked
    has logits that differ only by what 32 bits keep beside the mask's size."""
    return torch.where(bias == 0, logits, (logits.float() + bias.float()).double())


def _tri_mul(x, mask, p, first):
    d = x.shape[-1]
    xn = _ln(x, p["norm_in.weight"], p["norm_in.bias"])
    ab = (xn @ p["p_in.weight"].T) * torch.sigmoid(xn @ p["g_in.weight"].T) * mask[..., None]
    a, b = ab[..., :d].permute(2, 0, 1).contiguous(), ab[..., d:].permute(2, 0, 1).contiguous()
    o = a @ b.transpose(1, 2).contiguous() if first else a.transpose(1, 2).contiguous() @ b
    o = _ln(o.permute(1, 2, 0), p["norm_out.weight"], p["norm_out.bias"])
    return (o @ p["p_out.weight"].T) * torch.sigmoid(xn @ p["g_out.weight"].T)


def _tri_att(x, mask, p, first):
    if not first:
        return _tri_att(x.transpose(0, 1), mask.T, p, True).transpose(0, 1)
    n, c = x.shape[0], 32
    xn = _ln(x, p["layer_norm.weight"], p["layer_norm.bias"])
    bias = (xn @ p["linear.weight"].T).permute(2, 0, 1)
    out = []
    for i in range(0, n, 16):
        r = xn[i:i + 16]
        q, k, v = ((r @ p[f"mha.linear_{t}.weight"].T).view(-1, n, HEADS, c).transpose(1, 2) for t in "qkv")
        logits = (q / c ** 0.5) @ k.transpose(2, 3).contiguous() + bias
        a = torch.softmax(_masked(logits, (1e9 * (mask[i:i + 16] - 1))[:, None, None, :]), -1) @ v.contiguous()
        out.append(a.transpose(1, 2).reshape(-1, n, HEADS * c) * torch.sigmoid(r @ p["mha.linear_g.weight"].T))
    return torch.cat(out) @ p["mha.linear_o.weight"].T


def _transition(x, p):
    out = []
    for r in x.reshape(-1, x.shape[-1]).split(1 << 17):
        xn = _ln(r, p["norm.weight"], p["norm.bias"])
        h = torch.nn.functional.silu(xn @ p["fc1.weight"].T) * (xn @ p["fc2.weight"].T)
        out.append(h @ p["fc3.weight"].T)
    return torch.cat(out).view(x.shape)


def _pair(z, mask, p):
    z = z + _tri_mul(z, mask, _sub(p, "tri_mul_out"), True)
    z = z + _tri_mul(z, mask, _sub(p, "tri_mul_in"), False)
    z = z + _tri_att(z, mask, _sub(p, "tri_att_start"), True)
    z = z + _tri_att(z, mask, _sub(p, "tri_att_end"), False)
    return z + _transition(z, _sub(p, "transition_z"))


def _attention(s, bias, mask, p, heads):
    """s [B, N, c], bias [heads, N, N], mask [B, N]."""
    b, n, c = s.shape
    q, k, v, g = (s @ p[f"proj_{t}.weight"].T + (p["proj_q.bias"] if t == "q" else 0.0) for t in "qkvg")
    q, k, v = (t.view(b, n, heads, -1).transpose(1, 2) for t in (q, k, v))
    logits = q @ k.transpose(2, 3).contiguous() / (c // heads) ** 0.5 + bias
    o = torch.softmax(_masked(logits, ((1 - mask) * -1e6)[:, None, None, :]), -1) @ v.contiguous()
    return (torch.sigmoid(g) * o.transpose(1, 2).reshape(b, n, c)) @ p["proj_o.weight"].T


def _block(s, z, mask, pair_mask, p):
    z = _pair(z, pair_mask, p)
    zb = _ln(z, p["attention.proj_z.0.weight"], p["attention.proj_z.0.bias"]) @ p["attention.proj_z.1.weight"].T
    sn = _ln(s, p["pre_norm_s.weight"], p["pre_norm_s.bias"])
    s = s + _attention(sn, zb.permute(2, 0, 1), mask, _sub(p, "attention"), 16)
    return s + _transition(s, _sub(p, "transition_s")), z


def _msa(z, m, pair_mask, msa_mask, p):
    q = _sub(p, "pair_weighted_averaging")
    rows, n, _ = m.shape
    mn = _ln(m, q["norm_m.weight"], q["norm_m.bias"])
    logits = (_ln(z, q["norm_z.weight"], q["norm_z.bias"]) @ q["proj_z.weight"].T).permute(2, 0, 1)
    w = torch.softmax(_masked(logits, ((1 - pair_mask) * -1e6)[None]), -1)
    v = (mn @ q["proj_m.weight"].T).view(rows, n, 8, 32).permute(2, 1, 0, 3).reshape(8, n, rows * 32)
    o = (w @ v).view(8, n, rows, 32).permute(2, 1, 0, 3).reshape(rows, n, 256)
    m = m + (torch.sigmoid(mn @ q["proj_g.weight"].T) * o) @ q["proj_o.weight"].T
    m = m + _transition(m, _sub(p, "msa_transition"))
    q = _sub(p, "outer_product_mean")
    mn = _ln(m, q["norm.weight"], q["norm.bias"])
    a, b = ((mn @ q[f"proj_{t}.weight"].T * msa_mask[..., None]).reshape(rows, n * 32) for t in "ab")
    num = (msa_mask.T @ msa_mask).clamp(min=1)
    bt = b.contiguous()
    out = []
    for i in range(0, n, 32):
        k = min(32, n - i)
        o = (a[:, 32 * i:32 * (i + k)].T.contiguous() @ bt).view(k, 32, n, 32).transpose(1, 2).reshape(k, n, 1024)
        out.append((o / num[i:i + k, :, None]) @ q["proj_o.weight"].T + q["proj_o.bias"])
    return _pair(z + torch.cat(out), pair_mask, _sub(p, "pairformer_layer")), m


def _adaln(a, s, p):
    sn = _ln(s, p["s_norm.weight"])
    return torch.sigmoid(sn @ p["s_scale.weight"].T + p["s_scale.bias"]) * _ln(a) + sn @ p["s_bias.weight"].T


def _diffusion(a, s, bias, mask, p):
    gate = "output_projection_linear"
    b = _attention(_adaln(a, s, _sub(p, "adaln")), bias, mask, _sub(p, "pair_bias_attn"), DIFF_HEADS)
    a = a + torch.sigmoid(s @ p[f"{gate}.weight"].T + p[f"{gate}.bias"]) * b
    q, gate = _sub(p, "transition"), "output_projection.0"
    t = _adaln(a, s, _sub(q, "adaln"))
    x, g = (t @ q["swish_gate.0.weight"].T).chunk(2, -1)
    u = torch.nn.functional.silu(g) * x * (t @ q["a_to_b.weight"].T)
    return a + torch.sigmoid(s @ q[f"{gate}.weight"].T + q[f"{gate}.bias"]) * (u @ q["b_to_a.weight"].T)


def exact(case: dict, seed: int):
    p, x = _inputs(case, seed)
    x = {k: v.double() for k, v in x.items() if k != "bias"} | ({"bias": x["bias"]} if "bias" in x else {})
    p = {k: v.double() for k, v in p.items()}
    op, pair_mask = case["op"], x["pair_mask"][0]
    with torch.no_grad():
        if op == "diffusion":
            a = x["a"]
            for i in range(DIFF_DEPTH):
                bias = x["bias"][0, :, :, DIFF_HEADS * i:DIFF_HEADS * (i + 1)].permute(2, 0, 1).double()
                a = _diffusion(a, x["s"], bias, x["mask"], _sub(p, f"layers.{i}"))
            return a
        z = x["z"][0]
        if op == "layer":
            s, z = _block(x["s"], z, x["mask"], pair_mask, p)
            return s, z[None]
        if op == "trunk":
            s = x["s"]
            for i in range(case["blocks"]):
                s, z = _block(s, z, x["mask"], pair_mask, _sub(p, f"layers.{i}"))
            return s, z[None]
        if op == "template":
            for i in range(case["blocks"]):
                z = _pair(z, pair_mask, _sub(p, f"layers.{i}"))
            return z[None]
        if op == "msa":
            z, m = _msa(z, x["m"][0], pair_mask, x["msa_mask"][0], p)
            return z[None], m[None]
        return (_tri_att if op == "tri_att" else _tri_mul)(z, pair_mask, p, case["first"])[None]
