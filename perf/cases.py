"""The calls whose speed this package is judged by: what an AlphaFold 3 inference run has it do, from the smallest
crop to the largest, through the public entry points.

A case is a dict of plain values.  `op` names the entry point:

    attention   dot_product_attention_cpp on [B, H, L, D], float32 or bfloat16 arithmetic
    fp8         dot_product_attention_fp8 on bfloat16 tensors
    grid        GridSelfAttentionCpp.forward on a pair tensor [L, L, 128]: LayerNorm, pair bias, attention, gate, output projection
    self        self_attention_cpp on tokens [L, C] (or [B, L, C]: B diffusion samples of the same tokens)
    glu         gated_linear_unit_cpp on [L, L, C], the transition block of the pair tensor

The shapes are those of af3_kernels_amd/synthetic.py and of the tests; masks: "tail" drops the last tenth of the keys
(padding to a bucket), "random" drops 8 % of them at random, per batch row.
"""
import math

import torch

import af3_kernels_amd as af3

BF16 = torch.bfloat16


def _attention(name, B, H, L, D, dtype="bf16", mask="random"):
    return {"name": name, "op": "attention", "B": B, "H": H, "L": L, "D": D, "dtype": dtype, "mask": mask}


def listed():
    return [
        # triangle attention of a short peptide: launches and host time are all there is to it
        _attention("triangle_n37", 37, 4, 37, 32),
        # triangle attention of the starting node at a middling crop, padded to its bucket
        _attention("triangle_n384", 384, 4, 384, 32, mask="tail"),
        # the same at the largest training crop
        _attention("triangle_n768", 768, 4, 768, 32),
        # the same for a large complex of an odd number of tokens: the longest call of an inference run
        _attention("triangle_n1491", 1491, 4, 1491, 32),
        # a slab of triangle attention in float32, for callers that run the pair stack in full precision
        _attention("triangle_fp32_n768", 64, 4, 768, 32, dtype="fp32"),
        # single attention with pair bias of the pairformer (one sequence, 16 heads of 24)
        _attention("single_n768", 1, 16, 768, 24, mask="tail"),
        # the same for an odd number of tokens: bias rows start at any address
        _attention("single_n1491", 1, 16, 1491, 24),
        # token attention of the diffusion transformer (16 heads of 48) for a short sequence, called once a layer and step
        _attention("single_n128_d48", 1, 16, 128, 48),
        # five diffusion samples that share one pair bias, both products in e4m3
        {"name": "samples_fp8_n1536", "op": "fp8", "B": 5, "H": 16, "L": 1536, "D": 24, "mask": "tail"},
        # the whole grid self-attention block on the pair tensor of a middling crop
        {"name": "grid_n384", "op": "grid", "L": 384, "mask": "random"},
        # self-attention of the diffusion transformer with its projections and gate, one sample or several
        {"name": "self_n1536", "op": "self", "B": 1, "H": 16, "L": 1536, "C": 768, "mask": "random"},
        # the gated linear unit of the pair transition at the largest training crop
        {"name": "glu_n768", "op": "glu", "L": 768, "C": 128},
    ]


def _log(rng, low, high):
    """A whole number between low and high, spread over its logarithm; odd ones among them, and multiples of 8 (buckets) as often as not."""
    n = int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))
    if rng.random() < 0.4:
        n = (n + 7) // 8 * 8
    return max(low, min(high, n))


def draw(rng):
    mask = rng.choice(["random", "tail"])
    op = rng.choice(["triangle", "triangle", "triangle_fp32", "single", "single", "fp8", "grid", "self", "glu"])
    if op == "triangle":
        n = _log(rng, 32, 1491)
        case = _attention("", n, 4, n, 32, mask=mask)
    elif op == "triangle_fp32":
        case = _attention("", _log(rng, 2, 64), 4, _log(rng, 64, 768), 32, dtype="fp32", mask=mask)
    elif op == "single":
        case = _attention("", 1, 16, _log(rng, 32, 2048), rng.choice([24, 48]), mask=mask)
    elif op == "fp8":
        case = {"op": "fp8", "B": rng.randint(1, 8), "H": 16, "L": _log(rng, 128, 1536), "D": 24, "mask": mask}
    elif op == "grid":
        case = {"op": "grid", "L": _log(rng, 32, 1024), "mask": mask}
    elif op == "self":
        case = {"op": "self", "B": rng.choice([1, 1, 5]), "H": 16, "L": _log(rng, 64, 2048), "C": rng.choice([384, 768]), "mask": mask}
    else:
        case = {"op": "glu", "L": _log(rng, 32, 1024), "C": rng.choice([64, 128])}
    case.pop("name", None)
    return case


def _mask(kind, shape, gen):
    L = shape[-1]
    if kind == "tail":
        m = torch.ones(shape, dtype=torch.bool, device="cuda")
        m[..., L - L // 10:] = False
        return m
    m = torch.rand(shape, generator=gen, device="cuda") < 0.92
    m[..., 0] = True
    return m


def prepare(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)

    def normal(*shape, dtype=BF16, scale=1.0):
        t = torch.randn(shape, generator=gen, device="cuda", dtype=dtype)
        return t.mul_(scale) if scale != 1.0 else t

    op, L = case["op"], case["L"]
    if op in ("attention", "fp8"):
        B, H, D = case["B"], case["H"], case["D"]
        dtype = torch.float32 if case.get("dtype") == "fp32" else BF16
        q, k, v = (normal(B, H, L, D, dtype=dtype) for _ in range(3))
        bias = normal(H, L, L, dtype=dtype)
        # single sequences and samples of one sequence share one mask row; the rows of a pair tensor have one each
        mask = _mask(case["mask"], (L,) if op == "fp8" or B == 1 else (B, L), gen)
        fn = af3.dot_product_attention_fp8 if op == "fp8" else af3.dot_product_attention_cpp
        return fn, (q, k, v, mask, bias)
    if op == "grid":
        module = af3.GridSelfAttentionCpp(128, 4).to(device="cuda", dtype=BF16).eval().requires_grad_(False)
        for name, p in module.named_parameters():
            if p.dim() == 2:
                p.copy_(normal(*p.shape, scale=128 ** -0.5))
            else:
                p.copy_(normal(*p.shape, scale=0.1) + (1.0 if name.endswith("weight") else 0.0))
        return module, (normal(L, L, 128), _mask(case["mask"], (L, L), gen))
    C = case["C"]
    if op == "self":
        B, H = case["B"], case["H"]
        x = normal(L, C) if B == 1 else normal(B, L, C)
        wq, wk, wv, wg = (af3.vnni_repack_tensor(normal(C, C, scale=C ** -0.5), 2, C // H) for _ in range(4))
        return af3.self_attention_cpp, (x, _mask(case["mask"], (L,), gen), normal(H, L, L), wq, normal(C), wk, wv, wg, H)
    return af3.gated_linear_unit_cpp, (normal(L, L, C), normal(C, 8 * C, scale=C ** -0.5))


def run(state):
    fn, args = state
    return fn(*args)


def work(case):
    op, L = case["op"], case["L"]
    if op in ("attention", "fp8"):
        B, H, D = case["B"], case["H"], case["D"]
        size = 4 if case.get("dtype") == "fp32" else 2
        return {"bytes": size * (4 * B * H * L * D + H * L * L) + (L if op == "fp8" or B == 1 else B * L), "flops": 4 * B * H * L * L * D}
    if op == "grid":
        C = 128
        # pair in and out, mask, weights; bias projection, five C x C projections, both attention products
        return {"bytes": 2 * (2 * L * L * C + 5 * C * C + 6 * C) + L * L, "flops": L * L * C * (2 * 4 + 10 * C + 4 * L)}
    C = case["C"]
    if op == "self":
        B, H = case["B"], case["H"]
        return {"bytes": 2 * (2 * B * L * C + H * L * L + 4 * C * C + C) + L, "flops": B * L * C * (8 * C + 4 * L)}
    return {"bytes": 2 * (L * L * C + L * L * 4 * C + 8 * C * C), "flops": 2 * L * L * C * 8 * C}


def tolerance(case):
    if case.get("dtype") == "fp32":
        return {"rel": 1e-5}
    # e4m3 weights and values carry 4 significant bits, bf16 ones 8
    return {"rel": 2e-2 if case["op"] == "fp8" else 1e-2}
