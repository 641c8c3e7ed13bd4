"""The work whose time counts: single ops, blocks and one trunk of the Pairformer and MSA stacks.

Every case is one forward call through the public factories (or ``foldforge_amd.load``) on
resident tensors, as an inference program makes it: seeded fp32 master parameters, bf16
activations drawn from N(0, 1) (the ops normalise their input, so this is the distribution they
see), a key mask with ``real`` tokens out of ``n``. ``exact`` restates the same calls in plain
torch at 64 bits.
"""

from __future__ import annotations

import math

import torch
import torch.nn.functional as F

import foldforge_amd
from foldforge_amd import dispatch, factories
from foldforge_amd.adapter import place
from foldforge_amd.trunk import randomise

DEVICE = "cuda"

#: Template-stack blocks (pair 64): triangle attention form, head width, trimul hidden width,
#: transition factor. One per lineage that the block shapes of ``bench.py`` name.
TEMPLATE_STACKS = {
    "af3": dict(triangle_model="af3", d_head=16, d_tri=64, factor=2),
    "protenix": dict(triangle_model="protenix", d_head=32, d_tri=128, factor=2),
    "boltz2": dict(triangle_model="boltz2", d_head=32, d_tri=64, factor=4),
    "rf3": dict(triangle_model="rf3", d_head=64, d_tri=64, factor=4),
}


def listed() -> list[dict]:
    return [
        # one triangle attention at the smallest published op shape: launches and latency
        dict(name="triangle_attention_n128", kind="triangle_attention", model="af3", starting=True,
             n=128, real=128, batch=1),
        # an ordinary protein whose length is no multiple of anything, some tokens padded
        dict(name="triangle_multiplication_n300", kind="triangle_multiplication", outgoing=True,
             length_divided=False, n=300, real=263, batch=1),
        # the single track's attention of a small chain
        dict(name="single_attention_n201", kind="single_attention", n=201, real=201, batch=1),
        # the MSA track's transition: many short rows
        dict(name="transition_msa", kind="transition", width=64, factor=4, rows=512 * 256),
        # a standalone norm of MSA rows
        dict(name="layer_norm_msa", kind="layer_norm", width=64, rows=512 * 384, dtype="bf16"),
        # a peptide through a few trunk blocks with the single track: a whole call, launch-bound
        dict(name="trunk_n97", kind="trunk", blocks=3, n=97, real=97),
        # the headline: one pair-stack block, N = 512, ragged
        dict(name="pair_block_n512", kind="pair_block", model="af3", n=512, real=386, batch=1),
        # a large complex, the OpenFold lineage's form, no padding
        dict(name="pair_block_n1024", kind="pair_block", model="openfold3_preview2", n=1024, real=1024,
             batch=1),
        # four templates through a template-stack block
        dict(name="template_block_n384", kind="template_block", stack="af3", n=384, real=384, batch=4),
        # Chai-1's 256-wide trunk block
        dict(name="chai1_block_n384", kind="chai1_block", n=384, real=384, batch=1),
        # the MSA stack's two MSA-pair ops at the reference's op-table shapes
        dict(name="outer_product_mean_n384", kind="outer_product_mean", n=384, depth=512, fill=0.9),
        dict(name="msa_averaging_n256", kind="msa_averaging", n=256, depth=512, heads=8, d_head=8,
             real=256),
    ]


def _spread(rng, lo: int, hi: int) -> int:
    """A whole number of [lo, hi], spread over its logarithm."""
    return min(hi, max(lo, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def _real(rng, n: int) -> int:
    """Real tokens of a row of n: all of them, or a ragged share as in the benchmark (0.6 to 1)."""
    return n if rng.random() < 0.4 else max(1, round(n * rng.uniform(0.6, 1.0)))


def draw(rng) -> dict:
    kind = rng.choice(["triangle_attention", "triangle_multiplication", "single_attention", "transition",
                       "layer_norm", "trunk", "pair_block", "template_block", "chai1_block",
                       "outer_product_mean", "msa_averaging"])
    if kind == "triangle_attention":
        n = _spread(rng, 48, 768)
        return dict(kind=kind, model=rng.choice(["af3", "openfold3_preview2", "rf3"]),
                    starting=rng.random() < 0.5, n=n, real=_real(rng, n), batch=rng.choice([1, 1, 2]))
    if kind == "triangle_multiplication":
        n = _spread(rng, 48, 768)
        return dict(kind=kind, outgoing=rng.random() < 0.5, length_divided=rng.random() < 0.25, n=n,
                    real=_real(rng, n), batch=rng.choice([1, 1, 2]))
    if kind == "single_attention":
        n = _spread(rng, 48, 768)
        return dict(kind=kind, n=n, real=_real(rng, n), batch=rng.choice([1, 1, 5]))
    if kind == "transition":
        width, factor = rng.choice([(64, 2), (64, 4), (128, 4), (384, 4)])
        return dict(kind=kind, width=width, factor=factor,
                    rows=_spread(rng, 100, 2000) if width == 384 else _spread(rng, 2500, 260000))
    if kind == "layer_norm":
        width = rng.choice([64, 128, 256, 384, 768])
        return dict(kind=kind, width=width, rows=_spread(rng, 200, 25_000_000 // width),
                    dtype=rng.choice(["bf16", "bf16", "f32"]))
    if kind == "trunk":
        n = _spread(rng, 48, 320)
        return dict(kind=kind, blocks=rng.choice([2, 3]), n=n, real=_real(rng, n))
    if kind == "pair_block":
        n = _spread(rng, 64, 768)
        return dict(kind=kind, model=rng.choice(["af3", "openfold3_preview2"]), n=n, real=_real(rng, n),
                    batch=1)
    if kind == "template_block":
        n = _spread(rng, 64, 448)
        return dict(kind=kind, stack=rng.choice(sorted(TEMPLATE_STACKS)), n=n, real=_real(rng, n),
                    batch=rng.choice([1, 2, 4]))
    if kind == "chai1_block":
        n = _spread(rng, 64, 448)
        return dict(kind=kind, n=n, real=_real(rng, n), batch=1)
    if kind == "outer_product_mean":
        return dict(kind=kind, n=_spread(rng, 48, 448), depth=_spread(rng, 32, 1024),
                    fill=rng.choice([1.0, 0.9, 0.6]))
    n = _spread(rng, 48, 448)
    return dict(kind=kind, n=n, depth=_spread(rng, 32, 1024), heads=8, d_head=rng.choice([8, 32]),
                real=_real(rng, n))


# ------------------------------------------------------------------------------------ calls
def _module(case: dict, seed: int):
    """The case's module on the device with every op on the native kernels."""
    kind = case["kind"]
    if kind == "trunk":
        return foldforge_amd.load(blocks=case["blocks"], seed=seed, unsupported="error")
    if kind == "triangle_attention":
        module = factories.triangle_attention(128, 4, starting=case["starting"], model=case["model"])
    elif kind == "triangle_multiplication":
        module = factories.triangle_multiplication(128, outgoing=case["outgoing"],
                                                   divide_by_length=case["length_divided"])
    elif kind == "single_attention":
        module = factories.pairformer_block(d_pair=128, triangle_model="af3", d_single=384).single_attention
    elif kind == "transition":
        module = factories.transition(case["width"], case["factor"])
    elif kind == "layer_norm":
        module = factories.layer_norm(case["width"])
    elif kind == "pair_block":
        module = factories.pairformer_block(d_pair=128, triangle_model=case["model"])
    elif kind == "template_block":
        stack = TEMPLATE_STACKS[case["stack"]]
        module = factories.pairformer_block(
            d_pair=64, triangle_model=stack["triangle_model"], d_hidden_tri_attention=stack["d_head"],
            d_hidden_tri_multi=stack["d_tri"], pair_transition_n=stack["factor"])
    elif kind == "chai1_block":
        module = factories.pairformer_block(d_pair=256, triangle_model="chai1", d_hidden_tri_attention=64,
                                            pair_transition_n=2)
    elif kind == "outer_product_mean":
        module = factories.outer_product_mean(64, 128, 32, normalize_before_proj=False, count_offset=1e-3)
    else:
        module = factories.msa_pair_weighted_averaging(64, 128, case["heads"], case["d_head"])
    # blocks carry the bounded init of a deep stack; a single op the plain one (a larger update)
    module = place(randomise(module, seed, out_scale=0.25 if kind.endswith("_block") else None))
    dispatch.install(module, dispatch.Plan.of("hip", None, "error"), torch.device(DEVICE))
    return module


def _inputs(case: dict, seed: int) -> tuple:
    gen = torch.Generator(device=DEVICE).manual_seed(seed + 1)

    def normal(*shape: int, dtype=torch.bfloat16):
        return torch.randn(*shape, generator=gen, device=DEVICE).to(dtype)

    kind = case["kind"]
    if kind in ("transition", "layer_norm"):
        dtype = torch.float32 if case.get("dtype") == "f32" else torch.bfloat16
        return (normal(case["rows"], case["width"], dtype=dtype),)
    n, batch = case["n"], case.get("batch", 1)
    if kind == "outer_product_mean":
        keep = torch.rand(1, case["depth"], n, generator=gen, device=DEVICE) < case["fill"]
        return normal(1, case["depth"], n, 64), keep, normal(1, n, n, 128)
    mask = (torch.arange(n, device=DEVICE) < case["real"]).expand(batch, n).contiguous()
    pair = normal(batch, n, n, {"template_block": 64, "chai1_block": 256}.get(kind, 128))
    if kind == "single_attention":
        return normal(batch, n, 384), pair, mask
    if kind == "trunk":
        return pair, mask, normal(batch, n, 384)
    if kind == "msa_averaging":
        return normal(1, case["depth"], n, 64), pair, mask
    return pair, mask


def prepare(case: dict, seed: int) -> dict:
    return dict(module=_module(case, seed), args=_inputs(case, seed))


def run(state: dict):
    with torch.no_grad():
        return state["module"](*state["args"])


# ------------------------------------------------------------------------------------ the least work
def _attention_flops(tokens: float, queries: float, keys: float, width: int) -> float:
    return 4.0 * tokens * queries * keys * width


def _block_parts(n: int, c: int, hidden: int, width: int, factor: int, batch: int) -> tuple[float, float]:
    """FLOP of a pair block's five ops and its parameter bytes."""
    pairs = float(batch) * n * n
    trimul = pairs * (2 * 4 * hidden * c + 2 * n * hidden + 2 * hidden * c + 2 * c * c)
    att = pairs * (2 * 4 * width * c + 2 * 4 * c + 2 * width * c) + _attention_flops(batch * n, n, n, width)
    trans = pairs * 6 * factor * c * c
    params = 2 * (5 * hidden * c + c * c) + 2 * (5 * width * c + 4 * c) + 3 * factor * c * c
    return 2 * trimul + 2 * att + trans, 4.0 * params


def work(case: dict) -> dict:
    kind = case["kind"]
    if kind == "layer_norm":
        size = (4 if case["dtype"] == "f32" else 2) * case["rows"] * case["width"]
        return {"bytes": 2.0 * size, "flops": 8.0 * case["rows"] * case["width"]}
    if kind == "transition":
        d, f, rows = case["width"], case["factor"], case["rows"]
        return {"bytes": 4.0 * rows * d + 12.0 * f * d * d, "flops": 6.0 * rows * f * d * d}
    n, batch = case["n"], case.get("batch", 1)
    real = case.get("real", n)
    pairs = float(batch) * n * n
    pair_bytes = 2.0 * pairs * {"template_block": 64, "chai1_block": 256}.get(kind, 128)
    if kind == "triangle_attention":
        flops = pairs * (2 * 128 * 4 * 128 + 2 * 128 * 4 + 2 * 128 * 128) + _attention_flops(batch * n, n, real, 128)
        return {"bytes": 2 * pair_bytes + 4 * 5 * 128 * 128, "flops": flops}
    if kind == "triangle_multiplication":
        flops = pairs * (2 * 128 * 6 * 128) + 2.0 * pairs * real * 128
        return {"bytes": 2 * pair_bytes + 4 * 6 * 128 * 128, "flops": flops}
    single = 2.0 * batch * n * 384
    if kind == "single_attention":
        flops = 2.0 * batch * n * 5 * 384 * 384 + 2.0 * pairs * 128 * 16 + _attention_flops(batch, n, real, 384)
        return {"bytes": pair_bytes + 2 * single + 4 * 5 * 384 * 384, "flops": flops}
    if kind == "outer_product_mean":
        depth = case["depth"]
        flops = 2.0 * depth * n * 64 * 64 + 2.0 * depth * n * n * 1024 + 2.0 * n * n * 1024 * 128
        return {"bytes": 2.0 * depth * n * 64 + depth * n + 2 * pair_bytes + 4 * 1024 * 128, "flops": flops}
    if kind == "msa_averaging":
        depth, width = case["depth"], case["heads"] * case["d_head"]
        rows = float(depth) * n
        flops = 2 * rows * 64 * 3 * width + 2 * rows * real * width + 2 * pairs * 128 * case["heads"]
        return {"bytes": 4.0 * rows * 64 + pair_bytes + 4 * 3 * 64 * width, "flops": flops}
    if kind == "template_block":
        stack = TEMPLATE_STACKS[case["stack"]]
        flops, params = _block_parts(n, 64, stack["d_tri"], 4 * stack["d_head"], stack["factor"], batch)
    elif kind == "chai1_block":
        flops, params = _block_parts(n, 256, 256, 256, 2, batch)
    else:
        flops, params = _block_parts(n, 128, 128, 128, 4, batch)
    if kind == "trunk":
        track = 2.0 * n * (5 + 12) * 384 * 384 + 2.0 * pairs * 128 * 16 + _attention_flops(1, n, real, 384)
        return {"bytes": 2 * pair_bytes + 2 * single + case["blocks"] * (params + 4 * 17 * 384 * 384),
                "flops": case["blocks"] * (flops + track)}
    return {"bytes": 2 * pair_bytes + params, "flops": flops}


#: Four times the relative difference from ``exact`` that the calls were seen to have (the bf16
#: rounding of a residual output is 1.7e-3 of it; a block adds its intermediates').
TOLERANCE = {"trunk": 3e-2, "pair_block": 1.6e-2, "template_block": 1.6e-2, "chai1_block": 1.9e-2,
             "single_attention": 1.2e-2, "msa_averaging": 1.2e-2, "triangle_multiplication": 1.1e-2}


def tolerance(case: dict):
    if case.get("dtype") == "f32":
        return {"rel": 1e-5}
    return {"rel": TOLERANCE.get(case["kind"], 8e-3)}


# ------------------------------------------------------------------------------------ 64 bits
def _norm(x, p: dict, name: str, eps: float = 1e-5):
    return F.layer_norm(x, x.shape[-1:], p[name + ".weight"], p.get(name + ".bias"), eps)


def _lin(x, p: dict, name: str):
    return F.linear(x, p[name + ".weight"], p.get(name + ".bias"))


def _sub(p: dict, prefix: str) -> dict:
    return {k[len(prefix) + 1:]: v for k, v in p.items() if k.startswith(prefix + ".")}


def _exact_trimul(p: dict, z, mask, outgoing: bool, length_divided: bool = False):
    h = _norm(z, p, "ln_pair")
    keep = (mask[:, :, None] & mask[:, None, :])[..., None].to(z.dtype)
    a = (_lin(h, p, "to_left") * keep * torch.sigmoid(_lin(h, p, "to_left_gate"))).permute(0, 3, 1, 2)
    b = (_lin(h, p, "to_right") * keep * torch.sigmoid(_lin(h, p, "to_right_gate"))).permute(0, 3, 1, 2)
    a, b = (a, b.transpose(-1, -2)) if outgoing else (a.transpose(-1, -2), b)
    t = torch.matmul(a.contiguous(), b.contiguous()).permute(0, 2, 3, 1)
    if length_divided:
        t = t / mask.any(dim=0).sum().clamp_min(1)
    return z + _lin(_norm(t, p, "ln_out"), p, "to_out") * torch.sigmoid(_lin(h, p, "to_gate"))


def _exact_attend(q, k, v, bias, mask):
    """softmax(q k^T / sqrt(d) + bias) v over the real keys; q, k, v [rows, heads, n, d]."""
    logits = torch.matmul(q * q.shape[-1] ** -0.5, k.transpose(-1, -2).contiguous()) + bias
    return torch.matmul(logits.masked_fill(~mask, float("-inf")).softmax(dim=-1), v)


def _exact_triattn(p: dict, z, mask, heads: int, starting: bool, transposed_bias: bool, turned: bool = True):
    batch, n = z.shape[:2]
    h = _norm(z, p, "ln_pair")
    bias = _lin(h, p, "to_bias").permute(0, 3, 1, 2)
    if not starting:
        h = h.transpose(1, 2)
        bias = bias.transpose(-1, -2) if transposed_bias else bias
    o = torch.empty(*h.shape[:3], p["to_query.weight"].shape[0], dtype=z.dtype, device=z.device)
    rows = max(1, (1 << 28) // (n * n * heads))
    for b in range(batch):
        for r in range(0, n, rows):
            x = h[b, r:r + rows]
            q, k, v = (_lin(x, p, name).unflatten(-1, (heads, -1)).transpose(1, 2).contiguous()
                       for name in ("to_query", "to_key", "to_value"))
            o[b, r:r + rows] = _exact_attend(q, k, v, bias[b], mask[b]).transpose(1, 2).flatten(-2)
    y = _lin(torch.sigmoid(_lin(h, p, "to_gate")) * o, p, "to_out")
    return z + (y if starting or not turned else y.transpose(1, 2))


def _exact_transition(p: dict, x):
    h = _norm(x, p, "ln_in")
    return x + _lin(F.silu(_lin(h, p, "expand_a")) * _lin(h, p, "expand_b"), p, "squeeze")


def _exact_single(p: dict, s, z, mask, heads: int = 16):
    x = _norm(s, p, "ln_single")
    q, k, v = (_lin(x, p, name).unflatten(-1, (heads, -1)).transpose(1, 2).contiguous()
               for name in ("to_query", "to_key", "to_value"))
    bias = _lin(_norm(z, p, "ln_pair"), p, "to_bias").permute(0, 3, 1, 2)
    o = _exact_attend(q, k, v, bias, mask[:, None, None, :]).transpose(1, 2).flatten(-2)
    return s + _lin(torch.sigmoid(_lin(x, p, "to_gate")) * o, p, "to_out")


def _exact_block(p: dict, z, mask, heads: int = 4, transposed_bias: bool = False, turned: bool = True):
    z = _exact_trimul(_sub(p, "tri_multi_outgoing"), z, mask, True)
    z = _exact_trimul(_sub(p, "tri_multi_incoming"), z, mask, False)
    z = _exact_triattn(_sub(p, "tri_atten_starting"), z, mask, heads, True, transposed_bias)
    z = _exact_triattn(_sub(p, "tri_atten_ending"), z, mask, heads, False, transposed_bias, turned)
    return _exact_transition(_sub(p, "transition_pair"), z)


def exact(case: dict, seed: int):
    state = prepare(case, seed)
    p = {k: v.double() for k, v in state["module"].state_dict().items()}
    args = [t.double() if t.is_floating_point() else t for t in state["args"]]
    kind = case["kind"]
    with torch.no_grad():
        if kind == "layer_norm":
            return F.layer_norm(args[0], args[0].shape[-1:], p["weight"], p["bias"], 1e-5)
        if kind == "transition":
            return _exact_transition(p, args[0])
        if kind == "triangle_multiplication":
            return _exact_trimul(p, *args, case["outgoing"], case["length_divided"])
        if kind == "triangle_attention":
            return _exact_triattn(p, *args, 4, case["starting"], case["model"] == "openfold3_preview2")
        if kind == "single_attention":
            return _exact_single(p, *args)
        if kind == "pair_block":
            return _exact_block(p, *args, transposed_bias=case["model"] == "openfold3_preview2")
        if kind == "template_block":
            return _exact_block(p, *args, transposed_bias=case["stack"] in ("protenix", "boltz2"))
        if kind == "chai1_block":
            return _exact_block(p, *args, turned=False)
        if kind == "trunk":
            z, mask, s = args
            for i in range(case["blocks"]):
                block = _sub(p, f"blocks.{i}")
                z = _exact_block(block, z, mask)
                s = _exact_single(_sub(block, "single_attention"), s, z, mask)
                s = _exact_transition(_sub(block, "single_transition"), s)
            return z, s
        if kind == "outer_product_mean":
            m, keep, residual = args
            x, keep = _norm(m, p, "ln_msa"), keep.double()
            left, right = _lin(x, p, "to_left") * keep[..., None], _lin(x, p, "to_right") * keep[..., None]
            n, count = case["n"], torch.matmul(keep.transpose(1, 2).contiguous(), keep)
            o = torch.matmul(left[0].flatten(1).t().contiguous(), right[0].flatten(1))  # [(i c), (j e)]
            o = o.unflatten(0, (n, 32)).unflatten(2, (n, 32)).permute(0, 2, 1, 3).flatten(2)
            return residual + _lin(o[None], p, "to_out") / (count[..., None] + 1e-3)
        m, z, mask = args
        heads, x = case["heads"], _norm(m, p, "ln_msa")
        logits = _lin(_norm(z, p, "ln_pair"), p, "to_bias").permute(0, 3, 1, 2)
        w = logits.masked_fill(~mask[:, None, None, :], float("-inf")).softmax(dim=-1)[0]  # [heads, i, j]
        v = _lin(x, p, "to_value")[0].unflatten(-1, (heads, -1)).permute(2, 1, 0, 3)  # [heads, j, depth, d]
        o = torch.matmul(w, v.flatten(2).contiguous()).unflatten(2, v.shape[2:]).permute(2, 1, 0, 3).flatten(2)
        return m + _lin(torch.sigmoid(_lin(x, p, "to_gate")) * o[None], p, "to_out")
