"""The work that programs built on this package have it do, as cases to time and compare.

A case is a dict of plain values.  ``sets`` lists the wrapped Linears it covers,
``in>out,out;in>out``: each set is one input feeding one or more sibling
Linears.  Rows pick one of ``adapters`` adapters by a Zipf law (``base`` is the
share of rows on the base model) and adapters have ranks of max_rank, a half, a
quarter or an eighth of it.  Rows of more than one position are right-padded.
Routing, lengths and values all come from the seed.

``entry`` is the public entry point a pass goes through:

* ``apply``    sgmv.lora_apply, one Linear (``tiled`` False: lora_apply_rows,
               the kernels of PolyLoraConfig(use_triton_kernels=False))
* ``decode``   sgmv.lora_decode_stacked, one call per set
* ``fused``    sgmv.lora_fused_stacked, one call per set
* ``operator`` sgmv_lora_a_fwd + sgmv_lora_b_fwd on [adapters+1, K, R] tensors
* ``model``    PolyLoraModel.forward of a small decoder, returning its logits

Adapters are resident and the plan of the batch is built before the pass, as a
forward builds it once for all of its Linears; the model case does all of it
inside the pass.  Outputs are the Linears' outputs, updated in place.
"""

from __future__ import annotations

import math
import random

import torch
import torch.nn.functional as F
from torch import nn

from polylora_amd import GpuAdapterCache, PolyLoraConfig, PolyLoraModel, sgmv
from polylora_amd.cache import ModuleSpec
from polylora_amd.store import CpuAdapterStore, CpuLayerWeights

_DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
_QKV, _O, _GATE_UP, _DOWN = "4096>4096,1024,1024", "4096>4096", "4096>14336,14336", "14336>4096"


def _case(name, entry, dtype, rows, row_len, sets, adapters, max_rank, base=0.1, tiled=True):
    return {"name": name, "entry": entry, "dtype": dtype, "rows": rows, "row_len": row_len, "sets": sets,
            "adapters": adapters, "max_rank": max_rank, "base": base, "tiled": tiled}


def listed():
    return [
        # one request being decoded: the attention inputs of one layer, latency alone
        _case("decode_1_row", "decode", "bf16", 1, 1, _QKV, 32, 16, base=0.0),
        # a serving step of 256 requests over 64 adapters: every wrapped Linear of one layer
        _case("decode_256_rows", "decode", "bf16", 256, 1, ";".join((_QKV, _O, _GATE_UP, _DOWN)), 64, 64),
        # a small ragged batch with high-rank adapters, the longest reduction of a layer
        _case("decode_37_rows_r128", "apply", "fp16", 37, 1, _DOWN, 12, 128),
        # flattened tokens of mixed requests over 16 low-rank adapters
        _case("tokens_4096", "apply", "bf16", 4096, 1, _O, 16, 16),
        # the prompt of a single request
        _case("prompt_1500", "apply", "bf16", 1, 1500, "4096>14336", 4, 16, base=0.0),
        # the prompts of a full batch, the widest sibling pair of a layer
        _case("prefill_32x1024", "fused", "bf16", 32, 1024, _GATE_UP, 8, 32, base=0.0),
        # prompts with high-rank adapters
        _case("prefill_8x700_r128", "apply", "bf16", 8, 700, _O, 4, 128, base=0.0),
        # a batch through a small fp32 encoder: its feed-forward input
        _case("encoder_fp32_8x128", "apply", "fp32", 8, 128, "768>3072", 4, 16),
        # a head whose output count is no whole number of 16-byte chunks
        _case("odd_head_16x60", "apply", "bf16", 16, 60, "1024>1003", 6, 16),
        # the plain kernels (use_triton_kernels=False)
        _case("plain_kernels_16x64", "apply", "bf16", 16, 64, "1024>1024", 6, 16, tiled=False),
        # a decode step through the operators themselves, weights in the dense slot layout
        _case("operator_256_rows", "operator", "bf16", 256, 1, _O, 64, 64),
        # a whole forward: residency, plan, every wrapped Linear, logits
        _case("model_8x200", "model", "bf16", 8, 200, "1024>1024,256,256;1024>1024;1024>2816,2816;2816>1024", 6, 16),
    ]


def _spread(rng, lo, hi):
    return max(lo, min(hi, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def draw(rng):
    """One more case: decode steps, mixed tokens, prompts, encoders, odd sizes, the plain kernels, the operators."""
    half = rng.choice(("bf16", "bf16", "fp16"))
    wide = rng.choice((_QKV, _O, _GATE_UP, _DOWN, "2048>2048,512,512", "2048>8192,8192", "8192>2048", "3072>3072"))
    one = rng.choice((_O, "4096>14336", _DOWN, "2048>8192", "1024>1024", "3080>5000"))
    kind = rng.randrange(7)
    if kind == 0:
        c = _case("", "decode", half, _spread(rng, 1, 512), 1, wide, _spread(rng, 1, 64), rng.choice((8, 16, 32, 64)))
    elif kind == 1:
        c = _case("", "apply", half, _spread(rng, 1, 8192), 1, one, _spread(rng, 1, 64), rng.choice((8, 16, 64, 128)))
    elif kind == 2:
        rows = _spread(rng, 1, 16)
        c = _case("", "apply", half, rows, _spread(rng, 16, 1024), one, rng.randint(1, rows), rng.choice((8, 16, 64, 128)))
    elif kind == 3:
        c = _case("", "fused", half, _spread(rng, 4, 24), _spread(rng, 256, 1024), wide, rng.randint(1, 8),
                  rng.choice((8, 16, 32, 64)))
    elif kind == 4:
        c = _case("", "apply", "fp32", _spread(rng, 1, 16), _spread(rng, 8, 512),
                  rng.choice(("768>768", "768>3072", "3072>768")), rng.randint(1, 8), rng.choice((4, 8, 16, 32)))
    elif kind == 5:
        # odd sizes, or the plain kernels at any size
        odd = rng.random() < 0.5
        sizes = (rng.randint(100, 2000), rng.randint(50, 2000)) if odd else (rng.choice((768, 1024, 2048)), 1024)
        c = _case("", "apply", rng.choice(("bf16", "fp32")), _spread(rng, 1, 64), rng.choice((1, 17, 60)),
                  "%d>%d" % sizes, rng.randint(1, 8), rng.choice((4, 8, 16, 32)), tiled=odd)
    else:
        c = _case("", "operator", half, _spread(rng, 4, 64), rng.choice((1, 4, 33)), one, _spread(rng, 1, 64),
                  rng.choice((8, 16, 64)))
    c["base"] = round(rng.choice((0.0, 0.1, 0.3)), 2)
    del c["name"]
    return c


# ----------------------------------------------------------------------------- inputs


def _sets(case):
    """[(in, [out, ...], [module name, ...])] of a case."""
    out, n = [], 0
    for part in case["sets"].split(";"):
        fin, fouts = part.split(">")
        fouts = [int(v) for v in fouts.split(",")]
        out.append((int(fin), fouts, ["m%d" % (n + i) for i in range(len(fouts))]))
        n += len(fouts)
    return out


def _route(case, seed):
    """(rank of each adapter, adapter of each row or None, length of each row)."""
    rng = random.Random("%d:%d:%d" % (seed, case["rows"], case["adapters"]))
    top, n = case["max_rank"], case["adapters"]
    ranks = [top] + [max(1, top >> rng.randrange(4)) for _ in range(n - 1)]
    law = [1.0 / (i + 1) ** 1.1 for i in range(n)]
    rows = [None if rng.random() < case["base"] else rng.choices(range(n), law)[0] for _ in range(case["rows"])]
    if all(a is None for a in rows):
        rows[0] = 0
    m = case["row_len"]
    lens = [m if case["rows"] == 1 else rng.randint((m + 1) // 2, m) for _ in range(case["rows"])]
    return ranks, rows, lens


def _gen(seed, salt):
    return torch.Generator(device="cuda").manual_seed((seed * 1009 + salt) % (1 << 62))


def _weights(case, seed, ranks):
    """{module: [(A [rank, in], B [out, rank]) of each adapter]} in the case's dtype, N(0, 0.02)."""
    dt, g = _DTYPES[case["dtype"]], _gen(seed, 1)
    shapes = {n: (fin, fout) for fin, fouts, names in _sets(case) for n, fout in zip(names, fouts)}
    return {n: [((torch.randn(r, fin, generator=g, device="cuda") * 0.02).to(dt),
                 (torch.randn(fout, r, generator=g, device="cuda") * 0.02).to(dt)) for r in ranks]
            for n, (fin, fout) in shapes.items()}


def _activations(case, seed):
    """[(x [tokens, in], [y [tokens, out], ...])] of each set, N(0, 1)."""
    dt, g, t = _DTYPES[case["dtype"]], _gen(seed, 2), case["rows"] * case["row_len"]
    return [(torch.randn(t, fin, generator=g, device="cuda", dtype=dt),
             [torch.randn(t, fout, generator=g, device="cuda", dtype=dt) for fout in fouts])
            for fin, fouts, _ in _sets(case)]


def _store(weights, ranks):
    store = CpuAdapterStore()
    host = {n: [(a.t().contiguous().cpu(), b.t().contiguous().cpu()) for a, b in w] for n, w in weights.items()}
    for i, r in enumerate(ranks):
        store.add_adapter("a%d" % i, {n: CpuLayerWeights(A=w[i][0], B=w[i][1], rank=r, scale=2.0)
                                      for n, w in host.items()})
    return store


def prepare(case, seed):
    if case["entry"] == "model":
        return _prepare_model(case, seed)
    ranks, rows, lens = _route(case, seed)
    weights, acts = _weights(case, seed, ranks), _activations(case, seed)
    seq = torch.tensor(lens, dtype=torch.int32, device="cuda")
    s = {"entry": case["entry"], "tiled": case["tiled"], "acts": acts, "seq": seq, "row_len": case["row_len"],
         "names": [names for _, _, names in _sets(case)]}
    if case["entry"] == "operator":
        (fin, (fout,), (name,)), n, top = _sets(case)[0], case["adapters"] + 1, case["max_rank"]
        s["a"] = torch.zeros(n, fin, top, dtype=acts[0][0].dtype, device="cuda")
        s["b"] = torch.zeros(n, top, fout, dtype=acts[0][0].dtype, device="cuda")
        for i, (a, b) in enumerate(weights[name]):
            s["a"][i + 1, :, : ranks[i]] = a.t()
            s["b"][i + 1, : ranks[i]] = b.t()
        s["slots"] = torch.tensor([0 if r is None else r + 1 for r in rows], dtype=torch.int32, device="cuda")
        s["ranks"] = torch.tensor([0] + ranks, dtype=torch.int32, device="cuda")
        s["scales"] = torch.tensor([0.0] + [2.0] * len(ranks), device="cuda")
        s["x"] = acts[0][0].view(case["rows"], case["row_len"], fin)
        s["y"] = acts[0][1][0].view(case["rows"], case["row_len"], fout)
        return s
    specs = [ModuleSpec(n, fin, fout) for fin, fouts, names in _sets(case) for n, fout in zip(names, fouts)]
    config = PolyLoraConfig(max_gpu_adapters=case["adapters"], max_rank=case["max_rank"],
                            use_triton_kernels=case["tiled"])
    s["cache"] = GpuAdapterCache(_store(weights, ranks), specs, config, torch.device("cuda", 0), acts[0][0].dtype)
    s["slots"] = s["cache"].ensure_resident(["__base__" if r is None else "a%d" % r for r in rows])
    if case["tiled"]:
        s["plan"] = sgmv.SgmvPlan(s["slots"], seq, case["row_len"], s["cache"].num_slots,
                                  distinct_slots=len({r for r in rows if r is not None}))
    return s


def run(s):
    entry = s["entry"]
    if entry == "model":
        with torch.no_grad():
            return s["model"](input_ids=s["ids"], attention_mask=s["mask"], adapter_ids=s["adapter_ids"])
    if entry == "operator":
        t = sgmv.sgmv_lora_a_fwd(s["x"], s["a"], s["seq"], s["slots"], s["ranks"])
        return sgmv.sgmv_lora_b_fwd(t, s["b"], s["seq"], s["slots"], s["ranks"], s["scales"], s["y"])
    for (x, ys), names in zip(s["acts"], s["names"]):
        if entry == "decode":
            sgmv.lora_decode_stacked(x, ys, s["cache"], names, s["plan"])
        elif entry == "fused":
            sgmv.lora_fused_stacked(x, ys, s["cache"], names, s["plan"])
        elif s["tiled"]:
            sgmv.lora_apply(x, ys[0], s["cache"], names[0], s["plan"])
        else:
            sgmv.lora_apply_rows(x, ys[0], s["cache"], names[0], s["slots"], s["seq"], s["row_len"])
    return [ys for _, ys in s["acts"]]


# ----------------------------------------------------------------------------- the small decoder

_VOCAB, _HEAD, _LAYERS = 1000, 64, 2
_LINEARS = ("q_proj", "k_proj", "v_proj", "o_proj", "gate_proj", "up_proj", "down_proj")


def _norm(x, w):
    return F.rms_norm(x, (x.shape[-1],), w, 1e-5)


class _Block(nn.Module):
    def __init__(self, shapes):
        super().__init__()
        self.norm1 = nn.Parameter(torch.ones(shapes[0][0]))
        self.norm2 = nn.Parameter(torch.ones(shapes[0][0]))
        for name, (fin, fout) in zip(_LINEARS, shapes):
            setattr(self, name, nn.Linear(fin, fout, bias=False))

    def forward(self, h, attend):
        x = _norm(h, self.norm1)
        q, k, v = (p(x).unflatten(-1, (-1, _HEAD)).transpose(1, 2) for p in (self.q_proj, self.k_proj, self.v_proj))
        h = h + self.o_proj(attend(q, k, v).transpose(1, 2).flatten(2))
        x = _norm(h, self.norm2)
        return h + self.down_proj(F.silu(self.gate_proj(x)) * self.up_proj(x))


def _attend_fused(q, k, v):
    k, v = (t.repeat_interleave(q.shape[1] // t.shape[1], 1) for t in (k, v))
    with nn.attention.sdpa_kernel(nn.attention.SDPBackend.FLASH_ATTENTION):
        return F.scaled_dot_product_attention(q, k, v, is_causal=True)


def _attend_exact(q, k, v):
    k, v = (t.repeat_interleave(q.shape[1] // t.shape[1], 1).contiguous() for t in (k, v))
    s = q.contiguous() @ k.transpose(2, 3).contiguous() / math.sqrt(_HEAD)
    blocked = torch.ones(s.shape[-2:], dtype=torch.bool, device=s.device).triu(1)
    return s.masked_fill(blocked, float("-inf")).softmax(-1) @ v


class _Decoder(nn.Module):
    def __init__(self, shapes, attend=_attend_fused):
        super().__init__()
        self.embed = nn.Embedding(_VOCAB, shapes[0][0])
        self.blocks = nn.ModuleList(_Block(shapes) for _ in range(_LAYERS))
        self.norm = nn.Parameter(torch.ones(shapes[0][0]))
        self.head = nn.Linear(shapes[0][0], _VOCAB, bias=False)
        self.attend = attend

    def forward(self, input_ids, attention_mask=None):
        h = self.embed(input_ids)
        for block in self.blocks:
            h = block(h, self.attend)
        return self.head(_norm(h, self.norm))


def _model_parts(case, seed):
    """(decoder, {module: adapter weights}, ids, mask) of a model case."""
    ranks, rows, lens = _route(case, seed)
    shapes = [(fin, fout) for fin, fouts, _ in _sets(case) for fout in fouts]
    dt, g = _DTYPES[case["dtype"]], _gen(seed, 3)
    with torch.device("cuda"):
        model = _Decoder(shapes).to(dt).eval().requires_grad_(False)
    for p in model.parameters():
        if p.dim() > 1:
            p.copy_(torch.randn(p.shape, generator=g, device="cuda") * (1.0 if p.shape[0] == _VOCAB else 0.03))
    weights = {}
    for i in range(_LAYERS):
        w = _weights(case, seed * 16 + i, ranks)
        weights.update(("blocks.%d.%s" % (i, name), w["m%d" % j]) for j, name in enumerate(_LINEARS))
    model.head.weight.mul_(1 / math.sqrt(shapes[0][0]))
    ids = torch.randint(0, _VOCAB, (case["rows"], case["row_len"]), generator=g, device="cuda")
    mask = (torch.arange(case["row_len"], device="cuda") < torch.tensor(lens, device="cuda")[:, None]).long()
    return model, weights, ids, mask


def _prepare_model(case, seed):
    ranks, rows, _ = _route(case, seed)
    model, weights, ids, mask = _model_parts(case, seed)
    config = PolyLoraConfig(target_modules=list(_LINEARS), max_gpu_adapters=case["adapters"],
                            max_rank=case["max_rank"])
    pm = PolyLoraModel(model, config, adapter_store=_store(weights, ranks)).eval()
    return {"entry": "model", "model": pm, "ids": ids, "mask": mask,
            "adapter_ids": ["__base__" if r is None else "a%d" % r for r in rows]}


# ----------------------------------------------------------------------------- what a pass needs, and its answer


def work(case):
    """Active x rows read once per set, active y rows read and written, each used adapter's A and B read once."""
    ranks, rows, lens = _route(case, 0)
    es = 4 if case["dtype"] == "fp32" else 2
    active = [(a, n) for a, n in zip(rows, lens) if a is not None]
    t, used = sum(n for _, n in active), {a for a, _ in active}
    nbytes = flops = 0
    for fin, fouts, _ in _sets(case):
        nbytes += es * t * fin
        for fout in fouts:
            nbytes += es * (2 * t * fout + sum(ranks[a] for a in used) * (fin + fout))
            flops += 2 * sum(n * ranks[a] for a, n in active) * (fin + fout)
            if case["entry"] == "model":  # the base products too
                nbytes += es * fin * fout
                flops += 2 * case["rows"] * case["row_len"] * fin * fout
    if case["entry"] == "model":
        hidden, tokens = _sets(case)[0][0], case["rows"] * case["row_len"]
        return {"bytes": _LAYERS * nbytes + es * _VOCAB * (hidden + tokens), "flops": _LAYERS * flops + 2 * tokens * hidden * _VOCAB}
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    if case["entry"] == "model":
        return {"rel": 0.028}  # four times a bf16 forward's distance from its exact value
    # about four times the distance from the exact result (1.8e-3, 2.9e-4 and 3.5e-8): the output rounds once to the
    # element type, the intermediate once before it (fp32: sums of other orders as well)
    return {"rel": {"bf16": 8e-3, "fp16": 1.2e-3, "fp32": 1e-6}[case["dtype"]]}


def exact(case, seed):
    ranks, rows, lens = _route(case, seed)
    m = case["row_len"]
    if case["entry"] == "model":
        model, weights, ids, _ = _model_parts(case, seed)
        model = model.double()
        model.attend = _attend_exact

        def add(name):
            def hook(_, args, out):
                return _add_lora(args[0], out.clone(), weights[name], rows, lens)
            return hook

        for name in weights:
            model.get_submodule(name).register_forward_hook(add(name))
        with torch.no_grad():
            return model(ids)
    weights, out = _weights(case, seed, ranks), []
    for (x, ys), (_, _, names) in zip(_activations(case, seed), _sets(case)):
        x = x.view(case["rows"], m, -1)
        out.append([_add_lora(x, y.double().view(case["rows"], m, -1), weights[n], rows, lens).view(y.shape)
                    for y, n in zip(ys, names)])
    if case["entry"] == "operator":
        return out[0][0].view(case["rows"], m, -1)
    return out


def _add_lora(x, y, weights, rows, lens):
    for b, (a, n) in enumerate(zip(rows, lens)):
        if a is not None:
            wa, wb = (w.double() for w in weights[a])
            y[b, :n] += 2.0 * (x[b, :n].double() @ wa.t().contiguous()) @ wb.t().contiguous()
    return y
