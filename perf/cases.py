"""The calls whose speed this framework is judged by: what a program that serves a Qwen3-shaped model
with it makes, through the operator's own entry points (``megakernel.load()``), at the sizes of its
configurations, tests and benchmark.

``listed()`` names them, ``draw(rng)`` gives more of the same ranges, ``prepare`` builds what a program
holds before the call (weights, RoPE tables, caches, tokens, all on the GPU), ``run`` makes one call.
``work`` counts the bytes and operations the call cannot do without, ``tolerance`` states how far two
correct implementations may differ, and ``exact`` computes the same outputs in 64-bit floats with plain
torch.

The entry points are whole steps (there is no public single-layer call), so each case is a whole step of
a whole model. Their arithmetic carries activations and sums at fp32 accuracy; the only 16-bit roundings
on the way are those of the new K/V rows.
"""
import math
import os
import random
import sys

import torch

_PACKAGE = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "mega-kernel_amd")
if _PACKAGE not in sys.path:
    sys.path.insert(0, _PACKAGE)

# hidden, intermediate; 28 layers, 16 query and 8 K/V heads of 128, vocabulary 151936, tied embeddings
SHAPES = {"qwen3-0.6b": (1024, 3072), "qwen3-1.7b": (2048, 6144)}
LAYERS, HQ, HKV, D, VOCAB = 28, 16, 8, 128, 151936
EPS, THETA = 1e-6, 1e6


def listed():
    return [
        # One token of a chat in its first few hundred positions, one call per token: the smallest call.
        {"name": "decode", "op": "decode", "shape": "qwen3-0.6b", "position": 160, "max_seq": 512},
        # Several tokens in one call of the device-side loop (scoring given tokens).
        {"name": "decode-steps", "op": "steps", "shape": "qwen3-0.6b", "position": 301, "n": 16, "max_seq": 1024},
        # One token at the end of a long document, its cache in a shared pool of pages.
        {"name": "decode-paged-long", "op": "paged", "shape": "qwen3-0.6b", "position": 3700, "page": 64,
         "max_seq": 4096},
        # One token of the wider model.
        {"name": "decode-1.7b", "op": "decode", "shape": "qwen3-1.7b", "position": 640, "max_seq": 2048},
        # A short question: time to the first token.
        {"name": "prefill-32", "op": "prefill", "shape": "qwen3-0.6b", "n": 32, "position": 0, "max_seq": 512},
        # A paragraph, of a length that fills no tile.
        {"name": "prefill-131", "op": "prefill", "shape": "qwen3-0.6b", "n": 131, "position": 0, "max_seq": 512},
        # A page of text into the wider model.
        {"name": "prefill-512-1.7b", "op": "prefill", "shape": "qwen3-1.7b", "n": 512, "position": 0,
         "max_seq": 2048},
        # A long document at once: the largest call.
        {"name": "prefill-3584", "op": "prefill", "shape": "qwen3-0.6b", "n": 3584, "position": 0, "max_seq": 4096},
        # A later chunk of a long prompt, into pages.
        {"name": "prefill-chunk-paged", "op": "prefill_paged", "shape": "qwen3-0.6b", "n": 300, "position": 1801,
         "page": 16, "max_seq": 4096},
        # A server's step for a few users.
        {"name": "batch-8", "op": "batch", "shape": "qwen3-0.6b", "batch": 8, "ctx_lo": 33, "ctx_hi": 288,
         "max_seq": 512},
        # A busy server's step: the largest batch, conversations of very different lengths.
        {"name": "batch-64", "op": "batch", "shape": "qwen3-0.6b", "batch": 64, "ctx_lo": 64, "ctx_hi": 960,
         "max_seq": 1024},
        # The wider model, an odd number of longer conversations.
        {"name": "batch-13-1.7b", "op": "batch", "shape": "qwen3-1.7b", "batch": 13, "ctx_lo": 100, "ctx_hi": 1900,
         "max_seq": 2048},
    ]


def _spread(rng, lo, hi):
    """A whole number of [lo, hi], even over its logarithm."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    op = rng.choice(["decode", "steps", "paged", "prefill", "prefill", "prefill_paged", "batch", "batch", "batch"])
    shape = rng.choice(["qwen3-0.6b", "qwen3-0.6b", "qwen3-1.7b"])
    wide = shape == "qwen3-1.7b"
    c = {"op": op, "shape": shape}
    if op in ("decode", "steps", "paged"):
        c["max_seq"] = rng.choice([512, 1024, 2048, 4096])
        n = rng.randint(2, 16) if op == "steps" else 1
        c["position"] = _spread(rng, 2, c["max_seq"] - n)
        if op == "steps":
            c["n"] = n
        if op == "paged":
            c["page"] = rng.choice([16, 32, 64, 128])
    elif op == "prefill":
        c["n"] = _spread(rng, 3, 1024 if wide else 3584)
        c["position"] = 0
        c["max_seq"] = max(512, 1 << (c["n"] + 1).bit_length())
    elif op == "prefill_paged":
        c["n"] = _spread(rng, 3, 512)
        c["position"] = rng.randint(1, 3000)
        c["page"] = rng.choice([16, 32, 64, 128])
        c["max_seq"] = 4096
    else:
        c["batch"] = _spread(rng, 2, 64)
        c["max_seq"] = rng.choice([512, 1024, 2048])
        a, b = (_spread(rng, 4, c["max_seq"] - 1) for _ in range(2))
        c["ctx_lo"], c["ctx_hi"] = min(a, b), max(a, b)
    return c


def _contexts(case):
    """Earlier positions of each sequence of a batch: spread evenly from ctx_lo to ctx_hi."""
    B, lo, hi = case["batch"], case["ctx_lo"], case["ctx_hi"]
    return [lo + (hi - lo) * i // max(1, B - 1) for i in range(B)]


def _weights(shape, gen, dev):
    """Random weights of the shape (std 0.02 as Qwen3 initialises, norms about 1, embedding rows of
    different lengths as a trained table's are), flat in the operator's order: 11 tensors a layer."""
    H, I = SHAPES[shape]
    bf = torch.bfloat16

    def mat(n, k):
        return torch.randn(n, k, generator=gen, device=dev, dtype=bf).mul_(0.02)

    def norm(n):
        return (1 + 0.1 * torch.randn(n, generator=gen, device=dev)).to(bf)

    layers = []
    for _ in range(LAYERS):
        layers += [norm(H), mat(HQ * D, H), mat(HKV * D, H), mat(HKV * D, H), norm(D), norm(D), mat(H, HQ * D),
                   norm(H), mat(I, H), mat(I, H), mat(H, I)]
    embed = mat(VOCAB, H).mul_(torch.exp(0.5 * torch.randn(VOCAB, 1, generator=gen, device=dev)).to(bf))
    return layers, embed, norm(H)


def _rope(max_seq, dev):
    inv = 1.0 / THETA ** (torch.arange(0, D, 2, device=dev, dtype=torch.float32) / D)
    ang = torch.arange(max_seq, device=dev, dtype=torch.float32)[:, None] * inv[None, :]
    ang = torch.cat([ang, ang], dim=1)
    return ang.cos().to(torch.bfloat16).contiguous(), ang.sin().to(torch.bfloat16).contiguous()


def _inputs(case, seed):
    """Everything that the call reads, from the seed alone."""
    dev = torch.device("cuda:0")
    gen = torch.Generator(device=dev).manual_seed(int(seed))
    order = random.Random(int(seed))
    s = {"case": case}
    s["layers"], s["embed"], s["norm"] = _weights(case["shape"], gen, dev)
    T = case["max_seq"]
    s["cos"], s["sin"] = _rope(T, dev)
    op = case["op"]
    if op in ("paged", "prefill_paged"):
        pages = (T + case["page"] - 1) // case["page"]
        table = list(range(pages + 8))  # a pool a little larger than this sequence needs, in any order
        order.shuffle(table)
        s["table"] = torch.tensor(table[:pages], dtype=torch.int32, device=dev)
        dims = (LAYERS, pages + 8, HKV, case["page"], D)
    elif op == "batch":
        dims = (case["batch"], LAYERS, HKV, T, D)
    else:
        dims = (LAYERS, HKV, T, D)
    # keys as their norm and rotation leave them (about 1), values as a projection of a normalised row
    s["k"] = torch.randn(dims, generator=gen, device=dev, dtype=torch.bfloat16)
    s["v"] = torch.randn(dims, generator=gen, device=dev, dtype=torch.bfloat16).mul_(0.64)
    tokens = lambda n: [order.randrange(VOCAB) for _ in range(n)]  # noqa: E731
    if op in ("decode", "paged"):
        s["token"] = tokens(1)[0]
    elif op == "steps":
        s["tokens"] = torch.tensor(tokens(case["n"]) + [0], dtype=torch.int32, device=dev)
    elif op in ("prefill", "prefill_paged"):
        s["tokens"] = torch.tensor(tokens(case["n"]), dtype=torch.int32, device=dev)
    else:
        ctx = _contexts(case)
        order.shuffle(ctx)
        s["tokens"] = torch.tensor(tokens(case["batch"]), dtype=torch.int32, device=dev)
        s["positions"] = torch.tensor(ctx, dtype=torch.int32, device=dev)
    return s


def prepare(case, seed):
    import megakernel
    s = _inputs(case, seed)
    s["kernel"] = megakernel.load()
    return s


def run(s):
    """One call: the logits and the caches that it updated. The greedy token that each call also gives is
    the logits' argmax after rounding to bf16; it is made here as in a program, but not handed out to be
    compared, since a tie between two rounded logits turns on their last fp32 bits."""
    c, k = s["case"], s["kernel"]
    op = c["op"]
    model = (s["embed"], s["embed"], s["norm"], s["layers"], s["cos"], s["sin"], s["k"], s["v"])
    if op == "decode":
        logits, _ = k.decode_greedy(s["token"], *model, c["position"], c["max_seq"])
    elif op == "paged":
        logits, _ = k.decode_paged(s["token"], *model, s["table"], c["position"], c["max_seq"])
    elif op == "steps":
        logits = k.decode_steps(s["tokens"], c["n"], False, *model, c["position"], c["max_seq"])
    elif op == "prefill":
        logits, _ = k.prefill(s["tokens"], *model, c["position"], c["max_seq"])
    elif op == "prefill_paged":
        logits, _ = k.prefill_paged(s["tokens"], *model, s["table"], c["position"], c["max_seq"])
    else:
        logits, _ = k.decode_batch(s["tokens"], s["positions"], *model, c["max_seq"])
    return {"logits": logits, "k": s["k"], "v": s["v"]}


def work(case):
    H, I = SHAPES[case["shape"]]
    op = case["op"]
    matrices = LAYERS * (2 * HQ * D * H + 2 * HKV * D * H + 3 * I * H)
    weights = 2 * (matrices + LAYERS * (2 * H + 2 * D) + VOCAB * H + H)
    if op == "batch":
        ctx = [p + 1 for p in _contexts(case)]  # keys that each new token attends to
        read = sum(ctx) - len(ctx)
        rows = case["batch"]
    else:
        n = case.get("n", 1)
        ctx = [case["position"] + i + 1 for i in range(n)]
        read = case["position"]
        rows = n if op == "steps" else 1
    new = len(ctx)
    passes = case["n"] if op == "steps" else 1  # each step of the loop reads the weights and the cache again
    if op == "steps":
        read = sum(ctx) - new
    kv_row = 2 * LAYERS * HKV * D * 2
    logits_rows = rows if op == "batch" else 1
    heads = passes if op == "steps" else logits_rows
    return {"bytes": passes * weights + new * 2 * H + (read + new) * kv_row + 4 * VOCAB * logits_rows,
            "flops": 2.0 * matrices * new + 2.0 * VOCAB * H * heads + 4.0 * LAYERS * HQ * D * sum(ctx)}


def tolerance(case):
    """Sums in another order move a few of the new K/V rows across a bf16 rounding boundary (2^-8 of the
    value), and those differences travel through the layers that follow. Measured against `exact`: decode
    steps up to 6e-4 (a context of a few keys, where the new row weighs most), prefills up to 2e-3."""
    if case["op"].startswith("prefill"):
        return {"rel": 8e-3, "max": 0.15}
    return {"rel": 3e-3, "max": 0.06}


def _rms(x, w):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS) * w


def _rotate(x, cos, sin):
    """Rotate-half RoPE of [..., D] with the tables' rows (their first halves)."""
    a, b = x[..., :D // 2], x[..., D // 2:]
    c, s = cos[..., :D // 2], sin[..., :D // 2]
    return torch.cat([a * c - b * s, b * c + a * s], dim=-1)


def _exact_rows(s, tokens, positions, attend):
    """The last hidden rows (normalised) of `tokens` at `positions`, in 64 bits. attend(layer, q, k, v)
    takes the layer's rotated queries [n, HQ, D] and new K/V rows [n, HKV, D], keeps the rows in its
    cache and returns the attention's output [n, HQ * D]."""
    f = torch.float64
    H, I = SHAPES[s["case"]["shape"]]
    cos, sin = s["cos"][positions].to(f)[:, None], s["sin"][positions].to(f)[:, None]
    x = s["embed"][tokens].to(f)
    for layer in range(LAYERS):
        n1, wq, wk, wv, qn, kn, wo, n2, wg, wu, wd = (t.to(f) for t in s["layers"][11 * layer:11 * layer + 11])
        a = _rms(x, n1)
        q = _rotate(_rms((a @ wq.T).view(-1, HQ, D), qn), cos, sin)
        k = _rotate(_rms((a @ wk.T).view(-1, HKV, D), kn), cos, sin)
        x = x + attend(layer, q, k, (a @ wv.T).view(-1, HKV, D)) @ wo.T
        a = _rms(x, n2)
        x = x + (torch.nn.functional.silu(a @ wg.T) * (a @ wu.T)) @ wd.T
    return _rms(x, s["norm"].to(f))


def _softmax_rows(q, k, v, first):
    """Causal attention of q [n, HQ, D] at positions first .. over k, v [HKV, first + n, D]."""
    n, keys = q.shape[0], k.shape[1]
    out = torch.empty(n, HQ, D, dtype=q.dtype, device=q.device)
    later = torch.arange(keys, device=q.device)[None, :] > first + torch.arange(n, device=q.device)[:, None]
    for h in range(HQ):
        sc = (q[:, h] @ k[h // 2].T.contiguous()) / math.sqrt(D)
        out[:, h] = torch.softmax(sc.masked_fill_(later, -math.inf), dim=-1) @ v[h // 2]
    return out.view(n, HQ * D)


def exact(case, seed):
    s = _inputs(case, seed)
    f, op = torch.float64, case["op"]
    kept = torch.bfloat16  # the cache's type: attention reads the rows as the cache holds them
    table = s["embed"].to(f)
    k_out, v_out = s["k"].to(f), s["v"].to(f)
    if op == "batch":
        pos = s["positions"].tolist()

        def attend(layer, q, k, v):
            out = []
            for b, p in enumerate(pos):
                k_out[b, layer, :, p], v_out[b, layer, :, p] = k[b], v[b]
                kk, vv = s["k"][b, layer, :, :p + 1].to(f), s["v"][b, layer, :, :p + 1].to(f)
                kk[:, p], vv[:, p] = k[b].to(kept).to(f), v[b].to(kept).to(f)
                out.append(_softmax_rows(q[b:b + 1], kk, vv, p))
            return torch.cat(out)

        rows = _exact_rows(s, s["tokens"].long(), s["positions"].long(), attend)
        return {"logits": rows @ table.T, "k": k_out, "v": v_out}

    n, p = case.get("n", 1), case["position"]
    if op in ("paged", "prefill_paged"):
        at = torch.arange(p + n, device=table.device)
        page, off = s["table"].long()[at // case["page"]], at % case["page"]
    else:
        at = torch.arange(p + n, device=table.device)
        page = None

    def attend(layer, q, k, v):
        new = slice(p, p + n)
        if page is None:
            kk, vv = (t[layer, :, :p + n].to(f) for t in (s["k"], s["v"]))
            k_out[layer, :, new], v_out[layer, :, new] = k.transpose(0, 1), v.transpose(0, 1)
        else:
            kk, vv = (t[layer][page, :, off].transpose(0, 1).to(f) for t in (s["k"], s["v"]))
            k_out[layer, page[new], :, off[new]], v_out[layer, page[new], :, off[new]] = k, v
        kk[:, new], vv[:, new] = (t.transpose(0, 1).to(kept).to(f) for t in (k, v))
        return _softmax_rows(q, kk, vv, p)

    tokens = torch.tensor([s["token"]], device=table.device) if "token" in s else s["tokens"][:n].long()
    rows = _exact_rows(s, tokens, at[p:], attend)
    return {"logits": table @ rows[-1], "k": k_out, "v": v_out}
