"""The work that programs have this library do, as measurable cases.

A case is a dict of plain values; "path" says which public entry point it
takes:

* ``lse``: the torch.logsumexp drop-in (make_fuselse_logsumexp), forward or
  forward and backward, fp32 / fp16 / bf16;
* ``selective``: the fused selective log-softmax over shifted logits, forward
  and backward;
* ``int``: the fixed-point row kernels (Q16.16 of fp32 or int32, Q10.6);
* ``csr``: a sparse probabilistic-circuit sum layer with CSR edges, as an
  autograd layer in fp32 or its Q16.16 forward;
* ``block``: the same in pyjuice's block layout, as an autograd layer in fp32
  or through the forward dispatcher in fp32 or Q16.16.

``listed`` gives the cases, ``draw`` one more of the same ranges, ``prepare``
what a program holds before the call, ``run`` one pass, ``work`` the bytes and
operations a pass cannot do without, ``tolerance`` how far another correct
implementation may be off, and ``exact`` the results in 64 bits.
"""

import math

import torch

import fuselse_amd
from fuselse_amd import ext, pc

DEVICE = "cuda"
DTYPES = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}
LN2 = math.log(2.0)

# Most work of a drawn case: the largest listed one of its path.
MAX_DENSE = 512 * 128256
MAX_SELECTIVE = 8 * 1024 * 50257
MAX_CSR = 1_000_000 * 512
MAX_BLOCK = 8192 * 32 * 32 * 512


def listed():
    return [
        # A user's first call and the smallest in real use: a few short rows,
        # where the launch and the host side are all there is.
        {"name": "lse_small_f32", "path": "lse", "dtype": "f32", "robust": True, "grad": False, "rows": 32, "cols": 256},
        # Decoding: the log-normaliser of one step of a small batch over a
        # language model's vocabulary; few long rows.
        {"name": "lse_decode_f32", "path": "lse", "dtype": "f32", "robust": True, "grad": False, "rows": 8,
         "cols": 128256},
        # Many short rows in half precision (attention scores, class logits).
        {"name": "lse_short_f16", "path": "lse", "dtype": "f16", "robust": False, "grad": False, "rows": 65536,
         "cols": 256},
        # The training loss of a language model in fp32: forward and backward
        # over vocabulary logits, some of them masked to -inf.
        {"name": "lse_train_f32", "path": "lse", "dtype": "f32", "robust": True, "grad": True, "rows": 512,
         "cols": 128256},
        # The same in bf16 at a smaller vocabulary.
        {"name": "lse_train_bf16", "path": "lse", "dtype": "bf16", "robust": True, "grad": True, "rows": 4096,
         "cols": 32000},
        # RLHF: log-probabilities of the sampled tokens, forward and backward,
        # over logits[:, :-1] of an odd vocabulary (rows are not 16-byte
        # aligned, and the view is not contiguous).
        {"name": "selective_train_f32", "path": "selective", "batch": 8, "seq": 1024, "cols": 50257},
        # Fixed-point log-sum-exp of vocabulary logits quantised in the kernel.
        {"name": "int_q16_f32", "path": "int", "format": "q16_f32", "rows": 512, "cols": 128256},
        # Fixed-point at 16 bits, inputs quantised beforehand.
        {"name": "int_q10_6", "path": "int", "format": "q10_6", "rows": 1024, "cols": 32000},
        # A large probabilistic circuit's sum layer, one training step of it:
        # a million nodes, power-law fan-in, random children.
        {"name": "csr_train_f32", "path": "csr", "q16": False, "nodes": 1_000_000, "children": 1_000_000, "batch": 512},
        # Fixed-point inference of a middle-sized one at a ragged batch.
        {"name": "csr_q16", "path": "csr", "q16": True, "nodes": 200_000, "children": 150_000, "batch": 100},
        # pyjuice's block layout, one training step of a layer of 262144 nodes.
        {"name": "block_train_f32", "path": "block", "q16": False, "train": True, "blocks": 8192, "block_size": 32,
         "edges": 32, "elements": 262144, "batch": 512},
        # The forward dispatcher a pyjuice model is patched with, in fixed
        # point, as a hidden-Markov-like layer of latent size 32 calls it.
        {"name": "block_q16", "path": "block", "q16": True, "train": False, "blocks": 2048, "block_size": 32,
         "edges": 32, "elements": 65536, "batch": 512},
    ]


def _log_int(rng, lo, hi):
    """An integer of [lo, hi], spread over its logarithm."""
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    path = rng.choice(["lse", "lse", "lse", "selective", "int", "csr", "csr", "block", "block"])
    if path == "lse":
        cols = _log_int(rng, 2, 131072)
        return {"path": path, "dtype": rng.choice(["f32", "f32", "f16", "bf16"]), "robust": rng.random() < 0.7,
                "grad": rng.random() < 0.5, "rows": _log_int(rng, 1, min(65536, MAX_DENSE // cols)), "cols": cols}
    if path == "selective":
        batch = rng.randint(1, 16)
        cols = _log_int(rng, 1000, 131072)
        return {"path": path, "batch": batch, "seq": _log_int(rng, 2, min(2048, MAX_SELECTIVE // (batch * cols))),
                "cols": cols}
    if path == "int":
        cols = _log_int(rng, 2, 131072)
        return {"path": path, "format": rng.choice(["q16_f32", "q16_i32", "q10_6"]),
                "rows": _log_int(rng, 1, min(65536, MAX_DENSE // cols)), "cols": cols}
    if path == "csr":
        nodes = _log_int(rng, 1000, 1_000_000)
        return {"path": path, "q16": rng.random() < 0.4, "nodes": nodes,
                "children": _log_int(rng, max(500, nodes // 4), nodes),
                "batch": _log_int(rng, 1, min(512, MAX_CSR // nodes))}
    q16 = rng.random() < 0.4
    train = not q16 and rng.random() < 0.7
    block_size = rng.choice([1, 2, 4, 8, 16, 24, 32, 32, 64, 128])
    edges = _log_int(rng, 2, 128)
    batch = _log_int(rng, 1, 512)
    blocks = _log_int(rng, 16, max(16, min(16384, MAX_BLOCK // (block_size * edges * batch),
                                           MAX_CSR // (block_size * batch), MAX_CSR // (edges * batch))))
    return {"path": path, "q16": q16, "train": train, "blocks": blocks, "block_size": block_size, "edges": edges,
            "elements": _log_int(rng, max(edges, blocks * edges // 4), blocks * edges), "batch": batch}


# ---------------------------------------------------------------------------
# Inputs
# ---------------------------------------------------------------------------
def _generator(seed):
    gen = torch.Generator(device=DEVICE)
    gen.manual_seed(int(seed))
    return gen


def _logits(rows, cols, gen):
    """Vocabulary logits: N(0, 3^2), one in a thousand raised by 15."""
    x = torch.randn(rows, cols, device=DEVICE, generator=gen).mul_(3.0)
    spikes = torch.randint(0, rows * cols, (max(1, rows * cols // 1000),), device=DEVICE, generator=gen)
    x.view(-1)[spikes] = 15.0
    return x


def _prepare_lse(case, gen):
    x = _logits(case["rows"], case["cols"], gen)
    if case["robust"] and case["cols"] > 2:
        # one row in a hundred has half of its logits masked out
        x[::100, 1:(case["cols"] + 1) // 2] = float("-inf")
    x = x.to(DTYPES[case["dtype"]])
    g = torch.randn(case["rows"], device=DEVICE, generator=gen).to(x.dtype)
    fn = fuselse_amd.make_fuselse_logsumexp(ext, robust=case["robust"], half_inputs=case["dtype"] != "f32")
    return {"fn": fn, "x": x.requires_grad_(case["grad"]), "g": g}


def _prepare_selective(case, gen):
    b, s, v = case["batch"], case["seq"], case["cols"]
    full = _logits(b * s, v, gen).view(b, s, v)
    ids = torch.randint(0, v, (b, s), device=DEVICE, generator=gen)
    g = torch.randn(b, s - 1, device=DEVICE, generator=gen)
    return {"full": full, "logits": full[:, :-1].requires_grad_(True), "ids": ids, "g": g}


def _prepare_int(case, gen):
    x = torch.randn(case["rows"], case["cols"], device=DEVICE, generator=gen).mul_(2.0)
    if case["format"] == "q16_i32":
        x = torch.round(x * (65536.0 / LN2)).to(torch.int32)
    elif case["format"] == "q10_6":
        x = torch.round(x * (64.0 / LN2)).to(torch.int16)
    return {"x": x}


def _log_uniform(rows, batch, gen):
    """Log-probabilities log(U(0, 1)) of children."""
    return torch.rand(rows, batch, device=DEVICE, generator=gen).clamp_min_(1e-30).log_()


def _csr_edges(case, gen):
    """Fan-in k of [2, 256] with p(k) proportional to k^-2 (the distribution's
    quantiles in a random order, so a layer's edge count is a function of its
    sizes), children uniform, log-weights N(0, 1) less about their node's
    log-normaliser."""
    k = torch.arange(2, 257, dtype=torch.float64)
    cdf = torch.cumsum(k ** -2, 0)
    cdf = (cdf / cdf[-1]).to(DEVICE)
    u = (torch.arange(case["nodes"], device=DEVICE, dtype=torch.float64) + 0.5) / case["nodes"]
    fan = torch.searchsorted(cdf, u).clamp_max_(254) + 2
    fan = fan[torch.randperm(case["nodes"], device=DEVICE, generator=gen)]
    offsets = torch.zeros(case["nodes"] + 1, dtype=torch.int64, device=DEVICE)
    torch.cumsum(fan, 0, out=offsets[1:])
    edges = int(offsets[-1])
    ids = torch.randint(0, case["children"], (edges,), device=DEVICE, generator=gen, dtype=torch.int32)
    logw = torch.randn(edges, device=DEVICE, generator=gen)
    logw -= torch.repeat_interleave(torch.log(fan.float()) + 0.5, fan, output_size=edges)
    return offsets, ids, logw


def _prepare_csr(case, gen):
    offsets, ids, logw = _csr_edges(case, gen)
    child = _log_uniform(case["children"], case["batch"], gen)
    state = {"offsets": offsets, "ids": ids, "logw": logw, "child": child}
    if not case["q16"]:
        child.requires_grad_(True)
        logw.requires_grad_(True)
        state["g"] = torch.rand(case["nodes"], case["batch"], device=DEVICE, generator=gen)
        state["csc"] = ext.sparse_csr_transpose(offsets, ids, case["children"])
    return state


class _Layer:
    def __init__(self, block_size):
        self.block_size = block_size


def _prepare_block(case, gen):
    nb, bs, ne, nel = case["blocks"], case["block_size"], case["edges"], case["elements"]
    nids = torch.arange(nb, device=DEVICE, dtype=torch.int64) * bs
    cids = torch.randint(0, nel, (nb, ne), device=DEVICE, generator=gen, dtype=torch.int64)
    pids = (torch.arange(nb * ne, device=DEVICE, dtype=torch.int64) * bs).reshape(nb, ne)
    weights = torch.rand(nb * ne * bs, device=DEVICE, generator=gen).add_(1e-3).div_(ne / 2)
    elements = _log_uniform(nel, case["batch"], gen)
    state = {"nids": nids, "cids": cids, "pids": pids, "elements": elements, "nodes": nb * bs}
    if case["train"]:
        state["params"] = weights.log_().requires_grad_(True)
        elements.requires_grad_(True)
        state["g"] = torch.rand(nb * bs, case["batch"], device=DEVICE, generator=gen)
        state["plan"] = ext.sparse_blocked_transpose(nids, cids, pids, bs, nel)
    else:
        state["params"] = weights
        state["layer"] = _Layer(bs)
        state["call"] = pc.make_sparse_dispatcher(ext.sparse_forward_q16 if case["q16"] else ext.sparse_forward_float)
        state["out"] = torch.full((nb * bs, case["batch"]), float("-inf"), device=DEVICE)
    return state


def prepare(case, seed):
    gen = _generator(seed)
    make = {"lse": _prepare_lse, "selective": _prepare_selective, "int": _prepare_int, "csr": _prepare_csr,
            "block": _prepare_block}[case["path"]]
    state = make(case, gen)
    state["case"] = case
    return state


# ---------------------------------------------------------------------------
# One pass
# ---------------------------------------------------------------------------
_INT_CALLS = {"q16_f32": ext.batched_logsumexp, "q16_i32": ext.batched_logsumexp_q16_i32,
              "q10_6": ext.batched_logsumexp_q10_6}


def run(state):
    case = state["case"]
    path = case["path"]
    if path == "lse":
        y = state["fn"](state["x"], dim=-1)
        if not case["grad"]:
            return {"lse": y}
        (gx,) = torch.autograd.grad(y, state["x"], state["g"])
        return {"lse": y.detach(), "grad": gx}
    if path == "selective":
        y = fuselse_amd.selective_log_softmax(state["logits"], state["ids"][:, 1:])
        (gx,) = torch.autograd.grad(y, state["logits"], state["g"])
        return {"logp": y.detach(), "grad": gx}
    if path == "int":
        return {"lse": _INT_CALLS[case["format"]](state["x"])}
    if path == "csr":
        if case["q16"]:
            return {"out": ext.sparse_csr_forward(state["child"], state["offsets"], state["ids"], state["logw"], q16=True)}
        y = pc.sparse_csr_layer(state["child"], state["offsets"], state["ids"], state["logw"], csc=state["csc"])
        gc, gw = torch.autograd.grad(y, (state["child"], state["logw"]), state["g"])
        return {"out": y.detach(), "grad_child": gc, "grad_logw": gw}
    if case["train"]:
        y = pc.sparse_blocked_layer(state["elements"], state["params"], state["nids"], state["cids"], state["pids"],
                                    case["block_size"], state["nodes"], plan=state["plan"])
        ge, gp = torch.autograd.grad(y, (state["elements"], state["params"]), state["g"])
        return {"out": y.detach(), "grad_elements": ge, "grad_params": gp}
    state["call"](state["layer"], state["out"], state["elements"], state["params"], state["nids"], state["cids"],
                  state["pids"])
    return {"out": state["out"]}


# ---------------------------------------------------------------------------
# What a pass cannot do without
# ---------------------------------------------------------------------------
def work(case):
    """Each operand read once and each result written once per direction: a
    backward begins when its upstream gradient is there, so it reads the
    forward's inputs again.  Operations are counted per element or edge term
    as one multiply-add and one exponential."""
    path = case["path"]
    if path in ("lse", "int", "selective"):
        if path == "selective":
            rows, size = case["batch"] * (case["seq"] - 1), 4
        elif path == "lse":
            rows, size = case["rows"], 4 if case["dtype"] == "f32" else 2
        else:
            rows, size = case["rows"], 2 if case["format"] == "q10_6" else 4
        n = rows * case["cols"]
        forward = n * size + rows * (12 if path == "selective" else 4)
        if path == "int" or (path == "lse" and not case["grad"]):
            return {"bytes": forward, "flops": 3 * n}
        return {"bytes": forward + 2 * n * size + rows * 16, "flops": 6 * n}
    b = case["batch"]
    if path == "csr":
        # the mean of k over p(k) ~ k^-2 on [2, 256]
        ks = range(2, 257)
        mean = sum(1.0 / k for k in ks) / sum(1.0 / (k * k) for k in ks)
        edges = int(case["nodes"] * mean)
        used = case["children"] * (1.0 - math.exp(-edges / case["children"]))
        forward = used * b * 4 + case["nodes"] * (b * 4 + 8) + edges * 8
        if case["q16"]:
            return {"bytes": forward, "flops": 3 * edges * b}
        backward = (used + case["children"]) * b * 4 + case["nodes"] * b * 8 + edges * 16
        return {"bytes": forward + backward, "flops": 8 * edges * b}
    nodes, edges = case["blocks"] * case["block_size"], case["blocks"] * case["edges"]
    used = case["elements"] * (1.0 - math.exp(-edges / case["elements"]))
    terms = edges * case["block_size"]
    forward = used * b * 4 + nodes * b * 4 + edges * 16 + terms * 4
    if not case["train"]:
        return {"bytes": forward, "flops": 2 * terms * b}
    backward = (used + case["elements"]) * b * 4 + nodes * b * 8 + edges * 16 + terms * 8
    return {"bytes": forward + backward, "flops": 6 * terms * b}


def tolerance(case):
    if case["path"] == "int" or case.get("q16"):
        return "exact"  # the fixed-point arithmetic defines every bit
    # about four times the error measured against exact(): half-type results
    # and gradients are rounded to their type (2-norm 2.1e-4 in fp16, 1.9e-3
    # in bf16), fp32 gradients carry the rounding of x - lse (6.6e-7), the
    # circuits' parameter gradients their sums over the batch (3.3e-7)
    if case["path"] == "lse" and case["dtype"] == "f16":
        return {"rel": 1e-3, "max": 8e-3}
    if case["path"] == "lse" and case["dtype"] == "bf16":
        return {"rel": 8e-3, "max": 4e-2}
    return {"rel": 4e-6, "max": 1e-4}


# ---------------------------------------------------------------------------
# The same in 64 bits
# ---------------------------------------------------------------------------
def _row_chunks(rows, cols):
    step = max(1, (1 << 27) // cols)
    return [(r, min(rows, r + step)) for r in range(0, rows, step)]


def _exact_rows(x, g, index):
    """(lse or selected log-probability, gradient) of each row, chunk by chunk."""
    rows, cols = x.shape
    y = torch.empty(rows, dtype=torch.float64, device=x.device)
    gx = None if g is None else torch.empty(rows, cols, dtype=torch.float64, device=x.device)
    for r0, r1 in _row_chunks(rows, cols):
        xc = x[r0:r1].double()
        lse = torch.logsumexp(xc, -1)
        y[r0:r1] = lse if index is None else xc.gather(1, index[r0:r1, None])[:, 0] - lse
        if g is not None:
            p = torch.exp(xc - lse[:, None])
            if index is not None:
                p = -p
                p.scatter_add_(1, index[r0:r1, None], torch.ones_like(lse)[:, None])
            gx[r0:r1] = p * g[r0:r1, None].double()
    return y, gx


def _exact_int(case, x):
    scale = {"q16_f32": 1.0, "q16_i32": LN2 / 65536.0, "q10_6": LN2 / 64.0}[case["format"]]
    y = torch.empty(case["rows"], dtype=torch.float64, device=x.device)
    for r0, r1 in _row_chunks(case["rows"], case["cols"]):
        y[r0:r1] = torch.logsumexp(x[r0:r1].double() * scale, -1)
    return y


def _exact_csr(case, s):
    nodes, batch = case["nodes"], case["batch"]
    ids, logw = s["ids"].long(), s["logw"].detach().double()
    parent = torch.repeat_interleave(torch.arange(nodes, device=DEVICE), s["offsets"].diff())
    out = torch.empty(nodes, batch, dtype=torch.float64, device=DEVICE)
    train = not case["q16"]
    if train:
        gc = torch.zeros(case["children"], batch, dtype=torch.float64, device=DEVICE)
        gw = torch.zeros(logw.numel(), dtype=torch.float64, device=DEVICE)
    step = max(1, (1 << 27) // logw.numel())
    for b0 in range(0, batch, step):
        cols = slice(b0, min(batch, b0 + step))
        t = logw[:, None] + s["child"].detach()[:, cols].double()[ids]
        width = t.shape[1]
        top = torch.full((nodes, width), float("-inf"), dtype=torch.float64, device=DEVICE)
        top.scatter_reduce_(0, parent[:, None].expand(-1, width), t, "amax")
        total = torch.zeros(nodes, width, dtype=torch.float64, device=DEVICE)
        total.index_add_(0, parent, torch.exp(t - top[parent]))
        out[:, cols] = top + torch.log(total)
        if train:
            flow = torch.exp(t - out[:, cols][parent]) * s["g"][:, cols].double()[parent]
            gw += flow.sum(1)
            part = torch.zeros(case["children"], width, dtype=torch.float64, device=DEVICE)
            gc[:, cols] = part.index_add_(0, ids, flow)
    return {"out": out, "grad_child": gc, "grad_logw": gw} if train else {"out": out}


def _exact_block(case, s):
    nb, bs, ne, batch = case["blocks"], case["block_size"], case["edges"], case["batch"]
    x, w = s["elements"].detach(), s["params"].detach().double()
    logw = w if case["train"] else torch.log(w)
    train = case["train"]
    out = torch.empty(nb * bs, batch, dtype=torch.float64, device=DEVICE)
    if train:
        ge = torch.zeros(case["elements"], batch, dtype=torch.float64, device=DEVICE)
        gp = torch.empty(nb, ne, bs, dtype=torch.float64, device=DEVICE)
    lw = logw.view(nb, ne, bs).transpose(1, 2).contiguous()
    step = max(1, (1 << 26) // (max(bs, ne) * batch))
    for j0 in range(0, nb, step):
        j1 = min(nb, j0 + step)
        rows = s["cids"][j0:j1].reshape(-1)
        xe = x[rows].double().view(j1 - j0, ne, batch)
        top = xe.amax(1, keepdim=True)
        e, a = torch.exp(xe - top), torch.exp(lw[j0:j1])
        total = torch.matmul(a, e)
        out[j0 * bs:j1 * bs] = (top + torch.log(total)).reshape(-1, batch)
        if train:
            r = s["g"][j0 * bs:j1 * bs].double().view(j1 - j0, bs, batch) / total
            ge.index_add_(0, rows, (e * torch.matmul(a.transpose(1, 2).contiguous(), r)).view(-1, batch))
            p = a * torch.matmul(r, e.transpose(1, 2).contiguous())
            gp[j0:j1] = p.transpose(1, 2)
    return {"out": out, "grad_elements": ge, "grad_params": gp.reshape(-1)} if train else {"out": out}


def exact(case, seed):
    s = prepare(case, seed)
    if case["path"] == "lse":
        y, gx = _exact_rows(s["x"].detach(), s["g"] if case["grad"] else None, None)
        return {"lse": y, "grad": gx} if case["grad"] else {"lse": y}
    if case["path"] == "selective":
        x = s["logits"].detach().reshape(-1, case["cols"])
        y, gx = _exact_rows(x, s["g"].reshape(-1), s["ids"][:, 1:].reshape(-1))
        shape = (case["batch"], case["seq"] - 1)
        return {"logp": y.view(shape), "grad": gx.view(*shape, case["cols"])}
    if case["path"] == "int":
        return {"lse": _exact_int(case, s["x"])}
    return _exact_csr(case, s) if case["path"] == "csr" else _exact_block(case, s)
