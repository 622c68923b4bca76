"""The work a user of muon_amd has it do, as cases that can be timed: optimizer steps of whole models,
single matrices through the functional entry points, the three product operators and Adam.

A case is a dict of plain values; `kind` says which entry points it goes through:

  step      SingleDeviceMuonWithAuxAdam.step() of a transformer: `layers` blocks of `width` with
            key/value width `kv`, feed-forward width `ff` (two matrices, or three when `gated`), the query, key
            and value projections fused into one matrix when `fused_qkv`; Adam for the vocabulary
            matrix (`vocab` rows) and the norm weights
  convnet   the same class over the filters of a convolutional network of base width `channels` and two
            projections that are short and very long
  matrix    SingleDeviceMuon.step() over one matrix
  update    muon_update(grad, momentum) on one gradient (`kernel` > 0: a convolution filter)
  ns        zeropower_via_newtonschulz5(G) on a batch of matrices
  products  ns_line_1, ns_line_2, ns_line_3 with out= given: one iteration of a caller's own loop
  adam      adam_update(grad, exp_avg, exp_avg_sq) on one tensor

Model tensors are views into one flat buffer per role, as programs keep them that reduce or save them in
one piece, and the state is that of a run which is under way (momentum and moments are not zero).
"""
import torch

import muon_amd

DTYPES = {"fp32": torch.float32, "bf16": torch.bfloat16}
NS_COEFFS = (3.4445, -4.7750, 2.0315)
LR, WEIGHT_DECAY, MOMENTUM = 0.02, 0.01, 0.95
GRAD_STD, PARAM_STD = 1e-3, 0.02
ALIGN = 128                      # elements between the starts of two tensors in a flat buffer


def listed():
    def step(name, layers, width, kv, ff, gated, fused_qkv, vocab, dtype="fp32", variant="ns5", graph=False):
        return dict(name=name, kind="step", layers=layers, width=width, kv=kv, ff=ff, gated=gated, fused_qkv=fused_qkv,
                    vocab=vocab, dtype=dtype, variant=variant, graph=graph)

    return [
        # the smallest call: one small convolution filter through the functional update
        dict(name="update-64x64x3x3", kind="update", rows=64, cols=64, kernel=3, dtype="fp32"),
        # one feed-forward matrix of a small transformer, stepped by itself (a step hooked to each parameter)
        dict(name="matrix-768x3072", kind="matrix", rows=768, cols=3072, dtype="fp32"),
        # an odd-sized matrix, taller than wide, off every tile boundary
        dict(name="ns-1500x1100", kind="ns", batch=1, rows=1500, cols=1100, dtype="fp32"),
        # every filter of an image classifier and two projections of 128 x 16384
        dict(name="convnet-64", kind="convnet", channels=64, dtype="fp32"),
        # GPT-2-small: 48 matrices of 768 rows, the vocabulary and the norms with Adam
        step("gpt2-124m", 12, 768, 768, 3072, False, True, 50257),
        # a model of medium width, the four-iteration variant, its launches replayed from a graph
        step("decoder-1024-aol4-graph", 12, 1024, 1024, 4096, False, True, 32000, variant="aol4", graph=True),
        # widths that are no multiple of a 256 tile (as a width of 25 heads of 64 gives)
        step("decoder-1600", 6, 1600, 1600, 6400, False, True, 50257),
        # a model kept in bf16, grouped key/value heads, gated feed-forward of 21.5 tiles
        step("decoder-2048-bf16", 12, 2048, 512, 5504, True, False, 32000, dtype="bf16"),
        # the last quarter of Llama-3-8B with its output matrix (a pipeline stage): the largest
        step("llama3-8b-quarter", 8, 4096, 1024, 14336, True, False, 128256),
        # a batch of large square matrices, already bf16
        dict(name="ns-32x4096x4096-bf16", kind="ns", batch=32, rows=4096, cols=4096, dtype="bf16"),
        # the three operators on the feed-forward matrices of a small transformer
        dict(name="products-24x768x3072", kind="products", batch=24, m=768, n=3072, dtype="bf16"),
        # the vocabulary matrix of GPT-2-small through the functional Adam
        dict(name="adam-50257x768", kind="adam", rows=50257, cols=768, dtype="fp32"),
    ]


def draw(rng):
    def size(lo, hi):            # spread over the logarithm; odd sizes among them
        return int(round(lo * (hi / lo) ** rng.random()))

    kind = rng.choice(["step", "step", "step", "convnet", "matrix", "update", "ns", "ns", "products", "adam"])
    while True:
        if kind == "step":
            width = size(256, 4096)
            if rng.random() < 0.7:                               # mostly whole heads of 64, sometimes any width
                width = max(256, width // 64 * 64)
            gated = rng.random() < 0.5
            fused = not gated
            ff = 4 * width if not gated else int(width * rng.choice([8 / 3, 2.6875, 3.5])) // 8 * 8
            kv = width if fused else max(1, width // rng.choice([1, 4])) // 8 * 8
            dtype = rng.choice(["fp32", "fp32", "bf16"])
            variant = rng.choice(["ns5", "ns5", "ns5", "aol4"]) if dtype == "fp32" else "ns5"
            case = dict(kind=kind, layers=size(1, 16), width=width, kv=kv, ff=ff, gated=gated, fused_qkv=fused,
                        vocab=size(1000, 60000), dtype=dtype, variant=variant, graph=rng.random() < 0.25)
        elif kind == "convnet":
            case = dict(kind=kind, channels=size(24, 128), dtype="fp32")
        elif kind == "matrix":
            case = dict(kind=kind, rows=size(64, 4096), cols=size(64, 4096), dtype=rng.choice(["fp32", "bf16"]))
        elif kind == "update":
            kernel = rng.choice([0, 0, 3])
            hi = 2048 if not kernel else 512
            case = dict(kind=kind, rows=size(32, hi), cols=size(32, hi), kernel=kernel, dtype="fp32")
        elif kind == "ns":
            case = dict(kind=kind, batch=size(1, 32), rows=size(32, 4096), cols=size(32, 6000), dtype=rng.choice(["fp32", "bf16"]))
        elif kind == "products":
            m = size(128, 2048)
            case = dict(kind=kind, batch=size(1, 32), m=m, n=min(8192, m + size(1, 4 * m)), dtype="bf16")
        else:
            case = dict(kind=kind, rows=size(1, 60000), cols=size(64, 4096), dtype=rng.choice(["fp32", "bf16"]))
        w = work(case)
        if w["flops"] <= 4e13 and w["bytes"] <= 2e10:            # well under the largest listed case
            return case


# ---- the tensors of a case ---------------------------------------------------------------------------
def _shapes(case):
    """-> (Muon shapes, Adam shapes)"""
    k = case["kind"]
    if k == "step":
        w, kv, ff = case["width"], case["kv"], case["ff"]
        layer = [(w, 3 * w), (w, w)] if case["fused_qkv"] else [(w, w), (kv, w), (kv, w), (w, w)]
        layer += [(ff, w), (ff, w), (w, ff)] if case["gated"] else [(w, ff), (ff, w)]
        return layer * case["layers"], [(case["vocab"], w)] + [(w,)] * (2 * case["layers"] + 1)
    if k == "convnet":
        c = case["channels"]
        filters = [(c, 24), (4 * c, c), (4 * c, 4 * c), (4 * c, 4 * c), (8 * c, 4 * c), (8 * c, 8 * c), (8 * c, 8 * c), (8 * c, 8 * c)]
        return [(o, i, 3, 3) for o, i in filters] + [(2 * c, 256 * c), (256 * c, 2 * c)], [(24, 3, 2, 2), (10, 8 * c)]
    return [(case["rows"], case["cols"])], []


def _numel(shape):
    n = 1
    for s in shape:
        n *= s
    return n


def _flat(shapes, dtype, std, gen):
    """One buffer and its views, filled from the generator."""
    starts, end = [], 0
    for s in shapes:
        starts.append(end)
        end += -(-_numel(s) // ALIGN) * ALIGN
    buf = torch.empty(end, dtype=dtype, device="cuda").normal_(0.0, std, generator=gen)
    return buf, [buf[o:o + _numel(s)].view(s) for o, s in zip(starts, shapes)]


def prepare(case, seed):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    dtype, k = DTYPES[case["dtype"]], case["kind"]

    def normal(*shape, std=1.0):
        return torch.empty(*shape, dtype=dtype, device="cuda").normal_(0.0, std, generator=gen)

    if k in ("step", "convnet", "matrix"):
        muon, adam = _shapes(case)
        p_buf, p = _flat(muon, dtype, PARAM_STD, gen)
        g_buf, g = _flat(muon, dtype, GRAD_STD, gen)
        m_buf, m = _flat(muon, dtype, 0.3 * GRAD_STD, gen)
        params = [torch.nn.Parameter(t) for t in p]
        for q, grad in zip(params, g):
            q.grad = grad
        out = {"muon_params": p_buf, "momentum": m_buf}
        if k == "matrix":
            opt = muon_amd.SingleDeviceMuon(params, lr=LR, weight_decay=WEIGHT_DECAY, momentum=MOMENTUM)
        else:
            ap_buf, ap = _flat(adam, dtype, PARAM_STD, gen)
            ag_buf, ag = _flat(adam, dtype, GRAD_STD, gen)
            am_buf, am = _flat(adam, dtype, 0.3 * GRAD_STD, gen)
            av_buf, av = _flat(adam, dtype, GRAD_STD, gen)
            av_buf.square_()
            aux = [torch.nn.Parameter(t) for t in ap]
            for q, grad in zip(aux, ag):
                q.grad = grad
            opt = muon_amd.SingleDeviceMuonWithAuxAdam(
                [dict(params=params, use_muon=True, lr=LR, momentum=MOMENTUM, weight_decay=WEIGHT_DECAY),
                 dict(params=aux, use_muon=False, lr=3e-4, betas=(0.9, 0.95), eps=1e-10, weight_decay=WEIGHT_DECAY)],
                ns_variant=case.get("variant", "ns5"), use_graph=case.get("graph", False))
            for q, t, v in zip(aux, am, av):
                opt.state[q].update(exp_avg=t, exp_avg_sq=v, step=100)
            out.update(adam_params=ap_buf, exp_avg=am_buf, exp_avg_sq=av_buf)
        for q, t in zip(params, m):
            opt.state[q]["momentum_buffer"] = t
        return {"kind": k, "opt": opt, "out": out}
    if k == "update":
        shape = (case["rows"], case["cols"]) + ((case["kernel"],) * 2 if case["kernel"] else ())
        return {"kind": k, "grad": normal(*shape, std=GRAD_STD), "momentum": normal(*shape, std=0.3 * GRAD_STD)}
    if k == "ns":
        shape = (case["rows"], case["cols"]) if case["batch"] == 1 else (case["batch"], case["rows"], case["cols"])
        return {"kind": k, "G": normal(*shape)}
    if k == "products":
        b, m, n = case["batch"], case["m"], case["n"]
        # an iterate: singular values of at most about one
        X = normal(b, m, n, std=1.0 / (m ** 0.5 + n ** 0.5))
        return {"kind": k, "X": X, "A": torch.empty(b, m, m, dtype=dtype, device="cuda"),
                "B": torch.empty(b, m, m, dtype=dtype, device="cuda"), "C": torch.empty_like(X)}
    shape = (case["rows"], case["cols"])
    return {"kind": k, "grad": normal(*shape, std=GRAD_STD), "exp_avg": normal(*shape, std=0.3 * GRAD_STD),
            "exp_avg_sq": normal(*shape, std=GRAD_STD).square_()}


def run(state):
    k = state["kind"]
    if k in ("step", "convnet", "matrix"):
        state["opt"].step()
        return state["out"]
    if k == "update":
        return [muon_amd.muon_update(state["grad"], state["momentum"], beta=MOMENTUM), state["grad"], state["momentum"]]
    if k == "ns":
        return muon_amd.zeropower_via_newtonschulz5(state["G"], steps=5)
    if k == "products":
        a, b, c = NS_COEFFS
        A = muon_amd.ns_line_1(state["X"], out=state["A"])
        B = muon_amd.ns_line_2(A, alpha=c, beta=b, out=state["B"])
        return [A, B, muon_amd.ns_line_3(B, state["X"], a, out=state["C"])]
    upd = muon_amd.adam_update(state["grad"], state["exp_avg"], state["exp_avg_sq"], 100, (0.9, 0.95), 1e-10)
    return [upd, state["exp_avg"], state["exp_avg_sq"]]


# ---- what a pass cannot do without -------------------------------------------------------------------
def _ns_flops(rows, cols, steps=5):
    """Newton-Schulz on one matrix, the symmetric products counted once: per iteration A = X X^T,
    b A + c A A and a X + B X (the AOL variant: four such iterations)."""
    m, n = min(rows, cols), max(rows, cols)
    return steps * (m * (m + 1) * n + m * m * (m + 1) + 2 * m * m * n)


def work(case):
    e = 4 if case["dtype"] == "fp32" else 2
    k = case["kind"]
    if k in ("step", "convnet", "matrix"):
        muon, adam = _shapes(case)
        steps = 4 if case.get("variant") == "aol4" else 5
        return {"bytes": 5 * e * sum(map(_numel, muon)) + 7 * e * sum(map(_numel, adam)),
                "flops": sum(_ns_flops(s[0], _numel(s) // s[0], steps) for s in muon)}
    if k == "update":
        n = case["rows"] * case["cols"] * max(1, case["kernel"] ** 2)
        return {"bytes": n * (4 * e + 2), "flops": _ns_flops(case["rows"], n // case["rows"])}
    if k == "ns":
        return {"bytes": case["batch"] * case["rows"] * case["cols"] * (e + 2),
                "flops": case["batch"] * _ns_flops(case["rows"], case["cols"])}
    if k == "products":
        b, m, n = case["batch"], case["m"], case["n"]
        return {"bytes": b * 2 * (m * n + m * m + m * m + m * n), "flops": b * _ns_flops(m, n, 1)}
    return {"bytes": case["rows"] * case["cols"] * 6 * e, "flops": 12 * case["rows"] * case["cols"]}


def tolerance(case):
    """About four times what the path was seen to differ from itself with every sum in another order (rows
    and columns of each matrix permuted, and the result permuted back), over the listed cases and 24
    drawn ones; for Adam, from the same expressions in 64 bits.  The iteration amplifies bf16 rounding:
    its output differs by up to 2.0e-2 (the largest element by 0.16), and parameters by that times
    the share of a step in them (3.4e-4 and 1.4e-2 in fp32, 1.5e-3 and 1.2e-2 in bf16)."""
    k, fp32 = case["kind"], case["dtype"] == "fp32"
    if k in ("step", "convnet", "matrix"):
        return {"rel": 1.4e-3, "max": 0.06} if fp32 else {"rel": 6e-3, "max": 0.05}
    if k in ("update", "ns"):
        return {"rel": 0.03, "max": 0.6}
    if k == "products":                 # seen: 2.9e-4 and 1.4e-2
        return {"rel": 1.2e-3, "max": 0.06}
    return {"rel": 3e-7, "max": 2e-6} if fp32 else {"rel": 1.5e-2, "max": 0.1}
