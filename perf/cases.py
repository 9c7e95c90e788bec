"""The work a user of this package has it do, as measurable cases.

Every case is one pass through the public calls (``SparseLayout``, ``matmul``, ``softmax``, ``attention``):

    layout      a new block mask arrives: build its tables, gather a dense matrix into its block stack, scatter it back
    sdd|dsd|dds one block-sparse product, forward, or forward and both gradients (``train``)
    softmax     the masked row softmax over a block stack
    chain       scores = q k^T, softmax, probabilities times v, as three calls
    attention   the same as one call

Sizes are in blocks of 32: ``rows`` x ``cols`` is the block mask, ``dim`` the free dense dimension (head dim of
attention, tokens of a sparse linear layer), ``batch`` the flattened batch x heads.  ``shared``: one block-sparse
weight for the whole batch.  Masks are those of ``workloads.py``.  Run with the repository's root as the working
folder.
"""
import os
import random
import sys

import torch

sys.path.insert(0, os.path.abspath("experiments-pytorch-cuda-extension-for-sparse-matmul_amd"))

import sparse  # noqa: E402
import workloads as wl  # noqa: E402

BLOCK = 32
DTYPES = {"fp32": torch.float32, "fp16": torch.float16, "bf16": torch.bfloat16}
ITEM = {"fp32": 4, "fp16": 2, "bf16": 2}
DEFAULTS = {"train": False, "trans_a": False, "trans_b": False, "shared": False, "causal": False, "mask_seed": 1005}


def _case(name, path, dtype, mask, rows, batch, dim, **more):
    case = {"path": path, "dtype": dtype, "mask": mask, "rows": rows, "cols": rows, "batch": batch, "dim": dim}
    case.update(DEFAULTS)
    case.update(more)
    if name:
        case["name"] = name
    return case


def listed():
    return [
        # the smallest call: one head of 512 tokens in fp32, the reference's own type; latency of a single product
        _case("sdd_fp32_512", "sdd", "fp32", "random:0.25", 16, 1, 64, trans_b=True, mask_seed=1001),
        # probabilities times values of a sliding-window layer, 2048 tokens, 16 heads
        _case("dsd_fp16_local_2048", "dsd", "fp16", "local:2", 64, 16, 64),
        # the softmax of a training step, causal local + strided mask, 4096 tokens, 16 heads
        _case("softmax_train_fp16_4096", "softmax", "fp16", "causal:4:8", 128, 16, 64, causal=True, train=True),
        # dense times sparse over the columns of the same mask (a transposed activation against block-sparse scores)
        _case("dds_fp16_4096", "dds", "fp16", "causal:4:8", 128, 16, 64, trans_a=True),
        # inference over long documents with a local + global + random mask: 8192 tokens, 4 x 12 heads, three calls
        _case("chain_fp16_bigbird_8192", "chain", "fp16", "bigbird:1:2:3", 256, 48, 64),
        # a training step of the three-call chain, 4096 tokens, 16 heads
        _case("chain_train_fp16_4096", "chain", "fp16", "causal:4:8", 128, 16, 64, causal=True, train=True),
        # the same in the reference's own type at an ordinary size: 2048 tokens, 16 heads
        _case("chain_train_fp32_2048", "chain", "fp32", "causal:4:8", 64, 16, 64, causal=True, train=True),
        # scoring a ragged batch with the fused operator: 2976 tokens, 3 x 5 heads, nothing a power of two
        _case("attention_fp16_ragged", "attention", "fp16", "causal:5:7", 93, 15, 64, causal=True),
        # the largest: a training step of the fused operator over long documents in bf16, 8192 tokens, 4 x 12 heads
        _case("attention_train_bf16_8192", "attention", "bf16", "bigbird:1:2:3", 256, 48, 64, train=True),
        # a training step of the fused operator with heads of 128, 4096 tokens
        _case("attention_train_fp16_d128", "attention", "fp16", "causal:4:8", 128, 16, 128, causal=True, train=True),
        # a linear layer with a block-sparse weight, 2048 x 2048 at a quarter of its blocks, forward and gradients,
        # 4 sequences of 1056 tokens (33 blocks: no multiple of 64)
        _case("weight_train_bf16", "dds", "bf16", "random:0.25", 64, 4, 1056, shared=True, train=True),
        # a mask that changes from call to call: tables, gather and scatter of 8 matrices of 2048 x 2048
        _case("layout_fp16_2048", "layout", "fp16", "random:0.10", 64, 8, 2048),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, round(lo * (hi / lo) ** rng.random())))


def draw(rng: random.Random):
    path = rng.choice(["sdd", "dsd", "dds", "softmax", "chain", "chain", "attention", "attention", "attention",
                       "weight", "layout"])
    kind = rng.choice(["local", "causal", "causal", "bigbird", "random"])
    mask = {"local": lambda: f"local:{rng.randint(1, 4)}",
            "causal": lambda: f"causal:{rng.randint(2, 6)}:{rng.randint(5, 16)}",
            "bigbird": lambda: f"bigbird:1:{rng.randint(1, 2)}:{rng.randint(2, 4)}",
            "random": lambda: f"random:{rng.uniform(0.04, 0.25):.3f}"}[kind]()
    case = _case(None, path, rng.choice(["fp16", "fp16", "bf16", "fp32"]), mask,
                 _log_int(rng, 16, 128 if kind == "random" else 256), _log_int(rng, 1, 48), 64,
                 causal=kind == "causal", train=rng.random() < 0.5, mask_seed=rng.randrange(10 ** 6))
    if path == "attention":
        case["dtype"] = rng.choice(["fp16", "bf16"])
        case["dim"] = rng.choice([64, 64, 64, 128])
    elif path == "chain":
        case["dim"] = rng.choice([32, 64, 64, 96, 128])
    elif path in ("sdd", "dsd", "dds"):
        case["dim"] = BLOCK * rng.randint(1, 6)
        case["trans_a"], case["trans_b"] = rng.random() < 0.5, rng.random() < 0.5
        if kind == "random":
            case["cols"] = _log_int(rng, 16, 128)
    elif path == "weight":
        case.update(path="dds", shared=True, causal=False, mask=f"random:{rng.uniform(0.08, 0.3):.3f}",
                    rows=_log_int(rng, 16, 96), cols=_log_int(rng, 16, 96), batch=_log_int(rng, 1, 8),
                    dim=BLOCK * _log_int(rng, 2, 64))
    elif path == "layout":
        case.update(mask=f"random:{rng.uniform(0.04, 0.25):.3f}", train=False, causal=False,
                    batch=_log_int(rng, 1, 16), rows=_log_int(rng, 16, 128), cols=_log_int(rng, 16, 128))
    most = max(_cost(c) for c in listed())
    while _cost(case) > most:
        if case["batch"] > 1:
            case["batch"] = case["batch"] * 3 // 4
        else:
            case["rows"], case["cols"] = max(16, case["rows"] * 3 // 4), max(16, case["cols"] * 3 // 4)
    return case


def _cost(case):
    w = work(case)
    return max(w["bytes"], w["flops"] / 50)


def _mask(case):
    """The block mask of a case: a property of the model, the same for every seed of the data."""
    kind, *args = case["mask"].split(":")
    rows, cols = case["rows"], case["cols"]
    gen = torch.Generator().manual_seed(case["mask_seed"])
    if kind == "local":
        return wl.mask_local_window(rows, int(args[0]))
    if kind == "causal":
        return wl.mask_causal_local_strided(rows, int(args[0]), int(args[1]))
    if kind == "bigbird":
        return wl.mask_bigbird(rows, gen, int(args[0]), int(args[1]), int(args[2]))
    if rows == cols:
        return wl.mask_random_diag(rows, float(args[0]), gen)
    return (torch.rand(rows, cols, generator=gen) < float(args[0])).long().index_fill_(1, torch.tensor([0]), 1)


def _kept(case):
    """Blocks per row of the mask of the ``layout`` path, whose mask is an input and drawn from the seed."""
    return max(1, round(float(case["mask"].split(":")[1]) * case["cols"]))


def _blocks(case):
    return case["rows"] * _kept(case) if case["path"] == "layout" else int(_mask(case).sum())


def _dense_shape(case, mode, which):
    """Stored shape of the dense operand ``which`` (0: a, 1: b) of a product."""
    r, c, d = BLOCK * case["rows"], BLOCK * case["cols"], case["dim"]
    ta, tb = case["trans_a"], case["trans_b"]
    if mode == "sdd":                     # op(a) is r x d, op(b) is d x c
        return ((d, r) if ta else (r, d)) if which == 0 else ((c, d) if tb else (d, c))
    if mode == "dsd":                     # op(a) is the mask or its transpose, op(b) has as many rows as it has columns
        k = r if ta else c
        return (d, k) if tb else (k, d)
    k = c if tb else r                    # dds: op(b) is the mask or its transpose, op(a) is d x its rows
    return (k, d) if ta else (d, k)


def prepare(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    dtype = DTYPES[case["dtype"]]
    batch, rows, cols, dim = case["batch"], case["rows"], case["cols"], case["dim"]

    def normal(*shape, std=1.0, grad=False):
        x = torch.randn(*shape, generator=gen, device="cuda", dtype=torch.float32).mul_(std).to(dtype)
        return x.requires_grad_(grad)

    state = {"case": case}
    if case["path"] == "layout":
        keys = torch.rand(rows, cols, generator=gen, device="cuda")
        pattern = torch.zeros(rows, cols, dtype=torch.int64, device="cuda")
        state["pattern"] = pattern.scatter_(1, keys.topk(_kept(case), dim=1).indices, 1)
        state["x"] = normal(batch, BLOCK * rows, BLOCK * cols)
        return state

    layout = state["layout"] = sparse.SparseLayout(_mask(case).cuda())
    train, nnz = case["train"], layout.num_blocks
    if case["path"] in ("chain", "attention"):
        state["args"] = tuple(normal(batch, BLOCK * n, dim, grad=train) for n in (rows, cols, cols))
        grad_shape = (batch, BLOCK * rows, dim)
    elif case["path"] == "softmax":
        state["args"] = (normal(batch, nnz, BLOCK, BLOCK, std=2.0, grad=train),)
        grad_shape = (batch, nnz, BLOCK, BLOCK)
    else:
        mode, args = case["path"], []
        for which in (0, 1):
            if mode[1 + which] == "s":
                lead = () if case["shared"] else (batch,)
                args.append(normal(*lead, nnz, BLOCK, BLOCK, std=0.02 if case["shared"] else 0.1, grad=train))
            else:
                args.append(normal(batch, *_dense_shape(case, mode, which), grad=train))
        state["args"] = tuple(args)
        r, c = (BLOCK * n for n in (rows, cols))
        grad_shape = {"sdd": (batch, nnz, BLOCK, BLOCK), "dsd": (batch, c if case["trans_a"] else r, dim),
                      "dds": (batch, dim, r if case["trans_b"] else c)}[mode]
    if train:
        state["grad"] = normal(*grad_shape)
    return state


def _forward(case, layout, args):
    if case["path"] == "chain":
        q, k, v = args
        scores = sparse.matmul(q, k, "sdd", layout, False, True)
        probs = sparse.softmax(scores, layout, case["dim"] ** -0.5, case["causal"])
        return sparse.matmul(probs, v, "dsd", layout)
    if case["path"] == "attention":
        return sparse.attention(*args, layout, case["dim"] ** -0.5, case["causal"])
    if case["path"] == "softmax":
        return sparse.softmax(*args, layout, 0.125, case["causal"])
    return sparse.matmul(*args, case["path"], layout, case["trans_a"], case["trans_b"])


def run(state):
    case = state["case"]
    if case["path"] == "layout":
        layout = sparse.SparseLayout(state["pattern"])
        stack = layout.to_sparse(state["x"])
        return {"row": layout.row_layout, "col": layout.col_layout, "stack": stack, "dense": layout.to_dense(stack)}
    if not case["train"]:
        with torch.no_grad():
            return _forward(case, state["layout"], state["args"])
    out = _forward(case, state["layout"], state["args"])
    return (out,) + torch.autograd.grad(out, state["args"], state["grad"])


def work(case):
    """Bytes and operations of one pass: every operand of every call read once, every result written once."""
    es, batch, dim, nnz = ITEM[case["dtype"]], case["batch"], case["dim"], _blocks(case)
    rows, cols = BLOCK * case["rows"], BLOCK * case["cols"]
    stack, product = nnz * BLOCK * BLOCK, 2.0 * nnz * BLOCK * BLOCK * dim * batch
    q, kv = rows * dim * batch, cols * dim * batch
    if case["path"] == "layout":          # mask, two tables, the stored blocks twice in and out, the dense matrix once out
        return {"bytes": 8 * case["rows"] * case["cols"] + 16 * nnz + es * batch * (3 * stack + rows * cols), "flops": 0}
    if case["path"] == "softmax":
        return {"bytes": es * batch * stack * (4 if case["train"] else 2), "flops": 5.0 * batch * stack}
    if case["path"] == "chain":           # scores and probabilities are results of calls of their own
        items = 2 * q + 2 * kv + 4 * batch * stack
        if case["train"]:                 # dv, dp | ds | dq, dk
            items += (q + 2 * kv) + (2 * batch * stack) + (3 * batch * stack) + (2 * q + 2 * kv + batch * stack)
        return {"bytes": es * items, "flops": product * (6 if case["train"] else 2)}
    if case["path"] == "attention":
        items = 2 * q + 2 * kv
        if case["train"]:                 # the result and its gradient in, three gradients out; five more products
            items += 3 * q + 2 * kv
        return {"bytes": es * items, "flops": product * (7 if case["train"] else 2)}
    items = q + kv + stack * (1 if case["shared"] else batch)
    return {"bytes": es * items * (2 if case["train"] else 1), "flops": product * (3 if case["train"] else 1)}


def tolerance(case):
    """Four times the largest relative error that the calls show against the same products in float64, over the listed
    cases and forty drawn ones: the rounding of results, and in a chain of the block stacks between its calls."""
    if case["path"] == "layout":
        return "exact"
    seen = {"fp32": 2.9e-7, "fp16": 3.5e-4, "bf16": 2.9e-3}
    if case["path"] == "chain":
        seen = {"fp32": 4.0e-7, "fp16": 6.0e-4, "bf16": 4.5e-3}
    return {"rel": 4 * seen[case["dtype"]]}
