"""The work users of this package have it do, as cases that can be timed and compared.

Two kinds of case, both through the public entry points:

  ``ortho``  one call of an orthogonalization operator (``zeropower_via_newtonschulz5``, ``polar_express``,
             ``gram_newton_schulz``) on a batch of matrices, as a caller of the operators, or an optimizer of
             the caller's own, makes it;
  ``step``   one ``optimizer.step()`` of ``Muon`` / ``NorMuon`` / ``Dion2`` / ``NorDion2`` over the parameters of a
             transformer, with the embedding, head and norm parameters in an AdamW or Lion group where the case
             has a vocabulary.

A step starts from the state of a run under way (non-zero momentum and second moments).  Parameters and state of
one shape live in one allocation each, every tensor 256-byte aligned as the allocator would place it, so that a
pass returns a few whole buffers instead of several hundred tensors.
"""
import torch

import dion
from dion_amd import gram_newton_schulz, polar_express, zeropower_via_newtonschulz5

OPERATORS = {"ns5": zeropower_via_newtonschulz5, "polar_express": polar_express, "gram": gram_newton_schulz}
OPTIMIZERS = {"muon": dion.Muon, "normuon": dion.NorMuon, "dion2": dion.Dion2, "nordion2": dion.NorDion2}
DTYPES = {"bf16": torch.bfloat16, "fp32": torch.float32}
FRACTION = 0.25  # Dion2 / NorDion2: share of the slices that is selected
ITERATIONS = 5


def _ortho(name, batch, rows, cols, schedule, dtype):
    return {"name": name, "kind": "ortho", "batch": batch, "rows": rows, "cols": cols, "schedule": schedule,
            "dtype": dtype}


def _step(name, optimizer, schedule, layers, width, mlp, kv, *, fused=True, gated=False, heads=0, split=False,
          state="fp32", grad="bf16", nesterov=True, cautious=False, vocab=0, scalar="adamw"):
    """``kv``: rows of the key and of the value projection; ``fused``: query, key and value in one weight, which
    ``heads`` cuts into that many heads and ``split`` into its three projections; ``gated``: two up projections."""
    return {"name": name, "kind": "step", "optimizer": optimizer, "schedule": schedule, "layers": layers,
            "width": width, "mlp": mlp, "kv": kv, "fused": fused, "gated": gated, "heads": heads, "split": split,
            "state": state, "grad": grad, "nesterov": nesterov, "cautious": cautious, "vocab": vocab,
            "scalar": scalar}


def listed():
    return [
        # One matrix of a GPT-small MLP: the smallest call, a chain of dependent launches that cannot fill the chip
        # (trying the operator out, one parameter per call, the last parameters of a sharded group).
        _ortho("one_768x3072", 1, 768, 3072, "ns5", "bf16"),
        # Per-head orthogonalization of the fused attention weights of GPT-small: 12 layers of 36 heads of 64 x 768.
        _ortho("heads_432x64x768", 432, 64, 768, "polar_express", "bf16"),
        # fp32 gradients of a few weights whose sizes no tile divides (8/3 * 1000 hidden units), tall.
        _ortho("ragged_4x2730x1000", 4, 2730, 1000, "ns5", "fp32"),
        # The Gram-matrix form on the key / value projections of a 4096-wide model.
        _ortho("gram_8x1024x4096", 8, 1024, 4096, "gram", "bf16"),
        # A whole shape group of a 1.3B model in one call: GEMM-bound.
        _ortho("mlp_24x2048x8192", 24, 2048, 8192, "ns5", "bf16"),
        # A whole GPT-small step as a training script runs it, with embedding and head in an AdamW group.
        _step("muon_gpt_small", "muon", "polar_express", 12, 768, 3072, 768, vocab=50304),
        # The same model kept in bf16, with per-head attention weights.
        _step("muon_gpt_small_heads", "muon", "polar_express", 12, 768, 3072, 768, heads=36, state="bf16"),
        # A small gated model with grouped keys and values whose sizes fit no tile: a fused projection with
        # split_sizes, fp32 gradients, cautious weight decay, Lion for the rest.
        _step("muon_gated_ragged", "muon", "ns5", 6, 1000, 2730, 250, gated=True, split=True, grad="fp32",
              nesterov=False, cautious=True, vocab=32000, scalar="lion"),
        # The 1.3B model: NorMuon, and Dion2, whose step is mostly memory traffic.
        _step("normuon_gpt_1p3b", "normuon", "ns5", 24, 2048, 8192, 2048),
        _step("dion2_gpt_1p3b", "dion2", "polar_express", 24, 2048, 8192, 2048),
        # NorDion2 on the small model, bf16 state: many short launches between the orthogonalizations.
        _step("nordion2_gpt_small", "nordion2", "polar_express", 12, 768, 3072, 768, state="bf16"),
        # What one GPU of eight runs of a Llama-3-8B step: the largest matrices.
        _step("muon_llama3_8b_share8", "muon", "ns5", 4, 4096, 14336, 1024, fused=False, gated=True),
    ]


def _log_uniform(rng, lo, hi):
    return int(round(lo * (hi / lo) ** rng.random()))


def _extent(rng, lo, hi):
    """An extent as models have it: mostly a multiple of 64, now and then of 8, now and then anything."""
    v = _log_uniform(rng, lo, hi)
    grain = rng.choice((64, 64, 64, 8, 1))
    return max(grain, (v + grain // 2) // grain * grain)


def draw(rng):
    while True:
        case = _draw_ortho(rng) if rng.random() < 0.45 else _draw_step(rng)
        del case["name"]
        top = work(listed()[-1])
        w = work(case)
        if w["flops"] <= 0.8 * top["flops"] and w["bytes"] <= 0.8 * top["bytes"]:
            return case


def _draw_ortho(rng):
    schedule, dtype = rng.choice(("ns5", "polar_express", "polar_express", "gram")), rng.choice(("bf16", "bf16", "fp32"))
    if rng.random() < 0.35:  # attention heads: narrow matrices, many of them
        rows, cols, batch = rng.choice((32, 48, 64, 64, 80, 96, 128, 128)), _extent(rng, 256, 4096), _log_uniform(rng, 24, 1024)
    else:
        rows = _extent(rng, 128, 4096)
        cols = rows if rng.random() < 0.2 else max(1, int(rows * 4 ** rng.random()) // 8 * 8)
        batch = _log_uniform(rng, 1, 32)
    if rng.random() < 0.4:
        rows, cols = cols, rows
    return _ortho("", batch, rows, cols, schedule, dtype)


def _draw_step(rng):
    optimizer = rng.choice(("muon", "muon", "muon", "normuon", "dion2", "nordion2"))
    schedule = rng.choice(("polar_express", "polar_express", "ns5", "gram"))
    width, layers = _extent(rng, 256, 3072), _log_uniform(rng, 2, 24)
    gated = rng.random() < 0.5
    mlp = max(8, int(width * 8 / 3) // 2 * 2 if gated else 4 * width)
    fused = rng.random() < 0.6
    kv = max(1, width // rng.choice((1, 1, 4)))
    heads, split = 0, False
    if fused and optimizer in ("muon", "normuon") and rng.random() < 0.5:
        head = rng.choice((64, 64, 128))
        if (width + 2 * kv) % head == 0 and rng.random() < 0.6:
            heads = (width + 2 * kv) // head
        else:
            split = True
    vocab = rng.choice((0, 0, 32000, 50304))
    return _step("", optimizer, schedule, layers, width, mlp, kv, fused=fused, gated=gated, heads=heads, split=split,
                 state=rng.choice(("fp32", "fp32", "bf16")), grad=rng.choice(("bf16", "bf16", "fp32")),
                 nesterov=rng.random() < 0.5, cautious=optimizer in ("muon", "normuon") and rng.random() < 0.3,
                 vocab=vocab, scalar=rng.choice(("adamw", "adamw", "lion")))


def _weights(case):
    """[(rows, cols, count, option)] of the matrix weights of a ``step`` case, one entry per param group."""
    L, w, mlp, kv = case["layers"], case["width"], case["mlp"], case["kv"]
    if case["fused"]:
        option = {}
        if case["heads"]:
            option = {"num_heads": case["heads"]}
        elif case["split"]:
            option = {"split_sizes": (w, kv, kv)}
        out = [(w + 2 * kv, w, L, option), (w, w, L, {})]
    else:
        out = [(w, w, 2 * L, {}), (kv, w, 2 * L, {})]
    return out + [(mlp, w, (2 if case["gated"] else 1) * L, {}), (w, mlp, L, {})]


def _scalars(case):
    """[(shape, count)] of the parameters an AdamW / Lion group holds."""
    if not case["vocab"]:
        return []
    return [((case["vocab"], case["width"]), 2), ((case["width"],), 2 * case["layers"] + 1)]


def _arena(count, shape, dtype, gen, std):
    """``count`` tensors of ``shape`` in one allocation, each 256-byte aligned: (buffer, views)."""
    numel = 1
    for s in shape:
        numel *= s
    pitch = -(-numel // 128) * 128
    buf = torch.zeros(count, pitch, dtype=dtype, device="cuda")
    if std:
        # (the padding behind a tensor stays zero)
        buf[:, :numel] = torch.empty(count, numel, device="cuda").normal_(0.0, std, generator=gen)
    return buf, [buf[i, :numel].view(shape) for i in range(count)]


def _prepare_ortho(case, gen):
    G = torch.empty(case["batch"], case["rows"], case["cols"], device="cuda").normal_(0.0, 0.02, generator=gen)
    return {"operator": OPERATORS[case["schedule"]], "G": G.to(DTYPES[case["dtype"]])}


def _parameters(shape, count, case, gen, buffers):
    sdt, gdt = DTYPES[case["state"]], DTYPES[case["grad"]]
    buf, views = _arena(count, shape, sdt, gen, 0.02)
    buffers.append(buf)
    _g, grads = _arena(count, shape, gdt, gen, 0.02)
    params = []
    for x, g in zip(views, grads):
        p = torch.nn.Parameter(x)
        p.grad_dtype = None
        p.grad = g
        params.append(p)
    return params


def _prepare_step(case, gen):
    buffers, groups, owned = [], [], []
    for rows, cols, count, option in _weights(case):
        params = _parameters((rows, cols), count, case, gen, buffers)
        groups.append({"params": params, **option})
        owned.append((params, case["optimizer"]))
    scalars = []
    for shape, count in _scalars(case):
        params = _parameters(shape, count, case, gen, buffers)
        scalars += params
        owned.append((params, case["scalar"]))
    if scalars:
        groups.append({"params": scalars, "algorithm": case["scalar"], "lr": 0.001})
    kw = dict(lr=0.02, weight_decay=0.01, use_polar_express=case["schedule"] != "ns5",
              use_gram_newton_schulz=case["schedule"] == "gram")
    if case["optimizer"] in ("muon", "normuon"):
        kw.update(nesterov=case["nesterov"], cautious_wd=case["cautious"])
    else:
        kw.update(fraction=FRACTION)
    opt = OPTIMIZERS[case["optimizer"]](groups, **kw)
    # the state of a run under way
    for params, _algo in owned:
        for key, std in (("momentum", 0.05), ("variance", 4e-4), ("variance_neuron", 4e-4)):
            if key not in opt.state[params[0]]:
                continue
            old = opt.state[params[0]][key]
            buf, views = _arena(len(params), tuple(old.shape), old.dtype, gen, std)
            if key != "momentum":
                buf.abs_()
            buffers.append(buf)
            for p, v in zip(params, views):
                opt.state[p][key] = v
    return {"optimizer": opt, "buffers": buffers}


def prepare(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(int(seed))
    with torch.no_grad():
        return _prepare_ortho(case, gen) if case["kind"] == "ortho" else _prepare_step(case, gen)


def run(state):
    if "operator" in state:
        return state["operator"](state["G"])
    state["optimizer"].step()
    return state["buffers"]


def _ortho_flops(rows, cols, gram):
    """Products one orthogonalization cannot do without, half of each symmetric one."""
    m, n = float(min(rows, cols)), float(max(rows, cols))
    standard = ITERATIONS * (3 * m * m * n + m ** 3)
    if gram and n >= 3 * m:
        # two Gram matrices and two applications of an m x m matrix; per iteration R R, and between restarts T = Z R,
        # R = T Z and Q = Z Q
        return min(standard, 6 * m * m * n + 20 * m ** 3)
    return standard


def work(case):
    gram = case["schedule"] == "gram"
    if case["kind"] == "ortho":
        n = case["batch"] * case["rows"] * case["cols"]
        return {"bytes": float(n * ((2 if case["dtype"] == "bf16" else 4) + 2)),
                "flops": case["batch"] * _ortho_flops(case["rows"], case["cols"], gram)}
    s, g = (2 if case[k] == "bf16" else 4 for k in ("state", "grad"))
    nbytes = flops = 0.0
    for rows, cols, count, option in _weights(case):
        nbytes += count * rows * cols * (4 * s + g)  # parameter and momentum read and written, gradient read
        if option.get("num_heads"):
            parts = [(rows // option["num_heads"], cols)] * option["num_heads"]
        elif option.get("split_sizes"):
            parts = [(r, cols) for r in option["split_sizes"]]
        elif case["optimizer"] == "nordion2" or (case["optimizer"] == "dion2" and rows <= cols):
            parts = [(max(1, -int(-FRACTION * rows // 1)), cols)]
        elif case["optimizer"] == "dion2":
            parts = [(rows, max(1, -int(-FRACTION * cols // 1)))]
        else:
            parts = [(rows, cols)]
        flops += count * sum(_ortho_flops(r, c, gram) for r, c in parts)
    for shape, count in _scalars(case):
        numel = shape[0] * (shape[1] if len(shape) == 2 else 1)
        nbytes += count * numel * ((6 if case["scalar"] == "adamw" else 4) * s + g)
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    """About four times the distance to the same path with the orthogonalization in float64, measured on the listed
    and on drawn cases (largest seen).  Operators: ns5 5.0e-3 (largest element 2.6e-2 of the root mean square),
    Polar-Express 1.4e-2 (0.16) and Gram 1.9e-2 (0.17), whose steeper polynomials carry bf16 rounding further.
    Parameters after two steps: fp32 5.1e-4 (6.3e-3), bf16 2.7e-3 (1.6e-2: two units in the last place)."""
    if case["kind"] == "ortho":
        return {"rel": 0.02, "max": 0.11} if case["schedule"] == "ns5" else {"rel": 0.03, "max": 0.7}
    return {"rel": 2e-3, "max": 2.5e-2} if case["state"] == "fp32" else {"rel": 1e-2, "max": 6.4e-2}
