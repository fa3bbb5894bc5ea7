"""The work users of this framework have it do, as measurable cases.

Every case goes through the public surface (`rg.compile`, `rg.run`, a compiled program's call,
`nn`, `optim`, `random`, `workloads`). Tensors of this framework live in host memory between
calls, so a case's pass is a whole call: its inputs go to the device, the step loop (or the
program) runs there, and what it returns comes back. Training runs take as many steps as put the
device's work well above the transfers, as a training program does.

Kinds of work (a case's `kind`):
- linreg: full-batch gradient descent on a linear model, hundreds of tiny steps in one run; the
  smallest calls, bound by launches and latency.
- mlp: AdamW training of a three-layer GELU MLP on cycled batches; float32, or float64 as used
  where gradients are checked or curvature is computed.
- gpt: AdamW training of the character-level GPT (forward, backward, update) on cycled batches.
- attention: SGD on one self-attention layer and its input, past the context of the GPT cases.
- head: SGD on a final layer norm, a vocabulary projection and its input under cross-entropy.
- chain: SGD on the two inner matrices of a skinny matrix chain, written in the expensive order.
- logits: one serving call, token ids in, logits out, the weights constants of the program.
- generate: autoregressive sampling, one device step per token.

Training resumes from the state of a run under way (moments and step count set, biases away from
zero), which is what most steps of a run meet; the first moments of a fresh run would divide
rounding noise by itself wherever a gradient is exactly zero.
"""

import math

import numpy as np
import torch

import rustautograd_amd as rg
from rustautograd_amd import nn, optim, random, workloads

_LR, _DECAY, _B1, _B2, _EPS = 3e-4, 0.01, 0.9, 0.999, 1e-8
_COUNT = 1000.0     # optimizer steps behind the resumed state
_TEMPERATURE, _TOP_K = 0.8, 20


def listed():
    return [
        # The README's example: 500 steps of gradient descent on 256 x 8 in one run.
        {"name": "linreg 256x8", "kind": "linreg", "n": 256, "d": 8, "steps": 500},
        # The benchmark's MLP at its own sizes.
        {"name": "mlp 4096x512x2048", "kind": "mlp", "batch": 4096, "d_in": 512, "hidden": 2048, "dtype": "float32", "steps": 96},
        # Tabular regression: features and widths that no tile divides, a ragged batch.
        {"name": "mlp ragged 1000x77x500", "kind": "mlp", "batch": 1000, "d_in": 77, "hidden": 500, "dtype": "float32", "steps": 48},
        # The same model in double precision.
        {"name": "mlp f64 1024x128x512", "kind": "mlp", "batch": 1024, "d_in": 128, "hidden": 512, "dtype": "float64", "steps": 32},
        # The benchmark's small GPT (tied embeddings).
        {"name": "gpt d128 L4 T128", "kind": "gpt", "vocab": 96, "block": 128, "d": 128, "heads": 4, "layers": 4, "batch": 32, "tied": True,
         "steps": 60},
        # The headline: the benchmark's GPT.
        {"name": "gpt d256 L6 T256", "kind": "gpt", "vocab": 96, "block": 256, "d": 256, "heads": 8, "layers": 6, "batch": 32, "tied": False,
         "steps": 120},
        # A user's own GPT: a vocabulary and a context that divide by nothing.
        {"name": "gpt ragged d192 L3 T200", "kind": "gpt", "vocab": 101, "block": 200, "d": 192, "heads": 6, "layers": 3, "batch": 16,
         "tied": False, "steps": 32},
        # One attention layer at a longer context and a wider head.
        {"name": "attention T512 d512", "kind": "attention", "batch": 8, "block": 512, "d": 512, "heads": 8, "steps": 48},
        # The output layer of a language model with a word-piece vocabulary.
        {"name": "head 4096x256 V5000", "kind": "head", "rows": 4096, "d": 256, "vocab": 5000, "steps": 48},
        # The benchmark's matrix chain, its gradients applied.
        {"name": "chain 4096 k8", "kind": "chain", "n": 4096, "k": 8, "steps": 1000},
        # Scoring a few sequences with a trained GPT.
        {"name": "logits 8x256", "kind": "logits", "vocab": 96, "block": 256, "d": 256, "heads": 8, "layers": 6, "batch": 8, "length": 256},
        # Writing 64 characters with it.
        {"name": "generate 64 tokens", "kind": "generate", "vocab": 96, "block": 256, "d": 256, "heads": 8, "layers": 6, "tokens": 64},
    ]


def _log_int(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    kind = rng.choice(["linreg", "mlp", "mlp", "gpt", "gpt", "attention", "head", "chain", "logits", "generate"])
    if kind == "linreg":
        return {"kind": kind, "n": _log_int(rng, 64, 4096), "d": _log_int(rng, 3, 64), "steps": rng.randint(200, 500)}
    if kind == "mlp":
        dtype = rng.choice(["float32", "float32", "float64"])
        most = 4096 if dtype == "float32" else 1024
        hidden = _log_int(rng, 64, 1500 if dtype == "float32" else 512)
        return {"kind": kind, "batch": _log_int(rng, 100, most), "d_in": _log_int(rng, 16, 512), "hidden": hidden, "dtype": dtype,
                "steps": rng.randint(24, 48)}
    if kind == "chain":
        return {"kind": kind, "n": rng.choice([64 * rng.randint(8, 48), _log_int(rng, 500, 2500)]), "k": rng.randint(1, 16), "steps": rng.randint(50, 200)}
    if kind == "head":
        return {"kind": kind, "rows": _log_int(rng, 256, 4096), "d": 8 * rng.randint(8, 40), "vocab": _log_int(rng, 80, 5000),
                "steps": rng.randint(16, 48)}
    hd = rng.choice([16, 24, 32, 32, 64])
    if kind == "attention":
        return {"kind": kind, "batch": rng.randint(1, 8), "block": _log_int(rng, 48, 512), "d": 8 * hd if hd < 64 else 256,
                "heads": 8 if hd < 64 else 4, "steps": rng.randint(16, 48)}
    heads = rng.choice([2, 4, 6, 8] if hd <= 32 else [2, 3, 4])
    block = rng.choice([32 * rng.randint(1, 8), rng.randint(30, 256)])
    case = {"kind": kind, "vocab": rng.randint(65, 130), "block": block, "d": heads * hd, "heads": heads, "layers": rng.randint(1, 4)}
    if kind == "gpt":
        case.update(batch=rng.randint(4, 32), tied=rng.random() < 0.3, steps=rng.randint(16, 40))
    elif kind == "logits":
        case.update(batch=rng.randint(1, 16), length=rng.randint(max(8, block // 2), block))
    else:
        case.update(tokens=rng.randint(16, 64))
    return case


# ---- inputs and states ------------------------------------------------------------------------

def _normal(gen, shape, std, dtype=np.float32):
    return (gen.standard_normal(shape, dtype=np.float32) * np.float32(std)).astype(dtype)


def _dense(gen, d_in, d_out, bias=True, dtype=np.float32):
    """A trained layer's weights: fan-in scaled, biases near but not at zero."""
    w = {"w": _normal(gen, (d_in, d_out), 1.0 / math.sqrt(d_in), dtype)}
    if bias:
        w["b"] = _normal(gen, (d_out,), 0.05, dtype)
    return w


def _norm(gen, d):
    return {"scale": 1.0 + _normal(gen, (d,), 0.1), "shift": _normal(gen, (d,), 0.05)}


def _gpt_params(gen, c):
    d = c["d"]
    params = {"tok": {"table": _normal(gen, (c["vocab"], d), 0.3)}, "pos": {"table": _normal(gen, (c["block"], d), 0.1)}, "norm": _norm(gen, d),
              "blocks": [{"norm1": _norm(gen, d), "attn": {"qkv": _dense(gen, d, 3 * d), "out": _dense(gen, d, d)}, "norm2": _norm(gen, d),
                          "fc1": _dense(gen, d, 4 * d), "fc2": _dense(gen, 4 * d, d)} for _ in range(c["layers"])]}
    if not c.get("tied"):
        params["head"] = _dense(gen, d, c["vocab"], bias=False)
    return params


def _map(f, tree):
    if isinstance(tree, dict):
        return {k: _map(f, v) for k, v in tree.items()}
    if isinstance(tree, (list, tuple)):
        return [_map(f, v) for v in tree]
    return f(tree)


def _leaves(tree, path=""):
    """(path, leaf) in a fixed order."""
    if isinstance(tree, dict):
        return [x for k in sorted(tree) for x in _leaves(tree[k], f"{path}.{k}")]
    if isinstance(tree, (list, tuple)):
        return [x for i, v in enumerate(tree) for x in _leaves(v, f"{path}.{i}")]
    return [(path.lstrip("."), tree)]


def _adamw_state(gen, params, size):
    """Parameters with the optimizer state of a run whose gradients had about `size`, as numpy
    arrays."""
    dtype = _leaves(params)[0][1].dtype
    mu = _map(lambda p: _normal(gen, p.shape, 0.3 * size, dtype), params)
    nu = _map(lambda p: ((0.5 + gen.random(p.shape, dtype=np.float32)) * np.float32(size * size)).astype(dtype), params)
    return {"params": params, "opt": {"count": np.array(_COUNT, dtype), "mu": mu, "nu": nu}}


def _sgd(params, grads, lr):
    return rg.tree.map(lambda p, g: p - lr * g, params, grads)


# ---- the programs a user would write ------------------------------------------------------------

def _mlp_model(c):
    d, h, t = c["d_in"], c["hidden"], c["dtype"]
    return nn.Sequential(nn.Linear(d, h, dtype=t), nn.gelu, nn.Linear(h, h, dtype=t), nn.gelu, nn.Linear(h, 1, dtype=t))


def _adamw_step(loss):
    opt = optim.adamw(_LR, weight_decay=_DECAY)

    def step(state, data):
        value, grads = rg.value_and_grad(loss)(state["params"], *data)
        params, o = opt.update(grads, state["opt"], state["params"])
        return {"params": params, "opt": o}, value

    return step


def _sgd_step(loss, lr):
    def step(state, data):
        value, grads = rg.value_and_grad(loss)(state, *data)
        return _sgd(state, grads, lr), value

    return step


def _gpt_model(c):
    return workloads.GPT(c["vocab"], c["block"], c["d"], c["heads"], c["layers"], c.get("tied", False))


def _program(c):
    """The step a training case runs."""
    kind = c["kind"]
    if kind == "linreg":
        return _sgd_step(lambda w, x, y: nn.mse_loss(x @ w, y), 0.05)
    if kind == "mlp":
        model = _mlp_model(c)
        return _adamw_step(lambda p, x, t: nn.mse_loss(model(p, x), t))
    if kind == "gpt":
        model = _gpt_model(c)
        return _adamw_step(lambda p, x, y: nn.cross_entropy(model(p, x), y))
    if kind == "attention":
        layer, mask = nn.MultiHeadAttention(c["d"], c["heads"]), rg.tril(c["block"])
        return _sgd_step(lambda s, t: nn.mse_loss(s["x"] + layer(s["attn"], s["x"], mask), t), 0.5)
    if kind == "head":
        norm, head = nn.LayerNorm(c["d"]), nn.Linear(c["d"], c["vocab"])
        return _sgd_step(lambda s, y: nn.cross_entropy(head(s["head"], norm(s["norm"], s["x"])), y), 0.5)
    if kind == "chain":
        return _sgd_step(lambda s, a, d: (((a @ s["b"]) @ s["c"]) @ d).sum(), 0.001)
    raise ValueError(kind)


def _inputs(c, seed):
    """(state, batches) of a training case as numpy arrays, from the seed alone."""
    gen, kind = np.random.default_rng(seed), c["kind"]
    if kind == "linreg":
        x = _normal(gen, (c["n"], c["d"]), 1.0)
        return np.zeros(c["d"], np.float32), [(x, x @ np.arange(c["d"], dtype=np.float32))]
    if kind == "mlp":
        t = np.dtype(c["dtype"])
        params = {"0": _dense(gen, c["d_in"], c["hidden"], dtype=t), "2": _dense(gen, c["hidden"], c["hidden"], dtype=t),
                  "4": _dense(gen, c["hidden"], 1, dtype=t)}
        batches = []
        for _ in range(2):
            x = _normal(gen, (c["batch"], c["d_in"]), 1.0, t)
            batches.append((x, np.sin(x[:, :16]).sum(axis=1, keepdims=True).astype(t)))
        return _adamw_state(gen, params, 0.3), batches
    if kind == "gpt":
        state, batches = _adamw_state(gen, _gpt_params(gen, c), 2e-2), []
        for _ in range(2):
            ids = gen.integers(0, c["vocab"], (c["batch"], c["block"] + 1), dtype=np.int32)
            batches.append((np.ascontiguousarray(ids[:, :-1]), np.ascontiguousarray(ids[:, 1:])))
        return state, batches
    if kind == "attention":
        d, shape = c["d"], (c["batch"], c["block"], c["d"])
        return {"attn": {"qkv": _dense(gen, d, 3 * d), "out": _dense(gen, d, d)}, "x": _normal(gen, shape, 1.0)}, [(_normal(gen, shape, 1.0),)]
    if kind == "head":
        state = {"norm": _norm(gen, c["d"]), "head": _dense(gen, c["d"], c["vocab"]), "x": _normal(gen, (c["rows"], c["d"]), 1.0)}
        return state, [(gen.integers(0, c["vocab"], c["rows"], dtype=np.int32),)]
    n, k, sigma = c["n"], c["k"], 1.0 / math.sqrt(c["n"])
    a, b, m, d = (_normal(gen, s, sigma) for s in ((k, n), (n, n), (n, n), (n, k)))
    return {"b": b, "c": m}, [(a, d)]


def _tensors(tree):
    return _map(rg.tensor, tree)


def _sample_program(c, params):
    """One token of `workloads.Sampler`'s kind, the filtered logits it drew from beside it."""
    model = _gpt_model(c)

    def advance(state):
        carried, for_draw = random.split(state["key"])
        logits = model(params, state["ctx"])[:, -1, :] / _TEMPERATURE
        picked = random.categorical(for_draw, nn.top_k_logits(logits, _TOP_K))
        shifted = rg.concatenate([state["ctx"][:, 1:], picked.reshape(1, 1)], axis=1)
        return {"ctx": shifted, "key": carried}, (picked[0], logits)

    return advance


def _prompt(c, seed):
    gen = np.random.default_rng([seed, 1])
    return [int(t) for t in gen.integers(0, c["vocab"], c["block"])]


def _request(c, seed):
    return np.random.default_rng([seed, 1]).integers(0, c["vocab"], (c["batch"], c["length"]), dtype=np.int32)


def prepare(case, seed):
    c = case
    if c["kind"] == "logits":
        model, params, ids = _gpt_model(c), _tensors(_gpt_params(np.random.default_rng(seed), c)), rg.tensor(_request(c, seed))
        return {"case": c, "compiled": rg.compile(lambda idx: model(params, idx), (ids,), validate="basic"), "ids": ids}
    if c["kind"] == "generate":
        params = _tensors(_gpt_params(np.random.default_rng(seed), c))
        state = workloads.prompt_state(_prompt(c, seed), c["block"], seed)
        return {"case": c, "compiled": rg.compile(_sample_program(c, params), (state,), validate="basic"), "state": state}
    state, batches = _inputs(c, seed)
    state, batches = _tensors(state), [tuple(rg.tensor(x) for x in b) for b in batches]
    return {"case": c, "compiled": rg.compile(_program(c), (state, batches[0]), validate="basic"), "state": state, "batches": batches}


def _returned(tree):
    """The arrays of a state: matrices one by one; vectors joined, and all second moments joined,
    to keep their number small."""
    out, vectors, second = {}, [], []
    for path, leaf in _leaves(tree):
        if path.startswith("opt.nu"):
            second.append(leaf.reshape(-1))
        elif path.startswith(("params", "opt.mu")) and leaf.ndim < 2:
            vectors.append(leaf.reshape(-1))
        else:
            out[path] = leaf
    join = torch.cat if any(isinstance(v, torch.Tensor) for v in vectors + second) else np.concatenate
    if vectors:
        out["vectors"] = join(vectors)
    if second:
        out["second"] = join(second)
    return out


def run(state):
    c = state["case"]
    if c["kind"] == "logits":
        return {"logits": state["compiled"](state["ids"]).numpy()}
    if c["kind"] == "generate":
        r = rg.run(state["compiled"], state["state"], steps=c["tokens"])
        return {"tokens": np.array(r.history["aux.0"], np.int32), "logits": r.aux[1].numpy()}
    r = rg.run(state["compiled"], state["state"], state["batches"], steps=c["steps"])
    return {"loss": np.array(r.history["aux"]), **_returned(_map(lambda t: t.numpy(), r.state))}


# ---- what a pass cannot do without ----------------------------------------------------------------

def _gpt_flops(c, rows, length, grad):
    """Products of one pass over `rows` sequences of `length` tokens; attention's two per layer
    count the causal half."""
    d, tokens = c["d"], rows * length
    forward = c["layers"] * (tokens * 12 * d * d + tokens * (length + 1) * d) + tokens * d * c["vocab"]
    return 2.0 * forward * (3 if grad else 1)


def _gpt_size(c):
    d = c["d"]
    return c["vocab"] * d * (1 if c.get("tied") else 2) + c["block"] * d + 2 * d + c["layers"] * (12 * d * d + 13 * d)


def work(case):
    c = case
    kind, steps = c["kind"], c.get("steps", 1)
    if kind == "linreg":
        n, d = c["n"], c["d"]
        return {"bytes": steps * 4.0 * (n * d + n + 2 * d), "flops": steps * 4.0 * n * d}
    if kind == "mlp":
        b, d, h, item = c["batch"], c["d_in"], c["hidden"], 8 if c["dtype"] == "float64" else 4
        size = d * h + h * h + 3 * h + 1
        flops = 2.0 * b * (2 * d * h + 3 * h * h + 3 * h)
        return {"bytes": steps * item * (6.0 * size + b * (d + 1)), "flops": steps * flops}
    if kind == "gpt":
        return {"bytes": steps * (24.0 * _gpt_size(c) + 8.0 * c["batch"] * c["block"]),
                "flops": steps * _gpt_flops(c, c["batch"], c["block"], True)}
    if kind == "attention":
        b, t, d = c["batch"], c["block"], c["d"]
        return {"bytes": steps * 4.0 * (3 * b * t * d + 8 * d * d), "flops": steps * 6.0 * b * t * (4 * d * d + (t + 1) * d)}
    if kind == "head":
        n, d, v = c["rows"], c["d"], c["vocab"]
        return {"bytes": steps * 4.0 * (2 * n * d + 2 * d * v + n), "flops": steps * 6.0 * n * d * v}
    if kind == "chain":
        n, k = c["n"], c["k"]
        return {"bytes": steps * 4.0 * (4 * n * n + 2 * n * k), "flops": steps * 10.0 * n * n * k}
    if kind == "logits":
        return {"bytes": 4.0 * (_gpt_size(c) + c["batch"] * c["length"] * (1 + c["vocab"])), "flops": _gpt_flops(c, c["batch"], c["length"], False)}
    # A model that fixes the context's positions anew for every token scores the whole context.
    return {"bytes": c["tokens"] * 4.0 * _gpt_size(c), "flops": c["tokens"] * _gpt_flops(c, 1, c["block"], False)}


# ---- how far a correct implementation may be ------------------------------------------------------

# About four times the largest relative error against `exact` over the listed and some 50 drawn cases
# on an MI355X with float32 sums (gpt 7e-6, mlp 2e-6, attention 1e-6, the others 4e-7 to 8e-7, float64
# 6e-16); "max" is 40 times as much.
_TOLERANCE = {"linreg": 2e-6, "mlp": 1e-5, "gpt": 3e-5, "attention": 5e-6, "head": 3e-6, "chain": 4e-6, "logits": 4e-6, "generate": 4e-6}


def tolerance(case):
    if case.get("dtype") == "float64":
        return {"rel": 1e-14}
    if case["kind"] == "generate":
        # A token drawn between two equally likely ones may fall either way.
        return {"rel": _TOLERANCE["generate"], "differ": 0.01}
    return {"rel": _TOLERANCE[case["kind"]]}


# ---- the same in 64 bits, in plain torch ------------------------------------------------------------

_DEVICE = "cuda" if torch.cuda.is_available() else "cpu"


def _wide(x):
    x = torch.from_numpy(np.ascontiguousarray(x)).to(_DEVICE)
    return x.double() if x.is_floating_point() else x.long()


def _t_dense(p, x):
    y = x @ p["w"]
    return y + p["b"] if "b" in p else y


def _t_gelu(x):
    return torch.nn.functional.gelu(x, approximate="tanh")


def _t_norm(p, x):
    return torch.nn.functional.layer_norm(x, (x.shape[-1],), p["scale"], p["shift"], 1e-5)


def _t_attention(p, x, heads):
    b, t, d = x.shape
    q, k, v = _t_dense(p["qkv"], x).reshape(b, t, 3, heads, d // heads).permute(2, 0, 3, 1, 4).contiguous()
    scores = q @ k.transpose(-1, -2).contiguous() / math.sqrt(d // heads)
    hidden = torch.ones(t, t, dtype=torch.bool, device=x.device).triu(1)
    weights = torch.softmax(scores.masked_fill(hidden, -1e9), -1)
    return _t_dense(p["out"], (weights @ v).permute(0, 2, 1, 3).reshape(b, t, d))


def _t_gpt(c, p, ids):
    h = p["tok"]["table"][ids] + p["pos"]["table"][: ids.shape[1]]
    for q in p["blocks"]:
        h = h + _t_attention(q["attn"], _t_norm(q["norm1"], h), c["heads"])
        h = h + _t_dense(q["fc2"], _t_gelu(_t_dense(q["fc1"], _t_norm(q["norm2"], h))))
    h = _t_norm(p["norm"], h)
    return h @ p["tok"]["table"].T if c.get("tied") else _t_dense(p["head"], h)


def _t_loss(c, s, data):
    kind, f = c["kind"], torch.nn.functional
    if kind == "linreg":
        return ((data[0] @ s - data[1]) ** 2).mean()
    if kind == "mlp":
        hidden = _t_gelu(_t_dense(s["2"], _t_gelu(_t_dense(s["0"], data[0]))))
        return ((_t_dense(s["4"], hidden) - data[1]) ** 2).mean()
    if kind == "gpt":
        return f.cross_entropy(_t_gpt(c, s, data[0]).reshape(-1, c["vocab"]), data[1].reshape(-1))
    if kind == "attention":
        return ((s["x"] + _t_attention(s["attn"], s["x"], c["heads"]) - data[0]) ** 2).mean()
    if kind == "head":
        return f.cross_entropy(_t_dense(s["head"], _t_norm(s["norm"], s["x"])), data[0])
    return ((data[0] @ s["b"]) @ (s["c"] @ data[1])).sum()


def _train_exact(c, seed):
    state, batches = _inputs(c, seed)
    state, batches = _map(_wide, state), [tuple(_wide(x) for x in b) for b in batches]
    adamw = c["kind"] in ("mlp", "gpt")
    params = state["params"] if adamw else state
    lr = {"linreg": 0.05, "attention": 0.5, "head": 0.5, "chain": 0.001}.get(c["kind"])
    names = [n for n, _ in _leaves(params)]
    at = dict(_leaves(params))
    if adamw:
        count, mu, nu = _COUNT, dict(_leaves(state["opt"]["mu"])), dict(_leaves(state["opt"]["nu"]))
    losses = []
    for i in range(c["steps"]):
        for n in names:
            at[n] = at[n].detach().requires_grad_(True)
        value = _t_loss(c, _rebuild(params, at), batches[i % len(batches)])
        grads = torch.autograd.grad(value, [at[n] for n in names])
        losses.append(value.item())
        with torch.no_grad():
            if adamw:
                count += 1.0
                for n, g in zip(names, grads):
                    mu[n] = _B1 * mu[n] + (1.0 - _B1) * g
                    nu[n] = _B2 * nu[n] + (1.0 - _B2) * (g * g)
                    direction = (mu[n] / (1.0 - _B1 ** count)) / ((nu[n] / (1.0 - _B2 ** count)).sqrt() + _EPS)
                    if at[n].ndim > 1:
                        direction = direction + _DECAY * at[n]
                    at[n] = at[n] - _LR * direction
            else:
                for n, g in zip(names, grads):
                    at[n] = at[n] - lr * g
    new = _rebuild(params, at)
    if adamw:
        new = {"params": new, "opt": {"count": torch.tensor(count, dtype=torch.float64, device=_DEVICE), "mu": _rebuild(params, mu),
                                      "nu": _rebuild(params, nu)}}
    return {"loss": np.array(losses), **_returned(_map(lambda t: t.detach(), new))}


def _rebuild(tree, leaves, path=""):
    if isinstance(tree, dict):
        return {k: _rebuild(v, leaves, f"{path}.{k}") for k, v in tree.items()}
    if isinstance(tree, (list, tuple)):
        return [_rebuild(v, leaves, f"{path}.{i}") for i, v in enumerate(tree)]
    return leaves[path.lstrip(".")]


_MASK64 = (1 << 64) - 1


def _mix(z):
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9 & _MASK64
    z = (z ^ (z >> 27)) * 0x94D049BB133111EB & _MASK64
    return z ^ (z >> 31)


def _generate_exact(c, seed):
    """The published SplitMix64 streams drive the draws: key * gamma for a seed, one stream to
    split a key, one for uniform values of 24 bits."""
    params = _map(_wide, _gpt_params(np.random.default_rng(seed), c))
    context, key, logits = _prompt(c, seed), seed * 0x9E3779B97F4A7C15 & _MASK64, None
    for _ in range(c["tokens"]):
        carried, for_draw = (_mix(key + (j + 1) * 0xD1B54A32D192ED03 & _MASK64) for j in range(2))
        logits = _t_gpt(c, params, torch.tensor([context], device=_DEVICE))[0, -1] / _TEMPERATURE
        u = [(_mix(for_draw + (j + 1) * 0x9E3779B97F4A7C15 & _MASK64) >> 40) * 0.5 ** 24 for j in range(c["vocab"])]
        noise = torch.tensor([-math.log(-math.log(max(x, 1e-7))) for x in u], dtype=torch.float64, device=_DEVICE)
        kept = torch.where(logits >= logits.topk(_TOP_K).values[-1], logits, torch.full_like(logits, -1e9))
        context, key = context[1:] + [int((kept + noise).argmax())], carried
    return {"tokens": None, "logits": logits[None]}


@torch.no_grad()
def _logits_exact(c, seed):
    params = _map(_wide, _gpt_params(np.random.default_rng(seed), c))
    return {"logits": _t_gpt(c, params, _wide(_request(c, seed)))}


def exact(case, seed):
    if case["kind"] == "logits":
        return _logits_exact(case, seed)
    if case["kind"] == "generate":
        with torch.no_grad():
            return _generate_exact(case, seed)
    return _train_exact(case, seed)
