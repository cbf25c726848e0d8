"""What this framework's speed is judged on: calls through its public entry points
(``MorphoAttention``, ``SoftMorphAttention``, ``MultiHeadSelfAttention``), from the
smallest ones, where launches count, to the widest and longest configurations.

A case is a dict of plain values:

* ``kind``: ``attention`` (``MorphoAttention``), ``layer`` (``MultiHeadSelfAttention``
  under fp16 autocast, fp32 activations, as the image-classification harness of the
  reference trains it) or ``soft`` (``SoftMorphAttention``);
* ``train``: forward and backward with every gradient, else the forward under ``no_grad``;
* ``batch``, ``tokens``, ``heads``, ``cube`` (codes per head), ``head_dim`` (value columns
  per head), ``scale``, ``causal`` and the options of the modules.

Every tensor of the attention itself is float16, the only type that the entry points take.
"""

from __future__ import annotations

import math

import torch

DEVICE = "cuda"


def _case(name, kind, train, batch, tokens, heads, cube, head_dim, scale, causal, projection="sigmoid",
          mask_diag=False, deterministic=False, erosion=False, tau=0.5):
    c = {"kind": kind, "train": train, "batch": batch, "tokens": tokens, "heads": heads, "cube": cube,
         "head_dim": head_dim, "scale": scale, "causal": causal, "projection": projection, "mask_diag": mask_diag,
         "deterministic": deterministic, "erosion": erosion, "tau": tau}
    if name:
        c["name"] = name
    return c


def listed():
    return [
        # one short sequence through a small module: host time, launches and allocations
        _case("tiny_infer", "attention", False, 1, 100, 8, 16, 32, 1.0, False),
        # the smallest configuration of the tests, as a training step
        _case("tiny_train", "attention", True, 2, 128, 8, 16, 32, 1.0, False),
        # a small model's training step: about one round of workgroups in every kernel
        _case("short_train", "attention", True, 8, 1024, 8, 16, 64, 1.0, False),
        # a prompt of one user, of a length that nothing divides: the forward alone
        _case("prompt_infer", "attention", False, 1, 3001, 16, 16, 64, 1.0, True),
        # the headline training step
        _case("base_train", "attention", True, 4, 4096, 16, 16, 64, 1.0, True),
        # a long context on few sequences
        _case("long_train", "attention", True, 1, 16384, 16, 32, 64, 0.5, True),
        # the widest model: the most codes, heads and tokens
        _case("wide_train", "attention", True, 16, 2048, 32, 64, 64, 0.125, False),
        # the image classifier's layer: 14 x 14 patches and a class token, many images
        _case("image_train", "layer", True, 64, 197, 12, 64, 64, 0.125, False),
        # wide heads, a length off every tile edge
        _case("headwide_train", "attention", True, 3, 1500, 8, 32, 128, 0.5, True),
        # the soft max-plus aggregation at the headline size
        _case("soft_train", "soft", True, 4, 4096, 16, 16, 64, 1.0, True),
        # the soft min-plus aggregation at a small, ragged size
        _case("soft_erosion", "soft", True, 2, 1001, 8, 32, 64, 0.5, False, erosion=True, tau=1.0),
        # reproducible gradients with the other cube projection and the masked diagonal
        _case("variant_train", "attention", True, 4, 2000, 8, 16, 64, 1.0, False, projection="hardtanh01",
              mask_diag=True, deterministic=True),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["attention", "attention", "attention", "layer", "soft"])
    train = rng.random() < 0.7
    cube = rng.choice([16, 32, 64])
    head_dim = rng.choice([32, 64, 64, 128])
    heads = rng.choice([1, 2, 3, 4, 6, 8, 12, 16, 24, 32])
    while heads * head_dim > 2048:
        heads = heads // 2
    batch = _log_int(rng, 1, 64)
    tokens = _log_int(rng, 64, 16384)
    if rng.random() < 0.3:
        tokens -= tokens % 64
    causal = kind != "layer" and rng.random() < 0.5
    scale = cube ** -0.5 if kind == "layer" or rng.random() < 0.5 else rng.choice([0.25, 0.5, 1.0]) * 16 / cube
    projection, mask_diag, deterministic, erosion, tau = "sigmoid", False, False, False, 0.5
    if kind == "attention":
        if rng.random() < 0.2:
            projection = "hardtanh01"
        mask_diag = rng.random() < 0.1
        deterministic = train and rng.random() < 0.2
    elif kind == "soft":
        erosion = rng.random() < 0.5
        tau = rng.choice([0.5, 1.0, 2.0])
    c = _case(None, kind, train, batch, tokens, heads, cube, head_dim, scale, causal, projection, mask_diag,
              deterministic, erosion, tau)
    most = _flops(next(x for x in listed() if x["name"] == "soft_train")) if kind == "soft" else \
        _flops(next(x for x in listed() if x["name"] == "long_train"))
    # no more work than the listed cases of the kind, and no more values than the widest one
    while _flops(c) > most or c["batch"] * c["tokens"] * c["heads"] * (c["cube"] + c["head_dim"]) > 1 << 27:
        if c["batch"] > 1:
            c["batch"] = max(1, c["batch"] * 2 // 3)
        else:
            c["tokens"] = c["tokens"] * 3 // 4
    return c


def _flops(c):
    """Matrix work: one projection, scores and one value product forward; five products of the
    pairs and two of the projection backward. The layer adds its output projection."""
    B, N, H, m, dv = c["batch"], c["tokens"], c["heads"], c["cube"], c["head_dim"]
    T, D = B * N, H * dv
    pairs = B * H * (N * (N + 1) // 2 if c["causal"] else N * N)
    proj = 2.0 * T * D * (H * m + D)
    f = proj + 2.0 * pairs * (m + dv)
    if c["train"]:
        f += 2.0 * proj + 2.0 * pairs * (3 * m + 2 * dv)
    if c["kind"] == "layer":
        f += 2.0 * T * D * D * (3 if c["train"] else 1)
    return f


def work(case):
    B, N, H, m, dv = case["batch"], case["tokens"], case["heads"], case["cube"], case["head_dim"]
    D = H * dv
    act = 4 if case["kind"] == "layer" else 2            # bytes of one activation value
    x = B * N * D * act
    weights = (D * H * m + D * D + 2 * H * m) * 2
    if case["kind"] == "layer":
        weights += (D * D + D) * 4
    nbytes = x + weights + x
    if case["train"]:
        nbytes += x + x + weights                        # the output's gradient in, every gradient out
    return {"bytes": nbytes, "flops": _flops(case)}


def _gen(seed):
    return torch.Generator(device=DEVICE).manual_seed(seed)


def _tensors(case, seed):
    """x, the output's gradient and the parameters, from the seed alone. Weights as the modules
    initialise them, gates as training leaves them: around 1."""
    B, N, H, m, dv = case["batch"], case["tokens"], case["heads"], case["cube"], case["head_dim"]
    D = H * dv
    g = _gen(seed)

    def randn(*shape):
        return torch.randn(*shape, generator=g, device=DEVICE)

    t = {"x": randn(B, N, D).half(), "dout": randn(B, N, D).half(),
         "W_phi": (randn(D, H * m) * D ** -0.5).half(), "W_V": (randn(D, D) * D ** -0.5).half(),
         "gate_q": (1.0 + 0.1 * randn(H, m)).half(), "gate_k": (1.0 + 0.1 * randn(H, m)).half()}
    if case["kind"] == "layer":
        t["weight"] = randn(D, D) * D ** -0.5
        t["bias"] = 0.02 * randn(D)
    return t


PARAMS = ("W_phi", "gate_q", "gate_k", "W_V")


def prepare(case, seed):
    from morphottention_amd import MorphoAttention, SoftMorphAttention
    from morphottention_amd.layers import MultiHeadSelfAttention

    H, m, D = case["heads"], case["cube"], case["heads"] * case["head_dim"]
    t = _tensors(case, seed)
    if case["kind"] == "layer":
        module = MultiHeadSelfAttention(D, H, cube_m=m, scale=case["scale"], causal=case["causal"]).to(DEVICE)
        core = module.attn
    elif case["kind"] == "soft":
        module = core = SoftMorphAttention(D, H, m, scale=case["scale"], causal=case["causal"], tau=case["tau"],
                                           erosion=case["erosion"], projection=case["projection"],
                                           mask_diag=case["mask_diag"], device=DEVICE)
    else:
        module = core = MorphoAttention(D, H, m, scale=case["scale"], causal=case["causal"],
                                        projection=case["projection"], mask_diag=case["mask_diag"],
                                        deterministic=case["deterministic"], device=DEVICE)
    x, dout = t["x"], t["dout"]
    with torch.no_grad():
        for name in PARAMS:
            getattr(core, name).copy_(t[name])
        if case["kind"] == "layer":
            module.proj.weight.copy_(t["weight"])
            module.proj.bias.copy_(t["bias"])
            x, dout = x.float(), dout.float()
    wrt = [getattr(core, name) for name in PARAMS]
    if case["kind"] == "layer":
        wrt += [module.proj.weight, module.proj.bias]
    if case["kind"] == "soft":
        wrt.append(core.tau)
    if case["train"]:
        x.requires_grad_(True)
    return {"case": case, "module": module, "x": x, "dout": dout, "wrt": [x, *wrt]}


def _forward(state):
    if state["case"]["kind"] == "layer":
        x = state["x"]
        with torch.autocast("cuda", dtype=torch.float16):
            out, _ = state["module"](x, x, x)
        return out
    return state["module"](state["x"])


def run(state):
    if not state["case"]["train"]:
        with torch.no_grad():
            return {"out": _forward(state)}
    out = _forward(state)
    grads = torch.autograd.grad(out, state["wrt"], state["dout"].to(out.dtype))
    return {"out": out.detach(), "grads": list(grads)}


def tolerance(case):
    """About four times the error against 64 bits that float16 tensors and code products leave:
    3e-4 of the output, up to 1.7e-3 of the gradients; the soft aggregation's gate gradients
    cancel to a small rest and are up to 2.5e-3 off where few tokens add up."""
    if not case["train"]:
        return {"rel": 1.2e-3}
    return {"rel": 1e-2 if case["kind"] == "soft" else 7e-3}


def exact(case, seed):
    """The same outputs in 64 bits, in plain torch, one chunk of heads of one batch row at a time
    (differentiated by autograd; the chunks' gradients add up)."""
    B, N, H, m, dv = case["batch"], case["tokens"], case["heads"], case["cube"], case["head_dim"]
    if B * H * N * N > 6e9:
        return None
    t = {k: v.double() for k, v in _tensors(case, seed).items()}
    layer, soft, train = case["kind"] == "layer", case["kind"] == "soft", case["train"]
    D, scale = H * dv, case["scale"]
    idx = torch.arange(N, device=DEVICE)
    drop = torch.zeros(N, N, dtype=torch.bool, device=DEVICE)
    if case["causal"]:
        drop |= idx[None, :] > idx[:, None]
    if case["mask_diag"]:
        drop |= idx[None, :] == idx[:, None]
    dead = drop.all(1)[:, None]
    tau = torch.full((1,), case["tau"], dtype=torch.float64, device=DEVICE)
    leaves = {k: t[k].clone().requires_grad_(train) for k in PARAMS}
    tau.requires_grad_(train and soft)
    out = torch.zeros(B, N, D, dtype=torch.float64, device=DEVICE)
    dX = torch.zeros_like(out)
    datt = t["dout"] @ t["weight"] if layer else t["dout"]

    def heads_of(x, h0, h1):
        def split(w, width):
            return (x @ w[:, h0 * width:h1 * width]).view(N, h1 - h0, width).transpose(0, 1)

        z = split(leaves["W_phi"], m)
        phi = z.sigmoid() if case["projection"] == "sigmoid" else ((z + 1) / 2).clamp(0, 1)
        gate = (leaves["gate_q"] * leaves["gate_k"])[h0:h1, None, :]
        code = gate * phi
        bias = code.sum(-1)
        s = scale * (2 * phi @ code.transpose(1, 2).contiguous() - bias[:, :, None] - bias[:, None, :])
        s = s.masked_fill(drop, float("-inf")).masked_fill(dead, 0.0)
        v = split(leaves["W_V"], dv)
        if not soft:
            o = torch.softmax(s, -1) @ v
        else:
            sgn = -1.0 if case["erosion"] else 1.0
            u, w = sgn * s / tau, sgn * v / tau
            u = u.masked_fill(drop, float("-inf")).masked_fill(dead, 0.0)
            a, b = u.detach().amax(-1, keepdim=True), w.detach().amax(-2, keepdim=True)
            o = sgn * tau * (a + b + ((u - a).exp() @ (w - b).exp()).log())
        return o.masked_fill(dead, 0.0).transpose(0, 1).reshape(N, (h1 - h0) * dv)

    step = max(1, min(H, int(2.5e8 // (N * N))))
    for b in range(B):
        for h0 in range(0, H, step):
            h1 = min(H, h0 + step)
            cols = slice(h0 * dv, h1 * dv)
            x = t["x"][b].clone().requires_grad_(train)
            with torch.set_grad_enabled(train):
                o = heads_of(x, h0, h1)
            out[b, :, cols] = o.detach()
            if train:
                o.backward(datt[b, :, cols])
                dX[b] += x.grad
    y = torch.nn.functional.linear(out, t["weight"], t["bias"]) if layer else out
    if not train:
        return {"out": y}
    grads = [dX, *(leaves[k].grad for k in PARAMS)]
    if layer:
        flat = t["dout"].reshape(-1, D)
        grads += [flat.T.contiguous() @ out.reshape(-1, D), flat.sum(0)]
    if soft:
        grads.append(tau.grad)
    return {"out": y, "grads": grads}
