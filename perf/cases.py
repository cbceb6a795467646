"""The work a user of this framework has it do, as measurable cases.

Each case is one pass through a public entry point of `atlas_amd`: the memory
scan (forward, and forward + backward), the layer prologue, the sliding-window
attention of the MAG blocks, batched Polar-Express, and a whole model call.
Sizes are those of the repository's configurations (`bench.py` CONFIGS and
MODEL_CFGS, the `AtlasConfig` defaults) with the distributions of
`bench.make_layer_inputs`.

The chunk recurrence amplifies every rounding from chunk to chunk (two correct
fp32 evaluations of a long sequence end up O(1) apart), so the scan cases take
a segment of a few chunks: the first one of a sequence (model initial state)
or a later one (a state carried in).  Each chunk of a long sequence costs what
each chunk of a segment costs, and B*H streams run in parallel either way.
"""

import math
import os
import sys

import torch
import torch.nn.functional as F
import torch.utils.checkpoint

if os.path.join(os.getcwd(), "atlas-jax_amd") not in sys.path:
    sys.path.insert(0, os.path.join(os.getcwd(), "atlas-jax_amd"))

import atlas_amd as A  # noqa: E402

DT = {"fp32": torch.float32, "bf16": torch.bfloat16, "fp16": torch.float16}
BYTES = {"fp32": 4, "bf16": 2, "fp16": 2}


# ---------------------------------------------------------------------------
# The cases
# ---------------------------------------------------------------------------

def _scan(B, T, H, D, E, cs, w, io="bf16", init="carried", ns=5, gamma=True):
    return dict(op="scan", B=B, T=T, H=H, D=D, E=E, cs=cs, w=w, ns=ns, io=io, init=init, gamma=gamma)


def _train(B, T, H, D, E, cs, w, precision="f32", ns=5, gamma=True, ste=False):
    return dict(op="train", B=B, T=T, H=H, D=D, E=E, cs=cs, w=w, ns=ns, precision=precision, gamma=gamma, ste=ste)


def _attention(B, T, H, window, io="bf16", grad=False):
    return dict(op="attention", B=B, T=T, H=H, window=window, io=io, grad=grad)


def _prologue(B, T, H, D, w, io="bf16", grad=False):
    return dict(op="prologue", B=B, T=T, H=H, D=D, w=w, io=io, grad=grad)


def _polar(n, d1, d2, ns, io="fp32", muon=False):
    return dict(op="polar", n=n, d1=d1, d2=d2, ns=ns, io=io, muon=muon)


def _model(B, T, layers, C, H, expand, cs, w, vocab):
    return dict(op="model", B=B, T=T, layers=layers, C=C, H=H, expand=expand, cs=cs, w=w, vocab=vocab)


def listed():
    return [
        # The smallest memory layer in fp32 on one row: the call whose launches and latencies count.
        dict(_scan(1, 512, 4, 32, 32, 64, 16, io="fp32"), name="scan_small_fp32"),
        # The 59M language model's memory layer (8 rows, 8 heads), a later segment of its sequences.
        dict(_scan(8, 256, 8, 64, 128, 64, 32), name="scan_e128"),
        # The 170M model's memory layer (16 rows, 12 heads, fourfold memories), first segment, ragged length.
        dict(_scan(16, 250, 12, 64, 256, 64, 64, init="model"), name="scan_e256"),
        # Long context: one row, 16 heads, so few streams in parallel.
        dict(_scan(1, 256, 16, 64, 128, 64, 64), name="scan_one_row"),
        # The layer of the default AtlasConfig() (16 heads of 96), two rows.
        dict(_scan(2, 200, 16, 96, 192, 64, 16), name="scan_default_config"),
        # Training step of the 59M model's memory layer in the default (fp32) arithmetic: outputs and every gradient.
        dict(_train(8, 256, 8, 64, 128, 64, 32), name="train_e128"),
        # The same in the fp16 mode, one chunk.
        dict(_train(8, 64, 8, 64, 128, 64, 32, precision="f16"), name="train_e128_fp16"),
        # Prefill attention of the MAG transformer: 4 rows of 16 384 tokens, 12 heads, window 2048.
        dict(_attention(4, 16384, 12, 2048), name="attention_prefill"),
        # Attention of a MAG training step, forward and backward, odd length.
        dict(_attention(4, 4001, 12, 2048, grad=True), name="attention_train"),
        # Projections, convolutions, norms and gates of a training step of the 59M model, forward and backward.
        dict(_prologue(8, 4096, 8, 64, 32, grad=True), name="prologue_train"),
        # The reference's own Polar-Express benchmark: 65 536 matrices of 56 x 56, three steps, fp32.
        dict(_polar(65536, 56, 56, 3), name="polar_56"),
        # A short prompt through the whole 59M model: logits and the memory states.
        dict(_model(1, 60, 8, 512, 8, 2, 64, 32, 32768), name="model_prompt"),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    op = rng.choice(["scan", "scan", "scan", "train", "attention", "attention", "prologue", "polar", "model"])
    if op == "scan":
        H = rng.choice([4, 8, 12, 16])
        kind = rng.choice(["phase", "wide", "generic", "fp32"])
        cs = rng.choice([16, 64]) if kind == "generic" else rng.choice([32, 64, 64] + [128] * (kind != "fp32"))
        init = rng.choice(["model", "carried"])
        w = rng.choice([1, 16, 32, cs] if init == "carried" else [16, 32, cs])
        T = rng.randint(1, 4 * cs)
        # the zero initial memory comes with the window, as in the models (without it its first steps are ill-conditioned)
        gamma = init == "model" or rng.random() < 0.8
        io = rng.choice(["bf16", "bf16", "fp16"])
        if kind == "phase":
            D, E = rng.choice([(64, 128), (64, 128), (64, 64), (32, 64), (32, 128)])
            return _scan(_log(rng, 1, 16), T, H, D, E, cs, w, io, init, gamma=gamma)
        if kind == "wide":
            return _scan(_log(rng, 1, 8), T, H, 64, 256, cs, w, io, init, gamma=gamma)
        if kind == "generic":
            D, E = rng.choice([(96, 192), (48, 96), (96, 96)])
            return _scan(rng.randint(1, 2), T, H, D, E, cs, w, io, init, gamma=gamma)
        D, E = rng.choice([(32, 32), (32, 64), (64, 64), (64, 128)])
        return _scan(_log(rng, 1, 8), T, H, D, E, cs, w, "fp32", init, gamma=gamma)
    if op == "train":
        D, E = rng.choice([(32, 64), (64, 64), (64, 128), (64, 256)])
        H = rng.choice([4, 8, 12])
        B = _log(rng, 1, 2 if E == 256 else 8)
        if rng.random() < 0.5:
            cs = rng.choice([32, 64])
            return _train(B, rng.randint(cs // 2, 2 * cs), H, D, E, cs, rng.choice([1, 16, cs]),
                          ste=rng.random() < 0.25)
        cs = rng.choice([32, 48, 64, 96])
        if rng.random() < 0.5:   # straight-through Polar-Express: well conditioned at any length
            return _train(B, rng.randint(cs // 2, 2 * cs), H, D, E, cs, rng.choice([1, 16, cs]), "f16", ste=True)
        return _train(B, cs, H, D, min(E, 128), cs, rng.choice([32, cs]), "f16")
    if op == "attention":
        grad = rng.random() < 0.5
        T = _log(rng, 33, 4096 if grad else 16384)
        return _attention(rng.randint(1, 4), T, rng.choice([4, 8, 12, 16]), _log(rng, 16, 4096),
                          rng.choice(["bf16", "bf16", "fp16"]), grad)
    if op == "prologue":
        H, D = rng.choice([(8, 64), (12, 64), (4, 32), (16, 32)])
        return _prologue(rng.randint(1, 8), _log(rng, 17, 4096), H, D, rng.choice([1, 32]),
                         rng.choice(["bf16", "fp16", "fp32"]), rng.random() < 0.5)
    if op == "polar":
        d1, d2 = rng.randint(8, 64), _log(rng, 16, 250)
        if rng.random() < 0.5:
            d1, d2 = d2, d1
        n = max(8, min(_log(rng, 64, 65536), (1 << 27) // (d1 * d2)))
        return _polar(n, d1, d2, rng.choice([3, 5]), rng.choice(["fp32", "fp32", "bf16"]), rng.random() < 0.5)
    H = rng.choice([4, 8, 12])
    return _model(rng.randint(1, 2), rng.randint(3, 64), rng.randint(2, 8), 64 * H, H, rng.choice([2, 4]), 64,
                  rng.choice([16, 64]), rng.choice([8192, 32768]))


# ---------------------------------------------------------------------------
# Inputs and passes
# ---------------------------------------------------------------------------

def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _unit(x):
    return x / x.norm(dim=-1, keepdim=True)


def _layer_inputs(c, seed, io):
    g = _gen(seed)
    B, T, H, D, E = c["B"], c["T"], c["H"], c["D"], c["E"]

    def rnd(*s):
        return torch.randn(*s, device="cuda", generator=g)

    q, k, v = (x.to(io) for x in (_unit(rnd(B, T, H, D)), _unit(rnd(B, T, H, D)), rnd(B, T, H, D)))
    gates = [torch.sigmoid(rnd(B, T, H)) for _ in range(4)]
    gates[1] = gates[1] * 0.1
    if not c["gamma"]:
        gates[3] = None
    if c.get("init") == "model":
        W1, W2 = torch.zeros(B, H, D, E, device="cuda"), torch.zeros(B, H, E, D, device="cuda")
        W2[:, :, :D, :D] = torch.eye(D, device="cuda")
        S1, S2 = torch.zeros_like(W1), torch.zeros_like(W2)
    else:
        W1, W2 = rnd(B, H, D, E) / D ** 0.5, rnd(B, H, E, D) / D ** 0.5
        S1, S2 = 1e-3 * rnd(B, H, D, E), 1e-3 * rnd(B, H, E, D)
    return q, k, v, gates, A.DeepMemoryState(W1, W2, S1, S2)


def _model_of(c, seed):
    cfg = A.AtlasConfig(n_layer=c["layers"], n_embd=c["C"], n_head=c["H"], memory_expand=c["expand"],
                        chunk_size=c["cs"], omega_window=c["w"], ns_steps=5, poly_degree=2, vocab_size=c["vocab"])
    g = _gen(seed)
    model = A.Atlas(cfg, generator=g, device="cuda", dtype=torch.bfloat16)
    return model, torch.randint(0, c["vocab"], (c["B"], c["T"]), device="cuda", generator=g)


def prepare(case, seed):
    c, op = case, case["op"]
    s = {"case": c}
    if op == "scan":
        s["q"], s["k"], s["v"], s["gates"], s["state"] = _layer_inputs(c, seed, DT[c["io"]])
    elif op == "train":
        q, k, v, gates, st = _layer_inputs(c, seed, torch.float32)
        s["leaves"] = [None if t is None else t.requires_grad_(True) for t in (q, k, v, *gates, *st)]
        g = _gen(seed + 1000003)
        s["dy"] = torch.randn(q.shape, device="cuda", generator=g)
        s["dstate"] = [torch.randn(t.shape, device="cuda", generator=g) for t in st]
    elif op == "attention":
        g = _gen(seed)
        B, T, H = c["B"], c["T"], c["H"]
        qkv = torch.randn(B, T, 3, H, 64, device="cuda", generator=g).to(DT[c["io"]])
        s["cos"], s["sin"] = A.RotaryEmbedding(64)(T)
        s["qkv"] = qkv.requires_grad_(True) if c["grad"] else qkv
        if c["grad"]:
            s["dout"] = torch.randn(B, T, H, 64, device="cuda", generator=g).to(DT[c["io"]])
    elif op == "prologue":
        g = _gen(seed)
        B, T, H, D, io = c["B"], c["T"], c["H"], c["D"], DT[c["io"]]
        cfg = A.AtlasConfig(n_embd=H * D, n_head=H, omega_window=c["w"], poly_degree=2)
        s["layer"] = A.AtlasMemoryLayer(cfg, generator=g, device="cuda", dtype=torch.float32)
        with torch.no_grad():   # a trained convolution's taps, rather than the near-zero initial ones
            for conv in (s["layer"].conv_q, s["layer"].conv_k, s["layer"].conv_v):
                conv.weight.normal_(0.0, 0.5, generator=g)
        s["x"] = torch.randn(B, T, H * D, device="cuda", generator=g).to(io).requires_grad_(c["grad"])
        if c["grad"]:
            s["douts"] = [torch.randn(B, T, H, D, device="cuda", generator=g).to(io) for _ in range(3)] + \
                [torch.randn(B, T, H, device="cuda", generator=g) for _ in range(5 if c["w"] > 1 else 4)]
            s["params"] = _prologue_params(s["layer"])
    elif op == "polar":
        s["x"] = torch.randn(c["n"], c["d1"], c["d2"], device="cuda", generator=_gen(seed)).to(DT[c["io"]])
    else:
        s["model"], s["idx"] = _model_of(c, seed)
    return s


def _prologue_params(layer):
    gates = [layer.gate_alpha, layer.gate_eta, layer.gate_theta] + ([layer.gate_gamma] if layer.gate_gamma else [])
    return ([layer.c_q.weight, layer.c_k.weight, layer.c_v.weight] + [g.weight for g in gates] +
            [layer.retrieve_gate.weight] + [g.bias for g in gates] +
            [t for c in (layer.conv_q, layer.conv_k, layer.conv_v) for t in (c.weight, c.bias)] +
            [layer.poly_coeffs])


def run(s):
    c, op = s["case"], s["case"]["op"]
    if op == "scan":
        with torch.no_grad():
            y, st = A.memory_scan(s["q"], s["k"], s["v"], *s["gates"], s["state"], c["cs"], c["w"], c["ns"])
        return [y, *st]
    if op == "train":
        leaves = s["leaves"]
        y, st = A.memory_scan(*leaves[:7], A.DeepMemoryState(*leaves[7:]), c["cs"], c["w"], c["ns"],
                              pe_ste=c["ste"], train_precision=c["precision"])
        grads = torch.autograd.grad([y, *st], [t for t in leaves if t is not None], [s["dy"], *s["dstate"]])
        return [y, *st, *grads]
    if op == "attention":
        q, k, v = s["qkv"].unbind(2)
        out = A.swa_attention(q, k, v, c["window"], s["cos"], s["sin"])
        if not c["grad"]:
            return out
        return [out, *torch.autograd.grad(out, [s["qkv"]], s["dout"])]
    if op == "prologue":
        if not c["grad"]:
            with torch.no_grad():
                return [t for t in s["layer"].prologue(s["x"]) if t is not None]
        outs = [t for t in s["layer"].prologue(s["x"]) if t is not None]
        return outs + list(torch.autograd.grad(outs, [s["x"], *s["params"]], s["douts"]))
    if op == "polar":
        if c["muon"]:
            return A.muon_polar_express(s["x"], c["ns"])
        return A.polar_express(s["x"], c["ns"])
    with torch.no_grad():
        logits, states = s["model"](s["idx"])
    return [logits, *(t for st in states for t in st)]


# ---------------------------------------------------------------------------
# What a pass cannot do without
# ---------------------------------------------------------------------------

def _polar_flops(D, E, ns):
    return ns * (4 * D * D * E + 2 * D ** 3)


def _scan_work(c, io_bytes, layers=1):
    tok = c["B"] * c["T"] * c["H"] * layers
    D, E = c["D"], c["E"]
    flops = tok * (2 * _polar_flops(min(D, E), max(D, E), c["ns"]) + 12 * D * E)
    nbytes = tok * (4 * D * io_bytes + 16) + 8 * c["B"] * c["H"] * D * E * 4 * layers
    return flops, nbytes


def _pairs(T, window):
    w = min(window, T - 1)
    return w * (w + 1) // 2 + (T - w) * (w + 1)


def work(case):
    c, op = case, case["op"]
    if op == "scan":
        flops, nbytes = _scan_work(c, BYTES[c["io"]])
    elif op == "train":   # forward, and a backward of twice its products
        flops, nbytes = _scan_work(c, 4)
        flops, nbytes = 3 * flops, 3 * nbytes
    elif op == "attention":
        n = c["B"] * c["H"] * _pairs(c["T"], c["window"])
        x = c["B"] * c["T"] * c["H"] * 64 * BYTES[c["io"]]
        flops, nbytes = n * 64 * (14 if c["grad"] else 4), x * (8 if c["grad"] else 4)
    elif op == "prologue":
        C, n = c["H"] * c["D"], c["B"] * c["T"]
        cols = 3 * C + (5 if c["w"] > 1 else 4) * c["H"]
        flops = 2 * n * C * cols * (3 if c["grad"] else 1)
        nbytes = n * (4 * C * BYTES[c["io"]] + 4 * (cols - 3 * C)) * (2 if c["grad"] else 1) + 4 * C * cols
    elif op == "polar":
        D, E = min(c["d1"], c["d2"]), max(c["d1"], c["d2"])
        flops, nbytes = c["n"] * _polar_flops(D, E, c["ns"]), 2 * c["n"] * D * E * BYTES[c["io"]]
    else:
        C, n, L, V = c["C"], c["B"] * c["T"], c["layers"], c["vocab"]
        flops, nbytes = _scan_work(dict(c, D=64, E=64 * c["expand"], ns=5), 2, L)
        inner = int(C * 8 / 3)
        weights = L * (4 * C * C + 3 * C * inner) + C * V
        flops += 2 * n * weights
        nbytes += 2 * weights + 4 * n * V
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    """About four times the largest error measured against `exact` over these
    ranges (one implementation's rounding, grown over up to four or eight chunks
    in the scans), but at most 0.03: of the gradients of the fp16 training step
    eta's, a sum over tokens that largely cancels, is 3.5e-2 off by itself."""
    c, op = case, case["op"]
    if op == "scan":
        return {"rel": 3e-3 if c["io"] == "fp32" else 0.03}
    if op == "train":
        return {"rel": 2e-3 if c["precision"] == "f32" else 0.03}
    if op == "attention":
        return {"rel": 7e-3 if c["io"] == "bf16" else 2e-3}
    if op == "prologue":
        return {"rel": {"bf16": 1.5e-2, "fp16": 4e-3, "fp32": 1e-5}[c["io"]]}
    if op == "polar":
        return {"rel": 1.5e-5 if c["io"] == "fp32" or c["muon"] else 0.02}
    return {"rel": 0.03}


# ---------------------------------------------------------------------------
# The same in 64 bits, plain torch
# ---------------------------------------------------------------------------

COEFFS = A.POLAR_EXPRESS_COEFFS   # the five published quintics: data of the algorithm


def _gelu(x):
    return F.gelu(x, approximate="tanh")


def _gelu_slope(x):
    return 0.5 * (1 + torch.erf(x / math.sqrt(2))) + x * torch.exp(-x * x / 2) / math.sqrt(2 * math.pi)


def _polar64(X, ns, eps=1e-12):
    tall = X.shape[-2] > X.shape[-1]
    X = X.mT.contiguous() if tall else X
    X = X / (torch.sqrt((X * X).sum((-2, -1), keepdim=True) + eps) * 1.01 + 1e-6)
    for a, b, c in COEFFS[:ns]:
        G = X @ X.mT.contiguous()
        X = a * X + (b * G + c * (G @ G)) @ X
    return X.mT.contiguous() if tall else X


def _polar64_ste(X, ns):
    return X + (_polar64(X, ns) - X).detach()


def _recur(gate, x, h):
    """h_t = gate_t h_(t-1) + x_t over axis 1, every h_t."""
    out = []
    for t in range(x.shape[1]):
        h = gate[:, t, :, None, None] * h + x[:, t]
        out.append(h)
    return torch.stack(out, 1)


def _chunk64(W1, W2, S1, S2, q, k, v, al, et, th, ga, w, ns, ste):
    D, n = q.shape[-1], q.shape[1]
    h = torch.einsum("bhed,bthd->bthe", W2, k)
    act = _gelu(h)
    err = k + torch.einsum("bhde,bthe->bthd", W1, act) - v
    chain = torch.einsum("bhde,bthd->bthe", W1, err) * _gelu_slope(h)
    u1 = 2 / D * err.unsqueeze(-1) * act.unsqueeze(-2)
    u2 = 2 / D * chain.unsqueeze(-1) * k.unsqueeze(-2)
    if ga is not None and w > 1:
        i = torch.arange(n, device=q.device)
        band = ((i[None] <= i[:, None]) & (i[:, None] - i[None] < w)).to(q.dtype)
        u1, u2 = (torch.einsum("ti,bihde->bthde", band, ga[..., None, None] * u) for u in (u1, u2))
    S1a = _recur(th, -et[..., None, None] * u1, S1)
    S2a = _recur(th, -et[..., None, None] * u2, S2)
    polar = _polar64_ste if ste else _polar64
    W1a = _recur(al, polar(S1a, ns), W1)
    W2a = _recur(al, polar(S2a, ns), W2)
    y = q + torch.einsum("bthde,bthe->bthd", W1a, _gelu(torch.einsum("bthed,bthd->bthe", W2a, q)))
    return y, W1a[:, -1], W2a[:, -1], S1a[:, -1], S2a[:, -1]


def _scan64(q, k, v, al, et, th, ga, state, cs, w, ns, ste=False):
    T = q.shape[1]
    pad = -T % cs

    def fill(t, value):
        return t if t is None or not pad else F.pad(t, (0, 0) * (t.dim() - 2) + (0, pad), value=value)

    q, k, v, al, et, th, ga = fill(q, 0.0), fill(k, 0.0), fill(v, 0.0), fill(al, 1.0), fill(et, 0.0), fill(th, 0.0), \
        fill(ga, 0.0)
    ys = []
    for t in range(0, T + pad, cs):
        at = [x if x is None else x[:, t:t + cs] for x in (q, k, v, al, et, th, ga)]
        y, *state = torch.utils.checkpoint.checkpoint(_chunk64, *state, *at, w, ns, ste, use_reentrant=False)
        ys.append(y)
    return torch.cat(ys, 1)[:, :T], state


def _rows(f, n, step):
    return [f(i, min(n, i + step)) for i in range(0, n, step)]


def _d(t):
    return None if t is None else t.detach().double()


def _rms(x):
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + 1e-6)


def _prologue64(x, p, c):
    """q, k, v, the gates and the retrieve gate; p: _prologue_params in their order."""
    H, D = c["H"], c["D"]
    ng = 4 if c["w"] > 1 else 3
    ws, bs, conv, poly = p[:3 + ng + 1], p[4 + ng:4 + 2 * ng], p[4 + 2 * ng:-1], p[-1]
    B, T, C = x.shape

    def short(i):
        y = F.conv1d(F.pad((x @ ws[i].T).transpose(1, 2), (conv[2 * i].shape[-1] - 1, 0)), conv[2 * i],
                     conv[2 * i + 1], groups=C)
        return y.transpose(1, 2).reshape(B, T, H, D)

    def series(t):
        return sum(poly[j] * t ** (j + 1) for j in range(poly.shape[0]))

    q, k, v = short(0), short(1), short(2)
    gates = [torch.sigmoid(x @ ws[3 + i].T + bs[i]) * (0.1 if i == 1 else 1.0) for i in range(ng)]
    return [series(_rms(q)), _rms(series(k)), v, *gates, torch.sigmoid(x @ ws[3 + ng].T)]


def _attention64(qkv, cos, sin, window):
    """One row and head: (T, 3, 64) -> (T, 64), in blocks of queries."""
    T = qkv.shape[0]

    def turn(x):
        a, b = x[:, :32], x[:, 32:]
        return torch.cat([a * cos - b * sin, b * cos + a * sin], 1)

    q, k, v = turn(qkv[:, 0]), turn(qkv[:, 1]), qkv[:, 2]
    i = torch.arange(T, device=qkv.device)

    def block(a, b):
        s0 = max(0, a - window)
        sc = q[a:b] @ k[s0:b].T / 8.0
        far = i[a:b, None] - i[None, s0:b]
        return torch.softmax(sc.masked_fill((far < 0) | (far > window), -math.inf), -1) @ v[s0:b]

    return torch.cat(_rows(lambda a, b: torch.utils.checkpoint.checkpoint(block, a, b, use_reentrant=False), T, 2048))


def _model64(model, idx, c):
    P = {n: p.detach().double() for n, p in model.named_parameters()}
    B, T = idx.shape
    H, D, E = c["H"], 64, 64 * c["expand"]
    x = P["wte.weight"][idx]
    states = []
    for i in range(c["layers"]):
        n = f"blocks.{i}.memory."
        gates = ["alpha", "eta", "theta", "gamma"]
        p = [P[n + f"c_{a}.weight"] for a in "qkv"] + [P[n + f"gate_{g}.weight"] for g in gates] + \
            [P[n + "retrieve_gate.weight"]] + [P[n + f"gate_{g}.bias"] for g in gates] + \
            [P[n + f"conv_{a}.{b}"] for a in "qkv" for b in ("weight", "bias")] + [P[n + "poly_coeffs"]]
        q, k, v, al, et, th, ga, r = _prologue64(_rms(x), p, dict(H=H, D=D, w=c["w"]))
        W1, W2 = x.new_zeros(B, H, D, E), x.new_zeros(B, H, E, D)
        W2[:, :, :D, :D] = torch.eye(D, dtype=x.dtype, device=x.device)
        y, st = _scan64(q, k, v, al, et, th, ga, (W1, W2, W1 * 0, W2 * 0), c["cs"], c["w"], 5)
        states += st
        x = x + (y * r[..., None]).reshape(B, T, H * D) @ P[n + "c_proj.weight"].T
        a, b = (_rms(x) @ P[f"blocks.{i}.mlp.c_fc.weight"].T).chunk(2, -1)
        x = x + (F.silu(b) * a) @ P[f"blocks.{i}.mlp.c_proj.weight"].T
    return [(_rms(x) @ P["lm_head.weight"].T)[..., :c["vocab"]], *states]


def exact(case, seed):
    c, op = case, case["op"]
    s = prepare(case, seed)
    if op == "scan":
        with torch.no_grad():
            # a row at a time: every token's matrices are kept
            parts = _rows(lambda a, b: _scan64(*(_d(t if t is None else t[a:b]) for t in (s["q"], s["k"], s["v"],
                                                                                      *s["gates"])),
                                               [_d(t[a:b]) for t in s["state"]], c["cs"], c["w"], c["ns"]), c["B"], 4)
        return [torch.cat([y for y, _ in parts])] + [torch.cat([st[i] for _, st in parts]) for i in range(4)]
    if op == "train":
        def rows(a, b):
            ins = [None if t is None else _d(t[a:b]).requires_grad_(True) for t in s["leaves"]]
            y, st = _scan64(*ins[:7], ins[7:], c["cs"], c["w"], c["ns"], c["ste"])
            outs = [y, *st]
            g = torch.autograd.grad(outs, [t for t in ins if t is not None],
                                    [_d(t[a:b]) for t in (s["dy"], *s["dstate"])], allow_unused=True)
            g = [torch.zeros_like(t) if d is None else d for d, t in zip(g, [t for t in ins if t is not None])]
            return [t.detach() for t in (*outs, *g)]
        return [torch.cat(t) for t in zip(*_rows(rows, c["B"], 2))]
    if op == "attention":
        x, cos, sin = _d(s["qkv"]).requires_grad_(c["grad"]), _d(s["cos"]), _d(s["sin"])
        out = torch.stack([torch.stack([_attention64(x[b, :, :, h], cos, sin, c["window"]) for h in range(c["H"])], 1)
                           for b in range(c["B"])])
        if not c["grad"]:
            return out
        return [out.detach(), *torch.autograd.grad(out, [x], _d(s["dout"]))]
    if op == "prologue":
        p = [_d(t).requires_grad_(c["grad"]) for t in _prologue_params(s["layer"])]
        x = _d(s["x"]).requires_grad_(c["grad"])
        outs = _prologue64(x, p, c)
        if not c["grad"]:
            return [t.detach() for t in outs]
        return [t.detach() for t in outs] + list(torch.autograd.grad(outs, [x, *p], [_d(t) for t in s["douts"]]))
    if op == "polar":
        return torch.cat(_rows(lambda a, b: _polar64(_d(s["x"][a:b]), c["ns"], 0.0 if c["muon"] else 1e-12), c["n"],
                               8192))
    with torch.no_grad():
        return _model64(s["model"], s["idx"], c)
