"""The calls a user of this framework makes, with the sizes they make them at, for timing and for
comparing outputs.

Every case is a dict of plain values; ``kind`` names the public entry point it goes through:

  train    one attention sublayer, forward (state kept on the tape) and reverse-scan backward:
           ``HipSweepCell.layer_forward`` / ``layer_backward`` as a training engine drives them
  autograd the same through ``autograd.dm_layer`` and torch's autograd
  module   ``DualModAttention.forward`` without gradients: the exact scan (K = c)
  chunk    ``engine.chunk_cell_forward``: one chunk against a committed prefix
  decode   ``StaticTape.step``: one token per sequence on a static tape
  prompt   ``GraphDecoder.step`` over a prompt: a whole LM, one captured graph per token
  trunk    ``HipTrunk.train_step``: a whole LM's training step
  stack    ``HipLayerStack.step``: several attention sublayers, layer-batched

``exact`` restates the layer in 64-bit torch: RMSNorm, projections, RoPE on half-split pairs, per
chunk K Jacobi sweeps of attention over [committed rows | earlier rows of the chunk | the raw self
pair] followed by the gated refinement of the chunk's keys and values, and W_O.
"""

import math

import torch
import torch.nn.functional as F

DEV = "cuda"
EPS = 1e-5
THETA = 10000.0


# ---------------------------------------------------------------------------------------------
# the cases
# ---------------------------------------------------------------------------------------------

def listed():
    return [
        # the 340M model's layer in training: the headline workload of bench.py
        dict(name="train_340m", kind="train", d=1024, h=16, B=8, T=2048, c=64, K=4, mod="mult_res", dtype="bf16",
             window=0),
        # the 1.3B-class layer (16 heads of 128) at its training length
        dict(name="train_2048", kind="train", d=2048, h=16, B=4, T=4096, c=64, K=4, mod="mult_res", dtype="bf16",
             window=0),
        # fine-tuning on sequences that do not divide into chunks, under torch autograd, with the
        # configuration's default context operator
        dict(name="autograd_ragged", kind="autograd", d=1024, h=16, B=3, T=1000, c=64, K=4, mod="linear",
             dtype="bf16", window=0),
        # the small fp32 configuration people check gradients with: exact chunks of 16
        dict(name="train_fp32_small", kind="train", d=256, h=4, B=2, T=64, c=16, K=16, mod="mult_res", dtype="fp32",
             window=0),
        # evaluation through the module: the default configuration's width, the exact scan
        dict(name="module_exact", kind="module", d=512, h=8, B=2, T=300, mod="mult_res", dtype="bf16", window=0),
        # serving a prompt chunk by chunk against what is already committed
        dict(name="chunk_prefill", kind="chunk", d=1024, h=16, B=2, a=1984, c=64, K=4, mod="mult_res", dtype="bf16",
             window=0),
        # one interactive request: a single sequence, a short tape
        dict(name="decode_one", kind="decode", d=1024, h=16, B=1, P=2048, pos=777, mod="mult_res", dtype="bf16",
             window=0),
        # a modest serving batch of the wider layer
        dict(name="decode_16", kind="decode", d=2048, h=16, B=16, P=4096, pos=3001, mod="mult_res", dtype="bf16",
             window=0),
        # long-context batch decoding: bench.py's decode workload
        dict(name="decode_64_long", kind="decode", d=1024, h=16, B=64, P=33024, pos=32768, mod="mult_res",
             dtype="bf16", window=0),
        # a whole 340M-shape model stepping through a prompt, one graph replay per token
        dict(name="prompt_340m", kind="prompt", d=1024, h=16, layers=24, vocab=32000, B=8, P=512, n=12,
             mod="mult_res"),
        # a whole model's training step (embedding, attention, SwiGLU, head, loss)
        dict(name="trunk_step", kind="trunk", d=1024, h=16, layers=3, ffn=2816, vocab=32000, B=4, T=1024, c=64, K=4,
             mod="mult_res", wavefront=False),
        # several attention sublayers, layer-batched
        dict(name="stack_wave", kind="stack", d=1024, h=16, layers=8, B=8, T=512, c=64, K=4, mod="mult_res",
             dtype="bf16"),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _width(rng, lo=256, hi=2048):
    """(d_model, heads): head_dim 64 or 128, d_model a multiple of 256."""
    d = 256 * max(lo // 256, min(hi // 256, _log(rng, lo, hi) // 256))
    return d, d // (128 if rng.random() < 0.3 else 64)


def _mod(rng):
    return rng.choice(["mult_res", "mult_res", "mult_res", "linear", "mult", "fusion"])


def draw(rng):
    """One more case: the same entry points over the ranges the listed ones stand for."""
    kind = rng.choice(["train", "train", "autograd", "module", "chunk", "decode", "decode", "decode", "prompt",
                       "trunk", "stack"])
    if kind in ("train", "autograd"):
        d, h = _width(rng)
        fp32 = rng.random() < 0.25
        rows = _log(rng, 128, 16384 if not fp32 else 2048)      # B * T
        B = min(rng.randint(1, 8), rows)
        T = max(16, min(4096, rows // B))
        c = rng.choice([64, 64, 64, 32, 48])
        K = rng.choice([1, 2, 4, 4, 8])
        if B * T * K * d > 8 * 2048 * 4 * 1024:                  # no larger than the listed layers
            K = max(1, 8 * 2048 * 4 * 1024 // (B * T * d))
        return dict(kind=kind, d=d, h=h, B=B, T=T, c=c, K=K, mod=_mod(rng), dtype="fp32" if fp32 else "bf16",
                    window=rng.choice([0, 0, 0, 200]))
    if kind == "module":
        d, h = _width(rng, 256, 1024)
        return dict(kind=kind, d=d, h=h, B=rng.randint(1, 8), T=_log(rng, 20, 600), mod=_mod(rng),
                    dtype=rng.choice(["bf16", "bf16", "fp32"]), window=rng.choice([0, 0, 100]))
    if kind == "chunk":
        d, h = _width(rng)
        return dict(kind=kind, d=d, h=h, B=_log(rng, 1, 8), a=_log(rng, 1, 4096), c=rng.choice([64, 64, 37, 16]),
                    K=rng.choice([1, 4, 8, 16]), mod=_mod(rng), dtype=rng.choice(["bf16", "bf16", "fp32"]),
                    window=0)
    if kind == "decode":
        d, h = _width(rng)
        B = _log(rng, 1, 64)
        P = _log(rng, 64, min(33024, 33024 * 64 * 1024 // (B * d)))
        return dict(kind=kind, d=d, h=h, B=B, P=P, pos=rng.randint(P // 2, P - 1), mod=_mod(rng),
                    dtype=rng.choice(["bf16", "bf16", "bf16", "fp32"]) if B * P * d <= 2 ** 28 else "bf16",
                    window=rng.choice([0, 0, 0, 1000]))
    if kind == "prompt":
        d, h = _width(rng, 512, 1024)
        return dict(kind=kind, d=d, h=h, layers=rng.randint(2, 12), vocab=32000, B=_log(rng, 1, 64), P=512,
                    n=rng.randint(2, 12), mod=_mod(rng))
    if kind == "trunk":
        d, h = _width(rng, 256, 1024)
        return dict(kind=kind, d=d, h=h, layers=rng.randint(1, 3), ffn=128 * rng.randint(d // 64, 22 * d // 1024 + 1),
                    vocab=rng.choice([8000, 32000]), B=rng.randint(1, 4), T=64 * rng.randint(1, 16), c=64,
                    K=rng.choice([1, 2, 4]), mod=_mod(rng), wavefront=rng.random() < 0.3)
    d, h = _width(rng, 256, 1024)
    return dict(kind="stack", d=d, h=h, layers=rng.randint(2, 8), B=rng.randint(1, 8), T=64 * rng.randint(1, 8), c=64,
                K=rng.choice([1, 2, 4]), mod=_mod(rng), dtype="bf16")


# ---------------------------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------------------------

def _dtype(case):
    return torch.float32 if case.get("dtype") == "fp32" else torch.bfloat16


def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(1000003 * (seed + 1))


def _randn(g, *shape, scale=1.0, dtype=torch.float32):
    return (torch.randn(*shape, generator=g, device=DEV) * scale).to(dtype)


def _attn_params(case, g, dt, std=0.02):
    """One attention layer's parameters by their state-dict names; values of the storage dtype."""
    d = case["d"]
    w = lambda *s: _randn(g, *s, scale=std, dtype=dt)                         # noqa: E731
    one = lambda: (1.0 + _randn(g, d, scale=0.1)).to(dt)                      # noqa: E731
    p = {n + ".weight": w(d, d) for n in ("wq", "wk", "wv", "wo", "w_kctx", "w_vctx")}
    for n in ("w_gk", "w_gv"):
        p[n + ".weight"], p[n + ".bias"] = w(d, 2 * d), w(d)
    if case["mod"] in ("mult", "mult_res"):
        p["v_gate.weight"], p["v_gate.bias"], p["v_map.weight"] = w(d, d), w(d), w(d, d)
    elif case["mod"] == "fusion":
        p["v_pre.weight"] = w(d, 2 * d)
    p["norm_ctx.weight"], p["attn_norm.weight"] = one(), one()
    return p


def _block_params(case, g, dt, ffn, std=0.02):
    d = case["d"]
    p = {("attn." + k if k != "attn_norm.weight" else k): v for k, v in _attn_params(case, g, dt, std).items()}
    p["mlp_norm.weight"] = (1.0 + _randn(g, d, scale=0.1)).to(dt)
    p["mlp.w1.weight"] = _randn(g, ffn, d, scale=std, dtype=dt)
    p["mlp.w3.weight"] = _randn(g, ffn, d, scale=std, dtype=dt)
    p["mlp.w2.weight"] = _randn(g, d, ffn, scale=std, dtype=dt)
    return p


def _lm_params(case, g, ffn):
    """A whole LM's parameters: bf16 values held as fp32 masters."""
    sd = {"tok_emb.weight": _randn(g, case["vocab"], case["d"], scale=0.02, dtype=torch.bfloat16).float()}
    for l in range(case["layers"]):
        for k, v in _block_params(case, g, torch.bfloat16, ffn).items():
            sd[f"blocks.{l}.{k}"] = v.float()
    sd["norm_f.weight"] = (1.0 + _randn(g, case["d"], scale=0.1)).bfloat16().float()
    return sd


def _rope(n, dh):
    inv = 1.0 / THETA ** (torch.arange(0, dh, 2, dtype=torch.float64, device=DEV) / dh)
    f = torch.outer(torch.arange(n, dtype=torch.float64, device=DEV), inv)
    return f.cos().float(), f.sin().float()


def _schedule(T, c, K):
    return [(p, min(c, T - p), min(K, min(c, T - p))) for p in range(0, T, c)]


def _cfg(case, **kw):
    from dual_mod_public_amd.config import DualModConfig
    return DualModConfig(d_model=case["d"], n_heads=case["h"], ctx_mod=case["mod"],
                         local_window=case.get("window", 0), **kw)


def _inputs(case, seed):
    """The tensors of a case, from the seed alone (shared by prepare and exact)."""
    g, kind, dt = _gen(seed), case["kind"], _dtype(case)
    d, h, B = case["d"], case["h"], case["B"]
    dh = d // h
    if kind in ("train", "autograd"):
        i = dict(p=_attn_params(case, g, dt), x=_randn(g, B, case["T"], d, dtype=dt),
                 dy=_randn(g, B, case["T"], d, dtype=dt))
        i["cos"], i["sin"] = _rope(case["T"], dh)
    elif kind == "module":
        i = dict(p=_attn_params(case, g, dt), x=_randn(g, B, case["T"], d, dtype=dt))
        i["cos"], i["sin"] = _rope(case["T"], dh)
    elif kind == "chunk":
        i = dict(p=_attn_params(case, g, dt), x=_randn(g, B, case["c"], d, dtype=dt),
                 K=_randn(g, B, h, case["a"] + case["c"], dh, dtype=dt),
                 V=_randn(g, B, h, case["a"] + case["c"], dh, scale=0.6, dtype=dt))
        i["cos"], i["sin"] = _rope(case["a"] + case["c"], dh)
    elif kind == "decode":
        i = dict(p=_attn_params(case, g, dt), x=_randn(g, B, d, dtype=dt))
        i["K"] = torch.empty(B, h, case["P"], dh, device=DEV, dtype=dt)
        i["V"] = torch.empty_like(i["K"])
        for b in range(B):   # row by row: the fp32 draw of a long tape is never held whole
            i["K"][b] = _randn(g, h, case["P"], dh, dtype=dt)
            i["V"][b] = _randn(g, h, case["P"], dh, scale=0.6, dtype=dt)
        i["cos"], i["sin"] = _rope(case["P"], dh)
    elif kind == "prompt":
        i = dict(sd=_lm_params(case, g, _ffn_default(d)))
        i["tok"] = torch.randint(0, case["vocab"], (B, case["n"]), generator=g, device=DEV)
    elif kind == "trunk":
        i = dict(sd=_lm_params(case, g, case["ffn"]))
        i["idx"] = torch.randint(0, case["vocab"], (B, case["T"]), generator=g, device=DEV)
        i["targets"] = torch.randint(0, case["vocab"], (B, case["T"]), generator=g, device=DEV)
    else:
        i = dict(ps=[_attn_params(case, g, dt) for _ in range(case["layers"])],
                 x=_randn(g, B, case["T"], d, dtype=dt), dy=_randn(g, B, case["T"], d, dtype=dt))
        i["cos"], i["sin"] = _rope(case["T"], dh)
    return i


def _ffn_default(d):
    return int(round(d * 8 / 3 / 64) * 64)


def _lm(case, sd, ffn=0):
    """A DualModLM on the GPU with these parameters."""
    from dual_mod_public_amd.model import DualModLM
    cfg = _cfg(case, n_layers=case["layers"], vocab_size=case["vocab"],
               max_seq_len=max(case.get("P", 0), case.get("T", 0)), mlp_hidden_override=ffn)
    with torch.device(DEV):
        m = DualModLM(cfg).eval()
    m.load_state_dict(dict(sd, **{"lm_head.weight": sd["tok_emb.weight"]}))
    return m


# ---------------------------------------------------------------------------------------------
# prepare / run
# ---------------------------------------------------------------------------------------------

def prepare(case, seed):
    i, kind, dt = _inputs(case, seed), case["kind"], _dtype(case)
    s = dict(kind=kind, case=case)
    if kind in ("train", "autograd"):
        from dual_mod_public_amd.engine import HipSweepCell, LayerGrads
        cfg = _cfg(case, max_seq_len=case["T"])
        cell = HipSweepCell(cfg, case["B"], case["T"], device=DEV, dtype=dt).pack(i["p"])
        sched = _schedule(case["T"], case["c"], case["K"])
        s.update(cell=cell, sched=sched, x=i["x"], dy=i["dy"], cos=i["cos"], sin=i["sin"])
        if kind == "train":
            dh = case["d"] // case["h"]
            s["K"] = torch.zeros(case["B"], case["h"], case["T"], dh, device=DEV, dtype=dt)
            s["V"], s["ocat"] = torch.zeros_like(s["K"]), torch.empty_like(i["x"])
            s["y"], s["dx"] = torch.empty_like(i["x"]), torch.empty_like(i["x"])
            s["bufs"], s["tape"] = cell.new_bufs(case["T"]), cell.new_tape(sched)
            s["grads"] = LayerGrads(cfg, DEV)
        else:
            s["params"] = {k: v.requires_grad_() for k, v in i["p"].items()}
            s["x"] = i["x"].requires_grad_()
    elif kind in ("module", "chunk"):
        from dual_mod_public_amd.attention import DualModAttention
        n = case["T"] if kind == "module" else case["a"] + case["c"]
        with torch.device(DEV):
            m = DualModAttention(_cfg(case, max_seq_len=n))
        m.load_state_dict({k: v for k, v in i["p"].items() if k != "attn_norm.weight"})
        s.update(m=m.to(dt), x=i["x"], cos=i["cos"], sin=i["sin"], K=i.get("K"), V=i.get("V"))
    elif kind == "decode":
        from dual_mod_public_amd.decode import StaticTape
        sd = {k: v for k, v in i["p"].items() if k != "attn_norm.weight"}
        tape = StaticTape(_cfg(case, max_seq_len=case["P"]), case["B"], case["P"], device=DEV, dtype=dt, sd=sd)
        tape.K.copy_(i["K"])
        tape.V.copy_(i["V"])
        s.update(tape=tape, x=i["x"], cos=i["cos"], sin=i["sin"])
    elif kind == "prompt":
        from dual_mod_public_amd.graph_decode import GraphDecoder
        s.update(dec=GraphDecoder(_lm(case, i["sd"]), case["B"], case["P"]).capture(), tok=i["tok"])
    elif kind == "trunk":
        from dual_mod_public_amd.trunk import HipTrunk
        m = _lm(case, i["sd"], case["ffn"])
        tr = HipTrunk(m, case["B"], case["T"], schedule=_schedule(case["T"], case["c"], case["K"]),
                      wavefront=case["wavefront"])
        s.update(tr=tr, idx=i["idx"], targets=i["targets"])
    else:
        from dual_mod_public_amd.stack import HipLayerStack
        st = HipLayerStack(_cfg(case, max_seq_len=case["T"]), case["layers"], case["B"], case["T"],
                           schedule=_schedule(case["T"], case["c"], case["K"]), device=DEV, dtype=dt, wavefront=True)
        st.load(i["ps"], i["cos"], i["sin"])
        s.update(st=st, x=i["x"], dy=i["dy"])
    torch.cuda.synchronize()
    return s


def run(s):
    kind, case = s["kind"], s["case"]
    if kind == "train":
        c, g = s["cell"], s["grads"]
        c.layer_forward(s["x"], s["y"], s["cos"], s["sin"], s["sched"], s["K"], s["V"], s["ocat"], s["bufs"],
                        tape=s["tape"])
        g.zero_()
        c.layer_backward(s["x"], s["dy"], s["dx"], s["cos"], s["sin"], s["sched"], s["K"], s["V"], s["ocat"],
                         s["bufs"], g, tape=s["tape"])
        return dict(y=s["y"], dx=s["dx"], **{"d_" + k: v for k, v in g.t.items()})
    if kind == "autograd":
        from dual_mod_public_amd.autograd import dm_layer
        y = dm_layer(s["x"], s["cell"], s["params"], s["cos"], s["sin"], s["sched"])
        gr = torch.autograd.grad(y, [s["x"], *s["params"].values()], s["dy"])
        return dict(y=y.detach(), dx=gr[0], **{"d_" + k: v for k, v in zip(s["params"], gr[1:])})
    if kind == "module":
        with torch.no_grad():
            return s["m"](s["x"], s["cos"], s["sin"])
    if kind == "chunk":
        from dual_mod_public_amd.engine import chunk_cell_forward
        a = case["a"]
        with torch.no_grad():
            o, k, v = chunk_cell_forward(s["m"], s["x"], s["cos"][a:], s["sin"][a:], s["K"][:, :, :a],
                                         s["V"][:, :, :a], case["K"])
        return dict(o=o, k=k, v=v)
    if kind == "decode":
        t, pos = s["tape"], case["pos"]
        o, y = t.step(s["x"], pos, s["cos"], s["sin"], with_wo=True)
        # the step's outputs: the rows, and the slot of the tape it wrote
        return dict(o=o, y=y, k=t.K[:, :, pos], v=t.V[:, :, pos])
    if kind == "prompt":
        dec = s["dec"]
        dec.reset()
        out = []
        for p in range(case["n"]):
            dec.tok.copy_(s["tok"][:, p:p + 1])
            dec.step()
            out.append(dec.logits[:, 0].clone())
        return torch.stack(out, 1)
    if kind == "trunk":
        loss = s["tr"].train_step(s["idx"], s["targets"])
        return dict(loss=loss, **{"d_" + k: v for k, v in s["tr"].grad.items()})
    y, dx, grads = s["st"].step(s["x"], s["dy"])
    return dict(y=y, dx=dx, grads=s["st"].flat)   # every layer's gradients, in the buffer's order


# ---------------------------------------------------------------------------------------------
# the work a pass cannot do without
# ---------------------------------------------------------------------------------------------

def _nmats(mod):
    """Square d x d weight matrices of one layer: (projection, sweep GEMM 1, sweep GEMM 2)."""
    return (5, 4, 0) if mod == "linear" else (6, 4, 1)


def _layer_flops(case, T, c, K, a=0, wo=True):
    """Forward FLOPs per sequence of a layer over T rows in chunks of c, K sweeps, a rows before."""
    d = case["d"]
    npj, n1, n2 = _nmats(case["mod"])
    f = 2.0 * T * d * d * (npj + (1 if wo else 0)) + 2.0 * T * K * d * d * (n1 + n2)
    W = case.get("window", 0) or 10 ** 9
    comm = sum(min(p + a, W) * min(c, T - p) for p in range(0, T, c))     # committed (row, key) pairs
    intra = sum(min(c, T - p) * (min(c, T - p) + 1) / 2 for p in range(0, T, c))
    return f + 4.0 * d * (comm + K * intra)


def work(case):
    d, B, kind, mod = case["d"], case["B"], case["kind"], case["mod"]
    e = 4 if case.get("dtype") == "fp32" else 2
    wts = (sum(_nmats(mod)) + 1) * d * d                                   # elements of a layer's matrices
    if kind in ("train", "autograd", "stack"):
        n = case.get("layers", 1)
        f = 3.0 * n * B * _layer_flops(case, case["T"], case["c"], case["K"])
        x = B * case["T"] * d * e
        return dict(bytes=4.0 * x + n * wts * (e + 4), flops=f)
    if kind == "module":
        return dict(bytes=2.0 * B * case["T"] * d * e + wts * e,
                    flops=B * _layer_flops(case, case["T"], 64, min(64, case["T"])))
    if kind == "chunk":
        rd = 2.0 * B * case["a"] * d * e + 4.0 * B * case["c"] * d * e + (wts - d * d) * e
        return dict(bytes=rd, flops=B * _layer_flops(case, case["c"], case["c"], case["K"], case["a"], wo=False))
    if kind == "decode":
        P = min(case["pos"], case["window"] - 1) if case["window"] else case["pos"]
        return dict(bytes=2.0 * B * P * d * e + wts * e + 5.0 * B * d * e, flops=B * (2.0 * wts + 4.0 * d * P))
    if kind == "prompt":
        ffn = _ffn_default(d)
        w = case["layers"] * (wts + 3 * d * ffn) + case["vocab"] * d
        n = case["n"]
        return dict(bytes=n * (2.0 * w + 4.0 * B * case["vocab"]) + case["layers"] * 2.0 * B * d * n * n,
                    flops=2.0 * n * B * w)
    M = B * case["T"]
    f = 3.0 * case["layers"] * (B * _layer_flops(case, case["T"], case["c"], case["K"])
                                + 6.0 * M * d * case["ffn"]) + 6.0 * M * d * case["vocab"]
    nw = case["layers"] * (wts + 3 * d * case["ffn"]) + case["vocab"] * d
    return dict(bytes=6.0 * nw + 8.0 * M * d, flops=f)


def tolerance(case):
    """About four times the largest distance between a pass and ``exact`` measured over a kind's
    outputs (fp32: 1.3e-6; bf16: 0.003 for a step's rows, 0.004 for the exact scan, 0.012 for the
    gradients of a layer, 0.011 for the logits of 24 layers)."""
    if case.get("dtype") == "fp32":
        return {"rel": 6e-6}
    if case["kind"] in ("decode", "chunk", "module"):
        return {"rel": 1.4e-2}
    return {"rel": 3e-2}


# the order of a layer's gradients in HipLayerStack's flat buffer
GRAD_ORDER = ["wq.weight", "wk.weight", "wv.weight", "wo.weight", "w_kctx.weight", "w_vctx.weight", "w_gk.weight",
              "w_gv.weight", "w_gk.bias", "w_gv.bias", "norm_ctx.weight", "attn_norm.weight", "v_pre.weight",
              "v_gate.weight", "v_gate.bias", "v_map.weight"]


# ---------------------------------------------------------------------------------------------
# the same in 64 bits
# ---------------------------------------------------------------------------------------------

def _rms(x, w):
    return x * torch.rsqrt(x.pow(2).mean(-1, keepdim=True) + EPS) * w


def _rot(x, cos, sin):
    a, b = x.chunk(2, -1)
    return torch.cat([a * cos - b * sin, b * cos + a * sin], -1)


def _heads(x, h):
    return x.reshape(x.shape[0], x.shape[1], h, -1).transpose(1, 2)


def _merge(x):
    return x.transpose(1, 2).flatten(2)


def _refine(case, p, xhat, o, k, v):
    """Refined (unrotated) key and value rows from the attention output o of the same rows."""
    u = _rms(o, p["norm_ctx.weight"])
    xu = torch.cat([xhat, u], -1)
    gk = torch.sigmoid(F.linear(xu, p["w_gk.weight"], p["w_gk.bias"]))
    gv = torch.sigmoid(F.linear(xu, p["w_gv.weight"], p["w_gv.bias"]))
    vin = u
    if case["mod"] in ("mult", "mult_res"):
        vin = (torch.sigmoid(F.linear(xhat, p["v_gate.weight"], p["v_gate.bias"]))
               * torch.tanh(F.linear(u, p["v_map.weight"])))
        if case["mod"] == "mult_res":
            vin = u + vin
    elif case["mod"] == "fusion":
        vin = u + F.silu(F.linear(xu, p["v_pre.weight"]))
    return (gk * k + (1 - gk) * F.linear(u, p["w_kctx.weight"]),
            gv * v + (1 - gv) * F.linear(vin, p["w_vctx.weight"]))


def _cells(case, p, xhat, cos, sin, sched, K0=None, V0=None):
    """The chunked scan: o rows, and the refined rows of every chunk, against committed K0 / V0."""
    h = case["h"]
    dh = case["d"] // h
    W = case.get("window", 0)
    sc = 1.0 / math.sqrt(dh)
    q = _rot(_heads(F.linear(xhat, p["wq.weight"]), h), cos, sin)
    k, v = F.linear(xhat, p["wk.weight"]), F.linear(xhat, p["wv.weight"])
    ks, vs = _rot(_heads(k, h), cos, sin), _heads(v, h)
    Kc = q[:, :, :0] if K0 is None else K0
    Vc = q[:, :, :0] if V0 is None else V0
    outs, Kn, Vn = [], [], []
    for p0, c, n in sched:
        r = slice(p0, p0 + c)
        P = Kc.shape[2]
        i = torch.arange(c, device=DEV)[:, None]
        keep = torch.arange(c, device=DEV)[None] < i
        com = (q[:, :, r] @ Kc.transpose(-1, -2)) * sc
        if W > 1:
            com = com.masked_fill(torch.arange(P, device=DEV)[None] < P + i - W + 1, float("-inf"))
            keep = keep & (i - torch.arange(c, device=DEV)[None] <= W - 1)
        slf = (q[:, :, r] * ks[:, :, r]).sum(-1, keepdim=True) * sc
        # the committed part's row maximum and sums do not change from sweep to sweep
        m = torch.cat([com, slf], -1).amax(-1, keepdim=True).detach()
        ec = torch.exp(com - m)
        zc, oc = ec.sum(-1, keepdim=True), ec @ Vc
        zc, oc = zc + torch.exp(slf - m), oc + torch.exp(slf - m) * vs[:, :, r]
        Ki, Vi = ks[:, :, r], vs[:, :, r]
        for _ in range(n):
            si = ((q[:, :, r] @ Ki.transpose(-1, -2)) * sc).masked_fill(~keep, float("-inf"))
            ei = torch.exp(si - m)
            o = _merge((oc + ei @ Vi) / (zc + ei.sum(-1, keepdim=True)))
            kk, vv = _refine(case, p, xhat[:, r], o, k[:, r], v[:, r])
            Ki, Vi = _rot(_heads(kk, h), cos[r], sin[r]), _heads(vv, h)
        outs.append(o)
        Kn.append(Ki)
        Vn.append(Vi)
        Kc, Vc = torch.cat([Kc, Ki], 2), torch.cat([Vc, Vi], 2)
    return torch.cat(outs, 1), torch.cat(Kn, 2), torch.cat(Vn, 2)


def _sublayer(case, p, x, cos, sin, sched):
    xhat = _rms(x, p["attn_norm.weight"])
    return x + F.linear(_cells(case, p, xhat, cos, sin, sched)[0], p["wo.weight"])


def _mlp(p, x):
    hh = _rms(x, p["mlp_norm.weight"])
    return x + F.linear(F.silu(F.linear(hh, p["mlp.w1.weight"])) * F.linear(hh, p["mlp.w3.weight"]),
                        p["mlp.w2.weight"])


def _split(sd, l):
    pre = f"blocks.{l}."
    b = {k[len(pre):]: v for k, v in sd.items() if k.startswith(pre)}
    return {k.replace("attn.", "", 1): v for k, v in b.items()}


def _lm64(case, sd, idx, sched):
    """The whole model in 64 bits: logits of every position."""
    dh = case["d"] // case["h"]
    cos, sin = (t.double() for t in _rope(idx.shape[1], dh))
    x = sd["tok_emb.weight"][idx]
    for l in range(case["layers"]):
        p = _split(sd, l)
        x = _mlp(p, _sublayer(case, p, x, cos, sin, sched))
    return F.linear(_rms(x, sd["norm_f.weight"]), sd["tok_emb.weight"])


def exact(case, seed):
    i, kind = _inputs(case, seed), case["kind"]
    up = lambda t: t.double()                                                  # noqa: E731
    if kind in ("train", "autograd"):
        p = {k: up(v).requires_grad_() for k, v in i["p"].items()}
        x = up(i["x"]).requires_grad_()
        y = _sublayer(case, p, x, up(i["cos"]), up(i["sin"]), _schedule(case["T"], case["c"], case["K"]))
        gr = torch.autograd.grad(y, [x, *p.values()], up(i["dy"]))
        return dict(y=y.detach(), dx=gr[0], **{"d_" + k: v for k, v in zip(p, gr[1:])})
    with torch.no_grad():
        if kind == "module":
            p = {k: up(v) for k, v in i["p"].items()}
            o = _cells(case, p, up(i["x"]), up(i["cos"]), up(i["sin"]), _schedule(case["T"], 64, 64))[0]
            return F.linear(o, p["wo.weight"])
        if kind == "chunk":
            p, a = {k: up(v) for k, v in i["p"].items()}, case["a"]
            o, k, v = _cells(case, p, up(i["x"]), up(i["cos"][a:]), up(i["sin"][a:]), [(0, case["c"], case["K"])],
                             up(i["K"][:, :, :a]), up(i["V"][:, :, :a]))
            return dict(o=o, k=k, v=v)
        if kind == "decode":
            p, pos, W = {k: up(v) for k, v in i["p"].items()}, case["pos"], case["window"]
            lo = max(0, pos - W + 1) if W > 1 else 0
            cs, sn = up(i["cos"][pos:pos + 1]), up(i["sin"][pos:pos + 1])
            os, ks, vs = [], [], []
            for b in range(case["B"]):   # row by row: a long tape is never held whole in 64 bits
                o, k, v = _cells(dict(case, window=0), p, up(i["x"][b:b + 1, None]), cs, sn, [(0, 1, 1)],
                                 up(i["K"][b:b + 1, :, lo:pos]), up(i["V"][b:b + 1, :, lo:pos]))
                os.append(o[:, 0])
                ks.append(k[:, :, 0])
                vs.append(v[:, :, 0])
            o = torch.cat(os)
            return dict(o=o, y=F.linear(o, p["wo.weight"]), k=torch.cat(ks), v=torch.cat(vs))
        if kind == "prompt":
            return _lm64(case, {k: up(v) for k, v in i["sd"].items()}, i["tok"], [(0, case["n"], case["n"])])
    if kind == "trunk":
        sd = {k: up(v).requires_grad_() for k, v in i["sd"].items()}
        lg = _lm64(case, sd, i["idx"], _schedule(case["T"], case["c"], case["K"]))
        loss = F.cross_entropy(lg.flatten(0, 1), i["targets"].flatten())
        gr = torch.autograd.grad(loss, list(sd.values()))
        return dict(loss=loss.detach(), **{"d_" + n: v for n, v in zip(sd, gr)})
    ps = [{k: up(v).requires_grad_() for k, v in p.items()} for p in i["ps"]]
    x = up(i["x"]).requires_grad_()
    y = x
    for p in ps:
        y = _sublayer(case, p, y, up(i["cos"]), up(i["sin"]), _schedule(case["T"], case["c"], case["K"]))
    flat = [(l, k, v) for l, p in enumerate(ps) for k, v in p.items()]
    gr = torch.autograd.grad(y, [x] + [v for _, _, v in flat], up(i["dy"]))
    by = {(l, k): v for (l, k, _), v in zip(flat, gr[1:])}
    return dict(y=y.detach(), dx=gr[0],
                grads=torch.cat([by[l, k].flatten() for l in range(len(ps)) for k in GRAD_ORDER if (l, k) in by]))
