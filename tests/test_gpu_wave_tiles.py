"""The few-row forms against the forms they replace, bit for bit: a row's result does not depend on how
many rows a launch holds (every output sums its k in the same order), so the wave-tile products of few
rows must equal the same rows inside a larger call, exact cells run row by row must equal whole
Jacobi sweeps at K = c (which the tape keeps), and a short tape read in one launch must equal the split
read."""

from types import SimpleNamespace

import pytest
import torch

from dual_mod_public_amd import _lib as L
from dual_mod_public_amd.attention import DualModAttention
from dual_mod_public_amd.decode import StaticTape
from dual_mod_public_amd.engine import HipSweepCell, uniform_chunks
from dual_mod_public_amd.rope import build_rope_cache
from dual_mod_public_amd.synthetic import make_state_dict
from dual_mod_public_amd.trunk import MlpBufs, MlpWeights
from tests.hip_helpers import DEV, cfg_of, say

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _gpu():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    L.load()


def _rand(*shape, seed):
    g = torch.Generator(device=DEV).manual_seed(seed)
    return torch.randn(*shape, generator=g, device=DEV).bfloat16()


def _sd(cfg):
    return {k: v.to(DEV, torch.bfloat16) for k, v in make_state_dict(cfg, seed=5).items()}


def _same(a, b, what):
    torch.cuda.synchronize()
    assert torch.equal(a, b), f"{what}: {(a.float() - b.float()).abs().max().item():.3g} apart"


# B rows per step: one and several row tiles; T: whole chunks and a ragged last one
@pytest.mark.parametrize("B,T", [(1, 64), (2, 70), (9, 65), (17, 96), (33, 20)])
@pytest.mark.parametrize("mod,d,h,kw", [("mult_res", 256, 4, {}), ("linear", 256, 4, dict(local_window=9)),
                                        ("fusion", 512, 4, {}), ("mult", 256, 2, dict(v_clamp_tau=0.5))])
def test_exact_rows_equal_sweeps(B, T, mod, d, h, kw):
    say(f"exact rows B={B} T={T} {mod} d={d} h={h} {kw}")
    cfg = cfg_of(d, h, mod, T, **kw)
    cell = HipSweepCell(cfg, B, T, device=DEV, dtype=torch.bfloat16).pack(_sd(cfg))
    x = _rand(B, T, d, seed=B + T)
    cos, sin = (t.to(DEV) for t in build_rope_cache(T, cfg.head_dim, cfg.rope_theta))
    sched = uniform_chunks(T, 64)
    out = []
    for tape in (None, cell.new_tape(sched)):
        K = torch.full((B, h, T, cfg.head_dim), float("nan"), device=DEV, dtype=torch.bfloat16)
        V, ocat, y = K.clone(), torch.empty_like(x), torch.empty_like(x)
        cell.layer_forward(x, y, cos, sin, sched, K, V, ocat, cell.new_bufs(T), tape=tape)
        out.append((y, K, V, ocat))
    for a, b, what in zip(*out, ("y", "K", "V", "ocat")):
        _same(a, b, what)


# rows of the small call: edges of the 8-, 16- and 32-row tiles and of the wave-tile range
@pytest.mark.parametrize("n", [1, 8, 9, 16, 17, 32, 33, 63, 64, 65, 130, 256])
@pytest.mark.parametrize("mod,d,h", [("mult_res", 256, 4), ("linear", 1024, 16), ("fusion", 512, 4), ("mult", 1024, 8),
                                     ("mult_res", 2048, 32)])
def test_refine_rows_equal_larger_call(n, mod, d, h):
    say(f"refine rows n={n} {mod} d={d} h={h}")
    N = 320
    cfg = cfg_of(d, h, mod, N)
    m = DualModAttention(cfg)
    m.load_state_dict({k: v for k, v in _sd(cfg).items() if k != "attn_norm.weight"})
    m = m.to(DEV, torch.bfloat16)
    x, o, k, v = (_rand(1, N, d, seed=s) for s in (1, 2, 3, 4))
    with torch.no_grad():
        Ka, Va = m.refine_kv(x, o, k, v)
        Kb, Vb = m.refine_kv(*(t[:, :n].contiguous() for t in (x, o, k, v)))
    _same(Ka[:, :n], Kb, "K")
    _same(Va[:, :n], Vb, "V")


@pytest.mark.parametrize("T", [1, 8, 13, 16, 32, 40, 64, 100, 256])
@pytest.mark.parametrize("d,h", [(256, 4), (1024, 8), (1024, 16), (2048, 16), (2304, 36)])
def test_projection_rows_equal_larger_call(T, d, h):
    say(f"projection rows T={T} d={d} h={h}")
    N = 512
    cfg = cfg_of(d, h, "mult_res", N)
    cell = HipSweepCell(cfg, 1, N, device=DEV, dtype=torch.bfloat16).pack(_sd(cfg))
    cos, sin = (t.to(DEV) for t in build_rope_cache(N, cfg.head_dim, cfg.rope_theta))
    x = _rand(1, N, d, seed=7)
    a = cell.layer_proj(x, cell.new_bufs(N), cos, sin)
    b = cell.layer_proj(x[:, :T].contiguous(), cell.new_bufs(T), cos, sin)
    for n in ("xhat", "qr", "kraw", "kself", "vraw", "glogx", "sig"):
        ta, tb = getattr(a, n), getattr(b, n)
        _same(ta[:, :, :T] if ta.dim() == 4 else ta[:, :T], tb, n)


# A step at a host position reads at most 512 keys (head_dim 64: 1024) in one launch, in a quarter of the passes
# up to 128; at a device position the launch covers the whole tape, here five splits: the split grid. Keys at the
# edges of the passes, the splits and the rule; with a window also where it cuts the first split.
@pytest.mark.parametrize("P", [1, 127, 128, 129, 511, 512, 513, 640, 1024, 1025, 1600])
@pytest.mark.parametrize("W", [0, 600])
@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("d,h", [(256, 4), (512, 4)])
def test_short_read_equals_split_read(P, W, dt, d, h):
    say(f"short read P={P} W={W} {dt} d={d} h={h}")
    B, dh, T = 3, d // h, 2100
    cfg = cfg_of(d, h, "mult_res", T, local_window=W)
    sd = {k: v.to(DEV, dt) for k, v in make_state_dict(cfg, seed=5).items()}
    cos, sin = (t.to(DEV) for t in build_rope_cache(T, dh, cfg.rope_theta))
    tape = StaticTape(cfg, B, T, DEV, dt, sd=sd)
    tape.K.copy_(_rand(B, h, T, dh, seed=1))
    tape.V.copy_(_rand(B, h, T, dh, seed=2))
    x = _rand(B, d, seed=3).to(dt)
    host = tape.step(x, P, cos, sin)[0].clone()
    dev = tape.step(x, torch.tensor([P], device=DEV, dtype=torch.int32), cos, sin)[0]
    _same(host, dev, "o")


# mlp widths whose last k step is a half one (H = 32 mod 64), rows at the tiles' edges
@pytest.mark.parametrize("M", [1, 8, 9, 16, 17, 33, 64])
@pytest.mark.parametrize("d,H", [(128, 32), (512, 1376), (1024, 2752)])
def test_swiglu_rows_half_step(M, d, H):
    say(f"swiglu rows M={M} d={d} H={H}")
    x, w1, w3, w2 = (_rand(*s, seed=i) for i, s in enumerate([(M, d), (H, d), (H, d), (d, H)]))
    w1, w3, w2 = w1 * 0.05, w3 * 0.05, w2 * 0.05
    out = L.swiglu_rows(x, w1, w3, w2)
    torch.cuda.synchronize()
    g, u = x.float() @ w1.float().t(), x.float() @ w3.float().t()
    act = (torch.nn.functional.silu(g) * u).bfloat16().float()
    ref = act @ w2.float().t()
    # act and the output rounded to bf16 (2^-9 each, relative); act may round the other way where the
    # fp32 sums differ in the last bits: 4 * 2^-9
    err = ((out.float() - ref).norm() / ref.norm()).item()
    assert err < 4 * 2 ** -9, err


# a row's MLP output is the same in every batch: the split of each product's sum follows from its sizes alone
@pytest.mark.parametrize("d,H", [(128, 32), (512, 1376), (2048, 5504)])
def test_swiglu_rows_equal_in_every_batch(d, H):
    say(f"swiglu rows of 64 and of fewer, d={d} H={H}")
    x, w1, w3, w2 = (_rand(*s, seed=i) for i, s in enumerate([(64, d), (H, d), (H, d), (d, H)]))
    out = L.swiglu_rows(x, w1 * 0.05, w3 * 0.05, w2 * 0.05)
    for n in (1, 8, 9, 16, 17, 32, 33, 63):
        _same(L.swiglu_rows(x[:n].contiguous(), w1 * 0.05, w3 * 0.05, w2 * 0.05), out[:n], f"{n} rows")


# W_O and the MLP's down product sum eight chains of 32-wide steps (step j in chain j mod 8), its up products
# one chain per quarter of d: the rounding of these sums shows which. 2^24 swallows a 1 added to it.
@pytest.mark.parametrize("M", [1, 9, 17, 33, 64])
@pytest.mark.parametrize("K", [512, 1536])
def test_row_product_sum_order(M, K):
    say(f"order of the row products' sums, M={M} K={K}")
    bf = dict(device=DEV, dtype=torch.bfloat16)
    a, w = torch.zeros(K, **bf), torch.zeros(K, **bf)
    a[0] = a[256] = w[0] = 2.0 ** 12
    w[256] = -(2.0 ** 12)
    a[32:256:32] = w[32:256:32] = 1.0                     # steps 1 .. 7
    # W_O: a step without past rows returns its own value row, here x-hat itself
    cfg = cfg_of(K, K // 64, "mult_res", 8)
    sd = dict(_sd(cfg), **{"wv.weight": torch.eye(K, **bf), "wo.weight": w.expand(K, K).contiguous()})
    cos, sin = (t.to(DEV) for t in build_rope_cache(8, 64, cfg.rope_theta))
    y = StaticTape(cfg, M, 8, DEV, torch.bfloat16, sd=sd).step(a.expand(M, K).contiguous(), 0, cos, sin, with_wo=True)[1]
    _same(y, torch.full_like(y, 7.0), "W_O")
    # down: act = silu(64) * (a / 64)
    d = 128
    x, w1, w3 = torch.zeros(M, d, **bf), torch.zeros(K, d, **bf), torch.zeros(K, d, **bf)
    x[:, 0], w1[:, 0], w3[:, 0] = 1.0, 64.0, a / 64
    out = L.swiglu_rows(x, w1, w3, w.expand(d, K).contiguous())
    _same(out, torch.full_like(out, 7.0), "down")
    # up: 2^24 in the first quarter, 1 + 1 in the second, -2^24 in the third; the gate 64
    q, H = K // 4, 128
    x, w1, w3, w2 = (torch.zeros(*n, **bf) for n in ((M, K), (H, K), (H, K), (K, H)))
    x[:, 0], x[:, q], x[:, q + 32], x[:, 2 * q], x[:, K - 1] = 2.0 ** 12, 1.0, 1.0, -(2.0 ** 12), 1.0
    w3[:, 0], w3[:, q], w3[:, q + 32], w3[:, 2 * q], w1[:, K - 1] = 2.0 ** 12, 1.0, 1.0, 2.0 ** 12, 64.0
    w2[:, 0] = 1.0
    out = L.swiglu_rows(x, w1, w3, w2)
    _same(out, torch.full_like(out, 128.0), "up")


# dm_decode_step_norm against dm_decode_step and dm_residual_rmsnorm: the norm in GEMM 2's launch (bf16,
# B <= 64, no per-head norm), and where it follows the step (linear: one refine GEMM; B = 65; v_norm; fp32)
@pytest.mark.parametrize("dt,B,d,h,P0,kw", [
    (torch.bfloat16, 1, 256, 4, 0, {}), (torch.bfloat16, 9, 1024, 16, 700, dict(ctx_mod="mult")),
    (torch.bfloat16, 64, 512, 4, 520, dict(ctx_mod="fusion")), (torch.bfloat16, 3, 256, 4, 30, dict(ctx_mod="linear")),
    (torch.bfloat16, 65, 256, 4, 30, {}), (torch.bfloat16, 3, 256, 4, 30, dict(v_norm="rms")),
    (torch.float32, 5, 256, 4, 30, {})])
def test_step_norm_equals_two_calls(dt, B, d, h, P0, kw):
    say(f"decode step + norm in one call, {dt} B={B} d={d} P0={P0} {kw}")
    cfg = cfg_of(d=d, h=h, T=P0 + 4, **kw)
    dh = cfg.head_dim
    sd = {k: v.to(DEV, dt) for k, v in make_state_dict(cfg, seed=5).items()}
    cos, sin = (t.to(DEV) for t in build_rope_cache(P0 + 4, dh, 10000.0))
    tapes = [StaticTape(cfg, B, P0 + 4, DEV, dt, sd=sd) for _ in range(2)]
    for t in tapes:
        t.K.copy_(_rand(B, h, P0 + 4, dh, seed=1))
        t.V.copy_(_rand(B, h, P0 + 4, dh, seed=2))
    w = _rand(d, seed=3).float()
    xs = [_rand(B, d, seed=4).float() for _ in range(2)]
    for p in range(P0, P0 + 3):
        xh = _rand(B, d, seed=10 + p).to(dt)
        _, y = tapes[0].step(xh, p, cos, sin, with_wo=True)
        h0 = L.residual_rmsnorm(xs[0], y, w, dt)
        h1 = tapes[1].step_norm(xh, p, cos, sin, xs[1], w, torch.empty(B, d, device=DEV, dtype=dt), 1e-5)
        _same(h1, h0, "h")
        _same(xs[1], xs[0], "x")
    _same(tapes[1].K, tapes[0].K, "K tape")
    _same(tapes[1].V, tapes[0].V, "V tape")


# weight gradients whose row count is no multiple of the k-tile: whole k-tiles and the last rows by two launches
@pytest.mark.parametrize("M", [64, 65, 127, 130, 2049])
def test_weight_grad_last_rows(M):
    import ctypes
    say(f"weight gradients over M={M} rows")
    d, H, dt = 256, 384, torch.bfloat16
    blk = SimpleNamespace(mlp=SimpleNamespace(**{
        n: SimpleNamespace(weight=_rand(*s, seed=i) * 0.05)
        for i, (n, s) in enumerate([("w1", (H, d)), ("w3", (H, d)), ("w2", (d, H))])}),
        mlp_norm=SimpleNamespace(weight=_rand(d, seed=3)))
    mw = MlpWeights(d, H, DEV, dt)
    mw.pack(blk)
    mb = MlpBufs(1, M, d, H, DEV, dt)
    y, dz = _rand(M, d, seed=4), _rand(M, d, seed=5)
    z, dy = torch.empty_like(y), torch.empty_like(y)
    g = {k: torch.zeros(*s, device=DEV) for k, s in dict(w1=(H, d), w3=(H, d), w2=(d, H), norm_w=(d,)).items()}
    gs = L.dm_mlp_grads()
    for k in g:
        setattr(gs, k, L.ptr(g[k]))
    code = L.dtype_code(dt)
    L.check(L.lib().dm_mlp_fwd(code, ctypes.byref(mw.s), L.ptr(y), L.ptr(z), ctypes.byref(mb.s), M, d, H, 1e-5,
                               L.stream_ptr()))
    nb = L.lib().dm_mlp_workspace_bytes(code, M, d, H)
    ws = torch.empty(nb, device=DEV, dtype=torch.uint8)
    L.check(L.lib().dm_mlp_bwd(code, ctypes.byref(mw.s), L.ptr(y), L.ptr(dz), L.ptr(dy), ctypes.byref(mb.s),
                               ctypes.byref(gs), M, d, H, 1e-5, L.ptr(ws), nb, L.stream_ptr()))
    torch.cuda.synchronize()
    rows = lambda t: t.double().cpu().reshape(M, -1)
    dab, h = rows(mb.dab), rows(mb.h)
    w13 = (dab.t() @ h).reshape(-1, 2, 32, d)   # packed: 32 rows of w1, 32 of w3, ...
    for k, ref in (("w2", rows(dz).t() @ rows(mb.mid)), ("w1", w13[:, 0].reshape(H, d)),
                   ("w3", w13[:, 1].reshape(H, d))):
        err = ((g[k].double().cpu() - ref).norm() / ref.norm()).item()
        # fp32 sums of M exact products: at most M 2^-24 of sum |a b|, which is about sqrt(M) |sum a b|
        assert err < M ** 1.5 * 2 ** -24, (k, err)


# cross entropy rows and their gradient: vector rows, rows of no whole vectors, fewer columns than threads,
# ignored targets; against fp64
@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("M,V", [(1, 3), (5, 1000), (7, 2049), (33, 32000)])
def test_ce_rows(dt, M, V):
    say(f"cross entropy rows {dt} M={M} V={V}")
    x = (4 * _rand(M, V, seed=1).float()).to(dt)
    g = torch.Generator(device=DEV).manual_seed(2)
    t = torch.randint(0, V, (M,), generator=g, device=DEV)
    t[M // 2::3] = -1
    nv = (t >= 0).sum().clamp_min(1).float()
    leaf = x.double().cpu().requires_grad_(True)
    ref = torch.nn.functional.cross_entropy(leaf, t.cpu(), ignore_index=-1, reduction="none")
    (ref.sum() / nv.double().cpu()).backward()
    loss = L.ce_rows(x, t, nv)
    torch.cuda.synchronize()
    # fp32 sums of V exponentials (1 ulp each): 256 partial sums of V / 256 terms, then a tree
    tol = (V / 256 + 16) * 2 ** -23
    assert ((loss.double().cpu() - ref.detach()).abs() <= tol * (1 + ref.detach().abs())).all()
    d = (x.double().cpu() - leaf.grad).abs()
    rnd = 2 ** -8 if dt == torch.bfloat16 else 0.0   # the stored gradient's rounding
    # exp(x - lse): |x - lse| <= 64 rounded to 2^-19 absolute, then the sum's error
    assert (d <= leaf.grad.abs() * (rnd + tol + 2 ** -18) + 2 ** -22 / nv.item()).all(), d.max()


# infinities, NaN and both in a row: the loss and the gradient that torch gives
@pytest.mark.parametrize("V", [5, 2048, 2049])
def test_ce_rows_not_finite(V):
    say(f"cross entropy rows that are not finite, V={V}")
    inf, nan = float("inf"), float("nan")
    x = _rand(6, V, seed=1).float()
    x[0, 1], x[1, 1], x[2, 1] = inf, nan, -inf
    x[3, 1], x[3, V - 1] = inf, nan
    x[4, 1], x[4, 0] = nan, inf
    x[5] = -inf
    t = torch.full((6,), 2, device=DEV)
    leaf = x.double().cpu().requires_grad_(True)
    lse = torch.logsumexp(leaf, -1)
    ref = lse - leaf[:, 2]
    p = torch.exp(leaf - lse[:, None]).detach()
    p[:, 2] -= 1
    loss = L.ce_rows(x, t, torch.ones((), device=DEV))
    torch.cuda.synchronize()
    torch.testing.assert_close(loss.double().cpu(), ref.detach(), rtol=1e-5, atol=1e-5, equal_nan=True)
    torch.testing.assert_close(x.double().cpu(), p, rtol=1e-4, atol=1e-6, equal_nan=True)


# Embedding backward: repeated ids across the block's 256-token passes, one id for all, d beyond one pass and no
# multiple of the vector; above 4096 tokens by lists: ids of 1 to 256 tokens, frequent ones in pieces of 1024 and
# (70000 tokens) of 2048. Equal rows that no fp32 sum holds show how deep the sums are: one chain over the 4096
# rows of an id is 204 roundings off.
@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("rows", ["random", "equal"])
@pytest.mark.parametrize("M,d,n", [(1, 64, 5), (300, 128, 7), (700, 2176, 400), (513, 67, 1), (4096, 64, 1), (4097, 67, 50),
                                   (5000, 68, 3), (8192, 1100, 30), (5000, 260, 20000), (70000, 64, 300)])
def test_embed_bwd(dt, rows, M, d, n):
    say(f"embedding backward {dt} {rows} M={M} d={d} n={n}")
    dx = (_rand(M, d, seed=1) if rows == "random" else torch.full((M, d), 1 / 3, device=DEV)).to(dt)
    g = torch.Generator(device=DEV).manual_seed(2)
    idx = torch.randint(0, n, (M,), generator=g, device=DEV)
    if n == 300:   # every other token one id, the others from rare to frequent
        idx = torch.where(torch.rand(M, generator=g, device=DEV) < 0.5, 0, (idx.float() ** 2 / n).long())
    if n > 1000:
        idx[::3], idx[1::7] = -1, n   # left out
    out = _rand(n, d, seed=3).float()
    ok = ((idx >= 0) & (idx < n)).cpu()
    ref = out.double().cpu().index_add_(0, idx.cpu()[ok], dx.double().cpu()[ok])
    mag = out.abs().double().cpu().index_add_(0, idx.cpu()[ok], dx.abs().double().cpu()[ok])
    twice = out.clone()
    L.embed_bwd(dx, idx, out)
    L.embed_bwd(dx, idx, twice)
    _same(twice, out, "a second call")
    # additions a term goes through: its chain of 64, the chains of its block, the pieces, the gradient's
    span = M if M <= 4096 else 1024 * -(-M // 65536)
    depth = 64 + span // 64 + span // 256 + (0 if M <= 4096 else -(-M // span)) + 2
    assert ((out.double().cpu() - ref).abs() <= depth * 2 ** -24 * mag).all()


def test_captured_trunk_new_tokens():
    """A captured trunk step of 4096 tokens replayed with new ids each time, against eager steps between the
    replays (the ids are not sorted by a library call in the step), bit for bit."""
    from dual_mod_public_amd.trunk import HipTrunk
    from tests.test_gpu_trunk import _batch, _cfg, _model, _same as same_bits, _snapshot
    say("captured trunk, 4096 tokens, new ids per replay")
    cfg = _cfg(n_layers=1, max_seq_len=1024)
    B, T = 4, 1024
    m, _ = _model(cfg, torch.bfloat16)
    a, b = HipTrunk(m, B, T), HipTrunk(m, B, T)
    b.capture()
    for seed in (21, 22, 23, 24):
        idx, tg = (t.to(DEV) for t in _batch(cfg, B, T, seed=seed))
        a.train_step(idx, tg)
        b.train_step(idx, tg)
        torch.cuda.synchronize()
        assert same_bits(_snapshot(a), _snapshot(b)), seed
