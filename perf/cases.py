"""What is timed and compared when a kernel of this library changes: calls of a DeltaNet
layer's path through the package's public entry points, at the sizes a serving program makes
them -- one token, speculative verify blocks, short and long prompt windows -- and the whole
layer from in_proj to out_proj.

Sizes are the benchmark's: 16 k-heads and 48 v-heads of 128, 10240 conv channels, hidden
size 5120, 48 layers, prompt windows of up to 4096 tokens, verify blocks of 8 x 5 tokens.
A case is a dict of plain values; `kind` names the call (see prepare)."""
from __future__ import annotations

import math

import torch

import __graft_entry__

gdn = __graft_entry__.load_package()

D, HK, HV, HIDDEN = 128, 16, 48, 5120
C = (2 * HK + HV) * D
IN_ROWS = (C, HV * D, HV, HV)  # in_proj_qkv, in_proj_z, in_proj_a, in_proj_b
EPS = 1e-6
MAX_TOKENS = 4096


def listed():
    return [
        # one sequence generating: the recurrence of one layer, through the cache that holds
        # its state (fp32 o, as the gated norm behind it takes it)
        dict(name="decode_b1", kind="step", B=1, T=1, f32=True, fast=False),
        # the same step of a model's 48 DeltaNet layers in one launch
        dict(name="decode_48_layers", kind="layers", L=48, B=1, f32=False),
        # the reference's own call, delta::run: 32 sequences, q, k, v in fp32 and
        # head-expanded, gates computed by the caller
        dict(name="run_b32", kind="run", B=32, T=1, f32=True, collect=False),
        # speculative verify: 8 sequences of 5 tokens recorded, 3 of the 5 accepted
        dict(name="verify_b8_t5", kind="verify", B=8, T=5, n=3, f32=True),
        # a short prompt continued from a state
        dict(name="prefill_t100", kind="step", B=1, T=100, f32=True, fast=False),
        # four ragged prompts with q, k, v given, the fast precision, bf16 outputs
        dict(name="prefill_b4_t333_fast", kind="prefill", B=4, T=333, conv=False, f32=False, fast=True),
        # the longest prompt window
        dict(name="prefill_t4096", kind="prefill", B=1, T=4096, conv=True, f32=False, fast=False),
        # a generated token's four input projections
        dict(name="in_proj_m1", kind="in_proj", M=1),
        # a verify block's (8 x 5 rows)
        dict(name="in_proj_m40", kind="in_proj", M=40),
        # the gated norm and output projection of an odd prompt tail
        dict(name="out_proj_m333", kind="out_proj", M=333),
        # the input projections of the longest prompt window
        dict(name="in_proj_m4096", kind="in_proj", M=4096),
        # a whole DeltaNet layer over a 1024-token window: in_proj, the recurrence on its
        # cache, gated norm and out_proj
        dict(name="layer_t1024", kind="block", B=1, T=1024, fast=False),
    ]


def _log(rng, lo, hi):
    return min(hi, max(lo, int(math.exp(rng.uniform(math.log(lo), math.log(hi + 1))))))


def draw(rng):
    kind = rng.choice(["step", "step", "layers", "run", "verify", "prefill", "prefill", "in_proj", "in_proj",
                       "out_proj", "block"])
    f32, fast = rng.random() < 0.5, rng.random() < 0.4
    if kind == "step":
        T = 1 if rng.random() < 0.4 else _log(rng, 2, 1024)
        return dict(kind=kind, B=_log(rng, 1, max(1, min(32, MAX_TOKENS // T))), T=T, f32=f32, fast=fast)
    if kind == "layers":
        L = rng.randint(2, 48)
        return dict(kind=kind, L=L, B=_log(rng, 1, 4), f32=f32)
    if kind == "run":
        T = _log(rng, 1, 16)
        return dict(kind=kind, B=_log(rng, 1, max(1, 32 // T)), T=T, f32=f32, collect=rng.random() < 0.5)
    if kind == "verify":
        T = rng.randint(2, 8)
        return dict(kind=kind, B=_log(rng, 1, 16), T=T, n=rng.randint(0, T), f32=f32)
    if kind == "prefill":
        T = _log(rng, 16, MAX_TOKENS)
        return dict(kind=kind, B=_log(rng, 1, max(1, min(8, MAX_TOKENS // T))), T=T, conv=rng.random() < 0.7,
                    f32=f32, fast=fast)
    if kind == "block":
        return dict(kind=kind, B=_log(rng, 1, 4), T=_log(rng, 1, 512), fast=fast)
    return dict(kind=kind, M=_log(rng, 1, MAX_TOKENS))


# ---- inputs ----

def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _n(g, *shape):
    return torch.randn(shape, device="cuda", generator=g)


def _u(g, *shape):
    return torch.rand(shape, device="cuda", generator=g)


def _unit(g, *shape):
    x = _n(g, *shape)
    return x / x.norm(dim=-1, keepdim=True)


def _mat(g, n, k):
    """4-bit weights of standard deviation about 1/sqrt(k), quantized as a checkpoint's are:
    random nibbles, bf16 scales, and biases near each group's minimum."""
    w = torch.randint(-2 ** 31, 2 ** 31 - 1, (n, k // 8), dtype=torch.int32, device="cuda", generator=g)
    s = (0.5 + _u(g, n, k // 64)) / (4.6 * math.sqrt(k))
    b = -s * (7.0 + _u(g, n, k // 64))
    return gdn.QuantLinear(w, s.to(torch.bfloat16), b.to(torch.bfloat16))


def _gates(g, *rows):
    """a, b logits and the layer's A_log, dt_bias: decays from about 0.15 to 0.999 a token."""
    lead = rows[:1] if len(rows) == 3 else ()
    return dict(a=_n(g, *rows, HV).to(torch.bfloat16), b=_n(g, *rows, HV).to(torch.bfloat16),
                A_log=_u(g, *lead, HV) * 5 - 4, dt_bias=_n(g, *lead, HV) * 0.1)


def _x(g, *rows):
    return _n(g, *rows, C).to(torch.bfloat16)


def _conv(g, *lead):
    return (_n(g, *lead, 4, C) * 0.3).to(torch.bfloat16)


def _state(g, *lead):
    return _n(g, *lead, HV, D, D) * 0.02


def _tail(g, *lead):
    return _n(g, *lead, 3, C).to(torch.bfloat16)


def _cache(g, B, T, fast):
    """A layer's cache in the middle of a sequence, with a workspace for prompt blocks."""
    cache = gdn.DeltaCache(B, Hv=HV, Hk=HK, max_prefill_tokens=T,
                           prefill_precision=gdn.PREFILL_FAST if fast else gdn.PREFILL_ACCURATE)
    cache.state.copy_(_state(g, B))
    cache.conv.copy_(_tail(g, B))
    return cache


def _dtype(case):
    return torch.float32 if case["f32"] else torch.bfloat16


def prepare(case, seed):
    g = _gen(seed)
    kind = case["kind"]
    s = dict(case=case)
    if kind == "in_proj":
        s.update(mats=[_mat(g, n, HIDDEN) for n in IN_ROWS], x=_n(g, case["M"], HIDDEN).to(torch.bfloat16))
    elif kind == "out_proj":
        M, K = case["M"], HV * D
        s.update(mats=[_mat(g, HIDDEN, K)], o=_n(g, M, K) * 0.3, z=_n(g, M, K).to(torch.bfloat16),
                 gamma=_u(g, D) + 0.5)
    elif kind == "block":
        B, T = case["B"], case["T"]
        gates = _gates(g, B, 1)
        s.update(mats=[_mat(g, n, HIDDEN) for n in IN_ROWS], out=[_mat(g, HIDDEN, HV * D)], gamma=_u(g, D) + 0.5,
                 x=_n(g, B * T, HIDDEN).to(torch.bfloat16), conv_weight=_conv(g), A_log=gates["A_log"],
                 dt_bias=gates["dt_bias"], cache=_cache(g, B, T, case["fast"]))
    elif kind == "run":
        B, T = case["B"], case["T"]
        dt = _dtype(case)
        s.update(q=(_unit(g, B, T, HV, D) * D ** -0.5).to(dt), k=_unit(g, B, T, HV, D).to(dt),
                 v=_n(g, B, T, HV, D).to(dt), alpha=0.15 + 0.849 * _u(g, B, T, HV),
                 beta=torch.sigmoid(_n(g, B, T, HV)), S=_state(g, B))
    elif kind == "layers":
        L, B = case["L"], case["B"]
        s.update(_gates(g, L, B, 1), x=_x(g, L, B, 1), conv_weight=_conv(g, L), conv_in=_tail(g, L, B),
                 conv_out=torch.empty((L, B, 3, C), dtype=torch.bfloat16, device="cuda"), state=_state(g, L, B),
                 o=torch.empty((L, B, 1, HV, D), dtype=_dtype(case), device="cuda"))
        s["args"] = gdn.layer_args(B=B, T=1, Hk=HK, Hv=HV, n_layers=L, x=s["x"], conv_weight=s["conv_weight"],
                                   conv_state_in=s["conv_in"], conv_state_out=s["conv_out"], a=s["a"], b=s["b"],
                                   A_log=s["A_log"], dt_bias=s["dt_bias"], state_in=s["state"],
                                   state_out=s["state"], o=s["o"])
    elif kind == "prefill":
        B, T = case["B"], case["T"]
        s.update(_gates(g, B, T), state=_state(g, B))
        if case["conv"]:
            s.update(x=_x(g, B, T), conv_weight=_conv(g), conv_state=_tail(g, B))
        else:
            s.update(q=(_unit(g, B, T, HK, D) * D ** -0.5).to(torch.bfloat16),
                     k=_unit(g, B, T, HK, D).to(torch.bfloat16), v=_n(g, B, T, HV, D).to(torch.bfloat16))
        s["precision"] = gdn.PREFILL_FAST if case["fast"] else gdn.PREFILL_ACCURATE
        s["workspace"] = torch.empty(gdn.prefill_workspace_size(B, T, HK, HV, conv=case["conv"],
                                                                precision=s["precision"]),
                                     dtype=torch.uint8, device="cuda")
    else:  # step, verify
        B, T = case["B"], case["T"]
        s.update(_gates(g, B, T), x=_x(g, B, T), conv_weight=_conv(g),
                 cache=_cache(g, B, T if kind == "step" else 0, case.get("fast", False)))
    return s


def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "in_proj":
        return gdn.qlinear(s["mats"], s["x"])
    if kind == "out_proj":
        return gdn.qlinear(s["mats"], norm=(s["o"], s["z"], s["gamma"], EPS))
    if kind == "block":
        B, T, cache = case["B"], case["T"], s["cache"]
        qkv, z, a, b = gdn.qlinear(s["mats"], s["x"])
        o = cache.step(qkv.view(B, T, C), s["conv_weight"], a.view(B, T, HV), b.view(B, T, HV), s["A_log"],
                       s["dt_bias"], o_dtype=torch.float32)
        (y,) = gdn.qlinear(s["out"], norm=(o.view(B * T, HV * D), z, s["gamma"], EPS))
        return dict(y=y, state=cache.state, conv=cache.conv)
    if kind == "run":
        r = gdn.run(s["q"], s["k"], s["v"], s["alpha"], s["beta"], s["S"], collect=case["collect"])
        return dict(o=r.o, state=r.s_out, states=r.states)
    if kind == "layers":
        gdn.call_run(s["args"])
        return dict(o=s["o"], state=s["state"], conv=s["conv_out"])
    if kind == "prefill":
        r = gdn.prefill_chunked(x=s.get("x"), q=s.get("q"), k=s.get("k"), v=s.get("v"), a=s["a"], b=s["b"],
                                A_log=s["A_log"], dt_bias=s["dt_bias"], state=s["state"],
                                conv_weight=s.get("conv_weight"), conv_state=s.get("conv_state"),
                                o_dtype=_dtype(case), Hk=HK, Hv=HV, workspace=s["workspace"],
                                precision=s["precision"])
        return dict(o=r["o"], state=r["state"], conv=r["conv_state"] if case["conv"] else [])
    cache = s["cache"]
    cache.record = kind == "verify"
    o = cache.step(s["x"], s["conv_weight"], s["a"], s["b"], s["A_log"], s["dt_bias"], o_dtype=_dtype(case))
    if kind == "verify":
        cache.commit(case["n"])
    return dict(o=o, state=cache.state, conv=cache.conv)


# ---- what a pass cannot do without ----

def _proj_work(M, K, rows):
    return (sum(n * K // 2 + n * (K // 64) * 4 + M * n * 2 for n in rows), 2 * M * K * sum(rows))


def _layer_work(case, L, B, T, conv, o_bytes, states_written):
    state = L * B * HV * D * D * 4
    by = state * (1 + states_written) + L * (B * T * HV * (D * o_bytes + 4) + HV * 8)
    if conv:
        by += L * (B * T * C * 2 + 2 * B * 3 * C * 2 + 4 * C * 2)
    return by, L * B * T * HV * 6 * D * D  # k.S, the update, q.S


def work(case):
    kind = case["kind"]
    if kind == "in_proj":
        by, fl = _proj_work(case["M"], HIDDEN, IN_ROWS)
        return dict(bytes=by + case["M"] * HIDDEN * 2, flops=fl)
    if kind == "out_proj":
        by, fl = _proj_work(case["M"], HV * D, (HIDDEN,))
        return dict(bytes=by + case["M"] * HV * D * 6 + D * 4, flops=fl)
    B, T = case["B"], case.get("T", 1)
    if kind == "block":
        b1, f1 = _proj_work(B * T, HIDDEN, IN_ROWS)
        b2, f2 = _proj_work(B * T, HV * D, (HIDDEN,))
        inter = B * T * (sum(IN_ROWS)) * 2  # in_proj's outputs are not outputs of the layer
        state = 2 * B * HV * D * D * 4 + 2 * B * 3 * C * 2 + 4 * C * 2 + HV * 8
        return dict(bytes=b1 + b2 - inter + B * T * HIDDEN * 2 + D * 4 + state, flops=f1 + f2 + B * T * HV * 6 * D * D)
    o_bytes = 4 if case["f32"] else 2
    if kind == "run":
        el = 4 if case["f32"] else 2
        st = B * HV * D * D * 4
        by = st * (2 + (T if case["collect"] else 0)) + B * T * HV * (D * (3 * el + 4) + 8)
        return dict(bytes=by, flops=B * T * HV * 6 * D * D)
    if kind == "layers":
        by, fl = _layer_work(case, case["L"], B, 1, True, o_bytes, 1)
    elif kind == "verify":
        # every step's state is written: which one is kept is known only after the block
        by, fl = _layer_work(case, 1, B, T, True, o_bytes, T)
    elif kind == "prefill":
        by, fl = _layer_work(case, 1, B, T, case["conv"], o_bytes, 1)
        if not case["conv"]:
            by += B * T * (2 * HK + HV) * D * 2
    else:
        by, fl = _layer_work(case, 1, B, T, True, o_bytes, 1)
    return dict(bytes=by, flops=fl)


# ---- tolerances ----

def tolerance(case):
    kind = case["kind"]
    if kind in ("in_proj", "out_proj"):
        return dict(rel=7e-3)  # one bf16 rounding of the output: 1.7e-3 from exact
    if kind == "block":
        # bf16 between the steps, where a rounding may fall the other way: 2e-3 from exact
        return dict(rel=2e-2 if case["fast"] else 1e-2)
    if kind in ("step", "prefill") and case["T"] > 24:  # lengths the chunked form may take
        if case["fast"]:
            return dict(rel=1.4e-2)  # bf16 state products: 2.4e-3 (state), 3.4e-3 (outputs)
        return dict(rel=2.5e-3 if case["f32"] else 7e-3)  # bf16 operands in the readout: 6e-4
    if case["f32"]:
        return dict(rel=5e-4, max=0.1)  # fp32; a bf16 tie of the front end may fall the other way
    return dict(rel=7e-3)


# ---- the same values in 64 bits ----

def _rb(x):
    """Rounded to bf16: the path's own definition rounds here."""
    return x.to(torch.float32).to(torch.bfloat16).double()


def _exact_conv(x, tail, w, T):
    """Causal conv, SiLU, split, l2norm, q scale, each op rounded to bf16 as defined."""
    xp = torch.cat([tail, x], dim=-2).double()
    y = None
    for j in range(4):
        p = _rb(xp[..., j:j + T, :] * w[..., j, :].double().unsqueeze(-2).unsqueeze(-3) if w.dim() == 3
                else xp[..., j:j + T, :] * w[j].double())
        y = p if y is None else _rb(y + p)
    u = _rb(y * _rb(torch.sigmoid(y)))
    lead = u.shape[:-1]
    q, k, v = (u[..., :HK * D].reshape(*lead, HK, D), u[..., HK * D:2 * HK * D].reshape(*lead, HK, D),
               u[..., 2 * HK * D:].reshape(*lead, HV, D))

    def l2(t):
        ss = _rb(_rb(t * t).sum(-1, keepdim=True))
        den = _rb(ss + _rb(torch.tensor(1e-6, dtype=torch.float64, device=t.device)))
        return _rb(t * _rb(den.rsqrt()))

    scale = _rb(torch.tensor(D ** -0.5, dtype=torch.float64, device=x.device))
    return _rb(l2(q) * scale), l2(k), v, xp


def _exact_gates(s, a, b):
    A, dt = s["A_log"].double(), s["dt_bias"].double()
    if A.dim() == 2:
        A, dt = A[:, None, None], dt[:, None, None]
    t = a.double() + dt
    return torch.exp(-torch.exp(A) * torch.logaddexp(t, torch.zeros_like(t))), torch.sigmoid(b.double())


def _exact_steps(q, k, v, alpha, beta, S, keep=()):
    """The recurrence, token by token, over leading (.., T, H, D); `keep`: steps whose state to return too."""
    S = S.double()
    rep = v.shape[-2] // q.shape[-2]
    q, k, v = (t.double() for t in (q.repeat_interleave(rep, -2), k.repeat_interleave(rep, -2), v))
    T = q.shape[-3]
    o = torch.empty(v.shape, dtype=torch.float64, device=v.device)
    kept = {}
    for t in range(T):
        kt, qt, vt = k[..., t, :, :], q[..., t, :, :], v[..., t, :, :]
        at, bt = alpha[..., t, :, None], beta[..., t, :, None]
        kS = (S * kt.unsqueeze(-2)).sum(-1)
        S = at.unsqueeze(-1) * S + (bt * (vt - at * kS)).unsqueeze(-1) * kt.unsqueeze(-2)
        o[..., t, :, :] = (S * qt.unsqueeze(-2)).sum(-1)
        if t in keep:
            kept[t] = S
    return o, S, kept


def _exact_qlinear(x, m):
    shifts = torch.arange(0, 32, 4, device=x.device, dtype=torch.int32)
    n, g = m.scales.shape
    xd = x.double()
    y = torch.empty((x.shape[0], n), dtype=torch.float64, device=x.device)
    for r in range(0, n, 2048):
        w = ((m.w[r:r + 2048].unsqueeze(-1) >> shifts) & 15).reshape(-1, g, 64).double()
        w = w * m.scales[r:r + 2048].double().unsqueeze(-1) + m.biases[r:r + 2048].double().unsqueeze(-1)
        y[:, r:r + 2048] = xd @ w.reshape(w.shape[0], g * 64).t()
    return y


def _exact_norm(o, z, gamma):
    M, K = o.shape
    h = o.double().reshape(M, K // D, D)
    h = h * torch.rsqrt((h * h).mean(-1, keepdim=True) + EPS) * gamma.double()
    zd = z.double()
    return _rb(h.reshape(M, K) * zd * torch.sigmoid(zd))


def exact(case, seed):
    s = prepare(case, seed)
    kind = case["kind"]
    if kind == "in_proj":
        return [_exact_qlinear(s["x"], m) for m in s["mats"]]
    if kind == "out_proj":
        return [_exact_qlinear(_exact_norm(s["o"], s["z"], s["gamma"]), m) for m in s["mats"]]
    if kind == "run":
        T = case["T"]
        o, S, kept = _exact_steps(s["q"], s["k"], s["v"], s["alpha"].double(), s["beta"].double(), s["S"], range(T))
        return dict(o=o, state=S, states=[kept[t] for t in range(T)] if case["collect"] else [])
    B, T = case["B"], case.get("T", 1)
    if kind == "block":
        qkv, z, a, b = (_rb(_exact_qlinear(s["x"], m)) for m in s["mats"])
        cache = s["cache"]
        q, k, v, xp = _exact_conv(qkv.view(B, T, C), cache.conv.double(), s["conv_weight"], T)
        al, be = _exact_gates(s, a.view(B, T, HV), b.view(B, T, HV))
        o, S, _ = _exact_steps(q, k, v, al, be, cache.state)
        y = _exact_qlinear(_exact_norm(o.reshape(B * T, HV * D), z, s["gamma"]), s["out"][0])
        return dict(y=y, state=S, conv=xp[:, T:])
    al, be = _exact_gates(s, s["a"], s["b"])
    if kind == "prefill" and not case["conv"]:
        o, S, _ = _exact_steps(s["q"], s["k"], s["v"], al, be, s["state"])
        return dict(o=o, state=S, conv=[])
    if kind in ("layers", "prefill"):
        tail, S0 = (s["conv_in"] if kind == "layers" else s["conv_state"]), s["state"]
    else:
        tail, S0 = s["cache"].conv, s["cache"].state
    q, k, v, xp = _exact_conv(s["x"], tail, s["conv_weight"], T)
    n = case["n"] if kind == "verify" else T
    o, S, kept = _exact_steps(q, k, v, al, be, S0, (n - 1,))
    return dict(o=o, state=kept[n - 1] if n else S0.double(), conv=xp[..., n:n + 3, :])
