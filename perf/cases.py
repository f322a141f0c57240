"""The work whose speed counts: calls of the gated-delta-net operators as a serving or a
training program makes them, from one decoded token to packed and long prefills.

Sizes are those of the repository's own workloads (``avelang_amd.workloads``: 16 qk-heads ->
32 v-heads, K = V = 128, T = 8192 / 65536, 64 packed sequences, 256 decoding sequences), that
shape split by heads over several GPUs, and ragged sizes in between.

Case fields
    kind      decode | spec | layer_decode | prefill | layer_prefill | train
    seqs      sequences (batch rows; with ``packed`` the packed sequences of one row)
    tokens    tokens per sequence (with ``packed`` the largest length, ``least`` the smallest)
    hqk, hv   qk-heads and v-heads;  k, v: head sizes
    l2        use_qk_l2norm_in_kernel;  gated: the gates formed inside the call
    h0        an initial state is given;  decay: scale of the log-decay (0: per-head rates as a
              layer's A_log / dt_bias give them)
"""
import math

import torch
import torch.nn.functional as F

import avelang_amd as ave
from avelang_amd import layer_ops
from avelang_amd import workloads

DEV = "cuda"
C = 64   # chunk of the 64-bit form below
CONV_W = 4


def listed():
    full = dict(hqk=16, hv=32, k=128, v=128)
    return [
        # one user's next token: the smallest call, all latency
        dict(name="decode_one", kind="decode", seqs=1, tokens=1, l2=True, gated=True, h0=True,
             decay=0.0, **full),
        # a full decode batch, state in place: streams 1.08 GB of state
        dict(name="decode_256", kind="decode", seqs=256, tokens=1, l2=False, gated=False, h0=True,
             decay=0.1, **full),
        # the linear-attention part of a layer for a serving batch: convolution update, split,
        # recurrence over a pool of state slots with the gates formed inside, gated norm
        dict(name="layer_decode_48", kind="layer_decode", seqs=48, tokens=1, l2=True, gated=True,
             h0=True, decay=0.0, **full),
        # speculative decoding: four draft tokens per sequence, a state kept after each
        dict(name="spec_24x4", kind="spec", seqs=24, tokens=4, l2=True, gated=False, h0=True,
             decay=0.1, **full),
        # a short ragged prompt
        dict(name="prefill_449", kind="prefill", seqs=1, tokens=449, packed=False, l2=True,
             gated=True, h0=False, decay=0.0, **full),
        # the headline prefill
        dict(name="prefill_8k", kind="prefill", seqs=1, tokens=8192, packed=False, l2=False,
             gated=False, h0=True, decay=0.1, **full),
        # 64 prompts of 128 .. 4096 tokens packed into one call
        dict(name="prefill_packed_64", kind="prefill", seqs=64, tokens=4096, least=128,
             packed=True, l2=False, gated=False, h0=True, decay=0.1, **full),
        # a long document
        dict(name="prefill_64k", kind="prefill", seqs=1, tokens=65536, packed=False, l2=False,
             gated=False, h0=True, decay=0.01, **full),
        # one GPU's heads of a layer split over eight, a ragged long prompt
        dict(name="prefill_shard_20k", kind="prefill", seqs=1, tokens=20011, packed=False, l2=True,
             gated=True, h0=True, decay=0.0, hqk=2, hv=4, k=128, v=128),
        # the linear-attention part of a layer in a prefill: convolution, split, gated delta
        # rule, gated norm
        dict(name="layer_prefill_4k", kind="layer_prefill", seqs=1, tokens=4096, packed=False,
             l2=True, gated=True, h0=False, decay=0.0, **full),
        # a training step of the operator: forward and every gradient, the gates' included
        dict(name="train_8k", kind="train", seqs=1, tokens=8192, packed=False, l2=True, gated=True,
             h0=False, decay=0.0, **full),
        # training on packed documents of ragged length
        dict(name="train_packed_6", kind="train", seqs=6, tokens=1500, least=100, packed=True,
             l2=False, gated=False, h0=False, decay=0.1, **full),
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["decode", "spec", "layer_decode", "prefill", "prefill", "prefill",
                       "layer_prefill", "train", "train"])
    hqk, hv = rng.choice([(16, 32), (16, 32), (8, 16), (4, 8), (2, 4), (16, 16), (4, 16)])
    k, v = rng.choice([(128, 128), (128, 128), (128, 128), (64, 64)])
    c = dict(kind=kind, hqk=hqk, hv=hv, k=k, v=v, l2=rng.random() < 0.5,
             gated=rng.random() < 0.5, h0=rng.random() < 0.6,
             decay=rng.choice([0.0, 0.1, 0.01]))
    if kind == "decode":
        c.update(seqs=_log_int(rng, 1, 256), tokens=1, h0=True)
    elif kind == "spec":
        c.update(seqs=_log_int(rng, 1, 64), tokens=rng.randint(2, 6), h0=True, gated=False)
    elif kind == "layer_decode":
        c.update(seqs=_log_int(rng, 1, 256), tokens=1, h0=True, gated=True, l2=True, decay=0.0)
    elif kind == "layer_prefill":
        c.update(seqs=1, tokens=_log_int(rng, 65, 16384), packed=False, h0=False, gated=True,
                 l2=True, decay=0.0)
    elif kind == "train":
        seqs = rng.choice([1, 1, 2, rng.randint(3, 8)])
        c.update(seqs=seqs, tokens=_log_int(rng, 130, 8192 // seqs), packed=False)
        if seqs > 2:
            c.update(packed=True, least=rng.randint(1, c["tokens"]))
    else:
        seqs = rng.choice([1, 1, 2, 4, rng.randint(3, 64)])
        if seqs > 2 and rng.random() < 0.6:
            hi = _log_int(rng, 64, min(4096, 131072 // seqs))
            c.update(seqs=seqs, tokens=hi, least=rng.randint(1, hi), packed=True)
        else:
            c.update(seqs=seqs, tokens=_log_int(rng, 65, 65536 // seqs), packed=False)
    if not c["gated"] and c["decay"] == 0.0:
        c["decay"] = 0.1
    return c


def _lengths(case):
    """Sequence lengths of a case (packed ones as workloads.varlen_cu_seqlens draws them)."""
    if not case.get("packed"):
        return [case["tokens"]] * case["seqs"]
    cu = workloads.varlen_cu_seqlens(case["seqs"], case["least"], case["tokens"], 0)
    return [int(b - a) for a, b in zip(cu[:-1], cu[1:])]


# ------------------------------------------------------------------ inputs ----
def prepare(case, seed):
    gen = torch.Generator(device=DEV)
    gen.manual_seed(int(seed))

    def randn(*shape):
        return torch.randn(shape, generator=gen, device=DEV, dtype=torch.float32)

    def rand(*shape):
        return torch.rand(shape, generator=gen, device=DEV, dtype=torch.float32)

    bf = torch.bfloat16
    kind, N, hqk, hv, K, V = (case[x] for x in ("kind", "seqs", "hqk", "hv", "k", "v"))
    lens = _lengths(case)
    packed = case.get("packed", False)
    B, T = (1, sum(lens)) if packed else (N, case["tokens"])
    s = dict(case=dict(case))
    if packed:
        cu = [0]
        for x in lens:
            cu.append(cu[-1] + x)
        s["cu"] = torch.tensor(cu, dtype=torch.int32, device=DEV)
    if case["gated"]:
        # a layer's parameters: exp(A_log) uniform up to 16, dt_bias the inverse softplus of a
        # step between 1e-3 and 1e-1, and the small projections' outputs
        dt = torch.exp(rand(hv) * (math.log(0.1) - math.log(0.001)) + math.log(0.001))
        s["A_log"] = torch.log(rand(hv) * 16 + 0.01)
        s["dt_bias"] = dt + torch.log(-torch.expm1(-dt))
        s["a"] = (0.5 * randn(B, T, hv)).to(bf)
        s["b"] = randn(B, T, hv).to(bf)
        if not case["decay"] == 0.0:   # rates of the synthetic workloads instead
            s["A_log"] = torch.full((hv,), math.log(case["decay"]), device=DEV)
            s["dt_bias"] = torch.zeros(hv, device=DEV)
    else:
        s["g"] = -case["decay"] * F.softplus(randn(B, T, hv))
        s["beta"] = torch.sigmoid(randn(B, T, hv))
    if kind in ("layer_decode", "layer_prefill"):
        D = 2 * hqk * K + hv * V
        s["conv_w"] = (0.5 * randn(D, CONV_W)).to(bf)
        s["norm_w"] = (1 + 0.1 * randn(V)).to(bf)
        s["x"] = randn(B, T, D).to(bf)
        s["z"] = randn(B, T, hv, V).to(bf)
    else:
        q, k = randn(B, T, hqk, K), randn(B, T, hqk, K)
        if not case["l2"]:
            q, k = (x * torch.rsqrt((x * x).sum(-1, keepdim=True) + 1e-6) for x in (q, k))
        s["q"], s["k"], s["v"] = q.to(bf), k.to(bf), randn(B, T, hv, V).to(bf)
    if kind in ("spec", "layer_decode"):
        # a pool with spare slots, the sequences' slots scattered over it
        per = case["tokens"] if kind == "spec" else 1
        slots = N * per + 16
        order = torch.randperm(slots, generator=gen, device=DEV).to(torch.int32)[:N * per]
        s["pool"] = 0.01 * randn(slots, hv, K, V)
        if kind == "spec":
            s["slots"] = order.reshape(N, per).contiguous()
            s["accepted"] = torch.randint(1, per + 1, (N,), generator=gen, device=DEV,
                                          dtype=torch.int32)
        else:
            s["slots"] = order
            s["conv_state"] = randn(slots, s["x"].shape[-1], CONV_W - 1).to(bf)
    elif case["h0"]:
        s["h0"] = 0.01 * randn(N, hv, K, V)
    if kind == "train":
        s["leaves"] = [n for n in ("q", "k", "v", "a", "b", "A_log", "dt_bias", "g", "beta", "h0")
                       if n in s]
        for n in s["leaves"]:
            s[n].requires_grad_(True)
        s["do"] = randn(B, T, hv, V).to(bf)
    return s


# -------------------------------------------------------------------- call ----
def _split(case, y):
    """The convolution's output as the layer cuts it into q, k and v heads."""
    hqk, hv, K, V = (case[x] for x in ("hqk", "hv", "k", "v"))
    B, T, _ = y.shape
    q, k, v = torch.split(y, [hqk * K, hqk * K, hv * V], dim=-1)
    return q.reshape(B, T, hqk, K), k.reshape(B, T, hqk, K), v.reshape(B, T, hv, V)


def _core(case, s, q, k, v, **kw):
    if case["gated"]:
        return ave.chunk_gated_delta_rule_gated(
            q, k, v, s["a"], s["b"], s["A_log"], s["dt_bias"], initial_state=s.get("h0"),
            cu_seqlens=s.get("cu"), use_qk_l2norm_in_kernel=case["l2"], **kw)
    return ave.chunk_gated_delta_rule(
        q, k, v, s["g"], s["beta"], initial_state=s.get("h0"), cu_seqlens=s.get("cu"),
        use_qk_l2norm_in_kernel=case["l2"], **kw)


def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "decode":
        if case["gated"]:
            return ave.fused_recurrent_gated_delta_rule_gated(
                s["q"], s["k"], s["v"], s["a"], s["b"], s["A_log"], s["dt_bias"],
                initial_state=s["h0"], output_final_state=True,
                use_qk_l2norm_in_kernel=case["l2"])
        return ave.fused_recurrent_gated_delta_rule(
            s["q"], s["k"], s["v"], s["g"], s["beta"], initial_state=s["h0"],
            output_final_state=True, use_qk_l2norm_in_kernel=case["l2"])
    if kind == "spec":
        return ave.fused_recurrent_gated_delta_rule(
            s["q"], s["k"], s["v"], s["g"], s["beta"], initial_state=s["pool"],
            output_final_state=True, use_qk_l2norm_in_kernel=case["l2"],
            ssm_state_indices=s["slots"], num_accepted_tokens=s["accepted"])
    if kind == "layer_decode":
        y = layer_ops.causal_conv1d_update(s["x"][:, 0], s["conv_state"], s["conv_w"],
                                           activation="silu", conv_state_indices=s["slots"])
        q, k, v = _split(case, y.unsqueeze(1))
        o, pool = ave.fused_recurrent_gated_delta_rule_gated(
            q, k, v, s["a"], s["b"], s["A_log"], s["dt_bias"], initial_state=s["pool"],
            output_final_state=True, use_qk_l2norm_in_kernel=True, ssm_state_indices=s["slots"])
        return layer_ops.rms_norm_gated(o, s["z"], s["norm_w"]), pool, s["conv_state"]
    if kind == "layer_prefill":
        y, conv_state = layer_ops.causal_conv1d_fn(s["x"].transpose(1, 2), s["conv_w"],
                                                   return_final_states=True, activation="silu")
        q, k, v = _split(case, y.transpose(1, 2))
        o, ht = _core(case, s, q, k, v, output_final_state=True)
        return layer_ops.rms_norm_gated(o, s["z"], s["norm_w"]), ht, conv_state
    if kind == "train":
        o, _ = _core(case, s, s["q"], s["k"], s["v"])
        return (o,) + torch.autograd.grad(o, [s[n] for n in s["leaves"]], s["do"])
    return _core(case, s, s["q"], s["k"], s["v"], output_final_state=True)


# ------------------------------------------------------------- what it costs ----
def work(case):
    kind, N, hqk, hv, K, V = (case[x] for x in ("kind", "seqs", "hqk", "hv", "k", "v"))
    tok = sum(_lengths(case))
    qkv = tok * (2 * hqk * K + hv * V) * 2
    gates = tok * hv * (4 if case["gated"] else 8)
    state = N * hv * K * V * 4
    o = tok * hv * V * 2
    # S^T k, the rank-one update and S^T q per token and v-head
    flops = 6.0 * K * V * tok * hv
    if kind == "spec":
        return dict(bytes=qkv + gates + o + state * (1 + case["tokens"]), flops=flops)
    if kind == "decode":
        return dict(bytes=qkv + gates + o + 2 * state, flops=flops)
    if kind in ("layer_decode", "layer_prefill"):
        # x in, z in, the normed output, the convolution's states and the core's
        conv = N * (2 * hqk * K + hv * V) * (CONV_W - 1) * 2
        both = 2 if kind == "layer_decode" else 1
        return dict(bytes=qkv + 2 * o + gates + both * (conv + state), flops=flops)
    if kind == "train":
        # q, k, v, the gates and do in; o and a gradient of each input out
        return dict(bytes=2 * (qkv + gates) + 2 * o + (2 * state if case["h0"] else 0),
                    flops=3 * flops)
    return dict(bytes=qkv + gates + o + state * (2 if case["h0"] else 1), flops=flops)


def tolerance(case):
    """Four times the distance from 64 bits seen on this path: bf16 outputs (2^-9 each) of
    products with fp16 / bf16 operands, q and k rounded to bf16 where they are normalised in
    the call, and one more bf16 tensor between the layer's operators."""
    if case["kind"] in ("decode", "spec"):
        return {"rel": 7e-3}                 # 1.7e-3 seen: the output's rounding alone
    if case["kind"] in ("layer_decode", "layer_prefill", "train"):
        return {"rel": 1.6e-2}               # up to 4.1e-3 and 3.8e-3 seen
    return {"rel": 1.2e-2}                   # up to 3.0e-3 seen


# ------------------------------------------------------------------ 64 bits ----
def _norm64(x):
    return x * torch.rsqrt((x * x).sum(-1, keepdim=True) + 1e-6)


def _gates64(case, s):
    if not case["gated"]:
        return s["g"].double(), s["beta"].double()
    x = s["a"].double() + s["dt_bias"].double()
    return (-torch.exp(s["A_log"].double()) * F.softplus(x), torch.sigmoid(s["b"].double()))


def _chunked64(q, k, v, g, beta, S):
    """The delta rule by chunks: q, k [N, H, T, K], v [N, H, T, V], g, beta [N, H, T] with T a
    multiple of C and g = beta = 0 on padding; S [N, H, K, V].  Returns o and the last state."""
    N, H, T, K = q.shape
    n = T // C
    q, k = (x.reshape(N, H, n, C, K) for x in (q, k))
    v = v.reshape(N, H, n, C, v.shape[-1])
    g, beta = g.reshape(N, H, n, C).cumsum(-1), beta.reshape(N, H, n, C)
    low = torch.ones(C, C, dtype=torch.bool, device=q.device).tril()
    gam = (g[..., :, None] - g[..., None, :]).masked_fill(~low, -math.inf).exp()
    kT = k.transpose(-1, -2).contiguous()
    A = (beta[..., None] * (k @ kT) * gam).tril(-1)
    P = K ** -0.5 * (q @ kT) * gam
    eye = torch.eye(C, dtype=q.dtype, device=q.device).expand_as(A)
    Tb = torch.linalg.solve_triangular(A + eye, eye, upper=False, unitriangular=True)
    Tb = Tb * beta[..., None, :]
    U = Tb @ v
    W = Tb @ (k * g.exp()[..., None])
    Q = q * (K ** -0.5 * g.exp())[..., None]
    last = g[..., -1:]
    D = (k * (last - g).exp()[..., None]).transpose(-1, -2).contiguous()
    out = []
    for c in range(n):
        d = U[:, :, c] - W[:, :, c] @ S
        out.append(Q[:, :, c] @ S + P[:, :, c] @ d)
        S = last[:, :, c].exp()[..., None] * S + D[:, :, c] @ d
    return torch.stack(out, 2).reshape(N, H, T, -1), S


def _prefill64(case, s, q, k, v, g, beta, h0):
    """Packed or batched [B, T, H, D] inputs in 64 bits -> o [B, T, Hv, V], final state."""
    lens = _lengths(case)
    N, hv, K, V = case["seqs"], case["hv"], case["k"], case["v"]
    rep = hv // case["hqk"]
    if case["l2"]:
        q, k = _norm64(q), _norm64(k)
    pad = -(-max(lens) // C) * C

    def rows(x, heads):
        parts = x[0].split(lens) if case.get("packed") else x.unbind(0)
        out = torch.stack([F.pad(p.flatten(1), (0, 0, 0, pad - p.shape[0])) for p in parts])
        out = out.reshape(N, pad, heads, -1).transpose(1, 2)
        return out.repeat_interleave(hv // heads, dim=1) if heads != hv else out

    hq = case["hqk"] if rep > 1 else hv
    S = h0 if h0 is not None else torch.zeros(N, hv, K, V, dtype=torch.float64, device=DEV)
    o, S = _chunked64(rows(q, hq), rows(k, hq), rows(v, hv), rows(g, hv)[..., 0],
                      rows(beta, hv)[..., 0], S)
    o = o.transpose(1, 2)
    if case.get("packed"):
        return torch.cat([o[i, :x] for i, x in enumerate(lens)])[None], S
    return o[:, :case["tokens"]], S


def _steps64(case, q, k, v, g, beta, S):
    """Token by token: q, k [N, T, Hqk, K], v [N, T, Hv, V], g, beta [N, T, Hv], S [N, Hv, K, V].
    Returns o and the states after every token."""
    rep = case["hv"] // case["hqk"]
    if case["l2"]:
        q, k = _norm64(q), _norm64(k)
    q, k = (x.repeat_interleave(rep, dim=2) for x in (q, k))
    out, states = [], []
    for t in range(q.shape[1]):
        S = S * g[:, t, :, None, None].exp()
        d = beta[:, t, :, None] * (v[:, t] - (S * k[:, t, :, :, None]).sum(-2))
        S = S + k[:, t, :, :, None] * d[:, :, None, :]
        out.append(case["k"] ** -0.5 * (S * q[:, t, :, :, None]).sum(-2))
        states.append(S)
    return torch.stack(out, 1), states


def _gated_norm64(x, z, w):
    x, z, w = x.double(), z.double(), w.double()
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + 1e-6) * w * F.silu(z)


def exact(case, seed):
    s = prepare(case, seed)
    kind = case["kind"]
    with torch.set_grad_enabled(kind == "train"):
        return _exact(case, s, kind)


def _exact(case, s, kind):
    if kind == "train":
        raw = [s[n].detach().double().requires_grad_(True) for n in s["leaves"]]
        d = {**s, **dict(zip(s["leaves"], raw))}
        g, beta = _gates64(case, d)
        o, _ = _prefill64(case, d, d["q"], d["k"], d["v"], g, beta, d.get("h0"))
        return (o.detach(),) + torch.autograd.grad(o, raw, s["do"].double())
    g, beta = _gates64(case, s)
    if kind in ("decode", "spec", "layer_decode"):
        if kind == "layer_decode":
            x, w = s["x"].double(), s["conv_w"].double()
            slots = s["slots"].long()
            past = torch.cat([s["conv_state"][slots].double(), x.transpose(1, 2)], -1)
            q, k, v = _split(case, F.silu((past * w).sum(-1))[:, None])
            conv_state = s["conv_state"].double()
            conv_state[slots] = past[..., 1:]
        else:
            q, k, v = (s[n].double() for n in "qkv")
        if kind == "decode":
            o, states = _steps64(case, q, k, v, g, beta, s["h0"].double())
            return o, states[-1]
        pool = s["pool"].double()
        if kind == "layer_decode":
            o, states = _steps64(case, q, k, v, g, beta, pool[slots])
            pool[slots] = states[-1]
            return _gated_norm64(o, s["z"], s["norm_w"]), pool, conv_state
        slots = s["slots"].long()
        first = slots.gather(1, (s["accepted"].long() - 1)[:, None])[:, 0]
        o, states = _steps64(case, q, k, v, g, beta, pool[first])
        for t, S in enumerate(states):
            pool[slots[:, t]] = S
        return o, pool
    if kind == "layer_prefill":
        x, w = s["x"].double(), s["conv_w"].double()
        past = F.pad(x.transpose(1, 2), (CONV_W - 1, 0))
        y = sum(past[..., j:j + x.shape[1]] * w[:, j, None] for j in range(CONV_W))
        q, k, v = _split(case, F.silu(y).transpose(1, 2))
        o, S = _prefill64(case, s, q, k, v, g, beta, None)
        return _gated_norm64(o, s["z"], s["norm_w"]), S, past[..., -(CONV_W - 1):]
    h0 = s["h0"].double() if case["h0"] else None
    return _prefill64(case, s, *(s[n].double() for n in "qkv"), g, beta, h0)
