"""The workloads the library's speed is judged by, each through a public entry point of kairos_gdn.

Two families of head dims: the Kairos 4B layer's own (dk = 256, dv = 512, 20 heads, always with the
in-op L2 norm and slow per-head decays) and the op's headline dims (dk = dv = 128, unit-norm q and k).
``listed()`` names the fixed cases, ``draw(rng)`` gives one more of the same ranges.
"""
import math
import os
import sys

import torch

_PKG = os.path.join(os.getcwd(), "kairos-sensenova_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

import kairos_gdn as kg  # noqa: E402

DEV = "cuda"
CHUNK = 64
BF16, F32, F64 = torch.bfloat16, torch.float32, torch.float64
DTYPES = {"bf16": BF16, "fp32": F32, "fp16": torch.float16, "fp8": BF16}


def _case(kind, K, V, H, T, B=1, dtype="bf16", l2=False, carry=True, lens="", form=""):
    """carry: an initial state goes in (every streamed or split call hands one on); lens: packed
    sequence lengths (T is then their sum); form: which public calls a layer pass goes through."""
    return {"kind": kind, "K": K, "V": V, "H": H, "B": B, "T": T, "dtype": dtype, "l2": l2, "carry": carry,
            "lens": lens, "form": form}


def _packed(lens):
    return ",".join(str(n) for n in lens)


def listed():
    cases = {
        # the op in fp32 at its smallest documented size: a parity or debugging run, latency bound
        "op_fp32_small": _case("op", 64, 64, 4, 512, dtype="fp32", carry=False),
        # a whole 480P clip (21 latent frames of 1560 tokens) in one call at the headline head dims
        "op_clip": _case("op", 128, 128, 20, 32760),
        # clips of 1, 4, 8 and 21 frames packed into one varlen call
        "op_varlen": _case("op", 128, 128, 20, 53040, lens="1560,6240,12480,32760"),
        # one frame of a streaming rollout, 8 streams, fp8 q and k with per-head scales
        "op_stream_fp8": _case("op", 128, 128, 20, 1560, B=8, dtype="fp8"),
        # a training step of the op at the headline head dims: forward and backward through autograd
        "op_train": _case("train", 128, 128, 20, 8192),
        # a layer's inference call as the model makes it: a clip in eight sub-calls that hand the state on
        "layer_subcall": _case("op", 256, 512, 20, 4095, l2=True),
        # the whole clip in one call at the layer's head dims
        "layer_clip": _case("op", 256, 512, 20, 32760, l2=True, carry=False),
        # the same clip on one rank of four that split the layer's heads
        "layer_tp_clip": _case("op", 256, 512, 5, 32760, l2=True, carry=False),
        # clips of ragged lengths packed into one call at the layer's head dims
        "layer_varlen": _case("op", 256, 512, 20, 11047, lens="1560,37,3121,6329", l2=True),
        # a training step of the layer's op: five frames, forward and backward through autograd
        "layer_train": _case("train", 256, 512, 20, 7800, l2=True),
        # decoding: one token for each of eight streams through the short-sequence mode
        "layer_decode": _case("decode", 256, 512, 20, 1, B=8, l2=True),
        # one streamed frame through everything between a layer's projections: three short convolutions
        # with caches, gates, the op and the gated output norm
        "layer_mixer_frame": _case("mixer", 256, 512, 20, 1560, l2=True, form="modules"),
    }
    return [dict(c, name=n) for n, c in cases.items()]


_MOST_FWD, _MOST_FP32 = 655200, 40960                             # token-heads a drawn forward may have


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["op", "op", "layer", "layer", "varlen", "layer_varlen", "stream", "train", "layer_train",
                       "decode", "mixer"])
    if kind == "op":
        K, V = rng.choice([(128, 128), (128, 128), (64, 64), (64, 128)])
        dtype = rng.choice(["bf16", "bf16", "bf16", "fp32", "fp16"])
        H, B = rng.choice([4, 5, 8, 10, 16, 20]), rng.choice([1, 1, 1, 2, 4])
        most = min(32760, (_MOST_FWD if dtype == "bf16" else _MOST_FP32) // (H * B))
        return _case("op", K, V, H, _log_int(rng, 65, most), B=B, dtype=dtype, l2=rng.random() < 0.5,
                     carry=rng.random() < 0.5)
    if kind == "layer":
        H, B = rng.choice([5, 10, 20]), rng.choice([1, 1, 2])
        return _case("op", 256, 512, H, _log_int(rng, 65, min(32760, _MOST_FWD // (H * B))), B=B, l2=True,
                     carry=rng.random() < 0.5)
    if kind in ("varlen", "layer_varlen"):
        n = rng.randint(2, 8)
        lens = [_log_int(rng, 1, 32760 // n) for _ in range(n)]
        if kind == "varlen":
            return _case("op", 128, 128, 20, sum(lens), lens=_packed(lens), l2=rng.random() < 0.5)
        return _case("op", 256, 512, rng.choice([5, 10, 20]), sum(lens), lens=_packed(lens), l2=True)
    if kind == "stream":
        return _case("op", 128, 128, 20, rng.randint(390, 1560), B=rng.randint(1, 8), dtype="fp8")
    if kind == "train":
        H, B = rng.choice([10, 20]), rng.choice([1, 2])
        return _case("train", 128, 128, H, _log_int(rng, 500, 163840 // (H * B)), B=B, l2=rng.random() < 0.5,
                     carry=rng.random() < 0.5)
    if kind == "layer_train":
        H = rng.choice([5, 10, 20])
        return _case("train", 256, 512, H, _log_int(rng, 500, 7800), l2=True, carry=rng.random() < 0.5)
    if kind == "decode":
        K, V = rng.choice([(256, 512), (256, 512), (128, 128)])
        return _case("decode", K, V, rng.choice([5, 20]), rng.choice([1, 1, 1, 3, 17, 64]), B=rng.randint(1, 16),
                     l2=True)
    K, V = rng.choice([(256, 512), (256, 512), (128, 128)])
    return _case("mixer", K, V, rng.choice([5, 20]), _log_int(rng, 65, 4095), l2=True,
                 form=rng.choice(["modules", "norm_call", "conv_call"]))


def _lens(case):
    return [int(x) for x in case["lens"].split(",")] if case["lens"] else None


def _layer_gates(n, H, gen):
    """The layer's decay parameters at initialisation: A ~ U(0, 16), dt log-uniform in [1e-3, 1e-1]."""
    A = torch.empty(H, device=DEV).uniform_(0.05, 16, generator=gen)
    dt = torch.exp(torch.empty(H, device=DEV).uniform_(math.log(1e-3), math.log(1e-1), generator=gen))
    return torch.log(A), dt + torch.log(-torch.expm1(-dt))


def prepare(case, seed):
    gen = torch.Generator(device=DEV).manual_seed(seed)
    K, V, H, B, T = (case[x] for x in ("K", "V", "H", "B", "T"))
    dt = DTYPES[case["dtype"]]
    lens = _lens(case)
    N = len(lens) if lens else B

    def normal(*shape, dtype=F32, std=1.0):
        return torch.randn(shape, device=DEV, generator=gen).mul_(std).to(dtype)

    st = {"case": case, "cu": None, "h0": None, "q_scale": None, "k_scale": None}
    if lens:
        st["cu"] = torch.tensor([0] + lens, dtype=torch.int64).cumsum(0).to(DEV)
    if case["carry"]:
        st["h0"] = normal(N, H, K, V, std=0.02)
    A_log, dt_bias = _layer_gates(B * T, H, gen)
    if case["kind"] == "mixer":
        st["x"] = [normal(B, T, H * D, dtype=dt) for D in (K, K, V)]
        st["cache"] = [normal(N, H * D, 4, dtype=dt) for D in (K, K, V)]
        st["conv"] = [kg.ShortConvolution(H * D, 4, device=DEV, dtype=dt).requires_grad_(False) for D in (K, K, V)]
        for c in st["conv"]:
            c.weight.copy_(normal(*c.weight.shape, std=0.5))
        st["a"], st["b"] = normal(B, T, H, dtype=dt), normal(B, T, H, dtype=dt)
        st["A_log"], st["dt_bias"] = A_log, dt_bias
        st["gate"] = normal(B, T, H, V, dtype=dt)
        st["o_norm"] = kg.FusedRMSNormGated(V, device=DEV, dtype=dt).requires_grad_(False)
        st["o_norm"].weight.copy_(1 + 0.1 * normal(V))
        return st
    q, k = normal(B, T, H, K), normal(B, T, H, K)
    if not case["l2"]:
        q, k = (torch.nn.functional.normalize(x, dim=-1) for x in (q, k))
    if case["dtype"] == "fp8":
        for n, x in (("q", q), ("k", k)):
            s = x.abs().amax((0, 1, 3)) / 448
            st[n], st[n + "_scale"] = (x / s[:, None]).to(torch.float8_e4m3fn), s
    else:
        st["q"], st["k"] = q.to(dt), k.to(dt)
    st["v"] = normal(B, T, H, V, dtype=dt)
    st["beta"] = torch.sigmoid(normal(B, T, H)).to(dt)
    z = normal(B, T, H)
    if K == 256:
        st["g"] = -A_log.exp() * torch.nn.functional.softplus(z + dt_bias)
    else:
        st["g"] = -torch.nn.functional.softplus(z)
    if case["kind"] == "train":
        st["do"], st["dht"] = normal(B, T, H, V, dtype=dt), normal(N, H, K, V)
        for n in ("q", "k", "v", "g", "beta", "h0"):
            if st[n] is not None:
                st[n].requires_grad_()
    return st


def run(st):
    c = st["case"]
    if c["kind"] == "train":
        o, ht = kg.chunk_gated_delta_rule(st["q"], st["k"], st["v"], st["g"], st["beta"], initial_state=st["h0"],
                                          output_final_state=True, use_qk_l2norm_in_kernel=c["l2"])
        wrt = [st[n] for n in ("q", "k", "v", "g", "beta", "h0") if st[n] is not None]
        return [o.detach(), ht.detach(), *torch.autograd.grad([o, ht], wrt, [st["do"], st["dht"]])]
    with torch.no_grad():
        if c["kind"] == "decode":
            return kg.fused_recurrent_gated_delta_rule(
                st["q"], st["k"], st["v"], g=st["g"], beta=st["beta"], initial_state=st["h0"],
                output_final_state=True, use_qk_l2norm_in_kernel=c["l2"])
        if c["kind"] == "op":
            return kg.chunk_gated_delta_rule(
                st["q"], st["k"], st["v"], st["g"], st["beta"], initial_state=st["h0"], output_final_state=True,
                use_qk_l2norm_in_kernel=c["l2"], cu_seqlens=st["cu"], q_scale=st["q_scale"], k_scale=st["k_scale"])
        B, T, H = st["a"].shape
        g, beta = kg.gdn_gates(st["a"], st["b"], st["A_log"], st["dt_bias"])
        if c["form"] == "conv_call":
            o, ht, caches = kg.chunk_gated_delta_rule_conv(
                *st["x"], g, beta, *(m.weight for m in st["conv"]), initial_state=st["h0"], output_final_state=True,
                conv_state=tuple(st["cache"]), output_conv_state=True, use_qk_l2norm_in_kernel=c["l2"])
            return [st["o_norm"](o, st["gate"]), ht, *caches]
        got = [m(x, cache=s, output_final_state=True) for m, x, s in zip(st["conv"], st["x"], st["cache"])]
        q, k, v = (y.view(B, T, H, -1) for y, _ in got)
        if c["form"] == "norm_call":
            y, ht = kg.chunk_gated_delta_rule_gated_norm(
                q, k, v, g, beta, st["gate"], st["o_norm"].weight, initial_state=st["h0"], output_final_state=True,
                use_qk_l2norm_in_kernel=c["l2"], eps=st["o_norm"].eps)
        else:
            o, ht = kg.chunk_gated_delta_rule(q, k, v, g, beta, initial_state=st["h0"], output_final_state=True,
                                              use_qk_l2norm_in_kernel=c["l2"])
            y = st["o_norm"](o, st["gate"])
        return [y, ht, *(s for _, s in got)]


def work(case):
    """Algorithmic minimum: every input read once, every output written once, and the chunked form's
    contractions (6 dk dv + 6 C dk + 4 C dv per token-head forward, twice that backward); a decoding
    token takes its state through a rank-one update and two products instead."""
    K, V, H, B, T = (case[x] for x in ("K", "V", "H", "B", "T"))
    es = {"fp32": 4, "fp8": 2}.get(case["dtype"], 2)
    qk = 1 if case["dtype"] == "fp8" else es
    th, states = B * T * H, (len(_lens(case) or []) or B) * H * K * V * 4
    read = th * (2 * K * qk + V * es + 4 + es) + (states if case["carry"] else 0)
    wrote = th * V * es + states
    flops = th * (6 * K * V + 6 * CHUNK * K + 4 * CHUNK * V)
    if case["kind"] == "decode":
        return {"bytes": read + wrote, "flops": th * 7 * K * V}
    if case["kind"] == "train":                   # + do, dht in; dq, dk, dv, dg, dbeta, dh0 out
        more = th * V * es + states + th * (2 * K * es + V * es + 4 + es) + (states if case["carry"] else 0)
        return {"bytes": read + wrote + more, "flops": 3 * flops}
    if case["kind"] == "mixer":                   # a, b instead of g, beta; gate in; caches in and out
        more = th * (V * es - 4 + es) + 2 * B * H * (2 * K + V) * 4 * es
        return {"bytes": read + wrote + more, "flops": flops + th * (2 * K + V) * 8}
    return {"bytes": read + wrote, "flops": flops}


def tolerance(case):
    """About four times the distance from ``exact`` measured over these ranges: fp32 1.7e-6; fp16 outputs
    2e-4 (their rounding alone); bf16 forwards 3.3e-3 at the headline head dims and 3.9e-3 .. 4.8e-3 with the
    in-op L2 norm or fp8 q and k; gradients 3.8e-3, and 7.5e-3 (dg) under the layer's slow decays; a decoding
    token, whose arithmetic is fp32, 1.7e-3."""
    if case["dtype"] == "fp32":
        return {"rel": 1e-5}
    if case["dtype"] == "fp16":
        return {"rel": 1e-3}
    if case["kind"] == "decode":
        return {"rel": 7e-3}
    if case["kind"] == "train":
        return {"rel": 0.03 if case["K"] == 256 else 0.02}
    return {"rel": 0.015}


def _unit_lower_inverse(A):
    """(I + A)^-1 for strictly lower A [..., n, n], n a power of two, by halves."""
    n = A.shape[-1]
    if n == 1:
        return torch.ones_like(A)
    h = n // 2
    top, low = _unit_lower_inverse(A[..., :h, :h]), _unit_lower_inverse(A[..., h:, h:])
    return torch.cat([torch.cat([top, torch.zeros_like(top)], -1),
                      torch.cat([-(low @ A[..., h:, :h].contiguous() @ top), low], -1)], -2)


def _seq_exact(q, k, v, g, beta, scale, S):
    """One batch of equally long sequences in the chunked (WY) form: q, k, v [B, T, H, *] in 64 bits."""
    B, T, H, _ = q.shape
    n = -(-T // CHUNK)

    def chunks(x):                                 # [B, T, H, ...] -> [B, H, n, 64, ...], zero padded
        x = torch.nn.functional.pad(x.movedim(2, 1), (0, 0) * (x.dim() - 3) + (0, n * CHUNK - T))
        return x.reshape(B, H, n, CHUNK, *x.shape[3:])

    q, k, v, g, beta = (chunks(x) for x in (q * scale, k, v, g, beta))
    gc = g.cumsum(-1)
    tri = torch.ones(CHUNK, CHUNK, dtype=torch.bool, device=q.device).tril()
    decay = (gc[..., :, None] - gc[..., None, :]).masked_fill(~tri, -math.inf).exp()
    A = (beta[..., None] * (k @ k.transpose(-1, -2)) * decay).tril(-1)
    eg = gc.exp()[..., None]
    Ai = _unit_lower_inverse(A)
    w, u = Ai @ (beta[..., None] * eg * k), Ai @ (beta[..., None] * v)
    aqk, qe = (q @ k.transpose(-1, -2)) * decay, q * eg
    kd = (k * (gc[..., -1:] - gc).exp()[..., None]).transpose(-1, -2)
    last = gc[..., -1].exp()
    o = []
    for c in range(n):
        vn = u[:, :, c] - w[:, :, c] @ S
        o.append(qe[:, :, c] @ S + aqk[:, :, c] @ vn)
        S = last[:, :, c, None, None] * S + kd[:, :, c] @ vn
    return torch.stack(o, 2).reshape(B, H, n * CHUNK, -1)[:, :, :T].movedim(1, 2), S


def _op_exact(q, k, v, g, beta, h0, l2, lens=None):
    K, H, V = q.shape[-1], q.shape[2], v.shape[-1]
    if l2:
        q, k = (x * torch.rsqrt(x.square().sum(-1, keepdim=True) + 1e-6) for x in (q, k))
    if lens is None:
        S = h0 if h0 is not None else q.new_zeros(q.shape[0], H, K, V)
        return _seq_exact(q, k, v, g, beta, K ** -0.5, S)
    o, ht, at = [], [], 0
    for i, t in enumerate(lens):
        S = h0[i:i + 1] if h0 is not None else q.new_zeros(1, H, K, V)
        y, S = _seq_exact(*(x[:, at:at + t] for x in (q, k, v, g, beta)), K ** -0.5, S)
        o.append(y)
        ht.append(S)
        at += t
    return torch.cat(o, 1), torch.cat(ht, 0)


def exact(case, seed):
    st = prepare(case, seed)
    up = lambda x: None if x is None else x.detach().to(F64)  # noqa: E731
    if case["kind"] == "mixer":
        conv, caches = [], []
        for x, m, s in zip(st["x"], st["conv"], st["cache"]):
            ext = torch.cat([up(s).transpose(1, 2), up(x)], 1)
            w = up(m.weight)[:, 0]
            conv.append(torch.nn.functional.silu(sum(ext[:, 1 + i:1 + i + x.shape[1]] * w[:, i] for i in range(4))))
            caches.append(ext[:, -4:].transpose(1, 2))
        B, T, H = st["a"].shape
        q, k, v = (y.view(B, T, H, -1) for y in conv)
        g = -up(st["A_log"]).exp() * torch.nn.functional.softplus(up(st["a"]) + up(st["dt_bias"]))
        o, ht = _op_exact(q, k, v, g, torch.sigmoid(up(st["b"])), up(st["h0"]), case["l2"])
        norm = st["o_norm"]
        y = o * torch.rsqrt(o.square().mean(-1, keepdim=True) + norm.eps) * up(norm.weight)
        return [y * torch.nn.functional.silu(up(st["gate"])), ht, *caches]
    names = ("q", "k", "v", "g", "beta", "h0")
    x = {n: up(st[n]) for n in names}
    if case["dtype"] == "fp8":
        x["q"], x["k"] = x["q"] * up(st["q_scale"])[:, None], x["k"] * up(st["k_scale"])[:, None]
    if case["kind"] != "train":
        return _op_exact(*(x[n] for n in names), case["l2"], _lens(case))
    x = {n: t.requires_grad_() if t is not None else None for n, t in x.items()}
    o, ht = _op_exact(*(x[n] for n in names), case["l2"])
    grads = torch.autograd.grad([o, ht], [t for t in x.values() if t is not None], [up(st["do"]), up(st["dht"])])
    return [o.detach(), ht.detach(), *grads]
