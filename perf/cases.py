"""Workloads of the package as a speculative-decoding program meets them, for timing and comparison.

A target model is a stack of decoder layers whose projections are 4-bit MLX linears.  Per
generated block the program runs every layer on 16 tokens (the verify step) and rolls the
recurrent caches back to the accepted length; per prompt it runs them on the prompt; at the end
of an answer, and when it decodes without a draft, on one token or a short block.  Each case is
one of those calls on one layer (or, for the rollback, on all recurrent layers at once):

  call       one ``verify_matmul`` - the smallest thing a user can ask for
  dense      the projections of a dense layer: qkv, o, the gated MLP (``silu_gate_up``, down)
  gdn        a GatedDeltaNet layer: prompt, one token, or an armed block followed by its rollback
  attention  the attention layer of a 16-token block over a long KV cache, then the trim.  Prompt
             attention is not among the cases: it is torch's own operator, not this package's
  moe        the routed experts of a layer: gate/up in one gathered launch, then down
  rollback   arm, record in place, roll back every recurrent layer of the model

Shapes are those of the benchmark configurations (9B- and 27B-shaped dense stacks, the MoE
stack, 48 x 32-head recurrent layers, 8 x 256 KV heads) and generic ones around them.
"""
import math
import os

import torch
import torch.nn as nn

DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
SIZEOF = {"bf16": 2, "fp16": 2, "fp32": 4}
ATTENTION_HEADS = ((32, 8, 256), (16, 4, 256), (24, 4, 256), (16, 2, 256), (32, 8, 128), (40, 8, 128), (64, 8, 128),
                   (16, 8, 128))
GDN_HEADS = ((16, 32, 128), (16, 48, 128), (16, 16, 128), (8, 32, 128), (16, 64, 128), (4, 8, 64))
BLOCK = 16


def listed():
    return [
        # the smallest call: one narrow projection of one verify block; what counts is latency
        {"name": "call_1024x512", "kind": "call", "K": 1024, "N": 512, "group": 64, "dtype": "bf16"},
        # decoding without a draft: one token through a 9B-shaped layer
        {"name": "dense_9b_one_token", "kind": "dense", "rows": 1, "hidden": 4096, "qkv": 6144, "inter": 12288,
         "group": 64, "dtype": "bf16", "packed": False},
        # the verify step of a 27B-shaped layer: where a speculative decoder spends its time
        {"name": "dense_27b_verify", "kind": "dense", "rows": 16, "hidden": 5120, "qkv": 7168, "inter": 17408,
         "group": 64, "dtype": "bf16", "packed": False},
        # the same step of a 9B-shaped checkpoint quantised in groups of 32 instead of 64
        {"name": "dense_9b_verify_group32", "kind": "dense", "rows": 16, "hidden": 4096, "qkv": 6144, "inter": 12288,
         "group": 32, "dtype": "bf16", "packed": False},
        # a short chat turn: a prompt of an odd number of tokens
        {"name": "dense_9b_prompt77", "kind": "dense", "rows": 77, "hidden": 4096, "qkv": 6144, "inter": 12288,
         "group": 64, "dtype": "bf16", "packed": False},
        # a long prompt through a 27B-shaped layer: the largest call
        {"name": "dense_27b_prompt1024", "kind": "dense", "rows": 1024, "hidden": 5120, "qkv": 7168, "inter": 17408,
         "group": 64, "dtype": "bf16", "packed": False},
        # recurrent layer, verify block with tape, six of the drafts accepted
        {"name": "gdn_verify", "kind": "gdn", "tokens": 16, "hidden": 5120, "Hk": 16, "Hv": 32, "D": 128,
         "state": "fp32", "accepted": 6},
        # recurrent layer over a prompt that starts from an empty cache (whose state has the array dtype)
        {"name": "gdn_prompt1024", "kind": "gdn", "tokens": 1024, "hidden": 5120, "Hk": 16, "Hv": 32, "D": 128,
         "state": "bf16", "accepted": 0},
        # attention layer of a verify block, ordinary and long context
        {"name": "attention_4k", "kind": "attention", "prefix": 4096, "hidden": 5120, "Hq": 32, "Hk": 8, "D": 256},
        {"name": "attention_32k", "kind": "attention", "prefix": 32700, "hidden": 5120, "Hq": 32, "Hk": 8, "D": 256},
        # routed experts of a verify block
        {"name": "moe_verify", "kind": "moe", "tokens": 16, "experts": 256, "top_k": 8, "hidden": 2048, "inter": 512},
        # rollback of all recurrent layers after a verify step
        {"name": "rollback_48x32", "kind": "rollback", "layers": 48, "batch": 1, "Hk": 16, "Hv": 32, "D": 128,
         "state": "fp32", "accepted": 6, "arena": True},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _rows(rng, longest):
    """Tokens of a call: one, a last short block, a verify block, a prompt."""
    return rng.choice((1, rng.randint(2, BLOCK - 1), BLOCK, BLOCK, _log(rng, BLOCK + 1, longest), _log(rng, BLOCK + 1, longest)))


def draw(rng):
    kind = rng.choice(("call", "dense", "dense", "dense", "gdn", "gdn", "attention", "moe", "rollback"))
    if kind == "call":
        return {"kind": kind, "K": 128 * _log(rng, 2, 96), "N": 32 * _log(rng, 2, 384), "group": rng.choice((64, 64, 32, 128)),
                "dtype": rng.choice(("bf16", "bf16", "fp16"))}
    if kind == "dense":
        hidden = 256 * rng.randint(4, 20)
        inter = 128 * rng.randint(2 * hidden // 128, 17408 * hidden // 5120 // 128)
        return {"kind": kind, "rows": _rows(rng, 1024), "hidden": hidden, "qkv": 32 * rng.randint(hidden // 32, 7168 * hidden // 5120 // 32),
                "inter": inter, "group": rng.choice((64, 64, 64, 32, 128)), "dtype": rng.choice(("bf16", "bf16", "fp16")),
                "packed": rng.random() < 0.3}
    if kind == "gdn":
        hk, hv, d = rng.choice(GDN_HEADS)
        tokens = _rows(rng, 1024)
        return {"kind": kind, "tokens": tokens, "hidden": 256 * rng.randint(4, 20), "Hk": hk, "Hv": hv, "D": d,
                "state": rng.choice(("fp32", "bf16")), "accepted": rng.randint(0, max(0, min(tokens, BLOCK) - 2))}
    if kind == "attention":
        hq, hk, d = rng.choice(ATTENTION_HEADS)
        return {"kind": kind, "prefix": _log(rng, 1024, 32700), "hidden": 256 * rng.randint(4, 20), "Hq": hq, "Hk": hk, "D": d}
    if kind == "moe":
        experts = rng.choice((8, 32, 64, 128, 256))
        hidden, inter = 256 * rng.randint(4, 8), 128 * rng.randint(2, 4 if experts > 128 else 12)
        return {"kind": kind, "tokens": rng.choice((1, rng.randint(2, BLOCK), BLOCK, BLOCK, _log(rng, BLOCK + 1, 256))),
                "experts": experts, "top_k": rng.choice((2, 4, 8)), "hidden": hidden, "inter": inter}
    hk, hv, d = rng.choice(GDN_HEADS)
    batch = rng.choice((1, 1, 2))
    most = 48 * 32 * 128 * 128 // (batch * hv * d * d)
    return {"kind": kind, "layers": _log(rng, 3, min(64, most)), "batch": batch, "Hk": hk, "Hv": hv, "D": d,
            "state": rng.choice(("fp32", "fp32", "bf16")), "accepted": rng.randint(0, BLOCK - 2), "arena": rng.random() < 0.7}


# ---- inputs -----------------------------------------------------------------------------------
class _Random:
    """Seeded values on the GPU."""

    def __init__(self, seed):
        self.gen = torch.Generator(device="cuda")
        self.gen.manual_seed(seed)

    def normal(self, *shape, dtype=torch.float32, std=1.0):
        return (torch.randn(shape, generator=self.gen, device="cuda") * std).to(dtype)

    def triple(self, K, N, group, dtype, lead=()):
        """Codes, scales and biases as a 4-bit checkpoint holds them: weights of about N(0, 1/K), so that
        a projection of unit-size activations has unit-size results."""
        w = torch.randint(-2 ** 31, 2 ** 31, (*lead, N, K // 8), generator=self.gen, device="cuda", dtype=torch.int32)
        s = (0.5 + torch.rand((*lead, N, K // group), generator=self.gen, device="cuda")) * (0.2 * K ** -0.5)
        return w, s.to(dtype), (s * -7.5).to(dtype)

    def linear(self, K, N, group=64, dtype=torch.bfloat16):
        from dflash_mlx_amd.quantized import QuantizedLinear

        return QuantizedLinear(*self.triple(K, N, group, dtype), group_size=group, bits=4)


class _Dense(nn.Module):
    def __init__(self, r, case, dtype):
        super().__init__()
        h, inter, group = case["hidden"], case["inter"], case["group"]
        self.qkv_proj, self.o_proj = r.linear(h, case["qkv"], group, dtype), r.linear(h, h, group, dtype)
        self.gate_proj, self.up_proj = r.linear(h, inter, group, dtype), r.linear(h, inter, group, dtype)
        self.down_proj = r.linear(inter, h, group, dtype)


class _Layer(nn.Module):
    """A decoder layer of the hybrid model, as the hooks look for it: ``linear_attn`` or ``self_attn``."""

    def __init__(self, mixer, is_linear):
        super().__init__()
        self.is_linear = is_linear
        setattr(self, "linear_attn" if is_linear else "self_attn", mixer)


def _load(model):
    """What a program does with a model whose weights are on the device."""
    from dflash_mlx_amd.runtime import enable_verify_linears

    enable_verify_linears(model, {"num_hidden_layers": 64})


def _prepare_call(case, r, dtype):
    os.environ.setdefault("DFLASH_VERIFY_QMM", "1")
    return {"x": r.normal(1, BLOCK, case["K"], dtype=dtype), "w": r.triple(case["K"], case["N"], case["group"], dtype)}


def _prepare_dense(case, r, dtype):
    from dflash_mlx_amd.verify_linear import pack_verify_linears

    layer = _Dense(r, case, dtype)
    _load(layer)
    if case["packed"]:
        pack_verify_linears(layer)
    shape = (1, case["rows"], case["hidden"])
    return {"layer": layer, "x": r.normal(*shape, dtype=dtype), "attn": r.normal(*shape, dtype=dtype)}


def _prepare_gdn(case, r):
    from dflash_mlx_amd import gdn_layer
    from dflash_mlx_amd.recurrent_rollback_cache import RecurrentRollbackCache

    h, hk, hv, d, bf = case["hidden"], case["Hk"], case["Hv"], case["D"], torch.bfloat16
    conv_dim = 2 * hk * d + hv * d
    narrow = -(-hv // 16) * 16 if hv >= 16 else 16
    mixer = gdn_layer.GatedDeltaNet(
        h, num_k_heads=hk, num_v_heads=hv, head_k_dim=d, head_v_dim=d, in_proj_qkv=r.linear(h, conv_dim),
        in_proj_z=r.linear(h, hv * d), in_proj_b=_Narrow(r.linear(h, narrow), hv) if narrow != hv else r.linear(h, narrow),
        in_proj_a=_Narrow(r.linear(h, narrow), hv) if narrow != hv else r.linear(h, narrow), out_proj=r.linear(hv * d, h))
    mixer.conv1d.weight = nn.Parameter(r.normal(conv_dim, 4, 1, dtype=bf, std=0.5), requires_grad=False)
    mixer.A_log = nn.Parameter(torch.log(torch.rand(hv, generator=r.gen, device="cuda") * 2 + 0.2).to(bf), requires_grad=False)
    mixer.dt_bias = nn.Parameter(r.normal(hv, dtype=bf, std=0.3), requires_grad=False)
    layer = _Layer(mixer.to("cuda"), True)
    gdn_layer._install_exact_small_proj_hooks(mixer)
    gdn_layer._install_speculative_linear_cache_hook(mixer)
    _load(layer)
    cache = RecurrentRollbackCache(size=2, conv_kernel_size=4)
    if case["tokens"] <= BLOCK:  # a conversation is under way
        cache[0] = r.normal(1, 3, conv_dim, dtype=bf)
        cache[1] = r.normal(1, hv, d, d, dtype=DTYPES[case["state"]], std=0.1)
    return {"mixer": mixer, "x": r.normal(1, case["tokens"], h, dtype=bf), "cache": cache, "case": case}


class _Narrow(nn.Module):
    """The first outputs of a projection whose height the 4-bit format rounds up."""

    def __init__(self, inner, n):
        super().__init__()
        self.inner, self.n = inner, n

    def forward(self, x):
        return self.inner(x)[..., :self.n]


def _prepare_attention(case, r):
    from dflash_mlx_amd.attention_layer import GatedAttention, configure_full_attention_split
    from dflash_mlx_amd.cache import KVCache

    h, hq, hk, d, bf = case["hidden"], case["Hq"], case["Hk"], case["D"], torch.bfloat16
    attn = GatedAttention(num_attention_heads=hq, num_key_value_heads=hk, head_dim=d, q_proj=r.linear(h, 2 * hq * d),
                          k_proj=r.linear(h, hk * d), v_proj=r.linear(h, hk * d), o_proj=r.linear(hq * d, h)).to("cuda")
    for norm in (attn.q_norm, attn.k_norm):
        norm.weight = nn.Parameter((1 + r.normal(d, std=0.1)).to(bf), requires_grad=False)
    layer = _Layer(attn, False)
    configure_full_attention_split([layer], enabled=True)
    _load(layer)
    cache = KVCache()
    cache.update_and_fetch(r.normal(1, hk, case["prefix"], d, dtype=bf), r.normal(1, hk, case["prefix"], d, dtype=bf))
    return {"attn": attn, "x": r.normal(1, BLOCK, h, dtype=bf), "cache": cache}


def _prepare_moe(case, r):
    E, T, h, inter, bf = case["experts"], case["tokens"], case["hidden"], case["inter"], torch.bfloat16
    logits = r.normal(T, E)
    ids = torch.topk(torch.softmax(logits, dim=-1), case["top_k"], dim=-1).indices.to(torch.int32).reshape(-1)
    pairs = T * case["top_k"]
    return {"gate_up": r.triple(h, 2 * inter, 64, bf, (E,)), "down": r.triple(inter, h, 64, bf, (E,)), "ids": ids,
            "x": r.normal(pairs, h, dtype=bf), "hidden": r.normal(pairs, inter, dtype=bf)}


def _prepare_rollback(case, r):
    from dflash_mlx_amd.recurrent_rollback_cache import RecurrentRollbackCache, RollbackArena

    L, B, hk, hv, d, T = case["layers"], case["batch"], case["Hk"], case["Hv"], case["D"], BLOCK
    C = 2 * hk * d + hv * d
    k = r.normal(L, B, T, hk, d)
    tapes = {"tape": r.normal(L, B, T, hv, d, std=0.05), "k": (k / k.norm(dim=-1, keepdim=True)).to(torch.bfloat16),
             "g": torch.exp(-torch.nn.functional.softplus(r.normal(L, B, T, hv))), "qkv": r.normal(L, B, T, C, dtype=torch.bfloat16)}
    state, conv = r.normal(L, B, hv, d, d, dtype=DTYPES[case["state"]], std=0.1), r.normal(L, B, 3, C, dtype=torch.bfloat16)
    if case["arena"]:
        arena = RollbackArena(L, batch=B, Hk=hk, Hv=hv, Dk=d, Dv=d, conv_dim=C, state_dtype=DTYPES[case["state"]])
        for name, value in tapes.items():  # a forward writes its tape where the arena keeps it
            getattr(arena, name).copy_(value)
        arena.state[0].copy_(state)
        arena.conv[0].copy_(conv)
        caches = arena.caches()
        tapes = {name: [arena.tape_slots(i)[j] for i in range(L)] for j, name in enumerate(("tape", "k", "g", "qkv"))}
    else:
        arena, caches = None, [RecurrentRollbackCache(size=2, conv_kernel_size=4) for _ in range(L)]
        for i, c in enumerate(caches):
            c[0], c[1] = conv[i], state[i]
    return {"caches": caches, "arena": arena, "tapes": tapes, "accepted": case["accepted"]}


def prepare(case, seed):
    r, kind = _Random(seed), case["kind"]
    if kind in ("call", "dense"):
        made = (_prepare_call if kind == "call" else _prepare_dense)(case, r, DTYPES[case["dtype"]])
    else:
        made = {"gdn": _prepare_gdn, "attention": _prepare_attention, "moe": _prepare_moe, "rollback": _prepare_rollback}[kind](case, r)
    return dict(made, kind=kind, group=case.get("group", 64))


# ---- one pass ---------------------------------------------------------------------------------
def _run_dense(s):
    from dflash_mlx_amd.verify_linear import silu_gate_up

    layer, x = s["layer"], s["x"]
    qkv, o = layer.qkv_proj(x), layer.o_proj(s["attn"])
    hidden = silu_gate_up(layer, x)
    return qkv, o, hidden, layer.down_proj(hidden)


def _run_gdn(s):
    from dflash_mlx_amd.recurrent_rollback_cache import RecurrentRollbackCache

    case, cache = s["case"], s["cache"]
    if case["tokens"] > BLOCK:  # a new prompt has a new cache; an fp32 state is asked for by providing one
        cache = RecurrentRollbackCache(size=2, conv_kernel_size=4)
        if case["state"] == "fp32":
            cache[1] = torch.zeros((1, case["Hv"], case["D"], case["D"]), dtype=torch.float32, device="cuda")
    armed = 1 < case["tokens"] <= BLOCK
    if armed:
        cache.arm_rollback()
    y = s["mixer"](s["x"], cache=cache)
    if armed:
        cache.rollback(case["accepted"])
    return y, cache[0], cache[1]


def _run_attention(s):
    cache = s["cache"]
    y = s["attn"](s["x"], mask="causal", cache=cache)
    keys, values = cache.state
    cache.trim(BLOCK)
    return y, keys, values


def _run_rollback(s):
    from dflash_mlx_amd.engine import HybridGDNEngine

    engine, caches, tapes, arena = HybridGDNEngine(), s["caches"], s["tapes"], s["arena"]
    engine.arm_rollback(caches, prefix_len=0)
    for i, c in enumerate(caches):
        c.record_tape(tape=tapes["tape"][i], k=tapes["k"][i], g=tapes["g"][i], qkv=tapes["qkv"][i])
    engine.rollback(caches, target_len=0, acceptance_len=s["accepted"], drafted_tokens=BLOCK - 1)
    if arena is not None:
        return arena.state, arena.conv
    return [c[j] for c in caches[:32] for j in (0, 1)]


@torch.no_grad()
def run(state):
    kind = state["kind"]
    if kind == "call":
        from dflash_mlx_amd.verify_qmm import verify_matmul

        return verify_matmul(state["x"], *state["w"], group_size=state["group"], bits=4)
    if kind == "moe":
        from dflash_mlx_amd.verify_qmm import gather_qmm

        return (gather_qmm(state["x"], *state["gate_up"], state["ids"]), gather_qmm(state["hidden"], *state["down"], state["ids"]))
    return {"dense": _run_dense, "gdn": _run_gdn, "attention": _run_attention, "rollback": _run_rollback}[kind](state)


# ---- what a pass cannot do without ---------------------------------------------------------------
def _projection(rows, K, N, group=64):
    """(bytes, flops): codes, scales and biases, the activations and the results, once each."""
    return N * K // 2 + 4 * N * (K // group) + 2 * rows * (K + N), 2 * rows * K * N


def work(case):
    kind = case["kind"]
    if kind == "call":
        parts = [_projection(BLOCK, case["K"], case["N"], case["group"])]
    elif kind == "dense":
        h, inter, rows, g = case["hidden"], case["inter"], case["rows"], case["group"]
        parts = [_projection(rows, K, N, g) for K, N in ((h, case["qkv"]), (h, h), (h, 2 * inter), (inter, h))]
    elif kind == "gdn":
        h, hk, hv, d, rows = case["hidden"], case["Hk"], case["Hv"], case["D"], case["tokens"]
        conv_dim = 2 * hk * d + hv * d
        parts = [_projection(rows, h, conv_dim + hv * d + 2 * hv), _projection(rows, hv * d, h)]
        sweeps = rows + (case["accepted"] + 1 if 1 < rows <= BLOCK else 0)  # the forward's and the replay's steps
        parts.append((2 * hv * d * d * SIZEOF[case["state"]] + 12 * conv_dim, 6 * hv * d * d * sweeps))
    elif kind == "attention":
        h, hq, hk, d = case["hidden"], case["Hq"], case["Hk"], case["D"]
        keys = case["prefix"] + BLOCK
        parts = [_projection(BLOCK, h, 2 * hq * d + 2 * hk * d), _projection(BLOCK, hq * d, h),
                 (2 * hk * keys * d * 2, 4 * hq * BLOCK * keys * d)]
    elif kind == "moe":
        # the experts that at least one of the (token, expert) pairs picks, on average
        E, h, inter, pairs = case["experts"], case["hidden"], case["inter"], case["tokens"] * case["top_k"]
        busy = E * (1 - (1 - min(1.0, case["top_k"] / E)) ** case["tokens"])
        parts = []
        for K, N in ((h, 2 * inter), (inter, h)):
            parts.append((busy * (N * K // 2 + 4 * N * (K // 64)) + 2 * pairs * (K + N), 2 * pairs * K * N))
    else:
        L, B, hk, hv, d, steps = case["layers"], case["batch"], case["Hk"], case["Hv"], case["D"], case["accepted"] + 1
        C = 2 * hk * d + hv * d
        per_slot = hv * (2 * d * d * SIZEOF[case["state"]] + steps * (4 * d + 4)) + steps * hk * 2 * d + 2 * 3 * C * 2
        parts = [(L * B * per_slot, L * B * hv * steps * 3 * d * d)]
    return {"bytes": float(sum(p[0] for p in parts)), "flops": float(sum(p[1] for p in parts))}


def tolerance(case):
    if case["kind"] == "rollback" and case["state"] == "fp32":
        return {"rel": 1e-5}
    if case.get("dtype") == "fp16":
        return {"rel": 2e-3}
    return {"rel": 1e-2}
