"""Parity of the gfx950 GatedDeltaNet glue kernels (dflash_gdn_prepare, dflash_gdn_gated_norm)
against the CPU oracle, and of the layer's speculative call on the device against the same
layer evaluated with array operators on the host.

Bars: the next conv state is a copy - bit-exact; q, k, v, beta and the normed output agree
with the oracle to two steps of the array dtype's grid everywhere and exactly on
at least 97 % of the elements (device exp / log differ from the host's in the last fp32 bit,
which now and then moves a rounding); g (fp32) to 2e-5 relative in its exponent."""
import numpy as np
import pytest
import torch

from dflash_mlx_amd import gdn_layer as G
from dflash_mlx_amd.recurrent_rollback_cache import RecurrentRollbackCache
from oracle import dflash_oracle as O
from test_gdn_layer_glue import _inputs, _layer

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
TORCH = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
ULP = {"bf16": 2.0 ** -7, "fp16": 2.0 ** -10, "fp32": 2.0 ** -22}     # grid spacing relative to |x|, upper bound
TINY = {"bf16": 1e-7, "fp16": 2.0 ** -22, "fp32": 1e-7}     # two steps of the fp16 subnormal grid


def _dev(t, dtype, param_dtype=None):
    out = {}
    for key, val in t.items():
        dt = param_dtype if (param_dtype is not None and key in ("A_log", "dt_bias")) else dtype
        out[key] = None if val is None else torch.from_numpy(val).to(dt).to(DEV)
    return out


def _check(got, want, name):
    np.testing.assert_array_equal(got[0].float().cpu().numpy(), want[0])
    for what, a, b in zip(("q", "k", "v", "g", "beta"), got[1:], want[1:]):
        a = a.float().cpu().numpy()
        assert a.shape == b.shape, what
        if what == "g":
            np.testing.assert_allclose(np.log(a), np.log(b), rtol=2e-5, atol=1e-6)
            continue
        assert np.all(np.abs(a - b) <= 2 * ULP[name] * np.abs(b) + TINY[name]), what
        assert np.mean(a == b) > 0.97 or name == "fp32", what


@pytest.mark.parametrize("name", ["bf16", "fp16", "fp32"])
@pytest.mark.parametrize("S,with_state,masked", [(16, True, False), (16, False, True), (1, True, False),
                                                 (2, True, True), (3, False, False), (5, True, True)])
def test_prepare_against_the_oracle(native_lib, name, S, with_state, masked):
    t, dims = _inputs(B=2, S=S, Hk=2, Hv=4, Dk=128, Dv=128, seed=40 + S, with_state=with_state, dtype=name)
    mask = None
    if masked:
        mask = np.ones((2, S), bool)
        mask[1, S // 2] = False
    want = O.gdn_prepare(**t, **dims, mask=mask, dtype=name)
    d = _dev(t, TORCH[name])
    got = G.gdn_prepare(d["qkv"], d["conv_state"], d["conv_w"], d["a"], d["b"], d["A_log"], d["dt_bias"],
                        None if mask is None else torch.from_numpy(mask).to(DEV), **dims)
    torch.cuda.synchronize()
    assert got[1].dtype == TORCH[name] and got[4].dtype == torch.float32
    _check(got, want, name)


@pytest.mark.parametrize("dims", [dict(Hk=1, Hv=2, Dk=64, Dv=64), dict(Hk=2, Hv=2, Dk=256, Dv=128),
                                  dict(Hk=16, Hv=32, Dk=128, Dv=128), dict(Hk=2, Hv=4, Dk=128, Dv=192)])
def test_prepare_head_shapes_and_fp32_parameters(native_lib, dims):
    t, dims = _inputs(B=1, S=16, seed=50 + dims["Dk"], **dims)
    want = O.gdn_prepare(**t, **dims, dtype="bf16", bias_dtype="fp32")
    d = _dev(t, torch.bfloat16, param_dtype=torch.float32)
    got = G.gdn_prepare(d["qkv"], d["conv_state"], d["conv_w"].unsqueeze(-1), d["a"], d["b"], d["A_log"],
                        d["dt_bias"], None, **dims)
    torch.cuda.synchronize()
    _check(got, want, "bf16")


@pytest.mark.parametrize("K", [2, 3])
def test_prepare_shorter_conv_kernels(native_lib, K):
    t, dims = _inputs(B=1, S=5, Hk=1, Hv=2, Dk=128, Dv=64, K=K, seed=80 + K)
    want = O.gdn_prepare(**t, **dims, dtype="bf16")
    d = _dev(t, torch.bfloat16)
    got = G.gdn_prepare(d["qkv"], d["conv_state"], d["conv_w"], d["a"], d["b"], d["A_log"], d["dt_bias"], None, **dims)
    torch.cuda.synchronize()
    assert tuple(got[0].shape) == (1, K - 1, 2 * 128 + 2 * 64)
    _check(got, want, "bf16")


def test_prepare_takes_the_array_ops_for_other_head_sizes(native_lib):
    t, dims = _inputs(B=1, S=4, Hk=1, Hv=2, Dk=32, Dv=96, seed=60)
    want = O.gdn_prepare(**t, **dims, dtype="bf16")
    d = _dev(t, torch.bfloat16)
    got = G.gdn_prepare(d["qkv"], d["conv_state"], d["conv_w"], d["a"], d["b"], d["A_log"], d["dt_bias"], None, **dims)
    _check(got, want, "bf16")
    with pytest.raises(ValueError):
        G.gdn_prepare(d["qkv"][..., :-1], d["conv_state"], d["conv_w"], d["a"], d["b"], d["A_log"], d["dt_bias"],
                      None, **dims)


def test_prepare_rejects_bad_shapes_through_the_c_abi(native_lib):
    import dflash_mlx_amd._native as nat
    x = torch.zeros(4096, dtype=torch.bfloat16, device=DEV)
    g = torch.zeros(64, dtype=torch.float32, device=DEV)
    ptr = x.data_ptr()
    args = [ptr] * 7 + [None] + [ptr] * 4 + [g.data_ptr(), ptr]
    rc = native_lib.dflash_gdn_prepare(*args, 1, 1, 1, 1, 96, 64, 4, nat.BF16, nat.BF16, 1e-6, None)
    assert rc != 0 and b"multiples of 64" in native_lib.dflash_last_error()
    rc = native_lib.dflash_gdn_prepare(*args, 1, 1, 1, 1, 64, 64, 1, nat.BF16, nat.BF16, 1e-6, None)
    assert rc != 0
    rc = native_lib.dflash_gdn_gated_norm(ptr, ptr, ptr, ptr, 4, 100, nat.BF16, nat.BF16, 1e-6, None)
    assert rc != 0 and b"multiple of 64" in native_lib.dflash_last_error()
    torch.cuda.synchronize()


@pytest.mark.parametrize("name", ["bf16", "fp16", "fp32"])
@pytest.mark.parametrize("D", [64, 128, 256])
def test_gated_norm_against_the_oracle(native_lib, name, D):
    rng = np.random.default_rng(70 + D)
    r = lambda x: O.round_to(np.asarray(x, np.float32), name)
    x, z, w = r(rng.standard_normal((3, 16, 4, D)) * 3), r(rng.standard_normal((3, 16, 4, D))), r(1 + 0.1 * rng.standard_normal(D))
    want = O.gdn_gated_norm(x, z, w, name)
    got = G.gated_norm(*(torch.from_numpy(v).to(TORCH[name]).to(DEV) for v in (x, z, w)))
    torch.cuda.synchronize()
    a = got.float().cpu().numpy()
    assert np.all(np.abs(a - want) <= 2 * ULP[name] * np.abs(want) + TINY[name])
    assert np.mean(a == want) > 0.97 or name == "fp32"


def test_speculative_layer_call_on_the_device_matches_the_host(native_lib, monkeypatch):
    """The same layer, the same tokens: device kernels (projections through the verify qmm,
    fused glue, block recurrence) against the array operators on the host, then a rollback."""
    monkeypatch.setenv("DFLASH_VERIFY_QMM", "1")
    host = _layer(seed=8, hidden=512, Hk=2, Hv=4, D=128, dtype=torch.bfloat16, quantized=True)
    G._install_exact_small_proj_hooks(host)
    G._install_speculative_linear_cache_hook(host)
    import copy
    dev = copy.deepcopy(host).to(DEV)
    gen = torch.Generator().manual_seed(9)
    prompt = torch.randn((1, 7, 512), generator=gen).to(torch.bfloat16)
    block = torch.randn((1, 16, 512), generator=gen).to(torch.bfloat16)

    outs, caches = [], []
    for layer, to in ((host, lambda t: t), (dev, lambda t: t.to(DEV))):
        cache = RecurrentRollbackCache()
        layer(to(prompt), cache=cache)
        cache[1] = cache[1].float()                 # the serving configuration keeps S in fp32
        cache.arm_rollback(prefix_len=7)
        y = layer(to(block), cache=cache)
        tape = cache._tape.float().cpu()
        cache.rollback(9)
        outs.append((y.float().cpu(), tape))
        caches.append((cache[0].float().cpu(), cache[1].float().cpu()))
    torch.cuda.synchronize()
    rel = lambda a, b: float((a - b).norm() / b.norm())
    assert rel(outs[1][0], outs[0][0]) < 2e-2       # bf16 activations through five matmuls
    assert rel(outs[1][1], outs[0][1]) < 2e-2
    assert rel(caches[1][1], caches[0][1]) < 2e-2
    assert rel(caches[1][0], caches[0][0]) < 1e-2


def test_layer_hook_with_an_arena_cache_matches_the_per_layer_cache(native_lib, monkeypatch):
    """The documented set-up - RollbackArena with its defaults, the layer's speculative hook
    recording its fp32 tape into it, rollback_all - against a plain RecurrentRollbackCache."""
    import copy

    from dflash_mlx_amd.recurrent_rollback_cache import RollbackArena

    monkeypatch.setenv("DFLASH_VERIFY_QMM", "1")
    host = _layer(seed=18, hidden=512, Hk=2, Hv=4, D=128, dtype=torch.bfloat16, quantized=True)
    G._install_exact_small_proj_hooks(host)
    G._install_speculative_linear_cache_hook(host)
    layer = copy.deepcopy(host).to(DEV)
    gen = torch.Generator().manual_seed(19)
    prompt = torch.randn((1, 7, 512), generator=gen).to(torch.bfloat16).to(DEV)
    block = torch.randn((1, 16, 512), generator=gen).to(torch.bfloat16).to(DEV)
    conv_dim = 2 * 2 * 128 + 4 * 128

    plain = RecurrentRollbackCache()
    layer(prompt, cache=plain)
    plain[1] = plain[1].float()
    conv0, state0 = plain[0].clone(), plain[1].clone()
    plain.arm_rollback(prefix_len=7)
    y_plain = layer(block, cache=plain)
    plain.rollback(9)

    arena = RollbackArena(1, Hk=2, Hv=4, Dk=128, Dv=128, conv_dim=conv_dim, device=DEV)
    cache = arena.caches()[0]
    cache[0].copy_(conv0); cache[1].copy_(state0)
    arena.arm_all(prefix_len=7)
    y_arena = layer(block, cache=cache)
    assert cache._tape.dtype == torch.float32
    arena.rollback_all(torch.tensor(9, dtype=torch.int32, device=DEV))
    torch.cuda.synchronize()
    assert torch.equal(y_arena, y_plain)
    assert torch.equal(cache[1], plain[1]) and torch.equal(cache[0], plain[0])


@pytest.mark.parametrize("name", ["bf16", "fp16", "fp32"])
@pytest.mark.parametrize("B,S,Hk,Hv,Dk,Dv,K,masked", [(1, 1030, 16, 32, 128, 128, 4, False), (2, 333, 8, 16, 64, 192, 3, True),
                                                      (1, 700, 4, 8, 256, 64, 2, True), (3, 17, 2, 2, 128, 128, 4, True)])
def test_long_prompts_and_strided_projections(native_lib, name, B, S, Hk, Hv, Dk, Dv, K, masked):
    """Several tokens per wave and rows with a stride: the bits of blocks of at most 16 tokens (one token per wave) of
    contiguous arrays, their conv windows handed on; qkv_out is qkv without what the mask hides."""
    dt = TORCH[name]
    gen = torch.Generator(device=DEV).manual_seed(S)
    C = 2 * Hk * Dk + Hv * Dv
    joint = torch.randn((B, S, C + 64 + 2 * Hv), generator=gen, device=DEV).to(dt)
    qkv, b, a = joint[..., :C], joint[..., C + 64:C + 64 + Hv], joint[..., C + 64 + Hv:]
    conv_w = (torch.randn((C, K), generator=gen, device=DEV) * 0.5).to(dt)
    A_log, dt_bias = torch.randn(Hv, generator=gen, device=DEV).to(dt), torch.randn(Hv, generator=gen, device=DEV).to(dt)
    mask = torch.rand((B, S), generator=gen, device=DEV) > 0.2 if masked else None
    state = torch.randn((B, K - 1, C), generator=gen, device=DEV).to(dt)
    dims = dict(Hk=Hk, Hv=Hv, Dk=Dk, Dv=Dv)
    kept = torch.full((B, S, C), 7.0, dtype=dt, device=DEV)
    got = G.gdn_prepare(qkv, state, conv_w, a, b, A_log, dt_bias, mask, **dims, qkv_out=kept)
    assert torch.equal(kept, qkv if mask is None else torch.where(mask[..., None], qkv, torch.zeros_like(qkv)))
    pieces, window = [], state
    for s in range(0, S, 16):
        cut = slice(s, min(s + 16, S))
        part = G.gdn_prepare(qkv[:, cut].contiguous(), window, conv_w, a[:, cut].contiguous(), b[:, cut].contiguous(), A_log,
                             dt_bias, None if mask is None else mask[:, cut].contiguous(), **dims)
        window = part[0]
        pieces.append(part[1:])
    assert torch.equal(got[0], window)
    for whole, *parts in zip(got[1:], *pieces):
        assert torch.equal(whole, torch.cat(parts, dim=1))


@pytest.mark.parametrize("name", ["bf16", "fp32"])
@pytest.mark.parametrize("B,T,Hv,Dv,state", [(1, 16, 32, 128, "fp32"), (2, 16, 8, 128, "bf16"), (1, 1030, 16, 128, "fp32"),
                                             (2, 21, 4, 64, "fp32")])
def test_output_norm_reads_a_strided_gate(native_lib, name, B, T, Hv, Dv, state):
    """z as the columns of a joint product, through the block kernel, the prompt kernels and the norm of its own."""
    from dflash_mlx_amd.kernels import gated_delta_kernel_with_tape

    dt = TORCH[name]
    gen = torch.Generator(device=DEV).manual_seed(T)
    r = lambda *s: torch.randn(s, generator=gen, device=DEV)  # noqa: E731
    q, k, v = (r(B, T, h, Dv).mul(0.1).to(dt) for h in (Hv, Hv, Hv))
    g, beta = torch.rand((B, T, Hv), generator=gen, device=DEV), torch.sigmoid(r(B, T, Hv)).to(dt)
    joint = r(B, T, 96 + Hv * Dv + 32).to(dt)
    z = joint[..., 96:96 + Hv * Dv].reshape(B, T, Hv, Dv)
    assert not z.is_contiguous()
    weight, s0 = (1 + 0.1 * r(Dv)).to(dt), r(B, Hv, Dv, Dv).to(TORCH[state])
    got = gated_delta_kernel_with_tape(q, k, v, g, beta, s0, output_norm=(z, weight, 1e-6))
    want = gated_delta_kernel_with_tape(q, k, v, g, beta, s0, output_norm=(z.contiguous(), weight, 1e-6))
    assert all(torch.equal(x, y) for x, y in zip(got, want))
    plain = gated_delta_kernel_with_tape(q, k, v, g, beta, s0)[0]
    pieces = [G.gated_norm(plain[:, t:t + 16], z[:, t:t + 16], weight) for t in range(0, T, 16)]
    assert torch.equal(G.gated_norm(plain, z, weight), torch.cat(pieces, dim=1))
    assert torch.allclose(got[0].float(), torch.cat(pieces, dim=1).float(), rtol=4 * ULP[name], atol=1e-4)


class _Given(torch.nn.Module):
    def __init__(self, out):
        super().__init__()
        self.out = out

    def forward(self, x):
        return self.out


@pytest.mark.gpu
@pytest.mark.parametrize("state_dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("B,S,Hk,Hv,D,joint", [(1, 1, 2, 4, 128, True), (2, 16, 2, 2, 128, True), (1, 5, 1, 3, 128, False), (1, 2, 2, 4, 64, True),
                                               (3, 16, 1, 2, 64, False), (1, 15, 2, 4, 64, True), (1, 3, 4, 256, 128, True),
                                               (1, 16, 16, 512, 64, True)])
def test_a_block_in_one_launch(monkeypatch, state_dtype, B, S, Hk, Hv, D, joint):
    """The bits of the prepare kernel followed by the recurrence, for every state type, tokens fewer than taps, one row per lane and
    two, with and without windows, tapes, norms, joint products and fp32 gates; forms it does not have are left to them."""
    import dflash_mlx_amd._native as nat
    from dflash_mlx_amd import gdn_layer as G
    from dflash_mlx_amd.recurrent_rollback_cache import RecurrentRollbackCache

    gen = torch.Generator("cuda").manual_seed(S + D)

    def r(*shape, std=1.0, to=torch.bfloat16):
        return (torch.randn(shape, generator=gen, device="cuda") * std).to(to)

    C = 2 * Hk * D + Hv * D
    cut = (C, Hv * D, Hv, Hv)
    parts = r(B, S, sum(cut) + 8 - sum(cut) % 8)[..., :sum(cut)].split(cut, dim=-1) if joint else [r(B, S, n) for n in cut]
    mixer = G.GatedDeltaNet(8, num_k_heads=Hk, num_v_heads=Hv, head_k_dim=D, head_v_dim=D, in_proj_qkv=_Given(parts[0]),
                            in_proj_z=_Given(parts[1]), in_proj_b=_Given(parts[2]), in_proj_a=_Given(parts[3]),
                            out_proj=torch.nn.Identity()).cuda()
    mixer.conv1d.weight.data = r(C, 4, 1, std=0.5)
    mixer.norm.weight.data = 1 + r(D, std=0.1)
    x, window, state = torch.zeros((B, S, 8), device="cuda"), r(B, 3, C), r(B, Hv, D, D, std=0.1, to=state_dtype)
    served = []

    class Watched:
        def __init__(self, block):
            self.block = block

        def __call__(self):
            return self

        def __getattr__(self, name):
            def call(*args):
                out = None if name == "gdn_block" and not self.block else getattr(real, name)(*args)
                if name == "gdn_block" and self.block:
                    served.append(out is not None)
                return out

            return call

    real = nat.host()

    def run(block, window, state, record, mask=None):
        cache = RecurrentRollbackCache(size=2, conv_kernel_size=4)
        cache[0], cache[1] = window, state
        with monkeypatch.context() as m:
            m.setattr(nat, "host", Watched(block))
            if record:
                cache.arm_rollback()
            y = G._gdn_call(mixer, x, mask, cache, record)
        return y, cache[0], cache[1], cache._tape, cache._tape_k, cache._tape_g, cache._tape_qkv

    def same(expected, *args):
        del served[:]
        for got, want in zip(run(True, *args), run(False, *args)):
            assert (got is None) == (want is None)
            assert got is None or (got.shape == want.shape and got.dtype == want.dtype and torch.equal(got, want))
        assert served == expected

    for record in (True, False):
        same([True], window, state, record)
        same([True], None, None if state_dtype == torch.bfloat16 else state, record)
    for dtype in (torch.float32, torch.bfloat16):
        mixer.A_log.data, mixer.dt_bias.data = r(Hv, to=dtype), r(Hv, std=0.3, to=dtype)
        same([True], window, state, True)
    mixer.norm.weight.data = mixer.norm.weight.data.float()
    same([True], window, state, False)
    monkeypatch.setenv("DFLASH_GDN_FUSED_NORM", "0")
    same([True], window, state, False)
    monkeypatch.delenv("DFLASH_GDN_FUSED_NORM")
    same([], window, state, True, torch.ones((B, S), dtype=torch.bool, device="cuda"))
    shifted = torch.zeros(state.numel() + 1, dtype=state.dtype, device="cuda")
    shifted[1:] = state.reshape(-1)
    same([False], window, shifted[1:].view(state.shape), True)


@pytest.mark.parametrize("S", [3, 4, 6, 7, 8, 9, 13, 15])
def test_a_block_whose_last_wave_of_steps_is_not_full(monkeypatch, S):
    """Four steps to a wave, two to a lane: blocks that end at and within either, the kernels for both kinds of state."""
    for state_dtype in (torch.float32, torch.bfloat16):
        test_a_block_in_one_launch(monkeypatch, state_dtype, 1, S, 2, 4, 128, True)


@pytest.mark.parametrize("S", [1, 3, 4, 5, 13, 16])
@pytest.mark.parametrize("B,Hk,Hv", [(9, 16, 32), (1, 1, 258)])
def test_a_block_of_more_heads_than_compute_units(monkeypatch, S, B, Hk, Hv):
    """From 257 heads of fp32 states on a head is four waves' work, two heads at a time: the bits of the other form's parts."""
    test_a_block_in_one_launch(monkeypatch, torch.float32, B, S, Hk, Hv, 128, True)


@pytest.mark.parametrize("T,D,times", [(17, 128, 1), (40, 64, 1), (33, 128, 40)])
@pytest.mark.parametrize("normed", [True, False])
def test_a_prompt_that_starts_from_nothing(native_lib, T, D, times, normed):
    """No state is the state of zeros, bit for bit; what cannot start without one is left to the caller."""
    import dflash_mlx_amd._native as nat

    gen = torch.Generator("cuda").manual_seed(T)
    B, Hk, Hv = times, 1, 2
    q, k, v = (torch.randn((B, T, h, D), generator=gen, device=DEV).to(torch.bfloat16) * D ** -0.5 for h in (Hk, Hk, Hv))
    g, beta = torch.rand((B, T, Hv), generator=gen, device=DEV), torch.rand((B, T, Hv), generator=gen, device=DEV).to(torch.bfloat16)
    z, weight = torch.randn((B, T, Hv, D), generator=gen, device=DEV).to(torch.bfloat16), torch.ones(D, device=DEV, dtype=torch.bfloat16)
    norm = (z, weight, 1e-6) if normed else (None, None, 0.0)
    run = lambda state, *cut: nat.host().gdn_forward(*(t[:, :cut[0]].contiguous() if cut else t for t in (q, k, v, g, beta)), state,  # noqa: E731
                                                     *(norm if not cut else (None, None, 0.0)), True)
    zeros = torch.zeros((B, Hv, D, D), dtype=torch.bfloat16, device=DEV)
    for a, b in zip(run(None), run(zeros)):
        assert a.dtype == b.dtype and torch.equal(a, b)
    assert run(None, 16) is None and run(zeros, 16) is not None


@pytest.mark.parametrize("B,S,Hk,Hv,D,K,masked", [(1, 39, 16, 32, 128, 4, False), (1, 40, 16, 32, 128, 4, True), (1, 257, 16, 32, 128, 4, False),
                                                  (2, 41, 16, 32, 128, 3, True), (90, 2, 8, 16, 64, 4, True), (1, 515, 2, 4, 256, 2, False)])
def test_several_heads_per_wave(native_lib, B, S, Hk, Hv, D, K, masked):
    """Where several heads share a wave (640 waves of them and more), an odd or even number of tokens to each: the bits of one
    token and head per wave."""
    for name in ("bf16", "fp16"):
        test_long_prompts_and_strided_projections(native_lib, name, B, S, Hk, Hv, D, D, K, masked)


@pytest.mark.parametrize("B,S,Hk,Hv,D,K,masked", [(1, 321, 4, 8, 64, 4, False), (1, 700, 4, 8, 64, 3, True), (1, 645, 2, 4, 128, 4, True), (2, 643, 1, 2, 256, 2, False)])
def test_query_and_key_heads_in_one_wave(native_lib, B, S, Hk, Hv, D, K, masked):
    """Fewer q heads than a wave has room for: the same bits."""
    for name in ("bf16", "fp16"):
        test_long_prompts_and_strided_projections(native_lib, name, B, S, Hk, Hv, D, D, K, masked)


@pytest.mark.parametrize("name", ["bf16", "fp16"])
def test_activations_of_every_16_bit_number(native_lib, name):
    """The sigmoid behind beta, the conv's and the norm's silu and the attention's gate, for all 65536 numbers of the type.  Its fp32
    value is within two units of fp32 (one of the exponential, a half each of the sum and the quotient), so what is stored is the
    exact sigmoid's rounding or, where that is a tie to 2^-23, its other neighbour - down to the type's subnormal numbers."""
    from dflash_mlx_amd.attention_layer import GatedAttention, _finish

    dt = TORCH[name]
    every = torch.arange(-2 ** 15, 2 ** 15, dtype=torch.int32).to(torch.int16).view(dt)
    x64 = every.double()
    grow = torch.exp(-x64.abs())
    exact = torch.where(x64 < 0, grow, 1.0) / (1 + grow)
    slack = 2.0 ** -23 * exact
    rounded = [(v.clamp_min(0)).float().to(dt) for v in (exact - slack, exact + slack)]
    number = ~torch.isnan(x64)

    def check(got, low, high, what):
        got = got.cpu()
        assert torch.isnan(got[~number]).all(), what
        g, a, b = got[number].double(), low[number].double(), high[number].double()
        nan = torch.isnan(a) | torch.isnan(b)
        assert torch.equal(torch.isnan(g), nan), what
        wrong = ~nan & ~((g >= torch.minimum(a, b)) & (g <= torch.maximum(a, b)))
        assert not wrong.any(), (what, every[number][wrong][:8].tolist(), g[wrong][:8].tolist())

    silu = [(every.float() * s.float()).to(dt) for s in rounded]
    d = every.to(DEV)
    zeros = lambda *s: torch.zeros(s, dtype=dt, device=DEV)  # noqa: E731
    params = [zeros(1024), zeros(1024)]
    # beta: 1024 value heads, 64 tokens in one run; v: 1024 heads of 64, one token (and its conv only the last tap)
    dims = dict(Hk=1, Hv=1024, Dk=64, Dv=64)
    C = 128 + 1024 * 64
    taps = zeros(C, 4)
    taps[:, 3] = 1
    beta = G.gdn_prepare(zeros(1, 64, C), None, taps, zeros(1, 64, 1024), d.view(1, 64, 1024), *params, **dims)[5]
    check(beta.reshape(-1), *rounded, "beta")
    v = G.gdn_prepare(torch.cat([zeros(128), d]).view(1, 1, C), zeros(1, 3, C), taps, zeros(1, 1, 1024), zeros(1, 1, 1024), *params, **dims)[3]
    check(v.reshape(-1), *silu, "silu of the conv")
    # the norm of a row of ones, with eps 0, is the weight: 1
    normed = G.gated_norm(torch.ones((1024, 64), dtype=dt, device=DEV), d.view(1024, 64), torch.ones(64, dtype=dt, device=DEV), 0.0)
    check(normed.reshape(-1), *silu, "silu of the norm")
    # the gate of 64 heads of 128 behind an output of ones
    attn = GatedAttention(num_attention_heads=64, num_key_value_heads=64, head_dim=128, q_proj=None, k_proj=None, v_proj=None,
                          o_proj=torch.nn.Identity())
    gate = torch.cat([zeros(8, 64, 128), d.view(8, 64, 128)], dim=-1).view(1, 8, 64 * 256)
    check(_finish(attn, torch.ones((1, 64, 8, 128), dtype=dt, device=DEV), gate).reshape(-1), *rounded, "gate of the attention")


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("S,armed", [(1, False), (5, True), (16, True), (40, True), (40, False)])
@pytest.mark.parametrize("shifted", ["weight", "gate", "neither"])
def test_operands_that_start_on_any_element(native_lib, dtype, S, armed, shifted):
    """The output norm's weight, or its gate, off the 16-byte grid: the same call, with or without a state and a tape.  A block whose
    one launch declines it is the prepare kernel and the recurrence, whose bits are the same."""
    gen = torch.Generator(DEV).manual_seed(S)
    Hk, Hv, D = 2, 4, 128
    C = 2 * Hk * D + Hv * D

    def r(*shape, std=1.0):
        return (torch.randn(shape, generator=gen, device=DEV) * std).to(dtype)

    def off(t):
        return torch.cat([t.reshape(-1)[:1], t.reshape(-1)])[1:].view(t.shape)

    parts = [r(1, S, n) for n in (C, Hv * D, Hv, Hv)]
    weight, taps, window, s0 = 1 + r(D, std=0.1), r(C, 4, 1, std=0.5), r(1, 3, C), r(1, Hv, D, D, std=0.1)

    def run(shift, state):
        z = off(parts[1]) if shift == "gate" else parts[1]
        mixer = G.GatedDeltaNet(8, num_k_heads=Hk, num_v_heads=Hv, head_k_dim=D, head_v_dim=D, in_proj_qkv=_Given(parts[0]),
                                in_proj_z=_Given(z), in_proj_b=_Given(parts[2]), in_proj_a=_Given(parts[3]),
                                out_proj=torch.nn.Identity()).to(DEV)
        mixer.conv1d.weight.data, mixer.norm.weight.data = taps, off(weight) if shift == "weight" else weight
        assert (mixer.norm.weight.data_ptr() % 16 != 0) == (shift == "weight")
        cache = RecurrentRollbackCache(size=2, conv_kernel_size=4)
        if state:
            cache[0], cache[1] = window, s0
        if armed:
            cache.arm_rollback()
        y = G._gdn_call(mixer, torch.zeros((1, S, 8), device=DEV, dtype=dtype), None, cache, armed)
        return y, cache[0], cache[1], cache._tape

    for state in (False, True):
        for a, b in zip(run(shifted, state), run("neither", state)):
            assert (a is None) == (b is None)
            assert a is None or (a.shape == b.shape and a.dtype == b.dtype and torch.equal(a, b))


def test_a_first_block_makes_its_zeros_once(native_lib, monkeypatch):
    """A block that starts from nothing has its state of zeros filled once, also where the launch of the whole block declines it."""
    filled = []
    real = torch.zeros
    monkeypatch.setattr(torch, "zeros", lambda *a, **kw: (filled.append(a), real(*a, **kw))[1])
    for dtype, K in ((torch.float32, 4), (torch.bfloat16, 3), (torch.bfloat16, 4)):
        parts = [torch.randn((1, 5, n), device=DEV).to(dtype) for n in (512, 256, 2, 2)]
        mixer = G.GatedDeltaNet(8, num_k_heads=1, num_v_heads=2, head_k_dim=128, head_v_dim=128, in_proj_qkv=_Given(parts[0]),
                                in_proj_z=_Given(parts[1]), in_proj_b=_Given(parts[2]), in_proj_a=_Given(parts[3]),
                                out_proj=torch.nn.Identity(), conv_kernel_size=K, dtype=dtype).to(DEV)
        x = torch.randn((1, 5, 8), device=DEV).to(dtype)
        cache = RecurrentRollbackCache(size=2, conv_kernel_size=K)
        del filled[:]
        mixer(x, cache=cache)
        assert len(filled) <= 1 and cache[1].dtype == dtype, (dtype, K, filled)
