"""The one-launch glue of a gated attention layer (dflash_attn_prepare, dflash_attn_gate) against the array operators of the
same layer, and both against float64, at the edges of its range: one token, ragged prompts, every head size,
partial rotation, strided projections, caches that grow."""
import pytest
import torch

from dflash_mlx_amd import attention_layer as A
from dflash_mlx_amd.cache import KVCache

pytestmark = pytest.mark.gpu


class _Given(torch.nn.Module):
    """A projection whose output is given: columns lo .. hi of a joint product."""

    def __init__(self, out):
        super().__init__()
        self.out = out

    def forward(self, x):
        return self.out


def _layer(B, L, Hq, Hk, D, dims, dtype, wdtype, gen, joint):
    widths = (2 * Hq * D, Hk * D, Hk * D)
    full = torch.randn((B, L, sum(widths)), generator=gen, device="cuda").to(dtype)
    outs = torch.split(full, widths, dim=-1)
    if not joint:
        outs = [o.contiguous() for o in outs]
    attn = A.GatedAttention(num_attention_heads=Hq, num_key_value_heads=Hk, head_dim=D, q_proj=_Given(outs[0]),
                            k_proj=_Given(outs[1]), v_proj=_Given(outs[2]), o_proj=torch.nn.Identity(), rope_dims=dims)
    for norm in (attn.q_norm, attn.k_norm):
        norm.weight = torch.nn.Parameter((1 + 0.2 * torch.randn(D, generator=gen, device="cuda")).to(wdtype), requires_grad=False)
    return attn, outs


def _exact(head, weight, dims, offset, eps=1e-6):
    x = head.double()
    n = x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps) * weight.double()
    half = dims // 2
    freq = 10000.0 ** (-torch.arange(half, device=x.device, dtype=torch.float64) / half)
    angle = torch.arange(offset, offset + x.shape[1], device=x.device, dtype=torch.float64)[:, None] * freq
    c, s = torch.cos(angle)[None, :, None], torch.sin(angle)[None, :, None]
    a, b = n[..., :half], n[..., half:dims]
    return torch.cat([a * c - b * s, a * s + b * c, n[..., dims:]], dim=-1).transpose(1, 2)


@pytest.mark.parametrize("B,L,Hq,Hk,D,dims,prefix,dtype,wdtype,joint", [
    (1, 16, 32, 8, 256, 256, 4096, torch.bfloat16, torch.bfloat16, True),
    (1, 16, 16, 4, 256, 64, 240, torch.bfloat16, torch.float32, True),      # quarter rotation; the cache grows here
    (1, 1, 64, 8, 128, 128, 32700, torch.float16, torch.float16, False),    # one token, long angles
    (2, 77, 8, 2, 64, 64, 0, torch.bfloat16, torch.bfloat16, True),         # empty cache, two sequences
    (1, 5, 3, 1, 192, 96, 7, torch.float16, torch.bfloat16, False),         # three features per lane
    (1, 1030, 24, 4, 256, 256, 3, torch.bfloat16, torch.bfloat16, True),    # several heads per wave
])
def test_prepare_equals_the_array_operators(monkeypatch, B, L, Hq, Hk, D, dims, prefix, dtype, wdtype, joint):
    gen = torch.Generator(device="cuda").manual_seed(11)
    attn, outs = _layer(B, L, Hq, Hk, D, dims, dtype, wdtype, gen, joint)
    x = torch.empty((B, L, 8), device="cuda")
    before = [torch.randn((B, Hk, prefix, D), generator=gen, device="cuda").to(dtype) for _ in range(2)]
    caches = [KVCache(), KVCache()]
    for c in caches:
        if prefix:
            c.update_and_fetch(*before)
    queries, keys, values, gate, prev = A._project(attn, x, caches[0])
    assert gate is not None and gate.shape[-1] == 2 * Hq * D and prev == prefix  # the kernel took it
    monkeypatch.setattr(A, "_project_on_device", lambda *a: None)
    ref_q, ref_k, ref_v, ref_gate, _ = A._project(attn, x, caches[1])
    assert caches[0].offset == caches[1].offset == prefix + L and caches[0].keys.shape == caches[1].keys.shape
    assert torch.equal(values, ref_v) and torch.equal(keys[:, :, :prefix], ref_k[:, :, :prefix])
    # the sum of squares is taken in another order: a normed feature may fall on the next value of the type (eps of itself),
    # a turned one is the sum of two of them, rounded once more
    eps = torch.finfo(dtype).eps
    for got, ref, head, norm in ((queries, ref_q, outs[0].reshape(B, L, Hq, 2 * D)[..., :D], attn.q_norm),
                                 (keys[:, :, prefix:], ref_k[:, :, prefix:], outs[1].reshape(B, L, Hk, D), attn.k_norm)):
        exact = _exact(head, norm.weight, dims, prefix)
        size = exact.abs()
        pair = size.clone()
        pair[..., :dims // 2] += size[..., dims // 2:dims]
        pair[..., dims // 2:dims] += size[..., :dims // 2]
        assert ((got.double() - ref.double()).abs() <= 3 * eps * 1.5 * pair + 1e-6).all()
        err = [((t.double() - exact).norm() / exact.norm()).item() for t in (got, ref)]
        assert err[0] <= 1.01 * err[1]
    out = torch.randn((B, L, Hq, D), generator=gen, device="cuda").to(dtype)
    for o in (out.transpose(1, 2), out.transpose(1, 2).contiguous()):  # either order an attention may leave
        assert torch.equal(A._finish(attn, o, gate), A._finish(attn, o, ref_gate))


def test_what_the_kernel_does_not_cover_goes_to_the_array_operators():
    gen = torch.Generator(device="cuda").manual_seed(12)
    x = torch.empty((1, 4, 8), device="cuda")
    for change in ("hook", "cache", "grad", "fp32", "odd"):
        dtype = torch.float32 if change == "fp32" else torch.bfloat16
        attn, outs = _layer(1, 4, 4, 2, 96 if change == "odd" else 128, 64, dtype, dtype, gen, True)
        cache = KVCache()
        if change == "hook":
            attn.q_norm.register_forward_hook(lambda m, i, o: o)
        if change == "cache":
            cache = type("Other", (KVCache,), {})()
        if change == "grad":
            attn.q_proj.out = outs[0].clone().requires_grad_(True)
        queries, keys, _, gate, _ = A._project(attn, x, cache)
        assert gate.shape[-1] == queries.shape[1] * queries.shape[-1], change
        assert queries.requires_grad == (change == "grad")


@pytest.mark.parametrize("broken", ["values shorter", "offset behind the end", "offset without buffers", "negative offset"])
def test_rows_outside_the_cache_are_left_to_the_array_operators(monkeypatch, broken):
    """Buffers and offsets that do not belong together never reach the kernel: the caller gets what the array operators
    make of them, an error where the rows do not fit."""
    gen = torch.Generator(device="cuda").manual_seed(14)
    attn, _ = _layer(1, 16, 4, 2, 128, 128, torch.bfloat16, torch.bfloat16, gen, True)
    x = torch.empty((1, 16, 8), device="cuda")

    def launched(*args):
        raise AssertionError("the kernel was launched")

    monkeypatch.setattr(A._native.lib(), "dflash_attn_prepare", launched)
    cache = KVCache()
    if broken != "offset without buffers":
        cache.update_and_fetch(*(torch.zeros((1, 2, 100, 128), dtype=torch.bfloat16, device="cuda") for _ in range(2)))
    if broken == "values shorter":
        cache.values = cache.values[:, :, :100].contiguous()
    elif broken == "negative offset":
        cache.offset = -20
    else:
        cache.offset = 1000
    if broken == "negative offset":  # (they count from the end)
        assert A._project(attn, x, cache)[4] == -20 and cache.offset == -4
        return
    with pytest.raises(RuntimeError):
        A._project(attn, x, cache)


@pytest.mark.parametrize("B,Hq,Hk,D,N,dtype,masked,joint", [
    (1, 32, 8, 256, 4112, torch.bfloat16, False, True), (2, 16, 2, 128, 257, torch.float16, False, False),
    (1, 24, 4, 256, 1040, torch.bfloat16, True, True), (3, 5, 1, 128, 300, torch.bfloat16, False, True)])
def test_gate_behind_the_attention(B, Hq, Hk, D, N, dtype, masked, joint):
    """The gate where the key ranges meet: the bits of the attention followed by the gate of its own."""
    from dflash_mlx_amd.kernels import batched_sdpa_2pass_exact

    gen = torch.Generator(device="cuda").manual_seed(13)
    attn, outs = _layer(B, 16, Hq, Hk, D, D, dtype, dtype, gen, joint)
    q = torch.randn((B, Hq, 16, D), generator=gen, device="cuda").to(dtype)
    k, v = (torch.randn((B, Hk, N, D), generator=gen, device="cuda").to(dtype) for _ in range(2))
    mask = torch.randn((B, 1, 16, N), generator=gen, device="cuda").to(dtype) if masked else None
    plain = batched_sdpa_2pass_exact(q, k, v, D ** -0.5, mask)
    gated = batched_sdpa_2pass_exact(q, k, v, D ** -0.5, mask, q_proj_output=outs[0])
    assert gated.shape == (B, 16, Hq * D) and torch.equal(gated, A._finish(attn, plain, outs[0]))
    # one range of keys: nothing to ride on, the plain result
    short = batched_sdpa_2pass_exact(q, k[:, :, :100], v[:, :, :100], D ** -0.5, q_proj_output=outs[0])
    assert torch.equal(short, batched_sdpa_2pass_exact(q, k[:, :, :100], v[:, :, :100], D ** -0.5))


def test_a_refused_launch_leaves_the_cache_where_it_was(monkeypatch):
    gen = torch.Generator(device="cuda").manual_seed(15)
    attn, _ = _layer(1, 16, 4, 2, 128, 128, torch.bfloat16, torch.bfloat16, gen, True)
    x = torch.empty((1, 16, 8), device="cuda")
    for prefix in (0, 250):  # no buffers yet; buffers that are too short for the block
        cache = KVCache()
        before = [torch.randn((1, 2, prefix, 128), generator=gen, device="cuda").to(torch.bfloat16) for _ in range(2)]
        if prefix:
            cache.update_and_fetch(*before)
        with monkeypatch.context() as m:
            m.setattr(A._native.lib(), "dflash_attn_prepare", lambda *args: -1)
            with pytest.raises(A._native.NativeLibraryError):
                A._project(attn, x, cache)
        assert cache.offset == prefix
        _, keys, _, _, at = A._project(attn, x, cache)
        assert at == prefix and cache.offset == prefix + 16 and keys.shape[2] == prefix + 16
        if prefix:
            assert torch.equal(keys[:, :, :prefix], before[0])


@pytest.mark.parametrize("D,dims", [(128, 128), (128, 96), (192, 192), (192, 96), (256, 104), (64, 20)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_bits_of_the_array_operators_where_the_norms_sum_is_exact(monkeypatch, D, dims, dtype):
    """Small whole numbers: their squares add up exactly in any order, so that every bit that is left to differ is
    the rotation's or a rounding's."""
    gen = torch.Generator(device="cuda").manual_seed(16)
    attn, outs = _layer(1, 40, 6, 2, D, dims, dtype, dtype, gen, True)
    for o in outs:
        o.copy_(torch.randint(-8, 9, o.shape, generator=gen, device="cuda"))
    x = torch.empty((1, 40, 8), device="cuda")
    caches = [KVCache(), KVCache()]
    for c in caches:
        c.update_and_fetch(*(torch.zeros((1, 2, 3001, D), dtype=dtype, device="cuda") for _ in range(2)))
    got = A._project(attn, x, caches[0])
    assert got[3].shape[-1] == 2 * 6 * D  # the kernel took it
    monkeypatch.setattr(A, "_project_on_device", lambda *a: None)
    want = A._project(attn, x, caches[1])
    for a, b in zip(got[:3], want[:3]):
        assert torch.equal(a, b)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_both_gates_on_every_number(dtype):
    """The gate where the key ranges meet and the gate of its own, for all 65536 numbers of the type."""
    from dflash_mlx_amd.kernels import batched_sdpa_2pass_exact

    gen = torch.Generator(device="cuda").manual_seed(3)
    Hq, D, N = 32, 128, 400
    every = torch.arange(-2 ** 15, 2 ** 15, dtype=torch.int32).to(torch.int16).view(dtype).cuda().view(16, Hq, D)
    projected = torch.cat([torch.zeros_like(every), every], dim=-1).view(1, 16, Hq * 2 * D)
    attn, _ = _layer(1, 16, Hq, 8, D, D, dtype, dtype, gen, False)
    q = torch.randn((1, Hq, 16, D), generator=gen, device="cuda").to(dtype)
    k, v = (torch.randn((1, 8, N, D), generator=gen, device="cuda").to(dtype) for _ in range(2))
    gated = batched_sdpa_2pass_exact(q, k, v, D ** -0.5, q_proj_output=projected)
    assert gated.shape == (1, 16, Hq * D)
    want = A._finish(attn, batched_sdpa_2pass_exact(q, k, v, D ** -0.5), projected)
    nan = torch.isnan(want)
    assert torch.equal(torch.isnan(gated), nan) and torch.equal(gated[~nan], want[~nan])


def _block_layer(*args):
    """A layer whose verify blocks take the exact path behind any prefix."""
    attn, outs = _layer(*args)
    attn.q_proj.weight = torch.empty((outs[0].shape[-1], 1), device="cuda")  # (its height says that a gate rides along)
    A.configure_full_attention_split([type("L", (), {"is_linear": False, "self_attn": attn})()], enabled=True)
    attn._dflash_split_sdpa_exact_kv_threshold = 1
    return attn, outs


@pytest.mark.parametrize("B,Hq,Hk,D,dims,prefix,dtype,joint", [
    (1, 32, 8, 256, 256, 4096, torch.bfloat16, True),
    (1, 16, 2, 128, 128, 1025, torch.float16, True),    # eight heads of a key head, an odd prefix
    (2, 3, 1, 128, 64, 1039, torch.bfloat16, False),    # three heads, half of the features turned
    (1, 4, 4, 256, 64, 130, torch.float16, False),      # waves share a head four ways
    (1, 6, 2, 256, 128, 90, torch.bfloat16, True),      # one range: the launch has no form
    (1, 4, 2, 128, 128, 112, torch.bfloat16, True),
    (1, 6, 2, 256, 128, 1024, torch.bfloat16, True),    # the last range without a cached key
    (1, 4, 2, 128, 128, 1020, torch.bfloat16, True),    # ... with 12 of the block's own, four are the range's before it
    (2, 16, 2, 128, 64, 1015, torch.bfloat16, True),    # ... with seven
    (1, 8, 2, 256, 256, 250, torch.float16, False),     # the block's keys begin in one tile and end in the next
    (1, 32, 8, 256, 256, 32700, torch.bfloat16, True),
    (2, 16, 2, 128, 64, 1015, torch.float16, True),     # a key feature whose product falls between two numbers of fp16 once in fp32
    (8, 16, 16, 256, 64, 200, torch.float16, True),     # 524288 key features, one in 8192 of them such a one
])
def test_block_from_its_projections_in_the_launch_of_its_attention(monkeypatch, B, Hq, Hk, D, dims, prefix, dtype, joint):
    """Against the launch of its own for norms, rotation and cache rows, which is what a cache without room for the block
    takes: the same rows in the cache and the same bits of the attention, as close to 64 bits."""
    gen = torch.Generator(device="cuda").manual_seed(21)
    attn, outs = _block_layer(B, 16, Hq, Hk, D, dims, dtype, dtype, gen, joint)
    x = torch.empty((B, 16, 8), device="cuda")
    before = [torch.randn((B, Hk, prefix, D), generator=gen, device="cuda").to(dtype) for _ in range(2)]
    fused, real = [], A._native.host().attn_block
    results = []
    for in_one in (True, None, False):  # (None: no room)
        if in_one is False:
            monkeypatch.setattr(A, "_attend_in_one", lambda *a: None)
        elif in_one:
            spy = type("H", (), {"__getattr__": lambda self, n, h=A._native.host(): getattr(h, n),
                                 "attn_block": lambda self, *a: fused.append(real(*a)) or fused[-1]})()
            monkeypatch.setattr(A._native, "host", lambda: spy)
        cache = KVCache()
        cache.update_and_fetch(*before)
        if in_one is None:
            cache.keys, cache.values = (t[:, :, :prefix].contiguous() for t in (cache.keys, cache.values))
        elif cache.keys.shape[2] < prefix + 16:
            cache._make_room(B, Hk, 16, D, D, *before)
        y = attn(x, mask="causal" if in_one else None, cache=cache)
        assert cache.offset == prefix + 16
        results.append((y, *cache.state))
    assert fused and (fused[-1] is not None) == (prefix + 16 > 128)
    (got, keys, values), grown, (ref, ref_keys, ref_values) = results
    assert torch.equal(keys, ref_keys) and torch.equal(values, ref_values)
    assert torch.equal(got, ref) and all(torch.equal(a, b) for a, b in zip(grown, results[2]))
    q = A.rms_norm_ops(outs[0].reshape(B, 16, Hq, 2 * D)[..., :D], attn.q_norm.weight, attn.q_norm.eps).transpose(1, 2)
    q = attn.rope(q, offset=prefix).double()
    k, v = (t.double().repeat_interleave(Hq // Hk, dim=1) for t in (ref_keys, ref_values))
    scores = torch.matmul(q, k.transpose(2, 3).contiguous()) * attn.scale
    late = torch.arange(prefix + 16, device="cuda") > prefix + torch.arange(16, device="cuda")[:, None]
    o = torch.matmul(torch.softmax(scores.masked_fill(late, float("-inf")), dim=-1), v).transpose(1, 2)
    exact = (o * torch.sigmoid(outs[0].reshape(B, 16, Hq, 2 * D)[..., D:].double())).reshape(B, 16, Hq * D)
    err = [((t.double() - exact).norm() / exact.norm()).item() for t in (got, ref)]
    # (partial outputs, the output, the gate and their product are rounded to the type, each by eps / sqrt(48) on average)
    assert err[0] <= max(1.1 * err[1], 4 * torch.finfo(dtype).eps / 48 ** 0.5), err


def test_what_the_block_launch_does_not_cover_takes_the_launch_of_its_own(monkeypatch):
    """One range of keys, a rotation of 96 features, weights of another type, rows at odd addresses, a mask, no room."""
    for change in ("short", "rotation", "weights", "address", "mask", "room", "none"):
        gen = torch.Generator(device="cuda").manual_seed(22)
        prefix = 50 if change == "short" else 240 if change != "room" else 250
        attn, outs = _block_layer(1, 16, 4, 2, 128, 96 if change == "rotation" else 128, torch.bfloat16,
                                  torch.float32 if change == "weights" else torch.bfloat16, gen, True)
        if change == "address":
            attn.k_proj.out = torch.empty(16 * 256 + 4, dtype=torch.bfloat16, device="cuda")[4:].view(1, 16, 256).copy_(outs[1])
        cache = KVCache()
        cache.update_and_fetch(*(torch.randn((1, 2, prefix, 128), generator=gen, device="cuda").to(torch.bfloat16) for _ in range(2)))
        took = []
        real = A._attend_in_one
        with monkeypatch.context() as m:
            m.setattr(A, "_attend_in_one", lambda *a: took.append(real(*a)) or took[-1])
            mask = torch.zeros((1, 1, 16, prefix + 16), dtype=torch.bfloat16, device="cuda") if change == "mask" else "causal"
            y = attn(torch.empty((1, 16, 8), device="cuda"), mask=mask, cache=cache)
        assert y.shape == (1, 16, 4 * 128) and cache.offset == prefix + 16
        assert (not took or took[-1] is None) == (change != "none"), change


def test_a_refused_block_launch_leaves_the_cache_where_it_was(monkeypatch):
    gen = torch.Generator(device="cuda").manual_seed(23)
    attn, _ = _block_layer(1, 16, 4, 2, 128, 128, torch.bfloat16, torch.bfloat16, gen, True)
    cache = KVCache()
    cache.update_and_fetch(*(torch.zeros((1, 2, 240, 128), dtype=torch.bfloat16, device="cuda") for _ in range(2)))

    def refused(**kw):
        raise A._native.NativeLibraryError("refused")

    monkeypatch.setattr(A, "batched_sdpa_2pass_exact", refused)
    with pytest.raises(A._native.NativeLibraryError):
        attn(torch.empty((1, 16, 8), device="cuda"), mask="causal", cache=cache)
    assert cache.offset == 240
