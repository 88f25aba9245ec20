"""The native launch path: the bits of the Python it stands in for, over every form of a call; errors stay errors."""
import pytest
import torch

import dflash_mlx_amd._native as nat
from dflash_mlx_amd import gdn_layer as G
from dflash_mlx_amd import kernels as KN
from dflash_mlx_amd import verify_linear as VL
from dflash_mlx_amd import verify_qmm as VQ
from dflash_mlx_amd.recurrent_rollback_cache import RecurrentRollbackCache
from dflash_mlx_amd.workloads import make_qmm_case

BF, HF, FP = torch.bfloat16, torch.float16, torch.float32


class _Recorder:
    """Stands where ``_native.host`` does: notes which functions served a call, or lets none of them."""

    def __init__(self, serve):
        self.serve, self.served, self.real = serve, [], nat.host()

    def __call__(self):
        return self

    def __getattr__(self, name):
        def call(*args):
            out = getattr(self.real, name)(*args) if self.serve else None
            if out is not None:
                self.served.append(name)
            return out

        return call


def _outcome(monkeypatch, call, serve):
    recorder = _Recorder(serve)
    with monkeypatch.context() as m:
        m.setattr(nat, "host", recorder)
        try:
            out = call()
        except (ValueError, TypeError, RuntimeError) as error:
            return type(error), recorder.served
    torch.cuda.synchronize()
    return tuple(out) if isinstance(out, (tuple, list)) else (out,), recorder.served


def _same(monkeypatch, call, name, served):
    call()  # (a first call makes the scratch that both then find)
    got, by = _outcome(monkeypatch, call, True)
    want, none = _outcome(monkeypatch, call, False)
    assert not none and (name in by) == served, (name, by)
    _equal(got, want)


def _equal(got, want):
    if isinstance(want, type):
        assert got is want
        return
    assert len(got) == len(want)
    for a, b in zip(got, want):
        if b is None or a is None:
            assert a is b
            continue
        assert a.shape == b.shape and a.dtype == b.dtype and a.device == b.device and a.stride() == b.stride()
        assert torch.equal(a, b)


def _at(t, offset):
    """The same values ``offset`` elements behind an aligned address."""
    flat = torch.zeros(t.numel() + offset, dtype=t.dtype, device=t.device)
    flat[offset:] = t.reshape(-1)
    return flat[offset:].view(t.shape)


def _cut(t):
    """The same values as the first columns of something wider."""
    return torch.cat([t, t], dim=-1)[..., :t.shape[-1]]


def _triple(K, N, group, dtype, seed=5):
    c = make_qmm_case(K, N, seed, group_size=group).to("cuda")
    return c.w, c.scales.to(dtype), c.biases.to(dtype)


def _rows(lead, K, dtype, seed=6):
    return torch.randn((*lead, K), generator=torch.Generator("cuda").manual_seed(seed), device="cuda").to(dtype)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype,scales", [(BF, BF), (HF, HF), (BF, HF)])
@pytest.mark.parametrize("lead", [(1,), (1, 7), (2, 8), (16,), (17,), (3, 1, 30)])
@pytest.mark.parametrize("K,N,group", [(1024, 512, 64), (768, 96, 32), (640, 48, 128), (8192, 64, 64)])
def test_products(monkeypatch, dtype, scales, lead, K, N, group):
    w, s, b = _triple(K, N, group, scales)
    rows = 1
    for d in lead:
        rows *= d
    x = _rows(lead, K, dtype)
    forms = [(x, True), (torch.nn.Parameter(x, requires_grad=False), True), (_cut(x), rows == 1), (_at(x, 1), False), (_at(x, 8), True)]
    for enabled in (("0", "1") if rows == 16 else ("0",)):
        monkeypatch.setenv("DFLASH_VERIFY_QMM", enabled)
        for form, served in forms:
            if enabled == "1":
                if N % 32 == 0 and (K % 256 == 0 or not (K >= 8192 or N <= 8192)) and form.data_ptr() % 16 == 0:
                    _same(monkeypatch, lambda: VQ.verify_matmul(form, w, s, b, group_size=group), "qmm_m16", form.is_contiguous())
            elif rows <= 16:
                if rows < 16 or form.data_ptr() % 16 == 0:  # (a whole block that starts elsewhere is refused by the kernel)
                    _same(monkeypatch, lambda: VQ.small_m_matmul(form, w, s, b, group_size=group), "qmm_few",
                          form.is_contiguous() and form.data_ptr() % 16 == 0)
            if rows > 16 or form is x:
                _same(monkeypatch, lambda: VQ.rows_matmul(form, w, s, b, group_size=group), "qmm_rows",
                      form.is_contiguous() and form.data_ptr() % 16 == 0)
    # operands of another extent, type or place, and forms that are not the kernels': the same error or the same None
    call = VQ.rows_matmul if rows > 16 else VQ.small_m_matmul
    for bad in ((w[:, :-4], s, b), (w, s[:-1], b), (w, s.to(FP), b.to(FP)), (w, s, b.to(FP)), (w.cpu(), s, b), (w[None], s, b)):
        got, by = _outcome(monkeypatch, lambda: call(x, *bad, group_size=group), True)
        want, _ = _outcome(monkeypatch, lambda: call(x, *bad, group_size=group), False)
        assert not by
        _equal(got, want)
    # weights that are a view into a joint matrix, and ones that are not in one piece
    wide = [torch.cat([t, t], dim=0) for t in (w, s, b)]
    _same(monkeypatch, lambda: call(x, *(t[:N] for t in wide), group_size=group), "qmm_rows" if rows > 16 else "qmm_few", True)
    _same(monkeypatch, lambda: call(x, w, _cut(s), b, group_size=group), "qmm_rows" if rows > 16 else "qmm_few", False)


@pytest.mark.gpu
def test_products_that_something_watches(monkeypatch):
    """Calls that are differentiated, traced or batched, and subclasses, are not the native path's."""
    monkeypatch.setenv("DFLASH_VERIFY_QMM", "0")
    w, s, b = _triple(1024, 64, 64, BF)
    x = _rows((5,), 1024, BF)

    class Sub(torch.Tensor):
        pass

    for form in (x.clone().requires_grad_(True), x.as_subclass(Sub)):
        out, by = _outcome(monkeypatch, lambda: VQ.small_m_matmul(form, w, s, b), True)
        assert not by and out == (None,)
    host = nat.host()
    assert host.qmm_few(x.as_subclass(Sub), w, s, b, 64, 0, VQ._WORKSPACES) is None
    seen = []
    torch.vmap(lambda row: (seen.append(host.qmm_few(row, w, s, b, 64, 0, VQ._WORKSPACES)), row)[1])(x)
    assert seen == [None]
    assert host.columns(x.as_subclass(Sub), [(0, 4)]) is None and host.columns(x, [(0, 2000)]) is None


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [BF, HF])
@pytest.mark.parametrize("rows", [1, 16, 40])
def test_gated_activation_and_columns(monkeypatch, dtype, rows):
    from dflash_mlx_amd.quantized import QuantizedLinear

    monkeypatch.setenv("DFLASH_VERIFY_QMM", "1")
    for K, inter in ((1024, 256), (512, 96)):
        mlp = torch.nn.Module()
        for i, name in enumerate(("gate_proj", "up_proj")):
            setattr(mlp, name, QuantizedLinear(*_triple(K, inter, 64, dtype, seed=i), group_size=64, bits=4))
        model = torch.nn.Module()
        model.mlp = mlp
        assert VL.install_verify_linears(model) == 2 and VL.fuse_shared_input_linears(model) == 1
        for x in (_rows((1, rows), K, dtype), _rows((rows,), K, dtype, 8)):
            chained = rows == 16 and K % 1024 == 0
            _same(monkeypatch, lambda: VL.silu_gate_up(model.mlp, x), "chain_bind" if chained else "qmm_rows" if rows > 16
                  else "qmm_few_silu_mul", True)
            _same(monkeypatch, lambda: VL.shared_input_outputs(model.mlp, ("gate_proj", "up_proj"), x, columns=True), "columns", True)
        VL.pack_verify_linears(model)
        if rows == 16 and K % 1024 == 0:
            _same(monkeypatch, lambda: VL.shared_input_outputs(model.mlp, ("gate_proj", "up_proj"), x), "qmm_packed", True)
            _same(monkeypatch, lambda: VL.silu_gate_up(model.mlp, x), "chain_launch", True)


@pytest.mark.gpu
@pytest.mark.parametrize("pairs,E,K,N,group", [(1, 4, 512, 64, 64), (40, 8, 512, 96, 64), (300, 8, 640, 48, 32)])
def test_gathered_products(monkeypatch, pairs, E, K, N, group):
    w, s, b = (torch.stack(t) for t in zip(*(_triple(K, N, group, BF, seed=e) for e in range(E))))
    x, ids = _rows((pairs,), K, BF), torch.randint(0, E, (pairs,), device="cuda", dtype=torch.int32)
    for form, index, served in ((x, ids, True), (_cut(x), ids, pairs == 1), (x, ids.long(), False)):
        _same(monkeypatch, lambda: VQ.gather_qmm(form, w, s, b, index, group_size=group), "gather", served)
    for bad in ((x, w, s[:, :-1], b, ids), (x, w, s, b, ids[:-1]), (x, w, s, b, ids.cpu()), (x.float(), w, s, b, ids)):
        got, by = _outcome(monkeypatch, lambda: VQ.gather_qmm(*bad, group_size=group), True)
        assert not by and isinstance(got, type) and got is _outcome(monkeypatch, lambda: VQ.gather_qmm(*bad, group_size=group), False)[0]


@pytest.mark.gpu
@pytest.mark.parametrize("dtype,state_dtype", [(BF, FP), (HF, HF), (FP, FP), (BF, BF)])
@pytest.mark.parametrize("B,T,Hk,Hv,D", [(1, 1, 2, 4, 128), (2, 16, 2, 2, 64), (1, 5, 2, 4, 192), (1, 70, 4, 8, 128)])
def test_gated_delta_layer(monkeypatch, dtype, state_dtype, B, T, Hk, Hv, D):
    gen = torch.Generator("cuda").manual_seed(3)

    def r(*shape, std=1.0, to=dtype):
        return (torch.randn(shape, generator=gen, device="cuda") * std).to(to)

    C, dims = 2 * Hk * D + Hv * D, dict(Hk=Hk, Hv=Hv, Dk=D, Dv=D)
    joint = r(B, T, C + Hv * D + 2 * Hv)
    qkv, z, b, a = joint.split([C, Hv * D, Hv, Hv], dim=-1)
    taps, window, A, bias = r(C, 4, 1, std=0.5), r(B, 3, C), r(Hv, to=FP), r(Hv, to=FP)
    in_place = joint.stride(1) * joint.element_size() % 8 == 0
    for w, cs, out in ((taps, window, None), (taps[..., 0].contiguous(), None, torch.empty(B, T, C, dtype=dtype, device="cuda"))):
        _same(monkeypatch, lambda: G.gdn_prepare(qkv, cs, w, a, b, A, bias, qkv_out=out, **dims), "gdn_prepare", in_place)
    _same(monkeypatch, lambda: G.gdn_prepare(qkv.contiguous(), window, taps, a.contiguous(), b, A.to(BF), bias.to(BF), **dims), "gdn_prepare", True)
    _same(monkeypatch, lambda: G.gdn_prepare(qkv, window, taps, a, b, A, bias, torch.ones(B, T, dtype=torch.bool, device="cuda"), **dims),
          "gdn_prepare", False)
    _same(monkeypatch, lambda: G.gdn_prepare(qkv, _cut(window), taps, a, b, A, bias, **dims), "gdn_prepare", False)

    _, q, k, v, g, beta = G.gdn_prepare(qkv, window, taps, a, b, A, bias, **dims)
    state, weight, gate = r(B, Hv, D, D, std=0.1, to=state_dtype), r(D), z.reshape(B, T, Hv, D)
    for norm, tape in ((None, True), ((gate, weight, 1e-6), False), ((gate.contiguous(), weight.float(), 1e-6), True)):
        served = norm is None or (norm[0].data_ptr() | norm[0].stride(1) * norm[0].element_size() | norm[0].stride(0) * norm[0].element_size()) % 16 == 0
        call = lambda **kw: KN.gated_delta_kernel_with_tape(q, k, v, g, beta, state, output_norm=norm, with_tape=tape, **kw)  # noqa: E731
        _same(monkeypatch, call, "gdn_forward", served)
        _same(monkeypatch, lambda: call(mask=torch.ones(B, T, dtype=torch.bool, device="cuda")), "gdn_forward", False)
    _same(monkeypatch, lambda: KN.gated_delta_kernel_with_tape(q, k, v, g, beta, state.transpose(2, 3)), "gdn_forward", False)
    _same(monkeypatch, lambda: KN.gated_delta_kernel_with_tape(q, k, v, _at(g, 1), beta, _at(state, 1)), "gdn_forward", True)
    for bad in ((q, k, v, g[:, :, :-1], beta, state), (q, k, v, g, beta, state[:, :, :-1]), (q[:, :, :-1], k, v, g, beta, state)):
        got, by = _outcome(monkeypatch, lambda: KN.gated_delta_kernel_with_tape(*bad), True)
        assert not by and got is _outcome(monkeypatch, lambda: KN.gated_delta_kernel_with_tape(*bad), False)[0]

    tape = r(B, T, Hv, D, std=0.05, to=FP)

    def rolled(prev, tape=tape):
        cache = RecurrentRollbackCache(size=2, conv_kernel_size=4)
        cache[0], cache[1] = prev, state
        cache.arm_rollback()
        cache.record_tape(tape=tape, k=k, g=g, qkv=qkv)
        cache.rollback(T // 2)
        return cache[1], cache[0]

    fits = T * (3 * D + 1) * 4 + D * 4 <= 64 * 1024  # rows the replay can stage
    for prev, served in ((window, fits), (None, fits), (_cut(window), False)):
        _same(monkeypatch, lambda: rolled(prev), "rollback_layer", served)


@pytest.mark.gpu
@pytest.mark.parametrize("B,Hq,Hk,D,N,dtype", [(1, 32, 8, 256, 4112, BF), (2, 16, 2, 128, 257, HF), (1, 4, 4, 128, 20, BF)])
def test_attention_of_a_block(monkeypatch, B, Hq, Hk, D, N, dtype):
    q, kept = _rows((B, Hq, 16), D, dtype), _rows((B, Hk, N + 40), D, dtype, 9)
    k, v, gate = kept[:, :, :N], kept[:, :, 8:8 + N], _rows((B, 16), Hq * 2 * D, dtype, 10)
    turned = q.transpose(1, 2).contiguous().transpose(1, 2)
    for args, served in (((q, k, v), True), ((q, k.contiguous(), v), True), ((turned, k, v), False),
                         ((q, k.transpose(2, 3).contiguous().transpose(2, 3), v), False)):
        for extra in ({}, {"q_proj_output": gate}, {"q_proj_output": _at(gate, 1)}):
            _same(monkeypatch, lambda: KN.batched_sdpa_2pass_exact(*args, D ** -0.5, **extra), "sdpa_q16", served)
    masked = torch.zeros((B, 1, 16, N), dtype=dtype, device="cuda")
    _same(monkeypatch, lambda: KN.batched_sdpa_2pass_exact(q, k, v, D ** -0.5, masked), "sdpa_q16", False)
    for bad in ((q.float(), k, v), (q[:, :, :15], k, v), (q, k[:, :, :-1], v), (q, k.float(), v)):
        assert _outcome(monkeypatch, lambda: KN.batched_sdpa_2pass_exact(*bad, D ** -0.5), True) == ((None,), [])


def test_host_tensors_and_strangers_are_left_alone(native_lib):
    host, x = nat.host(), torch.zeros(16, 64)
    for name, count in (("qmm_m16", 7), ("qmm_packed", 9), ("qmm_few", 7), ("qmm_few_silu_mul", 7), ("qmm_rows", 7), ("columns", 2),
                        ("gather", 8), ("chain_bind", 4), ("chain_launch", 10), ("gdn_prepare", 13), ("gdn_forward", 10),
                        ("rollback_layer", 9), ("rollback_layers", 4), ("sdpa_q16", 6), ("attn_prepare", 11), ("first_rows", 3),
                        ("attn_block", 13)):
        for value in (x, x.to("meta"), None, 1, -1, 2 ** 70, 1.5, "x", {}):
            assert getattr(host, name)(*[value] * count) is None
        assert getattr(host, name)() is None


@pytest.mark.gpu
@pytest.mark.parametrize("B,L,Hq,Hk,D,rope,prefix", [(1, 16, 8, 2, 256, 256, 300), (2, 1, 4, 4, 128, 64, 5), (1, 40, 6, 3, 64, 32, 0),
                                                     (1, 16, 4, 2, 192, 192, 240)])
def test_what_stands_before_the_attention(monkeypatch, B, L, Hq, Hk, D, rope, prefix):
    from test_gpu_attn_glue import _layer

    from dflash_mlx_amd import attention_layer as A
    from dflash_mlx_amd.cache import KVCache

    gen = torch.Generator("cuda").manual_seed(4)
    attn, _ = _layer(B, L, Hq, Hk, D, rope, BF, BF, gen, True)
    x = torch.empty((B, L, 8), device="cuda")
    before = [torch.randn((B, Hk, prefix, D), generator=gen, device="cuda").to(BF) for _ in range(2)]

    def projected(served, change=None):
        cache = KVCache()
        if prefix:
            cache.update_and_fetch(*before)
        if change == "types":
            cache.keys, cache.values = cache.keys.to(HF), cache.values.to(HF)
        elif change == "order":
            cache.keys = cache.keys.transpose(2, 3).contiguous().transpose(2, 3)
        q, k, v, gate, at = A._project(attn, x, cache)
        return q, k.clone(), v.clone(), gate, torch.tensor([at, cache.offset])

    room = 0 < prefix and prefix + L <= -(-prefix // 256) * 256
    _same(monkeypatch, lambda: projected(room), "attn_prepare", room)
    if prefix:
        for change in ("types", "order"):
            _same(monkeypatch, lambda: projected(False, change), "attn_prepare", False)


@pytest.mark.gpu
@pytest.mark.parametrize("B,S,Hk,Hv,D,record", [(1, 1, 2, 4, 128, True), (1, 16, 2, 2, 64, True), (1, 16, 2, 4, 128, False), (2, 3, 1, 3, 64, True)])
def test_block_from_the_joint_product(monkeypatch, B, S, Hk, Hv, D, record):
    """The block's launch finds its operands in the product of the joined projections: the bits it has from views of them, and from
    tensors of their own; a product whose columns lie where it cannot read them is left to the others."""
    gen = torch.Generator("cuda").manual_seed(S)

    def r(*shape, std=1.0, to=BF):
        return (torch.randn(shape, generator=gen, device="cuda") * std).to(to)

    C = 2 * Hk * D + Hv * D
    cut = [0]
    for n in (C, Hv * D, Hv, Hv):
        cut.append(cut[-1] + n)
    bounds = list(zip(cut, cut[1:]))
    wide = r(B, S, cut[-1] + 8 - cut[-1] % 8)
    taps, window, A, bias, weight, state = r(C, 4, 1, std=0.5), r(B, 3, C), r(Hv, to=FP), r(Hv, to=FP), r(D), r(B, Hv, D, D, std=0.1, to=FP)
    rest = (Hk, Hv, D, D, 1e-6, 1e-6, record)

    def made(product, w=weight, bounds=bounds):
        return nat.host().gdn_block_of(product, bounds, window, taps, A, bias, w, state, *rest)

    qkv, z, b, a = (wide[..., lo:hi] for lo, hi in bounds)
    for w in (weight, None):
        got = made(wide, w)
        for own in (lambda t: t, lambda t: t.contiguous()):
            want = nat.host().gdn_block(own(qkv), window, taps, own(a), own(b), A, bias, None if w is None else own(z), w, state, *rest)
            for g, o in zip(got[:6], want[:6]):
                assert (g is None) == (o is None) and (g is None or torch.equal(g, o))
        assert got[0].shape == (B, S, Hv * D) and (got[6] is not None) == record and (not record or torch.equal(got[6], qkv))
    assert made(wide.half()) is None and made(wide[0]) is None and made(wide[..., :cut[-1] - 1]) is None
    assert made(wide, bounds=bounds[:3]) is None and made(wide, bounds=[(lo + 4, hi + 4) for lo, hi in bounds]) is None
    assert made(wide, bounds=bounds[:3] + [(cut[-1], cut[-1] + 99)]) is None and made(_at(wide, 1)) is None
    assert made(wide, bounds=[(lo - 8, hi - 8) for lo, hi in bounds]) is None  # (of the right widths, before the product)


@pytest.mark.gpu
def test_results_go_through_the_dispatcher_where_somebody_looks(monkeypatch):
    """A dispatch mode and the profiler see the results that the launches make, and memory is filled where that is asked for."""
    from torch.utils._python_dispatch import TorchDispatchMode

    monkeypatch.setenv("DFLASH_VERIFY_QMM", "1")
    w, s, b = _triple(1024, 512, 64, BF)
    x = _rows((1, 16), 1024, BF)
    want = VQ.verify_matmul(x, w, s, b)
    seen = []

    class Mode(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            seen.append(str(func))
            return func(*args, **(kwargs or {}))

    with Mode():
        got = VQ.verify_matmul(x, w, s, b)
    assert torch.equal(got, want) and any(name.startswith("aten.empty") for name in seen)
    with torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CPU]) as prof:
        got = VQ.verify_matmul(x, w, s, b)
    assert torch.equal(got, want) and any(e.key == "aten::empty" for e in prof.key_averages())
    before = torch.are_deterministic_algorithms_enabled()
    torch.use_deterministic_algorithms(True)
    try:
        got = VQ.verify_matmul(x, w, s, b)
    finally:
        torch.use_deterministic_algorithms(before)
    assert torch.equal(got, want)


@pytest.mark.gpu
@pytest.mark.parametrize("rows", [1, 15, 16, 17, 40])
@pytest.mark.parametrize("N", [16, 32, 48, 512])
def test_projection_module(monkeypatch, rows, N):
    """A projection's call reaches its launch with the bits that the operators behind it give."""
    monkeypatch.setenv("DFLASH_VERIFY_QMM", "1")
    w, s, b = _triple(1024, N, 64, BF)
    x, module = _rows((1, rows), 1024, BF), VL.VerifyQuantizedLinear.from_quantized(VL.QuantizedLinear(w, s, b, group_size=64, bits=4))
    call = VQ.verify_matmul if rows == 16 else VL.stock_matmul
    assert torch.equal(module(x), call(x, w, s, b, transpose=True, group_size=64, bits=4))
    with pytest.raises((ValueError, RuntimeError)):
        module(x.reshape(-1)[:rows * 512 * 2].reshape(2 * rows, 512))
