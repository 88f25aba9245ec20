"""Up to 16 rows through the streaming kernel's variants for every group size and K that is a multiple of 64
only, and through what is taken where no kernel is named, against the product of the same operands in fp64: last
chunks and last stages that are cut short in every way, ragged row blocks, one to sixteen rows, both activation types,
gathered experts."""
import pytest
import torch

from dflash_mlx_amd import verify_qmm as VQ
from dflash_mlx_amd.quantized import dequantize, stock_matmul
from dflash_mlx_amd.workloads import make_qmm_case

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
# the streaming kernel, and what calls take where no kernel is named (the one that keeps x in registers, where that has the shape)
each_kernel = pytest.mark.parametrize("kernel", ["auto", None])


def _choose(monkeypatch, kernel):
    if kernel is None:
        monkeypatch.delenv("DFLASH_QMM_KERNEL", raising=False)
    else:
        monkeypatch.setenv("DFLASH_QMM_KERNEL", kernel)


def _check(y, x, dense, K, dtype):
    exact = x.double() @ dense.t().contiguous()
    size = x.double().abs() @ dense.abs().t().contiguous()
    # half a unit in the last place of the result; fp32 sums over codes offset by 128 or 1024 (up to 70 times the
    # size of a centred code), whose errors add up like a random walk over K terms
    eps = 2.0 ** (-8 if dtype == torch.bfloat16 else -11)
    offset = 16.0 if dtype == torch.bfloat16 else 128.0
    assert ((y.double() - exact).abs() <= 1.01 * eps * exact.abs() + size * offset * 2.0 ** -24 * 4).all()
    assert (y.double() - exact).norm() <= eps * exact.norm()


@each_kernel
@pytest.mark.parametrize("K,N,group,dtype", [
    (512, 16, 32, torch.bfloat16), (576, 48, 32, torch.bfloat16), (640, 128, 64, torch.bfloat16), (768, 144, 64, torch.float16),
    (832, 272, 32, torch.float16), (896, 1040, 64, torch.bfloat16), (1024, 512, 32, torch.bfloat16),
    (1024, 512, 128, torch.bfloat16), (1152, 2064, 64, torch.bfloat16), (1280, 112, 128, torch.float16),
    (2176, 4096, 64, torch.bfloat16), (2816, 528, 128, torch.bfloat16), (4096, 6144, 32, torch.bfloat16),
    (5376, 144, 64, torch.bfloat16), (12288, 4096, 32, torch.bfloat16), (4352, 5120, 128, torch.bfloat16)])
def test_every_group_size_and_k(native_lib, monkeypatch, K, N, group, dtype, kernel):
    monkeypatch.setenv("DFLASH_VERIFY_QMM", "1")
    _choose(monkeypatch, kernel)
    c = make_qmm_case(K, N, 300 + K, group_size=group, dtype=dtype).to(DEV)
    dense = dequantize(c.w, c.scales, c.biases, group, 4, dtype=torch.float64)
    y = VQ._launch(c.x, c.w, c.scales, c.biases, K, N, group, "mma2big", 1)
    _check(y, c.x, dense, K, dtype)
    for rows in (1, 2, 7, 15, 16):  # and the same bits whatever shares the block with a row
        assert torch.equal(stock_matmul(c.x[:rows], c.w, c.scales, c.biases, group_size=group), y[:rows])
    torch.cuda.synchronize()
    VQ.raise_on_device_errors(torch.device(DEV))
    ws = VQ._workspace(torch.device(DEV), torch.cuda.current_stream().cuda_stream, 1)
    assert int((ws != 0).sum()) == 0


@each_kernel
@pytest.mark.parametrize("K,N,E,P", [(640, 144, 4, 37), (768, 256, 3, 16), (896, 2048, 8, 128), (1152, 272, 2, 250)])
def test_gathered_experts_of_any_k(native_lib, monkeypatch, K, N, E, P, kernel):
    _choose(monkeypatch, kernel)
    cases = [make_qmm_case(K, N, 500 + e).to(DEV) for e in range(E)]
    w, s, b = (torch.stack([getattr(c, n) for c in cases]) for n in ("w", "scales", "biases"))
    gen = torch.Generator().manual_seed(K)
    ids = torch.randint(-1, E + 1, (P,), generator=gen).to(torch.int32).to(DEV)  # some belong to no expert
    x = torch.randn(P, K, generator=gen).to(torch.bfloat16).to(DEV)
    y = VQ.gather_qmm(x, w, s, b, ids)
    for e in range(E):
        rows = ids == e
        if bool(rows.any()):
            _check(y[rows], x[rows], dequantize(w[e], s[e], b[e], 64, 4, dtype=torch.float64), K, torch.bfloat16)
    assert bool((y[(ids < 0) | (ids >= E)] == 0).all())
    assert torch.equal(y, VQ.gather_qmm(x, w, s, b, ids))


@each_kernel
@pytest.mark.parametrize("K,N,group,dtype", [
    (512, 32, 64, torch.bfloat16), (512, 16, 32, torch.bfloat16), (576, 48, 32, torch.float16), (896, 272, 64, torch.bfloat16),
    (1024, 1040, 64, torch.bfloat16), (1280, 112, 128, torch.float16), (1536, 4128, 64, torch.float16),
    (4096, 24576, 32, torch.bfloat16), (5120, 34816, 64, torch.bfloat16)])
def test_gated_activation_of_few_rows(native_lib, monkeypatch, K, N, group, dtype, kernel):
    """The silu-mul form (8 gate rows and their 8 up rows to a tile) against the joint product of the same matrix and the array
    operators, and both against float64."""
    monkeypatch.setenv("DFLASH_VERIFY_QMM", "1")
    _choose(monkeypatch, kernel)
    c = make_qmm_case(K, N, 700 + K, group_size=group, dtype=dtype).to(DEV)
    x = (c.x / (K ** 0.5 * c.scales.float().abs().mean() * 4)).to(dtype)  # gates of a few units
    assert VQ.small_m_silu_mul(x[:, :K - 64], c.w, c.scales, c.biases, group_size=group) is None
    y = VQ.small_m_silu_mul(x, c.w, c.scales, c.biases, group_size=group)
    assert y.shape == (16, N // 2)
    for rows in (1, 2, 9, 15):  # the same bits whatever shares the block with a row
        assert torch.equal(VQ.small_m_silu_mul(x[:rows], c.w, c.scales, c.biases, group_size=group), y[:rows])
    joint = VQ.small_m_matmul(x, c.w, c.scales, c.biases, group_size=group)
    gate, up = joint[:, :N // 2], joint[:, N // 2:]
    ref = (gate * torch.sigmoid(gate)) * up
    # K is cut between workgroups in other places: gate and up may fall on the next value of the type (eps of
    # themselves) and, where they cancel, move by the error of two fp32 sums over offset codes (``_check``); the slope of
    # silu is below 1.1, and three more roundings follow on either side
    eps = torch.finfo(dtype).eps
    dense = dequantize(c.w, c.scales, c.biases, group, 4, dtype=torch.float64)
    sums = (x.double().abs() @ dense.abs().t().contiguous()) * (16.0 if dtype == torch.bfloat16 else 128.0) * 2.0 ** -24 * 4 * 2
    g, u = gate.double(), up.double()
    s = g * torch.sigmoid(g)
    dg, du = eps * g.abs() + sums[:, :N // 2], eps * u.abs() + sums[:, N // 2:]
    assert ((y.double() - ref.double()).abs() <= 1.1 * dg * (u.abs() + du) + s.abs() * du + 3 * eps * (s * u).abs() + 1e-6).all()
    product = x.double() @ dense.t().contiguous()
    exact = product[:, :N // 2] * torch.sigmoid(product[:, :N // 2]) * product[:, N // 2:]
    assert (y.double() - exact).norm() <= 1.05 * (ref.double() - exact).norm()
    torch.cuda.synchronize()
    VQ.raise_on_device_errors(torch.device(DEV))
    ws = VQ._workspace(torch.device(DEV), torch.cuda.current_stream().cuda_stream, 1)
    assert int((ws != 0).sum()) == 0


@each_kernel
def test_few_rows_take_the_joint_launch(native_lib, monkeypatch, kernel):
    """One token and a short block through joined projections: the rows a block of 16 gets, also for members
    behind a wrapper that pads, and the members' own launches with DFLASH_STOCK_KERNEL=0 or once a member has left."""
    from dflash_mlx_amd import verify_linear as VL
    from dflash_mlx_amd.gdn_layer import _ExactSmallProjPad
    from dflash_mlx_amd.quantized import QuantizedLinear

    monkeypatch.setenv("DFLASH_VERIFY_QMM", "1")
    _choose(monkeypatch, kernel)
    parent = torch.nn.Module()
    widths = dict(in_proj_qkv=256, in_proj_z=128, in_proj_b=48, in_proj_a=48)
    for i, (name, n) in enumerate(widths.items()):
        c = make_qmm_case(1024, n, 900 + i).to(DEV)
        setattr(parent, name, QuantizedLinear(c.w, c.scales, c.biases, group_size=64, bits=4))
    parent.in_proj_b, parent.in_proj_a = _ExactSmallProjPad(parent.in_proj_b), _ExactSmallProjPad(parent.in_proj_a)
    VL.install_verify_linears(parent)
    assert VL.fuse_shared_input_linears(parent) == 1
    x = make_qmm_case(1024, 32, 950).to(DEV).x.reshape(1, 16, 1024)
    whole = VL.shared_input_outputs(parent, tuple(widths), x)
    group = parent._dflash_fused[0]
    for rows in (1, 5, 15):
        assert group.serves_few(parent, x[:, :rows])
        for got, want in zip(VL.shared_input_outputs(parent, tuple(widths), x[:, :rows]), whole):
            assert torch.equal(got, want[:, :rows])
    monkeypatch.setenv("DFLASH_STOCK_KERNEL", "0")
    assert not group.serves_few(parent, x[:, :1])
    monkeypatch.delenv("DFLASH_STOCK_KERNEL")
    parent.in_proj_z.to(torch.device(DEV), torch.bfloat16)
    parent.in_proj_z._apply(lambda t: t.clone())
    assert not group.serves_few(parent, x[:, :1])


@each_kernel
@pytest.mark.parametrize("rows", [1, 3, 15])
def test_few_rows_that_start_anywhere(native_lib, monkeypatch, rows, kernel):
    """The kernel loads x in pieces of 16 bytes; fewer rows than a block may start on any element all the same."""
    _choose(monkeypatch, kernel)
    for group, K, N in ((64, 1024, 256), (32, 576, 48), (128, 128, 16)):
        c = make_qmm_case(K, N, 960 + rows, group_size=group, M=rows).to(DEV)
        want = stock_matmul(c.x, c.w, c.scales, c.biases, group_size=group)
        for shift in (1, 4):
            held = torch.empty(rows * K + shift, dtype=c.x.dtype, device=DEV)
            x = held[shift:].view(rows, K)
            x.copy_(c.x)
            assert x.data_ptr() % 16 and x.is_contiguous()
            assert torch.equal(stock_matmul(x, c.w, c.scales, c.biases, group_size=group), want)


def test_hooks_of_joined_projections_run(native_lib, monkeypatch):
    """A member with a hook, or with a forward of its own, answers for itself; every length of call, the wrapper that pads
    included."""
    from dflash_mlx_amd import verify_linear as VL
    from dflash_mlx_amd.gdn_layer import _ExactSmallProjPad
    from dflash_mlx_amd.quantized import QuantizedLinear

    monkeypatch.setenv("DFLASH_VERIFY_QMM", "1")
    monkeypatch.delenv("DFLASH_QMM_KERNEL", raising=False)
    parent = torch.nn.Module()
    widths = dict(in_proj_qkv=256, in_proj_z=128, in_proj_b=48, in_proj_a=48)
    for i, (name, n) in enumerate(widths.items()):
        c = make_qmm_case(1024, n, 980 + i).to(DEV)
        setattr(parent, name, QuantizedLinear(c.w, c.scales, c.biases, group_size=64, bits=4))
    parent.in_proj_b, parent.in_proj_a = _ExactSmallProjPad(parent.in_proj_b), _ExactSmallProjPad(parent.in_proj_a)
    VL.install_verify_linears(parent)
    assert VL.fuse_shared_input_linears(parent) == 1
    seen = []

    def hook(module, args, *output):
        seen.append(module)

    places = [(parent.in_proj_z, "register_forward_hook"), (parent.in_proj_qkv, "register_forward_pre_hook"),
              (parent.in_proj_b, "register_forward_hook"), (parent.in_proj_b.linear, "register_forward_hook")]
    for rows in (1, 5, 16, 77):
        x = make_qmm_case(1024, 32, 990, M=rows).to(DEV).x.reshape(1, rows, 1024)
        for module, register in places:
            handle = getattr(module, register)(hook)
            VL.shared_input_outputs(parent, tuple(widths), x)
            handle.remove()
            assert seen == [module], (rows, register)
            seen.clear()
        every = torch.nn.modules.module.register_module_forward_hook(hook)
        VL.shared_input_outputs(parent, tuple(widths), x)
        every.remove()
        assert {id(m) for m in seen if isinstance(m, VL.VerifyQuantizedLinear)} == \
            {id(m) for m in (parent.in_proj_qkv, parent.in_proj_z, parent.in_proj_b.linear, parent.in_proj_a.linear)}
        seen.clear()
        z = parent.in_proj_z
        z.forward = lambda v: seen.append(z) or type(z).forward(z, v)  # as wrappers of a module's forward leave it
        VL.shared_input_outputs(parent, tuple(widths), x)
        del z.forward
        assert seen == [z]
        seen.clear()
        VL.shared_input_outputs(parent, tuple(widths), x)
        assert parent._dflash_fused[0]._holds(parent, x, padded=True) and not seen


@pytest.mark.parametrize("rows", [1, 5, 77])
def test_joined_outputs_of_prompts_and_short_blocks_are_tensors_of_their_own(native_lib, monkeypatch, rows):
    from dflash_mlx_amd import verify_linear as VL
    from dflash_mlx_amd.quantized import QuantizedLinear

    monkeypatch.setenv("DFLASH_VERIFY_QMM", "1")
    monkeypatch.delenv("DFLASH_QMM_KERNEL", raising=False)
    parent = torch.nn.Module()
    for i, (name, n) in enumerate(dict(q_proj=256, k_proj=64, v_proj=64).items()):
        c = make_qmm_case(512, n, 970 + i).to(DEV)
        setattr(parent, name, QuantizedLinear(c.w, c.scales, c.biases, group_size=64, bits=4))
    VL.install_verify_linears(parent)
    assert VL.fuse_shared_input_linears(parent) == 1
    x = make_qmm_case(512, 32, 975, M=rows).to(DEV).x.reshape(1, rows, 512)
    names = ("q_proj", "k_proj", "v_proj")
    for name, y in zip(names, VL.shared_input_outputs(parent, names, x)):
        n = getattr(parent, name).weight.shape[0]
        assert y.view(rows, n // 32, 32).shape == (rows, n // 32, 32) and y.is_contiguous()

    class Norm(torch.nn.Module):  # somebody's own
        def __init__(self, weight):
            super().__init__()
            self.weight = weight

        def forward(self, v):
            return v.view(-1, v.shape[-1]).view(v.shape) if v.shape[2] == 2 else v

    from dflash_mlx_amd.attention_layer import GatedAttention

    attn = GatedAttention(num_attention_heads=4, num_key_value_heads=2, head_dim=32, q_proj=parent.q_proj, k_proj=parent.k_proj,
                          v_proj=parent.v_proj, o_proj=torch.nn.Identity())
    object.__setattr__(attn, "_dflash_fused", parent._dflash_fused)
    attn.q_norm, attn.k_norm = Norm(attn.q_norm.weight), Norm(attn.k_norm.weight)
    assert attn(x).shape == (1, rows, 128)


@pytest.mark.parametrize("K,group", [(256, 64), (768, 32), (1280, 128), (2304, 64)])
def test_projections_join_where_k_is_a_multiple_of_256(verify_env, K, group):
    """The joint product against the members' own: two orders of the same fp32 sums (each within the bound of
    ``_check``), each rounded once to the array type.  The activation on top of that: its slope is below 1.1, its four operators
    round once each.  A variant asked for by name: the members themselves, bit for bit."""
    from dflash_mlx_amd.quantized import QuantizedLinear
    from dflash_mlx_amd.verify_linear import fuse_shared_input_linears, install_verify_linears, shared_input_outputs, silu_gate_up

    mlp, names = torch.nn.Module(), ("gate_proj", "up_proj")
    for i, name in enumerate(names):
        c = make_qmm_case(K, 288, 300 + i, group_size=group).to(DEV)
        setattr(mlp, name, QuantizedLinear(c.w, c.scales * 0.1, c.biases * 0.1, group_size=group, bits=4))
    model = torch.nn.Module()
    model.mlp = mlp
    assert install_verify_linears(model) == 2 and fuse_shared_input_linears(model) == 1
    for rows in (1, 5, 16, 40):
        x = (torch.randn((rows, K), generator=torch.Generator().manual_seed(rows)) * 0.5).to(torch.bfloat16).to(DEV)
        own = [getattr(model.mlp, n)(x) for n in names]
        dense = [dequantize(m.weight, m.scales, m.biases, group, 4, torch.float32) for m in (model.mlp.gate_proj, model.mlp.up_proj)]
        apart = [2.0 ** -7 * y.float().abs() + x.float().abs() @ w.abs().T * 16.0 * 2.0 ** -24 * 8 for y, w in zip(own, dense)]
        for got, want, slack in zip(shared_input_outputs(model.mlp, names, x), own, apart):
            assert ((got.float() - want.float()).abs() <= slack).all()
        gate, up = (y.float() for y in own)
        act = gate * torch.sigmoid(gate)
        slack = 1.1 * up.abs() * apart[0] + (act.abs() + apart[0]) * apart[1] + 5 * 2.0 ** -8 * (act * up).abs()
        assert ((silu_gate_up(model.mlp, x).float() - act * up).abs() <= slack).all()
    verify_env.setenv("DFLASH_VERIFY_VARIANT", "mma2big_pipe")
    x = torch.randn((16, K), generator=torch.Generator().manual_seed(9)).to(torch.bfloat16).to(DEV)
    joined = model._modules["mlp"]._dflash_fused[0].applies(model.mlp, x)
    assert joined == (K % 512 == 0)
    assert all(torch.equal(a, getattr(model.mlp, n)(x)) for n, a in zip(names, shared_input_outputs(model.mlp, names, x)))
