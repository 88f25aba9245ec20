"""The any-rows 4-bit product (prompts, calls outside the verify gate) against its operands in fp64:
tile edges in M, N and K, every group size, both activation types, split and whole tiles."""
import pytest
import torch

from dflash_mlx_amd.quantized import QuantizedLinear, dequantize, quantized_matmul
from dflash_mlx_amd.verify_qmm import rows_matmul
from dflash_mlx_amd.workloads import make_qmm_case

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("M,K,N,group,dtype", [
    (1, 64, 16, 64, torch.bfloat16), (3, 32, 48, 32, torch.bfloat16), (17, 1024, 512, 64, torch.bfloat16),
    (33, 96, 144, 32, torch.float16), (48, 320, 1040, 64, torch.bfloat16), (64, 384, 272, 128, torch.float16),
    (65, 4096, 256, 64, torch.bfloat16), (77, 2048, 6144, 32, torch.bfloat16), (81, 128, 64, 128, torch.bfloat16),
    (96, 1152, 528, 128, torch.bfloat16), (97, 640, 1296, 64, torch.float16), (112, 256, 16, 64, torch.bfloat16),
    (127, 4352, 2048, 64, torch.bfloat16), (128, 1024, 256, 64, torch.bfloat16), (129, 512, 4112, 64, torch.bfloat16),
    (300, 3072, 528, 32, torch.float16), (1024, 1280, 1040, 128, torch.bfloat16), (1500, 64, 4096, 64, torch.bfloat16),
])
def test_rows_against_fp64(native_lib, M, K, N, group, dtype):
    c = make_qmm_case(K, N, 1000 + M, group_size=group, dtype=dtype, M=M).to(DEV)
    y = rows_matmul(c.x, c.w, c.scales, c.biases, group_size=group)
    assert y is not None and y.shape == (M, N) and y.dtype == dtype
    assert torch.equal(y, quantized_matmul(c.x, c.w, c.scales, c.biases, group_size=group))  # and the same every time
    dense = dequantize(c.w, c.scales, c.biases, group, 4, dtype=dtype).double()
    exact = c.x.double() @ dense.t().contiguous()
    # half a unit in the last place of the result (8 and 11 significant bits), and fp32 sums of K products of size |x||w|
    eps = 2.0 ** (-8 if dtype == torch.bfloat16 else -11)
    size = c.x.double().abs() @ dense.abs().t().contiguous()
    # (q*s is exact in fp32, so both forms round the same weight: no term for it)
    assert ((y.double() - exact).abs() <= 1.01 * eps * exact.abs() + size * 2.0 ** -24 * K ** 0.5 + 1e-6).all()
    assert (y.double() - exact).norm() <= eps * exact.norm()


# (with MORE_SHAPES and REST_SHAPES) a call for every tile shape there is: K that ends inside a stage, N and M that end inside a tile, whole and sliced
TILE_SHAPES = [(17, 288, 16, 32), (17, 2080, 48, 32), (20, 96, 528, 32), (17, 160, 8208, 32), (17, 96, 6160, 32), (33, 288, 2064, 32),
               (45, 96, 2064, 32), (33, 160, 12432, 32), (65, 160, 3088, 32), (129, 160, 6160, 32), (129, 96, 12432, 32), (65, 96, 1552, 32),
               (400, 160, 8208, 32), (300, 96, 12432, 32), (97, 4416, 2064, 64), (200, 3136, 1552, 64), (1000, 1664, 5136, 128)]
TILE_SHAPES_SILU = [(17, 160, 32, 32), (31, 1056, 96, 32), (20, 96, 544, 32), (33, 160, 6176, 32), (40, 2080, 4128, 32), (400, 96, 16416, 32),
                    (65, 160, 6176, 32), (77, 2080, 4128, 32), (33, 96, 24864, 32), (193, 160, 16416, 32), (1000, 96, 16416, 32),
                    (200, 96, 16416, 32), (130, 1984, 4256, 64)]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("M,K,N,group,silu", [(*t, False) for t in TILE_SHAPES] + [(*t, True) for t in TILE_SHAPES_SILU])
def test_every_tile_shape_at_its_edges(native_lib, M, K, N, group, silu, dtype):
    c = make_qmm_case(K, N, 4000 + M, group_size=group, dtype=dtype, M=M).to(DEV)
    if silu:
        c.scales.mul_(0.05); c.biases.mul_(0.05)
    y = rows_matmul(c.x, c.w, c.scales, c.biases, group_size=group, epilogue="silu_mul" if silu else None)
    assert torch.equal(y, rows_matmul(c.x, c.w, c.scales, c.biases, group_size=group, epilogue="silu_mul" if silu else None))
    dense = dequantize(c.w, c.scales, c.biases, group, 4, dtype=dtype).double()
    exact, size = c.x.double() @ dense.t().contiguous(), c.x.double().abs() @ dense.abs().t().contiguous()
    eps = 2.0 ** (-8 if dtype == torch.bfloat16 else -11)
    err = size * 2.0 ** -24 * K ** 0.5 + 1e-6
    if silu:  # five roundings between the sums and the result, the sums' own errors with the slopes of the factors (silu's is below 1.1)
        (gate, up), (eg, eu) = exact.split(N // 2, dim=-1), err.split(N // 2, dim=-1)
        act = gate * torch.sigmoid(gate)
        err = 5 * eps * ((act * up).abs() + (gate * up).abs() * 0.25) + 1.1 * eg * up.abs() + eu * act.abs() + 1e-6
        exact = act * up
    else:
        err = err + 1.01 * eps * exact.abs()
    assert ((y.double() - exact).abs() <= err).all()


def test_leading_dimensions_and_switch(native_lib, monkeypatch):
    c = make_qmm_case(512, 96, 5, M=40).to(DEV)
    y = quantized_matmul(c.x.reshape(2, 20, 512), c.w, c.scales, c.biases)
    assert torch.equal(y.reshape(40, 96), quantized_matmul(c.x, c.w, c.scales, c.biases))
    monkeypatch.setenv("DFLASH_STOCK_KERNEL", "0")
    arrays = quantized_matmul(c.x, c.w, c.scales, c.biases)
    assert (y.reshape(40, 96).float() - arrays.float()).norm() <= 2 ** -8 * arrays.float().norm()


@pytest.mark.parametrize("M,K,N,group,dtype", [
    (17, 128, 32, 64, torch.bfloat16), (33, 1024, 544, 32, torch.float16), (77, 512, 1024, 64, torch.bfloat16),
    (112, 640, 96, 128, torch.bfloat16), (130, 1024, 2080, 64, torch.bfloat16), (600, 256, 8192, 64, torch.float16)])
def test_gated_activation_in_the_product(native_lib, M, K, N, group, dtype):
    """The silu-mul epilogue: the operators applied one by one to the product of the same rows.  The two products may
    be cut into different slices of K, so a result may differ by the rounding of a factor or two."""
    c = make_qmm_case(K, N, 2000 + M, group_size=group, dtype=dtype, M=M).to(DEV)
    c.scales.mul_(0.05); c.biases.mul_(0.05)
    h = rows_matmul(c.x, c.w, c.scales, c.biases, group_size=group, epilogue="silu_mul")
    gate, up = rows_matmul(c.x, c.w, c.scales, c.biases, group_size=group).split(N // 2, dim=-1)
    ops = ((gate * torch.sigmoid(gate)) * up).float()
    assert h.shape == (M, N // 2) and h.dtype == dtype
    eps = 2.0 ** (-8 if dtype == torch.bfloat16 else -11)
    assert ((h.float() - ops).abs() <= 4 * eps * ops.abs() + eps * (gate * up).abs().float() * 1e-2 + 1e-6).all()
    assert float((h.float() != ops).float().mean()) <= 2e-2


@pytest.mark.parametrize("M,K,N,group,dtype", [
    (1024, 1024, 12352, 64, torch.bfloat16),   # 392 tiles of 128 x 256: one round whole, the rest in slices
    (1000, 5120, 10000, 64, torch.bfloat16), (520, 2176, 33040, 32, torch.float16), (2048, 640, 17408, 128, torch.bfloat16)])
def test_more_tiles_than_the_chip_takes_at_once(native_lib, M, K, N, group, dtype):
    c = make_qmm_case(K, N, 3000 + M, group_size=group, dtype=dtype, M=M).to(DEV)
    y = rows_matmul(c.x, c.w, c.scales, c.biases, group_size=group)
    assert torch.equal(y, rows_matmul(c.x, c.w, c.scales, c.biases, group_size=group))
    dense = dequantize(c.w, c.scales, c.biases, group, 4, dtype=dtype).double()
    eps = 2.0 ** (-8 if dtype == torch.bfloat16 else -11)
    for lo in range(0, N, 4096):  # (as in the test above, some columns at a time)
        part = dense[lo:lo + 4096].t().contiguous()
        exact, size = c.x.double() @ part, c.x.double().abs() @ part.abs()
        got = y[:, lo:lo + 4096].double()
        assert ((got - exact).abs() <= 1.01 * eps * exact.abs() + size * 2.0 ** -24 * K ** 0.5 + 1e-6).all()
        assert (got - exact).norm() <= eps * exact.norm()


def _layer(widths, K, seed, dtype=torch.bfloat16):
    """A parent module whose swapped projections were joined."""
    from dflash_mlx_amd import verify_linear as VL

    parent = torch.nn.Module()
    for i, (name, n) in enumerate(widths.items()):
        c = make_qmm_case(K, n, seed + i, dtype=dtype).to(DEV)
        c.scales.mul_(0.05); c.biases.mul_(0.05)
        setattr(parent, name, QuantizedLinear(c.w, c.scales, c.biases, group_size=64, bits=4))
    VL.install_verify_linears(parent)
    assert VL.fuse_shared_input_linears(parent) == 1
    return parent


@pytest.mark.parametrize("rows", [1, 15, 17, 77])
def test_gradients_reach_the_activations(native_lib, rows):
    """A call that something differentiates keeps the array operators, whose graph autograd has: x + layer(x), joined
    projections, the gated activation, and the scales themselves."""
    from dflash_mlx_amd import verify_linear as VL

    c = make_qmm_case(512, 512, 50 + rows, M=rows).to(DEV)
    dense = dequantize(c.w, c.scales, c.biases, 64, 4, dtype=torch.bfloat16).double()
    x, g = c.x.clone().requires_grad_(True), torch.randn_like(c.x)
    layer = QuantizedLinear(c.w, c.scales, c.biases, group_size=64, bits=4)
    (x + layer(x)).backward(g)
    want = g.double() + g.double() @ dense
    # one rounding each of the product's part of the gradient and of the sum
    assert (x.grad.double() - want).norm() <= 2 * 2.0 ** -8 * want.norm()
    scales = c.scales.clone().requires_grad_(True)
    quantized_matmul(c.x, c.w, scales, c.biases).backward(g)
    assert scales.grad is not None and bool((scales.grad != 0).any())

    parent = _layer(dict(gate_proj=256, up_proj=256), 512, 60)
    for fn in (lambda v: VL.shared_input_outputs(parent, ("gate_proj", "up_proj"), v)[1], lambda v: VL.silu_gate_up(parent, v)):
        x.grad = None
        fn(x).float().square().sum().backward()
        assert x.grad is not None and bool((x.grad != 0).any())
    if rows > 16:
        parent.up_proj.scales.requires_grad_(True)
        VL.silu_gate_up(parent, c.x).float().square().sum().backward()
        assert parent.up_proj.scales.grad is not None


@pytest.mark.parametrize("rows", [5, 40])
def test_tangents_and_batched_calls_keep_the_array_operators(native_lib, rows):
    from torch.autograd import forward_ad

    from dflash_mlx_amd.verify_qmm import small_m_matmul, small_m_silu_mul

    c = make_qmm_case(512, 512, 70 + rows, M=rows).to(DEV)
    t = torch.randn_like(c.x)
    with forward_ad.dual_level():
        y = quantized_matmul(forward_ad.make_dual(c.x, t), c.w, c.scales, c.biases)
        tangent = forward_ad.unpack_dual(y).tangent
    assert tangent is not None
    want = t.double() @ dequantize(c.w, c.scales, c.biases, 64, 4, dtype=torch.bfloat16).double().t().contiguous()
    assert (tangent.double() - want).norm() <= 2.0 ** -8 * want.norm()

    def none_of_the_kernels(v):
        for kernel in (rows_matmul, small_m_matmul, small_m_silu_mul):
            assert kernel(v, c.w, c.scales, c.biases) is None
        return v

    torch.func.vmap(none_of_the_kernels)(torch.stack([c.x, t]))

    class Tagged(torch.Tensor):
        pass

    none_of_the_kernels(c.x.as_subclass(Tagged))
    assert rows_matmul(c.x, c.w, c.scales, c.biases) is not None

    layer = QuantizedLinear(c.w, c.scales, c.biases, group_size=64, bits=4)
    whole = torch.compile(layer, backend="eager", fullgraph=True)  # one graph of array operators, no break at a launch
    assert (whole(c.x).float() - layer(c.x).float()).norm() <= 2.0 ** -8 * layer(c.x).float().norm()


def test_activation_takes_the_bits_of_the_array_operators(native_lib):
    """Rows with a single 1 make every product exact (a dequantised weight), so that nothing but the activation is left to
    differ: every 16-bit gate a checkpoint's codes give, against the operators one by one."""
    for dtype in (torch.bfloat16, torch.float16):
        c = make_qmm_case(512, 2048, 80, dtype=dtype).to(DEV)
        c.scales.mul_(0.2); c.biases.mul_(0.2)
        x = torch.eye(512, dtype=dtype, device=DEV)
        gate, up = rows_matmul(x, c.w, c.scales, c.biases).split(1024, dim=-1)
        assert torch.equal(torch.cat([gate, up], dim=-1), dequantize(c.w, c.scales, c.biases, 64, 4, dtype=dtype).t())
        h = rows_matmul(x, c.w, c.scales, c.biases, epilogue="silu_mul")
        assert torch.equal(h, (gate * torch.sigmoid(gate)) * up)


# the shapes of more than four waves at the sizes where those of four do not serve, and those of four, whole and sliced
MORE_SHAPES = [(17, 1440, 16, 32), (33, 6080, 80, 32), (17, 1056, 8368, 32), (17, 4160, 2768, 32), (33, 2464, 4272, 32), (33, 672, 8224, 32),
               (33, 3168, 4112, 32), (97, 288, 8592, 32), (33, 2880, 8336, 32), (65, 288, 11024, 32), (65, 2880, 2784, 32), (130, 480, 10976, 32),
               (65, 2880, 8208, 32), (17, 6080, 8224, 32), (17, 2880, 8240, 32), (33, 1632, 432, 32), (17, 3168, 16, 32), (17, 288, 32832, 32),
               (600, 288, 8224, 32), (400, 480, 13232, 32)]
MORE_SHAPES_SILU = [(65, 2464, 8416, 32), (17, 3552, 11488, 32), (65, 288, 11040, 32), (33, 3168, 992, 32), (130, 480, 10912, 32), (65, 3168, 1376, 32),
                    (17, 2080, 32, 32), (33, 1632, 608, 32), (33, 288, 8224, 32), (17, 288, 32960, 32),
                    (400, 480, 13120, 32)]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("M,K,N,group,silu", [(*t, False) for t in MORE_SHAPES] + [(*t, True) for t in MORE_SHAPES_SILU])
def test_tile_shapes_of_four_and_eight_waves(native_lib, M, K, N, group, silu, dtype):
    test_every_tile_shape_at_its_edges(native_lib, M, K, N, group, silu, dtype)


# the shapes, whole and sliced, that the lists above do not reach as the choice is fitted now
REST_SHAPES = [(400, 5760, 144, 64), (65, 3616, 4240, 32), (97, 416, 8592, 32), (33, 5728, 5488, 32), (130, 960, 10992, 32), (17, 4416, 10912, 64),
               (400, 736, 13712, 32), (600, 1376, 13216, 32), (600, 96, 6432, 32), (97, 2880, 8288, 32), (300, 192, 1632, 32), (33, 5600, 1376, 32)]
REST_SHAPES_SILU = [(17, 192, 16736, 32), (33, 416, 17696, 32), (33, 3872, 8416, 32), (65, 992, 15136, 32), (65, 4672, 2848, 32),
                    (17, 2592, 16416, 32), (193, 224, 18720, 32), (65, 3424, 16608, 32), (200, 736, 22176, 32), (97, 4128, 16928, 32),
                    (65, 352, 21984, 32), (97, 3008, 8416, 64), (33, 4960, 16480, 32), (1000, 704, 16544, 32)]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("M,K,N,group,silu", [(*t, False) for t in REST_SHAPES] + [(*t, True) for t in REST_SHAPES_SILU])
def test_tile_shapes_that_the_choice_has_for_other_sizes(native_lib, M, K, N, group, silu, dtype):
    test_every_tile_shape_at_its_edges(native_lib, M, K, N, group, silu, dtype)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("M,K,N,group,silu", [(100, 3840, 528, 64, False), (90, 4096, 1056, 32, True), (400, 4352, 2320, 128, False),
                                              (1024, 2560, 8208, 64, False), (130, 1280, 4128, 32, True), (200, 12288, 272, 64, False),
                                              (300, 768, 12304, 128, False)])
def test_scales_past_the_registers(native_lib, M, K, N, group, silu, dtype):
    """Scales go from memory to LDS directly where rows of them start on four bytes: the bits of the other way, which scales at an odd
    element take, over groups that end inside a piece of eight; what lies behind a row stays in its own."""
    c = make_qmm_case(K, N, 7000 + M, group_size=group, dtype=dtype, M=M).to(DEV)

    def odd(t):
        moved = torch.empty(t.numel() + 1, dtype=t.dtype, device=t.device)[1:].view(t.shape)
        return moved.copy_(t)

    def product(scales, biases):
        return rows_matmul(c.x, c.w, scales, biases, group_size=group, epilogue="silu_mul" if silu else None)

    want = product(odd(c.scales), odd(c.biases))
    assert torch.equal(product(c.scales, c.biases), want)
    row = N // 2 - 3
    c.scales[row, 0] = float("nan")
    c.biases[row, -1] = float("inf")
    got = product(c.scales, c.biases)
    column = torch.arange(want.shape[1], device=DEV) != row
    assert torch.equal(got[:, column], want[:, column]) and got[:, row].isnan().all()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("M,K,N,group,silu", [(1, 1152, 160, 64, False), (16, 10496, 352, 64, False), (15, 4480, 224, 32, True), (8, 17024, 96, 64, False),
                                              (16, 2688, 2880, 32, False), (3, 1280, 1600, 32, True)])
def test_up_to_sixteen_rows_with_weights_in_registers(native_lib, M, K, N, group, silu, dtype):
    """K that the verify block's kernel does not take (an odd multiple of 128), or columns: rows that are not there, whole and in slices of K."""
    test_every_tile_shape_at_its_edges(native_lib, M, K, N, group, silu, dtype)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("M,K,N,group,silu", [
    (33, 3168, 4112, 32, False), (33, 3232, 2064, 32, False),           # an odd number of groups, K that ends inside a stage: sliced, whole
    (17, 10112, 416, 128, False), (100, 11904, 2048, 128, False),       # slices that begin inside a chunk of scales
    (100, 5440, 1040, 64, False), (70, 6432, 528, 32, False), (45, 4128, 1056, 32, True), (400, 4352, 2320, 128, False)])
def test_the_same_bits_call_after_call(native_lib, M, K, N, group, silu, dtype):
    """Waves read codes that other waves asked for: none of them may be filled again before.  Against fp64 once, then against itself."""
    test_every_tile_shape_at_its_edges(native_lib, M, K, N, group, silu, dtype)
    c = make_qmm_case(K, N, 8000 + M, group_size=group, dtype=dtype, M=M).to(DEV)
    want = rows_matmul(c.x, c.w, c.scales, c.biases, group_size=group, epilogue="silu_mul" if silu else None)
    for i in range(60):
        got = rows_matmul(c.x, c.w, c.scales, c.biases, group_size=group, epilogue="silu_mul" if silu else None)
        assert torch.equal(got, want), i
