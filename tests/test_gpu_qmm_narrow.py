"""Up to 16 rows through the kernel for matrices of few weights (csrc/qmm_narrow.hip): the edges of its rule, chunks that some waves
have and others do not, every group size and type, the packed images and the gated activation, against the product of the
same operands in fp64 and against the streaming kernel."""
import pytest
import torch

from dflash_mlx_amd import verify_qmm as VQ
from dflash_mlx_amd.quantized import dequantize, stock_matmul
from dflash_mlx_amd.workloads import make_qmm_case
from test_gpu_qmm_any_k import _check

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
BF, HF = torch.bfloat16, torch.float16
# one tile of rows (up to 4096 of them, K up to 3584 or, of up to 2304, 4864), two (up to 8192, K up to 2048), and just outside
EDGES = [(512, 16, 64), (640, 48, 32), (1024, 4096, 128), (1152, 80, 128), (2048, 4080, 64), (3584, 1040, 64), (3584, 112, 32),
         (3712, 2304, 128), (4736, 144, 64), (4864, 2304, 64), (512, 8192, 32), (1024, 4128, 64), (2048, 4128, 32), (1920, 6176, 128),
         (384, 64, 64), (576, 64, 64), (4992, 64, 64), (3712, 2320, 64), (2176, 4128, 64), (1024, 4112, 64), (512, 8224, 64)]


@pytest.mark.parametrize("K,N,group", EDGES)
@pytest.mark.parametrize("dtype,scales", [(BF, BF), (HF, HF), (BF, HF), (HF, BF)])
def test_products_at_the_edges(verify_env, native_lib, K, N, group, dtype, scales):
    c = make_qmm_case(K, N, K + N, group_size=group, dtype=dtype).to(DEV)
    s, b = c.scales.to(scales), c.biases.to(scales)
    dense = dequantize(c.w, s, b, group, 4, torch.float64)
    y = stock_matmul(c.x, c.w, s, b, group_size=group)
    _check(y, c.x, dense, K, dtype)
    for rows in (1, 2, 3, 15):  # a row's bits do not depend on the rows beside it
        assert torch.equal(stock_matmul(c.x[:rows].clone(), c.w, s, b, group_size=group), y[:rows])
    if N % 32 == 0 and K % 256 == 0:
        assert torch.equal(VQ.verify_matmul(c.x, c.w, s, b, group_size=group), y)
    if group == 64 and K % 1024 == 0 and N % 32 == 0:
        assert torch.equal(VQ.verify_matmul_packed(c.x, VQ.pack_weights(c.w, s, b)), y)
    # scales where a chunk's are not one aligned load: another kernel's, the same product
    shifted = [torch.cat([t.reshape(-1)[:1], t.reshape(-1)])[1:].view(t.shape) for t in (s, b)]
    _check(stock_matmul(c.x, c.w, *shifted, group_size=group), c.x, dense, K, dtype)
    if K % 256 == 0 and N % 32 == 0:  # and by name: the streaming or the tile kernel, a rounding apart
        for name in ("stream", "tile"):
            if name == "tile" or K % 512 == 0 and group == 64:
                verify_env.setenv("DFLASH_QMM_KERNEL", name)
                _check(stock_matmul(c.x, c.w, s, b, group_size=group), c.x, dense, K, dtype)


@pytest.mark.parametrize("K,N,group", [(512, 32, 64), (1024, 4096, 32), (2048, 8192, 64), (1280, 96, 128), (3584, 1056, 64), (1536, 4160, 128)])
@pytest.mark.parametrize("dtype", [BF, HF])
def test_gated_activation_at_the_edges(native_lib, K, N, group, dtype):
    """Against fp64: the slope of the activation is below 1.1, gate, up, sigmoid and two products are rounded once each."""
    c = make_qmm_case(K, N, K - N, group_size=group, dtype=dtype).to(DEV)
    s, b = (t * (2.0 / K ** 0.5) for t in (c.scales, c.biases))
    y = VQ.small_m_silu_mul(c.x, c.w, s, b, group_size=group)
    for rows in (1, 5, 15):
        assert torch.equal(VQ.small_m_silu_mul(c.x[:rows].clone(), c.w, s, b, group_size=group), y[:rows])
    dense = dequantize(c.w, s, b, group, 4, torch.float64)
    full, size = c.x.double() @ dense.T.contiguous(), c.x.double().abs() @ dense.abs().T.contiguous()
    eps, offset = 2.0 ** (-8 if dtype == BF else -11), 16.0 if dtype == BF else 128.0
    slack = 1.01 * eps * full.abs() + size * offset * 2.0 ** -24 * 4
    gate, up, dg, du = full[:, :N // 2], full[:, N // 2:], slack[:, :N // 2], slack[:, N // 2:]
    act = gate * torch.sigmoid(gate)
    tiny = 0.0 if dtype == BF else 2.0 ** -24  # (fp16 below its smallest normal number)
    bound = 1.1 * up.abs() * dg + (act.abs() + dg) * du + 4 * eps * (act * up).abs() + tiny * (1 + 2 * up.abs())
    assert ((y.double() - act * up).abs() <= bound).all()


@pytest.mark.parametrize("packed", [False, True])
@pytest.mark.parametrize("K,inter", [(1024, 512), (1024, 2048), (1024, 4096), (2048, 1536), (2048, 4096), (3072, 2048), (3072, 2112), (4096, 1024),
                                     (4096, 1152)])
def test_a_row_of_the_gated_activation_alone_and_in_its_block(verify_env, native_lib, K, inter, packed):
    """A token's hidden activation has the same bits decoded alone, in a last short block and in a verify block, with no
    kernel named, at widths that a chained launch serves (K a multiple of 1024, 64 rows) and on either side of this kernel's rule."""
    from dflash_mlx_amd import verify_linear as VL
    from dflash_mlx_amd.quantized import QuantizedLinear

    parent = torch.nn.Module()
    for name, seed in (("gate_proj", K), ("up_proj", K + 1)):
        c = make_qmm_case(K, inter, seed).to(DEV)
        setattr(parent, name, QuantizedLinear(c.w, c.scales * 0.05, c.biases * 0.05, group_size=64, bits=4))
    model = torch.nn.Module()
    model.mlp = parent
    assert VL.install_verify_linears(model) == 2 and VL.fuse_shared_input_linears(model) == 1
    if packed:
        assert VL.pack_verify_linears(model) == 1
    x = torch.randn((1, 16, K), generator=torch.Generator(DEV).manual_seed(inter), device=DEV).to(BF)
    block = VL.silu_gate_up(parent, x)
    assert parent._dflash_fused[0].silu_mul_ready(x) and block.shape == (1, 16, inter)
    for lo, hi in ((0, 1), (15, 16), (2, 4), (0, 15)):
        assert torch.equal(VL.silu_gate_up(parent, x[:, lo:hi].clone()), block[:, lo:hi]), (lo, hi)


@pytest.mark.parametrize("dtype", [BF, HF])
def test_gated_activation_of_two_tiles_in_groups_of_64(native_lib, dtype):
    """Two tiles of rows per workgroup at a K that no chained launch serves."""
    test_gated_activation_at_the_edges(native_lib, 1920, 8192, 64, dtype)


@pytest.mark.parametrize("K,N", [(1024, 512), (2048, 8192), (3072, 2048), (4096, 2048)])
def test_a_chain_beside_the_automatic_choice(verify_env, native_lib, K, N):
    """A chain is the streaming kernel's also where the automatic choice is this one: the same product, the bits of the kernel
    named."""
    c = make_qmm_case(K, N, K + 7).to(DEV)
    y = VQ.QmmChain([VQ.ChainProblem(c.x, c.w, c.scales, c.biases)])()[0]
    dense = dequantize(c.w, c.scales, c.biases, 64, 4, torch.float64)
    _check(y, c.x, dense, K, BF)
    _check(VQ.verify_matmul(c.x, c.w, c.scales, c.biases, group_size=64), c.x, dense, K, BF)
    verify_env.setenv("DFLASH_QMM_KERNEL", "stream")
    assert torch.equal(y, VQ.verify_matmul(c.x, c.w, c.scales, c.biases, group_size=64))
