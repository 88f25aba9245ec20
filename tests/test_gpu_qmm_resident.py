"""Up to 16 rows through the kernel that keeps x in registers (csrc/qmm_resident.h): widths that are whole chunks for every wave and
widths that are not, one to four slices of K, rings that go round and that do not, every group size and type, the packed
images and the gated activation, against the product of the same operands in fp64."""
import pytest
import torch

import dflash_mlx_amd._native as nat
from dflash_mlx_amd import verify_qmm as VQ
from dflash_mlx_amd.quantized import dequantize, stock_matmul
from dflash_mlx_amd.workloads import make_qmm_case
from test_gpu_qmm_any_k import _check
from test_gpu_qmm_narrow import test_gated_activation_at_the_edges as check_gated_activation
from test_gpu_qmm_rows import test_every_tile_shape_at_its_edges as check_rows_silu
from test_gpu_qmm_rows import test_rows_against_fp64 as check_rows

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
BF, HF = torch.bfloat16, torch.float16
# chunks of 128 k over 8 waves: 1, 1 and 2, 2, .., 6 each, then slices; one tile, a tile per compute unit and one more, nine tiles of some (two
# meetings and a last odd tile); three slices of two chunks, four with one round less than three have, a matrix left to the streaming kernel; narrow
# and wide ones whose waves would be half empty
SHAPES = [(1024, 4112, 64), (1152, 16, 64), (1920, 48, 32), (2048, 4112, 128), (2176, 32, 64), (2304, 36880, 64), (3072, 4096, 64), (3584, 80, 128),
          (4096, 4096, 64), (4096, 1040, 32), (4736, 2320, 64), (5120, 4128, 32), (5120, 12352, 64), (5376, 64, 128), (6144, 512, 64),
          (6144, 8224, 64), (6272, 112, 64), (8192, 4112, 64), (10240, 48, 32), (12288, 4096, 128), (12288, 1024, 64), (17408, 1040, 64),
          (1280, 2048, 64), (2560, 1040, 128), (1024, 24576, 64), (1280, 32768, 32), (17408, 5120, 64), (24576, 32, 64), (24704, 32, 64), (6144, 4096, 128), (14336, 4096, 64), (12800, 16384, 64)]


def _clean(native_lib):
    VQ.raise_on_device_errors(torch.device(DEV))
    ws = VQ._workspace(torch.device(DEV), nat.raw_stream(torch.device(DEV)), 1)
    return int((ws != 0).sum()) == 0


@pytest.mark.parametrize("K,N,group", SHAPES)
@pytest.mark.parametrize("dtype", [BF, HF])
def test_products(verify_env, native_lib, K, N, group, dtype):
    c = make_qmm_case(K, N, K + N, group_size=group, dtype=dtype).to(DEV)
    y = stock_matmul(c.x, c.w, c.scales, c.biases, group_size=group)
    _check(y, c.x, dequantize(c.w, c.scales, c.biases, group, 4, torch.float64), K, dtype)
    for rows in (1, 2, 5, 15):  # a row's bits do not depend on the rows beside it
        assert torch.equal(stock_matmul(c.x[:rows].clone(), c.w, c.scales, c.biases, group_size=group), y[:rows])
    if N % 32 == 0 and K % 256 == 0:
        assert torch.equal(VQ.verify_matmul(c.x, c.w, c.scales, c.biases, group_size=group), y)
    if group == 64 and K % 1024 == 0 and N % 32 == 0:
        assert torch.equal(VQ.verify_matmul_packed(c.x, VQ.pack_weights(c.w, c.scales, c.biases)), y)
    assert _clean(native_lib)  # (slices leave their tiles at zero)


@pytest.mark.parametrize("K,N,group", [(1024, 4128, 64), (1152, 32, 32), (3072, 2112, 64), (4096, 8224, 32), (5120, 4224, 64), (6144, 96, 128), (8192, 1056, 64),
                                       (12288, 2048, 64)])
@pytest.mark.parametrize("dtype", [BF, HF])
def test_gated_activation(native_lib, K, N, group, dtype):
    check_gated_activation(native_lib, K, N, group, dtype)
    assert _clean(native_lib)


@pytest.mark.parametrize("K,N,group", [(1024, 8192, 64), (4096, 4096, 64), (5120, 7168, 64), (4096, 6144, 32), (5120, 4096, 32), (3072, 8192, 32),
                                       (12288, 4096, 64), (17408, 4096, 64), (5120, 5120, 128)])
@pytest.mark.parametrize("dtype", [BF, HF])
def test_no_further_from_64_bits_than_the_streaming_kernel(verify_env, native_lib, K, N, group, dtype):
    """Results that are not the rounded ones of fp64: what fp32 sums leave in the last place.  A thousandth to a twentieth of all there; fewer here."""
    c = make_qmm_case(K, N, K + N, group_size=group, dtype=dtype).to(DEV)
    w = dequantize(c.w, c.scales, c.biases, group, 4, torch.float64)
    exact = (c.x.double() @ w.T).to(torch.float32).to(dtype)
    y = {}
    for kernel in (nat.QMM_KERNEL_AUTO, nat.QMM_KERNEL_FASTEST):
        y[kernel] = torch.empty((16, N), dtype=dtype, device=DEV)
        ws = VQ._workspace(torch.device(DEV), nat.raw_stream(torch.device(DEV)), 1)
        code = VQ._DTYPE_CODE[dtype]
        nat.check(native_lib.dflash_qmm_few(c.x.data_ptr(), c.w.data_ptr(), c.scales.data_ptr(), c.biases.data_ptr(), y[kernel].data_ptr(), ws.data_ptr(),
                                            ws.numel(), 16, K, N, group, code, code, kernel, nat.raw_stream(torch.device(DEV))), "dflash_qmm_few")
    off = {k: int((v != exact).sum()) for k, v in y.items()}
    assert off[nat.QMM_KERNEL_FASTEST] <= off[nat.QMM_KERNEL_AUTO], off
    if group == 64 and K <= 5120:  # the gathered form
        routed = VQ.gather_qmm(c.x, c.w[None], c.scales[None], c.biases[None], torch.zeros(16, dtype=torch.int32, device=DEV))
        assert int((routed != exact).sum()) <= off[nat.QMM_KERNEL_AUTO], off


@pytest.mark.parametrize("value", [float("inf"), float("-inf"), float("nan")])
def test_what_is_not_a_number_stays_in_its_row(verify_env, native_lib, value):
    """Rows are loaded together and padded chunks are multiplied with zeros: neither lets one row's values into another."""
    c = make_qmm_case(5248, 160, 3).to(DEV)  # (41 chunks over 8 waves)
    want = stock_matmul(c.x, c.w, c.scales, c.biases)
    x = c.x.clone()
    x[3, 5000] = value
    y = stock_matmul(x, c.w, c.scales, c.biases)
    assert not torch.isfinite(y[3]).any()
    keep = [r for r in range(16) if r != 3]
    assert torch.equal(y[keep], want[keep])
    scales = c.scales.clone()
    scales[17, 80] = value  # one row of W: one column of y
    y = stock_matmul(c.x, c.w, scales, c.biases)
    assert not torch.isfinite(y[:, 17]).any()
    cols = [n for n in range(160) if n != 17]
    assert torch.equal(y[:, cols], want[:, cols])


def test_a_slice_that_gives_up_says_so_and_the_launch_ends(verify_env, native_lib):
    """The wait for the other slices' tiles cut to one poll: as for the streaming kernel's adding workgroups."""
    c = make_qmm_case(17408, 5120, 41).to(DEV)
    good = VQ.verify_matmul(c.x, c.w, c.scales, c.biases)
    VQ.raise_on_device_errors(torch.device(DEV))
    assert native_lib.dflash_set_option(nat.OPT_QMM_SPIN_LIMIT, 1) == 0
    try:
        for _ in range(8):  # (320 tiles of workgroups that finish at different times)
            VQ.verify_matmul(c.x, c.w, c.scales, c.biases)
        torch.cuda.synchronize()
    finally:
        assert native_lib.dflash_set_option(nat.OPT_QMM_SPIN_LIMIT, 0) == 0
    with pytest.raises(nat.NativeLibraryError, match="partial tiles of row block"):
        VQ.raise_on_device_errors(torch.device(DEV))
    assert torch.equal(VQ.verify_matmul(c.x, c.w, c.scales, c.biases), good) and _clean(native_lib)


def test_sliced_launches_of_two_streams_beside_each_other(verify_env, native_lib):
    """The last slice of a product waits inside the launch for the others.  Two streams, each with such products of its own in flight:
    a workgroup waits for workgroups before it only, which wait for nobody, so neither stream can keep the other's from finishing."""
    cases = [make_qmm_case(17408, 5120, 51).to(DEV), make_qmm_case(14336, 4096, 52).to(DEV)]  # three slices, four slices
    alone = [VQ.verify_matmul(c.x, c.w, c.scales, c.biases) for c in cases]
    streams = [torch.cuda.Stream(), torch.cuda.Stream()]
    for s in streams:
        s.wait_stream(torch.cuda.current_stream())
    got = [[], []]
    for i in range(20):
        for k, s in enumerate(streams):
            with torch.cuda.stream(s):
                c = cases[(i + k) % 2]
                got[k].append(VQ.verify_matmul(c.x, c.w, c.scales, c.biases))
    torch.cuda.synchronize()
    VQ.raise_on_device_errors(torch.device(DEV))
    for k in range(2):
        for i, y in enumerate(got[k]):
            assert torch.equal(y, alone[(i + k) % 2]), (k, i)
    for s in streams:
        assert int((VQ._workspace(torch.device(DEV), s.cuda_stream, 1) != 0).sum()) == 0


# two to five tiles of 16 rows, full and not; one slice and more, whole and uneven chunks; fewer tiles than workgroups, one more, an odd number each
ROWS = [(17, 2048, 16, 64), (32, 4096, 4096, 64), (33, 2304, 4112, 64), (31, 5120, 12352, 64), (40, 3072, 3072, 32), (48, 4096, 6144, 64), (47, 6144, 2048, 128),
        (49, 3328, 4608, 64), (64, 4096, 6144, 32), (65, 4096, 6144, 64), (77, 8192, 5120, 64), (79, 3328, 4624, 64), (80, 12288, 4096, 64), (80, 4096, 6144, 128),
        (17, 17408, 2064, 64), (18, 2176, 8224, 64), (32, 4096, 36880, 64), (48, 3072, 12304, 64), (63, 2048, 12304, 64), (80, 2048, 12304, 64)]


@pytest.mark.parametrize("M,K,N,group", ROWS)
@pytest.mark.parametrize("dtype", [BF, HF])
def test_rows_of_short_prompts(native_lib, M, K, N, group, dtype):
    """Weights rounded to the activation type; the counters of the slices at zero again (the result is the same every time)."""
    check_rows(native_lib, M, K, N, group, dtype)


@pytest.mark.parametrize("M,K,N,group", [(17, 2048, 4128, 64), (32, 4096, 24576, 64), (45, 2304, 6912, 32), (64, 3072, 4096, 64), (77, 4096, 6176, 128),
                                         (80, 5120, 2080, 64)])
@pytest.mark.parametrize("dtype", [BF, HF])
def test_gated_activation_of_short_prompts(native_lib, M, K, N, group, dtype):
    check_rows_silu(native_lib, M, K, N, group, True, dtype)


# one, two, four and eight waves to a tile, even and uneven chunks; one tile of W, sets with one unit, with none, with two meetings and more; entries of one
# and of sixteen rows
@pytest.mark.parametrize("K,N,E,P", [(128, 16, 3, 7), (512, 2048, 256, 128), (640, 48, 5, 90), (768, 16, 300, 200), (1152, 80, 7, 33), (1280, 4112, 2, 16),
                                     (1408, 272, 9, 64), (2048, 1024, 64, 256), (2688, 96, 4, 40), (5120, 144, 3, 50), (1024, 16, 1, 1), (2560, 528, 600, 64),
                                     (640, 4112, 60, 150), (1152, 2064, 64, 200), (2304, 2064, 64, 100), (4096, 1040, 40, 70)])
@pytest.mark.parametrize("dtype", [BF, HF])
def test_routed_experts(native_lib, monkeypatch, K, N, E, P, dtype):
    monkeypatch.delenv("DFLASH_QMM_KERNEL", raising=False)
    gen = torch.Generator("cuda").manual_seed(K + P)
    w = torch.randint(-2 ** 31, 2 ** 31, (E, N, K // 8), generator=gen, device="cuda", dtype=torch.int32)
    s = (torch.rand((E, N, K // 64), generator=gen, device="cuda") * 0.02 + 1e-4).to(dtype)
    b = (s.float() * -8).to(dtype)
    x = torch.randn((P, K), generator=gen, device="cuda").to(dtype)
    ids = torch.randint(-1 if E > 1 else 0, E + (E > 1), (P,), generator=gen, device="cuda", dtype=torch.int32)
    y = VQ.gather_qmm(x, w, s, b, ids)
    assert (y[(ids < 0) | (ids >= E)] == 0).all()
    for e in range(E):
        mine = ids == e
        if mine.any():
            _check(y[mine], x[mine], dequantize(w[e], s[e], b[e], 64, 4, torch.float64), K, dtype)
    assert torch.equal(y, VQ.gather_qmm(x, w, s, b, ids))
    keep = torch.randperm(P, generator=gen, device="cuda")[:P // 2 + 1]  # a row's bits do not depend on the rows beside it
    assert torch.equal(VQ.gather_qmm(x[keep].contiguous(), w, s, b, ids[keep].contiguous()), y[keep])
