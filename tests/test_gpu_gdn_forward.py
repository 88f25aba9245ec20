"""Parity of the gfx950 GatedDeltaNet forward-with-tape kernel against the CPU oracle
(fp64 restatement of dflash_mlx/kernels.py:131-173), and its contract with the replay:
the tape it records, replayed for any prefix, gives the state the forward had there.

Bars: fp32 state and fp32 tape rel-L2 <= 2e-5; y (rounded to the input dtype) within one
rounding of the input dtype of the exact value; low-precision states compared against the
oracle run with the same per-step rounding."""
import numpy as np
import pytest
import torch

import dflash_mlx_amd._native as nat
from dflash_mlx_amd.gdn_layer import gated_norm
from dflash_mlx_amd.kernels import (_gated_delta_ops_with_tape, fused_output_norm_applies,
                                    gated_delta_kernel_with_tape, tape_replay_kernel)
from oracle import dflash_oracle as O

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _case(B=2, T=16, Hk=4, Hv=8, Dk=128, Dv=128, seed=0, g_per_dk=False, dtype=torch.bfloat16,
          state_dtype=torch.float32):
    g = torch.Generator().manual_seed(0xDF1A + seed)
    q = torch.randn((B, T, Hk, Dk), generator=g)
    k = torch.randn((B, T, Hk, Dk), generator=g)
    q = (q / q.norm(dim=-1, keepdim=True) * Dk ** -0.5).to(dtype)
    k = (k / k.norm(dim=-1, keepdim=True)).to(dtype)
    v = torch.randn((B, T, Hv, Dv), generator=g).to(dtype)
    gshape = (B, T, Hv, Dk) if g_per_dk else (B, T, Hv)
    gate = torch.exp(-torch.nn.functional.softplus(torch.randn(gshape, generator=g)))
    beta = torch.sigmoid(torch.randn((B, T, Hv), generator=g)).to(dtype)
    state = (torch.randn((B, Hv, Dv, Dk), generator=g) * 0.1).to(state_dtype)
    return q, k, v, gate, beta, state


def _f64(t):
    return t.detach().cpu().to(torch.float64).numpy()


def _rel(a, b):
    a, b = np.asarray(a, np.float64), np.asarray(b, np.float64)
    return float(np.linalg.norm(a - b) / max(np.linalg.norm(b), 1e-30))


def _run(args, mask=None):
    dev = [t.to(DEV) for t in args]
    y, s, tape = gated_delta_kernel_with_tape(*dev, mask=None if mask is None else mask.to(DEV))
    torch.cuda.synchronize()
    return y, s, tape


@pytest.mark.parametrize("g_per_dk", [False, True])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
def test_against_fp64_oracle(native_lib, g_per_dk, dtype):
    args = _case(seed=1 + int(g_per_dk), g_per_dk=g_per_dk, dtype=dtype)
    y, s, tape = _run(args)
    assert y.dtype == dtype and s.dtype == torch.float32 and tape.dtype == torch.float32
    yo, so, to = O.gated_delta_ops_with_tape(*[_f64(t) for t in args])
    assert _rel(_f64(s), so) <= 2e-5
    assert _rel(_f64(tape), to) <= 2e-5
    eps = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11, torch.float32: 2.0 ** -20}[dtype]
    assert np.all(np.abs(_f64(y) - yo) <= eps * np.abs(yo) + 2e-5 * np.abs(yo).max())


def test_config2_shape_all_heads(native_lib):
    """32 value heads of 128 x 128 with 16 key heads, 16 steps: the GDN layer shape of config[2]."""
    args = _case(B=3, Hk=16, Hv=32, seed=7)
    y, s, tape = _run(args)
    yo, so, to = O.gated_delta_ops_with_tape(*[_f64(t) for t in args])
    assert _rel(_f64(s), so) <= 2e-5 and _rel(_f64(tape), to) <= 2e-5 and _rel(_f64(y), yo) <= 4e-3


def test_mask_skips_steps(native_lib):
    args = _case(seed=3)
    mask = torch.tensor([[1, 1, 0, 1, 0, 0, 1, 1, 1, 0, 1, 1, 1, 1, 0, 1],
                         [0, 0, 1, 1, 1, 1, 1, 1, 1, 1, 1, 1, 1, 1, 1, 0]], dtype=torch.bool)
    y, s, tape = _run(args, mask)
    yo, so, to = O.gated_delta_ops_with_tape(*[_f64(t) for t in args], mask=mask.numpy())
    assert _rel(_f64(s), so) <= 2e-5 and _rel(_f64(tape), to) <= 2e-5
    off = ~mask
    assert torch.all(tape.cpu()[off] == 0) and torch.all(y.cpu()[off] == 0)


def test_recorded_tape_replays_to_every_prefix_state(native_lib):
    """The contract between the two kernels (dflash_mlx/recurrent_rollback_cache.py:160-167)."""
    q, k, v, gate, beta, state = _case(seed=5)
    y, s_full, tape = _run((q, k, v, gate, beta, state))
    kd, gd, sd = k.to(DEV), gate.to(DEV), state.to(DEV)
    for a in (0, 1, 7, 16):
        prefix = [t[:, :a] for t in (q, k, v, gate, beta)]
        if a == 0:
            want = sd
        else:
            _, want, _ = _run(prefix + [state])
        got = tape_replay_kernel(tape[:, :a], kd[:, :a], gd[:, :a], sd) if a else sd
        assert _rel(_f64(got), _f64(want)) <= 2e-5
    assert _rel(_f64(tape_replay_kernel(tape, kd, gd, sd)), _f64(s_full)) <= 2e-5


@pytest.mark.parametrize("state_dtype", [torch.bfloat16, torch.float16])
def test_low_precision_state_is_rounded_after_every_step(native_lib, state_dtype):
    """kernels.py:96-98: the state goes through its storage type after every step."""
    args = _case(B=1, Hk=2, Hv=2, seed=9, state_dtype=state_dtype)
    y, s, tape = _run(args)
    assert s.dtype == state_dtype
    # the same recurrence on the host, fp32 arithmetic, rounding through the state dtype per step
    q, k, v, gate, beta, state = args
    S = state.float()
    tapes = []
    for t in range(q.shape[1]):
        _, S, tp = _gated_delta_ops_with_tape(q[:, t:t + 1].float(), k[:, t:t + 1].float(), v[:, t:t + 1].float(),
                                              gate[:, t:t + 1], beta[:, t:t + 1].float(), S)
        S = S.to(state_dtype).float()
        tapes.append(tp)
    assert _rel(_f64(s), _f64(S)) <= 2e-3            # one unit of the state dtype here and there
    assert _rel(_f64(tape), _f64(torch.cat(tapes, dim=1))) <= 2e-3


@pytest.mark.parametrize("shape", [dict(Dk=64, Dv=64), dict(Dk=96, Dv=32, Hk=2, Hv=2), dict(Dk=128, Dv=64),
                                   dict(T=3), dict(T=40, Hk=1, Hv=2, B=1)])
def test_other_shapes(native_lib, shape):
    args = _case(seed=11, **shape)
    y, s, tape = _run(args)
    yo, so, to = O.gated_delta_ops_with_tape(*[_f64(t) for t in args])
    assert _rel(_f64(s), so) <= 2e-5 and _rel(_f64(tape), to) <= 2e-5 and _rel(_f64(y), yo) <= 4e-3


@pytest.mark.parametrize("T", [1, 2, 7, 15, 16])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_closed_form_block_lengths(native_lib, T, dtype):
    """Scalar gate, fp32 state, 128 x 128 heads, T <= 16: the block kernel on the matrix cores,
    every block length with a ragged mask, against the fp64 oracle."""
    args = _case(B=2, T=T, Hk=2, Hv=4, seed=20 + T, dtype=dtype)
    mask = torch.ones((2, T), dtype=torch.bool)
    mask[1, T // 2] = False
    y, s, tape = _run(args, mask)
    yo, so, to = O.gated_delta_ops_with_tape(*[_f64(t) for t in args], mask=mask.numpy())
    assert _rel(_f64(s), so) <= 2e-5 and _rel(_f64(tape), to) <= 2e-5
    eps = {torch.bfloat16: 2.0 ** -8, torch.float32: 2.0 ** -20}[dtype]
    assert np.all(np.abs(_f64(y) - yo) <= eps * np.abs(yo) + 2e-5 * np.abs(yo).max())


def test_closed_form_with_vanishing_gates(native_lib):
    """Gates near 1e-4 per step: the running product leaves the fp32 range after a few steps,
    the ratios c_t / c_s between neighbouring steps do not.  Also gates of exactly 0 and 1."""
    q, k, v, gate, beta, state = _case(B=2, Hk=2, Hv=4, seed=31)
    gate = gate * 1e-4
    gate[0, 3, 1] = 0.0
    gate[1, :, 2] = 1.0
    args = (q, k, v, gate, beta, state)
    y, s, tape = _run(args)
    yo, so, to = O.gated_delta_ops_with_tape(*[_f64(t) for t in args])
    assert np.all(np.isfinite(_f64(s))) and np.all(np.isfinite(_f64(tape)))
    assert _rel(_f64(s), so) <= 2e-5 and _rel(_f64(tape), to) <= 2e-5 and _rel(_f64(y), yo) <= 4e-3


def test_closed_form_equals_the_sequential_kernel(native_lib, monkeypatch):
    """The two kernels for the same shape differ only in the order of fp32 additions."""
    args = _case(B=2, Hk=4, Hv=8, seed=33)
    mask = torch.ones((2, 16), dtype=torch.bool)
    mask[0, 5:8] = False
    block = _run(args, mask)
    assert native_lib.dflash_set_option(nat.OPT_GDN_STEP_BY_STEP, 1) == 0
    try:
        steps = _run(args, mask)
    finally:
        native_lib.dflash_set_option(nat.OPT_GDN_STEP_BY_STEP, 0)
    for a, b in zip(block, steps):
        assert _rel(_f64(a), _f64(b)) <= 2e-5
    assert _rel(_f64(block[2]), _f64(steps[2])) > 0     # two different kernels did run


@pytest.mark.parametrize("spread", ["even", "wide"])
def test_bf16_arrays_take_the_16_bit_matrix_cores_without_losing_a_bit(native_lib, spread):
    """With bf16 q and k the block kernel multiplies the fp32 state (cut exactly into three bf16
    pieces) on the bf16 matrix cores; with fp16 arrays it keeps the fp32 matrix cores.  The same
    numbers handed over either way must come back equally close to the fp64 result: 5e-7, forty
    times below the bar of the other tests, and far below the 2^-9 a state piece left out or
    rounded instead of cut would cost.  `wide`: state entries from 1e-12 to 1e+3 in one head."""
    q, k, v, gate, beta, state = _case(seed=21, dtype=torch.bfloat16)
    q, k, v, beta = [(t.float().clamp(-4, 4)) for t in (q, k, v, beta)]
    tiny = q.abs() < 2.0 ** -10                      # fp16 would hold these with fewer bits than bf16
    q = torch.where(tiny, torch.zeros_like(q), q)
    k = torch.where(k.abs() < 2.0 ** -10, torch.zeros_like(k), k)
    v = torch.where(v.abs() < 2.0 ** -10, torch.zeros_like(v), v)
    if spread == "wide":
        g = torch.Generator().manual_seed(77)
        state = state * torch.pow(10.0, torch.randint(-11, 5, state.shape, generator=g).float())
    got = {}
    for dt in (torch.bfloat16, torch.float16):
        args = [q.to(dt), k.to(dt), v.to(dt), gate, beta.to(dt), state]
        for a, b in zip(args[:3], (q, k, v)):
            assert torch.equal(a.float(), b)         # the same numbers in both dtypes
        ref = O.gated_delta_ops_with_tape(*[_f64(t) for t in args])
        y, s, tape = _run(args)
        assert _rel(_f64(s), ref[1]) <= 5e-7 and _rel(_f64(tape), ref[2]) <= 5e-7, (dt, spread)
        got[dt] = (s, tape)
    assert _rel(_f64(got[torch.bfloat16][0]), _f64(got[torch.float16][0])) <= 5e-7
    assert _rel(_f64(got[torch.bfloat16][1]), _f64(got[torch.float16][1])) <= 5e-7
    # Element by element: the two routes add the same exact products in another order, so a state
    # entry may differ by the roundings of its partial sums, never by more.  An entry is a sum of
    # T + 1 terms, each with a rounding of its own and the roundings of the delta it is made from:
    #   S_T = c_T S_0 + sum_t (c_T / c_t) delta_t (x) k_t,   c_t = g_1 .. g_t
    # Bar: 8 units in the last place of fp32 at the size of the entry's terms (not at the size of
    # the entry itself, which cancellation can make much smaller); 2.5 units are seen.  The third
    # bf16 piece of a state entry left out would cost 2^-16 of a term, sixteen times the bar.
    g64, k64, tape64, s064 = _f64(gate), _f64(k), ref[2], _f64(state)
    B, T, Hv = g64.shape
    rep = Hv // k64.shape[2]
    c = np.cumprod(g64, axis=1)                                   # [B, T, Hv]
    size = np.abs(c[:, -1][:, :, None, None] * s064)
    for t in range(T):
        w = (c[:, -1] / c[:, t])[:, :, None, None]
        size += np.abs(w * tape64[:, t][:, :, :, None] * np.repeat(k64[:, t], rep, axis=1)[:, :, None, :])
    diff = np.abs(_f64(got[torch.bfloat16][0]) - _f64(got[torch.float16][0]))
    assert np.all(diff <= 2.0 ** -20 * size), float((diff / (2.0 ** -23 * size + 1e-300)).max())


@pytest.mark.parametrize("shape", [
    dict(T=17), dict(T=31, Hk=1, Hv=3), dict(T=32, Dk=64, Dv=64), dict(T=33, B=1), dict(T=63, Dk=64, Dv=48, Hk=2, Hv=2),
    dict(T=65, B=1, Hk=2, Hv=8, Dv=16), dict(T=200, B=1, Hk=1, Hv=2)])
@pytest.mark.parametrize("masked", [False, True])
def test_prompts_in_chunks(native_lib, shape, masked):
    """More than 16 tokens: chunks of 32 on the matrix cores.  One token to several chunks, last chunks
    of one token and full ones, state slices of one and of several waves, against the fp64 oracle; the
    three-piece products carry fp32 accuracy, so the bars are those of the 16-token kernel."""
    args = _case(seed=50 + shape["T"], **shape)
    B, T = args[0].shape[:2]
    mask = None
    if masked:
        mask = torch.rand((B, T), generator=torch.Generator().manual_seed(T)) > 0.3
    y, s, tape = _run(args, mask)
    yo, so, to = O.gated_delta_ops_with_tape(*[_f64(t) for t in args], mask=None if mask is None else mask.numpy())
    assert _rel(_f64(s), so) <= 2e-5 and _rel(_f64(tape), to) <= 2e-5
    assert np.all(np.abs(_f64(y) - yo) <= 2.0 ** -8 * np.abs(yo) + 2e-5 * np.abs(yo).max())
    if masked:
        assert torch.all(tape.cpu()[~mask] == 0) and torch.all(y.cpu()[~mask] == 0)


@pytest.mark.parametrize("state_dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("in_dtype", [torch.bfloat16, torch.float16])
def test_prompts_with_a_low_precision_state(native_lib, state_dtype, in_dtype):
    """bf16 arrays: the state is rounded once, behind the last token (half a unit of its type).  fp16
    arrays take the step-by-step kernel, whose state is rounded at every one of the 70 steps."""
    args = _case(B=1, T=70, Hk=2, Hv=2, seed=61, dtype=in_dtype, state_dtype=state_dtype)
    y, s, tape = _run(args)
    yo, so, to = O.gated_delta_ops_with_tape(*[_f64(t) for t in args])
    half = 2.0 ** (-9 if state_dtype == torch.bfloat16 else -12)
    # a rounding decays with the gates (0.2 to 0.9 a step, mean 0.5), so few steps' roundings are alive at a time
    bar = half if in_dtype == torch.bfloat16 else 4 * half
    assert s.dtype == state_dtype and _rel(_f64(s), so) <= bar
    assert _rel(_f64(tape), to) <= (2e-5 if in_dtype == torch.bfloat16 else 4 * half)


def test_errors_and_host_tensors(native_lib):
    q, k, v, gate, beta, state = _case(B=1, T=2, Hk=3, Hv=4, Dk=32, Dv=8)
    with pytest.raises(ValueError, match="Cannot align"):
        gated_delta_kernel_with_tape(q, k, v, gate, beta, state)
    q, k, v, gate, beta, state = _case(B=1, T=2, Hk=2, Hv=4, Dk=32, Dv=8)
    with pytest.raises(ValueError, match="Unsupported gating shape"):
        gated_delta_kernel_with_tape(q, k, v, gate[..., 0], beta, state)
    # host tensors: the array ops, as in the reference without its kernel
    y, s, tape = gated_delta_kernel_with_tape(q.float(), k.float(), v.float(), gate, beta.float(), state)
    yo, so, to = O.gated_delta_ops_with_tape(*[_f64(t) for t in (q, k, v, gate, beta, state)])
    assert _rel(_f64(s), so) <= 1e-5 and _rel(_f64(tape), to) <= 1e-5 and _rel(_f64(y), yo) <= 1e-5
    # the C entry point refuses aliasing and null pointers
    L = native_lib
    assert L.dflash_gdn_forward_tape(None, None, None, None, None, None, None, None, None, None,
                                     1, 1, 1, 1, 32, 8, 0, 2, 0, 2, 0, None) == -1


@pytest.mark.parametrize("accepted", [0, 5, 14])
def test_speculative_cycle_through_the_rollback_cache(native_lib, accepted):
    """One verify cycle of a GatedDeltaNet layer on the device (runtime.py:411-442, 878-907):
    arm, run the block with the tape recorded, roll back to `accepted` drafted tokens - the
    cache must hold what a run over only the committed accepted+1 tokens leaves."""
    from dflash_mlx_amd.recurrent_rollback_cache import RecurrentRollbackCache
    q, k, v, gate, beta, state = [t.to(DEV) for t in _case(B=1, Hk=4, Hv=8, seed=21)]
    C = 64
    gen = torch.Generator().manual_seed(5)
    conv0 = torch.randn((1, 3, C), generator=gen).to(torch.bfloat16).to(DEV)
    qkv = torch.randn((1, 16, C), generator=gen).to(torch.bfloat16).to(DEV)
    cache = RecurrentRollbackCache(size=2, conv_kernel_size=4)
    cache[0], cache[1] = conv0, state
    cache.arm_rollback()
    y, s_block, tape = gated_delta_kernel_with_tape(q, k, v, gate, beta, cache[1])
    cache.record_tape(tape=tape, k=k, g=gate, qkv=qkv)
    cache[0], cache[1] = qkv[:, -3:].clone(), s_block          # what the layer leaves after 16 tokens
    cache.rollback(accepted)
    torch.cuda.synchronize()
    n = accepted + 1
    y_n, s_n, _ = gated_delta_kernel_with_tape(q[:, :n], k[:, :n], v[:, :n], gate[:, :n], beta[:, :n], state)
    assert _rel(_f64(cache[1]), _f64(s_n)) <= 2e-5
    assert torch.equal(y[:, :n], y_n)                             # outputs of the kept tokens are the block's
    want_conv = torch.cat([conv0, qkv], dim=1)[:, n:n + 3]
    assert torch.equal(cache[0], want_conv)
    assert not cache._armed and cache._tape is None


@pytest.mark.parametrize("dtype,wdtype,state_dtype,T", [(torch.bfloat16, torch.bfloat16, torch.float32, 16),
                                                        (torch.float16, torch.float32, torch.float32, 16),
                                                        (torch.float32, torch.float32, torch.float32, 16),
                                                        (torch.bfloat16, torch.bfloat16, torch.float32, 5),
                                                        (torch.bfloat16, torch.bfloat16, torch.bfloat16, 16)])
def test_output_norm_in_the_same_launch(native_lib, dtype, wdtype, state_dtype, T):
    """silu(z) * rms_norm(y, weight) computed by the recurrence's launch: state and tape are those
    of the plain call bit for bit, and the output is the norm operator applied to the plain
    call's y - up to one rounding of the array dtype where the two add the squares in a different
    order (block kernel), exactly where the entry point runs the two kernels itself (bf16 state)."""
    args = [t.to(DEV) for t in _case(B=2, T=T, Hk=2, Hv=4, seed=40 + T, dtype=dtype, state_dtype=state_dtype)]
    g = torch.Generator().manual_seed(7)
    z = torch.randn((2, T, 4, 128), generator=g).to(dtype).to(DEV)
    weight = (1 + 0.2 * torch.randn(128, generator=g)).to(wdtype).to(DEV)
    mask = torch.ones((2, T), dtype=torch.bool)
    mask[1, T // 2] = False
    for m in (None, mask.to(DEV)):
        assert fused_output_norm_applies(args[0], args[2], args[5], z, weight)
        y, s_plain, tape_plain = gated_delta_kernel_with_tape(*args, mask=m)
        out, s_fused, tape_fused = gated_delta_kernel_with_tape(*args, mask=m, output_norm=(z, weight, 1e-6))
        torch.cuda.synchronize()
        assert torch.equal(s_plain, s_fused) and torch.equal(tape_plain, tape_fused)
        want = gated_norm(y, z, weight, 1e-6)
        if state_dtype != torch.float32:
            assert torch.equal(out, want)
        else:
            ulp = {torch.bfloat16: 2 ** -7, torch.float16: 2 ** -10, torch.float32: 2 ** -22}[dtype]
            w64, o64 = want.double(), out.double()
            assert bool(((o64 - w64).abs() <= 2 * ulp * w64.abs() + 1e-6).all())
            assert float((o64 - w64).norm() / w64.norm()) <= ulp / 4
        if m is not None:
            assert float(out[1, T // 2].abs().max()) == 0.0   # a masked step's output is zero, normed or not
    # a z of another shape is not taken
    assert not fused_output_norm_applies(args[0], args[2], args[5], z[..., :64], weight)
    with pytest.raises(ValueError):
        gated_delta_kernel_with_tape(*args, output_norm=(z[..., :64], weight, 1e-6))


def _same_values(got, want, bar):
    """NaN where the other has NaN, the same infinities, and finite values within ``bar`` of their norm."""
    got, want = got.detach().cpu().double(), want.detach().cpu().double()
    assert torch.equal(torch.isnan(got), torch.isnan(want))
    assert torch.equal(torch.isinf(got), torch.isinf(want)) and torch.equal(got[torch.isinf(got)], want[torch.isinf(want)])
    ok = torch.isfinite(want)
    assert float((got[ok] - want[ok]).norm()) <= bar * max(float(want[ok].norm()), 1e-30)


@pytest.mark.parametrize("shape", [dict(T=70, B=2), dict(T=100, B=1, Dk=64, Dv=48, Hk=2, Hv=2)])
@pytest.mark.parametrize("what", ["v", "k", "q", "g", "beta", "state"])
@pytest.mark.parametrize("value", [float("nan"), float("inf"), -float("inf")])
def test_a_non_finite_value_in_a_prompt_reaches_what_comes_after_it(native_lib, shape, what, value):
    """Token by token, a NaN or an infinity at one token touches that token and the ones behind it, in the rows of the state
    it enters; chunks of tokens must not hand it to the ones before or to other rows.  Against the array operators on the host."""
    args = list(_case(seed=70, **shape))
    for at in (5, 37):  # in the first chunk and in one that a state is carried into
        new = [t.clone() for t in args]
        which = ["q", "k", "v", "g", "beta", "state"].index(what)
        if what == "state":
            new[which][0, 1, 3, 7] = value
        elif what in ("g", "beta"):
            new[which][0, at, 1] = value
        else:
            new[which][0, at, 1, 9] = value
        y, s, tape = _run(new)
        wide = [t.double() for t in new]
        yo, so, to = _gated_delta_ops_with_tape(*wide)
        _same_values(y, yo, 4e-3)
        _same_values(s, so, 2e-5)
        _same_values(tape, to, 2e-5)


@pytest.mark.parametrize("T", [17, 70])
def test_what_a_mask_hides_in_a_prompt_has_no_effect(native_lib, T):
    """A masked token is skipped whatever it holds: the same bits as with ordinary values in its place."""
    args = _case(seed=71, T=T)
    mask = torch.rand((2, T), generator=torch.Generator().manual_seed(T)) > 0.4
    mask[:, 3], mask[:, 16] = False, False
    plain = _run(args, mask)
    for value in (float("nan"), float("inf")):
        hidden = [t.clone() for t in args]
        for t in hidden[:5]:
            t[~mask] = value
        for a, b in zip(_run(hidden, mask), plain):
            assert torch.equal(a, b)
    # and together with a value that counts
    last = int(torch.nonzero(mask[0])[-1])
    hidden[2][0, last, 1, 5] = float("nan")
    y, s, tape = _run(hidden, mask)
    assert bool(torch.isnan(s[0, 1, 5]).all()) and int(torch.isnan(s).sum()) == 128
    assert int(torch.isnan(y).sum()) == 1 and int(torch.isnan(tape).sum()) == 1


def test_magnitudes_whose_products_leave_the_range_of_fp32(native_lib):
    """Keys and values of 1e20 overflow in the closed form of a chunk (k . k) before they do token by token."""
    q, k, v, g, beta, state = _case(seed=72, T=40, Hk=2, Hv=2)
    k[0, 20] *= 1e20
    v[1, 30] *= 1e30
    wide = [t.float() for t in (q, k, v, g, beta, state)]
    yo, so, to = _gated_delta_ops_with_tape(*wide)
    y, s, tape = _run((q, k, v, g, beta, state))
    for before, (a, b) in ((20, (y[0], yo[0])), (20, (tape[0], to[0]))):
        _same_values(a[:before], b[:before], 4e-3)
        assert bool(torch.isfinite(a[:before]).all())
    _same_values(y[1], yo[1], 4e-3)
    _same_values(tape[1], to[1], 2e-5)
    _same_values(s[1], so[1], 2e-5)


@pytest.mark.parametrize("state_dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("B,T,Hk,Hv,Dk,Dv,dtype", [(1, 1, 2, 4, 128, 128, torch.bfloat16), (2, 16, 2, 4, 128, 48, torch.bfloat16),
                                                   (9, 7, 8, 16, 128, 128, torch.bfloat16), (1, 16, 4, 8, 64, 64, torch.bfloat16),
                                                   (1, 33, 1, 2, 64, 96, torch.float16), (9, 16, 16, 32, 64, 64, torch.float32),
                                                   (2, 17, 2, 2, 128, 64, torch.float32)])
def test_rows_of_the_state_in_registers(native_lib, state_dtype, B, T, Hk, Hv, Dk, Dv, dtype):
    """The kernel that spreads a head over workgroups of some of its rows: one and two rows per lane, blocks of 16
    steps and what is left of them, masked steps; against the recurrence in fp64 with the state rounded after every step."""
    args = _case(B=B, T=T, Hk=Hk, Hv=Hv, Dk=Dk, Dv=Dv, seed=B + T + Dk + Dv, dtype=dtype, state_dtype=state_dtype)
    q, k, v, gate, beta, state = (t.double() for t in args)
    mask = torch.rand((B, T), generator=torch.Generator().manual_seed(T)) > 0.25
    mask[0, -1] = True
    for m in (None, mask):
        y, s, tape = _run(args, m)
        assert s.dtype == state_dtype and y.dtype == dtype
        S, ys, tapes = state, [], []
        for t in range(T):
            yt, S, tp = _gated_delta_ops_with_tape(q[:, t:t + 1], k[:, t:t + 1], v[:, t:t + 1], gate[:, t:t + 1], beta[:, t:t + 1], S,
                                                   None if m is None else m[:, t:t + 1])
            S = S.to(state_dtype).double()
            ys.append(yt)
            tapes.append(tp)
        # one unit of a 16-bit state here and there (as for whole heads above); y is rounded to its own type
        tol = 2e-5 if state_dtype == torch.float32 else 2e-3
        tol_y = max(tol, {torch.bfloat16: 4e-3, torch.float16: 5e-4, torch.float32: 0.0}[dtype])
        assert _rel(_f64(s), _f64(S)) <= tol
        assert _rel(_f64(tape), _f64(torch.cat(tapes, dim=1))) <= tol
        assert _rel(_f64(y), _f64(torch.cat(ys, dim=1))) <= tol_y


@pytest.mark.parametrize("shape", [dict(T=70, B=2), dict(T=33, B=4, Dk=64, Dv=48), dict(T=40, B=2, Hk=1, Hv=1, Dv=16)])
@pytest.mark.parametrize("masked", [False, True])
@pytest.mark.parametrize("value", [0.5, float("nan"), float("inf")])
def test_prompts_of_few_heads_and_of_many(native_lib, shape, masked, value):
    """Up to 256 (head, 16 rows) a row of the state is spread over the waves of a workgroup, above that one wave holds it.  Batches of
    one kind, repeated into the other: sums in another order, each within the bar against fp64 (twice it between them),
    and one rounding of y each."""
    args = _case(seed=80 + shape["T"], **shape)
    args[2][0, 11, 0, 5] = value
    B, T, Hv, Dv = args[2].shape
    few, mask = B * Hv * (Dv // 16), None
    times = 256 // few + 1
    assert few <= 256 < few * times
    if masked:
        mask = torch.rand((B, T), generator=torch.Generator().manual_seed(T)) > 0.3
        mask[0, 11] = True
    y, s, tape = _run(args, mask)
    many = _run([torch.cat([t] * times) for t in args], None if mask is None else torch.cat([mask] * times))
    for i in range(times):
        y2, s2, tape2 = (t[i * B:(i + 1) * B] for t in many)
        _same_values(s2, s, 4e-5)
        _same_values(tape2, tape, 4e-5)
        _same_values(y2, y, 2.0 ** -7)


@pytest.mark.parametrize("shape", [dict(T=100, B=1), dict(T=33, B=33), dict(T=40, B=2, Hk=1, Hv=1, Dv=16), dict(T=32, B=2, Dk=64, Dv=48)])
@pytest.mark.parametrize("masked", [False, True])
@pytest.mark.parametrize("at", [None, 3, 31])
def test_a_prompt_without_its_tape_has_the_bits_of_one_with_it(native_lib, shape, masked, at):
    """Rows of a state on several waves and on one, chunks walked token by token (the first, with others behind it, and the last)."""
    args = _case(seed=90 + shape["T"], **shape)
    B, T, Hv, Dv = args[2].shape
    mask = None
    if masked:
        mask = torch.rand((B, T), generator=torch.Generator().manual_seed(T)) > 0.3
    if at is not None:
        args[2][0, at, 0, 5] = float("inf")
        args[1][-1, at, 0, 7] = 1e25  # k . k leaves the range, the recurrence does not
    on_device = [t.to(DEV) for t in args]
    m = None if mask is None else mask.to(DEV)
    y, state, tape = gated_delta_kernel_with_tape(*on_device, m)
    y2, state2, none = gated_delta_kernel_with_tape(*on_device, m, with_tape=False)
    assert none is None and tape is not None

    def bits(t):
        return t.view(torch.int16 if t.element_size() == 2 else torch.int32)

    for a, b in ((y, y2), (state, state2)):  # (a NaN is a NaN)
        assert torch.equal(torch.isnan(a), torch.isnan(b)) and torch.equal(bits(torch.nan_to_num(a)), bits(torch.nan_to_num(b)))
