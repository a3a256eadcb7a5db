"""GPU parity of the fused fp16 prologue (sl8_quantize_qk).

Its outputs must equal the separate kernels (k_mean, smooth+quantise, Q
quantise) and the oracle bit for bit, and its gate flag must equal the torch
evaluation the reference performs (reference superl8/quant/core.py:113-145).
"""
import numpy as np
import pytest
import torch

from oracle import quant as oqn
from superl8_amd import _C, ops, quant

pytestmark = pytest.mark.gpu

LOG2E = quant.LOG2E
# (B, Hq, Hkv, M, N, D): ragged key counts across mean chunks (512) and quantise
# blocks (128), M = 1 decode, more Q rows than the grid-stride cap covers at once
SHAPES = [(1, 8, 2, 512, 512, 64), (2, 6, 3, 33, 777, 128), (1, 4, 1, 5, 1, 256),
          (1, 2, 2, 1, 70001, 64), (1, 32, 8, 4096, 4096, 128), (2, 16, 2, 300, 1025, 256),
          (3, 4, 4, 1, 130, 128)]


def _np(x):
    return x.detach().cpu().numpy()


def _torch_gate(q, thr=12.0):
    a = q.float().abs()
    return bool(((a.amax(-1) / (a.median(-1).values + 1e-10)) > thr).any())


@pytest.mark.parametrize("B,Hq,Hkv,M,N,D", SHAPES)
def test_fused_prologue_matches_separate_kernels(device, B, Hq, Hkv, M, N, D):
    g = torch.Generator(device="cpu").manual_seed(B * 1000 + N + D)
    q = (torch.randn(B, Hq, M, D, generator=g) * 1.5).half().to(device)
    k = (torch.randn(B, Hkv, N, D, generator=g) * 2).half().to(device)
    k[..., 5] += 7.0
    mul = (1.0 / D ** 0.5) * LOG2E
    qi, qs, ki, ks, km, flag = _C.quantize_qk_fused(q, k, mul, 12.0)
    m_ref = _C.k_mean(k)
    qi_ref, qs_ref = _C.quantize_rows_centered(q, None, mul)
    ki_ref, ks_ref = _C.quantize_rows_centered(k, m_ref, 1.0)
    assert torch.equal(km, m_ref)
    assert torch.equal(qi, qi_ref) and torch.equal(qs, qs_ref)
    assert torch.equal(ki, ki_ref) and torch.equal(ks, ks_ref)
    assert bool(flag.item()) == _torch_gate(q)
    if q.numel() * k.numel() < 1 << 30 and N < 5000:
        rq, rqs, rk, rks, rm = oqn.quantize_qk(_np(q), _np(k))
        np.testing.assert_array_equal(_np(km), rm)
        np.testing.assert_array_equal(_np(qi), rq)
        np.testing.assert_array_equal(_np(qs), rqs)
        np.testing.assert_array_equal(_np(ki), rk)
        np.testing.assert_array_equal(_np(ks), rks)


@pytest.mark.parametrize("D", [64, 128, 256])
def test_fused_prologue_nonfinite_rows(device, D):
    """NaN and +-inf elements: the fused codes (reciprocal + exact-division
    fallback) equal the separate kernels' (IEEE division per element) bit for
    bit: a NaN element codes to -127 (the clamp fmaxf / fminf), an inf row has
    an inf scale, its inf element codes to -127 and its finite ones to 0."""
    g = torch.Generator(device="cpu").manual_seed(D + 7)
    q = torch.randn(1, 2, 40, D, generator=g).half().to(device)
    k = torch.randn(1, 1, 40, D, generator=g).half().to(device)
    q[0, 0, 3, 5] = float("nan")
    q[0, 1, 7, 0] = float("inf")
    q[0, 1, 8, D - 1] = float("-inf")
    q[0, 0, 9, :] = float("nan")
    qi, qs, _, _, _, _ = _C.quantize_qk_fused(q, k, 1.0, 0.0)
    qi_ref, qs_ref = _C.quantize_rows_centered(q, None, 1.0)
    assert torch.equal(qi, qi_ref)
    assert torch.equal(qs.isnan(), qs_ref.isnan()) and torch.equal(qs.nan_to_num(), qs_ref.nan_to_num())
    assert int(qi[0, 0, 3, 5]) == -127 and (qi[0, 0, 9] == -127).all()
    assert int(qi[0, 1, 7, 0]) == -127 and (qi[0, 1, 7, 1:] == 0).all()
    assert torch.isinf(qs[0, 1, 7]).all()
    # the finite rows are untouched by the others
    fin = torch.isfinite(q.float()).all(-1)
    qi2, qs2, _, _, _, _ = _C.quantize_qk_fused(torch.where(fin[..., None], q, 0), k, 1.0, 0.0)
    assert torch.equal(qi[fin], qi2[fin]) and torch.equal(qs[fin], qs2[fin])


@pytest.mark.parametrize("D", [64, 128, 256])
def test_fused_gate_decisions(device, D):
    torch.manual_seed(D)
    k = torch.randn(1, 2, 64, D, device=device, dtype=torch.float16)
    cases = []
    q = torch.randn(1, 4, 3000, D, device=device, dtype=torch.float16)
    cases.append(q.clone())                       # gaussian: ratio ~ 5
    q1 = q.clone(); q1[0, 3, 2999, 1] = 200.0     # one spike in the last row
    cases.append(q1)
    q2 = q.clone(); q2[0, 1, 17] = 0.0            # all-zero row: 0 / 1e-10 = 0
    cases.append(q2)
    q3 = q.clone(); q3[0, 2, 5, : D // 2 + 1] = 0.0; q3[0, 2, 5, D - 1] = 1e-3  # median 0
    cases.append(q3)
    q4 = q.clone(); q4[0, 0, 9, 0] = float("nan"); q4[0, 0, 9, 1] = 5e4  # NaN row never fires
    cases.append(q4)
    for c in cases:
        for thr in (3.0, 12.0, 1e6):
            _, _, _, _, _, flag = _C.quantize_qk_fused(c, k, 1.0, thr)
            ref, _ = _C.q_outlier_gate(c, thr)
            assert bool(flag.item()) == bool(ref.item()) == _torch_gate(c, thr), (thr,)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("B,Hq,Hkv,M,N,D", [(1, 4, 2, 37, 129, 32), (2, 3, 3, 196, 196, 72),
                                            (1, 2, 1, 61, 6145, 80), (1, 4, 2, 5, 777, 64),
                                            (1, 2, 2, 130, 6300, 128), (1, 2, 1, 33, 12400, 256)])
def test_fused_prologue_types_and_head_dims(device, dtype, B, Hq, Hkv, M, N, D):
    """Both storage types at every head dim, key counts around the growing mean chunks
    (6144 keys on), against the separate kernels and the torch gate, bit for bit."""
    g = torch.Generator(device="cpu").manual_seed(N + D)
    q = (torch.randn(B, Hq, M, D, generator=g) * 1.5).to(dtype).to(device)
    k = (torch.randn(B, Hkv, N, D, generator=g) * 2 + 3).to(dtype).to(device)
    q[0, 0, 0, :] = 0
    m_ref = _C.k_mean(k)
    qi_ref, qs_ref = _C.quantize_rows_centered(q, None, 0.3)
    ki_ref, ks_ref = _C.quantize_rows_centered(k, m_ref, 1.0)
    for spike in (False, True):
        if spike:
            q[-1, -1, -1, :] = 0.01
            q[-1, -1, -1, D - 1] = 90.0
            qi_ref, qs_ref = _C.quantize_rows_centered(q, None, 0.3)
        thr = 12.0 if D > 32 else 40.0   # 32 Gaussian values: the median is too loose for 12
        qi, qs, ki, ks, km, flag = _C.quantize_qk_fused(q, k, 0.3, thr)
        assert torch.equal(km, m_ref)
        assert torch.equal(qi, qi_ref) and torch.equal(qs, qs_ref)
        assert torch.equal(ki, ki_ref) and torch.equal(ks, ks_ref)
        assert bool(flag.item()) == _torch_gate(q, thr) == spike


def test_gate_boundary_exact(device):
    """Rows built so that max/median lands on either side of the threshold by one ulp."""
    D = 128
    torch.manual_seed(3)
    k = torch.randn(1, 1, 16, D, device=device, dtype=torch.float16)
    for med, mx in [(1.0, 12.0), (1.0, 12.0078125), (0.5, 6.0), (0.5, 6.00390625), (2.0, 24.0)]:
        row = torch.full((D,), med, dtype=torch.float16)
        row[: D // 2 - 1] = med / 2
        row[-1] = mx
        q = row.reshape(1, 1, 1, D).to(device)
        _, _, _, _, _, flag = _C.quantize_qk_fused(q, k, 1.0, 12.0)
        assert bool(flag.item()) == _torch_gate(q), (med, mx)


def test_attn_fwd_routes_on_fused_gate(device):
    torch.manual_seed(11)
    q = torch.randn(1, 4, 256, 64, device=device, dtype=torch.float16)
    k = torch.randn(1, 2, 256, 64, device=device, dtype=torch.float16)
    v = torch.randn(1, 2, 256, 64, device=device, dtype=torch.float16)
    ref = torch.nn.functional.scaled_dot_product_attention(q, k, v, is_causal=True, enable_gqa=True)
    o = ops.attn_int8_fwd(q, k, v, causal=True)
    assert (o.float() - ref.float()).abs().max().item() < 5e-2
    q[0, 1, 100, 7] = 300.0   # gate fires: the call returns full-precision SDPA exactly
    ref = torch.nn.functional.scaled_dot_product_attention(q, k, v, is_causal=True, enable_gqa=True)
    o = ops.attn_int8_fwd(q, k, v, causal=True)
    assert torch.equal(o, ref)


@pytest.mark.parametrize("dtype,D", [(torch.bfloat16, 128), (torch.bfloat16, 72), (torch.float16, 80)])
def test_attn_fwd_gate_of_new_prologue_forms(device, dtype, D):
    """bf16 and the head dims 72 / 80 take the deferred gate: quiet and firing calls, and
    inputs at an odd offset (the separate kernels) give the same codes and the same output."""
    torch.manual_seed(12)
    q, k, v = (torch.randn(1, h, 200, D, device=device).to(dtype) for h in (4, 2, 2))
    o = ops.attn_int8_fwd(q, k, v, causal=True)
    flat = torch.empty(q.numel() + 1, device=device, dtype=dtype)
    flat[1:] = q.reshape(-1)
    assert torch.equal(ops.attn_int8_fwd(flat[1:].view_as(q), k, v, causal=True), o)
    q[0, 1, 100, 7] = 300.0
    ref = torch.nn.functional.scaled_dot_product_attention(q, k, v, is_causal=True, enable_gqa=True)
    assert torch.equal(ops.attn_int8_fwd(q, k, v, causal=True), ref)


def test_fused_rejects(device):
    q = torch.randn(1, 1, 4, 96, device=device, dtype=torch.float16)
    with pytest.raises(RuntimeError):
        _C.quantize_qk_fused(q, q, 1.0)
    with pytest.raises(RuntimeError):
        _C.quantize_qk_fused(q.float()[..., :64].contiguous(), q.float()[..., :64].contiguous(), 1.0)


def test_gated_prefill_skips_or_matches(device):
    """sl8_attn_int8_fwd_gated through the C ABI: with the flag set every
    workgroup exits and the output buffer keeps its contents; with it clear the
    output is bit-identical to sl8_attn_int8_fwd's."""
    from superl8_amd import _lib
    from superl8_amd._lib import dtype_code

    torch.manual_seed(5)
    B, Hq, Hkv, M, N, D = 1, 4, 2, 200, 300, 128
    q = torch.randn(B, Hq, M, D, device=device, dtype=torch.float16)
    k = torch.randn(B, Hkv, N, D, device=device, dtype=torch.float16)
    v = torch.randn(B, Hkv, N, D, device=device, dtype=torch.float16)
    q_i8, qs, k_i8, ks, _ = quant.quantize_qk(q, k)
    qs, ks = qs.squeeze(-1).contiguous(), ks.squeeze(-1).contiguous()
    ref = _C.attn_int8_fwd(q_i8, qs, k_i8, ks, v, True)
    lib = _lib.load()
    stream = torch.cuda.current_stream().cuda_stream
    for flag_val in (1, 0):
        flag = torch.full((1,), flag_val, device=device, dtype=torch.int32)
        out = torch.full_like(ref, 7.0)
        rc = lib.sl8_attn_int8_fwd_gated(q_i8.data_ptr(), qs.data_ptr(), k_i8.data_ptr(),
                                         ks.data_ptr(), v.data_ptr(), dtype_code(v.dtype),
                                         out.data_ptr(), None, B, Hq, Hkv, M, N, D, 1, -1,
                                         None, 0, flag.data_ptr(), stream)
        assert rc == 0, lib.sl8_last_error()
        torch.cuda.synchronize()
        if flag_val:
            assert torch.equal(out, torch.full_like(ref, 7.0))
        else:
            assert torch.equal(out, ref)


def test_public_prefill_deferred_gate_is_the_two_step_path(device):
    """ops.attn_int8_fwd reads the fused prologue's gate flag after launching the
    attention: a call whose gate stays quiet returns exactly prologue + kernel."""
    torch.manual_seed(6)
    q = torch.randn(2, 8, 300, 128, device=device, dtype=torch.float16)
    k = torch.randn(2, 2, 300, 128, device=device, dtype=torch.float16)
    v = torch.randn(2, 2, 300, 128, device=device, dtype=torch.float16)
    o = ops.attn_int8_fwd(q, k, v, causal=True)
    q_i8, qs, k_i8, ks, _ = quant.quantize_qk(q, k)
    two_step = _C.attn_int8_fwd(q_i8, qs.squeeze(-1).contiguous(), k_i8,
                                ks.squeeze(-1).contiguous(), v, True)
    assert torch.equal(o, two_step)


def test_public_prefill_gate_read_back_to_back(device):
    """Calls issued back to back, alternating inputs whose gate fires and stays
    quiet: each call's decision is its own (the flag is read from a pinned copy
    made right after its prologue, while its attention may still be running)."""
    torch.manual_seed(8)
    q = torch.randn(1, 4, 256, 128, device=device, dtype=torch.float16)
    k = torch.randn(1, 2, 256, 128, device=device, dtype=torch.float16)
    v = torch.randn(1, 2, 256, 128, device=device, dtype=torch.float16)
    q_out = q.clone()
    q_out[0, 1, 7, 3] = 300.0  # one dominated row: the gate fires for this input
    quiet = ops.attn_int8_fwd(q, k, v, causal=True)
    loud = ops.attn_int8_fwd(q_out, k, v, causal=True)
    fp_loud = torch.nn.functional.scaled_dot_product_attention(
        q_out, k, v, is_causal=True, enable_gqa=True)
    assert torch.allclose(loud.float(), fp_loud.float(), atol=2e-3, rtol=0)
    assert not torch.equal(quiet, loud)
    outs = [ops.attn_int8_fwd(x, k, v, causal=True) for x in (q, q_out, q, q, q_out, q_out, q)]
    torch.cuda.synchronize()
    for x, o in zip((q, q_out, q, q, q_out, q_out, q), outs):
        assert torch.equal(o, quiet if x is q else loud)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("G,N,D", [(2, 1, 128), (3, 63, 64), (2, 777, 72), (1, 6200, 256), (4, 300, 32),
                                   (2, 4097, 128)])
def test_cache_build_matches_separate_kernels(device, dtype, G, N, D):
    """quantize_kv_cache's fused build (and V alone) against k_mean, the centred row quantiser and
    the element-wise column quantiser (reached with D = 2 D columns viewed apart), bit for bit."""
    g = torch.Generator(device="cpu").manual_seed(N + D)
    k, v = ((torch.randn(1, G, N, D, generator=g) * 2 + 1).to(dtype).to(device) for _ in range(2))
    v[..., 3] = 0            # an all-zero channel: scale 1
    v[0, 0, N // 2, 5] = float("nan")   # skipped by the maximum, coded -127
    v[0, G - 1, 0, 7] = float("inf")    # an infinite scale: 0, and -127 for the element itself
    ki, ks, vi, vs = ops.quantize_kv_cache(k, v)
    mean = _C.k_mean(k)
    ki_ref, ks_ref = _C.quantize_rows_centered(k, mean, 1.0)
    assert torch.equal(ki, ki_ref) and torch.equal(ks, ks_ref)
    v32 = v.float()
    vi_ref, vs_ref = _C.quantize_v_perchannel(v32)   # float32 input: the element-wise kernels
    assert vs.shape == (1, G, D)
    assert torch.equal(vs, vs_ref.squeeze(-2)) and torch.equal(vi, vi_ref)
    vi2, vs2 = _C.quantize_v_perchannel(v)
    assert torch.equal(vi2, vi_ref) and torch.equal(vs2, vs_ref)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("D", [32, 64, 128, 256])
def test_rotated_prologue_against_64_bits(device, dtype, D):
    """Q and the smoothed K through the in-register rotation, against the rotation in 64 bits
    rounded to the storage type: a neighbouring rounding moves a scale by at most one unit in the
    last place of the type and a code by at most one step."""
    ulp = 2.0 ** -10 if dtype == torch.float16 else 2.0 ** -7
    q, k = (torch.randn(1, 2, n, D, device=device).to(dtype) for n in (33, 130))
    h = torch.ones(1, 1, dtype=torch.float64, device=device)
    while h.shape[0] < D:
        h = torch.cat([torch.cat([h, h], 1), torch.cat([h, -h], 1)], 0)
    qi, qs, ki, ks, km = quant.quantize_qk(q, k, softmax_scale=1.0 / LOG2E, rotate=True)
    assert torch.equal(km, _C.k_mean(k))
    k_s = (k.float() - km).to(dtype)
    for x, c, s in ((q, qi, qs), (k_s, ki, ks)):
        ref = (x.double() @ h / D ** 0.5).to(dtype).double()
        s_ref = ref.abs().amax(-1, keepdim=True) / 127
        assert ((s.double() / s_ref - 1).abs() <= ulp).all()
        c_ref = (ref / s_ref).round().clamp(-127, 127)
        assert ((c.double() - c_ref).abs() <= 1).all() and (c.double() != c_ref).float().mean() <= 0.02


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("M,N,D", [(1, 1, 64), (300, 77, 128), (64, 512, 72), (700, 33, 256)])
def test_host_flag_follows_the_device_flag(device, dtype, M, N, D):
    g = torch.Generator(device=device).manual_seed(3)
    k = torch.randn(1, 2, N, D, device=device, generator=g).to(dtype)
    calm = torch.randn(1, 4, M, D, device=device, generator=g).clamp(-2, 2).to(dtype)
    calm[..., 0] = 2.0
    last, first = calm.clone(), calm.clone()
    last[0, -1, -1, -1] = 4000.0  # one row fires, in the last block
    first[0, 0, 0, 0] = -4000.0
    for q, fires in ((calm, 0), (last, 1), (calm, 0), (first, 1)):
        host = torch.zeros(1, dtype=torch.int32, pin_memory=True)
        flag = _C.quantize_qk_fused(q, k, 1.0, 24.0, host)[5]
        ready = torch.cuda.Event()
        ready.record()
        ready.synchronize()
        assert int(host[0]) == flag.item() == fires
    with pytest.raises(RuntimeError, match="pinned"):
        _C.quantize_qk_fused(calm, k, 1.0, 24.0, torch.zeros(1, dtype=torch.int32))


@pytest.mark.parametrize("D", [32, 64, 128, 256])
def test_rotated_bf16_rows_near_the_largest_float(device, D):
    """Rows whose unscaled sums pass the largest float while the normalised rotation does not:
    against the rotation in 64 bits (a bf16 rounding, 2^-8, moves a scale by at most that and a code
    by one step)."""
    x = torch.ones(1, 2, 5, D, dtype=torch.float64)
    x[:, :, 1] *= torch.where(torch.arange(D) % 3 == 0, -1.0, 1.0).double()
    x[:, :, 2:] = torch.randn(1, 2, 3, D, dtype=torch.float64).clamp(-3, 3) / 3
    q = (x * 3.0e38 / D ** 0.5).to(torch.bfloat16).to(device)
    k = torch.randn(1, 2, 5, D, device=device).to(torch.bfloat16)
    qi, qs, *_ = quant.quantize_qk(q, k, softmax_scale=1.0 / LOG2E, rotate=True)
    h = torch.ones(1, 1, dtype=torch.float64, device=device)
    while h.shape[0] < D:
        h = torch.cat([torch.cat([h, h], 1), torch.cat([h, -h], 1)], 0)
    ref = (q.double() @ h / D ** 0.5).to(torch.bfloat16).double()
    assert torch.isfinite(ref).all() and torch.isfinite(qs).all()
    s_ref = ref.abs().amax(-1) / 127
    assert ((qs.squeeze(-1).double() / s_ref - 1).abs() <= 2.0 ** -7).all()
    assert ((qi.double() - (ref / s_ref[..., None]).round()).abs() <= 1).all()
