"""The lean small-M kernel with two workgroups per CU (M <= 16 and more 16-column strips than CUs;
17..32 rows, at any width): whole outputs against a float64 evaluation on the device, and the bits of
the same columns from a call of at most one strip per CU (both forms add in one order). Every case
asks the plan that this kernel serves it."""

import ctypes

import pytest
import torch

from gpu_util import assert_gemm_close_dev, lib, stream, torch_ref_dev

pytestmark = pytest.mark.gpu

# M at the edges of 8-row copies and 16-row tiles; one strip past the CU count, a partial and a full
# second round, a full third, one strip past it; K below one stage per wave, one past a round of
# stages (16 waves x 2; two row tiles 16 x 1), long
CASES = [(1, 4112, 64), (1, 12288, 3072), (8, 8208, 640), (9, 8192, 2112), (16, 4144, 2112), (3, 12304, 64),
         (17, 1040, 64), (24, 4096, 1088), (32, 4112, 2112), (25, 8192, 1024), (18, 8208, 576), (30, 12288, 1088)]
LEAN, LEAN_PAIR = 3, 4


def _form(M, N, K, lora=0):
    ks = ctypes.c_int()
    assert lib().feather_scaled_mm_any_m_plan(M, N, K, ctypes.byref(ks)) == 10 and ks.value == 1
    return lib().feather_scaled_mm_any_m_smallm_form(M, N, K, lora)


@pytest.mark.parametrize("a_dtype,b_dtype,out_dtype", [
    (torch.float16, torch.float8_e5m2, torch.bfloat16), (torch.float16, torch.float8_e4m3fn, torch.float16),
    (torch.bfloat16, torch.float8_e5m2, torch.bfloat16)])
@pytest.mark.parametrize("M,N,K", CASES)
def test_small_m_pair(cuda, hk, M, N, K, a_dtype, b_dtype, out_dtype):
    e4m3 = b_dtype == torch.float8_e4m3fn
    assert _form(M, N, K) == LEAN_PAIR
    print("small-M pair", M, N, K, a_dtype, b_dtype, out_dtype, flush=True)
    g = torch.Generator(device=cuda).manual_seed(M + N + K)
    a = torch.randn(M, K, generator=g, device=cuda).to(a_dtype)
    w = torch.randn(N, K, generator=g, device=cuda) * 0.02
    s = (w.abs().max() / (448.0 if e4m3 else 57344.0)).float().reshape(1)
    bp = (w / s).to(b_dtype).view(N, K // 16, 16).permute(1, 0, 2).contiguous()
    bias = (torch.randn(N, generator=g, device=cuda) * 0.1).to(out_dtype)
    y = hk.scaled_mm_hip_any_m(a, bp, s, bias, out_dtype)
    ref = torch_ref_dev(a.half(), bp, s, bias, out_dtype, b_dtype=b_dtype)
    assert_gemm_close_dev(y, ref, out_dtype, f"{M}x{N}x{K}")
    n1 = 2048 if M <= 16 else 1024
    for n0 in range(0, N, n1):
        part = bp[:, n0:n0 + n1].contiguous()
        assert _form(M, part.shape[1], K) == (LEAN if M <= 16 else LEAN_PAIR)
        yp = hk.scaled_mm_hip_any_m(a, part, s, bias[n0:n0 + n1].contiguous(), out_dtype)
        assert torch.equal(yp.view(torch.int16), y[:, n0:n0 + n1].contiguous().view(torch.int16)), n0


@pytest.mark.parametrize("M,N,K,R", [(1, 4112, 1088, 32), (16, 8192, 2112, 64), (20, 4112, 64, 32), (32, 8208, 1088, 160)])
def test_small_m_pair_lora(cuda, hk, M, N, K, R):
    """The rank-R term is added to the finished result in the output type: the bits of the plain call
    plus the rounded product, up to the term's own rounding to the factors' type (fp32 sums of R terms)."""
    assert _form(M, N, K) == LEAN_PAIR and _form(M, N, K, lora=1) == LEAN_PAIR
    print("small-M pair lora", M, N, K, R, flush=True)
    g = torch.Generator(device=cuda).manual_seed(M + N + K)
    a = torch.randn(M, K, generator=g, device=cuda).bfloat16()
    bp = torch.randn(K // 16, N, 16, generator=g, device=cuda).to(torch.float8_e5m2)
    t = torch.randn(M, R, generator=g, device=cuda).bfloat16()
    u = torch.randn(N, R, generator=g, device=cuda).bfloat16()
    y0 = hk.scaled_mm_hip_any_m(a, bp, None, None, torch.bfloat16)
    y = hk.scaled_mm_hip_any_m_lora(a, bp, None, None, torch.bfloat16, t, u)
    want = y0.double() + t.double() @ u.double().T
    # two bf16 roundings: of the term (relative 2^-9) and of the sum
    bound = 2.0**-8 * ((t.double() @ u.double().T).abs() + want.abs()) + 1e-6
    assert ((y.double() - want).abs() <= bound).all()


STRIPS, WIDE = 1, 2


@pytest.mark.parametrize("M,N,K,form,split", [
    (31, 640, 9696, STRIPS, True), (17, 272, 11024, STRIPS, True), (32, 560, 8256, STRIPS, True),
    (26, 944, 10944, STRIPS, True), (29, 2736, 1824, STRIPS, False), (23, 9520, 752, WIDE, False),
    (41, 3616, 1056, STRIPS, False), (48, 4080, 400, STRIPS, False)])
def test_small_m_planned_forms(cuda, hk, M, N, K, form, split):
    """The other forms of 17..48 rows that the any-M plan hands to the launch (strip width and K split): whole
    outputs against float64, bf16 activations as their fp16 cast, and through the C entry without a workspace
    (K then split inside the workgroups only)."""
    ks = ctypes.c_int()
    assert lib().feather_scaled_mm_any_m_plan(M, N, K, ctypes.byref(ks)) == 10 and (ks.value > 1) == split
    assert lib().feather_scaled_mm_any_m_smallm_form(M, N, K, 0) == form
    assert (lib().feather_scaled_mm_any_m_workspace_size(M, N, K) > 0) == split
    print("small-M form", M, N, K, form, ks.value, flush=True)
    g = torch.Generator(device=cuda).manual_seed(M + N + K)
    ab = torch.randn(M, K, generator=g, device=cuda).bfloat16()
    a = ab.half()
    w = torch.randn(N, K, generator=g, device=cuda) * 0.02
    s = (w.abs().max() / 57344.0).float().reshape(1)
    bp = (w / s).to(torch.float8_e5m2).view(N, K // 16, 16).permute(1, 0, 2).contiguous()
    bias = (torch.randn(N, generator=g, device=cuda) * 0.1).half()
    ref = torch_ref_dev(a, bp, s, bias, torch.float16)
    y = hk.scaled_mm_hip_any_m(a, bp, s, bias, torch.float16)
    assert_gemm_close_dev(y, ref, torch.float16, f"{M}x{N}x{K}")
    for x in (ab, a):  # again, and with bf16 activations
        assert torch.equal(y.view(torch.int16), hk.scaled_mm_hip_any_m(x, bp, s, bias, torch.float16).view(torch.int16))
    c = torch.full((M, N), float("nan"), dtype=torch.float16, device=cuda)
    assert lib().feather_launch_scaled_mm_any_m(a.data_ptr(), 0, bp.data_ptr(), s.data_ptr(), bias.data_ptr(), c.data_ptr(),
                                                M, N, K, 1, 1, 1, 0, None, 0, stream(cuda))
    assert_gemm_close_dev(c, ref, torch.float16, f"{M}x{N}x{K} without a workspace")
