"""The any-M entry's planned tiles (32 x 64 up to 128 x 256, one and two K groups, K splits, any K): one
shape per tile and K remainder, whole outputs against a float64 evaluation on the device, under the
gate of gpu_util (fp32 sums in another order, two roundings to the output type)."""

import ctypes

import pytest
import torch

from gpu_util import assert_gemm_close_dev, lib, torch_ref_dev

pytestmark = pytest.mark.gpu

# (M, N, K, kernel id, K splits > 1): K a multiple of 128, of 64 only, of 16 only, below one stage
CASES = [
    (63, 224, 1152, 40, False), (77, 128, 1088, 40, False), (63, 240, 16, 40, False), (65, 256, 112, 40, False),
    (33, 128, 2480, 40, True), (48, 128, 2304, 40, True),
    (130, 5488, 128, 34, False), (130, 5664, 1232, 34, False), (17, 5456, 5648, 34, True),
    (191, 5024, 432, 30, False), (333, 1712, 3904, 30, False), (33, 2864, 4464, 30, True),
    (333, 2976, 1664, 41, False), (333, 3248, 4384, 41, False), (65, 3776, 5040, 41, True),
    (200, 5936, 80, 31, False), (777, 2160, 2816, 31, False), (97, 4160, 3984, 31, True),
    (333, 5504, 1264, 42, False), (333, 5408, 1728, 42, False), (200, 4640, 5520, 42, True),
    (500, 4384, 2352, 43, False), (500, 4416, 2368, 43, False), (200, 5504, 4528, 43, True),
    (2000, 4224, 80, 44, False), (1003, 4304, 896, 44, False), (777, 5056, 4880, 44, False),
    (200, 6112, 16, 45, False), (500, 5392, 128, 45, False), (777, 4064, 2704, 45, False),
    (777, 4688, 16, 46, False), (777, 5104, 64, 46, False), (1300, 3536, 2096, 46, False),
    (2000, 3088, 16, 47, False), (1300, 4576, 48, 47, False), (2000, 3712, 4528, 47, False),
    (1500, 4592, 1040, 47, False),
    # the split-K tiles on one group of waves (unsplit, K % 64 == 0 up to 1024): one stage of 64 K, fewer than
    # the ring's five, as many, one more, the longest; one round of workgroups and two
    (77, 128, 64, 30, False), (63, 224, 128, 30, False), (191, 5056, 320, 30, False), (97, 5040, 384, 30, False),
    (1003, 1632, 128, 30, False), (777, 4928, 64, 31, False), (200, 5952, 384, 31, False), (1578, 2544, 832, 31, False),
    (130, 5488, 1024, 34, False), (199, 8256, 192, 34, False),
]


@pytest.mark.parametrize("b_dtype,out_dtype", [(torch.float8_e5m2, torch.bfloat16), (torch.float8_e4m3fn, torch.float16)])
@pytest.mark.parametrize("M,N,K,kid,split", CASES)
def test_planned_tile(cuda, hk, M, N, K, kid, split, b_dtype, out_dtype):
    ks = ctypes.c_int()
    e4m3 = b_dtype == torch.float8_e4m3fn
    assert lib().feather_scaled_mm_any_m_plan(M, N, K, ctypes.byref(ks)) == kid
    assert (ks.value > 1) == split
    print("planned tile", M, N, K, "kernel", kid, "splits", ks.value, b_dtype, flush=True)
    g = torch.Generator(device=cuda).manual_seed(M + N + K)
    a = torch.randn(M, K, generator=g, device=cuda).half()
    w = torch.randn(N, K, generator=g, device=cuda) * 0.02
    s = (w.abs().max() / (448.0 if e4m3 else 57344.0)).float().reshape(1)
    bp = (w / s).to(b_dtype).view(N, K // 16, 16).permute(1, 0, 2).contiguous()
    bias = (torch.randn(N, generator=g, device=cuda) * 0.1).to(out_dtype)
    ref = torch_ref_dev(a, bp, s, bias, out_dtype, b_dtype=b_dtype)
    y = hk.scaled_mm_hip_any_m(a, bp, s, bias, out_dtype)
    assert_gemm_close_dev(y, ref, out_dtype, f"{M}x{N}x{K} kernel {kid}")
    assert torch.equal(y.view(torch.int16), hk.scaled_mm_hip_any_m(a, bp, s, bias, out_dtype).view(torch.int16))
    if not e4m3:  # bf16 activations: the bits of their fp16 cast (overflow, subnormals)
        ab = a.bfloat16()
        ab[0, :3] = torch.tensor([1.0e6, 3.0e-6, -5.0e-8], device=cuda)
        y = hk.scaled_mm_hip_any_m(ab, bp, s, bias, out_dtype)
        y16 = hk.scaled_mm_hip_any_m(ab.to(torch.float16), bp, s, bias, out_dtype)
        assert torch.equal(y.view(torch.int16), y16.view(torch.int16))
    # non-finite activations at both ends of K reach their own rows alone (the last stage's shared
    # part and chunks past K are zeroed in both operands)
    a[0, 0], a[M - 1, K - 1] = float("inf"), float("nan")
    ref = torch_ref_dev(a, bp, s, None, out_dtype, b_dtype=b_dtype)
    y = hk.scaled_mm_hip_any_m(a, bp, s, None, out_dtype)
    assert_gemm_close_dev(y, ref, out_dtype, f"{M}x{N}x{K} kernel {kid} non-finite")


# (M, N, K): one per planned tile and per place of the term's rounding, K splits, the lean small-M kernel (one and two
# row tiles), and the routes without a fused term
LORA_SHAPES = [
    (1, 4096, 1024), (16, 528, 512), (5, 13824, 5120), (31, 2048, 2048), (17, 1040, 1024),
    (63, 224, 128), (33, 128, 2480), (130, 5488, 128), (17, 5456, 5648), (333, 1712, 3904), (33, 2864, 4464),
    (333, 2976, 1664), (65, 3776, 5040), (777, 2160, 2816), (97, 4160, 3984), (333, 5408, 1728), (200, 4640, 5520),
    (500, 4416, 2368), (200, 5504, 4528), (1003, 4304, 896), (777, 5056, 4880), (1003, 1632, 128), (777, 4064, 2704),
    (777, 4928, 64), (1300, 3536, 2096), (2000, 3712, 4528), (2000, 6160, 128), (1300, 4640, 128), (2000, 4352, 1408),
    (2000, 4832, 128), (8, 2048, 12288),
]


def _check_lora(cuda, hk, M, N, K, R, out_dtype, f_dtype):
    g = torch.Generator(device=cuda).manual_seed(M + N + K + 1)
    a = torch.randn(M, K, generator=g, device=cuda).half()
    w = torch.randn(N, K, generator=g, device=cuda) * 0.02
    s = (w.abs().max() / 57344.0).float().reshape(1)
    bp = (w / s).to(torch.float8_e5m2).view(N, K // 16, 16).permute(1, 0, 2).contiguous()
    bias = (torch.randn(N, generator=g, device=cuda) * 0.1).to(out_dtype)
    t = (torch.randn(M, R, generator=g, device=cuda) * 0.2).to(f_dtype)
    u = (torch.randn(N, R, generator=g, device=cuda) * 0.05).to(f_dtype)
    print("planned tile, rank", R, "term", M, N, K, out_dtype, f_dtype, flush=True)
    y = hk.scaled_mm_hip_any_m_lora(a, bp, s, bias, out_dtype, t, u)
    term = t.double() @ u.double().t()
    if 20 <= hk.kernel_id(M, N, K, hk.any_m_config(M, N, K)) < 30:
        dec = bp.double().permute(0, 2, 1).reshape(K, N)
        ref = (((a.double() @ dec) * s.double() + term).to(out_dtype).float() + bias.float()).to(out_dtype)
    else:
        ref = torch_ref_dev(a, bp, s, bias, out_dtype)
        ref = (ref.float() + term.to(f_dtype).to(out_dtype).float()).to(out_dtype)
    assert_gemm_close_dev(y, ref, out_dtype, f"{M}x{N}x{K} rank {R}")
    y2 = hk.scaled_mm_hip_any_m_lora(a, bp, s, bias, out_dtype, t, u)
    assert torch.equal(y.view(torch.int16), y2.view(torch.int16))
    ab = a.bfloat16()  # bf16 activations: the bits of their fp16 cast
    yb = hk.scaled_mm_hip_any_m_lora(ab, bp, s, bias, out_dtype, t, u)
    y16 = hk.scaled_mm_hip_any_m_lora(ab.half(), bp, s, bias, out_dtype, t, u)
    assert torch.equal(yb.view(torch.int16), y16.view(torch.int16))


@pytest.mark.parametrize("out_dtype,f_dtype", [(torch.bfloat16, torch.bfloat16), (torch.float16, torch.float16),
                                               (torch.bfloat16, torch.float16), (torch.float16, torch.bfloat16)])
@pytest.mark.parametrize("M,N,K", LORA_SHAPES)
def test_planned_tile_lora(cuda, hk, M, N, K, out_dtype, f_dtype):
    """The rank-R term on every planned tile, against the whole output in float64 with the term in the
    accumulator (tuple route on a large tile) or rounded and added to the result (every other)."""
    _check_lora(cuda, hk, M, N, K, 32 * (1 + (M + N // 16) % 5), out_dtype, f_dtype)


# the lean kernel (loads of 128 ranks in flight; one and two row tiles, one and two workgroups per CU), the tiles whose
# stage buffer holds 64 ranks of both factors (three of those in flight), those that need two (two in flight) and a
# large tile (one)
MANY_RANK_SHAPES = [(5, 528, 512), (16, 4112, 512), (31, 1040, 1024), (63, 224, 128), (33, 128, 2480), (130, 5488, 128),
                    (333, 1712, 3904), (333, 2976, 1664), (97, 4160, 3984), (333, 5408, 1728), (500, 4416, 2368),
                    (777, 5056, 4880), (777, 4064, 2704), (777, 4928, 64), (2000, 6160, 128)]


@pytest.mark.parametrize("R", [96, 192, 224, 256, 320, 416, 1024])
@pytest.mark.parametrize("M,N,K", MANY_RANK_SHAPES)
def test_planned_tile_lora_many_ranks(cuda, hk, M, N, K, R):
    """Ranks around every number of 64-rank chunks in flight, stacks of several hundred among them."""
    _check_lora(cuda, hk, M, N, K, R, torch.bfloat16, torch.bfloat16)
