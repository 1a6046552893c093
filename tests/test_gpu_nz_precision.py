"""fp32-level error of the weight-quant kernels on NZ and [N, K] weights, on the GPU.

Columns k and k + 32 of x are equal and rows k and k + 32 of w opposite (in every 64), so every exact output is 0 and the output is
the error of the kernel's 32-bit sums alone (no 16-bit rounding hides it).  The kernels may sum x * (w + base) raw
over at most 128 rows before the scale and the base's share, base * sum x, come off: one rounding of such a sum errs
by at most u = 2^-24 * (base + max|w|) * sum of |x| over 128 rows.  A fold has 8 of them (four MFMAs for the products,
four for the sum of x) and the K / 128 folds' errors add up as a random walk, so the rms error stays below
8 * sqrt(K / 128) * u with a margin of about five; raw sums over all of K grow K / 128 times as large and miss it.
int8 operands need no base: what 32 rows add the next 32 take off, so the sums stay below 32 rows' |w * x| and each
MFMA errs by less than u0 = 2^-24 * max|w| * sum of |x| over 32 rows, K / 32 of them as a random walk.  With weights
this small a base of 128 makes the sums 64 times as large.
"""
import math

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.fixture(scope="module")
def ops():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import op_plugin_amd
    yield op_plugin_amd
    op_plugin_amd.debug_set_plan("")


def _rms_and_bar(ops, int4, layout, M, N, K, group, dtype, base, top, plan):
    print(f"[case] int4={int4} {layout} M={M} N={N} K={K} G={group} {dtype} plan={plan!r}", flush=True)
    g = torch.Generator().manual_seed(M + K)
    x = torch.randn((M, K // 64, 1, 32), generator=g).abs().to(dtype)
    x = x.expand(M, K // 64, 2, 32).reshape(M, K)
    w = torch.randint(-top, top + 1, (K // 64, 1, 32, N), generator=g, dtype=torch.int8)
    w = torch.cat([w, -w], 1).reshape(K, N)
    if layout == "nk":
        wd = w.t().contiguous().to(DEV).t()
    else:
        wd = ops.npu_convert_weight_to_int4pack(w.to(DEV)) if int4 else w.to(DEV)
        wd = ops.npu_format_cast(wd, ops.ACL_FORMAT_FRACTAL_NZ) if layout == "nz" else wd
    s = torch.ones((K // group, N) if group else (N,), dtype=torch.float16, device=DEV)
    ops.debug_set_plan(plan)
    out = ops.npu_weight_quant_batchmatmul(x.to(DEV), wd, s, antiquant_group_size=group)
    ops.debug_set_plan("")
    rows, roundings = (128, 8) if base else (32, 1)
    u = 2.0 ** -24 * (base + top) * rows * x.float().mean().item()
    rms, bar = out.float().square().mean().sqrt().item(), roundings * math.sqrt(K / rows) * u
    print(f"rms {rms:.3g} bar {bar:.3g}", flush=True)
    return rms, bar


@pytest.mark.parametrize("layout,M,K,group,dtype,base,plan", [
    ("nz", 20, 8192, 0, torch.float16, 1032, "nz_mid=1"),
    ("nz", 64, 8192, 0, torch.float16, 1032, "nz_mid=2"),
    ("nz", 100, 8192, 1024, torch.float16, 1032, "nz_mid=1"),
    ("nz", 40, 8192, 0, torch.bfloat16, 136, "nz_mid=1"),
    ("kn", 70, 8192, 2048, torch.float16, 1032, "nz_mid=1"),
    ("nz", 16, 8192, 0, torch.float16, 1032, ""),       # the decode kernel
    ("nz", 3, 128 * 43, 0, torch.float16, 1032, ""),    # its ragged form
])
def test_int4_long_groups(ops, layout, M, K, group, dtype, base, plan):
    rms, bar = _rms_and_bar(ops, True, layout, M, 272, K, group, dtype, base, 7, plan)
    assert rms <= bar, (rms, bar)


@pytest.mark.parametrize("layout,M,K,group,dtype,plan", [
    ("nz", 100, 8192, 0, torch.float16, "nz_mid=1"),
    ("nk", 40, 8192, 128, torch.bfloat16, "nz_mid=2"),
    ("kn", 70, 64 * 65, 0, torch.float16, "nz_mid=1"),
    ("nz", 200, 64 * 20, 64 * 5, torch.bfloat16, "nz_mid=1"),  # folds of four steps and one
    ("nz", 16, 4096, 0, torch.float16, ""),                    # the decode kernel, even form
    ("nz", 3, 64 * 65, 0, torch.bfloat16, ""),                 # its ragged form
    ("nk", 9, 128 * 43, 128, torch.float16, ""),
    ("nk", 40, 128 * 107, 0, torch.float16, "nz_mid=0"),
])
def test_int8_has_no_base(ops, layout, M, K, group, dtype, plan):
    rms, bar = _rms_and_bar(ops, False, layout, M, 272, K, group, dtype, 0, 2, plan)
    assert rms <= bar, (rms, bar)
