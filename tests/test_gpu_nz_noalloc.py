"""qk_weight_quant_bmm_noalloc on NZ and [N, K] weights, on the GPU: what its 16 MB scratch must not be asked for, and
what it runs where the planned workspace does not fit."""
import ctypes

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


def _run(ops, int4, layout, M, N, K, group, plan=""):
    """(query bytes, noalloc output, the op's output under `plan`)"""
    print(f"[case] int4={int4} {layout} M={M} N={N} K={K} G={group}", flush=True)
    g = torch.Generator(device=DEV).manual_seed(M + K)
    x = torch.randn((M, K), generator=g, device=DEV).bfloat16()
    w = torch.randint(*((-8, 8) if int4 else (-127, 128)), (K, N), generator=g, device=DEV, dtype=torch.int8)
    if layout == "nk":
        wd, code = w.t().contiguous().t(), ops.QK_I8_NK
    else:
        wd = ops.npu_format_cast(ops.npu_convert_weight_to_int4pack(w) if int4 else w, ops.ACL_FORMAT_FRACTAL_NZ)
        code = ops.QK_I4_NZ if int4 else ops.QK_I8_NZ
    s = ((5e-3 if int4 else 3e-4) * (1 + torch.rand((K // group, N) if group else (N,), generator=g, device=DEV))).half()
    L, n = ops.abi(), ctypes.c_size_t(0)
    assert L.qk_weight_quant_bmm_workspace_size(M, N, K, code, group, ctypes.byref(n)) == 0
    out = torch.empty((M, N), dtype=torch.bfloat16, device=DEV)
    rc = L.qk_weight_quant_bmm_noalloc(x.data_ptr(), ops.QK_BF16, wd.data_ptr(), code, s.data_ptr(), None, ops.QK_F16, M,
                                       N, K, group, None, 0, out.data_ptr(), ops.QK_BF16,
                                       torch.cuda.current_stream().cuda_stream)
    assert rc == 0, ops.last_error()
    ops.debug_set_plan(plan)
    ref = ops.npu_weight_quant_batchmatmul(x, wd, s, antiquant_group_size=group)
    ops.debug_set_plan("")
    return n.value, out, ref


@pytest.mark.parametrize("int4,M,N,K", [(True, 16, 11008, 4096), (False, 3, 4096, 64 * 65)])
def test_short_groups_need_no_scratch(ops, int4, M, N, K):
    """64-row groups, whose ND weight would exceed the scratch: the decode kernel, no workspace."""
    need, out, ref = _run(ops, int4, "nz", M, N, K, 64)
    assert need == 0 and K * N // (2 if int4 else 1) > ops.QK_NOALLOC_SCRATCH_BYTES
    assert torch.equal(out.view(torch.int16), ref.view(torch.int16))


@pytest.mark.parametrize("int4,layout,M,N,K", [
    (True, "nz", 60, 8192, 8192),    # the decode kernel
    (False, "nk", 90, 4096, 11008),  # its row chunks
])
def test_mid_splits_do_not_fit(ops, int4, layout, M, N, K):
    """The mid-M kernel's partial tiles exceed the scratch: the kernels without it, as with that kernel switched off."""
    need, out, ref = _run(ops, int4, layout, M, N, K, 128, plan="nz_mid=0")
    assert need > ops.QK_NOALLOC_SCRATCH_BYTES
    assert torch.equal(out.view(torch.int16), ref.view(torch.int16))
    mid = _run(ops, int4, layout, M, N, K, 128)[2]
    assert not torch.equal(mid.view(torch.int16), ref.view(torch.int16))
    torch.testing.assert_close(out.float(), mid.float(), rtol=1e-2, atol=1e-2)
