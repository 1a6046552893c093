"""npu_weight_quant_batchmatmul on NZ and [N, K] weights with operands that are not 16-byte aligned, on the GPU.

The workspace query knows only the shape, so it reports the room of the kernels that aligned operands run.  The op
copies what is not aligned (the aligned call's bits); the C entry point runs with the reported workspace whatever the
pointers' alignment.  Shapes of the decode kernel's ragged form, its row chunks and the mid-M kernel.
"""
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
    return op_plugin_amd


def _shift(t, elements=1):
    """The same values, `elements` past a 16-byte boundary, with t's strides."""
    buf = torch.empty(t.numel() + elements, dtype=t.dtype, device=t.device)
    v = buf[elements:].as_strided(t.shape, t.stride(), elements)
    v.copy_(t)
    assert v.data_ptr() % 16 != 0
    return v


def _inputs(ops, int4, layout, M, N, K, group):
    print(f"[case] int4={int4} {layout} M={M} N={N} K={K} G={group}", flush=True)
    g = torch.Generator(device=DEV).manual_seed(M + K)
    x = torch.randn((M, K), generator=g, device=DEV).bfloat16()
    w = torch.randint(*((-8, 8) if int4 else (-127, 128)), (K, N), generator=g, device=DEV, dtype=torch.int8)
    if layout == "nk":
        wd = w.t().contiguous().t()
    else:
        wd = ops.npu_format_cast(ops.npu_convert_weight_to_int4pack(w) if int4 else w, ops.ACL_FORMAT_FRACTAL_NZ)
    rows = (K // group, N) if group else (N,)
    s = ((5e-3 if int4 else 3e-4) * (1 + torch.rand(rows, generator=g, device=DEV))).half()
    o = (2 * torch.rand(rows, generator=g, device=DEV) - 1).half()
    return x, wd, s, o


CASES = [
    (True, "nz", 1, 4096, 11008, 128),    # the decode kernel's ragged form
    (True, "nz", 100, 272, 13696, 128),   # the mid-M kernel, K splits
    (True, "nz", 16, 272, 128 * 43, 64),
    (True, "nz", 20, 48, 256, 0),
    (False, "nz", 3, 272, 64 * 65, 0),
    (False, "nz", 100, 272, 64 * 13, 64),
    (False, "nk", 3, 272, 128 * 43, 128),
    (False, "nk", 130, 256, 128 * 5, 0),
]


@pytest.mark.parametrize("int4,layout,M,N,K,group", CASES)
def test_op(ops, int4, layout, M, N, K, group):
    x, w, s, o = _inputs(ops, int4, layout, M, N, K, group)
    call = lambda x, w, s, o: ops.npu_weight_quant_batchmatmul(x, w, s, o, antiquant_group_size=group)
    ref = call(x, w, s, o)
    for a in [(_shift(x), w, s, o), (x, w, _shift(s), o), (x, w, s, _shift(o, 4)), (_shift(x, 4), w, _shift(s), _shift(o))]:
        assert torch.equal(call(*a).view(torch.int16), ref.view(torch.int16))
    if layout == "nk":
        assert torch.equal(call(x, _shift(w.t(), 3).t(), s, o).view(torch.int16), ref.view(torch.int16))


@pytest.mark.parametrize("int4,layout,M,N,K,group", CASES)
def test_abi(ops, int4, layout, M, N, K, group):
    x, w, s, o = _inputs(ops, int4, layout, M, N, K, group)
    ref = ops.npu_weight_quant_batchmatmul(x, w, s, o, antiquant_group_size=group).float()
    code = ops.QK_I4_NZ if int4 else ops.QK_I8_NK if layout == "nk" else ops.QK_I8_NZ
    L, n = ops.abi(), ctypes.c_size_t(0)
    assert L.qk_weight_quant_bmm_workspace_size(M, N, K, code, group, ctypes.byref(n)) == 0
    ws = torch.empty(max(1, n.value), dtype=torch.uint8, device=DEV)
    out = torch.empty((M, N), dtype=torch.bfloat16, device=DEV)
    for a in [(_shift(x), w, s, o, out), (x, w, _shift(s), _shift(o), out), (x, w, s, o, _shift(out))]:
        a[-1].zero_()
        rc = L.qk_weight_quant_bmm(a[0].data_ptr(), ops.QK_BF16, a[1].data_ptr(), code, a[2].data_ptr(), a[3].data_ptr(),
                                   ops.QK_F16, M, N, K, group, None, 0, a[4].data_ptr(), ops.QK_BF16, ws.data_ptr(),
                                   n.value, torch.cuda.current_stream().cuda_stream)
        assert rc == 0, ops.last_error()
        torch.testing.assert_close(a[-1].float(), ref, rtol=1e-2, atol=1e-2)
