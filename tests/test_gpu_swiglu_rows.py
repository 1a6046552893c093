"""npu_quant_matmul_swiglu(_quant) on both sides of the row count up to which the ops run the small-M GEMMs and a
SwiGLU pass in place of the fused kernel: the op's bits equal the fused kernel's (through the C ABI)."""
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


@pytest.mark.parametrize("layout", ["kn", "nz"])
@pytest.mark.parametrize("M", [1, 17, 128, 129])
def test_swiglu_rows(ops, M, layout):
    print(f"[case] M={M} {layout}", flush=True)
    I, K = 384, 512
    g = torch.Generator().manual_seed(M)
    x = torch.randint(-128, 128, (M, K), generator=g, dtype=torch.int8).to(DEV)
    w = torch.randint(-128, 128, (K, 2 * I), generator=g, dtype=torch.int8).to(DEV)
    s = (1e-4 + 1e-3 * torch.rand(2 * I, generator=g)).to(DEV)
    pt = (1e-2 * torch.rand(M, generator=g)).to(DEV)
    nz = layout == "nz"
    wd = ops.npu_format_cast(w, ops.ACL_FORMAT_FRACTAL_NZ) if nz else w
    h = ops.npu_quant_matmul_swiglu(x, wd, s, pertoken_scale=pt, output_dtype=torch.bfloat16)
    q, qs = ops.npu_quant_matmul_swiglu_quant(x, wd, s, pertoken_scale=pt, output_dtype=torch.bfloat16)
    L, st = ops.abi(), torch.cuda.current_stream().cuda_stream
    fmt, ld = (ops.ACL_FORMAT_FRACTAL_NZ, 0) if nz else (ops.ACL_FORMAT_ND, 2 * I)
    h2 = torch.empty_like(h)
    assert L.qk_quant_matmul_swiglu(x.data_ptr(), K, wd.data_ptr(), fmt, ld, M, I, K, s.data_ptr(), 2 * I,
                                    pt.data_ptr(), h2.data_ptr(), ops.QK_BF16, st) == 0, ops.last_error()
    n = ctypes.c_size_t(0)
    assert L.qk_quant_matmul_swiglu_quant_workspace_size(M, I, ctypes.byref(n)) == 0
    ws = torch.empty(n.value, dtype=torch.uint8, device=DEV)
    q2, qs2 = torch.empty_like(q), torch.empty_like(qs)
    assert L.qk_quant_matmul_swiglu_quant(x.data_ptr(), K, wd.data_ptr(), fmt, ld, M, I, K, s.data_ptr(), 2 * I,
                                          pt.data_ptr(), ops.QK_BF16, q2.data_ptr(), qs2.data_ptr(), ws.data_ptr(),
                                          n.value, st) == 0, ops.last_error()
    assert torch.equal(h.view(torch.int16), h2.view(torch.int16))
    assert torch.equal(q, q2) and torch.equal(qs.view(torch.int32), qs2.view(torch.int32))
